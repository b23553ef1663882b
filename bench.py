#!/usr/bin/env python3
"""Benchmark: the RidgeFill late-layer fill of a Llama-3.1-8B-shaped 32K prompt on one MI355X.

Workload (synthetic, seeded; rfill.synth): hidden 4096, 32 query / 8 KV heads, head_dim 128, RoPE
theta 5e5, split at layer 16, 16 late layers each with a ridge map W_l = I + 0.02 N(0, 1/4096) and bias
N(0, 1e-3); prompt 32768 rows, exact tail 4096, so P = 28672 filled rows. One step = the fill of all
16 late layers from h_split already resident in HBM: per layer rf_map_apply (x = b W^T + c, with the
rows' RMSNorm statistics) then rf_norm_kv_write (RMSNorm, K / V projections, RoPE, cache write).

Reported: filled tokens/s = P * steps / elapsed; the dominant kernel's roofline (rf_map_apply, MFMA
bound, 2 P H^2 flop per launch over its mean HIP-event duration on the launch stream); the second
fill kernel and the standalone RoPE + KV-write kernel (HBM bound) beside it; library ceilings (a plain
hipBLASLt GEMM of the same shape and a device copy); and the CPU baseline: the oracle's fill (the
reference op sequence in torch on the host cores) timed on a bounded row sample.
"""
import argparse
import json
import os
import statistics
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
for p in (ROOT, ROOT / "ridgefill-data_amd"):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))

import torch  # noqa: E402

METRIC = "filled tokens/s (16-layer fill, 8B, 32K); MFMA % bf16 peak; HBM GB/s"
PEAK_BF16 = 2.5e15        # MI355X dense bf16 MFMA, FLOP/s
PEAK_HBM = 8.0e12         # MI355X HBM3E, B/s
N_ROWS, TAIL, SPLIT = 32768, 4096, 16


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


class KernelTimer:
    """Start / end HIP events around launches on the current stream; mean duration per name."""

    def __init__(self):
        self.ev = {}

    def run(self, name, fn):
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        out = fn()
        e.record()
        self.ev.setdefault(name, []).append((s, e))
        return out

    def mean_s(self, name):
        pairs = self.ev.get(name, [])
        return sum(s.elapsed_time(e) for s, e in pairs) / max(1, len(pairs)) / 1e3

    def median_s(self, name):
        ts = sorted(s.elapsed_time(e) for s, e in self.ev.get(name, []))
        return ts[len(ts) // 2] / 1e3 if ts else 0.0


def build_workload(dev):
    from rfill import synth
    from rfill.kva import Arm, Projector
    from rfill.model import FillModel
    cfg = synth.LLAMA_8B
    log("generating the synthetic workload on the GPU")
    w = synth.dense_fill(cfg, SPLIT, N_ROWS, TAIL, device=dev)
    model = FillModel(cfg, w["tensors"], dev, layers=w["layers"])
    arm = Arm("ridgefill", split=SPLIT, tail=TAIL, fill="proj", projector=Projector(SPLIT, w["maps"], w["biases"]))
    return cfg, w, model, arm


def fill_step(model, arm, b, pos, cs, xbuf, sbuf, caches, timer=None):
    """One step: the 16-layer fill (the hot path of finish() for the ridgefill arm, no exact rows),
    scheduled as fill_late schedules it (rfill.kva.serial with ATTN_GROUP): groups of consecutive late
    layers, each group's maps in one launch (rf_map_apply_batch), then the group's fused norm + K / V + RoPE
    cache writes in one launch (rf_norm_kv_write_batch), all on the current stream. Rows go to slot 0 of
    caches sized once, so every step writes the same slots."""
    from rfill import ops
    from rfill.kva import ATTN_GROUP
    layers = list(range(arm.split, model.n_layers))
    for g0 in range(0, len(layers), ATTN_GROUP):
        ids = layers[g0:g0 + ATTN_GROUP]
        n = len(ids)
        f = lambda: arm.projector.apply_batch(ids, b, xbuf[:n], sbuf[:n])    # noqa: E731
        f() if timer is None else timer.run("rf_map_apply_batch", f)
        g = lambda: ops.norm_kv_write_batch(  # noqa: E731
            xbuf[:n], sbuf[:n], model.eps, [model.W[i]["wkv"] for i in ids], model.n_kv, model.head_dim,
            [model.W[i].get("k_norm") for i in ids], model.knorm_kind, cs, [caches[i]["kbuf"] for i in ids],
            [caches[i]["vbuf"] for i in ids], 0)
        g() if timer is None else timer.run("rf_norm_kv_write_batch", g)


def ceilings(dev, P, H):
    """Library GEMM (hipBLASLt via torch) of the map's shape, a device-to-device copy, and the MFMA throughput
    the power limit allows (rf_mfma_ceiling: back-to-back bf16 MFMAs on register operands, 2 waves per SIMD)."""
    from rfill import ops
    a = torch.randn(P, H, device=dev, dtype=torch.bfloat16)
    w = torch.randn(H, H, device=dev, dtype=torch.bfloat16)
    out = torch.empty(P, H, device=dev, dtype=torch.bfloat16)
    # two forms of the same product (torch may route them to different library kernels); the faster median
    forms = {"matmul_out": lambda: torch.matmul(a, w.t(), out=out),
             "linear": lambda: torch.nn.functional.linear(a, w)}
    t = KernelTimer()
    for name, f in forms.items():
        for _ in range(3):
            f()
        torch.cuda.synchronize()
        for _ in range(10):
            t.run(name, f)
    torch.cuda.synchronize()
    gemm_form = min(forms, key=t.median_s)
    src_bytes = 1 << 30
    src = torch.empty(src_bytes, dtype=torch.uint8, device=dev)
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    for _ in range(10):
        t.run("copy", lambda: dst.copy_(src))
    del src, dst
    blocks, iters = 512, 20000
    acc = torch.empty(blocks * 256, dtype=torch.float32, device=dev)
    for _ in range(2):
        ops.mfma_ceiling(blocks, iters, acc)
    for _ in range(5):
        t.run("mfma", lambda: ops.mfma_ceiling(blocks, iters, acc))
    torch.cuda.synchronize()
    return {"hipblaslt_gemm_tflops": round(2 * P * H * H / t.median_s(gemm_form) / 1e12, 1),
            "gemm_form": gemm_form,
            "gemm_forms_tflops": {k: round(2 * P * H * H / t.median_s(k) / 1e12, 1) for k in forms},
            "copy_gbs": round(2 * src_bytes / t.mean_s("copy") / 1e9, 1),
            "gemm_shape": [P, H, H],
            "mfma_power_ceiling_tflops": round(blocks * 4 * 4 * iters * 32768 / t.mean_s("mfma") / 1e12, 1)}


def dequant_bench(dev, rows=2560, width=10240, maps=24):
    """Expansion of the release's i8_row128 maps (24 late layers of [2560, 10240] int8 codes with
    per-128-column bf16 scales) to bf16 maps: HBM bound, algorithmic bytes per map = codes (1 B per
    entry) + scales (2 B per 128 entries) read + the bf16 map (2 B per entry) written."""
    from rfill import ops
    g = torch.Generator(device=dev).manual_seed(30)
    codes = torch.randint(-128, 128, (rows, width), generator=g, device=dev, dtype=torch.int16).to(torch.int8)
    scale = (torch.rand(rows, width // 128, generator=g, device=dev) * 1e-3).to(torch.bfloat16)
    out = torch.empty(rows, width, dtype=torch.bfloat16, device=dev)
    for _ in range(3):
        ops.dequant_i8_rows(codes, scale, 128, out=out)
    torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(maps):
        ops.dequant_i8_rows(codes, scale, 128, out=out)
    e.record()
    torch.cuda.synchronize()
    sec = s.elapsed_time(e) / 1e3 / maps
    byts = rows * width * 3 + rows * (width // 128) * 2
    return {"kernel": "rf_dequant_i8_rows", "bound": "hbm", "achieved": round(byts / sec / 1e9, 1),
            "peak": PEAK_HBM / 1e9, "unit": "GB/s", "frac": round(byts / sec / PEAK_HBM, 4),
            "bytes_per_launch": byts, "mean_us": round(sec * 1e6, 2), "maps": maps,
            "ms_all_maps": round(sec * maps * 1e3, 3)}


def gguf_bench(dev, rows=5120, width=5120, maps=48):
    """rf_dequant_gguf_rows on the GGUF adapters' map tensors: Q8_0 (the fitted adapters) and F16 (the
    identity one), [5120, 5120] each (the 27B kit's width), HBM-bound: Q8_0 reads 34 bytes per 32 values
    and writes 2 bytes per value; F16 reads 2 and writes 2."""
    from rfill import ops
    g = torch.Generator(device=dev).manual_seed(33)
    out = torch.empty(rows, width, dtype=torch.bfloat16, device=dev)
    res = {}
    for name, gt, row_bytes in (("q8_0", 8, width // 32 * 34), ("f16", 1, 2 * width)):
        raw = torch.randint(0, 256, (rows, row_bytes), generator=g, device=dev, dtype=torch.int32).to(torch.uint8)
        if gt == 8:                                  # finite fp16 scales in every block's first two bytes
            blk = raw.view(rows, width // 32, 34)
            blk[:, :, 0] = 0
            blk[:, :, 1] = 0x20
        else:
            raw.view(rows, width, 2)[:, :, 1] &= 0x3F
        for _ in range(3):
            ops.dequant_gguf_rows(raw, gt, width, out=out)
        torch.cuda.synchronize()
        reps = 20
        s0, e0 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s0.record()
        for _ in range(reps):
            ops.dequant_gguf_rows(raw, gt, width, out=out)
        e0.record()
        torch.cuda.synchronize()
        sec = s0.elapsed_time(e0) / 1e3 / reps
        byts = rows * row_bytes + 2 * rows * width
        res[name] = {"mean_us": round(sec * 1e6, 1), "achieved": round(byts / sec / 1e9, 1), "unit": "GB/s",
                     "frac": round(byts / sec / PEAK_HBM, 4), "bytes_per_launch": byts,
                     "ms_per_adapter": round(sec * maps * 1e3, 3)}
    return {"kernel": "rf_dequant_gguf_rows", "bound": "hbm", "workload": f"{maps} GGUF maps [{rows}, {width}]", **res}


def window_mass_bench(dev, n=32768, w=64, hq=32, hkv=8, d=128, layers=4):
    """The qattn selector's mass (rf_window_mass) at the 8B 32K prompt: 64 window rows x 32 query heads over
    32768 cached keys, for each of the 4 exact lower layers. Algorithmic work per layer: the scores
    2 w hq n d FLOP; the kernel forms them twice (row statistics, then column sums)."""
    from rfill import ops
    g = torch.Generator(device=dev).manual_seed(31)
    q = (0.5 * torch.randn(w, hq * d, generator=g, device=dev)).to(torch.bfloat16)
    kb = (0.5 * torch.randn(hkv, n + 64, d, generator=g, device=dev)).to(torch.bfloat16)
    mass = torch.zeros(n, dtype=torch.float64, device=dev)
    ws = torch.empty(ops.window_mass_workspace_bytes(w, hq, hkv, d, n), dtype=torch.uint8, device=dev)
    for _ in range(3):
        ops.window_mass(q, n - w, kb, hq, d ** -0.5, mass, workspace=ws)
    torch.cuda.synchronize()
    reps = 20
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(reps):
        ops.window_mass(q, n - w, kb, hq, d ** -0.5, mass, workspace=ws)
    e.record()
    torch.cuda.synchronize()
    sec = s.elapsed_time(e) / 1e3 / reps
    flop = 2 * w * hq * n * d
    return {"kernel": "rf_window_mass", "workload": f"qattn mass: {w} window rows x {hq} heads over {n} keys, d {d}",
            "bound": "mfma", "mean_us": round(sec * 1e6, 1), "achieved_tflops": round(flop / sec / 1e12, 1),
            "frac": round(flop / sec / PEAK_BF16, 4), "flop_per_launch": flop,
            "ms_per_prompt": round(sec * layers * 1e3, 3), "layers": layers}


def kv_write_bench(model, dev, P, layer):
    """The standalone RoPE + K / V cache write (fill_kv) at the workload's shape: HBM bound,
    algorithmic bytes 4 Hkv d 2 per row (read pre-RoPE K, V; write post-RoPE K, V)."""
    from rfill import ops
    hkv, d = model.n_kv, model.head_dim
    k = torch.randn(P, hkv, d, device=dev).to(torch.bfloat16)
    v = torch.randn(P, hkv, d, device=dev).to(torch.bfloat16)
    cs = model.rope_table(torch.arange(P, device=dev))
    kb = torch.empty(hkv, P + 64, d, dtype=torch.bfloat16, device=dev)
    vb = torch.empty_like(kb)
    for _ in range(3):
        ops.rope_kv_write(k, v, cs, kb, vb, 0)
    torch.cuda.synchronize()
    reps = 50
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(reps):                 # back to back: the host enqueues faster than a launch runs
        ops.rope_kv_write(k, v, cs, kb, vb, 0)
    e.record()
    torch.cuda.synchronize()
    sec = s.elapsed_time(e) / 1e3 / reps
    byts = 4 * hkv * d * 2 * P
    return {"kernel": "rf_rope_kv_write", "bound": "hbm", "achieved": round(byts / sec / 1e9, 1),
            "peak": PEAK_HBM / 1e9, "unit": "GB/s", "frac": round(byts / sec / PEAK_HBM, 4),
            "bytes_per_launch": byts, "mean_us": round(sec * 1e6, 2)}


def _cpu_info():
    """(threads this process may use, the machine's CPU count, the CPU model name)."""
    try:
        usable = len(os.sched_getaffinity(0))
    except AttributeError:
        usable = os.cpu_count() or 1
    env = os.environ.get("OMP_NUM_THREADS")
    if env and env.isdigit() and int(env) > 0:
        usable = min(usable, int(env))
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return usable, os.cpu_count(), model


def cpu_baseline(cfg, w, layer, budget_s=8.0, rows=1024):
    """The oracle's fill (reference op sequence: F.linear map, rms_norm, K / V F.linear, RoPE, cache append) on
    the host, for `rows`-row blocks of one late layer until `budget_s` has passed, in bf16 (the reference's
    model dtype) and in fp32; scaled to filled tokens/s of the 16-layer fill. Threads: every core this
    process may use (the affinity mask, capped by OMP_NUM_THREADS)."""
    from oracle import model as OM
    threads, machine, model = _cpu_info()
    torch.set_num_threads(threads)
    t = {k: v.cpu() for k, v in w["tensors"].items() if f"layers.{layer}." in k}
    pos = torch.arange(rows)
    res = {}
    for dt in (torch.bfloat16, torch.float32):
        b = w["h_split"][:rows].cpu().to(dt)
        W, c = w["maps"][layer].cpu().to(dt), w["biases"][layer].cpu().to(dt)
        om = OM.OracleModel(cfg, t, dtype=dt, layers=[layer])
        done, t0 = 0, time.perf_counter()
        while True:
            cache = om.new_cache()
            x = torch.nn.functional.linear(b, W, c)
            om.fill(layer, x, pos, cache)
            done += rows
            el = time.perf_counter() - t0
            if el >= budget_s:
                break
        res[str(dt).split(".")[1]] = (done / el / (cfg["num_hidden_layers"] - SPLIT), done, el)
    rate, done, el = res["bfloat16"]
    return {"value": round(rate, 2), "unit": "filled tokens/s", "cores": threads, "kind": "port",
            "fp32_value": round(res["float32"][0], 2), "machine_cpus": machine, "cpu_model": model,
            "sample": f"oracle fill of one late layer (the reference's op sequence), {rows}-row blocks: "
                      f"bf16 {done // rows} blocks in {el:.1f} s, fp32 {res['float32'][1] // rows} blocks in "
                      f"{res['float32'][2]:.1f} s; scaled by 1/16 layers; torch {torch.__version__}"}


def cpu_exact_rows_baseline(n=32768, split=18, tail=4096, frac=0.01, reps=2):
    """The Qwen3-8B-shaped 32K fill with 1 % exact rows on the host, one late layer as the reference runs it
    (code/kva/kva.py:413-437): x = F.linear(b, W, c), x.index_copy(0, R, h_split[R]), then layer_rows (the
    fill of all P rows -- norm, K / V, k_norm, RoPE, cache append -- and the rows' full layer: queries,
    attention over the filled keys, o_proj, the MLP), in bf16, timed `reps` times and scaled to the 18 late
    layers; the same layer without exact rows (map + fill) for the plain fill's rate. The oracle's op
    sequence on every core this process may use."""
    from oracle import model as OM
    from rfill import synth
    threads, _, _ = _cpu_info()
    torch.set_num_threads(threads)
    cfg = synth.QWEN3_8B
    L = cfg["num_hidden_layers"] - split
    P = n - tail
    t, W, c = synth.layer_weights(cfg, split, "cpu", full=True)
    b = synth.hidden_states(n, cfg["hidden_size"])[:P]
    rows = torch.randperm(P, generator=torch.Generator().manual_seed(13))[:int(round(frac * P))].sort().values
    om = OM.OracleModel(cfg, t, dtype=torch.bfloat16, layers=[split])
    pos = torch.arange(P)
    times = {"plain": [], "exact": []}
    with torch.no_grad():
        for _ in range(reps):
            for name in ("plain", "exact"):
                cache = om.new_cache()
                t0 = time.perf_counter()
                x = torch.nn.functional.linear(b, W, c)
                if name == "exact":
                    x = x.index_copy(0, rows, b[rows])
                    om.layer_rows(split, x, pos, rows, cache)
                else:
                    om.fill(split, x, pos, cache)
                times[name].append(time.perf_counter() - t0)
    te, tp = min(times["exact"]), min(times["plain"])
    return {"value": round(P / (te * L), 2), "unit": "filled tokens/s", "cores": threads, "kind": "port",
            "value_without_exact_rows": round(P / (tp * L), 2), "exact_rows": len(rows),
            "sample": f"oracle layer {split} of the 32K Qwen3-8B-shaped fill ({P} rows, {len(rows)} exact), bf16: "
                      f"{te:.2f} s with the exact rows' layer_rows, {tp:.2f} s without (best of {reps}); scaled "
                      f"by {L} late layers"}


def cpu_hybrid_baseline(n=32768, split=24, tail=4096, seg=8192):
    """The Qwen3.5-shaped hybrid's 32K fill on the host, bounded: one 8192-row segment (GDN_ROWS,
    code/kva/model.py:31) of one GDN layer -- map, in-projections, causal conv, the chunked delta rule's
    Python chunk loop (code/kva/ops.py:199-262) -- and of one attention layer (map, K / V, RoPE, append),
    in bf16 with the fp32 recurrence, scaled by P / 8192 segments and the 18 GDN + 6 attention late layers.
    The oracle's op sequence on every core this process may use."""
    from oracle import model as OM
    from rfill import synth
    threads, _, _ = _cpu_info()
    torch.set_num_threads(threads)
    cfg = synth.QWEN35_HYBRID
    P = n - tail
    kinds = {i: ("gdn" if cfg["layer_types"][i] == "linear_attention" else "attn")
             for i in range(split, cfg["num_hidden_layers"])}
    g = next(i for i in kinds if kinds[i] == "gdn")
    a = next(i for i in kinds if kinds[i] == "attn")
    w = synth.hybrid_fill(cfg, split, seg, 0, device="cpu", only=(g, a))
    n_gdn = sum(k == "gdn" for k in kinds.values())
    n_attn = len(kinds) - n_gdn
    t = {k: v for k, v in w["tensors"].items() if f"layers.{g}." in k or f"layers.{a}." in k}
    om = OM.OracleModel(cfg, t, dtype=torch.bfloat16, layers=[g, a])
    b = w["h_split"][:seg]
    pos = torch.arange(seg)
    took = {}
    with torch.no_grad():
        for i in (g, a):
            cache = om.new_cache()
            t0 = time.perf_counter()
            om.fill(i, torch.nn.functional.linear(b, w["maps"][i], w["biases"][i]), pos, cache)
            took[i] = time.perf_counter() - t0
    total = P / seg * (n_gdn * took[g] + n_attn * took[a])
    return {"value": round(P / total, 2), "unit": "filled tokens/s", "cores": threads, "kind": "port",
            "sample": f"oracle fill of one {seg}-row segment, bf16: GDN layer {g} {took[g]:.2f} s (map, in-projections, "
                      f"conv, chunked delta rule), attention layer {a} {took[a]:.2f} s; scaled by {P / seg:.2f} "
                      f"segments x ({n_gdn} GDN + {n_attn} attention) late layers"}


def cpu_fit_baseline(d=4096, targets=16, block=8192, lams=(1e-4, 1e-3, 1e-2)):
    """The reference's fit on the host (code/kva/ridge.py:44-62, 80-105), bounded: one 8192-row block of
    centred fp32 GEMMs into fp64 (X^T X and the 16 X^T Y_l) scaled to the 256 blocks of 2,097,152 rows; the
    fp64 eigendecomposition timed in full, the solve of one target for 3 lambdas timed and scaled by 16."""
    from rfill import synth
    threads, _, _ = _cpu_info()
    torch.set_num_threads(threads)
    maps = synth.fit_maps(d, 1, device="cpu")
    x, ys = synth.fit_chunk(0, block, d, maps, device="cpu")
    xc = x.float() - x.float().mean(0)
    yc = ys[0].float() - ys[0].float().mean(0)
    sxx = torch.zeros(d, d, dtype=torch.float64)
    sxy = torch.zeros(d, d, dtype=torch.float64)
    t0 = time.perf_counter()
    sxx += (xc.T @ xc).double()
    sxy += (xc.T @ yc).double()
    t_two = time.perf_counter() - t0
    t_block = t_two / 2 * (1 + targets)
    n_blocks = 2097152 // block
    c = sxx + torch.eye(d, dtype=torch.float64) * float(sxx.diagonal().mean())
    t0 = time.perf_counter()
    e, v = torch.linalg.eigh(c)
    t_eigh = time.perf_counter() - t0
    t0 = time.perf_counter()
    a = v.T @ sxy
    for lam in lams:
        v @ (a / (e + lam * float(e.mean()))[:, None])
    t_target = time.perf_counter() - t0
    total = t_block * n_blocks + t_eigh + t_target * targets
    return {"value": round(total, 1), "unit": "s per fit", "cores": threads, "kind": "port",
            "accumulate_s": round(t_block * n_blocks, 1), "solve_s": round(t_eigh + t_target * targets, 1),
            "sample": f"one {block}-row block of 2 of the 17 fp32 GEMMs ({t_two:.2f} s) scaled to 17 GEMMs x "
                      f"{n_blocks} blocks; fp64 eigh of [{d}, {d}] ({t_eigh:.2f} s) + one target's solve for 3 "
                      f"lambdas ({t_target:.2f} s) x {targets}"}


def fit_bench(dev, chunks=3, rows=65536, d=4096, targets=16, lams=(1e-4, 1e-3, 1e-2)):
    """The closed-form fit at the 8B-width shape (d 4096, 16 targets, 64K-row chunks of Student-t rows):
    `chunks` of the 32 chunks of 2,097,152 rows are generated (untimed) and accumulated in the reference's
    8192-row blocks (timed: transposes with centring, column sums and the MFMA Gram / cross accumulation
    into fp64; X^T X on its block-upper tiles only, since it is symmetric). Chunk 0 also carries the one-time costs (the first block's statistics that pick the shifts
    and the centred channels, the accumulators' allocation); the later chunks are the steady state the
    projection uses. Then the fp64 solve of every target for 3 lambdas (timed cold, as a fit runs it, and once
    more with its device memory cached: the difference is the allocation of W and the workspace). Work per chunk:
    2 rows d^2 (1 + targets) flop counted (gram_tflops); executed, X^T X takes only its block-upper 256 x 256
    tiles (gram_executed_tflops)."""
    from rfill import ridge, synth
    maps = synth.fit_maps(d, targets, device=dev)
    stats = ridge.RidgeStats(0, list(range(targets)), d, device=dev)
    times = []
    for c in range(chunks):
        x, ys = synth.fit_chunk(c, rows, d, maps, device=dev)
        torch.cuda.synchronize()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        stats.add(x, dict(enumerate(ys)))
        e.record()
        torch.cuda.synchronize()
        times.append(s.elapsed_time(e) / 1e3)
        del x, ys
    steady = sum(times[1:]) / max(1, len(times) - 1)
    flop = 2.0 * rows * d * d * (1 + targets)
    tiles = d // 256
    flop_exec = 2.0 * rows * d * d * targets + 2.0 * rows * 256 * 256 * (tiles * tiles - tiles * (tiles - 1) // 2)
    t0 = time.perf_counter()
    fit = ridge.RidgeFit(stats.state(device=dev), device=dev)
    fit.layers(range(targets), lams)
    torch.cuda.synchronize()
    t_solve = time.perf_counter() - t0
    del fit
    t0 = time.perf_counter()                  # again, with the first solve's device memory cached by torch
    fit = ridge.RidgeFit(stats.state(device=dev), device=dev)
    fit.layers(range(targets), lams)
    torch.cuda.synchronize()
    t_warm = time.perf_counter() - t0
    return {"workload": f"ridge fit: d {d}, {targets} targets, {chunks} x {rows}-row chunks of 32 (timed sample), "
                        f"8192-row blocks",
            "first_chunk_s": round(times[0], 4), "steady_chunk_s": round(steady, 4),
            "gram_tflops": round(flop / steady / 1e12, 1), "gram_frac_bf16_peak": round(flop / steady / PEAK_BF16, 4),
            "gram_executed_tflops": round(flop_exec / steady / 1e12, 1),
            "gram_executed_frac_bf16_peak": round(flop_exec / steady / PEAK_BF16, 4),
            "centred_channels_x": stats.cen_x.s, "solve_s": round(t_solve, 3), "solve_warm_s": round(t_warm, 3),
            "projected_full_fit_s": round(times[0] + steady * 31 + t_solve, 2)}


def capture_bench(dev, split=SPLIT, n=8192, lams=9):
    """The fit's capture and lambda selection at the Llama-3.1-8B shape (32 layers, random weights): one
    n-token calibration document through the exact forward (layers 0 .. 30) with every input of layers
    16 .. 31 transposed into the Gram block, then the block's one MFMA Gram launch for split 16
    (X^T [H, n] times [H_16 .. H_31]^T: 2 n H (16 H) flop into fp64); and one n-token held-out document
    scored for `lams` maps + the identity on all 16 late layers (per layer and candidate: the map, the
    K | V reads GEMM and rf_read_cosine)."""
    from rfill import fit, synth
    from rfill.model import FillModel
    cfg = synth.LLAMA_8B
    model = FillModel(cfg, synth.full_model(cfg, device=dev), dev)
    L, H = cfg["num_hidden_layers"], cfg["hidden_size"]
    g = torch.Generator().manual_seed(17)
    doc = torch.randint(0, cfg["vocab_size"], (n,), generator=g)
    cap = fit.Capture(model, [split])
    cap.add_document(doc)                 # warm-up: packs the layers, allocates the block
    cap.flush()
    torch.cuda.synchronize()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
    ev[0].record()
    cap.add_document(doc)
    ev[1].record()
    cap.flush()
    ev[2].record()
    torch.cuda.synchronize()
    t_fwd, t_gram = ev[0].elapsed_time(ev[1]) / 1e3, ev[1].elapsed_time(ev[2]) / 1e3
    gram_flop = 2.0 * n * H * (L - split) * H
    del cap
    gm = torch.Generator(device=dev).manual_seed(18)
    maps = {lam: {i: ((torch.eye(H, device=dev) + 0.02 * torch.randn(H, H, generator=gm, device=dev) / H ** 0.5)
                      .to(torch.bfloat16), torch.zeros(H, dtype=torch.bfloat16, device=dev))
                  for i in range(split, L)} for lam in fit.LAMBDAS[:lams]}
    fit.read_scores(model, [doc[: n // 4]], split, maps)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    fit.read_scores(model, [doc], split, maps)
    torch.cuda.synchronize()
    t_sel = time.perf_counter() - t0
    return {"workload": f"llama-3.1-8b-shaped capture: {n}-token document, exact forward of layers 0..{L - 2}, "
                        f"Gram of split {split} over layers {split}..{L - 1}; selection of {lams} maps + identity "
                        f"on one {n}-token held-out document",
            "capture_tokens_per_s": round(n / (t_fwd + t_gram), 1), "ms_forward_and_transpose": round(t_fwd * 1e3, 2),
            "ms_gram": round(t_gram * 1e3, 2), "gram_tflops": round(gram_flop / t_gram / 1e12, 1),
            "gram_frac_bf16_peak": round(gram_flop / t_gram / PEAK_BF16, 4),
            "ms_select_per_doc": round(t_sel * 1e3, 1)}


def hybrid_bench(dev, reps=12, split=24, n_rows=32768, tail=4096):
    """The Gated-DeltaNet hybrid's late-layer fill (hidden 2048; layers 24..47 = 18 GDN + 6 attention;
    GDN 16 key / 32 value heads of 128, attention 2 KV heads of 256; P = 28672 filled rows from zero
    state), timed as finish() runs it (fill_late: groups of 8 late layers): per layer rf_map_apply, then the
    GDN fill (rf_norm_linear in-projection + the delta-rule fill, two GDN layers per rf_gdn_fill_batch) or
    the attention fill (rf_norm_kv_write). One cache serves every repetition (its K / V buffers allocated
    by the warm-up fill, then reset to no rows; GDN states start from zero), each repetition timed with HIP
    events on the launch stream; the figure is their median, and every repetition's time is reported.
    Counted work per filled row (the reference's accounting): GDN layer 2 H (2 nk dk + nv dv + 2 nv) + 2 H^2
    + 2 K C + 6 nv dk dv flop, attention layer 2 H^2 + 2 H (2 Hkv d). The per-layer means come from a
    second, layer-by-layer pass (one GDN layer at a time)."""
    from rfill import ops, synth
    from rfill.kva import Arm, Projector, fill_late
    from rfill.model import FillModel
    cfg = synth.QWEN35_HYBRID
    w = synth.hybrid_fill(cfg, split, n_rows, tail, device=dev)
    model = FillModel(cfg, w["tensors"], dev, layers=w["layers"])
    proj = Projector(split, w["maps"], w["biases"])
    arm = Arm("ridgefill", split=split, tail=tail, fill="proj", projector=proj)
    P, H = w["P"], cfg["hidden_size"]
    b = w["h_split"][:P]
    pos = torch.arange(P, device=dev)
    cs = model.rope_table(pos)
    x = torch.empty(P, H, dtype=torch.bfloat16, device=dev)
    ssq = torch.empty(P, ops.ssq_parts(H), dtype=torch.float32, device=dev)
    nk, nv, dk, dv = model.nk, model.nv, model.dk, model.dv
    C = 2 * nk * dk + nv * dv

    def step(timer=None):
        caches = model.new_cache()
        for i in w["layers"]:
            kind = model.layer_types[i]
            ws = model.gemm_workspace(P, H, H, dev, "produce")
            f_map = lambda: proj.apply(i, b, x, ssq, workspace=ws)                         # noqa: E731
            f_fill = lambda: model.fill(i, x, pos, caches, ssq=ssq, cs=cs)                 # noqa: E731
            for name, f in (("map", f_map), (kind, f_fill)):
                f() if timer is None else timer.run(name, f)
        return caches

    cache = model.new_cache()

    def reset():                                  # no rows; the attention layers keep their K / V buffers
        for i in w["layers"]:
            c = cache[i]
            cache[i] = dict(kbuf=c["kbuf"], vbuf=c["vbuf"], n=0) if "kbuf" in c else {}

    fill_late(model, w["h_split"], arm, cache=cache)
    torch.cuda.synchronize()
    rep_ms = []
    for _ in range(reps):
        reset()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        fill_late(model, w["h_split"], arm, cache=cache)
        e1.record()
        e1.synchronize()
        rep_ms.append(e0.elapsed_time(e1))
    el = statistics.median(rep_ms) / 1e3
    del cache
    t = KernelTimer()
    step(t)
    # one GDN layer's two kernels apart
    g = next(i for i in w["layers"] if model.layer_types[i] == "gdn")
    wg = model.W[g]
    proj.apply(g, b, x, ssq)
    pre = ops.norm_linear(x, ssq, model.eps, wg["w_in"])
    st = torch.zeros(nv, dk, dv, dtype=torch.float32, device=dev)
    for _ in range(reps):
        t.run("norm_linear", lambda: ops.norm_linear(x, ssq, model.eps, wg["w_in"], pre))
        st.zero_()
        t.run("gdn_fill", lambda: ops.gdn_fill(pre, nk, nv, dk, dv, wg["conv"], None, wg["a_log"], wg["dt_bias"], st))
    torch.cuda.synchronize()
    n_gdn = sum(model.layer_types[i] == "gdn" for i in w["layers"])
    n_attn = len(w["layers"]) - n_gdn
    f_gdn = 2 * H * (C + 2 * nv) + 2 * H * H + 2 * 4 * C + 6 * nv * dk * dv
    f_attn = 2 * H * H + 2 * H * 2 * model.n_kv * model.head_dim
    counted = P * (n_gdn * f_gdn + n_attn * f_attn)
    nl_flop = 2 * P * H * wg["w_in"].shape[0]
    return {"workload": f"qwen3.5-shaped hybrid fill: hidden {H}, late layers {split}..{cfg['num_hidden_layers'] - 1} "
                        f"({n_gdn} GDN + {n_attn} attention), {P} filled rows",
            "filled_tokens_per_s": round(P / el, 1), "ms_per_fill": round(el * 1e3, 3),
            "ms_per_fill_reps": [round(x, 3) for x in rep_ms], "timing": f"median of {reps} fills, HIP events",
            "counted_flop": counted, "counted_frac_bf16_peak": round(counted / el / PEAK_BF16, 4),
            "layer_mean_us": {k: round(t.mean_s(k) * 1e6, 1) for k in ("map", "gdn", "attn")},
            "gdn_kernels": {
                "rf_norm_linear": {"mean_us": round(t.mean_s("norm_linear") * 1e6, 1),
                                   "achieved_tflops": round(nl_flop / t.mean_s("norm_linear") / 1e12, 1),
                                   "flop_per_launch": nl_flop},
                "rf_gdn_fill": {"mean_us": round(t.mean_s("gdn_fill") * 1e6, 1),
                                "counted_flop_per_launch": P * (2 * 4 * C + 6 * nv * dk * dv)}}}


def hybrid_finish_bench(dev, reps=5, split=24, n_rows=32768, tail=4096):
    """The hybrid's whole late stack as finish() runs it, without the logits: the fill of layers 24..47
    (P = 28672 rows), then the 4096-row exact tail through every late layer -- GDN layers continue the
    filled conv and recurrent states (in-projection, rf_gdn_forward with outputs, gated norm, out_proj,
    MLP), attention layers attend over all 32768 keys with the output gate (head_dim 256). The fill and the
    tail are each the median of `reps` runs after one warm-up run; every run's tail is reported."""
    from rfill import ops, synth
    from rfill.kva import Arm, Projector, fill_late
    from rfill.model import FillModel
    cfg = synth.QWEN35_HYBRID
    w = synth.hybrid_fill(cfg, split, n_rows, tail, device=dev, full=True)
    model = FillModel(cfg, w["tensors"], dev, layers=w["layers"])
    arm = Arm("ridgefill", split=split, tail=tail, fill="proj", projector=Projector(split, w["maps"], w["biases"]))
    h = w["h_split"]
    P = w["P"]
    pos = torch.arange(P, n_rows, device=dev)
    cs = model.rope_table(pos)

    def run():
        cache = model.new_cache()
        for i in w["layers"]:
            if model.layer_types[i] == "attn":
                model.reserve(cache[i], n_rows, model.n_kv, model.head_dim, dev)
        t0 = time.perf_counter()
        fill_late(model, h, arm, cache=cache)
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        x, ssq = h[P:], ops.row_ssq(h[P:])
        for i in w["layers"]:
            x, ssq = model.layer(i, x, pos, cache, ssq=ssq, cs=cs)
        torch.cuda.synchronize()
        return t1 - t0, time.perf_counter() - t1

    run()
    runs = [run() for _ in range(reps)]
    tf = statistics.median(r[0] for r in runs)
    tt = statistics.median(r[1] for r in runs)
    return {"workload": f"qwen3.5-shaped hybrid late stack: fill of layers {split}..{cfg['num_hidden_layers'] - 1} "
                        f"({P} rows) + {tail}-row exact tail through every late layer (MLP 6144)",
            "prompt_tokens_per_s": round(n_rows / (tf + tt), 1), "ms_fill": round(tf * 1e3, 2),
            "ms_tail": round(tt * 1e3, 2), "ms_tail_reps": [round(r[1] * 1e3, 2) for r in runs],
            "timing": f"median of {reps} runs, host clock with a device synchronisation at each end"}


def sweep_bench(dev, reps=2, split=18, tail=4096, frac=0.01, lengths=(16384, 32768, 65536, 122880)):
    """The Qwen3-8B-shaped fill (hidden 4096, 32 / 8 heads, q_norm / k_norm, RoPE theta 1e6, layers 18..35,
    maps I + 0.02 N(0, 1/H)) over the prompt-length sweep 16K / 32K / 64K / 120K rows with a 4096-row exact
    tail, P = N - 4096 filled rows, with 1 % of them exact (round(0.01 P) seeded positions) run as finish()
    runs them -- every late layer's cache filled with the rows' inputs scattered in, each exact row through
    the layer (query projection, attention over the filled keys, o_proj, SwiGLU MLP) -- and the same fill
    without exact rows. One model for every length; the split-layer rows are the first N of one draw."""
    from rfill import synth
    from rfill.kva import Arm, Projector, fill_late
    from rfill.model import FillModel
    cfg = synth.QWEN3_8B
    n_max = max(lengths)
    w = synth.dense_fill(cfg, split, n_max, tail, device=dev, full=True)
    model = FillModel(cfg, w["tensors"], dev, layers=w["layers"])
    del w["tensors"]
    arm = Arm("ridgefill", split=split, tail=tail, fill="proj", projector=Projector(split, w["maps"], w["biases"]))
    L = len(w["layers"])
    out = {"workload": f"qwen3-8b-shaped fill: layers {split}..{cfg['num_hidden_layers'] - 1} ({L} late layers), "
                       f"exact tail {tail}, 1% of the filled rows exact", "lengths": {}}
    for n in lengths:
        P = n - tail
        rows = torch.randperm(P, generator=torch.Generator().manual_seed(13))[:int(round(frac * P))].sort().values
        h = w["h_split"][:n]
        res = {}
        for name, exact in (("plain", None), ("exact", rows.to(dev))):
            fill_late(model, h, arm, exact_rows=exact)          # warm-up (the caching allocator keeps the buffers)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(reps):
                fill_late(model, h, arm, exact_rows=exact)      # a new cache per fill, as finish() starts one
            torch.cuda.synchronize()
            res[name] = (time.perf_counter() - t0) / reps
        flop = 2.0 * P * L * (4096 * 4096 + 4096 * 2 * 8 * 128)
        out["lengths"][n] = {"filled_rows": P, "exact_rows": len(rows),
                             "filled_tokens_per_s": round(P / res["exact"], 1), "ms_per_fill": round(res["exact"] * 1e3, 2),
                             "ms_per_fill_without_exact_rows": round(res["plain"] * 1e3, 2),
                             "filled_tokens_per_s_without_exact_rows": round(P / res["plain"], 1),
                             "fill_mfma_frac_without_exact_rows": round(flop / res["plain"] / PEAK_BF16, 4),
                             "exact_rows_ms": round((res["exact"] - res["plain"]) * 1e3, 2)}
        log(f"sweep N={n}: {out['lengths'][n]}")
        torch.cuda.empty_cache()
    return out


def finish_bench(dev, reps=3, keep=TAIL):
    """The whole late stack of one ridgefill arm at the Llama-3.1-8B shape, as finish() runs it: the
    16-layer fill of P = 28672 rows, then the 4096-row exact tail through every late layer (K / V appended,
    causal attention over all 32768 keys, o_proj, SwiGLU MLP 14336) and the logits of its last `keep`
    rows (vocab 128256). Reported: prompt tokens/s through the late layers (N / time), the fill, tail and
    logits times apart, and the tail's counted work (its GEMMs 2 T (q + kv + o + 3 MLP) per layer and the
    attention's 4 d flop per (query head, visible key))."""
    from rfill import synth
    from rfill.kva import Arm, Projector, fill_late, finish
    from rfill.model import FillModel
    cfg = synth.LLAMA_8B
    w = synth.dense_fill(cfg, SPLIT, N_ROWS, TAIL, device=dev, full=True, head=True)
    model = FillModel(cfg, w["tensors"], dev, layers=w["layers"])
    arm = Arm("ridgefill", split=SPLIT, tail=TAIL, fill="proj", projector=Projector(SPLIT, w["maps"], w["biases"]))
    del w["tensors"]
    h = w["h_split"]
    ids = torch.zeros(N_ROWS, dtype=torch.long)
    finish(model, ids, h, None, arm, keep)
    torch.cuda.synchronize()
    times = {"finish": 0.0, "fill": 0.0, "logits": 0.0}
    for _ in range(reps):
        t0 = time.perf_counter()
        finish(model, ids, h, None, arm, keep)
        torch.cuda.synchronize()
        times["finish"] += (time.perf_counter() - t0) / reps
        t0 = time.perf_counter()
        cache = model.new_cache()
        for i in w["layers"]:
            model.reserve(cache[i], N_ROWS, model.n_kv, model.head_dim, dev)
        fill_late(model, h, arm, cache=cache)
        torch.cuda.synchronize()
        times["fill"] += (time.perf_counter() - t0) / reps
        t0 = time.perf_counter()
        model.logits(h[N_ROWS - keep:])
        torch.cuda.synchronize()
        times["logits"] += (time.perf_counter() - t0) / reps
    H, L, T, P = cfg["hidden_size"], len(w["layers"]), TAIL, w["P"]
    hq, hkv, d, inter = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["intermediate_size"]
    tail_gemm = 2 * T * H * (hq * d + 2 * hkv * d + hq * d + 3 * inter) * L
    keys = sum(P + j + 1 for j in range(T))
    tail_attn = 4 * d * hq * keys * L
    t_tail = times["finish"] - times["fill"] - times["logits"]
    return {"workload": f"llama-3.1-8b-shaped 32K finish(): fill of layers {SPLIT}..{cfg['num_hidden_layers'] - 1} "
                        f"({P} rows) + {T}-row exact tail through every late layer + logits of {keep} rows",
            "prompt_tokens_per_s": round(N_ROWS / times["finish"], 1), "ms_finish": round(times["finish"] * 1e3, 2),
            "ms_fill": round(times["fill"] * 1e3, 2), "ms_tail": round(t_tail * 1e3, 2),
            "ms_logits": round(times["logits"] * 1e3, 2),
            "tail_counted_flop": tail_gemm + tail_attn, "tail_attention_flop": tail_attn,
            "tail_tflops": round((tail_gemm + tail_attn) / t_tail / 1e12, 1)}


def traffic_from_profiles(kernel):
    """HBM bytes per launch from the committed rocprofv3 --pmc summary (FETCH_SIZE + WRITE_SIZE scaled
    by a copy kernel of known size), or None if it has not been measured."""
    f = ROOT / "profiles" / "traffic.json"
    if not f.exists():
        return None
    try:
        return json.loads(f.read_text()).get(kernel, {}).get("traffic_bytes")
    except (ValueError, OSError):
        return None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-extras", action="store_true", help="skip ceilings and the standalone KV-write leg")
    ap.add_argument("--no-fit", action="store_true", help="skip the closed-form fit leg")
    ap.add_argument("--no-hybrid", action="store_true", help="skip the Gated-DeltaNet hybrid fill leg")
    ap.add_argument("--no-exact", action="store_true", help="skip the Qwen3-8B prompt-length sweep with exact rows")
    ap.add_argument("--no-finish", action="store_true", help="skip the whole-finish() leg (fill + exact tail)")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build measures one GPU only (one MI355X per box); --gpus must be 1", file=sys.stderr)
        sys.exit(2)
    dev = torch.device("cuda")
    torch.cuda.set_device(0)
    cfg, w, model, arm = build_workload(dev)
    P = w["P"]
    H = cfg["hidden_size"]
    b = w["h_split"][:P]
    pos = torch.arange(P, device=dev)
    cs = model.rope_table(pos)
    from rfill.kva import ATTN_GROUP
    xbuf = [torch.empty(P, H, dtype=torch.bfloat16, device=dev) for _ in range(ATTN_GROUP)]
    sbuf = [torch.empty(P, H // 256, dtype=torch.float32, device=dev) for _ in range(ATTN_GROUP)]
    caches = model.new_cache()
    for i in w["layers"]:
        caches[i] = dict(kbuf=torch.empty(model.n_kv, P + 64, model.head_dim, dtype=torch.bfloat16, device=dev),
                         vbuf=torch.empty(model.n_kv, P + 64, model.head_dim, dtype=torch.bfloat16, device=dev), n=0)
    log(f"warmup {args.warmup} steps")
    for _ in range(args.warmup):
        fill_step(model, arm, b, pos, cs, xbuf, sbuf, caches)
    torch.cuda.synchronize()
    log(f"timing {args.steps} steps")
    timer = KernelTimer()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        fill_step(model, arm, b, pos, cs, xbuf, sbuf, caches, timer)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    L = len(w["layers"])
    # one launch covers ATTN_GROUP layers (L is a multiple of it here)
    map_s, kv_s = timer.mean_s("rf_map_apply_batch"), timer.mean_s("rf_norm_kv_write_batch")
    map_flop = 2 * P * H * H * ATTN_GROUP
    kv_flop = 2 * P * H * 2 * model.n_kv * model.head_dim * ATTN_GROUP
    step_flop = L * (map_flop + kv_flop) // ATTN_GROUP
    ms_step = elapsed / args.steps * 1e3
    out = {
        "metric": METRIC, "value": round(P * args.steps / elapsed, 1), "unit": "filled tokens/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms_step, 3), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "llama-3.1-8b-shaped 32K fill: 16 late layers (split 16), 28672 filled rows, tail 4096",
                   "hidden": H, "kv_heads": model.n_kv, "head_dim": model.head_dim, "late_layers": L,
                   "seq_len": N_ROWS, "filled_rows": P, "parallelism": "none (1 GPU)"},
        "roofline": {"kernel": "rf_map_apply_batch", "bound": "mfma",
                     "achieved": round(map_flop / map_s / 1e12, 1), "peak": PEAK_BF16 / 1e12, "unit": "TFLOP/s",
                     "frac": round(map_flop / map_s / PEAK_BF16, 4),
                     "traffic": traffic_from_profiles("rf_map_apply_batch"), "flop_per_launch": map_flop,
                     "layers_per_launch": ATTN_GROUP, "mean_us": round(map_s * 1e6, 1),
                     "mean_us_per_layer": round(map_s * 1e6 / ATTN_GROUP, 1)},
        "fill_mfma_frac": round(step_flop / (elapsed / args.steps) / PEAK_BF16, 4),
        "kernels": {"rf_norm_kv_write_batch": {"bound": "mfma", "mean_us": round(kv_s * 1e6, 1),
                                               "mean_us_per_layer": round(kv_s * 1e6 / ATTN_GROUP, 1),
                                               "layers_per_launch": ATTN_GROUP,
                                               "achieved_tflops": round(kv_flop / kv_s / 1e12, 1),
                                               "frac": round(kv_flop / kv_s / PEAK_BF16, 4),
                                               "flop_per_launch": kv_flop,
                                               "traffic": traffic_from_profiles("rf_norm_kv_write_batch")}},
    }
    if not args.no_extras:
        log("standalone RoPE + KV write and library ceilings")
        out["kernels"]["rf_rope_kv_write"] = kv_write_bench(model, dev, P, SPLIT)
        out["kernels"]["rf_dequant_i8_rows"] = dequant_bench(dev)
        out["kernels"]["rf_window_mass"] = window_mass_bench(dev)
        out["kernels"]["rf_dequant_gguf_rows"] = gguf_bench(dev)
        out["ceilings"] = c = ceilings(dev, P, H)
        rf = out["roofline"]
        rf["measured_ceilings_tflops"] = {"mfma_power": c["mfma_power_ceiling_tflops"],
                                          "hipblaslt_same_shape": c["hipblaslt_gemm_tflops"]}
        rf["frac_of_mfma_power_ceiling"] = round(rf["achieved"] / c["mfma_power_ceiling_tflops"], 4)
        rf["frac_of_hipblaslt"] = round(rf["achieved"] / c["hipblaslt_gemm_tflops"], 4)
    del caches, xbuf, sbuf
    torch.cuda.empty_cache()
    if not args.no_finish:
        log("finish(): fill + exact tail + logits")
        out["finish"] = finish_bench(dev)
        torch.cuda.empty_cache()
    if not args.no_exact:
        log("Qwen3-8B prompt-length sweep with 1% exact rows")
        out["qwen3_sweep"] = sweep_bench(dev)
        torch.cuda.empty_cache()
    if not args.no_hybrid:
        log("Gated-DeltaNet hybrid fill leg")
        out["hybrid"] = hybrid_bench(dev)
        torch.cuda.empty_cache()
        log("Gated-DeltaNet hybrid fill + exact tail")
        out["hybrid_finish"] = hybrid_finish_bench(dev)
        torch.cuda.empty_cache()
    if not args.no_fit:
        log("closed-form fit leg")
        out["fit"] = f = fit_bench(dev)
        if "ceilings" in out:                     # the Gram against the power-limited MFMA rate of this run
            f["gram_frac_of_mfma_power_ceiling"] = round(f["gram_tflops"] / out["ceilings"]["mfma_power_ceiling_tflops"], 4)
        torch.cuda.empty_cache()
        log("capture and lambda-selection leg")
        out["capture"] = capture_bench(dev)
        torch.cuda.empty_cache()
    if not args.no_cpu:
        log("CPU baseline (oracle fill on the host cores)")
        out["cpu_baseline"] = cpu_baseline(cfg, w, SPLIT)
        if not args.no_exact:
            log("CPU baseline of the Qwen3-8B 32K fill with 1% exact rows (one layer)")
            out["cpu_exact_rows_baseline"] = cpu_exact_rows_baseline()
        if not args.no_hybrid:
            log("CPU baseline of the hybrid fill (one 8192-row segment per layer kind)")
            out["cpu_hybrid_baseline"] = cpu_hybrid_baseline()
        if not args.no_fit:
            log("CPU baseline of the fit (bounded sample)")
            out["cpu_fit_baseline"] = cpu_fit_baseline()
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
