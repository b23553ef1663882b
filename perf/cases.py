"""The workloads that this framework's speed is judged on: a late layer's work in each of its forms, one whole
finish(), the exact-row selector and the two halves of the closed-form fit, at the shapes of rfill.synth's
configurations and of the small test model, over prompts from a few hundred rows to 32K.

A case names a kind (one of KINDS) and its sizes. prepare() builds the model, caches and inputs that a program
holds when it makes the call; run() is the call; exact() is the same computation in float64 by plain torch.
Prompt lengths, tails and exact-row counts are mostly odd: real prompts are not multiples of a tile.
"""
import math
import sys
from pathlib import Path

import torch

_ROOT = Path(__file__).resolve().parent.parent
if str(_ROOT / "ridgefill-data_amd") not in sys.path:
    sys.path.insert(0, str(_ROOT / "ridgefill-data_amd"))

DEV = "cuda"
SPLIT = 4                       # late layers begin here in the models below (only the late ones are built)
# the small test model: 3 late layers of 8, whole finish() in a few dozen short launches
SMALL = dict(model_type="llama", num_hidden_layers=8, hidden_size=256, intermediate_size=688, num_attention_heads=4,
             num_key_value_heads=2, head_dim=64, vocab_size=1024, rms_norm_eps=1e-5, rope_theta=1e4)
SMALL_SPLIT = 5
WINDOW = 64                     # the selector's window rows


def _arch(name):
    from rfill import synth
    return {"llama_8b": synth.LLAMA_8B, "qwen3_8b": synth.QWEN3_8B, "hybrid": synth.QWEN35_HYBRID, "small": SMALL}[name]


# ------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # The smallest whole call: finish() of a short prompt through the small model (fill of three late
        # layers, exact tail, logits). Its time is launches and host work.
        dict(name="finish_small", kind="finish_small", prompt=2048, tail=256),
        # An ordinary prompt's late-layer fill, four k_normed layers (one group of fill_late).
        dict(name="fill_dense_7k", kind="fill_dense", arch="qwen3_8b", layers=4, prompt=7181, tail=1021),
        # The longest prompt's fill at the 8B shape: 32K rows, a 4096-row exact tail, four layers of its sixteen.
        dict(name="fill_dense_32k", kind="fill_dense", arch="llama_8b", layers=4, prompt=32768, tail=4096),
        # The hybrid's fill: eight late layers (six Gated DeltaNet, two gated attention) of a 16K prompt.
        dict(name="fill_hybrid_16k", kind="fill_hybrid", layers=8, prompt=16411, tail=2048),
        # Exact rows: 1 % of a 12K prefix through one filled late layer.
        dict(name="rows_12k", kind="rows", arch="qwen3_8b", rows=119, prefix=11930),
        # A follow-up turn's few rows through one late layer over a short cache: weights and latency.
        dict(name="tail_short", kind="tail_attn", arch="llama_8b", rows=37, prefix=3001),
        # The exact tail of a 32K prompt through one late layer: 4096 queries over up to 32768 keys, and the MLP.
        dict(name="tail_long", kind="tail_attn", arch="llama_8b", rows=4096, prefix=28672),
        # The hybrid's gated attention layer (head_dim 256) over an ordinary tail.
        dict(name="tail_gated", kind="tail_attn", arch="hybrid", rows=1499, prefix=14003),
        # The hybrid's exact Gated DeltaNet layer over an ordinary tail, continuing the filled state.
        dict(name="tail_gdn", kind="tail_gdn", rows=1499),
        # Exact-row selection: the window's attention mass at two lower layers of a 32K prompt.
        dict(name="window_mass", kind="window_mass", layers=2, prompt=32768),
        # The fit's sums over three calibration documents: X^T X and four X^T Y, and the finished state.
        dict(name="fit_sums", kind="fit_sums", dim=4096, targets=4, docs="9001,7003,8190"),
        # The fit's solve: four targets for three ridge strengths.
        dict(name="fit_solve", kind="fit_solve", dim=4096, targets=4, lams="1e-4,1e-3,1e-2"),
    ]


KINDS = ("finish_small", "fill_dense", "fill_hybrid", "rows", "tail_attn", "tail_gdn", "window_mass", "fit_sums",
         "fit_solve")


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    if kind == "finish_small":
        prompt = _log_int(rng, 384, 2048)
        return dict(kind=kind, prompt=prompt, tail=_log_int(rng, 16, min(256, prompt // 2)))
    if kind == "fill_dense":
        prompt = _log_int(rng, 512, 32768)
        return dict(kind=kind, arch=rng.choice(("llama_8b", "qwen3_8b")), layers=rng.randint(1, 4), prompt=prompt,
                    tail=_log_int(rng, 64, min(4096, prompt // 2)))
    if kind == "fill_hybrid":
        prompt = _log_int(rng, 512, 16384)
        return dict(kind=kind, layers=rng.choice((4, 8)), prompt=prompt, tail=_log_int(rng, 64, min(4096, prompt // 2)))
    if kind == "rows":
        prefix = _log_int(rng, 2048, 28672)
        return dict(kind=kind, arch=rng.choice(("llama_8b", "qwen3_8b")), rows=_log_int(rng, 16, prefix // 20),
                    prefix=prefix)
    if kind == "tail_attn":
        return dict(kind=kind, arch=rng.choice(("llama_8b", "qwen3_8b", "hybrid")), rows=_log_int(rng, 16, 4096),
                    prefix=_log_int(rng, 512, 28672))
    if kind == "tail_gdn":
        return dict(kind=kind, rows=_log_int(rng, 16, 4096))
    if kind == "window_mass":
        return dict(kind=kind, layers=rng.choice((1, 2)), prompt=_log_int(rng, 512, 32768))
    if kind == "fit_sums":
        docs = [_log_int(rng, 300, 8500) for _ in range(rng.randint(1, 3))]
        return dict(kind=kind, dim=rng.choice((2048, 4096)), targets=rng.randint(1, 4),
                    docs=",".join(str(n) for n in docs))
    dim = rng.choice((1024, 2048, 2560, 4096))
    lams = (("1e-2",), ("1e-4", "1e-3", "1e-2"), ("1e-4", "3e-4", "1e-3", "3e-3", "0.01", "0.03", "0.1", "0.3", "1.0"))
    return dict(kind=kind, dim=dim, targets=rng.randint(1, 4),
                lams=",".join(lams[rng.randint(0, 1 if dim > 2560 else 2)]))


# ----------------------------------------------------------------------------------------- weights and inputs

class _Draws:
    """Seeded draws on the GPU, each from a generator of its own."""

    def __init__(self, seed):
        self.seed, self.k = seed, 0

    def gen(self):
        self.k += 1
        return torch.Generator(device=DEV).manual_seed((self.seed * 1000003 + self.k) & 0x7FFFFFFF)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.gen(), device=DEV) * std + mean

    def bf(self, *shape, std=1.0, mean=0.0):
        return self.normal(*shape, std=std, mean=mean).to(torch.bfloat16)

    def rand(self, *shape):
        return torch.rand(*shape, generator=self.gen(), device=DEV)


def _hidden(dr, n, h):
    """Split-layer rows: N(0, 1) x a log-normal(0, 0.5) channel gain, four outlier channels x 20."""
    gain = torch.exp(dr.normal(h, std=0.5))
    gain[torch.randperm(h, generator=dr.gen(), device=DEV)[:4]] *= 20.0
    return (dr.normal(n, h) * gain).to(torch.bfloat16)


def _layer(dr, cfg, i, full):
    """Checkpoint-named weights of layer i: matrices N(0, 0.02), norm gains 1 + N(0, 0.05) (zero-centred
    N(0, 0.05) for the hybrid); a GDN layer's conv U(-0.5, 0.5), A_log = log U(0, 16), dt_bias 1."""
    h, zc = cfg["hidden_size"], cfg["model_type"].startswith("qwen3_5")
    gain = lambda *s: dr.bf(*s, std=0.05, mean=0.0 if zc else 1.0)                      # noqa: E731
    mat = lambda *s: dr.bf(*s, std=0.02)                                                # noqa: E731
    p = f"model.layers.{i}."
    t = {p + "input_layernorm.weight": gain(h)}
    if zc and cfg["layer_types"][i] == "linear_attention":
        nk, nv = cfg["linear_num_key_heads"], cfg["linear_num_value_heads"]
        dk, dv = cfg["linear_key_head_dim"], cfg["linear_value_head_dim"]
        c, a = 2 * nk * dk + nv * dv, p + "linear_attn."
        t[a + "in_proj_qkv.weight"], t[a + "in_proj_b.weight"], t[a + "in_proj_a.weight"] = mat(c, h), mat(nv, h), mat(nv, h)
        t[a + "conv1d.weight"] = (dr.rand(c, 1, 4) - 0.5).to(torch.bfloat16)
        t[a + "A_log"] = torch.log(16 * dr.rand(nv).clamp_min(1e-6))
        t[a + "dt_bias"] = torch.ones(nv, device=DEV)
        if full:
            t[a + "in_proj_z.weight"] = mat(nv * dv, h)
            t[a + "norm.weight"] = dr.bf(dv, std=0.05, mean=1.0)
            t[a + "out_proj.weight"] = mat(h, nv * dv)
    else:
        hq, hkv, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        a = p + "self_attn."
        t[a + "k_proj.weight"], t[a + "v_proj.weight"] = mat(hkv * d, h), mat(hkv * d, h)
        if cfg["model_type"] != "llama":
            t[a + "k_norm.weight"] = gain(d)
        if full:
            t[a + "q_proj.weight"], t[a + "o_proj.weight"] = mat((2 if zc else 1) * hq * d, h), mat(h, hq * d)
            if cfg["model_type"] != "llama":
                t[a + "q_norm.weight"] = gain(d)
    if full:
        inter = cfg["intermediate_size"]
        t[p + "post_attention_layernorm.weight"] = gain(h)
        t[p + "mlp.gate_proj.weight"], t[p + "mlp.up_proj.weight"] = mat(inter, h), mat(inter, h)
        t[p + "mlp.down_proj.weight"] = mat(h, inter)
    return t


def _maps(dr, h, layers):
    """Ridge maps I + 0.02 N(0, 1/h) with biases N(0, 1e-3)."""
    W = {i: (torch.eye(h, device=DEV) + dr.normal(h, h, std=0.02 / h ** 0.5)).to(torch.bfloat16) for i in layers}
    return W, {i: dr.bf(h, std=1e-3) for i in layers}


def _cfg(case):
    """(config, late layers of the case) -- only the layers that the case runs exist."""
    kind = case["kind"]
    if kind == "finish_small":
        return SMALL, list(range(SMALL_SPLIT, SMALL["num_hidden_layers"]))
    arch = "hybrid" if kind in ("fill_hybrid", "tail_gdn") else case.get("arch", "llama_8b")
    cfg = dict(_arch(arch))
    if kind in ("fill_dense", "fill_hybrid"):
        cfg["num_hidden_layers"] = SPLIT + case["layers"]
        if "layer_types" in cfg:
            cfg["layer_types"] = cfg["layer_types"][:SPLIT + case["layers"]]
        return cfg, list(range(SPLIT, SPLIT + case["layers"]))
    if kind == "window_mass":
        return cfg, [3, 7][:case["layers"]]
    # one layer: the hybrid's attention layers are every fourth
    return cfg, [7 if arch == "hybrid" and kind == "tail_attn" else 4]


def _inputs(case, seed):
    """Everything drawn for a case, shared by prepare() and exact()."""
    dr, kind = _Draws(seed), case["kind"]
    if kind in ("fit_sums", "fit_solve"):
        return _fit_inputs(case, dr)
    cfg, layers = _cfg(case)
    h = cfg["hidden_size"]
    x = dict(cfg=cfg, layers=layers, tensors={})
    for i in layers:
        x["tensors"].update(_layer(dr, cfg, i, full=not kind.startswith("fill")))
    if kind in ("finish_small", "fill_dense", "fill_hybrid"):
        x["maps"], x["biases"] = _maps(dr, h, layers)
        x["h"] = _hidden(dr, case["prompt"], h)
        if kind == "finish_small":
            x["tensors"]["model.norm.weight"] = dr.bf(h, std=0.05, mean=1.0)
            x["tensors"]["lm_head.weight"] = dr.bf(cfg["vocab_size"], h, std=0.02)
        return x
    if kind == "tail_gdn":
        nk, nv = cfg["linear_num_key_heads"], cfg["linear_num_value_heads"]
        dk, dv = cfg["linear_key_head_dim"], cfg["linear_value_head_dim"]
        x["h"] = _hidden(dr, case["rows"], h)
        x["conv"] = dr.bf(3, 2 * nk * dk + nv * dv, std=0.02 * h ** 0.5)
        x["rec"] = dr.normal(nv, dk, dv, std=0.1)
        return x
    hkv, d = cfg["num_key_value_heads"], cfg["head_dim"]
    # the cached keys and values a filled layer holds: unit rows after k_norm, else the projections' spread
    kstd = 1.0 if cfg["model_type"] != "llama" else 0.02 * h ** 0.5
    if kind == "window_mass":
        x["win"] = {i: _hidden(dr, WINDOW, h) for i in layers}
        x["k"] = {i: dr.bf(hkv, case["prompt"], d, std=kstd) for i in layers}
        return x
    x["h"] = _hidden(dr, case["rows"], h)
    x["k"] = dr.bf(hkv, case["prefix"], d, std=kstd)
    x["v"] = dr.bf(hkv, case["prefix"], d, std=0.02 * h ** 0.5)
    if kind == "rows":
        x["rows"] = torch.randperm(case["prefix"], generator=dr.gen(), device=DEV)[:case["rows"]].sort().values
    return x


def _fit_inputs(case, dr):
    """Rows of Student-t(5) spread with four outlier channels x 20 and four channels whose mean exceeds their
    spread, and targets Y = X (I + 0.05 N(0, 1/d)) + 0.1 N(0, 1)."""
    d, L = case["dim"], list(range(case["targets"]))
    docs = [int(n) for n in case["docs"].split(",")] if case["kind"] == "fit_sums" else [2 * d]
    pick = torch.randperm(d, generator=dr.gen(), device=DEV)
    T = [torch.eye(d, device=DEV) + dr.normal(d, d, std=0.05 / d ** 0.5) for _ in L]
    out = []
    for n in docs:
        chi2 = sum(dr.normal(n, d) ** 2 for _ in range(5)) / 5
        x = dr.normal(n, d) * torch.rsqrt(chi2)
        x[:, pick[:4]] *= 20.0
        x[:, pick[4:8]] += 6.0
        x = x.to(torch.bfloat16)
        out.append((x, {i: (x.float() @ T[i] + dr.normal(n, d, std=0.1)).to(torch.bfloat16) for i in L}))
    return dict(dim=d, layers=L, docs=out)


def _sums(x, docs, block=8192):
    """The fit's sums in float64 about the first block's means (rounded to float32, as they are kept)."""
    L = x["layers"]
    cx = docs[0][0][:block].double().mean(0).float().double()
    cy = {i: docs[0][1][i][:block].double().mean(0).float().double() for i in L}
    z = dict(split=0, layers=L, dim=x["dim"], n=sum(a.shape[0] for a, _ in docs), cx=cx, cy=cy, sx=0.0, sxx=0.0,
             sy={i: 0.0 for i in L}, sxy={i: 0.0 for i in L})
    for a, ys in docs:
        a = a.double() - cx
        z["sx"], z["sxx"] = z["sx"] + a.sum(0), z["sxx"] + a.T @ a
        for i in L:
            y = ys[i].double() - cy[i]
            z["sy"][i], z["sxy"][i] = z["sy"][i] + y.sum(0), z["sxy"][i] + a.T @ y
    return z


# ------------------------------------------------------------------------------------------- prepare and run

def prepare(case, seed):
    x, kind = _inputs(case, seed), case["kind"]
    if kind == "fit_sums":
        return dict(kind=kind, x=x)
    if kind == "fit_solve":
        return dict(kind=kind, x=x, state=_sums(x, x["docs"]), lams=[float(v) for v in case["lams"].split(",")])
    from rfill import ops
    from rfill.kva import Arm, Projector
    from rfill.model import KV_RESERVE, FillModel
    cfg, layers = x["cfg"], x["layers"]
    model = FillModel(cfg, x["tensors"], DEV, layers=layers)
    s = dict(kind=kind, model=model, layers=layers)
    if "maps" in x:
        split = layers[0]
        s["arm"] = Arm("ridgefill", split=split, tail=case["tail"], fill="proj",
                       projector=Projector(split, x["maps"], x["biases"]))
        s["h"] = x["h"]
        if kind == "finish_small":
            s["ids"] = torch.zeros(case["prompt"], dtype=torch.int64)
        return s
    if kind == "tail_gdn":
        return dict(s, h=x["h"], ssq=ops.row_ssq(x["h"]), pos=torch.arange(case["rows"], device=DEV),
                    cache=dict(conv=x["conv"], rec=x["rec"], len=8192))

    def filled(k, v, room):
        """A cache dict whose first rows are k / v, with room for the coming ones."""
        hkv, n, d = k.shape
        kb = torch.zeros(hkv, n + room + KV_RESERVE, d, dtype=torch.bfloat16, device=DEV)
        vb = torch.zeros_like(kb)
        kb[:, :n], vb[:, :n] = k, v
        return dict(kbuf=kb, vbuf=vb, n=n, k=kb[:, :n], v=vb[:, :n])

    if kind == "window_mass":
        return dict(s, win=x["win"], cache={i: filled(x["k"][i], x["k"][i], 0) for i in layers})
    rows, prefix = case["rows"], case["prefix"]
    s.update(h=x["h"], ssq=ops.row_ssq(x["h"]))
    if kind == "rows":
        pos = torch.arange(prefix, device=DEV)
        return dict(s, rows=x["rows"], pos=pos, cs=model.rope_table(pos), cache=filled(x["k"], x["v"], 0))
    pos = torch.arange(prefix, prefix + rows, device=DEV)
    return dict(s, pos=pos, cs=model.rope_table(pos), cache=filled(x["k"], x["v"], rows))


def run(s):
    kind = s["kind"]
    if kind == "fit_sums":
        from rfill.ridge import RidgeStats
        x = s["x"]
        st = RidgeStats(0, x["layers"], x["dim"], DEV)
        for a, ys in x["docs"]:
            st.add(a, ys)
        z = st.state(device=DEV)
        return {k: z[k] for k in ("n", "cx", "cy", "sx", "sxx", "sy", "sxy")}
    if kind == "fit_solve":
        from rfill.ridge import RidgeFit
        got = RidgeFit(s["state"], DEV).layers(s["state"]["layers"], s["lams"])
        return [[got[i][lam] for lam in s["lams"]] for i in s["state"]["layers"]]
    model, layers = s["model"], s["layers"]
    if kind == "finish_small":
        from rfill.kva import finish
        logits, cache, _ = finish(model, s["ids"], s["h"], None, s["arm"], s["arm"].tail)
        return logits, [(cache[i]["k"], cache[i]["v"]) for i in layers]
    if kind in ("fill_dense", "fill_hybrid"):
        from rfill.kva import fill_late
        cache, _ = fill_late(model, s["h"], s["arm"])
        return [(cache[i]["k"], cache[i]["v"]) if "k" in cache[i] else (cache[i]["rec"], cache[i]["conv"])
                for i in layers]
    if kind == "window_mass":
        from rfill.select import window_mass
        return window_mass(model, s["win"], s["cache"], layers)
    i = layers[0]
    cache = {i: dict(s["cache"])}           # the call moves on its own copy of the cache's counters, so that the
    if kind == "rows":                      # next pass starts from the same prefix
        out = model.rows_over_fill(i, s["h"], s["ssq"], s["pos"], s["rows"], cache, s["cs"], full=True,
                                   rows_max=s["pos"].shape[0] - 1, qpos=s["rows"])
        return out, cache[i]["k"], cache[i]["v"]
    if kind == "tail_attn":
        out = model.layer(i, s["h"], s["pos"], cache, ssq=s["ssq"], cs=s["cs"])
        return out, cache[i]["k"], cache[i]["v"]
    out = model.layer(i, s["h"], s["pos"], cache, ssq=s["ssq"])
    return out, cache[i]["rec"], cache[i]["conv"]


# ------------------------------------------------------------------------------- the same in float64, plain torch

class _Layer64:
    """One layer's weights in float64 and its parts."""

    def __init__(self, x, i):
        self.cfg, self.i = x["cfg"], i
        p = f"model.layers.{i}."
        self.w = {k[len(p):]: v.double() for k, v in x["tensors"].items() if k.startswith(p)}
        c = self.cfg
        self.zc = c["model_type"].startswith("qwen3_5")
        self.gdn = self.zc and c["layer_types"][i] == "linear_attention"
        self.hq, self.hkv, self.d = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        rp = c.get("rope_parameters") or {}
        theta = rp.get("rope_theta", c.get("rope_theta"))
        self.rot = int(self.d * rp.get("partial_rotary_factor", 1.0))
        self.inv = (1.0 / (theta ** (torch.arange(0, self.rot, 2, dtype=torch.float32) / self.rot))).double().to(DEV)

    def norm(self, x, g):
        y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + self.cfg["rms_norm_eps"])
        return y * ((1.0 + g) if self.zc else g)

    def rope(self, x, pos):
        a = pos.double()[:, None] * self.inv
        c, s = a.cos()[:, None], a.sin()[:, None]
        h = self.rot // 2
        lo, hi = x[..., :h], x[..., h:self.rot]
        return torch.cat((lo * c - hi * s, hi * c + lo * s, x[..., self.rot:]), -1)

    def kv(self, xn, pos):
        """K (normed, rotated) and V of normed rows, [hkv, n, d]."""
        n = xn.shape[0]
        k = (xn @ self.w["self_attn.k_proj.weight"].T).view(n, self.hkv, self.d)
        if "self_attn.k_norm.weight" in self.w:
            k = self.norm(k, self.w["self_attn.k_norm.weight"])
        v = (xn @ self.w["self_attn.v_proj.weight"].T).view(n, self.hkv, self.d)
        return self.rope(k, pos).transpose(0, 1), v.transpose(0, 1)

    def queries(self, xn, pos):
        """(queries [n, hq, d], the output gate [n, hq, d] or None)."""
        n = xn.shape[0]
        q, gate = xn @ self.w["self_attn.q_proj.weight"].T, None
        if self.zc:
            q, gate = q.view(n, self.hq, 2, self.d).unbind(2)
        q = q.reshape(n, self.hq, self.d)
        if "self_attn.q_norm.weight" in self.w:
            q = self.norm(q, self.w["self_attn.q_norm.weight"])
        return self.rope(q, pos), gate

    def attend(self, q, k, v, qpos):
        """Causal attention [n, hq, d] of queries at positions qpos, a head and a block of queries at a time."""
        out, n, keys = torch.empty_like(q), q.shape[0], torch.arange(k.shape[1], device=DEV)
        step = max(1, (1 << 27) // k.shape[1])
        for h in range(self.hq):
            kh, vh = k[h // (self.hq // self.hkv)], v[h // (self.hq // self.hkv)]
            for a in range(0, n, step):
                s = (q[a:a + step, h] @ kh.T) * self.d ** -0.5
                s.masked_fill_(keys[None] > qpos[a:a + step, None], float("-inf"))
                out[a:a + step, h] = torch.softmax(s, -1) @ vh
        return out

    def rest(self, h, o):
        """The layer's output from its inputs h and mixed rows o: o_proj, the residual, the MLP."""
        w = self.w
        h = h + o @ (w["linear_attn.out_proj.weight"] if self.gdn else w["self_attn.o_proj.weight"]).T
        y = self.norm(h, w["post_attention_layernorm.weight"])
        g = y @ w["mlp.gate_proj.weight"].T
        return h + ((g * torch.sigmoid(g)) * (y @ w["mlp.up_proj.weight"].T)) @ w["mlp.down_proj.weight"].T

    def attn_layer(self, h, qpos, k, v):
        """The full layer of rows h at positions qpos over keys k / v that hold them already."""
        xn = self.norm(h, self.w["input_layernorm.weight"])
        q, gate = self.queries(xn, qpos)
        o = self.attend(q, k, v, qpos)
        if gate is not None:
            o = o * torch.sigmoid(gate)
        return self.rest(h, o.reshape(h.shape[0], -1))

    def gdn_mix(self, xn, conv, rec, want):
        """(delta-rule outputs [n, nv, dv] or None, state, conv state) of normed rows, chunk by chunk."""
        c, w = self.cfg, self.w
        nk, nv = c["linear_num_key_heads"], c["linear_num_value_heads"]
        dk, dv = c["linear_key_head_dim"], c["linear_value_head_dim"]
        n, a = xn.shape[0], "linear_attn."
        pre = xn @ w[a + "in_proj_qkv.weight"].T
        seq = torch.cat((torch.zeros(3, pre.shape[1], dtype=torch.float64, device=DEV) if conv is None
                         else conv.double(), pre), 0)
        cw = w[a + "conv1d.weight"][:, 0]
        y = sum(seq[j:j + n] * cw[:, j] for j in range(4))
        y = y * torch.sigmoid(y)
        q, k, v = y[:, :nk * dk].view(n, nk, dk), y[:, nk * dk:2 * nk * dk].view(n, nk, dk), y[:, 2 * nk * dk:].view(n, nv, dv)
        unit = lambda t: t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6)       # noqa: E731
        rep = nv // nk
        q = (unit(q) * dk ** -0.5).repeat_interleave(rep, 1).transpose(0, 1)
        k, v = unit(k).repeat_interleave(rep, 1).transpose(0, 1), v.transpose(0, 1)
        beta = torch.sigmoid(xn @ w[a + "in_proj_b.weight"].T).T
        g = -(w[a + "A_log"].exp() * torch.nn.functional.softplus(xn @ w[a + "in_proj_a.weight"].T + w[a + "dt_bias"])).T
        S = torch.zeros(nv, dk, dv, dtype=torch.float64, device=DEV) if rec is None else rec.double()
        outs, eye = [], torch.eye(64, dtype=torch.float64, device=DEV)
        for r in range(0, n, 64):
            m = min(64, n - r)
            qc, kc, vc, bc = q[:, r:r + m], k[:, r:r + m], v[:, r:r + m], beta[:, r:r + m, None]
            gam = g[:, r:r + m].cumsum(-1)
            gap = torch.tril(gam[:, :, None] - gam[:, None, :])
            decay = torch.tril(gap.exp())
            kT = kc.transpose(1, 2).contiguous()
            A = torch.tril(bc * torch.matmul(kc.contiguous(), kT) * decay, -1) + eye[:m, :m]
            rhs = bc * (vc - gam.exp()[..., None] * torch.matmul(kc.contiguous(), S))
            vn = torch.linalg.solve_triangular(A, rhs, upper=False, unitriangular=True)
            if want:
                outs.append(torch.matmul(qc * gam.exp()[..., None], S)
                            + torch.matmul(torch.matmul(qc.contiguous(), kT) * decay, vn))
            end = (gam[:, -1:] - gam).exp()[:, None, :]
            S = S * gam[:, -1].exp()[:, None, None] + torch.matmul(kT * end, vn)
        return (torch.cat(outs, 1).transpose(0, 1) if want else None), S, seq[n:]


def _ssq(y):
    return y.view(y.shape[0], -1, 256).square().sum(-1)


def exact(case, seed):
    """run()'s outputs in float64."""
    x, kind = _inputs(case, seed), case["kind"]
    if kind == "fit_sums":
        z = _sums(x, x["docs"])
        return {k: z[k] for k in ("n", "cx", "cy", "sx", "sxx", "sy", "sxy")}
    if kind == "fit_solve":
        z, out, L = _sums(x, x["docs"]), [], x["layers"]
        n, sx = z["n"], z["sx"]
        C = z["sxx"] - torch.outer(sx, sx) / n
        B = torch.cat([z["sxy"][i] - torch.outer(sx, z["sy"][i]) / n for i in L], 1)
        mx = z["cx"] + sx / n
        per = []
        for lam in (float(v) for v in case["lams"].split(",")):
            A = C + lam * C.diagonal().mean() * torch.eye(x["dim"], dtype=torch.float64, device=DEV)
            per.append(torch.cholesky_solve(B, torch.linalg.cholesky(A)))
        for j, i in enumerate(L):
            cols = slice(j * x["dim"], (j + 1) * x["dim"])
            my = z["cy"][i] + z["sy"][i] / n
            out.append([(W[:, cols].T, my - mx @ W[:, cols]) for W in per])
        return out
    layers = x["layers"]
    parts = {i: _Layer64(x, i) for i in layers}
    if kind in ("finish_small", "fill_dense", "fill_hybrid"):
        h = x["h"].double()
        n, P = h.shape[0], h.shape[0] - case["tail"]
        pos, out = torch.arange(n, device=DEV), []
        for i in layers:
            lay = parts[i]
            xn = lay.norm(h[:P] @ x["maps"][i].double().T + x["biases"][i].double(), lay.w["input_layernorm.weight"])
            out.append(lay.gdn_mix(xn, None, None, False)[1:] if lay.gdn else lay.kv(xn, pos[:P]))
        if kind != "finish_small":
            return out
        t, kept = h[P:], []
        for i, (k, v) in zip(layers, out):
            lay = parts[i]
            kt, vt = lay.kv(lay.norm(t, lay.w["input_layernorm.weight"]), pos[P:])
            k, v = torch.cat((k, kt), 1), torch.cat((v, vt), 1)
            kept.append((k, v))
            t = lay.attn_layer(t, pos[P:], k, v)
        lay = parts[layers[0]]
        return lay.norm(t, x["tensors"]["model.norm.weight"].double()) @ x["tensors"]["lm_head.weight"].double().T, kept
    if kind == "window_mass":
        n = case["prompt"]
        mass, keys, qpos = torch.zeros(n, dtype=torch.float64, device=DEV), torch.arange(n, device=DEV), \
            torch.arange(n - WINDOW, n, device=DEV)
        for i in layers:
            lay = parts[i]
            q, _ = lay.queries(lay.norm(x["win"][i].double(), lay.w["input_layernorm.weight"]), qpos)
            for h in range(lay.hq):
                s = (q[:, h] @ x["k"][i][h // (lay.hq // lay.hkv)].double().T) * lay.d ** -0.5
                mass += torch.softmax(s.masked_fill(keys[None] > qpos[:, None], float("-inf")), -1).sum(0)
        return mass.cpu()
    lay, h = parts[layers[0]], x["h"].double()
    xn = lay.norm(h, lay.w["input_layernorm.weight"])
    if kind == "tail_gdn":
        o, S, conv = lay.gdn_mix(xn, x["conv"], x["rec"], True)
        o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + lay.cfg["rms_norm_eps"]) * lay.w["linear_attn.norm.weight"]
        z = (xn @ lay.w["linear_attn.in_proj_z.weight"].T).view(o.shape)
        y = lay.rest(h, (o * (z * torch.sigmoid(z))).reshape(h.shape[0], -1))
        return (y, _ssq(y)), S, conv
    k, v = x["k"].double(), x["v"].double()
    if kind == "rows":
        qpos = x["rows"]
        k[:, qpos], v[:, qpos] = lay.kv(xn, qpos)
    else:
        qpos = torch.arange(case["prefix"], case["prefix"] + case["rows"], device=DEV)
        kt, vt = lay.kv(xn, qpos)
        k, v = torch.cat((k, kt), 1), torch.cat((v, vt), 1)
    y = lay.attn_layer(h, qpos, k, v)
    return (y, _ssq(y)), k, v


# ------------------------------------------------------------------------------------------ work and tolerance

def _layer_work(cfg, i, n, full, keys=0, seen=0):
    """(bytes, flops) of layer i on n rows: the fill's part, or with full the whole layer, its queries seeing
    `seen` (query, key) pairs over `keys` cached rows."""
    h = cfg["hidden_size"]
    if "layer_types" in cfg and cfg["layer_types"][i] == "linear_attention":
        nk, nv = cfg["linear_num_key_heads"], cfg["linear_num_value_heads"]
        dk, dv = cfg["linear_key_head_dim"], cfg["linear_value_head_dim"]
        w = (nk * dk + nv * dv + 2 * nv) * h
        f = 2 * n * w + n * nv * (64 * (dk + dv) + 6 * dk * dv)         # projections; the chunked rule's products
        b = 2 * w + 2 * 4 * nv * dk * dv
        if full:
            w2 = nk * dk * h + 2 * nv * dv * h
            f += 2 * n * w2 + n * nv * (64 * (dk + dv) + 2 * dk * dv)
            b += 2 * w2
    else:
        hq, hkv, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        w = 2 * hkv * d * h
        f, b = 2 * n * w, 2 * w + 2 * 2 * n * hkv * d
        if full:
            w2 = (3 if cfg["model_type"].startswith("qwen3_5") else 2) * hq * d * h
            f += 2 * n * w2 + 4 * d * hq * seen
            b += 2 * w2 + 2 * 2 * keys * hkv * d
    if full:
        f += 2 * n * 3 * h * cfg["intermediate_size"]
        b += 2 * 3 * h * cfg["intermediate_size"] + 2 * 2 * n * h
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "fit_sums":
        n, d, t = sum(int(v) for v in case["docs"].split(",")), case["dim"], case["targets"]
        return {"bytes": 2 * n * d * (1 + t) + 8 * d * d * (1 + t), "flops": n * d * d + 2 * n * d * d * t}
    if kind == "fit_solve":
        d, t, m = case["dim"], case["targets"], len(case["lams"].split(","))
        # a Cholesky factor per strength and two triangular solves per column
        return {"bytes": 8 * d * d * (1 + t) + 4 * d * d * t * m, "flops": m * (d ** 3 / 3 + 2 * d * d * d * t)}
    cfg, layers = _cfg(case)
    h = cfg["hidden_size"]
    if kind == "window_mass":
        hq, hkv, d, n = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], case["prompt"]
        return {"bytes": len(layers) * 2 * (hq * d * h + hkv * n * d) + 8 * n,
                "flops": len(layers) * (2 * WINDOW * h * hq * d + 2 * WINDOW * hq * n * d)}
    if kind in ("fill_dense", "fill_hybrid", "finish_small"):
        P, T = case["prompt"] - case["tail"], case["tail"]
        b, f = 2 * P * h, 0
        for i in layers:
            lb, lf = _layer_work(cfg, i, P, False)
            b, f = b + lb + 2 * h * h, f + lf + 2 * P * h * h
            if kind == "finish_small":
                lb, lf = _layer_work(cfg, i, T, True, P, T * P + T * (T + 1) // 2)
                b, f = b + lb, f + lf
        if kind == "finish_small":
            b, f = b + 2 * cfg["vocab_size"] * h + 4 * T * cfg["vocab_size"], f + 2 * T * h * cfg["vocab_size"]
        return {"bytes": b, "flops": f}
    n, P = case["rows"], case.get("prefix", 0)
    # exact rows lie anywhere in the prefix: half of its keys on average
    seen = n * P // 2 if kind == "rows" else n * P + n * (n + 1) // 2
    b, f = _layer_work(cfg, layers[0], n, True, P, seen)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the distance from exact() that each kind shows over the declared ranges: bf16 results (a
    few rounded products each) 3e-3 to 5e-3, the window's mass 5e-4 (bf16 queries, float32 softmax), the sums
    5e-7 (float32 over runs of 8192 rows), the solve's float32 weights 3e-8."""
    kind = case["kind"]
    if kind == "fit_sums":
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "fit_solve":
        return {"rel": 1.2e-7, "max": 2.5e-7}
    if kind == "window_mass":
        return {"rel": 2e-3, "max": 2e-2}
    # single entries: 2e-2 to 4e-2 of the result's spread; of a Gated DeltaNet state (sums over the prompt) 0.14
    return {"rel": 2e-2, "max": 0.5 if kind in ("fill_hybrid", "tail_gdn") else 0.15}
