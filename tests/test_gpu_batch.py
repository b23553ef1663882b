"""GPU tests of the batched fill launches (rf_map_apply_batch, rf_norm_kv_write_batch: the maps and the
K / V fills of several late layers in one launch each, on persistent tiles) and of fill_late's grouped
schedule.

Bar: bitwise for launches without a workspace and for rows in whole rounds of tiles. Every layer's x, row
statistics and K / V cache equal the per-layer launches' without a split-K workspace (the same tiles, the same
MFMA order, the same epilogue arithmetic); cache slots outside the written rows keep their contents. Rows left
over by whole rounds, which a workspace lets run as products of few rows with K split, are held to the rounding of
one bf16 value. The per-layer launches themselves are pinned to the oracle in test_gpu_fill.py."""
import pytest
import torch

from fill_cases import CASES, attn_config, case, inputs, random_tensors, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from rfill import _lib
    _lib.load()
    return torch.device("cuda")


def _maps(H, layers, seed):
    g = torch.Generator().manual_seed(seed)
    W = [(torch.eye(H) + 0.05 * torch.randn(H, H, generator=g) / H ** 0.5).to(torch.bfloat16) for _ in layers]
    B = [(1e-2 * torch.randn(H, generator=g)).to(torch.bfloat16) for _ in layers]
    return W, B


# Width-1024 configurations take the persistent K / V kernel (the CASES widths 256 / 512 take the per-tile
# kernel): its d-128 K epilogue without and with k_norm, and the generic one (d 256 with rot 64, d 64, and
# rot 8, whose table row is a single 16-byte chunk).
WIDE = {
    "w1024_llama_d128": ("llama", 1024, 2, 128, 5e5, {}),
    "w1024_qwen3_knorm": ("qwen3", 1024, 2, 128, 1e6, dict(eps=1e-6)),
    "w1024_qwen35_d256_rot64": ("qwen3_5", 1024, 2, 256, 1e7, dict(eps=1e-6, rot_frac=0.25)),
    "w1024_llama_d64": ("llama", 1024, 4, 64, 1e4, {}),
    "w1024_qwen35_d64_rot8": ("qwen3_5", 1024, 4, 64, 1e7, dict(eps=1e-6, rot_frac=0.125)),
}


def _case(name, layers):
    if name in CASES:
        return case(name, layers=layers)
    arch, h, hkv, d, theta, kw = WIDE[name]
    cfg = attn_config(arch, h, hkv, d, theta, layers=layers, **kw)
    return cfg, random_tensors(cfg, 0)


# P: 700 rows give fewer tiles than CUs for most cases (one tile per block); 20000 rows run every block
# over several tiles, with a ragged last tile row
@pytest.mark.parametrize("P", [700, 20000])
@pytest.mark.parametrize("name", sorted(CASES) + sorted(WIDE))
def test_batch_equals_per_layer(dev, name, P):
    from rfill import ops
    from rfill.model import FillModel
    nl = 3
    cfg, t = _case(name, nl)
    H, hkv, d = cfg["hidden_size"], cfg["num_key_value_heads"], cfg["head_dim"]
    layers = list(range(nl))
    m = FillModel(cfg, t, dev)
    b = inputs(P, H, seed=21).to(dev)
    W, B = _maps(H, layers, 22)
    W, B = [w.to(dev) for w in W], [c.to(dev) for c in B]
    pos = torch.arange(P, device=dev)
    cs = m.rope_table(pos)
    slot0, cap = 5, P + 5 + 64
    sentinel = -7.0
    ref_x, ref_s, ref_c = [], [], []
    for i in layers:
        x, s = ops.map_apply(b, W[i], B[i])
        w = m.W[i]
        kb = torch.full((hkv, cap, d), sentinel, dtype=torch.bfloat16, device=dev)
        vb = kb.clone()
        ops.norm_kv_write(x, s, m.eps, w["wkv"], hkv, d, w.get("k_norm"), m.knorm_kind, cs, kb, vb, slot0)
        ref_x.append(x)
        ref_s.append(s)
        ref_c.append((kb, vb))
    xs = [torch.empty(P, H, dtype=torch.bfloat16, device=dev) for _ in layers]
    ss = [torch.empty(P, H // 256, dtype=torch.float32, device=dev) for _ in layers]
    ops.map_apply_batch(b, W, B, xs, ss)
    kbs = [torch.full((hkv, cap, d), sentinel, dtype=torch.bfloat16, device=dev) for _ in layers]
    vbs = [k.clone() for k in kbs]
    ops.norm_kv_write_batch(xs, ss, m.eps, [m.W[i]["wkv"] for i in layers], hkv, d,
                            [m.W[i].get("k_norm") for i in layers], m.knorm_kind, cs, kbs, vbs, slot0)
    torch.cuda.synchronize()
    for i in layers:
        assert torch.equal(xs[i], ref_x[i]), f"layer {i}: x differs"
        assert torch.equal(ss[i], ref_s[i]), f"layer {i}: statistics differ"
        assert torch.equal(kbs[i], ref_c[i][0]), f"layer {i}: K differs"
        assert torch.equal(vbs[i], ref_c[i][1]), f"layer {i}: V differs"
        assert bool((kbs[i][:, :slot0] == sentinel).all()) and bool((kbs[i][:, slot0 + P:] == sentinel).all())
        assert bool((vbs[i][:, :slot0] == sentinel).all()) and bool((vbs[i][:, slot0 + P:] == sentinel).all())
    # layer 0's K / V against the oracle's fill of the same inputs (sampled rows at P = 20000)
    from oracle import model as OM
    sel = torch.arange(P) if P <= 1000 else torch.randperm(P, generator=torch.Generator().manual_seed(28))[:512].sort().values
    om = OM.OracleModel(cfg, t, dtype=torch.bfloat16)
    oc = om.new_cache()
    om.fill(0, ref_x[0][sel.to(dev)].cpu(), sel, oc)
    ek = rel_err(kbs[0][:, (slot0 + sel).to(dev)], oc[0]["k"])
    ev = rel_err(vbs[0][:, (slot0 + sel).to(dev)], oc[0]["v"])
    print(f"{name} P {P}: K rel err {ek:.2e}, V rel err {ev:.2e} vs the oracle")
    assert ek < 1e-2 and ev < 1e-2


def test_batch_c2_shape(dev):
    """Four late layers at the Llama-8B 32K shape (P = 28672; 7168 map tiles and 3584 K / V tiles, 28 and
    14 per block): bitwise the per-layer unsplit launches; 256 sampled rows of one layer's K / V against
    the oracle's fill of those rows."""
    from oracle import model as OM
    from rfill import ops, synth
    from rfill.model import FillModel
    cfg = synth.LLAMA_8B
    layers = [16, 17, 18, 19]
    tensors = {}
    for i in layers:
        t, _, _ = synth.layer_weights(cfg, i, with_map=False)
        tensors.update(t)
    P, H = 28672, cfg["hidden_size"]
    m = FillModel(cfg, tensors, dev, layers=layers)
    b = synth.hidden_states(P, H).to(dev)
    W, B = _maps(H, layers, 23)
    W, B = [w.to(dev) for w in W], [c.to(dev) for c in B]
    pos = torch.arange(P, device=dev)
    cs = m.rope_table(pos)
    xs = [torch.empty(P, H, dtype=torch.bfloat16, device=dev) for _ in layers]
    ss = [torch.empty(P, H // 256, dtype=torch.float32, device=dev) for _ in layers]
    ops.map_apply_batch(b, W, B, xs, ss)
    kbs = [torch.zeros(8, P + 64, 128, dtype=torch.bfloat16, device=dev) for _ in layers]
    vbs = [k.clone() for k in kbs]
    ops.norm_kv_write_batch(xs, ss, m.eps, [m.W[i]["wkv"] for i in layers], 8, 128, [None] * 4, 0, cs, kbs, vbs, 0)
    for n, i in enumerate(layers):
        x, s = ops.map_apply(b, W[n], B[n])
        assert torch.equal(xs[n], x) and torch.equal(ss[n], s), f"layer {i}: map differs"
        kb, vb = torch.zeros_like(kbs[n]), torch.zeros_like(vbs[n])
        ops.norm_kv_write(x, s, m.eps, m.W[i]["wkv"], 8, 128, None, 0, cs, kb, vb, 0)
        assert torch.equal(kbs[n], kb) and torch.equal(vbs[n], vb), f"layer {i}: K / V differ"
        del x, s, kb, vb
    sel = torch.randperm(P, generator=torch.Generator().manual_seed(24))[:256].sort().values
    om = OM.OracleModel(cfg, tensors, dtype=torch.bfloat16, layers=layers)
    oc = om.new_cache()
    om.fill(17, xs[1][sel.to(dev)].cpu(), sel, oc)
    ek = rel_err(kbs[1][:, sel.to(dev)], oc[17]["k"])
    ev = rel_err(vbs[1][:, sel.to(dev)], oc[17]["v"])
    print(f"C2 batch layer 17: K rel err {ek:.2e}, V rel err {ev:.2e}")
    assert ek < 1e-2 and ev < 1e-2


def test_fill_late_groups_equal_per_layer(dev):
    """fill_late's grouped schedule (ATTN_GROUP attention layers per map launch and K / V launch) gives every
    layer the caches of per-layer unsplit launches, bitwise, with given exact-row inputs scattered in (a width of
    512: the rows' sums are never split)."""
    from rfill import ops
    from rfill.kva import ATTN_GROUP, Arm, Projector, fill_late
    from rfill.model import FillModel
    L, split, N, tail = 8, 2, 3000, 200
    cfg, t = case("qwen3_knorm", layers=L)
    H = cfg["hidden_size"]
    P = N - tail
    late = list(range(split, L))
    assert len(late) > ATTN_GROUP                      # at least one full group and a remainder
    Wl, Bl = _maps(H, late, 25)
    W, B = dict(zip(late, Wl)), dict(zip(late, Bl))
    h = inputs(N, H, seed=26).to(dev)
    rows = torch.tensor([3, 64, 65, 700, 2799])
    hr = inputs(5, H, seed=27)
    m = FillModel(cfg, t, dev)
    arm = Arm("ridgefill", split=split, tail=tail, fill="proj", projector=Projector(split, W, B))
    cache, got_p = fill_late(m, h, arm, exact_rows=rows, hr=hr.to(dev))
    torch.cuda.synchronize()
    assert got_p == P
    pos = torch.arange(P, device=dev)
    cs = m.rope_table(pos)
    for i in late:
        x, s = ops.map_apply(h[:P], W[i].to(dev), B[i].to(dev))
        ops.row_scatter(x, s, rows.to(dev), hr.to(dev))
        w = m.W[i]
        kb = torch.zeros(cfg["num_key_value_heads"], P + 64, cfg["head_dim"], dtype=torch.bfloat16, device=dev)
        vb = kb.clone()
        ops.norm_kv_write(x, s, m.eps, w["wkv"], m.n_kv, m.head_dim, w.get("k_norm"), m.knorm_kind, cs, kb, vb, 0)
        assert cache[i]["n"] == P
        assert torch.equal(cache[i]["k"], kb[:, :P]), f"layer {i}: K differs"
        assert torch.equal(cache[i]["v"], vb[:, :P]), f"layer {i}: V differs"


def test_fill_late_hybrid_groups_equal_per_layer(dev):
    """A hybrid late stack (GDN, GDN, GDN, attention, GDN, GDN) at width 1024 filled by fill_late's grouped
    schedule (one map launch per group, paired GDN fills with one in-projection launch, batched attention
    fills) against per-layer unsplit launches: every GDN conv and recurrent state and the attention layer's K
    / V bitwise equal (2500 rows: no launch leaves rows over)."""
    from fill_cases import hybrid_config, hybrid_tensors
    from rfill import ops
    from rfill.kva import Arm, Projector, fill_late
    from rfill.model import FillModel
    kinds = ["gdn", "gdn", "gdn", "attn", "gdn", "gdn"]
    cfg = hybrid_config(kinds, hidden=1024)
    t = hybrid_tensors(cfg, seed=29)
    H, L, N, tail = cfg["hidden_size"], len(kinds), 2600, 100
    P = N - tail
    late = list(range(L))
    Wl, Bl = _maps(H, late, 30)
    W, B = dict(zip(late, Wl)), dict(zip(late, Bl))
    h = inputs(N, H, seed=31).to(dev)
    m = FillModel(cfg, t, dev)
    arm = Arm("ridgefill", split=0, tail=tail, fill="proj", projector=Projector(0, W, B))
    cache, _ = fill_late(m, h, arm)
    torch.cuda.synchronize()
    ref = m.new_cache()
    pos = torch.arange(P, device=dev)
    for i in late:
        x, s = ops.map_apply(h[:P], W[i].to(dev), B[i].to(dev))
        if kinds[i] == "attn":
            w = m.W[i]
            kb = torch.zeros(m.n_kv, P + 64, m.head_dim, dtype=torch.bfloat16, device=dev)
            vb = kb.clone()
            ops.norm_kv_write(x, s, m.eps, w["wkv"], m.n_kv, m.head_dim, w.get("k_norm"), m.knorm_kind,
                              m.rope_table(pos), kb, vb, 0)
            assert torch.equal(cache[i]["k"], kb[:, :P]) and torch.equal(cache[i]["v"], vb[:, :P]), f"layer {i}"
        else:
            m.fill(i, x, pos, ref, ssq=s)
            assert torch.equal(cache[i]["conv"], ref[i]["conv"]), f"layer {i}: conv state differs"
            assert torch.equal(cache[i]["rec"], ref[i]["rec"]), f"layer {i}: recurrent state differs"


def test_norm_linear_batch_ragged_entries(dev):
    """rf_norm_linear_batch with entries of different rows and widths in one launch (a GDN fill's two
    entries per layer: every row against the k | v | b | a rows, the last 3 rows against the q rows): each
    entry bitwise rf_norm_linear of it alone; the rows and columns outside the entries untouched."""
    from rfill import ops
    g = torch.Generator().manual_seed(21)
    P, H = 1000, 1024
    x = inputs(P, H, seed=22).to(dev)
    ssq = ops.row_ssq(x)
    w = [(torch.randn(n, H, generator=g) / H ** 0.5).to(torch.bfloat16).to(dev) for n in (768, 256, 512)]
    out = torch.full((P, 1280), 3.0, dtype=torch.bfloat16, device=dev)
    ops.norm_linear_batch([x, x[P - 3:], x[:130]], [ssq, ssq[P - 3:], ssq[:130]], 1e-6, w,
                          [out[:, 512:], out[P - 3:, :256], out[:130, :512]])
    torch.cuda.synchronize()
    assert torch.equal(out[:, 512:], ops.norm_linear(x, ssq, 1e-6, w[0]))
    assert torch.equal(out[P - 3:, :256], ops.norm_linear(x[P - 3:], ssq[P - 3:], 1e-6, w[1]))
    assert torch.equal(out[:130, :512], ops.norm_linear(x[:130], ssq[:130], 1e-6, w[2]))
    assert bool((out[130:P - 3, :512] == 3.0).all()) and bool((out[P - 3:, 256:512] == 3.0).all())


# Rows left over by whole rounds of tiles: 1 row, a row block and its edge, several row blocks, every row of a short
# prompt (3 layers of 1024 x 1024 maps: 12 map tiles a tile row, so 21 tile rows are a round; the linear entries: 32)
@pytest.mark.parametrize("P", [1, 160, 161, 448, 21 * 256 + 1, 21 * 256 + 30, 32 * 256 + 30])
@pytest.mark.parametrize("name", sorted(WIDE))
def test_batch_rows_left_over(dev, name, P):
    """Batched launches with a workspace against the same without: the rows of whole rounds keep their bits, the rest
    differ by the order of fp32 sums alone. A sum's two orders differ by at most K 2^-24 of its absolute terms, far
    below bf16's 2^-9, so a result moves by at most one bf16 spacing of the largest value that formed it, and few do:
    1e-3 relative Frobenius, single values within 2^-7 of the row's largest."""
    from rfill import ops
    from rfill.model import FillModel
    nl = 3
    cfg, t = _case(name, nl)
    H, hkv, d = cfg["hidden_size"], cfg["num_key_value_heads"], cfg["head_dim"]
    m = FillModel(cfg, t, dev)
    b = inputs(P, H, seed=41).to(dev)
    W, B = _maps(H, list(range(nl)), 42)
    W, B = [w.to(dev) for w in W], [c.to(dev) for c in B]
    cs = m.rope_table(torch.arange(P, device=dev))
    slot0, cap = 3, P + 3 + 64

    def run(ws_map, ws_kv, ws_lin, given=None):
        xs = [torch.empty(P, H, dtype=torch.bfloat16, device=dev) for _ in range(nl)]
        ss = [torch.empty(P, H // 256, dtype=torch.float32, device=dev) for _ in range(nl)]
        ops.map_apply_batch(b, W, B, xs, ss, ws_map)
        gx, gs = (xs, ss) if given is None else given    # the same inputs for both sides of what follows
        kb = [torch.full((hkv, cap, d), -7.0, dtype=torch.bfloat16, device=dev) for _ in range(nl)]
        vb = [k.clone() for k in kb]
        ops.norm_kv_write_batch(gx, gs, m.eps, [m.W[i]["wkv"] for i in range(nl)], hkv, d,
                                [m.W[i].get("k_norm") for i in range(nl)], m.knorm_kind, cs, kb, vb, slot0, ws_kv)
        lin = [torch.empty(P, H, dtype=torch.bfloat16, device=dev) for _ in range(2)]
        ops.norm_linear_batch([gx[0], gx[1], gx[0][:2]], [gs[0], gs[1], gs[0][:2]], m.eps, [W[1], W[2], W[0][:256]],
                              lin + [torch.empty(2, H, dtype=torch.bfloat16, device=dev)[:, :256]]
                              if P > 2 else lin + [torch.empty(1, H, dtype=torch.bfloat16, device=dev)[:, :256]], ws_lin)
        return xs, ss, kb, vb, lin

    n_kv, small = 2 * hkv * d, min(P, 2)
    need = [ops.batch_workspace_bytes(nl, P, H, H), ops.batch_workspace_bytes(nl, P, n_kv, H),
            ops.norm_linear_batch_workspace_bytes([P, P, small], [H, H, 256], H)]
    assert need[2] > 0 if P in (448, 32 * 256 + 30) else need[0] > 0
    ws = [torch.empty(n, dtype=torch.uint8, device=dev) if n else None for n in need]
    ref = run(None, None, None)
    got = run(*ws, given=ref[:2])
    torch.cuda.synchronize()
    whole = 21 * 256 if P > 21 * 256 else 0             # (P > 32 * 256: the maps' own plan may end later)
    for a, r in zip(got[0], ref[0]):
        assert torch.equal(a[:whole], r[:whole])

    def near(a, r):
        a, r = a.float(), r.float()
        assert float((a - r).norm()) <= 1e-3 * float(r.norm())
        assert bool(((a - r).abs() <= 2.0 ** -7 * r.abs().amax(-1, keepdim=True)).all())
    for group in (0, 2, 3, 4):
        for a, r in zip(got[group], ref[group]):
            near(a, r)
    for a, r in zip(got[1], ref[1]):
        assert torch.allclose(a, r, rtol=2e-2)          # sums of 256 squares of bf16 values, each within 2^-8
    for a in got[2] + got[3]:
        assert bool((a[:, :slot0] == -7).all()) and bool((a[:, slot0 + P:] == -7).all())


def _near(a, r):
    """One bf16 rounding apart, of the few values whose sums' order changed (test_batch_rows_left_over's bar)."""
    a, r = a.float(), r.float()
    assert float((a - r).norm()) <= 1e-3 * float(r.norm())
    assert bool(((a - r).abs() <= 2.0 ** -7 * r.abs().amax(-1, keepdim=True)).all())


def test_fill_late_with_rows_left_over(dev):
    """fill_late at a width and prompt whose launches leave rows over (33 tile rows, the last of 20 rows: K split two
    ways, the split count following the layers in the launch), in a group of four layers and one of two that share the
    call's workspace, against per-layer unsplit launches: rows of the whole rounds bitwise, the rest to one rounding."""
    from rfill import ops
    from rfill.kva import Arm, Projector, fill_late
    from rfill.model import FillModel
    L, split, tail = 8, 2, 100
    whole = 32 * 256
    P = whole + 20
    cfg, t = _case("w1024_qwen3_knorm", L)
    H, hkv, d = cfg["hidden_size"], cfg["num_key_value_heads"], cfg["head_dim"]
    for nl in (4, 2):
        assert ops.batch_workspace_bytes(nl, P, H, H) >= 2 * nl * 20 * H * 4
    assert ops.batch_workspace_bytes(4, P, 2 * hkv * d, H) >= 2 * 4 * 20 * 2 * hkv * d * 4
    late = list(range(split, L))
    Wl, Bl = _maps(H, late, 45)
    W, B = dict(zip(late, Wl)), dict(zip(late, Bl))
    h = inputs(P + tail, H, seed=46).to(dev)
    m = FillModel(cfg, t, dev)
    cache, got_p = fill_late(m, h, Arm("ridgefill", split=split, tail=tail, fill="proj", projector=Projector(split, W, B)))
    torch.cuda.synchronize()
    assert got_p == P
    cs = m.rope_table(torch.arange(P, device=dev))
    for i in late:
        x, s = ops.map_apply(h[:P], W[i].to(dev), B[i].to(dev))
        w = m.W[i]
        kb = torch.zeros(hkv, P + 64, d, dtype=torch.bfloat16, device=dev)
        vb = kb.clone()
        ops.norm_kv_write(x, s, m.eps, w["wkv"], m.n_kv, m.head_dim, w.get("k_norm"), m.knorm_kind, cs, kb, vb, 0)
        for got, want in ((cache[i]["k"], kb), (cache[i]["v"], vb)):
            assert torch.equal(got[:, :whole], want[:, :whole]), f"layer {i}"
            _near(got[:, whole:P], want[:, whole:P])


def test_fill_late_hybrid_with_rows_left_over(dev):
    """The hybrid's grouped schedule with rows left over in its map launch and in the GDN pairs' in-projections, which
    share the call's workspace: the attention layer's K / V as above; a GDN layer's states sum over all rows, of which
    the last 30 carry the changed roundings: 1e-3 of their norm."""
    from fill_cases import hybrid_config, hybrid_tensors
    from rfill import ops
    from rfill.kva import Arm, Projector, fill_late
    from rfill.model import FillModel
    kinds = ["gdn", "gdn", "gdn", "attn", "gdn", "gdn"]
    cfg = hybrid_config(kinds, hidden=1024)
    H, tail, whole = cfg["hidden_size"], 100, 32 * 256
    P = whole + 30
    late = list(range(len(kinds)))
    Wl, Bl = _maps(H, late, 50)
    W, B = dict(zip(late, Wl)), dict(zip(late, Bl))
    h = inputs(P + tail, H, seed=51).to(dev)
    m = FillModel(cfg, hybrid_tensors(cfg, seed=52), dev)
    m._layer(0, "gdn")
    n_in = m.W[0]["w_in"].shape[0] - m.nk * m.dk
    assert ops.batch_workspace_bytes(len(kinds), P, H, H) > 0
    assert ops.norm_linear_batch_workspace_bytes([P, 3, P, 3], [n_in, m.nk * m.dk] * 2, H) > 0
    cache, _ = fill_late(m, h, Arm("ridgefill", split=0, tail=tail, fill="proj", projector=Projector(0, W, B)))
    torch.cuda.synchronize()
    ref, pos = m.new_cache(), torch.arange(P, device=dev)
    for i in late:
        x, s = ops.map_apply(h[:P], W[i].to(dev), B[i].to(dev))
        if kinds[i] == "attn":
            w = m.W[i]
            kb = torch.zeros(m.n_kv, P + 64, m.head_dim, dtype=torch.bfloat16, device=dev)
            vb = kb.clone()
            ops.norm_kv_write(x, s, m.eps, w["wkv"], m.n_kv, m.head_dim, w.get("k_norm"), m.knorm_kind,
                              m.rope_table(pos), kb, vb, 0)
            _near(cache[i]["k"][:, :P], kb[:, :P])
            _near(cache[i]["v"][:, :P], vb[:, :P])
        else:
            m.fill(i, x, pos, ref, ssq=s)
            for part in ("conv", "rec"):
                assert rel_err(cache[i][part], ref[i][part]) < 1e-3, f"layer {i}: {part}"


@pytest.mark.parametrize("small", [1, 161, 200, 256])
def test_norm_linear_batch_small_entry_taller_than_the_rows_left(dev, small):
    """A small entry (at most 256 rows, all of them as few rows) beside 30 rows left over by the large one: its row
    blocks are taller than the plan's, one or two of them."""
    from rfill import ops
    P, H, n = 32 * 256 + 30, 1024, 2048
    g = torch.Generator().manual_seed(small)
    x = inputs(P, H, seed=53).to(dev)
    ssq = ops.row_ssq(x)
    w = [(torch.randn(k, H, generator=g) / H ** 0.5).to(torch.bfloat16).to(dev) for k in (n, 512)]
    need = ops.norm_linear_batch_workspace_bytes([P, small], [n, 512], H)
    assert need > 0 and need % (30 * n * 4 + small * 512 * 4) == 0
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    outs = [[torch.full((P + 1, n), 3.0, dtype=torch.bfloat16, device=dev) for _ in range(2)] for _ in range(2)]
    for o, space in zip(outs, (ws, None)):
        ops.norm_linear_batch([x, x[:small]], [ssq, ssq[:small]], 1e-6, w, [o[0][:P], o[1][:small, :512]], space)
    torch.cuda.synchronize()
    (a, b), (ra, rb) = outs
    assert torch.equal(a[:32 * 256], ra[:32 * 256])
    _near(a[32 * 256:P], ra[32 * 256:P])
    _near(b[:small, :512], rb[:small, :512])
    assert bool((a[P:] == 3.0).all()) and bool((b[small:] == 3.0).all()) and bool((b[:small, 512:] == 3.0).all())
