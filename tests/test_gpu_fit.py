"""GPU parity of the closed-form fit: rf_transpose (bit-exact, column sums), rf_gram_accumulate (fp32
over the block into fp64), RidgeStats on the device against the oracle's RidgeStats, and RidgeFit's
fp64 solve against the oracle's fp64 eigendecomposition solve. Bar for fitted maps: relative Frobenius
error <= 1e-5 against the fp64 reference solve."""
import pytest
import torch

from oracle import ridge as oridge

pytestmark = pytest.mark.gpu
MAP_TOL = 1e-5


def rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).norm() / b.norm())


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return torch.device("cuda")


def test_transpose_is_bit_exact_with_column_sums(dev):
    from rfill import ridge
    g = torch.Generator().manual_seed(0)
    x = torch.randn(1000, 512, generator=g).to(torch.bfloat16).to(dev)
    dst = torch.full((512, 1088), 5.0, dtype=torch.bfloat16, device=dev)
    part = torch.empty(1024 // 64, 512, dtype=torch.float32, device=dev)
    ridge._transpose(x, dst[:, :1024], part)
    torch.cuda.synchronize()
    assert torch.equal(dst[:, :1000], x.T)
    assert bool((dst[:, 1000:1024] == 0).all()) and bool((dst[:, 1024:] == 5.0).all())
    sums = torch.zeros(512, dtype=torch.float64, device=dev)
    ridge._colsum_fold(part, sums)
    assert rel(sums, x.double().sum(0)) < 1e-6


@pytest.mark.parametrize("fold_rows", [0, 128, 512])
def test_gram_accumulate_matches_fp64_products(dev, fold_rows):
    """fp32 runs of at most fold_rows added into fp64 in run order, against fp64 products; fold_rows 0 sums
    the whole K in fp32. The same bits run to run."""
    from rfill import ridge
    g = torch.Generator().manual_seed(1)
    a = torch.randn(384, 1024, generator=g).to(torch.bfloat16)
    b = (torch.randn(768, 1024, generator=g) * 3).to(torch.bfloat16)
    c0 = torch.randn(384, 768, generator=g, dtype=torch.float64)
    c = c0.to(dev)
    ridge.gram_accumulate(a.to(dev), b.to(dev), c, fold_rows)
    want = c0 + a.double() @ b.double().T
    err = rel(c, want)
    print(f"gram (fold_rows {fold_rows}) rel err {err:.2e}")
    assert err < 1e-6
    again = c0.to(dev)
    ridge.gram_accumulate(a.to(dev), b.to(dev), again, fold_rows)
    assert torch.equal(again, c)


@pytest.mark.parametrize("M,N,K,fold_rows", [(4104, 4352, 12288, 8192), (4352, 4096, 16384, 4096)])
def test_gram_run_split_schedule_is_bit_identical(dev, M, N, K, fold_rows):
    """Tile counts just past one round of the GPU's 256 CUs (a centred operand's extra rows / columns: 289
    and 272 tiles): with a workspace the tiles past the first 256 run as single runs whose fp32 sums a second
    kernel adds into C in run order. The same bits as every tile whole (no workspace, or one a byte short),
    nothing written past the workspace (a guard region after it), and fp64 products to 1e-6; the first
    shape's last run is shorter than fold_rows (12288 = 8192 + 4096)."""
    from rfill import _lib, ridge
    from rfill.ops import _ptr, _stream
    need = ridge.gram_workspace_bytes(M, N, K, fold_rows)
    assert need > 0
    g = torch.Generator(device=dev).manual_seed(3)
    a = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g, device=dev) * 2).to(torch.bfloat16)
    c0 = torch.randn(M, N, generator=g, device=dev, dtype=torch.float64)
    whole = c0.clone()
    _lib.call("rf_gram_accumulate", _ptr(a), a.stride(0), _ptr(b), b.stride(0), M, N, K, fold_rows, _ptr(whole),
              whole.stride(0), None, 0, _stream(a))
    guard = 1 << 20
    buf = torch.full((need + guard,), 0xFF, dtype=torch.uint8, device=dev)     # stale contents must not matter
    split = c0.clone()
    _lib.call("rf_gram_accumulate", _ptr(a), a.stride(0), _ptr(b), b.stride(0), M, N, K, fold_rows, _ptr(split),
              split.stride(0), _ptr(buf), need, _stream(a))
    short = c0.clone()                                                  # one byte short: every tile whole
    _lib.call("rf_gram_accumulate", _ptr(a), a.stride(0), _ptr(b), b.stride(0), M, N, K, fold_rows, _ptr(short),
              short.stride(0), _ptr(buf), need - 1, _stream(a))
    torch.cuda.synchronize()
    assert torch.equal(split, whole) and torch.equal(short, whole)
    assert bool((buf[need:] == 0xFF).all()), "the run-split schedule wrote past its workspace"
    err = rel(split - c0, a.double() @ b.double().T)
    print(f"gram {M} x {N} x {K} (fold {fold_rows}) run-split rel err {err:.2e}")
    assert err < 1e-6


@pytest.mark.parametrize("M,N,K,fold_rows", [(4104, 4352, 16384, 8192), (1024, 1024, 12288, 8192),
                                              (768, 1024, 2048, 0)])
def test_gram_upper_is_the_full_product_on_its_tiles(dev, M, N, K, fold_rows):
    """The symmetric X^T X on C's block-upper tiles (a centred X's 4104 rows against its 4352-row operand: 153
    of 289 tiles, each split into its two runs; a short last run; one run, whole tiles): those tiles
    bit-identical to rf_gram_accumulate of the same operands, the block-lower tiles untouched, the same bits
    with no workspace, nothing written past the workspace, and after mirror_block_upper the full product
    (fp64 products to 1e-6; the full launch's own lower tiles differ from the mirrored upper ones by fp32
    summation order only, about 1e-13 of C here)."""
    from rfill import _lib, ridge
    from rfill.ops import _ptr, _stream
    g = torch.Generator(device=dev).manual_seed(5)
    a = torch.randn(N, K, generator=g, device=dev).to(torch.bfloat16)
    a[M:] = 0                                                           # rows past M: a centred operand's padding
    c0 = torch.randn(M, N, generator=g, device=dev, dtype=torch.float64)
    c0[:, :M] += c0[:, :M].T.clone()                                    # a symmetric running sum, as RidgeStats'
    full = c0.clone()
    ridge.gram_accumulate(a[:M], a, full, fold_rows)
    need = ridge.gram_upper_workspace_bytes(M, N, K, fold_rows)
    assert (need > 0) == (fold_rows > 0)
    guard = 1 << 20
    buf = torch.full((need + guard,), 0xFF, dtype=torch.uint8, device=dev)
    up = c0.clone()
    _lib.call("rf_gram_accumulate_upper", _ptr(a), a.stride(0), M, N, K, fold_rows, _ptr(up), up.stride(0),
              _ptr(buf), need, _stream(a))
    whole = c0.clone()
    ridge.gram_accumulate_upper(a, M, whole, fold_rows, torch.empty(0, dtype=torch.uint8, device=dev))
    torch.cuda.synchronize()
    assert bool((buf[need:] == 0xFF).all()), "the upper schedule wrote past its workspace"
    assert torch.equal(whole, up)
    ti = torch.arange(M, device=dev)[:, None] // 256
    tj = torch.arange(N, device=dev)[None, :] // 256
    upper = tj >= ti
    assert torch.equal(up[upper], full[upper])
    assert torch.equal(up[~upper], c0[~upper])
    ridge.mirror_block_upper(up)
    sym = full[:, :M] - c0[:, :M]
    asym = float((sym - sym.T).abs().max())
    print(f"gram upper {M} x {N} x {K} (fold {fold_rows}): full product symmetric to {asym:.1e}")
    d = a[:M].double()
    want = d @ a.double().T
    assert torch.equal(up[:, M:], c0[:, M:])                           # products with the zero rows
    low = ~upper[:, :M]
    assert torch.equal(up[:, :M][low], (up[:, :M].T)[low])
    err = rel(up[:, :M][low] - c0[:, :M][low], want[:, :M][low])
    assert err < 1e-6, err


def test_gram_accumulate_refuses_bad_fold(dev):
    from rfill import ridge
    a = torch.zeros(256, 128, dtype=torch.bfloat16, device=dev)
    c = torch.zeros(256, 256, dtype=torch.float64, device=dev)
    with pytest.raises(ValueError, match="fold_rows"):
        ridge.gram_accumulate(a, a, c, 96)


def _student(n, d, seed):
    from rfill import synth
    g = torch.Generator().manual_seed(seed)
    x = synth.student_t((n, d), 5, g, "cpu")
    x[:, :4] *= 20
    return x.to(torch.bfloat16)


def test_ridge_stats_and_fit_match_the_oracle(dev):
    """Config-5-shaped data at a reduced size (d 512, 2 targets, 20000 rows, ragged last block): the
    device statistics against the oracle's (fp32 block GEMMs into fp64), and the maps fitted from each
    against the oracle's fp64 solve."""
    from rfill import ridge
    n, d = 20000, 512
    x = _student(n, d, 2)
    g = torch.Generator().manual_seed(3)
    ys = {}
    for i in (5, 6):
        t = torch.eye(d) + 0.05 * torch.randn(d, d, generator=g) / d ** 0.5
        ys[i] = (x.float() @ t + 0.1 * torch.randn(n, d, generator=g)).to(torch.bfloat16)
    mine = ridge.RidgeStats(4, [5, 6], d, device=dev)
    mine.add(x.to(dev), {i: y.to(dev) for i, y in ys.items()}, block=8192)
    ms = mine.state()
    ref = oridge.RidgeStats(4, [5, 6], d)
    ref.add(x, ys, block=8192)
    rs = ref.state()
    for k in ("sx", "sxx"):
        print(k, rel(ms[k], rs[k]))
        assert rel(ms[k], rs[k]) < 1e-5, k
    for i in (5, 6):
        assert rel(ms["sxy"][i], rs["sxy"][i]) < 1e-5
    ofit = oridge.RidgeFit(rs)
    same = ridge.RidgeFit(rs, device=dev)           # the solve alone, on the oracle's statistics
    full = ridge.RidgeFit(ms, device=dev)           # device statistics + device solve
    for lam in (1e-4, 1e-3, 1e-2):
        w_ref, b_ref = ofit.layer_f64(6, lam)
        w1, b1 = same.layer(6, (lam,))[lam]
        w2, b2 = full.layer(6, (lam,))[lam]
        e1, e2 = rel(w1, w_ref), rel(w2, w_ref)
        print(f"lam {lam:g}: solve-only rel err {e1:.2e}, stats+solve rel err {e2:.2e}")
        assert e1 < MAP_TOL and rel(b1, b_ref) < MAP_TOL
        assert e2 < MAP_TOL


def _centred(st, i):
    """Shift-free statistics of a state: the means of x and y_i, C = sxx - sx sx^T / n, Cxy = sxy - sx sy^T / n."""
    n = float(st["n"])
    sx, sy = st["sx"].double().cpu(), st["sy"][i].double().cpu()
    return dict(mx=st["cx"].double().cpu() + sx / n, my=st["cy"][i].double().cpu() + sy / n,
                c=st["sxx"].double().cpu() - torch.outer(sx, sx) / n,
                cxy=st["sxy"][i].double().cpu() - torch.outer(sx, sy) / n)


def test_resumed_statistics_continue_the_device_sums(dev):
    """RidgeStats.from_state on the device (the reference's resumable sufficient statistics,
    code/scripts/fit_sweep.py:20-25, :271-284): a state saved after the first 7000 rows, moved to the host
    and back as a saved file would be, then continued with the remaining rows, keeps the saved shifts and
    gives one pass's means, centred scatter and centred cross products (1e-6); a resume that adds layer 5
    only carries layer 6's saved sums unchanged; maps fitted from the resumed state agree with one pass's
    (1e-5)."""
    from rfill import ridge
    n, d = 20000, 512
    x = _student(n, d, 7)
    g = torch.Generator().manual_seed(8)
    ys = {}
    for i in (5, 6):
        t = torch.eye(d) + 0.05 * torch.randn(d, d, generator=g) / d ** 0.5
        ys[i] = (x.float() @ t + 0.1 * torch.randn(n, d, generator=g)).to(torch.bfloat16)
    xd, yd = x.to(dev), {i: y.to(dev) for i, y in ys.items()}
    one = ridge.RidgeStats(4, [5, 6], d, device=dev)
    one.add(xd, yd, block=8192)
    want = one.state()
    first = ridge.RidgeStats(4, [5, 6], d, device=dev)
    first.add(xd[:7000], {i: y[:7000] for i, y in yd.items()}, block=8192)
    saved = first.state(device="cpu")
    resumed = ridge.RidgeStats.from_state(saved, device=dev)
    resumed.add(xd[7000:], {i: y[7000:] for i, y in yd.items()}, block=8192)
    got = resumed.state()
    assert got["n"] == n and torch.equal(got["cx"].cpu(), saved["cx"].cpu())
    for i in (5, 6):
        assert torch.equal(got["cy"][i].cpu(), saved["cy"][i].cpu())
    # the shifts differ (the first 8192-row block's means against the first 7000 rows'), so compare the
    # statistics every shift gives alike: means, centred scatter and centred cross products
    for (k, a), (_, b) in zip(_centred(got, 5).items(), _centred(want, 5).items()):
        assert rel(a, b) < 1e-6, (k, rel(a, b))
    for (k, a), (_, b) in zip(_centred(got, 6).items(), _centred(want, 6).items()):
        assert rel(a, b) < 1e-6, (k, rel(a, b))
    part = ridge.RidgeStats.from_state(saved, device=dev)
    part.begin(xd[7000:], block=8192)
    part.add_layer(5, yd[5][7000:])
    ps = part.state()
    assert rel(_centred(ps, 5)["cxy"], _centred(want, 5)["cxy"]) < 1e-6
    for k in ("cy", "sy", "sxy"):
        assert torch.equal(ps[k][6].cpu(), saved[k][6].cpu()), k
    fa, fb = ridge.RidgeFit(got, device=dev), ridge.RidgeFit(want, device=dev)
    for lam in (1e-3, 1e-2):
        wa, ba = fa.layer(6, (lam,))[lam]
        wb, bb = fb.layer(6, (lam,))[lam]
        assert rel(wa, wb) < 1e-5 and rel(ba, bb) < 1e-5


@pytest.mark.parametrize("da,ea,db,eb,K,fold,upper", [
    (256, 0, 512, 0, 640, 256, False), (256, 2, 512, 6, 64, 0, False), (512, 256, 256, 250, 1088, 512, False),
    (512, 0, 512, 34, 2048, 0, False), (512, 66, 256, 0, 4160, 1024, False), (768, 8, 768, 8, 8192, 8192, True),
    (512, 162, 512, 162, 3136, 2048, True), (512, 0, 512, 0, 1088, 256, True)])
@pytest.mark.parametrize("init", [False, True])
def test_gram_centred_is_the_augmented_product(dev, da, ea, db, eb, K, fold, upper, init):
    """rf_gram_centred over its operands' main and extra rows (no extra rows, few, the most; one or two row blocks;
    K of one step, not a multiple of the splits; short last runs) against fp64 products: 1e-6 of their norm, the
    fp32 sums' bound as above. Columns past the extra ones stay untouched, with init the old values do not matter,
    and only the workspace it asks for is written."""
    from rfill import ridge
    g = torch.Generator(device=dev).manual_seed(da + ea + eb + K)
    a = torch.randn(da + 256, K + 64, generator=g, device=dev).to(torch.bfloat16)[:, :K]
    b = a if upper else (torch.randn(db + 256, K + 64, generator=g, device=dev) * 2).to(torch.bfloat16)[:, :K]
    c0 = torch.randn(da + ea, db + 256, generator=g, device=dev, dtype=torch.float64)
    need = ridge.gram_centred_workspace_bytes(da, ea, db, eb, K, fold, upper)
    buf = torch.full((need + 4096,), 0xFF, dtype=torch.uint8, device=dev)
    c = torch.full_like(c0, float("nan")) if init else c0.clone()
    old = c.clone()
    ridge.gram_centred(a, da, ea, b, db, eb, c, fold, upper, init, buf[:need] if need else None)
    torch.cuda.synchronize()
    assert bool((buf[need:] == 0xFF).all()), "wrote past its workspace"
    want = a[:da + ea].double() @ b[:db + eb].double().T + (0 if init else c0[:, :db + eb])
    ti = torch.arange(da + ea, device=dev)[:, None] // 256
    tj = torch.arange(db + eb, device=dev)[None, :] // 256
    live = tj >= ti if upper else torch.ones(da + ea, db + eb, dtype=torch.bool, device=dev)
    err = rel(c[:, :db + eb][live], want[live])
    print(f"gram centred rel err {err:.2e}")
    assert err < 1e-6
    assert torch.equal(c[:, db + eb:].isnan(), old[:, db + eb:].isnan())
    assert init or torch.equal(c[:, db + eb:], c0[:, db + eb:])


@pytest.mark.parametrize("cols,cap,given,kind", [(256, 128, False, "few"), (4096, 128, False, "many"), (1088, 3, True, "ties"),
                                                 (2048, 0, False, "many"), (3072, 128, False, "none"), (512, 512, False, "all")])
def test_centring_and_state_on_the_gpu_match_the_host_path(dev, cols, cap, given, kind):
    """rf_centre_select against Centring on the CPU from the same sums (nothing centred, few, more than the cap, equal
    ratios), every output equal; then rf_gram_state against centred_products and recentre on the CPU, to fp64
    rounding (4 parts and 3 rank-1 terms: 1e-14 of the largest term)."""
    from rfill import ridge
    g = torch.Generator().manual_seed(cols + cap)
    n, f64 = 1000, torch.float64
    mean = torch.randn(cols, generator=g, dtype=f64)
    spread = torch.rand(cols, generator=g, dtype=f64) + 0.5
    if kind == "few":
        mean *= torch.where(torch.arange(cols) % 50 == 7, 8.0, 0.1)
    elif kind == "ties":
        mean, spread = torch.full_like(mean, 2.0), torch.ones_like(spread)
    elif kind == "none":
        mean *= 0.01
    elif kind == "all":
        mean = mean.sign() * 4 + mean
    s1, s2 = mean * n, (spread ** 2 + mean ** 2) * n
    c = (mean * 1.01).float().double() if given else None
    want = ridge.Centring(s1, s2, n, c, cap)
    got = ridge.Centring(s1.to(dev), s2.to(dev), n, c, cap)
    for name in ("c", "shift", "lo_row", "idx", "delta"):
        assert torch.equal(getattr(got, name).cpu(), getattr(want, name)), name
    assert got.s == want.s and got.lo_rows == want.lo_rows
    if cols > 1100:
        return
    for upper in (False, True):
        rows = want.s if upper else min(want.s, 2)
        A = want if upper else ridge.Centring(s1[:320] if cols >= 320 else s1, s2[:320] if cols >= 320 else s2, n, None, rows)
        Ag = got if upper else ridge.Centring(s1[:A.c.numel()].to(dev), s2[:A.c.numel()].to(dev), n, None, rows)
        ca = A.c.numel()
        G = torch.randn(ca + 2 * A.s, cols + 2 * want.s + 8, generator=g, dtype=f64)
        if upper:                                   # symmetric over its stored part, the block-lower tiles not stored
            m = cols + 2 * want.s
            G[:, :m] += G[:, :m].T.clone()
        s1a, s1b = torch.randn(ca, generator=g, dtype=f64), torch.randn(cols, generator=g, dtype=f64)
        ref = ridge.recentre(ridge.centred_products(G, ca, A, cols, want), s1a, s1b, A.delta, want.delta, float(n))
        dG = G.to(dev)
        if upper:
            lower = torch.arange(G.shape[0])[:, None] // 256 > torch.arange(G.shape[1])[None, :] // 256
            dG[lower.to(dev)] = float("nan")
        out = ridge.centred_state(dG, ca, Ag, cols, got, s1a.to(dev), s1b.to(dev), float(n), upper)
        big = n * float((A.delta.abs().max() * want.delta.abs().max())) + 10
        assert float((out.cpu() - ref).abs().max()) < 1e-14 * big * 8, (upper, float((out.cpu() - ref).abs().max()))


def test_gram_and_state_refuse_what_the_kernels_do_not_check(dev):
    """Operands whose type, size or device the kernels take on trust: refused before a launch."""
    from rfill import ridge
    f64, d = torch.float64, 256
    a = torch.zeros(d + 8, 128, dtype=torch.bfloat16, device=dev)
    c = torch.zeros(d + 4, d + 8, dtype=f64, device=dev)
    for ws in (torch.empty(1 << 20, dtype=torch.float32, device=dev), torch.empty(1 << 20, dtype=torch.uint8)):
        with pytest.raises(ValueError):
            ridge.gram_centred(a, d, 4, a, d, 4, c, workspace=ws)
    sums = torch.full((d,), 100.0, dtype=f64, device=dev)
    sums[3] = 10000.0
    A = ridge.Centring(sums, sums * 120, 100, None, 2)
    cpu = ridge.Centring(sums.cpu(), sums.cpu() * 120, 100, None, 2)
    assert A.s == cpu.s == 1
    G = torch.zeros(d + 2, d + 2, dtype=f64, device=dev)
    assert ridge.centred_state(G, d, A, d, A, sums, sums, 100, True).shape == (d, d)
    for bad in ((G[:d + 1], A, sums, sums), (G[:, :d + 1], A, sums, sums), (G.float(), A, sums, sums),
                (G, cpu, sums, sums), (G, A, sums[:-1], sums), (G, A, sums, sums.float()), (G, A, sums.cpu(), sums)):
        g, op, s1a, s1b = bad
        with pytest.raises(ValueError):
            ridge.centred_state(g, d, op, d, op, s1a, s1b, 100)
    with pytest.raises(ValueError):
        ridge.Centring(sums, sums[1:], 100)
    with pytest.raises(ValueError):
        ridge.Centring(sums, sums, 100, torch.zeros(1, dtype=f64))
    # sums in another type or stride are read as the values they are
    wide = torch.stack((sums, sums * 120)).t().contiguous()
    B = ridge.Centring(wide[:, 0], wide[:, 1].float(), 100, None, 2)
    for name in ("c", "shift", "lo_row", "idx", "delta"):
        assert torch.equal(getattr(A, name), getattr(B, name))


@pytest.mark.parametrize("cols,cap", [(320, 1), (1024, 128), (4096, 128), (16448, 128), (16448, 0), (1025, 1024)])
def test_centring_past_its_cap(dev, cols, cap):
    """More channels qualify than the cap: equal ratios on both sides of it (taken in channel order), infinite ones (no
    variance), ones that differ in their last digits only; every output equal to the CPU's. Its time grows with the
    channels, not with their square: 16448 of them well under 5 ms (0.12 ms measured, 20 ms if each is ranked against
    all)."""
    import time
    from rfill import ridge
    g = torch.Generator().manual_seed(cols + cap)
    n = 1000
    mean = torch.randint(2, 6, (cols,), generator=g).double()       # ratios 4, 9, 16, 25 over unit variance, many of each
    var = torch.ones(cols, dtype=torch.float64)
    k = torch.arange(cols)
    var = torch.where(k % 7 == 0, 1 + 2.0 ** -40 * k.double(), var)
    var = torch.where(k % 97 == 5, 0.0, var)
    mean = torch.where(k % 97 == 5, 2.0 ** 20, mean)                # 2^40 / 1e-300: infinite
    mean = torch.where(k % 3 == 1, 0.25, mean)                      # these do not qualify
    s1, s2 = mean * n, (var + mean ** 2) * n
    want = ridge.Centring(s1, s2, n, None, cap)
    d1, d2 = s1.to(dev), s2.to(dev)
    for _ in range(3):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        got = ridge.Centring(d1, d2, n, None, cap)
        took = time.perf_counter() - t0
    assert got.s == want.s == min(cap, int((want.c ** 2 > var).sum()))
    for name in ("c", "shift", "lo_row", "idx", "delta"):
        assert torch.equal(getattr(got, name).cpu(), getattr(want, name)), name
    assert took < 5e-3


@pytest.mark.parametrize("init", [False, True])
@pytest.mark.parametrize("da,ea,db,eb,K,upper", [(256, 130, 256, 160, 1088, False), (512, 160, 512, 160, 640, True),
                                                 (256, 132, 256, 2, 2048, False)])
def test_gram_centred_with_one_tall_row_block(dev, da, ea, db, eb, K, upper, init):
    """130 to 160 extra rows (their count is even): one row block of five row tiles."""
    test_gram_centred_is_the_augmented_product(dev, da, ea, db, eb, K, 512, upper, init)
