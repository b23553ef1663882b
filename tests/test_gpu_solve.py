"""GPU parity of the ridge solve (rf_ridge_solve: the inverse of C + lam s I by block recursion on Schur
complements over a 128 x 128 Gauss-Jordan base, fp64 MFMA products) against torch.linalg.solve in fp64 on the
same device (the oracle), for sizes on and off the 128-multiple grid (the padded identity block), several
right-hand-side widths and lambdas, and the bias mean_y - mean_x W. Bar: 1e-10 relative Frobenius (fp64
arithmetic on matrices of condition number up to ~1e4)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 1e-10


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from rfill import _lib
    _lib.load()
    return torch.device("cuda")


def _spd(d, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(4 * d, d, generator=g, device=dev, dtype=torch.float64)
    x[:, :3] *= 20                                        # outlier channels, as in the fit workload
    xc = x - x.mean(0)
    return xc.T @ xc, g


def rel(a, b):
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("d,R", [(64, 64), (100, 2), (192, 200), (512, 1024), (1000, 130), (4096, 256)])
def test_ridge_solve_matches_fp64_solve(dev, d, R):
    from rfill.ridge import RidgeFit
    C, g = _spd(d, d, dev)
    B = torch.randn(d, R, generator=g, device=dev, dtype=torch.float64) * 50
    fit = RidgeFit.__new__(RidgeFit)
    fit.device, fit.cxx = dev, C.contiguous()
    fit.scale = C.diagonal().mean().item()
    fit.mean_x = torch.randn(d, generator=g, device=dev, dtype=torch.float64)
    mean_y = torch.randn(R, generator=g, device=dev, dtype=torch.float64)
    lams = (1e-4, 1e-2, 1.0)
    w, b = fit.solve(B, lams, mean_y)
    torch.cuda.synchronize()
    worst = 0.0
    for li, lam in enumerate(lams):
        want = torch.linalg.solve(C + lam * fit.scale * torch.eye(d, device=dev, dtype=torch.float64), B)
        worst = max(worst, rel(w[li], want), rel(b[li], mean_y - fit.mean_x @ want))
    print(f"rf_ridge_solve d {d}, R {R}: worst rel err {worst:.2e}")
    assert worst < TOL


# inverse: one leaf, an uneven split (128 + 64), two and three levels; weights: ragged last tiles, targets narrower
# than a tile and more than one launch's 64 of them, more than one batch of 8 lambdas
@pytest.mark.parametrize("d,width,targets,nlam", [(64, 2, 65, 1), (130, 200, 3, 9), (640, 130, 2, 2), (1000, 512, 1, 3)])
def test_weights_in_linear_layout(dev, d, width, targets, nlam):
    """RidgeFit.layers' weights (rf_ridge_solve_wt) against the fp64 solve's, transposed and rounded: the same fp64
    values up to their own rounding (1e-12 relative to the largest), so at most one fp32 spacing apart."""
    from rfill.ridge import RidgeFit
    C, g = _spd(d, d + 1, dev)
    fit = RidgeFit.__new__(RidgeFit)
    fit.device, fit.cxx, fit.scale = dev, C.contiguous(), C.diagonal().mean().item()
    fit.mean_x = torch.randn(d, generator=g, device=dev, dtype=torch.float64)
    B = torch.randn(d, targets * width, generator=g, device=dev, dtype=torch.float64) * 50
    my = torch.randn(targets * width, generator=g, device=dev, dtype=torch.float64)
    lams = [1e-3 * 2 ** k for k in range(nlam)]
    w, b = fit.solve(B, lams, my)
    wt, bt = fit._solve_wt(B, width, lams, my)
    assert torch.equal(b, bt) and len(wt) == targets
    for j in range(targets):
        want = w[:, :, j * width:(j + 1) * width].transpose(1, 2)
        diff = (wt[j].double() - want).abs()
        assert tuple(wt[j].shape) == (nlam, width, d)
        assert bool((diff <= 2.0 ** -23 * want.abs() + 1e-12 * want.abs().max()).all()), f"target {j}"


def test_ridge_solve_refuses(dev):
    from rfill.ridge import RidgeFit
    C, g = _spd(64, 1, dev)
    fit = RidgeFit.__new__(RidgeFit)
    fit.device, fit.cxx, fit.scale = dev, C.contiguous(), C.diagonal().mean().item()
    fit.mean_x = torch.zeros(64, device=dev, dtype=torch.float64)
    with pytest.raises(ValueError, match="positive"):
        fit.solve(torch.ones(64, 2, device=dev, dtype=torch.float64), (0.0,))
    with pytest.raises(ValueError, match="even"):
        fit.solve(torch.ones(64, 3, device=dev, dtype=torch.float64), (1.0,))
