"""``ttc_lqr_pad`` against torch's pad: whole vectors and matrices, edges of the four-element groups, both
storage types, and its argument checks."""
import ctypes

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,H,d,du,D", [(1, 1, 1, 1, 16), (3, 5, 15, 13, 16), (2, 3, 17, 16, 32), (257, 2, 24, 20, 32),
                                        (1, 7, 63, 64, 64), (5, 1, 33, 2, 64)])
def test_pad_equals_torch(dtype, N, H, d, du, D):
    from ttc.solvers.hip_lqr import _pad_tensors
    F = torch.nn.functional
    g = torch.Generator(device="cuda").manual_seed(d)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)  # noqa: E731
    xs = [mk(N, H, d), mk(N, d, du), mk(N, H, du), mk(N, H, d, d)]
    got = _pad_tensors(xs, [(D,), (D, D), (D,), (D, D)], [0, 0, 1, 0])
    want = [F.pad(xs[0], (0, D - d)), F.pad(xs[1], (0, D - du, 0, D - d)), F.pad(xs[2], (0, D - du), value=1.0),
            F.pad(xs[3], (0, D - d, 0, D - d))]
    for a, b in zip(got, want):
        assert a.dtype == dtype and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("d,du", [(5, 0), (0, 3), (0, 0)])
def test_sizes_without_elements(d, du):
    """No controls or no states: the solvers and the layer pad them like any other size, u is empty or zero
    and so are the gradients."""
    from ttc import TTCLayer
    from ttc.solvers.hip_lqr import hip_lqr_solve, hip_lqr_solve_factored
    N, H, r = 3, 2, 4
    ones = lambda *s: torch.ones(*s, device="cuda", requires_grad=True)  # noqa: E731
    lgs = [ones(N, H), ones(N, H, du), ones(N, H, d)]
    ins = [ones(N, H, d), ones(N, d, du), ones(N, d, d), ones(N, H, du), ones(N, H, d, d), *lgs, ones(N, H, d)]
    fact = [ones(N, H, d), ones(N, r), ones(N, r), ones(N, H, du), ones(N, H, r), *lgs, ones(N, H, d),
            ones(r, d, du), ones(r, d, d)]
    for solve, xs in ((hip_lqr_solve, ins), (hip_lqr_solve_factored, fact)):
        u = solve(*xs, 4)
        assert u.shape == (N, H, du) and not u.any()
        for x, g in zip(xs, torch.autograd.grad(u.sum(), xs)):
            assert g.shape == x.shape and not g.any()
    if d:
        layer = TTCLayer(8, 8, d, H, r, r, u_dim=du).cuda()
        x = torch.randn(N, 8, device="cuda", requires_grad=True)
        y = layer(x, T=4)
        y.sum().backward()
        assert y.shape == (N, 8) and not y.any() and not x.grad.any()


@pytest.mark.gpu
def test_pad_beyond_one_launch():
    """2^34 padded values and a few more, which are more than the 2^32 - 1 threads of one launch (four values
    each) write: both ends, and the seam of the two launches, hold the inputs and the fill."""
    from ttc.solvers.hip_lqr import _pad_tensors
    M = (1 << 22) + 5
    if torch.cuda.mem_get_info()[0] < 48 << 30:
        pytest.skip("needs 36 GB")
    x = torch.randn(M, 2, 3, device="cuda").to(torch.bfloat16)
    (got,) = _pad_tensors([x], [(64, 64)], [1])
    assert got.shape == (M, 64, 64)
    for part in (slice(0, 8), slice((1 << 22) - 8, M)):
        want = torch.nn.functional.pad(x[part], (0, 61, 0, 62), value=1.0)
        assert torch.equal(got[part], want)


def test_pad_argument_validation():
    from ttc.solvers._lib import lib
    p = (ctypes.c_void_p * 1)(64)
    call = lambda shape, n=1, size=4: lib.ttc_lqr_pad(p, p, (ctypes.c_int64 * 5)(*shape), (ctypes.c_float * 1)(0), n,  # noqa: E731
                                                      size, None)
    assert call((1, 1, 3, 1, 24)) == 1   # not a power of two
    assert call((1, 1, 17, 1, 16)) == 1  # larger than the padded size
    assert call((1, 1, 3, 1, 16), n=13) == 1
    assert call((1, 1, 3, 1, 16), size=8) == 1
    assert call((0, 1, 3, 1, 16)) == 0   # nothing to do
