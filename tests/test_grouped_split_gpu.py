"""The grouped expert projections as one launch over all experts (three exact bf16
planes on the matrix cores), at the edges of its tiles and runs, against float64."""
import pytest
import torch

from summa_amd import ops

pytestmark = pytest.mark.gpu


def _bound(K):
    """Relative to sum |a||b|: the plane products left out (below 3 x 2^-24) and
    half of the 6 K / 16 f32 additions, whose errors have either sign."""
    return 2.0 ** -21 + 2.0 ** -22 + (3 * K / 16 + 2) * 2.0 ** -24


# An empty first, middle and last expert; runs ending at and around the 64-k
# blocks and 128-row tiles; odd widths; more experts than one launch takes; one
# expert with every row (the wide tiles).
CASES = [([0, 63, 64, 65, 0, 127, 128, 129, 1, 0], 200, 333),
         ([40] * 70 + [0, 9], 96, 168),
         ([1000, 1, 999, 2100], 260, 1030),
         ([9000], 128, 2304)]


@pytest.mark.parametrize("counts,din,dout", CASES)
def test_grouped_linear_split_matches_f64(dev, counts, din, dout):
    R, E = sum(counts), len(counts)
    print(f"case grouped split R={R} E={E} {din}x{dout}", flush=True)
    assert R * din * dout >= 1 << 25  # the one-launch path
    g = torch.Generator(device=dev).manual_seed(R + din)
    x = torch.randn(R, din, generator=g, device=dev)
    x *= torch.exp2(torch.randint(-10, 11, (R, 1), generator=g, device=dev).float())
    w = torch.randn(E, din, dout, generator=g, device=dev) * 0.05
    dy = torch.randn(R, dout, generator=g, device=dev) / x.abs().amax(1, keepdim=True)
    y = ops.grouped_linear(x, w, counts)
    gx, gw = ops.grouped_linear_backward(x, w, dy, counts)
    at = 0
    for e, c in enumerate(counts):
        xe, ye, de, we = (t.double() for t in (x[at:at + c], y[at:at + c], dy[at:at + c], w[e]))
        gxe = gx[at:at + c].double()
        at += c
        if c == 0:
            assert (gw[e] == 0).all()
            continue
        assert ((ye - xe @ we).abs() <= _bound(din) * (xe.abs() @ we.abs())).all(), e
        assert ((gxe - de @ we.T).abs() <= _bound(dout) * (de.abs() @ we.abs().T)).all(), e
        mag = xe.abs().T @ de.abs()
        assert ((gw[e].double() - xe.T @ de).abs() <= _bound(c) * mag).all(), e


def test_grouped_weight_gradient_keeps_experts_apart(dev):
    """An expert whose rows are infinite, and one whose rows are 2^40 larger,
    change nothing in the other experts' weight gradients."""
    counts, din, dout = [200, 130, 300, 64, 9, 0, 40, 1], 224, 260
    assert sum(counts) * din * dout >= 1 << 25
    g = torch.Generator(device=dev).manual_seed(7)
    x = torch.randn(sum(counts), din, generator=g, device=dev)
    w = torch.randn(len(counts), din, dout, generator=g, device=dev)
    dy = torch.randn(sum(counts), dout, generator=g, device=dev)
    want = ops.grouped_linear_backward(x, w, dy, counts)[1]
    x[210] = float("inf")
    x[330:630] *= 2.0 ** 40
    got = ops.grouped_linear_backward(x, w, dy, counts)[1]
    assert not torch.isfinite(got[1]).any()
    assert torch.equal(got[2], want[2] * 2.0 ** 40)
    for e in (0, 3, 4, 5, 6, 7):
        assert torch.equal(got[e], want[e]), e


@pytest.mark.parametrize("big", ["x", "dy"])
def test_grouped_gradients_large_rows_without_a_gradient(dev, big):
    """A row of x 2^40 larger whose dy is zero changes nothing in its expert's
    weight gradient, nor a row of dy whose x is zero; weight columns 2^40 larger
    that every dy is zero at change nothing in grad_x."""
    counts, din, dout = [200, 312, 0, 5, 17, 64, 33, 128], 256, 512
    assert sum(counts) * din * dout >= 1 << 25
    print(f"case grouped split large {big}", flush=True)
    g = torch.Generator(device=dev).manual_seed(9)
    x = torch.randn(sum(counts), din, generator=g, device=dev)
    w = torch.randn(len(counts), din, dout, generator=g, device=dev)
    dy = torch.randn(sum(counts), dout, generator=g, device=dev)
    large, zero = (x, dy) if big == "x" else (dy, x)
    large[[9, 250]] *= 2.0 ** 40
    zero[[9, 250]] = 0.0
    w[:, :, 77] *= 2.0 ** 40
    dy[:, 77] = 0.0
    gx, gw = ops.grouped_linear_backward(x, w, dy, counts)
    at = 0
    for e, c in enumerate(counts):
        xe, de, we = x[at:at + c].double(), dy[at:at + c].double(), w[e].double()
        err = (gw[e].double() - xe.T @ de).abs()
        assert (err <= _bound(c) * (xe.abs().T @ de.abs())).all()
        err = (gx[at:at + c].double() - de @ we.T).abs()
        assert (err <= _bound(dout) * (de.abs() @ we.abs().T)).all()
        at += c


def test_grouped_swiglu_mlp_split_matches_small_problem_path(dev):
    """Forward and backward of the MLP on both paths (the plain entry points
    take no workspace): equal to f32 rounding."""
    from summa_amd._lib import call
    counts, d, width = [300, 0, 211, 513, 64, 1, 129, 70], 192, 224
    R, E = sum(counts), len(counts)
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(R, d, generator=g, device=dev)
    wi = torch.randn(E, d, 2 * width, generator=g, device=dev) * 0.05
    wd = torch.randn(E, width, d, generator=g, device=dev) * 0.05
    out, proj, hid = ops.grouped_swiglu_mlp(x, wi, wd, counts, width)
    import numpy as np
    c = np.asarray(counts, dtype=np.int64)
    st = torch.cuda.current_stream().cuda_stream
    out2, proj2, hid2 = (torch.empty_like(t) for t in (out, proj, hid))
    call("sm_grouped_swiglu_mlp", x.data_ptr(), wi.data_ptr(), wd.data_ptr(), c.ctypes.data, E, R,
         d, width, d, out2.data_ptr(), proj2.data_ptr(), hid2.data_ptr(), st)
    for a, b in ((out, out2), (proj, proj2), (hid, hid2)):
        assert float((a - b).norm() / b.norm()) < 2e-6
    dy = torch.randn(R, d, generator=g, device=dev)
    got = ops.grouped_swiglu_mlp_backward(x, wi, wd, counts, proj, hid, dy, width)
    want = [torch.empty_like(t) for t in got]
    scratch = torch.empty(R * 3 * width, device=dev)
    call("sm_grouped_swiglu_mlp_backward", x.data_ptr(), wi.data_ptr(), wd.data_ptr(),
         c.ctypes.data, E, R, d, width, d, proj.data_ptr(), hid.data_ptr(), dy.data_ptr(),
         want[0].data_ptr(), want[1].data_ptr(), want[2].data_ptr(), scratch.data_ptr(), st)
    for a, b in zip(got, want):
        assert float((a - b).norm() / b.norm()) < 2e-6
