"""The linear head + cross-entropy on split operands (three exact bf16 planes on
the matrix cores), at the sizes its tiles and K splits meet edges, against float64."""
import pytest
import torch
import torch.nn.functional as F

from summa_amd import _lib, ops
from summa_amd._lib import call

pytestmark = pytest.mark.gpu


def _bound(K):
    """Relative to sum |a||b|: the plane products left out (below 3 x 2^-24) and
    half of the 6 K / 16 f32 additions, whose errors have either sign."""
    return 2.0 ** -21 + 2.0 ** -22 + (3 * K / 16 + 2) * 2.0 ** -24


# Ragged in every direction at the smallest matrix-core size; a K of 8200 split
# over the chip and a last chunk of 76 rows; few rows against a long vocabulary.
@pytest.mark.parametrize("T,d,V,logical,chunk", [(257, 522, 1031, 1031, 1024),
                                                 (1100, 768, 8200, 8123, 1024),
                                                 (300, 96, 50304, 50304, 150)])
@pytest.mark.parametrize("bias", [True, False])
def test_split_linear_ce_matches_f64(dev, T, d, V, logical, chunk, bias):
    print(f"case split linear ce T={T} d={d} V={V} chunk={chunk} bias={bias}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + d + V)
    h = torch.randn(T, d, generator=g, device=dev)
    h *= torch.exp2(torch.randint(-12, 13, (T, 1), generator=g, device=dev).float())  # row scales
    w = torch.randn(V, d, generator=g, device=dev) * 0.02 / h.abs().amax()
    b = torch.randn(V, generator=g, device=dev) * 0.1 if bias else None
    t = torch.randint(0, logical, (T,), generator=g, device=dev, dtype=torch.int32)
    go = torch.full((1,), 3.0, device=dev)
    loss = ops.linear_cross_entropy(h, w, b, t, logical, chunk)
    gh, gw, gb = ops.linear_cross_entropy_backward(h, w, b, t, go, logical, chunk)
    h64, w64 = h.double().requires_grad_(True), w.double().requires_grad_(True)
    b64 = b.double().requires_grad_(True) if bias else None
    logits = F.linear(h64, w64, b64)[:, :logical]
    ref = F.cross_entropy(logits, t.long())
    (3.0 * ref).backward()
    # the error of a logit, and so the relative error of a probability (doubled)
    el = _bound(d) * float((h.double().abs() @ w.double().abs().T).amax()) + 1e-6
    G = (torch.softmax(logits, 1).detach() * 3.0 / T)
    G = G + F.one_hot(t.long(), logical) * 3.0 / T
    assert abs(float(loss) - float(ref.detach())) <= 2 * el
    for name, got, want, mag, K in (
            ("hidden", gh, h64.grad, G @ w64[:logical].abs(), V),
            ("weight", gw[:logical], w64.grad[:logical], G.T @ h64.abs(), T)):
        err = (got.double() - want).abs()
        assert (err <= (_bound(K) + 2 * el + 2e-6) * mag).all(), (name, float((err / mag).max()))
    assert (gw[logical:] == 0).all()
    if bias:
        assert (gb.double() - b64.grad).abs().max() <= (T * 2.0 ** -24 + 2 * el + 2e-6) * G.sum(0).max()
        assert (gb[logical:] == 0).all()


def test_small_workspace_keeps_the_unsplit_path(dev):
    """A workspace with room for the chunk's buffers alone is accepted, and the
    two paths agree: the same plane products in the same order, split once per
    call or in the K loop. The loss alone needs no more than its own query's bytes:
    the chunk's buffers, and W and hidden in split form where they are read so."""
    T, d, V, chunk = 1536, 512, 2048, 512
    g = torch.Generator(device=dev).manual_seed(3)
    h = torch.randn(T, d, generator=g, device=dev)
    w = torch.randn(V, d, generator=g, device=dev) * 0.05
    b = torch.randn(V, generator=g, device=dev) * 0.1
    t = torch.randint(0, V, (T,), generator=g, device=dev, dtype=torch.int32)
    st = torch.cuda.current_stream().cuda_stream
    full = int(_lib.lib().sm_linear_cross_entropy_workspace_bytes(T, d, V, chunk, 1))
    loss_only = int(_lib.lib().sm_linear_cross_entropy_forward_workspace_bytes(T, d, V, chunk, 1))
    # logits, log-probs, row scales, bias-gradient parts: each 256-byte aligned
    least = chunk * V * 4 + T * 4 + chunk * 4 + 64 * V * 4
    assert loss_only == least + 6 * d * (V + T) and full > loss_only
    ws = torch.empty(full + 256, dtype=torch.uint8, device=dev)
    base = (ws.data_ptr() + 255) // 256 * 256
    out = []
    for nbytes in (least, loss_only, full):
        loss, lp = torch.empty(1, device=dev), torch.empty(T, device=dev)
        call("sm_linear_cross_entropy", h.data_ptr(), w.data_ptr(), b.data_ptr(), t.data_ptr(), T,
             d, V, V, chunk, 1, loss.data_ptr(), lp.data_ptr(), base, nbytes, st)
        out.append(lp)
    assert torch.equal(out[0], out[1]) and torch.equal(out[1], out[2])


def test_split_linear_ce_infinity_and_zero_rows(dev):
    """An infinity spoils its own token only; a zero row is exact."""
    T, d, V = 1024, 512, 2048
    g = torch.Generator(device=dev).manual_seed(4)
    h = torch.randn(T, d, generator=g, device=dev)
    w = torch.randn(V, d, generator=g, device=dev) * 0.05
    b = torch.zeros(V, device=dev)
    t = torch.randint(0, V, (T,), generator=g, device=dev, dtype=torch.int32)
    _, clean = ops.linear_cross_entropy(h, w, b, t, want_logprob=True)
    h[7, 3], h[9] = float("inf"), 0.0
    _, lp = ops.linear_cross_entropy(h, w, b, t, want_logprob=True)
    assert not torch.isfinite(lp[7])
    assert abs(float(lp[9]) + torch.log(torch.tensor(float(V)))) < 1e-5
    keep = torch.ones(T, dtype=torch.bool, device=dev)
    keep[[7, 9]] = False
    assert torch.equal(lp[keep], clean[keep])


def _f64_grads(h, w, t, logical):
    logits = (h.double() @ w.double().T)[:, :logical]
    G = torch.softmax(logits, 1)
    G[torch.arange(len(t), device=h.device), t.long()] -= 1
    G /= len(t)
    return G, G @ w[:logical].double(), G.T @ h.double()


@pytest.mark.parametrize("case", ["padded rows", "saturated token", "unlikely row"])
def test_split_linear_ce_large_values_without_a_gradient(dev, case):
    """Finite values whose factor in a sum is exactly zero change nothing, however
    large: vocabulary rows past the logical size, the hidden row of a token whose
    softmax is saturated on its target, a vocabulary row that no token gives any
    probability. Against float64, as far as f32 sums of the other terms are off."""
    T, d, V, logical = 300, 512, 4096, 4000
    print(f"case split linear ce {case}", flush=True)
    g = torch.Generator(device=dev).manual_seed(11)
    h = torch.randn(T, d, generator=g, device=dev)
    w = torch.randn(V, d, generator=g, device=dev) * 0.02
    t = torch.randint(0, logical - 1, (T,), generator=g, device=dev, dtype=torch.int32)
    big = 2.0 ** 40
    if case == "padded rows":
        w[logical:] *= big
    elif case == "saturated token":
        w[:, :2], w[t[7].long(), 1] = 0.0, 1.0
        h[7], h[7, 0], h[7, 1] = 0.0, big, 256.0  # its logit 256, the others 0
    else:  # every token's logit of row logical - 1 is about -2^39
        h[:, 0] = h[:, 0].abs() + 0.5
        w[logical - 1] = 0.0
        w[logical - 1, 0] = -big
    G, want_h, want_w = _f64_grads(h, w, t, logical)
    quiet = G.abs() > 0  # the terms with a gradient
    gh, gw, _ = ops.linear_cross_entropy_backward(h, w, None, t, torch.ones(1, device=dev), logical)
    # G's own error: that of a logit, doubled (the saturated and unlikely ones are exact)
    live = torch.where((h.abs().amax(1) < big / 2 ** 20)[:, None], h.double(), 0.0).abs()
    rows = torch.where((w[:logical].abs().amax(1) < big / 2 ** 20)[:, None],
                       w[:logical].double(), 0.0).abs()
    el = 2 * _bound(d) * float((live @ rows.T).amax()) + 2e-6
    A = G.abs() + torch.nn.functional.one_hot(t.long(), logical) * quiet / T
    for name, got, want, mag, K in (("hidden", gh, want_h, A @ w[:logical].double().abs(), V),
                                    ("weight", gw[:logical], want_w, A.T @ h.double().abs(), T)):
        err = (got.double() - want).abs()
        assert (err <= (_bound(K) + el) * mag).all(), (name, float((err / (mag + 1e-300)).max()))
