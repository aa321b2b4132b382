"""The MoE layer at prefill and recompute sizes (many tokens): the router, the
three-launch route plan and the grouped projections on the
256-row tiles, against the small-batch kernels on slices and numpy."""
import numpy as np
import pytest
import torch

from summa_amd import _lib, ops

pytestmark = pytest.mark.gpu


# 4099: a last workgroup of three tokens; 2, 32 and 64 experts.
@pytest.mark.parametrize("E", [2, 32, 64])
@pytest.mark.parametrize("kind", ["pair", "f16", "f32"])
def test_router_many_tokens_equals_slices(dev, E, kind):
    T, d = 4099, 2048
    print(f"case router rows T={T} E={E} {kind}", flush=True)
    g = torch.Generator(device=dev).manual_seed(E)
    h = torch.randn(T, d, generator=g, device=dev)
    h = ops.f16_pair(h) if kind == "pair" else h.half() if kind == "f16" else h
    r = torch.randn(E, d, generator=g, device=dev) / d ** 0.5
    r[E - 1] = r[0]  # exact ties keep the lower index
    got = ops.moe_top2_indices(h, r, want_logits=True, pair=kind == "pair")
    parts = [ops.moe_top2_indices(h[a:a + 1000].contiguous(), r, want_logits=True,
                                  pair=kind == "pair") for a in range(0, T, 1000)]
    for i in range(3):  # indices, weights, logits: the same bits
        assert torch.equal(got[i], torch.cat([p[i] for p in parts]))
    ref = (ops.unpair(h) if kind == "pair" else h).double() @ r.double().T
    bound = (d + 8) * 2.0 ** -24 * (ops.unpair(h) if kind == "pair" else h).double().abs().sum(1) \
        * float(r.abs().max())
    assert ((got[2].double() - ref).abs().amax(1) <= bound).all()


# Just over one workgroup's routes, a last workgroup of nearly twice its share,
# whole workgroups, more of them than the scan has parts; one expert alone.
@pytest.mark.parametrize("T,k,E,used", [(513, 2, 32, 32), (1023, 2, 64, 64), (2047, 1, 8, 5),
                                        (2048, 2, 32, 32), (70000, 2, 64, 60), (3000, 1, 4, 1)])
def test_route_plan_many_routes(dev, T, k, E, used):
    print(f"case plan T={T} k={k} E={E} used={used}", flush=True)
    rng = np.random.default_rng(T + E)
    idx = rng.choice(E, used, replace=False)[rng.integers(0, used, (T, k))].astype(np.int32)
    R = T * k
    assert R > 1024
    plan = ops.moe_route_plan(torch.from_numpy(idx).to(dev), E)
    flat = idx.ravel()
    order = np.argsort(flat, kind="stable")
    counts = np.bincount(flat, minlength=E)
    inverse = np.empty(R, dtype=np.int64)
    inverse[order] = np.arange(R)
    np.testing.assert_array_equal(plan.counts.cpu().numpy(), counts)
    np.testing.assert_array_equal(plan.offsets.cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
    np.testing.assert_array_equal(plan.order.cpu().numpy(), order)
    np.testing.assert_array_equal(plan.inverse.cpu().numpy(), inverse)
    np.testing.assert_array_equal(plan.src_rows.cpu().numpy(), order // k)
    assert int(plan.error.item()) == 0
    w, at = plan.words.cpu().numpy(), 2 * E + 1 + 3 * R
    for rows in (16, 128):
        tiles = [(e, r) for e in range(E) for r in range(0, counts[e], rows)]
        assert w[at] == len(tiles)
        np.testing.assert_array_equal(w[at + 1:at + 1 + 2 * len(tiles)].reshape(-1, 2), tiles)
        at += 1 + 2 * (-(-R // rows) + E)


def test_route_plan_many_routes_flags_bad_index(dev):
    idx = torch.randint(0, 8, (2000, 2), device=dev, dtype=torch.int32)
    idx[5, 1], idx[1999, 0] = 8, -1
    plan = ops.moe_route_plan(idx, 8)
    assert int(plan.error.item()) == 1
    inv = plan.inverse.cpu().numpy()
    assert inv[11] == -1 and inv[3998] == -1 and (np.delete(inv, [11, 3998]) >= 0).all()
    assert sorted(np.delete(inv, [11, 3998])) == list(range(3998))
    assert int(plan.counts.sum()) == 3998


# Ragged last row tiles and column tiles; an expert without rows and one with a
# single row beside large ones; plain f16 and pairs, gathered rows and not.
@pytest.mark.parametrize("mode", ["pair_swiglu", "pair_store", "f16_swiglu", "f16_store"])
def test_grouped_wide_tiles_equal_dense_projection(dev, mode):
    counts, n, k = [1500, 0, 1, 255, 2043, 257, 2600, 512], 1800, 384
    E, R = len(counts), sum(counts)
    print(f"case grouped wide R={R} n={n} k={k} {mode}", flush=True)
    assert R >= 192 * E and (R // 256 + E // 2) * -(-n // 256) >= 128  # the 256-row tiles
    g = torch.Generator(device=dev).manual_seed(7)
    flat = torch.repeat_interleave(torch.arange(E, device=dev), torch.tensor(counts, device=dev))
    flat = flat[torch.randperm(R, generator=g, device=dev)].int()
    plan = ops.moe_route_plan(flat[:, None].contiguous(), E)
    experts = [ops.Q4Weight.quantize(torch.randn(n, k, generator=g, device=dev) * 0.02)
               for _ in range(E)]
    bank = ops.ExpertBank(experts)
    pair, swiglu = mode.startswith("pair"), mode.endswith("swiglu")
    epi = (_lib.SM_EPI_SWIGLU_F16X2 if pair else _lib.SM_EPI_SWIGLU_F16) if swiglu \
        else _lib.SM_EPI_STORE_F32
    x = torch.randn(R, k, generator=g, device=dev)
    x = ops.f16_pair(x) if pair else x.half()
    got = ops.grouped_q4_matmul(bank, x, plan, gather=swiglu, epilogue=epi, pair=pair)
    rows = x[plan.src_rows.long()] if swiglu else x
    at = 0
    for e, c in enumerate(counts):
        if c >= 256:  # the dense batch kernels accumulate in the same order
            want = ops.q4_matmul(experts[e], rows[at:at + c].contiguous(), epilogue=epi, pair=pair)
            assert torch.equal(got[at:at + c], want), e
        elif c:
            want = ops.q4_matmul(experts[e], rows[at:at + c].contiguous(), epilogue=epi, pair=pair)
            torch.testing.assert_close(got[at:at + c].float(), want.float(), rtol=2e-3, atol=2e-4)
        at += c
