"""The dense f32 projection (sm_gemm_f32, summa-llm/src/model/matmul.rs:57-66)
over the tile sizes its dispatch picks from, against float64."""
import numpy as np
import pytest
import torch

from summa_amd._lib import call

pytestmark = pytest.mark.gpu

STORE, ADD = 0, 2


# One output; whole and ragged 8-row tiles; more columns than one k slice and a
# ragged one; the last size of the 8-row tile (4096 tiles) and the first of the
# 16-row one; the last of the 16-row one (16384) and ragged 32-row tiles.
@pytest.mark.parametrize("M,N,K,pad", [(1, 1, 1, 0), (8, 8, 128, 0), (9, 17, 130, 0),
                                       (32, 257, 77, 3), (32, 256, 1024, 4), (128, 2048, 36, 0),
                                       (129, 2048, 66, 2), (512, 2048, 64, 0), (515, 2049, 99, 1)])
@pytest.mark.parametrize("epilogue", [STORE, ADD])
def test_gemm_f32_matches_f64(dev, M, N, K, pad, epilogue):
    print(f"case gemm_f32 M={M} N={N} K={K} pad={pad} epilogue={epilogue}", flush=True)
    rng = np.random.default_rng(M * 7 + N + K)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    w = rng.normal(0, 1, (N, K)).astype(np.float32)
    y0 = rng.normal(0, 1, (M, N)).astype(np.float32)
    xp = torch.full((M, K + pad), float("nan"), device=dev)  # padding is never read
    xp[:, :K] = torch.from_numpy(x).to(dev)
    yp = torch.full((M, N + pad), 7.0, device=dev)
    yp[:, :N] = torch.from_numpy(y0).to(dev)
    wd = torch.from_numpy(w).to(dev)
    call("sm_gemm_f32", wd.data_ptr(), N, K, xp.data_ptr(), M, K + pad, yp.data_ptr(), N + pad,
         epilogue, torch.cuda.current_stream().cuda_stream)
    got = yp.cpu().numpy().astype(np.float64)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    mag = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    if epilogue == ADD:
        want, mag = want + y0, mag + np.abs(y0)
    # K + 1 roundings of at most 2^-24 of the running magnitude
    assert (np.abs(got[:, :N] - want) <= (K + 1) * 2.0 ** -24 * mag).all()
    assert (got[:, N:] == 7.0).all()


# sm_gemm_ex's small products, each transpose pair: ragged tiles of every size
# (one, two and four 8-row blocks a wave), odd leading dimensions, and a long k.
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K,pad", [(1, 1, 1, 0), (13, 9, 131, 1), (64, 64, 128, 0),
                                       (20, 36, 4100, 4), (515, 520, 67, 0), (1030, 1027, 33, 0)])
def test_small_gemm_ex_matches_f64(dev, ta, tb, M, N, K, pad):
    print(f"case small gemm_ex ta={ta} tb={tb} M={M} N={N} K={K} pad={pad}", flush=True)
    rng = np.random.default_rng(M + N + K + 2 * ta + tb)
    a, b = rng.normal(0, 1, (M, K)).astype(np.float32), rng.normal(0, 1, (K, N)).astype(np.float32)
    c0 = rng.normal(0, 1, (M, N)).astype(np.float32)

    def padded(x):
        t = torch.full((x.shape[0], x.shape[1] + pad), float("nan"), device=dev)
        t[:, :x.shape[1]] = torch.from_numpy(np.ascontiguousarray(x)).to(dev)
        return t
    A, B, C = padded(a.T if ta else a), padded(b.T if tb else b), padded(c0)
    call("sm_gemm_ex", ta, tb, M, N, K, 0.5, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0),
         2.0, C.data_ptr(), C.stride(0), torch.cuda.current_stream().cuda_stream)
    got = C[:, :N].cpu().numpy().astype(np.float64)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = 0.5 * (a64 @ b64) + 2.0 * c0
    mag = 0.5 * (np.abs(a64) @ np.abs(b64)) + 2.0 * np.abs(c0)
    assert (np.abs(got - want) <= (K + 3) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("d,heads,kv_heads,hd,ffn,vocab", [(256, 4, 2, 64, 1024, 1000),
                                                           (132, 2, 1, 64, 200, 333)])
def test_fp32_decode_batches_equal_larger_ones(dev, d, heads, kv_heads, hd, ffn, vocab):
    """Few rows run SwiGLU, RoPE and the cache append inside their projections,
    more rows the separate kernels: the log-probs of the same sequences are the
    same bits."""
    from summa_amd.model import Model, ModelConfig
    cfg = ModelConfig(layers=2, d_model=d, heads=heads, kv_heads=kv_heads, head_dim=hd, ffn=ffn,
                      vocab=vocab, max_seq=40, quantized=False)
    m = Model(cfg)
    m.init_random(3, std=0.05)
    gen = torch.Generator().manual_seed(2)
    prompts = torch.randint(0, vocab, (600, 5), generator=gen, dtype=torch.int32).to(dev)
    tokens = torch.randint(0, vocab, (600, 20), generator=gen, dtype=torch.int32).to(dev)
    many = m.logprobs(prompts, tokens)  # 14400 rows: more than 4096 8 x 8 tiles
    few = torch.cat([m.logprobs(prompts[i:i + 1], tokens[i:i + 1]) for i in (0, 1, 599)])
    assert torch.equal(few, many[[0, 1, 599]])
