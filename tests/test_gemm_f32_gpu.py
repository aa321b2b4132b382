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
