"""The workgroup map of the prefill attention (csrc/prefill_map.hpp), walked on the
CPU: every (KV head, place) exactly once, and the eight XCDs, to which workgroups go
in turn, evenly loaded however few KV heads there are."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "prefill_map.hpp"
// groups, per -> most and least work of an XCD, times each (group, place) is taken
int main(int argc, char** argv) {
  for (int a = 1; a + 1 < argc; a += 2) {
    const uint32_t groups = atoi(argv[a]), per = atoi(argv[a + 1]);
    const sm::PrefillMap map(groups, per);
    std::vector<int> seen((size_t)groups * per, 0);
    long load[8] = {}, once = 1, whole = 1;
    std::vector<int> home(groups, -1);
    for (long w = 0; w < map.workgroups(); ++w) {
      uint32_t g, p;
      if (!map.at((uint32_t)w, g, p)) continue;
      if (g >= groups || p >= per) return 1;
      seen[(size_t)g * per + p]++;
      load[w % 8]++;
      if (g < groups / 8 * 8) {
        if (home[g] >= 0 && home[g] != w % 8) whole = 0;
        home[g] = (int)(w % 8);
      }
    }
    for (int n : seen) if (n != 1) once = 0;
    long most = 0, least = load[0];
    for (long n : load) { most = n > most ? n : most; least = n < least ? n : least; }
    printf("%ld %ld %ld %ld %lld\n", most, least, once, whole, (long long)map.workgroups());
  }
  return 0;
}
"""

CASES = [(1, 1), (1, 64), (1, 1031), (2, 128), (3, 48), (4, 256), (5, 7), (6, 33), (7, 12),
         (8, 64), (9, 512), (12, 36), (15, 1), (16, 3), (129, 40), (1000, 5)]


@pytest.fixture(scope="module")
def loads(tmp_path_factory):
    d = tmp_path_factory.mktemp("prefill_map")
    src = d / "map.cpp"
    src.write_text(PROGRAM)
    exe = d / "map"
    cxx = shutil.which("g++") or shutil.which("c++")
    subprocess.run([cxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    str(ROOT / "summa_amd" / "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    args = [str(v) for c in CASES for v in c]
    out = subprocess.run([str(exe), *args], check=True, capture_output=True, text=True,
                         timeout=60).stdout.split("\n")
    return {c: tuple(map(int, line.split())) for c, line in zip(CASES, out)}


@pytest.mark.parametrize("groups,per", CASES)
def test_prefill_map_covers_once_and_evenly(loads, groups, per):
    most, least, once, whole, total = loads[(groups, per)]
    assert once, "a (KV head, place) is taken twice or never"
    assert whole, "one of the whole eights of groups is spread over XCDs"
    # the whole eights load every XCD alike, what is left by at most one workgroup
    assert most - least <= 1 and most == -(-groups * per // 8)
    assert groups * per <= total < groups * per + 16


# One and two sequences of few KV heads over many row tiles (dealt over the XCDs),
# an eight with one and with four left over, an odd number of row tiles.
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,KVH,S", [(1, 8, 1, 1300), (1, 8, 2, 1025), (1, 12, 3, 700),
                                       (2, 8, 2, 640), (3, 6, 3, 300), (5, 5, 1, 390),
                                       (6, 4, 2, 260)])
@pytest.mark.parametrize("causal", [True, False])
def test_attention_with_few_kv_heads(dev, B, H, KVH, S, causal):
    import torch

    from summa_amd import ops
    print(f"case attention B={B} H={H} KVH={KVH} S={S} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(B + H + S)
    q, k, v = (torch.randn(B, n, S, 64, generator=g).bfloat16() for n in (H, KVH, KVH))
    out = ops.attention(q.to(dev), k.to(dev), v.to(dev), causal=causal).cpu().double()
    kr, vr = (t.double().repeat_interleave(H // KVH, 1) for t in (k, v))
    sc = torch.matmul(q.double(), kr.transpose(2, 3).contiguous()) / 8.0
    if causal:
        sc = sc.masked_fill(torch.ones(S, S, dtype=torch.bool).triu(1), float("-inf"))
    ref = torch.matmul(torch.softmax(sc, -1), vr)
    # one rounding of the f32-accumulated output to bf16
    assert bool(((out - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4).all())


@pytest.mark.gpu
def test_attention_takes_many_single_rows(dev):
    """2^24 workgroups, more than one grid dimension holds: the largest batch and
    head count, one position each. Its one probability is 1, so the output is V."""
    import torch

    from summa_amd import ops
    B, H = 65535, 256
    print("case attention 65535 x 256 x 1", flush=True)
    g = torch.Generator(device=dev).manual_seed(0)
    q = torch.randn(B, H, 1, 64, generator=g, device=dev, dtype=torch.bfloat16)
    v = torch.randint(-8, 9, (B, 1, 1, 64), generator=g, device=dev).bfloat16() / 4
    out = ops.attention(q, v, v, causal=True)
    assert torch.equal(out, v.expand(B, H, 1, 64))
