"""The launch rules of csrc/rules.h, compiled with the host compiler and checked on the CPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "minicpm5-vllm-tpu_amd", "csrc")

SRC = r"""
#include "rules.h"
extern "C" void fit(const size_t* in, size_t* out, int spare, int hd, int S) {
  mk::PrefetchRanges pf{};
  for (int r = 0; r < 4; ++r) pf.p[r] = in[r] ? in : nullptr, pf.bytes[r] = in[r];
  const mk::PrefetchRanges f = mk::prefetch_fit(pf, spare, hd, S);
  for (int r = 0; r < 4; ++r) out[r] = f.bytes[r] && !f.p[r] ? ~(size_t)0 : f.bytes[r];
}
extern "C" int gemm_tile(int silu, int in, int M, int N, int kb) {
  return mk::gemm_tile(silu, (mk::GemmIn)in, M, N, kb);
}
extern "C" int gemm_tile_built(int id, int silu, int in) { return mk::gemm_tile_built(id, silu, (mk::GemmIn)in); }
extern "C" int attn_waves(int items8, int ncu, int hd, int B, int prefetch) {
  return mk::attn_waves(items8, ncu, hd, B, prefetch);
}
extern "C" int lm_head_skinny(int rows, int V, int K) { return mk::lm_head_skinny(rows, V, K); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SRC)
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "rules.cpp"), "-o",
                    str(d / "rules.so")], check=True)
    return ctypes.CDLL(str(d / "rules.so"))


# bytes of a layer's gate/up, O, next QKV and down weights (W8A8 gate/up and QKV, bf16 O and down)
WEIGHTS = {"1b": (14155776, 6291456, 3932160, 14155776), "2b": (25165824, 8388608, 5242880, 25165824)}


def _fit(rules, ranges, spare, hd, S):
    a, out = (ctypes.c_size_t * 4)(*ranges), (ctypes.c_size_t * 4)()
    rules.fit(a, out, spare, hd, S)
    return tuple(out)


@pytest.mark.parametrize("arch", ["1b", "2b"])
@pytest.mark.parametrize("hd", [96, 128])
def test_prefetch_within_the_launch(rules, arch, hd):
    """Whole ranges only, and never more than the spare workgroups read (at most 75 KB/us each) while the launch
    runs (8 us and 1.25 us per key tile at hd 128): 8 spare workgroups beside 31 sequences of 128 tokens took
    111 us for the 2B layer's 64 MB."""
    w = WEIGHTS[arch]
    for spare in (0, 1, 8, 16, 40, 64, 96, 128, 240):
        for S in (64, 128, 1024, 1920, 3968):
            got = _fit(rules, w, spare, hd, S)
            assert all(g in (0, b) for g, b in zip(got, w))
            assert sum(got) <= spare * 75 * 1024 * (8 + 1.25 * hd / 128 * (S // 64))


def test_prefetch_takes_what_fits(rules):
    w1, w2 = WEIGHTS["1b"], WEIGHTS["2b"]
    assert _fit(rules, w2, 8, 128, 128) == (0, 0, 5242880, 0)
    assert _fit(rules, w2, 128, 128, 128) == w2 and _fit(rules, w1, 240, 128, 128) == w1
    assert _fit(rules, w2, 16, 128, 1920) == w2[:3] + (0,)
    assert _fit(rules, (0, 0, 0, 0), 8, 128, 128) == (0, 0, 0, 0)


@pytest.mark.parametrize("rows,V,K,skinny", [
    (1, 1000, 256, True), (1, 8192, 1536, True), (2, 1000, 4096, True), (8, 8192, 1536, True), (8, 8192, 256, True),
    (12, 4096, 1536, True), (16, 1000, 4096, True), (1, 16384, 1536, True),
    (17, 1000, 4096, False), (16, 8192, 1536, False), (33, 1000, 1536, False), (1, 20480, 1536, False),
    (2, 20480, 2048, False), (1, 130560, 1536, False), (1, 130560, 2048, True), (2, 130560, 2048, True),
    (2, 65536, 2048, False), (3, 130560, 2048, False), (40, 130560, 1536, False)])
def test_lm_head_kernel_choice(rules, rows, V, K, skinny):
    """Few rows over a vocabulary whose 64-column workgroups run in one round, and one or two rows over long rows,
    take the skinny kernel (measured faster there), the rest the batch kernel."""
    assert bool(rules.lm_head_skinny(rows, V, K)) == skinny


@pytest.mark.parametrize("B,S,hd,prefetch,waves", [
    (1, 2048, 64, False, 4), (16, 128, 96, True, 4), (1, 3136, 128, False, 4), (1, 3456, 128, False, 4),
    (1, 3840, 128, False, 4), (2, 1088, 128, False, 4), (2, 1472, 128, False, 4), (1, 3072, 128, True, 4),
    (1, 3904, 128, False, 8), (1, 3136, 128, True, 8), (1, 3840, 128, True, 8), (2, 1536, 128, False, 8),
    (2, 1088, 128, True, 8), (1, 2112, 96, False, 8), (2, 1088, 64, False, 8), (3, 704, 128, False, 8),
    (4, 768, 128, False, 8), (1, 4096, 128, False, 8), (1, 8192, 128, True, 8)])
def test_attention_waves(rules, B, S, hd, prefetch, waves):
    """Waves per attention workgroup on 256 CUs (2 kv heads, 32-token q tiles)."""
    assert rules.attn_waves(B * 2 * (S // 32), 256, hd, B, int(prefetch)) == waves


I8, BF16, F8 = 0, 1, 2      # GemmIn


def test_gemm_tile_is_built(rules):
    """The dispatch rule picks a tile that is built for the operands and epilogue, and one of whole-line stages only
    for K of whole lines, over sizes from one row to 70000."""
    sizes = [1, 2, 31, 33, 63, 64, 65, 127, 129, 256, 257, 511, 700, 1000, 1537, 2048, 3000, 4097, 6000, 8192, 10923,
             16384, 30000, 70000]
    for silu in (0, 1):
        for in_type in (I8, BF16, F8):
            for M in sizes:
                for N in (64, 128, 512, 1536, 1920, 2048, 2560, 4096, 9216, 12288, 40000):
                    for kb in (64, 128, 192, 448, 960, 1024, 1088, 1536, 2048, 4096, 4160, 9216, 12288):
                        t = rules.gemm_tile(silu, in_type, M, N, kb)
                        assert rules.gemm_tile_built(t, silu, in_type), (silu, in_type, M, N, kb, t)
                        assert kb % 128 == 0 or not (t == 6 or t >= 9), (silu, in_type, M, N, kb, t)


def test_gate_up_tile_of_two_rows(rules):
    """int8 gate/up of 385 .. 512 rows: two rows of 256x128 tiles, not three of 192x128, one workgroup per CU."""
    assert [rules.gemm_tile(1, I8, m, 9216, 1536) for m in (384, 385, 400, 512, 513)] == [3, 2, 2, 2, 12]
    assert rules.gemm_tile(1, I8, 3072, 1536, 256) == 12


def test_gemm_tile_of_tested_shapes(rules):
    """The GPU tests reach the tiles that they name."""
    from test_gpu_kernels import SILU_SHAPES, TILE_SHAPES

    for t, M, N, kb in TILE_SHAPES:
        assert [rules.gemm_tile(0, i, M, N, kb) for i in (I8, BF16, F8)] == [t] * 3, (t, M, N, kb)
    for t, M, N, kb in SILU_SHAPES:
        assert [rules.gemm_tile(1, i, M, N, kb) for i in (BF16, F8)] == [t] * 2, (t, M, N, kb)
    assert {t for t, *_ in TILE_SHAPES} == {2, 3, 6, 7, 9, 10, 11, 13} and {t for t, *_ in SILU_SHAPES} == {3, 4, 7, 12}
    # ping-pong stages and the routed QKV projection of the model tests (N = 1280 and 1920)
    for N, t in ((1536, 5), (2048, 4), (2560, 8)):
        for kb in (64, 128, 192, 384, 448, 1600, 4160):
            assert [rules.gemm_tile(0, i, 8100, N, kb) for i in (I8, BF16)] == [t] * 2, (N, kb)
    assert rules.gemm_tile(0, F8, 8100, 2560, 192) == 5
    assert rules.gemm_tile(0, I8, 8192, 1920, 1536) == 4 and rules.gemm_tile(0, I8, 8192, 2560, 1536) == 8
    assert [rules.gemm_tile(0, BF16, 1000, 1536, 2 * k) for k in (4608, 2080, 544)] == [11, 7, 7]
    assert [rules.gemm_tile(0, BF16, 4096, 1536, 2 * k) for k in (4608, 2080, 544)] == [13, 2, 2]
    assert rules.gemm_tile(0, I8, 4096, 1280, 256) == 13 and rules.gemm_tile(0, BF16, 4096, 1280, 512) == 13
    assert rules.gemm_tile(0, F8, 2304, 1920, 384) == 13
