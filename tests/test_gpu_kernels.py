"""Per-kernel parity of libmk's HIP kernels against the oracle (GPU; calls go through the C ABI).

  * attention (super_gqa_v2 numerics): vs the FP32 reference attention.  Tolerance: max |err| <= 0.02,
    mean |err| <= 5e-4 -- about 2x the error of the oracle's own bf16-rounding emulation of the same
    kernel (0.0093 / 2.3e-4 at S = 1024..4096, hd 96), and below the TPU reference's own rounding
    (0.013 / 3.0e-4 with its bf16 exp2 and bf16 RoPE products).  At S <= 1024 also vs the restatement of
    the reference's short-sequence kernel (attention_small): max <= 0.03, mean <= 1e-3.
  * row quantisation: bit-exact int8 and f32 scales (same f32 operations).
  * int8 GEMM: bit-exact int32 accumulators (exact integer arithmetic), dequant epilogues within
    1 bf16 ulp of the oracle (f32 products identical up to the row scale's last bit).
  * bf16 GEMM: f32 accumulation in a different order than the CPU: relative error <= 1e-2 of the
    output scale, bf16 rounding of the result dominating.
  * activation quantisation in the fp8d / int8 / fp8 modes: bit-exact codes (the static modes with
    RMSNorm round x * rstd to bf16, so an rstd one f32 ulp off may move a code by one step: at most
    0.1% of codes, each by one step); f32 -> e4m3 conversion bit-exact over every finite bf16 value.
  * fp8 GEMM: the fp8 MFMAs sum their products at reduced internal precision.  Measured on MI355X with
    v_mfma_f32_32x32x64_f8f6f4 (the K = 16 instructions give the same): max error 6.2e-5 of sum|products| at
    K = 64, 1.2e-5 at K = 448, 2.2e-6 at K = 4608, 1.5e-5 in 2-norm at every K.  So the bound is
    1e-4 * sum|products| of the exact (float64) result; dequant epilogues within 1 bf16 ulp + that bound.
"""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _dev():
    assert torch.cuda.is_available(), "GPU test needs a visible MI355X"
    return torch.device("cuda:0")


def _attn_inputs(B, S, hd, n_q=16, n_kv=2):
    gens = [torch.Generator().manual_seed(i) for i in range(3)]
    q = torch.randn(B, S, n_q * hd, generator=gens[0])
    k = torch.randn(B, S, n_kv * hd, generator=gens[1])
    v = torch.randn(B, S, n_kv * hd, generator=gens[2])
    return torch.cat([q, k, v], -1).to(BF16)


@pytest.mark.parametrize("B,S,hd,theta", [(1, 256, 64, 1e4), (2, 512, 96, 1e4), (1, 1024, 128, 5e6),
                                           (3, 128, 128, 5e6), (2, 384, 96, 1e4), (1, 640, 128, 5e6),
                                           (1, 8192, 96, 1e4), (1, 8192, 128, 5e6), (3, 2048, 128, 5e6),
                                           (1, 3136, 128, 5e6)])
def test_attention_vs_fp32(B, S, hd, theta):
    from minicpm5_mk import ops
    from minicpm5_mk.mk_weights import rope_tables
    from oracle import emulate

    dev = _dev()
    print(f"[attn] B={B} S={S} hd={hd}", flush=True)
    qkv = _attn_inputs(B, S, hd)
    cos, sin = rope_tables(S, hd, theta)
    sm = 1.0 / math.sqrt(hd)
    out = ops.attn_prefill(qkv.to(dev), cos.to(dev), sin.to(dev), 16, 2, hd, sm_scale=sm)
    torch.cuda.synchronize()
    out = out.float().cpu()
    ref = emulate.attention_fp32(qkv, cos, sin, 16, 2, hd, sm)
    err = (out - ref).abs()
    print(f"[attn] max {err.max():.4g} mean {err.mean():.4g}", flush=True)
    assert torch.isfinite(out).all()
    assert err.max() <= 0.02 and err.mean() <= 5e-4, (float(err.max()), float(err.mean()))



@pytest.mark.parametrize("B,S,hd", [(1, 128, 128), (2, 512, 96), (1, 1024, 128)])
def test_attention_vs_reference_short_kernel(B, S, hd):
    """At S <= 1024 the reference runs another kernel (attn_fused_small, mk_jax.py:58-175: exact row max,
    f32 exp and sum, P normalised to bf16 before the PV product); this build runs the long-sequence
    algorithm at every length.  The two agree to the bf16 rounding of their P and RoPE products: on the
    CPU the restatements differ by max 0.016 / mean 6e-4 (S = 128..1024), each within 0.013 of FP32.
    Tolerance: max |err| <= 0.03, mean |err| <= 1e-3 against the reference kernel's restatement."""
    from minicpm5_mk import ops
    from minicpm5_mk.mk_weights import rope_tables
    from oracle import emulate

    dev = _dev()
    print(f"[attn-short] B={B} S={S} hd={hd}", flush=True)
    qkv = _attn_inputs(B, S, hd)
    cos, sin = rope_tables(S, hd, 5e6)
    sm = 1.0 / math.sqrt(hd)
    out = ops.attn_prefill(qkv.to(dev), cos.to(dev), sin.to(dev), 16, 2, hd, sm_scale=sm)
    torch.cuda.synchronize()
    ref = emulate.attention_small(qkv, cos, sin, 16, 2, hd, sm).float()
    err = (out.float().cpu() - ref).abs()
    print(f"[attn-short] max {err.max():.4g} mean {err.mean():.4g}", flush=True)
    assert err.max() <= 0.03 and err.mean() <= 1e-3, (float(err.max()), float(err.mean()))

def test_attention_deterministic():
    from minicpm5_mk import ops
    from minicpm5_mk.mk_weights import rope_tables

    dev = _dev()
    qkv = _attn_inputs(1, 2048, 128).to(dev)
    cos, sin = (t.to(dev) for t in rope_tables(2048, 128, 5e6))
    a = ops.attn_prefill(qkv, cos, sin, 16, 2, 128)
    b = ops.attn_prefill(qkv, cos, sin, 16, 2, 128)
    assert torch.equal(a, b)


@pytest.mark.parametrize("B,S,hd", [(2, 4096, 128), (4, 2048, 96), (3, 2048, 128), (4, 768, 96), (4, 768, 64),
                                    (2, 2560, 128), (2, 3392, 128), (2, 1216, 128)])
def test_attention_batch_invariant(B, S, hd):
    """Each sequence of a batch equals the same sequence run alone, bit for bit.  (2, 4096) and
    (4, 2048) launch 256 tile pairs (B * 2 kv heads * S / 64) and take the static pair mapping;
    (3, 2048) launches 384 items on 256 persistent workgroups, so workgroups take several items and
    drain the other kv head's queue; the single-sequence runs have no more items than CUs and take the
    direct mapping (workgroup i computes item i, no queue).  (4, 768) launches 192 items of 8 waves, its
    single sequences items of 4 waves.  The single sequences of (2, 2560) and (2, 3392), and the batch
    (2, 1216), launch more 4-wave items than there are CUs and take them from the queues."""
    from minicpm5_mk import ops
    from minicpm5_mk.mk_weights import rope_tables

    dev = _dev()
    print(f"[attn-batch] B={B} S={S} hd={hd}", flush=True)
    qkv = _attn_inputs(B, S, hd).to(dev)
    cos, sin = (t.to(dev) for t in rope_tables(S, hd, 5e6))
    full = ops.attn_prefill(qkv, cos, sin, 16, 2, hd)
    for b in range(B):
        one = ops.attn_prefill(qkv[b:b + 1].contiguous(), cos, sin, 16, 2, hd)
        assert torch.equal(full[b:b + 1], one), b


@pytest.mark.parametrize("T,H,norm,recip,f32", [(300, 1536, True, True, False), (64, 2048, False, False, False),
                                                (129, 4608, False, True, True), (8192, 1536, True, True, False),
                                                (77, 256, True, True, False), (5, 1280, True, False, True)])
def test_row_quant_bitexact(T, H, norm, recip, f32):
    from minicpm5_mk import ops
    from oracle import emulate

    dev = _dev()
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g) * 3
    x[0, :7] = 0.0
    x = x if f32 else x.to(BF16)
    a = torch.rand(H, generator=g) + 0.5
    q, sx = ops.row_quant(x.to(dev), a.to(dev), 1e-6, norm, recip)
    qr, sxr = emulate.row_quant(x.float(), a, 1e-6, norm, recip)
    assert torch.equal(q.cpu(), qr)
    if norm:   # rstd: different summation order of mean(x^2) -> a few f32 ulps
        torch.testing.assert_close(sx.cpu(), sxr, rtol=4e-7, atol=0)
    else:
        assert torch.equal(sx.cpu(), sxr)


def _rowquant_tree_sx(x: np.ndarray, a: np.ndarray, eps: float) -> np.ndarray:
    """The fused prologue's per-token scale sx = max(amax(x a) / 127, 1e-6) * rsqrt(mean(x^2) + eps) with the
    sum of squares added in the kernel's order: lane L (of 64) sums chunks L + 64 i (8 elements each) with
    FMAs, then the DPP tree (partners L^1, L^2, the 8-lane mirror, the 16-lane mirror) and
    (L0 + L16) + (L32 + L48).  Float32 throughout; a bf16 square is exact in float64, so
    f32(f64(v)^2 + f64(s)) is the FMA."""
    f32 = np.float32
    T, H = x.shape
    nc = H // 8
    out = np.empty(T, dtype=f32)
    for t in range(T):
        lanes = np.zeros(64, dtype=f32)
        for L in range(64):
            s = f32(0.0)
            for c in range(L, nc, 64):
                for e in range(8):
                    v = np.float64(x[t, 8 * c + e])
                    s = f32(v * v + np.float64(s))
            lanes[L] = s
        for part in (lambda l: l ^ 1, lambda l: l ^ 2, lambda l: (l & ~7) | (7 - (l & 7)),
                     lambda l: (l & ~15) | (15 - (l & 15))):
            lanes = np.array([f32(lanes[l] + lanes[part(l)]) for l in range(64)], dtype=f32)
        ss = f32(f32(lanes[0] + lanes[16]) + f32(lanes[32] + lanes[48]))
        rstd = f32(1.0) / np.sqrt(f32(ss / f32(H)) + f32(eps), dtype=f32)
        am = np.max(np.abs(x[t].astype(f32) * a.astype(f32)))
        out[t] = f32(max(f32(am * f32(1.0 / 127.0)), f32(1e-6)) * rstd)
    return out


@pytest.mark.parametrize("T,H", [(9, 1536), (7, 2048), (3, 1280)])
def test_row_quant_scale_tree_bitexact(T, H):
    """sx bit for bit against a restatement of the kernel's summation order (per-lane FMAs over chunks
    L + 64 i, then the DPP tree), rows with 2, 3 and 4 chunks per lane (the last one partly past the row)."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(T * H)
    x = (torch.randn(T, H, generator=g) * 3).to(BF16)
    a = torch.rand(H, generator=g) + 0.5
    _, sx = ops.row_quant(x.to(dev), a.to(dev), 1e-6, True, True)
    ref = _rowquant_tree_sx(x.float().numpy(), a.numpy(), 1e-6)
    assert np.array_equal(sx.cpu().numpy().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("M,N,K", [(256, 128, 64), (300, 200, 1536), (8192, 1920, 1536), (8192, 2560, 1536),
                                   (1000, 1536, 4608), (1000, 1536, 1088)])
def test_gemm_int8_exact(M, N, K):
    """Exact int32 products; (8192, 1920) and (8192, 2560) are the QKV projections at hd 96 and 128, on the
    256x256 and on the 256x320 tile, whose epilogue stages its 64x160 wave tiles in two column chunks."""
    from minicpm5_mk import ops
    from oracle import emulate

    dev = _dev()
    g = torch.Generator().manual_seed(M * 7 + N)
    a = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    b = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    acc = ops.gemm(a.to(dev), b.to(dev), "i32").cpu()
    ref = emulate.int_matmul(a, b.t().contiguous())
    assert torch.equal(acc.to(torch.int64), ref)


def test_gemm_int8_skinny_exact():
    from minicpm5_mk import ops
    from oracle import emulate

    dev = _dev()
    g = torch.Generator().manual_seed(5)
    for M in (1, 7, 32):
        a = torch.randint(-127, 128, (M, 2048), generator=g, dtype=torch.int8)
        b = torch.randint(-127, 128, (4096 + 96, 2048), generator=g, dtype=torch.int8)
        acc = ops.gemm(a.to(dev), b.to(dev), "i32").cpu()
        assert torch.equal(acc.to(torch.int64), emulate.int_matmul(a, b.t().contiguous()))


def test_fused_qkv_epilogue():
    """fused_qkv (mk_mlp.py:161-170) through row_quant + int8 GEMM with the DQ epilogue."""
    from minicpm5_mk import ops
    from oracle import emulate

    dev = _dev()
    g = torch.Generator().manual_seed(11)
    T, H, D = 1024, 1536, 2560
    x = torch.randn(T, H, generator=g).to(BF16)
    w = torch.randint(-127, 128, (H, D), generator=g, dtype=torch.int8)
    s_w = torch.rand(D, generator=g) * 1e-3
    a = torch.rand(H, generator=g) + 0.5
    q, sx = ops.row_quant(x.to(dev), a.to(dev), 1e-6, True, True)
    out = ops.gemm(q, w.t().contiguous().to(dev), "dq_bf16", rs=sx, cs=s_w.to(dev)).float().cpu()
    ref = emulate.fused_qkv(x, w, s_w, a, 1e-6).float()
    ulp = ref.abs().clamp(min=1e-30) * 2.0 ** -7
    assert ((out - ref).abs() <= ulp).all()


@pytest.mark.parametrize("M,N,K", [(512, 1536, 2048), (8192, 1536, 4608), (100, 512, 1536)])
def test_gemm_bf16(M, N, K):
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(M + K)
    a = torch.randn(M, K, generator=g).to(BF16)
    b = (torch.randn(N, K, generator=g) * 0.02).to(BF16)
    out = ops.gemm(a.to(dev), b.to(dev), "f32").cpu()
    ref = a.float() @ b.float().t()
    torch.testing.assert_close(out, ref, rtol=1e-4, atol=1e-4 * ref.abs().max().item())
    outb = ops.gemm(a.to(dev), b.to(dev), "bf16").float().cpu()
    assert ((outb - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-3 * ref.abs().max()).all()


@pytest.mark.parametrize("N,K", [(1536, 4608), (1536, 2080), (1536, 544)])
def test_gemm_bf16_rows_independent_of_tile(N, K):
    """The first 1000 rows of a 4096-row product alone, on a 64x128 tile (loader waves at K = 4608, the two-stage
    loop with an odd stage count at K = 2080 and at K = 544, 17 stages, the fewest it is chosen for), and on
    128x128 pairs or 256x128 tiles inside the big product: identical f32 bits."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(K)
    a = torch.randn(4096, K, generator=g).to(BF16).to(dev)
    b = (torch.randn(N, K, generator=g) * 0.02).to(BF16).to(dev)
    big = ops.gemm(a, b, "f32")
    small = ops.gemm(a[:1000].contiguous(), b, "f32")
    assert torch.equal(small.view(torch.int32), big[:1000].view(torch.int32))


@pytest.mark.parametrize("M,N,K", [(33, 72, 64), (40, 1536, 192), (250, 1504, 4608), (321, 1528, 128), (500, 1504, 320),
                                   (1000, 1512, 2112), (600, 1512, 2048), (2000, 1512, 2112), (1100, 1512, 2048)])
def test_gemm_short_problem_tiles(M, N, K):
    """Whole-line tiles of short problems (32x64, 64x64, 64x128, 128x128: K loops of one stage, fewer stages
    than ring slots, an odd and an even count; ragged rows and columns): bf16 rows bitwise equal to the same rows of a
    product of 9000 rows on a wide tile and within 64 eps sum|products| of float64; int8 exact."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(M + N + K)
    print(f"[short tiles] {M}x{N}x{K}", flush=True)
    a = torch.randn(9000, K, generator=g).to(BF16).to(dev)
    b = (torch.randn(N, K, generator=g) * 0.02).to(BF16).to(dev)
    out, big = ops.gemm(a[:M].contiguous(), b, "f32"), ops.gemm(a, b, "f32")
    assert torch.equal(out.view(torch.int32), big[:M].view(torch.int32))
    ref = a[:M].double() @ b.double().t()
    assert ((out.double() - ref).abs() <= 64 * 2.0 ** -24 * (a[:M].double().abs() @ b.double().abs().t())).all()
    x = torch.randn(M, N, generator=g).to(BF16).to(dev)
    res = ops.gemm(a[:M].contiguous(), b, "res_f32add", res=x.clone())
    assert torch.equal(res.view(torch.int16), (x.float() + out).to(BF16).view(torch.int16))
    ai = torch.randint(-127, 128, (M, 2 * K), generator=g, dtype=torch.int8).to(dev)
    bi = torch.randint(-127, 128, (N, 2 * K), generator=g, dtype=torch.int8).to(dev)
    assert torch.equal(ops.gemm(ai, bi, "i32").double(), ai.double() @ bi.double().t())


@pytest.mark.parametrize("M,N,K", [(2900, 1528, 64), (4000, 1536, 128), (2300, 2008, 1536), (2300, 2008, 192)])
def test_gemm_mid_size_tiles(M, N, K):
    """128x128 workgroup pairs (257 .. 512 tiles; K loops of one, two, three and many stages, ragged rows and
    columns): bf16 rows bitwise equal to those of a product of 9000 rows and within 64 eps sum|products| of
    float64, int8 exact, fp8 within 1e-4 sum|products|."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(M + K)
    print(f"[mid tiles] {M}x{N}x{K}", flush=True)
    a = torch.randn(9000, K, generator=g).to(BF16).to(dev)
    b = (torch.randn(N, K, generator=g) * 0.02).to(BF16).to(dev)
    out = ops.gemm(a[:M].contiguous(), b, "f32")
    assert torch.equal(out.view(torch.int32), ops.gemm(a, b, "f32")[:M].view(torch.int32))
    ref = a[:M].double() @ b.double().t()
    assert ((out.double() - ref).abs() <= 64 * 2.0 ** -24 * (a[:M].double().abs() @ b.double().abs().t())).all()
    ai = torch.randint(-127, 128, (M, 2 * K), generator=g, dtype=torch.int8).to(dev)
    bi = torch.randint(-127, 128, (N, 2 * K), generator=g, dtype=torch.int8).to(dev)
    assert torch.equal(ops.gemm(ai, bi, "i32").double(), ai.double() @ bi.double().t())
    af, bf = (t.to(dev) for t in _fp8_pair(M, N, 2 * K, 6))
    err = (ops.gemm(af, bf, "f32").double() - af.double() @ bf.double().t()).abs()
    assert (err <= 1e-4 * (af.double().abs() @ bf.double().abs().t())).all()


@pytest.mark.parametrize("M,N,K", [(200, 9216, 1536), (1500, 12288, 256), (1400, 12288, 128), (5990, 9216, 384)])
def test_gate_up_tiles_match(M, N, K):
    """SiLU epilogue on the tiles chosen for short and mid-size gate/up problems (128x128, 192x128 pairs with an
    even, a single and an odd number of stages): rows bitwise equal to the same rows of a product of 8192."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(M + N)
    print(f"[gate/up tiles] {M}x{N}x{K}", flush=True)
    a = torch.randint(-127, 128, (8192, K), generator=g, dtype=torch.int8).to(dev)
    b = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(dev)
    rs, cs = (torch.rand(8192, generator=g) * 1e-2).to(dev), (torch.rand(N, generator=g) * 1e-2).to(dev)
    big = ops.gemm(a, b, "dq_silu", rs=rs, cs=cs)
    out = ops.gemm(a[:M].contiguous(), b, "dq_silu", rs=rs[:M].contiguous(), cs=cs)
    assert torch.equal(out.view(torch.int16), big[:M].view(torch.int16))


# (tile configuration, M, N, K bytes): the tile is checked against the dispatch rule on the CPU (test_launch_rules)
TILE_SHAPES = [
    (10, 33, 72, 128), (10, 250, 1504, 4608), (9, 321, 1528, 256), (9, 500, 1504, 640), (11, 1000, 1512, 4224),
    (6, 2000, 1512, 4224), (13, 2300, 2008, 384), (7, 512, 2560, 1024), (7, 512, 2560, 1088), (7, 512, 2560, 1536),
    (3, 1500, 1528, 128), (3, 1500, 1528, 192), (3, 1500, 1528, 256), (3, 1500, 1528, 960), (2, 40000, 128, 192),
    (2, 40000, 128, 320)]


@pytest.mark.parametrize("tile,M,N,kb", TILE_SHAPES)
def test_gemm_every_tile(tile, M, N, kb):
    """Every tile below the ping-pong ones, each loop with one stage, fewer stages than ring slots, odd, even and many
    (fp8 takes a stage in one wide k-step, so its loops differ): fp8 and bf16 bits equal to the same rows of a
    product of 9000 rows, fp8 within 1e-4 and bf16 within 64 eps of sum|products| of float64, int8 exact."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(M + N + kb)
    rows = max(M, 9000)
    print(f"[tile {tile}] {M}x{N} K bytes {kb}", flush=True)

    def same(a, b):
        out, other = ops.gemm(a[:M].contiguous(), b, "f32"), ops.gemm(a[:9000].contiguous(), b, "f32")
        n = min(M, 9000)
        assert torch.equal(out[:n].view(torch.int32), other[:n].view(torch.int32))
        return out.double(), a[:M].double() @ b.double().t(), a[:M].double().abs() @ b.double().abs().t()

    out, ref, mag = same(*(t.to(dev) for t in _fp8_pair(rows, N, kb, 7)))
    assert ((out - ref).abs() <= 1e-4 * mag).all()
    a = torch.randn(rows, kb // 2, generator=g).to(BF16).to(dev)
    b = (torch.randn(N, kb // 2, generator=g) * 0.02).to(BF16).to(dev)
    out, ref, mag = same(a, b)
    assert ((out - ref).abs() <= 64 * 2.0 ** -24 * mag).all()
    ai = torch.randint(-127, 128, (M, kb), generator=g, dtype=torch.int8).to(dev)
    bi = torch.randint(-127, 128, (N, kb), generator=g, dtype=torch.int8).to(dev)
    assert torch.equal(ops.gemm(ai, bi, "i32").double(), ai.double() @ bi.double().t())


SILU_SHAPES = [(7, 100, 9216, 1536), (3, 200, 9216, 1536), (12, 576, 9216, 1536), (12, 1500, 12288, 256),
               (12, 1400, 12288, 128), (12, 5990, 9216, 384), (4, 1792, 9216, 1536)]


@pytest.mark.parametrize("tile,M,N,kb", SILU_SHAPES)
def test_gate_up_tiles_match_float(tile, M, N, kb):
    """SILU_BF16 with fp8 operands (dequantised) and with bf16 ones on each gate/up tile: rows bitwise equal to the
    same rows of a product of 8192."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(M + N + kb)
    print(f"[gate/up tile {tile}] {M}x{N} K bytes {kb}", flush=True)
    a, b = (t.to(dev) for t in _fp8_pair(8192, N, kb, 8))
    rs, cs = (torch.rand(8192, generator=g) * 1e-3).to(dev), (torch.rand(N, generator=g) * 1e-3).to(dev)
    big = ops.gemm(a, b, "silu_bf16", rs=rs, cs=cs)
    out = ops.gemm(a[:M].contiguous(), b, "silu_bf16", rs=rs[:M].contiguous(), cs=cs)
    assert torch.equal(out.view(torch.int16), big[:M].view(torch.int16))
    a = torch.randn(8192, kb // 2, generator=g).to(BF16).to(dev)
    b = (torch.randn(N, kb // 2, generator=g) * 0.1).to(BF16).to(dev)
    big, out = ops.gemm(a, b, "silu_bf16"), ops.gemm(a[:M].contiguous(), b, "silu_bf16")
    assert torch.equal(out.view(torch.int16), big[:M].view(torch.int16))


@pytest.mark.parametrize("N", [1536, 2048, 2560])
@pytest.mark.parametrize("kb", [64, 128, 192, 384, 448, 1600, 4160])
def test_gemm_ping_pong_stages(N, kb):
    """256x192, 256x256 and 256x320 (bf16, int8) ping-pong tiles (M = 8100, ragged): K of 64 bytes up to 65 times
    that, over every remainder of the unrolled loops, on 128-byte stages with whole and half last ones and (256x320
    in bf16 and with half lines of K) on 64-byte stages: int8 exact, bf16 within 64 eps sum|products| of float64, fp8 within 1e-4 sum|products| (the fp8
    unit's own precision)."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(N + kb)
    M = 8100
    print(f"[ping-pong] {M}x{N} K bytes {kb}", flush=True)
    a = torch.randn(M, kb // 2, generator=g).to(BF16).to(dev)
    b = torch.randn(N, kb // 2, generator=g).to(BF16).to(dev)
    err = (ops.gemm(a, b, "f32").double() - a.double() @ b.double().t()).abs()
    assert (err <= 64 * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t())).all()
    ai = torch.randint(-127, 128, (M, kb), generator=g, dtype=torch.int8).to(dev)
    bi = torch.randint(-127, 128, (N, kb), generator=g, dtype=torch.int8).to(dev)
    assert torch.equal(ops.gemm(ai, bi, "i32").double(), ai.double() @ bi.double().t())
    af, bf = (t.to(dev) for t in _fp8_pair(M, N, kb, 5))
    err = (ops.gemm(af, bf, "f32").double() - af.double() @ bf.double().t()).abs()
    assert (err <= 1e-4 * (af.double().abs() @ bf.double().abs().t())).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("N", [1536, 2048, 2560])
@pytest.mark.parametrize("kb", [64, 192, 1600])
def test_gemm_operand_column_range(N, kb, fp8):
    """Operands that are the last columns of wider matrices (row stride K + 80 bytes, the last row ends with the
    allocation), K bytes an odd multiple of 64: the ping-pong tiles' half stage stops at K, f32 bits equal to those
    of contiguous copies."""
    import ctypes

    from minicpm5_mk import _lib, ops

    dev = _dev()
    g = torch.Generator().manual_seed(N + kb)
    dt, esz = (torch.float8_e4m3fn, 1) if fp8 else (BF16, 2)
    M, K, pad = 8100, kb // esz, 80 // esz
    ld = K + pad
    print(f"[column range] {M}x{N} K bytes {kb} {dt}", flush=True)
    a = torch.randn(M, ld, generator=g).to(dt).to(dev)[:, pad:]
    b = torch.randn(N, ld, generator=g).to(dt).to(dev)[:, pad:]
    out = torch.empty(M, N, dtype=torch.float32, device=dev)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _lib.check(_lib.load().mk_gemm(2 if fp8 else 0, _lib.EPI["f32"], ptr(a), ld, ptr(b), ld, M, N, K, ptr(out), N, None,
                                   0, None, None, None, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "mk_gemm")
    ref = ops.gemm(a.contiguous(), b.contiguous(), "f32")
    assert torch.equal(out.view(torch.int32), ref.view(torch.int32))


@pytest.mark.parametrize("epi", ["f32", "bf16", "res_f32add", "res_bf16add"])
def test_gemm_wide_tile_rows_match(epi):
    """M = 8192, N = 2560 takes the 256x320 tile (one round of 256 CUs; 64x160 wave tiles, the epilogue
    staged in a 128- and a 32-column chunk, the offsets of later async loads recomputed per load), M = 1000
    the 128x128 one: the first 1000 rows are bitwise equal for each epilogue, and the f32 products match
    a float64 reference on rows at both ends."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(2560)
    M, N, K = 8192, 2560, 1536
    a = torch.randn(M, K, generator=g).to(BF16)
    b = (torch.randn(N, K, generator=g) * 0.02).to(BF16)
    x = torch.randn(M, N, generator=g).to(BF16)
    ad, bd = a.to(dev), b.to(dev)
    if epi.startswith("res"):
        big = ops.gemm(ad, bd, epi, res=x.clone().to(dev))
        small = ops.gemm(ad[:1000].contiguous(), bd, epi, res=x[:1000].clone().to(dev))
    else:
        big = ops.gemm(ad, bd, epi)
        small = ops.gemm(ad[:1000].contiguous(), bd, epi)
    assert torch.equal(small.view(torch.int16 if small.dtype == BF16 else torch.int32),
                       big[:1000].view(torch.int16 if big.dtype == BF16 else torch.int32))
    if epi == "f32":
        rows = torch.cat([torch.arange(300), torch.arange(M - 300, M)])
        ref = a[rows].double() @ b.double().t()
        torch.testing.assert_close(big.cpu()[rows].double(), ref, rtol=1e-4, atol=1e-4 * ref.abs().max().item())


_RAGGED_WIDE = r"""
import sys, torch
sys.path[:0] = [sys.argv[1], sys.argv[2]]
from minicpm5_mk import ops
from oracle import emulate
dev = torch.device("cuda:0")
g = torch.Generator().manual_seed(77)
bad = []
for M, N, K in [(300, 200, 1536), (1000, 600, 64), (257, 328, 128), (8292, 2568, 1536)]:
    a = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    b = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    print(f"[wide ragged] int8 {M}x{N}x{K}", flush=True)
    acc = ops.gemm(a.to(dev), b.to(dev), "i32").cpu().to(torch.int64)
    if not torch.equal(acc, emulate.int_matmul(a, b.t().contiguous())):
        bad.append(("i32", M, N, K))
for M, N, K, epi in [(300, 200, 1536, "f32"), (1000, 600, 2048, "f32"), (333, 640, 512, "res_f32add")]:
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(M, N, generator=g).to(torch.bfloat16)
    print(f"[wide ragged] bf16 {epi} {M}x{N}x{K}", flush=True)
    ref = a.double() @ b.double().t()
    if epi == "f32":
        out = ops.gemm(a.to(dev), b.to(dev), "f32").cpu().double()
        ok = ((out - ref).abs() <= 1e-4 * ref.abs().max()).all()
    else:
        out = ops.gemm(a.to(dev), b.to(dev), epi, res=x.clone().to(dev)).cpu().float()
        exp = (x.float() + ref.float())
        ok = ((out - exp).abs() <= exp.abs() * 2.0 ** -7 + 1e-3).all()
    if not bool(ok):
        bad.append((epi, M, N, K))
print("BAD", bad, flush=True)
sys.exit(1 if bad else 0)
"""


def test_gemm_wide_tile_ragged_shapes():
    """The 256x320 tile forced for every GEMM (MK_GEMM_CFG=8, a fresh process: the override is read once)
    on shapes that are not tile multiples -- rows past M and columns past N take the clamped load offsets
    of the lean addressing and the bounds checks of the chunked epilogue: exact int32 products against the
    oracle, bf16 products and the f32 residual epilogue against float64."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, MK_GEMM_CFG="8")
    r = subprocess.run([sys.executable, "-c", _RAGGED_WIDE, root, os.path.join(root, "minicpm5-vllm-tpu_amd")],
                       env=env, capture_output=True, text=True, timeout=240)
    print(r.stdout[-2000:], r.stderr[-2000:])
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]


def test_gemm_residual_epilogues():
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(3)
    M, N, K = 512, 256, 512
    a = torch.randn(M, K, generator=g).to(BF16)
    b = (torch.randn(N, K, generator=g) * 0.05).to(BF16)
    x = torch.randn(M, N, generator=g).to(BF16)
    acc = ops.gemm(a.to(dev), b.to(dev), "f32").cpu()
    r1 = ops.gemm(a.to(dev), b.to(dev), "res_bf16add", res=x.clone().to(dev)).cpu()
    exp1 = (x.float() + acc.to(BF16).float()).to(BF16)
    assert torch.equal(r1, exp1)
    r2 = ops.gemm(a.to(dev), b.to(dev), "res_f32add", res=x.clone().to(dev)).cpu()
    exp2 = (x.float() + acc).to(BF16)
    assert torch.equal(r2, exp2)


def test_gate_up_silu_epilogue():
    """fused_mlp gate/up (mk_mlp.py:79-84): packed in [32 gate | 32 up] blocks, h = silu(g) * u.  One
    8192-row launch (256x128 tiles) vs the oracle on its first and last 640 rows, and 100- and 640-row
    launches (64x128 and 256x128 tiles) equal to its first rows, bit for bit."""
    from minicpm5_mk import ops
    from minicpm5_mk.mk_weights import interleave_gu, mlp_chunk
    from oracle import emulate

    dev = _dev()
    g = torch.Generator().manual_seed(21)
    T, H, inter = 8192, 1536, 4608
    x = torch.randn(T, H, generator=g).to(BF16)
    w = torch.randint(-127, 128, (H, 2, inter), generator=g, dtype=torch.int8)
    s = torch.rand(2, inter, generator=g) * 2e-3
    a = torch.rand(H, generator=g) + 0.5
    ic = mlp_chunk(inter)
    w_il, s_il = interleave_gu(w, s, ic)                       # reference layout (H, 2I), (1, 2I)
    wp = ops.pack_weight(w_il.to(dev), map_gu=True, ic=ic, inter=inter)     # (2I, H) packed
    s_p = _pack_gu_scales(s_il, inter).to(dev)
    q, sx = ops.row_quant(x.to(dev), a.to(dev), 1e-6, True, True)
    h = ops.gemm(q, wp, "dq_silu", rs=sx, cs=s_p)
    for M in (100, 640):
        hm = ops.gemm(q[:M].contiguous(), wp, "dq_silu", rs=sx[:M].contiguous(), cs=s_p)
        assert torch.equal(hm, h[:M]), M
    rows = torch.cat([torch.arange(640), torch.arange(T - 640, T)])
    h = h.float().cpu()[rows]
    qr, _ = emulate.row_quant(x[rows].float(), a, 1e-6, True, True)
    gu = (emulate.int_matmul(qr, w.reshape(H, -1)).float() * sx.cpu()[rows][:, None]) * s.reshape(1, -1)
    ref = emulate.silu_f32(gu[:, :inter]) * gu[:, inter:]
    err = (h - ref).abs()
    assert (err <= ref.abs() * 2.0 ** -7 + 1e-6).all(), float(err.max())


def test_lm_head():
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator(device=dev).manual_seed(9)
    w = (torch.randn(130560, 1536, generator=g, device=dev) * 0.02).to(BF16)
    for B in (1, 5, 40):
        hdn = torch.randn(B, 1536, generator=g, device=dev).to(BF16)
        out = ops.lm_head(hdn, w)
        ref = hdn.float() @ w.float().t()          # f32 torch reference for a floating-point kernel
        torch.testing.assert_close(out, ref, rtol=1e-4, atol=2e-4)


def _pack_gu_scales(s_il, inter):
    """Per-column scales of the chunk-interleaved gate/up matrix in the packed order: packed row p holds
    [32 gate | 32 up] block p // 64, half (p // 32) % 2, intermediate column 32 (p // 64) + p % 32."""
    from minicpm5_mk.mk_weights import mlp_chunk

    ic = mlp_chunk(inter)
    p = torch.arange(2 * inter)
    n = (p // 64) * 32 + p % 32
    src = (n // ic) * 2 * ic + ((p // 32) % 2) * ic + n % ic
    return s_il.reshape(-1)[src].contiguous()


@pytest.mark.parametrize("V,H", [(1000, 1536), (1000, 2048), (520, 256), (520, 1152), (16392, 256), (16400, 2048)])
def test_lm_head_batches(V, H):
    """Batches at the edges of the LM head's 16-row groups and 64-row passes (H = 1152: no whole 256-element
    chunks, the 32-row kernel; above V = 16384 the batch kernel takes fewer than 17 rows too): f32 sums of exact bf16 products, so each logit is within 32 eps sum|products|
    of the float64 one, and a row's bits do not depend on the batch."""
    from minicpm5_mk import ops

    dev = _dev()
    g = torch.Generator().manual_seed(V + H)
    x = torch.randn(129, H, generator=g).to(BF16).to(dev)
    w = (torch.randn(V, H, generator=g) * 0.02).to(BF16).to(dev)
    full = ops.lm_head(x, w)
    ref = x.double() @ w.double().t()
    bound = 32 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    for B in (1, 2, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 128):
        out = ops.lm_head(x[:B].contiguous(), w)
        assert ((out.double() - ref[:B]).abs() <= bound[:B]).all(), B
        # few rows, or one over more than 1536 k, take the skinny kernel: same sums, same bits
        assert torch.equal(out.view(torch.int32), full[:B].view(torch.int32)), B


@pytest.mark.parametrize("smooth", [False, True])
def test_decoder_block_int8(smooth):
    """Quantised decoder block at its full size (8192 tokens, MiniCPM5-1B hd-96 shapes): fused RMSNorm +
    QKV (mk_mlp.py:161-170), int8d O projection + bf16 residual (mk_jax.py:243-265, :394), fused MLP with
    int8 gate/up and int8 down (mk_mlp.py:68-97).  X ~ N(0, 1) from seed 3, weights ~ N(0, 0.02) from
    seed 0 quantised per output channel; activations per-token dynamic int8 with a = gamma (= 1), or
    SmoothQuant a = 1 / s with s from X's and the weight's per-channel amax (mk_weights.py:229-252).
    Checked stage by stage against the oracle's restatement of the same algebra: QKV within one bf16 ulp,
    the O residual bit-exact, the block output within bf16 rounding (SiLU's exp differs in the last f32
    bits, which can move an int8 code of h)."""
    from minicpm5_mk import ops
    from minicpm5_mk.mk_weights import interleave_gu, mlp_chunk, quantize_w
    from oracle import emulate

    dev = _dev()
    T, H, hd, n_q, n_kv, inter, eps = 8192, 1536, 96, 16, 2, 4608, 1e-6
    D, qd = (n_q + 2 * n_kv) * hd, n_q * hd
    print(f"[block] T={T} smooth={smooth}", flush=True)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(3)).to(BF16)
    g0 = torch.Generator().manual_seed(0)
    w_qkv, w_o, w_gu, w_dn = (torch.randn(r, c, generator=g0) * 0.02 for r, c in
                              ((H, D), (qd, H), (H, 2 * inter), (inter, H)))
    ones = lambda n: torch.ones(n)  # noqa: E731

    def smooth_of(xa, w):
        if not smooth:
            return ones(w.shape[0])
        s = xa.float().abs().amax(0).pow(0.5) / w.abs().amax(1).clamp_min(1e-12).pow(0.5)
        return s.clamp(1e-4, 1e4)

    s1 = smooth_of(x, w_qkv)
    q_qkv, sc_qkv = quantize_w(w_qkv * s1[:, None], "int8d", 1.0)
    a_qkv = 1.0 / s1
    q_o, sc_o = quantize_w(w_o, "int8d", 1.0)
    q_gu, sc_gu = quantize_w(w_gu * s1[:, None], "int8d", 1.0)
    q_dn, sc_dn = quantize_w(w_dn, "int8d", 1.0)
    ic = mlp_chunk(inter)
    q_gu_il, sc_gu_il = interleave_gu(q_gu.view(H, 2, inter), sc_gu.view(2, inter), ic)
    a_o, a_dn = ones(qd), ones(inter)

    # ---- GPU, launched as the model's layer does
    xd = x.to(dev)
    q8, sx = ops.row_quant(xd, a_qkv.to(dev), eps, True, True)
    qkv = ops.gemm(q8, ops.pack_weight(q_qkv.to(dev)), "dq_bf16", rs=sx, cs=sc_qkv.reshape(-1).to(dev))
    att = qkv[:, :qd].contiguous()          # stands in for the attention output (same shape)
    q8, sx = ops.row_quant(att, a_o.to(dev), 0.0, False, False)
    x1 = ops.gemm(q8, ops.pack_weight(q_o.to(dev)), "dq_res_bf16add", rs=sx, cs=sc_o.reshape(-1).to(dev),
                  res=xd.clone())
    q8, sx = ops.row_quant(x1, a_qkv.to(dev), eps, True, True)
    wgu = ops.pack_weight(q_gu_il.to(dev), map_gu=True, ic=ic, inter=inter)
    h = ops.gemm(q8, wgu, "dq_silu_f32a", rs=sx, cs=_pack_gu_scales(sc_gu_il, inter).to(dev), aux=a_dn.to(dev))
    q8, sx = ops.row_quant(h, None, 0.0, False, True)
    x2 = ops.gemm(q8, ops.pack_weight(q_dn.to(dev)), "dq2_res_f32add", rs=sx, cs=sc_dn.reshape(-1).to(dev),
                  res=x1.clone())
    torch.cuda.synchronize()
    qkv, x1, x2 = qkv.cpu(), x1.cpu(), x2.float().cpu()

    # ---- oracle, stage by stage on the GPU's own inputs to each stage.  RMSNorm's sum of squares runs
    # in a different order on the GPU, so rstd (and the dequantised QKV / gate-up values) may differ by
    # one f32 ulp: QKV within one bf16 ulp, the O stage bit-exact
    def within_ulp(a, b):   # one bf16 ulp is at most 2^-7 of the value
        return bool(((a.float() - b.float()).abs() <= b.float().abs() * 2.0 ** -7 + 1e-30).all())

    qkv_r = emulate.fused_qkv(x, q_qkv, sc_qkv, a_qkv, eps)
    assert within_ulp(qkv, qkv_r)
    o_r = emulate.linear(qkv[:, :qd], q_o, sc_o, a_o, "int8d")
    x1_r = emulate.bf(x.float() + o_r.float()).to(BF16)
    assert torch.equal(x1, x1_r)
    x2_r = emulate.fused_mlp(x1, q_gu_il, sc_gu_il, a_qkv, q_dn, sc_dn, a_dn, eps, ic).float()
    err = (x2 - x2_r).abs()
    print(f"[block] out max {err.max():.4g} mean {err.mean():.4g}; |out| max {x2_r.abs().max():.3g}", flush=True)
    assert (err <= x2_r.abs() * 2.0 ** -7 + 2e-2).all() and err.mean() <= 1e-3, (float(err.max()), float(err.mean()))


# ------------------------------------------------------------------------------------ fp8 / static int8
@pytest.mark.parametrize("mode,norm,recip,smul", [("fp8d", True, False, True), ("fp8d", False, True, True),
                                                  ("int8d", True, False, True), ("int8", True, False, False),
                                                  ("int8", False, False, False), ("fp8", True, False, False),
                                                  ("fp8", False, False, False)])
def test_act_quant_modes(mode, norm, recip, smul):
    from minicpm5_mk import ops
    from oracle import emulate

    dev = _dev()
    print(f"[act_quant] {mode} norm={norm} recip={recip} smul={smul}", flush=True)
    g = torch.Generator().manual_seed(len(mode) * 10 + norm)
    T, H = 777, 1536
    x = (torch.randn(T, H, generator=g) * 3).to(BF16)
    x[0] = 0.0                                      # all-zero row: dynamic scale floor 1e-6
    x[1, :5] = torch.tensor([1e-30, -5e-3, 300.0, -7.0, 2.0 ** -12]).to(BF16)
    # static modes: per-channel factors a = 1 / s_x, as prepared weights carry them (large enough to clip)
    a = (torch.rand(H, generator=g) + 0.5) * (40.0 if mode in ("int8", "fp8") else 1.0)
    q, sx = ops.act_quant(x.to(dev), a.to(dev), mode, 1e-6, norm, recip, smul)
    qr, sxr = emulate.act_quant(x.float(), a, 1e-6, mode, norm, recip, smul)
    q, sx = q.cpu(), sx.cpu()
    assert q.dtype == qr.dtype
    if mode.endswith("d"):
        assert torch.equal(q.view(torch.uint8), qr.view(torch.uint8))
        if norm:
            torch.testing.assert_close(sx, sxr, rtol=4e-7, atol=0)
        else:
            assert torch.equal(sx, sxr)
    else:
        assert torch.equal(sx, torch.ones(T))
        if mode == "int8":
            d = (q.to(torch.int32) - qr.to(torch.int32)).abs()
        else:   # adjacent e4m3 codes of one sign differ by one in their magnitude bits
            d = (q.view(torch.uint8).to(torch.int32) - qr.view(torch.uint8).to(torch.int32)).abs()
        if norm:
            assert d.max() <= 1 and (d > 0).float().mean() <= 1e-3, (int(d.max()), float((d > 0).float().mean()))
        else:
            assert d.max() == 0


def test_fp8_conversion_exhaustive():
    """Every finite bf16 value, clipped to +-448, through the hardware e4m3 conversion (static fp8, a = 1)
    vs torch's round-to-nearest-even float8_e4m3fn cast."""
    from minicpm5_mk import ops

    dev = _dev()
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    x = bits.view(BF16).reshape(256, 256).clone()
    x[~torch.isfinite(x.float())] = 0.0
    q, _ = ops.act_quant(x.to(dev), None, "fp8", 0.0, False)
    ref = torch.clamp(x.float(), -448.0, 448.0).to(torch.float8_e4m3fn)
    qb, rb = q.cpu().view(torch.uint8), ref.view(torch.uint8)
    bad = (qb != rb).nonzero()
    assert bad.numel() == 0, [(float(x[i, j]), int(qb[i, j]), int(rb[i, j])) for i, j in bad[:8].tolist()]


def _fp8_pair(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    a = (torch.randn(M, K, generator=g) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    b = (torch.randn(N, K, generator=g) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    return a, b


@pytest.mark.parametrize("M,N,K", [(256, 128, 64), (300, 200, 1536), (8192, 1920, 1536), (13, 4096, 2048)])
def test_gemm_fp8(M, N, K):
    from minicpm5_mk import ops
    from oracle import emulate

    dev = _dev()
    a, b = _fp8_pair(M, N, K, M + N)
    out = ops.gemm(a.to(dev), b.to(dev), "f32").cpu()
    ref = emulate.fp8_matmul(a, b.t().contiguous())
    bound = a.to(torch.float64).abs() @ b.to(torch.float64).abs().t()
    err = (out.double() - ref.double()).abs()
    assert (err <= 1e-4 * bound).all(), float((err / bound.clamp(min=1e-30)).max())


@pytest.mark.parametrize("epi", ["dq2_bf16", "dq2_res_bf16add", "dq_res_bf16add", "silu_bf16"])
def test_gemm_fp8_epilogues(epi):
    from minicpm5_mk import ops
    from oracle import emulate

    dev = _dev()
    M, N, K = 1000, 512, 1536
    a, b = _fp8_pair(M, N, K, 17)
    g = torch.Generator().manual_seed(18)
    rs = torch.rand(M, generator=g) * 1e-3
    cs = torch.rand(N, generator=g) * 1e-3
    acc = emulate.fp8_matmul(a, b.t().contiguous())
    bound = (a.to(torch.float64).abs() @ b.to(torch.float64).abs().t()).float() * 1e-4
    x = torch.randn(M, N, generator=g).to(BF16)
    kw = dict(rs=rs.to(dev), cs=cs.to(dev))
    if epi == "dq2_bf16":
        out = ops.gemm(a.to(dev), b.to(dev), epi, **kw).float().cpu()
        ref = acc * (rs[:, None] * cs[None, :])
        scale = rs[:, None] * cs[None, :]
    elif epi == "silu_bf16":
        out = ops.gemm(a.to(dev), b.to(dev), epi, **kw).float().cpu()   # (M, N/2), 32-column g/u blocks
        gu = (acc * (rs[:, None] * cs[None, :])).to(BF16).float().view(M, -1, 2, 32)
        gv, uv = gu[:, :, 0].reshape(M, -1), gu[:, :, 1].reshape(M, -1)
        ref = (gv / (1 + torch.exp(-gv))).to(BF16).float() * uv
        tol = ref.abs() * 2.0 ** -6 + 1e-6
        assert ((out - ref).abs() <= tol).all()
        return
    else:
        out = ops.gemm(a.to(dev), b.to(dev), epi, res=x.clone().to(dev), **kw).float().cpu()
        o = acc * (rs[:, None] * cs[None, :]) if epi == "dq2_res_bf16add" else (acc * rs[:, None]) * cs[None, :]
        ref = (x.float() + o.to(BF16).float())
        scale = rs[:, None] * cs[None, :]
        tol = (x.float().abs() + o.abs()) * 2.0 ** -7 + bound * scale + 1e-30
        assert ((out - ref).abs() <= tol).all()
        return
    tol = ref.abs() * 2.0 ** -7 + bound * scale + 1e-30
    assert ((out - ref).abs() <= tol).all()
