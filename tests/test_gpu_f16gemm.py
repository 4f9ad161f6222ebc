"""The FP16-activation dequant GEMM (ifr_quant_gemm_f16: the reference's
default GPU linear, quant_gemm_forward_usm, quant_gemm.cpp:359-2153) on the
device against the oracle's restatement, bit for bit: fp32 accumulation in
ascending k, w = (scale * alpha) * canonical codebook value, fp32 weights and
fused steps at M == 1, fp16-rounded weights at M > 1.  The oracle is pinned
in tests/test_oracle.py (numpy float32 step by step; exact rational fma)."""
import ctypes as C

import numpy as np
import pytest

import intfer_amd as ia
from oracle import pyoracle as po
from oracle.pyoracle import ptr
from tests.conftest import announce

pytestmark = pytest.mark.gpu
L = ia.lib()


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("N,K", [(256, 1024), (144, 3072)])
def test_qgemm_f16_matches_oracle(dev, bits, N, K):
    rng = np.random.default_rng(bits * 7 + K)
    lin = ia.make_linear(N, K, bits, rng)
    dl = C.c_void_p()
    ia.check(L.ifr_linear_upload(dev.ctx, C.byref(lin.struct), C.byref(dl)), "upload")
    try:
        for M, alpha in ((1, 1.0), (1, 0.37), (3, 1.0), (64, 2.5), (130, 1.0)):
            a = (rng.standard_normal((M, K)) * 2).astype(np.float16)
            ad = dev.upload(a.view(np.uint16))
            od = dev.alloc(M * N * 2)
            announce(f"fp16 GEMM bits={bits} N={N} K={K} M={M}")
            ia.check(L.ifr_quant_gemm_f16(dev.ctx, dl, ad.p, M, C.c_float(alpha), od.p), "f16 gemm")
            got = dev.download(od, np.uint16, (M, N))
            ref = np.empty((M, N), np.uint16)
            po.oracle().or_qgemm_f16(ptr(a.view(np.uint16)), M, C.byref(lin.struct), np.float32(alpha), ptr(ref))
            assert np.array_equal(got, ref), (M, alpha)
            ad.free()
            od.free()
    finally:
        L.ifr_linear_free(dev.ctx, dl)


def test_qgemm_f16_declines_non_codebook_and_pairs(dev):
    rng = np.random.default_rng(3)
    N, K = 64, 256
    gen = ia.make_linear(N, K, 2, rng, zero=rng.uniform(0, 3, size=(N, K // 128)))
    g, u = ia.make_linear(N, K, 2, rng), ia.make_linear(N, K, 2, rng)
    d1, d2 = C.c_void_p(), C.c_void_p()
    ia.check(L.ifr_linear_upload(dev.ctx, C.byref(gen.struct), C.byref(d1)), "upload")
    ia.check(L.ifr_linear_upload_pair(dev.ctx, C.byref(g.struct), C.byref(u.struct), C.byref(d2)), "pair")
    a = dev.alloc(4 * K * 2)
    o = dev.alloc(4 * N * 2 * 2)
    try:
        for d in (d1, d2):
            assert L.ifr_quant_gemm_f16(dev.ctx, d, a.p, 4, C.c_float(1.0), o.p) == ia.IFR_EDECLINE
    finally:
        L.ifr_linear_free(dev.ctx, d1)
        L.ifr_linear_free(dev.ctx, d2)


@pytest.mark.parametrize("bits,N,K,M,shift", [(2, 16, 128, 2, 0), (4, 80, 256, 17, 0), (2, 1024, 128, 361, 0),
                                              (4, 1024, 128, 800, 0), (8, 1024, 128, 801, 0), (2, 144, 256, 33, 2),
                                              (4, 48, 128, 1, 2)])
def test_qgemm_f16_row_blocks_and_unaligned_rows(dev, bits, N, K, M, shift):
    """Each row-block size the launch picks (16, 32 and 64 rows), partial last
    blocks and column tiles, and activations that start off a 16-byte
    boundary, bit for bit against the oracle."""
    rng = np.random.default_rng(bits * 11 + M)
    lin = ia.make_linear(N, K, bits, rng)
    dl = C.c_void_p()
    ia.check(L.ifr_linear_upload(dev.ctx, C.byref(lin.struct), C.byref(dl)), "upload")
    a = (rng.standard_normal((M, K)) * 2).astype(np.float16)
    ad = dev.upload(np.concatenate([np.zeros(shift // 2, np.uint16), a.view(np.uint16).reshape(-1)]))
    od = dev.alloc(M * N * 2)
    try:
        announce(f"fp16 GEMM bits={bits} N={N} K={K} M={M} shift={shift}")
        ia.check(L.ifr_quant_gemm_f16(dev.ctx, dl, C.c_void_p(ad.p.value + shift), M, C.c_float(0.37), od.p), "f16 gemm")
        ref = np.empty((M, N), np.uint16)
        po.oracle().or_qgemm_f16(ptr(a.view(np.uint16)), M, C.byref(lin.struct), np.float32(0.37), ptr(ref))
        assert np.array_equal(dev.download(od, np.uint16, (M, N)), ref)
    finally:
        ad.free()
        od.free()
        L.ifr_linear_free(dev.ctx, dl)


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("M", [1, 2, 100])
def test_qgemm_f16_rounding_of_every_step(dev, bits, M):
    """The second half of a row meets the first half's weights negated, so the
    exact sums are 0 and an output is what the roundings of its 512 steps left:
    it pins the order of the products inside and between the matrix
    instructions and the single rounding of each step (fp32 weights at one
    row).  fp16 subnormal activations among them."""
    rng = np.random.default_rng(70 + bits)
    N, K = 48, 512
    half = ia.make_linear(N, K // 2, bits, rng, scale_sigma=0.5)
    vals = np.concatenate([half.values, ((1 << bits) - 1) - half.values], 1)
    twice = lambda x: np.concatenate([x.reshape(N, -1)] * 2, 1)
    lin = ia.HostLinear(N, K, bits, ia.pack_codes(vals, bits), twice(half.scale), twice(half.zero), vals, 0.0)
    a = rng.standard_normal((M, K // 2)) * 10.0 ** rng.integers(-3, 4, size=(M, K // 2))
    a[:, ::16] *= 1e-6
    a = np.concatenate([a, a], 1).astype(np.float16)
    assert ((a != 0) & (np.abs(a) < 6.1e-5)).any()
    alpha = np.float32(3.7)
    ref, rev = np.empty((M, N), np.uint16), np.empty((M, N), np.uint16)
    po.oracle().or_qgemm_f16(ptr(a.view(np.uint16)), M, C.byref(lin.struct), alpha, ptr(ref))
    # the test can tell orders apart: the halves swapped sum to something else
    b = np.ascontiguousarray(a[:, ::-1])
    back = ia.HostLinear(N, K, bits, ia.pack_codes(np.ascontiguousarray(vals[:, ::-1]), bits), twice(half.scale)[:, ::-1].copy(),
                         lin.zero, vals, 0.0)
    po.oracle().or_qgemm_f16(ptr(b.view(np.uint16)), M, C.byref(back.struct), alpha, ptr(rev))
    assert (ref != rev).mean() > 0.5
    dl = C.c_void_p()
    ia.check(L.ifr_linear_upload(dev.ctx, C.byref(lin.struct), C.byref(dl)), "upload")
    ad, od = dev.upload(a.view(np.uint16)), dev.alloc(M * N * 2)
    try:
        announce(f"fp16 GEMM rounding bits={bits} M={M}")
        ia.check(L.ifr_quant_gemm_f16(dev.ctx, dl, ad.p, M, C.c_float(alpha), od.p), "f16 gemm")
        assert np.array_equal(dev.download(od, np.uint16, (M, N)), ref)
    finally:
        ad.free()
        od.free()
        L.ifr_linear_free(dev.ctx, dl)
