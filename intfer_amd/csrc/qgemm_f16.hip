// FP16-activation dequant GEMM: the reference's default GPU linear path
// (quant_gemm_forward_usm, src/gemm/quant_gemm.cpp:359-2153), on the device
// weight layout of this library.
//
//   out(m, n) = fp16_rne( sum_k a(m, k) * w(n, k) )     fp32, k ascending
//   w(n, k)   = (scale(n, g) * alpha) * cb(code(n, k))  g = k / 128
//   cb(c)     = the canonical codebook (2c - C) / C as an fp32 constant
//               ({-1, -1/3, 1/3, 1} for INT2; canon_value, :139-144)
//
// M == 1 follows the decode kernels (:1026-1080 for INT2, :2022-2066): the
// weight stays fp32 and every step is acc = fma(a, w, acc) (the reference's
// `acc += av * w` contracted, as its device compiler's default fp model
// does).  M > 1 follows the tiled kernel (:2069-2150): the weight tile is
// rounded to fp16 when staged, so each product a * w of two halves is exact
// in fp32 and the step is one rounded add (fma gives the same bits).
//
// This path holds no integer T; it is the reference's fp16 operating point
// beside the W2A8 path (qgemm.hip), for parity with the reference's default
// numerics.  The accumulation order is the reference's: the products go
// through v_mfma_f32_16x16x4_f32, which adds its four products to the
// accumulator in ascending k, each step one fused multiply-add with a single
// rounding (test_qgemm_f16_rounding_of_every_step: sums that cancel, full-width
// fp32 weights and fp16 subnormals, bit for bit against the sequential loop).
#include "ifr_dev.h"
#include "ifr_kernels.h"

namespace ifrk {
namespace {

// Codes in the fragment-major layout (pack_linear_host): column tile n / 16,
// K step k / 64, lane 16 (k % 64 / 16) + n % 16, code j = k % 16 of that
// lane in operand dword j / 4, byte j % 4 (INT8 stored as c ^ 0x80).

template <int BITS>
__device__ __forceinline__ float canon(int c) {
  if constexpr (BITS == 2) {
    return c == 0 ? -1.0f : c == 1 ? -1.0f / 3.0f : c == 2 ? 1.0f / 3.0f : 1.0f;
  } else {
    constexpr float C = (float)((1 << BITS) - 1);
    return (2.0f * (float)c - C) / C;
  }
}

// scale(n, g) * alpha, the reference's `s` (fp32)
__device__ __forceinline__ float group_scale(const F16Args& p, int n, int g) {
  const uint32_t zw = p.sz[((size_t)(n >> 4) * p.ng + g) * 16 + (n & 15)];
  return ifrd::h2f((uint16_t)(zw & 0xFFFFu)) * p.alpha;
}

// One workgroup: BM = 16 WM rows x 4 column tiles, one tile per wave, over the
// whole K; per 128-wide K group the A rows are converted to fp32 once and
// staged in LDS (two buffers, one barrier per group), the weights are decoded
// by the wave that uses them.
//
// Bound: the fp32 matrix rate (32 multiply-adds per cycle and SIMD; 130 TFLOP/s
// reached here) for many rows, the chain of dependent MFMAs (40 cycles per 4 k)
// for few.  The vector ALU it replaces runs 16 per cycle, and its 64 x 64
// blocks left most CUs idle at N = 1024..4096: 0.8B QKV (K 1024, N 4096), INT2,
// M = 361: 132.8 -> 38.2 us (79 TFLOP/s); M = 16: 97 -> 11.6 us; M = 1: 15.2 ->
// 11.6 us.
//
// MFMA i of a group takes k = 4 i + q in lane group q = lane / 16.  In the
// fragment-major code layout those are byte q of the packed dwords of the four
// 16-code chunks of a K step, so a lane loads each chunk's dwords (one address
// per column, shared by the four lane groups) and shifts its byte down.
template <int BITS, int WM, bool M1>
__global__ __launch_bounds__(256) void qgemm_f16_mfma(F16Args p, int avec) {
  constexpr int BM = 16 * WM;
  // LDS, 16-byte units: chunk qq (16 k) at qq * PITCH, then [q][row]: the four
  // values k = 16 qq + 4 jj + q, jj = 0..3, of a row.  The pitch spreads the
  // eight chunks a row's threads write over all banks.
  constexpr int PITCH = 4 * BM + 1, BUF = 8 * PITCH;
  constexpr int NU = 8 * BM, UPT = (NU + 255) / 256;  // (row, chunk) units, per thread
  extern __shared__ v4f sA[];
  // 2 and 4 bits: each wave's weights of the group, [code][column], so that a
  // code costs two address operations and one LDS read (the vector ALU and the
  // fp32 MFMA do not overlap here); 8 bits: the codebook values
  constexpr int NT = BITS == 8 ? 256 : 4 * 16 << BITS;
  __shared__ float tab[NT];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int t = min((int)blockIdx.x * 4 + wave, p.N / 16 - 1);  // past the last tile: not stored
  const int m0 = blockIdx.y * BM;
  float* const wt = BITS == 8 ? tab : tab + (wave * 16 << BITS);
  constexpr int TE = BITS == 8 ? 1 : (1 << BITS) / 4;  // table entries per lane: codes q, q + 4, ..
  float cv[TE];
  if constexpr (BITS == 8)
    for (int i = threadIdx.x; i < 256; i += 256) tab[i] = canon<8>(i);
  else
#pragma unroll
    for (int e = 0; e < TE; ++e) cv[e] = canon<BITS>(q + 4 * e);

  uint4 av[UPT][2];
  auto load_a = [&](int g) {
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      const int u = threadIdx.x + 256 * j;
      if (NU % 256 != 0 && u >= NU) break;
      const uint16_t* src = p.a + (size_t)min(m0 + (u >> 3), p.M - 1) * p.K + 128 * g + 16 * (u & 7);
      if (avec) {
        av[j][0] = reinterpret_cast<const uint4*>(src)[0];
        av[j][1] = reinterpret_cast<const uint4*>(src)[1];
      } else {  // the caller's rows are not 16-byte aligned
        uint32_t w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = (uint32_t)src[2 * i] | ((uint32_t)src[2 * i + 1] << 16);
        av[j][0] = make_uint4(w[0], w[1], w[2], w[3]);
        av[j][1] = make_uint4(w[4], w[5], w[6], w[7]);
      }
    }
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      const int u = threadIdx.x + 256 * j;
      if (NU % 256 != 0 && u >= NU) break;
      const uint32_t w[8] = {av[j][0].x, av[j][0].y, av[j][0].z, av[j][0].w,
                             av[j][1].x, av[j][1].y, av[j][1].z, av[j][1].w};
      v4f* dst = sA + buf * BUF + (u & 7) * PITCH + (u >> 3);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v4f x;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)  // half 4 jj + e
          x[jj] = ifrd::h2f((uint16_t)(w[2 * jj + (e >> 1)] >> (16 * (e & 1))));
        dst[e * BM] = x;
      }
    }
  };
  // the group's packed dwords of this lane's column, chunk by chunk
  struct Codes {
    uint32_t w[8][BITS / 2];
    float sc;
  };
  auto load_w = [&](Codes& o, int g) {
    const uint32_t* src = p.codes + (((size_t)t * p.nsteps + 2 * g) * 64 + c) * (BITS / 2);
#pragma unroll
    for (int qq = 0; qq < 8; ++qq)
#pragma unroll
      for (int i = 0; i < BITS / 2; ++i) o.w[qq][i] = src[16 * qq * (BITS / 2) + i];
    o.sc = group_scale(p, 16 * t + c, g);
  };
  // fp32 weights k = 16 qq + 4 jj + q, jj = 0..3 (rounded to fp16 unless M1)
  auto rnd = [](float x) { return M1 ? x : ifrd::fp16r(x); };
  auto decode = [&](const uint32_t (&w)[BITS / 2], float sc, float (&b)[4]) {
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      if constexpr (BITS == 8) {
        b[jj] = rnd(sc * tab[((w[jj] >> (8 * q)) & 0xFFu) ^ 0x80u]);
      } else {
        const uint32_t x = BITS == 2 ? (w[0] >> (8 * q + 2 * jj)) & 3u : (w[jj >> 1] >> (8 * q + 4 * (jj & 1))) & 15u;
        b[jj] = wt[16 * x + c];
      }
    }
  };

  const int ng = p.ng;
  Codes cur, nxt;
  load_a(0);
  load_w(cur, 0);
  store_a(0);
  v4f acc[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) acc[i] = (v4f){0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  for (int g = 0; g < ng; ++g) {
    const int gn = min(g + 1, ng - 1);
    load_a(gn);
    load_w(nxt, gn);
    const v4f* A = sA + (g & 1) * BUF + q * BM + c;
    if constexpr (BITS != 8) {
      ifrd::wave_sync();  // the wave's reads of the previous group's weights
#pragma unroll
      for (int e = 0; e < TE; ++e) wt[16 * (q + 4 * e) + c] = rnd(cur.sc * cv[e]);
      ifrd::wave_sync();
    }
    float b[2][4];
    decode(cur.w[0], cur.sc, b[0]);
#pragma unroll
    for (int qq = 0; qq < 8; ++qq) {
      v4f a[WM];
#pragma unroll
      for (int i = 0; i < WM; ++i) a[i] = A[qq * PITCH + 16 * i];
      if (qq < 7) decode(cur.w[qq + 1], cur.sc, b[(qq + 1) & 1]);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int i = 0; i < WM; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][jj], b[qq & 1][jj], acc[i], 0, 0, 0);
    }
    // the other buffer's readers passed the barrier of the group before
    store_a((g + 1) & 1);
    cur = nxt;
    __syncthreads();
  }
  if ((int)blockIdx.x * 4 + wave >= p.N / 16) return;
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + 16 * i + 4 * q + r;
      if (m < p.M) p.out[(size_t)m * p.N + 16 * t + c] = ifrd::f2h(acc[i][r]);
    }
}

template <int BITS, int WM, bool M1>
hipError_t launch_mfma(const F16Args& p, hipStream_t st) {
  constexpr int BM = 16 * WM;
  const size_t lds = (size_t)2 * 8 * (4 * BM + 1) * sizeof(v4f);
  static bool attr_set = false;
  if (lds > 64 * 1024 && !attr_set) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(qgemm_f16_mfma<BITS, WM, M1>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((qgemm_f16_mfma<BITS, WM, M1>), dim3((p.N / 16 + 3) / 4, (p.M + BM - 1) / BM), dim3(256), lds, st,
                     p, (int)(reinterpret_cast<uintptr_t>(p.a) % 16 == 0));
  return hipGetLastError();
}

template <int BITS>
hipError_t launch_f16_bits(const F16Args& p, hipStream_t st) {
  if (p.M == 1) return launch_mfma<BITS, 1, true>(p, st);
  // 16, 32 or 64 rows per workgroup: the fewest rounds of the 256 CUs, a round
  // of the three costing about 7 : 13 : 22 (K = 1024: 7.5, 12.5 and 22 us; the
  // weights are decoded once per workgroup).  One size for all would cost, at
  // N = 4096, M = 32 / 256 / 576: 16 rows 11.7 / 31.0 / 63.5, 32 rows 15.6 /
  // 27.3 / 60.1, 64 rows 25.2 / 27.6 / 67.9 us.
  auto cost = [&](long bm, long unit) {
    return unit * (((p.N / 16 + 3) / 4 * ((p.M + bm - 1) / bm) + 255) / 256);
  };
  const long c1 = cost(16, 7), c2 = cost(32, 13), c4 = cost(64, 22);
  if (c1 <= c2 && c1 <= c4) return launch_mfma<BITS, 1, false>(p, st);
  return c2 <= c4 ? launch_mfma<BITS, 2, false>(p, st) : launch_mfma<BITS, 4, false>(p, st);
}

}  // namespace

hipError_t launch_qgemm_f16(const F16Args& p, hipStream_t st) {
  if (p.M <= 0) return hipSuccess;
  if (!p.a || !p.codes || !p.sz || !p.out || p.N % 16 != 0 || p.K % 128 != 0 || p.ng != p.K / 128 ||
      p.nsteps != p.K / 64)
    return hipErrorInvalidValue;
  switch (p.bits) {
    case 2: return launch_f16_bits<2>(p, st);
    case 4: return launch_f16_bits<4>(p, st);
    case 8: return launch_f16_bits<8>(p, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ifrk
