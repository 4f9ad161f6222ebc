// lm_head (tied embedding) as an int8 x int8 MFMA GEMM fused with a
// first-max-wins argmax.
//
// Weights: per-row symmetric int8 with an fp16 row scale, quantized at load
// exactly as the reference's INT8 lm_head upload (examples/intfer_cli/
// main.cpp:1745-1761).  Activations: final-normed rows quantized per 64-wide
// slice with round-to-nearest-even (the reference lm_head act-quant,
// main.cpp:2445-2451, dashq.hpp:61-78).  Per 64-slice s:
//     T = sum a_q * w_q (int32), acc = fma((float)T, as(m,s), acc)
// logit = acc * ws(v).  Argmax: strict '>' scanning the vocabulary in order
// (main.cpp:8289-8312); ties keep the lower index.
#include "ifr_dev.h"
#include "ifr_kernels.h"

namespace ifrk {
namespace {

constexpr int kWN = 2;  // column tiles per wave

struct LmP {
  const int8_t* a;
  const float* as;
  const uint32_t* w;
  const uint16_t* ws;
  float* logits;
  float* pv;
  int32_t* pi;
  int W, V, H, nsteps;
};

__device__ __forceinline__ bool better(float v, int i, float bv, int bi) {
  return v > bv || (v == bv && i < bi);
}

template <int WM, int R>
__global__ __launch_bounds__(256) void lmhead_kernel(LmP p) {
  extern __shared__ float as_l[];  // [16 WM rows][nsteps] activation scales of the block
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lrow = lane & 15, lgrp = lane >> 4;
  const int ntiles = p.V >> 4;
  const int part = blockIdx.x * 4 + wave;
  const int tile0 = part * kWN;
  const int row0 = blockIdx.y * 16 * WM;
  int tl[kWN];
#pragma unroll
  for (int j = 0; j < kWN; ++j) tl[j] = min(tile0 + j, ntiles - 1);
  const int8_t* arow[WM];  // A tiles: one 1 KB tile per (16 rows, K step)
#pragma unroll
  for (int i = 0; i < WM; ++i)
    arow[i] = p.a + ((size_t)(min(row0 + 16 * i, p.W - 1) >> 4) * p.nsteps << 10) + 16 * lane;
  // the block's activation scales, staged once (rows past W read row W - 1):
  // per K step a lane then reads its 4 WM scales from LDS instead of memory
  for (int e = threadIdx.x; e < 16 * WM * p.nsteps; e += 256) {
    const int r = e / p.nsteps, s = e - r * p.nsteps;
    as_l[e] = p.as[(size_t)min(row0 + r, p.W - 1) * p.nsteps + s];
  }
  __syncthreads();
  v4f acc[WM][kWN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < kWN; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  // R K steps of the weight stream in flight per wave beside the A rows of two
  // (L2).  One step at a time reaches the stream's rate while many waves share a
  // SIMD (32 rows with the argmax reduce: 38.7 us, with 4 steps 47.8); the
  // 64-row block holds fewer and needs them: 64 rows 76.3 -> 64.6 us, of which
  // the reduce is 5 (launch_lmhead: where its waves take no more rounds for it).
  v4i Bq[R][kWN];
  auto load_b = [&](v4i (&B)[kWN], int s) {
    s = min(s, p.nsteps - 1);
#pragma unroll
    for (int j = 0; j < kWN; ++j)
      B[j] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p.w) +
                                        ((size_t)tl[j] * p.nsteps + s) * 64 + lane);
  };
  auto load_a = [&](v4i (&A)[WM], int s) {
    s = min(s, p.nsteps - 1);
#pragma unroll
    for (int i = 0; i < WM; ++i) A[i] = *reinterpret_cast<const v4i*>(arow[i] + 1024 * s);
  };
  auto mac = [&](const v4i (&A)[WM], const v4i (&B)[kWN], int s) {
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      float asr[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) asr[r] = as_l[(16 * i + 4 * lgrp + r) * p.nsteps + s];
#pragma unroll
      for (int j = 0; j < kWN; ++j) {
        const v4i T = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[i], B[j], (v4i){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf((float)T[r], asr[r], acc[i][j][r]);
      }
    }
  };
  if constexpr (R == 1) {
    for (int s = 0; s < p.nsteps; ++s) {
      v4i A[WM];
      load_a(A, s);
      load_b(Bq[0], s);
      mac(A, Bq[0], s);
    }
  } else {
    v4i Aq[2][WM];
    load_a(Aq[0], 0);
#pragma unroll
    for (int d = 0; d < R; ++d) load_b(Bq[d], d);
    for (int s0 = 0; s0 < p.nsteps; s0 += R) {
#pragma unroll
      for (int d = 0; d < R; ++d) {
        if (s0 + d >= p.nsteps) break;
        load_a(Aq[(d + 1) & 1], s0 + d + 1);
        mac(Aq[d & 1], Bq[d], s0 + d);
        load_b(Bq[d], s0 + d + R);
      }
    }
  }
  float wsv[kWN];
#pragma unroll
  for (int j = 0; j < kWN; ++j) wsv[j] = ifrd::h2f(p.ws[16 * tl[j] + lrow]);
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 16 * i + 4 * lgrp + r;
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < kWN; ++j) {
        const int col = 16 * (tile0 + j) + lrow;
        if (tile0 + j >= ntiles) continue;
        const float lg = acc[i][j][r] * wsv[j];
        if (p.logits && row < p.W) p.logits[(size_t)row * p.V + col] = lg;
        if (better(lg, col, bv, bi)) { bv = lg; bi = col; }
      }
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
      }
      if (lrow == 0 && row < p.W) {
        // row-major [row][part] (part count = 4 gridDim.x): the final
        // reduce reads each row's partials contiguously
        const size_t at = (size_t)row * (4 * gridDim.x) + part;
        p.pv[at] = bv;
        p.pi[at] = bi;
      }
    }
}

// Reduce the per-wave (value, index) partials of each row.  Bound by the
// latency of reading them: 1024 threads, four partials of each in flight (V =
// 151936, 4748 partials a row: lm_head and reduce of 8 rows 38.0 -> 33.4 us
// against 256 threads with one in flight).
__global__ __launch_bounds__(1024) void argmax_final_kernel(const float* pv, const int32_t* pi,
                                                            int nparts, int W, int32_t* best) {
  const int row = blockIdx.x, lane = threadIdx.x & 63;
  pv += (size_t)row * nparts;
  pi += (size_t)row * nparts;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int q0 = threadIdx.x; q0 < nparts; q0 += 4 * 1024) {
    float v[4];
    int i[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // past the end: this thread's first partial again
      const int q = q0 + 1024 * k < nparts ? q0 + 1024 * k : q0;
      v[k] = pv[q];
      i[k] = pi[q];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (better(v[k], i[k], bv, bi)) { bv = v[k]; bi = i[k]; }
  }
  auto wave_best = [&] {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
    }
  };
  __shared__ float sv[16];
  __shared__ int si[16];
  wave_best();
  if (lane == 0) {
    sv[threadIdx.x >> 6] = bv;
    si[threadIdx.x >> 6] = bi;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;  // (after the only barrier)
  bv = sv[lane & 15];
  bi = si[lane & 15];
  wave_best();
  // The reference starts from -1e30 with strict '>': a row whose logits are
  // all <= -1e30 reports -1.
  if (threadIdx.x == 0) best[row] = (bv > -1e30f) ? bi : -1;
}

template <int WM, int R>
hipError_t launch_wm(const LmP& p, int nparts, int nrb, hipStream_t st) {
  const size_t lds = (size_t)16 * WM * p.nsteps * sizeof(float);
  if (lds > 64 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL((lmhead_kernel<WM, R>), dim3(nparts / 4, nrb), dim3(256), lds, st, p);
  return hipGetLastError();
}

}  // namespace

int lmhead_nparts(int V) {
  const int ntiles = V / 16;
  const int waves = (ntiles + kWN - 1) / kWN;
  return ((waves + 3) / 4) * 4;
}

hipError_t launch_lmhead(LmHeadArgs& a, hipStream_t st) {
  if (a.W <= 0) return hipSuccess;
  if (a.V % 16 != 0 || a.H % 64 != 0 || !a.a || !a.as || !a.wcodes || !a.wscale || !a.part_val ||
      !a.part_idx || !a.best)
    return hipErrorInvalidValue;
  a.nparts = lmhead_nparts(a.V);
  LmP p{a.a, a.as, a.wcodes, a.wscale, a.logits, a.part_val, a.part_idx, a.W, a.V, a.H, a.H / 64};
  hipError_t e;
  // Four steps in flight take 164 VGPRs: three waves a SIMD, 3072 on the chip,
  // where one step holds four.  A round of three costs about 0.7 of one of
  // four (0.8 at 16 K steps and fewer), so the whole rounds decide (us with the
  // reduce, four steps / one: H 1024, V 32000, 192 rows' 3000 waves 37.8 / 40.9,
  // 256 rows' 4000 waves 60.5 / 48.0; V 151936, 64 rows 64.4 / 76.5, 256 rows 197 /
  // 188, and at H 2048 312 / 316).
  const int nrb = (a.W + 63) / 64;
  const long waves = (long)a.nparts * nrb, r3 = (waves + 3071) / 3072, r4 = (waves + 4095) / 4096;
  if (a.W <= 16) e = launch_wm<1, 1>(p, a.nparts, 1, st);
  else if (a.W <= 32) e = launch_wm<2, 1>(p, a.nparts, 1, st);
  else if (r3 * (p.nsteps > 16 ? 7 : 8) <= r4 * 10) e = launch_wm<4, 4>(p, a.nparts, nrb, st);
  else e = launch_wm<4, 1>(p, a.nparts, nrb, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(argmax_final_kernel, dim3(a.W), dim3(1024), 0, st, a.part_val, a.part_idx,
                     a.nparts, a.W, a.best);
  return hipGetLastError();
}

}  // namespace ifrk
