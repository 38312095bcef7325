// gemv_fused.hip -- vec_dot in one launch: every workgroup quantizes the f32 input itself.
//
// vec_dot_* (src/gemma.rs:66-95) takes the f32 input, so a call used to be a quantizer launch
// (2.2-2.7 us for 4-14 K elements) and a GEMV that waits for it.  Here a workgroup of eight waves
// issues its share of the input's loads, then its weight loads, and quantizes the input into LDS
// (the same per-block operations as the quantizer kernels, so the same bytes) while the weights are
// in flight; each lane then takes its activation slice from LDS and reduces its rows as
// gemv_kernel does (the same units per lane, the same sums: the same bits).
//
// What bounds it: the weight stream, and before it the round trip of the input, which every
// workgroup reads whole (16 KB at 4096 elements, from L2).  Eight waves share that read and fill the
// CU in twos: four waves read the input twice as often (4096 -> 12288 Q4_K_R 10.6 against 8.9 us),
// sixteen wait at one barrier (9.0; 4096 -> 4096 5.7 against 5.3), and so do twice the rows per wave
// (9.8).  Per call in a graph, quantizer + GEMV before and this kernel now: Q4_K_R 4096 -> 4096 5.8
// and 5.3 us, 4096 -> 12288 8.7 and 8.9, 2048 -> 8192 5.9 and 4.8; Q8_0 4096 -> 4096 7.3 and 6.4;
// Q4_0 4096 -> 11008 9.3 and 8.2.  Enqueued call by call, the second launch costs the host 3 us more.
#include "gemv.h"

#include "gemv_dot.h"
#include "quantize.h"
#include "runtime.h"

namespace jero {

constexpr int kFusedWaves = 8;
constexpr int kFusedThreads = kFusedWaves * kWave;
// Input groups of 256 elements that a wave quantizes at most: rows up to 8192 elements.
constexpr int kFusedGroups = 4;

// Input groups per wave of a row of `elems` elements.
__host__ __device__ constexpr int fused_groups(int elems) {
  return ((elems + 255) / 256 + kFusedWaves - 1) / kFusedWaves;
}

// LDS bytes of a quantized group: one Q8_K block, or eight ACT_Q8 blocks.
__host__ __device__ constexpr int group_bytes(int f) { return is_kquant(f) ? 292 : 288; }

template <int F, int LPR, int UPL, int R, bool NT>
__global__ void __launch_bounds__(kFusedThreads) gemv_fused_kernel(const uint8_t* __restrict__ w, int64_t rb, int U,
                                                                   int64_t N, const float* __restrict__ x, int n_in,
                                                                   float* __restrict__ y) {
  using Ut = Unit<F>;
  constexpr int G = kWave / LPR;
  // groups of a row of LPR * UPL units, shared by the waves
  constexpr int XG = fused_groups(LPR * UPL * Ut::kElems);
  static_assert(XG <= kFusedGroups, "row too long for the staged input");
  extern __shared__ __attribute__((aligned(16))) uint8_t s_act[];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int g = lane / LPR, c = lane % LPR;
  const int64_t row0 = (int64_t(blockIdx.x) * kFusedWaves + wv) * (G * R);

  // the input first: its loads retire before the weights'.  Groups past the row read its last
  // elements and are not stored (of a partial last group, the elements past the row count as 0).
  float4 xv[XG];
#pragma unroll
  for (int i = 0; i < XG; i++)
    xv[i] = *reinterpret_cast<const float4*>(x + min((wv + kFusedWaves * i) * 256 + 4 * lane, n_in - 4));

  typename Ut::W wt[R][UPL];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t row = min(row0 + r * G + g, N - 1);
#pragma unroll
    for (int t = 0; t < UPL; t++) load_unit<F, NT>(wt[r][t], w, rb, N, U, row, min(c + LPR * t, U - 1));
  }

#pragma unroll
  for (int i = 0; i < XG; i++) {
    const int grp = wv + kFusedWaves * i;
    if (grp * 256 < n_in) {
      const bool in = grp * 256 + 4 * lane < n_in;
      const float e[4] = {in ? xv[i].x : 0.f, in ? xv[i].y : 0.f, in ? xv[i].z : 0.f, in ? xv[i].w : 0.f};
      if constexpr (is_kquant(F)) q8k_block_wave(e, lane, s_act + grp * 292);
      else actq8_blocks_wave(e, lane, s_act + grp * 288);
    }
  }
  lds_barrier();  // the LDS writes only, not the weight loads
  if (row0 >= N) return;
  typename Ut::Act act[UPL];
#pragma unroll
  for (int t = 0; t < UPL; t++) Ut::load_act(act[t], s_act, min(c + LPR * t, U - 1));
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t row = row0 + r * G + g;
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < UPL; t++) {
      const float d = Ut::dot(wt[r][t], act[t], nullptr);
      acc += c + LPR * t < U ? d : 0.0f;
    }
    acc = group_sum_last<LPR>(acc);
    if (c == LPR - 1 && row < N) y[row] = acc;
  }
}

namespace {

template <int F, int LPR, int UPL>
bool fused_one(int R, const uint8_t* w, int64_t k, int64_t N, const float* x, float* y, hipStream_t s) {
  if constexpr (fused_groups(LPR * UPL * Unit<F>::kElems) > kFusedGroups) {
    return false;
  } else {
    const int64_t rows = int64_t(kWave / LPR) * kFusedWaves * R;
    const dim3 grid(unsigned((N + rows - 1) / rows)), block(kFusedThreads);
    const size_t shm = size_t((k + 255) / 256) * group_bytes(F);
    const int64_t rb = row_bytes(F, k);
    const int U = units_per_row(F, k);
    if (R == 2)
      hipLaunchKernelGGL((gemv_fused_kernel<F, LPR, UPL, 2, nt_capable(F)>), grid, block, shm, s, w, rb, U, N, x,
                         int(k), y);
    else
      hipLaunchKernelGGL((gemv_fused_kernel<F, LPR, UPL, 1, nt_capable(F)>), grid, block, shm, s, w, rb, U, N, x,
                         int(k), y);
    return true;
  }
}

template <int F>
bool fused_fmt(const uint8_t* w, int64_t k, int64_t N, const float* x, float* y, hipStream_t s) {
  // lanes per row and units per lane as in launch_fmt (gemv.hip): the same sums
  const int U = units_per_row(F, k);
  const int lpr = U > 32 ? 64 : U > 16 ? 32 : U > 4 ? 16 : 4;
  const int G = kWave / lpr;
  const int64_t groups = (N + G - 1) / G;
  const int64_t cus = device_info().cus;
  // Where the quantizer and the GEMV stay apart: long rows of few outputs, where a workgroup's
  // quantizing is not hidden by its weights (us apart and fused: Q6_K_R 8192 -> 2048 7.5 and 8.8,
  // Q4_K_R 8192 -> 4096 9.1 and 8.1, 12288 -> 4096 9.3 and 11.4), and outputs beyond 96 rows per
  // lane group and CU, which run four rows per wave and repeat the quantizing too often (Q4_K_R
  // 4096 -> 48000 23.2 and 23.3; 4096 -> 24000 of Q6_K_R 19.8 and 17.7).
  if (groups > cus * 96 || k > 8192 || (k > 4096 && N < 4096)) return false;
  const int R = groups >= cus * 8 && (k < 8192 || is_planar(F)) ? 2 : 1;
  switch (lpr) {
    case 4: return fused_one<F, 4, 1>(R, w, k, N, x, y, s);
    case 16: return fused_one<F, 16, 1>(R, w, k, N, x, y, s);
    case 32: return fused_one<F, 32, 1>(R, w, k, N, x, y, s);
  }
  switch ((U + 63) / 64) {
    case 1: return fused_one<F, 64, 1>(R, w, k, N, x, y, s);
    case 2: return fused_one<F, 64, 2>(R, w, k, N, x, y, s);
    case 3: return fused_one<F, 64, 3>(R, w, k, N, x, y, s);
    case 4: return fused_one<F, 64, 4>(R, w, k, N, x, y, s);
  }
  return false;
}

}  // namespace

bool launch_vec_dot_fused(int quant, const void* w, int64_t n_in, int64_t n_out, const float* x, float* y,
                          hipStream_t s) {
  const uint8_t* wb = static_cast<const uint8_t*>(w);
  switch (quant) {
    case JERO_Q4_K: return fused_fmt<JERO_Q4_K>(wb, n_in, n_out, x, y, s);
    case JERO_Q4_K_R: return fused_fmt<JERO_Q4_K_R>(wb, n_in, n_out, x, y, s);
    case JERO_Q6_K: return fused_fmt<JERO_Q6_K>(wb, n_in, n_out, x, y, s);
    case JERO_Q6_K_R: return fused_fmt<JERO_Q6_K_R>(wb, n_in, n_out, x, y, s);
    case JERO_Q8_0: return fused_fmt<JERO_Q8_0>(wb, n_in, n_out, x, y, s);
    case JERO_Q4_0: return fused_fmt<JERO_Q4_0>(wb, n_in, n_out, x, y, s);
  }
  return false;
}

}  // namespace jero
