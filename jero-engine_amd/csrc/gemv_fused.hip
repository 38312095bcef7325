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
// (9.8).  Per call in a graph, quantizer + GEMV and this kernel: Q4_K_R 4096 -> 4096 6.0 and 5.3 us,
// 4096 -> 12288 8.9 and 8.9, 2048 -> 8192 5.9 and 4.9; Q8_0 4096 -> 4096 7.1 and 6.1; Q4_0 4096 ->
// 11000 9.0 and 8.1.  Enqueued call by call, the second launch costs the host 3 us more, which at 4096
// -> 12288 is the whole gain.  The rule (fused_pays) goes by the graph's times, the device's own, but
// for calls so short that the host's launches bound them when they are enqueued one by one.
#include "gemv.h"

#include "gemv_dot.h"
#include "quantize.h"
#include "runtime.h"

namespace jero {

constexpr int kFusedWaves = 8;
constexpr int kFusedThreads = kFusedWaves * kWave;

// Longest row that a format runs fused (fused_pays): 8192 elements at most, which is four input groups
// of 256 elements per wave.
__host__ __device__ constexpr int fused_max_k(int f) {
  return f == JERO_Q6_K ? 4096 : f == JERO_Q6_K_R ? 5120 : f == JERO_Q4_K ? 7936 : 8192;
}

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
  if constexpr (LPR * (UPL - 1) * Unit<F>::kElems >= fused_max_k(F)) {
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

// Whether one launch is at most as long as the quantizer and the GEMV (us apart and fused, in a graph).
// Every workgroup quantizes the whole input, so it loses where that is not hidden by its weights: long
// rows of few outputs (Q6_K_R 8192 -> 2048 7.5 and 8.8, Q4_K_R 12288 -> 4096 9.3 and 11.4), and outputs
// beyond 96 rows per lane group and CU, where the GEMV runs four rows per wave (Q4_K_R 4096 -> 48000 23.2
// and 23.3).  And its 8-wave workgroups fill the chip in coarser rounds than the GEMV's of four waves:
// `tail`, a short last round (less than 65 % of the CUs), costs up to 10 % of long rows (Q4_K_R 4096 ->
// 10000 7.9 and 8.5, -> 11000 8.6 and 8.7, -> 12288 8.9 and 8.9; Q6_K_R 4096 -> 10000 9.8 and 10.3, -> 8192
// 8.9 and 8.9).  Up to 4096 -> 8192 that is the smaller loss: one launch is up to 9 % longer in a graph
// (Q4_K_R 4096 -> 4128 6.0 and 6.4, Q6_K_R 6.9 and 7.5) and a third shorter call by call (Q4_K_R 10.4 and
// 6.2 or, with the host's present two launches, 7.4).
template <int F>
bool fused_pays(int64_t k, int64_t N, bool tail) {
  if (k > fused_max_k(F) || (k > 4096 && N < 4096)) return false;
  if (k <= 4096 && N <= 8192) return true;
  switch (F) {
    // 3072 -> 20000 10.7 and 11.3, -> 14000 8.8 and 9.0; 5120 -> 10000 12.1 and 11.6, -> 14000 16.4 and
    // 14.4, -> 24576 20.4 and 21.4; 6144 -> 6000 10.1 and 9.8, -> 10000 12.3 and 13.0, -> 12288 16.2 and
    // 13.6, -> 14000 17.1 and 16.4; 8192 -> 6000 11.0 and 11.6, -> 12288 18.0 and 16.0
    case JERO_Q4_K_R:
      if (k <= 2048) return true;
      if (N >= 16384) return false;
      if (k <= 3072) return !tail || N <= 12288;
      if (k <= 4096 || k == 8192) return !tail;
      return k <= 5120 || !tail || N <= 8192 || N > 12288;
    // 5120 -> 6000 10.2 and 10.1, -> 12288 15.9 and 14.2; 6144 -> 6000 10.7 and 11.2, -> 10000 14.7 and
    // 15.0, -> 12288 17.3 and 15.7, -> 14000 19.1 and 18.7, -> 24576 27.1 and 27.4; 8192 -> 12288 19.7 and 19.7
    case JERO_Q4_K: return k <= 5120 || (N <= 16384 && (!tail || N > 12288));
    // 5120 -> 6000 9.9 and 10.6, -> 12288 16.0 and 15.0; 5632 -> 8192 11.9 and 12.3, -> 10000 13.7 and 15.6
    case JERO_Q6_K_R: return k <= 3072 || !tail;
    // 4096 -> 12288 16.0 and 13.1; 4352 -> 12288 16.4 and 21.8, 6144 -> 10000 16.1 and 24.3
    case JERO_Q6_K: return true;
    // 5120 -> 4128 6.9 and 6.8; 7168 -> 4128 8.1 and 8.6, -> 6000 10.0 and 9.4, -> 14000 16.5 and 15.8; 8192
    // -> 8192 12.1 and 11.5, -> 14000 16.5 and 17.5
    case JERO_Q4_0: return k <= 7168 || N <= 8192;
    // 4096 -> 4128 7.8 and 7.4, 8192 -> 10000 19.8 and 17.8
    default: return true;
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
  if (groups > cus * 96) return false;
  const int R = groups >= cus * 8 && (k < 8192 || is_planar(F)) ? 2 : 1;
  const int64_t wgs = (groups + kFusedWaves * R - 1) / (kFusedWaves * R), last = wgs % cus;
  if (!fused_pays<F>(k, N, wgs > cus && last && 100 * last < 65 * cus)) return false;
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
