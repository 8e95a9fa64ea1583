// The SPLADE training loss on the head's output, on gfx950 (reference training/train.py:73-88,
// combined at :164-197). For query reps Q [Bq,V] and document reps R [Bd,V] (row-major, the
// head's reps dtype):
//   S      = Q R^T / T                                   in-batch scores
//   CE     = mean_i ( logsumexp_j S[i,j] - S[i,i] )       InfoNCE with labels arange(Bq) (:73-77)
//   L1(X)  = mean_b sum_v |X[b,v]|                        (:80-82)
//   FL(X)  = mean_v ( sum_b X[b,v] )^2                    (:85-87)
//   total  = w_ce CE + w_l1 (L1(Q) + L1(R)) + w_fl (FL(Q) + FL(R))    (:196-197)
// R may be absent (Bd = 0): then CE, L1(R) and FL(R) are 0.
//
// Forward, three launches:
//   loss_partial_kernel   one workgroup per 64-column vocabulary slice: stages the slice of Q
//                         and R as fp32 in LDS and writes the slice's partial S (4x4 or 2x2
//                         register tiles), each row's partial sum |X| and the slice's
//                         sum_v (sum_b X)^2;
//   loss_slice_sum_kernel those partials summed over the slices in a fixed order;
//   loss_final_kernel     one workgroup: the rows' softmax, CE, the means, total, and
//                         P = (softmax(S) - I) / (Bq T), which the backward uses.
// Backward, one launch (loss_bwd_kernel, one workgroup per slice), with the upstream
// gradients g[0..5] of (total, CE, L1(Q), L1(R), FL(Q), FL(R)) read from device memory:
//   dQ = (g0 w_ce + g1) P R + (g0 w_l1 + g2) sign(Q) / Bq + (g0 w_fl + g4) 2 colsum(Q) / V
//   dR = (g0 w_ce + g1) P^T Q + (g0 w_l1 + g3) sign(R) / Bd + (g0 w_fl + g5) 2 colsum(R) / V
// Everything accumulates in fp32 in a fixed order, so results are bitwise reproducible.
// The whole loss moves each of Q and R once forward and once backward: HBM-bound, small.

#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "sparton_common.h"

namespace sparton {
namespace loss {

constexpr int SLICE = 64;            // vocabulary columns per workgroup, one per lane
constexpr int NWAVES = 4;
constexpr int NT = 64 * NWAVES;
constexpr int MAX_B = 64;            // rows of Q and of R (past it the GEMM kernels are faster)
constexpr int LD = SLICE + 4;        // LDS row stride (floats) of a staged slice
constexpr int SUM_WAVES = 16;        // slice reduction: 64 entries x 16 waves per workgroup

__host__ __device__ constexpr int round4(int x) { return (x + 3) & ~3; }

// Rows [0, Bq) of Q then [0, Bd) of R, columns [c0, c0 + 64), as fp32 into sq / sd, zeros past
// V and in the padding rows up to a multiple of 4. Wave w stages rows w, w + 4, ...; lane l
// column c0 + l (one 128-byte segment per row for 16-bit types). All of a wave's loads are
// issued before the first is used, so they share one round trip: every lane loads from a
// clamped, valid address and the values of padding rows and columns past V are replaced by
// zeros afterwards (a load under a per-lane condition is waited for before the next one is
// issued). Bq >= 1, and R is read only when Bd > 0. Then row_fn(isq, row, x) runs for every
// real row with the lane's value (wave-uniform control flow).
template <typename T, int MB, typename F>
__device__ __forceinline__ void stage_slice(const T* __restrict__ Q, const T* __restrict__ R, int Bq,
                                            int Bd, int V, int c0, float* sq, float* sd, F row_fn) {
  constexpr int RPW = 2 * MB / NWAVES;  // rows per wave at most (Q and R padded to MB each)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = c0 + lane;
  const int cl = min(c, V - 1);
  const int Bqp = round4(Bq), Bdp = round4(Bd);
  T raw[RPW];
#pragma unroll
  for (int k = 0; k < RPW; ++k) {
    const int r = wave + k * NWAVES;
    const bool isq = r < Bqp || Bd == 0;
    const int row = isq ? min(r, Bq - 1) : min(r - Bqp, Bd - 1);
    raw[k] = (isq ? Q : R)[(size_t)row * V + cl];
  }
#pragma unroll
  for (int k = 0; k < RPW; ++k) {
    const int r = wave + k * NWAVES;
    if (r >= Bqp + Bdp) break;
    const bool isq = r < Bqp;
    const int row = isq ? r : r - Bqp;
    if (!(row < (isq ? Bq : Bd) && c < V)) raw[k] = T(0.0f);
    const float x = to_f32(raw[k]);
    (isq ? sq : sd)[row * LD + lane] = x;
    if (row < (isq ? Bq : Bd)) row_fn(isq, row, x);
  }
}

// Partials of one slice, at part + slice * K:
//   [0, Bq Bd)                     S without the 1/T (only when Bd > 0)
//   [o, o + Bq), [o + Bq, o + Bq + Bd)   sum over the slice of |Q[i,:]|, |R[j,:]|
//   o + Bq + Bd, o + Bq + Bd + 1   sum over the slice of colsum(Q)^2, colsum(R)^2
template <typename T, int MB, int TM>
__global__ __launch_bounds__(NT) void loss_partial_kernel(const T* __restrict__ Q,
                                                          const T* __restrict__ R, int Bq, int Bd,
                                                          int V, float* __restrict__ part, int K) {
  __shared__ __attribute__((aligned(16))) float sq[MB * LD];
  __shared__ __attribute__((aligned(16))) float sd[MB * LD];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float* out = part + (size_t)blockIdx.x * K;
  const int o = Bq * Bd;
  stage_slice<T, MB>(Q, R, Bq, Bd, V, blockIdx.x * SLICE, sq, sd, [&](bool isq, int row, float x) {
    const float s = wave_sum(fabsf(x));
    if (lane == 0) out[o + (isq ? 0 : Bq) + row] = s;
  });
  __syncthreads();
  if (wave < 2) {  // wave 0: Q's column sums, wave 1: R's
    const float* s = wave == 0 ? sq : sd;
    const int nrows = wave == 0 ? Bq : Bd;
    float cs = 0.0f;
    for (int r = 0; r < nrows; ++r) cs += s[r * LD + lane];
    const float t = wave_sum(cs * cs);
    if (lane == 0) out[o + Bq + Bd + wave] = t;
  }
  if (Bd == 0) return;
  // S tiles of TM x TM (TM = 2 when 4 x 4 tiles would leave threads idle)
  const int nbi = round4(Bq) / TM, nbj = round4(Bd) / TM;
  for (int blk = threadIdx.x; blk < nbi * nbj; blk += NT) {
    const int i0 = (blk / nbj) * TM, j0 = (blk % nbj) * TM;
    float acc[TM][TM];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b) acc[a][b] = 0.0f;
#pragma unroll 4
    for (int cc = 0; cc < SLICE; cc += 4) {
      f32x4 qa[TM], rb[TM];
#pragma unroll
      for (int k = 0; k < TM; ++k) {
        qa[k] = *(const f32x4*)(sq + (i0 + k) * LD + cc);
        rb[k] = *(const f32x4*)(sd + (j0 + k) * LD + cc);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int b = 0; b < TM; ++b) acc[a][b] = fmaf(qa[a][e], rb[b][e], acc[a][b]);
    }
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b)
        if (i0 + a < Bq && j0 + b < Bd) out[(i0 + a) * Bd + j0 + b] = acc[a][b];
  }
}

// sums[k] = sum over slices of part[slice][k]. Workgroup g owns entries [64 g, 64 g + 64), one
// per lane; wave w sums slices [w S, (w + 1) S) in order (S = ceil(nslice / 16)), eight loads
// in flight, and wave 0 adds the 16 wave sums in wave order.
__global__ __launch_bounds__(64 * SUM_WAVES) void loss_slice_sum_kernel(const float* __restrict__ part,
                                                                       int nslice, int K,
                                                                       float* __restrict__ sums) {
  __shared__ float wsum[SUM_WAVES][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int k = blockIdx.x * 64 + lane;
  const int seg = (nslice + SUM_WAVES - 1) / SUM_WAVES;
  const int beg = min(nslice, wave * seg), end = min(nslice, beg + seg);
  float acc = 0.0f;
  if (k < K) {
    for (int s0 = beg; s0 < end; s0 += 8) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = part[(size_t)min(s0 + j, end - 1) * K + k];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc += s0 + j < end ? v[j] : 0.0f;
    }
  }
  wsum[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && k < K) {
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < SUM_WAVES; ++w) t += wsum[w][lane];
    sums[k] = t;
  }
}

// One workgroup. Wave w takes score rows w, w + 4, ...; lane l holds columns l and l + 64.
// out = (total, CE, L1(Q), L1(R), FL(Q), FL(R)); probs[i][j] = (softmax_j(S[i,:]) - [i == j]) / (Bq T).
__global__ __launch_bounds__(NT) void loss_final_kernel(const float* __restrict__ sums, int Bq, int Bd,
                                                        int V, float inv_t, float w_ce, float w_l1,
                                                        float w_fl, float* __restrict__ out,
                                                        float* __restrict__ probs) {
  __shared__ float row_loss[MAX_B];
  __shared__ float tail[2 * MAX_B + 2];  // the row sums of |x| and the two FLOPS sums
  __shared__ float ss[MAX_B * MAX_B];     // S without the 1/T
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int o = Bq * Bd, n = o + Bq + Bd + 2;
  for (int k0 = 0; k0 < n; k0 += 8 * NT) {  // every load of a round issued before any store
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[u] = sums[min(k0 + u * NT + (int)threadIdx.x, n - 1)];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = k0 + u * NT + threadIdx.x;
      if (k < o) ss[k] = v[u];
      else if (k < n) tail[k - o] = v[u];
    }
  }
  __syncthreads();
  if (Bd > 0) {
    const float pscale = inv_t / (float)Bq;
    for (int i = wave; i < Bq; i += NWAVES) {
      const float* srow = ss + i * Bd;
      const bool h0 = lane < Bd, h1 = lane + 64 < Bd;
      const float x0 = h0 ? srow[lane] * inv_t : -INFINITY;
      const float x1 = h1 ? srow[lane + 64] * inv_t : -INFINITY;
      const float m = wave_max(fmaxf(x0, x1));
      const float e0 = h0 ? expf(x0 - m) : 0.0f, e1 = h1 ? expf(x1 - m) : 0.0f;
      const float s = wave_sum(e0 + e1);
      if (lane == 0) row_loss[i] = m + logf(s) - srow[i] * inv_t;
      const float rs = 1.0f / s;
      if (h0) probs[(size_t)i * Bd + lane] = (e0 * rs - (lane == i ? 1.0f : 0.0f)) * pscale;
      if (h1) probs[(size_t)i * Bd + lane + 64] = (e1 * rs - (lane + 64 == i ? 1.0f : 0.0f)) * pscale;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float ce = 0.0f, l1q = 0.0f, l1d = 0.0f;
    for (int i = 0; i < (Bd > 0 ? Bq : 0); ++i) ce += row_loss[i];
    for (int i = 0; i < Bq; ++i) l1q += tail[i];
    for (int j = 0; j < Bd; ++j) l1d += tail[Bq + j];
    ce = Bd > 0 ? ce / (float)Bq : 0.0f;
    l1q /= (float)Bq;
    l1d = Bd > 0 ? l1d / (float)Bd : 0.0f;
    const float flq = tail[Bq + Bd] / (float)V, fld = tail[Bq + Bd + 1] / (float)V;
    out[0] = w_ce * ce + w_l1 * (l1q + l1d) + w_fl * (flq + fld);
    out[1] = ce;
    out[2] = l1q;
    out[3] = l1d;
    out[4] = flq;
    out[5] = fld;
  }
}

// The upstream gradients of the six outputs: each a device fp32 scalar, or NULL for 0.
struct Grads6 {
  const float* p[6];
};
__device__ __forceinline__ float grad_of(const Grads6& g, int k) {
  return g.p[k] != nullptr ? *g.p[k] : 0.0f;
}

// One workgroup per slice: stages Q, R and P, the slice's column sums, then 4x4 tiles of
// dQ (rows i0..i0+3 x 4 columns) and dR (rows j0..j0+3 x 4 columns), each thread a tile.
template <typename T, int MB>
__global__ __launch_bounds__(NT) void loss_bwd_kernel(const T* __restrict__ Q, const T* __restrict__ R,
                                                      const float* __restrict__ P,
                                                      const Grads6 g, int Bq, int Bd,
                                                      int V, float w_ce, float w_l1, float w_fl,
                                                      T* __restrict__ GQ, T* __restrict__ GR) {
  constexpr int PLD = MB + 4;
  __shared__ __attribute__((aligned(16))) float sq[MB * LD];
  __shared__ __attribute__((aligned(16))) float sd[MB * LD];
  __shared__ __attribute__((aligned(16))) float sp[MB * PLD];
  __shared__ float colsum[2][SLICE];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c0 = blockIdx.x * SLICE;
  const int Bqp = round4(Bq), Bdp = round4(Bd);
  // P, zero-padded to Bqp x Bdp: its loads are issued first, so that they are in flight
  // together with the slice's (clamped addresses, padding zeroed afterwards; P exists only
  // when Bd > 0)
  constexpr int PPT = MB * MB / NT;  // P entries per thread at most
  float pr[PPT];
  if (Bdp > 0) {
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
      const int e = u * NT + threadIdx.x;
      const int i = e / Bdp, j = e - i * Bdp;
      pr[u] = P[(size_t)min(i, Bq - 1) * Bd + min(j, Bd - 1)];
    }
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
      const int e = u * NT + threadIdx.x;
      const int i = e / Bdp, j = e - i * Bdp;
      if (!(e < Bqp * Bdp && i < Bq && j < Bd)) pr[u] = 0.0f;
    }
  }
  stage_slice<T, MB>(Q, R, Bq, Bd, V, c0, sq, sd, [](bool, int, float) {});
#pragma unroll
  for (int u = 0; u < PPT; ++u) {
    const int e = u * NT + threadIdx.x;
    if (Bdp > 0 && e < Bqp * Bdp) sp[(e / Bdp) * PLD + e % Bdp] = pr[u];
  }
  __syncthreads();
  if (wave < 2) {
    const float* s = wave == 0 ? sq : sd;
    const int nrows = wave == 0 ? Bq : Bd;
    float cs = 0.0f;
    for (int r = 0; r < nrows; ++r) cs += s[r * LD + lane];
    colsum[wave][lane] = cs;
  }
  __syncthreads();
  const float g0 = grad_of(g, 0);
  const float c_ce = g0 * w_ce + grad_of(g, 1);
  const float c_sq = (g0 * w_l1 + grad_of(g, 2)) / (float)Bq;
  const float c_sd = Bd > 0 ? (g0 * w_l1 + grad_of(g, 3)) / (float)Bd : 0.0f;
  const float c_fq = 2.0f * (g0 * w_fl + grad_of(g, 4)) / (float)V;
  const float c_fd = 2.0f * (g0 * w_fl + grad_of(g, 5)) / (float)V;
  const int nbi = Bqp / 4, nbj = Bdp / 4;
  constexpr int CT = SLICE / 4;  // column tiles per slice
  for (int t = threadIdx.x; t < (nbi + nbj) * CT; t += NT) {
    const bool isq = t < nbi * CT;
    const int tt = isq ? t : t - nbi * CT;
    const int r0 = (tt / CT) * 4, cc = (tt % CT) * 4;
    float acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = 0.0f;
    if (isq) {  // sum_j P[i][j] R[j][c]
      for (int j = 0; j < Bd; ++j) {
        const f32x4 rv = *(const f32x4*)(sd + j * LD + cc);
        float p[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) p[a] = sp[(r0 + a) * PLD + j];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int b = 0; b < 4; ++b) acc[a][b] = fmaf(p[a], rv[b], acc[a][b]);
      }
    } else {  // sum_i P[i][j] Q[i][c]
      for (int i = 0; i < Bq; ++i) {
        const f32x4 qv = *(const f32x4*)(sq + i * LD + cc);
        const f32x4 p = *(const f32x4*)(sp + i * PLD + r0);
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int b = 0; b < 4; ++b) acc[a][b] = fmaf(p[a], qv[b], acc[a][b]);
      }
    }
    const float* own = isq ? sq : sd;
    const float* cs = colsum[isq ? 0 : 1];
    const float c_s = isq ? c_sq : c_sd, c_f = isq ? c_fq : c_fd;
    const int nrows = isq ? Bq : Bd;
    T* G = isq ? GQ : GR;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int row = r0 + a;
      if (row >= nrows) continue;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int c = c0 + cc + b;
        if (c >= V) continue;
        const float x = own[row * LD + cc + b];
        const float sg = x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f);
        G[(size_t)row * V + c] = from_f32<T>(c_ce * acc[a][b] + c_s * sg + c_f * cs[cc + b]);
      }
    }
  }
}

static int64_t slices(int64_t V) { return cdiv(V, (int64_t)SLICE); }
static int64_t entries(int64_t Bq, int64_t Bd) { return Bq * Bd + Bq + Bd + 2; }

template <typename T, int MB>
static void launch_fwd(const void* q, const void* d, int Bq, int Bd, int V, float* part, int K,
                       hipStream_t st) {
  const dim3 grid((unsigned)slices(V));
  if ((round4(Bq) / 4) * (round4(Bd) / 4) >= NT)
    hipLaunchKernelGGL((loss_partial_kernel<T, MB, 4>), grid, dim3(NT), 0, st, (const T*)q,
                       (const T*)d, Bq, Bd, V, part, K);
  else
    hipLaunchKernelGGL((loss_partial_kernel<T, MB, 2>), grid, dim3(NT), 0, st, (const T*)q,
                       (const T*)d, Bq, Bd, V, part, K);
}
template <typename T, int MB>
static void launch_bwd(const void* q, const void* d, const float* P, const Grads6& g, int Bq, int Bd,
                       int V, float w_ce, float w_l1, float w_fl, void* gq, void* gd, hipStream_t st) {
  hipLaunchKernelGGL((loss_bwd_kernel<T, MB>), dim3((unsigned)slices(V)), dim3(NT), 0, st,
                     (const T*)q, (const T*)d, P, g, Bq, Bd, V, w_ce, w_l1, w_fl, (T*)gq, (T*)gd);
}

template <typename T>
static void fwd_partial(const void* q, const void* d, int Bq, int Bd, int V, float* part, int K,
                        hipStream_t st) {
  const int mb = Bq > Bd ? Bq : Bd;
  if (mb <= 32) launch_fwd<T, 32>(q, d, Bq, Bd, V, part, K, st);
  else launch_fwd<T, MAX_B>(q, d, Bq, Bd, V, part, K, st);
}
template <typename T>
static void bwd_all(const void* q, const void* d, const float* P, const Grads6& g, int Bq, int Bd,
                    int V, float w_ce, float w_l1, float w_fl, void* gq, void* gd, hipStream_t st) {
  const int mb = Bq > Bd ? Bq : Bd;
  if (mb <= 32) launch_bwd<T, 32>(q, d, P, g, Bq, Bd, V, w_ce, w_l1, w_fl, gq, gd, st);
  else launch_bwd<T, MAX_B>(q, d, P, g, Bq, Bd, V, w_ce, w_l1, w_fl, gq, gd, st);
}

// ---- batches past MAX_B rows ---------------------------------------------------------------
//
// The kernels above stage every row of a 64-column slice and keep per-slice partials of all
// Bq x Bd scores; their per-thread work grows with the rows, and past 64 rows a side the
// kernels below are faster (V 30522, fwd+bwd device time: 96 rows 134 us against 81 us, 128
// rows 190 against 90; 64 rows 62 against 70). Larger batches take GEMM-shaped kernels; the
// score and gradient kernels further down run on the 16-bit matrix cores, those here on the fp32
// ones (v_mfma_f32_32x32x2f32: the products of any reps dtype are exact in fp32, and the sums
// accumulate in fp32, as above), which tests compare them with and which the tiles of fp32 and
// fp16 reps with an entry that is not finite take:
//   forward   loss_stats_kernel   per 128-column slice: each row's sum of |x| over the slice,
//                                 and sum_v (sum_b x)^2 of Q and of R;
//             loss_score_kernel   S = Q R^T in 128 x 128 tiles, the vocabulary split into
//                                 chunks (one partial S per chunk);
//             loss_slice_sum_kernel (above) sums both sets of partials in a fixed order;
//             loss_rows_kernel    one wave per query row: softmax, the row's CE term, P;
//             loss_final_large_kernel the six scalars.
//   backward  loss_bwd_large_kernel, one workgroup per 64 vocabulary columns: the columns'
//             sums over Q and R, then dQ = c P R + ... tile by tile over 128 query rows and
//             dR = c P^T Q + ... over 128 document rows, K (the other side's rows) streamed
//             through LDS in stages of 32. No workspace.
// Operand tiles sit in LDS as fp32 [k][m]; an MFMA takes A[m][k] from lane m + 32 k and B[k][n]
// from lane n + 32 k, so both reads are consecutive floats. The row strides 161 and 97 are
// 33 mod 64 banks, so the transposing stores and the two lane halves' reads barely conflict.
namespace big {
constexpr int TM = 128;   // score tile rows and columns; gradient rows per tile
constexpr int KS = 32;    // K per LDS stage
constexpr int LDA = 161;  // floats per k row of a [KS][128] tile
constexpr int NC = 64;    // backward: vocabulary columns per workgroup
constexpr int LDB = 97;   // floats per k row of a [KS][64] tile
constexpr int ST_ROWS = 32;  // stats: rows whose loads are in flight together per wave
constexpr int ST_COLS = 128;  // and columns per workgroup

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.0f;
  return z;
}

// K-contiguous source X[m][k] (row stride ld): rows [m0, m0 + 128), k in [k0, k0 + KS); zero past
// M rows or past kend. Thread t holds k = t % 32 of rows t / 32 + 8 u.
template <typename T>
__device__ __forceinline__ void load_kc(const T* __restrict__ X, int64_t ld, int m0, int M, int k0,
                                        int kend, T (&v)[16]) {
  const int t = threadIdx.x, k = k0 + (t & 31), rb = t >> 5;
  // every load from a clamped place, zeroed afterwards: a load under its own condition would be
  // waited for before the next
#pragma unroll
  for (int u = 0; u < 16; ++u) v[u] = X[(int64_t)min(m0 + rb + 8 * u, M - 1) * ld + min(k, kend - 1)];
#pragma unroll
  for (int u = 0; u < 16; ++u)
    if (!(m0 + rb + 8 * u < M && k < kend)) v[u] = T(0.0f);
}
template <typename T>
__device__ __forceinline__ void store_kc(float* s, const T (&v)[16]) {
  const int t = threadIdx.x, kk = t & 31, rb = t >> 5;
#pragma unroll
  for (int u = 0; u < 16; ++u) s[kk * LDA + rb + 8 * u] = to_f32(v[u]);
}

// N-contiguous source X[k][n] (row stride ld): k in [k0, k0 + KS) below kend, n in [n0, n0 + NN)
// below nend, into s[k][n] (row stride LD). Thread t holds n = t % NN of k rows t / NN + (NT/NN) u.
template <typename T, int NN>
__device__ __forceinline__ void load_nc(const T* __restrict__ X, int64_t ld, int k0, int kend, int n0,
                                        int nend, T (&v)[KS * NN / NT]) {
  constexpr int KSTEP = NT / NN;
  const int t = threadIdx.x, n = n0 + t % NN, kb = t / NN;
#pragma unroll
  for (int u = 0; u < KS / KSTEP; ++u)
    v[u] = X[(int64_t)min(k0 + kb + KSTEP * u, kend - 1) * ld + min(n, nend - 1)];
#pragma unroll
  for (int u = 0; u < KS / KSTEP; ++u)
    if (!(k0 + kb + KSTEP * u < kend && n < nend)) v[u] = T(0.0f);
}
template <typename T, int NN, int LD>
__device__ __forceinline__ void store_nc(float* s, const T (&v)[KS * NN / NT]) {
  constexpr int KSTEP = NT / NN;
  const int t = threadIdx.x, n = t % NN, kb = t / NN;
#pragma unroll
  for (int u = 0; u < KS / KSTEP; ++u) s[(kb + KSTEP * u) * LD + n] = to_f32(v[u]);
}

// acc[bi][bj] += A[am0 + 32 bi .., :] B[:, bn0 + 32 bj ..] over one stage (KS values of k).
template <int BI, int BJ, int LDa, int LDb>
__device__ __forceinline__ void mma_stage(const float* sA, int am0, const float* sB, int bn0,
                                          f32x16 (&acc)[BI][BJ]) {
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
#pragma unroll 4
  for (int ks = 0; ks < KS / 2; ++ks) {
    const int k = 2 * ks + h;
    float a[BI], b[BJ];
#pragma unroll
    for (int i = 0; i < BI; ++i) a[i] = sA[k * LDa + am0 + 32 * i + l32];
#pragma unroll
    for (int j = 0; j < BJ; ++j) b[j] = sB[k * LDb + bn0 + 32 * j + l32];
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
  }
}

// Row of accumulator register r of a 32 x 32 block held by lane half h (the lane holds column
// lane % 32).
__device__ __forceinline__ int acc_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// acc += Q R^T over columns [kc0, kc1) for the 128 x 128 tile at (i0, j0), in [KS][LDA] tiles.
template <typename T>
__device__ __forceinline__ void score_tile(float* sA, float* sB, const T* __restrict__ Q,
                                           const T* __restrict__ R, int Bq, int Bd, int V, int i0, int j0,
                                           int kc0, int kc1, f32x16 (&acc)[2][2]) {
  const int wave = threadIdx.x >> 6, wm = wave >> 1, wn = wave & 1;
  T ra[16], rb[16];
  load_kc(Q, V, i0, Bq, kc0, kc1, ra);
  load_kc(R, V, j0, Bd, kc0, kc1, rb);
  for (int k0 = kc0; k0 < kc1; k0 += KS) {
    __syncthreads();  // the previous stage is read
    store_kc(sA, ra);
    store_kc(sB, rb);
    __syncthreads();
    if (k0 + KS < kc1) {  // the next stage's loads run under this stage's MFMAs
      load_kc(Q, V, i0, Bq, k0 + KS, kc1, ra);
      load_kc(R, V, j0, Bd, k0 + KS, kc1, rb);
    }
    mma_stage<2, 2, LDA, LDA>(sA, wm * 64, sB, wn * 64, acc);
  }
}

// Partial S = Q R^T over the vocabulary chunk blockIdx.y (columns [chunk y, chunk (y+1))) for
// the 128 x 128 tile blockIdx.x, at part + y Bq Bd. Four waves of 64 x 64 (2 x 2 blocks).
template <typename T>
__global__ __launch_bounds__(NT) void loss_score_kernel(const T* __restrict__ Q, const T* __restrict__ R,
                                                        int Bq, int Bd, int V, int chunk,
                                                        float* __restrict__ part) {
  __shared__ float sA[KS * LDA];
  __shared__ float sB[KS * LDA];
  const int tj = (Bd + TM - 1) / TM;
  const int i0 = (blockIdx.x / tj) * TM, j0 = (blockIdx.x % tj) * TM;
  const int kc0 = blockIdx.y * chunk, kc1 = min(V, kc0 + chunk);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, wm = wave >> 1, wn = wave & 1;
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero16();
  score_tile(sA, sB, Q, R, Bq, Bd, V, i0, j0, kc0, kc1, acc);
  float* out = part + (size_t)blockIdx.y * Bq * Bd;
  const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj) {
      const int j = j0 + wn * 64 + 32 * bj + l32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = i0 + wm * 64 + 32 * bi + acc_row(r, h);
        if (i < Bq && j < Bd) out[(size_t)i * Bd + j] = acc[bi][bj][r];
      }
    }
}

typedef __attribute__((ext_vector_type(2))) float f32x2;
template <typename T> using Two = T __attribute__((ext_vector_type(2)));

// N rows r0, r0 + step, .. (r0 uniform) of X at columns c, c + 1 (c even), two to a load where rows
// and columns allow it (pair: V even, X aligned to two elements). Rows past K read zero; columns
// past V whatever is there (nothing of theirs is stored).
template <typename T, int N>
__device__ __forceinline__ void load_x(const T* __restrict__ X, bool pair, int K, int r0, int step, int c,
                                       int V, Two<T> (&v)[N]) {
  if (pair) {  // uniform
    const uint32_t cc = (uint32_t)min(c, V - 2);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const T* row = X + (int64_t)min(r0 + step * i, K - 1) * V;
      v[i] = *(const Two<T>*)(row + cc);
    }
  } else {
    const uint32_t ca = (uint32_t)min(c, V - 1), cb = (uint32_t)min(c + 1, V - 1);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const T* row = X + (int64_t)min(r0 + step * i, K - 1) * V;
      v[i] = Two<T>{row[ca], row[cb]};
    }
  }
  if (r0 + step * (N - 1) >= K)
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (r0 + step * i >= K) v[i] = Two<T>{T(0.0f), T(0.0f)};
}
// Side blockIdx.y (Q, R) of the 128-column slice blockIdx.x, at part + slice K: entries [0, Bq) and
// [Bq, Bq + Bd) the rows' sums of |x| over the slice, Bq + Bd and Bq + Bd + 1 the slice's
// sum_v (sum_b x)^2 of Q and of R. Wave w takes rows w, w + 4, ..., two columns a lane; column sums
// are added over the waves in order. Bound by the loads' latency: a workgroup for each side, and
// ST_ROWS rows' loads in flight (256 x 512 x 30522 fp16: 28 -> 20 us).
template <typename T>
__global__ __launch_bounds__(NT) void loss_stats_kernel(const T* __restrict__ Q, const T* __restrict__ R,
                                                        bool pair, int Bq, int Bd, int V,
                                                        float* __restrict__ part, int K) {
  __shared__ f32x2 cpart[4][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = blockIdx.x * ST_COLS + 2 * lane, side = blockIdx.y;
  const T* X = side ? R : Q;
  const int rows = side ? Bd : Bq, o = side ? Bq : 0;
  float* out = part + (size_t)blockIdx.x * K;
  f32x2 cs = {0.0f, 0.0f};
  for (int b0 = wave; b0 < rows; b0 += 4 * ST_ROWS) {
    Two<T> v[ST_ROWS];
    load_x<T>(X, pair, rows, b0, 4, c, V, v);
#pragma unroll
    for (int u = 0; u < ST_ROWS; ++u) {
      const int b = b0 + 4 * u;
      if (b < rows) {  // uniform
        const float x0 = c < V ? to_f32((T)v[u][0]) : 0.0f, x1 = c + 1 < V ? to_f32((T)v[u][1]) : 0.0f;
        cs[0] += x0;
        cs[1] += x1;
        const float a = wave_sum(fabsf(x0) + fabsf(x1));
        if (lane == 0) out[o + b] = a;
      }
    }
  }
  cpart[wave][lane] = cs;
  __syncthreads();
  if (wave == 0) {
    const f32x2 tot = ((cpart[0][lane] + cpart[1][lane]) + cpart[2][lane]) + cpart[3][lane];
    const float sq = wave_sum(tot[0] * tot[0] + tot[1] * tot[1]);
    if (lane == 0) out[Bq + Bd + side] = sq;
  }
}

// One wave per query row i: x = S[i, :] / T, the row's CE term logsumexp(x) - x[i] and
// P[i, j] = (softmax(x)_j - [i == j]) / (Bq T).
__global__ __launch_bounds__(NT) void loss_rows_kernel(const float* __restrict__ S, int Bq, int Bd,
                                                       float inv_t, float* __restrict__ row_loss,
                                                       float* __restrict__ probs) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + wave;
  if (i >= Bq) return;
  const float* srow = S + (size_t)i * Bd;
  float m = -INFINITY;
  for (int j = lane; j < Bd; j += 64) m = fmaxf(m, srow[j] * inv_t);
  m = wave_max(m);
  float s = 0.0f;
  for (int j = lane; j < Bd; j += 64) s += expf(srow[j] * inv_t - m);
  s = wave_sum(s);
  if (lane == 0) row_loss[i] = m + logf(s) - srow[i] * inv_t;
  const float rs = 1.0f / s, pscale = inv_t / (float)Bq;
  for (int j = lane; j < Bd; j += 64)
    probs[(size_t)i * Bd + j] = (expf(srow[j] * inv_t - m) * rs - (j == i ? 1.0f : 0.0f)) * pscale;
}

// One wave: the six scalars from the row CE terms and the summed statistics.
__global__ __launch_bounds__(64) void loss_final_large_kernel(const float* __restrict__ row_loss,
                                                              const float* __restrict__ stats, int Bq,
                                                              int Bd, int V, float w_ce, float w_l1,
                                                              float w_fl, float* __restrict__ out) {
  const int lane = threadIdx.x;
  float ce = 0.0f, l1q = 0.0f, l1d = 0.0f;
  if (Bd > 0)
    for (int i = lane; i < Bq; i += 64) ce += row_loss[i];
  for (int i = lane; i < Bq; i += 64) l1q += stats[i];
  for (int j = lane; j < Bd; j += 64) l1d += stats[Bq + j];
  ce = wave_sum(ce);
  l1q = wave_sum(l1q);
  l1d = wave_sum(l1d);
  if (lane == 0) {
    ce = Bd > 0 ? ce / (float)Bq : 0.0f;
    l1q /= (float)Bq;
    l1d = Bd > 0 ? l1d / (float)Bd : 0.0f;
    const float flq = stats[Bq + Bd] / (float)V, fld = stats[Bq + Bd + 1] / (float)V;
    out[0] = w_ce * ce + w_l1 * (l1q + l1d) + w_fl * (flq + fld);
    out[1] = ce;
    out[2] = l1q;
    out[3] = l1d;
    out[4] = flq;
    out[5] = fld;
  }
}

// 128 rows of one gradient over the workgroup's 64 columns: acc = sum_k A[m][k] B[k][n] with A
// from a K-contiguous (P rows, dQ) or N-contiguous (P columns, dR) source; wave w owns rows
// 32 w .. 32 w + 31 (two 32 x 32 blocks). Then G = c_ce acc + c_s sign(X) + c_f colsum, in T.
template <typename T, bool A_KC>
__device__ __forceinline__ void grad_tile(float* sA, float* sB, const float* __restrict__ P,
                                          int Bq, int Bd, const T* __restrict__ Bsrc, int K,
                                          const T* __restrict__ X, int rows, int m0, int c0, int V,
                                          float c_ce, float c_s, float c_f, const float* colsum,
                                          T* __restrict__ G) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  f32x16 acc[1][2] = {{zero16(), zero16()}};
  if (K > 0) {
    float pa[16];
    T rbv[KS * NC / NT];
    auto load_a = [&](int k0) {
      if (A_KC) {  // A[m][k] = P[m0 + m][k]: rows of P (dQ)
        load_kc(P, Bd, m0, Bq, k0, K, pa);
      } else {     // A[m][k] = P[k][m0 + m]: columns of P (dR)
        load_nc<float, TM>(P, Bd, k0, K, m0, Bd, pa);
      }
    };
    load_a(0);
    load_nc<T, NC>(Bsrc, V, 0, K, c0, V, rbv);
    for (int k0 = 0; k0 < K; k0 += KS) {
      __syncthreads();
      if (A_KC) store_kc(sA, pa);
      else store_nc<float, TM, LDA>(sA, pa);
      store_nc<T, NC, LDB>(sB, rbv);
      __syncthreads();
      if (k0 + KS < K) {
        load_a(k0 + KS);
        load_nc<T, NC>(Bsrc, V, k0 + KS, K, c0, V, rbv);
      }
      mma_stage<1, 2, LDA, LDB>(sA, wave * 32, sB, 0, acc);
    }
  }
#pragma unroll
  for (int bj = 0; bj < 2; ++bj) {
    const int cl = 32 * bj + l32, c = c0 + cl;
    T xv[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = m0 + wave * 32 + acc_row(r, h);
      xv[r] = (i < rows && c < V) ? X[(int64_t)i * V + c] : T(0.0f);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = m0 + wave * 32 + acc_row(r, h);
      if (i < rows && c < V) {
        const float x = to_f32(xv[r]);
        const float sg = x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f);
        G[(int64_t)i * V + c] = from_f32<T>(c_ce * acc[0][bj][r] + c_s * sg + c_f * colsum[cl]);
      }
    }
  }
}

// ---- score and gradients on 16-bit MFMAs ----
//
// A product of two bf16 (or two fp16) values is exact in fp32, so for 16-bit reps the score
// GEMM runs on v_mfma_f32_32x32x16_{bf16,f16}: 8 times the k per instruction of the fp32
// MFMA, in the same 32 x 32 output layout. The stage's operands are kept in LDS as [row][k]
// 16-bit values, rows LDH apart: 80 bytes, so the 16 rows of one ds_read_b128 phase fall in
// distinct banks. A lane's MFMA operand (8 consecutive k of one row) is one 16-byte read.
// Other operands are taken as sums of bf16 parts, x = x0 + x1 + ... (each part rounds what
// the ones before it left to nearest even; the remainders are exact): three parts hold an
// fp32 value's 24 bits, two an fp16 value's 11, and bf16 has fp32's exponents, so no scales
// are needed. A product takes the pairs of parts down to 2^-24 of it:
//   scores     fp32 reps 3 x 3 parts, 6 MFMAs per step (against 8 fp32 ones of twice the time)
//   gradients  P (fp32) against bf16 reps 2 x 1 parts (p within 2^-17), 2 MFMAs; fp16 reps
//              3 x 2 parts, 5; fp32 reps 3 x 3, 6
// The products of the lower parts have accumulators of their own, added at the end: the main
// sums then round once per 16 k (the fp32 MFMA's: 8 times), and over batches of 65 to 500 rows
// and V 257 to 30522 the gradients' rms error against fp64 is that of the fp32 MFMAs or below
// (0.65 to 1.0 of it, also where it is all sums; with one set of accumulators it was twice that).
// Every load of a row goes two elements at a time: a row of V elements starts on any 2- or
// 4-byte boundary, and 16-byte loads off theirs took 1.6 times as long (256 x 512 x 30522 fp16
// score 42.6 us against 27.2).
// Forward and backward of 256 x 512 x 30522, before (fp32 MFMAs, bf16 reps on bf16 ones) -> now:
// fp16 398 -> 184 us, bf16 326 -> 154, fp32 436 -> 236; 512 x 1024 bf16 972 -> 400, fp32
// 1448 -> 710; 65 x 130 and 128 x 128, where the launches weigh most, 93-112 -> 90-109.
constexpr int LDH = 40;

template <typename T> struct Mfma16;
template <> struct Mfma16<bf16> {
  static __device__ __forceinline__ f32x16 run(const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma16<f16> {
  static __device__ __forceinline__ f32x16 run(const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

template <typename T> __device__ __forceinline__ uint16_t bits16(T x) {
  return __builtin_bit_cast(uint16_t, x);
}

// Parts of the reps in the score GEMM, of P and of the reps in the gradients.
template <typename T> struct Parts {
  static constexpr int S = sizeof(T) == 4 ? 3 : 1;
  static constexpr int P = std::is_same<T, bf16>::value ? 2 : 3;
  static constexpr int X = sizeof(T) == 4 ? 3 : std::is_same<T, f16>::value ? 2 : 1;
  typedef typename std::conditional<sizeof(T) == 4, bf16, T>::type ST;  // the score MFMA's type
  // Scale of P in the gradients, exact: the parts of a value under 2^-110 fall below bf16's smallest
  // (probabilities of e^-83, and gradients of nothing else, came out with errors of 2e-4).
  static constexpr float PS = X > 1 ? 0x1p48f : 1.0f;
};

// Two values as N parts, a pair of bf16 each.
template <int N>
__device__ __forceinline__ void parts2(f32x2 r, uint32_t (&p)[N]) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    p[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
    r = r - f32x2{__uint_as_float(p[i] << 16), __uint_as_float(p[i] & 0xffff0000u)};
  }
}
// Eight consecutive k of one row as N parts, 16 bytes each.
template <int N>
__device__ __forceinline__ void parts8(const float (&x)[8], u32x4 (&p)[N]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t w[N];
    parts2<N>(f32x2{x[2 * q], x[2 * q + 1]}, w);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i][q] = w[i];
  }
}

// A stage of a K-contiguous operand X[m][k] (row stride V): thread t holds k = k0 + 2 (t % 16), + 1
// of rows m0 + t / 16 + 16 u, two to a load where rows lie on 4-byte boundaries (`pair`); from
// clamped places otherwise and at the end of K, zero past it. Rows past M repeat the last one
// (nothing of theirs is stored).
template <typename T>
__device__ __forceinline__ void load_rows(const T* __restrict__ X, bool pair, int V, int m0, int M, int k0,
                                          int kend, Two<T> (&v)[8]) {
  const int t = threadIdx.x, k = k0 + 2 * (t & 15);
  typedef Two<T> __attribute__((aligned(4))) two;
  if (pair && k0 + KS <= kend) {  // uniform
#pragma unroll
    for (int u = 0; u < 8; ++u)
      v[u] = *(const two*)(X + (int64_t)min(m0 + (t >> 4) + 16 * u, M - 1) * V + k);
  } else {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const T* row = X + (int64_t)min(m0 + (t >> 4) + 16 * u, M - 1) * V;
      const T a = row[min(k, kend - 1)], b = row[min(k + 1, kend - 1)];
      v[u] = Two<T>{k < kend ? a : T(0.0f), k + 1 < kend ? b : T(0.0f)};
    }
  }
}
// Into [rows][KS] tiles, one per part, TM * LDH apart.
template <int N, typename T>
__device__ __forceinline__ void store_rows(uint16_t* s, const Two<T> (&v)[8]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    uint16_t* to = s + ((t >> 4) + 16 * u) * LDH + 2 * (t & 15);
    if constexpr (N == 1) {
      *(uint32_t*)to = __builtin_bit_cast(uint32_t, v[u]);
    } else {
      uint32_t p[N];
      parts2<N>(v[u], p);
#pragma unroll
      for (int i = 0; i < N; ++i) *(uint32_t*)(to + i * TM * LDH) = p[i];
    }
  }
}

// The operand of lane (l32, h) for k step s of a stage: row `row`, k = 16 s + 8 h .. + 7.
__device__ __forceinline__ u32x4 frag16(const uint16_t* s, int row, int ks) {
  const int h = (threadIdx.x & 63) >> 5;
  return *(const u32x4*)(s + row * LDH + 16 * ks + 8 * h);
}

// acc[bi][bj] += A[am0 + 32 bi .., :] B[bn0 + 32 bj .., :]^T over one stage, A in NA parts and B
// in NB (tiles of 128 rows): the pairs (i, j) with i + j < max(NA, NB), smallest first.
template <typename T, int NA, int NB, bool SPLIT>
__device__ __forceinline__ void mma16_stage(const uint16_t* sA, int am0, const uint16_t* sB, int bn0,
                                            f32x16 (&acc)[2][2], f32x16 (&low)[2][2]) {
  constexpr int W = NA > NB ? NA : NB;
  const int l32 = threadIdx.x & 31;
#pragma unroll
  for (int ks = 0; ks < KS / 16; ++ks) {
    u32x4 a[NA][2], b[NB][2];
#pragma unroll
    for (int p = 0; p < NA; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i) a[p][i] = frag16(sA + p * TM * LDH, am0 + 32 * i + l32, ks);
#pragma unroll
    for (int p = 0; p < NB; ++p)
#pragma unroll
      for (int j = 0; j < 2; ++j) b[p][j] = frag16(sB + p * TM * LDH, bn0 + 32 * j + l32, ks);
#pragma unroll
    for (int d = W - 1; d >= 0; --d)
#pragma unroll
      for (int p = 0; p < NA; ++p) {
        const int q = d - p;
        if (q < 0 || q >= NB) continue;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            f32x16& to = d > 0 && SPLIT ? low[i][j] : acc[i][j];
            to = Mfma16<T>::run(a[p][i], b[q][j], to);
          }
      }
  }
}

__device__ __forceinline__ void zero4(f32x16 (&acc)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero16();
}
__device__ __forceinline__ void add4(f32x16 (&acc)[2][2], const f32x16 (&low)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] += low[i][j];
}

// Whether any sum of the workgroup's is not finite (every thread calls it). A part of an infinite
// value, or of one that rounds to infinity in bf16, is infinite and its remainder no number: such a
// tile is done again on the fp32 MFMAs, whose products are those of the values themselves.
__device__ __forceinline__ bool any_nonfinite(const f32x16 (&acc)[2][2]) {
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) bad |= !(fabsf(acc[i][j][r]) < INFINITY);
  return __syncthreads_or(bad);
}

// loss_score_kernel on the 16-bit MFMAs.
template <typename T>
__global__ __launch_bounds__(NT, 2) void loss_score16_kernel(const T* __restrict__ Q,
                                                          const T* __restrict__ R, bool pair, int Bq,
                                                          int Bd, int V, int chunk,
                                                          float* __restrict__ part) {
  constexpr int NS = Parts<T>::S;
  __shared__ __attribute__((aligned(16))) uint16_t sA[NS * TM * LDH];
  __shared__ __attribute__((aligned(16))) uint16_t sB[NS * TM * LDH];
  static_assert(NS == 1 || sizeof(sA) >= KS * LDA * sizeof(float), "score_tile's tiles");
  // Workgroups go round the 8 XCDs in launch order: a chunk's tiles share one, so its columns of Q
  // and R come into one L2 once.
  const int tj = (Bd + TM - 1) / TM, tiles = tj * ((Bq + TM - 1) / TM), slot = blockIdx.x >> 3;
  const int tile = slot % tiles, c = 8 * (slot / tiles) + (blockIdx.x & 7);
  const int i0 = (tile / tj) * TM, j0 = (tile % tj) * TM;
  const int64_t kc = (int64_t)c * chunk;
  if (kc >= V) return;  // uniform
  const int kc0 = (int)kc, kc1 = min(V, kc0 + chunk);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, wm = wave >> 1, wn = wave & 1;
  f32x16 acc[2][2], low[2][2];
  zero4(acc);
  zero4(low);
  // Two stages of loads are in flight where registers allow: a stage's MFMAs are shorter than the
  // loads' way.
  constexpr int ST = NS > 1 ? 1 : 2;
  Two<T> ra[ST][8], rb[ST][8];
  auto load = [&](int k0, int b) {
    if (k0 >= kc1) return;  // uniform
    load_rows(Q, pair, V, i0, Bq, k0, kc1, ra[b]);
    load_rows(R, pair, V, j0, Bd, k0, kc1, rb[b]);
  };
  auto stage = [&](int k0, int b) {
    if (k0 >= kc1) return;
    __syncthreads();  // the previous stage is read
    store_rows<NS>(sA, ra[b]);
    store_rows<NS>(sB, rb[b]);
    __syncthreads();
    load(k0 + ST * KS, b);
    mma16_stage<typename Parts<T>::ST, NS, NS, (NS > 1)>(sA, wm * 64, sB, wn * 64, acc, low);
  };
  load(kc0, 0);
  if (ST > 1) load(kc0 + KS, ST - 1);
  for (int k0 = kc0; k0 < kc1; k0 += ST * KS) {
    stage(k0, 0);
    if (ST > 1) stage(k0 + KS, ST - 1);
  }
  if (NS > 1) add4(acc, low);
  if (NS > 1 && any_nonfinite(acc)) {
    zero4(acc);
    score_tile((float*)sA, (float*)sB, Q, R, Bq, Bd, V, i0, j0, kc0, kc1, acc);
  }
  float* out = part + (size_t)c * Bq * Bd;
  const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj) {
      const int j = j0 + wn * 64 + 32 * bj + l32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = i0 + wm * 64 + 32 * bi + acc_row(r, h);
        if (i < Bq && j < Bd) out[(size_t)i * Bd + j] = acc[bi][bj][r];
      }
    }
}

// ---- gradients as one tiled GEMM grid ----
//
// Both gradients are GEMMs over the other side's rows plus per-element terms:
//   dQ = c_ce P R + ...  (K = Bd),   dR = c_ce P^T Q + ...  (K = Bq).
// A workgroup owns GC columns of one 128-row tile of dQ or of dR, four waves of 64 x 64. It sums
// its own side's columns (the FLOPS term) while the first stages of the GEMM load. No workspace:
// everything stays in the workgroup.
// Two workgroups fit a CU, so what bounds it is the latency that a stage does not hide, in turn
// with the parts' vector arithmetic and the MFMAs (25% of the time for fp16): two stages are in
// flight, from uniform addresses at constant distances, and the sums' and the epilogue's loads
// are issued all at once. 256 x 512 x 30522 fp16, each with what comes before: parts in place of
// fp32 MFMAs 273 -> 174 us, two stages 155, uniform addresses and one side a workgroup 128,
// loads at once 105 (114 in a profile of whole passes); fp32 132, bf16 78.
constexpr int GC = 128;

static_assert(GC == TM, "one tile shape for both operands");
static_assert(KS == 32 && NT == 256, "the loaders' thread mappings");

// A stage of A = P rows m0.. (A_KC: thread t holds k = 8 (t % 4) .. + 7 of rows t / 4 + 64 u) or
// of P's columns m0.. (row t % 128, k = 8 (t / 128 + 2 u) .. + 7). k past P reads zero; rows past P
// repeat its last one (nothing of theirs is stored). A whole stage is loaded at constant distances
// from a uniform address, so it costs no vector arithmetic.
template <bool A_KC>
__device__ __forceinline__ void load_p(const float* __restrict__ P, int Bq, int Bd, int m0, int k0,
                                       float (&v)[2][8]) {
  const int t = threadIdx.x, K = A_KC ? Bd : Bq;
  typedef f32x4 __attribute__((aligned(4))) f32x4_any;
  const bool whole = k0 + KS <= K;  // uniform
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (A_KC) {
      const uint32_t m = (uint32_t)min(m0 + (t >> 2) + 64 * u, Bq - 1), k = 8 * (t & 3);
      if (whole) {
        const uint32_t off = m * (uint32_t)Bd + k;  // Bq Bd fits an int
        const f32x4 a = *(const f32x4_any*)(P + k0 + off), b = *(const f32x4_any*)(P + k0 + 4 + off);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[u][i] = a[i];
          v[u][4 + i] = b[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int kk = k0 + (int)k + i;
          const float x = P[m * (uint32_t)Bd + (uint32_t)min(kk, K - 1)];
          v[u][i] = kk < K ? x : 0.0f;
        }
      }
    } else {
      const int k = k0 + 8 * (__builtin_amdgcn_readfirstlane(t >> 7) + 2 * u);
      const uint32_t m = (uint32_t)min(m0 + (t & 127), Bd - 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float* row = P + (int64_t)min(k + i, K - 1) * Bd;
        v[u][i] = row[m];
      }
      if (!whole)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (k + i >= K) v[u][i] = 0.0f;
    }
  }
}
template <typename T, bool A_KC, int N>
__device__ __forceinline__ void store_p(uint16_t* s, const float (&v)[2][8]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int m = A_KC ? (t >> 2) + 64 * u : t & 127, kg = A_KC ? t & 3 : (t >> 7) + 2 * u;
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = v[u][i] * Parts<T>::PS;
    u32x4 p[N];
    parts8<N>(x, p);
#pragma unroll
    for (int i = 0; i < N; ++i) *(u32x4*)(s + i * TM * LDH + m * LDH + 8 * kg) = p[i];
  }
}

// Sums of X's columns c0 .. c0 + GC - 1 into sum: thread t adds columns 2 (t % 64), + 1 over rows
// t / 64 + 4 i, the four waves' shares are added in wave order. Every thread of the workgroup.
template <typename T>
__device__ __forceinline__ void column_sums(const T* __restrict__ X, bool pair, int K, int c0, int V,
                                            float (&share)[4][GC], float (&sum)[GC]) {
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), c = 2 * (t & 63);
  float a = 0.0f, b = 0.0f;
  constexpr int N = 128 / sizeof(T);  // loads in flight
  for (int k0 = 0; k0 < K; k0 += 4 * N) {
    Two<T> v[N];
    load_x<T>(X, pair, K, k0 + wave, 4, c0 + c, V, v);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      a += to_f32((T)v[i][0]);
      b += to_f32((T)v[i][1]);
    }
  }
  share[wave][c] = a;
  share[wave][c + 1] = b;
  __syncthreads();
  if (t < GC) sum[t] = ((share[0][t] + share[1][t]) + share[2][t]) + share[3][t];
  __syncthreads();
}

// A stage of X: thread t holds columns c0 + 2 (t % 64), + 1 of rows k0 + 8 (t / 64) .. + 7.
template <typename T, int N>
__device__ __forceinline__ void store_x(uint16_t* s, const Two<T> (&v)[8]) {
  const int t = threadIdx.x, kg = t >> 6, n = 2 * (t & 63);
#pragma unroll
  for (int col = 0; col < 2; ++col) {
    uint16_t* to = s + (n + col) * LDH + 8 * kg;
    if constexpr (N == 1) {
      u32x4 w;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        w[q] = (uint32_t)bits16<T>(v[2 * q][col]) | ((uint32_t)bits16<T>(v[2 * q + 1][col]) << 16);
      *(u32x4*)to = w;
    } else {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = to_f32((T)v[i][col]);
      u32x4 p[N];
      parts8<N>(x, p);
#pragma unroll
      for (int i = 0; i < N; ++i) *(u32x4*)(to + i * GC * LDH) = p[i];
    }
  }
}

// One GEMM tile: acc += A B^T over k in [0, K), A = P rows m0.. (A_KC) or P columns m0..,
// B = X[k][c0 ..], times PS. `meanwhile` (barriers in it are reached by every thread) runs under the first
// loads.
template <typename T, bool A_KC, typename F>
__device__ __forceinline__ void gemm16(uint16_t* sA, uint16_t* sB, const float* __restrict__ P, int Bq,
                                       int Bd, const T* __restrict__ X, bool pair, int K, int m0, int c0,
                                       int V, f32x16 (&acc)[2][2], const F& meanwhile) {
  f32x16 low[2][2];
  zero4(low);
  constexpr int NP = Parts<T>::P, NX = Parts<T>::X;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave >> 1, wn = wave & 1;
  // Two stages of loads are in flight: a stage's MFMAs are shorter than the loads' way.
  float pa0[2][8], pa1[2][8];
  Two<T> xv0[8], xv1[8];
  auto load = [&](int k0, float (&p)[2][8], Two<T> (&x)[8]) __attribute__((always_inline)) {
    if (k0 >= K) return;  // uniform
    load_p<A_KC>(P, Bq, Bd, m0, k0, p);
    load_x<T>(X, pair, K, k0 + 8 * wave, 1, c0 + 2 * (t & 63), V, x);
  };
  auto stage = [&](int k0, float (&p)[2][8], Two<T> (&x)[8]) __attribute__((always_inline)) {
    if (k0 >= K) return;
    __syncthreads();  // the previous stage is read
    store_p<T, A_KC, NP>(sA, p);
    store_x<T, NX>(sB, x);
    __syncthreads();
    load(k0 + 2 * KS, p, x);
    mma16_stage<bf16, NP, NX, (NX > 1)>(sA, wm * 64, sB, wn * 64, acc, low);
  };
  load(0, pa0, xv0);
  load(KS, pa1, xv1);
  meanwhile();
  for (int k0 = 0; k0 < K; k0 += 2 * KS) {
    stage(k0, pa0, xv0);
    stage(k0 + KS, pa1, xv1);
  }
  if (NX > 1) add4(acc, low);
}

// G[i][c] = c_ce acc / PS + c_s sign(X[i][c]) + c_f colsum[c] for the tile's rows below `rows`.
template <typename T>
__device__ __forceinline__ void grad16_epilogue(const f32x16 (&acc)[2][2], const T* __restrict__ X,
                                                int rows, int m0, int c0, int V, float c_ce,
                                                float c_s, float c_f, const float* colsum,
                                                T* __restrict__ G) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  T xv[2][2][16];  // every load issued, from clamped places, before any is used
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = m0 + wm * 64 + 32 * bi + acc_row(r, h), c = c0 + wn * 64 + 32 * bj + l32;
        xv[bi][bj][r] = X[(int64_t)min(i, rows - 1) * V + min(c, V - 1)];
      }
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj) {
      const int cl = wn * 64 + 32 * bj + l32, c = c0 + cl;
      const float add = c_f * colsum[cl];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = m0 + wm * 64 + 32 * bi + acc_row(r, h);
        if (i < rows && c < V) {
          const float x = to_f32(xv[bi][bj][r]);
          const float sg = x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f);
          G[(int64_t)i * V + c] = from_f32<T>(c_ce * (acc[bi][bj][r] * (1.0f / Parts<T>::PS)) + c_s * sg + add);
        }
      }
    }
}

template <typename T>
__global__ __launch_bounds__(NT, 2) void loss_grad16_kernel(const T* __restrict__ Q,
                                                            const T* __restrict__ R,
                                                            const float* __restrict__ P, const Grads6 g,
                                                            bool pair, int Bq, int Bd, int V, float w_ce,
                                                            float w_l1, float w_fl,
                                                            T* __restrict__ GQ,
                                                            T* __restrict__ GR) {
  __shared__ __attribute__((aligned(16))) uint16_t sA[Parts<T>::P * TM * LDH];
  __shared__ __attribute__((aligned(16))) uint16_t sB[Parts<T>::X * GC * LDH];
  __shared__ float share[4][GC];
  __shared__ float colsum[GC];
  // One bf16 part (bf16 reps) is the value itself.
  constexpr bool REDO = Parts<T>::X > 1;
  static_assert(!REDO || (sizeof(sA) >= KS * LDA * sizeof(float) && sizeof(sB) >= KS * LDB * sizeof(float)),
                "grad_tile's tiles");
  // Workgroups go round the 8 XCDs in launch order: the tiles of one side and column tile share an
  // XCD, so what they stream comes into one L2 once. The side with the longer GEMMs goes first.
  const int nq = (Bq + TM - 1) / TM, nd = (Bd + TM - 1) / TM, cols8 = (V + 8 * GC - 1) / (8 * GC);
  const bool q_first = Bd >= Bq;
  const int n0 = q_first ? nq : nd, n1 = q_first ? nd : nq;
  int slot = blockIdx.x >> 3;
  const bool second = slot >= cols8 * n0;  // uniform, as all below
  if (second) slot -= cols8 * n0;
  const int n = second ? n1 : n0;
  const int c0 = (8 * (slot / n) + (int)(blockIdx.x & 7)) * GC, m0 = (slot % n) * TM;
  if (c0 >= V) return;
  const float g0 = grad_of(g, 0);
  const float c_ce = g0 * w_ce + grad_of(g, 1);
  f32x16 acc[2][2];
  zero4(acc);
  if (second != q_first) {
    gemm16<T, true>(sA, sB, P, Bq, Bd, R, pair, Bd, m0, c0, V, acc,
                    [&] { column_sums<T>(Q, pair, Bq, c0, V, share, colsum); });
    const float c_s = (g0 * w_l1 + grad_of(g, 2)) / (float)Bq;
    const float c_f = 2.0f * (g0 * w_fl + grad_of(g, 4)) / (float)V;
    if (REDO && any_nonfinite(acc)) {
      for (int c = 0; c < GC && c0 + c < V; c += NC)
        grad_tile<T, true>((float*)sA, (float*)sB, P, Bq, Bd, R, Bd, Q, Bq, m0, c0 + c, V, c_ce, c_s, c_f,
                           colsum + c, GQ);
      return;
    }
    grad16_epilogue(acc, Q, Bq, m0, c0, V, c_ce, c_s, c_f, colsum, GQ);
  } else {
    gemm16<T, false>(sA, sB, P, Bq, Bd, Q, pair, Bq, m0, c0, V, acc,
                     [&] { column_sums<T>(R, pair, Bd, c0, V, share, colsum); });
    const float c_s = (g0 * w_l1 + grad_of(g, 3)) / (float)Bd;
    const float c_f = 2.0f * (g0 * w_fl + grad_of(g, 5)) / (float)V;
    if (REDO && any_nonfinite(acc)) {
      for (int c = 0; c < GC && c0 + c < V; c += NC)
        grad_tile<T, false>((float*)sA, (float*)sB, P, Bq, Bd, Q, Bq, R, Bd, m0, c0 + c, V, c_ce, c_s, c_f,
                            colsum + c, GR);
      return;
    }
    grad16_epilogue(acc, R, Bd, m0, c0, V, c_ce, c_s, c_f, colsum, GR);
  }
}

template <typename T>
__global__ __launch_bounds__(NT) void loss_bwd_large_kernel(const T* __restrict__ Q, const T* __restrict__ R,
                                                            const float* __restrict__ P, const Grads6 g,
                                                            int Bq, int Bd, int V, float w_ce, float w_l1,
                                                            float w_fl, T* __restrict__ GQ,
                                                            T* __restrict__ GR) {
  __shared__ float sA[KS * LDA];
  __shared__ float sB[KS * LDB];
  __shared__ float cpart[2][4][NC];
  __shared__ float colsum[2][NC];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c0 = blockIdx.x * NC;
  // the columns' sums over Q's and R's rows: wave w sums rows w, w + 4, ... in order
  {
    const int c = c0 + lane;
    const bool cv = c < V;
    for (int side = 0; side < 2; ++side) {
      const T* X = side ? R : Q;
      const int rows = side ? Bd : Bq;
      float cs = 0.0f;
      for (int b0 = wave; b0 < rows; b0 += 4 * ST_ROWS) {
        T v[ST_ROWS];
#pragma unroll
        for (int u = 0; u < ST_ROWS; ++u)
          v[u] = X[(int64_t)min(b0 + 4 * u, rows - 1) * V + min(c, V - 1)];
#pragma unroll
        for (int u = 0; u < ST_ROWS; ++u)
          if (!(b0 + 4 * u < rows && cv)) v[u] = T(0.0f);
#pragma unroll
        for (int u = 0; u < ST_ROWS; ++u) cs += to_f32(v[u]);
      }
      cpart[side][wave][lane] = cs;
    }
  }
  __syncthreads();
  if (threadIdx.x < 2 * NC) {
    const int side = threadIdx.x / NC, l = threadIdx.x % NC;
    colsum[side][l] = ((cpart[side][0][l] + cpart[side][1][l]) + cpart[side][2][l]) + cpart[side][3][l];
  }
  __syncthreads();
  const float g0 = grad_of(g, 0);
  const float c_ce = g0 * w_ce + grad_of(g, 1);
  const float c_sq = (g0 * w_l1 + grad_of(g, 2)) / (float)Bq;
  const float c_sd = Bd > 0 ? (g0 * w_l1 + grad_of(g, 3)) / (float)Bd : 0.0f;
  const float c_fq = 2.0f * (g0 * w_fl + grad_of(g, 4)) / (float)V;
  const float c_fd = 2.0f * (g0 * w_fl + grad_of(g, 5)) / (float)V;
  for (int i0 = 0; i0 < Bq; i0 += TM)  // dQ = c_ce P R + ...
    grad_tile<T, true>(sA, sB, P, Bq, Bd, R, Bd, Q, Bq, i0, c0, V, c_ce, c_sq, c_fq, colsum[0], GQ);
  for (int j0 = 0; j0 < Bd; j0 += TM)  // dR = c_ce P^T Q + ...
    grad_tile<T, false>(sA, sB, P, Bq, Bd, Q, Bq, R, Bd, j0, c0, V, c_ce, c_sd, c_fd, colsum[1], GR);
}

// Score chunking: about 512 workgroups, chunks of whole LDS stages.
struct ScorePlan {
  int tiles, chunk, nchunk;
};
static ScorePlan score_plan(int64_t Bq, int64_t Bd, int64_t V) {
  ScorePlan p;
  p.tiles = (int)(cdiv(Bq, TM) * cdiv(Bd, TM));
  const int64_t want = cdiv(512, p.tiles);
  const int64_t nc = want < 1 ? 1 : (want > cdiv(V, 256) ? cdiv(V, 256) : want);
  p.chunk = (int)round_up(cdiv(V, nc), KS);
  p.nchunk = (int)cdiv(V, p.chunk);
  return p;
}
static int64_t stats_entries(int64_t Bq, int64_t Bd) { return Bq + Bd + 2; }
// Workspace (floats): partial S per chunk, S, partial stats per slice, stats, row CE terms.
static int64_t workspace_floats(int64_t Bq, int64_t Bd, int64_t V) {
  const int64_t s = Bd > 0 ? (int64_t)score_plan(Bq, Bd, V).nchunk * Bq * Bd + Bq * Bd : 0;
  return s + (slices(V) + 1) * stats_entries(Bq, Bd) + Bq;
}

// SPARTON_LOSS_MFMA16=0 takes the fp32 MFMAs throughout (tests compare the two).
static bool mfma16_on() {
  const char* e = getenv("SPARTON_LOSS_MFMA16");
  return e == nullptr || strcmp(e, "0") != 0;
}

// Two columns to a load: rows of an even number of elements, from a place aligned to two.
template <typename T>
static bool pairs(const void* q, const void* d, int V) {
  return V % 2 == 0 && ((uintptr_t)q | (uintptr_t)d) % (2 * sizeof(T)) == 0;
}

template <typename T>
static void fwd(const void* q, const void* d, int Bq, int Bd, int V, float inv_t, float w_ce,
                float w_l1, float w_fl, float* out, float* probs, float* ws, hipStream_t st) {
  float* spart = ws;
  float* S = nullptr;
  if (Bd > 0) {
    const ScorePlan p = score_plan(Bq, Bd, V);
    S = spart + (size_t)p.nchunk * Bq * Bd;
    if (mfma16_on()) {
      const dim3 grid((unsigned)(p.tiles * round_up(p.nchunk, 8)));
      const bool pair = V * sizeof(T) % 4 == 0 && ((uintptr_t)q | (uintptr_t)d) % 4 == 0;
      hipLaunchKernelGGL((loss_score16_kernel<T>), grid, dim3(NT), 0, st, (const T*)q, (const T*)d,
                         pair, Bq, Bd, V, p.chunk, spart);
    } else {
      hipLaunchKernelGGL((loss_score_kernel<T>), dim3((unsigned)p.tiles, (unsigned)p.nchunk), dim3(NT),
                         0, st, (const T*)q, (const T*)d, Bq, Bd, V, p.chunk, spart);
    }
    const int K = Bq * Bd;
    hipLaunchKernelGGL(loss_slice_sum_kernel, dim3((unsigned)cdiv(K, 64)), dim3(64 * SUM_WAVES), 0, st,
                       (const float*)spart, p.nchunk, K, S);
  }
  float* tpart = Bd > 0 ? S + (size_t)Bq * Bd : ws;
  const int KS2 = (int)stats_entries(Bq, Bd), ns = (int)cdiv(V, ST_COLS);
  float* stats = tpart + (size_t)ns * KS2;
  float* row_loss = stats + KS2;
  hipLaunchKernelGGL((loss_stats_kernel<T>), dim3((unsigned)ns, 2), dim3(NT), 0, st, (const T*)q,
                     (const T*)d, pairs<T>(q, d, V), Bq, Bd, V, tpart, KS2);
  hipLaunchKernelGGL(loss_slice_sum_kernel, dim3((unsigned)cdiv(KS2, 64)), dim3(64 * SUM_WAVES), 0, st,
                     (const float*)tpart, ns, KS2, stats);
  if (Bd > 0)
    hipLaunchKernelGGL(loss_rows_kernel, dim3((unsigned)cdiv(Bq, 4)), dim3(NT), 0, st, (const float*)S,
                       Bq, Bd, inv_t, row_loss, probs);
  hipLaunchKernelGGL(loss_final_large_kernel, dim3(1), dim3(64), 0, st, (const float*)row_loss,
                     (const float*)stats, Bq, Bd, V, w_ce, w_l1, w_fl, out);
}

template <typename T>
static void bwd(const void* q, const void* d, const float* P, const Grads6& g, int Bq, int Bd, int V,
                float w_ce, float w_l1, float w_fl, void* gq, void* gd, hipStream_t st) {
  if (mfma16_on()) {
    const dim3 grid((unsigned)(round_up(cdiv(V, GC), 8) * (cdiv(Bq, TM) + cdiv(Bd, TM))));
    hipLaunchKernelGGL(loss_grad16_kernel<T>, grid, dim3(NT), 0, st, (const T*)q, (const T*)d, P, g,
                       pairs<T>(q, d, V), Bq, Bd, V, w_ce, w_l1, w_fl, (T*)gq, (T*)gd);
    return;
  }
  hipLaunchKernelGGL((loss_bwd_large_kernel<T>), dim3((unsigned)cdiv(V, NC)), dim3(NT), 0, st,
                     (const T*)q, (const T*)d, P, g, Bq, Bd, V, w_ce, w_l1, w_fl, (T*)gq, (T*)gd);
}
}  // namespace big

// Batches with more than MAX_B rows on either side take the kernels in `big`.
static bool is_big(int64_t Bq, int64_t Bd) { return Bq > MAX_B || Bd > MAX_B; }

}  // namespace loss
}  // namespace sparton

using namespace sparton;

static int loss_check(int64_t Bq, int64_t Bd, int64_t V, int dtype) {
  if (dtype < SPARTON_F32 || dtype > SPARTON_F16) return SPARTON_EINVAL;
  if (Bq < 1 || Bd < 0 || V < 1) return SPARTON_EINVAL;
  // int offsets: the scores and their per-chunk partials, and row * V + column
  if (V > INT32_MAX || Bq > INT32_MAX / 8 || Bd > INT32_MAX / 8 ||
      (Bd > 0 && Bq * Bd * (int64_t)loss::big::score_plan(Bq, Bd, V).nchunk > INT32_MAX) ||
      (Bq + Bd) * V > ((int64_t)1 << 62))
    return SPARTON_EUNSUPPORTED;
  if (Bd > 0 && Bq > Bd) return SPARTON_EINVAL;  // labels arange(Bq) index R's rows
  return SPARTON_OK;
}

extern "C" __attribute__((visibility("default"))) size_t sparton_loss_workspace_bytes(int64_t Bq,
                                                                                      int64_t Bd,
                                                                                      int64_t V) {
  if (Bq < 1 || Bd < 0 || V < 1) return 0;
  if (loss::is_big(Bq, Bd)) return (size_t)loss::big::workspace_floats(Bq, Bd, V) * sizeof(float);
  return (size_t)((loss::slices(V) + 1) * loss::entries(Bq, Bd)) * sizeof(float);
}

extern "C" __attribute__((visibility("default"))) int sparton_loss_fwd(
    const void* q, const void* d, int64_t Bq, int64_t Bd, int64_t V, float temperature, float w_ce,
    float w_l1, float w_flops, float* out, float* probs, void* workspace, size_t workspace_bytes,
    int dtype, void* stream) {
  const int rc = loss_check(Bq, Bd, V, dtype);
  if (rc != SPARTON_OK) return rc;
  if (q == nullptr || out == nullptr || (Bd > 0 && (d == nullptr || probs == nullptr)))
    return SPARTON_EINVAL;
  if (Bd > 0 && !(temperature > 0.0f && temperature < INFINITY)) return SPARTON_EINVAL;
  if (workspace == nullptr || workspace_bytes < sparton_loss_workspace_bytes(Bq, Bd, V))
    return SPARTON_EWORKSPACE;
  if ((uintptr_t)workspace % 16 != 0) return SPARTON_EALIGN;
  hipStream_t st = (hipStream_t)stream;
  if (loss::is_big(Bq, Bd)) {
    const float inv_t = Bd > 0 ? 1.0f / temperature : 0.0f;
    float* ws = (float*)workspace;
    switch (dtype) {
      case SPARTON_BF16:
        loss::big::fwd<bf16>(q, d, (int)Bq, (int)Bd, (int)V, inv_t, w_ce, w_l1, w_flops, out, probs, ws, st);
        break;
      case SPARTON_F16:
        loss::big::fwd<f16>(q, d, (int)Bq, (int)Bd, (int)V, inv_t, w_ce, w_l1, w_flops, out, probs, ws, st);
        break;
      default:
        loss::big::fwd<float>(q, d, (int)Bq, (int)Bd, (int)V, inv_t, w_ce, w_l1, w_flops, out, probs, ws, st);
        break;
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SPARTON_OK : (int)e;
  }
  const int K = (int)loss::entries(Bq, Bd), ns = (int)loss::slices(V);
  float* part = (float*)workspace;
  float* sums = part + (size_t)ns * K;
  switch (dtype) {
    case SPARTON_BF16: loss::fwd_partial<bf16>(q, d, (int)Bq, (int)Bd, (int)V, part, K, st); break;
    case SPARTON_F16: loss::fwd_partial<f16>(q, d, (int)Bq, (int)Bd, (int)V, part, K, st); break;
    default: loss::fwd_partial<float>(q, d, (int)Bq, (int)Bd, (int)V, part, K, st); break;
  }
  hipLaunchKernelGGL(loss::loss_slice_sum_kernel, dim3((unsigned)cdiv((int64_t)K, (int64_t)64)),
                     dim3(64 * loss::SUM_WAVES), 0, st, (const float*)part, ns, K, sums);
  hipLaunchKernelGGL(loss::loss_final_kernel, dim3(1), dim3(loss::NT), 0, st, (const float*)sums,
                     (int)Bq, (int)Bd, (int)V, Bd > 0 ? 1.0f / temperature : 0.0f, w_ce, w_l1,
                     w_flops, out, probs);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SPARTON_OK : (int)e;
}

static int loss_bwd_run(const void* q, const void* d, const float* probs, const loss::Grads6& grad_out,
                        int64_t Bq, int64_t Bd, int64_t V, float w_ce, float w_l1, float w_flops,
                        void* grad_q, void* grad_d, int dtype, void* stream) {
  const int rc = loss_check(Bq, Bd, V, dtype);
  if (rc != SPARTON_OK) return rc;
  if (q == nullptr || grad_q == nullptr ||
      (Bd > 0 && (d == nullptr || probs == nullptr || grad_d == nullptr)))
    return SPARTON_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (loss::is_big(Bq, Bd)) {
    switch (dtype) {
      case SPARTON_BF16:
        loss::big::bwd<bf16>(q, d, probs, grad_out, (int)Bq, (int)Bd, (int)V, w_ce, w_l1, w_flops, grad_q,
                             grad_d, st);
        break;
      case SPARTON_F16:
        loss::big::bwd<f16>(q, d, probs, grad_out, (int)Bq, (int)Bd, (int)V, w_ce, w_l1, w_flops, grad_q,
                            grad_d, st);
        break;
      default:
        loss::big::bwd<float>(q, d, probs, grad_out, (int)Bq, (int)Bd, (int)V, w_ce, w_l1, w_flops, grad_q,
                              grad_d, st);
        break;
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SPARTON_OK : (int)e;
  }
  switch (dtype) {
    case SPARTON_BF16:
      loss::bwd_all<bf16>(q, d, probs, grad_out, (int)Bq, (int)Bd, (int)V, w_ce, w_l1, w_flops, grad_q,
                          grad_d, st);
      break;
    case SPARTON_F16:
      loss::bwd_all<f16>(q, d, probs, grad_out, (int)Bq, (int)Bd, (int)V, w_ce, w_l1, w_flops, grad_q,
                         grad_d, st);
      break;
    default:
      loss::bwd_all<float>(q, d, probs, grad_out, (int)Bq, (int)Bd, (int)V, w_ce, w_l1, w_flops,
                           grad_q, grad_d, st);
      break;
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SPARTON_OK : (int)e;
}

extern "C" __attribute__((visibility("default"))) int sparton_loss_bwd(
    const void* q, const void* d, const float* probs, const float* grad_out, int64_t Bq, int64_t Bd,
    int64_t V, float w_ce, float w_l1, float w_flops, void* grad_q, void* grad_d, int dtype,
    void* stream) {
  if (grad_out == nullptr) return SPARTON_EINVAL;
  const loss::Grads6 g{{grad_out, grad_out + 1, grad_out + 2, grad_out + 3, grad_out + 4, grad_out + 5}};
  return loss_bwd_run(q, d, probs, g, Bq, Bd, V, w_ce, w_l1, w_flops, grad_q, grad_d, dtype, stream);
}

extern "C" __attribute__((visibility("default"))) int sparton_loss_bwd_terms(
    const void* q, const void* d, const float* probs, const float* const* grad_terms, int64_t Bq,
    int64_t Bd, int64_t V, float w_ce, float w_l1, float w_flops, void* grad_q, void* grad_d,
    int dtype, void* stream) {
  if (grad_terms == nullptr) return SPARTON_EINVAL;
  loss::Grads6 g;
  for (int k = 0; k < 6; ++k) g.p[k] = grad_terms[k];
  return loss_bwd_run(q, d, probs, g, Bq, Bd, V, w_ce, w_l1, w_flops, grad_q, grad_d, dtype, stream);
}
