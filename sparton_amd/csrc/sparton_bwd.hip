// SpartonHead backward on gfx950: atomic-free on floating-point data, deterministic,
// HBM-bound.
//
// Only entries (b,v) with reps > 0, G != 0 and mask[b,I] != 0 carry gradient
// (g' = G*exp(-reps)*mask[b,I]). The reference scatters them with fp32 atomics into
// zero-filled dH/dW/dbias (src/sparton/sparton_kernel.py:473-565, :676-678). Here
// every output row is summed in a fixed order by one workgroup:
//
//   dW / dbias  row v gathers H[b, I[b,v], :] for b ascending. For B <= 128 and S <= 65536 a
//               workgroup stages g' and I of all batch rows for 32 consecutive ids in LDS
//               (coalesced loads) and its waves gather the H rows of one id at a time;
//               bwd_dw_wide_kernel and bwd_dw_kernel take larger batches.
//   dH          bucket_run sorts each batch row's entries by position, at most 16 runs of
//               consecutive ids per batch row; then bwd_dh_kernel's 16-lane groups sum
//               g' * W[v,:] over a row's entries, run by run, ids ascending.
//
// The bucketing and the staged dW share a launch (neither needs the other), so a backward is
// two launches. At most 64 dH rows take the few-row path instead.
// Measured against the kernels it replaced, which sorted by 64-id blocks and gave each dH row
// one wave, 4 rows of W in flight (backward kernels, one box): dense gradients, 16 x 256 rows
// bf16 into fp32 341 -> 186 us, 8 x 128 rows fp32 557 -> 153 us; 5% dense, 32 x 256 rows
// 47 -> 48 us, 8 x 512 rows 23 -> 24 us, V = 250002 337 -> 290 us, D = 4096 515 -> 425 us.
// The only atomics are integer counts in LDS, which are order-independent.
//
// Gradients are written as fp32 (what the reference returns) or in the input dtype
// (what autograd would cast them to for bf16/fp16 parameters), rounded once from
// the fp32 sums.

#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "sparton_common.h"

extern __shared__ __attribute__((aligned(16))) unsigned char sparton_bwd_smem[];

namespace sparton {
namespace bwd {

constexpr int BK_WAVES = 8;         // waves of a bucketing or dW workgroup
constexpr int BK_ROUNDS = 8;        // rounds of 64 ids whose loads a bucketing wave has in flight
constexpr int BK_IDS = 64 * BK_ROUNDS * BK_WAVES;  // ids of a workgroup's turn
constexpr int BK_RUNS = 16;         // bucketing workgroups (runs) per batch row, at most
constexpr int MAX_S = 4096;         // positions per dH window (LDS: S counters per wave)
constexpr int64_t MAX_ROWS = 1 << 20;  // dH rows per pass (bounds the run offsets)
constexpr int64_t MAX_B = 8192;     // and batch rows (bounds the runs, 8 V bytes each)
constexpr int MAX_NP = 16;          // D up to 16 * 256 per register pass

// How a batch row's ids are cut: `runs` runs of `cap` ids (a multiple of BK_IDS).
struct Cut {
  int64_t runs, cap;
};
static Cut cut_ids(int64_t V) {
  Cut c;
  c.cap = BK_IDS * std::max<int64_t>(1, cdiv(V, (int64_t)BK_IDS * BK_RUNS));
  c.runs = std::max<int64_t>(1, cdiv(V, c.cap));
  return c;
}

struct Layout {
  size_t off, run, total;
};
static Layout layout(int64_t B, int64_t S, int64_t V) {
  Layout L;
  size_t at = 0;
  auto take = [&](size_t bytes) { size_t o = at; at += (size_t)round_up((int64_t)bytes, 256); return o; };
  L.off = take((size_t)(B * (S + 1) * cut_ids(V).runs) * 4);  // [B][S + 1][runs] a position's first entry
  L.run = take((size_t)(B * V) * 8);  // [B][V] (v, g'): run c from id c cap on, by position, then v
  L.total = at;
  return L;
}

// A launch holds fewer than 2^32 threads (past that, workgroups were left out without an error):
// the workgroups of a dH launch, and of one with dW's.
constexpr int64_t MAX_THREADS = ((int64_t)1 << 32) - 1;
constexpr int64_t DH_MAX_WG = MAX_THREADS / 256, BK_MAX_WG = MAX_THREADS / (64 * BK_WAVES);

// Batch rows and positions of one dH pass: 16 rows a workgroup, for each 256-byte slice of theirs.
struct Pass {
  int64_t b, s;
};
static Pass pass_of(int64_t B, int64_t S, int64_t D) {
  const int64_t rows = std::max<int64_t>(16, std::min<int64_t>(MAX_ROWS, 16 * (DH_MAX_WG / cdiv(D * 4, 256))));
  Pass p;
  p.s = std::min<int64_t>({S, MAX_S, rows});
  p.b = std::min<int64_t>({B, MAX_B, std::max<int64_t>(1, rows / std::max<int64_t>(1, p.s))});
  return p;
}

static int64_t mask_elem_bytes(int mdt) {
  switch (mdt) {
    case SPARTON_MASK_I64: return 8;
    case SPARTON_MASK_I32:
    case SPARTON_MASK_F32: return 4;
    case SPARTON_MASK_U8: return 1;
    default: return 2;
  }
}

// Entry (b, v): whether it carries gradient, its coefficient g' and index s.
// Activity is decided by comparisons of loaded values only (never by the float
// product), so the bucketing's count and its write agree on every entry; an index outside
// [0, S) makes the entry inactive, so it can never turn into an out-of-bounds access.
// g' = G * exp(-reps) (src/sparton/sparton_kernel.py:531) times mask[b, I], the torch
// head's d x / d logits (training/model.py:60); 1 for a 0/1 mask.
template <typename T, typename RT>
__device__ __forceinline__ bool entry(T g_raw, RT r_raw, int s, const float* maskf, int S,
                                      float* g_out) {
  *g_out = 0.0f;
  const float r = to_f32(r_raw);
  if (!(r > 0.0f) || s < 0 || s >= S) return false;
  const float g = to_f32(g_raw);
  if (g == 0.0f) return false;
  const float m = maskf[s];
  if (m == 0.0f) return false;
  *g_out = g * expf(-r) * m;
  return true;
}

// ---- bucketing --------------------------------------------------------------
//
// The active entries of each batch row are sorted by position, ids ascending, a run of
// consecutive ids at a time: workgroup (b, c) takes run c (at most BK_RUNS of them, so that
// a 16-lane group can look at all runs of its row at once), wave w of it a contiguous share.
// It counts the share's entries per (wave, position) in LDS, a scan over (position, wave)
// turns the counts into slots, and each entry goes to its slot, ranked among the equal
// positions of its 64: a stable counting sort. off[b][s][c] is the run's first entry of
// position s. One launch and no exchange between workgroups; dW's workgroups share the
// launch (dW reads only the inputs) and hide it.
//
// A share is taken BK_ROUNDS rounds of 64 ids at a time: their 3 * BK_ROUNDS loads are issued
// up front and unconditionally (ids past V re-read id V - 1 and are inactive), no value
// converted or tested until all are in flight. A share of one turn (V <= 65536) keeps its
// entries in registers between counting and writing; longer ones read them again.
template <typename T, typename RT>
__device__ __forceinline__ void bucket_run(const T* __restrict__ grad, const RT* __restrict__ reps,
                                           const int32_t* __restrict__ idx,
                                           const void* __restrict__ mask, int mdt, int S, int V,
                                           int64_t b, int c, int runs, int cap, int* __restrict__ off,
                                           int2* __restrict__ run, int s0, int S_row) {
  constexpr int NT = 64 * BK_WAVES;
  int* wsum = (int*)sparton_bwd_smem;  // [BK_WAVES]
  int* carry = wsum + BK_WAVES;
  float* maskf = (float*)(carry + 1);  // [S]
  int* all = (int*)(maskf + S);        // [BK_WAVES][S]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int* cur = all + wave * S;
  const int share = cap / BK_WAVES, v_beg = c * cap + wave * share;
  const int turns = share / (64 * BK_ROUNDS);
  float g[BK_ROUNDS];
  int s[BK_ROUNDS];  // position in the window, -1: inactive
  T gr[BK_ROUNDS];
  RT rr[BK_ROUNDS];
  auto load = [&](int t) {
#pragma unroll
    for (int j = 0; j < BK_ROUNDS; ++j) {
      const int64_t o = b * V + max(0, min(v_beg + (t * BK_ROUNDS + j) * 64 + lane, V - 1));
      gr[j] = grad[o];
      rr[j] = reps[o];
      s[j] = idx[o];
    }
  };
  auto decide = [&](int t) {
#pragma unroll
    for (int j = 0; j < BK_ROUNDS; ++j) {
      // Positions relative to the window (wrapping: an index outside it lands outside [0, S)
      // and the entry is inactive).
      const int sw = (int)((unsigned)s[j] - (unsigned)s0);
      const bool act = v_beg + (t * BK_ROUNDS + j) * 64 + lane < V && entry(gr[j], rr[j], sw, maskf, S, &g[j]);
      s[j] = act ? sw : -1;
    }
  };
  if (V > 0) load(0);
  for (int i = tid; i < S; i += NT) maskf[i] = load_mask(mask, mdt, b * S_row + s0 + i);
  for (int i = tid; i < BK_WAVES * S; i += NT) all[i] = 0;
  if (tid == 0) *carry = 0;
  __syncthreads();
  for (int t = 0; t < turns && V > 0; ++t) {
    if (t > 0) load(t);
    decide(t);
#pragma unroll
    for (int j = 0; j < BK_ROUNDS; ++j)
      if (s[j] >= 0) atomicAdd(&cur[s[j]], 1);
  }
  __syncthreads();
  int* ob = off + b * (S + 1) * runs + c;
  for (int p0 = 0; p0 < S; p0 += NT) {
    const int p = p0 + tid;
    int k[BK_WAVES], tot = 0;
#pragma unroll
    for (int w = 0; w < BK_WAVES; ++w) {
      k[w] = p < S ? all[w * S + p] : 0;
      tot += k[w];
    }
    int incl = tot;  // inclusive scan over p: within the wave, then across waves
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int at = *carry + incl - tot;
    for (int w = 0; w < wave; ++w) at += wsum[w];
    if (p < S) {
      ob[(int64_t)p * runs] = at;
      if (p == S - 1) ob[(int64_t)S * runs] = at + tot;
      int slot = at;
#pragma unroll
      for (int w = 0; w < BK_WAVES; ++w) {
        all[w * S + p] = slot;
        slot += k[w];
      }
    }
    __syncthreads();
    if (tid == NT - 1) *carry = at + tot;
    __syncthreads();
  }
  // Lanes with equal s are found with one ballot per bit of s: `same` keeps the lanes that
  // agree with this lane on every bit. A slot is the cursor of its position plus the lower
  // lanes of its group; all lanes read the cursor, then each group's lowest lane advances it
  // (one wave's LDS accesses complete in program order).
  const uint64_t lt = (1ull << lane) - 1ull;
  const int sbits = S > 1 ? 32 - __builtin_clz((unsigned)(S - 1)) : 0;
  int2* out = run + b * V + c * cap;
  for (int t = 0; t < turns && V > 0; ++t) {
    if (turns > 1) {
      load(t);
      decide(t);
    }
#pragma unroll
    for (int j = 0; j < BK_ROUNDS; ++j) {
      const bool act = s[j] >= 0;
      uint64_t same = __ballot(act);
      if (same != 0) {  // uniform
        const int sj = act ? s[j] : 0;
        for (int k = 0; k < sbits; ++k) {
          const bool bit = ((sj >> k) & 1) != 0;
          const uint64_t ones = __ballot(bit);
          same &= bit ? ones : ~ones;
        }
        const int at = act ? cur[sj] : 0;
        if (act) out[at + __popcll(same & lt)] = make_int2(v_beg + (t * BK_ROUNDS + j) * 64 + lane, __float_as_int(g[j]));
        if (act && (same & lt) == 0) cur[sj] = at + __popcll(same);
      }
    }
  }
}

// Store four fp32 values as O. The gradients are written once and read by nothing in the
// backward, so the stores are nontemporal: they stream to memory instead of evicting from
// L2 the W and H rows that the gathers re-read (cfg 4 backward 342 -> 320 us, cfg 5
// 535 -> 482 us).
__device__ __forceinline__ void store4(float* p, const f32x4& a) {
  __builtin_nontemporal_store(a, (f32x4*)p);
}
__device__ __forceinline__ void store4(bf16* p, const f32x4& a) {
  const bf16x4 v = bf16x4{(bf16)a[0], (bf16)a[1], (bf16)a[2], (bf16)a[3]};
  __builtin_nontemporal_store(__builtin_bit_cast(uint64_t, v), (uint64_t*)p);
}
__device__ __forceinline__ void store4(f16* p, const f32x4& a) {
  const f16x4 v = f16x4{(f16)a[0], (f16)a[1], (f16)a[2], (f16)a[3]};
  __builtin_nontemporal_store(__builtin_bit_cast(uint64_t, v), (uint64_t*)p);
}

// Four consecutive elements of a row, loaded raw (8 bytes for 16-bit types, 16 for
// fp32) so that a batch of loads is issued before any conversion.
template <typename T> struct Raw4;
template <> struct Raw4<float> {
  f32x4 v;
  __device__ __forceinline__ void load(const float* p) { v = *(const f32x4*)p; }
  __device__ __forceinline__ void zero() { v = f32x4{0.f, 0.f, 0.f, 0.f}; }
  __device__ __forceinline__ f32x4 f() const { return v; }
};
template <> struct Raw4<bf16> {
  bf16x4 v;
  __device__ __forceinline__ void load(const bf16* p) { v = *(const bf16x4*)p; }
  __device__ __forceinline__ void zero() { v = bf16x4{(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f}; }
  __device__ __forceinline__ f32x4 f() const { return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]}; }
};
template <> struct Raw4<f16> {
  f16x4 v;
  __device__ __forceinline__ void load(const f16* p) { v = *(const f16x4*)p; }
  __device__ __forceinline__ void zero() { v = f16x4{(f16)0.f, (f16)0.f, (f16)0.f, (f16)0.f}; }
  __device__ __forceinline__ f32x4 f() const { return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]}; }
};

// The order every dH row is summed in (the few-row path aside): the row's entries, in v
// order, are taken DH_BATCH at a time (the last batch may hold fewer); a batch's partial is
// P = fma(g_u, W[v_u], P) over its entries from P = 0. Partials are added in order in blocks of
// FOLD entries, those in blocks of FOLD2 and these in order (below). So a row is the same bits
// whether one lane group sums it or a workgroup shares its batches.
constexpr int DH_BATCH = 4;

// Rows gathered per batch: all their loads are in flight together (about 24 per lane).
template <int NP> struct Batch { static constexpr int U = NP <= 3 ? 8 : NP <= 6 ? 4 : NP <= 8 ? 3 : 2; };
// The staged dW kernel gathers the rows of IDC of a wave's ids together, U rows at a
// time. For 16-bit rows of up to 768 elements one id and 4 rows keep it within 64 VGPRs:
// two 16-wave workgroups per CU, so config 2's 477 workgroups run in one round instead
// of two (measured: 4 ids x 6 rows at 128 VGPRs, 55.0 us for the backward; 1 x 4, 49.8).
template <typename T, int NP> struct DwBatch {
  static constexpr int IDC = sizeof(T) == 2 ? 1 : NP > 3 ? 1 : 2;
  static constexpr int U = sizeof(T) == 2 && NP <= 3 ? 4 : IDC > 1 ? 6 : Batch<NP>::U;
};
// Register passes of the staged dW kernel: at most 8 (16-bit) or 4 (fp32), so that one
// id's accumulators and a batch of rows fit 128 VGPRs; longer rows loop over D.
template <typename T, int NP> struct DwPasses {
  static constexpr int CAP = sizeof(T) == 2 ? 8 : 4;
  static constexpr int value = NP < CAP ? NP : CAP;
};

// ---- dH ---------------------------------------------------------------------
// A row of D elements is cut into slices of DH_LANES 16-byte chunks, and 16 lanes (one DPP
// row) sum one slice of one row, a chunk each, over the row's entries. The lanes look up 16
// entries together, one each, and hand them round with row broadcasts; then the 16 W chunks
// are loaded, 256 bytes of a W row per lane group.
// What bounds it: with dense gradients the W rows' way from the MALL into the L2s (every
// entry's row is read once, 5.3 to 6.5 TB/s), with sparse ones the round trips of the longest row. So
// many lane groups are in flight, each with 16 rows of W.
constexpr int DH_LANES = 16;
constexpr int DH_WAVES = 4;
constexpr int DH_GROUPS = 64 / DH_LANES * DH_WAVES;  // lane groups (rows) of a workgroup

template <typename T> struct Chunk {
  static constexpr int E = 16 / (int)sizeof(T);  // elements of a 16-byte chunk
  static constexpr int COLS = DH_LANES * E;      // columns of a slice
};
template <typename T>
__device__ __forceinline__ void chunk_f32(const u32x4& c, float* f);
template <> __device__ __forceinline__ void chunk_f32<float>(const u32x4& c, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(c[i]);
}
template <> __device__ __forceinline__ void chunk_f32<bf16>(const u32x4& c, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(c[i] << 16);
    f[2 * i + 1] = __uint_as_float(c[i] & 0xffff0000u);
  }
}
template <> __device__ __forceinline__ void chunk_f32<f16>(const u32x4& c, float* f) {
  const f16x8 h = __builtin_bit_cast(f16x8, c);
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = (float)h[i];
}

// Lane U of the 16-lane row, to all its lanes (which must be active together).
template <int U> __device__ __forceinline__ uint32_t row_bcast(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x150 + U, 0xF, 0xF, true);  // row_newbcast:U
}
template <int I, int N, typename F> __device__ __forceinline__ void static_for(F f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// The entries of one dH row, spread over the batch row's runs: lane l of the group holds run
// l's. Entry i of the row (ids ascending) lies in the run q that holds the i-th of the
// running total, at place base_q + i of the batch row's runs.
struct RowEntries {
  int incl, base, total;
  __device__ __forceinline__ void load(const int* off, int runs, int cap, int l) {
    const int o0 = l < runs ? off[l] : 0, o1 = l < runs ? off[runs + l] : 0;
    incl = o1 - o0;
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xF, 0xF, true);  // row_shr:1
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xF, 0xF, true);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xF, 0xF, true);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xF, 0xF, true);
    base = l * cap + o0 - (incl - (o1 - o0));
    total = (int)row_bcast<15>((uint32_t)incl);
  }
  __device__ __forceinline__ int place(int i, int runs) const {
    int q = 0;
    static_for<0, 8>([&](auto k) { q += (int)row_bcast<decltype(k)::value>((uint32_t)incl) <= i ? 1 : 0; });
    if (runs > 8)  // uniform
      static_for<8, 15>([&](auto k) { q += (int)row_bcast<decltype(k)::value>((uint32_t)incl) <= i ? 1 : 0; });
    return i + __builtin_amdgcn_ds_bpermute((((int)threadIdx.x & 48) + min(q, 15)) * 4, base);
  }
};

// 16 entries of a row, one per lane: g' (0 past the row's end) and the place of the W row in
// 16-byte units (the last entry's past its end). WIDE: a W of 64 GiB or more, whose places need
// more than 32 bits; the second half's broadcasts cost 1.5% (16 x 256 dense bf16 rows), so
// smaller ones do without.
template <bool WIDE> struct Entries {
  uint32_t lo, hi;
  float g;
  __device__ __forceinline__ void load(const int2* run, const RowEntries& re, int runs, int e,
                                       uint64_t row16, int l) {
    const int2 x = run[re.place(min(e + l, re.total - 1), runs)];
    if constexpr (WIDE) {
      const uint64_t at = (uint64_t)(uint32_t)x.x * row16;
      lo = (uint32_t)at;
      hi = (uint32_t)(at >> 32);
    } else {
      lo = (uint32_t)x.x * (uint32_t)row16;
    }
    g = e + l < re.total ? __int_as_float(x.y) : 0.0f;
  }
  // Byte offset of entry U's W row.
  template <int U> __device__ __forceinline__ uint64_t at() const {
    uint64_t u = row_bcast<U>(lo);
    if constexpr (WIDE) u |= (uint64_t)row_bcast<U>(hi) << 32;
    return u << 4;
  }
};
constexpr uint64_t DH_WIDE_16 = 1ull << 32;  // 16-byte units of W from which on it is WIDE

// The partials P of the DH_BATCHes of entries 0 .. N - 1 over one chunk of their W rows (wp:
// the chunk in row 0), handed to put(batch, P) in order. With MASKED only the first `left`
// count; the others add 0 * 0, which leaves the sums as they are.
template <typename T, bool MASKED, int N, bool WIDE, typename Put>
__device__ __forceinline__ void dh_partials(const char* wp, const Entries<WIDE>& en, int left, Put put) {
  constexpr int E = Chunk<T>::E;
  u32x4 w[N];
  static_for<0, N>([&](auto u) {
    w[u] = *(const u32x4*)(wp + en.template at<decltype(u)::value>());
  });
  static_for<0, N / DH_BATCH>([&](auto a) {
    float P[E];
#pragma unroll
    for (int i = 0; i < E; ++i) P[i] = 0.0f;
    static_for<0, DH_BATCH>([&](auto k) {
      constexpr int u = decltype(a)::value * DH_BATCH + decltype(k)::value;
      const float g = __uint_as_float(row_bcast<u>(__float_as_uint(en.g)));
      u32x4 x = w[u];
      if (MASKED && u >= left) x = u32x4{0u, 0u, 0u, 0u};
      float f[E];
      chunk_f32<T>(x, f);
#pragma unroll
      for (int i = 0; i < E; ++i) P[i] = __builtin_fmaf(g, f[i], P[i]);
    });
    put(decltype(a)::value, P);
  });
}
// The same for the last `left` < DH_LANES entries, no more of them loaded than a few.
template <typename T, bool WIDE, typename Put>
__device__ __forceinline__ void dh_partials_tail(const char* wp, const Entries<WIDE>& en, int left, Put put) {
  if (left > 8) dh_partials<T, true, 16>(wp, en, left, put);
  else if (left > 4) dh_partials<T, true, 8>(wp, en, left, put);
  else dh_partials<T, true, 4>(wp, en, left, put);
}

template <typename O, int E>
__device__ __forceinline__ void store_chunk(O* out, const float* a) {
#pragma unroll
  for (int i = 0; i < E; i += 4) store4(out + i, f32x4{a[i], a[i + 1], a[i + 2], a[i + 3]});
}

// Hot rows: a lane group sums a row serially, so one that holds many times the entries of
// the others (a [CLS]-like position wins most ids), or any row of a launch with few rows,
// would outlast the launch. A workgroup's lane groups therefore share such rows: each step
// every group computes the batch partials of 16 consecutive entries into LDS, and the
// slice's columns add them in batch order: the same sums. A workgroup takes DH_GROUPS rows,
// of which those past max(HOT_MIN, HOT_REL times its mean) are shared, or one row, which is
// unless it is short (HOT_FEW).
constexpr int HOT_MIN = 128;
constexpr int HOT_REL = 4;
constexpr int HOT_FEW = 32;
constexpr int HOT_NB = DH_LANES / DH_BATCH;  // partials per lane group and step

// A row's partials are summed in blocks of FOLD entries, those in blocks of FOLD2 and these in
// order: a row may hold every id, and one chain over thousands of them has the larger error. fp32
// dH against fp64, rms, one chain -> these blocks (the kernels before, per-wave parts):
// 3 x 60 x 1024 x 180001 5.6e-7 -> 0.63e-7 (1.8e-7), 40 x 20 x 1024 x 40001 6.0e-7 -> 0.76e-7
// (2.3e-7), 2 x 50 x 772 x 200000 with 5% of the gradients 1.3e-7 -> 0.85e-7 (0.94e-7); the time
// is the same.
constexpr int FOLD = 64, FOLD2 = 1024;

template <typename T>
struct HotSmem {
  __attribute__((aligned(16))) float part[DH_GROUPS * HOT_NB][Chunk<T>::COLS];
  int total[DH_GROUPS];
};

template <typename T, typename O, bool WIDE>
__global__ __launch_bounds__(64 * DH_WAVES) void bwd_dh_kernel(
    const T* __restrict__ W, const int* __restrict__ off, const int2* __restrict__ run,
    O* __restrict__ dH, int B, int S, int D, int V, int runs, int cap, int S_row, int n_slices, int n16,
    int dense, int hot_min) {
  constexpr int E = Chunk<T>::E;
  static_assert(Chunk<T>::COLS <= 64 * DH_WAVES, "one thread per column");
  static_assert(FOLD % DH_LANES == 0 && DH_GROUPS * DH_LANES % FOLD == 0 &&
                    FOLD2 % (DH_GROUPS * DH_LANES) == 0,
                "blocks of whole steps");
  __shared__ HotSmem<T> sm;
  const int slice = (int)blockIdx.x % n_slices, blk = (int)blockIdx.x / n_slices;
  const int tid = threadIdx.x, grp = tid / DH_LANES, l = tid % DH_LANES;
  // n16 workgroups of DH_GROUPS rows a slice, then, with dense >= 0, one for each row: a batch
  // row's positions go to those where it holds more than `dense` entries (dh_dense).
  const bool single = blk >= n16;
  const int rpw = single ? 1 : DH_GROUPS;
  auto many_entries = [&](int64_t b) {  // (lane l of each group adds run l's)
    int n = l < runs ? off[(b * (S + 1) + S) * runs + l] : 0;
    n += __builtin_amdgcn_update_dpp(0, n, 0x111, 0xF, 0xF, true);  // row_shr:1
    n += __builtin_amdgcn_update_dpp(0, n, 0x112, 0xF, 0xF, true);
    n += __builtin_amdgcn_update_dpp(0, n, 0x114, 0xF, 0xF, true);
    n += __builtin_amdgcn_update_dpp(0, n, 0x118, 0xF, 0xF, true);
    return (int)row_bcast<15>((uint32_t)n) > dense;
  };
  const int64_t n_rows = (int64_t)B * S, row0 = single ? blk - n16 : (int64_t)blk * DH_GROUPS;
  if (single && !many_entries(row0 / S)) return;  // workgroup-uniform
  const uint64_t row16 = (uint64_t)D * sizeof(T) / 16;  // 16-byte units per row
  const int d0 = slice * Chunk<T>::COLS;
  // Lanes past the row's end work on its last chunk (the row broadcasts need them) and do not
  // store.
  const int d = d0 + l * E;
  const char* wp = (const char*)(W + min(d, D - E));
  auto entries_of = [&](int64_t row, RowEntries& re) {  // returns the batch row's runs
    const int64_t b = row / S;
    re.load(off + (b * (S + 1) + (row - b * S)) * runs, runs, cap, l);
    return run + b * V;
  };
  auto out_of = [&](int64_t row) {
    const int64_t b = row / S;
    return dH + (b * S_row + (row - b * S)) * D;
  };
  bool live = grp < rpw && row0 + grp < n_rows;
  if (live && !single && dense >= 0) live = !many_entries((row0 + grp) / S);  // uniform in a group
  RowEntries re;
  re.total = 0;
  const int2* rb = nullptr;
  if (live) rb = entries_of(row0 + grp, re);
  if (l == 0) sm.total[grp] = re.total;
  __syncthreads();
  int lim = HOT_FEW;
  if (rpw == DH_GROUPS) {
    int sum = 0;
#pragma unroll
    for (int k = 0; k < DH_GROUPS; ++k) sum += sm.total[k];
    lim = max(HOT_MIN, HOT_REL * (sum / DH_GROUPS));
  }
  if (hot_min >= 0) lim = hot_min;
  if (live && re.total <= lim) {
    float acc[E], sum[E], all[E];
#pragma unroll
    for (int i = 0; i < E; ++i) acc[i] = sum[i] = all[i] = 0.0f;
    if (re.total > 0) {
      auto add = [&](int, const float* P) {
#pragma unroll
        for (int i = 0; i < E; ++i) acc[i] += P[i];
      };
      Entries<WIDE> next;
      next.load(rb, re, runs, 0, row16, l);
      int e = 0;
      for (; e + DH_LANES <= re.total; e += DH_LANES) {
        const Entries<WIDE> en = next;
        next.load(rb, re, runs, e + DH_LANES, row16, l);
        dh_partials<T, false, DH_LANES>(wp, en, DH_LANES, add);
        if ((e + DH_LANES) % FOLD == 0)
#pragma unroll
          for (int i = 0; i < E; ++i) {
            sum[i] += acc[i];
            acc[i] = 0.0f;
          }
        if ((e + DH_LANES) % FOLD2 == 0)
#pragma unroll
          for (int i = 0; i < E; ++i) {
            all[i] += sum[i];
            sum[i] = 0.0f;
          }
      }
      if (e < re.total) dh_partials_tail<T>(wp, next, re.total - e, add);
#pragma unroll
      for (int i = 0; i < E; ++i) all[i] += sum[i] + acc[i];
    }
    if (d < D) store_chunk<O, E>(out_of(row0 + grp) + d, all);
  }
  for (int k = 0; k < rpw; ++k) {
    const int n = __builtin_amdgcn_readfirstlane(sm.total[k]);
    if (n <= lim) continue;  // workgroup-uniform
    RowEntries rk;
    const int2* rbk = entries_of(row0 + k, rk);
    float sum = 0.0f, all = 0.0f;  // column `tid` of the slice
    Entries<WIDE> next;
    next.load(rbk, rk, runs, grp * DH_LANES, row16, l);
    for (int e0 = 0; e0 < n; e0 += DH_GROUPS * DH_LANES) {
      const int e = e0 + grp * DH_LANES;
      const Entries<WIDE> en = next;
      next.load(rbk, rk, runs, e + DH_GROUPS * DH_LANES, row16, l);
      if (e < n) {
        auto put = [&](int p, const float* P) {
#pragma unroll
          for (int j = 0; j < E; j += 4)
            *(f32x4*)&sm.part[grp * HOT_NB + p][l * E + j] = f32x4{P[j], P[j + 1], P[j + 2], P[j + 3]};
        };
        if (n - e >= DH_LANES) dh_partials<T, false, DH_LANES>(wp, en, DH_LANES, put);
        else dh_partials_tail<T>(wp, en, n - e, put);
      }
      __syncthreads();
      const int m = min(DH_GROUPS * HOT_NB, (n - e0 + DH_BATCH - 1) / DH_BATCH);
      if (tid < Chunk<T>::COLS)
        for (int j0 = 0; j0 < m; j0 += FOLD / DH_BATCH) {
          float acc = 0.0f;
          for (int j = j0; j < min(m, j0 + FOLD / DH_BATCH); ++j) acc += sm.part[j][tid];
          sum += acc;
        }
      if ((e0 + DH_GROUPS * DH_LANES) % FOLD2 == 0 || e0 + DH_GROUPS * DH_LANES >= n) {
        all += sum;
        sum = 0.0f;
      }
      __syncthreads();  // the partials are rewritten next step
    }
    if (tid < Chunk<T>::COLS && d0 + tid < D) out_of(row0 + k)[d0 + tid] = from_f32<O>(all);
  }
}

// Entries (b_i, v) for N batch rows (b_i >= B or v >= V: inactive): g' (0 if inactive) and
// s. Three raw loads per row, issued together; then the mask of the candidates, issued
// together; then the coefficients. Inactive entries get s = 0.
template <typename T, typename RT, int N>
__device__ __forceinline__ void entries_n(const T* grad, const RT* reps, const int32_t* idx,
                                          const void* mask, int mdt, const int* bs, int v, int B,
                                          int S, int V, float* g, int* s) {
  T gr[N];
  RT rr[N];
  int ss[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int64_t o = (int64_t)min(bs[i], B - 1) * V + min(v, V - 1);
    gr[i] = grad[o];
    rr[i] = reps[o];
    ss[i] = idx[o];
  }
  bool cand[N];
  int64_t moff[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    cand[i] = bs[i] < B && v < V && to_f32(rr[i]) > 0.0f && ss[i] >= 0 && ss[i] < S &&
              to_f32(gr[i]) != 0.0f;
    moff[i] = cand[i] ? (int64_t)bs[i] * S + ss[i] : 0;
  }
  float mv[N];
  load_mask_n<N>(mask, mdt, moff, mv);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const bool act = cand[i] && mv[i] != 0.0f;
    g[i] = act ? to_f32(gr[i]) * expf(-to_f32(rr[i])) * mv[i] : 0.0f;
    s[i] = act ? ss[i] : 0;
  }
}

// ---- dW and dbias -------------------------------------------------------------
// One wave per vocab row v: lanes hold batch rows b (64 per pass), a ballot lists the
// active ones, and their H rows are gathered in ascending b, two at a time. Lanes past the
// row end load the row's last group (D >= 4 whenever D > 0), so the loads carry no per-lane
// condition and are in flight together; those lanes' sums are never stored.
template <typename T, typename O, int NP, typename RT>
__global__ __launch_bounds__(256) void bwd_dw_kernel(
    const T* __restrict__ grad, const RT* __restrict__ reps,
    const int32_t* __restrict__ idx, const void* __restrict__ mask, int mdt,
    const T* __restrict__ H, O* __restrict__ dW, O* __restrict__ dbias, int B, int S, int D,
    int V) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int v = blockIdx.x * 4 + wave;
  if (v >= V) return;
  const int dend = max(D, 1);  // one pass even when D == 0, for dbias
  for (int d0 = 0; d0 < dend; d0 += NP * 256) {
    f32x4 acc[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) acc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.0f;
    for (int b0 = 0; b0 < B; b0 += 64) {
      const int bb = b0 + lane;
      float g;
      int s;
      entries_n<T, RT, 1>(grad, reps, idx, mask, mdt, &bb, v, B, S, V, &g, &s);
      uint64_t pending = __ballot(g != 0.0f);
      while (pending) {
        const int l0 = __ffsll((unsigned long long)pending) - 1;
        pending &= pending - 1;
        const int s0 = __builtin_amdgcn_readlane(s, l0);
        const float g0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), l0));
        const T* h0 = H + ((int64_t)(b0 + l0) * S + s0) * D;
        bsum += g0;
        if (pending) {
          const int l1 = __ffsll((unsigned long long)pending) - 1;
          pending &= pending - 1;
          const int s1 = __builtin_amdgcn_readlane(s, l1);
          const float g1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), l1));
          const T* h1 = H + ((int64_t)(b0 + l1) * S + s1) * D;
          bsum += g1;
          if (D > 0) {  // (H may be null without columns)
            f32x4 x0[NP], x1[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) {
              const int d = min(d0 + p * 256 + lane * 4, D - 4);
              x0[p] = load4(h0 + d);
              x1[p] = load4(h1 + d);
            }
#pragma unroll
            for (int p = 0; p < NP; ++p) acc[p] += g0 * x0[p] + g1 * x1[p];
          }
        } else if (D > 0) {
          f32x4 x0[NP];
#pragma unroll
          for (int p = 0; p < NP; ++p) x0[p] = load4(h0 + min(d0 + p * 256 + lane * 4, D - 4));
#pragma unroll
          for (int p = 0; p < NP; ++p) acc[p] += g0 * x0[p];
        }
      }
    }
    if (d0 == 0 && dbias != nullptr && lane == 0) dbias[v] = from_f32<O>(bsum);
    if (dW != nullptr) {
      O* out = dW + (int64_t)v * D;
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int d = d0 + p * 256 + lane * 4;
        if (d < D) store4(out + d, acc[p]);
      }
    }
  }
}

// ---- dW and dbias, staged (B <= DW_STAGE_B) ---------------------------------
constexpr int DW_STAGE_B = 128;
// The staged dW: a workgroup of NW waves owns NIDS consecutive vocab ids (NIDS / NW per
// wave). It loads G, reps and I of all batch rows for them (each load instruction reads
// NIDS consecutive elements of 64 / NIDS rows) and keeps g' (0 = inactive) and I in LDS;
// then each wave handles its ids: lanes scan the batch rows, ballots list the active
// ones, and their H rows are gathered up to U at a time and accumulated, each id in
// ascending b. I is kept as 16 bits: the staged kernels take S <= DW_STAGE_S.
constexpr int DW_WAVES = 16;  // of the wide kernel
constexpr int DW_IDS = 4 * BK_WAVES;  // ids of a staged workgroup
constexpr int DW_LD = DW_STAGE_B + 1;  // odd row stride: conflict-free column and row access
constexpr int DW_STAGE_S = 1 << 16;

template <typename T, typename RT, int NIDS, int NW, int LD = DW_LD>
__device__ __forceinline__ void dw_stage(float* gl, uint16_t* sl, const T* __restrict__ grad,
                                         const RT* __restrict__ reps,
                                         const int32_t* __restrict__ idx,
                                         const void* __restrict__ mask, int mdt, int B, int S,
                                         int V, int v0, int wave, int lane) {
  constexpr int RPL = 64 / NIDS;  // batch rows per load instruction
  const int idl = lane % NIDS, rsub = lane / NIDS;
  // Each wave takes 2 * RPL batch rows at a time, their loads in flight together.
  for (int b0 = wave * 2 * RPL; b0 < B; b0 += NW * 2 * RPL) {
    const int bs[2] = {b0 + rsub, b0 + RPL + rsub};
    float g[2];
    int s[2];
    entries_n<T, RT, 2>(grad, reps, idx, mask, mdt, bs, v0 + idl, B, S, V, g, s);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (bs[i] < B) {
        gl[idl * LD + bs[i]] = g[i];
        sl[idl * LD + bs[i]] = (uint16_t)s[i];
      }
    }
  }
}

template <typename T, typename O, int NP, typename RT, int NIDS, int NW, int LD = DW_LD>
__device__ __forceinline__ void dw_gather(const float* gl, const uint16_t* sl,
                                          const T* __restrict__ H, O* __restrict__ dW,
                                          O* __restrict__ dbias, int B, int S, int D, int V,
                                          int v0, int wave, int lane) {
  // IDC of the wave's ids at a time are gathered together: batches of U rows are taken
  // from their active (id, b) pairs in (id, b) order, so each id still sums its rows in
  // ascending b.
  constexpr int IDS = NIDS / NW;  // ids per wave
  constexpr int IDC = DwBatch<T, NP>::IDC;
  constexpr int U = DwBatch<T, NP>::U;
  static_assert(IDS % IDC == 0, "ids per wave");
  const int dend = max(D, 1);  // one pass even when D == 0, for dbias
  for (int i0 = 0; i0 < IDS; i0 += IDC) {
    if (v0 + wave * IDS + i0 >= V) break;
    for (int d0 = 0; d0 < dend; d0 += NP * 256) {
      f32x4 acc[IDC][NP];
      float bsum[IDC];
#pragma unroll
      for (int i = 0; i < IDC; ++i) {
        bsum[i] = 0.0f;
#pragma unroll
        for (int p = 0; p < NP; ++p) acc[i][p] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      for (int b0 = 0; b0 < B; b0 += 64) {
        const int bb = b0 + lane;
        float g[IDC];
        int s[IDC];
        uint64_t pend[IDC];
        int left = 0;
#pragma unroll
        for (int i = 0; i < IDC; ++i) {
          const int vl = wave * IDS + i0 + i;
          const bool in = bb < B && v0 + vl < V;
          g[i] = in ? gl[vl * LD + bb] : 0.0f;
          s[i] = in ? (int)sl[vl * LD + bb] : 0;
          pend[i] = __ballot(g[i] != 0.0f);
          left += __popcll(pend[i]);
        }
        while (left > 0) {
          const int nb = min(U, left);  // rows in this batch (uniform)
          left -= nb;
          Raw4<T> x[U][NP];
          float gu[U];
          int iu[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            gu[u] = 0.0f;
            iu[u] = -1;
            if (u < nb) {
              int l = 0, su = 0;
              float gg = 0.0f;
              bool taken = false;
#pragma unroll
              for (int i = 0; i < IDC; ++i) {  // the first id with rows left (uniform)
                if (!taken && pend[i] != 0) {
                  taken = true;
                  iu[u] = i;
                  l = __ffsll((unsigned long long)pend[i]) - 1;
                  pend[i] &= pend[i] - 1;
                  gg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g[i]), l));
                  su = __builtin_amdgcn_readlane(s[i], l);
                }
              }
              gu[u] = gg;
              const T* hr = H + ((int64_t)(b0 + l) * S + su) * D;
#pragma unroll
              for (int p = 0; p < NP; ++p) {
                const int d = d0 + p * 256 + lane * 4;
                if (d < D) x[u][p].load(hr + d);
                else x[u][p].zero();
              }
            }
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int i = 0; i < IDC; ++i) {
              if (iu[u] == i) {
                bsum[i] += gu[u];
#pragma unroll
                for (int p = 0; p < NP; ++p) acc[i][p] += gu[u] * x[u][p].f();
              }
            }
          }
        }
      }
#pragma unroll
      for (int i = 0; i < IDC; ++i) {
        const int v = v0 + wave * IDS + i0 + i;
        if (v >= V) break;
        if (d0 == 0 && dbias != nullptr && lane == 0) dbias[v] = from_f32<O>(bsum[i]);
        if (dW != nullptr) {
          O* out = dW + (int64_t)v * D;
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            const int d = d0 + p * 256 + lane * 4;
            if (d < D) store4(out + d, acc[i][p]);
          }
        }
      }
    }
  }
}

// The bucketing's workgroups (n_bucket of them), then dW's, DW_IDS ids each: dW reads only the
// inputs, so both run side by side. Either part may be empty. grad, reps, idx and mask start
// at the pass's first batch row.
template <typename T, typename O, int NP, typename RT>
__global__ __launch_bounds__(64 * BK_WAVES) void bwd_bucket_dw_kernel(
    const T* __restrict__ grad, const RT* __restrict__ reps, const int32_t* __restrict__ idx,
    const void* __restrict__ mask, int mdt, const T* __restrict__ H, O* __restrict__ dW,
    O* __restrict__ dbias, int B, int S, int D, int V, int n_bucket, int runs, int cap, int win_s0,
    int win_s, int* __restrict__ off, int2* __restrict__ run) {
  const int blk = blockIdx.x;
  if (blk < n_bucket) {  // workgroup-uniform
    bucket_run<T, RT>(grad, reps, idx, mask, mdt, win_s, V, blk / runs, blk % runs, runs, cap, off, run,
                      win_s0, S);
    return;
  }
  float* gl = (float*)sparton_bwd_smem;
  uint16_t* sl = (uint16_t*)(gl + DW_IDS * DW_LD);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int v0 = (blk - n_bucket) * DW_IDS;
  dw_stage<T, RT, DW_IDS, BK_WAVES>(gl, sl, grad, reps, idx, mask, mdt, B, S, V, v0, wave, lane);
  __syncthreads();
  dw_gather<T, O, NP, RT, DW_IDS, BK_WAVES>(gl, sl, H, dW, dbias, B, S, D, V, v0, wave, lane);
}

// dW / dbias for DW_STAGE_B < B <= DW_WIDE_B and S <= DW_STAGE_S: the staged kernel with
// fewer ids per workgroup, so that every batch row of them fits LDS (NIDS ids x (ROWS + 1)
// x 6 bytes, ~99 KB: 64 ids up to 256 rows, 32 up to 512, 16 up to 1024). The rows are
// staged once and each id sums its rows in ascending b, as above.
constexpr int DW_WIDE_IDS_ROWS = 16384;  // NIDS x ROWS
constexpr int DW_WIDE_B = 1024;
template <typename T, typename O, int NP, typename RT, int NIDS>
__global__ __launch_bounds__(64 * DW_WAVES) void bwd_dw_wide_kernel(
    const T* __restrict__ grad, const RT* __restrict__ reps,
    const int32_t* __restrict__ idx, const void* __restrict__ mask, int mdt,
    const T* __restrict__ H, O* __restrict__ dW, O* __restrict__ dbias, int B, int S, int D,
    int V) {
  constexpr int LD = DW_WIDE_IDS_ROWS / NIDS + 1;  // odd: conflict-free
  __shared__ float gl[NIDS * LD];
  __shared__ uint16_t sl[NIDS * LD];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int v0 = blockIdx.x * NIDS;
  dw_stage<T, RT, NIDS, DW_WAVES, LD>(gl, sl, grad, reps, idx, mask, mdt, B, S, V, v0, wave, lane);
  __syncthreads();
  dw_gather<T, O, NP, RT, NIDS, DW_WAVES, LD>(gl, sl, H, dW, dbias, B, S, D, V, v0, wave, lane);
}

// Register passes for a row of D elements (4 per lane, 256 per pass), capped at MAX_NP
// (longer rows loop over D in chunks of MAX_NP * 256).
static int passes_for(int64_t D) {
  return (int)std::min<int64_t>(MAX_NP, std::max<int64_t>(1, cdiv(D, 256)));
}

// From this many rows on every dH workgroup takes 16: they fill the chip then. A launch of fewer
// also holds a workgroup for each row, last, and a batch row's positions get one each where it
// holds more than 48 entries a position, or less in proportion under 1024 rows; the workgroups of
// the other kind end at once. Backward with bf16 rows of 768, V = 30522, at 16 rows / 1 row a
// workgroup: 12 x 150 with 9 entries a position 42 / 54 us, 38 61 / 66, 190 180 / 140; 16 x 64 with
// 22 45 / 50, 90 76 / 62, 440 248 / 164; 16 x 32 with 9 34 / 40, 45 43 / 44, 180 75 / 59; 4 x 64
// with 24 36 / 33.
constexpr int64_t DH_MANY_ROWS = 2048;
static int64_t dh_dense(int64_t S, int64_t rows) { return S * 48 * std::min<int64_t>(rows, 1024) / 1024; }
static_assert(DH_MAX_WG == MAX_THREADS / (64 * DH_WAVES), "workgroups of a dH launch");
// SPARTON_BWD_HOT_MIN sets the number of entries past which a row is shared (tests compare
// shared and unshared rows).
static int dh_hot_min() {
  const char* e = getenv("SPARTON_BWD_HOT_MIN");
  return e != nullptr ? atoi(e) : -1;
}
// ---- few dH rows (B * S <= FEW_ROWS) ------------------------------------------------------
//
// With few dH rows every W row serves several of them (config 1: each of the 30522 ids is
// active in both batch rows), so gathering W rows per dH row reads W once per batch row.
// Here one launch does all of the backward: a workgroup owns a range of vocabulary ids and
// a 256-column slice of D, and walks the range tile by tile (FEW_TILE ids), reading each W
// row of its slice once.
//   dH: wave w holds dH rows FEW_RPW w .. FEW_RPW w + FEW_RPW - 1 of the slice in registers
//   (lane l: columns 4 l .. 4 l + 3), indexed statically. A row b S + s takes the tile's
//   ids whose entry (b, id) is active with index s (one ballot), in ascending v, so its
//   partial sum runs over the range in ascending v; bwd_few_sum_kernel adds the ranges'
//   partials in range order. These sums are this path's own order (they agree with every
//   other path to fp32 rounding, not bitwise).
//   dW, dbias: wave w also owns the tile's ids 8 w .. 8 w + 7 and sums their active entries'
//   H rows (the slice of all B S rows sits in LDS) in ascending b, exactly as the staged dW
//   kernel does (same operations in the same order: the results are bitwise the same).
//
// The tile's W rows travel HBM -> registers -> LDS: they are loaded during the previous
// tile and written to LDS at the start of this one, so the loads overlap a whole tile's
// work. (Direct-to-LDS copies would not: the compiler cannot tell the copy's target from
// the buffer being read and waits for every copy before each LDS read.)
constexpr int FEW_ROWS = 64;                          // dH rows held per workgroup
constexpr int FEW_TILE = 64;                          // vocabulary ids per tile (one per lane)
constexpr int FEW_WAVES = 8;
constexpr int FEW_THREADS = 64 * FEW_WAVES;
constexpr int FEW_COLS = 256;                         // columns of D per slice (4 per lane)
constexpr int FEW_RPW = FEW_ROWS / FEW_WAVES;         // dH rows per wave
constexpr int FEW_IPW = FEW_TILE / FEW_WAVES;         // dW ids per wave
constexpr int FEW_IDC = 8;                            // dW ids summed together
constexpr int FEW_NJ = FEW_ROWS * FEW_TILE / FEW_THREADS;  // entry rounds: batch rows per wave
constexpr int FEW_ES_LD = 68;   // bytes per id of the index table: 17 words, odd, so a wave's
                                // 64 ids fall in 64 different banks
constexpr uint8_t FEW_NONE = 0xff;  // index table: inactive entry (S <= FEW_ROWS < 255)

// SPARTON_BWD_FEW=0 sends few-row batches to the bucketing and bwd_dh_kernel instead (tests
// compare the two).
static bool few_enabled() {
  const char* e = getenv("SPARTON_BWD_FEW");
  return e == nullptr || strcmp(e, "0") != 0;
}

struct FewPlan {
  bool fits;       // the shape qualifies (the workspace is sized for it whatever the switch)
  int slices, ranges, range_len;
  size_t part_bytes;
};
static FewPlan few_plan(int64_t B, int64_t S, int64_t D, int64_t V) {
  FewPlan p{};
  p.fits = B * S > 0 && B * S <= FEW_ROWS && D > 0 && V > 0;
  if (!p.fits) return p;
  p.slices = (int)cdiv(D, FEW_COLS);
  // about one workgroup per CU: each reads range_len W rows of its slice once
  const int64_t want = std::max<int64_t>(1, 256 / p.slices);
  p.range_len = (int)(cdiv(cdiv(V, FEW_TILE), want) * FEW_TILE);
  p.ranges = (int)cdiv(V, p.range_len);
  p.part_bytes = (size_t)p.ranges * (size_t)(B * S) * (size_t)D * 4;
  return p;
}

// Workgroup barrier once this wave's LDS operations are complete. Global loads in flight
// (the next tile's, into registers) are not waited for; the memory clobber keeps the
// compiler from moving memory accesses across it.
__device__ __forceinline__ void few_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Rows of a matrix with row stride D, slice columns c0 .. c0 + FEW_COLS - 1, in 16-byte
// chunks: chunk q = i * FEW_THREADS + thread is row q / CPR, chunk q % CPR of the row, so
// consecutive threads read consecutive bytes. Chunks past D re-read the slice's first chunk
// (those columns are never stored); D * sizeof(T) is a multiple of 16.
template <typename T>
struct FewChunks {
  static constexpr int CPR = FEW_COLS * (int)sizeof(T) / 16;  // chunks per row
  static constexpr int PER = 16 / (int)sizeof(T);             // elements per chunk
  static __device__ __forceinline__ u32x4 load(const T* __restrict__ M, int row, int q, int D,
                                               int c0) {
    const int col = c0 + (q % CPR) * PER;
    return *(const u32x4*)(M + (int64_t)row * D + (col < D ? col : c0));
  }
};

// One tile's W rows (ids past V re-read id V-1: their entries are inactive), held in
// registers between their load and their store to LDS.
template <typename T>
struct FewStage {
  static constexpr int NL = FEW_TILE * FewChunks<T>::CPR / FEW_THREADS;  // chunks per thread
  u32x4 c[NL];
  __device__ __forceinline__ void load(const T* __restrict__ W, int v0, int V, int D, int c0,
                                       int t) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int q = i * FEW_THREADS + t;
      c[i] = FewChunks<T>::load(W, min(v0 + q / FewChunks<T>::CPR, V - 1), q, D, c0);
    }
  }
  __device__ __forceinline__ void store(T* wt, int t) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) ((u32x4*)wt)[i * FEW_THREADS + t] = c[i];
  }
};

template <typename T, typename O, typename RT>
__global__ __launch_bounds__(FEW_THREADS) void bwd_few_kernel(
    const T* __restrict__ grad, const RT* __restrict__ reps, const int32_t* __restrict__ idx,
    const void* __restrict__ mask, int mdt, const T* __restrict__ H, const T* __restrict__ W,
    float* __restrict__ part, O* __restrict__ dW, O* __restrict__ dbias, int B, int S, int D,
    int V, int slices, int range_len) {
  // Each table has one more row, of zeros (row FEW_TILE, FEW_ROWS): a pass points a row or
  // id with no entry left at it, and adding g' * w = +0 * +0 changes no sum.
  __shared__ __attribute__((aligned(16))) T wt[FEW_TILE + 1][FEW_COLS];  // the tile's W rows
  __shared__ __attribute__((aligned(16))) T hs[FEW_ROWS + 1][FEW_COLS];  // H's B*S rows, this slice
  __shared__ float eg[FEW_ROWS][FEW_TILE + 1];  // g' of entry (b, v0 + id) at [b][id], 0 = inactive
  __shared__ uint8_t es[FEW_TILE][FEW_ES_LD];       // its index s, FEW_NONE = inactive
  __shared__ float maskf[FEW_ROWS];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform: scalar registers, branches
  const int range = (int)blockIdx.x / slices, slice = (int)blockIdx.x - range * slices;
  const int c0 = slice * FEW_COLS;
  const int BS = B * S;
  const int v_beg = range * range_len, v_end = min(V, v_beg + range_len);
  const bool dw_on = dW != nullptr || dbias != nullptr;
  for (int i = t; i < BS; i += FEW_THREADS) maskf[i] = load_mask(mask, mdt, i);
  for (int i = t; i < FEW_COLS; i += FEW_THREADS) {
    wt[FEW_TILE][i] = T(0.0f);
    hs[FEW_ROWS][i] = T(0.0f);
  }
  for (int i = t; i < FEW_ROWS; i += FEW_THREADS) eg[i][FEW_TILE] = 0.0f;
  if (dW != nullptr) {  // (H may be absent when only dbias is asked for)
    for (int q = t; q < BS * FewChunks<T>::CPR; q += FEW_THREADS)
      ((u32x4*)&hs[0][0])[q] = FewChunks<T>::load(H, q / FewChunks<T>::CPR, q, D, c0);
  }
  // This wave's dH rows: batch row and index of each (rows past B*S take none).
  int rb[FEW_RPW], rs[FEW_RPW];
#pragma unroll
  for (int r = 0; r < FEW_RPW; ++r) {
    const int row = wave * FEW_RPW + r;
    rb[r] = row < BS ? row / S : 0;
    rs[r] = row < BS ? row - rb[r] * S : -1;
  }
  f32x4 acc[FEW_RPW];
#pragma unroll
  for (int r = 0; r < FEW_RPW; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The tile's W rows and entries (b, v0 + lane), loaded one tile ahead; round j of wave w
  // holds batch row b = FEW_WAVES j + w (B <= FEW_ROWS).
  FewStage<T> stage;
  T gr[FEW_NJ];
  RT rr[FEW_NJ];
  int sr[FEW_NJ];
  auto load_entries = [&](int v0) {
    const int v = min(v0 + lane, V - 1);
#pragma unroll
    for (int j = 0; j < FEW_NJ; ++j) {
      const int b = FEW_WAVES * j + wave;
      if (b < B) {  // uniform per wave
        const int64_t o = (int64_t)b * V + v;
        gr[j] = grad[o];
        rr[j] = reps[o];
        sr[j] = idx[o];
      }
    }
  };
  stage.load(W, v_beg, V, D, c0, t);
  load_entries(v_beg);
  const T* wcol = &wt[0][lane * 4];
  const int c = c0 + lane * 4;
  for (int v0 = v_beg; v0 < v_end; v0 += FEW_TILE) {
    // the previous tile's rows and ids are done: wt, eg and es are free
    few_barrier();
    stage.store(&wt[0][0], t);
    const bool more = v0 + FEW_TILE < v_end;
    // The next tile's W rows load under all of this tile's work; its entries load once
    // this tile's are used, below. (The next tile's first wait is for all of them, and for
    // this tile's dW stores: stores and loads share one counter.)
    if (more) stage.load(W, v0 + FEW_TILE, V, D, c0, t);
    const int v = v0 + lane;
#pragma unroll
    for (int j = 0; j < FEW_NJ; ++j) {
      const int b = FEW_WAVES * j + wave;
      if (b < B) {  // uniform per wave
        float gp;
        const int si = sr[j];
        const bool act = v < v_end && entry(gr[j], rr[j], si, maskf + b * S, S, &gp) &&
                         gp != 0.0f;
        eg[b][lane] = act ? gp : 0.0f;
        es[lane][b] = act ? (uint8_t)si : FEW_NONE;
      }
    }
    if (more) load_entries(v0 + FEW_TILE);
    few_barrier();
    // dW, dbias: this wave's ids, FEW_IDC at a time, pass k taking each id's k-th active
    // batch row (ascending); an id with none left takes the zero rows.
    if (dw_on) {
#pragma unroll 1
      for (int i0 = 0; i0 < FEW_IPW; i0 += FEW_IDC) {
        uint64_t p[FEW_IDC];
        int npass = 0;
#pragma unroll
        for (int i = 0; i < FEW_IDC; ++i) {
          const int il = wave * FEW_IPW + i0 + i;
          // eg holds +0.0 for every inactive entry
          p[i] = __ballot(lane < B && __float_as_int(eg[min(lane, FEW_ROWS - 1)][il]) != 0);
          npass = max(npass, __popcll(p[i]));
        }
        f32x4 ad[FEW_IDC];
        float bsum[FEW_IDC];
#pragma unroll
        for (int i = 0; i < FEW_IDC; ++i) {
          ad[i] = f32x4{0.f, 0.f, 0.f, 0.f};
          bsum[i] = 0.0f;
        }
        for (int k = 0; k < npass; ++k) {
          float g[FEW_IDC];
          f32x4 h[FEW_IDC];
#pragma unroll
          for (int i = 0; i < FEW_IDC; ++i) {
            const bool on = p[i] != 0;  // uniform
            const int b = on ? (int)__builtin_ctzll(p[i]) : 0;
            p[i] &= ~(1ull << b);
            const int iv = wave * FEW_IPW + i0 + i;
            g[i] = eg[b][on ? iv : FEW_TILE];
            const int hr = on ? b * S + (int)es[iv][b] : FEW_ROWS;
            h[i] = load4(&hs[hr][lane * 4]);
          }
#pragma unroll
          for (int i = 0; i < FEW_IDC; ++i) {
            ad[i] = f32x4{fmaf(g[i], h[i][0], ad[i][0]), fmaf(g[i], h[i][1], ad[i][1]),
                          fmaf(g[i], h[i][2], ad[i][2]), fmaf(g[i], h[i][3], ad[i][3])};
            bsum[i] += g[i];
          }
        }
#pragma unroll
        for (int i = 0; i < FEW_IDC; ++i) {
          const int vi = v0 + wave * FEW_IPW + i0 + i;
          if (vi < v_end) {
            if (dW != nullptr && c < D) store4(dW + (int64_t)vi * D + c, ad[i]);
            if (dbias != nullptr && slice == 0 && lane == 0) dbias[vi] = from_f32<O>(bsum[i]);
          }
        }
      }
    }
    // dH: this wave's rows, pass k taking each row's k-th id (ascending); a row with none
    // left takes the zero rows. Straight-line passes: the ids are scalar, the coefficients
    // come by broadcast LDS reads, and a pass's reads are independent of each other.
    {
      uint64_t m[FEW_RPW];
      int npass = 0;
#pragma unroll
      for (int r = 0; r < FEW_RPW; ++r) {
        m[r] = __ballot((int)es[lane][rb[r]] == rs[r]);
        npass = max(npass, __popcll(m[r]));
      }
      for (int k = 0; k < npass; ++k) {
        float g[FEW_RPW];
        f32x4 w[FEW_RPW];
#pragma unroll
        for (int r = 0; r < FEW_RPW; ++r) {
          const int id = m[r] != 0 ? (int)__builtin_ctzll(m[r]) : FEW_TILE;  // uniform
          m[r] &= ~(1ull << (id & 63));
          g[r] = eg[rb[r]][id];
          w[r] = load4(wcol + id * FEW_COLS);
        }
#pragma unroll
        for (int r = 0; r < FEW_RPW; ++r)
          acc[r] = f32x4{fmaf(g[r], w[r][0], acc[r][0]), fmaf(g[r], w[r][1], acc[r][1]),
                         fmaf(g[r], w[r][2], acc[r][2]), fmaf(g[r], w[r][3], acc[r][3])};
      }
    }
  }
  if (c < D) {
    float* out = part + (int64_t)range * BS * D + c;
#pragma unroll
    for (int r = 0; r < FEW_RPW; ++r) {
      const int row = wave * FEW_RPW + r;
      if (row < BS) *(f32x4*)(out + (int64_t)row * D) = acc[r];
    }
  }
}

// dH = the ranges' partial rows added in range order, in the output dtype. A workgroup
// takes 256 elements (4 per lane of a wave); its FEW_SUM_WAVES waves sum consecutive
// groups of the ranges, and the groups are added in order.
constexpr int FEW_SUM_WAVES = 8;
template <typename O>
__global__ __launch_bounds__(64 * FEW_SUM_WAVES) void bwd_few_sum_kernel(
    const float* __restrict__ part, O* __restrict__ dH, int64_t n, int ranges) {
  __shared__ f32x4 red[FEW_SUM_WAVES - 1][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t i = ((int64_t)blockIdx.x * 64 + lane) * 4;
  const int q = (ranges + FEW_SUM_WAVES - 1) / FEW_SUM_WAVES;
  const int k0 = min(ranges, wave * q), k1 = min(ranges, k0 + q);
  f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
  if (i < n) {  // n is a multiple of 4
    int k = k0;
    for (; k + 4 <= k1; k += 4) {
      f32x4 x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = *(const f32x4*)(part + (int64_t)(k + j) * n + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) s += x[j];
    }
    for (; k < k1; ++k) s += *(const f32x4*)(part + (int64_t)k * n + i);
  }
  if (wave > 0) red[wave - 1][lane] = s;
  __syncthreads();
  if (wave == 0 && i < n) {
#pragma unroll
    for (int w = 0; w < FEW_SUM_WAVES - 1; ++w) s += red[w][lane];
    store4(dH + i, s);
  }
}

// dW's workgroups run in the bucketing's launch
// (SPARTON_BWD_DW_MERGE=0 keeps them apart; tests compare the two).
constexpr int64_t DW_MERGE_S = 1024;
static bool dw_merge_on() {
  const char* e = getenv("SPARTON_BWD_DW_MERGE");
  return e == nullptr || strcmp(e, "0") != 0;
}

// The wide staged dW with 16 ids per workgroup (B <= DW_WIDE_B), for 16-bit types: fp32
// rows gather two ids at a time, which 16 ids over 16 waves cannot give. Returns whether it
// launched.
template <typename T, typename O, int DNP, typename RT>
static bool wide16(const T* g, const RT* r, const int32_t* idx, const void* mask, int mdt,
                   const T* H, O* dW, O* dbias, int64_t B, int64_t S, int64_t D, int64_t V,
                   hipStream_t st) {
  if constexpr (sizeof(T) == 2) {
    if (B <= DW_WIDE_B && S <= DW_STAGE_S) {
      hipLaunchKernelGGL((bwd_dw_wide_kernel<T, O, DNP, RT, 16>), dim3((unsigned)cdiv(V, 16)),
                         dim3(64 * DW_WAVES), 0, st, g, r, idx, mask, mdt, H, dW, dbias, (int)B,
                         (int)S, (int)D, (int)V);
      return true;
    }
  }
  return false;
}

template <typename T, typename O, int NP, typename RT>
static void launch_rows(const T* g, const RT* r, const int32_t* idx, const void* mask,
                        int mdt, const T* H, const T* W, O* dH, O* dW, O* dbias, void* ws,
                        int64_t B, int64_t S, int64_t D, int64_t V, hipStream_t st) {
  const FewPlan few = few_plan(B, S, D, V);
  if (few.fits && few_enabled() && dH != nullptr) {
    float* part = (float*)ws;
    hipLaunchKernelGGL((bwd_few_kernel<T, O, RT>), dim3((unsigned)(few.ranges * few.slices)),
                       dim3(FEW_THREADS), 0, st, g, r, idx, mask, mdt, H, W, part, dW, dbias,
                       (int)B, (int)S, (int)D, (int)V, few.slices, few.range_len);
    const int64_t n = B * S * D;
    hipLaunchKernelGGL((bwd_few_sum_kernel<O>), dim3((unsigned)cdiv(n, 256)), dim3(64 * FEW_SUM_WAVES),
                       0, st,
                       (const float*)part, dH, n, few.ranges);
    return;
  }
  constexpr int DNP = DwPasses<T, NP>::value;
  const bool need_dw = (dW != nullptr || dbias != nullptr) && V > 0;
  const bool staged = B <= DW_STAGE_B && S <= DW_STAGE_S;
  const size_t dw_lds = (size_t)DW_IDS * DW_LD * 6;
  const int n_dw = need_dw && staged ? (int)cdiv(V, DW_IDS) : 0;
  bool dw_done = false;
  if (dH != nullptr && B * S > 0 && D > 0) {
    // Batch rows in chunks and positions in windows (pass_of): each pass buckets the
    // entries of rows [b0, b0 + nb) and positions [s0, s0 + sw) (entries whose index lies
    // outside the window are inactive) and sums its dH rows, so every dH row is written by
    // exactly one pass. The workspace holds one pass; the passes reuse it in stream order.
    const Pass pass = pass_of(B, S, D);
    const int64_t Bc = pass.b, Sc = pass.s;
    const Layout L = layout(Bc, Sc, V);
    const Cut c = cut_ids(V);
    int* off = (int*)((char*)ws + L.off);
    int2* run = (int2*)((char*)ws + L.run);
    const int64_t n_slices = cdiv(D, Chunk<T>::COLS);
    for (int64_t b0 = 0; b0 < B; b0 += Bc) {
      const int64_t nb = std::min(Bc, B - b0);
      for (int64_t s0 = 0; s0 < S; s0 += Sc) {
        const int64_t sw = std::min(Sc, S - s0);
        const int nbk = (int)(nb * c.runs);
        // dW's workgroups join where the bucketing's counters take little more LDS than dW's.
        const bool with_dw = n_dw > 0 && S <= DW_MERGE_S && nb == B && nbk + (int64_t)n_dw <= BK_MAX_WG &&
                             dw_merge_on();
        const size_t lds = (size_t)(BK_WAVES + 1 + (BK_WAVES + 1) * sw) * 4;
        hipLaunchKernelGGL((bwd_bucket_dw_kernel<T, O, DNP, RT>), dim3((unsigned)(nbk + (with_dw ? n_dw : 0))),
                           dim3(64 * BK_WAVES), with_dw ? std::max(lds, dw_lds) : lds, st, g + b0 * V,
                           r + b0 * V, idx + b0 * V, (const char*)mask + b0 * S * mask_elem_bytes(mdt), mdt,
                           H, dW, dbias, (int)B, (int)S, (int)D, (int)V, nbk, (int)c.runs, (int)c.cap,
                           (int)s0, (int)sw, off, run);
        dw_done |= with_dw;
        const int64_t rows = nb * sw, n16 = cdiv(rows, DH_GROUPS);
        // (rows so long that a launch cannot hold a workgroup for each share them all)
        const bool singles = rows < DH_MANY_ROWS && (n16 + rows) * n_slices <= DH_MAX_WG;
        const bool wide = (uint64_t)V * ((uint64_t)D * sizeof(T) / 16) > DH_WIDE_16;
        hipLaunchKernelGGL((wide ? bwd_dh_kernel<T, O, true> : bwd_dh_kernel<T, O, false>),
                           dim3((unsigned)((n16 + (singles ? rows : 0)) * n_slices)),
                           dim3(64 * DH_WAVES), 0, st, W, (const int*)off, (const int2*)run,
                           dH + (b0 * S + s0) * D, (int)nb, (int)sw, (int)D, (int)V, (int)c.runs, (int)c.cap,
                           (int)S, (int)n_slices, (int)n16, singles ? (int)dh_dense(sw, rows) : -1, dh_hot_min());
      }
    }
  }
  if (need_dw && !dw_done) {
    if (staged)
      hipLaunchKernelGGL((bwd_bucket_dw_kernel<T, O, DNP, RT>), dim3((unsigned)n_dw), dim3(64 * BK_WAVES),
                         dw_lds, st, g, r, idx, mask, mdt, H, dW, dbias, (int)B, (int)S, (int)D, (int)V,
                         0, 1, 0, 0, 0, nullptr, nullptr);
    else if (B <= DW_WIDE_IDS_ROWS / 64 && S <= DW_STAGE_S)
      hipLaunchKernelGGL((bwd_dw_wide_kernel<T, O, DNP, RT, 64>), dim3((unsigned)cdiv(V, 64)),
                         dim3(64 * DW_WAVES), 0, st, g, r, idx, mask, mdt, H, dW, dbias, (int)B,
                         (int)S, (int)D, (int)V);
    else if (B <= DW_WIDE_IDS_ROWS / 32 && S <= DW_STAGE_S)
      hipLaunchKernelGGL((bwd_dw_wide_kernel<T, O, DNP, RT, 32>), dim3((unsigned)cdiv(V, 32)),
                         dim3(64 * DW_WAVES), 0, st, g, r, idx, mask, mdt, H, dW, dbias, (int)B,
                         (int)S, (int)D, (int)V);
    else if (!wide16<T, O, DNP, RT>(g, r, idx, mask, mdt, H, dW, dbias, B, S, D, V, st))
      hipLaunchKernelGGL((bwd_dw_kernel<T, O, NP, RT>), dim3((unsigned)cdiv(V, 4)), dim3(256), 0, st,
                         g, r, idx, mask, mdt, H, dW, dbias, (int)B, (int)S, (int)D, (int)V);
  }
}

template <typename T, typename O>
static int launch(const void* grad, const void* r, int rdt, const int32_t* idx, const void* mask,
                  int mdt, const void* H, const void* W, void* dH, void* dW, void* dbias,
                  void* ws, int64_t B, int64_t S, int64_t D, int64_t V, hipStream_t st) {
  const T* g = (const T*)grad;
  const T* h = (const T*)H;
  const T* w = (const T*)W;
#define SPARTON_ROWS(NP)                                                                        \
  (rdt == SPARTON_F32                                                                           \
       ? launch_rows<T, O, NP, float>(g, (const float*)r, idx, mask, mdt, h, w, (O*)dH, (O*)dW, \
                                      (O*)dbias, ws, B, S, D, V, st)                            \
       : launch_rows<T, O, NP, T>(g, (const T*)r, idx, mask, mdt, h, w, (O*)dH, (O*)dW,         \
                                  (O*)dbias, ws, B, S, D, V, st))
  switch (passes_for(D)) {
    case 1: SPARTON_ROWS(1); break;
    case 2: SPARTON_ROWS(2); break;
    case 3: SPARTON_ROWS(3); break;
    case 4: SPARTON_ROWS(4); break;
    case 5: case 6: SPARTON_ROWS(6); break;
    case 7: case 8: SPARTON_ROWS(8); break;
    case 9: case 10: case 11: case 12: SPARTON_ROWS(12); break;
    default: SPARTON_ROWS(16); break;
  }
#undef SPARTON_ROWS
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SPARTON_OK : (int)e;
}

}  // namespace bwd
}  // namespace sparton

using namespace sparton;

extern "C" __attribute__((visibility("default"))) size_t sparton_bwd_workspace_bytes(
    int64_t B, int64_t S, int64_t D, int64_t V) {
  if (B <= 0 || S <= 0 || D <= 0 || V < 0) return 0;
  const bwd::FewPlan few = bwd::few_plan(B, S, D, V);
  const bwd::Pass p = bwd::pass_of(B, S, D);
  return std::max(bwd::layout(p.b, p.s, V).total, few.fits ? few.part_bytes : (size_t)0);
}

extern "C" __attribute__((visibility("default"))) int sparton_bwd(
    const void* grad_reps, const void* reps, int reps_dtype, const int32_t* argmax,
    const void* mask, int mask_dtype, const void* hidden, const void* weight, void* d_hidden,
    void* d_weight, void* d_bias, int grad_dtype, void* workspace, size_t workspace_bytes,
    int64_t B, int64_t S, int64_t D, int64_t V, int dtype, void* stream) {
  if (B < 0 || S < 0 || D < 0 || V < 0) return SPARTON_EINVAL;
  if (dtype < SPARTON_F32 || dtype > SPARTON_F16) return SPARTON_EINVAL;
  if (reps_dtype != SPARTON_F32 && reps_dtype != dtype) return SPARTON_EINVAL;
  if (grad_dtype != SPARTON_F32 && grad_dtype != dtype) return SPARTON_EINVAL;
  if (mask_dtype < SPARTON_MASK_I64 || mask_dtype > SPARTON_MASK_F16) return SPARTON_EINVAL;
  if (B * V > 0 && (grad_reps == nullptr || reps == nullptr || argmax == nullptr || mask == nullptr))
    return SPARTON_EINVAL;
  const bool need_dh = d_hidden != nullptr && B * S > 0 && D > 0;
  const bool need_dw = (d_weight != nullptr || d_bias != nullptr) && V > 0;
  if (need_dh && weight == nullptr) return SPARTON_EINVAL;
  if (need_dw && d_weight != nullptr && D > 0 && B * S > 0 && hidden == nullptr) return SPARTON_EINVAL;
  const int64_t esz = dtype == SPARTON_F32 ? 4 : 2;
  if ((D * esz) % 16 != 0) return SPARTON_EINVAL;
  if (((uintptr_t)hidden | (uintptr_t)weight) % 16 != 0) return SPARTON_EALIGN;
  // Outputs are written 4 elements at a time: 16 bytes (fp32) or 8 bytes (16-bit).
  const uintptr_t oalign = grad_dtype == SPARTON_F32 ? 16 : 8;
  if (((uintptr_t)d_hidden | (uintptr_t)d_weight) % oalign != 0) return SPARTON_EALIGN;
  if (D > INT32_MAX || V > INT32_MAX || B * S > INT32_MAX || B * V > INT32_MAX)
    return SPARTON_EUNSUPPORTED;
  if (need_dh) {
    if (workspace == nullptr) return SPARTON_EWORKSPACE;
    if (workspace_bytes < sparton_bwd_workspace_bytes(B, S, D, V)) return SPARTON_EWORKSPACE;
    if ((uintptr_t)workspace % 256 != 0) return SPARTON_EALIGN;
  }
  if (!need_dh && !need_dw) return SPARTON_OK;
  hipStream_t st = (hipStream_t)stream;
  void* dh = need_dh ? d_hidden : nullptr;
  const bool f32out = grad_dtype == SPARTON_F32;
#define SPARTON_BWD(T)                                                                           \
  (f32out ? bwd::launch<T, float>(grad_reps, reps, reps_dtype, argmax, mask, mask_dtype, hidden, \
                                  weight, dh, d_weight, d_bias, workspace, B, S, D, V, st)       \
          : bwd::launch<T, T>(grad_reps, reps, reps_dtype, argmax, mask, mask_dtype, hidden,     \
                              weight, dh, d_weight, d_bias, workspace, B, S, D, V, st))
  switch (dtype) {
    case SPARTON_BF16: return SPARTON_BWD(bf16);
    case SPARTON_F16: return SPARTON_BWD(f16);
    default: return SPARTON_BWD(float);
  }
#undef SPARTON_BWD
}
