// SnapKV observation-window scores for gfx950 (the baseline path of the reference,
// flash_evict/baselines.py:15-25, `snap_scores`):
//
//   W = min(window, N); the last W query positions of every query head observe all keys
//   logits = (q[:, :, -W:] @ repeat_interleave(k, G)^T) in the input dtype     (:21)
//   logits = float(logits) * D^-0.5, causal mask key > query position -> -inf   (:22-25)
//   p = softmax(logits) in FP32; scores[b, j, n] = mean over the G heads of group j of
//   sum over the W window rows of p                                               (:26-27)
//
// The dot products accumulate in FP32 on MFMA and are rounded to the input dtype before
// the FP32 softmax, as the native-dtype matmul of the reference does. Two kernels:
//   snap_stats_kernel    per key block: partial row max and sum of exponentials of every
//                        window row of the group (lanes hold rows)
//   snap_scores_kernel   per key block: merges the partials into each row's max and 1/sum,
//                        then p summed over the rows in-lane (lanes hold keys), / G, one
//                        store per key
// Both take the same key blocks in the same order, so the second read of a block's K finds it
// in the L2 of the XCD that read it first. Many partials (long prompts of few KV heads, wide windows)
// are merged once, in snap_combine_kernel between the two, instead of in every block.
// No atomics: every score is written once, in a fixed summation order.
//
// What bounds it: K is read once from HBM (33.5 MB at N = 32768, 4 KV heads: 7 us) and each
// logit takes two exponentials (2 x 29 M at 28 heads x 32 rows, 10 us of vector work); launches
// and the latency of each step make the rest. Layout: a wave keeps the K fragments of its keys in
// registers and runs over the row tiles, whose Q the block holds in LDS, eight tiles at a time. (One
// row tile per wave against a strip of K, 64-thread blocks, read K once per row tile and left a combine
// kernel of few threads with a serial loop over the strips: 47.9 + 37.1 + 35.3 us at 28/4 heads,
// N = 32768, D = 128, window 32, against 18.6 + 23.8 us here.)
#include <math.h>
#include <string>

#include "fe_attn.h"
#include "fe_internal.h"
#include "../../include/flash_evict.h"

namespace fe {

// Waves of a block: KG key groups x (waves / KG) row parts. Above tile dim 128 the K fragments of
// 64 keys take 128 registers: one wave per SIMD.
constexpr int snap_waves(int DP) { return DP > 128 ? 4 : 8; }
constexpr int kSnapChunk = 8;        // row tiles between two merges of the key groups' partials
constexpr int kSnapLdsRows = 2048;   // rows per group whose statistics a scores block keeps in LDS
// Partials of a group up to which each scores block merges them itself (128 KiB through L2 a
// block: about the 4.6 us of another launch). More go through snap_combine_kernel. Calls with a limit of
// 4096 / 8192 / 16384 / 32768 / 131072 partials, us: Hq8/Hkv2 D64 N65536 window 16 19.1 / 17.2 / 17.3 / 17.3 /
// 17.1, Hq28/Hkv4 D128 N32768 window 64 63.7 / 63.5 / 63.4 / 67.8 / 67.9, Hq32/Hkv8 N65536 window 64 157 / 156 / 157 /
// 182 / 182, Hq14/Hkv2 D64 N30000 window 64 39 / 39 / 39 / 39 / 82; nine more shapes the same to 16384, and 0-18%
// slower at 32768.
constexpr int kSnapMergeMax = 16384;

// Row tiles of partials up to which each key block has its own (16 MiB): every window of at most 128
// rows to 131072 keys, or of 1024 rows to 32768, at 32/8 heads. Rows x key blocks grow with the window
// times the prompt (1.1 GB for 32768 rows and keys), so beyond it a partial covers several key blocks
// and row parts keep the CUs busy: 25 MB and 23.2 ms there (28.5 with 1.1 GB and no key block left out), 18 MB
// and 14.0 ms (13.2 with 538 MB) for 4096 rows and 131072 keys.
constexpr long long kSnapPartTiles = 65536;

struct SnapArgs {
  const u16* q;
  const u16* k;
  float* scores;
  float2* part;          // [BH][S][Rp] (max, sum) partials
  float2* stats;         // [BH][Rp] (max, sum), where snap_combine_kernel runs
  long long qs[4], ks[4];
  int N, D, G, Hkv, BH;
  int W, R, RT, Rp;      // window rows per head, rows per group (G*W), 32-row tiles, 32 * RT
  int NB, KG;            // key blocks per (b, kv head), key groups (of KT 32-key halves) per block
  int S, per;            // partials per (b, kv head), each of `per` consecutive key blocks
  int part_tiles;        // row tiles of a statistics block (all of a group's, or some chunks)
  float scale_log2;      // D^-0.5 * log2 e
};

// Row r of a group: head g = r / W of the group, query position N - W + r % W.
__device__ __forceinline__ void snap_row(const SnapArgs& a, int hkv, int r, int& head, int& qpos) {
  const int g = r / a.W;
  head = hkv * a.G + g;
  qpos = a.N - a.W + (r - g * a.W);
}

// The 16 dot products of an accumulator rounded to the input type, in place.
template <typename E>
__device__ __forceinline__ void round_logits(f32x16& x) {
#pragma unroll
  for (int i = 0; i < 16; i += 2) {
    const u32 p = E::pack2(x[i], x[i + 1]);
    x[i] = E::to_f32((unsigned short)(p & 0xffffu));
    x[i + 1] = E::to_f32((unsigned short)(p >> 16));
  }
}

// Rows in LDS: DP / 8 16-byte chunks per row, chunk ch of row r at position ch ^ snap_swz(r), so
// that the 16 lanes of a read phase (one chunk of 16 rows) hit every bank once. Rows come from
// HBM whole, consecutive lanes on consecutive chunks: read as fragments straight from global
// memory (32-byte pieces of 32 rows per load, 128 KiB in flight per CU for 32 KiB of L1) they took
// 41.8 + 34.0 us at 28/4 heads, N = 32768, window 32.
template <int DP>
__device__ __forceinline__ int snap_swz(int r) {
  return DP == 64 ? (r >> 1) & 7 : r & 15;
}
template <int DP>
__device__ __forceinline__ u32x4 snap_frag(const u32x4* rows, int r, int ch) {
  return rows[r * (DP / 8) + (ch ^ snap_swz<DP>(r))];
}

// Orders a wave's LDS accesses before and after it for lanes that read each other's data. The hardware
// completes them in order, so this emits no wait of its own; it keeps the compiler, which sees one
// thread's addresses only, from moving a lane's loads above its stores or its next stores above them.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// The wave's K fragments of keys kb .. kb+31 through its own 32 rows of LDS (zeros past N).
template <int DP, int VEC>
__device__ __forceinline__ void snap_load_keys(const SnapArgs& a, const u16* kbase, int kb, u32x4* rows, u32x4 (&f)[DP / 16]) {
  constexpr int CPR = DP / 8, NL = 32 * CPR / 64;
  const int lane = threadIdx.x & 63;
  u32x4 v[NL];
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int i = lane + 64 * j, key = kb + i / CPR;
    const bool ok = key < a.N;
    v[j] = ok ? load8(kbase + (long long)key * a.ks[2], a.ks[3], 8 * (i % CPR), a.D, VEC) : (u32x4){0u, 0u, 0u, 0u};
    if (!VEC) __builtin_amdgcn_sched_barrier(0);   // element loads: one chunk's addresses at a time
  }
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int i = lane + 64 * j;
    rows[(i / CPR) * CPR + ((i % CPR) ^ snap_swz<DP>(i / CPR))] = v[j];
  }
  wave_lds_order();
#pragma unroll
  for (int c = 0; c < DP / 16; ++c) f[c] = snap_frag<DP>(rows, lane & 31, 2 * c + (lane >> 5));
  wave_lds_order();   // the next call writes these rows
}

// Row tiles rt0 .. rt0 + kSnapChunk - 1 of the group's query rows into LDS by the whole block
// (zeros past the last row).
template <int DP, int VEC, int NT>
__device__ __forceinline__ void snap_load_rows(const SnapArgs& a, int b, int hkv, int rt0, u32x4* rows) {
  constexpr int CPR = DP / 8, NL = kSnapChunk * 32 * CPR / NT, U = VEC ? (NL < 8 ? NL : 8) : 1;
  static_assert(NL % U == 0, "row chunk");
  for (int j0 = 0; j0 < NL; j0 += U) {
    if (rt0 * 32 + (NT * j0) / CPR >= a.Rp) break;   // past the last tile
    u32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = (int)threadIdx.x + NT * (j0 + u), r = rt0 * 32 + i / CPR;
      int head = 0, qpos = 0;
      if (r < a.R) snap_row(a, hkv, r, head, qpos);
      v[u] = r < a.R ? load8(a.q + b * a.qs[0] + head * a.qs[1] + (long long)qpos * a.qs[2], a.qs[3], 8 * (i % CPR), a.D, VEC)
                     : (u32x4){0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = (int)threadIdx.x + NT * (j0 + u);
      rows[(i / CPR) * CPR + ((i % CPR) ^ snap_swz<DP>(i / CPR))] = v[u];
    }
  }
}

// Position of the group's row r (-1: padding of the last tile).
__device__ __forceinline__ int snap_qpos(const SnapArgs& a, int r) {
  return r < a.R ? a.N - a.W + r % a.W : -1;
}

// Largest position among the group's rows r0 .. r1 (r1 below R).
__device__ __forceinline__ int snap_last(const SnapArgs& a, int r0, int r1) {
  return r0 / a.W == r1 / a.W ? a.N - a.W + r1 % a.W : a.N - 1;
}

// exp(scale * x) for x <= 0, a difference of two rounded logits (exact in FP32 unless one is
// 2^13 times the other): one product by scale * log2 e and v_exp_f32. Against 64 bits the scores
// are as close as with expf(scale * logit - scale * max): 7.3e-7 to 3.6e-6 relative over ten shapes
// of 2144 to 54886 keys, the two within 0.5% of each other on each (most of it is logits that FP32
// sums round the other way).
__device__ __forceinline__ float snap_exponent(const SnapArgs& a, float x) { return x * a.scale_log2; }
__device__ __forceinline__ float snap_exp(const SnapArgs& a, float x) { return fast_exp2(snap_exponent(a, x)); }

// exp2 down to the smallest subnormal: v_exp_f32 returns 0 below 2^-126. Sums of exponentials, which
// hold a term of 1, need nothing below that; the probabilities do, as keys are ranked by them.
__device__ __forceinline__ float exp2_subnormal(float y) {
  const bool sub = y < -126.f;
  return fast_exp2(sub ? y + 64.f : y) * (sub ? 0x1p-64f : 1.f);
}

// What a partial's exponentials are taken against: its maximum, or 0 where no logit is above -inf. Then
// the sum is 0 over -inf logits (a partial without a visible key), and NaN, which reaches the row's
// sum through every merge, where the maximum passed over NaN logits only.
__device__ __forceinline__ float snap_ref(float m) { return m == -__builtin_huge_valf() ? 0.f : m; }

// Merge of two softmax partials.
__device__ __forceinline__ void snap_merge(const SnapArgs& a, float& m, float& l, float m2, float l2) {
  const float mn = fmaxf(m, m2), ref = snap_ref(mn);
  l = l * snap_exp(a, m - ref) + l2 * snap_exp(a, m2 - ref);
  m = mn;
}

template <typename E, int DP, int VEC, int KT>
__global__ __launch_bounds__(64 * snap_waves(DP)) void snap_stats_kernel(const SnapArgs a) {
  constexpr int NDC = DP / 16, NW = snap_waves(DP);
  constexpr float NEG_INF = -__builtin_huge_valf();
  __shared__ u32x4 rows[kSnapChunk * 32 * (DP / 8)];   // K on the way to registers, then Q
  __shared__ float2 sm[NW][kSnapChunk * 32];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wv % a.KG, rp = wv / a.KG, RP = NW / a.KG;
  const int bh = (int)(blockIdx.x % (unsigned)a.BH), idx = (int)(blockIdx.x / (unsigned)a.BH);
  const int part = idx % a.S, rt_lo = idx / a.S * a.part_tiles, rt_hi = min(a.RT, rt_lo + a.part_tiles);
  const int b = bh / a.Hkv, hkv = bh - b * a.Hkv;
  const u16* kbase = a.k + b * a.ks[0] + hkv * a.ks[1];

  // key blocks up to the last of the part's rows (one at least, which writes the partial)
  int blk_hi = min(a.NB, (part + 1) * a.per);
  if (a.per > 1) blk_hi = max(part * a.per + 1, min(blk_hi, snap_last(a, rt_lo * 32, min(rt_hi * 32, a.R) - 1) / (a.KG * 32 * KT) + 1));
  for (int blk = part * a.per; blk < blk_hi; ++blk) {
    const int kb = (blk * a.KG + kg) * 32 * KT;
    u32x4 kf[KT][NDC];                            // K fragments (A operand) of the wave's keys
#pragma unroll
    for (int s = 0; s < KT; ++s)
      snap_load_keys<DP, VEC>(a, kbase, kb + 32 * s, rows + wv * 32 * (DP / 8), kf[s]);
    __syncthreads();
    const bool masked = kb + 32 * KT > a.N - a.W;   // some key of the wave is past some row
    for (int rt0 = rt_lo; rt0 < rt_hi; rt0 += kSnapChunk) {
      snap_load_rows<DP, VEC, 64 * NW>(a, b, hkv, rt0, rows);
      __syncthreads();
      for (int rt = rt0 + rp; rt < min(rt0 + kSnapChunk, rt_hi); rt += RP) {
        f32x16 x[KT];
#pragma unroll
        for (int c = 0; c < NDC; ++c) {
          const u32x4 qf = snap_frag<DP>(rows, (rt - rt0) * 32 + l32, 2 * c + hh);
#pragma unroll
          for (int s = 0; s < KT; ++s)
            x[s] = c == 0 ? E::mfma(kf[s][0], qf, (f32x16){}) : E::mfma(kf[s][c], qf, x[s]);
        }
        // lanes hold query row rt*32 + l32; register i of half s holds key kb + 32s + 8(i/4) + 4h + i%4
        float m = NEG_INF, l = 0.f;
#pragma unroll
        for (int s = 0; s < KT; ++s) {
          round_logits<E>(x[s]);
          if (masked) {
            const int rel = snap_qpos(a, rt * 32 + l32) - kb - 32 * s - 4 * hh;
#pragma unroll
            for (int i = 0; i < 16; ++i) x[s][i] = 8 * (i >> 2) + (i & 3) <= rel ? x[s][i] : NEG_INF;
          }
#pragma unroll
          for (int i = 0; i < 16; ++i) m = fmaxf(m, x[s][i]);
        }
        m = half_swap_max(m);
        const float ref = snap_ref(m);
#pragma unroll
        for (int s = 0; s < KT; ++s) {
#pragma unroll
          for (int i = 0; i < 16; ++i) l += snap_exp(a, x[s][i] - ref);
        }
        l = half_swap_sum(l);
        if (hh == 0) sm[kg][(rt - rt0) * 32 + l32] = make_float2(m, l);
      }
      __syncthreads();
      const int nrows = min(kSnapChunk, rt_hi - rt0) * 32;
      for (int r = tid; r < nrows; r += 64 * NW) {
        float m = sm[0][r].x, l = sm[0][r].y;
        for (int g = 1; g < a.KG; ++g) snap_merge(a, m, l, sm[g][r].x, sm[g][r].y);
        float2* out = a.part + ((long long)bh * a.S + part) * a.Rp + rt0 * 32 + r;
        if (blk > part * a.per) snap_merge(a, m, l, out->x, out->y);   // this thread's own of the block before
        *out = make_float2(m, l);
      }
      __syncthreads();
    }
  }
}

// (max, sum) of row r of a group from partials s0, s0 + step, ... of its key blocks; four loads
// in flight.
__device__ __forceinline__ void snap_merge_parts(const SnapArgs& a, int bh, int r, int s0, int step, float& m, float& l) {
  const float2* p = a.part + (long long)bh * a.S * a.Rp + r;
  m = -__builtin_huge_valf();
  l = 0.f;
  for (int s = s0; s < a.S; s += 4 * step) {
    float2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = s + u * step < a.S ? p[(long long)(s + u * step) * a.Rp] : make_float2(-__builtin_huge_valf(), 0.f);
    float mn = m;
#pragma unroll
    for (int u = 0; u < 4; ++u) mn = fmaxf(mn, v[u].x);
    const float ref = snap_ref(mn);
    l *= snap_exp(a, m - ref);
#pragma unroll
    for (int u = 0; u < 4; ++u) l += v[u].y * snap_exp(a, v[u].x - ref);
    m = mn;
  }
}

// 32 rows per block, each by 32 threads that take every 32nd partial (B1 Hq7/Hkv1, N = 40831, window
// 128: 319 partials of 896 rows).
__global__ __launch_bounds__(1024) void snap_combine_kernel(const SnapArgs a) {
  __shared__ float2 sm[32][33];
  const int r32 = threadIdx.x & 31, part = threadIdx.x >> 5;
  const int tiles = a.Rp / 32;
  const int bh = (int)(blockIdx.x / (unsigned)tiles), r = (int)(blockIdx.x % (unsigned)tiles) * 32 + r32;
  float m, l;
  snap_merge_parts(a, bh, r, part, 32, m, l);
  sm[part][r32] = make_float2(m, l);
  __syncthreads();
  if (part == 0) {
    for (int p = 1; p < 32; ++p) snap_merge(a, m, l, sm[p][r32].x, sm[p][r32].y);
    a.stats[(long long)bh * a.Rp + r] = make_float2(m, l);
  }
}

template <typename E, int DP, int VEC, int KT>
__global__ __launch_bounds__(64 * snap_waves(DP)) void snap_scores_kernel(const SnapArgs a) {
  constexpr int NDC = DP / 16, NW = snap_waves(DP), NT = 64 * NW;
  __shared__ u32x4 qrows[kSnapChunk * 32 * (DP / 8)];  // K on the way to registers, then Q
  __shared__ __attribute__((aligned(16))) float st_m[kSnapLdsRows], st_il[kSnapLdsRows];
  __shared__ float2 sm[NT];
  __shared__ float red[NW][64];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wv % a.KG, rp = wv / a.KG, RP = NW / a.KG;
  const int bh = (int)(blockIdx.x % (unsigned)a.BH), blk = (int)(blockIdx.x / (unsigned)a.BH);
  const int b = bh / a.Hkv, hkv = bh - b * a.Hkv;
  const int kb = (blk * a.KG + kg) * 32 * KT;
  const u16* kbase = a.k + b * a.ks[0] + hkv * a.ks[1];

  u32x4 kf[KT][NDC];                              // K fragments (B operand) of the wave's keys
#pragma unroll
  for (int s = 0; s < KT; ++s)
    snap_load_keys<DP, VEC>(a, kbase, kb + 32 * s, qrows + wv * 32 * (DP / 8), kf[s]);
  const bool masked = kb + 32 * KT > a.N - a.W;
  // max and 1/sum of row r; rows whose every logit is -inf contribute nothing
  auto put = [&](int r, float m, float l) {
    const bool live = r < a.R && l != 0.f;
    st_m[r % kSnapLdsRows] = live ? m : 0.f;
    st_il[r % kSnapLdsRows] = live ? 1.f / l : 0.f;
  };
  // score of the wave's key 32hh + l32 (row part 0 only), times G
  const int key = kb + 32 * hh + l32;
  const bool store = rp == 0 && hh < KT && key < a.N;
  auto score = [&](auto exp2_fn) __attribute__((always_inline)) {
    float acc[KT] = {};
    for (int r0 = 0; r0 < a.Rp; r0 += kSnapLdsRows) {
      // statistics of rows r0 .. r0 + rows - 1 into LDS
      const int rows = min(kSnapLdsRows, a.Rp - r0);
      if (a.stats) {
        if (snap_last(a, r0, min(r0 + rows, a.R) - 1) < blk * a.KG * 32 * KT) continue;   // keys past all of them
        if (r0 > 0) __syncthreads();
        for (int r = tid; r < rows; r += NT) {
          const float2 v = a.stats[(long long)bh * a.Rp + r0 + r];
          put(r0 + r, v.x, v.y);
        }
      } else {
        // Rp <= kSnapLdsRows: few rows share the block's threads, each taking every P-th partial
        int P = 1;
        while (P < 8 && 2 * P * rows <= NT) P *= 2;
        for (int i = tid; i < P * rows; i += NT) {
          const int r = i % rows, part = i / rows;
          float m, l;
          snap_merge_parts(a, bh, r, part, P, m, l);
          if (P > 1)
            sm[i] = make_float2(m, l);
          else
            put(r, m, l);
        }
        if (P > 1) {
          __syncthreads();
          if (tid < rows) {
            float m = sm[tid].x, l = sm[tid].y;
            for (int p = 1; p < P; ++p) snap_merge(a, m, l, sm[p * rows + tid].x, sm[p * rows + tid].y);
            put(tid, m, l);
          }
        }
      }
      for (int rt0 = r0 / 32; rt0 < (r0 + rows) / 32; rt0 += kSnapChunk) {
        __syncthreads();                             // the buffer's last readers are done
        snap_load_rows<DP, VEC, NT>(a, b, hkv, rt0, qrows);
        __syncthreads();
        for (int rt = rt0 + rp; rt < min(rt0 + kSnapChunk, a.RT); rt += RP) {
          f32x16 x[KT];
#pragma unroll
          for (int c = 0; c < NDC; ++c) {
            const u32x4 qf = snap_frag<DP>(qrows, (rt - rt0) * 32 + l32, 2 * c + hh);
#pragma unroll
            for (int s = 0; s < KT; ++s)
              x[s] = c == 0 ? E::mfma(qf, kf[s][0], (f32x16){}) : E::mfma(qf, kf[s][c], x[s]);
          }
          // padding rows are left out by their position: their zero query gives NaN against a key with an
          // infinite channel, which 1/sum = 0 would not take out of the key's score
          const bool sel = masked || (rt + 1) * 32 > a.R;
          const int qpos = sel ? snap_qpos(a, rt * 32 + l32) : 0;
#pragma unroll
          for (int s = 0; s < KT; ++s) round_logits<E>(x[s]);
          // lanes hold key kb + 32s + l32; register i holds row 8(i/4) + 4h + i%4 of the tile
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int rj = rt * 32 - r0 + 8 * j + 4 * hh;
            const float4 m4 = *(const float4*)(st_m + rj), il4 = *(const float4*)(st_il + rj);
            const float mr[4] = {m4.x, m4.y, m4.z, m4.w}, ilr[4] = {il4.x, il4.y, il4.z, il4.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int qp = sel ? __shfl(qpos, 8 * j + 4 * hh + e) : 0;
#pragma unroll
              for (int s = 0; s < KT; ++s) {
                const float p = exp2_fn(snap_exponent(a, x[s][4 * j + e] - mr[e])) * ilr[e];
                acc[s] += !sel || kb + 32 * s + l32 <= qp ? p : 0.f;
              }
            }
          }
        }
      }
    }
    // lanes h = 0 and 1 hold the two halves of the rows of each key, the row parts' waves the
    // other row tiles; lane l of half s holds key kb + 32s + l32
    const float t0 = half_swap_sum(acc[0]), t1 = half_swap_sum(acc[KT - 1]);
    red[wv][lane] = hh == 0 ? t0 : t1;
    __syncthreads();
    float t = 0.f;
    if (store) {
      t = red[kg][lane];
      for (int p = 1; p < RP; ++p) t += red[p * a.KG + kg][lane];
    }
    return t;
  };
  float t = score([](float y) { return fast_exp2(y); });
  // v_exp_f32 returns 0 below 2^-126. The R terms of a sum of at least R * 2^-102 miss less than 2^-24
  // of it by that; where a key's sum is smaller, the block runs once more with exp2_subnormal. Against
  // the fast exponential alone 39.2 -> 40.0 us a call at 28/4 heads, N = 32768, D = 128, window 32,
  // and 0.5-1.2% at window 128; choosing the exponential in every row tile took 3-5%.
  if (__syncthreads_or(store && t < (float)a.R * 0x1p-102f)) t = score([](float y) { return exp2_subnormal(y); });
  if (store) a.scores[(long long)bh * a.N + key] = t / (float)a.G;
}

struct SnapKernel {
  const void* fn;
  const char* name;
};

// Index ((dtype * 3 + tile dim 64, 128, 256) * 2 + VEC) * 4 + 2 * (KT - 1) (+1 for the scores
// kernel); VEC = 1: 16-byte row loads (channel stride 1, 16-byte aligned rows), 0: element loads.
#define FE_SNAP_KT(E, DP, V, KT, TAG)                                                                       \
  {(const void*)snap_stats_kernel<E, DP, V, KT>, "snap_stats_kernel<" TAG "," #DP "," #V "," #KT ">"},       \
      {(const void*)snap_scores_kernel<E, DP, V, KT>, "snap_scores_kernel<" TAG "," #DP "," #V "," #KT ">"}
#define FE_SNAP_VEC(E, DP, V, TAG) FE_SNAP_KT(E, DP, V, 1, TAG), FE_SNAP_KT(E, DP, V, 2, TAG)
#define FE_SNAP_DIM(E, DP, TAG) FE_SNAP_VEC(E, DP, 0, TAG), FE_SNAP_VEC(E, DP, 1, TAG)
#define FE_SNAP_TYPE(E, TAG) FE_SNAP_DIM(E, 64, TAG), FE_SNAP_DIM(E, 128, TAG), FE_SNAP_DIM(E, 256, TAG)

const SnapKernel kSnapKernels[] = {
    FE_SNAP_TYPE(F16, "f16"),
    FE_SNAP_TYPE(BF16, "bf16"),
    {(const void*)snap_combine_kernel, "snap_combine_kernel"},
};
#undef FE_SNAP_TYPE
#undef FE_SNAP_DIM
#undef FE_SNAP_VEC
#undef FE_SNAP_KT

void append_snap_resources(std::string& out) {
  for (const auto& e : kSnapKernels) {
    hipFuncAttributes attr;
    if (hipFuncGetAttributes(&attr, e.fn) != hipSuccess) continue;
    char buf[512];
    snprintf(buf, sizeof(buf),
             "{\"kernel\":\"%s\",\"registers_per_thread\":%d,\"lds_static_bytes\":%zu,"
             "\"lds_dynamic_bytes\":0,\"scratch_bytes_per_thread\":%zu,\"max_threads_per_block\":%d},",
             e.name, attr.numRegs, (size_t)attr.sharedSizeBytes, (size_t)attr.localSizeBytes,
             attr.maxThreadsPerBlock);
    out += buf;
  }
}

// Key blocks: KG groups of KT 32-key halves each. The largest block (512 keys, each K fragment in
// registers serving every row tile) that still gives every CU one; short prompts take fewer keys
// per block and give the waves different row tiles instead. Blocks per (b, kv head): the result.
int snap_split(long long BH, long long N, int waves, int& KG, int& KT) {
  KG = waves;
  KT = 2;
  auto blocks = [&]() { return (N + 32 * KG * KT - 1) / (32 * KG * KT); };
  while (KG > 1 && BH * blocks() < 256) KG /= 2;
  if (KG == 1 && BH * blocks() < 256) KT = 1;
  return (int)blocks();
}

// Partials per (b, kv head): one per key block, fewer where they would exceed kSnapPartTiles row tiles.
int snap_parts(long long BH, long long NB, long long RT) {
  const long long tiles = BH * RT;
  if (tiles < 1 || tiles > kSnapPartTiles) return 1;   // below 1: sizes past 64 bits, refused by the call
  return (int)(NB < kSnapPartTiles / tiles ? NB : kSnapPartTiles / tiles);
}

bool snap_vec(const void* p, const int64_t* st, int64_t D) {
  return st[3] == 1 && D % 8 == 0 && ((uintptr_t)p % 16) == 0 && st[0] % 8 == 0 && st[1] % 8 == 0 &&
         st[2] % 8 == 0;
}

}  // namespace fe

using namespace fe;

extern "C" size_t fe_snap_scores_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t window) {
  if (B < 1 || Hq < 1 || Hkv < 1 || N < 1 || window < 1 || Hq % Hkv != 0) return 0;
  const long long W = window < N ? window : N;
  const long long BH = B * Hkv, R = (Hq / Hkv) * W, RT = (R + 31) / 32;
  int KG, KT;
  const int S = snap_parts(BH, snap_split(BH, N, snap_waves(256), KG, KT), RT);   // the most of any head dim
  return (size_t)(BH * RT * 32) * sizeof(float2) * (size_t)(S + 1);
}

extern "C" int fe_snap_scores(const void* q, const void* k, float* scores, int64_t B, int64_t Hq, int64_t Hkv,
                              int64_t N, int64_t D, const int64_t* q_strides, const int64_t* k_strides, int dtype,
                              int64_t window, void* workspace, size_t workspace_bytes, void* hip_stream) {
  clear_error();
  if (!q || !k || !scores || !q_strides || !k_strides) {
    set_error("fe_snap_scores: null pointer argument");
    return FE_ERR_INVALID;
  }
  if (B < 1 || Hq < 1 || Hkv < 1 || N < 1 || D < 1 || Hq % Hkv != 0 || window < 1) {
    set_error("fe_snap_scores: expected nonempty shapes, Hq divisible by Hkv and window >= 1");
    return FE_ERR_INVALID;
  }
  if (D > 256) {
    set_error("fe_snap_scores: head dimension must be <= 256");
    return FE_ERR_INVALID;
  }
  if (dtype != FE_DTYPE_F16 && dtype != FE_DTYPE_BF16) {
    set_error("fe_snap_scores: dtype must be FE_DTYPE_F16 or FE_DTYPE_BF16");
    return FE_ERR_INVALID;
  }
  for (int i = 0; i < 4; ++i)
    if (q_strides[i] < 0 || k_strides[i] < 0) {
      set_error("fe_snap_scores: negative strides are not supported");
      return FE_ERR_INVALID;
    }
  const long long W = window < N ? window : N;
  const long long G = Hq / Hkv, BH = B * Hkv, R = G * W, RT = (R + 31) / 32;
  // each grid within 31 bits: at most one block per 64 keys or per row tile (32 keys only below 256 blocks)
  if (N > (1LL << 30) || R > (1LL << 30) || BH * RT > 0x7fffffffLL || BH * ((N + 63) / 64) > 0x7fffffffLL) {
    set_error("fe_snap_scores: problem too large");
    return FE_ERR_UNSUPPORTED;
  }
  int KG, KT;
  const int waves = snap_waves(D <= 128 ? 128 : 256), NB = snap_split(BH, N, waves, KG, KT);
  const int most = snap_parts(BH, NB, RT), per = (NB + most - 1) / most, S = (NB + per - 1) / per;
  // statistics blocks: one per partial, or, where a partial covers several key blocks, row parts (of whole
  // chunks) to make 1024 blocks. Fewer read K less often and end later: with 512 a window of 1024 rows
  // takes 1% less, one of 32768 rows 16% more.
  const long long chunks = (RT + kSnapChunk - 1) / kSnapChunk;
  long long RS = 1;
  if (per > 1) RS = (1024 + BH * S - 1) / (BH * S);
  const long long part_chunks = (chunks + (RS < chunks ? RS : chunks) - 1) / (RS < chunks ? RS : chunks);
  RS = (chunks + part_chunks - 1) / part_chunks;
  const size_t need = fe_snap_scores_workspace_bytes(B, Hq, Hkv, N, window);
  if (!workspace || workspace_bytes < need) {
    set_error("fe_snap_scores: needs a workspace of fe_snap_scores_workspace_bytes() bytes");
    return FE_ERR_WORKSPACE;
  }
  SnapArgs a;
  a.q = (const u16*)q;
  a.k = (const u16*)k;
  a.scores = scores;
  a.part = (float2*)workspace;
  a.stats = RT * 32 > kSnapLdsRows || RT * 32 * S > kSnapMergeMax ? a.part + BH * RT * 32 * S : nullptr;
  for (int i = 0; i < 4; ++i) {
    a.qs[i] = q_strides[i];
    a.ks[i] = k_strides[i];
  }
  a.N = (int)N;
  a.D = (int)D;
  a.G = (int)G;
  a.Hkv = (int)Hkv;
  a.BH = (int)BH;
  a.W = (int)W;
  a.R = (int)R;
  a.RT = (int)RT;
  a.Rp = (int)(RT * 32);
  a.NB = NB;
  a.KG = KG;
  a.S = S;
  a.per = per;
  a.part_tiles = (int)(part_chunks * kSnapChunk);
  a.scale_log2 = (float)(1.4426950408889634 * pow((double)D, -0.5));
  const int vec = snap_vec(q, q_strides, D) && snap_vec(k, k_strides, D) ? 1 : 0;
  const int bf = dtype == FE_DTYPE_BF16 ? 1 : 0;
  const int ki = ((bf * 3 + (D <= 64 ? 0 : (D <= 128 ? 1 : 2))) * 2 + vec) * 4 + 2 * (KT - 1);
  const void* stats_fn = kSnapKernels[ki].fn;
  const void* scores_fn = kSnapKernels[ki + 1].fn;
  hipStream_t stream = (hipStream_t)hip_stream;
  void* kargs[] = {&a};
  const dim3 block(64 * waves);
  hipError_t err = hipLaunchKernel(stats_fn, dim3((unsigned)(BH * S * RS)), block, kargs, 0, stream);
  if (err == hipSuccess && a.stats) {
    const long long rows = BH * RT * 32;
    err = hipLaunchKernel((const void*)snap_combine_kernel, dim3((unsigned)(rows / 32)), dim3(1024), kargs, 0, stream);
  }
  if (err == hipSuccess) err = hipLaunchKernel(scores_fn, dim3((unsigned)(BH * NB)), block, kargs, 0, stream);
  if (err != hipSuccess) {
    set_error(std::string("fe_snap_scores: launch: ") + hipGetErrorString(err));
    return FE_ERR_HIP;
  }
  return FE_OK;
}
