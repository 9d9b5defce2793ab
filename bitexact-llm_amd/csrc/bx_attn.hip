// Exact integer attention for gfx950: paged limb-plane KV store, paged decode attention, and fused prefill
// attention over a contiguous integer cache.
//
// What is computed (src/bitexact/exact/ops.py:133-143, src/bitexact/vllm_plugin/tri_exact_attn.py:1-15):
//   raw[i, s] = sum_d q[i, d] K[s, d]                 exact int64 (|q|, |K| within 3 signed base-256 limbs)
//   mx[i]     = max over visible keys s <= qpos[i] of raw[i, s]
//   zf        = min(rshc(mx - raw, FK + 3 - sh[i] - FZ), 48 << FZ); t = rshc(zf l2e, 28)
//   p         = exp2neg_lut(t, lut, FP)   (2^-f table at 2^60 + linear interpolation; 0 for hidden keys)
//   den[i]    = sum_s p,   num[i, d] = sum_s p V[s, d]                  exact int64
// Two sweeps over the keys are required (the quantized exp table does not allow online rescaling,
// src/bitexact/vllm_plugin/tri_paged.py:16-19). Maxima and sums are exact in any order, so the key split and
// the tiling never change a bit.
//
// Kernel shape: one block of 256 threads per (query tile, key range). 64-key tiles are staged in LDS as
// int32 K / V rows (paged caches hold int8 limb planes that are joined on the way in). Thread t = (wave w,
// lane l) owns key l of the tile for the scores of queries w, w + 4, ... and output dims l, l + 64 of the
// same queries for p V, so query-indexed LDS reads are wave-uniform broadcasts and key/dim-indexed reads
// hit distinct banks (rows padded by one word).
#include "bx_common.h"
#include "bx_rope.h"
#include "bx_introws.h"

#include <algorithm>
#include <type_traits>

namespace bx {

BX_PHASE_TABLE

constexpr int kFK = 17, kFZ = 26, kFP = 22, kFT2 = 26, kExp2Bits = 14, kExp2One = 60;

// A weight is exactly 0 once n >= FP + 2: the interpolated table value v lies in [0, 2^60] (the table falls
// from 2^60), and rshc(v, 60 - FP + n) with a shift of at least 62 rounds it to 0 whatever entry was read. Such
// scores (most of them: softmax weights are mostly negligible) read entry 0, so their loads share one cache
// line instead of scattering over the 128 KiB table.
constexpr int64_t kZeroN = kFP + 2;

// attn_weight in two halves, so that a caller can issue the table loads of many scores before using any:
// WeightAt holds the table position of one score (always inside the table: 0 <= idx < 2^14, whatever z is,
// so loads for hidden keys are safe and their weight is discarded).
struct WeightAt {
  int64_t n, rr;
  int idx;
};

__device__ __forceinline__ WeightAt weight_at(int64_t z, int64_t zshift, int64_t l2e) {
  int64_t zf = rshc(z, zshift);
  zf = imin(zf, 48LL << kFZ);
  const int64_t t = rshc(mul_wrap(zf, l2e), kFZ + 28 - kFT2);
  const int64_t f = t & ((1LL << kFT2) - 1);
  WeightAt w;
  w.n = t >> kFT2;
  w.idx = w.n < kZeroN ? (int)(f >> (kFT2 - kExp2Bits)) : 0;
  w.rr = f & ((1LL << (kFT2 - kExp2Bits)) - 1);
  return w;
}

__device__ __forceinline__ int64_t weight_of(const WeightAt& w, int64_t a, int64_t b) {
  const int64_t v = add_wrap(a, rshc(mul_wrap(b - a, w.rr), kFT2 - kExp2Bits));
  return rshc(v, kExp2One - kFP + w.n);
}

// softmax_w's weight of one visible key (src/bitexact/exact/ops.py:133-143 over exp2neg_lut, 108-116).
__device__ __forceinline__ int64_t attn_weight(int64_t z, int64_t zshift, const int64_t* lut, int64_t l2e) {
  int64_t zf = rshc(z, zshift);
  zf = imin(zf, 48LL << kFZ);
  const int64_t t = rshc(mul_wrap(zf, l2e), kFZ + 28 - kFT2);
  const int64_t n = t >> kFT2;
  const int64_t f = t & ((1LL << kFT2) - 1);
  const int64_t idx = n < kZeroN ? f >> (kFT2 - kExp2Bits) : 0;
  const int64_t rr = f & ((1LL << (kFT2 - kExp2Bits)) - 1);
  const int64_t a = lut[idx];
  const int64_t v = add_wrap(a, rshc(mul_wrap(lut[idx + 1] - a, rr), kFT2 - kExp2Bits));
  return rshc(v, kExp2One - kFP + n);
}

// int8-mode weight of a visible key (int8.segs.softmax, src/bitexact/int8/segs.py:90-99; tri_paged._zscale,
// src/bitexact/vllm_plugin/tri_paged.py:93-99): d = raw - mx <= 0 at 2 FQ bits, z = rsh(d, zsh) (head_dim 64)
// or rsh(max(d, -2^38) zmul, zsh) (head_dim 128, zmul = round(2^24 / sqrt 2)); the weight is the table entry
// rsh(e^z 2^FE, FE - FP) of z at step 2^-FA over [EXP_MIN, 0], 0 below it.
constexpr int64_t kI8ZClamp = -(1LL << 38);
constexpr int64_t kI8ZLo = -32LL * 4096;         // EXP_MIN << FA: table index 0
// The table index of int8_weight (negative: weight 0).
__device__ __forceinline__ int64_t int8_index(int64_t d, int zsh, int64_t zmul) {
  const int64_t z = zmul == 0 ? rsh64(d, zsh) : rsh64(mul_wrap(imax(d, kI8ZClamp), zmul), zsh);
  return imax(z, kI8ZLo - 1) - kI8ZLo;
}

__device__ __forceinline__ int64_t int8_weight(int64_t d, int zsh, int64_t zmul, const int32_t* ptab) {
  const int64_t idx = int8_index(d, zsh, zmul);
  return idx >= 0 ? (int64_t)ptab[idx] : 0;
}

// int32 value -> the value of its first three signed base-256 digits (what a 3-limb split keeps).
__device__ __forceinline__ int32_t keep3(int32_t x) {
  const int32_t a0 = limb_lo(x);
  int32_t r = (x - a0) >> 8;
  const int32_t a1 = limb_lo(r);
  r = (r - a1) >> 8;
  const int32_t a2 = limb_lo(r);
  return a0 + a1 * 256 + a2 * 65536;
}

struct AttnArgs {
  // queries
  const int32_t* q;
  int64_t sq_tile, sq_row;        // element strides: between query groups (z or (r,h)) and between queries
  const int64_t* sh;              // per query exponent, index = group * sh_tile + query
  int64_t sh_tile;
  const int64_t* qpos;            // per query position: qpos[(group / qpos_div) * qpos_tile + query * qpos_row]
  int64_t qpos_tile, qpos_row;
  int qpos_div;
  int nq;                         // queries per group (decode M <= 4, prefill gT)
  // keys: paged limb planes or contiguous int32
  const int8_t* cache;            // [nb, HKV, bs, 8 HD]
  int64_t sc_nb, sc_h, sc_bs;
  const int32_t* bt;
  int64_t sbt;
  const int64_t* rmap;
  int bs, hkv;
  int nblk;                       // paged: block-table entries per row
  const int32_t* K;               // contiguous: [Z, S, HD] with strides
  const int32_t* V;
  int64_t sk_z, sk_s, sv_z, sv_s;
  int S;                          // contiguous: keys available
  // table, scale (exact mode)
  const int64_t* lut;
  int64_t l2e;
  // int8 mode: int64 queries and the weight table (wrule 1)
  const int64_t* q64;
  const int32_t* ptab;
  int wrule, zsh;
  int64_t zmul;
  // outputs
  int64_t* num;
  int64_t* den;
  int64_t snum_tile, snum_row;
  int64_t sden_tile;
  // split-KV state
  int nsplit;
  int64_t* mx_ws;                 // [groups, nq] running maxima stored as mx - NEG (0 = none yet)
  int64_t* num_ws;                // [groups, nq, HD]
  int64_t* den_ws;                // [groups, nq]
  int32_t* sem;                   // [groups]
  int64_t* raw;                   // split launches that keep the scores (null: K read in both)
  int one_keys;                   // there: a tile with at most this many keys is one block's
  const int32_t* list;            // attn_dec_kernel's LIST form: count, then token rows
  uint64_t exch_ticks;            // attn_dec_exch_kernel: longest wait for the other splits' maxima (100 MHz ticks)
};

template <int QT, int HD>
struct AttnSmem {
  int32_t Qs[QT][HD];
  int32_t Ks[64][HD + 1];
  int32_t Vs[64][HD + 1];
  int32_t Ps[QT][65];
  int64_t qpos[QT];
  int64_t shift[QT];              // per query: FK + 3 - FZ - sh
  int64_t mx[QT];
  int s_last;
};

template <int QT, int HD, bool PAGED>
__device__ __forceinline__ void load_kv_tile(const AttnArgs& p, AttnSmem<QT, HD>& sm, int group, int h, int key0, int nkeys,
                                             bool want_v) {
  constexpr int UNITS = 64 * (HD / 16);          // (key, 16-dim chunk) units per tile
  for (int u = threadIdx.x; u < UNITS; u += 256) {
    const int kk = u / (HD / 16), c = u % (HD / 16);
    const int s = key0 + kk;
    int32_t kv[16], vv[16];
    if (kk < nkeys) {
      if (PAGED) {
        const int64_t brow = p.rmap ? p.rmap[group / p.hkv] : group / p.hkv;
        const int blk = p.bt[brow * p.sbt + s / p.bs];
        const int8_t* row = p.cache + (int64_t)blk * p.sc_nb + (int64_t)h * p.sc_h + (int64_t)(s % p.bs) * p.sc_bs;
        const v4i k0 = *(const v4i*)(row + c * 16), k1 = *(const v4i*)(row + HD + c * 16),
                  k2 = *(const v4i*)(row + 2 * HD + c * 16);
        v4i v0 = {0, 0, 0, 0}, v1 = v0, v2 = v0;
        if (want_v) {
          v0 = *(const v4i*)(row + 3 * HD + c * 16);
          v1 = *(const v4i*)(row + 4 * HD + c * 16);
          v2 = *(const v4i*)(row + 5 * HD + c * 16);
        }
        const int8_t* pk0 = (const int8_t*)&k0;
        const int8_t* pk1 = (const int8_t*)&k1;
        const int8_t* pk2 = (const int8_t*)&k2;
        const int8_t* pv0 = (const int8_t*)&v0;
        const int8_t* pv1 = (const int8_t*)&v1;
        const int8_t* pv2 = (const int8_t*)&v2;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          kv[e] = (int32_t)pk0[e] + (int32_t)pk1[e] * 256 + (int32_t)pk2[e] * 65536;
          vv[e] = (int32_t)pv0[e] + (int32_t)pv1[e] * 256 + (int32_t)pv2[e] * 65536;
        }
      } else {
        const int32_t* kr = p.K + (int64_t)group * p.sk_z + (int64_t)s * p.sk_s + c * 16;
        const int32_t* vr = p.V + (int64_t)group * p.sv_z + (int64_t)s * p.sv_s + c * 16;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          kv[e] = keep3(kr[e]);
          vv[e] = want_v ? keep3(vr[e]) : 0;
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) kv[e] = vv[e] = 0;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      sm.Ks[kk][c * 16 + e] = kv[e];
      if (want_v) sm.Vs[kk][c * 16 + e] = vv[e];
    }
  }
}

// raw scores of this thread's queries (w + 4 j) against key lane l of the staged tile
template <int QT, int HD>
__device__ __forceinline__ void tile_scores(const AttnSmem<QT, HD>& sm, int64_t (&raw)[QT / 4]) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < QT / 4; ++j) raw[j] = 0;
#pragma unroll 8
  for (int d = 0; d < HD; ++d) {
    const int64_t kd = sm.Ks[l][d];
#pragma unroll
    for (int j = 0; j < QT / 4; ++j) raw[j] += (int64_t)sm.Qs[w + 4 * j][d] * kd;
  }
}

// Stage queries of the tile (3-limb values), their exponents / positions; returns the visible key count.
template <int QT, int HD>
__device__ __forceinline__ int64_t stage_queries(const AttnArgs& p, AttnSmem<QT, HD>& sm, int group, int q0, int nvalid) {
  for (int u = threadIdx.x; u < QT * HD; u += 256) {
    const int i = u / HD, d = u % HD;
    const int64_t qi = group * p.sq_tile + (int64_t)(q0 + i) * p.sq_row + d;
    sm.Qs[i][d] = i < nvalid ? keep3(p.q64 ? (int32_t)p.q64[qi] : p.q[qi]) : 0;
  }
  if (threadIdx.x < QT) {
    const int i = threadIdx.x;
    const bool ok = i < nvalid;
    sm.qpos[i] = ok ? p.qpos[(group / p.qpos_div) * p.qpos_tile + (int64_t)(q0 + i) * p.qpos_row] : -1;
    sm.shift[i] = ok && p.sh ? (int64_t)(kFK + 3 - kFZ) - p.sh[group * p.sh_tile + q0 + i] : 0;
    sm.mx[i] = kNeg;
  }
  __syncthreads();
  int64_t kend = 0;
  for (int i = 0; i < QT; ++i) kend = imax(kend, sm.qpos[i] + 1);
  return kend;
}

// Sweep 1: per-query maxima over visible keys in [lo, hi) into sm.mx (LDS atomic max).
template <int QT, int HD, bool PAGED>
__device__ void sweep_max(const AttnArgs& p, AttnSmem<QT, HD>& sm, int group, int h, int64_t lo, int64_t hi) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  int64_t best[QT / 4];
#pragma unroll
  for (int j = 0; j < QT / 4; ++j) best[j] = kNeg;
  for (int64_t k0 = lo; k0 < hi; k0 += 64) {
    const int nk = (int)imin(64, hi - k0);
    __syncthreads();
    load_kv_tile<QT, HD, PAGED>(p, sm, group, h, (int)k0, nk, false);
    __syncthreads();
    int64_t raw[QT / 4];
    tile_scores<QT, HD>(sm, raw);
#pragma unroll
    for (int j = 0; j < QT / 4; ++j) {
      const bool vis = l < nk && k0 + l <= sm.qpos[w + 4 * j];
      if (vis) best[j] = imax(best[j], raw[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < QT / 4; ++j) {
    const int64_t m = wave_max64(best[j]);
    if (l == 0) atomicMax((long long*)&sm.mx[w + 4 * j], (long long)m);
  }
  __syncthreads();
}

// Sweep 2: weights from the maxima in sm.mx; accumulates den / num for the thread's queries.
template <int QT, int HD, bool PAGED>
__device__ void sweep_acc(const AttnArgs& p, AttnSmem<QT, HD>& sm, int group, int h, int64_t lo, int64_t hi,
                          int64_t (&den)[QT / 4], int64_t (&num)[QT / 4][HD / 64]) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < QT / 4; ++j) {
    den[j] = 0;
#pragma unroll
    for (int c = 0; c < HD / 64; ++c) num[j][c] = 0;
  }
  for (int64_t k0 = lo; k0 < hi; k0 += 64) {
    const int nk = (int)imin(64, hi - k0);
    __syncthreads();
    load_kv_tile<QT, HD, PAGED>(p, sm, group, h, (int)k0, nk, true);
    __syncthreads();
    int64_t raw[QT / 4];
    tile_scores<QT, HD>(sm, raw);
#pragma unroll
    for (int j = 0; j < QT / 4; ++j) {
      const int i = w + 4 * j;
      const bool vis = l < nk && k0 + l <= sm.qpos[i];
      int64_t pw = 0;
      if (vis)
        pw = p.wrule == 0 ? attn_weight(sm.mx[i] - raw[j], sm.shift[i], p.lut, p.l2e)
                          : int8_weight(raw[j] - sm.mx[i], p.zsh, p.zmul, p.ptab);
      den[j] += pw;
      sm.Ps[i][l] = (int32_t)pw;
    }
    __syncthreads();
#pragma unroll 4
    for (int s = 0; s < nk; ++s) {
#pragma unroll
      for (int c = 0; c < HD / 64; ++c) {
        const int64_t vd = sm.Vs[s][l + 64 * c];
#pragma unroll
        for (int j = 0; j < QT / 4; ++j) num[j][c] += (int64_t)sm.Ps[w + 4 * j][s] * vd;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < QT / 4; ++j) den[j] = wave_sum64(den[j]);
}

// Key range [lo, hi) of split `sp` of [0, kend) in 64-key multiples.
__device__ __forceinline__ void split_range(int64_t kend, int nsplit, int sp, int64_t& lo, int64_t& hi) {
  const int64_t chunk = ((kend + nsplit - 1) / nsplit + 63) / 64 * 64;
  lo = imin(kend, sp * chunk);
  hi = imin(kend, lo + chunk);
}

// grid (groups * query tiles, nsplit). nsplit == 1: both sweeps, outputs written directly.
// nsplit > 1 and PHASE 0: maxima only (atomic max into mx_ws). PHASE 1: sums into the workspace; the last
// block of a group writes the outputs and restores the workspace (maxima, sums and counter back to 0).
template <int QT, int HD, bool PAGED, int PHASE>
__global__ __launch_bounds__(256) void attn_kernel(AttnArgs p) {
  extern __shared__ __align__(16) char smem_raw[];
  AttnSmem<QT, HD>& sm = *(AttnSmem<QT, HD>*)smem_raw;
  const int tiles = (p.nq + QT - 1) / QT;
  const int group = blockIdx.x / tiles, q0 = (blockIdx.x % tiles) * QT;
  const int nvalid = min(QT, p.nq - q0);
  const int h = PAGED ? group % p.hkv : 0;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t kend = stage_queries<QT, HD>(p, sm, group, q0, nvalid);
  int64_t lo, hi;
  split_range(kend, gridDim.y, blockIdx.y, lo, hi);

  if (gridDim.y == 1) {
    sweep_max<QT, HD, PAGED>(p, sm, group, h, lo, hi);
    int64_t den[QT / 4], num[QT / 4][HD / 64];
    sweep_acc<QT, HD, PAGED>(p, sm, group, h, lo, hi, den, num);
#pragma unroll
    for (int j = 0; j < QT / 4; ++j) {
      const int i = w + 4 * j;
      if (i < nvalid) {
#pragma unroll
        for (int c = 0; c < HD / 64; ++c)
          p.num[group * p.snum_tile + (int64_t)(q0 + i) * p.snum_row + l + 64 * c] = num[j][c];
        if (l == 0) p.den[group * p.sden_tile + q0 + i] = den[j];
      }
    }
    return;
  }
  const int64_t gq = (int64_t)group * p.nq + q0;   // workspace row of the tile's first query
  if (PHASE == 0) {
    sweep_max<QT, HD, PAGED>(p, sm, group, h, lo, hi);
    if (threadIdx.x < nvalid && hi > lo)
      atomicMax((long long*)&p.mx_ws[gq + threadIdx.x], (long long)(sm.mx[threadIdx.x] - kNeg));
    return;
  }
  if (threadIdx.x < QT) sm.mx[threadIdx.x] = threadIdx.x < nvalid ? p.mx_ws[gq + threadIdx.x] + kNeg : kNeg;
  __syncthreads();
  int64_t den[QT / 4], num[QT / 4][HD / 64];
  sweep_acc<QT, HD, PAGED>(p, sm, group, h, lo, hi, den, num);
  if (hi > lo) {
#pragma unroll
    for (int j = 0; j < QT / 4; ++j) {
      const int i = w + 4 * j;
      if (i < nvalid) {
#pragma unroll
        for (int c = 0; c < HD / 64; ++c)
          atomicAdd((unsigned long long*)&p.num_ws[(gq + i) * HD + l + 64 * c], (unsigned long long)num[j][c]);
        if (l == 0) atomicAdd((unsigned long long*)&p.den_ws[gq + i], (unsigned long long)den[j]);
      }
    }
  }
  // every split arrives (empty ones too), the last one publishes and restores the workspace
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int tile_id = blockIdx.x;
    const bool last = atomicAdd(&p.sem[tile_id], 1) == (int)gridDim.y - 1;
    if (last) atomicExch(&p.sem[tile_id], 0);
    sm.s_last = last;
  }
  __syncthreads();
  if (!sm.s_last) return;
  for (int u = threadIdx.x; u < nvalid * HD; u += 256) {
    const int i = u / HD, d = u % HD;
    p.num[group * p.snum_tile + (int64_t)(q0 + i) * p.snum_row + d] =
        (int64_t)atomicExch((unsigned long long*)&p.num_ws[(gq + i) * HD + d], 0ull);
  }
  if (threadIdx.x < nvalid) {
    p.den[group * p.sden_tile + q0 + threadIdx.x] =
        (int64_t)atomicExch((unsigned long long*)&p.den_ws[gq + threadIdx.x], 0ull);
    atomicExch((unsigned long long*)&p.mx_ws[gq + threadIdx.x], 0ull);
  }
}

// ---- paged decode attention on MFMA ----
// Grid (query tiles of <= 4 queries, key splits); a block is 8 independent waves, wave w taking the 16-key blocks
// w, w + 8, ... of the block's key range, with the next block's limb loads in flight while one is used.
// Scores: v_mfma_i32_16x16x64_i8 with the queries' limbs as A (row m = 4 query + limb; the fourth row of each
// query is zero) and one K limb plane as B straight from the cache (lane: key lane & 15, dims of chunk
// lane >> 4 -- the key row is contiguous along the MFMA depth). Lane l receives query l >> 4's limb rows for key
// l & 15 and joins them in int64: raw = sum_j sum_i acc_j[i] 2^(8 (i + j)) (|acc| <= HD 2^14, exact in int32).
// Sweep 1 keeps per-lane maxima. Sweep 2 turns scores into weights, puts the block's weights and joined V rows
// in the wave's own LDS slice and accumulates p V in int64 with one lane per dimension. Waves, then splits,
// are summed in a fixed order: partial maxima and sums go to per-split workspace slots with plain stores and the
// last block of a tile (counter) combines them, so no value is accumulated with atomics.
constexpr int kDecWaves = 8;
constexpr int kDecMaxSplit = 64;
constexpr int64_t kDecWsSplitBudget = 4096;
constexpr uint64_t kDecExchTicks = 20000;     // the exchange kernel's longest wait: 200 us at 100 MHz
constexpr int kDecExchBlocks = 256;           // the exchange kernel: at most one block per compute unit   // the workspace query sizes for min(64, 4096 / tiles) splits

template <int HD>
struct DecSmem {
  union {
    int32_t Vs[kDecWaves][16][HD + 1];   // sweep 2: each wave's joined V rows
    int64_t red[kDecWaves][4][HD];        // after it: each wave's p V sums
  };
  alignas(16) int32_t Ps[kDecWaves][16][4];   // sweep 2: [wave][key][query], one 16-byte read per key
  int64_t qpos[4];
  int64_t shift[4];
  int64_t mx[4];
  int64_t den[kDecWaves][4];
  int s_last;
};

template <int HD>
struct KvRegs {
  v4i k[3][HD / 64];
  v4i v[3][HD / 64];
};

// The cache block of key s (the block table entry: one load, issued an iteration ahead of the rows it locates).
__device__ __forceinline__ int dec_page(const AttnArgs& p, int64_t brow, int s) { return p.bt[brow * p.sbt + s / p.bs]; }

template <int HD, bool WANT_K, bool WANT_V>
__device__ __forceinline__ void dec_rows(const AttnArgs& p, int blk, int h, int s, KvRegs<HD>& r) {
  const int c = (threadIdx.x & 63) >> 4;
  const int8_t* row = p.cache + (int64_t)blk * p.sc_nb + (int64_t)h * p.sc_h + (int64_t)(s % p.bs) * p.sc_bs + c * 16;
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int kk = 0; kk < HD / 64; ++kk) {
      if (WANT_K) r.k[j][kk] = *(const v4i*)(row + j * HD + kk * 64);
      if (WANT_V) r.v[j][kk] = *(const v4i*)(row + (3 + j) * HD + kk * 64);
    }
}

template <int HD>
__device__ __forceinline__ int64_t dec_score(const v4i (&qa)[HD / 64], const KvRegs<HD>& r) {
  int64_t raw = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    v4i acc = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < HD / 64; ++kk) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa[kk], r.k[j][kk], acc, 0, 0, 0);
    const int64_t t = (int64_t)acc[0] + ((int64_t)acc[1] << 8) + ((int64_t)acc[2] << 16);
    raw += t << (8 * j);
  }
  return raw;
}

// workspace slots of tile t (per split sp): maxima (stored as mx - kNeg), p V sums, weight sums; then counters
struct DecWs {
  int64_t* mx;    // [T][NS][4]
  int64_t* num;   // [T][NS][4][HD]
  int64_t* den;   // [T][NS][4]
  int32_t* sem;   // [T]
};
__host__ __device__ __forceinline__ int64_t dec_ws_bytes(int64_t T, int64_t NS, int HD) {
  return T * NS * 4 * 8 * (2 + HD) + T * 4 + 256;
}

__device__ __forceinline__ DecWs dec_ws(const AttnArgs& p, int T, int NS, int HD) {
  const int64_t slots = (int64_t)T * NS * 4;
  char* b = (char*)p.mx_ws;
  DecWs w;
  w.mx = (int64_t*)b;
  w.num = (int64_t*)(b + slots * 8);
  w.den = (int64_t*)(b + slots * 8 * (1 + HD));
  w.sem = (int32_t*)(b + slots * 8 * (2 + HD));
  return w;
}

// The MFMA A operand of a tile's queries: limb (m & 3) of query (m >> 2), m = lane & 15, dims kk 64 +
// (lane >> 4) 16 + [0, 16); the fourth row of each query and queries past nvalid are 0. In two steps, so that a
// caller can issue the query loads first and use them after its other requests: dec_q_load reads the lane's 16
// values per 64 dims (16-byte loads when q is 16-byte aligned), dec_q_limbs packs the lane's limb.
template <int HD>
struct DecQ {
  int32_t x[HD / 64][16];
};

template <int HD>
__device__ __forceinline__ void dec_q_load(const AttnArgs& p, int group, int q0, int nvalid, int lane, DecQ<HD>& q) {
  const int m = lane & 15, qi = m >> 2, li = m & 3, c = lane >> 4;
  const bool live = qi < nvalid && li < 3;
  const int64_t base = group * p.sq_tile + (int64_t)(q0 + qi) * p.sq_row + c * 16;
  const bool vec = !p.q64 && ((reinterpret_cast<uintptr_t>(p.q + base)) & 15) == 0;
#pragma unroll
  for (int kk = 0; kk < HD / 64; ++kk) {
    if (vec) {
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const v4i v = live ? *(const v4i*)(p.q + base + kk * 64 + e4 * 4) : v4i{0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; ++e) q.x[kk][e4 * 4 + e] = v[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t qidx = base + kk * 64 + e;
        q.x[kk][e] = live ? (p.q64 ? (int32_t)p.q64[qidx] : p.q[qidx]) : 0;
      }
    }
  }
}

template <int HD>
__device__ __forceinline__ void dec_q_limbs(const DecQ<HD>& q, int lane, v4i (&qa)[HD / 64]) {
  const int li = lane & 3;
#pragma unroll
  for (int kk = 0; kk < HD / 64; ++kk) {
    int32_t word[4];
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      uint32_t wv = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int32_t x = q.x[kk][e4 * 4 + e];
        const int32_t a0 = limb_lo(x);
        x = (x - a0) >> 8;
        const int32_t a1 = limb_lo(x);
        x = (x - a1) >> 8;
        const int32_t a2 = limb_lo(x);
        const int32_t v = li == 0 ? a0 : li == 1 ? a1 : li == 2 ? a2 : 0;
        wv |= (uint32_t)(v & 255) << (8 * e);
      }
      word[e4] = (int32_t)wv;
    }
    qa[kk] = v4i{word[0], word[1], word[2], word[3]};
  }
}

template <int HD>
__device__ __forceinline__ void dec_qa(const AttnArgs& p, int group, int q0, int nvalid, int lane, v4i (&qa)[HD / 64]) {
  DecQ<HD> q;
  dec_q_load<HD>(p, group, q0, nvalid, lane, q);
  dec_q_limbs<HD>(q, lane, qa);
}

// The block's p V and weight sums (waves added in order) to the outputs (one split) or to the split's workspace
// slots; the last block of a tile (counter) adds the slots in split order, writes the outputs and puts the
// workspace back to zero (maxima slots included).
template <int HD>
__device__ __forceinline__ void dec_finish(const AttnArgs& p, DecSmem<HD>& sm, const DecWs& ws, int64_t den,
                                           int64_t (&num)[4][HD / 64], int tile, int sp, int NS, int group, int q0,
                                           int nvalid) {
  constexpr int KK = HD / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, kl = lane & 15, qo = lane >> 4;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) den += __shfl_xor(den, o, 64);
  if (kl == 0) sm.den[w][qo] = den;
  __syncthreads();                                 // red overlays the waves' V rows
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) sm.red[w][i][lane + 64 * kk] = num[i][kk];
  __syncthreads();
  // the block's sums, waves in order: thread u -> (query u / HD, dim u % HD)
  for (int u = threadIdx.x; u < 4 * HD + 4; u += kDecWaves * 64) {
    int64_t t = 0;
    if (u < 4 * HD) {
      for (int ww = 0; ww < kDecWaves; ++ww) t += sm.red[ww][u / HD][u % HD];
    } else {
      for (int ww = 0; ww < kDecWaves; ++ww) t += sm.den[ww][u - 4 * HD];
    }
    const int i = u < 4 * HD ? u / HD : u - 4 * HD;
    if (i >= nvalid) continue;
    if (NS == 1) {
      if (u < 4 * HD) p.num[group * p.snum_tile + (int64_t)(q0 + i) * p.snum_row + u % HD] = t;
      else p.den[group * p.sden_tile + q0 + i] = t;
    } else {
      const int64_t slot = (int64_t)tile * NS + sp;
      if (u < 4 * HD) ws_store(&ws.num[(slot * 4 + i) * HD + u % HD], t);
      else ws_store(&ws.den[slot * 4 + i], t);
    }
  }
  if (NS == 1) return;
  // every split arrives (its slot stores complete first); the last one adds the slots in split order
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    const bool last = atomicAdd(&ws.sem[tile], 1) == NS - 1;
    if (last) atomicExch(&ws.sem[tile], 0);
    sm.s_last = last;
  }
  __syncthreads();
  if (!sm.s_last) return;
  // every (split, entry) slot is read at once and added into LDS (exact in any order); the slots go back to
  // zero, so the workspace is left as it was found
  int64_t* fin = &sm.red[0][0][0];                 // 4 HD + 4 sums
  for (int u = threadIdx.x; u < 4 * HD + 4; u += kDecWaves * 64) fin[u] = 0;
  __syncthreads();
  constexpr int NT = kDecWaves * 64, UB = 8;      // UB slot loads in flight per thread
  const int nslot = NS * (4 * HD + 4);
  for (int u0 = threadIdx.x; u0 < nslot; u0 += NT * UB) {
    int64_t v[UB];
    int64_t* src[UB];
#pragma unroll
    for (int b = 0; b < UB; ++b) {
      const int u = u0 + b * NT;
      const int k = u / (4 * HD + 4), e = u % (4 * HD + 4);
      const int64_t slot = (int64_t)tile * NS + k;
      src[b] = e < 4 * HD ? &ws.num[slot * 4 * HD + e] : &ws.den[slot * 4 + (e - 4 * HD)];
      v[b] = u < nslot ? ws_load(src[b]) : 0;
    }
#pragma unroll
    for (int b = 0; b < UB; ++b) {
      const int u = u0 + b * NT;
      if (u < nslot) {
        atomicAdd((unsigned long long*)&fin[u % (4 * HD + 4)], (unsigned long long)v[b]);
        ws_store(src[b], 0);
      }
    }
  }
  for (int u = threadIdx.x; u < NS * 4; u += kDecWaves * 64) ws_store(&ws.mx[(int64_t)tile * NS * 4 + u], 0);
  __syncthreads();
  for (int u = threadIdx.x; u < nvalid * HD; u += kDecWaves * 64)
    p.num[group * p.snum_tile + (int64_t)(q0 + u / HD) * p.snum_row + u % HD] = fin[u];
  if (threadIdx.x < nvalid) p.den[group * p.sden_tile + q0 + threadIdx.x] = fin[4 * HD + threadIdx.x];
}

// The decode step's attention output stage (segs.attn_out: div_round + regroup + quant, src/bitexact/exact/segs.py
// and ops.py; the standalone form is attn_out_kernel in csrc/bx_rows.hip) fused into the one-block decode
// attention: ws_p int64 [R, H HD] (scratch) and ws_e int64 [R] / cnt int32 [R] (zero-filled workspace, left zero)
// are the exchange, q int32 [R, ldq] and sh int64 [R] the outputs.
struct AoArgs {
  int64_t* ws_p;
  int64_t* ws_e;
  int32_t* cnt;
  int32_t* q;
  int64_t ldq;
  int64_t* sh;
  int8_t* planes;   // optional: q's signed int8 limb planes [3][R][H HD] (limb i of q[n][c] at i plane + n H HD + c)
  int64_t plane;    // R H HD
  int FR, FV;
};

// The block's sums as dec_finish forms them (waves in order), then its queries' quotients P = div_round(num, FR -
// FV, den) (0 where den = 0), their exponent maximum into the token's slot (atomicMax of emax - kNegBig + 1) and the
// quotients into the token's row of ws_p (agent-scope stores, complete before the count); the token's last block
// quantizes the whole row against the row maximum (rshc(P, shr + FR), shr = max(emax - kQB, NEG_BIG)) and resets
// the slot and the count. No block waits for another.
template <int HD>
__device__ __forceinline__ void dec_finish_ao(const AttnArgs& p, const AoArgs& ao, DecSmem<HD>& sm, int64_t den,
                                              int64_t (&num)[4][HD / 64], int group, int nvalid) {
  constexpr int KK = HD / 64, NT = kDecWaves * 64;
  __shared__ int64_t s_den[4];
  __shared__ int64_t s_red[NT / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, kl = lane & 15, qo = lane >> 4;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) den += __shfl_xor(den, o, 64);
  if (kl == 0) sm.den[w][qo] = den;
  __syncthreads();                                 // red overlays the waves' V rows
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) sm.red[w][i][lane + 64 * kk] = num[i][kk];
  if (threadIdx.x < 4) {
    int64_t t = 0;
    for (int ww = 0; ww < kDecWaves; ++ww) t += sm.den[ww][threadIdx.x];
    s_den[threadIdx.x] = t;
  }
  __syncthreads();
  const int n = group / p.hkv, h = group % p.hkv, G = p.nq;
  const int64_t W = (int64_t)p.hkv * G * HD;
  int64_t emax = kNegBig;
  for (int u = threadIdx.x; u < nvalid * HD; u += NT) {
    const int i = u / HD, d = u % HD;
    int64_t t = 0;
    for (int ww = 0; ww < kDecWaves; ++ww) t += sm.red[ww][i][d];
    const int64_t dn = s_den[i];                   // >= 1 whenever the query sees a key (itself)
    const int64_t v = dn > 0 ? div_round64(t, ao.FR - ao.FV, dn, 1.0 / (double)dn) : 0;
    ws_store(&ao.ws_p[n * W + (int64_t)(h * G + i) * HD + d], v);
    if (v != 0) emax = imax(emax, bitlen(v < 0 ? -v : v) - ao.FR);
  }
  emax = block_max64(emax, s_red);
  if (threadIdx.x == 0) atomicMax((unsigned long long*)&ao.ws_e[n], (unsigned long long)(emax - kNegBig + 1));
  __builtin_amdgcn_s_waitcnt(0);                   // this thread's stores and atomic are complete before the count
  __syncthreads();
  if (threadIdx.x == 0) sm.s_last = atomicAdd(&ao.cnt[n], 1) == p.hkv - 1;
  __syncthreads();
  if (!sm.s_last) return;
  const int64_t em = (int64_t)ws_load(&ao.ws_e[n]) + kNegBig - 1;
  const int64_t shr = imax(em - kQB, kNegBig);
  for (int64_t c = threadIdx.x; c < W; c += NT) {
    const int32_t qv = (int32_t)rshc(ws_load(&ao.ws_p[n * W + c]), shr + ao.FR);
    ao.q[n * ao.ldq + c] = qv;
    if (ao.planes != nullptr) {   // the exact linear's activation planes (split_q_kernel's limbs)
      int32_t r = qv;
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        const int32_t lo = limb_lo(r);
        ao.planes[l * ao.plane + n * W + c] = (int8_t)lo;
        r = (r - lo) >> 8;
      }
    }
  }
  if (threadIdx.x == 0) {
    ao.sh[n] = shr;
    ws_store(&ao.ws_e[n], 0);
    atomicExch(&ao.cnt[n], 0);
  }
}

// RAW (split launches): phase 0 writes every score to p.raw ([tile][key][query] int64, p.S keys a tile) and phase 1
// reads them back, 32 bytes a key instead of K's 3 HD again. With splits for about two blocks a CU in both launches
// this is the form of long contexts and of grids that neither fill the chip unsplit nor fit the exchange kernel.
// The host chooses it by the table's width; a tile whose context is short (p.one_keys) is one block's in phase 1, as
// the exchange between the phases costs more than its keys: 128 tiles of 128 keys (heads of 64) 14.3 -> 11.7 us, of
// 256 16.0 -> 14.6; at 384 both take 17.4, and heads of 128 cross at half the keys.
// LIST: the token rows of p.list, whose number only the device knows: block b takes tile b % T of T and split b / T, with
// as many splits as make kDecListBlocks blocks (at least 128 keys of the table each); one split: phase 1 alone.
constexpr int kDecListBlocks = 512;
template <int HD, int PHASE, bool RAW, bool LIST = false>
__global__ __launch_bounds__(kDecWaves * 64) void attn_dec_kernel(AttnArgs p) {
  __shared__ DecSmem<HD> sm;
  constexpr int KK = HD / 64;
  const int tiles = (p.nq + 3) / 4;
  int tile = blockIdx.x, T = gridDim.x, sp = blockIdx.y, NS = gridDim.y;
  if constexpr (LIST) {
    T = p.list[0] * p.hkv;
    if (T == 0) return;
    NS = max(min(min(kDecListBlocks / T, kDecMaxSplit), p.S / 128), 1);
    sp = tile / T;
    tile -= sp * T;
    if (sp >= NS || (PHASE == 0 && NS == 1)) return;         // block-uniform
  }
  int64_t* raws = RAW ? p.raw + (int64_t)tile * p.S * 4 : nullptr;
  const int group = LIST ? p.list[1 + tile / p.hkv] * p.hkv + tile % p.hkv : tile / tiles;
  const int q0 = LIST ? 0 : (tile % tiles) * 4;
  const int nvalid = min(4, p.nq - q0);
  const int h = group % p.hkv;
  const int64_t brow = p.rmap ? p.rmap[group / p.hkv] : group / p.hkv;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int kl = lane & 15, qo = lane >> 4;
  DecWs ws = dec_ws(p, T, NS, HD);
  if constexpr (LIST) ws.sem = p.sem;                // (a place that does not depend on T)

  if (threadIdx.x < 4) {
    const int i = threadIdx.x;
    const bool ok = i < nvalid;
    sm.qpos[i] = ok ? p.qpos[(group / p.qpos_div) * p.qpos_tile + (int64_t)(q0 + i) * p.qpos_row] : -1;
    sm.shift[i] = ok && p.sh ? (int64_t)(kFK + 3 - kFZ) - p.sh[group * p.sh_tile + q0 + i] : 0;
    sm.mx[i] = kNeg;
  }
  v4i qa[KK];
  dec_qa<HD>(p, group, q0, nvalid, lane, qa);
  __syncthreads();
  int64_t kend = 0;
  for (int i = 0; i < 4; ++i) kend = imax(kend, sm.qpos[i] + 1);
  if (RAW || LIST) kend = imin(kend, p.S);         // (qpos < the block table's keys: the scores' bound in any case)
  if (RAW) {
    if (kend <= p.one_keys) {                      // block-uniform: phase 1's split 0 alone, both sweeps
      if (PHASE == 0 || sp > 0) return;
      NS = 1;
    }
  }
  int64_t lo64, hi64;
  split_range(kend, NS, sp, lo64, hi64);
  const int lo = (int)lo64, hi = (int)hi64;
  const int64_t my_qpos = sm.qpos[qo];
  const int nb16 = (hi - lo + 15) / 16;

  // ---- sweep 1: maxima over visible keys ----
  if (PHASE == 0 || NS == 1) {
    int64_t best = kNeg;
    KvRegs<HD> cur, nxt;
    // pipeline per wave: rows of block b + 8 and the page of block b + 16 are requested while block b is used
    int pg = 0;
    if (w < nb16) dec_rows<HD, true, false>(p, dec_page(p, brow, min(lo + w * 16 + kl, hi - 1)), h,
                                            min(lo + w * 16 + kl, hi - 1), cur);
    if (w + kDecWaves < nb16) pg = dec_page(p, brow, min(lo + (w + kDecWaves) * 16 + kl, hi - 1));
    for (int b = w; b < nb16; b += kDecWaves) {
      const int s = lo + b * 16 + kl;
      if (b + kDecWaves < nb16) dec_rows<HD, true, false>(p, pg, h, min(s + 16 * kDecWaves, hi - 1), nxt);
      if (b + 2 * kDecWaves < nb16) pg = dec_page(p, brow, min(s + 32 * kDecWaves, hi - 1));
      const int64_t raw = dec_score<HD>(qa, cur);
      if (RAW && s < hi) raws[(int64_t)s * 4 + qo] = raw;
      if (s < hi && s <= my_qpos) best = imax(best, raw);
      cur = nxt;
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) best = imax(best, __shfl_xor(best, o, 64));
    if (kl == 0) atomicMax((long long*)&sm.mx[qo], (long long)best);
    __syncthreads();
    if (NS > 1) {                       // PHASE 0: this split's maxima (kNeg: none) into its slot
      if (threadIdx.x < 4) ws_store(&ws.mx[((int64_t)tile * NS + sp) * 4 + threadIdx.x], sm.mx[threadIdx.x] - kNeg);
      return;
    }
  } else {                              // PHASE 1 of a split launch: the maxima over every split
    __syncthreads();                    // sm.mx holds kNeg
    for (int u = threadIdx.x; u < NS * 4; u += kDecWaves * 64)      // every split's slot at once
      atomicMax((long long*)&sm.mx[u & 3], (long long)(ws_load(&ws.mx[(int64_t)tile * NS * 4 + u]) + kNeg));
    __syncthreads();
  }

  // ---- sweep 2: weights, den, num ----
  const int64_t mx = sm.mx[qo];
  const int64_t shift = sm.shift[qo];
  int64_t den = 0;
  int64_t num[4][KK];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) num[i][kk] = 0;
  KvRegs<HD> cur, nxt;
  int pg = 0;
  int64_t rcur = 0, rnxt = 0;
  if (w < nb16) {
    const int s = min(lo + w * 16 + kl, hi - 1);
    if (RAW) rcur = raws[(int64_t)s * 4 + qo];
    dec_rows<HD, !RAW, true>(p, dec_page(p, brow, s), h, s, cur);
  }
  if (w + kDecWaves < nb16) pg = dec_page(p, brow, min(lo + (w + kDecWaves) * 16 + kl, hi - 1));
  for (int b = w; b < nb16; b += kDecWaves) {
    const int s = lo + b * 16 + kl;
    const int64_t raw = RAW ? rcur : dec_score<HD>(qa, cur);
    // the weight's table loads go out before the next block's requests (loads complete in order: waiting for
    // them then does not wait for the prefetch) and unconditionally (a hidden key's weight is discarded)
    WeightAt wat;
    int64_t ta = 0, tb = 0, i8 = 0;
    if (p.wrule == 0) {
      wat = weight_at(mx - raw, shift, p.l2e);
      ta = p.lut[wat.idx];
      tb = p.lut[wat.idx + 1];
    } else {
      i8 = int8_index(raw - mx, p.zsh, p.zmul);
      ta = p.ptab[imin(imax(i8, 0), -kI8ZLo)];   // a visible key has d <= 0, so idx <= -kI8ZLo (z = 0)
    }
    if (b + kDecWaves < nb16) {
      dec_rows<HD, !RAW, true>(p, pg, h, min(s + 16 * kDecWaves, hi - 1), nxt);
      if (RAW) rnxt = raws[(int64_t)min(s + 16 * kDecWaves, hi - 1) * 4 + qo];
    }
    if (b + 2 * kDecWaves < nb16) pg = dec_page(p, brow, min(s + 32 * kDecWaves, hi - 1));
    int64_t pw = p.wrule == 0 ? weight_of(wat, ta, tb) : (i8 >= 0 ? ta : 0);
    if (!(qo < nvalid && s < hi && s <= my_qpos)) pw = 0;
    den += pw;
    sm.Ps[w][kl][qo] = (int32_t)pw;
    const int c = lane >> 4;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const int32_t w0 = cur.v[0][kk][e4], w1 = cur.v[1][kk][e4], w2 = cur.v[2][kk][e4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int32_t b0 = (w0 << (24 - 8 * e)) >> 24, b1 = (w1 << (24 - 8 * e)) >> 24, b2 = (w2 << (24 - 8 * e)) >> 24;
          sm.Vs[w][kl][kk * 64 + c * 16 + e4 * 4 + e] = b0 + b1 * 256 + b2 * 65536;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);           // lgkmcnt(0): this wave's LDS writes are done
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      int64_t vd[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) vd[kk] = sm.Vs[w][k][lane + 64 * kk];
      const v4i pk = *(const v4i*)&sm.Ps[w][k][0];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t pv = pk[i];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) num[i][kk] += pv * vd[kk];
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
    cur = nxt;
    rcur = rnxt;
  }
  dec_finish<HD>(p, sm, ws, den, num, tile, sp, NS, group, q0, nvalid);
}

// A key's weight in two halves: dec_w_issue sends the table loads of one score (always inside the table,
// whatever the score: a hidden key's weight is discarded), dec_w_value forms the weight once they are in.
struct DecW {
  WeightAt wat;
  int64_t ta, tb, i8;
};

__device__ __forceinline__ DecW dec_w_issue(const AttnArgs& p, int64_t raw, int64_t mx, int64_t shift) {
  DecW d;
  d.tb = 0;
  d.i8 = 0;
  if (p.wrule == 0) {
    d.wat = weight_at(mx - raw, shift, p.l2e);
    d.ta = p.lut[d.wat.idx];
    d.tb = p.lut[d.wat.idx + 1];
  } else {
    d.i8 = int8_index(raw - mx, p.zsh, p.zmul);
    d.ta = p.ptab[imin(imax(d.i8, 0), -kI8ZLo)];   // a visible key has d <= 0, so idx <= -kI8ZLo (z = 0)
  }
  return d;
}

__device__ __forceinline__ int64_t dec_w_value(const AttnArgs& p, const DecW& d) {
  return p.wrule == 0 ? weight_of(d.wat, d.ta, d.tb) : (d.i8 >= 0 ? d.ta : 0);
}

// p V of one 16-key block of a wave: the weights (lane: key kl, query qo) and the joined V rows (from the three
// limb planes the lane holds: key kl, dims of chunk lane >> 4) meet in the wave's LDS slice; lane l then adds
// sum_k p[k][i] V[k][l + 64 kk] for the four queries i.
template <int HD>
__device__ __forceinline__ void dec_pv(DecSmem<HD>& sm, int w, int lane, int64_t pw, const v4i (&v)[3][HD / 64],
                                       int64_t (&num)[4][HD / 64]) {
  constexpr int KK = HD / 64;
  const int kl = lane & 15, qo = lane >> 4, c = lane >> 4;
  sm.Ps[w][kl][qo] = (int32_t)pw;
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      const int32_t w0 = v[0][kk][e4], w1 = v[1][kk][e4], w2 = v[2][kk][e4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int32_t b0 = (w0 << (24 - 8 * e)) >> 24, b1 = (w1 << (24 - 8 * e)) >> 24, b2 = (w2 << (24 - 8 * e)) >> 24;
        sm.Vs[w][kl][kk * 64 + c * 16 + e4 * 4 + e] = b0 + b1 * 256 + b2 * 65536;
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);           // lgkmcnt(0): this wave's LDS writes are done
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    int64_t vd[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) vd[kk] = sm.Vs[w][k][lane + 64 * kk];
    const v4i pk = *(const v4i*)&sm.Ps[w][k][0];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t pv = pk[i];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) num[i][kk] += pv * vd[kk];
    }
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_wave_barrier();
}

// One key row's three limb planes (K: planes 0-2, V: planes 3-5 of the cache row) for the lane: key s of cache
// block pg, dims of chunk lane >> 4.
template <int HD>
__device__ __forceinline__ void dec_planes(const AttnArgs& p, int pg, int h, int s, int first, v4i (&r)[3][HD / 64]) {
  const int c = (threadIdx.x & 63) >> 4;
  const int8_t* row = p.cache + (int64_t)pg * p.sc_nb + (int64_t)h * p.sc_h + (int64_t)(s % p.bs) * p.sc_bs + c * 16;
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int kk = 0; kk < HD / 64; ++kk) r[j][kk] = *(const v4i*)(row + (first + j) * HD + kk * 64);
}

template <int HD>
__device__ __forceinline__ int64_t dec_score_k(const v4i (&qa)[HD / 64], const v4i (&k)[3][HD / 64]) {
  int64_t raw = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    v4i acc = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < HD / 64; ++kk) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa[kk], k[j][kk], acc, 0, 0, 0);
    const int64_t t = (int64_t)acc[0] + ((int64_t)acc[1] << 8) + ((int64_t)acc[2] << 16);
    raw += t << (8 * j);
  }
  return raw;
}

// ---- paged decode attention, one block per query tile, up to kDecRawKeys keys ----
// The tile's block-table entries are copied to LDS first, so locating a key row costs an LDS read rather than a
// memory round trip. Each wave keeps the limb rows of its next DR 16-key blocks in flight (a register ring, the
// loop unrolled by DR). Sweep 1 streams K, keeps every score in LDS and the per-query maxima; sweep 2 streams V
// and forms weights and p V from the kept scores, so K and V are each read once.
// RP (decode steps with one token per sequence): the block first runs the rope kernel's work for its (token, KV
// head): waves 0 .. nq - 1 RoPE and quantize the group's q heads into LDS, waves 4 and 5 RoPE the k head and
// store the k and v limbs at the token's cache slot (each waits for its stores before the barrier, so the
// sweeps read them back). The launch then replaces the standalone rope kernel.
constexpr int kDecDepth = 3;
template <int HD, bool RP = false, bool AO = false>
__global__ __launch_bounds__(kDecWaves * 64) void attn_dec_raw_kernel(AttnArgs p, RopeArgs r, AoArgs ao) {
  static_assert(!RP || kDecWaves >= 6, "the rope prologue uses waves 0-3 (q heads), 4 (k) and 5 (v)");
  BX_PHASE(1, 0);
  __shared__ DecSmem<HD> sm;
  extern __shared__ __align__(16) int64_t raw_cache[];     // [4][p.S] scores, then the block-table entries
  constexpr int KK = HD / 64, DR = kDecDepth;
  const int tiles = (p.nq + 3) / 4;
  const int tile = blockIdx.x;
  const int group = tile / tiles, q0 = (tile % tiles) * 4;
  const int nvalid = min(4, p.nq - q0);
  const int h = group % p.hkv;
  const int64_t brow = p.rmap ? p.rmap[group / p.hkv] : group / p.hkv;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kl = lane & 15, qo = lane >> 4;
  int32_t* spg = (int32_t*)(raw_cache + 4 * (int64_t)p.S);
  __shared__ int32_t s_q[RP ? 4 : 1][RP ? HD : 1];
  __shared__ int64_t s_shq[4];

  DecQ<HD> qv;
  if constexpr (!RP) dec_q_load<HD>(p, group, q0, nvalid, lane, qv);
  // the block-table row (every entry the launch may reach: p.S / bs + 1), independent of the positions
  const int npg = p.S / p.bs + 1 < p.nblk ? p.S / p.bs + 1 : p.nblk;
  for (int i = threadIdx.x; i < npg; i += kDecWaves * 64) spg[i] = p.bt[brow * p.sbt + i];
  // RP: the wave's first DR key blocks that lie wholly below the token's position (no prologue store touches
  // them) are requested before the prologue, straight from the block table; the sweep loads the rest
  v4i kr[DR][3][KK];
  int npre = 0;                                             // wave-uniform: kr[0 .. npre) already requested
  if constexpr (RP) {
    const int64_t pos0 = r.pos[(int64_t)(group / p.hkv) * r.spb];
    const int64_t pe = pos0 < p.S ? pos0 : p.S - 1;        // the last visible key
#pragma unroll
    for (int d = 0; d < DR; ++d) {
      const int i = w + d * kDecWaves;
      if (npre == d && pos0 >= 0 && (int64_t)(i + 1) * 16 <= pe) {   // wave-uniform
        const int s = i * 16 + kl;
        dec_planes<HD>(p, p.bt[brow * p.sbt + s / p.bs], h, s, 0, kr[d]);
        npre = d + 1;
      }
    }
  }
  int64_t qp[4];
  if constexpr (RP) {
    // token group / hkv, KV head h, its nq q heads h nq ..; one position for the group (the token's)
    const int n = group / p.hkv;
    const int64_t pos_raw = r.pos[(int64_t)n * r.spb];
    bool bad = pos_raw < 0 || pos_raw >= r.npos;        // the reference's table index would fail: flagged
    const int64_t pos = imin(imax(pos_raw, 0), r.npos - 1);
    int64_t out[KK];
    if (w < nvalid) {
      rope_row<HD>(r, n, h * p.nq + w, pos, lane, out, bad);
      const int64_t shq = rope_q_shift<HD>(r, out, bad);
#pragma unroll
      for (int e = 0; e < KK; ++e) s_q[w][lane + 64 * e] = (int32_t)rshc(out[e], shq + r.FR + r.FT);
      if (lane == 0) s_shq[w] = shq;
    } else if (w == 4 || w == 5) {
      const int hr = r.H + (w - 4) * r.HKV + h;
      rope_row<HD>(r, n, hr, pos, lane, out, bad);
      rope_kv_store<HD>(r, n, hr, lane, out, bad);
      __builtin_amdgcn_s_waitcnt(0);                     // the cache stores are complete before the barrier
    }
    if (wave_or(bad ? 1 : 0) && lane == 0) r.err[0] = 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) qp[i] = i < nvalid ? pos_raw : -1;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      qp[i] = i < nvalid ? p.qpos[(group / p.qpos_div) * p.qpos_tile + (int64_t)(q0 + i) * p.qpos_row] : -1;
  }
  const int kend = (int)imin(imax(imax(qp[0], qp[1]), imax(qp[2], qp[3])) + 1, p.S);   // qpos < nblk bs <= p.S
  const int64_t my_qpos = qo == 0 ? qp[0] : qo == 1 ? qp[1] : qo == 2 ? qp[2] : qp[3];
  if (threadIdx.x < 4) sm.mx[threadIdx.x] = kNeg;
  int64_t shift = 0;
  if constexpr (!RP) shift = qo < nvalid && p.sh ? (int64_t)(kFK + 3 - kFZ) - p.sh[group * p.sh_tile + q0 + qo] : 0;
  __syncthreads();
  if constexpr (RP) {
    // the queries from LDS in dec_q_load's lane layout: query (lane & 15) >> 2, dims 16 (lane >> 4) + e
    const int m = lane & 15, qi = m >> 2, c = lane >> 4;
    const bool live = qi < nvalid && (m & 3) < 3;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int e = 0; e < 16; ++e) qv.x[kk][e] = live ? s_q[qi][kk * 64 + c * 16 + e] : 0;
    shift = qo < nvalid ? (int64_t)(kFK + 3 - kFZ) - s_shq[qo] : 0;
  }
  v4i qa[KK];
  dec_q_limbs<HD>(qv, lane, qa);
  const int nb16 = (kend + 15) / 16;
  BX_PHASE(1, 1);
  auto rows = [&](int i, int first, v4i (&r)[3][KK]) {
    const int s = min(i * 16 + kl, kend - 1);
    dec_planes<HD>(p, spg[s / p.bs], h, s, first, r);
  };

  // ---- sweep 1: K, scores into LDS, maxima ----
  {
#pragma unroll
    for (int d = 0; d < DR; ++d)
      if (d >= npre && w + d * kDecWaves < nb16) rows(w + d * kDecWaves, 0, kr[d]);
    int64_t best = kNeg;
    for (int b0 = w; b0 < nb16; b0 += DR * kDecWaves) {
#pragma unroll
      for (int d = 0; d < DR; ++d) {
        const int i = b0 + d * kDecWaves;
        if (i < nb16) {                              // wave-uniform
          const int64_t raw = dec_score_k<HD>(qa, kr[d]);
          if (i + DR * kDecWaves < nb16) rows(i + DR * kDecWaves, 0, kr[d]);
          const int s = i * 16 + kl;
          if (s < kend) raw_cache[qo * p.S + s] = raw;
          if (s < kend && s <= my_qpos) best = imax(best, raw);
        }
      }
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) best = imax(best, __shfl_xor(best, o, 64));
    if (kl == 0) atomicMax((long long*)&sm.mx[qo], (long long)best);
  }
  BX_PHASE(1, 2);
  // the first V rows go out before the maxima are complete
  v4i vr[DR][3][KK];
#pragma unroll
  for (int d = 0; d < DR; ++d)
    if (w + d * kDecWaves < nb16) rows(w + d * kDecWaves, 3, vr[d]);
  __builtin_amdgcn_s_waitcnt(0xc07f);             // LDS only (lgkmcnt(0)): the V loads stay in flight
  asm volatile("s_barrier" ::: "memory");

  BX_PHASE(1, 3);
  // ---- sweep 2: V, weights from the kept scores, den, p V ----
  const int64_t mx = sm.mx[qo];
  int64_t den = 0;
  int64_t num[4][KK];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) num[i][kk] = 0;
  for (int b0 = w; b0 < nb16; b0 += DR * kDecWaves) {
#pragma unroll
    for (int d = 0; d < DR; ++d) {
      const int i = b0 + d * kDecWaves;
      if (i < nb16) {                                // wave-uniform
        const int s = i * 16 + kl;
        const int64_t raw = s < kend ? raw_cache[qo * p.S + s] : 0;
        const DecW wt = dec_w_issue(p, raw, mx, shift);
        int64_t pw = dec_w_value(p, wt);
        if (!(qo < nvalid && s < kend && s <= my_qpos)) pw = 0;
        den += pw;
        dec_pv<HD>(sm, w, lane, pw, vr[d], num);
        if (i + DR * kDecWaves < nb16) rows(i + DR * kDecWaves, 3, vr[d]);
      }
    }
  }
  BX_PHASE(1, 4);
  if constexpr (AO)
    dec_finish_ao<HD>(p, ao, sm, den, num, group, nvalid);
  else
    dec_finish<HD>(p, sm, DecWs{}, den, num, tile, 0, 1, group, q0, nvalid);
  BX_PHASE(1, 5);
}

// ---- paged decode attention, key splits in one launch ----
// Grid (query tiles, key splits), every block normally resident at once (the host takes this kernel for at most
// one block per compute unit). A block's key range is at most 16 NBW kDecWaves keys, so wave w holds the K and V
// limb rows of its NBW 16-key blocks in registers: the block-table entries, then every K and V row, are requested
// at once, before the queries are read. Scores stay in registers. The splits of a tile exchange their maxima
// through the workspace: each publishes its own (as mx - kNeg + 1; 0 = not yet published) and waits for the
// others' for at most p.exch_ticks of the 100 MHz real-time counter; a block that has not seen them all by then
// computes the maxima over the tile's keys itself, so the wait always ends and the integers never depend on which
// blocks ran together. Weights, p V and the split sums then follow attn_dec_kernel's sweep 2 and dec_finish,
// so K and V are each read once.
template <int HD, int NBW>
__global__ __launch_bounds__(kDecWaves * 64) void attn_dec_exch_kernel(AttnArgs p) {
  BX_PHASE(0, 0);
  __shared__ DecSmem<HD> sm;
  __shared__ int64_t s_best[kDecWaves][4];
  constexpr int KK = HD / 64;
  const int tiles = (p.nq + 3) / 4;
  const int tile = blockIdx.x, T = gridDim.x, sp = blockIdx.y, NS = gridDim.y;
  const int group = tile / tiles, q0 = (tile % tiles) * 4;
  const int nvalid = min(4, p.nq - q0);
  const int h = group % p.hkv;
  const int64_t brow = p.rmap ? p.rmap[group / p.hkv] : group / p.hkv;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kl = lane & 15, qo = lane >> 4;
  const DecWs ws = dec_ws(p, T, NS, HD);

  DecQ<HD> qv;                                     // the queries first: used after every other request
  dec_q_load<HD>(p, group, q0, nvalid, lane, qv);
  // the tile's query positions, read by every lane (the key range needs their maximum)
  int64_t qp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    qp[i] = i < nvalid ? p.qpos[(group / p.qpos_div) * p.qpos_tile + (int64_t)(q0 + i) * p.qpos_row] : -1;
  const int64_t kend = imax(imax(qp[0], qp[1]), imax(qp[2], qp[3])) + 1;
  const int64_t my_qpos = qo == 0 ? qp[0] : qo == 1 ? qp[1] : qo == 2 ? qp[2] : qp[3];
  int64_t lo64, hi64;
  split_range(kend, NS, sp, lo64, hi64);
  const int lo = (int)lo64, hi = (int)hi64;
  const int nb16 = (hi - lo + 15) / 16;            // <= NBW kDecWaves (the host's bound on the split size)
  int pg[NBW];
#pragma unroll
  for (int t = 0; t < NBW; ++t)
    pg[t] = w + t * kDecWaves < nb16 ? dec_page(p, brow, min(lo + (w + t * kDecWaves) * 16 + kl, hi - 1)) : 0;
  KvRegs<HD> kv[NBW];
#pragma unroll
  for (int t = 0; t < NBW; ++t)
    if (w + t * kDecWaves < nb16)
      dec_rows<HD, true, true>(p, pg[t], h, min(lo + (w + t * kDecWaves) * 16 + kl, hi - 1), kv[t]);
  if (threadIdx.x < 4) sm.mx[threadIdx.x] = kNeg;
  const int64_t shift = qo < nvalid && p.sh ? (int64_t)(kFK + 3 - kFZ) - p.sh[group * p.sh_tile + q0 + qo] : 0;
  v4i qa[KK];
  dec_q_limbs<HD>(qv, lane, qa);

  // scores and this split's maxima
  int64_t raw[NBW];
  int64_t best = kNeg;
#pragma unroll
  for (int t = 0; t < NBW; ++t) {
    raw[t] = 0;
    if (w + t * kDecWaves < nb16) {                // wave-uniform
      const int s = lo + (w + t * kDecWaves) * 16 + kl;
      raw[t] = dec_score<HD>(qa, kv[t]);
      if (s < hi && s <= my_qpos) best = imax(best, raw[t]);
    }
  }
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) best = imax(best, __shfl_xor(best, o, 64));
  if (kl == 0) s_best[w][qo] = best;
  __syncthreads();
  BX_PHASE(0, 1);
  if (threadIdx.x < 4) {
    int64_t m = kNeg;
    for (int ww = 0; ww < kDecWaves; ++ww) m = imax(m, s_best[ww][threadIdx.x]);
    ws_store(&ws.mx[((int64_t)tile * NS + sp) * 4 + threadIdx.x], m - kNeg + 1);
  }
  bool seen = true;
  if (threadIdx.x < NS * 4) {
    int64_t* a = &ws.mx[(int64_t)tile * NS * 4 + threadIdx.x];
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    int64_t v = ws_load(a);
    while (v == 0 && __builtin_amdgcn_s_memrealtime() - t0 < p.exch_ticks) {
      __builtin_amdgcn_s_sleep(1);
      v = ws_load(a);
    }
    seen = v != 0;
    if (seen) atomicMax((long long*)&sm.mx[threadIdx.x & 3], (long long)(v - 1 + kNeg));
  }
  if (!__syncthreads_and(seen)) {
    // maxima over every key of the tile, from the cache (rows of 16 keys, the waves in turn)
    const int nall = (int)((kend + 15) / 16);
    int64_t b2 = kNeg;
    for (int i = w; i < nall; i += kDecWaves) {
      const int s = min(i * 16 + kl, (int)kend - 1);
      KvRegs<HD> r;
      dec_rows<HD, true, false>(p, dec_page(p, brow, s), h, s, r);
      const int64_t sc = dec_score<HD>(qa, r);
      if (i * 16 + kl < kend && s <= my_qpos) b2 = imax(b2, sc);
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) b2 = imax(b2, __shfl_xor(b2, o, 64));
    if (kl == 0) atomicMax((long long*)&sm.mx[qo], (long long)b2);
    __syncthreads();
  }

  BX_PHASE(0, 2);
  // weights (every table load first), den, p V
  const int64_t mx = sm.mx[qo];
  int64_t pw[NBW];
  {
    WeightAt wat[NBW];
    int64_t ta[NBW], tb[NBW], i8[NBW];
#pragma unroll
    for (int t = 0; t < NBW; ++t) {
      if (p.wrule == 0) {
        wat[t] = weight_at(mx - raw[t], shift, p.l2e);
        ta[t] = p.lut[wat[t].idx];
        tb[t] = p.lut[wat[t].idx + 1];
      } else {
        i8[t] = int8_index(raw[t] - mx, p.zsh, p.zmul);
        ta[t] = p.ptab[imin(imax(i8[t], 0), -kI8ZLo)];   // a visible key has d <= 0, so idx <= -kI8ZLo (z = 0)
      }
    }
#pragma unroll
    for (int t = 0; t < NBW; ++t) {
      const int s = lo + (w + t * kDecWaves) * 16 + kl;
      pw[t] = p.wrule == 0 ? weight_of(wat[t], ta[t], tb[t]) : (i8[t] >= 0 ? ta[t] : 0);
      if (!(w + t * kDecWaves < nb16 && qo < nvalid && s < hi && s <= my_qpos)) pw[t] = 0;
    }
  }
  int64_t den = 0;
  int64_t num[4][KK];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) num[i][kk] = 0;
  const int c = lane >> 4;
#pragma unroll
  for (int t = 0; t < NBW; ++t) {
    if (w + t * kDecWaves >= nb16) break;          // wave-uniform
    den += pw[t];
    sm.Ps[w][kl][qo] = (int32_t)pw[t];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const int32_t w0 = kv[t].v[0][kk][e4], w1 = kv[t].v[1][kk][e4], w2 = kv[t].v[2][kk][e4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int32_t b0 = (w0 << (24 - 8 * e)) >> 24, b1 = (w1 << (24 - 8 * e)) >> 24, b2 = (w2 << (24 - 8 * e)) >> 24;
          sm.Vs[w][kl][kk * 64 + c * 16 + e4 * 4 + e] = b0 + b1 * 256 + b2 * 65536;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);           // lgkmcnt(0): this wave's LDS writes are done
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      int64_t vd[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) vd[kk] = sm.Vs[w][k][lane + 64 * kk];
      const v4i pk = *(const v4i*)&sm.Ps[w][k][0];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t pv = pk[i];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) num[i][kk] += pv * vd[kk];
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
  }
  BX_PHASE(0, 3);
  dec_finish<HD>(p, sm, ws, den, num, tile, sp, NS, group, q0, nvalid);
  BX_PHASE(0, 4);
}

// ---- fused prefill attention on MFMA (contiguous int32 K / V) ----
// A block (4 waves) owns 64 consecutive query rows of one group z; wave w owns rows 16 w .. 16 w + 15. Keys go
// in 64-key tiles staged in LDS as int8 limb planes: K row-major (Ks[j][key][dim], the QK B operand: a lane's
// 16 bytes are 16 dims of one key) and V transposed (Vt[j][dim][key], the PV B operand: 16 keys of one dim).
// QK: for each 16-key block, A = limb i of the wave's 16 queries (registers), B = K limb plane j; the nine limb
// products accumulate by weight i + j in five int32 sets, joined in int64 per score (lane: query rows
// 4 (lane >> 4) + e, key lane & 15). Sweep 1 keeps per-row maxima; sweep 2 turns scores into weights p, writes
// p's three limbs to the wave's LDS slice (Pl[i][query][key]) and runs PV on MFMA: A = limb i of p (16
// queries x 64 keys), B = V limb plane j (64 keys x 16 dims), five int32 sets per 16-dim block, exact while
// S 3 2^14 < 2^31 (S < 43690), joined in int64 at the end.
template <int HD>
struct PreSmem {
  int8_t Ks[3][64][HD + 16];
  int8_t Vt[3][HD][64 + 16];
  int8_t Pl[4][3][16][64 + 16];
};

// A tile's K / V rows in registers (thread -> K: (key, 16-dim chunk) units; V: (4 keys, 4 dims) units), loaded
// while the previous tile is computed, then split into limb planes in LDS.
template <int HD>
struct PreRegs {
  v4i k[HD / 64][4];
  v4i v[HD / 64][4];
};

template <int HD>
__device__ __forceinline__ void pre_load(const AttnArgs& p, PreRegs<HD>& r, int z, int key0, int kend, bool want_v) {
#pragma unroll
  for (int t = 0; t < HD / 64; ++t) {
    const int u = threadIdx.x + t * 256;
    const int kk = u / (HD / 16), c = u % (HD / 16);
    const int s = min(key0 + kk, kend - 1);
    const int32_t* kr = p.K + (int64_t)z * p.sk_z + (int64_t)s * p.sk_s + c * 16;
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) r.k[t][e4] = *(const v4i*)(kr + e4 * 4);
    if (want_v) {
      const int kq = u % 16, dq = u / 16;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int sv = min(key0 + 4 * kq + m, kend - 1);
        r.v[t][m] = *(const v4i*)(p.V + (int64_t)z * p.sv_z + (int64_t)sv * p.sv_s + dq * 4);
      }
    }
  }
}

template <int HD>
__device__ __forceinline__ void pre_store(PreSmem<HD>& sm, const PreRegs<HD>& r, bool want_v) {
#pragma unroll
  for (int t = 0; t < HD / 64; ++t) {
    const int u = threadIdx.x + t * 256;
    const int kk = u / (HD / 16), c = u % (HD / 16);
    uint32_t w0[4], w1[4], w2[4];
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) split3(r.k[t][e4], w0[e4], w1[e4], w2[e4]);
    *(v4i*)&sm.Ks[0][kk][c * 16] = v4i{(int)w0[0], (int)w0[1], (int)w0[2], (int)w0[3]};
    *(v4i*)&sm.Ks[1][kk][c * 16] = v4i{(int)w1[0], (int)w1[1], (int)w1[2], (int)w1[3]};
    *(v4i*)&sm.Ks[2][kk][c * 16] = v4i{(int)w2[0], (int)w2[1], (int)w2[2], (int)w2[3]};
    if (want_v) {
      const int kq = u % 16, dq = u / 16;
      uint32_t l[4][3];
#pragma unroll
      for (int m = 0; m < 4; ++m) split3(r.v[t][m], l[m][0], l[m][1], l[m][2]);
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t word = ((l[0][j] >> (8 * d)) & 255) | (((l[1][j] >> (8 * d)) & 255) << 8) |
                                (((l[2][j] >> (8 * d)) & 255) << 16) | (((l[3][j] >> (8 * d)) & 255) << 24);
          *(uint32_t*)&sm.Vt[j][dq * 4 + d][kq * 4] = word;
        }
    }
  }
}

template <int HD>
__device__ __forceinline__ void pre_scores(const PreSmem<HD>& sm, const v4i (&qa)[3][HD / 64], int kb, int64_t (&raw)[4]) {
  const int lane = threadIdx.x & 63;
  v4i acc[5];
#pragma unroll
  for (int w = 0; w < 5; ++w) acc[w] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int kk = 0; kk < HD / 64; ++kk)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const v4i b = *(const v4i*)&sm.Ks[j][kb * 16 + (lane & 15)][kk * 64 + (lane >> 4) * 16];
#pragma unroll
      for (int i = 0; i < 3; ++i) acc[i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa[i][kk], b, acc[i + j], 0, 0, 0);
    }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    int64_t r = 0;
#pragma unroll
    for (int w = 0; w < 5; ++w) r += (int64_t)acc[w][e] << (8 * w);
    raw[e] = r;
  }
}

template <int HD>
__global__ __launch_bounds__(256, HD == 64 ? 2 : 1) void attn_pre_kernel(AttnArgs p) {
  extern __shared__ __align__(16) char smem_raw[];
  PreSmem<HD>& sm = *(PreSmem<HD>*)smem_raw;
  constexpr int KK = HD / 64, DB = HD / 16;
  const int tiles = (p.nq + 63) / 64;
  const int z = blockIdx.x / tiles, q0 = (blockIdx.x % tiles) * 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // A operands: limb i of query q0 + 16 w + (lane & 15), dims kk 64 + (lane >> 4) 16 + [0, 16)
  v4i qa[3][KK];
  {
    const int qr = min(q0 + 16 * w + (lane & 15), p.nq - 1);
    const int32_t* qp = p.q + (int64_t)z * p.sq_tile + (int64_t)qr * p.sq_row;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      uint32_t l[3][4];
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        split3(*(const v4i*)(qp + kk * 64 + (lane >> 4) * 16 + e4 * 4), l[0][e4], l[1][e4], l[2][e4]);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) qa[i][kk] = v4i{(int)l[i][0], (int)l[i][1], (int)l[i][2], (int)l[i][3]};
    }
  }
  // this lane's output rows: 16 w + 4 (lane >> 4) + e
  int64_t qpos[4], shift[4], mx[4];
  int64_t kend = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = q0 + 16 * w + 4 * (lane >> 4) + e;
    const bool ok = r < p.nq;
    qpos[e] = ok ? p.qpos[(z / p.qpos_div) * p.qpos_tile + (int64_t)r * p.qpos_row] : -1;
    shift[e] = ok ? (int64_t)(kFK + 3 - kFZ) - p.sh[z * p.sh_tile + r] : 0;
    mx[e] = kNeg;
    kend = imax(kend, qpos[e] + 1);
  }
  // the block's key range: the largest visible key of its rows (bounded by the cache)
  __shared__ int64_t s_kend;
  if (threadIdx.x == 0) s_kend = 0;
  __syncthreads();
  atomicMax((long long*)&s_kend, (long long)kend);
  __syncthreads();
  const int kb_end = (int)imin(s_kend, (int64_t)p.S);
  const int ntile = (kb_end + 63) / 64;

  // ---- sweep 1: row maxima ----
  PreRegs<HD> kv;
  if (ntile > 0) pre_load<HD>(p, kv, z, 0, kb_end, false);
  for (int t = 0; t < ntile; ++t) {
    __syncthreads();
    pre_store<HD>(sm, kv, false);
    __syncthreads();
    if (t + 1 < ntile) pre_load<HD>(p, kv, z, (t + 1) * 64, kb_end, false);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      int64_t raw[4];
      pre_scores<HD>(sm, qa, kb, raw);
      const int s = t * 64 + kb * 16 + (lane & 15);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (s < kb_end && s <= qpos[e]) mx[e] = imax(mx[e], raw[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) mx[e] = imax(mx[e], __shfl_xor(mx[e], o, 64));

  // ---- sweep 2: weights, den, PV ----
  int64_t den[4] = {0, 0, 0, 0};
  v4i pacc[DB][5];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int ww = 0; ww < 5; ++ww) pacc[d][ww] = v4i{0, 0, 0, 0};
  if (ntile > 0) pre_load<HD>(p, kv, z, 0, kb_end, true);
  for (int t = 0; t < ntile; ++t) {
    __syncthreads();
    pre_store<HD>(sm, kv, true);
    __syncthreads();
    if (t + 1 < ntile) pre_load<HD>(p, kv, z, (t + 1) * 64, kb_end, true);
    // per 16-key block, its 8 table loads are issued before any weight is formed (a load under a per-score
    // branch would wait alone); NKB blocks at a time
    constexpr int NKB = 1;
#pragma unroll
    for (int kb2 = 0; kb2 < 4; kb2 += NKB) {
      WeightAt wa[NKB][4];
      int64_t ta[NKB][4], tb[NKB][4];
#pragma unroll
      for (int h = 0; h < NKB; ++h) {
        int64_t raw[4];
        pre_scores<HD>(sm, qa, kb2 + h, raw);
#pragma unroll
        for (int e = 0; e < 4; ++e) wa[h][e] = weight_at(mx[e] - raw[e], shift[e], p.l2e);
      }
#pragma unroll
      for (int h = 0; h < NKB; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ta[h][e] = p.lut[wa[h][e].idx];
          tb[h][e] = p.lut[wa[h][e].idx + 1];
        }
#pragma unroll
      for (int h = 0; h < NKB; ++h) {
      const int kb = kb2 + h;
      const int s = t * 64 + kb * 16 + (lane & 15);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t w8 = weight_of(wa[h][e], ta[h][e], tb[h][e]);
        const int64_t pw = (s < kb_end && s <= qpos[e]) ? w8 : 0;
        den[e] += pw;
        int32_t x = (int32_t)pw;                         // 0 <= p <= 2^22: three limbs
        const int32_t a0 = limb_lo(x);
        x = (x - a0) >> 8;
        const int32_t a1 = limb_lo(x);
        x = (x - a1) >> 8;
        const int row = 4 * (lane >> 4) + e, col = kb * 16 + (lane & 15);
        sm.Pl[w][0][row][col] = (int8_t)a0;
        sm.Pl[w][1][row][col] = (int8_t)a1;
        sm.Pl[w][2][row][col] = (int8_t)limb_lo(x);
      }
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);                  // this wave's LDS writes are done
    __builtin_amdgcn_wave_barrier();
    v4i pa[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) pa[i] = *(const v4i*)&sm.Pl[w][i][lane & 15][(lane >> 4) * 16];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const v4i b = *(const v4i*)&sm.Vt[j][d * 16 + (lane & 15)][(lane >> 4) * 16];
#pragma unroll
        for (int i = 0; i < 3; ++i) pacc[d][i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pa[i], b, pacc[d][i + j], 0, 0, 0);
      }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) den[e] += __shfl_xor(den[e], o, 64);
  // outputs: lane holds rows 4 (lane >> 4) + e of the wave, dims d 16 + (lane & 15)
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = q0 + 16 * w + 4 * (lane >> 4) + e;
    if (r >= p.nq) continue;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      int64_t v = 0;
#pragma unroll
      for (int ww = 0; ww < 5; ++ww) v += (int64_t)pacc[d][ww][e] << (8 * ww);
      p.num[z * p.snum_tile + (int64_t)r * p.snum_row + d * 16 + (lane & 15)] = v;
    }
    if ((lane & 15) == 0) p.den[z * p.sden_tile + r] = den[e];
  }
}

// ---- fused prefill attention, limb-plane form (contiguous int32 K / V, with a scratch buffer) ----
// pre_split_kernel writes K and V once as int8 limb planes, padded with zeros to Sp (a multiple of 64 keys):
// Kp [Z][3][Sp][HD] (key rows: the QK A operand) and Vp [Z][3][HD][Sp] (dim rows: the PV B operand), the keys of
// every 64-key tile of Vp in MFMA k order: position 16 c + 4 kb + e holds key 16 kb + 4 c + e. That is the order in
// which the transposed QK product leaves the weights in the lanes (below), so the weights go from registers
// straight into the PV A operand.
__device__ __forceinline__ int pre_vpos(int key) {   // tile key -> its Vp position
  return ((key >> 2) & 3) * 16 + ((key >> 4) & 3) * 4 + (key & 3);
}

// The 2^-f table as the main kernel keeps it in LDS: U[i] = floor((2^60 - lut[i]) / 2^29), 32 bits an entry (64 KiB
// for the table instead of the 128 KiB of its int64 entries, so it fits beside the ring). pre_table_block (one block
// per 256 entries) writes it to scratch with one word per block: 1 when its entries can take the short weight rule,
// i.e. 2^59 <= lut[i] <= 2^60, 0 <= U[i + 1] - U[i] < 2^20 and U[i + 1] > 0 (true of the 2^-f table; any other table
// takes the general rule).
constexpr int kTabN = 1 << kExp2Bits;                  // entries [0, kTabN]
constexpr int kTabBlocks = kTabN / 256;
constexpr int kTabPad = kTabN + 4;                     // words of U in scratch and LDS (16-byte multiple)
// Factors of the table in float64: lut[128 h + l] is within 2^10 of F[h] F[129 + l] (F[h] = lut[128 h], F[129 + l] =
// lut[l] / 2^60; three roundings of 2^-53 and the table's own), checked for every entry by pre_table_block.
constexpr int kTabF = 129 + 128;
__device__ __forceinline__ double pre_f(const int64_t* lut, int j) {
  return j < 129 ? (double)lut[j * 128] : ldexp((double)lut[j - 129], -kExp2One);
}
__device__ __forceinline__ uint32_t pre_u(int64_t a) {
  const bool in = a >= (1LL << 59) && a <= (1LL << 60);
  return in ? (uint32_t)(((1LL << 60) - a) >> 29) : 0xffffffffu;
}
__device__ __forceinline__ void pre_table_block(const int64_t* lut, uint32_t* tab, int b) {
  const int i = b * 256 + threadIdx.x;
  const uint32_t u0 = pre_u(lut[i]), u1 = pre_u(lut[i + 1]);
  tab[i] = u0;
  if (i == kTabN - 1) {
#pragma unroll
    for (int j = 0; j < kTabPad - kTabN; ++j) tab[kTabN + j] = u1;
  }
  const double df = pre_f(lut, i >> 7) * pre_f(lut, 129 + (i & 127)) - (double)(lut[i] & ~1023LL);
  const double de = pre_f(lut, (i + 1) >> 7) * pre_f(lut, 129 + ((i + 1) & 127)) - (double)(lut[i + 1] & ~1023LL);
  const bool ok = u0 != 0xffffffffu && u1 != 0xffffffffu && u1 - u0 < (1u << 20) && u1 > 0 && df >= -1024.0 &&
                  df <= 2048.0 && de >= -1024.0 && de <= 2048.0;
  const bool all = __syncthreads_and(ok);
  if (threadIdx.x == 0) tab[kTabPad + b] = all ? 1u : 0u;
}

__global__ __launch_bounds__(256) void pre_split_kernel(AttnArgs p, int8_t* kp, int8_t* vp, uint32_t* tab, int Z, int Sp,
                                                        int HD) {
  if (blockIdx.x < kTabBlocks) {
    pre_table_block(p.lut, tab, blockIdx.x);
    return;
  }
  const int CR = HD / 16;
  const int64_t nk = (int64_t)Z * Sp * CR;          // K units: (z, key, 16-dim chunk)
  const int64_t nv = (int64_t)Z * (Sp / 4) * (HD / 4);   // V units: (z, 4 keys, 4 dims)
  for (int64_t u = (blockIdx.x - kTabBlocks) * 256LL + threadIdx.x; u < nk + nv;
       u += (int64_t)(gridDim.x - kTabBlocks) * 256) {
    if (u < nk) {
      const int c = (int)(u % CR), s = (int)((u / CR) % Sp), z = (int)(u / ((int64_t)CR * Sp));
      uint32_t l[3][4];
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const v4i v = s < p.S ? *(const v4i*)(p.K + (int64_t)z * p.sk_z + (int64_t)s * p.sk_s + c * 16 + e4 * 4)
                              : v4i{0, 0, 0, 0};
        split3(v, l[0][e4], l[1][e4], l[2][e4]);
      }
#pragma unroll
      for (int j = 0; j < 3; ++j)
        *(v4i*)(kp + (((int64_t)z * 3 + j) * Sp + s) * HD + c * 16) =
            v4i{(int)l[j][0], (int)l[j][1], (int)l[j][2], (int)l[j][3]};
    } else {
      const int64_t w = u - nk;
      const int d4 = (int)(w % (HD / 4)), s4 = (int)((w / (HD / 4)) % (Sp / 4)), z = (int)(w / ((int64_t)(HD / 4) * (Sp / 4)));
      uint32_t l[4][3];   // [key m][plane j]: the 4 dims' limbs
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int s = s4 * 4 + m;
        const v4i v = s < p.S ? *(const v4i*)(p.V + (int64_t)z * p.sv_z + (int64_t)s * p.sv_s + d4 * 4) : v4i{0, 0, 0, 0};
        split3(v, l[m][0], l[m][1], l[m][2]);
      }
      const int key0 = (s4 * 4) & 63, tile0 = (s4 * 4) & ~63;
      const int pos = tile0 + pre_vpos(key0);      // the 4 keys stay consecutive
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t word = ((l[0][j] >> (8 * d)) & 255) | (((l[1][j] >> (8 * d)) & 255) << 8) |
                                (((l[2][j] >> (8 * d)) & 255) << 16) | (((l[3][j] >> (8 * d)) & 255) << 24);
          *(uint32_t*)(vp + (((int64_t)z * 3 + j) * HD + d4 * 4 + d) * Sp + pos) = word;
        }
    }
  }
}

// ---- the same attention over the paged cache, for steps of many tokens per sequence ----
// rows_group_kernel sorts the step's token rows by their block-table row (stable) and cuts each sequence's into
// tiles of TT tokens; paged_planes_kernel writes the sequences' cached K and V limbs as the planes above;
// attn_pre2_kernel then runs a (tile, KV head) per block. One block per table row s counts the tokens of smaller rows
// (its start in perm) and its own, then writes them in order. Tile slots [start / TT + s, (start + count) / TT + s + 1)
// belong to sequence s: at least ceil(count / TT) of them, never two sequences' (the spare ones hold 0 tokens).
// Tokens whose row is not in the table (padding) form a last sequence, s = nrow, that sees no key: their outputs are
// 0, and every slot and every entry of perm is written whatever rmap holds.
// A sequence of fewer than kFewTokens tokens (one that decodes beside another's prefill chunk) gets no tile and no
// planes: laying out all its keys and a block over them cost more than its tokens. Its token rows go on a list that
// attn_dec_kernel works off, scores kept (heads of 64, 8 KV heads; every sequence grouped / none / so): a chunk of 512
// and 31 tokens past 4096 keys 465 / 258 / 200 us, 256 and 15 past 4096 313 / 147 / 103, 512 and 63 past 1024 276 / 197
// / 124. The line: 32 sequences of 4 past 4096 433 grouped and 341 not, of 8 451 and 632; 8 sequences of 8 276 and
// 157, of 12 283 and 244. Steps without such sequences pay for the empty list (8 of 32 tokens 23.8 -> 29.0, 8 of 512 the
// same as before with the faster grouping).
constexpr int kFewTokens = 8;
struct RowMap {
  const int32_t* perm;      // [R] token rows, sorted
  const int4* slots;        // [nslot] (start in perm, tokens, table row or nrow, 0)
  int nslot, nrow, M, hkv;
};

// Each wave takes a quarter of the token rows, kRowU loads in flight: bound by their latency (R = 4096: two round trips;
// 8 sequences of 512 tokens: 9.4 us; one wave a sequence with 8 in flight took 17).
constexpr int kRowU = 16;
__device__ __forceinline__ void rows_load(const int64_t* rmap, int i0, int i1, int nrow, int (&r)[kRowU]) {
  int64_t v[kRowU];
#pragma unroll
  for (int u = 0; u < kRowU; ++u) v[u] = rmap[min(i0 + u * 64, i1 - 1)];
#pragma unroll
  for (int u = 0; u < kRowU; ++u)        // past the wave's part: no sequence's
    r[u] = i0 + u * 64 >= i1 ? nrow + 1 : v[u] >= 0 && v[u] < nrow ? (int)v[u] : nrow;
}
__global__ __launch_bounds__(256) void rows_group_kernel(const int64_t* rmap, const int64_t* qpos, int64_t sqpos, int R,
                                                         int M, int nrow, int S, int TT, int nslot, int32_t* perm,
                                                         int4* slots, int32_t* klen, int2* few) {
  __shared__ int s_lt[4], s_eq[4];
  __shared__ int64_t s_kmax[4];
  const int s = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i0 = (int)((int64_t)R * w / 4), i1 = (int)((int64_t)R * (w + 1) / 4);
  const bool held = i1 - i0 <= 64 * kRowU;           // one pass over the part: its rows stay in registers
  int lt = 0, eq = 0, r[kRowU];
  for (int i = i0; i < i1; i += 64 * kRowU) {
    rows_load(rmap, i + lane, i1, nrow, r);
#pragma unroll
    for (int u = 0; u < kRowU; ++u) {
      lt += __popcll(__builtin_amdgcn_ballot_w64(r[u] < s));
      eq += __popcll(__builtin_amdgcn_ballot_w64(r[u] == s));
    }
  }
  if (lane == 0) {
    s_lt[w] = lt;
    s_eq[w] = eq;
  }
  __syncthreads();
  lt = s_lt[0] + s_lt[1] + s_lt[2] + s_lt[3];
  int at = lt;
  for (int u = 0; u < w; ++u) at += s_eq[u];
  int64_t kmax = -1;
  for (int i = i0; eq > 0 && i < i1; i += 64 * kRowU) {
    if (!held) rows_load(rmap, i + lane, i1, nrow, r);
#pragma unroll
    for (int u = 0; u < kRowU; ++u) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(r[u] == s);
      if (r[u] == s) {
        const int64_t row = i + u * 64 + lane;
        perm[at + __popcll(m & ((1ULL << lane) - 1))] = (int)row;
        for (int j = 0; s < nrow && j < M; ++j) kmax = imax(kmax, qpos[row * sqpos + j]);
      }
      at += __popcll(m);
    }
  }
  kmax = wave_max64(kmax);
  if (lane == 0) s_kmax[w] = kmax;
  __syncthreads();
  kmax = imax(imax(s_kmax[0], s_kmax[1]), imax(s_kmax[2], s_kmax[3]));
  eq = s_eq[0] + s_eq[1] + s_eq[2] + s_eq[3];
  const int first = lt / TT + s, next = s < nrow ? (lt + eq) / TT + s + 1 : nslot;
  const bool is_few = s < nrow && eq < kFewTokens;
  for (int j = first + threadIdx.x; j < next; j += 256) {
    const int o = (j - first) * TT;
    slots[j] = int4{lt + o, is_few ? 0 : min(max(eq - o, 0), TT), s, 0};
  }
  if (threadIdx.x == 0 && s < nrow) {
    klen[s] = is_few ? 0 : (int)imin(kmax + 1, S);
    few[s] = int2{lt, is_few ? eq : 0};
  }
}

// Block kTabBlocks of paged_planes_kernel: the token rows of the sequences with few tokens, in table order, after their
// number, and their kernel's counters set to 0.
__device__ void rows_list_block(const int32_t* perm, const int2* few, int nrow, int32_t* list, int32_t* sem) {
  __shared__ int s_at;
  const int lane = threadIdx.x & 63;
  if (threadIdx.x == 0) s_at = 0;
  for (int u = threadIdx.x; u < kDecListBlocks; u += 256) sem[u] = 0;
  __syncthreads();
  for (int s0 = 0; s0 < nrow; s0 += 256) {           // 256 sequences at a time, a lane each; waves in turn
    const int s = s0 + threadIdx.x;
    const int2 f = s < nrow ? few[s] : int2{0, 0};
    int incl = f.y;                                  // counts up to this lane's
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    int base = 0;
    for (int w = 0; w < 4; ++w) {
      if ((int)(threadIdx.x >> 6) == w) {
        base = s_at;
        if (lane == 63) s_at = base + incl;
      }
      __syncthreads();
    }
    for (int j = 0; j < f.y; ++j) list[1 + base + incl - f.y + j] = perm[f.x + j];
  }
  if (threadIdx.x == 0) list[0] = s_at;
}

// Block kTabBlocks + 1 + ((row HKV + h) ntile + tile): 64 keys of one (sequence, KV head). K rows are copied as they
// stand; V goes 4 keys x 4 dims at a time through a byte transpose. Keys past klen are left as they are: no query
// sees them, so their weights are 0.
template <int HD>
__global__ __launch_bounds__(256) void paged_planes_kernel(AttnArgs p, const int32_t* klen, int8_t* kp, int8_t* vp,
                                                           uint32_t* tab, int Sp, int ntile, const int32_t* perm,
                                                           const int2* few, int nrow, int32_t* list) {
  if (blockIdx.x < kTabBlocks) {
    pre_table_block(p.lut, tab, blockIdx.x);
    return;
  }
  if (blockIdx.x == kTabBlocks) {
    rows_list_block(perm, few, nrow, list, p.sem);
    return;
  }
  const int b = blockIdx.x - kTabBlocks - 1, z = b / ntile, k0 = (b - z * ntile) * 64;
  const int row = z / p.hkv, h = z - row * p.hkv;
  const int nk = min(klen[row] - k0, 64);
  if (nk <= 0) return;
  __shared__ int64_t s_off[64];
  if (threadIdx.x < 64) {
    const int s = k0 + min((int)threadIdx.x, nk - 1);
    s_off[threadIdx.x] = (int64_t)p.bt[row * p.sbt + s / p.bs] * p.sc_nb + (int64_t)h * p.sc_h + (int64_t)(s % p.bs) * p.sc_bs;
  }
  __syncthreads();
  constexpr int CH = 3 * HD / 16;
  for (int u = threadIdx.x; u < 64 * CH; u += 256) {
    const int k = u / CH, ch = u - k * CH, j = ch / (HD / 16), cc = ch - j * (HD / 16);
    if (k < nk)
      *(v4i*)(kp + (((int64_t)z * 3 + j) * Sp + k0 + k) * HD + cc * 16) = *(const v4i*)(p.cache + s_off[k] + ch * 16);
  }
  for (int u = threadIdx.x; u < 16 * 3 * (HD / 4); u += 256) {
    const int s4 = u & 15, jd = u >> 4, j = jd / (HD / 4), d4 = jd - j * (HD / 4);
    uint32_t y[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) y[m] = *(const uint32_t*)(p.cache + s_off[s4 * 4 + m] + (3 + j) * HD + d4 * 4);
    const uint32_t a0 = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u), a1 = __builtin_amdgcn_perm(y[1], y[0], 0x07030602u);
    const uint32_t b0 = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u), b1 = __builtin_amdgcn_perm(y[3], y[2], 0x07030602u);
    const uint32_t o[4] = {__builtin_amdgcn_perm(b0, a0, 0x05040100u), __builtin_amdgcn_perm(b0, a0, 0x07060302u),
                           __builtin_amdgcn_perm(b1, a1, 0x05040100u), __builtin_amdgcn_perm(b1, a1, 0x07060302u)};
    int8_t* dst = vp + (((int64_t)z * 3 + j) * HD + d4 * 4) * Sp + k0 + pre_vpos(s4 * 4);
#pragma unroll
    for (int d = 0; d < 4; ++d) *(uint32_t*)(dst + (int64_t)d * Sp) = o[d];
  }
}

// The three signed base-256 limbs of four values 0 <= x <= 2^22, each as one word of four bytes: byte i of x + 0x8080
// is limb i + 128 for i = 0, 1 and limb 2 for i = 2 (the adds' carries are the digits' borrows); the bytes of the
// four words are transposed with seven v_perm_b32.
__device__ __forceinline__ void limb_words(const int32_t (&x)[4], uint32_t& l0, uint32_t& l1, uint32_t& l2) {
  uint32_t y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = (uint32_t)x[e] + 0x8080u;
  const uint32_t a = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u);   // y0.0 y1.0 y0.1 y1.1
  const uint32_t b = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u);
  const uint32_t c = __builtin_amdgcn_perm(y[1], y[0], 0x0c0c0602u);   // y0.2 y1.2 0 0
  l0 = __builtin_amdgcn_perm(b, a, 0x05040100u) ^ 0x80808080u;
  l1 = __builtin_amdgcn_perm(b, a, 0x07060302u) ^ 0x80808080u;
  l2 = __builtin_amdgcn_perm(y[3], y[2], 0x06020c0cu) | c;             // 0 0 y2.2 y3.2
}

template <int HD>
struct Pre2 {
  static constexpr int KK = HD / 64, CR = HD / 16;
  static constexpr int PB = 3 * 64 * HD;             // one operand's three planes of a tile (bytes): a ring slot
  static constexpr int SLOTS = 3;                    // ring: K of tile t, V of tile t, K of tile t + 1, V of t + 1, ...
  static constexpr int KI = PB / 1024;               // 1 KiB instructions per slot
  // Waves that share 16 query rows, and waves of a block: two waves per SIMD (198 and 213 registers). Measured at
  // head_dim 64 (4 x 1024 tokens): 8 waves 198 us, 12 waves (168 registers, spills) 305, 12 waves of pairs (156
  // registers) 221; at head_dim 128 (1337 tokens): 8 waves of pairs 157 us, 4 single waves (one per SIMD) 234.
  static constexpr int SW = HD == 64 ? 1 : 2;
  static constexpr int NW = 8;
  static constexpr int LP = (KI + NW - 1) / NW;      // instructions per issuing wave and slot
  static constexpr int KB = 4 / SW, DB = HD / 16 / SW;   // 16-key blocks and 16-dim blocks of a wave
  static constexpr int QR = 16 * NW / SW;            // query rows per block
  static constexpr int XB = SW == 1 ? 0 : 3 * 16 * QR * 4;   // p exchange between the waves of a pair (bytes)
  // LDS: the table first (its reads then need no address add), the ring, the exchange, the table's factors
  static constexpr int RO = 4 * kTabPad, XO = RO + SLOTS * PB, FO = XO + XB;
  static constexpr size_t LDS = FO + 8 * kTabF;
  static_assert(RO % 16 == 0 && FO % 8 == 0, "LDS alignment");
  static_assert(KI % LP == 0, "a wave issues LP instructions or none");
};

__device__ __forceinline__ int pre_swzk(int k, int HD) { return HD == 64 ? (k >> 2) & 3 : (k >> 1) & 7; }
__device__ __forceinline__ int pre_swzv(int d) { return (d >> 2) & 3; }

// An empty use: the value is formed where it stands (no branch around its computation).
__device__ __forceinline__ void pin_v(int32_t& x) { asm("" : "+v"(x)); }
__device__ __forceinline__ void pin_v(uint32_t& x) { asm("" : "+v"(x)); }

// attn_pre2_kernel: SW waves own 16 consecutive query rows of one group z (SW = 2: each forms the scores and weights
// of half of a tile's keys and p V of half of the dims, the weights' limbs meet in LDS; accumulators per wave halve).
// The 64-key tiles of the limb planes stream through a 3-slot LDS ring filled by buffer_load ... lds
// (1 KiB per wave instruction; 16-byte chunks XOR-swizzled by row so the 16 rows an MFMA operand read touches fall
// in distinct bank groups). QK is computed transposed: A = K limb plane j (16 keys x 64 dims), B = limb i of the
// 16 queries (registers), so lane l receives query l & 15's scores for keys 16 kb + 4 (l >> 4) + e; the
// nine limb products accumulate by weight i + j in five int32 sets, joined in int64. Sweep 1 keeps the per-query
// maxima. Sweep 2 forms the weights in the same lanes; their three limbs, packed in key order 4 kb + e, are the
// PV A operand as they stand (16 queries x 64 keys in Vp's order), and B = V limb plane j (64 keys x 16 dims):
// five int32 sets per 16-dim block (exact while S 3 2^14 < 2^31), joined in int64 at the end. The next key block's
// MFMAs are issued before a block's weights are formed.
//
// The short weight rule (`fast`: no query of the wave has a negative exponent shift, 0 <= l2e < 2^31, and the table
// passed pre_table_block's check). With U the LDS table, y = (2^60 - v) / 2^29 of the interpolated value v lies in [Uc
// - 2^-30, Uc + 2) for Uc = U0 + ((U1 - U0) rr >> 12): both entries (fractions at most 1 - 2^-29) and the product are
// floors, v's own rounding is 2^-30 of the unit. The weight rshc(v, 38 + n) = floor((2^31 + 2^(8+n) - y) / 2^(9+n))
// for n <= 22 is then 2^(22-n) + (T >> (9+n)), T = 2^(8+n) - Uc, whatever y is, unless T mod 2^(9+n) <= 1: such a
// score (2 in 2^(9+n)) takes its value from the table's float64 factors, and from the int64 table where even that is
// within 2^-25 of a rounding boundary. From n = 23 the weight is 0, v being below 2^60, except at the single position
// n = 23, f = 0 (Uc = 0: T = 2^31 marks it).
// Before, every score gathered its 16-byte table pair through L1: with attention scores of unit spread that was 140 of
// 341 us (4 x 1024 tokens, 32 / 8 heads of 64), the lanes' lines missing the 32 KiB L1. Now 198 us (1337 tokens, heads
// of 128: 233 -> 157): bound by the integer work per score (54 VALU instructions over both sweeps), with sweep 1 about
// 55 us of it. The second-step values come from LDS too because one wave's memory round trip holds its block at the
// tile's barrier (238 us).
// ROWS: the paged form. Block (slot, KV head h); the block's query i is query i % M of the slot's token i / M.
template <int HD, bool ROWS>
__global__ __launch_bounds__(64 * Pre2<HD>::NW, 1) void attn_pre2_kernel(AttnArgs p, const int8_t* planes, int Z,
                                                                         int Sp, const uint32_t* tab, RowMap rm) {
  using C = Pre2<HD>;
  constexpr int QR = C::QR, SW = C::SW;
  constexpr int KK = C::KK, DB = C::DB, SL = C::SLOTS;
  extern __shared__ __align__(16) char smem[];
  uint32_t* U = (uint32_t*)smem;
  char* ring = smem + C::RO;
  __shared__ int s_kend;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kl = lane & 15, c = lane >> 4;
  const int wr = w / SW, wp = w % SW;                // row group, part of it
  // the group z of the planes, and where query i of the block lives: (token row, query) group g, row r
  int z, q0 = 0, h = 0;
  int4 slot = {};
  if constexpr (ROWS) {
    slot = rm.slots[rm.nslot - 1 - (int)(blockIdx.x / rm.hkv)];            // late (long) tiles of a sequence first
    if (slot.y == 0) return;                         // the whole block: a spare slot
    h = blockIdx.x % rm.hkv;
    z = slot.z * rm.hkv + h;
  } else {
    const int tiles = (p.nq + QR - 1) / QR;
    z = blockIdx.x % Z;
    q0 = (tiles - 1 - blockIdx.x / Z) * QR;          // late (long) row tiles first
  }
  auto locate = [&](int i, int64_t& g, int& r) {     // false: no such query (g, r then name a readable one)
    if constexpr (ROWS) {
      const int tok = i / rm.M;
      r = i - tok * rm.M;
      g = (int64_t)rm.perm[slot.x + min(tok, slot.y - 1)] * rm.hkv + h;
      return tok < slot.y;
    } else {
      r = min(q0 + i, p.nq - 1);
      g = z;
      return q0 + i < p.nq;
    }
  };
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(planes), (short)0, kBufRange, 0x00020000);
  const int64_t vbase = (int64_t)Z * 3 * Sp * HD;

  // the lane's query (B operand rows) and its position / exponent
  int64_t qg;
  int qr;
  const bool live = locate(16 * wr + kl, qg, qr), keys = !ROWS || slot.z < rm.nrow;   // keys: the query's row has some
  v4i qb[3][KK];
  {
    const int32_t* qp = p.q + qg * p.sq_tile + (int64_t)qr * p.sq_row;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      uint32_t l[3][4];
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) split3(*(const v4i*)(qp + kk * 64 + c * 16 + e4 * 4), l[0][e4], l[1][e4], l[2][e4]);
#pragma unroll
      for (int i = 0; i < 3; ++i) qb[i][kk] = v4i{(int)l[i][0], (int)l[i][1], (int)l[i][2], (int)l[i][3]};
    }
  }
  // (positions past S - 1 see every key, negative ones, whatever their 64 bits, none: the clamp changes neither)
  const int my_qpos =
      live && keys ? (int)imax(imin(p.qpos[(qg / p.qpos_div) * p.qpos_tile + (int64_t)qr * p.qpos_row], (int64_t)p.S), -1)
                   : -1;
  const int64_t shift = live ? (int64_t)(kFK + 3 - kFZ) - p.sh[qg * p.sh_tile + qr] : 0;
  if (threadIdx.x == 0) s_kend = 0;
  __syncthreads();
  const int wmax_qpos = (int)wave_max64(my_qpos);    // the rows' largest position
  const int wmin_qpos = (int)-wave_max64(-(int64_t)my_qpos);      // and smallest
  if (lane == 0) atomicMax(&s_kend, wmax_qpos + 1);
  __syncthreads();
  const int kend = min(s_kend, p.S);                 // keys [0, kend) are visible to some row of the block
  const int ntile = (kend + 63) / 64;

  // DMA offsets of the wave's instructions of a K and of a V slot at tile 0 (a tile further: 64 HD and 64 bytes)
  int offk[C::LP], offv[C::LP];
  const bool issuer = w * C::LP < C::KI;
#pragma unroll
  for (int i = 0; i < C::LP; ++i) {
    const int n = min(w * C::LP + i, C::KI - 1), j = n / (C::KI / 3), o = (n % (C::KI / 3)) * 1024 + lane * 16;
    const int k = o / HD, kc = ((o % HD) / 16) ^ pre_swzk(k, HD);
    offk[i] = (int)((((int64_t)z * 3 + j) * Sp + k) * HD + kc * 16);
    const int d = o / 64, vc = ((o % 64) / 16) ^ pre_swzv(d);
    offv[i] = (int)(vbase + (((int64_t)z * 3 + j) * HD + d) * Sp + vc * 16);
  }
  auto issue = [&](const int (&off)[C::LP], int step, int slot) {
    if (!issuer) return;
#pragma unroll
    for (int i = 0; i < C::LP; ++i) buf_lds16(rs, ring + slot * C::PB + (w * C::LP + i) * 1024, off[i] + step, 0);
  };
  // the nine limb products of 16-key block kb of the staged tile with the lane's query: keys 16 kb + 4 c + e
  const int ksw = pre_swzk(kl, HD);                  // (of key 16 kb + kl: the same for every kb)
  auto qk = [&](const int8_t* kbase, int kb, v4i (&acc)[5]) {
#pragma unroll
    for (int u = 0; u < 5; ++u) acc[u] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const v4i a = *(const v4i*)(kbase + j * 64 * HD + (kb * 16 + kl) * HD + (((kk * 4 + c) ^ ksw) * 16));
#pragma unroll
        for (int i = 0; i < 3; ++i) acc[i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, qb[i][kk], acc[i + j], 0, 0, 0);
      }
  };
  // |acc| <= 64 KK 2^14 = 2^(20 + KK - 1): the pairs acc0 + 2^8 acc1 and acc2 + 2^8 acc3 are exact in int32; the
  // second joins by one 32 x 32 + 64-bit multiply-add (k64k: 2^16 the compiler cannot see)
  int32_t k64k = 65536;
  asm("" : "+s"(k64k));
  auto join = [&](const v4i (&acc)[5], int64_t (&raw)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int32_t lo = acc[0][e] + (acc[1][e] << 8), mid = acc[2][e] + (acc[3][e] << 8);
      const uint64_t base = ((uint64_t)(uint32_t)(acc[4][e] + (lo >> 31)) << 32) | (uint32_t)lo;
      raw[e] = (int64_t)mid * k64k + (int64_t)base;
    }
  };

  // ---- sweep 1: the lane's query maximum over its keys ----
  int64_t mx = kNeg;
  if (ntile > 0) issue(offk, 0, 0);
  if (ntile > 1) issue(offk, 64 * HD, 1);
  // the weight table into LDS behind the first tiles: sweep 2 reads it
  {
    const auto rt = buf_rsrc(tab);
    constexpr int TI = kTabN * 4 / 1024;             // 64 instructions; the last words follow by plain stores
    for (int i = w; i < TI; i += C::NW) buf_lds16(rt, (char*)U + i * 1024, i * 1024 + lane * 16, 0);
    if (threadIdx.x < kTabPad - kTabN) U[kTabN + threadIdx.x] = tab[kTabN + threadIdx.x];
  }
  double* F = (double*)(smem + C::FO);
  for (int i = threadIdx.x; i < kTabF; i += 64 * C::NW) F[i] = pre_f(p.lut, i);
  const bool tab_ok = __builtin_amdgcn_ballot_w64(tab[kTabPad + lane] == 0) == 0;
  static_assert(kTabBlocks == 64, "one table check word per lane");
  for (int t = 0, sl = 0; t < ntile; ++t) {
    if (t == 0 || t + 1 >= ntile) ring_barrier<0>();
    else ring_barrier<C::LP>();
    if (t + 2 < ntile) issue(offk, (t + 2) * 64 * HD, sl == 0 ? 2 : sl - 1);
    const int8_t* kbase = (const int8_t*)ring + sl * C::PB;
    sl = sl == 2 ? 0 : sl + 1;
    auto scan = [&](auto full_t) {
#pragma unroll
      for (int i = 0; i < C::KB; ++i) {
        const int kb = wp * C::KB + i;
        v4i acc[5];
        int64_t raw[4];
        qk(kbase, kb, acc);
        join(acc, raw);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (decltype(full_t)::value || t * 64 + kb * 16 + 4 * c + e <= my_qpos) mx = imax(mx, raw[e]);
      }
    };
    if (t * 64 + 63 <= wmin_qpos) scan(std::true_type{});     // wave-uniform: every key is visible to every row
    else if (t * 64 <= wmax_qpos) scan(std::false_type{});    // some key is visible to some row
  }
  mx = imax(mx, __shfl_xor(mx, 16, 64));
  mx = imax(mx, __shfl_xor(mx, 32, 64));
  ring_barrier<0>();                                 // every wave is done with the ring
  if constexpr (SW == 2) {                           // the pair's maxima meet in slot 2 (free until K of tile 1)
    int64_t* xm = (int64_t*)(ring + 2 * C::PB);
    if (lane < 16) xm[w * 16 + lane] = mx;
    ring_barrier<0>();
    mx = imax(mx, xm[(w ^ 1) * 16 + kl]);
  }

  // ---- sweep 2: weights, den, p V ----
  const bool fast = tab_ok && __builtin_amdgcn_ballot_w64(shift < 0) == 0 && p.l2e >= 0 && p.l2e < (1LL << 31);
  int64_t den = 0;
  v4i pacc[DB][5];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int u = 0; u < 5; ++u) pacc[d][u] = v4i{0, 0, 0, 0};
  if (ntile > 0) {
    issue(offk, 0, 0);
    issue(offv, 0, 1);
  }
  // fast: zf = rshc(mx - raw, s) = (cz - raw) >> s with cz = mx + 2^(s - 1) (wrapping, as rshc's add), s clamped
  // to 62 as rshc clamps it
  const int s62 = (int)imin(imax(shift, 0), 62);
  const int64_t cz = add_wrap(mx, s62 > 0 ? (1LL << (s62 - 1)) : 0);
  // the general rule: four weights, or one
  auto weights_gen = [&](const int64_t (&raw)[4], int32_t (&x)[4]) {
    WeightAt wa[4];
    int64_t ta[4], tb[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      wa[e] = weight_at(mx - raw[e], shift, p.l2e);
      ta[e] = p.lut[wa[e].idx];
      tb[e] = p.lut[wa[e].idx + 1];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = (int32_t)weight_of(wa[e], ta[e], tb[e]);
  };
  auto weight_gen = [&](int64_t raw) { return (int32_t)attn_weight(mx - raw, shift, p.lut, p.l2e); };
  auto weights_fast = [&](const int64_t (&raw)[4], int32_t (&x)[4]) {
    uint32_t f[4], ph[4], u0[4], u1[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint64_t zf = (uint64_t)((cz - raw[e]) >> s62);
      zf = zf < (48ULL << kFZ) ? zf : (48ULL << kFZ);      // hidden keys (negative) clamp too: inside the table
      const uint64_t prod = (uint64_t)(uint32_t)zf * (uint64_t)(uint32_t)p.l2e + (1ULL << 27);
      // t = prod >> 28: n = t >> 26 = prod >> 54 and f = t mod 2^26 from the product's two words
      ph[e] = (uint32_t)(prod >> 32);
      f[e] = __builtin_amdgcn_alignbit(ph[e], (uint32_t)prod, 28);        // t mod 2^32
      pin_v(ph[e]);
      const uint32_t* u = (const uint32_t*)((const char*)U + ((ph[e] >> 6) & (4 * kTabN - 4)));
      u0[e] = u[0];
      u1[e] = u[1];
    }
    bool amb[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t n = ph[e] >> 22;
      const uint32_t uc = u0[e] + __umulhi(u1[e] - u0[e], f[e] << 20);
      const uint32_t sb = (n < 22u ? n : 22u) + 9;         // n > 22: the weight is 0, T only marks the exception
      const int32_t T = (int32_t)((256u << (n & 31)) - uc);
      int32_t wf = (int32_t)(0x400000u >> (n & 31)) + (T >> sb);
      pin_v(wf);
      x[e] = n > 22u ? 0 : wf;
      amb[e] = __builtin_amdgcn_ubfe((uint32_t)T, 0, sb) < 2u;
    }
    if (__builtin_amdgcn_ballot_w64(amb[0] | amb[1] | amb[2] | amb[3]) != 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (__builtin_amdgcn_ballot_w64(amb[e]) != 0) {
          // the value from the table's float64 factors: v within 2^12, so v 2^-(38+n) + 1/2 within 2^-26 decides the
          // weight unless it lies that close to an integer (then the int64 table itself)
          const uint32_t i0 = (f[e] >> 12) & (kTabN - 1), i1 = i0 + 1;
          const double a = F[i0 >> 7] * F[129 + (i0 & 127)], b = F[i1 >> 7] * F[129 + (i1 & 127)];
          const double v = a + (b - a) * ((double)(int32_t)(f[e] & 4095u) * (1.0 / 4096.0));
          const double tt = ldexp(v, -(kExp2One - kFP) - (int)(ph[e] >> 22)) + 0.5;
          const int32_t wi = (int32_t)tt;
          const double fr = tt - (double)wi;
          x[e] = amb[e] ? wi : x[e];
          if (__builtin_amdgcn_ballot_w64(amb[e] && (fr < 0x1p-25 || fr > 1.0 - 0x1p-25)) != 0)
            x[e] = amb[e] ? weight_gen(raw[e]) : x[e];
        }
    }
  };
  auto sweep2 = [&](auto fast_t) {
    constexpr bool kFast = decltype(fast_t)::value;
    uint32_t* xp = (uint32_t*)(smem + C::XO) + wr * (3 * 16 * 16);   // the pair's p limbs
    int ks = 0;                                      // slot of K of this tile; V's is the next, K's of t + 1 the third
    for (int t = 0; t < ntile; ++t) {
      const int vs = ks == 2 ? 0 : ks + 1, ns = vs == 2 ? 0 : vs + 1;
      // K of this tile is in and every wave is done with V of the tile before
      ring_barrier<C::LP>();
      if (t + 1 < ntile) issue(offk, (t + 1) * 64 * HD, ns);
      const int8_t* kbase = (const int8_t*)ring + ks * C::PB;
      const int8_t* vbs = (const int8_t*)ring + vs * C::PB;
      const bool some = t * 64 <= wmax_qpos;         // wave-uniform
      const bool full = t * 64 + 63 <= wmin_qpos;    // wave-uniform: every key of the tile is visible to every query
      v4i pa[3] = {v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}};
      if (some) {
        int32_t dt = 0;                              // the tile's weight sum: <= 64 2^22, exact in int32
        uint32_t pw[3][C::KB];
        v4i acc[2][5];
        qk(kbase, wp * C::KB, acc[0]);
#pragma unroll
        for (int i = 0; i < C::KB; ++i) {
          const int kb = wp * C::KB + i;
          int64_t raw[4];
          int32_t x[4];
          if (i + 1 < C::KB) qk(kbase, kb + 1, acc[(i + 1) & 1]);
          join(acc[i & 1], raw);
          if constexpr (kFast) weights_fast(raw, x);
          else weights_gen(raw, x);
          if (!full) {
            const int key0 = t * 64 + kb * 16 + 4 * c;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = key0 + e <= my_qpos ? x[e] : 0;
          }
          dt += x[0] + x[1];
          dt += x[2] + x[3];
          limb_words(x, pw[0][i], pw[1][i], pw[2][i]);
        }
        den += dt;
#pragma unroll
        for (int l = 0; l < 3; ++l)
          if constexpr (SW == 1) {
            pa[l] = v4i{(int)pw[l][0], (int)pw[l][C::KB - 3], (int)pw[l][C::KB - 2], (int)pw[l][C::KB - 1]};
          } else {
            // 16 bytes per (limb, query, chunk): word kb of lane (query kl, chunk c)
            *(uint2*)&xp[((l * 16 + kl) * 4 + (c ^ ((kl >> 2) & 3))) * 4 + wp * 2] = uint2{pw[l][0], pw[l][1]};
          }
      }
      // V of this tile is in and every wave is done with K of this tile
      if (t + 1 < ntile) ring_barrier<C::LP>();
      else ring_barrier<0>();
      if (t + 1 < ntile) issue(offv, (t + 1) * 64, ks);
      ks = ns;
      if (some) {
        if constexpr (SW == 2) {
#pragma unroll
          for (int l = 0; l < 3; ++l) pa[l] = *(const v4i*)&xp[((l * 16 + kl) * 4 + (c ^ ((kl >> 2) & 3))) * 4];
        }
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          const int row = (wp * DB + d) * 16 + kl;
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const v4i b = *(const v4i*)(vbs + j * HD * 64 + row * 64 + ((c ^ pre_swzv(row)) * 16));
#pragma unroll
            for (int i = 0; i < 3; ++i) pacc[d][i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pa[i], b, pacc[d][i + j], 0, 0, 0);
          }
        }
      }
    }
  };
  if (fast)
    sweep2(std::true_type{});
  else
    sweep2(std::false_type{});
  den += __shfl_xor(den, 16, 64);
  den += __shfl_xor(den, 32, 64);
  if constexpr (SW == 2) {                           // the pair's weight sums (the ring is free: after every wave's last read)
    int64_t* xd = (int64_t*)ring;
    ring_barrier<0>();
    if (lane < 16) xd[w * 16 + lane] = den;
    ring_barrier<0>();
    den += xd[(w ^ 1) * 16 + kl];
  }
  // outputs: lane holds queries 4 c + e of the rows, dims 16 d + kl
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int qw = 4 * c + e;
    const int64_t dq = __shfl(den, qw, 64);
    int64_t g;
    int r;
    if (!locate(16 * wr + qw, g, r)) continue;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      int64_t v = 0;
#pragma unroll
      for (int u = 0; u < 5; ++u) v += (int64_t)pacc[d][u][e] << (8 * u);
      p.num[g * p.snum_tile + (int64_t)r * p.snum_row + (wp * DB + d) * 16 + kl] = v;
    }
    if (kl == 0 && wp == 0) p.den[g * p.sden_tile + r] = dq;
  }
}

// ---- KV store into the limb-plane cache (tri_paged.store, src/bitexact/vllm_plugin/tri_paged.py:311-335) ----
template <typename T>
__global__ __launch_bounds__(128) void kv_store_kernel(int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs,
                                                       const int64_t* slot, const T* k, int64_t skn, int64_t skh,
                                                       const T* v, int64_t svn, int64_t svh, int HD, int bs) {
  const int64_t n = blockIdx.x, h = blockIdx.y;
  const int64_t sl = slot[n];
  if (sl < 0) return;                                  // dummy / padded tokens carry slot -1
  int8_t* base = cache + (sl / bs) * sc_nb + h * sc_h + (sl % bs) * sc_bs;
  for (int d = threadIdx.x; d < HD; d += blockDim.x) {
    int32_t kr = (int32_t)k[n * skn + h * skh + d], vr = (int32_t)v[n * svn + h * svh + d];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int32_t k0 = limb_lo(kr), v0 = limb_lo(vr);
      base[i * HD + d] = (int8_t)k0;
      base[(3 + i) * HD + d] = (int8_t)v0;
      kr = (kr - k0) >> 8;
      vr = (vr - v0) >> 8;
    }
  }
}

}  // namespace bx

using namespace bx;

// ======================================== C ABI ========================================

static void allow_lds_attn(const void* k, size_t lds) {
  if (lds > 64 * 1024) hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

template <int QT, int HD, bool PAGED>
static int launch_attn(AttnArgs& p, int groups, hipStream_t st) {
  const int tiles = (p.nq + QT - 1) / QT;
  const size_t lds = sizeof(AttnSmem<QT, HD>);
  dim3 grid(groups * tiles, p.nsplit);
  if (lds > 64 * 1024) {
    hipFuncSetAttribute((const void*)attn_kernel<QT, HD, PAGED, 0>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipFuncSetAttribute((const void*)attn_kernel<QT, HD, PAGED, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  }
  if (p.nsplit > 1) {
    attn_kernel<QT, HD, PAGED, 0><<<grid, 256, lds, st>>>(p);
    if (int rc = check_launch("attn_kernel(max)")) return rc;
  }
  attn_kernel<QT, HD, PAGED, 1><<<grid, 256, lds, st>>>(p);
  return check_launch("attn_kernel");
}

constexpr int kDecRawKeys = 2048;               // single-launch score cache: 4 x 2048 x 8 B of LDS
constexpr int kDecOneKeys = 256 * 64;           // kept scores: keys x head_dim of a tile that is one block's

template <int HD>
static int launch_dec(AttnArgs& p, int groups, int64_t max_keys, hipStream_t st) {
  const int tiles = (p.nq + 3) / 4;
  dim3 grid(groups * tiles, p.nsplit);
  const int64_t chunk = ((max_keys + p.nsplit - 1) / p.nsplit + 63) / 64 * 64;   // keys per split, at most
  if (p.raw == nullptr && p.nsplit > 1 && chunk <= 64 * kDecWaves && (int64_t)grid.x * grid.y <= kDecExchBlocks) {
    // BX_ATTN_EXCH_TICKS (tests): a shorter wait, down to 0, where blocks compute the maxima they have not seen
    const char* et = getenv("BX_ATTN_EXCH_TICKS");
    p.exch_ticks = et ? (uint64_t)strtoull(et, nullptr, 10) : kDecExchTicks;
    if (chunk <= 32 * kDecWaves) attn_dec_exch_kernel<HD, 2><<<grid, kDecWaves * 64, 0, st>>>(p);
    else attn_dec_exch_kernel<HD, 4><<<grid, kDecWaves * 64, 0, st>>>(p);
    return check_launch("attn_dec_exch_kernel");
  }
  if (p.raw != nullptr) {
    p.S = (int)max_keys;
    p.one_keys = kDecOneKeys / HD;
    attn_dec_kernel<HD, 0, true><<<grid, kDecWaves * 64, 0, st>>>(p);
    if (int rc = check_launch("attn_dec_kernel(scores)")) return rc;
    attn_dec_kernel<HD, 1, true><<<grid, kDecWaves * 64, 0, st>>>(p);
    return check_launch("attn_dec_kernel");
  }
  if (p.nsplit > 1) {
    attn_dec_kernel<HD, 0, false><<<grid, kDecWaves * 64, 0, st>>>(p);
    if (int rc = check_launch("attn_dec_kernel(max)")) return rc;
    attn_dec_kernel<HD, 1, false><<<grid, kDecWaves * 64, 0, st>>>(p);
    return check_launch("attn_dec_kernel");
  }
  if (max_keys <= kDecRawKeys) {
    p.S = (int)((max_keys + 15) / 16 * 16);
    const size_t lds = (size_t)4 * p.S * 8 + ((size_t)p.S / p.bs + 2) * 4;   // scores + block-table entries
    hipFuncSetAttribute((const void*)attn_dec_raw_kernel<HD>, hipFuncAttributeMaxDynamicSharedMemorySize,
                        (int)(4 * kDecRawKeys * 8 + (kDecRawKeys + 2) * 4));
    attn_dec_raw_kernel<HD><<<grid, kDecWaves * 64, lds, st>>>(p, RopeArgs{}, AoArgs{});
    return check_launch("attn_dec_raw_kernel");
  }
  attn_dec_kernel<HD, 1, false><<<grid, kDecWaves * 64, 0, st>>>(p);
  return check_launch("attn_dec_kernel");
}

// split-KV workspace: mx [Gq] + num [Gq, HD] + den [Gq] + counters [tiles]; zero-filled = idle
static int64_t attn_ws_bytes(int64_t gq, int64_t tiles, int HD) { return gq * 8 * (2 + HD) + tiles * 4 + 256; }

static void bind_attn_ws(AttnArgs& p, void* ws, int64_t gq, int HD) {
  char* b = (char*)ws;
  p.mx_ws = (int64_t*)b;
  p.num_ws = (int64_t*)(b + gq * 8);
  p.den_ws = (int64_t*)(b + gq * 8 * (1 + HD));
  p.sem = (int32_t*)(b + gq * 8 * (2 + HD));
}

static int64_t dec_split_cap(int64_t T) { return std::max<int64_t>(1, std::min<int64_t>(kDecMaxSplit, kDecWsSplitBudget / std::max<int64_t>(T, 1))); }

extern "C" int64_t bx_attn_paged_workspace(int32_t R, int32_t HKV, int32_t M, int32_t HD) {
  const int64_t T = (int64_t)R * HKV * ((M + 3) / 4);                                  // query tiles
  return dec_ws_bytes(T, dec_split_cap(T), HD);
}

// The kept-scores form's scratch (`tmp` of the *_scores entries): every (tile, key, query) score
extern "C" int64_t bx_attn_paged_scores_scratch(int32_t R, int32_t HKV, int32_t M, int32_t keys) {
  if (R <= 0 || HKV <= 0 || M <= 0 || keys <= 0) return 0;
  return (int64_t)R * HKV * ((M + 3) / 4) * keys * 32;
}

static int bind_scores(AttnArgs& p, int64_t T, int64_t keys, void* tmp, int64_t tmp_bytes) {
  BX_REQUIRE(p.nsplit > 1, "the kept-scores form needs nsplit > 1");
  BX_REQUIRE(tmp_bytes >= T * keys * 32 && ((uintptr_t)tmp & 7) == 0, "scratch too small (%lld < %lld)",
             (long long)tmp_bytes, (long long)(T * keys * 32));
  p.raw = (int64_t*)tmp;
  return BX_OK;
}

static int exact_paged(const int32_t* q, const int64_t* sh, const int64_t* qpos, int64_t sqpos_r,
                       const int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs,
                       const int32_t* bt, int64_t sbt, int32_t nblk, const int64_t* rmap, const int64_t* lut,
                       int64_t l2e, int64_t* num, int64_t* den, int32_t R, int32_t HKV, int32_t M,
                       int32_t HD, int32_t nsplit, void* ws, int64_t ws_bytes, void* tmp, int64_t tmp_bytes,
                       bx_stream_t stream) {
  BX_REQUIRE(R >= 0 && HKV > 0 && M >= 1 && M <= 4, "need 1 <= M <= 4 queries per (row, KV head)");
  BX_REQUIRE(HD == 64 || HD == 128, "head_dim must be 64 or 128");
  BX_REQUIRE((int64_t)nblk * bs < 43690, "keys per row must stay below 43690");
  BX_REQUIRE(nsplit >= 1 && nsplit <= 64, "nsplit in [1, 64]");
  BX_REQUIRE(sc_bs >= 6 * HD && sc_nb % 16 == 0 && sc_h % 16 == 0 && sc_bs % 16 == 0 && ((uintptr_t)cache & 15) == 0,
             "cache rows must hold the 6 HD limb bytes, 16-byte aligned");
  BX_REQUIRE(q && sh && qpos && bt && rmap && lut && num && den, "null pointer");
  if (R == 0) return BX_OK;
  AttnArgs p = {};
  p.q = q; p.sq_tile = (int64_t)M * HD; p.sq_row = HD;
  p.sh = sh; p.sh_tile = M;
  p.qpos = qpos; p.qpos_tile = sqpos_r; p.qpos_row = 1; p.qpos_div = HKV; p.nq = M;
  p.cache = cache; p.sc_nb = sc_nb; p.sc_h = sc_h; p.sc_bs = sc_bs; p.bt = bt; p.sbt = sbt; p.rmap = rmap;
  p.bs = bs; p.hkv = HKV; p.nblk = nblk;
  p.lut = lut; p.l2e = l2e;
  p.num = num; p.den = den; p.snum_tile = (int64_t)M * HD; p.snum_row = HD; p.sden_tile = M;
  p.nsplit = nsplit;
  if (nsplit > 1) {
    const int64_t T = (int64_t)R * HKV * ((M + 3) / 4);
    const int64_t need = dec_ws_bytes(T, nsplit, HD);
    BX_REQUIRE(ws != nullptr && ws_bytes >= need, "workspace too small for %d splits (%lld < %lld)", nsplit,
               (long long)ws_bytes, (long long)need);
    BX_REQUIRE(((uintptr_t)ws & 7) == 0, "workspace must be 8-byte aligned");
    p.mx_ws = (int64_t*)ws;
  }
  const int64_t max_keys = (int64_t)nblk * bs;     // qpos < nblk bs: the block table's reach
  if (tmp != nullptr)
    if (int rc = bind_scores(p, (int64_t)R * HKV * ((M + 3) / 4), max_keys, tmp, tmp_bytes)) return rc;
  return HD == 64 ? launch_dec<64>(p, R * HKV, max_keys, (hipStream_t)stream)
                  : launch_dec<128>(p, R * HKV, max_keys, (hipStream_t)stream);
}

extern "C" int bx_exact_attn_paged(const int32_t* q, const int64_t* sh, const int64_t* qpos, int64_t sqpos_r,
                                   const int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs,
                                   const int32_t* bt, int64_t sbt, int32_t nblk, const int64_t* rmap, const int64_t* lut,
                                   int64_t l2e, int64_t* num, int64_t* den, int32_t R, int32_t HKV, int32_t M,
                                   int32_t HD, int32_t nsplit, void* ws, int64_t ws_bytes, bx_stream_t stream) {
  return exact_paged(q, sh, qpos, sqpos_r, cache, sc_nb, sc_h, sc_bs, bs, bt, sbt, nblk, rmap, lut, l2e, num, den, R, HKV,
                     M, HD, nsplit, ws, ws_bytes, nullptr, 0, stream);
}

extern "C" int bx_exact_attn_paged_scores(const int32_t* q, const int64_t* sh, const int64_t* qpos, int64_t sqpos_r,
                                          const int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs,
                                          const int32_t* bt, int64_t sbt, int32_t nblk, const int64_t* rmap,
                                          const int64_t* lut, int64_t l2e, int64_t* num, int64_t* den, int32_t R,
                                          int32_t HKV, int32_t M, int32_t HD, int32_t nsplit, void* ws,
                                          int64_t ws_bytes, void* tmp, int64_t tmp_bytes, bx_stream_t stream) {
  BX_REQUIRE(tmp != nullptr || R == 0, "null scratch");
  return exact_paged(q, sh, qpos, sqpos_r, cache, sc_nb, sc_h, sc_bs, bs, bt, sbt, nblk, rmap, lut, l2e, num, den, R, HKV,
                     M, HD, nsplit, ws, ws_bytes, tmp, tmp_bytes, stream);
}

static int attn_rope_common(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spos, const int64_t* cos,
                            const int64_t* sin, int32_t npos, int32_t H, int32_t FR, int32_t FT, int32_t FK, int32_t FV,
                            int32_t FZ, const int64_t* slot, int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs,
                            int32_t bs, const int32_t* bt, int64_t sbt, int32_t nblk, const int64_t* rmap,
                            const int64_t* lut, int64_t l2e, int64_t* num, int64_t* den, int32_t R, int32_t HKV,
                            int32_t HD, int32_t* err, const AoArgs* ao, hipStream_t st) {
  BX_REQUIRE(R >= 0 && HKV > 0 && H % HKV == 0 && H / HKV >= 1 && H / HKV <= 4, "need 1 <= H / HKV <= 4");
  BX_REQUIRE(HD == 64 || HD == 128, "head_dim must be 64 or 128");
  BX_REQUIRE(FK == kFK && FZ == kFZ, "the attention's fixed-point formats (FK, FZ) are compiled in");
  BX_REQUIRE((int64_t)nblk * bs <= kDecRawKeys, "the fused form takes at most %d keys per row", kDecRawKeys);
  BX_REQUIRE(ldy >= (int64_t)(H + 2 * HKV) * HD && npos > 0, "bad qkv rows or rope tables");
  BX_REQUIRE(sc_bs >= 6 * HD && sc_nb % 16 == 0 && sc_h % 16 == 0 && sc_bs % 16 == 0 && ((uintptr_t)cache & 15) == 0,
             "cache rows must hold the 6 HD limb bytes, 16-byte aligned");
  BX_REQUIRE(sc_h >= (int64_t)bs * sc_bs && sc_nb >= (int64_t)HKV * sc_h, "cache strides");
  BX_REQUIRE(y && pos && cos && sin && slot && bt && rmap && lut && err, "null pointer");
  BX_REQUIRE(ao != nullptr || (num && den), "null pointer");
  if (R == 0) return BX_OK;
  const int M = H / HKV;
  AttnArgs p = {};
  p.nq = M;
  p.cache = cache; p.sc_nb = sc_nb; p.sc_h = sc_h; p.sc_bs = sc_bs; p.bt = bt; p.sbt = sbt; p.rmap = rmap;
  p.bs = bs; p.hkv = HKV; p.nblk = nblk;
  p.lut = lut; p.l2e = l2e;
  p.num = num; p.den = den; p.snum_tile = (int64_t)M * HD; p.snum_row = HD; p.sden_tile = M;
  p.nsplit = 1;
  RopeArgs r = {y, ldy, pos, spos, 0, cos, sin, npos, R, 1, H, HKV, HD, FR, FT, FK, FV, FZ, nullptr, nullptr, nullptr,
                nullptr, err, cache, sc_nb, sc_h, sc_bs, slot, bs};
  const int64_t max_keys = (int64_t)nblk * bs;
  p.S = (int)((max_keys + 15) / 16 * 16);
  const size_t lds = (size_t)4 * p.S * 8 + ((size_t)p.S / p.bs + 2) * 4;   // scores + block-table entries
  const dim3 grid(R * HKV, 1);
  const int maxlds = (int)(4 * kDecRawKeys * 8 + (kDecRawKeys + 2) * 4);
#define BX_RAW_ROPE(HDV, AOV)                                                                                       \
  do {                                                                                                           \
    hipFuncSetAttribute((const void*)attn_dec_raw_kernel<HDV, true, AOV>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                        maxlds);                                                                                 \
    attn_dec_raw_kernel<HDV, true, AOV><<<grid, kDecWaves * 64, lds, st>>>(p, r, ao ? *ao : AoArgs{});              \
  } while (0)
  if (HD == 64 && ao) BX_RAW_ROPE(64, true);
  else if (HD == 64) BX_RAW_ROPE(64, false);
  else if (ao) BX_RAW_ROPE(128, true);
  else BX_RAW_ROPE(128, false);
#undef BX_RAW_ROPE
  return check_launch("attn_dec_raw_kernel(rope)");
}

extern "C" int bx_exact_attn_paged_rope(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spos,
                                        const int64_t* cos, const int64_t* sin, int32_t npos, int32_t H, int32_t FR,
                                        int32_t FT, int32_t FK, int32_t FV, int32_t FZ, const int64_t* slot,
                                        int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs,
                                        const int32_t* bt, int64_t sbt, int32_t nblk, const int64_t* rmap,
                                        const int64_t* lut, int64_t l2e, int64_t* num, int64_t* den, int32_t R,
                                        int32_t HKV, int32_t HD, int32_t* err, bx_stream_t stream) {
  return attn_rope_common(y, ldy, pos, spos, cos, sin, npos, H, FR, FT, FK, FV, FZ, slot, cache, sc_nb, sc_h, sc_bs, bs,
                          bt, sbt, nblk, rmap, lut, l2e, num, den, R, HKV, HD, err, nullptr, (hipStream_t)stream);
}

extern "C" int64_t bx_attn_rope_out_workspace(int32_t R) {
  if (R <= 0) return 0;
  return (int64_t)R * 12 + 256;
}

extern "C" int64_t bx_attn_rope_out_scratch(int32_t R, int32_t H, int32_t HD) {
  if (R <= 0 || H <= 0 || HD <= 0) return 0;
  return (int64_t)R * H * HD * 8;
}

static int attn_rope_out(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spos, const int64_t* cos,
                         const int64_t* sin, int32_t npos, int32_t H, int32_t FR, int32_t FT, int32_t FK, int32_t FV,
                         int32_t FZ, const int64_t* slot, int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs,
                         int32_t bs, const int32_t* bt, int64_t sbt, int32_t nblk, const int64_t* rmap,
                         const int64_t* lut, int64_t l2e, int32_t* q, int64_t ldq, int64_t* sh, int8_t* planes,
                         int32_t R, int32_t HKV, int32_t HD, int32_t* err, void* ws, int64_t ws_bytes, void* tmp,
                         int64_t tmp_bytes, hipStream_t stream) {
  BX_REQUIRE(q && sh && ldq >= (int64_t)H * HD, "null q / sh or ldq too small");
  BX_REQUIRE(ws && ws_bytes >= bx_attn_rope_out_workspace(R) && ((uintptr_t)ws & 7) == 0,
             "workspace too small (%lld < %lld)", (long long)ws_bytes, (long long)bx_attn_rope_out_workspace(R));
  BX_REQUIRE(tmp && tmp_bytes >= bx_attn_rope_out_scratch(R, H, HD) && ((uintptr_t)tmp & 7) == 0,
             "scratch too small (%lld < %lld)", (long long)tmp_bytes, (long long)bx_attn_rope_out_scratch(R, H, HD));
  BX_REQUIRE(FR - FV >= 0 && FR - FV <= 62, "FR - FV outside [0, 62]");
  AoArgs ao;
  ao.ws_p = (int64_t*)tmp;
  ao.ws_e = (int64_t*)ws;
  ao.cnt = (int32_t*)(ao.ws_e + R);
  ao.q = q; ao.ldq = ldq; ao.sh = sh; ao.FR = FR; ao.FV = FV;
  ao.planes = planes; ao.plane = (int64_t)R * H * HD;
  return attn_rope_common(y, ldy, pos, spos, cos, sin, npos, H, FR, FT, FK, FV, FZ, slot, cache, sc_nb, sc_h, sc_bs, bs,
                          bt, sbt, nblk, rmap, lut, l2e, nullptr, nullptr, R, HKV, HD, err, &ao, stream);
}

extern "C" int bx_exact_attn_paged_rope_out(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spos,
                                            const int64_t* cos, const int64_t* sin, int32_t npos, int32_t H,
                                            int32_t FR, int32_t FT, int32_t FK, int32_t FV, int32_t FZ,
                                            const int64_t* slot, int8_t* cache, int64_t sc_nb, int64_t sc_h,
                                            int64_t sc_bs, int32_t bs, const int32_t* bt, int64_t sbt, int32_t nblk,
                                            const int64_t* rmap, const int64_t* lut, int64_t l2e, int32_t* q,
                                            int64_t ldq, int64_t* sh, int32_t R, int32_t HKV, int32_t HD, int32_t* err,
                                            void* ws, int64_t ws_bytes, void* tmp, int64_t tmp_bytes,
                                            bx_stream_t stream) {
  return attn_rope_out(y, ldy, pos, spos, cos, sin, npos, H, FR, FT, FK, FV, FZ, slot, cache, sc_nb, sc_h, sc_bs, bs, bt,
                       sbt, nblk, rmap, lut, l2e, q, ldq, sh, nullptr, R, HKV, HD, err, ws, ws_bytes, tmp, tmp_bytes,
                       (hipStream_t)stream);
}

extern "C" int bx_exact_attn_paged_rope_out_planes(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spos,
                                                   const int64_t* cos, const int64_t* sin, int32_t npos, int32_t H,
                                                   int32_t FR, int32_t FT, int32_t FK, int32_t FV, int32_t FZ,
                                                   const int64_t* slot, int8_t* cache, int64_t sc_nb, int64_t sc_h,
                                                   int64_t sc_bs, int32_t bs, const int32_t* bt, int64_t sbt,
                                                   int32_t nblk, const int64_t* rmap, const int64_t* lut, int64_t l2e,
                                                   int32_t* q, int64_t ldq, int64_t* sh, int8_t* planes, int32_t R,
                                                   int32_t HKV, int32_t HD, int32_t* err, void* ws, int64_t ws_bytes,
                                                   void* tmp, int64_t tmp_bytes, bx_stream_t stream) {
  BX_REQUIRE(planes, "null planes");
  return attn_rope_out(y, ldy, pos, spos, cos, sin, npos, H, FR, FT, FK, FV, FZ, slot, cache, sc_nb, sc_h, sc_bs, bs, bt,
                       sbt, nblk, rmap, lut, l2e, q, ldq, sh, planes, R, HKV, HD, err, ws, ws_bytes, tmp, tmp_bytes,
                       (hipStream_t)stream);
}

static int int8_paged(const int64_t* q, const int64_t* qpos, int64_t sqpos_r, const int8_t* cache, int64_t sc_nb,
                      int64_t sc_h, int64_t sc_bs, int32_t bs, const int32_t* bt, int64_t sbt, int32_t nblk,
                      const int32_t* ptab, int32_t ptab_len, int64_t* num, int64_t* den, int32_t R, int32_t HKV,
                      int32_t M, int32_t HD, int32_t nsplit, void* ws, int64_t ws_bytes, void* tmp, int64_t tmp_bytes,
                      bx_stream_t stream) {
  BX_REQUIRE(R >= 0 && HKV > 0 && M >= 1, "need M >= 1 queries per (row, KV head)");
  BX_REQUIRE(HD == 64 || HD == 128, "head_dim must be 64 or 128");
  BX_REQUIRE((int64_t)nblk * bs < 43690, "keys per row must stay below 43690");
  BX_REQUIRE(nsplit >= 1 && nsplit <= 64, "nsplit in [1, 64]");
  BX_REQUIRE(ptab_len >= (int32_t)(-kI8ZLo) + 1, "weight table needs 2^17 + 1 entries");
  BX_REQUIRE(sc_bs >= 6 * HD && sc_nb % 16 == 0 && sc_h % 16 == 0 && sc_bs % 16 == 0 && ((uintptr_t)cache & 15) == 0,
             "cache rows must hold the 6 HD limb bytes, 16-byte aligned");
  BX_REQUIRE(q && qpos && bt && ptab && num && den, "null pointer");
  if (R == 0) return BX_OK;
  AttnArgs p = {};
  p.q64 = q; p.sq_tile = (int64_t)M * HD; p.sq_row = HD;
  p.qpos = qpos; p.qpos_tile = sqpos_r; p.qpos_row = 1; p.qpos_div = HKV; p.nq = M;
  p.cache = cache; p.sc_nb = sc_nb; p.sc_h = sc_h; p.sc_bs = sc_bs; p.bt = bt; p.sbt = sbt; p.rmap = nullptr;
  p.bs = bs; p.hkv = HKV; p.nblk = nblk;
  // int8.segs.score_rule (src/bitexact/int8/segs.py:29-37): FQ = 14, FA = 12; head_dim 128 scales by 2^-1/2
  p.wrule = 1; p.ptab = ptab;
  p.zsh = 2 * 14 + 3 - 12 + (HD == 128 ? 24 : 0);
  p.zmul = HD == 128 ? 11863283 : 0;
  p.num = num; p.den = den; p.snum_tile = (int64_t)M * HD; p.snum_row = HD; p.sden_tile = M;
  p.nsplit = nsplit;
  if (nsplit > 1) {
    const int64_t T = (int64_t)R * HKV * ((M + 3) / 4);
    const int64_t need = dec_ws_bytes(T, nsplit, HD);
    BX_REQUIRE(ws != nullptr && ws_bytes >= need, "workspace too small for %d splits (%lld < %lld)", nsplit,
               (long long)ws_bytes, (long long)need);
    BX_REQUIRE(((uintptr_t)ws & 7) == 0, "workspace must be 8-byte aligned");
    p.mx_ws = (int64_t*)ws;
  }
  const int64_t max_keys = (int64_t)nblk * bs;     // qpos < nblk bs: the block table's reach
  if (tmp != nullptr)
    if (int rc = bind_scores(p, (int64_t)R * HKV * ((M + 3) / 4), max_keys, tmp, tmp_bytes)) return rc;
  return HD == 64 ? launch_dec<64>(p, R * HKV, max_keys, (hipStream_t)stream)
                  : launch_dec<128>(p, R * HKV, max_keys, (hipStream_t)stream);
}

extern "C" int bx_int8_attn_paged(const int64_t* q, const int64_t* qpos, int64_t sqpos_r, const int8_t* cache,
                                  int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs, const int32_t* bt, int64_t sbt,
                                  int32_t nblk, const int32_t* ptab, int32_t ptab_len, int64_t* num, int64_t* den,
                                  int32_t R, int32_t HKV, int32_t M, int32_t HD, int32_t nsplit, void* ws,
                                  int64_t ws_bytes, bx_stream_t stream) {
  return int8_paged(q, qpos, sqpos_r, cache, sc_nb, sc_h, sc_bs, bs, bt, sbt, nblk, ptab, ptab_len, num, den,
                    R, HKV, M, HD, nsplit, ws, ws_bytes, nullptr, 0, stream);
}

extern "C" int bx_int8_attn_paged_scores(const int64_t* q, const int64_t* qpos, int64_t sqpos_r, const int8_t* cache,
                                  int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs, const int32_t* bt, int64_t sbt,
                                  int32_t nblk, const int32_t* ptab, int32_t ptab_len, int64_t* num, int64_t* den,
                                  int32_t R, int32_t HKV, int32_t M, int32_t HD, int32_t nsplit, void* ws,
                                  int64_t ws_bytes, void* tmp, int64_t tmp_bytes,
                                  bx_stream_t stream) {
  BX_REQUIRE(tmp != nullptr || R == 0, "null scratch");
  return int8_paged(q, qpos, sqpos_r, cache, sc_nb, sc_h, sc_bs, bs, bt, sbt, nblk, ptab, ptab_len, num, den,
                    R, HKV, M, HD, nsplit, ws, ws_bytes, tmp, tmp_bytes, stream);
}

// the limb-plane form's scratch: K and V planes, 3 Z Sp HD bytes each (Sp = S rounded up to 64 keys), and the weight table
static int64_t pre2_planes(int64_t Z, int64_t S, int64_t HD) { return 2 * 3 * Z * ((S + 63) / 64 * 64) * HD; }
static int64_t pre2_scratch(int64_t Z, int64_t S, int64_t HD) {
  return pre2_planes(Z, S, HD) + (4LL * (kTabPad + kTabBlocks) + 255) / 256 * 256;
}

extern "C" int64_t bx_attn_prefill_scratch(int32_t Z, int32_t S, int32_t HD) {
  if (Z <= 0 || S <= 0 || (HD != 64 && HD != 128)) return 0;
  const int64_t b = pre2_scratch(Z, S, HD);
  return b < kBufRange - 16 ? b : 0;                 // larger: the register-staged form (no scratch)
}

// bx_exact_attn_paged_rows's scratch: the token order, the tile slots and key counts, the rows of sequences with few
// tokens and their splits' workspace, the weight table, the planes
struct RowsLayout {
  int TT, nslot, Sp, nfew;                   // nfew: at most so many rows of sequences with few tokens
  int64_t slots, klen, few, list, sem, ws, raw, tab, planes, total;   // byte offsets (perm at 0; raw -1: no kept scores)
};
constexpr int64_t kFewScoresMax = 1LL << 28;
static RowsLayout rows_layout(int64_t R, int64_t nrow, int64_t HKV, int64_t M, int64_t HD, int64_t keys) {
  RowsLayout l;
  l.TT = (HD == 64 ? Pre2<64>::QR : Pre2<128>::QR) / (int)M;
  l.nslot = (int)(R / l.TT + nrow + 1);
  l.Sp = (int)((keys + 63) / 64 * 64);
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  l.slots = up(R * 4);
  l.klen = l.slots + up(l.nslot * 16LL);
  l.nfew = (int)std::min(R, nrow * (kFewTokens - 1));
  l.few = l.klen + up(nrow * 4);
  l.list = l.few + up(nrow * 8);
  l.sem = l.list + up(4LL * (1 + l.nfew));
  l.ws = l.sem + up(4LL * kDecListBlocks);
  l.raw = l.ws + up(dec_ws_bytes(kDecListBlocks, 1, (int)HD));
  const int64_t scores = 32LL * l.nfew * HKV * keys;
  l.tab = l.raw + (scores <= kFewScoresMax ? up(scores) : 0);
  if (scores > kFewScoresMax) l.raw = -1;
  l.planes = l.tab + up(4LL * (kTabPad + kTabBlocks));
  l.total = l.planes + 6 * nrow * HKV * l.Sp * HD;
  return l;
}
constexpr int64_t kRowsScratchMax = 1LL << 30;

extern "C" int64_t bx_attn_paged_rows_scratch(int32_t R, int32_t nrow, int32_t HKV, int32_t M, int32_t HD, int32_t keys) {
  if (R <= 0 || nrow <= 0 || HKV <= 0 || M < 1 || M > 4 || (HD != 64 && HD != 128) || keys <= 0 || keys >= 43690) return 0;
  const int64_t b = rows_layout(R, nrow, HKV, M, HD, keys).total;
  return b <= kRowsScratchMax ? b : 0;
}

template <int HD, bool RAW>
static int launch_few(const AttnArgs& p, int nfew, hipStream_t st) {
  const int grid = std::max(nfew * p.hkv, kDecListBlocks);
  attn_dec_kernel<HD, 0, RAW, true><<<grid, kDecWaves * 64, 0, st>>>(p);
  if (int rc = check_launch("attn_dec_kernel(list, scores)")) return rc;
  attn_dec_kernel<HD, 1, RAW, true><<<grid, kDecWaves * 64, 0, st>>>(p);
  return check_launch("attn_dec_kernel(list)");
}

extern "C" int bx_exact_attn_paged_rows(const int32_t* q, const int64_t* sh, const int64_t* qpos, int64_t sqpos_r,
                                        const int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs,
                                        const int32_t* bt, int64_t sbt, int32_t nrow, int32_t nblk, const int64_t* rmap,
                                        const int64_t* lut, int64_t l2e, int64_t* num, int64_t* den, int32_t R,
                                        int32_t HKV, int32_t M, int32_t HD, void* tmp, int64_t tmp_bytes,
                                        bx_stream_t stream) {
  BX_REQUIRE(R >= 0 && nrow >= 0 && HKV > 0 && M >= 1 && M <= 4, "need 1 <= M <= 4 queries per (row, KV head)");
  BX_REQUIRE(HD == 64 || HD == 128, "head_dim must be 64 or 128");
  BX_REQUIRE(nblk >= 0 && bs > 0 && (int64_t)nblk * bs < 43690, "keys per row must stay below 43690");
  BX_REQUIRE(sc_bs >= 6 * HD && sc_nb % 16 == 0 && sc_h % 16 == 0 && sc_bs % 16 == 0 && ((uintptr_t)cache & 15) == 0,
             "cache rows must hold the 6 HD limb bytes, 16-byte aligned");
  BX_REQUIRE(q && sh && qpos && bt && rmap && lut && num && den, "null pointer");
  BX_REQUIRE(((uintptr_t)q & 15) == 0, "q must be 16-byte aligned");
  if (R == 0) return BX_OK;
  BX_REQUIRE(nrow > 0 && nblk > 0, "empty block table");
  const RowsLayout l = rows_layout(R, nrow, HKV, M, HD, (int64_t)nblk * bs);
  BX_REQUIRE(l.total <= kRowsScratchMax, "limb planes above %lld bytes: use bx_exact_attn_paged", (long long)kRowsScratchMax);
  BX_REQUIRE(tmp && tmp_bytes >= l.total && ((uintptr_t)tmp & 15) == 0, "scratch too small (%lld < %lld) or not 16-byte aligned",
             (long long)tmp_bytes, (long long)l.total);
  char* t = (char*)tmp;
  int32_t* perm = (int32_t*)t;
  int4* slots = (int4*)(t + l.slots);
  int32_t *klen = (int32_t*)(t + l.klen), *list = (int32_t*)(t + l.list);
  int2* few = (int2*)(t + l.few);
  uint32_t* tab = (uint32_t*)(t + l.tab);
  int8_t* kp = (int8_t*)(t + l.planes);
  int8_t* vp = kp + 3LL * nrow * HKV * l.Sp * HD;
  AttnArgs p = {};
  p.q = q; p.sq_tile = (int64_t)M * HD; p.sq_row = HD;
  p.sh = sh; p.sh_tile = M;
  p.qpos = qpos; p.qpos_tile = sqpos_r; p.qpos_row = 1; p.qpos_div = HKV; p.nq = M;
  p.cache = cache; p.sc_nb = sc_nb; p.sc_h = sc_h; p.sc_bs = sc_bs; p.bt = bt; p.sbt = sbt;
  p.bs = bs; p.hkv = HKV; p.nblk = nblk; p.S = nblk * bs;
  p.lut = lut; p.l2e = l2e;
  p.num = num; p.den = den; p.snum_tile = (int64_t)M * HD; p.snum_row = HD; p.sden_tile = M;
  p.nsplit = 1;
  p.rmap = rmap; p.list = list; p.sem = (int32_t*)(t + l.sem); p.mx_ws = (int64_t*)(t + l.ws);
  p.raw = l.raw < 0 ? nullptr : (int64_t*)(t + l.raw);
  p.one_keys = kDecOneKeys / HD;
  hipStream_t st = (hipStream_t)stream;
  rows_group_kernel<<<nrow + 1, 256, 0, st>>>(rmap, qpos, sqpos_r, R, M, nrow, p.S, l.TT, l.nslot, perm, slots, klen, few);
  if (int rc = check_launch("rows_group_kernel")) return rc;
  const int ntile = l.Sp / 64, Z = nrow * HKV;
  const RowMap rm = {perm, slots, l.nslot, nrow, M, HKV};
  if (HD == 64) {
    paged_planes_kernel<64><<<kTabBlocks + 1 + Z * ntile, 256, 0, st>>>(p, klen, kp, vp, tab, l.Sp, ntile, perm, few, nrow, list);
    if (int rc = check_launch("paged_planes_kernel")) return rc;
    allow_lds_attn((const void*)attn_pre2_kernel<64, true>, Pre2<64>::LDS);
    attn_pre2_kernel<64, true><<<l.nslot * HKV, 64 * Pre2<64>::NW, Pre2<64>::LDS, st>>>(p, kp, Z, l.Sp, tab, rm);
  } else {
    paged_planes_kernel<128><<<kTabBlocks + 1 + Z * ntile, 256, 0, st>>>(p, klen, kp, vp, tab, l.Sp, ntile, perm, few, nrow, list);
    if (int rc = check_launch("paged_planes_kernel")) return rc;
    allow_lds_attn((const void*)attn_pre2_kernel<128, true>, Pre2<128>::LDS);
    attn_pre2_kernel<128, true><<<l.nslot * HKV, 64 * Pre2<128>::NW, Pre2<128>::LDS, st>>>(p, kp, Z, l.Sp, tab, rm);
  }
  if (int rc = check_launch("attn_pre2_kernel(rows)")) return rc;
  if (l.raw < 0) return HD == 64 ? launch_few<64, false>(p, l.nfew, st) : launch_few<128, false>(p, l.nfew, st);
  return HD == 64 ? launch_few<64, true>(p, l.nfew, st) : launch_few<128, true>(p, l.nfew, st);
}

extern "C" int bx_exact_attn_prefill(const int32_t* qg, int64_t sq_z, int64_t sq_row, const int64_t* shg,
                                     int64_t ssh_z, const int64_t* qpos, int64_t sqpos_z, int64_t sqpos_row,
                                     const int32_t* K, int64_t sk_z, int64_t sk_s, const int32_t* V, int64_t sv_z,
                                     int64_t sv_s, int32_t S, const int64_t* lut, int64_t l2e, int64_t* num,
                                     int64_t* den, int32_t Z, int32_t gT, int32_t HD, void* tmp, int64_t tmp_bytes,
                                     bx_stream_t stream) {
  BX_REQUIRE(Z >= 0 && gT >= 0 && S >= 0, "negative size");
  BX_REQUIRE(HD == 64 || HD == 128, "head_dim must be 64 or 128");
  BX_REQUIRE(S < 43690, "keys must stay below 43690");
  BX_REQUIRE(qg && shg && qpos && K && V && lut && num && den, "null pointer");
  BX_REQUIRE(ssh_z == gT, "shg must be [Z, gT, 1] contiguous");
  BX_REQUIRE(((uintptr_t)qg & 15) == 0 && ((uintptr_t)K & 15) == 0 && ((uintptr_t)V & 15) == 0 && sq_z % 4 == 0 &&
                 sq_row % 4 == 0 && sk_z % 4 == 0 && sk_s % 4 == 0 && sv_z % 4 == 0 && sv_s % 4 == 0,
             "qg, K, V: 16-byte aligned rows (base and strides multiples of 4 elements)");
  if (Z == 0 || gT == 0) return BX_OK;
  AttnArgs p = {};
  p.q = qg; p.sq_tile = sq_z; p.sq_row = sq_row;
  p.sh = shg; p.sh_tile = ssh_z;
  p.qpos = qpos; p.qpos_tile = sqpos_z; p.qpos_row = sqpos_row; p.qpos_div = 1; p.nq = gT;
  p.K = K; p.V = V; p.sk_z = sk_z; p.sk_s = sk_s; p.sv_z = sv_z; p.sv_s = sv_s; p.S = S;
  p.lut = lut; p.l2e = l2e;
  p.num = num; p.den = den; p.snum_tile = (int64_t)gT * HD; p.snum_row = HD; p.sden_tile = gT;
  p.nsplit = 1;
  // keys visible to a query never exceed the cache length S: qpos beyond S - 1 is the caller's contract
  hipStream_t st = (hipStream_t)stream;
  if (tmp != nullptr && S > 0) {
    const int64_t need = pre2_scratch(Z, S, HD);
    BX_REQUIRE(need < kBufRange - 16, "limb planes above 2 GiB: call without scratch");
    BX_REQUIRE(tmp_bytes >= need && ((uintptr_t)tmp & 15) == 0, "scratch too small (%lld < %lld) or not 16-byte aligned",
               (long long)tmp_bytes, (long long)need);
    const int Sp = (S + 63) / 64 * 64;
    int8_t* pl = (int8_t*)tmp;
    const int64_t units = (int64_t)Z * Sp * (HD / 16) + (int64_t)Z * (Sp / 4) * (HD / 4);
    uint32_t* tab = (uint32_t*)(pl + pre2_planes(Z, S, HD));
    pre_split_kernel<<<kTabBlocks + (int)std::min<int64_t>((units + 255) / 256, 8192), 256, 0, st>>>(
        p, pl, pl + (int64_t)Z * 3 * Sp * HD, tab, Z, Sp, HD);
    if (int rc = check_launch("pre_split_kernel")) return rc;
    if (HD == 64) {
      allow_lds_attn((const void*)attn_pre2_kernel<64, false>, Pre2<64>::LDS);
      attn_pre2_kernel<64, false><<<Z * ((gT + Pre2<64>::QR - 1) / Pre2<64>::QR), 64 * Pre2<64>::NW, Pre2<64>::LDS, st>>>(
          p, pl, Z, Sp, tab, RowMap{});
    } else {
      allow_lds_attn((const void*)attn_pre2_kernel<128, false>, Pre2<128>::LDS);
      attn_pre2_kernel<128, false><<<Z * ((gT + Pre2<128>::QR - 1) / Pre2<128>::QR), 64 * Pre2<128>::NW, Pre2<128>::LDS, st>>>(
          p, pl, Z, Sp, tab, RowMap{});
    }
    return check_launch("attn_pre2_kernel");
  }
  const int tiles = (gT + 63) / 64;
  if (HD == 64) {
    allow_lds_attn((const void*)attn_pre_kernel<64>, sizeof(PreSmem<64>));
    attn_pre_kernel<64><<<Z * tiles, 256, sizeof(PreSmem<64>), st>>>(p);
  } else {
    allow_lds_attn((const void*)attn_pre_kernel<128>, sizeof(PreSmem<128>));
    attn_pre_kernel<128><<<Z * tiles, 256, sizeof(PreSmem<128>), st>>>(p);
  }
  return check_launch("attn_pre_kernel");
}

extern "C" int bx_kv_store(int8_t* cache, int64_t sc_nb, int64_t sc_h, int64_t sc_bs, int32_t bs, const int64_t* slot,
                           const void* k, int64_t skn, int64_t skh, const void* v, int64_t svn, int64_t svh,
                           int32_t elem_bytes, int32_t N, int32_t HKV, int32_t HD, bx_stream_t stream) {
  BX_REQUIRE(N >= 0 && HKV > 0 && HD > 0 && bs > 0, "bad sizes");
  BX_REQUIRE(elem_bytes == 4 || elem_bytes == 8, "k / v must be int32 or int64");
  BX_REQUIRE(sc_bs >= 6 * HD, "cache rows must hold the 6 HD limb bytes");
  if (N == 0) return BX_OK;
  BX_REQUIRE(cache && slot && k && v, "null pointer");
  dim3 grid(N, HKV);
  if (elem_bytes == 8)
    kv_store_kernel<int64_t><<<grid, 128, 0, (hipStream_t)stream>>>(cache, sc_nb, sc_h, sc_bs, slot, (const int64_t*)k,
                                                                   skn, skh, (const int64_t*)v, svn, svh, HD, bs);
  else
    kv_store_kernel<int32_t><<<grid, 128, 0, (hipStream_t)stream>>>(cache, sc_nb, sc_h, sc_bs, slot, (const int32_t*)k,
                                                                   skn, skh, (const int32_t*)v, svn, svh, HD, bs);
  return check_launch("kv_store_kernel");
}

BX_PHASE_DEFINE(attn)
