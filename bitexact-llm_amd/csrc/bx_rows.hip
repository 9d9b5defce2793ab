// Row-wise integer stages around the GEMMs and the attention, one block per row (1024 threads for few rows, as in a
// decode step, so each row spreads over a whole CU; smaller blocks for many; softmax rows use 256; the SiLU stage of
// few rows goes over column chunks, that of many walks rows with its table in LDS) with DPP wavefront int64
// reductions: RMSNorm + per-row quantization (segs.norm_quant, optionally after the residual add or the embedding
// gather), SiLU gating + quantization (segs.silu_y + quant_silu), the masked softmax weights (segs.softmax), and the
// attention output rule (segs.attn_out = div_round + regroup + quant).
#include "bx_common.h"
#include "bx_introws.h"

#include <algorithm>

namespace bx {

BX_PHASE_TABLE


constexpr int kRowThreads = 1024;

// ---- segs.norm_quant (src/bitexact/exact/segs.py:59-63) over ops.rms (src/bitexact/exact/ops.py:92-105) and
// ops.quant (src/bitexact/exact/ops.py:82-89), on the residual row the block first forms:
//   SRC_X    the row of x as it is;
//   SRC_ADD  x + y (segs.add_y, src/bitexact/exact/segs.py:40-41), written back to x;
//   SRC_EMB  emb[ids[row]] widened to int64 (the model's `emb[ids].long()`, exact/model.py:130), written to x.
// With gm null only the residual row is formed and bound-checked (the last layer's add). The row and P stay in LDS between the
// passes. ----
enum RowSrc { SRC_X = 0, SRC_ADD = 1, SRC_EMB = 2 };

struct NormArgs {
  int64_t* x;
  int64_t ldx;
  const int64_t* y;
  int64_t ldy;
  const int32_t* emb;
  const int64_t* ids;
  const int64_t* gm;
  const int64_t* ge;
  int32_t* q;
  int64_t ldq;
  int64_t* sh;
  int D, lg, FR, FN;
  int32_t* err;
  int8_t* planes;   // optional: q's signed int8 limb planes [3][M][D] (limb i of q[m][k] at i M D + m D + k)
  int64_t plane;    // M D
  bool vec;         // pairs of columns by 16-byte accesses (set by launch_norm)
};

// Pairs of columns i, i + 1: 16-byte loads where `vec` (host: aligned bases, even strides), else one by one; columns
// past D read as 0.
typedef int64_t v2l __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2l ld_pair(const int64_t* a, int i, int D, bool vec) {
  if (vec) return i < D ? *(const v2l*)(a + i) : v2l{0, 0};
  return v2l{i < D ? a[i] : 0, i + 1 < D ? a[i + 1] : 0};
}
__device__ __forceinline__ void st_q_pair(int32_t* q, int i, int D, bool vec, int32_t a, int32_t b) {
  if (vec) {
    if (i < D) *(int2*)(q + i) = int2{a, b};
  } else {
    if (i < D) q[i] = a;
    if (i + 1 < D) q[i + 1] = b;
  }
}
__device__ __forceinline__ void st_limbs(int8_t* dst, int64_t plane, int32_t r) {   // split_q_kernel's limbs
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    const int32_t lo = limb_lo(r);
    dst[l * plane] = (int8_t)lo;
    r = (r - lo) >> 8;
  }
}
// max over the block of non-negative float64 values (their bit patterns order as integers)
template <int NW>
__device__ __forceinline__ double block_fmax(double v, int64_t* slot) {
  return __builtin_bit_cast(double, block_reduce64_dpp<true, NW>(__builtin_bit_cast(int64_t, v), slot, 0));
}

// The row's rule in int64 as the reference states it, on x as it stands in memory: taken by rows the float64 form
// cannot hold (a value of 2^52 or more, a quotient of 2^50 or more). The quotients are formed twice.
template <int NT>
__device__ void norm_row_general(const NormArgs& p, const int64_t* xr) {
  constexpr int NW = NT / 64;
  __shared__ int64_t gbuf[3][NW];
  const int D = p.D;
  int64_t amax = 0;
  for (int i = threadIdx.x; i < D; i += NT) amax = imax(amax, xr[i] < 0 ? -xr[i] : xr[i]);
  amax = block_reduce64_dpp<true, NW>(amax, gbuf[0], 0);
  if (threadIdx.x == 0 && amax >= (1LL << 40)) p.err[0] = 1;
  if (p.gm == nullptr) return;
  const int64_t shx = imax(bitlen(imax(amax, 1)) - 25, -6);
  int64_t S = 0;
  for (int i = threadIdx.x; i < D; i += NT) {
    const int64_t xs = rshc(xr[i], shx);
    S = add_wrap(S, mul_wrap(xs, xs));
  }
  S = block_reduce64_dpp<false, NW>(S, gbuf[1], 0);
  const int64_t T = add_wrap(S, rshc(kEps60 * (int64_t)D, 60 - 2 * (p.FR - shx)));
  const int64_t m = fdiv(62 + p.lg - bitlen(T), 2);
  const int64_t s = 2 * m - p.lg;
  const int64_t V = s >= 0 ? shl(T, s) : sar(T, -s);
  const int64_t r = isqrt64(V), er = shx - p.FR - m;
  const double rinv = 1.0 / (double)r;
  int64_t emax = kNegBig;
  for (int i = threadIdx.x; i < D; i += NT) {
    const int64_t P = div_round64(mul_wrap(xr[i], p.gm[i]), p.ge[i] - p.FR - er + p.FN, r, rinv);
    if (P != 0) emax = imax(emax, bitlen(P < 0 ? -P : P) - p.FN);
  }
  emax = block_reduce64_dpp<true, NW>(emax, gbuf[2], kNegBig);
  const int64_t shr = imax(emax - kQB, kNegBig);
  for (int i = threadIdx.x; i < D; i += NT) {
    const int64_t P = div_round64(mul_wrap(xr[i], p.gm[i]), p.ge[i] - p.FR - er + p.FN, r, rinv);
    const int32_t qv = (int32_t)rshc(P, shr + p.FN);
    p.q[(int64_t)blockIdx.x * p.ldq + i] = qv;
    if (p.planes != nullptr) st_limbs(p.planes + (int64_t)blockIdx.x * D + i, p.plane, qv);
  }
  if (threadIdx.x == 0) p.sh[blockIdx.x] = shr;
}

// One block of NT threads per row, EPT elements of it in a thread's registers. The arithmetic runs in float64, which
// holds every integer of the rule exactly in the rows' ordinary range (|x| < 2^52, quotients below 2^50; other rows
// take norm_row_general): the division by the rms is one estimate, a fused remainder and a correction, the
// quantization a scale, half and floor. NT = 1024 (2 elements a thread) for few rows, where one row's latency
// counts; NT = 256 (8 a thread, 8 blocks a CU) from two rows per CU: 4096 rows of 2048 measured 74 us with one
// 1024-thread block of integer arithmetic a row, 57 us (add, 235 MB) and 40 us (embedding, 134 MB) so, near HBM's
// rate for reads and writes mixed; a decode step's 32 launches together 39 us less.
template <int SRC, int NT, int EPT>
__global__ __launch_bounds__(NT) void norm_quant_kernel(NormArgs p) {
  BX_PHASE(0, 0);
  constexpr int NW = NT / 64, H = EPT / 2;
  __shared__ int64_t sbuf[3][NW];
  const int D = p.D;
  const bool vec = p.vec;
  int64_t* xr = p.x + (int64_t)blockIdx.x * p.ldx;
  const int32_t* er_row = nullptr;
  if (SRC == SRC_EMB) er_row = p.emb + p.ids[blockIdx.x] * (int64_t)D;
  const int64_t* yr = SRC == SRC_ADD ? p.y + (int64_t)blockIdx.x * p.ldy : nullptr;
  double X[EPT];
  v2l gm2[H], ge2[H];
  {
    v2l v[H], y[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int i = 2 * (h * NT + threadIdx.x);
      if (SRC == SRC_EMB) {
        if (vec) {
          const int2 e = i < D ? *(const int2*)(er_row + i) : int2{0, 0};
          v[h] = v2l{e.x, e.y};
        } else {
          v[h] = v2l{i < D ? er_row[i] : 0, i + 1 < D ? er_row[i + 1] : 0};
        }
      } else {
        v[h] = ld_pair(xr, i, D, vec);
        if (SRC == SRC_ADD) y[h] = ld_pair(yr, i, D, vec);
      }
    }
    if (EPT <= 4 && p.gm != nullptr) {   // the gamma pairs, requested with the row (wide rows: after its sum)
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const int i = 2 * (h * NT + threadIdx.x);
        gm2[h] = ld_pair(p.gm, i, D, vec);
        ge2[h] = ld_pair(p.ge, i, D, vec);
      }
    }
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int i = 2 * (h * NT + threadIdx.x);
      if (SRC == SRC_ADD) v[h] = v2l{add_wrap(v[h][0], y[h][0]), add_wrap(v[h][1], y[h][1])};
      if (SRC != SRC_X) {
        if (vec) {
          if (i < D) *(v2l*)(xr + i) = v[h];
        } else {
          if (i < D) xr[i] = v[h][0];
          if (i + 1 < D) xr[i + 1] = v[h][1];
        }
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) X[2 * h + e] = (double)v[h][e];
    }
  }
  double am = 0;
#pragma unroll
  for (int k = 0; k < EPT; ++k) am = __builtin_fmax(am, __builtin_fabs(X[k]));
  BX_PHASE(0, 1);
  am = block_fmax<NW>(am, sbuf[0]);
  if (am >= 0x1p52) {                                // block-uniform: the int64 rule (the row is written: see it whole)
    __syncthreads();
    norm_row_general<NT>(p, xr);
    return;
  }
  if (threadIdx.x == 0 && am >= 0x1p40) p.err[0] = 1;
  if (p.gm == nullptr) return;
  const int shx = am > 0 ? (int)imax(bitlen_f64(am) - 25, -6) : -6;
  const double xsc = ldexp(1.0, -shx);
  int64_t S = 0;
#pragma unroll
  for (int k = 0; k < EPT; ++k) {                    // rshc(x, shx): |.| <= 2^25, exact in float64
    const int32_t xs = (int32_t)__builtin_floor(__builtin_fma(X[k], xsc, 0.5));
    S += (int64_t)xs * xs;
  }
  S = block_reduce64_dpp<false, NW>(S, sbuf[1], 0);
  if (EPT > 4) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int i = 2 * (h * NT + threadIdx.x);
      gm2[h] = ld_pair(p.gm, i, D, vec);
      ge2[h] = ld_pair(p.ge, i, D, vec);
    }
  }
  const int64_t T = add_wrap(S, rshc(kEps60 * (int64_t)D, 60 - 2 * (p.FR - shx)));
  const int64_t m = (62 + p.lg - bitlen(T)) >> 1;
  const int64_t s = 2 * m - p.lg;
  const int64_t V = s >= 0 ? shl(T, s) : sar(T, -s);
  const int64_t r = isqrt64(V), er = shx - p.FR - m;
  const double rf = (double)r, rinv = 1.0 / rf;
  BX_PHASE(0, 2);
  double pm = 0;
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const int64_t gm = gm2[k >> 1][k & 1], pe = ge2[k >> 1][k & 1] - p.FR - er + p.FN;
    const double A0 = X[k] * (double)gm;
    const bool ok = (__builtin_fabs(A0) < 0x1p52 && pe >= 0 && pe <= 62) || 2 * ((k >> 1) * NT + (int)threadIdx.x) + (k & 1) >= D;
    X[k] = div_round_f64(ldexp(A0, (int)pe), rf, rinv);   // (a column past D: 0)
    const double mag = __builtin_fabs(X[k]);
    pm = __builtin_fmax(pm, ok && mag < 0x1p50 ? mag : __builtin_inf());
  }
  BX_PHASE(0, 3);
  if (r <= 0 || r >= (1LL << 34)) pm = __builtin_inf();
  pm = block_fmax<NW>(pm, sbuf[2]);
  if (pm == __builtin_inf()) {
    __syncthreads();
    norm_row_general<NT>(p, xr);
    return;
  }
  const int64_t shr = pm > 0 ? imax(bitlen_f64(pm) - p.FN - kQB, kNegBig) : kNegBig;
  const double qsc = ldexp(1.0, (int)-imin(imax(shr + p.FN, -62), 62));
  int32_t* qr = p.q + (int64_t)blockIdx.x * p.ldq;
#pragma unroll
  for (int h = 0; h < H; ++h) {                      // rshc(P, shr + FN)
    const int i = 2 * (h * NT + threadIdx.x);
    int32_t qv[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) qv[e] = (int32_t)__builtin_floor(__builtin_fma(X[2 * h + e], qsc, 0.5));
    st_q_pair(qr, i, D, vec, qv[0], qv[1]);
    if (p.planes != nullptr && i < D) {              // (planes: D % 16 == 0)
      int8_t* dst = p.planes + (int64_t)blockIdx.x * D + i;
      if (vec) {
        // byte i of q + 0x808080 is limb i + 128 (the adds' carries are the digits' borrows)
        const uint32_t y0 = ((uint32_t)qv[0] + 0x808080u) ^ 0x808080u, y1 = ((uint32_t)qv[1] + 0x808080u) ^ 0x808080u;
#pragma unroll
        for (int l = 0; l < 3; ++l)
          *(uint16_t*)(dst + l * p.plane) = (uint16_t)(((y0 >> (8 * l)) & 255u) | (((y1 >> (8 * l)) & 255u) << 8));
      } else {
        st_limbs(dst, p.plane, qv[0]);
        st_limbs(dst + 1, p.plane, qv[1]);
      }
    }
  }
  if (threadIdx.x == 0) p.sh[blockIdx.x] = shr;
  BX_PHASE(0, 4);
}

// ---- segs.silu_y + segs.quant_silu (src/bitexact/exact/segs.py:120-128) over ops.silu_mul
// (src/bitexact/exact/ops.py:119-130): per row of gu = [gate | up] at FR, P = silu(gate) up at 2 FR exactly,
// then the row quantization at eps = -2 FR. err[0] = 1 where silu_mul's ok is false (|g| > 2^32, or an element
// with bitlen(|s|) + bitlen(|u|) > 62). ----
__global__ __launch_bounds__(kRowThreads) void silu_quant_kernel(const int64_t* gu, int64_t ldgu, int ff, const int64_t* lut,
                                                         int FR, int32_t* q, int64_t ldq, int64_t* sh, int32_t* err) {
  extern __shared__ __align__(16) char smem[];
  int64_t* Ps = (int64_t*)smem;
  __shared__ int64_t sbuf[16];
  const int64_t* row = gu + (int64_t)blockIdx.x * ldgu;
  const int eps = -2 * FR;
  int64_t emax = kNegBig;
  int bad = 0;
  // kSiluU elements per thread at a time: their row loads, then their table loads, are issued together (one
  // element after another, each waited for its own two dependent loads)
  constexpr int kSiluU = 4;
  for (int i0 = threadIdx.x; i0 < ff; i0 += kSiluU * kRowThreads) {
  int64_t gv[kSiluU], uv[kSiluU], la[kSiluU], lb[kSiluU];
#pragma unroll
  for (int k = 0; k < kSiluU; ++k) {
    const int i = min(i0 + k * kRowThreads, ff - 1);
    gv[k] = row[i];
    uv[k] = row[ff + i];
  }
#pragma unroll
  for (int k = 0; k < kSiluU; ++k) {
    const int idx = silu_index(gv[k], FR);
    la[k] = lut[idx];
    lb[k] = lut[idx + 1];
  }
#pragma unroll
  for (int k = 0; k < kSiluU; ++k) {
    const int i = i0 + k * kRowThreads;
    if (i >= ff) continue;
    const int64_t P = silu_any(gv[k], uv[k], la[k], lb[k], FR, bad);
    Ps[i] = P;
    if (P != 0) emax = imax(emax, bitlen(P < 0 ? (int64_t)(0 - (uint64_t)P) : P) + eps);
  }
  }
  if (bad) err[0] = 1;
  emax = block_max64(emax, sbuf);
  const int64_t shr = imax(emax - kQB, kNegBig);
  for (int i = threadIdx.x; i < ff; i += kRowThreads) q[(int64_t)blockIdx.x * ldq + i] = (int32_t)rshc(Ps[i], shr - eps);
  if (threadIdx.x == 0) sh[blockIdx.x] = shr;
}

// ---- the same stage for many rows (FR = 24): one 1024-thread block per CU walks rows with the 2^-f table in LDS ----
// A row-per-block launch gathered two 8-byte table entries an element through L1 (the 128 KiB table misses its 32
// KiB) and divided twice per element, once for each sign of g: 4096 rows of 2 x 8192 took 337 us against 134 us
// for their bytes at 5 TB/s. Here the gathers are LDS reads, the quotient is one float64 estimate, a thread keeps its
// products in registers (8 columns a chunk of 8192) and the next chunk's 16-byte loads are in flight while this one
// is worked: 121 us (5.5 TB/s of the bytes it must move), bound by HBM.
constexpr int kSiluTab = 16385;
__device__ __forceinline__ uint64_t wave_or64(uint64_t v) {
  v |= (uint64_t)dpp64<0x121>((int64_t)v);
  v |= (uint64_t)dpp64<0x122>((int64_t)v);
  v |= (uint64_t)dpp64<0x124>((int64_t)v);
  v |= (uint64_t)dpp64<0x128>((int64_t)v);
  return (uint64_t)(readlane64((int64_t)v, 0) | readlane64((int64_t)v, 16) | readlane64((int64_t)v, 32) |
                    readlane64((int64_t)v, 48));
}
template <int NCH>
__global__ __launch_bounds__(1024) void silu_rows_kernel(const int64_t* gu, int64_t ldgu, int ff, const int64_t* lut,
                                                         int32_t* q, int64_t ldq, int64_t* sh, int M, int32_t* err) {
  extern __shared__ __align__(16) int64_t T[];       // the table
  __shared__ uint64_t sor[2][16];
  constexpr int FR = 24, eps = -2 * FR;
  const int tid = threadIdx.x;
  v2l G[4], V[4];
  auto load = [&](int r, int ch) {                   // columns past the row: its last pair (their products are not used)
    const int64_t* row = gu + (int64_t)r * ldgu;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int c = min(ch * 8192 + (k * 1024 + tid) * 2, ff - 2);
      G[k] = __builtin_nontemporal_load((const v2l*)(row + c));
      V[k] = __builtin_nontemporal_load((const v2l*)(row + ff + c));
    }
  };
  load(blockIdx.x, 0);
  for (int i = tid; i < kSiluTab; i += 1024) T[i] = lut[i];
  __syncthreads();
  int par = 0;
  for (int r = blockIdx.x; r < M; r += gridDim.x, par ^= 1) {
    int64_t P[NCH * 8];
    uint64_t any = 0;                                // the products' magnitudes ored: the row's bit length
    int bad = 0;
    bool least = false;                              // a product of -2^63, whose magnitude wraps (bitlen 0)
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        SiluAt a[2];
        int64_t la[2], lb[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          a[e] = silu_at24(G[k][e]);
          la[e] = T[a[e].idx];
          lb[e] = T[a[e].idx + 1];
        }
        const bool in = ch * 8192 + (k * 1024 + tid) * 2 < ff;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          int64_t v;
          const bool ok = silu_short24(G[k][e], V[k][e], a[e], la[e], lb[e], v);
          if (!ok) {
            int b = 0;
            v = silu_elem(G[k][e], V[k][e], la[e], lb[e], FR, b);
            if (in) bad |= b;
            if (in && v == INT64_MIN) least = true;
          }
          P[ch * 8 + k * 2 + e] = v;
          const uint64_t m = v < 0 ? 0 - (uint64_t)v : (uint64_t)v;
          if (in) any |= m & (uint64_t)INT64_MAX;
        }
      }
      if (ch + 1 < NCH) load(r, ch + 1);
      else if (r + (int)gridDim.x < M) load(r + gridDim.x, 0);
    }
    if (bad) err[0] = 1;
    any = wave_or64(any) | (wave_or(least ? 1 : 0) ? 1ULL << 63 : 0);
    if ((tid & 63) == 0) sor[par][tid >> 6] = any;
    lds_sync();                                      // the other buffer serves the next row, so one barrier a row
    any = wave_or64(sor[par][tid & 15]);
    const int64_t len = 64 - __clzll((long long)(any & (uint64_t)INT64_MAX));
    const int64_t emax = (any & (uint64_t)INT64_MAX) != 0 ? len + eps : any != 0 ? eps : kNegBig;
    const int64_t shr = imax(emax - kQB, kNegBig);
    const int64_t s = imin(imax(shr - eps, -62), 62);
    int32_t* qr = q + (int64_t)r * ldq;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int c = ch * 8192 + (k * 1024 + tid) * 2;
        if (c < ff) *(int2*)(qr + c) = int2{(int)rshc(P[ch * 8 + k * 2], s), (int)rshc(P[ch * 8 + k * 2 + 1], s)};
      }
    if (tid == 0) sh[r] = shr;
  }
}

// ---- intops.first_argmax (src/bitexact/intops.py:55-59): index of the first maximum of each int64 row. A lane
// keeps its first maximum (columns rise along its loop, only a strictly larger value replaces it); the block
// then takes the row maximum and the smallest index holding it. Integer max / min: no order dependence. ----
__global__ __launch_bounds__(1024) void first_argmax_kernel(const int64_t* v, int64_t ldv, int N, int64_t* out) {
  __shared__ int64_t smax[16], sidx[16];
  const int64_t* row = v + (int64_t)blockIdx.x * ldv;
  int64_t best = INT64_MIN, idx = N;
  constexpr int U = 8;                             // loads in flight per thread
  int i0 = threadIdx.x;
  for (; i0 + (U - 1) * 1024 < N; i0 += U * 1024) {
    int64_t x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = __builtin_nontemporal_load(row + i0 + u * 1024);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (x[u] > best || idx == N) { best = x[u]; idx = i0 + u * 1024; }
  }
  for (int i = i0; i < N; i += 1024) {
    const int64_t x = row[i];
    if (x > best || idx == N) { best = x; idx = i; }
  }
  int64_t m = best;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = imax(m, __shfl_xor(m, o, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) smax[wave] = m;
  __syncthreads();
  int64_t rm = smax[0];
  for (int w = 1; w < 16; ++w) rm = imax(rm, smax[w]);
  int64_t cand = (best == rm) ? idx : N;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) cand = imin(cand, __shfl_xor(cand, o, 64));
  if (lane == 0) sidx[wave] = cand;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t r = sidx[0];
    for (int w = 1; w < 16; ++w) r = imin(r, sidx[w]);
    out[blockIdx.x] = r;
  }
}

// ---- segs.softmax (src/bitexact/exact/segs.py:102-105) over ops.softmax_w: key s visible iff s <= qpos ----
__global__ __launch_bounds__(256) void softmax_kernel(const int64_t* raw, int64_t ldr, const int64_t* qpos,
                                                      const int64_t* sh, int S, int kbits, const int64_t* lut,
                                                      int64_t l2e, int fp, int32_t* p, int64_t ldp, int64_t* den) {
  __shared__ int64_t sbuf[16];
  const int64_t row = blockIdx.x;
  const int64_t* rr = raw + row * ldr;
  const int64_t qp = qpos[row];
  int64_t mx = kNeg;
  for (int i = threadIdx.x; i < S; i += 256)
    if (i <= qp) mx = imax(mx, rr[i]);
  mx = block_max64(mx, sbuf);
  const int64_t zshift = kbits + 3 - sh[row] - 26;
  int64_t sum = 0;
  for (int i = threadIdx.x; i < S; i += 256) {
    const int64_t w = i <= qp ? weight64(mx - rr[i], zshift, lut, l2e, fp) : 0;
    p[row * ldp + i] = (int32_t)w;
    sum += w;
  }
  sum = block_sum64(sum, sbuf);
  if (threadIdx.x == 0) den[row] = sum;
}

// ---- segs.attn_out (src/bitexact/exact/segs.py:108-113, 187-188): o = div_round(num, FR - FV, den), regrouped to
// one row of H HD values per token, then quantized per row with eps = -FR. Output row o, head hh:
// group = (o / T) HKV + hh / g, query = (hh % g) T + o % T, with g = H / HKV. ----
__global__ __launch_bounds__(kRowThreads) void attn_out_kernel(const int64_t* num, int64_t sn_group, int64_t sn_query,
                                                       const int64_t* den, int64_t sd_group, int T, int HKV, int g,
                                                       int HD, int FR, int FV, int32_t* q, int64_t ldq, int64_t* sh) {
  extern __shared__ __align__(16) char smem[];
  int64_t* Os = (int64_t*)smem;
  __shared__ int64_t sbuf[16];
  const int o = blockIdx.x;
  const int W = HKV * g * HD;
  int64_t emax = kNegBig;
  for (int c = threadIdx.x; c < W; c += kRowThreads) {
    const int hh = c / HD, d = c % HD;
    const int64_t group = (int64_t)(o / T) * HKV + hh / g, query = (int64_t)(hh % g) * T + o % T;
    const int64_t dn = den[group * sd_group + query];   // >= 1 whenever the query sees a key (itself)
    const int64_t v = dn > 0 ? div_round64(num[group * sn_group + query * sn_query + d], FR - FV, dn, 1.0 / (double)dn) : 0;
    Os[c] = v;
    if (v != 0) emax = imax(emax, bitlen(v < 0 ? -v : v) - FR);
  }
  emax = block_max64(emax, sbuf);
  const int64_t shr = imax(emax - kQB, kNegBig);
  for (int c = threadIdx.x; c < W; c += kRowThreads) q[(int64_t)o * ldq + c] = (int32_t)rshc(Os[c], shr + FR);
  if (threadIdx.x == 0) sh[o] = shr;
}

// The same stage with the row in registers (EPT elements a thread, pairs of columns of one head) and the quotients in
// float64 (div_round_f64): rows of at most NT EPT columns, even head_dim, 16-byte aligned. A row that float64 does
// not hold (|num| 2^(FR - FV) of 2^52 or more, den of 2^34 or more, a quotient of 2^50 or more) forms its quotients
// in int64, twice. NT = 256 from two rows per CU on: 4096 rows of 2048 took 59 us with one 1024-thread block a row
// (a float64 division and an int64 one per element), 27 us so (101 MB of HBM traffic).
template <int NT, int EPT>
__global__ __launch_bounds__(NT) void attn_out_regs_kernel(const int64_t* num, int64_t sn_group, int64_t sn_query,
                                                           const int64_t* den, int64_t sd_group, int T, int HKV, int g,
                                                           int HD, int FR, int FV, int32_t* q, int64_t ldq, int64_t* sh) {
  constexpr int NW = NT / 64, H = EPT / 2;
  __shared__ int64_t sbuf[2][NW];
  const int o = blockIdx.x, b = o / T, t = o - b * T;
  const int W = HKV * g * HD;
  auto where = [&](int c, int64_t& nm, int64_t& dn) {   // element offsets of column c's num and its head's den
    const int hh = c / HD, d = c - hh * HD, kv = hh / g;
    const int64_t group = (int64_t)b * HKV + kv, query = (int64_t)(hh - kv * g) * T + t;
    nm = group * sn_group + query * sn_query + d;
    dn = group * sd_group + query;
  };
  v2l n2[H];
  int64_t d1[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    int64_t nm, dn;
    where(min(2 * (h * NT + (int)threadIdx.x), W - 2), nm, dn);
    n2[h] = *(const v2l*)(num + nm);
    d1[h] = den[dn];
  }
  const double up = ldexp(1.0, FR - FV);
  double P[EPT], pm = 0;
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const bool in = 2 * (h * NT + (int)threadIdx.x) < W;
    const double r = (double)d1[h];
    double x = __builtin_amdgcn_rcp(r);               // 1 / r: two Newton steps
    x = __builtin_fma(x, __builtin_fma(-r, x, 1.0), x);
    x = __builtin_fma(x, __builtin_fma(-r, x, 1.0), x);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const double A = (double)n2[h][e];
      const double v = d1[h] > 0 ? div_round_f64(A * up, r, x) : 0.0;   // den = 0: no visible key
      const double mag = __builtin_fabs(v);
      P[2 * h + e] = v;
      if (in) pm = __builtin_fmax(pm, __builtin_fabs(A) < 0x1p52 && d1[h] < (1LL << 34) && mag < 0x1p48 ? mag : __builtin_inf());
    }
  }
  pm = block_fmax<NW>(pm, sbuf[0]);
  int32_t* qr = q + (int64_t)o * ldq;
  if (pm == __builtin_inf()) {                       // block-uniform
    auto quot = [&](int c) {
      int64_t nm, dn;
      where(c, nm, dn);
      return den[dn] > 0 ? div_round64(num[nm], FR - FV, den[dn], 1.0 / (double)den[dn]) : 0;
    };
    int64_t emax = kNegBig;
    for (int c = threadIdx.x; c < W; c += NT) {
      const int64_t v = quot(c);
      if (v != 0) emax = imax(emax, bitlen(v < 0 ? -v : v) - FR);
    }
    emax = block_reduce64_dpp<true, NW>(emax, sbuf[1], kNegBig);
    const int64_t shr = imax(emax - kQB, kNegBig);
    for (int c = threadIdx.x; c < W; c += NT) qr[c] = (int32_t)rshc(quot(c), shr + FR);
    if (threadIdx.x == 0) sh[o] = shr;
    return;
  }
  const int64_t shr = pm > 0 ? imax(bitlen_f64(pm) - FR - kQB, kNegBig) : kNegBig;
  const double qsc = ldexp(1.0, (int)-imin(imax(shr + FR, -62), 62));
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int c = 2 * (h * NT + (int)threadIdx.x);
    if (c < W)
      *(int2*)(qr + c) = int2{(int)__builtin_floor(__builtin_fma(P[2 * h], qsc, 0.5)),
                              (int)__builtin_floor(__builtin_fma(P[2 * h + 1], qsc, 0.5))};
  }
  if (threadIdx.x == 0) sh[o] = shr;
}

// The same stage split over column chunks for few rows (one block per row would leave most CUs idle while each
// streams its 16 ff bytes of gate | up): grid (C, M), chunk index fastest, chunks of about 1024 columns.
constexpr int kSiluPartThreads = 256;
// Block (m, c) keeps its chunk's P in LDS, publishes the chunk's exponent maximum
// (as emax - kNegBig + 1; 0 = not yet published) and waits for the other chunks of its row for at most `ticks` of
// the 100 MHz real-time counter. A block that has not seen them all by then forms the row's maximum itself from
// gu (the same integers, slower), so the wait always ends. The row's last block to finish reading resets its
// slots and counter: the zero-filled workspace is left as it was found.
constexpr uint64_t kSiluTicks = 20000;   // 200 us
__global__ __launch_bounds__(kSiluPartThreads) void silu_fused_kernel(const int64_t* gu, int64_t ldgu, int ff,
                                                                      int chunk, const int64_t* lut, int FR,
                                                                      int64_t* slots, int32_t* cnt, uint64_t ticks,
                                                                      int32_t* q, int64_t ldq, int64_t* sh,
                                                                      int8_t* planes, int32_t* err) {
  extern __shared__ __align__(16) int64_t Ps[];   // [chunk]
  __shared__ int64_t sbuf[16];
  __shared__ int64_t s_row;
  const int m = blockIdx.y, c = blockIdx.x, C = gridDim.x;   // chunk index fastest: a row's chunks run together
  const int64_t* row = gu + (int64_t)m * ldgu;
  const int i_lo = c * chunk, i_hi = min(ff, i_lo + chunk);
  const int eps = -2 * (int)FR;
  int64_t emax = kNegBig;
  int bad = 0;
  constexpr int U = 4;
  for (int i0 = i_lo + threadIdx.x; i0 < i_hi; i0 += U * kSiluPartThreads) {
    int64_t gv[U], uv[U], la[U], lb[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int i = min(i0 + k * kSiluPartThreads, i_hi - 1);
      gv[k] = row[i];
      uv[k] = row[ff + i];
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int idx = silu_index(gv[k], FR);
      la[k] = lut[idx];
      lb[k] = lut[idx + 1];
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int i = i0 + k * kSiluPartThreads;
      if (i >= i_hi) continue;
      const int64_t v = silu_any(gv[k], uv[k], la[k], lb[k], FR, bad);
      Ps[i - i_lo] = v;
      if (v != 0) emax = imax(emax, bitlen(v < 0 ? (int64_t)(0 - (uint64_t)v) : v) + eps);
    }
  }
  if (bad) err[0] = 1;
  emax = block_max64(emax, sbuf);
  if (threadIdx.x == 0) {
    s_row = emax;
    ws_store(&slots[(int64_t)m * C + c], emax - kNegBig + 1);
  }
  lds_sync();
  bool seen = true;
  if ((int)threadIdx.x < C && (int)threadIdx.x != c) {
    int64_t* a = &slots[(int64_t)m * C + threadIdx.x];
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    int64_t v = ws_load(a);
    while (v == 0 && __builtin_amdgcn_s_memrealtime() - t0 < ticks) {
      __builtin_amdgcn_s_sleep(1);
      v = ws_load(a);
    }
    seen = v != 0;
    if (seen) atomicMax((long long*)&s_row, (long long)(v - 1 + kNegBig));
  }
  const bool all = __syncthreads_and(seen);
  // Thread 0's own publish (an agent-scope store) is complete before its count (s_waitcnt), so no publish can
  // arrive after the row's last block has reset the slots. (An agent-scope release / acquire fence would write back
  // and invalidate the whole L2 on this chip; the waits on the coherent stores are all that is needed.)
  if (threadIdx.x == 0) __builtin_amdgcn_s_waitcnt(0);
  if (threadIdx.x == 0 && atomicAdd(&cnt[m], 1) == C - 1) {
    for (int j = 0; j < C; ++j) ws_store(&slots[(int64_t)m * C + j], 0);
    atomicExch(&cnt[m], 0);
  }
  int64_t rmax = s_row;
  if (!all) {   // the row's maximum from gu (blocks of the row that did not run alongside this one)
    int64_t e2 = kNegBig;
    int bad2 = 0;
    for (int i = threadIdx.x; i < ff; i += kSiluPartThreads) {
      const int64_t g = row[i];
      const int idx = silu_index(g, FR);
      const int64_t v = silu_elem(g, row[ff + i], lut[idx], lut[idx + 1], FR, bad2);
      if (v != 0) e2 = imax(e2, bitlen(v < 0 ? (int64_t)(0 - (uint64_t)v) : v) + eps);
    }
    rmax = block_max64(e2, sbuf);
  }
  const int64_t shr = imax(rmax - kQB, kNegBig);
  const int64_t plane = (int64_t)gridDim.y * ff;
  for (int i = i_lo + threadIdx.x; i < i_hi; i += kSiluPartThreads) {
    const int32_t qv = (int32_t)rshc(Ps[i - i_lo], shr - eps);
    q[(int64_t)m * ldq + i] = qv;
    if (planes != nullptr) {
      int32_t r = qv;
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        const int32_t lo = limb_lo(r);
        planes[l * plane + (int64_t)m * ff + i] = (int8_t)lo;
        r = (r - lo) >> 8;
      }
    }
  }
  if (c == 0 && threadIdx.x == 0) sh[m] = shr;
}


// first_argmax split over column chunks for few rows (one block per row streams the whole row on one CU):
// argmax_part_kernel, grid (M, C), writes each chunk's (maximum, its first index) to scratch slots; argmax_fin_kernel
// takes, per row, the first chunk holding the row maximum (chunks in column order, so ties keep the smallest index).
constexpr int kArgThreads = 256;
__global__ __launch_bounds__(kArgThreads) void argmax_part_kernel(const int64_t* v, int64_t ldv, int N, int chunk,
                                                                  int64_t* slots) {
  __shared__ int64_t smax[kArgThreads / 64], sidx[kArgThreads / 64];
  const int m = blockIdx.x, c = blockIdx.y, C = gridDim.y;
  const int64_t* row = v + (int64_t)m * ldv;
  const int i_lo = c * chunk, i_hi = min(N, i_lo + chunk);
  int64_t best = INT64_MIN, idx = N;
  constexpr int U = 8;
  int i0 = i_lo + threadIdx.x;
  for (; i0 + (U - 1) * kArgThreads < i_hi; i0 += U * kArgThreads) {
    int64_t x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = __builtin_nontemporal_load(row + i0 + u * kArgThreads);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (x[u] > best || idx == N) { best = x[u]; idx = i0 + u * kArgThreads; }
  }
  for (int i = i0; i < i_hi; i += kArgThreads) {
    const int64_t x = row[i];
    if (x > best || idx == N) { best = x; idx = i; }
  }
  int64_t mx = best;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = imax(mx, __shfl_xor(mx, o, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) smax[wave] = mx;
  __syncthreads();
  int64_t rm = smax[0];
  for (int w = 1; w < kArgThreads / 64; ++w) rm = imax(rm, smax[w]);
  int64_t cand = (best == rm) ? idx : N;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) cand = imin(cand, __shfl_xor(cand, o, 64));
  if (lane == 0) sidx[wave] = cand;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t ri = sidx[0];
    for (int w = 1; w < kArgThreads / 64; ++w) ri = imin(ri, sidx[w]);
    slots[((int64_t)m * C + c) * 2] = rm;
    slots[((int64_t)m * C + c) * 2 + 1] = ri;
  }
}

__global__ __launch_bounds__(64) void argmax_fin_kernel(const int64_t* slots, int M, int N, int C, int64_t* out) {
  const int m = blockIdx.x * 64 + threadIdx.x;
  if (m >= M) return;
  int64_t best = INT64_MIN, idx = N;
  for (int c = 0; c < C; ++c) {
    const int64_t sv = slots[((int64_t)m * C + c) * 2], si = slots[((int64_t)m * C + c) * 2 + 1];
    if (sv > best || idx == N) { best = sv; idx = si; }
  }
  out[m] = idx;
}

// A greedy decode step's next inputs, one thread per sequence: ids = the step's first-max tokens, pos + 1, and the
// cache slot of the new position through the block table (slot = bt[rmap, pos / bs] bs + pos % bs).
__global__ void decode_advance_kernel(const int64_t* next, int64_t* ids, int64_t* pos, int64_t* slot, const int32_t* bt,
                                      int64_t sbt, const int64_t* rmap, int bs, int N) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int64_t p = pos[n] + 1;
  ids[n] = next[n];
  pos[n] = p;
  slot[n] = (int64_t)bt[rmap[n] * sbt + p / bs] * bs + p % bs;
}

}  // namespace bx

using namespace bx;

static void allow_lds_rows(const void* k, size_t lds) {
  if (lds > 64 * 1024) hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

static int launch_norm(NormArgs& p, int src, int32_t M, bx_stream_t stream) {
  int lg = 0;
  while ((1 << lg) < p.D) ++lg;
  BX_REQUIRE(p.D > 0 && (1 << lg) == p.D && lg <= 12, "row length a power of two <= 4096");
  BX_REQUIRE(M >= 0 && p.ldx >= p.D, "bad sizes");
  BX_REQUIRE(p.x && p.err, "null pointer");
  BX_REQUIRE(!p.gm || (p.ge && p.q && p.sh && p.ldq >= p.D), "gamma given without the quantized outputs");
  if (M == 0) return BX_OK;
  p.lg = lg;
  hipStream_t st = (hipStream_t)stream;
  auto al = [](const void* a, unsigned m) { return ((uintptr_t)a & m) == 0; };
  p.vec = p.D >= 2 && al(p.x, 15) && p.ldx % 2 == 0 && al(p.y, 15) && p.ldy % 2 == 0 && al(p.emb, 7) && al(p.gm, 15) &&
          al(p.ge, 15) && al(p.q, 7) && p.ldq % 2 == 0 && al(p.planes, 1);
  const bool many = M >= 2 * device_cus();
#define BX_NORM(SRCV)                                                                        \
  do {                                                                                       \
    if (!many && p.D <= 2048) norm_quant_kernel<SRCV, 1024, 2><<<M, 1024, 0, st>>>(p);       \
    else if (!many) norm_quant_kernel<SRCV, 1024, 4><<<M, 1024, 0, st>>>(p);                 \
    else if (p.D <= 1024) norm_quant_kernel<SRCV, 256, 4><<<M, 256, 0, st>>>(p);             \
    else if (p.D <= 2048) norm_quant_kernel<SRCV, 256, 8><<<M, 256, 0, st>>>(p);             \
    else norm_quant_kernel<SRCV, 512, 8><<<M, 512, 0, st>>>(p);                              \
  } while (0)
  if (src == SRC_ADD) BX_NORM(SRC_ADD);
  else if (src == SRC_EMB) BX_NORM(SRC_EMB);
  else BX_NORM(SRC_X);
#undef BX_NORM
  return check_launch("norm_quant_kernel");
}

extern "C" int bx_rmsnorm_quant(const int64_t* x, int64_t ldx, const int64_t* gm, const int64_t* ge, int32_t* q,
                                int64_t ldq, int64_t* sh, int32_t M, int32_t D, int32_t FR, int32_t FN, int32_t* err,
                                bx_stream_t stream) {
  BX_REQUIRE(gm && ge && q && sh, "null pointer");
  NormArgs p = {const_cast<int64_t*>(x), ldx, nullptr, 0, nullptr, nullptr, gm, ge, q, ldq, sh, D, 0, FR, FN, err, nullptr, 0, false};
  return launch_norm(p, SRC_X, M, stream);
}

extern "C" int bx_add_rmsnorm_quant(int64_t* x, int64_t ldx, const int64_t* y, int64_t ldy, const int64_t* gm,
                                    const int64_t* ge, int32_t* q, int64_t ldq, int64_t* sh, int32_t M, int32_t D,
                                    int32_t FR, int32_t FN, int32_t* err, bx_stream_t stream) {
  BX_REQUIRE(y && ldy >= D, "y: null or ldy too small");
  NormArgs p = {x, ldx, y, ldy, nullptr, nullptr, gm, ge, q, ldq, sh, D, 0, FR, FN, err, nullptr, 0, false};
  return launch_norm(p, SRC_ADD, M, stream);
}

extern "C" int bx_add_rmsnorm_quant_planes(int64_t* x, int64_t ldx, const int64_t* y, int64_t ldy, const int64_t* gm,
                                           const int64_t* ge, int32_t* q, int64_t ldq, int64_t* sh, int8_t* planes,
                                           int32_t M, int32_t D, int32_t FR, int32_t FN, int32_t* err,
                                           bx_stream_t stream) {
  BX_REQUIRE(!y || ldy >= D, "ldy too small");
  BX_REQUIRE(gm && ge && q && sh && planes, "null pointer");
  BX_REQUIRE(D % 16 == 0, "D %% 16 != 0 (the limb planes are the exact GEMM's K-major operand)");
  NormArgs p = {x, ldx, y, ldy, nullptr, nullptr, gm, ge, q, ldq, sh, D, 0, FR, FN, err, planes, (int64_t)M * D, false};
  return launch_norm(p, y ? SRC_ADD : SRC_X, M, stream);   // y null: the norm of x as it is (x not written)
}

extern "C" int bx_embed_rmsnorm_quant(const int32_t* emb, const int64_t* ids, int64_t* x, int64_t ldx,
                                      const int64_t* gm, const int64_t* ge, int32_t* q, int64_t ldq, int64_t* sh,
                                      int32_t M, int32_t D, int32_t FR, int32_t FN, int32_t* err, bx_stream_t stream) {
  BX_REQUIRE(emb && ids, "null pointer");
  NormArgs p = {x, ldx, nullptr, 0, emb, ids, gm, ge, q, ldq, sh, D, 0, FR, FN, err, nullptr, 0, false};
  return launch_norm(p, SRC_EMB, M, stream);
}

extern "C" int bx_embed_rmsnorm_quant_planes(const int32_t* emb, const int64_t* ids, int64_t* x, int64_t ldx,
                                             const int64_t* gm, const int64_t* ge, int32_t* q, int64_t ldq,
                                             int64_t* sh, int8_t* planes, int32_t M, int32_t D, int32_t FR,
                                             int32_t FN, int32_t* err, bx_stream_t stream) {
  BX_REQUIRE(emb && ids && gm && ge && q && sh && planes, "null pointer");
  BX_REQUIRE(D % 16 == 0, "D %% 16 != 0 (the limb planes are the exact GEMM's K-major operand)");
  NormArgs p = {x, ldx, nullptr, 0, emb, ids, gm, ge, q, ldq, sh, D, 0, FR, FN, err, planes, (int64_t)M * D, false};
  return launch_norm(p, SRC_EMB, M, stream);
}

extern "C" int bx_silu_quant(const int64_t* gu, int64_t ldgu, int32_t ff, const int64_t* lut, int32_t FR, int32_t* q,
                             int64_t ldq, int64_t* sh, int32_t M, int32_t* err, bx_stream_t stream) {
  BX_REQUIRE(M >= 0 && ff > 0 && ldgu >= 2 * (int64_t)ff && ldq >= ff, "bad sizes");
  BX_REQUIRE(ff <= 16384, "ff > 16384 (row kept in LDS)");
  BX_REQUIRE(FR >= 0 && FR <= 24, "FR outside [0, 24]");
  BX_REQUIRE(gu && lut && q && sh && err, "null pointer");
  if (M == 0) return BX_OK;
  // many rows, whole pairs of columns, 16-byte rows: the table-in-LDS kernel (one block per CU; below 2 rows a block the
  // table's 128 KiB copy costs what it saves)
  const int cus = device_cus();
  if (FR == 24 && M >= 2 * cus && ff >= 2048 && ff % 2 == 0 && ldgu % 2 == 0 && ldq % 2 == 0 &&
      ((uintptr_t)gu & 15) == 0 && ((uintptr_t)q & 7) == 0) {
    constexpr size_t tl = kSiluTab * 8 + 8;
    const dim3 grid(std::min(M, cus));
    if (ff <= 8192) {
      allow_lds_rows((const void*)silu_rows_kernel<1>, tl);
      silu_rows_kernel<1><<<grid, 1024, tl, (hipStream_t)stream>>>(gu, ldgu, ff, lut, q, ldq, sh, M, err);
    } else {
      allow_lds_rows((const void*)silu_rows_kernel<2>, tl);
      silu_rows_kernel<2><<<grid, 1024, tl, (hipStream_t)stream>>>(gu, ldgu, ff, lut, q, ldq, sh, M, err);
    }
    return check_launch("silu_rows_kernel");
  }
  const size_t lds = (size_t)ff * 8;
  allow_lds_rows((const void*)silu_quant_kernel, lds);
  silu_quant_kernel<<<M, kRowThreads, lds, (hipStream_t)stream>>>(gu, ldgu, ff, lut, FR, q, ldq, sh, err);
  return check_launch("silu_quant_kernel");
}

// silu chunks: about 1024 elements each, at most 64 per row
static int silu_chunks(int ff) { return std::min(64, std::max(1, (ff + 1023) / 1024)); }

extern "C" int64_t bx_silu_quant_scratch(int32_t M, int32_t ff) {
  if (M <= 0 || ff <= 0) return 0;
  return (int64_t)M * silu_chunks(ff) * 8 + (int64_t)M * 4;
}

extern "C" int bx_silu_quant_ws(const int64_t* gu, int64_t ldgu, int32_t ff, const int64_t* lut, int32_t FR, int32_t* q,
                                int64_t ldq, int64_t* sh, int8_t* planes, int32_t M, int32_t* err, void* tmp,
                                int64_t tmp_bytes, bx_stream_t stream) {
  BX_REQUIRE(M >= 0 && ff > 0 && ldgu >= 2 * (int64_t)ff && ldq >= ff, "bad sizes");
  BX_REQUIRE(FR >= 0 && FR <= 24, "FR outside [0, 24]");
  BX_REQUIRE(gu && lut && q && sh && err, "null pointer");
  if (M == 0) return BX_OK;
  BX_REQUIRE(tmp && tmp_bytes >= bx_silu_quant_scratch(M, ff) && ((uintptr_t)tmp & 7) == 0,
             "scratch too small (%lld < %lld)", (long long)tmp_bytes, (long long)bx_silu_quant_scratch(M, ff));
  BX_REQUIRE(!planes || ff % 16 == 0, "limb planes need ff %% 16 == 0");
  const int C = silu_chunks(ff), chunk = (ff + C - 1) / C;
  // dynamic LDS (the chunk's products) plus the kernel's static LDS must stay within the default 64 KiB
  BX_REQUIRE((int64_t)chunk * 8 <= 63 * 1024, "ff too large for the one-launch form");
  int64_t* slots = (int64_t*)tmp;
  int32_t* cnt = (int32_t*)(slots + (int64_t)M * C);
  // BX_SILU_TICKS (tests): a shorter wait, down to 0, where blocks form the row maximum they have not seen
  const char* et = getenv("BX_SILU_TICKS");
  const uint64_t ticks = et ? (uint64_t)strtoull(et, nullptr, 10) : kSiluTicks;
  silu_fused_kernel<<<dim3(C, M), kSiluPartThreads, (size_t)chunk * 8, (hipStream_t)stream>>>(
      gu, ldgu, ff, chunk, lut, FR, slots, cnt, ticks, q, ldq, sh, planes, err);
  return check_launch("silu_fused_kernel");
}

extern "C" int bx_first_argmax(const int64_t* v, int64_t ldv, int32_t M, int32_t N, int64_t* out, bx_stream_t stream) {
  BX_REQUIRE(M >= 0 && N > 0 && ldv >= N, "bad sizes");
  BX_REQUIRE(v && out, "null pointer");
  if (M == 0) return BX_OK;
  first_argmax_kernel<<<M, 1024, 0, (hipStream_t)stream>>>(v, ldv, N, out);
  return check_launch("first_argmax_kernel");
}

static int argmax_chunks(int N) { return std::min(64, std::max(1, (N + 8191) / 8192)); }

extern "C" int64_t bx_first_argmax_scratch(int32_t M, int32_t N) {
  if (M <= 0 || N <= 0) return 0;
  return (int64_t)M * argmax_chunks(N) * 16;
}

extern "C" int bx_first_argmax_ws(const int64_t* v, int64_t ldv, int32_t M, int32_t N, int64_t* out, void* tmp,
                                  int64_t tmp_bytes, bx_stream_t stream) {
  BX_REQUIRE(M >= 0 && N > 0 && ldv >= N, "bad sizes");
  BX_REQUIRE(v && out, "null pointer");
  if (M == 0) return BX_OK;
  BX_REQUIRE(tmp && tmp_bytes >= bx_first_argmax_scratch(M, N) && ((uintptr_t)tmp & 7) == 0,
             "scratch too small (%lld < %lld)", (long long)tmp_bytes, (long long)bx_first_argmax_scratch(M, N));
  const int C = argmax_chunks(N), chunk = (N + C - 1) / C;
  int64_t* slots = (int64_t*)tmp;
  argmax_part_kernel<<<dim3(M, C), kArgThreads, 0, (hipStream_t)stream>>>(v, ldv, N, chunk, slots);
  if (int rc = check_launch("argmax_part_kernel")) return rc;
  argmax_fin_kernel<<<(M + 63) / 64, 64, 0, (hipStream_t)stream>>>(slots, M, N, C, out);
  return check_launch("argmax_fin_kernel");
}

extern "C" int bx_softmax_w(const int64_t* raw, int64_t ldr, const int64_t* qpos, const int64_t* sh, int32_t rows,
                            int32_t S, int32_t kbits, const int64_t* lut, int64_t l2e, int32_t fp, int32_t* p,
                            int64_t ldp, int64_t* den, bx_stream_t stream) {
  BX_REQUIRE(rows >= 0 && S >= 0 && ldr >= S && ldp >= S, "bad sizes");
  BX_REQUIRE(raw && qpos && sh && lut && p && den, "null pointer");
  if (rows == 0) return BX_OK;
  softmax_kernel<<<rows, 256, 0, (hipStream_t)stream>>>(raw, ldr, qpos, sh, S, kbits, lut, l2e, fp, p, ldp, den);
  return check_launch("softmax_kernel");
}

extern "C" int bx_attn_out(const int64_t* num, int64_t sn_group, int64_t sn_query, const int64_t* den,
                           int64_t sd_group, int32_t rows, int32_t T, int32_t HKV, int32_t g, int32_t HD, int32_t FR,
                           int32_t FV, int32_t* q, int64_t ldq, int64_t* sh, bx_stream_t stream) {
  BX_REQUIRE(rows >= 0 && T > 0 && HKV > 0 && g > 0 && HD > 0 && rows % T == 0, "bad sizes");
  BX_REQUIRE(ldq >= (int64_t)HKV * g * HD, "ldq too small");
  BX_REQUIRE(num && den && q && sh, "null pointer");
  if (rows == 0) return BX_OK;
  const int64_t W = (int64_t)HKV * g * HD;
  if (W <= 4096 && HD % 2 == 0 && FR >= FV && FR - FV <= 62 && ((uintptr_t)num & 15) == 0 && sn_group % 2 == 0 &&
      sn_query % 2 == 0 && ((uintptr_t)q & 7) == 0 && ldq % 2 == 0) {
    hipStream_t st = (hipStream_t)stream;
    const bool many = rows >= 2 * device_cus();
#define BX_AOUT(NT, EPT) \
  attn_out_regs_kernel<NT, EPT><<<rows, NT, 0, st>>>(num, sn_group, sn_query, den, sd_group, T, HKV, g, HD, FR, FV, q, ldq, sh)
    if (!many && W <= 2048) BX_AOUT(1024, 2);
    else if (!many) BX_AOUT(1024, 4);
    else if (W <= 2048) BX_AOUT(256, 8);
    else BX_AOUT(512, 8);
#undef BX_AOUT
    return check_launch("attn_out_regs_kernel");
  }
  const size_t lds = (size_t)W * 8;
  allow_lds_rows((const void*)attn_out_kernel, lds);
  attn_out_kernel<<<rows, kRowThreads, lds, (hipStream_t)stream>>>(num, sn_group, sn_query, den, sd_group, T, HKV, g, HD, FR,
                                                          FV, q, ldq, sh);
  return check_launch("attn_out_kernel");
}

BX_PHASE_DEFINE(rows)

extern "C" int bx_decode_advance(const int64_t* next, int64_t* ids, int64_t* pos, int64_t* slot, const int32_t* bt,
                                 int64_t sbt, int32_t nblk, const int64_t* rmap, int32_t bs, int32_t N,
                                 bx_stream_t stream) {
  BX_REQUIRE(N >= 0 && bs > 0 && nblk > 0 && sbt >= nblk, "bad sizes");
  if (N == 0) return BX_OK;
  BX_REQUIRE(next && ids && pos && slot && bt && rmap, "null pointer");
  decode_advance_kernel<<<(N + 255) / 256, 256, 0, (hipStream_t)stream>>>(next, ids, pos, slot, bt, sbt, rmap, bs, N);
  return check_launch("decode_advance_kernel");
}
