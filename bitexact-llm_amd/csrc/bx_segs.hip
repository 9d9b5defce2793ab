// Element-wise segments between the matrix products:
//  * exact mode: RoPE of the qkv linear output, per-(token, head) quantization of q and the regroup by KV head,
//    fused in one pass (segs.rope_y + segs.q_group, src/bitexact/exact/segs.py:66-99);
//  * int8 mode: per-row quantization of the GEMM input with the limbs written as the stacked int8 rows the
//    GEMM reads (int8.ops.quant_rows + intops.stack_limbs, src/bitexact/int8/ops.py:24-35,
//    src/bitexact/intops.py:73-79), and the linear post-segment (int8.segs.post, src/bitexact/int8/segs.py:62-67).
// All arithmetic is int64 with the reference's wrapping and shift rules; every reduction is a maximum.
#include "bx_common.h"
#include "bx_rope.h"

namespace bx {


// intops.rdiv (src/bitexact/intops.py:41-43): floor((2a + b) / (2b)), b > 0.
__device__ __forceinline__ int64_t rdiv64(int64_t a, int64_t b) { return fdiv(add_wrap(2 * a, b), 2 * b); }

__device__ __forceinline__ int64_t seg_block_max(int64_t v, int64_t* sbuf) {
  v = wave_max64(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sbuf[wave] = v;
  __syncthreads();
  int64_t r = sbuf[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) r = imax(r, sbuf[i]);
  return r;
}

// Grid (token, group of head rows): HD / 2 lanes take a head row, lane l its dims l and l + HD / 2 (a RoPE pair), so a
// wave works 64 / (HD / 2) rows at a time with one cos / sin pair per lane and token, and RU of them with all their
// loads in flight. Before, one lane per dim read every pair twice and every row its own cos / sin: 4096 tokens of 32
// + 8 + 8 heads of 64 took 104 us, so 44 us (168 MB). Products are 32 x 32 bits: rows with a value of 2^31 or more
// (flagged) or tables past 32 bits take the wrapping 64-bit products.
template <int HD, int RU>
__global__ __launch_bounds__(256) void rope_qgroup_kernel(RopeArgs p) {
  constexpr int HALF = HD / 2, RW = 64 / HALF;
  const int token = blockIdx.x, b = token / p.T, t = token - b * p.T;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, d = lane % HALF, sub = lane / HALF;
  const int64_t pos_raw = p.pos[(int64_t)b * p.spb + (int64_t)t * p.spt];
  bool bad = pos_raw < 0 || pos_raw >= p.npos;          // the reference's table index would fail: flagged
  const int64_t pos = imin(imax(pos_raw, 0), p.npos - 1);
  const int64_t c = p.cos[pos * HALF + d], sn = p.sin[pos * HALF + d];
  const bool fit = c == (int32_t)c && sn == (int32_t)sn && (int32_t)sn != INT32_MIN;
  const int g = p.H / p.HKV, rows = p.H + 2 * p.HKV;
  const int64_t eps = -(int64_t)(p.FR + p.FT);
  const int64_t* y = p.y + (int64_t)token * p.ldy;
  const int r0 = (blockIdx.y * RU * 4 + wave) * RW + sub;
  int64_t x1[RU], x2[RU];
#pragma unroll
  for (int u = 0; u < RU; ++u) {
    const int64_t* x = y + (int64_t)min(r0 + u * 4 * RW, rows - 1) * HD;
    x1[u] = x[d];
    x2[u] = x[d + HALF];
  }
#pragma unroll
  for (int u = 0; u < RU; ++u) {
    const int hr = r0 + u * 4 * RW;
    const bool live = hr < rows;
    const bool in = x1[u] < (1LL << 31) && x1[u] > -(1LL << 31) && x2[u] < (1LL << 31) && x2[u] > -(1LL << 31);
    bad |= live && !in;
    int64_t o1 = x1[u], o2 = x2[u];
    if (hr < p.H + p.HKV) {
      // _rope_full (src/bitexact/exact/segs.py:66-69): (x1 c - x2 s, x2 c + x1 s)
      if (in && fit) {
        const int32_t a = (int32_t)x1[u], e = (int32_t)x2[u], ci = (int32_t)c, si = (int32_t)sn;
        o1 = (int64_t)a * ci + (int64_t)e * -si;
        o2 = (int64_t)e * ci + (int64_t)a * si;
      } else {
        o1 = add_wrap(mul_wrap(x1[u], c), -mul_wrap(x2[u], sn));
        o2 = add_wrap(mul_wrap(x2[u], c), mul_wrap(x1[u], sn));
      }
    }
    // the magnitudes ored over the row's lanes: the row's bit length (-2^63 sets bit 63 alone: a bit length of 0)
    uint64_t any = (o1 < 0 ? 0 - (uint64_t)o1 : (uint64_t)o1) | (o2 < 0 ? 0 - (uint64_t)o2 : (uint64_t)o2);
    any |= (uint64_t)dpp64<0x121>((int64_t)any);
    any |= (uint64_t)dpp64<0x122>((int64_t)any);
    any |= (uint64_t)dpp64<0x124>((int64_t)any);
    any |= (uint64_t)dpp64<0x128>((int64_t)any);
    any |= (uint64_t)__shfl_xor((long long)any, 16, 64);
    if (HD == 128) any |= (uint64_t)__shfl_xor((long long)any, 32, 64);
    if (!live) continue;
    if (hr < p.H) {
      // q head: ops.quant(Pq, -(FR + FT)) over its HD values, stored at its grouped row
      const uint64_t low = any & (uint64_t)INT64_MAX;
      const int64_t emax = low != 0 ? bitlen((int64_t)low) + eps : any != 0 ? eps : kSegNegBig;
      const int64_t shq = imax(emax - kSegQB, kSegNegBig);
      bad |= shq > p.FK + 3 - p.FZ;
      const int kvh = hr / g, gi = hr - kvh * g;
      const int64_t row = ((int64_t)b * p.HKV + kvh) * ((int64_t)g * p.T) + (int64_t)gi * p.T + t;
      p.qg[row * HD + d] = (int32_t)rshc(o1, shq - eps);
      p.qg[row * HD + d + HALF] = (int32_t)rshc(o2, shq - eps);
      if (d == 0) p.shg[row] = shq;
    } else {
      const bool isk = hr < p.H + p.HKV;
      const int h = isk ? hr - p.H : hr - p.H - p.HKV, down = isk ? p.FR + p.FT - p.FK : p.FR - p.FV;
      const int64_t v1 = rshc(o1, down), v2 = rshc(o2, down);
      bad |= v1 > kLim3 || v1 < -kLim3 || v2 > kLim3 || v2 < -kLim3;
      int64_t* dst = isk ? p.k : p.v;
      if (dst) {
        dst += ((int64_t)token * p.HKV + h) * HD;
        dst[d] = v1;
        dst[d + HALF] = v2;
      }
      store_limbs(p, token, h, isk ? 0 : 3, d, v1);
      store_limbs(p, token, h, isk ? 0 : 3, d + HALF, v2);
    }
  }
  if (wave_or(bad ? 1 : 0) && lane == 0) p.err[0] = 1;
}

// int8 quant_rows + stack_limbs: one block per row. amax is brought to 30 bits (sh), as_ = rsh(amax, sh),
// q = rdiv(rsh(z, sh) qmax, as_); limb i of q[m] goes to stacked row i M + m. With mant / e given, also the
// row scale of segs.pre_plain: (mant, e) = norm24(as_, sh - FR) (src/bitexact/int8/segs.py:56-59,
// src/bitexact/int8/ops.py:73-76).
__global__ __launch_bounds__(256) void int8_quant_rows_kernel(const int64_t* z, int64_t ldz, int M, int K, int nl,
                                                              int FR, int8_t* a, int64_t* as_out, int64_t* sh_out,
                                                              int64_t* mant, int64_t* e) {
  __shared__ int64_t sbuf[4];
  const int m = blockIdx.x;
  const int64_t* zr = z + (int64_t)m * ldz;
  int64_t amax = 0;
  for (int k = threadIdx.x; k < K; k += 256) {
    const int64_t x = zr[k];
    amax = imax(amax, x < 0 ? -x : x);
  }
  amax = imax(seg_block_max(amax, sbuf), 1);
  const int64_t sh = bitlen(amax) - 30;
  const int64_t as = rsh64(amax, sh);
  const int64_t qmax = 127LL << (8 * (nl - 1));
  for (int k = threadIdx.x; k < K; k += 256) {
    int64_t r = rdiv64(mul_wrap(rsh64(zr[k], sh), qmax), as);
    for (int i = 0; i < nl; ++i) {
      const int64_t lo = limb_lo64(r);
      a[((int64_t)i * M + m) * K + k] = (int8_t)lo;
      r = (r - lo) >> 8;
    }
  }
  if (threadIdx.x == 0) {
    as_out[m] = as;
    sh_out[m] = sh;
    if (mant) {
      const int64_t b = bitlen(as) - 24;
      mant[m] = rsh64(as, b);
      e[m] = sh - FR + b;
    }
  }
}

// int8.segs.post: t = rsh(acc m_c, fmsh) (flag when |t| >= 2^38), y = rsh(t mant_r, 24 - FR - e_r).
__global__ __launch_bounds__(256) void int8_post_kernel(const int64_t* acc, int64_t ldacc, const int64_t* mc, int fmsh,
                                                        const int64_t* mant, const int64_t* e, int FR, int64_t* y,
                                                        int64_t ldy, int M, int N, int32_t* flag) {
  const int64_t total = (int64_t)M * N;
  bool big = false;
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int m = (int)(i / N), n = (int)(i - (int64_t)m * N);
    const int64_t t = rsh64(mul_wrap(acc[(int64_t)m * ldacc + n], mc[n]), fmsh);
    big |= t >= (1LL << 38) || t <= -(1LL << 38);
    y[(int64_t)m * ldy + n] = rsh64(mul_wrap(t, mant[m]), 24 - FR - e[m]);
  }
  if (wave_or(big ? 1 : 0) && (threadIdx.x & 63) == 0) flag[0] = 1;
}

// wmm.epilogue over segs.lin_y's inputs (src/bitexact/exact/wmm.py:132-150, src/bitexact/exact/segs.py:25-32):
// T = sum of the split partials, B = dense residual or the ELL gather sum_j q[m, ec[n, j]] ev[n, j], then the
// one rounding at p = sh[m] + g[n] - d[n] + FR; flag[0] = 1 where the checked rule fails.
__global__ __launch_bounds__(256) void exact_epilogue_kernel(const int64_t* T, int64_t ldt, int64_t sts, int nsplit,
                                                             const int64_t* B, int64_t ldb, const int32_t* q,
                                                             int64_t ldq, int K, const int32_t* ec, const int64_t* ev,
                                                             int R, const int64_t* d, const int64_t* g,
                                                             const int64_t* sh, int FR, int checked, int64_t* y,
                                                             int64_t ldy, int M, int N, int32_t* flag) {
  const int64_t total = (int64_t)M * N;
  bool bad_any = false, corrupt = false;
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int m = (int)(i / N), n = (int)(i - (int64_t)m * N);
    int64_t t = 0;
    for (int s = 0; s < nsplit; ++s) t = add_wrap(t, T[s * sts + (int64_t)m * ldt + n]);
    int64_t b = 0;
    if (B) {
      b = B[(int64_t)m * ldb + n];
    } else {
      for (int j = 0; j < R; ++j) {
        // valid ELL columns are in [0, K); a corrupt one reads column 0 and raises the flag
        const uint32_t c0 = (uint32_t)ec[(int64_t)n * R + j];
        const bool out = c0 >= (uint32_t)K;
        corrupt |= out;
        const int c = out ? 0 : (int)c0;
        b = add_wrap(b, mul_wrap((int64_t)q[(int64_t)m * ldq + c], ev[(int64_t)n * R + j]));
      }
    }
    const int64_t dn = d[n];
    bool bad;
    y[(int64_t)m * ldy + n] = exact_round(t, b, dn, sh[m] + g[n] - dn + FR, bad);
    bad_any |= bad;
  }
  if (wave_or(((checked && bad_any) || corrupt) ? 1 : 0) && flag != nullptr && (threadIdx.x & 63) == 0) flag[0] = 1;
}

}  // namespace bx

using namespace bx;

static int rope_common(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spb, int64_t spt,
                       const int64_t* cos, const int64_t* sin, int32_t npos, int32_t B, int32_t T, int32_t H,
                       int32_t HKV, int32_t HD, int32_t FR, int32_t FT, int32_t FK, int32_t FV, int32_t FZ,
                       int32_t* qg, int64_t* shg, int64_t* k, int64_t* v, int32_t* err, int8_t* cache, int64_t sc_nb,
                       int64_t sc_h, int64_t sc_bs, const int64_t* slot, int32_t bs, hipStream_t stream);

extern "C" int bx_rope_qgroup(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spb, int64_t spt,
                              const int64_t* cos, const int64_t* sin, int32_t npos, int32_t B, int32_t T, int32_t H,
                              int32_t HKV, int32_t HD, int32_t FR, int32_t FT, int32_t FK, int32_t FV, int32_t FZ,
                              int32_t* qg, int64_t* shg, int64_t* k, int64_t* v, int32_t* err, bx_stream_t stream) {
  BX_REQUIRE(k && v, "null pointer");
  return rope_common(y, ldy, pos, spb, spt, cos, sin, npos, B, T, H, HKV, HD, FR, FT, FK, FV, FZ, qg, shg, k, v, err,
                     nullptr, 0, 0, 0, nullptr, 1, (hipStream_t)stream);
}

extern "C" int bx_rope_qgroup_store(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spb, int64_t spt,
                                    const int64_t* cos, const int64_t* sin, int32_t npos, int32_t B, int32_t T,
                                    int32_t H, int32_t HKV, int32_t HD, int32_t FR, int32_t FT, int32_t FK, int32_t FV,
                                    int32_t FZ, int32_t* qg, int64_t* shg, int64_t* k, int64_t* v, int8_t* cache,
                                    int64_t sc_nb, int64_t sc_h, int64_t sc_bs, const int64_t* slot, int32_t bs,
                                    int32_t* err, bx_stream_t stream) {
  BX_REQUIRE(cache && slot && bs > 0, "null cache / slot");
  BX_REQUIRE(sc_bs >= 8LL * HD && sc_h >= (int64_t)bs * sc_bs && sc_nb >= (int64_t)HKV * sc_h, "cache strides");
  return rope_common(y, ldy, pos, spb, spt, cos, sin, npos, B, T, H, HKV, HD, FR, FT, FK, FV, FZ, qg, shg, k, v, err,
                     cache, sc_nb, sc_h, sc_bs, slot, bs, (hipStream_t)stream);
}

static int rope_common(const int64_t* y, int64_t ldy, const int64_t* pos, int64_t spb, int64_t spt,
                       const int64_t* cos, const int64_t* sin, int32_t npos, int32_t B, int32_t T, int32_t H,
                       int32_t HKV, int32_t HD, int32_t FR, int32_t FT, int32_t FK, int32_t FV, int32_t FZ,
                       int32_t* qg, int64_t* shg, int64_t* k, int64_t* v, int32_t* err, int8_t* cache, int64_t sc_nb,
                       int64_t sc_h, int64_t sc_bs, const int64_t* slot, int32_t bs, hipStream_t stream) {
  BX_REQUIRE(B >= 0 && T >= 0 && H > 0 && HKV > 0 && H % HKV == 0, "bad head counts");
  BX_REQUIRE(HD == 64 || HD == 128, "head_dim 64 or 128");
  BX_REQUIRE(ldy >= (int64_t)(H + 2 * HKV) * HD, "ldy too small");
  BX_REQUIRE(npos > 0, "empty rope tables");
  if (B == 0 || T == 0) return BX_OK;
  BX_REQUIRE(y && pos && cos && sin && qg && shg && err, "null pointer");
  RopeArgs p = {y, ldy, pos, spb, spt, cos, sin, npos, B, T, H, HKV, HD, FR, FT, FK, FV, FZ, qg, shg, k, v, err,
                cache, sc_nb, sc_h, sc_bs, slot, bs};
  // many tokens: a block takes a whole token's rows, 3 a wave in flight; few: a block per 4 waves' rows
  const int rows = H + 2 * HKV, per = 4 * (128 / HD);
  hipStream_t st = (hipStream_t)stream;
  if ((int64_t)B * T >= 2 * device_cus()) {
    const dim3 blocks(B * T, (rows + 3 * per - 1) / (3 * per));
    if (HD == 64) rope_qgroup_kernel<64, 3><<<blocks, 256, 0, st>>>(p);
    else rope_qgroup_kernel<128, 3><<<blocks, 256, 0, st>>>(p);
  } else {
    const dim3 blocks(B * T, (rows + per - 1) / per);
    if (HD == 64) rope_qgroup_kernel<64, 1><<<blocks, 256, 0, st>>>(p);
    else rope_qgroup_kernel<128, 1><<<blocks, 256, 0, st>>>(p);
  }
  return check_launch("rope_qgroup_kernel");
}

extern "C" int bx_int8_quant_rows(const int64_t* z, int64_t ldz, int32_t M, int32_t K, int32_t nl, int32_t FR,
                                  int8_t* a, int64_t* as_, int64_t* sh, int64_t* mant, int64_t* e,
                                  bx_stream_t stream) {
  BX_REQUIRE(M >= 0 && K >= 0 && ldz >= K, "bad sizes");
  BX_REQUIRE(nl >= 1 && nl <= 3, "nl must be 1, 2 or 3");
  if (M == 0) return BX_OK;
  BX_REQUIRE(z && a && as_ && sh, "null pointer");
  BX_REQUIRE((mant == nullptr) == (e == nullptr), "mant and e come together");
  int8_quant_rows_kernel<<<M, 256, 0, (hipStream_t)stream>>>(z, ldz, M, K, nl, FR, a, as_, sh, mant, e);
  return check_launch("int8_quant_rows_kernel");
}

extern "C" int bx_int8_post(const int64_t* acc, int64_t ldacc, const int64_t* m, int32_t fmsh, const int64_t* mant,
                            const int64_t* e, int32_t FR, int64_t* y, int64_t ldy, int32_t M, int32_t N, int32_t* flag,
                            bx_stream_t stream) {
  BX_REQUIRE(M >= 0 && N >= 0 && ldacc >= N && ldy >= N, "bad sizes");
  if (M == 0 || N == 0) return BX_OK;
  BX_REQUIRE(acc && m && mant && e && y && flag, "null pointer");
  const int64_t total = (int64_t)M * N;
  const int blocks = (int)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
  int8_post_kernel<<<blocks, 256, 0, (hipStream_t)stream>>>(acc, ldacc, m, fmsh, mant, e, FR, y, ldy, M, N, flag);
  return check_launch("int8_post_kernel");
}

extern "C" int bx_exact_epilogue(const int64_t* T, int64_t ldt, int64_t sts, int32_t nsplit, const int64_t* B,
                                 int64_t ldb, const int32_t* q, int64_t ldq, int32_t K, const int32_t* ell_col,
                                 const int64_t* ell_val, int32_t R, const int64_t* d, const int64_t* g,
                                 const int64_t* sh, int32_t FR, int32_t checked, int64_t* y, int64_t ldy, int32_t M,
                                 int32_t N, int32_t* flag, bx_stream_t stream) {
  BX_REQUIRE(M >= 0 && N >= 0 && nsplit >= 1 && ldt >= N && ldy >= N, "bad sizes");
  BX_REQUIRE(B == nullptr || ldb >= N, "ldb too small");
  BX_REQUIRE(B != nullptr || R == 0 || (q && ell_col && ell_val && K > 0 && ldq >= K), "residual missing");
  BX_REQUIRE(!checked || flag, "checked needs a flag pointer");
  if (M == 0 || N == 0) return BX_OK;
  BX_REQUIRE(T && d && g && sh && y, "null pointer");
  const int64_t total = (int64_t)M * N;
  const int blocks = (int)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192);
  exact_epilogue_kernel<<<blocks, 256, 0, (hipStream_t)stream>>>(T, ldt, sts, nsplit, B, ldb, q, ldq, K, ell_col,
                                                                ell_val, B ? 0 : R, d, g, sh, FR, checked, y, ldy, M,
                                                                N, flag);
  return check_launch("exact_epilogue_kernel");
}
