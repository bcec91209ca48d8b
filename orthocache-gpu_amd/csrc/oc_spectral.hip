// The 512-token block spectra of orthocache_forward(mode='compact') and its
// stream compaction (declared in include/orthocache_hip.h).
//
// The normalised 512-point Walsh-Hadamard transform along tokens, X =
// H512 K / sqrt(512) in natural (Hadamard) order, factors over the token
// index t = 64 th + tl and the sequency u = 64 uh + ul as H512[u, t] =
// H8[uh, th] H64[ul, tl].  With Z_uh[tl] = sum_th H8[uh, th] K[64 th + tl]
// (an 8-point transform across the block's eight 64-token chunks),
// X[64 uh + ul] = (H64 Z_uh)[ul] / sqrt(512), and by Parseval over ul
//   sum_ul ||X[64 uh + ul]||^2 = ||Z_uh||_F^2 / 8.
// So the bands [64, 256) (uh = 1..3) and [256, 512) (uh = 4..7) are sums of
// squares of the 8-point outputs, computed in registers as the block
// streams in; the band [1, 64) is, by Parseval over tl, what is left of
// Z_0 without its mean, 64 sum_tl (Z_0[tl] - mean)^2, from the registers too
// (the generic head_dim path does the 64-point transform per column from
// LDS).  Every band energy is a sum of squares, so near-zero bands stay
// exact-ish instead of cancelling.
#include <hip/hip_runtime.h>

#include <cmath>

#include "oc_kernels.h"
#include "oc_status.h"
#include "orthocache_hip.h"

namespace oc {
namespace {

constexpr int kSpThreads = 256;
constexpr int kBlock = 512;
constexpr int kMaxD = 256;

struct SpecArgs {
  const char* k;
  int64_t k_ts, k_hs;  // byte strides: token, head
  int32_t H, d, nb, dtype;
  const char* q;       // (Sq, H, d) or null
  int64_t q_ss, q_hs;  // byte strides
  int32_t Sq, q_dtype;
  float* e_low;
  float* e_mid;
  float* e_high;
  float* zeta;
  float* e_ac;
  float* energy;
  float* mean;        // (nb, H, d) block mean = DC / sqrt(512), or null
  float* bounds;      // (Sq, nb, H) or null
  float* max_bound;   // (nb, H) or null
  float* q_norm_max;  // (H,) max_s ||q_s|| or null
};

// 16-byte pieces of one token position: the eight chunk values (th) of a
// thread's columns (eight 16-bit or four float32), fetched raw so that no use
// of the loaded words (no wait) sits among the loads
template <int DT>
struct SpRaw {
  static constexpr int COLS = DT == OC_F32 ? 4 : 8;
  u32x4 w[8];
};

// K streams past the caches (32 heads x 32K x 128 in bfloat16 52.9 us with
// plain loads, 48.5 streamed; x 16K in float32 48.2 / 42.1).  The compact
// pipeline's decode, which reads the retained half again, then takes 54 us
// where it took 49, so the two together are level; callers of the spectra
// alone keep the gain.
template <int DT>
__device__ __forceinline__ void sp_fetch(const char* p, int64_t th_stride, SpRaw<DT>& r) {
#pragma unroll
  for (int th = 0; th < 8; ++th)
    r.w[th] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + th * th_stride));
}

// column c of chunk th as float
template <int DT>
__device__ __forceinline__ float sp_elem(const SpRaw<DT>& r, int th, int c) {
  if constexpr (DT == OC_F32) {
    return __uint_as_float(r.w[th][c]);
  } else {
    const uint32_t x = r.w[th][c >> 1];
    if constexpr (DT == OC_BF16) return __uint_as_float((c & 1) ? (x & 0xFFFF0000u) : (x << 16));
    else return (float)__builtin_bit_cast(_Float16, (uint16_t)((c & 1) ? (x >> 16) : (x & 0xFFFFu)));
  }
}

// Energies of one token position's columns and the 8-point transform over the
// chunks th; z0[c] receives Z_0.
template <int DT>
__device__ __forceinline__ void sp_consume(const SpRaw<DT>& r, float& energy, float& e_mid, float& e_high,
                                           float (&z0)[SpRaw<DT>::COLS]) {
#pragma unroll
  for (int c = 0; c < SpRaw<DT>::COLS; ++c) {
    float z[8];
#pragma unroll
    for (int th = 0; th < 8; ++th) {
      z[th] = sp_elem<DT>(r, th, c);
      energy = __builtin_fmaf(z[th], z[th], energy);
    }
    // natural-order 8-point Walsh-Hadamard transform over th (unnormalised)
#pragma unroll
    for (int m = 1; m < 8; m <<= 1)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (!(i & m)) {
          const float u = z[i], v = z[i + m];
          z[i] = u + v;
          z[i + m] = u - v;
        }
#pragma unroll
    for (int uh = 1; uh < 4; ++uh) e_mid = __builtin_fmaf(z[uh], z[uh], e_mid);
#pragma unroll
    for (int uh = 4; uh < 8; ++uh) e_high = __builtin_fmaf(z[uh], z[uh], e_high);
    z0[c] = z[0];
    asm volatile("" : "+v"(z0[c]), "+v"(energy), "+v"(e_mid), "+v"(e_high));  // column by column: few live registers
  }
}

__device__ __forceinline__ float block_max(float v, float* sh_red) {
  v = wave_max(v);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh_red[w] = v;
  __syncthreads();
  float s = sh_red[0];
  for (int i = 1; i < kSpThreads / 64; ++i) s = fmaxf(s, sh_red[i]);
  return s;
}

// a q element's raw bits (zero-extended 16-bit, or float32) and its value
__device__ __forceinline__ float sp_q_value(uint32_t bits, int dtype) {
  if (dtype == OC_F32) return __uint_as_float(bits);
  if (dtype == OC_BF16) return __uint_as_float(bits << 16);
  return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}

// The band energies of one (block, head) from its four sums, written by one thread.
__device__ __forceinline__ float sp_write(const SpecArgs& a, int64_t o, float mid, float high, float low, float energy,
                                          bool write) {
  const float s_mid = mid * 0.125f;
  const float s_high = high * 0.125f;
  const float s_ac = low + s_mid + s_high;
  if (write) {
    if (a.e_low) a.e_low[o] = low;
    if (a.e_mid) a.e_mid[o] = s_mid;
    if (a.e_high) a.e_high[o] = s_high;
    if (a.zeta) a.zeta[o] = s_high / (low + 1e-6f);
    if (a.e_ac) a.e_ac[o] = s_ac;
    if (a.energy) a.energy[o] = energy;
  }
  return s_ac;
}

// Eight consecutive elements of a q row, raw: 16-byte loads where every row
// allows them, else element by element.
__device__ __forceinline__ void sp_q8(const char* p, int dtype, bool vec, u32x4 (&r)[2]) {
  if (vec) {
    r[0] = *reinterpret_cast<const u32x4*>(p);
    if (dtype == OC_F32) r[1] = *reinterpret_cast<const u32x4*>(p + 16);
  } else if (dtype == OC_F32) {
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i >> 2][i & 3] = reinterpret_cast<const uint32_t*>(p)[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint16_t* e = reinterpret_cast<const uint16_t*>(p) + 2 * i;
      r[0][i] = (uint32_t)e[0] | ((uint32_t)e[1] << 16);
    }
  }
}

// element c of them as float
__device__ __forceinline__ float sp_q8_value(const u32x4 (&r)[2], int dtype, int c) {
  if (dtype == OC_F32) return __uint_as_float(r[c >> 2][c & 3]);
  const uint32_t x = r[0][c >> 1];
  return sp_q_value((c & 1) ? (x >> 16) : (x & 0xFFFFu), dtype);
}

// head_dim 64 and 128: one workgroup per (head, block), HBM-bound.  A thread
// keeps its positions' Z_0 in registers, so the workgroup needs no Z_0 in LDS
// and stays below 128 registers a thread (16 wavefronts per CU).  With Z_0 in
// LDS and the 64-point transform done by half the threads, at 12 wavefronts,
// 32 heads x 32K x 128 took 53.3 us in bfloat16 and x 16K in float32 52.7, now
// 48.5 (5.5 TB/s) and 42.1 (6.4 TB/s).  Resident workgroups that walk over the
// blocks, the next one's loads in flight over the reductions, were slower
// (58-61 us).
template <int DT, int D>
__global__ __launch_bounds__(kSpThreads, 4) void block_spectrum_kernel(const SpecArgs a) {
  constexpr int COLS = SpRaw<DT>::COLS;
  constexpr int CG = D / COLS;          // threads side by side over a token row (whole rows per instruction)
  constexpr int TG = kSpThreads / CG;   // token positions at once
  constexpr int TPT = 64 / TG;          // positions per thread
  constexpr int WAVES = kSpThreads / 64;
  static_assert(CG >= 8 && CG <= 32 && TPT >= 2, "lane layout of the column sums");
  __shared__ float sh_col[WAVES][D];  // column sums of Z_0 per wave
  __shared__ float sh_mean[D];
  __shared__ float sh_sum[WAVES][4];
  __shared__ float sh_red[WAVES];
  const int tid = threadIdx.x;
  const int cg = tid % CG;
  const int tg = tid / CG;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  // consecutive workgroups take the heads of one block, so the workgroups
  // in flight together read whole token rows of the (S, H, d) cache
  const int h = blockIdx.x;
  const int blk = blockIdx.y;
  const char* kb = a.k + (int64_t)blk * kBlock * a.k_ts + (int64_t)h * a.k_hs + (int64_t)cg * 16 + (int64_t)tg * a.k_ts;
  // the bounds: D / 8 lanes per query, eight columns each; the wave's first
  // queries are requested before the block streams in
  constexpr int LPQ = D / 8, QPW = 64 / LPQ;
  const int qc = (lane % LPQ) * 8;
  const int qs = wave * QPW + lane / LPQ;
  const int qes = a.q_dtype == OC_F32 ? 4 : 2;
  const bool q_vec = (((uintptr_t)a.q | (uintptr_t)a.q_ss | (uintptr_t)a.q_hs) & 15) == 0;
  u32x4 q0[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
  const char* qbase = a.q + (int64_t)h * a.q_hs + (int64_t)qc * qes;
  if (a.q && qs < a.Sq) sp_q8(qbase + (int64_t)qs * a.q_ss, a.q_dtype, q_vec, q0);
  const int64_t th_stride = 64 * a.k_ts;
  SpRaw<DT> rb[2];
  sp_fetch<DT>(kb, th_stride, rb[0]);
  // the next position's loads are issued before the current one is consumed
  float e_mid = 0.f, e_high = 0.f, energy = 0.f;
  float z0[TPT][COLS];
#pragma unroll
  for (int i = 0; i < TPT; ++i) {
    if (i + 1 < TPT) sp_fetch<DT>(kb + (int64_t)((i + 1) * TG) * a.k_ts, th_stride, rb[(i + 1) & 1]);
    sp_consume<DT>(rb[i & 1], energy, e_mid, e_high, z0[i]);
    // the next position but one is not requested before this one is finished
    // (else the compiler requests every position at once and spills)
    asm volatile("" : : : "memory");
  }
  // column sums over tl, in pairs throughout (a constant column's mean, and
  // with it E_low = 0, is then exact): the thread's positions, the wave's
  // lanes of the same columns, the waves
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    float t[TPT];
#pragma unroll
    for (int i = 0; i < TPT; ++i) t[i] = z0[i][c];
#pragma unroll
    for (int m = 1; m < TPT; m <<= 1)
#pragma unroll
      for (int i = 0; i < TPT; ++i)
        if (!(i & (2 * m - 1))) t[i] += t[i + m];
    float x = t[0], lo, hi;
    if constexpr (CG == 8) x += dpp<0x128>(x);  // row_ror:8
    if constexpr (CG <= 16) {
      row_pair<16>(x, lo, hi);
      x = lo + hi;
    }
    row_pair<32>(x, lo, hi);
    x = lo + hi;
    if (lane < CG) sh_col[wave][lane * COLS + c] = x;
  }
  __syncthreads();
  auto col_sum = [&](int c) { return (sh_col[0][c] + sh_col[1][c]) + (sh_col[2][c] + sh_col[3][c]); };
  if (tid < D) {
    const float m = col_sum(tid) * (1.0f / 512.0f);  // DC / sqrt(512) with DC = sum_t k_t / sqrt(512)
    sh_mean[tid] = m;
    if (a.mean) a.mean[((int64_t)blk * a.H + h) * D + tid] = m;
  }
  float e_low = 0.f;
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    const float m = col_sum(cg * COLS + c) * (1.0f / 64.0f);
#pragma unroll
    for (int i = 0; i < TPT; ++i) {
      const float x = z0[i][c] - m;
      e_low = __builtin_fmaf(x, x, e_low);
    }
  }
  // the four band sums in one reduction: lanes, then the four waves in LDS
  float r4[4] = {e_mid, e_high, e_low, energy};
#pragma unroll
  for (int j = 0; j < 4; ++j) r4[j] = wave_sum(r4[j]);
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) sh_sum[wave][j] = r4[j];
  }
  __syncthreads();  // also: sh_mean complete
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r4[j] = sh_sum[0][j];
    for (int w = 1; w < WAVES; ++w) r4[j] += sh_sum[w][j];
  }
  if (__builtin_isnan(r4[2])) {
    // K that is not finite (uniform over the workgroup): the transform's rows
    // 1..63 of a column with one infinity are all infinite, of one with more,
    // or with a NaN, some are NaN; without its mean both are NaN
    int* cnt = reinterpret_cast<int*>(&sh_col[0][0]);
    if (tid < D) cnt[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < COLS; ++c)
#pragma unroll
      for (int i = 0; i < TPT; ++i)
        if (!__builtin_isfinite(z0[i][c])) atomicAdd(&cnt[cg * COLS + c], __builtin_isnan(z0[i][c]) ? 2 : 1);
    __syncthreads();
    bool nan = false;
    for (int c = 0; c < D; ++c) nan = nan || cnt[c] > 1;
    r4[2] = nan ? __builtin_nanf("") : __builtin_inff();
  }
  const int64_t o = (int64_t)blk * a.H + h;
  const float s_ac = sp_write(a, o, r4[0], r4[1], r4[2] * 0.125f, r4[3], tid == 0);  // 64 / 512
  if (!a.q) return;
  // query-aware bounds: (q . mean + ||q|| sqrt(E_ac)) / sqrt(d)
  const float inv_sd = 1.0f / __builtin_sqrtf((float)D);
  const float sq_ac = __builtin_sqrtf(fmaxf(s_ac, 0.f));
  float mean[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) mean[c] = sh_mean[qc + c];
  float best = -__builtin_inff();
  float qbest = 0.f;
  for (int s = qs; s < a.Sq; s += WAVES * QPW) {
    if (s != qs) sp_q8(qbase + (int64_t)s * a.q_ss, a.q_dtype, q_vec, q0);
    float dot = 0.f, nn = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float qv = sp_q8_value(q0, a.q_dtype, c);
      dot = __builtin_fmaf(qv, mean[c], dot);
      nn = __builtin_fmaf(qv, qv, nn);
    }
    // (the lanes of one query leave the loop together)
    if constexpr (LPQ == 16) {
      dot += xpair<8>(dot);
      nn += xpair<8>(nn);
    }
    dot += xpair<4>(dot);
    nn += xpair<4>(nn);
    dot += xpair<2>(dot);
    nn += xpair<2>(nn);
    dot += xpair<1>(dot);
    nn += xpair<1>(nn);
    const float qn = __builtin_sqrtf(nn);
    const float bnd = dot * inv_sd + qn * sq_ac * inv_sd;
    if (a.bounds && qc == 0) a.bounds[((int64_t)s * a.nb + blk) * a.H + h] = bnd;
    best = fmaxf(best, bnd);
    qbest = fmaxf(qbest, qn);
  }
  best = block_max(best, sh_red);
  if (tid == 0 && a.max_bound) a.max_bound[o] = best;
  if (blk == 0 && a.q_norm_max) {
    qbest = block_max(qbest, sh_red);
    if (tid == 0) a.q_norm_max[h] = qbest;
  }
}

// Any other head_dim (a multiple of 8 up to kMaxD).
template <int DT>
__global__ __launch_bounds__(kSpThreads) void block_spectrum_any_kernel(const SpecArgs a) {
  constexpr int DMAX = kMaxD;
  constexpr int COLS = SpRaw<DT>::COLS;
  // Z_0[tl][c]; once the transform has read it (after the barrier that
  // follows), row 0 holds the block mean (each thread writes its own
  // column) and entries d .. d + 20 the reduction scratch, so the whole
  // workgroup's LDS is 32 KiB at d = 128 (five workgroups per CU)
  __shared__ float sh_z[64 * DMAX];
  float* sh_mean = sh_z;
  float (*sh_sum)[4] = reinterpret_cast<float (*)[4]>(sh_z + a.d);
  float* sh_red = sh_z + a.d + 4 * (kSpThreads / 64);
  // consecutive workgroups take the heads of one block, so the workgroups
  // in flight together read whole token rows of the (S, H, d) cache
  const int h = blockIdx.x;
  const int blk = blockIdx.y;
  const int d = a.d;
  const int CG = d / COLS;
  const int TG = kSpThreads / CG;
  const int tid = threadIdx.x;
  const int cg = tid % CG;
  const int tg = tid / CG;
  const char* kb = a.k + (int64_t)blk * kBlock * a.k_ts + (int64_t)h * a.k_hs + (int64_t)cg * 16;
  // the bounds: wave w takes queries w, w + 4, ..., lane l columns l, l + 64, ...;
  // the wave's first query is requested before the block streams in
  constexpr int QPL = (DMAX + 63) / 64;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  // raw bits, converted where used: columns past d read column d - 1 (in
  // bounds) and are zeroed at the conversion
  auto load_q = [&](int s, uint32_t (&qr_bits)[QPL]) {
    const char* qr = a.q + (int64_t)s * a.q_ss + (int64_t)h * a.q_hs;
    if (a.q_dtype == OC_F32) {
#pragma unroll
      for (int k = 0; k < QPL; ++k)
        qr_bits[k] = *reinterpret_cast<const uint32_t*>(qr + (int64_t)min(lane + 64 * k, d - 1) * 4);
    } else {
#pragma unroll
      for (int k = 0; k < QPL; ++k)
        qr_bits[k] = *reinterpret_cast<const uint16_t*>(qr + (int64_t)min(lane + 64 * k, d - 1) * 2);
    }
  };
  uint32_t q0[QPL];
#pragma unroll
  for (int k = 0; k < QPL; ++k) q0[k] = 0u;
  if (a.q && wave < a.Sq) load_q(wave, q0);
  float e_mid = 0.f, e_high = 0.f, energy = 0.f;
  const int64_t th_stride = 64 * a.k_ts;
  if (tg < TG) {
    // positions tg, tg + TG, ... < 64; the threads past TG * CG (when CG does
    // not divide 256) take none
    for (int tl = tg; tl < 64; tl += TG) {
      SpRaw<DT> r;
      float z0[COLS];
      sp_fetch<DT>(kb + (int64_t)tl * a.k_ts, th_stride, r);
      sp_consume<DT>(r, energy, e_mid, e_high, z0);
#pragma unroll
      for (int c = 0; c < COLS; ++c) sh_z[tl * d + COLS * cg + c] = z0[c];
    }
  }
  __syncthreads();
  // 64-point transform of Z_0 along tl, one column per thread
  float e_low = 0.f;
  if (tid < d) {
    float y[64];
#pragma unroll
    for (int i = 0; i < 64; ++i) y[i] = sh_z[i * d + tid];  // consecutive threads, consecutive words
#pragma unroll
    for (int m = 1; m < 64; m <<= 1)
#pragma unroll
      for (int i = 0; i < 64; ++i)
        if (!(i & m)) {
          const float u = y[i], v = y[i + m];
          y[i] = u + v;
          y[i + m] = u - v;
        }
#pragma unroll
    for (int i = 1; i < 64; ++i) e_low = __builtin_fmaf(y[i], y[i], e_low);
    sh_mean[tid] = y[0] * (1.0f / 512.0f);  // DC / sqrt(512) with DC = sum_t k_t / sqrt(512)
  }
  // the four band sums in one reduction: lanes, then the four waves in LDS
  float r4[4] = {e_mid, e_high, e_low, energy};
#pragma unroll
  for (int j = 0; j < 4; ++j) r4[j] = wave_sum(r4[j]);
  __syncthreads();  // every column of Z_0 has been read: the scratch entries are free
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) sh_sum[wave][j] = r4[j];
  }
  __syncthreads();  // also: sh_mean complete
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r4[j] = sh_sum[0][j];
    for (int w = 1; w < kSpThreads / 64; ++w) r4[j] += sh_sum[w][j];
  }
  const int64_t o = (int64_t)blk * a.H + h;
  const float s_ac = sp_write(a, o, r4[0], r4[1], r4[2] * (1.0f / 512.0f), r4[3], tid == 0);
  if (a.mean && tid < d) a.mean[o * d + tid] = sh_mean[tid];
  if (!a.q) return;
  // query-aware bounds: (q . mean + ||q|| sqrt(E_ac)) / sqrt(d)
  const float inv_sd = 1.0f / __builtin_sqrtf((float)d);
  const float sq_ac = __builtin_sqrtf(fmaxf(s_ac, 0.f));
  float best = -__builtin_inff();
  float qbest = 0.f;
  for (int s = wave; s < a.Sq; s += kSpThreads / 64) {
    uint32_t qb[QPL];
    if (s == wave) {
#pragma unroll
      for (int k = 0; k < QPL; ++k) qb[k] = q0[k];
    } else {
      load_q(s, qb);
    }
    float dot = 0.f, nn = 0.f;
#pragma unroll
    for (int k = 0; k < QPL; ++k) {
      const int c = lane + 64 * k;
      if (c < d) {
        const float qv = sp_q_value(qb[k], a.q_dtype);
        dot = __builtin_fmaf(qv, sh_mean[c], dot);
        nn = __builtin_fmaf(qv, qv, nn);
      }
    }
    dot = wave_sum(dot);
    nn = wave_sum(nn);
    const float qn = __builtin_sqrtf(nn);
    const float bnd = dot * inv_sd + qn * sq_ac * inv_sd;
    if (a.bounds && lane == 0) a.bounds[((int64_t)s * a.nb + blk) * a.H + h] = bnd;
    best = fmaxf(best, bnd);
    qbest = fmaxf(qbest, qn);
  }
  best = block_max(best, sh_red);
  if (tid == 0 && a.max_bound) a.max_bound[o] = best;
  if (blk == 0 && a.q_norm_max) {
    qbest = block_max(qbest, sh_red);
    if (tid == 0) a.q_norm_max[h] = qbest;
  }
}

constexpr int kGateLds = 2048;   // (block, head) entries staged in LDS by the gate kernel
constexpr int kGateHeads = 256;  // query norms staged with them
constexpr int kGateBlocks = 2048;  // blocks whose per-block results the gate kernel keeps in LDS
constexpr int kGateWaves = 16;

// N values reduced over the 1024-thread workgroup at once: a DPP reduction
// per wave, then the 16 wave results from LDS (bit j of max_mask: maximum,
// else sum; identical result in every thread, fixed order).
template <int N>
__device__ __forceinline__ void gate_reduce(float (&v)[N], unsigned max_mask, float (*sh)[8]) {
  static_assert(N <= 8, "at most eight values per reduction");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] = ((max_mask >> j) & 1) ? wave_max(v[j]) : wave_sum(v[j]);
  __syncthreads();  // the previous reduction's reads of sh are done
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < N; ++j) sh[wave][j] = v[j];
  }
  __syncthreads();
  // every wave combines the 16 results over the lanes of its rows (read one
  // by one by all 1024 threads, the LDS reads were most of the reduction)
#pragma unroll
  for (int j = 0; j < N; ++j) {
    float t = sh[lane & (kGateWaves - 1)][j];
    if ((max_mask >> j) & 1) {
      t = fmaxf(t, xpair<8>(t));
      t = fmaxf(t, xpair<4>(t));
      t = fmaxf(t, xpair<2>(t));
      t = fmaxf(t, xpair<1>(t));
    } else {
      t = row16_sum(t);
    }
    v[j] = t;
  }
}

// The compact pipeline's gates and statistics in one workgroup over the
// (block, head) table (pipeline.py:458-527): tau (given, or mean - unbiased
// std of the max bounds), the two-gate mask, the any-head block mask and its
// tile expansion, the zeta statistics of the per-block head means, the
// retained count, the largest retained bound and the perfect / statistical
// regimes of the evicted blocks.  stats: [tau, zeta mean, zeta std, zeta
// min, zeta max, retained, perfect, statistical, z_max].
//
// STAGED: at most kGateLds entries and kGateHeads heads, and the tables are
// read from LDS.  Latency-bound: the masks are stored once per-block results
// are in LDS, for a wait for any of the loop's reads is one for its earlier
// stores too (64 blocks of 32 heads: 9.8 us with the stores in the loop and
// reads that may go to either memory, 6.0 now).
template <bool STAGED>
__global__ __launch_bounds__(1024) void compact_gate_kernel(const float* mb, const float* zeta, const float* energy,
                                                            const float* qmax, int nb, int H, int d, float tau_in,
                                                            int tau_auto, float zeta_max, float underflow,
                                                            int tiles_per_block, uint8_t* unified,
                                                            uint8_t* tile_mask, float* stats) {
  __shared__ float sh_f[kGateWaves][8];
  // the (block, head) tables and the query norms, every load in flight at once
  __shared__ float sh_mb[STAGED ? kGateLds : 1], sh_zeta[STAGED ? kGateLds : 1], sh_en[STAGED ? kGateLds : 1],
      sh_qmax[STAGED ? kGateHeads : 1];
  // per-block results of the first pass (any head kept, head-mean zeta, beta)
  __shared__ float sh_za[kGateBlocks], sh_beta[kGateBlocks];
  __shared__ uint8_t sh_any[kGateBlocks];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int n = nb * H;
  const bool cache_blk = STAGED || nb <= kGateBlocks;
  if constexpr (STAGED) {
#pragma unroll
    for (int k = 0; k < kGateLds / 1024; ++k) {
      const int i = tid + 1024 * k;
      if (i < n) {
        sh_mb[i] = mb[i];
        sh_zeta[i] = zeta[i];
        sh_en[i] = energy[i];
      }
    }
    if (tid < H) sh_qmax[tid] = qmax[tid];
    __syncthreads();
  }
  auto mb_at = [&](int64_t i) { return STAGED ? sh_mb[STAGED ? i : 0] : mb[i]; };
  auto zeta_at = [&](int64_t i) { return STAGED ? sh_zeta[STAGED ? i : 0] : zeta[i]; };
  auto energy_at = [&](int64_t i) { return STAGED ? sh_en[STAGED ? i : 0] : energy[i]; };
  auto qmax_at = [&](int64_t i) { return STAGED ? sh_qmax[STAGED ? i : 0] : qmax[i]; };
  float tau = tau_in;
  if (tau_auto) {
    float s[1] = {0.f};
    for (int i = tid; i < n; i += 1024) s[0] += mb_at(i);
    gate_reduce<1>(s, 0u, sh_f);
    const float mean = s[0] / (float)n;
    float v[1] = {0.f};
    for (int i = tid; i < n; i += 1024) v[0] = __builtin_fmaf(mb_at(i) - mean, mb_at(i) - mean, v[0]);
    gate_reduce<1>(v, 0u, sh_f);
    const float var = v[0] / (float)(n - 1);  // n = 1: NaN, as torch.std
    tau = mean - __builtin_sqrtf(var);
  }
  // per block (one 16-lane row per block, lanes over heads; a wave per block
  // left half its lanes idle at 32 heads and cost 1 us per 16 blocks): any
  // head retained, head-mean zeta, largest bound, beta = max_h qmax_h sqrt(E)
  // / sqrt(d)
  const int j = tid & 15, row = tid >> 4;
  constexpr int kRows = 64;
  auto row_max = [](float x) {
    x = fmaxf(x, xpair<8>(x));
    x = fmaxf(x, xpair<4>(x));
    x = fmaxf(x, xpair<2>(x));
    return fmaxf(x, xpair<1>(x));
  };
  const float isd = 1.0f / __builtin_sqrtf((float)d);
  struct Blk {
    bool any;
    float za, bmx, beta;
  };
  auto block_stats = [&](int b) {
    bool any = false;
    float zsum = 0.f, bmx = -__builtin_inff(), beta = -__builtin_inff();
    for (int h = j; h < H; h += 16) {
      const float m = mb_at((int64_t)b * H + h), z = zeta_at((int64_t)b * H + h);
      any = any || (m >= tau && z <= zeta_max);
      zsum += z;
      bmx = fmaxf(bmx, m);
      beta = fmaxf(beta, qmax_at(h) * __builtin_sqrtf(fmaxf(energy_at((int64_t)b * H + h), 0.f)) * isd);
    }
    return Blk{((__ballot(any) >> (lane & 48)) & 0xFFFFu) != 0, row16_sum(zsum) / (float)H, row_max(bmx),
               row_max(beta)};
  };
  // r1: zeta sum, retained (sums); -zeta min, zeta max, best retained bound (maxima)
  float r1[5] = {0.f, 0.f, -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
  for (int b = row; b < nb; b += kRows) {
    const Blk k = block_stats(b);
    if (!cache_blk)
      for (int t = j; t < tiles_per_block; t += 16) tile_mask[(int64_t)b * tiles_per_block + t] = k.any ? 1 : 0;
    if (j == 0) {
      if (!cache_blk) unified[b] = k.any ? 1 : 0;
      if (cache_blk) {
        sh_any[b] = k.any ? 1 : 0;
        sh_za[b] = k.za;
        sh_beta[b] = k.beta;
      }
      r1[0] += k.za;
      r1[1] += k.any ? 1.f : 0.f;
      r1[2] = fmaxf(r1[2], -k.za);
      r1[3] = fmaxf(r1[3], k.za);
      if (k.any) r1[4] = fmaxf(r1[4], k.bmx);
    }
  }
  gate_reduce<5>(r1, 0x1Cu, sh_f);  // its barriers also publish sh_any / sh_za / sh_beta
  if (cache_blk) {
    for (int b = tid; b < nb; b += 1024) unified[b] = sh_any[b];
    for (int64_t t = tid; t < (int64_t)nb * tiles_per_block; t += 1024) tile_mask[t] = sh_any[t / tiles_per_block];
  }
  const float zmean = r1[0] / (float)nb;
  const float retained = r1[1];
  const float zmin = -r1[2], zmx = r1[3];
  const float zmax_ret = retained == 0.f ? 0.f : r1[4];
  // r2: squared zeta deviations, perfect and statistical evictions
  float r2[3] = {0.f, 0.f, 0.f};
  auto regime = [&](bool any, float za, float beta) {
    r2[0] = __builtin_fmaf(za - zmean, za - zmean, r2[0]);
    if (!any) {
      if (zmax_ret - beta >= underflow) r2[1] += 1.f;
      else r2[2] += 1.f;
    }
  };
  if (cache_blk) {
    for (int b = tid; b < nb; b += 1024) regime(sh_any[b] != 0, sh_za[b], sh_beta[b]);
  } else {
    for (int b = row; b < nb; b += kRows) {
      const Blk k = block_stats(b);
      if (j == 0) regime(k.any, k.za, k.beta);
    }
  }
  gate_reduce<3>(r2, 0u, sh_f);
  if (tid == 0) {
    stats[0] = tau;
    stats[1] = zmean;
    stats[2] = __builtin_sqrtf(r2[0] / (float)(nb - 1));
    stats[3] = zmin;
    stats[4] = zmx;
    stats[5] = retained;
    stats[6] = r2[1];
    stats[7] = r2[2];
    stats[8] = zmax_ret;
  }
}

// NaN-propagating maximum (torch.max semantics): a NaN operand wins
__device__ __forceinline__ float nan_max(float a, float b) { return (a != a || a >= b) ? a : b; }

// Eviction regimes of a block table (perfect_eviction.py:75-186 as
// orthocache_forward and its callers use it), one workgroup:
//   qn[h]   = max_s q_norms[s, h]                       (NaN propagates)
//   b[b, h] = qn[h] * sqrt(E[b, h] clamped at 0) / sqrt_d  (float32, NaN kept)
//   beta[b] = max_h b[b, h];  gap[b] = z - beta[b]
//   regime  = 0 when any of the block's mask entries is set (retained);
//             else 1 when gap >= underflow, 2 when gap < underflow, and 0
//             when gap is NaN (neither compare holds)
// counts = (regime-1 blocks, regime-2 blocks, retained blocks).  z is the
// largest of z_vec[0 .. z_count) when given (NaN propagates), else z_scalar.
__global__ __launch_bounds__(1024) void block_regimes_kernel(const float* qnorms, int sq, int H, const float* energy,
                                                             int nb, float sqrt_d, float z_scalar, const float* z_vec,
                                                             int z_count, const uint8_t* mask, int mask_heads,
                                                             float underflow, int32_t* regime, float* beta,
                                                             float* gap, float* beta_full, int32_t* counts) {
  __shared__ float sh_qn[kGateHeads];
  __shared__ float sh_f[kGateWaves][8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // z: the reduction runs in every wave over the same lanes, so each wave
  // ends with the same value (no barrier needed)
  float z = z_scalar;
  if (z_vec) {
    float m = -__builtin_inff();
    for (int i = lane; i < z_count; i += 64) m = nan_max(m, z_vec[i]);
    for (int o = 32; o > 0; o >>= 1) m = nan_max(m, __shfl_xor(m, o, 64));
    z = m;
  }
  // per-head query norm maxima; heads past the LDS table are re-derived
  // where they are used
  auto head_qmax = [&](int h) {
    float m = -__builtin_inff();
    for (int s = 0; s < sq; ++s) m = nan_max(m, qnorms[(int64_t)s * H + h]);
    return m;
  };
  for (int h = threadIdx.x; h < H && h < kGateHeads; h += 1024) sh_qn[h] = head_qmax(h);
  __syncthreads();
  // one wave per block, lanes over heads
  float cnt[3] = {0.f, 0.f, 0.f};
  for (int b = wave; b < nb; b += kGateWaves) {
    float bm = -__builtin_inff();
    bool kept = false;
    for (int h = lane; h < H; h += 64) {
      const float e = energy[(int64_t)b * H + h];
      const float qn = h < kGateHeads ? sh_qn[h] : head_qmax(h);
      const float x = qn * __builtin_sqrtf(e < 0.f ? 0.f : e) / sqrt_d;
      if (beta_full) beta_full[(int64_t)b * H + h] = x;
      bm = nan_max(bm, x);
      if (mask_heads > 1) kept = kept || mask[(int64_t)b * mask_heads + h] != 0;
    }
    for (int o = 32; o > 0; o >>= 1) bm = nan_max(bm, __shfl_xor(bm, o, 64));
    kept = mask_heads > 1 ? __ballot(kept) != 0 : mask[b] != 0;
    if (lane == 0) {
      const float g = z - bm;
      const int r = kept ? 0 : (g >= underflow ? 1 : (g < underflow ? 2 : 0));
      regime[b] = r;
      beta[b] = bm;
      gap[b] = g;
      cnt[0] += r == 1 ? 1.f : 0.f;
      cnt[1] += r == 2 ? 1.f : 0.f;
      cnt[2] += kept ? 1.f : 0.f;
    }
  }
  gate_reduce<3>(cnt, 0u, sh_f);  // exact: counts below 2^24
  if (threadIdx.x == 0) {
    counts[0] = (int32_t)cnt[0];
    counts[1] = (int32_t)cnt[1];
    counts[2] = (int32_t)cnt[2];
  }
}

// Active-first stable order of n blocks (stream compaction): out[r] = the
// r-th retained block, then the evicted ones in order; *num_active = the
// retained count.  One workgroup of 1024 threads, chunked prefix sums.
__global__ __launch_bounds__(1024) void stream_compact_kernel(const uint8_t* mask, int n, int64_t* out,
                                                              int32_t* num_active) {
  __shared__ int sh[1024];
  __shared__ int sh_total;
  const int tid = threadIdx.x;
  int cnt = 0;
  for (int i = tid; i < n; i += 1024) cnt += mask[i] ? 1 : 0;
  for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
  if (tid == 0) sh_total = 0;
  __syncthreads();
  if ((tid & 63) == 0) atomicAdd(&sh_total, cnt);
  __syncthreads();
  const int total = sh_total;
  int base_a = 0;
  for (int c0 = 0; c0 < n; c0 += 1024) {
    const int i = c0 + tid;
    const int f = (i < n && mask[i]) ? 1 : 0;
    sh[tid] = f;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {  // inclusive Hillis-Steele scan
      const int v = tid >= off ? sh[tid - off] : 0;
      __syncthreads();
      sh[tid] += v;
      __syncthreads();
    }
    const int incl = sh[tid];
    const int chunk_a = sh[1023];
    if (i < n) {
      const int ra = base_a + incl - f;           // retained before i
      const int r = f ? ra : total + (i - ra);     // evicted before i: i - ra
      out[r] = i;
    }
    base_a += chunk_a;
    __syncthreads();
  }
  if (tid == 0 && num_active) *num_active = total;
}

template <int DT>
int launch_spectrum(const SpecArgs& a, hipStream_t s) {
  if (a.d == 128)
    hipLaunchKernelGGL((block_spectrum_kernel<DT, 128>), dim3(a.H, a.nb), dim3(kSpThreads), 0, s, a);
  else if (a.d == 64)
    hipLaunchKernelGGL((block_spectrum_kernel<DT, 64>), dim3(a.H, a.nb), dim3(kSpThreads), 0, s, a);
  else
    hipLaunchKernelGGL(block_spectrum_any_kernel<DT>, dim3(a.H, a.nb), dim3(kSpThreads), 0, s, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? OC_OK : hip_fail(e, "block-spectrum launch");
}

}  // namespace
}  // namespace oc

using namespace oc;

extern "C" int oc_block_spectra(const oc_spectra_params* p, void* stream) {
  if (!p || !p->k) return fail(OC_ERR_INVALID, "NULL pointer");
  if (p->dtype != OC_F32 && p->dtype != OC_F16 && p->dtype != OC_BF16) return fail(OC_ERR_INVALID, "dtype %d", p->dtype);
  if (p->block_size != kBlock) return fail(OC_ERR_UNSUPPORTED, "block_size %d (the transform is 512-point)", p->block_size);
  if (p->head_dim < 8 || p->head_dim > kMaxD || p->head_dim % 8)
    return fail(OC_ERR_UNSUPPORTED, "head_dim %d (a multiple of 8 up to %d)", p->head_dim, kMaxD);
  if (p->num_blocks < 0 || p->num_heads < 0 || p->q_len < 0) return fail(OC_ERR_INVALID, "bad sizes");
  const int es = p->dtype == OC_F32 ? 4 : 2;
  if ((p->k_token_stride * es) % 16 || (p->k_head_stride * es) % 16 || ((uintptr_t)p->k % 16))
    return fail(OC_ERR_INVALID, "K rows must be 16-byte aligned");
  if (p->q && p->q_dtype != OC_F32 && p->q_dtype != OC_F16 && p->q_dtype != OC_BF16)
    return fail(OC_ERR_INVALID, "q dtype %d", p->q_dtype);
  if ((p->bounds || p->max_bound || p->q_norm_max) && !p->q) return fail(OC_ERR_INVALID, "bounds need q");
  if (p->num_blocks == 0 || p->num_heads == 0) return OC_OK;
  if (p->num_blocks > 65535) return fail(OC_ERR_UNSUPPORTED, "num_blocks > 65535 (33553920 tokens)");
  SpecArgs a{};
  a.k = (const char*)p->k;
  a.k_ts = p->k_token_stride * es, a.k_hs = p->k_head_stride * es;
  a.H = p->num_heads, a.d = p->head_dim, a.nb = p->num_blocks, a.dtype = p->dtype;
  a.q = (const char*)p->q;
  const int qes = p->q_dtype == OC_F32 ? 4 : 2;
  a.q_ss = p->q_token_stride * qes, a.q_hs = p->q_head_stride * qes;
  a.Sq = p->q ? p->q_len : 0;
  a.q_dtype = p->q_dtype;
  a.e_low = p->e_low, a.e_mid = p->e_mid, a.e_high = p->e_high, a.zeta = p->zeta;
  a.e_ac = p->e_ac, a.energy = p->energy, a.mean = p->block_mean;
  a.bounds = p->bounds, a.max_bound = p->max_bound, a.q_norm_max = p->q_norm_max;
  const hipStream_t s = (hipStream_t)stream;
  switch (p->dtype) {
    case OC_F32: return launch_spectrum<OC_F32>(a, s);
    case OC_F16: return launch_spectrum<OC_F16>(a, s);
    default: return launch_spectrum<OC_BF16>(a, s);
  }
}

extern "C" int oc_stream_compact(const uint8_t* block_mask, int32_t num_blocks, int64_t* indices,
                                 int32_t* num_active, void* stream) {
  if (!block_mask || !indices) return fail(OC_ERR_INVALID, "NULL pointer");
  if (num_blocks < 0) return fail(OC_ERR_INVALID, "bad sizes");
  if (num_blocks == 0) return OC_OK;
  hipLaunchKernelGGL(stream_compact_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, block_mask, num_blocks,
                     indices, num_active);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? OC_OK : hip_fail(e, "stream-compact launch");
}

extern "C" int oc_compact_gate(const float* max_bound, const float* zeta, const float* energy, const float* q_norm_max,
                               int32_t num_blocks, int32_t num_heads, int32_t head_dim, double tau, int32_t tau_auto,
                               double zeta_max, double underflow, int32_t tiles_per_block, uint8_t* block_mask,
                               uint8_t* tile_mask, float* stats, void* stream) {
  if (!max_bound || !zeta || !energy || !q_norm_max || !block_mask || !tile_mask || !stats)
    return fail(OC_ERR_INVALID, "NULL pointer");
  if (num_blocks < 1 || num_heads < 1 || head_dim < 1 || tiles_per_block < 1) return fail(OC_ERR_INVALID, "bad sizes");
  const bool staged = (int64_t)num_blocks * num_heads <= kGateLds && num_heads <= kGateHeads;
  hipLaunchKernelGGL(staged ? compact_gate_kernel<true> : compact_gate_kernel<false>, dim3(1), dim3(1024), 0,
                     (hipStream_t)stream, max_bound, zeta, energy, q_norm_max, num_blocks, num_heads, head_dim, (float)tau, tau_auto, (float)zeta_max,
                     (float)underflow, tiles_per_block, block_mask, tile_mask, stats);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? OC_OK : hip_fail(e, "compact-gate launch");
}

extern "C" int oc_block_regimes(const float* q_norms, int32_t q_len, int32_t num_heads, const float* energy,
                                int32_t num_blocks, int32_t head_dim, double z_max, const float* z_values,
                                int32_t z_count, const uint8_t* block_mask, int32_t mask_heads, double underflow,
                                int32_t* regime, float* beta, float* gap, float* beta_full, int32_t* counts,
                                void* stream) {
  if (!q_norms || !energy || !block_mask || !regime || !beta || !gap || !counts)
    return fail(OC_ERR_INVALID, "NULL pointer");
  if (q_len < 1 || num_heads < 1 || num_blocks < 0 || head_dim < 1 || (z_values && z_count < 1))
    return fail(OC_ERR_INVALID, "bad sizes");
  if (mask_heads != 1 && mask_heads != num_heads)
    return fail(OC_ERR_INVALID, "mask_heads %d must be 1 or num_heads %d", mask_heads, num_heads);
  if (num_blocks >= (1 << 24)) return fail(OC_ERR_UNSUPPORTED, "num_blocks %d >= 2^24", num_blocks);
  // the divisor as the reference forms it: math.sqrt(head_dim) taken to float32
  const float sqrt_d = (float)std::sqrt((double)head_dim);
  hipLaunchKernelGGL(block_regimes_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, q_norms, q_len, num_heads,
                     energy, num_blocks, sqrt_d, (float)z_max, z_values, z_count, block_mask, mask_heads,
                     (float)underflow, regime, beta, gap, beta_full, counts);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? OC_OK : hip_fail(e, "block-regimes launch");
}

extern "C" size_t oc_spectra_params_bytes(void) { return sizeof(oc_spectra_params); }
