// tq_q16.h -- the MSE quantizer of bf16 / fp16 rows of 64 or 128 dims, a wave per 16 rows,
// shared by the kernels that write its codes as bit planes, into a cache or into pools.
//
// What is computed is quantize_kernel<false>'s result bit for bit: n = round(||x||),
// u = round(x / max(n, eps)), y_j = the fp32 sum of u_k R_jk (R rounded to the input type)
// by fused multiply-adds in increasing k, code = #{boundary < round(y_j)}.  A wave forms y
// on v_mfma_f32_16x16x32_{bf16,f16} (exact products, fp32 sums in another order) and
// compares it with the fp32 thresholds T_i for which round(y) > boundary_i <=> y > T_i.  Both
// sums lie within  (d + 33 d/32) 2^-24 ||u|| ||R_j||  of each other: the sequential sum's error is
// at most 2^-24 of every partial sum, each at most ||u|| ||R_j|| (Cauchy-Schwarz), the matrix
// cores' at most 2^-24 of the largest addend for each of an instruction's 33 (measured: up
// to 16 an instruction).  A coordinate whose y is farther than that from every threshold has
// its code; the others (about one in 1,000) are summed again in the sequential order, a
// lane each.
//
// Why: the fp32 rotation of 16-bit rows on the vector ALUs took 422 us for 262,147 rows of
// 128 dims (20 TFLOP/s; the rows themselves are 84 MB, 17 us at a copy's rate).
#pragma once

#include "tq_common.h"

#include <type_traits>

namespace tq {
namespace q16 {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8hf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v8f __attribute__((ext_vector_type(8)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

// Waves per workgroup: with D = 128 the R operand (128 registers) stays in LDS, and two
// workgroups of eight waves share a CU; with D = 64 its 32 registers are held.
template <int D> constexpr int waves() { return D == 128 ? 8 : 4; }
constexpr int kCells = 64;     // cells of the threshold table
constexpr int kCopies = 32;    // its copies: lanes l and l + 32 share one, conflict-free
constexpr float kMargin = 0.05f;

// One matrix's tables.  cell(y) = round(clamp(v(y), 0, 63)) with v(y) = y s + off, monotone in
// y.  A cell's entry is its threshold, the one, if any, whose v lies in the cell or within
// kMargin of it (NaN for none), with the number of lower thresholds in the last four
// mantissa bits: those are below every y of the cell, the other thresholds above, all by at
// least about kMargin / s.  A y within 2^-19 |T| of T counts as undecided, which covers the
// mantissa bits.
template <int D>
struct Lds {
  // R rounded to the input type, row j at at(j).  Sixteen lanes read rows 4 ct + r + 32 i
  // (i, r = 0..3) or 16 ct + m: either way the 16 rows start on 16 distinct bank quads.
  alignas(16) uint16_t r[D * (D + 8) + 96];
  static __device__ __forceinline__ int at(int j) { return j * (D + 8) + 32 * (j / (D / 4)); }
  uint32_t lut[kCells][kCopies];
  float thr[16];                       // T_i
  float bnd[16];                       // boundaries rounded to the input type
  float rr[D];                         // ||R_j||^2
  uint32_t shared_cell;                // a cell with two thresholds: the table is not used
  uint32_t irregular;                  // unsorted or non-finite boundaries: every code exact
};
// A wave's unit rows, for the sequential sums.
template <int D>
struct WaveLds {
  alignas(16) uint16_t u[16][D + 8];
};

template <bool BF>
__device__ __forceinline__ float widen(uint32_t h) {
  if constexpr (BF) return __uint_as_float(h << 16);
  else return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// The largest fp32 y whose rounding to the 16-bit type is not above b: midway to the next
// value up where the tie goes to b (b's last bit even), just below the midpoint otherwise.
template <bool BF>
__device__ __forceinline__ float threshold_of(float b) {
  uint32_t h;  // b's 16 bits
  if constexpr (BF) h = __float_as_uint(b) >> 16;
  else h = __builtin_bit_cast(uint16_t, (_Float16)b);
  if ((h & 0x7fffu) == 0) h = 0;  // -0
  const uint32_t up = (h & 0x8000u) ? (h == 0x8001u ? 0u : h - 1) : h + 1;
  const float mid = 0.5f * (widen<BF>(h) + widen<BF>(up));
  if ((h & 1u) == 0) return mid;
  const uint32_t m = __float_as_uint(mid);  // mid != 0: only h = 0 has a zero neighbour below
  if ((m & 0x7fffffffu) == 0) return -1e-45f;
  return __uint_as_float((m & 0x80000000u) ? m + 1 : m - 1);
}

// cell(y) = v(y) rounded to an integer and clamped to 0..63, from the low bits of
// y s + off + 1.5 2^23 (off a whole number).
struct Map {
  static constexpr float kMagic = 12582912.f;
  float s, off;
  __device__ __forceinline__ float v(float y) const { return fmaf(y, s, off); }
  // byte offset of the cell's entry in a copy; lane_off = 4 (lane % kCopies)
  __device__ __forceinline__ uint32_t entry(float y, uint32_t lane_off) const {
    const float c = __builtin_amdgcn_fmed3f(fmaf(y, s, off + kMagic), kMagic, kMagic + 63.f);
    return (__float_as_uint(c) - __float_as_uint(kMagic)) * (4 * kCopies) + lane_off;
  }
};

// Output column of D tile row m = 4 g + r of column tile ct.  ROWS: lane group g holds the
// D/4 consecutive dims D/4 g + 4 ct + r; else the dims 16 ct + 4 g + r (r = 0..3).
template <int D, bool ROWS>
__device__ __forceinline__ int column(int ct, int m) {
  return ROWS ? (D / 4) * (m >> 2) + 4 * ct + (m & 3) : 16 * ct + m;
}

template <int D, bool BF, bool ROWS>
struct Quantizer {
  static constexpr int KS = D / 32, CT = D / 16;
  using v8 = typename std::conditional<BF, v8bf, v8hf>::type;
  static constexpr int DT = BF ? TQ_BF16 : TQ_F16;
  static constexpr bool kHold = D == 64;
  static constexpr int W = waves<D>(), kThreads = 64 * W;
  v8 a[kHold ? CT : 1][KS];  // R[column(ct, c16)][32 s + 8 g ..]
  Map map;
  float ebound;  // (D + 33 D / 32) 2^-24 max_j ||R_j||
  float eabs;    // 2^-19 max_i |T_i|
  bool exact_all, no_table;

  // The workgroup's tables (every thread calls it; ends with a barrier).
  // `more` issues the caller's own first loads, behind the tables' and before any wait.
  template <typename F>
  static __device__ __forceinline__ void fill(Lds<D>& t, const float* __restrict__ rot,
                                              const float* __restrict__ bnd, int nb, F more) {
    constexpr int NF = D * D / 4 / kThreads;  // float4 pieces per thread
    const int tid = threadIdx.x;
    if (tid == 0) t.shared_cell = t.irregular = 0;
    float bt = 0.f;
    if (tid < nb) bt = bnd[tid];
    v4f p[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i) p[i] = reinterpret_cast<const v4f*>(rot)[i * kThreads + tid];
    more();
    if (tid < 16) {
      const float b = round_to(bt, DT);
      t.bnd[tid] = b;
      t.thr[tid] = tid < nb ? threshold_of<BF>(b) : __builtin_inff();
    }
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const int f = i * kThreads + tid, j = 4 * f / D, k = 4 * f % D;
      typedef typename std::conditional<BF, __bf16, _Float16>::type h1;
      typedef h1 h4 __attribute__((ext_vector_type(4)));
      *reinterpret_cast<v2u*>(&t.r[Lds<D>::at(j) + k]) = __builtin_bit_cast(v2u, __builtin_convertvector(p[i], h4));
      float rr = fmaf(p[i][0], p[i][0], p[i][1] * p[i][1]) + fmaf(p[i][2], p[i][2], p[i][3] * p[i][3]);
#pragma unroll
      for (int o = 1; o < D / 4; o <<= 1) rr += __shfl_xor(rr, o, 64);  // a row's D / 4 threads
      if (k == 0) t.rr[j] = rr;
    }
    __syncthreads();
    const Map m = make_map(t, nb);
    const int c = tid & (kCells - 1);
    float th = __uint_as_float(0x7fc00000u);
    uint32_t below = 0, own = 0;
#pragma unroll
    for (int i = 0; i < 15; ++i) {
      if (i >= nb) break;
      const float vi = m.v(t.thr[i]);
      if (vi <= (float)c - (0.5f + kMargin)) ++below;
      else if (vi < (float)c + (0.5f + kMargin)) { th = t.thr[i]; ++own; }
    }
    if (own > 1) t.shared_cell = 1;
    if (tid < nb) {
      const float lim = BF ? 3e38f : 6e4f;
      if (!(fabsf(t.bnd[tid]) < lim) || (tid > 0 && !(t.bnd[tid - 1] <= t.bnd[tid]))) t.irregular = 1;
      if (!(m.s > 0.f && m.s < 1e30f && fabsf(m.off) < 1e6f)) t.shared_cell = 1;
    }
    for (int k = tid / kCells; k < kCopies; k += kThreads / kCells) t.lut[c][k] = (__float_as_uint(th) & ~15u) | below;
    __syncthreads();
  }

  static __device__ __forceinline__ Map make_map(const Lds<D>& t, int nb) {
    const float lo = t.thr[0], hi = t.thr[nb - 1];
    Map m;
    m.s = hi > lo ? 61.f / (hi - lo) : 1.f;
    m.off = rintf(1.f - lo * m.s);
    return m;
  }

  __device__ __forceinline__ void load(const Lds<D>& t, int nb) {
    const int lane = threadIdx.x & 63;
    map = make_map(t, nb);
    exact_all = t.irregular != 0;
    no_table = t.shared_cell != 0;
    eabs = 0x1p-19f * fmaxf(fabsf(t.thr[0]), fabsf(t.thr[nb - 1]));
    float big = 0.f;
#pragma unroll
    for (int j = 0; j < D; j += 64) {
      const float rr = t.rr[j + lane];
      big = fmaxf(big, rr < 1e30f ? rr : __builtin_inff());  // NaN and infinity: every code exact
    }
    if constexpr (kHold) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int s = 0; s < KS; ++s) a[ct][s] = operand(t, ct, s);
    }
    ebound = (float)(D + 33 * KS) * 0x1p-24f * 1.02f * sqrtf(wave_max(big));
  }

  static __device__ __forceinline__ v8 operand(const Lds<D>& t, int ct, int s) {
    const int lane = threadIdx.x & 63;
    return __builtin_bit_cast(v8, *reinterpret_cast<const v4u*>(
                                      &t.r[Lds<D>::at(column<D, ROWS>(ct, lane & 15)) + 32 * s + 8 * (lane >> 4)]));
  }

  // x[s]: dims 32 s + 8 g .. + 7 of the lane's row c16 (zeros for a row that is not there).
  // Returns the row's rounded norm; code[ct] holds the codes of the four columns
  // column(ct, 4 g + r) in its bytes r.
  __device__ __forceinline__ float tile(const Lds<D>& t, WaveLds<D>& wl, int nb, const v4u (&x)[KS],
                                        uint32_t (&code)[CT]) const {
    const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    auto el = [&](int s, int i) { return widen<BF>(i & 1 ? x[s][i >> 1] >> 16 : x[s][i >> 1] & 0xffffu); };
    auto across = [](float v, bool by32) {  // v + the partner lane's
      const uint32_t b = __float_as_uint(v);
      const v2u r = by32 ? __builtin_bit_cast(v2u, __builtin_amdgcn_permlane32_swap(b, b, false, false))
                         : __builtin_bit_cast(v2u, __builtin_amdgcn_permlane16_swap(b, b, false, false));
      return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
    // ---- norm, the sum of squares in any order: within 40 2^-24 (of nonnegative terms) of the
    // sum below, so its rounded root is the norm unless a rounding boundary lies that near
    float ss = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = fmaf(el(s, i), el(s, i), ss);
    ss = across(across(ss, true), false);
    float nrm = round_to(sqrtf(ss * (1.f + 0x1p-17f)), DT);
    if (__any(!(ss == 0.f || (ss > 1e-30f && ss < 1e37f && nrm == round_to(sqrtf(ss * (1.f - 0x1p-17f)), DT))))) {
      // dims l and l + 64 by fma, then the wave sum's tree over l = 0..63 (partners l ^ 32,
      // ^ 16, ..., ^ 1): l = 32 (s % 2) + 8 g + i, so ^ 32 and ^ 4, 2, 1 stay in the lane
      // and ^ 16, ^ 8 cross the lane groups
      float q[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float p[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          p[s] = el(s, i) * el(s, i);
          if constexpr (D == 128) p[s] = fmaf(el(s + 2, i), el(s + 2, i), p[s]);
        }
        q[i] = across(across(p[0] + p[1], true), false);
      }
      ss = ((q[0] + q[4]) + (q[2] + q[6])) + ((q[1] + q[5]) + (q[3] + q[7]));
      nrm = round_to(sqrtf(ss), DT);
    }
    const float den = fmaxf(nrm, round_to(1e-10f, DT));
    // ---- unit row, and a bound of its norm (1.02: the norm's and the elements' rounding)
    v8 b[KS];
    float uu = 1.04f;
    if (!__any(!(nrm > 0x1p-10f && nrm < 0x1p60f))) {
      const float y0 = __builtin_amdgcn_rcpf(den), y = fmaf(fmaf(-den, y0, 1.f), y0, y0);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        v8f u;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float xv = el(s, i);
          // bf16: a quotient of two 8-bit significands is no rounding midpoint and at least
          // 2^-17 from one, the product within 2^-22 of it.  fp16: the correctly rounded
          // quotient (as qm_div).
          u[i] = xv * y;
          if constexpr (!BF) u[i] = fmaf(fmaf(-u[i], den, xv), y, u[i]);
        }
        b[s] = __builtin_convertvector(u, v8);
      }
    } else {
      uu = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        v8f u;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          u[i] = round_to(el(s, i) / den, DT);
          uu = fmaf(u[i], u[i], uu);
        }
        b[s] = __builtin_convertvector(u, v8);
      }
      uu = across(across(uu, true), false);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) mfma_operand_fence(b[s]);
    // a zero row's sums are 0 in any order and a NaN row's NaN: nothing to repeat
    const float eps = uu > 0.f ? fmaf(ebound * 1.01f, sqrtf(uu), eabs) : -1.f;
    // ---- y = R u and codes
    uint32_t amb = 0;  // bit 4 CT - 1 - (4 ct + r): coordinate (ct, r) is within eps of a threshold
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        v8 op;
        if constexpr (kHold) op = a[ct][s];
        else op = operand(t, ct, s);
        if constexpr (BF) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op, b[s], acc, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, b[s], acc, 0, 0, 0);
      }
      uint32_t cd[4];
      if (!no_table) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t e = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(t.lut) +
                                                                map.entry(acc[r], 4 * (lane & (kCopies - 1))));
          const float th = __uint_as_float(e);
          cd[r] = e + (acc[r] > th ? 1u : 0u);  // at most 15 in the low four bits
          // the sign of |y - T| - eps
          amb = __builtin_amdgcn_alignbit(amb, __float_as_uint(fabsf(acc[r] - th) - eps), 31);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          uint32_t am = 0;
          cd[r] = 0;
#pragma unroll 1
          for (int i = 0; i < nb; ++i) {
            cd[r] += acc[r] > t.thr[i] ? 1u : 0u;
            am |= __float_as_uint(fabsf(acc[r] - t.thr[i]) - eps) >> 31;
          }
          amb = amb << 1 | am;
        }
      }
      const uint32_t lo = __builtin_amdgcn_perm(cd[1], cd[0], 0x0c0c0400u);
      const uint32_t hi = __builtin_amdgcn_perm(cd[3], cd[2], 0x0c0c0400u);
      code[ct] = (lo | hi << 16) & 0x0f0f0f0fu;
    }
    if (exact_all || eps > 0.9f * kMargin / map.s) amb = CT * 4 == 32 ? 0xffffffffu : (1u << (CT * 4)) - 1u;
    if (__any(amb != 0)) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
        *reinterpret_cast<v4u*>(&wl.u[c16][32 * s + 8 * g]) = __builtin_bit_cast(v4u, b[s]);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      while (__any(amb != 0)) {
        const int bit = amb ? __builtin_ctz(amb) : 0;
        const int idx = CT * 4 - 1 - bit, ct = idx >> 2, r = idx & 3;
        const int j = column<D, ROWS>(ct, 4 * g + r);
        float y = 0.f;
#pragma unroll 4
        for (int k = 0; k < D; k += 8) {
          const v4u uw = *reinterpret_cast<const v4u*>(&wl.u[c16][k]);
          const v4u rw = *reinterpret_cast<const v4u*>(&t.r[Lds<D>::at(j) + k]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            y = fmaf(widen<BF>(uw[e] & 0xffffu), widen<BF>(rw[e] & 0xffffu), y);
            y = fmaf(widen<BF>(uw[e] >> 16), widen<BF>(rw[e] >> 16), y);
          }
        }
        uint32_t c = (uint32_t)count_below(t.bnd, nb + 1, round_to(y, DT));
        if (amb) {
#pragma unroll
          for (int q2 = 0; q2 < CT; ++q2)
            if (q2 == ct) code[q2] = (code[q2] & ~(0xffu << (8 * r))) | c << (8 * r);
          amb &= amb - 1;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // wl.u is rewritten by the wave's next tile
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    return nrm;
  }
};

// Bit p of the eight codes of two code words (bytes, dim order) as a bit-plane byte, the
// first dim at bit 7.
__device__ __forceinline__ uint32_t nibbles8(uint32_t lo, uint32_t hi) {
  // pair bytes (even dim in the high nibble) of dims 0..7
  const uint32_t a = lo << 4 | lo >> 8, b = hi << 4 | hi >> 8;
  return __builtin_amdgcn_perm(b, a, 0x06040200u);
}
__device__ __forceinline__ uint32_t plane8(uint32_t nib, int p) {
  uint32_t t = (nib >> p) & 0x11111111u;  // per byte: even dim at bit 4, odd at bit 0
  t = (t | t >> 3) & 0x03030303u;
  return (t * 0x40100401u) >> 24;         // the four bytes' bit pairs, first byte on top
}

}  // namespace q16
}  // namespace tq
