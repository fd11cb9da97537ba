// tq_dequant.hip -- packed codes back to rows: round(round(c[codes] R) norm), d = 64 / 128
// (reference.py:320-367), from bit-plane rows, or from a decode-layout cache straight into
// the tensors a model's attention takes (history, then the new tokens as they are).
//
// A wave takes 32 tokens at a time.  The rows' centroids are the B operand of the MFMAs (a
// 256-entry table of centroid pairs turns a byte of two codes into two operand elements)
// and R^T, in LDS, the A operand, so a lane's results are consecutive columns of its token's
// row and leave in 16-byte stores.  bf16 / fp16 results: v_mfma_f32_16x16x32_{bf16,f16} on
// operands rounded to that type, as the reference rounds them; fp32: v_mfma_f32_16x16x4f32.
// Value tiles hold a dim's codes of several tokens per byte: they are transposed to rows of
// code pairs in LDS, a lane pair's two dims at a time.
//
// Why: a vector-ALU contraction of 16-row tiles took 479 us for 262,144 rows of 128 dims,
// after a pass (140 us) back to bit planes and before a copy (46 us) into the result.  Both
// sides of such a history (4096 tokens, 8 x 8 heads of 128 dims, bf16), one token added to it:
// 109 us a layer update with the tables' loads waited for one by one and an unroll that
// spilled 376 bytes a lane, 67 us with neither (72 over several states, caches cold).

#include "tq_common.h"

#include <algorithm>
#include <type_traits>

namespace tq {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8hf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

constexpr int kDqWaves = 8, kDqThreads = 64 * kDqWaves;
constexpr int kDqUnit = 32;    // tokens per wave step
constexpr int kPairCopies = 16;
constexpr int kPlanes = 0, kKeys = 1;  // row sources; 2-4: value tiles of that many bits

struct DqSide {
  const uint8_t* src;  // bit-plane rows [n], key pair bytes or value tiles [streams][t_cap ..]
  const void* norms;   // [streams][t_cap], norm_dt
  const float* cen;
  const float* rot;
  void* out;           // [streams][t_out][D]
  const void* fresh;   // new tokens, element (b, h, s, j) at b sb + h sh + s ss + j
  int64_t sb, sh, ss;
  int bits;            // kPlanes: bits of the codes
};
struct DqArgs {
  DqSide side[2];
  int64_t streams, t_cap, T, t_out;
  int norm_dt;
  int heads;           // streams = batch x heads
};

template <int D, int OUT>
struct DqLds {
  static constexpr bool k16 = OUT != TQ_F32;
  // R^T: row = output column.  16-bit rows start at at(col): the 16 columns a lane group
  // reads (32 p + 8 i + 4 e + r) start on 16 distinct bank quads.
  alignas(16) uint16_t r16[k16 ? D * (D + 8) + 2 * D : 8];
  float r32[k16 ? 1 : D * (D + 1)];
  static __device__ __forceinline__ int at(int col) { return col * (D + 8) + 32 * (col >> 4); }
  alignas(16) uint32_t pair[k16 ? 256 : 1][kPairCopies];  // (c[hi nibble], c[lo nibble])
  float cen[k16 ? 1 : 16][32];
  uint32_t spread[256];                       // kPlanes: a plane byte's bits in eight nibbles
  uint8_t rows[kDqWaves][kDqUnit][D / 2 + 4]; // value tiles as code pairs
};

template <int D, int OUT, int SRC>
__device__ __forceinline__ void dequant_side(const DqArgs& a, const DqSide& sd, DqLds<D, OUT>& t) {
  constexpr bool k16 = OUT != TQ_F32, BF = OUT == TQ_BF16;
  constexpr int KS = D / 32, CT = D / 16;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
  const int nlev = 1 << (SRC == kPlanes ? sd.bits : SRC == kKeys ? 4 : SRC);

  const int64_t per = (a.T + kDqUnit - 1) / kDqUnit, units = a.streams * per;
  const int64_t step = (int64_t)gridDim.x * kDqWaves;
  // A unit's packed codes as loaded: keys and bit planes, lane (token 16 u + c16, g): dims
  // D/4 g ..; value tiles, lane L: the words of its dims (SRC words per half and unit at
  // most 4) of the unit's 32 tokens
  constexpr int NR = SRC >= 2 ? 4 * (D / 64) : 8;
  struct Raw {
    uint32_t w[NR];
    float n[2];
  };
  auto load = [&](int64_t unit, Raw& r) {
    const int64_t s = unit / per, t0 = (unit - s * per) * kDqUnit;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t tk = t0 + 16 * u + c16;
      // a cache's fp32 norms are rounded to a 16-bit result's type first; bit-plane rows' are taken as given
      const float n = tk < a.T ? load_as_f32(sd.norms, s * a.t_cap + tk, a.norm_dt) : 0.f;
      r.n[u] = SRC == kPlanes ? n : round_to(n, OUT);
      if constexpr (SRC == kKeys) {
        const uint8_t* p = sd.src + (s * a.t_cap + (tk < a.T ? tk : a.T - 1)) * (D / 2) + (D / 8) * g;
#pragma unroll
        for (int i = 0; i < KS; ++i) r.w[4 * u + i] = reinterpret_cast<const uint32_t*>(p)[i];
      } else if constexpr (SRC == kPlanes) {
        const uint8_t* p = sd.src + (s * a.t_cap + (tk < a.T ? tk : a.T - 1)) * (sd.bits * (D / 8)) + (D / 32) * g;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          r.w[4 * u + b] = 0;
          if (b < sd.bits) {
            if constexpr (D == 128) r.w[4 * u + b] = *reinterpret_cast<const uint32_t*>(p + b * (D / 8));
            else r.w[4 * u + b] = *reinterpret_cast<const uint16_t*>(p + b * (D / 8));
          }
        }
      }
    }
    if constexpr (SRC >= 2) {
      const int64_t tile = s * (a.t_cap >> 6) + (t0 >> 6);
      const int G = (int)(t0 >> 5) & 1;
#pragma unroll
      for (int h = 0; h < D / 64; ++h) {
        const uint8_t* p = sd.src + (tile * (D / 64) + h) * (512 * SRC);
        uint32_t* w = r.w + 4 * h;
        if constexpr (SRC == 4) {
          const v4u v = *reinterpret_cast<const v4u*>(p + 1024 * G + 16 * lane);
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] = v[i];
        } else if constexpr (SRC == 2) {
          const v2u v = *reinterpret_cast<const v2u*>(p + 16 * lane + 8 * G);
          w[0] = v[0]; w[1] = v[1]; w[2] = w[3] = 0;
        } else {  // words 3 G .. 3 G + 2: words 0-3 at 16 L, 4-5 at 1024 + 8 L
          const v2u v = *reinterpret_cast<const v2u*>(G ? p + 1024 + 8 * lane : p + 16 * lane);
          const uint32_t x = *reinterpret_cast<const uint32_t*>(p + 16 * lane + (G ? 12 : 8));
          w[0] = G ? x : v[0]; w[1] = G ? v[0] : v[1]; w[2] = G ? v[1] : x; w[3] = 0;
        }
      }
    }
  };

  // ---- tables: everything they are made of requested at once, then the first unit
  __shared__ float cen_s[16];
  float cv0 = 0.f;
  if (tid < nlev) cv0 = sd.cen[tid];
  int64_t unit = (int64_t)blockIdx.x * kDqWaves + wave;
  Raw nx;
  if constexpr (k16) {
    constexpr int NP = D * D / 8 / kDqThreads > 0 ? D * D / 8 / kDqThreads : 1;
    v4f p[NP], q[NP];  // rows j, j + 1, columns 4 c ..
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int e = i * kDqThreads + tid, j = 2 * (e / (D / 4)), c = 4 * (e % (D / 4));
      if (e < D * D / 8) {
        p[i] = *reinterpret_cast<const v4f*>(sd.rot + j * D + c);
        q[i] = *reinterpret_cast<const v4f*>(sd.rot + (j + 1) * D + c);
      }
    }
    if (unit < units) load(unit, nx);
    if (tid < 16) cen_s[tid] = cv0;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int e = i * kDqThreads + tid, j = 2 * (e / (D / 4)), c = 4 * (e % (D / 4));
      if (e >= D * D / 8) continue;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        typedef typename std::conditional<BF, __bf16, _Float16>::type h1;
        typedef h1 h2 __attribute__((ext_vector_type(2)));
        *reinterpret_cast<uint32_t*>(&t.r16[DqLds<D, OUT>::at(c + k) + j]) =
            __builtin_bit_cast(uint32_t, (h2){(h1)p[i][k], (h1)q[i][k]});
      }
    }
    __syncthreads();
    for (int e = tid; e < 256 * kPairCopies / 4; e += kDqThreads) {
      typedef typename std::conditional<BF, __bf16, _Float16>::type h1;
      typedef h1 h2 __attribute__((ext_vector_type(2)));
      const int idx = e / (kPairCopies / 4);  // the even dim is the high nibble
      const uint32_t v = __builtin_bit_cast(uint32_t, (h2){(h1)cen_s[idx >> 4], (h1)cen_s[idx & 15]});
      *reinterpret_cast<v4u*>(&t.pair[idx][4 * (e % (kPairCopies / 4))]) = (v4u){v, v, v, v};
    }
  } else {
    if (unit < units) load(unit, nx);
    if (tid < 16) cen_s[tid] = cv0;
#pragma unroll 8
    for (int e = tid; e < D * D; e += kDqThreads) t.r32[(e % D) * (D + 1) + e / D] = sd.rot[e];
    __syncthreads();
    for (int e = tid; e < 16 * 32; e += kDqThreads) t.cen[e >> 5][e & 31] = cen_s[e >> 5];
  }
  if constexpr (SRC == kPlanes) {
    if (tid < 256) {  // dim i of eight at bit 7 - i; nibbles: the even dim of a byte high
      uint32_t v = 0;
      for (int i = 0; i < 8; ++i) v |= ((tid >> (7 - i)) & 1u) << (4 * (i ^ 1));
      t.spread[tid] = v;
    }
  }
  __syncthreads();
  for (; unit < units; unit += step) {
    const Raw cur = nx;
    if (unit + step < units) load(unit + step, nx);
    const int64_t s = unit / per, t0 = (unit - s * per) * kDqUnit;
    // ---- codes of lane (token, g) as nibbles, eight dims per word
    uint32_t nib[2][KS];
    if constexpr (SRC == kKeys) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < KS; ++i) nib[u][i] = cur.w[4 * u + i];
    } else if constexpr (SRC == kPlanes) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < KS; ++i) {
          nib[u][i] = 0;
#pragma unroll
          for (int b = 0; b < 4; ++b) nib[u][i] |= t.spread[(cur.w[4 * u + b] >> (8 * i)) & 255u] << b;
        }
    } else {
      const int sl = lane >> 4, odd = lane & 1;
      uint8_t* row0 = &t.rows[wave][4 * sl][(lane & 15) >> 1];
      constexpr int RS = D / 2 + 4;  // row stride
#pragma unroll
      for (int h = 0; h < D / 64; ++h) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = cur.w[4 * h + i];
        if constexpr (SRC == 2) {  // word mm: byte dg, token t of four at bits 2 t
#pragma unroll
          for (int mm = 0; mm < 2; ++mm) {
            const uint32_t n = (uint32_t)__builtin_amdgcn_mov_dpp((int)w[mm], 0xB1, 0xf, 0xf, true);  // lane ^ 1
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
              const int t2 = 2 * tt + odd;
              const uint32_t x = (w[mm] >> (2 * t2)) & 0x03030303u, y = (n >> (2 * t2)) & 0x03030303u;
              const uint32_t v = odd ? y << 4 | x : x << 4 | y;
#pragma unroll
              for (int dg = 0; dg < 4; ++dg) row0[(16 * mm + t2) * RS + 32 * h + 8 * dg] = (uint8_t)(v >> (8 * dg));
            }
          }
        } else {
          if constexpr (SRC == 3) {  // pair indices of 3-bit codes -> nibble pairs
            w[3] = ((w[0] >> 6) & 0x03030303u) | ((w[1] >> 4) & 0x0c0c0c0cu) | ((w[2] >> 2) & 0x30303030u);
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = (w[i] & 0x07070707u) | (w[i] & 0x38383838u) << 1;
          }
          // word dg: byte k, tokens 16 (k / 2) + 4 sl + 2 (k % 2) + e in nibble e
#pragma unroll
          for (int dg = 0; dg < 4; ++dg) {
            const uint32_t n = (uint32_t)__builtin_amdgcn_mov_dpp((int)w[dg], 0xB1, 0xf, 0xf, true);
            const uint32_t v = odd ? (n & 0xf0f0f0f0u) | ((w[dg] >> 4) & 0x0f0f0f0fu)
                                   : (w[dg] & 0x0f0f0f0fu) << 4 | (n & 0x0f0f0f0fu);
#pragma unroll
            for (int k = 0; k < 4; ++k)
              row0[(16 * (k >> 1) + 2 * (k & 1) + odd) * RS + 32 * h + 8 * dg] = (uint8_t)(v >> (8 * k));
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < KS; ++i)
          nib[u][i] = *reinterpret_cast<const uint32_t*>(&t.rows[wave][16 * u + c16][(D / 8) * g + 4 * i]);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the next unit rewrites the rows
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // ---- rows = R^T c[codes]; k order: dim D/4 g + 8 i + e of lane group g
    const int64_t tk0 = t0 + c16, tk1 = t0 + 16 + c16;
    if constexpr (k16) {
      using v8 = typename std::conditional<BF, v8bf, v8hf>::type;
      v8 b[2][KS];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < KS; ++i) {
          v4u w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = t.pair[(nib[u][i] >> (8 * e)) & 255u][lane & (kPairCopies - 1)];
          b[u][i] = __builtin_bit_cast(v8, w);
        }
      uint16_t* o0 = static_cast<uint16_t*>(sd.out) + (s * a.t_out + tk0) * D + 8 * g;
#pragma unroll
      for (int p = 0; p < CT / 2; ++p) {
        __builtin_amdgcn_sched_barrier(0);  // bounds the operand reads in flight (they spilled)
        v4f acc[2][2];  // [token group][column half]
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          acc[0][e] = acc[1][e] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < KS; ++i) {
            const int col = 32 * p + 8 * (c16 >> 2) + 4 * e + (c16 & 3);
            const v8 op = __builtin_bit_cast(v8, *reinterpret_cast<const v4u*>(&t.r16[DqLds<D, OUT>::at(col) + (D / 4) * g + 8 * i]));
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              if constexpr (BF) acc[u][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op, b[u][i], acc[u][e], 0, 0, 0);
              else acc[u][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, b[u][i], acc[u][e], 0, 0, 0);
            }
          }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          typedef typename std::conditional<BF, __bf16, _Float16>::type h1;
          typedef h1 h8 __attribute__((ext_vector_type(8)));
          typedef float v8f __attribute__((ext_vector_type(8)));
          v8f f;
#pragma unroll
          for (int r = 0; r < 8; ++r) f[r] = (float)(h1)acc[u][r >> 2][r & 3] * cur.n[u];
          if ((u ? tk1 : tk0) < a.T)
            *reinterpret_cast<v4u*>(o0 + u * 16 * D + 32 * p) = __builtin_bit_cast(v4u, __builtin_convertvector(f, h8));
        }
      }
    } else {
      float cv[2][D / 4];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) cv[u][8 * i + e] = t.cen[(nib[u][i] >> (4 * (e ^ 1))) & 15u][lane & 31];
      float* o0 = static_cast<float*>(sd.out) + (s * a.t_out + tk0) * D + 4 * g;
#pragma unroll 1
      for (int ct = 0; ct < CT; ++ct) {
        v4f acc[2];
        acc[0] = acc[1] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < D / 4; ++k) {
          const float op = t.r32[(16 * ct + c16) * (D + 1) + (D / 4) * g + k];
#pragma unroll
          for (int u = 0; u < 2; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(op, cv[u][k], acc[u], 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
          if ((u ? tk1 : tk0) < a.T) *reinterpret_cast<v4f*>(o0 + u * 16 * D + 16 * ct) = acc[u] * cur.n[u];
      }
    }
  }
  // ---- new tokens, copied as they are
  const int64_t s_new = a.t_out - a.T;
  if (sd.fresh && s_new > 0) {
    constexpr int V = 16 / (k16 ? 2 : 4), PR = D / V;  // 16-byte pieces per row
    constexpr int64_t es = k16 ? 2 : 4;
    const int64_t total = a.streams * s_new * PR;
    for (int64_t e = (int64_t)blockIdx.x * kDqThreads + tid; e < total; e += (int64_t)gridDim.x * kDqThreads) {
      const int pc = (int)(e % PR);
      const int64_t r = e / PR, s = r / s_new, i = r - s * s_new, b = s / a.heads, h = s - b * a.heads;
      const char* from = static_cast<const char*>(sd.fresh) + (b * sd.sb + h * sd.sh + i * sd.ss + pc * V) * es;
      char* to = static_cast<char*>(sd.out) + ((s * a.t_out + a.T + i) * D + pc * V) * es;
      *reinterpret_cast<v4u*>(to) = *reinterpret_cast<const v4u*>(from);
    }
  }
}

// A cache's keys (blockIdx.y 0) and values (1).
template <int D, int OUT, int VB>
__global__ __launch_bounds__(kDqThreads, OUT == TQ_F32 ? 2 : 4) void dequant_cache_kernel(DqArgs a) {
  __shared__ DqLds<D, OUT> t;
  if (blockIdx.y == 0) dequant_side<D, OUT, kKeys>(a, a.side[0], t);
  else dequant_side<D, OUT, VB>(a, a.side[1], t);
}

template <int D, int OUT>
__global__ __launch_bounds__(kDqThreads, OUT == TQ_F32 ? 2 : 4) void dequant_rows_kernel(DqArgs a) {
  __shared__ DqLds<D, OUT> t;
  dequant_side<D, OUT, kPlanes>(a, a.side[0], t);
}

unsigned dq_grid(const DqArgs& a, int out_dt, int sides) {
  const int64_t units = a.streams * ((a.T + kDqUnit - 1) / kDqUnit);
  const int64_t want = std::max<int64_t>(1, (units + kDqWaves - 1) / kDqWaves);
  const int64_t cap = (int64_t)device_cu_count() * (out_dt == TQ_F32 ? 1 : 2) / sides;
  return (unsigned)std::min(want, cap);
}

template <int D, int OUT>
void launch_cache(int vb, dim3 grid, const DqArgs& a, hipStream_t st) {
  if (vb == 2) hipLaunchKernelGGL((dequant_cache_kernel<D, OUT, 2>), grid, dim3(kDqThreads), 0, st, a);
  else if (vb == 3) hipLaunchKernelGGL((dequant_cache_kernel<D, OUT, 3>), grid, dim3(kDqThreads), 0, st, a);
  else hipLaunchKernelGGL((dequant_cache_kernel<D, OUT, 4>), grid, dim3(kDqThreads), 0, st, a);
}

bool aligned(const void* p, size_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

}  // namespace

// Bit-plane rows of d = 64 / 128 (tq_dequantize_mse); false where the shapes or addresses
// are not this kernel's.
bool dequant_rows_mfma(const uint8_t* packed, const float* norms, int64_t n, int d, int bits, const float* cen,
                       const float* rot, int out_dt, void* out, hipStream_t st) {
  if ((d != 64 && d != 128) || !aligned(packed, 4) || !aligned(out, 16) || !aligned(rot, 16)) return false;
  DqArgs a{};
  a.side[0] = DqSide{packed, norms, cen, rot, out, nullptr, 0, 0, 0, bits};
  a.streams = 1; a.t_cap = n; a.T = n; a.t_out = n; a.norm_dt = TQ_F32; a.heads = 1;
  const dim3 grid(dq_grid(a, out_dt, 1));
#define TQ_DQ_ROWS(D, OUT) hipLaunchKernelGGL((dequant_rows_kernel<D, OUT>), grid, dim3(kDqThreads), 0, st, a)
  if (d == 64) {
    if (out_dt == TQ_F32) TQ_DQ_ROWS(64, TQ_F32);
    else if (out_dt == TQ_BF16) TQ_DQ_ROWS(64, TQ_BF16);
    else TQ_DQ_ROWS(64, TQ_F16);
  } else {
    if (out_dt == TQ_F32) TQ_DQ_ROWS(128, TQ_F32);
    else if (out_dt == TQ_BF16) TQ_DQ_ROWS(128, TQ_BF16);
    else TQ_DQ_ROWS(128, TQ_F16);
  }
#undef TQ_DQ_ROWS
  return true;
}

}  // namespace tq

using namespace tq;

extern "C" int tq_dequantize_cache_dl(const uint8_t* kpairs, const void* knorms, const uint8_t* vtiles,
                                      const void* vnorms, tq_dtype norm_dtype, int64_t batch, int32_t heads,
                                      int32_t d, int64_t t_cap, int64_t T, int32_t vbits, const float* kcentroids,
                                      const float* krotation, const float* vcentroids, const float* vrotation,
                                      const void* key_new, const int64_t* key_strides, const void* value_new,
                                      const int64_t* value_strides, int64_t n_new, tq_dtype out_dtype, void* keys,
                                      void* values, void* stream) {
  TQ_REQUIRE(batch >= 0 && heads >= 1 && T >= 0 && n_new >= 0, "bad sizes");
  TQ_REQUIRE(d == 64 || d == 128, "dim must be 64 or 128, got %d", d);
  TQ_REQUIRE(vbits >= 2 && vbits <= 4, "value bits must be 2-4, got %d", vbits);
  TQ_REQUIRE(t_cap % 64 == 0 && T <= t_cap, "the capacity must be a multiple of 64 and hold T tokens");
  TQ_REQUIRE(valid_dtype(norm_dtype) && valid_dtype(out_dtype), "unknown dtype");
  if (batch == 0 || T + n_new == 0) return TQ_OK;
  TQ_REQUIRE(kcentroids && krotation && vcentroids && vrotation && keys && values, "null pointer argument");
  TQ_REQUIRE(T == 0 || (kpairs && knorms && vtiles && vnorms), "null pointer argument");
  TQ_REQUIRE(n_new == 0 || (key_new && key_strides && value_new && value_strides), "null pointer argument");
  TQ_REQUIRE(aligned(keys, 16) && aligned(values, 16) && aligned(kpairs, 16) && aligned(vtiles, 16) &&
                 aligned(krotation, 16) && aligned(vrotation, 16),
             "outputs, caches and rotations must be 16-byte aligned");
  DqArgs a{};
  a.side[0] = DqSide{kpairs, knorms, kcentroids, krotation, keys, n_new ? key_new : nullptr, 0, 0, 0, 4};
  a.side[1] = DqSide{vtiles, vnorms, vcentroids, vrotation, values, n_new ? value_new : nullptr, 0, 0, 0, vbits};
  if (n_new) {
    const int64_t piece = 16 / (int64_t)dtype_size(out_dtype);
    const int64_t* sv[2] = {key_strides, value_strides};
    for (int i = 0; i < 2; ++i) {
      TQ_REQUIRE(aligned(a.side[i].fresh, 16) && sv[i][0] % piece == 0 && sv[i][1] % piece == 0 && sv[i][2] % piece == 0,
                 "new tokens' rows must be 16-byte aligned");
      a.side[i].sb = sv[i][0]; a.side[i].sh = sv[i][1]; a.side[i].ss = sv[i][2];
    }
  }
  a.streams = batch * heads; a.t_cap = t_cap; a.T = T; a.t_out = T + n_new; a.norm_dt = (int)norm_dtype;
  a.heads = heads;
  const dim3 grid(dq_grid(a, out_dtype, 2), 2);
  hipStream_t st = as_stream(stream);
  if (d == 64) {
    if (out_dtype == TQ_F32) launch_cache<64, TQ_F32>(vbits, grid, a, st);
    else if (out_dtype == TQ_BF16) launch_cache<64, TQ_BF16>(vbits, grid, a, st);
    else launch_cache<64, TQ_F16>(vbits, grid, a, st);
  } else {
    if (out_dtype == TQ_F32) launch_cache<128, TQ_F32>(vbits, grid, a, st);
    else if (out_dtype == TQ_BF16) launch_cache<128, TQ_BF16>(vbits, grid, a, st);
    else launch_cache<128, TQ_F16>(vbits, grid, a, st);
  }
  TQ_LAUNCH_CHECK("dequant_cache_kernel");
  return TQ_OK;
}
