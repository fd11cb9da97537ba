// tq_append.hip -- bf16 / fp16 keys and values quantized straight into a decode-layout cache
// or its paged pools: one launch in the place of a quantize, a layout pass and a norm store
// for each of K and V (csrc/tq_q16.h computes the codes; tq_rotate_and_quantize followed by
// tq_pack_decode_layout / tq_paged_store* gives the same bytes).
//
// A wave quantizes 16 rows.  Keys: lane (row, g) holds D/4 consecutive dims' codes, which are
// D/8 whole pair bytes.  Values: lane (row, g) holds the codes of dims 16 dg + 4 g + r, whose
// four dg meet in one word of the value tile (2 bits) or in 16-bit shares of its words (3 and
// 4 bits), a token's bits at its own place in them.  Where the 16 rows are the 16 tokens of a
// sub-block (positions 16 q .. 16 q + 15 of a sequence), four lanes hold the four tokens of
// every word: they are merged by two DPP steps, each lane stores one of the four words, and
// nothing is read.  Tokens that come alone are merged into the stored words.

#include "tq_common.h"
#include "tq_q16.h"

#include <algorithm>

namespace tq {
namespace {

using q16::v4u;

// A value word's share of one token: codes (byte r of code[4 h + dg], dims 64 h + 16 dg +
// 4 g + r) at the bits of token t = position % 4.  VB 2: s[0] is the word.  VB 4: 16-bit shares
// dg 0, 1 in s[0], dg 2, 3 in s[1].  VB 3: shares of words 0, 1 in s[0] and 2 in s[1], dim
// group 3 still in s[1]'s upper half until fold3.
template <int VB>
struct Share {
  uint32_t s[VB == 2 ? 1 : 2];
};
__device__ __forceinline__ int share_shift(int VB, int t) {
  return VB == 2 ? 2 * t : VB == 4 ? 4 * t : 8 * (t >> 1) + 3 * (t & 1);
}
template <int VB>
__device__ __forceinline__ Share<VB> make_share(uint32_t bytes, int t) {  // bytes: dg 0..3
  Share<VB> o;
  const int sh = share_shift(VB, t);
  if constexpr (VB == 2) {
    o.s[0] = bytes << sh;
  } else {
    o.s[0] = __builtin_amdgcn_perm(0, bytes, 0x0c010c00u) << sh;
    o.s[1] = __builtin_amdgcn_perm(0, bytes, 0x0c030c02u) << sh;
  }
  return o;
}
template <int VB>
__device__ __forceinline__ Share<VB> field_mask(int t) {  // the bits token t owns
  return make_share<VB>(VB == 2 ? 0x03030303u : VB == 3 ? 0x07070707u : 0x0f0f0f0fu, t);
}
template <int VB>
__device__ __forceinline__ void fold3(Share<VB>& o) {
  if constexpr (VB == 3) {
    const uint32_t q = o.s[1] >> 16;
    o.s[0] |= (q & 0x0303u) << 6 | ((q >> 2) & 0x0303u) << 22;
    o.s[1] = (o.s[1] & 0xffffu) | ((q >> 4) & 0x0303u) << 6;
  }
}
__device__ __forceinline__ uint32_t quad_or(uint32_t v) {
  v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true);  // lane ^ 1
  v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xf, 0xf, true);  // lane ^ 2
  return v;
}
// Bytes r of four code words as a word, dg 0..3
template <int CT>
__device__ __forceinline__ uint32_t gather_byte(const uint32_t (&code)[CT], int h, int r) {
  const uint32_t sel = (uint32_t)r | (uint32_t)(r + 4) << 8 | 0x0c0c0000u;
  const uint32_t a = __builtin_amdgcn_perm(code[4 * h + 1], code[4 * h], sel);
  const uint32_t b = __builtin_amdgcn_perm(code[4 * h + 3], code[4 * h + 2], sel);
  return a | b << 16;
}
// Byte offset of share j (VB 2: of the word) of lane L's words, sub-block m of its tile.  In a
// 64-token tile: the word 4 m (VB 2), 16 bits of word (VB 4: 4, VB 3: 3) (m / 2) + j; in a
// 16-token sub-block's own 128 VB bytes (SUB): 4 L; 8 L + 2 j; 4 L + 2 j, the third at 256 + 2 L.
template <int VB, bool SUB>
__device__ __forceinline__ int share_off(int L, int m, int j) {
  if constexpr (SUB) {
    if (VB == 2) return 4 * L;
    if (VB == 4) return 8 * L + 2 * j;
    return j < 2 ? 4 * L + 2 * j : 256 + 2 * L;
  } else {
    if (VB == 2) return 16 * L + 4 * m;
    const int w = (VB == 4 ? 4 : 3) * (m >> 1) + j, k = 2 * (m & 1);
    return w < 4 ? 16 * L + 4 * w + k : 1024 + (8 * VB - 16) * L + 4 * (w - 4) + k;
  }
}
template <int VB>
__device__ __forceinline__ uint32_t share_of(const Share<VB>& o, int j) {
  return VB == 2 ? o.s[0] : (o.s[j >> 1] >> (16 * (j & 1))) & 0xffffu;
}

// Merges a 16-bit share at byte offset `off` into its word while the word's other half may be
// written the same way by another wave: whole-word atomics, the bits outside `mask` untouched.
__device__ __forceinline__ void merge_share(uint8_t* base, int off, uint32_t mask, uint32_t bits) {
  uint32_t* q = reinterpret_cast<uint32_t*>(base + (off & ~3));
  const int sh = 8 * (off & 2);
  atomicAnd(q, ~(mask << sh));
  atomicOr(q, bits << sh);
}

// Stores a 16-token sub-block's words of half h: row c16 is token c16 of the sub-block (live
// or not), m its number in the 64-token tile.  `base`: the tile's half, or the sub-block.
// In a tile, words of 3 and 4 bits hold two sub-blocks, a 16-bit share each.  `atomic`: single
// tokens of the other one may be merged (whole-word atomics) meanwhile; a plain 16-bit store
// would race with those on the word, so the share is merged like them.  Else the other
// sub-block is not written by this launch, or by plain 16-bit stores to its own bytes.
template <int VB, bool SUB, int CT>
__device__ __forceinline__ void store_sub_block(const uint32_t (&code)[CT], int h, bool live, int m,
                                                uint8_t* base, bool atomic = false) {
  const int lane = threadIdx.x & 63, g = lane >> 4, sl = (lane & 15) >> 2, t = lane & 3;
  Share<VB> mask = field_mask<VB>(t), mine{};
  constexpr int NS = VB == 2 ? 1 : 2;
#pragma unroll
  for (int i = 0; i < NS; ++i) mask.s[i] = quad_or(live ? mask.s[i] : 0u);
  fold3<VB>(mask);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    Share<VB> o = make_share<VB>(gather_byte(code, h, r), t);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      o.s[i] = quad_or(live ? o.s[i] : 0u);
      if (t == r) mine.s[i] = o.s[i];
    }
  }
  fold3<VB>(mine);
  const int L = 16 * sl + 4 * g + t;
  constexpr uint32_t kFull = VB == 2 ? 0xffffffffu : 0xffffu;
#pragma unroll
  for (int j = 0; j < (VB == 2 ? 1 : VB); ++j) {
    const uint32_t mk = share_of<VB>(mask, j), v = share_of<VB>(mine, j);
    if (mk == 0) continue;
    if constexpr (VB != 2 && !SUB) {
      if (atomic) {
        merge_share(base, share_off<VB, SUB>(L, m, j), mk, v);
        continue;
      }
    }
    uint8_t* p = base + share_off<VB, SUB>(L, m, j);
    if constexpr (VB == 2) {
      uint32_t* q = reinterpret_cast<uint32_t*>(p);
      *q = mk == kFull ? v : (*q & ~mk) | v;
    } else {
      uint16_t* q = reinterpret_cast<uint16_t*>(p);
      *q = (uint16_t)(mk == kFull ? v : (*q & ~mk) | v);
    }
  }
}

// Merges the lane's own token (position `at` in its 64-token tile) into half h's words.
// ATOMIC: other tokens of the same words may be written by other waves of this launch.
template <int VB, bool SUB, bool ATOMIC, int CT>
__device__ __forceinline__ void store_token(const uint32_t (&code)[CT], int h, int at, uint8_t* base) {
  const int g = (threadIdx.x & 63) >> 4, sl = (at >> 2) & 3, t = at & 3, m = at >> 4;
  Share<VB> mask = field_mask<VB>(t);
  fold3<VB>(mask);
  Share<VB> o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    o[r] = make_share<VB>(gather_byte(code, h, r), t);
    fold3<VB>(o[r]);
  }
  constexpr int NJ = VB == 2 ? 1 : VB;
  if constexpr (ATOMIC) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const uint32_t mk = share_of<VB>(mask, j);
        if (mk == 0) continue;
        merge_share(base, share_off<VB, SUB>(16 * sl + 4 * g + r, m, j), mk, share_of<VB>(o[r], j));
      }
  } else {
    uint32_t old[4][NJ];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const uint8_t* p = base + share_off<VB, SUB>(16 * sl + 4 * g + r, m, j);
        if constexpr (VB == 2) old[r][j] = *reinterpret_cast<const uint32_t*>(p);
        else old[r][j] = *reinterpret_cast<const uint16_t*>(p);
      }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        uint8_t* p = base + share_off<VB, SUB>(16 * sl + 4 * g + r, m, j);
        const uint32_t v = (old[r][j] & ~share_of<VB>(mask, j)) | share_of<VB>(o[r], j);
        if constexpr (VB == 2) *reinterpret_cast<uint32_t*>(p) = v;
        else *reinterpret_cast<uint16_t*>(p) = (uint16_t)v;
      }
  }
}

// The 3- / 4-bit codes of 16 streams' tokens (row s: stream s0 + s, all at position `at` of
// tile `tile`) merged into their value tiles: the codes pass through LDS, and then lane
// (c = lane / 4, i = lane % 4) owns word (VB 4: 4, VB 3: 3) (at / 32) + i of tile lane
// 16 sl + c, so a stream's words of a half are one 256-byte access (VB 3: 192 bytes in one
// or two pieces).  Merging from the codes' own lanes, 16 bytes apart over 16 streams at a time,
// took 25 us instead of 16 for 512 streams of 128 dims.
template <int D, int VB, int CT>
__device__ __forceinline__ void store_streams(const uint32_t (&code)[CT], q16::WaveLds<D>& wl, int64_t s0,
                                              int64_t streams, int64_t tiles, int64_t tile, int at, uint8_t* codes) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15, c = lane >> 2, i = lane & 3;
  constexpr int NW = VB == 4 ? 4 : 3, H = D / 64, RS = 2 * (D + 8);
  const int sl = (at >> 2) & 3, m = at >> 4, G = m >> 1, k = 2 * (m & 1) + ((at >> 1) & 1), e = at & 1;
  const int off = share_off<VB, false>(16 * sl + c, 2 * G, i);
  const int ns = (int)(streams - s0 < 16 ? streams - s0 : 16);
  uint8_t* lds = reinterpret_cast<uint8_t*>(wl.u);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) *reinterpret_cast<uint32_t*>(lds + c16 * RS + 16 * ct + 4 * g) = code[ct];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // bits of byte k: the token's field, and at 3 bits its bits of dim 48 + c in the byte's top two
  uint32_t mask = (VB == 4 ? 15u : 7u) << (VB * e);
  int top[2] = {0, 0};
  if constexpr (VB == 3) {
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      top[h2] = 2 * i + h2 - 3 * e;  // bit of the code at byte bit 6 + h2
      if (top[h2] >= 0 && top[h2] < 3) mask |= 64u << h2;
    }
  }
  if (i < NW) {
#pragma unroll
    for (int q0 = 0; q0 < 16; q0 += 8) {
      uint32_t old[8][H];
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int h = 0; h < H; ++h)
          old[q][h] = q0 + q < ns ? *reinterpret_cast<const uint32_t*>(
                                        codes + (((s0 + q0 + q) * tiles + tile) * H + h) * (512 * VB) + off)
                                  : 0u;
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const uint8_t* cr = lds + (q0 + q) * RS + 64 * h + c;
          uint32_t b = (uint32_t)cr[16 * i] << (VB * e);
          if constexpr (VB == 3) {
            const uint32_t c48 = cr[48];
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2)
              if (top[h2] >= 0 && top[h2] < 3) b |= ((c48 >> top[h2]) & 1u) << (6 + h2);
          }
          if (q0 + q < ns)
            *reinterpret_cast<uint32_t*>(codes + (((s0 + q0 + q) * tiles + tile) * H + h) * (512 * VB) + off) =
                (old[q][h] & ~(mask << (8 * k))) | b << (8 * k);
        }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();  // the next tile rewrites the LDS rows
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int D, int CT>
__device__ __forceinline__ void store_key(const uint32_t (&code)[CT], uint8_t* row) {
  const int g = (threadIdx.x & 63) >> 4;
  if constexpr (D == 128) {
    v4u w;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = q16::nibbles8(code[2 * i], code[2 * i + 1]);
    *reinterpret_cast<v4u*>(row + 16 * g) = w;
  } else {
    *reinterpret_cast<q16::v2u*>(row + 8 * g) =
        (q16::v2u){q16::nibbles8(code[0], code[1]), q16::nibbles8(code[2], code[3])};
  }
}

// wide: every row starts at a multiple of 16 bytes.
template <int KS>
__device__ __forceinline__ void load_row(const uint16_t* row, bool live, bool wide, v4u (&x)[KS]) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int s = 0; s < KS; ++s) x[s] = (v4u){0, 0, 0, 0};
  if (!live) return;
  if (wide) {
#pragma unroll
    for (int s = 0; s < KS; ++s) x[s] = *reinterpret_cast<const v4u*>(row + 32 * s + 8 * g);
  } else {
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) x[s][i >> 1] |= (uint32_t)row[32 * s + 8 * g + i] << (16 * (i & 1));
  }
}

// ------------------------------------------------------------------ contiguous caches
struct AppendSide {
  const uint16_t* x;   // element (b, h, i, j) at b sb + h sh + i ss + j
  int64_t sb, sh, ss;
  bool wide;           // rows 16-byte aligned
  const float* rot;
  const float* bnd;
  uint8_t* codes;      // [streams][t_cap][D / 2], or [streams][t_cap / 64][512 VB (D / 64)]
  void* norms;         // [streams][t_cap], norm_dt
};
struct AppendArgs {
  AppendSide side[2];
  int64_t streams;     // batch x heads
  int heads;
  int64_t n;           // new tokens per stream
  int64_t t_cap, pos;
  int norm_dt;
};

// One new token per stream: a tile is 16 streams.  More: 16 positions 16 q .. of a stream.
template <int D, bool BF, bool KEYS, int VB, bool ONE>
__device__ __forceinline__ void append_side(const AppendArgs& a, const AppendSide& sd, q16::Lds<D>& t,
                                            q16::WaveLds<D>* wl) {
  using Q = q16::Quantizer<D, BF, KEYS>;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int nb = KEYS ? 15 : (1 << VB) - 1;
  const int64_t q0 = a.pos >> 4, per = ONE ? 1 : ((a.pos + a.n + 15) >> 4) - q0;
  const int64_t ntiles = ONE ? (a.streams + 15) / 16 : a.streams * per;
  const int64_t step = (int64_t)gridDim.x * Q::W;
  int64_t tile = (int64_t)blockIdx.x * Q::W + wave;
  v4u x[Q::KS];
  auto where = [&](int64_t tl, int64_t& s, int64_t& tk) {  // the lane's row; whether there is one
    if constexpr (ONE) {
      s = tl * 16 + c16;
      tk = a.pos;
      return s < a.streams;
    } else {
      s = tl / per;
      tk = (q0 + (tl - s * per)) * 16 + c16;
      return tk >= a.pos && tk < a.pos + a.n;
    }
  };
  auto load = [&](int64_t tl) {
    int64_t s, tk;
    const bool live = where(tl, s, tk);
    const int64_t b = s / a.heads, h = s - b * a.heads;
    load_row(sd.x + b * sd.sb + h * sd.sh + (tk - a.pos) * sd.ss, live, sd.wide, x);
  };
  Q::fill(t, sd.rot, sd.bnd, nb, [&] { if (tile < ntiles) load(tile); });
  if (tile >= ntiles) return;  // no barrier follows
  Q q;
  q.load(t, nb);
  for (; tile < ntiles; tile += step) {
    v4u xc[Q::KS];
#pragma unroll
    for (int s = 0; s < Q::KS; ++s) xc[s] = x[s];
    if (tile + step < ntiles) load(tile + step);
    uint32_t code[Q::CT];
    const float nrm = q.tile(t, wl[wave], nb, xc, code);
    int64_t s, tk;
    const bool live = where(tile, s, tk);
    if (g == 0 && live) store_from_f32(sd.norms, s * a.t_cap + tk, nrm, a.norm_dt);
    if constexpr (KEYS) {
      if (live) store_key<D>(code, sd.codes + (s * a.t_cap + tk) * (D / 2));
    } else if constexpr (ONE && VB >= 3) {
      store_streams<D, VB>(code, wl[wave], tile * 16, a.streams, a.t_cap >> 6, a.pos >> 6, (int)(a.pos & 63), sd.codes);
    } else {
      uint8_t* base = sd.codes + (s * (a.t_cap >> 6) + (tk >> 6)) * (int64_t)(512 * VB * (D / 64));
#pragma unroll
      for (int h = 0; h < D / 64; ++h) {
        if constexpr (ONE) {
          if (live) store_token<VB, false, false>(code, h, (int)(tk & 63), base + h * 512 * VB);
        } else {
          store_sub_block<VB, false>(code, h, live, (int)(tk >> 4) & 3, base + h * 512 * VB);
        }
      }
    }
  }
}

template <int D, bool BF, int VB, bool ONE>
__global__ __launch_bounds__(64 * q16::waves<D>(), 4) void append_kernel(AppendArgs a) {
  __shared__ q16::Lds<D> t;
  __shared__ q16::WaveLds<D> wl[q16::waves<D>()];
  if (blockIdx.y == 0) append_side<D, BF, true, VB, ONE>(a, a.side[0], t, wl);
  else append_side<D, BF, false, VB, ONE>(a, a.side[1], t, wl);
}

template <int D, bool BF, int VB>
void launch_append(const AppendArgs& a, hipStream_t st) {
  const int64_t per = ((a.pos + a.n + 15) >> 4) - (a.pos >> 4);
  const int64_t tiles = D == 128 && a.n == 1 ? (a.streams + 15) / 16 : a.streams * per;
  const int w = q16::waves<D>();
  const int64_t cap = (int64_t)device_cu_count() * (D == 128 ? 1 : 2);
  const dim3 grid((unsigned)std::min((tiles + w - 1) / w, cap), 2);
  // (one token per stream at d = 64: tq_cache_append_dl)
  if (D == 128 && a.n == 1) hipLaunchKernelGGL((append_kernel<128, BF, VB, true>), grid, dim3(64 * w), 0, st, a);
  else hipLaunchKernelGGL((append_kernel<D, BF, VB, false>), grid, dim3(64 * w), 0, st, a);
}
template <int D, bool BF>
void launch_append_vb(int vb, const AppendArgs& a, hipStream_t st) {
  if (vb == 2) launch_append<D, BF, 2>(a, st);
  else if (vb == 3) launch_append<D, BF, 3>(a, st);
  else launch_append<D, BF, 4>(a, st);
}

// ------------------------------------------------------------------ paged pools (d = 64)
struct PagedArgs {
  const uint16_t* x[2];   // keys, values [n][heads][64]
  const float* rot[2];
  const float* bnd[2];
  uint8_t* pool[2];       // [blocks][heads][bs][32], value tiles or sub-blocks
  float* norms[2];        // [blocks][heads][bs]
  const int64_t* slots;   // [n]; outside [0, num_slots): skipped
  int64_t n, num_slots;
  int heads, bs_log2;
  bool wide[2];           // rows 16-byte aligned
};

// Window w of 16 new tokens of one head.  Tokens that fill a 16-aligned run of slots (a prompt's
// body) are taken as whole sub-blocks: the run that holds the window's first token, shifted
// back to the run's start, when all of its 16 tokens are in the batch; the window before
// leaves those tokens out.  The window's remaining tokens are merged one by one.  A batch names
// a slot once: the tokens of a whole run are the only ones of its sub-block.
template <bool BF, bool KEYS, int VB, bool SUB>
__device__ __forceinline__ void paged_side(const PagedArgs& a, q16::Lds<64>& t, q16::WaveLds<64>* wl) {
  using Q = q16::Quantizer<64, BF, KEYS>;
  constexpr int SD = KEYS ? 0 : 1;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int nb = KEYS ? 15 : (1 << VB) - 1;
  const int64_t windows = (a.n + 15) / 16, tasks = windows * a.heads;
  const int64_t step = (int64_t)gridDim.x * Q::W;
  Q::fill(t, a.rot[SD], a.bnd[SD], nb, [] {});
  Q q;
  int64_t task = (int64_t)blockIdx.x * Q::W + wave;
  if (task >= tasks) return;  // no barrier follows
  q.load(t, nb);
  // the first token of window w's whole run, -1 without one
  auto run_of = [&](int64_t w) -> int64_t {
    const int64_t i = 16 * w;
    if (KEYS || i >= a.n) return -1;
    const int64_t s0 = a.slots[i];
    const int64_t b = i - (s0 & 15);
    const bool in = s0 >= 0 && b >= 0 && b + 16 <= a.n;
    const int64_t s = in ? a.slots[b + c16] : -1;
    return __all(in && s == (s0 & ~(int64_t)15) + c16 && s < a.num_slots) ? b : -1;
  };
  // whether the other sub-block of run b's value words is a whole run of this batch, too (then
  // its window takes it as one and no single token of it is merged)
  auto paired = [&](int64_t b) {
    const int64_t s0 = a.slots[b], o = (s0 & 16) ? b - 16 : b + 16;
    const bool in = o >= 0 && o + 16 <= a.n;
    const int64_t s = in ? a.slots[o + c16] : -1;
    return (bool)__all(in && s == (s0 ^ 16) + c16);
  };
  auto block_of = [&](int64_t slot, int h) { return ((slot >> a.bs_log2) * a.heads + h) << a.bs_log2; };
  for (; task < tasks; task += step) {
    const int64_t w = task / a.heads;
    const int h = (int)(task - w * a.heads);
    const int64_t run = run_of(w), next = run_of(w + 1);
    for (int pass = run >= 0 ? 0 : 1; pass < 2; ++pass) {  // the run, then single tokens
      const int64_t i = pass == 0 ? run + c16 : 16 * w + c16;
      bool live = i < a.n;
      if (pass == 1 && ((run >= 0 && i >= run && i < run + 16) || (next >= 0 && i >= next))) live = false;
      const int64_t slot = live ? a.slots[i] : -1;
      live = live && slot >= 0 && slot < a.num_slots;
      if (!__any(live)) continue;
      v4u x[Q::KS];
      load_row(a.x[SD] + (i * a.heads + h) * 64, live, a.wide[SD], x);
      uint32_t code[Q::CT];
      const float nrm = q.tile(t, wl[wave], nb, x, code);
      const int64_t row = block_of(slot, h) + (slot & ((1 << a.bs_log2) - 1));
      if (g == 0 && live) a.norms[SD][row] = nrm;
      if constexpr (KEYS) {
        if (live) store_key<64>(code, a.pool[SD] + row * 32);
      } else {
        uint8_t* base = a.pool[SD] + (SUB ? (row >> 4) * (128 * VB) : (row >> 6) * (512 * VB));
        if (pass == 0) {
          store_sub_block<VB, SUB>(code, 0, true, (int)(row >> 4) & 3, base, !SUB && VB != 2 && !paired(run));
        }
        else if (live) store_token<VB, SUB, true>(code, 0, (int)(row & 63), base);
      }
    }
  }
}

template <bool BF, int VB, bool SUB>
__global__ __launch_bounds__(64 * q16::waves<64>(), 4) void paged_write_kernel(PagedArgs a) {
  __shared__ q16::Lds<64> t;
  __shared__ q16::WaveLds<64> wl[q16::waves<64>()];
  if (blockIdx.y == 0) paged_side<BF, true, VB, SUB>(a, t, wl);
  else paged_side<BF, false, VB, SUB>(a, t, wl);
}

template <bool BF, int VB>
void launch_paged(const PagedArgs& a, hipStream_t st) {
  const int w = q16::waves<64>();
  const int64_t tasks = (a.n + 15) / 16 * a.heads, cap = (int64_t)device_cu_count() * 2;
  const dim3 grid((unsigned)std::min((tasks + w - 1) / w, cap), 2);
  if (a.bs_log2 < 6) hipLaunchKernelGGL((paged_write_kernel<BF, VB, true>), grid, dim3(64 * w), 0, st, a);
  else hipLaunchKernelGGL((paged_write_kernel<BF, VB, false>), grid, dim3(64 * w), 0, st, a);
}
template <bool BF>
void launch_paged_vb(int vb, const PagedArgs& a, hipStream_t st) {
  if (vb == 2) launch_paged<BF, 2>(a, st);
  else if (vb == 3) launch_paged<BF, 3>(a, st);
  else launch_paged<BF, 4>(a, st);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace tq

using namespace tq;

extern "C" {

int tq_cache_append_tokens_dl(const void* key, const int64_t* key_strides, const void* value,
                              const int64_t* value_strides, tq_dtype in_dtype, int64_t batch, int32_t heads,
                              int64_t n, int32_t d, const float* krotation, const float* kboundaries,
                              const float* vrotation, const float* vboundaries, int32_t vbits, uint8_t* kpairs,
                              void* knorms, uint8_t* vtiles, void* vnorms, tq_dtype norm_dtype, int64_t t_cap,
                              int64_t pos, void* stream) {
  TQ_REQUIRE(in_dtype == TQ_BF16 || in_dtype == TQ_F16, "keys and values must be bf16 or fp16");
  TQ_REQUIRE(d == 64 || d == 128, "dim must be 64 or 128, got %d", d);
  TQ_REQUIRE(vbits >= 2 && vbits <= 4, "value bits must be 2-4, got %d", vbits);
  TQ_REQUIRE(valid_dtype(norm_dtype), "unknown norm dtype");
  TQ_REQUIRE(batch >= 0 && heads >= 1 && n >= 0 && t_cap >= 0 && t_cap % 64 == 0 && pos >= 0 && pos + n <= t_cap,
             "bad position or capacity");
  if (batch == 0 || n == 0) return TQ_OK;
  TQ_REQUIRE(key && key_strides && value && value_strides && krotation && kboundaries && vrotation && vboundaries &&
                 kpairs && knorms && vtiles && vnorms,
             "null pointer argument");
  TQ_REQUIRE(aligned16(krotation) && aligned16(vrotation) && aligned16(kpairs) && aligned16(vtiles),
             "rotations and caches must be 16-byte aligned");
  auto wide = [&](const void* p, const int64_t* st) {
    return aligned16(p) && st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0;
  };
  AppendArgs a{};
  a.side[0] = AppendSide{static_cast<const uint16_t*>(key), key_strides[0], key_strides[1], key_strides[2],
                         wide(key, key_strides), krotation, kboundaries, kpairs, knorms};
  a.side[1] = AppendSide{static_cast<const uint16_t*>(value), value_strides[0], value_strides[1], value_strides[2],
                         wide(value, value_strides), vrotation, vboundaries, vtiles, vnorms};
  a.streams = batch * heads; a.heads = heads; a.n = n; a.t_cap = t_cap; a.pos = pos; a.norm_dt = (int)norm_dtype;
  hipStream_t st = as_stream(stream);
  if (d == 64) {
    if (in_dtype == TQ_BF16) launch_append_vb<64, true>(vbits, a, st);
    else launch_append_vb<64, false>(vbits, a, st);
  } else {
    if (in_dtype == TQ_BF16) launch_append_vb<128, true>(vbits, a, st);
    else launch_append_vb<128, false>(vbits, a, st);
  }
  TQ_LAUNCH_CHECK("append_kernel");
  return TQ_OK;
}

int tq_paged_write_dl(const void* key, const void* value, tq_dtype in_dtype, int64_t n_tokens, int32_t hkv,
                      const float* krotation, const float* kboundaries, const float* vrotation,
                      const float* vboundaries, const int64_t* slot_mapping, uint8_t* kpairs_pool,
                      float* knorm_pool, uint8_t* vtile_pool, float* vnorm_pool, int64_t num_blocks,
                      int32_t block_size, int32_t vbits, void* stream) {
  TQ_REQUIRE(in_dtype == TQ_BF16 || in_dtype == TQ_F16, "keys and values must be bf16 or fp16");
  TQ_REQUIRE(n_tokens >= 0 && hkv >= 1 && num_blocks >= 0, "bad sizes");
  TQ_REQUIRE(vbits >= 2 && vbits <= 4, "value tiles hold 2-4 bit codes, got %d", vbits);
  int bsl = 0;
  while ((1 << bsl) < block_size) ++bsl;
  TQ_REQUIRE(block_size >= 16 && (1 << bsl) == block_size,
             "value tiles need a power-of-two block_size >= 16, got %d", block_size);
  if (n_tokens == 0) return TQ_OK;
  TQ_REQUIRE(key && value && krotation && kboundaries && vrotation && vboundaries && slot_mapping && kpairs_pool &&
                 knorm_pool && vtile_pool && vnorm_pool,
             "null pointer argument");
  TQ_REQUIRE(aligned16(krotation) && aligned16(vrotation) && aligned16(kpairs_pool) && aligned16(vtile_pool),
             "rotations and pools must be 16-byte aligned");
  PagedArgs a{};
  a.wide[0] = aligned16(key); a.wide[1] = aligned16(value);
  a.x[0] = static_cast<const uint16_t*>(key); a.x[1] = static_cast<const uint16_t*>(value);
  a.rot[0] = krotation; a.rot[1] = vrotation;
  a.bnd[0] = kboundaries; a.bnd[1] = vboundaries;
  a.pool[0] = kpairs_pool; a.pool[1] = vtile_pool;
  a.norms[0] = knorm_pool; a.norms[1] = vnorm_pool;
  a.slots = slot_mapping; a.n = n_tokens; a.num_slots = num_blocks << bsl; a.heads = hkv; a.bs_log2 = bsl;
  if (in_dtype == TQ_BF16) launch_paged_vb<true>(vbits, a, as_stream(stream));
  else launch_paged_vb<false>(vbits, a, as_stream(stream));
  TQ_LAUNCH_CHECK("paged_write_kernel");
  return TQ_OK;
}

}  // extern "C"
