// tq_row_filter.h -- top-k over bit-plane rows of any dim, and over prod rows (bit planes or
// pair rows beside QJL signs), filtered on the matrix cores.  Included by tq_scan.hip, whose
// exact scans (scan_kernel, pair_scan_kernel) it stands in for and falls back to.
//
// As the multi-query pair filter above: approximate scores with a proven error bound, every row
// whose upper bound reaches a threshold tau listed, the listed rows rescored with the exact
// scan's arithmetic (same products, same order, same rounding) and ranked, so ids and scores
// are the exact scan's.  A pass serves 16 queries (one 16-row MFMA operand).
//   rf_query   q_rot (and S q) per query with the exact scan's sums; fp16 operands scaled by a
//              power of two per query; beta1, beta2 with
//                |approx - exact| <= |n| (beta1 + |gamma| beta2) + 2^-100
//   rf_sample  lower bounds of evenly spaced 64-row groups; per query a bucket's largest (a bucket
//              is 16 rows where there are few groups, else a group or several)
//   rf_tau     tau = the k-th largest bucket maximum (k distinct rows score at least it)
//   rf_filter  every row against tau; rf_merge  rescoring and ranking
// A query with more listed rows than the lists hold is flagged and answered by the exact scan.
//
// beta1 = (||q_rot||_1 (e_c (1 + 2^-11) + max|c| (2^-11 + 2^-14)) + d (max|c| + e_c) 2^-25 / s1)
// (1 + 2^-9): the fp16 query costs 2^-11 relative, or 2^-25 / s1 absolute below fp16's normal
// range, the fp16 centroids e_c; 2^-14 covers fp32 sums of 256 products on the matrix cores
// (2^-15), the exact scan's own sequential sum (2^-16) and the few multiplies after them; the
// last factor the rounding of the bound itself.  beta2 the same for the signs, which are exact:
// (||S q||_1 (2^-11 + 2^-13) + d 2^-25 / s2) sqrt(pi/2)/d (1 + 2^-9), 2^-13 covering also the
// exact scan's four-sign table entries, their scaling and the fma with gamma.
//
// Why: the exact scan reads a per-query table in LDS for every dim of every row (two queries
// per pass at 200 dims: 390,001 rows x 16 queries 715 us, for 42 MB of rows); here a dim's
// centroid pair is looked up once for 16 queries.

constexpr int kRfQ = 16;             // queries per pass
constexpr int kRfThreads = 512, kRfWaves = kRfThreads / 64;
constexpr int kRfCap = 64;           // listed rows per (block, query)
constexpr int kRfMaxBuckets = 2048;
constexpr int kRfMergeCap = 6144, kRfMergeCapBig = 10240;
constexpr int kRfPairCopies = 16;

struct RfArgs {
  const uint8_t* rows;   // [n][bits bpp] bit planes, or pair rows of the same width
  const float* norms;    // [n]
  const uint8_t* signs;  // prod: [n][bpp]
  const float* gammas;   // prod: [n]
  int64_t n;
  const void* q;         // [nq][d]
  int q_dt, nq, d, bpp, bits, k;
  const float* rot;
  const float* qjl;
  const float* cen;
  float qjl_scale;
  float* qrot;           // [nq][256] rotated queries; [nq][256] S q follows
  uint32_t* qa;          // per pass: [1 or 2][KT][64 lanes][4 words] fp16 operands
  float4* qpar;          // [passes 16] {1 / s1, beta1, qjl_scale / s2, beta2}
  float* buckets;        // [passes 16][nbk]
  float* tau;            // [passes 16]
  int nbk, per_bucket, sstride, nsgroups, nb;
  bool wide;             // rot and qjl are read 16 bytes at a time
  int* cnt;              // [passes][nb][16]
  float* chi;            // [passes][nb][16][kRfCap]
  float* clo;
  int* cid;
  int* flag;             // [nq]
  float* out_s;
  int64_t* out_i;
};

// Sums of one query per block: thread j (of each matrix's 256) the dim j, in the exact scan's
// order; then the operand.  Rows of R and S pass through LDS 64 columns at a time, read
// coalesced, two chunks requested before the first is used (a block waits on memory only:
// 16 us at 200 dims with each thread reading its own rows, 20 us with 32 columns one ahead).
template <int KT, bool PROD>
__global__ __launch_bounds__(PROD ? 512 : 256) void rf_query_kernel(RfArgs a) {
#pragma clang fp contract(off)
  constexpr int NM = PROD ? 2 : 1, C = 64;
  __shared__ __attribute__((aligned(16))) float qs[256];
  __shared__ float mt[NM][256][C + 1];
  __shared__ float red[2][2][4];
  const int qi = blockIdx.x, mi = threadIdx.x >> 8, j = threadIdx.x & 255, d = a.d;
  const bool real = qi < a.nq;
  const float* __restrict__ mat = mi ? a.qjl : a.rot;
  const bool wide = a.wide;
  const int nch = real ? (d + C - 1) / C : 0;  // uniform
  // thread j's pieces of a chunk: row r = 16 i + j / 16, columns 4 (j % 16) ..
  struct Chunk {
    fs_v4f p[16];
  };
  auto load = [&](int ch, Chunk& c) {
    const int k = C * ch + 4 * (j & 15);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 16 * i + (j >> 4);
      c.p[i] = (fs_v4f){0.f, 0.f, 0.f, 0.f};
      if (r < d) {
        if (wide && k < d) c.p[i] = *reinterpret_cast<const fs_v4f*>(mat + (size_t)r * d + k);
        else if (!wide)
          for (int e = 0; e < 4; ++e)
            if (k + e < d) c.p[i][e] = mat[(size_t)r * d + k + e];
      }
    }
  };
  float v = 0.f;
  auto sums = [&](int ch, Chunk& c) {  // chunk ch's share of the sums; requests chunk ch + 2
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) mt[mi][16 * i + (j >> 4)][4 * (j & 15) + e] = c.p[i][e];
    if (ch + 2 < nch) load(ch + 2, c);
    __syncthreads();
    const int n = d - C * ch < C ? d - C * ch : C;
    if (j < d) {
      if (mi == 0) {
#pragma unroll 8
        for (int k = 0; k < n; ++k) v = v + qs[C * ch + k] * mt[0][j][k];
      } else {
#pragma unroll 8
        for (int k = 0; k < n; ++k) v = fmaf(qs[C * ch + k], mt[NM - 1][j][k], v);
      }
    }
  };
  Chunk c0, c1;
  if (nch > 0) load(0, c0);
  if (nch > 1) load(1, c1);
  if (mi == 0) qs[j] = real && j < d ? load_as_f32(a.q, (int64_t)qi * d + j, a.q_dt) : 0.f;
  for (int ch = 0; ch < nch; ch += 2) {
    sums(ch, c0);
    if (ch + 1 < nch) sums(ch + 1, c1);
  }
  if (real) a.qrot[((size_t)mi * a.nq + qi) * 256 + j] = v;
  // max |.| and 1-norm of each
  const int wave = j >> 6, lane = j & 63;
  const float am = wave_max(fabsf(v)), l1 = wave_sum(fabsf(v));
  if (lane == 0) { red[mi][0][wave] = am; red[mi][1][wave] = l1; }
  __syncthreads();
  float cmax = 0.f, ec = 0.f;
  for (int i = 0; i < (1 << a.bits); ++i) {
    const float c = a.cen[i];
    cmax = fmaxf(cmax, fabsf(c));
    ec = fmaxf(ec, fabsf(c - (float)(_Float16)c));
  }
  if (!(cmax < INFINITY)) ec = INFINITY;
  const int tile = qi / kRfQ, m16 = qi % kRfQ;
  const float amax = fmaxf(fmaxf(red[mi][0][0], red[mi][0][1]), fmaxf(red[mi][0][2], red[mi][0][3]));
  const float l = (red[mi][1][0] + red[mi][1][1]) + (red[mi][1][2] + red[mi][1][3]);
  int ex = 0;
  // a zero query has nothing to scale; a NaN or infinity makes the 1-norm no number below it
  const bool zero = l == 0.f, scalable = amax > 0.f && amax < INFINITY && l < INFINITY;
  if (scalable) frexpf(amax, &ex);
  const bool ok = zero || (scalable && ex > -60 && ex < 60);
  const float scale = ok && !zero ? ldexpf(1.f, 15 - ex) : 0.f, inv = ok && !zero ? ldexpf(1.f, ex - 15) : 0.f;
  float beta = INFINITY;
  if (ok) {
    beta = mi == 0 ? l * (ec * (1.f + 0x1p-11f) + cmax * (0x1p-11f + 0x1p-14f)) + (float)d * (cmax + ec) * 0x1p-25f * inv
                   : (l * (0x1p-11f + 0x1p-13f) + (float)d * 0x1p-25f * inv) * a.qjl_scale;
    beta *= 1.f + 0x1p-9f;
    if (!(beta < INFINITY) || !(ec < INFINITY)) beta = INFINITY;
  }
  // dim j: octet j / 8 = KT g + kt of lane group g, element j % 8
  if (j < 32 * KT) {
    const int o = j >> 3, g = o / KT, kt = o - g * KT, e = j & 7;
    uint16_t* dst = reinterpret_cast<uint16_t*>(a.qa + (((size_t)tile * NM + mi) * KT + kt) * 256);
    dst[(16 * g + m16) * 8 + e] = __builtin_bit_cast(uint16_t, (_Float16)(v * scale));
  }
  if (j == 0) {
    float2* par = reinterpret_cast<float2*>(a.qpar + qi);
    par[mi] = make_float2(mi ? inv * a.qjl_scale : inv, real ? beta : 0.f);
    if (!PROD) par[1] = make_float2(0.f, 0.f);
  }
}

// Eight bytes at p + off of a region that ends at `end` (at least 8), zeros past it.
__device__ __forceinline__ u32x2 rf_load8_tail(const uint8_t* p, int64_t off, int64_t end) {
  const int64_t at = off < end - 8 ? off : end - 8;
  uint64_t v;
  __builtin_memcpy(&v, p + at, 8);
  const int sh = (int)(off - at) * 8;
  v = sh < 64 ? v >> sh : 0;
  return (u32x2){(uint32_t)v, (uint32_t)(v >> 32)};
}

// A wave's 64-row group on its way to the operands.  Bit planes (rows of any byte count): the
// group's bytes are contiguous and start at a multiple of 64 bytes, so they come in 16-byte
// pieces a group ahead (load), go to the wave's LDS (stage), and lane (i, g) reads its row's
// octets KT g .. KT g + KT - 1 of a plane from there as whole words (octets).  Reading
// them from memory, eight bytes at any address, took 19 us per step of a CU's waves at 200 dims
// instead of 4.  Pair rows: MqRows' words and whole sign words straight from memory.
template <int BITS, int KT, bool PROD, bool PAIRS>
struct RfLds {
  static constexpr int PMAX = BITS * 4 * KT, SMAX = 4 * KT;  // bytes per row and sign row
  uint8_t rows[PAIRS ? 16 : 64 * PMAX + 16];
  uint8_t signs[PROD && !PAIRS ? 64 * SMAX + 16 : 16];
};

template <int BITS, int KT, bool PROD, bool PAIRS>
struct RfRows {
  static constexpr int NC = PAIRS ? 1 : (BITS * KT + 3) / 4, NS = PROD && !PAIRS ? (KT + 3) / 4 : 1;
  u32x4 c[NC], sc[NS];
  MqRows<32 * (KT == 2 || KT == 4 ? KT : 4), BITS, true> pr;  // pair rows
  uint32_t sg[PROD && PAIRS ? 4 : 1];
  float n, gam;
  __device__ __forceinline__ void load(const RfArgs& a, int64_t g, int lane) {
    const int64_t r0 = g * 64, mine = r0 + lane;
    n = mine < a.n ? a.norms[mine] : 0.f;
    gam = PROD && mine < a.n ? a.gammas[mine] : 0.f;
    if constexpr (PAIRS) {
      MqArgs m{};
      m.rows = a.rows; m.norms = a.norms; m.n = a.n;
      pr.load(m, (uint32_t)g, 0u, buf_rsrc(a.rows, 0), buf_rsrc(a.norms, 0), lane, 0);
      if constexpr (PROD) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          const int64_t row = r0 + 16 * rt + (lane & 15);
          const uint8_t* p = a.signs + (row < a.n ? row : a.n - 1) * (4 * KT) + KT * (lane >> 4);
          sg[rt] = KT == 4 ? *reinterpret_cast<const uint32_t*>(p) : *reinterpret_cast<const uint16_t*>(p);
        }
      }
    } else if (r0 + 64 <= a.n) {  // uniform; the last, partial group is read when it is staged
      const int P = BITS * a.bpp;
#pragma unroll
      for (int k = 0; k < NC; ++k)
        if (lane + 64 * k < 4 * P) c[k] = reinterpret_cast<const u32x4*>(a.rows + r0 * P)[lane + 64 * k];
      if constexpr (PROD) {
#pragma unroll
        for (int k = 0; k < NS; ++k)
          if (lane + 64 * k < 4 * a.bpp) sc[k] = reinterpret_cast<const u32x4*>(a.signs + r0 * a.bpp)[lane + 64 * k];
      }
    }
  }
  __device__ __forceinline__ void stage(const RfArgs& a, int64_t g, int lane, RfLds<BITS, KT, PROD, PAIRS>& l) const {
    if constexpr (!PAIRS) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the previous group's reads are done
      const int64_t r0 = g * 64;
      const int P = BITS * a.bpp;
      if (r0 + 64 <= a.n) {
#pragma unroll
        for (int k = 0; k < NC; ++k)
          if (lane + 64 * k < 4 * P) reinterpret_cast<u32x4*>(l.rows)[lane + 64 * k] = c[k];
        if constexpr (PROD) {
#pragma unroll
          for (int k = 0; k < NS; ++k)
            if (lane + 64 * k < 4 * a.bpp) reinterpret_cast<u32x4*>(l.signs)[lane + 64 * k] = sc[k];
        }
      } else {
        const int64_t left = a.n - r0;
#pragma unroll 1
        for (int b = lane; b < left * P; b += 64) l.rows[b] = a.rows[r0 * P + b];
        if constexpr (PROD) {
#pragma unroll 1
          for (int b = lane; b < left * a.bpp; b += 64) l.signs[b] = a.signs[r0 * a.bpp + b];
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
};

// KT bytes at byte `at` of an LDS buffer of whole words (up to 12 bytes read)
template <int KT>
__device__ __forceinline__ void rf_octets(const uint8_t* lds, int at, uint32_t (&o)[2]) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(lds + (at & ~3));
  const uint32_t w0 = w[0], w1 = w[1];
  o[0] = __builtin_amdgcn_alignbyte(w1, w0, at & 3);
  o[1] = 0;
  if constexpr (KT > 4) o[1] = __builtin_amdgcn_alignbyte(w[2], w1, at & 3);
}

struct RfTables {
  uint32_t pair[256][kRfPairCopies];  // fp16 (c[hi nibble], c[lo nibble])
  u32x4 sign[256];                    // eight +-1 of a sign byte
  uint32_t spread[256];               // a plane byte's bits in eight nibbles, even dims high
};
template <bool PROD>
__device__ __forceinline__ void rf_fill(RfTables& t, const RfArgs& a, int tid) {
  const int nlev = 1 << a.bits;
  for (int e = tid; e < 256 * kRfPairCopies; e += kRfThreads) {
    const int idx = e / kRfPairCopies, hi = idx >> 4, lo = idx & 15;
    const uint16_t h = __builtin_bit_cast(uint16_t, (_Float16)(hi < nlev ? a.cen[hi] : 0.f));
    const uint16_t l = __builtin_bit_cast(uint16_t, (_Float16)(lo < nlev ? a.cen[lo] : 0.f));
    t.pair[idx][e % kRfPairCopies] = h | (uint32_t)l << 16;
  }
  if (tid < 256) {
    uint32_t v = 0;
    for (int i = 0; i < 8; ++i) v |= (((uint32_t)tid >> (7 - i)) & 1u) << (4 * (i ^ 1));
    t.spread[tid] = v;
    if constexpr (PROD) {
      u32x4 s;
      for (int i = 0; i < 4; ++i)
        s[i] = ((tid >> (7 - 2 * i)) & 1 ? 0x3c00u : 0xbc00u) | ((tid >> (6 - 2 * i)) & 1 ? 0x3c000000u : 0xbc000000u);
      t.sign[tid] = s;
    }
  }
}

// A wave's operands and the lane's four queries' parameters.
template <int KT, bool PROD>
struct RfQuery {
  fs_v8h a1[KT], a2[PROD ? KT : 1];
  float4 par[4];  // queries 4 g + r
  __device__ __forceinline__ void load(const RfArgs& a, int tile, int lane) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      a1[kt] = __builtin_bit_cast(fs_v8h, *reinterpret_cast<const u32x4*>(
                                              a.qa + (((size_t)tile * (PROD ? 2 : 1)) * KT + kt) * 256 + lane * 4));
      if constexpr (PROD)
        a2[kt] = __builtin_bit_cast(fs_v8h, *reinterpret_cast<const u32x4*>(
                                                a.qa + (((size_t)tile * 2 + 1) * KT + kt) * 256 + lane * 4));
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) par[r] = a.qpar[tile * kRfQ + 4 * (lane >> 4) + r];
  }
};

// The unscaled sums of row tile rt: query 4 (lane >> 4) + r, row 16 rt + (lane & 15)
template <int BITS, int KT, bool PROD, bool PAIRS>
__device__ __forceinline__ void rf_scores(const RfRows<BITS, KT, PROD, PAIRS>& rb, int rt,
                                          const RfQuery<KT, PROD>& q, const RfTables& t,
                                          const RfLds<BITS, KT, PROD, PAIRS>& l, int bpp, int lane, fs_v4f& s1,
                                          fs_v4f& s2) {
  s1 = s2 = (fs_v4f){0.f, 0.f, 0.f, 0.f};
  uint32_t pl[BITS][2], sg[2];
  const int row = 16 * rt + (lane & 15), oct = KT * (lane >> 4);
  if constexpr (!PAIRS) {
#pragma unroll
    for (int p = 0; p < BITS; ++p) rf_octets<KT>(l.rows, row * BITS * bpp + p * bpp + oct, pl[p]);
    if constexpr (PROD) rf_octets<KT>(l.signs, row * bpp + oct, sg);
  } else if constexpr (PROD) {
    sg[0] = rb.sg[rt];
    sg[1] = 0;
  }
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    uint32_t nib = 0;
    if constexpr (PAIRS) {
      const uint32_t x = mq_pair_indices<32 * KT, BITS, true>(rb.pr, rt, kt, (uint32_t)lane);
      constexpr uint32_t lo = BITS == 3 ? 0x07070707u : 0x03030303u;
      nib = (x & lo) | ((x & (lo << BITS)) << (4 - BITS));
    } else {
#pragma unroll
      for (int p = 0; p < BITS; ++p) nib |= t.spread[(pl[p][kt >> 2] >> (8 * (kt & 3))) & 255u] << p;
    }
    u32x4 b;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = t.pair[(nib >> (8 * e)) & 255u][lane & (kRfPairCopies - 1)];
    s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(q.a1[kt], __builtin_bit_cast(fs_v8h, b), s1, 0, 0, 0);
    if constexpr (PROD) {
      const u32x4 sv = t.sign[(sg[kt >> 2] >> (8 * (kt & 3))) & 255u];
      s2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(q.a2[kt], __builtin_bit_cast(fs_v8h, sv), s2, 0, 0, 0);
    }
  }
}

// approx and its bound of (query r, row): mid -+ bound
template <int KT, bool PROD>
__device__ __forceinline__ void rf_bounds(const RfQuery<KT, PROD>& q, int r, float s1, float s2, float n, float gam,
                                          float& mid, float& bound) {
  float t = s1 * q.par[r].x, b = q.par[r].y;
  if constexpr (PROD) {
    t = __builtin_fmaf(gam, s2 * q.par[r].z, t);
    b = __builtin_fmaf(fabsf(gam), q.par[r].w, b);
  }
  mid = n * t;
  bound = __builtin_fmaf(fabsf(n), b, 0x1p-100f);
}

// FINE: a bucket per 16 rows (per_bucket 1), else per per_bucket groups.
template <int BITS, int KT, bool PROD, bool PAIRS, bool FINE>
__global__ __launch_bounds__(kRfThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void rf_sample_kernel(RfArgs a) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) RfTables t;
  __shared__ __attribute__((aligned(16))) RfLds<BITS, KT, PROD, PAIRS> lds[kRfWaves];
  const int tid = threadIdx.x, lane = tid & 63, tile = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bucket = blockIdx.x * kRfWaves + wave;
  RfRows<BITS, KT, PROD, PAIRS> rb;
  if (bucket * a.per_bucket < a.nsgroups) rb.load(a, (int64_t)bucket * a.per_bucket * a.sstride, lane);
  RfQuery<KT, PROD> q;
  q.load(a, tile, lane);
  rf_fill<PROD>(t, a, tid);
  __syncthreads();
  float bmax[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) bmax[r] = -INFINITY;
  auto store = [&](int at) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = row_max16(bmax[r]);
      if ((lane & 15) == 0) a.buckets[(size_t)(tile * kRfQ + 4 * (lane >> 4) + r) * a.nbk + at] = v;
      if (FINE) bmax[r] = -INFINITY;
    }
  };
  for (int u = 0; u < a.per_bucket; ++u) {
    const int s = bucket * a.per_bucket + u;
    if (s >= a.nsgroups) break;  // uniform
    const int64_t g = (int64_t)s * a.sstride;
    if (u) rb.load(a, g, lane);
    rb.stage(a, g, lane, lds[wave]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      __builtin_amdgcn_sched_barrier(0);
      fs_v4f s1, s2;
      rf_scores<BITS, KT, PROD, PAIRS>(rb, rt, q, t, lds[wave], a.bpp, lane, s1, s2);
      const float n = __shfl(rb.n, 16 * rt + (lane & 15)), gam = PROD ? __shfl(rb.gam, 16 * rt + (lane & 15)) : 0.f;
      const bool valid = g * 64 + 16 * rt + (lane & 15) < a.n;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float mid, b;
        rf_bounds<KT, PROD>(q, r, s1[r], s2[r], n, gam, mid, b);
        const float lo = mid - b;  // no bound from an overflowed one
        if (valid && lo < INFINITY) bmax[r] = fmaxf(bmax[r], lo);
      }
      if (FINE) store(4 * bucket + rt);
    }
  }
  if (!FINE && bucket < a.nbk) store(bucket);
}

// One block per query: tau = its k-th largest bucket maximum, by bits of an order-preserving key
// (one wave per query, 32 keys a lane, took 16 to 32 us at 1,523 buckets).
__global__ __launch_bounds__(kRfThreads) void rf_tau_kernel(RfArgs a) {
  constexpr int PER = kRfMaxBuckets / kRfThreads;
  __shared__ int cnt[32];
  const int q = blockIdx.x, tid = threadIdx.x;
  const float* src = a.buckets + (size_t)q * a.nbk;
  uint32_t u[PER];
  if (tid < 32) cnt[tid] = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = j * kRfThreads + tid;
    const float v = e < a.nbk ? src[e] : -INFINITY;
    u[j] = v > -INFINITY ? fs_fkey(v) : 0u;
  }
  __syncthreads();
  uint32_t x = 0;
#pragma unroll 1
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t tr = x | (1u << bit);
    int c = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) c += __popcll(__ballot(u[j] >= tr));
    if ((tid & 63) == 0 && c) atomicAdd(&cnt[bit], c);
    __syncthreads();
    if (cnt[bit] >= a.k) x = tr;
  }
  if (tid == 0) a.tau[q] = x ? fs_unkey(x) : -INFINITY;
}

template <int BITS, int KT, bool PROD, bool PAIRS>
__global__ __launch_bounds__(kRfThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void rf_filter_kernel(RfArgs a) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) RfTables t;
  __shared__ __attribute__((aligned(16))) RfLds<BITS, KT, PROD, PAIRS> lds[kRfWaves];
  __shared__ int cnt_s[kRfQ];
  const int tid = threadIdx.x, lane = tid & 63, tile = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t W = (int64_t)gridDim.x * kRfWaves, ngroups = (a.n + 63) / 64;
  int64_t g = (int64_t)blockIdx.x * kRfWaves + wave;
  RfRows<BITS, KT, PROD, PAIRS> nx;
  if (g < ngroups) nx.load(a, g, lane);
  RfQuery<KT, PROD> q;
  q.load(a, tile, lane);
  float th[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int qi = tile * kRfQ + 4 * (lane >> 4) + r;
    th[r] = a.tau[qi];
  }
  if (tid < kRfQ) cnt_s[tid] = 0;
  rf_fill<PROD>(t, a, tid);
  __syncthreads();
  const size_t lbase = ((size_t)tile * a.nb + blockIdx.x) * kRfQ;
  for (; g < ngroups; g += W) {
    const RfRows<BITS, KT, PROD, PAIRS> rb = nx;
    rb.stage(a, g, lane, lds[wave]);
    if (g + W < ngroups) nx.load(a, g + W, lane);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      __builtin_amdgcn_sched_barrier(0);
      fs_v4f s1, s2;
      rf_scores<BITS, KT, PROD, PAIRS>(rb, rt, q, t, lds[wave], a.bpp, lane, s1, s2);
      const float n = __shfl(rb.n, 16 * rt + (lane & 15)), gam = PROD ? __shfl(rb.gam, 16 * rt + (lane & 15)) : 0.f;
      const int64_t row = g * 64 + 16 * rt + (lane & 15);
      float mid[4], b[4];
      uint32_t hit = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        rf_bounds<KT, PROD>(q, r, s1[r], s2[r], n, gam, mid[r], b[r]);
        const bool real = tile * kRfQ + 4 * (lane >> 4) + r < a.nq;
        hit |= (uint32_t)(real & (row < a.n) & !(mid[r] + b[r] < th[r])) << r;  // NaN bounds are listed
      }
      if (__any(hit != 0)) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if ((hit >> r) & 1u) {
            const int ql = 4 * (lane >> 4) + r, slot = atomicAdd(&cnt_s[ql], 1);
            if (slot < kRfCap) {
              const size_t e = (lbase + ql) * kRfCap + slot;
              a.chi[e] = mid[r] + b[r];
              a.clo[e] = mid[r] - b[r];
              a.cid[e] = (int)row;
            }
          }
      }
    }
  }
  __syncthreads();
  if (tid < kRfQ) a.cnt[lbase + tid] = cnt_s[tid];
}

// The exact scan's score of a listed row: products q_rot[j] c[code] (ptab) added in dim
// order, then gamma times the sign table's sum, then the norm.
template <int BITS, bool PROD, bool PAIRS>
__device__ __forceinline__ float rf_exact(const RfArgs& a, int64_t id, const float* ptab, const float* stab) {
#pragma clang fp contract(off)
  constexpr int NL = 1 << BITS;
  const int P = BITS * a.bpp, d = a.d;
  const float nrm = a.norms[id], gam = PROD ? a.gammas[id] : 0.f;
  float acc = 0.f, sacc = 0.f;
  if constexpr (PAIRS) {  // d = 64 / 128: codes of dims 32 t .. in BITS words (layouts above pmp_row)
    for (int t = 0; t < d / 32; ++t) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < BITS; ++i) w[i] = *reinterpret_cast<const uint32_t*>(a.rows + id * P + 4 * (BITS * t + i));
      if constexpr (BITS == 3)
        w[3] = ((w[0] >> 6) & 0x03030303u) | ((w[1] >> 4) & 0x0C0C0C0Cu) | ((w[2] >> 2) & 0x30303030u);
#pragma unroll
      for (int e = 0; e < 32; ++e) {  // 3 bits: pair e / 2 in byte (e / 2) % 4 of word e / 8
        const uint32_t code = BITS == 3 ? (w[e >> 3] >> (8 * ((e >> 1) & 3) + (e & 1 ? 0 : 3))) & 7u
                                        : (w[e >> 4] >> (8 * ((e >> 2) & 3) + 6 - 2 * (e & 3))) & 3u;
        acc = acc + ptab[(32 * t + e) * NL + code];
      }
    }
  }
  for (int o0 = 0; o0 < a.bpp; o0 += 8) {
    u32x2 w[BITS], sg;
    if constexpr (!PAIRS) {
#pragma unroll
      for (int p = 0; p < BITS; ++p) w[p] = rf_load8_tail(a.rows, id * P + p * a.bpp + o0, a.n * P);
    }
    if constexpr (PROD) sg = rf_load8_tail(a.signs, id * a.bpp + o0, a.n * a.bpp);
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      if (o0 + o >= a.bpp) break;
      if constexpr (!PAIRS) {
        uint32_t by[BITS];
#pragma unroll
        for (int p = 0; p < BITS; ++p) by[p] = w[p][o >> 2] >> (8 * (o & 3));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int j = 8 * (o0 + o) + i;
          if (j >= d) break;
          uint32_t code = 0;
#pragma unroll
          for (int p = 0; p < BITS; ++p) code |= ((by[p] >> (7 - i)) & 1u) << p;
          acc = acc + ptab[j * NL + code];
        }
      }
      if constexpr (PROD) {
        const uint32_t s = sg[o >> 2] >> (8 * (o & 3));
        sacc = sacc + stab[(2 * (o0 + o)) * 16 + ((s >> 4) & 15u)];
        sacc = sacc + stab[(2 * (o0 + o) + 1) * 16 + (s & 15u)];
      }
    }
  }
  if constexpr (PROD) acc = fmaf(gam, sacc, acc);
  return acc * nrm;
}

template <int BITS, bool PROD, bool PAIRS, int MCAP>
__global__ __launch_bounds__(kRfThreads) void rf_merge_kernel(RfArgs a) {
#pragma clang fp contract(off)
  constexpr int NL = 1 << BITS;
  __shared__ __attribute__((aligned(16))) float ehi[MCAP];
  __shared__ __attribute__((aligned(16))) float elo[MCAP];
  __shared__ __attribute__((aligned(16))) int eid[MCAP];
  __shared__ float ptab[256 * NL];
  __shared__ float stab[PROD ? 64 * 16 : 1];
  __shared__ int off_s[kRfThreads + 1];
  __shared__ int part[kRfWaves];
  __shared__ int tcnt[32];
  __shared__ int bad_s, m2_s, nvalid_s, shi_s[2];
  __shared__ float ts_s;
  const int q = blockIdx.x, ql = q % kRfQ, tile = q / kRfQ;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nb = a.nb, k = a.k, d = a.d;
  int c = 0;
  if (tid < nb) c = a.cnt[((size_t)tile * nb + tid) * kRfQ + ql];
  if (tid == 0) { bad_s = 0; m2_s = 0; nvalid_s = 0; }
  if (tid < 32) tcnt[tid] = 0;
  // the exact scan's tables of this query
  for (int e = tid; e < d * NL; e += kRfThreads) ptab[e] = a.qrot[(size_t)q * 256 + e / NL] * a.cen[e % NL];
  if constexpr (PROD) {
    const float* qs = a.qrot + ((size_t)a.nq + q) * 256;
    for (int e = tid; e < 64 * 16; e += kRfThreads) {
      const int g = e >> 4, v = e & 15;
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = 4 * g + i < d ? qs[4 * g + i] : 0.f;
        s += ((v >> (3 - i)) & 1) ? x : -x;
      }
      stab[e] = s * a.qjl_scale;
    }
  }
  __syncthreads();
  if (c > kRfCap) bad_s = 1;
  int incl = c;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(incl, off);
    if (lane >= off) incl += y;
  }
  if (lane == 63) part[wave] = incl;
  __syncthreads();
  int wofs = 0;
  for (int w = 0; w < wave; ++w) wofs += part[w];
  off_s[tid] = wofs + incl - c;
  if (tid == kRfThreads - 1) off_s[kRfThreads] = wofs + incl;
  __syncthreads();
  const int M = off_s[kRfThreads];
  if (bad_s || M > MCAP) {  // uniform
    if (tid == 0) a.flag[q] = 1;
    return;
  }
  if (tid == 0) a.flag[q] = 0;
  for (int e = tid; e < M; e += kRfThreads) {
    int lo = 0, hi = nb;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (off_s[mid] <= e) lo = mid; else hi = mid;
    }
    const size_t src = (((size_t)tile * nb + lo) * kRfQ + ql) * kRfCap + (e - off_s[lo]);
    const float l = a.clo[src];
    ehi[e] = a.chi[src];
    elo[e] = l == l ? l : -INFINITY;
    eid[e] = a.cid[src];
  }
  __syncthreads();
  // tau' = the k-th best listed lo (up to one entry per thread every entry is rescored anyway)
  constexpr int EPT = (MCAP + kRfThreads - 1) / kRfThreads;
  uint32_t x = 0;
  if (M > kRfThreads) {  // uniform
    uint32_t u[EPT];
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int e = j * kRfThreads + tid;
      u[j] = (e < M && elo[e] > -INFINITY) ? fs_fkey(elo[e]) : 0u;
    }
#pragma unroll 1
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t tr = x | (1u << bit);
      int cc = 0;
#pragma unroll
      for (int j = 0; j < EPT; ++j)
        if (j * kRfThreads < M) cc += __popcll(__ballot(u[j] >= tr));
      if (lane == 0 && cc) atomicAdd(&tcnt[bit], cc);
      __syncthreads();
      if (tcnt[bit] >= k) x = tr;
    }
  }
  const float tau2 = fmaxf(a.tau[q], x ? fs_unkey(x) : -INFINITY);
  int my[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = j * kRfThreads + tid;
    my[j] = (e < M && !(ehi[e] < tau2)) ? eid[e] : -1;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < EPT; ++j)
    if (my[j] >= 0) eid[atomicAdd(&m2_s, 1)] = my[j];
  __syncthreads();
  const int m2 = m2_s;
  for (int s = tid; s < m2; s += kRfThreads) {
    const float sc = rf_exact<BITS, PROD, PAIRS>(a, eid[s], ptab, stab);
    const bool ok = !__builtin_isnan(sc);
    ehi[s] = ok ? sc : -INFINITY;
    if (!ok) eid[s] = INT_MAX;
    else atomicAdd(&nvalid_s, 1);
  }
  for (int s = m2 + tid; s < ((m2 + 3) & ~3); s += kRfThreads) { ehi[s] = -INFINITY; eid[s] = INT_MAX; }
  int* rk = reinterpret_cast<int*>(elo);
  const int m3 = rank_best<kRfThreads, EPT>(ehi, eid, m2, k, rk, tid, &ts_s, shi_s);
  float* os = a.out_s + (size_t)q * k;
  int64_t* oi = a.out_i + (size_t)q * k;
  for (int s = tid; s < m3; s += kRfThreads) {
    const int id = eid[s], rank = rk[s];
    if ((id != INT_MAX) & (rank < k)) { os[rank] = ehi[s]; oi[rank] = id; }
  }
  for (int e = nvalid_s + tid; e < k; e += kRfThreads) { os[e] = -INFINITY; oi[e] = -1; }
}
