// Backward of the block-sparse masked attention (gfx950, f16 / bf16, D = 64 or 128).
//
// The reference has no backward (gpu/triton_attn.py:9-10, README.md:118); this is the
// textbook gradient of o = softmax(scale q k^T, masked) v with the forward's row
// log-sum-exp saved: with P = exp(scale q k^T - lse) on live pairs (0 elsewhere),
//   dV = P^T dO,  dP = dO V^T,  dS = P * (dP - rowsum(dO * O)),
//   dQ = scale dS K,  dK = scale dS^T Q.
// Rows with no live key have P = 0 and get no gradient.
//
// Tiles are 64 x 64 (query block x key block), from the block index built at
// BQ = A = 64 and its transpose (pa_index_transpose).  Two passes, no atomics: dK / dV per
// (key block, head), dQ per (query block, head), each a work-group that walks its list with
// the next tile moving into LDS by DMA while the current one is consumed.  A wave owns one
// 32 x 32 quadrant of every tile from the scores to the accumulators, so nothing passes
// between waves inside a tile.
// Partial tiles are masked from element bitmaps when given, else by evaluating the mask in
// original coordinates (perm_q / perm_kv map index-space rows to them, as in the forward).
#include <math.h>

#include <type_traits>

#include "lds_rows.hpp"

namespace pa {
namespace {

constexpr int kBT = 64;  // tile side (query rows = key rows)

struct BwdK {
  const char* q;
  const char* k;
  const char* v;
  const char* o;
  const char* dout;
  char* dq;
  char* dk;
  char* dv;
  int64_t sb, sn;          // element strides shared by every [BH, N, D] tensor
  const float* lse;        // [BH, N], natural log
  float* dvec;             // [BH, N]: rowsum(dO * O)
  int64_t lse_sb;
  int32_t N, nb;           // nb = N / 64
  float c;                 // scale * log2(e)
  float scale;
  const int32_t* kv_idx;   // [nb, pitch] key blocks of each query block
  const int32_t* kv_num;
  const int8_t* kv_partial;
  int64_t pitch;
  const int32_t* q_idx;    // [nb, tpitch] query blocks of each key block
  const int32_t* q_num;
  const int8_t* q_partial;
  int64_t tpitch;
  const int32_t* kv_bits_off;  // [nb, pitch] bitmap word offsets (-1: full), or NULL
  const uint32_t* kv_bits;     // 64 rows x 2 words per partial tile, row-major
  const int32_t* q_bits_off;   // [nb, tpitch], same offsets in the transposed lists
  const uint32_t* q_bits;      // the same bitmaps transposed (64 columns x 2 words)
  int32_t accumulate;          // add into dq / dk / dv
  // > 0: the tensors (and lse, dvec) are in ORIGINAL order and index-space
  // row r lives at row (r mod 2^qlog2) s + r div 2^qlog2 (the residue-s permutation in
  // closed form); a 64-row tile is then 64 rows s apart
  int32_t residue_s, residue_qlog2;
  const int32_t* kv_order;     // issue order of the key blocks in the dK / dV pass, or NULL
  Pred pred;
};

// Memory row of index-space row r.
__device__ __forceinline__ int64_t mem_row(const BwdK& a, int r) {
  return a.residue_s ? (int64_t)(r & ((1 << a.residue_qlog2) - 1)) * a.residue_s + (r >> a.residue_qlog2) : r;
}

// rowsum(dO * O) in fp32: a row per D / 8 lanes, 16 bytes of each tensor per lane (the
// loads of a wave cover whole rows), summed across the row's lanes.
template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_pre_kernel(const BwdK a, int64_t rows) {
  constexpr int LPR = D / 8;  // lanes per row
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t r = g / LPR;
  const int u = (int)(g % LPR);
  float acc = 0.f;
  if (r < rows) {
    const int64_t bh = r / a.N, i = r - bh * a.N;
    const int64_t off = (bh * a.sb + i * a.sn) * (int64_t)sizeof(T) + 16 * u;
    typedef T t8 __attribute__((ext_vector_type(8)));
    const f32x8 x = __builtin_convertvector(*reinterpret_cast<const t8*>(a.o + off), f32x8);
    const f32x8 y = __builtin_convertvector(*reinterpret_cast<const t8*>(a.dout + off), f32x8);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = __builtin_fmaf(x[e], y[e], acc);
  }
#pragma unroll
  for (int o = LPR / 2; o >= 1; o >>= 1) acc += __shfl_xor(acc, o);
  if (r < rows && u == 0) {
    const int64_t bh = r / a.N, i = r - bh * a.N;
    a.dvec[bh * a.lse_sb + i] = acc;
  }
}

__device__ __forceinline__ int32_t orig_of(const int32_t* perm, int32_t r) { return perm ? perm[r] : r; }

// ---- staged tiles ------------------------------------------------------------------
// A tile of 64 rows of two tensors is brought into LDS by LDS DMA (no staging registers,
// no LDS stores; layout in lds_rows.hpp), two stages deep: the next listed tile moves while
// the current one is consumed, behind one wait and one barrier per tile.
// LDS of both kernels: two stages of two tiles, then per stage 1 KB of row vectors (at 0 and
// 256: two vectors of 64 floats; at 512: the partial tile's bitmap, or without bitmaps the
// original numbers of the tile's rows, and in stage 0 at 768 the mask's terms).
template <int D>
struct Tile : Rows<D> {
  static constexpr int TB = kBT * Rows<D>::ROW;          // bytes of a staged tile
  static constexpr int STAGE = 2 * TB;
  static constexpr int VEC = 1024;
  static constexpr int VEC_OFF = 2 * STAGE;
  static constexpr int TERMS_OFF = VEC_OFF + 768;
  static constexpr int END = VEC_OFF + 2 * VEC;
  static_assert(PA_MAX_TERMS * sizeof(pa_term) <= 256, "the terms fit beside the row numbers");
};

typedef const __attribute__((address_space(3))) int32_t lds_i32;
typedef __attribute__((address_space(3))) float lds_fw;
typedef const __attribute__((address_space(4))) int8_t cbyte;

// DMA of rows 16 w .. 16 w + 15 of a tile of two tensors (heads applied; the tile's first
// row at byte r0b, its rows `pitch` bytes apart: the row pitch, or s times it when the tile
// is gathered through the residue-s basis) into the stage at LDS m0 (dvoff: dma_offsets).
template <int D>
__device__ __forceinline__ void dma_tiles(uint32_t m0, const char* g0, const char* g1, int64_t pitch, int64_t r0b, int w,
                                          const uint32_t* dvoff) {
  const char* a0 = g0 + r0b + 16 * w * pitch;
  const char* a1 = g1 + r0b + 16 * w * pitch;
  const uint32_t mw = m0 + (uint32_t)(16 * w * Tile<D>::ROW);
#pragma unroll
  for (int i = 0; i < Tile<D>::NI; ++i) {
    dma_x4(mw + i * 1024, a0 + Tile<D>::RPI * i * pitch, dvoff[i]);
    dma_x4(mw + Tile<D>::TB + i * 1024, a1 + Tile<D>::RPI * i * pitch, dvoff[i]);
  }
}

// Score elements dead in `word` (bit c of it = row or column c of the 32 the lane's
// elements come from; element i is 8 (i / 4) + 4 G + i % 4) become 0.
__device__ __forceinline__ void mask16(f32x16& p, uint32_t word, int G) {
  const int32_t wv = (int32_t)(word >> (4 * G));
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float pv = p[i];  // (a scalar copy: bit-casting the vector element itself reads element 0)
    const int32_t keep = __builtin_amdgcn_sbfe(wv, 8 * (i >> 2) + (i & 3), 1);
    p[i] = __builtin_bit_cast(float, __builtin_bit_cast(int32_t, pv) & keep);
  }
}

// The lane's 32-bit word of live pairs of a partial tile without bitmaps: bit 8 (i / 4) +
// 4 G + i % 4 set when pair i is live; q_at / k_at give the pair's original positions.
template <typename QF, typename KF>
__device__ __forceinline__ uint32_t live_word(const BwdK& a, const pa_term* terms, int G, QF q_at, KF k_at) {
  uint32_t word = 0u;
#pragma unroll 1
  for (int i = 0; i < 16; ++i) {
    const int b = 8 * (i >> 2) + 4 * G + (i & 3);
    if (pred_live_rolled(terms, a.pred.n_include, a.pred.n_exclude, q_at(b), k_at(b), a.pred.dense_bits,
                         a.pred.dense_words))
      word |= 1u << b;
  }
  return word;
}

// A row's exponent offset -lse log2 e, -inf for a row with no live key (its P is then 0).
__device__ __forceinline__ float neg_lse2(float lse) {
  return lse == -INFINITY ? -INFINITY : -lse * 1.4426950408889634f;
}

template <typename T>
__device__ __forceinline__ void to_frags(const f32x16& x, typename Mma<T>::frag* f) {
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    f32x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = x[8 * c + e];
    f[c] = Mma<T>::cvt(v);
  }
}

// The gradient rows of a work-group: each of its waves holds a partial X^T of one 32-row
// half (half = the rows' half, part = which of the 2 NG partials), block db element
// (i4, e) = column 32 db + 8 i4 + 4 G + e of row 32 half + m.  The partials go through LDS
// (fp32, 16-byte units swizzled by row), are added, scaled, and leave as whole rows.
// Thread t takes 8 columns of row (t + NT j) / (D / 8); with accumulate the stored rows are
// loaded ahead (OldRows), so that their latency runs beside the last tile and the exchange.
template <typename T, int D, int NG>
struct OldRows {
  static constexpr int NT = 256 * NG;
  static constexpr int N = kBT * (D / 8) / NT;
  typedef T t8 __attribute__((ext_vector_type(8)));
  u32x4 x[N];
  __device__ __forceinline__ static t8* at(const BwdK& a, char* head, int row0, int tid, int j) {
    const int g = tid + NT * j, r = g / (D / 8), u = g % (D / 8);
    return reinterpret_cast<t8*>(head + mem_row(a, row0 + r) * a.sn * 2 + 16 * u);
  }
  __device__ __forceinline__ void load(const BwdK& a, char* head, int row0, int tid) {
    if (a.accumulate) {
#pragma unroll
      for (int j = 0; j < N; ++j) x[j] = *reinterpret_cast<const u32x4*>(at(a, head, row0, tid, j));
    }
  }
};
template <typename T, int D, int NG>
__device__ __forceinline__ void store_rows(const BwdK& a, char* smem, const f32x16* acc, int half, int part, int tid,
                                           char* head, int row0, float scale, const OldRows<T, D, NG>& old) {
  constexpr int NDB = D / 32, FU = D / 4;  // 16-byte units of a row of floats
  using O = OldRows<T, D, NG>;
  const int lane = tid & 63, G = lane >> 5, m = lane & 31;
  lds_char_t* st = (lds_char_t*)smem;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4 x = {acc[db][4 * i4], acc[db][4 * i4 + 1], acc[db][4 * i4 + 2], acc[db][4 * i4 + 3]};
      *(lds_f4w*)(st + ((part * 2 + half) * 32 + m) * (D * 4) + 16 * ((8 * db + 2 * i4 + G) ^ (m & 15))) = x;
    }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < O::N; ++j) {
    const int g = tid + O::NT * j, r = g / (D / 8), u = g % (D / 8);
    f32x8 x;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int at = r * (D * 4) + 16 * ((2 * u + k) ^ (r & 15));
      f32x4 y = *(lds_f4*)(st + at);
#pragma unroll
      for (int pt = 1; pt < 2 * NG; ++pt) y += *(lds_f4*)(st + pt * kBT * FU * 16 + at);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * k + e] = y[e] * scale;
    }
    if (a.accumulate) x += __builtin_convertvector(__builtin_bit_cast(typename O::t8, old.x[j]), f32x8);
    *O::at(a, head, row0, tid, j) = __builtin_convertvector(x, typename O::t8);
  }
}

// ---------------------------------------------------------------------------------
// dK / dV.  Work-group: 4 waves, one key block of 64; wave (kh, qh) takes keys 32 kh ..
// +31 and, of every listed query block (a staged tile of Q and dO), rows 32 qh .. +31:
//   S = Q K^T, P = exp(scale S - lse) (masked), dP = dO V^T, dS = P (dP - rowsum(dO O)),
//   dV^T += dO^T P, dK^T += Q^T dS,
// all on 32x32 MFMAs with the keys along the lanes, so P and dS are formed in the layout
// the transposed products take them in: nothing passes between waves inside a tile, and
// the one barrier per tile is the stage's.  The two query halves' partials are added
// through LDS at the end.
//
// What bounds it: on long lists the MFMAs (causal, 32 heads x 8192, D = 128, bf16: both
// kernels together 1.9 ms, 1.0 PFLOP/s of the 14 D per pair they issue, 80% of a large
// torch matmul's rate); on short lists each item's start and end and its rows' bytes (band and
// lattice below, lists of about 7 tiles: matrix cores busy 24% of the SIMDs' clocks in the
// band's launches and 33% in the lattice's).  Two waves per SIMD is what the registers allow
// at D = 128 (dK and dV take 128 of 256; K in registers, V in LDS but for one fragment, address
// halves recomputed: 247 with bitmaps, 251 without, none spilled).  Without bitmaps at D = 64
// three waves with 8 spilled registers take 360 us where two with none take 370 (causal, 15 x
// 8192).
// Splitting a tile by quadrants replaced a pair of waves per 32 keys, one for P and dV and
// one for dP and dK, that met at a barrier in the middle of every tile with P in LDS
// (D = 128), and register-staged tiles that evaluated the mask and waited for each tile
// (D = 64).  Measured: 32 heads x 16384 of band-256 | lattice-16 in bf16, D = 128, 1625 ->
// 1260 us; causal, 8 heads x 4032 in f16, D = 64, 402 -> 100 us.
//
// NG groups of 4 waves share a work-group's list, group g taking tiles g, g + NG, ...; the
// groups' partials are added with the halves'.  See launch_bwd for when.
// The phases of a tile kept apart for the scheduler at D = 64 (108.6 -> 104 us of the causal
// case above); at D = 128 it does better left alone (1302 -> 1289 us of the band and lattice).
#define PA_FENCE() \
  if constexpr (D == 64) __builtin_amdgcn_sched_barrier(0)
template <int D>
constexpr int v_in_regs() { return D == 64 ? 4 : 1; }  // V fragments kept in registers
template <int D, int NG>
constexpr int dkdv_smem() { return NG * Tile<D>::END + 2 * (D / 16 - v_in_regs<D>()) * 1024; }

template <typename T, int D, bool BITS, int NG>
__global__ __launch_bounds__(256 * NG) __attribute__((amdgpu_waves_per_eu(D == 64 && NG == 1 ? 3 : 2)))
void bwd_dkdv_kernel(const BwdK a) {
  using Frag = typename Mma<T>::frag;
  using TL = Tile<D>;
  constexpr int ESZ = 2, NKC = D / 16, NDB = D / 32;
  constexpr int NVR = v_in_regs<D>(), NVL = NKC - NVR;
  extern __shared__ __attribute__((aligned(256))) char smem[];
  pa_term* terms_s = reinterpret_cast<pa_term*>(smem + TL::TERMS_OFF);
  if constexpr (!BITS) {
#pragma unroll
    for (int i = 0; i < PA_MAX_TERMS; ++i)  // (constant indices into the argument block)
      if (threadIdx.x == i) terms_s[i] = a.pred.terms[i];
  }

  const int tid = threadIdx.x, lane = tid & 63, G = lane >> 5, m = lane & 31;
  const int wg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = NG == 1 ? 0 : wg >> 2, w = wg & 3;
  char* gsm = smem + grp * TL::END;  // this group's stages and vectors
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char_t*)gsm;
  lds_cptr lds = (lds_cptr)gsm;
  const int kh = w >> 1, qh = w & 1;
  const int64_t id = xcd_remap(blockIdx.x, (int64_t)gridDim.x);
  const int kr = snake((int)(id % a.nb), a.nb);
  const int kb = a.kv_order ? ((cint*)a.kv_order)[kr] : kr;
  const int64_t bh = gridDim.x / a.nb - 1 - id / a.nb;
  const int key = kb * kBT + kh * 32 + m;
  const int key_o = orig_of(a.pred.perm_kv, key);
  const int64_t rowb = a.sn * ESZ;
  const int rs = a.residue_s ? a.residue_s : 1;
  const int64_t pitch = rs * rowb;
  const char* hq = a.q + bh * a.sb * ESZ;
  const char* hdo = a.dout + bh * a.sb * ESZ;
  const float* hlse = a.lse + bh * a.lse_sb;
  const char* hdvec = reinterpret_cast<const char*>(a.dvec + bh * a.lse_sb);
  const char* hperm = reinterpret_cast<const char*>(a.pred.perm_q);

  uint32_t dvoff[TL::NI];
  dma_offsets<D>(dvoff, pitch, lane);
  // Query block qb into stage S: the rows of Q and dO by every wave, rowsum(dO O) by wave 1,
  // a partial tile's bitmap (bo >= 0) by waves 2 and 3 or, without bitmaps, the original row
  // numbers by wave 2.  The lse goes through registers (lse_n): once it has arrived, put_lse
  // writes it as the exponent offset (wave 0) and keeps which of the wave's 32 rows have no
  // weight (lse = -inf: P is 0 also where their scores are NaN).
  float lse_n = 0.f;
  uint32_t dead_n = 0u;
  auto dma = [&](int qb, int bo, int S) __attribute__((always_inline)) {
    const int64_t r0 = mem_row(a, qb * kBT);
    lse_n = hlse[r0 + rs * lane];
    dma_tiles<D>(lds0 + S * TL::STAGE, hq, hdo, pitch, r0 * rowb, w, dvoff);
    const uint32_t mv = lds0 + TL::VEC_OFF + S * TL::VEC;
    if (w == 1) dma_x1(mv + 256, hdvec + r0 * 4, 4u * rs * lane);
    if constexpr (BITS) {
      if (w >= 2 && bo >= 0)
        dma_x1(mv + 512 + 256 * (w - 2), reinterpret_cast<const char*>(a.q_bits + bo) + 256 * (w - 2), 4u * lane);
    } else if (hperm && w == 2) {
      dma_x1(mv + 512, hperm + (int64_t)qb * 256, 4u * lane);
    }
  };
  auto put_lse = [&](int S) __attribute__((always_inline)) {
    if (w == 0) *(lds_fw*)((lds_char_t*)gsm + TL::VEC_OFF + S * TL::VEC + 4 * lane) = neg_lse2(lse_n);
    dead_n = (uint32_t)(__ballot(lse_n == -INFINITY) >> (32 * qh));
  };

  const TileReads<D> rd = tile_reads<D>(lds + 32 * qh * TL::ROW, lane);
  lds_cptr vrow = lds + TL::VEC_OFF + 128 * qh + 16 * G;  // row vector entries 8 j + 4 G + 0..3

  // K in registers; V partly in registers, the rest in LDS in fragment order (the
  // accumulators of dK and dV already take half of a wave's registers).  Their rows come
  // through stage 1, moved beside the first tile.
  Frag kf[NKC], vf[NKC];
  lds_char_t* vl = (lds_char_t*)smem + NG * TL::END + kh * NVL * 1024 + lane * 16;
  f32x16 dkt[NDB], dvt[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) dkt[i] = dvt[i] = f32x16{0};

  auto tile = [&](auto SC, bool partial, int qb, uint32_t dead) __attribute__((always_inline)) {
    constexpr int S = decltype(SC)::value;
    constexpr int SO = S * TL::STAGE;
    // element i of the lane: query row 32 qh + 8 (i / 4) + 4 G + i % 4, key `key`
    f32x16 s = f32x16{0}, dp = f32x16{0};
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc)
      s = Mma<T>::mma(__builtin_bit_cast(Frag, *(lds_u4*)(rd.row(kc) + SO)), kf[kc], s);
    PA_FENCE();
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc) {
      const Frag vx = kc < NVR ? vf[kc] : __builtin_bit_cast(Frag, *(lds_u4*)(vl + (kc - NVR) * 1024));
      dp = Mma<T>::mma(__builtin_bit_cast(Frag, *(lds_u4*)(rd.row(kc) + SO + TL::TB)), vx, dp);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 nl = *(lds_f4*)(vrow + S * TL::VEC + 32 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        s[4 * j + e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * j + e], a.c, nl[e]));
    }
    // (dead rows with the bitmap where there is one, apart where the mask is evaluated: the
    // other way round costs 2% at D = 128 and spills 8 registers)
    if (partial || (BITS && dead != 0u)) {
      uint32_t word = ~0u;
      if constexpr (BITS) {
        if (partial) word = *(lds_u32*)(lds + TL::VEC_OFF + S * TL::VEC + 512 + (32 * kh + m) * 8 + 4 * qh);
        word &= ~dead;
      } else {
        lds_i32* qo = (lds_i32*)(lds + TL::VEC_OFF + S * TL::VEC + 512 + 128 * qh);
        word = live_word(a, terms_s, G, [&](int b) { return hperm ? qo[b] : qb * kBT + 32 * qh + b; },
                         [&](int) { return key_o; });
      }
      mask16(s, word, G);
    }
    if (!BITS && dead != 0u) mask16(s, ~dead, G);
    PA_FENCE();
    Frag pf[2], sf[2];
    to_frags<T>(s, pf);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int db = 0; db < NDB; ++db)
        dvt[db] = Mma<T>::mma(tr_frag<T, D>(rd, db, SO + TL::TB + 16 * c * TL::ROW), pf[c], dvt[db]);
    PA_FENCE();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 dv = *(lds_f4*)(vrow + S * TL::VEC + 256 + 32 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * j + e] *= dp[4 * j + e] - dv[e];
    }
    to_frags<T>(s, sf);
    PA_FENCE();
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int db = 0; db < NDB; ++db)
        dkt[db] = Mma<T>::mma(tr_frag<T, D>(rd, db, SO + 16 * c * TL::ROW), sf[c], dkt[db]);
  };

  const int nl = ((cint*)a.q_num)[kb];
  cint* qlist = (cint*)(a.q_idx + (int64_t)kb * a.tpitch);
  cbyte* plist = (cbyte*)(a.q_partial + (int64_t)kb * a.tpitch);
  cint* olist = (cint*)(BITS ? a.q_bits_off + (int64_t)kb * a.tpitch : a.q_idx);
  auto tile_of = [&](int t, int& qb, int& bo) __attribute__((always_inline)) {
    qb = qlist[t];
    bo = BITS ? olist[t] : (plist[t] != 0 ? 0 : -1);
  };
  int qb_c = 0, bo_c = -1, qb_n = 0, bo_n = -1;
  if (nl > 0) {
    if (grp < nl) {
      tile_of(grp, qb_c, bo_c);
      dma(qb_c, bo_c, 0);
    }
    dma_tiles<D>(lds0 + TL::STAGE, a.k + bh * a.sb * ESZ, a.v + bh * a.sb * ESZ, pitch, mem_row(a, kb * kBT) * rowb, w,
                 dvoff);
    put_lse(0);
    if (NG + grp < nl) tile_of(NG + grp, qb_n, bo_n);
    dma_wait_all();
    __syncthreads();
    const TileReads<D> kd = tile_reads<D>(lds + TL::STAGE + 32 * kh * TL::ROW, lane);
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc) {
      kf[kc] = __builtin_bit_cast(Frag, *(lds_u4*)(kd.row(kc)));
      vf[kc] = __builtin_bit_cast(Frag, *(lds_u4*)(kd.row(kc) + TL::TB));
    }
    if (grp == 0 && qh == 0) {
#pragma unroll
      for (int kc = NVR; kc < NKC; ++kc) *(lds_u4w*)(vl + (kc - NVR) * 1024) = __builtin_bit_cast(u32x4, vf[kc]);
    }
  }
  auto step = [&](auto SC, int t) __attribute__((always_inline)) {
    constexpr int S = decltype(SC)::value;
    dma_wait_all();
    __syncthreads();  // stage S is in; every wave is past stage S ^ 1
    if (t + NG < nl) dma(qb_n, bo_n, S ^ 1);
    const int qb = qb_c;
    const uint32_t dead = dead_n;
    const bool partial = bo_c >= 0;
    qb_c = qb_n;
    bo_c = bo_n;
    if (t + 2 * NG < nl) tile_of(t + 2 * NG, qb_n, bo_n);
    if (NG == 1 || t < nl) tile(SC, partial, qb, dead);
    if (t + NG < nl) put_lse(S ^ 1);
  };
  // (every group takes every step: the last one may have no tile for it)
  const int ns = (nl + NG - 1) / NG;
  int t = 0;
  for (; t + 1 < ns; t += 2) {
    step(std::integral_constant<int, 0>{}, t * NG + grp);
    step(std::integral_constant<int, 1>{}, (t + 1) * NG + grp);
  }
  if (t < ns) step(std::integral_constant<int, 0>{}, t * NG + grp);

  char* hdv = a.dv + bh * a.sb * ESZ;
  char* hdk = a.dk + bh * a.sb * ESZ;
  OldRows<T, D, NG> odv, odk;
  odv.load(a, hdv, kb * kBT, tid);
  odk.load(a, hdk, kb * kBT, tid);
  __syncthreads();  // every wave is past its tiles
  store_rows<T, D, NG>(a, smem, dvt, kh, 2 * grp + qh, tid, hdv, kb * kBT, 1.f, odv);
  __syncthreads();
  store_rows<T, D, NG>(a, smem, dkt, kh, 2 * grp + qh, tid, hdk, kb * kBT, a.scale, odk);
}

// ---------------------------------------------------------------------------------
// dQ, the same with the roles of queries and keys exchanged (the forward's layout): wave
// (qh, kh) takes query rows 32 qh .. +31 of the work-group's block and, of every listed key
// block (a staged tile of K and V), keys 32 kh .. +31:
//   S^T = K Q^T, dP^T = V dO^T, dQ^T += K^T dS^T,
// with the queries along the lanes; the two key halves' partials are added at the end.
template <typename T, int D, bool BITS, int NG>
__global__ __launch_bounds__(256 * NG) __attribute__((amdgpu_waves_per_eu(D == 64 && NG == 1 ? 3 : 2)))
void bwd_dq_kernel(const BwdK a) {
  using Frag = typename Mma<T>::frag;
  using TL = Tile<D>;
  constexpr int ESZ = 2, NKC = D / 16, NDB = D / 32;
  extern __shared__ __attribute__((aligned(256))) char smem[];
  pa_term* terms_s = reinterpret_cast<pa_term*>(smem + TL::TERMS_OFF);
  if constexpr (!BITS) {
#pragma unroll
    for (int i = 0; i < PA_MAX_TERMS; ++i)
      if (threadIdx.x == i) terms_s[i] = a.pred.terms[i];
  }

  const int tid = threadIdx.x, lane = tid & 63, G = lane >> 5, m = lane & 31;
  const int wg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = NG == 1 ? 0 : wg >> 2, w = wg & 3;
  char* gsm = smem + grp * TL::END;  // this group's stages and vectors
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char_t*)gsm;
  lds_cptr lds = (lds_cptr)gsm;
  const int qh = w >> 1, kh = w & 1;
  const int64_t id = xcd_remap(blockIdx.x, (int64_t)gridDim.x);
  // the last query blocks first: a causal mask's lists grow along the sequence, and the
  // longest should not be the last to start
  const int qb = a.nb - 1 - snake((int)(id % a.nb), a.nb);
  const int64_t bh = id / a.nb;
  const int row = qb * kBT + qh * 32 + m;  // this lane's query row (index space)
  const int q_o = orig_of(a.pred.perm_q, row);
  const int64_t row_m = mem_row(a, row);
  const int64_t rowb = a.sn * ESZ;
  const int rs = a.residue_s ? a.residue_s : 1;
  const int64_t pitch = rs * rowb;
  const char* hk = a.k + bh * a.sb * ESZ;
  const char* hv = a.v + bh * a.sb * ESZ;
  const char* hperm = reinterpret_cast<const char*>(a.pred.perm_kv);

  uint32_t dvoff[TL::NI];
  dma_offsets<D>(dvoff, pitch, lane);
  // key block kb into stage S: the rows of K and V by every wave, a partial tile's bitmap
  // (bo >= 0) by waves 0 and 1 or, without bitmaps, the original key numbers by wave 0
  auto dma = [&](int kb, int bo, int S) __attribute__((always_inline)) {
    dma_tiles<D>(lds0 + S * TL::STAGE, hk, hv, pitch, mem_row(a, kb * kBT) * rowb, w, dvoff);
    const uint32_t mv = lds0 + TL::VEC_OFF + S * TL::VEC + 512;
    if constexpr (BITS) {
      if (w < 2 && bo >= 0) dma_x1(mv + 256 * w, reinterpret_cast<const char*>(a.kv_bits + bo) + 256 * w, 4u * lane);
    } else if (hperm && w == 0) {
      dma_x1(mv, hperm + (int64_t)kb * 256, 4u * lane);
    }
  };

  const TileReads<D> rd = tile_reads<D>(lds + 32 * kh * TL::ROW, lane);

  // Q and dO in registers: their rows come through stage 1, moved beside the first tile
  Frag qf[NKC], df[NKC];
  const float nl2 = neg_lse2(a.lse[bh * a.lse_sb + row_m]);
  const float dr = a.dvec[bh * a.lse_sb + row_m];
  const bool dead = nl2 == -INFINITY;  // a row with no weight: P is 0 also where its scores are NaN
  const bool any_dead = __ballot(dead) != 0ull;
  f32x16 dqt[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) dqt[i] = f32x16{0};

  auto tile = [&](auto SC, bool partial, int kb) __attribute__((always_inline)) {
    constexpr int S = decltype(SC)::value;
    constexpr int SO = S * TL::STAGE;
    // element i of the lane: key 32 kh + 8 (i / 4) + 4 G + i % 4, query `row`
    f32x16 s = f32x16{0}, dp = f32x16{0};
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc)
      s = Mma<T>::mma(__builtin_bit_cast(Frag, *(lds_u4*)(rd.row(kc) + SO)), qf[kc], s);
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc)
      dp = Mma<T>::mma(__builtin_bit_cast(Frag, *(lds_u4*)(rd.row(kc) + SO + TL::TB)), df[kc], dp);
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.c, nl2));
    if (partial) {
      uint32_t word;
      if constexpr (BITS) {
        word = *(lds_u32*)(lds + TL::VEC_OFF + S * TL::VEC + 512 + (32 * qh + m) * 8 + 4 * kh);
      } else {
        lds_i32* ko = (lds_i32*)(lds + TL::VEC_OFF + S * TL::VEC + 512 + 128 * kh);
        word = live_word(a, terms_s, G, [&](int) { return q_o; },
                         [&](int b) { return hperm ? ko[b] : kb * kBT + 32 * kh + b; });
      }
      mask16(s, word, G);
    }
    if (any_dead) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = dead ? 0.f : s[i];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] *= dp[i] - dr;
    Frag sf[2];
    to_frags<T>(s, sf);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int db = 0; db < NDB; ++db)
        dqt[db] = Mma<T>::mma(tr_frag<T, D>(rd, db, SO + 16 * c * TL::ROW), sf[c], dqt[db]);
  };

  const int nl = ((cint*)a.kv_num)[qb];
  cint* klist = (cint*)(a.kv_idx + (int64_t)qb * a.pitch);
  cbyte* plist = (cbyte*)(a.kv_partial + (int64_t)qb * a.pitch);
  cint* olist = (cint*)(BITS ? a.kv_bits_off + (int64_t)qb * a.pitch : a.kv_idx);
  auto tile_of = [&](int t, int& kb, int& bo) __attribute__((always_inline)) {
    kb = klist[t];
    bo = BITS ? olist[t] : (plist[t] != 0 ? 0 : -1);
  };
  int kb_c = 0, bo_c = -1, kb_n = 0, bo_n = -1;
  if (nl > 0) {
    if (grp < nl) {
      tile_of(grp, kb_c, bo_c);
      dma(kb_c, bo_c, 0);
    }
    dma_tiles<D>(lds0 + TL::STAGE, a.q + bh * a.sb * ESZ, a.dout + bh * a.sb * ESZ, pitch, mem_row(a, qb * kBT) * rowb, w,
                 dvoff);
    if (NG + grp < nl) tile_of(NG + grp, kb_n, bo_n);
    dma_wait_all();
    __syncthreads();
    const TileReads<D> qd = tile_reads<D>(lds + TL::STAGE + 32 * qh * TL::ROW, lane);
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc) {
      qf[kc] = __builtin_bit_cast(Frag, *(lds_u4*)(qd.row(kc)));
      df[kc] = __builtin_bit_cast(Frag, *(lds_u4*)(qd.row(kc) + TL::TB));
    }
  }
  auto step = [&](auto SC, int t) __attribute__((always_inline)) {
    constexpr int S = decltype(SC)::value;
    dma_wait_all();
    __syncthreads();
    if (t + NG < nl) dma(kb_n, bo_n, S ^ 1);
    const int kb = kb_c;
    const bool partial = bo_c >= 0;
    kb_c = kb_n;
    bo_c = bo_n;
    if (t + 2 * NG < nl) tile_of(t + 2 * NG, kb_n, bo_n);
    if (NG == 1 || t < nl) tile(SC, partial, kb);
  };
  // (every group takes every step: the last one may have no tile for it)
  const int ns = (nl + NG - 1) / NG;
  int t = 0;
  for (; t + 1 < ns; t += 2) {
    step(std::integral_constant<int, 0>{}, t * NG + grp);
    step(std::integral_constant<int, 1>{}, (t + 1) * NG + grp);
  }
  if (t < ns) step(std::integral_constant<int, 0>{}, t * NG + grp);

  char* hdq = a.dq + bh * a.sb * ESZ;
  OldRows<T, D, NG> odq;
  odq.load(a, hdq, qb * kBT, tid);
  __syncthreads();  // every wave is past its tiles
  store_rows<T, D, NG>(a, smem, dqt, qh, 2 * grp + kh, tid, hdq, qb * kBT, a.scale, odq);
}

// Transposed block lists: for key block kb, the query blocks whose list holds kb, in
// ascending order, with the partial flag.  One thread per key block; each query block's
// list is sorted, so membership is a binary search.  q_idx == nullptr: counts only.
__global__ __launch_bounds__(256) void transpose_kernel(const int32_t* kv_idx, const int32_t* kv_num,
                                                        const int8_t* kv_partial, const int32_t* kv_bits_off,
                                                        int32_t nq, int64_t pitch, int32_t nk, int32_t* q_num,
                                                        int32_t* q_idx, int8_t* q_partial, int32_t* q_bits_off,
                                                        int64_t tp) {
  const int kb = blockIdx.x * 256 + threadIdx.x;
  if (kb >= nk) return;
  int n = 0;
  for (int qb = 0; qb < nq; ++qb) {
    const int32_t* row = kv_idx + (int64_t)qb * pitch;
    int lo = 0, hi = kv_num[qb];
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (row[mid] < kb)
        lo = mid + 1;
      else
        hi = mid;
    }
    if (lo < kv_num[qb] && row[lo] == kb) {
      if (q_idx && n < tp) {
        q_idx[(int64_t)kb * tp + n] = qb;
        q_partial[(int64_t)kb * tp + n] = kv_partial[(int64_t)qb * pitch + lo];
        if (q_bits_off) q_bits_off[(int64_t)kb * tp + n] = kv_bits_off[(int64_t)qb * pitch + lo];
      }
      ++n;
    }
  }
  q_num[kb] = n;
}

// One 64 x 64 bitmap per work-group of 64 threads (listed tile j of query block i, when
// kv_bits_off[i, j] >= 0): thread k assembles column k from the 64 row words.
__global__ __launch_bounds__(64) void bits_transpose_kernel(const int32_t* kv_bits_off, int64_t pitch,
                                                             const uint32_t* kv_bits, uint32_t* q_bits) {
  const int64_t off = kv_bits_off[(int64_t)blockIdx.y * pitch + blockIdx.x];
  if (off < 0) return;
  const int k = threadIdx.x;
  uint32_t col[2] = {0u, 0u};
#pragma unroll 8
  for (int r = 0; r < 64; ++r) col[r >> 5] |= ((kv_bits[off + 2 * r + (k >> 5)] >> (k & 31)) & 1u) << (r & 31);
  q_bits[off + 2 * k] = col[0];
  q_bits[off + 2 * k + 1] = col[1];
}

template <typename T, int D, bool BITS, int NG>
int launch_bwd_t(const BwdK& k, int64_t BH, hipStream_t s) {
  constexpr int kv_smem = dkdv_smem<D, NG>(), q_smem = NG * Tile<D>::END;
  // the dynamic LDS limit is raised once per device
  static unsigned long long configured = 0ull;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev >= 64 || !((configured >> dev) & 1ull)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&bwd_dkdv_kernel<T, D, BITS, NG>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kv_smem);
    if (e == hipSuccess)
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(&bwd_dq_kernel<T, D, BITS, NG>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, q_smem);
    if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(bwd kernels)");
    if (dev < 64) configured |= 1ull << dev;
  }
  const unsigned grid = (unsigned)(k.nb * BH);
  hipLaunchKernelGGL((bwd_dkdv_kernel<T, D, BITS, NG>), dim3(grid), dim3(256 * NG), kv_smem, s, k);
  PA_LAUNCH_CHECK("bwd_dkdv_kernel");
  hipLaunchKernelGGL((bwd_dq_kernel<T, D, BITS, NG>), dim3(grid), dim3(256 * NG), q_smem, s, k);
  PA_LAUNCH_CHECK("bwd_dq_kernel");
  return PA_OK;
}

// Two groups of waves per list where one would leave the chip waiting for its longest
// lists: a work-group for every CU or fewer, or up to two with a list of 32 tiles or more.
// One group / two, both kernels and the pre-pass, causal f16 D = 64: 64 work-groups (longest
// list 32) 54.0 / 39.3 us, 504 (63) 107.6 / 101.4 us; window 512, bf16, 448 work-groups
// (9): 33.5 / 38.8 us; causal, 1024 work-groups (64): 162.6 / 179.4 us.
template <typename T, int D>
int launch_bwd(const BwdK& k, int64_t BH, bool dvec_given, hipStream_t s) {
  const int64_t rows = BH * k.N;
  if (!dvec_given) {
    hipLaunchKernelGGL((bwd_pre_kernel<T, D>), dim3((unsigned)((rows * (D / 8) + 255) / 256)), dim3(256), 0, s, k,
                       rows);
    PA_LAUNCH_CHECK("bwd_pre_kernel");
  }
  if (!k.q_bits) return launch_bwd_t<T, D, false, 1>(k, BH, s);
  const int64_t grid = k.nb * BH, longest = k.tpitch > k.pitch ? k.tpitch : k.pitch;
  const bool two = grid <= 256 || (grid <= 512 && longest >= 32);
  return two ? launch_bwd_t<T, D, true, 2>(k, BH, s) : launch_bwd_t<T, D, true, 1>(k, BH, s);
}

}  // namespace
}  // namespace pa

extern "C" int pa_index_transpose(const int32_t* kv_idx, const int32_t* kv_num, const int8_t* kv_partial,
                                  const int32_t* kv_bits_off, int32_t nq, int64_t pitch, int32_t nk, int32_t* q_num,
                                  int32_t* q_idx, int8_t* q_partial, int32_t* q_bits_off, int64_t tpitch,
                                  void* stream) {
  PA_CHECK_ARG(kv_num && q_num && nq >= 1 && nk >= 1 && pitch >= 0 && tpitch >= 0, "pa_index_transpose: bad arguments");
  PA_CHECK_ARG(pitch == 0 || (kv_idx && kv_partial), "pa_index_transpose: null kv_idx / kv_partial");
  PA_CHECK_ARG(!q_idx || q_partial, "pa_index_transpose: q_idx needs q_partial");
  PA_CHECK_ARG(!q_bits_off || (kv_bits_off && q_idx), "pa_index_transpose: q_bits_off needs kv_bits_off and q_idx");
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(pa::transpose_kernel, dim3((unsigned)((nk + 255) / 256)), dim3(256), 0, s, kv_idx, kv_num,
                     kv_partial, kv_bits_off, nq, pitch, nk, q_num, q_idx, q_partial, q_bits_off, tpitch);
  PA_LAUNCH_CHECK("transpose_kernel");
  return PA_OK;
}

extern "C" int pa_index_bits_transpose(const int32_t* kv_bits_off, int32_t nq, int64_t pitch, const uint32_t* kv_bits,
                                       uint32_t* q_bits, void* stream) {
  PA_CHECK_ARG(nq >= 1 && nq <= 65535 && pitch >= 0 && pitch < (1ll << 31), "pa_index_bits_transpose: nq=%d pitch=%lld",
               nq, (long long)pitch);
  if (pitch == 0) return PA_OK;
  PA_CHECK_ARG(kv_bits_off && kv_bits && q_bits, "pa_index_bits_transpose: null array");
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(pa::bits_transpose_kernel, dim3((unsigned)pitch, (unsigned)nq), dim3(64), 0, s, kv_bits_off,
                     pitch, kv_bits, q_bits);
  PA_LAUNCH_CHECK("bits_transpose_kernel");
  return PA_OK;
}

extern "C" int pa_attn_bwd(const pa_attn_bwd_args* x, void* stream) {
  PA_CHECK_ARG(x, "pa_attn_bwd: null arguments");
  PA_CHECK_ARG(x->dtype == PA_BF16 || x->dtype == PA_F16, "pa_attn_bwd: dtype must be f16 or bf16");
  PA_CHECK_ARG(x->D == 64 || x->D == 128, "pa_attn_bwd: D=%d (64 or 128)", x->D);
  PA_CHECK_ARG(x->BH >= 1 && x->BH <= 65535, "pa_attn_bwd: BH=%lld", (long long)x->BH);
  PA_CHECK_ARG(x->N >= 64 && x->N % 64 == 0 && x->N < (1ll << 31), "pa_attn_bwd: N=%lld must be a multiple of 64",
               (long long)x->N);
  PA_CHECK_ARG(x->q && x->k && x->v && x->o && x->dout && x->dq && x->dk && x->dv && x->lse && x->dvec,
               "pa_attn_bwd: null tensor");
  PA_CHECK_ARG(x->kv_num && x->q_num && (x->pitch == 0 || (x->kv_idx && x->kv_partial)) &&
                   (x->tpitch == 0 || (x->q_idx && x->q_partial)),
               "pa_attn_bwd: null index array");
  PA_CHECK_ARG(x->lse_sb >= x->N, "pa_attn_bwd: lse_sb=%lld < N=%lld (lse and dvec rows must not overlap)",
               (long long)x->lse_sb, (long long)x->N);
  PA_CHECK_ARG(x->sn >= x->D && x->sb >= x->sn && x->sn < (1ll << 28), "pa_attn_bwd: strides sb=%lld sn=%lld",
               (long long)x->sb, (long long)x->sn);
  PA_CHECK_ARG((x->N / 64) * x->BH < (1ll << 31), "pa_attn_bwd: %lld blocks x %lld heads exceed one launch",
               (long long)(x->N / 64), (long long)x->BH);
  auto al = [&](const void* p) { return (reinterpret_cast<uintptr_t>(p) % 16) == 0; };
  PA_CHECK_ARG(al(x->q) && al(x->k) && al(x->v) && al(x->o) && al(x->dout) && al(x->dq) && al(x->dk) && al(x->dv) &&
                   (x->sn * 2) % 16 == 0 && (x->sb * 2) % 16 == 0,
               "pa_attn_bwd: rows must be 16-byte aligned");
  const int rc = pa::check_mask(&x->mask, x->N);
  if (rc) return rc;
  pa::BwdK k;
  k.q = static_cast<const char*>(x->q);
  k.k = static_cast<const char*>(x->k);
  k.v = static_cast<const char*>(x->v);
  k.o = static_cast<const char*>(x->o);
  k.dout = static_cast<const char*>(x->dout);
  k.dq = static_cast<char*>(x->dq);
  k.dk = static_cast<char*>(x->dk);
  k.dv = static_cast<char*>(x->dv);
  k.sb = x->sb;
  k.sn = x->sn;
  k.lse = x->lse;
  k.dvec = x->dvec;
  k.lse_sb = x->lse_sb;
  k.N = (int32_t)x->N;
  k.nb = (int32_t)(x->N / 64);
  k.scale = x->scale > 0.f ? x->scale : 1.f / sqrtf((float)x->D);
  k.c = k.scale * 1.4426950408889634f;
  k.kv_idx = x->kv_idx;
  k.kv_num = x->kv_num;
  k.kv_partial = x->kv_partial;
  k.pitch = x->pitch;
  k.q_idx = x->q_idx;
  k.q_num = x->q_num;
  k.q_partial = x->q_partial;
  k.tpitch = x->tpitch;
  const bool nb_ = !x->kv_bits_off, nk_ = !x->kv_bits, qo_ = !x->q_bits_off, qk_ = !x->q_bits;
  PA_CHECK_ARG(nb_ == nk_ && nb_ == qo_ && nb_ == qk_, "pa_attn_bwd: the four bitmap arrays are all NULL or all given");
  k.kv_bits_off = x->kv_bits_off;
  k.kv_bits = x->kv_bits;
  k.q_bits_off = x->q_bits_off;
  k.q_bits = x->q_bits;
  PA_CHECK_ARG((x->flags & ~(PA_BWD_ACCUMULATE | PA_BWD_DVEC_GIVEN)) == 0, "pa_attn_bwd: unknown flags %d", x->flags);
  k.accumulate = (x->flags & PA_BWD_ACCUMULATE) != 0;
  k.residue_s = 0;
  k.residue_qlog2 = 0;
  k.kv_order = x->kv_order;
  if (x->residue_s > 1) {
    const int64_t per = x->N / x->residue_s;
    PA_CHECK_ARG(x->D == 128 && x->N % x->residue_s == 0 && (per & (per - 1)) == 0 && per % 64 == 0,
                 "pa_attn_bwd: residue_s=%d needs D = 128 and N / s a power of two and a multiple of 64 (N=%lld)",
                 x->residue_s, (long long)x->N);
    PA_CHECK_ARG((int64_t)x->residue_s * x->sn * 2 * 4 < (1ll << 32), "pa_attn_bwd: residue_s=%d rows too far apart",
                 x->residue_s);
    k.residue_s = x->residue_s;
    while ((1ll << k.residue_qlog2) < per) ++k.residue_qlog2;
  }
  const bool dg = (x->flags & PA_BWD_DVEC_GIVEN) != 0;
  k.pred = pa::make_pred(x->mask);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (x->dtype == PA_BF16)
    return x->D == 128 ? pa::launch_bwd<__bf16, 128>(k, x->BH, dg, s) : pa::launch_bwd<__bf16, 64>(k, x->BH, dg, s);
  return x->D == 128 ? pa::launch_bwd<_Float16, 128>(k, x->BH, dg, s) : pa::launch_bwd<_Float16, 64>(k, x->BH, dg, s);
}
