// Block-sparse attention forward for f16 / bf16 on block lists as they are (no step
// descriptors, bitmaps optional): D = 64 or 128, BQ = 64 or 128, any A.
//
// Same contract and numerics as attn_fwd_kernel (the replacement of the Triton kernel
// _attn_fwd, gpu/triton_attn.py:62-182): scores transposed (S^T = K Q^T) on 32x32x16 MFMAs,
// online softmax with the finite -1e30 sentinel and a lazy rescale, probabilities rounded
// to 16 bits only as MFMA operands (their sum is taken in fp32 before), the l > 0 guard, and
// the log-sum-exp merge with a previous partial (narrower query blocks: attn_narrow.hip).
// attn_fwd_kernel stages K and V through registers and keeps the rest: f32, K / V gathered
// through a permutation table, class-B emulation.
//
// A work-group is RG row groups (one wave of 32 query rows each; all of the query block's, or
// with H = 2 half of them) times KG key groups.  Key group g takes the 64-column steps g,
// g + KG, ... of the query block's list, its K and V rows by LDS DMA into a two-stage ring of
// its own (layout in lds_rows.hpp), the next step's while this one is computed, behind one
// wait and one barrier per step.  The key groups' states (max, sum, O^T) are merged through
// LDS at the end.
//
// What bounds it: at D = 64 a step's 16 MFMAs take 512 clocks of a SIMD and its exponentials,
// maxima, sums and packing about 850.  With every CU full (causal, 32 heads x 8192, f16: 375
// us, 730 TFLOP/s, about 1500 clocks per wave's step) the VALU is busy 61% of the SIMDs'
// clocks and the matrix cores 33%, less than half of that at the same time: the issue of the
// two, hardly overlapped (2.2 waves per SIMD on average).  On smaller launches the latency of
// a wave's step: causal, 8 x 4096, has 1.1 waves per SIMD, VALU 26%, matrix cores 13%, and
// waits for its longest lists; lattice-8 in its basis, 8 x 16384, 1.5 waves, 40% and 20%.
// Against attn_fwd_kernel: the first case 798 us; 8 heads x
// 4096 causal, 128x128 tiles, f16, D = 64 (no bitmaps) 138 -> 44 us; lattice-8 in its basis,
// 8 heads x 16384, 128x32 tiles 155 -> 64 us; causal, bf16, D = 128, 8 x 4096, 128x128 tiles
// 209 -> 77 us.  A step's scalar work decides much of it (the scalar unit is shared by the
// SIMDs): the list read entry by entry, with its codes worked out per step, took 64 us where
// 16 steps at a time took 55.
//
// The list is held 16 steps at a time, a 16-column segment per lane; a partial block's mask
// word (32 columns of the lane's query row) is loaded from the bitmaps one step ahead, or
// evaluated from the predicate when the index has no bitmaps.
#include <type_traits>

#include "lds_rows.hpp"

namespace pa {
namespace {

template <int D, int KG>
constexpr int tile_smem_bytes() { return KG * 4 * 64 * Rows<D>::ROW; }

// Waves per SIMD that the registers allow (163 to 168 and 246 to 254 in use by the
// instantiations, none spilled; 2 to 27 scalars are).
template <int D>
constexpr int tile_waves() { return D == 64 ? 3 : 2; }

template <typename T, int D, int RG, int KG, int H>
__global__ __launch_bounds__(64 * RG * KG) __attribute__((amdgpu_waves_per_eu(tile_waves<D>())))
void attn_tile_kernel(const AttnK a) {
  using Frag = typename Mma<T>::frag;
  using R = Rows<D>;
  constexpr int ESZ = 2, NQF = D / 16, NDB = D / 32;
  constexpr int TB = 64 * R::ROW;      // a staged tensor
  constexpr int STAGE = 2 * TB;        // K, then V
  constexpr int SPW = 4 / RG;          // 16-row segments a wave moves
  static_assert(4 % RG == 0, "a wave moves whole segments");

  extern __shared__ __attribute__((aligned(256))) char smem[];
  __shared__ pa_term terms_s[PA_MAX_TERMS];

  const int tid = threadIdx.x, lane = tid & 63, G = lane >> 5, m = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = KG == 1 ? 0 : wv / RG, w = KG == 1 ? wv : wv % RG;
  char* ring = smem + kg * 2 * STAGE;
  const uint32_t ring0 = (uint32_t)(uintptr_t)(lds_char_t*)ring;

  const uint32_t lid = xcd_remap32(blockIdx.x, gridDim.x);
  const int np = H * a.nq;  // pieces of a head
  const uint32_t bh_l = lid / (uint32_t)np;
  const int64_t bh = a.heads_desc ? a.BH - 1 - bh_l : bh_l;
  const int p_lin = (int)(lid - bh_l * (uint32_t)np);
  // (without an order, the last query blocks first: a causal mask's lists grow along the
  // sequence, and the longest should not be the last to start: 456 -> 375 us for 32 heads of
  // 8192 in f16, D = 64.  Up to 1024 work-groups, which mostly start at once, are also dealt
  // to the CUs long with short: 69.5 -> 64.5 us for the lattice-8 mask below; beyond that it
  // costs 3% of L2 reuse.  An order that the caller gives, as a split plan's, is taken as it
  // is.)
  const int p = a.qblock_order ? p_lin : np - 1 - (gridDim.x <= 1024 ? snake(p_lin, np) : p_lin);
  const int qb = a.qblock_order ? ((cint*)a.qblock_order)[p / H] : p / H;
  const int wb = (p % H) * RG + w;  // this wave's row group in the query block

  const int A = a.A, spt_log2 = a.spt_log2, spt_mask = (1 << spt_log2) - 1;
  const int ncg = A >= 32 ? (A >> 5) : 1;   // 32-column groups per tile
  const int wpr = (A + 31) >> 5;            // bitmap words per row
  const int64_t row0 = (int64_t)qb * a.pitch;
  const int n_ent = ((cint*)a.kv_num)[qb];
  const int n_seg = n_ent << spt_log2;
  const int n_all = (n_seg + 3) >> 2;                // 64-column steps of the list
  const int n_steps = (n_all + KG - 1) / KG;         // of every key group

  // index-space position -> original position
  const bool closed = a.residue_s != 0;
  const int32_t rmask = (1 << a.residue_qlog2) - 1;
  auto orig_closed = [&](int p) __attribute__((always_inline)) -> int {
    return (p & rmask) * a.residue_s + (p >> a.residue_qlog2);
  };
  const bool has_pq = closed || a.pred.perm_q;
  const bool gather_kv = a.gather_kv && closed;
  const int r_idx = qb * (32 * RG * H) + wb * 32 + m;  // index-space query row of this lane
  int q_orig = r_idx;
  if (has_pq) q_orig = closed ? orig_closed(r_idx) : a.pred.perm_q[r_idx];
  const int r_load = (a.gather_q && has_pq) ? q_orig : r_idx;

  const bool use_bits = a.kv_bits != nullptr;
  if (!use_bits) {
#pragma unroll
    for (int i = 0; i < PA_MAX_TERMS; ++i)  // constant indices into the argument block
      if (tid == i) terms_s[i] = a.pred.terms[i];
  }

  // ---- Q fragments (B operand of S^T = K Q^T) --------------------------------
  Frag qf[NQF];
  {
    const char* qrow = a.q + (bh * a.q_sb + (int64_t)r_load * a.q_sn) * ESZ;
#pragma unroll
    for (int kc = 0; kc < NQF; ++kc)
      qf[kc] = __builtin_bit_cast(Frag, *reinterpret_cast<const uint4*>(qrow + (16 * kc + 8 * G) * ESZ));
  }

  // ---- K / V staging -------------------------------------------------------------
  const char* kbase = a.k + bh * a.k_sb * ESZ;
  const char* vbase = a.v + bh * a.v_sb * ESZ;
  const int64_t krow_b = a.k_sn * ESZ, vrow_b = a.v_sn * ESZ;
  const int rstride = gather_kv ? a.residue_s : 1;
  uint32_t koff[R::NI], voff[R::NI];
  dma_offsets<D>(koff, rstride * krow_b, lane);
  dma_offsets<D>(voff, rstride * vrow_b, lane);
  const uint32_t kstep = (uint32_t)(R::RPI * rstride * krow_b), vstep = (uint32_t)(R::RPI * rstride * vrow_b);
#pragma unroll
  for (int i = 1; i < R::NI; ++i) {
    koff[i] += i * kstep;
    voff[i] += i * vstep;
  }

  // The list, 16 of this key group's steps at a time: lane 4 u + t holds segment t (16
  // columns) of step 16 c + u, its first column, its row in memory and its bitmap offset; the
  // segments' codes for this wave are two 64-bit words (bit 4 u + t: some pair live / every
  // pair live).  A step then costs a few scalar operations.  The next 16 steps' entries are
  // loaded (raw) halfway through these.
  // (row offsets inside a head are 32-bit, checked on the host: they go into the lanes'
  // addresses, and the 64-bit bases stay as they are: window 1024, 64x64, bf16 D = 128,
  // 16 x 8192, 179.5 -> 172.5 us)
  int32_t c_col = 0, c_boff = -1;   // current 16 steps
  uint32_t c_koff = 0u, c_voff = 0u;
  uint64_t c_live = 0ull, c_full = 0ull;
  int32_t r_idx_ = 0, r_boff = -1;  // raw entries of the next 16
  uint32_t r_code = 0u;
  auto seg_of = [&](int c) __attribute__((always_inline)) -> int {
    return 4 * ((16 * c + (lane >> 2)) * KG + kg) + (lane & 3);
  };
  auto load_raw = [&](int c) __attribute__((always_inline)) {
    const int e = seg_of(c) >> spt_log2;
    r_idx_ = 0;
    r_code = 0u;
    r_boff = -1;
    if (e < n_ent) {
      r_idx_ = a.kv_idx[row0 + e];
      r_code = a.kv_wave_bits ? a.kv_wave_bits[row0 + e] : (a.kv_partial[row0 + e] ? 0x55555555u : 0xffffffffu);
      if (use_bits) r_boff = a.kv_bits_off[row0 + e];
    }
  };
  auto take_raw = [&](int c) __attribute__((always_inline)) {
    const int seg = seg_of(c);
    const int within = seg & spt_mask;
    const bool in = seg < n_seg;
    const uint32_t code = in ? r_code >> (2 * (wb * ncg + (A >= 32 ? within >> 1 : 0))) : 0u;
    c_live = __ballot((code & 1u) != 0u);
    c_full = __ballot((code & 2u) != 0u);
    c_col = r_idx_ * A + within * 16;
    // (a segment past the list holds its step's first segment again, with code 0: rows this
    // query block meets anyway)
    const int first = __shfl(c_col, lane & ~3);
    if (!in) c_col = first;
    const int row = gather_kv ? orig_closed(c_col) : c_col;
    c_koff = (uint32_t)row * (uint32_t)krow_b;
    c_voff = (uint32_t)row * (uint32_t)vrow_b;
    c_boff = r_boff >= 0 ? r_boff + ((within * 16) >> 5) : -1;
  };

  // One step of this wave: its place among the 16, bit t of live / full: segment t has a live
  // pair / is all live.
  struct Step {
    int u4;
    uint32_t live, full;
  };
  auto dma = [&](int u4, int S) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < SPW; ++u) {
      const int at = SPW * w + u;
      const uint32_t ko = (uint32_t)__builtin_amdgcn_readlane((int)c_koff, u4 + at);
      const uint32_t vo = (uint32_t)__builtin_amdgcn_readlane((int)c_voff, u4 + at);
      const uint32_t m0 = ring0 + (uint32_t)(S * STAGE + at * 16 * R::ROW);
#pragma unroll
      for (int i = 0; i < R::NI; ++i) {
        dma_x4(m0 + i * 1024, kbase, koff[i] + ko);
        dma_x4(m0 + TB + i * 1024, vbase, voff[i] + vo);
      }
    }
  };
  // mask words of a step's two 32-column blocks for this lane's row: ones for a full segment,
  // zeros for a dead one, the bitmap's bits for a partial one
  auto words = [&](const Step& s, uint32_t* wd) __attribute__((always_inline)) {
    if (!use_bits || s.full == 15u) return;
    const uint32_t* rowp = a.kv_bits + (int64_t)(wb * 32 + m) * wpr;
#pragma unroll
    for (int lb = 0; lb < 2; ++lb) {
      const uint32_t lv = (s.live >> (2 * lb)) & 3u, fl = (s.full >> (2 * lb)) & 3u;
      if (lv != 0u && fl != 3u) {
        const int b0 = __builtin_amdgcn_readlane(c_boff, s.u4 + 2 * lb);
        if (A >= 32) {
          wd[lb] = b0 >= 0 ? rowp[b0] : 0u;
        } else {
          // one bitmap word of 16 columns per segment
          const int b1 = __builtin_amdgcn_readlane(c_boff, s.u4 + 2 * lb + 1);
          const uint32_t lo = (fl & 1u) ? 0xffffu : ((lv & 1u) && b0 >= 0) ? rowp[b0] & 0xffffu : 0u;
          const uint32_t hi = (fl & 2u) ? 0xffffu : ((lv & 2u) && b1 >= 0) ? rowp[b1] & 0xffffu : 0u;
          wd[lb] = lo | (hi << 16);
        }
      }
    }
  };
  // the same by evaluating the predicate (index without bitmaps); col: the block's columns,
  // column m's on lane m
  auto eval_word = [&](uint32_t lv, uint32_t fl, int col) __attribute__((always_inline)) -> uint32_t {
    const int ko_m = closed ? orig_closed(col) : a.pred.perm_kv ? a.pred.perm_kv[col] : col;
    uint32_t word = 0u;
#pragma unroll 1
    for (int i = 0; i < 16; ++i) {
      const int b = 8 * (i >> 2) + 4 * G + (i & 3);
      const int ko = __shfl(ko_m, b);
      if (((fl >> (b >> 4)) & 1u) ||
          (((lv >> (b >> 4)) & 1u) && pred_live_rolled(terms_s, a.pred.n_include, a.pred.n_exclude, q_orig, ko,
                                                       a.pred.dense_bits, a.pred.dense_words)))
        word |= 1u << b;
    }
    return word;
  };

  const TileReads<D> rd = tile_reads<D>((lds_cptr)ring, lane);

  f32x16 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) acc[i] = f32x16{0};
  float m_run = kSentinel, l_part = 0.f;

  // A step in stage SC, with `rest` segments of the list left from its first on.  FULL: every
  // pair of it live for this wave (no masking, no branch).
  auto compute = [&](auto SC, auto FULL, const Step& s, const uint32_t* wd, int rest, int col0, int col1)
                     __attribute__((always_inline)) {
    constexpr int SO = decltype(SC)::value * STAGE;
    constexpr bool ALL = decltype(FULL)::value;
    f32x16 sc[2];
    float mx = -INFINITY;
    Frag vf[2 * NDB];  // the first block's V fragments, read behind the scores
    if constexpr (ALL) {
      // both blocks' scores, K reads running ahead of their MFMAs
      u32x4 ka[2][NQF];
#pragma unroll
      for (int lb = 0; lb < 2; ++lb)
#pragma unroll
        for (int kc = 0; kc < NQF; ++kc) ka[lb][kc] = *(lds_u4*)(rd.row(kc) + SO + 32 * lb * R::ROW);
#pragma unroll
      for (int lb = 0; lb < 2; ++lb) {
        sc[lb] = Mma<T>::mma(__builtin_bit_cast(Frag, ka[lb][0]), qf[0], f32x16{0});
#pragma unroll
        for (int kc = 1; kc < NQF; ++kc) sc[lb] = Mma<T>::mma(__builtin_bit_cast(Frag, ka[lb][kc]), qf[kc], sc[lb]);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int db = 0; db < NDB; ++db) vf[NDB * c + db] = tr_frag<T, D>(rd, db, SO + TB + 16 * c * R::ROW);
      constexpr int AHEAD = 6;
      __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
      for (int q_ = 0; q_ < 2 * NQF; ++q_) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 4 * NDB, 0);
#pragma unroll
      for (int lb = 0; lb < 2; ++lb)
#pragma unroll
        for (int i = 0; i < 16; i += 2) mx = nan_max(mx, nan_max(sc[lb][i], sc[lb][i + 1]));
    } else {
#pragma unroll
      for (int lb = 0; lb < 2; ++lb) {
        const uint32_t lv = (s.live >> (2 * lb)) & 3u, fl = (s.full >> (2 * lb)) & 3u;
        if (!ALL && lv == 0u) continue;
        f32x16 x = f32x16{0};
#pragma unroll
        for (int kc = 0; kc < NQF; ++kc)
          x = Mma<T>::mma(__builtin_bit_cast(Frag, *(lds_u4*)(rd.row(kc) + SO + 32 * lb * R::ROW)), qf[kc], x);
        if (!ALL && fl != 3u) {
          const uint32_t word = (use_bits ? wd[lb] : eval_word(lv, fl, lb ? col1 : col0)) >> (4 * G);
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float xv = x[i];  // (a scalar copy: bit-casting the vector element reads element 0)
            const int32_t keep = __builtin_amdgcn_sbfe((int32_t)word, 8 * (i >> 2) + (i & 3), 1);
            x[i] = __builtin_bit_cast(float, (__builtin_bit_cast(int32_t, xv) & keep) |
                                                 (int32_t)(0xff800000u & ~(uint32_t)keep));
          }
        }
#pragma unroll
        for (int i = 0; i < 16; i += 2) mx = nan_max(mx, nan_max(x[i], x[i + 1]));
        sc[lb] = x;
      }
    }
    const float m_new = nan_max(m_run, row_nan_max(mx) * a.c);
    if (__ballot(m_new > m_run + kLazy) != 0ull) {
      const float alpha = exp2f(m_run - m_new);
      m_run = m_new;
      l_part *= alpha;
#pragma unroll
      for (int i = 0; i < NDB; ++i) acc[i] *= alpha;
    }
    const float neg_m = -m_run;
#pragma unroll
    for (int lb = 0; lb < 2; ++lb) {
      if (!ALL && ((s.live >> (2 * lb)) & 3u) == 0u) continue;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        // (a segment past the list has no pairs, and 0 times its V rows, which are another
        // segment's, is no 0 where they hold an infinity)
        if (!ALL && c == 1 && 2 * lb + 1 >= rest) continue;
        f32x8 pv;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[lb][8 * c + e], a.c, neg_m));
          l_part += pv[e];
        }
        const Frag pf = Mma<T>::cvt(pv);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
          acc[db] = Mma<T>::mma(ALL && lb == 0 ? vf[NDB * c + db]
                                               : tr_frag<T, D>(rd, db, SO + TB + (32 * lb + 16 * c) * R::ROW),
                                pf, acc[db]);
      }
    }
    if constexpr (ALL) {
      // the second block's V reads and exponentials beside the first block's products
      __builtin_amdgcn_sched_group_barrier(0x002, 56, 1);
#pragma unroll
      for (int q_ = 0; q_ < 4 * NDB; ++q_) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
        __builtin_amdgcn_sched_group_barrier(0x002, 112 / (3 * NDB), 1);
      }
    }
  };

  // ---- the list ------------------------------------------------------------------
  Step s_n{0, 0u, 0u};
  uint32_t w_n[2] = {~0u, ~0u};
  auto prefetch = [&](int j, int S) __attribute__((always_inline)) {
    if ((j & 15) == 0) take_raw(j >> 4);
    if ((j & 15) == 8) load_raw((j >> 4) + 1);
    s_n.u4 = 4 * (j & 15);
    s_n.live = (uint32_t)(c_live >> s_n.u4) & 15u;
    s_n.full = (uint32_t)(c_full >> s_n.u4) & 15u;
    // (a key group's step past the list moves and computes nothing)
    if (j * KG + kg < n_all) {
      words(s_n, w_n);
      dma(s_n.u4, S);
    }
  };
  auto step = [&](auto SC, int j) __attribute__((always_inline)) {
    constexpr int S = decltype(SC)::value;
    dma_wait_all();
    // (uses that make the compiler's own waits for its loads fall here, before the next
    // step's DMA is issued)
    asm volatile("" ::"v"(w_n[0]), "v"(w_n[1]), "v"(r_idx_), "v"(r_code), "v"(r_boff));
#pragma unroll
    for (int kc = 0; kc < NQF; ++kc) asm volatile("" ::"v"(qf[kc]));
    __syncthreads();  // stage S is in; every wave is past stage S ^ 1
    const Step s = s_n;
    const uint32_t wd[2] = {w_n[0], w_n[1]};
    int col0 = 0, col1 = 0;
    if (!use_bits && s.full != s.live) {
      // the original columns a partial block's predicate is evaluated at
      col0 = __shfl(c_col, s.u4 + (m >> 4)) + (m & 15);
      col1 = __shfl(c_col, s.u4 + 2 + (m >> 4)) + (m & 15);
    }
    if (j + 1 < n_steps) prefetch(j + 1, S ^ 1);
    const int rest = n_seg - 4 * (j * KG + kg);
    if (s.full == 15u)
      compute(SC, std::true_type{}, s, wd, rest, col0, col1);
    else if (s.live != 0u)
      compute(SC, std::false_type{}, s, wd, rest, col0, col1);
  };
  if (n_steps > 0) {
    load_raw(0);
    prefetch(0, 0);
  }
  int j = 0;
  for (; j + 1 < n_steps; j += 2) {
    step(std::integral_constant<int, 0>{}, j);
    step(std::integral_constant<int, 1>{}, j + 1);
  }
  if (j < n_steps) step(std::integral_constant<int, 0>{}, j);

  // ---- merge of the key groups ------------------------------------------------------
  float l_tot = row_sum(l_part);
  if constexpr (KG > 1) {
    __syncthreads();  // every wave is past its ring
    lds_char_t* ex = (lds_char_t*)smem;
    constexpr int WB = NDB * 4 * 1024 + 512;  // a wave's state: O^T, then max and sum per lane
    typedef __attribute__((address_space(3))) float lds_fw;
    if (kg > 0) {
      lds_char_t* at = ex + ((kg - 1) * RG + w) * WB;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const f32x4 x = {acc[db][4 * i4], acc[db][4 * i4 + 1], acc[db][4 * i4 + 2], acc[db][4 * i4 + 3]};
          *(lds_f4w*)(at + (4 * db + i4) * 1024 + 16 * lane) = x;
        }
      *(lds_fw*)(at + NDB * 4096 + 4 * lane) = m_run;
      *(lds_fw*)(at + NDB * 4096 + 256 + 4 * lane) = l_tot;
    }
    __syncthreads();
    if (kg > 0) return;  // (no barrier follows)
#pragma unroll
    for (int g = 1; g < KG; ++g) {
      lds_char_t* at = ex + ((g - 1) * RG + w) * WB;
      const float mg = *(lds_fw*)(at + NDB * 4096 + 4 * lane), lg = *(lds_fw*)(at + NDB * 4096 + 256 + 4 * lane);
      const float mn = fmaxf(m_run, mg);
      const float f0 = exp2f(m_run - mn), f1 = exp2f(mg - mn);
      m_run = mn;
      l_tot = l_tot * f0 + lg * f1;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const f32x4 x = *(lds_f4*)(at + (4 * db + i4) * 1024 + 16 * lane);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[db][4 * i4 + e] = acc[db][4 * i4 + e] * f0 + x[e] * f1;
        }
    }
  }

  // ---- epilogue (as attn_fwd_kernel) -------------------------------------------------
  const bool has = l_tot > 0.f;
  float lse_v = has ? (m_run + log2f(l_tot)) * kLn2 : -INFINITY;
  float a_own = has ? 1.f / l_tot : 0.f;
  float a_prev = 0.f;
  const int srow = (a.scatter_o && has_pq) ? q_orig : r_idx;
  if (a.prev_o) {
    const float lp = a.prev_lse[bh * a.lse_sb + srow];
    const float M = fmaxf(lse_v, lp);
    if (M == -INFINITY) {
      a_own = 0.f;
      lse_v = -INFINITY;
    } else {
      const float w1 = has ? expf(lse_v - M) : 0.f;
      const float w2 = lp == -INFINITY ? 0.f : expf(lp - M);
      const float den = w1 + w2;
      a_own = has ? (w1 / den) / l_tot : 0.f;
      a_prev = w2 / den;
      lse_v = M + logf(den);
    }
  }
  char* orow = a.o + (bh * a.o_sb + (int64_t)srow * a.o_sn) * ESZ;
  const int psz = a.prev_dtype == PA_F32 ? 4 : 2;
  const char* prow = a.prev_o ? a.prev_o + (bh * a.prev_sb + (int64_t)srow * a.prev_sn) * psz : nullptr;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int d0 = 32 * db + 8 * i4 + 4 * G;
      f32x4 x = {acc[db][4 * i4], acc[db][4 * i4 + 1], acc[db][4 * i4 + 2], acc[db][4 * i4 + 3]};
      x *= a_own;
      if (prow && a_prev != 0.f) x += a_prev * load4_any(prow + d0 * psz, a.prev_dtype);
      Mma<T>::store4(orow + d0 * ESZ, x);
    }
  }
  if (a.lse && G == 0) a.lse[bh * a.lse_sb + srow] = lse_v;
}

template <typename T, int D, int RG, int KG, int H>
int launch_tile_t(const AttnK& a, hipStream_t s) {
  constexpr int smem = tile_smem_bytes<D, KG>();
  static unsigned long long configured = 0ull;  // the dynamic LDS limit is raised once per device
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev >= 64 || !((configured >> dev) & 1ull)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_tile_kernel<T, D, RG, KG, H>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(attn_tile_kernel)");
    if (dev < 64) configured |= 1ull << dev;
  }
  hipLaunchKernelGGL((attn_tile_kernel<T, D, RG, KG, H>), dim3((unsigned)(H * a.total_wg)), dim3(64 * RG * KG), smem,
                     s, a);
  PA_LAUNCH_CHECK("attn_tile_kernel");
  return PA_OK;
}

// How many key groups a list is given and into how many pieces of 64 rows a block of 128 is
// cut.  A second group halves what a launch of up to one work-group per CU waits for; beyond
// that it pays where a few lists are much longer than the rest (uneven: a covering mask in
// order), and costs where all are alike.  Measured (us; f16, lists of tiles with bitmaps / by
// the predicate where two figures stand; w: a window), by one key group of 128 rows / two /
// pieces of 64 rows by two / by four:
//   D = 64, work-groups of 128 rows:
//     64 (causal, 2 x 4096)   - / 50.5 / 41.8 / 33.2      128 (causal, 1 x 16384) - / 183 / 153 / 111
//     128 (w 200, 4 x 4096) - / 10.7 / 9.3 / 9.3     128 (w 1024) - / 18.4 / 15.2 / 13.5
//     256 (causal, 8 x 4096) 73.2 / 51.7 / 43.5 / 53.6    256 (causal, 4 x 8192) - / 91.6 / 76.2 / 96.7
//     256 (32 x 1024) - / 21.1 / 22.1 / 30.2      256 (w 4096, 4 x 8192) - / 49.5 / 50.5 / 57.7
//     320 (w 200) 14.3 55.0 / 18.0 58.3 / 16.7 58.3 / 22.1 66.5, (w 2048) 46.4 68.4 / 41.7 56.3
//     384 (causal, 12 x 4096) 93.8 / 63.9 / 60.8 / 74.0   512 (causal, 16 x 4096) - / 64.4 / 72.2 / 94.3
//     512 (w 64) 11.0 27.3 / 15.1 36.3, (w 300) 16.5 51.7 / 20.8 70.8, (w 1536) 39.2 59.5 / 43.6 63.4,
//     (lattice 8 in its basis) 37.1 48.9 / 46.7 61.5, (band and lattice 16 in the lattice's) 68.8 / 74.4
//   so four key groups and pieces up to 128 work-groups, which then fit one to a CU; two groups
//   up to 256, and on long lists a quarter more; up to 512 two groups on uneven lists, in
//   pieces up to 384 (a CU takes a long and a short one);
//   D = 128: 64 (2 x 4096) - / 70.8 / 58.8, 128 (4 x 4096) - / 71.3 / 60.1, 128 (w 200)
//     - / 39.9 / 32.4, 160 (5 x 4096) - / 72.2 / 71.0, 160 (10 x 2048) - / 42.6 / 47.0, 256
//     107 / 74.7 / 89.0 (one work-group of two groups per CU by its LDS).
// Blocks of 64 rows, one key group / two / four:
//   D = 64:  128 (8 x 1024) - / 18.4 / 16.9, 256 (8 x 2048) - / 26.6 / 22.6, 256 (4 x 4096) - /
//     42.6 / 33.9, 512 (8 x 4096) 71.8 / 43.4 / 53.6, 768 (w 128) 10.4 22.1 / 14.8 36.2, 1024 (w 300)
//     15.7 36.9 / 19.0 51.2, 2048 (w 1024) 85 / 105 / -;
//   D = 128: 512 (causal, 8 x 4096) 87.4 / 78.2, (causal, 16 x 2048) 60.8 / 38.6, (w 128) 13.1 24.4 /
//     19.1 38.7, (w 1024) 37.2 48.1 / 40.2 59.6, (band and lattice 16 in the lattice's basis) 60.2 355
//     / 83.4 460; 2048 (w 1024) 172 / 227.
template <typename T, int D>
int launch_tile_d(const AttnK& a, hipStream_t s) {
  const int64_t wgs = a.total_wg, longest = a.pitch * a.A;
  // (in a residue basis a covering mask's lists are about equally long)
  const bool uneven = longest >= 2048 && 4 * longest >= 3 * (int64_t)a.N && !a.residue_s && !a.pred.perm_q;
  if constexpr (D == 64) {
    if (a.BQ == 64) {
      if (wgs <= 256) return launch_tile_t<T, D, 2, 4, 1>(a, s);
      if (wgs <= 512 || (wgs <= 1024 && uneven)) return launch_tile_t<T, D, 2, 2, 1>(a, s);
      return launch_tile_t<T, D, 2, 1, 1>(a, s);
    }
    if (wgs <= 128) return launch_tile_t<T, D, 2, 4, 2>(a, s);
    if (wgs <= 384 && uneven) return launch_tile_t<T, D, 2, 2, 2>(a, s);
    if (wgs <= 256 || (wgs <= 320 && longest >= 1536) || (wgs <= 512 && uneven))
      return launch_tile_t<T, D, 4, 2, 1>(a, s);
  } else {
    if (a.BQ == 64) {
      if (wgs <= 256 || (wgs <= 512 && uneven)) return launch_tile_t<T, D, 2, 2, 1>(a, s);
      return launch_tile_t<T, D, 2, 1, 1>(a, s);
    }
    if (wgs <= 128) return launch_tile_t<T, D, 2, 2, 2>(a, s);
    if (wgs <= 256) return launch_tile_t<T, D, 4, 2, 1>(a, s);
  }
  return launch_tile_t<T, D, 4, 1, 1>(a, s);
}

}  // namespace

// 2-byte types, rows gathered in index space or through the closed-form basis, a head's K
// and V within 4 GiB
bool attn_tile_takes(const AttnK& a, int dtype) {
  const int64_t row = 2 * (a.k_sn > a.v_sn ? a.k_sn : a.v_sn);
  return (dtype == PA_F16 || dtype == PA_BF16) && a.gather_mult <= 1 && !(a.gather_kv && a.residue_s == 0) &&
         a.k_sn >= 0 && a.v_sn >= 0 && a.N * row < (1ll << 32);
}

int launch_attn_narrow(const AttnK& a, int dtype, int D, hipStream_t s);

int launch_attn_tile(const AttnK& a, int dtype, int D, hipStream_t s) {
  if (a.BQ < 64) return launch_attn_narrow(a, dtype, D, s);
  if (dtype == PA_BF16) return D == 64 ? launch_tile_d<__bf16, 64>(a, s) : launch_tile_d<__bf16, 128>(a, s);
  return D == 64 ? launch_tile_d<_Float16, 64>(a, s) : launch_tile_d<_Float16, 128>(a, s);
}

}  // namespace pa
