// Block-sparse attention forward for f16 / bf16 on narrow query blocks: BQ = 16 or 32, any A,
// D = 64 or 128, on block lists as they are (bitmaps optional).
//
// Same contract and numerics as attn_fwd_kernel (the replacement of the Triton kernel
// _attn_fwd, gpu/triton_attn.py:62-182), which gives a 16-row block a wave of 32-row MFMAs
// (half of them padding) and stages K and V through registers.  Here a wave owns 16 query
// rows (half a block for BQ = 32) and walks the list 32 columns at a time on 16x16x32 MFMAs,
// with nothing shared between the waves of a work-group and no barrier:
//
//  * S^T = K Q^T of two 16-column segments: lane (q = l % 16, g = l / 16) holds columns
//    4 g + 0..3 of each for its row.  K rows are loaded straight into the A operand
//    registers, a step ahead;
//  * the two segments' P values of a lane are, in that order, 8 consecutive contraction
//    indices of P^T as the B operand of O^T += V^T P^T; V^T comes from transposed LDS reads
//    of V rows that the LDS DMA moved into the wave's own two-stage ring.  The rows are
//    unpadded; 16-byte unit u of row r sits at u ^ 2 (r % 8) (D = 128) or u ^ 2 ((r / 2) % 4)
//    (D = 64, two rows to a bank window), so the 8 rows x 2 units that half a wave reads are
//    16 different units of the 256-byte window;
//  * the list is held 32 steps at a time, a segment per lane.
//
// What bounds it: the latency of a wave's step, whose loads are issued one step ahead and all
// waited for.  Lattice-8 in its basis, 8 heads x 8192, 16x16 tiles, D = 64, is one round of
// work-groups; a step of its longest lists takes some 2900 clocks, of which the 8 MFMAs are
// 128, and waves wait on a counter 56% of theirs (2.5 waves per SIMD on average, VALU 23%,
// matrix cores 7% of the SIMDs' clocks).  Every wave reads its own K and V rows: 8 KB per 16 x
// 32 pairs at D = 64 and 16 KB at D = 128, from the L1 and L2.  118 registers at D = 64 (four
// waves per SIMD), 182 at D = 128 (two).  Against
// attn_fwd_kernel, f16: lattice-8 in its basis, 8 heads x 8192, 16x16 tiles, D = 64 211 ->
// 45 us (191 live TFLOP/s); window 256, 8 x 8192: 16x16 140 -> 29 us, D = 128 286 -> 54;
// 32x32 89 -> 31, D = 128 171 -> 58; causal, 8 x 2048: 16x16 128 -> 42, D = 128 241 -> 79;
// 32x32, D = 128 157 -> 81.
#include <type_traits>

#include "lds_rows.hpp"

namespace pa {
namespace {

template <typename T>
__device__ __forceinline__ f32x4 mma16x32(typename Mma<T>::frag a, typename Mma<T>::frag b, f32x4 c) {
  if constexpr (__is_same(T, __bf16))
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// max / sum over the four lanes l % 16 + 16 g that hold one query row
__device__ __forceinline__ float quad_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
  return row_nan_max(nan_max(__builtin_bit_cast(float, (int)r[0]), __builtin_bit_cast(float, (int)r[1])));
}
__device__ __forceinline__ float quad_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
  return row_sum(__builtin_bit_cast(float, (int)r[0]) + __builtin_bit_cast(float, (int)r[1]));
}

constexpr int kNarrowWaves = 4;

template <typename T, int D>
__global__ __launch_bounds__(64 * kNarrowWaves) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2)))
void attn_narrow_kernel(const AttnK a, int units, int groups) {
  using Frag = typename Mma<T>::frag;
  using R = Rows<D>;
  constexpr int ESZ = 2, NK = D / 32, NDB = D / 16;
  constexpr int SEG = 16 * R::ROW, STAGE = 2 * SEG;  // V rows of a segment, of a step

  __shared__ __attribute__((aligned(256))) char ring_s[kNarrowWaves * 2 * STAGE];
  __shared__ pa_term terms_s[PA_MAX_TERMS];

  const int tid = threadIdx.x, lane = tid & 63, q16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool use_bits = a.kv_bits != nullptr;
  if (!use_bits) {
#pragma unroll
    for (int i = 0; i < PA_MAX_TERMS; ++i)  // constant indices into the argument block
      if (tid == i) terms_s[i] = a.pred.terms[i];
    __syncthreads();  // (the only one: before any wave leaves)
  }

  // work-group = four consecutive 16-row units of a head; without an issue order the last
  // first (a causal mask's longest), launches that mostly start at once long with short
  const uint32_t lid = xcd_remap32(blockIdx.x, gridDim.x);
  const uint32_t bh_l = lid / (uint32_t)groups;
  const int64_t bh = a.heads_desc ? a.BH - 1 - bh_l : bh_l;
  int gi = (int)(lid - bh_l * (uint32_t)groups);
  if (!a.qblock_order) gi = groups - 1 - (gridDim.x <= 1024 ? snake(gi, groups) : gi);
  const int unit = gi * kNarrowWaves + w;
  if (unit >= units) return;
  const int upb = a.BQ >> 4;  // units per query block
  const int ub = unit / upb;
  const int qb = a.qblock_order ? ((cint*)a.qblock_order)[ub] : ub;
  const int half = unit - ub * upb;

  const int A = a.A, spt_log2 = a.spt_log2, spt_mask = (1 << spt_log2) - 1;
  const int wpr = (A + 31) >> 5;
  const int64_t row0 = (int64_t)qb * a.pitch;
  const int n_ent = ((cint*)a.kv_num)[qb];
  const int n_seg = n_ent << spt_log2;
  const int n_steps = (n_seg + 1) >> 1;

  const bool closed = a.residue_s != 0;
  const int32_t rmask = (1 << a.residue_qlog2) - 1;
  auto orig_closed = [&](int p) __attribute__((always_inline)) -> int {
    return (p & rmask) * a.residue_s + (p >> a.residue_qlog2);
  };
  const bool has_pq = closed || a.pred.perm_q;
  const bool gather_kv = a.gather_kv && closed;
  const int row_b = half * 16 + q16;            // the lane's row in its block
  const int r_idx = qb * a.BQ + row_b;          // index-space query row of this lane
  int q_orig = r_idx;
  if (has_pq) q_orig = closed ? orig_closed(r_idx) : a.pred.perm_q[r_idx];
  const int r_load = (a.gather_q && has_pq) ? q_orig : r_idx;

  Frag qf[NK];
  {
    const char* qrow = a.q + (bh * a.q_sb + (int64_t)r_load * a.q_sn) * ESZ + 16 * g;
#pragma unroll
    for (int kc = 0; kc < NK; ++kc) qf[kc] = __builtin_bit_cast(Frag, *reinterpret_cast<const uint4*>(qrow + 64 * kc));
  }

  const char* kbase = a.k + bh * a.k_sb * ESZ;
  const char* vbase = a.v + bh * a.v_sb * ESZ;
  const int64_t krow_b = a.k_sn * ESZ, vrow_b = a.v_sn * ESZ;
  const int rstride = gather_kv ? a.residue_s : 1;
  const uint32_t koff = (uint32_t)(q16 * rstride * krow_b) + 16u * (uint32_t)g;
  // V: instruction i moves rows RPI i + l / UPR of a segment
  uint32_t voff[R::NI];
#pragma unroll
  for (int i = 0; i < R::NI; ++i) {
    const int r = R::RPI * i + lane / R::UPR;
    const int sw = D == 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3);
    voff[i] = (uint32_t)(r * rstride * vrow_b) + 16u * (uint32_t)((lane % R::UPR) ^ sw);
  }
  const uint32_t ring0 = (uint32_t)(uintptr_t)(lds_char_t*)ring_s + (uint32_t)(w * 2 * STAGE);
  // transposed reads of 16 columns (block db) of rows 4 g + q16 / 4 of a segment
  lds_cptr vptr[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    const int r = 4 * g + (q16 >> 2);
    const int sw = D == 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3);
    vptr[db] = (lds_cptr)ring_s + w * 2 * STAGE + r * R::ROW + 16 * ((2 * db + ((q16 & 3) >> 1)) ^ sw) + 8 * (q16 & 1);
    asm volatile("" : "+v"(vptr[db]));
  }

  // 32 steps of the list: lane l holds segment 64 c + l (its first column, its bitmap
  // offset); bit l of live / full: it has a live pair / is all live.  The next 32 steps'
  // entries are loaded (raw) halfway through these.
  // (row offsets inside a head are 32-bit, checked on the host: they go into the lanes'
  // addresses, and the 64-bit bases stay as they are; 64-bit products and sums per step on
  // the scalar unit took 48.5 us of causal 16x16, 8 x 2048, against 41.9)
  int32_t c_col = 0, c_boff = -1, r_tile = 0, r_boff = -1;
  uint32_t c_koff = 0u, c_voff = 0u;
  uint32_t r_code = 0u;
  uint64_t c_live = 0ull, c_full = 0ull;
  auto load_raw = [&](int c) __attribute__((always_inline)) {
    const int e = (64 * c + lane) >> spt_log2;
    r_tile = 0;
    r_code = 0u;
    r_boff = -1;
    if (e < n_ent) {
      r_tile = a.kv_idx[row0 + e];
      r_code = a.kv_wave_bits ? a.kv_wave_bits[row0 + e] : (a.kv_partial[row0 + e] ? 0x55555555u : 0xffffffffu);
      if (use_bits) r_boff = a.kv_bits_off[row0 + e];
    }
  };
  auto take_raw = [&](int c) __attribute__((always_inline)) {
    const int seg = 64 * c + lane;
    const int within = seg & spt_mask;
    const bool in = seg < n_seg;
    const uint32_t code = in ? r_code >> (2 * (A >= 32 ? within >> 1 : 0)) : 0u;
    c_live = __ballot((code & 1u) != 0u);
    c_full = __ballot((code & 2u) != 0u);
    c_col = r_tile * A + within * 16;
    // (a segment past the list holds its step's other one again, with code 0)
    const int first = __shfl(c_col, lane & ~1);
    if (!in) c_col = first;
    const int row = gather_kv ? orig_closed(c_col) : c_col;
    c_koff = (uint32_t)row * (uint32_t)krow_b;
    c_voff = (uint32_t)row * (uint32_t)vrow_b;
    c_boff = r_boff >= 0 ? r_boff + ((within * 16) >> 5) : -1;
  };

  struct Step {
    int col[2];
    uint32_t live, full;  // 2 bits each
  };
  struct Data {  // what a step needs in registers
    u32x4 k[2][NK];
    uint32_t word[2];
  };
  auto prefetch = [&](int j, int S, Step& s, Data& d) __attribute__((always_inline)) {
    if ((j & 31) == 0) take_raw(j >> 5);
    if ((j & 31) == 16) load_raw((j >> 5) + 1);
    const int l0 = 2 * (j & 31);
    s.live = (uint32_t)(c_live >> l0) & 3u;
    s.full = (uint32_t)(c_full >> l0) & 3u;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (!use_bits) s.col[t] = __builtin_amdgcn_readlane(c_col, l0 + t);
      const uint32_t ko = koff + (uint32_t)__builtin_amdgcn_readlane((int)c_koff, l0 + t);
      const uint32_t vo = (uint32_t)__builtin_amdgcn_readlane((int)c_voff, l0 + t);
#pragma unroll
      for (int kc = 0; kc < NK; ++kc) d.k[t][kc] = *reinterpret_cast<const u32x4*>(kbase + ko + 64 * kc);
      if (use_bits && s.full != 3u) {
        const int bo = __builtin_amdgcn_readlane(c_boff, l0 + t);
        d.word[t] = ((s.full >> t) & 1u)                ? ~0u
                    : (((s.live >> t) & 1u) && bo >= 0) ? a.kv_bits[(int64_t)bo + row_b * wpr] >> (A >= 32 ? 16 * t : 0)
                                                        : 0u;
      }
#pragma unroll
      for (int i = 0; i < R::NI; ++i) dma_x4(ring0 + S * STAGE + t * SEG + i * 1024, vbase, voff[i] + vo);
    }
  };
  // bits 4 g + 0..3 of a partial segment by evaluating the predicate (index without bitmaps)
  auto eval_word = [&](int col) __attribute__((always_inline)) -> uint32_t {
    const int c = col + q16;
    const int ko_m = closed ? orig_closed(c) : a.pred.perm_kv ? a.pred.perm_kv[c] : c;
    uint32_t word = 0u;
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
      const int b = 4 * g + i;
      const int ko = __shfl(ko_m, b);
      if (pred_live_rolled(terms_s, a.pred.n_include, a.pred.n_exclude, q_orig, ko, a.pred.dense_bits,
                           a.pred.dense_words))
        word |= 1u << b;
    }
    return word;
  };

  f32x4 acc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kSentinel, l_part = 0.f;

  auto compute = [&](int S, const Step& s, const Data& d) __attribute__((always_inline)) {
    if (s.live == 0u) return;
    f32x4 x[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      x[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < NK; ++kc) x[t] = mma16x32<T>(__builtin_bit_cast(Frag, d.k[t][kc]), qf[kc], x[t]);
    }
    if (s.full != 3u) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if ((s.full >> t) & 1u) continue;
        const uint32_t word = (use_bits ? d.word[t] : ((s.live >> t) & 1u) ? eval_word(s.col[t]) : 0u) >> (4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (!((word >> i) & 1u)) x[t][i] = -INFINITY;
      }
    }
    const float mx = quad_max(nan_max(nan_max(nan_max(x[0][0], x[0][1]), nan_max(x[0][2], x[0][3])),
                                      nan_max(nan_max(x[1][0], x[1][1]), nan_max(x[1][2], x[1][3]))));
    const float m_new = nan_max(m_run, mx * a.c);
    if (__ballot(m_new > m_run + kLazy) != 0ull) {
      const float alpha = exp2f(m_run - m_new);
      m_run = m_new;
      l_part *= alpha;
#pragma unroll
      for (int i = 0; i < NDB; ++i) acc[i] *= alpha;
    }
    const float neg_m = -m_run;
    f32x8 pv;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(x[e >> 2][e & 3], a.c, neg_m));
      l_part += pv[e];
    }
    const Frag pf = Mma<T>::cvt(pv);
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const s16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vptr[db] + S * STAGE));
      const s16x4 x2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vptr[db] + S * STAGE + SEG));
      const uint4 vx = {__builtin_bit_cast(uint2, x1).x, __builtin_bit_cast(uint2, x1).y,
                        __builtin_bit_cast(uint2, x2).x, __builtin_bit_cast(uint2, x2).y};
      acc[db] = mma16x32<T>(__builtin_bit_cast(Frag, vx), pf, acc[db]);
    }
  };

  Step s0{}, s1{};
  Data d0{}, d1{};
  // The step's V rows are in LDS and its K rows in registers once everything issued is done.
  // The memory clobber keeps the ring's reads on their side of the wait (no barrier does),
  // and the last step's are done before the next DMA into their stage; the uses make the
  // compiler's own wait fall here, before the next step's loads.
  auto arrive = [&](const Data& d) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int kc = 0; kc < NK; ++kc) asm volatile("" ::"v"(d.k[t][kc]));
      asm volatile("" ::"v"(d.word[t]));
    }
    asm volatile("" ::"v"(r_tile), "v"(r_code), "v"(r_boff));
  };
  // A list of an odd number of segments: its last step's second one is past it, with no
  // pairs and V rows that are the first one's again, and 0 times an infinity is no 0.
  auto clear_past = [&](int S) __attribute__((always_inline)) {
    if (n_seg & 1) {
#pragma unroll
      for (int i = 0; i < R::NI; ++i)
        *(lds_u4w*)((lds_char_t*)ring_s + w * 2 * STAGE + S * STAGE + SEG + i * 1024 + 16 * lane) = u32x4{0u, 0u, 0u, 0u};
    }
  };
  if (n_steps > 0) {
    load_raw(0);
    prefetch(0, 0, s0, d0);
  }
  int j = 0;
  for (; j + 1 < n_steps; j += 2) {
    arrive(d0);
    prefetch(j + 1, 1, s1, d1);
    compute(0, s0, d0);
    arrive(d1);
    if (j + 2 < n_steps)
      prefetch(j + 2, 0, s0, d0);
    else
      clear_past(1);
    compute(1, s1, d1);
  }
  if (j < n_steps) {
    arrive(d0);
    clear_past(0);
    compute(0, s0, d0);
  }

  // ---- epilogue (as attn_fwd_kernel) -------------------------------------------------
  const float l_tot = quad_sum(l_part);
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
    const int dd = 16 * db + 4 * g;
    f32x4 x = acc[db] * a_own;
    if (prow && a_prev != 0.f) x += a_prev * load4_any(prow + dd * psz, a.prev_dtype);
    Mma<T>::store4(orow + dd * ESZ, x);
  }
  if (a.lse && g == 0) a.lse[bh * a.lse_sb + srow] = lse_v;
}

template <typename T, int D>
int launch_narrow_t(const AttnK& a, hipStream_t s) {
  const int units = a.N / 16, groups = (units + kNarrowWaves - 1) / kNarrowWaves;
  const int64_t grid = a.BH * groups;
  PA_CHECK_ARG(grid <= 0x7fffffffll, "attn_narrow_kernel: %lld work-groups exceed the grid limit", (long long)grid);
  hipLaunchKernelGGL((attn_narrow_kernel<T, D>), dim3((unsigned)grid), dim3(64 * kNarrowWaves), 0, s, a, units, groups);
  PA_LAUNCH_CHECK("attn_narrow_kernel");
  return PA_OK;
}

}  // namespace

int launch_attn_narrow(const AttnK& a, int dtype, int D, hipStream_t s) {
  if (dtype == PA_BF16) return D == 64 ? launch_narrow_t<__bf16, 64>(a, s) : launch_narrow_t<__bf16, 128>(a, s);
  return D == 64 ? launch_narrow_t<_Float16, 64>(a, s) : launch_narrow_t<_Float16, 128>(a, s);
}

}  // namespace pa
