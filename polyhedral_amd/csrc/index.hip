// Block-index builder on the GPU: mask predicate -> per-query-block lists of live
// KV tiles.  Replaces gpu/blockindex.py:32-51 (build), which materialises the N x N
// mask on the host and tiles it with numpy any/all.
//
// Phase 1 (classify): work-groups (query block, column split) walk the KV columns in
// chunks of 256 (split j takes chunks j, j + splits, ...) and fold the predicate over
// the block's BQ rows into per-tile codes: 2 bits (some live / all live) per wave group
// of 32 query rows x min(A, 32) columns.  Most blocks of 32 rows x a wave's 64 columns are
// live or dead as a whole, which the ranges of their original positions (and, for strided
// terms, their common residues) decide, and most chunks of columns in order so too; the
// rest are evaluated pair by pair (an explicit matrix: every pair).  Wave ballots
// do the column reduction; a query block's list length is summed over its splits.
// Evaluating every pair was bound by the VALU: the classification of a prefix-LM at N =
// 16256, 128x32 tiles, took 304 us against 50, at 65536 4810 against 130, lattice-16 outside
// a band in its basis at 16384 533 against 114; what remains is the mixed blocks and, in a
// table basis, the ranges.
// Phase 2 (compact): one work-group per query block scans the tile codes and
// writes the ascending, zero-padded kv_idx / kv_partial / kv_wave_bits rows.
#include "common.hpp"

namespace pa {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 256;  // columns per pass, one per thread

__global__ void zero_totals_kernel(unsigned long long* totals, int32_t* kv_num, int32_t nq) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 3) totals[i] = 0ull;
  if (i < nq) kv_num[i] = 0;
}

// The listed tiles and the longest list, once every split has added its count.
__global__ void max_list_kernel(const int32_t* kv_num, int32_t nq, unsigned long long* totals) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int32_t v = i < nq ? kv_num[i] : 0;
  unsigned long long sum = (unsigned long long)v;
  for (int off = 32; off > 0; off >>= 1) {
    v = max(v, __shfl_down(v, off, 64));
    sum += __shfl_down(sum, off, 64);
  }
  if ((threadIdx.x & 63) == 0 && v > 0) {
    atomicAdd(&totals[0], sum);
    atomicMax(&totals[2], (unsigned long long)v);
  }
}

// What a set of pairs is under a term or the whole predicate: kMixed = not decided here.
enum Verdict { kDead, kLive, kMixed };

// A block of rows and columns in original positions: their ranges, and for a stride p
// whether each side has one residue (rq, rk).
struct Range {
  int32_t q0, q1, k0, k1;
};

// Decides a term for every pair of the block at once where its ranges allow; `same(p)` is 1
// when all rows and all columns have one residue mod p, 0 when each side has one and they
// differ, -1 otherwise.
template <typename F>
__device__ __forceinline__ Verdict term_verdict(const pa_term& t, const Range& r, F same) {
  const int64_t d0 = (int64_t)r.q0 - r.k1, d1 = (int64_t)r.q1 - r.k0;  // range of q - kv
  auto strided = [&](int32_t p) -> Verdict {                           // d % p == 0, given d >= 0
    const int s = same(p);
    return s == 1 ? kLive : s == 0 ? kDead : kMixed;
  };
  switch (t.kind) {
    case PA_FULL:
      return kLive;
    case PA_PREFIX_LM:
      if (d0 >= 0 || (r.q1 < t.p0 && r.k1 < t.p0)) return kLive;
      return (d1 < 0 && (r.q0 >= t.p0 || r.k0 >= t.p0)) ? kDead : kMixed;
    case PA_DENSE:
      return kMixed;
    default:
      break;
  }
  // the other kinds are causal
  if (d1 < 0) return kDead;
  if (t.kind == PA_DILATED) {
    const Verdict v = strided(t.p0);
    return (v == kLive && d0 < 0) ? kMixed : v;
  }
  if (d0 < 0) {
    // pairs on both sides of the diagonal: dead only where no d >= 0 of the range is live
    return kMixed;
  }
  switch (t.kind) {
    case PA_CAUSAL:
      return kLive;
    case PA_WINDOW:
      return d1 < t.p0 ? kLive : d0 >= t.p0 ? kDead : kMixed;
    case PA_LOCAL_STRIDED:
      if (d1 < t.p0) return kLive;
      {
        const Verdict v = strided(t.p1);
        return v == kLive ? kLive : d0 >= t.p0 ? v : kMixed;
      }
    case PA_TWOBAND: {
      // (the band's end wraps as term_live's 32-bit sum does)
      const int64_t b0 = t.p1, b1 = (int32_t)((uint32_t)t.p1 + (uint32_t)t.p2);
      if (d1 < t.p0 || (d0 >= b0 && d1 < b1)) return kLive;
      return (d0 >= t.p0 && (d0 >= b1 || d1 < b0)) ? kDead : kMixed;
    }
    case PA_SINKS:
      if (d1 < t.p0 || r.k1 < t.p1) return kLive;
      return (d0 >= t.p0 && r.k0 >= t.p1) ? kDead : kMixed;
    default:
      return kMixed;
  }
}

// The whole predicate: live where an include term is and no exclude term is.  The terms come
// from LDS in a rolled loop: unrolled over the argument block, the two uses below held 263
// spilled scalars (118 now) beside the pairs' evaluation.  With that and with ranges taken by
// shuffles, a build in a random permutation, where hardly a block is decided here, took 7 to
// 12% longer than evaluating every pair alone (16x16 tiles, N = 16256, window 300: 1158 us
// against 1043; now 1051).
template <typename F>
__device__ __forceinline__ Verdict pred_verdict(const pa_term* terms, int n_include, int n_exclude, const Range& r,
                                                F same) {
  Verdict inc = kDead, exc = kDead;
#pragma unroll 1
  for (int i = 0; i < n_include + n_exclude; ++i) {
    pa_term t;  // (the same in every lane)
    t.kind = __builtin_amdgcn_readfirstlane(terms[i].kind);
    t.p0 = __builtin_amdgcn_readfirstlane(terms[i].p0);
    t.p1 = __builtin_amdgcn_readfirstlane(terms[i].p1);
    t.p2 = __builtin_amdgcn_readfirstlane(terms[i].p2);
    const Verdict v = term_verdict(t, r, same);
    Verdict& to = i < n_include ? inc : exc;
    if (v == kLive || to == kLive)
      to = kLive;
    else if (v == kMixed)
      to = kMixed;
  }
  if (inc == kDead || exc == kLive) return kDead;
  return (inc == kLive && exc == kDead) ? kLive : kMixed;
}

// Minimum over a wave, in every lane (cross-lane moves of the VALU: in a table basis it is
// taken for every 64 columns, and shuffles through LDS wait for one another).
template <int CTRL>
__device__ __forceinline__ int32_t dpp_min(int32_t x) {
  return min(x, __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ int32_t wave_min(int32_t x) {
  x = dpp_min<0x140>(x);  // row_mirror
  x = dpp_min<0x141>(x);  // row_half_mirror
  x = dpp_min<0x4e>(x);   // quad_perm [2, 3, 0, 1]
  x = dpp_min<0xb1>(x);   // quad_perm [1, 0, 3, 2]
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  x = min((int32_t)r[0], (int32_t)r[1]);
  const auto h = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return min((int32_t)h[0], (int32_t)h[1]);
}
__device__ __forceinline__ int32_t wave_max_i(int32_t x) { return ~wave_min(~x); }

__global__ __launch_bounds__(kThreads) void classify_kernel(const Pred pred, int32_t N, int32_t BQ,
                                                             int32_t A, uint32_t* __restrict__ codes,
                                                             int32_t* __restrict__ kv_num,
                                                             unsigned long long* __restrict__ totals) {
  __shared__ int32_t q_orig[128];
  __shared__ uint32_t tile_code[kChunk / 16];
  __shared__ int32_t red_live[kThreads / 64];
  __shared__ int32_t red_tiles;
  __shared__ int32_t q_lo[4], q_hi[4];
  __shared__ pa_term terms_s[PA_MAX_TERMS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int qb = blockIdx.x;
  const int split = blockIdx.y, splits = gridDim.y;
  const int nk = N / A;
  const int rg_rows = BQ < 32 ? BQ : 32;   // rows per wave group
  const int n_rg = BQ / rg_rows;
  const int cw = A < 32 ? A : 32;          // columns per wave group
  const int ncg = A / cw;

  if (tid < BQ) {
    const int r = qb * BQ + tid;
    q_orig[tid] = pred.perm_q ? pred.perm_q[r] : r;
  }
  if (tid == 0) red_tiles = 0;
#pragma unroll
  for (int i = 0; i < PA_MAX_TERMS; ++i)  // (constant indices into the argument block)
    if (tid == i) terms_s[i] = pred.terms[i];
  __syncthreads();
  if (wave < n_rg) {
    // the row groups' ranges (their rows, one per lane; lanes past them repeat)
    const int32_t qo = q_orig[wave * rg_rows + (lane & (rg_rows - 1))];
    const int32_t lo = wave_min(qo), hi = wave_max_i(qo);
    if (lane == 0) {
      q_lo[wave] = lo;
      q_hi[wave] = hi;
    }
  }
  __syncthreads();

  int32_t live_count = 0;
  int32_t tiles_listed = 0;  // meaningful in thread 0 only
  // pairs and tiles of the chunks decided at once (thread 0's count)
  long long live_whole = 0;
  int32_t tiles_whole = 0;
  const int log2a = 31 - __builtin_clz((unsigned)A), log2cw = 31 - __builtin_clz((unsigned)cw);
  Range rw;
  rw.q0 = q_lo[0];
  rw.q1 = q_hi[0];
  for (int g = 1; g < n_rg; ++g) {
    rw.q0 = min(rw.q0, q_lo[g]);
    rw.q1 = max(rw.q1, q_hi[g]);
  }
  const uint32_t all_code = n_rg * ncg == 16 ? ~0u : (1u << (2 * n_rg * ncg)) - 1u;

  for (int c0 = split * kChunk; c0 < N; c0 += splits * kChunk) {
    if (!pred.perm_kv) {
      // a chunk of columns in order that is live or dead as a whole (uniform: no barrier)
      rw.k0 = c0;
      rw.k1 = min(c0 + kChunk, N) - 1;
      const Verdict v =
          pred_verdict(terms_s, pred.n_include, pred.n_exclude, rw, [](int32_t p) -> int { return p == 1 ? 1 : -1; });
      if (v != kMixed) {
        const int cols = rw.k1 - c0 + 1, tiles = cols >> log2a;
        if (tid < tiles) codes[(int64_t)qb * nk + (c0 >> log2a) + tid] = v == kLive ? all_code : 0u;
        if (v == kLive) {
          live_whole += (long long)cols * BQ;
          tiles_whole += tiles;
        }
        continue;
      }
    }
    if (tid < kChunk / 16) tile_code[tid] = 0u;
    __syncthreads();

    const int col = c0 + tid;
    const bool valid = col < N;
    uint32_t any_rg = 0u, all_rg = 0u;
    if (c0 + wave * 64 < N) {  // (uniform; lane 0's column is then valid)
      int32_t ko = valid ? (pred.perm_kv ? pred.perm_kv[col] : col) : 0;
      const int32_t ko0 = __shfl(ko, 0);
      if (!valid) ko = ko0;  // a lane past the end stands for a column of the block
      Range r;
      if (pred.perm_kv) {
        r.k0 = wave_min(ko);
        r.k1 = wave_max_i(ko);
      } else {
        r.k0 = c0 + wave * 64;
        r.k1 = min(c0 + wave * 64 + 64, N) - 1;
      }
      // columns from all over the sequence (a random permutation): hardly a block is decided
      const bool wide = pred.perm_kv && r.k1 - r.k0 >= N >> 1;
      for (int g = 0; g < n_rg; ++g) {
        const int32_t qo = q_orig[g * rg_rows + (lane & (rg_rows - 1))];
        r.q0 = q_lo[g];
        r.q1 = q_hi[g];
        auto same = [&](int32_t p) -> int {
          const int32_t rq = qo % p, rk = ko % p;
          const int32_t rq0 = __builtin_amdgcn_readfirstlane(rq), rk0 = __builtin_amdgcn_readfirstlane(rk);
          if (__ballot(rq != rq0 || rk != rk0) != 0ull) return -1;
          return rq0 == rk0 ? 1 : 0;
        };
        const Verdict v = wide ? kMixed : pred_verdict(terms_s, pred.n_include, pred.n_exclude, r, same);
        bool any = v == kLive, all = v == kLive;
        if (v == kMixed) {
          all = true;
          int32_t n = 0;
          for (int rr = 0; rr < rg_rows; ++rr) {
            const bool live = pred_live(pred, q_orig[g * rg_rows + rr], ko);
            any |= live;
            all &= live;
            n += live ? 1 : 0;
          }
          if (valid) live_count += n;
        } else if (v == kLive && valid) {
          live_count += rg_rows;
        }
        any_rg |= (any ? 1u : 0u) << g;
        all_rg |= (all ? 1u : 0u) << g;
      }
    }
    // Column reduction inside each wave: a column group never straddles a wave.
    const int wave_col0 = c0 + wave * 64;
    for (int g = 0; g < n_rg; ++g) {
      const unsigned long long b_any = __ballot((any_rg >> g) & 1u);
      const unsigned long long b_all = __ballot((all_rg >> g) & 1u);
      const int ngroups_in_wave = 64 / cw;
      if (lane < ngroups_in_wave) {
        const int gc0 = wave_col0 + lane * cw;  // first column of this column group
        if (gc0 < N) {
          const unsigned long long gm = (cw == 64 ? ~0ull : ((1ull << cw) - 1ull)) << (lane * cw);
          const bool gany = (b_any & gm) != 0ull;
          const bool gall = (b_all & gm) == gm;
          const int cg = (gc0 & (A - 1)) >> log2cw;
          const int code_g = g * ncg + cg;
          const uint32_t bits = (gany ? 1u : 0u) << (2 * code_g) | (gall ? 1u : 0u) << (2 * code_g + 1);
          if (bits) atomicOr(&tile_code[(gc0 - c0) >> log2a], bits);
        }
      }
    }
    __syncthreads();
    const int tiles_in_chunk = kChunk >> log2a;
    if (tid < tiles_in_chunk) {
      const int kb = (c0 >> log2a) + tid;
      if (kb < nk) {
        const uint32_t code = tile_code[tid];
        codes[(int64_t)qb * nk + kb] = code;
        if (code & 0x55555555u) atomicAdd(&red_tiles, 1);
      }
    }
    __syncthreads();
  }

  // live pairs: wave reduce, then one atomic per work-group
  for (int off = 32; off > 0; off >>= 1) live_count += __shfl_down(live_count, off, 64);
  if (lane == 0) red_live[wave] = live_count;
  __syncthreads();
  if (tid == 0) {
    long long tot = live_whole;
    for (int i = 0; i < kThreads / 64; ++i) tot += red_live[i];
    tiles_listed = red_tiles + tiles_whole;
    if (tiles_listed) atomicAdd(&kv_num[qb], tiles_listed);
    if (tot) atomicAdd(&totals[1], (unsigned long long)tot);
  }
}

__global__ __launch_bounds__(kThreads) void compact_kernel(const uint32_t* __restrict__ codes,
                                                            const int32_t* __restrict__ kv_num,
                                                            int32_t N, int32_t BQ, int32_t A,
                                                            uint32_t full_mask,
                                                            int32_t* __restrict__ kv_idx,
                                                            int8_t* __restrict__ kv_partial,
                                                            uint32_t* __restrict__ kv_wave_bits,
                                                            int64_t pitch) {
  __shared__ int32_t wave_tot[kThreads / 64];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int qb = blockIdx.x;
  const int nk = N / A;
  const int64_t row = (int64_t)qb * pitch;
  int base = 0;
  for (int k0 = 0; k0 < nk; k0 += kThreads) {
    const int kb = k0 + tid;
    const uint32_t code = kb < nk ? codes[(int64_t)qb * nk + kb] : 0u;
    const bool listed = (code & 0x55555555u) != 0u;
    const unsigned long long bal = __ballot(listed);
    const int before_in_wave = __popcll(bal & ((1ull << lane) - 1ull));
    if (lane == 0) wave_tot[wave] = __popcll(bal);
    __syncthreads();
    int before = base + before_in_wave;
    int chunk_total = 0;
    for (int i = 0; i < kThreads / 64; ++i) {
      if (i < wave) before += wave_tot[i];
      chunk_total += wave_tot[i];
    }
    if (listed && before < pitch) {  // pitch >= kv_num is the caller's contract; never write past it
      kv_idx[row + before] = kb;
      kv_partial[row + before] = ((code & full_mask) == full_mask) ? 0 : 1;
      if (kv_wave_bits) kv_wave_bits[row + before] = code;
    }
    base += chunk_total;
    __syncthreads();
  }
  // zero padding up to the pitch (gpu/blockindex.py:44-45 allocates with np.zeros)
  const int n = kv_num[qb];
  for (int64_t j = n + tid; j < pitch; j += kThreads) {
    kv_idx[row + j] = 0;
    kv_partial[row + j] = 0;
    if (kv_wave_bits) kv_wave_bits[row + j] = 0u;
  }
}

// Partial tiles of each query block, then their exclusive prefix sum.
__global__ __launch_bounds__(kThreads) void part_count_kernel(const uint32_t* __restrict__ codes, int32_t nk,
                                                               uint32_t full_mask, int64_t* __restrict__ part_base) {
  __shared__ int32_t tot[kThreads / 64];
  const int tid = threadIdx.x;
  const uint32_t* row = codes + (int64_t)blockIdx.x * nk;
  int32_t n = 0;
  for (int k = tid; k < nk; k += kThreads) {
    const uint32_t c = row[k];
    n += ((c & 0x55555555u) != 0u && (c & full_mask) != full_mask) ? 1 : 0;
  }
  for (int off = 32; off > 0; off >>= 1) n += __shfl_down(n, off, 64);
  if ((tid & 63) == 0) tot[tid >> 6] = n;
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < kThreads / 64; ++i) n += tot[i];
    part_base[blockIdx.x] = n;
  }
}

__global__ __launch_bounds__(kThreads) void part_scan_kernel(int64_t* part_base, int32_t nq) {
  __shared__ long long wave_tot[kThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  long long base = 0;
  for (int i0 = 0; i0 < nq; i0 += kThreads) {
    const int i = i0 + tid;
    const long long n = i < nq ? (long long)part_base[i] : 0;
    long long sum = n;  // inclusive within the wave
    for (int off = 1; off < 64; off <<= 1) {
      const long long y = __shfl_up(sum, off, 64);
      if (lane >= off) sum += y;
    }
    if (lane == 63) wave_tot[wave] = sum;
    __syncthreads();
    long long before = base, total = 0;
    for (int u = 0; u < kThreads / 64; ++u) {
      if (u < wave) before += wave_tot[u];
      total += wave_tot[u];
    }
    if (i < nq) part_base[i] = before + sum - n;
    base += total;
    __syncthreads();
  }
  if (tid == 0) part_base[nq] = base;
}

// The codes' all-live bits of a tile.
uint32_t full_mask_of(int32_t BQ, int32_t A) {
  const int ngroups = (BQ / (BQ < 32 ? BQ : 32)) * (A / (A < 32 ? A : 32));
  uint32_t m = 0u;
  for (int g = 0; g < ngroups; ++g) m |= 2u << (2 * g);
  return m;
}

bool tile_ok(int32_t x) { return x == 16 || x == 32 || x == 64 || x == 128; }

}  // namespace
}  // namespace pa

extern "C" int pa_index_classify(const pa_mask* mask, int64_t N, int32_t BQ, int32_t A,
                                 uint32_t* tile_codes, int32_t* kv_num, unsigned long long* totals,
                                 void* stream) {
  PA_CHECK_ARG(mask != nullptr && tile_codes && kv_num && totals, "pa_index_classify: null argument");
  PA_CHECK_ARG(N >= 1 && N <= (1ll << 30), "pa_index_classify: N=%lld out of range", (long long)N);
  PA_CHECK_ARG(pa::tile_ok(BQ) && pa::tile_ok(A),
               "pa_index_classify: BQ=%d A=%d must each be one of 16, 32, 64, 128", BQ, A);
  PA_CHECK_ARG(N % BQ == 0 && N % A == 0, "pa_index_classify: N=%lld not divisible by BQ=%d and A=%d",
               (long long)N, BQ, A);
  if (int rc = pa::check_mask(mask, N)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const pa::Pred pred = pa::make_pred(*mask);
  const int64_t nq = N / BQ;
  hipLaunchKernelGGL(pa::zero_totals_kernel, dim3((unsigned)((nq + 3 + 255) / 256)), dim3(256), 0, s, totals, kv_num,
                     (int32_t)nq);
  PA_LAUNCH_CHECK("zero_totals_kernel");
  // enough column splits for about 2048 work-groups (the chip holds ~2048 of 256 threads;
  // 1024 were 10 to 45% slower)
  const int64_t chunks = (N + pa::kChunk - 1) / pa::kChunk;
  int64_t splits = (2048 + nq - 1) / nq;
  if (splits > chunks) splits = chunks;
  if (splits < 1) splits = 1;
  hipLaunchKernelGGL(pa::classify_kernel, dim3((unsigned)nq, (unsigned)splits), dim3(pa::kThreads), 0, s, pred,
                     (int32_t)N, BQ, A, tile_codes, kv_num, totals);
  PA_LAUNCH_CHECK("classify_kernel");
  hipLaunchKernelGGL(pa::max_list_kernel, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, s, kv_num,
                     (int32_t)nq, totals);
  PA_LAUNCH_CHECK("max_list_kernel");
  return PA_OK;
}

extern "C" int pa_index_part_base(const uint32_t* tile_codes, int64_t N, int32_t BQ, int32_t A, int64_t* part_base,
                                  void* stream) {
  PA_CHECK_ARG(tile_codes && part_base, "pa_index_part_base: null argument");
  PA_CHECK_ARG(N >= 1 && N <= (1ll << 30), "pa_index_part_base: N=%lld out of range", (long long)N);
  PA_CHECK_ARG(pa::tile_ok(BQ) && pa::tile_ok(A) && N % BQ == 0 && N % A == 0,
               "pa_index_part_base: bad tile shape BQ=%d A=%d for N=%lld", BQ, A, (long long)N);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int32_t nq = (int32_t)(N / BQ);
  hipLaunchKernelGGL(pa::part_count_kernel, dim3((unsigned)nq), dim3(pa::kThreads), 0, s, tile_codes, (int32_t)(N / A),
                     pa::full_mask_of(BQ, A), part_base);
  PA_LAUNCH_CHECK("part_count_kernel");
  hipLaunchKernelGGL(pa::part_scan_kernel, dim3(1), dim3(pa::kThreads), 0, s, part_base, nq);
  PA_LAUNCH_CHECK("part_scan_kernel");
  return PA_OK;
}

extern "C" int pa_index_compact(const uint32_t* tile_codes, const int32_t* kv_num, int64_t N, int32_t BQ,
                                int32_t A, int32_t* kv_idx, int8_t* kv_partial, uint32_t* kv_wave_bits,
                                int64_t pitch, void* stream) {
  PA_CHECK_ARG(tile_codes && kv_num, "pa_index_compact: null argument");
  PA_CHECK_ARG(N >= 1 && N <= (1ll << 30), "pa_index_compact: N=%lld out of range", (long long)N);
  PA_CHECK_ARG(pa::tile_ok(BQ) && pa::tile_ok(A) && N % BQ == 0 && N % A == 0,
               "pa_index_compact: bad tile shape BQ=%d A=%d for N=%lld", BQ, A, (long long)N);
  PA_CHECK_ARG(pitch >= 0, "pa_index_compact: negative pitch");
  if (pitch == 0) return PA_OK;  // every query block is empty: nothing to write
  PA_CHECK_ARG(kv_idx && kv_partial, "pa_index_compact: null output");
  const uint32_t full_mask = pa::full_mask_of(BQ, A);
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(pa::compact_kernel, dim3((unsigned)(N / BQ)), dim3(pa::kThreads), 0, s, tile_codes,
                     kv_num, (int32_t)N, BQ, A, full_mask, kv_idx, kv_partial, kv_wave_bits, pitch);
  PA_LAUNCH_CHECK("compact_kernel");
  return PA_OK;
}

// ---------------------------------------------------------------------------
// Element bitmaps of the listed partial tiles (phase 3).  One work-group per query block
// takes its list 256 entries at a time, one per thread: the flags are ranked with ballots
// (one dependent load per 256 entries, not per entry) and the partial tiles collected in
// LDS; then each gets BQ x ceil(A/32) words, one thread per word, 32 predicate evaluations
// per word.
namespace pa {
namespace {

__global__ __launch_bounds__(kThreads) void bits_kernel(const Pred pred, int32_t N, int32_t BQ, int32_t A,
                                                         const int32_t* __restrict__ kv_idx,
                                                         const int32_t* __restrict__ kv_num,
                                                         const int8_t* __restrict__ kv_partial, int64_t pitch,
                                                         const int64_t* __restrict__ part_base,
                                                         int32_t* __restrict__ kv_bits_off,
                                                         uint32_t* __restrict__ pool) {
  __shared__ int32_t q_orig[128];
  const int tid = threadIdx.x;
  const int qb = blockIdx.x;
  const int wpr = (A + 31) >> 5;
  const int words = BQ * wpr;
  if (tid < BQ) {
    const int r = qb * BQ + tid;
    q_orig[tid] = pred.perm_q ? pred.perm_q[r] : r;
  }
  __syncthreads();
  __shared__ int32_t part_kb[kThreads];
  __shared__ int32_t wave_tot[kThreads / 64];
  const int lane = tid & 63, wave = tid >> 6;
  const int n = kv_num[qb];
  const int64_t row = (int64_t)qb * pitch;
  int64_t rank = part_base[qb];
  for (int j0 = 0; j0 < n; j0 += kThreads) {
    const int j = j0 + tid;
    const bool partial = j < n && kv_partial[row + j] != 0;
    const unsigned long long bal = __ballot(partial);
    if (lane == 0) wave_tot[wave] = __popcll(bal);
    __syncthreads();
    int before = __popcll(bal & ((1ull << lane) - 1ull)), total = 0;
    for (int i = 0; i < kThreads / 64; ++i) {
      if (i < wave) before += wave_tot[i];
      total += wave_tot[i];
    }
    if (j < n) kv_bits_off[row + j] = partial ? (int32_t)((rank + before) * words) : -1;
    if (partial) part_kb[before] = kv_idx[row + j];
    __syncthreads();
    for (int x = tid; x < total * words; x += kThreads) {
      const int u = x / words, wi = x - u * words;
      const int rr = wi / wpr, cw = wi % wpr;
      const int c0 = part_kb[u] * A + cw * 32;
      const int ncol = A - cw * 32 < 32 ? A - cw * 32 : 32;
      uint32_t bits = 0u;
      for (int c = 0; c < ncol; ++c) {
        const int col = c0 + c;
        const int32_t ko = pred.perm_kv ? pred.perm_kv[col] : col;
        bits |= (pred_live(pred, q_orig[rr], ko) ? 1u : 0u) << c;
      }
      pool[(rank + u) * words + wi] = bits;
    }
    __syncthreads();  // part_kb and wave_tot are read
    rank += total;
  }
  for (int64_t j = n + tid; j < pitch; j += kThreads) kv_bits_off[row + j] = -1;
}

}  // namespace
}  // namespace pa

extern "C" int pa_index_bits(const pa_mask* mask, int64_t N, int32_t BQ, int32_t A, const int32_t* kv_idx,
                             const int32_t* kv_num, const int8_t* kv_partial, int64_t pitch,
                             const int64_t* part_base, int32_t* kv_bits_off, uint32_t* pool, void* stream) {
  PA_CHECK_ARG(mask && kv_num && part_base, "pa_index_bits: null argument");
  PA_CHECK_ARG(N >= 1 && N <= (1ll << 30), "pa_index_bits: N=%lld out of range", (long long)N);
  PA_CHECK_ARG(pa::tile_ok(BQ) && pa::tile_ok(A) && N % BQ == 0 && N % A == 0,
               "pa_index_bits: bad tile shape BQ=%d A=%d for N=%lld", BQ, A, (long long)N);
  if (pitch == 0) return PA_OK;
  PA_CHECK_ARG(kv_idx && kv_partial && kv_bits_off, "pa_index_bits: null list");
  if (int rc = pa::check_mask(mask, N)) return rc;
  const pa::Pred pred = pa::make_pred(*mask);
  hipLaunchKernelGGL(pa::bits_kernel, dim3((unsigned)(N / BQ)), dim3(pa::kThreads), 0,
                     static_cast<hipStream_t>(stream), pred, (int32_t)N, BQ, A, kv_idx, kv_num, kv_partial,
                     pitch, part_base, kv_bits_off, pool);
  PA_LAUNCH_CHECK("bits_kernel");
  return PA_OK;
}

// ---------------------------------------------------------------------------
// Step descriptors of the streaming attention kernel: one thread per (query block,
// step of 64 kv columns), 64 bytes out, written as four 16-byte stores.
namespace pa {
namespace {

__global__ __launch_bounds__(kThreads) void steps_kernel(const int32_t* __restrict__ kv_idx,
                                                          const int32_t* __restrict__ kv_num,
                                                          const int8_t* __restrict__ kv_partial,
                                                          const uint32_t* __restrict__ kv_wave_bits,
                                                          const int32_t* __restrict__ kv_bits_off, int64_t pitch,
                                                          int32_t nq, int32_t BQ, int32_t A, int32_t residue_s,
                                                          int32_t residue_qlog2, const int32_t* __restrict__ order,
                                                          int32_t* __restrict__ steps, int64_t steps_pitch) {
  const int64_t gid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (gid >= (int64_t)nq * steps_pitch) return;
  const int pos = (int)(gid / steps_pitch);  // issue position of the list
  const int qb = order ? order[pos] : pos;
  const int j = (int)(gid % steps_pitch);
  const int spt = A >> 4;                    // 16-column segments per tile
  const int n_seg = kv_num[qb] * spt;
  const int ncg = A >= 32 ? A >> 5 : 1;      // 32-column groups per tile
  const int ngr = BQ >= 32 ? BQ >> 5 : 1;    // 32-row groups per query block
  int32_t d[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) d[i] = 0;
  uint32_t code = 0u;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int seg = 4 * j + t;
    int32_t base = 0, boff = -1;
    uint32_t c8 = 0u;
    if (seg < n_seg) {
      const int64_t ti = (int64_t)qb * pitch + seg / spt;
      const int within = seg % spt;
      base = kv_idx[ti] * A + within * 16;
      if (residue_s > 0) {
        const int32_t rmask = (1 << residue_qlog2) - 1;
        base = (base & rmask) * residue_s + (base >> residue_qlog2);
      }
      if (kv_wave_bits) {
        const int cg = A >= 32 ? within >> 1 : 0;
        const uint32_t wb = kv_wave_bits[ti];
        for (int g = 0; g < ngr && g < 4; ++g) c8 |= ((wb >> (2 * (g * ncg + cg))) & 3u) << (2 * g);
      } else {
        c8 = kv_partial[ti] ? 0x55u : 0xffu;
      }
      if (kv_bits_off && kv_bits_off[ti] >= 0) boff = kv_bits_off[ti] + ((within * 16) >> 5);
    }
    d[t] = base;
    d[5 + t] = boff;
    code |= c8 << (8 * t);
  }
  d[4] = (int32_t)code;
  d[13] = qb;
  d[14] = (kv_num[qb] * A + 63) >> 6;
  d[15] = residue_s > 0 ? residue_s : 0;
  int4* dst = reinterpret_cast<int4*>(steps + gid * 16);
#pragma unroll
  for (int i = 0; i < 4; ++i) dst[i] = int4{d[4 * i], d[4 * i + 1], d[4 * i + 2], d[4 * i + 3]};
}

}  // namespace
}  // namespace pa

extern "C" int pa_index_steps(const int32_t* kv_idx, const int32_t* kv_num, const int8_t* kv_partial,
                              const uint32_t* kv_wave_bits, const int32_t* kv_bits_off, int64_t pitch, int64_t N,
                              int32_t BQ, int32_t A, int32_t residue_s, int32_t residue_qlog2,
                              const int32_t* order, int32_t* steps, int64_t steps_pitch, void* stream) {
  PA_CHECK_ARG(kv_num, "pa_index_steps: null kv_num");
  PA_CHECK_ARG(N >= 1 && N <= (1ll << 30), "pa_index_steps: N=%lld out of range", (long long)N);
  PA_CHECK_ARG(pa::tile_ok(BQ) && pa::tile_ok(A) && N % BQ == 0 && N % A == 0,
               "pa_index_steps: bad tile shape BQ=%d A=%d for N=%lld", BQ, A, (long long)N);
  PA_CHECK_ARG(pitch >= 0, "pa_index_steps: negative pitch");
  PA_CHECK_ARG(residue_s <= 0 || (residue_qlog2 >= 4 && residue_qlog2 < 31 &&
                                  (int64_t)residue_s << residue_qlog2 == N),
               "pa_index_steps: residue_s=%d with N/s = 2^%d does not match N=%lld", residue_s, residue_qlog2,
               (long long)N);
  PA_CHECK_ARG(steps_pitch >= (pitch * A + 63) / 64,
               "pa_index_steps: steps_pitch=%lld < ceil(pitch * A / 64) = %lld", (long long)steps_pitch,
               (long long)((pitch * A + 63) / 64));
  const int64_t nq = N / BQ;
  const int64_t total = nq * steps_pitch;
  if (total == 0) return PA_OK;
  PA_CHECK_ARG(steps, "pa_index_steps: null steps");
  PA_CHECK_ARG(pitch == 0 || (kv_idx && kv_partial), "pa_index_steps: null list");
  PA_CHECK_ARG((reinterpret_cast<uintptr_t>(steps) & 15) == 0, "pa_index_steps: steps must be 16-byte aligned");
  PA_CHECK_ARG(total / pa::kThreads < 0x7fffffffll, "pa_index_steps: too many steps");
  hipLaunchKernelGGL(pa::steps_kernel, dim3((unsigned)((total + pa::kThreads - 1) / pa::kThreads)),
                     dim3(pa::kThreads), 0, static_cast<hipStream_t>(stream), kv_idx, kv_num, kv_partial,
                     kv_wave_bits, kv_bits_off, pitch, (int32_t)nq, BQ, A, residue_s > 0 ? residue_s : 0,
                     residue_qlog2, order, steps, steps_pitch);
  PA_LAUNCH_CHECK("steps_kernel");
  return PA_OK;
}

namespace pa {
namespace {

// One work-group of 64 threads per item: its run rows are its list's steps (from the
// descriptors of its piece) with the K / V rows moved to the item's head, the bitmap
// offsets moved to the piece's part of a shared pool, and the item written into words
// 9 to 11.
struct RunPieces {
  const int32_t* steps[2];
  int64_t pitch[2];
  int32_t boff_base[2];
};

__global__ __launch_bounds__(64) void run_kernel(const RunPieces pcs, int64_t N, const int32_t* __restrict__ item_piece,
                                                 const int32_t* __restrict__ item_bh,
                                                 const int32_t* __restrict__ item_qb,
                                                 const int32_t* __restrict__ item_sync,
                                                 const int32_t* __restrict__ item_off, int32_t* __restrict__ run) {
  const int i = blockIdx.x;
  const int pc = item_piece ? item_piece[i] : 0;
  const int32_t bh = item_bh[i], qb = item_qb[i];
  const int32_t sg = item_sync ? item_sync[i] : -1;
  const int32_t r0 = item_off[i], len = item_off[i + 1] - r0;
  const int32_t* list = (pc ? pcs.steps[1] : pcs.steps[0]) + (int64_t)qb * (pc ? pcs.pitch[1] : pcs.pitch[0]) * 16;
  const int32_t bbase = pc ? pcs.boff_base[1] : pcs.boff_base[0];
  const int32_t n_list = list[14];  // the list's number of steps (0: an empty list)
  const int32_t head_row = (int32_t)(bh * N);
  for (int j = threadIdx.x; j < len; j += 64) {
    int32_t d[16];
    if (j < n_list) {
      const int4* src = reinterpret_cast<const int4*>(list + (int64_t)j * 16);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int4 x = src[u];
        d[4 * u] = x.x;
        d[4 * u + 1] = x.y;
        d[4 * u + 2] = x.z;
        d[4 * u + 3] = x.w;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (d[5 + t] >= 0) d[5 + t] += bbase;
    } else {
      // the one step of an empty list: every code 0 (the scores are -inf), rows 0 of the
      // head (valid memory), no bitmaps
#pragma unroll
      for (int u = 0; u < 16; ++u) d[u] = 0;
#pragma unroll
      for (int t = 0; t < 4; ++t) d[5 + t] = -1;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) d[t] += head_row;
    d[9] = (j == 0 ? 1 : 0) | (j == len - 1 ? 2 : 0) | (pc ? 4 : 0) | (qb << 3);
    d[10] = bh;
    d[11] = sg;
    int4* dst = reinterpret_cast<int4*>(run + ((int64_t)r0 + j) * 16);
#pragma unroll
    for (int u = 0; u < 4; ++u) dst[u] = int4{d[4 * u], d[4 * u + 1], d[4 * u + 2], d[4 * u + 3]};
  }
}

}  // namespace
}  // namespace pa

extern "C" int pa_index_run(const int32_t* const* steps, const int64_t* steps_pitch, const int32_t* boff_base,
                            int32_t n_pieces, int64_t N, const int32_t* item_piece, const int32_t* item_bh,
                            const int32_t* item_qb, const int32_t* item_sync, const int32_t* item_off, int32_t n_items,
                            int32_t* run, void* stream) {
  PA_CHECK_ARG(n_items >= 0, "pa_index_run: n_items=%d", n_items);
  if (n_items == 0) return PA_OK;
  PA_CHECK_ARG(n_pieces == 1 || n_pieces == 2, "pa_index_run: n_pieces=%d (1 or 2)", n_pieces);
  PA_CHECK_ARG(steps && steps_pitch && item_bh && item_qb && item_off && run, "pa_index_run: null argument");
  PA_CHECK_ARG(n_pieces == 1 || item_piece, "pa_index_run: two pieces need item_piece");
  PA_CHECK_ARG(N >= 1 && N <= (1ll << 30), "pa_index_run: N=%lld out of range", (long long)N);
  pa::RunPieces pcs{};
  for (int p = 0; p < n_pieces; ++p) {
    PA_CHECK_ARG(steps[p] && steps_pitch[p] >= 1, "pa_index_run: piece %d has no descriptors", p);
    PA_CHECK_ARG((reinterpret_cast<uintptr_t>(steps[p]) & 15) == 0, "pa_index_run: steps not 16-byte aligned");
    pcs.steps[p] = steps[p];
    pcs.pitch[p] = steps_pitch[p];
    pcs.boff_base[p] = boff_base ? boff_base[p] : 0;
    PA_CHECK_ARG(pcs.boff_base[p] >= 0, "pa_index_run: negative bitmap base");
  }
  PA_CHECK_ARG((reinterpret_cast<uintptr_t>(run) & 15) == 0, "pa_index_run: run must be 16-byte aligned");
  hipLaunchKernelGGL(pa::run_kernel, dim3((unsigned)n_items), dim3(64), 0, static_cast<hipStream_t>(stream), pcs, N,
                     item_piece, item_bh, item_qb, item_sync, item_off, run);
  PA_LAUNCH_CHECK("run_kernel");
  return PA_OK;
}
