// Block selection and cross-head pattern sharing on the device, with no host synchronisation.
// Replaces the torch-op chains of shareprefill/attn/attention_sharing.py:169-364 and :94-103 and the
// helpers of shareprefill/attn/utils.py:26-128.
//
// Canonical arithmetic shared with the CPU oracle:
//   * order = (value descending, index ascending), compared on the fp32 bit pattern (sp_sort_key);
//   * cumulative mass = exact integer sums of values truncated to 2^-48 fixed point (sp_to_fixed),
//     so every comparison against a threshold is independent of summation order (integer atomics
//     and scans may associate freely).
// Two primitives:
//   * radix mass descent for long vectors (per-token vectors of length N, the nb*nb pooled map), from (count, mass)
//     histograms over the key's bits: one workgroup per vector in four levels of 8/8/8/7 bits up to GSEL_ONE_LEN values
//     and GSEL_ONE_NB blocks, many workgroups per vector in three levels of 11/11/10 bits beyond;
//   * rank sort for short vectors (rows of length nb): rank by pairwise comparison in LDS, scatter to
//     sorted order, integer prefix scan -- a literal sort / cumsum / threshold.
#include <cstring>

#include "sp_block_probs.h"
#include "sp_pool.h"
#include "sp_repack.h"
#include "sp_rows.h"

#define SEL_THREADS 1024
#define SEL_BINS 2048

// ------------------------------------------------------------------------------------------------
// radix mass descent: shared state of the per-vector pick step (one workgroup of SEL_THREADS threads)
// ------------------------------------------------------------------------------------------------
struct SelShared {
  unsigned long long sum[SEL_BINS];
  uint32_t cnt[SEL_BINS];
  unsigned long long sum_above;
  uint32_t cnt_above;
  int32_t bin;
  uint32_t bin_cnt;
  unsigned long long bin_sum;
};

// suffix-inclusive scan of sh.sum over SEL_BINS bins (bin b <- sum of bins >= b), all SEL_THREADS threads.
// Thread t owns bins t and t + SEL_THREADS.  Inside a wave (64 consecutive bins of either half) the suffix sums come
// from lane shuffles; the waves' totals meet in LDS.  Integer sums: any association gives the same result.
__device__ static void sel_suffix_scan(SelShared& sh) {
  __shared__ unsigned long long wave_tot[2][SEL_THREADS / SP_WAVE];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  unsigned long long v0 = sh.sum[t], v1 = sh.sum[t + SEL_THREADS];
#pragma unroll
  for (int off = 1; off < SP_WAVE; off <<= 1) {
    const unsigned long long a0 = __shfl_down(v0, off, SP_WAVE), a1 = __shfl_down(v1, off, SP_WAVE);
    if (lane + off < SP_WAVE) {
      v0 += a0;
      v1 += a1;
    }
  }
  if (lane == 0) {
    wave_tot[0][wave] = v0;
    wave_tot[1][wave] = v1;
  }
  __syncthreads();
  unsigned long long above0 = 0, above1 = 0;  // bins of the same half in higher waves
#pragma unroll
  for (int w = 0; w < SEL_THREADS / SP_WAVE; ++w) {
    if (w > wave) {
      above0 += wave_tot[0][w];
      above1 += wave_tot[1][w];
    }
    above0 += wave_tot[1][w];  // the whole upper half lies above every bin of the lower half
  }
  sh.sum[t] = v0 + above0;
  sh.sum[t + SEL_THREADS] = v1 + above1;
  __syncthreads();
}

// ---- score_cover_idx (attn/utils.py:53-57) on [nb][nb] maps, written into bit masks -----------------
// Multi-workgroup radix mass descent over the LOWER TRIANGLE of each map (entries above the diagonal are
// exactly zero in the reference's maps and cannot be selected; they are ignored here).  Per level: many
// workgroups per vector build LDS histograms of their rows and merge them into a global (count, mass)
// histogram with integer atomics; one workgroup per vector then picks the bin in which the running mass
// crosses the budget.  A row-parallel kernel writes the mask bits.  Only when the boundary falls inside a
// group of equal values that is taken partially (lowest indices first) a sequential kernel ranks them.
#define GSEL_SPLIT 64     // workgroups per vector in the histogram / emit kernels
#define GSEL_THREADS 256

struct GselState {
  unsigned long long rem;   // budget left after the bins / groups above the current prefix
  uint32_t prefix;          // key bits fixed so far
  uint32_t above;           // elements with key above the cut
  uint32_t n_equal, n_take; // boundary group
  int32_t all;              // 1: the whole vector is kept
  int32_t enabled;
  uint32_t pad[8];
};

__device__ static inline bool gsel_enabled(const int32_t* enable, int enable_match, int v) {
  if (!enable) return true;
  const int e = enable[v];
  return enable_match < 0 ? (e != 0) : (e == enable_match);
}

__global__ void sp_gsel_init_kernel(GselState* st, uint32_t* cnt, unsigned long long* sum, const int32_t* enable,
                                    int enable_match, int n_vec, long long t_le, uint64_t* mask, int nb, int nbw) {
  const int v = blockIdx.x;
  for (int i = threadIdx.x; i < SEL_BINS; i += blockDim.x) {
    cnt[(int64_t)v * SEL_BINS + i] = 0;
    sum[(int64_t)v * SEL_BINS + i] = 0;
  }
  if (threadIdx.x == 0) {
    GselState s;
    s.rem = t_le < 0 ? 0ull : (unsigned long long)t_le;
    s.prefix = 0;
    s.above = 0;
    s.n_equal = 0;
    s.n_take = 0;
    s.all = 0;
    s.enabled = (gsel_enabled(enable, enable_match, v) && t_le >= 0) ? 1 : 0;
    for (int i = 0; i < 8; ++i) s.pad[i] = 0;
    st[v] = s;
    if (mask != nullptr && gsel_enabled(enable, enable_match, v))  // block (0,0): the padding id of the reference
      atomicOr(reinterpret_cast<uint32_t*>(mask + (int64_t)v * nb * nbw), 1u);
  }
}

template <int LEVEL>
__global__ __launch_bounds__(GSEL_THREADS) void sp_gsel_hist_kernel(const float* __restrict__ x, int nb,
                                                                    const GselState* __restrict__ st,
                                                                    uint32_t* __restrict__ gcnt,
                                                                    unsigned long long* __restrict__ gsum) {
  __shared__ unsigned long long lsum[SEL_BINS];
  __shared__ uint32_t lcnt[SEL_BINS];
  const int v = blockIdx.y;
  const GselState s = st[v];
  if (!s.enabled || s.all) return;
  constexpr int shift = LEVEL == 0 ? 21 : (LEVEL == 1 ? 10 : 0);
  constexpr int width = LEVEL == 2 ? 10 : 11;
  constexpr int pshift = LEVEL == 0 ? 32 : (LEVEL == 1 ? 21 : 10);
  for (int i = threadIdx.x; i < SEL_BINS; i += GSEL_THREADS) {
    lsum[i] = 0;
    lcnt[i] = 0;
  }
  __syncthreads();
  const float* xv = x + (int64_t)v * nb * nb;
  for (int r = blockIdx.x; r < nb; r += GSEL_SPLIT) {
    const float* row = xv + (int64_t)r * nb;
    for (int c = threadIdx.x; c <= r; c += GSEL_THREADS) {
      const float val = row[c];
      const uint32_t key = sp_sort_key(val);
      if (pshift < 32 && (key >> (pshift & 31)) != s.prefix) continue;
      const uint32_t b = (key >> shift) & ((1u << width) - 1u);
      atomicAdd(&lcnt[b], 1u);
      const unsigned long long fx = sp_to_fixed(val);
      if (fx) atomicAdd(&lsum[b], fx);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < (1 << width); i += GSEL_THREADS) {
    if (lcnt[i]) atomicAdd(&gcnt[(int64_t)v * SEL_BINS + i], lcnt[i]);
    if (lsum[i]) atomicAdd(&gsum[(int64_t)v * SEL_BINS + i], lsum[i]);
  }
}

// One level of the descent on a histogram that sits in sh.sum / sh.cnt: finds the bin in which the running mass
// (from the top bin down) first exceeds the budget left, and moves the state below it.  Called by all SEL_THREADS
// threads of a workgroup with the same `s`; every thread returns with the same updated `s`.  sh may be refilled
// afterwards (the function ends with a barrier).
template <int LEVEL>
__device__ static void sel_pick_level(SelShared& sh, GselState& s) {
  const int t = threadIdx.x;
  constexpr int width = LEVEL == 2 ? 10 : 11;
  const int nbins = 1 << width;
  if (t == 0) {
    sh.bin = -1;
    sh.cnt_above = 0;
  }
  __syncthreads();
  const unsigned long long own0 = sh.sum[t], own1 = sh.sum[t + SEL_THREADS];
  __syncthreads();
  sel_suffix_scan(sh);
#pragma unroll
  for (int rep = 0; rep < 2; ++rep) {
    const int b = t + rep * SEL_THREADS;
    if (b < nbins) {
      const unsigned long long incl = sh.sum[b];
      const unsigned long long excl = (b + 1 < SEL_BINS) ? sh.sum[b + 1] : 0ull;
      if (incl > s.rem && excl <= s.rem) {
        sh.bin = b;
        sh.sum_above = excl;
        sh.bin_sum = rep ? own1 : own0;
        sh.bin_cnt = sh.cnt[b];
      }
    }
  }
  __syncthreads();
  const int bin = sh.bin;
  if (bin < 0) {  // the running mass never exceeds the budget (top level only): keep everything
    s.all = 1;
    __syncthreads();
    return;
  }
  uint32_t c = 0;
#pragma unroll
  for (int rep = 0; rep < 2; ++rep) {
    const int b = t + rep * SEL_THREADS;
    if (b < nbins && b > bin) c += sh.cnt[b];
  }
  if (c) atomicAdd(&sh.cnt_above, c);
  __syncthreads();
  s.prefix = (s.prefix << width) | (uint32_t)bin;
  s.above += sh.cnt_above;
  s.rem -= sh.sum_above;
  if (LEVEL == 2) {
    s.n_equal = sh.bin_cnt;
    const unsigned long long each = sh.bin_sum / (sh.bin_cnt ? sh.bin_cnt : 1u);
    unsigned long long take = each ? s.rem / each : (unsigned long long)s.n_equal;
    if (take > s.n_equal) take = s.n_equal;
    s.n_take = (uint32_t)take;
  }
  __syncthreads();
}

template <int LEVEL>
__global__ __launch_bounds__(SEL_THREADS) void sp_gsel_pick_kernel(GselState* __restrict__ st,
                                                                   uint32_t* __restrict__ gcnt,
                                                                   unsigned long long* __restrict__ gsum) {
  __shared__ SelShared sh;
  const int v = blockIdx.x, t = threadIdx.x;
  GselState s = st[v];
  if (!s.enabled || s.all) return;
  uint32_t* gc = gcnt + (int64_t)v * SEL_BINS;
  unsigned long long* gs = gsum + (int64_t)v * SEL_BINS;
  sh.sum[t] = gs[t];
  sh.sum[t + SEL_THREADS] = gs[t + SEL_THREADS];
  sh.cnt[t] = gc[t];
  sh.cnt[t + SEL_THREADS] = gc[t + SEL_THREADS];
  gs[t] = 0;  // ready for the next level
  gs[t + SEL_THREADS] = 0;
  gc[t] = 0;
  gc[t + SEL_THREADS] = 0;
  sel_pick_level<LEVEL>(sh, s);
  if (t == 0) st[v] = s;
}

// ---- the same descent by ONE workgroup per vector, histograms in LDS only -------------------------------------------
// The multi-workgroup descent is ten launches, most of them a few microseconds of launch latency.  Here one workgroup of
// CS_THREADS threads makes the passes over its vector itself; keys, fixed-point masses, pick rule and tie rule are the
// same integers, so both paths select the same entries.
// What bounds it: LDS atomics on equal addresses (the values of a probability vector share few exponents, so the lanes of
// a wave meet in a handful of bins) and the barriers of the workgroup.  Hence four levels of 8, 8, 8 and 7 key bits
// with CS_COPIES histograms side by side, lane % CS_COPIES choosing one (at most four lanes of a wave on an address),
// two barriers per level, and a pick that every wave makes for itself from the 256 folded bins, without another barrier.
// Vectors of at most CS_ITEMS entries per thread stay in registers for all levels; longer ones are read again.
// 64 vectors, one launch against three levels of 2048 bins (one workgroup up to 16384 values, ten launches above): 3001
// values 16.7 -> 11.0 us, 16384 25.9 -> 14.5, 32768 58 -> 25, 131072 80 -> 75; at 262144 the ten launches take 106 us and
// one would take 109, hence GSEL_ONE_LEN (few vectors: cover_one_launch).  32 maps of 64 x 64 blocks 20.2 -> 12.8 us, 256 x 256
// 72 -> 41 (one map 42 -> 40) and, what most layers meet, no map enabled 30.6 -> 6.7; at 512 x 512 the ten launches are ahead
// (96 us against 227 with the entries read again in each level), hence GSEL_ONE_NB.
#define CS_THREADS 1024
#define CS_BINS 256
#define CS_COPIES 16
#define CS_ITEMS 16
struct CoverShared {
  unsigned long long sum[CS_BINS * CS_COPIES];
  uint32_t cnt[CS_BINS * CS_COPIES];
  unsigned long long bin_sum[CS_BINS];
  uint32_t bin_cnt[CS_BINS];
};

__device__ static inline GselState sel_fresh_state(long long t_le, bool enabled) {
  GselState s;
  s.rem = t_le < 0 ? 0ull : (unsigned long long)t_le;
  s.prefix = 0;
  s.above = 0;
  s.n_equal = 0;
  s.n_take = 0;
  s.all = 0;
  s.enabled = (enabled && t_le >= 0) ? 1 : 0;
  for (int i = 0; i < 8; ++i) s.pad[i] = 0;
  return s;
}

// Lane exchanges of the fold and the pick go through DPP moves: as LDS permutes (30 per level, times 16 waves) they cost
// more than everything else in a level.
template <int CTRL, int ROW_MASK = 0xf>
__device__ static __forceinline__ uint32_t cs_dpp(uint32_t v) {  // lanes without a source (or outside ROW_MASK) get 0
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}
template <int CTRL, int ROW_MASK = 0xf>
__device__ static __forceinline__ unsigned long long cs_dpp64(unsigned long long v) {
  return ((unsigned long long)cs_dpp<CTRL, ROW_MASK>((uint32_t)(v >> 32)) << 32) | cs_dpp<CTRL, ROW_MASK>((uint32_t)v);
}
template <int CTRL, int ROW_MASK = 0xf>
__device__ static __forceinline__ void cs_scan_step(uint32_t& c, unsigned long long& m) {
  c += cs_dpp<CTRL, ROW_MASK>(c);
  m += cs_dpp64<CTRL, ROW_MASK>(m);
}
__device__ static __forceinline__ uint32_t cs_lane(uint32_t v, int src) {  // src uniform
  return (uint32_t)__builtin_amdgcn_readlane((int)v, src);
}

// sp_to_fixed of a value whose key is normal or infinite (no sign, no NaN, no zero): one 64-bit shift
__device__ static __forceinline__ unsigned long long cs_fixed(uint32_t key) {
  const int right = 140 - (int)(key >> 23);  // floor(m 2^(e - 102)) = (m << 38) >> (140 - e), m < 2^24
  const unsigned long long m = (unsigned long long)((key & 0x7fffffu) | 0x800000u) << 38;
  return right < 0 ? SP_FX_SAT : m >> (right < 63 ? right : 63);
}

// histograms zero; ends with a barrier
__device__ static inline void cover_begin(CoverShared& sh) {
  for (int i = threadIdx.x; i < CS_BINS * CS_COPIES; i += CS_THREADS) {
    sh.sum[i] = 0;
    sh.cnt[i] = 0;
  }
  __syncthreads();
}

// One level: for_each(f) calls f(value) for each of this thread's values.  Called by all CS_THREADS threads with the same
// `s` and zero histograms; returns the same updated `s` to every thread and leaves the histograms zero again.
template <typename ForEach>
__device__ static inline void cover_level(CoverShared& sh, GselState& s, int level, ForEach&& for_each) {
  const int width = level == 3 ? 7 : 8;
  const int shift = level == 3 ? 0 : 23 - 8 * level;  // (the sign bit of a key is never set)
  const int t = threadIdx.x, lane = t & 63;
  const int copy = t & (CS_COPIES - 1);
  const uint32_t prefix = s.prefix;
  for_each([&](float val) {
    const uint32_t key = sp_sort_key(val);
    if ((key >> (shift + width)) != prefix || key < 0x00800000u) return;  // (zeros carry no mass: never the cut)
    const uint32_t at = ((key >> shift) & ((1u << width) - 1u)) * CS_COPIES + copy;
    atomicAdd(&sh.cnt[at], 1u);
    atomicAdd(&sh.sum[at], cs_fixed(key));
  });
  __syncthreads();
  {  // four threads fold a bin's copies and leave them zero; the masses of empty bins are not read
    const int bin = t >> 2, part = t & 3;
    uint4* pc = reinterpret_cast<uint4*>(sh.cnt + bin * CS_COPIES + part * 4);
    ulonglong2* ps = reinterpret_cast<ulonglong2*>(sh.sum + bin * CS_COPIES + part * 4);
    const uint4 c4 = *pc;
    uint32_t c = (c4.x + c4.y) + (c4.z + c4.w);
    unsigned long long m = 0;
    if (c) {
      const ulonglong2 s0 = ps[0], s1 = ps[1];
      m = (s0.x + s0.y) + (s1.x + s1.y);
      *pc = make_uint4(0, 0, 0, 0);
      ps[0] = ps[1] = make_ulonglong2(0, 0);
    }
    cs_scan_step<0xB1>(c, m);  // quad_perm [1, 0, 3, 2]
    cs_scan_step<0x4E>(c, m);  // quad_perm [2, 3, 0, 1]
    if (part == 0) {
      sh.bin_cnt[bin] = c;
      sh.bin_sum[bin] = m;
    }
  }
  __syncthreads();
  // every wave by itself: lane l owns bins 255 - 4 l .. 252 - 4 l, the running mass comes from the top.  (The next level's
  // fold overwrites the bins only behind that level's first barrier, which this wave reaches after its pick.)
  uint32_t c[4];
  unsigned long long m[4];
  {
    const uint4 c4 = *reinterpret_cast<const uint4*>(sh.bin_cnt + (CS_BINS - 4 - 4 * lane));
    const ulonglong2 lo = *reinterpret_cast<const ulonglong2*>(sh.bin_sum + (CS_BINS - 4 - 4 * lane));
    const ulonglong2 hi = *reinterpret_cast<const ulonglong2*>(sh.bin_sum + (CS_BINS - 2 - 4 * lane));
    c[0] = c4.w, c[1] = c4.z, c[2] = c4.y, c[3] = c4.x;
    m[0] = hi.y, m[1] = hi.x, m[2] = lo.y, m[3] = lo.x;
  }
  uint32_t c_incl = (c[0] + c[1]) + (c[2] + c[3]);
  unsigned long long m_incl = (m[0] + m[1]) + (m[2] + m[3]);
  const uint32_t c_own = c_incl;
  const unsigned long long m_own = m_incl;
  cs_scan_step<0x111>(c_incl, m_incl);       // row_shr 1, 2, 4, 8: inclusive scan of each row of 16 lanes
  cs_scan_step<0x112>(c_incl, m_incl);
  cs_scan_step<0x114>(c_incl, m_incl);
  cs_scan_step<0x118>(c_incl, m_incl);
  cs_scan_step<0x142, 0xa>(c_incl, m_incl);  // row_bcast15 into rows 1 and 3
  cs_scan_step<0x143, 0xc>(c_incl, m_incl);  // row_bcast31 into rows 2 and 3
  uint32_t c_above = c_incl - c_own, found = 0, f_above = 0, f_cnt = 0;
  unsigned long long m_above = m_incl - m_own, f_mass = 0;
  int f_bin = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {  // the first bin behind which the running mass exceeds what is left
    if (!found && m_above <= s.rem && m_above + m[u] > s.rem) {
      found = 1;
      f_bin = CS_BINS - 1 - 4 * lane - u;
      f_above = c_above;
      f_mass = m_above;
      f_cnt = c[u];
    }
    c_above += c[u];
    m_above += m[u];
  }
  const unsigned long long who = __ballot(found != 0);
  if (who == 0ull) {  // the running mass never exceeds the budget (top level only): keep everything
    s.all = 1;
    return;
  }
  const int src = __ffsll((long long)who) - 1;
  f_bin = (int)cs_lane((uint32_t)f_bin, src);
  f_above = cs_lane(f_above, src);
  f_cnt = cs_lane(f_cnt, src);
  f_mass = ((unsigned long long)cs_lane((uint32_t)(f_mass >> 32), src) << 32) | cs_lane((uint32_t)f_mass, src);
  s.prefix = (prefix << width) | (uint32_t)f_bin;
  s.above += f_above;
  s.rem -= f_mass;
  s.n_equal = f_cnt;
  if (level == 3) {  // the bin is one value: as many of its entries as the budget left holds
    const unsigned long long each = sp_to_fixed(__uint_as_float(s.prefix));
    unsigned long long take = each ? s.rem / each : (unsigned long long)f_cnt;
    if (take > f_cnt) take = f_cnt;
    s.n_take = (uint32_t)take;
  }
}

// COUNT: only the number of entries is wanted.  A bin of one entry then ends the descent: its mass exceeds what is left, so it is
// not taken (n_take 0).  Of a few thousand entries the third level's bin rarely holds two: layers of 3001 tokens 112.4 -> 110.7 us,
// 6177 of 64 channels 126.0 -> 123.3, 10007 of 28 heads 243.4 -> 241.3 (with the pivots' decisions asked for earlier in the
// attention of the first two).
template <bool COUNT = false, typename ForEach>
__device__ static inline void cover_descent(CoverShared& sh, GselState& s, ForEach&& for_each) {
  cover_begin(sh);
  // (a loop, not four instances: code that runs once per launch is paid for in instruction fetches)
#pragma unroll 1
  for (int level = 0; level < 4 && !s.all && !(COUNT && s.n_equal == 1); ++level) cover_level(sh, s, level, for_each);  // (uniform)
}

// flat vectors (score_cover_topk, the budgets): vectors 0..n0-1 are rows of x0, the others rows of x1
struct CoverCountArgs {
  const float *x0, *x1;
  int n0, len;
  long long t_le;
  int32_t *out0, *out1;
  int bs, minb, maxb;
};

__device__ static void cover_count_vector(CoverShared& sh, const CoverCountArgs& a, int v) {
  const float* xv = v < a.n0 ? a.x0 + (int64_t)v * a.len : a.x1 + (int64_t)(v - a.n0) * a.len;
  GselState s = sel_fresh_state(a.t_le, true);
  const int t = threadIdx.x, len = a.len;
  if (s.enabled) {
    float val[CS_ITEMS];
    auto load = [&](int i0) {  // CS_ITEMS loads in flight
#pragma unroll
      for (int i = 0; i < CS_ITEMS; ++i) {
        const int at = i0 + i * CS_THREADS + t;
        val[i] = at < len ? xv[at] : 0.f;
      }
    };
    auto each = [&](int i0, auto&& f) {
#pragma unroll
      for (int i = 0; i < CS_ITEMS; ++i) {
        if (i0 + i * CS_THREADS >= len) break;  // (uniform)
        f(val[i]);  // (past the end: zeros, which are left out of the histograms)
      }
    };
    if (len <= CS_ITEMS * CS_THREADS) {
      load(0);
      cover_descent<true>(sh, s, [&](auto&& f) { each(0, f); });
    } else {
      cover_descent<true>(sh, s, [&](auto&& f) {
        for (int i0 = 0; i0 < len; i0 += CS_ITEMS * CS_THREADS) {
          load(i0);
          each(i0, f);
        }
      });
    }
  }
  if (t == 0) {  // as sp_gsel_count_kernel
    long long m = 0;
    if (a.t_le >= 0) m = s.all ? (long long)len : (long long)s.above + s.n_take;
    long long r = m + 1;
    if (a.bs > 0) {
      r = r / a.bs + 1;
      if (r < a.minb) r = a.minb;
      if (r > a.maxb) r = a.maxb;
    }
    if (v < a.n0)
      a.out0[v] = (int32_t)r;
    else
      a.out1[v - a.n0] = (int32_t)r;
  }
}

#define GSEL_ONE_LEN 131072
// One workgroup per vector, or the many-workgroup descent: the first costs the same for any number of vectors the chip holds at
// once, the second grows with them.  us, one launch / ten: 2 vectors 32768 values 26 / 35, 65001 43 / 36; 8 vectors 65001 43 /
// 40; 28 vectors 65001 43 / 52, 131072 79 / 58; 64 vectors 131072 79 / 84.
static bool cover_one_launch(int64_t len, int n_vec) {
  return len <= GSEL_ONE_LEN && len <= 49152 + 1280 * (int64_t)n_vec;
}
__global__ __launch_bounds__(CS_THREADS) void sp_cover_count_kernel(CoverCountArgs a) {
  __shared__ __attribute__((aligned(16))) CoverShared sh;
  cover_count_vector(sh, a, blockIdx.x);
}

// lower triangle of an [nb][nb] map (score_cover_idx), nb <= NB: 128 or GSEL_ONE_NB
#define GSEL_ONE_NB 256
template <int NB>
__device__ static __forceinline__ void cover_select_map(CoverShared& sh, uint32_t* row_ties /* LDS [GSEL_ONE_NB] */,
                                                        const float* __restrict__ xv,
                                                        int nb, int nbw, long long t_le, uint64_t* __restrict__ mv) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int WAVES = CS_THREADS / SP_WAVE;
  GselState s = sel_fresh_state(t_le, true);
  if (s.enabled) {
    // Rows p and nb - 1 - p of the triangle together have nb + 1 entries: entry j of pair p.  A wave takes pairs wave,
    // wave + 16, ..., 64 entries at a time, so that hardly any lane idles above the diagonal.  All of a thread's entries are
    // read once, in one go, and stay in registers for the four levels (256 x 256 blocks, one map: read again in each level,
    // eight at a time, and the mask written word by word 68 us, so 40; ten launches of the other descent 42).
    constexpr int CHUNKS = NB / SP_WAVE + 1, ITEMS = NB / 2 / WAVES * CHUNKS;  // of up to NB + 1 entries
    const int pairs = (nb + 1) / 2;
    float val[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int p = wave + WAVES * (i / CHUNKS), j = SP_WAVE * (i % CHUNKS) + lane, r = nb - 1 - p;
      const bool low = j <= p;
      const int row = low ? p : r, col = low ? j : j - p - 1;
      val[i] = p < pairs && (low || (j <= nb && r != p)) ? xv[row * nb + col] : 0.f;  // (zeros are left out of the histograms)
    }
    cover_descent(sh, s, [&](auto&& f) {
#pragma unroll
      for (int i = 0; i < ITEMS; ++i)
        if (wave + WAVES * (i / CHUNKS) < pairs && SP_WAVE * (i % CHUNKS) <= nb) f(val[i]);  // (uniform)
    });
  }
  // the boundary group of equal values is taken partially: its n_take lowest indices (row-major) win
  const bool ranked = s.enabled && !s.all && s.n_take != 0 && s.n_take < s.n_equal;
  const bool take_all_equal = s.all || s.n_take >= s.n_equal;
  if (ranked) {
    for (int r = wave; r < nb; r += WAVES) {
      uint32_t cnt = 0;
      for (int c0 = 0; c0 <= r; c0 += SP_WAVE) {
        const int c = c0 + lane;
        cnt += __popcll(__ballot(c <= r && sp_sort_key(xv[(int64_t)r * nb + c]) == s.prefix));
      }
      if (lane == 0) row_ties[r] = cnt;
    }
    __syncthreads();
  }
  constexpr int WORDS = NB / SP_WAVE, ROWS = 4;  // rows of a wave at a time: their entries and mask words are read in one go
  uint32_t before_rows = 0;  // members of the boundary group in the rows in front of row `counted` (uniform per wave)
  int counted = 0;
  for (int r0 = wave; r0 < nb; r0 += WAVES * ROWS) {
    float x[ROWS][WORDS];
    uint64_t old[ROWS];  // lane u: word u of the row
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int r = r0 + i * WAVES;
#pragma unroll
      for (int u = 0; u < WORDS; ++u) {
        const int c = u * SP_WAVE + lane;
        x[i][u] = s.enabled && r < nb && c <= r ? xv[r * nb + c] : 0.f;
      }
      old[i] = r < nb && lane < WORDS && lane * SP_WAVE <= r ? mv[r * nbw + lane] : 0ull;
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int r = r0 + i * WAVES;
      if (r >= nb) break;  // (uniform)
      if (ranked)
        for (; counted < r; ++counted) before_rows += row_ties[counted];
      uint32_t before = before_rows;
      uint64_t mine = 0;  // lane u: what word u of the row gains
#pragma unroll
      for (int u = 0; u < WORDS; ++u) {
        if (u * SP_WAVE > r) break;  // (uniform)
        const bool in = s.enabled && u * SP_WAVE + lane <= r;
        const uint32_t key = sp_sort_key(x[i][u]);
        const bool eq = in && key == s.prefix;
        bool sel = in && (s.all || key > s.prefix || (eq && take_all_equal));
        if (ranked) {
          const unsigned long long eqb = __ballot(eq);
          if (eq && before + (uint32_t)__popcll(eqb & ((1ull << lane) - 1ull)) < s.n_take) sel = true;
          before += (uint32_t)__popcll(eqb);
        }
        unsigned long long bal = __ballot(sel);
        if (r == 0 && u == 0) bal |= 1ull;  // block (0,0): the padding id of the reference
        if (lane == u) mine = bal;
      }
      // this wave alone writes the words of its rows (the kernels that wrote the mask before have finished)
      if (mine) mv[r * nbw + lane] = old[i] | mine;
    }
  }
}

template <int NB>
__global__ __launch_bounds__(CS_THREADS) void sp_cover_select_kernel(const float* __restrict__ x,
                                                                      const int32_t* __restrict__ enable,
                                                                      int enable_match, int nb, int nbw, long long t_le,
                                                                      uint64_t* __restrict__ mask) {
  __shared__ __attribute__((aligned(16))) CoverShared sh;
  __shared__ uint32_t row_ties[GSEL_ONE_NB];
  const int v = blockIdx.x;
  if (!gsel_enabled(enable, enable_match, v)) return;
  cover_select_map<NB>(sh, row_ties, x + (int64_t)v * nb * nb, nb, nbw, t_le, mask + (int64_t)v * nb * nbw);
}

__global__ __launch_bounds__(GSEL_THREADS) void sp_gsel_emit_kernel(const float* __restrict__ x, int nb, int nbw,
                                                                    const GselState* __restrict__ st,
                                                                    uint64_t* __restrict__ mask) {
  const int v = blockIdx.y;
  const GselState s = st[v];
  if (!s.enabled) return;
  const bool take_all_equal = s.all || s.n_take >= s.n_equal;
  const float* xv = x + (int64_t)v * nb * nb;
  uint64_t* mv = mask + (int64_t)v * nb * nbw;
  for (int r = blockIdx.x; r < nb; r += GSEL_SPLIT) {
    const float* row = xv + (int64_t)r * nb;
    for (int c0 = 0; c0 <= r; c0 += GSEL_THREADS) {  // uniform trip count per workgroup: every lane votes
      const int c = c0 + threadIdx.x;
      bool sel = false;
      if (c <= r) {
        const uint32_t key = sp_sort_key(row[c]);
        sel = s.all || key > s.prefix || (key == s.prefix && take_all_equal);
      }
      const unsigned long long bal = __ballot(sel);
      if ((threadIdx.x & 63) == 0 && bal)
        atomicOr(reinterpret_cast<unsigned long long*>(mv) + (int64_t)r * nbw + (c >> 6), bal);
    }
  }
}

// Boundary group taken partially: the n_take lowest indices (row-major) of the equal-valued entries win.  The
// rows are cut into GSEL_SPLIT contiguous segments: a first kernel counts each segment's members of the group, the
// second gives every segment the count of the segments before it and ranks inside the segment only.
__device__ static inline void gsel_segment(int nb, int seg, int& r_lo, int& r_hi) {
  const int per = (nb + GSEL_SPLIT - 1) / GSEL_SPLIT;
  r_lo = seg * per < nb ? seg * per : nb;
  r_hi = r_lo + per < nb ? r_lo + per : nb;
}

__device__ static inline bool gsel_ranked_needed(const GselState& s) {
  return s.enabled && !s.all && s.n_take != 0 && s.n_take < s.n_equal;
}

__global__ __launch_bounds__(GSEL_THREADS) void sp_gsel_tie_count_kernel(const float* __restrict__ x, int nb,
                                                                         const GselState* __restrict__ st,
                                                                         uint32_t* __restrict__ tie_cnt) {
  __shared__ uint32_t total;
  const int v = blockIdx.y, seg = blockIdx.x;
  const GselState s = st[v];
  if (!gsel_ranked_needed(s)) return;
  if (threadIdx.x == 0) total = 0;
  __syncthreads();
  int r_lo, r_hi;
  gsel_segment(nb, seg, r_lo, r_hi);
  const float* xv = x + (int64_t)v * nb * nb;
  uint32_t mine = 0;
  for (int r = r_lo; r < r_hi; ++r)
    for (int c = threadIdx.x; c <= r; c += GSEL_THREADS) mine += sp_sort_key(xv[(int64_t)r * nb + c]) == s.prefix;
  if (mine) atomicAdd(&total, mine);
  __syncthreads();
  if (threadIdx.x == 0) tie_cnt[(int64_t)v * SEL_BINS + seg] = total;
}

__global__ __launch_bounds__(GSEL_THREADS) void sp_gsel_emit_ranked_kernel(const float* __restrict__ x, int nb, int nbw,
                                                                           const GselState* __restrict__ st,
                                                                           const uint32_t* __restrict__ tie_cnt,
                                                                           uint64_t* __restrict__ mask) {
  __shared__ uint32_t wave_cnt[GSEL_THREADS / SP_WAVE];
  const int v = blockIdx.y, seg = blockIdx.x;
  const GselState s = st[v];
  if (!gsel_ranked_needed(s)) return;
  uint32_t running = 0;  // members of the group in front of the current chunk (uniform)
  for (int i = 0; i < seg; ++i) running += tie_cnt[(int64_t)v * SEL_BINS + i];
  if (running >= s.n_take) return;
  int r_lo, r_hi;
  gsel_segment(nb, seg, r_lo, r_hi);
  const float* xv = x + (int64_t)v * nb * nb;
  uint32_t* mv = reinterpret_cast<uint32_t*>(mask + (int64_t)v * nb * nbw);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int r = r_lo; r < r_hi; ++r) {
    for (int c0 = 0; c0 <= r; c0 += GSEL_THREADS) {  // uniform trip count: every lane votes
      const int c = c0 + threadIdx.x;
      const bool eq = c <= r && sp_sort_key(xv[(int64_t)r * nb + c]) == s.prefix;
      const unsigned long long bal = __ballot(eq);
      const uint32_t before = __popcll(bal & ((1ull << lane) - 1ull));
      __syncthreads();  // the previous chunk's counts have been read
      if (lane == 0) wave_cnt[wave] = __popcll(bal);
      __syncthreads();
      uint32_t off = running, tot = 0;
#pragma unroll
      for (int w = 0; w < GSEL_THREADS / SP_WAVE; ++w) {
        if (w < wave) off += wave_cnt[w];
        tot += wave_cnt[w];
      }
      if (eq && off + before < s.n_take)
        atomicOr(&mv[((int64_t)r * nbw + (c >> 6)) * 2 + ((c >> 5) & 1)], 1u << (c & 31));
      running += tot;
      if (running >= s.n_take) return;  // uniform
    }
  }
}

// ---- score_cover_topk (attn/utils.py:47-50) on flat vectors: the same descent, the count instead of the set ----
// (its own launch shape: a flat vector is cut into FLAT_SPLIT strided shares of FLAT_THREADS-wide rows; few fat workgroups,
// all resident at once, instead of 64 x 256 threads: every workgroup pays for clearing and flushing 2048 bins)
#define FLAT_SPLIT 16
#define FLAT_THREADS 1024
template <int LEVEL>
__global__ __launch_bounds__(FLAT_THREADS) void sp_gsel_hist_flat_kernel(const float* __restrict__ x0,
                                                                         const float* __restrict__ x1, int n0,
                                                                         int64_t len,
                                                                         const GselState* __restrict__ st,
                                                                         uint32_t* __restrict__ gcnt,
                                                                         unsigned long long* __restrict__ gsum) {
  __shared__ unsigned long long lsum[SEL_BINS];
  __shared__ uint32_t lcnt[SEL_BINS];
  const int v = blockIdx.y;
  const GselState s = st[v];
  if (!s.enabled || s.all) return;
  constexpr int shift = LEVEL == 0 ? 21 : (LEVEL == 1 ? 10 : 0);
  constexpr int width = LEVEL == 2 ? 10 : 11;
  constexpr int pshift = LEVEL == 0 ? 32 : (LEVEL == 1 ? 21 : 10);
  for (int i = threadIdx.x; i < SEL_BINS; i += FLAT_THREADS) {
    lsum[i] = 0;
    lcnt[i] = 0;
  }
  __syncthreads();
  const float* xv = v < n0 ? x0 + (int64_t)v * len : x1 + (int64_t)(v - n0) * len;  // vectors n0.. live in x1
  for (int64_t i0 = (int64_t)blockIdx.x * FLAT_THREADS; i0 < len; i0 += (int64_t)FLAT_SPLIT * FLAT_THREADS) {
    const int64_t i = i0 + threadIdx.x;
    bool live = i < len;
    uint32_t b = 0;
    unsigned long long fx = 0;
    if (live) {
      const float val = xv[i];
      const uint32_t key = sp_sort_key(val);
      live = !(pshift < 32 && (key >> (pshift & 31)) != s.prefix);
      b = (key >> shift) & ((1u << width) - 1u);
      fx = sp_to_fixed(val);
    }
    if (live) {
      atomicAdd(&lcnt[b], 1u);
      if (fx) atomicAdd(&lsum[b], fx);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < (1 << width); i += FLAT_THREADS) {
    if (lcnt[i]) atomicAdd(&gcnt[(int64_t)v * SEL_BINS + i], lcnt[i]);
    if (lsum[i]) atomicAdd(&gsum[(int64_t)v * SEL_BINS + i], lsum[i]);
  }
}

__global__ void sp_gsel_count_kernel(const GselState* __restrict__ st, int n_vec, long long t_le, int64_t len,
                                     int32_t* __restrict__ out0, int32_t* __restrict__ out1, int n0, int bs,
                                     int minb, int maxb) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n_vec) return;
  const GselState s = st[v];
  long long m = 0;
  if (t_le >= 0) m = s.all ? (long long)len : (long long)s.above + s.n_take;
  long long r = m + 1;
  if (bs > 0) {  // budgets: tokens // bs + 1, clamped (attention_sharing.py:169-176)
    r = r / bs + 1;
    if (r < minb) r = minb;
    if (r > maxb) r = maxb;
  }
  if (v < n0)
    out0[v] = (int32_t)r;
  else
    out1[v - n0] = (int32_t)r;
}

static int gsel_count_run(const float* x0, const float* x1, int n0, int n_vec, int64_t len, float thr, int32_t* out0,
                          int32_t* out1, int bs, int minb, int maxb, void* workspace, size_t workspace_bytes,
                          hipStream_t s, const char* who);

extern "C" size_t sp_cover_select_workspace_bytes(int32_t n_vec) {
  if (n_vec <= 0) return 0;
  return (size_t)n_vec * (sizeof(GselState) + SEL_BINS * (sizeof(uint32_t) + sizeof(unsigned long long)));
}

static int gsel_run(const float* x, const int32_t* enable, int enable_match, int n_vec, int nb, float score,
                    uint64_t* mask, void* workspace, size_t workspace_bytes, hipStream_t s, const char* who) {
  SP_REQUIRE(workspace && workspace_bytes >= sp_cover_select_workspace_bytes(n_vec) && ((uintptr_t)workspace % 8) == 0,
             SP_ERR_WORKSPACE, "%s: workspace missing, misaligned or too small", who);
  const int nbw = (nb + 63) / 64;
  if (nb <= GSEL_ONE_NB) {  // one workgroup per map does the whole descent and writes the bits
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(n_vec), dim3(CS_THREADS), 0, s, x, enable, enable_match, nb, nbw,
                         (long long)sp_thr_le(score), mask);
    };
    nb <= 128 ? launch(sp_cover_select_kernel<128>) : launch(sp_cover_select_kernel<GSEL_ONE_NB>);
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  GselState* st = reinterpret_cast<GselState*>(workspace);
  unsigned long long* gsum = reinterpret_cast<unsigned long long*>(st + n_vec);
  uint32_t* gcnt = reinterpret_cast<uint32_t*>(gsum + (size_t)n_vec * SEL_BINS);
  hipLaunchKernelGGL(sp_gsel_init_kernel, dim3(n_vec), dim3(256), 0, s, st, gcnt, gsum, enable, enable_match, n_vec,
                     (long long)sp_thr_le(score), mask, nb, nbw);
  SP_LAUNCH_CHECK();
  const dim3 hgrid(GSEL_SPLIT, n_vec);
  hipLaunchKernelGGL(sp_gsel_hist_kernel<0>, hgrid, dim3(GSEL_THREADS), 0, s, x, nb, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_pick_kernel<0>, dim3(n_vec), dim3(SEL_THREADS), 0, s, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_hist_kernel<1>, hgrid, dim3(GSEL_THREADS), 0, s, x, nb, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_pick_kernel<1>, dim3(n_vec), dim3(SEL_THREADS), 0, s, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_hist_kernel<2>, hgrid, dim3(GSEL_THREADS), 0, s, x, nb, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_pick_kernel<2>, dim3(n_vec), dim3(SEL_THREADS), 0, s, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_emit_kernel, hgrid, dim3(GSEL_THREADS), 0, s, x, nb, nbw, st, mask);
  // (the histogram counters are free after the last pick: the segments' tie counts go there)
  hipLaunchKernelGGL(sp_gsel_tie_count_kernel, hgrid, dim3(GSEL_THREADS), 0, s, x, nb, st, gcnt);
  hipLaunchKernelGGL(sp_gsel_emit_ranked_kernel, hgrid, dim3(GSEL_THREADS), 0, s, x, nb, nbw, st,
                     (const uint32_t*)gcnt, mask);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// vectors 0..n0-1 are rows of x0 (results to out0), vectors n0..n_vec-1 rows of x1 (results to out1)
static int gsel_count_run(const float* x0, const float* x1, int n0, int n_vec, int64_t len, float thr, int32_t* out0,
                          int32_t* out1, int bs, int minb, int maxb, void* workspace, size_t workspace_bytes,
                          hipStream_t s, const char* who) {
  SP_REQUIRE(workspace && workspace_bytes >= sp_cover_select_workspace_bytes(n_vec) && ((uintptr_t)workspace % 8) == 0,
             SP_ERR_WORKSPACE, "%s: workspace missing, misaligned or too small", who);
  GselState* st = reinterpret_cast<GselState*>(workspace);
  unsigned long long* gsum = reinterpret_cast<unsigned long long*>(st + n_vec);
  uint32_t* gcnt = reinterpret_cast<uint32_t*>(gsum + (size_t)n_vec * SEL_BINS);
  const long long t_le = (long long)sp_thr_le(thr);
  if (cover_one_launch(len, n_vec)) {  // one workgroup per vector, one launch
    const CoverCountArgs a = {x0, x1, n0, (int)len, t_le, out0, out1, bs, minb, maxb};
    hipLaunchKernelGGL(sp_cover_count_kernel, dim3(n_vec), dim3(CS_THREADS), 0, s, a);
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  hipLaunchKernelGGL(sp_gsel_init_kernel, dim3(n_vec), dim3(256), 0, s, st, gcnt, gsum, (const int32_t*)nullptr, -1,
                     n_vec, t_le, (uint64_t*)nullptr, 0, 0);
  SP_LAUNCH_CHECK();
  const dim3 hgrid(FLAT_SPLIT, n_vec);
  hipLaunchKernelGGL(sp_gsel_hist_flat_kernel<0>, hgrid, dim3(FLAT_THREADS), 0, s, x0, x1, n0, len, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_pick_kernel<0>, dim3(n_vec), dim3(SEL_THREADS), 0, s, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_hist_flat_kernel<1>, hgrid, dim3(FLAT_THREADS), 0, s, x0, x1, n0, len, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_pick_kernel<1>, dim3(n_vec), dim3(SEL_THREADS), 0, s, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_hist_flat_kernel<2>, hgrid, dim3(FLAT_THREADS), 0, s, x0, x1, n0, len, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_pick_kernel<2>, dim3(n_vec), dim3(SEL_THREADS), 0, s, st, gcnt, gsum);
  hipLaunchKernelGGL(sp_gsel_count_kernel, dim3((n_vec + 63) / 64), dim3(64), 0, s, st, n_vec, t_le, len, out0, out1, n0,
                     bs, minb, maxb);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_cover_count(const float* x, int32_t n_vec, int64_t len, float thr, int32_t* out, void* workspace,
                              size_t workspace_bytes, sp_stream_t stream) {
  SP_REQUIRE(x && out && n_vec > 0 && len > 0, SP_ERR_INVALID_ARGUMENT, "sp_cover_count: bad arguments");
  return gsel_count_run(x, x, n_vec, n_vec, len, thr, out, out, 0, 0, 0, workspace, workspace_bytes,
                        (hipStream_t)stream, "sp_cover_count");
}

// both vectors of every head in one descent: 2*hq vectors
extern "C" int sp_cover_budgets(const float* vert_tok, const float* slash_tok, int32_t hq, int64_t n, int32_t bs,
                                float pattern_threshold, int32_t min_blocks, int32_t max_blocks, int32_t* nv,
                                int32_t* ns, void* workspace, size_t workspace_bytes, sp_stream_t stream) {
  SP_REQUIRE(vert_tok && slash_tok && nv && ns && hq > 0 && n > 0 && bs > 0, SP_ERR_INVALID_ARGUMENT,
             "sp_cover_budgets: bad arguments");
  return gsel_count_run(vert_tok, slash_tok, hq, 2 * hq, n, pattern_threshold, nv, ns, bs, min_blocks, max_blocks,
                        workspace, workspace_bytes, (hipStream_t)stream, "sp_cover_budgets");
}

extern "C" int sp_cover_select_global(const float* x, const int32_t* enable, int32_t n_vec, int32_t nb, float score,
                                      uint64_t* mask, void* workspace, size_t workspace_bytes, sp_stream_t stream) {
  SP_REQUIRE(x && mask && n_vec > 0 && nb > 0, SP_ERR_INVALID_ARGUMENT, "sp_cover_select_global: bad arguments");
  return gsel_run(x, enable, -1, n_vec, nb, score, mask, workspace, workspace_bytes, (hipStream_t)stream,
                  "sp_cover_select_global");
}

// ------------------------------------------------------------------------------------------------
// score_cover_idx_each_row (attn/utils.py:60-76): sp_rows.h
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(RS_THREADS) void sp_cover_select_rows_kernel(const float* __restrict__ x, int nb, int nbw,
                                                                          long long t_lt,
                                                                          uint64_t* __restrict__ pattern) {
  extern __shared__ __attribute__((aligned(16))) char rs_lds[];
  const RowShared sh = rs_carve<RS_THREADS>(rs_lds, nb);
  const int r = blockIdx.x;
  const int keep = rs_row_keep<RS_THREADS>(x + (int64_t)r * nb, nb, t_lt, sh);
  uint32_t* prow = reinterpret_cast<uint32_t*>(pattern + (int64_t)r * nbw);
  for (int w = threadIdx.x; w < nbw * 2; w += RS_THREADS) {
    uint32_t bits = 0;
    for (int b = 0; b < 32; ++b) {
      const int c = w * 32 + b;
      if (c < nb && c <= r && sh.rank[c] < keep) bits |= 1u << b;
    }
    if (r == 0 && w == 0) bits |= 1u;
    prow[w] = bits;
  }
}

extern "C" int sp_cover_select_rows(const float* x, int32_t nb, float thr, uint64_t* pattern, sp_stream_t stream) {
  SP_REQUIRE(x && pattern && nb > 0, SP_ERR_INVALID_ARGUMENT, "sp_cover_select_rows: bad arguments");
  SP_REQUIRE(nb <= RS_MAX, SP_ERR_UNSUPPORTED, "sp_cover_select_rows: nb=%d exceeds %d", nb, RS_MAX);
  hipLaunchKernelGGL(sp_cover_select_rows_kernel, dim3(nb), dim3(RS_THREADS), rs_lds_bytes(nb), (hipStream_t)stream, x, nb,
                     (nb + 63) / 64, (long long)sp_thr_lt(thr), pattern);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ------------------------------------------------------------------------------------------------
// sqrt Jensen-Shannon divergence (attn/utils.py:26-30), one wave, fixed summation order
// ------------------------------------------------------------------------------------------------
__device__ static float wave_sqrt_js(const float* __restrict__ p, const float* __restrict__ q, int n, int lane) {
  float sp = 0.f, sq = 0.f;
  for (int i = lane; i < n; i += SP_WAVE) {
    const float a = p[i], b = q[i];
    const float m = (a + b) / 2.f;
    sp += a * logf(a / m);
    sq += b * logf(b / m);
  }
  sp = sp_wave_sum(sp);
  sq = sp_wave_sum(sq);
  return sqrtf(0.5f * sp + 0.5f * sq);
}

// ------------------------------------------------------------------------------------------------
// query-aware test (attention_sharing.py:193-202)
// ------------------------------------------------------------------------------------------------
#define QA_THREADS 1024
struct QaArgs {
  const sp_bf16 *q, *kbar;
  const float* vert_blk;
  int64_t n, sq_n, sq_h;
  int hq, hkv, d, bs, nb;
  uint32_t flags;
  float inv_sqrt_d, thr;
  float* avg_qk;
  float* js_qa;
  int32_t* use_qa;
};
static inline size_t qa_lds_bytes(int d, int nb) { return (size_t)(d + (nb > 16 * d ? nb : 16 * d)) * sizeof(float); }

// Head h, by all QA_THREADS threads.  wave_extra(w): what waves 1.. do while wave 0 forms the divergence (no barrier in it).
template <typename Extra>
__device__ static __forceinline__ void queryaware_head(const QaArgs& a, int h, float* qa_lds, Extra&& wave_extra) {
  const sp_bf16 *__restrict__ q = a.q, *__restrict__ kbar = a.kbar;
  const float* __restrict__ vert_blk = a.vert_blk;
  const int64_t n = a.n, sq_n = a.sq_n, sq_h = a.sq_h;
  const int hq = a.hq, hkv = a.hkv, d = a.d, bs = a.bs, nb = a.nb;
  const uint32_t flags = a.flags;
  const float inv_sqrt_d = a.inv_sqrt_d;
  float* qmean = qa_lds;       // [d]
  float* logit = qa_lds + d;   // [nb]
  __shared__ float red[QA_THREADS / SP_WAVE];
  __shared__ float bcast;
  const int kvh = h / (hq / hkv);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // mean over the last bs queries of bf16(q / sqrt(d)), rounded to bf16 (last_q.mean(1), :197-199): thread
  // (row group rg, chunk of 8 channels) sums its rows rg, rg + 16, ..., the 16 partials meet in LDS in a fixed order
  {
    float* part = logit;  // [16][d] partial sums, reused for the logits afterwards (nb >= 1: sized max(nb, 16 d) by the host)
    const int nchunk = d >> 3;
    for (int item = threadIdx.x; item < 16 * nchunk; item += QA_THREADS) {
      const int ch = item % nchunk, rg = item / nchunk;
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int i = rg; i < bs; i += 16) {
        const uint4 raw = *reinterpret_cast<const uint4*>(q + (int64_t)h * sq_h + (n - bs + i) * sq_n + ch * 8);
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[2 * j] += sp_round_bf16(__uint_as_float(w[j] << 16) * inv_sqrt_d);
          acc[2 * j + 1] += sp_round_bf16(__uint_as_float(w[j] & 0xffff0000u) * inv_sqrt_d);
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) part[rg * d + ch * 8 + j] = acc[j];
    }
    __syncthreads();
    for (int c = threadIdx.x; c < d; c += QA_THREADS) {
      float sum = 0.f;
#pragma unroll
      for (int rg = 0; rg < 16; ++rg) sum += part[rg * d + c];
      qmean[c] = sp_round_bf16(sum / (float)bs);
    }
    __syncthreads();
  }
  // logits against the pooled keys: four threads per key (32 channels each), partials folded in a fixed order
  float lmax = -INFINITY;
  const int quarter = threadIdx.x & 3;
  for (int b0 = 0; b0 < nb; b0 += QA_THREADS / 4) {
    const int b = b0 + (threadIdx.x >> 2);
    float sacc = 0.f;
    if (b < nb) {
      const sp_bf16* kr = kbar + ((int64_t)b * hkv + kvh) * d;
      for (int c = quarter * 8; c < d; c += 32) {
        const uint4 raw = *reinterpret_cast<const uint4*>(kr + c);
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          sacc += qmean[c + 2 * j] * __uint_as_float(w[j] << 16);
          sacc += qmean[c + 2 * j + 1] * __uint_as_float(w[j] & 0xffff0000u);
        }
      }
    }
    const float s1 = sacc + __shfl_xor(sacc, 1, SP_WAVE);
    float sfull = s1 + __shfl_xor(s1, 2, SP_WAVE);
    if (b < nb && quarter == 0) {  // (the partial sums that shared `logit` were consumed before the barrier above)
      if (flags & SP_FLAG_LOGITS_BF16) sfull = sp_round_bf16(sfull);
      logit[b] = sfull;
      lmax = fmaxf(lmax, sfull);
    }
  }
  lmax = sp_wave_max(lmax);
  if (lane == 0) red[wave] = lmax;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = red[0];
    for (int w = 1; w < QA_THREADS / SP_WAVE; ++w) m = fmaxf(m, red[w]);
    bcast = m;
  }
  __syncthreads();
  const float gmax = bcast;
  float lsum = 0.f;
  for (int b = threadIdx.x; b < nb; b += QA_THREADS) {
    const float e = expf(logit[b] - gmax);
    logit[b] = e;
    lsum += e;
  }
  lsum = sp_wave_sum(lsum);
  __syncthreads();
  if (lane == 0) red[wave] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int w = 0; w < QA_THREADS / SP_WAVE; ++w) s += red[w];
    bcast = s;
  }
  __syncthreads();
  const float gsum = bcast;
  for (int b = threadIdx.x; b < nb; b += QA_THREADS) {
    const float p = logit[b] / gsum;
    logit[b] = p;
    a.avg_qk[(int64_t)h * nb + b] = p;
  }
  __syncthreads();
  if (wave == 0) {
    const float js = wave_sqrt_js(logit, vert_blk + (int64_t)h * nb, nb, lane);
    if (lane == 0) {
      a.js_qa[h] = js;
      a.use_qa[h] = (js < a.thr) ? 1 : 0;  // NaN compares false
    }
  } else {
    wave_extra(wave);
  }
}

__global__ __launch_bounds__(QA_THREADS) void sp_queryaware_test_kernel(QaArgs a) {
  extern __shared__ float qa_lds[];
  queryaware_head(a, blockIdx.x, qa_lds, [](int) {});
}

static int queryaware_args(QaArgs* a, const void* q, const void* kbar, const float* vert_blk, int64_t n, int32_t hq,
                           int32_t hkv, int32_t d, int64_t q_stride_n, int64_t q_stride_h, int32_t bs, uint32_t flags,
                           float queryaware_threshold, float* avg_qk, float* js_qa, int32_t* use_qa) {
  SP_REQUIRE(q && kbar && vert_blk && avg_qk && js_qa && use_qa, SP_ERR_INVALID_ARGUMENT,
             "sp_queryaware_test_bf16: null pointer");
  SP_REQUIRE(hq > 0 && hkv > 0 && hq % hkv == 0 && d % 8 == 0 && n >= bs && bs > 0, SP_ERR_INVALID_ARGUMENT,
             "sp_queryaware_test_bf16: bad shape");
  const int nb = (int)sp_ceil_div(n, bs);
  SP_REQUIRE(d <= 256, SP_ERR_UNSUPPORTED, "sp_queryaware_test_bf16: head_dim %d too large", d);
  SP_REQUIRE(q_stride_n % 8 == 0 && q_stride_h % 8 == 0 && ((uintptr_t)q % 16) == 0 && ((uintptr_t)kbar % 16) == 0,
             SP_ERR_UNSUPPORTED, "sp_queryaware_test_bf16: q / kbar must be 16-byte aligned with strides multiple of 8");
  SP_REQUIRE(qa_lds_bytes(d, nb) <= 60000, SP_ERR_UNSUPPORTED, "sp_queryaware_test_bf16: nb=%d too large", nb);
  *a = QaArgs{(const sp_bf16*)q, (const sp_bf16*)kbar, vert_blk, n, q_stride_n, q_stride_h, hq, hkv, d, bs, nb, flags,
              sp_inv_sqrt_dim(flags, d), queryaware_threshold, avg_qk, js_qa, use_qa};
  return SP_OK;
}

extern "C" int sp_queryaware_test_bf16(const void* q, const void* kbar, const float* vert_blk, int64_t n, int32_t hq,
                                       int32_t hkv, int32_t d, int64_t q_stride_n, int64_t q_stride_h, int32_t bs,
                                       uint32_t flags, float queryaware_threshold, float* avg_qk, float* js_qa,
                                       int32_t* use_qa, sp_stream_t stream) {
  QaArgs a;
  const int rc = queryaware_args(&a, q, kbar, vert_blk, n, hq, hkv, d, q_stride_n, q_stride_h, bs, flags,
                                 queryaware_threshold, avg_qk, js_qa, use_qa);
  if (rc != SP_OK) return rc;
  hipLaunchKernelGGL(sp_queryaware_test_kernel, dim3(hq), dim3(QA_THREADS), qa_lds_bytes(d, a.nb), (hipStream_t)stream, a);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ------------------------------------------------------------------------------------------------
// top-k sets of the pooled vertical / slash vectors (attention_sharing.py:231-251, :303-329)
// cols[c] = 1 for the nv best columns (column 0 forced), dists[dd] = 1 for the ns best distances
// (distance 0 forced); slash index i holds distance nb-1-i.
// ------------------------------------------------------------------------------------------------
// Membership in the top k of the order (key descending, index ascending), for every element at once, by selection
// instead of ranking: four 8-bit radix passes over the keys find the k-th key T (a 256-bin histogram in LDS and one
// wave that walks it from the top), then an element is in iff key > T, or key == T and fewer than `take` equal keys
// have a lower index (ballots and per-wave counts give that index order).  O(nb) per workgroup where ranking every
// element against every other was O(nb^2 / threads) -- 50 us of a 1024-thread workgroup at nb = 1024.
// Every thread of the workgroup calls it (nthreads = blockDim.x, a multiple of 64); flags[map(i)] = 1 / 0 for i < nb
// with map(i) = reverse ? nb - 1 - i : i.
__device__ static void vs_topk_flags(const uint32_t* keys, int nb, int k, uint8_t* flags, bool reverse, int nthreads) {
  __shared__ uint32_t hist[256];
  __shared__ uint32_t wave_cnt[16];
  __shared__ uint32_t s_prefix, s_take, s_base;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = nthreads >> 6;
  if (k >= nb || k <= 0) {  // (uniform) everything or nothing
    for (int i = threadIdx.x; i < nb; i += nthreads) flags[reverse ? nb - 1 - i : i] = k > 0;
    __syncthreads();
    return;
  }
  if (threadIdx.x == 0) {
    s_prefix = 0u;
    s_take = (uint32_t)k;
  }
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    for (int b = threadIdx.x; b < 256; b += nthreads) hist[b] = 0u;
    __syncthreads();
    const uint32_t prefix = s_prefix;
    for (int i = threadIdx.x; i < nb; i += nthreads) {
      const uint32_t key = keys[i];
      if (pass == 0 || (key >> (shift + 8)) == (prefix >> (shift + 8))) atomicAdd(&hist[(key >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (wave == 0) {  // the bin where the running count from the top reaches the number still to take
      uint32_t c[4], tot = 0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        c[u] = hist[255 - (4 * lane + u)];  // lane 0 holds the four top bins
        tot += c[u];
      }
      uint32_t incl = tot;  // inclusive scan over lanes
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
      }
      uint32_t above = incl - tot;
      const uint32_t take = s_take;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (above < take && above + c[u] >= take) {  // exactly one (lane, u) satisfies this
          s_prefix = prefix | ((uint32_t)(255 - (4 * lane + u)) << shift);
          s_take = take - above;
        }
        above += c[u];
      }
    }
    __syncthreads();
  }
  const uint32_t T = s_prefix, take = s_take;  // take >= 1 keys equal to T belong, lowest indices first
  if (threadIdx.x == 0) s_base = 0u;
  __syncthreads();
  for (int i0 = 0; i0 < nb; i0 += nthreads) {  // (uniform trip count: every lane votes)
    const int i = i0 + threadIdx.x;
    const uint32_t key = i < nb ? keys[i] : 0u;
    const bool eq = i < nb && key == T;
    const unsigned long long bal = __ballot(eq);
    if (lane == 0) wave_cnt[wave] = __popcll(bal);
    __syncthreads();
    uint32_t before = s_base, tot = 0;
    for (int w = 0; w < nwaves; ++w) {
      if (w < wave) before += wave_cnt[w];
      tot += wave_cnt[w];
    }
    before += __popcll(bal & ((1ull << lane) - 1ull));
    if (i < nb) flags[reverse ? nb - 1 - i : i] = key > T || (eq && before < take);
    __syncthreads();  // counts and base have been read
    if (threadIdx.x == 0) s_base += tot;
    __syncthreads();
  }
}

// The same sets by ranking, for both vectors at once: an element is in iff fewer than k come before it in the order.  Four
// lanes share an element's comparisons (16-byte reads that 16 lanes have in common), a wave takes 16 elements at a time: no
// barrier but the one behind the keys, where the radix passes are two dozen of them.  O(nb^2 / threads): up to VS_RANK_NB
// blocks (at 1024 it would be the slower one again).
// Mask launch of a layer: 3001 tokens (24 blocks) 11.0 -> 4.0 us, 8192 with Q pooled beside 23.6 -> 16.4, 32768 (256 blocks)
// 14.0 -> 11.8.
#define VS_RANK_NB 256
__device__ static void vs_rank_sets(const float* __restrict__ vert, const float* __restrict__ slash, int nb, int nv, int ns,
                                    uint32_t* keys /* LDS [2 VS_RANK_NB], 16-byte aligned */, uint8_t* cols, uint8_t* dists,
                                    int nthreads) {
  const uint32_t inf_key = 0x7f800000u;
  for (int i = threadIdx.x; i < 2 * VS_RANK_NB; i += nthreads) {  // (zeros behind the vectors come before nothing)
    const int e = i & (VS_RANK_NB - 1);
    const bool v = i < VS_RANK_NB;
    keys[i] = e >= nb ? 0u : e == (v ? 0 : nb - 1) ? inf_key : sp_sort_key(v ? vert[e] : slash[e]);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, part = lane >> 4;
  const int groups = (nb + 15) / 16;
  for (int gi = wave; gi < 2 * groups; gi += nthreads >> 6) {
    const bool v = gi < groups;  // (uniform)
    const int i = (v ? gi : gi - groups) * 16 + (lane & 15);
    const uint32_t* ks = keys + (v ? 0 : VS_RANK_NB);
    const uint32_t key = ks[i];
    int rank = 0;
    for (int j = 4 * part; j < nb; j += 16) {
      const uint4 o = *reinterpret_cast<const uint4*>(ks + j);
      rank += (o.x > key || (o.x == key && j < i)) + (o.y > key || (o.y == key && j + 1 < i)) +
              (o.z > key || (o.z == key && j + 2 < i)) + (o.w > key || (o.w == key && j + 3 < i));
    }
    rank += __shfl_xor(rank, 16, SP_WAVE);
    rank += __shfl_xor(rank, 32, SP_WAVE);
    if (part == 0 && i < nb) {
      if (v)
        cols[i] = rank < nv;
      else
        dists[nb - 1 - i] = rank < ns;
    }
  }
  __syncthreads();
}

__device__ static void vs_sets(const float* __restrict__ vert, const float* __restrict__ slash, int nb, int nv,
                               int ns, uint32_t* keys /* LDS [RS_MAX], 16-byte aligned */, uint8_t* cols,
                               uint8_t* dists, int nthreads) {
  if (nb <= VS_RANK_NB) {  // (uniform)
    vs_rank_sets(vert, slash, nb, nv, ns, keys, cols, dists, nthreads);
    return;
  }
  const uint32_t inf_key = 0x7f800000u;
  for (int i = threadIdx.x; i < nb; i += nthreads) keys[i] = (i == 0) ? inf_key : sp_sort_key(vert[i]);
  __syncthreads();
  vs_topk_flags(keys, nb, nv, cols, false, nthreads);
  for (int i = threadIdx.x; i < nb; i += nthreads) keys[i] = (i == nb - 1) ? inf_key : sp_sort_key(slash[i]);
  __syncthreads();
  vs_topk_flags(keys, nb, ns, dists, true, nthreads);
}

// ------------------------------------------------------------------------------------------------
// pivot election / share test (attention_sharing.py:204-301): three launches.
//   similarity : one workgroup per head, its sqrt-JS against the cluster's stored pivot (one wave per vector);
//   decide     : one thread per head; the election's ascending order is resolved by looking at the lower heads;
//   keep       : one workgroup per head; the newly elected pivots store their pooled vectors and their own
//                vertical-slash sets.
// ------------------------------------------------------------------------------------------------
#define DEC_THREADS 256
#define DEC_MAX_HEADS 256
// head_cluster[h] names a slot of the state only inside [0, n_clusters); -1 (no shared cluster) and anything a
// caller got wrong must never be used as an index into the slabs

// sqrt-JS of head h's pooled vector (0: vertical, 1: slash) against its cluster's stored pivot (pivots of EARLIER layers
// only: the launch precedes the layer's election); NaN where there is none.  One wave.
__device__ static __forceinline__ float share_similarity(const sp_cluster_state& st, int c, int h, int which,
                                                         const float* __restrict__ blk, int lane) {
  if (!sp_slot_ok(st, c) || st.info[c * 8 + 0] < 0 || st.info[c * 8 + 1] == 0) return NAN;
  return wave_sqrt_js((which == 0 ? st.vert : st.slash) + (int64_t)c * st.nb, blk + (int64_t)h * st.nb, st.nb, lane);
}
__global__ __launch_bounds__(2 * SP_WAVE) void sp_share_similarity_kernel(
    sp_cluster_state st, const int32_t* __restrict__ head_cluster, const float* __restrict__ vert_blk,
    const float* __restrict__ slash_blk, const int32_t* __restrict__ use_qa, float* __restrict__ js_v,
    float* __restrict__ js_s) {
  const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float js = NAN;
  if (!use_qa[h]) js = share_similarity(st, head_cluster[h], h, wave, wave == 0 ? vert_blk : slash_blk, lane);
  if (lane == 0) (wave == 0 ? js_v : js_s)[h] = js;
}

// the cluster's pivot is this head, elected in this layer
__device__ static __forceinline__ bool share_elected(const sp_cluster_state& st, int c, int h, int layer_idx) {
  return sp_slot_ok(st, c) && st.info[c * 8 + 0] == h && st.info[c * 8 + 4] == layer_idx;
}
__device__ static __forceinline__ void share_elect(const sp_cluster_state& st, int c, int h, int layer_idx, int nv, int ns) {
  st.info[c * 8 + 0] = h;
  st.info[c * 8 + 2] = nv;
  st.info[c * 8 + 3] = ns;
  st.info[c * 8 + 4] = layer_idx;
}
__global__ __launch_bounds__(DEC_MAX_HEADS) void sp_share_decide_kernel(
    sp_cluster_state st, const int32_t* __restrict__ head_cluster, int layer_idx, int hq,
    const int32_t* __restrict__ use_qa, const int32_t* __restrict__ nv, const int32_t* __restrict__ ns, int minb,
    float sim_thr, double fb_thr, int32_t* __restrict__ decision, float* __restrict__ js_v,
    float* __restrict__ js_s, int32_t* __restrict__ nv_f, int32_t* __restrict__ ns_f) {
  // The reference walks the heads in ascending order (attention_sharing.py:209-295): the first head of a shared
  // cluster that is not query-aware and finds no pivot becomes the pivot; its later siblings of the same layer find
  // a pivot without a pattern and fall back; heads of clusters with a pattern take the share test.  One thread per
  // head reaches the same decisions: "first" = no lower head of the same cluster is a candidate too.
  __shared__ int s_slot[DEC_MAX_HEADS];
  __shared__ int s_cand[DEC_MAX_HEADS];
  const int h = threadIdx.x;
  int c = -1, qa = 0;
  bool member = false, candidate = false;
  if (h < hq) {
    c = head_cluster[h];
    qa = use_qa[h];
    member = !qa && sp_slot_ok(st, c);
    candidate = member && st.info[c * 8 + 0] < 0;  // the state as the previous layers left it
  }
  s_slot[h] = c;
  s_cand[h] = candidate ? 1 : 0;
  __syncthreads();  // every read of the pivot slots precedes the writes below
  if (h >= hq) return;
  int dec = SP_DEC_VS;
  if (qa) {
    dec = SP_DEC_QA;
    js_v[h] = js_s[h] = NAN;  // (formed beside the query-aware test for every head)
  } else if (candidate) {
    bool first = true;
    for (int h2 = 0; h2 < h; ++h2) first = first && !(s_cand[h2] && s_slot[h2] == c);
    if (first) {
      share_elect(st, c, h, layer_idx, nv[h], ns[h]);
      dec = SP_DEC_DENSE;
    }
  } else if (member && st.info[c * 8 + 1] != 0) {
    if (js_v[h] < sim_thr && js_s[h] < sim_thr && st.ratio[c] < fb_thr) dec = SP_DEC_SHARE;
  }
  decision[h] = dec;
  const bool reset = (dec == SP_DEC_QA || dec == SP_DEC_SHARE);
  nv_f[h] = reset ? minb : nv[h];
  ns_f[h] = reset ? minb : ns[h];
}

// a newly elected pivot keeps its pooled vectors and its own
// vertical-slash sets (:223-263); every thread of the workgroup calls it
__device__ static __forceinline__ void share_keep(const sp_cluster_state& st, int c, int h,
                                                  const float* __restrict__ vert_blk, const float* __restrict__ slash_blk,
                                                  int nv, int ns, uint32_t* keys, int nthreads) {
  const int nb = st.nb;
  for (int i = threadIdx.x; i < nb; i += nthreads) {
    st.vert[(int64_t)c * nb + i] = vert_blk[(int64_t)h * nb + i];
    st.slash[(int64_t)c * nb + i] = slash_blk[(int64_t)h * nb + i];
  }
  vs_sets(vert_blk + (int64_t)h * nb, slash_blk + (int64_t)h * nb, nb, nv, ns, keys, st.cols + (int64_t)c * nb,
          st.dists + (int64_t)c * nb, nthreads);
}
__global__ __launch_bounds__(DEC_THREADS) void sp_share_keep_kernel(
    sp_cluster_state st, const int32_t* __restrict__ head_cluster, int layer_idx,
    const float* __restrict__ vert_blk, const float* __restrict__ slash_blk, const int32_t* __restrict__ decision,
    const int32_t* __restrict__ nv, const int32_t* __restrict__ ns) {
  __shared__ __attribute__((aligned(16))) uint32_t s_keys[RS_MAX];
  const int h = blockIdx.x;
  if (decision[h] != SP_DEC_DENSE || !share_elected(st, head_cluster[h], h, layer_idx)) return;  // (uniform)
  share_keep(st, head_cluster[h], h, vert_blk, slash_blk, nv[h], ns[h], s_keys, DEC_THREADS);
}

extern "C" int sp_share_decide(const sp_cluster_state* state, const int32_t* head_cluster, int32_t layer_idx,
                               int32_t hq, const float* vert_blk, const float* slash_blk, const int32_t* use_qa,
                               const int32_t* nv, const int32_t* ns, int32_t min_blocks, float similarity_threshold,
                               double fallback_threshold, int32_t* decision, float* js_v, float* js_s,
                               int32_t* nv_final, int32_t* ns_final, sp_stream_t stream) {
  SP_REQUIRE(state, SP_ERR_INVALID_ARGUMENT, "sp_share_decide: null cluster state");
  int rc = check_state(state, state->nb, "sp_share_decide");
  if (rc) return rc;
  SP_REQUIRE(head_cluster && vert_blk && slash_blk && use_qa && nv && ns && decision && js_v && js_s && nv_final &&
                 ns_final,
             SP_ERR_INVALID_ARGUMENT, "sp_share_decide: null pointer");
  SP_REQUIRE(hq > 0 && hq <= DEC_MAX_HEADS, SP_ERR_UNSUPPORTED, "sp_share_decide: hq=%d unsupported (max %d)", hq,
             DEC_MAX_HEADS);
  SP_REQUIRE(state->nb <= RS_MAX, SP_ERR_UNSUPPORTED, "sp_share_decide: nb=%d exceeds %d", state->nb, RS_MAX);
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(sp_share_similarity_kernel, dim3(hq), dim3(2 * SP_WAVE), 0, s, state_by_value(state), head_cluster, vert_blk,
                     slash_blk, use_qa, js_v, js_s);
  SP_LAUNCH_CHECK();
  hipLaunchKernelGGL(sp_share_decide_kernel, dim3(1), dim3(DEC_MAX_HEADS), 0, s, state_by_value(state), head_cluster, layer_idx, hq, use_qa,
                     nv, ns, min_blocks, similarity_threshold, fallback_threshold, decision, js_v, js_s, nv_final,
                     ns_final);
  SP_LAUNCH_CHECK();
  hipLaunchKernelGGL(sp_share_keep_kernel, dim3(hq), dim3(DEC_THREADS), 0, s, state_by_value(state), head_cluster, layer_idx, vert_blk,
                     slash_blk, decision, nv, ns);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ------------------------------------------------------------------------------------------------
// mask construction (attention_sharing.py:303-337 and attn/utils.py:99-128 as a set)
// ------------------------------------------------------------------------------------------------
#define MASK_THREADS 1024
#define MASK_SPLIT 8  // workgroups per head: each ranks the head's vectors itself and writes a share of the rows
// What the whole-layer selection adds to the mask launch: nothing of it depends on the mask, and each would be a launch of
// its own (2 to 2.7 us of the stream if it had nothing to do).
struct MaskBesides {
  int layer_idx;    // pivots elected in this layer store their vectors and sets
  PoolArgs qpool;   // query-aware heads: the averages of Q's blocks
  float* zero;      // [hq][nb][nb] cleared, or null
  // the decisions themselves, where the launch makes them
  const int32_t *use_qa, *nv, *ns;
  int minb;
  float sim_thr;
  double fb_thr;
  int32_t *decision, *nv_f, *ns_f;
  float *js_v, *js_s;
};
// sp_share_decide_kernel's decision for head h, by every workgroup of the head for itself: "first" only looks at lower heads of its
// cluster that are not query-aware.  The state stays as the previous layers left it until the next launch (share_elect in
// sp_queryaware_small_kernel), so no workgroup can see another's election.  Every thread of the workgroup calls it.  Layers with the
// election as a launch of one workgroup in between / with it here, us: 3001 tokens 110.1 / 107.7, 6177 of 64 channels 122.3 / 120.0,
// 10007 258.4 / 255.5.
__device__ static __forceinline__ int mask_decide(const sp_cluster_state& st, const int32_t* __restrict__ head_cluster, int h,
                                                  const MaskBesides& a) {
  const int t = threadIdx.x, c = head_cluster[h], qa = a.use_qa[h];
  const int tc = t < h ? head_cluster[t] : 0, tqa = t < h ? a.use_qa[t] : 1;
  const float js_v = a.js_v[h], js_s = a.js_s[h];
  if (qa) return SP_DEC_QA;
  if (!sp_slot_ok(st, c)) return SP_DEC_VS;
  const int pivot = st.info[c * 8 + 0], pattern = st.info[c * 8 + 1];
  if (pivot < 0) return __syncthreads_or(t < h && tc == c && !tqa) ? SP_DEC_VS : SP_DEC_DENSE;
  return pattern != 0 && js_v < a.sim_thr && js_s < a.sim_thr && st.ratio[c] < a.fb_thr ? SP_DEC_SHARE : SP_DEC_VS;
}
// q blocks of one query-aware head, share `part_no` of MASK_SPLIT: a chunk of 8 channels by four waves, 64 / (d / 8) blocks
// at a time for each four waves
__device__ static void mask_pool_q(const PoolArgs& a, int h, int nb, int part_no, char* lds) {
  const int t = threadIdx.x % POOL_THREADS, set = threadIdx.x / POOL_THREADS;
  const int lane = t % POOL_CHUNKS, sub = t / POOL_CHUNKS, dchunks = a.d / 8;
  float(*part)[POOL_CHUNKS][8] = reinterpret_cast<float(*)[POOL_CHUNKS][8]>(lds) + set * POOL_SPLIT;
  const int at_once = POOL_CHUNKS / dchunks, d0 = lane % dchunks * 8;  // (lanes beyond at_once * dchunks idle)
  const int per = (nb + MASK_SPLIT - 1) / MASK_SPLIT, b_end = min(nb, (part_no + 1) * per);
  for (int b0 = part_no * per; b0 < b_end; b0 += at_once * (MASK_THREADS / POOL_THREADS)) {
    const int blk = b0 + set * at_once + lane / dchunks;
    const bool active = lane / dchunks < at_once && blk < b_end;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (active) pool_quarter<SP_POOL_AVG>(a.x + (int64_t)h * a.sx_h + d0, a.sx_n, (int64_t)blk * a.bs, a.n, a.bs, sub, acc);
    __syncthreads();  // the previous round's partial sums have been read
#pragma unroll
    for (int j = 0; j < 8; ++j) part[sub][lane][j] = acc[j];
    __syncthreads();
    if (sub == 0 && active) {
      const int64_t rem = a.n - (int64_t)blk * a.bs;
      pool_store<SP_POOL_AVG>(part, lane, rem < a.bs ? (int)rem : a.bs, a.bs, a.tail_mode, a.y + ((int64_t)blk * a.h + h) * a.d + d0);
    }
  }
}

// BESIDES: grid (hq, 2 MASK_SPLIT), the second half of which pools and clears.  DECIDE (up to 128 blocks): the launch makes the
// decisions too.
template <bool BESIDES, bool DECIDE>
__global__ __launch_bounds__(MASK_THREADS) void sp_build_mask_kernel(
    sp_cluster_state st, const int32_t* __restrict__ head_cluster, const int32_t* __restrict__ decision,
    const float* __restrict__ vert_blk, const float* __restrict__ slash_blk, const int32_t* __restrict__ nv_f,
    const int32_t* __restrict__ ns_f, int nb, int nbw, uint64_t* __restrict__ mask, MaskBesides extra) {
  __shared__ __attribute__((aligned(16))) uint32_t s_keys[BESIDES ? MASK_THREADS * 8 : RS_MAX];
  __shared__ uint8_t s_cols[RS_MAX], s_dists[RS_MAX];
  const int h = blockIdx.x;
  const bool pools = BESIDES && blockIdx.y >= MASK_SPLIT;
  int dec, n_v = 0, n_s = 0;
  if constexpr (DECIDE) {
    static_assert(BESIDES && MASK_THREADS >= DEC_MAX_HEADS, "");
    dec = pools ? (extra.use_qa[h] ? SP_DEC_QA : SP_DEC_VS) : mask_decide(st, head_cluster, h, extra);
    if (!pools) {
      const bool reset = dec == SP_DEC_QA || dec == SP_DEC_SHARE;
      n_v = reset ? extra.minb : extra.nv[h];
      n_s = reset ? extra.minb : extra.ns[h];
      if (blockIdx.y == 0 && threadIdx.x == 0) {
        extra.decision[h] = dec;
        extra.nv_f[h] = n_v;
        extra.ns_f[h] = n_s;
        if (dec == SP_DEC_QA) extra.js_v[h] = extra.js_s[h] = NAN;  // (formed beside the query-aware test for every head)
      }
    }
  } else {
    dec = decision[h];
    if (!pools) n_v = nv_f[h], n_s = ns_f[h];
  }
  if constexpr (BESIDES) {
    static_assert(MASK_THREADS * 8 >= RS_MAX, "");
    if (pools) {
      const int part_no = blockIdx.y - MASK_SPLIT;
      if (extra.zero != nullptr) {  // (in shares of the whole array: a head's part is 4-byte aligned only)
        const int64_t all = (int64_t)gridDim.x * nb * nb, shares = (int64_t)gridDim.x * MASK_SPLIT;
        const int64_t per = (all / 4 + shares - 1) / shares, i0 = ((int64_t)h * MASK_SPLIT + part_no) * per;
        const int64_t i1 = min(all / 4, i0 + per);
        float4* z = reinterpret_cast<float4*>(extra.zero);
        for (int64_t i = i0 + threadIdx.x; i < i1; i += MASK_THREADS) z[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (h == 0 && part_no == 0 && threadIdx.x < (all & 3)) extra.zero[(all & ~3ll) + threadIdx.x] = 0.f;
      }
      if (dec == SP_DEC_QA) mask_pool_q(extra.qpool, h, nb, part_no, reinterpret_cast<char*>(s_keys));
      return;
    }
    if (dec == SP_DEC_DENSE && blockIdx.y == 0 && (DECIDE || share_elected(st, head_cluster[h], h, extra.layer_idx)))
      share_keep(st, head_cluster[h], h, vert_blk, slash_blk, n_v, n_s, s_keys, MASK_THREADS);  // (nothing here reads what it writes)
  }
  if (dec != SP_DEC_DENSE)
    vs_sets(vert_blk + (int64_t)h * nb, slash_blk + (int64_t)h * nb, nb, n_v, n_s, s_keys, s_cols, s_dists,
            MASK_THREADS);
  const uint64_t* pat = nullptr;
  // a SHARE decision without a valid slot (only a caller's own decision vector can hold one) adds no pattern
  if (dec == SP_DEC_SHARE && sp_slot_ok(st, head_cluster[h])) pat = st.pattern + (int64_t)head_cluster[h] * nb * nbw;
  uint64_t* mh = mask + (int64_t)h * nb * nbw;
  // Both sets as bit strings: colw = the columns, dstw = the distances in the order of the slash index i = nb - 1 - d.
  // Row r, columns c0 .. c0 + 63 then want distance bits i = nb - 1 - r + c0 .. + 63: a 64-bit window of dstw, so a mask
  // word is two shifts and an OR instead of 64 pairs of byte look-ups.
  __shared__ uint64_t colw[RS_MAX / 64], dstw[RS_MAX / 64 + 1];
  if (dec != SP_DEC_DENSE) {
    const int lane = threadIdx.x & 63;
    for (int i0 = 0; i0 < nbw * 64; i0 += MASK_THREADS) {  // (uniform trip count: every lane votes)
      const int i = i0 + threadIdx.x;
      const unsigned long long cb = __ballot(i < nb && s_cols[i] != 0);
      const unsigned long long db = __ballot(i < nb && s_dists[nb - 1 - i] != 0);
      if (lane == 0 && i < nbw * 64) {
        colw[i >> 6] = cb;
        dstw[i >> 6] = db;
      }
    }
    if (threadIdx.x == 0) dstw[nbw] = 0ull;
    __syncthreads();
  }
  const int rows_per = (nb + MASK_SPLIT - 1) / MASK_SPLIT;
  const int r_begin = blockIdx.y * rows_per, r_end = min(nb, r_begin + rows_per);
  for (int idx = r_begin * nbw + threadIdx.x; idx < r_end * nbw; idx += MASK_THREADS) {
    const int r = idx / nbw, w = idx - r * nbw;
    const int c0 = w * 64;
    const int cend = min(c0 + 64, r + 1);
    // the causal part of the word: columns c0 .. cend - 1
    const uint64_t causal = cend <= c0 ? 0ull : ((cend - c0 == 64) ? ~0ull : ((1ull << (cend - c0)) - 1ull));
    uint64_t bits = causal;
    if (dec != SP_DEC_DENSE) {
      bits = 0ull;
      if (causal) {
        const int start = nb - 1 - r + c0;  // >= 0; bits past nb - 1 belong to columns beyond r
        const int k = start >> 6, sh = start & 63;
        uint64_t win = dstw[k] >> sh;
        if (sh) win |= dstw[k + 1] << (64 - sh);
        bits = (colw[w] | win) & causal;
      }
      if (pat) bits |= pat[idx];
    }
    if (idx == 0) bits |= 1ull;
    mh[idx] = bits;
  }
}

extern "C" int sp_build_mask(const sp_cluster_state* state, const int32_t* head_cluster, const int32_t* decision,
                             const float* vert_blk, const float* slash_blk, const int32_t* nv_final,
                             const int32_t* ns_final, int32_t hq, int32_t nb, uint64_t* mask, sp_stream_t stream) {
  int rc = check_state(state, nb, "sp_build_mask");
  if (rc) return rc;
  SP_REQUIRE(head_cluster && decision && vert_blk && slash_blk && nv_final && ns_final && mask,
             SP_ERR_INVALID_ARGUMENT, "sp_build_mask: null pointer");
  SP_REQUIRE(hq > 0 && nb > 0 && nb <= RS_MAX, SP_ERR_UNSUPPORTED, "sp_build_mask: nb=%d unsupported (max %d)", nb,
             RS_MAX);
  hipLaunchKernelGGL((sp_build_mask_kernel<false, false>), dim3(hq, MASK_SPLIT), dim3(MASK_THREADS), 0, (hipStream_t)stream,
                     state_by_value(state), head_cluster, decision, vert_blk, slash_blk, nv_final, ns_final, nb, (nb + 63) / 64, mask,
                     MaskBesides{});
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ------------------------------------------------------------------------------------------------
// query-aware heads: pooled block probabilities (attention_sharing.py:350-360)
// ------------------------------------------------------------------------------------------------
#define BP_THREADS 256
__global__ __launch_bounds__(BP_THREADS) void sp_block_probs_kernel(
    const sp_bf16* __restrict__ qbar, const sp_bf16* __restrict__ kbar, const int32_t* __restrict__ decision, int hq,
    int hkv, int d, int nb, uint32_t flags, float inv_sqrt_d, float* __restrict__ probs) {
  extern __shared__ float bp_lds[];
  float* qs = bp_lds;          // [d]
  float* logit = bp_lds + d;   // [nb]
  __shared__ float red[BP_THREADS / SP_WAVE];
  __shared__ float bcast;
  const int r = blockIdx.x, h = blockIdx.y;
  if (decision[h] != SP_DEC_QA) return;
  const int kvh = h / (hq / hkv);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int c = threadIdx.x; c < d; c += BP_THREADS)
    qs[c] = sp_round_bf16(sp_bf16_to_f32(qbar[((int64_t)r * hq + h) * d + c]) * inv_sqrt_d);
  __syncthreads();
  float lmax = -INFINITY;
  for (int b = threadIdx.x; b <= r; b += BP_THREADS) {
    const sp_bf16* kr = kbar + ((int64_t)b * hkv + kvh) * d;
    float s = 0.f;
    for (int c = 0; c < d; c += 8) {
      const uint4 raw = *reinterpret_cast<const uint4*>(kr + c);
      const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s += qs[c + 2 * j] * __uint_as_float(w[j] << 16);
        s += qs[c + 2 * j + 1] * __uint_as_float(w[j] & 0xffff0000u);
      }
    }
    if (flags & SP_FLAG_LOGITS_BF16) s = sp_round_bf16(s);
    logit[b] = s;
    lmax = fmaxf(lmax, s);
  }
  lmax = sp_wave_max(lmax);
  if (lane == 0) red[wave] = lmax;
  __syncthreads();
  if (threadIdx.x == 0) {
    float m = red[0];
    for (int w = 1; w < BP_THREADS / SP_WAVE; ++w) m = fmaxf(m, red[w]);
    bcast = m;
  }
  __syncthreads();
  const float gmax = bcast;
  float lsum = 0.f;
  for (int b = threadIdx.x; b <= r; b += BP_THREADS) {
    const float e = expf(logit[b] - gmax);
    logit[b] = e;
    lsum += e;
  }
  lsum = sp_wave_sum(lsum);
  __syncthreads();
  if (lane == 0) red[wave] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int w = 0; w < BP_THREADS / SP_WAVE; ++w) s += red[w];
    bcast = s;
  }
  __syncthreads();
  const float gsum = bcast;
  float* out = probs + ((int64_t)h * nb + r) * nb;
  for (int b = threadIdx.x; b < nb; b += BP_THREADS) out[b] = (b <= r) ? logit[b] / gsum : 0.f;
}

// Up to 128 blocks (16384 tokens at block size 128) a head's map is one row tile of bpm_rows, and the head's probabilities and
// its selection are one workgroup and one launch: the map is read back by the workgroup that wrote it.  Beyond, a head's
// row tiles are workgroups of a launch of their own.  Bound by latency (one K tile, two passes over it, the descent's
// barriers) and, in layers without a query-aware head, by being a launch at all: against two launches a layer without one takes
// 2 us less (3001 tokens, 6177 of 64 channels, 10007 of 28 / 4 heads), one with all 32 heads query-aware 3 us (8192 tokens).
struct ElectArgs {  // pivots that the mask launch has decided on and the state does not know yet (st.info null: none)
  sp_cluster_state st;
  const int32_t *head_cluster, *nv, *ns;
  int layer_idx;
};
template <int D>
__global__ __launch_bounds__(CS_THREADS) void sp_queryaware_small_kernel(const sp_bf16* qbar, const sp_bf16* kbar,
                                                                         const int32_t* __restrict__ decision, int hq, int hkv,
                                                                         int nb, int nbw, uint32_t flags, float inv_sqrt_d,
                                                                         float* probs, long long t_le, uint64_t* mask,
                                                                         ElectArgs elect) {
  __shared__ union {
    BpmLds<D> rows;
    struct {
      __attribute__((aligned(16))) CoverShared cover;
      uint32_t row_ties[GSEL_ONE_NB];
    } sel;
  } lds;
  static_assert(CS_THREADS % BPM_THREADS == 0 && LQ_TILE <= GSEL_ONE_NB, "");
  const int h = blockIdx.x, dec = decision[h];
  if (dec == SP_DEC_DENSE && elect.st.info != nullptr && threadIdx.x == 0)
    share_elect(elect.st, elect.head_cluster[h], h, elect.layer_idx, elect.nv[h], elect.ns[h]);
  if (dec != SP_DEC_QA) return;
  bpm_rows<D, CS_THREADS / BPM_THREADS>(lds.rows, qbar, kbar, 0, h, hq, hkv, nb, flags, inv_sqrt_d, probs);
  __syncthreads();  // the map is written, the tile's LDS is free
  cover_select_map<LQ_TILE>(lds.sel.cover, lds.sel.row_ties, probs + (int64_t)h * nb * nb, nb, nbw, t_le, mask + (int64_t)h * nb * nbw);
}

// score = pattern_threshold * nb: the product of the caller's DOUBLE threshold and the block count, evaluated in
// double as Python evaluates it (attention_sharing.py:361), then taken to fp32 as the comparison with an fp32
// tensor takes it (utils.py:56).  A threshold that had been rounded to fp32 first would give a score one fp32 ulp
// away for about a fifth of the block counts.
extern "C" float sp_queryaware_select_score(double pattern_threshold, int32_t nb) {
  volatile double product = pattern_threshold * (double)nb;  // one rounding to double, then one to float
  return (float)product;
}

static bool queryaware_small(int32_t d, int32_t nb) { return (d == 128 || d == 64) && nb <= LQ_TILE; }
static int queryaware_small_launch(const void* qbar, const void* kbar, const int32_t* decision, int32_t hq, int32_t hkv, int32_t d,
                                   int32_t nb, uint32_t flags, float score, float* probs, uint64_t* mask, const ElectArgs& elect,
                                   hipStream_t s) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(hq), dim3(CS_THREADS), 0, s, (const sp_bf16*)qbar, (const sp_bf16*)kbar, decision, (int)hq, (int)hkv,
                       (int)nb, (int)((nb + 63) / 64), flags, sp_inv_sqrt_dim(flags, d), probs, (long long)sp_thr_le(score), mask,
                       elect);
  };
  d == 64 ? launch(sp_queryaware_small_kernel<64>) : launch(sp_queryaware_small_kernel<128>);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_queryaware_select_bf16(const void* qbar, const void* kbar, const int32_t* decision, int32_t hq,
                                         int32_t hkv, int32_t d, int32_t nb, uint32_t flags, double pattern_threshold,
                                         float* probs, uint64_t* mask, void* workspace, size_t workspace_bytes,
                                         sp_stream_t stream) {
  SP_REQUIRE(qbar && kbar && decision && probs && mask, SP_ERR_INVALID_ARGUMENT,
             "sp_queryaware_select_bf16: null pointer");
  SP_REQUIRE(hq > 0 && hkv > 0 && hq % hkv == 0 && d % 8 == 0 && nb > 0, SP_ERR_INVALID_ARGUMENT,
             "sp_queryaware_select_bf16: bad shape");
  const size_t lds = (size_t)(d + nb) * sizeof(float);
  SP_REQUIRE(lds <= 60000, SP_ERR_UNSUPPORTED, "sp_queryaware_select_bf16: nb=%d too large", nb);
  const float score = sp_queryaware_select_score(pattern_threshold, nb);
  if (queryaware_small(d, nb)) {
    SP_REQUIRE(workspace && workspace_bytes >= sp_cover_select_workspace_bytes(hq) && ((uintptr_t)workspace % 8) == 0,
               SP_ERR_WORKSPACE, "sp_queryaware_select_bf16: workspace missing, misaligned or too small");  // (unused here)
    return queryaware_small_launch(qbar, kbar, decision, hq, hkv, d, nb, flags, score, probs, mask, ElectArgs{}, (hipStream_t)stream);
  }
  if (d == 128 || d == 64) {  // two passes on the matrix core, 128 rows per workgroup
    const int rc = sp_block_probs_mfma_launch(qbar, kbar, decision, hq, hkv, d, nb, flags, probs, (hipStream_t)stream);
    if (rc != SP_OK) return rc;
  } else {  // one row per workgroup, fp32 dot products
    hipLaunchKernelGGL(sp_block_probs_kernel, dim3(nb, hq), dim3(BP_THREADS), lds, (hipStream_t)stream,
                       (const sp_bf16*)qbar, (const sp_bf16*)kbar, decision, hq, hkv, d, nb, flags,
                       sp_inv_sqrt_dim(flags, d), probs);
    SP_LAUNCH_CHECK();
  }
  return gsel_run(probs, decision, SP_DEC_QA, hq, nb, score, mask, workspace, workspace_bytes, (hipStream_t)stream,
                  "sp_queryaware_select_bf16");
}

// ------------------------------------------------------------------------------------------------
// the selection of one layer (attention_sharing.py:105-366) in one call
// ------------------------------------------------------------------------------------------------
// The stages above, with the launches folded that do not wait for each other: K's averages beside the score statistics, the
// query-aware test and the share similarities beside the budgets, Q's averages, the pivots' own sets and the clearing of the
// map beside the masks.  Same device code, same results.  A launch that has nothing to do costs 2 to 2.7 us of the stream;
// against 15 launches, seven (five up to 128 blocks since) take 21 to 23 us off a layer (3001 tokens, 6177 of 64 channels, 10007
// of 28 / 4 heads).
struct HeadArgs {
  CoverCountArgs cover;
  int n_cover;  // workgroups 0 .. n_cover - 1: the budgets (0: made by other launches); then one per head
  QaArgs qa;
  sp_cluster_state st;
  const int32_t* head_cluster;
  const float* slash_blk;
  float *js_v, *js_s;
  // Behind the heads: a workgroup per tile of V (repack.nb 0: none).  The budgets and the query-aware test are 3 hq workgroups of
  // latency, the repack is bytes and depends on v alone; the two in one launch against two, us: 10007 tokens 4 kv heads 16 / 26,
  // 16384 (8 kv heads) 24 / 35, 32768 43 / 61, 65001 78 / 108.
  RepackArgs repack;
};
#define HEAD_LDS_BYTES(d, nb) (qa_lds_bytes(d, nb) > sizeof(CoverShared) ? qa_lds_bytes(d, nb) : sizeof(CoverShared))
__global__ __launch_bounds__(CS_THREADS) void sp_layer_heads_kernel(HeadArgs a) {
  extern __shared__ __attribute__((aligned(16))) char head_lds[];
  static_assert(CS_THREADS == QA_THREADS, "");
  if ((int)blockIdx.x < a.n_cover) {
    cover_count_vector(*reinterpret_cast<CoverShared*>(head_lds), a.cover, blockIdx.x);
    return;
  }
  const int h = (int)blockIdx.x - a.n_cover, lane = threadIdx.x & 63;
  if (h >= a.qa.hq) {
    const int tile = h - a.qa.hq;
    repack_v_tile<CS_THREADS>(a.repack, tile % a.repack.nb, tile / a.repack.nb, reinterpret_cast<sp_bf16*>(head_lds));
    return;
  }
  // (for a head that turns out query-aware too: the decision drops it)
  queryaware_head(a.qa, h, reinterpret_cast<float*>(head_lds), [&](int wave) {
    if (wave > 2) return;
    const float js = share_similarity(a.st, a.head_cluster[h], h, wave - 1, wave == 1 ? a.qa.vert_blk : a.slash_blk, lane);
    if (lane == 0) (wave == 1 ? a.js_v : a.js_s)[h] = js;
  });
}

// scratch of the call, each part 256-byte aligned
enum { LY_VERT_TOK, LY_SLASH_TOK, LY_VERT_BLK, LY_SLASH_BLK, LY_AVG_QK, LY_JS_QA, LY_JS_V, LY_JS_S, LY_USE_QA, LY_KBAR, LY_QBAR,
       LY_LASTQ, LY_COVER, LY_PARTS };
static size_t layer_scratch(int64_t n, int32_t hq, int32_t hkv, int32_t d, int32_t bs, size_t (&at)[LY_PARTS]) {
  const size_t nb = (size_t)sp_ceil_div(n, bs), tok = (size_t)hq * n * 4, blk = (size_t)hq * nb * 4, head = (size_t)hq * 4;
  const size_t bytes[LY_PARTS] = {tok, tok, blk, blk, blk, head, head, head, head, nb * hkv * d * 2, nb * hq * d * 2,
                                  sp_lastq_scores_workspace_bytes(n, hq, bs), sp_cover_select_workspace_bytes(2 * hq)};
  size_t sum = 0;
  for (int i = 0; i < LY_PARTS; ++i) {
    at[i] = sum;
    sum += (bytes[i] + 255) / 256 * 256;
  }
  return sum;
}

extern "C" size_t sp_select_layer_scratch_bytes(int64_t n, int32_t hq, int32_t hkv, int32_t d, int32_t bs, int64_t* offsets) {
  if (n <= 0 || hq <= 0 || hkv <= 0 || d <= 0 || bs <= 0) return 0;
  size_t at[LY_PARTS];
  const size_t sum = layer_scratch(n, hq, hkv, d, bs, at);
  for (int i = 0; offsets != nullptr && i <= LY_KBAR; ++i) offsets[i] = (int64_t)at[i];
  return sum;
}

static int select_layer(const char* who, const void* q, const void* k, int64_t n, int32_t hq, int32_t hkv, int32_t d,
                                    int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h, int32_t bs,
                                    uint32_t flags, const sp_cluster_state* state, const int32_t* head_cluster,
                                    int32_t layer_idx, int32_t min_blocks, int32_t max_blocks, double pattern_threshold,
                                    float similarity_threshold, double fallback_threshold, float queryaware_threshold,
                                    void* scratch, size_t scratch_bytes, float* qa_probs, int32_t* per_head, uint64_t* mask,
                                    float* avg_attn, const RepackArgs& repack, sp_stream_t stream) {
  SP_REQUIRE(state && head_cluster && scratch && qa_probs && per_head && mask, SP_ERR_INVALID_ARGUMENT,
             "%s: null pointer", who);
  SP_REQUIRE(n > 0 && hq > 0 && hkv > 0 && bs > 0 && d > 0, SP_ERR_INVALID_ARGUMENT, "%s: bad shape", who);
  SP_REQUIRE(hq <= DEC_MAX_HEADS, SP_ERR_UNSUPPORTED, "%s: hq=%d unsupported (max %d)", who, hq, DEC_MAX_HEADS);
  SP_REQUIRE(sp_ceil_div(n, bs) <= RS_MAX, SP_ERR_UNSUPPORTED, "%s: n=%lld needs more than %d blocks", who,
             (long long)n, RS_MAX);
  SP_REQUIRE(((uintptr_t)avg_attn % 16) == 0, SP_ERR_UNSUPPORTED, "%s: avg_attn must be 16-byte aligned", who);
  const int nb = (int)sp_ceil_div(n, bs);
  int rc = check_state(state, nb, who);
  if (rc) return rc;
  size_t at[LY_PARTS];
  SP_REQUIRE(scratch_bytes >= layer_scratch(n, hq, hkv, d, bs, at) && ((uintptr_t)scratch % 256) == 0, SP_ERR_WORKSPACE,
             "%s: scratch too small or not 256-byte aligned", who);
  auto part = [&](int i) { return (char*)scratch + at[i]; };
  auto floats = [&](int i) { return (float*)part(i); };
  float *vert_tok = floats(LY_VERT_TOK), *slash_tok = floats(LY_SLASH_TOK), *vert_blk = floats(LY_VERT_BLK),
        *slash_blk = floats(LY_SLASH_BLK);
  int32_t *use_qa = (int32_t*)part(LY_USE_QA), *decision = per_head, *nv = per_head + hq, *ns = nv + hq, *nv_f = ns + hq,
          *ns_f = nv_f + hq;
  hipStream_t s = (hipStream_t)stream;
  HeadArgs a = {};
  rc = queryaware_args(&a.qa, q, part(LY_KBAR), vert_blk, n, hq, hkv, d, q_stride_n, q_stride_h, bs, flags,
                       queryaware_threshold, floats(LY_AVG_QK), floats(LY_JS_QA), use_qa);
  if (rc != SP_OK) return rc;
  rc = sp_lastq_scores_run(q, k, n, hq, hkv, d, q_stride_n, q_stride_h, k_stride_n, k_stride_h, bs, flags, part(LY_LASTQ),
                           sp_lastq_scores_workspace_bytes(n, hq, bs), vert_tok, slash_tok, vert_blk, slash_blk, part(LY_KBAR), s);
  if (rc != SP_OK) return rc;
  if (n <= GSEL_ONE_LEN) {  // (with the heads beside them one launch is ahead for few vectors too: 14 heads, 131072 335 / 347)
    a.n_cover = 2 * hq;
    a.cover = CoverCountArgs{vert_tok, slash_tok, hq, (int)n, (long long)sp_thr_le((float)pattern_threshold), nv, ns, bs,
                             min_blocks, max_blocks};
  } else {
    rc = gsel_count_run(vert_tok, slash_tok, hq, 2 * hq, n, (float)pattern_threshold, nv, ns, bs, min_blocks, max_blocks,
                        part(LY_COVER), sp_cover_select_workspace_bytes(2 * hq), s, who);
    if (rc != SP_OK) return rc;
  }
  a.st = state_by_value(state);
  a.head_cluster = head_cluster;
  a.slash_blk = slash_blk;
  a.js_v = floats(LY_JS_V);
  a.js_s = floats(LY_JS_S);
  a.repack = repack;
  static_assert(sizeof(CoverShared) >= RP_LDS_BYTES, "");
  hipLaunchKernelGGL(sp_layer_heads_kernel, dim3((unsigned)(a.n_cover + hq + repack.nb * repack.hkv)), dim3(CS_THREADS),
                     HEAD_LDS_BYTES(d, nb), s, a);
  SP_LAUNCH_CHECK();
  const bool small = queryaware_small(d, nb);
  if (!small) {
    hipLaunchKernelGGL(sp_share_decide_kernel, dim3(1), dim3(DEC_MAX_HEADS), 0, s, a.st, head_cluster, layer_idx, hq, use_qa, nv,
                       ns, min_blocks, similarity_threshold, fallback_threshold, decision, a.js_v, a.js_s, nv_f, ns_f);
    SP_LAUNCH_CHECK();
  }
  const MaskBesides besides = {layer_idx,
                               pool_args(q, part(LY_QBAR), n, hq, d, q_stride_n, q_stride_h, bs, SP_POOL_TAIL_RESCALE, use_qa),
                               avg_attn, use_qa, nv, ns, min_blocks, similarity_threshold, fallback_threshold, decision, nv_f, ns_f,
                               a.js_v, a.js_s};
  auto launch_masks = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(hq, 2 * MASK_SPLIT), dim3(MASK_THREADS), 0, s, a.st, head_cluster, decision, vert_blk, slash_blk,
                       nv_f, ns_f, nb, (nb + 63) / 64, mask, besides);
  };
  small ? launch_masks(sp_build_mask_kernel<true, true>) : launch_masks(sp_build_mask_kernel<true, false>);
  SP_LAUNCH_CHECK();
  if (small)
    return queryaware_small_launch(part(LY_QBAR), part(LY_KBAR), decision, hq, hkv, d, nb, flags,
                                   sp_queryaware_select_score(pattern_threshold, nb), qa_probs, mask,
                                   ElectArgs{a.st, head_cluster, nv, ns, layer_idx}, s);
  return sp_queryaware_select_bf16(part(LY_QBAR), part(LY_KBAR), decision, hq, hkv, d, nb, flags, pattern_threshold, qa_probs,
                                   mask, part(LY_COVER), sp_cover_select_workspace_bytes(2 * hq), stream);
}

extern "C" int sp_select_layer_bf16(const void* q, const void* k, int64_t n, int32_t hq, int32_t hkv, int32_t d,
                                    int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h, int32_t bs,
                                    uint32_t flags, const sp_cluster_state* state, const int32_t* head_cluster,
                                    int32_t layer_idx, int32_t min_blocks, int32_t max_blocks, double pattern_threshold,
                                    float similarity_threshold, double fallback_threshold, float queryaware_threshold,
                                    void* scratch, size_t scratch_bytes, float* qa_probs, int32_t* per_head, uint64_t* mask,
                                    float* avg_attn, sp_stream_t stream) {
  return select_layer("sp_select_layer_bf16", q, k, n, hq, hkv, d, q_stride_n, q_stride_h, k_stride_n, k_stride_h, bs, flags, state, head_cluster,
                      layer_idx, min_blocks, max_blocks, pattern_threshold, similarity_threshold, fallback_threshold, queryaware_threshold,
                      scratch, scratch_bytes, qa_probs, per_head, mask, avg_attn, RepackArgs{}, stream);
}

extern "C" int sp_select_layer_repack_bf16(const void* q, const void* k, int64_t n, int32_t hq, int32_t hkv, int32_t d,
                                    int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h, int32_t bs,
                                    uint32_t flags, const sp_cluster_state* state, const int32_t* head_cluster,
                                    int32_t layer_idx, int32_t min_blocks, int32_t max_blocks, double pattern_threshold,
                                    float similarity_threshold, double fallback_threshold, float queryaware_threshold,
                                    void* scratch, size_t scratch_bytes, float* qa_probs, int32_t* per_head, uint64_t* mask,
                                    float* avg_attn, const void* v, int64_t v_stride_n, int64_t v_stride_h, void* vt, size_t vt_bytes,
                                    sp_stream_t stream) {
  RepackArgs repack;
  const int rc = repack_args(&repack, "sp_select_layer_repack_bf16", v, n, hkv, d, v_stride_n, v_stride_h, bs, vt, vt_bytes);
  if (rc != SP_OK) return rc;
  return select_layer("sp_select_layer_repack_bf16", q, k, n, hq, hkv, d, q_stride_n, q_stride_h, k_stride_n, k_stride_h, bs, flags, state, head_cluster,
                      layer_idx, min_blocks, max_blocks, pattern_threshold, similarity_threshold, fallback_threshold, queryaware_threshold,
                      scratch, scratch_bytes, qa_probs, per_head, mask, avg_attn, repack, stream);
}

// ------------------------------------------------------------------------------------------------
// pivot state update (attention_sharing.py:94-103 and the vs_ratio of :278-286, computed eagerly)
// ------------------------------------------------------------------------------------------------
// one workgroup per (row, head)
__global__ __launch_bounds__(RS_THREADS) void sp_pivot_rows_kernel(PivotArgs a, const float* __restrict__ avg_attn) {
  __shared__ PivotRowShared sh;
  extern __shared__ __attribute__((aligned(16))) char rs_lds[];
  if (a.decision[blockIdx.y] != SP_DEC_DENSE) return;
  pivot_row<RS_THREADS>(a, sh, rs_lds, avg_attn, blockIdx.x, blockIdx.y);
}

extern "C" int sp_pivot_update(const sp_cluster_state* state, const int32_t* head_cluster, const int32_t* decision,
                               const float* avg_attn, int32_t hq, int32_t nb, float pattern_threshold,
                               sp_stream_t stream) {
  int rc = check_state(state, nb, "sp_pivot_update");
  if (rc) return rc;
  SP_REQUIRE(head_cluster && decision && avg_attn, SP_ERR_INVALID_ARGUMENT, "sp_pivot_update: null pointer");
  SP_REQUIRE(hq > 0 && hq <= 1024 && nb > 0 && nb <= RS_MAX, SP_ERR_UNSUPPORTED,
             "sp_pivot_update: hq=%d nb=%d unsupported", hq, nb);
  if (state->n_clusters == 0) return SP_OK;
  const PivotArgs a = {state_by_value(state), head_cluster, decision, hq, nb, (nb + 63) / 64,
                       (long long)sp_thr_lt(pattern_threshold)};
  hipLaunchKernelGGL(sp_pivot_rows_kernel, dim3(nb, hq), dim3(RS_THREADS), rs_lds_bytes(nb), (hipStream_t)stream, a, avg_attn);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ------------------------------------------------------------------------------------------------
// CSR row pointers of a mask (triton_column_count_cumsum, shareprefill_attn.py:226-269)
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void sp_mask_row_pointers_kernel(const uint64_t* __restrict__ mask, int nb, int nbw,
                                                                   int32_t* __restrict__ row_ptr) {
  __shared__ int32_t cnt[RS_MAX];
  const int h = blockIdx.x;
  const uint64_t* mh = mask + (int64_t)h * nb * nbw;
  for (int r = threadIdx.x; r < nb; r += 256) {
    int c = 0;
    for (int w = 0; w < nbw; ++w) c += __popcll(mh[(int64_t)r * nbw + w]);
    cnt[r] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t* out = row_ptr + (int64_t)h * (nb + 1);
    int acc = 0;
    out[0] = 0;
    for (int r = 0; r < nb; ++r) {
      acc += cnt[r];
      out[r + 1] = acc;
    }
  }
}

extern "C" int sp_mask_row_pointers(const uint64_t* mask, int32_t hq, int32_t nb, int32_t* row_ptr,
                                    sp_stream_t stream) {
  SP_REQUIRE(mask && row_ptr && hq > 0 && nb > 0, SP_ERR_INVALID_ARGUMENT, "sp_mask_row_pointers: bad arguments");
  SP_REQUIRE(nb <= RS_MAX, SP_ERR_UNSUPPORTED, "sp_mask_row_pointers: nb=%d exceeds %d", nb, RS_MAX);
  hipLaunchKernelGGL(sp_mask_row_pointers_kernel, dim3(hq), dim3(256), 0, (hipStream_t)stream, mask, nb,
                     (nb + 63) / 64, row_ptr);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ------------------------------------------------------------------------------------------------
// The reference's block_idx form of a layer's selection (shareprefill_attn.py:484-486, 528-540): per head a list
// of flat block ids row * nb + col, in any order, padded with values outside the grid (the reference pads with
// nb * (nb + 1)).
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void sp_fill_u64_kernel(uint64_t* __restrict__ p, int64_t n, uint64_t value) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = value;
}

__global__ __launch_bounds__(256) void sp_block_idx_to_mask_kernel(const int64_t* __restrict__ idx, int64_t stride_h,
                                                                   int64_t k, int nb, int nbw,
                                                                   uint64_t* __restrict__ mask) {
  const int h = blockIdx.y;
  const int64_t cells = (int64_t)nb * nb;
  unsigned long long* mh = reinterpret_cast<unsigned long long*>(mask) + (int64_t)h * nb * nbw;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < k; i += (int64_t)gridDim.x * 256) {
    const int64_t id = idx[(int64_t)h * stride_h + i];
    if (id < 0 || id >= cells) continue;  // padding
    const int r = (int)(id / nb), c = (int)(id % nb);
    if (c > r) continue;  // above the diagonal: the kernel's causal mask leaves nothing of such a block
    atomicOr(mh + (int64_t)r * nbw + (c >> 6), 1ull << (c & 63));
  }
}

extern "C" int sp_block_idx_to_mask(const int64_t* block_idx, int64_t idx_stride_h, int64_t k, int32_t hq, int32_t nb,
                                    uint64_t* mask, sp_stream_t stream) {
  SP_REQUIRE(mask && hq > 0 && nb > 0 && k >= 0 && (block_idx || k == 0), SP_ERR_INVALID_ARGUMENT,
             "sp_block_idx_to_mask: bad arguments");
  SP_REQUIRE(hq <= 65535, SP_ERR_UNSUPPORTED, "sp_block_idx_to_mask: hq=%d exceeds 65535", hq);
  const int nbw = (nb + 63) / 64;
  const int64_t words = (int64_t)hq * nb * nbw;
  // a fill kernel rather than a memset node, so that the call can be recorded into a graph
  const unsigned fill_grid = (unsigned)(sp_ceil_div(words, 256) < 4096 ? sp_ceil_div(words, 256) : 4096);
  hipLaunchKernelGGL(sp_fill_u64_kernel, dim3(fill_grid), dim3(256), 0, (hipStream_t)stream, mask, words,
                     (uint64_t)0);
  SP_LAUNCH_CHECK();
  if (k > 0) {
    const unsigned gx = (unsigned)(sp_ceil_div(k, 256) < 1024 ? sp_ceil_div(k, 256) : 1024);
    hipLaunchKernelGGL(sp_block_idx_to_mask_kernel, dim3(gx, hq), dim3(256), 0, (hipStream_t)stream, block_idx,
                       idx_stride_h, k, nb, nbw, mask);
    SP_LAUNCH_CHECK();
  }
  return SP_OK;
}

// CSR row pointers of id lists (count_kernel, shareprefill_attn.py:187-223: a histogram of id / nb, then its running
// sum).  Duplicates count as often as they occur and the order of the ids does not matter, as in the reference.
__global__ __launch_bounds__(256) void sp_block_idx_row_pointers_kernel(const int64_t* __restrict__ idx,
                                                                        int64_t stride_h, int64_t k, int nb,
                                                                        int32_t* __restrict__ row_ptr) {
  __shared__ int32_t cnt[RS_MAX];
  __shared__ int32_t part[256];
  const int h = blockIdx.x;
  const int64_t cells = (int64_t)nb * nb;
  for (int r = threadIdx.x; r < nb; r += 256) cnt[r] = 0;
  __syncthreads();
  for (int64_t i = threadIdx.x; i < k; i += 256) {
    const int64_t id = idx[(int64_t)h * stride_h + i];
    if (id >= 0 && id < cells) atomicAdd(&cnt[(int)(id / nb)], 1);
  }
  __syncthreads();
  // running sum: every thread owns a contiguous run of rows
  const int per = (nb + 255) / 256;
  const int r0 = threadIdx.x * per, r1 = (r0 + per < nb) ? r0 + per : nb;
  int s = 0;
  for (int r = r0; r < r1; ++r) s += cnt[r];
  part[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int t = 0; t < 256; ++t) {
      const int v = part[t];
      part[t] = acc;
      acc += v;
    }
  }
  __syncthreads();
  int32_t* out = row_ptr + (int64_t)h * (nb + 1);
  int acc = part[threadIdx.x];
  for (int r = r0; r < r1; ++r) {
    acc += cnt[r];
    out[r + 1] = acc;
  }
  if (threadIdx.x == 0) out[0] = 0;
}

extern "C" int sp_block_idx_row_pointers(const int64_t* block_idx, int64_t idx_stride_h, int64_t k, int32_t hq,
                                         int32_t nb, int32_t* row_ptr, sp_stream_t stream) {
  SP_REQUIRE(row_ptr && hq > 0 && nb > 0 && k >= 0 && (block_idx || k == 0), SP_ERR_INVALID_ARGUMENT,
             "sp_block_idx_row_pointers: bad arguments");
  SP_REQUIRE(nb <= RS_MAX, SP_ERR_UNSUPPORTED, "sp_block_idx_row_pointers: nb=%d exceeds %d", nb, RS_MAX);
  hipLaunchKernelGGL(sp_block_idx_row_pointers_kernel, dim3(hq), dim3(256), 0, (hipStream_t)stream, block_idx,
                     idx_stride_h, k, nb, row_ptr);
  SP_LAUNCH_CHECK();
  return SP_OK;
}
