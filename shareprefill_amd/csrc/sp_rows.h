// What the rows of a pivot's block-average map turn into: the per-row selection (score_cover_idx_each_row,
// attn/utils.py:60-76) and the pivot state update (attention_sharing.py:94-103 and the vs_ratio of :278-286), a workgroup per
// row.  Included by the kernels that do it in a launch of their own and by those that have just made the row.
#pragma once
#include <cstring>
#include "sp_common.h"

// rank sort for short vectors (length <= RS_MAX)
#define RS_THREADS 256  // of the kernels that do nothing else
#define RS_MAX 4096

// ---- score_cover_idx_each_row (attn/utils.py:60-76) -------------------------------------------------
// keep[r] = first (count(cumsum < thr) + 1) entries of the sorted row, or exactly one if thr is never reached
// Views into the kernel's dynamic LDS, carved for rows of n entries (rs_lds_bytes(n) bytes: 14 KiB at nb = 1024
// instead of the 58 KiB a layout for the longest supported row takes, i.e. eight workgroups per CU instead of two).
struct RowShared {
  uint32_t* keys;                 // [n4], 16-byte aligned
  uint16_t* rank;                 // [n4]
  unsigned long long* sorted_fx;  // [n4]
  unsigned long long* chunk_sum;  // [threads]
  uint32_t* below;
  int* n_eff;
};
__host__ __device__ static inline size_t rs_lds_bytes(int n, int threads = RS_THREADS) {
  const size_t n4 = (size_t)((n + 3) & ~3);
  return n4 * 8 + threads * 8 + n4 * 4 + n4 * 2 + 16;
}
template <int THREADS>
__device__ static __forceinline__ RowShared rs_carve(char* base, int n) {
  const size_t n4 = (size_t)((n + 3) & ~3);
  RowShared sh;
  sh.sorted_fx = reinterpret_cast<unsigned long long*>(base);
  sh.chunk_sum = sh.sorted_fx + n4;
  sh.keys = reinterpret_cast<uint32_t*>(sh.chunk_sum + THREADS);
  sh.rank = reinterpret_cast<uint16_t*>(sh.keys + n4);
  sh.below = reinterpret_cast<uint32_t*>(base + n4 * 8 + THREADS * 8 + n4 * 4 + n4 * 2);
  sh.n_eff = reinterpret_cast<int*>(sh.below + 1);
  return sh;
}

// rank[i] for i < m among keys[0 .. m-1], four keys per LDS read; keys[m .. (m + 3) & ~3) must be zero
template <int THREADS>
__device__ static __forceinline__ void rs_ranks4(const uint32_t* keys, int m, uint16_t* rank, int tid) {
  const int m4 = (m + 3) & ~3;
  for (int i = tid; i < m; i += THREADS) {
    const uint32_t ki = keys[i];
    int r = 0;
    for (int j = 0; j < m4; j += 4) {
      const uint4 kj = *reinterpret_cast<const uint4*>(keys + j);
      r += (kj.x > ki) || (kj.x == ki && j < i);
      r += (kj.y > ki) || (kj.y == ki && j + 1 < i);
      r += (kj.z > ki) || (kj.z == ki && j + 2 < i);
      r += (kj.w > ki) || (kj.w == ki && j + 3 < i);
    }
    rank[i] = (uint16_t)r;
  }
}

// Only the row's entries up to its last non-zero key take part in the sort: the zero keys behind it sort last in
// index order whatever stands before them (rank[i] = i), add nothing to any cumulative mass and cannot be the
// crossing entry, so ranks, count and the "never reached -> keep one" rule come out as over the whole row.  Row r of
// a pivot's block-average map ends at column r: a third of the comparisons of the full square on average.
template <int THREADS>
__device__ static __forceinline__ int rs_row_keep(const float* __restrict__ row, int n, long long t_lt, const RowShared& sh, int tid = threadIdx.x) {
  if (tid == 0) {
    *sh.below = 0;
    *sh.n_eff = 0;
  }
  __syncthreads();
  int last = 0;
  for (int i = tid; i < n; i += THREADS) {
    const uint32_t key = sp_sort_key(row[i]);
    sh.keys[i] = key;
    if (key) last = i + 1;
  }
  if (last) atomicMax(sh.n_eff, last);
  __syncthreads();
  const int m = *sh.n_eff;
  for (int i = m + tid; i < ((m + 3) & ~3); i += THREADS) sh.keys[i] = 0;  // (past the row's end too)
  for (int i = m + tid; i < n; i += THREADS) sh.rank[i] = (uint16_t)i;
  __syncthreads();
  rs_ranks4<THREADS>(sh.keys, m, sh.rank, tid);
  __syncthreads();
  for (int i = tid; i < m; i += THREADS) sh.sorted_fx[sh.rank[i]] = sp_to_fixed(row[i]);
  __syncthreads();
  // inclusive scan of sorted_fx in contiguous per-thread chunks
  const int per = (m + THREADS - 1) / THREADS;
  const int lo = min(tid * per, m), hi = min(lo + per, m);
  unsigned long long s = 0;
  for (int i = lo; i < hi; ++i) s += sh.sorted_fx[i];
  unsigned long long incl = s;  // (integers: any order of the sums is the same)
#pragma unroll
  for (int o = 1; o < SP_WAVE; o <<= 1) {
    const unsigned long long below = __shfl_up(incl, o, SP_WAVE);
    if ((int)(tid & 63) >= o) incl += below;
  }
  if ((tid & 63) == 63) sh.chunk_sum[tid >> 6] = incl;
  __syncthreads();
  unsigned long long off = incl - s;
  for (int w = 0; w < (int)(tid >> 6); ++w) off += sh.chunk_sum[w];
  uint32_t cnt = 0;
  if (t_lt >= 0) {
    for (int i = lo; i < hi; ++i) {
      off += sh.sorted_fx[i];
      cnt += (off <= (unsigned long long)t_lt);
    }
  }
  if (cnt) atomicAdd(sh.below, cnt);
  __syncthreads();
  const int c = (int)*sh.below;
  return c < m ? c + 1 : 1;
}

// ---- pivot state update -----------------------------------------------------------------------------
__device__ __forceinline__ bool sp_slot_ok(const sp_cluster_state& st, int c) { return c >= 0 && c < st.n_clusters; }

// The struct a kernel receives by value.  A caller built against the first layout of the struct (it ended with
// `accum`; struct_bytes 0 or SP_CLUSTER_STATE_V1_BYTES) has no avg_map member: nothing behind `accum` is read.
static sp_cluster_state state_by_value(const sp_cluster_state* st) {
  sp_cluster_state v;
  memset(&v, 0, sizeof v);
  const bool full = st->struct_bytes >= (int32_t)sizeof(sp_cluster_state);
  memcpy(&v, st, full ? sizeof v : (size_t)SP_CLUSTER_STATE_V1_BYTES);
  if (!full) v.avg_map = nullptr;
  return v;
}

static int check_state(const sp_cluster_state* st, int nb, const char* who) {
  SP_REQUIRE(st != nullptr, SP_ERR_INVALID_ARGUMENT, "%s: null cluster state", who);
  SP_REQUIRE(st->struct_bytes == 0 || st->struct_bytes == (int32_t)SP_CLUSTER_STATE_V1_BYTES ||
                 st->struct_bytes >= (int32_t)sizeof(sp_cluster_state),
             SP_ERR_INVALID_ARGUMENT, "%s: cluster state struct_bytes=%d is neither 0, %d nor >= %d", who,
             st->struct_bytes, (int)SP_CLUSTER_STATE_V1_BYTES, (int)sizeof(sp_cluster_state));
  SP_REQUIRE(st->n_clusters >= 0 && st->nb == nb && st->nbw == (nb + 63) / 64, SP_ERR_INVALID_ARGUMENT,
             "%s: cluster state sized for nb=%d, call uses nb=%d", who, st->nb, nb);
  if (st->n_clusters > 0) {
    SP_REQUIRE(st->info && st->ratio && st->vert && st->slash && st->cols && st->dists && st->pattern && st->accum,
               SP_ERR_INVALID_ARGUMENT, "%s: cluster state has null slabs", who);
  }
  return SP_OK;
}

struct PivotRowShared {
  unsigned long long cov, tot;
  unsigned long long pad[16];
  int last;
};

// Row r of dense head h, by all THREADS threads of a workgroup.  The workgroup that finishes a head's last row (a counter in the cluster's info
// slot 5, which is zero between calls) turns the accumulated masses into the coverage ratio, publishes the pattern
// and leaves counter and accumulators zero again.  Invariant: state.accum and info[.][5] are zero on entry; the
// caller's slabs start zeroed and every completed call restores that.
struct PivotArgs {
  sp_cluster_state st;
  const int32_t *head_cluster, *decision;
  int hq, nb, nbw;
  long long t_lt;
};
template <int THREADS>
__device__ static __forceinline__ void pivot_row(const PivotArgs& a, PivotRowShared& sh, char* lds /* rs_lds_bytes(nb, THREADS) */,
                                                 const float* avg_attn, int r, int h) {
  const sp_cluster_state& st = a.st;
  const int32_t *const head_cluster = a.head_cluster, *const decision = a.decision;
  const int hq = a.hq, nb = a.nb, nbw = a.nbw;
  unsigned long long* const accum = reinterpret_cast<unsigned long long*>(st.accum);
  const RowShared rsh = rs_carve<THREADS>(lds, nb);
  const int c = head_cluster[h];
  if (!sp_slot_ok(st, c)) return;  // a dense head outside every shared cluster keeps no pattern
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (a caller's loop over rows would keep a dozen addresses made of it in registers)
  // One head per cluster and call: the election flags one, but a caller's own flags may name several heads of a
  // cluster.  The reference stores them one after the other, so the highest head's map is what stays
  // (attention_sharing.py:96-103); here the lower ones leave, or their rows would share the cluster's row counter
  // and accumulators with the highest head's.
  if (tid == 0) sh.last = 0;
  __syncthreads();
  bool later = false;
  for (int h2 = h + 1 + tid; h2 < hq; h2 += THREADS)
    later = later || (decision[h2] == SP_DEC_DENSE && head_cluster[h2] == c);
  if (later) sh.last = 1;
  __syncthreads();
  if (sh.last) return;
  const float* row = avg_attn + ((int64_t)h * nb + r) * nb;
  const int keep = rs_row_keep<THREADS>(row, nb, a.t_lt, rsh, tid);
  uint32_t* prow = reinterpret_cast<uint32_t*>(st.pattern + ((int64_t)c * nb + r) * nbw);
  for (int w = tid; w < nbw * 2; w += THREADS) {
    uint32_t bits = 0;
    for (int b = 0; b < 32; ++b) {
      const int col = w * 32 + b;
      if (col < nb && col <= r && rsh.rank[col] < keep) bits |= 1u << b;
    }
    if (r == 0 && w == 0) bits |= 1u;
    prow[w] = bits;
  }
  // vs_ratio pieces: mass under the pivot's own vertical / slash sets (a block in both counts twice) and the total
  if (tid == 0) {
    sh.cov = 0;
    sh.tot = 0;
  }
  __syncthreads();
  const uint8_t* cols = st.cols + (int64_t)c * nb;
  const uint8_t* dists = st.dists + (int64_t)c * nb;
  unsigned long long cov = 0, tot = 0;
  float* keep_row = st.avg_map ? st.avg_map + ((int64_t)c * nb + r) * nb : nullptr;
  for (int col = tid; col < nb; col += THREADS) {
    const float val = row[col];
    if (keep_row) keep_row[col] = val;  // the pivot's map itself, for get_pivotal_attn
    const unsigned long long fx = sp_to_fixed(val);
    tot += fx;
    if (col <= r) cov += fx * (unsigned long long)((cols[col] ? 1 : 0) + (dists[r - col] ? 1 : 0));
  }
  if (cov) atomicAdd(&sh.cov, cov);
  if (tot) atomicAdd(&sh.tot, tot);
  __syncthreads();
  if (tid == 0) {
    if (sh.cov) atomicAdd(&accum[c * 2 + 0], sh.cov);
    if (sh.tot) atomicAdd(&accum[c * 2 + 1], sh.tot);
    __threadfence();  // this row's pattern words and masses are visible before the row is counted
    sh.last = atomicAdd(&st.info[c * 8 + 5], 1) == nb - 1;
  }
  __syncthreads();
  if (!sh.last) return;
  // ---- the head's last row: every other row of it has been counted, so its atomics and stores are visible ----
  __threadfence();
  // every out-of-range slash / vertical slot of the reference's id list is the padding id 0
  unsigned long long pad = 0;
  for (int i = tid; i < nb; i += THREADS) {
    if (cols[i]) pad += (unsigned long long)i;
    if (dists[i]) pad += (unsigned long long)i;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) pad += __shfl_xor(pad, o, SP_WAVE);
  if ((tid & 63) == 0) sh.pad[tid >> 6] = pad;
  __syncthreads();
  if (tid == 0) {
    pad = 0;
    for (int w = 0; w < THREADS / SP_WAVE; ++w) pad += sh.pad[w];
    const unsigned long long acc_cov = atomicAdd(&accum[c * 2 + 0], 0ull), acc_tot = atomicAdd(&accum[c * 2 + 1], 0ull);
    const unsigned long long a00 = sp_to_fixed(avg_attn[(int64_t)h * nb * nb]);
    // one IEEE operation at a time (no fused multiply-add), so the value is reproducible on a CPU
    const double covd = __dadd_rn((double)acc_cov, __dmul_rn((double)pad, (double)a00));
    const double totd = (double)acc_tot;
    st.ratio[c] = totd > 0.0 ? __ddiv_rn(covd, totd) : (double)NAN;
    accum[c * 2 + 0] = 0;
    accum[c * 2 + 1] = 0;
    st.info[c * 8 + 5] = 0;
    __threadfence();
    st.info[c * 8 + 1] = 1;
  }
}
