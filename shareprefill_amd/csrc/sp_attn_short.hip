// Block-sparse causal attention for short prompts (same operation as sp_attn.hip, which takes the long ones).
//
// A launch over a few thousand tokens is bound by latency, not by the matrix cores: the persistent kernel's work item --
// two rows of up to 128 keys per block step, a ticket, a block list, two barriers and an epilogue around it -- is too
// large a part of the launch (3001 tokens, 32 heads: 384 items of up to 16 block steps on 256 CUs), and the launches that
// prepare it (V repack, tickets, pairing) cost as much as the arithmetic of a short prompt.  This kernel needs none of
// them and cuts the work finer:
//   * one workgroup per (128-query block, head), 4 waves of 32 queries, two workgroups per CU (three with 64 channels): K and
//     V tiles of 64 keys double-buffered in LDS, one barrier per tile, and a plain loop of S, softmax and P.V.  Workgroups of
//     different rows run out of step, so one's matrix instructions fall into another's softmax; the persistent kernel's
//     software pipeline inside the wave was built here too and measured the same (a wave alone issues an instruction about
//     every 8 cycles, whatever it is), at twice the code;
//   * a row's keys split over two sets of four waves, merged through LDS, halve the chain of tiles; that was worth 6 % up to 700
//     tokens and cost 4 % at 2048 (32 heads: 25.0 -> 23.6 us, 1500 44.5 -> 44.0, 2048 57.3 -> 59.4) and gave other bits than the
//     persistent kernel's, so it was taken out;
//   * workgroups are dispatched heaviest row first, all heads of one row before the next; a CU that finishes a row takes
//     the next one, which balances causal rows without tickets.  The query heads of a kv group share an XCD (one L2) for a
//     row; the XCDs trade groups from row to row, or heads that keep more blocks than others would leave the other XCDs idle
//     (8192 tokens, masks at coverage 0.95: 319 us with a fixed assignment, 178 with the rotating one);
//   * V is read as it is: the tile is row-major in LDS and the V^T operand comes from the transposing LDS read
//     (ds_read_b64_tr_b16: the 16 lanes of a group address 4 keys x 16 channels and each receives 4 keys of its channel).
//     S^T = K . Q^T leaves a lane with keys 4g .. 4g+3 of every 16-key tile (g = lane / 16), which is exactly what two such
//     reads deliver, so P^T is the S^T accumulators converted to bf16 in place;
//   * a pivot head's block-average map is made by the same workgroup at the end of its row (no second kernel), and so is the
//     row's pattern in the sharing state, which needs nothing but that row (a launch in every layer, of which all but one per
//     cluster had nothing to do: 2.4 us of a layer of 3001 tokens, 1.4 of 6177 with 64 channels); a call without decisions
//     has its maps cleared here (a fill launch in front of the kernel costs its caller 5 us of host time, 2.6 us of a layer of
//     700 tokens).
// Two rows sharing one K / V tile, as in the persistent kernel, halve the tile traffic per flop, which is why that one
// stays for long prompts; sp_short_attn_max_tokens holds the lines between the two and the figures.  Both give the same bits.
#include "sp_rows.h"

#include <type_traits>

struct AsArgs {
  const sp_bf16 *q, *k, *v;
  const uint64_t* mask;      // [hq][nb][nbw]
  const int32_t* decision;   // [hq] or null
  sp_bf16* out;              // [n][hq][D]
  float* avg_attn;           // [hq][nb][nb], written for pivot heads
  float* block_sums;         // [slots][nb (nb + 1) / 2][128] of pivot heads
  int slots;                 // pivot heads there is room for; -1: no maps wanted
  int64_t n, sq_n, sq_h, sk_n, sk_h, sv_n, sv_h;
  int hq, group, nb, nbw;
  int zero_maps;             // 1: no decisions, every row of avg_attn is cleared
  float scale_log2;
};
struct AsPivotArgs : AsArgs {
  PivotArgs pivot;
};

typedef __bf16 as_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 as_bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 as_bf16x2 __attribute__((ext_vector_type(2)));
typedef float as_floatx4 __attribute__((ext_vector_type(4)));
typedef float as_floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t as_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t as_u32x2 __attribute__((ext_vector_type(2)));

#define AS_BS 128
#define AS_TILE 64      // keys per step
#define AS_THREADS 256  // 4 waves x 32 queries
#define AS_WAVES 4
#define AS_MAX_NB 512     // blocks a row's list holds
#define AS_LDS_BYTES(D) (4 * AS_TILE * (D) * 2)
#define AS_NO_MAX (-1.0e30f)         // "no key seen yet": finite, so exp2(S * scale - m) is +inf or 0, never NaN
#define AS_P_TOO_LARGE 0x40004000u   // bf16 pair: exponent >= 128 in either half

typedef __attribute__((address_space(3))) void* as_lds_ptr;
typedef const __attribute__((address_space(1))) void* as_gbl_ptr;

// K and V tiles are [64 keys][D] bf16 in 16-byte chunks, the chunk index XOR-swizzled by the row so that both kinds of
// operand read are free of bank conflicts: the K read (one chunk of 16 consecutive rows) and the transposing V read (two
// neighbouring chunks of 16 consecutive rows).  Rows of 64 channels are half a bank cycle long: two rows share a swizzle.
template <int D>
__device__ __forceinline__ int as_swz(int row) {
  return D == 128 ? (row & 15) : ((row >> 1) & 7);
}

__device__ __forceinline__ uint32_t as_pack2(float a, float b) {
  as_floatx2 f;
  f[0] = a;
  f[1] = b;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, as_bf16x2));
}

// One tile by direct global -> LDS 128-bit loads: a wave-instruction fills 1 KiB (lane i writes chunk base + i and fetches
// whichever chunk belongs there).  Row and swizzle of a lane are the same in every instruction up to a uniform step, so a
// lane's address is a uniform base plus an offset made once; only the tile that reaches past the sequence clamps its rows
// onto the last key (such keys lie behind every stored query).
template <int D>
__device__ __forceinline__ uint32_t as_lane_off(int64_t stride_n, int wave, int lane) {
  constexpr int CHUNKS = D / 8, ROWS = 64 / CHUNKS;  // chunks per row, rows per wave-instruction
  const int row = wave * ROWS + lane / CHUNKS;
  return (uint32_t)(row * (int)stride_n + ((lane % CHUNKS) ^ as_swz<D>(row)) * 8) * 2u;
}
template <int D>
__device__ __forceinline__ void as_issue(const sp_bf16* __restrict__ x, int64_t stride_n, int64_t key0, int64_t n,
                                         uint32_t lane_off, char* tile, int wave, int lane) {
  constexpr int CHUNKS = D / 8, ROWS = 64 / CHUNKS;
  constexpr int STEP = ROWS * AS_WAVES, ITS = AS_TILE / STEP;  // rows per instruction of all waves (a multiple of the swizzle's period)
  if (key0 + AS_TILE <= n) {
    const char* base = reinterpret_cast<const char*>(x + key0 * stride_n);
#pragma unroll
    for (int it = 0; it < ITS; ++it)
      __builtin_amdgcn_global_load_lds((as_gbl_ptr)(base + (int64_t)it * STEP * 2 * stride_n + lane_off),
                                       (as_lds_ptr)(tile + (it * AS_WAVES + wave) * 1024), 16, 0, 0);
  } else {
    int ln = lane;
    asm volatile("" : "+v"(ln));  // (keeps this rare path's lane arithmetic out of the tile loop)
#pragma unroll 1
    for (int it = 0; it < ITS; ++it) {
      const int seg = it * AS_WAVES + wave, row = seg * ROWS + ln / CHUNKS;
      int64_t key = key0 + row;
      if (key > n - 1) key = n - 1;
      __builtin_amdgcn_global_load_lds((as_gbl_ptr)(x + key * stride_n + ((ln % CHUNKS) ^ as_swz<D>(row)) * 8),
                                       (as_lds_ptr)(tile + seg * 1024), 16, 0, 0);
    }
  }
}

// Transposing LDS read the compiler does not track (valid after as_wait_v on the same registers).  Through the builtin it
// waits for every direct-to-LDS load in flight before each of these reads -- the next tile's whole memory latency in
// every step: 1.6 us per 64 keys where the arithmetic takes half of that.
template <int IMM>
__device__ __forceinline__ as_u32x2 as_read_tr(uint32_t addr) {
  as_u32x2 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(IMM));
  return r;
}
template <int N>
__device__ __forceinline__ void as_wait_v(as_u32x2 (&r)[8]) {  // all but the N youngest LDS reads have landed
  asm volatile("s_waitcnt lgkmcnt(%8)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]), "+v"(r[6]), "+v"(r[7])
               : "n"(N));
}
// The same for a K operand (16 bytes of a lane's row).  Left to itself the compiler waits for each pair of these reads where it
// uses them.
template <int IMM>
__device__ __forceinline__ as_u32x4 as_read_k(uint32_t addr) {
  as_u32x4 r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(IMM));
  return r;
}
template <int N>
__device__ __forceinline__ void as_wait_k(as_u32x4 (&r)[4]) {
  asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]) : "n"(N));
}
template <int N>
__device__ __forceinline__ void as_wait_k(as_u32x4 (&r)[2]) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(r[0]), "+v"(r[1]) : "n"(N));
}
template <int K, int N, typename F>
__device__ __forceinline__ void as_static_for(F&& f) {
  if constexpr (K < N) {
    f(std::integral_constant<int, K>{});
    as_static_for<K + 1, N>(f);
  }
}

// max over the lanes l, l ^ 16, l ^ 32, l ^ 48 that share a query
__device__ __forceinline__ float as_groupmax(float v) {
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = fmaxf(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
  u = __builtin_bit_cast(uint32_t, v);
  const auto b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)b[0]), __builtin_bit_cast(float, (uint32_t)b[1]));
}

// Args = AsPivotArgs: with the pivots' patterns (an instance of its own: prompts that select nothing, whose launch is the
// whole layer, run 1.5 % slower with that code in theirs).
template <int D, typename Args>
__global__ __launch_bounds__(AS_THREADS, 2) void sp_attn_short_kernel(Args a) {
  constexpr int QT = 2;                             // 16-query tiles per wave
  constexpr int KS = D / 32, CT = D / 16;           // channel steps of S, channel tiles of O
  constexpr int WAVES = AS_WAVES, THREADS = AS_THREADS, WQ = 16 * QT;
  constexpr int TILE_BYTES = AS_TILE * D * 2;
  extern __shared__ __attribute__((aligned(1024))) char lds[];  // [buffer][K | V]
  __shared__ uint16_t list[AS_MAX_NB];
  const int t = threadIdx.x, lane = t & 63, lq = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // query band
  const uint32_t lds_base = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)lds;
  int h, rr;  // head, rank of the row (0 = the last, heaviest one)
  if ((a.hq & 7) == 0) {
    const int per = a.hq >> 3, i = blockIdx.x >> 3;
    rr = i / per;
    h = ((blockIdx.x + rr) & 7) * per + i % per;
  } else {
    h = blockIdx.x % a.hq;
    rr = blockIdx.x / a.hq;
  }
  const int r = a.nb - 1 - rr;
  const int kvh = h / a.group;
  const sp_bf16* kh = a.k + (int64_t)kvh * a.sk_h;
  const sp_bf16* vh = a.v + (int64_t)kvh * a.sv_h;

  const int dec = a.slots >= 0 ? a.decision[h] : 0;  // (asked for up here: its way from memory passes under the mask's)

  const int q_off = wave * WQ + lq;  // the first of the lane's queries; the others are 16 further each
  const int64_t qrow = (int64_t)r * AS_BS + q_off;
  as_bf16x8 qb[QT][KS];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int64_t qr = qrow + 16 * qt < a.n ? qrow + 16 * qt : a.n - 1;
    const sp_bf16* src = a.q + (int64_t)h * a.sq_h + qr * a.sq_n + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qb[qt][ks] = __builtin_bit_cast(as_bf16x8, *reinterpret_cast<const uint4*>(src + 32 * ks));
  }
  const uint32_t k_lane = as_lane_off<D>(a.sk_n, wave, lane), v_lane = as_lane_off<D>(a.sv_n, wave, lane);
  auto issue = [&](int c, int half, int buf) {
    const int64_t key0 = (int64_t)c * AS_BS + half * AS_TILE;
    // (a last block that ends in its first half: the second half is all beyond the sequence; its one key is the last)
    const int64_t k0 = key0 < a.n ? key0 : a.n - 1;
    as_issue<D>(kh, a.sk_n, k0, a.n, k_lane, lds + buf * 2 * TILE_BYTES, wave, lane);
    as_issue<D>(vh, a.sv_n, k0, a.n, v_lane, lds + buf * 2 * TILE_BYTES + TILE_BYTES, wave, lane);
  };
  // the row's kept blocks, ascending: every wave counts the (uniform) mask words, wave w compacts its share of them
  int n_blk = 0, c = 0;
  {
    const uint64_t* row = a.mask + ((int64_t)h * a.nb + r) * a.nbw;
    for (int wi = 0; wi <= (r >> 6); ++wi) {
      uint64_t x = row[wi];
      if (wi == (r >> 6) && (r & 63) != 63) x &= (2ull << (r & 63)) - 1ull;
      if (n_blk == 0 && x != 0ull) {  // the first tile is on its way while the list is made
        c = wi * 64 + __builtin_ctzll(x);
        issue(c, 0, 0);
      }
      if (wi % WAVES == wave && ((x >> lane) & 1ull))
        list[n_blk + __builtin_popcountll(x & ((1ull << lane) - 1ull))] = (uint16_t)(wi * 64 + lane);
      n_blk += __builtin_popcountll(x);
    }
    n_blk = __builtin_amdgcn_readfirstlane(n_blk);
  }
  // the list is complete (a plain __syncthreads would wait for the first tile as well)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  as_floatx4 o[CT][QT], l[QT];  // l: row sums (ones . P, every row of the tile holds the sum)
  float m[QT], l_mark[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) o[ct][qt] = (as_floatx4){0, 0, 0, 0};
    l[qt] = (as_floatx4){0, 0, 0, 0};
    m[qt] = AS_NO_MAX;
    l_mark[qt] = 0.f;
  }
  const as_bf16x8 ones = __builtin_bit_cast(as_bf16x8, (as_u32x4){0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  // pivot heads: this row's sums per block, [column][128 queries], in the slab of the head's rank among them
  const bool pivot = a.slots >= 0 && dec == SP_DEC_DENSE;  // (uniform)
  float* pu = nullptr;
  if (pivot) {
    int slot = 0;
    for (int i = 0; i < h; i += SP_WAVE)
      slot += __builtin_popcountll(__ballot(i + lane < h && a.decision[i + lane < h ? i + lane : 0] == SP_DEC_DENSE));
    if (slot < a.slots)
      pu = a.block_sums + ((int64_t)slot * ((int64_t)a.nb * (a.nb + 1) / 2) + (int64_t)r * (r + 1) / 2) * AS_BS;
  }

  // LDS byte offsets of the lane's operands: K row lq, logical chunk 4 ks + g; V row 4 g + lq / 4, 8-byte piece lq % 4 of the
  // 32 bytes of channel tile ct.  Rows 16 further have the same swizzle.
  const int koff = lq * (D * 2), kswz = as_swz<D>(lq);
  const int vrow = 4 * g + (lq >> 2);
  const int voff = vrow * (D * 2) + 8 * (lq & 1), vswz = as_swz<D>(vrow), vhalf = (lq >> 1) & 1;

  int c_next = 0;
  // One step per tile, two per block.  The block list is read a block ahead of its use.
  for (int st = 0; st < 2 * n_blk; ++st) {
    const int i = st >> 1, half = st & 1, buf = half;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's loads of the tile have landed
    __syncthreads();                     // ... everybody's; and the other buffer's readers are done
    if (half == 0) {
      issue(c, 1, buf ^ 1);
      c_next = (int)list[i + 1 < n_blk ? i + 1 : i];
    } else if (i + 1 < n_blk) {
      c_next = __builtin_amdgcn_readfirstlane(c_next);
      issue(c_next, 0, buf ^ 1);
    }
    const bool diag = c == r;
    if (!diag || half * AS_TILE <= wave * WQ + WQ - 1) {  // (else: every key of the tile lies behind the wave's queries)
      // Operands are fetched ahead of the matrix instructions that take them: K two 16-key groups ahead, the first of V's in
      // front of the softmax, the others a group ahead.  With every operand waited for where it is used a step of a workgroup alone
      // on its CU took 3800 cycles, ten LDS latencies among them; now 3400 (700 tokens 23.8 -> 22.2 us, 3001 115.4 -> 112.5, 6400
      // 178 -> 173; 64 channels 1000 tokens 23.5 -> 22.7, 20000 347 -> 342).  Of them the next tile's loads take 700 (32 KiB at the CU's
      // 64 bytes a cycle); spread between the matrix instructions or put behind them they cost more (700 tokens 24.2 and 23.5).
      const uint32_t kt_addr = lds_base + (uint32_t)(buf * 2 * TILE_BYTES);
      const uint32_t vt_addr = lds_base + (uint32_t)(buf * 2 * TILE_BYTES + TILE_BYTES + voff);
      constexpr int GR = CT / 4;  // groups of four channel tiles
      as_u32x2 vr[2][8];
      auto fetch_v = [&](auto hc, auto gc) {  // group gc of half hc, into vr[gc & 1] (the first of the next half: where it is free)
        constexpr int hh = decltype(hc)::value, gi = decltype(gc)::value, to = GR == 1 ? hh & 1 : gi & 1;
        as_static_for<0, 4>([&](auto uc) {
          constexpr int u = decltype(uc)::value;
          const uint32_t ad = vt_addr + (uint32_t)(((2 * (4 * gi + u) + vhalf) ^ vswz) << 4);
          vr[to][2 * u] = as_read_tr<hh * 32 * (D * 2)>(ad);
          vr[to][2 * u + 1] = as_read_tr<hh * 32 * (D * 2) + 16 * (D * 2)>(ad);
        });
      };
      as_floatx4 s[4][QT];
      {
        as_u32x4 kr[2][KS];
        auto fetch_k = [&](auto kc) {
          constexpr int kt = decltype(kc)::value;
          as_static_for<0, KS>([&](auto sc) {
            constexpr int ks = decltype(sc)::value;
            kr[kt & 1][ks] = as_read_k<kt * 16 * (D * 2)>(kt_addr + (uint32_t)(koff + (((4 * ks + g) ^ kswz) << 4)));
          });
        };
        fetch_k(std::integral_constant<int, 0>{});
        fetch_k(std::integral_constant<int, 1>{});
        as_static_for<0, 4>([&](auto kc) {
          constexpr int kt = decltype(kc)::value;
          as_wait_k<(kt < 3 ? KS : 0)>(kr[kt & 1]);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) s[kt][qt] = (as_floatx4){0, 0, 0, 0};
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
              s[kt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(as_bf16x8, kr[kt & 1][ks]), qb[qt][ks], s[kt][qt], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (kt + 2 < 4) fetch_k(std::integral_constant<int, kt + 2>{});
        });
      }
      if (diag) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (half * AS_TILE + 16 * kt + 4 * g + j > q_off + 16 * qt) s[kt][qt][j] = -INFINITY;
      }
      fetch_v(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
      uint32_t pk[QT][8];
      auto softmax = [&](int qt, int hh) {  // half hh: 32 keys
#pragma unroll
        for (int kt = 2 * hh; kt < 2 * hh + 2; ++kt) {
          float e[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) e[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][qt][j], a.scale_log2, -m[qt]));
          pk[qt][2 * kt] = as_pack2(e[0], e[1]);
          pk[qt][2 * kt + 1] = as_pack2(e[2], e[3]);
        }
      };
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        softmax(qt, 0);
        softmax(qt, 1);
      }
      as_static_for<0, 2>([&](auto hc) {
        constexpr int hh = decltype(hc)::value;
        // The running max is lazy, as in the persistent kernel and in its steps of 32 keys, which gives its bits: it moves
        // only when some probability came out at 2 or more (or is inf: a row's first keys), and then the probabilities are
        // formed again before they are used.
        uint32_t det = 0u;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
          for (int i = 4 * hh; i < 4 * hh + 4; i += 2) det |= pk[qt][i] | pk[qt][i + 1];
        as_wait_v<0>(vr[GR == 1 ? hh & 1 : 0]);  // the half's first group (no read may be in flight across the branch)
        if (__ballot((det & AS_P_TOO_LARGE) != 0u) != 0ull) {
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) {
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 2 * hh; kt < 2 * hh + 2; ++kt)
              mx = fmaxf(mx, fmaxf(fmaxf(s[kt][qt][0], s[kt][qt][1]), fmaxf(s[kt][qt][2], s[kt][qt][3])));
            const float m_new = fmaxf(m[qt], as_groupmax(mx * a.scale_log2));
            const float alpha = __builtin_amdgcn_exp2f(m[qt] - m_new);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) o[ct][qt] *= alpha;
            l[qt] *= alpha;
            l_mark[qt] *= alpha;
            m[qt] = m_new;
            softmax(qt, hh);
            if constexpr (hh == 0) softmax(qt, 1);
          }
        }
        // O += V^T . P: groups of four channel tiles, the next group's operands on their way
        as_bf16x8 p[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
          p[qt] = __builtin_bit_cast(as_bf16x8, (as_u32x4){pk[qt][4 * hh], pk[qt][4 * hh + 1], pk[qt][4 * hh + 2], pk[qt][4 * hh + 3]});
        as_static_for<0, GR>([&](auto gc) {
          constexpr int gi = decltype(gc)::value, from = GR == 1 ? hh & 1 : gi & 1;
          if constexpr (gi > 0) as_wait_v<0>(vr[from]);
          if constexpr (gi + 1 < GR)
            fetch_v(hc, std::integral_constant<int, gi + 1>{});
          else if constexpr (hh == 0)
            fetch_v(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const as_u32x4 raw = __builtin_shufflevector(vr[from][2 * u], vr[from][2 * u + 1], 0, 1, 2, 3);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
              o[4 * gi + u][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(as_bf16x8, raw), p[qt], o[4 * gi + u][qt], 0, 0, 0);
          }
          if constexpr (gi == 0) {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) l[qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, p[qt], l[qt], 0, 0, 0);
          }
        });
      });
    }
    if (pu != nullptr && half == 1) {  // pivot head: the block's softmax mass, log2 units
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const float u = __builtin_amdgcn_logf(l[qt][0] - l_mark[qt]) + m[qt];
        l_mark[qt] = l[qt][0];
        if (g == 0) pu[(int64_t)c * AS_BS + q_off + 16 * qt] = u;
      }
    }
    if (half == 1) c = c_next;
  }

  float inv_l[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    inv_l[qt] = 1.0f / l[qt][0];
    if (qrow + 16 * qt < a.n) {
      sp_bf16* dst = a.out + ((qrow + 16 * qt) * a.hq + h) * D + 4 * g;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        *reinterpret_cast<uint2*>(dst + ct * 16) = make_uint2(as_pack2(o[ct][qt][0] * inv_l[qt], o[ct][qt][1] * inv_l[qt]),
                                                              as_pack2(o[ct][qt][2] * inv_l[qt], o[ct][qt][3] * inv_l[qt]));
    }
  }
  if (a.zero_maps)
    for (int i = t; i < a.nb; i += THREADS) a.avg_attn[((int64_t)h * a.nb + r) * a.nb + i] = 0.f;
  if (!pivot) return;  // (uniform)
  if (pu == nullptr) {  // more pivots than the caller made room for: no map, and visibly so
    for (int i = t; i < n_blk; i += THREADS) a.avg_attn[((int64_t)h * a.nb + r) * a.nb + (int)list[i]] = NAN;
    return;
  }
  // pivot head: avg[r][c] = mean over the block's valid queries of exp2(u - m[q]) / l[q].  A wave
  // reads back its own sums (its own stores), folds its queries, and the waves meet in LDS.
  float* const part = reinterpret_cast<float*>(lds);  // [block][wave]
  __syncthreads();                                    // LDS is free, the stores of pu have left
  for (int i = 0; i < n_blk; ++i) {
    const int c = (int)list[i];
    float x = 0.f;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
      if (qrow + 16 * qt < a.n) {
        x += __builtin_amdgcn_exp2f(pu[(int64_t)c * AS_BS + q_off + 16 * qt] - m[qt]) * inv_l[qt];
      }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) x += __shfl_xor(x, off, SP_WAVE);
    if (lane == 0) part[i * WAVES + wave] = x;
  }
  __syncthreads();
  const int64_t rem = a.n - (int64_t)r * AS_BS;
  const float inv_q = 1.0f / (float)(rem < AS_BS ? (int)rem : AS_BS);
  for (int i = t; i < n_blk; i += THREADS) {
    float x = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) x += part[i * WAVES + w];
    a.avg_attn[((int64_t)h * a.nb + r) * a.nb + (int)list[i]] = x * inv_q;
  }
  if constexpr (std::is_same<Args, AsPivotArgs>::value) {
    __shared__ PivotRowShared pivot_sh;
    __syncthreads();  // the row is written, LDS is free
    pivot_row<THREADS>(a.pivot, pivot_sh, lds, a.avg_attn, r, h);
  }
}

// ---- host ---------------------------------------------------------------------------------------------
// The lines between this kernel and the persistent one, where the latter's shared tiles outweigh its fixed costs.  Whole layers,
// us here / there, in one call (two runs of one side within 0.5 %).  128 channels:
//   masks of the selection, 32 query / 8 kv heads: coverage 0.65 6656 tokens 180 / 189, 8192 198 / 202, 10007 243 / 256; 0.95 201 / 210,
//   226 / 236, 282 / 285; 0.99 257 / 257, 324 / 315, 451 / 433; every head query-aware 209 / 220, 243 / 251, 306 / 312;
//   28 / 4 heads, the same coverages at 6656 and 8192: 166 / 189, 183 / 198; 184 / 199, 208 / 220; 239 / 237, 299 / 287; 8 / 2 heads: 88 /
//   101, 91 / 99; 132 / 146, 142 / 138; 178 / 180, 205 / 207;
//   every block kept: 32 / 8 heads 5120 220 / 242, 5632 263 / 273, 6177 318 / 317, 6656 358 / 347; 28 / 4 5632 234 / 260, 6656 316 / 331;
//   8 / 2 6656 148 / 156.
// So up to 6656 tokens this kernel is never behind by more than 1 %, whatever the coverage; beyond, it is ahead at low coverage and
// behind at 0.99.  (The line of dense masks stands a little low: 5632 is this kernel's too.)
// 64 channels, where the persistent kernel computes on zero-padded tiles (padding counted), 32 / 8 heads: 0.65 8192 148 / 254, 32768
// 448 / 810, 49152 715 / 1244; 0.95 143 / 253, 583 / 907, 1268 / 1692; 0.99 147 / 261, 1177 / 1422, 2970 / 3100; every block kept 311 / 409,
// 4920 / 5135, 10775 / 11010; 14 / 2 heads 0.95 32768 333 / 462, every block 2062 / 2198.  The line is where both were once even without
// the padding; what lies beyond it is not measured but for these lengths, and each pivot's block sums take 16.8 MB there.
extern "C" int64_t sp_short_attn_max_tokens(int32_t d) {
  return d == 64 ? 32768 : 6656;
}
extern "C" int64_t sp_short_attn_max_dense_tokens(int32_t d) {
  return d == 64 ? 32768 : 5120;
}

extern "C" size_t sp_short_attn_workspace_bytes(int64_t n, int32_t hq) {
  return n <= 0 || hq <= 0 ? 0 : (size_t)hq * sp_attn_pivot_scratch_bytes(n, AS_BS);
}

static int as_launch(const char* who, const void* q, const void* k, const void* v, int64_t n, int32_t hq, int32_t hkv,
                                      int32_t d, int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                                      int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h, float softmax_scale,
                                      const uint64_t* mask, const int32_t* decision, void* out, float* avg_attn,
                                      void* workspace, size_t workspace_bytes, const PivotArgs* pivot, sp_stream_t stream) {
  SP_REQUIRE(q && k && v && mask && out, SP_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
  SP_REQUIRE(n > 0 && hq > 0 && hkv > 0 && hq % hkv == 0, SP_ERR_INVALID_ARGUMENT,
             "%s: bad shape n=%lld hq=%d hkv=%d", who, (long long)n, hq, hkv);
  SP_REQUIRE(softmax_scale > 0.f, SP_ERR_INVALID_ARGUMENT, "%s: softmax_scale must be > 0", who);
  SP_REQUIRE(d == 128 || d == 64, SP_ERR_UNSUPPORTED, "%s: head_dim %d unsupported (64 or 128)", who, d);
  SP_REQUIRE((q_stride_n | q_stride_h | k_stride_n | k_stride_h | v_stride_n | v_stride_h) % 8 == 0 &&
                 ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) % 16 == 0,
             SP_ERR_UNSUPPORTED, "%s: tensors must be 16-byte aligned, strides multiple of 8", who);
  SP_REQUIRE(k_stride_n >= 0 && v_stride_n >= 0 && AS_BS * k_stride_n < (1ll << 31) && AS_BS * v_stride_n < (1ll << 31),
             SP_ERR_UNSUPPORTED, "%s: token strides %lld / %lld unsupported", who, (long long)k_stride_n,
             (long long)v_stride_n);
  const int64_t nb = sp_ceil_div(n, AS_BS);
  SP_REQUIRE(nb <= AS_MAX_NB && nb * hq < (1ll << 31), SP_ERR_UNSUPPORTED, "%s: n=%lld hq=%d too large", who,
             (long long)n, hq);
  const bool maps = decision != nullptr && avg_attn != nullptr;
  SP_REQUIRE(!maps || workspace_bytes == 0 || (workspace && ((uintptr_t)workspace % 4) == 0), SP_ERR_WORKSPACE,
             "%s: workspace missing or misaligned", who);
  const size_t room = workspace_bytes / sp_attn_pivot_scratch_bytes(n, AS_BS);
  const int slots = !maps ? -1 : room < (size_t)hq ? (int)room : hq;
  const AsArgs a = {(const sp_bf16*)q, (const sp_bf16*)k, (const sp_bf16*)v, mask, decision, (sp_bf16*)out, avg_attn,
                    (float*)workspace, slots, n, q_stride_n, q_stride_h, k_stride_n, k_stride_h, v_stride_n,
                    v_stride_h, hq, hq / hkv, (int)nb, (int)((nb + 63) / 64), decision == nullptr && avg_attn != nullptr,
                    softmax_scale * 1.4426950408889634f};
  static_assert(AS_LDS_BYTES(64) >= AS_MAX_NB * 14 + AS_THREADS * 8 + 16, "");  // rs_lds_bytes(AS_MAX_NB, AS_THREADS)
  const dim3 grid((unsigned)(nb * hq));
  static bool attr_set[64] = {false};  // per device, once (idempotent)
  int dev = 0;
  SP_HIP(hipGetDevice(&dev));
  SP_REQUIRE(dev >= 0 && dev < 64, SP_ERR_UNSUPPORTED, "%s: device index %d", who, dev);
  if (!attr_set[dev]) {
    const void* kernels[4] = {
        (const void*)sp_attn_short_kernel<64, AsArgs>, (const void*)sp_attn_short_kernel<128, AsArgs>,
        (const void*)sp_attn_short_kernel<64, AsPivotArgs>, (const void*)sp_attn_short_kernel<128, AsPivotArgs>};
    for (const void* f : kernels)
      SP_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, AS_LDS_BYTES(128)));
    attr_set[dev] = true;
  }
  auto launch = [&](auto kernel, const auto& args) {
    hipLaunchKernelGGL(kernel, grid, dim3(AS_THREADS), AS_LDS_BYTES(d), (hipStream_t)stream, args);
  };
  auto pick = [&](const auto& args) {
    using Args = std::decay_t<decltype(args)>;
    d == 64 ? launch(sp_attn_short_kernel<64, Args>, args) : launch(sp_attn_short_kernel<128, Args>, args);
  };
  if (pivot != nullptr) {
    AsPivotArgs with;
    static_cast<AsArgs&>(with) = a;
    with.pivot = *pivot;
    pick(with);
  } else {
    pick(a);
  }
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_short_attn_fwd_bf16(const void* q, const void* k, const void* v, int64_t n, int32_t hq, int32_t hkv,
                                      int32_t d, int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                                      int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h, float softmax_scale,
                                      const uint64_t* mask, const int32_t* decision, void* out, float* avg_attn,
                                      void* workspace, size_t workspace_bytes, sp_stream_t stream) {
  return as_launch("sp_short_attn_fwd_bf16", q, k, v, n, hq, hkv, d, q_stride_n, q_stride_h, k_stride_n, k_stride_h, v_stride_n,
                   v_stride_h, softmax_scale, mask, decision, out, avg_attn, workspace, workspace_bytes, nullptr, stream);
}

extern "C" int sp_short_attn_pivot_fwd_bf16(const void* q, const void* k, const void* v, int64_t n, int32_t hq, int32_t hkv,
                                            int32_t d, int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                                            int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h, float softmax_scale,
                                            const uint64_t* mask, const int32_t* decision, void* out, float* avg_attn,
                                            void* workspace, size_t workspace_bytes, const sp_cluster_state* state,
                                            const int32_t* head_cluster, float pattern_threshold, sp_stream_t stream) {
  SP_REQUIRE(decision && avg_attn && head_cluster, SP_ERR_INVALID_ARGUMENT, "sp_short_attn_pivot_fwd_bf16: null pointer");
  const int nb = (int)sp_ceil_div(n, AS_BS);
  int rc = check_state(state, nb, "sp_short_attn_pivot_fwd_bf16");
  if (rc) return rc;
  SP_REQUIRE(hq <= 1024, SP_ERR_UNSUPPORTED, "sp_short_attn_pivot_fwd_bf16: hq=%d unsupported", hq);
  const PivotArgs pivot = {state_by_value(state), head_cluster, decision, hq, nb, (nb + 63) / 64,
                           (long long)sp_thr_lt(pattern_threshold)};
  return as_launch("sp_short_attn_pivot_fwd_bf16", q, k, v, n, hq, hkv, d, q_stride_n, q_stride_h, k_stride_n, k_stride_h, v_stride_n,
                   v_stride_h, softmax_scale, mask, decision, out, avg_attn, workspace, workspace_bytes, state->n_clusters > 0 ? &pivot : nullptr, stream);
}
