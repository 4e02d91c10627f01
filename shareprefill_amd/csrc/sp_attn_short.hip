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
  int rotate;                // grid of (8, hq / 8, rows): heads rotate over the XCDs from row to row
  uint32_t group_mul;        // h / group = (h * group_mul) >> 32, or 0: divide
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
#define AS_MAX_NB 1024    // blocks of a row: a lane holds a word of its mask, its maps fit the tiles' LDS
#define AS_LDS_BYTES(D) (4 * AS_TILE * (D) * 2)
#define AS_NO_MAX (-1.0e30f)         // "no key seen yet": finite, so exp2(S * scale - m) is +inf or 0, never NaN
#define AS_P_TOO_LARGE 0x40004000u   // bf16 pair: exponent >= 128 in either half

typedef __attribute__((address_space(3))) void* as_lds_ptr;

// K and V tiles are [64 keys][D] bf16 in 16-byte chunks, the chunk index XOR-swizzled by the row so that each kind of operand read
// is free of bank conflicts.  The LDS serves 256 bytes a cycle: 16 lanes of a K read (one chunk of 16 consecutive rows), so K's
// chunks are permuted by the row; 32 lanes of a transposing V read (two neighbouring chunks of 8 consecutive rows), so V's pairs
// of chunks are: by the single chunks rows 2i and 2i + 1 met in the same banks, a third of the LDS's active cycles.  Rows of 64
// channels are half a bank cycle long: two rows share a swizzle.
template <int D>
__device__ __forceinline__ int as_swz(int row) {
  return D == 128 ? (row & 15) : ((row >> 1) & 7);
}

template <int D>
__device__ __forceinline__ int as_swz_v(int row) {
  return D == 128 ? 2 * (row & 7) : 2 * ((row >> 1) & 3);
}

__device__ __forceinline__ uint32_t as_pack2(float a, float b) {
  as_floatx2 f;
  f[0] = a;
  f[1] = b;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, as_bf16x2));
}

// One tile by direct memory -> LDS 128-bit loads: a wave-instruction fills 1 KiB (lane i writes chunk base + i and fetches
// whichever chunk belongs there).  A block is a buffer of its own, so that a load is a lane offset made once, a scalar offset
// that only depends on where in the block it stands, and the LDS address in m0; only the tiles of a block that ends with the
// sequence clamp their rows onto the last key (such keys lie behind every stored query).
// What stands between a tile's barrier and its first matrix instruction is in series: with 64-bit addresses made for every load, the
// kept blocks in a list in LDS and V's bank conflicts a step took some hundred cycles of 3300 more (layers, us: 700 tokens 21.9 -> 21.4,
// 3001 105.0 -> 103.7, 6600 at coverage 0.99 255.4 -> 252.9; 64 channels 6177 tokens 120.4 -> 119.0, 20000 at 0.99 514 -> 499).  Of the
// rest the loads' issue is 600; spread over the products, rings of three and four tiles, 16 queries a wave in twice the waves (the LDS's
// reads double: 8 % slower), tiles of 32 keys with a third workgroup on the CU (15 %) and products between the probabilities' arithmetic
// (a wave alone issues no faster) gain nothing.  The two descriptors beside the walk spill 16 scalars of the 128-channel instance to
// vector lanes (42 with the pivots' patterns), of which 6 and 8 are read back per block.
template <int D, bool V>
__device__ __forceinline__ uint32_t as_lane_off(int64_t stride_n, int wave, int lane) {
  constexpr int CHUNKS = D / 8, ROWS = 64 / CHUNKS;  // chunks per row, rows per wave-instruction
  const int row = wave * ROWS + lane / CHUNKS;
  return (uint32_t)(row * (int)stride_n + ((lane % CHUNKS) ^ (V ? as_swz_v<D>(row) : as_swz<D>(row))) * 8) * 2u;
}
template <int D, bool V>
__device__ __forceinline__ void as_issue(__amdgpu_buffer_rsrc_t block, uint32_t row_bytes, int rows /* of the block */, int part,
                                         uint32_t lane_off, uint32_t tile /* LDS offset, the wave's */, int wave, int lane) {
  constexpr int CHUNKS = D / 8, ROWS = 64 / CHUNKS;
  constexpr int STEP = ROWS * AS_WAVES, ITS = AS_TILE / STEP;  // rows per instruction of all waves (a multiple of the swizzle's period)
  if (rows == AS_BS) {
#pragma unroll
    for (int it = 0; it < ITS; ++it)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(block, (as_lds_ptr)(uintptr_t)(tile + it * AS_WAVES * 1024), 16, (int)lane_off,
                                               (int)((part * ITS + it) * (STEP * row_bytes)), 0, 0);
  } else {
    int ln = lane;
    asm volatile("" : "+v"(ln));  // (keeps this rare path's lane arithmetic out of the tile loop)
#pragma unroll 1
    for (int it = 0; it < ITS; ++it) {
      const int in_tile = (it * AS_WAVES + wave) * ROWS + ln / CHUNKS;
      const int row = part * AS_TILE + in_tile < rows ? part * AS_TILE + in_tile : rows - 1;
      const int chunk = (ln % CHUNKS) ^ (V ? as_swz_v<D>(in_tile) : as_swz<D>(in_tile));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(block, (as_lds_ptr)(uintptr_t)(tile + it * AS_WAVES * 1024), 16,
                                               (int)((uint32_t)row * row_bytes + 16u * chunk), 0, 0, 0);
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
// RAISE: the products go before the other workgroups' softmax and loads on the SIMD (as_raise).
template <int D, typename Args, bool RAISE>
__device__ __forceinline__ void as_row(const Args a) {
  constexpr int QT = 2;                             // 16-query tiles per wave
  constexpr int KS = D / 32, CT = D / 16;           // channel steps of S, channel tiles of O
  constexpr int WAVES = AS_WAVES, THREADS = AS_THREADS, WQ = 16 * QT;
  constexpr int TILE_BYTES = AS_TILE * D * 2;
  extern __shared__ __attribute__((aligned(1024))) char lds[];  // [buffer][K | V]
  const int t = threadIdx.x, lane = t & 63, lq = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // query band
  const uint32_t lds_base = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)lds;
  // Head and rank of the row (0 = the last, heaviest one); the grid is (8, hq / 8, rows) or (hq, 1, rows).  An integer division
  // costs a wave that has its SIMD to itself some 300 cycles in front of its first load, hence the grid's form and the multiplier.
  const int rr = blockIdx.z, r = a.nb - 1 - rr;
  const int h = a.rotate ? ((blockIdx.x + rr) & 7) * gridDim.y + blockIdx.y : blockIdx.x;
  const int kvh = a.group_mul ? (int)__umulhi((uint32_t)h, a.group_mul) : h / a.group;
  const sp_bf16* kh = a.k + (int64_t)kvh * a.sk_h;
  const sp_bf16* vh = a.v + (int64_t)kvh * a.sv_h;

  const int dec = a.slots >= 0 ? a.decision[h] : 0;  // (asked for up here: its way from memory passes under the mask's)

  const uint32_t k_lane = as_lane_off<D, false>(a.sk_n, wave, lane), v_lane = as_lane_off<D, true>(a.sv_n, wave, lane);
  const uint32_t k_row = (uint32_t)a.sk_n * 2u, v_row = (uint32_t)a.sv_n * 2u;  // bytes
  const int last_rows = (int)(a.n - (int64_t)(a.nb - 1) * AS_BS);
  __amdgpu_buffer_rsrc_t k_blk, v_blk;  // the block whose tiles are being fetched
  int blk_rows = 0;
  auto open_block = [&](int c) {
    blk_rows = c == a.nb - 1 ? last_rows : AS_BS;
    auto block = [&](const sp_bf16* x, uint32_t row_bytes) {
      const char* p = (const char*)x + (uint64_t)(uint32_t)c * (uint64_t)(AS_BS * row_bytes);
      return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)((uint32_t)(blk_rows - 1) * row_bytes + 2u * D), 0x00027000);
    };
    k_blk = block(kh, k_row);
    v_blk = block(vh, v_row);
  };
  const uint32_t lds_wave = lds_base + wave * 1024;
  auto issue = [&](int part, int buf) {
    const uint32_t at = lds_wave + (uint32_t)(buf * 2 * TILE_BYTES);
    as_issue<D, false>(k_blk, k_row, blk_rows, part, k_lane, at, wave, lane);
    as_issue<D, true>(v_blk, v_row, blk_rows, part, v_lane, at + TILE_BYTES, wave, lane);
  };
  // The row's mask, one word per lane; the kept blocks are walked bit by bit in scalar registers.  The first tile of block 0, which
  // nearly every row keeps, is asked for before the word is looked at (a row that does not keep it fetches its own into the same place:
  // loads land in order); with 64 channels before the word is there: us, with its trimming in front / behind the tile, 300 tokens 10.4 /
  // 10.2, 700 17.9 / 17.5, 1024 22.9 / 22.4.  With 128 the trimming is a branch in front of the tile, which waits for the word: without
  // the wait nothing is won (the tile's loads take 600 cycles to issue), and the code of the other form runs 0.5 to 1 % slower, with the wait
  // or without (700 23.3 / 23.5, 1024 31.1 / 31.3).
  const uint64_t* const mask_row = a.mask + ((int64_t)h * a.nb + r) * a.nbw;
  const int last_w = r >> 6;
  uint64_t lane_word = 0;
  if (lane <= last_w) lane_word = mask_row[lane];
  if constexpr (D == 128)
    if (lane == last_w && (r & 63) != 63) lane_word &= (2ull << (r & 63)) - 1ull;
  open_block(0);
  issue(0, 0);
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
  if constexpr (D == 64) lane_word &= lane == last_w ? ~0ull >> (63 - (r & 63)) : ~0ull;  // (no branch: one would wait in front of the loads)
  const uint32_t word_lo = (uint32_t)lane_word, word_hi = (uint32_t)(lane_word >> 32);
  auto word = [&](int w) {
    return (uint64_t)(uint32_t)__builtin_amdgcn_readlane(word_lo, w) | (uint64_t)(uint32_t)__builtin_amdgcn_readlane(word_hi, w) << 32;
  };
  int n_blk = 0;
  for (int w = 0; w <= last_w; ++w) n_blk += __builtin_popcountll(word(w));
  struct Walk {
    uint64_t x;
    int w;
  };
  auto next_block = [&](Walk& k) {  // (there is one)
    while (k.x == 0ull) k.x = word(++k.w);
    const int c = k.w * 64 + __builtin_ctzll(k.x);
    k.x &= k.x - 1ull;
    return c;
  };
  Walk walk = {word(0), 0};
  int c = 0;
  if (n_blk > 0) {
    c = next_block(walk);
    if (c != 0) {
      open_block(c);
      issue(0, 0);
    }
  } else {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // (vmcnt(0): no load may outlive the wave)
  }

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
  const int voff = vrow * (D * 2) + 8 * (lq & 1), vswz = as_swz_v<D>(vrow), vhalf = (lq >> 1) & 1;

  int c_next = 0;
  // One step per tile, two per block, a buffer for either; the block behind is opened when its first tile is asked for.
  for (int st = 0; st < 2 * n_blk; ++st) {
    const int half = st & 1, buf = half;
    // this wave's loads of the tile have landed, and everybody's; the other buffer's readers are done
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (half == 0) {
      issue(1, 1);
    } else if (st + 1 < 2 * n_blk) {
      c_next = next_block(walk);
      open_block(c_next);
      issue(0, 0);
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
        if constexpr (RAISE) __builtin_amdgcn_s_setprio(1);
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
      if constexpr (RAISE) __builtin_amdgcn_s_setprio(0);
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
      if constexpr (RAISE) __builtin_amdgcn_s_setprio(1);
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
    if constexpr (RAISE) __builtin_amdgcn_s_setprio(0);
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
    // (lane groups 2i and 2i + 1 trade halves of two neighbouring channel tiles: 16 bytes a store, 64 contiguous ones a row)
    sp_bf16* dst = a.out + ((qrow + 16 * qt) * a.hq + h) * D + 16 * (g & 1) + 8 * (g >> 1);
#pragma unroll
    for (int ct = 0; ct < CT; ct += 2) {
      uint32_t w[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        w[u][0] = as_pack2(o[ct + u][qt][0] * inv_l[qt], o[ct + u][qt][1] * inv_l[qt]);
        w[u][1] = as_pack2(o[ct + u][qt][2] * inv_l[qt], o[ct + u][qt][3] * inv_l[qt]);
      }
      const auto lo = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
      const auto hi = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
      if (qrow + 16 * qt < a.n) *reinterpret_cast<uint4*>(dst + ct * 16) = make_uint4(lo[0], hi[0], lo[1], hi[1]);
    }
  }
  if (a.zero_maps)
    for (int i = t; i < a.nb; i += THREADS) a.avg_attn[((int64_t)h * a.nb + r) * a.nb + i] = 0.f;
  if (!pivot) return;  // (uniform)
  if (pu == nullptr) {  // more pivots than the caller made room for: no map, and visibly so
    for (int i = t; i <= r; i += THREADS)
      if ((mask_row[i >> 6] >> (i & 63)) & 1ull) a.avg_attn[((int64_t)h * a.nb + r) * a.nb + i] = NAN;
    return;
  }
  // pivot head: avg[r][c] = mean over the block's valid queries of exp2(u - m[q]) / l[q].  A wave
  // reads back its own sums (its own stores), folds its queries, and the waves meet in LDS.
  float* const part = reinterpret_cast<float*>(lds);  // [column][wave]
  __syncthreads();                                    // LDS is free, the stores of pu have left
  walk = {word(0), 0};
  for (int i = 0; i < n_blk; ++i) {
    const int c = next_block(walk);
    float x = 0.f;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
      if (qrow + 16 * qt < a.n) {
        x += __builtin_amdgcn_exp2f(pu[(int64_t)c * AS_BS + q_off + 16 * qt] - m[qt]) * inv_l[qt];
      }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) x += __shfl_xor(x, off, SP_WAVE);
    if (lane == 0) part[c * WAVES + wave] = x;
  }
  __syncthreads();
  const int64_t rem = a.n - (int64_t)r * AS_BS;
  const float inv_q = 1.0f / (float)(rem < AS_BS ? (int)rem : AS_BS);
  for (int i = t; i <= r; i += THREADS) {
    if (!((mask_row[i >> 6] >> (i & 63)) & 1ull)) continue;
    float x = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) x += part[i * WAVES + w];
    a.avg_attn[((int64_t)h * a.nb + r) * a.nb + i] = x * inv_q;
  }
  if constexpr (std::is_same<Args, AsPivotArgs>::value) {
    __shared__ PivotRowShared pivot_sh;
    __syncthreads();  // the row is written, LDS is free
    pivot_row<THREADS>(a.pivot, pivot_sh, lds, a.avg_attn, r, h);
  }
}

template <int D, typename Args>
__global__ __launch_bounds__(AS_THREADS, 2) void sp_attn_short_kernel(Args a) {
  as_row<D, Args, true>(a);
}
template <int D, typename Args>
__global__ __launch_bounds__(AS_THREADS, 2) void sp_attn_short_level_kernel(Args a) {
  as_row<D, Args, false>(a);
}

// ---- host ---------------------------------------------------------------------------------------------
// Whether a wave raises its priority around S and P . V, by the rows of the launch.  Where rows wait for a place it lets a CU's workgroups
// take turns with the matrix core (attention, us, without / with: every block kept, 32 / 8 heads of 128 3001 tokens 98.7 / 92.1, 40 / 8 2432
// 82.9 / 76.3; 64 channels 4500 125 / 110, 14 / 2 9984 234 / 213; half of them, 28 / 4 of 128 4500 117 / 108).  Where every row is resident
// from the start, or nearly, the long rows wait for the short ones: 28 / 4 3200 tokens (700 rows) 90.8 / 95.2, 32 / 8 2048 58.6 / 60.1; 64
// channels 3001 62.5 / 65.6, 14 / 2 6656 (728 rows) 119 / 128, 16128 of 8 / 2 (1008) 304 / 320.  With 128 channels there are 512 places and 720 to
// 760 rows are even, with 64 768 and 1008 to 1064: a third beyond is taken in by the rows that end first.  A row alone on its CU has nobody to go before; the instance with the
// priority is 0.3 to 1 % ahead there.  (Around S alone it does nothing, around P . V alone half; behind a condition in the kernel the
// branches cost what it gives.)
static bool as_raise(int d, int64_t rows) { return rows <= 256 || rows > (d == 64 ? 1024 : 736); }

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
// (These lines hold for any layer; where none of its heads can be elected see sp_short_attn_max_steady_tokens.)
// 64 channels, where the persistent kernel computes on zero-padded tiles (padding counted), 32 / 8 heads: 0.65 8192 148 / 254, 32768
// 448 / 810, 49152 715 / 1244; 0.95 143 / 253, 583 / 907, 1268 / 1692; 0.99 147 / 261, 1177 / 1422, 2970 / 3100; every block kept 311 / 409,
// 4920 / 5135, 10775 / 11010; 14 / 2 heads 0.95 32768 333 / 462, every block 2062 / 2198.  The line is where both were once even without
// the padding; layers with pivots beyond it are slower here at low coverage (below), and each pivot's block sums take 16.8 MB there.
extern "C" int64_t sp_short_attn_max_tokens(int32_t d) {
  return d == 64 ? 32768 : 6656;
}
// The same where no pivot is elected, by the coverage the masks are made at (share of the softmax mass: what the density grows with).
// A pivot's rows keep every block, which the persistent kernel's rows of two share out better: whole passes of an electing layer and a
// steady one, us here / there, 32 / 8 heads of 128 channels 8192 tokens at 0.95 709 / 665, 9000 at 0.9 775 / 681; 64 channels 40000 at 0.95
// 4462 / 4666, 100000 at 0.65 19754 / 17016.
// Query-aware heads keep far more blocks at the same coverage (0.86 of them at 0.9, 0.53 at 0.65 where vertical-slash heads keep 0.2 to
// 0.3) and are known on the device alone, so a line lies where a layer of nothing else is even.  Steady layers, 128 channels, 32 / 8 and
// 28 / 4 heads:
//   query-aware     0.9 7424 474 / 484, 438 / 474, 7680 506 / 505, 457 / 496, 8192 562 / 552, 492 / 531, 10240 807 / 783, 719 / 701;
//                   0.65 10241 593 / 603, 536 / 551, 11264 672 / 678, 602 / 616, 12288 759 / 749, 661 / 673, 16384 1201 / 1157, 1056 / 1031;
//   vertical-slash  0.9 7000 181 / 198, 156 / 177, 10240 248 / 266, 229 / 248; 0.65 8192 200 / 209, 182 / 202, 16384 354 / 375, 321 / 330;
//   at 0.95 8192 237 / 249, 222 / 232, but 1162 / 1140 of a decoder layer's half with query-aware heads there: not taken.
// A minimum budget sets a floor of its own: of a quarter of 10241 tokens at 0.65 437 / 432, of half of 8192 426 / 414, of half of 16384 1518 /
// 1401, of a sixth 344 / 353, 383 / 387 at 11264 (that much is asked of the caller).
// 64 channels, 32 / 8 and 14 / 2 heads: vertical-slash 0.65 36000 546 / 961, 291 / 479, 131072 1965 / 3287, 941 / 1497; 0.95 36000 745 / 1113,
// 402 / 576, 131072 11717 / 12320, 5784 / 5969; 0.99 65536 5500 / 5627, 2406 / 2780, 90001 11976 / 11675, 5534 / 5696; query-aware 0.65 131072
// 33557 / 34114, 0.9 65536 15790 / 16352, 131072 60853 / 60756, 27383 / 27736, 0.95 131072 67357 / 67303, 30320 / 30424, 0.99 65536 18809 / 19347;
// a minimum budget of half of 131072 54434 / 54978.
extern "C" int64_t sp_short_attn_max_steady_tokens(int32_t d, float pattern_threshold) {
  if (d == 64) return pattern_threshold <= 0.951f ? AS_MAX_NB * AS_BS : pattern_threshold <= 0.991f ? 65536 : sp_short_attn_max_tokens(d);
  return pattern_threshold <= 0.651f ? 11264 : pattern_threshold <= 0.901f ? 7680 : sp_short_attn_max_tokens(d);
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
  const bool rotate = hq % 8 == 0 && hq / 8 <= 65535;
  // (h * group_mul) >> 32 is h / group while h * group < 2^32
  const uint32_t group_mul = hq < 65536 && hq > hkv ? (uint32_t)((1ull << 32) / (uint32_t)(hq / hkv)) + 1u : 0u;
  const AsArgs a = {(const sp_bf16*)q, (const sp_bf16*)k, (const sp_bf16*)v, mask, decision, (sp_bf16*)out, avg_attn,
                    (float*)workspace, slots, n, q_stride_n, q_stride_h, k_stride_n, k_stride_h, v_stride_n,
                    v_stride_h, hq, hq / hkv, (int)nb, (int)((nb + 63) / 64), rotate, group_mul, decision == nullptr && avg_attn != nullptr,
                    softmax_scale * 1.4426950408889634f};
  static_assert(AS_LDS_BYTES(64) >= AS_MAX_NB * 14 + AS_THREADS * 8 + 16, "");  // rs_lds_bytes(AS_MAX_NB, AS_THREADS)
  const dim3 grid(rotate ? 8 : (unsigned)hq, rotate ? (unsigned)(hq / 8) : 1, (unsigned)nb);
  static bool attr_set[64] = {false};  // per device, once (idempotent)
  int dev = 0;
  SP_HIP(hipGetDevice(&dev));
  SP_REQUIRE(dev >= 0 && dev < 64, SP_ERR_UNSUPPORTED, "%s: device index %d", who, dev);
  if (!attr_set[dev]) {
    const void* kernels[8] = {
        (const void*)sp_attn_short_kernel<64, AsArgs>, (const void*)sp_attn_short_kernel<128, AsArgs>,
        (const void*)sp_attn_short_kernel<64, AsPivotArgs>, (const void*)sp_attn_short_kernel<128, AsPivotArgs>,
        (const void*)sp_attn_short_level_kernel<64, AsArgs>, (const void*)sp_attn_short_level_kernel<128, AsArgs>,
        (const void*)sp_attn_short_level_kernel<64, AsPivotArgs>, (const void*)sp_attn_short_level_kernel<128, AsPivotArgs>};
    for (const void* f : kernels)
      SP_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, AS_LDS_BYTES(128)));
    attr_set[dev] = true;
  }
  auto launch = [&](auto kernel, const auto& args) {
    hipLaunchKernelGGL(kernel, grid, dim3(AS_THREADS), AS_LDS_BYTES(d), (hipStream_t)stream, args);
  };
  auto pick = [&](const auto& args) {
    using Args = std::decay_t<decltype(args)>;
    if (as_raise(d, nb * hq))
      d == 64 ? launch(sp_attn_short_kernel<64, Args>, args) : launch(sp_attn_short_kernel<128, Args>, args);
    else
      d == 64 ? launch(sp_attn_short_level_kernel<64, Args>, args) : launch(sp_attn_short_level_kernel<128, Args>, args);
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
