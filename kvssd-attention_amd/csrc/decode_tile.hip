// Tiled matrix-core decode kernel for the shapes the fp16-weight kernels do
// not take: head_dim 64, 128 or 256 (and 96 with INT4 codes), up to 16 groups
// per head, blocks of a multiple of 16 tokens, any GQA ratio.  fp32-grade
// arithmetic, as the general kernel it stands in for: codes enter the matrix
// core as the exact integers c - mid, the query and the softmax weights as sums
// of fp16 parts, and every scale multiplies in fp32.
//
// Semantics: ReferenceAttentionBackend.run (src/kvssd/backends/reference.py:22-50)
// and csrc/fused_decode.cu:12-90 (element addressing :50-56, GQA map :34).
//
// Measured against the vector kernel on the same arrays (fp16 queries, split
// and merge): 32K tokens in 32-token blocks, 8 kv heads, GQA 4, head_dim 128
// 372 -> 16.3 us (37.7 MB of codes and scales); 24K tokens, 4 kv heads, GQA 6,
// head_dim 256, groups of 64, bf16 222 -> 21.3 us; 16K tokens, head_dim 64 (the
// kernel alone) 60 -> 10 us.  Output error against float64 (rms over 192 to 1,600
// heads of a shape): INT4 0.53-0.89 times the vector kernel's, INT2 0.82-1.08.
// What bounds it now: a workgroup's start and end (argument, table and query
// round trips, the waves' merge), and in between the VALU: of the 32K-token
// decode above, 1,180 instructions a wave and 4 waves a SIMD, 7.9 us of issue
// (the matrix cores are busy for 1.3 us); 1M tokens in 32-token blocks, 128
// passes a SIMD, come in at 3.7 TB/s.
//
// Work split.  A workgroup of 4 waves owns one kv head, up to 16 / Gp of its
// query heads (Gp: groups per head, rounded up to a power of two) and one
// split's run of blocks, taken as one sequence of token slots: wave w works on
// slots 64 w, 64 w + 256, ... 64 at a time, wherever block ends fall.  The
// waves' states meet in LDS at the end, one partial per query head.
//
// QK (v_mfma_f32_16x16x32_f16): A = query, row r = (head, group) holding that
//   head masked to that group, scaled by a power of two; B = the codes of 16
//   tokens, lane (li, lq) the lq-th quarter of token li's row.  Lane (li, lq)
//   ends with rows 4 lq .. 4 lq + 3 of token li, applies each row's K scale and
//   adds the groups of a head: in registers up to 4 groups, across lane rows
//   beyond.
// Softmax: running (m, l) in log2 units per lane row and head, m a whole number,
//   so that every rescaling is exact.  The weights W = 2^(s - m) scale_v 2^k carry
//   a whole exponent k per row (head, group) that follows the row's largest, so
//   that one lies in [2^12, 2^13) whatever the scales, and W, as two fp16 parts,
//   is off by at most 2^-23 of itself or 2^-37 of the row's largest.  (One k for a
//   head's groups left a group of V scales 2^-18 times the head's largest with 8
//   times the vector kernel's error.)
// PV: A = W (rows (head, group), K = 32 tokens, hi and lo parts through LDS),
//   B = V codes from a nibble transpose read (ds_read_b64_tr_b4) of the rows
//   staged in LDS.  Of a column (dim), the rows of its own group count.
// Token <-> K slot of PV, shared by both operands: K step kk, lane group q,
//   slot s -> token 16 (s & 3) + 4 q + 2 kk + (s >> 2) of the wave's 64.
#include "staged_ops.hpp"

namespace kvssd {
namespace {

constexpr int kTileWaves = 4;
constexpr int kTileThreads = kWave * kTileWaves;
constexpr int kChunkTok = 64;               // token slots of a wave's pass
constexpr int kWRowBytes = 2 * kChunkTok + 16;  // one W row: 64 fp16 slots and a pad

// Kernel arguments beyond the preloaded ones (query, pk, pv, sk, sv and four
// dwords).  The first pass's addresses wait for a fetch of these: the block
// table and the constants that find block ends are among them.
struct TileTail {
  const int32_t* table;
  const int32_t* valid;
  float* part_o;
  float* part_ml;
  float* split_note;                   // where to note `splits`, or nullptr
  int query_heads, num_blocks, gq, heads_per_wg;
  int head_chunks, query_dtype, splits;
  uint32_t chunk_magic;                // ceil(2^32 / head_chunks), head_chunks > 1
  uint32_t bt_magic;                   // ceil(2^20 / block_tokens), block_tokens < 256
  uint32_t group_magic;                // ceil(2^16 / group_size)
  float scale_log2;                    // sm_scale * log2(e)
};
// shape argument: kv_heads in bits 0-15, groups per head in 16-20, log2 of
// their count rounded up in 21-23, bit 24 set when there is a block table
inline uint32_t pack_shape(int kv_heads, int groups, int group_shift, bool has_table) {
  return static_cast<uint32_t>(kv_heads) | (static_cast<uint32_t>(groups) << 16) |
         (static_cast<uint32_t>(group_shift) << 21) | (has_table ? kHasTable : 0u);
}

// workgroups resident on a CU (4 waves each, one per SIMD), by registers and,
// for head_dim 256, by LDS: what the register budget and the split plan count on
// (of INT2, one-part, head_dim 256 with four or more groups, 158 registers and
// 43 KB, three would fit)
constexpr int tile_workgroups_per_cu(int head_dim, int hs, int parts) {
  return parts == 1 && (head_dim == 64 || (head_dim == 128 && hs == 1)) ? 4 : head_dim <= 128 ? 3 : 2;
}

struct TileParams {
  const uint8_t* pk;
  const uint8_t* pv;
  const uint16_t* sk;
  const uint16_t* sv;
  int kv_heads, groups, group_shift;
  uint32_t block_tokens;
  bool has_table;
};

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// A code c at bit b of an fp16 whose exponent field is that of 1024 reads as
// 1024 + 2^b c; one packed fp16 FMA turns the pair into c - mid, exactly.
__device__ __forceinline__ uint32_t magic1024(uint32_t x, uint32_t mask) {
  return __builtin_amdgcn_bitop3_b32(x, mask, 0x64006400u, 0xEA);  // (x & mask) | 1024-pairs
}
template <int SHIFT, int MID>
__device__ __forceinline__ uint32_t centre(uint32_t v) {
  const half2_t h = __builtin_bit_cast(half2_t, v);
  const _Float16 f = static_cast<_Float16>(1.0f / (1 << SHIFT));
  const _Float16 o = static_cast<_Float16>(-(1024.0f / (1 << SHIFT)) - MID);
  if constexpr (SHIFT == 0) return __builtin_bit_cast(uint32_t, h + half2_t{o, o});
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(h, half2_t{f, f}, half2_t{o, o}));
}
template <int SHIFT>
__device__ __forceinline__ uint32_t pair4(uint32_t x, uint32_t opaque_zero) {
  return centre<SHIFT, 8>(magic1024(x, (0x000F000Fu << SHIFT) | opaque_zero));
}
template <int SHIFT>
__device__ __forceinline__ uint32_t pair2(uint32_t x, uint32_t opaque_zero) {
  return centre<SHIFT, 2>(magic1024(x, (0x00030003u << SHIFT) | opaque_zero));
}

// INT4 word (nibbles n0..n7): slot s holds n_i - 8, i = (s >> 1) + 4 (s & 1)
__device__ __forceinline__ u32x4 ints4(uint32_t x, uint32_t oz) {
  const uint32_t y = x >> 8;
  return u32x4{pair4<0>(x, oz), pair4<4>(x, oz), pair4<0>(y, oz), pair4<4>(y, oz)};
}
// INT2 word (codes c0..c15), half o: slot s holds c_i - 2, i = 4 o + (s >> 1) + 8 (s & 1)
__device__ __forceinline__ u32x4 ints2(uint32_t x, int o, uint32_t oz) {
  if (o == 0) return u32x4{pair2<0>(x, oz), pair2<2>(x, oz), pair2<4>(x, oz), pair2<6>(x, oz)};
  const uint32_t y = x >> 8;
  return u32x4{pair2<0>(y, oz), pair2<2>(y, oz), pair2<4>(y, oz), pair2<6>(y, oz)};
}
// INT2 transpose-read word (nibble i: the codes of dims 2j and 2j + 1 of token
// row i): slot s holds the even (par 0) or odd (par 1) code of row
// (s >> 1) + 4 (s & 1), less 2
__device__ __forceinline__ u32x4 ints2_tr(uint32_t x, int par, uint32_t oz) {
  const uint32_t y = x >> 8;
  if (par == 0) return u32x4{pair2<0>(x, oz), pair2<4>(x, oz), pair2<0>(y, oz), pair2<4>(y, oz)};
  return u32x4{pair2<2>(x, oz), pair2<6>(x, oz), pair2<2>(y, oz), pair2<6>(y, oz)};
}

// position of dim d in a query row laid out by K slots: lane group q's quarter
// of the row at q D / 4, its K step m at 8 m, slot s
template <int BITS, int D>
__device__ __forceinline__ int query_slot(int d) {
  const int q = d / (D / 4), r = d % (D / 4);
  if (BITS == 4) return q * (D / 4) + (r & ~7) + 2 * (r & 3) + ((r >> 2) & 1);
  return q * (D / 4) + (r & ~15) + 8 * ((r >> 2) & 1) + 2 * (r & 3) + ((r >> 3) & 1);
}

// x = hi + lo, both fp16 (pairs).  An infinite x leaves a finite lo part
// (inf - inf is NaN, which fmaxf drops), so that x c stays infinite.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t& hi, uint32_t& lo) {
  hi = __builtin_bit_cast(uint32_t, half2_t{static_cast<_Float16>(x0), static_cast<_Float16>(x1)});
  // the remainders are taken from these very bits: where x is a product the
  // compiler may otherwise round it to fp16 a second way for the subtraction,
  // and a value near a rounding tie then loses a whole fp16 step
  asm("" : "+v"(hi));
  const half2_t l = {static_cast<_Float16>(fmaxf(x0 - half_lo(hi), -65504.0f)),
                     static_cast<_Float16>(fmaxf(x1 - half_hi(hi), -65504.0f))};
  lo = __builtin_bit_cast(uint32_t, l);
}

template <int BITS, int D, int HS, int QSPLIT = 1>
struct TileGeo {
  static constexpr int PD = D * BITS / 8;        // packed bytes of a row
  static constexpr int KW = PD / 16;             // dwords of a quarter row
  static constexpr int KS = D / 32;              // QK K steps
  static constexpr int NTR = PD / 8;             // transpose reads (8 bytes of a row each)
  static constexpr int NPAR = BITS == 4 ? 1 : 2; // output tiles per transpose read
  static constexpr int NT = NTR * NPAR;          // 16-column output tiles
  static constexpr int NG = 4 / HS;              // groups per head held by a lane
  // V rows in LDS: 8-byte unit n of token t at t VS + 8 (n ^ v_phi(t)).  A
  // transpose read takes one unit of tokens 16 a + c, a < 4, of 8 values of c
  // per 32 lanes; the swizzle (a pad where the row is not a power of two)
  // spreads them over the banks
  static constexpr bool V_XOR = (PD & (PD - 1)) == 0;
  static constexpr int VS = V_XOR ? PD : PD + ((PD / 8) % 2 == 0 ? 8 : 0);
  static constexpr int V_BYTES = kChunkTok * VS;
  static constexpr int WAVE_BYTES = V_BYTES + 2 * 16 * kWRowBytes;
  static constexpr int HEADS = 4 * HS;           // most query heads of a workgroup
  static constexpr int X_BYTES = kTileWaves * HEADS * D * 4;   // the waves' outputs at the end
  static constexpr int Q_ROW = 2 * D + 16;       // one query operand row and a pad
  static constexpr int Q_BYTES = QSPLIT * 16 * Q_ROW;
  static constexpr int Q_OFF = WAVE_BYTES * kTileWaves;
  static constexpr int LDS = Q_OFF + Q_BYTES > X_BYTES ? Q_OFF + Q_BYTES : X_BYTES;
  static_assert(WAVE_BYTES % 16 == 0 && V_BYTES % 16 == 0, "aligned LDS regions");
};

// Registers of one pass's loads: 4 tiles of 16 tokens, a quarter row and the
// scales of this lane's groups (fp16 pairs) each.
template <int BITS, int D, int HS>
struct TileLoads {
  static constexpr int SW = HS == 1 ? 2 : 1;
  uint32_t k[4][TileGeo<BITS, D, HS>::KW], v[4][TileGeo<BITS, D, HS>::KW];
  uint32_t sk[4][SW], sv[4][SW];
  uint32_t ok;  // bit tau: tile tau's token li is a valid one
};
__device__ __forceinline__ uint16_t scale_bits(const uint32_t* w, int i) {
  return static_cast<uint16_t>(i & 1 ? w[i >> 1] >> 16 : w[i >> 1] & 0xFFFFu);
}

template <int PD>
__device__ __forceinline__ int v_phi(int t) {
  if constexpr (PD == 128) return ((t >> 1) & 3) | (((t >> 4) & 3) << 2);
  else if constexpr (PD == 64) return ((t >> 2) & 1) | (((t >> 4) & 3) << 1);
  else if constexpr (PD == 32) return (t >> 4) & 3;
  else if constexpr (PD == 16) return (t >> 4) & 1;
  else return 0;
}

template <int BYTES>
__device__ __forceinline__ void load_bytes(void* dst, const void* src) {
  constexpr int kAlign = BYTES % 16 == 0 ? 16 : BYTES % 8 == 0 ? 8 : BYTES % 4 == 0 ? 4 : 2;
  __builtin_memcpy(dst, __builtin_assume_aligned(src, kAlign), BYTES);
}

// head_dim 96: rows past the last of 3, 6 or 12 groups re-read the scales of
// groups before; their K scales count as zeros (their sums are zeros, and 0
// times an infinite scale would not be)
template <int D, int HS>
constexpr bool kPadRows = D == 96 && HS == 1;

// the scales of a lane's NG groups, from group gbase on
template <int NG, bool NARROW>
__device__ __forceinline__ void load_scales(uint32_t* dst, const uint16_t* row, int gbase, int groups, bool wide) {
  if constexpr (NG == 1) {
    dst[0] = row[0];
  } else if (!NARROW || wide) {
    load_bytes<2 * NG>(dst, row + gbase);
  } else {
    uint16_t h[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) h[i] = row[min(gbase + i, groups - 1)];
#pragma unroll
    for (int i = 0; i < NG; i += 2) dst[i >> 1] = h[i] | (static_cast<uint32_t>(h[i + 1]) << 16);
  }
}

// a uniform index read through the scalar cache (the kernel never writes these arrays)
__device__ __forceinline__ int scalar_read(const int32_t* a, int i) {
  typedef const __attribute__((address_space(4))) int32_t* const_ptr;
  return ((const_ptr)a)[__builtin_amdgcn_readfirstlane(i)];
}

// The loads of the pass that starts base_off slots into block base_unit of the
// split (its blocks u0 .. u0 + n_units - 1, taken as one sequence of slots).
// Blocks hold whole 16-token tiles, so block id, row and valid count of a tile
// are scalars, read through the scalar cache: their waits never hold up a wave
// behind its code loads.  Tiles past the end read the last block again; tokens
// past their block's valid count read their own (stale) row.
template <int BITS, int D, int HS>
__device__ __forceinline__ void load_pass(TileLoads<BITS, D, HS>& ld, const TileParams& p, const TileTail& r, int u0,
                                          int n_units, int base_unit, uint32_t base_off, int kvh, int li, int lq,
                                          int gbase, bool wide_scales) {
  using G = TileGeo<BITS, D, HS>;
  const uint32_t bt = p.block_tokens;
  int blk[4], count[4];
  uint32_t off[4], live[4];  // live: all ones, 0 for a tile past the end (masks, so that no load sits under a branch)
  // a tile's block and offset: base_off < bt, so with blocks of 256 or more at
  // most one block end is within reach (bt_magic is 0); below, x < 512 and the
  // magic quotient is exact
  const uint32_t one_end = bt >= 256u ? bt : 0xFFFFFFFFu;
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) {
    const uint32_t x = base_off + static_cast<uint32_t>(16 * tau);
    const uint32_t q = ((x * r.bt_magic) >> 20) + (x >= one_end ? 1u : 0u);
    const int u = base_unit + static_cast<int>(q);
    live[tau] = u < n_units ? 0xFFFFFFFFu : 0u;
    off[tau] = x - q * bt;
    blk[tau] = u0 + min(u, n_units - 1);
  }
  if (p.has_table) {
    int id[4];
#pragma unroll
    for (int tau = 0; tau < 4; ++tau) id[tau] = scalar_read(r.table, blk[tau]);
#pragma unroll
    for (int tau = 0; tau < 4; ++tau) {  // ids are checked on the host; never read out of bounds
      const uint32_t ok = static_cast<uint32_t>(id[tau]) < static_cast<uint32_t>(r.num_blocks) ? 0xFFFFFFFFu : 0u;
      live[tau] &= ok;
      blk[tau] = static_cast<int>(static_cast<uint32_t>(id[tau]) & ok);
    }
  }
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) count[tau] = scalar_read(r.valid, blk[tau]);
  // a lane's offsets within a tile: token li's row, quarter lq
  const uint32_t ko = static_cast<uint32_t>(li * p.kv_heads * G::PD + 4 * G::KW * lq);
  const uint32_t so = static_cast<uint32_t>(2 * li * p.kv_heads * p.groups);
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) {
    // (rows of the batch below 2^31: checked on the host)
    const uint32_t row = (static_cast<uint32_t>(blk[tau]) * bt + off[tau]) * static_cast<uint32_t>(p.kv_heads) +
                         static_cast<uint32_t>(kvh);
    load_bytes<4 * G::KW>(ld.k[tau], p.pk + static_cast<size_t>(row) * G::PD + ko);
    load_bytes<4 * G::KW>(ld.v[tau], p.pv + static_cast<size_t>(row) * G::PD + ko);
    const size_t srow = static_cast<size_t>(row) * static_cast<uint32_t>(p.groups);
    const uint8_t* skb = reinterpret_cast<const uint8_t*>(p.sk + srow) + so;
    const uint8_t* svb = reinterpret_cast<const uint8_t*>(p.sv + srow) + so;
    load_scales<G::NG, D == 96>(ld.sk[tau], reinterpret_cast<const uint16_t*>(skb), gbase, p.groups, wide_scales);
    load_scales<G::NG, D == 96>(ld.sv[tau], reinterpret_cast<const uint16_t*>(svb), gbase, p.groups, wide_scales);
  }
  ld.ok = 0u;
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) {
    const int left = (clamp_valid(count[tau], static_cast<int>(bt)) - static_cast<int>(off[tau])) &
                     static_cast<int>(live[tau]);
    ld.ok |= li < left ? 1u << tau : 0u;
  }
}

// Per lane row and head (m, l); per row the exponent k that its accumulators carry
template <int NT, int HS>
struct TileState {
  float m[HS], l[HS];
  int k[4];
  f32x4 acc[NT];
};
constexpr int kMostExponent = 123;  // 2^k and 2^-k are normal numbers; weights below 2^-110 lose bits
constexpr int kFar = -1000;         // an exponent that ldexpf turns any finite value into 0 by

// m - to as a whole number, m <= to whole (kFar where they are infinite)
__device__ __forceinline__ int whole_diff(float m, float to) {
  return static_cast<int>(fmaxf(m - to, static_cast<float>(kFar)));
}

template <int BITS, int D, int HS, int QSPLIT>
__device__ __forceinline__ void tile_pass(const TileLoads<BITS, D, HS>& ld, uint8_t* v_lds, uint8_t* w_lds,
                                          const uint8_t* q_lds, const float* q_scale, float scale_log2,
                                          const uint32_t (&k_mask)[TileLoads<BITS, D, HS>::SW],
                                          TileState<TileGeo<BITS, D, HS>::NT, HS>& st, int group_shift, int li,
                                          int lq, uint32_t oz) {
  using G = TileGeo<BITS, D, HS, QSPLIT>;
  constexpr int NG = G::NG;
  // LDS offsets are formed anew in each pass: hoisted out of the loop they
  // would hold ~40 registers, i.e. a resident wave
  asm volatile("" : "+v"(li), "+v"(lq));
  // V rows to LDS (this wave's own region: its earlier reads are done, LDS
  // operations of a wave complete in order)
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) {
    const int t = 16 * tau + li;
    uint8_t* dst = v_lds + t * G::VS;
    if constexpr (G::KW % 2 == 0) {
#pragma unroll
      for (int j = 0; j < G::KW; j += 2)
        *reinterpret_cast<u32x2*>(dst + 8 * ((G::KW / 2 * lq + j / 2) ^ v_phi<G::PD>(t))) =
            u32x2{ld.v[tau][j], ld.v[tau][j + 1]};
    } else {
#pragma unroll
      for (int j = 0; j < G::KW; ++j)
        *reinterpret_cast<uint32_t*>(dst + ((4 * (G::KW * lq + j)) ^ (8 * v_phi<G::PD>(t)))) = ld.v[tau][j];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // -------------------------------------------------------------------- QK
  float score[HS][4];
  // the small query parts have sums of their own: added to the large ones step
  // by step they would cost a rounding each (1.2-1.6x the output error of the
  // vector kernel at one group per head, 0.6-1.1x this way)
  f32x4 c[4], rest[4];
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) c[tau] = rest[tau] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int m = 0; m < G::KS; ++m) {
    u32x4 qa[QSPLIT];
#pragma unroll
    for (int sp = 0; sp < QSPLIT; ++sp)
      qa[sp] = *reinterpret_cast<const u32x4*>(q_lds + (16 * sp + li) * G::Q_ROW + 2 * (lq * (D / 4) + 8 * m));
#pragma unroll
    for (int tau = 0; tau < 4; ++tau) {
      const u32x4 b = BITS == 4 ? ints4(ld.k[tau][m], oz) : ints2(ld.k[tau][m >> 1], m & 1, oz);
      c[tau] = mfma16(qa[0], b, c[tau]);
#pragma unroll
      for (int sp = 1; sp < QSPLIT; ++sp) rest[tau] = mfma16(qa[sp], b, rest[tau]);
    }
    __builtin_amdgcn_sched_barrier(0);  // (unpacking further ahead costs registers, i.e. resident waves)
  }
  const f32x4 row_scale = *reinterpret_cast<const f32x4*>(q_scale + 4 * lq);  // of this lane's query rows
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) {
    if constexpr (QSPLIT > 1) c[tau] += rest[tau];
    uint32_t sk[TileLoads<BITS, D, HS>::SW];
#pragma unroll
    for (int i = 0; i < TileLoads<BITS, D, HS>::SW; ++i) sk[i] = kPadRows<D, HS> ? ld.sk[tau][i] & k_mask[i] : ld.sk[tau][i];
#pragma unroll
    for (int hs = 0; hs < HS; ++hs) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const float k = half_bits_to_float(scale_bits(sk, i));
        const float ci = c[tau][hs * NG + i] * row_scale[hs * NG + i];  // (a power of two: exact)
        s = i == 0 ? k * ci : __builtin_fmaf(k, ci, s);
      }
      score[hs][tau] = s;
    }
    if constexpr (HS == 1) {  // 8 or 16 groups: a head's rows lie in 2 or 4 lane rows
      if (group_shift >= 3) score[0][tau] += __shfl_xor(score[0][tau], 16, kWave);
      if (group_shift >= 4) score[0][tau] += __shfl_xor(score[0][tau], 32, kWave);
    }
  }
  // --------------------------------------------------------------- softmax
  float sv[4][NG];  // V scales, 0 for masked tokens (a stale scale may not be finite)
  bool ok[4];
#pragma unroll
  for (int tau = 0; tau < 4; ++tau) {
    ok[tau] = (ld.ok >> tau) & 1u;
#pragma unroll
    for (int i = 0; i < NG; ++i) sv[tau][i] = half_bits_to_float(ok[tau] ? scale_bits(ld.sv[tau], i) : static_cast<uint16_t>(0));
  }
  // W rows 4 lq + i: this lane's four tokens in slots 4 u .. 4 u + 3
  const int u = 8 * ((li >> 1) & 1) + 2 * (li >> 2) + (li & 1);
  int shift[4];  // log2 of what the accumulators so far count relative to the new references
#pragma unroll
  for (int hs = 0; hs < HS; ++hs) {
    float sc[4], mx = -INFINITY;
#pragma unroll
    for (int tau = 0; tau < 4; ++tau) {
      sc[tau] = ok[tau] ? score[hs][tau] * scale_log2 : -INFINITY;
      mx = fmaxf(mx, sc[tau]);
    }
    const float m_new = fmaxf(st.m[hs], ceilf(row_max16(mx)));
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    const int dm = whole_diff(st.m[hs], m_use);
    st.m[hs] = m_new;
    float sum = 0.0f;
#pragma unroll
    for (int tau = 0; tau < 4; ++tau) {
      sc[tau] = __builtin_amdgcn_exp2f(sc[tau] - m_use);
      sum += sc[tau];
    }
    st.l[hs] = ldexpf(st.l[hs], dm) + sum;
#pragma unroll
    for (int gi = 0; gi < NG; ++gi) {
      const int i = hs * NG + gi;
      float w[4];
#pragma unroll
      for (int tau = 0; tau < 4; ++tau) w[tau] = sc[tau] * sv[tau][gi];
      const float big = row_max16(fmaxf(fmaxf(fabsf(w[0]), fabsf(w[1])), fmaxf(fabsf(w[2]), fabsf(w[3]))));
      // (big in [2^(e - 1), 2^e), e its frexp exponent)
      const int most = big > 0.0f ? 13 - __builtin_amdgcn_frexp_expf(big) : kMostExponent;
      const int k = min(min(st.k[i] - dm, most), kMostExponent);
      shift[i] = dm + k - st.k[i];
      st.k[i] = k;
      u32x2 hi, lo;
      uint32_t h, l;
      split_pair(ldexpf(w[0], k), ldexpf(w[1], k), h, l);
      hi[0] = h;
      lo[0] = l;
      split_pair(ldexpf(w[2], k), ldexpf(w[3], k), h, l);
      hi[1] = h;
      lo[1] = l;
      uint8_t* dst = w_lds + (4 * lq + i) * kWRowBytes + 8 * u;
      *reinterpret_cast<u32x2*>(dst) = hi;
      *reinterpret_cast<u32x2*>(dst + 16 * kWRowBytes) = lo;
    }
  }
  if (__any((shift[0] | shift[1] | shift[2] | shift[3]) != 0)) {
#pragma unroll
    for (int n = 0; n < G::NT; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) st.acc[n][i] = ldexpf(st.acc[n][i], shift[i]);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // -------------------------------------------------------------------- PV
  u32x4 wa[2][2];  // [part][K step]
#pragma unroll
  for (int sp = 0; sp < 2; ++sp)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      wa[sp][kk] = *reinterpret_cast<const u32x4*>(w_lds + (16 * sp + li) * kWRowBytes + 64 * kk + 16 * lq);
  // transpose-read row of this lane: kk = li >> 3, nibble rho = li & 7 in slot
  // s = 2 (rho & 3) + (rho >> 2)
  const int rho = li & 7;
  const int s_tr = ((rho & 3) << 1) | (rho >> 2);
  const int t_tr = 16 * (s_tr & 3) + 4 * lq + 2 * (li >> 3) + (s_tr >> 2);
#pragma unroll
  for (int n = 0; n < G::NTR; ++n) {
    const i32x2 tr = lds_read_tr4(v_lds, t_tr * G::VS + 8 * (n ^ v_phi<G::PD>(t_tr)));
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int par = 0; par < G::NPAR; ++par) {
        const uint32_t x = static_cast<uint32_t>(tr[kk]);
        const u32x4 b = BITS == 4 ? ints4(x, oz) : ints2_tr(x, par, oz);
        f32x4& a = st.acc[G::NPAR * n + par];
        a = mfma16(wa[0][kk], b, a);
        a = mfma16(wa[1][kk], b, a);
      }
    if (n % 2 == 1) __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_wave_barrier();  // the next pass's LDS writes stay behind these reads
}

// v[e], of dim lane + 64 e of a head, becomes the largest of v >= 0 over the
// dim's group `own` (HS == 4: over the head).  Without branches, under which the pass's loads in flight
// would cost registers, where head_dim is a power of two.  `scratch`: an LDS
// word a group, the wave's own.
template <int D, int HS, int QE>
__device__ __forceinline__ void group_max(float (&v)[QE], const int (&own)[QE], int* scratch, int group_size) {
  const int lane = threadIdx.x & (kWave - 1);
  if constexpr (HS == 4) {
    float m = v[0];
#pragma unroll
    for (int e = 1; e < QE; ++e) m = fmaxf(m, v[e]);
    m = wave_max(m);
#pragma unroll
    for (int e = 0; e < QE; ++e) v[e] = m;
  } else if constexpr (HS == 2 && D % 128 == 0) {  // two groups of whole waves
    constexpr int kPer = QE / 2;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      float m = v[g * kPer];
#pragma unroll
      for (int e = 1; e < kPer; ++e) m = fmaxf(m, v[g * kPer + e]);
      m = wave_max(m);
#pragma unroll
      for (int e = 0; e < kPer; ++e) v[g * kPer + e] = m;
    }
  } else if (D % kWave == 0 || (group_size & (group_size - 1)) == 0) {  // runs of 4 to 64 lanes, a power of two
#pragma unroll
    for (int e = 0; e < QE; ++e) {
      float m = fmaxf(v[e], quad_lane<0xB1>(v[e]));
      m = fmaxf(m, quad_lane<0x4E>(m));
      const float m8 = fmaxf(m, quad_lane<0x141>(m));  // with the other quad of 8
      m = group_size > 4 ? m8 : m;
      const float m16 = fmaxf(m, quad_lane<0x140>(m));  // with the other half of 16
      m = group_size > 8 ? m16 : m;
      const float m01 = fmaxf(lane_value(m, 0), lane_value(m, 16)), m23 = fmaxf(lane_value(m, 32), lane_value(m, 48));
      v[e] = group_size > 32 ? fmaxf(m01, m23) : group_size > 16 ? (lane < 32 ? m01 : m23) : m;
    }
  } else {  // head_dim 96 in other groups: the largest bits (lanes past the row's end repeat its last value)
    const int groups = D / group_size;
    if (lane < groups) scratch[lane] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int e = 0; e < QE; ++e)
      __hip_atomic_fetch_max(scratch + own[e], __builtin_bit_cast(int, v[e]), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int e = 0; e < QE; ++e) v[e] = __builtin_bit_cast(float, scratch[own[e]]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

template <int BITS, int D, int HS, int QSPLIT>
__global__ __launch_bounds__(kTileThreads, tile_workgroups_per_cu(D, HS, QSPLIT)) void decode_tile_kernel(
    const void* query, const uint8_t* pk, const uint8_t* pv, const uint16_t* sk, const uint16_t* sv, uint32_t shape,
    uint32_t block_tokens, int blocks_per_split, int units, TileTail r) {
  using G = TileGeo<BITS, D, HS, QSPLIT>;
  constexpr int NG = G::NG;
  __shared__ __attribute__((aligned(16))) uint8_t lds[G::LDS];
  __shared__ __attribute__((aligned(16))) float ml[4][HS][2][kTileWaves];  // [lane row][head][m, l][wave]
  __shared__ __attribute__((aligned(16))) float q_scale[16];  // what a query row's operand counts by
  const TileParams p{pk, pv, sk, sv, static_cast<int>(shape & 0xFFFFu), static_cast<int>((shape >> 16) & 0x1Fu),
                     static_cast<int>((shape >> 21) & 7u), block_tokens, (shape & kHasTable) != 0};

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 15;
  const int lq = lane >> 4;

  // XCD-aware placement: consecutive workgroup ids go to different XCDs; the
  // kv heads and head chunks of one split, which share cache lines and rows,
  // get ids 8 apart (grid (8, kv heads x chunks, splits / 8)), i.e. one XCD and
  // its L2
  const int split = static_cast<int>(blockIdx.z) * 8 + static_cast<int>(blockIdx.x);
  const int u0 = split * blocks_per_split;
  if (u0 >= units) return;  // padding ids of the last round (splits = ceil(units / blocks_per_split))
  const int n_units = min(units - u0, blocks_per_split);
  int kvh = static_cast<int>(blockIdx.y), chunk = 0;
  if (r.head_chunks > 1) {
    const uint32_t y = blockIdx.y;
    kvh = static_cast<int>(__umulhi(y, r.chunk_magic));
    chunk = static_cast<int>(y) - kvh * r.head_chunks;
  }
  const int head0 = kvh * r.gq + chunk * r.heads_per_wg;
  const int nh = min(r.heads_per_wg, r.gq - chunk * r.heads_per_wg);

  // ------------------------------------------------------------------ loads
  // the query rows first (this wave's heads: wave, wave + 4, ...), then this
  // wave's first pass
  constexpr int QE = (D + kWave - 1) / kWave;
  const int group_shift = p.group_shift;
  float qx[HS][QE];
  auto load_rows = [&](auto type) {
    using QT = decltype(type);
#pragma unroll
    for (int i = 0; i < HS; ++i)
#pragma unroll
      for (int e = 0; e < QE; ++e) {
        // (rows past the last head re-read the last one and count as zeros below)
        const int h = min(wave + kTileWaves * i, nh - 1), d = min(lane + kWave * e, D - 1);
        qx[i][e] = load_query<QT>(query, (head0 + h) * D + d);
      }
  };
  if constexpr (QSPLIT == 1) {
    if (r.query_dtype == KVSSD_DTYPE_F16) load_rows(_Float16{});
    else load_rows(uint16_t{});
  } else {
    if (r.query_dtype == KVSSD_DTYPE_F32) load_rows(float{});
    else load_rows(double{});
  }
  const int span_shift = group_shift > 2 ? group_shift - 2 : 0;  // lane rows per head: 2^span_shift
  const bool wide_scales = D != 96 || p.groups % NG == 0;  // this lane's groups in one aligned load
  int gbase = NG == 4 ? 4 * (lq & ((1 << span_shift) - 1)) : 0;
  uint32_t k_mask[TileLoads<BITS, D, HS>::SW];
#pragma unroll
  for (int i = 0; i < TileLoads<BITS, D, HS>::SW; ++i)
    k_mask[i] = (gbase + 2 * i < p.groups ? 0xFFFFu : 0u) | (gbase + 2 * i + 1 < p.groups ? 0xFFFF0000u : 0u);
  if (wide_scales) gbase = min(gbase, p.groups - NG);

  const uint32_t bt = block_tokens;
  int base_unit = 0;
  uint32_t base_off = static_cast<uint32_t>(kChunkTok * wave);
  base_unit = static_cast<int>((base_off * r.bt_magic) >> 20);  // (below 256: 0 in blocks of 256 or more)
  base_off -= static_cast<uint32_t>(base_unit) * bt;
  TileLoads<BITS, D, HS> ld;
  bool have = base_unit < n_units;
  if (have) load_pass<BITS, D, HS>(ld, p, r, u0, n_units, base_unit, base_off, kvh, li, lq, gbase, wide_scales);

  // ------------------------------------------------------------------ query
  // A operand rows (head, group) in LDS, in K-slot order: a head's values in
  // the row of their group, zeros in its other rows.  Values are scaled by
  // 2^(kTop - ex), ex the exponent of the largest: over the head for 16-bit
  // queries, of which one part holds fp16 values exactly and bf16 values down to
  // 2^-32 of the largest (below, to 2^-40 of it); over the row for the three
  // parts of wider ones, which leave at most 2^-39 of the row's largest.  (Rows
  // for all of them: 0.4-0.8 us of 17-22.)
  constexpr int kTop = QSPLIT == 1 ? 15 : 14;
  const int group_size = D % kWave == 0 ? D >> group_shift : D / p.groups;
  uint8_t* q_lds = lds + G::Q_OFF;
#pragma unroll
  for (int i = 0; i < HS; ++i) {
    const int h = wave + kTileWaves * i;
    if (h >= (16 >> group_shift)) break;
    int own[QE];
    float mx[QE];
#pragma unroll
    for (int e = 0; e < QE; ++e) {
      own[e] = static_cast<int>((static_cast<uint32_t>(min(lane + kWave * e, D - 1)) * r.group_magic) >> 16);
      if (h >= nh) qx[i][e] = 0.0f;
      const float x = fabsf(qx[i][e]);
      mx[e] = x < INFINITY ? x : 0.0f;
    }
    group_max<D, QSPLIT == 1 ? 4 : HS>(mx, own, reinterpret_cast<int*>(q_scale) + (h << group_shift), group_size);
    // (rows past the last of 3, 6 or 12 groups hold zeros: any finite factor)
    if (D == 96 && lane < (1 << group_shift)) q_scale[(h << group_shift) + lane] = 1.0f;
#pragma unroll
    for (int e = 0; e < QE; ++e) {
      const int d = lane + kWave * e;
      if (D % kWave != 0 && d >= D) break;
      const int ex = (mx[e] > 0.0f ? __builtin_amdgcn_frexp_expf(mx[e]) - 1 : 0) - kTop;  // mx in [2^ex, 2^(ex + 1))
      q_scale[(h << group_shift) + own[e]] = ldexpf(1.0f, ex);
      float rem = ldexpf(qx[i][e], -ex);
      _Float16 part[QSPLIT];
#pragma unroll
      for (int sp = 0; sp < QSPLIT; ++sp) {
        part[sp] = static_cast<_Float16>(rem);
        rem = fmaxf(rem - static_cast<float>(part[sp]), -65504.0f);
      }
      uint8_t* dst = q_lds + (h << group_shift) * G::Q_ROW + 2 * query_slot<BITS, D>(d);
      for (int g = 0; g < (1 << group_shift); ++g, dst += G::Q_ROW)
#pragma unroll
        for (int sp = 0; sp < QSPLIT; ++sp)
          *reinterpret_cast<_Float16*>(dst + 16 * sp * G::Q_ROW) = g == own[e] ? part[sp] : static_cast<_Float16>(0.0f);
    }
  }
  __syncthreads();
  TileState<G::NT, HS> st;
#pragma unroll
  for (int i = 0; i < 4; ++i) st.k[i] = kMostExponent;
#pragma unroll
  for (int hs = 0; hs < HS; ++hs) {
    st.m[hs] = -INFINITY;
    st.l[hs] = 0.0f;
  }
#pragma unroll
  for (int n = 0; n < G::NT; ++n) st.acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // 0, but opaque: keeps the unpack masks in VGPRs (a three-operand VALU op
  // reads one scalar at most)
  const uint32_t oz = static_cast<uint32_t>(lane) & static_cast<uint32_t>(units >> 30);
  uint8_t* v_lds = lds + wave * G::WAVE_BYTES;
  uint8_t* w_lds = v_lds + G::V_BYTES;
  while (have) {
    tile_pass<BITS, D, HS, QSPLIT>(ld, v_lds, w_lds, q_lds, q_scale, r.scale_log2, k_mask, st, group_shift, li, lq, oz);
    base_off += kTileThreads;  // (64 slots per wave and pass)
    const uint32_t q = ((base_off * r.bt_magic) >> 20) + (bt >= 256u && base_off >= bt ? 1u : 0u);
    base_unit += static_cast<int>(q);
    base_off -= q * bt;
    have = base_unit < n_units;
    if (have) load_pass<BITS, D, HS>(ld, p, r, u0, n_units, base_unit, base_off, kvh, li, lq, gbase, wide_scales);
  }

  // --------------------------------------------- the waves' states, merged
  // (a wave without a valid token has l = 0 and counts for nothing; a NaN l stays)
#pragma unroll
  for (int hs = 0; hs < HS; ++hs) {
    const float l = row_sum16(st.l[hs]);
    if (li == 0) {
      ml[lq][hs][0][wave] = l != 0.0f ? st.m[hs] : -INFINITY;
      ml[lq][hs][1][wave] = l;
    }
  }
  __syncthreads();  // (m, l) of every wave; every V, W and query region is free
  const int span = 1 << span_shift;
  // the largest m of a head: over the waves and its lane rows, whose m differ
  // by a rounding (and so at most by one, past a whole number)
  auto head_max = [&](int row, int hs) {
    float big = -INFINITY;
    for (int i = 0; i < span; ++i) {
      const f32x4 m = *reinterpret_cast<const f32x4*>(ml[row + i][hs][0]);
      big = fmaxf(fmaxf(fmaxf(big, m[0]), fmaxf(m[1], m[2])), m[3]);
    }
    return big;
  };
  float* xo = reinterpret_cast<float*>(lds);  // [wave][head][D]
#pragma unroll
  for (int hs = 0; hs < HS; ++hs) {
    const int h = HS == 1 ? lq >> span_shift : HS * lq + hs;
    const float big = head_max(lq & ~(span - 1), hs);
    const bool some = ml[lq][hs][1][wave] != 0.0f;
    const int dm = whole_diff(st.m[hs], big);
    if (h < nh) {
      float* xrow = xo + (wave * G::HEADS + h) * D;
#pragma unroll
      for (int n = 0; n < G::NTR; ++n)
#pragma unroll
        for (int par = 0; par < G::NPAR; ++par) {
          const int dim = BITS == 4 ? 16 * n + li : 32 * n + 2 * li + par;
          const int gt = static_cast<int>((static_cast<uint32_t>(dim) * r.group_magic) >> 16);
          const f32x4 a = st.acc[G::NPAR * n + par];
          float o = a[hs * NG];
          int k = st.k[hs * NG];
#pragma unroll
          for (int i = 1; i < NG; ++i) {
            o = (gt & (NG - 1)) == i ? a[hs * NG + i] : o;
            k = (gt & (NG - 1)) == i ? st.k[hs * NG + i] : k;
          }
          const bool mine = NG < 4 || (gt >> 2) == (lq & (span - 1));
          if (mine) xrow[dim] = some ? ldexpf(o, dm - k) : 0.0f;
        }
    }
  }
  __syncthreads();
  const long prow = static_cast<long>(split) * r.query_heads + head0;
  for (int i = tid; i < nh * D; i += kTileThreads) {
    float o = 0.0f;
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) o += xo[w * G::HEADS * D + i];
    r.part_o[prow * D + i] = o;
  }
  if (tid < nh) {
    // a head's first lane row holds its l
    const int row = HS == 1 ? tid << span_shift : tid / HS;
    const int hs = HS == 1 ? 0 : tid % HS;
    const float big = head_max(row, hs);
    float l = 0.0f;
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) {
      const float lw = ml[row][hs][1][w];
      l += lw != 0.0f ? lw * __builtin_amdgcn_exp2f(ml[row][hs][0][w] - big) : 0.0f;
    }
    r.part_ml[2 * (prow + tid)] = big;
    r.part_ml[2 * (prow + tid) + 1] = l;
  }
  if (r.split_note != nullptr && split == 0 && blockIdx.y == 0 && tid == 0) *r.split_note = -static_cast<float>(r.splits);
}

int ceil_log2(int n) {
  int s = 0;
  while ((1 << s) < n) ++s;
  return s;
}

struct TileLaunch {
  const DecodeArgs& a;
  uint32_t shape;
  int group_shift, blocks_per_split;
  dim3 grid;
  TileTail tail;
};

template <int BITS, int D, int HS, int QSPLIT>
void launch_parts(const TileLaunch& t) {
  const DecodeArgs& a = t.a;
  hipLaunchKernelGGL((decode_tile_kernel<BITS, D, HS, QSPLIT>), t.grid, dim3(kTileThreads), 0, a.stream, a.query,
                     a.packed_k, a.packed_v, a.scales_k, a.scales_v, t.shape,
                     static_cast<uint32_t>(a.desc.block_tokens), t.blocks_per_split, a.units, t.tail);
}

// an fp16 query is one fp16 part, a bf16 one too once its head's largest value
// is normalised; fp32 and fp64 ones (as fp32) take three
int tile_query_parts(int dtype) { return dtype == KVSSD_DTYPE_F16 || dtype == KVSSD_DTYPE_BF16 ? 1 : 3; }

template <int BITS, int D, int HS>
void launch_hs(const TileLaunch& t) {
  if (tile_query_parts(t.a.desc.query_dtype) == 1) launch_parts<BITS, D, HS, 1>(t);
  else launch_parts<BITS, D, HS, 3>(t);
}

template <int BITS, int D>
void launch_dim(const TileLaunch& t) {
  if (t.group_shift >= 2) launch_hs<BITS, D, 1>(t);
  else if (t.group_shift == 1) launch_hs<BITS, D, 2>(t);
  else launch_hs<BITS, D, 4>(t);
}

// query heads of a workgroup: as many as a 16-row operand holds
int tile_head_chunks(const kvssd_decode_desc& d, int* rows) {
  *rows = 16 >> ceil_log2(d.head_dim / d.group_size);
  return (d.query_heads / d.kv_heads + *rows - 1) / *rows;
}

}  // namespace

bool tile_supported(const kvssd_decode_desc& d) {
  const bool dim = d.head_dim == 64 || d.head_dim == 128 || d.head_dim == 256 || (d.head_dim == 96 && d.bits == 4);
  if (!dim || d.head_dim / d.group_size > 16 || d.block_tokens % 16) return false;
  if (static_cast<int64_t>(d.num_blocks) * d.block_tokens > 0x7FFFFFFF / d.kv_heads) return false;  // 32-bit row indices
  int rows = 0;
  return static_cast<int64_t>(d.kv_heads) * tile_head_chunks(d, &rows) <= 0xFFFF;  // grid limit
}

// Splits of the tile kernel: a pass of all four waves covers 256 slots and costs
// ~2 us, a workgroup's start and end ~5 us.  So the grid is one round of
// resident workgroups, each of at least one full pass, and longer contexts get
// more passes per workgroup; never more splits than plan_splits, which the
// workspace is sized for.
SplitPlan tile_splits(const kvssd_decode_desc& d, int units, const SplitPlan& most) {
  int rows = 0;
  const int64_t items = static_cast<int64_t>(d.kv_heads) * tile_head_chunks(d, &rows);
  const int hs = rows == 16 ? 4 : rows == 8 ? 2 : 1;
  const int64_t resident = 256LL * tile_workgroups_per_cu(d.head_dim, hs, tile_query_parts(d.query_dtype));
  const int64_t slots = static_cast<int64_t>(units) * d.block_tokens;
  const int64_t passes = (slots * items + 256 * resident - 1) / (256 * resident);
  const int64_t per = (256 * passes + d.block_tokens - 1) / d.block_tokens;
  SplitPlan plan = most;
  if (per > most.blocks_per_split) {
    plan.blocks_per_split = static_cast<int>(per < units ? per : units);
    plan.splits = (units + plan.blocks_per_split - 1) / plan.blocks_per_split;
  }
  return plan;
}

bool tile_aligned(const DecodeArgs& a) {
  auto ok = [](const void* ptr, uintptr_t n) { return (reinterpret_cast<uintptr_t>(ptr) % n) == 0; };
  return ok(a.packed_k, 16) && ok(a.packed_v, 16) && ok(a.scales_k, 8) && ok(a.scales_v, 8);
}

int launch_tile(const DecodeArgs& a, const SplitPlan& plan, SplitPartials parts) {
  const kvssd_decode_desc& d = a.desc;
  const int gq = d.query_heads / d.kv_heads;
  const int groups = d.head_dim / d.group_size;
  int rows = 0;
  const int chunks = tile_head_chunks(d, &rows);
  TileLaunch t{a};
  t.group_shift = ceil_log2(groups);
  t.shape = pack_shape(d.kv_heads, groups, t.group_shift, a.table != nullptr);
  t.blocks_per_split = plan.blocks_per_split;
  t.grid = dim3(8, static_cast<unsigned>(d.kv_heads * chunks), static_cast<unsigned>((plan.splits + 7) / 8));
  TileTail& r = t.tail;
  r.table = a.table;
  r.valid = a.valid;
  r.part_o = parts.o;
  r.part_ml = parts.ml;
  r.query_heads = d.query_heads;
  r.num_blocks = d.num_blocks;
  r.gq = gq;
  r.heads_per_wg = (gq + chunks - 1) / chunks;
  r.head_chunks = chunks;
  r.query_dtype = d.query_dtype;
  r.splits = plan.splits;
  r.split_note = a.split_note;
  r.chunk_magic = chunks > 1 ? static_cast<uint32_t>(((1ull << 32) + chunks - 1) / chunks) : 0u;
  r.bt_magic = d.block_tokens < 256 ? ((1u << 20) + d.block_tokens - 1) / d.block_tokens : 0u;
  r.group_magic = (65536u + d.group_size - 1) / d.group_size;
  r.scale_log2 = static_cast<float>(d.sm_scale) * kLog2e;
  switch (d.head_dim) {
    case 64: d.bits == 4 ? launch_dim<4, 64>(t) : launch_dim<2, 64>(t); break;
    case 96: launch_dim<4, 96>(t); break;
    case 128: d.bits == 4 ? launch_dim<4, 128>(t) : launch_dim<2, 128>(t); break;
    default: d.bits == 4 ? launch_dim<4, 256>(t) : launch_dim<2, 256>(t); break;
  }
  return hip_status(hipGetLastError(), "decode_tile launch");
}

}  // namespace kvssd
