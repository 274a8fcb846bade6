// CRC-32 on the GPU, shared by the v1 record codec (records.hip) and the
// vLLM block codec (vllm_codec.hip).
//
// CRC-32 is zlib's: reflected polynomial 0xEDB88320, register preset to all
// ones, output complemented.  Polynomials over GF(2) are held bit-reflected
// (bit 31 is the coefficient of x^0).  The raw register update (preset 0, no
// complement) is linear: crc_raw(A || B) = x^(8|B|) crc_raw(A) + crc_raw(B)
// (mod P), and leading zero bytes do not change crc_raw, so a payload is
// virtually left-padded with zeros to a whole number of pieces.  Finally
// crc32(D) = x^(8|D|) * 0xFFFFFFFF + crc_raw(D) + 0xFFFFFFFF.
//
// Chunked form (payloads of a multiple of 16 bytes whose arrays are too, the
// usual case): a workgroup of 1024 threads covers a record in 16-byte chunks,
// chunk c = j * 1024 + t belonging to thread t, and takes the CRC on the matrix
// cores.  A raw CRC is a product over GF(2) of a constant bit matrix with the
// message bits, so one v_mfma_f32_32x32x64_f8f6f4 of 0/1 values in fp4 counts,
// for 32 CRC bits (rows) and 32 columns, the set message bits of 64 (a dword of
// lane n's chunk and one of lane n + 32's); the counts' parities are the CRC
// bits.  Four rows j of chunks accumulate before the parities are taken (their
// matrices differ by powers of x^(8 * 16384)); a fifth matrix carries a column's
// CRC so far over the next four rows.  One multiply per column by its distance
// to the end of the message and an XOR reduction end it.  Bits need no
// unpacking: the four bits of a nibble, masked out one at a time, read as the
// fp4 values 0.5, 1 and 2 (the top bit shifted down first), and the matrix
// holds the factor that makes each product 1.
// Measured (1024 records of 148 KiB, with the copy into the arrays): 93 us with
// 16 table lookups in LDS per chunk (their bank conflicts, ~40 us of it), 66
// us in this form; the copy alone takes 54.
// Other layouts take the general form: 1024 contiguous segments through a
// slicing-by-4 walk and a 10-level fold.  All tables are built at compile time.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace kvssd {
namespace {

constexpr uint32_t kPoly = 0xEDB88320u;
constexpr int kCrcThreads = 1024;          // segments per record
constexpr int kCrcLevels = 10;             // log2(kCrcThreads)

// a * b mod P (reflected representation)
__host__ __device__ constexpr uint32_t gf_mul(uint32_t a, uint32_t b) {
  uint32_t p = 0;
  for (int i = 0; i < 32; ++i) {
    if (a & (0x80000000u >> i)) p ^= b;
    b = (b & 1u) ? (b >> 1) ^ kPoly : b >> 1;  // b *= x
  }
  return p;
}

// x^(8 n) mod P
__host__ __device__ constexpr uint32_t x_pow_bytes(uint64_t n) {
  uint32_t r = 0x80000000u;   // x^0
  uint32_t sq = 0x00800000u;  // x^8
  while (n) {
    if (n & 1u) r = gf_mul(r, sq);
    sq = gf_mul(sq, sq);
    n >>= 1;
  }
  return r;
}

constexpr int kChunkBytes = 16;
constexpr int kStrideBytes = kChunkBytes * kCrcThreads;  // one row of chunks

// slice[k][n]: raw register after byte n followed by k zero bytes
struct CrcTables {
  uint32_t slice[4][256];
};

constexpr CrcTables make_crc_tables() {
  CrcTables t{};
  for (uint32_t n = 0; n < 256; ++n) {
    uint32_t c = n;
    for (int i = 0; i < 8; ++i) c = (c & 1u) ? (c >> 1) ^ kPoly : c >> 1;
    t.slice[0][n] = c;
  }
  for (int k = 1; k < 4; ++k)
    for (uint32_t n = 0; n < 256; ++n) {
      const uint32_t c = t.slice[k - 1][n];
      t.slice[k][n] = t.slice[0][c & 0xFFu] ^ (c >> 8);  // one more zero byte
    }
  return t;
}

__device__ const CrcTables kCrcTables = make_crc_tables();

// Position multipliers of the chunked form: chunk[t] = x^(8 * 16 * (1023 - t)),
// row[t] = x^(8 * 16384 * (1023 - t)) -- the shift of piece t of 1024 equal
// pieces to the end of the message they form.
// word[t] = that of the last dword of thread t's column in the dword layout (below).
struct PosTables {
  uint32_t chunk[kCrcThreads];
  uint32_t row[kCrcThreads];
  uint32_t word[kCrcThreads];
};

constexpr PosTables make_pos_tables() {
  PosTables p{};
  const uint32_t sc = x_pow_bytes(16), sr = x_pow_bytes(16384);
  p.chunk[kCrcThreads - 1] = 0x80000000u;  // x^0
  p.row[kCrcThreads - 1] = 0x80000000u;
  for (int t = kCrcThreads - 1; t > 0; --t) {
    p.chunk[t - 1] = gf_mul(p.chunk[t], sc);
    p.row[t - 1] = gf_mul(p.row[t], sr);
  }
  const uint32_t sw = x_pow_bytes(4);
  for (int t = kCrcThreads - 1; t >= 0; --t)
    p.word[t] = (t & 31) == 31 ? p.chunk[t | 63] : gf_mul(p.word[t + 1], sw);
  return p;
}

__device__ const PosTables kPosTables = make_pos_tables();

// a * b mod P without branches (device)
__device__ __forceinline__ uint32_t gf_mul_dev(uint32_t a, uint32_t b) {
  uint32_t p = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    p ^= b & (0u - ((a >> (31 - i)) & 1u));
    b = (b >> 1) ^ (kPoly & (0u - (b & 1u)));
  }
  return p;
}

// raw register after byte n followed by k zero bytes (slicing-by-4 table k)
__device__ __forceinline__ uint32_t crc_table_entry(int k, uint32_t n) { return kCrcTables.slice[k][n]; }

struct CrcPlan {
  uint32_t seg_bytes;           // L: bytes per segment (multiple of 4)
  uint32_t pad;                 // virtual leading zero bytes
  uint32_t len;                 // payload bytes covered
  uint32_t x_len;               // x^(8 len) mod P
  uint32_t level[kCrcLevels];   // x^(8 L 2^k) mod P
};

CrcPlan make_crc_plan(uint32_t len) {
  CrcPlan c{};
  const uint32_t per = (len + kCrcThreads - 1) / kCrcThreads;
  c.seg_bytes = (per + 3u) & ~3u;
  c.pad = c.seg_bytes * kCrcThreads - len;
  c.len = len;
  c.x_len = x_pow_bytes(len);
  for (int k = 0; k < kCrcLevels; ++k) c.level[k] = x_pow_bytes(static_cast<uint64_t>(c.seg_bytes) << k);
  return c;
}

// zlib CRC-32 of data[0 .. plan.len), data 4-byte aligned; every thread of a
// kCrcThreads workgroup calls it; tab = the four slicing tables in LDS,
// seg = kCrcThreads words of LDS.  Returns the CRC in every thread.
__device__ uint32_t block_crc32(const uint8_t* data, const CrcPlan& plan, const uint32_t (*tab)[256], uint32_t* seg) {
  const int tid = threadIdx.x;
  const int64_t v0 = static_cast<int64_t>(tid) * plan.seg_bytes - plan.pad;  // first real byte of the segment
  uint32_t crc = 0;
  if ((plan.len & 3u) == 0) {
    // pad is then a multiple of 4: whole dwords, real or virtual zeros
    for (uint32_t i = 0; i < plan.seg_bytes; i += 4) {
      const int64_t at = v0 + i;
      if (at < 0) continue;  // leading zeros keep the raw register at 0
      crc ^= *reinterpret_cast<const uint32_t*>(data + at);
      crc = tab[3][crc & 0xFFu] ^ tab[2][(crc >> 8) & 0xFFu] ^ tab[1][(crc >> 16) & 0xFFu] ^ tab[0][crc >> 24];
    }
  } else {
    for (uint32_t i = 0; i < plan.seg_bytes; ++i) {
      const int64_t at = v0 + i;
      if (at < 0) continue;
      crc = tab[0][(crc ^ data[at]) & 0xFFu] ^ (crc >> 8);
    }
  }
  seg[tid] = crc;
  for (int k = 0; k < kCrcLevels; ++k) {
    __syncthreads();
    const int span = 1 << k;
    if ((tid & (2 * span - 1)) == 0) seg[tid] = gf_mul(plan.level[k], seg[tid]) ^ seg[tid + span];
  }
  __syncthreads();
  const uint32_t raw = seg[0];
  __syncthreads();  // seg may be reused by the caller
  return gf_mul(plan.x_len, 0xFFFFFFFFu) ^ raw ^ 0xFFFFFFFFu;
}

__device__ __forceinline__ void fill_crc_tables(uint32_t (*tab)[256]) {
  for (int i = threadIdx.x; i < 4 * 256; i += blockDim.x) tab[i >> 8][i & 255] = crc_table_entry(i >> 8, i & 255);
}

// ----------------------------------------------------------- chunked form ---
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kGroupRows = 4;  // rows of chunks between two parity steps

// Matrices of the chunked form as A operands, one u32x4 per lane: lane (r, half)
// holds bit r of the CRC contributions of 32 message bits, nibble i of dword p
// that of bit 4 i + p.  data[j][w]: dword w of a chunk in row j of a group, in
// lane half 0 (32 chunks before half 1's).  In the dword layout a wave's 1 KiB
// of a row is four runs of 64 dwords instead, lane l holding dword l of each:
// data[j][w] is run w, and half 0's dword lies 32 dwords before half 1's.
// carry: the column's raw CRC before the group, bits split over the halves as
// the parities are.
struct BitMatrices {
  uint32_t data[kGroupRows][4][64][4];
  uint32_t carry[64][4];
};

// the CRC bits a lane half holds after a parity step
constexpr uint32_t kHalfBits = 0x0F0F0F0Fu;

constexpr uint32_t fp4_factor(int plane) { return plane == 0 ? 4u : plane == 1 ? 2u : 1u; }  // 2, 1, 0.5

constexpr BitMatrices make_bit_matrices(bool words) {
  BitMatrices m{};
  uint32_t row_pow[kGroupRows] = {};
  row_pow[kGroupRows - 1] = 0x80000000u;  // x^0
  const uint32_t stride = x_pow_bytes(kStrideBytes);
  for (int j = kGroupRows - 1; j > 0; --j) row_pow[j - 1] = gf_mul(row_pow[j], stride);
  const uint32_t over = gf_mul(row_pow[0], stride);  // a whole group of rows
  const uint32_t half_pow = x_pow_bytes(32 * (words ? 4 : kChunkBytes));
  // byte b of dword w, to the end of the chunk (the last run): its own 8 shifts and the bytes after it
  uint32_t byte_pow[kChunkBytes] = {};
  byte_pow[kChunkBytes - 1] = 0x00800000u;
  const uint32_t run = words ? x_pow_bytes(4 * 64) : x_pow_bytes(4);
  for (int b = kChunkBytes - 1; b > 0; --b)
    byte_pow[b - 1] = (b & 3) != 0 ? gf_mul(byte_pow[b], 0x00800000u) : gf_mul(byte_pow[b + 3], run);
  for (int bit = 0; bit < 32; ++bit) {
    const int plane = bit & 3;
    const uint32_t value = fp4_factor(plane) << (4 * (bit >> 2));
    for (int w = 0; w < 4; ++w) {
      const uint32_t c = gf_mul(1u << (bit & 7), byte_pow[4 * w + bit / 8]);
      for (int j = 0; j < kGroupRows; ++j) {
        uint32_t v = gf_mul(c, row_pow[j]);
        for (int half = 1; half >= 0; --half) {
          for (int r = 0; r < 32; ++r)
            if ((v >> r) & 1u) m.data[j][w][32 * half + r][plane] |= value;
          v = gf_mul(v, half_pow);
        }
      }
    }
    const int half = (kHalfBits >> bit) & 1u ? 0 : 1;  // the half that holds this CRC bit
    const uint32_t v = gf_mul(1u << bit, over);
    for (int r = 0; r < 32; ++r)
      if ((v >> r) & 1u) m.carry[32 * half + r][plane] |= value;
  }
  return m;
}

__device__ const BitMatrices kBitMatrices = make_bit_matrices(false);
__device__ const BitMatrices kWordMatrices = make_bit_matrices(true);

struct ChunkLds {
  u32x4 data[kGroupRows][4][64];
  u32x4 carry[64];
  uint32_t seg[kCrcThreads / 64];
};

// by a workgroup of kCrcThreads / PARTS threads
template <int PARTS = 1>
__device__ __forceinline__ void load_chunk_tables(ChunkLds& l, const BitMatrices& m = kBitMatrices) {
  constexpr int threads = kCrcThreads / PARTS;
  const u32x4* src = reinterpret_cast<const u32x4*>(&m);
  u32x4* dst = &l.data[0][0][0];  // data then carry: 1024 + 64 entries
  u32x4 v[PARTS];
#pragma unroll
  for (int i = 0; i < PARTS; ++i) v[i] = src[threadIdx.x + i * threads];
  if (threadIdx.x < 64) dst[kCrcThreads + threadIdx.x] = src[kCrcThreads + threadIdx.x];
#pragma unroll
  for (int i = 0; i < PARTS; ++i) dst[threadIdx.x + i * threads] = v[i];
}

// 16 bytes at a 4-byte aligned address
__device__ __forceinline__ u32x4 load16(const uint8_t* p) {
  u32x4 v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, 4), 16);
  return v;
}

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// acc += A x (the 32 bits of x in every lane, as fp4 values)
__device__ __forceinline__ f32x16 count_bits(u32x4 a, uint32_t x, f32x16 acc) {
  const i32x8 A = {static_cast<int>(a[0]), static_cast<int>(a[1]), static_cast<int>(a[2]), static_cast<int>(a[3]), 0, 0, 0, 0};
  const i32x8 B = {static_cast<int>(x & 0x11111111u), static_cast<int>(x & 0x22222222u),
                   static_cast<int>(x & 0x44444444u), static_cast<int>((x >> 1) & 0x44444444u), 0, 0, 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B, acc, 4, 4, 0, 127, 0, 127);  // fp4, block scales 2^0
}

// Counts of a group of rows, from the column state h (this lane half's bits of
// the column's raw CRC) carried over it.  Every lane of the wave takes part.
__device__ __forceinline__ f32x16 crc_begin(const ChunkLds& l, uint32_t h) {
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 8388608.0f;  // 2^23: a count's parity is the lowest bit
  return count_bits(l.carry[threadIdx.x & 63], h, acc);
}

// ... with row j of the group
__device__ __forceinline__ f32x16 crc_row(const ChunkLds& l, f32x16 acc, int j, u32x4 v) {
#pragma unroll
  for (int w = 0; w < 4; ++w) acc = count_bits(l.data[j][w][threadIdx.x & 63], v[w], acc);
  return acc;
}

// ... and the column state after it
__device__ __forceinline__ uint32_t crc_end(f32x16 acc) {
  // register i holds CRC bit 8 (i / 4) + i % 4, + 4 in lane half 1
  uint32_t p = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float count = acc[i];  // (a bit cast of acc[i] itself reads acc[0])
    p |= (__builtin_bit_cast(uint32_t, count) & 1u) << (8 * (i >> 2) + (i & 3));
  }
  return p << (((threadIdx.x & 63) >> 5) * 4);
}

// A group of rows v, the first `first` of them zeros.
__device__ __forceinline__ uint32_t crc_group(const ChunkLds& l, uint32_t h, const u32x4 (&v)[kGroupRows], int first) {
  f32x16 acc = crc_begin(l, h);
#pragma unroll
  for (int j = 0; j < kGroupRows; ++j)
    if (j >= first) acc = crc_row(l, acc, j, v[j]);
  return crc_end(acc);
}

// Chunk geometry of a payload of `len` bytes (a multiple of 16): `rows` rows of
// 1024 chunks, the first `pad` bytes virtual zeros.
struct ChunkPlan {
  int rows;
  int64_t pad;
  uint32_t x_len;  // x^(8 len) mod P
};

ChunkPlan make_chunk_plan(uint32_t len) {
  ChunkPlan c{};
  c.rows = static_cast<int>((len + kStrideBytes - 1) / kStrideBytes);
  c.pad = static_cast<int64_t>(c.rows) * kStrideBytes - len;
  c.x_len = x_pow_bytes(len);
  return c;
}

// byte offset (into the payload) of chunk row j of this thread; negative = virtual zeros
__device__ __forceinline__ int64_t chunk_offset(const ChunkPlan& c, int j) {
  return (static_cast<int64_t>(j) * kCrcThreads + threadIdx.x) * kChunkBytes - c.pad;
}

// Fold the column states h of crc_group over the workgroup, thread t holding
// those of threads t, t + 1024 / PARTS, ... of 1024: a column ends with its
// half-1 chunk (pos[t] = the shift of piece t to the end).  The raw register
// value of the whole message is returned in every thread.
template <int PARTS>
__device__ __forceinline__ uint32_t fold_columns(ChunkLds& l, const uint32_t* pos, const uint32_t (&h)[PARTS]) {
  constexpr int threads = kCrcThreads / PARTS;
  const int tid = threadIdx.x;
  uint32_t v = 0;
#pragma unroll
  for (int i = 0; i < PARTS; ++i) {
    const uint32_t column = h[i] | static_cast<uint32_t>(__shfl_xor(static_cast<int>(h[i]), 32, 64));
    v ^= gf_mul_dev(pos[(tid + i * threads) | 32], column);
  }
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) v ^= static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), off, 64));
  if ((tid & 63) == 0) l.seg[tid >> 6] = v;
  __syncthreads();
  uint32_t raw = 0;
#pragma unroll
  for (int w = 0; w < threads / 64; ++w) raw ^= l.seg[w];
  __syncthreads();  // seg may be reused by the caller
  return raw;
}

__device__ __forceinline__ uint32_t fold_columns(ChunkLds& l, const uint32_t* pos, uint32_t h) {
  const uint32_t one[1] = {h};
  return fold_columns<1>(l, pos, one);
}

// Fold one value per thread, thread t's piece followed by the pieces of threads
// t + 1 .. 1023.  The raw register value is returned in every thread.
__device__ uint32_t fold_pos(uint32_t* seg, const uint32_t* pos, uint32_t h) {
  const int tid = threadIdx.x;
  uint32_t v = gf_mul_dev(pos[tid], h);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v ^= static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), off, 64));
  if ((tid & 63) == 0) seg[tid >> 6] = v;
  __syncthreads();
  uint32_t raw = 0;
#pragma unroll
  for (int w = 0; w < kCrcThreads / 64; ++w) raw ^= seg[w];
  __syncthreads();  // seg may be reused by the caller
  return raw;
}

// zlib's CRC-32 of a message of x_len = x^(8 len) from its raw register value
__host__ __device__ inline uint32_t crc_from_raw(uint32_t x_len, uint32_t raw) {
  return gf_mul(x_len, 0xFFFFFFFFu) ^ raw ^ 0xFFFFFFFFu;
}

// Fold the column states of a payload: its zlib CRC-32, returned in every thread.
__device__ uint32_t fold_chunks(ChunkLds& l, const ChunkPlan& c, uint32_t h) {
  return crc_from_raw(c.x_len, fold_columns(l, kPosTables.chunk, h));
}

}  // namespace
}  // namespace kvssd
