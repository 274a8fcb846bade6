// GPU codec of the v1 KV block record (src/kvssd/format.py:14-177):
//
// * gather: raw records (as read from the store, copied to HBM in one span)
//   -> the PackedBatch arrays, with decode_record's header, layout and
//   payload CRC-32 checks (format.py:134-177); replaces the loader's per-block
//   payload clones and the pipeline's per-array stacking
//   (src/kvssd/loader.py:73-91, src/kvssd/pipeline.py:98-108);
// * quantize: bit-exact twin of quantize_tensor (src/kvssd/quant.py:49-65);
// * encode: KVCacheStore.create's block loop for one layer (zero-padded last
//   block, src/kvssd/store.py:46-63) -- quantise keys and values and write
//   whole records with their CRC-32 (encode_record, format.py:104-131); one
//   fused kernel for the common layouts, else a payload and a header pass.
//
// CRC-32 machinery (zlib's CRC, chunked and general forms): crc32.hpp.
#include "crc32.hpp"
#include "decode.hpp"

namespace kvssd {
namespace {

constexpr int kHeaderBytes = 52;      // "<8sIIIIIIIIIII"
constexpr int kRecordAlign = 4096;
constexpr uint32_t kMagic0 = 0x5353564Bu;  // "KVSS", little-endian
constexpr uint32_t kMagic1 = 0x31303044u;  // "D001"

// bytes [0, len) from src to dst, dwords when both ends allow
__device__ __forceinline__ void copy_region(const uint8_t* src, uint8_t* dst, int64_t len) {
  if (((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) | static_cast<uintptr_t>(len)) & 3u) == 0) {
    const uint32_t* s = reinterpret_cast<const uint32_t*>(src);
    uint32_t* d = reinterpret_cast<uint32_t*>(dst);
    for (int64_t i = threadIdx.x; i < len / 4; i += blockDim.x) d[i] = s[i];
  } else {
    for (int64_t i = threadIdx.x; i < len; i += blockDim.x) dst[i] = src[i];
  }
}

struct Layout {
  int bits, block_tokens, kv_heads, head_dim, group_size;
  __host__ __device__ int64_t scale_bytes() const { return static_cast<int64_t>(block_tokens) * kv_heads * (head_dim / group_size) * 2; }
  __host__ __device__ int64_t packed_bytes() const { return static_cast<int64_t>(block_tokens) * kv_heads * head_dim * bits / 8; }
  __host__ __device__ int64_t payload_bytes() const { return 2 * scale_bytes() + 2 * packed_bytes(); }
  __host__ __device__ int64_t record_bytes() const {
    const int64_t n = kHeaderBytes + payload_bytes();
    return (n + kRecordAlign - 1) / kRecordAlign * kRecordAlign;
  }
};

// ------------------------------------------------------------------ gather ---
struct GatherParams {
  const uint8_t* records;
  int64_t stride;
  const int32_t* rows;  // record r lies in row rows[r] of num_records; nullptr: in row r
  int n, num_records, verify;
  Layout lay;
  CrcPlan plan;
  uint8_t *pk, *pv, *sk, *sv;
  int32_t* valid;
  int32_t* status;
};

// record r's bytes, or nullptr for a row outside the records
__device__ __forceinline__ const uint8_t* record_of(const GatherParams& p, int r) {
  int row = r;
  if (p.rows != nullptr) {
    row = p.rows[r];
    if (static_cast<uint32_t>(row) >= static_cast<uint32_t>(p.num_records)) return nullptr;
  }
  return p.records + static_cast<int64_t>(row) * p.stride;
}

// a record that is not there: bad header, no valid token
__device__ __forceinline__ void reject_row(const GatherParams& p, int r) {
  p.status[r] = 1;
  p.valid[r] = 0;
}

__device__ __forceinline__ int header_status(const uint32_t* hdr, const Layout& lay) {
  if (hdr[0] != kMagic0 || hdr[1] != kMagic1 || hdr[2] != 1u) return 1;
  if (hdr[6] != static_cast<uint32_t>(lay.bits) || hdr[7] != static_cast<uint32_t>(lay.block_tokens) ||
      hdr[8] != static_cast<uint32_t>(lay.kv_heads) || hdr[9] != static_cast<uint32_t>(lay.head_dim) ||
      hdr[10] != static_cast<uint32_t>(lay.group_size))
    return 2;
  return 0;
}

// one workgroup per record; status: 0 ok, 1 invalid header (magic / version),
// 2 layout differs from the expected one, 3 payload length or CRC mismatch
__global__ __launch_bounds__(kCrcThreads) void gather_records_kernel(GatherParams p) {
  __shared__ uint32_t tab[4][256];
  __shared__ uint32_t seg[kCrcThreads];
  __shared__ uint32_t hdr[kHeaderBytes / 4];
  const int r = blockIdx.x;
  const uint8_t* rec = record_of(p, r);
  if (rec == nullptr) {
    if (threadIdx.x == 0) reject_row(p, r);
    return;
  }
  fill_crc_tables(tab);
  if (threadIdx.x < kHeaderBytes / 4) hdr[threadIdx.x] = reinterpret_cast<const uint32_t*>(rec)[threadIdx.x];
  __syncthreads();
  int status = header_status(hdr, p.lay);
  const int64_t s = p.lay.scale_bytes(), pb = p.lay.packed_bytes();
  const uint8_t* pay = rec + kHeaderBytes;
  copy_region(pay, p.sk + r * s, s);
  copy_region(pay + s, p.sv + r * s, s);
  copy_region(pay + 2 * s, p.pk + r * pb, pb);
  copy_region(pay + 2 * s + pb, p.pv + r * pb, pb);
  if (p.verify && status == 0) {
    // a record written for this layout has exactly the layout's payload
    if (hdr[11] != p.plan.len) {
      status = 3;
    } else {
      const uint32_t crc = block_crc32(pay, p.plan, tab, seg);
      if (crc != hdr[12]) status = 3;
    }
  }
  if (threadIdx.x == 0) {
    p.status[r] = status;
    p.valid[r] = static_cast<int32_t>(hdr[5]);
  }
}

// chunked form of gather_records_kernel (same statuses), for layouts whose
// four arrays are 16-byte multiples and 16-byte aligned destinations.  Each
// thread takes its chunks four rows at a time, from memory to the arrays and
// through the CRC, in at most 64 registers: two workgroups share a CU, and the
// loads of some waves cover the matrix work of the others.  The records may lie
// in page-locked host memory: every byte is read once (128 records of 148 KiB
// over PCIe: 389 us, 50 GB/s; 1,024: 55 GB/s, a copy engine's 57).
__global__ __launch_bounds__(kCrcThreads, 8) void gather_chunked_kernel(GatherParams p, ChunkPlan c) {
  __shared__ ChunkLds lds;
  __shared__ uint32_t hdr[kHeaderBytes / 4];
  const int r = blockIdx.x;
  const uint8_t* rec = record_of(p, r);
  if (rec == nullptr) {
    if (threadIdx.x == 0) reject_row(p, r);
    return;
  }
  const uint8_t* pay = rec + kHeaderBytes;
  if (threadIdx.x < kHeaderBytes / 4) hdr[threadIdx.x] = reinterpret_cast<const uint32_t*>(rec)[threadIdx.x];
  if (p.verify) load_chunk_tables(lds);
  __syncthreads();
  const int64_t sb = p.lay.scale_bytes(), pb = p.lay.packed_bytes();
  uint32_t h = 0;
  const int lead = (kGroupRows - c.rows % kGroupRows) % kGroupRows;  // zero rows of the first group
  for (int j0 = -lead; j0 < c.rows; j0 += kGroupRows) {
    u32x4 v[kGroupRows];
#pragma unroll
    for (int j = 0; j < kGroupRows; ++j) {
      v[j] = u32x4{0u, 0u, 0u, 0u};
      const int64_t o = chunk_offset(c, j0 + j);
      if (o >= 0) v[j] = load16(pay + o);
    }
#pragma unroll
    for (int j = 0; j < kGroupRows; ++j) {
      const int64_t o = chunk_offset(c, j0 + j);
      if (o >= 0) {
        uint8_t* dst;
        if (o < sb) dst = p.sk + r * sb + o;
        else if (o < 2 * sb) dst = p.sv + r * sb + (o - sb);
        else if (o < 2 * sb + pb) dst = p.pk + r * pb + (o - 2 * sb);
        else dst = p.pv + r * pb + (o - 2 * sb - pb);
        *reinterpret_cast<u32x4*>(dst) = v[j];
      }
    }
    if (p.verify) h = crc_group(lds, h, v, j0 < 0 ? -j0 : 0);
  }
  int status = header_status(hdr, p.lay);
  // status, p.verify and the header are the same in every thread, so the
  // fold's barriers are reached by the whole workgroup or by none of it
  if (p.verify && status == 0) {
    if (hdr[11] != p.plan.len || fold_chunks(lds, c, h) != hdr[12]) status = 3;
  }
  if (threadIdx.x == 0) {
    p.status[r] = status;
    p.valid[r] = static_cast<int32_t>(hdr[5]);
  }
}

// ---------------------------------------------------------------- quantize ---
template <typename T>
__device__ __forceinline__ float to_f32(T v) {
  return static_cast<float>(v);
}
template <>
__device__ __forceinline__ float to_f32<uint16_t>(uint16_t v) {  // bfloat16 bits
  return __builtin_bit_cast(float, static_cast<uint32_t>(v) << 16);
}

// one group (group_size consecutive values) -> packed bytes + fp16 scale, as
// quantize_tensor: scale32 = max|x| (at least 1e-8) / (2^(bits-1) - 1) with
// IEEE division, code = clamp(rint(x / scale32), -mid, mid - 1) + mid, codes
// packed low bits first, scale stored as fp16 (round to nearest even).  A
// null src reads zeros (padding tokens).
template <typename T>
__device__ __forceinline__ void quantize_group(const T* src, int group_size, int bits, uint8_t* packed, uint16_t* scale) {
  float amax = 0.0f;
  for (int i = 0; i < group_size; ++i) amax = fmaxf(amax, fabsf(src ? to_f32(src[i]) : 0.0f));
  const int mid = 1 << (bits - 1);
  const float s32 = fmaxf(amax, 1e-8f) / static_cast<float>(mid - 1);
  const int per = 8 / bits;
  for (int b = 0; b < group_size / per; ++b) {
    uint32_t byte = 0;
    for (int j = 0; j < per; ++j) {
      const float x = src ? to_f32(src[b * per + j]) : 0.0f;
      const float c = fminf(fmaxf(rintf(x / s32), static_cast<float>(-mid)), static_cast<float>(mid - 1));
      byte |= static_cast<uint32_t>(static_cast<int>(c) + mid) << (j * bits);
    }
    packed[b] = static_cast<uint8_t>(byte);
  }
  *scale = __builtin_bit_cast(uint16_t, static_cast<_Float16>(s32));
}

constexpr int kRegGroup = 32;  // the fused encode's group size

// A word of codes, low bits first: clamp(rint(x / s32), -mid, mid - 1) + mid
// with x / s32 rounded as IEEE division does, |x| <= (mid - 1) s32 (1 + 2^-23) or
// x NaN (code 0).  Two roundings around a reciprocal stand in for the division
// (~12 instructions a value):
// * 16-bit values: q = x r, then q + (x - q s32) r, off x / s32 by at most
//   2^-46 relative before its own rounding.  The codes could then differ only
//   where x / s32 lies that close to half an ulp off some k + 0.5; with x and
//   the group's largest value in 16 bits, both quotients in question are at
//   least 2^-38 apart (checked over every such pair in float16 and bfloat16);
// * 32-bit values: q = x r is off by less than 2^-19, so that its nearest
//   integer is right unless q lies within 2^-18 of some k + 0.5; then, and for
//   scales whose reciprocal is subnormal or zero, the division itself.
// Only the division's form needs the clamp, for NaN: a NaN shows in the sums.
template <typename T, int BITS>
__device__ __forceinline__ uint32_t code_word(const float (&x)[32 / BITS], float s32) {
  constexpr int kCodes = 32 / BITS, n = kCodes / 2;
  constexpr float mid = static_cast<float>(1 << (BITS - 1));
  constexpr float radix = static_cast<float>(1 << BITS);
  float half[2];  // 16 bits at a time as an exact float sum
  bool done = false;
  if (s32 < 0x1p120f) {
    const float r0 = __builtin_amdgcn_rcpf(s32);
    const float r = __builtin_fmaf(__builtin_fmaf(-s32, r0, 1.0f), r0, r0);
    float off = 0.0f;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float t = 0.0f;
#pragma unroll
      for (int i = n - 1; i >= 0; --i) {
        const float v = x[k * n + i];
        float q = v * r;
        if constexpr (sizeof(T) == 2) q = __builtin_fmaf(__builtin_fmaf(-q, s32, v), r, q);
        const float c = rintf(q);  // within +-(mid - 1), or NaN, and then so is the sum
        if constexpr (sizeof(T) != 2) off = fmaxf(off, fabsf(q - c));
        t = i == n - 1 ? c : __builtin_fmaf(t, radix, c);
      }
      half[k] = t + static_cast<float>(BITS == 4 ? 0x8888 : 0xAAAA);  // mid for every code
    }
    done = half[0] == half[0] && half[1] == half[1] && (sizeof(T) == 2 || off < 0.5f - 0x1p-18f);
  }
  if (!done) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      half[k] = 0.0f;
#pragma unroll
      for (int i = n - 1; i >= 0; --i)
        half[k] = __builtin_fmaf(half[k], radix, fminf(fmaxf(rintf(x[k * n + i] / s32), -mid), mid - 1.0f) + mid);
    }
  }
  return static_cast<uint32_t>(half[0]) | (static_cast<uint32_t>(half[1]) << 16);
}

// max(amax, 1e-8) / (mid - 1), IEEE: a quotient by 7 lies at least 1/14 ulp from
// the middle of two floats, which two roundings around 1/7 resolve (checked over
// every mantissa); large values, where the remainder may not be finite, divide.
template <int BITS>
__device__ __forceinline__ float group_scale(float amax) {
  const float a = fmaxf(amax, 1e-8f);
  if constexpr (BITS == 2) return a;
  if (!(a < 0x1p120f)) return a / 7.0f;
  const float q = a * (1.0f / 7.0f);
  return __builtin_fmaf(__builtin_fmaf(-7.0f, q, a), 1.0f / 7.0f, q);
}

template <int CTRL>
__device__ __forceinline__ float max_across(float v) {
  return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true)));
}

// largest of v over each run of `lanes` (a power of two) lanes
__device__ __forceinline__ float lanes_max(float v, int lanes) {
  if (lanes > 1) v = max_across<0xB1>(v);    // lane ^ 1
  if (lanes > 2) v = max_across<0x4E>(v);    // lane ^ 2
  if (lanes > 4) v = max_across<0x141>(v);   // the other quad of 8
  if (lanes > 8) v = max_across<0x140>(v);   // the other half of 16
  for (int m = 16; m < lanes; m <<= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
  return v;
}

// The word form: a lane takes the 8 (INT4) or 16 (INT2) values of one word of
// codes, `lanes` of them (a power of two) a group, so that loads and stores are
// contiguous over the wave.  Measured (131,072 x 8 x
// 128 bfloat16 keys and values into records, INT4): groups of 64, which went
// through a thread a group with a load per value, 10.2 -> 0.23 ms; groups of 32
// in 32-token blocks, before by a lane a group in registers, 0.31 -> 0.26 ms.
template <typename T, int BITS>
__device__ __forceinline__ void quantize_word(const T* src, int lanes, uint8_t* packed, uint16_t* scale) {
  constexpr int kVals = 32 / BITS;
  float x[kVals], amax = 0.0f;
  if (src != nullptr) {
    T v[kVals];
    __builtin_memcpy(v, __builtin_assume_aligned(src, 16), sizeof(v));
#pragma unroll
    for (int i = 0; i < kVals; ++i) x[i] = to_f32(v[i]);
  } else {
#pragma unroll
    for (int i = 0; i < kVals; ++i) x[i] = 0.0f;
  }
#pragma unroll
  for (int i = 0; i < kVals; ++i) amax = fmaxf(amax, fabsf(x[i]));
  const float s32 = group_scale<BITS>(lanes_max(amax, lanes));
  const uint32_t word = code_word<T, BITS>(x, s32);
  __builtin_memcpy(__builtin_assume_aligned(packed, 4), &word, 4);
  if ((threadIdx.x & (lanes - 1)) == 0) *scale = __builtin_bit_cast(uint16_t, static_cast<_Float16>(s32));
}

// lanes of a group in the word form, 0 where it does not apply: whole words, a
// power of two of them within a wave
inline int word_lanes(int group_size, int bits) {
  const int lanes = group_size * bits % 32 == 0 ? group_size * bits / 32 : 0;
  return lanes <= 64 && (lanes & (lanes - 1)) == 0 ? lanes : 0;
}

// lanes == 0: a thread a group, any size and alignment (quantize_group);
// else the word form, a thread a word
template <typename T, int BITS>
__global__ __launch_bounds__(256) void quantize_kernel(const T* __restrict__ x, int64_t count, int group_size, int lanes,
                                                       uint8_t* __restrict__ packed, uint16_t* __restrict__ scales) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  if (lanes == 0) {
    quantize_group(x + i * group_size, group_size, BITS, packed + i * (group_size * BITS / 8), scales + i);
  } else {
    quantize_word<T, BITS>(x + i * (32 / BITS), lanes, packed + 4 * i, scales + i / lanes);
  }
}

// ------------------------------------------------------------------ encode ---
struct EncodeParams {
  const void* keys;
  const void* values;
  int64_t tokens;
  int n, layer, first_block;
  Layout lay;
  CrcPlan plan;
  uint8_t* records;
  uint32_t* crcs;
};

// phase 1: every (record, key/value, token, kv head, group) quantised into
// the record's payload; tokens past the end read as zeros.
template <typename T>
__global__ __launch_bounds__(256) void encode_payload_kernel(EncodeParams p) {
  const Layout& L = p.lay;
  const int G = L.head_dim / L.group_size;
  const int64_t per_record = static_cast<int64_t>(L.block_tokens) * L.kv_heads * G;  // groups per array
  const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= 2 * per_record * p.n) return;
  const int r = static_cast<int>(g / (2 * per_record));
  const int64_t rest = g % (2 * per_record);
  const bool is_v = rest >= per_record;
  const int64_t q = is_v ? rest - per_record : rest;  // (token, head, group) within the block
  const int64_t row = q / G;                          // token * kv_heads + head
  const int gi = static_cast<int>(q % G);
  const int64_t token = static_cast<int64_t>(r) * L.block_tokens + row / L.kv_heads;
  const T* base = static_cast<const T*>(is_v ? p.values : p.keys);
  const T* src = token < p.tokens ? base + (token * L.kv_heads + row % L.kv_heads) * L.head_dim + gi * L.group_size
                                  : nullptr;
  uint8_t* pay = p.records + static_cast<int64_t>(r) * L.record_bytes() + kHeaderBytes;
  const int64_t s = L.scale_bytes(), pb = L.packed_bytes();
  uint16_t* scale = reinterpret_cast<uint16_t*>(pay + (is_v ? s : 0)) + q;
  uint8_t* packed = pay + 2 * s + (is_v ? pb : 0) + q * (L.group_size * L.bits / 8);
  quantize_group(src, L.group_size, L.bits, packed, scale);
}

// phase 1 in the word form: grid y is (record, key/value), whose values and
// words lie in one run each
template <typename T, int BITS>
__global__ __launch_bounds__(256) void encode_words_kernel(EncodeParams p, int lanes) {
  const Layout& L = p.lay;
  const int64_t w = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;  // of the array
  const int64_t s = L.scale_bytes(), pb = L.packed_bytes();
  if (4 * w >= pb) return;
  const int r = static_cast<int>(blockIdx.y >> 1);
  const bool is_v = blockIdx.y & 1;
  const int64_t row = static_cast<int64_t>(L.kv_heads) * L.head_dim;
  const int64_t at = r * (L.block_tokens * row) + w * (32 / BITS);  // of the layer's values
  const T* base = static_cast<const T*>(is_v ? p.values : p.keys);
  uint8_t* pay = p.records + static_cast<int64_t>(r) * L.record_bytes() + kHeaderBytes;
  quantize_word<T, BITS>(at < p.tokens * row ? base + at : nullptr, lanes, pay + 2 * s + (is_v ? pb : 0) + 4 * w,
                         reinterpret_cast<uint16_t*>(pay + (is_v ? s : 0)) + w / lanes);
}

// phase 2: one workgroup per record -- CRC of the payload, header, padding.
// CHUNKED: the payload is a 16-byte multiple.
struct WalkLds {
  uint32_t tab[4][256];
  uint32_t seg[kCrcThreads];
};

template <bool CHUNKED>
__global__ __launch_bounds__(kCrcThreads) void encode_header_kernel(EncodeParams p, ChunkPlan c) {
  __shared__ union {
    ChunkLds lds;
    WalkLds walk;
  } shared;
  ChunkLds& lds = shared.lds;
  WalkLds& walk = shared.walk;
  const Layout& L = p.lay;
  const int r = blockIdx.x;
  uint8_t* rec = p.records + static_cast<int64_t>(r) * L.record_bytes();
  uint32_t crc;
  if constexpr (CHUNKED) {
    const uint8_t* pay = rec + kHeaderBytes;
    load_chunk_tables(lds);
    __syncthreads();
    uint32_t h = 0;
    const int lead = (kGroupRows - c.rows % kGroupRows) % kGroupRows;
    for (int j0 = -lead; j0 < c.rows; j0 += kGroupRows) {
      u32x4 v[kGroupRows];
#pragma unroll
      for (int j = 0; j < kGroupRows; ++j) {
        v[j] = u32x4{0u, 0u, 0u, 0u};
        const int64_t o = chunk_offset(c, j0 + j);
        if (o >= 0) v[j] = load16(pay + o);
      }
      h = crc_group(lds, h, v, j0 < 0 ? -j0 : 0);
    }
    crc = fold_chunks(lds, c, h);
  } else {
    fill_crc_tables(walk.tab);
    __syncthreads();
    crc = block_crc32(rec + kHeaderBytes, p.plan, walk.tab, walk.seg);
  }
  const int64_t start = static_cast<int64_t>(r) * L.block_tokens;
  const int64_t valid = p.tokens - start < L.block_tokens ? p.tokens - start : L.block_tokens;
  if (threadIdx.x < kHeaderBytes / 4) {
    uint32_t v = 0;
    switch (threadIdx.x) {
      case 0: v = kMagic0; break;
      case 1: v = kMagic1; break;
      case 2: v = 1u; break;
      case 3: v = static_cast<uint32_t>(p.layer); break;
      case 4: v = static_cast<uint32_t>(p.first_block + r); break;
      case 5: v = static_cast<uint32_t>(valid); break;
      case 6: v = static_cast<uint32_t>(L.bits); break;
      case 7: v = static_cast<uint32_t>(L.block_tokens); break;
      case 8: v = static_cast<uint32_t>(L.kv_heads); break;
      case 9: v = static_cast<uint32_t>(L.head_dim); break;
      case 10: v = static_cast<uint32_t>(L.group_size); break;
      case 11: v = p.plan.len; break;
      default: v = crc; break;
    }
    reinterpret_cast<uint32_t*>(rec)[threadIdx.x] = v;
  }
  for (int64_t i = kHeaderBytes + L.payload_bytes() + threadIdx.x; i < L.record_bytes(); i += blockDim.x) rec[i] = 0;
  if (threadIdx.x == 0) p.crcs[r] = crc;
}

// One kernel for the common layout (group size 32, the scale region [Ks | Vs]
// and the code region [Kc | Vc] each a whole number of 16 KiB rows of the
// chunked CRC form, so no virtual zeros): one workgroup of 1024 threads per
// record.  A record's codes are those of its keys, then its values, in memory
// order, so wave w of code row k takes the 1 KiB piece 16 k + w as four runs of
// 64 words: a lane reads the 8 (INT4) or 16 (INT2) values of its word, a group
// is 4 or 2 lanes, loads and stores are contiguous over the wave, and the words
// go through the CRC in its dword layout as they are made.  The scales collect
// in LDS; after a barrier they are stored and take a CRC of their own, moved
// before the codes' by one multiply, so the payload is never read back.
// Measured (1,024 records of 8 kv heads, head_dim 128, bfloat16, 688 MB moved):
// a lane a group, reading 64 bytes of its own, and IEEE divisions 222 us, 166
// us in this form.
struct FusedPlan {
  int rows_s, rows_c;  // rows of scale / code chunks
  uint32_t x_codes;    // x^(8 * code bytes) mod P
};

constexpr int kComputeUnits = 256;
constexpr int kLdsBytes = 160 * 1024;  // of a CU
constexpr int kMaxScaleRows = kGroupRows;  // scale region <= 64 KiB of LDS, one group of rows

// PARTS: the workgroup has 1024 / PARTS threads, each taking the parts of PARTS
// in turn.
template <typename T, int BITS, int PARTS>
__global__ __launch_bounds__(kCrcThreads / PARTS) void encode_fused_kernel(EncodeParams p, ChunkPlan c, FusedPlan f) {
  constexpr int kThreads = kCrcThreads / PARTS;
  __shared__ ChunkLds lds;
  extern __shared__ __attribute__((aligned(16))) uint16_t scales[];  // the record's scale region
  constexpr int kVals = 32 / BITS;                                   // values of a word of codes
  constexpr int kRunBytes = 64 * 4;
  constexpr int kRaw = kVals * static_cast<int>(sizeof(T)) / 4;      // dwords of those values
  constexpr int kAhead = kRaw <= 4 ? 4 : kRaw <= 8 ? 2 : 1;          // runs loaded at a time
  const Layout& L = p.lay;
  const int r = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  uint8_t* rec = p.records + static_cast<int64_t>(r) * L.record_bytes();
  uint8_t* pay = rec + kHeaderBytes;
  const int64_t code0 = 2 * L.scale_bytes(), array = L.packed_bytes();
  // the record's first value of keys and of values, and how many follow before the last token's end
  const int64_t block = static_cast<int64_t>(L.block_tokens) * L.kv_heads * L.head_dim;
  const int64_t left = p.tokens * L.kv_heads * L.head_dim - r * block;
  // the values of runs u0 .. u0 + kAhead - 1 of code row k's piece
  auto piece_of = [&](int k, int part) {
    return (static_cast<int64_t>(k) * kCrcThreads + part * kThreads + (tid & ~63)) * kChunkBytes;
  };
  auto load_runs = [&](int k, int part, int u0, uint32_t (&raw)[kAhead][kRaw]) {
    // codes of keys or of values (arrays are whole pieces)
    const int64_t piece = piece_of(k, part);
    const bool is_v = piece >= array;
    const T* base = static_cast<const T*>(is_v ? p.values : p.keys) + r * block;
    const int64_t at = (is_v ? piece - array : piece) * (8 / BITS) + lane * kVals;  // of the block's values
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      const int64_t e = at + (u0 + a) * 64 * kVals;
      const bool in = e < left;
      __builtin_memcpy(raw[a], __builtin_assume_aligned(base + (in ? e : 0), 16), sizeof(raw[a]));
#pragma unroll
      for (int i = 0; i < kRaw; ++i) raw[a][i] = in ? raw[a][i] : 0u;  // tokens past the end are zeros
    }
  };
  uint32_t next[kAhead][kRaw];
  load_runs(0, 0, 0, next);
  load_chunk_tables<PARTS>(lds, kWordMatrices);
  __syncthreads();  // the CRC matrices are in LDS
  uint32_t codes[PARTS], sums[PARTS];  // column states of the codes, of the scales
  const int lead = (kGroupRows - f.rows_c % kGroupRows) % kGroupRows;  // zero rows of the first group
#pragma unroll 1
  for (int part = 0; part < PARTS; ++part) {
    uint32_t h = 0;
    for (int k0 = -lead; k0 < f.rows_c; k0 += kGroupRows) {
      f32x16 acc = crc_begin(lds, h);
#pragma unroll 1
      for (int j = k0 < 0 ? -k0 : 0; j < kGroupRows; ++j) {
        const int k = k0 + j;
        const int64_t piece = piece_of(k, part);
        u32x4 words;
#pragma unroll
        for (int u0 = 0; u0 < 4; u0 += kAhead) {
          uint32_t raw[kAhead][kRaw];
          __builtin_memcpy(raw, next, sizeof(raw));
          // the next runs' loads are in flight while these are quantised
          if (u0 + kAhead < 4) load_runs(k, part, u0 + kAhead, next);
          else if (k + 1 < f.rows_c) load_runs(k + 1, part, 0, next);
          else if (part + 1 < PARTS) load_runs(0, part + 1, 0, next);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int a = 0; a < kAhead; ++a) {
            const int u = u0 + a;
            T v[kVals];
            __builtin_memcpy(v, raw[a], sizeof(v));
            float x[kVals], amax = 0.0f;
#pragma unroll
            for (int i = 0; i < kVals; ++i) {
              x[i] = to_f32(v[i]);
              amax = fmaxf(amax, fabsf(x[i]));
            }
            const float s32 = group_scale<BITS>(lanes_max(amax, BITS));
            const uint32_t word = code_word<T, BITS>(x, s32);
            words[u] = word;
            if ((lane & (BITS - 1)) == 0)
              scales[piece / (4 * BITS) + u * (64 / BITS) + lane / BITS] =
                  __builtin_bit_cast(uint16_t, static_cast<_Float16>(s32));
            __builtin_memcpy(__builtin_assume_aligned(pay + code0 + piece + u * kRunBytes + 4 * lane, 4), &word, 4);
            __builtin_amdgcn_sched_barrier(0);  // (runs quantised side by side would not fit the registers)
          }
        }
        acc = crc_row(lds, acc, j, words);
      }
      h = crc_end(acc);
    }
    if (part == 0) codes[0] = h;
    else codes[PARTS - 1] = h;
  }
  __syncthreads();  // every scale is in LDS
#pragma unroll
  for (int part = 0; part < PARTS; ++part) {
    u32x4 v[kGroupRows];
#pragma unroll
    for (int j = 0; j < kGroupRows; ++j) {
      v[j] = u32x4{0u, 0u, 0u, 0u};
      const int row = j + f.rows_s - kGroupRows;
      if (row >= 0) {
        const int64_t piece = piece_of(row, part);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t word = reinterpret_cast<const uint32_t*>(scales)[piece / 4 + u * 64 + lane];
          __builtin_memcpy(__builtin_assume_aligned(pay + piece + u * kRunBytes + 4 * lane, 4), &word, 4);
          v[j][u] = word;
        }
      }
    }
    sums[part] = crc_group(lds, 0u, v, kGroupRows - f.rows_s);
  }
  // the scales come before the codes in the message
  const uint32_t raw_s = fold_columns<PARTS>(lds, kPosTables.word, sums);
  const uint32_t raw_c = fold_columns<PARTS>(lds, kPosTables.word, codes);
  const uint32_t crc = crc_from_raw(c.x_len, gf_mul_dev(f.x_codes, raw_s) ^ raw_c);
  const int64_t start = static_cast<int64_t>(r) * L.block_tokens;
  const int64_t valid = p.tokens - start < L.block_tokens ? p.tokens - start : L.block_tokens;
  if (tid < kHeaderBytes / 4) {
    uint32_t v = 0;
    switch (tid) {
      case 0: v = kMagic0; break;
      case 1: v = kMagic1; break;
      case 2: v = 1u; break;
      case 3: v = static_cast<uint32_t>(p.layer); break;
      case 4: v = static_cast<uint32_t>(p.first_block + r); break;
      case 5: v = static_cast<uint32_t>(valid); break;
      case 6: v = static_cast<uint32_t>(L.bits); break;
      case 7: v = static_cast<uint32_t>(L.block_tokens); break;
      case 8: v = static_cast<uint32_t>(L.kv_heads); break;
      case 9: v = static_cast<uint32_t>(L.head_dim); break;
      case 10: v = static_cast<uint32_t>(L.group_size); break;
      case 11: v = p.plan.len; break;
      default: v = crc; break;
    }
    reinterpret_cast<uint32_t*>(rec)[tid] = v;
  }
  for (int64_t i = kHeaderBytes + L.payload_bytes() + tid; i < L.record_bytes(); i += kThreads) rec[i] = 0;
  if (tid == 0) p.crcs[r] = crc;
}

// the fused form applies: scale and code
// regions whole rows of the chunked CRC form, scales within the LDS copy
bool fused_layout(const Layout& L, FusedPlan* f) {
  const int64_t sr = 2 * L.scale_bytes(), cr = 2 * L.packed_bytes();
  if (L.group_size != kRegGroup || sr % kStrideBytes || cr % kStrideBytes) return false;
  f->rows_s = static_cast<int>(sr / kStrideBytes);
  f->rows_c = static_cast<int>(cr / kStrideBytes);
  f->x_codes = x_pow_bytes(static_cast<uint64_t>(cr));
  return f->rows_s >= 1 && f->rows_s <= kMaxScaleRows && f->rows_c >= 1;
}

// the chunked CRC / gather form applies: all four arrays 16-byte multiples
bool chunked_layout(const Layout& L) {
  return L.scale_bytes() % kChunkBytes == 0 && L.packed_bytes() % kChunkBytes == 0;
}

int check_layout(const kvssd_record_layout* l, Layout* out) {
  if (l == nullptr) return arg_error("record layout is NULL");
  if (l->bits != 2 && l->bits != 4) return arg_error("bits must be 2 or 4");
  if (l->block_tokens <= 0 || l->kv_heads <= 0 || l->head_dim <= 0)
    return arg_error("all cache dimensions must be positive");
  if (l->group_size <= 0 || l->head_dim % l->group_size) return arg_error("head_dim must be divisible by group_size");
  if (l->group_size % (8 / l->bits)) return arg_error("group_size must be positive and pack-aligned");
  *out = Layout{l->bits, l->block_tokens, l->kv_heads, l->head_dim, l->group_size};
  if (out->payload_bytes() > 0x7FFFFFFFLL) return arg_error("record payload too large");
  return 0;
}

// the word form's loads and stores: a 16-byte aligned source, 4-byte aligned codes
inline bool word_aligned(const void* src, const void* packed) {
  return (reinterpret_cast<uintptr_t>(src) & 15u) == 0 && (reinterpret_cast<uintptr_t>(packed) & 3u) == 0;
}

// threads of one launch, 2^34 INT4 values of the word form (a grid holds less than 2^32
// of them, and of one of more only the rest runs, without an error)
constexpr int64_t kMaxThreads = int64_t{1} << 31;

template <typename T>
void launch_quantize_t(const void* x, int64_t groups, int group_size, int bits, uint8_t* packed, uint16_t* scales,
                       hipStream_t s) {
  const int lanes = word_aligned(x, packed) ? word_lanes(group_size, bits) : 0;
  const int64_t most = lanes > 0 ? kMaxThreads / lanes : kMaxThreads;  // (lanes is a power of two)
  for (int64_t g0 = 0; g0 < groups; g0 += most) {
    const int64_t n = groups - g0 < most ? groups - g0 : most;
    const int64_t count = lanes > 0 ? n * lanes : n;
    const dim3 grid(static_cast<unsigned>((count + 255) / 256));
    const T* src = static_cast<const T*>(x) + g0 * group_size;
    uint8_t* codes = packed + g0 * (group_size * bits / 8);
    if (bits == 4)
      hipLaunchKernelGGL((quantize_kernel<T, 4>), grid, dim3(256), 0, s, src, count, group_size, lanes, codes, scales + g0);
    else
      hipLaunchKernelGGL((quantize_kernel<T, 2>), grid, dim3(256), 0, s, src, count, group_size, lanes, codes, scales + g0);
  }
}

template <typename T, int PARTS>
void launch_fused_parts(const EncodeParams& p, const ChunkPlan& c, const FusedPlan& f, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(p.n));
  const size_t scale_lds = static_cast<size_t>(2 * p.lay.scale_bytes());
  if (p.lay.bits == 4)
    hipLaunchKernelGGL((encode_fused_kernel<T, 4, PARTS>), grid, dim3(kCrcThreads / PARTS), scale_lds, s, p, c, f);
  else
    hipLaunchKernelGGL((encode_fused_kernel<T, 2, PARTS>), grid, dim3(kCrcThreads / PARTS), scale_lds, s, p, c, f);
}

// Past one record per CU, workgroups of 512 threads: their registers let two
// share a CU, and one's start and end pass under the other's work (128-token
// records of 8 kv heads: 257 of them 71 -> 66 us a call, 400 79 -> 74, 1,024
// 174 -> 170).  Up to there 1024 threads finish a record sooner (256: 42 us
// against 47, 16: 33 against 37), and so they do where the LDS of two does not
// fit a CU (64 KiB of scales, 32 kv heads: 300 records 256 us against 338, 600
// 404 against 518).
template <typename T>
void launch_fused_t(const EncodeParams& p, const ChunkPlan& c, const FusedPlan& f, hipStream_t s) {
  const bool two_fit = 2 * (2 * p.lay.scale_bytes() + static_cast<int64_t>(sizeof(ChunkLds))) <= kLdsBytes;
  if (p.n > kComputeUnits && two_fit) launch_fused_parts<T, 2>(p, c, f, s);
  else launch_fused_parts<T, 1>(p, c, f, s);
}

// One workgroup a record pays off while a record is short, or where records
// fill the chip.  Past 8 code rows (8 kv heads of 128 tokens, INT4) the two
// passes, which spread a record over the chip, are faster for few records (16
// kv heads, INT4, bfloat16: 64 records 39 us against 58, 256 103 against 82;
// 32 heads: 64 64 against 102, 600 461 against 404), and at any count for INT2
// codes or fp32 values, whose quantising outweighs the payload read back (24
// kv heads, 300 records: INT2 bfloat16 124 us against 158, fp32 211 against
// 288; INT4 fp32 238 against 294).
bool fused_pays(const FusedPlan& f, int bits, int dtype, int n) {
  return f.rows_c <= 8 || (bits == 4 && dtype != KVSSD_DTYPE_F32 && n > kComputeUnits / 2);
}

// records of one launch of the word form, whose (record, key/value) pairs are
// grid y (65,535 at most): calls of more take several launches (1,048,576
// tokens in 32-token blocks, 32,768 records: 9.3 ms by a thread a group, 1.9 ms in two launches)
constexpr int kMaxWordRecords = 32767;

template <typename T>
void launch_encode_t(const EncodeParams& p, hipStream_t s) {
  const int lanes = word_lanes(p.lay.group_size, p.lay.bits);
  const int64_t row = static_cast<int64_t>(p.lay.kv_heads) * p.lay.head_dim;
  // (records are 4-byte aligned, checked; the codes after them too where the scales are whole words)
  if (lanes > 0 && word_aligned(p.keys, p.records) && word_aligned(p.values, p.records) &&
      2 * p.lay.scale_bytes() % 4 == 0 && p.lay.packed_bytes() % 4 == 0 && p.lay.block_tokens * row % 16 == 0) {
    const unsigned tiles = static_cast<unsigned>((p.lay.packed_bytes() / 4 + 255) / 256);
    for (int64_t r0 = 0; r0 < p.n; r0 += kMaxWordRecords) {
      EncodeParams slice = p;
      const int64_t skip = r0 * p.lay.block_tokens;  // tokens before the slice
      slice.n = static_cast<int>(p.n - r0 < kMaxWordRecords ? p.n - r0 : kMaxWordRecords);
      slice.tokens = p.tokens - skip;
      slice.keys = static_cast<const T*>(p.keys) + skip * row;
      slice.values = static_cast<const T*>(p.values) + skip * row;
      slice.records = p.records + r0 * p.lay.record_bytes();
      const dim3 words(tiles, static_cast<unsigned>(2 * slice.n));
      if (p.lay.bits == 4) hipLaunchKernelGGL((encode_words_kernel<T, 4>), words, dim3(256), 0, s, slice, lanes);
      else hipLaunchKernelGGL((encode_words_kernel<T, 2>), words, dim3(256), 0, s, slice, lanes);
    }
  } else {
    const int64_t groups = 2 * p.lay.block_tokens * row / p.lay.group_size * p.n;
    const dim3 grid(static_cast<unsigned>((groups + 255) / 256));
    hipLaunchKernelGGL(encode_payload_kernel<T>, grid, dim3(256), 0, s, p);
  }
}

}  // namespace

int record_bytes_of(const kvssd_record_layout* layout, size_t* bytes) {
  Layout L{};
  if (int rc = check_layout(layout, &L)) return rc;
  if (bytes == nullptr) return arg_error("bytes output pointer is NULL");
  *bytes = static_cast<size_t>(L.record_bytes());
  return 0;
}

int launch_gather_records(const kvssd_record_layout* layout, const uint8_t* records, size_t stride, int num_records,
                          const int32_t* rows, int n, int verify_crc, uint8_t* packed_k, uint8_t* packed_v, uint16_t* scales_k,
                          uint16_t* scales_v, int32_t* valid, int32_t* status, hipStream_t stream) {
  Layout L{};
  if (int rc = check_layout(layout, &L)) return rc;
  if (n < 0 || num_records < 0) return arg_error("record count must be non-negative");
  if (n == 0) return 0;
  if (rows != nullptr && reinterpret_cast<uintptr_t>(rows) % 4) return arg_error("record rows must be 4-byte aligned");
  if (!records || !packed_k || !packed_v || !scales_k || !scales_v || !valid || !status)
    return arg_error("a required buffer pointer is NULL");
  if (stride < static_cast<size_t>(L.record_bytes()) || (stride % 4) || (reinterpret_cast<uintptr_t>(records) % 4))
    return arg_error("records must be 4-byte aligned and at least record_bytes apart");
  GatherParams p{};
  p.records = records;
  p.stride = static_cast<int64_t>(stride);
  p.rows = rows;
  p.n = n;
  p.num_records = num_records;
  p.verify = verify_crc != 0;
  p.lay = L;
  p.plan = make_crc_plan(static_cast<uint32_t>(L.payload_bytes()));
  p.pk = packed_k;
  p.pv = packed_v;
  p.sk = reinterpret_cast<uint8_t*>(scales_k);
  p.sv = reinterpret_cast<uint8_t*>(scales_v);
  p.valid = valid;
  p.status = status;
  const bool aligned16 = ((reinterpret_cast<uintptr_t>(packed_k) | reinterpret_cast<uintptr_t>(packed_v) |
                           reinterpret_cast<uintptr_t>(scales_k) | reinterpret_cast<uintptr_t>(scales_v)) & 15u) == 0;
  if (aligned16 && chunked_layout(L)) {
    const ChunkPlan c = make_chunk_plan(p.plan.len);
    hipLaunchKernelGGL(gather_chunked_kernel, dim3(static_cast<unsigned>(n)), dim3(kCrcThreads), 0, stream, p, c);
  } else {
    hipLaunchKernelGGL(gather_records_kernel, dim3(static_cast<unsigned>(n)), dim3(kCrcThreads), 0, stream, p);
  }
  return hip_status(hipGetLastError(), "gather_records launch");
}

int launch_quantize(const void* x, int dtype, int64_t rows, int head_dim, int bits, int group_size, uint8_t* packed,
                    uint16_t* scales, hipStream_t stream) {
  if (bits != 2 && bits != 4) return arg_error("bits must be 2 or 4");
  if (group_size <= 0 || group_size % (8 / bits)) return arg_error("group_size must be positive and pack-aligned");
  if (head_dim <= 0 || head_dim % group_size) return arg_error("last dimension must be divisible by group_size");
  if (rows < 0) return arg_error("row count must be non-negative");
  if (rows == 0) return 0;
  if (!x || !packed || !scales) return arg_error("a required buffer pointer is NULL");
  const int64_t groups = rows * (head_dim / group_size);
  switch (dtype) {
    case KVSSD_DTYPE_F16:
      launch_quantize_t<_Float16>(x, groups, group_size, bits, packed, scales, stream);
      break;
    case KVSSD_DTYPE_BF16:
      launch_quantize_t<uint16_t>(x, groups, group_size, bits, packed, scales, stream);
      break;
    case KVSSD_DTYPE_F32:
      launch_quantize_t<float>(x, groups, group_size, bits, packed, scales, stream);
      break;
    case KVSSD_DTYPE_F64:
      launch_quantize_t<double>(x, groups, group_size, bits, packed, scales, stream);
      break;
    default:
      return arg_error("quantization input must be floating point");
  }
  return hip_status(hipGetLastError(), "quantize launch");
}

int launch_encode_records(const kvssd_record_layout* layout, int dtype, const void* keys, const void* values,
                          int64_t tokens, int layer, int first_block, uint8_t* records, uint32_t* crcs,
                          hipStream_t stream) {
  Layout L{};
  if (int rc = check_layout(layout, &L)) return rc;
  if (tokens < 0) return arg_error("token count must be non-negative");
  if (tokens == 0) return 0;
  if (!keys || !values || !records || !crcs) return arg_error("a required buffer pointer is NULL");
  if (reinterpret_cast<uintptr_t>(records) % 4) return arg_error("records must be 4-byte aligned");
  EncodeParams p{};
  p.keys = keys;
  p.values = values;
  p.tokens = tokens;
  p.n = static_cast<int>((tokens + L.block_tokens - 1) / L.block_tokens);
  p.layer = layer;
  p.first_block = first_block;
  p.lay = L;
  p.plan = make_crc_plan(static_cast<uint32_t>(L.payload_bytes()));
  p.records = records;
  p.crcs = crcs;
  const uint32_t len = p.plan.len;
  const ChunkPlan c = make_chunk_plan(len);
  FusedPlan f{};
  // (fp64 input keeps the two-kernel form: its fused INT2 instance would spill)
  if (fused_layout(L, &f) && fused_pays(f, L.bits, dtype, p.n) && word_aligned(keys, records) && word_aligned(values, records) &&
      (dtype == KVSSD_DTYPE_F16 || dtype == KVSSD_DTYPE_BF16 || dtype == KVSSD_DTYPE_F32)) {
    if (dtype == KVSSD_DTYPE_F16) launch_fused_t<_Float16>(p, c, f, stream);
    else if (dtype == KVSSD_DTYPE_BF16) launch_fused_t<uint16_t>(p, c, f, stream);
    else launch_fused_t<float>(p, c, f, stream);
    return hip_status(hipGetLastError(), "encode_records launch");
  }
  switch (dtype) {
    case KVSSD_DTYPE_F16:
      launch_encode_t<_Float16>(p, stream);
      break;
    case KVSSD_DTYPE_BF16:
      launch_encode_t<uint16_t>(p, stream);
      break;
    case KVSSD_DTYPE_F32:
      launch_encode_t<float>(p, stream);
      break;
    case KVSSD_DTYPE_F64:
      launch_encode_t<double>(p, stream);
      break;
    default:
      return arg_error("quantization input must be floating point");
  }
  if (int rc = hip_status(hipGetLastError(), "encode_records launch")) return rc;
  if (len % kChunkBytes == 0) {
    hipLaunchKernelGGL(encode_header_kernel<true>, dim3(static_cast<unsigned>(p.n)), dim3(kCrcThreads), 0, stream, p, c);
  } else {
    hipLaunchKernelGGL(encode_header_kernel<false>, dim3(static_cast<unsigned>(p.n)), dim3(kCrcThreads), 0, stream, p, c);
  }
  return hip_status(hipGetLastError(), "encode_records launch");
}

}  // namespace kvssd
