// loader.hip - delimited text (TPC-H .tbl rows) to typed columns, on the
// device.  Restates the reference's loaders (TC_data_process.cu:20-100:
// getline, strtok on the delimiter, atoi per field, one packed tuple per
// row) as two HBM passes over the text once it is resident:
//
//  1. row ends: tiles of 512 threads x 128 bytes turn the newlines into
//     bits, count them, scan the counts across the block and take the tile's
//     offset from a decoupled look-back, then store the position of every
//     newline in text order;
//  2. fields: a block of 128 rows stages their text (one contiguous span)
//     in LDS; a thread per row splits it at the delimiters; then each wave
//     converts field f of 64 rows by the type spec[f] into column f.
//
// Field conversions (C semantics): integers as atoi/atol (leading spaces,
// a sign, digits up to the first other byte; wrapping), decimals as the
// digits before and after one '.' (the value mantissa / 10^k, one IEEE
// division, so the result is the correctly rounded one while the mantissa
// stays below 2^53), dates YYYY-MM-DD as seconds since 1970 in Date.h's
// calendar, a char as its first byte.  A '\r' before the newline is not
// part of the last field.
#include "mapfilter_dev.h"
#include "rfx_internal.h"

namespace rfx {
namespace {

constexpr int kLNT = 512;
// Bytes per thread: 64 KB tiles.  Tiles take turns at one ticket word (12 ns
// each) and at the look-back, so small tiles wait for those; large ones take
// longer to read where there are few.  Row ends of 133 MB of text in tiles of
// 32 / 64 / 128 KB 67 / 50 / 42 us, of 16 MB 17 / 13 / 12, of 1.09 MB 8.2 / 9.1 / 10.8,
// of 64 KB 8.7 / 9.0 / 10.6: 64 KB is the middle (128 KB from 16 MB on would be
// faster still).
constexpr int kLBytes = 128;
constexpr int kLTile = kLNT * kLBytes;
constexpr int kMaxFields = RFX_TBL_MAX_COLS;

// Which of 4 bytes equal pat's (one byte four times): bits 0 to 3.
__device__ __forceinline__ uint32_t byte_bits4(uint32_t w, uint32_t pat) {
  const uint32_t x = w ^ pat;
  // 0x80 in every zero byte (exact), moved together by one multiplication.
  const uint32_t z = ~(((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x | 0x7F7F7F7Fu);
  return ((z >> 7) * 0x10204080u) >> 28;
}
__device__ __forceinline__ uint32_t byte_bits16(uint4 v, uint32_t pat) {
  return byte_bits4(v.x, pat) | byte_bits4(v.y, pat) << 4 | byte_bits4(v.z, pat) << 8 |
         byte_bits4(v.w, pat) << 12;
}

__global__ __launch_bounds__(kLNT) void k_tbl_rows(const uint8_t* __restrict__ text,
                                                   uint64_t bytes, uint64_t* __restrict__ ends,
                                                   uint64_t cap, uint32_t ntiles,
                                                   uint64_t* __restrict__ counts,
                                                   uint64_t* __restrict__ rows,
                                                   uint64_t* __restrict__ status,
                                                   uint32_t* __restrict__ ticket) {
  __shared__ uint32_t s_scan[kLNT / kWave + 1];
  __shared__ uint32_t s_tile;
  __shared__ uint64_t s_prefix;
  __shared__ __attribute__((aligned(8))) uint16_t s_bits[kLTile / 16];
  const uint32_t tid = threadIdx.x, lane = lane_id(), w = wave_id();
  if (tid == 0) s_tile = atomicAdd(ticket, 1u);
  __syncthreads();
  const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);  // block-uniform: scalar from here
  // Places count from the 16-byte word that holds the first byte: the text is
  // [head, stop) of them.
  const uint32_t head = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(text) % 16);
  const uint8_t* const t0 = text - head;
  const uint64_t stop = head + bytes;
  const uint64_t tile_at = static_cast<uint64_t>(tile) * kLTile;
  const uint64_t at = tile_at + static_cast<uint64_t>(tid) * kLBytes;
  // Neighbouring lanes load neighbouring 16 bytes; the newlines of each
  // become 16 bits in LDS, where a thread then reads its own bytes' bits.
  const uint4* t = reinterpret_cast<const uint4*>(t0 + tile_at) + tid;
  uint4 v[kLBytes / 16];
  if (tile_at >= head && tile_at + kLTile <= stop) {  // uniform
#pragma unroll
    for (int j = 0; j < kLBytes / 16; ++j) v[j] = t[j * kLNT];
#pragma unroll
    for (int j = 0; j < kLBytes / 16; ++j)
      s_bits[tid + j * kLNT] = static_cast<uint16_t>(byte_bits16(v[j], 0x0A0A0A0Au));
  } else {
    // The first tile of an unaligned text and the last one: words inside the
    // text by the same loads, the two that its ends cut byte by byte.  (The
    // whole tile byte by byte is 128 loads in a row: a text of 16 KB 20 us,
    // 64 KB less a byte 34, 1.09 MB 27, 16 MB unaligned 74; now 7, 9, 9 and 13.)
#pragma unroll
    for (int j = 0; j < kLBytes / 16; ++j) {
      const uint64_t p = tile_at + 16ull * (tid + j * kLNT);
      v[j] = make_uint4(0, 0, 0, 0);
      if (p >= head && p + 16 <= stop) v[j] = t[j * kLNT];
    }
#pragma unroll
    for (int j = 0; j < kLBytes / 16; ++j) {
      const uint64_t p = tile_at + 16ull * (tid + j * kLNT);
      uint32_t bits = byte_bits16(v[j], 0x0A0A0A0Au);
      if (p < stop && (p < head || p + 16 > stop)) {  // the first word or the last
        for (int b = 0; b < 16; ++b)
          if (p + b >= head && p + b < stop && t0[p + b] == '\n') bits |= 1u << b;
      }
      s_bits[tid + j * kLNT] = static_cast<uint16_t>(bits);
    }
  }
  __syncthreads();
  uint64_t mask[kLBytes / 64];  // bit b of word q: byte 64 q + b is a newline
#pragma unroll
  for (int q = 0; q < kLBytes / 64; ++q)
    mask[q] = reinterpret_cast<const uint64_t*>(s_bits)[tid * (kLBytes / 64) + q];
  uint32_t mine = 0;
#pragma unroll
  for (int q = 0; q < kLBytes / 64; ++q) mine += static_cast<uint32_t>(__popcll(mask[q]));
  uint32_t total = 0;
  const uint32_t excl = block_excl_scan<kLNT>(mine, s_scan, &total);
  if (w == 0) {
    if (tile == 0) {
      if (lane == 0) {
        status_store64(status, kFlagIncl64 | total);
        s_prefix = 0;
      }
    } else {
      if (lane == 0) status_store64(status + tile, kFlagAgg64 | total);
      const uint64_t prev = wave_lookback64(status, tile);
      if (lane == 0) {
        status_store64(status + tile, kFlagIncl64 | (prev + total));
        s_prefix = prev;
      }
    }
  }
  __syncthreads();
  uint64_t k = s_prefix + excl;
#pragma unroll
  for (int q = 0; q < kLBytes / 64; ++q) {
    while (mask[q]) {
      const int b = __builtin_ctzll(mask[q]);
      mask[q] &= mask[q] - 1;
      if (k < cap) ends[k] = at + 64 * q + b - head;
      ++k;
    }
  }
  if (tile == ntiles - 1 && tid == 0) {
    // The text's rows: a last one may end without a newline.
    const uint64_t newlines = s_prefix + total;
    const uint64_t n = newlines + (text[bytes - 1] != '\n' ? 1 : 0);
    counts[0] = newlines;
    counts[1] = n;
    *rows = n;
  }
}

// The newlines alone, without their places: no order, so no ticket and no
// look-back (133 MB: 29 us against 50 by the pass above).  counts[0] is 0
// before; the last block to finish turns it into the rows.
constexpr int kCNT = 512;
__global__ __launch_bounds__(kCNT) void k_tbl_count(const uint8_t* __restrict__ text,
                                                    uint64_t bytes, bool aligned,
                                                    uint64_t* __restrict__ counts,
                                                    uint64_t* __restrict__ rows,
                                                    uint32_t* __restrict__ finished) {
  __shared__ uint32_t s_sum[kCNT / kWave];
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kCNT;
  const uint64_t g = static_cast<uint64_t>(blockIdx.x) * kCNT + threadIdx.x;
  uint32_t mine = 0;
  uint64_t done = 0;
  if (aligned) {
    const uint4* t = reinterpret_cast<const uint4*>(text);
    const uint64_t vecs = bytes / 16;
    uint64_t i = g;
    for (; i + 3 * stride < vecs; i += 4 * stride) {
      uint4 v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = t[i + j * stride];
#pragma unroll
      for (int j = 0; j < 4; ++j) mine += __popc(byte_bits16(v[j], 0x0A0A0A0Au));
    }
    for (; i < vecs; i += stride) mine += __popc(byte_bits16(t[i], 0x0A0A0A0Au));
    done = vecs * 16;
  }
  for (uint64_t i = done + g; i < bytes; i += stride) mine += text[i] == '\n';
  const uint32_t w = wave_incl_scan(mine);
  if (lane_id() == kWave - 1) s_sum[wave_id()] = w;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t sum = 0;
    for (int i = 0; i < kCNT / kWave; ++i) sum += s_sum[i];
    // The old value is waited for: the sum is in before the block is counted.
    const uint64_t old = atomicAdd(reinterpret_cast<unsigned long long*>(counts), sum);
    asm volatile("" ::"v"(old) : "memory");
    if (atomicAdd(finished, 1u) == gridDim.x - 1)
      *rows = status_load64(counts) + (text[bytes - 1] != '\n' ? 1 : 0);
  }
}

struct TblCols {
  void* p[kMaxFields];
  uint8_t t[kMaxFields];
};

__device__ __forceinline__ void tbl_store(const TblCols& c, int f, uint64_t row, int64_t iv,
                                          double dv) {
  void* p = c.p[f];
  switch (c.t[f]) {
    case RFX_TBL_I32: case RFX_TBL_U32: static_cast<uint32_t*>(p)[row] = static_cast<uint32_t>(iv); break;
    case RFX_TBL_I64: case RFX_TBL_DATE: static_cast<int64_t*>(p)[row] = iv; break;
    case RFX_TBL_U8: case RFX_TBL_CHAR: static_cast<uint8_t*>(p)[row] = static_cast<uint8_t>(iv); break;
    case RFX_TBL_F64: static_cast<double*>(p)[row] = dv; break;
    case RFX_TBL_STR: static_cast<int64_t*>(p)[row] = iv; break;
    default: break;
  }
}

__device__ const double kPow10[23] = {1e0,  1e1,  1e2,  1e3,  1e4,  1e5,  1e6,  1e7,
                                      1e8,  1e9,  1e10, 1e11, 1e12, 1e13, 1e14, 1e15,
                                      1e16, 1e17, 1e18, 1e19, 1e20, 1e21, 1e22};

constexpr int kFNT = 256;
constexpr int kFRows = 128;           // rows per block
constexpr int kStage = 24 * 1024;     // staged text bytes per block

// Parse row r ([pos, end) of the text) into the columns; at(q) gives byte
// q and scan(q, e) the first delimiter in [q, e) (e if none).  Each field's
// end is found first and its value parsed from its own bytes only, as
// splitting the row at the delimiters and then reading each field would
// (so a space, sign, point or digit delimiter never joins two fields).
template <class At, class Scan>
__device__ __forceinline__ void parse_row(At at, Scan scan, uint8_t* text, uint64_t bytes,
                                          uint64_t r, uint64_t pos, uint64_t end, int n_fields,
                                          const TblCols& cols, uint64_t* short_rows) {
  if (end > pos && at(end - 1) == '\r') --end;
  int f = 0;
  while (f < n_fields) {
    const int t = cols.t[f];
    const uint64_t fe = scan(pos, end);
    int64_t iv = 0;
    double dv = 0.0;
    if (t == RFX_TBL_CHAR) {
      iv = pos < fe ? at(pos) : 0;
    } else if (t == RFX_TBL_DATE) {
      // YYYY-MM-DD: each '-'-separated part read as atoi reads it
      // (leading spaces, a '+', digits up to the first other byte).
      int part[3] = {0, 0, 0}, k = 0, state = 0;  // 0 leading, 1 digits, 2 done
      for (uint64_t q = pos; q < fe && k < 3; ++q) {
        const uint8_t c = at(q);
        if (c == '-') {
          ++k;
          state = 0;
        } else if (c >= '0' && c <= '9' && state < 2) {
          part[k] = part[k] * 10 + (c - '0');
          state = 1;
        } else if (!(state == 0 && (c == ' ' || c == '+'))) {
          state = 2;
        }
      }
      iv = static_cast<int64_t>(date2int(part[0], part[1], part[2]));
    } else if (t != RFX_TBL_SKIP && t != RFX_TBL_STR) {
      uint64_t q = pos;
      while (q < fe && at(q) == ' ') ++q;
      bool neg = false;
      if (q < fe && (at(q) == '-' || at(q) == '+')) neg = at(q++) == '-';
      uint64_t m = 0;
      int frac = -1;  // digits after the point
      for (; q < fe; ++q) {
        const uint8_t c = at(q);
        if (c >= '0' && c <= '9') {
          m = m * 10 + (c - '0');
          if (frac >= 0) ++frac;
        } else if (c == '.' && t == RFX_TBL_F64 && frac < 0) {
          frac = 0;
        } else {
          break;
        }
      }
      iv = neg ? -static_cast<int64_t>(m) : static_cast<int64_t>(m);
      if (t == RFX_TBL_F64) {
        const double mag = static_cast<double>(m) / kPow10[frac > 0 ? (frac < 22 ? frac : 22) : 0];
        dv = neg ? -mag : mag;
      }
    } else if (t == RFX_TBL_STR) {
      // The field's address; its end (delimiter, '\r' or newline) becomes
      // its terminating NUL.  A field running to the end of the text has
      // nowhere to end: it reads as the null pointer (the empty string).
      iv = fe < bytes ? static_cast<int64_t>(reinterpret_cast<uintptr_t>(text + pos)) : 0;
      if (fe < bytes) text[fe] = 0;
    }
    tbl_store(cols, f, r, iv, dv);
    ++f;
    pos = fe;
    if (pos >= end) break;
    ++pos;  // past the delimiter
  }
  if (f < n_fields) {
    atomicAdd(reinterpret_cast<unsigned long long*>(short_rows), 1ull);
    for (; f < n_fields; ++f) tbl_store(cols, f, r, 0, 0.0);  // missing fields read 0
  }
}

// 8 bytes of the staged text from byte q (the stage ends in 16 spare bytes).
__device__ __forceinline__ uint64_t lds8(const uint4* stage, uint32_t q) {
  const uint64_t* w = reinterpret_cast<const uint64_t*>(stage) + (q >> 3);
  const uint32_t sh = (q & 7) * 8;
  const uint64_t lo = w[0], hi = w[1];
  return lo >> sh | (hi << 1) << (63 - sh);
}

// The first n (1 to 8) bytes of w as decimal digits: value, and whether all
// of them are digits.
__device__ __forceinline__ bool digits8(uint64_t w, uint32_t n, uint32_t* value) {
  const uint32_t pad = 8 * (8 - n);
  const uint64_t x = (w ^ 0x3030303030303030ull) << pad;  // zeros first, then the digits
  const uint64_t bad = (x | (x + 0x7676767676767676ull)) & 0x8080808080808080ull;
  uint32_t four[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t y = static_cast<uint32_t>(x >> (32 * h));
    const uint32_t two = (y & 0x00FF00FFu) * 10 + ((y >> 8) & 0x00FF00FFu);
    four[h] = (two & 0xFFFFu) * 100 + (two >> 16);
  }
  *value = four[0] * 10000 + four[1];
  return !bad;
}

// A field's bytes one at a time, from a register refilled every 8.
struct FieldBytes {
  const uint4* stage;
  uint32_t q, e, left = 0;
  uint64_t w = 0;
  __device__ __forceinline__ bool more() const { return q < e; }
  __device__ __forceinline__ uint8_t peek() {
    if (!left) {
      w = lds8(stage, q);
      left = 8;
    }
    return static_cast<uint8_t>(w);
  }
  __device__ __forceinline__ void skip() {  // after peek
    ++q;
    w >>= 8;
    --left;
  }
};

// Staged field [s, e) as type t (uniform over the wave): the well-formed
// ones by words, the others byte by byte, as parse_row reads them.
__device__ __forceinline__ void parse_staged(const uint4* stage, uint32_t s, uint32_t e, int t,
                                             int64_t* iv, double* dv) {
  const uint32_t len = e - s;
  if (t == RFX_TBL_CHAR) {
    *iv = len ? reinterpret_cast<const uint8_t*>(stage)[s] : 0;
    return;
  }
  const uint64_t w = lds8(stage, s);
  if (t == RFX_TBL_DATE) {
    uint32_t y, m, d;
    const bool fine = len == 10 && static_cast<uint8_t>(w >> 32) == '-' &&
                      static_cast<uint8_t>(w >> 56) == '-' && digits8(w, 4, &y) &&
                      digits8(w >> 40, 2, &m) && digits8(lds8(stage, s + 8), 2, &d);
    if (fine) {
      *iv = static_cast<int64_t>(date2int(static_cast<int>(y), static_cast<int>(m),
                                          static_cast<int>(d)));
      return;
    }
    FieldBytes b{stage, s, e};
    int part[3] = {0, 0, 0}, k = 0, state = 0;  // 0 leading, 1 digits, 2 done
    for (; b.more() && k < 3; b.skip()) {
      const uint8_t c = b.peek();
      if (c == '-') {
        ++k;
        state = 0;
      } else if (c >= '0' && c <= '9' && state < 2) {
        const int digit = c - '0';
        if (k == 0) part[0] = part[0] * 10 + digit;
        else if (k == 1) part[1] = part[1] * 10 + digit;
        else part[2] = part[2] * 10 + digit;
        state = 1;
      } else if (!(state == 0 && (c == ' ' || c == '+'))) {
        state = 2;
      }
    }
    *iv = static_cast<int64_t>(date2int(part[0], part[1], part[2]));
    return;
  }
  uint32_t whole, part;
  if (t == RFX_TBL_F64) {
    // Up to 8 digits, or up to 7, a point and one or two more.
    const uint64_t x = w ^ 0x2E2E2E2E2E2E2E2Eull;
    const uint64_t z = (x - 0x0101010101010101ull) & ~x & 0x8080808080808080ull;
    const uint32_t dot = z ? static_cast<uint32_t>(__builtin_ctzll(z)) >> 3 : 8;
    const uint32_t after = len - dot - 1;  // digits after the point
    if (dot >= len) {
      if (len >= 1 && len <= 8 && digits8(w, len, &whole)) {
        *dv = static_cast<double>(whole);
        return;
      }
    } else if (dot >= 1 && dot < 8 && (after == 1 || after == 2) && digits8(w, dot, &whole) &&
               digits8(lds8(stage, s + dot + 1), after, &part)) {
      const uint32_t ten = after == 1 ? 10u : 100u;
      *dv = static_cast<double>(whole * ten + part) / static_cast<double>(ten);
      return;
    }
  } else if (len >= 1 && len <= 8 && digits8(w, len, &whole)) {
    *iv = whole;
    return;
  }
  FieldBytes b{stage, s, e};
  while (b.more() && b.peek() == ' ') b.skip();
  bool neg = false;
  if (b.more() && (b.peek() == '-' || b.peek() == '+')) {
    neg = b.peek() == '-';
    b.skip();
  }
  uint64_t m = 0;
  int frac = -1;  // digits after the point
  for (; b.more(); b.skip()) {
    const uint8_t c = b.peek();
    if (c >= '0' && c <= '9') {
      m = m * 10 + (c - '0');
      if (frac >= 0) ++frac;
    } else if (c == '.' && t == RFX_TBL_F64 && frac < 0) {
      frac = 0;
    } else {
      break;
    }
  }
  *iv = neg ? -static_cast<int64_t>(m) : static_cast<int64_t>(m);
  if (t == RFX_TBL_F64) {
    const double mag = static_cast<double>(m) / kPow10[frac > 0 ? (frac < 22 ? frac : 22) : 0];
    *dv = neg ? -mag : mag;
  }
}

// The fields that have a column, and how many fields a row is split into.
struct TblTasks {
  int n, fields;
  uint8_t f[kMaxFields];
};

// Rows [128 b, 128 b + 128) of block b.  Their text is one contiguous span:
// when it fits, the block stages it in LDS with 16-byte loads, one bit per
// byte for the delimiters beside it; a thread per row walks those bits to
// the ends of its fields; then each wave takes one field of 64 rows at a
// time, so that its lanes convert texts of one type and their stores are
// neighbours.  (A thread walking and converting a whole row was bound by its
// chain of byte loads from LDS and by divergence, 12 waves per CU: 1 M
// lineitem rows 144 us; now 99.)  Otherwise every thread parses a row
// from global memory.
constexpr uint16_t kNoField = 0xFFFF;  // past the fields that a row has

__global__ __launch_bounds__(kFNT) void k_tbl_fields(uint8_t* __restrict__ text,
                                                     uint64_t bytes, bool aligned,
                                                     const uint64_t* __restrict__ ends,
                                                     uint64_t n_newlines, uint64_t rows,
                                                     uint8_t delim, TblTasks tasks, TblCols cols,
                                                     uint64_t* __restrict__ short_rows) {
  __shared__ uint4 s_text[kStage / 16 + 1];
  __shared__ __attribute__((aligned(8))) uint16_t s_bits[kStage / 16 + 4];
  __shared__ uint16_t s_start[kFRows];
  __shared__ uint64_t s_span[2];
  extern __shared__ uint16_t s_ends[];  // [fields][kFRows]
  const uint32_t tid = threadIdx.x;
  const uint64_t r0 = static_cast<uint64_t>(blockIdx.x) * kFRows;
  if (tid == 0) {
    const uint64_t last = r0 + kFRows - 1 < rows ? r0 + kFRows - 1 : rows - 1;
    s_span[0] = r0 == 0 ? 0 : ends[r0 - 1] + 1;
    s_span[1] = last < n_newlines ? ends[last] : bytes;
  }
  const uint64_t r = r0 + tid;
  const bool mine = tid < kFRows && r < rows;
  uint64_t pos = 0, end = 0;
  if (mine) {
    pos = r == 0 ? 0 : ends[r - 1] + 1;
    end = r < n_newlines ? ends[r] : bytes;
  }
  __syncthreads();
  const uint64_t base = s_span[0] & ~15ull, stop = s_span[1];
  if (!aligned || stop - base > static_cast<uint64_t>(kStage)) {
    if (mine) {
      auto scan = [&](uint64_t q, uint64_t e) -> uint64_t {
        while (q < e && text[q] != delim) ++q;
        return q;
      };
      parse_row([&](uint64_t q) -> uint8_t { return text[q]; }, scan, text, bytes, r, pos, end,
                tasks.fields, cols, short_rows);
    }
    return;
  }
  constexpr int kVecs = kStage / 16 / kFNT;
  const uint32_t nvec = static_cast<uint32_t>((stop - base + 15) / 16);
  uint4 v[kVecs];
#pragma unroll
  for (int j = 0; j < kVecs; ++j) {
    const uint32_t i = tid + j * kFNT;
    const uint64_t off = base + 16ull * i;
    v[j] = make_uint4(0, 0, 0, 0);
    if (i < nvec) {
      if (off + 16 <= bytes) {
        v[j] = *reinterpret_cast<const uint4*>(text + off);
      } else {
        uint32_t w[4] = {0, 0, 0, 0};
        for (int b = 0; off + b < bytes && b < 16; ++b)
          w[b >> 2] |= static_cast<uint32_t>(text[off + b]) << (8 * (b & 3));
        v[j] = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
  }
  const uint32_t pat = 0x01010101u * delim;
#pragma unroll
  for (int j = 0; j < kVecs; ++j) {
    const uint32_t i = tid + j * kFNT;
    if (i < nvec) {
      s_text[i] = v[j];
      s_bits[i] = static_cast<uint16_t>(byte_bits16(v[j], pat));
    }
  }
  __syncthreads();
  const uint8_t* lds = reinterpret_cast<const uint8_t*>(s_text);
  if (mine) {
    const uint32_t p = static_cast<uint32_t>(pos - base);
    uint32_t e = static_cast<uint32_t>(end - base);
    if (e > p && lds[e - 1] == '\r') --e;
    s_start[tid] = static_cast<uint16_t>(p);
    const uint64_t* bits = reinterpret_cast<const uint64_t*>(s_bits);
    uint32_t word = p >> 6;
    uint64_t m = bits[word] & (~0ull << (p & 63));
    int f = 0;
    for (;;) {
      while (!m && (word + 1) * 64 < e) m = bits[++word];
      const uint32_t d0 = m ? word * 64 + static_cast<uint32_t>(__builtin_ctzll(m)) : e;
      const uint32_t d = d0 < e ? d0 : e;
      s_ends[f * kFRows + tid] = static_cast<uint16_t>(d);
      if (++f == tasks.fields) break;
      if (d == e) {
        atomicAdd(reinterpret_cast<unsigned long long*>(short_rows), 1ull);
        for (; f < tasks.fields; ++f) s_ends[f * kFRows + tid] = kNoField;
        break;
      }
      m &= m - 1;
    }
  }
  __syncthreads();
  constexpr int kHalves = kFRows / kWave;
  for (int c = static_cast<int>(wave_id()); c < tasks.n * kHalves; c += kFNT / kWave) {
    const int f = tasks.f[c / kHalves];
    const uint32_t row = static_cast<uint32_t>(c % kHalves) * kWave + lane_id();
    if (r0 + row >= rows) continue;
    const uint32_t fe = s_ends[f * kFRows + row];
    int64_t iv = 0;
    double dv = 0.0;
    if (fe != kNoField) {  // missing fields read 0
      const uint32_t fs = f ? s_ends[(f - 1) * kFRows + row] + 1u : s_start[row];
      const int t = cols.t[f];
      if (t == RFX_TBL_STR) {
        // The field's address; its end (delimiter, '\r' or newline) becomes
        // its terminating NUL.  A field running to the end of the text has
        // nowhere to end: it reads as the null pointer (the empty string).
        if (base + fe < bytes) {
          iv = static_cast<int64_t>(reinterpret_cast<uintptr_t>(text + base + fs));
          text[base + fe] = 0;
        }
      } else {
        parse_staged(s_text, fs, fe, t, &iv, &dv);
      }
    }
    tbl_store(cols, f, r0 + row, iv, dv);
  }
}

}  // namespace
}  // namespace rfx

using namespace rfx;

extern "C" int rfx_tbl_parse(rfx_ctx* ctx, void* text, uint64_t bytes, char delim,
                             const int* types, int n_fields, void* const* columns,
                             uint64_t capacity, uint64_t* rows, uint64_t* short_rows) {
  if (!ctx || !rows || !short_rows || (bytes && !text) || (n_fields && (!types || !columns)))
    return fail(RFX_EINVAL, "rfx_tbl_parse: null argument");
  if (n_fields < 0 || n_fields > kMaxFields)
    return fail(RFX_EINVAL, "rfx_tbl_parse: %d fields (at most %d)", n_fields, kMaxFields);
  if (delim == '\n') return fail(RFX_EINVAL, "rfx_tbl_parse: the delimiter cannot be a newline");
  if (bytes >= (1ull << 40)) return fail(RFX_ERANGE, "rfx_tbl_parse: text too large");
  TblCols cols{};
  for (int f = 0; f < n_fields; ++f) {
    if (types[f] < RFX_TBL_SKIP || types[f] > RFX_TBL_STR)
      return fail(RFX_EINVAL, "rfx_tbl_parse: field %d type %d", f, types[f]);
    if (types[f] != RFX_TBL_SKIP && capacity && !columns[f])
      return fail(RFX_EINVAL, "rfx_tbl_parse: field %d has no column", f);
    cols.p[f] = types[f] == RFX_TBL_SKIP ? nullptr : columns[f];
    cols.t[f] = static_cast<uint8_t>(types[f]);
  }
  // Row ends are kept for the rows that are parsed (the count covers all).
  const uint64_t head = reinterpret_cast<uintptr_t>(text) % 16;
  const uint64_t ntiles = bytes ? (head + bytes + kLTile - 1) / kLTile : 0;
  const uint64_t ecap = !capacity ? 1 : capacity < bytes ? capacity + 1 : (bytes ? bytes : 1);
  Carve c(nullptr);
  c.take<uint64_t>(ecap);
  c.take<uint64_t>(ntiles ? ntiles : 1);
  c.take<uint32_t>(1);
  c.take<uint64_t>(2);
  RFX_TRY(ensure_workspace(ctx, c.off));
  Carve w(ctx->ws);
  uint64_t* ends = w.take<uint64_t>(ecap);
  uint64_t* status = w.take<uint64_t>(ntiles ? ntiles : 1);
  uint32_t* ticket = w.take<uint32_t>(1);
  uint64_t* counts = w.take<uint64_t>(2);  // newlines, rows
  RFX_TRY(fill_u32(ctx, reinterpret_cast<uint32_t*>(status),
                   (reinterpret_cast<char*>(counts + 2) - reinterpret_cast<char*>(status)) / 4, 0));
  RFX_TRY(fill_u32(ctx, reinterpret_cast<uint32_t*>(short_rows), 2, 0));
  if (!ntiles) RFX_TRY(fill_u32(ctx, reinterpret_cast<uint32_t*>(rows), 2, 0));
  if (ntiles && !capacity) {
    RFX_PROF(ctx, "tbl.rows");
    const uint64_t most = static_cast<uint64_t>(ctx->device_cus) * 4;
    const uint64_t blocks = (bytes + 16 * kCNT - 1) / (16 * kCNT);
    k_tbl_count<<<static_cast<uint32_t>(blocks < most ? blocks : most), kCNT, 0, ctx->stream>>>(
        static_cast<const uint8_t*>(text), bytes, reinterpret_cast<uintptr_t>(text) % 16 == 0,
        counts, rows, ticket);
    RFX_LAUNCHED();
  } else if (ntiles) {
    RFX_PROF(ctx, "tbl.rows");
    k_tbl_rows<<<static_cast<uint32_t>(ntiles), kLNT, 0, ctx->stream>>>(
        static_cast<const uint8_t*>(text), bytes, ends, ecap, static_cast<uint32_t>(ntiles), counts,
        rows, status, ticket);
    RFX_LAUNCHED();
  }
  // The row count sizes the field pass: read it back.
  uint64_t got[2] = {0, 0};
  if (ntiles && capacity && n_fields)
    RFX_HIP(hipMemcpyAsync(got, counts, 16, hipMemcpyDeviceToHost, ctx->stream));
  RFX_HIP(hipStreamSynchronize(ctx->stream));
  const uint64_t newlines = got[0], n = got[1];
  const uint64_t todo = n < capacity ? n : capacity;
  if (todo && n_fields) {
    RFX_PROF(ctx, "tbl.fields");
    TblTasks tasks{};
    tasks.fields = n_fields;
    for (int f = 0; f < n_fields; ++f)
      if (types[f] != RFX_TBL_SKIP) tasks.f[tasks.n++] = static_cast<uint8_t>(f);
    k_tbl_fields<<<static_cast<uint32_t>((todo + kFRows - 1) / kFRows), kFNT,
                   n_fields * kFRows * sizeof(uint16_t), ctx->stream>>>(
        static_cast<uint8_t*>(text), bytes, reinterpret_cast<uintptr_t>(text) % 16 == 0,
        ends, newlines, todo, static_cast<uint8_t>(delim), tasks, cols, short_rows);
    RFX_LAUNCHED();
    RFX_HIP(hipStreamSynchronize(ctx->stream));
  }
  return RFX_OK;
}
