// strings.hip - sorted search over string keys (find_bounds_string,
// ModernGPUJoin.cu:213-312) for gfx950.
//
// Keys are device addresses of NUL-terminated strings, each side sorted by
// compare_string2 (ModernGPUJoin.cu:72-97): bytes compared as signed char
// up to the first NUL of either, a proper prefix ordered first.  A block of
// left keys first narrows the right side to the range that its first and
// last key span; one thread per left key then finds its lower bound in that
// range (every probe a string comparison in global memory) and takes its
// upper bound from its neighbour's lower bound; the counts are turned into
// their exclusive prefix sums by a tile scan with decoupled look-back, whose
// last tile writes the total.  The outputs are those of rfx_join_find_bounds, so rfx_join_main
// expands them into row pairs.
#include "rfx_device.h"
#include "rfx_internal.h"

namespace rfx {
namespace {

constexpr uint64_t kLow7 = 0x7F7F7F7F7F7F7F7Full;

// 0x80 in every byte of v that is zero (exact: no false flags).
__device__ __forceinline__ uint64_t zero_bytes(uint64_t v) {
  return ~(((v & kLow7) + kLow7) | v | kLow7);
}
// 0x80 in every byte of v that is not zero.
__device__ __forceinline__ uint64_t nonzero_bytes(uint64_t v) {
  return (((v & kLow7) + kLow7) | v) & ~kLow7;
}

// The 8 bytes at address p (little-endian), read as aligned words: the
// word after the first is read only when the first holds no NUL at or
// after p, so every word read holds a byte of the string (an aligned word
// does not cross a page).  Bytes after a NUL are don't-cares.
__device__ __forceinline__ uint64_t load8(uint64_t p) {
  const uint64_t* w = reinterpret_cast<const uint64_t*>(p & ~7ull);
  const uint32_t sh = static_cast<uint32_t>(p & 7) * 8;
  uint64_t v = w[0] >> sh;
  if (sh && !(zero_bytes(v | (~0ull << (64 - sh))))) v |= w[1] << (64 - sh);
  return v;
}

// compare_string2: a < b, 8 bytes per step.  A null address reads as the
// empty string.
__device__ __forceinline__ bool str_less(uint64_t pa, uint64_t pb) {
  if (!pa || !pb) return !pa && pb && *reinterpret_cast<const uint8_t*>(pb) != 0;
  for (;; pa += 8, pb += 8) {
    const uint64_t va = load8(pa), vb = load8(pb);
    const uint64_t m = zero_bytes(va) | zero_bytes(vb) | nonzero_bytes(va ^ vb);
    if (m) {
      const uint32_t sh = static_cast<uint32_t>(__builtin_ctzll(m)) & ~7u;
      const uint8_t x = static_cast<uint8_t>(va >> sh), y = static_cast<uint8_t>(vb >> sh);
      if (x == 0 || y == 0) return x == 0 && y != 0;
      return static_cast<int8_t>(x) < static_cast<int8_t>(y);
    }
  }
}

constexpr int kSNT = 256;

// First index in [lo, hi) whose string is not below key (UPPER: above key),
// by one wave: 64 probes a round, of which the ones below form a prefix.
template <bool UPPER>
__device__ __forceinline__ uint64_t wave_bound(const uint64_t* __restrict__ right, uint64_t lo,
                                               uint64_t hi, uint64_t key) {
  const uint32_t lane = lane_id();
  while (lo < hi) {
    const uint64_t len = hi - lo;
    // Probe points, spread evenly; the same point may be taken twice.
    const uint64_t at = lo + len * (lane + 1) / (kWave + 1);
    const bool below = UPPER ? !str_less(key, right[at]) : str_less(right[at], key);
    const uint32_t c = static_cast<uint32_t>(__popcll(ballot(below)));
    const uint64_t old = lo;
    if (c) lo = old + len * c / (kWave + 1) + 1;
    if (c < kWave) hi = old + len * (c + 1) / (kWave + 1);
  }
  return lo;
}

// Searches are chains of dependent loads, so what counts is their length: at
// 2^18 left and 2^22 right keys a search of all right keys is 22 probes and
// the upper bound as many again.  The block's range costs 4 rounds of 64
// probes for its first and last key (one wave each) and saves about log2 of
// the blocks, so it is looked for where it saves more rounds than it takes
// (300,000 x 10 of 287 bytes 86 us, 573 without; 20 x 10 13 and 10).  Inside it a thread bisects: several probes a round are as many
// comparisons one after the other (three: 300,000 x 150,000 names 136 us, 20 x
// 10 30; one: 93 and 16).  The upper bound is the next key's lower bound,
// which one comparison confirms (a right key that no left key equals may lie
// in between: then the run's end is searched for).
constexpr uint64_t kGallopFrom = 1024;
__global__ __launch_bounds__(kSNT) void k_str_bounds(const uint64_t* __restrict__ left, uint64_t nl,
                                                     const uint64_t* __restrict__ right,
                                                     uint64_t nr, int32_t* __restrict__ lower,
                                                     int32_t* __restrict__ count) {
  __shared__ uint64_t s_range[2];
  __shared__ uint64_t s_lo[kSNT];
  const uint64_t i0 = static_cast<uint64_t>(blockIdx.x) * kSNT;
  const uint64_t i = i0 + threadIdx.x;
  const uint64_t last = (i0 + kSNT < nl ? i0 + kSNT : nl) - 1;
  const uint32_t w = wave_id();
  const int rounds = (69 - __clzll(static_cast<long long>(nr | 1))) / 6;  // of 64 probes
  if (31 - __clz(static_cast<int>(gridDim.x)) <= rounds) {  // uniform
    if (threadIdx.x < 2) s_range[threadIdx.x] = threadIdx.x ? nr : 0;
  } else if (w < 2) {
    const uint64_t r = w == 0 ? wave_bound<false>(right, 0, nr, left[i0])
                              : wave_bound<true>(right, 0, nr, left[last]);
    if (lane_id() == 0) s_range[w] = r;
  }
  __syncthreads();
  const uint64_t b0 = s_range[0], b1 = s_range[1];
  const uint64_t key = i < nl ? left[i] : 0;
  uint64_t lo = b0, hi = i < nl ? b1 : b0;  // first right key not below key
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (str_less(right[mid], key)) lo = mid + 1;
    else hi = mid;
  }
  s_lo[threadIdx.x] = lo;
  __syncthreads();
  if (i >= nl) return;
  // The right keys before `next` are below the next left key (for the last
  // one, not above the block's last), so the run of keys equal to this one ends
  // there or before, unless the next left key is this one again (next == lo).
  const uint64_t next = i == last ? b1 : s_lo[threadIdx.x + 1];
  uint64_t up = lo, end = b1;
  if (lo < b1) {  // one comparison for all lanes alike
    const uint64_t at = next > lo ? next - 1 : lo;
    const bool above = str_less(key, right[at]);
    if (!above) up = at + 1;
    if (above) end = at;
    else if (next > lo) end = up;
  }
  if (end - up > kGallopFrom) {
    uint64_t step = 1;
    while (up < b1) {
      const uint64_t at = up + step - 1 < b1 ? up + step - 1 : b1 - 1;
      if (str_less(key, right[at])) {
        end = at;
        break;
      }
      up = at + 1;
      step <<= 1;
    }
  }
  while (up < end) {
    const uint64_t mid = (up + end) >> 1;
    if (str_less(key, right[mid])) end = mid;
    else up = mid + 1;
  }
  lower[i] = static_cast<int32_t>(lo);
  count[i] = static_cast<int32_t>(up - lo);
}

// count[] -> exclusive prefix sums in place, tiles of 256 x 8; *total gets
// the sum.
constexpr int kCVT = 8;
constexpr int kCTile = kSNT * kCVT;

__global__ __launch_bounds__(kSNT) void k_count_scan(int32_t* __restrict__ count, uint64_t n,
                                                     uint32_t ntiles, uint64_t* __restrict__ total,
                                                     uint64_t* __restrict__ status,
                                                     uint32_t* __restrict__ ticket) {
  __shared__ uint64_t s_scan[kSNT / kWave + 1];
  __shared__ uint32_t s_tile;
  __shared__ uint64_t s_prefix;
  const uint32_t tid = threadIdx.x, lane = lane_id(), w = wave_id();
  if (tid == 0) s_tile = atomicAdd(ticket, 1u);
  __syncthreads();
  const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);  // block-uniform: scalar from here
  const uint64_t at = static_cast<uint64_t>(tile) * kCTile + static_cast<uint64_t>(tid) * kCVT;
  uint64_t v[kCVT], sum = 0;
#pragma unroll
  for (int j = 0; j < kCVT; ++j) {
    v[j] = at + j < n ? static_cast<uint32_t>(count[at + j]) : 0u;
    sum += v[j];
  }
  uint64_t tile_sum = 0;
  const uint64_t excl = block_excl_scan<kSNT>(sum, s_scan, &tile_sum);
  if (w == 0) {
    if (tile == 0) {
      if (lane == 0) {
        status_store64(status, kFlagIncl64 | tile_sum);
        s_prefix = 0;
      }
    } else {
      if (lane == 0) status_store64(status + tile, kFlagAgg64 | tile_sum);
      const uint64_t prev = wave_lookback64(status, tile);
      if (lane == 0) {
        status_store64(status + tile, kFlagIncl64 | (prev + tile_sum));
        s_prefix = prev;
      }
    }
  }
  __syncthreads();
  uint64_t run = s_prefix + excl;
#pragma unroll
  for (int j = 0; j < kCVT; ++j) {
    if (at + j < n) count[at + j] = static_cast<int32_t>(run);
    run += v[j];
  }
  if (tile == ntiles - 1 && tid == 0) *total = s_prefix + tile_sum;
}

// 8 bytes of a string as 8 order-preserving codes, first byte most
// significant: the terminator and what follows it 0, then signed chars
// -128..-1, 1..127 as 1..255 (compare_string2's order).
__device__ __forceinline__ uint64_t str_codes(uint64_t v) {
  const uint64_t z = zero_bytes(v);
  if (z) v &= (1ull << (static_cast<uint32_t>(__builtin_ctzll(z)) & ~7u)) - 1;
  const uint64_t some = (nonzero_bytes(v) >> 7) * 0xFFull;
  // No carry leaves a byte: 0xFF becomes 0x7F + 1.
  const uint64_t c = ((v ^ 0x8080808080808080ull) + ((v >> 7) & 0x0101010101010101ull)) & some;
  return __builtin_bswap64(c);
}

// Walks a string 8 bytes at a time: the codes of the next 8 bytes, 0 past
// the end.
struct StrWalk {
  uint64_t p;  // 0: ended
  __device__ __forceinline__ explicit StrWalk(uint64_t addr) : p(addr) {}
  __device__ __forceinline__ uint64_t next() {
    if (!p) return 0;
    const uint64_t v = load8(p);
    p = zero_bytes(v) ? 0 : p + 8;
    return str_codes(v);
  }
};

// The bits of the strings' codes in which any string differs from the first
// one, for the first kVaryWords words of 8 codes, and the number of words of
// the longest string.
constexpr int kVaryWords = 32;
struct StrStats {
  unsigned long long vary[kVaryWords];
  unsigned long long words;
};

__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  int x = static_cast<int>(v);
  x |= __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x |= __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x |= __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x |= __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x |= __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x |= __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(x, kWave - 1));
}

__global__ __launch_bounds__(kSNT) void k_str_stats(const uint64_t* __restrict__ addr, uint64_t n,
                                                    StrStats* __restrict__ out) {
  __shared__ unsigned long long s_vary[kVaryWords];
  __shared__ uint32_t s_words;
  for (uint32_t q = threadIdx.x; q < kVaryWords; q += kSNT) s_vary[q] = 0;
  if (threadIdx.x == 0) s_words = 0;
  __syncthreads();
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kSNT;
  const uint64_t first = addr[0];
  // Whole waves go round together; the last rows are repeated.
  for (uint64_t i0 = static_cast<uint64_t>(blockIdx.x) * kSNT; i0 < n; i0 += stride) {
    const uint64_t i = i0 + threadIdx.x < n ? i0 + threadIdx.x : n - 1;
    StrWalk me(addr[i]), ref(first);
    uint32_t c = 0;
    while (ballot(me.p != 0 || ref.p != 0)) {
      const uint64_t d = me.next() ^ ref.next();
      if (c < kVaryWords) {
        const uint64_t any = static_cast<uint64_t>(wave_or(static_cast<uint32_t>(d >> 32))) << 32 |
                             wave_or(static_cast<uint32_t>(d));
        if (lane_id() == 0 && any) atomicOr(&s_vary[c], any);
      }
      ++c;
    }
    if (lane_id() == 0) atomicMax(&s_words, c);
  }
  __syncthreads();
  // Atomics of all blocks on one word take turns (10 ns each): with many, only
  // a block that adds something makes them (300,000 empty strings 42 -> 30 us,
  // 1.5 M names 194 -> 161); with few, looking first is the longer way.
  auto adds = [&](unsigned long long* word, unsigned long long mine, bool bits) {
    if (!mine || gridDim.x <= kWave) return mine != 0;
    const unsigned long long now = status_load64(reinterpret_cast<uint64_t*>(word));
    return bits ? (mine & ~now) != 0 : mine > now;
  };
  for (uint32_t q = threadIdx.x; q < kVaryWords; q += kSNT)
    if (adds(&out->vary[q], s_vary[q], true)) atomicOr(&out->vary[q], s_vary[q]);
  if (threadIdx.x == 0 && adds(&out->words, s_words, false))
    atomicMax(&out->words, static_cast<unsigned long long>(s_words));
}

// A sort key of up to 64 bits: pieces of the strings' code words, most
// significant first.
struct StrPiece {
  uint32_t word;
  uint8_t shift, bits;
};
struct StrKey {
  int pieces;
  StrPiece p[64];
};

// Each string's key.  With rows, element i is the string of row rows[i].
template <class K>
__global__ __launch_bounds__(kSNT) void k_str_key(const uint64_t* __restrict__ addr,
                                                  const uint32_t* __restrict__ rows, uint64_t n,
                                                  StrKey key, K* __restrict__ out) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kSNT + threadIdx.x;
  if (i >= n) return;
  StrWalk s(addr[rows ? rows[i] : i]);
  uint64_t k = 0, codes = s.next();
  uint32_t at = 0;
  for (int q = 0; q < key.pieces; ++q) {
    const StrPiece p = key.p[q];
    for (; at < p.word; ++at) codes = s.next();
    k = p.bits < 64 ? (k << p.bits) | ((codes >> p.shift) & ((1ull << p.bits) - 1)) : codes;
  }
  out[i] = static_cast<K>(k);
}

// Run heads of sorted strings: 1 where a string differs from the one
// before it (sorted, so where the one before is less), 0 elsewhere.
__global__ __launch_bounds__(kSNT) void k_str_heads(const uint64_t* __restrict__ addr, uint64_t n,
                                                    int32_t* __restrict__ head) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kSNT + threadIdx.x;
  if (i >= n) return;
  head[i] = i == 0 || str_less(addr[i - 1], addr[i]) ? 1 : 0;
}

// After the exclusive scan of the heads: group of row i = heads up to and
// including i, less one (the scan of row i + 1, or the total for the last).
__global__ __launch_bounds__(kSNT) void k_str_groups(const int32_t* __restrict__ excl, uint64_t n,
                                                     const uint64_t* __restrict__ total,
                                                     uint32_t* __restrict__ group) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kSNT + threadIdx.x;
  if (i >= n) return;
  const uint64_t incl = i + 1 < n ? static_cast<uint32_t>(excl[i + 1]) : *total;
  group[i] = static_cast<uint32_t>(incl - 1);
}

}  // namespace
}  // namespace rfx

using namespace rfx;

extern "C" int rfx_string_groups(rfx_ctx* ctx, const uint64_t* sorted, uint64_t n, uint32_t* group,
                                 int32_t* scratch, uint64_t* n_groups) {
  if (!ctx || !n_groups || (n && (!sorted || !group || !scratch)))
    return fail(RFX_EINVAL, "rfx_string_groups: null argument");
  if (n >= (1ull << 31)) return fail(RFX_ERANGE, "rfx_string_groups: more than 2^31 - 1 rows");
  if (n == 0) return fill_u32(ctx, reinterpret_cast<uint32_t*>(n_groups), 2, 0);
  const uint32_t grid = static_cast<uint32_t>((n + kSNT - 1) / kSNT);
  k_str_heads<<<grid, kSNT, 0, ctx->stream>>>(sorted, n, scratch);
  RFX_LAUNCHED();
  const uint64_t ntiles = (n + kCTile - 1) / kCTile;
  Carve c(nullptr);
  c.take<uint64_t>(ntiles);
  c.take<uint32_t>(1);
  RFX_TRY(ensure_workspace(ctx, c.off));
  Carve w(ctx->ws);
  uint64_t* status = w.take<uint64_t>(ntiles);
  uint32_t* ticket = w.take<uint32_t>(1);
  RFX_TRY(fill_u32(ctx, reinterpret_cast<uint32_t*>(status),
                   (reinterpret_cast<char*>(ticket + 1) - reinterpret_cast<char*>(status)) / 4, 0));
  k_count_scan<<<static_cast<uint32_t>(ntiles), kSNT, 0, ctx->stream>>>(
      scratch, n, static_cast<uint32_t>(ntiles), n_groups, status, ticket);
  RFX_LAUNCHED();
  k_str_groups<<<grid, kSNT, 0, ctx->stream>>>(scratch, n, n_groups, group);
  RFX_LAUNCHED();
  return RFX_OK;
}

namespace rfx {
namespace {

// Sort rows (or, without rows, the addresses themselves) by their strings.
// Of each of the first kVaryWords words only the bits that differ between
// strings go into the sort keys (in each code from its lowest to its highest
// such bit), so names like Supplier#000012345 sort by one key of 4 bits a
// varying digit instead of three 64-bit keys; later words go in whole.  LSD
// over keys of up to 64 bits, least significant key first; each pass is a
// stable sort of (key, payload) pairs.
int sort_by_string(rfx_ctx* ctx, const uint64_t* addr, uint64_t* moved, uint32_t* rows,
                   uint64_t* scratch, uint64_t n) {
  RFX_TRY(ensure_workspace(ctx, sizeof(StrStats)));
  StrStats* stats = static_cast<StrStats*>(ctx->ws);
  RFX_TRY(fill_u32(ctx, reinterpret_cast<uint32_t*>(stats), sizeof(StrStats) / 4, 0));
  const uint64_t blocks = (n + kSNT - 1) / kSNT, most = static_cast<uint64_t>(ctx->device_cus) * 16;
  k_str_stats<<<static_cast<uint32_t>(blocks < most ? blocks : most), kSNT, 0, ctx->stream>>>(
      addr, n, stats);
  RFX_LAUNCHED();
  StrStats h;
  RFX_HIP(hipMemcpyAsync(&h, stats, sizeof h, hipMemcpyDeviceToHost, ctx->stream));
  RFX_HIP(hipStreamSynchronize(ctx->stream));
  // Pieces from the least significant end, cut into keys of up to 64 bits.
  StrKey key{};
  uint32_t bits = 0;
  auto flush = [&]() -> int {
    if (!bits) return RFX_OK;
    for (int a = 0, b = key.pieces - 1; a < b; ++a, --b) {
      const StrPiece t = key.p[a];
      key.p[a] = key.p[b];
      key.p[b] = t;
    }
    const int kb = bits <= 32 ? 4 : 8;
    if (kb == 4)
      k_str_key<uint32_t><<<static_cast<uint32_t>(blocks), kSNT, 0, ctx->stream>>>(
          addr, rows, n, key, reinterpret_cast<uint32_t*>(scratch));
    else
      k_str_key<uint64_t><<<static_cast<uint32_t>(blocks), kSNT, 0, ctx->stream>>>(addr, rows, n,
                                                                                   key, scratch);
    RFX_LAUNCHED();
    RFX_TRY(rfx_sort_pairs(ctx, scratch, rows ? static_cast<void*>(rows) : moved, n, kb,
                           static_cast<int>(bits), rows ? 4 : 8));
    key.pieces = 0;
    bits = 0;
    return RFX_OK;
  };
  auto piece = [&](uint64_t word, uint32_t shift, uint32_t width) -> int {
    if (bits + width > 64) RFX_TRY(flush());
    key.p[key.pieces++] = {static_cast<uint32_t>(word), static_cast<uint8_t>(shift),
                           static_cast<uint8_t>(width)};
    bits += width;
    return RFX_OK;
  };
  for (uint64_t c = h.words; c-- > 0;) {
    if (c >= kVaryWords) {
      RFX_TRY(piece(c, 0, 64));
      continue;
    }
    for (uint32_t sh = 0; sh < 64; sh += 8) {
      const uint32_t v = static_cast<uint32_t>(h.vary[c] >> sh) & 0xFFu;
      if (!v) continue;
      const uint32_t lo = static_cast<uint32_t>(__builtin_ctz(v));
      RFX_TRY(piece(c, sh + lo, 32u - static_cast<uint32_t>(__builtin_clz(v)) - lo));
    }
  }
  return flush();
}

}  // namespace
}  // namespace rfx

extern "C" int rfx_sort_strings(rfx_ctx* ctx, uint64_t* addresses, uint64_t* scratch, uint64_t n) {
  if (!ctx || (n && (!addresses || !scratch)))
    return fail(RFX_EINVAL, "rfx_sort_strings: null argument");
  if (n < 2) return RFX_OK;
  if (n >= (1ull << 40)) return fail(RFX_ERANGE, "rfx_sort_strings: too many strings");
  return sort_by_string(ctx, addresses, addresses, nullptr, scratch, n);
}

extern "C" int rfx_sort_strings_rows(rfx_ctx* ctx, const uint64_t* addresses, uint32_t* rows,
                                     uint64_t* scratch, uint64_t n) {
  if (!ctx || (n && (!addresses || !rows || !scratch)))
    return fail(RFX_EINVAL, "rfx_sort_strings_rows: null argument");
  if (n >= (1ull << 32)) return fail(RFX_ERANGE, "rfx_sort_strings_rows: too many rows");
  if (n < 2) return RFX_OK;
  return sort_by_string(ctx, addresses, nullptr, rows, scratch, n);
}

extern "C" int rfx_join_find_bounds_string(rfx_ctx* ctx, int32_t* lower_bound, int32_t* left_count,
                                           uint64_t* total, const uint64_t* left, uint64_t nl,
                                           const uint64_t* right, uint64_t nr) {
  if (!ctx || !total || (nl && (!lower_bound || !left_count || !left)) || (nr && !right))
    return fail(RFX_EINVAL, "rfx_join_find_bounds_string: null argument");
  if (nl >= (1ull << 31) || nr >= (1ull << 31))
    return fail(RFX_ERANGE, "rfx_join_find_bounds_string: more than 2^31 - 1 keys");
  if (nl == 0) return fill_u32(ctx, reinterpret_cast<uint32_t*>(total), 2, 0);
  const uint64_t ntiles = (nl + kCTile - 1) / kCTile;
  Carve c(nullptr);
  c.take<uint64_t>(ntiles);
  c.take<uint32_t>(1);
  RFX_TRY(ensure_workspace(ctx, c.off));
  Carve w(ctx->ws);
  uint64_t* status = w.take<uint64_t>(ntiles);
  uint32_t* ticket = w.take<uint32_t>(1);
  RFX_TRY(fill_u32(ctx, reinterpret_cast<uint32_t*>(status),
                   (reinterpret_cast<char*>(ticket + 1) - reinterpret_cast<char*>(status)) / 4, 0));
  {
    RFX_PROF(ctx, "join.find_bounds_string");
    k_str_bounds<<<static_cast<uint32_t>((nl + kSNT - 1) / kSNT), kSNT, 0, ctx->stream>>>(
        left, nl, right, nr, lower_bound, left_count);
    RFX_LAUNCHED();
  }
  k_count_scan<<<static_cast<uint32_t>(ntiles), kSNT, 0, ctx->stream>>>(
      left_count, nl, static_cast<uint32_t>(ntiles), total, status, ticket);
  RFX_LAUNCHED();
  return RFX_OK;
}
