// sort.hip - stable LSD radix sort for gfx950: one upfront histogram pass
// over the keys for all digit positions, then one "onesweep" kernel per
// digit that ranks a tile in registers/LDS, obtains its global digit offsets
// by decoupled look-back and scatters through an LDS reorder buffer.  Digits
// are 8 bits, or 6 to 10 where key_bits makes an even number of passes of
// them and they are faster (auto_digit): wider digits take fewer passes over
// the data at the cost of more bins per tile (more ranking ballots and
// look-back words, shorter runs per bin in the scatter), narrower ones save
// the copy back after an odd number of passes.
//
// Replaces redfox::sort_pair / sort_key (b40cSort.cu:58-1021: b40c LSD
// radix, 4-5 bit digits, upsweep + spine + downsweep per digit, pong
// buffers cudaMalloc'd per call) and the mergesort variants
// (ModernGPUSort.cu:238-574).  Both are stable, so for the same key bits
// they produce exactly the order this sort produces.
//
// Everything after the launch is decided on the device: a digit position
// whose histogram has one full bucket is an identity permutation and is
// skipped; which of the two buffers holds the data is tracked in a device
// word, and a final kernel copies back only if it is the pong buffer.  No
// host round trip, so a sort can be captured into a HIP graph.
#include <type_traits>

#include "rfx_device.h"
#include "rfx_internal.h"

namespace rfx {
namespace {

// Digit width DB: 1 << DB bins.
template <int DB>
constexpr int kBinsOf = 1 << DB;

// Tile shape of the large sorts: NT threads x IPT keys per thread.  LDS per
// block is about kMax*TILE (reorder) + 2*bins*NT/64 (wave counters) +
// 4*bins.  The pass is bound by the cache lines that it writes in part, one
// or two per tile, digit and column, so the tile is as large as the
// registers allow with two blocks per CU (128 VGPRs; whole sorts of 2^28
// u32 pairs: 512 x 16 4.81 ms, 512 x 20 4.74, 512 x 24 4.52, 512 x 32 4.65
// with spills; 2^28 u32 keys alone: 512 x 16 1.81 ms at 2^27, 512 x 32
// 1.62).  8-byte elements: two 512 x 14 blocks or, where the digits are 10
// bits wide or keys and values are both 8 bytes, one block of 1024 (2^25
// u32 keys of 20 bits with f64 values: 0.65 -> 0.57 ms; 2^26 u64 pairs
// 3.97 -> 3.79 ms; u64 keys with u32 values 6.16 -> 7.1 ms, so not there).
// 4-byte elements beside narrower ones take the tile of 24 as well past
// mid_rows rows (2^28 rows, 16 -> 24: 2-byte keys with 4-byte values 2.48 ->
// 2.08 ms, 4-byte keys with one-byte values 4.50 -> 3.82); at 1 M rows it is
// too few tiles (0.073 against 0.083 ms).
template <int KB, int VB, int DB>
struct SortTune {
  static constexpr int kMax = KB > VB ? KB : VB;
  static constexpr bool kWide = kMax == 8 && (DB == 10 || (KB == 8 && VB == 8));
  static constexpr int NT = kWide ? 1024 : 512;
  static constexpr int IPT = kMax >= 16                       ? 8
                             : kMax >= 8                      ? (kWide && DB <= 8 ? 12 : 14)
                             : KB >= 2 && VB > 0 && kMax == 4 ? 24
                             : KB == 4 && VB == 0             ? (DB <= 8 ? 32 : 24)
                                                              : 16;
  // Up to mid_rows, in shapes that have no tile of kMidNT x kMidIPT.
  static constexpr int kFewIPT = kMax >= 8 ? IPT : 16;
};

// Look-back window (status words per round trip): every extra word polled
// costs a large sort (2^28 u32 pairs 4.79 ms with 2, 4.81 with 4, 4.95 with
// 8).
constexpr int kWindow = 2;

// Tile of the sorts whose large tiles would not fill the chip: kMidNT
// threads x 4 keys (12 x 512 for 9 and 10 bit digits, whose counters fill
// the LDS), up to kMidTiles such tiles per CU.  All of them run at once, and
// their look-back goes by groups of tiles (kGroups) instead of a window.
// 1 M u64 keys with u32 values: 178 us with tiles of 7168 and a window of
// 4, 168 with tiles of 4096, 145 with groups as well.
constexpr int kMidNT = 1024;
constexpr int kMidIPT = 4;
constexpr uint64_t kMidTiles = 2;
constexpr int kGroups = 0;  // as a look-back window
constexpr uint64_t mid_rows(uint64_t cus, uint64_t tile) { return cus * kMidTiles * tile; }

// Consecutive tiles that one XCD's queue takes at a time.  Fewer share fewer
// lines; more keep the chunks after them waiting in their look-back (2^26
// u64 pairs, tiles of 12288: 8 3.74 ms, 16 4.03; 2^27 u64 keys with u32
// values, tiles of 7168: 8 6.20 ms, 16 6.10).
template <int TILE>
constexpr uint32_t kChunkOf = TILE >= 12288 ? 8 : 16;
constexpr uint32_t kMinChunk = 8;

// Look-back status words: 32 bits (2 flag bits, a 30-bit count) for up to
// 2^30 - 1 rows, 64 bits (flags in bits 62-63) beyond, up to 2^31 - 1.
template <class S>
struct StatusWord;
template <>
struct StatusWord<uint32_t> {
  static constexpr uint32_t kAgg = kFlagAgg, kIncl = kFlagIncl, kMask = kCountMask;
};
template <>
struct StatusWord<uint64_t> {
  static constexpr uint64_t kAgg = kFlagAgg64, kIncl = kFlagIncl64, kMask = kCountMask64;
};

template <class S>
__device__ __forceinline__ void sw_store(S* p, S v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class S>
__device__ __forceinline__ S sw_load(const S* p) {
  return __hip_atomic_load(const_cast<S*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Exclusive prefix of column `col` of tile `tile` (stride words between
// tiles), polling W predecessors per round trip: they are consumed in
// order up to the first word not yet published (polled again from there)
// or the first inclusive prefix.  Tiles before tile 0 count as an
// inclusive prefix of 0.
template <int W, class S>
__device__ __forceinline__ uint32_t sort_lookback(const S* status, uint32_t tile, uint32_t stride,
                                                  uint32_t col) {
  using SW = StatusWord<S>;
  uint32_t excl = 0;
  int64_t k = static_cast<int64_t>(tile) - 1;
  while (true) {
    S v[W];
#pragma unroll
    for (int i = 0; i < W; ++i)
      v[i] = (k - i >= 0) ? sw_load(status + static_cast<uint64_t>(k - i) * stride + col) : SW::kIncl;
    bool stop = false, fin = false;
    int used = 0;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const S f = v[i] & ~SW::kMask;
      const bool take = !stop && f != 0;
      excl += take ? static_cast<uint32_t>(v[i] & SW::kMask) : 0u;
      used += take;
      fin |= take && f == SW::kIncl;
      stop |= (f == 0) || (take && f == SW::kIncl);
    }
    if (fin) return excl;
    k -= used;
    if (used < W) __builtin_amdgcn_s_sleep(1);
  }
}

// Hides x's value from the optimiser, so that what is computed from it
// before is computed again afterwards instead of being kept in registers.
template <class T>
__device__ __forceinline__ void opaque(T& x) {
  if constexpr (sizeof(T) <= 4) {
    uint32_t t = x;
    asm volatile("" : "+v"(t));
    x = static_cast<T>(t);
  } else if constexpr (sizeof(T) == 8) {
    asm volatile("" : "+v"(x));
  } else {
    asm volatile("" : "+v"(x.lo), "+v"(x.hi));
  }
}

// The same prefix when every tile of the sort runs at once: the tiles have
// all published their aggregates and none has a prefix yet, so a walk back
// reads most of them (1 M rows: 245 tiles, 10 us of an 18 us pass).  Instead
// the last tile of each group of kGroup adds up its group's aggregates and
// publishes the sum; a tile adds the aggregates before it in its group and
// the sums of the groups before.  Tiles only wait for lower ones.
constexpr uint32_t kGroup = 16;

template <class S>
__device__ __forceinline__ uint32_t sum_words(const S* p, uint32_t count, uint32_t stride) {
  using SW = StatusWord<S>;
  uint32_t sum = 0;
  for (uint32_t i = 0; i < count; i += 8) {
    S v[8];
    bool all;
    do {
      all = true;
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j)
        v[j] = i + j < count ? sw_load(p + static_cast<uint64_t>(i + j) * stride) : SW::kAgg;
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) all &= (v[j] & ~SW::kMask) != 0;
    } while (!all);
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) sum += static_cast<uint32_t>(v[j] & SW::kMask);
  }
  return sum;
}

template <class S>
__device__ __forceinline__ uint32_t sort_lookback_groups(const S* status, S* sums, uint32_t tile,
                                                         uint32_t stride, uint32_t col,
                                                         uint32_t own) {
  using SW = StatusWord<S>;
  const uint32_t g = tile / kGroup, in = tile % kGroup;
  const uint32_t before =
      sum_words(status + static_cast<uint64_t>(tile - in) * stride + col, in, stride);
  if (in == kGroup - 1)
    sw_store<S>(sums + static_cast<uint64_t>(g) * stride + col,
                SW::kAgg | static_cast<S>(before + own));
  return before + sum_words(sums + col, g, stride);
}

// ---- tiles -----------------------------------------------------------------
// The pass's blocks are persistent and take tiles until none is left, except
// where there are as many as tiles and one ticket: then each takes one.  With
// first == 0 every tile comes from one ticket.  Otherwise blocks are split
// over kQueues queues by blockIdx, which the hardware deals out to the XCDs
// in turn, and a queue hands out chunks of consecutive tiles (`first` tiles,
// one for each of its blocks, then kChunk at a time): their runs of one
// digit are neighbours in the output, so the cache lines that two tiles
// share are completed in one XCD's L2 instead of being written twice, in
// part, from two of them.
//
// A chunk's first tile (plus 1) is kept in the queue's list.  It comes from
// the global ticket: chunk 0's with the queue's first tile, chunk k + 1's
// with the first tile of chunk k, so that it is there when chunk k + 1
// begins.  Whoever numbers chunk k + 1 has waited for chunk k's number, so
// a queue's chunks are in increasing order.
//
// Progress: a queue hands out its tiles in increasing order, to any block of
// the queue that is running, and a block exits only when its queue's next
// chunk lies past the last tile.  So the lowest unfinished tile is either
// held by a running block, whose predecessors are all done, or the next tile
// of a queue whose blocks hold only lower tiles, all done: one of them takes
// it.  Nothing depends on how many blocks are resident.
constexpr uint32_t kQueues = 8;
constexpr uint32_t kCtrLine = 32;  // words between counters (128 bytes)
constexpr uint32_t kCtrWords = (2 + kQueues) * kCtrLine;

// Chunks that one queue's list has room for: a queue that hands out all of
// them, and the ones past the end that its blocks ask for.
constexpr uint64_t queue_list(uint64_t tiles) { return tiles / kMinChunk + 4; }

template <uint32_t kChunk>
struct TileQueue {
  uint32_t* ctr;   // [0] ticket, [kCtrLine] finished blocks, then the queues' counters
  uint32_t* list;  // [kQueues][list_len]
  uint32_t list_len;
  uint32_t first;
  // Ask for a tile (the answer is not waited for) ...
  __device__ __forceinline__ uint32_t ask() const {
    return atomicAdd(first ? ctr + (2 + blockIdx.x % kQueues) * kCtrLine : ctr, 1u);
  }
  // ... and the tile that the answer stands for (past the last one: none).
  __device__ __forceinline__ uint32_t tile(uint32_t i) const {
    if (!first) return i;
    uint32_t* l = list + (blockIdx.x % kQueues) * list_len;
    const uint32_t k = i < first ? 0 : 1 + (i - first) / kChunk;
    const uint32_t in = i < first ? i : (i - first) % kChunk;
    if (k >= list_len) return ~0u;
    if (i == 0) sw_store(l, atomicAdd(ctr, first) + 1);
    uint32_t t;
    while ((t = sw_load(l + k)) == 0) __builtin_amdgcn_s_sleep(1);
    if (in == 0 && k + 1 < list_len) sw_store(l + k + 1, atomicAdd(ctr, kChunk) + 1);
    return t - 1 + in;
  }
};

// Rows of status words of one pass: the tiles, then the groups of a sort
// whose tiles all run at once (at most kGroupedTiles; a larger sort has rows
// for as many, so that more tiles never need fewer rows).
constexpr uint64_t kGroupedTiles = 2048;
__host__ __device__ constexpr uint64_t status_rows(uint64_t tiles) {
  return tiles + ((tiles < kGroupedTiles ? tiles : kGroupedTiles) + kGroup - 1) / kGroup;
}

// Tiles per resident block from which the queues pay.  Their chunks wait for
// one another in the look-back, so with few of them, or where a tile writes
// little, one ticket is faster (whole sorts, ms by queues / by one ticket):
// (4, 4) 14 M rows 0.306 / 0.274, 30 M 0.573 / 0.620; (8, 4) 14 M 0.805 / 0.755,
// 20 M 1.093 / 1.168; (4, 1) 30 M 0.500 / 0.483, 64 M 0.981 / 0.993; (16, 0) 14 M
// 2.06 / 1.97, 30 M 4.16 / 4.65; (8, 0) 64 M 2.58 / 2.51, 134 M 5.06 / 5.23;
// (4, 0) 64 M 0.825 / 0.764, 268 M 2.97 / 2.89.
template <int KB, int VB>
constexpr uint64_t kQueueFrom = VB >= 4             ? 4
                                : VB > 0 || KB == 16 ? 8
                                : KB == 8            ? 24
                                                     : 64;

struct SortLayout {
  uint32_t* hist;    // [P][bins]
  uint32_t* base;    // [P][bins] exclusive global digit offsets
  uint32_t* ctrs;    // [P][kCtrWords] tile queues
  uint32_t* lists;   // [P][kQueues][queue_list(tiles)] their chunks
  uint32_t* skip;    // [P]
  uint32_t* sel;     // [1]      0: data in caller's buffers, 1: in pong
  void* status;      // [P][status_rows(tiles)][bins] status words of S
  void* pong_keys;
  void* pong_vals;
  uint64_t zero_words;  // words from hist to the end of status
};

static void carve_sort(Carve& c, uint64_t n, int kb, int vb, int passes, uint64_t tiles,
                       uint32_t bins, SortLayout* L, bool wide = false) {
  // The zeroed block comes first so it is one contiguous range.
  const uint64_t status_words = static_cast<uint64_t>(passes) * status_rows(tiles) * bins;
  L->hist = c.take<uint32_t>(static_cast<uint64_t>(passes) * bins);
  L->base = c.take<uint32_t>(static_cast<uint64_t>(passes) * bins);
  L->ctrs = c.take<uint32_t>(static_cast<uint64_t>(passes) * kCtrWords);
  L->lists = c.take<uint32_t>(static_cast<uint64_t>(passes) * kQueues * queue_list(tiles));
  L->skip = c.take<uint32_t>(static_cast<uint64_t>(passes));
  L->sel = c.take<uint32_t>(1);
  L->status = wide ? static_cast<void*>(c.take<uint64_t>(status_words))
                   : static_cast<void*>(c.take<uint32_t>(status_words));
  L->zero_words = (c.off - (reinterpret_cast<uintptr_t>(L->hist) - c.base)) / 4;
  L->pong_keys = c.take<char>(n * kb);
  L->pong_vals = vb ? c.take<char>(n * vb) : nullptr;
}

template <int DB>
__device__ __forceinline__ uint32_t pass_mask(int pass, uint32_t key_bits) {
  uint32_t width = key_bits - static_cast<uint32_t>(DB * pass);
  if (width > DB) width = DB;
  return (1u << width) - 1u;
}

// Digit of key k at `shift`.  8-bit digits never straddle a 32-bit half of
// a 64-bit key (digit_of's fast form); wider ones may, and take the
// 64-bit shift.
template <int DB, class K>
__device__ __forceinline__ uint32_t dig(K k, uint32_t shift, uint32_t m) {
  if constexpr (DB == 8 || sizeof(K) <= 4) {
    return digit_of(k, shift, m);
  } else {
    static_assert(sizeof(K) == 8, "digits wider than 8 bits are for keys of up to 8 bytes");
    return static_cast<uint32_t>(k >> shift) & m;
  }
}

// Histogram of every digit position in one read of the keys.  With an
// aligned key pointer each thread reads 16 bytes at a time.  Blocks are
// large and few, since each adds its bins to the global ones by atomics
// (1 M u64 keys: 245 blocks of 256 threads 18.7 us, mostly those adds).  The
// last block to finish scans every digit's bins into offsets and flags the
// identity passes.
constexpr int kHistNT = 1024;
template <int KB, bool VEC, int DB>
__global__ __launch_bounds__(kHistNT) void k_radix_hist(
    const typename Elem<KB>::T* __restrict__ keys, uint64_t n, int passes, uint32_t key_bits,
    uint32_t* __restrict__ hist, uint32_t* __restrict__ base, uint32_t* __restrict__ skip,
    uint32_t* __restrict__ finished) {
  using K = typename Elem<KB>::T;
  constexpr int kBins = kBinsOf<DB>;
  constexpr int PER = (VEC && KB < 16) ? 16 / KB : 1;
  __shared__ bool s_last;
  __shared__ uint32_t lh[(8 * KB + DB - 1) / DB * kBins];
  for (int i = threadIdx.x; i < passes * kBins; i += kHistNT) lh[i] = 0;
  __syncthreads();
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kHistNT;
  const uint64_t gtid = blockIdx.x * static_cast<uint64_t>(kHistNT) + threadIdx.x;
  auto count = [&](K k) {
    for (int p = 0; p < passes; ++p)
      atomicAdd(&lh[p * kBins + dig<DB>(k, DB * p, pass_mask<DB>(p, key_bits))], 1u);
  };
  uint64_t done = 0;
  if constexpr (PER > 1) {
    // A 16-byte vector whose keys share a digit adds once; when every lane's
    // vector shares one digit (sorted or low-cardinality keys), the first
    // lane adds for the whole wave instead of 64 lanes hitting one word.
    struct alignas(16) Vec { K k[PER]; };
    const Vec* kv = reinterpret_cast<const Vec*>(keys);
    const uint64_t nvec = n / PER;
    for (uint64_t v = gtid; v < nvec; v += stride) {
      const Vec x = kv[v];
      const uint64_t active = ballot(true);
      for (int p = 0; p < passes; ++p) {
        const uint32_t sh = DB * p, m = pass_mask<DB>(p, key_bits);
        const uint32_t d = dig<DB>(x.k[0], sh, m);
        bool same = true;
#pragma unroll
        for (int e = 1; e < PER; ++e) same &= dig<DB>(x.k[e], sh, m) == d;
        if (ballot(same) == active) {
          const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
          if (ballot(d != d0) == 0) {
            if (mbcnt(active) == 0)
              atomicAdd(&lh[p * kBins + d], static_cast<uint32_t>(PER * __popcll(active)));
            continue;
          }
        }
        if (same) {
          atomicAdd(&lh[p * kBins + d], static_cast<uint32_t>(PER));
        } else {
#pragma unroll
          for (int e = 0; e < PER; ++e) atomicAdd(&lh[p * kBins + dig<DB>(x.k[e], sh, m)], 1u);
        }
      }
    }
    done = nvec * PER;
  }
  for (uint64_t i = done + gtid; i < n; i += stride) count(keys[i]);
  __syncthreads();
  // The adds' old values are waited for, so a block counts as finished only
  // when its adds are done (a release fence would write the whole L2 back,
  // in every wave: 12 M keys 0.30 -> 0.36 ms).
  uint32_t old = 0;
  for (int i = threadIdx.x; i < passes * kBins; i += kHistNT)
    if (lh[i]) old |= atomicAdd(&hist[i], lh[i]);
  asm volatile("" ::"v"(old) : "memory");
  __syncthreads();
  if (threadIdx.x == 0) s_last = atomicAdd(finished, 1u) == gridDim.x - 1;
  __syncthreads();
  if (!s_last) return;
  // One wave per digit, kBins / 64 consecutive bins per lane.
  constexpr int PL = kBins / kWave;
  for (int p = static_cast<int>(wave_id()); p < passes; p += kHistNT / kWave) {
    const uint32_t at = p * kBins + lane_id() * PL;
    uint32_t c[PL], sum = 0;
    bool one = false;  // every key has the same digit here
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      c[j] = sw_load(hist + at + j);
      sum += c[j];
      one |= c[j] == n;
    }
    uint32_t run = wave_incl_scan(sum) - sum;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      base[at + j] = run;
      run += c[j];
    }
    if (one) skip[p] = 1u;  // at most one lane: the bins add up to n
  }
}

// The lanes whose digit is this lane's.  acc collects, per lane, the lanes
// whose digit differs in some bit: x is the lane's bit b as 0 or all ones,
// and acc | (bb ^ x) is one bitop3 per 32-bit half (table 0xDE with acc in
// the middle operand is the same under either operand order of the truth
// table).  Bits above a narrow last digit are zero everywhere and change
// nothing.
template <int DB>
__device__ __forceinline__ uint64_t same_digit(uint32_t d) {
  uint32_t acc_lo = 0, acc_hi = 0;
#pragma unroll
  for (int b = 0; b < DB; ++b) {
    const uint32_t x = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(d), b, 1));
    // The ballot of x itself (a plain ballot(x != 0) is rewritten into a
    // second shift-and-compare of d); 33 is the not-equal predicate.  Lanes
    // outside exec give 0, as a ballot does.
    const uint64_t bb = __builtin_amdgcn_uicmp(x, 0u, 33);
    acc_lo = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(bb), acc_lo, x, 0xDE);
    acc_hi = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(bb >> 32), acc_hi, x, 0xDE);
  }
  return ~((static_cast<uint64_t>(acc_hi) << 32) | acc_lo);
}

// A whole sort in one block: rows in registers, every pass's exchange
// through LDS.  Seven launches and the trips of a look-back are what a small
// sort costs otherwise (u32 pairs, the call alone: 1,000 rows 35 -> 11 us,
// 4,099 39 -> 20, 8,000 45 -> 27; past that one CU takes longer than the
// passes do).  Digits in which no two keys differ are left out.
constexpr int kBlockNT = 1024;
template <int KB, int VB>
constexpr int kBlockIPT = (KB > VB ? KB : VB) >= 16 ? 4 : 8;

template <int KB, int VB>
__global__ __launch_bounds__(kBlockNT) void k_sort_block(typename Elem<KB>::T* __restrict__ keys,
                                                         typename Elem<VB>::T* __restrict__ vals,
                                                         uint32_t n, uint32_t key_bits) {
  using K = typename Elem<KB>::T;
  using V = typename Elem<VB>::T;
  constexpr int IPT = kBlockIPT<KB, VB>;
  constexpr int NW = kBlockNT / kWave, kBins = 256, NBW = kBins / kWave;
  __shared__ __attribute__((aligned(16))) K kbuf[kBlockNT * IPT];
  __shared__ __attribute__((aligned(16))) V vbuf[VB > 0 ? kBlockNT * IPT : 1];
  __shared__ __attribute__((aligned(16))) uint16_t wcnt[NW][kBins];
  __shared__ uint32_t s_scan[NBW];
  __shared__ uint32_t s_vary[4];  // bits in which some key differs from the first
  const uint32_t tid = threadIdx.x, lane = lane_id(), w = wave_id();
  // Wave w holds rows w*64*ipt .. of the present order, 64 to a step.
  const uint32_t ipt = (n + kBlockNT - 1) / kBlockNT;
  const uint32_t row0 = w * ipt * kWave + lane;
  if (tid < 4) s_vary[tid] = 0;
  const K first = keys[0];
  K k[IPT];
  V v[IPT];
  u128 vary{0, 0};
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = row0 + j * kWave;
    if (static_cast<uint32_t>(j) < ipt && i < n) {
      k[j] = keys[i];
      if constexpr (VB > 0) v[j] = vals[i];
      const u128 a = to128(k[j]), b = to128(first);
      vary.lo |= a.lo ^ b.lo;
      if constexpr (KB == 16) vary.hi |= a.hi ^ b.hi;
    }
  }
  __syncthreads();
  {
    const uint32_t words[4] = {static_cast<uint32_t>(vary.lo), static_cast<uint32_t>(vary.lo >> 32),
                               static_cast<uint32_t>(vary.hi), static_cast<uint32_t>(vary.hi >> 32)};
#pragma unroll
    for (int q = 0; q < (KB + 3) / 4; ++q) {
      uint32_t x = words[q];
#pragma unroll
      for (int d = kWave / 2; d > 0; d >>= 1) x |= __shfl_xor(x, d, kWave);
      if (lane == 0 && x) atomicOr(&s_vary[q], x);
    }
  }
  for (uint32_t shift = 0; shift < key_bits; shift += 8) {
    const uint32_t dmask = key_bits - shift < 8 ? (1u << (key_bits - shift)) - 1u : 0xFFu;
    __syncthreads();  // the last exchange is read (before the first digit: s_vary is written)
    if (!((s_vary[shift / 32] >> (shift % 32)) & dmask)) continue;  // uniform
#pragma unroll
    for (int q = 0; q < NW * kBins / 2 / kBlockNT; ++q)
      reinterpret_cast<uint32_t*>(&wcnt[0][0])[tid + q * kBlockNT] = 0;
    __syncthreads();
    uint32_t pos[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      if (static_cast<uint32_t>(j) < ipt) {
        const bool valid = row0 + j * kWave < n;
        const uint32_t d = digit_of(k[j], shift, dmask);
        const uint64_t m = ballot(valid) & same_digit<8>(d);
        const uint32_t below = mbcnt(m);
        uint32_t prior = 0;
        if (valid) {
          prior = wcnt[w][d];
          const uint32_t cnt = __popcll(m);
          if (below == cnt - 1) wcnt[w][d] = static_cast<uint16_t>(prior + cnt);
        }
        pos[j] = prior + below;
      }
    }
    __syncthreads();
    uint32_t total = 0;
    if (tid < kBins) {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) total += wcnt[ww][tid];
    }
    uint32_t start = wave_incl_scan(total);
    if (w < NBW && lane == kWave - 1) s_scan[w] = start;
    start -= total;
    __syncthreads();
    if (tid < kBins) {
#pragma unroll
      for (int i = 0; i < NBW; ++i) start += static_cast<uint32_t>(i) < w ? s_scan[i] : 0u;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        const uint32_t c = wcnt[ww][tid];
        wcnt[ww][tid] = static_cast<uint16_t>(start);
        start += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      if (static_cast<uint32_t>(j) < ipt && row0 + j * kWave < n) {
        const uint32_t at = pos[j] + wcnt[w][digit_of(k[j], shift, dmask)];
        kbuf[at] = k[j];
        if constexpr (VB > 0) vbuf[at] = v[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint32_t i = row0 + j * kWave;
      if (static_cast<uint32_t>(j) < ipt && i < n) {
        k[j] = kbuf[i];
        if constexpr (VB > 0) v[j] = vbuf[i];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = row0 + j * kWave;
    if (static_cast<uint32_t>(j) < ipt && i < n) {
      keys[i] = k[j];
      if constexpr (VB > 0) vals[i] = v[j];
    }
  }
}

template <int KB, int VB, int NT, int IPT, int DB, int LBW, class S>
__global__ __launch_bounds__(NT, 4) void k_onesweep(
    typename Elem<KB>::T* __restrict__ k0, typename Elem<KB>::T* __restrict__ k1,
    typename Elem<VB>::T* __restrict__ v0, typename Elem<VB>::T* __restrict__ v1, uint64_t n,
    int pass, uint32_t key_bits, const uint32_t* __restrict__ base, uint32_t* __restrict__ ctrs,
    const uint32_t* __restrict__ skip, uint32_t* __restrict__ sel, S* __restrict__ status,
    uint32_t ntiles, uint32_t first, uint32_t* __restrict__ lists, uint32_t list_len) {
  using K = typename Elem<KB>::T;
  using V = typename Elem<VB>::T;
  constexpr int NW = NT / kWave;
  constexpr int TILE = NT * IPT;
  constexpr int RB = (KB > VB ? KB : VB) * TILE;
  constexpr int kBins = kBinsOf<DB>;
  constexpr int BPT = (kBins + NT - 1) / NT;  // bins per thread in the per-bin steps
  constexpr int NBW = (kBins < NT ? kBins : NT) / kWave;  // waves that hold bins
  constexpr int kScatterBatch = 8;  // scattered at a time: bounds the registers in flight
  // Wave counters and tile positions stay below TILE: 16 bits hold them,
  // which keeps the wider digits' counters within LDS.
  using WC = uint16_t;
  static_assert(TILE <= 65535 && IPT % 2 == 0, "16-bit wave counters, packed positions");

  if (skip[pass]) return;
  const uint32_t cur = *sel;
  const K* __restrict__ kin = cur ? k1 : k0;
  K* __restrict__ kout = cur ? k0 : k1;
  const V* __restrict__ vin = cur ? v1 : v0;
  V* __restrict__ vout = cur ? v0 : v1;

  __shared__ uint32_t s_tile;
  __shared__ __attribute__((aligned(16))) WC wcnt[NW][kBins];
  __shared__ uint32_t gdelta[kBins];
  __shared__ uint32_t s_scan[BPT][NBW];
  __shared__ __attribute__((aligned(16))) unsigned char rbuf[RB];

  const uint32_t n32 = static_cast<uint32_t>(n);
  const uint32_t shift = static_cast<uint32_t>(DB * pass);
  const uint32_t dmask = pass_mask<DB>(pass, key_bits);

  uint32_t tid = threadIdx.x, lane = lane_id();
  const uint32_t w = wave_id();
  const TileQueue<kChunkOf<TILE>> queue{ctrs + pass * kCtrWords, lists + pass * kQueues * list_len, list_len, first};
  if (tid == 0) s_tile = queue.tile(queue.ask());
  // One tile per block: as many blocks as tiles, by the ticket.
  const bool once = first == 0 && gridDim.x == ntiles;
  using SW = StatusWord<S>;
  S* st = status + (static_cast<uint64_t>(pass) * status_rows(ntiles)) * kBins;

  // Every tile but the last is full: its copy of the body has no per-key
  // bounds checks.
  auto body = [&](uint32_t tile, auto full_tag) {
    constexpr bool FULL = decltype(full_tag)::value;
    const uint64_t tile_base = static_cast<uint64_t>(tile) * TILE;
    const uint64_t wave_base = tile_base + static_cast<uint64_t>(w) * kWave * IPT;
    // Keys only: values are read after the keys are ranked, which keeps
    // the ranking phase's register footprint small.
    K keys[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint64_t idx = wave_base + static_cast<uint64_t>(j) * kWave + lane;
      if (FULL) keys[j] = kin[idx];
      else keys[j] = idx < n ? kin[idx] : K{};
    }

    // Stable rank within the wave: lanes sharing a digit are found by one
    // ballot per digit bit; the highest such lane bumps the wave counter.
    // (An LDS atomic per group leader, issued for all keys before any
    // result is used, measured slower on MI355X: 1.67 against 1.45 ms per
    // pass.)
    uint32_t pos[IPT / 2];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint64_t idx = wave_base + static_cast<uint64_t>(j) * kWave + lane;
      const bool valid = FULL || idx < n;
      const uint32_t d = dig<DB>(keys[j], shift, dmask);
      const uint64_t m = (FULL ? ~0ull : ballot(valid)) & same_digit<DB>(d);
      const uint32_t below = mbcnt(m);
      const uint32_t cnt = __popcll(m);
      uint32_t prior = 0;
      if (valid) {
        prior = wcnt[w][d];
        if (below == cnt - 1) wcnt[w][d] = static_cast<WC>(prior + cnt);
      }
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t r = prior + below;
      pos[j / 2] = (j & 1) ? (pos[j / 2] | (r << 16)) : r;
    }
    __syncthreads();

    // The digits and counter addresses of the ranking are not kept (90 -> 80
    // registers at 16 keys).
#pragma unroll
    for (int j = 0; j < IPT; ++j) opaque(keys[j]);
    // Per-digit tile totals and wave prefixes; publish the tile aggregate.
    // wcnt[w][d] becomes the tile position of wave w's first key of digit
    // d: the digit's start in the tile plus the waves before w.
    // Thread t handles bins t, t + NT, ... (one bin, or none, for 8 and 9
    // bits).
    uint32_t total_d[BPT], bs[BPT];
    uint32_t wpre[BPT][NW];
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const uint32_t bin = tid + q * NT;
      total_d[q] = 0;
      if (bin < kBins) {
        uint32_t run = 0;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) {
          wpre[q][ww] = run;
          run += wcnt[ww][bin];
        }
        total_d[q] = run;
        sw_store<S>(st + static_cast<uint64_t>(tile) * kBins + bin,
                    (tile == 0 ? SW::kIncl : SW::kAgg) | static_cast<S>(run));
      }
    }
    // Each digit's start in the tile: scans within the waves, then the
    // totals of the waves before.
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const uint32_t incl = wave_incl_scan(total_d[q]);
      if (w < NBW && lane == kWave - 1) s_scan[q][w] = incl;
      bs[q] = incl - total_d[q];
    }
    __syncthreads();
    {
      uint32_t carry = 0;
#pragma unroll
      for (int q = 0; q < BPT; ++q) {
        uint32_t all = 0;
#pragma unroll
        for (int i = 0; i < NBW; ++i) {
          const uint32_t x = s_scan[q][i];
          bs[q] += static_cast<uint32_t>(i) < w ? x : 0u;
          all += x;
        }
        bs[q] += carry;
        carry += all;
      }
    }
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const uint32_t bin = tid + q * NT;
      if (bin < kBins) {
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) wcnt[ww][bin] = static_cast<WC>(bs[q] + wpre[q][ww]);
      }
    }
    __syncthreads();

    // Work that does not need the global offsets goes before the look-back
    // so it overlaps the wait: the LDS reorder of the keys and the value
    // loads.
    K* kbuf = reinterpret_cast<K*>(rbuf);
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint64_t idx = wave_base + static_cast<uint64_t>(j) * kWave + lane;
      if (FULL || idx < n) {
        const uint32_t d = dig<DB>(keys[j], shift, dmask);
        const uint32_t off = wcnt[w][d];
        const uint32_t at = ((j & 1) ? (pos[j / 2] >> 16) : (pos[j / 2] & 0xFFFFu)) + off;
        pos[j / 2] += (j & 1) ? (off << 16) : off;
        kbuf[at] = keys[j];
      }
    }
    V vals[IPT];
    if constexpr (VB > 0) {
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const uint64_t idx = wave_base + static_cast<uint64_t>(j) * kWave + lane;
        if (FULL || idx < n) vals[j] = vin[idx];
      }
    }
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const uint32_t bin = tid + q * NT;
      if (bin < kBins) {
        uint32_t excl = 0;
        if constexpr (LBW == kGroups) {
          excl = sort_lookback_groups<S>(st, st + static_cast<uint64_t>(ntiles) * kBins, tile,
                                         kBins, bin, total_d[q]);
        } else if (tile > 0) {
          excl = sort_lookback<LBW>(st, tile, kBins, bin);
          sw_store<S>(st + static_cast<uint64_t>(tile) * kBins + bin,
                      SW::kIncl | static_cast<S>(excl + total_d[q]));
        }
        gdelta[bin] = base[pass * kBins + bin] + excl - bs[q];
      }
    }
    __syncthreads();

    const uint32_t tile_n =
        FULL ? static_cast<uint32_t>(TILE)
             : static_cast<uint32_t>((n - tile_base) < TILE ? (n - tile_base) : TILE);
    uint32_t dst[IPT];
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
      if (k % kScatterBatch == 0) __builtin_amdgcn_sched_barrier(0);
      const uint32_t i = k * NT + tid;
      if (FULL || i < tile_n) {
        const K key = kbuf[i];
        const uint32_t d = dig<DB>(key, shift, dmask);
        dst[k] = gdelta[d] + i;
        if (dst[k] < n32) kout[dst[k]] = key;  // always true when ranks are right
      }
    }
    // The next tile is asked for while this one is still being stored.
    uint32_t next = 0;
    if constexpr (VB == 0) {
      if (tid == 0 && !once) s_tile = queue.tile(queue.ask());
    }
    if constexpr (VB > 0) {
      __syncthreads();  // every key is out of kbuf
      V* vbuf = reinterpret_cast<V*>(rbuf);
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const uint64_t idx = wave_base + static_cast<uint64_t>(j) * kWave + lane;
        if (FULL || idx < n) vbuf[(j & 1) ? (pos[j / 2] >> 16) : (pos[j / 2] & 0xFFFFu)] = vals[j];
      }
      __syncthreads();
      if (tid == 0 && !once) next = queue.ask();
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
        if (k % kScatterBatch == 0) __builtin_amdgcn_sched_barrier(0);
        const uint32_t i = k * NT + tid;
        if (FULL || i < tile_n) {
          if (dst[k] < n32) vout[dst[k]] = vbuf[i];
        }
      }
      if (tid == 0 && !once) s_tile = queue.tile(next);
    }
  };
  for (;;) {
    // Opaque to the compiler in each round: addresses made of them are
    // worked out where they are used, not kept in registers around the loop.
    opaque(tid);
    opaque(lane);
    for (uint32_t i = tid; i < NW * kBins / 2; i += NT)
      reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0;
    __syncthreads();
    const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);  // block-uniform: scalar from here
    if (tile >= ntiles) break;
    if (static_cast<uint64_t>(tile) * TILE + TILE <= n) body(tile, std::true_type{});
    else body(tile, std::false_type{});
    if (once) break;
  }

  // The last block to finish flips the buffer selector.  Every block read
  // *sel before arriving here, so nobody reads the new value this pass.
  if (tid == 0) {
    const uint32_t prev = atomicAdd(&queue.ctr[kCtrLine], 1u);
    if (prev == gridDim.x - 1)
      __hip_atomic_store(sel, cur ^ 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <int KB, int VB>
__global__ __launch_bounds__(256) void k_copyback(typename Elem<KB>::T* __restrict__ k0,
                                                  const typename Elem<KB>::T* __restrict__ k1,
                                                  typename Elem<VB>::T* __restrict__ v0,
                                                  const typename Elem<VB>::T* __restrict__ v1,
                                                  uint64_t n, const uint32_t* __restrict__ sel) {
  if (*sel == 0) return;
  uint64_t stride = static_cast<uint64_t>(gridDim.x) * 256;
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += stride) {
    k0[i] = k1[i];
    if constexpr (VB > 0) v0[i] = v1[i];
  }
}

// Tunable tile shapes: the autotuner may pick 8, 12 or 16 keys per thread
// (of 512) for 4- and 8-byte keys with 0-, 4- or 8-byte values; other shapes
// keep the default.  The smallest tile needs the most look-back status
// words.
template <int KB, int VB>
constexpr bool kSortTunable = (KB == 4 || KB == 8) && (VB == 0 || VB == 4 || VB == 8);
constexpr int kTuneNT = 512;
constexpr int kSortMinIPT = 8;

uint64_t sort_ws_tile(uint64_t n, int kb, int vb, int key_bits, uint64_t tile, int db,
                      bool wide = false) {
  const int passes = (key_bits + db - 1) / db;
  const uint64_t tiles = (n + tile - 1) / tile;
  Carve s(nullptr);
  SortLayout L;
  carve_sort(s, n, kb, vb, passes, tiles, 1u << db, &L, wide);
  return s.off;
}

// Sorts of more than 2^30 - 1 rows take 64-bit look-back status words, at
// the default tile and 8-bit digits.
constexpr uint64_t kSortMaxRows = (1ull << 31) - 1;

// Digit width chosen for key_bits when the context does not set one.  An
// odd number of passes leaves the data in the pong buffer and costs a copy
// back (about 0.87 ms for 2^28 u32 pairs, a full read and write), so 17-20
// bit keys take two passes of 9 or 10 bits instead of three of 8: 2^28
// pairs, 18 bits 3.36 ms against 5.04, 20 bits 4.04 against 4.90.  Wider
// keys keep 8 bits (26 bits: 5.51 ms against 5.65 with 9; 32 bits: 5.56
// against 6.29).
// Narrower digits have fewer bins per tile, so fewer lines written in part:
// 25-28 bit keys take four passes of 7 bits, and 21-24 bit keys, from the
// rows on where four passes of 6 bits are faster than three of 8 and the copy
// (24 bits, ms by 6 / by 8 bits: u32 pairs 1.5 M rows 0.086 / 0.071, 16 M 0.293 /
// 0.268, 24 M 0.433 / 0.441, 64 M 1.01 / 1.05; u32 keys alone 24 M 0.298 / 0.275,
// 64 M 0.686 / 0.700).
constexpr uint64_t six_bits_from(int val_bytes) { return val_bytes ? 20'000'000 : 64'000'000; }
constexpr int auto_digit(int key_bits, uint64_t n, int val_bytes) {
  return key_bits >= 17 && key_bits <= 18   ? 9
         : key_bits >= 19 && key_bits <= 20 ? 10
         : key_bits >= 21 && key_bits <= 24 ? (n < six_bits_from(val_bytes) ? 8 : 6)
         : key_bits >= 25 && key_bits <= 28 ? 7
                                            : 8;
}

// Workspace for any tile shape the context may be tuned to, at the digit
// width chosen for key_bits (a context tuned to other digit widths grows
// its own workspace on first use).
template <int KB, int VB>
uint64_t sort_ws_bytes(uint64_t n, int key_bits) {
  using Tn = SortTune<KB, VB, 8>;
  const uint64_t tile = static_cast<uint64_t>(Tn::NT) * Tn::IPT;
  if (n > kCountMask) {
    // 64-bit words for larger tiles: no less than the most rows with 32-bit
    // words and the smallest tile take.
    const uint64_t wide = sort_ws_tile(n, KB, VB, key_bits, tile, 8, true);
    const uint64_t narrow = sort_ws_bytes<KB, VB>(kCountMask, key_bits);
    return wide > narrow ? wide : narrow;
  }
  constexpr uint64_t kMinTile = kTuneNT * (kSortTunable<KB, VB> ? kSortMinIPT : Tn::kFewIPT);
  uint64_t ws = sort_ws_tile(n, KB, VB, key_bits, kMinTile < tile ? kMinTile : tile, 8);
  const int digit = auto_digit(key_bits, n, VB);
  if (kSortTunable<KB, VB> && digit != 8) {
    const uint64_t w2 =
        sort_ws_tile(n, KB, VB, key_bits, digit > 8 ? kTuneNT * 12ull : kMinTile, digit);
    if (w2 > ws) ws = w2;
  }
  return ws;
}

template <int KB, int VB, int NT, int IPT, int DB, int LBW = kWindow, class S = uint32_t>
int sort_impl(rfx_ctx* ctx, void* keys, void* vals, uint64_t n, int key_bits) {
  using K = typename Elem<KB>::T;
  using V = typename Elem<VB>::T;
  constexpr int TILE = NT * IPT;
  constexpr bool kWide = sizeof(S) == 8;
  if (n < 2) return RFX_OK;
  if (n > (kWide ? kSortMaxRows : static_cast<uint64_t>(kCountMask)))
    return fail(RFX_ERANGE, "sort: %llu rows exceeds 2^31-1", static_cast<unsigned long long>(n));
  constexpr uint32_t kBins = kBinsOf<DB>;
  const int passes = (key_bits + DB - 1) / DB;
  const uint64_t tiles = (n + TILE - 1) / TILE;
  RFX_TRY(ensure_workspace(ctx, sort_ws_tile(n, KB, VB, key_bits, TILE, DB, kWide)));
  Carve c(ctx->ws);
  SortLayout L;
  carve_sort(c, n, KB, VB, passes, tiles, kBins, &L, kWide);
  RFX_TRY(fill_u32(ctx, L.hist, L.zero_words, 0u));

  // 8 rows a thread up to one block per CU (1 M u64 keys: 137 us the whole
  // sort, 144 with 16), then 16, up to two blocks.
  const uint64_t cus = static_cast<uint64_t>(ctx->device_cus);
  uint64_t hb = (n + kHistNT * 8 - 1) / (kHistNT * 8);
  if (hb > cus) hb = hb / 2 > cus ? hb / 2 : cus;
  if (hb > 2 * cus) hb = 2 * cus;
  {
    RFX_PROF(ctx, "sort.hist");
    if (reinterpret_cast<uintptr_t>(keys) % 16 == 0)
      k_radix_hist<KB, true, DB><<<static_cast<uint32_t>(hb), kHistNT, 0, ctx->stream>>>(
          static_cast<const K*>(keys), n, passes, static_cast<uint32_t>(key_bits), L.hist, L.base,
          L.skip, L.ctrs + 1);
    else
      k_radix_hist<KB, false, DB><<<static_cast<uint32_t>(hb), kHistNT, 0, ctx->stream>>>(
          static_cast<const K*>(keys), n, passes, static_cast<uint32_t>(key_bits), L.hist, L.base,
          L.skip, L.ctrs + 1);
    RFX_LAUNCHED();
  }
  static const int per_cu = [] {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &b, reinterpret_cast<const void*>(k_onesweep<KB, VB, NT, IPT, DB, LBW, S>), NT, 0) !=
            hipSuccess || b < 1)
      b = 1;
    return b;
  }();
  const uint64_t slots = static_cast<uint64_t>(ctx->device_cus) * per_cu;
  // A server's context (its workspace is the request's) shares the GPU with
  // other requests' kernels: there each block takes one tile and gives its
  // slot back, since blocks that stay until the pass ends keep the others
  // waiting.  The saturated served mix: 1,103 requests/s with blocks that
  // stay, 1,369 with one tile each (1,254 before there were any that stay);
  // one request at a time, where nothing waits: 993 and 982.
  const bool shared = ctx->ws_borrowed;
  const uint32_t grid = static_cast<uint32_t>(tiles < slots || shared ? tiles : slots);
  const uint32_t first =
      tiles > kQueueFrom<KB, VB> * slots && !shared ? (grid + kQueues - 1) / kQueues : 0;
  for (int p = 0; p < passes; ++p) {
    RFX_PROF(ctx, "sort.onesweep");
    k_onesweep<KB, VB, NT, IPT, DB, LBW, S><<<grid, NT, 0, ctx->stream>>>(
        static_cast<K*>(keys), static_cast<K*>(L.pong_keys), static_cast<V*>(vals),
        static_cast<V*>(L.pong_vals), n, p, static_cast<uint32_t>(key_bits), L.base, L.ctrs,
        L.skip, L.sel, static_cast<S*>(L.status), static_cast<uint32_t>(tiles), first, L.lists,
        static_cast<uint32_t>(queue_list(tiles)));
    RFX_LAUNCHED();
  }
  uint64_t cb = (n + 255) / 256;
  if (cb > 8192) cb = 8192;
  k_copyback<KB, VB><<<static_cast<uint32_t>(cb), 256, 0, ctx->stream>>>(
      static_cast<K*>(keys), static_cast<const K*>(L.pong_keys), static_cast<V*>(vals),
      static_cast<const V*>(L.pong_vals), n, L.sel);
  RFX_LAUNCHED();
  return RFX_OK;
}

// At one digit width: the large tile, or for a sort whose large tiles would
// not fill the chip, a small one.
template <int KB, int VB, int DB>
int sort_digits(rfx_ctx* ctx, void* keys, void* vals, uint64_t n, int key_bits) {
  using Tn = SortTune<KB, VB, DB>;
  constexpr int NT = DB > 8 ? kTuneNT : kMidNT, IPT = DB > 8 ? 12 : kMidIPT;
  if constexpr (kSortTunable<KB, VB>) {
    if (n <= mid_rows(ctx->device_cus, NT * IPT))
      return sort_impl<KB, VB, NT, IPT, DB, kGroups>(ctx, keys, vals, n, key_bits);
  } else if constexpr (Tn::kFewIPT != Tn::IPT) {
    if (n <= mid_rows(ctx->device_cus, kMidNT * kMidIPT))
      return sort_impl<KB, VB, Tn::NT, Tn::kFewIPT, DB>(ctx, keys, vals, n, key_bits);
  }
  return sort_impl<KB, VB, Tn::NT, Tn::IPT, DB>(ctx, keys, vals, n, key_bits);
}

template <int KB, int VB>
int sort_tuned(rfx_ctx* ctx, void* keys, void* vals, uint64_t n, int key_bits) {
  using Tn = SortTune<KB, VB, 8>;
  // More than 2^30 - 1 rows (or the sort.status knob at 64): 64-bit status
  // words, default tile, 8-bit digits.
  if (n > kCountMask || ctx->tune_sort_status == 64)
    return sort_impl<KB, VB, Tn::NT, Tn::IPT, 8, kWindow, uint64_t>(ctx, keys, vals, n,
                                                                         key_bits);
  if (n <= static_cast<uint64_t>(kBlockNT) * kBlockIPT<KB, VB> && !ctx->tune_sort_ipt &&
      !ctx->tune_sort_digit) {
    if (n < 2) return RFX_OK;
    RFX_PROF(ctx, "sort.block");
    k_sort_block<KB, VB><<<1, kBlockNT, 0, ctx->stream>>>(
        static_cast<typename Elem<KB>::T*>(keys), static_cast<typename Elem<VB>::T*>(vals),
        static_cast<uint32_t>(n), static_cast<uint32_t>(key_bits));
    RFX_LAUNCHED();
    return RFX_OK;
  }
  if constexpr (kSortTunable<KB, VB>) {
    // Knob value 0 takes the digit width chosen for key_bits; tiles of a set
    // number of keys exist for 8 bits and wider.
    const int ipt = ctx->tune_sort_ipt;
    int digit = ctx->tune_sort_digit;
    if (!digit) {
      digit = auto_digit(key_bits, n, VB);
      if (ipt && digit < 8) digit = 8;
    }
    if (digit == 6) return sort_digits<KB, VB, 6>(ctx, keys, vals, n, key_bits);
    if (digit == 7) return sort_digits<KB, VB, 7>(ctx, keys, vals, n, key_bits);
    if (digit == 9)
      return ipt == 12 ? sort_impl<KB, VB, kTuneNT, 12, 9>(ctx, keys, vals, n, key_bits)
                       : sort_digits<KB, VB, 9>(ctx, keys, vals, n, key_bits);
    if (digit == 10)
      return ipt == 12 ? sort_impl<KB, VB, kTuneNT, 12, 10>(ctx, keys, vals, n, key_bits)
                       : sort_digits<KB, VB, 10>(ctx, keys, vals, n, key_bits);
    if (ipt == 8) return sort_impl<KB, VB, kTuneNT, 8, 8>(ctx, keys, vals, n, key_bits);
    if (ipt == 12) return sort_impl<KB, VB, kTuneNT, 12, 8>(ctx, keys, vals, n, key_bits);
    if (ipt == 16) return sort_impl<KB, VB, kTuneNT, 16, 8>(ctx, keys, vals, n, key_bits);
  }
  return sort_digits<KB, VB, 8>(ctx, keys, vals, n, key_bits);
}

template <int KB>
int sort_dispatch_v(rfx_ctx* ctx, void* keys, void* vals, uint64_t n, int key_bits, int vb) {
  switch (vb) {
    case 0: return sort_tuned<KB, 0>(ctx, keys, nullptr, n, key_bits);
    case 1: return sort_tuned<KB, 1>(ctx, keys, vals, n, key_bits);
    case 2: return sort_tuned<KB, 2>(ctx, keys, vals, n, key_bits);
    case 4: return sort_tuned<KB, 4>(ctx, keys, vals, n, key_bits);
    case 8: return sort_tuned<KB, 8>(ctx, keys, vals, n, key_bits);
    case 16: return sort_tuned<KB, 16>(ctx, keys, vals, n, key_bits);
    default: return fail(RFX_EINVAL, "sort: value width %d", vb);
  }
}

template <int KB>
uint64_t ws_dispatch_v(uint64_t n, int key_bits, int vb) {
  switch (vb) {
    case 0: return sort_ws_bytes<KB, 0>(n, key_bits);
    case 1: return sort_ws_bytes<KB, 1>(n, key_bits);
    case 2: return sort_ws_bytes<KB, 2>(n, key_bits);
    case 4: return sort_ws_bytes<KB, 4>(n, key_bits);
    case 8: return sort_ws_bytes<KB, 8>(n, key_bits);
    case 16: return sort_ws_bytes<KB, 16>(n, key_bits);
    default: return 0;
  }
}

}  // namespace
}  // namespace rfx

using namespace rfx;

extern "C" int rfx_sort_pairs(rfx_ctx* ctx, void* keys, void* vals, uint64_t n, int key_bytes,
                              int key_bits, int val_bytes) {
  if (!ctx) return fail(RFX_EINVAL, "rfx_sort_pairs: null context");
  if (!valid_width(key_bytes)) return fail(RFX_EINVAL, "rfx_sort_pairs: key width %d", key_bytes);
  if (val_bytes != 0 && !valid_width(val_bytes))
    return fail(RFX_EINVAL, "rfx_sort_pairs: value width %d", val_bytes);
  if (key_bits <= 0 || key_bits > 8 * key_bytes)
    return fail(RFX_EINVAL, "rfx_sort_pairs: key_bits %d for %d-byte keys", key_bits, key_bytes);
  if (n && !keys) return fail(RFX_EINVAL, "rfx_sort_pairs: null keys");
  if (n && val_bytes && !vals) return fail(RFX_EINVAL, "rfx_sort_pairs: null values");
  switch (key_bytes) {
    case 1: return sort_dispatch_v<1>(ctx, keys, vals, n, key_bits, val_bytes);
    case 2: return sort_dispatch_v<2>(ctx, keys, vals, n, key_bits, val_bytes);
    case 4: return sort_dispatch_v<4>(ctx, keys, vals, n, key_bits, val_bytes);
    case 8: return sort_dispatch_v<8>(ctx, keys, vals, n, key_bits, val_bytes);
    case 16: return sort_dispatch_v<16>(ctx, keys, vals, n, key_bits, val_bytes);
  }
  return fail(RFX_EINVAL, "rfx_sort_pairs: key width %d", key_bytes);
}

extern "C" uint64_t rfx_sort_workspace(uint64_t n, int key_bytes, int key_bits, int val_bytes) {
  if (!valid_width(key_bytes) || key_bits <= 0 || key_bits > 8 * key_bytes) return 0;
  switch (key_bytes) {
    case 1: return ws_dispatch_v<1>(n, key_bits, val_bytes);
    case 2: return ws_dispatch_v<2>(n, key_bits, val_bytes);
    case 4: return ws_dispatch_v<4>(n, key_bits, val_bytes);
    case 8: return ws_dispatch_v<8>(n, key_bits, val_bytes);
    case 16: return ws_dispatch_v<16>(n, key_bits, val_bytes);
  }
  return 0;
}
