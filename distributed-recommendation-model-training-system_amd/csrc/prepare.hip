// prepare.hip -- device-side dedup of pushed occurrences by row.
//
// The reference dedups on the host with a hash map in first-occurrence order
// (PrepareFeature, src/access/batch_access.cpp:32-36; ReduceGradients, :73-93)
// and ships either reduced rows or a host-built CSR to the device
// (BuildCompactGradients, src/access/compact_gradients.cpp:43-72).  Here the
// grouping is a stable LSD radix sort of 32-bit keys (key index << row_bits |
// slot), so equal rows end up adjacent in occurrence order -- exactly the CSR
// order of the reference's references (repeats kept, (feature, bag, position)
// order).
//
// A push names its tables, so their key indices need no sorting: the features
// are laid out table by table (in call order within a table) and each table's
// run of occurrences, a segment, is sorted by slot alone.
//
//   keygen : one block per tile of up to 4,096 occurrences of one feature ->
//            key, packed (gradient row | scale) reference word, the tile's
//            digit counts for every pass, its valid count, max |scale|.  Rows
//            not on this device get the sentinel key and are not counted.
//   passes : onesweep (one launch per digit): per-tile stable ranking with
//            wavefront ballots, the digit prefix over the segment's earlier
//            tiles, LDS-staged scatter so each digit run is written
//            contiguously.  The first pass reads the prefix from keygen's
//            counts (its tiles are keygen's); the later ones look back over
//            the tiles' published counts (two levels: tiles, groups of 16).
//            The first pass drops the sentinels, the last one closes the gaps
//            they left between the tables and writes the class boundaries.
//   unique : first-occurrence ranks (PrepareFeature's unique order) from a
//            head-flag scan in occurrence space.
//
// A push of up to 4,096 occurrences is prepared by one block in one launch
// (SmallPrepareKernel): sorted in LDS, hot rows listed on the way out.
//
// Every launch is a chain of dependent steps on about one tile a CU, so what
// counts is their number: sorting whole keys (25 bits for 26 tables of
// 1,000,000 rows) in three 9-bit passes of 256-thread blocks, key generation,
// a clearing launch before it and one position a thread in the hot-row list
// took 116 us for 1.1 M occurrences; 20 bits in two passes of 1,024-thread
// blocks take 70.  4 x 8.4 M occurrences: 1.73 -> 1.27 ms; 65,536: 63 -> 50
// us.  (A pass of the larger blocks still spends 3.5 us on its launch, ~2 on
// ranking, ~2.5 on its tile's loads and ~2-5 on the look-back.)
#include "prepare.hpp"

#include <algorithm>

namespace eps_hip {

namespace {

constexpr uint32_t kSortWaves = kSortBlock / kWave;
constexpr uint32_t kFlagAggregate = 1u << 30;
constexpr uint32_t kFlagInclusive = 2u << 30;
constexpr uint32_t kValueMask = (1u << 30) - 1;
constexpr uint32_t kLookWindow = 8;   // predecessor tiles or groups read per look-back round
constexpr uint32_t kKeyBlock = 1024;    // threads of a keygen block
constexpr uint32_t kKeyItems = kSortTile / kKeyBlock;
// Bag offsets a keygen block stages in LDS: a tile's bags (at most its
// occurrences, runs of empty bags aside) and the search's last step.
constexpr uint32_t kSearchStep = 256, kStageBags = kSortTile + kSearchStep + 1;
constexpr uint32_t kProbes = 128;        // offsets probed in a round of a block's bag search
// Largest number of keygen tiles of a table whose counts a pass's blocks add
// up themselves (each thread one digit, eight loads in flight).  Above it one
// more launch adds them up per table (CountSumKernel), and the first pass
// looks back like the others: 131,000 references on a table of a million rows
// take 43 us with the blocks adding and 54 with the launch, 26 tables of 43,000
// 67 and 77.  Past 32 tiles it depends: 200,000 on one table 48 and 63, but
// 400,000 on each of four 123 and 110.
constexpr uint32_t kDirectTiles = 32;

struct PrepFeature {
  const uint64_t* indices;
  const uint64_t* offsets;
  const uint64_t* lengths;
  const float* weights;
  uint64_t occurrences, bags, table_rows;
  uint32_t occ_begin;   // of the feature in call order: its occurrence indices
  uint32_t sort_begin;  // of the feature in the sort's input
  uint32_t key_index, pooling, block_begin, feature;
};
struct PrepArgs {
  PrepFeature f[EPS_HIP_MAX_FEATURES];  // by table key index, then call order
  uint32_t count, row_bits, sentinel, passes, digits;
  uint32_t shift[kMaxPasses], bits[kMaxPasses];
  Control* ctrl;
  TileInfo* info;
  uint16_t* counts;    // [pass][tile][digit]
  uint32_t tiles;
  uint32_t* keys;
  uint32_t* vals;
  uint64_t* refscale;  // reference words with their scales (8 bytes), or
  uint32_t* refs;      // without (4 bytes: no weighted-sum feature; the scale is derived)
  // Words that keygen's blocks clear beside the control block, for the passes:
  // the look-back flags (and the per-table counts when CountSumKernel runs).
  uint32_t* zero;
  uint64_t zero_words;
};
static_assert(sizeof(PrepArgs) <= 4096, "keygen arguments fit the kernel-argument segment");

// What the last pass needs to put each reference word's scale back (pushes
// with no weighted-sum feature sort 4-byte words without it): the mean
// features and their valid lengths.  The scale is then exactly what keygen
// computes: 1.0f / (float)len for a mean bag of nonzero length, else 1.0f.
struct ScaleArgs {
  const uint64_t* lengths[EPS_HIP_MAX_FEATURES];
  uint32_t mean_mask;  // bit f: feature f is mean-pooled
};

// Clears the control block for a new push, but the status history (its last
// word): nothing else touches the block before the launch that calls this
// has ended.
__device__ __forceinline__ void ClearControl(Control* ctrl, uint32_t threads) {
  for (uint32_t i = threadIdx.x; i < kHistoryWord; i += threads) reinterpret_cast<uint32_t*>(ctrl)[i] = 0;
}

__global__ void __launch_bounds__(kKeyBlock) __attribute__((amdgpu_waves_per_eu(8))) KeygenKernel(PrepArgs args) {
  const PrepFeature f = args.f[PartOf(args.f, args.count)];
  __shared__ uint32_t s_hist[kAllDigits];  // [pass][digit]
  __shared__ uint32_t s_misc[3];           // [0] status bits, [1] max scale, [2] valid occurrences
  __shared__ uint32_t s_off[kStageBags];   // offsets[b0 .. b0 + staged)
  __shared__ uint32_t s_probe[kProbes / kWave][2];
  if (blockIdx.x == 0) ClearControl(args.ctrl, kKeyBlock);
  for (uint64_t i = uint64_t(blockIdx.x) * kKeyBlock + threadIdx.x; i < args.zero_words;
       i += uint64_t(gridDim.x) * kKeyBlock)
    args.zero[i] = 0;
  const uint32_t all_digits = args.passes * args.digits;
  for (uint32_t i = threadIdx.x; i < all_digits; i += kKeyBlock) s_hist[i] = 0;
  if (threadIdx.x < 3) s_misc[threadIdx.x] = 0;

  const uint64_t local0 = uint64_t(blockIdx.x - f.block_begin) * kSortTile;
  uint32_t scale_max = 0;
  bool bad = false;
  // The thread's occurrences are independent: their slot loads, bag searches
  // and scale loads proceed interleaved, so each dependent step has all of
  // them in flight instead of one.
  uint64_t slot[kKeyItems];
  uint32_t lo[kKeyItems];  // bag of the occurrence: largest b < bags with offsets[b] <= li
  const uint32_t here = uint32_t(min<uint64_t>(kSortTile, f.occurrences - local0));  // occurrences of the tile
  auto item = [&](uint32_t k) { return k * kKeyBlock + threadIdx.x; };               // within the tile
#pragma unroll
  for (uint32_t k = 0; k < kKeyItems; ++k) {
    slot[k] = f.indices[local0 + min(item(k), here - 1)];
    lo[k] = 0;
  }
  if (f.pooling != EPS_HIP_POOL_SEQUENCE) {
    // Bag of each occurrence: the largest b < bags with offsets[b] <= li.
    // The block's occurrences are consecutive, so the block first finds a bag
    // b0 at most kSearchStep before that of its first occurrence and one past
    // that of its last (each round probes 128 evenly spaced offsets at once
    // and keeps the segment that the probes at or below the first point at:
    // one round for 32,768 bags), then stages the offsets between them in LDS,
    // where each occurrence is searched.  (1,024 probes a round: 4 x 8.4 M
    // occurrences in 262,144 bags each took 238 us against 184, a line read per
    // probe.)
    const uint64_t first = local0, last = min(local0 + kSortTile, f.occurrences) - 1;
    uint64_t b0 = 0, span = f.bags;  // answer in [b0, b0 + span); offsets[b0] <= first or b0 == 0
    uint64_t upper = f.bags;         // offsets[upper] > last, or bags
    while (span > kSearchStep) {
      const uint64_t step = (span + kProbes - 1) / kProbes;
      const uint64_t q = uint64_t(threadIdx.x) * step;
      const bool probing = threadIdx.x < kProbes && q < span;
      const uint64_t offset = probing ? f.offsets[b0 + q] : ~0ull;
      const uint64_t below = __ballot(offset <= first), inside = __ballot(offset <= last);
      __syncthreads();  // the round before has been read
      if ((threadIdx.x & (kWave - 1)) == 0 && threadIdx.x < kProbes) {
        s_probe[threadIdx.x / kWave][0] = uint32_t(__popcll(below));
        s_probe[threadIdx.x / kWave][1] = uint32_t(__popcll(inside));
      }
      __syncthreads();
      uint32_t count = 0, reach = 0;
#pragma unroll
      for (uint32_t w = 0; w < kProbes / kWave; ++w) {
        count += s_probe[w][0];
        reach += s_probe[w][1];
      }
      if (uint64_t(reach) * step < span) upper = b0 + uint64_t(reach) * step;
      const uint64_t keep = count ? count - 1 : 0;
      b0 += keep * step;
      span = min(step, span - keep * step);
    }
    const uint32_t staged = uint32_t(min<uint64_t>(kStageBags, max(upper, b0 + 1) + 1 - b0));
    // Offsets relative to the block's first occurrence (those before it are
    // 0, which orders them as well, those far past it the largest value).
    for (uint32_t i = threadIdx.x; i < staged; i += kKeyBlock) {
      const uint64_t o = f.offsets[b0 + i];
      s_off[i] = o <= first ? 0u : uint32_t(min<uint64_t>(o - first, 0xffffffffu));
    }
    __syncthreads();
    // Covered when the staged offsets reach past the block's last occurrence
    // (or reach offsets[bags], which is past every occurrence); else (runs of
    // empty bags longer than the stage) fall back to searching global memory.
    if (b0 + staged == f.bags + 1 || s_off[staged - 1] > last - first) {
      uint32_t r[kKeyItems];
#pragma unroll
      for (uint32_t k = 0; k < kKeyItems; ++k) r[k] = 0;
      // Answer in [0, staged - 1): offsets[b0 + staged - 1] > last unless it is offsets[bags].
      for (uint32_t len = staged - 1; len > 1;) {
        const uint32_t half = len >> 1;
#pragma unroll
        for (uint32_t k = 0; k < kKeyItems; ++k) r[k] = s_off[r[k] + half] <= item(k) ? r[k] + half : r[k];
        len -= half;
      }
#pragma unroll
      for (uint32_t k = 0; k < kKeyItems; ++k) lo[k] = uint32_t(b0) + r[k];
    } else {
      // Branch-free binary search with a trip count that is uniform over the
      // block: each step issues all of the thread's offset loads before it
      // waits on them.  The probe lo + half stays below lo + len <= bags.
      for (uint32_t len = uint32_t(f.bags); len > 1;) {
        const uint32_t half = len >> 1;
        uint64_t probe[kKeyItems];
#pragma unroll
        for (uint32_t k = 0; k < kKeyItems; ++k) probe[k] = f.offsets[lo[k] + half];
#pragma unroll
        for (uint32_t k = 0; k < kKeyItems; ++k) lo[k] = probe[k] <= local0 + item(k) ? lo[k] + half : lo[k];
        len -= half;
      }
    }
  } else {
    __syncthreads();
  }
  // Per-occurrence scale, loaded for all items before any is used (the pooling
  // mode is uniform over the block; indices are clamped into range).
  float scale[kKeyItems];
#pragma unroll
  for (uint32_t k = 0; k < kKeyItems; ++k) scale[k] = 1.0f;
  if (f.pooling == EPS_HIP_POOL_MEAN) {
    // A push without weighted sums sorts words without scales: the last pass
    // derives them, and 1 / length never exceeds 1.
    if (!args.refs) {
      uint64_t len[kKeyItems];
#pragma unroll
      for (uint32_t k = 0; k < kKeyItems; ++k) len[k] = f.lengths[lo[k]];
#pragma unroll
      for (uint32_t k = 0; k < kKeyItems; ++k)
        if (len[k]) scale[k] = 1.0f / (float)len[k];  // batch_access.cpp:79-80
    }
  } else if (f.pooling == EPS_HIP_POOL_WEIGHTED_SUM) {
#pragma unroll
    for (uint32_t k = 0; k < kKeyItems; ++k)
      scale[k] = f.weights[local0 + min(item(k), here - 1)];
  }
  uint32_t valid = 0;
#pragma unroll
  for (uint32_t k = 0; k < kKeyItems; ++k) {
    if (item(k) >= here) continue;
    uint64_t s = slot[k];
    if (s != kHole && s >= f.table_rows) { bad = true; s = kHole; }
    const uint32_t li = uint32_t(local0) + item(k), at = f.sort_begin + li;
    uint32_t key = args.sentinel;
    if (s != kHole) {
      key = (f.key_index << args.row_bits) | uint32_t(s);
      scale_max = max(scale_max, AbsBits(scale[k]));
      ++valid;
      for (uint32_t p = 0; p < args.passes; ++p)
        atomicAdd(&s_hist[p * args.digits + ((key >> args.shift[p]) & ((1u << args.bits[p]) - 1))], 1u);
    }
    const uint32_t row = f.pooling == EPS_HIP_POOL_SEQUENCE ? li : lo[k];
    args.keys[at] = key;
    if (args.vals) args.vals[at] = f.occ_begin + li;
    const uint32_t ref = (f.feature << kRefRowBits) | row;
    if (args.refs) args.refs[at] = ref;
    else args.refscale[at] = (uint64_t(__float_as_uint(scale[k])) << 32) | ref;
  }
  if (bad) s_misc[0] = EPS_HIP_STATUS_BAD_INDEX;
  // Only scales above 1.0 matter to the guard (it bounds with max(1, |scale|)),
  // so sum and mean pooling never reach the atomics below.
  scale_max = WaveMax(scale_max);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) valid += uint32_t(__shfl_xor(int(valid), o));
  if ((threadIdx.x & (kWave - 1)) == 0) {
    if (scale_max > 0x3f800000u) atomicMax(&s_misc[1], scale_max);
    atomicAdd(&s_misc[2], valid);
  }
  __syncthreads();
  // The tile's digit counts, two to a word (a tile has at most 4,096 of any;
  // digit counts are powers of two, at least 2).
  for (uint32_t i = threadIdx.x * 2; i < all_digits; i += kKeyBlock * 2) {
    const uint32_t p = i / args.digits, d = i - p * args.digits;
    uint32_t* to = reinterpret_cast<uint32_t*>(args.counts + (uint64_t(p) * args.tiles + blockIdx.x) * args.digits + d);
    *to = s_hist[i] | (s_hist[i + 1] << 16);
  }
  if (threadIdx.x == 0) args.info[blockIdx.x] = TileInfo{s_misc[2], s_misc[1], s_misc[0], 0u};
}

// Digit counts of each table over its keygen tiles: hist[table][pass][digit]
// (zeroed by keygen) from counts[pass][tile][digit].  A block adds up
// kSumTiles tiles of one table.
constexpr uint32_t kSumTiles = 64;
struct CountSumArgs {
  struct Part { uint32_t block_begin, tile_begin, tile_end, segment; } part[EPS_HIP_MAX_TABLES];
  uint32_t parts, passes, digits, tiles;
  const uint16_t* counts;
  uint32_t* hist;
};
__global__ void __launch_bounds__(kBlock) CountSumKernel(CountSumArgs a) {
  const auto& part = a.part[PartOf(a.part, a.parts)];
  const uint32_t first = part.tile_begin + (blockIdx.x - part.block_begin) * kSumTiles;
  const uint32_t n = min(kSumTiles, part.tile_end - first);
  for (uint32_t i = threadIdx.x; i < a.passes * a.digits; i += kBlock) {
    const uint32_t p = i / a.digits, d = i - p * a.digits;
    const uint16_t* c = a.counts + (uint64_t(p) * a.tiles + first) * a.digits + d;
    uint32_t sum = 0;
    for (uint32_t k = 0; k < n; k += 16) {
      uint32_t v[16];
#pragma unroll
      for (uint32_t q = 0; q < 16; ++q) v[q] = c[uint64_t(min(k + q, n - 1)) * a.digits];
#pragma unroll
      for (uint32_t q = 0; q < 16; ++q) sum += k + q < n ? v[q] : 0u;
    }
    if (sum) atomicAdd(&a.hist[(part.segment * a.passes + p) * a.digits + d], sum);
  }
}

// Exclusive scan of one value per thread over a 256-thread block.
__device__ __forceinline__ uint32_t BlockExclusiveScan(uint32_t x, uint32_t* s_wave) {
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  uint32_t inc = x;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(inc, o);
    if (lane >= uint32_t(o)) inc += y;
  }
  if (lane == kWave - 1) s_wave[wave] = inc;
  __syncthreads();
  uint32_t before = 0;
  for (uint32_t w = 0; w < wave; ++w) before += s_wave[w];
  __syncthreads();
  return before + inc - x;
}

// Inclusive scan over a wavefront with DPP moves: within rows of 16 lanes, then
// the last lane of row 0 (2) into row 1 (3), then lane 31 into rows 2 and 3.
__device__ __forceinline__ uint32_t WaveScan(uint32_t x) {
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x111, 0xf, 0xf, false));  // row_shr:1
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x112, 0xf, 0xf, false));  // row_shr:2
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x114, 0xf, 0xf, false));  // row_shr:4
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x118, 0xf, 0xf, false));  // row_shr:8
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x142, 0xa, 0xf, false));  // row_bcast:15, rows 1 and 3
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x143, 0xc, 0xf, false));  // row_bcast:31, rows 2 and 3
  return x;
}

// Exclusive scans of two values per thread over a sort block (one barrier).
__device__ __forceinline__ void SortScan2(uint32_t& x, uint32_t& y, uint32_t (*s_wave)[2]) {
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const uint32_t ix = WaveScan(x), iy = WaveScan(y);
  if (lane == kWave - 1) { s_wave[wave][0] = ix; s_wave[wave][1] = iy; }
  __syncthreads();
  uint32_t bx = 0, by = 0;
#pragma unroll
  for (uint32_t w = 0; w < kSortWaves; ++w)
    if (w < wave) { bx += s_wave[w][0]; by += s_wave[w][1]; }
  x = bx + ix - x;
  y = by + iy - y;
}

// Stable rank of each of a wavefront's items among the wavefront's earlier
// items of the same digit; s_count[digit] (this wavefront's row, zeroed) ends
// with the wavefront's digit counts.  Items are ranked i = 0, 1, ..., lanes in
// order within each.
// (`items`, uniform: later items are not ranked.)
__device__ __forceinline__ void RankDigits(const uint32_t (&digit)[kSortItems], const bool (&valid)[kSortItems],
                                           uint32_t bits, uint16_t* s_count, uint32_t (&rank)[kSortItems],
                                           uint32_t items = kSortItems) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint64_t lt_mask = (1ull << lane) - 1;
  // Lanes of the item's digit: per bit, the lanes whose bit is this lane's
  // (match & ~(ones ^ mine), one v_bitop3 a half).
  uint32_t lo[kSortItems], hi[kSortItems];
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    const uint64_t in = __ballot(valid[i]);
    lo[i] = uint32_t(in);
    hi[i] = uint32_t(in >> 32);
  }
  for (uint32_t b = 0; b < bits; ++b) {
#pragma unroll
    for (uint32_t i = 0; i < kSortItems; ++i) {
      if (i >= items) break;
      const uint32_t mine = uint32_t(__builtin_amdgcn_sbfe(digit[i], b, 1u));  // 0 or ~0
      const uint64_t ones = __ballot(mine != 0);
      lo[i] = __builtin_amdgcn_bitop3_b32(lo[i], uint32_t(ones), mine, 0x90);
      hi[i] = __builtin_amdgcn_bitop3_b32(hi[i], uint32_t(ones >> 32), mine, 0x90);
    }
  }
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    rank[i] = 0;
    if (i >= items) break;
    if (valid[i]) {
      const uint64_t match = lo[i] | (uint64_t(hi[i]) << 32);
      const uint32_t before = s_count[digit[i]];
      rank[i] = before + uint32_t(__popcll(match & lt_mask));
      if ((match & lt_mask) == 0) s_count[digit[i]] = uint16_t(before + uint32_t(__popcll(match)));
    }
    // The next item reads what this one wrote (one wavefront: LDS accesses
    // are performed in order, only the compiler has to keep them so).
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  }
}

// kVals: the occurrence indices travel with the keys (for eps_hip_unique and
// eps_hip_reduce, which map sorted positions back to occurrences); a push
// needs only the keys and reference words.  kWords: the reference words are
// 8 bytes with their scales (kWide), 4 bytes without (kNarrow), or 4 bytes
// in and 8 bytes out (kWiden, the last pass of a sort of 4-byte words, which
// puts each word's scale back from ScaleArgs).
enum WordForm : int { kWide = 0, kNarrow = 1, kWiden = 2 };
template <int kWords> struct WordTypes;
template <> struct WordTypes<kWide> { typedef uint64_t In; typedef uint64_t Out; };
template <> struct WordTypes<kNarrow> { typedef uint32_t In; typedef uint32_t Out; };
template <> struct WordTypes<kWiden> { typedef uint32_t In; typedef uint64_t Out; };

// A pass's tiles.  Spans of the first pass are features (its tiles are
// keygen's), of the later ones tables; `begin` and `count` are elements of the
// sort's arrays (the later passes: room for every occurrence, of which the
// table's valid ones come first).
struct SortSpan { uint32_t begin, count, segment; };
constexpr uint32_t kMaxSpans =
    EPS_HIP_MAX_TABLES > EPS_HIP_MAX_FEATURES ? EPS_HIP_MAX_TABLES : EPS_HIP_MAX_FEATURES;
struct SortArgs {
  uint32_t span_tile[kMaxSpans];  // first tile of each span (~0 past the last)
  SortSpan span[kMaxSpans];
  // Per segment (a table with occurrences, by key index): first element,
  // first keygen tile (and the ends), key index.
  uint32_t seg_begin[EPS_HIP_MAX_TABLES], seg_tile[EPS_HIP_MAX_TABLES + 1], seg_key[EPS_HIP_MAX_TABLES];
  uint32_t segments, shift, bits, digits, pass, passes, count_tiles, sentinel;
  uint32_t direct;  // counts are added up by the block (no CountSumKernel ran)
  uint32_t class_key[kClasses + 1];  // first table key index of each class (+ table count)
  const uint16_t* counts;
  const uint32_t* hist;
  const TileInfo* info;
  uint32_t* look;
  uint32_t* group_look;
  Control* ctrl;
  const uint32_t* keys_in;
  const uint32_t* vals_in;
  uint32_t* keys_out;
  uint32_t* vals_out;
  const void* rs_in;
  void* rs_out;
};

// (Two blocks a CU: 64 registers.)
template <bool kVals, int kWords>
__global__ void __launch_bounds__(kSortBlock) __attribute__((amdgpu_waves_per_eu(8))) RadixPassKernel(SortArgs a, ScaleArgs sc) {
  typedef typename WordTypes<kWords>::In InWord;
  typedef typename WordTypes<kWords>::Out OutWord;
  const InWord* rs_in = static_cast<const InWord*>(a.rs_in);
  OutWord* rs_out = static_cast<OutWord*>(a.rs_out);
  // The wavefronts' digit counts, then (after the ranks are final) the tile in
  // digit order.
  struct Sorted { uint32_t keys[kSortTile], vals[kVals ? kSortTile : 1]; InWord rs[kSortTile]; };
  __shared__ union { uint16_t count[kSortWaves][kDigits]; Sorted sorted; } sh;
  __shared__ uint32_t s_tile_start[kDigits], s_global[kDigits];
  __shared__ uint32_t s_wave[kSortWaves][2], s_sum[2];
  __shared__ uint32_t s_tile;

  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  const bool first_pass = a.pass == 0, last_pass = a.pass + 1 == a.passes;
  // Tiles that wait on earlier ones are claimed in order, so that what a tile
  // waits on has started; the first pass of a small sort waits on nothing.
  const bool looks = !(first_pass && a.direct);
  if (t == 0) s_tile = looks ? atomicAdd(&a.ctrl->tile_counter[a.pass], 1u) : blockIdx.x;
  if (t < 2) s_sum[t] = 0;
  for (uint32_t d = lane * 2; d < a.digits; d += kWave * 2) *reinterpret_cast<uint32_t*>(&sh.count[wave][d]) = 0;
  __syncthreads();
  const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);
  uint32_t part = 0;
#pragma unroll
  for (uint32_t k = 1; k < kMaxSpans; ++k) part += tile >= a.span_tile[k] ? 1u : 0u;
  const SortSpan span = a.span[part];
  const uint32_t seg = span.segment, local = tile - a.span_tile[part];
  const uint32_t begin = span.begin + local * kSortTile;
  const uint32_t room = min(kSortTile, span.count - local * kSortTile);
  const uint32_t base = wave * (kSortTile / kSortWaves) + lane;
  uint32_t key[kSortItems], val[kSortItems], digit[kSortItems], rank[kSortItems];
  InWord rs[kSortItems];
  bool valid[kSortItems];
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    const uint32_t q = base + i * kWave;
    valid[i] = q < room;
    const uint32_t p = begin + (valid[i] ? q : 0u);
    key[i] = a.keys_in[p];
    val[i] = kVals ? a.vals_in[p] : 0u;
    rs[i] = rs_in[p];
  }
  // Valid occurrences of this segment and of the segments before it.
  const uint32_t seg_first = a.seg_tile[seg], seg_last = a.seg_tile[seg + 1];
  if (!first_pass || last_pass) {
    uint32_t before = 0, mine = 0;
    const uint32_t from = last_pass ? 0u : seg_first;
    for (uint32_t i = from + t; i < seg_last; i += kSortBlock) {
      const uint32_t v = a.info[i].valid;
      if (i < seg_first) before += v; else mine += v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      before += uint32_t(__shfl_xor(int(before), o));
      mine += uint32_t(__shfl_xor(int(mine), o));
    }
    if (lane == 0) {
      if (before) atomicAdd(&s_sum[0], before);
      if (mine) atomicAdd(&s_sum[1], mine);
    }
  }
  // Digit counts of the whole segment, and (first pass of a small sort) of
  // its tiles before this one: thread t has digit t.
  uint32_t digit_count = 0, exclusive = 0;
  if (t < a.digits) {
    if (a.direct) {
      const uint16_t* c = a.counts + (uint64_t(a.pass) * a.count_tiles + seg_first) * a.digits + t;
      const uint32_t n = seg_last - seg_first, mine = tile - seg_first;
      for (uint32_t k = 0; k < n; k += 8) {
        uint32_t v[8];
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) v[q] = c[min(k + q, n - 1) * a.digits];
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) {
          const uint32_t x = k + q < n ? v[q] : 0u;
          digit_count += x;
          if (first_pass && k + q < mine) exclusive += x;
        }
      }
    } else {
      digit_count = a.hist[(seg * a.passes + a.pass) * a.digits + t];
    }
  }
  __syncthreads();
  // Valid elements of the tile: the first pass drops the sentinels, the later
  // ones end with the segment's valid occurrences.
  const uint32_t seg_valid = s_sum[1];
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    if (first_pass) valid[i] = valid[i] && key[i] != a.sentinel;
    else valid[i] = local * kSortTile + base + i * kWave < seg_valid;
    digit[i] = (key[i] >> a.shift) & ((1u << a.bits) - 1);
  }
  RankDigits(digit, valid, a.bits, sh.count[wave], rank);
  __syncthreads();
  // Per digit: wave prefixes and tile total.
  uint32_t total = 0;
  if (t < a.digits) {
#pragma unroll
    for (uint32_t w = 0; w < kSortWaves; ++w) {
      const uint32_t c = sh.count[w][t];
      sh.count[w][t] = uint16_t(total);
      total += c;
    }
  }
  if (looks && t < a.digits) {
    // Two-level look-back over the segment's tiles.  Tiles form groups of
    // kGroupTiles; every tile publishes its digit counts.  A tile's exclusive
    // prefix is the counts of the tiles before it in its group plus the
    // prefix of the segment's groups before its group.  The group's last tile
    // publishes the group total, then (after its own walk) the group's
    // inclusive prefix.  The walk over groups is windowed and stops at the
    // first inclusive prefix, as a tile-level look-back would, but the chain
    // runs through groups, not tiles.  A tile waits only on tiles claimed
    // before it (the tile counter hands tiles out in order), so the waits
    // always end.
    const uint32_t at = first_pass ? tile - seg_first : local;  // tile within its segment
    const uint32_t row0 = tile - at;                            // the segment's first tile
    const uint32_t in_seg = first_pass ? seg_last - seg_first : (span.count + kSortTile - 1) / kSortTile;
    const uint32_t group = at / kGroupTiles, first = group * kGroupTiles;
    const bool leader = at + 1 == min(first + kGroupTiles, in_seg);
    __hip_atomic_store(a.look + uint64_t(tile) * a.digits + t, kFlagAggregate | total, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    // Counts of the tiles before this one in its group (all published or about to be).
    uint32_t within = 0;
    for (uint32_t half = 0; half < at - first; half += kLookWindow) {
      const uint32_t* row = a.look + uint64_t(row0 + first + half) * a.digits + t;
      uint32_t missing = (1u << min(at - first - half, kLookWindow)) - 1;  // bit w: tile w of the half still to add
      while (missing) {
        uint32_t v[kLookWindow];
#pragma unroll
        for (uint32_t w = 0; w < kLookWindow; ++w)
          v[w] = (missing >> w) & 1u ? __hip_atomic_load(row + w * a.digits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                     : 0u;
#pragma unroll
        for (uint32_t w = 0; w < kLookWindow; ++w) {
          if (!((missing >> w) & 1u) || !(v[w] & ~kValueMask)) continue;
          within += v[w] & kValueMask;
          missing &= ~(1u << w);
        }
      }
    }
    // The segment's group rows follow those of the segments before it, which
    // have at most one group per started 16 tiles each.
    uint32_t* groups = a.group_look + uint64_t(row0 / kGroupTiles + seg) * a.digits + t;
    uint32_t* group_mine = groups + uint64_t(group) * a.digits;
    if (leader)
      __hip_atomic_store(group_mine, (group == 0 ? kFlagInclusive : kFlagAggregate) | (within + total),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // Windowed walk over the groups before this one: each round reads the next
    // kLookWindow predecessors at once and adds their counts, nearest first,
    // up to the first inclusive prefix (done) or the first group that has not
    // published yet (read again from there).  Group 0 always publishes an
    // inclusive prefix, so the walk ends at or before it; reads before group 0
    // are never issued.
    int64_t next = int64_t(group) - 1;
    bool done = group == 0;
    while (!done) {
      uint32_t v[kLookWindow];
#pragma unroll
      for (uint32_t w = 0; w < kLookWindow; ++w) {
        const int64_t q = next - int64_t(w);
        v[w] = q >= 0 ? __hip_atomic_load(groups + uint64_t(q) * a.digits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                      : kFlagInclusive;
      }
      bool stop = false;
      uint32_t taken = 0;
#pragma unroll
      for (uint32_t w = 0; w < kLookWindow; ++w) {
        const uint32_t flag = v[w] & ~kValueMask;
        if (!stop) {
          if (flag == 0) {
            stop = true;  // not published yet
          } else {
            exclusive += v[w] & kValueMask;
            ++taken;
            if (flag == kFlagInclusive) stop = done = true;
          }
        }
      }
      next -= int64_t(taken);
    }
    if (leader && group != 0)
      __hip_atomic_store(group_mine, kFlagInclusive | (exclusive + within + total), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    exclusive += within;
  }
  // Exclusive scans in digit order.  Elements go to the segment's own room, in
  // the last pass to where the valid occurrences of the segments before it end.
  uint32_t digit_base = digit_count, tile_start = total;
  SortScan2(digit_base, tile_start, s_wave);
  if (t < a.digits) {
    s_tile_start[t] = tile_start;
    s_global[t] = (last_pass ? s_sum[0] : a.seg_begin[seg]) + digit_base + exclusive - tile_start;
  }
  __syncthreads();
  uint32_t place[kSortItems];
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i)
    if (valid[i]) place[i] = s_tile_start[digit[i]] + sh.count[wave][digit[i]] + rank[i];
  __syncthreads();  // the counts make room for the sorted tile
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    if (!valid[i]) continue;
    sh.sorted.keys[place[i]] = key[i];
    if (kVals) sh.sorted.vals[place[i]] = val[i];
    sh.sorted.rs[place[i]] = rs[i];
  }
  // The tile's valid elements: the scan's end.
  uint32_t tile_n = 0;
#pragma unroll
  for (uint32_t w = 0; w < kSortWaves; ++w) tile_n += s_wave[w][1];
  __syncthreads();
  // Scatter of the digit-sorted tile: all LDS reads, then the stores.  The
  // reference words travel with their keys through every pass, so the last
  // pass needs no gather by occurrence index.  Entries past the tile's end
  // read stale LDS (in bounds) and are not stored.
  uint32_t dest[kSortItems];
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    const uint32_t q = i * kSortBlock + t;
    key[i] = sh.sorted.keys[q];
    if (kVals) val[i] = sh.sorted.vals[q];
    rs[i] = sh.sorted.rs[q];
    dest[i] = s_global[(key[i] >> a.shift) & ((1u << a.bits) - 1)] + q;
  }
  uint64_t len[kSortItems];
  if (kWords == kWiden) {
    // Each word's scale: the valid length of a mean feature's bag (all
    // loaded before any is used), as keygen computed it.
#pragma unroll
    for (uint32_t i = 0; i < kSortItems; ++i) {
      const uint32_t feature = uint32_t(rs[i]) >> kRefRowBits;
      const bool mean = i * kSortBlock + t < tile_n && ((sc.mean_mask >> feature) & 1u);
      len[i] = mean ? sc.lengths[feature][uint32_t(rs[i]) & ((1u << kRefRowBits) - 1u)] : 0ull;
    }
  }
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    if (i * kSortBlock + t >= tile_n) continue;
    a.keys_out[dest[i]] = key[i];
    if (kVals) a.vals_out[dest[i]] = val[i];
    if (kWords == kWiden) {
      const float scale = len[i] ? 1.0f / (float)len[i] : 1.0f;  // batch_access.cpp:79-80
      rs_out[dest[i]] = OutWord((uint64_t(__float_as_uint(scale)) << 32) | uint32_t(rs[i]));
    } else {
      rs_out[dest[i]] = OutWord(rs[i]);
    }
  }
  // One block of the last pass writes what the tiles found: the class
  // boundaries (first sorted position of each class, the valid count last),
  // the prepare-time findings and the largest scale.
  if (last_pass && tile == 0) {
    __shared__ uint32_t s_class[kClasses], s_found[2], s_seg_tile[EPS_HIP_MAX_TABLES], s_seg_class[EPS_HIP_MAX_TABLES];
    if (t < kClasses) s_class[t] = 0;
    if (t < a.segments) {
      s_seg_tile[t] = a.seg_tile[t + 1];
      uint32_t c = 0;
#pragma unroll
      for (uint32_t k = 1; k < kClasses; ++k) c += a.seg_key[t] >= a.class_key[k];
      s_seg_class[t] = c;
    }
    if (t < 2) s_found[t] = 0;
    __syncthreads();
    uint32_t scale = 0, status = 0;
    for (uint32_t i = t; i < a.count_tiles; i += kSortBlock) {
      const TileInfo x = a.info[i];
      scale = max(scale, x.scale);
      status |= x.status;
      uint32_t s = 0;
      while (s + 1 < a.segments && i >= s_seg_tile[s]) ++s;
      if (x.valid) atomicAdd(&s_class[s_seg_class[s]], x.valid);
    }
    if (scale) atomicMax(&s_found[0], scale);
    if (status) atomicOr(&s_found[1], status);
    __syncthreads();
    if (t <= kClasses) {
      uint32_t start = 0;
      for (uint32_t c = 0; c < t; ++c) start += s_class[c];
      a.ctrl->class_start[t] = start;
      if (t == kClasses) a.ctrl->valid_count = start;
    }
    if (t == 0) {
      if (s_found[0]) a.ctrl->scale_slots[0] = s_found[0];
      if (s_found[1]) a.ctrl->prep_status = s_found[1];
    }
  }
}

// ---- first-occurrence ranking ----
__global__ void HeadFlagKernel(const uint32_t* keys, const uint32_t* vals, const Control* ctrl,
                               uint32_t* flags, uint32_t n) {
  const uint32_t valid = ctrl->valid_count;
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n && p < valid;
       p += blockDim.x * gridDim.x)
    if (p == 0 || keys[p] != keys[p - 1]) flags[vals[p]] = 1;
}

__global__ void ScanBlockSumsKernel(const uint32_t* flags, uint32_t* block_sums, uint32_t n) {
  __shared__ uint32_t s_wave[4];
  const uint32_t b = blockIdx.x;
  uint32_t sum = 0;
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t i = b * 1024 + k * kBlock + threadIdx.x;
    if (i < n) sum += flags[i];
  }
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane == 0) s_wave[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) block_sums[b] = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
}

__global__ void ScanTopKernel(uint32_t* block_sums, uint32_t blocks, Control* ctrl,
                              uint64_t* unique_count) {
  __shared__ uint32_t s_scan[4];
  __shared__ uint32_t s_carry;
  if (threadIdx.x == 0) s_carry = 0;
  __syncthreads();
  for (uint32_t start = 0; start < blocks; start += kBlock) {
    const uint32_t i = start + threadIdx.x;
    const uint32_t x = i < blocks ? block_sums[i] : 0;
    const uint32_t ex = BlockExclusiveScan(x, s_scan);
    const uint32_t carry = s_carry;
    if (i < blocks) block_sums[i] = carry + ex;
    __syncthreads();
    if (threadIdx.x == kBlock - 1) s_carry = carry + ex + x;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    ctrl->unique_count = s_carry;
    if (unique_count) *unique_count = s_carry;
  }
}

__global__ void ScanApplyKernel(const uint32_t* flags, const uint32_t* block_sums, uint32_t* ranks,
                                uint32_t n) {
  __shared__ uint32_t s_scan[4];
  __shared__ uint32_t s_carry;
  const uint32_t b = blockIdx.x;
  if (threadIdx.x == 0) s_carry = block_sums[b];
  __syncthreads();
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t i = b * 1024 + k * kBlock + threadIdx.x;
    const uint32_t x = i < n ? flags[i] : 0;
    const uint32_t ex = BlockExclusiveScan(x, s_scan);
    const uint32_t carry = s_carry;
    if (i < n) ranks[i] = carry + ex;
    __syncthreads();
    if (threadIdx.x == kBlock - 1) s_carry = carry + ex + x;
    __syncthreads();
  }
}

// ---- hot rows: segments of more than kLongRefs references ----
// Keys are sorted, so a segment that starts at p has more than kLongRefs
// references exactly when keys[p + kLongRefs] == keys[p]: one test per
// position, no scan.  Only vector dimension classes are listed (the generic
// class keeps its own kernel).  The list order is irrelevant: rows are
// independent.
struct HotArgs {
  const uint32_t* keys;
  HotEntry* hot;
  Control* ctrl;
  uint32_t n, capacity;
  uint32_t generic_key;  // first key of the generic class (its tables come last; ~0: none)
};

// The row whose first position p of `keys` is hot (its positions and key) goes
// to one of the lists of the XCD that owns that eighth of the push's n
// positions (the update kernels split their work the same way); its length
// picks the list (eight ranges, from 65,536 or more references down), so the
// hot-row kernel can deal the longest rows out first.
__device__ __forceinline__ void ListHotRow(const HotArgs& a, uint32_t p, uint32_t end, uint32_t key) {
  const uint32_t refs = end - p;
  // Lists by length, longest first: >= 65536, 16384, 4096, 2048, 1024, 512, 256, fewer.
  const uint32_t bucket = refs >= 65536 ? 0u : refs >= 16384 ? 1u : refs >= 4096 ? 2u : refs >= 2048 ? 3u :
                          refs >= 1024 ? 4u : refs >= 512 ? 5u : refs >= 256 ? 6u : 7u;
  const uint32_t list = uint32_t(uint64_t(p) * kXcds / a.n) * kHotBuckets + bucket;
  // Sorted keys give each hot row one first position, so a list never holds
  // more than n / 129 entries; the bound keeps the write inside the list
  // whatever the keys (the readers clamp the counts to the capacity too).
  const uint32_t at = atomicAdd(&a.ctrl->long_count[list], 1u);
  if (at < a.capacity) a.hot[uint64_t(list) * a.capacity + at] = HotEntry{p, end, key, 0u};
}

// Lists the hot rows that start at `start` (~0: none) of a wavefront's lanes,
// one after another, the wavefront searching each row's end together: each
// round probes 64 positions, the first one at a stride of 64, then strides
// that grow by 64 until a probe misses, then back down to single positions.
__device__ __forceinline__ void ListHotRows(const HotArgs& a, const uint32_t* keys, uint32_t valid, uint32_t start,
                                            uint32_t row_key) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  for (uint64_t todo = __ballot(start != ~0u); todo; todo &= todo - 1) {
    const uint32_t owner = uint32_t(__ffsll((unsigned long long)todo) - 1);
    const uint32_t p = __shfl(start, int(owner)), key = __shfl(row_key, int(owner));
    // keys[at] == key; the end lies in (at, valid].
    uint32_t at = p + kLongRefs, stride = kWave;
    bool missed = false;  // a probe at `stride` missed: the end is within 64 strides
    for (;;) {
      const uint64_t q = uint64_t(at) + uint64_t(lane + 1) * stride;
      const bool hit = q < valid && keys[q < valid ? q : at] == key;
      const uint32_t hits = uint32_t(__popcll(__ballot(hit)));  // hits come first: the row is one run
      at += hits * stride;
      missed = missed || hits < kWave;
      if (!missed) { if (stride < (1u << 24)) stride *= kWave; continue; }
      if (stride == 1) break;
      stride /= kWave;
    }
    if (lane == owner) ListHotRow(a, p, at + 1, key);
  }
}

// Four sorted positions a thread, their keys and the keys kLongRefs further on
// in one 16-byte load each.
constexpr uint32_t kHotItems = 4;
__global__ void __launch_bounds__(kBlock) HotListKernel(HotArgs a) {
  const uint32_t valid = min(a.ctrl->valid_count, a.n);
  const uint32_t p = (blockIdx.x * kBlock + threadIdx.x) * kHotItems;
  if (blockIdx.x * kBlock * kHotItems + kLongRefs >= valid) return;  // uniform over the block
  typedef uint32_t U4 __attribute__((ext_vector_type(4)));
  // p is a multiple of four and the key buffers are 256-byte aligned; the last
  // quad may reach past the valid keys, not past its buffer's padding.
  const U4 mine = *reinterpret_cast<const U4*>(a.keys + (p < valid ? p : 0u));
  U4 ahead;
  if (p + kLongRefs + kHotItems <= valid) {
    ahead = *reinterpret_cast<const U4*>(a.keys + p + kLongRefs);
  } else {
#pragma unroll
    for (uint32_t k = 0; k < kHotItems; ++k) ahead[k] = a.keys[min(p + kLongRefs + k, valid - 1)];
  }
  const uint32_t before = p && p < valid ? a.keys[p - 1] : ~mine[0];
  // At most one of a thread's positions starts a hot row (they are longer
  // than a quad).
  uint32_t start = ~0u, row_key = 0;
#pragma unroll
  for (uint32_t k = 0; k < kHotItems; ++k) {
    const uint32_t key = mine[k], prev = k ? mine[k - 1] : before, at = p + k;
    if (key == prev || key >= a.generic_key || at + kLongRefs >= valid || ahead[k] != key) continue;
    start = at;
    row_key = key;
  }
  ListHotRows(a, a.keys, valid, start, row_key);
}

// ---- a small push, prepared by one block ----
struct SmallFeature {
  const uint64_t* indices;
  const uint64_t* offsets;
  const uint64_t* lengths;
  const float* weights;
  uint64_t table_rows;
  uint32_t occ_begin, bags, off_begin, key_index, pooling, reserved;
};
struct SmallArgs {
  SmallFeature f[EPS_HIP_MAX_FEATURES];
  uint32_t count, n, row_bits, sentinel, passes, shift[kMaxPasses], bits[kMaxPasses];
  uint32_t class_key[kClasses + 1];
  uint32_t* keys;
  uint32_t* vals;  // NULL: not wanted
  uint64_t* rs;
  HotArgs hot;
};
static_assert(sizeof(SmallArgs) <= 4096, "small prepare arguments fit the kernel-argument segment");

// Keys, reference words and hot rows of a push of up to kSmallOccurrences
// occurrences, sorted in LDS by whole keys (equal keys stay in occurrence
// order; the sentinel sorts last).  What bounds it is latency, so it is one
// launch: key generation, each radix pass and the hot-row list as launches of
// their own took 30 us and the gaps between six launches for 256 occurrences
// of two tables, this 13 us.
__global__ void __launch_bounds__(kSortBlock) SmallPrepareKernel(SmallArgs a) {
  __shared__ uint16_t s_count[kSortWaves][kDigits];
  __shared__ uint64_t s_word[kSmallOccurrences];
  __shared__ uint32_t s_key[kSmallOccurrences];
  __shared__ uint16_t s_occ[kSmallOccurrences];
  __shared__ uint32_t s_off[kSmallOffsets];  // the pooled features' offsets, one feature after another
  __shared__ uint32_t s_start[kDigits], s_wave[kSortWaves][2];
  __shared__ SmallFeature s_f[EPS_HIP_MAX_FEATURES];
  __shared__ uint32_t s_found[2], s_valid;
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  for (uint32_t i = t; i < a.count * sizeof(SmallFeature) / 4; i += kSortBlock)
    reinterpret_cast<uint32_t*>(s_f)[i] = reinterpret_cast<const uint32_t*>(a.f)[i];
  ClearControl(a.hot.ctrl, kSortBlock);
  if (t < 2) s_found[t] = 0;
  if (t == 0) s_valid = 0;
  __syncthreads();
  // Each wavefront has `items` times 64 occurrences, as few as hold the push;
  // item i of a thread is number 64 * i + lane of its wavefront's, so that
  // ranks in (wavefront, item, lane) order are ranks in occurrence order.
  const uint32_t items = (a.n + kSortBlock - 1) / kSortBlock;
  auto place = [&](uint32_t i) { return (wave * items + i) * kWave + lane; };
  uint32_t key[kSortItems], occ[kSortItems];
  uint64_t slot[kSortItems];
  uint32_t feat[kSortItems], li[kSortItems];
  bool in[kSortItems];
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    occ[i] = place(i);
    in[i] = i < items && occ[i] < a.n;
    feat[i] = 0;
    for (uint32_t f = 1; f < a.count; ++f) feat[i] += occ[i] >= s_f[f].occ_begin ? 1u : 0u;
    li[i] = occ[i] - s_f[feat[i]].occ_begin;
    slot[i] = in[i] ? s_f[feat[i]].indices[li[i]] : kHole;
  }
  for (uint32_t f = 0; f < a.count; ++f) {
    if (s_f[f].pooling == EPS_HIP_POOL_SEQUENCE) continue;
    for (uint32_t b = t; b <= s_f[f].bags; b += kSortBlock)
      s_off[s_f[f].off_begin + b] = uint32_t(min<uint64_t>(s_f[f].offsets[b], 0xffffffffu));
  }
  __syncthreads();
  uint32_t scale_max = 0, valid = 0;
  bool bad = false;
  float scale[kSortItems];
  uint32_t row[kSortItems];
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    const SmallFeature& f = s_f[feat[i]];
    scale[i] = 1.0f;
    row[i] = li[i];
    if (!in[i] || f.pooling == EPS_HIP_POOL_SEQUENCE) continue;
    uint32_t lo = 0;  // bag: the largest b < bags with offsets[b] <= li
    for (uint32_t len = f.bags; len > 1;) {
      const uint32_t half = len >> 1;
      lo = s_off[f.off_begin + lo + half] <= li[i] ? lo + half : lo;
      len -= half;
    }
    row[i] = lo;
    if (f.pooling == EPS_HIP_POOL_MEAN) {
      const uint64_t len = f.lengths[lo];
      if (len) scale[i] = 1.0f / (float)len;  // batch_access.cpp:79-80
    } else if (f.pooling == EPS_HIP_POOL_WEIGHTED_SUM) {
      scale[i] = f.weights[li[i]];
    }
  }
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    key[i] = a.sentinel;
    if (!in[i]) continue;
    const SmallFeature& f = s_f[feat[i]];
    uint64_t s = slot[i];
    if (s != kHole && s >= f.table_rows) { bad = true; s = kHole; }
    if (s != kHole) {
      key[i] = (f.key_index << a.row_bits) | uint32_t(s);
      scale_max = max(scale_max, AbsBits(scale[i]));
      ++valid;
    }
    s_word[occ[i]] = (uint64_t(__float_as_uint(scale[i])) << 32) | (feat[i] << kRefRowBits) | row[i];
  }
  if (bad) s_found[1] = EPS_HIP_STATUS_BAD_INDEX;
  if (scale_max > 0x3f800000u) atomicMax(&s_found[0], scale_max);
  if (valid) atomicAdd(&s_valid, valid);
  for (uint32_t p = 0; p < a.passes; ++p) {
    const uint32_t digits = 1u << a.bits[p];
    for (uint32_t i = lane; i < digits; i += kWave) s_count[wave][i] = 0;
    uint32_t digit[kSortItems], rank[kSortItems];
#pragma unroll
    for (uint32_t i = 0; i < kSortItems; ++i) digit[i] = (key[i] >> a.shift[p]) & (digits - 1);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    RankDigits(digit, in, a.bits[p], s_count[wave], rank, items);
    __syncthreads();
    uint32_t total = 0, none = 0;
    if (t < digits) {
#pragma unroll
      for (uint32_t w = 0; w < kSortWaves; ++w) {
        const uint32_t c = s_count[w][t];
        s_count[w][t] = uint16_t(total);
        total += c;
      }
    }
    SortScan2(total, none, s_wave);
    if (t < digits) s_start[t] = total;
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kSortItems; ++i) {
      if (!in[i]) continue;
      const uint32_t at = s_start[digit[i]] + s_count[wave][digit[i]] + rank[i];
      s_key[at] = key[i];
      s_occ[at] = uint16_t(occ[i]);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kSortItems; ++i) {
      const uint32_t q = place(i);
      if (!in[i]) continue;  // the elements stay the first n
      key[i] = s_key[q];
      occ[i] = s_occ[q];
    }
  }
  const uint32_t n = s_valid;  // valid occurrences: the first n of the sorted ones
#pragma unroll
  for (uint32_t i = 0; i < kSortItems; ++i) {
    const uint32_t q = place(i);
    if (!in[i]) continue;
    a.keys[q] = key[i];
    if (a.vals) a.vals[q] = occ[i];
    a.rs[q] = s_word[occ[i]];
  }
  // Hot rows, as HotListKernel finds them.
  if (n > kLongRefs) {
#pragma unroll
    for (uint32_t i = 0; i < kSortItems; ++i) {
      const uint32_t q = place(i);
      const bool hot = in[i] && q + kLongRefs < n && key[i] < a.hot.generic_key && s_key[q + kLongRefs] == key[i] &&
                       (q == 0 || s_key[q - 1] != key[i]);
      ListHotRows(a.hot, s_key, n, hot ? q : ~0u, key[i]);
    }
  }
  // Class boundaries: the first position of a key at or past the class's first.
  if (t <= kClasses) {
    uint32_t lo = 0, hi = n;
    const uint64_t from = uint64_t(a.class_key[t]) << a.row_bits;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) / 2;
      if (s_key[mid] < from) lo = mid + 1; else hi = mid;
    }
    if (t == kClasses) lo = n;
    a.hot.ctrl->class_start[t] = lo;
    if (t == kClasses) a.hot.ctrl->valid_count = n;
  }
  if (t == 0) {
    if (s_found[0]) a.hot.ctrl->scale_slots[0] = s_found[0];
    if (s_found[1]) a.hot.ctrl->prep_status = s_found[1];
  }
}

struct UniqueArgs {
  uint32_t table_of_key[EPS_HIP_MAX_TABLES];
};

__global__ void UniqueWriteKernel(const uint32_t* keys, const uint32_t* vals, const uint32_t* ranks,
                                  const Control* ctrl, uint32_t n, uint32_t row_bits,
                                  UniqueArgs args, uint64_t* unique_slots, uint32_t* unique_tables,
                                  uint64_t* occurrence_to_unique) {
  const uint32_t valid = ctrl->valid_count;
  __shared__ uint32_t s_table[EPS_HIP_MAX_TABLES];
#pragma unroll
  for (uint32_t i = 0; i < EPS_HIP_MAX_TABLES; ++i)
    if (threadIdx.x == i) s_table[i] = args.table_of_key[i];
  __syncthreads();
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n && p < valid;
       p += blockDim.x * gridDim.x) {
    const uint32_t key = keys[p];
    uint32_t lo = 0, hi = p;  // first index with this key (lower bound) in [lo, hi]
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (keys[mid] < key) lo = mid + 1; else hi = mid;
    }
    const uint32_t u = ranks[vals[lo]];
    occurrence_to_unique[vals[p]] = u;
    if (lo == p) {
      unique_slots[u] = key & ((1u << row_bits) - 1);
      unique_tables[u] = s_table[key >> row_bits];
    }
  }
}

unsigned Grid(uint64_t n, unsigned cap) {
  const uint64_t b = (n + kBlock - 1) / kBlock;
  return unsigned(std::max<uint64_t>(1, std::min<uint64_t>(b, cap)));
}

uint32_t BitLength(uint64_t x) {
  uint32_t b = 0;
  while (x) { ++b; x >>= 1; }
  return b;
}

}  // namespace

int PlanPush(const eps_hip_table* tables, uint32_t table_count,
             const eps_hip_push_feature* features, uint32_t feature_count, PushPlan& plan) {
  if (!tables || table_count == 0 || table_count > EPS_HIP_MAX_TABLES)
    return Fail(EPS_HIP_INVALID_ARGUMENT, "push needs 1..32 tables");
  if (!features || feature_count == 0 || feature_count > EPS_HIP_MAX_FEATURES)
    return Fail(EPS_HIP_INVALID_ARGUMENT, "push needs 1..32 features");
  uint64_t max_rows = 1;
  for (uint32_t t = 0; t < table_count; ++t) {
    if (!tables[t].state || tables[t].dim == 0 || tables[t].dim > 65536)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid push table");
    if (reinterpret_cast<uintptr_t>(tables[t].state) % 16)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "table state must be 16-byte aligned");
    max_rows = std::max<uint64_t>(max_rows, tables[t].rows);
  }
  plan.row_bits = std::max<uint32_t>(1, BitLength(max_rows - 1));
  // Table key indices ordered by dimension class, so each class is one
  // contiguous range of the sorted keys (tables of a class in call order).
  uint32_t keyed = 0;
  for (uint32_t c = 0; c < kClasses; ++c)
    for (uint32_t t = 0; t < table_count; ++t)
      if (DimClass(tables[t].dim) == c) plan.table_of_key[keyed++] = t;
  for (uint32_t i = 0; i < table_count; ++i) plan.key_index[plan.table_of_key[i]] = i;
  const auto& order = plan.table_of_key;
  for (uint32_t c = 0; c <= kClasses; ++c) {
    uint32_t k = 0;
    while (k < table_count && DimClass(tables[order[k]].dim) < c) ++k;
    plan.class_start[c] = k;
  }
  const uint64_t max_valid = (uint64_t(table_count - 1) << plan.row_bits) | (max_rows - 1);
  plan.key_bits = BitLength(max_valid + 1);
  if (plan.key_bits > 32) return Fail(EPS_HIP_CAPACITY_EXCEEDED, "table rows exceed 32-bit sort keys");
  plan.occurrences = 0;
  uint64_t staged = 0;  // bag offsets a one-block preparation would stage
  plan.class_occurrences.fill(0);
  for (uint32_t i = 0; i < feature_count; ++i) {
    const auto& f = features[i];
    if (f.table >= table_count || f.pooling > EPS_HIP_POOL_WEIGHTED_SUM)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid push feature");
    if (f.occurrences && !f.indices) return Fail(EPS_HIP_INVALID_ARGUMENT, "null feature indices");
    if (f.pooling != EPS_HIP_POOL_SEQUENCE && (!f.offsets || (f.pooling == EPS_HIP_POOL_MEAN && !f.valid_lengths)))
      return Fail(EPS_HIP_INVALID_ARGUMENT, "pooled feature needs offsets (and lengths for mean)");
    if (f.pooling != EPS_HIP_POOL_SEQUENCE && f.occurrences && !f.bags)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "pooled feature with occurrences but no bags");
    if (f.pooling == EPS_HIP_POOL_WEIGHTED_SUM && f.occurrences && !f.weights)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "weighted feature needs weights");
    const uint64_t rows = f.pooling == EPS_HIP_POOL_SEQUENCE ? f.occurrences : f.bags;
    if (rows >= (1ull << kRefRowBits)) return Fail(EPS_HIP_CAPACITY_EXCEEDED, "feature has too many rows");
    plan.occurrences += f.occurrences;
    if (f.pooling != EPS_HIP_POOL_SEQUENCE && f.occurrences) staged += f.bags + 1;
    plan.class_occurrences[DimClass(tables[f.table].dim)] += f.occurrences;
  }
  if (plan.occurrences >= (1ull << 30)) return Fail(EPS_HIP_CAPACITY_EXCEEDED, "too many occurrences");
  plan.small = plan.occurrences <= kSmallOccurrences && staged <= kSmallOffsets;
  // A small push is sorted by whole keys, a larger one by slots within each
  // table.
  const uint32_t bits = plan.small ? plan.key_bits : plan.row_bits;
  const uint32_t passes = (bits + kRadixBits - 1) / kRadixBits;
  if (passes > kMaxPasses) return Fail(EPS_HIP_CAPACITY_EXCEEDED, "sort keys need too many passes");
  uint32_t at = 0;
  for (uint32_t p = 0; p < passes; ++p) {
    const uint32_t remaining = bits - at, left = passes - p;
    plan.bits[p] = (remaining + left - 1) / left;
    plan.shift[p] = at;
    at += plan.bits[p];
  }
  plan.passes = plan.small ? 1 : passes;
  plan.small_passes = plan.small ? passes : 0;
  return EPS_HIP_OK;
}

// Final sorted buffers after `passes` passes starting from A.
inline bool SortedInB(uint32_t passes) { return passes % 2 == 1; }

}  // namespace eps_hip

using namespace eps_hip;

extern "C" {

uint64_t eps_hip_push_workspace_bytes(uint64_t occurrences) {
  return PushLayout(occurrences).total;
}

}  // extern "C"

namespace eps_hip {
namespace {
// The one-block preparation of a small push.
int PrepareSmall(const eps_hip_table* tables, uint32_t table_count, const eps_hip_push_feature* features,
                 uint32_t feature_count, const PushPlan& plan, const PushLayout& L, uint8_t* ws, hipStream_t s,
                 bool with_vals, const HotArgs& hot, uint32_t sentinel) {
  SmallArgs a{};
  a.count = feature_count;
  a.n = uint32_t(plan.occurrences);
  a.row_bits = plan.row_bits;
  a.sentinel = sentinel;
  a.passes = plan.small_passes;
  for (uint32_t p = 0; p < kMaxPasses; ++p) { a.shift[p] = plan.shift[p]; a.bits[p] = plan.bits[p]; }
  for (uint32_t c = 0; c < kClasses; ++c) a.class_key[c] = plan.class_start[c];
  a.class_key[kClasses] = table_count;
  uint32_t occ = 0, off = 0;
  for (uint32_t i = 0; i < feature_count; ++i) {
    const auto& in = features[i];
    SmallFeature& f = a.f[i];
    f.indices = in.indices; f.offsets = in.offsets; f.lengths = in.valid_lengths; f.weights = in.weights;
    f.table_rows = tables[in.table].rows;
    f.occ_begin = occ; f.bags = uint32_t(in.bags); f.off_begin = off;
    f.key_index = plan.key_index[in.table];
    f.pooling = in.occurrences ? in.pooling : EPS_HIP_POOL_SEQUENCE;  // no offsets are read without occurrences
    occ += uint32_t(in.occurrences);
    if (f.pooling != EPS_HIP_POOL_SEQUENCE) off += uint32_t(in.bags + 1);
  }
  a.keys = reinterpret_cast<uint32_t*>(ws + L.keys_b);
  a.vals = with_vals ? reinterpret_cast<uint32_t*>(ws + L.vals_b) : nullptr;
  a.rs = reinterpret_cast<uint64_t*>(ws + L.sorted_rs);
  a.hot = hot;
  hipLaunchKernelGGL(SmallPrepareKernel, dim3(1), dim3(kSortBlock), 0, s, a);
  EPS_HIP_LAUNCHED("small prepare");
  return EPS_HIP_OK;
}

int Prepare(const eps_hip_table* tables, uint32_t table_count, const eps_hip_push_feature* features,
            uint32_t feature_count, void* workspace, uint64_t workspace_bytes, void* stream, bool with_vals) {
  PushPlan plan;
  EPS_HIP_TRY(PlanPush(tables, table_count, features, feature_count, plan));
  const PushLayout L(plan.occurrences);
  if (!workspace || workspace_bytes < L.total)
    return Fail(EPS_HIP_CAPACITY_EXCEEDED, "push workspace too small");
  auto* ws = static_cast<uint8_t*>(workspace);
  auto* ctrl = reinterpret_cast<Control*>(ws);
  const hipStream_t s = AsStream(stream);
  // The control block (but its status history) starts at zero: the first
  // launch of a preparation clears it.
  if (!plan.occurrences)
    return LaunchFill(reinterpret_cast<uint32_t*>(ws), 0, sizeof(Control) / 4, s, kHistoryWord);
  const uint32_t n = uint32_t(plan.occurrences);
  const uint32_t sentinel = plan.key_bits >= 32 ? 0xffffffffu : ((1u << plan.key_bits) - 1);
  uint32_t* keys[2] = {reinterpret_cast<uint32_t*>(ws + L.keys_a), reinterpret_cast<uint32_t*>(ws + L.keys_b)};
  uint32_t* vals[2] = {reinterpret_cast<uint32_t*>(ws + L.vals_a), reinterpret_cast<uint32_t*>(ws + L.vals_b)};
  HotArgs ha{};
  ha.keys = keys[plan.passes % 2];
  ha.hot = reinterpret_cast<HotEntry*>(ws + L.long_list);
  ha.ctrl = ctrl;
  ha.n = n;
  ha.capacity = uint32_t(L.HotCapacity());
  ha.generic_key = plan.class_start[kClasses - 1] < table_count
                       ? uint32_t(uint64_t(plan.class_start[kClasses - 1]) << plan.row_bits) : 0xffffffffu;
  if (plan.small)
    return PrepareSmall(tables, table_count, features, feature_count, plan, L, ws, s, with_vals, ha, sentinel);

  PrepArgs args{};
  args.count = feature_count;
  args.row_bits = plan.row_bits;
  args.sentinel = sentinel;
  args.passes = plan.passes;
  args.digits = 1u << plan.bits[0];  // the widest pass
  for (uint32_t p = 0; p < kMaxPasses; ++p) { args.shift[p] = plan.shift[p]; args.bits[p] = plan.bits[p]; }
  args.ctrl = ctrl;
  args.info = reinterpret_cast<TileInfo*>(ws + L.info);
  args.counts = reinterpret_cast<uint16_t*>(ws + L.counts);
  args.keys = keys[0];
  args.vals = with_vals ? vals[0] : nullptr;
  // Reference words ping-pong between two buffers through the passes and
  // end in sorted_rs: keygen writes them where an even number of swaps
  // before the end starts.  A push with no weighted-sum feature sorts them
  // as 4-byte words without their scales (a third less sort traffic) and the
  // last pass puts the scales back.
  uint64_t* rs[2] = {reinterpret_cast<uint64_t*>(ws + (plan.passes % 2 ? L.refscale : L.sorted_rs)),
                     reinterpret_cast<uint64_t*>(ws + (plan.passes % 2 ? L.sorted_rs : L.refscale))};
  ScaleArgs sc{};
  bool narrow = true;
  for (uint32_t i = 0; i < feature_count; ++i) {
    if (features[i].pooling == EPS_HIP_POOL_WEIGHTED_SUM) narrow = false;
    if (features[i].pooling == EPS_HIP_POOL_MEAN) {
      sc.mean_mask |= 1u << i;
      sc.lengths[i] = features[i].valid_lengths;
    }
  }
  args.refscale = narrow ? nullptr : rs[0];
  args.refs = narrow ? reinterpret_cast<uint32_t*>(rs[0]) : nullptr;

  // Features table by table (call order within a table), their tiles, and the
  // segments they make up.
  uint32_t occ_begin[EPS_HIP_MAX_FEATURES];
  uint64_t occ = 0;
  for (uint32_t i = 0; i < feature_count; ++i) {
    occ_begin[i] = uint32_t(occ);
    occ += features[i].occurrences;
  }
  SortArgs first{}, later{};
  uint32_t blocks = 0, later_blocks = 0, at = 0, used = 0, segments = 0, most_tiles = 0;
  for (uint32_t k = 0; k < table_count; ++k) {
    const uint32_t seg_at = at, seg_block = blocks;
    for (uint32_t i = 0; i < feature_count; ++i) {
      const auto& in = features[i];
      if (in.table != plan.table_of_key[k] || !in.occurrences) continue;
      first.span_tile[used] = blocks;
      first.span[used] = SortSpan{at, uint32_t(in.occurrences), segments};
      PrepFeature& f = args.f[used++];
      f.indices = in.indices; f.offsets = in.offsets; f.lengths = in.valid_lengths; f.weights = in.weights;
      f.occurrences = in.occurrences; f.bags = in.bags; f.table_rows = tables[in.table].rows;
      f.occ_begin = occ_begin[i]; f.sort_begin = at; f.key_index = k; f.pooling = in.pooling; f.feature = i;
      f.block_begin = blocks;
      at += uint32_t(in.occurrences);
      blocks += uint32_t((in.occurrences + kSortTile - 1) / kSortTile);
    }
    if (at == seg_at) continue;
    first.seg_begin[segments] = seg_at;
    first.seg_tile[segments] = seg_block;
    first.seg_key[segments] = k;
    later.span_tile[segments] = later_blocks;
    later.span[segments] = SortSpan{seg_at, at - seg_at, segments};
    later_blocks += (at - seg_at + kSortTile - 1) / kSortTile;
    most_tiles = std::max(most_tiles, blocks - seg_block);
    first.seg_tile[++segments] = blocks;
  }
  if (std::max(blocks, later_blocks) > L.tiles) return Fail(EPS_HIP_RUN_FAILED, "push tiles exceed the workspace");
  args.count = used;
  args.tiles = blocks;
  const bool direct = most_tiles <= kDirectTiles;
  // The look-back flags of the passes that look back (per pass: its tiles'
  // rows, then its groups') start at zero, and the per-table counts that lie
  // before them.
  const uint64_t look_words = uint64_t(args.digits) * (std::max(blocks, later_blocks) + L.groups);
  uint32_t* look = reinterpret_cast<uint32_t*>(ws + L.look);
  args.zero = direct ? look + look_words : reinterpret_cast<uint32_t*>(ws + L.hist);
  args.zero_words = uint64_t(look + look_words * plan.passes - args.zero);
  hipLaunchKernelGGL(KeygenKernel, dim3(blocks), dim3(kKeyBlock), 0, s, args);
  EPS_HIP_LAUNCHED("keygen");
  if (!direct) {
    CountSumArgs ca{};
    uint32_t sum_blocks = 0;
    for (uint32_t g = 0; g < segments; ++g) {
      ca.part[g] = {sum_blocks, first.seg_tile[g], first.seg_tile[g + 1], g};
      sum_blocks += (first.seg_tile[g + 1] - first.seg_tile[g] + kSumTiles - 1) / kSumTiles;
    }
    ca.parts = segments;
    ca.passes = plan.passes;
    ca.digits = args.digits;
    ca.tiles = blocks;
    ca.counts = args.counts;
    ca.hist = reinterpret_cast<uint32_t*>(ws + L.hist);
    hipLaunchKernelGGL(CountSumKernel, dim3(sum_blocks), dim3(kBlock), 0, s, ca);
    EPS_HIP_LAUNCHED("digit counts");
  }
  for (uint32_t i = used; i < kMaxSpans; ++i) first.span_tile[i] = ~0u;
  for (uint32_t i = segments; i < kMaxSpans; ++i) later.span_tile[i] = ~0u;
  for (uint32_t g = 0; g <= segments; ++g) later.seg_tile[g] = first.seg_tile[g];
  for (uint32_t g = 0; g < segments; ++g) {
    later.seg_begin[g] = first.seg_begin[g];
    later.seg_key[g] = first.seg_key[g];
  }
  for (uint32_t p = 0; p < plan.passes; ++p) {
    SortArgs a = p == 0 ? first : later;
    const uint32_t grid = p == 0 ? blocks : later_blocks;
    a.segments = segments;
    a.shift = plan.shift[p];
    a.bits = plan.bits[p];
    a.digits = args.digits;
    a.pass = p;
    a.passes = plan.passes;
    a.count_tiles = blocks;
    a.sentinel = sentinel;
    a.direct = direct ? 1u : 0u;
    for (uint32_t c = 0; c < kClasses; ++c) a.class_key[c] = plan.class_start[c];
    a.class_key[kClasses] = table_count;
    a.counts = args.counts;
    a.hist = reinterpret_cast<const uint32_t*>(ws + L.hist);
    a.info = args.info;
    a.look = look + look_words * p;
    a.group_look = a.look + uint64_t(args.digits) * grid;
    a.ctrl = ctrl;
    a.keys_in = keys[p % 2];
    a.vals_in = vals[p % 2];
    a.keys_out = keys[(p + 1) % 2];
    a.vals_out = vals[(p + 1) % 2];
    a.rs_in = rs[p % 2];
    a.rs_out = rs[(p + 1) % 2];
    const int form = !narrow ? kWide : (p + 1 < plan.passes ? kNarrow : kWiden);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(kSortBlock), 0, s, a, sc); };
    if (form == kWide)
      launch(with_vals ? RadixPassKernel<true, kWide> : RadixPassKernel<false, kWide>);
    else if (form == kNarrow)
      launch(with_vals ? RadixPassKernel<true, kNarrow> : RadixPassKernel<false, kNarrow>);
    else
      launch(with_vals ? RadixPassKernel<true, kWiden> : RadixPassKernel<false, kWiden>);
    EPS_HIP_LAUNCHED("radix pass");
  }
  // Hot rows of the sorted keys.
  if (n > kLongRefs) {
    hipLaunchKernelGGL(HotListKernel, dim3((n + kBlock * kHotItems - 1) / (kBlock * kHotItems)), dim3(kBlock), 0, s,
                       ha);
    EPS_HIP_LAUNCHED("hot rows");
  }
  return EPS_HIP_OK;
}
}  // namespace

int PrepareWithOccurrences(const eps_hip_table* tables, uint32_t table_count,
                           const eps_hip_push_feature* features, uint32_t feature_count, void* workspace,
                           uint64_t workspace_bytes, void* stream) {
  return Prepare(tables, table_count, features, feature_count, workspace, workspace_bytes, stream, true);
}
}  // namespace eps_hip

extern "C" {

int eps_hip_prepare(const eps_hip_table* tables, uint32_t table_count,
                    const eps_hip_push_feature* features, uint32_t feature_count,
                    void* workspace, uint64_t workspace_bytes, void* stream) {
  return Prepare(tables, table_count, features, feature_count, workspace, workspace_bytes, stream, false);
}

int eps_hip_unique(const eps_hip_table* tables, uint32_t table_count,
                   const eps_hip_push_feature* features, uint32_t feature_count,
                   void* workspace, uint64_t workspace_bytes, uint64_t* unique_slots,
                   uint32_t* unique_tables, uint64_t* occurrence_to_unique,
                   uint64_t* unique_count, void* stream) {
  PushPlan plan;
  EPS_HIP_TRY(PlanPush(tables, table_count, features, feature_count, plan));
  const PushLayout L(plan.occurrences);
  if (!workspace || workspace_bytes < L.total)
    return Fail(EPS_HIP_CAPACITY_EXCEEDED, "push workspace too small");
  if (!unique_slots || !unique_tables || !occurrence_to_unique)
    return Fail(EPS_HIP_INVALID_ARGUMENT, "null unique outputs");
  EPS_HIP_TRY(PrepareWithOccurrences(tables, table_count, features, feature_count, workspace, workspace_bytes,
                                     stream));
  auto* ws = static_cast<uint8_t*>(workspace);
  auto* ctrl = reinterpret_cast<Control*>(ws);
  const hipStream_t s = AsStream(stream);
  const uint32_t n = uint32_t(plan.occurrences);
  // Holes keep UINT64_MAX (include/eps/types.hpp:139; cache_backend.cu:281).
  EPS_HIP_TRY(LaunchFill(reinterpret_cast<uint32_t*>(occurrence_to_unique), 0xffffffffu, 2ull * n, s));
  if (!n) {
    if (unique_count) EPS_HIP_TRY(LaunchFill(reinterpret_cast<uint32_t*>(unique_count), 0, 2, s));
    return EPS_HIP_OK;
  }
  const bool in_b = SortedInB(plan.passes);
  const auto* keys = reinterpret_cast<const uint32_t*>(ws + (in_b ? L.keys_b : L.keys_a));
  const auto* vals = reinterpret_cast<const uint32_t*>(ws + (in_b ? L.vals_b : L.vals_a));
  auto* flags = reinterpret_cast<uint32_t*>(ws + L.flags);
  auto* ranks = reinterpret_cast<uint32_t*>(ws + L.ranks);
  auto* sums = reinterpret_cast<uint32_t*>(ws + L.block_sums);
  const uint32_t scan_blocks = (n + 1023) / 1024;
  EPS_HIP_TRY(LaunchFill(flags, 0, n, s));
  if (unique_count) EPS_HIP_TRY(LaunchFill(reinterpret_cast<uint32_t*>(unique_count), 0, 2, s));
  hipLaunchKernelGGL(HeadFlagKernel, dim3(Grid(n, 8192)), dim3(kBlock), 0, s, keys, vals, ctrl, flags, n);
  EPS_HIP_LAUNCHED("head flags");
  hipLaunchKernelGGL(ScanBlockSumsKernel, dim3(scan_blocks), dim3(kBlock), 0, s, flags, sums, n);
  EPS_HIP_LAUNCHED("scan sums");
  hipLaunchKernelGGL(ScanTopKernel, dim3(1), dim3(kBlock), 0, s, sums, scan_blocks, ctrl, unique_count);
  EPS_HIP_LAUNCHED("scan top");
  hipLaunchKernelGGL(ScanApplyKernel, dim3(scan_blocks), dim3(kBlock), 0, s, flags, sums, ranks, n);
  EPS_HIP_LAUNCHED("scan apply");
  UniqueArgs uargs{};
  for (uint32_t k = 0; k < table_count; ++k) uargs.table_of_key[k] = plan.table_of_key[k];
  hipLaunchKernelGGL(UniqueWriteKernel, dim3(Grid(n, 8192)), dim3(kBlock), 0, s, keys, vals, ranks,
                     ctrl, n, plan.row_bits, uargs, unique_slots, unique_tables,
                     occurrence_to_unique);
  EPS_HIP_LAUNCHED("unique write");
  return EPS_HIP_OK;
}

}  // extern "C"
