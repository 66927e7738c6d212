// gather.hip -- pooled gather (pull), row-state movement and initialisation.
//
// Pull = one launch for up to 32 features.  A block owns a tile of output rows
// (bags, or positions for sequence pooling) of one feature.  It stages the
// tile's bag offsets and row slots in LDS (one coalesced pass, unique->slot
// remap and range checks done once per occurrence), then sub-wavefront groups
// of G lanes (dim / V rounded up to a power of two, 4..64) each own one output
// row: lane l holds columns [V*l, V*l+V) (and those 64*V further on, for rows
// wider than a wavefront) and adds the bag's rows with loads of V floats,
// strictly in occurrence order from +0.0f, as the reference does (GatherKernel,
// src/cuda/cache_backend.cu:81-94; PrepareFeature,
// src/access/batch_access.cpp:41-50).  V is the widest of 4, 2 and 1 that the
// dimension, the stride and the buffers' alignment allow.  The mean divide of the client
// (src/client/distributed_client.cpp:227-232; NormalizeMean,
// src/cuda/cache_backend.cu:134-139) is fused into the store.
#include "common.hpp"

#include <algorithm>
#include <cfloat>
#include <mutex>
#include <type_traits>

namespace eps_hip {

static thread_local std::string g_error;
void SetError(const std::string& message) { g_error = message; }
int Fail(int code, const std::string& message) { g_error = message; return code; }
int Check(hipError_t e, const char* what) {
  if (e == hipSuccess) return EPS_HIP_OK;
  g_error = std::string(what) + ": " + hipGetErrorString(e);
  return e == hipErrorOutOfMemory ? EPS_HIP_CAPACITY_EXCEEDED : EPS_HIP_RUN_FAILED;
}

namespace {

constexpr uint32_t kIdCap = 1024;     // occurrences staged in LDS per tile (LDS sets the occupancy)
constexpr uint32_t kGatherBatch = 8;  // source rows in flight per lane group
constexpr int kBufferWord3 = 0x00020000;         // raw buffer resource, dword data (gfx9 family)
// An offset past every buffer range, also with the columns of a row of up to
// kBufferDim floats added to it.
constexpr uint32_t kBufferOutside = 0xFFFE0000u, kBufferDim = 16384;
typedef int EpsI4 __attribute__((ext_vector_type(4)));

struct GatherDesc {
  const float* source;
  const uint64_t* indices;
  const uint64_t* remap;
  const uint64_t* offsets;
  const uint64_t* lengths;
  const float* weights;
  float* output;
  uint64_t stride, rows, source_rows, remap_count;
  uint32_t dim, pooling, block_begin;
  uint16_t log2g, rows_per_block, width, reserved;  // width: floats of a load
  uint32_t pieces_magic;  // sequence parts: 2^32 / (dim / width), rounded up
  // Bytes of the source when they fit a 32-bit buffer range (0: they do not):
  // the row loads then go through a buffer resource, and the slots of a batch
  // past the bag's end (or holes) take an offset outside the range, which
  // returns zeros without a memory request.  Rows read with the range's whole
  // stride lie inside it, whatever the dimension.
  uint32_t buffer_bytes;
};
struct GatherArgs {
  GatherDesc part[EPS_HIP_MAX_GATHER_PARTS];
  uint32_t count;
  uint32_t* status;
};
static_assert(sizeof(GatherArgs) <= 4096, "gather arguments fit the kernel-argument segment");

// Slot of an occurrence's index (or kHole); range failures are reported and skipped.
__device__ __forceinline__ uint64_t ResolveSlot(const GatherDesc& d, uint64_t idx, bool& bad) {
  if (idx == kHole) return kHole;
  if (d.remap) {
    if (idx >= d.remap_count) { bad = true; return kHole; }
    idx = d.remap[idx];
  }
  if (idx >= d.source_rows) { bad = true; return kHole; }
  return idx;
}

// V floats of a row: a load, and a load through the part's buffer resource.
template <uint32_t V> struct Columns { float c[V]; };
template <uint32_t V>
__device__ __forceinline__ Columns<V> LoadColumns(const float* p) {
  Columns<V> r;
  if constexpr (V == 4) {
    const float4 x = Load4(p);
    r.c[0] = x.x; r.c[1] = x.y; r.c[2] = x.z; r.c[3] = x.w;
  } else if constexpr (V == 2) {
    typedef float F2 __attribute__((ext_vector_type(2)));
    const F2 x = *(const EPS_GLOBAL F2*)(p);
    r.c[0] = x.x; r.c[1] = x.y;
  } else {
    r.c[0] = LoadF(p);
  }
  return r;
}
template <uint32_t V>
__device__ __forceinline__ Columns<V> LoadColumns(__amdgpu_buffer_rsrc_t rsrc, uint32_t at) {
  Columns<V> r;
  if constexpr (V == 4) {
    const EpsI4 q = __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, 0);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) r.c[k] = __int_as_float(q[k]);
  } else if constexpr (V == 2) {
    const auto q = __builtin_amdgcn_raw_buffer_load_b64(rsrc, at, 0, 0);
    r.c[0] = __int_as_float(int(q[0]));
    r.c[1] = __int_as_float(int(q[1]));
  } else {
    r.c[0] = __int_as_float(int(__builtin_amdgcn_raw_buffer_load_b32(rsrc, at, 0, 0)));
  }
  return r;
}
template <uint32_t V>
__device__ __forceinline__ void StoreColumns(float* p, const Columns<V>& r) {
  if constexpr (V == 4) {
    Store4(p, make_float4(r.c[0], r.c[1], r.c[2], r.c[3]));
  } else if constexpr (V == 2) {
    typedef float F2 __attribute__((ext_vector_type(2)));
    *(EPS_GLOBAL F2*)(p) = F2{r.c[0], r.c[1]};
  } else {
    StoreF(p, r.c[0]);
  }
}

// Where each staged occurrence's row starts: its byte offset in the part's
// buffer range (kBufferOutside: a hole), or, for sources past such a range,
// its 64-bit byte offset (kHole: a hole).
struct GatherShared {
  uint64_t off[kBlock / 4 + 1];
  union {
    uint32_t at32[kIdCap + kGatherBatch];
    uint64_t at64[kIdCap];
  };
  float weight[kIdCap + kGatherBatch];
  uint32_t bad;
};

// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ uint64_t Uniform(uint64_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(x)), hi = __builtin_amdgcn_readfirstlane(uint32_t(x >> 32));
  return lo | (uint64_t(hi) << 32);
}

// Orders a wavefront's LDS accesses before and after it (they are performed in
// order: the compiler is held).
__device__ __forceinline__ void WaveLdsFence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Stages the row of one occurrence, of index `idx`, as entry `k`.
__device__ __forceinline__ void StageRow(const GatherDesc& d, GatherShared& sh, uint32_t k, uint64_t idx, bool& bad) {
  const uint64_t slot = ResolveSlot(d, idx, bad);
  if (d.buffer_bytes) sh.at32[k] = slot == kHole ? kBufferOutside : uint32_t(slot * d.stride * 4);
  else sh.at64[k] = slot == kHole ? kHole : slot * d.stride * 4;
}

// Stages occurrences [first, first + n) of a part (n <= kIdCap): the remap and
// the range check are done once per occurrence.
__device__ __forceinline__ void StageOccurrences(const GatherDesc& d, GatherShared& sh, uint64_t first, uint32_t n,
                                                 bool& bad) {
  for (uint32_t k = threadIdx.x; k < n; k += kBlock) {
    StageRow(d, sh, k, d.indices[first + k], bad);
    if (d.pooling == EPS_HIP_POOL_WEIGHTED_SUM) sh.weight[k] = d.weights[first + k];
  }
}

// The output rows row0 .. row0 + nrows of a pooled part, a group of 2^log2g
// lanes per row (at most one row a group) and V columns a lane.  The block's
// occurrences [occ_begin, occ_end) are staged at once when there are up to
// kIdCap of them.  In a block with more, each group stages its own bag's, its
// share of the entries (four a lane) at a time; when one bag has them all
// (kOneBag), the whole block stages them for its group, kIdCap at a time.
// Each is staged as the offset of its row, so that a load costs a lane one LDS
// read and an add instead of a 64-bit multiply per row and lane, which bound
// the launch: 26 x 4,096 bags of 1-20 rows of dim 64, 46 -> 41 us; 4 x 262,144
// bags of 32 rows of dim 128 (38 GB of state, past a buffer range), 1,775 ->
// 1,071 us.
template <uint32_t V, bool kWeighted, bool kBuffered, bool kOneBag>
__device__ __forceinline__ void PoolRows(const GatherDesc& d, GatherShared& sh, uint64_t row0, uint32_t nrows,
                                         uint64_t occ_begin, uint64_t occ_end, bool none, bool& bad) {
  const uint32_t G = 1u << d.log2g;
  const uint32_t lig = threadIdx.x & (G - 1);
  const uint32_t r = threadIdx.x >> d.log2g;
  const bool once = !kOneBag && occ_end - occ_begin <= kIdCap;  // (uniform over the block)
  if (once) {
    StageOccurrences(d, sh, occ_begin, uint32_t(occ_end - occ_begin), bad);
    __syncthreads();
  }
  // A mean's divisor (0: none), asked for before the rows.
  float divisor = 0.f;
  if (d.pooling == EPS_HIP_POOL_MEAN && d.lengths && r < nrows) divisor = (float)d.lengths[row0 + r];
  constexpr uint32_t kOwn = kIdCap / kBlock;  // entries of a lane
  const uint32_t room = kOwn << d.log2g;      // entries of a group
  // A bag of one row of several steps is a copy of it (through +0.0f): its
  // steps' loads go out together, without the rest of a batch (10,000 bags of
  // dim 258, 12.7 us as sums, 7.8 so; of dim 300, 10.4 and 7.8).
  const uint64_t first = sh.off[r] - occ_begin;
  if (once && G * V < d.dim && r < nrows && sh.off[r + 1] - sh.off[r] == 1 && sh.off[r + 1] <= occ_end &&
      first < kIdCap && (kBuffered || sh.at64[first] != kHole)) {  // (staged, whatever the offsets)
    const uint32_t at = kBuffered ? sh.at32[first] : 0u;  // (a hole reads zeros)
    const float weight = !kWeighted ? 1.f : kBuffered && at == kBufferOutside ? 0.f : sh.weight[first];
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(d.source), (short)0, int(d.buffer_bytes), kBufferWord3);
    const float* row = d.source + (kBuffered ? 0 : sh.at64[first] / 4);
    float* out = d.output + (row0 + r) * d.dim;
#pragma unroll 4
    for (uint32_t c = lig * V; c < d.dim; c += G * V) {
      Columns<V> x;
      if constexpr (kBuffered) x = LoadColumns<V>(rsrc, at + c * 4);
      else x = LoadColumns<V>(row + c);
#pragma unroll
      for (uint32_t q = 0; q < V; ++q) {
        x.c[q] = 0.f + (kWeighted ? x.c[q] * weight : x.c[q]);
        if (divisor != 0.f) x.c[q] = x.c[q] / divisor;
      }
      StoreColumns<V>(out + c, x);
    }
    return;
  }
  // One step for rows of up to 64 * V columns.
  for (uint32_t c0 = 0; c0 < d.dim; c0 += G * V) {
    const uint32_t c = c0 + lig * V;
    const bool active = c < d.dim;
    Columns<V> acc;
#pragma unroll
    for (uint32_t k = 0; k < V; ++k) acc.c[k] = 0.f;
    auto add = [&](const Columns<V>& x, float a) {
#pragma unroll
      for (uint32_t k = 0; k < V; ++k) {
        if (kWeighted) acc.c[k] += x.c[k] * a;
        else acc.c[k] += x.c[k];
      }
    };
    // Adds the staged entries [first, e), kBatch rows in flight.
    auto add_staged = [&](auto batch, uint32_t first, uint32_t e) {
      constexpr uint32_t kBatch = decltype(batch)::value;
      if constexpr (kBuffered) {
        // Through the buffer range: occurrences past the bag and holes read
        // zeros without a memory request, and adding them (weighted: zero
        // times a weight of zero) changes no sum, since one that starts at
        // +0.0f is never -0.0f.  The loads of a batch are issued before any
        // is added.
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(d.source), (short)0, int(d.buffer_bytes), kBufferWord3);
        for (uint32_t pos = first; pos < e; pos += kBatch) {
          Columns<V> v[kBatch];
          uint32_t at[kBatch];
#pragma unroll
          for (uint32_t u = 0; u < kBatch; ++u) at[u] = sh.at32[pos + u];
#pragma unroll
          for (uint32_t u = 0; u < kBatch; ++u) {
            at[u] = pos + u < e ? at[u] : kBufferOutside;
            v[u] = LoadColumns<V>(rsrc, at[u] + c * 4);
          }
#pragma unroll
          for (uint32_t u = 0; u < kBatch; ++u)
            add(v[u], !kWeighted ? 1.f : at[u] != kBufferOutside ? sh.weight[pos + u] : 0.f);
        }
      } else if (d.source_rows) {  // (without rows every occurrence is a hole)
        // No branch around a load: a hole or a position past the bag reads
        // row 0 and is dropped.
        const char* source = reinterpret_cast<const char*>(d.source + c);
        for (uint32_t pos = first; pos < e; pos += kBatch) {
          Columns<V> v[kBatch];
          bool ok[kBatch];
#pragma unroll
          for (uint32_t u = 0; u < kBatch; ++u) {
            const uint64_t at = sh.at64[min(pos + u, e - 1)];
            ok[u] = pos + u < e && at != kHole;
            v[u] = LoadColumns<V>(reinterpret_cast<const float*>(source + (ok[u] ? at : 0)));
          }
#pragma unroll
          for (uint32_t u = 0; u < kBatch; ++u)
            if (ok[u]) add(v[u], kWeighted ? sh.weight[pos + u] : 1.f);
        }
      }
    };
    if constexpr (kOneBag) {
      for (uint64_t chunk = occ_begin; chunk < occ_end; chunk += kIdCap) {
        const uint32_t n = uint32_t(min<uint64_t>(kIdCap, occ_end - chunk));
        __syncthreads();  // the chunk before has been added
        StageOccurrences(d, sh, chunk, n, bad);
        __syncthreads();
        if (active && sh.off[r] == occ_begin && sh.off[r + 1] == occ_end)
          add_staged(std::integral_constant<uint32_t, kGatherBatch>{}, 0u, n);
      }
    } else if (once) {
      // (Kept inside the staged entries, whatever the offsets.)
      const uint64_t from = max(sh.off[r], occ_begin), to = min(sh.off[r + 1], occ_end);
      if (active && from < to)
        add_staged(std::integral_constant<uint32_t, kGatherBatch>{}, uint32_t(from - occ_begin),
                   uint32_t(to - occ_begin));
    } else if (!none) {
      // A group lies in one wavefront, whose LDS accesses are performed in
      // order, so no barrier comes between the groups: with the block staging
      // kIdCap occurrences between two barriers, one bag of a block was added
      // at a time (1,000 bags of 1,500 rows of dim 64, 16 bags a block: 1,036
      // us, 128 so; 64 of 2,000 of dim 4, a block: 3,860, 257 so).  A block's
      // only bag is better off with that (20,000 rows of dim 3: 0.99 ms, its
      // group alone 2.65; 500,000 of dim 64: 23, 29).
      const uint32_t entry = r * room;
      for (uint64_t from = max(sh.off[r], occ_begin); from < min(sh.off[r + 1], occ_end); from += room) {
        const uint32_t n = uint32_t(min<uint64_t>(room, min(sh.off[r + 1], occ_end) - from));
        uint64_t idx[kOwn];
#pragma unroll
        for (uint32_t k = 0; k < kOwn; ++k) idx[k] = d.indices[from + min(k * G + lig, n - 1)];
#pragma unroll
        for (uint32_t k = 0; k < kOwn; ++k) {
          const uint32_t at = k * G + lig;
          if (at < n) StageRow(d, sh, entry + at, idx[k], bad);
        }
        if constexpr (kWeighted) {
          __builtin_amdgcn_sched_barrier(0);  // (all at once, they cost the launch a wavefront a SIMD)
          float weight[kOwn];
#pragma unroll
          for (uint32_t k = 0; k < kOwn; ++k) weight[k] = d.weights[from + min(k * G + lig, n - 1)];
#pragma unroll
          for (uint32_t k = 0; k < kOwn; ++k)
            if (k * G + lig < n) sh.weight[entry + k * G + lig] = weight[k];
        }
        WaveLdsFence();
        if (active) add_staged(std::integral_constant<uint32_t, V == 4 && kWeighted ? 6 : kGatherBatch>{}, entry, entry + n);
        WaveLdsFence();  // the entries have been read
      }
    }
    if (r >= nrows || !active) continue;
    if (divisor != 0.f) {
#pragma unroll
      for (uint32_t k = 0; k < V; ++k) acc.c[k] = acc.c[k] / divisor;
    }
    StoreColumns<V>(d.output + (row0 + r) * d.dim + c, acc);
  }
}

// The output rows row0 .. row0 + nrows of a sequence part, each a copy of one
// source row (through +0.0f, as a sum of one; zeros for a hole).  The block's
// rows are one run of pieces of V columns, kGatherBatch of them in flight a
// thread: with a lane group per row a group had one load in flight and most
// lanes of a row wider than a wavefront's columns were idle (five tables of
// 20,011 bags of dims 16 to 300, one of them 130,000 sequence rows of dim 300:
// the launch 127 us, now 55).
template <uint32_t V>
__device__ __forceinline__ void CopyRows(const GatherDesc& d, const GatherShared& sh, uint64_t row0, uint32_t nrows) {
  const uint32_t per_row = d.dim / V, total = nrows * per_row;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(d.source), (short)0, int(d.buffer_bytes), kBufferWord3);
  float* out = d.output + row0 * d.dim;
  for (uint32_t first = threadIdx.x; first < total; first += kBlock * kGatherBatch) {
    Columns<V> v[kGatherBatch];
    bool ok[kGatherBatch];
#pragma unroll
    for (uint32_t u = 0; u < kGatherBatch; ++u) {
      const uint32_t e = min(first + u * kBlock, total - 1);
      // e / per_row: exact for the at most 2^14 pieces of a block (or one row).
      const uint32_t r = per_row == 1 ? e : nrows > 1 ? __umulhi(e, d.pieces_magic) : 0u;
      const uint32_t col = (e - r * per_row) * V;
      if (d.buffer_bytes) {
        v[u] = LoadColumns<V>(rsrc, sh.at32[r] + col * 4);  // a hole reads zeros
        ok[u] = true;
      } else {
        const uint64_t at = sh.at64[r];
        ok[u] = at != kHole;
#pragma unroll
        for (uint32_t k = 0; k < V; ++k) v[u].c[k] = 0.f;
        if (d.source_rows)  // else every row is a hole
          v[u] = LoadColumns<V>(reinterpret_cast<const float*>(reinterpret_cast<const char*>(d.source) + (ok[u] ? at : 0)) +
                                (ok[u] ? col : 0u));
      }
    }
#pragma unroll
    for (uint32_t u = 0; u < kGatherBatch; ++u) {
      if (first + u * kBlock >= total) continue;
#pragma unroll
      for (uint32_t k = 0; k < V; ++k) v[u].c[k] = ok[u] ? 0.f + v[u].c[k] : 0.f;
      StoreColumns<V>(out + uint64_t(first + u * kBlock) * V, v[u]);
    }
  }
}

__global__ void __launch_bounds__(kBlock) GatherKernel(GatherArgs args) {
  const GatherDesc d = args.part[PartOf(args.part, args.count)];

  __shared__ GatherShared sh;

  const bool seq = d.pooling == EPS_HIP_POOL_SEQUENCE;
  const uint64_t row0 = uint64_t(blockIdx.x - d.block_begin) * d.rows_per_block;
  if (row0 >= d.rows) return;
  const uint32_t nrows = uint32_t(min<uint64_t>(d.rows_per_block, d.rows - row0));
  if (threadIdx.x == 0) sh.bad = 0;
  bool bad = false;
  if (seq) {
    StageOccurrences(d, sh, row0, nrows, bad);
    __syncthreads();
    if (d.width == 4) CopyRows<4>(d, sh, row0, nrows);
    else if (d.width == 2) CopyRows<2>(d, sh, row0, nrows);
    else CopyRows<1>(d, sh, row0, nrows);
  } else {
    // (Groups past the rows have empty bags.)
    for (uint32_t r = threadIdx.x; r <= kBlock / 4; r += kBlock) sh.off[r] = d.offsets[row0 + min(r, nrows)];
    __syncthreads();
    const uint64_t occ_begin = Uniform(sh.off[0]);
    // A part without indices has no occurrences (every bag empty): nothing is
    // read, and offsets that claim occurrences are reported as bad indices.
    const bool none = d.indices == nullptr;
    if (none && sh.off[nrows] != occ_begin && threadIdx.x == 0) sh.bad = 1;
    const uint64_t occ_end = none ? occ_begin : Uniform(sh.off[nrows]);
    const bool one_bag = occ_end - occ_begin > kIdCap && !none &&
                         __syncthreads_or(sh.off[threadIdx.x & (kBlock / 4 - 1)] == occ_begin &&
                                          sh.off[(threadIdx.x & (kBlock / 4 - 1)) + 1] == occ_end);
    auto pool = [&](auto v, auto weighted, auto through) {
      auto rows = [&](auto one) {
        PoolRows<decltype(v)::value, decltype(weighted)::value, decltype(through)::value, decltype(one)::value>(
            d, sh, row0, nrows, occ_begin, occ_end, none, bad);
      };
      if (one_bag) rows(std::true_type{});
      else rows(std::false_type{});
    };
    auto with_width = [&](auto weighted, auto through) {
      if (d.width == 4) pool(std::integral_constant<uint32_t, 4>{}, weighted, through);
      else if (d.width == 2) pool(std::integral_constant<uint32_t, 2>{}, weighted, through);
      else pool(std::integral_constant<uint32_t, 1>{}, weighted, through);
    };
    auto with_weights = [&](auto through) {
      if (d.pooling == EPS_HIP_POOL_WEIGHTED_SUM) with_width(std::true_type{}, through);
      else with_width(std::false_type{}, through);
    };
    if (d.buffer_bytes) with_weights(std::true_type{});
    else with_weights(std::false_type{});
  }
  if (bad) sh.bad = 1;
  __syncthreads();
  if (threadIdx.x == 0 && sh.bad && args.status) atomicOr(args.status, EPS_HIP_STATUS_BAD_INDEX);
}

__global__ void AddContributionKernel(float* output, const float* source, const uint64_t* positions,
                                      uint64_t values, uint32_t dim) {
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < values;
       i += uint64_t(blockDim.x) * gridDim.x) {
    const uint64_t target = positions ? positions[i / dim] * dim + i % dim : i;
    output[target] += source[i];
  }
}

// NormalizeMean (src/cuda/cache_backend.cu:134-139): output[r, d] /= len[r]
// for len[r] != 0, an IEEE float divide by the length converted to float.
__global__ void NormalizeMeanKernel(float* output, const uint64_t* lengths, uint64_t rows,
                                    uint32_t dim) {
  const uint64_t values = rows * dim;
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < values;
       i += uint64_t(blockDim.x) * gridDim.x) {
    const uint64_t len = lengths[i / dim];
    if (len) output[i] = output[i] / (float)len;
  }
}

// target[i] = value for i < count, except i == keep (kept as it is).
__global__ void FillKernel(uint32_t* target, uint32_t value, uint64_t count, uint64_t keep) {
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count;
       i += uint64_t(blockDim.x) * gridDim.x)
    if (i != keep) target[i] = value;
}

__device__ __forceinline__ uint64_t Mix(uint64_t x) {
  x += 0x9e3779b97f4a7c15ULL;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ULL;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebULL;
  return x ^ (x >> 31);
}

__device__ __forceinline__ void BoundMax(Bounds* bounds, uint32_t w, uint32_t m, uint32_t v) {
  w = WaveMax(w); m = WaveMax(m); v = WaveMax(v);
  if ((threadIdx.x & (kWave - 1)) == 0 && bounds) {
    uint32_t* slot = bounds->v[(blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave) % kBoundSlots];
    if (w) atomicMax(slot + 0, w);
    if (m) atomicMax(slot + 1, m);
    if (v) atomicMax(slot + 2, v);
  }
}

// ShardStore::Ensure's initializer (src/store/shard_store.cpp:104-112) for
// key = key_base + slot * key_stride; salt = Mix(seed) ^ Mix(table id).
__global__ void InitRowsKernel(float* state, uint32_t dim, uint64_t first, uint64_t count,
                               uint64_t key_base, uint64_t key_stride, uint64_t salt,
                               double lo, double hi, int32_t bounded, float wmin, float wmax,
                               Bounds* bounds) {
  uint32_t wmax_bits = 0;
  const uint64_t total = count * dim;
  for (uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
       e += uint64_t(blockDim.x) * gridDim.x) {
    const uint64_t slot = first + e / dim;
    const uint32_t col = uint32_t(e % dim);
    const uint64_t key = key_base + slot * key_stride;
    const uint64_t bits = Mix(key ^ salt ^ Mix(uint64_t(col)));
    const double u = double(bits >> 11) * 0x1.0p-53;
    float w = float((1 - u) * lo + u * hi);
    if (bounded) w = Clamp(w, wmin, wmax);
    float* row = state + slot * uint64_t(dim) * 3;
    row[col] = w;
    row[dim + col] = 0.f;
    row[2 * dim + col] = 0.f;
    wmax_bits = max(wmax_bits, AbsBits(w));
  }
  BoundMax(bounds, wmax_bits, 0, 0);
}

// ScatterState (src/cuda/cache_backend.cu:69-74): packed [w|m|v] rows -> slots.
// From pinned host memory the host link bounds it, and the link is slower with
// more reads waiting on it than fill it: 4,096 rows of dim 64 (3.1 MB) take 128
// us with 8 blocks of 16-byte loads, 68 with 16, 60 with 32 or 64, 64 with 256
// and 79 with 768, a thread a load (a copy of that size 69).  The other widths
// and counts gain as much or nothing: 65,536 rows of dim 4 77 -> 59, 262,144 262
// -> 223, 1,024 6.5 either way; 16,384 rows of dim 256 957 -> 879.  Loads of 4
// bytes keep a thread a load.
constexpr unsigned kHostReadGrid = 64;
__global__ void ScatterRowsKernel(float* state, uint32_t dim, const uint64_t* slots,
                                  const float* packed, uint64_t count, Bounds* bounds) {
  uint32_t bw = 0, bm = 0, bv = 0;
  const uint64_t width = uint64_t(dim) * 3;
  if ((dim & 3) == 0) {
    const uint64_t w4 = width / 4, total = count * w4;
    for (uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
         e += uint64_t(blockDim.x) * gridDim.x) {
      const uint64_t row = e / w4, col = (e % w4) * 4;
      const float4 x = Load4(packed + row * width + col);
      Store4(state + slots[row] * width + col, x);
      const uint32_t a = max(max(AbsBits(x.x), AbsBits(x.y)), max(AbsBits(x.z), AbsBits(x.w)));
      if (col < dim) bw = max(bw, a); else if (col < 2 * dim) bm = max(bm, a); else bv = max(bv, a);
    }
  } else {
    const uint64_t total = count * width;
    for (uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
         e += uint64_t(blockDim.x) * gridDim.x) {
      const uint64_t row = e / width, col = e % width;
      const float x = packed[e];
      state[slots[row] * width + col] = x;
      if (col < dim) bw = max(bw, AbsBits(x)); else if (col < 2 * dim) bm = max(bm, AbsBits(x));
      else bv = max(bv, AbsBits(x));
    }
  }
  BoundMax(bounds, bw, bm, bv);
}

// ReadStateKernel (src/cuda/cache_backend.cu:75-80): slots -> packed rows.
__global__ void GatherRowsKernel(const float* state, uint32_t dim, const uint64_t* slots,
                                 float* packed, uint64_t count) {
  const uint64_t width = uint64_t(dim) * 3;
  if ((dim & 3) == 0) {
    const uint64_t w4 = width / 4, total = count * w4;
    for (uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
         e += uint64_t(blockDim.x) * gridDim.x) {
      const uint64_t row = e / w4, col = (e % w4) * 4;
      Store4(packed + row * width + col, Load4(state + slots[row] * width + col));
    }
  } else {
    const uint64_t total = count * width;
    for (uint64_t e = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
         e += uint64_t(blockDim.x) * gridDim.x)
      packed[e] = state[slots[e / width] * width + e % width];
  }
}

// Row moves of several tables in one launch (admissions: packed -> slots,
// like ScatterRowsKernel; write-backs: slots -> packed, like
// GatherRowsKernel).  A part's 16-byte pieces (scalar floats when dim % 4)
// form chunks of kBlock * kMovePerThread; the launch's blocks take the chunks
// of all parts in turn (chunk c, c + gridDim.x, ...).  When one side is host
// memory the grid is small: each block's loads wait microseconds on the host
// link, and a few blocks keep enough bytes in flight for it without holding
// wave slots the step's own kernels need.
constexpr uint32_t kMovePerThread = 4;
constexpr uint32_t kHostLinkGrid = 16;  // blocks of a move that crosses the host link (best of 8-64 on
                                         // config 5: fewer slow the moves, more slow the step)
struct MoveDesc {
  float* state;
  float* packed;
  const uint64_t* slots;
  uint64_t count;
  uint32_t dim, block_begin;  // block_begin: the part's first chunk
};
struct MoveArgs {
  MoveDesc part[EPS_HIP_MAX_TABLES];
  uint32_t count, chunks;
  uint32_t write_back;
  Bounds* bounds;
};

__global__ void __launch_bounds__(kBlock) MoveRowsKernel(MoveArgs a) {
  uint32_t bw = 0, bm = 0, bv = 0;
  for (uint32_t chunk = blockIdx.x; chunk < a.chunks; chunk += gridDim.x) {
    const MoveDesc d = a.part[PartOf(a.part, a.count, chunk)];
    const uint64_t width = uint64_t(d.dim) * 3;
    const bool vec = (d.dim & 3) == 0;
    const uint64_t per_row = vec ? width / 4 : width;
    const uint64_t items = d.count * per_row;
    const uint64_t first = uint64_t(chunk - d.block_begin) * kBlock * kMovePerThread;
    // Every load of the thread is issued before any store: one side may be
    // host memory, microseconds away over the host link.
    const float* src[kMovePerThread];
    float* dst[kMovePerThread];
    uint64_t col[kMovePerThread];
    bool ok[kMovePerThread];
#pragma unroll
    for (uint32_t k = 0; k < kMovePerThread; ++k) {
      const uint64_t e = first + uint64_t(k) * kBlock + threadIdx.x;
      ok[k] = e < items;
      const uint64_t row = ok[k] ? e / per_row : 0, piece = ok[k] ? e % per_row : 0;
      col[k] = vec ? piece * 4 : piece;
      float* slot_row = d.state + (ok[k] ? d.slots[row] : 0) * width + col[k];
      float* packed = d.packed + row * width + col[k];
      src[k] = a.write_back ? slot_row : packed;
      dst[k] = a.write_back ? packed : slot_row;
    }
    if (vec) {
      float4 x[kMovePerThread];
#pragma unroll
      for (uint32_t k = 0; k < kMovePerThread; ++k) x[k] = ok[k] ? Load4(src[k]) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (uint32_t k = 0; k < kMovePerThread; ++k) {
        if (!ok[k]) continue;
        Store4(dst[k], x[k]);
        const uint32_t m = max(max(AbsBits(x[k].x), AbsBits(x[k].y)), max(AbsBits(x[k].z), AbsBits(x[k].w)));
        if (col[k] < d.dim) bw = max(bw, m); else if (col[k] < 2 * d.dim) bm = max(bm, m); else bv = max(bv, m);
      }
    } else {
      float x[kMovePerThread];
#pragma unroll
      for (uint32_t k = 0; k < kMovePerThread; ++k) x[k] = ok[k] ? LoadF(src[k]) : 0.f;
#pragma unroll
      for (uint32_t k = 0; k < kMovePerThread; ++k) {
        if (!ok[k]) continue;
        StoreF(dst[k], x[k]);
        if (col[k] < d.dim) bw = max(bw, AbsBits(x[k])); else if (col[k] < 2 * d.dim) bm = max(bm, AbsBits(x[k]));
        else bv = max(bv, AbsBits(x[k]));
      }
    }
  }
  if (!a.write_back) BoundMax(a.bounds, bw, bm, bv);
}

unsigned GridFor(uint64_t n, unsigned cap = 65536) {
  const uint64_t blocks = (n + kBlock - 1) / kBlock;
  return unsigned(blocks < 1 ? 1 : (blocks > cap ? cap : blocks));
}

uint64_t HostMix(uint64_t x) {
  x += 0x9e3779b97f4a7c15ULL;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ULL;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebULL;
  return x ^ (x >> 31);
}

// Device-visible address of a row buffer: device memory as is, pinned host
// memory through its mapped device pointer; pageable host memory is refused
// (a kernel must never dereference an unmapped host address).
int DeviceAddress(const void* p, const void** out, bool* host = nullptr) {
  hipPointerAttribute_t attr;
  if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
    (void)hipGetLastError();
    return Fail(EPS_HIP_INVALID_ARGUMENT, "row buffer must be device memory or pinned host memory");
  }
  if (host) *host = attr.type == hipMemoryTypeHost;
  if (attr.type == hipMemoryTypeHost) {
    if (!attr.devicePointer) return Fail(EPS_HIP_INVALID_ARGUMENT, "pinned host buffer is not mapped");
    *out = attr.devicePointer;
  } else {
    *out = p;
  }
  return EPS_HIP_OK;
}

int CheckTable(const eps_hip_table* t) {
  if (!t || !t->state) return Fail(EPS_HIP_INVALID_ARGUMENT, "null table");
  if (t->dim == 0 || t->dim > 65536) return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid dimension");
  if (reinterpret_cast<uintptr_t>(t->state) % 16)
    return Fail(EPS_HIP_INVALID_ARGUMENT, "table state must be 16-byte aligned");
  return EPS_HIP_OK;
}

}  // namespace

int LaunchFill(uint32_t* target, uint32_t value, uint64_t count, hipStream_t stream, uint64_t keep) {
  if (!count) return EPS_HIP_OK;
  hipLaunchKernelGGL(FillKernel, dim3(GridFor(count, 4096)), dim3(kBlock), 0, stream, target,
                     value, count, keep);
  EPS_HIP_LAUNCHED("fill");
  return EPS_HIP_OK;
}

}  // namespace eps_hip

using namespace eps_hip;

extern "C" {

int eps_hip_abi_version(void) { return EPS_HIP_ABI_VERSION; }
const char* eps_hip_last_error(void) { return g_error.c_str(); }

int eps_hip_device_check(int device) {
  EPS_HIP_TRY(Check(hipSetDevice(device), "hipSetDevice"));
  hipDeviceProp_t prop;
  EPS_HIP_TRY(Check(hipGetDeviceProperties(&prop, device), "hipGetDeviceProperties"));
  if (std::string(prop.gcnArchName).rfind("gfx950", 0) != 0)
    return Fail(EPS_HIP_UNAVAILABLE, std::string("device is ") + prop.gcnArchName + ", not gfx950");
  return EPS_HIP_OK;
}

uint64_t eps_hip_bounds_bytes(void) { return sizeof(Bounds); }

int eps_hip_bounds_reset(void* bounds, void* stream) {
  if (!bounds) return Fail(EPS_HIP_INVALID_ARGUMENT, "null bounds");
  return LaunchFill(static_cast<uint32_t*>(bounds), 0, sizeof(Bounds) / 4, AsStream(stream));
}

int eps_hip_fill_u32(uint32_t* target, uint32_t value, uint64_t count, void* stream) {
  if (!target && count) return Fail(EPS_HIP_INVALID_ARGUMENT, "null target");
  return LaunchFill(target, value, count, AsStream(stream));
}

int eps_hip_init_rows(const eps_hip_table* t, uint64_t first, uint64_t count, uint64_t key_base,
                      uint64_t key_stride, uint64_t seed, float init_min, float init_max,
                      int32_t bounded, float weight_min, float weight_max, void* bounds,
                      void* stream) {
  EPS_HIP_TRY(CheckTable(t));
  if (first > t->rows || count > t->rows - first)
    return Fail(EPS_HIP_INVALID_ARGUMENT, "initialised slots exceed table rows");
  if (!count) return EPS_HIP_OK;
  const uint64_t salt = HostMix(seed) ^ HostMix(uint64_t(t->id));
  hipLaunchKernelGGL(InitRowsKernel, dim3(GridFor(count * t->dim)), dim3(kBlock), 0,
                     AsStream(stream), t->state, t->dim, first, count, key_base, key_stride, salt,
                     double(init_min), double(init_max), bounded, weight_min, weight_max,
                     static_cast<Bounds*>(bounds));
  EPS_HIP_LAUNCHED("init rows");
  return EPS_HIP_OK;
}

int eps_hip_scatter_rows(const eps_hip_table* t, const uint64_t* slots, const float* packed,
                         uint64_t count, void* bounds, void* stream) {
  EPS_HIP_TRY(CheckTable(t));
  if (!count) return EPS_HIP_OK;
  if (!slots || !packed) return Fail(EPS_HIP_INVALID_ARGUMENT, "null scatter buffers");
  const void* source = nullptr;
  bool host = false;
  EPS_HIP_TRY(DeviceAddress(packed, &source, &host));
  packed = static_cast<const float*>(source);
  const bool vec = t->dim % 4 == 0;
  const uint64_t work = vec ? count * t->dim * 3 / 4 : count * t->dim * 3;
  const unsigned grid = host && vec ? GridFor(work, kHostReadGrid) : GridFor(work);
  hipLaunchKernelGGL(ScatterRowsKernel, dim3(grid), dim3(kBlock), 0, AsStream(stream),
                     t->state, t->dim, slots, packed, count, static_cast<Bounds*>(bounds));
  EPS_HIP_LAUNCHED("scatter rows");
  return EPS_HIP_OK;
}

int eps_hip_gather_rows(const eps_hip_table* t, const uint64_t* slots, float* packed,
                        uint64_t count, void* stream) {
  EPS_HIP_TRY(CheckTable(t));
  if (!count) return EPS_HIP_OK;
  if (!slots || !packed) return Fail(EPS_HIP_INVALID_ARGUMENT, "null gather buffers");
  const void* target = nullptr;
  EPS_HIP_TRY(DeviceAddress(packed, &target));
  packed = static_cast<float*>(const_cast<void*>(target));
  const uint64_t work = (t->dim % 4 == 0) ? count * t->dim * 3 / 4 : count * t->dim * 3;
  hipLaunchKernelGGL(GatherRowsKernel, dim3(GridFor(work)), dim3(kBlock), 0, AsStream(stream),
                     t->state, t->dim, slots, packed, count);
  EPS_HIP_LAUNCHED("gather rows");
  return EPS_HIP_OK;
}

int eps_hip_move_rows(const eps_hip_row_batch* batches, uint32_t count, int32_t write_back, void* bounds,
                      void* stream) {
  if (count > EPS_HIP_MAX_TABLES) return Fail(EPS_HIP_INVALID_ARGUMENT, "too many row batches");
  if (count && !batches) return Fail(EPS_HIP_INVALID_ARGUMENT, "null row batches");
  MoveArgs args{};
  args.write_back = write_back ? 1u : 0u;
  args.bounds = static_cast<Bounds*>(bounds);
  uint64_t blocks = 0;
  bool host_link = false;
  for (uint32_t i = 0; i < count; ++i) {
    const eps_hip_row_batch& b = batches[i];
    if (!b.count) continue;
    if (!b.state || !b.slots || !b.packed || b.dim == 0 || b.dim > 65536)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid row batch");
    if (reinterpret_cast<uintptr_t>(b.state) % 16) return Fail(EPS_HIP_INVALID_ARGUMENT, "table state must be 16-byte aligned");
    const void* packed = nullptr;
    bool host = false;
    EPS_HIP_TRY(DeviceAddress(b.packed, &packed, &host));
    host_link = host_link || host;
    if ((b.dim & 3) == 0 && reinterpret_cast<uintptr_t>(packed) % 16)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "packed rows must be 16-byte aligned");
    MoveDesc& d = args.part[args.count++];
    d.state = b.state;
    d.packed = static_cast<float*>(const_cast<void*>(packed));
    d.slots = b.slots;
    d.count = b.count;
    d.dim = b.dim;
    d.block_begin = uint32_t(blocks);
    const uint64_t per_row = (b.dim & 3) == 0 ? uint64_t(b.dim) * 3 / 4 : uint64_t(b.dim) * 3;
    blocks += (b.count * per_row + kBlock * kMovePerThread - 1) / (kBlock * kMovePerThread);
    if (blocks >= (1ull << 31)) return Fail(EPS_HIP_CAPACITY_EXCEEDED, "row move grid too large");
  }
  if (!blocks) return EPS_HIP_OK;
  args.chunks = uint32_t(blocks);
  const uint64_t grid = std::min<uint64_t>(blocks, host_link ? kHostLinkGrid : 65536);
  hipLaunchKernelGGL(MoveRowsKernel, dim3(unsigned(grid)), dim3(kBlock), 0, AsStream(stream), args);
  EPS_HIP_LAUNCHED("move rows");
  return EPS_HIP_OK;
}

int eps_hip_gather(const eps_hip_gather_part* parts, uint32_t count, uint32_t* status,
                   void* stream) {
  if (count > EPS_HIP_MAX_GATHER_PARTS) return Fail(EPS_HIP_INVALID_ARGUMENT, "too many gather parts");
  GatherArgs args{};
  args.status = status;
  uint32_t blocks = 0, used = 0;
  for (uint32_t p = 0; p < count; ++p) {
    const auto& in = parts[p];
    if (in.dim == 0 || in.pooling > EPS_HIP_POOL_WEIGHTED_SUM)
      return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid gather part");
    if (in.rows == 0) continue;
    // indices (and weights) may be NULL only for a pooled part whose bags are
    // all empty; offsets that claim occurrences then raise the bad-index bit.
    if (!in.source || !in.output || (in.pooling == EPS_HIP_POOL_SEQUENCE && !in.indices) ||
        (in.pooling != EPS_HIP_POOL_SEQUENCE && !in.offsets) ||
        (in.pooling == EPS_HIP_POOL_WEIGHTED_SUM && in.indices && !in.weights))
      return Fail(EPS_HIP_INVALID_ARGUMENT, "null gather buffer");
    GatherDesc& d = args.part[used++];
    d.source = in.source; d.indices = in.indices; d.remap = in.remap; d.offsets = in.offsets;
    d.lengths = in.valid_lengths; d.weights = in.weights; d.output = in.output;
    d.stride = in.stride; d.rows = in.rows; d.source_rows = in.source_rows;
    d.remap_count = in.remap_count; d.dim = in.dim; d.pooling = in.pooling;
    const uint64_t source_bytes = in.source_rows * in.stride * 4;
    d.buffer_bytes = source_bytes && source_bytes <= kBufferOutside && in.source_rows < (1ull << 32) &&
                             in.stride <= kBufferOutside && in.dim <= kBufferDim
                         ? uint32_t(source_bytes) : 0u;
    // The widest load that every row and the output allow.
    auto fits = [&](uint32_t v) {
      return in.dim % v == 0 && in.stride % v == 0 && reinterpret_cast<uintptr_t>(in.source) % (4 * v) == 0 &&
             reinterpret_cast<uintptr_t>(in.output) % (4 * v) == 0;
    };
    const uint32_t width = fits(4) ? 4u : fits(2) ? 2u : 1u;
    uint32_t log2g = 2;
    while (log2g < 6 && (width << log2g) < in.dim) ++log2g;
    d.width = uint16_t(width);
    d.log2g = uint16_t(log2g);
    d.rows_per_block = uint16_t(kBlock >> log2g);  // one bag per lane group
    if (in.pooling == EPS_HIP_POOL_SEQUENCE) {
      // A batch of pieces per thread, staged slots permitting.
      const uint32_t per_row = in.dim / width;
      d.rows_per_block = uint16_t(std::min(std::max(kBlock * kGatherBatch / per_row, 1u), kIdCap));
      d.pieces_magic = uint32_t((uint64_t(1) << 32) / per_row + (per_row > 1));
    }
    d.block_begin = blocks;
    const uint64_t b = (in.rows + d.rows_per_block - 1) / d.rows_per_block;
    if (b > (1ull << 31) - blocks) return Fail(EPS_HIP_CAPACITY_EXCEEDED, "gather grid too large");
    blocks += uint32_t(b);
  }
  args.count = used;
  if (!blocks) return EPS_HIP_OK;
  hipLaunchKernelGGL(GatherKernel, dim3(blocks), dim3(kBlock), 0, AsStream(stream), args);
  EPS_HIP_LAUNCHED("gather");
  return EPS_HIP_OK;
}

int eps_hip_normalize_mean(float* output, const uint64_t* lengths, uint64_t rows, uint32_t dim,
                           void* stream) {
  if (!rows) return EPS_HIP_OK;
  if (!output || !lengths || !dim) return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid mean normalisation");
  hipLaunchKernelGGL(NormalizeMeanKernel, dim3(GridFor(rows * dim)), dim3(kBlock), 0,
                     AsStream(stream), output, lengths, rows, dim);
  EPS_HIP_LAUNCHED("normalize mean");
  return EPS_HIP_OK;
}

int eps_hip_add_contribution(float* output, const float* source, const uint64_t* positions,
                             uint64_t values, uint32_t dim, void* stream) {
  if (!values) return EPS_HIP_OK;
  if (!output || !source || !dim) return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid contribution");
  hipLaunchKernelGGL(AddContributionKernel, dim3(GridFor(values)), dim3(kBlock), 0,
                     AsStream(stream), output, source, positions, values, dim);
  EPS_HIP_LAUNCHED("add contribution");
  return EPS_HIP_OK;
}

}  // extern "C"
