// adam.hip -- duplicate-id aggregation fused with sparse (Lazy)Adam.
//
// Per unique row, one sub-wavefront group of G lanes (lane l owns columns
// [4l, 4l+4)) sums the row's references in order from +0.0f -- acc = acc +
// src * scale, separate multiply and add -- (ReduceGradients,
// src/access/batch_access.cpp:73-93; ExpandCompactGradients,
// src/access/compact_gradients.cpp:31-36; ReduceFeatureGradients,
// src/cuda/cache_backend.cu:115-125), then reads the row's w, m, v once, applies
//   m' = b1*m + (1-b1)*g;  v' = b2*v + ((1-b2)*g)*g;  w' = w - (lr_t*m')/(sqrt(v')+eps)
// and the clamp (src/update/lazy_adam.cpp:31-35; AdamKernel,
// src/cuda/cache_backend.cu:95-114), and writes w, m, v once.
//
// All-or-nothing without a second pass over the state.  The reference
// validates every element before any write, with a second full state pass
// (ValidateLazyAdam then ApplyLazyAdam; AdamKernel twice).  Here a guard decides
// before the update whether overflow is impossible:
//   * bounds domain: running maxima W >= |w|, M >= |m|, V >= v of every value
//     this library ever wrote (init, admission, updates);
//   * G >= |g| for every reduced gradient: max|source| * max(1, max|scale|) *
//     references * (1+2^-24)^(references+2) (rounding growth of a sequential sum);
//   * then |m'| <= b1*M + (1-b1)*G, v' <= b2*V + (1-b2)*G^2 and
//     |w'| <= W + lr_t*|m'|/eps (since sqrt(v') + eps >= eps), each widened by 1%.
// If every bound stays below 1e30 (far below FLT_MAX) no element can overflow and
// the single fused pass runs ("fused").  Otherwise the same kernel runs in
// validate-only mode and a second launch applies only if nothing failed
// ("checked") -- the reference's two-pass behaviour.  A non-finite gradient value
// or an out-of-range slot rejects the whole update before anything is written.
#include "prepare.hpp"

#include <hip/hip_ext.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <type_traits>

namespace eps_hip {

namespace {

constexpr uint32_t kFallbackGrid = 2048;
// Blocks of a CSR packet's tail, which has nothing to do for many packets (2,000
// rows without a long one: 512 blocks 15.0 us a call, 1,024 15.8); packets of
// kTailRows rows and more take twice as many.
constexpr uint32_t kTailGrid = 512;
constexpr uint64_t kTailRows = 1ull << 15;

// ---------------------------------------------------------------------------
// Gradient scan (GradMaxKernel), the first kernel of an update.  Its spans are
// the guarded input arrays: gradient values, reference scales, 64-bit caller
// indices that must all be below `limit`, and (a push) the sorted keys of the
// prepared workspace, whose table indices and slots must name the push's
// tables and rows.  It records max |gradient| and max |scale| for the guard
// and any range failure as a prepare-time finding, all before anything is
// written; block 0 also copies the bounds-domain maxima into the control
// block, the snapshot the guard decides from.  (The reference words are
// checked where the update kernels decode them: a word naming no gradient row
// of the push is never used as an address, and the rows it feeds are not
// written.)
enum SpanKind : uint32_t { kGradientSpan = 0, kScaleSpan = 1, kIndexSpan = 2, kSortedSpan = 3 };
struct Span {
  const float* p;
  uint64_t count;
  uint32_t block_begin, kind;
  uint64_t limit;
};
// What the sorted keys are checked against (key index order for tables).
struct SortedCheck {
  const uint32_t* keys;
  uint64_t table_rows[EPS_HIP_MAX_TABLES];
  uint32_t row_bits, tables;
};
struct GuardArgs {
  Span span[EPS_HIP_MAX_FEATURES + 4];
  uint32_t spans;
  Control* ctrl;
  const Bounds* bounds;  // snapshot source (NULL: no snapshot)
  SortedCheck sorted;
};
static_assert(sizeof(GuardArgs) <= 4096, "gradient scan arguments fit the kernel-argument segment");
constexpr uint32_t kMaxItems = 16;     // float4 per thread per block (all issued before any is used)
constexpr uint32_t kSortedItems = 16;  // sorted keys per thread per block
constexpr uint32_t kIndexItems = 16;   // caller indices per thread per block

__global__ void __launch_bounds__(kBlock) GradMaxKernel(GuardArgs a) {
  __shared__ uint32_t s_max[4];
  __shared__ uint64_t s_rows[EPS_HIP_MAX_TABLES];
  if (blockIdx.x == 0 && threadIdx.x < kWave && a.bounds) {
    const uint32_t lane = threadIdx.x;
    const uint32_t w = WaveMax(a.bounds->v[lane][0]), m = WaveMax(a.bounds->v[lane][1]),
                   v = WaveMax(a.bounds->v[lane][2]);
    if (lane == 0) {
      a.ctrl->snap[0] = w;
      a.ctrl->snap[1] = m;
      a.ctrl->snap[2] = v;
    }
  }
  if (!a.spans) return;
  const Span sp = a.span[PartOf(a.span, a.spans)];
  uint32_t m = 0;
  uint32_t found = 0;  // prepare-status bits this thread found
  if (sp.kind == kSortedSpan) {
    const SortedCheck& c = a.sorted;
    if (threadIdx.x < EPS_HIP_MAX_TABLES) s_rows[threadIdx.x] = c.table_rows[threadIdx.x];
    __syncthreads();
    // Positions past the valid count hold keys of rows not on this device,
    // which no update kernel reads.
    const uint64_t per_block = uint64_t(kBlock) * kSortedItems;
    const uint64_t begin = uint64_t(blockIdx.x - sp.block_begin) * per_block;
    {
      // Every load is issued before any is used (and before the valid count
      // is known): positions past the span read the block's first position,
      // and positions past the valid count are not judged.
      uint32_t key[kSortedItems];
#pragma unroll
      for (uint32_t k = 0; k < kSortedItems; ++k) {
        const uint64_t i = begin + uint64_t(k) * kBlock + threadIdx.x;
        key[k] = c.keys[i < sp.count ? i : begin];
      }
      const uint64_t valid = min<uint64_t>(sp.count, a.ctrl->valid_count);
      bool bad = false;
#pragma unroll
      for (uint32_t k = 0; k < kSortedItems; ++k) {
        const uint64_t i = begin + uint64_t(k) * kBlock + threadIdx.x;
        const KeyParts kp = SplitKey(key[k], c.row_bits);
        bad |= i < valid && !KeyInRange(kp, c.tables, s_rows[min(kp.table, EPS_HIP_MAX_TABLES - 1u)]);
      }
      if (bad) found = EPS_HIP_STATUS_BAD_INDEX;
    }
  } else if (sp.kind == kIndexSpan) {
    // All of a thread's loads are issued before any is compared (positions
    // past the span read the block's first index): a loop over 64 indices a
    // thread, one load in flight each, made this the longest part of the scan
    // (40,003 slots beside 20 MB of gradients: 20.1 -> 6.1 us).
    const uint64_t per_block = uint64_t(kBlock) * kIndexItems;
    const uint64_t begin = uint64_t(blockIdx.x - sp.block_begin) * per_block;
    const uint64_t* idx = reinterpret_cast<const uint64_t*>(sp.p);
    uint64_t x[kIndexItems];
#pragma unroll
    for (uint32_t k = 0; k < kIndexItems; ++k) {
      const uint64_t i = begin + uint64_t(k) * kBlock + threadIdx.x;
      x[k] = idx[i < sp.count ? i : begin];
    }
    bool bad = false;
#pragma unroll
    for (uint32_t k = 0; k < kIndexItems; ++k) bad |= x[k] >= sp.limit;
    if (bad) found = EPS_HIP_STATUS_BAD_INDEX;
  } else {
    const uint64_t per_block = uint64_t(kBlock) * kMaxItems * 4;
    const uint64_t begin = uint64_t(blockIdx.x - sp.block_begin) * per_block;
    const uint64_t end = min(begin + per_block, sp.count);
    if (reinterpret_cast<uintptr_t>(sp.p) % 16 == 0) {
      const uint64_t vend = begin + ((end - begin) & ~uint64_t(3));
      // Every load is issued before any is used (a branch around each would
      // make the compiler wait for each pair): quads past the vector part
      // read the block's first quad and count as zeros.
      float4 x[kMaxItems];
      if (vend > begin) {  // uniform over the block
#pragma unroll
        for (uint32_t k = 0; k < kMaxItems; ++k) {
          const uint64_t i = begin + (uint64_t(k) * kBlock + threadIdx.x) * 4;
          x[k] = Load4(sp.p + (i < vend ? i : begin));
        }
#pragma unroll
        for (uint32_t k = 0; k < kMaxItems; ++k) {
          const uint64_t i = begin + (uint64_t(k) * kBlock + threadIdx.x) * 4;
          if (i >= vend) x[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
      } else {
#pragma unroll
        for (uint32_t k = 0; k < kMaxItems; ++k) x[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      uint32_t neg = 0;  // any value below zero (not -0.0)
#pragma unroll
      for (uint32_t k = 0; k < kMaxItems; ++k) {
        m = max(m, max(max(AbsBits(x[k].x), AbsBits(x[k].y)), max(AbsBits(x[k].z), AbsBits(x[k].w))));
        neg |= (x[k].x < 0.f) | (x[k].y < 0.f) | (x[k].z < 0.f) | (x[k].w < 0.f);
      }
      for (uint64_t i = vend + threadIdx.x; i < end; i += kBlock) {
        m = max(m, AbsBits(sp.p[i]));
        neg |= sp.p[i] < 0.f;
      }
      if (sp.kind == kScaleSpan && neg) found = EPS_HIP_STATUS_BAD_SCALE;
    } else {
      for (uint64_t i = begin + threadIdx.x; i < end; i += kBlock) {
        m = max(m, AbsBits(sp.p[i]));
        if (sp.kind == kScaleSpan && sp.p[i] < 0.f) found = EPS_HIP_STATUS_BAD_SCALE;
      }
    }
    // A compact scale must be finite and >= 0 (compact_gradients.cpp:21).
    if (sp.kind == kScaleSpan && m >= 0x7f800000u) found = EPS_HIP_STATUS_BAD_SCALE;
  }
  if (found) atomicOr(&a.ctrl->prep_status, found);
  m = WaveMax(m);
  if ((threadIdx.x & (kWave - 1)) == 0) s_max[threadIdx.x / kWave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t bm = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
    if (bm)
      atomicMax(sp.kind == kScaleSpan ? &a.ctrl->scale_slots[blockIdx.x % kSrcSlots]
                                      : &a.ctrl->src_slots[blockIdx.x % kSrcSlots], bm);
  }
}

// ---------------------------------------------------------------------------
// Shared per-row arithmetic.
struct TableDesc {
  float* state;
  uint64_t rows;     // slots of the table (sorted keys must name one)
  uint32_t dim;
  float beta1, beta2, omb1, omb2, lr, eps, lo, hi;
  uint32_t bounded;  // lo/hi are the table's weight bounds (else -FLT_MAX/FLT_MAX)
};

// Running maxima of magnitude bits over a thread's elements: of the reduced
// gradients (bg), and of m, v and w (before and after the clamp) as computed.
// A maximum at or above the infinity pattern means a non-finite value; the
// m, v, w maxima of what a launch writes feed the bounds domain.
struct RowStats {
  uint32_t err = 0, bg = 0, bw = 0, bm = 0, bv = 0;
};

// Block-wide copy of a kernel-argument array to LDS, one 32-bit word per
// thread per step (the arrays are read in place from the argument segment).
template <uint32_t kThreads = kBlock>
__device__ __forceinline__ void CopyWords(void* dst, const void* src, uint32_t bytes) {
  const uint32_t* from = static_cast<const uint32_t*>(src);
  uint32_t* to = static_cast<uint32_t*>(dst);
  for (uint32_t i = threadIdx.x; i < bytes / 4; i += kThreads) to[i] = from[i];
}

// Correctly rounded square root.  For x in [2^-96, infinity) it is the
// hardware estimate s corrected to s - 1 ulp or s + 1 ulp by the signs of the
// residuals fma(-(s -/+ ulp), s, x): the steps hipcc emits for sqrtf once its
// range handling (scaling of tiny inputs, zero and infinity) is out of the
// way, so both give the same bits.  Other inputs take sqrtf.
__device__ __forceinline__ float SqrtRn(float x) {
  const uint32_t b = __float_as_uint(x);
  if (b - 0x0f800000u < 0x7f800000u - 0x0f800000u) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float below = __uint_as_float(__float_as_uint(s) - 1u);
    const float above = __uint_as_float(__float_as_uint(s) + 1u);
    const float r = fmaf(-below, s, x) <= 0.f ? below : s;
    return fmaf(-above, s, x) > 0.f ? above : r;
  }
  return sqrtf(x);
}

// One element: Adam in the reference's operation order, w clamped to the
// table's bounds (kClamp false: an unbounded table, whose clamp to
// -FLT_MAX..FLT_MAX changes no finite w, and a non-finite w is an error that
// nothing is written for).  vn is +0 or more, or NaN (v >= 0 and
// (omb2 * g) * g >= 0), so its raw bits order like its magnitude.
template <bool kClamp = true>
__device__ __forceinline__ void AdamElement(const TableDesc& T, float g, float& w, float& m,
                                            float& v, RowStats& st) {
  const float mn = T.beta1 * m + T.omb1 * g;
  const float vn = T.beta2 * v + (T.omb2 * g) * g;
  const float wn = w - (T.lr * mn) / (SqrtRn(vn) + T.eps);
  st.bg = max(st.bg, AbsBits(g));
  st.bm = max(st.bm, AbsBits(mn));
  st.bv = max(st.bv, __float_as_uint(vn));
  if (kClamp) {
    w = Clamp(wn, T.lo, T.hi);
    st.bw = max(st.bw, max(AbsBits(wn), AbsBits(w)));
  } else {
    w = wn;
    st.bw = max(st.bw, AbsBits(wn));
  }
  m = mn;
  v = vn;
}

// Vector row update: lane owns columns [c, c+4).
__device__ __forceinline__ void AdamRow4(const TableDesc& T, uint64_t slot, uint32_t c, float4 g,
                                         bool write, RowStats& st) {
  float* row = T.state + slot * uint64_t(T.dim) * 3;
  float4 w = Load4(row + c), m = Load4(row + T.dim + c), v = Load4(row + 2 * T.dim + c);
  AdamElement(T, g.x, w.x, m.x, v.x, st);
  AdamElement(T, g.y, w.y, m.y, v.y, st);
  AdamElement(T, g.z, w.z, m.z, v.z, st);
  AdamElement(T, g.w, w.w, m.w, v.w, st);
  if (write) {
    Store4(row + c, w);
    Store4(row + T.dim + c, m);
    Store4(row + 2 * T.dim + c, v);
  }
}

__device__ __forceinline__ void AdamRow1(const TableDesc& T, uint64_t slot, uint32_t c, float g,
                                         bool write, RowStats& st) {
  float* row = T.state + slot * uint64_t(T.dim) * 3;
  float w = LoadF(row + c), m = LoadF(row + T.dim + c), v = LoadF(row + 2 * T.dim + c);
  AdamElement(T, g, w, m, v, st);
  if (write) {
    StoreF(row + c, w); StoreF(row + T.dim + c, m); StoreF(row + 2 * T.dim + c, v);
  }
}

__device__ __forceinline__ void Accumulate4(float4& acc, float4 x, float s) {
  acc.x = acc.x + x.x * s;
  acc.y = acc.y + x.y * s;
  acc.z = acc.z + x.z * s;
  acc.w = acc.w + x.w * s;
}

// The guard decision (see the file comment), made by every block of the first
// kernel of an update from inputs that earlier kernels wrote and nothing
// changes while the update runs: the gradient maxima, the prepare-time
// findings and the bounds snapshot the gradient scan took (never the live
// bounds domain, which the update's own finished blocks raise).  So every
// block -- of either kernel, when two decide on two streams -- takes the same
// decision.  Block 0 publishes the mode and the status bits for the kernels
// after it.  Runs in wavefront 0 (one gradient slot and one table per lane);
// returns the mode to every thread.
static_assert(kSrcSlots == kWave, "one guard slot per lane");
struct GuardScalars {
  uint64_t refs;       // references summed into one reduced gradient, at most; 0: the prepared count
  uint32_t tables;
};
// What the decision is made from, loaded at once and before the tables are
// staged, so that a block's start waits for one memory latency and not for one
// per value.
struct GuardInputs { uint32_t grad, scale, status, w, m, v, valid; };
__device__ __forceinline__ GuardInputs LoadGuard(const Control* ctrl) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  return GuardInputs{ctrl->src_slots[lane], ctrl->scale_slots[lane], ctrl->prep_status, ctrl->snap[0],
                     ctrl->snap[1],         ctrl->snap[2],           ctrl->valid_count};
}
__device__ uint32_t DecideBlock(Control* ctrl, const GuardInputs& in, const TableDesc* t, const GuardScalars& gs,
                                uint32_t* s_mode) {
  if (threadIdx.x < kWave) {
    const uint32_t lane = threadIdx.x;
    const uint32_t gb = WaveMax(in.grad);
    const uint32_t scale_bits = WaveMax(in.scale);
    uint32_t status = in.status;
    uint32_t mode = kFused;
    if (status & (EPS_HIP_STATUS_BAD_INDEX | EPS_HIP_STATUS_BAD_SCALE)) {
      mode = kReject;
    } else if (gb >= 0x7f800000u) {
      status |= EPS_HIP_STATUS_NONFINITE_GRAD;
      mode = kReject;
    } else if (scale_bits >= 0x7f800000u) {  // a non-finite weight or scale
      status |= EPS_HIP_STATUS_BAD_SCALE;
      mode = kReject;
    } else {
      const double W = __uint_as_float(in.w), M = __uint_as_float(in.m), V = __uint_as_float(in.v);
      const double refs = double(gs.refs ? gs.refs : uint64_t(in.valid));
      const double G = GuardGradBound(__uint_as_float(gb), __uint_as_float(scale_bits), refs);
      bool table_safe = true;  // one table per lane
      if (lane < gs.tables) {
        const TableDesc& T = t[lane];
        table_safe = GuardTableSafe(T.beta1, T.beta2, T.lr, T.eps, W, M, V, G);
      }
      if (!(G < kGuardLimit) || __ballot(!table_safe) != 0) {
        mode = kChecked;
        status |= EPS_HIP_STATUS_CHECKED_PATH;
      }
    }
    if (mode == kReject) status |= EPS_HIP_STATUS_REJECTED;
    if (lane == 0) {
      *s_mode = mode;
      if (blockIdx.x == 0) {
        ctrl->mode = mode;
        ReportStatus(ctrl, status);
      }
    }
  }
  __syncthreads();
  return *s_mode;
}

// Role of a launch in an update.  The first kernel decides (DecideBlock);
// the primary kernels after it follow that decision; the fallback (the apply
// pass of the checked path) runs only when the decision was "checked" and the
// validate-only pass found nothing.
enum Role : uint32_t { kDecide = 0, kFollow = 1, kFallback = 2 };

// Whether this launch has work, and whether it writes (uniform over the
// block).  s_t must hold the launch's tables; every thread calls it.
// `in` (LoadGuard) is used by a deciding launch only.
__device__ bool LaunchGate(Control* ctrl, const GuardInputs& in, const TableDesc* s_t, const GuardScalars& gs,
                           uint32_t role, uint32_t* s_mode, bool& write) {
  if (role == kDecide) {
    __syncthreads();  // s_t is staged
    const uint32_t mode = DecideBlock(ctrl, in, s_t, gs, s_mode);
    write = mode == kFused;
    return mode != kReject;
  }
  const uint32_t mode = ctrl->mode, status = ctrl->status;
  if (role == kFollow) {
    // A stall in an earlier kernel of a fused update stops every later write.
    write = mode == kFused;
    return mode != kReject && !(status & EPS_HIP_STATUS_STALLED);
  }
  if (mode != kChecked) return false;
  if (status & (kErrorBits | EPS_HIP_STATUS_STALLED)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) ReportStatus(ctrl, EPS_HIP_STATUS_REJECTED);
    return false;
  }
  write = true;
  return true;
}

// Block-level fold of the per-lane statistics: error bits (with those the
// maxima imply) to the status word, written maxima to one slot of the bounds
// domain.
template <uint32_t kWaves = kBlock / kWave>
__device__ void FinishBlock(const RowStats& st, Control* ctrl, Bounds* bounds, bool wrote) {
  __shared__ uint32_t s_red[kWaves][4];
  uint32_t e = st.err;
  if (st.bg >= 0x7f800000u) e |= EPS_HIP_STATUS_REDUCE_OVERFLOW;
  if (max(st.bw, max(st.bm, st.bv)) >= 0x7f800000u) e |= EPS_HIP_STATUS_ADAM_OVERFLOW;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) e |= uint32_t(__shfl_xor(int(e), o));
  const uint32_t w = WaveMax(st.bw), m = WaveMax(st.bm), v = WaveMax(st.bv);
  const uint32_t wave = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) {
    s_red[wave][0] = e; s_red[wave][1] = w; s_red[wave][2] = m; s_red[wave][3] = v;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t E = 0, W = 0, M = 0, V = 0;
    for (uint32_t i = 0; i < kWaves; ++i) {
      E |= s_red[i][0]; W = max(W, s_red[i][1]); M = max(M, s_red[i][2]); V = max(V, s_red[i][3]);
    }
    ReportStatus(ctrl, E);
    if (wrote && bounds) {
      uint32_t* slot = bounds->v[blockIdx.x % kBoundSlots];
      if (W) atomicMax(slot + 0, W);
      if (M) atomicMax(slot + 1, M);
      if (V) atomicMax(slot + 2, V);
    }
  }
}

// ---------------------------------------------------------------------------
// Long rows of the sorted driver: one row's references summed by a whole block.
// A group's own loop keeps four gradient rows in flight, so a row of thousands
// of references would hold its group (and the launch) for a memory latency per
// four of them.  Here the block's threads load the gradient rows of a tile of
// 4,096 products together (2,048 in scalar columns), two tiles ahead, scale
// them and stage the products in one of two LDS tiles as [reference][column];
// thread c adds column c of the other tile in reference order meanwhile, its
// LDS reads a step ahead of its adds.  The sum is the group loop's, bit for
// bit: acc = acc + src * scale, in order, from +0 (products past the row's end
// are staged as -0.0f, the identity).  What bounds it is the adding waves:
// their adds, their share of the staging and a barrier per tile: 16 ns a
// reference of dim 64 (a tile of 8,192 products 13, but two blocks a CU).  Rows
// past 256 columns take 16-byte loads too, where their alignment allows them.
// Dedup and reduce of six tables of dims 10 to 300, 10,600 references each, the
// longest rows ~1,000: 2,057 us with a group a row, 328 with 4-byte loads and
// one tile of 16 references in flight, 202 so, 168 with the short rows launched
// apart and units of 128 columns (below).
// Rows with more references are summed by the block.  (Reduce of six tables of
// dims 10 to 300, 10,600 references each: 95 us with 16, 100 with 32, 107 with
// 64; 200,000 references of dim 64 in rows of 24 133, 123 and 123, in rows of 48
// 112, 112 and 129.)
constexpr uint32_t kBlockRowRefs = 32;
constexpr uint32_t kLongTile = 4096;     // floats of a staged tile (of two)
// Columns of a row that one block sums; wider rows are units of as many, on
// different blocks.  (43,000 references of dim 300, Zipf of 1.05, pushed: units
// of 256 columns 273 us, of 128 163.  Of 64, 133, but a CSR packet of 200,000
// references in rows of 65, dim 256, 110 instead of 76.)
constexpr uint32_t kLongColumns = 128;

// Waits for this wave's LDS accesses, then for the block's other waves: unlike
// __syncthreads it leaves global loads in flight.
__device__ __forceinline__ void LdsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The references of one row of the sorted array: Load reads reference i's
// word, Source decodes it to column `at` of its gradient row (`safe` and ok
// false when it names none of the push) and scale.
struct SortedRefs {
  typedef uint64_t Word;
  const uint64_t* rs;
  const float* const* grad;
  const uint64_t* rows;  // gradient rows per feature
  const float* safe;
  uint32_t features, dim;
  __device__ __forceinline__ Word Load(uint32_t i) const { return rs[i]; }
  __device__ __forceinline__ const float* Source(Word w, uint32_t at, float& scale, bool& ok) const {
    const RefParts rp = SplitRef(w);
    const uint32_t f = min(rp.feature, features - 1);
    const bool in = RefInRange(rp, features, rows[f]);
    if (!in) ok = false;
    scale = __uint_as_float(uint32_t(w >> 32));
    return in ? grad[f] + uint64_t(rp.row) * dim + at : safe;
  }
};

// The references of one row of a CSR packet (already range-checked by the
// gradient scan).
struct CsrRefs {
  struct Word { uint64_t row; float scale; };
  const uint64_t* sources;
  const float* scales;
  const float* src;
  uint32_t dim;
  __device__ __forceinline__ Word Load(uint32_t i) const { return Word{sources[i], scales[i]}; }
  __device__ __forceinline__ const float* Source(Word w, uint32_t at, float& scale, bool&) const {
    scale = w.scale;
    return src + w.row * dim + at;
  }
};

// `acc` plus the first `count` rows of a staged tile's column `col`, kPitch
// floats a row, in order.  Rows from `count` to the next multiple of kAddRows
// hold -0.0f.
template <uint32_t kPitch, uint32_t kAddRows>
__device__ __forceinline__ float AddTile(const float* col, uint32_t count, float acc) {
  float x[kAddRows], y[kAddRows];
  auto read = [&](float (&v)[kAddRows], uint32_t r) {
#pragma unroll
    for (uint32_t k = 0; k < kAddRows; ++k) v[k] = col[r * kPitch + k * kPitch];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto add = [&](const float (&v)[kAddRows]) {
#pragma unroll
    for (uint32_t k = 0; k < kAddRows; ++k) acc = acc + v[k];
    __builtin_amdgcn_sched_barrier(0);
  };
  read(x, 0);
#pragma clang loop unroll(disable)
  for (uint32_t r = 0; r < count; r += 2 * kAddRows) {
    if (r + kAddRows < count) read(y, r + kAddRows);
    add(x);
    if (r + kAddRows >= count) break;
    if (r + 2 * kAddRows < count) read(x, r + 2 * kAddRows);
    add(y);
  }
  return acc;
}

// Scratch of BlockRowSum: two staged tiles, and where the references of two
// groups lie.
constexpr uint32_t kRefGroup = 128;
struct RowSumShared {
  __align__(16) float tile[2][kLongTile];
  const float* src[2][kRefGroup];
  float scale[2][kRefGroup];
};

// `acc` plus references [0, count) of column c0 + threadIdx.x (`acc` past the
// unit's columns).  kVec: rows are 16-byte aligned and dim % 4 == 0.
// `ok` turns false in any thread that met a reference of no gradient row.
// Called by the whole block.  A thread each decodes the references of a group
// of 128 to LDS, a group ahead of the row loads, so that these wait for no
// reference word: loads return in issue order, and a wait for a word would
// wait for the rows in flight before it.
template <bool kVec, class Refs>
__device__ __forceinline__ float BlockRowSum(RowSumShared& sh, const Refs& refs, uint32_t count, uint32_t dim,
                                             uint32_t c0, float acc, bool& ok) {
  constexpr uint32_t kCols = kVec ? 4 : 1;                       // columns of a load
  constexpr uint32_t kTile = kVec ? kLongTile : kLongTile / 2;   // floats of a tile
  constexpr uint32_t kLoads = kTile / (kBlock * kCols);          // loads of a thread per tile
  constexpr uint32_t kDepth = 2;                                 // tiles of rows in flight
  constexpr uint32_t kAddRows = kVec ? 16 : 8;
  static_assert(kTile / kLongColumns % kAddRows == 0 && kTile / (kVec ? 32 : 16) <= kRefGroup, "tiles of whole steps, in a group");
  static_assert(kDepth % 2 == 0, "a slot's tiles lie in one half of the LDS");
  const uint32_t cols = min(dim - c0, kLongColumns);
  uint32_t log2g = kVec ? 3 : 4;                                 // lanes of a reference
  while ((kCols << log2g) < cols) ++log2g;
  const uint32_t pitch = kCols << log2g;                         // 16 to 128
  const uint32_t per_step = kBlock >> log2g, tile_refs = kTile / pitch;
  const uint32_t sub = threadIdx.x >> log2g, e = (threadIdx.x & ((1u << log2g) - 1)) * kCols;
  const uint32_t at = e < cols ? e : 0u;
  struct Rows {
    float4 x[kLoads];
    float scale[kLoads];
  } rows[kDepth];
  // References past the row's end repeat its last one.
  typename Refs::Word word;
  auto load_word = [&](uint32_t group) { word = refs.Load(min(group * kRefGroup + threadIdx.x % kRefGroup, count - 1)); };
  auto decode = [&](uint32_t group) {
    if (threadIdx.x >= kRefGroup) return;
    float scale;
    sh.src[group % 2][threadIdx.x] = refs.Source(word, c0, scale, ok);
    sh.scale[group % 2][threadIdx.x] = scale;
  };
  // The rows of the tile of references from `base` on.
  auto load_rows = [&](Rows& r, uint32_t base) {
    const uint32_t half = base / kRefGroup % 2, first = base % kRefGroup + sub;
    const float* src[kLoads];
#pragma unroll
    for (uint32_t k = 0; k < kLoads; ++k) {
      src[k] = sh.src[half][first + k * per_step] + at;
      r.scale[k] = sh.scale[half][first + k * per_step];
    }
#pragma unroll
    for (uint32_t k = 0; k < kLoads; ++k) {
      if constexpr (kVec) r.x[k] = Load4(src[k]);
      else r.x[k].x = LoadF(src[k]);
    }
  };
  // Their products, into LDS.
  auto stage = [&](float* tile, const Rows& r, uint32_t base) {
    if (e >= cols) return;  // (the padding columns are never added)
    const bool whole = base + tile_refs <= count;
#pragma unroll
    for (uint32_t k = 0; k < kLoads; ++k) {
      float* to = tile + (k * per_step + sub) * pitch + e;
      const bool in = whole || base + k * per_step + sub < count;
      const float4 x = r.x[k];
      const float s = r.scale[k];
      if constexpr (kVec)
        *reinterpret_cast<float4*>(to) =
            make_float4(in ? x.x * s : -0.f, in ? x.y * s : -0.f, in ? x.z * s : -0.f, in ? x.w * s : -0.f);
      else
        *to = in ? x.x * s : -0.f;
    }
  };
  // `ahead`: the first reference whose row is not yet asked for.  Where it
  // starts a group, that group is decoded already; the next one is now, and
  // the words of the one after it go out before the rows.
  uint32_t ahead = 0;
  auto next_rows = [&](Rows& r) {
    if (ahead % kRefGroup == 0) {
      decode(ahead / kRefGroup + 1);
      load_word(ahead / kRefGroup + 2);
    }
    load_rows(r, ahead);
    ahead += tile_refs;
  };
  load_word(0);
  LdsBarrier();  // what an earlier call left in LDS has been read
  decode(0);
  load_word(1);
#pragma unroll
  for (uint32_t d = 0; d < kDepth; ++d) {
    if (ahead % kRefGroup == 0) LdsBarrier();
    next_rows(rows[d]);
  }
  stage(sh.tile[0], rows[0], 0);
  LdsBarrier();  // tile 0 is staged, and a group's references decoded (and read)
  next_rows(rows[0]);
  // Tile t (of slot d = t % kDepth) is added, and tile t + 1 staged beside it.
#pragma clang loop unroll(disable)
  for (uint32_t base = 0; base < count;) {
#pragma unroll
    for (uint32_t d = 0; d < kDepth; ++d) {
      if (base >= count) break;  // uniform
      LdsBarrier();  // tile t is staged, tile t - 1 added
      if (threadIdx.x < cols) {
        const float* col = sh.tile[d % 2] + threadIdx.x;
        const uint32_t n = min(tile_refs, count - base);
        switch (pitch) {
          case 16: acc = AddTile<16, kAddRows>(col, n, acc); break;
          case 32: acc = AddTile<32, kAddRows>(col, n, acc); break;
          case 64: acc = AddTile<64, kAddRows>(col, n, acc); break;
          default: acc = AddTile<128, kAddRows>(col, n, acc); break;
        }
      }
      base += tile_refs;
      if (base < count) {
        Rows& r = rows[(d + 1) % kDepth];
        stage(sh.tile[(d + 1) % 2], r, base);
        next_rows(r);
      }
    }
  }
  return acc;
}

// ---------------------------------------------------------------------------
// Sorted driver: segments are runs of equal keys in the sorted key array.
struct FusedArgs {
  TableDesc t[EPS_HIP_MAX_TABLES];   // by key index
  const float* grad[EPS_HIP_MAX_FEATURES];
  uint64_t grad_rows[EPS_HIP_MAX_FEATURES];
  const uint32_t* keys;
  const uint64_t* rs;
  const uint32_t* vals;              // reduce mode: sorted occurrence indices
  const uint64_t* occ2u;             // reduce mode
  float* reduce_out;
  uint64_t reduce_stride;
  Control* ctrl;
  Bounds* bounds;
  GuardScalars gs;
  uint32_t row_bits, cls, cls_end, role, tables, features;  // classes [cls, cls_end)
  uint32_t n;     // occurrences of the push (sorted positions, occurrence indices)
  uint32_t wide;  // every gradient array is 16-byte aligned: rows of dim % 4 == 0 too
  // The short rows' windows: log2 of their positions per class, and each
  // class's first block (and the total).  The long rows': log2 of theirs, and
  // the units of columns of the widest table's.
  uint32_t window_bits[kClasses], class_block[kClasses + 1], long_bits, long_slices;
};
static_assert(sizeof(FusedArgs) <= 4096, "update arguments fit the kernel-argument segment");

struct SortedShared {
  TableDesc t[EPS_HIP_MAX_TABLES];
  const float* grad[EPS_HIP_MAX_FEATURES];
  uint64_t rows[EPS_HIP_MAX_FEATURES];  // gradient rows per feature
  uint32_t heads[kBlock];
  uint32_t wave_heads[kBlock / kWave];
  uint32_t mode;
};
struct LongRowShared {
  uint32_t heads[kBlock], count[3], bad;
  RowSumShared sum;
};
__device__ __forceinline__ void StageSorted(const FusedArgs& a, SortedShared& sh) {
  CopyWords(sh.t, a.t, sizeof(a.t));
  CopyWords(sh.grad, a.grad, sizeof(a.grad));
  CopyWords(sh.rows, a.grad_rows, sizeof(a.grad_rows));
}

// The row that starts at sorted position `sb`.  A key or reference naming
// nothing of the push (a damaged workspace) is not used as an address: its
// loads read zero and the row is not written.  The reference checks see the
// same words in every lane.
struct SortedRow { KeyParts kp; bool ok; uint64_t u; };
template <bool kReduce>
__device__ __forceinline__ SortedRow RowAt(const FusedArgs& a, const SortedShared& sh, uint32_t sb) {
  SortedRow r;
  r.kp = SplitKey(a.keys[sb], a.row_bits);
  r.ok = KeyInRange(r.kp, a.tables, sh.t[min(r.kp.table, a.tables - 1)].rows);
  r.u = 0;
  if (kReduce) {
    const uint32_t occ = a.vals[sb];
    r.ok = r.ok && occ < a.n;
    r.u = r.ok ? a.occ2u[occ] : 0;
  }
  return r;
}

// The rows of up to kBlockRowRefs references whose first position lies in the
// windows of 2^window_bits positions that blocks vb, vb + step, ... of the
// positions [start, end) own: a group of 2^log2g lanes a row (kGeneric: a
// wavefront over scalar columns).  Only references of the row are loaded: a
// batch filled up with repeats of the last one cost rows of one reference up
// to twice their time (200,000 of dim 300 reduced, 306 -> 555 us).
template <bool kGeneric, bool kReduce>
__device__ __forceinline__ void ShortRows(const FusedArgs& a, SortedShared& sh, uint32_t start, uint32_t end,
                                          uint32_t log2g, uint32_t window_bits, uint32_t vb, uint32_t step, bool write,
                                          RowStats& st) {
  const uint32_t G = kGeneric ? kWave : (1u << log2g);
  const uint32_t lig = threadIdx.x & (G - 1);
  const uint32_t gid = threadIdx.x / G, ngroups = kBlock / G;
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const float* safe = reinterpret_cast<const float*>(a.ctrl);
  const uint32_t window = 1u << window_bits, windows = (end - start + window - 1) >> window_bits;
  for (; vb < windows; vb += step) {
    const uint32_t p0 = start + (vb << window_bits);
    const uint32_t p1 = min(p0 + window, end);
    // Head positions of this window, in order.
    const uint32_t p = p0 + threadIdx.x;
    const bool head = threadIdx.x < window && p < p1 && (p == start || a.keys[p] != a.keys[p - 1]);
    const uint64_t ballot = __ballot(head);
    if (lane == 0) sh.wave_heads[wave] = uint32_t(__popcll(ballot));
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; ++w) before += sh.wave_heads[w];
    const uint32_t nheads = sh.wave_heads[0] + sh.wave_heads[1] + sh.wave_heads[2] + sh.wave_heads[3];
    if (head) sh.heads[before + uint32_t(__popcll(ballot & ((1ull << lane) - 1)))] = p;
    __syncthreads();
    for (uint32_t h = gid; h < nheads; h += ngroups) {
      const uint32_t sb = sh.heads[h];
      uint32_t se;
      if (h + 1 < nheads) {
        se = sh.heads[h + 1];
      } else {  // the window's last row: it may go on past the window
        const uint32_t key = a.keys[sb];
        if (sb + kBlockRowRefs < end && a.keys[sb + kBlockRowRefs] == key) continue;
        se = SegmentEndSearch(a.keys, p1, min(end, sb + kBlockRowRefs), key);
      }
      const uint32_t cnt = se - sb;
      if (cnt > kBlockRowRefs) continue;  // (LongRows)
      const SortedRow row = RowAt<kReduce>(a, sh, sb);
      const TableDesc& T = sh.t[min(row.kp.table, a.tables - 1)];
      const uint32_t dim = T.dim;
      const SortedRefs refs{a.rs + sb, sh.grad, sh.rows, safe, a.features, dim};
      bool ok = row.ok;
      if (!kGeneric) {
        const uint32_t c = lig * 4;
        const bool active = c < dim;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t base = 0; base < cnt; base += G) {
          const uint32_t here = min(G, cnt - base);
          const uint64_t my = lig < here ? refs.Load(base + lig) : 0ull;
          for (uint32_t k = 0; k < here; k += 4) {
            float4 x[4];
            float s[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
              const uint64_t w = __shfl(my, int(k + q), int(G));
              bool in = true;
              const float* src = refs.Source(w, active ? c : 0u, s[q], in);
              const bool mine = k + q < here;
              if (mine && !in) ok = false;
              x[q] = mine && active ? Load4(src) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
              if (k + q < here) Accumulate4(acc, x[q], s[q]);
          }
        }
        if (!ok) st.err |= EPS_HIP_STATUS_BAD_INDEX;
        if (!active || !ok) continue;
        if (kReduce) {
          if (!(Finite(acc.x) && Finite(acc.y) && Finite(acc.z) && Finite(acc.w)))
            st.err |= EPS_HIP_STATUS_REDUCE_OVERFLOW;
          Store4(a.reduce_out + row.u * a.reduce_stride + c, acc);
        } else {
          AdamRow4(T, row.kp.slot, c, acc, write, st);
        }
      } else {
        // Lane l decodes reference l; the others take it from there.
        static_assert(kBlockRowRefs <= kWave, "a reference a lane");
        const uint32_t count = __builtin_amdgcn_readfirstlane(cnt);
        float scale = 0.f;
        bool in = true;
        uint64_t src = 0;
        if (lane < count) src = reinterpret_cast<uint64_t>(refs.Source(refs.Load(lane), 0, scale, in));
        if (__ballot(!in)) ok = false;
        auto source = [&](uint32_t k) {
          const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(src), k);
          const uint32_t hi = __builtin_amdgcn_readlane(uint32_t(src >> 32), k);
          return reinterpret_cast<const float*>(lo | (uint64_t(hi) << 32));
        };
        auto scale_of = [&](uint32_t k) {
          return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(scale), k));
        };
        if (!ok) {
          st.err |= EPS_HIP_STATUS_BAD_INDEX;
          continue;
        }
        for (uint32_t c = lane; c < dim; c += kWave) {
          float acc = 0.f;
          uint32_t k = 0;
          for (; k + 4 <= count; k += 4) {
            float x[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) x[q] = LoadF(source(k + q) + c);
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) acc = acc + x[q] * scale_of(k + q);
          }
          for (; k < count; ++k) acc = acc + LoadF(source(k) + c) * scale_of(k);
          if (kReduce) {
            if (!Finite(acc)) st.err |= EPS_HIP_STATUS_REDUCE_OVERFLOW;
            a.reduce_out[row.u * a.reduce_stride + c] = acc;
          } else {
            AdamRow1(T, row.kp.slot, c, acc, write, st);
          }
        }
      }
    }
    __syncthreads();
  }
}

// The rows of more than kBlockRowRefs references whose first position lies in
// the windows of 2^long_bits positions (at most kBlock) that blocks vb, vb +
// step, ... of the positions [start, end) own, one after another, each by the
// whole block (a unit of its columns).  False when there is none: nothing was
// staged then.
template <bool kReduce>
__device__ __forceinline__ bool LongRows(const FusedArgs& a, SortedShared& sh, LongRowShared& lsh, bool staged,
                                         uint32_t start, uint32_t end, uint32_t vb, uint32_t step, bool write,
                                         RowStats& st) {
  const float* safe = reinterpret_cast<const float*>(a.ctrl);
  const uint32_t window = 1u << a.long_bits, windows = (end - start + window - 1) >> a.long_bits;
  bool found = false;
  if (threadIdx.x == 0) lsh.count[0] = lsh.bad = 0;
  __syncthreads();
  // (The counts go round three words, so that no thread still reads the one
  // that another clears.)
  for (uint32_t i = 0; vb < windows * a.long_slices; vb += step, i = i == 2 ? 0 : i + 1) {
    const uint32_t slice = vb / windows, c0 = slice * kLongColumns;
    const uint32_t p = start + ((vb - slice * windows) << a.long_bits) + threadIdx.x;
    if (threadIdx.x < window && p + kBlockRowRefs < end) {
      const uint32_t key = a.keys[p], ahead = a.keys[p + kBlockRowRefs], before = p == start ? ~key : a.keys[p - 1];
      if (key == ahead && key != before) lsh.heads[atomicAdd(&lsh.count[i], 1u)] = p;
    }
    if (threadIdx.x == 0) lsh.count[i == 2 ? 0 : i + 1] = 0;
    __syncthreads();
    const uint32_t rows = lsh.count[i];
    if (rows && !found && !staged) {
      StageSorted(a, sh);
      __syncthreads();
    }
    found = found || rows;
    for (uint32_t h = 0; h < rows; ++h) {
      const uint32_t sb = lsh.heads[h], se = SegmentEndSearch(a.keys, sb + kBlockRowRefs + 1, end, a.keys[sb]);
      const SortedRow row = RowAt<kReduce>(a, sh, sb);
      const TableDesc& T = sh.t[min(row.kp.table, a.tables - 1)];
      const SortedRefs refs{a.rs + sb, sh.grad, sh.rows, safe, a.features, T.dim};
      if (c0 >= T.dim) continue;  // uniform
      // (Vector classes load 16 bytes wherever their gradients lie, as their own kernels do.)
      bool ok = row.ok;
      const float acc = T.dim % 4 == 0 && (T.dim <= 256 || a.wide)
                            ? BlockRowSum<true>(lsh.sum, refs, se - sb, T.dim, c0, 0.f, ok)
                            : BlockRowSum<false>(lsh.sum, refs, se - sb, T.dim, c0, 0.f, ok);
      if (!ok) lsh.bad = 1;
      __syncthreads();
      ok = lsh.bad == 0;
      __syncthreads();
      if (threadIdx.x == 0) lsh.bad = 0;
      if (!ok) st.err |= EPS_HIP_STATUS_BAD_INDEX;
      const uint32_t c = c0 + threadIdx.x;
      if (threadIdx.x >= kLongColumns || c >= T.dim || !ok) continue;
      if (kReduce) {
        if (!Finite(acc)) st.err |= EPS_HIP_STATUS_REDUCE_OVERFLOW;
        a.reduce_out[row.u * a.reduce_stride + c] = acc;
      } else {
        AdamRow1(T, row.kp.slot, c, acc, write, st);
      }
    }
  }
  return found;
}

// The sorted positions of classes [first, last), from the workspace, kept
// inside the push's.
__device__ __forceinline__ uint2 ClassRange(const FusedArgs& a, uint32_t first, uint32_t last) {
  const uint32_t begin = a.ctrl->class_start[first], stop = a.ctrl->class_start[last];
  const uint32_t end = min(stop, a.n);
  return make_uint2(min(begin, end), end);
}

// Which rows a launch of the sorted driver takes.  Long rows need 40 KB of LDS
// and about 140 registers, three blocks a CU; rows of a few references are a
// chain of memory latencies, and want more of them.  So the rows of more than
// kBothBlocks windows, whose blocks would wait for room, are taken by two
// launches: 43,000 uniform references on each of 26 tables of dim 64 reduced,
// 422 us with both in one, 275 apart; 200,000 of dim 300 pushed, 909 and 425
// (20,000 of dim 50, 2,500 windows, 33 and 28).  Fewer take one, and save a
// launch: 400 or 4,000 references of dim 50, 15 us and 18 apart.  The two do
// not overlap, which costs skewed ids what the long rows took beside the short
// ones (43,000 of dim 10, Zipf of 1.05, 75 -> 87).
enum SortedPart : uint32_t { kShortPart = 1, kLongPart = 2, kBothParts = 3 };

// Adam of the generic class (one wavefront per row, scalar columns), and the
// checked apply of every class.
template <uint32_t kPart>
__device__ __forceinline__ void SortedUpdate(const FusedArgs& a) {
  // The checked apply nearly always has nothing to do.
  if (a.role == kFallback && a.ctrl->mode != kChecked) return;
  __shared__ SortedShared sh;
  Control* ctrl = a.ctrl;
  const GuardInputs in = LoadGuard(ctrl);
  if (kPart & kShortPart) StageSorted(a, sh);
  bool write = true;
  if (!LaunchGate(ctrl, in, sh.t, a.gs, a.role, &sh.mode, write)) return;
  const uint2 range = ClassRange(a, a.cls, a.cls_end);
  RowStats st;
  __syncthreads();
  if constexpr (kPart & kShortPart)
    ShortRows<true, false>(a, sh, range.x, range.y, 6, a.window_bits[kClasses - 1], blockIdx.x, gridDim.x, write, st);
  if constexpr (kPart & kLongPart) {
    __shared__ LongRowShared lsh;
    const bool found = LongRows<false>(a, sh, lsh, kPart & kShortPart, range.x, range.y, blockIdx.x, gridDim.x, write,
                                       st);
    if (!found && !(kPart & kShortPart)) return;
  }
  FinishBlock(st, ctrl, a.bounds, write);
}
__global__ void __launch_bounds__(kBlock) SortedUpdateKernel(FusedArgs a) { SortedUpdate<kShortPart>(a); }
__global__ void __launch_bounds__(kBlock) LongUpdateKernel(FusedArgs a) { SortedUpdate<kLongPart>(a); }
__global__ void __launch_bounds__(kBlock) SortedLongUpdateKernel(FusedArgs a) { SortedUpdate<kBothParts>(a); }

// Reduced gradients of every class in one launch: the short rows of class c
// have the blocks [class_block[c], class_block[c + 1]), the long rows of every
// class all of them.
template <uint32_t kPart>
__device__ __forceinline__ void SortedReduce(const FusedArgs& a) {
  __shared__ SortedShared sh;
  Control* ctrl = a.ctrl;
  RowStats st;
  if constexpr (kPart & kShortPart) {
    StageSorted(a, sh);
    uint32_t cls = 0;
#pragma unroll
    for (uint32_t c = 1; c < kClasses; ++c) cls += blockIdx.x >= a.class_block[c];
    const uint2 range = ClassRange(a, cls, cls + 1);
    const uint32_t block = blockIdx.x - a.class_block[cls], grid = a.class_block[cls + 1] - a.class_block[cls];
    __syncthreads();
    if (cls + 1 == kClasses)
      ShortRows<true, true>(a, sh, range.x, range.y, 6, a.window_bits[cls], block, grid, false, st);
    else
      ShortRows<false, true>(a, sh, range.x, range.y, cls + 2, a.window_bits[cls], block, grid, false, st);
  }
  if constexpr (kPart & kLongPart) {
    __shared__ LongRowShared lsh;
    const uint2 range = ClassRange(a, 0, kClasses);
    const bool found = LongRows<true>(a, sh, lsh, kPart & kShortPart, range.x, range.y, blockIdx.x, gridDim.x, false,
                                      st);
    if (!found && !(kPart & kShortPart)) return;
  }
  FinishBlock(st, ctrl, nullptr, false);
}
__global__ void __launch_bounds__(kBlock) SortedReduceKernel(FusedArgs a) { SortedReduce<kShortPart>(a); }
__global__ void __launch_bounds__(kBlock) LongReduceKernel(FusedArgs a) { SortedReduce<kLongPart>(a); }
__global__ void __launch_bounds__(kBlock) SortedLongReduceKernel(FusedArgs a) { SortedReduce<kBothParts>(a); }

// ---------------------------------------------------------------------------
// Vector-class update (dim % 4 == 0, dim <= 256).  Two kernels:
//
//  * HotSliceKernel: rows with more than kLongRefs references (listed at
//    prepare time).  Work unit = (hot row, kSlice-column slice); a block
//    works through a stream of units chunk by chunk (64 references; 256 for
//    16-column units, so a chunk's tile holds the same 4,096 products).
//    Wave 0 adds: lane c < kSlice owns column col0 + c, adds the chunk's
//    products in reference order (one dependent add per reference) and
//    applies Adam after the unit's last chunk.  Waves 1..kProducers produce:
//    producer p loads the gradient rows of every kProducers-th chunk (16
//    contiguous bytes per lane), multiplies them by their scales and stores
//    the products into one of kHotRing LDS tiles [column][reference], with
//    the unit's w, m, v when the chunk is its last.  Tiles change hands
//    through two LDS counters per tile (staged / added), so the waves never
//    meet at a block barrier, and each producer keeps two chunks of rows in
//    flight (one of the longer 16-column chunks).  For very long rows the slices are narrow (32 columns) so that a
//    hot row's chain data spreads over several CUs: a block's producers then
//    move half of a 64-column chunk's bytes through their CU per chunk, and
//    the adding wave's serial chain, not the CU's memory pipeline, sets the
//    rate; a 32-column slice of a reference is one whole 128-byte line, so
//    no line is fetched for part of its bytes.  Small pushes with very long
//    rows (their gradient rows stay in the caches) take 16-column slices.
//  * RowRunKernel: every other row.  A block owns a window of sorted
//    positions (RunPositions: 256, or 128 / 64 for 32- / 64-lane groups, so
//    every group has a few rows per window whatever the width); it stages
//    their keys and reference words (plus kLongRefs positions of look-ahead)
//    in LDS with coalesced loads, finds the segment heads with a ballot, and a
//    group of G = dim/4 lanes per row (lane = 4 columns) loads the row's w, m,
//    v together with its gradient rows, sums them in order and applies Adam.
constexpr uint32_t kHotBlock = 256;                       // threads of a hot-row block
constexpr uint32_t kHotRing = 4;                          // chunks staged in LDS per block
constexpr uint32_t kUnitCache = 512;                      // unit headers a block stages in LDS
// Shape of a hot-row unit of kS columns (16, 32 or 64) in chunks of kC
// references (kS * kC = 4,096 or fewer products a tile): lanes per reference
// in a producer's row load, references per row load, row loads per producer
// lane per chunk, reference words per producer lane per chunk, floats per
// tile row (one column), and the parts the adding wave reads a tile in (of
// kPart references: 32 for 16-column units, whose 256-reference chunks would
// otherwise need more registers than the kernel has, 64 for the others).
template <uint32_t kS, uint32_t kC>
struct HotShape {
  static constexpr uint32_t kQuads = kS / 4;
  static constexpr uint32_t kRefsPerLoad = kWave / kQuads;
  static constexpr uint32_t kLoads = kC / kRefsPerLoad;
  static constexpr uint32_t kWords = kC / kWave;
  static constexpr uint32_t kPitch = kC + 4;
  static constexpr uint32_t kPart = kS < 32 ? kWave / 2 : kWave;
  // Own chunks each producer keeps in flight: two (four measured no faster,
  // and for the HBM-bound chains of 4 x 8.4 M references three or four made
  // the step 9.8 -> 11.3-11.7 ms), one for 16-column units, whose chunks of
  // 256 references keep as many bytes in flight and leave the registers for
  // their longer reference lists.
  static constexpr uint32_t kDepth = kS < 32 ? 1 : 2;
  static constexpr uint32_t kParts = kC / kPart;
  static_assert(kC % kWave == 0 && kS <= kWave && kWave % kQuads == 0 && kLoads % 4 == 0 &&
                    kLoads <= 16 && kS * kC <= kWave * kWave,
                "hot-row tile shape");
};
constexpr uint32_t kProducers = kHotBlock / kWave - 1;

// Sorted positions per row-run window for groups of 2^log2g lanes: about 5
// rows per group at the usual ~3 references per row.  Wider groups take
// narrower windows, so a class of wide rows still spreads over many blocks.
// (RunWindowBits, below: the windows of a push too small to fill the chip.)
constexpr uint32_t RunPositions(uint32_t log2g) { return log2g <= 4 ? 256u : (log2g == 5 ? 128u : 64u); }
constexpr uint32_t kRunPositions = RunPositions(2);  // the widest window
static_assert(kRunPositions <= kBlock, "one thread per staged position finds the row heads");
constexpr uint32_t kRefBatch = 4;                       // gradient rows in flight per group

struct VecArgs {
  TableDesc t[EPS_HIP_MAX_TABLES];   // by key index
  const float* grad[EPS_HIP_MAX_FEATURES];
  uint64_t grad_rows[EPS_HIP_MAX_FEATURES];
  const uint32_t* keys;
  const uint64_t* rs;
  const HotEntry* hot;
  Control* ctrl;
  Bounds* bounds;
  GuardScalars gs;
  uint32_t row_bits, cls, role, slice_bits, hot_capacity, tables, features;
  uint32_t n;           // sorted positions of the push (hot-row entries are clamped to them)
  uint32_t spin_limit;  // polls of a hot-row hand-over wait (0: give up at once)
  uint32_t class_block[kClasses], class_grid[kClasses];  // RowRunClassesKernel's blocks per class
  uint32_t window_bits[kClasses];                        // log2 of each class's row-run window
};
static_assert(sizeof(VecArgs) <= 4096, "update arguments fit the kernel-argument segment");

// Position of (column c, reference r) in a hot-row tile of kPitch floats a
// column.  Groups of four references are rotated by the column's 16-column
// group (XOR; the identity for slices of 16 columns), so a producer's stores
// of one row load hit distinct banks, and the adding wave's 16-byte reads of
// four consecutive references stay aligned.
template <uint32_t kPitch>
__device__ __forceinline__ uint32_t TileAt(uint32_t c, uint32_t r) {
  return c * kPitch + 4u * ((r >> 2) ^ (c >> 4)) + (r & 3u);
}

__device__ __forceinline__ const float* RefSource(const float* const* grad, uint64_t word,
                                                  uint32_t dim, uint32_t col, float& scale) {
  const uint32_t ref = uint32_t(word);
  scale = __uint_as_float(uint32_t(word >> 32));
  return grad[ref >> kRefRowBits] + uint64_t(ref & ((1u << kRefRowBits) - 1)) * dim + col;
}

// Copies the per-launch tables to LDS and decides whether this launch writes;
// returns false when it has nothing to do (uniform over the block).
template <uint32_t kThreads = kBlock>
__device__ __forceinline__ bool VecPrologue(const VecArgs& a, TableDesc* s_t, const float** s_grad,
                                            uint32_t* s_mode, bool& write, uint64_t* s_rows) {
  const GuardInputs in = LoadGuard(a.ctrl);
  CopyWords<kThreads>(s_t, a.t, a.tables * uint32_t(sizeof(TableDesc)));
  CopyWords<kThreads>(s_grad, a.grad, a.features * uint32_t(sizeof(a.grad[0])));
  CopyWords<kThreads>(s_rows, a.grad_rows, a.features * uint32_t(sizeof(a.grad_rows[0])));
  return LaunchGate(a.ctrl, in, s_t, a.gs, a.role, s_mode, write);
}

// One chunk of a hot work unit: positions [cbase, cbase + chunk) of the
// row whose references are the sorted positions [start, end), for the kSlice
// columns from col0.  `ok` is false past the stream's last unit.  Every field
// is the same in all lanes of a wavefront.
struct HotSlot {
  uint32_t start, end, key, col0, cbase;
  bool ok;
};

// A producer's loads of one chunk in flight.  Row load k brings columns
// 4*quad .. 4*quad+3 of reference kHotRefsPerLoad*k + sub, with its scale;
// wmv is lane l's column of the unit's w, m, v (used when the chunk ends its
// unit).
template <uint32_t kS, uint32_t kC>
struct HotRows {
  HotSlot c;
  float4 x[HotShape<kS, kC>::kLoads];
  float s[HotShape<kS, kC>::kLoads];
  float wmv[3];
};

// A producer's row pointers and scales of one chunk, staged in LDS in the
// order the row loads use them: entry [sub][k] is reference
// kHotRefsPerLoad*k + sub, so a lane reads its kHotLoads pointers and scales
// with a few 16-byte reads.
template <uint32_t kS, uint32_t kC>
struct HotRefs {
  const float* src[HotShape<kS, kC>::kRefsPerLoad][HotShape<kS, kC>::kLoads];
  float scale[HotShape<kS, kC>::kRefsPerLoad][HotShape<kS, kC>::kLoads];
};

// s_waitcnt operand that waits for LDS (and scalar memory) accesses only:
// vmcnt and expcnt at their maxima, lgkmcnt 0.
constexpr int kLgkmZero = 0xC07F;

// Waits until the LDS counter reaches `target` (all lanes read the same word).
// Returns false on a timeout: a wait that has not been satisfied after `limit`
// polls marks the push failed and stops waiting, so a block always finishes
// (limit 0: every wait times out at once, the host-driven test of that path).
__device__ __forceinline__ bool WaitCounter(const uint32_t* counter, uint32_t target, uint32_t sleep,
                                            uint32_t limit) {
  if (limit == 0) return false;
  for (uint32_t spins = 0;; ++spins) {
    const uint32_t v = uint32_t(__builtin_amdgcn_readfirstlane(
        int(__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))));
    if (v >= target) break;
    if (spins >= limit) return false;
    if (sleep) __builtin_amdgcn_s_sleep(1);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  return true;
}

// Publishes `value` after this wave's earlier LDS accesses.
__device__ __forceinline__ void PostCounter(uint32_t* counter, uint32_t value) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if ((threadIdx.x & (kWave - 1)) == 0)
    __hip_atomic_store(counter, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

constexpr uint32_t kLongDepth = 2;  // own chunks of rows a producer of a long unit keeps in flight (even)

// One unit on a block of its own: the kS columns from col0 of a row of very
// many references.  There is no stream to walk, and a chunk is always 4,096
// products, so the adding wave is held up once per 4,096 / kS references.
// Each producer has a tile of its own ([reference][column], which it writes
// with 16-byte stores as the rows arrive), two own chunks of rows in flight
// and the reference words of a third; the adding wave reads a tile a part of
// 64 references at a time into one register buffer while it adds the other.
// What bounds it is the adding wave's instruction rate (about one per six
// cycles, whatever their kind): an add and half an LDS read a reference.  4 x
// 8.4 M references, the hottest rows 977,000: 7.4 ns a reference in 64-reference
// chunks with the stream walked between them (hot-row kernel 7.1 ms), 5.7 so
// (5.6 ms; with one chunk of rows in flight 10, 9.8 ms).
template <uint32_t kS>
struct LongShape {
  static constexpr uint32_t kChunk = 4096 / kS;            // references of a chunk
  static constexpr uint32_t kQuads = kS / 4;
  static constexpr uint32_t kRefsPerLoad = kWave / kQuads;
  static constexpr uint32_t kLoads = kChunk / kRefsPerLoad;  // row loads of a producer lane per chunk
  static constexpr uint32_t kParts = kChunk / kWave;
  static constexpr uint32_t kWords = kChunk / kWave;  // reference words of a producer lane per chunk
  static_assert(kLoads == 16 && kParts % 2 == 0, "long unit shape");
};
template <uint32_t kS>
struct LongShared {
  __align__(16) float tile[kProducers][4096];
  // A producer's decoded references: entry [sub][i] is what its row load i
  // brings to the lanes of `sub`.
  const float* src[kProducers][LongShape<kS>::kRefsPerLoad][LongShape<kS>::kLoads];
  float scale[kProducers][LongShape<kS>::kRefsPerLoad][LongShape<kS>::kLoads];
  uint32_t ready[kProducers], used[kProducers];
};

template <uint32_t kS>
__device__ void LongUnit(const VecArgs& a, LongShared<kS>& sh, const TableDesc* s_t, const float* const* s_grad,
                         const uint64_t* s_rows, uint32_t* s_bad, uint32_t start, uint32_t end, uint32_t key,
                         uint32_t col0, bool write, RowStats& st) {
  using Shape = LongShape<kS>;
  constexpr uint32_t kChunk = Shape::kChunk;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave)));
  start = __builtin_amdgcn_readfirstlane(start);
  end = __builtin_amdgcn_readfirstlane(end);
  const KeyParts kp = SplitKey(__builtin_amdgcn_readfirstlane(key), a.row_bits);
  const TableDesc& T = s_t[min(kp.table, a.tables - 1)];
  const bool key_ok = KeyInRange(kp, a.tables, T.rows);
  const uint32_t dim = T.dim;
  const uint32_t chunks = (end - start + kChunk - 1) / kChunk;
  const float* idle = reinterpret_cast<const float*>(a.rs);
  bool stalled = false;
  if (wave == 0) {
    __builtin_amdgcn_s_setprio(2);
    const uint32_t c = lane % kS;
    const bool mine = lane < kS && col0 + c < dim;
    float* row = T.state + uint64_t(key_ok ? kp.slot : 0u) * dim * 3 + (mine ? col0 + c : 0u);
    float w = 0.f, m = 0.f, v = 0.f;
    if (key_ok) { w = LoadF(row); m = LoadF(row + dim); v = LoadF(row + 2 * dim); }
    float acc = 0.f;
    float xa[kWave], xb[kWave];
    // Part h of tile t: rows kStep apart lie 256 bytes apart, so that a pair of
    // them is one LDS access; one address a residue (opaque to the compiler,
    // which would pair neighbours and take an address for each eight rows).
    constexpr uint32_t kStep = kWave / kS;
    uint32_t at[kStep];
#pragma unroll
    for (uint32_t k = 0; k < kStep; ++k) {
      at[k] = k * kS + c;
      if constexpr (kStep > 1) asm volatile("" : "+v"(at[k]));
    }
    auto read = [&](uint32_t t, uint32_t h, uint32_t r) {
      return (&sh.tile[0][0])[at[r % kStep] + t * 4096 + h * (kWave * kS) + r / kStep * kWave];
    };
    // Chunk j lies in tile j % kProducers, whose number is a constant of the
    // unrolled loop.  uses = j / kProducers + 1.
    auto add_chunk = [&](uint32_t t, uint32_t j, uint32_t uses) {
      const uint32_t next = (t + 1) % kProducers, next_uses = t + 1 == kProducers ? uses + 1 : uses;
      uint32_t peek = 0;
#pragma unroll
      for (uint32_t h = 0; h < Shape::kParts; ++h) {
        float* cur = h % 2 ? xb : xa;
        float* nxt = h % 2 ? xa : xb;
        const bool last = h + 1 == Shape::kParts;
        // The part to add has arrived before the next part's reads go out.
        __builtin_amdgcn_s_waitcnt(kLgkmZero);
        __builtin_amdgcn_sched_barrier(0);
        if (last) {
          if (j + 1 < chunks && uint32_t(__builtin_amdgcn_readfirstlane(int(peek))) < next_uses &&
              !WaitCounter(&sh.ready[next], next_uses, 0, a.spin_limit)) {
            stalled = true;
            return;
          }
          // Every value of this tile is in registers: its producer may have it
          // back.  (A part past the last chunk is read all the same, from a
          // tile in LDS, and dropped.  The LDS accesses of one wavefront are
          // performed in order: the fence only holds the compiler.)
          if (lane == 0)
            __hip_atomic_store(&sh.used[t], uses, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        } else if (h + 2 == Shape::kParts) {
          // The next chunk's readiness is read along with the last part.
          peek = __hip_atomic_load(&sh.ready[next], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        __builtin_amdgcn_sched_barrier(0);
        // The next part's reads go out among the adds, two rows a read.
#pragma unroll
        for (uint32_t r = 0; r < kWave; r += 2 * kStep) {
#pragma unroll
          for (uint32_t k = r; k < r + 2 * kStep; ++k) nxt[k] = last ? read(next, 0, k) : read(t, h + 1, k);
#pragma unroll
          for (uint32_t k = r; k < r + 2 * kStep; ++k) acc = acc + cur[k];
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("" : "+v"(acc));
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (!WaitCounter(&sh.ready[0], 1, 0, a.spin_limit)) {
      stalled = true;
    } else {
#pragma unroll
      for (uint32_t r = 0; r < kWave; ++r) xa[r] = read(0, 0, r);
    }
    for (uint32_t j = 0, uses = 1; j < chunks && !stalled; j += kProducers, ++uses) {
#pragma unroll
      for (uint32_t t = 0; t < kProducers; ++t)
        if (j + t < chunks && !stalled) add_chunk(t, j + t, uses);
    }
    if (!key_ok) *s_bad = 1;
    if (mine && key_ok && !stalled) {
      AdamElement(T, acc, w, m, v, st);
      if (write && !*s_bad) {
        StoreF(row, w); StoreF(row + dim, m); StoreF(row + 2 * dim, v);
      }
    }
  } else {
    const uint32_t p = wave - 1;
    const uint32_t quad = lane % Shape::kQuads, sub = lane / Shape::kQuads;
    // Lanes whose columns lie past the row's dimension read the slice's first.
    const uint32_t at = col0 + 4 * quad < dim ? 4 * quad : 0u;
    float4 x[kLongDepth][Shape::kLoads];
    float scale[kLongDepth][Shape::kLoads];
    uint64_t word[2][Shape::kWords];  // lane l: references l, l + 64, ... of a chunk
    float* tile = sh.tile[p] + sub * kS + 4 * quad;
    // Own chunk k is chunk p + kProducers * k; past the row's end its words are
    // the row's last, its products -0.0f (the identity of addition).
    auto first_of = [&](uint32_t k) { return start + (p + kProducers * k) * kChunk; };  // (positions stay below 2^30)
    auto load_words = [&](uint32_t k, uint64_t (&w)[Shape::kWords]) {
#pragma unroll
      for (uint32_t i = 0; i < Shape::kWords; ++i) w[i] = a.rs[min(first_of(k) + kWave * i + lane, end - 1)];
    };
    auto decode = [&](const uint64_t (&w)[Shape::kWords]) {
#pragma unroll
      for (uint32_t i = 0; i < Shape::kWords; ++i) {
        const uint32_t r = kWave * i + lane;
        const RefParts rp = SplitRef(w[i]);
        const uint32_t f = min(rp.feature, a.features - 1);
        const bool ok = RefInRange(rp, a.features, s_rows[f]);
        if (!ok) *s_bad = 1;
        sh.src[p][r % Shape::kRefsPerLoad][r / Shape::kRefsPerLoad] =
            ok ? s_grad[f] + uint64_t(rp.row) * dim + col0 : idle;
        sh.scale[p][r % Shape::kRefsPerLoad][r / Shape::kRefsPerLoad] = __uint_as_float(uint32_t(w[i] >> 32));
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    auto load_rows = [&](float4 (&xr)[Shape::kLoads], float (&sr)[Shape::kLoads]) {
#pragma unroll
      for (uint32_t i = 0; i < Shape::kLoads; ++i) xr[i] = Load4(sh.src[p][sub][i] + at);
#pragma unroll
      for (uint32_t i = 0; i < Shape::kLoads; ++i) sr[i] = sh.scale[p][sub][i];
    };
    const uint32_t own = chunks > p ? (chunks - p + kProducers - 1) / kProducers : 0u;
    if (own) {
      // Loads return in issue order, so the words of own chunk k + D + 1 go out
      // before the rows of own chunk k + D: decoding them waits for no row.
      load_words(0, word[0]);
#pragma unroll
      for (uint32_t k = 0; k < kLongDepth; ++k) {
        decode(word[k % 2]);
        load_words(k + 1, word[(k + 1) % 2]);
        load_rows(x[k], scale[k]);
      }
      auto stage = [&](uint32_t k, uint32_t slot, uint64_t (&w)[Shape::kWords], uint64_t (&next)[Shape::kWords]) {
        float4(&xr)[Shape::kLoads] = x[slot];
        float(&sr)[Shape::kLoads] = scale[slot];
        if (!stalled && !WaitCounter(&sh.used[p], k, 1, a.spin_limit)) stalled = true;
        if (stalled) return;
        const uint32_t first = first_of(k);
        if (first + kChunk <= end) {
#pragma unroll
          for (uint32_t i = 0; i < Shape::kLoads; ++i)
            *reinterpret_cast<float4*>(tile + i * (Shape::kRefsPerLoad * kS)) =
                make_float4(xr[i].x * sr[i], xr[i].y * sr[i], xr[i].z * sr[i], xr[i].w * sr[i]);
        } else {
#pragma unroll
          for (uint32_t i = 0; i < Shape::kLoads; ++i) {
            const bool in = first + Shape::kRefsPerLoad * i + sub < end;
            *reinterpret_cast<float4*>(tile + i * (Shape::kRefsPerLoad * kS)) =
                make_float4(in ? xr[i].x * sr[i] : -0.f, in ? xr[i].y * sr[i] : -0.f, in ? xr[i].z * sr[i] : -0.f,
                            in ? xr[i].w * sr[i] : -0.f);
          }
        }
        PostCounter(&sh.ready[p], k + 1);
        decode(w);                               // own chunk k + D
        load_words(k + kLongDepth + 1, next);
        load_rows(xr, sr);                       // own chunk k + D
      };
      for (uint32_t k = 0; k < own && !stalled; k += kLongDepth) {
#pragma unroll
        for (uint32_t d = 0; d < kLongDepth; ++d)
          if (k + d < own) stage(k + d, d, word[(d + kLongDepth) % 2], word[(d + kLongDepth + 1) % 2]);
      }
    }
  }
  if (stalled) st.err |= EPS_HIP_STATUS_STALLED;
}

template <uint32_t kSlice, uint32_t kChunk>
__global__ void __launch_bounds__(kHotBlock) __attribute__((amdgpu_waves_per_eu(kSlice == 32 ? 2 : 1)))
HotSliceKernel(VecArgs a) {
  using Shape = HotShape<kSlice, kChunk>;
  constexpr uint32_t kHotQuads = Shape::kQuads;
  constexpr uint32_t kHotRefsPerLoad = Shape::kRefsPerLoad;
  constexpr uint32_t kHotLoads = Shape::kLoads;
  constexpr uint32_t kPitch = Shape::kPitch;
  constexpr uint32_t kPart = Shape::kPart;
  constexpr uint32_t kParts = Shape::kParts;
  constexpr uint32_t kDepth = Shape::kDepth;
  __shared__ TableDesc s_t[EPS_HIP_MAX_TABLES];
  __shared__ const float* s_grad[EPS_HIP_MAX_FEATURES];
  // Pushes with very long rows (narrow units) give the longest a block each.
  constexpr bool kLong = kSlice < kWave;
  struct Tiles { __align__(16) float tile[kHotRing][kSlice * kPitch]; };
  __shared__ union { Tiles t; std::conditional_t<kLong, LongShared<kLong ? kSlice : 32>, uint32_t> lone; } s_tiles;
  auto& s_tile = s_tiles.t.tile;
  __shared__ float s_wmv[kHotRing][3][kSlice];
  __shared__ __align__(16) HotRefs<kSlice, kChunk> s_ref[kProducers];
  // ready[t]: chunks staged in tile t so far; used[t]: chunks added from it.
  __shared__ uint32_t s_ready[kHotRing], s_used[kHotRing];
  __shared__ uint4 s_unit[kUnitCache];  // {start, end, key, col0} of the block's first units
  __shared__ uint32_t s_mode;
  // Set when a hot-row entry, key or reference names nothing of the push (a
  // damaged workspace): the block writes nothing from then on.
  __shared__ uint32_t s_bad;
  __shared__ uint64_t s_rows[EPS_HIP_MAX_FEATURES];  // gradient rows per feature
  bool write = false;
  if (!VecPrologue<kHotBlock>(a, s_t, s_grad, &s_mode, write, s_rows)) return;
  if (threadIdx.x < kHotRing) {
    s_ready[threadIdx.x] = 0;
    s_used[threadIdx.x] = 0;
  }
  if (threadIdx.x == 0) s_bad = 0;
  Control* ctrl = a.ctrl;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave)));
  RowStats st;
  __syncthreads();
  // XCD x takes its hot-row lists: the hot rows of the x-th eighth of the
  // sorted positions, whose gradient rows the row runs of that XCD also read.
  // Work units are (row, slice) in list order, longest rows first.  Units of
  // the first list (rows of 65,536 or more references) each get a block of
  // their own, when there are fewer of them than the XCD has blocks: one such
  // unit can take longer than all the shorter units spread over the other
  // blocks (4 x 8.4 M references: 15,200 chunks vs ~1,800 a block), so its
  // block takes nothing else.  The other units are dealt to the remaining
  // blocks in snake order (round r goes left to right when r is even, right
  // to left when odd), so the per-block totals stay close.
  const uint32_t xcd = blockIdx.x % kXcds;
  const uint32_t xcd_blocks = gridDim.x / kXcds;
  const uint32_t me = blockIdx.x / kXcds;
  const uint32_t slice_mask = (1u << a.slice_bits) - 1;
  uint32_t bucket_end[kHotBuckets];
  uint32_t units = 0;
#pragma unroll
  for (uint32_t b = 0; b < kHotBuckets; ++b) {
    const uint32_t count = uint32_t(__builtin_amdgcn_readfirstlane(int(ctrl->long_count[xcd * kHotBuckets + b])));
    units += min(count, a.hot_capacity) << a.slice_bits;
    bucket_end[b] = units;
  }
  // The block's unit u of round r (units or more: none), and where its
  // hot-row entry lies.
  const uint32_t own = bucket_end[0] < xcd_blocks ? bucket_end[0] : 0u;  // blocks with a unit of their own
  const uint32_t shared = xcd_blocks - own, mine = me - own;
  auto unit_of = [&](uint32_t r) {
    if (me < own) return r == 0 ? me : units;
    return own + r * shared + ((r & 1) ? shared - 1 - mine : mine);
  };
  // An entry's positions, kept inside the push's sorted positions (start < end
  // <= n), so a damaged list can neither read past them nor run unbounded.
  auto sane = [&](uint32_t& start, uint32_t& end) {
    if (start < end && end <= a.n) return true;
    start = min(start, a.n - 1);
    end = min(max(end, start + 1), a.n);
    return false;
  };
  auto entry_of = [&](uint32_t u, uint32_t& col0) {
    uint32_t b = 0;
#pragma unroll
    for (uint32_t k = 0; k + 1 < kHotBuckets; ++k) b += u >= bucket_end[k];
    const uint32_t local = u - (b ? bucket_end[b - 1] : 0u);
    col0 = (local & slice_mask) * kSlice;
    return uint64_t(xcd * kHotBuckets + b) * a.hot_capacity + (local >> a.slice_bits);
  };
  if constexpr (kLong) {
    if (me < own) {
      uint32_t col0;
      HotEntry e = a.hot[entry_of(me, col0)];
      if (!sane(e.start, e.end)) s_bad = 1;
      if (threadIdx.x < kProducers) s_tiles.lone.ready[threadIdx.x] = s_tiles.lone.used[threadIdx.x] = 0;
      __syncthreads();
      if (col0 < s_t[min(e.key >> a.row_bits, a.tables - 1)].dim)
        LongUnit<kSlice>(a, s_tiles.lone, s_t, s_grad, s_rows, &s_bad, e.start, e.end, e.key, col0, write, st);
      __syncthreads();
      if (s_bad) st.err |= EPS_HIP_STATUS_BAD_INDEX;
      FinishBlock<kHotBlock / kWave>(st, ctrl, a.bounds, write);
      return;
    }
  }
  // The headers of the block's first kUnitCache units are staged in LDS once,
  // so walking the stream costs each wave an LDS read per unit.  (A scalar
  // load per unit would stall every wave's next LDS wait until it returns:
  // scalar loads and LDS accesses share one wait counter.)  Later units, if
  // any, are read through the scalar cache.
  for (uint32_t r = threadIdx.x; r < kUnitCache; r += kHotBlock) {
    const uint32_t u = unit_of(r);
    if (u < units) {
      uint32_t col0;
      HotEntry e = a.hot[entry_of(u, col0)];
      if (!sane(e.start, e.end)) s_bad = 1;
      s_unit[r] = make_uint4(e.start, e.end, e.key, col0);
    }
  }
  __syncthreads();
  const auto* hot = reinterpret_cast<const __attribute__((address_space(4))) HotEntry*>(
      reinterpret_cast<uintptr_t>(a.hot));
  // The block's stream of chunks; every wave walks it the same way.
  uint32_t round = 0;
  HotEntry next_entry{0, 0, 0, 0};
  uint32_t next_col0 = 0;
  bool next_ok = false;
  auto fetch = [&]() {  // header of the block's next unit
    const uint32_t r = round++;
    const uint32_t u = unit_of(r);
    next_ok = u < units;  // unit indices grow with the round: past the end stays past
    if (!next_ok) return;
    if (r < kUnitCache) {
      const uint4 e = s_unit[r];
      next_entry = HotEntry{e.x, e.y, e.z, 0u};
      next_col0 = e.w;
      return;
    }
    const auto& e = hot[entry_of(u, next_col0)];
    next_entry = HotEntry{e.start, e.end, e.key, 0u};
    if (!sane(next_entry.start, next_entry.end)) s_bad = 1;
  };
  auto take = [&]() {  // the next unit's first chunk; slices past a row's dimension are skipped
    for (;;) {
      HotSlot t{next_entry.start, next_entry.end, next_entry.key, next_col0, next_entry.start, next_ok};
      const uint32_t dim = uint32_t(__builtin_amdgcn_readfirstlane(
          int(s_t[min(next_entry.key >> a.row_bits, a.tables - 1)].dim)));
      const bool usable = !next_ok || next_col0 < dim;
      fetch();
      if (usable) return t;
    }
  };
  auto after = [&](const HotSlot& c) {  // the chunk that follows c in the stream
    if (c.ok && c.cbase + kChunk < c.end) {
      HotSlot t = c;
      t.cbase += kChunk;
      return t;
    }
    return take();
  };
  // A hand-over wait timed out: this wave stops waiting, staging, adding and
  // writing, and the push reports a failure.
  bool stalled = false;

  if (wave == 0) {
    // The adding wave: chunk j is the (j / kHotRing)-th use of tile j % kHotRing.
    // Chunk j + 1's tile is read while chunk j is added, and the readiness
    // of chunk j + 2 is polled at the same time; scheduling barriers keep the
    // compiler from moving those LDS accesses (or their waits) before the adds.
    __builtin_amdgcn_s_setprio(2);
    fetch();
    HotSlot c = take();          // chunk j
    HotSlot cn = after(c);       // chunk j + 1
    HotSlot cnn = after(cn);     // chunk j + 2
    float acc = 0.f;
    // Part h (references kPart * h onwards) of chunk j's tile into x.  With
    // one part a chunk, lanes past the slice read nothing.  With several,
    // they read a copy of a slice column and drop it: every lane then writes
    // all of x, so no old contents of a buffer stay live from part to part
    // (which would make the compiler copy whole buffers).
    const uint32_t sl = lane % kSlice;
    auto read_part = [&](uint32_t j, uint32_t h, float4* x) {
      const float* tile = s_tile[j % kHotRing];
      if (kParts > 1 || lane < kSlice) {
#pragma unroll
        for (uint32_t g = 0; g < kPart / 4; ++g)
          x[g] = *reinterpret_cast<const float4*>(tile + TileAt<kPitch>(sl, kPart * h + 4 * g));
      }
    };
    auto ready = [&](uint32_t j) {
      if (!stalled && !WaitCounter(&s_ready[j % kHotRing], j / kHotRing + 1, 0, a.spin_limit)) stalled = true;
    };
    // Adds chunk j (chunk c) part by part: part h is in x for even h and in y
    // for odd h, and each part's adds overlap the reads of the next part (of
    // chunk j + 1's first part after the last), which go to the other buffer.
    // So a chunk of an even number of parts starts and ends in x.  The
    // hand-over (tile release, readiness poll, walk to the next chunk) comes
    // once per chunk, whatever its length.  With several parts a chunk, the
    // next tile is read after the stream's last chunk all the same (plain LDS
    // reads, dropped), for the same reason.
    auto add = [&](uint32_t j, float4* x, float4* y) {
      const uint32_t t = j % kHotRing;
      float w = 0.f, m = 0.f, v = 0.f;
      uint32_t peek = 0;
#pragma unroll
      for (uint32_t h = 0; h < kParts; ++h) {
        const float4* cur = h % 2 ? y : x;
        float4* nxt = h % 2 ? x : y;
        // cur arrived during the previous adds.  Wait for it here, before more
        // reads are issued: the LDS counter tracks at most 15 accesses, so a
        // wait placed after the next part's 16 reads would wait for those too.
        __builtin_amdgcn_s_waitcnt(kLgkmZero);
        __builtin_amdgcn_sched_barrier(0);
        if (h + 1 < kParts) {
          read_part(j, h + 1, nxt);
        } else {
          w = s_wmv[t][0][sl];
          m = s_wmv[t][1][sl];
          v = s_wmv[t][2][sl];
          peek = __hip_atomic_load(&s_ready[(j + 2) % kHotRing], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          if (kParts > 1 || cn.ok) read_part(j + 1, 0, nxt);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t g = 0; g < kPart / 4; ++g) {
          acc = acc + cur[g].x;
          acc = acc + cur[g].y;
          acc = acc + cur[g].z;
          acc = acc + cur[g].w;
        }
        // With several parts, each part's sum is taken here: otherwise the
        // compiler sinks every part's adds below the last part's reads, which
        // then holds all the chunk's values in registers at once.
        if constexpr (kParts > 1) asm volatile("" : "+v"(acc));
        __builtin_amdgcn_sched_barrier(0);
      }
      // Tile t is free once chunk j's values and w, m, v are read: they were
      // read before tile j + 1's reads, and a wavefront's LDS accesses are
      // performed in order, so the counter store needs no wait for the reads
      // still in flight (the wavefront-scope fence keeps the compiler from
      // moving the reads after it).
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      if (lane == 0)
        __hip_atomic_store(&s_used[t], j / kHotRing + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __builtin_amdgcn_sched_barrier(0);
      if (c.cbase + kChunk >= c.end) {  // the unit's last chunk
        const KeyParts kp = SplitKey(c.key, a.row_bits);
        const TableDesc& T = s_t[min(kp.table, a.tables - 1)];
        if (!KeyInRange(kp, a.tables, T.rows)) s_bad = 1;
        if (lane < kSlice && c.col0 + lane < T.dim && !stalled) {
          AdamElement(T, acc, w, m, v, st);
          if (write && !s_bad) {
            float* row = T.state + uint64_t(kp.slot) * T.dim * 3 + c.col0 + lane;
            StoreF(row, w); StoreF(row + T.dim, m); StoreF(row + 2 * T.dim, v);
          }
        }
        acc = 0.f;
      }
      // Chunk j + 2 (if any) must be staged before the next call reads it.
      if (cnn.ok && uint32_t(__builtin_amdgcn_readfirstlane(int(peek))) < (j + 2) / kHotRing + 1)
        ready(j + 2);
      else
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      c = cn;
      cn = cnn;
      cnn = after(cnn);
    };
    float4 xa[kPart / 4], xb[kPart / 4];
    if (c.ok) {
      ready(0);
      read_part(0, 0, xa);
      if (cn.ok) ready(1);
    }
    for (uint32_t j = 0; c.ok && !stalled; j += 2) {
      add(j, xa, xb);
      if (!c.ok || stalled) break;
      if constexpr (kParts % 2 == 1)
        add(j + 1, xb, xa);
      else
        add(j + 1, xa, xb);
    }
  } else {
    // Producer p stages chunks p, p + kProducers, ... (its own chunks, counted
    // by o).  At own chunk o it stages rows(o), decodes the words of o + D
    // into its LDS reference slots, loads the words of o + 2D and then the
    // rows of o + D (D = kDepth).  Loads complete in issue order, so each wait
    // waits only for what it needs.  Every chunk issues the same loads, also
    // past the stream's end (then from the start of the reference words, never
    // used), so the number of loads between any two points is fixed.
    const uint32_t p = wave - 1;
    const uint32_t quad = lane % kHotQuads, sub = lane / kHotQuads;
    const float* idle = reinterpret_cast<const float*>(a.rs);
    HotRefs<kSlice, kChunk>& slots = s_ref[p];
    fetch();
    HotSlot cur = take();  // cursor over the stream, at chunk jc
    uint32_t jc = 0, total = cur.ok ? ~0u : 0u;
    auto advance = [&](uint32_t by) {
      for (uint32_t i = 0; i < by; ++i) {
        cur = after(cur);
        ++jc;
        if (!cur.ok && total == ~0u) total = jc;
      }
    };
    // Reference words of one chunk in flight (lane l: references l, l + 64, ...).
    struct Words {
      HotSlot c;
      uint64_t word[Shape::kWords];
    };
    HotSlot dc{};  // chunk whose references are in the LDS slots
    auto load_words = [&](Words& w) {
      w.c = cur;
#pragma unroll
      for (uint32_t k = 0; k < Shape::kWords; ++k) {
        const uint32_t pos = cur.ok ? min(cur.cbase + kWave * k + lane, cur.end - 1) : 0u;  // end <= n (sane)
        w.word[k] = a.rs[pos];
      }
    };
    // Lane l decodes the words of references l, l + 64, ...: their gradient
    // rows (from the slice's first column) and scales.
    auto decode = [&](const Words& w) {
      const HotSlot& wc = w.c;
      dc = wc;
      const TableDesc& T = s_t[min(wc.key >> a.row_bits, a.tables - 1)];
#pragma unroll
      for (uint32_t k = 0; k < Shape::kWords; ++k) {
        const uint32_t r = kWave * k + lane;
        const RefParts rp = SplitRef(w.word[k]);
        const bool ref_ok = RefInRange(rp, a.features, s_rows[min(rp.feature, a.features - 1)]);
        if (wc.ok && !ref_ok) s_bad = 1;
        float scale;
        const float* src = RefSource(s_grad, w.word[k], T.dim, wc.col0, scale);
        slots.src[r % kHotRefsPerLoad][r / kHotRefsPerLoad] = wc.ok && ref_ok ? src : idle;
        slots.scale[r % kHotRefsPerLoad][r / kHotRefsPerLoad] = scale;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    // Lanes whose columns lie past the row's dimension read the slice's first
    // columns; their products are never stored by the adding wave.
    auto load_rows = [&](HotRows<kSlice, kChunk>& r) {
      r.c = dc;
      const KeyParts kp = SplitKey(dc.key, a.row_bits);
      const TableDesc& T = s_t[min(kp.table, a.tables - 1)];
      const bool key_ok = KeyInRange(kp, a.tables, T.rows);
      const uint32_t dim = T.dim;
      const uint32_t off = dc.col0 + 4 * quad < dim ? 4 * quad : 0u;
      const uint32_t step = dc.ok ? off : 0u;
      const float* src[kHotLoads];
#pragma unroll
      for (uint32_t k = 0; k < kHotLoads; k += 2) {
        const uint4 two = *reinterpret_cast<const uint4*>(&slots.src[sub][k]);
        src[k] = reinterpret_cast<const float*>(uint64_t(two.x) | (uint64_t(two.y) << 32));
        src[k + 1] = reinterpret_cast<const float*>(uint64_t(two.z) | (uint64_t(two.w) << 32));
      }
#pragma unroll
      for (uint32_t k = 0; k < kHotLoads; k += 4) {
        const float4 four = *reinterpret_cast<const float4*>(&slots.scale[sub][k]);
        r.s[k] = four.x; r.s[k + 1] = four.y; r.s[k + 2] = four.z; r.s[k + 3] = four.w;
      }
#pragma unroll
      for (uint32_t k = 0; k < kHotLoads; ++k) r.x[k] = Load4(src[k] + step);
      const uint32_t wcol = dc.col0 + (lane < kSlice && dc.col0 + lane < dim ? lane : 0u);
      const float* row = dc.ok && key_ok ? T.state + uint64_t(kp.slot) * dim * 3 + wcol : idle;
      const uint32_t ms = dc.ok && key_ok ? dim : 0u;
      r.wmv[0] = LoadF(row); r.wmv[1] = LoadF(row + ms); r.wmv[2] = LoadF(row + 2 * ms);
    };
    auto stage = [&](const HotRows<kSlice, kChunk>& r, uint32_t j) {
      const uint32_t t = j % kHotRing;
      if (!stalled && !WaitCounter(&s_used[t], j / kHotRing, 1, a.spin_limit)) stalled = true;
      if (stalled) return;  // nothing more is staged
      // Load k brings columns 4*quad .. 4*quad+3 of reference
      // kHotRefsPerLoad*k + sub; each lands at TileAt(column, reference).
      float* tile = s_tile[t];
      if (r.c.cbase + kChunk <= r.c.end) {  // every reference inside the row
#pragma unroll
        for (uint32_t k = 0; k < kHotLoads; ++k) {
          const float sv = r.s[k];
          float* q = tile + TileAt<kPitch>(4 * quad, kHotRefsPerLoad * k + sub);
          q[0] = r.x[k].x * sv;
          q[kPitch] = r.x[k].y * sv;
          q[2 * kPitch] = r.x[k].z * sv;
          q[3 * kPitch] = r.x[k].w * sv;
        }
      } else {  // references past the row's end add -0.0f, the identity
#pragma unroll
        for (uint32_t k = 0; k < kHotLoads; ++k) {
          const bool in = r.c.cbase + kHotRefsPerLoad * k + sub < r.c.end;
          const float sv = r.s[k];
          float* q = tile + TileAt<kPitch>(4 * quad, kHotRefsPerLoad * k + sub);
          q[0] = in ? r.x[k].x * sv : -0.f;
          q[kPitch] = in ? r.x[k].y * sv : -0.f;
          q[2 * kPitch] = in ? r.x[k].z * sv : -0.f;
          q[3 * kPitch] = in ? r.x[k].w * sv : -0.f;
        }
      }
      if (lane < kSlice) {
        s_wmv[t][0][lane] = r.wmv[0];
        s_wmv[t][1][lane] = r.wmv[1];
        s_wmv[t][2][lane] = r.wmv[2];
      }
      PostCounter(&s_ready[t], j / kHotRing + 1);
    };
    // kDepth own chunks of rows and of reference words in flight.  The
    // prologue leaves the loads in the loop's own order (words(D), rows(0),
    // words(D+1), rows(1), ...), so the compiler's load waits inside the loop
    // can be exact.
    HotRows<kSlice, kChunk> rows[kDepth];
    Words words[kDepth];
    advance(p);  // own chunk 0
#pragma unroll
    for (uint32_t k = 0; k < kDepth; ++k) {  // words(0 .. D-1)
      load_words(words[k]);
      advance(kProducers);
    }
#pragma unroll
    for (uint32_t k = 0; k < kDepth; ++k) {  // words(D + k), then rows(k) from the slots of own chunk k
      decode(words[k]);
      load_words(words[k]);
      advance(kProducers);
      load_rows(rows[k]);
    }
    // Own chunk o (chunk j = p + kProducers*o), buffers b = o % D: stage
    // rows(o), decode words(o + D), load words(o + 2D) and rows(o + D).
    // Words and rows both get D own chunks to arrive (the decode needs no
    // wait of its own: its words were issued before the rows the stage
    // waited for).  D own chunks per pass keep the buffers static.
    auto own = [&](HotRows<kSlice, kChunk>& r, Words& w, uint32_t j) {
      stage(r, j);
      decode(w);
      load_words(w);
      advance(kProducers);
      load_rows(r);
    };
    uint32_t j = p;
    for (; j + (kDepth - 1) * kProducers < total; j += kDepth * kProducers) {  // one exit: every part runs
#pragma unroll
      for (uint32_t k = 0; k < kDepth; ++k) own(rows[k], words[k], j + k * kProducers);
    }
#pragma unroll
    for (uint32_t k = 0; k + 1 < kDepth; ++k)
      if (j + k * kProducers < total) stage(rows[k], j + k * kProducers);
  }
  if (stalled) st.err |= EPS_HIP_STATUS_STALLED;
  __syncthreads();
  if (s_bad) st.err |= EPS_HIP_STATUS_BAD_INDEX;
  FinishBlock<kHotBlock / kWave>(st, ctrl, a.bounds, write);
}

// LDS of a row-run block, sized for the widest window.
struct RunShared {
  uint32_t key[kRunPositions + kLongRefs + 1];  // key[i + 1] = key at position p0 + i
  const float* src[kRunPositions + kLongRefs];  // gradient row of position p0 + i
  float scale[kRunPositions + kLongRefs];
  uint32_t heads[kRunPositions];
  uint32_t wave_heads[kBlock / kWave];
  uint32_t next;  // next unclaimed row (head index) of the window
  uint32_t bad;
};

// The rows of a dimension class (groups of 2^kLog2G lanes) at the sorted
// positions `range`, for block `block` of the `grid` blocks the class has, in
// windows of 2^window_bits positions (at most RunPositions(kLog2G)).
template <uint32_t kLog2G>
__device__ __forceinline__ void RowRuns(const VecArgs& a, RunShared& sh, const TableDesc* s_t,
                                        const float* const* s_grad, const uint64_t* s_rows, uint2 range,
                                        uint32_t block, uint32_t grid, uint32_t window_bits, bool write,
                                        RowStats& st) {
  constexpr uint32_t G = 1u << kLog2G;
  constexpr uint32_t ngroups = kBlock / G;
  static_assert(RunPositions(kLog2G) <= kRunPositions, "row-run window fits its LDS");
  const uint32_t window = 1u << window_bits;
  // Safe address for reads a damaged workspace would point elsewhere: the
  // control block and what follows it (far more than a row of 3 x 256 floats).
  const float* safe = reinterpret_cast<const float*>(a.ctrl);
  // The class's sorted positions, from the workspace: kept inside the push's
  // positions, so a damaged workspace cannot send the staging reads past them.
  const uint32_t end = min(range.y, a.n), begin = min(range.x, end);
  const uint32_t row_mask = (1u << a.row_bits) - 1;
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const uint32_t lig = threadIdx.x & (G - 1), gid = threadIdx.x >> kLog2G;
  const uint32_t c = lig * 4;
  // The class's positions are cut into kXcds contiguous ranges, one per XCD
  // (the class's blocks start at a multiple of kXcds and number a multiple of
  // it, and blocks reach the XCDs round robin): the gradient rows a range
  // references then come from a few features and stay in that XCD's L2 for
  // all their references.  Rows that straddle a cut belong to the range
  // holding their first position.
  const uint32_t xcd = block % kXcds, per_xcd = grid / kXcds;
  const uint32_t span = ((end - begin + kXcds - 1) / kXcds + window - 1) >> window_bits << window_bits;
  const uint32_t xbegin = min(begin + xcd * span, end), xend = min(xbegin + span, end);
  for (uint32_t p0 = xbegin + (block / kXcds) * window; p0 < xend; p0 += per_xcd * window) {
    const uint32_t p1 = min(p0 + window, xend);
    const uint32_t lim = min(p1 + kLongRefs, end);
    const uint32_t staged = lim - p0;
    __syncthreads();  // previous iteration's readers are done
    // Stage keys and, per position, the gradient row it references and its
    // scale (one coalesced pass; the table and feature lookups happen here
    // once per position instead of once per lane).
    if (threadIdx.x == 0) {
      sh.key[0] = p0 > begin ? a.keys[p0 - 1] : ~a.keys[p0];
      sh.next = ngroups;
    }
    for (uint32_t i = threadIdx.x; i < staged; i += kBlock) {
      const uint32_t key = a.keys[p0 + i];
      const uint64_t word = a.rs[p0 + i];
      sh.key[i + 1] = key;
      // A key or reference that names no table, slot, feature or gradient row
      // of the push (a damaged workspace) is read from a safe address instead,
      // and the block writes nothing from then on.
      const KeyParts kp = SplitKey(key, a.row_bits);
      const RefParts rp = SplitRef(word);
      const uint32_t ti = min(kp.table, a.tables - 1);
      const uint32_t fi = min(rp.feature, a.features - 1);
      const bool ok = KeyInRange(kp, a.tables, s_t[ti].rows) && RefInRange(rp, a.features, s_rows[fi]);
      float scale;
      const float* src = RefSource(s_grad, word, s_t[ti].dim, 0, scale);
      sh.src[i] = ok ? src : safe;
      sh.scale[i] = scale;
      if (!ok) sh.bad = 1;
    }
    __syncthreads();
    const bool window_ok = sh.bad == 0;
    const bool head = threadIdx.x < p1 - p0 && sh.key[threadIdx.x + 1] != sh.key[threadIdx.x];
    const uint64_t ballot = __ballot(head);
    if (lane == 0) sh.wave_heads[wave] = uint32_t(__popcll(ballot));
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; ++w) before += sh.wave_heads[w];
    uint32_t nheads = 0;
    for (uint32_t w = 0; w < kBlock / kWave; ++w) nheads += sh.wave_heads[w];
    if (head) sh.heads[before + uint32_t(__popcll(ballot & ((1ull << lane) - 1)))] = threadIdx.x;
    __syncthreads();
    // Groups take rows in order from a shared counter (claimed at the top of
    // a row, used at its end), so a group held up by a row with many
    // references does not hold up the rows behind it.
    for (uint32_t h = gid; h < nheads;) {
      uint32_t claim = 0;
      if (lig == 0) claim = atomicAdd(&sh.next, 1u);
      const uint32_t sb = sh.heads[h];
      const uint32_t key = sh.key[sb + 1];
      // Hot rows (more than kLongRefs references) belong to HotSliceKernel.
      if (sb + kLongRefs < staged && sh.key[sb + kLongRefs + 1] == key) {
        h = uint32_t(__shfl(int(claim), 0, int(G)));
        continue;
      }
      uint32_t se = h + 1 < nheads ? sh.heads[h + 1] : p1 - p0;
      while (se < staged && sh.key[se + 1] == key) ++se;
      const TableDesc& T = s_t[min(key >> a.row_bits, a.tables - 1)];
      const uint32_t dim = T.dim;
      const bool active = c < dim;
      const uint32_t cl = active ? c : 0;  // inactive lanes read column 0 and drop it
      float* row = window_ok ? T.state + uint64_t(key & row_mask) * dim * 3 : const_cast<float*>(safe);
      const float4 w0 = Load4Stream(row + cl), m0 = Load4Stream(row + dim + cl),
                   v0 = Load4Stream(row + 2 * dim + cl);
      float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
      // Every slot of a batch loads (slots past the row repeat its last
      // reference, an in-bounds row of the same table); only real references
      // are added, in order.  The first batch is straight-line code so its
      // loads go out together with w, m and v; longer rows loop.
      auto batch = [&](uint32_t j0) {
        float4 x[kRefBatch];
        float s[kRefBatch];
#pragma unroll
        for (uint32_t k = 0; k < kRefBatch; ++k) {
          const uint32_t j = min(j0 + k, se - 1);
          s[k] = sh.scale[j];
          x[k] = Load4(sh.src[j] + cl);
        }
#pragma unroll
        for (uint32_t k = 0; k < kRefBatch; ++k) {
          float4 t = g;
          Accumulate4(t, x[k], s[k]);
          if (j0 + k < se) g = t;
        }
      };
      batch(sb);
      for (uint32_t j0 = sb + kRefBatch; j0 < se; j0 += kRefBatch) batch(j0);
      if (active) {
        float4 w = w0, m = m0, v = v0;
        if (T.bounded) {
          AdamElement<true>(T, g.x, w.x, m.x, v.x, st);
          AdamElement<true>(T, g.y, w.y, m.y, v.y, st);
          AdamElement<true>(T, g.z, w.z, m.z, v.z, st);
          AdamElement<true>(T, g.w, w.w, m.w, v.w, st);
        } else {
          AdamElement<false>(T, g.x, w.x, m.x, v.x, st);
          AdamElement<false>(T, g.y, w.y, m.y, v.y, st);
          AdamElement<false>(T, g.z, w.z, m.z, v.z, st);
          AdamElement<false>(T, g.w, w.w, m.w, v.w, st);
        }
        if (write && window_ok) {
          Store4Stream(row + c, w);
          Store4Stream(row + dim + c, m);
          Store4Stream(row + 2 * dim + c, v);
        }
      }
      h = uint32_t(__shfl(int(claim), 0, int(G)));
    }
  }
}

// Seven waves per SIMD (72 registers) where that needs no spill: more rows'
// loads in flight per CU.
template <uint32_t kLog2G>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kLog2G == 2 || kLog2G == 6 ? 6 : 7)))
RowRunKernel(VecArgs a) {
  __shared__ TableDesc s_t[EPS_HIP_MAX_TABLES];
  __shared__ const float* s_grad[EPS_HIP_MAX_FEATURES];
  __shared__ RunShared sh;
  __shared__ uint32_t s_mode;
  __shared__ uint64_t s_rows[EPS_HIP_MAX_FEATURES];  // gradient rows per feature
  bool write = false;
  const uint2 range = make_uint2(a.ctrl->class_start[a.cls], a.ctrl->class_start[a.cls + 1]);
  if (!VecPrologue(a, s_t, s_grad, &s_mode, write, s_rows)) return;
  RowStats st;
  if (threadIdx.x == 0) sh.bad = 0;
  __syncthreads();
  RowRuns<kLog2G>(a, sh, s_t, s_grad, s_rows, range, blockIdx.x, gridDim.x, a.window_bits[kLog2G - 2], write,
                  st);
  if (sh.bad) st.err |= EPS_HIP_STATUS_BAD_INDEX;
  FinishBlock(st, a.ctrl, a.bounds, write);
}

// Every vector class of a push in one launch: class c has the blocks
// [class_block[c], class_block[c] + class_grid[c]) (starts and counts are
// multiples of kXcds; absent classes have none), so the classes' rows run
// side by side instead of one launch (and its tail) after another.
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6)))
RowRunClassesKernel(VecArgs a) {
  __shared__ TableDesc s_t[EPS_HIP_MAX_TABLES];
  __shared__ const float* s_grad[EPS_HIP_MAX_FEATURES];
  __shared__ RunShared sh;
  __shared__ uint32_t s_mode;
  __shared__ uint64_t s_rows[EPS_HIP_MAX_FEATURES];
  bool write = false;
  uint32_t cls = 0;
#pragma unroll
  for (uint32_t c = 1; c + 1 < kClasses; ++c)
    if (a.class_grid[c] && blockIdx.x >= a.class_block[c]) cls = c;
  const uint2 range = make_uint2(a.ctrl->class_start[cls], a.ctrl->class_start[cls + 1]);
  if (!VecPrologue(a, s_t, s_grad, &s_mode, write, s_rows)) return;
  RowStats st;
  if (threadIdx.x == 0) sh.bad = 0;
  __syncthreads();
  const uint32_t block = blockIdx.x - a.class_block[cls], grid = a.class_grid[cls];
  const uint32_t bits = a.window_bits[cls];
  switch (cls) {
    case 0: RowRuns<2>(a, sh, s_t, s_grad, s_rows, range, block, grid, bits, write, st); break;
    case 1: RowRuns<3>(a, sh, s_t, s_grad, s_rows, range, block, grid, bits, write, st); break;
    case 2: RowRuns<4>(a, sh, s_t, s_grad, s_rows, range, block, grid, bits, write, st); break;
    case 3: RowRuns<5>(a, sh, s_t, s_grad, s_rows, range, block, grid, bits, write, st); break;
    default: RowRuns<6>(a, sh, s_t, s_grad, s_rows, range, block, grid, bits, write, st); break;
  }
  if (sh.bad) st.err |= EPS_HIP_STATUS_BAD_INDEX;
  FinishBlock(st, a.ctrl, a.bounds, write);
}

// ---------------------------------------------------------------------------
// Row driver: explicit unique rows (ApplyHost) or CSR references (ApplyCompact).
// 43,000 references of 14,700 rows of dim 64, the longest 3,787: 751 us with a
// group a row and one reference in flight, 75 so (short rows 14, long rows 60).
struct RowArgs {
  TableDesc t;
  const uint64_t* slots;
  const uint64_t* offsets;   // NULL: row r has exactly gradient row r (ApplyHost)
  const uint64_t* sources;
  const float* scales;
  const float* src;
  uint64_t rows;
  Control* ctrl;
  Bounds* bounds;
  GuardScalars gs;
  uint32_t log2g, vblocks, role, short_refs;
};

template <bool kGeneric>
__global__ void __launch_bounds__(kBlock) RowUpdateKernel(RowArgs a) {
  __shared__ TableDesc s_t[1];
  __shared__ uint32_t s_mode;
  Control* ctrl = a.ctrl;
  const GuardInputs in = LoadGuard(ctrl);
  if (threadIdx.x == 0) s_t[0] = a.t;
  bool write = false;
  if (!LaunchGate(ctrl, in, s_t, a.gs, a.role, &s_mode, write)) return;
  const TableDesc T = a.t;
  const uint32_t dim = T.dim;
  const uint32_t G = kGeneric ? kWave : (1u << a.log2g);
  const uint32_t lig = threadIdx.x & (G - 1);
  const uint32_t gid = threadIdx.x / G, ngroups = kBlock / G;
  RowStats st;
  for (uint32_t vb = blockIdx.x; vb < a.vblocks; vb += gridDim.x) {
    const uint64_t r = uint64_t(vb) * ngroups + gid;
    if (r >= a.rows) continue;
    const uint64_t slot = a.slots[r];
    if (!kGeneric) {
      const uint32_t c = lig * 4;
      const bool active = c < dim;
      const float4 g = active ? Load4(a.src + r * dim + c) : make_float4(0.f, 0.f, 0.f, 0.f);
      if (active) AdamRow4(T, slot, c, g, write, st);
    } else {
      for (uint32_t c = lig; c < dim; c += kWave) AdamRow1(T, slot, c, a.src[r * dim + c], write, st);
    }
  }
  FinishBlock(st, ctrl, a.bounds, write);
}

// Rows of more references than this are summed by a block each.  A large packet
// has groups enough for longer rows (200,000 references in rows of 33, dim 64:
// 25 us with 64, 49 with 32; of 300, 28 both ways), a small one waits for them
// (200 mean bags, dim 128, the longest row 182 references: 25 us with 64, 22
// with 32).
constexpr uint64_t kCsrLargeRefs = 1ull << 16;
constexpr uint32_t CsrShortRefs(uint64_t references) { return references >= kCsrLargeRefs ? 64u : 32u; }
constexpr uint64_t kCsrPiece = 1ull << 30;  // references of one BlockRowSum (it counts in 32 bits)

// CSR rows, a group of 2^log2g lanes a row (kGeneric: a wavefront over scalar
// columns), four gradient rows in flight; rows of more than
// short_refs references are left out when `short_only`.
template <bool kGeneric>
__device__ __forceinline__ void CsrShortRows(const RowArgs& a, bool short_only, bool write, RowStats& st) {
  const TableDesc T = a.t;
  const uint32_t dim = T.dim;
  const uint32_t G = kGeneric ? kWave : (1u << a.log2g);
  const uint32_t lig = threadIdx.x & (G - 1);
  const uint32_t gid = threadIdx.x / G, ngroups = kBlock / G;
  for (uint32_t vb = blockIdx.x; vb < a.vblocks; vb += gridDim.x) {
    const uint64_t r = uint64_t(vb) * ngroups + gid;
    if (r >= a.rows) continue;
    const uint64_t slot = a.slots[r], b = a.offsets[r], e = max(a.offsets[r + 1], b);
    if (short_only && e - b > a.short_refs) continue;  // (CsrTailKernel)
    if (!kGeneric) {
      const uint32_t c = lig * 4;
      const bool active = c < dim;
      float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
      for (uint64_t j = b; j < e; j += 4) {
        float4 x[4];
        float s[4];
        uint64_t source[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
          const bool mine = j + q < e;
          source[q] = mine ? a.sources[j + q] : 0ull;
          s[q] = mine ? a.scales[j + q] : 0.f;
        }
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
          x[q] = j + q < e && active ? Load4(a.src + source[q] * dim + c) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
          if (j + q < e) Accumulate4(g, x[q], s[q]);
      }
      if (active) AdamRow4(T, slot, c, g, write, st);
    } else {
      for (uint32_t c = lig; c < dim; c += kWave) {
        float g = 0.f;
        uint64_t j = b;
        for (; j + 4 <= e; j += 4) {
          float x[4], s[4];
#pragma unroll
          for (uint32_t q = 0; q < 4; ++q) {
            s[q] = a.scales[j + q];
            x[q] = LoadF(a.src + a.sources[j + q] * dim + c);
          }
#pragma unroll
          for (uint32_t q = 0; q < 4; ++q) g = g + x[q] * s[q];
        }
        for (; j < e; ++j) g = g + LoadF(a.src + a.sources[j] * dim + c) * a.scales[j];
        AdamRow1(T, slot, c, g, write, st);
      }
    }
  }
}

// CSR rows of more than short_refs references, a block a unit of columns.  A packet lists its rows in first-occurrence order,
// so its long rows crowd at its start: neighbours (groups of 2^spread_bits of
// them, one in packets of up to kSpreadRows rows) go to different blocks.
constexpr uint64_t kSpreadRows = 1ull << 18;
struct CsrLongShared {
  uint64_t rows[kBlock];
  uint32_t count[3];
  RowSumShared sum;
};
template <bool kGeneric>
__device__ __forceinline__ bool CsrLongRows(const RowArgs& a, CsrLongShared& sh, RowStats& st) {
  const TableDesc T = a.t;
  const uint32_t dim = T.dim, slices = (dim + kLongColumns - 1) / kLongColumns;
  const uint32_t slice = blockIdx.x % slices, c0 = slice * kLongColumns, part = blockIdx.x / slices, parts = gridDim.x / slices;
  const uint32_t spread = a.rows <= kSpreadRows ? 0u : 3u;
  bool found = false;
  if (threadIdx.x == 0) sh.count[0] = 0;
  __syncthreads();
  uint32_t turn = 0;
  for (uint64_t first = 0; first < a.rows; first += uint64_t(kBlock) * parts, turn = turn == 2 ? 0 : turn + 1) {
    const uint64_t piece = (threadIdx.x >> spread) * uint64_t(parts) + part;
    const uint64_t r = first + (piece << spread) + (threadIdx.x & ((1u << spread) - 1));
    if (r < a.rows) {
      const uint64_t b = a.offsets[r], e = a.offsets[r + 1];
      if (e > b && e - b > a.short_refs) sh.rows[atomicAdd(&sh.count[turn], 1u)] = r;
    }
    if (threadIdx.x == 0) sh.count[turn == 2 ? 0 : turn + 1] = 0;  // (three in turn: one is still read)
    __syncthreads();
    const uint32_t rows = sh.count[turn];
    found = found || rows;
    for (uint32_t i = 0; i < rows; ++i) {
      const uint64_t row = sh.rows[i], b = a.offsets[row], e = a.offsets[row + 1];
      float g = 0.f;
      bool ok = true;  // the gradient scan has checked every source
      for (uint64_t at = b; at < e; at += kCsrPiece)
        g = BlockRowSum<!kGeneric>(sh.sum, CsrRefs{a.sources + at, a.scales + at, a.src, dim},
                                   uint32_t(min(e - at, kCsrPiece)), dim, c0, g, ok);
      const uint32_t c = c0 + threadIdx.x;
      if (threadIdx.x < kLongColumns && c < dim) AdamRow1(T, a.slots[row], c, g, true, st);
    }
  }
  return found;
}

// The update of a CSR packet decides; the fused one leaves long rows to the
// tail, the validate-only one looks at every row.
template <bool kGeneric>
__global__ void __launch_bounds__(kBlock) CsrUpdateKernel(RowArgs a) {
  __shared__ TableDesc s_t[1];
  __shared__ uint32_t s_mode;
  Control* ctrl = a.ctrl;
  const GuardInputs in = LoadGuard(ctrl);
  if (threadIdx.x == 0) s_t[0] = a.t;
  bool write = false;
  if (!LaunchGate(ctrl, in, s_t, a.gs, kDecide, &s_mode, write)) return;
  RowStats st;
  CsrShortRows<kGeneric>(a, write, write, st);
  FinishBlock(st, ctrl, a.bounds, write);
}

// After it: the long rows of a fused update, every row of a checked one that
// found nothing.  (In one kernel with the short rows, the tile's LDS and the
// registers of the long ones cost a packet of 200,000 rows of one reference of
// dim 16 more than half its rate, 46 -> 107 us, and rows of 33 references, one
// block's one after another, 43 -> 184.)
template <bool kGeneric>
__global__ void __launch_bounds__(kBlock) CsrTailKernel(RowArgs a) {
  __shared__ CsrLongShared sh;
  Control* ctrl = a.ctrl;
  const uint32_t mode = ctrl->mode, status = ctrl->status;
  if (mode == kReject) return;
  RowStats st;
  if (mode == kChecked) {
    if (status & (kErrorBits | EPS_HIP_STATUS_STALLED)) {
      if (blockIdx.x == 0 && threadIdx.x == 0) ReportStatus(ctrl, EPS_HIP_STATUS_REJECTED);
      return;
    }
    CsrShortRows<kGeneric>(a, true, true, st);
  }
  const bool found = CsrLongRows<kGeneric>(a, sh, st);
  if (!found && mode != kChecked) return;
  FinishBlock(st, ctrl, a.bounds, true);
}

// ---------------------------------------------------------------------------
TableDesc MakeTable(const eps_hip_table& t, const eps_hip_optimizer& o) {
  TableDesc d;
  d.state = t.state;
  d.rows = t.rows;
  d.dim = t.dim;
  d.beta1 = o.beta1;
  d.beta2 = o.beta2;
  d.omb1 = 1.0f - o.beta1;  // (1 - o.beta1) in float, lazy_adam.cpp:31
  d.omb2 = 1.0f - o.beta2;
  // lr_t in float exactly as lazy_adam.cpp:27 / cache_backend.cu:341.
  d.lr = o.learning_rate * std::sqrt(1 - o.beta2_power) / (1 - o.beta1_power);
  d.eps = o.epsilon;
  d.lo = o.bounded ? o.weight_min : -FLT_MAX;
  d.hi = o.bounded ? o.weight_max : FLT_MAX;
  d.bounded = o.bounded ? 1u : 0u;
  return d;
}

int CheckOptimizer(const eps_hip_optimizer& o) {
  // UpdateContext validation, src/cuda/cache_backend.cu:321-325.
  if (!(std::isfinite(o.learning_rate) && o.learning_rate > 0 && o.beta1_power >= 0 &&
        o.beta1_power < 1 && o.beta2_power >= 0 && o.beta2_power < 1))
    return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid update context");
  if (o.bounded && !(std::isfinite(o.weight_min) && std::isfinite(o.weight_max) &&
                     o.weight_min <= o.weight_max))
    return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid optimizer weight bounds");
  const float lr = o.learning_rate * std::sqrt(1 - o.beta2_power) / (1 - o.beta1_power);
  if (!std::isfinite(lr)) return Fail(EPS_HIP_INVALID_ARGUMENT, "optimizer learning-rate overflow");
  return EPS_HIP_OK;
}

uint32_t Log2G(uint32_t dim) {
  uint32_t log2g = 2;
  while ((1u << log2g) < dim / 4) ++log2g;
  return log2g;
}

// A launch that also records `done` when the kernel completes (nullptr: a
// plain launch).  The event then rides on the kernel's own completion signal,
// with no marker packet after it in the stream.  For the join of the side
// stream: 26 tables of ~43,000 references, 0.2723 -> 0.2687 ms a step over six
// paired runs on one box (each faster than its pair), 0.2708 -> 0.2701 over
// four on another; 65,536 pairs on one table 0.111 -> 0.109 ms.
template <typename... Args>
void LaunchRecording(void (*kernel)(Args...), dim3 grid, dim3 block, hipStream_t s, hipEvent_t done,
                     Args... args) {
  if (done)
    hipExtLaunchKernelGGL(kernel, grid, block, 0, s, nullptr, done, 0, args...);
  else
    hipLaunchKernelGGL(kernel, grid, block, 0, s, args...);
}

// The gradient scan.  It always runs (one block at least), since its block 0
// takes the bounds snapshot the guard decides from; the decision itself is
// made by the first kernel of the update (DecideBlock).
int LaunchGuard(const GuardArgs& g, uint64_t blocks, hipStream_t s, hipEvent_t done = nullptr) {
  LaunchRecording(GradMaxKernel, dim3(unsigned(std::max<uint64_t>(blocks, 1))), dim3(kBlock), s, done, g);
  EPS_HIP_LAUNCHED("gradient guard");
  return EPS_HIP_OK;
}

uint64_t SpanBlocks(uint64_t count, SpanKind kind = kGradientSpan) {
  const uint64_t per = uint64_t(kBlock) * (kind == kSortedSpan  ? kSortedItems
                                           : kind == kIndexSpan ? kIndexItems
                                                                : kMaxItems * 4);
  return (count + per - 1) / per;
}

// The hot-row kernel's side stream and fork/join events, per calling thread
// and device (created on first use, default priority, never destroyed), so
// concurrent callers never share an event.
struct Overlap {
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
int ThreadOverlap(Overlap** out) {
  constexpr int kDevices = 64;
  thread_local Overlap per_device[kDevices];
  int device = 0;
  EPS_HIP_TRY(Check(hipGetDevice(&device), "hipGetDevice"));
  if (device < 0 || device >= kDevices) return Fail(EPS_HIP_UNAVAILABLE, "device ordinal out of range");
  Overlap& o = per_device[device];
  if (!o.side) {
    EPS_HIP_TRY(Check(hipStreamCreateWithFlags(&o.side, hipStreamNonBlocking), "hot-row stream"));
    EPS_HIP_TRY(Check(hipEventCreateWithFlags(&o.fork, hipEventDisableTiming), "hot-row fork event"));
    EPS_HIP_TRY(Check(hipEventCreateWithFlags(&o.join, hipEventDisableTiming), "hot-row join event"));
  }
  *out = &o;
  return EPS_HIP_OK;
}

// The hot-row kernel runs beside the row kernels (on a side stream): its
// serial chains then overlap the row traffic instead of preceding it
// (measured on MI355X: 65,536 pairs on one table, 167 -> 133 us a push; 4 x
// 8.4 M references, 13.4 -> 11.6 ms; 26 tables of ~43,000 references with
// 64-column units on 256 blocks, 245 -> 236 us a step).  Pushes with a table
// of at least this many references take 32- or 16-column units on 512 blocks,
// so a very long row's chain data spreads over several CUs.
constexpr uint64_t kOverlapTableRefs = 1ull << 16;
constexpr uint32_t kFineSlice = 16, kNarrowSlice = 32, kWideSlice = 64;  // columns per hot-row unit
// References per hot-row chunk of each unit width.  16-column units take
// chunks of 256 references (a tile of 4,096 products, like a 64-column
// chunk), so their blocks hand a tile over (release, readiness poll, walk to
// the next chunk) once per 256 references instead of once per 64: 65,536
// pairs on one table, fused update 98-102 -> 84-91 us.  32-column units keep
// 64: with 128 the kernel needs 256 registers and 84 KB of LDS, one block per
// CU instead of two, and 4 x 8.4 M references lost (update 7.4-8.2 -> 8.1-8.3
// ms).
constexpr uint32_t kFineChunk = 256, kNarrowChunk = 64, kWideChunk = 64;
// Pushes with very long rows but fewer vector references than this take
// 16-column units (below).
constexpr uint64_t kFinePushRefs = 1ull << 18;

std::atomic<uint32_t> g_spin_limit{1u << 22};
uint32_t SpinLimit() { return g_spin_limit.load(std::memory_order_relaxed); }
// Whether this thread's pushes run the hot-row kernel on the side stream.
thread_local bool t_hot_row_overlap = true;

// Phases of a push (kPrimary: the fused update; kSecond: the checked apply)
// and kOneStream: every kernel on the caller's stream, the hot-row kernel
// before the row kernels (no side stream or event is created or used, so the
// push can be captured in a graph).
// kForked: the gradient scan has recorded the thread's fork event.
constexpr int kPrimary = 1, kSecond = 2, kOneStream = 4, kForked = 8;
constexpr uint64_t kVectorGrid = 4096;  // persistent grid cap of the vector kernels
constexpr uint64_t kSecondGrid = 32;      // grid cap of the checked apply: it usually exits at
                                          // once, and a small grid launches faster
constexpr uint32_t kApplyWindowBits = 5;  // its windows of sorted positions
constexpr uint64_t kBothBlocks = 1024;    // windows up to which one launch takes short and long rows
constexpr uint64_t kLongGrid = 2048;      // grid cap of the long rows' launches
// Grid cap of a class's short rows: six classes in one launch stay below the
// 2^32 threads that one can have.
constexpr uint64_t kSortedGrid = 1ull << 21;
// Blocks of the 16- and 32-column hot-row kernels.  A CU holds one of the
// former (87 KB of LDS) and two of the latter (68 KB).  4 x 8.4 M references:
// 256 blocks 8.64 ms a push, 512 5.67, 1,024 5.72; the 16-column kernel takes as
// long with any of them (65,536 pairs 67 to 68 us: its hottest row is one block
// a unit).
constexpr uint64_t kHotGrid = 512;
// Blocks of the 64-column hot-row kernel beside the row kernels: enough to
// finish the hot rows well before the row kernels do, few enough to leave
// them most of the GPU (26 tables of ~43,000 references: 64 blocks 259 us a
// step of pull + push, 256 blocks 236, 512 blocks 240).
constexpr uint64_t kWideHotGrid = 256;

// log2 of each class's row-run window.  A push of fewer than kRunBlocks windows
// (two a CU) halves them until it has as many, down to one position a lane
// group: with whole windows a group works through several rows, one memory
// latency after another, while CUs stand idle.  256 pairs of dim 32 34.3 ->
// 31.2 us a step; eight tables of 1,500 references, dims 16 to 256, 107 -> 94; four of
// 4,400 of dim 128 112 -> 97; 20,000 pairs of dim 256 109 -> 106.  (Up to 1,024
// windows: four tables of 22,000 references of dim 4 97 -> 101, since every
// window stages kLongRefs positions of look-ahead.)
constexpr uint64_t kRunBlocks = 512;
void RunWindowBits(const std::array<uint64_t, kClasses>& positions, uint32_t* bits) {
  uint64_t windows = 0;
  for (uint32_t c = 0; c + 1 < kClasses; ++c) windows += (positions[c] + RunPositions(c + 2) - 1) / RunPositions(c + 2);
  uint32_t halvings = 0;
  while (windows << halvings < kRunBlocks && halvings < 6) ++halvings;
  for (uint32_t c = 0; c + 1 < kClasses; ++c) {
    const uint32_t window = std::max(RunPositions(c + 2) >> halvings, kBlock >> (c + 2));
    bits[c] = 0;
    while ((1u << bits[c]) < window) ++bits[c];
  }
}

template <uint32_t kLog2G>
int LaunchRowRun(unsigned grid, const VecArgs& a, hipStream_t s, hipEvent_t done) {
  LaunchRecording(RowRunKernel<kLog2G>, dim3(grid), dim3(kBlock), s, done, a);
  EPS_HIP_LAUNCHED("row update");
  return EPS_HIP_OK;
}

// Hot rows (any vector class) when `hot_slice`, else the other rows of class
// `cls`; `done` (if any) is recorded when the launch completes.
int LaunchVectorUpdate(uint32_t cls, uint32_t hot_slice, unsigned grid, const VecArgs& a, hipStream_t s,
                       hipEvent_t done = nullptr) {
  if (hot_slice) {
    if (hot_slice == kWideSlice)
      LaunchRecording(HotSliceKernel<kWideSlice, kWideChunk>, dim3(grid), dim3(kHotBlock), s, done, a);
    else if (hot_slice == kFineSlice)
      LaunchRecording(HotSliceKernel<kFineSlice, kFineChunk>, dim3(grid), dim3(kHotBlock), s, done, a);
    else
      LaunchRecording(HotSliceKernel<kNarrowSlice, kNarrowChunk>, dim3(grid), dim3(kHotBlock), s, done, a);
    EPS_HIP_LAUNCHED("hot row update");
    return EPS_HIP_OK;
  }
  switch (cls) {
    case 0: return LaunchRowRun<2>(grid, a, s, done);
    case 1: return LaunchRowRun<3>(grid, a, s, done);
    case 2: return LaunchRowRun<4>(grid, a, s, done);
    case 3: return LaunchRowRun<5>(grid, a, s, done);
    case 4: return LaunchRowRun<6>(grid, a, s, done);
    default: return Fail(EPS_HIP_INVALID_ARGUMENT, "no vector kernel for this dimension class");
  }
}

// Bound on the hot rows of a push: a hot row takes more than kLongRefs
// references of its own table, so no table adds more hot rows than its
// references allow; a push with no such table (a few hundred pairs) launches no
// hot-row kernel and no events.  `table_refs`: references per table.
uint64_t HotRowBound(const eps_hip_table* tables, uint32_t table_count, const eps_hip_push_feature* features,
                     uint32_t feature_count, uint64_t* table_refs) {
  std::fill(table_refs, table_refs + EPS_HIP_MAX_TABLES, 0);
  for (uint32_t f = 0; f < feature_count; ++f) table_refs[features[f].table] += features[f].occurrences;
  uint64_t rows = 0;
  for (uint32_t t = 0; t < table_count; ++t)
    if (DimClass(tables[t].dim) < kClasses - 1) rows += table_refs[t] / (kLongRefs + 1);
  return rows;
}

int RunSorted(const eps_hip_table* tables, const eps_hip_optimizer* optimizers, uint32_t table_count,
              const eps_hip_push_feature* features, uint32_t feature_count, const PushPlan& plan,
              const PushLayout& L, uint8_t* ws, bool reduce, const uint64_t* occ2u, float* out,
              uint64_t stride, Bounds* bounds, hipStream_t s, int phases) {
  FusedArgs a{};
  const bool in_b = plan.passes % 2 == 1;
  a.keys = reinterpret_cast<const uint32_t*>(ws + (in_b ? L.keys_b : L.keys_a));
  a.vals = reinterpret_cast<const uint32_t*>(ws + (in_b ? L.vals_b : L.vals_a));
  a.rs = reinterpret_cast<const uint64_t*>(ws + L.sorted_rs);
  a.occ2u = occ2u;
  a.reduce_out = out;
  a.reduce_stride = stride;
  a.ctrl = reinterpret_cast<Control*>(ws);
  a.bounds = bounds;
  a.row_bits = plan.row_bits;
  a.tables = table_count;
  a.features = feature_count;
  a.n = uint32_t(plan.occurrences);
  a.gs = GuardScalars{0, table_count};  // refs: the prepared valid count
  // The first kernel of the primary phase makes the guard decision.
  uint32_t role = kDecide;
  bool overlap = false;  // hot rows (on the side stream, joined before the checked apply)
  Overlap* ov = nullptr;
  for (uint32_t k = 0; k < table_count; ++k) {
    const uint32_t t = plan.table_of_key[k];
    eps_hip_optimizer o{};
    if (optimizers) o = optimizers[t];
    else { o.learning_rate = 1; o.beta1 = 0; o.beta2 = 0; o.epsilon = 1; }
    a.t[k] = MakeTable(tables[t], o);
  }
  a.wide = 1;
  for (uint32_t f = 0; f < feature_count; ++f) {
    a.grad[f] = features[f].gradients;
    if (reinterpret_cast<uintptr_t>(features[f].gradients) % 16) a.wide = 0;
    a.grad_rows[f] = features[f].pooling == EPS_HIP_POOL_SEQUENCE ? features[f].occurrences : features[f].bags;
  }
  if (!reduce) {
    // Vector classes: hot rows (sliced) first, then the other rows per class.
    VecArgs va{};
    for (uint32_t k = 0; k < table_count; ++k) va.t[k] = a.t[k];
    for (uint32_t f = 0; f < feature_count; ++f) {
      va.grad[f] = a.grad[f];
      va.grad_rows[f] = a.grad_rows[f];
    }
    va.tables = table_count;
    va.features = feature_count;
    va.n = a.n;
    va.keys = a.keys;
    va.rs = a.rs;
    va.hot = reinterpret_cast<const HotEntry*>(ws + L.long_list);
    va.hot_capacity = uint32_t(L.HotCapacity());
    va.ctrl = a.ctrl;
    va.bounds = bounds;
    va.gs = a.gs;
    va.spin_limit = SpinLimit();
    va.row_bits = plan.row_bits;
    uint64_t table_refs[EPS_HIP_MAX_TABLES];
    const uint64_t hot_rows = HotRowBound(tables, table_count, features, feature_count, table_refs);
    const uint64_t most_refs = *std::max_element(table_refs, table_refs + table_count);
    const bool long_rows = most_refs >= kOverlapTableRefs;
    uint64_t vector_occurrences = 0;
    for (uint32_t cls = 0; cls + 1 < kClasses; ++cls) vector_occurrences += plan.class_occurrences[cls];
    // Slice width: pushes with very long hot rows (some table with 65,536 or
    // more references) cut each row into 32-column units, so one row's chain
    // data spreads over several CUs (4 x 8.4 M references: 16-column units
    // 13.8 ms a step, 32-column units, each a whole line per reference, 12.8);
    // small pushes of that kind, whose time is their hottest row's chain and
    // whose gradient rows stay in the caches, take 16-column units, so each
    // chunk moves half the bytes through its producers (65,536 pairs on one
    // table: 100.6 -> 97.0 us an update; a ragged 8-table push of 525,000
    // references lost with them, 270 -> 295 us, and with 256-reference chunks
    // it still did, 264 -> 296 us, as did 4 x 8.4 M references, 9.9 -> 10.8 ms
    // a step); otherwise 64-column units,
    // whose fewer and fuller units a block's producers stage with less
    // bookkeeping per column (26 tables of ~43,000 references: 47 -> 41 us a
    // push).
    const uint32_t slice =
        !long_rows ? kWideSlice : (vector_occurrences < kFinePushRefs ? kFineSlice : kNarrowSlice);
    // Units per hot row: the widest vector table's slices, rounded up to a
    // power of two (units past a row's dimension are skipped in the kernel).
    uint32_t slices = 1;
    for (uint32_t t = 0; t < table_count; ++t)
      if (DimClass(tables[t].dim) < kClasses - 1)
        slices = std::max(slices, (tables[t].dim + slice - 1) / slice);
    va.slice_bits = 0;
    while ((1u << va.slice_bits) < slices) ++va.slice_bits;
    const uint64_t hot_units = hot_rows << va.slice_bits;
    overlap = hot_units != 0 && !(phases & kOneStream) && t_hot_row_overlap;
    if (phases & kPrimary) {
      // Grids are multiples of kXcds (the kernels split their work by XCD).
      auto xcd_grid = [](uint64_t b) { return (b + kXcds - 1) / kXcds * kXcds; };
      // The hot-row kernel and the row runs side by side on two streams,
      // joined before the checked apply: the longer of the two stays on this
      // stream and the other goes to the side stream, so this stream waits
      // for no event while the longer part runs.  The hot rows are the longer
      // part when some table takes 65,536 or more references (its hottest
      // rows' chains outlast the row runs: 65,536 pairs on one table, hot rows
      // 80 us against row runs 49 us); otherwise the row runs are.  (Below that
      // it turns on the skew, which the host does not know: with the row runs
      // on the side stream, eight tables of 64,000 references take 109 us a
      // push instead of 115 when their ids are Zipf of 1.05 and 115 instead of
      // 134 at 1.2, but fourteen of 20,000 take 89 instead of 71, eight of
      // 43,000 94 instead of 86, and two of 64,000 uniform ids 74 instead of
      // 62.)  Both sides make the guard decision themselves, from the same
      // snapshot, so they decide the same.
      const bool rows_beside = overlap && long_rows;
      const uint64_t hot_blocks =
          hot_units ? xcd_grid(std::min<uint64_t>(hot_units, long_rows ? kHotGrid : kWideHotGrid)) : 0;
      if (overlap) {
        EPS_HIP_TRY(ThreadOverlap(&ov));
        if (!(phases & kForked)) EPS_HIP_TRY(Check(hipEventRecord(ov->fork, s), "update fork"));
        // With the rows beside, the hot rows (the longer part) go out on this
        // stream before the side stream's wait is set up (the wait on a
        // pending event takes ~14 us of host time): they use no class fields
        // of `va`, and they decide from the same snapshot as the rows.
        if (hot_units && rows_beside) {
          va.role = role;
          EPS_HIP_TRY(LaunchVectorUpdate(0, slice, unsigned(hot_blocks), va, s));
        }
        EPS_HIP_TRY(Check(hipStreamWaitEvent(ov->side, ov->fork, 0), "update fork wait"));
      }
      // The side stream's last kernel records the join as it completes.
      bool joined = false;
      if (hot_units && !rows_beside) {
        va.role = role;
        EPS_HIP_TRY(LaunchVectorUpdate(0, slice, unsigned(hot_blocks), va, overlap ? ov->side : s,
                                       overlap ? ov->join : nullptr));
        joined = overlap;
        if (!overlap) role = kFollow;  // one stream: the hot rows first, deciding; the row kernels follow
      }
      const hipStream_t rs = rows_beside ? ov->side : s;
      // The row runs: one launch per present vector class, or one launch
      // for all of them when there are several.
      uint32_t present = 0;
      uint64_t total_blocks = 0;
      RunWindowBits(plan.class_occurrences, va.window_bits);
      for (uint32_t cls = 0; cls + 1 < kClasses; ++cls) {
        va.class_block[cls] = uint32_t(total_blocks);
        va.class_grid[cls] = 0;
        if (!plan.class_occurrences[cls]) continue;
        const uint64_t window = 1ull << va.window_bits[cls];
        const uint64_t blocks =
            xcd_grid(std::min<uint64_t>((plan.class_occurrences[cls] + window - 1) / window, kVectorGrid));
        va.class_grid[cls] = uint32_t(blocks);
        total_blocks += blocks;
        ++present;
      }
      va.class_block[kClasses - 1] = uint32_t(total_blocks);
      va.class_grid[kClasses - 1] = 0;
      // With the rows beside, their launch is the side stream's last (one
      // launch at most: several classes share one).
      const hipEvent_t rows_done = rows_beside ? ov->join : nullptr;
      if (present > 1) {
        va.role = role;
        role = kFollow;
        LaunchRecording(RowRunClassesKernel, dim3(unsigned(total_blocks)), dim3(kBlock), rs, rows_done, va);
        EPS_HIP_LAUNCHED("row update (all classes)");
        joined |= rows_beside;
      } else {
        for (uint32_t cls = 0; cls + 1 < kClasses; ++cls) {
          if (!va.class_grid[cls]) continue;
          va.cls = cls;
          va.role = role;
          role = kFollow;
          EPS_HIP_TRY(LaunchVectorUpdate(cls, 0, va.class_grid[cls], va, rs, rows_done));
          joined |= rows_beside;
        }
      }
      if (overlap && !joined) EPS_HIP_TRY(Check(hipEventRecord(ov->join, ov->side), "update join"));
    }
  }
  // The sorted driver's launches.  Whether a table of classes [first, kClasses)
  // has references enough for a long row:
  auto may_be_long = [&](uint32_t first) {
    uint64_t refs[EPS_HIP_MAX_TABLES] = {};
    for (uint32_t f = 0; f < feature_count; ++f) refs[features[f].table] += features[f].occurrences;
    for (uint32_t t = 0; t < table_count; ++t)
      if (DimClass(tables[t].dim) >= first && refs[t] > kBlockRowRefs) return true;
    return false;
  };
  for (uint32_t cls = 0; cls < kClasses; ++cls) {
    a.window_bits[cls] = 0;
    while ((2u << a.window_bits[cls]) <= PositionsPerBlock(cls)) ++a.window_bits[cls];
  }
  // Long rows' windows: as many positions as threads to look at them, fewer
  // where that leaves blocks idle.
  a.long_slices = 1;
  for (uint32_t t = 0; t < table_count; ++t)
    a.long_slices = std::max(a.long_slices, (tables[t].dim + kLongColumns - 1) / kLongColumns);
  auto long_grid = [&](uint64_t positions) {
    a.long_bits = positions >= (kLongGrid << 8) ? 8 : 6;
    return unsigned(std::min<uint64_t>(((positions + (1u << a.long_bits) - 1) >> a.long_bits) * a.long_slices, kLongGrid));
  };
  if (reduce) {
    uint64_t blocks = 0;
    for (uint32_t cls = 0; cls < kClasses; ++cls) {
      a.class_block[cls] = uint32_t(blocks);
      blocks += std::min<uint64_t>((plan.class_occurrences[cls] + PositionsPerBlock(cls) - 1) / PositionsPerBlock(cls),
                                   kSortedGrid);
    }
    a.class_block[kClasses] = uint32_t(blocks);
    const unsigned grid = long_grid(plan.occurrences);
    const bool apart = blocks > kBothBlocks;
    if (!may_be_long(0) || apart)
      hipLaunchKernelGGL(SortedReduceKernel, dim3(unsigned(blocks)), dim3(kBlock), 0, s, a);
    else
      hipLaunchKernelGGL(SortedLongReduceKernel, dim3(unsigned(blocks)), dim3(kBlock), 0, s, a);
    EPS_HIP_LAUNCHED("sorted reduce");
    if (may_be_long(0) && apart) {
      hipLaunchKernelGGL(LongReduceKernel, dim3(grid), dim3(kBlock), 0, s, a);
      EPS_HIP_LAUNCHED("sorted reduce (long rows)");
    }
    return EPS_HIP_OK;
  }
  // The generic class.
  if ((phases & kPrimary) && plan.class_occurrences[kClasses - 1]) {
    const uint64_t positions = plan.class_occurrences[kClasses - 1];
    const uint64_t blocks = (positions + PositionsPerBlock(kClasses - 1) - 1) / PositionsPerBlock(kClasses - 1);
    a.cls = kClasses - 1;
    a.cls_end = kClasses;
    a.role = role;
    const unsigned grid = long_grid(positions);
    const bool apart = blocks > kBothBlocks, any_long = may_be_long(kClasses - 1);
    auto kernel = any_long && !apart ? SortedLongUpdateKernel : SortedUpdateKernel;
    hipLaunchKernelGGL(kernel, dim3(unsigned(std::min<uint64_t>(blocks, kSortedGrid))), dim3(kBlock), 0, s, a);
    EPS_HIP_LAUNCHED("sorted update");
    if (any_long && apart) {
      a.role = kFollow;
      hipLaunchKernelGGL(LongUpdateKernel, dim3(grid), dim3(kBlock), 0, s, a);
      EPS_HIP_LAUNCHED("sorted update (long rows)");
    }
  }
  if (overlap && (phases & kPrimary)) EPS_HIP_TRY(Check(hipStreamWaitEvent(s, ov->join, 0), "hot-row join wait"));
  // The checked apply (after a validate-only pass) is one launch over every
  // class, one wavefront per row: it usually exits at once, and when it runs
  // it adds each row's references in the same order as the passes above.
  if (phases & kSecond) {
    a.cls = 0;
    a.cls_end = kClasses;
    a.role = kFallback;
    a.window_bits[kClasses - 1] = kApplyWindowBits;
    a.long_bits = 8;
    const uint64_t windows = (plan.occurrences + (1u << kApplyWindowBits) - 1) >> kApplyWindowBits;
    if (windows) {
      hipLaunchKernelGGL(SortedLongUpdateKernel, dim3(unsigned(std::min<uint64_t>(windows, kSecondGrid))),
                         dim3(kBlock), 0, s, a);
      EPS_HIP_LAUNCHED("sorted update (checked apply)");
    }
  }
  return EPS_HIP_OK;
}

}  // namespace
}  // namespace eps_hip

using namespace eps_hip;

extern "C" {

// Shared validation of the push entry points.
static int PushSetup(const eps_hip_table* tables, const eps_hip_optimizer* optimizers,
                     uint32_t table_count, const eps_hip_push_feature* features,
                     uint32_t feature_count, void* workspace, uint64_t workspace_bytes,
                     void* bounds, PushPlan& plan) {
  EPS_HIP_TRY(PlanPush(tables, table_count, features, feature_count, plan));
  const PushLayout L(plan.occurrences);
  if (!workspace || workspace_bytes < L.total)
    return Fail(EPS_HIP_CAPACITY_EXCEEDED, "push workspace too small");
  if (!optimizers || !bounds) return Fail(EPS_HIP_INVALID_ARGUMENT, "push needs optimizers and bounds");
  for (uint32_t t = 0; t < table_count; ++t) EPS_HIP_TRY(CheckOptimizer(optimizers[t]));
  for (uint32_t f = 0; f < feature_count; ++f) {
    const auto& in = features[f];
    const uint64_t rows = in.pooling == EPS_HIP_POOL_SEQUENCE ? in.occurrences : in.bags;
    if (rows && !in.gradients) return Fail(EPS_HIP_INVALID_ARGUMENT, "null feature gradient");
  }
  return EPS_HIP_OK;
}

// The gradient scan of a push; `done` (if any) is recorded as it completes.
static int PushScan(const eps_hip_table* tables, uint32_t table_count, const eps_hip_push_feature* features,
                    uint32_t feature_count, const PushPlan& plan, void* workspace, void* bounds, void* stream,
                    hipEvent_t done) {
  GuardArgs g{};
  uint64_t blocks = 0;
  auto add = [&](const void* p, uint64_t count, SpanKind kind) {
    if (!count) return;
    g.span[g.spans++] = Span{static_cast<const float*>(p), count, uint32_t(blocks), kind, 0};
    blocks += SpanBlocks(count, kind);
  };
  for (uint32_t f = 0; f < feature_count; ++f) {
    const auto& in = features[f];
    const uint64_t rows = in.pooling == EPS_HIP_POOL_SEQUENCE ? in.occurrences : in.bags;
    add(in.gradients, rows * tables[in.table].dim, kGradientSpan);
  }
  // The prepared keys, checked before the update uses them as addresses.
  const PushLayout L(plan.occurrences);
  auto* ws = static_cast<uint8_t*>(workspace);
  g.sorted.keys = reinterpret_cast<const uint32_t*>(ws + (plan.passes % 2 == 1 ? L.keys_b : L.keys_a));
  for (uint32_t k = 0; k < table_count; ++k) g.sorted.table_rows[k] = tables[plan.table_of_key[k]].rows;
  g.sorted.row_bits = plan.row_bits;
  g.sorted.tables = table_count;
  add(nullptr, plan.occurrences, kSortedSpan);
  g.ctrl = static_cast<Control*>(workspace);
  g.bounds = static_cast<const Bounds*>(bounds);
  return LaunchGuard(g, blocks, AsStream(stream), done);
}

int eps_hip_push_begin(const eps_hip_table* tables, const eps_hip_optimizer* optimizers,
                       uint32_t table_count, const eps_hip_push_feature* features,
                       uint32_t feature_count, void* workspace, uint64_t workspace_bytes,
                       void* bounds, void* stream) {
  PushPlan plan;
  EPS_HIP_TRY(PushSetup(tables, optimizers, table_count, features, feature_count, workspace,
                        workspace_bytes, bounds, plan));
  return PushScan(tables, table_count, features, feature_count, plan, workspace, bounds, stream, nullptr);
}

static int PushPhase(const eps_hip_table* tables, const eps_hip_optimizer* optimizers,
                     uint32_t table_count, const eps_hip_push_feature* features,
                     uint32_t feature_count, void* workspace, uint64_t workspace_bytes,
                     void* bounds, void* stream, int phase) {
  PushPlan plan;
  EPS_HIP_TRY(PushSetup(tables, optimizers, table_count, features, feature_count, workspace,
                        workspace_bytes, bounds, plan));
  if (!plan.occurrences) return EPS_HIP_OK;
  const PushLayout L(plan.occurrences);
  return RunSorted(tables, optimizers, table_count, features, feature_count, plan, L,
                   static_cast<uint8_t*>(workspace), false, nullptr, nullptr, 0,
                   static_cast<Bounds*>(bounds), AsStream(stream), phase);
}

int eps_hip_push_apply(const eps_hip_table* tables, const eps_hip_optimizer* optimizers,
                       uint32_t table_count, const eps_hip_push_feature* features,
                       uint32_t feature_count, void* workspace, uint64_t workspace_bytes,
                       void* bounds, void* stream) {
  return PushPhase(tables, optimizers, table_count, features, feature_count, workspace,
                   workspace_bytes, bounds, stream, kPrimary);
}

int eps_hip_push_end(const eps_hip_table* tables, const eps_hip_optimizer* optimizers,
                     uint32_t table_count, const eps_hip_push_feature* features,
                     uint32_t feature_count, void* workspace, uint64_t workspace_bytes,
                     void* bounds, void* stream) {
  return PushPhase(tables, optimizers, table_count, features, feature_count, workspace,
                   workspace_bytes, bounds, stream, kSecond);
}

// A whole push: scan, update and checked apply from one plan.  Nothing of the
// caller's can come between the scan and the update, so the side stream is
// forked from the scan's own completion, without a marker packet behind it
// (which also holds the row kernels up: 26 tables of ~43,000 references, scan
// end to row kernel start 11-14 -> 5 us).
static int PushWhole(const eps_hip_table* tables, const eps_hip_optimizer* optimizers, uint32_t table_count,
                     const eps_hip_push_feature* features, uint32_t feature_count, void* workspace,
                     uint64_t workspace_bytes, void* bounds, void* stream, int phases) {
  PushPlan plan;
  EPS_HIP_TRY(PushSetup(tables, optimizers, table_count, features, feature_count, workspace,
                        workspace_bytes, bounds, plan));
  uint64_t table_refs[EPS_HIP_MAX_TABLES];
  Overlap* ov = nullptr;
  if (!(phases & kOneStream) && t_hot_row_overlap &&
      HotRowBound(tables, table_count, features, feature_count, table_refs)) {
    EPS_HIP_TRY(ThreadOverlap(&ov));
    phases |= kForked;
  }
  EPS_HIP_TRY(PushScan(tables, table_count, features, feature_count, plan, workspace, bounds, stream,
                       ov ? ov->fork : nullptr));
  if (!plan.occurrences) return EPS_HIP_OK;
  const PushLayout L(plan.occurrences);
  return RunSorted(tables, optimizers, table_count, features, feature_count, plan, L,
                   static_cast<uint8_t*>(workspace), false, nullptr, nullptr, 0, static_cast<Bounds*>(bounds),
                   AsStream(stream), phases);
}

}  // extern "C"

namespace eps_hip {
int PushOneStream(const eps_hip_table* tables, const eps_hip_optimizer* optimizers, uint32_t table_count,
                  const eps_hip_push_feature* features, uint32_t feature_count, void* workspace,
                  uint64_t workspace_bytes, void* bounds, void* stream) {
  return PushWhole(tables, optimizers, table_count, features, feature_count, workspace, workspace_bytes, bounds,
                   stream, kPrimary | kSecond | kOneStream);
}
}  // namespace eps_hip

extern "C" {

int eps_hip_push(const eps_hip_table* tables, const eps_hip_optimizer* optimizers,
                 uint32_t table_count, const eps_hip_push_feature* features,
                 uint32_t feature_count, void* workspace, uint64_t workspace_bytes, void* bounds,
                 void* stream) {
  return PushWhole(tables, optimizers, table_count, features, feature_count, workspace, workspace_bytes, bounds,
                   stream, kPrimary | kSecond);
}

int eps_hip_reduce(const eps_hip_table* tables, uint32_t table_count,
                   const eps_hip_push_feature* features, uint32_t feature_count,
                   void* workspace, uint64_t workspace_bytes, const uint64_t* occurrence_to_unique,
                   float* values, uint64_t row_stride, void* stream) {
  PushPlan plan;
  EPS_HIP_TRY(PlanPush(tables, table_count, features, feature_count, plan));
  const PushLayout L(plan.occurrences);
  if (!workspace || workspace_bytes < L.total)
    return Fail(EPS_HIP_CAPACITY_EXCEEDED, "push workspace too small");
  if (!occurrence_to_unique || !values) return Fail(EPS_HIP_INVALID_ARGUMENT, "null reduce buffers");
  uint32_t max_dim = 0;
  for (uint32_t t = 0; t < table_count; ++t) max_dim = std::max(max_dim, tables[t].dim);
  if (row_stride < max_dim || (row_stride % 4 && max_dim % 4 == 0 && max_dim <= 256))
    return Fail(EPS_HIP_INVALID_ARGUMENT, "row stride must cover every dimension (multiple of 4)");
  EPS_HIP_TRY(PrepareWithOccurrences(tables, table_count, features, feature_count, workspace, workspace_bytes,
                                     stream));
  if (!plan.occurrences) return EPS_HIP_OK;
  auto* ws = static_cast<uint8_t*>(workspace);
  return RunSorted(tables, nullptr, table_count, features, feature_count, plan, L, ws, true,
                   occurrence_to_unique, values, row_stride, nullptr, AsStream(stream), kPrimary);
}

uint64_t eps_hip_update_workspace_bytes(void) { return sizeof(Control); }

static int RunRows(const eps_hip_table* table, const eps_hip_optimizer* optimizer,
                   const uint64_t* slots, uint64_t rows, const uint64_t* offsets,
                   const uint64_t* sources, const float* scales, const float* src,
                   uint64_t src_values, uint64_t references, void* workspace, void* bounds,
                   void* stream) {
  if (!table || !table->state || table->dim == 0 || table->dim > 65536)
    return Fail(EPS_HIP_INVALID_ARGUMENT, "invalid update table");
  if (!optimizer || !workspace || !bounds) return Fail(EPS_HIP_INVALID_ARGUMENT, "null update argument");
  EPS_HIP_TRY(CheckOptimizer(*optimizer));
  const hipStream_t s = AsStream(stream);
  auto* ctrl = static_cast<Control*>(workspace);
  // The control block starts at zero, except the status history (its last word).
  static_assert(kHistoryWord + 1 == sizeof(Control) / 4, "history is the control block's last word");
  EPS_HIP_TRY(LaunchFill(reinterpret_cast<uint32_t*>(ctrl), 0, kHistoryWord, s));
  if (!rows) return EPS_HIP_OK;
  if (!slots || !src) return Fail(EPS_HIP_INVALID_ARGUMENT, "null update buffers");
  GuardArgs g{};
  uint64_t blocks = 0;
  auto add = [&](const void* p, uint64_t count, SpanKind kind, uint64_t limit) {
    if (!count) return;
    g.span[g.spans++] = Span{static_cast<const float*>(p), count, uint32_t(blocks), kind, limit};
    blocks += SpanBlocks(count, kind);
  };
  add(src, src_values, kGradientSpan, 0);
  if (scales) add(scales, references, kScaleSpan, 0);
  // Caller-provided indices are range-checked before the update, so a bad
  // slot or reference rejects it instead of touching memory out of range.
  add(slots, rows, kIndexSpan, table->rows);
  if (offsets) {
    add(offsets, rows + 1, kIndexSpan, references + 1);
    add(sources, references, kIndexSpan, src_values / table->dim);
  }
  const TableDesc d = MakeTable(*table, *optimizer);
  g.ctrl = ctrl;  // the index checks report to its prepare status
  g.bounds = static_cast<const Bounds*>(bounds);
  EPS_HIP_TRY(LaunchGuard(g, blocks, s));
  RowArgs a{};
  a.t = d;
  a.slots = slots;
  a.offsets = offsets;
  a.sources = sources;
  a.scales = scales;
  a.src = src;
  a.rows = rows;
  a.ctrl = ctrl;
  a.bounds = static_cast<Bounds*>(bounds);
  a.gs = GuardScalars{std::max<uint64_t>(1, offsets ? references : 1), 1};
  const uint32_t cls = DimClass(table->dim);
  const bool generic = cls == 5 || reinterpret_cast<uintptr_t>(src) % 16 != 0;
  a.log2g = generic ? 6 : Log2G(table->dim);
  const uint32_t groups = kBlock >> a.log2g;
  const uint64_t vb = (rows + groups - 1) / groups;
  if (vb > 0xffffffffull) return Fail(EPS_HIP_CAPACITY_EXCEEDED, "too many rows");
  a.vblocks = uint32_t(vb);
  if (offsets) {
    a.short_refs = CsrShortRefs(references);
    hipLaunchKernelGGL(generic ? CsrUpdateKernel<true> : CsrUpdateKernel<false>, dim3(a.vblocks), dim3(kBlock), 0, s, a);
    EPS_HIP_LAUNCHED("csr update");
    // (Whole turns of the column units.)
    const uint32_t slices = (table->dim + kLongColumns - 1) / kLongColumns;
    const uint64_t most = rows >= kTailRows ? 2 * kTailGrid : kTailGrid;
    const uint64_t parts = std::min<uint64_t>(rows, std::max<uint64_t>(most / slices, 1));
    hipLaunchKernelGGL(generic ? CsrTailKernel<true> : CsrTailKernel<false>, dim3(unsigned(parts * slices)), dim3(kBlock),
                       0, s, a);
    EPS_HIP_LAUNCHED("csr update (long rows, checked apply)");
    return EPS_HIP_OK;
  }
  auto kernel = generic ? RowUpdateKernel<true> : RowUpdateKernel<false>;
  a.role = kDecide;
  hipLaunchKernelGGL(kernel, dim3(a.vblocks), dim3(kBlock), 0, s, a);
  EPS_HIP_LAUNCHED("row update");
  a.role = kFallback;
  hipLaunchKernelGGL(kernel, dim3(std::min<uint32_t>(a.vblocks, kFallbackGrid)), dim3(kBlock), 0, s, a);
  EPS_HIP_LAUNCHED("row update (checked apply)");
  return EPS_HIP_OK;
}

int eps_hip_adam_rows(const eps_hip_table* table, const eps_hip_optimizer* optimizer,
                      const uint64_t* slots, const float* gradients, uint64_t rows,
                      void* workspace, void* bounds, void* stream) {
  const uint64_t values = table ? rows * table->dim : 0;
  return RunRows(table, optimizer, slots, rows, nullptr, nullptr, nullptr, gradients, values,
                 0, workspace, bounds, stream);
}

int eps_hip_adam_compact(const eps_hip_table* table, const eps_hip_optimizer* optimizer,
                         const uint64_t* slots, uint64_t rows, const uint64_t* row_offsets,
                         const uint64_t* source_rows, const float* scales,
                         const float* source_values, uint64_t source_count, uint64_t references,
                         void* workspace, void* bounds, void* stream) {
  if (rows && (!row_offsets || (references && (!source_rows || !scales))))
    return Fail(EPS_HIP_INVALID_ARGUMENT, "null compact buffers");
  const uint64_t values = table ? source_count * table->dim : 0;
  return RunRows(table, optimizer, slots, rows, row_offsets, source_rows, scales, source_values,
                 values, references, workspace, bounds, stream);
}

uint32_t* eps_hip_status_word(void* workspace) {
  return workspace ? &static_cast<Control*>(workspace)->status : nullptr;
}

uint32_t* eps_hip_status_history_word(void* workspace) {
  return workspace ? &static_cast<Control*>(workspace)->history : nullptr;
}

int eps_hip_set_hot_row_overlap(int enabled) {
  t_hot_row_overlap = enabled != 0;
  return EPS_HIP_OK;
}

int eps_hip_debug_set_spin_limit(uint32_t polls) {
  g_spin_limit.store(polls, std::memory_order_relaxed);
  return EPS_HIP_OK;
}

int eps_hip_read_status(void* workspace, uint32_t* status, void* stream) {
  if (!workspace || !status) return Fail(EPS_HIP_INVALID_ARGUMENT, "null status arguments");
  EPS_HIP_TRY(Check(hipStreamSynchronize(AsStream(stream)), "hipStreamSynchronize"));
  EPS_HIP_TRY(Check(hipMemcpy(status, &static_cast<Control*>(workspace)->status, 4,
                              hipMemcpyDeviceToHost), "status copy"));
  return EPS_HIP_OK;
}

}  // extern "C"
