// hawk_team.hip — the cross-sample team stages of hawk's gfx950 target,
// written by hand for CDNA4 (wave64, 160 KiB LDS per workgroup, 8 XCDs).
//
// Two reductions whose bits must not depend on the launch: the fixed-tree
// ordered sum (reference hawk/emit/team.py:208-278 `_block_part` and
// :173-192 `_block`, gp form) and the keyed ordered scatter (reference
// hawk/emit/team.py:322-460 with the chunk rule of hawk/_lane_bind.py:111-114).
// Neither uses a floating-point atomic: every addition happens in the order
// the reference's serial host walk makes it, so the results are bit-identical
// to that walk.  Build flags keep -ffp-contract=off.

#include "hawk_core.h"
#include "hawk_internal.h"

#include <hip/hip_runtime.h>
#include <cstdint>
#include <mutex>
#include <string>

namespace {

// ---------------------------------------------------------------------------
// Fixed-tree ordered sum.
// ---------------------------------------------------------------------------
constexpr int kVirtualLanes = 65536;   // reference hawk/emit/team.py:21-23
constexpr int kFoldLanes = 1024;
constexpr int kGroups = 64;            // reference hawk/ir/team.py:649 GROUPS
constexpr int kLaneBlock = 256;
// Rows of a batch: 32, and 64 in float32 past 64 rows a lane (2^26 float rows:
// 58 us in batches of 32, 47 of 64, 88 with one batch at a time).
constexpr int kSumBatch = 32;
constexpr int kSumLong = 64;

// Scratch layout (bytes): lanes[65536] f64 | gp[64] f64 | ticket u32 (+pad).
constexpr size_t kLanesBytes = sizeof(double) * kVirtualLanes;
constexpr size_t kGpBytes = sizeof(double) * kGroups;
constexpr size_t kSumScratch = kLanesBytes + kGpBytes + 256;

// Virtual lane l = blockIdx.x*256 + threadIdx.x adds u[l], u[l+65536], ... in
// order from +0.0.  A batch of rows is in flight while the one
// before it is added (one wave a SIMD holds the lanes, so nothing else covers
// the loads' latency); Once: all rows are one batch.  A row past the end adds
// +0.0, which leaves a sum that is never -0.0 as it is, and a group of eight
// rows past every lane's end is neither tested row by row nor added (testing
// 64 loads that read nothing cost 1.5 us of a float sum of 524 289 to
// 5 000 000 rows).  The fold's ticket is cleared here, one launch ahead of
// the fold that takes it, so a sum never depends on what an earlier call left
// in its scratch.
template <class T, int Batch, bool Once>
__global__ __launch_bounds__(kLaneBlock) void hawk_sum_lanes(const T* __restrict__ u,
                                                              long long n,
                                                              T* __restrict__ lanes,
                                                              unsigned* __restrict__ ticket) {
    const long long l = static_cast<long long>(blockIdx.x) * kLaneBlock + threadIdx.x;
    if (l == 0) *ticket = 0u;
    constexpr long long kStep = kVirtualLanes;
    const long long rows = (n + kStep - 1) / kStep;         // of the first lane, the longest
    T s = T(0);
    auto load = [&](long long r, T (&a)[Batch]) {
        const T* p = u + r * kStep + l;
        if (!Once && (r + Batch) * kStep <= n) {
#pragma unroll
            for (int k = 0; k < Batch; ++k) a[k] = __builtin_nontemporal_load(p + k * kStep);
        } else if (r < rows) {
            const int left = n - r * kStep - l <= 0 ? 0 : static_cast<int>((n - r * kStep - l + kStep - 1) / kStep);
            const int held = static_cast<int>(rows - r);
#pragma unroll
            for (int k8 = 0; k8 < Batch; k8 += 8) {
                if (k8 >= held) break;                       // the whole grid
#pragma unroll
                for (int k = k8; k < k8 + 8; ++k) a[k] = k < left ? __builtin_nontemporal_load(p + k * kStep) : T(0);
            }
        }
    };
    auto add = [&](long long r, const T (&a)[Batch]) {
        const long long held = rows - r;
#pragma unroll
        for (int k8 = 0; k8 < Batch; k8 += 8) {
            if (k8 >= held) break;                           // the whole grid
#pragma unroll
            for (int k = k8; k < k8 + 8; ++k) s += a[k];
        }
    };
    T a[Batch];
    load(0, a);
    if constexpr (Once) {
        add(0, a);
    } else {
        T b[Batch];
        for (long long r = 0; r < rows; r += 2 * Batch) {
            load(r + Batch, b);
            add(r, a);
            load(r + 2 * Batch, a);
            add(r + Batch, b);
        }
    }
    lanes[l] = s;
}

// Group g of 1024 lanes folded by s[i] += s[i+w], w = 512..1, into gp[g]; the
// last group to finish folds the 64 group values by the same tree, w = 32..1,
// and stores the result.  The ticket is left at zero for the next call.
// Thread t holds lanes t, t+256, t+512 and t+768, so levels 512 and 256 are
// its own adds; levels 128 and 64 cross waves through LDS, and levels 32..1
// run in wave 0, lane i adding lane i+w's value taken by a permute: the same
// additions in the same order as the tree over an LDS array, with two
// barriers in place of ten.
template <class T>
__global__ __launch_bounds__(256) void hawk_sum_fold(const T* __restrict__ lanes,
                                                     T* __restrict__ gp,
                                                     unsigned* __restrict__ ticket,
                                                     T* __restrict__ out) {
    static_assert(kFoldLanes == 1024 && kGroups == 64, "four lanes a thread, one wave of group values");
    __shared__ T up128[128];
    __shared__ T up64[64];
    __shared__ unsigned last;
    const int g = blockIdx.x;
    const int t = threadIdx.x;
    const T* src = lanes + static_cast<long long>(g) * kFoldLanes;
    const T x0 = src[t], x1 = src[t + 256], x2 = src[t + 512], x3 = src[t + 768];
    T a = (x0 + x2) + (x1 + x3);                 // w = 512 (lanes t and t+256), then w = 256
    if (t >= 128) up128[t - 128] = a;
    __syncthreads();
    if (t < 128) a = a + up128[t];               // w = 128
    if (t >= 64 && t < 128) up64[t - 64] = a;
    __syncthreads();
    if (t < 64) {
        a = a + up64[t];                         // w = 64
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) a = a + __shfl_down(a, w, 64);
        if (t == 0) {
            gp[g] = a;
            __threadfence();
            last = atomicAdd(ticket, 1u);
        }
    }
    __syncthreads();
    if (last != kGroups - 1 || t >= 64) return;
    __threadfence();   // acquire: every group's gp store is visible
    T b = __builtin_nontemporal_load(gp + t);
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) b = b + __shfl_down(b, w, 64);
    if (t == 0) {
        *out = b;
        *ticket = 0u;
    }
}

// ---------------------------------------------------------------------------
// Banded reductions (the banded scalar mode; reference hawk/emit/wrapper.py:140
// `BANDED`, hawk/emit/team.py:26-49 and :225-245): every partial is a band, a
// normalised double-double (h, l) with |l| <= ulp(h)/2, folded in the same
// fixed order as the float64 stages, and the stored cell is the final band's
// h.  Two bands join as in Hida, Li and Bailey's QD library: TwoSum of the
// leading and of the low parts and two quick renormalisations; Knuth's TwoSum
// is exact in either operand order, so the add is symmetric.  A virtual
// lane's run of terms accumulates by Neumaier's compensated sum and becomes a
// band at its end (lane_add, lane_band).  A non-finite leading sum drops the
// low part, so Inf and NaN follow IEEE through h.
// ---------------------------------------------------------------------------
struct Band {
    double h, l;
};

__device__ __forceinline__ Band band_two(double a, double b) {
    const double s = a + b;
    const double bb = s - a;
    return Band{s, (a - (s - bb)) + (b - bb)};
}

__device__ __forceinline__ Band band_quick(double a, double b) {
    const double s = a + b;
    return Band{s, b - (s - a)};
}

// A virtual lane's run of rows (the banded ordered sum): Neumaier's
// compensated sum, the running sum s one addition a row and each addition's
// exact error added to c beside it, so a row costs the chain one dependent
// add; renormalised into a band once, at the run's end, by TwoSum of (s, c);
// a non-finite s drops c.
struct LaneSum {
    double s, c;
};

__device__ __forceinline__ void lane_add(LaneSum& a, double x) {
    // the error by TwoSum: the exact error of t = s + x whichever operand is
    // larger, so the same value as Neumaier's branch on |s| >= |x|, without a
    // compare and select
    const double t = a.s + x;
    const double bb = t - a.s;
    a.c = a.c + ((a.s - (t - bb)) + (x - bb));
    a.s = t;
}

__device__ __forceinline__ Band lane_band(LaneSum a) {
    const Band b = band_two(a.s, a.c);
    const bool finite = (a.s - a.s) == 0.0;
    return Band{finite ? b.h : a.s, finite ? b.l : 0.0};
}

__device__ __forceinline__ Band band_add(Band a, Band b) {
    Band s = band_two(a.h, b.h);
    if (!((s.h - s.h) == 0.0)) return Band{s.h, 0.0};
    const Band t = band_two(a.l, b.l);
    s = band_quick(s.h, s.l + t.h);
    return band_quick(s.h, s.l + t.l);
}

// The banded ordered sum's geometry, reference hawk/emit/team.py:26-30
// (BAND_LANES, BAND_VIRTUAL_LANES) and :225-245: group g's 128 virtual lanes
// l = g*128 + t each add rows l, l + 8192, ... as terms of one band.
constexpr int kBandLanes = 128;
constexpr int kBandVirtual = kBandLanes * kGroups;   // 8192
constexpr size_t kBandLanesBytes = sizeof(Band) * kBandVirtual;
constexpr size_t kBandGpBytes = sizeof(Band) * kGroups;
constexpr size_t kBandSumScratch = kBandLanesBytes + kBandGpBytes + 256;

// One workgroup per kBandChains virtual lanes: wave 0 is the chains (lane c
// < kBandChains adds column c of each stage, kBandStage row blocks of
// kBandChains contiguous values, to its lane sum, row after row) and the
// kBandLoaders threads after it read the rows.  A stage reaches the loaders'
// registers kBandAhead stages before the chains add it and their LDS ring
// (kBandSlots stages) two stages before; the chain wave reads each stage into
// registers one stage ahead, so neither the rows' nor the LDS's latency
// meets the chain.  Clears the fold's ticket one launch ahead of the fold.
// Measured on MI355X at N = 2^26: 0.204 ms, against 0.227 for a two-stage
// ring of 64-row stages read after each barrier with 256 loaders, and 0.209
// with 256 loaders here (two loader waves leave the chains' SIMD to them).
// Chains spread over two or four waves measured slower (282 and 358 us
// against 236 in the two-stage form).
constexpr int kBandChains = 32;
constexpr int kBandStage = 32;
constexpr int kBandSlots = 3;
constexpr int kBandAhead = 6;                 // stages a row read has before its chain adds it
constexpr int kBandSets = kBandAhead - 2;     // loader register sets: stage s read at s - 6, stored at s - 2
constexpr int kBandLoaders = 128;
constexpr int kBandThreads = 64 + kBandLoaders;
constexpr int kBandPer = kBandStage * kBandChains / kBandLoaders;   // values a loader reads a stage
static_assert(kBandVirtual % kBandChains == 0 && kBandSets == 4, "whole workgroups of chains, four register sets");

__global__ __launch_bounds__(kBandThreads) void hawk_band_sum_lanes(const double* __restrict__ u, long long n,
                                                                     Band* __restrict__ lanes,
                                                                     unsigned* __restrict__ ticket) {
    __shared__ double buf[kBandSlots][kBandStage * kBandChains];
    const int t = threadIdx.x;
    const bool loader = t >= 64;
    const int lt = t - 64;
    const bool chain = t < kBandChains;
    const long long l0 = static_cast<long long>(blockIdx.x) * kBandChains;
    if (blockIdx.x == 0 && t == 0) *ticket = 0u;
    // row blocks of lane l0, the workgroup's longest lane, and its stages
    const long long blocks = n > l0 ? (n - l0 + kBandVirtual - 1) / kBandVirtual : 0;
    const long long stages = (blocks + kBandStage - 1) / kBandStage;
    double ld[kBandSets][kBandPer];
    auto load = [&](long long st, double (&reg)[kBandPer]) {
        if (!loader || st >= stages) return;
#pragma unroll
        for (int q = 0; q < kBandPer; ++q) {
            const int i = lt + q * kBandLoaders;
            const long long r = (st * kBandStage + i / kBandChains) * kBandVirtual + l0 + i % kBandChains;
            reg[q] = r < n ? __builtin_nontemporal_load(u + r) : 0.0;
        }
    };
    auto store = [&](long long st, const double (&reg)[kBandPer]) {
        if (!loader || st >= stages) return;
        double* slot = buf[st % kBandSlots];
#pragma unroll
        for (int q = 0; q < kBandPer; ++q) slot[lt + q * kBandLoaders] = reg[q];
    };
    const long long mine = chain && l0 + t < n ? (n - l0 - t + kBandVirtual - 1) / kBandVirtual : 0;
    LaneSum acc{0.0, 0.0};
    double v[2][kBandStage];
    auto fetch = [&](long long st, double (&v)[kBandStage]) {
        if (!chain || st >= stages) return;
        const double* slot = buf[st % kBandSlots];
#pragma unroll
        for (int k = 0; k < kBandStage; ++k) v[k] = slot[k * kBandChains + t];
    };
    auto add = [&](long long st, const double (&v)[kBandStage]) {
        if (!chain) return;
        const long long left = mine - st * kBandStage;
        if (left >= kBandStage) {
#pragma unroll
            for (int k = 0; k < kBandStage; ++k) lane_add(acc, v[k]);
        } else {
#pragma unroll
            for (int k = 0; k < kBandStage; ++k)
                if (k < left) lane_add(acc, v[k]);
        }
    };
    // stages 0 .. 3 into the loaders' registers, 0 and 1 into the ring
#pragma unroll
    for (int j = 0; j < kBandSets; ++j) load(j, ld[j]);
    store(0, ld[0]);
    store(1, ld[1]);
    load(kBandSets, ld[0]);
    load(kBandSets + 1, ld[1]);
    __syncthreads();
    fetch(0, v[0]);
    // iteration s: the chains read stage s + 1 and add stage s; the loaders
    // store stage s + 2 (set (s + 2) % 4) and read stage s + 6 into that set
    for (long long s0 = 0; s0 < stages; s0 += kBandSets) {
#pragma unroll
        for (int j = 0; j < kBandSets; ++j) {
            const long long s = s0 + j;
            if (s < stages) {
                fetch(s + 1, v[(j + 1) & 1]);
                add(s, v[j & 1]);
                store(s + 2, ld[(j + 2) % kBandSets]);
                load(s + kBandAhead, ld[(j + 2) % kBandSets]);
            }
            __syncthreads();
        }
    }
    if (chain) lanes[l0 + t] = lane_band(acc);
}

// Group g's 128 lane bands by the halving tree into gp[g]; the last group
// to finish folds the 64 group bands by the same tree and stores h.
__global__ __launch_bounds__(256) void hawk_band_sum_fold(const Band* __restrict__ lanes, Band* __restrict__ gp,
                                                          unsigned* __restrict__ ticket, double* __restrict__ out) {
    __shared__ Band sh[kBandLanes];
    __shared__ unsigned last;
    const int g = blockIdx.x;
    const int t = threadIdx.x;
    for (int i = t; i < kBandLanes; i += 256) sh[i] = lanes[g * kBandLanes + i];
    __syncthreads();
    for (int w = kBandLanes / 2; w > 0; w >>= 1) {
        for (int i = t; i < w; i += 256) sh[i] = band_add(sh[i], sh[i + w]);
        __syncthreads();
    }
    if (t == 0) {
        gp[g] = sh[0];
        __threadfence();
        last = atomicAdd(ticket, 1u);
    }
    __syncthreads();
    if (last != kGroups - 1) return;
    __threadfence();
    if (t < kGroups) {
        sh[t].h = __builtin_nontemporal_load(&gp[t].h);
        sh[t].l = __builtin_nontemporal_load(&gp[t].l);
    }
    __syncthreads();
    for (int w = kGroups / 2; w > 0; w >>= 1) {
        if (t < w) sh[t] = band_add(sh[t], sh[t + w]);
        __syncthreads();
    }
    if (t == 0) {
        *out = sh[0].h;
        *ticket = 0u;
    }
}

// ---------------------------------------------------------------------------
// The default-policy sample sum's finish.  The per-sample stage leaves one
// compensated (hi, comp) pair per row of 32 samples; the cell is those rows
// folded in the canonical ordered tree of reference hawk/_cells.py:71-119:
// leaves of 4096 rows, each leaf's 256 slots adding rows slot, slot + 256,
// ... (16 terms) with Neumaier's compensated add, the leaf's slots folded by
// the halving tree, then the leaves folded pairwise level by level (an odd
// last one carried up), and hi + comp at the end.  A non-finite partial drops
// its compensation, so Inf and NaN follow IEEE through hi.
// ---------------------------------------------------------------------------
constexpr int kRowSlots = 256;
constexpr int kRowTerms = 16;
constexpr long long kRowLeaf = static_cast<long long>(kRowSlots) * kRowTerms;

template <class T>
__device__ __forceinline__ bool finite_bits(T x) { return (x - x) == T(0); }

// The exact residual of s == a + b, a zero residual +0, NaN when s is not
// finite (reference hawk/_cells.py:46-52, Fast2Sum on the operands ordered by
// magnitude).  Knuth's TwoSum gives the same exact residual for any finite
// a and b without the ordering's compare and selects.
template <class T>
__device__ __forceinline__ T two_sum_err(T a, T b, T s) {
    const T bb = s - a;
    return finite_bits(s) ? ((a - (s - bb)) + (b - bb)) + T(0) : T(__builtin_nan(""));
}

// Neumaier's add of (x, xc) onto (h, c) (reference hawk/_cells.py:55-58).
template <class T>
__device__ __forceinline__ void neumaier_add(T& h, T& c, T x, T xc) {
    const T s = h + x;
    const bool fin = finite_bits(s);
    c = fin ? c + two_sum_err(h, x, s) : T(0);
    c = fin ? c + xc : T(0);
    h = s;
}

// Two partials combined (reference hawk/_cells.py:61-63).
template <class T>
__device__ __forceinline__ void pair_add(T& h, T& c, T h2, T c2) {
    const T s = h + h2;
    c = finite_bits(s) ? (c + c2) + two_sum_err(h, h2, s) : T(0);
    h = s;
}

// A reduction's finish: its rows (hi, and comp or a band's low parts), its cell
// and its rule.  Every reduction of a stage has the same number of rows, so one
// launch folds the leaves of all of them and one their levels (one launch in
// all where the rows are a single leaf): five reductions of a stage took ten
// launches, 9 to 10 us a reduction.
enum RowsOp { kRowsSum = 0, kRowsMax = 1, kRowsMin = 2, kRowsBand = 3 };
struct RowsJob {
    const void* hi;
    const void* lo;
    void* out;
    int op;
};
constexpr int kRowsJobs = 16;                    // reductions a launch takes
struct RowsJobs {
    RowsJob job[kRowsJobs];
};

// The rule of each reduction over partials (h, c): `first` of a slot's first
// row, `add` of a further row, `join` of two partials, and the cell's `value`.
//
// * the default sum: Neumaier's add and the compensated join (above);
// * hawk.max / hawk.min (reference hawk/_cells.py:66-71 and `finish`): every
//   add the extreme a > b ? a : b (max) or a < b ? a : b (min) of (the earlier
//   partial, the later); exact, and a NaN partial on the left gives way to the
//   right one;
// * the banded sum: every add a band add, the cell the final band's h.
template <class T, int Op>
struct RowsRule {
    __device__ static __forceinline__ T first_c(T h, T c) { return Op == kRowsSum && !finite_bits(h) ? T(0) : c; }
    __device__ static __forceinline__ void add(T& h, T& c, T x, T xc) {
        if constexpr (Op == kRowsSum) neumaier_add(h, c, x, xc);
        else join(h, c, x, xc);
    }
    __device__ static __forceinline__ void join(T& h, T& c, T h2, T c2) {
        if constexpr (Op == kRowsSum) {
            pair_add(h, c, h2, c2);
        } else if constexpr (Op == kRowsBand) {
            const Band b = band_add(Band{h, c}, Band{h2, c2});
            h = b.h;
            c = b.l;
        } else {
            h = Op == kRowsMax ? (h > h2 ? h : h2) : (h < h2 ? h : h2);
        }
    }
    __device__ static __forceinline__ T value(T h, T c) { return Op == kRowsSum && finite_bits(h) ? h + c : h; }
};

// Leaf j of a reduction: rows [j*4096, min((j+1)*4096, rows)), thread = slot.
// T is the rows' type: the finish runs in it, as the reference's finish runs in
// the rows' dtype.  A slot's sixteen rows load together, then add in order; the
// tree's levels 128 and 64 cross waves through LDS, 32 .. 1 run in one wave.  A
// slot past the rows joins nothing.
template <class T, int Op>
__device__ __forceinline__ void rows_leaf(const RowsJob& job, long long rows, T* buf, long long leaves, T* sh, T* sc) {
    typedef RowsRule<T, Op> Rule;
    constexpr bool kPair = Op == kRowsSum || Op == kRowsBand;
    const int s = threadIdx.x;
    const long long lo = static_cast<long long>(blockIdx.x) * kRowLeaf;
    const T* hi = static_cast<const T*>(job.hi) + lo;
    const T* comp = kPair ? static_cast<const T*>(job.lo) + lo : nullptr;
    const long long rest = rows - lo;
    const int cnt = rest < kRowLeaf ? static_cast<int>(rest) : static_cast<int>(kRowLeaf);
    const int live = cnt < kRowSlots ? cnt : kRowSlots;
    T x[kRowTerms], y[kRowTerms];
#pragma unroll
    for (int k = 0; k < kRowTerms; ++k) x[k] = y[k] = T(0);
    if (cnt == kRowLeaf) {
#pragma unroll
        for (int k = 0; k < kRowTerms; ++k) {
            x[k] = hi[k * kRowSlots + s];
            if constexpr (kPair) y[k] = comp[k * kRowSlots + s];
        }
    } else {
#pragma unroll
        for (int k = 0; k < kRowTerms; ++k)
            if (k * kRowSlots + s < cnt) {
                x[k] = hi[k * kRowSlots + s];
                if constexpr (kPair) y[k] = comp[k * kRowSlots + s];
            }
    }
    T h = x[0], c = Rule::first_c(x[0], y[0]);
#pragma unroll
    for (int k = 1; k < kRowTerms; ++k)
        if (k * kRowSlots + s < cnt) Rule::add(h, c, x[k], y[k]);
    auto lim = [&](int off) { return live > off ? (off < live - off ? off : live - off) : 0; };
#pragma unroll
    for (int off = kRowSlots / 2; off > 32; off >>= 1) {
        if (s >= off && s < 2 * off) {
            sh[s] = h;
            sc[s] = c;
        }
        __syncthreads();
        if (s < lim(off)) Rule::join(h, c, sh[s + off], sc[s + off]);
    }
    if (s >= 64) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const T h2 = __shfl_down(h, off, 64), c2 = __shfl_down(c, off, 64);
        if (s < lim(off)) Rule::join(h, c, h2, c2);
    }
    if (s != 0) return;
    if (leaves == 1) {
        *static_cast<T*>(job.out) = Rule::value(h, c);
    } else {
        buf[blockIdx.x] = h;
        buf[leaves + blockIdx.x] = c;
    }
}

// The rows' rule picked once a workgroup; the band rule is double only.
#define HK_ROWS_RULE(op, call)                                  \
    if ((op) == kRowsSum) call(kRowsSum);                       \
    else if ((op) == kRowsMax) call(kRowsMax);                  \
    else if ((op) == kRowsMin) call(kRowsMin);                  \
    else if constexpr (sizeof(T) == 8) call(kRowsBand)

template <class T>
__global__ __launch_bounds__(kRowSlots) void hawk_rows_leaves(RowsJobs jobs, long long rows, T* __restrict__ buf,
                                                              long long leaves) {
    __shared__ T sh[kRowSlots], sc[kRowSlots];
    const RowsJob job = jobs.job[blockIdx.y];
    T* mine = buf + 4 * leaves * blockIdx.y;
#define HK_LEAF(op) rows_leaf<T, op>(job, rows, mine, leaves, sh, sc)
    HK_ROWS_RULE(job.op, HK_LEAF);
#undef HK_LEAF
}

// The leaves folded pairwise level by level by one workgroup a reduction: in
// the scratch's two halves while they are more than kLevelLds, then in LDS, the
// last 128 by one wave with no barrier.
constexpr int kLevelLds = 1024;
template <class T, int Op>
__device__ __forceinline__ void rows_levels(const RowsJob& job, T* buf, long long leaves, T* sh, T* sc) {
    typedef RowsRule<T, Op> Rule;
    const int t = threadIdx.x;
    T* vh = buf;
    T* vc = buf + leaves;
    T* nh = buf + 2 * leaves;
    T* nc = buf + 3 * leaves;
    long long m = leaves;
    while (m > kLevelLds) {
        const long long pairs = m / 2;
        for (long long p = t; p < pairs; p += 256) {
            T h = vh[2 * p], c = vc[2 * p];
            Rule::join(h, c, vh[2 * p + 1], vc[2 * p + 1]);
            nh[p] = h;
            nc[p] = c;
        }
        if ((m & 1) && t == 0) {
            nh[pairs] = vh[m - 1];
            nc[pairs] = vc[m - 1];
        }
        __syncthreads();
        T* th = vh; vh = nh; nh = th;
        T* tc = vc; vc = nc; nc = tc;
        m = pairs + (m & 1);
    }
    for (int p = t; p < m; p += 256) {
        sh[p] = vh[p];
        sc[p] = vc[p];
    }
    __syncthreads();
    int left = static_cast<int>(m);
    while (left > 128) {
        const int pairs = left / 2;
        T h[kLevelLds / 512], c[kLevelLds / 512];
#pragma unroll
        for (int q = 0; q < kLevelLds / 512; ++q) {
            const int p = t + 256 * q;
            if (p < pairs) {
                h[q] = sh[2 * p];
                c[q] = sc[2 * p];
                Rule::join(h[q], c[q], sh[2 * p + 1], sc[2 * p + 1]);
            } else if (p == pairs && (left & 1)) {
                h[q] = sh[left - 1];
                c[q] = sc[left - 1];
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kLevelLds / 512; ++q) {
            const int p = t + 256 * q;
            if (p < pairs + (left & 1)) {
                sh[p] = h[q];
                sc[p] = c[q];
            }
        }
        __syncthreads();
        left = pairs + (left & 1);
    }
    if (t >= 64) return;
    while (left > 1) {                       // a lane a pair; the wave's reads precede its writes
        const int pairs = left / 2;
        T h = T(0), c = T(0);
        if (t < pairs) {
            h = sh[2 * t];
            c = sc[2 * t];
            Rule::join(h, c, sh[2 * t + 1], sc[2 * t + 1]);
        }
        const T lh = sh[left - 1], lc = sc[left - 1];
        __builtin_amdgcn_wave_barrier();
        if (t < pairs) {
            sh[t] = h;
            sc[t] = c;
        }
        if ((left & 1) && t == 0) {
            sh[pairs] = lh;
            sc[pairs] = lc;
        }
        __builtin_amdgcn_wave_barrier();
        left = pairs + (left & 1);
    }
    if (t == 0) *static_cast<T*>(job.out) = Rule::value(sh[0], sc[0]);
}

template <class T>
__global__ __launch_bounds__(256) void hawk_rows_levels(RowsJobs jobs, T* __restrict__ buf, long long leaves) {
    __shared__ T sh[kLevelLds], sc[kLevelLds];
    const RowsJob job = jobs.job[blockIdx.x];
    T* mine = buf + 4 * leaves * blockIdx.x;
#define HK_LEVELS(op) rows_levels<T, op>(job, mine, leaves, sh, sc)
    HK_ROWS_RULE(job.op, HK_LEVELS);
#undef HK_LEVELS
}

// hawk.sum(x, over=<trailing lane axes>) under the default policy: key k's
// `group` consecutive values are summed as a sample sum of their own.  Rows
// of 32 run from the key's first value (a ragged last row padded with +0),
// each a compensated (hi, comp) pair by the pairs (l, l ^ 16), ..., (l, l ^ 1);
// the rows fold in the canonical tree above (leaves of 4096 rows over 256
// slots with Neumaier's add, the halving tree, the leaves pairwise level by
// level) and the key's cell is hi + comp.
//
// Eight lanes hold a row, four samples each (samples j, j + 8, j + 16, j + 24
// of lane j of the row), so a wave sums eight rows at a time: the levels 16 and
// 8 join in registers and the levels 4, 2, 1 are DPP moves, with j's bits
// reversed over the lanes (level 4 is lane ^ 1, level 2 lane ^ 2, both quad
// permutations; by level 1 a quad's lanes are equal, so the mirrored lane of
// the half row stands for lane ^ 4).  A half-wave a row with five __shfl_xor
// levels before: 20000 keys of 500 samples 42 us in float64 and 27 in float32,
// 10^6 keys of 10 262 us, 10 keys of 100000 226 us.
//
// A row or slot past the key's rows holds (+0, +0), which every add leaves as
// it is but for the sign of a zero hi, and hi + comp (comp is never -0) ends
// in +0 either way: the bits of the tree over the live rows alone.
constexpr long long kKeyedCompLeaves = kRowSlots;        // leaves a key may span

template <class T, int Ctrl>
__device__ __forceinline__ T dpp_move(T x) {
    if constexpr (sizeof(T) == 4) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), Ctrl, 0xf, 0xf, false));
    } else {
        const long long b = __double_as_longlong(x);
        const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), Ctrl, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), Ctrl, 0xf, 0xf, false);
        return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
    }
}

// The sample of its row that lane q of eight reads first, and the row's sum
// from its four samples a lane: every lane of the eight ends with the row's
// (h, c).
__device__ __forceinline__ int row_sample(int q) { return ((q & 1) << 2) | (q & 2) | ((q >> 2) & 1); }

template <class T>
__device__ __forceinline__ void row_of_eight(const T (&x)[4], T& h, T& c) {
    T h1 = x[1], c1 = T(0);
    h = x[0];
    c = T(0);
    pair_add(h, c, x[2], T(0));                             // level 16
    pair_add(h1, c1, x[3], T(0));
    pair_add(h, c, h1, c1);                                 // level 8
    pair_add(h, c, dpp_move<T, 0xb1>(h), dpp_move<T, 0xb1>(c));       // level 4: quad_perm 1,0,3,2
    pair_add(h, c, dpp_move<T, 0x4e>(h), dpp_move<T, 0x4e>(c));       // level 2: quad_perm 2,3,0,1
    pair_add(h, c, dpp_move<T, 0x141>(h), dpp_move<T, 0x141>(c));     // level 1: row_half_mirror
}

// Keys of at most 64 rows (2048 samples), a wave a key in Steps = 1, 2, 4 or 8
// steps of eight rows; a key of at most four rows shares its wave's step with
// 8 / G - 1 others (G = 2^ceil(log2 rows)).  Row 8 s + g is step s's lanes
// 8g .. 8g + 7, so the halving tree's levels 32, 16 and 8 join steps in
// registers and the levels 4, 2 and 1 lane groups.
template <class T, int Steps>
__global__ __launch_bounds__(256) void hawk_keyed_comp_wave(const T* __restrict__ u, long long group, int G,
                                                            long long keys, T* __restrict__ out) {
    const int lane = threadIdx.x & 63, g = lane >> 3, j = row_sample(lane & 7);
    const long long wave = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const long long k = Steps > 1 ? wave : wave * (8 / G) + g / G;
    const int row = Steps > 1 ? g : g & (G - 1);
    const T* __restrict__ mine = u + (k < keys ? k : 0) * group;
    const int len = k < keys ? static_cast<int>(group) : 0;
    const T* __restrict__ from = mine + row * 32 + j;
    T x[Steps][4];
#pragma unroll
    for (int s = 0; s < Steps; ++s) {
        if (Steps > 1 && (s + 1) * 256 <= len) {            // eight whole rows of the wave's key
#pragma unroll
            for (int v = 0; v < 4; ++v) x[s][v] = __builtin_nontemporal_load(from + s * 256 + 8 * v);
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                x[s][v] = s * 256 + row * 32 + j + 8 * v < len ? __builtin_nontemporal_load(from + s * 256 + 8 * v)
                                                               : T(0);
        }
    }
    T h[Steps], c[Steps];
#pragma unroll
    for (int s = 0; s < Steps; ++s) row_of_eight<T>(x[s], h[s], c[s]);
#pragma unroll
    for (int off = Steps / 2; off > 0; off >>= 1)
#pragma unroll
        for (int s = 0; s < off; ++s) pair_add(h[s], c[s], h[s + off], c[s + off]);
#pragma unroll
    for (int off = 4; off > 0; off >>= 1)
        if (Steps > 1 || G > off) pair_add(h[0], c[0], __shfl_xor(h[0], 8 * off, 64), __shfl_xor(c[0], 8 * off, 64));
    if ((lane & 7) == 0 && row == 0 && k < keys) out[k] = finite_bits(h[0]) ? h[0] + c[0] : h[0];
}

// Longer keys, a workgroup of Waves waves a key: lane group i of 8 * Waves
// keeps slots i, i + 8 Waves, ... of each leaf in registers and adds their rows
// in order; the slots join in registers, then over the groups in the first
// wave.  Four waves where the keys fill the chip, sixteen where they do not or
// are long (4 / 16 waves, fp64: 2000 keys of 5000 samples 19.4 / 21.7 us, 600
// of 20000 28.1 / 23.6, 10 of 100000 79 / 29).
template <class T, int Waves>
__global__ __launch_bounds__(64 * Waves) void hawk_keyed_comp(const T* __restrict__ u, long long group,
                                                              T* __restrict__ out) {
    constexpr int kGroups8 = 8 * Waves;                  // lane groups
    constexpr int kOwn = kRowSlots / kGroups8;           // slots a lane group keeps
    static_assert(kGroups8 == 32 || kGroups8 == 128, "a wave folds the groups' slots");
    __shared__ T sh[kGroups8], sc[kGroups8], lh[kKeyedCompLeaves], lc[kKeyedCompLeaves];
    const int t = threadIdx.x, lane = t & 63, j = row_sample(t & 7), mine8 = t >> 3;
    const int wave8 = __builtin_amdgcn_readfirstlane(mine8 & ~7);        // the wave's first lane group
    const T* __restrict__ mine = u + static_cast<long long>(blockIdx.x) * group;
    const long long rows = (group + 31) / 32;
    const long long leaves = (rows + kRowLeaf - 1) / kRowLeaf;
    for (long long leaf = 0; leaf < leaves; ++leaf) {
        const long long first = leaf * kRowLeaf;
        const int cnt = static_cast<int>(rows - first < kRowLeaf ? rows - first : kRowLeaf);
        T h[kOwn], c[kOwn];
#pragma unroll
        for (int i = 0; i < kOwn; ++i) h[i] = c[i] = T(0);
        for (int r0 = 0; r0 < cnt; r0 += kRowSlots) {
            T x[kOwn][4];
            const long long base = (first + r0) * 32;
            const T* __restrict__ from = mine + base + mine8 * 32 + j;
            if (base + kRowSlots * 32 <= group) {               // whole rows, a row a slot
#pragma unroll
                for (int i = 0; i < kOwn; ++i)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        x[i][v] = __builtin_nontemporal_load(from + kGroups8 * i * 32 + 8 * v);
            } else {
                const int left = static_cast<int>(group - base) - mine8 * 32 - j;
#pragma unroll
                for (int i = 0; i < kOwn; ++i)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        x[i][v] = kGroups8 * i * 32 + 8 * v < left
                                      ? __builtin_nontemporal_load(from + kGroups8 * i * 32 + 8 * v) : T(0);
            }
#pragma unroll
            for (int i = 0; i < kOwn; ++i) {
                if (r0 + wave8 + kGroups8 * i >= cnt) break;             // no rows for the whole wave
                T rh, rc;
                row_of_eight<T>(x[i], rh, rc);
                neumaier_add(h[i], c[i], rh, rc);
            }
        }
#pragma unroll
        for (int off = kOwn / 2; off > 0; off >>= 1)
#pragma unroll
            for (int i = 0; i < off; ++i) pair_add(h[i], c[i], h[i + off], c[i + off]);
        if ((t & 7) == 0) {
            sh[mine8] = h[0];
            sc[mine8] = c[0];
        }
        __syncthreads();
        if (t < 64) {
            T a = lane < kGroups8 ? sh[lane] : T(0), b = lane < kGroups8 ? sc[lane] : T(0);
            if constexpr (kGroups8 == 128) pair_add(a, b, sh[lane + 64], sc[lane + 64]);
#pragma unroll
            for (int off = kGroups8 == 128 ? 32 : 16; off > 0; off >>= 1)
                pair_add(a, b, __shfl_down(a, off, 64), __shfl_down(b, off, 64));
            if (t == 0) {
                lh[leaf] = a;
                lc[leaf] = b;
            }
        }
        __syncthreads();
    }
    if (t == 0) {
        long long m = leaves;
        while (m > 1) {               // in place: pair p reads slots 2p, 2p + 1 >= p
            const long long pairs = m / 2;
            for (long long p = 0; p < pairs; ++p) {
                T h = lh[2 * p], c = lc[2 * p];
                pair_add(h, c, lh[2 * p + 1], lc[2 * p + 1]);
                lh[p] = h;
                lc[p] = c;
            }
            if (m & 1) {
                lh[pairs] = lh[m - 1];
                lc[pairs] = lc[m - 1];
            }
            m = pairs + (m & 1);
        }
        out[blockIdx.x] = finite_bits(lh[0]) ? lh[0] + lc[0] : lh[0];
    }
}

// ---------------------------------------------------------------------------
// Keyed fixed-tree sum: hawk.sum(x, over=<trailing lane axes>, policy=
// "ordered").  Key k's rows are the `group` consecutive values
// u[k*group .. (k+1)*group), and each key takes the ordered sum's tree
// (reference hawk/emit/team.py:115-205 with its gp stage): virtual lane l of
// 65536 adds rows l, l + 65536, ... from +0.0, groups of 1024 lanes fold by
// the halving tree, then the 64 group values by the same tree.
//
// Only the first lv = min(group, 65536) lanes of a key can hold rows; the
// others are +0.0, and so are the groups past ceil(lv / 1024).  No lane value
// or tree sum is ever -0.0 (each starts at +0.0; a round-to-nearest sum is
// -0.0 only from two -0.0 operands), so adding +0.0 is the identity and the
// trees need only the lanes and group values that hold rows, the others +0.0:
// the bits of the full trees.
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ int pow2_at_least(long long x) {
    int p = 1;
    while (p < x) p <<= 1;
    return p;
}

// The halving tree over a wave's lanes, lane i adding lane i + w's value for
// w = P/2 .. 1 (P a power of 2; only lanes below w carry on): lane 0 of each
// P lanes ends with their tree's sum.  Rows of 16 lanes shift by DPP.
template <class T>
__device__ __forceinline__ T wave_tree(T x, int P) {
    if (P > 32) x = x + __shfl_down(x, 32, 64);
    if (P > 16) x = x + __shfl_down(x, 16, 64);
    if (P > 8) x = x + dpp_move<T, 0x108>(x);            // row_shl:8
    if (P > 4) x = x + dpp_move<T, 0x104>(x);
    if (P > 2) x = x + dpp_move<T, 0x102>(x);
    if (P > 1) x = x + dpp_move<T, 0x101>(x);
    return x;
}

// 64 J consecutive values from u, `left` of them live: lane l's x[j] is value
// l + 64 j, or +0.0 past the live ones.  A whole run loads without a test a
// value: testing each took 16384 keys of 4096 rows from 75 to 110 us.
template <class T, int J>
__device__ __forceinline__ void wave_rows(T (&x)[J], const T* __restrict__ u, long long left) {
    const int lane = threadIdx.x & 63;
    if (left >= 64 * J) {
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = __builtin_nontemporal_load(u + lane + 64 * j);
        return;
    }
    const int most = static_cast<int>(left);
#pragma unroll
    for (int j = 0; j < J; ++j) x[j] = lane + 64 * j < most ? __builtin_nontemporal_load(u + lane + 64 * j) : T(0);
}

// The halving tree over 64 J values held as wave_rows holds them: the levels
// from 32 J down to 64 join registers and the rest are wave_tree's, with no LDS
// and no barrier.  Lane 0 returns the sum.
template <class T, int J>
__device__ __forceinline__ T rows_tree(T (&v)[J]) {
#pragma unroll
    for (int off = J / 2; off > 0; off >>= 1)
#pragma unroll
        for (int j = 0; j < off; ++j) v[j] = v[j] + v[j + off];
    return wave_tree(v[0], 64);
}

// Keys of 65 to 1024 rows (64 J or fewer): a wave a key.  A workgroup a key
// with the tree through LDS took 103 us where this takes 23 (100000 keys of 100
// rows, fp64) and 25 where it takes 11.5 (20000 of 500: 7.0 TB/s).
template <class T, int J>
__global__ __launch_bounds__(256) void hawk_keyed_wave(const T* __restrict__ u, long long group, long long keys,
                                                       T* __restrict__ out) {
    const long long k = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (k >= keys) return;                               // the whole wave
    T v[J];
    wave_rows<T, J>(v, u + k * group, group);
#pragma unroll
    for (int j = 0; j < J; ++j) v[j] = T(0) + v[j];
    const T s = rows_tree<T, J>(v);
    if ((threadIdx.x & 63) == 0) out[k] = s;
}

// Keys of at most 65536 rows: a workgroup a key, its waves the key's groups of
// 1024 lanes in turn (the next group's rows in flight during a group's tree),
// then the group values' tree in the first wave.  Four waves where the keys
// fill the chip; sixteen for few keys of at most 16 groups, and for the plain
// ordered sum of at most 16384 rows.
template <class T, int Waves>
__global__ __launch_bounds__(64 * Waves) void hawk_keyed_rows(const T* __restrict__ u, long long group,
                                                              T* __restrict__ out) {
    __shared__ T gp[kGroups];
    const int t = threadIdx.x;
    const int used = static_cast<int>((group + kFoldLanes - 1) / kFoldLanes);
    const T* mine = u + static_cast<long long>(blockIdx.x) * group;
    T x[16];
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    if (w < used) wave_rows<T, 16>(x, mine + w * kFoldLanes, group - w * kFoldLanes);
    for (int g = w; g < used; g += Waves) {
        T v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = T(0) + x[j];
        if (g + Waves < used) wave_rows<T, 16>(x, mine + (g + Waves) * kFoldLanes, group - (g + Waves) * kFoldLanes);
        const T s = rows_tree<T, 16>(v);
        if ((t & 63) == 0) gp[g] = s;
    }
    __syncthreads();
    if (t < 64) {
        const T total = wave_tree(t < used ? gp[t] : T(0), kGroups);
        if (t == 0) out[blockIdx.x] = total;
    }
}

// Longer keys, and few keys of more than 16 groups: a wave a (key, group),
// virtual lane m adding rows m, m + 65536, ... (the next ones in flight), each
// group's sum into gp[key][group]; then a wave a key for the group values'
// tree.
template <class T>
__global__ __launch_bounds__(256) void hawk_keyed_groups(const T* __restrict__ u, long long group, int used,
                                                         long long keys, T* __restrict__ gp) {
    const long long i = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const long long k = i / used, g = i % used;
    if (k >= keys) return;                               // the whole wave
    const T* mine = u + k * group + g * kFoldLanes;
    const long long rows = group - g * kFoldLanes;
    T x[16], v[16];
    wave_rows<T, 16>(x, mine, rows);
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = T(0);
    for (long long r = 0; r < rows; r += kVirtualLanes) {
        T a[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = x[j];
        if (r + kVirtualLanes < rows) wave_rows<T, 16>(x, mine + r + kVirtualLanes, rows - r - kVirtualLanes);
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = v[j] + a[j];
    }
    const T s = rows_tree<T, 16>(v);
    if ((threadIdx.x & 63) == 0) gp[k * kGroups + g] = s;
}
template <class T>
__global__ __launch_bounds__(256) void hawk_keyed_top(const T* __restrict__ gp, int used, long long keys,
                                                      T* __restrict__ out) {
    const long long k = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (k >= keys) return;                               // the whole wave
    const int lane = threadIdx.x & 63;
    const T s = wave_tree(lane < used ? gp[k * kGroups + lane] : T(0), kGroups);
    if (lane == 0) out[k] = s;
}

// Keys of at most 64 rows: a wave holds 64 / P keys, P = 2^ceil(log2 group),
// in segments of P lanes (lane j of a segment holds row j, 0.0 + u, or +0.0
// past the key's rows), and each segment runs the halving tree.  The group
// tree has one value, which it returns unchanged.  A wave takes four such sets,
// their loads in flight together.
constexpr int kSmallSets = 4;
template <class T>
__global__ __launch_bounds__(256) void hawk_keyed_small(const T* __restrict__ u, long long group, int P,
                                                        long long keys, T* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int per_wave = 64 / P;
    const int j = lane & (P - 1);
    const long long k0 = (static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * (kSmallSets * per_wave) +
                         lane / P;
    T x[kSmallSets];
#pragma unroll
    for (int q = 0; q < kSmallSets; ++q) {
        const long long k = k0 + q * per_wave;
        x[q] = k < keys && j < group ? T(0) + __builtin_nontemporal_load(u + k * group + j) : T(0);
    }
#pragma unroll
    for (int q = 0; q < kSmallSets; ++q) x[q] = wave_tree(x[q], P);
#pragma unroll
    for (int q = 0; q < kSmallSets; ++q)
        if (j == 0 && k0 + q * per_wave < keys) out[k0 + q * per_wave] = x[q];
}

// ---------------------------------------------------------------------------
// Keyed ordered scatter.
//
// parts[b][k] is the in-lane-order sum (from +0.0) of chunk b's values with
// key k; cell k then adds parts[0][k], parts[1][k], ... in chunk order from
// +0.0 and adds that onto target[k].  Two walks make those additions, the
// split walk (a workgroup a chunk) and the wide walk (a workgroup a chunk and
// key range, for few chunks or many cells); in both every accumulator is in
// LDS while its chunk is walked.
// ---------------------------------------------------------------------------
constexpr int kScatterChunks = 256;    // reference hawk/_lane_bind.py:108
constexpr int kWalkThreads = 1024;
constexpr int kWalkWaves = kWalkThreads / 64;
constexpr int kWalkItems = 4;                      // lanes per thread per tile
constexpr int kTile = kWalkThreads * kWalkItems;   // 4096 lanes per tile

// Inclusive scan over the 64 lanes of a wave in DPP moves, no LDS: within
// each row of 16 lanes by row shifts 1, 2, 4, 8 (a lane past the row's start
// adds 0), then row 15's total into rows 1 and 3 and lane 31's into rows 2
// and 3 (row broadcasts).
__device__ __forceinline__ unsigned wave_inclusive_scan(unsigned x) {
    x += __builtin_amdgcn_update_dpp(0u, x, 0x111, 0xf, 0xf, false);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0u, x, 0x112, 0xf, 0xf, false);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0u, x, 0x114, 0xf, 0xf, false);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0u, x, 0x118, 0xf, 0xf, false);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0u, x, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1, 3
    x += __builtin_amdgcn_update_dpp(0u, x, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2, 3
    return x;
}

// Lane base + wave*256 + j*64 + lane goes to thread slot j: every load
// instruction of a wave reads 64 consecutive lanes.  Lanes past `hi` read as
// the skip key -1.
template <class T>
__device__ __forceinline__ void walk_load(const int* __restrict__ key, const T* __restrict__ v, long long base,
                                          long long hi, int (&kk)[kWalkItems], T (&vv)[kWalkItems]) {
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < kWalkItems; ++j) {
        const long long i = base + wave * (kWalkItems * 64) + j * 64 + lane;
        const bool in = i < hi;
        kk[j] = in ? __builtin_nontemporal_load(key + i) : -1;
        vv[j] = in ? __builtin_nontemporal_load(v + i) : T(0);
    }
}

// Cell c adds its chunk partials in chunk order from +0.0, then onto the
// target: target[c] += sum (reference hawk/emit/team.py:437-460).  Two blocks
// of kAhead chunks are in flight while a third is added: 64 loads a thread,
// since a grid of one thread per cell (65536 at the split walk's largest)
// holds only a wave or two per SIMD to cover HBM's latency.  Few: at most
// kAhead chunks, one block, by the groups of 8 chunks it holds.  Otherwise a
// whole block reads all its chunks with no test among the loads (256 chunks,
// fp64, every block by groups / this: 64 cells 13.6 / 7.5 us, 1000 cells 15.7 /
// 10.2, 65536 cells 28.5 / 24.6; with both forms in one kernel, 16 chunks of
// 262144 cells took 9.5 us instead of 8.3).
constexpr int kAhead = 32;
template <class T, bool Few>
__global__ __launch_bounds__(256) void hawk_scatter_cells(const T* __restrict__ parts, long long cells,
                                                          int chunks, T* __restrict__ target) {
    const long long c = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    if (c >= cells) return;
    auto fetch = [&](int b, T (&x)[kAhead]) {
        if (!Few && b + kAhead <= chunks) {
#pragma unroll
            for (int q = 0; q < kAhead; ++q) x[q] = parts[static_cast<long long>(b + q) * cells + c];
            return;
        }
#pragma unroll
        for (int q = 0; q < kAhead; ++q) x[q] = T(0);
#pragma unroll
        for (int q8 = 0; q8 < kAhead; q8 += 8) {
            if (b + q8 >= chunks) break;                      // the whole grid
#pragma unroll
            for (int q = q8; q < q8 + 8; ++q) {
                // past the last chunk a partial reads as +0.0, which adds
                // nothing to a sum that is never -0.0
                const int bq = b + q < chunks ? b + q : chunks - 1;
                const T p = parts[static_cast<long long>(bq) * cells + c];
                x[q] = b + q < chunks ? p : T(0);
            }
        }
    };
    T x0[kAhead];
    T s = T(0);
    fetch(0, x0);
    if constexpr (Few) {
#pragma unroll
        for (int q = 0; q < kAhead; ++q) s = s + x0[q];
    } else {
        T x1[kAhead];
        fetch(kAhead, x1);
        for (int b = 0; b < chunks; b += kAhead) {
            T x2[kAhead];
            fetch(b + 2 * kAhead, x2);
#pragma unroll
            for (int q = 0; q < kAhead; ++q) s = s + x0[q];
#pragma unroll
            for (int q = 0; q < kAhead; ++q) {
                x0[q] = x1[q];
                x1[q] = x2[q];
            }
        }
    }
    target[c] = target[c] + s;
}

// ---- the split walk: the ordered scatter into at most 65536 cells ----------
// Each (chunk, key) sum in lane order from +0.0, every accumulator in LDS:
//
// * hawk_split_hot: one workgroup per chunk, keys [0, kSplitHot) in LDS.  Each
//   tile of 4096 lanes is split stably into buckets in one pass: window keys
//   0..31 each a bucket of their own, keys 32..kSplitHot-1 fifteen classes by
//   (key - 32) % 15, and keys from kSplitHot up one bucket per tail range of
//   kTailRange keys.  Waves 0..7 then add the head buckets' chains, four a
//   wave, and wave w > 0 folds class w - 1 (64 entries at a time: equal keys
//   find each other, and the lowest lane adds its group in lane order onto the
//   key's accumulator; a wave's LDS operations complete in issue order, so a
//   key's groups meet the accumulator window after window).
//   The tail buckets go from registers to the tile's slot of the chunk's bin,
//   with the offset of each range.
// * hawk_split_tail: one workgroup of 8 waves per (chunk, tail range), the
//   range's keys in LDS, two workgroups a CU; it reads the range's segment of
//   every slot in tile order (lane order), a batch of 2048 entries at a time,
//   and folds them in eight classes by key & 7 as above.
//
// Both write every key's accumulator of their window to parts[b] (+0.0 for a
// key no lane named); hawk_scatter_cells then adds the partials in chunk order.
constexpr int kSplitHot = 12288;                 // keys hawk_split_hot keeps in LDS (96 KiB of accumulators)
constexpr int kTailRange = 6144;                 // keys a hawk_split_tail workgroup keeps in LDS (48 KiB)
constexpr long long kSplitCells = 65536;         // the split walk's largest cell count
constexpr int kSplitMaxRanges = static_cast<int>((kSplitCells - kSplitHot + kTailRange - 1) / kTailRange);  // 9
constexpr int kSplitHeads = 32;                  // buckets 0..31: window keys 0..31, a chain each
constexpr int kSplitClassBase = kSplitHeads;     // classes from bucket 32 (hot: 32..46; tail: 32..39)
constexpr int kSplitTailBase = kSplitClassBase + 16;   // 48..56: hawk_split_hot's tail ranges
constexpr int kSplitNone = 63;                   // a lane that adds nothing (skip key, bad key, padding)
constexpr int kHotStride = kSplitTailBase + kSplitMaxRanges + 3;   // 60: a wave's row of bucket counts
constexpr int kTailClassBits = 3;                // hawk_split_tail's classes: key & 7
constexpr int kTailClasses = 1 << kTailClassBits;
constexpr int kTailStride = kSplitClassBase + kTailClasses + 8;   // 48
constexpr int kTailWaves = kTailClasses;         // a wave per class
constexpr int kTailThreads = 64 * kTailWaves;
constexpr int kTailBatch = kTailThreads * kWalkItems;   // 2048 entries a batch

static_assert(kSplitHot - kSplitHeads < (1 << 15), "hot_class_index is exact below 2^15");
static_assert((kSplitHot - kSplitHeads) / 15 < 1024, "fold_class matches ten bits of hawk_split_hot's class index");
static_assert(kHotStride >= kSplitTailBase + kSplitMaxRanges + 1, "bucket starts need one past the last bucket");
static_assert(kTailStride >= kSplitClassBase + kTailClasses + 1, "bucket starts need one past the last bucket");
static_assert(kSplitNone >= kHotStride && kSplitNone >= kTailStride, "the no-bucket code is outside the count rows");
static_assert(kTailRange < (1 << 16), "bins hold window-local keys as u16");

constexpr int kSplitPad = 72;                    // entries read (and ignored) past a run's end
constexpr int kPeerBlock = 4;                    // a key's peers read at once (at most kPeerBlock - 1 past their run)
constexpr unsigned kPeerSlots = 128;             // hawk_split_hot's match slots a wave: class-index bits 0..6

// A split walk workgroup's LDS: Waves waves, Window accumulators, count rows
// of Stride buckets, and the split tile (Waves * 256 entries); Peers match
// slots a wave for the folds.
template <class T, int Waves, int Window, int Stride, unsigned Peers = kPeerSlots>
struct SplitShared {
    static constexpr int kWaves = Waves;
    static constexpr int kStride = Stride;
    static constexpr int kWindow = Window;
    static constexpr unsigned kPeers = Peers;
    static constexpr int kSpan = Waves * 64 * kWalkItems;
    T acc[Window];                              // the window's accumulators
    T val[kSpan + kSplitPad];                   // the tile's values, bucket order
    unsigned short key[kSpan + kSplitPad];      // their window-local keys
    union {                                     // one phase at a time:
        unsigned long long win[Waves][Stride];                 // split: a match table per wave
        struct {
            unsigned long long peer[Waves][Peers];             // fold: per-wave match masks
        } f;
    };
    unsigned cnt[Waves][Stride];                // bucket counts, a row per wave (lane b reads word b)
    unsigned bstart[Stride + 1];                // bucket d holds [bstart[d], bstart[d+1])
};
template <class T>
using HotShared = SplitShared<T, kWalkWaves, kSplitHot, kHotStride>;      // 157 KiB (float64)
template <class T, int Window>
using TailShared = SplitShared<T, kTailWaves, Window, kTailStride, 64>;
static_assert(sizeof(TailShared<double, kTailRange>) <= 80 * 1024, "two tail workgroups share a CU's 160 KiB");

// The bucket of window-local key kl (0 <= kl < window) in hawk_split_hot:
// keys 0..31 a head bucket each; keys from 32 up one of fifteen classes by
// (kl - 32) % 15, so the fifteen class waves share the window evenly.
__device__ __forceinline__ unsigned hot_class_index(unsigned kl) {   // (kl - 32) / 15, exact below 2^15
    return ((kl - static_cast<unsigned>(kSplitHeads)) * 34953u) >> 19;
}
// hawk_split_tail keeps a class's accumulators together (class c = kl & 7 at
// [K c, K c + K), K = Window / 8, key index m = kl >> 3), so a class wave's
// reads and writes of distinct keys spread over the LDS banks; in key order all
// of a class's keys sit 64 bytes apart, on four bank positions.  m is XORed
// with 8c, which keeps it below K (a multiple of 64) and turns the final
// store's reads (eight classes a wave) from eight-way bank conflicts into
// two-way ones.
template <int Window>
__device__ __forceinline__ unsigned tail_slot(unsigned kl) {
    static_assert(Window % (64 * kTailClasses) == 0, "the XOR stays inside a class");
    const unsigned c = kl & (kTailClasses - 1u);
    return c * static_cast<unsigned>(Window / kTailClasses) + ((kl >> kTailClassBits) ^ (c << 3));
}
__device__ __forceinline__ int split_bucket(unsigned kl) {
    const unsigned u = kl - static_cast<unsigned>(kSplitHeads);
    return kl < static_cast<unsigned>(kSplitHeads) ? static_cast<int>(kl)
                                                   : kSplitClassBase + static_cast<int>(u - 15u * hot_class_index(kl));
}

// Where hawk_split_hot's split puts the tile's tail entries: straight from
// registers into the tile's slot of the chunk's bin, in bucket order, with
// the offset of each tail range in the tile's row of bin_off.
template <class T>
struct TailSink {
    unsigned short* key = nullptr;
    T* val = nullptr;
    unsigned* off = nullptr;
    int ranges = 0;
};

// Stable split of the tile held in registers (thread slot j of wave w is tile
// position w*256 + j*64 + lane) into nb buckets: sh.key/sh.val in bucket order,
// lane order within a bucket; bucket bounds in sh.bstart.  Each wave matches
// its four windows one after another in one table, so a lane's rank is the
// count of its bucket in the wave's earlier windows plus the lanes below it
// in its own.  Every wave then forms its own positions from all waves'
// counts.  With Sink, entries of a tail bucket go to the sink instead of LDS.
// Starts and ends with every thread of the workgroup.
template <class T, class Sh, bool Sink>
__device__ void split_tile(Sh& sh, const unsigned (&kl)[kWalkItems], const int (&d)[kWalkItems],
                           const T (&vv)[kWalkItems], int nb, const TailSink<T>& sink) {
    const int t = threadIdx.x;
    const int wave = t >> 6;
    const int lane = t & 63;
    const unsigned long long me = 1ull << lane;
    unsigned long long own[kWalkItems], mine[kWalkItems];
    // Window j: clear the table, OR every lane's bit into its bucket's slot,
    // read the lane's own slot and (lane b) slot b.  The four windows' LDS
    // operations run back to back: a wave's LDS operations complete in issue
    // order, so each window's reads see its own ORs and precede the next
    // window's clear.
    unsigned long long* tab = sh.win[wave];
    const int b = lane < Sh::kStride ? lane : 0;
#pragma unroll
    for (int j = 0; j < kWalkItems; ++j) {
        if (lane < Sh::kStride) tab[lane] = 0ull;
        __builtin_amdgcn_wave_barrier();
        if (d[j] != kSplitNone) atomicOr(&tab[d[j]], me);
        __builtin_amdgcn_wave_barrier();
        own[j] = tab[d[j] != kSplitNone ? d[j] : 0];
        mine[j] = tab[b];
        __builtin_amdgcn_wave_barrier();
    }
    // lane b: bucket b's count in each window and the running count before
    // each; each item later takes its bucket's position from lane d (a
    // permute) and adds the lanes below it in its window
    unsigned run[kWalkItems], below[kWalkItems];
    unsigned total = 0u;
#pragma unroll
    for (int j = 0; j < kWalkItems; ++j) {
        run[j] = total;
        total += static_cast<unsigned>(__popcll(mine[j]));
        below[j] = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(own[j] >> 32),
                                             __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(own[j]), 0u));
    }
    if (lane < Sh::kStride) sh.cnt[wave][lane] = total;
    __syncthreads();
    // lane b: bucket b's total over the waves, the earlier waves' share of it,
    // and (a scan over the lanes) where bucket b starts
    unsigned before = 0u, sum = 0u;
    if (lane < nb) {
        // word b of every wave's row: consecutive lanes, consecutive banks
#pragma unroll
        for (int w = 0; w < Sh::kWaves; ++w) {
            const unsigned c = sh.cnt[w][lane];
            before += w < wave ? c : 0u;
            sum += c;
        }
    }
    const unsigned start = wave_inclusive_scan(sum) - sum;
    if (wave == 0 && lane <= nb) sh.bstart[lane] = start;
    const unsigned base = start + before;
    unsigned ts = 0u;
    if constexpr (Sink) {
        ts = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(start), kSplitTailBase));
        if (sink.ranges > 0 && wave == 0 && lane >= kSplitTailBase && lane <= kSplitTailBase + sink.ranges)
            sink.off[lane - kSplitTailBase] = start - ts;
    }
#pragma unroll
    for (int j = 0; j < kWalkItems; ++j) {
        const int dj = d[j] != kSplitNone ? d[j] : 0;
        const unsigned p =
                static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(dj << 2, static_cast<int>(base + run[j]))) + below[j];
        if (d[j] != kSplitNone) {
            if (Sink && d[j] >= kSplitTailBase) {
                sink.key[p - ts] = static_cast<unsigned short>(kl[j]);
                sink.val[p - ts] = vv[j];
            } else {
                sh.key[p] = static_cast<unsigned short>(kl[j]);
                sh.val[p] = vv[j];
            }
        }
    }
    __syncthreads();
}

// Lane `lane`'s T, to every lane (two readlanes: the lane select is uniform).
__device__ __forceinline__ double lane_value(double x, int lane) {
    const long long bits = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane(static_cast<int>(bits), lane);
    const int hi = __builtin_amdgcn_readlane(static_cast<int>(bits >> 32), lane);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
__device__ __forceinline__ float lane_value(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// a + x0 + x1 + ... + x15, one addition at a time, x_q the value lane q of
// each row of 16 lanes holds: every row adds its own lanes' values, each
// handed to the whole row by the add itself (DPP row_newbcast), so a value
// costs one instruction and no LDS read: 4.9 cycles an add on MI355X (5.6
// in float32), where a chain fed from LDS takes 11 to 25 and one fed by
// readlane 13.5.  The fp64 add is the fused x * 1 + a, which rounds x + a once.
// The leading s_nop covers a DPP read's wait on the lane's last write of x.
__device__ __forceinline__ double row_chain(double a, double x) {
    const double one = 1.0;
#define HK_STEP(q) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #q " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" HK_STEP(0) HK_STEP(1) HK_STEP(2) HK_STEP(3) HK_STEP(4) HK_STEP(5) HK_STEP(6) HK_STEP(7)
        HK_STEP(8) HK_STEP(9) HK_STEP(10) HK_STEP(11) HK_STEP(12) HK_STEP(13) HK_STEP(14) HK_STEP(15)
        : "+v"(a) : "v"(x), "v"(one));
#undef HK_STEP
    return a;
}
__device__ __forceinline__ float row_chain(float a, float x) {
#define HK_STEP(q) "v_add_f32_dpp %0, %1, %0 row_newbcast:" #q " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" HK_STEP(0) HK_STEP(1) HK_STEP(2) HK_STEP(3) HK_STEP(4) HK_STEP(5) HK_STEP(6) HK_STEP(7)
        HK_STEP(8) HK_STEP(9) HK_STEP(10) HK_STEP(11) HK_STEP(12) HK_STEP(13) HK_STEP(14) HK_STEP(15)
        : "+v"(a) : "v"(x));
#undef HK_STEP
    return a;
}

// The chains of the split tile's head buckets c .. c + 3 (a key each: one
// contiguous run, lane order), by one wave: row r of 16 lanes adds bucket
// c + r onto acc[c + r], one addition at a time through row_chain, 64 values a
// step with the next step's reads in flight.  The wave runs as long as the
// longest of its four runs; a run that has ended adds +0.0, which changes no
// sum (none is ever -0.0: each started at +0.0).  A lane a chain, 32 values of
// its own ahead, took 2^23 lanes into 64 Zipf cells 80.7 us against 72.2.
template <class T, class Sh>
__device__ __forceinline__ void fold_heads(Sh& sh, int c) {
    const int lane = threadIdx.x & 63;
    const int k = c + (lane >> 4);
    const int s = static_cast<int>(sh.bstart[k]) + (lane & 15);
    const int e = static_cast<int>(sh.bstart[k + 1]);
    const int own = static_cast<int>(sh.bstart[k + 1] - sh.bstart[k]);
    const int top = max(__builtin_amdgcn_readlane(own, 0), __builtin_amdgcn_readlane(own, 16));
    const int low = max(__builtin_amdgcn_readlane(own, 32), __builtin_amdgcn_readlane(own, 48));
    const int longest = max(top, low);
    if (longest == 0) return;
    T a = sh.acc[k];
    T x[4];
    auto load = [&](int m) {                         // in bounds past the run: its end is at most the tile's
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = sh.val[min(s + m + 16 * q, e)];
    };
    load(0);
    for (int m = 0; m < longest; m += 64) {
        T y[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] = s + m + 16 * q < e ? x[q] : T(0);
        load(m + 64);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (m + 16 * q < longest) a = row_chain(a, y[q]);
    }
    if ((lane & 15) == 0) sh.acc[k] = a;
}

// The caller's wave folds class c of the split tile, 64 entries a window in
// lane order.  Within a class a key is named by its index m (hot: (kl - 32)
// / 15; tail: kl >> 3), below 1024.  Equal keys of a window find each other
// through the wave's match table: bits 0..6 of m pick one of kPeerSlots
// slots, every lane ORs its bit into its slot, and three ballots over bits
// 7..9 keep the lanes whose whole key is equal.  The lowest lane of each key
// adds its own value onto the accumulator it read with the match.  Where no
// key has more than one peer, the peer then adds its value onto what that lane
// left.  Otherwise every key's peers move, in lane order, to a run of their own
// in the window's place (a scan over the keys' peer counts gives the runs'
// starts), and the lowest lane adds its run from consecutive reads: finding
// each peer in the match mask instead (count trailing zeros, clear the bit)
// took most of a window's instructions.  In the widest tail window a window of
// one key alone is a chain by rows (3*10^7 sorted lanes into 65537 cells 1586 ->
// 816 us, five keys 1640 -> 634).  A wave's LDS operations complete in issue
// order, so a key's windows meet its accumulator one after another.
// With the head chains by rows, on MI355X in float64: 2^23 lanes into 64
// uniform cells 120.5 -> 82.1 us, into 64 Zipf cells 99.0 -> 72.2, into 4096
// uniform cells 84.6 -> 73.7, 2^26 Zipf lanes into 65536 cells 571 -> 524, and
// the wide walk's 2^22 lanes into 2^18 cells 74.0 -> 68.4.
template <class T, class Sh, bool Hot>
__device__ void fold_class(Sh& sh, int c) {
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const unsigned long long me = 1ull << lane;
    const int s = static_cast<int>(sh.bstart[kSplitClassBase + c]);
    const int e = static_cast<int>(sh.bstart[kSplitClassBase + c + 1]);
    if (s >= e) return;
    // bits below kLow pick the match slot, bits kLow .. kBits - 1 are balloted
    constexpr int kKeys = Hot ? 1024 : Sh::kWindow / kTailClasses;
    constexpr int kLow = Sh::kPeers == 64 ? 6 : 7;
    constexpr int kBits = kKeys > 512 ? 10 : kKeys > 256 ? 9 : kKeys > 128 ? 8 : 7;
    static_assert(Sh::kPeers == (1u << kLow) && kKeys <= (1 << kBits), "class matching covers every key");
    constexpr bool kChains = !Hot && Sh::kWindow == kTailRange;      // the others have no registers to spare
    unsigned long long* peer = sh.f.peer[wave];
    unsigned k = sh.key[s + lane];
    T x = sh.val[s + lane];
    for (int base = s; base < e; base += 64) {
        const bool valid = base + lane < e;
        unsigned nk = 0u;
        T nx = T(0);
        if (base + 64 < e) {
            nk = sh.key[base + 64 + lane];
            nx = sh.val[base + 64 + lane];
        }
        const unsigned kv = valid ? k : 0u;
        const unsigned m = Hot ? hot_class_index(kv) : (kv >> kTailClassBits);
        const unsigned h = m & (Sh::kPeers - 1u);
        if (valid) atomicOr(&peer[h], me);
        __builtin_amdgcn_wave_barrier();
        unsigned long long pm = valid ? peer[h] : 0ull;
        const unsigned ai = Hot ? kv : tail_slot<Sh::kWindow>(kv);
        const T a0 = valid ? sh.acc[ai] : T(0);
        __builtin_amdgcn_wave_barrier();
        if (valid) peer[h] = 0ull;
#pragma unroll
        for (int bit = kLow; bit < kBits; ++bit) {
            const unsigned long long ones = __ballot(valid && ((m >> bit) & 1u));
            const unsigned long long own = 0ull - static_cast<unsigned long long>((m >> bit) & 1u);
            pm &= ~(ones ^ own);
        }
        // equal keys below this lane: 0 for a key's lowest lane (and a lane past the run)
        const unsigned rank = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(pm >> 32),
                                                        __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(pm), 0u));
        T a = a0 + x;
        const unsigned long long more = __ballot(rank > 1u);
        if (more != 0ull) {
            if (kChains && __ballot(valid && rank == 0u) == 1ull) {
                // one key: its chain by rows, no peer looked for, and on through
                // the whole windows of the same key that follow (sorted keys)
                a = lane_value(a0, 0);
                T r[4];
                auto rows = [&](int at) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int i = at + 16 * q + (lane & 15);
                        const T v = sh.val[i];                   // up to 63 entries past the run (the padding)
                        r[q] = i < e ? v : T(0);
                    }
                };
                rows(base);
                const unsigned one = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(kv)));
                while (base + 128 <= e && __ballot(nk == one) == ~0ull) {
                    T y[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) y[q] = r[q];
                    base += 64;
                    rows(base);
                    if (base + 64 < e) {
                        nk = sh.key[base + 64 + lane];
                        nx = sh.val[base + 64 + lane];
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) a = row_chain(a, y[q]);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (base + 16 * q < e) a = row_chain(a, r[q]);
            } else {
                // a key has several peers: each key's to a run of their own in the window's place
                const int peers = valid && rank == 0u ? static_cast<int>(__popcll(pm)) - 1 : 0;
                const int start = static_cast<int>(wave_inclusive_scan(static_cast<unsigned>(peers))) - peers;
                const int low = pm != 0ull ? static_cast<int>(__builtin_ctzll(pm)) : 0;
                const int run = __builtin_amdgcn_ds_bpermute(low << 2, start);
                if (rank != 0u) sh.val[base + run + static_cast<int>(rank) - 1] = x;
                __builtin_amdgcn_wave_barrier();
                const T* y = sh.val + base + start;
                for (int left = peers; left > 0; left -= kPeerBlock, y += kPeerBlock) {
                    T r[kPeerBlock];
#pragma unroll
                    for (int q = 0; q < kPeerBlock; ++q) r[q] = y[q];
#pragma unroll
                    for (int q = 0; q < kPeerBlock; ++q) a = a + (q < left ? r[q] : T(0));
                }
            }
        }
        if (valid && rank == 0u) {
            sh.acc[ai] = a;
        }
        __builtin_amdgcn_wave_barrier();
        // at most one peer a key: it adds onto what its key's lowest lane left
        if (more == 0ull && rank != 0u) sh.acc[ai] = sh.acc[ai] + x;
        __builtin_amdgcn_wave_barrier();
        k = nk;
        x = nx;
    }
}

// The split tile's folds in hawk_split_hot: wave w the chains of the head keys
// 4w .. 4w + 3 (w < 8), then (w > 0) class w - 1: a skewed histogram's first
// four keys run longest, and wave 0 has nothing but them.  A class wave first
// clears its match table (it shares LDS with the split's tables); each window
// leaves it clear.
template <class T>
__device__ void split_fold(HotShared<T>& sh) {
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    if (4 * wave < kSplitHeads) fold_heads<T>(sh, 4 * wave);
    if (wave == 0) return;
#pragma unroll
    for (unsigned i = 0; i < kPeerSlots; i += 64) sh.f.peer[wave][i + lane] = 0ull;
    __builtin_amdgcn_wave_barrier();
    fold_class<T, HotShared<T>, true>(sh, wave - 1);
}

// hawk_split_tail's folds: wave w folds class w (keys with kl & 7 == w).
template <class T, int Window>
__device__ void split_fold_tail(TailShared<T, Window>& sh) {
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (unsigned i = 0; i < TailShared<T, Window>::kPeers; i += 64) sh.f.peer[wave][i + lane] = 0ull;
    __builtin_amdgcn_wave_barrier();
    fold_class<T, TailShared<T, Window>, false>(sh, wave);
}

// The window's partials of chunk b, every key [klo, klo+window): a key no
// lane named holds +0.0, the walk's starting value.
template <class T, class Sh>
__device__ void split_store(Sh& sh, long long b, long long cells, long long klo, int window,
                            T* __restrict__ parts) {
    __syncthreads();
    T* row = parts + b * cells + klo;
    for (int k = threadIdx.x; k < window; k += Sh::kWaves * 64) row[k] = sh.acc[k];
}

template <class T, class Sh>
__device__ void split_clear(Sh& sh, int window) {
    for (int k = threadIdx.x; k < window; k += Sh::kWaves * 64) sh.acc[k] = T(0);
    __syncthreads();
}

// Chunk b = blockIdx.x: lanes [b*span, min((b+1)*span, n)), keys below
// kSplitHot folded here, the others written to the chunk's bin (slot = tile,
// offsets of the `ranges` tail ranges in bin_off[b][tile][0..ranges]).
template <class T>
__global__ __launch_bounds__(kWalkThreads) void hawk_split_hot(
        const int* __restrict__ key, const T* __restrict__ v, long long n, long long cells, long long span,
        int tiles, int ranges, unsigned short* __restrict__ bin_key, T* __restrict__ bin_val,
        unsigned* __restrict__ bin_off, T* __restrict__ parts, int* __restrict__ status) {
    __shared__ HotShared<T> sh;
    const int t = threadIdx.x;
    const long long b = blockIdx.x;
    const long long lo = b * span;
    const long long hi = lo + span < n ? lo + span : n;
    const int window = cells < kSplitHot ? static_cast<int>(cells) : kSplitHot;
    const int nb = kSplitTailBase + ranges;
    split_clear<T>(sh, window);
    bool bad = false;
    int nk[kWalkItems];
    T nv[kWalkItems];
    if (lo < hi) walk_load(key, v, lo, hi, nk, nv);
    int tile = 0;
    for (long long base = lo; base < hi; base += kTile, ++tile) {
        unsigned kl[kWalkItems];
        int d[kWalkItems];
        T vv[kWalkItems];
        // each lane's bucket, without branches: a skip or bad key none, a
        // window key its head bucket or class, a tail key its range
#pragma unroll
        for (int j = 0; j < kWalkItems; ++j) {
            const unsigned u = static_cast<unsigned>(nk[j]);
            vv[j] = nv[j];
            const bool valid = u < static_cast<unsigned>(cells);
            bad = bad | ((nk[j] != -1) & !valid);
            const unsigned tl = u - static_cast<unsigned>(kSplitHot);
            const unsigned r = tl / static_cast<unsigned>(kTailRange);
            const bool in_win = u < static_cast<unsigned>(window);
            const int dw = split_bucket(u);
            d[j] = !valid ? kSplitNone : in_win ? dw : kSplitTailBase + static_cast<int>(r);
            kl[j] = in_win ? u : tl - r * static_cast<unsigned>(kTailRange);
        }
        if (base + kTile < hi) walk_load(key, v, base + kTile, hi, nk, nv);
        {
            TailSink<T> sink;
            if (ranges > 0) {
                const long long slot = (b * tiles + tile) * kTile;
                sink.key = bin_key + slot;
                sink.val = bin_val + slot;
                sink.off = bin_off + (b * tiles + tile) * (ranges + 1);
                sink.ranges = ranges;
            }
            split_tile<T, HotShared<T>, true>(sh, kl, d, vv, nb, sink);
        }
        split_fold(sh);
        __syncthreads();
    }
    // a chunk with fewer tiles than `tiles` (the last, short one) leaves its
    // later slots empty
    if (ranges > 0)
        for (int i = t; i < (tiles - tile) * (ranges + 1); i += kWalkThreads)
            bin_off[(b * tiles + tile) * (ranges + 1) + i] = 0u;
    split_store<T>(sh, b, cells, 0, window, parts);
    // the status plane: chunk b's flag, and from chunk 0 the cell count and the
    // flags of the chunks past the last
    const int any = __syncthreads_or(bad ? 1 : 0);
    if (t == 0) status[1 + b] = any ? 1 : 0;
    if (b == 0) {
        if (t == 0) status[0] = static_cast<int>(cells);
        for (int i = static_cast<int>(gridDim.x) + t; i < kScatterChunks; i += kWalkThreads) status[1 + i] = 0;
    }
}

// The tail ranges' stream: for workgroup (chunk b, range r), the range's
// segment of each tile slot of the chunk, slot after slot (lane order).  Each
// wave holds a group of up to kTailGroup segments in registers: lane l,
// register k describes segment g = 64k + l by its first stream position
// P[k] and the offset that turns a stream position q of it into its bin
// entry, base + A[k] + q (base: the group's first slot).  Segments past the group's end start at the group's
// length, so no position of the group falls in them.
constexpr int kTailGroup = 128;

struct TailSegs {
    unsigned P[kTailGroup / 64];
    int A[kTailGroup / 64];
    long long base;        // the group's first slot
    unsigned count;        // entries in the group
    int n;                 // segments in the group
};

__device__ __forceinline__ unsigned tail_reg(const unsigned (&x)[kTailGroup / 64], int m) {
    static_assert(kTailGroup == 128, "two registers a lane");
    const unsigned v = m < 64 ? x[0] : x[1];
    return static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v), m & 63));
}
__device__ __forceinline__ int tail_reg(const int (&x)[kTailGroup / 64], int m) {
    const int v = m < 64 ? x[0] : x[1];
    return __builtin_amdgcn_readlane(v, m & 63);
}

// Group [g0, g0 + gn) of chunk b's slots, range r: every wave reads the
// group's bounds (hawk_split_hot wrote 0 <= o[r] <= o[r+1] <= 4096; the
// clamps keep every read inside its slot whatever the plane holds).
__device__ __forceinline__ TailSegs tail_segs(const unsigned* __restrict__ bin_off, long long b, int tiles, int row,
                                              int r, int g0, int gn) {
    const int lane = threadIdx.x & 63;
    TailSegs S;
    unsigned carry = 0u;
#pragma unroll
    for (int k = 0; k < kTailGroup / 64; ++k) {
        const int g = k * 64 + lane;
        unsigned lo = 0u, hi = 0u;
        if (g < gn) {
            const unsigned* o = bin_off + (b * tiles + g0 + g) * row;
            const unsigned a = o[r], z = o[r + 1];
            lo = a < static_cast<unsigned>(kTile) ? a : static_cast<unsigned>(kTile);
            hi = z < lo ? lo : (z < static_cast<unsigned>(kTile) ? z : static_cast<unsigned>(kTile));
        }
        const unsigned c = hi - lo;
        const unsigned incl = wave_inclusive_scan(c) + carry;
        S.P[k] = incl - c;
        S.A[k] = g * kTile + static_cast<int>(lo) - static_cast<int>(S.P[k]);
        carry = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(incl), 63));
    }
    S.count = carry;
    S.n = gn;
    S.base = (b * tiles + g0) * kTile;
#pragma unroll
    for (int k = 0; k < kTailGroup / 64; ++k)
        if (k * 64 + lane >= gn) S.P[k] = carry;
    return S;
}

// A wave's entries from stream position q0 (wave-uniform): slot j takes
// position q0 + j*64 + lane (positions past the group's end read as nothing).
// Each window of 64 positions finds the segment of its first position with
// two ballots, then steps over the segments that start inside it.  Keys: read
// the entries' keys too.
template <class T, bool Keys = true>
__device__ __forceinline__ void tail_load(const TailSegs& S, const unsigned short* __restrict__ bin_key,
                                          const T* __restrict__ bin_val, unsigned q0, unsigned (&kk)[kWalkItems],
                                          T (&vv)[kWalkItems]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < kWalkItems; ++j) {
        const unsigned qw = q0 + static_cast<unsigned>(j * 64);
        const unsigned q = qw + static_cast<unsigned>(lane);
        kk[j] = 0u;
        vv[j] = T(0);
        if (qw >= S.count) continue;
        int g = -1;
#pragma unroll
        for (int k = 0; k < kTailGroup / 64; ++k) g += __popcll(__ballot(S.P[k] <= qw));
        int a = tail_reg(S.A, g);
        for (int m = g + 1; m < S.n; ++m) {
            // both reads with every lane active: the lane read from must
            // have computed its register select
            const unsigned pm = tail_reg(S.P, m);
            if (pm > qw + 63u) break;
            const int am = tail_reg(S.A, m);
            a = q >= pm ? am : a;
        }
        if (q < S.count) {
            const long long at = S.base + a + static_cast<long long>(q);
            if constexpr (Keys) kk[j] = bin_key[at];
            vv[j] = bin_val[at];
        }
    }
}

// The key ranges a walk's bins hold.  The split walk: `ranges` ranges of
// `width` keys from `first` up (singles 0, octaves 0).  The wide walk: keys
// 0..7 a range each (singles 8), then octaves [8, 16), [16, 32), ... up to
// `first` = 8 * 2^octaves, then ranges of `width` keys.
struct TailRanges {
    long long cells, first;      // keys 0 .. cells - 1 of this pass, its cell 0 at parts[0]
    long long stride;            // cells of a chunk's row of parts
    int ranges, singles, octaves, width;
    int row;                     // words a tile's row of bin_off has
};
constexpr int kWideSingles = kTailWaves;         // 8: a wave each
constexpr int kWideOctaves = 7;                  // [8, 16) .. [512, 1024)

// Chunk b's chain of single key k, by one wave: the key's segment of every
// tile slot in tile order, 256 values a step through the wave's LDS (so each
// row of lanes holds the same 16 values at a time), the next two steps' reads
// in flight while a step is added.  Positions past the end read as +0.0, which
// adds nothing to a sum that is never -0.0.
template <class T>
__device__ __forceinline__ T wide_chain(const T* __restrict__ bin_val, const unsigned* __restrict__ bin_off,
                                        long long b, int tiles, int row, int k, T* buf) {
    const int lane = threadIdx.x & 63;
    constexpr unsigned kStep = 64 * kWalkItems;
    T a = T(0);
    for (int g0 = 0; g0 < tiles; g0 += kTailGroup) {
        const int gn = tiles - g0 < kTailGroup ? tiles - g0 : kTailGroup;
        const TailSegs S = tail_segs(bin_off, b, tiles, row, k, g0, gn);
        unsigned none[kWalkItems];
        auto load = [&](unsigned q, T (&v)[kWalkItems]) {
            if (q < S.count) tail_load<T, false>(S, nullptr, bin_val, q, none, v);
        };
        auto step = [&](unsigned q, T (&v)[kWalkItems]) {
            if (q >= S.count) return;
#pragma unroll
            for (int j = 0; j < kWalkItems; ++j) buf[j * 64 + lane] = v[j];
            __builtin_amdgcn_wave_barrier();
            load(q + 2 * kStep, v);
            const int left = static_cast<int>(S.count - q < kStep ? S.count - q : kStep);
            for (int m = 0; m < left; m += 64) {
                T x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = buf[m + 16 * e + (lane & 15)];
#pragma unroll
                for (int e = 0; e < 4; ++e) a = row_chain(a, x[e]);
            }
            __builtin_amdgcn_wave_barrier();
        };
        T v0[kWalkItems], v1[kWalkItems];
        load(0u, v0);
        load(kStep, v1);
        for (unsigned q = 0; q < S.count; q += 2 * kStep) {
            step(q, v0);
            step(q + kStep, v1);
        }
    }
    return a;
}

// The chains of a split tile's buckets c, c + step, ... below `keys` (each the
// run of one key, lane order), by one wave, 64 values a round.
template <class T, class Sh>
__device__ __forceinline__ void fold_rows(Sh& sh, int c, int step, int keys) {
    const int lane = threadIdx.x & 63;
    for (; c < keys; c += step) {
        const int s = static_cast<int>(sh.bstart[c]), e = static_cast<int>(sh.bstart[c + 1]);
        if (s >= e) continue;
        T a = sh.acc[c];
        for (int m = s; m < e; m += 64) {
            T x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int at = m + 16 * q + (lane & 15);
                const T v = sh.val[at];                      // up to 63 entries past the run (the padding)
                x[q] = at < e ? v : T(0);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (m + 16 * q < e) a = row_chain(a, x[q]);
        }
        if (lane == 0) sh.acc[c] = a;
    }
}

// Range r of chunk b, read as a stream from the bin's slots in tile order,
// kTailBatch entries a batch, the next batch's reads in flight while a batch
// is split and folded: in eight classes, or, for a range of at most 32 keys,
// in a bucket a key (a chain a key: few keys share many lanes).  Workgroups
// chunk by chunk, range after range; with
// single keys (the wide walk) the first `chunks` workgroups are the chunks'
// chains, a wave a key, and with a status plane they also gather the chunk's
// bad-key flags, which hawk_wide_bin left behind each tile's
// offsets.  Windows up to 3072 keys leave three workgroups a CU, larger two.
template <class T, int Window>
__global__ __launch_bounds__(kTailThreads, Window <= 3072 ? 6 : 4) void hawk_split_tail(
        TailRanges R, int chunks, int tiles, const unsigned short* __restrict__ bin_key,
        const T* __restrict__ bin_val, const unsigned* __restrict__ bin_off, T* __restrict__ parts,
        int* __restrict__ status) {
    __shared__ __align__(16) TailShared<T, Window> sh;
    const int t = threadIdx.x;
    const int i = static_cast<int>(blockIdx.x);
    const long long b = i % chunks;
    if (R.singles > 0 && i < chunks) {
        const int k = t >> 6;
        const T a = wide_chain<T>(bin_val, bin_off, b, tiles, R.row, k, sh.val + k * (64 * kWalkItems));
        if ((t & 63) == 0 && k < R.cells) parts[b * R.stride + k] = a;
        if (status == nullptr) return;
        unsigned bad = 0u;
        for (int g = t; g < tiles; g += kTailThreads) bad |= bin_off[(b * tiles + g) * R.row + R.row - 1];
        const int any = __syncthreads_or(bad ? 1 : 0);
        if (t == 0) status[1 + b] = any;
        if (b == 0)
            for (int c = chunks + t; c < kScatterChunks; c += kTailThreads) status[1 + c] = 0;
        if (i == 0 && t == 0) status[0] = static_cast<int>(R.stride);
        return;
    }
    const int r = R.singles + i / chunks - (R.singles > 0 ? 1 : 0);
    const int u = r - R.singles - R.octaves;
    const long long klo = u < 0 ? static_cast<long long>(kWideSingles) << (r - R.singles)
                                : R.first + static_cast<long long>(R.width) * u;
    const long long size = u < 0 ? klo : R.width;
    // past the last pass's cells a range holds no key (and its window none)
    const int window = static_cast<int>(klo + size < R.cells ? size : R.cells - klo);
    const bool few = size <= kSplitHeads;
    split_clear<T>(sh, Window);
    for (int g0 = 0; g0 < tiles; g0 += kTailGroup) {
        const int gn = tiles - g0 < kTailGroup ? tiles - g0 : kTailGroup;
        const TailSegs S = tail_segs(bin_off, b, tiles, R.row, r, g0, gn);
        const unsigned w0 = static_cast<unsigned>((t >> 6) * (kWalkItems * 64));
        unsigned nk[kWalkItems];
        T nv[kWalkItems];
        if (S.count > 0u) tail_load(S, bin_key, bin_val, w0, nk, nv);
        for (unsigned qb = 0; qb < S.count; qb += kTailBatch) {
            unsigned kl[kWalkItems];
            int d[kWalkItems];
            T vv[kWalkItems];
#pragma unroll
            for (int j = 0; j < kWalkItems; ++j) {
                const unsigned q = qb + w0 + static_cast<unsigned>(j * 64 + (t & 63));
                kl[j] = nk[j];
                vv[j] = nv[j];
                const unsigned in = few ? kl[j] & (kSplitHeads - 1u) : kSplitClassBase + (kl[j] & (kTailClasses - 1u));
                d[j] = q < S.count ? static_cast<int>(in) : kSplitNone;
            }
            if (qb + kTailBatch < S.count) tail_load(S, bin_key, bin_val, qb + kTailBatch + w0, nk, nv);
            split_tile<T, TailShared<T, Window>, false>(sh, kl, d, vv, kSplitClassBase + kTailClasses, TailSink<T>());
            if (few) fold_rows<T>(sh, t >> 6, kTailWaves, static_cast<int>(size));
            else split_fold_tail<T, Window>(sh);
            __syncthreads();
        }
    }
    __syncthreads();
    T* row = parts + b * R.stride + klo;
    for (int k = t; k < window; k += kTailThreads) row[k] = sh.acc[few ? static_cast<unsigned>(k) : tail_slot<Window>(static_cast<unsigned>(k))];
}

// ---- the wide walk ----------------------------------------------------------
// hawk_split_hot walks a chunk in one workgroup, so a scatter of few chunks
// (n / cells of them, at most 256) leaves most of the chip idle, and its
// window and buckets end at 65536 cells.  The wide walk splits first and walks
// after: hawk_wide_bin splits every tile of every chunk on its own (a workgroup
// a tile, no order between them) into the key ranges' bins, and
// hawk_split_tail folds every (chunk, range) in lane order, a workgroup each:
// the same additions.  A skewed histogram's head keys 0..7 are chains of their
// own, a wave each, and the ranges above them grow by octaves, so a Zipf
// histogram's ranges hold about equal shares of its other lanes.  More than
// kWideCells cells take a pass (both launches) per kWideCells of them.
constexpr int kWideBuckets = 62;                 // ranges a tile splits into (bucket 63 is a lane that adds nothing)
constexpr int kWideStride = 63;
constexpr long long kWideCells = (static_cast<long long>(kWideSingles) << kWideOctaves) +
                                 static_cast<long long>(kWideBuckets - kWideSingles - kWideOctaves) * kTailRange;
constexpr int kWideGroups = 2048;                // workgroups hawk_split_tail gets where the cells allow it

// Which walk: the wide one where the split walk cannot go (more than 65536
// cells) and where its workgroup a chunk leaves the chip idle for longer than
// a second pass over the lanes takes.  Measured (fp64, uniform keys, split /
// wide, us; Zipf keys and float32 cross at about the same chunks): 65536 cells
// in 16 chunks 105 / 32, in 64 124 / 67, in 128 149 / 121, in 191 178 / 172; 20000
// in 96 62 / 43, in 191 66 / 67.  Few lanes in the tail make the split walk's
// second pass short: 14000 cells in 96 chunks 42 / 40, in 128 45 / 45; 12289 in
// 64 36 / 34, in 96 38 / 41, and with sorted keys (a chunk's lanes all in one
// range's workgroup) in 64 83 / 128, in 160 90 / 182.  Up to 12288 cells (no
// tail ranges) a chunk is at most three tiles: 10500 cells in 20 chunks 24 / 21,
// in 31 25 / 26; 4000 cells in 16 chunks 16 / 18.  Past 65536 cells, against a
// sorted walk of each chunk (a serial one past 2^19 cells): 2^18 cells, 2^22
// lanes 1470 us -> 68 uniform, 1395 -> 166 Zipf; 10^3 lanes into 10^8 cells, 346
// passes, 5.2 ms -> 4.9; 65537 cells, 3*10^7 sorted lanes 885 -> 816, 8*10^6
// 499 -> 554.
bool wide_walk(int64_t cells, int chunks) {
    return cells > kSplitCells ||
           chunks < (cells > kSplitHot + kTile ? 192 : cells > kSplitHot ? 96 : cells > 2 * kTile ? 32 : 0);
}

template <class T>
using WideShared = SplitShared<T, kWalkWaves, 1, kWideStride, 1>;        // 54 KiB (float64): two a CU
static_assert(kWideBuckets < kWideStride && kSplitNone >= kWideStride, "bucket starts need one past the last bucket");

// Tile g of chunk b (blockIdx.x = b * tiles + g): its entries in range order
// into the tile's slot of the bins, the ranges' offsets and a flag for a key
// that is neither a cell nor -1 into the tile's row of bin_off.  The pass takes
// keys [key0, key0 + R.cells).  magic is floor(2^32 / width): the quotient it
// gives is exact or one short.
template <class T>
__global__ __launch_bounds__(kWalkThreads) void hawk_wide_bin(
        const int* __restrict__ key, const T* __restrict__ v, long long n, long long span, int tiles, TailRanges R,
        unsigned key0, unsigned magic, unsigned short* __restrict__ bin_key, T* __restrict__ bin_val,
        unsigned* __restrict__ bin_off) {
    __shared__ WideShared<T> sh;
    const int t = threadIdx.x;
    const long long b = blockIdx.x / static_cast<unsigned>(tiles);
    const long long g = blockIdx.x % static_cast<unsigned>(tiles);
    const long long lo = b * span + g * kTile;
    const long long end = (b + 1) * span < n ? (b + 1) * span : n;
    const long long hi = lo + kTile < end ? lo + kTile : end;
    int kk[kWalkItems];
    T vv[kWalkItems];
    walk_load(key, v, lo, hi, kk, vv);
    unsigned kl[kWalkItems];
    int d[kWalkItems];
    bool bad = false;
    const unsigned first = static_cast<unsigned>(R.first), width = static_cast<unsigned>(R.width);
#pragma unroll
    for (int j = 0; j < kWalkItems; ++j) {
        bad = bad | ((kk[j] != -1) & !(static_cast<unsigned>(kk[j]) < static_cast<unsigned>(R.stride)));
        // a key below key0 wraps past the pass's cells
        const unsigned u = static_cast<unsigned>(kk[j]) - key0;
        const bool mine = (kk[j] >= 0) & (u < static_cast<unsigned>(R.cells));
        const unsigned w = u - first;
        unsigned q = __umulhi(w, magic);
        unsigned rem = w - q * width;
        if (rem >= width) {
            q += 1u;
            rem -= width;
        }
        const int o = 31 - __builtin_clz(u | 1u);            // key u's octave, 2^o <= u
        const bool single = u < static_cast<unsigned>(kWideSingles);
        const int low = single ? static_cast<int>(u) : kWideSingles + o - 3;
        d[j] = !mine ? kSplitNone : u < first ? low : kWideSingles + R.octaves + static_cast<int>(q);
        kl[j] = u < first ? (single ? 0u : u - (1u << o)) : rem;
    }
    static_assert(kWideSingles == 8, "the first octave is [8, 16)");
    split_tile<T, WideShared<T>, false>(sh, kl, d, vv, R.ranges, TailSink<T>());
    const long long slot = b * tiles + g;
    const unsigned count = sh.bstart[R.ranges];
    for (unsigned i = t; i < count; i += kWalkThreads) {
        bin_key[slot * kTile + i] = sh.key[i];
        bin_val[slot * kTile + i] = sh.val[i];
    }
    unsigned* row = bin_off + slot * R.row;
    if (t <= R.ranges) row[t] = sh.bstart[t];
    const int any = __syncthreads_or(bad ? 1 : 0);
    if (t == 0) row[R.row - 1] = static_cast<unsigned>(any);
}

// The ordered scatter's scratch, in this order (each part 256-byte aligned):
// parts[chunks][cells] f64; and for the split walk with tail ranges and the
// wide walk, the bin offsets [chunks][tiles][row] u32 (a range's and one more;
// the wide walk's row ends in a bad-key flag), the bin keys
// [chunks][tiles][4096] u16 and the bin values [chunks][tiles][4096] f64.
struct ScatterLayout {
    int chunks = 1;
    long long span = 0;
    bool wide = false;             // the wide walk, else the split walk
    int tiles = 0;
    int ranges = 0;                // key ranges the bins hold
    int octaves = 0, width = 0;    // the wide walk's octaves, and keys a range past them
    int row = 0;                   // words a tile's row of bin_off has
    size_t parts = 0, bin_off = 0, bin_key = 0, bin_val = 0, bytes = 0;
};

size_t align256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

ScatterLayout scatter_layout(int64_t n, int64_t cells, int chunks) {
    ScatterLayout L;
    L.chunks = chunks;
    L.span = (n + chunks - 1) / chunks;
    L.wide = wide_walk(cells, chunks);
    const size_t c = static_cast<size_t>(chunks);
    size_t at = 0;
    L.parts = at;
    at += align256(sizeof(double) * c * static_cast<size_t>(cells));
    const long long tiles = (L.span + kTile - 1) / kTile;
    L.tiles = static_cast<int>(tiles < 1 ? 1 : tiles);
    if (L.wide) {
        // octaves up to the pass's cells; past them enough ranges for
        // kWideGroups workgroups of hawk_split_tail, no more than the buckets,
        // none narrower than 64 keys
        const long long pass = cells < kWideCells ? cells : kWideCells;
        while (L.octaves < kWideOctaves && (static_cast<long long>(kWideSingles) << L.octaves) < pass) ++L.octaves;
        const long long rest = pass - (static_cast<long long>(kWideSingles) << L.octaves);
        if (rest > 0) {
            long long want = kWideGroups / chunks;
            const long long most = kWideBuckets - kWideSingles - L.octaves;
            const long long least = (rest + kTailRange - 1) / kTailRange;
            if (want > (rest + 63) / 64) want = (rest + 63) / 64;
            if (want < least) want = least;
            if (want > most) want = most;
            L.width = static_cast<int>((rest + want - 1) / want);
            L.ranges = static_cast<int>((rest + L.width - 1) / L.width);
        }
        L.ranges += kWideSingles + L.octaves;
    } else {
        L.ranges = cells > kSplitHot ? static_cast<int>((cells - kSplitHot + kTailRange - 1) / kTailRange) : 0;
    }
    L.row = L.ranges + (L.wide ? 2 : 1);
    if (L.ranges > 0) {
        const size_t slots = c * static_cast<size_t>(L.tiles);
        L.bin_off = at;
        at += align256(sizeof(unsigned) * slots * static_cast<size_t>(L.row));
        L.bin_key = at;
        at += align256(sizeof(unsigned short) * slots * kTile);
        L.bin_val = at;
        at += align256(sizeof(double) * slots * kTile);
    }
    L.bytes = at;
    return L;
}

// ---- the ordered gradient's log fold ----------------------------------------
// reference hawk/emit/team.py:281-312 (`_fold`) and hawk/ir/team.py:684-693
// (`fold_spec`): pair (key k, slot e) adds the key's `rows` contributions
// v[e * stride + k * rows + r], r = 0, 1, ..., in lane order from +0.0, and
// STORES the sum into out[cell_of[e * keys + k]].  Pairs run slot-major
// (pair = e * keys + k), so neighbouring pairs read neighbouring runs of one
// component plane.  A cell outside [0, cells) is not stored and sets status
// bit 0; a cell that a second pair names sets bit 1 and lowers status[1] to
// it (claims counts the pairs naming each cell): such stores race, as they do
// in the reference, and the caller is told.

template <class T>
__device__ __forceinline__ void log_fold_store(T s, int c, long long cells, T* __restrict__ out,
                                               int* __restrict__ claims, int* __restrict__ status) {
    if (c < 0 || c >= cells) {
        atomicOr(status, 1);
        return;
    }
    if (atomicAdd(claims + c, 1) != 0) {
        atomicOr(status, 2);
        atomicMin(status + 1, c);
    }
    out[c] = s;
}

// One thread per pair: the thread reads its run 16 rows at a time (then 8,
// then one), each batch's loads in flight before its adds.  Measured on
// MI355X over 805 MB of log: 4.6 TB/s at 64 rows a run, against 4.0 with
// batches of 8; staging the runs through LDS, or a wave reading whole lines,
// did no better.
template <class T>
__global__ __launch_bounds__(256) void hawk_log_fold_lanes(const T* __restrict__ v, long long stride,
                                                           const int* __restrict__ cell_of, long long keys,
                                                           long long rows, long long pairs,
                                                           T* __restrict__ out, long long cells,
                                                           int* __restrict__ claims, int* __restrict__ status) {
    const long long t = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    if (t >= pairs) return;
    const long long e = t / keys, k = t - e * keys;
    const T* __restrict__ p = v + e * stride + k * rows;
    T s = T(0);
    long long r = 0;
    for (; r + 16 <= rows; r += 16) {
        T x[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] = p[r + q];
#pragma unroll
        for (int q = 0; q < 16; ++q) s = s + x[q];
    }
    if (r + 8 <= rows) {
        T x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = p[r + q];
#pragma unroll
        for (int q = 0; q < 8; ++q) s = s + x[q];
        r += 8;
    }
    for (; r < rows; ++r) s = s + p[r];
    log_fold_store(s, cell_of[t], cells, out, claims, status);
}

// One wave per pair, for long runs of few pairs: the wave loads 64 consecutive rows (one
// 512-byte read) while it adds the previous 64 in lane order, every lane
// holding the same running sum; lane 0 stores it.
template <class T>
__global__ __launch_bounds__(256) void hawk_log_fold_waves(const T* __restrict__ v, long long stride,
                                                           const int* __restrict__ cell_of, long long keys,
                                                           long long rows, long long pairs,
                                                           T* __restrict__ out, long long cells,
                                                           int* __restrict__ claims, int* __restrict__ status) {
    const long long pair = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (pair >= pairs) return;                 // the whole wave
    const int lane = threadIdx.x & 63;
    const long long e = pair / keys, k = pair - e * keys;
    const T* __restrict__ p = v + e * stride + k * rows;
    T s = T(0);
    T x = lane < rows ? p[lane] : T(0);
    long long r0 = 0;
    for (; r0 + 64 <= rows; r0 += 64) {
        const T cur = x;
        x = r0 + 64 + lane < rows ? p[r0 + 64 + lane] : T(0);
#pragma unroll
        for (int j = 0; j < 64; ++j) s = s + lane_value(cur, j);
    }
    const int tail = static_cast<int>(rows - r0);
    for (int j = 0; j < tail; ++j) s = s + lane_value(x, j);
    if (lane == 0) log_fold_store(s, cell_of[pair], cells, out, claims, status);
}

__global__ __launch_bounds__(256) void hawk_log_fold_clear(int* __restrict__ claims, long long cells,
                                                           int* __restrict__ status) {
    const long long i0 = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    if (i0 == 0) {
        status[0] = 0;
        status[1] = 0x7fffffff;
    }
    for (long long i = i0; i < cells; i += static_cast<long long>(gridDim.x) * 256) claims[i] = 0;
}

int launch_error(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hawk_internal::set_hip_error(what, e);
    return HK_OK;
}

}  // namespace

// The scratch of hk_ordered_sum_f64_noalloc: the ordered sum's 65536 lane
// partials, 64 group values and ticket, kSumScratch bytes (512 KiB + 768 B)
// whatever the number of samples.  Each GPU the library runs on holds its own
// copy until the process ends.  In host code `scratch` names a host-side
// stand-in, never the device memory: launches take the per-device address
// that scratch_of() obtains with hipGetSymbolAddress.
static __device__ __align__(256) unsigned char scratch[kSumScratch];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the GPU that runs `stream` (the current
// device for the null stream), looked up once per device with that device
// current.
int scratch_of(hipStream_t stream, void** out) {
    int dev = 0;
    hipError_t e = stream ? hipStreamGetDevice(stream, &dev) : hipGetDevice(&dev);
    if (e != hipSuccess) return hawk_internal::set_hip_error("hk_ordered_sum_f64_noalloc: the stream's device", e);
    if (dev < 0 || dev >= kMaxDevices)
        return hawk_internal::set_error(HK_EVALUE, "hk_ordered_sum_f64_noalloc: device " + std::to_string(dev) +
                                                       " is past the " + std::to_string(kMaxDevices) +
                                                       " devices it keeps a scratch address for");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        int current = 0;
        e = hipGetDevice(&current);
        if (e != hipSuccess) return hawk_internal::set_hip_error("hk_ordered_sum_f64_noalloc: hipGetDevice", e);
        if (current != dev && (e = hipSetDevice(dev)) != hipSuccess)
            return hawk_internal::set_hip_error("hk_ordered_sum_f64_noalloc: hipSetDevice", e);
        void* ptr = nullptr;
        const hipError_t got = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (current != dev && (e = hipSetDevice(current)) != hipSuccess)
            return hawk_internal::set_hip_error("hk_ordered_sum_f64_noalloc: hipSetDevice", e);
        if (got != hipSuccess)
            return hawk_internal::set_hip_error("hk_ordered_sum_f64_noalloc: hipGetSymbolAddress(scratch)", got);
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return HK_OK;
}

// Fewer keys than this leave CUs idle at four waves a key; below a quarter of
// it long keys go group by group (10 keys of 60000 rows: 40 us a workgroup a
// key, 7.4 group by group; 400 of 20000: 12 a workgroup a key).
constexpr long long kFewKeys = 512;
// The rows a sixteen-wave workgroup sums in one launch: a group of 1024 a wave
// (1000 rows: 7.1 us as lanes and fold, 4.6 in one launch; 60000 rows, four
// groups a wave: 7.1 and 9.8).
constexpr long long kOneLaunchRows = 16 * kFoldLanes;

// Waves a key of hawk_keyed_comp: sixteen for few or long keys (see there), four
// otherwise and where sixteen would pass a launch's 2^32 - 1 threads.
constexpr int keyed_comp_waves(long long keys, long long group) {
    return (keys < kFewKeys || group > 8192) && keys * 1024 < (1LL << 32) ? 16 : 4;
}
static_assert(keyed_comp_waves(600, 8193) == 16 && keyed_comp_waves((1LL << 22) - 1, 8193) == 16 &&
              keyed_comp_waves(1LL << 22, 8193) == 4 && keyed_comp_waves((1LL << 24) - 1, 8193) == 4,
              "up to 2^24 - 1 keys of any length fit a launch");

// Whether a keyed ordered sum goes group by group, its group values in scratch.
constexpr bool keyed_by_groups(long long keys, long long group) {
    return group > (keys < kFewKeys / 4 ? kOneLaunchRows : kVirtualLanes);
}

// The ordered sum in T (hk_ordered_sum_f64 / _f32): the lanes, then the fold;
// up to kOneLaunchRows rows one launch of the keyed sum's kernel.
// A float sum keeps the double layout's offsets, its data in the front of
// each region.
template <class T>
int ordered_sum(const T* u, int64_t n, T* out, void* scratch, void* stream, const char* name) {
    if (n < 0) return hawk_internal::set_error(HK_EVALUE, std::string(name) + ": n must be >= 0");
    if ((n > 0 && !u) || !out || !scratch)
        return hawk_internal::set_error(HK_EVALUE, std::string(name) + ": u, out and scratch are required");
    auto* base = static_cast<unsigned char*>(scratch);
    auto* lanes = reinterpret_cast<T*>(base);
    auto* gp = reinterpret_cast<T*>(base + kLanesBytes);
    auto* ticket = reinterpret_cast<unsigned*>(base + kLanesBytes + kGpBytes);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (n <= kOneLaunchRows) {
        hipLaunchKernelGGL((hawk_keyed_rows<T, 16>), dim3(1), dim3(1024), 0, s, u, static_cast<long long>(n), out);
        return launch_error("hawk_keyed_rows launch");
    }
    const dim3 grid(kVirtualLanes / kLaneBlock), block(kLaneBlock);
    const long long len = n;
    auto rows_up_to = [n](int rows) { return n <= rows * static_cast<int64_t>(kVirtualLanes); };
    if (rows_up_to(kSumBatch))
        hipLaunchKernelGGL((hawk_sum_lanes<T, kSumBatch, true>), grid, block, 0, s, u, len, lanes, ticket);
    else if (sizeof(T) == 8 || rows_up_to(2 * kSumBatch))
        hipLaunchKernelGGL((hawk_sum_lanes<T, kSumBatch, false>), grid, block, 0, s, u, len, lanes, ticket);
    else
        hipLaunchKernelGGL((hawk_sum_lanes<T, kSumLong, false>), grid, block, 0, s, u, len, lanes, ticket);
    int rc = launch_error("hawk_sum_lanes launch");
    if (rc != HK_OK) return rc;
    hipLaunchKernelGGL(hawk_sum_fold<T>, dim3(kGroups), dim3(256), 0, s, lanes, gp, ticket, out);
    return launch_error("hawk_sum_fold launch");
}

// The keyed ordered sum in T (hk_keyed_ordered_sum_f64 / _f32).
template <class T>
int keyed_ordered_sum(const T* u, int64_t n, int64_t group, T* out, void* scratch, void* stream, const char* name) {
    const std::string who(name);
    if (n < 0 || group <= 0) return hawk_internal::set_error(HK_EVALUE, who + ": n must be >= 0 and group >= 1");
    if (n % group != 0)
        return hawk_internal::set_error(HK_EVALUE, who + ": n (" + std::to_string(n) +
                                                       ") is not a whole number of groups of " + std::to_string(group));
    if (n == 0) return HK_OK;
    if (!u || !out || !scratch) return hawk_internal::set_error(HK_EVALUE, who + ": u, out and scratch are required");
    if (n == group) return ordered_sum<T>(u, n, out, scratch, stream, name);    // one key: the ordered sum
    const long long keys = n / group;
    if (keys > 0x7fffffffLL) return hawk_internal::set_error(HK_EVALUE, who + ": too many keys");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const long long len = group;
    auto blocks_of = [](long long waves) { return dim3(static_cast<unsigned>((waves + 3) / 4)); };
    if (group <= 64) {
        const int P = pow2_at_least(group);
        const long long per_wave = kSmallSets * (64 / P);
        hipLaunchKernelGGL(hawk_keyed_small<T>, blocks_of((keys + per_wave - 1) / per_wave), dim3(256), 0, s, u, len, P,
                           keys, out);
        return launch_error("hawk_keyed_small launch");
    }
    if (group <= kFoldLanes) {
        const dim3 grid = blocks_of(keys);
        if (group <= 128) hipLaunchKernelGGL((hawk_keyed_wave<T, 2>), grid, dim3(256), 0, s, u, len, keys, out);
        else if (group <= 256) hipLaunchKernelGGL((hawk_keyed_wave<T, 4>), grid, dim3(256), 0, s, u, len, keys, out);
        else if (group <= 512) hipLaunchKernelGGL((hawk_keyed_wave<T, 8>), grid, dim3(256), 0, s, u, len, keys, out);
        else hipLaunchKernelGGL((hawk_keyed_wave<T, 16>), grid, dim3(256), 0, s, u, len, keys, out);
        return launch_error("hawk_keyed_wave launch");
    }
    if (!keyed_by_groups(keys, group)) {
        const dim3 grid(static_cast<unsigned>(keys));
        if (keys < kFewKeys && group <= kOneLaunchRows)
            hipLaunchKernelGGL((hawk_keyed_rows<T, 16>), grid, dim3(1024), 0, s, u, len, out);
        else
            hipLaunchKernelGGL((hawk_keyed_rows<T, 4>), grid, dim3(256), 0, s, u, len, out);
        return launch_error("hawk_keyed_rows launch");
    }
    auto* gp = static_cast<T*>(scratch);
    const long long used = (group + kFoldLanes - 1) / kFoldLanes < kGroups ? (group + kFoldLanes - 1) / kFoldLanes
                                                                           : kGroups;
    hipLaunchKernelGGL(hawk_keyed_groups<T>, blocks_of(keys * used), dim3(256), 0, s, u, len, static_cast<int>(used),
                       keys, gp);
    int rc = launch_error("hawk_keyed_groups launch");
    if (rc != HK_OK) return rc;
    hipLaunchKernelGGL(hawk_keyed_top<T>, blocks_of(keys), dim3(256), 0, s, gp, static_cast<int>(used), keys, out);
    return launch_error("hawk_keyed_top launch");
}

// The finishes of `count` reductions of `rows` rows each, in T: the leaves of
// all of them, then the levels (kRowsJobs reductions a launch).
template <class T>
int rows_finish(const hk_rows_job* jobs, int count, int64_t rows, void* scratch, void* stream, const char* name) {
    const std::string who(name);
    if (rows < 1) return hawk_internal::set_error(HK_EVALUE, who + ": rows must be >= 1");
    if (count < 0 || (count > 0 && (!jobs || !scratch)))
        return hawk_internal::set_error(HK_EVALUE, who + ": jobs and scratch are required");
    for (int i = 0; i < count; ++i) {
        const int32_t op = jobs[i].op;
        if (op < kRowsSum || op > kRowsBand || (op == kRowsBand && sizeof(T) != 8))
            return hawk_internal::set_error(HK_EVALUE, who + ": op must be 0 (sum), 1 (max), 2 (min) or, in float64, "
                                                             "3 (band)");
        if (!jobs[i].hi || !jobs[i].out || ((op == kRowsSum || op == kRowsBand) && !jobs[i].lo))
            return hawk_internal::set_error(HK_EVALUE, who + ": a job's hi, lo (of a sum) and out are required");
    }
    const long long leaves = (rows + kRowLeaf - 1) / kRowLeaf;
    if (leaves > 0x7fffffffLL) return hawk_internal::set_error(HK_EVALUE, who + ": too many rows");
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int first = 0; first < count; first += kRowsJobs) {
        const int here = count - first < kRowsJobs ? count - first : kRowsJobs;
        RowsJobs all{};
        for (int i = 0; i < here; ++i)
            all.job[i] = RowsJob{jobs[first + i].hi, jobs[first + i].lo, jobs[first + i].out, jobs[first + i].op};
        T* buf = static_cast<T*>(scratch) + 4 * leaves * first;
        hipLaunchKernelGGL(hawk_rows_leaves<T>, dim3(static_cast<unsigned>(leaves), static_cast<unsigned>(here)),
                           dim3(kRowSlots), 0, s, all, static_cast<long long>(rows), buf, leaves);
        int rc = launch_error("hawk_rows_leaves launch");
        if (rc != HK_OK || leaves == 1) {
            if (rc != HK_OK) return rc;
            continue;
        }
        hipLaunchKernelGGL(hawk_rows_levels<T>, dim3(static_cast<unsigned>(here)), dim3(256), 0, s, all, buf, leaves);
        rc = launch_error("hawk_rows_levels launch");
        if (rc != HK_OK) return rc;
    }
    return HK_OK;
}

// One reduction's finish, refusing by its own entry's argument names.
template <class T>
int rows_finish_one(const T* hi, const T* lo, int32_t op, int64_t rows, T* out, void* scratch, void* stream,
                    const char* name, const char* planes) {
    const std::string who(name);
    if (rows < 1) return hawk_internal::set_error(HK_EVALUE, who + ": rows must be >= 1");
    if (!hi || !out || !scratch || ((op == kRowsSum || op == kRowsBand) && !lo))
        return hawk_internal::set_error(HK_EVALUE, who + ": " + planes + ", out and scratch are required");
    const hk_rows_job job{hi, lo, out, op};
    return rows_finish<T>(&job, 1, rows, scratch, stream, name);
}

// The rows' extreme in T (op 1 max, 2 min).
template <class T>
int rows_extreme(const T* hi, int64_t rows, int32_t op, T* out, void* scratch, void* stream, const char* name) {
    if (rows >= 1 && op != kRowsMax && op != kRowsMin)
        return hawk_internal::set_error(HK_EVALUE, std::string(name) + ": op must be 1 (max) or 2 (min)");
    return rows_finish_one<T>(hi, nullptr, op, rows, out, scratch, stream, name, "hi");
}

// The keyed default-policy sum in T (hk_keyed_sample_sum_f64 / _f32).
template <class T>
int keyed_sample_sum(const T* u, int64_t n, int64_t group, T* out, void* stream, const char* name) {
    const std::string who(name);
    if (n < 0 || group <= 0)
        return hawk_internal::set_error(HK_EVALUE, who + ": n must be >= 0 and group >= 1");
    if (n % group != 0)
        return hawk_internal::set_error(HK_EVALUE, who + ": n (" + std::to_string(n) +
                                                       ") is not a whole number of groups of " + std::to_string(group));
    if ((group + 31) / 32 > kRowLeaf * kKeyedCompLeaves)
        return hawk_internal::set_error(HK_EVALUE, who + ": a key of " + std::to_string(group) +
                                                       " samples spans more than 256 leaves of 4096 rows; sum it "
                                                       "with policy='ordered'");
    if (n == 0) return HK_OK;
    if (!u || !out) return hawk_internal::set_error(HK_EVALUE, who + ": u and out are required");
    const long long keys = n / group;
    if (keys > 0x7fffffffLL) return hawk_internal::set_error(HK_EVALUE, who + ": too many keys");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const long long len = group;
    if (group <= 64 * 32) {
        const int rows = static_cast<int>((group + 31) / 32);
        const int G = rows > 8 ? 8 : pow2_at_least(rows);           // rows of a key in one step
        const long long waves = rows > 8 ? keys : (keys + 8 / G - 1) / (8 / G);
        const dim3 grid(static_cast<unsigned>((waves + 3) / 4)), block(256);
        if (rows <= 8) hipLaunchKernelGGL((hawk_keyed_comp_wave<T, 1>), grid, block, 0, s, u, len, G, keys, out);
        else if (rows <= 16) hipLaunchKernelGGL((hawk_keyed_comp_wave<T, 2>), grid, block, 0, s, u, len, G, keys, out);
        else if (rows <= 32) hipLaunchKernelGGL((hawk_keyed_comp_wave<T, 4>), grid, block, 0, s, u, len, G, keys, out);
        else hipLaunchKernelGGL((hawk_keyed_comp_wave<T, 8>), grid, block, 0, s, u, len, G, keys, out);
        return launch_error("hawk_keyed_comp_wave launch");
    }
    const dim3 grid(static_cast<unsigned>(keys));
    if (keyed_comp_waves(keys, group) == 16)
        hipLaunchKernelGGL((hawk_keyed_comp<T, 16>), grid, dim3(1024), 0, s, u, len, out);
    else hipLaunchKernelGGL((hawk_keyed_comp<T, 4>), grid, dim3(256), 0, s, u, len, out);
    return launch_error("hawk_keyed_comp launch");
}

// The ordered gradient's log fold in T (hk_keyed_log_fold_f64 / _f32).
template <class T>
int keyed_log_fold(const T* values, int64_t stride, const int32_t* cells_log, int64_t keys, int64_t rows,
                   int32_t width, T* out, int64_t cells, void* scratch, int32_t* status, void* stream,
                   const char* name) {
    const std::string who(name);
    if (keys < 0 || rows < 1 || width < 1 || cells < 0)
        return hawk_internal::set_error(HK_EVALUE, who + ": keys and cells must be >= 0, rows and width >= 1");
    if (stride < keys * rows)
        return hawk_internal::set_error(HK_EVALUE, who + ": stride (" + std::to_string(stride) +
                                                       ") is shorter than keys * rows (" +
                                                       std::to_string(keys * rows) + ")");
    if (!status) return hawk_internal::set_error(HK_EVALUE, who + ": status is required");
    const long long pairs = keys * static_cast<long long>(width);
    if (pairs > 0 && (!values || !cells_log || !out || (cells > 0 && !scratch)))
        return hawk_internal::set_error(HK_EVALUE,
                                        who + ": values, cells_log, out and scratch are required");
    if (cells > 0x7fffffffLL)
        return hawk_internal::set_error(HK_EVALUE, who + ": more than 2^31-1 cells");
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto* claims = static_cast<int*>(scratch);
    const long long clear = (cells + 255) / 256 < 1 ? 1 : ((cells + 255) / 256 < 4096 ? (cells + 255) / 256 : 4096);
    hipLaunchKernelGGL(hawk_log_fold_clear, dim3(static_cast<unsigned>(clear)), dim3(256), 0, s, claims,
                       static_cast<long long>(cells), status);
    int rc = launch_error("hawk_log_fold_clear launch");
    if (rc != HK_OK || pairs == 0) return rc;
    if (rows <= 64 || pairs >= 65536) {          // enough pairs for a thread each to fill the chip
        const long long blocks = (pairs + 255) / 256;
        if (blocks > 0x7fffffffLL) return hawk_internal::set_error(HK_EVALUE, who + ": too many pairs");
        hipLaunchKernelGGL(hawk_log_fold_lanes<T>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, values,
                           static_cast<long long>(stride), cells_log, static_cast<long long>(keys),
                           static_cast<long long>(rows), pairs, out, static_cast<long long>(cells), claims, status);
        return launch_error("hawk_log_fold_lanes launch");
    }
    const long long blocks = (pairs + 3) / 4;
    if (blocks > 0x7fffffffLL) return hawk_internal::set_error(HK_EVALUE, who + ": too many pairs");
    hipLaunchKernelGGL(hawk_log_fold_waves<T>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, values,
                       static_cast<long long>(stride), cells_log, static_cast<long long>(keys),
                       static_cast<long long>(rows), pairs, out, static_cast<long long>(cells), claims, status);
    return launch_error("hawk_log_fold_waves launch");
}

template <class T, int Window>
int split_tail(const TailRanges& R, int chunks, int tiles, const unsigned short* bin_key, const T* bin_val,
               const unsigned* bin_off, T* parts, int32_t* status, hipStream_t s) {
    // the wide walk's single keys share a workgroup a chunk
    const int groups = R.singles > 0 ? R.ranges - R.singles + 1 : R.ranges;
    hipLaunchKernelGGL((hawk_split_tail<T, Window>), dim3(static_cast<unsigned>(chunks * groups)),
                       dim3(kTailThreads), 0, s, R, chunks, tiles, bin_key, bin_val, bin_off, parts, status);
    return launch_error("hawk_split_tail launch");
}

// The ordered scatter in T (hk_ordered_scatter_f64 / _f32).
template <class T>
int ordered_scatter(const int32_t* key, const T* v, int64_t n, T* target, int64_t cells, void* scratch,
                    int32_t* status, void* stream, const char* name) {
    const std::string who(name);
    if (n < 0 || cells < 0)
        return hawk_internal::set_error(HK_EVALUE, who + ": n and cells must be >= 0");
    if (cells == 0) return HK_OK;   // a scatter into no cells adds nothing (reference hawk/runtime.py:727)
    if ((n > 0 && (!key || !v)) || !target || !scratch || !status)
        return hawk_internal::set_error(HK_EVALUE,
                                        who + ": key, v, target, scratch and status are required");
    if (cells > 0x7fffffffLL)
        return hawk_internal::set_error(HK_EVALUE, who + ": more than 2^31-1 cells");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int chunks = hk_scatter_chunks(n, cells);
    const ScatterLayout L = scatter_layout(n, cells, chunks);
    unsigned char* base = static_cast<unsigned char*>(scratch);
    auto* parts = reinterpret_cast<T*>(base + L.parts);     // a float scatter uses the front of each region
    auto* bin_off = reinterpret_cast<unsigned*>(base + L.bin_off);
    auto* bin_key = reinterpret_cast<unsigned short*>(base + L.bin_key);
    auto* bin_val = reinterpret_cast<T*>(base + L.bin_val);
    int rc = HK_OK;
    if (L.wide) {
        const long long slots = static_cast<long long>(chunks) * L.tiles;
        if (slots > 0x7fffffffLL) return hawk_internal::set_error(HK_EVALUE, who + ": too many samples");
        // with no width every key is below `first`
        const unsigned magic = L.width > 1 ? static_cast<unsigned>((1ull << 32) / static_cast<unsigned>(L.width))
                                           : 0xffffffffu;
        for (long long key0 = 0; key0 < cells; key0 += kWideCells) {
            const TailRanges R{cells - key0 < kWideCells ? cells - key0 : kWideCells,
                               static_cast<long long>(kWideSingles) << L.octaves, static_cast<long long>(cells),
                               L.ranges, kWideSingles, L.octaves, L.width, L.row};
            hipLaunchKernelGGL(hawk_wide_bin<T>, dim3(static_cast<unsigned>(slots)), dim3(kWalkThreads), 0, s, key, v,
                               static_cast<long long>(n), L.span, L.tiles, R, static_cast<unsigned>(key0), magic,
                               bin_key, bin_val, bin_off);
            rc = launch_error("hawk_wide_bin launch");
            if (rc != HK_OK) return rc;
            T* row = parts + key0;
            int32_t* flags = key0 == 0 ? status : nullptr;
            rc = L.width <= 1024   ? split_tail<T, 1024>(R, chunks, L.tiles, bin_key, bin_val, bin_off, row, flags, s)
                 : L.width <= 3072 ? split_tail<T, 3072>(R, chunks, L.tiles, bin_key, bin_val, bin_off, row, flags, s)
                                   : split_tail<T, kTailRange>(R, chunks, L.tiles, bin_key, bin_val, bin_off, row,
                                                               flags, s);
            if (rc != HK_OK) return rc;
        }
    } else {
        hipLaunchKernelGGL(hawk_split_hot<T>, dim3(static_cast<unsigned>(chunks)), dim3(kWalkThreads), 0, s, key, v,
                           static_cast<long long>(n), static_cast<long long>(cells), L.span, L.tiles, L.ranges,
                           bin_key, bin_val, bin_off, parts, status);
        rc = launch_error("hawk_split_hot launch");
        if (rc != HK_OK) return rc;
        if (L.ranges > 0) {
            const TailRanges R{static_cast<long long>(cells), kSplitHot, static_cast<long long>(cells), L.ranges, 0, 0,
                               kTailRange, L.row};
            rc = split_tail<T, kTailRange>(R, chunks, L.tiles, bin_key, bin_val, bin_off, parts, nullptr, s);
            if (rc != HK_OK) return rc;
        }
    }
    const long long grid = (cells + 255) / 256;
    if (chunks <= kAhead)
        hipLaunchKernelGGL((hawk_scatter_cells<T, true>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, s, parts,
                           static_cast<long long>(cells), chunks, target);
    else
        hipLaunchKernelGGL((hawk_scatter_cells<T, false>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, s, parts,
                           static_cast<long long>(cells), chunks, target);
    return launch_error("hawk_scatter_cells launch");
}

}  // namespace

extern "C" {

size_t hk_ordered_sum_scratch_bytes(void) { return kSumScratch; }

int hk_ordered_fold_f64(const double* lanes, double* out, void* scratch, void* stream) {
    if (!lanes || !out || !scratch)
        return hawk_internal::set_error(HK_EVALUE, "hk_ordered_fold_f64: lanes, out and scratch are required");
    auto* base = static_cast<unsigned char*>(scratch);
    auto* gp = reinterpret_cast<double*>(base + kLanesBytes);
    auto* ticket = reinterpret_cast<unsigned*>(base + kLanesBytes + kGpBytes);
    hipLaunchKernelGGL(hawk_sum_fold<double>, dim3(kGroups), dim3(256), 0, static_cast<hipStream_t>(stream),
                       lanes, gp, ticket, out);
    return launch_error("hawk_sum_fold launch");
}

int hk_ordered_sum_f64(const double* u, int64_t n, double* out, void* scratch, void* stream) {
    return ordered_sum<double>(u, n, out, scratch, stream, "hk_ordered_sum_f64");
}

int hk_ordered_sum_f32(const float* u, int64_t n, float* out, void* scratch, void* stream) {
    return ordered_sum<float>(u, n, out, scratch, stream, "hk_ordered_sum_f32");
}

size_t hk_ordered_sum_noalloc_scratch_bytes(void) { return kSumScratch; }

int hk_ordered_sum_f64_noalloc(const double* u, int64_t n, double* out, void* stream) {
    if (n < 0) return hawk_internal::set_error(HK_EVALUE, "hk_ordered_sum_f64_noalloc: n must be >= 0");
    if ((n > 0 && !u) || !out)
        return hawk_internal::set_error(HK_EVALUE, "hk_ordered_sum_f64_noalloc: u and out are required");
    void* ptr = nullptr;
    const int rc = scratch_of(static_cast<hipStream_t>(stream), &ptr);
    if (rc != HK_OK) return rc;
    return hk_ordered_sum_f64(u, n, out, ptr, stream);    // the same kernels, on the static scratch
}

size_t hk_keyed_ordered_sum_scratch_bytes(int64_t n, int64_t group) {
    if (n <= 0 || group <= 0 || n % group != 0) return 0;
    if (n == group) return kSumScratch;
    if (!keyed_by_groups(n / group, group)) return 256;      // the keys read their rows directly
    // group values; for keys past 65536 rows the entry's size, a lane partial each, stays
    return sizeof(double) * static_cast<size_t>(n / group) *
               static_cast<size_t>(group > kVirtualLanes ? kVirtualLanes : kGroups) + 256;
}

int hk_keyed_ordered_sum_f64(const double* u, int64_t n, int64_t group, double* out, void* scratch, void* stream) {
    return keyed_ordered_sum<double>(u, n, group, out, scratch, stream, "hk_keyed_ordered_sum_f64");
}

int hk_keyed_ordered_sum_f32(const float* u, int64_t n, int64_t group, float* out, void* scratch, void* stream) {
    return keyed_ordered_sum<float>(u, n, group, out, scratch, stream, "hk_keyed_ordered_sum_f32");
}

int hk_keyed_sample_sum_f64(const double* u, int64_t n, int64_t group, double* out, void* stream) {
    return keyed_sample_sum<double>(u, n, group, out, stream, "hk_keyed_sample_sum_f64");
}

int hk_keyed_sample_sum_f32(const float* u, int64_t n, int64_t group, float* out, void* stream) {
    return keyed_sample_sum<float>(u, n, group, out, stream, "hk_keyed_sample_sum_f32");
}

size_t hk_rows_finish_scratch_bytes(int64_t rows) {
    if (rows <= 0) return 0;
    const long long leaves = (rows + kRowLeaf - 1) / kRowLeaf;
    return sizeof(double) * 4 * static_cast<size_t>(leaves);
}

int hk_rows_finish_f64(const double* hi, const double* comp, int64_t rows, double* out, void* scratch,
                       void* stream) {
    return rows_finish_one<double>(hi, comp, kRowsSum, rows, out, scratch, stream, "hk_rows_finish_f64", "hi, comp");
}

int hk_rows_finish_f32(const float* hi, const float* comp, int64_t rows, float* out, void* scratch,
                       void* stream) {
    return rows_finish_one<float>(hi, comp, kRowsSum, rows, out, scratch, stream, "hk_rows_finish_f32", "hi, comp");
}

int hk_rows_extreme_f64(const double* hi, int64_t rows, int32_t op, double* out, void* scratch, void* stream) {
    return rows_extreme(hi, rows, op, out, scratch, stream, "hk_rows_extreme_f64");
}

int hk_rows_extreme_f32(const float* hi, int64_t rows, int32_t op, float* out, void* scratch, void* stream) {
    return rows_extreme(hi, rows, op, out, scratch, stream, "hk_rows_extreme_f32");
}

size_t hk_band_rows_finish_scratch_bytes(int64_t rows) { return hk_rows_finish_scratch_bytes(rows); }

int hk_band_rows_finish_f64(const double* hi, const double* lo, int64_t rows, double* out, void* scratch,
                            void* stream) {
    return rows_finish_one<double>(hi, lo, kRowsBand, rows, out, scratch, stream, "hk_band_rows_finish_f64", "hi, lo");
}

size_t hk_rows_finish_many_scratch_bytes(int64_t rows, int32_t count) {
    return count <= 0 ? 0 : hk_rows_finish_scratch_bytes(rows) * static_cast<size_t>(count);
}

int hk_rows_finish_many_f64(const hk_rows_job* jobs, int32_t count, int64_t rows, void* scratch, void* stream) {
    return rows_finish<double>(jobs, count, rows, scratch, stream, "hk_rows_finish_many_f64");
}

int hk_rows_finish_many_f32(const hk_rows_job* jobs, int32_t count, int64_t rows, void* scratch, void* stream) {
    return rows_finish<float>(jobs, count, rows, scratch, stream, "hk_rows_finish_many_f32");
}

size_t hk_band_ordered_sum_scratch_bytes(void) { return kBandSumScratch; }

int hk_band_ordered_sum_f64(const double* u, int64_t n, double* out, void* scratch, void* stream) {
    if (n < 0) return hawk_internal::set_error(HK_EVALUE, "hk_band_ordered_sum_f64: n must be >= 0");
    if ((n > 0 && !u) || !out || !scratch)
        return hawk_internal::set_error(HK_EVALUE, "hk_band_ordered_sum_f64: u, out and scratch are required");
    auto* base = static_cast<unsigned char*>(scratch);
    auto* lanes = reinterpret_cast<Band*>(base);
    auto* gp = reinterpret_cast<Band*>(base + kBandLanesBytes);
    auto* ticket = reinterpret_cast<unsigned*>(base + kBandLanesBytes + kBandGpBytes);
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(hawk_band_sum_lanes, dim3(kBandVirtual / kBandChains), dim3(kBandThreads), 0, s, u,
                       static_cast<long long>(n), lanes, ticket);
    int rc = launch_error("hawk_band_sum_lanes launch");
    if (rc != HK_OK) return rc;
    hipLaunchKernelGGL(hawk_band_sum_fold, dim3(kGroups), dim3(256), 0, s, lanes, gp, ticket, out);
    return launch_error("hawk_band_sum_fold launch");
}

int hk_scatter_chunks(int64_t n, int64_t cells) {
    if (n <= 0) return 1;
    const int64_t fit = n / (cells < 1 ? 1 : cells);
    return static_cast<int>(fit < 1 ? 1 : (fit > kScatterChunks ? kScatterChunks : fit));
}

size_t hk_ordered_scatter_scratch_bytes(int64_t n, int64_t cells) {
    if (cells <= 0) return 0;
    return scatter_layout(n, cells, hk_scatter_chunks(n, cells)).bytes;
}

int hk_ordered_scatter_f64(const int32_t* key, const double* v, int64_t n, double* target, int64_t cells,
                           void* scratch, int32_t* status, void* stream) {
    return ordered_scatter<double>(key, v, n, target, cells, scratch, status, stream, "hk_ordered_scatter_f64");
}

int hk_ordered_scatter_f32(const int32_t* key, const float* v, int64_t n, float* target, int64_t cells,
                           void* scratch, int32_t* status, void* stream) {
    return ordered_scatter<float>(key, v, n, target, cells, scratch, status, stream, "hk_ordered_scatter_f32");
}

size_t hk_keyed_log_fold_scratch_bytes(int64_t cells) {
    return cells <= 0 ? 0 : sizeof(int) * static_cast<size_t>(cells);
}

int hk_keyed_log_fold_f64(const double* values, int64_t stride, const int32_t* cells_log, int64_t keys,
                          int64_t rows, int32_t width, double* out, int64_t cells, void* scratch,
                          int32_t* status, void* stream) {
    return keyed_log_fold<double>(values, stride, cells_log, keys, rows, width, out, cells, scratch, status, stream,
                                  "hk_keyed_log_fold_f64");
}

int hk_keyed_log_fold_f32(const float* values, int64_t stride, const int32_t* cells_log, int64_t keys,
                          int64_t rows, int32_t width, float* out, int64_t cells, void* scratch,
                          int32_t* status, void* stream) {
    return keyed_log_fold<float>(values, stride, cells_log, keys, rows, width, out, cells, scratch, status, stream,
                                 "hk_keyed_log_fold_f32");
}

}  // extern "C"
