// Dense traversal: one workgroup per (query, partition) computes, for EVERY point
// of the partition, the outer step at which the loop of
// dci_query_single_point_by_block (src/dci_cuda_kernel.cu:401-626) would promote
// it, and from those steps the stop step, the candidates and their k best.
//
// It is the kernel for traversals that visit a large part of the index before
// they stop (hundreds or thousands of promotions per partition): there the batch
// kernel's cost per promotion (a rank by 2L binary searches, a replay) dominates,
// while the work here does not depend on where the loop stops.  Facts used, the
// same as in the batch kernel: a composite index consumes its windows in
// ascending (priority, simple index, order within the simple index), window
// number r at outer step r; a point is promoted under a composite at the step of
// the last of the L windows that hold it and is a candidate at its earliest
// (step, composite); the loop stops at the first step t with c0(t) >= k and
// (t + 1 >= outer * L or c0(t) >= max_candidates), c0 counting candidates whose
// promoting window held them in lane 0 (:598-607).
//
// Per composite index: the priorities |key[clamped window start] - q| (:572-590)
// of all its windows are laid out by (simple index, order within it) and sorted
// stably in LDS, which gives every window its step; every point then looks up the
// steps of its L windows (positions from the inverse permutation) and keeps the
// largest.  A histogram of the steps of lane-0 candidates yields the stop step;
// points promoted up to it get their exact distances (rows read by whole
// wavefronts) and go through a k-best filter.  Shapes that do not fit the tables
// are left to the other kernels through the same hand-over list.
#include <type_traits>

#include "bucket_core.h"
#include "common.h"
#include "kernels.h"
#include "radix_core.h"
#include "traverse_common.h"

namespace dcih {

namespace {

constexpr uint32_t kNever = 0xffffu;     // step field of a point that is never promoted

enum DMisc {   // 32-bit scalars shared by the workgroup
    dWin = 0, dArmed, dMaxc, dCand, dProbes, dMore, dOr, dAnd, dMaxW, dMaxBits, dUse8, dNoStep, dSlot,
    dMiscWords = 16
};

// Partitions of few points: workgroups of one wavefront, or an item would mostly wait for its own chain of
// reads and barriers.
constexpr int64_t kNarrowPoints = 512;
constexpr size_t kLdsBytes = 160 * 1024;

struct DenseLayout {
    int nt;           // threads per workgroup
    int ipt;          // windows per thread the sort holds (cap = nt * ipt per composite)
    int off_idx;      // per simple index: p, qp, left start, right start   (4 * I words)
    int off_seg;      // per composite: 2L + 1 segment starts, 2L stream numbers, 2L table places of window 0
    int off_q;        // query row
    int off_time;     // uint16 per point: step << 1 | lane-0 flag
    int off_sort;     // k best + pending candidates, 64-bit words
    int off_stage;
    int off_misc, off_wlist;
    int whole_bytes;  // room from off_stage on for the results of one round
    int sort_cap, quota;
    int front8, quota8;   // the same buffer where rows are compared by their codes: words kept, entries per wavefront between two merges
    int tiles;        // 1: rows of at most 128 elements, 16-byte aligned, distances wanted: whole batches of 64 rows
    int by_windows;   // 1: candidates are found by the windows' first lanes and the rows of near tiles, no time is kept per point
    int off_tab, tab_cap;   // then the step tables of all composites, uint16 per window, and
    int off_hist;     // the histogram of steps
    size_t lds_bytes;
};

// Buckets of the windows' ranking: about as many as windows, 4096 at most: twice as many rank 7021 windows no
// faster, and their 8 KB can be what keeps a second workgroup out of a CU (14000 points: 7.0 and 10.2 ms).
constexpr int dense_bucket_bits(int cap) {
    return cap <= 320 ? 8 : (cap <= 1280 ? 10 : (cap <= 2560 ? 11 : 12));
}
constexpr int kWlist = 2 * kWave;        // candidates a wavefront keeps listed
// Whether a partition's items compare rows by their codes: one word per partition, the number of items that
// had to give up on the codes less those that did not, while there is any doubt.  At kGiveUp the codes rest for
// kRest items, then one item tries them again: a partition whose rows lie too close together for their codes
// costs one wasted attempt in kRest + 1, and a query far outside the data costs its own items only.  Items
// that change the word together may count too few or too many; the rest is cut to kRest where it is counted down.
// (One load and one addition at the item's end: with an operation for each case the compiler's registers for the
// whole kernel came out worse, 75.4 instead of 73.1 ms for 512 queries on 10M unit vectors.)
constexpr int kGiveUp = 16, kRest = 64, kTrying = 1 << 20;      // kTrying: one item is at it
// How an item takes the codes (misc[dUse8]): not at all, with no doubt about them, with some, as the one that tries again.
// kCodesFailed is added when they did not do.
enum { kCodesOff = 0, kCodesOn, kCodesDoubted, kCodesTried, kCodesFailed };
constexpr int kBins = 256;               // of the histogram of scores, which lies at the start of the staging words

// Upper bound of the windows of one composite index: per simple index at most
// ceil((p+1)/T) + floor((n+T-3-p)/T) + 1 <= n/T + 3.  (A layout holds that many, so every item fits it.)
int64_t dense_max_windows(const QueryArgs& a) { return (int64_t)a.L * (a.ppb / a.T + 3); }

// (point_rows are there where the rules of point_rows_fit and point_rows_pay say so)
bool by_windows(const QueryArgs& a) { return a.picked && a.near_bounds && a.point_rows && dense_max_windows(a) <= 9 * 512 && a.M * (dense_max_windows(a) + 1) < 32768; }

DenseLayout dense_layout_for(const QueryArgs& a, int nt, int ipt, bool windows_only) {
    DenseLayout y;
    const int I = a.M * a.L;
    y.nt = nt;
    y.ipt = ipt;
    const int waves = y.nt / kWave;
    int o = dMiscWords * 4 + 64 * 4;      // scalars, then scratch of the block scans
    y.off_misc = 0;
    y.off_idx = o;      o += 4 * I * 4;
    y.off_seg = o;      o += (6 * a.L + 2) * 4;
    y.off_q = o;        o += ((a.dim + 3) & ~3) * 4;
    y.by_windows = windows_only ? 1 : 0;
    y.off_time = y.off_tab = y.off_hist = o;
    y.tab_cap = (int)((dense_max_windows(a) + 1) & ~(int64_t)1);
    if (y.by_windows) {
        o += 2 * a.M * y.tab_cap;
        o = (o + 3) & ~3;
        y.off_hist = o; o += 2 * y.tab_cap + 8;
    } else {
        o += (int)(((a.ppb + 1) & ~(int64_t)1) * 2);
    }
    o = (o + 15) & ~15;
    // k best plus room for candidates that beat the current k-th: the wavefronts fill
    // a quota each between two merges
    y.tiles = (!a.blind && a.dim <= 128 && (a.dim & 3) == 0 &&
               (reinterpret_cast<uintptr_t>(a.data) & 15) == 0) ? 1 : 0;
    // (a wavefront's share takes at least one whole batch of 64 candidates, of eight where rows are
    //  read eight at a time; compared by their codes, at least twice as many as the k best and 64 are kept)
    y.sort_cap = 64;
    while (y.sort_cap < max(a.kcap + waves * (y.tiles || a.blind ? 96 : 16), a.rows8 ? 2 * a.kcap + 64 + waves * 64 : 0)) y.sort_cap <<= 1;
    y.quota = (y.sort_cap - a.kcap) / waves;
    y.quota8 = max(64, (y.sort_cap - 2 * a.kcap - 64) / waves);
    y.front8 = y.sort_cap - waves * y.quota8;
    // staging words (later the step table, then the step histogram), behind them the buckets' counters, and
    // behind those what the window ranking does not need meanwhile: the radix passes' counters, which are
    // larger, reach into it
    y.off_stage = o;    o += (nt * ipt + 4) * 4;
    const int counters = o;
    o += ((1 << dense_bucket_bits(nt * ipt)) / 2 + 4) * 4;
    // The ranking is over when the first candidate is kept: where its room holds the buffer of kept ones twice,
    // the buffer lies in its upper half and the results of one round in its lower one.  (22223 points, 2640
    // windows, k = 50: 74576 bytes, two workgroups per CU, 1.60 ms for 4096 items; with the buffer
    // behind everything 82768 bytes, one, and 2.25.)
    const bool inside = o - y.off_stage >= y.sort_cap * 8 + max(y.sort_cap * 8, kBins * 4);
    y.off_sort = inside ? o - y.sort_cap * 8 : o + waves * kWlist * 2;
    y.whole_bytes = (inside ? y.off_sort : o) - y.off_stage;
    y.off_wlist = o;    o += waves * kWlist * 2;
    if (!inside) o += y.sort_cap * 8;
    o = max(o, counters + 8 * nt * 4);
    y.lds_bytes = (size_t)o;
    return y;
}

// Threads per workgroup and windows per thread; ipt = 0: too many windows.  With up to fifteen windows per
// thread 128 registers do, which allow 16 wavefronts per CU, and the kernel needs them all to hide its chains
// of LDS and memory reads: one per workgroup where partitions are small, four where four workgroups' tables
// fit a CU's LDS, else eight (7021 windows per composite, items taken up by strides: 22.2 ms; four wavefronts per
// workgroup and eight per CU 25.8).  With more, 128 registers spill in the ranking (17: 46 ms), so there eight wavefronts per CU, of
// two workgroups as far as a thread can hold the windows.
DenseLayout dense_layout(const QueryArgs& a, bool windows_only) {
    const int64_t windows = dense_max_windows(a);
    if (a.ppb <= kNarrowPoints)
        for (int i : {5, 9})
            if (windows <= (int64_t)64 * i) return dense_layout_for(a, 64, i, windows_only);
    for (int i : {5, 9})
        if (windows <= (int64_t)256 * i) {
            const DenseLayout y = dense_layout_for(a, 256, i, windows_only);
            if (4 * y.lds_bytes <= kLdsBytes) return y;
            break;
        }
    for (int i : {5, 9, 13, 15})
        if (windows <= (int64_t)512 * i) return dense_layout_for(a, 512, i, windows_only);
    if (windows <= (int64_t)256 * 33) return dense_layout_for(a, 256, 33, windows_only);
    if (windows <= (int64_t)512 * 21) return dense_layout_for(a, 512, 21, windows_only);
    DenseLayout none;
    none.ipt = 0;
    return none;
}
constexpr size_t kMostDenseLds = 160 * 1024 - 512;
// By windows only where that fits: the step tables of many composites can take more room than the points' times.
DenseLayout make_dense_layout(const QueryArgs& a) {
    if (by_windows(a)) {
        const DenseLayout y = dense_layout(a, true);
        if (y.ipt > 0 && y.lds_bytes <= kMostDenseLds) return y;
    }
    return dense_layout(a, false);
}

// Sums of N rows' lane values over a group of N lanes at once: on entry lane s of the group
// holds v[r] = its share of row r; on return it holds the total of row s.  Each level pairs
// the lanes s and s ^ H and halves the rows a lane carries, adding exactly the operands the
// butterfly  v += shfl_xor(v, H)  of wave_sum adds for that row, in the same order of levels,
// so every total has the bits wave_row_dists gives (N - 1 exchanges for N rows, not N log N).
template <int N, class V>
__device__ inline V group_row_sums(V (&v)[N], int s) {
    if constexpr (N == 1) {
        return v[0];
    } else {
        constexpr int H = N / 2;
        const bool upper = (s & H) != 0;
        V nv[H];
#pragma unroll
        for (int i = 0; i < H; i++) {
            const V send = upper ? v[i] : v[i + H];
            const V keep = upper ? v[i + H] : v[i];
            nv[i] = keep + lane_xor<H>(send);
        }
        return group_row_sums<H>(nv, s);
    }
}

// The first lane's value, in scalar registers.
__device__ inline float uniform_f32(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ inline unsigned long long uniform_u64(unsigned long long v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Workgroup g of its die takes the items from g * first on, every step-th one, below g * first + len.
struct DenseArgs { QueryArgs a; DenseLayout y; int first, step; int64_t len; };

// Where the workgroup's tables lie in LDS.
struct DenseTables {
    int* p;                       // per simple index: position of the query, its projection,
    float* qp;
    int* tabbase;                 // where its windows start in the step table (there they lie in the order of the
    int* shift;                   // positions they cover), and the shift that makes (position + shift) / T a window's place among them
    int* seg;                     // 2L + 1 segment starts (layout order)
    int* segstream;               // stream (2h + side) of a segment
    int* segw;                    // table place of a segment's window 0
    float* q;
    uint16_t* time;
    unsigned long long* sortbuf;
    uint32_t* stage;
    uint16_t* rank16;
    uint16_t* wlist;              // per wavefront: kWlist candidates
    template <class A, class Y>
    __device__ __forceinline__ DenseTables(unsigned char* smem, const A& a, const Y& y) {
        const int I = a.M * a.L;
        p = reinterpret_cast<int*>(smem + y.off_idx);
        qp = reinterpret_cast<float*>(p + I);
        tabbase = reinterpret_cast<int*>(qp + I);
        shift = tabbase + I;
        seg = reinterpret_cast<int*>(smem + y.off_seg);
        segstream = seg + 2 * a.L + 1;
        segw = segstream + 2 * a.L;
        q = reinterpret_cast<float*>(smem + y.off_q);
        time = reinterpret_cast<uint16_t*>(smem + y.off_time);
        sortbuf = reinterpret_cast<unsigned long long*>(smem + y.off_sort);
        stage = reinterpret_cast<uint32_t*>(smem + y.off_stage);
        rank16 = reinterpret_cast<uint16_t*>(stage);
        wlist = reinterpret_cast<uint16_t*>(smem + y.off_wlist);
    }
};

// WAVES: wavefronts per SIMD the registers are shared out for.  kPicked: the items are those of a call's round.  (Both in one
// kernel cost whole calls 3 %: 5000 items of 1350 rows, 418 and 429 us.)
// kWindows: of these, where few points are the first lane of a window and only the rows of near tiles can be results.
enum DenseKind { kWhole, kPicked, kWindows };
template <int NT, int IPT, int WAVES, int KIND>
__global__ __launch_bounds__(NT, WAVES) void traverse_dense_kernel(DenseArgs) {
    constexpr bool PICKED = KIND != kWhole, WINDOWS = KIND == kWindows;
    // The arguments are read where they are used, through a pointer that every phase makes opaque again:
    // read once, ahead of the loop over the items, they would be carried through it in spilled registers.
    typedef const DenseArgs __attribute__((address_space(4)))* ArgsPtr;
    // (Loops that may end for some threads only begin with a pointer of their own.)
    auto fresh_args = [&]() -> ArgsPtr {
        ArgsPtr p = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(p));
        return p;
    };
    ArgsPtr args = fresh_args();
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int kWaves = NT / kWave;
    constexpr int kBucketBits = dense_bucket_bits(NT * IPT);
    uint32_t* misc = reinterpret_cast<uint32_t*>(smem);
    uint32_t* scan_tmp = misc + dMiscWords;                           // 64 words
    DenseTables tb(smem, args->a, args->y);

    // The thread numbers are made opaque again at the start of every phase, and every phase ends
    // in an exit that is never taken but that the compiler cannot rule out (PHASE_END): otherwise
    // each phase's lane groupings, per-thread addresses and loop-invariant loads are computed
    // once, ahead of the loop over the items, and carried through every other phase in registers
    // or scratch.
    int tid = threadIdx.x;
    int lane = tid & (kWave - 1);
    int wave = tid / kWave;
    auto fresh_thread_ids = [&]() {
        asm volatile("" : "+v"(tid));
        lane = tid & (kWave - 1);
        wave = tid / kWave;
    };
#define PHASE_END(which)                                 \
    do {                                                 \
        phase(which);                                    \
        int leave_now = 0;                               \
        asm volatile("" : "+s"(leave_now));              \
        if (leave_now) return;                           \
        fresh_thread_ids();                              \
        args = fresh_args();                             \
        tb = DenseTables(smem, args->a, args->y);        \
    } while (0)
    const int I = args->a.M * args->a.L;
    const int T = args->a.T;
    const int X = args->a.xcds;
    const int xcd = (int)(blockIdx.x % X);
    const int64_t g0 = blockIdx.x / X;
    int64_t my_count;
    const int32_t* my_items = nullptr;
    if constexpr (PICKED) {
        my_count = picked_run(args->a, xcd, my_items);
    } else if (args->a.dense_items != nullptr && args->a.mode != 3) {
        my_count = (int64_t)args->a.dense_count[xcd];
        my_items = args->a.dense_items + (int64_t)xcd * args->a.dense_cap;
    } else {
        my_count = block_items(X, args->a.B, args->a.q_count) / X;
    }
    const int slot_first = (int)g0 * args->first, slot_end = (int)min(my_count, (int64_t)slot_first + args->len);

    // optional phase profile: thread 0 adds the 100 MHz ticks each phase took
    unsigned long long tick = 0ull;
    auto phase = [&](int which) {
        if (args->a.phase_ticks && tid == 0) {
            const unsigned long long now = wall_clock64();
            atomicAdd(&args->a.phase_ticks[which], now - tick);
            tick = now;
        }
    };

    // (a die's items number below 2^28; the step is read where it is used: one more scalar carried through the loop
    //  costs 1 % where a call is a few rounds of items)
    // The items of a round, whose number the launch does not know, are handed out in order as workgroups come to ask for one: the
    // last ones that start do, those before them take one item each.
    auto next_slot = [&](int slot) -> int {
        if constexpr (!PICKED) return slot + fresh_args()->step;
        if (slot < fresh_args()->step || slot_end <= (int)(gridDim.x / (unsigned)X)) return 0x7fffffff;      // (or none is left over)
        if (tid == 0) misc[dSlot] = atomicAdd(&fresh_args()->a.picked_ticket[xcd * kTicketStride], 1u);
        __syncthreads();
        const int taken = __builtin_amdgcn_readfirstlane((int)misc[dSlot]);
        __syncthreads();
        return (int)(gridDim.x / (unsigned)X) + taken;
    };
    for (int slot = slot_first; slot < slot_end; slot = next_slot(slot)) {
        ArgsPtr args = fresh_args();
        DenseTables tb(smem, args->a, args->y);
        int b, qi;
        if (PICKED || my_items) {
            const int64_t item = my_items[slot];
            b = (int)(item % args->a.B);
            qi = (int)(item / args->a.B);
        } else {
            if (!block_item((int64_t)slot * X + xcd, X, args->a.B, args->a.q_count, b, qi)) continue;
            qi += args->a.q_first;
        }
        b = __builtin_amdgcn_readfirstlane(b);      // (what is the same for all threads stays in scalar registers)
        qi = __builtin_amdgcn_readfirstlane(qi);
        const int64_t item = (int64_t)qi * args->a.B + b;
        const int64_t off = (int64_t)b * args->a.ppb;
        const int n = (int)min(args->a.N - off, args->a.ppb);
        unsigned long long* part_out = args->a.part + item * args->a.kcap;
        __syncthreads();                         // the previous item's tables are done with
        if (n <= 0) {
            for (int j = tid; j < args->a.kcap; j += NT) part_out[j] = ~0ull;
            continue;
        }

        // ---- set-up: query row, positioning searches (:279-297) -------------------
        if (args->a.phase_ticks) tick = wall_clock64();
        if (tid < dMiscWords) misc[tid] = 0;
        for (int j = tid; j < args->a.dim; j += NT) tb.q[j] = args->a.query[(int64_t)qi * args->a.dim + j];
        if constexpr (!WINDOWS) for (int pt = tid; pt < n; pt += NT) tb.time[pt] = (uint16_t)((kNever << 1) & 0xffffu);
        uint32_t probes = 0;
        {
            const int per_wave = (I + kWaves - 1) / kWaves;
            const int lg = min(3, floor_log2(kWave / per_wave > 0 ? kWave / per_wave : 1)), Gq = 1 << lg;
            const int slots = kWave >> lg;
            for (int i0 = 0; i0 < I; i0 += slots * kWaves) {
                const int sl = lane >> lg, i = i0 + wave * slots + sl;
                const bool active = i < I;
                const float* key = args->a.skeys + (int64_t)(active ? i : 0) * args->a.N + off;
                const float qp = active ? args->a.qproj[(int64_t)i * args->a.nq + qi] : 0.f;
                const int lo = group_partition_point(0, n, active, lg, sl * Gq, lane - sl * Gq,
                                                     [&](int j) { return key[j] < qp; }, probes);
                if (active && lane == sl * Gq) { tb.p[i] = lo - 1; tb.qp[i] = qp; }
            }
        }
        if (args->a.rows8 && tid == 0) {          // (other items change the word meanwhile: one thread decides)
            int* doubt = reinterpret_cast<int*>(args->a.rows8_bounds) + 2 * args->a.B + b;
            int have = __hip_atomic_load(doubt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t use = have <= 0 ? kCodesOn : (have < kGiveUp ? kCodesDoubted : kCodesOff);
            for (int tries = 0; tries < 8 && use == kCodesOff && have >= kGiveUp && have < kTrying; tries++) {      // counts the rest down
                const int was = atomicCAS(doubt, have, have == kGiveUp ? kTrying : min(have, kGiveUp + kRest) - 1);
                if (was == have) {
                    if (have == kGiveUp) use = kCodesTried;
                    break;
                }
                have = was;
            }
            misc[dUse8] = use;
        }
        __syncthreads();
        PHASE_END(0);

        unsigned long long maxw = 0;             // most windows any composite has a step for
        for (int m = 0; m < args->a.M; m++) {
            ArgsPtr args = fresh_args();
            DenseTables tb(smem, args->a, args->y);
            // ---- layout of the composite's windows: per simple index its left stream, then
            // its right one; where the query lies above every key the single (ghost) right
            // window comes first, as dci_next_closest_proj orders it (:264-265)
            // (one lane per simple index, the first wavefront: L <= 64)
            if (wave == 0) {
                const int h = lane;
                int nl = 0, nr = 0, p = 0;
                if (h < args->a.L) {
                    p = tb.p[m * args->a.L + h];
                    nl = stream_windows(n, T, p, 0);
                    nr = stream_windows(n, T, p, 1);
                }
                int incl = nl + nr;
#pragma unroll
                for (int o = 1; o < kWave; o <<= 1) {
                    const int t2 = __shfl_up(incl, o, kWave);
                    if (lane >= o) incl += t2;
                }
                const int at = incl - (nl + nr);
                if (h < args->a.L) {
                    const int i = m * args->a.L + h;
                    const bool corner = p == n - 1 && T >= 2;
                    // In the table the index's windows lie by the positions they cover: left
                    // window j at place nl - 1 - j, right window j at nl + j; a position pos
                    // belongs to the window at place (pos + nl * T - p - 1) / T and is its first
                    // lane where that division leaves no remainder.
                    // (by windows both in one word)
                    tb.tabbase[i] = at;
                    tb.shift[i] = (nl * T - p - 1) | (WINDOWS ? (at + m * args->y.tab_cap) << 16 : 0);
                    const int w_left = at + nl - 1, w_right = at + nl;
                    if (corner) {
                        tb.seg[2 * h] = at; tb.segstream[2 * h] = 2 * h + 1; tb.segw[2 * h] = w_right;
                        tb.seg[2 * h + 1] = at + nr; tb.segstream[2 * h + 1] = 2 * h; tb.segw[2 * h + 1] = w_left;
                    } else {
                        tb.seg[2 * h] = at; tb.segstream[2 * h] = 2 * h; tb.segw[2 * h] = w_left;
                        tb.seg[2 * h + 1] = at + nl; tb.segstream[2 * h + 1] = 2 * h + 1; tb.segw[2 * h + 1] = w_right;
                    }
                }
                const int total = __shfl(incl, args->a.L - 1, kWave);
                if (lane == 0) {
                    misc[dMaxBits] = 0;
                    misc[dNoStep] = 0;
                    tb.seg[2 * args->a.L] = total;
                    misc[dWin] = (uint32_t)total;
                    misc[dOr] = 0; misc[dAnd] = 0xffffffffu;
                }
            }
            __syncthreads();
            const int W = __builtin_amdgcn_readfirstlane((int)misc[dWin]);
            // (where the composite's steps go: a table of its own, or the room of the ranking's lists)
            auto step_table = [&](const DenseTables& tb) __attribute__((always_inline)) {
                if constexpr (!WINDOWS) return tb.rank16;
                ArgsPtr args = fresh_args();
                return reinterpret_cast<uint16_t*>(smem + args->y.off_tab) + m * args->y.tab_cap;
            };

            // The step of every window is its place in the order of priorities, stored doubled with bit 0
            // set: a lookup subtracts one where the point is not the window's first lane, which
            // leaves the lane-0 flag beside the step.  A window whose priority is not finite (rows that hold
            // infinities or NaN) is never reached: the loop takes the first minimum below infinity (:466-478).
            // Such windows come last in the order and get kNever; their number is misc[dNoStep].
            bool few_windows = false;
            if constexpr (IPT <= 9) if (W <= 2 * NT) {
                // ---- few windows: one or two per thread, as (priority, layout index, table place) words; the
                // layout index makes equal priorities keep their order.  Sorted in registers, up to 256 words
                // by one wavefront: bound by vector issue, and the exchanges inside a lane are done once, not
                // by both sides.
                few_windows = true;
                const int np = W <= 4 * kWave ? (W <= kWave ? kWave : (W <= 2 * kWave ? 2 * kWave : 4 * kWave)) : (W <= NT ? NT : 2 * NT);
                unsigned long long* s64 = reinterpret_cast<unsigned long long*>(tb.stage);
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int idx = e * NT + tid;
                    unsigned long long word = ~0ull;
                    if (idx < W) {
                        int lo = 0, hi = 2 * args->a.L - 1;      // the first segment that ends behind idx
                        while (lo < hi) {
                            const int mid = (lo + hi) >> 1;
                            if (tb.seg[mid + 1] <= idx) lo = mid + 1; else hi = mid;
                        }
                        const int sidx = tb.segstream[lo], j = idx - tb.seg[lo], h = sidx >> 1;
                        const int p = tb.p[m * args->a.L + h];
                        const int pos = sidx & 1 ? p + 1 + j * T : p - T + 1 - j * T;
                        const int place = sidx & 1 ? tb.segw[lo] + j : tb.segw[lo] - j;
                        const float key = args->a.skeys[(int64_t)(m * args->a.L + h) * args->a.N + off + min(max(pos, 0), n - 1)];
                        const float prio = fabsf(key - tb.qp[m * args->a.L + h]);
                        word = ((unsigned long long)__builtin_bit_cast(uint32_t, prio) << 32) | ((uint32_t)idx << 16) | (uint32_t)place;
                        if (__builtin_bit_cast(uint32_t, prio) >= kInfBits) atomicAdd(&misc[dNoStep], 1u);
                        probes++;
                    }
                    if (idx < np) s64[idx] = word;
                }
                __syncthreads();
                PHASE_END(1);
                auto step_of = [&](unsigned long long word, int at) {
                    return (uint32_t)(word >> 32) < kInfBits ? (uint16_t)((at << 1) | 1) : (uint16_t)kNever;
                };
                auto by_one_wave = [&](auto etag) __attribute__((always_inline)) {
                    constexpr int E = decltype(etag)::value;
                    if (wave == 0) {
                        unsigned long long v[E];
#pragma unroll
                        for (int i = 0; i < E; i++) v[i] = s64[lane * E + i];
                        wave_sort_u64(v, lane);
                        __builtin_amdgcn_wave_barrier();                // the table takes the words' room
                        uint16_t* steps = step_table(tb);
#pragma unroll
                        for (int i = 0; i < E; i++)
                            if (v[i] != ~0ull) steps[(uint32_t)v[i] & 0xffffu] = step_of(v[i], lane * E + i);
                    }
                };
                if (np == kWave) by_one_wave(std::integral_constant<int, 1>{});
                else if (np == 2 * kWave) by_one_wave(std::integral_constant<int, 2>{});
                else if constexpr (NT > kWave) {
                    if (np == 4 * kWave) {
                        by_one_wave(std::integral_constant<int, 4>{});
                    } else {
                        if constexpr (NT > 4 * kWave) if (np == NT) bitonic_sort_u64_regs<1, NT>(s64, tid);
                        if (np == 2 * NT) bitonic_sort_u64_regs<2, NT>(s64, tid);
                        unsigned long long mine[2];
#pragma unroll
                        for (int e = 0; e < 2; e++) mine[e] = e * NT < np ? s64[e * NT + tid] : 0ull;
                        __syncthreads();                    // the table takes the sorted words' room
                        uint16_t* steps = step_table(tb);
#pragma unroll
                        for (int e = 0; e < 2; e++)
                            if (e * NT + tid < W) steps[(uint32_t)mine[e] & 0xffffu] = step_of(mine[e], e * NT + tid);
                    }
                }
            }
            // ---- priorities of the windows, blocked: thread t holds layout indices t*IPT.. ----
            // (formed a second time in the rare case that the ranking by buckets gives up)
            for (bool by_radix = false; !few_windows; by_radix = true) {
            ArgsPtr args = fresh_args();
            DenseTables tb(smem, args->a, args->y);
            uint32_t k[IPT], rp[IPT];
            {
                int seg = 0;
                const int first = tid * IPT;
                {   // the first segment that ends behind `first` (empty segments are skipped)
                    int lo = 0, hi = 2 * args->a.L - 1;
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if (tb.seg[mid + 1] <= first) lo = mid + 1; else hi = mid;
                    }
                    seg = lo;
                }
                // (offsets from the composite's first slice; all reads are issued before any is used)
                const float* kbase = args->a.skeys + (int64_t)m * args->a.L * args->a.N + off;
                uint32_t koff[IPT];
                float qv[IPT];
                // Per segment: where its windows' keys lie and which way they run.  Window j of
                // a right stream starts at position p + 1 + j * T and takes table place
                // seg_w + j; of a left stream, p - T + 1 - j * T and seg_w - j; the key read is
                // the one at that position moved into the slice.
                int seg_end, pos_cur, pos_step, w_cur, w_step;
                uint32_t h_base;
                float q_seg;
                auto enter = [&](int idx) {
                    seg_end = tb.seg[seg + 1];
                    const int sidx = tb.segstream[seg], j = idx - tb.seg[seg], h = sidx >> 1;
                    const int p = tb.p[m * args->a.L + h];
                    q_seg = tb.qp[m * args->a.L + h];
                    h_base = (uint32_t)h * (uint32_t)args->a.N;
                    if (sidx & 1) { pos_step = T; pos_cur = p + 1 + j * T; w_step = 1; w_cur = tb.segw[seg] + j; }
                    else { pos_step = -T; pos_cur = p - T + 1 - j * T; w_step = -1; w_cur = tb.segw[seg] - j; }
                };
                enter(first);
#pragma unroll
                for (int r = 0; r < IPT; r++) {
                    const int idx = first + r;
                    if (idx >= seg_end && seg < 2 * args->a.L - 1) {
                        do { seg++; } while (seg < 2 * args->a.L - 1 && tb.seg[seg + 1] <= idx);
                        enter(idx);
                    }
                    koff[r] = h_base + (uint32_t)(idx < W ? min(max(pos_cur, 0), n - 1) : 0);
                    qv[r] = q_seg;
                    rp[r] = (uint32_t)(idx < W ? w_cur : 0);    // the sort's payload: the window's place in the table
                    pos_cur += pos_step;
                    w_cur += w_step;
                }
                float kv[IPT];
#pragma unroll
                for (int r = 0; r < IPT; r++) kv[r] = kbase[koff[r]];
                int most = 0;
#pragma unroll
                for (int r = 0; r < IPT; r++) {
                    const int idx = first + r;
                    const uint32_t bits = __builtin_bit_cast(uint32_t, fabsf(kv[r] - qv[r]));
                    k[r] = idx < W ? bits : 0xffffffffu;      // pads sort last and stay last
                    most = max(most, idx < W ? (int)bits : 0);
                }
                probes += IPT;
                most = wave_max_i32(most);
                if (lane == 0) atomicMax(&misc[dMaxBits], (uint32_t)most);
            }
            __syncthreads();
            PHASE_END(1);
            const uint32_t max_bits = (uint32_t)__builtin_amdgcn_readfirstlane((int)misc[dMaxBits]);
            const float scale = 4294966016.0f / __builtin_bit_cast(float, max_bits);
            bool ranked = false;
            int fix_rank;
            uint32_t fix_place;
            if (!by_radix && max_bits < kInfBits && scale < 4e38f) {      // (else, or if priorities cluster, the radix passes)
                // two windows of equal list words: windows of one stream keep their order, others are
                // compared by their priorities, then by their order in the layout
                auto before = [&](int x, int z) __attribute__((always_inline)) {
                    auto seg_of = [&](int idx) {
                        int lo = 0, hi = 2 * args->a.L - 1;
                        while (lo < hi) {
                            const int mid = (lo + hi) >> 1;
                            if (tb.seg[mid + 1] <= idx) lo = mid + 1; else hi = mid;
                        }
                        return lo;
                    };
                    const int gx = seg_of(x), gz = seg_of(z);
                    if (gx == gz) return x < z;
                    auto prio = [&](int idx, int g) {
                        const int sidx = tb.segstream[g], i = m * args->a.L + (sidx >> 1);
                        Stream st;
                        st.key = args->a.skeys + (int64_t)i * args->a.N + off;
                        st.n = n; st.T = T; st.p = tb.p[i]; st.side = sidx & 1; st.q = tb.qp[i];
                        return stream_prio_bits(st, idx - tb.seg[g]);
                    };
                    const uint32_t bx = prio(x, gx), bz = prio(z, gz);
                    return bx != bz ? bx < bz : x < z;
                };
                ranked = lds_bucket_ranks<NT, IPT, kBucketBits>(
                    k, rp, W, scale, tb.stage, tb.stage + IPT * NT + 4, scan_tmp, reinterpret_cast<unsigned long long*>(tb.wlist),
                    kWaves * kWlist * 2 / 8, tid, fix_rank, fix_place, before);
                if (ranked) {
                    __syncthreads();                    // the table takes the lists' room
                    uint16_t* steps = step_table(tb);
                    int own = W - tid * IPT;            // (opaque: no lane masks kept for it across the ranking)
                    asm volatile("" : "+v"(own));
#pragma unroll
                    for (int r = 0; r < IPT; r++)
                        if (r < own) steps[rp[r] & 0xffffu] = (uint16_t)(((rp[r] >> 16) << 1) | 1);
                    __syncthreads();
                    if (fix_rank >= 0) steps[fix_place] = (uint16_t)((fix_rank << 1) | 1);
                }
            }
            if (ranked) break;
            if (by_radix) {
                uint32_t vor = 0, vand = 0xffffffffu;
                int own = W - tid * IPT;
                asm volatile("" : "+v"(own));
#pragma unroll
                for (int r = 0; r < IPT; r++) {
                    const bool real = r < own;
                    vor |= real ? k[r] : 0u;
                    vand &= real ? k[r] : 0xffffffffu;
                }
                for (int o = 32; o > 0; o >>= 1) {
                    vor |= (uint32_t)__shfl_xor((int)vor, o, kWave);
                    vand &= (uint32_t)__shfl_xor((int)vand, o, kWave);
                }
                if (lane == 0) { atomicOr(&misc[dOr], vor); atomicAnd(&misc[dAnd], vand); }
                __syncthreads();
                // (the pads need no pass of their own: they start behind every window, every
                //  digit of theirs is the largest, and the passes are stable)
                const uint32_t varying = misc[dOr] ^ misc[dAnd];
                lds_radix_passes<NT, IPT>(k, rp, tb.stage, tb.stage + IPT * NT + 4, scan_tmp, varying);
                __syncthreads();
                uint16_t* steps = step_table(tb);
                uint32_t no_step = 0;
#pragma unroll
                for (int r = 0; r < IPT; r++) {
                    const int sp = tid * IPT + r;
                    const bool never = k[r] >= kInfBits;
                    if (sp < W) steps[rp[r] & 0xffffu] = never ? (uint16_t)kNever : (uint16_t)((sp << 1) | 1);      // (the first W sorted items are the windows)
                    no_step += sp < W && never ? 1u : 0u;
                }
                if (no_step) atomicAdd(&misc[dNoStep], no_step);
                break;
            }
            __syncthreads();
            }
            __syncthreads();
            maxw = max(maxw, (unsigned long long)(misc[dWin] - misc[dNoStep]));
            PHASE_END(2);

            // ---- every point: the latest of the steps of its L windows ------------------
            // A thread takes eight consecutive points at a time: their positions in one simple
            // index are one 16-byte read of the inverse permutation (slices start on 2-byte
            // boundaries; the reads need no more).  The reads for two simple indices make a
            // group, and the reads of three groups are in flight while one group is looked up
            // (the rows read for distances by the CU's other workgroup keep the memory system
            // busy: a read takes microseconds).  The last chunk of a slice is moved back to end at the
            // slice's end: some points are then looked up twice, with the same result.  The
            // phase is bound by vector-ALU issue, so the lookups are kept branch-free and short:
            // for a power-of-two T two points at a time in packed 16-bit arithmetic, otherwise
            // with 24-bit multiplies (32-bit ones run at a quarter of the rate).
            if constexpr (!WINDOWS) {
            const uint16_t* invm = args->a.inv + (int64_t)m * args->a.L * args->a.N + off;
            auto store_time = [&](int pt, uint32_t b) __attribute__((always_inline)) {
                const uint32_t old = tb.time[pt];      // ties: the earlier composite stays
                if ((b >> 1) < (old >> 1)) tb.time[pt] = (uint16_t)b;
            };
            if (n < 8) {
                for (int pt = tid; pt < n; pt += NT) {
                    uint32_t best = 0u;
                    for (int h = 0; h < args->a.L; h++) {
                        const int i = m * args->a.L + h;
                        const uint32_t x = (uint32_t)invm[(int64_t)h * args->a.N + pt] + (uint32_t)tb.shift[i];
                        const uint32_t w = T > 1 ? __umulhi(x, args->a.T_magic) : x;
                        best = max(best, (uint32_t)tb.rank16[tb.tabbase[i] + w] - (x - w * (uint32_t)T != 0u ? 1u : 0u));
                    }
                    store_time(pt, best);
                }
            } else {
                auto run = [&](auto path_tag) __attribute__((always_inline)) {
                    constexpr int kPath = decltype(path_tag)::value;     // 0: T = 2^s; 1: any other T
                    constexpr int kH = 2, kD = 4, kChunk = NT * 8;
                    const int ngrp = (args->a.L + kH - 1) / kH;
                    // (a wavefront whose points of a chunk all lie past the slice's end has no part in that chunk)
                    const int own_chunks = max(0, (n - 8 * kWave * __builtin_amdgcn_readfirstlane(wave) + kChunk - 1) / kChunk);
                    const int NG = own_chunks * ngrp;
                    const uint32_t tab0 = (uint32_t)(uintptr_t)(lds_u16*)tb.rank16;      // LDS address
                    // path 0
                    const uint16_t sh = (uint16_t)floor_log2(T);
                    const u16x2 sh_pk = {sh, sh};
                    const u16x2 mask_pk = {(uint16_t)(T - 1), (uint16_t)(T - 1)};
                    const u16x2 one_pk = {1, 1};
                    // path 1: d / T for 0 <= d < 65536 is the upper 32 bits of (d << q_sh) *
                    // ceil(2^(32 - q_sh) / T); rounding the factor up adds less than 1 / T to d / T,
                    // which never reaches the next integer; q_sh = 8 serves 2 <= T <= 256, q_sh = 0
                    // the wider windows, and both factors stay below 2^24 either way.
                    const uint32_t q_sh = T <= 256 ? 8u : 0u;
                    const uint32_t q_magic = (uint32_t)(((1ull << (32 - q_sh)) + (uint32_t)T - 1) / (uint32_t)T);
                    const uint32_t q_T = (uint32_t)T << q_sh;
                    uint32_t best[kPath == 0 ? 4 : 8];     // path 0: two points a word
                    auto chunk_start = [&](int c0) { return min(c0 + 8 * tid, n - 8); };
                    auto issue = [&](int c0, int h0, u32x4 (&pv)[kH]) __attribute__((always_inline)) {
#pragma unroll
                        for (int hh = 0; hh < kH; hh++) {
                            const uint16_t* invh = invm + (int64_t)min(h0 + hh, args->a.L - 1) * args->a.N;
                            __builtin_memcpy(&pv[hh], invh + (uint32_t)chunk_start(c0), 16);
                        }
                    };
                    auto consume = [&](int c0, int h0, const u32x4 (&pv)[kH]) __attribute__((always_inline)) {
                        if (h0 == 0) {
#pragma unroll
                            for (int e = 0; e < (kPath == 0 ? 4 : 8); e++) best[e] = 0u;
                        }
                        // every table read of the group is issued before the first is used
                        uint32_t tv[kH][8];
                        u16x2 rem[kH][4];
#pragma unroll
                        for (int hh = 0; hh < kH; hh++) {
                            const int i = m * args->a.L + min(h0 + hh, args->a.L - 1);   // (past L: the last index again)
                            const uint32_t shift = (uint32_t)tb.shift[i];
                            const uint32_t tab = tab0 + 2 * (uint32_t)tb.tabbase[i];
                            const uint32_t wd[4] = {pv[hh].x, pv[hh].y, pv[hh].z, pv[hh].w};
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                if constexpr (kPath == 0) {
                                    const u16x2 shift_pk = {(uint16_t)shift, (uint16_t)shift};
                                    const u16x2 x = __builtin_bit_cast(u16x2, wd[j]) + shift_pk;
                                    const u16x2 w = x >> sh_pk;
                                    // (spelled out: the compiler's own form of min(r, 1) is
                                    //  two compares, two selects and a byte permute)
                                    asm("v_pk_min_u16 %0, %1, %2" : "=v"(rem[hh][j]) : "v"(x & mask_pk), "v"(one_pk));
                                    // (one instruction takes a window's place out of its half, doubles it and
                                    //  adds the table's address)
                                    uint32_t a0, a1;
                                    asm("v_mad_u32_u16 %0, %1, 2, %2" : "=v"(a0) : "v"(w), "v"(tab));
                                    asm("v_mad_u32_u16 %0, %1, 2, %2 op_sel:[1,0,0,0]" : "=v"(a1) : "v"(w), "v"(tab));
                                    tv[hh][2 * j] = *(const lds_u16*)a0;
                                    tv[hh][2 * j + 1] = *(const lds_u16*)a1;
                                } else {
#pragma unroll
                                    for (int e = 0; e < 2; e++) {
                                        const uint32_t pos = e ? wd[j] >> 16 : wd[j] & 0xffffu;
                                        const uint32_t xs = (pos << q_sh) + (shift << q_sh);
                                        uint32_t w;
                                        asm("v_mul_hi_u32_u24 %0, %1, %2" : "=v"(w) : "s"(q_magic), "v"(xs));
                                        tv[hh][2 * j + e] = *(const lds_u16*)(tab + 2 * w);
                                        const uint32_t off_lane = (uint32_t)((uint32_t)__umul24(w, q_T) != xs);
                                        if (e) rem[hh][j].y = (uint16_t)off_lane; else rem[hh][j].x = (uint16_t)off_lane;
                                    }
                                }
                            }
                        }
#pragma unroll
                        for (int hh = 0; hh < kH; hh++)
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                if constexpr (kPath == 0) {
                                    const u16x2 val =
                                        __builtin_bit_cast(u16x2, tv[hh][2 * j] | (tv[hh][2 * j + 1] << 16)) - rem[hh][j];
                                    best[j] = __builtin_bit_cast(uint32_t,
                                        __builtin_elementwise_max(__builtin_bit_cast(u16x2, best[j]), val));
                                } else {
                                    best[2 * j] = max(best[2 * j], tv[hh][2 * j] - (uint32_t)rem[hh][j].x);
                                    best[2 * j + 1] = max(best[2 * j + 1], tv[hh][2 * j + 1] - (uint32_t)rem[hh][j].y);
                                }
                            }
                        if (h0 + kH >= args->a.L) {
                            // (read, choose, write back unconditionally: a point that two threads
                            //  hold, at the moved-back end of a slice, gets the same value from both)
                            const int pt0 = chunk_start(c0);
                            uint32_t old[8];
#pragma unroll
                            for (int e = 0; e < 8; e++) old[e] = tb.time[pt0 + e];
#pragma unroll
                            for (int e = 0; e < 8; e++) {
                                uint32_t b;
                                if constexpr (kPath == 0) b = (best[e >> 1] >> ((e & 1) * 16)) & 0xffffu;
                                else b = best[e];
                                // ties: the earlier composite stays
                                tb.time[pt0 + e] = (uint16_t)((b >> 1) < (old[e] >> 1) ? b : old[e]);
                            }
                        }
                    };
                    // A ring of kD groups: the reads of the next kD - 1 groups are in flight while
                    // one group is looked up.  The loop body has no branch (the counters of reads
                    // under way are only exact in straight-line code): past the last group the reads
                    // repeat the slice's last chunk and the lookups change nothing that is stored.
                    int cc = 0, hc = 0, ci = 0, hi = 0;     // (chunk base, first simple index) of the group to consume / to issue
                    auto advance = [&](int& c, int& h) { h += kH; if (h >= args->a.L) { h = 0; c += kChunk; } };
                    u32x4 pv[kD][kH];
                    if (NG == 0) return;
#pragma unroll
                    for (int d = 0; d < kD; d++) {
                        issue(ci, hi, pv[d]);
                        advance(ci, hi);
                    }
                    for (int g = 0; g < NG; g += kD) {
#pragma unroll
                        for (int d = 0; d < kD; d++) {
                            consume(cc, hc, pv[d]);
                            advance(cc, hc);
                            issue(ci, hi, pv[d]);
                            advance(ci, hi);
                        }
                    }
                };
                if ((T & (T - 1)) == 0) run(std::integral_constant<int, 0>{});
                else run(std::integral_constant<int, 1>{});
            }
            __syncthreads();
            PHASE_END(3);
            }
        }
        // ---- by windows: a point's windows in a composite end at the latest of their steps, and what the stop counts are the windows whose
        // first lane is a point none of whose other windows there comes later.  So the first lanes of all windows are looked up instead of
        // all points, and later the points of near tiles (25000 points, windows of 128, 24 simple indices: 4700 first lanes, 600000 positions).
        // A point's positions lie side by side (point_rows), eight at a time: 16 bytes for each look-up of a composite.  Bound by the
        // reads, each from a line of its own, and their latency: several points a lane are under way together.  Without a time per point an
        // item takes 28 instead of 75 KB of LDS: four workgroups of four wavefronts to a CU instead of two of eight.  (512 queries on 10M unit
        // vectors of 96, 51700 items: 12.8 -> 6.6 ms in all, with the candidates of near tiles listed together, below.)
        const int lp = (args->a.L + 7) & ~7;
        // the latest (doubled, with bit 0 set, or kNever) of the steps of the windows that hold points pts under composites ms
        auto latest = [&](auto utag, const int (&pts)[decltype(utag)::value], const int (&ms)[decltype(utag)::value],
                          uint32_t (&late)[decltype(utag)::value]) __attribute__((always_inline)) {
            constexpr int U = decltype(utag)::value;
            ArgsPtr args = fresh_args();
            const int L = args->a.L, M = args->a.M;
            const uint16_t* rows = args->a.point_rows + off * M * lp;
            const uint32_t tab_at = (uint32_t)(uintptr_t)(lds_u16*)reinterpret_cast<uint16_t*>(smem + args->y.off_tab);
            const uint32_t q_sh = T <= 256 ? 8u : 0u, q_magic = (uint32_t)(((1ull << (32 - q_sh)) + (uint32_t)T - 1) / (uint32_t)T);
#pragma unroll
            for (int u = 0; u < U; u++) late[u] = 0;
            for (int h0 = 0; h0 < L; h0 += 8) {
                u32x4 v[U];
#pragma unroll
                for (int u = 0; u < U; u++) v[u] = *reinterpret_cast<const u32x4*>(rows + (uint32_t)((pts[u] * M + ms[u]) * lp + h0));
                auto four = [&](int half) __attribute__((always_inline)) {
                    uint32_t at[4][U];                       // the windows' places in the tables, then their steps
#pragma unroll
                    for (int e = 0; e < 4; e++) {
#pragma unroll
                        for (int u = 0; u < U; u++) {
                            const int i = ms[u] * L + min(h0 + 4 * half + e, L - 1);      // (past the last: that one again, here and in the table)
                            const uint32_t place = (uint32_t)tb.shift[i];
                            const uint32_t wd = half ? (e < 2 ? v[u].z : v[u].w) : (e < 2 ? v[u].x : v[u].y);
                            const uint32_t xs = ((e & 1 ? wd >> 16 : wd & 0xffffu) + (place & 0xffffu)) << q_sh;
                            uint32_t w;
                            asm("v_mul_hi_u32_u24 %0, %1, %2" : "=v"(w) : "s"(q_magic), "v"(xs));
                            at[e][u] = tab_at + 2 * (w + (place >> 16));
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int u = 0; u < U; u++) late[u] = max(late[u], (uint32_t)*(const lds_u16*)at[e][u]);
                };
                four(0);
                if (h0 + 4 < L) four(1);
            }
        };
        // ---- stop step from the histogram of the steps of lane-0 candidates -----------
        const int HW = ((int)maxw + 2) / 2;                 // 32-bit words of the histogram (two steps each)
        uint32_t* hist = WINDOWS ? reinterpret_cast<uint32_t*>(smem + args->y.off_hist) : tb.stage;
        for (int w = tid; w < HW; w += NT) hist[w] = 0;
        if (tid == 0) { misc[dArmed] = 0xffffffffu; misc[dMaxc] = 0xffffffffu; misc[dMore] = 0; }
        __syncthreads();
        if constexpr (WINDOWS) {
            // (step, composite, point) of the first lanes that are promoted there, then of those those that no composite promotes sooner
            constexpr int kListed = NT * IPT / 2, U = 4;
            constexpr unsigned long long kSooner = 1ull << 63;
            unsigned long long* list = reinterpret_cast<unsigned long long*>(tb.stage);
            const uint16_t* tab = reinterpret_cast<const uint16_t*>(smem + args->y.off_tab);
            const int M = args->a.M, L = args->a.L;
            auto sooner = [&](uint32_t late, int m, uint32_t step, int own) { return (late >> 1) < step || ((late >> 1) == step && m < own); };
            const int parts = n / (T * kWave) + 1, wave_s = __builtin_amdgcn_readfirstlane(wave);      // (of 64 windows, of a simple index)
            for (int c0 = wave_s * U; c0 < I * parts; c0 += kWaves * U) {
                int pts[U], ms[U];
                uint32_t mine[U], late[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int c = min(c0 + u, I * parts - 1), i = c / parts;
                    const uint32_t place = (uint32_t)tb.shift[i];
                    const int shift = (int)(place & 0xffffu);
                    const int j = (shift + T - 1) / T + (c - i * parts) * kWave + lane, at = j * T - shift;
                    mine[u] = c0 + u < I * parts && at < n ? (uint32_t)tab[(place >> 16) + (uint32_t)j] : kNever;
                    ms[u] = i / L;
                    pts[u] = args->a.sids[(int64_t)i * args->a.N + off + min(at, n - 1)];
                }
#pragma unroll
                for (int u = 0; u < U; u++) pts[u] -= (int)off;
                latest(std::integral_constant<int, U>{}, pts, ms, late);
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const bool in = mine[u] != kNever && late[u] <= mine[u];
                    const unsigned long long all = __ballot(in);
                    if (all == 0) continue;
                    uint32_t first = 0;
                    if (lane == 0) first = atomicAdd(&misc[dMore], (uint32_t)__popcll(all));
                    first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
                    const uint32_t slot = first + (uint32_t)__popcll(all & ((1ull << lane) - 1ull));
                    if (in && slot < (uint32_t)kListed)
                        list[slot] = ((unsigned long long)(mine[u] >> 1) << 32) | ((uint32_t)ms[u] << 16) | (uint32_t)pts[u];
                    if (first + (uint32_t)__popcll(all) > (uint32_t)kListed) {      // (no room left: looked at here)
                        bool real = in && slot >= (uint32_t)kListed;
                        for (int m = 0; m < M; m++) {
                            const int one_pt[1] = {pts[u]}, one_m[1] = {m};
                            uint32_t l1[1];
                            latest(std::integral_constant<int, 1>{}, one_pt, one_m, l1);
                            if (m != ms[u] && sooner(l1[0], m, mine[u] >> 1, ms[u])) real = false;
                        }
                        if (real) atomicAdd(&hist[mine[u] >> 2], 1u << ((mine[u] >> 1 & 1u) * 16));
                    }
                }
            }
            __syncthreads();
            const int listed = min((int)misc[dMore], kListed), pairs = listed * (M - 1);      // (with every other composite)
            for (int e0 = 0; e0 < pairs; e0 += NT * U) {
                int pts[U], ms[U], es[U];
                uint32_t late[U], step[U], own[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int e = min(e0 + u * NT + tid, pairs - 1), other = e / listed;
                    es[u] = e - other * listed;
                    const unsigned long long v = list[es[u]];
                    pts[u] = (int)((uint32_t)v & 0xffffu);
                    own[u] = (uint32_t)v >> 16;
                    step[u] = (uint32_t)(v >> 32) & 0x7fffu;
                    ms[u] = (int)own[u] + 1 + other;
                    if (ms[u] >= M) ms[u] -= M;
                }
                latest(std::integral_constant<int, U>{}, pts, ms, late);
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (sooner(late[u], ms[u], step[u], (int)own[u])) reinterpret_cast<uint32_t*>(list)[2 * es[u] + 1] = (uint32_t)(kSooner >> 32);
            }
            if (pairs > 0) __syncthreads();
            for (int e = tid; e < listed; e += NT) {
                const uint32_t step = (uint32_t)(list[e] >> 32);
                if (!(step >> 31)) atomicAdd(&hist[step >> 1], 1u << ((step & 1u) * 16));
            }
        } else {
            for (int pt = tid; pt < n; pt += NT) {
                const uint32_t v = tb.time[pt];
                if ((v & 1u) && (v >> 1) != (kNever & 0x7fffu)) atomicAdd(&hist[v >> 2], 1u << (((v >> 1) & 1u) * 16));
            }
        }
        __syncthreads();
        {
            const int per = (HW + NT - 1) / NT;           // words per thread, contiguous
            const int w0 = tid * per, w1 = min(HW, w0 + per);
            uint32_t sum = 0;
            for (int w = w0; w < w1; w++) { const uint32_t v = hist[w]; sum += (v & 0xffffu) + (v >> 16); }
            uint32_t incl = sum;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t t2 = (uint32_t)__shfl_up((int)incl, o, kWave);
                if (lane >= o) incl += t2;
            }
            if (lane == kWave - 1) scan_tmp[wave] = incl;
            __syncthreads();
            uint32_t run = incl - sum;
            for (int w2 = 0; w2 < wave; w2++) run += scan_tmp[w2];
            const uint32_t need_k = (uint32_t)args->a.k_stop;
            const uint32_t need_c = (uint32_t)min((int64_t)0x7fffffff, max((int64_t)1, args->a.max_cand));
            for (int w = w0; w < w1; w++) {
                const uint32_t v = hist[w];
                const uint32_t c_lo = run + (v & 0xffffu), c_hi = c_lo + (v >> 16);
                if (run < need_k && c_lo >= need_k) atomicMin(&misc[dArmed], (uint32_t)(2 * w));
                else if (c_lo < need_k && c_hi >= need_k) atomicMin(&misc[dArmed], (uint32_t)(2 * w + 1));
                if (run < need_c && c_lo >= need_c) atomicMin(&misc[dMaxc], (uint32_t)(2 * w));
                else if (c_lo < need_c && c_hi >= need_c) atomicMin(&misc[dMaxc], (uint32_t)(2 * w + 1));
                run = c_hi;
            }
        }
        __syncthreads();
        const uint32_t t_armed = (uint32_t)__builtin_amdgcn_readfirstlane((int)misc[dArmed]);
        const uint32_t t_maxc = (uint32_t)__builtin_amdgcn_readfirstlane((int)misc[dMaxc]);
        const bool stop = t_armed != 0xffffffffu;
        unsigned long long t_stop = ~0ull;                  // candidates: promoted at a step <= t_stop
        if (stop) {
            const unsigned long long last_needed = args->a.stop_at > 0 ? (unsigned long long)(args->a.stop_at - 1) : 0ull;
            const unsigned long long by_count = t_maxc != 0xffffffffu ? (unsigned long long)t_maxc : ~0ull;
            t_stop = max((unsigned long long)t_armed, min(last_needed, by_count));
        }
        const uint32_t t_lim = (uint32_t)min(t_stop, (unsigned long long)0x7ffe);   // every real step is below 0x7fff
        __syncthreads();                                    // the histogram's room is free again
        PHASE_END(4);

        // ---- distances of the candidates, k best ---------------------------------------
        // Every wavefront walks its share of the points and lists its candidates, a batch at a
        // time; entries that may be among the k best wait in the wavefront's share of the buffer
        // until the next merge.
        typedef float v4f __attribute__((ext_vector_type(4)));
        const bool vec4 = rows_vec4(args->a.data, args->a.dim);
        const int chunk = (n + kWaves - 1) / kWaves;
        const int wave_u = __builtin_amdgcn_readfirstlane(wave);
        const int at_end = min(n, (wave_u + 1) * chunk);
        int at = wave_u * chunk;                            // next point of this wavefront
        uint16_t* wl = tb.wlist + wave_u * kWlist;             // this wavefront's candidates
        int list_len = 0, list_pos = 0;
        uint32_t ncand = 0;
        int topn = 0;
        // In a call's rounds only the tiles of rows that can hold one of the round's wanted distances are gone through (one bit
        // each, in words of the scan's scratch that this phase does not use): 13000 candidates of 96 elements, k = 100, of 25000
        // rows in 196 tiles, a handful of them near: 76 -> 12 us per item.
        uint32_t* near_bits = scan_tmp + 48;
        const bool near = PICKED && args->a.near_bounds != nullptr;
        const int near_shift = args->a.near_shift;
        uint16_t* near_list = reinterpret_cast<uint16_t*>(tb.stage);      // the near tiles
        if (near) {
            if (tid < 16) near_bits[tid] = 0;
            if (tid == 0) { misc[dMore] = 0; misc[dWin] = 0; }
            __syncthreads();
            const float most = args->a.near_limit[(int64_t)qi * args->a.near_stride];
            const uint32_t* bounds = args->a.near_bounds + (int64_t)b * args->a.near_tiles * args->a.nq + qi;
            const int tiles = (n + (1 << near_shift) - 1) >> near_shift;
            for (int t = tid; t < tiles; t += NT)
                if (!(__builtin_bit_cast(float, bounds[(int64_t)t * args->a.nq]) > most)) {
                    atomicOr(&near_bits[t >> 5], 1u << (t & 31));
                    near_list[atomicAdd(&misc[dMore], 1u)] = (uint16_t)t;
                }
            __syncthreads();
        }
        // lists at least `want` candidates, while points are left
        auto list_more = [&](int want) {
            while (list_len - list_pos < want && at < at_end) {
                int end = at_end;
                if (near) {
                    const int t = at >> near_shift;
                    end = min(at_end, (t + 1) << near_shift);
                    if (!((uint32_t)__builtin_amdgcn_readfirstlane((int)near_bits[t >> 5]) >> (t & 31) & 1u)) { at = end; continue; }
                }
                if (list_pos > 0) {      // what is left moves to the front (one wavefront: its LDS operations keep their order)
                    const int rest = list_len - list_pos;
                    const uint16_t v = lane < rest ? wl[list_pos + lane] : (uint16_t)0;
                    __builtin_amdgcn_wave_barrier();
                    if (lane < rest) wl[lane] = v;
                    list_len = rest;
                    list_pos = 0;
                }
                const int pt = at + lane;
                uint32_t v = 0xffffu;
                if constexpr (WINDOWS) {
                    const int pts[1] = {min(pt, end - 1)};
                    for (int m = 0; m < fresh_args()->a.M; m++) {
                        const int ms[1] = {m};
                        uint32_t late[1];
                        latest(std::integral_constant<int, 1>{}, pts, ms, late);
                        v = min(v, late[0]);
                    }
                    if (pt >= end) v = 0xffffu;
                } else if (pt < end) {
                    v = tb.time[pt];
                }
                const bool is_cand = (v >> 1) <= t_lim;
                const unsigned long long m = __ballot(is_cand);
                if (is_cand) wl[list_len + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)pt;
                list_len += __popcll(m);
                at = near ? min(at + kWave, end) : at + kWave;
                ncand += (uint32_t)__popcll(m);
            }
            __builtin_amdgcn_wave_barrier();
        };
        // Distances of eight rows by one wavefront, all eight reads under way together: the sums and
        // their order are those of wave_row_dists, level by level; lane l has that of row l >> 3.
        auto eight_rows = [&](const int (&pts)[8]) -> float {
            float acc[8];
            const float* rows[8];                               // (the points are the same for all lanes: addresses in scalar registers)
            const float* data = args->a.data;
            const int dim = args->a.dim;
#pragma unroll
            for (int r = 0; r < 8; r++) { acc[r] = 0.f; rows[r] = data + (off + __builtin_amdgcn_readfirstlane(pts[r])) * dim; }
            if (vec4) {
                for (int j = lane * 4; j < dim; j += kWave * 4) {
                    v4f x[8];
#pragma unroll
                    for (int r = 0; r < 8; r++) x[r] = *reinterpret_cast<const v4f*>(rows[r] + j);
                    const float q0 = tb.q[j], q1 = tb.q[j + 1], q2 = tb.q[j + 2], q3 = tb.q[j + 3];
#pragma unroll
                    for (int r = 0; r < 8; r++) {
                        float dd = x[r].x - q0; acc[r] = __builtin_fmaf(dd, dd, acc[r]);
                        dd = x[r].y - q1; acc[r] = __builtin_fmaf(dd, dd, acc[r]);
                        dd = x[r].z - q2; acc[r] = __builtin_fmaf(dd, dd, acc[r]);
                        dd = x[r].w - q3; acc[r] = __builtin_fmaf(dd, dd, acc[r]);
                    }
                }
            } else {
                for (int j = lane; j < dim; j += kWave) {
                    float x[8];
#pragma unroll
                    for (int r = 0; r < 8; r++) x[r] = rows[r][j];
                    const float qj = tb.q[j];
#pragma unroll
                    for (int r = 0; r < 8; r++) { const float dd = x[r] - qj; acc[r] = __builtin_fmaf(dd, dd, acc[r]); }
                }
            }
            float v4[4], v2[2];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const bool up = (lane & 32) != 0;
                v4[i] = (up ? acc[i + 4] : acc[i]) + lane_xor<32>(up ? acc[i] : acc[i + 4]);
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const bool up = (lane & 16) != 0;
                v2[i] = (up ? v4[i + 2] : v4[i]) + lane_xor<16>(up ? v4[i] : v4[i + 2]);
            }
            const bool up = (lane & 8) != 0;
            float v = (up ? v2[1] : v2[0]) + lane_xor<8>(up ? v2[0] : v2[1]);
            v += lane_xor<4>(v); v += lane_xor<2>(v); v += lane_xor<1>(v);
            return sqrtf(v);
        };
        auto pack = [&](uint32_t score, int pt) { return ((unsigned long long)score << 32) | (uint32_t)(off + pt); };

        // Candidates by their rows' 8-bit codes (rows8.hip).  The distance d~ between coded row and coded
        // query is off by at most the two coding errors (their sum: err) and by the rounding of its square
        // (delta), so a candidate more than 2 err + delta's part behind the k-th smallest d~ cannot be
        // among the k best: the others -- k and some -- are kept, and only their rows are read.
        // What d~ may be at most, given the k-th smallest:
        const int rec = args->a.rows8_rec, code_bytes = (args->a.dim + 15) & ~15;
        const unsigned char* qrec = args->a.query8 + (int64_t)qi * (16 + 2 * code_bytes);
        enum { kBlind = 1, kRows = 8, kRows16 = 16, kRows32 = 32, kCodes8 = 108, kCodes16 = 116, kCodes64 = 164 };
        int path = args->a.blind ? kBlind : (!args->y.tiles ? kRows : (args->a.dim <= 64 ? kRows16 : kRows32));
        float q_scale = 0.f, q_n2 = 0.f, err = 0.f, delta = 0.f;
        if (args->a.rows8) {
            const float* qh = reinterpret_cast<const float*>(qrec);
            q_scale = qh[0]; q_n2 = qh[1];
            err = __builtin_bit_cast(float, args->a.rows8_bounds[2 * b]) + qh[2];
            delta = (__builtin_bit_cast(float, args->a.rows8_bounds[2 * b + 1]) + q_n2) * 9.5367431640625e-7f;   // 2^-20
            q_scale = uniform_f32(q_scale); q_n2 = uniform_f32(q_n2); err = uniform_f32(err); delta = uniform_f32(delta);
            if (__builtin_amdgcn_readfirstlane((int)misc[dUse8]) != kCodesOff) {
                if (err < 1e30f && delta < 1e30f) path = code_bytes <= 128 ? kCodes8 : (code_bytes <= 256 ? kCodes16 : kCodes64);
                else if (tid == 0) misc[dUse8] |= kCodesFailed;      // (no useful codes of these rows, or of this query)
            }
        }
        auto limit = [&](float d) {
            const float part = d * d > 4.0f * delta ? 2.0f * delta / d : 4.0f * sqrtf(delta);
            return (d + 2.0f * err + part) * 1.0001f;
        };
        // One batch of nb candidates (listed at cur) by their codes: G lanes read a record, 16 codes
        // each; the integer sums are exact.  Lane c has the entry (d~, point) of candidate c.
        auto batch_codes = [&](auto gtag, const uint16_t* cur, int nb) -> unsigned long long {
            constexpr int G = decltype(gtag)::value;            // lanes per record
            constexpr int RB = G < 32 ? G : 32;                 // records per lane group and batch
            constexpr int CB = kWave / G * RB;                  // candidates per batch
            constexpr int kInFlight = RB < 8 ? RB : 8;
            const int grp = lane / G, sl = lane & (G - 1);
            const bool has = sl * 16 < code_bytes;
            const int my_off = 16 + (has ? sl * 16 : 0);
            u32x4 qh = *reinterpret_cast<const u32x4*>(qrec + my_off);
            u32x4 ql = *reinterpret_cast<const u32x4*>(qrec + code_bytes + my_off);
            if (!has) qh = ql = u32x4{0, 0, 0, 0};              // (idle lanes add nothing)
            const unsigned char* base = args->a.rows8 + off * rec;
            const int mypt = (int)cur[min(lane & (CB - 1), nb - 1)];
            const float2 head = *reinterpret_cast<const float2*>(base + (uint32_t)mypt * (uint32_t)rec);
            int acc[RB];
#pragma unroll
            for (int r0 = 0; r0 < RB; r0 += kInFlight) {
                u32x4 x[kInFlight];
#pragma unroll
                for (int r = 0; r < kInFlight; r++) {
                    const int pt = (int)cur[min(grp * RB + r0 + r, nb - 1)];
                    x[r] = *reinterpret_cast<const u32x4*>(base + ((uint32_t)pt * (uint32_t)rec + (uint32_t)my_off));
                }
#pragma unroll
                for (int r = 0; r < kInFlight; r++) {
                    int dh = __builtin_amdgcn_sdot4((int)x[r].x, (int)qh.x, 0, false);
                    dh = __builtin_amdgcn_sdot4((int)x[r].y, (int)qh.y, dh, false);
                    dh = __builtin_amdgcn_sdot4((int)x[r].z, (int)qh.z, dh, false);
                    dh = __builtin_amdgcn_sdot4((int)x[r].w, (int)qh.w, dh, false);
                    int dl = __builtin_amdgcn_sdot4((int)x[r].x, (int)ql.x, dh << 7, false);
                    dl = __builtin_amdgcn_sdot4((int)x[r].y, (int)ql.y, dl, false);
                    dl = __builtin_amdgcn_sdot4((int)x[r].z, (int)ql.z, dl, false);
                    acc[r0 + r] = __builtin_amdgcn_sdot4((int)x[r].w, (int)ql.w, dl, false);
                }
            }
            if constexpr (G > RB) {
#pragma unroll
                for (int r = 0; r < RB; r++) acc[r] += lane_xor<32>(acc[r]);
            }
            const int dot = group_row_sums<RB>(acc, sl);           // of candidate lane (mod CB)
            const float d2 = head.y + q_n2 - 2.0f * (head.x * q_scale * (float)dot);
            const float d = sqrtf(fmaxf(d2, 0.0f));
            return ((unsigned long long)__builtin_bit_cast(uint32_t, d) << 32) | (uint32_t)mypt;
        };
        // The same by whole rows of at most 4 * GL elements: GL lanes read a row (16 bytes each), every
        // lane group takes GL rows; the partial sums a lane ends up with are reduced for all its rows
        // together, which leaves lane c of the wavefront with the distance of candidate c.
        auto batch_rows = [&](auto gtag, const uint16_t* cur, int nb) -> unsigned long long {
            constexpr int GL = decltype(gtag)::value;
            constexpr int kInFlight = 8;                        // row reads under way per lane
            const int grp = lane / GL, sl = lane & (GL - 1);
            const int j = sl * 4;
            const bool has = j < args->a.dim;
            float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
            if (has) { q0 = tb.q[j]; q1 = tb.q[j + 1]; q2 = tb.q[j + 2]; q3 = tb.q[j + 3]; }
            const float* base = args->a.data + off * args->a.dim + (has ? j : 0);
            float acc[GL];
#pragma unroll
            for (int r0 = 0; r0 < GL; r0 += kInFlight) {
                v4f x[kInFlight];
#pragma unroll
                for (int r = 0; r < kInFlight; r++) {
                    // (lanes beyond the row's end read its head and add nothing: a load
                    //  under a condition would wait for the loads before it)
                    const int pt = (int)cur[min(grp * GL + r0 + r, nb - 1)];
                    x[r] = *reinterpret_cast<const v4f*>(base + pt * args->a.dim);
                }
#pragma unroll
                for (int r = 0; r < kInFlight; r++) {
                    float s2 = 0.f;
                    float dd = x[r].x - q0; s2 = __builtin_fmaf(dd, dd, s2);
                    dd = x[r].y - q1; s2 = __builtin_fmaf(dd, dd, s2);
                    dd = x[r].z - q2; s2 = __builtin_fmaf(dd, dd, s2);
                    dd = x[r].w - q3; s2 = __builtin_fmaf(dd, dd, s2);
                    acc[r0 + r] = has ? s2 : 0.f;
                }
            }
            const float total = group_row_sums<GL>(acc, sl);      // of candidate grp * GL + sl = lane
            return pack(__builtin_bit_cast(uint32_t, sqrtf(total)), (int)cur[min(lane, nb - 1)]);
        };
        // Every wavefront goes through its batches; entries that may still be among the k best go to its share
        // of the buffer.  What may be is known from a histogram of the scores seen so far (256 bins over
        // the range of every wavefront's first batch, one for all, without a barrier: a count that is
        // read late only loosens the cut): the upper edge of the bin that holds the k-th smallest bounds it.  A share that is full
        // is cleared of what has fallen behind the cut meanwhile; where that makes no room, the round
        // ends: the shares are sorted in with what is held.  Nearly always there is one such sort, at the end.
        // Compared by codes, the kept entries get their exact distances before that sort.
        // Bound by the latency of the records' reads (eight 16-byte reads per lane under way).  12801 candidates
        // of 96 elements, k = 100, two workgroups per CU: 75 us per item, 140 by whole rows; 1285 of 960
        // elements, k = 10: 55, and 198 by whole rows.
        unsigned long long* res = tb.sortbuf;                      // where the result lies
        // ---- few candidates in near tiles, as nearly always: all wavefronts list them together, form their distances, eight rows and more to a
        // wavefront under way, and sort them.  (3.5 tiles of 128 rows and 230 candidates an item, k = 100: 51 us when every wavefront kept to its
        // share of the points, most of them waiting for one.)
        bool few = false;
        if (near) {
            const int tiles = (int)misc[dMore];
            // room: the tiles, the results, the candidates
            const int tile_bytes = (2 * tiles + 7) & ~7;
            int room = NT;
            while (room < 1024 && tile_bytes + 2 * room * 10 <= args->y.whole_bytes) room <<= 1;
            res = reinterpret_cast<unsigned long long*>(reinterpret_cast<unsigned char*>(tb.stage) + tile_bytes);
            uint16_t* cand = reinterpret_cast<uint16_t*>(res + room);
            if (tile_bytes + room * 10 <= args->y.whole_bytes) {
                constexpr int U = WINDOWS ? 2 : 1;
                const int rows = tiles << near_shift;
                for (int r0 = 0; r0 < rows; r0 += NT * U) {
                    int pts[U];
                    uint32_t v[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int r = r0 + u * NT + tid;
                        const int pt = r < rows ? ((int)near_list[r >> near_shift] << near_shift) + (r & ((1 << near_shift) - 1)) : n;
                        v[u] = pt < n ? 0u : 0xffffu;
                        pts[u] = min(pt, n - 1);
                    }
                    if constexpr (WINDOWS) {
                        uint32_t first[U];
#pragma unroll
                        for (int u = 0; u < U; u++) first[u] = 0xffffu;
                        for (int m = 0; m < fresh_args()->a.M; m++) {
                            int ms[U];
                            uint32_t late[U];
#pragma unroll
                            for (int u = 0; u < U; u++) ms[u] = m;
                            latest(std::integral_constant<int, U>{}, pts, ms, late);
#pragma unroll
                            for (int u = 0; u < U; u++) first[u] = min(first[u], late[u]);
                        }
#pragma unroll
                        for (int u = 0; u < U; u++) v[u] = max(v[u], first[u]);
                    } else {
#pragma unroll
                        for (int u = 0; u < U; u++) v[u] = max(v[u], (uint32_t)tb.time[pts[u]]);
                    }
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const bool in = (v[u] >> 1) <= t_lim;
                        const unsigned long long all = __ballot(in);
                        if (all == 0) continue;
                        uint32_t slot = 0;
                        if (lane == 0) slot = atomicAdd(&misc[dWin], (uint32_t)__popcll(all));
                        slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)slot) + (uint32_t)__popcll(all & ((1ull << lane) - 1ull));
                        if (in && slot < (uint32_t)room) cand[slot] = (uint16_t)pts[u];
                    }
                }
                __syncthreads();
                const int count = __builtin_amdgcn_readfirstlane((int)misc[dWin]);
                if (count <= room) {
                    few = true;
                    fresh_thread_ids();
                    // GL lanes to a row of at most 4 GL elements, eight rows to a lane group; the sums and their order are those of wave_row_dists
                    auto some_rows = [&](auto gtag) __attribute__((always_inline)) {
                        constexpr int GL = decltype(gtag)::value, kRows8 = 8 * (kWave / GL);
                        const int grp = lane / GL, sl = lane & (GL - 1), j = sl * 4;
                        const bool has = j < args->a.dim;
                        float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
                        if (has) { q0 = tb.q[j]; q1 = tb.q[j + 1]; q2 = tb.q[j + 2]; q3 = tb.q[j + 3]; }
                        const float* base = args->a.data + off * args->a.dim + (has ? j : 0);
                        for (int c0 = wave * kRows8; c0 < count; c0 += kWaves * kRows8) {
                            float acc[8];
                            v4f x[8];
#pragma unroll
                            for (int r = 0; r < 8; r++) x[r] = *reinterpret_cast<const v4f*>(base + (int)cand[min(c0 + grp * 8 + r, count - 1)] * args->a.dim);
#pragma unroll
                            for (int r = 0; r < 8; r++) {
                                float s2 = 0.f;
                                float dd = x[r].x - q0; s2 = __builtin_fmaf(dd, dd, s2);
                                dd = x[r].y - q1; s2 = __builtin_fmaf(dd, dd, s2);
                                dd = x[r].z - q2; s2 = __builtin_fmaf(dd, dd, s2);
                                dd = x[r].w - q3; s2 = __builtin_fmaf(dd, dd, s2);
                                acc[r] = has ? s2 : 0.f;
                            }
                            float v4[4], v2[2];
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                const bool up = (sl & (GL / 2)) != 0;
                                v4[i] = (up ? acc[i + 4] : acc[i]) + lane_xor<GL / 2>(up ? acc[i] : acc[i + 4]);
                            }
#pragma unroll
                            for (int i = 0; i < 2; i++) {
                                const bool up = (sl & (GL / 4)) != 0;
                                v2[i] = (up ? v4[i + 2] : v4[i]) + lane_xor<GL / 4>(up ? v4[i] : v4[i + 2]);
                            }
                            const bool up = (sl & (GL / 8)) != 0;
                            float v = (up ? v2[1] : v2[0]) + lane_xor<GL / 8>(up ? v2[0] : v2[1]);
                            if constexpr (GL > 16) v += lane_xor<2>(v);
                            v += lane_xor<1>(v);
                            const int c = c0 + grp * 8 + sl / (GL / 8);
                            if ((sl & (GL / 8 - 1)) == 0 && c < count) res[c] = pack(__builtin_bit_cast(uint32_t, sqrtf(v)), (int)cand[c]);
                        }
                    };
                    if (!args->y.tiles) {
                        for (int c0 = wave_u * 8; c0 < count; c0 += kWaves * 8) {
                            int pts[8];
#pragma unroll
                            for (int r = 0; r < 8; r++) pts[r] = (int)cand[min(c0 + r, count - 1)];
                            const float d = eight_rows(pts);
                            const int c = c0 + (lane >> 3);
                            if ((lane & 7) == 0 && c < count) res[c] = pack(__builtin_bit_cast(uint32_t, d), (int)cand[c]);
                        }
                    } else if (args->a.dim <= 64) {
                        some_rows(std::integral_constant<int, 16>{});
                    } else {
                        some_rows(std::integral_constant<int, 32>{});
                    }
                    int np = count <= kWave ? kWave : NT;
                    while (np < count) np <<= 1;
                    for (int j = count + tid; j < np; j += NT) res[j] = ~0ull;
                    if (NT > kWave && np == kWave) {
                        __syncthreads();
                        if (wave == 0) {
                            unsigned long long v[1] = {res[lane]};
                            wave_sort_u64(v, lane);
                            res[lane] = v[0];
                        }
                        __syncthreads();
                    } else {
                        bitonic_sort_u64_by<NT, NT == 64 ? 4 : 2>(res, np, tid);
                    }
                    topn = min(count, args->a.kcap);
                    if (wave == 0) ncand = (uint32_t)count;
                    if (tid == 0 && misc[dUse8] == kCodesDoubted) misc[dUse8] = kCodesOn;      // (the codes were not asked)
                    if (tid == 0 && misc[dUse8] == kCodesTried) misc[dUse8] = kCodesTried + kCodesFailed;
                }
            }
            __syncthreads();
        }
        uint32_t* bins = tb.stage;
        unsigned long long cut = ~0ull;                         // entries above it are out
        unsigned long long pend = ~0ull;                        // lane's entry of a batch that did not fit the share
        bool have_pend = false, first = true, last = false;
        float h_lo = 0.f, h_scale = 0.f;                        // (no histogram while the scale is 0)
        int batches = 0;
        while (!few) {
            const bool codes = path >= kCodes8;
            const int front = codes ? args->y.front8 : args->a.kcap, quota = codes ? args->y.quota8 : args->y.quota;
            const int CB = path == kRows ? 8 : (path == kCodes64 ? 32 : kWave);
            unsigned long long* my_slots = tb.sortbuf + front + wave_u * quota;
            auto score = [&](unsigned long long e) {
                return args->a.blind ? (float)(uint32_t)(e >> 32) : __builtin_bit_cast(float, (uint32_t)(e >> 32));
            };
            // (compared as a number before it becomes a bin: a NaN, which sorts behind everything, must not
            //  be counted among the nearest, where the conversion would put it)
            auto count = [&](bool keep, unsigned long long e) {
                const float at_bin = (score(e) - h_lo) * h_scale;
                if (keep && at_bin < (float)kBins) atomicAdd(&bins[max(0, (int)at_bin)], 1u);
            };
            auto tighten = [&]() {
                const u32x4 c = reinterpret_cast<const u32x4*>(bins)[lane];
                const uint32_t c1 = c.x + c.y, c2 = c1 + c.z, upto = wave_scan_u32(c2 + c.w), before = upto - (c2 + c.w);
                const uint32_t want = (uint32_t)args->a.kcap;
                const unsigned long long m = __ballot(upto >= want);
                if (m) {
                    const int bin = 4 * lane + (before + c.x >= want ? 0 : (before + c1 >= want ? 1 : (before + c2 >= want ? 2 : 3)));
                    const float edge = (h_lo + (float)(__shfl(bin, __ffsll((long long)m) - 1, kWave) + 1) / h_scale) * 1.00001f;
                    const uint32_t top = codes ? __builtin_bit_cast(uint32_t, limit(edge))
                                               : (args->a.blind ? (uint32_t)edge : __builtin_bit_cast(uint32_t, edge));
                    cut = uniform_u64(min(cut, ((unsigned long long)top << 32) | 0xffffffffull));
                }
            };
            int mine = 0, added = 0;
            bool any_more = false;
            // drops what has fallen behind the cut from the wavefront's share
            auto clear_share = [&]() {
                int kept = 0;
                for (int j0 = 0; j0 < mine; j0 += kWave) {
                    const unsigned long long v = j0 + lane < mine ? my_slots[j0 + lane] : ~0ull;
                    const bool stay = v != ~0ull && v <= cut;
                    const unsigned long long m = __ballot(stay);
                    __builtin_amdgcn_wave_barrier();
                    if (stay) my_slots[kept + __popcll(m & ((1ull << lane) - 1ull))] = v;
                    kept += __popcll(m);
                }
                __builtin_amdgcn_wave_barrier();
                mine = kept;
            };
            if (!last) {
                auto push = [&](bool keep, unsigned long long e) -> bool {
                    const unsigned long long m = __ballot(keep);
                    if (mine + __popcll(m) > quota) return false;
                    if (keep) my_slots[mine + __popcll(m & ((1ull << lane) - 1ull))] = e;
                    mine += __popcll(m);
                    return true;
                };
                if (have_pend) {
                    if (batches == 1 && h_scale > 0.f) count(pend != ~0ull, pend);      // (the first batch: now there is a histogram)
                    push(pend != ~0ull && pend <= cut, pend);      // (a share takes a whole batch)
                }
                have_pend = false;
                for (;;) {
                    list_more(CB);
                    const int nb = min(CB, list_len - list_pos);
                    if (nb <= 0) break;
                    const uint16_t* cur = wl + list_pos;
                    using std::integral_constant;
                    unsigned long long e;
                    bool valid = lane < nb;
                    // (opaque, or the compiler makes a copy of the whole loop, sorts included, for every path)
                    int how = path;
                    asm volatile("" : "+v"(how));
                    how = __builtin_amdgcn_readfirstlane(how);
                    fresh_thread_ids();      // (nor are lane-derived addresses of all paths kept across the batches)
                    if (how == kCodes8) e = batch_codes(integral_constant<int, 8>{}, cur, nb);
                    else if (how == kCodes16) e = batch_codes(integral_constant<int, 16>{}, cur, nb);
                    else if (how == kCodes64) e = batch_codes(integral_constant<int, 64>{}, cur, nb);
                    else if (how == kRows16) e = batch_rows(integral_constant<int, 16>{}, cur, nb);
                    else if (how == kRows32) e = batch_rows(integral_constant<int, 32>{}, cur, nb);
                    else if (how == kRows) {
                        int pts[8];
#pragma unroll
                        for (int r = 0; r < 8; r++) pts[r] = (int)cur[min(r, nb - 1)];
                        const float d = eight_rows(pts);
                        e = pack(__builtin_bit_cast(uint32_t, d), (int)cur[min(lane >> 3, nb - 1)]);
                        valid = (lane & 7) == 0 && (lane >> 3) < nb;
                    } else {      // blind: scored by the promoting step (:498-505), no row is read
                        const int pt = (int)cur[min(lane, nb - 1)];
                        e = pack(WINDOWS ? 0u : (uint32_t)tb.time[pt] >> 1, pt);
                    }
                    list_pos += nb;
                    batches++;
                    bool keep = valid && e <= cut;
                    if (first) { pend = keep ? e : ~0ull; have_pend = true; break; }
                    if (h_scale > 0.f) {
                        count(keep, e);
                        if (batches <= 4 || (batches & 3) == 0) {
                            tighten();
                            keep = keep && e <= cut;
                        }
                    }
                    if (!push(keep, e)) {
                        clear_share();
                        if (!push(keep, e)) { pend = keep ? e : ~0ull; have_pend = true; break; }
                    }
                }
                if (first) {      // the range of the histogram, and an empty one
                    const uint32_t bits = have_pend && pend != ~0ull ? __builtin_bit_cast(uint32_t, score(pend)) : 0x7fffffffu;
                    const uint32_t least = wave_min_u32(bits);
                    const int most = wave_max_i32(bits == 0x7fffffffu ? 0 : (int)bits);
                    if (lane == 0) { scan_tmp[24 + wave] = least; scan_tmp[40 + wave] = (uint32_t)most; }
                    for (int j = tid; j < kBins; j += NT) bins[j] = 0;
                    __syncthreads();
                    uint32_t lo = 0x7fffffffu, hi = 0;
                    for (int w2 = 0; w2 < kWaves; w2++) { lo = min(lo, scan_tmp[24 + w2]); hi = max(hi, scan_tmp[40 + w2]); }
                    const float f_lo = __builtin_bit_cast(float, lo), width = __builtin_bit_cast(float, hi) - f_lo;
                    if (lo < hi && hi < kInfBits && width > 1e-30f && width < 1e30f) { h_lo = uniform_f32(f_lo); h_scale = uniform_f32((float)kBins / width); }
                    first = false;
                    continue;
                }
                if (lane == 0) {
                    scan_tmp[8 + wave] = (uint32_t)mine;
                    scan_tmp[16 + wave] = have_pend || list_pos < list_len || at < at_end ? 1u : 0u;
                }
                __syncthreads();
                for (int w2 = 0; w2 < kWaves; w2++) { added += (int)scan_tmp[8 + w2]; any_more = any_more || scan_tmp[16 + w2] != 0u; }
                added = __builtin_amdgcn_readfirstlane(added);
                any_more = __builtin_amdgcn_readfirstlane((int)any_more) != 0;
            }
            int words = args->y.sort_cap;
            res = tb.sortbuf;
            bool whole = false;                                 // one round did: what is left fits the tables' room, side by side
            int left = topn;                                    // entries to be given their exact distances (codes)
            if (!last && !any_more && topn == 0) {
                if (h_scale > 0.f) tighten();
                clear_share();
                if (lane == 0) scan_tmp[wave] = (uint32_t)mine;
                __syncthreads();
                int base = 0;
                added = 0;
                for (int w2 = 0; w2 < kWaves; w2++) { const int c = (int)scan_tmp[w2]; if (w2 < wave_u) base += c; added += c; }
                added = __builtin_amdgcn_readfirstlane(added);
                int np = added <= kWave ? kWave : NT;
                while (np < added) np <<= 1;
                if (np * 8 <= args->y.whole_bytes) {
                    whole = true;
                    left = added;
                    words = np;
                    res = reinterpret_cast<unsigned long long*>(tb.stage);
                    for (int j = lane; j < mine; j += kWave) res[base + j] = my_slots[j];
                    for (int j = added + tid; j < np; j += NT) res[j] = ~0ull;
                    if (codes) __syncthreads();
                }
            }
            if (!whole && !last) {
                for (int j = mine + lane; j < quota; j += kWave) my_slots[j] = ~0ull;
                for (int j = topn + tid; j < front; j += NT) tb.sortbuf[j] = ~0ull;
                for (int j = front + kWaves * quota + tid; j < args->y.sort_cap; j += NT) tb.sortbuf[j] = ~0ull;
            } else if (codes) {
                for (int j0 = wave * 8; j0 < left; j0 += 8 * kWaves) {
                    int pts[8];
#pragma unroll
                    for (int r = 0; r < 8; r++) pts[r] = (int)(uint32_t)res[min(j0 + r, left - 1)];
                    const float d = eight_rows(pts);
                    const int j = j0 + (lane >> 3);
                    int mypt = pts[0];
#pragma unroll
                    for (int r = 1; r < 8; r++) mypt = (lane >> 3) == r ? pts[r] : mypt;
                    if ((lane & 7) == 0 && j < left) res[j] = pack(__builtin_bit_cast(uint32_t, d), mypt);
                }
                if (last) for (int j = topn + tid; j < args->y.sort_cap; j += NT) tb.sortbuf[j] = ~0ull;
            }
            if (NT > kWave && words == kWave) {
                __syncthreads();
                if (wave == 0) {
                    unsigned long long v[1] = {res[lane]};
                    wave_sort_u64(v, lane);
                    res[lane] = v[0];
                }
                __syncthreads();
            } else {
                bitonic_sort_u64_by<NT, NT == 64 ? 4 : (IPT > 9 ? 1 : 2)>(res, words, tid);
            }
            if (whole) { topn = min(added, args->a.kcap); break; }
            topn += added;
            if (last) { topn = min(topn, args->a.kcap); break; }
            if (topn >= args->a.kcap) {
                const unsigned long long kth = tb.sortbuf[args->a.kcap - 1];
                if (codes) {
                    cut = ((unsigned long long)__builtin_bit_cast(uint32_t, limit(__builtin_bit_cast(float, (uint32_t)(kth >> 32)))) << 32) | 0xffffffffull;
                    cut = uniform_u64(cut);
                    int lo = args->a.kcap, hi = topn;                     // words ascend: the first one past the cut
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if (tb.sortbuf[mid] <= cut) lo = mid + 1; else hi = mid;
                    }
                    topn = __builtin_amdgcn_readfirstlane(lo);
                } else {
                    cut = uniform_u64(kth);
                    topn = args->a.kcap;
                }
            }
            __syncthreads();
            if (topn > front) {
                // more has to be kept than the buffer holds: these rows lie too close together, as seen from this
                // query, for their codes; whole rows for this item
                if (tid == 0) misc[dUse8] |= kCodesFailed;
                path = !args->y.tiles ? kRows : (args->a.dim <= 64 ? kRows16 : kRows32);
                at = wave_u * chunk;
                list_len = list_pos = topn = batches = 0;
                ncand = 0;
                have_pend = false;
                first = true;
                h_scale = 0.f;
                cut = ~0ull;
                continue;
            }
            if (!any_more) {
                if (!codes) break;
                last = true;
            }
        }
        if (lane == 0) atomicAdd(&misc[dCand], ncand);
        for (int j = tid; j < args->a.kcap; j += NT) part_out[j] = j < topn ? res[j] : ~0ull;
        PHASE_END(5);
        if (args->a.phase_ticks && tid == 0) atomicAdd(&args->a.phase_ticks[9], 1ull);
        if (tid == 0 && misc[dUse8] > kCodesOn) {
            const uint32_t use = misc[dUse8];
            int* doubt = reinterpret_cast<int*>(args->a.rows8_bounds) + 2 * args->a.B + b;
            const int have = __hip_atomic_load(doubt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            int change = have > 0 && have < kGiveUp ? -1 : 0;                                      // they did, doubted
            if (use > kCodesFailed) change = have < kGiveUp ? (have < kGiveUp - 1 ? max(1, 1 - have) : kRest + 1) : 0;
            if (use == kCodesTried) change = -kTrying;
            if (use == kCodesTried + kCodesFailed) change = kGiveUp + kRest - kTrying;
            if (change != 0) atomicAdd(doubt, change);
        }
        if (args->a.phase_ticks && tid == 0 && misc[dUse8] - 1u < kCodesFailed - 1u) atomicAdd(&args->a.phase_ticks[15], 1ull);

        // ---- hints for the batch kernel's routing, counters -----------------------------
        __syncthreads();
        const unsigned long long bound = (unsigned long long)n * args->a.L * T;
        unsigned long long steps = min(bound, maxw + 1);
        if (stop) steps = min(t_stop + 1, steps);
        if (args->a.stop_hint && tid == 0 && stop) record_stop(args->a.stop_hint, args->a.B, b, qi, (float)(t_stop + 1), (float)misc[dCand]);
        if (args->a.counters) {
            probes = wave_sum_u32(probes);
            if (lane == 0) atomicAdd(&misc[dProbes], probes);
            __syncthreads();
            if (tid == 0) {
                atomicAdd(&args->a.counters[(int64_t)qi * 4 + 0], (unsigned long long)n * I);
                atomicAdd(&args->a.counters[(int64_t)qi * 4 + 1], (unsigned long long)misc[dCand]);
                atomicAdd(&args->a.counters[(int64_t)qi * 4 + 2], (unsigned long long)misc[dProbes]);
                atomicAdd(&args->a.counters[(int64_t)qi * 4 + 3], steps);
            }
        }
    }
}

#undef PHASE_END

template <int NT, int IPT, int WAVES, int KIND>
int launch_dense(const DenseArgs& args, unsigned grid, hipStream_t s) {
    static DeviceOnce once;
    const int rc = once.run([]() -> int {
        DCIH_HIP(hipFuncSetAttribute((const void*)traverse_dense_kernel<NT, IPT, WAVES, KIND>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        return 0;
    });
    if (rc) return rc;
    hipLaunchKernelGGL((traverse_dense_kernel<NT, IPT, WAVES, KIND>), dim3(grid), dim3(NT), args.y.lds_bytes, s, args);
    DCIH_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// By windows: n / T + 3 first lanes of every simple index cost two reads from random lines and L look-ups each, by points
// every one of the n costs one look-up that a coalesced read feeds; a read of a line of its own takes as long as a dozen look-ups.
// What decides beyond that is the LDS: a time for every point takes room that leaves fewer workgroups to a CU, two from about 16000 points on.  1000 queries on 1M
// rows, us by points and by windows: unit vectors, 8 indices, windows of 128, partitions of 8000 points 1437, 1297; 10000 1602, 1462; 12500 1826, 1638; 16129
// 2393, 1818.  Normal rows, 12 indices, windows of 96: 1360, 1223; 1664, 1422; 2105, 1622; 3778, 2400.  A noisy manifold, 12 indices, windows of 64: 1550, 1577; 1602,
// 1573; 2539, 2437; 3948, 3944.  Shorter partitions give between 0.80 and 1.07 of their times by points, and calls that wait for single items lose a tenth.
bool point_rows_pay(const QueryArgs& a) {
    return a.pick_rule == 2 || (a.ppb >= 8000 && (double)a.nq * (double)a.B * a.share >= 4096.0);
}
bool point_rows_fit(int64_t ppb, int M, int L, int T) {
    return ppb <= 32766 && (double)(ppb / T + 3) * (double)(L + 24) < 0.7 * (double)ppb && (int64_t)L * (ppb / T + 3) <= 9 * 512 && M <= 64 && L <= 64;
}

bool dense_traversal_supported(const QueryArgs& a, size_t* lds_bytes) {
    if (!a.inv || a.ppb > 32766 || a.T < 1) return false;
    if (a.M > 64 || a.L > 64 || a.kcap > 512 || (int64_t)a.L * a.N >= 0x7fffffffLL) return false;
    if (dense_max_windows(a) >= 0x7fff || a.ppb + (int64_t)a.T >= 65536) return false;
    if (a.xcds < 1 || a.xcds > 32 || (int64_t)a.nq * (a.B + a.xcds) >= 0x7fffffffLL) return false;
    const DenseLayout y = make_dense_layout(a);
    if (y.ipt == 0) return false;
    if (lds_bytes) *lds_bytes = y.lds_bytes;
    return y.lds_bytes <= kMostDenseLds;
}

int query_dense_items(const QueryArgs& a_in, hipStream_t s) {
    QueryArgs a = a_in;
    const DenseLayout y = make_dense_layout(a);
    if (y.ipt == 0) return fail(-4, "query: this shape does not fit the dense traversal kernel");
    a.q_first = 0;
    a.q_count = a.nq;
    // Items whose number only the device knows (a list), and few items, are shared out by strides among enough
    // workgroups to fill the device.  Else one workgroup takes one item, or as short a run of neighbouring ones
    // as a launch of 2^32 - 1 threads covers: workgroups start in order, so a die's resident ones work on
    // neighbouring queries of one partition and its slices stay in the L2, where resident workgroups that stride
    // over everything drift apart into several partitions (20M points, 900 partitions, 2000 queries: 984 ms by
    // strides, 608 in order).  From eight times as many items as the die holds at a time in order is 0 to 13 %
    // faster; below, starting more workgroups can cost up to 5 % (2000 points, 3200 items: 211 and 222 us), and
    // so it can where registers leave one workgroup to a CU, which nothing covers while the next one
    // starts (10000 points, 10030 windows: 390 and 397 ms).
    const int by_regs = (y.ipt > 15 ? 512 : 1024) / y.nt;
    const int per_cu = (int)max((size_t)1, min((size_t)by_regs, kLdsBytes / y.lds_bytes));
    const bool listed = a.picked || (a.dense_items && a.mode != 3);
    const int64_t most = a.picked || !listed ? block_items(a.xcds, a.B, a.nq) / a.xcds : (int64_t)a.dense_cap;
    int64_t per_xcd = max((int64_t)1, min((int64_t)32 * per_cu * 2, most));
    DenseArgs args{a, y, 1, (int)per_xcd, most};
    if (!listed && y.ipt <= 15 && most >= (int64_t)32 * per_cu * 8) {
        const int64_t fit = 0xffffffffLL / ((int64_t)a.xcds * y.nt);
        args.first = (int)((most + fit - 1) / fit);
        args.len = args.first;
        args.step = 1;
        per_xcd = (most + args.first - 1) / args.first;
    }
    // A round's items: as many workgroups as the device holds, each asks for the next one.  500 queries, 100 partitions of 2000 rows of 960, all
    // of them in the first round: 10.3 ms by strides, 7.7 so; rows that bounds tell apart, 1.28 and 1.17.  To ask takes the time in which no wavefront
    // of the workgroup works, so of as many items as in order the expected number have a workgroup each before these (10000 queries,
    // 400 partitions of 25000 unit vectors of 96, a million items: 410 ms all asking, 387 so; 512 queries, 49000 items:
    // 15.3 and 15.0; a million mixture rows in 100 partitions, 1000 queries, 10000 items: 2.40, 2.38).
    // None asks where each workgroup has had its item, and the dies' words lie on lines of their own: 4000 workgroups at one line took
    // 40 us (1385 queries, 83 partitions of 72 rows: 300 us, 256 so).
    if (a.picked) {
        const int64_t resident = min((int64_t)32 * per_cu, most);
        const int64_t fit = 0xffffffffLL / ((int64_t)a.xcds * y.nt), expect = min(min(fit, most), a.picked_expect / a.xcds);
        per_xcd = y.ipt <= 15 && expect >= resident * 8 ? expect : resident;
        args.step = (int)(per_xcd - resident);
    }
    const unsigned grid = (unsigned)(per_xcd * a.xcds);
    if (y.by_windows) ++*a.window_launches;
#define DCIH_DENSE(NT, IPT, WAVES) \
    rc = y.by_windows && IPT <= 9 ? launch_dense<NT, IPT, WAVES, IPT <= 9 ? kWindows : kPicked>(args, grid, s) \
         : (a.picked ? launch_dense<NT, IPT, WAVES, kPicked>(args, grid, s) : launch_dense<NT, IPT, WAVES, kWhole>(args, grid, s))
    int rc;
    if (y.nt == 64) {
        if (y.ipt == 5) DCIH_DENSE(64, 5, 4); else DCIH_DENSE(64, 9, 4);
    } else if (y.nt == 256) {
        if (y.ipt == 5) DCIH_DENSE(256, 5, 4); else if (y.ipt == 9) DCIH_DENSE(256, 9, 4); else DCIH_DENSE(256, 33, 2);
    } else if (y.ipt <= 9) {
        if (y.ipt == 5) DCIH_DENSE(512, 5, 4); else DCIH_DENSE(512, 9, 4);
    } else if (y.ipt <= 15) {
        if (y.ipt == 13) DCIH_DENSE(512, 13, 4); else DCIH_DENSE(512, 15, 4);
    } else {
        DCIH_DENSE(512, 21, 2);
    }
#undef DCIH_DENSE
    return rc;
}

}  // namespace dcih
