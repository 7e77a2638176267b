// Full ranking: num_neighbours beyond what the traversal's top-k tables hold.
//
// dci_query (src/dci_cuda_kernel.cu:777-875) with num_neighbours up to the
// number of indexed points, which is what dciknn_cuda/core.py:84-85 asks for
// when the caller leaves num_neighbours at -1.  The stop rule (:598-607) needs
// c0 >= num_neighbours, and c0 counts promotions inside ONE partition, so with
// num_neighbours above the points per partition no partition ever stops early:
// every window of every simple index is consumed (the loop bound of :458 is
// never below the number of windows), every point is promoted, and the result
// is the num_neighbours closest of ALL points by (distance, id).  That closed
// form is computed here directly: exact distances of every (query, point) pair,
// one sort per query with the build's segmented sort, first num_neighbours
// columns copied out.  The traversal counters have closed forms too: every
// index entry is visited once, every point is a candidate, and the outer steps
// follow from the window counts on either side of the positioning search.
#include <type_traits>

#include "bucket_core.h"
#include "common.h"
#include "kernels.h"
#include "radix_core.h"
#include "traverse_common.h"

namespace dcih {

namespace {

typedef const __attribute__((address_space(4))) float cfloat;

constexpr int kExRows = 64;       // rows per workgroup, one wavefront
constexpr int kExCols = 32;       // columns staged per LDS tile
constexpr int kExPitch = 36;      // row pitch in LDS: conflict-free 16-byte reads
typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_any __attribute__((aligned(4)));      // a 16-byte read that may start at any float
typedef const __attribute__((address_space(4))) v4f_any cv4f;

// out[q][row] = || data[row] - query[q] ||, the squares summed one after the
// other in index order like compute_dist_device (src/dci_cuda_kernel.cu:36-44);
// multiply and add rounded separately, as a CPU build of that loop does.
// A wavefront takes 64 rows and QN queries: the rows go through LDS 32 columns at
// a time (eight lanes read a row's 128 bytes; a lane reading its row straight from
// memory asks for 64 lines per instruction), the next columns' reads in flight
// meanwhile, and every lane keeps its row's QN sums; the queries' values are the
// same for all lanes and come through the scalar cache.  Bound by vector issue, three
// instructions per element and query, once enough wavefronts run, hence fewer queries per
// wavefront where rows and queries are few.  (500 queries, 3000 rows of 100:
// 86 us before, 22 now; 4000 queries, 9582 rows: 440 us with the queries read where they are used, 364 ahead.)
template <int QN>
__device__ __forceinline__ void exact_tile(float* tile, const float* __restrict__ data, int64_t N, int dim, int64_t row0, int lane,
                                           const cfloat* (&qv)[QN], float (&acc)[QN]) {
#pragma clang fp contract(off)     // no fused multiply-add: product and sum are rounded separately
    constexpr int kTpr = kExCols / 4, kLoads = kTpr;      // lanes per row; 16-byte reads per lane and chunk
    const int kq = (lane % kTpr) * 4, r_in = lane / kTpr;
    v4f pre[kLoads];
    auto prefetch = [&](int k0) {      // (past the last row: that row again; past the row's end: its last 16 bytes)
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            const float* x = data + min(row0 + j * kTpr + r_in, N - 1) * dim;
            if (dim >= 4) pre[j] = *reinterpret_cast<const v4f_any*>(x + min(k0 + kq, dim - 4));
            else pre[j] = v4f{x[0], x[min(1, dim - 1)], x[min(2, dim - 1)], 0.0f};
        }
    };
    prefetch(0);
#pragma unroll 1
    for (int k0 = 0; k0 < dim; k0 += kExCols) {
        const int kc = min(kExCols, dim - k0);
        __syncthreads();
        if (k0 + kq + 4 <= dim || dim < 4) {
#pragma unroll
            for (int j = 0; j < kLoads; j++) *reinterpret_cast<v4f*>(&tile[(j * kTpr + r_in) * kExPitch + kq]) = pre[j];
        } else {      // the row's last quad, or a repetition of it: to the columns it holds
            const int col = dim - 4 - k0;
#pragma unroll
            for (int j = 0; j < kLoads; j++) {
                float* t = &tile[(j * kTpr + r_in) * kExPitch + col];
                if (col >= 0) t[0] = pre[j].x;
                if (col >= -1) t[1] = pre[j].y;
                if (col >= -2) t[2] = pre[j].z;
                t[3] = pre[j].w;
            }
        }
        if (k0 + kExCols < dim) prefetch(k0 + kExCols);
        __syncthreads();
        const float* x = &tile[lane * kExPitch];
        int kk = 0;
        // The queries' next four elements are read while the present four are worked on.  (Scalar reads
        // return in any order, so a wait is for all of them: the present ones are made to arrive first.)
        auto fetch = [&](int at, v4f (&q)[QN]) __attribute__((always_inline)) {
            const int c = min(at, max(dim - 4, 0));
#pragma unroll
            for (int j = 0; j < QN; j++) q[j] = *(cv4f*)(qv[j] + c);
        };
        auto arrived = [&](v4f (&q)[QN]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < QN; j++) asm volatile("" :: "s"(q[j]));
            __builtin_amdgcn_sched_barrier(0);
        };
        auto add = [&](const v4f& v, const v4f (&q)[QN]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < QN; j++) {
                float d = v.x - q[j].x; acc[j] = acc[j] + d * d;
                d = v.y - q[j].y; acc[j] = acc[j] + d * d;
                d = v.z - q[j].z; acc[j] = acc[j] + d * d;
                d = v.w - q[j].w; acc[j] = acc[j] + d * d;
            }
        };
        if (kc >= 4) {
            v4f qa[QN], qb[QN];
            fetch(k0, qa);
            v4f va = *reinterpret_cast<const v4f*>(x), vb;
#pragma unroll 1
            for (; kk + 8 <= kc; kk += 8) {
                arrived(qa);
                fetch(k0 + kk + 4, qb);
                vb = *reinterpret_cast<const v4f*>(x + kk + 4);
                __builtin_amdgcn_sched_barrier(0);
                add(va, qa);
                arrived(qb);
                fetch(k0 + kk + 8, qa);
                va = *reinterpret_cast<const v4f*>(x + min(kk + 8, kExCols - 4));
                __builtin_amdgcn_sched_barrier(0);
                add(vb, qb);
            }
            if (kk + 4 <= kc) { add(va, qa); kk += 4; }
        }
#pragma unroll 1
        for (; kk < kc; kk++) {
            const float v = x[kk];
#pragma unroll
            for (int j = 0; j < QN; j++) {
                const float d = v - qv[j][k0 + kk];
                acc[j] = acc[j] + d * d;
            }
        }
    }
}
template <int QN>
__global__ __launch_bounds__(kExRows) void exact_dists_kernel(
    const float* __restrict__ data, int64_t N, int dim, const float* __restrict__ query, int nq,
    float* __restrict__ out) {
    __shared__ float tile[kExRows * kExPitch];
    const int lane = threadIdx.x;
    const int64_t row0 = (int64_t)blockIdx.x * kExRows;
    const int q0 = blockIdx.y * QN;
    float acc[QN];
    const cfloat* qv[QN];             // wave-uniform: read through the scalar cache
#pragma unroll
    for (int j = 0; j < QN; j++) {
        acc[j] = 0.0f;
        qv[j] = (const cfloat*)(uintptr_t)(query + (int64_t)min(q0 + j, nq - 1) * dim);
    }
    exact_tile<QN>(tile, data, N, dim, row0, lane, qv, acc);
    const int64_t row = row0 + lane;
    if (row >= N) return;
#pragma unroll
    for (int j = 0; j < QN; j++)
        // (the square root taken in double and rounded once more is the correctly rounded
        //  single-precision root: 53 bits are more than twice 24 plus two)
        if (q0 + j < nq) out[(int64_t)(q0 + j) * N + row] = (float)sqrt((double)acc[j]);
}

// The kc smallest (distance, id) pairs of one piece of one query's row of distances, ascending,
// as packed words to part[query][piece][kc]; a piece has at most kSelLen entries and kc <= 256.
// The row is read once, into registers; the kc-th smallest of the threads' own smallest entries
// bounds the kc-th best from above, and only what lies below that bound (kc entries and few
// more) is sorted.  (Sorting the whole row of 3000: 32 us for 500 queries, and 5 us to cut it.)
constexpr int kSelThreads = 256, kSelItems = 16, kSelLen = kSelThreads * kSelItems, kSelCap = 2048;
constexpr int kSelMaxK = kSelThreads;
__device__ __forceinline__ void select_piece(unsigned long long* buf, uint32_t& s_count, const float* row, int n, int kc) {
    const int tid = threadIdx.x;
    uint32_t v[kSelItems];       // (distances are not negative: their bits order as they do)
    uint32_t least = 0xffffffffu;
    int at = 0;
#pragma unroll
    for (int r = 0; r < kSelItems; r++) {
        const int j = r * kSelThreads + tid;
        v[r] = j < n ? __builtin_bit_cast(uint32_t, row[j]) : 0xffffffffu;
    }
#pragma unroll
    for (int r = 0; r < kSelItems; r++)
        if (v[r] < least) { least = v[r]; at = r * kSelThreads + tid; }
    buf[tid] = ((unsigned long long)least << 32) | (uint32_t)at;
    if (tid == 0) s_count = 0;
    bitonic_sort_u64_by256(buf, kSelThreads);
    const unsigned long long bound = buf[kc - 1];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSelItems; r++) {
        const int j = r * kSelThreads + tid;
        const unsigned long long e = ((unsigned long long)v[r] << 32) | (uint32_t)j;
        if (j < n && e <= bound) {
            const uint32_t slot = atomicAdd(&s_count, 1u);
            if (slot < (uint32_t)kSelCap) buf[slot] = e;
        }
    }
    __syncthreads();
    int count = (int)s_count;
    if (count > kSelCap) {       // (most of the piece lies below the bound, kc near the number of threads: in two goes)
        __syncthreads();
        for (int half = 0; half < 2; half++) {
            // the best of the first half stay at the front, the other half is sorted in behind them
            const int keep = half ? kSelMaxK : 0;
#pragma unroll
            for (int r = 0; r < kSelItems / 2; r++) {
                const int j = (half * (kSelItems / 2) + r) * kSelThreads + tid;
                const uint32_t bits = half ? v[kSelItems / 2 + r] : v[r];
                const int slot = keep + r * kSelThreads + tid;
                if (slot < kSelCap) buf[slot] = j < n ? ((unsigned long long)bits << 32) | (uint32_t)j : ~0ull;
            }
            bitonic_sort_u64_by256(buf, kSelCap);
            __syncthreads();
            if (half) {     // (the entries the second go had no room for)
                const int j = (kSelItems - 1) * kSelThreads + tid;
                buf[keep + tid] = j < n ? ((unsigned long long)v[kSelItems - 1] << 32) | (uint32_t)j : ~0ull;
                bitonic_sort_u64_by256(buf, 2 * kSelMaxK);
            }
        }
    } else {
        int np = kWave;
        while (np < count || np < kc) np <<= 1;
        for (int j = count + tid; j < np; j += kSelThreads) buf[j] = ~0ull;
        if (np >= kSelThreads) bitonic_sort_u64_by256(buf, np); else bitonic_sort_u64(buf, np);
    }
}
__global__ __launch_bounds__(kSelThreads) void select_rows_kernel(const float* __restrict__ dists, int64_t N, int len,
                                                                  int kc, unsigned long long* __restrict__ part,
                                                                  int32_t* __restrict__ out_ids, float* __restrict__ out_dists,
                                                                  int float_ids) {
    __shared__ unsigned long long buf[kSelCap];
    __shared__ uint32_t s_count;
    const int tid = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * len;
    const int n = (int)min((int64_t)len, N - first);
    unsigned long long* out = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kc;
    select_piece(buf, s_count, dists + (int64_t)blockIdx.y * N + first, n, kc);
    for (int j = tid; j < kc; j += kSelThreads) {
        const unsigned long long e = buf[j];
        if (out_ids) {               // (the only piece of the row, and kc = k: these are the results)
            const int64_t at_out = (int64_t)blockIdx.y * kc + j;
            const int32_t id = (int32_t)(uint32_t)e;
            out_ids[at_out] = float_ids ? __builtin_bit_cast(int32_t, (float)id) : id;
            out_dists[at_out] = __builtin_bit_cast(float, (uint32_t)(e >> 32));
        } else {
            out[j] = e == ~0ull ? e : e + (unsigned long long)first;      // (ids of the whole row; no carry into the distance)
        }
    }
}


// The same for the queries of a list whose length is known on the device only (nearest.hip's, of bounds that say too little): left[0] of them, their
// numbers, and a counter for every eight, zero.  A workgroup takes a piece of the rows and eight queries, forms their distances into `rows`, selects the
// piece's best, and whoever finishes a query's last piece merges them.  (200 queries, 200000 rows of 64, one query not finite: 164 us in all, 4930 where the
// query's workgroup went through all rows by itself; all of them: 1144, 4820; distances of all from the beginning: 300.)
constexpr int kListed = 8, kListedLen = 2048;
__host__ __device__ inline int listed_pieces(int64_t N) { return (int)((N + kListedLen - 1) / kListedLen); }
__global__ __launch_bounds__(kSelThreads) void listed_rows_kernel(const float* __restrict__ data, int64_t N, int dim, const float* __restrict__ query, int nq,
                                                                  int k, int float_ids, float* rows, unsigned long long* part,
                                                                  uint32_t* left, int32_t* __restrict__ out_ids, float* __restrict__ out_dists) {
    __shared__ __align__(16) float tile[kSelThreads / kWave][kExRows * kExPitch];
    __shared__ unsigned long long buf[kSelCap];
    __shared__ uint32_t s_count, s_last;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t count = left[0];
    const int pieces = listed_pieces(N);
    const int64_t tasks = (int64_t)((count + kListed - 1) / kListed) * pieces;
    for (int64_t t = blockIdx.x; t < tasks; t += gridDim.x) {
        const int group = (int)(t / pieces), piece = (int)(t % pieces), here = min(kListed, (int)count - group * kListed);
        const int64_t first = (int64_t)piece * kListedLen;
        const int n = (int)min((int64_t)kListedLen, N - first);
        auto distances = [&](auto qn) __attribute__((always_inline)) {
            constexpr int QN = decltype(qn)::value;
            int q[QN];
            const cfloat* qv[QN];
#pragma unroll
            for (int j = 0; j < QN; j++) {
                q[j] = __builtin_amdgcn_readfirstlane((int)left[1 + group * kListed + min(j, here - 1)]);
                qv[j] = (const cfloat*)(uintptr_t)(query + (int64_t)q[j] * dim);
            }
            for (int i = 0; i < n; i += kSelThreads) {      // (the same number of times for every wavefront)
                float acc[QN] = {};
                const int64_t row0 = first + i + wave * kExRows, row = row0 + lane;
                exact_tile<QN>(tile[wave], data, N, dim, row0, lane, qv, acc);
#pragma unroll
                for (int j = 0; j < QN; j++)
                    if (j < here && row < first + n) rows[(int64_t)q[j] * N + row] = (float)sqrt((double)acc[j]);
            }
        };
        if (here <= 2) distances(std::integral_constant<int, 2>()); else distances(std::integral_constant<int, kListed>());
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (read again by this workgroup only)
        __syncthreads();
        for (int j = 0; j < here; j++) {
            const int qj = (int)left[1 + group * kListed + j];
            select_piece(buf, s_count, rows + (int64_t)qj * N + first, n, k);
            unsigned long long* out = part + ((int64_t)(group * kListed + j) * pieces + piece) * k;
            for (int e = tid; e < k; e += kSelThreads)
                __hip_atomic_store(&out[e], buf[e] == ~0ull ? buf[e] : buf[e] + (unsigned long long)first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
        }
        // (The pieces of a query are of several dies.  Their entries are written and read past the dies' own caches and have arrived before they are
        // counted; a fence would write back all of a die's cache, distances and all.)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) s_last = atomicAdd(&left[1 + nq + group], 1u) == (uint32_t)pieces - 1 ? 1u : 0u;
        __syncthreads();
        if (s_last) {
            for (int j = 0; j < here; j++) {
                const int64_t qj = left[1 + group * kListed + j];
                const unsigned long long* from = part + (int64_t)(group * kListed + j) * pieces * k;
                keep_smallest(buf, s_count, (int64_t)pieces * k, k, [&](int64_t at, int m) {
                    if (tid < m) buf[kKeepAt + tid] = __hip_atomic_load(&from[at + tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                });
                for (int e = tid; e < k; e += kSelThreads) {
                    const int32_t id = (int32_t)(uint32_t)buf[e];
                    out_ids[qj * k + e] = float_ids ? __builtin_bit_cast(int32_t, (float)id) : id;
                    out_dists[qj * k + e] = __builtin_bit_cast(float, (uint32_t)(buf[e] >> 32));
                }
            }
        }
        __syncthreads();      // (the next task's tables)
    }
}

// One row of distances per workgroup, ranked in LDS by buckets (bucket_core.h; by radix passes where the distances
// cluster) and written out in order, the first k of them.  Such calls are few rows, so what counts is one
// row's time: sixteen wavefronts on it, the whole LDS for it, no kernel to cut and convert the result after
// it.  (20 rows of 9582: 22 us; the segmented sort and that kernel 39 + 4.)  Beyond 16 items per thread 128
// registers do not hold them and eight wavefronts take as long as the segmented sort (20000: 63 and 62 us).
constexpr int rank_bits(int items) { return items <= 2048 ? 11 : (items <= 4096 ? 12 : (items <= 8192 ? 13 : 14)); }
constexpr int rank_counter_words(int nt, int ipt) {
    return (1 << rank_bits(nt * ipt)) / 2 + 4 > 8 * nt ? (1 << rank_bits(nt * ipt)) / 2 + 4 : 8 * nt;
}
constexpr size_t rank_lds(int nt, int ipt) {
    return (size_t)(64 + nt * ipt + 4 + rank_counter_words(nt, ipt)) * 4 + (size_t)nt * 8;
}
template <int NT, int IPT>
__global__ __launch_bounds__(NT, NT / 256) void rank_row_kernel(const float* __restrict__ dists, int n, int k, int float_ids,
                                                                   int32_t* __restrict__ out_ids, float* __restrict__ out_vals) {
    extern __shared__ __align__(16) unsigned char rank_smem[];
    uint32_t* misc = reinterpret_cast<uint32_t*>(rank_smem);             // 32 words for the ranking, then the extremes
    unsigned long long* work = reinterpret_cast<unsigned long long*>(misc + 64);
    uint32_t* list = reinterpret_cast<uint32_t*>(work + NT);
    uint32_t* cnt = list + NT * IPT + 4;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const float* row = dists + (int64_t)blockIdx.x * n;
    out_ids += (int64_t)blockIdx.x * k;
    out_vals += (int64_t)blockIdx.x * k;
    if (tid == 0) { misc[32] = 0xffffffffu; misc[33] = 0; misc[34] = 0; misc[35] = 0xffffffffu; }
    __syncthreads();
    uint32_t key[IPT], rp[IPT];
    {
        uint32_t least = 0xffffffffu, most = 0;
#pragma unroll
        for (int r = 0; r < IPT; r++) {
            const int j = r * NT + tid;
            key[r] = __builtin_bit_cast(uint32_t, row[min(j, n - 1)]);
            rp[r] = (uint32_t)j;
            least = min(least, key[r]);
            most = max(most, key[r]);
        }
        least = wave_min_u32(least);
        most = ~wave_min_u32(~most);
        if (lane == 0) { atomicMin(&misc[32], least); atomicMax(&misc[33], most); }
    }
    __syncthreads();
    const uint32_t lo_bits = misc[32], hi_bits = misc[33];
    const float lo = __builtin_bit_cast(float, lo_bits), width = __builtin_bit_cast(float, hi_bits) - lo;
    const float scale = 4294966016.0f / width;
    int fix_rank = -1;
    uint32_t fix_item = 0;
    bool ranked = false;
    if (hi_bits < kInfBits && scale < 4e38f) {
        auto before = [&](int x, int z) __attribute__((always_inline)) {
            const uint32_t bx = __builtin_bit_cast(uint32_t, row[x]), bz = __builtin_bit_cast(uint32_t, row[z]);
            return bx != bz ? bx < bz : x < z;
        };
#pragma unroll
        for (int r = 0; r < IPT; r++) key[r] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, key[r]) - lo);
        ranked = lds_bucket_ranks<NT, IPT, rank_bits(NT * IPT), true>(key, rp, n, scale, list, cnt, misc, work, NT, tid, fix_rank,
                                                                 fix_item, before);
    }
    auto store = [&](int at, uint32_t bits, uint32_t item) {
        if (at >= k) return;
        out_vals[at] = __builtin_bit_cast(float, bits);
        out_ids[at] = float_ids ? __builtin_bit_cast(int32_t, (float)(int)item) : (int)item;
    };
    __syncthreads();
    if (ranked) {
        // through LDS, so that the results leave in order: the row's numbers first, from which the values follow
        uint16_t* order = reinterpret_cast<uint16_t*>(list);
        int own = n > tid ? (n - tid + NT - 1) / NT : 0;
        asm volatile("" : "+v"(own));
#pragma unroll
        for (int r = 0; r < IPT; r++)
            if (r < own) order[rp[r] >> 16] = (uint16_t)(r * NT + tid);
        __syncthreads();
        if (fix_rank >= 0) order[fix_rank] = (uint16_t)fix_item;
        __syncthreads();
        const int end = min(n, k);
        for (int j = tid; j < end; j += NT) {
            const uint32_t item = order[j];
            store(j, __builtin_bit_cast(uint32_t, row[item]), item);
        }
        return;
    }
    uint32_t vor = 0, vand = 0xffffffffu;
#pragma unroll
    for (int r = 0; r < IPT; r++) {
        const int j = tid * IPT + r;
        key[r] = j < n ? __builtin_bit_cast(uint32_t, row[j]) : 0xffffffffu;      // (pads stay behind everything: the passes are stable)
        rp[r] = (uint32_t)j;
        vor |= j < n ? key[r] : 0u;
        vand &= j < n ? key[r] : 0xffffffffu;
    }
    for (int o = 32; o > 0; o >>= 1) {
        vor |= (uint32_t)__shfl_xor((int)vor, o, kWave);
        vand &= (uint32_t)__shfl_xor((int)vand, o, kWave);
    }
    if (lane == 0) { atomicOr(&misc[34], vor); atomicAnd(&misc[35], vand); }
    __syncthreads();
    lds_radix_passes<NT, IPT>(key, rp, list, cnt, misc, misc[34] ^ misc[35]);
#pragma unroll
    for (int r = 0; r < IPT; r++)
        if (tid * IPT + r < n) store(tid * IPT + r, key[r], rp[r] & 0xffffu);
}
// Rows fewer than CUs, of 8192 to 32768 items: `parts` workgroups to a row, each of which finds the part of the order that is its own,
// lists that part's items in LDS and ranks them there as above.  The parts are cut at bins of an even division of the row's range:
// every workgroup counts all of the row, 4096 bins, and cuts where the bins pass p / parts of it.  Where a part does not fit
// (distances that cluster) or a distance is not finite, its first and last item are found by their digits instead, eight bits of
// (distance, number) at a time.  Bound by vector issue and LDS operations, of the passes over the row and of the ranking.
// (Ranks of 64 rows of 20000: 61 us by the segmented sort, 30 in four parts each; read again by each of the four passes: 34.  16 rows of
// 16000: 30 -> 16 us.  Whole-number rows, whose distances are often equal, 64 of 20480: 44.  Few different distances, 49 of 40 rows of 20480: 72 -> 96.)
constexpr int kRankMaxN = 1024 * 16;
constexpr int kPartThreads = 1024, kPartBins = 4096, kPartMaxN = 32768;
constexpr int part_work(int ipt) { return ipt <= 6 ? 4096 : 2048; }      // (what LDS leaves; a power of two)
constexpr size_t part_lds(int ipt) {
    const size_t items = (size_t)kPartThreads * ipt;
    return 160 * 4 + (size_t)part_work(ipt) * 8 + (2 * items + 4 + rank_counter_words(kPartThreads, ipt)) * 4 + items * 2;
}
template <int IPT, int ROW>      // ROW: items of the whole row per thread, in registers
__global__ __launch_bounds__(kPartThreads, 4) void rank_part_kernel(const float* __restrict__ dists, int n, int k, int float_ids,
                                                                 int32_t* __restrict__ out_ids, float* __restrict__ out_vals) {
    constexpr int NT = kPartThreads, kItems = NT * IPT, kWaves = NT / kWave;
    static_assert(kItems >= kPartBins, "the bins are where the items are listed later");
    extern __shared__ __align__(16) unsigned char rank_smem[];
    uint32_t* misc = reinterpret_cast<uint32_t*>(rank_smem);             // 32 words for the ranking
    uint32_t* extremes = misc + 32;                                      // of the row, of the part; digits that differ
    uint32_t* wave_sum = misc + 40;                                      // [kWaves]
    uint32_t* cut = misc + 64;                                           // [parts + 1] bins, parts at most 32,
    uint32_t* cut_at = misc + 112;                                       // and the items before them
    unsigned long long* work = reinterpret_cast<unsigned long long*>(misc + 160);
    uint32_t* list = reinterpret_cast<uint32_t*>(work + part_work(IPT));      // [kItems + 4]; the bins first
    uint32_t* cnt = list + kItems + 4;                                   // [rank_counter_words]
    uint32_t* bits = cnt + rank_counter_words(NT, IPT);                                       // [kItems]: the part's distances, in order of their numbers
    uint16_t* number = reinterpret_cast<uint16_t*>(bits + kItems);       // [kItems]
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int part = blockIdx.x, parts = gridDim.x;
    const float* row = dists + (int64_t)blockIdx.y * n;
    out_ids += (int64_t)blockIdx.y * k;
    out_vals += (int64_t)blockIdx.y * k;
    const int share = (n + kWaves - 1) / kWaves, from = min(n, wave * share), to = min(n, from + share);      // this wavefront's items
    uint32_t w[ROW];
#pragma unroll
    for (int r = 0; r < ROW; r++) w[r] = __builtin_bit_cast(uint32_t, row[min(from + r * kWave + lane, n - 1)]);
    auto each = [&](auto use) __attribute__((always_inline)) {           // use(number, bits, whether there is one): all lanes, in order
#pragma unroll
        for (int r = 0; r < ROW; r++) {
            if (from + r * kWave >= to) break;
            use(from + r * kWave + lane, w[r], from + r * kWave + lane < to);
        }
    };
    // One more of `what`; the first lane's by a single addition for all lanes that have it (rows of few distinct distances: one word's additions queue up).
    auto count_in = [&](uint32_t what, bool in) __attribute__((always_inline)) {
        const unsigned long long have = __ballot(in);
        if (have == 0) return;
        const int lead = (int)__builtin_ctzll(have);
        const uint32_t lead_what = (uint32_t)__builtin_amdgcn_readlane((int)what, lead);
        const unsigned long long same = __ballot(in && what == lead_what);
        if (lane == lead) atomicAdd(&list[what], (uint32_t)__popcll(same));
        if (in && what != lead_what) atomicAdd(&list[what], 1u);
    };
    // Exclusive sum over the workgroup's threads.
    auto scan = [&](uint32_t sum) {
        uint32_t incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = (uint32_t)__shfl_up((int)incl, o, 64);
            if (lane >= o) incl += t;
        }
        __syncthreads();
        if (lane == 63) wave_sum[wave] = incl;
        __syncthreads();
        for (int w = 0; w < wave; w++) incl += wave_sum[w];
        return incl - sum;
    };
    if (tid < 8) extremes[tid] = (tid & 1) ? 0u : 0xffffffffu;
    for (int j = tid; j < kPartBins; j += NT) list[j] = 0;
    __syncthreads();
    {
        uint32_t least = 0xffffffffu, most = 0;
        each([&](int, uint32_t b, bool) { least = min(least, b); most = max(most, b); });      // (the row's last item again does no harm)
        least = wave_min_u32(least);
        most = ~wave_min_u32(~most);
        if (lane == 0) { atomicMin(&extremes[0], least); atomicMax(&extremes[1], most); }
    }
    __syncthreads();
    const uint32_t hi_bits = extremes[1];
    const float lo = __builtin_bit_cast(float, extremes[0]), scale = 4294966016.0f / (__builtin_bit_cast(float, hi_bits) - lo);
    bool even = hi_bits < kInfBits && scale < 4e38f;                     // (the same for all of a row's workgroups)
    auto bin_of = [&](uint32_t b) { return (uint32_t)((__builtin_bit_cast(float, b) - lo) * scale) >> 20; };
    auto cut_of = [&](int p) { return (uint32_t)((int64_t)n * p / parts); };
    if (even) {
        // (where the wavefront's first items lie in one bin by the half dozen; else the test for each costs more than it saves: 64 normal rows of
        // 20000 44.1 us with it, 42.7 without, 20 of 32768 45, 40.7; half of a row at one distance takes 111, 244 where each item is added by itself)
        const uint32_t some = bin_of(w[0]);
        if (__popcll(__ballot(some == (uint32_t)__builtin_amdgcn_readfirstlane((int)some))) >= 6)
            each([&](int, uint32_t b, bool in) { count_in(bin_of(b), in); });
        else
            each([&](int, uint32_t b, bool in) { if (in) atomicAdd(&list[bin_of(b)], 1u); });
        __syncthreads();
        constexpr int kPer = kPartBins / NT;
        uint32_t v[kPer], sum = 0;
#pragma unroll
        for (int i = 0; i < kPer; i++) { v[i] = list[tid * kPer + i]; sum += v[i]; }
        uint32_t run = scan(sum);
#pragma unroll
        for (int i = 0; i < kPer; i++) { list[tid * kPer + i] = run; run += v[i]; }
        __syncthreads();
        if (tid <= parts) {      // the first bin that begins at the part's share or behind it
            int a = 0, b = kPartBins;
            while (a < b) {
                const int mid = (a + b) >> 1;
                if (list[mid] < cut_of(tid)) a = mid + 1; else b = mid;
            }
            cut[tid] = (uint32_t)a;
            cut_at[tid] = a < kPartBins ? list[a] : (uint32_t)n;
        }
        __syncthreads();
        for (int p = 0; p < parts; p++) even = even && cut_at[p + 1] - cut_at[p] <= (uint32_t)kItems;
    }
    unsigned long long item0 = 0, item1 = ~0ull;                         // (distance, number): the part's first, and the first behind it
    // (by their bits as in rank_row_kernel, in rows too long for it by value as in the segmented sort: NaN of either sign)
    const uint32_t negative = n > kRankMaxN ? 0xffffffffu : 0u, positive = n > kRankMaxN ? 0x80000000u : 0u;
    auto order_of = [&](uint32_t b) { return b ^ (b >> 31 ? negative : positive); };
    auto item_of = [&](uint32_t b, int j) { return ((unsigned long long)order_of(b) << 16) | (uint32_t)j; };
    uint32_t first = cut_of(part);
    if (even) {
        first = cut_at[part];
    } else {
        uint32_t place[2] = {first, cut_of(part + 1)};      // the items with so many others before them, both at once
        unsigned long long found[2] = {0, 0};
        const bool wanted[2] = {place[0] != 0, place[1] != (uint32_t)n};
#pragma unroll 1
        for (int shift = 40; shift >= 0; shift -= 8) {
            __syncthreads();
            if (tid < 512) list[tid] = 0;
            __syncthreads();
            each([&](int j, uint32_t b, bool in) {
                const unsigned long long e = item_of(b, j);
#pragma unroll
                for (int end = 0; end < 2; end++)
                    if (wanted[end]) count_in(256u * end + ((uint32_t)(e >> shift) & 255u), in && (e >> shift >> 8) == found[end]);
            });
            __syncthreads();
#pragma unroll
            for (int end = 0; end < 2; end++) {
                if (!wanted[end]) continue;
                const uint32_t v = tid < 256 ? list[256 * end + tid] : 0, run = scan(v);
                if (run <= place[end] && place[end] < run + v) { extremes[6] = (uint32_t)tid; extremes[7] = place[end] - run; }      // (one thread)
                __syncthreads();
                found[end] = found[end] << 8 | extremes[6];
                place[end] = extremes[7];
                __syncthreads();
            }
        }
        if (wanted[0]) item0 = found[0];
        if (wanted[1]) item1 = found[1];
    }
    if (first >= (uint32_t)k) return;
    // The part's items, in order of their numbers.
    const uint32_t bin0 = even ? cut[part] : 0, bin1 = even ? cut[part + 1] : 0;
    auto mine = [&](int j, uint32_t b) {
        if (even) { const uint32_t bin = bin_of(b); return bin >= bin0 && bin < bin1; }
        const unsigned long long e = item_of(b, j);
        return e >= item0 && e < item1;
    };
    uint32_t have = 0;
    each([&](int j, uint32_t b, bool in) { have += in && mine(j, b) ? 1u : 0u; });
    uint32_t at = scan(have);      // (lane 0's is the wavefront's)
    at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    int count = 0;
    for (int w = 0; w < kWaves; w++) count += (int)wave_sum[w];
    {
        uint32_t least = 0xffffffffu, most = 0, all_or = 0, all_and = 0xffffffffu;
        each([&](int j, uint32_t b, bool in) {
            const bool take = in && mine(j, b);
            const unsigned long long m = __ballot(take);
            if (take) {
                const uint32_t to_at = at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                bits[to_at] = b;
                number[to_at] = (uint16_t)j;
                least = min(least, b); most = max(most, b);
                all_or |= order_of(b); all_and &= order_of(b);
            }
            at += (uint32_t)__popcll(m);
        });
        least = wave_min_u32(least);
        most = ~wave_min_u32(~most);
        for (int o = 32; o > 0; o >>= 1) {
            all_or |= (uint32_t)__shfl_xor((int)all_or, o, kWave);
            all_and &= (uint32_t)__shfl_xor((int)all_and, o, kWave);
        }
        if (lane == 0) { atomicMin(&extremes[2], least); atomicMax(&extremes[3], most); atomicAnd(&extremes[4], all_and); atomicOr(&extremes[5], all_or); }
    }
    __syncthreads();
    if (count == 0) return;
    uint32_t key[IPT], rp[IPT];
    int fix_rank = -1;
    uint32_t fix_item = 0;
    bool ranked = false;
    int sorted = 0;
    const float part_lo = __builtin_bit_cast(float, extremes[2]), part_scale = 4294966016.0f / (__builtin_bit_cast(float, extremes[3]) - part_lo);
    if (extremes[3] < kInfBits && part_scale < 4e38f) {
#pragma unroll
        for (int r = 0; r < IPT; r++) {
            const int j = r * NT + tid;
            key[r] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, bits[min(j, count - 1)]) - part_lo);
            rp[r] = (uint32_t)j;
        }
        auto before = [&](int x, int z) __attribute__((always_inline)) { return bits[x] != bits[z] ? bits[x] < bits[z] : x < z; };
        ranked = lds_bucket_ranks<NT, IPT, rank_bits(kItems), true, true>(key, rp, count, part_scale, list, cnt, misc, work, part_work(IPT), tid, fix_rank,
                                                                          fix_item, before, [&](int x) { return bits[x]; }, &sorted);
    }
    auto store = [&](uint32_t place, uint32_t b, uint32_t item) {
        if (place >= (uint32_t)k) return;
        out_vals[place] = __builtin_bit_cast(float, b);
        out_ids[place] = float_ids ? __builtin_bit_cast(int32_t, (float)(int)item) : (int)item;
    };
    __syncthreads();
    if (ranked) {      // through LDS, so that the results leave in order
        uint16_t* order = reinterpret_cast<uint16_t*>(list);
        int own = count > tid ? (count - tid + NT - 1) / NT : 0;
        asm volatile("" : "+v"(own));
#pragma unroll
        for (int r = 0; r < IPT; r++)
            if (r < own) order[rp[r] >> 16] = (uint16_t)(r * NT + tid);
        __syncthreads();
        if (fix_rank >= 0) order[fix_rank] = (uint16_t)fix_item;
        for (int i = tid; i < sorted; i += NT) order[sorted_place(work, i)] = (uint16_t)(work[i] & ((1u << kSortedNumberBits) - 1u));
        __syncthreads();
        for (int j = tid; j < count; j += NT) store(first + (uint32_t)j, bits[order[j]], number[order[j]]);
        return;
    }
#pragma unroll
    for (int r = 0; r < IPT; r++) {
        const int j = tid * IPT + r;
        key[r] = j < count ? order_of(bits[j]) : 0xffffffffu;      // (pads stay behind everything: the passes are stable)
        rp[r] = (uint32_t)j;
    }
    lds_radix_passes<NT, IPT>(key, rp, list, cnt, misc, extremes[4] ^ extremes[5]);
#pragma unroll
    for (int r = 0; r < IPT; r++)
        if (tid * IPT + r < count) store(first + (uint32_t)(tid * IPT + r), bits[rp[r] & 0xffffu], number[rp[r] & 0xffffu]);
}
static bool rank_fits(int64_t n) { return n <= kRankMaxN; }
static int rank_rows_in_lds(const float* d_dist, int rows, int n, int k, int float_ids, int32_t* out_ids, float* out_vals,
                            hipStream_t s) {
#define DCIH_RANK(NT, IPT)                                                                              \
    do {                                                                                            \
        static DeviceOnce once;                                                                     \
        const int rc_attr = once.run([]() -> int {                                                  \
            DCIH_HIP(hipFuncSetAttribute((const void*)rank_row_kernel<NT, IPT>,                         \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));  \
            return 0;                                                                               \
        });                                                                                         \
        if (rc_attr) return rc_attr;                                                                \
        hipLaunchKernelGGL((rank_row_kernel<NT, IPT>), dim3((unsigned)rows), dim3(NT), rank_lds(NT, IPT), s, d_dist, n, k, \
                           float_ids, out_ids, out_vals);                                           \
    } while (0)
    if (n <= 1024 * 2) DCIH_RANK(1024, 2); else if (n <= 1024 * 4) DCIH_RANK(1024, 4); else if (n <= 1024 * 8) DCIH_RANK(1024, 8);
    else if (n <= 1024 * 12) DCIH_RANK(1024, 12); else DCIH_RANK(1024, 16);
#undef DCIH_RANK
    DCIH_HIP(hipGetLastError());
    return 0;
}

template <int IPT, int ROW>
static int launch_parts(const float* d_dist, int parts, int rows, int n, int k, int float_ids, int32_t* out_ids, float* out_vals, hipStream_t s) {
    static DeviceOnce once;
    const int rc = once.run([]() -> int {
        DCIH_HIP(hipFuncSetAttribute((const void*)rank_part_kernel<IPT, ROW>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        return 0;
    });
    if (rc) return rc;
    hipLaunchKernelGGL((rank_part_kernel<IPT, ROW>), dim3((unsigned)parts, (unsigned)rows), dim3(kPartThreads), part_lds(IPT), s, d_dist, n, k,
                       float_ids, out_ids, out_vals);
    DCIH_HIP(hipGetLastError());
    return 0;
}
// How many workgroups to a row: as many as leave one to a CU, if they hold it; 1: the kernels for whole rows.  (With rows on the device
// twice, 64 of 16000, 4 / 6 parts: 33 / 52 us.  Short rows lose by the passes over the whole, 64 of 4000: 16 us whole, 18 in parts; 9582:
// 28, 26.  More than 16 gain nothing.  Rows that do not stay in registers, past 32768, would be read again by every pass: 16 of 40000, whole 79 us, in parts 65;
// 32, 87 and 95; 16 whose distances are few different numbers, 78 and 164.)
constexpr int part_items(int64_t n, int parts) { return (int)(n / parts) * 21 / 20 + 64; }      // (bins are a few items)
static int rank_parts(int64_t n, int rows) {
    const int parts = (int)min((int64_t)16, (int64_t)256 / rows);
    return n >= 8192 && n <= kPartMaxN && parts > 1 && part_items(n, parts) <= kPartThreads * 10 ? parts : 1;
}
static int rank_rows_in_parts(const float* d_dist, int parts, int rows, int n, int k, int float_ids, int32_t* out_ids, float* out_vals, hipStream_t s) {
    const int most = part_items(n, parts);
    const auto launch = n <= 20480 ? (most <= 4096 ? launch_parts<4, 20> : most <= 6144 ? launch_parts<6, 20> : launch_parts<10, 20>)
                                   : (most <= 4096 ? launch_parts<4, 32> : most <= 6144 ? launch_parts<6, 32> : launch_parts<10, 32>);
    return launch(d_dist, parts, rows, n, k, float_ids, out_ids, out_vals, s);
}

// The first k columns of every sorted row.  Columns past the end of a row and, when
// asked, entries whose value is +inf (points that never became candidates) read as
// "no result": id -1, +inf.
__global__ __launch_bounds__(256) void take_columns_kernel(
    const float* __restrict__ skeys, const int32_t* __restrict__ sids, int64_t N, int k,
    int inf_is_empty, int float_ids, int32_t* __restrict__ out_ids, float* __restrict__ out_vals) {
    const int q = blockIdx.y;
    for (int j = blockIdx.x * 256 + threadIdx.x; j < k; j += gridDim.x * 256) {
        const float v = j < N ? skeys[(int64_t)q * N + j] : __builtin_inff();
        const bool empty = j >= N || (inf_is_empty && v == __builtin_inff());
        const int32_t id = empty ? -1 : sids[(int64_t)q * N + j];
        out_ids[(int64_t)q * k + j] = float_ids ? __builtin_bit_cast(int32_t, (float)id) : id;
        if (out_vals) out_vals[(int64_t)q * k + j] = v;
    }
}

__global__ void fill_f32_kernel(float* p, int64_t n, float v) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) p[e] = v;
}

// Counters of a traversal that runs every partition dry, one wavefront per
// (query, partition): the positioning search (:279-318) gives p, the largest
// position with key < projection; the left stream then has ceil((p+1)/T)
// windows and the right one ceil((n+T-1 - (p+1))/T) (starts below n+T-1, :250-273);
// a composite needs as many steps as its L indices have windows, and the loop
// runs one idle step more unless its bound n*L*T (:458) ends it first.
__global__ __launch_bounds__(kWave) void exhaustive_counters_kernel(QueryArgs a) {
    const int lane = threadIdx.x;
    const int b = (int)(blockIdx.x % a.B);
    const int qi = (int)(blockIdx.x / a.B);
    const int64_t off = (int64_t)b * a.ppb;
    const int n = (int)min(a.N - off, a.ppb);
    if (n <= 0) return;
    unsigned long long probes = 0, maxw = 0;
    for (int m = 0; m < a.M; m++) {
        unsigned long long w = 0;
        for (int h = lane; h < a.L; h += kWave) {
            const int i = m * a.L + h;
            const float* key = a.skeys + (int64_t)i * a.N + off;
            const float qp = a.qproj[(int64_t)i * a.nq + qi];
            int start_pos = -1, end_pos = n - 1;
            int cur_pos = (start_pos + end_pos + 2) / 2;
            while (start_pos < end_pos) {
                probes++;
                if (key[cur_pos] < qp) start_pos = cur_pos; else end_pos = cur_pos - 1;
                cur_pos = (start_pos + end_pos + 2) / 2;
            }
            const int64_t p1 = (int64_t)start_pos + 1;
            const int64_t rem = (int64_t)n + a.T - 1 - p1;
            w += (unsigned long long)((p1 + a.T - 1) / a.T) +
                 (unsigned long long)(rem > 0 ? (rem + a.T - 1) / a.T : 0);
        }
        for (int o = kWave / 2; o > 0; o >>= 1) w += __shfl_xor(w, o, kWave);
        maxw = max(maxw, w);
    }
    for (int o = kWave / 2; o > 0; o >>= 1) probes += __shfl_xor(probes, o, kWave);
    if (lane == 0) {
        const unsigned long long bound = (unsigned long long)n * a.L * a.T;
        atomicAdd(&a.counters[(int64_t)qi * 4 + 0], (unsigned long long)n * a.M * a.L);
        atomicAdd(&a.counters[(int64_t)qi * 4 + 1], (unsigned long long)n);
        atomicAdd(&a.counters[(int64_t)qi * 4 + 2], probes);
        atomicAdd(&a.counters[(int64_t)qi * 4 + 3], min(bound, maxw + 1));
    }
}

__global__ void zero_counters_kernel(unsigned long long* p, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) p[e] = 0;
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace

int exhaustive_chunk(int64_t N, int nq) {
    // 64 M (query, point) pairs at a time: 1.8 GB of scratch
    return (int)max((int64_t)1, min(min((int64_t)nq, (int64_t)32768), ((int64_t)1 << 26) / N));
}

// Few results: selected from the row of distances instead of sorting it.
static bool exhaustive_selects(int k) { return k <= kSelMaxK; }
struct ExSelect { int pieces, len, kc; };
static ExSelect exhaustive_select(int64_t N, int k) {
    ExSelect e;
    e.pieces = (int)((N + kSelLen - 1) / kSelLen);
    e.len = (int)((N + e.pieces - 1) / e.pieces);
    e.pieces = (int)((N + e.len - 1) / e.len);
    e.kc = min(k, e.len);
    return e;
}

// What is selected of every piece, or the smallest bounds of every 32 rows.
static size_t select_bytes(int64_t N, int chunk, int k) {
    const ExSelect e = exhaustive_select(N, k);
    return align256(max((size_t)chunk * max((size_t)e.pieces, k <= 128 ? (size_t)listed_pieces(N) : 0) * e.kc * sizeof(unsigned long long),
                        nearest_least_bytes(N, chunk)));
}

size_t exhaustive_ws_bytes(int64_t N, int chunk, int k) {
    const size_t cells = (size_t)chunk * (size_t)N;
    if (exhaustive_selects(k)) {
        return align256(cells * 4) + select_bytes(N, chunk, k) + align256(nearest_left_bytes(chunk));
    }
    return 3 * align256(cells * 4) + align256(segsort_tmp_bytes(chunk, N, 1));
}

float* rank_rows_input(void* ws) { return (float*)ws; }

int fill_rows(float* d_rows, int64_t cells, float value, hipStream_t s) {
    hipLaunchKernelGGL(fill_f32_kernel, dim3((unsigned)min((int64_t)8192, (cells + 255) / 256)), dim3(256), 0, s,
                       d_rows, cells, value);
    DCIH_HIP(hipGetLastError());
    return 0;
}

int rank_rows(void* ws, int chunk, int rows, int64_t N, int k, bool inf_is_empty, bool float_ids,
              int32_t* out_ids, float* out_vals, hipStream_t s) {
    const size_t cells = (size_t)chunk * (size_t)N;
    char* base = (char*)ws;
    float* d_in = (float*)base;
    float* d_sorted = (float*)(base + align256(cells * 4));
    int32_t* d_sids = (int32_t*)(base + 2 * align256(cells * 4));
    void* d_tmp = segsort_tmp_bytes(chunk, N, 1) ? (void*)(base + 3 * align256(cells * 4)) : nullptr;
    if (k == N && !inf_is_empty)       // the sorted rows are the results
        return segsort(d_in, N, rows, N, 1, out_vals, out_ids, nullptr, nullptr, d_tmp, s, float_ids, true);
    const int rc = segsort(d_in, N, rows, N, 1, d_sorted, d_sids, nullptr, nullptr, d_tmp, s, false, true);
    if (rc) return rc;
    hipLaunchKernelGGL(take_columns_kernel, dim3((unsigned)min(1024, (k + 255) / 256), (unsigned)rows),
                       dim3(256), 0, s, d_sorted, d_sids, N, k, inf_is_empty ? 1 : 0, float_ids ? 1 : 0,
                       out_ids, out_vals);
    DCIH_HIP(hipGetLastError());
    return 0;
}

template <int QN>
static void launch_dists(const QueryArgs& a, int q0, int nqc, float* d_dist, hipStream_t s) {
    hipLaunchKernelGGL(exact_dists_kernel<QN>,
                       dim3((unsigned)((a.N + kExRows - 1) / kExRows), (unsigned)((nqc + QN - 1) / QN)), dim3(kExRows),
                       0, s, a.data, a.N, a.dim, a.query + (int64_t)q0 * a.dim, nqc, d_dist);
}

int query_exhaustive(const QueryArgs& a, void* ws, int chunk, hipStream_t s) {
    if (a.nq <= 0) return 0;
    if ((a.N + kExRows - 1) / kExRows > 0x7fffffffLL || (int64_t)a.nq * a.B > 0x7fffffffLL)
        return fail(-4, "query: too many points for the full-ranking path");
    float* d_dist = rank_rows_input(ws);
    const int64_t row_groups = (a.N + kExRows - 1) / kExRows;
    const bool select = exhaustive_selects(a.k);
    const ExSelect sel = exhaustive_select(a.N, a.k);
    for (int q0 = 0; q0 < a.nq; q0 += chunk) {
        const int nqc = min(chunk, a.nq - q0);
        if (a.pick_rule != 1 && nearest_supported(a.N, a.dim, a.k) && (a.pick_rule == 2 || nearest_pays(a.N, a.dim, a.k, nqc))) {
            char* rest = (char*)ws + align256((size_t)chunk * (size_t)a.N * 4);
            uint32_t* left = (uint32_t*)(rest + select_bytes(a.N, chunk, a.k));
            bool leaves = false;
            const int rc = query_nearest(a, q0, nqc, d_dist, (float*)rest, left, s, leaves);
            if (rc) return rc;
            if (leaves) {      // (as many workgroups as the device holds at a time, at most)
                const int64_t tasks = (int64_t)((nqc + kListed - 1) / kListed) * listed_pieces(a.N);
                hipLaunchKernelGGL(listed_rows_kernel, dim3((unsigned)min((int64_t)a.xcds * 32 * 3, tasks)), dim3(kSelThreads), 0, s, a.data, a.N, a.dim,
                                   a.query + (int64_t)q0 * a.dim, nqc, a.k, a.float_ids, d_dist, (unsigned long long*)rest, left,
                                   a.out_ids + (int64_t)q0 * a.k, a.out_dists + (int64_t)q0 * a.k);
                DCIH_HIP(hipGetLastError());
            }
            if (a.selected) *a.selected += nqc;
            continue;
        }
        // as many queries per wavefront as leave a wavefront to every SIMD (a row is read once for all of them)
        const auto waves = [&](int qn) { return row_groups * ((nqc + qn - 1) / qn); };
        if (waves(8) >= 1024) launch_dists<8>(a, q0, nqc, d_dist, s);
        else if (waves(4) >= 1024) launch_dists<4>(a, q0, nqc, d_dist, s);
        else if (waves(2) >= 1024) launch_dists<2>(a, q0, nqc, d_dist, s);
        else launch_dists<1>(a, q0, nqc, d_dist, s);
        DCIH_HIP(hipGetLastError());
        int32_t* out_ids = a.out_ids + (int64_t)q0 * a.k;
        float* out_dists = a.out_dists + (int64_t)q0 * a.k;
        if (select) {
            unsigned long long* part = (unsigned long long*)((char*)ws + align256((size_t)chunk * (size_t)a.N * 4));
            const bool done = sel.pieces == 1 && sel.kc == a.k;      // (3000 rows, 500 queries: no merge, 5 us of 40)
            hipLaunchKernelGGL(select_rows_kernel, dim3((unsigned)sel.pieces, (unsigned)nqc), dim3(kSelThreads), 0, s,
                               d_dist, a.N, sel.len, sel.kc, part, done ? out_ids : nullptr, out_dists, a.float_ids);
            DCIH_HIP(hipGetLastError());
            if (done) continue;
            QueryArgs m = a;
            m.nq = nqc; m.part = part; m.B = sel.pieces; m.kcap = sel.kc;
            m.out_ids = out_ids; m.out_dists = out_dists;
            const int rc = merge_lists(m, s);
            if (rc) return rc;
            continue;
        }
        const int parts = rank_parts(a.N, nqc);
        const int rc = parts > 1 ? rank_rows_in_parts(d_dist, parts, nqc, (int)a.N, a.k, a.float_ids, out_ids, out_dists, s)
            : rank_fits(a.N)
            ? rank_rows_in_lds(d_dist, nqc, (int)a.N, a.k, a.float_ids, out_ids, out_dists, s)
            : rank_rows(ws, chunk, nqc, a.N, a.k, false, a.float_ids != 0, out_ids, out_dists, s);
        if (rc) return rc;
    }
    if (a.counters) {
        const int64_t cellsc = (int64_t)a.nq * 4;
        hipLaunchKernelGGL(zero_counters_kernel, dim3((unsigned)((cellsc + 255) / 256)), dim3(256), 0, s,
                           a.counters, cellsc);
        hipLaunchKernelGGL(exhaustive_counters_kernel, dim3((unsigned)((int64_t)a.nq * a.B)), dim3(kWave),
                           0, s, a);
        DCIH_HIP(hipGetLastError());
    }
    return 0;
}

}  // namespace dcih
