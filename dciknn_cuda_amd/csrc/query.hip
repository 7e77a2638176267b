// Query path: prioritized traversal of one partition per wavefront, exact
// distances of the promoted points, k best per partition, then a per-query
// merge over partitions.
//
// Stands in for dci_query (src/dci_cuda_kernel.cu:777-875) and the kernels it
// launches once per query: init_dist / init_counts / init_candidate_dists
// (:703-716, :357-382), dci_query_single_point_by_block (:401-626) with
// search_index / init_index_priority / dci_next_closest_proj (:250-355), and
// get_top_candidates (:691-701).
//
// All queries run in one launch: workgroup = one 64-lane wavefront = one
// (query, partition) pair.  The visit counters the reference keeps in global
// memory and re-initialises for every query (4*M*N + 4*N bytes per query) live
// in LDS as packed bit fields, sized by the partition, plus one "seen" bit per
// point; when a partition is too large for LDS they fall back to a per-
// workgroup slice of global scratch.  A window of T sorted entries is visited
// by T lanes at once (in 64-lane slabs when T > 64); promoted points are found
// with a ballot and their rows are read by the whole wavefront.
#include <math.h>

#include "common.h"
#include "kernels.h"

namespace dcih {

namespace {

constexpr int kMaxLds = 160 * 1024;       // LDS per workgroup on gfx950
constexpr int kLdsMargin = 1024;
constexpr int kTopkLdsMax = 2048;         // k up to which the per-partition top-k stays in LDS
constexpr int kMaxSlots = 4096;           // resident workgroups in the global-counter fallback
constexpr int kMergeThreads = 256;

__host__ __device__ inline int counter_bits(int L) {
    return L <= 15 ? 4 : (L <= 255 ? 8 : (L <= 65535 ? 16 : 32));
}

struct Layout {
    int cbits;          // bits per visit counter
    int wpc;            // 32-bit words per composite index counter array
    int seen_words;
    int counter_words;  // M * wpc + seen_words
    int state_bytes;    // left/right/cur/prio/qp + query row
    int topk_bytes;     // 0 when the top-k lives in global memory
    bool lds_counters;
    size_t lds_bytes;
};

Layout make_layout(const QueryArgs& a) {
    Layout y;
    y.cbits = counter_bits(a.L);
    const int64_t fpw = 32 / y.cbits;
    y.wpc = (int)((a.ppb + fpw - 1) / fpw);
    y.seen_words = (int)((a.ppb + 31) / 32);
    const int64_t cw = (int64_t)a.M * y.wpc + y.seen_words;
    y.counter_words = (int)cw;
    const int I = a.M * a.L;
    y.state_bytes = 5 * I * 4 + ((a.dim + 3) & ~3) * 4;
    y.topk_bytes = a.kcap <= kTopkLdsMax ? a.kcap * 8 : 0;
    const int64_t fixed = y.state_bytes + y.topk_bytes + 64;
    y.lds_counters = fixed + cw * 4 <= kMaxLds - kLdsMargin;
    y.lds_bytes = (size_t)(fixed + (y.lds_counters ? cw * 4 : 0));
    return y;
}

// dci_next_closest_proj (src/dci_cuda_kernel.cu:250-273)
__device__ inline int next_window(const float* __restrict__ key, int n, int T, int& left,
                                  int& right, float q) {
    const int lower = -T, upper = n + T - 1;
    int cur;
    if (left <= lower && right >= upper) {
        cur = lower;
    } else if (left <= lower) {
        cur = right; right += T;
    } else if (right >= upper) {
        cur = left; left -= T;
    } else if (key[min(right, n - 1)] - q < q - key[max(left, 0)]) {
        cur = right; right += T;
    } else {
        cur = left; left -= T;
    }
    return cur;
}

// Priority of the window starting at cur (src/dci_cuda_kernel.cu:572-590).
__device__ inline float window_priority(const float* __restrict__ key, int n, int T, int& cur,
                                        float q) {
    int position;
    if (cur < 0 && cur > -T) position = 0;
    else if (cur < n + T - 1 && cur >= n) position = n - 1;
    else position = cur;
    if (position >= 0 && position < n) return fabsf(key[position] - q);
    cur = -T;
    return __builtin_inff();
}

template <bool LDS_COUNTERS>
__global__ __launch_bounds__(kWave) void traverse_kernel(QueryArgs a, Layout y) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int I = a.M * a.L;
    const int lane = threadIdx.x;
    int* s_left = reinterpret_cast<int*>(smem);
    int* s_right = s_left + I;
    int* s_cur = s_right + I;
    float* s_prio = reinterpret_cast<float*>(s_cur + I);
    float* s_qp = s_prio + I;
    float* s_q = s_qp + I;
    unsigned long long* s_top =
        reinterpret_cast<unsigned long long*>(smem + ((y.state_bytes + 15) & ~15));
    uint32_t* s_cnt = reinterpret_cast<uint32_t*>(smem + ((y.state_bytes + 15) & ~15) + y.topk_bytes);

    const int64_t items = a.item_list ? (int64_t)*a.item_count : (int64_t)a.nq * a.B;
    const uint32_t cmask = y.cbits == 32 ? 0xffffffffu : ((1u << y.cbits) - 1u);
    const int fshift = y.cbits == 4 ? 3 : (y.cbits == 8 ? 2 : (y.cbits == 16 ? 1 : 0));  // log2(fields/word)

    for (int64_t slot = blockIdx.x; slot < items; slot += gridDim.x) {
        const int64_t item = a.item_list ? (int64_t)a.item_list[slot] : slot;
        const int b = (int)(item % a.B);
        const int qi = (int)(item / a.B);
        const int64_t off = (int64_t)b * a.ppb;
        const int n = (int)min(a.N - off, a.ppb);
        unsigned long long* top = y.topk_bytes ? s_top : a.part + item * a.kcap;
        unsigned long long* part_out = a.part + item * a.kcap;
        if (n <= 0) {   // empty partition (src/dci_cuda_kernel.cu:429)
            if (!a.dense)
                for (int j = lane; j < a.kcap; j += kWave) part_out[j] = ~0ull;
            continue;
        }
        uint32_t* cnt = LDS_COUNTERS ? s_cnt
                                     : a.gscratch + (size_t)blockIdx.x * (size_t)y.counter_words;
        uint32_t* seen = cnt + (size_t)a.M * y.wpc;

        __syncthreads();
        for (int w = lane; w < y.counter_words; w += kWave) cnt[w] = 0;
        for (int j = lane; j < a.dim; j += kWave) s_q[j] = a.query[(int64_t)qi * a.dim + j];
        if (!LDS_COUNTERS) __threadfence();

        // positioning search (:279-318) and first window of every simple index (:320-355)
        unsigned long long probes = 0;
        for (int i = lane; i < I; i += kWave) {
            const float* key = a.skeys + (int64_t)i * a.N + off;
            const float qp = a.qproj[(int64_t)i * a.nq + qi];
            int start_pos = -1, end_pos = n - 1;
            int cur_pos = (start_pos + end_pos + 2) / 2;
            while (start_pos < end_pos) {
                probes++;
                if (key[cur_pos] < qp) start_pos = cur_pos; else end_pos = cur_pos - 1;
                cur_pos = (start_pos + end_pos + 2) / 2;
            }
            int left = start_pos - a.T + 1;
            int right = left + a.T;
            int cur = next_window(key, n, a.T, left, right, qp);
            const float pr = window_priority(key, n, a.T, cur, qp);
            s_left[i] = left; s_right[i] = right; s_cur[i] = cur; s_prio[i] = pr; s_qp[i] = qp;
        }
        __syncthreads();

        const int64_t bound = (int64_t)n * a.L * a.T;     // :458
        int64_t kk = 0, c0 = 0;
        unsigned long long visited = 0, ncand = 0, steps = 0;
        int tk_count = 0;                 // entries in `top`
        unsigned long long tk_max = 0;    // largest packed entry once full
        int tk_maxslot = 0;

        while (kk < bound) {
            bool any = false;
            for (int m = 0; m < a.M; m++) {
                // first strict minimum of the L priorities (:466-478)
                uint32_t best = 0x7f800000u;   // +inf: an exhausted simple index never wins
                int best_h = 0x7fffffff;
                for (int h = lane; h < a.L; h += kWave) {
                    const uint32_t p = __builtin_bit_cast(uint32_t, s_prio[m * a.L + h]);
                    if (p < best) { best = p; best_h = h; }
                }
                const uint32_t wbest = wave_min_u32(best);
                if (wbest >= 0x7f800000u) continue;
                const int top_h = (int)wave_min_u32(best == wbest ? (uint32_t)best_h : 0x7fffffffu);
                any = true;
                const int i = m * a.L + top_h;
                const int position = s_cur[i];
                const int32_t* ids = a.sids + (int64_t)i * a.N + off;
                uint32_t* mcnt = cnt + (size_t)m * y.wpc;

                for (int t0 = 0; t0 < a.T; t0 += kWave) {     // :487-562
                    const int t = t0 + lane;
                    const int cur_index = position + t;
                    const bool valid = t < a.T && cur_index >= 0 && cur_index < n;
                    int pt = -1;
                    bool promoted = false;
                    if (valid) {
                        pt = ids[cur_index];
                        const uint32_t local = (uint32_t)(pt - off);
                        const uint32_t sh = (local & ((1u << fshift) - 1u)) * y.cbits;
                        const uint32_t old = atomicAdd(&mcnt[local >> fshift], 1u << sh);
                        if (((old >> sh) & cmask) + 1u == (uint32_t)a.L) {
                            const uint32_t bit = 1u << (local & 31);
                            promoted = (atomicOr(&seen[local >> 5], bit) & bit) == 0;
                        }
                    }
                    visited += __popcll(__ballot(valid));
                    unsigned long long pm = __ballot(promoted);
                    while (pm) {
                        const int src = __ffsll((long long)pm) - 1;
                        pm &= pm - 1;
                        const int cpt = __shfl(pt, src, kWave);
                        uint32_t score;
                        if (a.blind) {
                            score = (uint32_t)kk;     // (:498-505: recorded, no distance)
                        } else {
                            // exact distance (:36-44), row read by the whole wavefront
                            const float* const rows1[1] = {a.data + (int64_t)cpt * a.dim};
                            float dist1[1];
                            wave_row_dists<1>(rows1, s_q, a.dim, rows_vec4(a.data, a.dim), dist1);
                            score = __builtin_bit_cast(uint32_t, dist1[0]);
                        }
                        const unsigned long long e = ((unsigned long long)score << 32) | (uint32_t)cpt;
                        ncand++;
                        if (t0 + src == 0) c0++;          // only lane 0's promotions count (:413, :598)
                        if (a.dense) {
                            // every candidate is kept: its score goes to its own cell of the query's row
                            if (lane == 0)
                                a.dense[(int64_t)qi * a.N + cpt] =
                                    a.blind ? (float)score : __builtin_bit_cast(float, score);
                        } else if (tk_count < a.kcap) {
                            if (lane == 0) top[tk_count] = e;
                            if (tk_count == 0 || e > tk_max) { tk_max = e; tk_maxslot = tk_count; }
                            tk_count++;
                        } else if (e < tk_max) {
                            if (lane == 0) top[tk_maxslot] = e;
                            __syncthreads();
                            if (!y.topk_bytes) __threadfence();
                            unsigned long long mx = 0;
                            for (int j = lane; j < a.kcap; j += kWave) {
                                const unsigned long long v = top[j];
                                if (v > mx) mx = v;
                            }
                            mx = wave_max_u64(mx);
                            int slot = 0x7fffffff;
                            for (int j = lane; j < a.kcap; j += kWave)
                                if (top[j] == mx) slot = min(slot, j);
                            tk_max = mx;
                            tk_maxslot = (int)wave_min_u32((uint32_t)slot);
                        }
                    }
                }
                __syncthreads();
                if (lane == 0) {        // :566-591
                    const float* key = a.skeys + (int64_t)i * a.N + off;
                    int left = s_left[i], right = s_right[i];
                    const float qp = s_qp[i];
                    int cur = next_window(key, n, a.T, left, right, qp);
                    const float pr = window_priority(key, n, a.T, cur, qp);
                    s_left[i] = left; s_right[i] = right; s_cur[i] = cur; s_prio[i] = pr;
                }
                __syncthreads();
            }
            steps++;
            if (c0 >= a.k_stop && (kk + 1 >= a.stop_at || c0 >= a.max_cand)) break;   // :598-607
            if (!any) break;   // every simple index exhausted: nothing can change any more
            kk++;
        }

        __syncthreads();
        if (!y.topk_bytes) __threadfence();
        if (!a.dense && y.topk_bytes) {      // in ascending order, as the merge takes them (no entry occurs twice)
            for (int j = lane; j < tk_count; j += kWave) {
                const unsigned long long v = top[j];
                int rank = 0;
                for (int o = 0; o < tk_count; o++) rank += top[o] < v ? 1 : 0;
                part_out[rank] = v;
            }
        }
        for (int j = lane + (y.topk_bytes ? tk_count : 0); j < (a.dense ? 0 : a.kcap); j += kWave)
            part_out[j] = j < tk_count ? top[j] : ~0ull;
        if (a.counters) {
            for (int o = 32; o > 0; o >>= 1) probes += __shfl_xor(probes, o, kWave);
            if (lane == 0) {
                atomicAdd(&a.counters[(int64_t)qi * 4 + 0], visited);
                atomicAdd(&a.counters[(int64_t)qi * 4 + 1], ncand);
                atomicAdd(&a.counters[(int64_t)qi * 4 + 2], probes);
                atomicAdd(&a.counters[(int64_t)qi * 4 + 3], steps);
            }
        }
    }
}

// One result of a query: the id (as float32 where the caller takes ids that way) and the distance.
__device__ inline void store_result(const QueryArgs& a, int qi, int j, unsigned long long v) {
    const bool empty = v == ~0ull;
    const int32_t id = empty ? -1 : (int32_t)(uint32_t)v;
    a.out_ids[(int64_t)qi * a.k + j] = a.float_ids ? __builtin_bit_cast(int32_t, (float)id) : id;
    if (a.out_dists)
        a.out_dists[(int64_t)qi * a.k + j] =
            empty ? __builtin_inff()
                  : (a.blind ? (float)(uint32_t)(v >> 32) : __builtin_bit_cast(float, (uint32_t)(v >> 32)));
}

// k best of the B*kcap per-partition results of one query (get_top_candidates,
// src/dci_cuda_kernel.cu:691-701), more than 256 of them: repeated LDS bitonic sorts of the running
// best k (kept at buf[0, k)) plus as many new entries as fit cap words; k <= cap / 2.
__device__ inline void merge_by_sorting(unsigned long long* buf, int cap, int k, const unsigned long long* src, int64_t total) {
    const int room = cap - k;
    for (int j = threadIdx.x; j < k; j += blockDim.x) buf[j] = ~0ull;
    for (int64_t p = 0; p < total; p += room) {
        const int m = (int)min((int64_t)room, total - p);
        __syncthreads();
        for (int j = threadIdx.x; j < room; j += blockDim.x)
            buf[k + j] = j < m ? src[p + j] : ~0ull;
        bitonic_sort_u64(buf, cap);
    }
    __syncthreads();
}

__global__ __launch_bounds__(kMergeThreads) void merge_topk_kernel(QueryArgs a, int cap) {
    extern __shared__ unsigned long long buf[];
    const int qi = blockIdx.x;
    if (a.only && a.only[qi] != a.only_round) return;
    merge_by_sorting(buf, cap, a.k, a.part + (int64_t)qi * a.B * a.kcap, (int64_t)a.B * a.kcap);
    for (int j = threadIdx.x; j < a.k; j += blockDim.x) store_result(a, qi, j, buf[j]);
}

// The same for k <= NT.  The lists ascend, so the k-th smallest of their first few entries is an
// upper bound of the k-th best, and only the entries up to it -- k and a few more, all near the
// lists' beginnings -- are read and sorted.  (The bound comes from the `heads` first entries of
// every list, at least 2 k in all; where those are more than NT, from the smallest of each thread's
// share of them.)  Bound by its chain of reads, sorts and barriers: one wavefront per query where
// the heads fit two per lane.  10000 queries of 58 lists of 10: 171 us with the sorts of 1024 words above.
template <int NT, bool ROUNDS>      // ROUNDS: some queries' results stay as they are
__global__ __launch_bounds__(NT) void merge_heads_kernel(QueryArgs a, int heads) {
    constexpr int kCap = NT == kWave ? 256 : 2048, kAhead = 4;
    __shared__ unsigned long long buf[kCap];
    __shared__ uint32_t s_count;
    const int tid = threadIdx.x, qi = blockIdx.x;
    if (ROUNDS && a.only[qi] != a.only_round) return;
    const unsigned long long* src = a.part + (int64_t)qi * a.B * a.kcap;
    const int nheads = a.B * heads;
    unsigned long long best = ~0ull;
    for (int e = tid; e < nheads; e += NT) {
        const unsigned long long v = src[(int64_t)(e / heads) * a.kcap + e % heads];
        best = v < best ? v : best;
    }
    buf[tid] = best;
    if (tid == 0) s_count = 0;
    if constexpr (NT == kWave) bitonic_sort_u64(buf, NT); else bitonic_sort_u64_by256(buf, NT);
    const unsigned long long bound = buf[a.k - 1];       // (nothing at all in some list heads: ~0, every entry passes)
    __syncthreads();
    // (as many threads to a list as there are, every one with its own entries: two lists of 100, 17 -> 10 us)
    int lg = 0;
    while ((2 * a.B << lg) <= NT) lg++;
    for (int l = tid >> lg; l < a.B; l += NT >> lg) {
        const unsigned long long* list = src + (int64_t)l * a.kcap;
        for (int j0 = (tid & ((1 << lg) - 1)) * kAhead; j0 < a.kcap; j0 += kAhead << lg) {
            unsigned long long v[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++) v[u] = list[min(j0 + u, a.kcap - 1)];
            bool more = true;
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const bool take = j0 + u < a.kcap && v[u] <= bound && v[u] != ~0ull;
                if (take) {
                    const uint32_t slot = atomicAdd(&s_count, 1u);
                    if (slot < (uint32_t)kCap) buf[slot] = v[u];
                }
                more = more && take;
            }
            if (!more) break;
        }
    }
    __syncthreads();
    const int count = (int)s_count;
    if (count > kCap) {      // a few lists hold nearly all of the best: the lists as a whole
        merge_by_sorting(buf, kCap, a.k, src, (int64_t)a.B * a.kcap);
    } else {
        int n = kWave;
        while (n < count || n < a.k) n <<= 1;
        for (int j = count + tid; j < n; j += NT) buf[j] = ~0ull;
        if (NT == kMergeThreads && n >= kMergeThreads) bitonic_sort_u64_by256(buf, n);
        else bitonic_sort_u64(buf, n);
    }
    for (int j = tid; j < a.k; j += NT) store_result(a, qi, j, buf[j]);
}

// Clears n 64-bit words at p and also_n 32-bit words at `also` (either may be null / 0).
__global__ void zero_u64_kernel(unsigned long long* p, int64_t n, uint32_t* also, int also_n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += stride) p[e] = 0;
    if (also && blockIdx.x == 0 && (int)threadIdx.x < also_n) also[threadIdx.x] = 0;
}

// Words of the merge's sort buffer: room for the k best plus at least as many new entries, and
// no more than the per-partition lists hold in all (a sort of 2048 words for 590 entries would
// spend most of its stages on padding).
int merge_cap(int k, int64_t total) {
    int cap = 2048;
    while (cap < 2 * k) cap <<= 1;
    int need = 64;
    while ((int64_t)need < (int64_t)k + total && need < cap) need <<= 1;
    return need < cap ? need : cap;
}

}  // namespace

// The traversal and merge kernels may use all of a CU's LDS.
static int allow_full_lds() {
    static DeviceOnce once;
    return once.run([]() -> int {
        DCIH_HIP(hipFuncSetAttribute((const void*)traverse_kernel<true>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
        DCIH_HIP(hipFuncSetAttribute((const void*)traverse_kernel<false>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
        DCIH_HIP(hipFuncSetAttribute((const void*)merge_topk_kernel,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
        return 0;
    });
}

int zero_words64(void* d_p, int64_t n, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(zero_u64_kernel, dim3((unsigned)max((int64_t)1, min((int64_t)1024, (n + 255) / 256))),
                       dim3(256), 0, s, (unsigned long long*)d_p, n, (uint32_t*)nullptr, 0);
    DCIH_HIP(hipGetLastError());
    return 0;
}

size_t query_part_bytes(const QueryArgs& a) {
    return (size_t)a.nq * a.B * a.kcap * sizeof(unsigned long long);
}

static int64_t traverse_grid(const QueryArgs& a, const Layout& y) {
    const int64_t items = (int64_t)a.nq * a.B;
    if (y.lds_counters) return min(items, step_grid_cap());   // the kernel strides over its items
    return min(items, (int64_t)kMaxSlots);
}

size_t query_gscratch_bytes(const QueryArgs& a) {
    const Layout y = make_layout(a);
    if (y.lds_counters) return 0;
    return (size_t)traverse_grid(a, y) * (size_t)y.counter_words * 4;
}

// Left to choose: from the number of promotions at which the dense kernel is the cheaper one for sure,
// and where it is estimated to be, every item goes straight to it (no hints needed: also a first call is
// routed right).  The estimates mostly decide for small partitions (69 points, L = 7, 390 items: 26 us
// against the batch kernel's 156) and for calls of few items, which wait for the batch kernel's chain of epochs.
bool takes_dense_kernel(const QueryArgs& a) {
    if (a.mode == 3) return true;
    if (a.mode != 0 || a.dense_min_promos <= 0) return false;
    const double promotions = fmin(expected_promotions(a), (double)a.ppb);
    if (promotions >= (double)a.dense_min_promos) return true;
    if (!a.dense_by_cost) return false;
    // (of all items, in rounds too: where bounds rule nothing out every item comes after all, and the dense kernel, chosen for few items,
    // takes up to five times as long.  5 results of 300 queries, 100 partitions of 10000 rows of 300, normal rows: 4.2 ms whole, 19.4 in
    // rounds by the dense kernel, 4.6 by the batch kernel; a manifold's rows of 128, 10 results: 4.4, 3.5, 4.1.)
    QueryArgs whole = a;
    whole.share = 1.0;
    const TraversalCosts c = traversal_costs(whole, promotions);
    return c.dense < c.batch;
}

// Whether a round's items go through confirm.hip first.  That takes about 0.02 us of an item where items fill the device, a traversal 0.03 to 0.25; it loses where
// partitions are short (137 rows of 41, windows of 10: 427 us without, 466 with; 127 of 675: 1.50 ms, 2.48; 947 of 168: 4.99, 1.07) and where it has to leave
// too many (331 rows, a sixth of the items left: 2.64, 3.15; 2818 rows, a twelfth: 9.19, 5.86).  Calls that are over soon have to be answered as a whole, or
// they wait for a traversal as well (455 items, 25 left: 278 us, 444; 5800, a fifth left: 1.44, 1.55 ms), and the positions by the first simple index, which
// it reads, are not formed for the first small call of an index (one that is formed anew for a few lookups).
// may_pay: whether it can be so for such a call at all, whatever the index's calls so far.
static bool confirm_pays(const QueryArgs& a, double items, bool by_dense, int& may_pay) {
    may_pay = 1;
    if (a.pick_rule == 2) return true;
    const double item = by_dense ? traversal_costs(a, 0.0).dense_item : 1.0;
    may_pay = item >= 0.024;
    if (!may_pay) return false;
    if (items <= 4096.0 && confirm_scans(a) && !*a.rpos_ready && a.index_calls == 0) return false;
    const double may = items <= 16384.0 ? 1.0 / 256.0 : fmin(1.0, (item - 0.022) / 0.02);
    return (double)a.confirm_lost <= (items <= 16384.0 ? 0.0 : 16.0) + may * (double)a.confirm_had;
}

bool plan_rounds(QueryArgs& a) {
    a.pick_rounds = a.pick_near = a.pick_confirm = a.pick_sample = 0;
    a.pick_parts = 1;
    a.share = 1.0;
    if (a.mode != 0 || a.pick_rule == 1 || !bounds_supported(a)) return false;
    // The r nearest rows of a query lie in about B (1 - e^(-r/B)) partitions (rows in no particular order).  Round 1
    // takes those of the k nearest, and where traversals find most of them the later rounds add a tenth.  A call of so few items
    // that twice as many partitions are one more item for some workgroups takes those of the 2 k nearest instead: a second
    // round is then mostly empty, and waiting for one more item would take longer.
    const double B = (double)a.B;
    auto parts_of = [&](double r) { return fmin(B, B * (1.0 - exp(-r / B)) + 0.5); };
    const bool few = (double)a.nq * parts_of(2.0 * (double)a.k) <= 1024.0;
    const int rank = few ? 2 * a.k : a.k + a.k / 16;      // (a few are missed: 10M unit vectors, k = 100: 111 pairs a query at 100, 102 at 110)
    const double first = parts_of((double)rank);
    const double share = fmin(1.0, (few ? first : 1.1 * first + 0.2) / B);
    const bool can_dense = dense_traversal_supported(a, nullptr), can_block = block_traversal_supported(a, nullptr);
    bool fits = true;
    auto time = [&](double part) {
        QueryArgs p = a;
        p.share = part;
        const TraversalCosts c = traversal_costs(p, fmin(expected_promotions(a), (double)a.ppb));
        const bool dense = can_dense && takes_dense_kernel(p);
        fits = fits && (dense || (can_block && block_takes_lists(a)));      // (the step-by-step kernel takes no round's items)
        return dense ? c.dense : c.batch;
    };
    const double whole = time(1.0), traversals = time(first / B) + (few ? 15.0 : time(share - first / B)), rounds = traversals + bounds_cost(a) + 30.0;
    (void)time(share);
    // Traversals that stop after less than one promotion of fifty points find rows further away than the bounds of most partitions where
    // distances lie close together, and every partition is traversed after all.  Such queries then take all in one round (unit vectors
    // of 241 elements, 42 partitions, 985 queries: 0.95 ms whole, 2.2 in rounds, 1.03 so), and rounds have to promise more.
    const bool short_stops = expected_promotions(a) < 0.02 * (double)a.ppb;
    // Traversals that stop after less than a twentieth of their partition (and those of the batch kernel) may find too little for bounds to rule
    // anything out; a sample of the queries says so (bounds.hip).  That takes as long as an item does, and each round waits for its
    // slowest item too, so calls of less than 25 times that are traversed whole.  (1215 shapes: without this rule and the sample 110 took more than
    // 3 % longer than whole, up to five times as long; with them the sample costs what takes everything 2 to 7 %.)
    const bool by_batch = !(can_dense && takes_dense_kernel(a));
    const bool sampled = by_batch || expected_promotions(a) < 0.05 * (double)a.ppb;
    if (sampled && a.pick_rule == 0 && whole < 25.0 * time(1.0 / ((double)a.nq * B))) return false;
    if (!fits || (a.pick_rule == 0 && rounds > (short_stops ? 0.6 : 0.85) * whole)) return false;
    // One to three results of traversals that leave out near rows bound little: everything else follows in the later rounds (32 queries, 64
    // partitions of 8000 normal rows of 32, k = 3: 539 us whole, 710 in rounds; of 6000, k = 1: 378, 415; k = 10: 401, 229), and calls of
    // one item for every workgroup gain less than that costs (14 queries, 64 partitions of 4000, k = 1: 155, 193; 32 queries: 295, 189).
    if (a.pick_rule == 0 && a.k < 4 && (whole < 250.0 || expected_promotions(a) < 0.3 * (double)a.ppb)) return false;
    a.pick_flat = short_stops ? 1.3f : 0.0f;
    a.pick_rounds = few ? 2 : (whole > 1500.0 || a.pick_rule == 2 ? (by_batch ? 3 : kMostRounds) : 2);
    a.pick_rank = rank;
    a.pick_first = first;
    a.share = share;
    a.pick_near = !sampled;
    a.may_confirm = 0;
    a.pick_confirm = confirm_supported(a) && confirm_pays(a, (double)a.nq * first, can_dense && takes_dense_kernel(a), a.may_confirm) ? 1 : 0;
    // Where the tiles' bounds take more than their room, the dense kernel's calls come as parts of the queries that keep within it, one after the other.  All that
    // each does again is to read the rows once.  (10000 queries on 10M unit vectors of 96: 397 ms without these bounds, 144 in parts; on 20M normal rows of 64 221, 153;
    // 60000 on 1M rows of 128 at the defaults 132, 22.4, with room for all 21.6; 20000 on 3M unit vectors 407, 172; where bounds rule out little, 30000 on 2M
    // normal rows of 64, 3124, 3187.)  A part of the batch kernel's calls takes its own sample and waits for its own slowest items: 60000 queries, windows
    // of 2, 46.0 ms without the tiles' bounds, 48.9 in two parts.
    // Left to choose, only parts that would go in rounds with these bounds themselves, and whose reading of the rows again and launches take less
    // than a third of what the traversals are estimated to: that much, and mostly more, these bounds saved above.
    const size_t near = near_bytes(a);
    if (near > a.near_room) {
        if (a.pick_near) {
            QueryArgs part = a;
            int parts = (int)std::min<size_t>((size_t)a.nq, (near + a.near_room - 1) / a.near_room);
            for (;; parts += 1 + parts / 8) {      // (few queries' tiles can be smaller ones, and their bounds more)
                parts = std::min(parts, a.nq);
                part.nq = (a.nq + parts - 1) / parts;
                if (part.nq == 1 || near_bytes(part) <= a.near_room) break;
            }
            bool pays = a.pick_rule == 2;
            if (!pays && near_bytes(part) <= a.near_room) {
                const double again = (double)(parts - 1) * (bounds_cost(part) + 60.0) + bounds_cost(part) - bounds_cost(a);
                pays = again < 0.3 * traversals && plan_rounds(part) && part.pick_near;
            }
            if (pays) a.pick_parts = parts;
        }
        a.pick_near = a.pick_confirm = a.may_confirm = 0;
    }
    a.pick_sample = sampled ? std::min(a.nq, std::max(2, std::min(16, 1024 / a.B))) : 0;
    // Up to which share of the sample's pairs rounds pay: the fewer results, the further away the k-th of the first rounds lies than
    // that of all.  (Five kinds of rows, 16 to 300 elements, 30000 to a million: shares from which rounds begin to take longer are 0.31 to
    // 0.37 for 5 results, 0.39 to 0.51 for 10 and 0.75 for 30; all of them at a share of 0.7, 10 results: 0.69 to 0.94 of whole calls' rate.)
    a.pick_most = a.pick_rule == 2 ? 2.0f : (float)(0.75 * (double)a.k / ((double)a.k + 7.5));
    return true;
}

int merge_lists(const QueryArgs& a, hipStream_t s) {
    // (the lists of the step-by-step kernel ascend as long as its top-k stays in LDS)
    // (after a round only the lists of the partitions taken so far, about pick_first of them, hold anything)
    const double lists = a.pick_rounds ? fmax(1.0, a.pick_first) : (double)a.B;
    const int heads = min(a.kcap, (int)ceil((a.pick_rounds ? 3.0 : 2.0) * (double)a.k / lists));
    if (a.k <= 32 && (int64_t)a.B * heads <= 2 * kWave) {
        hipLaunchKernelGGL((a.only ? merge_heads_kernel<kWave, true> : merge_heads_kernel<kWave, false>), dim3((unsigned)a.nq), dim3(kWave), 0, s, a, heads);
    } else if (a.k <= kMergeThreads && (int64_t)a.B * heads < 0x7fffffffLL) {
        hipLaunchKernelGGL((a.only ? merge_heads_kernel<kMergeThreads, true> : merge_heads_kernel<kMergeThreads, false>), dim3((unsigned)a.nq),
                           dim3(kMergeThreads), 0, s, a, heads);
    } else {
        const int cap = merge_cap(a.k, (int64_t)a.B * a.kcap);
        hipLaunchKernelGGL(merge_topk_kernel, dim3((unsigned)a.nq), dim3(kMergeThreads),
                           (size_t)cap * sizeof(unsigned long long), s, a, cap);
    }
    DCIH_HIP(hipGetLastError());
    return 0;
}

int query(const QueryArgs& a_in, void* bounds_ws, hipStream_t s, hipEvent_t* ev, bool* ran) {
    QueryArgs a = a_in;
    if (a.nq <= 0) return 0;
    if (a.k > 8192)
        return fail(-4, a.blind ? "query: more than 8192 blind candidates per query are not supported"
                                : "query: num_neighbours above 8192 is not supported");
    if (a.blind && (int64_t)a.L * (a.ppb + 2 * (int64_t)a.T) >= 0x7fffffffLL)
        return fail(-4, "query: blind querying needs step numbers that fit 31 bits");
    if ((int64_t)a.M * a.ppb * 8 > 0x7fffffffLL)
        return fail(-4, "query: partition too large for the visit counters; use a larger block_size");
    const Layout y = make_layout(a);
    if (y.lds_bytes > (size_t)kMaxLds)
        return fail(-4, "query: dim / num_indices / num_neighbours too large for LDS state");
    const bool can_block = block_traversal_supported(a, nullptr);
    const bool can_dense = dense_traversal_supported(a, nullptr);
    if (a.mode == 2 && !can_block)
        return fail(-4, "query: this shape does not fit the batch traversal kernel");
    if (a.mode == 3 && !can_dense)
        return fail(-4, "query: this shape does not fit the dense traversal kernel");
    if (can_dense && takes_dense_kernel(a)) a.mode = 3;
    // An item that is already under way in the batch kernel is worth moving only from twice the number of
    // promotions at which a whole call is routed to the dense kernel: below that, finishing it there is
    // cheaper than starting over here.  By cost: from one and a half times the promotions that take as long as the
    // dense kernel takes for all (1000 points, T = 2, L = 15, k = 1, 20000 items: 1.8 ms, 13.5 ms at a fixed 320;
    // at one half of them calls whose traversals mostly stop soon after take up to twice as long).
    a.hand_over_at = 2 * a.dense_min_promos;
    if (a.dense_by_cost) {
        const TraversalCosts c = traversal_costs(a, 0.0);
        a.hand_over_at = (int)fmin((double)a.hand_over_at, fmax(16.0, 1.5 * c.dense_item / c.batch_per_promotion));
    }
    const bool use_block = a.mode != 1 && a.mode != 3 && can_block;
    // the batch kernel hands items that need many promotions to the dense kernel
    if (!(use_block && a.mode == 0 && can_dense && a.dense_items && a.dense_min_promos > 0)) {
        if (a.mode != 3) a.dense_items = nullptr;
    }
    {
        const int rc = allow_full_lds();
        if (rc) return rc;
    }
    auto traverse = [&](QueryArgs a) -> int {
        const bool lists = a.mode != 3;         // the dense kernel alone leaves no item to another
        if (lists || a.counters) {   // zero the counters and the list lengths with a kernel (safe under graph capture);
            // the dense lists' lengths follow the hand-over list's
            const int64_t cells = a.counters ? (int64_t)a.nq * 4 : 0;
            hipLaunchKernelGGL(zero_u64_kernel, dim3((unsigned)max((int64_t)1, min((int64_t)1024, (cells + 255) / 256))),
                               dim3(256), 0, s, a.counters, cells, a.redo_count, kListCountWords);
        }
        a.item_list = nullptr;
        a.item_count = nullptr;
        if (use_block || a.mode == 3) {
            if (use_block) {
                if (a.rpos_ready && !*a.rpos_ready) {      // the first batch traversal over this index
                    const int rc = fill_positions_by_first(a.sids, a.inv, const_cast<uint16_t*>(a.rpos), a.N, a.M, a.L, a.ppb, a.B, s);
                    if (rc) return rc;
                    if (!a.recorded) *a.rpos_ready = 1;
                }
                const int rc = query_block(a, s);
                if (rc) return rc;
                if (ev) (void)hipEventRecord(ev[1], s);
                if (ran) ran[0] = true;
            }
            if (a.mode == 3 || a.dense_items) {
                QueryArgs d = a;
                if (use_block) { d.picked = nullptr; d.near_bounds = nullptr; }      // what the batch kernel handed over
                const int rc = query_dense_items(d, s);
                if (rc) return rc;
                if (ev) (void)hipEventRecord(ev[2], s);
                if (ran) ran[1] = true;
            }
        }
        if (use_block) {
            // whatever the batch kernel handed back goes through the step-by-step kernel
            a.item_list = a.redo_items;
            a.item_count = a.redo_count;
            if (y.lds_counters) {
                const int64_t grid = min((int64_t)a.nq * a.B, (int64_t)1024);
                hipLaunchKernelGGL(traverse_kernel<true>, dim3((unsigned)grid), dim3(kWave), y.lds_bytes, s, a, y);
            } else {      // partitions whose visit counters do not fit LDS: a slice of global scratch per workgroup
                if (!a.gscratch) return fail(-1, "query: counter scratch missing");
                const int64_t grid = min(traverse_grid(a, y), (int64_t)1024);
                hipLaunchKernelGGL(traverse_kernel<false>, dim3((unsigned)grid), dim3(kWave), y.lds_bytes, s, a, y);
            }
        } else if (a.mode != 3) {
            const int64_t grid = traverse_grid(a, y);
            if (y.lds_counters) {
                hipLaunchKernelGGL(traverse_kernel<true>, dim3((unsigned)grid), dim3(kWave), y.lds_bytes, s, a, y);
            } else {
                if (!a.gscratch) return fail(-1, "query: counter scratch missing");
                hipLaunchKernelGGL(traverse_kernel<false>, dim3((unsigned)grid), dim3(kWave), y.lds_bytes, s, a, y);
            }
        }
        DCIH_HIP(hipGetLastError());
        return 0;
    };
    if (ev && ev[0]) (void)hipEventRecord(ev[0], s);
    if (!a.pick_rounds) {
        const int rc = traverse(a);
        if (rc) return rc;
    } else {      // rounds (bounds.hip): the results of one bound what the next has to take
        int rc = pack_bounds(a, bounds_ws, s);
        if (a.pick_sample && !rc) {
            Picked p;
            rc = sample_items(a, bounds_ws, p, s);
            if (rc) return rc;
            a.picked = p.items;
            a.picked_count = p.count;
            a.picked_ticket = p.ticket;
            a.picked_exact = a.picked_cover = (int64_t)a.pick_sample * a.B;
            a.picked_expect = 0;
            rc = traverse(a);
            a.only = p.last_round;
            a.only_round = kSampleRound;
            if (!rc) rc = merge_lists(a, s);
            if (!rc) rc = sample_decide(a, bounds_ws, s);
            if (a.round_items && !rc)
                DCIH_HIP(hipMemcpyAsync(a.round_items + kMostRounds, p.count + (kSkipWord - kSampleWord), 2 * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
            a.picked_exact = 0;
            a.only = nullptr;
        }
        if (!rc) rc = partition_bounds(a, bounds_ws, s);
        for (int round = 0; round < a.pick_rounds && !rc; round++) {
            if (round > 0) rc = merge_lists(a, s);
            if (!rc) rc = pick_items(a, bounds_ws, round, a.pick_rounds, s);
            const Picked p = picked_items(a, bounds_ws, round);
            a.picked = p.items;
            a.picked_count = p.count;
            a.picked_ticket = p.ticket;
            if (a.round_items && !rc) DCIH_HIP(hipMemcpyAsync(a.round_items + round, p.count, sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
            a.near_bounds = p.near_bounds; a.near_limit = p.near_limit; a.near_stride = p.near_stride;
            a.near_shift = p.near_shift; a.near_tiles = p.near_tiles;
            // The batch kernel's first launch covers all that may come in the first round, where queries whose bounds lie close together take
            // every partition: strides over the rest take up to twice as long, a workgroup without an item 0.5 ns.  (4000 queries, 58 partitions
            // of 17242 normal rows of 128: 15.2 ms whole, 18.9 in rounds that covered 131072 items.)
            a.picked_cover = round ? std::max((int64_t)(0.3 * (double)a.nq * (double)a.B), (int64_t)65536) : (int64_t)a.nq * a.B;
            if (a.pick_confirm && round) a.picked_cover = std::min(a.picked_cover, (int64_t)16384);
            a.picked_expect = round ? 0 : (int64_t)((double)a.nq * a.pick_first);
            if (a.pick_confirm && !rc) {
                if (confirm_scans(a) && a.rpos_ready && !*a.rpos_ready) {
                    rc = fill_positions_by_first(a.sids, a.inv, const_cast<uint16_t*>(a.rpos), a.N, a.M, a.L, a.ppb, a.B, s);
                    if (!rc && !a.recorded) *a.rpos_ready = 1;
                }
                a.near_limit = p.confirm_limit;
                if (!rc) rc = confirm_round(a, bounds_ws, s);
                a.near_limit = p.near_limit;
                a.picked_expect = 0;
                if (!a.pick_near) a.near_bounds = nullptr;
            }
            if (!rc) rc = traverse(a);
            a.left = nullptr;
            a.only = round > 0 ? p.last_round : nullptr;
            a.only_round = (uint32_t)round;
        }
        if (rc) return rc;
    }
    DCIH_HIP(hipGetLastError());
    if (ev) (void)hipEventRecord(ev[3], s);
    {
        const int rc = merge_lists(a, s);
        if (rc) return rc;
    }
    if (ev) (void)hipEventRecord(ev[4], s);
    DCIH_HIP(hipGetLastError());
    return 0;
}

int query_dense(const QueryArgs& a_in, const float* d_dirs, void* ws, int chunk, hipStream_t s) {
    if (a_in.nq <= 0) return 0;
    const int I = a_in.M * a_in.L;
    if ((int64_t)a_in.M * a_in.ppb * 8 > 0x7fffffffLL)
        return fail(-4, "query: partition too large for the visit counters; use a larger block_size");
    // blind scores are step numbers stored as floats: they must stay exact
    if (a_in.blind && (int64_t)a_in.L * (a_in.ppb + 2 * (int64_t)a_in.T) >= (1 << 24))
        return fail(-4, "query: this many blind results need step numbers below 2^24; use a larger block_size");
    {
        const int rc = allow_full_lds();
        if (rc) return rc;
    }
    const size_t qp_bytes = ((size_t)I * chunk * sizeof(float) + 255) & ~(size_t)255;
    float* d_qproj = (float*)ws;
    void* ws_rank = (char*)ws + qp_bytes;
    for (int q0 = 0; q0 < a_in.nq; q0 += chunk) {
        QueryArgs a = a_in;             // this chunk's queries as a query batch of their own
        a.nq = min(chunk, a_in.nq - q0);
        a.query = a_in.query + (int64_t)q0 * a.dim;
        a.qproj = d_qproj;
        a.counters = a_in.counters ? a_in.counters + (int64_t)q0 * 4 : nullptr;
        a.kcap = 1;                     // no per-partition lists
        a.part = nullptr;
        a.item_list = nullptr;
        a.item_count = nullptr;
        a.dense = rank_rows_input(ws_rank);
        int rc = project(d_dirs, I, a.query, a.nq, a.dim, d_qproj, a.nq, s);
        if (rc) return rc;
        rc = fill_rows(a.dense, (int64_t)a.nq * a.N, __builtin_inff(), s);
        if (rc) return rc;
        const Layout y = make_layout(a);
        if (y.lds_bytes > (size_t)kMaxLds)
            return fail(-4, "query: dim / num_indices too large for LDS state");
        const int64_t cells = a.counters ? (int64_t)a.nq * 4 : 0;
        hipLaunchKernelGGL(zero_u64_kernel, dim3((unsigned)max((int64_t)1, min((int64_t)1024, (cells + 255) / 256))),
                           dim3(256), 0, s, a.counters, cells, (uint32_t*)nullptr, 0);
        const int64_t grid = traverse_grid(a, y);
        if (y.lds_counters) {
            hipLaunchKernelGGL(traverse_kernel<true>, dim3((unsigned)grid), dim3(kWave), y.lds_bytes, s, a, y);
        } else {
            if (!a.gscratch) return fail(-1, "query: counter scratch missing");
            hipLaunchKernelGGL(traverse_kernel<false>, dim3((unsigned)grid), dim3(kWave), y.lds_bytes, s, a, y);
        }
        DCIH_HIP(hipGetLastError());
        rc = rank_rows(ws_rank, chunk, a.nq, a.N, a_in.k, true, a_in.float_ids != 0, a_in.out_ids + (int64_t)q0 * a_in.k,
                       a_in.out_dists ? a_in.out_dists + (int64_t)q0 * a_in.k : nullptr, s);
        if (rc) return rc;
    }
    return 0;
}

}  // namespace dcih
