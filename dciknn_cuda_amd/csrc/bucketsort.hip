// Segmented sort of one slice per workgroup by ONE distribution into buckets in LDS and a repair of what the buckets leave unsorted,
// where the radix kernels of segsort.hip need eight digit passes.
//
// A monotone map takes every key to one of about as many buckets as the slice has points, a point or two to a bucket: linear inside each of
// kSegs pieces of the keys' range, whose shares of the buckets are their shares of the points, so that bell-shaped, clustered and lopsided
// projections come out as even as uniform ones.  One returning atomic per key counts its bucket and numbers it there, one scan gives the
// buckets' starts, and keys and ids go to start + number.  The list that this leaves is ordered but for points of one bucket, so a point's
// place is off by less than the fullest bucket holds, and is set right by counting: every thread holds a run of the list and its
// neighbourhood in registers and compares each pair within that distance once.  Equal keys keep the list's order there and are put in the
// order of their ids when the keys are written out.
//
// Where most points share a piece, because others lie far out, the pieces' widths grow with the distance from the median instead.
//
// A slice whose fullest bucket holds more than kMostInBucket points (keys that repeat), or whose keys are not all
// finite, is left alone and marked by an id of -1 in its first place: the caller has the radix kernels sort what is marked.
//
// Bound by LDS and vector issue, a third to two thirds as fast as memory alone would allow: a key costs six randomly addressed LDS operations
// (the radix kernels 44 to 58) and about 80 instructions, its slice is read once and written once.  20M Gaussian keys, us, by digits and so: slices of 277 points
// 526, 70; 1111 285, 70; 4000 229, 72; 8000 240, 81; 10000 220, 83; 13000 218, 98; 17142 246, 103; 25000 304, 127.  Slices that are left cost
// the attempt on top: rows that are there 32 times each, one after the other (all slices left), slices of 100 points 256, 498; 277 531, 427; 1111 281, 324;
// 2000 203, 334; 4000 220, 363; 8000 231, 372; 17142 249, 367; 25000 292, 468.  20 different keys in 17142 237, 265.
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace dcih {

namespace {

constexpr int kMostInBucket = 16;

template <int NT, int IPT>
struct BucketShape {
    static constexpr int kCap = NT * IPT;                   // points
    static constexpr int kWords = (IPT - 1) / 2;            // counters' words per thread, two counters each
    static constexpr int kBuckets = 2 * kWords * NT;
    static constexpr int kSegs = NT >= 512 ? 512 : (NT >= 256 ? 256 : 128);
    static constexpr int kWaves = NT / kWave;
    // LDS words: pads and keys, then counters (later the ids), the pieces of the map, scratch
    static constexpr int kKeys = kMostInBucket, kCounters = kKeys + kCap + kMostInBucket;
    static constexpr int kMap = (kCounters + (kCap + 1) / 2 + 3) & ~3;
    static constexpr int kScratch = kMap + 2 * kSegs;
    static constexpr int kLdsWords = kScratch + 4 * kWaves + 8;
    static_assert(2 * kWords * 2 <= IPT * 2, "the counters lie in the ids' room");
};

__device__ __forceinline__ float wave_min_f(float v) {
    v = fminf(v, lane_xor<32>(v)); v = fminf(v, lane_xor<16>(v)); v = fminf(v, lane_xor<8>(v));
    v = fminf(v, lane_xor<4>(v)); v = fminf(v, lane_xor<2>(v)); return fminf(v, lane_xor<1>(v));
}
__device__ __forceinline__ float wave_max_f(float v) {
    v = fmaxf(v, lane_xor<32>(v)); v = fmaxf(v, lane_xor<16>(v)); v = fmaxf(v, lane_xor<8>(v));
    v = fmaxf(v, lane_xor<4>(v)); v = fmaxf(v, lane_xor<2>(v)); return fmaxf(v, lane_xor<1>(v));
}

// A thread's run of the list, keys k[0, IPT) at places first .., compared with all within the distances d .. D below `most`: lo[e] is the key
// at place first - 1 - e, hi[e] at first + IPT + e.  move[r] becomes the distance of key r from its place to where it belongs.
template <int d, int IPT, int D>
__device__ __forceinline__ void repair(const uint32_t* list, int first, const uint32_t (&k)[IPT], uint32_t (&lo)[D], uint32_t (&hi)[D],
                                       int (&move)[IPT], int most) {
    if (d >= most) return;                                   // (the same for all threads)
    lo[d - 1] = list[first - d];
    hi[d - 1] = list[first + IPT + d - 1];
#pragma unroll
    for (int r = 0; r < IPT; r++) {
        if (r + d < IPT) {
            const bool c = k[r + d] < k[r];
            move[r] += c ? 1 : 0;
            move[r + d] -= c ? 1 : 0;
        } else {
            move[r] += hi[r + d - IPT] < k[r] ? 1 : 0;
        }
        if (r < d) move[r] -= k[r] < lo[d - r - 1] ? 1 : 0;
    }
    if constexpr (d < D) repair<d + 1, IPT, D>(list, first, k, lo, hi, move, most);
}

template <int NT, int IPT>
__global__ __launch_bounds__(NT, NT == 512 ? 4 : 1) void bucketsort_kernel(const float* __restrict__ keys, int64_t kstride, int64_t n_all, int64_t ppb, int B,
                                                        float* __restrict__ skeys, int32_t* __restrict__ sids, uint16_t* __restrict__ inv) {
    typedef BucketShape<NT, IPT> S;
    extern __shared__ __align__(16) uint32_t lds[];
    uint32_t* list = lds + S::kKeys;
    uint32_t* cnt32 = lds + S::kCounters;
    uint16_t* cnt = reinterpret_cast<uint16_t*>(cnt32);
    uint16_t* ids = cnt;
    float2* map = reinterpret_cast<float2*>(lds + S::kMap);
    uint32_t* hist = lds + S::kMap;                          // [kSegs], while the sample is counted
    uint32_t* scratch = lds + S::kScratch;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int b = (int)(blockIdx.x % B);
    const int64_t i = blockIdx.x / B, off = (int64_t)b * ppb, base = i * n_all + off;
    const int n = (int)min(n_all - off, ppb);
    if (n <= 0) return;
    const float* kin = keys + i * kstride + off;

    // ---- keys, all reads under way at once
    float x[IPT];
#pragma unroll
    for (int r = 0; r < IPT; r++) x[r] = kin[min(r * NT + tid, n - 1)];
#pragma unroll
    for (int w = 0; w < S::kWords; w++) cnt32[w * NT + tid] = 0;
    for (int s = tid; s < S::kSegs; s += NT) hist[s] = 0;
    if (tid < kMostInBucket) { lds[tid] = 0; list[S::kCap + tid] = 0xffffffffu; }
    float least = x[0], largest = x[0], odd = 0.0f;          // odd: NaN where a key is not finite
#pragma unroll
    for (int r = 0; r < IPT; r++) {
        x[r] += 0.0f;                                        // (-0.0 ties with +0.0 on the id)
        least = fminf(least, x[r]);
        largest = fmaxf(largest, x[r]);
        odd = __builtin_fmaf(x[r], 0.0f, odd);
    }
    least = wave_min_f(least);
    largest = wave_max_f(largest);
    odd = __any(odd != 0.0f) ? 1.0f : 0.0f;                  // (NaN differs from everything)
    float* f_scratch = reinterpret_cast<float*>(scratch);
    if (S::kWaves > 1 && lane == 0) { f_scratch[wave] = least; f_scratch[S::kWaves + wave] = largest; f_scratch[2 * S::kWaves + wave] = odd; }
    __syncthreads();
    if constexpr (S::kWaves > 1) {
#pragma unroll
        for (int w = 0; w < S::kWaves; w++) {
            least = fminf(least, f_scratch[w]);
            largest = fmaxf(largest, f_scratch[S::kWaves + w]);
            odd = fmaxf(odd, f_scratch[2 * S::kWaves + w]);
        }
    }
    const float range = largest - least;
    if (odd != 0.0f || !(range > 1e-30f && range < 1e38f)) {
        if (tid == 0) sids[base] = -1;
        return;
    }
    // ---- the map: a key's piece of the range and its place inside it, pieces of equal widths or (WIDE) of widths that grow with the distance
    // from the median, eight (four) to a factor of two.  Pieces, then the buckets of each: no more or less than its points' share.
    const float scale = (float)S::kSegs * 0.999999f / range;
    constexpr int kFine = S::kSegs == 512 ? 20 : (S::kSegs == 256 ? 21 : 21);      // bits of a float below a piece
    float median = 0.0f;
    uint32_t nearest = 0;                                    // float bits below which distances are not told apart
    auto piece_of = [&](auto wide, float v, float& inside) __attribute__((always_inline)) {
        if constexpr (decltype(wide)::value) {
            const float d = v - median;
            const uint32_t t = __builtin_bit_cast(uint32_t, d) & 0x7fffffffu;
            const int above = (int)(max(t, nearest) - nearest), g = d < 0.0f ? ~above : above;
            inside = (float)(g & ((1 << kFine) - 1)) * (1.0f / (float)(1 << kFine));
            return (uint32_t)(S::kSegs / 2 + (g >> kFine));
        } else {
            const float f = (v - least) * scale;
            inside = __builtin_amdgcn_fractf(f);
            return (uint32_t)f;
        }
    };
    // true where one piece holds most of the points
    auto make_map = [&](auto wide) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < IPT; r++) {
            // (straight-line code, so that the operations are under way together: a pad adds nothing, each to another word)
            const bool real = r * NT + tid < n;
            float inside;
            const uint32_t piece = piece_of(wide, x[r], inside);
            atomicAdd(&hist[real ? piece : (uint32_t)tid & (S::kSegs - 1)], real ? 1u : 0u);
        }
        __syncthreads();
        if (wave == 0) {
            constexpr int kPer = S::kSegs / kWave;           // pieces per lane, neighbours
            uint32_t c[kPer], sum = 0, most = 0;
#pragma unroll
            for (int u = 0; u < kPer; u++) { c[u] = hist[lane * kPer + u]; sum += c[u]; most = max(most, c[u]); }
            uint32_t before = wave_scan_u32(sum) - sum;
            const float per = (float)(S::kBuckets - 1) / (float)n;
            float2 e[kPer];
#pragma unroll
            for (int u = 0; u < kPer; u++) {
                const float from = floorf((float)before * per);
                before += c[u];
                e[u] = make_float2(from, floorf((float)before * per) - from);
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int u = 0; u < kPer; u++) map[lane * kPer + u] = e[u];
            if (lane == 0) f_scratch[3 * S::kWaves] = 0.0f;
            if (__any(most > (uint32_t)n / 2u)) f_scratch[3 * S::kWaves] = 1.0f;
        }
        __syncthreads();
        return f_scratch[3 * S::kWaves] != 0.0f;
    };
    // x's bucket << 16 | its number in the bucket
    uint32_t at[IPT];
    auto count = [&](auto wide) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < IPT; r++) {
            float inside;
            const float2 e = map[piece_of(wide, x[r], inside)];
            // (rounding keeps the order: what lies in a piece stays at or below the next one's first bucket)
            const uint32_t bucket = (uint32_t)__builtin_fmaf(inside, e.y, e.x);
            const uint32_t sh = (bucket & 1u) * 16u;
            const bool real = r * NT + tid < n;
            const uint32_t old = atomicAdd(&cnt32[real ? bucket >> 1 : (uint32_t)tid], real ? 1u << sh : 0u);
            at[r] = (bucket << 16) | ((old >> sh) & 0xffffu);
            if ((r & 7) == 7) __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (!make_map(std::false_type{})) {
        count(std::false_type{});
    } else {
        // most points share a piece, for others lie far out: pieces by the distance from the median of 64 points
        if (wave == 0) {
            unsigned long long v = f2ord(kin[(int)((uint32_t)lane * (uint32_t)n / kWave)] + 0.0f);
            bitonic_wave_steps<2, 1>(v, lane, kWave);
            if (lane == kWave / 2) f_scratch[0] = ord2f((uint32_t)v);
        }
        for (int s = tid; s < S::kSegs; s += NT) hist[s] = 0;
        __syncthreads();
        median = f_scratch[0];
        const uint32_t furthest = __builtin_bit_cast(uint32_t, fmaxf(largest - median, median - least));
        const uint32_t whole = (uint32_t)(S::kSegs / 2) << kFine;
        nearest = furthest >= whole ? furthest - whole + 1u : 0u;
        if (make_map(std::true_type{})) {
            if (tid == 0) sids[base] = -1;
            return;
        }
        count(std::true_type{});
    }
    __syncthreads();
    uint32_t fullest = 0;
    {
        uint32_t v[S::kWords], sum = 0;
#pragma unroll
        for (int w = 0; w < S::kWords; w++) {
            v[w] = cnt32[tid * S::kWords + w];
            const uint32_t p = v[w] & 0xffffu, q = v[w] >> 16;
            sum += p + q;
            fullest = max(fullest, max(p, q));
        }
        const uint32_t upto = wave_scan_u32(sum);
        fullest = (uint32_t)wave_max_i32((int)fullest);
        if (S::kWaves > 1 && lane == 63) { scratch[wave] = upto; scratch[S::kWaves + wave] = fullest; }
        __syncthreads();
        uint32_t run = upto - sum;
        if constexpr (S::kWaves > 1) {
#pragma unroll
            for (int w = 0; w < S::kWaves; w++) {
                run += w < wave ? scratch[w] : 0u;
                fullest = max(fullest, scratch[S::kWaves + w]);
            }
        }
#pragma unroll
        for (int w = 0; w < S::kWords; w++) {
            const uint32_t p = v[w] & 0xffffu, q = v[w] >> 16;
            cnt32[tid * S::kWords + w] = run | ((run + p) << 16);
            run += p + q;
        }
    }
    fullest = (uint32_t)__builtin_amdgcn_readfirstlane((int)fullest);
    if (fullest > (uint32_t)kMostInBucket) {
        if (tid == 0) sids[base] = -1;
        return;
    }
    __syncthreads();

    // ---- into the list
#pragma unroll
    for (int r = 0; r < IPT; r++) {
        const int j = r * NT + tid;
        const uint32_t place = j < n ? (uint32_t)cnt[at[r] >> 16] + (at[r] & 0xffffu) : (uint32_t)j;
        list[place] = j < n ? f2ord(x[r]) : 0xffffffffu;
        at[r] = place;
        if ((r & 7) == 7) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; r++) ids[at[r]] = (uint16_t)(r * NT + tid);
    __syncthreads();

    // ---- repaired
    {
        const int first = tid * IPT;
        uint32_t k[IPT], lo[kMostInBucket - 1], hi[kMostInBucket - 1];
        int move[IPT];
#pragma unroll
        for (int r = 0; r < IPT; r++) { k[r] = list[first + r]; move[r] = 0; }
        repair<1, IPT, kMostInBucket - 1>(list, first, k, lo, hi, move, (int)fullest);
        uint32_t id[IPT];
#pragma unroll
        for (int r = 0; r < IPT; r++) id[r] = ids[first + r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < IPT; r++) {
            list[first + r + move[r]] = k[r];
            ids[first + r + move[r]] = (uint16_t)id[r];
        }
    }
    __syncthreads();

    // ---- out: keys four at a time, equal ones' ids put in order; then ids; then the inverse permutation, turned round in the keys' room
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    for (int j = 4 * tid; j < n; j += 4 * NT) {
        const v4u k = *reinterpret_cast<const v4u*>(list + j);
        const uint32_t before = list[j - 1], behind = list[j + 4];
        const bool pairs = k.x == k.y || k.y == k.z || k.z == k.w || k.w == behind;
        if (pairs) {
            uint32_t prev = j > 0 ? before : 0u;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t own = list[j + e];
                if (own != prev && j + e < n) {              // a run may begin here
                    int end = j + e + 1;
                    while (end < n && list[end] == own) end++;
                    for (int p = j + e + 1; p < end; p++) {
                        const uint16_t v = ids[p];
                        int q = p;
                        for (; q > j + e && ids[q - 1] > v; q--) ids[q] = ids[q - 1];
                        ids[q] = v;
                    }
                }
                prev = own;
            }
        }
        const float f[4] = {ord2f(k.x), ord2f(k.y), ord2f(k.z), ord2f(k.w)};
        if (j + 4 <= n) {
            __builtin_memcpy(skeys + base + j, f, 16);
        } else {
#pragma unroll
            for (int e = 0; e < 3; e++) if (j + e < n) skeys[base + j + e] = f[e];
        }
    }
    __syncthreads();
    uint16_t* pos = reinterpret_cast<uint16_t*>(list);
    for (int j = 4 * tid; j < n; j += 4 * NT) {
        uint16_t p[4];
        __builtin_memcpy(p, ids + j, 8);
        const int32_t o = (int32_t)off;
        const int32_t g[4] = {o + p[0], o + p[1], o + p[2], o + p[3]};
        if (j + 4 <= n) {
            __builtin_memcpy(sids + base + j, g, 16);
#pragma unroll
            for (int e = 0; e < 4; e++) pos[p[e]] = (uint16_t)(j + e);
        } else {
#pragma unroll
            for (int e = 0; e < 3; e++) if (j + e < n) { sids[base + j + e] = g[e]; pos[p[e]] = (uint16_t)(j + e); }
        }
    }
    if (!inv) return;
    __syncthreads();
    for (int j = 4 * tid; j < n; j += 4 * NT) {
        uint16_t p[4];
        __builtin_memcpy(p, pos + j, 8);
        if (j + 4 <= n) {
            __builtin_memcpy(inv + base + j, p, 8);
        } else {
#pragma unroll
            for (int e = 0; e < 3; e++) if (j + e < n) inv[base + j + e] = p[e];
        }
    }
}

template <int NT, int IPT>
int launch(const float* d_keys, int64_t kstride, int num_indices, int64_t n, int64_t ppb, int B, float* d_skeys, int32_t* d_sids,
           uint16_t* d_inv, hipStream_t s) {
    constexpr int kLds = BucketShape<NT, IPT>::kLdsWords * 4;
    static DeviceOnce once;
    const int rc = once.run([]() -> int {
        DCIH_HIP(hipFuncSetAttribute((const void*)bucketsort_kernel<NT, IPT>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
        return 0;
    });
    if (rc) return rc;
    hipLaunchKernelGGL((bucketsort_kernel<NT, IPT>), dim3((unsigned)((int64_t)num_indices * B)), dim3(NT), kLds, s,
                       d_keys, kstride, n, ppb, B, d_skeys, d_sids, d_inv);
    DCIH_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// (Up to 64 points the bitonic sort of one wavefront is the whole work; above 25600 keys and ids do not fit a CU's LDS.)
bool bucketsort_supported(int64_t ppb) { return ppb > 64 && ppb <= 1024 * 25; }

int bucketsort(const float* d_keys, int64_t kstride, int num_indices, int64_t n, int64_t ppb, int B, float* d_skeys, int32_t* d_sids,
               uint16_t* d_inv, hipStream_t s) {
    // As many threads as keep about a dozen items each; 512 threads up to what lets two workgroups into a CU's LDS (9967 points: 83 us, 112 with
    // 1024 threads).  An odd number of items per thread keeps the reads of the list free of bank conflicts.
#define DCIH_BUCKETS(NT, IPT) \
    if (ppb <= (int64_t)(NT) * (IPT)) return launch<NT, IPT>(d_keys, kstride, num_indices, n, ppb, B, d_skeys, d_sids, d_inv, s)
    DCIH_BUCKETS(64, 5); DCIH_BUCKETS(64, 9); DCIH_BUCKETS(64, 13); DCIH_BUCKETS(64, 17); DCIH_BUCKETS(64, 21);
    DCIH_BUCKETS(256, 9); DCIH_BUCKETS(256, 13); DCIH_BUCKETS(256, 17);
    DCIH_BUCKETS(512, 13); DCIH_BUCKETS(512, 17); DCIH_BUCKETS(512, 21); DCIH_BUCKETS(512, 25);
    DCIH_BUCKETS(1024, 13); DCIH_BUCKETS(1024, 17); DCIH_BUCKETS(1024, 21); DCIH_BUCKETS(1024, 25);
#undef DCIH_BUCKETS
    return fail(-1, "bucketsort: slice too long");
}

}  // namespace dcih
