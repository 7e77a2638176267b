// Ranks of items held in registers by a workgroup, by one distribution into buckets in LDS
// instead of the eight digit passes of radix_core.h.
#pragma once

#include "common.h"

namespace dcih {
namespace {

constexpr int kBucketMost = 48;          // items one bucket may hold before the radix passes are the cheaper way

// Thread t holds the items t*IPT .. t*IPT+IPT-1 (STRIDED: t, t+NT, t+2*NT ...) of W (the rest are pads): k[r] the bits of a
// non-negative finite float, rp[r] a payload of 16 bits.  On return the item's place in the ascending
// order of (k, item number) is in rp[r]'s high half, the payload still in its low half; k is used up.
//
// x * scale (scale maps the largest x below 2^32) grows with x; its upper NBITS bits name a bucket,
// so every item's place is the number of items in the buckets below plus its rank inside its own,
// a couple of items.  One returning atomic counts and gives the item a slot; the buckets' starts come
// from one scan; the products are listed bucket by bucket, and an item's rank is the number of smaller
// words from its bucket's first on (words of later buckets are larger: no test for the bucket's end).
// Items whose product is another's too are put on the list `work` and ordered among themselves by
// `before(item number, item number)`, which is exact: at the end thread t has in (fix_rank, fix_payload)
// the place and payload of the t-th of them (fix_rank < 0: none), to be stored over what rp says.
//
// Bound by vector issue (about 100 instructions per item) and randomly addressed LDS operations (about
// nine), where eight radix passes take some 150 and 56; the operations' round trips overlap because
// four items at a time go through straight-line code, pads included (a pad adds nothing to some
// counter).  7021 items by 256 threads, two workgroups per CU: 43 us against 68 us by radix passes.
// Returns false, with k and rp undefined, if some bucket or the list `work` is too long.  SORTED (items numbered below 2^14): where the list is
// longer than some hundred items it is sorted instead, by (place, order_of(item number), item number), and `sorted` receives its length; the caller takes
// their places with sorted_place.  (Whole-number rows have many equal distances: 64 rows of 20480 in parts of 5120, 95 us by radix passes, 44 so.)
//
// LDS: `list` IPT * NT + 4 words, `cnt32` (1 << NBITS) / 2 + 1 words, `misc` 32 words, `work` work_cap <= NT
// 64-bit words.  All threads call this; it ends with reads of `list` under way (callers need a
// barrier before they reuse it).
struct NoOrder { __device__ uint32_t operator()(int) const { return 0; } };
constexpr int kSortedNumberBits = 14;
// The place of item i of the sorted list (its own word names it: the low bits), which begins with the place all items of its product share.
__device__ inline int sorted_place(const unsigned long long* work, int i) {
    const uint32_t place = (uint32_t)(work[i] >> (32 + kSortedNumberBits));
    int lo = 0, hi = i;      // the first of that place
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((uint32_t)(work[mid] >> (32 + kSortedNumberBits)) < place) lo = mid + 1; else hi = mid;
    }
    return (int)place + i - lo;
}
template <int NT, int IPT, int NBITS, bool STRIDED = false, bool SORTED = false, class Before, class Order = NoOrder>
__device__ inline bool lds_bucket_ranks(uint32_t (&k)[IPT], uint32_t (&rp)[IPT], int W, float scale,
                                        uint32_t* list, uint32_t* cnt32, uint32_t* misc, unsigned long long* work,
                                        int work_cap, int tid, int& fix_rank, uint32_t& fix_payload, Before before,
                                        Order order_of = Order(), int* sorted = nullptr) {
    static_assert(NT * IPT <= (1 << 15), "places of 16 bits");
    constexpr int kWords = (1 << NBITS) / 2, kPer = kWords / NT, kGroup = 4;
    const int lane = tid & 63, wave = tid >> 6;
    const uint16_t* cnt = reinterpret_cast<const uint16_t*>(cnt32);
    // items of this thread that are no pads; made opaque again for every pass, or the compiler keeps the
    // IPT comparisons with it as lane masks across all of them
    int own = STRIDED ? (W > tid ? (W - tid + NT - 1) / NT : 0) : min(max(W - tid * IPT, 0), IPT);
    auto number = [&](int r) { return STRIDED ? r * NT + tid : tid * IPT + r; };
    auto fresh = [&]() { asm volatile("" : "+v"(own)); };
#pragma unroll
    for (int w = 0; w < kPer; w++) cnt32[tid + w * NT] = 0;
    if (tid < 4) list[IPT * NT + tid] = 0xffffffffu;
    if (tid == 0) { cnt32[kWords] = (uint32_t)W; misc[16] = 0; misc[17] = 0; }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; r++) {
        const bool real = r < own;
        k[r] = real ? (uint32_t)(__builtin_bit_cast(float, k[r]) * scale) : 0u;
        const uint32_t b = k[r] >> (32 - NBITS), sh = (b & 1u) * 16u;
        const uint32_t old = atomicAdd(&cnt32[real ? b >> 1 : (uint32_t)tid], real ? 1u << sh : 0u);
        rp[r] = (rp[r] & 0xffffu) | (((old >> sh) & 0xffffu) << 16);
        if ((r & 7) == 7) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    {   // exclusive scan of the counters, and the longest bucket
        uint32_t v[kPer], sum = 0, most = 0;
#pragma unroll
        for (int w = 0; w < kPer; w++) {
            v[w] = cnt32[tid * kPer + w];
            const uint32_t lo = v[w] & 0xffffu, hi = v[w] >> 16;
            sum += lo + hi;
            most = max(most, max(lo, hi));
        }
        uint32_t incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = (uint32_t)__shfl_up((int)incl, o, 64);
            if (lane >= o) incl += t;
        }
        if (lane == 63) misc[wave] = incl;
        if (most > (uint32_t)kBucketMost) misc[16] = 1;
        __syncthreads();
        uint32_t run = incl - sum;
        for (int w2 = 0; w2 < wave; w2++) run += misc[w2];
#pragma unroll
        for (int w = 0; w < kPer; w++) {
            const uint32_t lo = v[w] & 0xffffu, hi = v[w] >> 16;
            cnt32[tid * kPer + w] = run | ((run + lo) << 16);
            run += lo + hi;
        }
    }
    __syncthreads();
    if (misc[16]) return false;
    fresh();
#pragma unroll
    for (int r = 0; r < IPT; r++) {
        // (a pad's word goes to its own place behind the items)
        const bool real = r < own;
        const uint32_t at = (uint32_t)cnt[k[r] >> (32 - NBITS)] + (rp[r] >> 16);
        list[real ? at : (uint32_t)number(r)] = real ? k[r] : 0xffffffffu;
        if ((r & 7) == 7) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
#pragma unroll
    for (int r0 = 0; r0 < IPT; r0 += kGroup) {
        uint32_t first[kGroup], len[kGroup], upto[kGroup];
#pragma unroll
        for (int g = 0; g < kGroup; g++) {
            if (r0 + g >= IPT) break;
            const uint32_t b = k[r0 + g] >> (32 - NBITS);
            first[g] = cnt[b];
            len[g] = cnt[b + 1];
        }
        uint32_t w[kGroup][4];
#pragma unroll
        for (int g = 0; g < kGroup; g++) {
            if (r0 + g >= IPT) break;
#pragma unroll
            for (int u = 0; u < 4; u++) w[g][u] = list[first[g] + u];
            len[g] -= first[g];
        }
        bool equal = false;
#pragma unroll
        for (int g = 0; g < kGroup; g++) {
            if (r0 + g >= IPT) break;
            const uint32_t mine = k[r0 + g];
            uint32_t below = 0;
            upto[g] = 0;
#pragma unroll
            for (int u = 0; u < 4; u++) { below += w[g][u] < mine ? 1u : 0u; upto[g] += w[g][u] <= mine ? 1u : 0u; }
            for (uint32_t p = 4; __any(p < len[g]); p += 4) {
                const uint32_t at = first[g] + min(p, len[g]);      // (past the bucket: words of later ones)
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t v = list[min(at + u, (uint32_t)(IPT * NT))];
                    below += v < mine ? 1u : 0u;
                    upto[g] += v <= mine ? 1u : 0u;
                }
            }
            rp[r0 + g] = (rp[r0 + g] & 0xffffu) | ((first[g] + below) << 16);
            upto[g] -= below;
            equal = equal || upto[g] > 1u;
        }
        if (equal) {
            fresh();
#pragma unroll
            for (int g = 0; g < kGroup; g++) {
                if (r0 + g >= IPT) break;
                if (upto[g] > 1u && r0 + g < own) {
                    const uint32_t slot = atomicAdd(&misc[17], 1u);
                    if (slot < (uint32_t)work_cap)
                        work[slot] = ((unsigned long long)rp[r0 + g] << 32) | (uint32_t)number(r0 + g);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    fix_rank = -1;
    fix_payload = 0;
    const int listed = (int)misc[17];
    if (listed > work_cap) return false;
    if constexpr (SORTED) {
        static_assert(NT * IPT <= (1 << kSortedNumberBits), "numbers of items");
        *sorted = listed > 256 ? listed : 0;
        if (listed > 256) {
            int np = NT;
            while (np < listed) np <<= 1;
            __syncthreads();
            for (int i = tid; i < np; i += NT) {
                const unsigned long long e = i < listed ? work[i] : ~0ull;
                work[i] = i < listed ? (e >> 48) << (32 + kSortedNumberBits) | (unsigned long long)order_of((int)(uint32_t)e) << kSortedNumberBits | (uint32_t)e : ~0ull;
            }
            __syncthreads();
            bitonic_sort_u64_by<NT, 4>(work, np, tid);
            __syncthreads();
            return true;
        }
    }
    if (tid < listed) {
        // (items of one product have the same place so far)
        const unsigned long long e = work[tid];
        const uint32_t place = (uint32_t)(e >> 48);
        fix_rank = (int)place;
        for (int o = 0; o < listed; o++) {
            const unsigned long long v = work[o];
            if (o != tid && (uint32_t)(v >> 48) == place && before((int)(uint32_t)v, (int)(uint32_t)e)) fix_rank++;
        }
        fix_payload = (uint32_t)(e >> 32) & 0xffffu;
    }
    return true;
}

}  // namespace
}  // namespace dcih
