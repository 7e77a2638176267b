// The k nearest of all rows of each query, k up to kNearestMaxK: what a query's answer is where no partition stops
// early (exhaustive.hip says when).  Lower bounds of all distances come from products on the matrix cores, and the distances
// themselves, formed and rounded as exact_dists_kernel forms them, only of the rows whose bound is within the k-th of
// them: the results are the same to the bit.
// (A distance of every pair costs three vector instructions an element.)
//
// The bound.  Rows and queries less a common centre are split into two 16-bit floats of eight bits each, x' = h + l + r with
// |r| <= 2^-18 |x'|, and x'.q' taken as h.h + h.l + l.h: what is left out is at most 2^-16 |x'||q'|, and every addition is off by
// 2^-23 of what limits a partial sum or less.  These 16-bit floats have a float's range, so no scale has to be found first; the split instead of
// one float keeps rows apart that lie far from the centre and close together.  The centre, the middle of three rows in every
// column, needs no pass over the rows either.
#include "common.h"
#include "half_core.h"
#include "kernels.h"

namespace dcih {

namespace {

typedef __bf16 v2b __attribute__((ext_vector_type(2)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kNearestMaxK = 128, kNearestMaxDim = 4096;

// out[q][row] = a lower bound of || data[row] - query[q] ||, least[q][row / 32] = the smallest of 32 of them.  A workgroup of four wavefronts takes
// 64 RT rows and as many queries, splits both, 64 OCT columns at a time, into LDS in the order the matrix instructions take them,
// and each wavefront multiplies a quarter; the next columns are under way meanwhile.  The queries are the products' columns: a lane holds 16 rows
// of one query, their smallest is its own to find and four neighbours one store.  Bound by vector issue (splitting an element
// is seven instructions, its 64 RT products three eighths of one each), below 500 tiles by what precedes and follows the products.
// (500 queries, 3000 rows of 100: 11 us, 20 with one 16-bit float an element, the scale and centre from a sample; distances of all 19.)
template <int RT, int OCT, bool OCTETS>
__global__ __launch_bounds__(kPackThreads, 2) void bound_rows_kernel(const float* __restrict__ data, int64_t N, int dim,
                                                                  const float* __restrict__ query, int nq, float* __restrict__ out,
                                                                  float* __restrict__ least, uint32_t* __restrict__ left) {
    constexpr int T = 64 * RT, kGroups = 2 * T / 32;            // groups of eight rows or queries per wavefront
    constexpr int kColumns = 64 * OCT, kSteps = kColumns / kStep;
    constexpr int kHalf = 4 * RT * kSteps * 64;
    extern __shared__ __align__(16) unsigned char smem[];
    const int width = (dim + kColumns - 1) / kColumns * kColumns;
    v8b* s_high = reinterpret_cast<v8b*>(smem);                 // [4 RT tiles of 32][kSteps][64]
    v8b* s_low = s_high + kHalf;
    float* s_sq = reinterpret_cast<float*>(s_low + kHalf);      // [2 T]
    float* s_ulp = s_sq + 2 * T;                                // [2 T]
    float* s_centre = s_ulp + 2 * T;                            // [width]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (left)      // what the kernels below take as cleared: the length of the list of queries, and their counters
        for (int e = (int)blockIdx.x * kPackThreads + tid; e <= nq; e += (int)gridDim.x * kPackThreads) left[e ? nq + e : 0] = 0;
    // Tiles in order, all queries' of some rows first, an eighth of the order to each XCD (workgroups go round them): its L2 then reads
    // an eighth of the rows.
    const uint32_t tile = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8, q_tiles = ((uint32_t)nq + T - 1) / T;
    const int64_t row0 = (int64_t)(tile / q_tiles) * T;
    const int q0 = (int)(tile % q_tiles) * T;
    if (row0 >= N) return;
    float next[kGroups][OCT][8];
    auto read = [&](int k0) {
#pragma unroll
        for (int g = 0; g < kGroups; g++) {
            const int r = (g * 4 + wave) * 8 + (lane & 7);      // (the first half are rows, in every wavefront)
            const float* x = g < kGroups / 2 ? data + min(row0 + r, N - 1) * dim : query + (int64_t)min(q0 + r - T, nq - 1) * dim;
#pragma unroll
            for (int c = 0; c < OCT; c++) load_octet<OCTETS>(x, dim, k0 + c * 64 + (lane >> 3) * 8, next[g][c]);
        }
    };
    read(0);
    for (int j = tid; j < width; j += kPackThreads) {
        const float* x = data + min(j, dim - 1);
        const float c = __builtin_amdgcn_fmed3f(x[N / 6 * dim], x[N / 2 * dim], x[(N - 1 - N / 6) * dim]);
        s_centre[j] = j < dim && fabsf(c) < 3e38f ? c : 0.0f;
    }
    float sq[kGroups] = {};
    v16f acc[RT][RT], cross[RT][RT];
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
        for (int b = 0; b < RT; b++) acc[a][b] = cross[a][b] = v16f{};
    const int wq = wave >> 1, wr = wave & 1;
    lds_barrier();
    for (int k0 = 0; k0 < width; k0 += kColumns) {
#pragma unroll
        for (int c = 0; c < OCT; c++) {
            const int o = c * 8 + (lane >> 3);
            float centre[8];
#pragma unroll
            for (int i = 0; i < 8; i++) centre[i] = s_centre[k0 + o * 8 + i];
#pragma unroll
            for (int g = 0; g < kGroups; g++) {
                const int r = (g * 4 + wave) * 8 + (lane & 7);
                if (k0 + c * 64 + 64 > dim) place_octet<OCTETS>(dim, k0 + o * 8, next[g][c]);
                v8b high, low;
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    const v2f x = {next[g][c][i] - centre[i], next[g][c][i + 1] - centre[i + 1]};
                    const v2b h = __builtin_convertvector(x, v2b);
                    const v2f back = __builtin_convertvector(h, v2f), off = {x.x - back.x, x.y - back.y};
                    const v2b l = __builtin_convertvector(off, v2b);
                    high[i] = h[0]; high[i + 1] = h[1];
                    low[i] = l[0]; low[i + 1] = l[1];
                    sq[g] = __builtin_fmaf(x.x, x.x, sq[g]);
                    sq[g] = __builtin_fmaf(x.y, x.y, sq[g]);
                }
                const int at = ((r >> 5) * kSteps + (o >> 1)) * 64 + (o & 1) * 32 + (r & 31);
                s_high[at] = high;
                s_low[at] = low;
            }
        }
        lds_barrier();
        read(min(k0 + kColumns, width - kColumns));
#pragma unroll
        for (int s = 0; s < kSteps; s++) {
            v8b xh[RT], xl[RT], qh[RT], ql[RT];
#pragma unroll
            for (int b = 0; b < RT; b++) {
                const int at = ((wr * RT + b) * kSteps + s) * 64 + lane;
                xh[b] = s_high[at]; xl[b] = s_low[at];
            }
#pragma unroll
            for (int a = 0; a < RT; a++) {
                const int at = ((2 * RT + wq * RT + a) * kSteps + s) * 64 + lane;
                qh[a] = s_high[at]; ql[a] = s_low[at];
            }
#pragma unroll
            for (int a = 0; a < RT; a++)
#pragma unroll
                for (int b = 0; b < RT; b++) {
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh[b], qh[a], acc[a][b], 0, 0, 0);
                    cross[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xl[b], qh[a], cross[a][b], 0, 0, 0);
                    cross[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh[b], ql[a], cross[a][b], 0, 0, 0);
                }
        }
        lds_barrier();
    }
    // Of a row or query: its squared length, less what (|x|^2 + |q|^2, of which 2 |x||q| is at most the whole) times the error of the
    // product is: its additions, twice 2^-23 each at most with those of the squared lengths, and what the split left out.  Minus infinity where
    // a sum may pass the largest float: nothing is known then.  And what the subtraction of the centre may be off by, an ulp.
    const float sum_error = 1.6f * sum_error_of(width) + 1.1f * 0x1p-16f, factor = distance_factor(dim) * 0.999999f;
#pragma unroll
    for (int g = 0; g < kGroups; g++) {
        float s2 = sq[g];
        s2 += lane_xor<32>(s2); s2 += lane_xor<16>(s2); s2 += lane_xor<8>(s2);
        if (lane < 8) {
            const int r = (g * 4 + wave) * 8 + lane;
            s_sq[r] = s2 < 1e36f ? s2 - s2 * sum_error : -__builtin_inff();
            s_ulp[r] = sqrtf(s2) * 0x1p-22f;
        }
    }
    __syncthreads();
    const int64_t groups = (N + 31) / 32;
    const int half = lane >> 5;
#pragma unroll
    for (int b = 0; b < RT; b++) {
        const int r0 = (wr * RT + b) * kTile + half * 4;        // the lane's rows: four from here, and from eight on, ...
        const int64_t row = row0 + r0;
#pragma unroll
        for (int a = 0; a < RT; a++) {
            const int at = (wq * RT + a) * kTile + (lane & 31), q = q0 + at;
            const float y = s_sq[T + at], ey = s_ulp[T + at];
            float* to = out + (int64_t)q * N + row;
            uint32_t low = kInf;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const v4f x = *reinterpret_cast<const v4f*>(s_sq + r0 + i * 8), ex = *reinterpret_cast<const v4f*>(s_ulp + r0 + i * 8);
                v4f d;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float d2 = __builtin_fmaf(-2.0f, acc[a][b][i * 4 + j] + cross[a][b][i * 4 + j], x[j] + y);
                    float v = __builtin_fmaf(__builtin_amdgcn_sqrtf(fmaxf(d2, 0.0f)), factor, -(ex[j] + ey));
                    v = v > 1e-14f ? v : 0.0f;      // (squares below the smallest float count as nothing in the distances)
                    if (row + i * 8 + j < N) low = min(low, __builtin_bit_cast(uint32_t, v));
                    d[j] = v;
                }
                if (q < nq) {
                    if (row + i * 8 + 4 <= N) *reinterpret_cast<v4f_any*>(to + i * 8) = d;
                    else
#pragma unroll
                        for (int j = 0; j < 3; j++) if (row + i * 8 + j < N) to[i * 8 + j] = d[j];
                }
            }
            low = min(low, lane_xor<32>(low));
            if (half == 0 && q < nq && row < N) least[(int64_t)q * groups + row / 32] = __builtin_bit_cast(float, low);
        }
    }
}

// sum + (x - q)^2, every step rounded.  The operands stand as they do in exact_dists_kernel: which NaN comes out of two, and with which
// sign, depends on their order, and the sign decides where its row is sorted.
__device__ __forceinline__ float add_square(float sum, float x, float q) {
    float d, out;
    asm("v_subrev_f32_e32 %0, %1, %2" : "=v"(d) : "v"(q), "v"(x));
    asm("v_mul_f32_e32 %0, %1, %1" : "=v"(d) : "v"(d));
    asm("v_add_f32_e32 %0, %1, %2" : "=v"(out) : "v"(d), "v"(sum));
    return out;
}

constexpr int kCap = 1024, kGroupCap = 1024, kPatch = 2304;      // (floats of rows per wavefront at a time)
// The distances of entries [from, to) of a list of row numbers, by a whole workgroup.  A wavefront takes 8 to 64 rows, few where there are few, and
// 256 to 32 columns of them at a time through LDS (`mine`: kPatch floats of its own), the next ones' reads under way; then each lane adds up its own row's.
__device__ __forceinline__ void list_distances(unsigned long long* buf, int from, int to, float* mine, const float* s_q, const float* __restrict__ data,
                                               int dim, int wave, int lane) {
    const int quarter = (to - from + 3) / 4, wide = quarter > 32 ? 3 : quarter > 16 ? 4 : quarter > 8 ? 5 : 6;
    const int per = 512 >> wide, columns = 4 << wide, pitch = columns + 4;
    const int kq = (lane & ((1 << wide) - 1)) * 4, r_in = lane >> wide, r_step = 64 >> wide;
    for (int g0 = from + wave * per; g0 < to; g0 += 4 * per) {
        const int count = min(per, to - g0), loads = (count + r_step - 1) / r_step;
        const float* x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = data + (int64_t)(uint32_t)buf[g0 + min(i * r_step + r_in, count - 1)] * dim;
        v4f pre[8];
        auto fetch = [&](int k0) {      // (past the row's end: its last 16 bytes)
#pragma unroll
            for (int i = 0; i < 8; i++) if (i < loads) pre[i] = *reinterpret_cast<const v4f_any*>(x[i] + min(k0 + kq, dim - 4));
        };
        fetch(0);
        float sum = 0.0f;
        for (int k0 = 0; k0 < dim; k0 += columns) {
            __builtin_amdgcn_wave_barrier();
            const int col = min(k0 + kq, dim - 4) - k0;     // (a row's last quad may begin before its place, its head is then there already)
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (i < loads) {
                    float* t = mine + (i * r_step + r_in) * pitch + col;
                    if (k0 + kq + 4 <= dim) {
                        *reinterpret_cast<v4f*>(t) = pre[i];
                    } else {
                        if (col >= 0) t[0] = pre[i].x;
                        if (col >= -1) t[1] = pre[i].y;
                        if (col >= -2) t[2] = pre[i].z;
                        if (col >= -3) t[3] = pre[i].w;
                    }
                }
            if (k0 + columns < dim) fetch(k0 + columns);
            __builtin_amdgcn_wave_barrier();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const float* t = mine + min(lane, per - 1) * pitch;
            const int kc = min(columns, dim - k0);
            int kk = 0;
#pragma unroll 4
            for (; kk + 4 <= kc; kk += 4) {
                const v4f v = *reinterpret_cast<const v4f*>(t + kk), y = *reinterpret_cast<const v4f*>(s_q + k0 + kk);
                sum = add_square(sum, v.x, y.x);
                sum = add_square(sum, v.y, y.y);
                sum = add_square(sum, v.z, y.z);
                sum = add_square(sum, v.w, y.w);
            }
            for (; kk < kc; kk++) sum = add_square(sum, t[kk], s_q[k0 + kk]);
        }
        if (lane < count)      // (the square root: as in exact_dists_kernel)
            buf[g0 + lane] = ((unsigned long long)__builtin_bit_cast(uint32_t, (float)sqrt((double)sum)) << 32) | (uint32_t)buf[g0 + lane];
    }
}
// One query per workgroup.  The rows whose bound is among the k smallest, and some further ones, are listed, their distances
// formed, and the k-th of these says which other rows have to be listed too: hardly ever any.  Bounds are read only of groups of 32 rows
// whose smallest one counts.  More than the lists take (rows that cannot be told apart, or whose squares no float holds): all rows, in tables of
// fewer than kAloneRows here, else by query_listed (exhaustive.hip).  Bound by the five reads that wait for each other (500 queries, 3000 rows: 9 us).
// (500 queries, one of them not finite, 3000 rows of 100: 118 us with a sort for every 256 rows, 94 now, 29 from all distances.)
constexpr int kAloneRows = 8192;
__global__ __launch_bounds__(kPackThreads) void nearest_rows_kernel(const float* __restrict__ bounds, const float* __restrict__ least,
                                                                    const float* __restrict__ data, int64_t N,
                                                                    int dim, const float* __restrict__ query, int k, int float_ids,
                                                                    int32_t* __restrict__ out_ids, float* __restrict__ out_dists,
                                                                    uint32_t* __restrict__ left) {
    __shared__ unsigned long long buf[kCap];
    __shared__ __align__(16) float patch[4][kPatch];
    __shared__ uint32_t s_count, s_groups, s_limit;
    extern __shared__ __align__(16) float s_q[];                // [dim rounded up to 4]
    uint32_t* s_group = reinterpret_cast<uint32_t*>(patch[0]);  // [kGroupCap]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t groups = (N + 31) / 32;
    const float* row = bounds + (int64_t)blockIdx.x * N;
    const float* group_least = least + (int64_t)blockIdx.x * groups;
    const float* q = query + (int64_t)blockIdx.x * dim;
    uint32_t mine_least = 0xffffffffu;      // (bounds are not negative: their bits order as they do)
    float first[2];                         // kept for the second look at them
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int64_t g = i * kPackThreads + tid;
        first[i] = g < groups ? group_least[g] : __builtin_inff();
        mine_least = min(mine_least, g < groups ? __builtin_bit_cast(uint32_t, first[i]) : 0xffffffffu);
    }
#pragma unroll 4
    for (int64_t g = 2 * kPackThreads + tid; g < groups; g += kPackThreads) mine_least = min(mine_least, __builtin_bit_cast(uint32_t, group_least[g]));
    for (int j = tid; j < dim; j += kPackThreads) s_q[j] = q[j];
    if (tid == 0) s_count = 0;
    buf[tid] = (unsigned long long)mine_least << 32;
    // the k-th smallest of the threads' smallest is at least the k-th smallest of all (there are 2 k groups or more)
    if (k <= 32) {
        __syncthreads();
        if (wave == 0) {      // (of four threads' smallest: as good where there are few, a sort of one wavefront)
            unsigned long long v[1] = {groups <= 64 ? buf[lane] : min(min(buf[lane], buf[64 + lane]), min(buf[128 + lane], buf[192 + lane]))};
            wave_sort_u64(v, lane);
            if (lane == k - 1) s_limit = (uint32_t)(v[0] >> 32);
        }
    } else {
        bitonic_sort_u64_by256(buf, kPackThreads);
        if (tid == 0) s_limit = (uint32_t)(buf[k - 1] >> 32);
    }
    __syncthreads();
    const float listed = __builtin_bit_cast(float, s_limit) * 1.003f;      // (at least k groups: finite)
    auto list = [&](float above, float upto) {                  // appends the rows with a bound in (above, upto]; false: too many groups
        __syncthreads();
        if (tid == 0) s_groups = 0;
        __syncthreads();
        const auto take = [&](int64_t g) {
            const uint32_t slot = atomicAdd(&s_groups, 1u);
            if (slot < (uint32_t)kGroupCap) s_group[slot] = (uint32_t)g;
        };
#pragma unroll
        for (int i = 0; i < 2; i++)
            if (i * kPackThreads + tid < groups && !(first[i] > upto)) take(i * kPackThreads + tid);
#pragma unroll 4
        for (int64_t g = 2 * kPackThreads + tid; g < groups; g += kPackThreads)
            if (!(group_least[g] > upto)) take(g);
        __syncthreads();
        const int n = (int)s_groups;
        if (n > kGroupCap) return false;
#pragma unroll 2
        for (int i = tid >> 5; i < n; i += kPackThreads / 32) {
            const int64_t j = (int64_t)s_group[i] * 32 + (tid & 31);
            const float b = j < N ? row[j] : 0.0f;
            if (j < N && b > above && !(b > upto)) {
                const uint32_t slot = atomicAdd(&s_count, 1u);
                if (slot < (uint32_t)kCap) buf[slot] = (uint32_t)j;
            }
        }
        __syncthreads();
        return s_count <= (uint32_t)kCap;
    };
    auto distances = [&](int from, int to) {
        list_distances(buf, from, to, patch[wave], s_q, data, dim, wave, lane);
        __syncthreads();
    };
    auto sort = [&](int count) {
        int np = kWave;
        while (np < count) np <<= 1;
        for (int j = count + tid; j < np; j += kPackThreads) buf[j] = ~0ull;
        __syncthreads();
        if (np == kWave) {
            if (wave == 0) {
                unsigned long long v[1] = {buf[lane]};
                wave_sort_u64(v, lane);
                buf[lane] = v[0];
            }
            __syncthreads();
        } else if (np == 128) {
            bitonic_sort_u64(buf, np);
        } else {
            bitonic_sort_u64_by256(buf, np);
        }
    };
    bool fits = list(-1.0f, listed);      // (the same for all threads, as what follows)
    if (fits) {
        const int count = (int)s_count;
        distances(0, count);
        sort(count);
        const float kth = __builtin_bit_cast(float, (uint32_t)(buf[k - 1] >> 32));
        if (!(kth <= listed)) {
            __syncthreads();      // (the sorted entries stay, more are appended)
            fits = list(listed, kth);
            const int more = (int)s_count;
            if (fits && more > count) {
                distances(count, more);
                sort(more);
            }
        }
    }
    if (!fits) {
        if (N >= kAloneRows) {
            if (tid == 0) left[1 + atomicAdd(&left[0], 1u)] = blockIdx.x;
            return;
        }
        keep_smallest(buf, s_count, N, k, [&](int64_t first, int n) {
            buf[kKeepAt + tid] = (unsigned long long)(uint32_t)(first + tid);
            __syncthreads();
            list_distances(buf, kKeepAt, kKeepAt + n, patch[wave], s_q, data, dim, wave, lane);
        });
    }
    for (int j = tid; j < k; j += kPackThreads) {
        const unsigned long long e = buf[j];
        const int32_t id = (int32_t)(uint32_t)e;
        out_ids[(int64_t)blockIdx.x * k + j] = float_ids ? __builtin_bit_cast(int32_t, (float)id) : id;
        out_dists[(int64_t)blockIdx.x * k + j] = __builtin_bit_cast(float, (uint32_t)(e >> 32));
    }
}

template <int RT, int OCT, bool OCTETS>
int launch_bounds(const float* data, int64_t N, int dim, const float* query, int nq, float* out, float* least, uint32_t* left, hipStream_t s) {
    constexpr int T = 64 * RT, columns = 64 * OCT;
    const size_t lds = (size_t)2 * 2 * T * columns * 2 + 2 * 2 * T * 4 + (size_t)((dim + columns - 1) / columns * columns) * 4;
    static DeviceOnce once;
    const int rc = once.run([]() -> int {
        DCIH_HIP(hipFuncSetAttribute((const void*)bound_rows_kernel<RT, OCT, OCTETS>, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024));
        return 0;
    });
    if (rc) return rc;
    const int64_t tiles = ((N + T - 1) / T) * ((nq + T - 1) / T);
    hipLaunchKernelGGL((bound_rows_kernel<RT, OCT, OCTETS>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(kPackThreads), lds, s,
                       data, N, dim, query, nq, out, least, left);
    DCIH_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// (64 rows and more for each result: twice as many groups of 32 as results, or most groups are looked into)
bool nearest_supported(int64_t N, int dim, int k) {
    return k <= kNearestMaxK && dim >= 8 && dim <= kNearestMaxDim && N >= 64 * (int64_t)k && N >= 1024;
}
// Whether that is faster than all distances and a selection from them.  Few rows: those are a kernel of a few microseconds, until the
// distances take as long as a second kernel's start (rows x dim, queries, all distances / this, us: 3000 x 100, 64: 15 / 17, 256: 22 / 17;
// 1500 x 64 never gains, 4096: 59 / 64).  Many rows: one query gains nothing from a tile of 64 (60000 x 300, 4: 41 / 46, 16: 53 / 46,
// 256: 637 / 75; 200000 x 64, 16: 42 / 53, 64: 102 / 60; 10000 x 32, 1: 15 / 13), of short rows fewer still (100000 x 16, 32: 28 / 32, 64:
// 38 / 34).  Long rows: few workgroups, one after another through the columns, wait longer than all distances take, until there are some
// dozens of tiles (2048 x 960, 48: 44 / 55, 128: 68 / 56; 8192 x 300, 4: 24 / 26, 16: 28 / 26).
// More results than the sort of one wavefront takes need more work to pay for theirs (8500 x 900, 128 results, 12: 70 / 108; 45000 x 64, 64, 24: 27 / 30),
// many queries rows that cost more than their own sorts (2500 x 16, 36, 4000: 55 / 83), and large tables a third launch's time.  (9213 shapes, 2100 to
// 150000 rows of 16 to 900, 10 to 128 results: by a rule that does not look at k 692 took more than 2 % longer than all distances, the worst half as long
// again; by this one 70, the worst 18 %.)
// A thousand million products pay for two dozen queries' tiles whatever the rest is (150000 x 300, 64, 36: all distances 389, 99; 87722 x 772, 96, 36: 378,
// 166; of the same shapes none that takes longer is added, of fewer queries some: 70000 x 900, 128, 16: 146 / 199).
bool nearest_pays(int64_t N, int dim, int k, int nq) {
    const bool many = k >= 32;
    const double pairs = (double)N * (double)nq, work = pairs * (double)dim;
    if (N < kAloneRows)
        return N >= 2048 && (double)N * dim >= (many ? 2e5 : 8e4) && pairs >= (many ? 3.75e5 : 2.5e5) && work >= (many ? 9e7 : 6e7);
    if (nq >= 24 && work >= 1e9) return true;
    return (double)nq * (dim < 64 ? 2048.0 : 4096.0) >= (many ? 2.0 : 1.0) * (double)N && work >= (many ? 8e7 : 2e7) &&
           (dim <= 100 || pairs >= (many ? 2e5 : 1e5)) && (dim <= 600 || pairs >= (many ? 8e5 : 4e5));
}
size_t nearest_least_bytes(int64_t N, int nq) { return (size_t)nq * (size_t)((N + 31) / 32) * 4; }
size_t nearest_left_bytes(int nq) { return (2 * (size_t)nq + 1) * 4; }

int query_nearest(const QueryArgs& a, int q0, int nq, float* d_bounds, float* d_least, uint32_t* d_left, hipStream_t s, bool& leaves) {
    const float* query = a.query + (int64_t)q0 * a.dim;
    leaves = a.N >= kAloneRows;
    uint32_t* left = leaves ? d_left : nullptr;
    const bool octets = a.dim % 8 == 0, large = ((a.N + 127) / 128) * ((nq + 127) / 128) >= 512;
    const auto bounds = large ? (octets ? launch_bounds<2, 1, true> : launch_bounds<2, 1, false>)
                      : a.dim > 64 ? (octets ? launch_bounds<1, 2, true> : launch_bounds<1, 2, false>)
                                   : octets ? launch_bounds<1, 1, true> : launch_bounds<1, 1, false>;
    const int rc = bounds(a.data, a.N, a.dim, query, nq, d_bounds, d_least, left, s);
    if (rc) return rc;
    hipLaunchKernelGGL(nearest_rows_kernel, dim3((unsigned)nq), dim3(kPackThreads), (size_t)((a.dim + 3) & ~3) * 4, s, d_bounds, d_least, a.data, a.N,
                       a.dim, query, a.k, a.float_ids, a.out_ids + (int64_t)q0 * a.k, a.out_dists + (int64_t)q0 * a.k, left);
    DCIH_HIP(hipGetLastError());
    return 0;
}

}  // namespace dcih
