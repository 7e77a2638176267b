// 8-bit codes of the indexed rows and of a batch of queries, for the dense traversal's distance
// phase: a candidate row is read as dim bytes instead of 4 * dim, its distance is known from the
// codes within a proven margin, and only the few candidates within the margin of the k best are
// read whole (traverse_dense.hip).  Results do not depend on the codes.
//
// A row x is coded as c = round(x / s), s = max |x_j| / 127, one scale per row; its record is
//   { float s; float n2 = |s c|^2; 8 unused bytes; int8 c[dim], zeros to a multiple of 16 bytes
//     or, up to dim = 112, to one 128-byte line }.
// Per partition the largest |x - s c| and the largest n2 of its rows are kept (they bound the margin).
// A query q is coded in 15 bits, q ~ sq (128 hi + lo), two bytes per element:
//   { float sq; float n2; float e >= |q - sq (128 hi + lo)|; 4 unused bytes; int8 hi[..], lo[..] }.
#include "common.h"
#include "kernels.h"

namespace dcih {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_any __attribute__((aligned(4)));
constexpr int kThreads = 256;
constexpr int kQuads = 4;          // quads of a row per lane at most: 16 lanes take rows of up to 256 elements, 64 of up to 1024
constexpr int kRows = 8;           // rows one lane group codes

template <int LPR> __device__ inline float group_max(float v) {
    if constexpr (LPR == 64) { v = fmaxf(v, lane_xor<32>(v)); v = fmaxf(v, lane_xor<16>(v)); }
    v = fmaxf(v, lane_xor<8>(v)); v = fmaxf(v, lane_xor<4>(v)); v = fmaxf(v, lane_xor<2>(v)); v = fmaxf(v, lane_xor<1>(v));
    return v;
}
template <int LPR> __device__ inline float group_sum(float v) {
    if constexpr (LPR == 64) { v += lane_xor<32>(v); v += lane_xor<16>(v); }
    v += lane_xor<8>(v); v += lane_xor<4>(v); v += lane_xor<2>(v); v += lane_xor<1>(v);
    return v;
}

// A lane's elements of a row: quad q holds elements (q * LPR + sl) * 4 .. + 3, zeros past the end.
template <int LPR, int NQ> __device__ inline void load_quads(const float* x, int dim, int sl, float (&v)[NQ][4]) {
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int j = (q * LPR + sl) * 4;
        if (j + 4 <= dim) {
            const v4f t = *reinterpret_cast<const v4f_any*>(x + j);
            v[q][0] = t.x; v[q][1] = t.y; v[q][2] = t.z; v[q][3] = t.w;
        } else {
#pragma unroll
            for (int c = 0; c < 4; c++) v[q][c] = j + c < dim ? x[j + c] : 0.0f;
        }
    }
}

// Bound by memory: every row read once, its record written once.  A workgroup takes kRows consecutive rows
// per lane group and keeps the partition's bounds in registers meanwhile: one atomic per row and its
// division by ppb took thirty times that (666k rows of 96: 2.1 ms, now 67 us).
template <int LPR, int NQ>
__global__ __launch_bounds__(kThreads) void code_rows_kernel(const float* __restrict__ data, int64_t n, int dim,
                                                             int64_t ppb, unsigned char* __restrict__ recs, int rec_bytes,
                                                             uint32_t* __restrict__ bounds) {
    constexpr int kGroups = kThreads / LPR;
    __shared__ uint32_t s_e[kGroups], s_n2[kGroups], s_part[kGroups];
    const int sl = threadIdx.x & (LPR - 1), grp = threadIdx.x / LPR;
    const int64_t first = (int64_t)blockIdx.x * (kGroups * kRows);
    uint32_t part = (uint32_t)(first / ppb);
    int64_t part_end = ((int64_t)part + 1) * ppb;
    uint32_t most_e = 0, most_n2 = 0;       // of the rows of `part` so far (not negative: their bits order as they do)
    auto flush = [&](uint32_t p, uint32_t e, uint32_t n2) {
        if (e > 0) atomicMax(&bounds[2 * p], e);
        if (n2 > 0) atomicMax(&bounds[2 * p + 1], n2);
    };
    for (int i = 0; i < kRows; i++) {
        const int64_t row = first + i * kGroups + grp;
        if (row >= n) break;
        float v[NQ][4];
        load_quads<LPR, NQ>(data + row * dim, dim, sl, v);
        float most = 0.0f;
        bool finite = true;
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
            for (int c = 0; c < 4; c++) { most = fmaxf(most, fabsf(v[q][c])); finite = finite && fabsf(v[q][c]) < 3e38f; }
        most = group_max<LPR>(finite ? most : __builtin_inff());
        // (rows too large or too small for float32 squares are left without useful codes: an infinite error)
        const bool usable = most < 1e15f && (most > 1e-15f || most == 0.0f);
        const float s = usable ? most / 127.0f : 0.0f, inv = usable && most > 0.0f ? 127.0f / most : 0.0f;
        float err = 0.0f, sq = 0.0f;
        unsigned char* rec = recs + row * rec_bytes;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int j = (q * LPR + sl) * 4;
            uint32_t word = 0;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float code = fminf(127.0f, fmaxf(-127.0f, rintf(v[q][c] * inv)));
                const float d = __builtin_fmaf(-s, code, v[q][c]);
                err = __builtin_fmaf(d, d, err);
                sq = __builtin_fmaf(code, code, sq);
                word |= ((uint32_t)(int)code & 0xffu) << (8 * c);
            }
            if (j < rec_bytes - 16) *reinterpret_cast<uint32_t*>(rec + 16 + j) = word;
        }
        err = group_sum<LPR>(err);
        sq = group_sum<LPR>(sq);
        if (sl == 0) {
            const float n2 = (float)((double)s * (double)s * (double)sq);      // (the sum of squares of codes is exact)
            float4 h;
            h.x = s; h.y = n2; h.z = 0.0f; h.w = 0.0f;
            *reinterpret_cast<float4*>(rec) = h;
            const float e = usable ? sqrtf(err) * 1.001f + 1e-30f : __builtin_inff();
            if (row >= part_end) {
                flush(part, most_e, most_n2);
                do { part++; part_end += ppb; } while (row >= part_end);
                most_e = most_n2 = 0;
            }
            most_e = max(most_e, __builtin_bit_cast(uint32_t, e));
            most_n2 = max(most_n2, __builtin_bit_cast(uint32_t, n2));
        }
    }
    if (sl == 0) { s_e[grp] = most_e; s_n2[grp] = most_n2; s_part[grp] = part; }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t p = s_part[0], e = s_e[0], n2 = s_n2[0];
        for (int g = 1; g < kGroups; g++) {
            if (s_part[g] != p) { flush(p, e, n2); p = s_part[g]; e = n2 = 0; }
            e = max(e, s_e[g]);
            n2 = max(n2, s_n2[g]);
        }
        flush(p, e, n2);
    }
}

template <int LPR>
__global__ __launch_bounds__(kThreads) void code_queries_kernel(const float* __restrict__ query, int nq, int dim,
                                                                unsigned char* __restrict__ recs, int code_bytes) {
    const int sl = threadIdx.x & (LPR - 1);
    const int row = (int)(((int64_t)blockIdx.x * kThreads + threadIdx.x) / LPR);
    const bool in = row < nq;
    float v[kQuads][4];
    load_quads<LPR, kQuads>(query + (int64_t)min(row, nq - 1) * dim, dim, sl, v);
    float most = 0.0f;
    bool finite = true;
#pragma unroll
    for (int q = 0; q < kQuads; q++)
#pragma unroll
        for (int c = 0; c < 4; c++) { most = fmaxf(most, fabsf(v[q][c])); finite = finite && fabsf(v[q][c]) < 3e38f; }
    most = group_max<LPR>(finite ? most : __builtin_inff());
    const bool usable = most < 1e15f && (most > 1e-15f || most == 0.0f);
    const float s = usable ? most / 16256.0f : 0.0f, inv = usable && most > 0.0f ? 16256.0f / most : 0.0f;
    float err = 0.0f;
    double sq = 0.0;
    unsigned char* rec = recs + (int64_t)min(row, nq - 1) * (16 + 2 * code_bytes);
#pragma unroll
    for (int q = 0; q < kQuads; q++) {
        const int j = (q * LPR + sl) * 4;
        uint32_t wh = 0, wl = 0;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int code = (int)fminf(16256.0f, fmaxf(-16256.0f, rintf(v[q][c] * inv)));
            const int hi = (code + 64) >> 7, lo = code - 128 * hi;          // hi in [-127, 127], lo in [-64, 63]
            const float d = __builtin_fmaf(-s, (float)code, v[q][c]);
            err = __builtin_fmaf(d, d, err);
            sq += (double)code * (double)code;
            wh |= ((uint32_t)hi & 0xffu) << (8 * c);
            wl |= ((uint32_t)lo & 0xffu) << (8 * c);
        }
        if (in && j < code_bytes) {
            *reinterpret_cast<uint32_t*>(rec + 16 + j) = wh;
            *reinterpret_cast<uint32_t*>(rec + 16 + code_bytes + j) = wl;
        }
    }
    err = group_sum<LPR>(err);
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
    if (in && sl == 0) {
        float4 h;
        h.x = s; h.y = (float)((double)s * (double)s * sq); h.w = 0.0f;
        h.z = usable ? sqrtf(err) * 1.001f + 1e-30f : __builtin_inff();
        *reinterpret_cast<float4*>(rec) = h;
    }
}

}  // namespace

// Rows of fewer than 96 elements span at most three 128-byte lines: reading them whole costs less than
// their record, a longer list and the rows of what is kept (1111 candidates each, k = 50; 64 elements: 24 us of
// distances per item by whole rows, 48 by codes; 512 elements: 102 and 70).
bool rows8_supported(int dim) { return dim >= 96 && dim <= 1024; }
// (a record that fits one 128-byte line gets one to itself)
int rows8_record_bytes(int dim) { const int b = 16 + ((dim + 15) & ~15); return b <= 128 ? 128 : b; }
int rows8_query_bytes(int dim) { return 16 + 2 * ((dim + 15) & ~15); }

int code_rows(const float* d_data, int64_t n, int dim, int64_t ppb, int B, unsigned char* d_recs, uint32_t* d_bounds,
              hipStream_t s) {
    if (n <= 0) return 0;
    const int rc = zero_words64(d_bounds, (int64_t)B + ((int64_t)B + 1) / 2, s);
    if (rc) return rc;
    const int lpr = dim <= 256 ? 16 : 64, quads = (dim + 4 * lpr - 1) / (4 * lpr);
    const int64_t per_block = (int64_t)(kThreads / lpr) * kRows, blocks = (n + per_block - 1) / per_block;
    if (blocks > 0x7fffffffLL) return fail(-1, "code_rows: too many rows for one launch");
#define DCIH_CODE_ROWS(LPR, NQ)                                                                                       \
    hipLaunchKernelGGL((code_rows_kernel<LPR, NQ>), dim3((unsigned)blocks), dim3(kThreads), 0, s, d_data, n, dim, ppb, \
                       d_recs, rows8_record_bytes(dim), d_bounds)
    if (lpr == 16) {
        if (quads <= 2) DCIH_CODE_ROWS(16, 2); else if (quads == 3) DCIH_CODE_ROWS(16, 3); else DCIH_CODE_ROWS(16, 4);
    } else {
        if (quads <= 2) DCIH_CODE_ROWS(64, 2); else if (quads == 3) DCIH_CODE_ROWS(64, 3); else DCIH_CODE_ROWS(64, 4);
    }
#undef DCIH_CODE_ROWS
    DCIH_HIP(hipGetLastError());
    return 0;
}

int code_queries(const float* d_query, int nq, int dim, unsigned char* d_recs, hipStream_t s) {
    if (nq <= 0) return 0;
    const int lpr = dim <= 256 ? 16 : 64, code_bytes = (dim + 15) & ~15;
    const unsigned blocks = (unsigned)(((int64_t)nq * lpr + kThreads - 1) / kThreads);
    if (lpr == 16)
        hipLaunchKernelGGL(code_queries_kernel<16>, dim3(blocks), dim3(kThreads), 0, s, d_query, nq, dim, d_recs, code_bytes);
    else
        hipLaunchKernelGGL(code_queries_kernel<64>, dim3(blocks), dim3(kThreads), 0, s, d_query, nq, dim, d_recs, code_bytes);
    DCIH_HIP(hipGetLastError());
    return 0;
}

}  // namespace dcih
