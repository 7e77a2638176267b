// Rows rounded to 16-bit floats for the matrix cores, with what a bound of a distance needs to know about the rounding
// (bounds.hip says how the bound is made up).  Workgroups of kPackThreads threads where samples are taken.
#pragma once

#include "common.h"

namespace dcih {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_any __attribute__((aligned(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kPackThreads = 256;
constexpr int kTile = 32;                 // rows and queries of one matrix instruction
constexpr int kStep = 16;                 // elements of one
constexpr int kSample = 16;               // rows and queries the scales are taken from
constexpr float kHalfMax = 65504.0f, kHalfMin = 6.103515625e-05f;       // largest, and smallest normal, 16-bit float
constexpr uint32_t kInf = 0x7f800000u;

// 2^e with the sample's largest value at 64 .. 128: outliers of five hundred times that still fit, and what is
// flushed to zero is 2^-20 of it.  The exponent is limited so that no sum below can overflow.
__device__ inline float scale_for(float most) {
    if (!(most > 0.0f)) return 1.0f;
    const int e = (int)(__builtin_bit_cast(uint32_t, most) >> 23) - 127;
    const int up = min(40, max(-40, 6 - e));
    return __builtin_bit_cast(float, (uint32_t)(up + 127) << 23);
}

__device__ inline float block_max(float v, float* tmp) {
    v = __builtin_bit_cast(float, wave_max_i32(__builtin_bit_cast(int, v)));      // (not negative)
    __syncthreads();
    if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(tmp[0], tmp[1]), fmaxf(tmp[2], tmp[3]));
}
// Of some rows, a column per thread and all of them under way together: sum, smallest and largest value of each column that are finite.
template <class F>
__device__ inline void sample_columns(const float* base, int64_t rows, int dim, F use) {
    const int take = (int)min((int64_t)kSample, rows);
    for (int j = threadIdx.x; j < dim; j += kPackThreads) {
        float x[kSample], sum = 0.0f, lo = 3e38f, hi = -3e38f;
#pragma unroll
        for (int r = 0; r < kSample; r++) x[r] = base[(rows * min(r, take - 1) / take) * dim + j];
#pragma unroll
        for (int r = 0; r < kSample; r++) {
            const bool in = r < take && fabsf(x[r]) < 3e38f;
            sum += in ? x[r] : 0.0f;
            lo = in ? fminf(lo, x[r]) : lo;
            hi = in ? fmaxf(hi, x[r]) : hi;
        }
        use(j, sum / (float)take, lo, hi);
    }
}
// The common centre: the mean of some rows, in steps of 2^-7 of the power of two at their largest magnitude, so that whole numbers stay
// whole.  Returns those rows' largest magnitude less the centre.  s_centre: 3 * width floats, of which the first `width` are the centre.
__device__ inline float sample_centre(const float* base, int64_t rows, int dim, int width, float* s_centre, float* tmp) {
    float* s_lo = s_centre + width;
    float* s_hi = s_lo + width;
    float most = 0.0f;
    sample_columns(base, rows, dim, [&](int j, float mean, float lo, float hi) {
        s_centre[j] = mean; s_lo[j] = lo; s_hi[j] = hi;
        most = fmaxf(most, lo <= hi ? fmaxf(fabsf(lo), fabsf(hi)) : 0.0f);
    });
    most = block_max(most, tmp);
    const float step = __builtin_bit_cast(float, (uint32_t)max(1, (int)(__builtin_bit_cast(uint32_t, most) >> 23) - 7) << 23);
    float away = 0.0f;
    for (int j = threadIdx.x; j < width; j += kPackThreads) {      // (the thread's own columns)
        const float mean = j < dim ? rintf(s_centre[j] / step) * step : 0.0f;
        const float centre = fabsf(mean) <= most ? mean : 0.0f;
        if (j < dim && s_lo[j] <= s_hi[j]) away = fmaxf(away, fmaxf(fabsf(s_lo[j] - centre), fabsf(s_hi[j] - centre)));
        s_centre[j] = centre;
    }
    return block_max(away, tmp);
}

// Eight consecutive elements of a row, j a multiple of eight, zeros past its end; dim >= 8.  Rows of
// whole octets are read as such; else the last octet is read from the row's end and moved down.
template <bool OCTETS>
__device__ inline void load_octet(const float* row, int dim, int j, float (&x)[8]) {
    const int from = OCTETS ? min(j, dim - 8) : max(0, min(j, dim - 8));
    const v4f lo = *reinterpret_cast<const v4f_any*>(row + from), hi = *reinterpret_cast<const v4f_any*>(row + from + 4);
    x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w;
    x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
}
template <bool OCTETS>
__device__ inline void place_octet(int dim, int j, float (&x)[8]) {
    const int shift = j - max(0, min(j, dim - 8));
    if constexpr (!OCTETS) {
        const bool s4 = (shift & 4) != 0, s2 = (shift & 2) != 0, s1 = (shift & 1) != 0;
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = s4 ? (i + 4 < 8 ? x[i + 4] : 0.0f) : x[i];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = s2 ? (i + 2 < 8 ? x[i + 2] : 0.0f) : x[i];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = s1 ? (i + 1 < 8 ? x[i + 1] : 0.0f) : x[i];
    }
    if (shift >= 8)
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = 0.0f;
}
// Rounds x - centre to 16 bits and sums the squares of the rounded values and of what was rounded off (the subtraction's
// own rounding is allowed for where the sums are used).  No rounded value is larger than `most`: where the sum of an octet's squares
// does not say so, its values are cut to that one by one, and to zero what is not finite, which makes the second sum infinite.
// (16-bit floats below 2^-14, which the matrix cores may take as zeros, are allowed for in rounding_floor.)
__device__ inline v8h round_octet(const float (&x)[8], const float (&centre)[8], float scale, float most, float& sq, float& err) {
    v8h out;
    float s2 = 0.0f, e2 = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const float a = (x[i] - centre[i]) * scale, b = (x[i + 1] - centre[i + 1]) * scale;
        v2h h;
        h[0] = (_Float16)a; h[1] = (_Float16)b;
        out[i] = h[0]; out[i + 1] = h[1];
        s2 = __builtin_amdgcn_fdot2(h, h, s2, false);
        const float oa = __builtin_fmaf((float)h[0], -1.0f, a), ob = __builtin_fmaf((float)h[1], -1.0f, b);
        e2 = __builtin_fmaf(oa, oa, e2);
        e2 = __builtin_fmaf(ob, ob, e2);
    }
    if (!(s2 < most * most && e2 < 1e30f)) {
        s2 = e2 = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float v = (x[i] - centre[i]) * scale;
            if (!(fabsf(v) < 3e38f)) { v = 0.0f; e2 = __builtin_inff(); }
            out[i] = (_Float16)fminf(most, fmaxf(-most, v));
            const float back = (float)out[i], off = v - back;
            s2 = __builtin_fmaf(back, back, s2);
            e2 = __builtin_fmaf(off, off, e2);
        }
    }
    sq += s2;
    err += e2;
    return out;
}
// The largest length of what the values below 2^-14 make up, scaled.
__device__ inline float rounding_floor(int elements) { return sqrtf((float)elements) * kHalfMin; }
// An upper bound of |x - x'|, scaled, from the two sums: of what was rounded off (a float32 sum), of the values below 2^-14, and of the
// subtraction of the centre, a float32 ulp or less of what it gave.
__device__ inline float rounding_error(float sq, float err, int elements) {
    return sqrtf(err) * 1.001f + rounding_floor(elements) + sqrtf(sq + err) * 0x1p-22f;
}

// By how much a product's sum may be off, relative to what limits it (1.5 |x|^2 + 2 |x||q| + 0.5 |q|^2), and a factor that lowers a bound
// by the relative error of a distance formed in float32.  (Every addition off by 2^-23 of the largest magnitude a partial sum can
// have, twice what rounding to nearest allows; the squared lengths by half of that.)
__device__ inline float sum_error_of(int elements) { return (float)(elements + 32) * 0x1p-23f; }
__device__ inline float distance_factor(int dim) { return 1.0f - (float)(dim + 32) * 0x1p-23f; }
// A barrier that waits for the wavefront's LDS accesses only: __syncthreads() would wait for the reads from memory under way as well,
// which are to arrive in registers during what follows.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace
}  // namespace dcih
