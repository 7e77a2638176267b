// Which partitions of a query have to be traversed at all.
//
// A query's answer is the k best of all partitions' candidates (get_top_candidates,
// src/dci_cuda_kernel.cu:691-701), and a partition none of whose rows lies nearer than the k-th of
// them adds nothing to it, whatever its traversal would promote.  So a call of many items first
// bounds, for every (query, partition), the distance of the partition's nearest row from below --
// a matrix product on the matrix cores whose epilogue keeps a minimum -- and then traverses
//   first the partitions whose bound is within what the query's k nearest rows are bounded by,
//   then, as far as their bound does not exceed the k-th distance found so far, those within the bounds of the 2 k nearest and, the
//     dense kernel's, of the 4 k nearest,
//   last all others whose bound does not exceed it.
// What is left out lies further than that, so the results are those of traversing everything; where
// traversals miss near rows (low recall), or a bound is poor, the later rounds are larger, up to everything.
// (123457 normal rows of 67 elements, 37 partitions, 7 results, half of the pairs needed: 27 pairs a query in three rounds, 22 in
// four.  The batch kernel's calls take three: a fourth traversed 0.03 ms' worth of 8.9 on a million rows and
// cost as much again in launches.  Calls of about a millisecond take the first and the last round only: a round's launches would cost more than the pairs it saves.)
// The k nearest rows are told apart by bounds of parts of a partition: among S of them, k nearest rows that fall into
// the same part are k^2 / 2 S, which is what the first limit is too large by.
//
// The bounds of all tiles of 64 or 128 rows are kept where they fit.  By them most picked items are answered without a traversal (confirm.hip), and
// the dense kernel forms the distances of those candidates only whose
// tile can hold one that matters: in the first round one within the bounds of the 32 k nearest rows (a query whose k-th result turns out
// further away has those partitions taken again), later one within the k-th distance found.  Alone that gave 512 queries on 10M unit vectors of 96 21.4 -> 15.3 ms,
// 500 on 1M rows of 960 3.2 -> 2.6.
//
// Traversals that stop after a small part of a partition may find rows that lie further away than most partitions' bounds: then everything is
// traversed all the same, in rounds that each wait for their slowest item, behind bounds that ruled nothing out.  Whether that is so depends
// on the rows.  So such a call first traverses all partitions of a few of its queries, compares their results with bounds of a
// few partitions, and where these rule out too little for rounds to pay takes everything at once, without the other bounds
// (sample_decide_kernel; the device's own decision, nobody waits for it).
//
// The bound.  Rows and queries, less a common centre, are rounded to 16-bit floats x', q' (scaled by powers of two, so that
// nothing overflows; what does, or is not finite, has an unbounded error).  |x - q| >= |x' - q'| - |x - x'| - |q - q'|,
// the two errors being summed where the rounding is done, and |x' - q'|^2 = |x'|^2 + |q'|^2 - 2 x'.q' comes
// from 16-bit products added up in float32, lowered by what those additions can be off (the less, the nearer the data
// lies to the centre: on 1M rows of 128 elements of 0 to 300 a bound of 0.25 % below the distance takes 12 % more pairs).  The distance
// the traversal kernels compute is a float32 sum itself; the bound is lowered by its relative error too.
#include "common.h"
#include "half_core.h"
#include "kernels.h"

namespace dcih {

namespace {

constexpr int kWholeDim = 256;            // rows up to here can be kept in LDS whole
constexpr int kMostParts = 2048;           // bounds kept per query
constexpr int kLimits = kMostRounds;       // per query: of the rounds but the last, and how far a near row of round 1 may be
constexpr int kMostDies = 32;             // tickets cleared
constexpr int kListQueries = 1024;        // queries of a partition listed by one workgroup

struct Header { float row_scale, query_scale; };      // the centre follows, kCentre floats in
constexpr int kCentre = 16;

// The first workgroups round 32 queries each, into the order the matrix instructions take them
// ([32 queries][16 elements]: 64 lanes of 8), times -2; all of them clear what the later launches
// take as cleared: the bounds (infinite), the bounds of near tiles where they are formed by atomics (infinite), and the
// partitions' lists of results (empty).
struct PackArgs {
    const float* query; const float* data;
    int64_t n;
    int nq, dim, steps, tiles;            // steps: of 16 elements; tiles: of 32 queries
    Header* header;
    float2* qinfo;                        // [tiles * 32]: |q'|^2 and an upper bound of |q - q'|
    _Float16* frags;
    uint32_t* bounds; int64_t num_bounds;
    uint32_t* near; int64_t num_near;     // (only where they are formed by atomics)
    unsigned long long* part; int64_t num_part;
};
template <bool OCTETS>
__global__ __launch_bounds__(kPackThreads) void pack_queries_kernel(PackArgs a) {
    __shared__ float tmp[4];
    extern __shared__ float s_centre[];                       // [3][steps * 16]
    const int tid = threadIdx.x;
    const int64_t at = (int64_t)blockIdx.x * kPackThreads + tid, all = (int64_t)gridDim.x * kPackThreads;
    for (int64_t e = at; e < a.num_bounds; e += all) a.bounds[e] = kInf;
    for (int64_t e = at; e < a.num_near; e += all) a.near[e] = kInf;
    for (int64_t e = at; e < a.num_part; e += all) a.part[e] = ~0ull;
    if ((int)blockIdx.x >= a.tiles) return;
    const int width = a.steps * kStep;
    const float row_scale = scale_for(sample_centre(a.data, a.n, a.dim, width, s_centre, tmp));
    float most = 0.0f;
    sample_columns(a.query, a.nq, a.dim, [&](int j, float, float lo, float hi) {
        if (lo <= hi) most = fmaxf(most, fmaxf(fabsf(lo - s_centre[j]), fabsf(hi - s_centre[j])));
    });
    const float scale = scale_for(block_max(most, tmp));
    if (blockIdx.x == 0) {
        if (tid == 0) { a.header->row_scale = row_scale; a.header->query_scale = scale; }
        for (int j = tid; j < width; j += kPackThreads) reinterpret_cast<float*>(a.header)[kCentre + j] = s_centre[j];
    }
    const int qt = tid >> 3, q = (int)blockIdx.x * kTile + qt;
    const float* row = a.query + (int64_t)min(q, a.nq - 1) * a.dim;
    float sq = 0.0f, err = 0.0f;
    for (int o = tid & 7; o < 2 * a.steps; o += 8) {
        float x[8];
        load_octet<OCTETS>(row, a.dim, o * 8, x);
        place_octet<OCTETS>(a.dim, o * 8, x);
        float centre[8];
#pragma unroll
        for (int i = 0; i < 8; i++) centre[i] = s_centre[o * 8 + i];
        v8h h = round_octet(x, centre, scale, 0.5f * kHalfMax, sq, err);
#pragma unroll
        for (int i = 0; i < 8; i++) h[i] = (_Float16)((float)h[i] * -2.0f);      // (exact, and finite: half the largest at most)
        *reinterpret_cast<v8h*>(a.frags + (((int64_t)blockIdx.x * a.steps + (o >> 1)) * 64 + (o & 1) * 32 + qt) * 8) = h;
    }
    sq += lane_xor<4>(sq); sq += lane_xor<2>(sq); sq += lane_xor<1>(sq);
    err += lane_xor<4>(err); err += lane_xor<2>(err); err += lane_xor<1>(err);
    if ((tid & 7) == 0) {
        const float inv = 1.0f / scale;
        a.qinfo[q] = make_float2(sq * inv * inv, rounding_error(sq, err, a.steps * kStep) * inv);
    }
}

struct BoundArgs {
    const float* data;
    int64_t n, ppb, step;                 // step: rows from a partition to the next one taken (ppb, or more for a sample of them)
    int dim, steps, nq, tiles;
    int column_steps;                     // staged at a time (even)
    int next_part, next_tile;             // from a workgroup's row tile to its next one
    int num_parts, row_tiles, parts;      // partitions, row tiles of each, and the parts of each that bounds are kept for
    const Header* header; const float2* qinfo; const _Float16* frags;
    uint32_t* bounds;                     // [B * parts][nq] float bits
    uint32_t* tile_bounds;                // null, or the same of every near_rows(RT) rows
    const uint32_t* skip;                 // null, or where it says so nothing is formed
};

// The rows a near tile holds: one wavefront's, 64 at least.
__host__ __device__ constexpr int near_rows(int rt) { return kTile * (rt < 2 ? 2 : rt); }

// What the kernels below share.  A workgroup of WR wavefronts along the rows and WC along the queries takes tiles of R = 32 RT WR
// rows of a partition, each wavefront RT x CT accumulators of 32 x 32.  A row's squared length is where its
// accumulators start (or is added at their end), so what is left to do with a sum is to keep the smallest, in the lane that holds the
// query's column.
// QD: steps of the queries that are under way.  A step is multiplied in 256 cycles, less than a read from the L2 takes, and where rows are streamed one
// wavefront of a SIMD multiplies: with two steps ahead 512 queries on 10M rows of 96 take 1956 us, with six 1872; 500 on 1M rows of 960, two and four,
// 1483, 1430.  (Two stretches of rows under way instead of one change nothing: the multiplying side is the slower one.  Without the
// multiplications 1169 and 807 us, with every tile reading the same rows 1814 and 1255.)
template <int RT, int CT, int WR, int WC, int COLUMNS, bool OCTETS, int QD = 2>
struct BoundTile {
    static constexpr int kWaves = WR * WC, R = kTile * RT * WR, kGroups = R / 8 / kWaves, kOctets = COLUMNS / 64;
    static_assert(kGroups >= 1 && kOctets >= 1, "eight rows per wavefront at least");
    typedef float Octets[kGroups][kOctets][8];
    const BoundArgs& a;
    const int lane;
    const bool reads;                     // (streamed rows: the first kWaves wavefronts read, the others multiply)
    const int wave, wr, wc;
    const float row_scale, query_scale;
    const float* base;                    // of the tile: its first row, number of rows, and its bounds
    int rows;
    uint32_t* out;
    int64_t tile_out;                     // (where the tile's own ones begin)

    __device__ __forceinline__ BoundTile(const BoundArgs& args)
        : a(args), lane((int)(threadIdx.x & 63)), reads(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) < kWaves),
          wave(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) % kWaves), wr(wave / WC), wc(wave % WC),
          row_scale(args.header->row_scale), query_scale(args.header->query_scale), base(nullptr), rows(0), out(nullptr), tile_out(0) {}

    // Row tile rt of partition b.
    __device__ __forceinline__ void take(int b, int rt) {
        const int64_t off = (int64_t)b * a.step, first = off + (int64_t)rt * R;
        rows = (int)min((int64_t)R, min(a.n, off + a.ppb) - first);
        base = a.data + first * a.dim;
        out = a.bounds + ((int64_t)b * a.parts + rt * a.parts / a.row_tiles) * a.nq;
        tile_out = (((int64_t)b * a.row_tiles + rt) * (R / near_rows(RT)) + wr * RT * kTile / near_rows(RT)) * a.nq;
    }
    // Columns [16 s0 + 8 o0, ..) of the tile's rows, kOctets octets per lane of each of its kGroups rows: read, then rounded into LDS in
    // the order the matrix instructions take them.  A lane group of eight takes eight rows, so that its stores hit different banks; eight
    // such groups read 256 bytes of a row.  All of a wavefront's reads are under way before the first is used.
    __device__ __forceinline__ void read(Octets& x, int s0, int o0, int octets) const {
#pragma unroll
        for (int g = 0; g < kGroups; g++) {
            const int r = (g * kWaves + wave) * 8 + (lane & 7);
            const float* row = base + (int64_t)min(r, rows - 1) * a.dim;
#pragma unroll
            for (int u = 0; u < kOctets; u++) load_octet<OCTETS>(row, a.dim, s0 * kStep + min(o0 + 8 * u + (lane >> 3), octets - 1) * 8, x[g][u]);
        }
    }
    __device__ __forceinline__ void place(Octets& x, v8h* to, const float* s_centre, int pitch, int s0, int o0, int octets,
                                          float (&sq)[kGroups], float (&err)[kGroups]) const {
#pragma unroll
        for (int u = 0; u < kOctets; u++) {
            const int o = o0 + 8 * u + (lane >> 3);
            if (o < octets) {
                float centre[8];
                const v4f lo = *reinterpret_cast<const v4f*>(s_centre + s0 * kStep + o * 8), hi = *reinterpret_cast<const v4f*>(s_centre + s0 * kStep + o * 8 + 4);
                centre[0] = lo.x; centre[1] = lo.y; centre[2] = lo.z; centre[3] = lo.w;
                centre[4] = hi.x; centre[5] = hi.y; centre[6] = hi.z; centre[7] = hi.w;
#pragma unroll
                for (int g = 0; g < kGroups; g++) {
                    const int r = (g * kWaves + wave) * 8 + (lane & 7);
                    place_octet<OCTETS>(a.dim, s0 * kStep + o * 8, x[g][u]);
                    to[((r >> 5) * pitch + (o >> 1)) * 64 + (o & 1) * 32 + (r & 31)] = round_octet(x[g][u], centre, row_scale, kHalfMax, sq[g], err[g]);
                }
            }
        }
    }
    // The centre into LDS, by the whole workgroup.
    __device__ __forceinline__ void copy_centre(float* s_centre) const {
        for (int j = threadIdx.x; j < a.steps * kStep; j += blockDim.x) s_centre[j] = reinterpret_cast<const float*>(a.header)[kCentre + j];
        __syncthreads();
    }
    // Squared lengths, scaled as the products are (infinite past the last row), and the wavefront's largest length and error.
    __device__ __forceinline__ void put_sums(const float (&sq)[kGroups], const float (&err)[kGroups], float* s_n, float* s_red) const {
        const float to_sum = query_scale / row_scale;
        float mn = 0.0f, me = 0.0f;
#pragma unroll
        for (int g = 0; g < kGroups; g++) {
            const int r = (g * kWaves + wave) * 8 + (lane & 7);
            float s2 = sq[g], e2 = err[g];
            s2 += lane_xor<32>(s2); s2 += lane_xor<16>(s2); s2 += lane_xor<8>(s2);
            e2 += lane_xor<32>(e2); e2 += lane_xor<16>(e2); e2 += lane_xor<8>(e2);
            if (r < rows) { mn = fmaxf(mn, s2); me = fmaxf(me, e2); }
            if (lane < 8) s_n[r] = r < rows ? s2 * to_sum : __builtin_inff();
        }
        mn = fmaxf(mn, lane_xor<4>(mn)); mn = fmaxf(mn, lane_xor<2>(mn)); mn = fmaxf(mn, lane_xor<1>(mn));
        me = fmaxf(me, lane_xor<4>(me)); me = fmaxf(me, lane_xor<2>(me)); me = fmaxf(me, lane_xor<1>(me));
        if (lane == 0) { s_red[wave] = mn; s_red[kWaves + wave] = me; }
    }
    // Largest squared length and largest error of the tile's rows.
    __device__ __forceinline__ float2 most(const float* s_red) const {
        float n = 0.0f, e = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; w++) { n = fmaxf(n, s_red[w]); e = fmaxf(e, s_red[kWaves + w]); }
        const float inv = 1.0f / row_scale;
        return make_float2(n * inv * inv, rounding_error(n, e, a.steps * kStep) * inv);
    }
    __device__ __forceinline__ v16f lengths(const float* s_n, int r) const {      // of row tile r of this wavefront
        v16f v;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const v4f t = *reinterpret_cast<const v4f*>(s_n + (wr * RT + r) * kTile + 8 * i + 4 * (lane >> 5));
            v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
        }
        return v;
    }
    // The queries' steps in the order a wavefront multiplies them: all of tiles first .. first + CT - 1, then of those kPass
    // further on, and from the beginning again.  q8 holds the next QD; a step's registers take the step QD further on once it has
    // been multiplied, no sooner, or the compiler copies them, which waits for what is under way.
    struct Queries {
        v8h q8[QD][CT];
        uint32_t at, group, left;         // bytes from a.frags on: the step read next and its tiles' first one; steps left of those
        uint32_t first, end, stride;      // the first tiles; past the last; from tiles to the next tiles
        uint32_t mine[CT];                // the lane's place in a step
    };
    __device__ __forceinline__ void read_queries(Queries& y, v8h (&q)[CT]) const {
#pragma unroll
        for (int c = 0; c < CT; c++) q[c] = *reinterpret_cast<const v8h*>(reinterpret_cast<const char*>(a.frags) + (y.at + y.mine[c]));
    }
    __device__ __forceinline__ void next_step(Queries& y) const {
        y.left--;
        const uint32_t on = y.group + y.stride, group = on < y.end ? on : y.first;
        const bool over = y.left == 0;
        y.at = over ? group : y.at + 1024;
        y.group = over ? group : y.group;
        y.left = over ? (uint32_t)a.steps : y.left;
    }
    __device__ __forceinline__ void start_queries(Queries& y, int tile) const {
        constexpr int kPass = CT * WC;
        const uint32_t bytes = (uint32_t)a.steps * 1024u;
        y.first = (uint32_t)tile * bytes;
        y.end = (uint32_t)a.tiles * bytes;
        y.stride = kPass * bytes;
        y.at = y.group = y.first;
        y.left = (uint32_t)a.steps;
#pragma unroll
        for (int c = 0; c < CT; c++) y.mine[c] = c * bytes + lane * 16;
#pragma unroll
        for (int u = 0; u < QD; u++) {
            read_queries(y, y.q8[u]);
            next_step(y);
        }
    }
    // The next ns (a multiple of QD) steps.
    __device__ __forceinline__ void multiply_steps(v16f (&acc)[RT][CT], const v8h* rows_at, int pitch, Queries& y, int ns) const {
        v8h x8[2][RT];
#pragma unroll
        for (int r = 0; r < RT; r++) x8[0][r] = rows_at[r * pitch * 64];
        auto one = [&](const v8h* next_rows, v8h (&x)[RT], v8h (&x_next)[RT], v8h (&q)[CT]) {
#pragma unroll
            for (int r = 0; r < RT; r++) x_next[r] = next_rows[r * pitch * 64];
            Queries then = y;
            next_step(then);
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int c = 0; c < CT; c++) acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[r], q[c], acc[r][c], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            read_queries(y, q);
            __builtin_amdgcn_sched_barrier(0);
            y.at = then.at; y.group = then.group; y.left = then.left;
        };
        static_assert(QD % 2 == 0, "the rows' steps take two turns");
        for (int s = 0; s < ns; s += QD) {
#pragma unroll
            for (int u = 0; u < QD; u++) one(rows_at + min(s + u + 1, ns - 1) * 64, x8[u & 1], x8[(u + 1) & 1], y.q8[u]);
        }
    }
    // The smallest sum of each of 32 CT queries over the wavefront's rows -> their bounds; q: the lane's query of the first 64.
    __device__ __forceinline__ void finish(const v16f (&acc)[RT][CT], int q, bool mine, const float2 (&info)[(CT + 1) / 2],
                                           const uint32_t (&have)[(CT + 1) / 2], float2 most) const {
        const float unscale = 1.0f / (row_scale * query_scale);
        const float sum_error = sum_error_of(a.steps * kStep), dist_error = distance_factor(a.dim);
        float best[CT];
#pragma unroll
        for (int c = 0; c < CT; c++) {      // (four chains each: a single one would wait for every result)
            float part[4];
#pragma unroll
            for (int i = 0; i < 4; i++) part[i] = fminf(fminf(acc[0][c][i], acc[0][c][i + 4]), acc[0][c][i + 8]);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                part[i] = fminf(part[i], acc[0][c][i + 12]);
#pragma unroll
                for (int r = 1; r < RT; r++) {
                    part[i] = fminf(fminf(part[i], acc[r][c][i]), acc[r][c][i + 4]);
                    part[i] = fminf(fminf(part[i], acc[r][c][i + 8]), acc[r][c][i + 12]);
                }
            }
            best[c] = fminf(fminf(part[0], part[1]), fminf(part[2], part[3]));
        }
#pragma unroll
        for (int c = 0; c < CT; c++) best[c] = fminf(best[c], lane_xor<32>(best[c]));
#pragma unroll
        for (int c = 0; c < (CT + 1) / 2; c++) {
            const float v = CT >= 2 && lane >= 32 ? best[min(2 * c + 1, CT - 1)] : best[2 * c];
            const float d2 = v * unscale + info[c].x - sum_error * (1.5f * most.x + 2.0f * sqrtf(most.x * info[c].x) + 0.5f * info[c].x);
            float d = sqrtf(fmaxf(d2, 0.0f)) - most.y - info[c].y;
            d = fmaxf(d, 0.0f) * dist_error;
            if (!(d > 1e-14f)) d = 0.0f;                      // (squares below the smallest float count as nothing in the distances)
            const uint32_t bits = __builtin_bit_cast(uint32_t, d);
            if (mine && q + 64 * c < a.nq) {
                if (a.tile_bounds) {
                    if constexpr (RT * kTile < near_rows(RT)) atomicMin(&a.tile_bounds[tile_out + q + 64 * c], bits);
                    else a.tile_bounds[tile_out + q + 64 * c] = bits;
                }
                if (bits < have[c]) atomicMin(&out[q + 64 * c], bits);
            }
        }
    }
};

// Many queries, rows of at most kWholeDim elements: a workgroup keeps one row tile in LDS and takes all queries past it.  Bound by
// the matrix cores and the reads of the queries from L2 (32 bytes per CU and clock at the full rate).
template <int RT, int CT, int WC, int WAVES, bool OCTETS>
__global__ __launch_bounds__(64 * WC, WAVES) void bounds_resident_kernel(BoundArgs a) {
    typedef BoundTile<RT, CT, 1, WC, 128, OCTETS> Tile;
    extern __shared__ __align__(16) unsigned char smem[];
    float* s_n = reinterpret_cast<float*>(smem);
    float* s_red = s_n + Tile::R;
    float* s_centre = s_red + 2 * Tile::kWaves;
    v8h* s_rows = reinterpret_cast<v8h*>(s_centre + a.steps * kStep);
    if (a.skip && *a.skip) return;
    Tile y(a);
    y.take((int)(blockIdx.x / (unsigned)a.row_tiles), (int)(blockIdx.x % (unsigned)a.row_tiles));
    if (y.rows <= 0) return;
    const int lane = y.lane;
    y.copy_centre(s_centre);
    {
        float sq[Tile::kGroups] = {}, err[Tile::kGroups] = {};
        for (int o0 = 0; o0 < 2 * a.steps; o0 += 8 * Tile::kOctets) {
            typename Tile::Octets x;
            y.read(x, 0, o0, 2 * a.steps);
            y.place(x, s_rows, s_centre, a.steps, 0, o0, 2 * a.steps, sq, err);
        }
        y.put_sums(sq, err, s_n, s_red);
    }
    __syncthreads();
    const float2 most = y.most(s_red);
    constexpr int kPass = CT * WC;                            // query tiles of one pass
    const int first = y.wc * CT;
    if (first >= a.tiles) return;
    typename Tile::Queries queries;
    y.start_queries(queries, first);
    for (int t = first; t < a.tiles; t += kPass) {
        const int q = (t + (lane >> 5)) * kTile + (lane & 31);
        const bool mine = q < a.nq && (CT == 2 || lane < 32);
        const float2 info[1] = {a.qinfo[min(q, a.nq - 1)]};
        const uint32_t have[1] = {y.out[min(q, a.nq - 1)]};
        v16f acc[RT][CT];
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const v16f start = y.lengths(s_n, r);
#pragma unroll
            for (int c = 0; c < CT; c++) acc[r][c] = start;
        }
        y.multiply_steps(acc, s_rows + lane, a.steps, queries, a.steps);
        y.finish(acc, q, mine, info, have, most);
    }
}

// Fewer queries, or longer rows: the rows are streamed through two halves of LDS, COLUMNS columns of a tile at a time, by four wavefronts
// that read and round, while four others multiply what the first have placed before; a workgroup goes on from tile to tile.
// (One set of wavefronts for both cannot: their reads of the queries would wait for the reads of rows issued before them,
// 592 us for 512 queries on 2M rows of 96.)  ONE: a row is no longer than COLUMNS, and all queries are taken past it while it lies there;
// else its columns come once for every pass over 32 CT WC queries.
template <int RT, int CT, int WR, int WC, int COLUMNS, int WAVES, bool ONE, bool OCTETS, int QD>
__global__ __launch_bounds__(128 * WR * WC, WAVES) void bounds_stream_kernel(BoundArgs a) {
    typedef BoundTile<RT, CT, WR, WC, COLUMNS, OCTETS, QD> Tile;
    constexpr int kPass = CT * WC;
    extern __shared__ __align__(16) unsigned char smem[];
    const int pitch = a.column_steps, half = Tile::R * pitch * 2;      // 16-byte words
    float* s_n = reinterpret_cast<float*>(smem);              // [2][R], by turns of tiles
    float* s_red = s_n + 2 * Tile::R;                         // [2][2 * kWaves]
    float* s_centre = s_red + 4 * Tile::kWaves;
    v8h* s_rows = reinterpret_cast<v8h*>(s_centre + a.steps * kStep);
    if (a.skip && *a.skip) return;
    Tile y(a);
    y.copy_centre(s_centre);
    int b = (int)(blockIdx.x / (unsigned)a.row_tiles), rt = (int)(blockIdx.x % (unsigned)a.row_tiles);
    auto go_on = [&]() {                                      // the workgroup's next tile that has rows
        do {
            b += a.next_part;
            rt += a.next_tile;
            if (rt >= a.row_tiles) { rt -= a.row_tiles; b++; }
            if (b < a.num_parts) y.take(b, rt);
        } while (b < a.num_parts && y.rows <= 0);
    };
    y.take(b, rt);
    if (y.rows <= 0) go_on();
    if (b >= a.num_parts) return;
    int side = 0, turn = 0;
    if (y.reads) {
        // ---- reads and rounds: what comes next is under way while the others multiply what lies in LDS.  (One place that reads, and
        // under no condition: registers that come together from two are copied, which waits for them.)
        const int passes = ONE ? 1 : (a.tiles + kPass - 1) / kPass;
        typename Tile::Octets next;
        float sq[Tile::kGroups], err[Tile::kGroups];
        int s0 = 0, pass = 0;
        y.read(next, 0, 0, 2 * pitch);
        for (;;) {
            if (s0 == 0)
#pragma unroll
                for (int g = 0; g < Tile::kGroups; g++) sq[g] = err[g] = 0.0f;
            y.place(next, s_rows + side * half, s_centre, pitch, s0, 0, 2 * min(pitch, a.steps - s0), sq, err);
            s0 += pitch;
            if (s0 >= a.steps) {
                s0 = 0;
                if (pass == 0) y.put_sums(sq, err, s_n + turn * Tile::R, s_red + turn * 2 * Tile::kWaves);
                if (++pass == passes) { pass = 0; turn ^= 1; go_on(); }
            }
            y.read(next, s0, 0, 2 * min(pitch, a.steps - s0));      // (past the last tile: its columns again)
            side ^= 1;
            lds_barrier();
            if (b >= a.num_parts) return;
        }
    }
    // ---- multiplies
    const int lane = y.lane, first = y.wc * CT;
    typename Tile::Queries queries;
    y.start_queries(queries, min(first, a.tiles - CT));
    for (; b < a.num_parts; go_on(), turn ^= 1) {
        const float* n_here = s_n + turn * Tile::R;
        const float* red_here = s_red + turn * 2 * Tile::kWaves;
        float2 most;
        if constexpr (ONE) {
            lds_barrier();
            most = y.most(red_here);
        }
        for (int t0 = 0; t0 < a.tiles; t0 += kPass) {
            const int t = t0 + first;
            const bool busy = t < a.tiles;
            if (ONE && !busy) break;
            const int q = (t + (lane >> 5)) * kTile + (lane & 31);
            const bool mine = busy && q < a.nq && (CT >= 2 || lane < 32);
            float2 info[(CT + 1) / 2];
            uint32_t have[(CT + 1) / 2];
#pragma unroll
            for (int c = 0; c < (CT + 1) / 2; c++) { const int qc = min(q + 64 * c, a.nq - 1); info[c] = a.qinfo[qc]; have[c] = y.out[qc]; }
            v16f acc[RT][CT];
#pragma unroll
            for (int r = 0; r < RT; r++) {
                v16f start = {};
                if constexpr (ONE) start = y.lengths(n_here, r);
#pragma unroll
                for (int c = 0; c < CT; c++) acc[r][c] = start;
            }
            if constexpr (ONE) {
                y.multiply_steps(acc, s_rows + side * half + y.wr * RT * pitch * 64 + lane, pitch, queries, a.steps);
            } else {
                for (int s0 = 0; s0 < a.steps; s0 += pitch) {
                    lds_barrier();
                    if (busy)
                        y.multiply_steps(acc, s_rows + side * half + y.wr * RT * pitch * 64 + lane, pitch, queries, min(pitch, a.steps - s0));
                    side ^= 1;
                }
                most = y.most(red_here);
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    const v16f n2 = y.lengths(n_here, r);
#pragma unroll
                    for (int c = 0; c < CT; c++)
#pragma unroll
                        for (int i = 0; i < 16; i++) acc[r][c][i] += n2[i];
                }
            }
            y.finish(acc, q, mine, info, have, most);
        }
        if constexpr (ONE) side ^= 1;
    }
}

// Of each query's S bounds about the j-th, the 2 j-th, the 4 j-th and the near_rank-th smallest, one wavefront per query: the
// largest in the histogram's bins up to the one that holds it, 1024 bins over the range of those that are finite.  A workgroup reads the
// bounds of `per` neighbouring queries into LDS first.  (Bit by bit, with a ballot per bit, limit and 64 bounds: 3 times as long.)
template <int V>
__global__ __launch_bounds__(256) void pick_limits_kernel(const uint32_t* __restrict__ bounds, int S, int nq, int per, int j, int near_rank, int tight_rank, float flat,
                                                          uint32_t* __restrict__ limits, uint32_t* __restrict__ last_round, uint32_t* __restrict__ blind) {
    constexpr int kBins = 1024, kMine = kBins / 64;
    __shared__ uint32_t s_hist[4][kBins];
    extern __shared__ uint32_t s_b[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q0 = (int)blockIdx.x * per, pitch = per + 1;
    bool all_blind = true;
#pragma unroll 4
    for (int e = threadIdx.x; e < S * per; e += 256) {
        const int i = e / per, q = e - i * per;
        s_b[i * pitch + q] = bounds[(int64_t)i * nq + min(q0 + q, nq - 1)];
    }
    __syncthreads();
    uint32_t* hist = s_hist[wave];
    for (int q = wave; q < per; q += 4) {      // (each wavefront its own histogram; no barrier below)
        uint32_t v[V], lo = kInf;
        int hi = 0;
#pragma unroll
        for (int i = 0; i < V; i++) {
            v[i] = i * 64 + lane < S ? s_b[(i * 64 + lane) * pitch + q] : kInf;
            lo = min(lo, v[i]);
            hi = max(hi, v[i] < kInf ? (int)v[i] : 0);
        }
        const float f_lo = __builtin_bit_cast(float, wave_min_u32(lo));
        const float range = __builtin_bit_cast(float, wave_max_i32(hi)) - f_lo;
        const float scale = range > 1e-30f ? (float)kBins / range : 0.0f;
        auto bin = [&](uint32_t x) { return x < kInf ? min(kBins - 1, (int)((__builtin_bit_cast(float, x) - f_lo) * scale)) : kBins; };
#pragma unroll
        for (int i = 0; i < kMine; i++) hist[i * 64 + lane] = 0;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < V; i++) if (v[i] < kInf) atomicAdd(&hist[bin(v[i])], 1u);
        __builtin_amdgcn_wave_barrier();
        uint32_t mine[kMine], sum = 0;
#pragma unroll
        for (int i = 0; i < kMine; i++) { mine[i] = hist[lane * kMine + i]; sum += mine[i]; }
        const uint32_t upto = wave_scan_u32(sum);
        uint32_t limit[kLimits + 1];          // (the last one: of confirm.hip's first round)
#pragma unroll
        for (int w = 0; w < kLimits + 1; w++) {
            const uint32_t rank = (uint32_t)(w == kLimits ? tight_rank : (w == kLimits - 1 ? near_rank : j << w));
            uint32_t run = upto - sum;
            int at = kBins - 1;
#pragma unroll
            for (int i = 0; i < kMine; i++) { run += mine[i]; at = run >= rank ? min(at, lane * kMine + i) : at; }
            at = (int)wave_min_u32((uint32_t)at);
            int most = 0;
#pragma unroll
            for (int i = 0; i < V; i++) most = max(most, bin(v[i]) <= at ? (int)v[i] : 0);
            most = wave_max_i32(most);
            limit[w] = __ballot(upto >= rank) ? (uint32_t)most : kInf;          // (infinite where there are fewer)
        }
        // Bounds that say nothing of the nearest: candidates of any distance are wanted, or round 2 would take them all again.  (1000 queries, 100
        // partitions of 10000 rows of 128 in clusters a thousand times further apart than they are wide: 32 ms whole, 67 with whole rows read twice,
        // 33 once and, from the second call on, by the rows' codes, which near rows do without otherwise.)
        if (limit[0] == 0) limit[kLimits - 1] = limit[kLimits] = kInf; else all_blind = false;
        // Bounds too close together for what a short traversal finds: the first round would find no distance that rules a partition out.
        if (f_lo + range < flat * __builtin_bit_cast(float, limit[0])) limit[0] = limit[1] = limit[2] = kInf;
        if (q0 + q < nq) {
            if (lane <= kLimits) limits[(int64_t)lane * nq + q0 + q] = lane == 0 ? limit[0] : (lane == 1 ? limit[1] : (lane == 2 ? limit[2] : (lane == 3 ? limit[3] : limit[4])));
            if (lane == 0) last_round[q0 + q] = 0;
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (blind && all_blind && wave < per && lane == 0) *reinterpret_cast<volatile uint32_t*>(blind) = 1;
}

// Lists the (query, partition) pairs of a round by partition, then query: each die takes one run of the list, so that its
// resident workgroups work on one partition and its slices stay in the die's L2, whatever partitions the pairs are of.  (In the order in
// which workgroups came to reserve their places, a die's 832 items of 17242 points were of five partitions, and took twice as long.)
// One workgroup per kListQueries queries of a partition; the first launch counts, the second adds up the counts before its own.
struct ListArgs {
    const uint32_t* bounds; const uint32_t* limits; const uint32_t* skip;
    const float* worst; int64_t worst_stride;      // the k-th distance each query has so far
    uint32_t* last_round;                          // the round that last took a partition of the query
    int B, parts, nq, groups, round, rounds, near;
    uint32_t* rests; unsigned long long* confirm_word; uint32_t confirm_tag; int confirm_dies;      // (0: confirm.hip has no part in the call)
    const float* near_then; float* near_now;       // how far rows counted in the round before, and in this one
    int32_t* items; uint32_t* count; uint32_t* part_counts; uint32_t* ticket;
};
__device__ inline bool takes_item(const ListArgs& a, int b, int q) {
    if (a.skip && *a.skip) return a.round == 0;
    uint32_t v = a.bounds[(int64_t)b * a.parts * a.nq + q];
    for (int p = 1; p < a.parts; p++) v = min(v, a.bounds[((int64_t)b * a.parts + p) * a.nq + q]);
    // a round takes what lies between two limits, the last one everything above the last limit
    if (a.round + 1 < a.rounds && v > a.limits[(int64_t)a.round * a.nq + q]) return false;
    if (a.round == 0) return true;
    // (what is infinite or NaN so far is bounded by nothing)
    const float worst = a.worst[(int64_t)q * a.worst_stride];
    if (__builtin_bit_cast(float, v) > worst) return false;
    if (v > a.limits[(int64_t)(a.round - 1) * a.nq + q]) return true;
    // the round before took no candidates further away than its limit: where the k-th so far is, its partitions and those before are taken again
    // (by the traversals alone only round 1's limit can be that)
    const float wide = __builtin_bit_cast(float, a.limits[(int64_t)(kLimits - 1) * a.nq + q]);
    if (a.confirm_dies == 0) return a.near && a.round == 1 && !(worst <= wide);
    return !(worst <= (a.round == 1 && a.rests[1] ? wide : a.near_then[q]));
}
template <bool COUNT>
__global__ __launch_bounds__(256) void list_items_kernel(ListArgs a) {
    __shared__ uint32_t s_wave[4], s_before[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int b = blockIdx.x / a.groups, q0 = (int)(blockIdx.x % a.groups) * kListQueries, q1 = min(a.nq, q0 + kListQueries);
    unsigned long long m[kListQueries / 256];
    uint32_t mine = 0;
#pragma unroll
    for (int i = 0; i < kListQueries / 256; i++) {      // (a wavefront's queries are consecutive)
        const int q = q0 + wave * (kListQueries / 4) + i * 64 + lane;
        m[i] = __ballot(q < q1 && takes_item(a, b, min(q, a.nq - 1)));
        mine += (uint32_t)__popcll(m[i]);
    }
    uint32_t before = 0;
    if (!COUNT) {
        for (int e = tid; e < (int)blockIdx.x; e += 256) before += a.part_counts[e];
        before = wave_sum_u32(before);
    }
    if (lane == 0) { s_wave[wave] = mine; s_before[wave] = before; }
    __syncthreads();
    if (COUNT) {
        if (tid == 0) a.part_counts[blockIdx.x] = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
        return;
    }
    uint32_t at = s_before[0] + s_before[1] + s_before[2] + s_before[3];
    // What confirm.hip has made of the items it counts, in earlier rounds: for it, and for later calls.
    if (a.confirm_dies > 0 && blockIdx.x == 0 && wave == 3) {
        const uint32_t* left = a.ticket + (kLeftWord - kTicketWord) + (lane & (kMostDies - 1)) * kTicketStride;
        const uint32_t had = wave_sum_u32(a.round > 0 && lane < a.confirm_dies ? left[1] + left[kConfirmPass + 1] : 0u);
        const uint32_t lost = wave_sum_u32(a.round > 0 && lane < a.confirm_dies ? left[2] : 0u);
        if (lane == 0) {
            a.rests[0] = lost > 16 + had ? 1u : 0u;
            if (a.round == 0) a.rests[1] = 0;
            if (a.confirm_word && a.round > 0) {
                // (one store, so that the host reads what belongs together; their ratio is what matters)
                uint32_t h = had, l = lost;
                while ((h | l) >> 24) { h >>= 1; l >>= 1; }
                *reinterpret_cast<volatile unsigned long long*>(a.confirm_word) = (unsigned long long)a.confirm_tag << 48 | (unsigned long long)l << 24 | h;
            }
        }
    }
    if (blockIdx.x == 0 && tid < kMostDies) {
        uint32_t* left = a.ticket + (kLeftWord - kTicketWord) + tid * kTicketStride;
        a.ticket[tid * kTicketStride] = left[0] = left[kConfirmPass] = 0;
        if (a.round == 0) left[1] = left[2] = left[kConfirmPass + 1] = left[kConfirmPass + 2] = left[kConfirmPilot + 1] = left[kConfirmPilot + 2] = 0;
    }
    // (of queries that have no k results yet, rows as near as round 1's partitions may hold: all rows come in the last round)
    if (a.confirm_dies > 0 && a.round > 0 && b == 0)
        for (int q = q0 + tid; q < q1; q += 256) {
            const float worst = a.worst[(int64_t)q * a.worst_stride], wide = __builtin_bit_cast(float, a.limits[(int64_t)(kLimits - 1) * a.nq + q]);
            a.near_now[q] = a.round + 1 < a.rounds && !(worst < __builtin_inff()) ? wide : worst;
        }
    if (blockIdx.x + 1 == gridDim.x && tid == 0) *a.count = at + s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
    for (int w = 0; w < wave; w++) at += s_wave[w];
#pragma unroll
    for (int i = 0; i < kListQueries / 256; i++) {
        const int q = q0 + wave * (kListQueries / 4) + i * 64 + lane;
        if ((m[i] >> lane) & 1ull) {
            a.items[at + (uint32_t)__popcll(m[i] & ((1ull << lane) - 1ull))] = (int32_t)((int64_t)q * a.B + b);
            if (a.round > 0) a.last_round[q] = (uint32_t)a.round;
        }
        at += (uint32_t)__popcll(m[i]);
    }
}

// How the product is cut: row tiles and query tiles per wavefront, wavefronts along rows and queries; rows streamed or a tile of them
// resident, and read once or once for every pass over the queries.  Up to 128 queries the rows' bytes bound it (512 columns: 160 us
// for 819 MB, 5.1 TB/s), so all queries are taken in one pass with as few accumulators as hold them, and with them as many reading
// wavefronts; above, the matrix cores, and a wavefront of 4x2 tiles reads 6 fragments for 8 products, one of 2x2 4 for 4.  us on 400000
// rows in 10 partitions, columns/queries, the cut taken first:
//   1x1 against 1x2 tiles:            64/32 28, 29    128/32 48, 50    512/32 160, 170    and at 48 queries 1x2 30, 44; 49, 65; 168, 274
//   1x2 against 2x2 (2x2 wavefronts): 64/64 30, 45    128/64 49, 53    512/64 167, 158    and at 128 queries 2x2 46, 40; 56, 65; 181, 289
//   2x2 against 4x2:                  64/128 46, 47   128/128 56, 59   200/128 82, 90     and at 192 queries 4x2 49, 62; 60, 80; 98, 131
//   2x2 against 2x4, past 256 columns (rows are not kept whole there): 512/128 181, 268; at 192 queries 2x4 288, 276; 512 320, 567
//   streamed against resident rows:   64/192 49, 53   64/1024 113, 95  200/1024 236, 202  and at 4096 queries resident 260, 349; 404, 505; 622, 798
// (resident rows are up to 16 % the faster ones from 512 queries on where there are as many rows; streamed ones keep fewer rows' workgroups busy).
// Rows of up to 128 columns are rounded once, whole; longer ones a stretch at a time.
struct Shape { int rt, ct, wr, wc; bool stream, one; };
Shape shape_of(const QueryArgs& a) {
    if (a.nq <= 32) return {1, 1, 4, 1, true, a.dim <= 128};
    if (a.nq <= 64) return {1, 2, 4, 1, true, a.dim <= 128};
    if (a.nq <= 128) return {2, 2, 2, 2, true, a.dim <= 128};
    if (a.dim > kWholeDim) return {2, 4, 1, 4, true, false};
    if (a.nq <= 1024) return {4, 2, 1, 4, true, true};
    return {4, 2, 1, 4, false, true};
}

// The sample of a call's queries: every (nq / S)-th, and all their partitions as a round's items, by partition, then query.
__device__ inline int sample_query(int s, int S, int nq) { return (int)((int64_t)nq * s / S); }
__global__ __launch_bounds__(256) void sample_items_kernel(const float* __restrict__ query, int nq, int dim, int B, int S, float* __restrict__ rows,
                                                           int32_t* __restrict__ items, uint32_t* __restrict__ count, uint32_t* __restrict__ ticket, uint32_t* __restrict__ last_round) {
    const int at = blockIdx.x * 256 + threadIdx.x, all = gridDim.x * 256;
    for (int e = at; e < S * dim; e += all) rows[e] = query[(int64_t)sample_query(e / dim, S, nq) * dim + e % dim];
    for (int e = at; e < S * B; e += all) items[e] = sample_query(e % S, S, nq) * B + e / S;
    // (nearest query of the sample from below, and whether it is this one)
    for (int q = at; q < nq; q += all) {
        const int s = (int)(((int64_t)q * S + S - 1) / nq);
        last_round[q] = s < S && sample_query(s, S, nq) == q ? kSampleRound : 0u;
    }
    if (at == 0) *count = (uint32_t)(S * B);
    if (at < kMostDies) ticket[at * kTicketStride] = 0;
}
// Whether more than `most` of the sample's (query, partition) pairs have bounds within the query's k-th result.
__global__ __launch_bounds__(256) void sample_decide_kernel(const uint32_t* __restrict__ bounds, int S, int nq, int B, int parts, const float* __restrict__ worst,
                                                            int64_t worst_stride, float most, uint32_t* __restrict__ skip) {
    __shared__ uint32_t s_need;
    if (threadIdx.x == 0) s_need = 0;
    __syncthreads();
    uint32_t need = 0;
    for (int e = threadIdx.x; e < B * S; e += 256) {
        const int b = e / S, s = e % S;
        uint32_t v = kInf;
        for (int p = 0; p < parts; p++) v = min(v, bounds[((int64_t)b * parts + p) * S + s]);
        need += __builtin_bit_cast(float, v) > worst[(int64_t)sample_query(s, S, nq) * worst_stride] ? 0u : 1u;
    }
    need = wave_sum_u32(need);
    if ((threadIdx.x & 63) == 0) atomicAdd(&s_need, need);
    __syncthreads();
    if (threadIdx.x == 0) { skip[0] = (float)s_need > most * (float)(B * S) ? 1u : 0u; skip[1] = s_need; }
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct Room { size_t header, counts, qinfo, frags, bounds, limits, last, items, part_counts, near, left, sample, sample_rows, total; int steps, tiles, parts; };
// The sample as a call of its own, over every (B / kSampleParts)-th partition.
constexpr int kSampleParts = 12;
int sample_stride(const QueryArgs& a) { return a.B / min(a.B, kSampleParts); }
QueryArgs sample_call(const QueryArgs& a, const float* rows) {
    QueryArgs c = a;
    c.query = rows;
    c.nq = a.pick_sample;
    c.B = (a.B + sample_stride(a) - 1) / sample_stride(a);
    c.k = 1;
    c.kcap = 0;                           // (nothing of it is kept, so nothing to clear)
    c.part = nullptr;
    c.pick_sample = c.pick_near = c.pick_confirm = 0;
    return c;
}
// Items a die's run of a round's list holds at most.
int64_t left_cap(const QueryArgs& a) { return ((int64_t)a.nq * a.B + a.xcds - 1) / a.xcds; }
Room room_of(const QueryArgs& a) {
    Room r;
    r.steps = (a.dim + 2 * kStep - 1) / (2 * kStep) * 2;       // an even number of them
    // (whole groups of the query tiles a wavefront takes at a time)
    const int group = shape_of(a).ct;
    r.tiles = (a.nq + kTile * group - 1) / (kTile * group) * group;
    // parts of a partition: 64 k in all, as far as that leaves them a row tile each and a query 2048 of them
    const int64_t row_tiles = max((int64_t)1, a.ppb / 128);
    r.parts = 1;
    while (2 * r.parts <= row_tiles && (int64_t)a.B * r.parts < 64 * (int64_t)a.k && (int64_t)a.B * r.parts * 2 <= kMostParts) r.parts *= 2;
    size_t o = 0;
    r.header = o; o += align256((size_t)(kCentre + r.steps * kStep) * 4);
    r.counts = o; o += align256(kPickCountWords * 4);
    r.qinfo = o;  o += align256((size_t)r.tiles * kTile * sizeof(float2));
    r.frags = o;  o += align256((size_t)r.tiles * r.steps * 64 * 16);
    r.bounds = o; o += align256((size_t)a.B * r.parts * a.nq * 4);
    r.limits = o; o += align256((size_t)(kLimits + 3) * a.nq * 4);
    r.last = o;   o += align256((size_t)a.nq * 4);
    r.items = o;  o += align256((size_t)a.nq * a.B * 4);
    r.part_counts = o; o += align256((size_t)a.B * ((a.nq + kListQueries - 1) / kListQueries) * 4);
    r.near = o;   o += a.pick_near || a.pick_confirm ? align256(near_bytes(a)) : 0;
    r.left = o;   o += a.pick_confirm ? align256((size_t)2 * left_cap(a) * a.xcds * 4) : 0;
    r.sample = r.sample_rows = o;
    if (a.pick_sample) {
        o += room_of(sample_call(a, nullptr)).total;
        r.sample_rows = o; o += align256((size_t)a.pick_sample * a.dim * 4);
    }
    r.total = o;
    return r;
}

}  // namespace

bool bounds_supported(const QueryArgs& a) {
    return !a.blind && !a.counters && a.dim >= 8 && a.dim <= 4096 && a.nq >= 1 && a.B >= 2 && a.B <= kMostParts &&
           ((int64_t)a.nq + 128) * (a.dim + 32) < (1LL << 30) &&      // (the rounded queries are addressed by 32 bits)
           (int64_t)a.nq * a.B < 0x7fffffffLL && (a.ppb + kTile - 1) / kTile * (int64_t)a.B < 0x7fffffffLL;
}

// Of a partition, those of its last row tile that hold no rows among them.
static int64_t near_tiles_of(const QueryArgs& a) {
    const Shape y = shape_of(a);
    const int R = kTile * y.rt * y.wr;
    return (a.ppb + R - 1) / R * (R / near_rows(y.rt));
}

size_t bounds_bytes(const QueryArgs& a) { return room_of(a).total; }

size_t near_bytes(const QueryArgs& a) {
    return (size_t)near_tiles_of(a) * a.B * a.nq * 4;
}

// us.  The constants are half of what the product reaches (400000 rows of 128, 4096 queries: 1.04 PFLOP/s; 512 columns, 32 queries: 5.1 TB/s;
// 10M rows of 96, 512 queries, with the bounds of near tiles: 0.51 PFLOP/s and 1.9 TB/s): listing and limits come to the rest, and rounds
// are not to be chosen where they gain little.  12 us: packing the queries and the launches.
double bounds_cost(const QueryArgs& a) {
    const Shape y = shape_of(a);
    const int R = kTile * y.rt * y.wr;
    const double dim = (double)((a.dim + 2 * kStep - 1) / (2 * kStep) * 2 * kStep);
    const double rows = (double)((a.ppb + R - 1) / R * R) * (double)a.B;
    const double passes = y.one ? 1.0 : ceil((double)a.nq / (double)(kTile * y.ct * y.wc));
    const double queries = ceil((double)a.nq / (kTile * y.ct)) * (kTile * y.ct);
    return 12.0 + fmax(2.0 * rows * queries * dim / 500e6, passes * rows * (double)a.dim * 4.0 / 3e6);
}

static int pack(const QueryArgs& a, const Room& r, char* ws, hipStream_t s) {
    PackArgs p{a.query, a.data, a.N, a.nq, a.dim, r.steps, r.tiles, (Header*)(ws + r.header),
               (float2*)(ws + r.qinfo), (_Float16*)(ws + r.frags), (uint32_t*)(ws + r.bounds), (int64_t)a.B * r.parts * a.nq, (uint32_t*)(ws + r.near),
               (a.pick_near || a.pick_confirm) && shape_of(a).rt * kTile < near_rows(shape_of(a).rt) ? (int64_t)near_bytes(a) / 4 : 0,
               a.part, (int64_t)a.nq * a.B * a.kcap};
    const int64_t clear = (p.num_part + p.num_bounds + p.num_near + kPackThreads * 16 - 1) / (kPackThreads * 16);
    const unsigned blocks = (unsigned)max((int64_t)r.tiles, min((int64_t)2048, clear));
    const size_t lds = (size_t)3 * r.steps * kStep * 4;
    if (a.dim % 8 == 0) hipLaunchKernelGGL(pack_queries_kernel<true>, dim3(blocks), dim3(kPackThreads), lds, s, p);
    else hipLaunchKernelGGL(pack_queries_kernel<false>, dim3(blocks), dim3(kPackThreads), lds, s, p);
    DCIH_HIP(hipGetLastError());
    return 0;
}

template <int RT, int CT, int WR, int WC, int COLUMNS, int WAVES, bool ONE, int QD = 2>
static int launch_stream(const BoundArgs& p, int xcds, hipStream_t s) {
    constexpr int R = kTile * RT * WR, NT = 128 * WR * WC, kColumnSteps = COLUMNS / kStep;
    BoundArgs a = p;
    // stretches of columns of about the same length
    const int stretches = ONE ? 1 : (p.steps + kColumnSteps - 1) / kColumnSteps;
    a.column_steps = (p.steps + QD * stretches - 1) / (QD * stretches) * QD;
    const size_t lds = (size_t)2 * R * 4 + 4 * WR * WC * 4 + (size_t)p.steps * kStep * 4 + (size_t)2 * R * a.column_steps * kStep * 2;
    a.row_tiles = (int)((p.ppb + R - 1) / R);
    // as many workgroups as the device holds at a time
    const int per_cu = max(1, min((int)(160 * 1024 / lds), WAVES * 4 / (NT / 64)));
    const int64_t grid = min((int64_t)a.row_tiles * a.num_parts, (int64_t)xcds * 32 * per_cu);
    a.next_part = (int)(grid / a.row_tiles);
    a.next_tile = (int)(grid % a.row_tiles);
    static DeviceOnce once;
    const int rc = once.run([]() -> int {
        DCIH_HIP(hipFuncSetAttribute((const void*)bounds_stream_kernel<RT, CT, WR, WC, COLUMNS, WAVES, ONE, true, QD>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        DCIH_HIP(hipFuncSetAttribute((const void*)bounds_stream_kernel<RT, CT, WR, WC, COLUMNS, WAVES, ONE, false, QD>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        return 0;
    });
    if (rc) return rc;
    if (p.dim % 8 == 0) hipLaunchKernelGGL((bounds_stream_kernel<RT, CT, WR, WC, COLUMNS, WAVES, ONE, true, QD>), dim3((unsigned)grid), dim3(NT), lds, s, a);
    else hipLaunchKernelGGL((bounds_stream_kernel<RT, CT, WR, WC, COLUMNS, WAVES, ONE, false, QD>), dim3((unsigned)grid), dim3(NT), lds, s, a);
    DCIH_HIP(hipGetLastError());
    return 0;
}

static int products(const QueryArgs& a, const Room& r, char* ws, int64_t step, const uint32_t* skip, hipStream_t s) {
    BoundArgs p{a.data, a.N, a.ppb, step, a.dim, r.steps, a.nq, r.tiles, 0, 0, 0, a.B, 0, r.parts,
                (const Header*)(ws + r.header), (const float2*)(ws + r.qinfo), (const _Float16*)(ws + r.frags),
                (uint32_t*)(ws + r.bounds), a.pick_near || a.pick_confirm ? (uint32_t*)(ws + r.near) : nullptr, skip};
    const Shape y = shape_of(a);
    if (!y.stream) {
        constexpr int R = 128;
        p.row_tiles = (int)((p.ppb + R - 1) / R);
        const dim3 grid((unsigned)((int64_t)p.row_tiles * a.B));
        const size_t lds = (size_t)R * 4 + 2 * 4 * 4 + (size_t)p.steps * kStep * 4 + (size_t)R * p.steps * kStep * 2;
        static DeviceOnce once;
        const int rc_attr = once.run([]() -> int {
            DCIH_HIP(hipFuncSetAttribute((const void*)bounds_resident_kernel<4, 2, 4, 2, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            DCIH_HIP(hipFuncSetAttribute((const void*)bounds_resident_kernel<4, 2, 4, 2, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            return 0;
        });
        if (rc_attr) return rc_attr;
        if (a.dim % 8 == 0) hipLaunchKernelGGL((bounds_resident_kernel<4, 2, 4, 2, true>), grid, dim3(256), lds, s, p);
        else hipLaunchKernelGGL((bounds_resident_kernel<4, 2, 4, 2, false>), grid, dim3(256), lds, s, p);
        DCIH_HIP(hipGetLastError());
        return 0;
    }
    // (COLUMNS is what the registers hold that are read ahead into; longer rows come in stretches)
    const int columns = r.steps * kStep;
    if (y.ct == 1) {
        if (columns <= 64) return launch_stream<1, 1, 4, 1, 64, 4, true>(p, a.xcds, s);
        return columns <= 128 ? launch_stream<1, 1, 4, 1, 128, 4, true>(p, a.xcds, s) : launch_stream<1, 1, 4, 1, 64, 4, false>(p, a.xcds, s);
    }
    if (y.wr == 4) {
        if (columns <= 64) return launch_stream<1, 2, 4, 1, 64, 4, true>(p, a.xcds, s);
        return columns <= 128 ? launch_stream<1, 2, 4, 1, 128, 4, true>(p, a.xcds, s) : launch_stream<1, 2, 4, 1, 64, 4, false>(p, a.xcds, s);
    }
    if (y.wr == 2) return columns <= 128 ? launch_stream<2, 2, 2, 2, 128, 3, true>(p, a.xcds, s) : launch_stream<2, 2, 2, 2, 64, 4, false>(p, a.xcds, s);
    // (these have one multiplying wavefront per SIMD: as many steps of the queries ahead as divide the rows' steps)
    const bool fours = r.steps % 4 == 0;
    if (y.ct == 4) return fours ? launch_stream<2, 4, 1, 4, 256, 2, false, 4>(p, a.xcds, s) : launch_stream<2, 4, 1, 4, 256, 2, false>(p, a.xcds, s);
    if (columns <= 128) {
        if (fours) return launch_stream<4, 2, 1, 4, 128, 2, true, 4>(p, a.xcds, s);
        return r.steps % 6 == 0 ? launch_stream<4, 2, 1, 4, 128, 2, true, 6>(p, a.xcds, s) : launch_stream<4, 2, 1, 4, 128, 2, true>(p, a.xcds, s);
    }
    return fours ? launch_stream<4, 2, 1, 4, 256, 2, true, 4>(p, a.xcds, s) : launch_stream<4, 2, 1, 4, 256, 2, true>(p, a.xcds, s);
}

int pack_bounds(const QueryArgs& a, void* ws, hipStream_t s) { return pack(a, room_of(a), (char*)ws, s); }

int partition_bounds(const QueryArgs& a, void* ws_, hipStream_t s) {
    char* ws = (char*)ws_;
    const Room r = room_of(a);
    return products(a, r, ws, a.ppb, a.pick_sample ? (const uint32_t*)(ws + r.counts) + kSkipWord : nullptr, s);
}

int sample_items(const QueryArgs& a, void* ws_, Picked& p, hipStream_t s) {
    char* ws = (char*)ws_;
    const Room r = room_of(a);
    uint32_t* count = (uint32_t*)(ws + r.counts) + kSampleWord;
    hipLaunchKernelGGL(sample_items_kernel, dim3(32), dim3(256), 0, s, a.query, a.nq, a.dim, a.B, a.pick_sample, (float*)(ws + r.sample_rows),
                       (int32_t*)(ws + r.items), count, (uint32_t*)(ws + r.counts) + kTicketWord, (uint32_t*)(ws + r.last));
    DCIH_HIP(hipGetLastError());
    p = Picked{(const int32_t*)(ws + r.items), count, (const uint32_t*)(ws + r.last), (uint32_t*)(ws + r.counts) + kTicketWord, nullptr, nullptr, nullptr, 0, 0, 0};
    return 0;
}

int sample_decide(const QueryArgs& a, void* ws_, hipStream_t s) {
    char* ws = (char*)ws_;
    const Room r = room_of(a);
    const QueryArgs c = sample_call(a, (const float*)(ws + r.sample_rows));
    const Room rc_room = room_of(c);
    char* ws_c = ws + r.sample;
    int rc = pack(c, rc_room, ws_c, s);
    if (!rc) rc = products(c, rc_room, ws_c, (int64_t)sample_stride(a) * a.ppb, nullptr, s);
    if (rc) return rc;
    hipLaunchKernelGGL(sample_decide_kernel, dim3(1), dim3(256), 0, s, (const uint32_t*)(ws_c + rc_room.bounds), c.nq, a.nq, c.B, rc_room.parts,
                       (const float*)a.out_dists + (a.k - 1), (int64_t)a.k, a.pick_most, (uint32_t*)(ws + r.counts) + kSkipWord);
    DCIH_HIP(hipGetLastError());
    return 0;
}

// How far rows count in a round of confirm.hip's: in round 1 as picked, later one of two rows in turn.
static float* near_limits(char* ws, const Room& r, int nq, int round) {
    return (float*)(ws + r.limits) + (int64_t)(round <= 0 ? kLimits : kLimits + 1 + (round & 1)) * nq;
}
int pick_items(const QueryArgs& a, void* ws_, int round, int rounds, hipStream_t s) {
    char* ws = (char*)ws_;
    const Room r = room_of(a);
    uint32_t* bounds = (uint32_t*)(ws + r.bounds);
    uint32_t* limits = (uint32_t*)(ws + r.limits);
    uint32_t* last = (uint32_t*)(ws + r.last);
    if (round == 0) {
        const int S = a.B * r.parts, per = a.nq >= 8192 && S <= 512 ? 16 : 4;
        const dim3 grid((unsigned)((a.nq + per - 1) / per));
        const int near_rank = min(32 * a.pick_rank, max(4 * a.pick_rank, S / 2));
        const int tight_rank = 4 * a.pick_rank;
#define DCIH_LIMITS(V)                                                                                              \
    hipLaunchKernelGGL(pick_limits_kernel<V>, grid, dim3(256), (size_t)S * (per + 1) * 4, s, bounds, S, a.nq, per, \
                       a.pick_rank, near_rank, a.pick_confirm ? tight_rank : near_rank, a.pick_flat, limits, last, \
                       a.blind_word)
        if (S <= 64) DCIH_LIMITS(1); else if (S <= 128) DCIH_LIMITS(2); else if (S <= 256) DCIH_LIMITS(4);
        else if (S <= 512) DCIH_LIMITS(8); else if (S <= 1024) DCIH_LIMITS(16); else DCIH_LIMITS(32);
#undef DCIH_LIMITS
        DCIH_HIP(hipGetLastError());
    }
    const int groups = (a.nq + kListQueries - 1) / kListQueries;
    ListArgs p{bounds, limits, a.pick_sample ? (const uint32_t*)(ws + r.counts) + kSkipWord : nullptr, a.out_dists + (a.k - 1), a.k, last, a.B, r.parts, a.nq, groups, round, rounds, a.pick_near,
                 (uint32_t*)(ws + r.counts) + kRestsWord, a.pick_confirm ? a.confirm_word : nullptr, a.confirm_tag, a.pick_confirm ? a.xcds : 0, near_limits(ws, r, a.nq, round - 1), near_limits(ws, r, a.nq, round),
               (int32_t*)(ws + r.items), (uint32_t*)(ws + r.counts) + round, (uint32_t*)(ws + r.part_counts),
               (uint32_t*)(ws + r.counts) + kTicketWord};
    const dim3 grid((unsigned)((int64_t)a.B * groups));
    hipLaunchKernelGGL(list_items_kernel<true>, grid, dim3(256), 0, s, p);
    hipLaunchKernelGGL(list_items_kernel<false>, grid, dim3(256), 0, s, p);
    DCIH_HIP(hipGetLastError());
    return 0;
}

int confirm_round(QueryArgs& a, void* ws_, hipStream_t s) {
    char* ws = (char*)ws_;
    const Room r = room_of(a);
    uint32_t* counts = (uint32_t*)(ws + r.counts);
    a.left = nullptr;
    const int rc = confirm_items(a, a.pick_sample ? counts + kSkipWord : nullptr, counts + kRestsWord, (int32_t*)(ws + r.left), counts + kLeftWord, left_cap(a), s);
    a.left = (const int32_t*)(ws + r.left);
    a.left_count = counts + kLeftWord;
    a.left_cap = left_cap(a);
    return rc;
}

Picked picked_items(const QueryArgs& a, void* ws_, int round) {
    char* ws = (char*)ws_;
    const Room r = room_of(a);
    Picked p{(const int32_t*)(ws + r.items), (const uint32_t*)(ws + r.counts) + round, (const uint32_t*)(ws + r.last),
             (uint32_t*)(ws + r.counts) + kTicketWord, nullptr, nullptr, nullptr, 0, 0, 0};
    if (a.pick_near || a.pick_confirm) {
        p.near_bounds = (const uint32_t*)(ws + r.near);
        // (later rounds': the k-th distance found so far, as list_items_kernel has noted it for confirm.hip)
        p.confirm_limit = near_limits(ws, r, a.nq, round);
        p.near_limit = round == 0 ? (const float*)(ws + r.limits) + (int64_t)(kLimits - 1) * a.nq : (a.pick_confirm ? p.confirm_limit : a.out_dists + (a.k - 1));
        p.near_stride = round && !a.pick_confirm ? a.k : 1;
        p.near_shift = near_rows(shape_of(a).rt) == 64 ? 6 : 7;
        p.near_tiles = (int)near_tiles_of(a);
    }
    return p;
}

}  // namespace dcih
