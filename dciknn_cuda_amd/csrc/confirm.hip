// Items of a call's rounds (bounds.hip) that need no traversal: one workgroup per (query, partition) finds the rows that can matter to
// the round and whether the traversal would promote them before it stops.
//
// In a round only rows no further away than the query's limit count, one or two of a partition.  Under composite m such a row is promoted
// with the last of its L windows, whose priority is the largest of theirs.  All windows up to that priority, of which 2L binary searches
// give the number, are consumed by the step that promotes the row, and it is a candidate unless the loop of dci_query_single_point_by_block
// (src/dci_cuda_kernel.cu:401-626) stops before.  That takes at least max(k, max_candidates) promotions by a window's first lane
// (k of them once the step limit is reached, :598-607) among as many windows of every composite.  These cover one run of
// places of every simple index's slice, and their promotions are the points that lie inside all L runs of a composite.  Near rows come early, so these
// points are few, mostly fewer than a stop takes: then all near rows are candidates, and nothing has to be ordered, replayed or looked
// up point by point.  Where they are not, the promotions' steps are found one by one (2L searches each) and the stop with them, if the tables here hold them;
// else, and where more rows are near than they hold, the item is left to the traversal kernels, in a list per die.
//
// The count may be too high, never too low: each composite's windows are those up to some priority that takes at least as many steps as the
// last near row, and a point counts once per composite.
//
// Bound by chains of dependent reads (searches, then rows, then positions), hence by the items a CU holds: few registers, little LDS.
// 10000 queries on 1M rows of 128, 58 partitions, windows of 2: 113000 items, 6.1 ms of the batch kernel, 2.5 ms of one wavefront each here and 0.4 by
// eight for 600 of them.  1000 queries at the defaults, 10200 items of 10000 points: 1.85 ms of the dense kernel, 0.19 ms.  Of the 2.0 ms that 97000
// items take: starting them and near tiles 0.3, rows 0.2, searches 0.5, scan 0.6, promotions in order 0.3.
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "traverse_common.h"

namespace dcih {

namespace {

constexpr int kNearTiles = 16;       // near tiles and
constexpr int kNearRows = 32;        // near rows that an item may have
constexpr int kRuns = 4;             // rows of positions that the scan of a run tests together
// What the tables of a workgroup of NT threads hold: rows to compare, or places that the first rows of positions leave; points inside all runs;
// and of those where they have to be put in order.  One wavefront's are small: 24 of them to a CU, what takes longer is the larger workgroups'.
constexpr int listed_cap(int nt) { return nt == kWave ? 1024 : 4096; }
constexpr int found_cap(int nt) { return nt == kWave ? 512 : 2048; }
constexpr int event_cap(int nt) { return nt == kWave ? 64 : (nt == 256 ? 128 : 512); }

struct ConfirmLayout { int off_idx, off_consumed, off_near, off_comp, off_list, off_found; size_t lds_bytes; };
enum CMisc { cTiles = 0, cRows, cNear, cListed, cCount, cFound, cTry, cArmed, cMost, cMiscWords = 12 };

ConfirmLayout confirm_layout(const QueryArgs& a, int nt) {
    const int I = a.M * a.L;
    ConfirmLayout y;
    int o = cMiscWords * 4 + kNearTiles * 4;
    y.off_idx = o;      o += 6 * I * 4;                      // per simple index: position, projection, the run's first place and its end
    y.off_consumed = o; o += 2 * 2 * I * 4;                  // per stream: windows consumed, and those of a trial
    y.off_comp = o;     o += 5 * a.M * 4;                    // per composite: priority, windows consumed, those of a trial, near rows, points found
    o = (o + 15) & ~15;
    y.off_near = o;     o += kNearRows * 8 + kNearRows * a.M * 4;      // near rows: (distance, point), and their priorities by composite
    y.off_list = o;     o += listed_cap(nt) * 2;
    y.off_found = o;    o += found_cap(nt) * 2;
    y.lds_bytes = (size_t)((o + 15) & ~15);
    return y;
}

struct ConfirmArgs {
    const float* skeys; const int32_t* sids; const uint16_t* inv; const uint16_t* rpos;
    const float* data; const float* query; const float* qproj;
    int64_t N, ppb, stop_at, max_cand;
    int dim, M, L, B, T, nq, k_stop, kcap, xcds;
    unsigned T_magic;
    unsigned long long* part;
    struct { const int32_t* picked; const uint32_t* picked_count; const int32_t* left; const uint32_t* left_count; int64_t left_cap; int xcds; } from;
    const uint32_t* skip;
    uint32_t* rests;                      // (set before the launch where earlier rounds have left most of their items), and whether round 1's rested
    int pilot;                            // 1: a few items ahead, only to be counted; 2: the launch after that one
    const uint32_t* near_bounds; const float* near_limit; int64_t near_stride;
    int near_shift, near_tiles;
    int32_t* left; uint32_t* left_count; int64_t left_cap;
    int64_t second_cap;                   // items of a die that the second pass takes
    int pilot_at, stats_at;               // where from left_count on the pilot's counts lie, and those that later rounds go by
    ConfirmLayout y;
};

// SCAN: the points are looked for where windows alone do not settle it.
template <int NT, bool SCAN>
__device__ __forceinline__ bool confirm_item(const ConfirmArgs& a, unsigned char* smem, const int b, const int qi) {
    constexpr int kWaves = NT / kWave, kListed = listed_cap(NT), kFound = found_cap(NT), kEvents = event_cap(NT);
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(1))) const u32x4 g_u32x4;
    const int I = a.M * a.L, M = a.M, L = a.L, T = a.T, S = 2 * a.L;
    uint32_t* misc = reinterpret_cast<uint32_t*>(smem);
    uint32_t* tiles = misc + cMiscWords;
    int* s_p = reinterpret_cast<int*>(smem + a.y.off_idx);
    float* s_qp = reinterpret_cast<float*>(s_p + I);
    int* s_lo = reinterpret_cast<int*>(s_qp + I);
    int* s_hi = s_lo + I;
    uint32_t* s_lo2 = reinterpret_cast<uint32_t*>(s_hi + I);      // the same as packed 16-bit pairs: first place and length less one, twice
    uint32_t* s_len2 = s_lo2 + I;
    int* s_c = reinterpret_cast<int*>(smem + a.y.off_consumed);
    int* s_try = s_c + 2 * I;
    float* s_rho = reinterpret_cast<float*>(smem + a.y.off_comp);
    uint32_t* s_have = reinterpret_cast<uint32_t*>(s_rho + M);
    uint32_t* s_sum = s_have + M;
    uint32_t* s_rows = s_sum + M;
    uint32_t* s_found = s_rows + M;
    unsigned long long* near = reinterpret_cast<unsigned long long*>(smem + a.y.off_near);
    uint32_t* prio = reinterpret_cast<uint32_t*>(near + kNearRows);
    uint16_t* list = reinterpret_cast<uint16_t*>(smem + a.y.off_list);
    uint16_t* found = reinterpret_cast<uint16_t*>(smem + a.y.off_found);
    uint32_t* ev_prio = reinterpret_cast<uint32_t*>(list);      // (when the list is done with)
    uint32_t* ev_window = ev_prio + kEvents;
    uint32_t* ev_point = ev_window + kEvents;
    uint32_t* ev_step = ev_point + kEvents;
    static_assert(kListed * 2 >= kEvents * 16, "room of the promotions");

    // (made opaque again in every phase, so that what derives from them is not computed ahead and carried through the others)
    int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    auto next_phase = [&]() {
        int leave_now = 0;
        asm volatile("" : "+s"(leave_now));
        asm volatile("" : "+v"(tid));
        lane = tid & (kWave - 1);
        return leave_now != 0;      // (never)
    };
    const int64_t item = (int64_t)qi * a.B + b, off = (int64_t)b * a.ppb;
    const int n = (int)min(a.N - off, a.ppb);
    unsigned long long* part_out = a.part + item * a.kcap;
    auto div_T = [&](int d) { return T > 1 ? (int)__umulhi((uint32_t)d, a.T_magic) : d; };
    // the window of simple index i that holds position pos, its first position and the place in it
    auto window_of = [&](int i, int pos, int& side, int& j, int& t) {
        const int p = s_p[i];
        int start;
        if (pos > p) {
            const int d = pos - (p + 1);
            side = 1; j = div_T(d); start = p + 1 + j * T;
        } else {
            side = 0; j = div_T(p - pos); start = p - T + 1 - j * T;
        }
        t = pos - start;
        return max(start, 0);
    };

    // ---- near tiles, the query's positions (:279-297) -----------------------------
    __syncthreads();
    if (tid < cMiscWords) misc[tid] = 0;
    __syncthreads();
    const float most = a.near_limit[(int64_t)qi * a.near_stride];
    if (n > 0) {
        const uint32_t* bounds = a.near_bounds + (int64_t)b * a.near_tiles * a.nq + qi;
        const int all = (n + (1 << a.near_shift) - 1) >> a.near_shift;
        for (int t = tid; t < all; t += NT)
            if (!(__builtin_bit_cast(float, bounds[(int64_t)t * a.nq]) > most)) {
                const uint32_t slot = atomicAdd(&misc[cTiles], 1u);
                if (slot < (uint32_t)kNearTiles) tiles[slot] = (uint32_t)t;
            }
    }
    __syncthreads();
    const int ntiles = (int)misc[cTiles];
    auto nothing = [&]() { for (int j = tid; j < a.kcap; j += NT) part_out[j] = ~0ull; };
    if (ntiles == 0) { nothing(); return true; }
    if (ntiles > kNearTiles) return false;

    if (next_phase()) return false;
    // ---- near rows: by the squares of their first 32 elements, which rule out most of a tile, then whole -----------
    const bool vec4 = rows_vec4(a.data, a.dim);
    const float* q = a.query + (int64_t)qi * a.dim;
    const float* base = a.data + off * a.dim;
    const int rows = ntiles << a.near_shift, in_tile = (1 << a.near_shift) - 1;
    {
        // (what a distance is rounded by is far below the factor; squares that underflow say nothing; a limit that is not a number is none)
        const float most2 = most == most ? fmaxf(most * most * 1.0001f, 1e-30f) : __builtin_inff();
        const bool head = vec4 && a.dim >= 64;
        const int sl = lane & 7;
        float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
        if (head) { q0 = q[4 * sl]; q1 = q[4 * sl + 1]; q2 = q[4 * sl + 2]; q3 = q[4 * sl + 3]; }
        constexpr int U = 8;
        for (int r0 = wave * 8 * U; r0 < rows; r0 += kWaves * 8 * U) {
            int pts[U];
            float s2[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int r = min(r0 + u * 8 + (lane >> 3), rows - 1);
                pts[u] = (int)(tiles[r >> a.near_shift] << a.near_shift) + (r & in_tile);
                s2[u] = 0.f;
            }
            if (head) {
                v4f x[U];
#pragma unroll
                for (int u = 0; u < U; u++) x[u] = *reinterpret_cast<const v4f*>(base + (int64_t)min(pts[u], n - 1) * a.dim + 4 * sl);
#pragma unroll
                for (int u = 0; u < U; u++) {
                    float d = x[u].x - q0; s2[u] = __builtin_fmaf(d, d, s2[u]);
                    d = x[u].y - q1; s2[u] = __builtin_fmaf(d, d, s2[u]);
                    d = x[u].z - q2; s2[u] = __builtin_fmaf(d, d, s2[u]);
                    d = x[u].w - q3; s2[u] = __builtin_fmaf(d, d, s2[u]);
                    s2[u] += lane_xor<4>(s2[u]); s2[u] += lane_xor<2>(s2[u]); s2[u] += lane_xor<1>(s2[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (sl == 0 && r0 + u * 8 + (lane >> 3) < rows && pts[u] < n && !(s2[u] > most2)) {
                    const uint32_t slot = atomicAdd(&misc[cRows], 1u);
                    if (slot < (uint32_t)kListed) list[slot] = (uint16_t)pts[u];
                }
            }
        }
    }
    __syncthreads();
    const int compared = (int)misc[cRows];
    if (compared > kListed) return false;
    // (the sums and their order are those of wave_row_dists)
    auto keep = [&](float d, int pt) {
        if (d > most) return;
        const uint32_t slot = atomicAdd(&misc[cNear], 1u);
        if (slot < (uint32_t)kNearRows) near[slot] = ((unsigned long long)__builtin_bit_cast(uint32_t, d) << 32) | (uint32_t)(off + pt);
    };
    if (compared > 4 * kWaves && vec4 && a.dim <= 128) {
        // 32 lanes to a row, eight rows each
        const int grp = lane >> 5, sl = lane & 31, j = sl * 4;
        const bool has = j < a.dim;
        float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
        if (has) { q0 = q[j]; q1 = q[j + 1]; q2 = q[j + 2]; q3 = q[j + 3]; }
        const float* from = base + (has ? j : 0);
        for (int c0 = wave * 16; c0 < compared; c0 += kWaves * 16) {
            v4f x[8];
            float acc[8];
#pragma unroll
            for (int r = 0; r < 8; r++) x[r] = *reinterpret_cast<const v4f*>(from + (int64_t)list[min(c0 + grp * 8 + r, compared - 1)] * a.dim);
#pragma unroll
            for (int r = 0; r < 8; r++) {
                float s2 = 0.f;
                float d = x[r].x - q0; s2 = __builtin_fmaf(d, d, s2);
                d = x[r].y - q1; s2 = __builtin_fmaf(d, d, s2);
                d = x[r].z - q2; s2 = __builtin_fmaf(d, d, s2);
                d = x[r].w - q3; s2 = __builtin_fmaf(d, d, s2);
                acc[r] = has ? s2 : 0.f;
            }
            float v4[4], v2[2];
            const bool u16 = (sl & 16) != 0, u8 = (sl & 8) != 0, u4 = (sl & 4) != 0;
#pragma unroll
            for (int i = 0; i < 4; i++) v4[i] = (u16 ? acc[i + 4] : acc[i]) + lane_xor<16>(u16 ? acc[i] : acc[i + 4]);
#pragma unroll
            for (int i = 0; i < 2; i++) v2[i] = (u8 ? v4[i + 2] : v4[i]) + lane_xor<8>(u8 ? v4[i] : v4[i + 2]);
            float v = (u4 ? v2[1] : v2[0]) + lane_xor<4>(u4 ? v2[0] : v2[1]);
            v += lane_xor<2>(v);
            v += lane_xor<1>(v);
            const int c = c0 + grp * 8 + sl / 4;
            if ((sl & 3) == 0 && c < compared) keep(sqrtf(v), (int)list[c]);
        }
    } else {
        for (int c0 = wave * 4; c0 < compared; c0 += kWaves * 4) {
            const float* at[4];
            int pts[4];
            float d[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                pts[r] = __builtin_amdgcn_readfirstlane((int)list[min(c0 + r, compared - 1)]);
                at[r] = base + (int64_t)pts[r] * a.dim;
            }
            wave_row_dists<4>(at, q, a.dim, vec4, d, lane);
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (lane == 0 && c0 + r < compared) keep(d[r], pts[r]);
        }
    }
    __syncthreads();
    const int R = (int)misc[cNear];
    if (R == 0) { nothing(); return true; }
    if (R > kNearRows) return false;

    if (next_phase()) return false;
    // ---- where the query stands in every simple index -----------------------------
    // Searches by groups of lanes are shorter chains, by single lanes fewer instructions: where items fill the device, one wavefront each.
    auto lanes_for = [&](int searches) {
        int lg = NT == kWave ? 0 : 3;
        while (lg > 0 && (searches << lg) > NT) lg--;
        return lg;
    };
    uint32_t probes = 0;
    {
        const int lg = lanes_for(I), slots = kWave >> lg;
        for (int i0 = 0; i0 < I; i0 += slots * kWaves) {
            const int sl = lane >> lg, i = i0 + wave * slots + sl;
            const bool active = i < I;
            const float* key = a.skeys + (int64_t)(active ? i : 0) * a.N + off;
            const float qp = active ? a.qproj[(int64_t)i * a.nq + qi] : 0.f;
            int lo = 0;
            if (lg == 0) {
                for (int hi = active ? n : 0; lo < hi;) {
                    const int mid = (lo + hi) >> 1;
                    if (key[mid] < qp) lo = mid + 1; else hi = mid;
                }
            } else {
                lo = group_partition_point(0, n, active, lg, sl << lg, lane - (sl << lg), [&](int j) { return key[j] < qp; }, probes);
            }
            if (active && lane == (sl << lg)) { s_p[i] = lo - 1; s_qp[i] = qp; }
        }
    }
    for (int e = tid; e < R * M; e += NT) prio[e] = 0;
    for (int e = tid; e < 5 * M; e += NT) s_have[e - M] = 0;
    __syncthreads();
    if (next_phase()) return false;
    // ---- the last of the windows of every near row, per composite: the largest priority ------------------------------
    for (int e = tid; e < R * I; e += NT) {
        const int r = e / I, i = e - r * I, m = i / L;
        const int pos = (int)a.inv[(int64_t)i * a.N + off + (int)((uint32_t)near[r] - (uint32_t)off)];
        int side, j, t;
        const int kp = window_of(i, pos, side, j, t);
        atomicMax(&prio[r * M + m], __builtin_bit_cast(uint32_t, fabsf(a.skeys[(int64_t)i * a.N + off + kp] - s_qp[i])));
    }
    __syncthreads();
    if (next_phase()) return false;
    // ---- every near row by the composite of its smallest one: the priorities up to which windows are consumed ------------
    if (tid < R) {
        uint32_t least = kInfBits;
        int at = 0;
        for (int m = 0; m < M; m++)
            if (prio[tid * M + m] < least) { least = prio[tid * M + m]; at = m; }
        atomicMax(reinterpret_cast<uint32_t*>(&s_rho[at]), least);
        atomicAdd(&s_rows[at], 1u);
        atomicMax(&misc[cTry], least);
    }
    __syncthreads();
    if (misc[cTry] >= kInfBits) return false;      // (a row that no composite promotes)
    if (tid < M && s_rows[tid] == 0) s_rho[tid] = __builtin_bit_cast(float, misc[cTry]);
    if (next_phase()) return false;
    // ---- their number; a composite without near rows, or with earlier ones only, goes on until it has as many as the one that has most ---------
    uint32_t steps = 0;
    bool accept = false;
    uint32_t t_stop = 0xffffffffu;
    int64_t need = 0;
    // (a second time, where these take in more points than the tables hold, only those up to a part of the priority: the loop may have stopped by then)
    const float rho_all = __builtin_bit_cast(float, misc[cTry]);
    bool partial = false;
    for (;;) {
        constexpr int kTrials = 7;
        for (int trial = 0; trial < kTrials; trial++) {
            __syncthreads();
            const bool final = trial == kTrials - 1;
            auto open = [&](int m) {
                return trial == 0 || (!partial && (s_have[m] < steps || (s_rows[m] == 0 && trial < 3 && s_have[m] > steps + steps / 32 + 8)));
            };
            int order = 0, which = 0;      // (the open composites, four bits each)
            for (int m = 0; m < M; m++)
                if (open(m)) which |= m << (4 * order++);
            if (order == 0) break;      // (the same for every thread)
            const int units = order * S;
            const int lg = lanes_for(units), slots = kWave >> lg;
            for (int u0 = 0; u0 < units; u0 += slots * kWaves) {
                const int sl = lane >> lg, e = u0 + wave * slots + sl, at = min(e, units - 1) / S;
                const int m = (which >> (4 * at)) & 15, s = m * S + min(e, units - 1) - at * S;
                const uint32_t bits = __builtin_bit_cast(uint32_t, s_rho[m]);
                Stream st;
                st.key = a.skeys + (int64_t)(s >> 1) * a.N + off;
                st.n = n; st.T = T; st.p = s_p[s >> 1]; st.side = s & 1; st.q = s_qp[s >> 1];
                // (the last trial takes all windows)
                const int ns = stream_windows(n, T, st.p, st.side);
                int c = ns;
                if (!final) {
                    if (lg == 0) c = e < units ? count_below(st, bits, false, 0, ns, probes) : 0;
                    else c = group_partition_point(0, ns, e < units, lg, sl << lg, lane - (sl << lg), [&](int j) { return stream_prio_bits(st, j) <= bits; }, probes);
                }
                if (e < units && lane == (sl << lg)) {
                    s_try[s] = c;
                    atomicAdd(&s_sum[m], (uint32_t)c);
                }
            }
            __syncthreads();
            if (trial == 0 && !partial) {
                for (int m = 0; m < M; m++)
                    if (s_rows[m]) steps = max(steps, s_sum[m]);
                need = (int64_t)steps < a.stop_at ? max((int64_t)a.k_stop, a.max_cand) : (int64_t)a.k_stop;
                accept = (int64_t)M * steps < need;      // (a window promotes one point by its first lane at most)
                if (accept) break;
            }
            // (a trial that falls short is no use; of two that do not the smaller is kept)
            auto better = [&](int m) { return trial == 0 || (open(m) && (final || (s_sum[m] >= steps && (s_have[m] < steps || s_sum[m] < s_have[m])))); };
            for (int s = tid; s < M * S; s += NT)
                if (better(s / S)) s_c[s] = s_try[s];
            bool take = false;
            float rho = 0.f;
            uint32_t sum = 0;
            if (tid < M) {
                take = better(tid);
                sum = s_sum[tid];
                rho = s_rho[tid] * fminf(fmaxf(((float)steps + 1.0f) / ((float)sum + 1.0f), 0.25f), 4.0f) * (1.01f + 0.03f * (float)trial);
            }
            __syncthreads();
            if (tid < M) {
                if (take) s_have[tid] = sum;
                s_rho[tid] = rho;
                s_sum[tid] = 0;
            }
        }
        __syncthreads();
        if (!SCAN && !accept) return false;
        if (!accept) {
            if (next_phase()) return false;
            // ---- the runs of places they cover -----------------------------------------
            for (int i = tid; i < I; i += NT) {
                const int p1 = s_p[i] + 1;
                s_lo[i] = (int)max((int64_t)0, (int64_t)p1 - (int64_t)s_c[2 * i] * T);
                s_hi[i] = (int)min((int64_t)n, (int64_t)p1 + (int64_t)s_c[2 * i + 1] * T);
                s_lo2[i] = (uint32_t)s_lo[i] * 0x10001u;
                s_len2[i] = ((uint32_t)(s_hi[i] - s_lo[i] - 1) & 0xffffu) * 0x10001u;
            }
            {
                if (next_phase()) return false;
                uint32_t too_many = 0;
                // ---- the points inside all runs of a composite -------------
                // First the places of its first simple index's run, eight at a time, that lie inside the runs of the next few, as many as
                // leave about a hundred.
                bool all_rows = false;      // (too many were left: once more, by all rows)
                for (int m = 0; m < M; m++) {
                    __syncthreads();
                    if (tid == 0) misc[cListed] = 0;
                    bool empty = false;
                    int stage = 0;
                    float expect = 1.0f;
                    for (int h = 0; h < L; h++) {
                        const int len = s_hi[m * L + h] - s_lo[m * L + h];
                        empty = empty || len <= 0;
                        if (h == 0) expect = (float)len;
                        else if (h <= 2 || expect > 100.0f) { expect *= (float)len / (float)n; stage = h; }
                    }
                    stage = all_rows ? L - 1 : (stage <= kRuns ? min(L - 1, kRuns) : stage);
                    __syncthreads();
                    if (empty) continue;
                    const int64_t first_row = (int64_t)m * L * a.N + off;
                    const int run_lo = s_lo[m * L], run_hi = s_hi[m * L];
                    // (16-byte reads on their boundaries where the slices of all simple indices can be aligned together)
                    const int start = run_lo - ((a.N & 7) == 0 ? (int)((off + run_lo) & 7) : 0);
                    const int chunks = (run_hi - start + 7) >> 3;
                    const uint16_t* rp = a.rpos + first_row + start;
                    // (the rows of two chunks under way together; what is the same for all lanes in scalar registers)
                    const char* rows[kRuns];
                    u16x2 lo[kRuns], len[kRuns];
#pragma unroll
                    for (int u = 0; u < kRuns; u++) {
                        const int h = min(1 + u, stage);
                        rows[u] = reinterpret_cast<const char*>(rp + (int64_t)h * a.N);
                        lo[u] = __builtin_bit_cast(u16x2, __builtin_amdgcn_readfirstlane((int)s_lo2[m * L + h]));
                        len[u] = __builtin_bit_cast(u16x2, __builtin_amdgcn_readfirstlane((int)s_len2[m * L + h]));
                    }
                    auto read = [&](int c, u32x4 (&x)[kRuns]) {
                        const uint32_t from = (uint32_t)min(c, chunks - 1) * 16u;
#pragma unroll
                        for (int u = 0; u < kRuns; u++) x[u] = *(g_u32x4*)(rows[u] + from);
                    };
                    auto test = [&](u16x2 (&worst)[4], const u32x4& x, u16x2 lo, u16x2 len) {
                        const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                        for (int g = 0; g < 4; g++)
                            worst[g] = __builtin_elementwise_max(worst[g], __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, w[g]) - lo, len));
                    };
                    auto one_chunk = [&](int c, const u32x4 (&x)[kRuns]) {
                        u16x2 worst[4];
#pragma unroll
                        for (int g = 0; g < 4; g++) worst[g] = u16x2{0, 0};
                        if (c == 0 || c == chunks - 1) {      // places before the run's first or past its last
#pragma unroll
                            for (int g = 0; g < 4; g++) {
                                const int at = start + 8 * c + 2 * g;
                                worst[g] = u16x2{(uint16_t)(at < run_lo || at >= run_hi ? 0xffff : 0), (uint16_t)(at + 1 < run_lo || at + 1 >= run_hi ? 0xffff : 0)};
                            }
                        }
#pragma unroll
                        for (int u = 0; u < kRuns; u++) test(worst, x[u], lo[u], len[u]);
                        // the places that have passed: bit g the first one of pair g, bit 16 + g its second one
                        auto passed_of = [&]() {
                            uint32_t p = 0;
#pragma unroll
                            for (int g = 0; g < 4; g++) {
                                const uint32_t out = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(worst[g], u16x2{1, 1}));
                                p |= out << g;
                            }
                            return p ^ 0x000f000fu;
                        };
                        uint32_t passed = passed_of();
                        for (int h = kRuns + 1; h <= stage && passed; h++) {
                            const u32x4 one = *(g_u32x4*)(reinterpret_cast<const char*>(rp + (int64_t)h * a.N) + (uint32_t)c * 16u);
                            test(worst, one, __builtin_bit_cast(u16x2, s_lo2[m * L + h]), __builtin_bit_cast(u16x2, s_len2[m * L + h]));
                            passed = passed_of();
                        }
                        if (!passed) return;
                        uint32_t slot = atomicAdd(&misc[cListed], (uint32_t)__popc(passed));
                        for (; passed; passed &= passed - 1, slot++) {
                            const int bit = __ffs(passed) - 1;
                            if (slot < (uint32_t)kListed) list[slot] = (uint16_t)(start + 8 * c + 2 * (bit & 15) + (bit >> 4));
                        }
                    };
                    u32x4 x0[kRuns], x1[kRuns];
                    read(tid, x0);
                    for (int c = tid; c < chunks; c += 2 * NT) {
                        read(c + NT, x1);
                        one_chunk(c, x0);
                        read(c + 2 * NT, x0);
                        if (c + NT < chunks) one_chunk(c + NT, x1);
                    }
                    __syncthreads();
                    const int listed = (int)misc[cListed];
                    if (listed > kListed) {
                        if (NT < 512) return false;
                        if (stage == L - 1) {
                            too_many = (uint32_t)listed;
                            break;
                        }
                        all_rows = true;
                        m--;
                        continue;
                    }
                    if (next_phase()) return false;
                    // ---- then of those the ones inside all others
                    for (int e = tid; e < listed; e += NT) {
                        const int place = (int)list[e];
                        bool inside = true;
                        for (int h0 = stage + 1; h0 < L && inside; h0 += 4) {
                            int pos[4];
#pragma unroll
                            for (int u = 0; u < 4; u++) pos[u] = (int)a.rpos[first_row + (int64_t)min(h0 + u, L - 1) * a.N + place];
#pragma unroll
                            for (int u = 0; u < 4; u++) {
                                const int i = m * L + min(h0 + u, L - 1);
                                inside = inside && pos[u] >= s_lo[i] && pos[u] < s_hi[i];
                            }
                        }
                        if (!inside) continue;
                        const uint32_t slot = atomicAdd(&misc[cFound], 1u);
                        atomicAdd(&s_found[m], 1u);
                        if (slot < (uint32_t)kFound) found[slot] = (uint16_t)place;
                    }
                }
                __syncthreads();
                const int all = too_many ? (int)too_many : (int)misc[cFound];
                accept = !partial && !too_many && all < need;
                if (!accept && !too_many && all <= kFound && (!partial || all <= kEvents)) {
                    if (next_phase()) return false;
                    // ---- as many as a stop may take: of those only the ones whose last window holds them in its first lane count --------
                    // The last window of each, the largest (priority, simple index), and whether it holds the point in its first lane.
                    for (int e = tid; e < all; e += NT) {
                        int m = 0;
                        for (uint32_t end = s_found[0]; (uint32_t)e >= end; end += s_found[++m]) {}
                        const int place = (int)found[e];
                        const int64_t first_row = (int64_t)m * L * a.N + off + place;
                        const uint32_t pt = (uint32_t)(a.sids[first_row] - (int32_t)off);
                        uint32_t most_bits = 0, window = 0;
                        for (int h0 = 0; h0 < L; h0 += 4) {
                            uint32_t w4[4];
                            float kv[4];
#pragma unroll
                            for (int u = 0; u < 4; u++) {
                                const int h = min(h0 + u, L - 1), i = m * L + h;
                                int side, j, t;
                                const int kp = window_of(i, h == 0 ? place : (int)a.rpos[first_row + (int64_t)h * a.N], side, j, t);
                                kv[u] = a.skeys[(int64_t)i * a.N + off + kp];
                                w4[u] = (uint32_t)(t == 0 ? 1 << 22 : 0) | (uint32_t)h << 17 | (uint32_t)side << 16 | (uint32_t)j;
                            }
#pragma unroll
                            for (int u = 0; u < 4; u++) {
                                const uint32_t bits = __builtin_bit_cast(uint32_t, fabsf(kv[u] - s_qp[m * L + min(h0 + u, L - 1)]));
                                if (bits >= most_bits) { most_bits = bits; window = w4[u]; }
                            }
                        }
                        if (window >> 22) atomicAdd(&misc[cCount], 1u);
                        if (e < kEvents) {
                            ev_prio[e] = most_bits;
                            ev_window[e] = window;
                            ev_point[e] = pt | (uint32_t)m << 16;
                            ev_step[e] = 0;
                        }
                    }
                    __syncthreads();
                    accept = !partial && (int64_t)misc[cCount] < need;
                }
                if (!accept && (too_many || all > kEvents)) {
                    // (as many as promote by the stop, by the power law of the priority)
                    if (NT < 512 || partial || 1.5f * (float)need * (float)T > (float)kEvents) return false;
                    partial = true;
                    __syncthreads();
                    const float cut = fast_pow(0.6f * (float)kEvents / (float)all, 1.0f / (float)L);
                    for (int m = tid; m < M; m += NT) {
                        s_rho[m] = rho_all * cut;
                        s_have[m] = s_sum[m] = s_found[m] = 0;
                    }
                    if (tid == 0) misc[cFound] = misc[cCount] = 0;
                    continue;
                }
                if (!accept) {
                    if (next_phase()) return false;
                    // ---- still as many: the promotions in order, as the loop sees them ---------------------
                    // Their steps: the windows of the composite ordered before that one.
                    // (four searches to a lane under way together)
                    constexpr int U = 4;
                    for (int u0 = tid; u0 < all * S; u0 += NT * U) {
                        int lo[U], hi[U], at[U];
                        uint32_t bits[U];
                        bool strict[U];
#pragma unroll
                        for (int u = 0; u < U; u++) {
                            const int x = min(u0 + u * NT, all * S - 1), e = x / S, s = x - e * S;
                            const int m = (int)(ev_point[e] >> 16), i = m * L + (s >> 1), side = s & 1;
                            const uint32_t window = ev_window[e];
                            const int w_h = (int)(window >> 17) & 31, w_side = (int)(window >> 16) & 1, w_j = (int)(window & 0xffffu);
                            bits[u] = ev_prio[e];
                            at[u] = 2 * i + side;
                            lo[u] = 0;
                            hi[u] = s_c[m * S + s];
                            strict[u] = (s >> 1) > w_h;
                            if ((s >> 1) == w_h) {
                                const bool corner = s_p[i] == n - 1 && T >= 2;      // (the ghost window comes first, :264-265)
                                strict[u] = w_side == 0;
                                if (side == w_side) lo[u] = hi[u] = w_j;
                                else if (corner) lo[u] = hi[u] = w_side ? 0 : stream_windows(n, T, s_p[i], side);
                            }
                        }
                        for (;;) {
                            bool any = false;
#pragma unroll
                            for (int u = 0; u < U; u++) {
                                if (lo[u] >= hi[u]) continue;
                                any = true;
                                const int mid = (lo[u] + hi[u]) >> 1, i = at[u] >> 1;
                                Stream st;
                                st.key = a.skeys + (int64_t)i * a.N + off;
                                st.n = n; st.T = T; st.p = s_p[i]; st.side = at[u] & 1; st.q = s_qp[i];
                                const uint32_t v = stream_prio_bits(st, mid);
                                if (strict[u] ? v < bits[u] : v <= bits[u]) lo[u] = mid + 1; else hi[u] = mid;
                            }
                            if (!any) break;
                        }
#pragma unroll
                        for (int u = 0; u < U; u++)
                            if (u0 + u * NT < all * S) atomicAdd(&ev_step[(u0 + u * NT) / S], (uint32_t)lo[u]);
                    }
                    __syncthreads();
                    // Of a point's promotions the earliest counts (ties: the first composite), if it was in its window's first lane.
                    // (every loop below reads the same words on all lanes, eight at a time and without branches)
                    for (int e = tid; e < all; e += NT) {
                        const uint32_t own = ev_step[e], id = ev_point[e];
                        uint32_t sooner = 0;
#pragma unroll 8
                        for (int x = 0; x < all; x++) {
                            const uint32_t other = ev_point[x], s = ev_step[x];
                            sooner |= (uint32_t)(((other ^ id) & 0xffffu) == 0) & ((uint32_t)(s < own) | ((uint32_t)(s == own) & (uint32_t)(other < id)));
                        }
                        ev_prio[e] = sooner == 0 && (ev_window[e] >> 22) ? own : 0xffffffffu;      // the step by which it is counted
                    }
                    if (tid == 0) misc[cArmed] = misc[cMost] = 0xffffffffu;
                    __syncthreads();
                    // The first steps at which k of them, and max_candidates, have been counted.
                    const uint32_t need_k = (uint32_t)a.k_stop, need_c = (uint32_t)min((int64_t)0x7fffffff, max((int64_t)1, a.max_cand));
                    for (int e = tid; e < all; e += NT) {
                        const uint32_t own = ev_prio[e];
                        uint32_t c0 = 0;
#pragma unroll 8
                        for (int x = 0; x < all; x++) c0 += (uint32_t)(ev_prio[x] <= own);
                        if (own != 0xffffffffu && c0 >= need_k) atomicMin(&misc[cArmed], own);
                        if (own != 0xffffffffu && c0 >= need_c) atomicMin(&misc[cMost], own);
                    }
                    __syncthreads();
                    const uint32_t armed = misc[cArmed], by_count = misc[cMost];
                    if (armed != 0xffffffffu) {
                        const uint32_t last_needed = (uint32_t)min((int64_t)0xfffffffe, max((int64_t)0, a.stop_at - 1));
                        t_stop = max(armed, min(last_needed, by_count));
                    }
                    if (partial) {      // (what is promoted by the fewest windows that any composite has consumed is known)
                        uint32_t known = 0xffffffffu;
                        for (int m = 0; m < M; m++) known = min(known, s_have[m]);
                        if (t_stop >= known) return false;
                    }
                    // The near rows among them that are promoted by then.  (All of them are among them, or else come later.)
                    for (int r = tid; r < R; r += NT) {
                        const uint32_t pt = (uint32_t)near[r] - (uint32_t)off;
                        uint32_t in = 0;
#pragma unroll 8
                        for (int x = 0; x < all; x++) in |= (uint32_t)((ev_point[x] & 0xffffu) == pt) & (uint32_t)(ev_step[x] <= t_stop);
                        if (!in) near[r] = ~0ull;
                    }
                    __syncthreads();
                    accept = true;
                }
            }
        }
        break;
    }
    if (!accept) return false;
    if (next_phase()) return false;
    // ---- the nearest kcap near rows, in order ------------
    if (wave == 0) {
        unsigned long long v[1] = {lane < R ? near[lane] : ~0ull};
        wave_sort_u64(v, lane);
        if (lane < a.kcap) part_out[lane] = v[0];
    }
    for (int j = kWave + tid; j < a.kcap; j += NT) part_out[j] = ~0ull;
    return true;
}

template <int NT, bool SCAN>
__global__ __launch_bounds__(NT, 6) void confirm_kernel(ConfirmArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t* misc = reinterpret_cast<uint32_t*>(smem);
    const int X = a.xcds, die = (int)(blockIdx.x % (unsigned)X);
    uint32_t* left_count = a.left_count + die * kTicketStride;
    uint32_t skip = (a.skip ? *a.skip : 0u) | a.rests[0];
    const int32_t* items;
    int64_t count = picked_run(a.from, die, items);
    if (a.pilot == 1) {
        if (skip) return;
        count = min(count, (int64_t)kPilotItems);
    } else if (a.pilot == 2) {      // (the pilot's counts stand: the workgroups decide alike)
        uint32_t had = 0, lost = 0;
        for (int x = 0; x < X; x++) {
            had += a.left_count[x * kTicketStride + a.pilot_at + 1];
            lost += a.left_count[x * kTicketStride + a.pilot_at + 2];
        }
        const bool rests = lost > had;
        if (rests && blockIdx.x == 0 && threadIdx.x == 0) {      // (seen by the rounds after this, and by later calls)
            a.rests[1] = 1;
            a.left_count[a.stats_at + 2] = lost + 17;
        }
        skip |= rests ? 1u : 0u;
    }
    if (skip) {      // everything is traversed at once, or this is no use here: the round's own list stays
        if (blockIdx.x < (unsigned)X && threadIdx.x == 0) *left_count = kAllLeft;
        return;
    }
    // Many that the first pass left can take longer here than a traversal: then they go on as they are, in order.
    if (NT == 512 && count > a.second_cap) {
        if (blockIdx.x < (unsigned)X) {
            for (int64_t e = threadIdx.x; e < count; e += NT) a.left[(int64_t)die * a.left_cap + e] = items[e];
            if (threadIdx.x == 0) { left_count[0] = (uint32_t)count; left_count[2] += (uint32_t)(count / 8); }
        }
        return;
    }
    // Workgroups start in order, so a die's resident ones work on neighbouring queries of one partition; what a launch does not cover they take by
    // strides.  (No tickets: a word that all of a die's items add to takes 20 ns each time, 1 ms of 95000 items.)
    for (int64_t slot = blockIdx.x / (unsigned)X; slot < count; slot += gridDim.x / (unsigned)X) {
        const int32_t item = __builtin_amdgcn_readfirstlane(items[slot]);
        // Some are counted; where nearly all of these had to be left only they are tried.  (One thread reads the counts: others change them meanwhile, and
        // the workgroup has to decide alike.)
        const bool counted = count < 512 || (slot & 7) == 0;
        __syncthreads();
        if (threadIdx.x == 0) misc[cTry] = counted || left_count[2] < 16 + 3 * left_count[1] ? 1u : 0u;
        __syncthreads();
        const bool tried = misc[cTry] != 0;
        const bool done = tried && confirm_item<NT, SCAN>(a, smem, item % a.B, item / a.B);
        if (threadIdx.x == 0) {
            if (!done && a.pilot != 1) a.left[(int64_t)die * a.left_cap + atomicAdd(left_count, 1u)] = item;
            if (counted) atomicAdd(left_count + (done ? 1 : 2), 1u);
        }
    }
}

template <int NT>
int launch_confirm(const QueryArgs& a, ConfirmArgs c, int64_t items, hipStream_t s) {
    c.y = confirm_layout(a, NT);
    const int64_t most = ((int64_t)a.nq * a.B + a.xcds - 1) / a.xcds;
    const int per_cu = std::max(1, std::min((int)(160 * 1024 / c.y.lds_bytes), 24 / (NT / 64)));
    const int64_t grid = std::min(std::max((int64_t)32 * per_cu, items / a.xcds), most) * a.xcds;
    if (confirm_scans(a)) hipLaunchKernelGGL((confirm_kernel<NT, true>), dim3((unsigned)grid), dim3(NT), c.y.lds_bytes, s, c);
    else hipLaunchKernelGGL((confirm_kernel<NT, false>), dim3((unsigned)grid), dim3(NT), c.y.lds_bytes, s, c);
    DCIH_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// Wide windows promote many points by the time a near row comes (25000 unit vectors, windows of 128: 3600), which the scan would list and put in
// order one by one; but where all windows are fewer than the first-lane promotions that a stop takes, there is nothing to scan for.
bool confirm_scans(const QueryArgs& a) { return a.T < 32; }

bool confirm_supported(const QueryArgs& a) {
    const int64_t windows = (int64_t)a.M * a.L * (a.ppb / a.T + 3);
    return (confirm_scans(a) || windows < max((int64_t)a.k_stop, a.max_cand)) && a.inv && a.rpos && a.rpos_ready && a.ppb <= 32766 && a.M <= 8 && a.L >= 2 && a.L <= 32 && a.M * a.L <= 64 && a.T < 32768 &&
           (int64_t)a.L * a.N < 0x7fffffffLL && a.xcds >= 1 && a.xcds <= 32 && confirm_layout(a, 512).lds_bytes <= 40 * 1024;
}


int confirm_items(const QueryArgs& a, const uint32_t* skip, uint32_t* rests, int32_t* left, uint32_t* left_count, int64_t left_cap, hipStream_t s) {
    ConfirmArgs c;
    c.skeys = a.skeys; c.sids = a.sids; c.inv = a.inv; c.rpos = a.rpos;
    c.data = a.data; c.query = a.query; c.qproj = a.qproj;
    c.N = a.N; c.ppb = a.ppb; c.stop_at = a.stop_at; c.max_cand = a.max_cand;
    c.dim = a.dim; c.M = a.M; c.L = a.L; c.B = a.B; c.T = a.T; c.nq = a.nq; c.k_stop = a.k_stop; c.kcap = a.kcap; c.xcds = a.xcds;
    c.T_magic = a.T_magic; c.part = a.part; c.skip = skip;
    c.near_bounds = a.near_bounds; c.near_limit = a.near_limit; c.near_stride = a.near_stride; c.near_shift = a.near_shift; c.near_tiles = a.near_tiles;
    c.left_cap = left_cap;
    c.rests = rests;
    c.from.picked = a.picked; c.from.picked_count = a.picked_count; c.from.xcds = a.xcds; c.from.left = nullptr; c.from.left_count = nullptr; c.from.left_cap = 0;
    // Calls of few items wait for their slowest: four wavefronts to an item.  Items that fill the device several times over are one wavefront's, which takes
    // fewer instructions (10000 items: 192 us, 261 by four), and what its tables do not hold eight wavefronts' (1400 of 113000: 422 us, 638 by four).
    const double expect = (double)a.nq * a.pick_first;
    const bool many = expect > (double)(a.xcds * 32 * 16);
    // (an item takes 0.24 us there where its promotions fill the tables: 17000 of 53000 items of 1272 points, windows of 10, 7 indices, 4.0 ms, 1.6 by the dense kernel;
    // 18000 of 36000 of 2818, 12 indices, with the second pass 5.9 ms in all, 7.1 without)
    c.second_cap = a.mode != 2 && takes_dense_kernel(a) && traversal_costs(a, 0.0).dense_item < 0.08 ? 256 : left_cap;
    // Nothing on record: a few items go ahead, and where most of those have to be left (their rows are promoted late, or not at all) no others are tried.
    c.pilot = 0;
    if (a.confirm_had + a.confirm_lost == 0 && confirm_scans(a) && a.picked_expect > 0 && expect > (double)(a.xcds * kPilotItems * 2)) {
        c.pilot = 1;
        c.left = nullptr;
        c.left_count = left_count + kConfirmPilot;
        const int rc = launch_confirm<256>(a, c, (int64_t)a.xcds * kPilotItems, s);
        if (rc) return rc;
        c.pilot = 2;
    }
    if (many) {
        c.left = left + a.xcds * left_cap;
        c.left_count = left_count + kConfirmPass;
        c.pilot_at = kConfirmPilot - kConfirmPass;
        c.stats_at = -kConfirmPass;
        const int rc = launch_confirm<kWave>(a, c, a.picked_expect, s);
        if (rc) return rc;
        c.from.left = c.left; c.from.left_count = c.left_count; c.from.left_cap = left_cap;
    }
    c.left = left;
    c.left_count = left_count;
    c.pilot_at = kConfirmPilot;
    c.stats_at = 0;
    return many ? launch_confirm<512>(a, c, 0, s) : launch_confirm<256>(a, c, a.picked_expect, s);
}

}  // namespace dcih
