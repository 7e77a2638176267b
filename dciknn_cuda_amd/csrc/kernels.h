// Internal launch interface between the kernel translation units and api.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace dcih {

// out[r][c] = sum_k rows[c][k] * dirs[r][k]; row r of out starts at d_out + r * out_stride
// (out_stride >= num_rows).
int project(const float* d_dirs, int num_dirs, const float* d_rows, int64_t num_rows,
            int dim, float* d_out, int64_t out_stride, hipStream_t s);

// Sorts every (simple index, partition) slice of the keys by (key, id); the keys of
// index i start at d_keys + i * key_stride (key_stride >= n), the outputs are
// [num_indices][n].  d_tmp is scratch of segsort_tmp_bytes() bytes (may be null when
// that is 0).
size_t segsort_tmp_bytes(int num_indices, int64_t n, int block_size);
// d_inv: null, or [num_indices][n] receiving each point's position inside its
// sorted slice (the inverse of d_sids) as a 16-bit value (only meaningful when a partition
// holds at most 65536 points).  d_lids: null, or [num_indices][n] receiving the ids relative
// to their partition's first point as 16-bit values (no kernel reads them any more; the
// index does not keep them).  values: the keys are distances, many of which may be equal or infinite, and not projections: always sorted by digits.
int segsort(const float* d_keys, int64_t key_stride, int num_indices, int64_t n, int block_size,
            float* d_skeys, int32_t* d_sids, uint16_t* d_inv, uint16_t* d_lids, void* d_tmp,
            hipStream_t s, bool float_ids = false, bool values = false);

// The same for slices of ppb <= 25600 points by one distribution into buckets (bucketsort.hip); a slice that it does not suit is left alone
// but for an id of -1 in its first place.
bool bucketsort_supported(int64_t ppb);
int bucketsort(const float* d_keys, int64_t key_stride, int num_indices, int64_t n, int64_t ppb, int B, float* d_skeys, int32_t* d_sids,
               uint16_t* d_inv, hipStream_t s);

// Appending: the index over n1 points from the sorted arrays of the index over their first
// n0 points (same block_size) and the unsorted keys of the others (index i's key of point id
// at d_keys + i * key_stride + id): old slices are split into runs of the new ones, the new
// points sorted, the runs merged; nothing of the old part is sorted again.  Outputs as
// segsort's; d_tmp = segsort_append_tmp_bytes() bytes.
bool segsort_append_supported(int64_t n0, int64_t n1, int block_size);
size_t segsort_append_tmp_bytes(int num_indices, int64_t n1);
int segsort_append(const float* d_old_skeys, const int32_t* d_old_sids, int64_t n0,
                   const float* d_keys, int64_t key_stride, int num_indices, int64_t n1, int block_size,
                   float* d_skeys, int32_t* d_sids, uint16_t* d_inv, uint16_t* d_lids, void* d_tmp,
                   hipStream_t s);

// rpos (above inv's layout, [I][n] 16-bit values): rpos[i][e] = inv[i][sids[first(i)][e]], first(i) = the first simple
// index of i's composite; the rows of the first simple indices themselves are left alone (the identity).
int fill_positions_by_first(const int32_t* d_sids, const uint16_t* d_inv, uint16_t* d_rpos, int64_t n, int M, int L, int64_t ppb, int B,
                            hipStream_t s);

// point_rows from inv (see QueryArgs), and whether the dense kernel's calls in rounds are better off with them.
size_t point_rows_bytes(int64_t n, int M, int L);
int fill_point_rows(const uint16_t* d_inv, uint16_t* d_rows, int64_t n, int M, int L, hipStream_t s);
bool point_rows_fit(int64_t ppb, int M, int L, int T);

struct QueryArgs {
    const float* skeys;      // [I][N] sorted projections
    const int32_t* sids;     // [I][N] point ids in the same order
    const uint16_t* inv;     // [I][N] position of every point inside its sorted slice (null if ppb > 65536)
    const uint16_t* rpos;    // [I][N] the same positions in the order of the composite's FIRST simple index: entry s of a
                             // slice is the position, in this simple index, of the point that stands at place s of the
                             // first one's slice (null if ppb > 65536; filled on the first use, see fill_positions_by_first)
    int* rpos_ready;         // host flag of the index: rpos has been filled
    const uint16_t* point_rows;   // null, or [N][M][L up to a multiple of 8] inv's positions, a point's side by side (the last one of a composite repeated)
    int recorded;            // 1: the call is recorded into a graph, its kernels do not run now
    const float* data;       // [N][dim]
    const float* query;      // [nq][dim]
    const float* qproj;      // [I][nq]
    int64_t N;
    int64_t ppb;             // points per partition = ceil(N / B)
    int dim, M, L, B, T, nq;
    int k;                   // results per query
    int k_stop;              // promotions by a window's first lane that arm the stop rule (num_neighbours)
    int blind;               // 1: a candidate is scored by the step that promoted it, no distance is computed
    unsigned T_magic;        // ceil(2^32 / T) for T > 1: d / T == mulhi(d, T_magic) for 0 <= d < 65536
    int kcap;                // min(k, ppb): results kept per (query, partition)
    int64_t stop_at;         // num_outer_iterations * L
    int64_t max_cand;
    unsigned long long* part;      // [nq][B][kcap] packed (dist bits << 32 | id); blind: (step << 32 | id)
    unsigned long long* counters;  // null or [nq][4]
    uint32_t* gscratch;      // global visit counters when they do not fit LDS
    int32_t* redo_items;     // [nq*B] (query, partition) pairs the batch kernel hands back
    uint32_t* redo_count;    // their number
    const int32_t* item_list;    // step-by-step kernel: null = all nq*B items, else this list
    const uint32_t* item_count;  // ... of this length
    float* stop_hint;        // null, or [3][B] per partition: running averages of the stop step and of the promotions at the stop, stops seen
    int hints_cold;          // the table was cleared for this call: nothing is known yet about where traversals stop
    unsigned long long* phase_ticks;  // null, or 16 accumulators for the batch kernel's phases
    int mode;                // 0 = pick, 1 = step-by-step kernel, 2 = batch kernel, 3 = dense kernel
    // hand-over from the batch kernel to the dense kernel: one list of items per die
    int32_t* dense_items;    // null, or [xcds][dense_cap]
    uint32_t* dense_count;   // [xcds]
    int64_t dense_cap;
    int dense_by_cost;       // 1: the estimates below decide, too, and say when an item is handed over
    int hand_over_at;        // promotions from which the batch kernel hands an item over
    int dense_min_promos;    // promotions per (query, partition) from which the dense kernel is the cheaper one
    // second pass of the batch kernel: items that outgrow its compact per-item tables are listed and
    // taken up again by the variant with the full tables
    int32_t* wide_items;     // null, or [wide_cap]
    uint32_t* wide_count;
    int64_t wide_cap;
    const int32_t* block_list;        // null = the launch covers queries q_first .. q_first + q_count; else workgroup w takes block_list[w]
    const uint32_t* block_list_count; // ... for w below this number
    float expect_steps, expect_promotions;      // the batch kernel's first guess at where a full partition's traversal stops
    int few_items;           // 1: the batch kernel gives every item four wavefronts or more; 2: and larger tables
    int full_tables;         // 1: the batch kernel keeps its per-point flags as bits whatever the shape
    // dense kernel: the rows' and the queries' 8-bit codes (rows8.hip; null = read whole rows)
    const unsigned char* rows8;      // [N][rows8_rec]
    int rows8_rec;                   // bytes per record
    uint32_t* rows8_bounds;          // [B][2]: largest coding error and largest squared norm of a partition's rows (float
                                     // bits), then [B]: how many items the codes did not do for lately (traverse_dense.hip)
    const unsigned char* query8;     // [nq][rows8_query_bytes(dim)]
    int xcds;                // accelerator dies of the device (each has an L2 of its own)
    int q_first, q_count;    // batch kernel: the queries one launch covers
    int32_t* out_ids;        // [nq][k]
    int float_ids;           // 1: ids are stored as float32 values in the same place
    float* out_dists;        // [nq][k]; blind: null, or the promoting steps as floats
    // a call in rounds (bounds.hip)
    const int32_t* picked;   // null = all nq * B items, else the round's, of which every die takes one run
    const uint32_t* picked_count;
    const int32_t* left;     // null, or per die of these those that confirm.hip has left, and how many (kAllLeft: all of them, not listed)
    const uint32_t* left_count;
    int64_t left_cap;
    uint32_t* round_items;   // null, or device words for the number of items of every round, then the sample's decision
    uint32_t* blind_word;    // null, or (the host's memory) set where bounds say nothing of queries' nearest rows
    unsigned long long* confirm_word;   // null, or (the host's memory) confirm_tag << 48 | items that confirm.hip left << 24 | answered, of those it counts
    uint32_t confirm_tag;
    int64_t* selected;       // (host) counts the queries that nearest.hip answers
    int64_t* window_launches;   // (host) counts the launches of the dense kernel that look up first lanes of windows
    uint32_t* picked_ticket; // a zeroed word per die: the dense kernel's workgroups take their items by it
    int64_t picked_exact;    // their number, where it is known: 0 otherwise
    int64_t picked_expect;   // about how many there are, 0: few
    int64_t picked_cover;    // how many there seldom are more of: what a launch of the batch kernel covers by a workgroup each
    const uint32_t* only;    // merge: null, or only the queries whose word here is only_round
    uint32_t only_round;
    // dense kernel, in rounds: lower bounds per tile of 2^near_shift rows ([B * near_tiles][nq]) and the distance of each query from
    // which on a candidate does not matter to the round; null = all candidates' distances are wanted
    const uint32_t* near_bounds;
    const float* near_limit;
    int64_t near_stride;
    int near_shift, near_tiles;
    int pick_near;           // 1: a call in rounds goes to the dense kernel and keeps those bounds
    int pick_confirm;        // 1: rounds' items go through confirm.hip first, which needs those bounds too
    int may_confirm;         // 1: a later call like this one may
    size_t near_room;        // what the tiles' bounds of a call may take
    int pick_parts;          // above 1: what plan_rounds would do with the call if it came in so many parts
    int pick_sample;         // 0, or: so many queries are traversed whole first, and decide
    float pick_most;         // share of pairs that rounds may have to take: where the sample's bounds leave more, everything is taken at once
    int pick_rounds;         // 0: everything is traversed at once
    int pick_rank;           // the first round takes the partitions of so many nearest rows
    uint32_t confirm_had, confirm_lost;   // of the items that confirm.hip counted in the last call of this shape that it was part of, those that it answered and left
    int index_calls;         // queries of this index before
    int pick_rule;           // DCIH_OPT_ROUNDS value
    double pick_first;       // partitions per query the first round is expected to take
    double share;            // share of all items that are expected to be traversed (1 but for such calls)
    float pick_flat;         // a query whose furthest bound is within this factor of round 1's limit takes every partition at once
    float* dense;            // null, or [nq][N]: the step-by-step kernel stores every candidate's score here instead of keeping a top-k
};
// About how many promotions a partition's traversal takes before it stops: k_stop of them by a window's
// first lane, which takes about k_stop * T in all.  The step limit can ask for more: a traversal
// that must consume the fraction f of a composite's windows before it may stop has by then promoted about
// f^L of the partition (a point needs all L of its windows; nearby windows come first, so this is on
// the low side), unless max_cand first-lane promotions end it earlier.
inline double expected_promotions(const QueryArgs& a) {
    const double windows = (double)a.L * ((double)a.ppb / (double)a.T);
    const double f = fmin(1.0, (double)a.stop_at / fmax(1.0, windows));
    const double by_steps = fmin((double)a.ppb * pow(f, (double)a.L), (double)a.max_cand * (double)a.T);
    return fmax((double)a.k_stop * (double)a.T, by_steps);
}
// About the step at which a partition's traversal stops, by the same reasoning (0.55 to 1.0 of this in
// Gaussian rows, unit vectors, manifolds and mixtures of 0.4 to 1 million rows, mostly above 0.9).
inline double expected_stop(const QueryArgs& a) {
    const double windows = (double)a.L * ((double)a.ppb / (double)a.T);
    auto fraction = [&](double promotions) { return fmin(1.0, pow(promotions * (double)a.T / (double)a.ppb, 1.0 / (double)a.L)); };
    const double by_steps = fmin((double)a.stop_at / fmax(1.0, windows), fraction((double)a.max_cand));
    return windows * fmin(1.0, fmax(fraction((double)a.k_stop), by_steps));
}
// What the two kernels take, in us on an MI355X: a time one item takes from end to end, and a time per item
// once they fill the device.  The dense kernel's grow with the windows it ranks and the points it looks up,
// the batch kernel's with the promotions it replays.  Fitted to Gaussian rows (24 to 4000 points per partition,
// T 2 to 64, L 7 and 15); today's kernels are faster than this by about a tenth (dense) and a quarter (batch),
// which leaves the choice where it was: over 692 shapes of 24 to 20000 points, T 1 to 64, L 3 to 15, M 1 to 3
// (profiles/kernel_choice.txt) a call left to choose takes 1.3 % longer than the best of batch, dense and the
// two together in the geometric mean, and more than a tenth longer in 27, mostly at M = 1; factors of their
// own for each M would make that 0.9 % and 19.
struct TraversalCosts { double dense_item, batch_item, batch_per_promotion, dense, batch; };
inline TraversalCosts traversal_costs(const QueryArgs& a, double promotions) {
    TraversalCosts c;
    const double ppb = (double)a.ppb, windows = (double)a.L * (ppb / (double)a.T + 3.0);
    const double size = (double)a.M / 2.0, length = (double)a.L / 7.0, items = (double)a.nq * (double)a.B * a.share;
    c.dense_item = (0.0086 + 1.8e-5 * windows + 1.1e-6 * (double)a.L * ppb) * size;
    c.batch_per_promotion = 1.37e-3 * length * size;
    c.batch_item = 0.0063 * length * size + c.batch_per_promotion * promotions;
    c.dense = 45.0 + (0.0115 * windows + 0.005 * ppb) * size + items * c.dense_item;
    c.batch = 153.0 + 7.0 * promotions * length * sqrt(length) * size + items * c.batch_item;
    return c;
}
// The query scratch keeps its list lengths in 64 consecutive words that one kernel clears: the
// step-by-step kernel's redo list, one hand-over list per die (up to 32), and in the last word
// the batch kernel's second-pass list.
constexpr int kListCountWords = 64;

// Work order of the batch kernel.  Workgroups go to the XCDs round-robin by their
// number and every XCD has an L2 of its own, so XCD x is given the partitions x,
// x + X, ... and works through them one after the other, all queries of a
// partition before the next: the workgroups an XCD runs at any moment share one
// partition's slices.  The B mod X partitions that do not fill a round are spread
// over all X dies as equal runs of the (partition, query) list, so no die idles.
// block_items = workgroups one launch over nq queries needs; block_item maps a
// workgroup to its partition b and query q (false: nothing to do).
__host__ __device__ inline int64_t block_items(int X, int B, int nq) {
    const int full = B / X, rest = B - full * X;
    return (int64_t)X * ((int64_t)full * nq + ((int64_t)rest * nq + X - 1) / X);
}
__host__ __device__ inline bool block_item(int64_t block, int X, int B, int nq, int& b, int& q) {
    const int xcd = (int)(block % X);
    const int64_t seq = block / X;
    const int full = B / X, rest = B - full * X;
    const int64_t full_items = (int64_t)full * nq;
    if (seq < full_items) {
        b = xcd + X * (int)(seq / nq);
        q = (int)(seq % nq);
        return true;
    }
    const int64_t run = ((int64_t)rest * nq + X - 1) / X;
    const int64_t e = (seq - full_items) + (int64_t)xcd * run;
    if (seq - full_items >= run || e >= (int64_t)rest * nq) return false;
    b = X * full + (int)(e / nq);
    q = (int)(e % nq);
    return true;
}
// Queries one launch of the batch kernel may cover: a launch is limited to 2^32 - 1
// threads in all (256 per workgroup).
__host__ __device__ inline int block_queries_per_launch(int X, int B, int nq) {
    const int64_t max_items = 0xffffffffLL / 256;
    const int64_t per_query = (int64_t)B + X;          // upper bound of block_items / nq
    const int64_t fit = max_items / per_query;
    return (int)(fit < 1 ? 0 : (fit < nq ? fit : nq));
}
// Workgroups of the step-by-step kernel: it strides over its items, and a launch is
// limited to 2^32 - 1 threads in all (64 per workgroup).
__host__ __device__ inline int64_t step_grid_cap() { return (int64_t)1 << 20; }

size_t query_part_bytes(const QueryArgs& a);
// Clears n 64-bit words with a kernel (a memset node is not safe in a captured graph).
int zero_words64(void* d_p, int64_t n, hipStream_t s);
// Bytes of global counter scratch the traversal needs (0 when LDS suffices).
size_t query_gscratch_bytes(const QueryArgs& a);
// Batch traversal (traverse_block.hip): whether the shape fits its fixed LDS
// tables, and the launch itself.
bool block_traversal_supported(const QueryArgs& a, size_t* lds_bytes);
bool block_takes_lists(const QueryArgs& a);
int query_block(const QueryArgs& a, hipStream_t s);
// Dense traversal (traverse_dense.hip): every point's promoting step at once.  Works
// through the lists the batch kernel filled (a.dense_items) or, with a.mode == 3,
// through all items.
bool dense_traversal_supported(const QueryArgs& a, size_t* lds_bytes);
bool point_rows_pay(const QueryArgs& a);
int query_dense_items(const QueryArgs& a, hipStream_t s);

// 8-bit codes of rows and queries (rows8.hip); bounds: 3 * B words.
bool rows8_supported(int dim);
int rows8_record_bytes(int dim);
int rows8_query_bytes(int dim);
int code_rows(const float* d_data, int64_t n, int dim, int64_t ppb, int B, unsigned char* d_recs, uint32_t* d_bounds,
              hipStream_t s);
int code_queries(const float* d_query, int nq, int dim, unsigned char* d_recs, hipStream_t s);

// The run of a list of `count` items that die x of X takes: its first item and their number.
__device__ inline int64_t run_of_die(int64_t count, int x, int X, int64_t& first) {
    const int64_t each = (count + X - 1) / X;
    first = each * x;
    return min(each, max((int64_t)0, count - first));
}
// Calls in rounds (bounds.hip): lower bounds of every (query, partition)'s nearest distance, and the items each
// round takes.  Scratch of bounds_bytes(); bounds_cost: about how long the bounds take, us.  pack_bounds
// comes first and also clears a.part.
constexpr int kPickCountWords = 64 + 2 * 32 * 32, kMostRounds = 4;
// of the count words: the sample's items, whether rounds are skipped, the pairs that says so by, whether confirm.hip rests, and did so in round 1; per die a ticket, and the items that confirm.hip left, then of some those that it answered and left
constexpr int kSampleWord = 8, kSkipWord = 9, kRestsWord = 12, kRestedWord = 13, kTicketWord = 64, kTicketStride = 32, kLeftWord = kTicketWord + 32 * 32, kConfirmPass = 8, kConfirmPilot = 16;      // (where the counts of confirm.hip's first pass, and of its pilot, lie in a die's words)
constexpr int kPilotItems = 64;      // tried ahead, per die, where nothing is known yet
// A round's items of die x: its run of the round's list, or what confirm.hip has left of that.
constexpr uint32_t kAllLeft = 0xffffffffu;
template <class A>
__device__ inline int64_t picked_run(const A& a, int x, const int32_t*& items) {
    const uint32_t left = a.left ? a.left_count[x * kTicketStride] : kAllLeft;
    if (left != kAllLeft) {
        items = a.left + x * a.left_cap;
        return (int64_t)left;
    }
    int64_t first;
    const int64_t count = run_of_die(*a.picked_count, x, a.xcds, first);
    items = a.picked + first;
    return count;
}
constexpr uint32_t kSampleRound = 0x10000;         // of the sample's queries while their results are merged
struct Picked {
    const int32_t* items; const uint32_t* count; const uint32_t* last_round; uint32_t* ticket;
    const uint32_t* near_bounds; const float* near_limit; const float* confirm_limit; int64_t near_stride; int near_shift, near_tiles;
};
bool bounds_supported(const QueryArgs& a);
size_t bounds_bytes(const QueryArgs& a);
size_t near_bytes(const QueryArgs& a);      // the part of it that pick_near adds
double bounds_cost(const QueryArgs& a);
int pack_bounds(const QueryArgs& a, void* ws, hipStream_t s);
int partition_bounds(const QueryArgs& a, void* ws, hipStream_t s);
// Where a.pick_sample is set, after pack_bounds: all items of that many queries, and, once they are traversed and merged, whether the
// bounds are formed at all (else everything comes in round 1).
int sample_items(const QueryArgs& a, void* ws, Picked& p, hipStream_t s);
int sample_decide(const QueryArgs& a, void* ws, hipStream_t s);
int pick_items(const QueryArgs& a, void* ws, int round, int rounds, hipStream_t s);
// Answers those of a round's items that need no traversal (confirm.hip); a.left.. become the others.
bool confirm_supported(const QueryArgs& a);
bool confirm_scans(const QueryArgs& a);      // whether that needs rpos
int confirm_items(const QueryArgs& a, const uint32_t* skip, uint32_t* rests, int32_t* left, uint32_t* left_count, int64_t left_cap, hipStream_t s);
int confirm_round(QueryArgs& a, void* ws, hipStream_t s);
Picked picked_items(const QueryArgs& a, void* ws, int round);
// Whether a call is worth its rounds; sets a.pick_rounds, a.pick_first and a.share.
bool plan_rounds(QueryArgs& a);

// Full ranking (exhaustive.hip) for num_neighbours above the points per partition,
// where the traversal provably visits everything: queries are processed `chunk` at
// a time in `ws` (exhaustive_ws_bytes(N, chunk, k) bytes); a.qproj is needed only when
// a.counters is set.
int exhaustive_chunk(int64_t N, int nq);
size_t exhaustive_ws_bytes(int64_t N, int chunk, int k);
int query_exhaustive(const QueryArgs& a, void* ws, int chunk, hipStream_t s);
// The same for few results (nearest.hip): distances only of the rows whose lower bound says that they can be among them.
// d_bounds: [nq][N] floats; d_least: nearest_least_bytes.
bool nearest_supported(int64_t N, int dim, int k);
bool nearest_pays(int64_t N, int dim, int k, int nq);
size_t nearest_least_bytes(int64_t N, int nq);
// Queries whose bounds rule out too little are left in large tables (`leaves`): d_left receives their number, then their numbers, then as many
// words as queries that are zero.
size_t nearest_left_bytes(int nq);
int query_nearest(const QueryArgs& a, int q0, int nq, float* d_bounds, float* d_least, uint32_t* d_left, hipStream_t s, bool& leaves);
// The pieces of it that the dense-row traversal (query_dense) shares: rows of N values
// at rank_rows_input(ws), `rows` <= chunk of them; rank_rows sorts every row by (value,
// column) and writes the first k columns (id = column, or -1 for +inf when asked).
float* rank_rows_input(void* ws);
int fill_rows(float* d_rows, int64_t cells, float value, hipStream_t s);
int rank_rows(void* ws, int chunk, int rows, int64_t N, int k, bool inf_is_empty, bool float_ids,
              int32_t* out_ids, float* out_vals, hipStream_t s);
// k best of the B ascending lists of kcap packed words per query at a.part, to a.out_ids / a.out_dists.
int merge_lists(const QueryArgs& a, hipStream_t s);
// More results per query than the top-k tables hold, early stops possible: the
// step-by-step kernel writes every candidate's score into a dense row of its query
// (+inf = not a candidate), rank_rows does the rest.  Projects the queries itself
// (d_dirs), chunk by chunk; ws = I*chunk floats + exhaustive_ws_bytes(N, chunk, N) bytes.
int query_dense(const QueryArgs& a, const float* d_dirs, void* ws, int chunk, hipStream_t s);

// Whether a call goes to the dense kernel as a whole (given that the shape fits it).
bool takes_dense_kernel(const QueryArgs& a);

// bounds_ws: bounds_bytes(a) of scratch where a.pick_rounds is set.
// ev: null, or five events recorded before the traversal, after the batch kernel (if it
// ran: ran[0]), after the dense kernel (if it ran: ran[1]), between traversal and merge,
// and after the merge.
int query(const QueryArgs& a, void* bounds_ws, hipStream_t s, hipEvent_t* ev, bool* ran);

}  // namespace dcih
