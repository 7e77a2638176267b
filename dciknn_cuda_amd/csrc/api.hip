// Host side of libdci_hip.so: the C-ABI declared in include/dci_hip.h (and the
// inspection entry points of include/dci_hip_debug.h).
//
// Mirrors the host functions of the reference (dci_init, dci_add, dci_query,
// dci_clear, dci_reset, dci_free: src/dci_cuda_kernel.cu:77-187, :777-899) but
// returns status codes instead of asserting, takes a stream, frees what it
// allocates, and launches a constant number of kernels per call instead of
// several per query.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "../../include/dci_hip.h"
#include "../../include/dci_hip_debug.h"
#include "common.h"
#include "kernels.h"

namespace dcih {

static thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}

namespace {

// splitmix64 -> xoshiro256** -> Box-Muller in double: the same seed gives the
// same directions on every machine.
struct Rng {
    uint64_t s[4];
    bool have_spare = false;
    double spare = 0.0;
    explicit Rng(uint64_t seed) {
        uint64_t x = seed;
        for (int i = 0; i < 4; i++) {
            x += 0x9e3779b97f4a7c15ull;
            uint64_t z = x;
            z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
            z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
            s[i] = z ^ (z >> 31);
        }
    }
    static uint64_t rotl(uint64_t v, int k) { return (v << k) | (v >> (64 - k)); }
    uint64_t next() {
        const uint64_t r = rotl(s[1] * 5, 7) * 9;
        const uint64_t t = s[1] << 17;
        s[2] ^= s[0]; s[3] ^= s[1]; s[1] ^= s[2]; s[0] ^= s[3];
        s[2] ^= t; s[3] = rotl(s[3], 45);
        return r;
    }
    double uniform() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }  // (0,1)
    double normal() {
        if (have_spare) { have_spare = false; return spare; }
        const double u = uniform(), v = uniform();
        const double r = std::sqrt(-2.0 * std::log(u));
        const double th = 6.283185307179586476925 * v;
        spare = r * std::sin(th);
        have_spare = true;
        return r * std::cos(th);
    }
};

struct DeviceGuard {
    int prev = -1;
    bool ok;
    explicit DeviceGuard(int dev) {
        ok = hipGetDevice(&prev) == hipSuccess && hipSetDevice(dev) == hipSuccess;
    }
    ~DeviceGuard() { if (prev >= 0) (void)hipSetDevice(prev); }
};

}  // namespace
}  // namespace dcih

using namespace dcih;

// Scratch of dcih_query_noalloc: part of the code object, so every device the library
// runs on holds its own copy from the moment the library is loaded there until the
// process ends.  Host code never uses this name as an address (on the host it is only a
// stand-in for the symbol): dcih_create asks the runtime where the array lives on its
// device and keeps that pointer.  (The host code's use of the name below is what gives the
// device symbol external linkage, which the runtime's lookup by name needs: a `used`
// attribute would keep it local to the code object and the lookup would abort.)
constexpr size_t kScratchBytes = DCIH_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
constexpr int kMaxXcds = 32;      // dies per device the query scratch has list lengths for (256 bytes: 1 + 32 words used)
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on `device`, which must be the current device.
int resolve_scratch(int device) {
    if (device < 0 || device >= kMaxDevices) return fail(DCIH_EINVAL, "device number out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return 0;
    void* ptr = nullptr;
    DCIH_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return fail(DCIH_EHIP, "hipGetSymbolAddress returned no address for the scratch array");
    g_scratch_ptr[device] = ptr;
    return 0;
}

void* scratch_of(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return device >= 0 && device < kMaxDevices ? g_scratch_ptr[device] : nullptr;
}
}  // namespace

// What confirm.hip has made of queries of one shape, for the plans of the next ones of that shape (other numbers of results, stops and windows leave
// other items).  Forgotten when the index is formed anew, or for a fifth shape.
constexpr int kNearRecords = 4;
struct NearRecord {
    int k = 0, outer = 0, T = 0, maxc = 0;   // the shape (zeros: none)
    uint32_t tag = 0;                   // what its words have to bear: calls still under way may write those of an earlier record
    int rests = 0;                      // calls in rounds that went without confirm.hip, since the last one with it
    uint64_t last = 0;                  // the last call
};
// Words that the device writes and the host reads when it plans a call: they steer work, never results.
struct HostWords {
    uint32_t blind;                     // set by queries in rounds whose bounds said nothing: the next ones use the rows' codes
    uint32_t pad;
    uint64_t near[kNearRecords];        // tag << 48 | items left << 24 | items answered, of those that confirm.hip counts
};

struct dcih_index {
    int dim = 0, M = 0, L = 0, device = 0;
    int xcds = 8;                       // accelerator dies of the device
    uint64_t seed = 0;
    uint64_t draws = 0;                 // direction sets drawn so far
    std::vector<float> h_dirs;          // [I][dim]
    float* d_dirs = nullptr;
    const float* d_data = nullptr;      // borrowed
    int64_t n = 0;
    int block_size = 0;
    float* d_skeys = nullptr;           // [I][n]
    int32_t* d_sids = nullptr;          // [I][n]
    uint16_t* d_inv = nullptr;          // [I][n] position of each point in its sorted slice (partitions <= 65536 points)
    uint16_t* d_rpos = nullptr;         // [I][n] the same, in the order of each composite's first simple index (room kept by the
                                        // build, filled by the first query that runs the batch traversal kernel)
    int rpos_ready = 0;
    // every point's positions side by side (where windows are wide): room taken and filled by a call in rounds, once such calls
    // have asked for more than that costs
    uint16_t* d_point_rows = nullptr;
    size_t point_rows_room = 0;
    int point_rows_ready = 0;
    bool point_rows_no_room = false;    // there was no memory for them: not asked for again until the next build
    double point_rows_demand = 0.0;     // points looked at by such calls so far, in indexes' worth
    // 8-bit codes of the rows and the partitions' bounds behind them (rows8.hip): room taken and codes formed
    // once the dense kernel's calls have asked for more candidate rows than forming them costs
    unsigned char* d_rows8 = nullptr;
    size_t rows8_bytes = 0;
    double rows8_demand = 0.0;          // candidate rows asked for so far
    bool rows8_ready = false;           // formed, or under way on some stream:
    hipEvent_t rows8_event = nullptr;   // ... until this is over,
    bool rows8_settled = false;         // ... as has been seen
    bool rows8_no_room = false;         // there was no memory for them: not asked for again until the next build
    float* d_own = nullptr;             // rows copied in by dcih_append (the index owns these)
    float* d_ukeys = nullptr;           // [I][own_rows] unsorted projections of the rows in d_own
    int64_t own_rows = 0;               // capacity of d_own / d_ukeys in rows
    int64_t ukeys_rows = 0;             // leading rows of d_own whose projections d_ukeys holds
    // the end of the last call that reads rows the index owns, on its stream, and through it of all before it:
    // what comes after dcih_clear, on whatever stream, is put behind it
    hipEvent_t busy = nullptr;
    bool busy_set = false;
    bool recorded = false;              // such a call was recorded into a graph: when it runs is not known
    float* d_stop_hint = nullptr;       // [3][block_size] epoch-size hints learnt from earlier queries
    int hint_k = 0, hint_outer = 0, hint_T = 0, hint_maxc = 0;   // query shape the hints belong to (zeros: none, as after a build)
    int traversal = 0;                  // DCIH_OPT_TRAVERSAL value
    int dense_min_promos = 160;         // DCIH_OPT_DENSE_MIN_PROMOTIONS value
    int dense_by_cost = 1;              // until that option is set
    int append_mode = 0;                // DCIH_OPT_APPEND value
    int rounds = 0;                     // DCIH_OPT_ROUNDS value
    int64_t route[4] = {0, 0, 0, 0};    // dcih_debug_route
    int64_t plan[3] = {0, 0, 0};        // the first of dcih_debug_plan's values
    NearRecord near_records[kNearRecords];
    int near_last = -1;                 // the one of the last call that confirm.hip was part of
    uint32_t near_tag = 0;              // of the last record that was begun
    uint64_t near_calls = 0;            // calls that had a record
    int index_calls = 0;                // queries since the index was formed
    size_t near_room = (size_t)1 << 30; // what the bounds of a call's tiles may take
    volatile HostWords* words = nullptr;   // (pinned, from the first query in rounds that writes them)
    uint32_t* d_round_items = nullptr;  // dcih_debug_round_items
    unsigned long long* d_phase_ticks = nullptr;   // optional profile of the batch kernel
    // grow-only workspace: query scratch, and the unsorted keys during a build
    void* ws = nullptr;
    size_t ws_bytes = 0;
    // grow-only arenas the sorted arrays and the hint table are carved from; kept
    // across dcih_clear so that a rebuild allocates nothing.  The index lives in
    // arena[cur]; dcih_append builds the next one in the other and then switches, so
    // a failed append leaves the index as it was.
    void* arena[2] = {nullptr, nullptr};
    size_t arena_bytes[2] = {0, 0};
    int cur = 0;
    // optional per-kernel timing: ev[2*t], ev[2*t+1] bracket timer t
    bool profiling = false;
    hipEvent_t ev[2 * DCIH_NUM_TIMERS] = {};
    bool ev_valid[DCIH_NUM_TIMERS] = {};
};

namespace {

int num_indices(const dcih_index* h) { return h->M * h->L; }

// Draws direction set number h->draws from the handle's seed and uploads it.
int draw_directions(dcih_index* h) {
    const int I = num_indices(h);
    Rng rng(h->seed + 0x632be59bd9b4e019ull * h->draws);
    h->draws++;
    h->h_dirs.resize((size_t)I * h->dim);
    for (auto& v : h->h_dirs) v = (float)rng.normal();
    // unit rows: sequential fp32 sum of squares, sqrtf, divide
    // (normalize_proj_vecs, src/dci_cuda_kernel.cu:52-73)
    for (int r = 0; r < I; r++) {
        float* row = h->h_dirs.data() + (size_t)r * h->dim;
        float sq = 0.0f;
        for (int k = 0; k < h->dim; k++) sq += row[k] * row[k];
        const float norm = sqrtf(sq);
        for (int k = 0; k < h->dim; k++) row[k] /= norm;
    }
    DCIH_HIP(hipMemcpy(h->d_dirs, h->h_dirs.data(), h->h_dirs.size() * sizeof(float),
                       hipMemcpyHostToDevice));
    return 0;
}

// The rows change: their codes are formed anew, in the same room if it holds them.
void forget_rows8(dcih_index* h) {
    h->rows8_ready = h->rows8_no_room = false;
    if (h->words) h->words->blind = 0;
    h->rows8_demand = 0.0;
}

void forget_point_rows(dcih_index* h) {
    h->point_rows_ready = 0;
    h->point_rows_no_room = false;
    h->point_rows_demand = 0.0;
}
// For an index of n points: the room goes where it does not hold the points' positions, or none would be looked up.
void fit_point_rows(dcih_index* h, int64_t n, int block_size, int thread_size) {
    if (!h->d_point_rows) return;
    if (point_rows_fit((n + block_size - 1) / block_size, h->M, h->L, thread_size) && point_rows_bytes(n, h->M, h->L) <= h->point_rows_room) return;
    (void)hipFree(h->d_point_rows);
    h->d_point_rows = nullptr;
    h->point_rows_room = 0;
    h->point_rows_ready = 0;
}
// Whether the positions are there for a call on stream `s`; fills the table when calls have asked for enough.
constexpr double kPointRowsDemand = 16.0;
int use_point_rows(dcih_index* h, double points, bool recorded, hipStream_t s, bool& use) {
    use = h->point_rows_ready != 0;
    h->point_rows_demand += points;
    if (use || h->point_rows_demand < kPointRowsDemand || h->point_rows_no_room) return 0;
    const size_t need = point_rows_bytes(h->n, h->M, h->L);
    if (need > h->point_rows_room) {
        if (recorded) return 0;
        if (h->d_point_rows) { DCIH_HIP(hipFree(h->d_point_rows)); h->d_point_rows = nullptr; h->point_rows_room = 0; }
        if (hipMalloc((void**)&h->d_point_rows, need) != hipSuccess) {      // points' times do as well
            (void)hipGetLastError();
            h->d_point_rows = nullptr;
            h->point_rows_no_room = true;
            return 0;
        }
        h->point_rows_room = need;
    }
    const int rc = fill_point_rows(h->d_inv, h->d_point_rows, h->n, h->M, h->L, s);
    if (rc) return rc;
    if (!recorded) h->point_rows_ready = 1;
    use = true;
    return 0;
}

int find_near_record(const dcih_index* h, int k, int outer, int T, int maxc) {
    for (int i = 0; i < kNearRecords; i++) {
        const NearRecord& r = h->near_records[i];
        if (r.k == k && r.outer == outer && r.T == T && r.maxc == maxc) return i;
    }
    return -1;
}
int begin_near_record(dcih_index* h, int k, int outer, int T, int maxc) {
    int at = 0;
    for (int i = 1; i < kNearRecords; i++)
        if (h->near_records[i].last < h->near_records[at].last) at = i;
    h->near_tag = h->near_tag % 0xffffu + 1u;
    NearRecord r;
    r.k = k; r.outer = outer; r.T = T; r.maxc = maxc; r.tag = h->near_tag;
    h->near_records[at] = r;
    return at;
}
// The items that were answered and left, as far as calls have written them.
void read_near_record(const dcih_index* h, int at, uint32_t& had, uint32_t& lost) {
    had = lost = 0;
    if (at < 0 || !h->words) return;
    const uint64_t w = h->words->near[at];
    if ((uint32_t)(w >> 48) != h->near_records[at].tag) return;
    had = (uint32_t)w & 0xffffffu;
    lost = (uint32_t)(w >> 24) & 0xffffffu;
}
void forget_near_records(dcih_index* h) {
    for (NearRecord& r : h->near_records) r = NearRecord();
    h->near_last = -1;
}

void release_rows8(dcih_index* h) {
    forget_rows8(h);
    if (h->d_rows8) { (void)hipFree(h->d_rows8); h->d_rows8 = nullptr; h->rows8_bytes = 0; }
}

// Drops the sorted arrays (their arena stays allocated for the next build) but keeps the rows.
int release_sorted(dcih_index* h) {
    h->d_skeys = nullptr;
    h->d_sids = nullptr;
    h->d_inv = nullptr;
    h->d_rpos = nullptr;
    h->rpos_ready = 0;
    forget_point_rows(h);
    forget_rows8(h);
    h->d_stop_hint = nullptr;
    return 0;
}

int release_arena(dcih_index* h) {
    (void)release_sorted(h);
    for (int j = 0; j < 2; j++)
        if (h->arena[j]) { (void)hipFree(h->arena[j]); h->arena[j] = nullptr; h->arena_bytes[j] = 0; }
    return 0;
}

void release_rows(dcih_index* h) {
    if (h->d_own) { (void)hipFree(h->d_own); h->d_own = nullptr; }
    if (h->d_ukeys) { (void)hipFree(h->d_ukeys); h->d_ukeys = nullptr; }
    h->own_rows = 0;
}

// The index is empty; the room of owned rows stays for the next appends.
int release_index(dcih_index* h) {
    const int rc = release_sorted(h);
    h->ukeys_rows = 0;
    h->d_data = nullptr;
    h->n = 0;
    h->block_size = 0;
    return rc;
}

// True while `s` is recording into a graph: nothing may be allocated or freed then.
bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// Puts what follows on stream `s` behind the calls so far that read owned rows.
int after_readers(dcih_index* h, hipStream_t s) {
    if (h->busy_set) DCIH_HIP(hipStreamWaitEvent(s, h->busy, 0));
    return 0;
}
// Marks the end of such a call; where that cannot be done, waits for it.
void mark_reader(dcih_index* h, hipStream_t s, bool recording) {
    if (recording) { h->recorded = true; return; }
    h->busy_set = h->busy && hipEventRecord(h->busy, s) == hipSuccess;
    if (!h->busy_set) { (void)hipGetLastError(); (void)hipDeviceSynchronize(); }
}
// The host waits for them.
int wait_for_readers(dcih_index* h) {
    if (h->busy_set) DCIH_HIP(hipEventSynchronize(h->busy));
    h->busy_set = false;
    return 0;
}

int ensure_ws(dcih_index* h, size_t bytes, hipStream_t s) {
    if (bytes <= h->ws_bytes) return 0;
    if (capturing(s))
        return fail(DCIH_ESTATE, "the workspace would have to grow while the stream is being captured: "
                                 "run the same call once outside the capture first");
    if (h->ws) { DCIH_HIP(hipFree(h->ws)); h->ws = nullptr; h->ws_bytes = 0; }
    DCIH_HIP(hipMalloc(&h->ws, bytes));
    h->ws_bytes = bytes;
    return 0;
}

size_t align_up(size_t v) { return (v + 255) & ~(size_t)255; }

// Makes arena `which` at least `bytes` large.  Growing frees that arena first, so it must
// not hold the live index.
int ensure_arena(dcih_index* h, int which, size_t bytes) {
    if (bytes <= h->arena_bytes[which]) return 0;
    if (h->arena[which]) { DCIH_HIP(hipFree(h->arena[which])); h->arena[which] = nullptr; h->arena_bytes[which] = 0; }
    DCIH_HIP(hipMalloc(&h->arena[which], bytes));
    h->arena_bytes[which] = bytes;
    return 0;
}

// Where the arrays of an index of n points lie inside an arena.
struct ArenaLayout {
    size_t keys, ids, inv, rpos, hint, total;   // byte offsets, and the size of it all
    bool small_parts;                           // partitions of at most 65536 points: 16-bit tables exist
};
ArenaLayout arena_layout(int I, int64_t n, int block_size) {
    ArenaLayout y;
    const size_t cells = (size_t)I * (size_t)n;
    y.small_parts = (n + block_size - 1) / block_size <= 65536;
    const size_t b_keys = align_up(cells * sizeof(float));
    const size_t b_ids = align_up(cells * sizeof(int32_t));
    // +16: the traversal reads whole 16-byte chunks of positions, also at the very end
    const size_t b_inv = y.small_parts ? align_up((cells + 16) * sizeof(uint16_t)) : 0;
    const size_t b_hint = align_up((size_t)3 * block_size * sizeof(float));   // stop step, promotions at the stop, stops seen
    y.keys = 0;
    y.ids = b_keys;
    y.inv = y.ids + b_ids;
    y.rpos = y.inv + b_inv;
    y.hint = y.rpos + b_inv;
    y.total = y.hint + b_hint;
    return y;
}

size_t rows8_records(const dcih_index* h, int64_t n) { return align_up((size_t)n * rows8_record_bytes(h->dim)); }
size_t rows8_room(const dcih_index* h, int64_t n, int block_size) {
    return rows8_records(h, n) + align_up((size_t)3 * block_size * sizeof(uint32_t) + 8);
}

// Whether a call on stream `s` that goes to the dense kernel may compare rows by their codes; forms
// the codes when they have become worth it: a candidate read by its code saves three quarters of its row,
// forming the codes reads every row and writes a quarter of it, so from twice as many candidates as rows on.
// Until they have been seen to be there, calls are put behind their event, whatever the stream.
bool rows8_there(dcih_index* h, hipStream_t s) {
    if (h->rows8_settled) return true;
    // (the event is no part of a capture under way: asking after it is all right there)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool recording = capturing(s) && hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    h->rows8_settled = hipEventQuery(h->rows8_event) == hipSuccess;
    if (!h->rows8_settled) (void)hipGetLastError();
    if (recording) (void)hipThreadExchangeStreamCaptureMode(&mode);
    return h->rows8_settled;
}
int use_rows8(dcih_index* h, double candidates, bool may_form, hipStream_t s, bool& use) {
    use = false;
    if (!rows8_supported(h->dim) || h->rows8_no_room) return 0;
    h->rows8_demand += candidates;
    if (!h->rows8_ready) {
        if (!may_form || h->rows8_demand < 2.0 * (double)h->n || capturing(s)) return 0;
        if (!h->rows8_event) DCIH_HIP(hipEventCreateWithFlags(&h->rows8_event, hipEventDisableTiming));
        const size_t need = rows8_room(h, h->n, h->block_size);
        if (need > h->rows8_bytes) {
            if (h->d_rows8) { DCIH_HIP(hipFree(h->d_rows8)); h->d_rows8 = nullptr; h->rows8_bytes = 0; }
            if (hipMalloc((void**)&h->d_rows8, need) != hipSuccess) {      // whole rows do as well
                (void)hipGetLastError();
                h->d_rows8 = nullptr;
                h->rows8_no_room = true;
                return 0;
            }
            h->rows8_bytes = need;
        }
        const int64_t ppb = (h->n + h->block_size - 1) / h->block_size;
        const int rc = code_rows(h->d_data, h->n, h->dim, ppb, h->block_size, h->d_rows8,
                                 (uint32_t*)(h->d_rows8 + rows8_records(h, h->n)), s);
        if (rc) return rc;
        DCIH_HIP(hipEventRecord(h->rows8_event, s));
        h->rows8_ready = true;
        h->rows8_settled = false;
    } else if (!rows8_there(h, s)) {
        if (capturing(s)) return 0;
        DCIH_HIP(hipStreamWaitEvent(s, h->rows8_event, 0));
    }
    use = true;
    return 0;
}

// Records the start (which = 0) or end (1) event of timer t when profiling.
void mark(dcih_index* h, int t, int which, hipStream_t s) {
    if (!h->profiling) return;
    (void)hipEventRecord(h->ev[2 * t + which], s);
    if (which) h->ev_valid[t] = true;
}

}  // namespace

extern "C" {

const char* dcih_last_error(void) { return g_last_error.c_str(); }

int dcih_abi_version(void) { return 2; }

int dcih_create(int dim, int num_comp_indices, int num_simp_indices, int device,
                uint64_t seed, dcih_index** out) {
    if (!out) return fail(DCIH_EINVAL, "dcih_create: out is null");
    *out = nullptr;
    if (dim <= 0 || num_comp_indices <= 0 || num_simp_indices <= 0)
        return fail(DCIH_EINVAL, "dcih_create: dim and index counts must be positive");
    if ((int64_t)num_comp_indices * num_simp_indices > (1 << 20))
        return fail(DCIH_EINVAL, "dcih_create: too many simple indices");
    int ndev = 0;
    DCIH_HIP(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return fail(DCIH_EINVAL, "dcih_create: no such device");
    DeviceGuard guard(device);
    if (!guard.ok) return fail(DCIH_EHIP, "dcih_create: cannot select device");
    dcih_index* h = new (std::nothrow) dcih_index();
    if (!h) return fail(DCIH_EHIP, "dcih_create: out of host memory");
    h->dim = dim; h->M = num_comp_indices; h->L = num_simp_indices;
    h->device = device; h->seed = seed;
    {   // dies with an L2 of their own: the batch traversal orders its work by them
        int xcds = 0;
        // (the per-die list lengths of the query scratch have room for kMaxXcds dies; a device
        //  that reports more, or none, is treated as one of 8)
        if (hipDeviceGetAttribute(&xcds, hipDeviceAttributeNumberOfXccs, device) == hipSuccess &&
            xcds >= 1 && xcds <= kMaxXcds)
            h->xcds = xcds;
        (void)hipGetLastError();
    }
    if (const int rc_s = resolve_scratch(device)) { delete h; return rc_s; }
    const size_t bytes = (size_t)num_indices(h) * dim * sizeof(float);
    if (hipMalloc(&h->d_dirs, bytes) != hipSuccess) {
        delete h;
        return fail(DCIH_EHIP, "dcih_create: hipMalloc of the directions failed");
    }
    const int rc = draw_directions(h);
    if (rc) { (void)hipFree(h->d_dirs); delete h; return rc; }
    *out = h;
    return DCIH_OK;
}

int dcih_get_directions(const dcih_index* h, float* h_dirs) {
    if (!h || !h_dirs) return fail(DCIH_EINVAL, "dcih_get_directions: null argument");
    std::memcpy(h_dirs, h->h_dirs.data(), h->h_dirs.size() * sizeof(float));
    return DCIH_OK;
}

int dcih_set_directions(dcih_index* h, const float* h_dirs) {
    if (!h || !h_dirs) return fail(DCIH_EINVAL, "dcih_set_directions: null argument");
    if (h->n > 0) return fail(DCIH_ESTATE, "dcih_set_directions: index is not empty");
    DeviceGuard guard(h->device);
    const int rc = wait_for_readers(h);
    if (rc) return rc;
    std::memcpy(h->h_dirs.data(), h_dirs, h->h_dirs.size() * sizeof(float));
    DCIH_HIP(hipMemcpy(h->d_dirs, h_dirs, h->h_dirs.size() * sizeof(float), hipMemcpyHostToDevice));
    return DCIH_OK;
}

// Sorts the projections of `num_points` rows (index i's at d_keys + i * key_stride) into
// arena `which`, which must already be large enough, and makes the result the handle's
// index over the rows at d_data.  Synchronises the stream before returning; on failure the
// handle's fields are untouched.
// With merge_from > 0 the live index (over the first merge_from points, in the other arena) is
// merged with the sorted new points instead of everything being sorted again.
static int sort_into(dcih_index* h, int which, const float* d_keys, int64_t key_stride,
                     int64_t num_points, const float* d_data, int block_size, void* d_tmp,
                     hipStream_t s, int64_t merge_from = 0) {
    const int I = num_indices(h);
    const ArenaLayout y = arena_layout(I, num_points, block_size);
    char* base = (char*)h->arena[which];
    float* skeys = (float*)(base + y.keys);
    int32_t* sids = (int32_t*)(base + y.ids);
    uint16_t* inv = y.small_parts ? (uint16_t*)(base + y.inv) : nullptr;
    float* hint = (float*)(base + y.hint);
    int rc;
    mark(h, DCIH_T_SEGSORT, 0, s);
    if (merge_from > 0)
        rc = segsort_append(h->d_skeys, h->d_sids, merge_from, d_keys, key_stride, I, num_points, block_size,
                            skeys, sids, inv, nullptr, d_tmp, s);
    else
        rc = segsort(d_keys, key_stride, I, num_points, block_size, skeys, sids, inv, nullptr, d_tmp, s);
    mark(h, DCIH_T_SEGSORT, 1, s);
    // like the reference's dci_add, the call returns when the index is complete
    const hipError_t se = hipStreamSynchronize(s);
    if (rc == DCIH_OK && se != hipSuccess)
        rc = fail(DCIH_EHIP, std::string("build: ") + hipGetErrorString(se));
    if (rc) return rc;
    h->d_skeys = skeys; h->d_sids = sids; h->d_inv = inv; h->d_stop_hint = hint;
    h->d_rpos = y.small_parts ? (uint16_t*)(base + y.rpos) : nullptr;
    h->rpos_ready = 0;
    h->index_calls = 0;
    forget_near_records(h);
    forget_point_rows(h);
    forget_rows8(h);
    h->cur = which;
    h->d_data = d_data;
    h->n = num_points;
    h->block_size = block_size;
    h->hint_k = h->hint_outer = h->hint_T = h->hint_maxc = 0;
    return DCIH_OK;
}

int dcih_add(dcih_index* h, int dim, int64_t num_points, const float* d_data,
             int block_size, int thread_size, void* stream) {
    if (!h) return fail(DCIH_EINVAL, "dcih_add: null handle");
    if (dim != h->dim) return fail(DCIH_EINVAL, "dcih_add: dim differs from the index's");
    if (h->n > 0) return fail(DCIH_ESTATE, "dcih_add: index already holds points; clear it first");
    if (num_points <= 0 || !d_data) return fail(DCIH_EINVAL, "dcih_add: no points given");
    if (num_points > 0x7fffffffLL) return fail(DCIH_EINVAL, "dcih_add: more than 2^31-1 points");
    if (block_size <= 0 || thread_size <= 0)
        return fail(DCIH_EINVAL, "dcih_add: block_size and thread_size must be positive");
    DeviceGuard guard(h->device);
    hipStream_t s = (hipStream_t)stream;
    const int I = num_indices(h);
    // one arena for what the index keeps, the workspace for what only the build needs
    // (the unsorted keys): a rebuild of the same size allocates and frees nothing
    const size_t b_keys = align_up((size_t)I * num_points * sizeof(float));
    const size_t tmp_bytes = segsort_tmp_bytes(I, num_points, block_size);
    int rc = wait_for_readers(h);
    if (rc) return rc;
    release_rows(h);                // (rows of appends before a clear: this index borrows its rows)
    if (h->rows8_bytes < rows8_room(h, num_points, block_size)) release_rows8(h);
    fit_point_rows(h, num_points, block_size, thread_size);
    rc = ensure_arena(h, h->cur, arena_layout(I, num_points, block_size).total);
    if (rc == DCIH_OK) rc = ensure_ws(h, b_keys + align_up(tmp_bytes), s);
    if (rc == DCIH_OK) {
        float* d_keys = (float*)h->ws;
        mark(h, DCIH_T_PROJECT, 0, s);
        rc = project(h->d_dirs, I, d_data, num_points, dim, d_keys, num_points, s);
        mark(h, DCIH_T_PROJECT, 1, s);
        if (rc == DCIH_OK)
            rc = sort_into(h, h->cur, d_keys, num_points, num_points, d_data, block_size,
                           tmp_bytes ? (void*)((char*)h->ws + b_keys) : nullptr, s);
        else
            (void)hipStreamSynchronize(s);
    }
    if (rc) (void)release_index(h);
    return rc;
}

int dcih_append(dcih_index* h, int dim, int64_t num_points, const float* d_data,
                int block_size, int thread_size, void* stream) {
    if (!h) return fail(DCIH_EINVAL, "dcih_append: null handle");
    if (dim != h->dim) return fail(DCIH_EINVAL, "dcih_append: dim differs from the index's");
    if (num_points <= 0 || !d_data) return fail(DCIH_EINVAL, "dcih_append: no points given");
    if (block_size <= 0 || thread_size <= 0)
        return fail(DCIH_EINVAL, "dcih_append: block_size and thread_size must be positive");
    if (h->n > 0 && block_size != h->block_size)
        return fail(DCIH_EINVAL, "dcih_append: block_size differs from the one the index was built with");
    const int64_t total = h->n + num_points;
    if (total > 0x7fffffffLL) return fail(DCIH_EINVAL, "dcih_append: more than 2^31-1 points");
    DeviceGuard guard(h->device);
    hipStream_t s = (hipStream_t)stream;
    const int I = num_indices(h);
    const size_t row_bytes = (size_t)dim * sizeof(float);

    // Everything that can fail for lack of memory happens before the index is touched:
    // room for the rows and their projections (both owned by the index, capacity doubles
    // so that copies amortise), for the next index in the spare arena, and for the sort.
    int64_t have_keys = (h->n > 0 && h->d_data == h->d_own) ? std::min(h->ukeys_rows, h->n) : 0;
    const int spare = 1 - h->cur;
    // Merging the old slices with the sorted new points instead of sorting everything again.
    // Both are built; left to choose, the append sorts: the one-pass LDS sort moves 16 bytes per
    // index entry, split + merge + inverse move 40, and on an MI355X the sort is the faster of the
    // two at every size of the incremental workload (8.7 against 9.0 ms for 1M onto 19M points).
    const bool merge = h->n > 0 && h->append_mode == 2 && h->d_inv != nullptr &&
                       segsort_append_supported(h->n, total, block_size);
    if (h->append_mode == 2 && h->n > 0 && !merge)
        return fail(DCIH_EUNSUPPORTED, "dcih_append: this shape cannot be appended by merging (partitions too long)");
    // (a release to the device is all its waiters need: they overwrite what was read)
    if (!h->busy) DCIH_HIP(hipEventCreateWithFlags(&h->busy, hipEventDisableTiming | hipEventReleaseToDevice));
    // (calls that read borrowed rows are not marked)
    if (h->n > 0 && h->d_data != h->d_own) DCIH_HIP(hipDeviceSynchronize());
    int rc = after_readers(h, s);
    if (rc) return rc;
    // An empty index has no rows to keep: room of earlier ones that does not hold the new ones goes first.
    if (h->n == 0 && h->own_rows < total) release_rows(h);
    float* rows = h->d_own;
    float* ukeys = h->d_ukeys;
    int64_t cap = h->own_rows;
    // (codes of the rows so far are not the next index's; their room goes where it will not hold its codes)
    if (h->rows8_bytes < rows8_room(h, total, block_size)) release_rows8(h);
    float* fresh_rows = nullptr;
    float* fresh_keys = nullptr;
    if (!rows || cap < total) {
        cap = std::max<int64_t>(total, 2 * h->own_rows);
        if (hipMalloc(&fresh_rows, (size_t)cap * row_bytes) != hipSuccess ||
            hipMalloc(&fresh_keys, (size_t)I * cap * sizeof(float)) != hipSuccess) {
            (void)hipGetLastError();
            if (fresh_rows) (void)hipFree(fresh_rows);
            return fail(DCIH_EHIP, "dcih_append: out of device memory for the rows (the index is unchanged)");
        }
        rows = fresh_rows;
        ukeys = fresh_keys;
    }
    const size_t tmp_bytes = merge ? segsort_append_tmp_bytes(I, total) : segsort_tmp_bytes(I, total, block_size);
    rc = ensure_arena(h, h->n > 0 ? spare : h->cur,
                          std::max(arena_layout(I, total, block_size).total, arena_layout(I, cap, block_size).total));
    if (rc == DCIH_OK && tmp_bytes) rc = ensure_ws(h, align_up(tmp_bytes), s);
    hipError_t e = hipSuccess;
    if (rc == DCIH_OK && h->n > 0 && rows != h->d_data)        // rows (and projections) indexed so far
        e = hipMemcpyAsync(rows, h->d_data, (size_t)h->n * row_bytes, hipMemcpyDeviceToDevice, s);
    if (rc == DCIH_OK && e == hipSuccess && have_keys > 0 && ukeys != h->d_ukeys)
        e = hipMemcpy2DAsync(ukeys, (size_t)cap * sizeof(float), h->d_ukeys, (size_t)h->own_rows * sizeof(float),
                             (size_t)have_keys * sizeof(float), (size_t)I, hipMemcpyDeviceToDevice, s);
    if (rc == DCIH_OK && e == hipSuccess)
        e = hipMemcpyAsync(rows + (size_t)h->n * dim, d_data, (size_t)num_points * row_bytes,
                           hipMemcpyDeviceToDevice, s);
    if (rc == DCIH_OK && e != hipSuccess) rc = fail(DCIH_EHIP, std::string("dcih_append: ") + hipGetErrorString(e));
    if (rc == DCIH_OK) {
        // only rows without kept projections are projected: the new ones, after a plain
        // dcih_add (which keeps none) all of them
        mark(h, DCIH_T_PROJECT, 0, s);
        rc = project(h->d_dirs, I, rows + (size_t)have_keys * dim, total - have_keys, dim,
                     ukeys + have_keys, cap, s);
        mark(h, DCIH_T_PROJECT, 1, s);
    }
    if (rc == DCIH_OK)
        // the partition boundaries move with the total, so every slice is formed again
        rc = sort_into(h, h->n > 0 ? spare : h->cur, ukeys, cap, total, rows, block_size,
                       tmp_bytes ? h->ws : nullptr, s, merge ? h->n : 0);
    else
        (void)hipStreamSynchronize(s);
    h->busy_set = false;            // (the stream was waited for, and was behind them)
    if (rc) {       // the index stays as it was
        if (fresh_rows) (void)hipFree(fresh_rows);
        if (fresh_keys) (void)hipFree(fresh_keys);
        return rc;
    }
    if (fresh_rows) {
        if (h->d_own) (void)hipFree(h->d_own);
        if (h->d_ukeys) (void)hipFree(h->d_ukeys);
        h->d_own = fresh_rows;
        h->d_ukeys = fresh_keys;
        h->own_rows = cap;
    }
    h->ukeys_rows = total;
    fit_point_rows(h, total, block_size, thread_size);
    return DCIH_OK;
}

// dcih_query and dcih_query_noalloc.  `fixed` = take every byte of scratch from the
// device's static array and refuse what does not fit, instead of growing the handle's
// workspace.
static int query_impl(dcih_index* h, int dim, int num_queries, const float* d_query,
                      int num_neighbours, int blind, int num_outer_iterations,
                      int max_num_candidates, int block_size, int thread_size,
                      int32_t* d_nn, float* d_dists, uint64_t* d_counters, void* stream,
                      bool fixed, bool float_ids, const char* who, bool whole = false, bool later_part = false) {
    const std::string me(who);
    if (!h) return fail(DCIH_EINVAL, me + ": null handle");
    if (dim != h->dim) return fail(DCIH_EINVAL, me + ": dim differs from the index's");
    if (h->n <= 0) return fail(DCIH_ESTATE, me + ": index is empty");
    if (num_neighbours <= 0 || num_neighbours > h->n)
        return fail(DCIH_EINVAL, me + ": num_neighbours must be in [1, num_points]");
    if (num_queries < 0 || (num_queries > 0 && (!d_query || !d_nn || (!blind && !d_dists))))
        return fail(DCIH_EINVAL, me + ": null buffer");
    // blind: as many candidates per query as the reference's result buffer holds (:782-783)
    const int64_t num_results =
        blind ? std::min<int64_t>(max_num_candidates, num_outer_iterations) : num_neighbours;
    if (num_results <= 0)
        return fail(DCIH_EINVAL, me + ": blind querying needs positive max_num_candidates and num_outer_iterations");
    if (thread_size <= 0) return fail(DCIH_EINVAL, me + ": thread_size must be positive");
    if (block_size != h->block_size)
        return fail(DCIH_EINVAL, me + ": block_size differs from the one the index was built with");
    if (num_queries == 0) return DCIH_OK;
    DeviceGuard guard(h->device);
    hipStream_t s = (hipStream_t)stream;
    // Under capture nothing runs: what this call's kernels fill or clear for later calls has not been when it returns.
    const bool recorded = capturing(s);
    struct Reader {                 // (whatever way the call ends)
        dcih_index* h;
        hipStream_t s;
        bool recording;
        ~Reader() { if (h) mark_reader(h, s, recording); }
    } reader{h->d_data == h->d_own ? h : nullptr, s, recorded};
    if (reader.h && !recorded) {
        const int rc = after_readers(h, s);
        if (rc) return rc;
    }
    const int I = num_indices(h);
    // the scratch of this call: the handle's workspace, grown as needed, or the static array
    char* ws_base = nullptr;
    auto get_ws = [&](size_t bytes) -> int {
        if (!fixed) {
            const int rc = ensure_ws(h, bytes, s);
            ws_base = (char*)h->ws;
            return rc;
        }
        ws_base = (char*)scratch_of(h->device);
        if (!ws_base) return fail(DCIH_ESTATE, me + ": the scratch array of this device was not located");
        if (bytes > kScratchBytes)
            return fail(DCIH_EINVAL, me + ": this call needs " + std::to_string(bytes) +
                                     " bytes of scratch and the fixed array holds " +
                                     std::to_string(kScratchBytes) + "; pass fewer queries per call");
        return 0;
    };

    h->ev_valid[DCIH_T_BATCH] = h->ev_valid[DCIH_T_DENSE] = false;
    for (int64_t& r : h->route) r = 0;
    if (!later_part) h->plan[0] = h->plan[2] = 0;
    if (!later_part) h->plan[1] = 1;
    QueryArgs a;
    a.skeys = h->d_skeys; a.sids = h->d_sids; a.inv = h->d_inv; a.data = h->d_data; a.query = d_query;
    a.rpos = h->d_rpos; a.rpos_ready = &h->rpos_ready; a.recorded = recorded ? 1 : 0;
    a.point_rows = nullptr;
    a.hints_cold = 0;
    a.mode = h->traversal; a.item_list = nullptr; a.item_count = nullptr; a.dense = nullptr;
    a.xcds = h->xcds; a.q_first = 0; a.q_count = num_queries;
    a.dense_items = nullptr; a.dense_count = nullptr; a.dense_cap = 0;
    a.wide_items = nullptr; a.wide_count = nullptr; a.wide_cap = 0;
    a.block_list = nullptr; a.block_list_count = nullptr; a.full_tables = a.few_items = 0;
    a.dense_min_promos = h->dense_min_promos;
    a.dense_by_cost = h->dense_by_cost;
    a.hand_over_at = 0;
    a.expect_steps = a.expect_promotions = 0.0f;
    a.rows8 = nullptr; a.rows8_rec = 0; a.rows8_bounds = nullptr; a.query8 = nullptr;
    a.picked = nullptr; a.picked_count = nullptr; a.picked_exact = a.picked_cover = a.picked_expect = 0; a.picked_ticket = nullptr; a.left = nullptr; a.left_count = nullptr; a.left_cap = 0; a.only = nullptr; a.only_round = 0;
    a.share = 1.0; a.pick_first = 0.0; a.pick_rounds = a.pick_rank = a.pick_near = a.pick_confirm = a.may_confirm = a.pick_sample = 0; a.pick_most = 1.0f;
    a.near_bounds = nullptr; a.near_limit = nullptr; a.near_stride = 0; a.near_shift = a.near_tiles = 0; a.pick_rule = fixed || whole ? 1 : h->rounds;
    a.phase_ticks = h->d_phase_ticks;
    a.near_room = h->near_room;
    a.pick_parts = 1;
    a.round_items = h->d_round_items;
    a.blind_word = nullptr;
    a.confirm_word = nullptr;
    a.confirm_tag = 0;
    a.confirm_had = a.confirm_lost = 0;
    a.index_calls = 0;
    a.selected = &h->route[3];
    a.window_launches = &h->plan[2];
    a.stop_hint = nullptr;
    a.N = h->n;
    a.ppb = (h->n + block_size - 1) / block_size;
    a.dim = dim; a.M = h->M; a.L = h->L; a.B = block_size; a.T = thread_size;
    a.T_magic = thread_size > 1 ? (unsigned)((0x100000000ull + (unsigned)thread_size - 1u) / (unsigned)thread_size) : 0u;
    a.nq = num_queries; a.k = (int)std::min<int64_t>(num_results, 0x7fffffff);
    a.k_stop = num_neighbours; a.blind = blind ? 1 : 0;
    a.kcap = (int)std::min<int64_t>(num_results, a.ppb);
    a.stop_at = (int64_t)num_outer_iterations * h->L;
    a.max_cand = max_num_candidates;
    a.counters = (unsigned long long*)d_counters;
    a.out_ids = d_nn; a.out_dists = d_dists; a.float_ids = float_ids ? 1 : 0;

    if (fixed && num_results > 8192)
        return fail(DCIH_EUNSUPPORTED, me + ": more than 8192 results per query need the row-per-query "
                                            "workspace of dcih_query");
    if (num_results > 8192 &&
        (blind || num_neighbours < a.ppb || (num_neighbours == a.ppb && d_counters))) {
        // More results than the top-k tables hold while partitions may still stop early: the
        // step-by-step traversal records every candidate in a dense row per query, which is
        // then sorted like the full ranking below.
        const int chunk = exhaustive_chunk(h->n, num_queries);
        QueryArgs probe = a;
        probe.nq = chunk; probe.kcap = 1;
        const size_t qp_bytes = align_up((size_t)I * chunk * sizeof(float));
        const size_t rank_bytes = align_up(exhaustive_ws_bytes(h->n, chunk, (int)std::min<int64_t>(h->n, 0x7fffffff)));
        const size_t gs_bytes = align_up(query_gscratch_bytes(probe));
        int rc = get_ws(qp_bytes + rank_bytes + gs_bytes);
        if (rc) return rc;
        a.gscratch = gs_bytes ? (uint32_t*)(ws_base + qp_bytes + rank_bytes) : nullptr;
        mark(h, DCIH_T_TRAVERSE, 0, s);
        rc = query_dense(a, h->d_dirs, ws_base, chunk, s);
        mark(h, DCIH_T_TRAVERSE, 1, s);
        return rc;
    }
    // The stop rule (:598-607) can also never fire when a partition has fewer points than
    // max_num_candidates and fewer windows per simple index (at most ppb / T + 3) than
    // num_outer_iterations: the loop then runs every partition dry, as in the reference's own
    // example (3000 points in 100 partitions, 5000 iterations).  Left to pick, the engine
    // computes that answer directly as well (not with the fixed scratch, which a million
    // points per query would overrun: there the traversal kernels give the same neighbours).
    const bool runs_dry = !blind && !fixed && h->traversal == 0 && a.ppb < (int64_t)max_num_candidates &&
                          a.ppb / thread_size + 4 < (int64_t)num_outer_iterations;
    if (!blind && (num_neighbours > 8192 || runs_dry)) {
        // With more neighbours asked for than a partition holds, no partition can stop early
        // (c0 counts promotions of one partition, :598-607), so the answer is the full ranking
        // and is computed as such.  (With exactly as many, the results are the same but the
        // last step may end the loop before its idle pass: the counters then come from the
        // traversal above.)
        const int chunk = exhaustive_chunk(h->n, num_queries);
        const size_t qp_bytes = d_counters ? align_up((size_t)I * num_queries * sizeof(float)) : 0;
        int rc = get_ws(qp_bytes + exhaustive_ws_bytes(h->n, chunk, a.k));
        if (rc) return rc;
        if (d_counters) {
            rc = project(h->d_dirs, I, d_query, num_queries, dim, (float*)ws_base, num_queries, s);
            if (rc) return rc;
            a.qproj = (float*)ws_base;
        }
        mark(h, DCIH_T_TRAVERSE, 0, s);
        rc = query_exhaustive(a, ws_base + qp_bytes, chunk, s);
        mark(h, DCIH_T_TRAVERSE, 1, s);
        return rc;
    }

    // (where earlier calls' items had to be left, every 256th call tries again, as if nothing were on record: a few items go ahead)
    int record = find_near_record(h, num_neighbours, num_outer_iterations, thread_size, max_num_candidates);
    read_near_record(h, record, a.confirm_had, a.confirm_lost);
    if (record >= 0 && h->near_records[record].rests >= 255) a.confirm_had = a.confirm_lost = 0;
    a.index_calls = h->index_calls++;
    (void)plan_rounds(a);
    if (a.pick_parts > 1) {
        const int part = (num_queries + a.pick_parts - 1) / a.pick_parts;
        for (int q = 0; q < num_queries; q += part) {
            const int rc = query_impl(h, dim, std::min(part, num_queries - q), d_query + (size_t)q * dim, num_neighbours, blind, num_outer_iterations, max_num_candidates,
                                      block_size, thread_size, d_nn + (size_t)q * num_neighbours, d_dists + (size_t)q * num_neighbours, d_counters, stream, fixed, float_ids, who,
                                      whole, later_part || q > 0);
            if (rc) return rc;
        }
        h->plan[1] = a.pick_parts;
        return DCIH_OK;
    }
    if (a.pick_confirm) {
        if (record < 0) record = begin_near_record(h, num_neighbours, num_outer_iterations, thread_size, max_num_candidates);
        h->near_records[record].rests = 0;
        h->near_last = record;
    } else if (record >= 0 && a.pick_rounds) {
        h->near_records[record].rests++;
    }
    if (record >= 0) h->near_records[record].last = ++h->near_calls;
    if (a.pick_near || a.pick_confirm) {
        if (!h->words && !recorded) {
            void* p = nullptr;
            if (hipHostMalloc(&p, sizeof(HostWords), hipHostMallocDefault) == hipSuccess) { std::memset(p, 0, sizeof(HostWords)); h->words = (volatile HostWords*)p; }
            else (void)hipGetLastError();
        }
        void* p = nullptr;
        if (h->words && hipHostGetDevicePointer(&p, (void*)h->words, 0) == hipSuccess) {
            HostWords* d_words = (HostWords*)p;
            if (a.pick_near) a.blind_word = &d_words->blind;
            if (a.pick_confirm) { a.confirm_word = (unsigned long long*)&d_words->near[record]; a.confirm_tag = h->near_records[record].tag; }
        }
    }
    const bool bounds_failed = h->words && h->words->blind;      // (of earlier calls)
    size_t q8_bytes = 0;
    if (!blind && (!a.pick_near || bounds_failed) && dense_traversal_supported(a, nullptr)) {      // (near rows only: few enough to be read whole)
        const bool all_dense = takes_dense_kernel(a);
        bool use = false;
        const double per_item = std::min((double)a.ppb, expected_promotions(a));
        const int rc8 = use_rows8(h, all_dense ? (double)num_queries * block_size * per_item * (bounds_failed ? 1.0 : a.share) : 0.0, all_dense && !fixed, s, use);
        if (rc8) return rc8;
        if (use) {
            a.rows8 = h->d_rows8; a.rows8_rec = rows8_record_bytes(dim); a.rows8_bounds = (uint32_t*)(h->d_rows8 + rows8_records(h, h->n));
            if (dense_traversal_supported(a, nullptr)) q8_bytes = align_up((size_t)num_queries * rows8_query_bytes(dim));
            else a.rows8 = nullptr;      // (no room for the longer list of what is kept)
        }
    }
    // The hints, which only the batch kernel reads, describe where traversals of one query shape stop;
    // forget them when it changes (cleared by a kernel: a memset node is not safe in a captured graph; the
    // table's room is a multiple of 256 bytes, so whole 64-bit words may be cleared)
    if (!(dense_traversal_supported(a, nullptr) && takes_dense_kernel(a))) {
        if (h->hint_k != num_neighbours || h->hint_outer != num_outer_iterations ||
            h->hint_T != thread_size || h->hint_maxc != max_num_candidates) {
            const int rc = zero_words64(h->d_stop_hint, (int64_t)(((size_t)3 * block_size * sizeof(float) + 7) / 8), s);
            if (rc) return rc;
            if (!recorded) {
                h->hint_k = num_neighbours; h->hint_outer = num_outer_iterations;
                h->hint_T = thread_size; h->hint_maxc = max_num_candidates;
            }
            a.hints_cold = 1;
        }
        a.stop_hint = h->d_stop_hint;
    }
    const size_t qp_bytes = align_up((size_t)I * num_queries * sizeof(float));
    const size_t part_bytes = align_up(query_part_bytes(a));
    const size_t gs_bytes = align_up(query_gscratch_bytes(a));
    const size_t redo_bytes = align_up((size_t)num_queries * block_size * sizeof(int32_t));
    // per die one list of the items the batch kernel leaves to the dense kernel
    a.dense_cap = (int64_t)num_queries * (block_size / h->xcds + 1) + 64;
    const bool dense_lists = h->traversal == 0 && h->dense_min_promos > 0 &&
                             dense_traversal_supported(a, nullptr) && block_traversal_supported(a, nullptr);
    const size_t dense_bytes = dense_lists ? align_up((size_t)h->xcds * a.dense_cap * sizeof(int32_t)) : 0;
    // (the second pass may have to take every item, up to what one launch of 256-thread workgroups covers)
    a.wide_cap = std::min((int64_t)num_queries * block_size, (int64_t)1 << 23);
    const size_t wide_bytes = align_up((size_t)a.wide_cap * sizeof(int32_t));
    const size_t ws_bytes = qp_bytes + part_bytes + gs_bytes + redo_bytes + 256 + dense_bytes + wide_bytes;
    if (fixed && ws_bytes + q8_bytes > kScratchBytes) { a.rows8 = nullptr; q8_bytes = 0; }
    // (room for confirm.hip also where this call goes without it: the next one like it may not, and may be recorded, when nothing can grow)
    const size_t need = ws_bytes + q8_bytes + (a.pick_rounds ? bounds_bytes(a) : 0);
    size_t most = need;
    if (a.pick_rounds && a.may_confirm && !a.pick_confirm) {
        QueryArgs with = a;
        with.pick_confirm = 1;
        most = ws_bytes + q8_bytes + bounds_bytes(with);
    }
    int rc = get_ws(most);
    if (rc && most > need) {
        (void)hipGetLastError();
        rc = get_ws(need);
    }
    if (rc && a.pick_rounds) {      // no room for the bounds: everything is traversed, which needs less (the same results)
        (void)hipGetLastError();
        return query_impl(h, dim, num_queries, d_query, num_neighbours, blind, num_outer_iterations, max_num_candidates,
                          block_size, thread_size, d_nn, d_dists, d_counters, stream, fixed, float_ids, who, true);
    }
    if (rc) return rc;
    // A point's positions side by side for the dense kernel's near rows.  To form them takes as long as the look-ups of all points by eight queries.
    if (a.pick_rounds && a.pick_near && point_rows_fit(a.ppb, a.M, a.L, a.T) && point_rows_pay(a)) {
        bool use = false;
        rc = use_point_rows(h, (double)num_queries * a.share, recorded, s, use);
        if (rc) return rc;
        if (use) a.point_rows = h->d_point_rows;
    }
    h->plan[0] = a.pick_rounds ? a.pick_confirm : 0;
    h->route[0] = a.pick_rounds; h->route[1] = a.pick_near; h->route[2] = a.pick_sample;
    char* base = ws_base;
    float* d_qproj = (float*)base;
    a.qproj = d_qproj;
    a.part = (unsigned long long*)(base + qp_bytes);
    a.gscratch = gs_bytes ? (uint32_t*)(base + qp_bytes + part_bytes) : nullptr;
    a.redo_items = (int32_t*)(base + qp_bytes + part_bytes + gs_bytes);
    a.redo_count = (uint32_t*)(base + qp_bytes + part_bytes + gs_bytes + redo_bytes);
    a.dense_count = a.redo_count + 1;         // one length per die, cleared together with redo_count
    a.dense_items = dense_lists ? (int32_t*)(base + qp_bytes + part_bytes + gs_bytes + redo_bytes + 256) : nullptr;
    a.wide_count = a.redo_count + kListCountWords - 1;      // (the last of the list lengths that are cleared together)
    a.wide_items = (int32_t*)(base + qp_bytes + part_bytes + gs_bytes + redo_bytes + 256 + dense_bytes);

    mark(h, DCIH_T_QPROJECT, 0, s);
    rc = project(h->d_dirs, I, d_query, num_queries, dim, d_qproj, num_queries, s);
    mark(h, DCIH_T_QPROJECT, 1, s);
    if (rc) return rc;
    if (a.rows8) {
        unsigned char* q8 = (unsigned char*)(base + qp_bytes + part_bytes + gs_bytes + redo_bytes + 256 + dense_bytes + wide_bytes);
        rc = code_queries(d_query, num_queries, dim, q8, s);
        if (rc) return rc;
        a.query8 = q8;
    }
    // events in the order query() records them: traversal start, batch kernel end, dense
    // kernel end, traversal end, merge end
    // (of a call in parts the traversal starts with the first one's)
    hipEvent_t qev[5] = {later_part ? nullptr : h->ev[2 * DCIH_T_TRAVERSE], h->ev[2 * DCIH_T_BATCH + 1], h->ev[2 * DCIH_T_DENSE + 1],
                         h->ev[2 * DCIH_T_TRAVERSE + 1], h->ev[2 * DCIH_T_MERGE + 1]};
    bool ran[2] = {false, false};
    rc = query(a, base + ws_bytes + q8_bytes, s, h->profiling ? qev : nullptr, ran);
    if (rc == DCIH_OK && h->profiling) {
        h->ev_valid[DCIH_T_TRAVERSE] = h->ev_valid[DCIH_T_MERGE] = true;
        h->ev_valid[DCIH_T_BATCH] = ran[0];
        h->ev_valid[DCIH_T_DENSE] = ran[1];
    }
    return rc;
}

int dcih_query(dcih_index* h, int dim, int num_queries, const float* d_query,
               int num_neighbours, int blind, int num_outer_iterations,
               int max_num_candidates, int block_size, int thread_size,
               int32_t* d_nn, float* d_dists, uint64_t* d_counters, void* stream) {
    return query_impl(h, dim, num_queries, d_query, num_neighbours, blind, num_outer_iterations,
                      max_num_candidates, block_size, thread_size, d_nn, d_dists, d_counters, stream,
                      false, false, "dcih_query");
}

int dcih_query_float_ids(dcih_index* h, int dim, int num_queries, const float* d_query,
                         int num_neighbours, int blind, int num_outer_iterations,
                         int max_num_candidates, int block_size, int thread_size,
                         float* d_nn, float* d_dists, uint64_t* d_counters, void* stream) {
    return query_impl(h, dim, num_queries, d_query, num_neighbours, blind, num_outer_iterations,
                      max_num_candidates, block_size, thread_size, (int32_t*)d_nn, d_dists, d_counters, stream,
                      false, true, "dcih_query_float_ids");
}

int dcih_query_noalloc(dcih_index* h, int dim, int num_queries, const float* d_query,
                       int num_neighbours, int blind, int num_outer_iterations,
                       int max_num_candidates, int block_size, int thread_size,
                       int32_t* d_nn, float* d_dists, uint64_t* d_counters, void* stream) {
    return query_impl(h, dim, num_queries, d_query, num_neighbours, blind, num_outer_iterations,
                      max_num_candidates, block_size, thread_size, d_nn, d_dists, d_counters, stream,
                      true, false, "dcih_query_noalloc");
}

int64_t dcih_debug_launch_map(int xcds, int block_size, int num_queries, int64_t block,
                              int* b, int* q, int* queries_per_launch) {
    if (xcds < 1 || block_size < 1 || num_queries < 1) return -1;
    const int per_launch = block_queries_per_launch(xcds, block_size, num_queries);
    if (queries_per_launch) *queries_per_launch = per_launch;
    if (per_launch < 1) return -1;
    const int nq = std::min(per_launch, num_queries);
    const int64_t items = block_items(xcds, block_size, nq);
    if (b && q && block >= 0 && block < items) {
        int bb = -1, qq = -1;
        if (!block_item(block, xcds, block_size, nq, bb, qq)) bb = qq = -1;
        *b = bb; *q = qq;
    }
    return items;
}

int dcih_debug_positions(dcih_index* h, uint16_t* d_inv, uint16_t* d_rpos, void* stream) {
    if (!h) return fail(DCIH_EINVAL, "dcih_debug_positions: null handle");
    if (h->n <= 0) return fail(DCIH_ESTATE, "dcih_debug_positions: the index is empty");
    if (!h->d_inv || !h->d_rpos) return fail(DCIH_EUNSUPPORTED, "dcih_debug_positions: this index keeps no position tables");
    DeviceGuard guard(h->device);
    hipStream_t s = (hipStream_t)stream;
    const size_t cells = (size_t)num_indices(h) * (size_t)h->n;
    if (d_inv) DCIH_HIP(hipMemcpyAsync(d_inv, h->d_inv, cells * sizeof(uint16_t), hipMemcpyDeviceToDevice, s));
    if (d_rpos) {
        if (!h->rpos_ready) {
            // (rows of the first simple indices are never written: clear the table so that they read as zeros)
            DCIH_HIP(hipMemsetAsync(h->d_rpos, 0, cells * sizeof(uint16_t), s));
            const int rc = fill_positions_by_first(h->d_sids, h->d_inv, h->d_rpos, h->n, h->M, h->L, (h->n + h->block_size - 1) / h->block_size, h->block_size, s);
            if (rc) return rc;
            h->rpos_ready = 1;
        }
        DCIH_HIP(hipMemcpyAsync(d_rpos, h->d_rpos, cells * sizeof(uint16_t), hipMemcpyDeviceToDevice, s));
    }
    DCIH_HIP(hipStreamSynchronize(s));
    return DCIH_OK;
}

int dcih_set_option(dcih_index* h, int option, int value) {
    if (!h) return fail(DCIH_EINVAL, "dcih_set_option: null handle");
    if (option == DCIH_OPT_TRAVERSAL && value >= 0 && value <= 3) {
        h->traversal = value;
        return DCIH_OK;
    }
    if (option == DCIH_OPT_DENSE_MIN_PROMOTIONS && value >= 0) {
        h->dense_min_promos = value;
        h->dense_by_cost = 0;
        return DCIH_OK;
    }
    if (option == DCIH_OPT_APPEND && value >= 0 && value <= 2) {
        h->append_mode = value;
        return DCIH_OK;
    }
    if (option == DCIH_OPT_ROUNDS && value >= 0 && value <= 2) {
        h->rounds = value;
        return DCIH_OK;
    }
    if (option == DCIH_OPT_FORGET_HINTS) {
        h->hint_k = h->hint_outer = h->hint_T = h->hint_maxc = 0;     // the next query clears the table
        return DCIH_OK;
    }
    return fail(DCIH_EINVAL, "dcih_set_option: unknown option or value");
}

int dcih_debug_route(const dcih_index* h, int64_t* route) {
    if (!h || !route) return fail(DCIH_EINVAL, "dcih_debug_route: null argument");
    for (int i = 0; i < 4; i++) route[i] = h->route[i];
    return DCIH_OK;
}

int dcih_debug_round_items(dcih_index* h, uint32_t* d_items) {
    if (!h) return fail(DCIH_EINVAL, "dcih_debug_round_items: null handle");
    h->d_round_items = d_items;
    return DCIH_OK;
}

int dcih_debug_confirmed(const dcih_index* h, uint32_t* counts) {
    if (!h || !counts) return fail(DCIH_EINVAL, "dcih_debug_confirmed: null argument");
    read_near_record(h, h->near_last, counts[0], counts[1]);
    return DCIH_OK;
}

int dcih_debug_plan(const dcih_index* h, int64_t* plan) {
    if (!h || !plan) return fail(DCIH_EINVAL, "dcih_debug_plan: null argument");
    for (int i = 0; i < 3; i++) plan[i] = h->plan[i];
    return DCIH_OK;
}

int dcih_debug_near_room(dcih_index* h, int64_t bytes) {
    if (!h || bytes < 1) return fail(DCIH_EINVAL, "dcih_debug_near_room: null handle or no room");
    h->near_room = (size_t)bytes;
    return DCIH_OK;
}

int dcih_phase_profile(dcih_index* h, uint64_t* d_ticks) {
    if (!h) return fail(DCIH_EINVAL, "dcih_phase_profile: null handle");
    h->d_phase_ticks = (unsigned long long*)d_ticks;
    return DCIH_OK;
}

int dcih_profile(dcih_index* h, int enable) {
    if (!h) return fail(DCIH_EINVAL, "dcih_profile: null handle");
    DeviceGuard guard(h->device);
    if (enable && !h->ev[0]) {
        for (auto& e : h->ev) DCIH_HIP(hipEventCreate(&e));
    }
    h->profiling = enable != 0;
    for (auto& v : h->ev_valid) v = false;
    return DCIH_OK;
}

int dcih_last_timings(dcih_index* h, float* h_ms) {
    if (!h || !h_ms) return fail(DCIH_EINVAL, "dcih_last_timings: null argument");
    if (!h->profiling) return fail(DCIH_ESTATE, "dcih_last_timings: profiling is off");
    DeviceGuard guard(h->device);
    for (int t = 0; t < DCIH_NUM_TIMERS; t++) {
        h_ms[t] = -1.0f;
        if (!h->ev_valid[t]) continue;
        // timers that start where another one ends: the merge after the traversal, the batch
        // kernel at the traversal's start, the dense kernel after the batch kernel
        hipEvent_t a = h->ev[2 * t];
        if (t == DCIH_T_MERGE) a = h->ev[2 * DCIH_T_TRAVERSE + 1];
        if (t == DCIH_T_BATCH) a = h->ev[2 * DCIH_T_TRAVERSE];
        if (t == DCIH_T_DENSE) a = h->ev_valid[DCIH_T_BATCH] ? h->ev[2 * DCIH_T_BATCH + 1] : h->ev[2 * DCIH_T_TRAVERSE];
        hipEvent_t b = h->ev[2 * t + 1];
        DCIH_HIP(hipEventSynchronize(b));
        DCIH_HIP(hipEventElapsedTime(&h_ms[t], a, b));
    }
    return DCIH_OK;
}

int dcih_get_index(const dcih_index* h, float* h_keys, int32_t* h_ids) {
    if (!h) return fail(DCIH_EINVAL, "dcih_get_index: null handle");
    if (h->n <= 0) return fail(DCIH_ESTATE, "dcih_get_index: index is empty");
    DeviceGuard guard(h->device);
    const size_t cells = (size_t)num_indices(h) * h->n;
    DCIH_HIP(hipDeviceSynchronize());
    if (h_keys) DCIH_HIP(hipMemcpy(h_keys, h->d_skeys, cells * sizeof(float), hipMemcpyDeviceToHost));
    if (h_ids) DCIH_HIP(hipMemcpy(h_ids, h->d_sids, cells * sizeof(int32_t), hipMemcpyDeviceToHost));
    return DCIH_OK;
}

int64_t dcih_num_points(const dcih_index* h) { return h ? h->n : 0; }

int dcih_clear(dcih_index* h) {
    if (!h) return fail(DCIH_EINVAL, "dcih_clear: null handle");
    DeviceGuard guard(h->device);
    // Borrowed rows are the caller's again when this returns, so nothing may be reading them.  Rows the index
    // owns stay with it: what comes next is put behind the calls that read them, unless they are in a graph.
    if (h->recorded || h->d_data != h->d_own) {
        DCIH_HIP(hipDeviceSynchronize());
        h->busy_set = h->recorded = false;
    }
    return release_index(h);
}

int dcih_reset(dcih_index* h) {
    int rc = dcih_clear(h);
    if (rc) return rc;
    DeviceGuard guard(h->device);
    rc = wait_for_readers(h);
    return rc ? rc : draw_directions(h);
}

int dcih_free(dcih_index* h) {
    if (!h) return DCIH_OK;
    DeviceGuard guard(h->device);
    (void)hipDeviceSynchronize();
    (void)release_index(h);
    release_rows(h);
    release_rows8(h);
    if (h->d_point_rows) (void)hipFree(h->d_point_rows);
    (void)release_arena(h);
    if (h->ws) (void)hipFree(h->ws);
    if (h->d_dirs) (void)hipFree(h->d_dirs);
    for (auto& e : h->ev) if (e) (void)hipEventDestroy(e);
    if (h->busy) (void)hipEventDestroy(h->busy);
    if (h->rows8_event) (void)hipEventDestroy(h->rows8_event);
    if (h->words) (void)hipHostFree((void*)h->words);
    delete h;
    return DCIH_OK;
}

int dcih_project(const float* d_dirs, int num_idx, const float* d_rows, int64_t num_rows,
                 int dim, float* d_out, void* stream) {
    if (!d_dirs || !d_rows || !d_out || num_idx <= 0 || num_rows < 0 || dim <= 0)
        return fail(DCIH_EINVAL, "dcih_project: bad argument");
    return project(d_dirs, num_idx, d_rows, num_rows, dim, d_out, num_rows, (hipStream_t)stream);
}

int dcih_segsort(const float* d_keys, int num_idx, int64_t num_points, int block_size,
                 float* d_skeys, int32_t* d_sids, void* stream) {
    if (!d_keys || !d_skeys || !d_sids || num_idx <= 0 || num_points <= 0 || block_size <= 0)
        return fail(DCIH_EINVAL, "dcih_segsort: bad argument");
    hipStream_t s = (hipStream_t)stream;
    const size_t tmp_bytes = segsort_tmp_bytes(num_idx, num_points, block_size);
    void* d_tmp = nullptr;
    if (tmp_bytes) DCIH_HIP(hipMalloc(&d_tmp, tmp_bytes));
    const int rc = segsort(d_keys, num_points, num_idx, num_points, block_size, d_skeys, d_sids, nullptr, nullptr, d_tmp, s);
    if (d_tmp) {
        (void)hipStreamSynchronize(s);
        (void)hipFree(d_tmp);
    }
    return rc;
}

}  // extern "C"
