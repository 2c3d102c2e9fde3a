// Resident forward simulation: ONE cooperative launch for the whole run.
//
// Workgroup g owns elements [g*span, (g+1)*span): their state and propagators
// live in registers, their slice of the delay ring in LDS, from the first step
// to the last.  Per step a workgroup
//   1. folds the arrivals of slot t-1 (LDS) into y1 and runs the GLIF3 update
//      from registers, then publishes its wavefronts' spike ballots;
//   2. pulls the spikes of step t-1: it scans the ballots every workgroup
//      published before the previous barrier and, for each neuron that fired,
//      reads ITS OWN segment of that neuron's synapse row (rows are sorted by
//      target; a per-row offset table gives the segment bounds) and adds the
//      weights into its LDS ring slice with LDS atomics; external input events
//      of step t-1 are pulled the same way;
//   3. on the way, once every wavefront's ballot store of step t has been
//      acknowledged (an explicit wait on the vector memory counter, taken
//      together with the pull's first loads), signals the grid barrier of
//      step t, which then fills while the pull runs;
//   4. waits for the barrier where the spikes behind it are needed.
// Nothing but spike ballots, segment offsets and the synapses actually used
// crosses the memory system: no global atomics, no state traffic.
//
// That is the form for runs with slack (below), and without where the caller does
// not ask for lists.  Without slack the workgroups exchange lists of fired neurons
// and meet at no grid barrier: sim_resident_lists_kernel, further down.
//
// Ballots live in a history of D rows, row t%D for step t.  With D = 3 a
// workgroup waits for the barrier of step t at the end of step t: row t%3 is
// read in step t+1 and next overwritten in step t+3, which a workgroup can only
// reach after the barrier of step t+2, i.e. after every workgroup finished
// reading it.  With a fourth row the wait moves to where the barrier is needed,
// just before the pull in step t+1: the update of step t+1 needs no spike newer
// than step t-1 (delays are at least one step, and arrivals enter y1 a step
// late), so it runs while the barrier of step t fills, and the wait is
// normally over before it begins.  A workgroup writing row t%4 is then at most
// two steps ahead of one still reading row (t-3)%4.
//
// With a delay offset B (tables hold delays shortened by B steps) step t pulls
// the spikes of step t-1-B from a history of D rows, and a workgroup only has
// to know that everybody has published step t-B before it starts step t+1: it
// waits for the barrier of S = min(B, D-3-B, 31) steps ago, so workgroups drift
// up to S steps apart and the wait is normally over before it begins.  Because
// of the drift one running count cannot tell who has arrived where: there is a
// counter per step, 64 of them used in turn (the fastest workgroup is at most
// 2S+1 < 64 steps ahead of a waiting one), each compared with the number of
// workgroups times the number of rounds it has served.  Row t%D is
// overwritten in step t+D; by then its writer has seen every workgroup arrive
// at the barrier of step t+D-1-S, hence finish the pull of step t+D-2-S, which
// read the spikes of step t+D-3-S-B >= t.
//
// Every wait is bounded: a workgroup that spins too long on the barrier raises
// the abort word, every other workgroup sees it and all leave the loop, so the
// grid always drains.
#include <stdlib.h>

#include "fired_lists.hpp"
#include "glif3_update.hpp"
#include "sim_internal.hpp"

namespace bmtk {

constexpr int kResBlock = 1024;
constexpr unsigned kMaxSpin = 4000000u;  // polls of the barrier word before giving up (seconds)
constexpr int kBarrierWords = 64;        // per-step arrival counters, used round-robin
// Words between two counters.  The arrivals of one step are a burst of one atomic per workgroup on one address,
// which the memory side works off one after the other (a few microseconds for 248 of them); a look at the
// counter of the step before must not queue up behind that burst, so every counter lives in a memory channel
// of its own rather than side by side in one cache line.
constexpr int kBarrierStride = BMTK_RES_SYNC_STRIDE;
// For the same reason a step's arrivals are spread over kWays counters (the workgroups of one XCD share one) and
// a look adds them up: the burst on one address is then an eighth as long, and so is the time the barrier takes
// to fill.  Counter (slot i, way x) is word (x * kBarrierWords + i) * kBarrierStride of the counter area.
constexpr int kWays = BMTK_RES_SYNC_WAYS;
constexpr int kWayStride = kBarrierWords * kBarrierStride;
static_assert(BMTK_RES_SYNC_WORDS >= (1 + kWays * kBarrierWords) * kBarrierStride, "res_sync too small");
constexpr int kMaxSlack = 31;

#ifdef BMTK_RES_PROFILE
__device__ unsigned long long g_prof[8];
__device__ unsigned long long g_prof_blk[256][4];  // per workgroup: update, pull, wait, segment pull
#define PROF_BLK(i, a, b) if (threadIdx.x == 0) atomicAdd(&g_prof_blk[blockIdx.x & 255][i], (unsigned long long)((b) - (a)))
#define PROF_T(var) const long long var = wall_clock64()
#define PROF_ADD(i, a, b) if (threadIdx.x == 0 && blockIdx.x == 0) atomicAdd(&g_prof[i], (unsigned long long)((b) - (a)))
#else
#define PROF_T(var)
#define PROF_ADD(i, a, b)
#define PROF_BLK(i, a, b)
#endif

struct Resident {
    int64_t step0, n_steps;
    int span, n_groups;
    int offset, hist, slack;  // B, D, S of the note above
    int check;                // the arrival counters are looked at every `check` steps (1 when S = 0)
    int row_cap;              // lists: rows of a step that there is room for
};

__device__ __forceinline__ unsigned load_agent(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wait until every vector memory operation this wavefront has issued is complete: its loads have returned and
// its stores -- the write-through, device-coherent ballot store among them -- have been acknowledged.  A release
// fence of workgroup scope does NOT do this: on this target it waits for LDS and scalar operations only, because
// the wavefronts of a workgroup share one vector cache.
//
// THE GRID BARRIER'S CONTRACT.  Three kinds of words in device memory are written by one workgroup and read by
// others during a launch; every such access is a relaxed atomic of AGENT scope (it passes the compute unit's
// vector cache and the XCD's L2 and is served where all XCDs see the same value), and the order between them is
// made by hand, because HIP's memory model offers no fence of the needed kind that does not also invalidate the
// XCD's L2 every step:
//   work_bits   (ballots)   written by: lane 0 of every wavefront that owns elements, right after its update of
//                           step t (row t % hist).  Read by: every workgroup's pull of step t, after it has seen
//                           the barrier of step t complete.
//   arrival counters        written by: thread 0 of a workgroup, one increment per step, on the counter of (step,
//                           the workgroup's XCD), AFTER every wavefront of the workgroup has executed
//                           wait_vector_memory() and the workgroup has passed __syncthreads().  Read by: one look
//                           per workgroup and step (the eight counters of the step added up), repeated within a
//                           bounded spin.
//   abort word              written by: any workgroup whose spin ran out.  Read by: every workgroup inside its spin
//                           and at the start of a launch.  Sticky: only the host clears it.
// The one ordering that makes the barrier a barrier: a workgroup's ballot stores of step t are
// ACKNOWLEDGED (wait_vector_memory in every wavefront that stored, then the workgroup barrier) before its arrival
// for step t is sent.  A reader that has counted all arrivals of step t therefore loads ballots that
// are already where agent-scope loads look.  Nothing else is assumed: readers do not rely on the order of two
// stores of another workgroup, and no acquire fence runs inside the loop (every read of another workgroup's words
// is an agent-scope load, which is not served from a copy that an earlier read left in the compute unit's cache).
// If the wait before the arrival were lost (a compiler that moved or dropped the asm, a fence mistaken for it),
// a reader could see the arrival before a ballot word and miss a spike of that step: the tests that run many
// workgroups for many steps against a driver without this barrier would differ in single synaptic segments --
// tests/test_gpu_simulate.py::test_v1_scale_resident_equals_per_step_launches and
// ::test_lists_of_fired_neurons_equal_the_ballots, tests/test_gpu_random_networks.py::
// test_many_workgroups_with_volleys_and_delay_offsets.
// (The lists of sim_resident_lists_kernel need none of this: every word of theirs carries its step.)
__device__ __forceinline__ void wait_vector_memory()
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// add the weights of one row's synapses that target this workgroup's group,
// positions [seg_row[g], seg_row[g+1]) of the packed table, to the LDS ring
// slice.  Every lane of a wavefront reads a different cache line here, and the
// address unit serialises such requests, so the number of requests is what
// costs: the two bounds come in one 8-byte load, and only lanes that really
// have a k-th synapse issue the k-th load (a segment holds 1.2 on average).
struct __attribute__((packed, aligned(4))) SegBounds {
    uint32_t lo, hi;
};

struct RingSlice {
    float *origin;     // the slice's origin less e0
    unsigned span_v;   // in a vector register once, not before every multiply
    unsigned q_lo, q_wrap;

    // additions to the slots behind slot0
    __device__ __forceinline__ RingSlice(float *ring_l, int span, int e0, int L, int slot0)
        : origin(ring_l - e0), q_lo((unsigned)slot0 * 4u), q_wrap((unsigned)slot0 * 4u - 4u * (unsigned)L)
    {
        asm("v_mov_b32 %0, %1" : "=v"(span_v) : "s"(span));
    }
    // An LDS float atomic costs about three clocks per LANE on gfx950 (its lanes are worked off one after the
    // other), an integer compare-and-swap a few clocks per INSTRUCTION.  Where most lanes of a wavefront take
    // part -- the first synapse of the segments -- the addition is therefore a compare-and-swap loop (a
    // lane repeats only if another thread changed its cell in between, which is rare among 23,000 cells); the
    // thinly populated later ones keep the float atomic.  The sum is the same either way.
    // ring cell of a synapse: the record's upper byte is delay*4 + receptor, so (slot0 + delay) % L * 4 + receptor
    // = min(u, u - 4L) with u = slot0*4 + that byte (unsigned), times the span, plus the target's place in it.
    // Instruction issue is what the pull is short of (every lane walks its own segment, so each addition is a
    // wavefront instruction for a handful of lanes): the cell's address takes six instructions -- two byte adds, min,
    // mask, one 24-bit multiply-add, one shift-add onto the slice's origin less e0 -- and a synapse's load a compare
    // against the segment's length and an immediate offset.
    __device__ __forceinline__ void add(const uint2 sy, bool crowded) const
    {
        const unsigned dq = sy.x >> 24;
        const unsigned plane = min(dq + q_lo, dq + q_wrap);
        float *cell = origin + mad_u24(plane, span_v, sy.x & 0xFFFFFFu);
        const float w = __uint_as_float(sy.y);
        if (!crowded) {
            atomicAdd(cell, w);
            return;
        }
        unsigned *bits = reinterpret_cast<unsigned *>(cell);
        unsigned old = *bits;  // only seeds the loop: a stale value costs one more round
        while (true) {
            const unsigned seen = atomicCAS(bits, old, __float_as_uint(__uint_as_float(old) + w));
            if (seen == old) break;
            old = seen;
        }
    }
};

__device__ __forceinline__ void pull_bounds(uint32_t lo, uint32_t len, uint32_t part, uint32_t team,
                                            const bmtk_synapse *__restrict__ tab, const RingSlice &ring)
{
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(tab) + lo;
    // all of a segment's loads go out together: a loop of dependent loads for the few long segments would
    // hold up the whole wavefront (1 in 25 segments has more than 3 synapses, 1 in 5000 more than 6); measured at V1
    // scale: four together and the compare-and-swap for the first only, 5.35 us per step; six and two, 5.43
    constexpr int kTogether = 4;
    for (uint32_t q = part; q < len; q += kTogether * team) {
        uint2 sy[kTogether];
#pragma unroll
        for (int u = 0; u < kTogether; ++u)
            if (q + u * team < len) sy[u] = rows[q + u * team];
#pragma unroll
        for (int u = 0; u < kTogether; ++u)
            if (q + u * team < len) ring.add(sy[u], u < 1);
    }
}

__device__ __forceinline__ void pull_segment(const uint32_t *__restrict__ seg_row, int g,
                                             const bmtk_synapse *__restrict__ tab, float *ring_l, int span, int e0,
                                             int L, int slot0)
{
    const SegBounds sb = *reinterpret_cast<const SegBounds *>(seg_row + g);
    pull_bounds(sb.lo, sb.hi - sb.lo, 0u, 1u, tab, RingSlice(ring_l, span, e0, L, slot0));  // the offsets never decrease
}

constexpr int kScanWords = 4;   // ballot words per thread and round
constexpr unsigned kInputTag = 0x80000000u;

// Spikes and input events of one step, read from row `hist_row` of the ballot
// history and handed over as if emitted in the step whose ring slot is `slot0`
// (the step they were emitted in plus the delay offset) -> this workgroup's
// ring slice.
// Pass by pass: every thread reads kScanWords ballot words and one input
// event (independent loads), a workgroup-wide prefix sum packs the rows that
// fired into one LDS list, then one thread per listed row pulls this
// workgroup's segment of it.  Must be called by all threads of the workgroup.
// `arrival`, when not null, is the grid barrier counter this workgroup still has to bump for the step whose
// ballots its wavefronts have just stored: the bump may only happen once every one of those stores has been
// acknowledged, and the cheapest place to wait for that is where each wavefront waits for its scan loads anyway.
// Returns true when the bump has been made.
// kUnified: the input rows follow the recurrent rows in ONE table (inp_seg = rec_seg + n_neurons*(n_groups+1), both
// sets of offsets index rec_packed), so a listed row needs no choice between two tables.
template <bool kUnified>
__device__ __forceinline__ bool pull_step(const bmtk_glif3_sim &s, const Resident &r, int g, int hist_row, int slot0,
                                          float *ring_l, unsigned *act, unsigned *scan_l, int e0, int words,
                                          int64_t k0, int64_t k1, unsigned *arrival = nullptr)
{
    const int tid = threadIdx.x;
    const int L = s.ring_slots;
    const int wave = tid / kWave;
    const bool has_rec = s.rec_seg != nullptr;
    // one thread per listed row pulls this workgroup's segment of it
    auto pull_listed = [&](unsigned total) {
        for (unsigned a = tid; a < total; a += kResBlock) {
            // one code path for both kinds of rows: a wavefront nearly always holds some of each, and a
            // branch would make it walk the two chains of dependent loads one after the other
            const unsigned entry = act[a];
            if (kUnified) {  // rows * (n_groups + 1) stays below 2^32 (checked before the launch)
                pull_segment(s.rec_seg + mul_u24(entry, (unsigned)(r.n_groups + 1)), g, s.rec_packed, ring_l, r.span,
                             e0, L, slot0);
            } else {
                const int64_t row = entry & ~kInputTag;
                const bool is_input = (entry & kInputTag) != 0u;
                const uint32_t *seg = is_input ? s.inp_seg : s.rec_seg;
                const bmtk_synapse *tab = is_input ? s.inp_packed : s.rec_packed;
                pull_segment(seg + row * (r.n_groups + 1), g, tab, ring_l, r.span, e0, L, slot0);
            }
        }
    };
    const unsigned long long *bits =
        reinterpret_cast<const unsigned long long *>(s.work_bits) + (int64_t)hist_row * (words + 1);
    // 32-bit counters wherever the sizes allow: the loop is short of scalar registers
    const int n_words = has_rec ? words : 0;
    const int word_rounds = (n_words + kScanWords * kResBlock - 1) / (kScanWords * kResBlock);
    const int event_rounds = (int)((k1 - k0 + kResBlock - 1) / kResBlock);  // a step's events are below 2^31
    const int rounds = word_rounds > event_rounds ? word_rounds : event_rounds;
    for (int round = 0; round < rounds; ++round) {
        const int w0 = round * kScanWords * kResBlock;
        PROF_T(p0);
        unsigned long long v[kScanWords];
        unsigned cnt = 0;
        // words past the end are read from the row's last word, which nothing ever writes (it stays zero):
        // no branch round the loads
        if (has_rec) {
#pragma unroll
            for (int u = 0; u < kScanWords; ++u) {
                const unsigned w = min((unsigned)w0 + (unsigned)(u * kResBlock + tid), (unsigned)words);
                v[u] = __hip_atomic_load(bits + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else {
#pragma unroll
            for (int u = 0; u < kScanWords; ++u) v[u] = 0ull;
        }
        const int64_t ke = k0 + (round * kResBlock + tid);
        const bool has_event = ke < k1;
        const unsigned event_row = has_event ? (unsigned)s.in_events[ke] : 0u;
#pragma unroll
        for (int u = 0; u < kScanWords; ++u) cnt += (unsigned)__popcll(v[u]);
        cnt += has_event ? 1u : 0u;
        const unsigned inc = wave_inclusive_scan(cnt);
        if (lane_id() == kWave - 1) scan_l[wave] = inc;
        if (arrival && round == 0) wait_vector_memory();  // the loads are back already; this is for the ballot store
        __syncthreads();
        if (arrival && round == 0 && tid == 0)
            __hip_atomic_fetch_add(arrival, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        PROF_T(p1);
        // prefix over the 16 wavefront sums: one LDS read per lane and one more scan instead of 16 reads
        const unsigned part = wave_inclusive_scan(lane_id() < kResBlock / kWave ? scan_l[lane_id()] : 0u);
        const unsigned total = (unsigned)bcast_i((int)part, kResBlock / kWave - 1);
        const unsigned base = wave > 0 ? (unsigned)__shfl((int)part, wave - 1, kWave) : 0u;
        const bool listed = total <= (unsigned)kActCap;  // workgroup-uniform
        if (listed) {
            unsigned pos = base + inc - cnt;
#pragma unroll
            for (int u = 0; u < kScanWords; ++u) {
                unsigned long long x = v[u];
                const unsigned j0 = (unsigned)(w0 + u * kResBlock + tid) << 6;
                while (x) {
                    const int bit = __ffsll((long long)x) - 1;
                    x &= x - 1ull;
                    act[pos++] = j0 + (unsigned)bit;
                }
            }
            if (has_event) act[pos] = kUnified ? event_row + (unsigned)s.n_neurons : event_row | kInputTag;
        } else {
            // more rows than the list holds: every thread pulls what it found itself, unbalanced but correct
            for (int u = 0; u < kScanWords; ++u) {
                unsigned long long x = v[u];
                const int64_t j0 = (int64_t)(w0 + u * kResBlock + tid) << 6;
                while (x) {
                    const int bit = __ffsll((long long)x) - 1;
                    x &= x - 1ull;
                    pull_segment(s.rec_seg + (j0 + bit) * (r.n_groups + 1), g, s.rec_packed, ring_l, r.span, e0, L,
                                 slot0);
                }
            }
            if (has_event) {
                if (kUnified)
                    pull_segment(s.rec_seg + (s.n_neurons + (int64_t)event_row) * (r.n_groups + 1), g, s.rec_packed, ring_l,
                                 r.span, e0, L, slot0);
                else
                    pull_segment(s.inp_seg + (int64_t)event_row * (r.n_groups + 1), g, s.inp_packed, ring_l, r.span, e0,
                                 L, slot0);
            }
        }
        __syncthreads();
        PROF_T(p2);
        if (listed) pull_listed(total);
        __syncthreads();
        PROF_T(p3);
        PROF_ADD(4, p0, p1);
        PROF_ADD(5, p1, p2);
        PROF_ADD(6, p2, p3);
        PROF_BLK(3, p2, p3);
    }
    return arrival != nullptr && rounds > 0;
}

// kLate: the run has slack (S > 0), see the loop body.  kForm: what the launch asks for beyond the simulation
// itself.  The loop is short of scalar registers (98 spilled in the general form; every use in the loop is a lane
// read), so the pointers and counters a launch does not use are taken out of it at compile time:
//   kFormLean    spike bits only, and the two tables are one (pull_step);
//   kFormRecord  the same with the spike record (what the PyNEST-shaped front end and the configuration runner
//                ask for), no membrane potential probes;
//   kFormAny     everything: probes, record, two tables.
enum { kFormAny = 0, kFormRecord = 1, kFormLean = 2 };
template <bool kLate, int kForm>
__global__ __launch_bounds__(kResBlock) void sim_resident_kernel(bmtk_glif3_sim s, Resident r)
{
    constexpr bool kUnifiedTables = kForm != kFormAny;
    if (kForm != kFormAny) {
        s.probe_col = nullptr;
        s.inp_seg = nullptr;
        s.inp_packed = nullptr;
    }
    if (kForm == kFormLean) s.spike_count = nullptr;
    extern __shared__ float ring_l[];  // [L*4][span], then the active-row list
    __shared__ int go_on;
    __shared__ unsigned scan_l[kResBlock / kWave];
    __shared__ unsigned fired_n[2];  // how many fired in this step and the one before
    const int tid = threadIdx.x;
    const int lane = lane_id();
    // Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD
    // b % 8).  Give each XCD a run of consecutive groups so that the segments
    // of a synapse row its workgroups read -- and their offsets -- are
    // contiguous and are fetched into that XCD's L2 once.
    const int per_xcd = (int)gridDim.x >> 3;
    const int g = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    const int ne = (int)s.n_neurons;  // batch 1, at most 1024 elements per compute unit
    const int words = (ne + 63) >> 6;
    const int L = s.ring_slots;
    const int span = r.span;
    const int e0 = g * span;
    const int mine = max(0, min(span, ne - e0));  // groups past the end own nothing
    const bool own = tid < mine;
    const int e = e0 + tid;
    unsigned *act = reinterpret_cast<unsigned *>(ring_l + s.ring_slots * GLIF3_NREC * r.span);
    unsigned *abort_word = s.res_sync + 1;
    unsigned *arrivals = s.res_sync + kBarrierStride;  // [kBarrierWords] counters, kBarrierStride words apart
    // a run before this one gave up and nobody has looked yet: do nothing, so that the failure is still there to see
    // (one thread looks for the whole workgroup, so that all of its threads take the same way)
    if (tid == 0) {
        go_on = load_agent(abort_word) == 0u;
        fired_n[0] = fired_n[1] = 0u;
    }
    __syncthreads();
    if (!go_on) return;
    __syncthreads();  // go_on is written again in the loop

    for (int c = tid; c < L * GLIF3_NREC * span; c += kResBlock) {
        const int dr = c / span, i = c - dr * span;
        ring_l[c] = i < mine ? s.ring[(int64_t)dr * ne + e0 + i] : 0.0f;
    }
    Glif3Elem st{};
    Glif3Prop p{};
    float I = 0.0f;
    if (own) {
        const int64_t col = s.class_id ? (int64_t)s.class_id[e] : e;
        p.load(s.prop, s.prop_stride, col);
        glif3_load(st, s.V, s.asc, s.y1, s.y2, s.ref, ne, e);
        I = s.i_ext ? s.i_ext[e] : 0.0f;
    }
    __syncthreads();

    // membrane potential probes: this thread's column, and where in the sampling period the call begins
    const int probe_col = (own && s.probe_col) ? s.probe_col[e] : -1;
    int probe_phase = s.probe_col ? (int)((r.step0 + 1) % s.probe_every) : 1;  // 0: sample after this step
    int64_t probe_row = 0;
    const float zero[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f};
    bool aborted = false;
    int done = 0;  // steps whose update has run
    // the spike record may be split into several lists, one per group of workgroups
    const unsigned rec_ways = s.spike_ways > 1 ? (unsigned)s.spike_ways : 1u;
    const unsigned long long rec_way = blockIdx.x & (rec_ways - 1u), rec_cap = (unsigned long long)s.spike_cap / rec_ways;
    // With as many lists as workgroups this one appends to its list alone: its count lives in a register of every
    // thread (first loaded, written back at the end), a spike's place is that count plus the spike's rank among the
    // workgroup's spikes of the step (an LDS atomic), and no wavefront
    // waits for an atomic on device memory, which the arrivals of a step would queue up behind.
    const bool own_record = !kLate && s.spike_count != nullptr && rec_ways >= gridDim.x;
    unsigned long long rec_count = own_record ? s.spike_count[rec_way * BMTK_RECORD_COUNT_STRIDE] : 0ull;
    // the input events of the step pulled in step t, u = t-1-B, are in_events[ka, kb); the bound for the
    // next step is fetched a step ahead.  Steps before 0 have no events (in_ptr[0] = 0).
    const int B = r.offset;
    auto in_bound = [&](int64_t i) -> int64_t { return (s.in_ptr && i > 0) ? s.in_ptr[i] : 0; };
    int opaque_zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(opaque_zero));
    int64_t ka = 0, kb = in_bound(r.step0 - B);
#ifdef BMTK_RES_PROFILE
    long long prof_prev = 0, prof_c1 = 0;
#endif
    // Wait until every workgroup has arrived at the barrier of step j of this call (all threads call it;
    // false = the run was given up).  No acquire fence: it would invalidate this XCD's L2 every step, and
    // the only data other workgroups write during the run are the ballots, which are read with agent-scope
    // loads that bypass the non-coherent caches.
    auto counter_of = [&](int j) { return arrivals + ((j < 0 ? 0 : j) & (kBarrierWords - 1)) * kBarrierStride; };
    auto poll = [&](int j) -> int {  // one thread: 1 = everybody arrived at step j, 0 = given up
        const unsigned *word = counter_of(j);
        const unsigned target = j < 0 ? 0u : gridDim.x * (unsigned)(j / kBarrierWords + 1);
        unsigned spins = 0;
        auto arrived = [&]() {  // the loads of a look travel together
            unsigned n[kWays];
#pragma unroll
            for (int x = 0; x < kWays; ++x) n[x] = load_agent(word + x * kWayStride);
            unsigned sum = 0;
#pragma unroll
            for (int x = 0; x < kWays; ++x) sum += n[x];
            return sum;
        };
        while (arrived() < target) {
            if (load_agent(abort_word) != 0u) return 0;
            if (++spins > (s.res_spin_limit ? s.res_spin_limit : kMaxSpin)) {
                __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return 0;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        return 1;
    };
    auto wait_for = [&](int j) -> bool {
        if (tid == 0) go_on = poll(j);
        __syncthreads();
        return go_on != 0;
    };
    // Without slack, the pull of step t-1-B (in step t) is all that needs the barrier of step t-1, and the
    // update of step t needs neither: when the history has a row to spare (D >= B + 4) the wait for the barrier
    // of step t-1 moves from the end of step t-1 to just before that pull.  By then every workgroup arrived an
    // update and a pull ago, so the wait is over before it begins.  A workgroup writing row t%D may then be up
    // to two steps ahead of one still reading row (t-3-B)%D, hence the spare row.
    const bool defer = !kLate && r.hist >= B + 4;
    // The look itself is taken by the last wavefront, while the others update: its 64 threads own no elements
    // when the span is 960 or less, and the answer, a memory round trip away, is there when the workgroup meets
    // after the update.
    constexpr int kLooker = kResBlock - kWave;
    // ring slot of step t-1 and history rows of steps t and t-1-B, counted along instead of taking three
    // 64-bit remainders per step (every instruction of the loop costs all 16 wavefronts an issue slot)
    auto wrap = [](int64_t a, int m) { return (int)(((a % m) + m) % m); };
    int next_slot_prev = wrap(r.step0 - 1, L), next_row_t = wrap(r.step0, r.hist),
        next_row_p = wrap(r.step0 - 1 - B, r.hist);
    const int n_steps = (int)r.n_steps;
    for (int k = 0; k < n_steps; ++k) {
        const int64_t t = r.step0 + k;
        const int slot_prev = next_slot_prev, row_t = next_row_t, row_p = next_row_p;
        next_slot_prev = slot_prev + 1 == L ? 0 : slot_prev + 1;
        next_row_t = row_t + 1 == r.hist ? 0 : row_t + 1;
        next_row_p = row_p + 1 == r.hist ? 0 : row_p + 1;
        PROF_T(c0);
#ifdef BMTK_RES_PROFILE
        if (k > 0) PROF_ADD(1, prof_prev, c0);
#endif
        // The bound of the next step's events is asked for now and looked at after the pull.  The address gets a
        // zero the compiler cannot see through: a load it knows to be the same in every lane is moved to a scalar
        // register on the spot, and every wavefront would wait for the answer here, at the top of the step.
        const int64_t in_next = t + 1 - B;
        long long kn_lanes = 0;
        if (s.in_ptr && in_next > 0) kn_lanes = s.in_ptr[in_next + opaque_zero];
        if (defer && k > 0 && tid == kLooker) go_on = poll(k - 1);
        // 1. fold the arrivals of slot t-1 and update
        bool spike = false;
        float frac = 0.0f;
        if (own) {
            if (k > 0) {
                float *prev = ring_l + slot_prev * GLIF3_NREC * span + tid;
#pragma unroll
                for (int q = 0; q < GLIF3_NREC; ++q) {
                    const float a = prev[q * span];
                    prev[q * span] = 0.0f;
                    st.y1[q] = st.y1[q] + a * p.psc0[q];
                }
            }
            spike = glif3_update(st, p, s.h, zero, I, &frac);
        }
        if (s.probe_col) {
            if (probe_phase == 0) {
                if (probe_col >= 0) s.probe_v[probe_row * s.probe_stride + probe_col] = st.V;
                ++probe_row;
            }
            probe_phase = probe_phase + 1 == s.probe_every ? 0 : probe_phase + 1;
        }
        const unsigned long long m = __ballot(spike);
        // only the wavefronts that cover this workgroup's span own a ballot word
        if (lane == 0 && tid < span && (e & ~(kWave - 1)) < ne) {
            __hip_atomic_store(reinterpret_cast<unsigned long long *>(s.work_bits) + (int64_t)row_t * (words + 1) + (e >> 6),
                               m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (s.spike_bits) s.spike_bits[k * s.spike_bits_stride + (e >> 6)] = m;
        }
        // Spike record: a wavefront with spikes takes its places in the list with ONE atomic, whose answer is a
        // memory round trip away.  It is only asked for here and looked at after the pull, so that no wavefront
        // stops for it in the update (which every other wavefront of the workgroup would wait out at the next
        // barrier).
        if (own_record && m != 0ull && spike) {
            const unsigned at = atomicAdd(&fired_n[k & 1], 1u);
            if (rec_count + at < rec_cap) {
                const unsigned long long idx = rec_way * rec_cap + rec_count + at;
                s.spike_step[idx] = (int32_t)t;
                s.spike_elem[idx] = (int32_t)e;
                if (s.spike_frac) s.spike_frac[idx] = frac;
            }
        }
        unsigned long long rec_base = 0ull;
        if (s.spike_count && !own_record && m != 0ull && lane == __ffsll((long long)m) - 1)
            rec_base = atomicAdd(s.spike_count + rec_way * BMTK_RECORD_COUNT_STRIDE, (unsigned long long)__popcll(m));
        done = k + 1;
        // With no slack (S = 0) the arrival is signalled early in the pull so that the barrier fills while
        // the pull runs.  With slack nobody is waiting for this step yet: the arrival moves behind the pull,
        // which saves a workgroup barrier, and the counters are only looked at every `check` steps.
        constexpr bool late = kLate;
        const int check = late ? r.check : 1;
        unsigned *const my_counter = counter_of(k) + (blockIdx.x & (kWays - 1)) * kWayStride;
        if (!late) {
            // the workgroup meets, so that the looker's answer can be read
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __syncthreads();
            PROF_T(c1);
            PROF_ADD(0, c0, c1);
            PROF_BLK(0, c0, c1);
#ifdef BMTK_RES_PROFILE
            prof_c1 = c1;
#endif
            if (defer && k > 0 && !go_on) {  // written before the workgroup met above
                aborted = true;
                break;
            }
            // the number of this step, complete since the workgroup met; the other one, last read a barrier ago and next added
            // to a barrier on, back to zero
            if (own_record) rec_count += fired_n[k & 1];
            if (own_record && tid == 0) fired_n[(k + 1) & 1] = 0u;
        }
        PROF_T(c2);
#ifdef BMTK_RES_PROFILE
        if (!kLate) PROF_ADD(7, prof_c1, c2);
#endif
        // 2. + 3. pull the spikes and input events of step t-1-B (the first step of a call pulls nothing: the
        //    call before it closed with that pull) and, without slack, arrive at the barrier of step t on the
        //    way, so that the barrier fills while the pull runs.  The arrival tells the other workgroups that
        //    this one's ballots of step t can be read: it must not move before every wavefront's ballot store
        //    (a write-through, device-coherent store) has been acknowledged, which each wavefront waits for
        //    together with the first loads of the pull.  No L2 write-back is needed: nothing else written
        //    inside the loop is read by another workgroup before the kernel ends.
        bool arrived = false;
        if (k > 0 && t - 1 - B >= 0 && mine > 0)
            arrived = pull_step<kUnifiedTables>(s, r, g, row_p, slot_prev, ring_l, act, scan_l, e0, words, ka, kb,
                                               late ? nullptr : my_counter);
        if (!late && !arrived) {
            wait_vector_memory();
            __syncthreads();
            if (tid == 0) __hip_atomic_fetch_add(my_counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        ka = kb;
        kb = ((int64_t)__builtin_amdgcn_readfirstlane((int)(kn_lanes >> 32)) << 32) |
             (int64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)kn_lanes);
        if (s.spike_count && !own_record && m != 0ull) {  // the places asked for above: the answer has long arrived
            unsigned long long idx = bcast_u64(rec_base, __ffsll((long long)m) - 1) + (unsigned long long)lane_prefix(m);
            if (spike && idx < rec_cap) {
                idx += rec_way * rec_cap;  // this workgroup's list
                s.spike_step[idx] = (int32_t)t;
                s.spike_elem[idx] = (int32_t)e;
                if (s.spike_frac) s.spike_frac[idx] = frac;
            }
        }
        if (late) {
            // every wavefront's ballot store has been acknowledged before the workgroup meets and arrives
            wait_vector_memory();
            __syncthreads();
        }
        // (without slack no workgroup barrier is needed here: pull_step ends with one, and the word thread 0
        //  writes below was last read before the barrier that precedes the arrival)
        PROF_T(c3);
        if (late && tid == 0) __hip_atomic_fetch_add(my_counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // 4. every `check` steps (each step without slack) wait until every workgroup has published
        //    step k - S + (check - 1): enough for the steps up to the next look
        if (late && k % check != check - 1 && k + 1 < n_steps) continue;
        bool ok = true;
        if (!defer) {
            int j = late ? k - r.slack + (check - 1) : k;  // step of this call everybody must have published
            ok = wait_for(j < k ? j : k);
        }
        PROF_T(c4);
        PROF_ADD(2, c2, c3);
        PROF_ADD(3, c3, c4);
        PROF_BLK(1, c2, c3);
        PROF_BLK(2, c3, c4);
#ifdef BMTK_RES_PROFILE
        prof_prev = c4;
#endif
        if (!ok) {
            aborted = true;
            break;
        }
    }
    // with the deferred wait the closing pull is the first to need the barrier of the last step
    if (defer && !aborted && done > 0 && !wait_for(done - 1)) aborted = true;

    if (!aborted && done > 0) {
        // closing: spikes and inputs of the last step (less the delay offset), then fold the last slot
        const int64_t tl = r.step0 + done - 1;
        if (tl - B >= 0 && mine > 0)
            pull_step<kUnifiedTables>(s, r, g, wrap(tl - B, r.hist), wrap(tl, L), ring_l, act, scan_l, e0, words, ka,
                                              kb);
        __syncthreads();
        if (own) {
            float *prev = ring_l + (int)(tl % L) * GLIF3_NREC * span + tid;
#pragma unroll
            for (int q = 0; q < GLIF3_NREC; ++q) {
                const float a = prev[q * span];
                prev[q * span] = 0.0f;
                st.y1[q] = st.y1[q] + a * p.psc0[q];
            }
        }
        __syncthreads();
    }
    if (own) glif3_store(st, s.V, s.asc, s.y1, s.y2, s.ref, ne, e);
    if (own_record && tid == 0) s.spike_count[rec_way * BMTK_RECORD_COUNT_STRIDE] = rec_count;
    for (int c = tid; c < L * GLIF3_NREC * span; c += kResBlock) {
        const int dr = c / span, i = c - dr * span;
        if (i < mine) s.ring[(int64_t)dr * ne + e0 + i] = ring_l[c];
    }
}

// The form without slack (delay offset 0), several workgroups.  What sets its pace is a chain through memory: a spike of
// step t has to be in every workgroup's ring slice before the update of step t+2.  Here little but that chain is left of
// the exchange.  The neurons that fired travel in lists that carry their step (fired_lists.hpp): no acknowledgement, no
// arrival, no barrier over the grid.  And the wavefronts divide the memory traffic, because a wavefront's accesses complete
// in the order issued (one that waits for a load waits for its stores before it, and a store is acknowledged after a trip
// to the far side of the L2):
//   reader (the last)       asks for the lists of step t until every workgroup's are there and puts the rows that fired, and
//                           those of the step's input events, into one list in LDS.  Stores nothing.
//   writer (last but one)   stores what the workgroup leaves in LDS: its list first, ballots, the spike record.  Pulls
//                           nothing.
//   the others              pull: a thread takes a row, reads the bounds of this workgroup's segment of it and adds the
//                           segment's synapses to the ring slice.
// All but the reader (the reader too at spans above 960) own neurons and update them.  A round k of the loop:
//     fold slot k-1, update; who fired -> LDS; writer: list of step k   (reader: lists of step k-1 -> rows)
//   --------------------------------- the workgroup meets --------------------------------------------------
//     pull step k-1                                                     (reader: on to the lists of step k)
//   ------------------ all but the reader wait for one another's pulls (a count in LDS) --------------------
// A workgroup that publishes step t has seen everybody's step t-2, so four rows of lists are enough.
//
// The reader waits half a thousand clocks before its first look: lists looked at while they are being written cost the
// writers' stores, and the pulls, more than the look brings (120,000 neurons: 4.2 us per step looking at once, 3.9 so).
// A look then finds all lists there nearly always.
//
// A row's segment is read by a team of neighbouring lanes, as many as a segment holds synapses on average, rounded up, if
// the step has threads for it (a small network has few rows a step and long segments).
//
// Steps in which more than 39 neurons of a workgroup fire, or whose rows have no room, are crowded: all sixteen wavefronts read the
// lists (or ballots) and work the rows off.  A network's usual few Hz are far below that; us per step, ballots behind a grid barrier /
// the reader taking lists of up to 19 neurons and 3,808 rows / of 39 and all that LDS holds: 60,000 neurons at 35, 45, 56, 71, 92 Hz
// 8.9 / 8.5 / 7.9, 10.3 / 12.2 / 9.3, 12.1 / 14.5 / 10.8, 14.2 / 17.1 / 13.0, 17.4 / 20.7 / 17.5; 230,924 neurons at 24, 35, 46, 60 Hz
// 17.3 / 19.4 / 18.4, 23.1 / 33.8 / 29.0, 38.4 / 41.7 / 36.5, 47.0 / 52.1 / 45.4 (crowded from 25 Hz on).
//
// Measured per step, ballots or lists behind a grid barrier -> this: 10,007 neurons of in-degree 600 3.27 -> 2.16 us; 60,000 of
// 660 4.15 -> 2.88; 120,000 of 440 4.63 -> 3.92; the V1 network's 230,924 of 335 5.46 -> 4.96.  What it spends there: update
// 0.5, list out 0.5, pull 2.5 (two dependent trips to memory for 700 rows), and 1.1 until the slowest wavefront has pulled.
// Bounds and first synapses of a segment in one 16-byte cell (a gigabyte): 4.89 us at V1, slower elsewhere, dropped; flags in
// LDS in place of the meeting, so that the list need not be out before the pull begins: 5.4 us, the pulls and the reader
// then share the way to memory; another order of rows for each workgroup of an XCD: no difference.
constexpr int kReader = kResBlock / kWave - 1, kWriter = kReader - 1;
constexpr int kPullThreads = kWriter * kWave;
constexpr int kReaderEvents = 8;    // input events a lane of the reader asks for ahead
// LDS behind the ring slice, `bytes` of it: rows of two steps, a place per lane of the reader for what is none, the neurons of this
// workgroup that fired and, for a record, their crossing fractions.  At least kActCap words (3,808 rows of a step, with a record 3,296),
// and all that the ring slice leaves, up to four times as many: crowded steps cost half as much again.
constexpr int row_cap(size_t bytes, bool record)
{
    return (int)((bytes - 2 * kResBlock - (record ? 4 * kResBlock : 0) - 4 * kWave) / 8);
}

template <int kForm, bool kReaderOwns>
__global__ __launch_bounds__(kResBlock) void sim_resident_lists_kernel(bmtk_glif3_sim s, Resident r)
{
    constexpr bool kUnified = kForm != kFormAny, kRecord = kForm != kFormLean;
    const unsigned row_cap = (unsigned)r.row_cap;
    if (kForm != kFormAny) {
        s.probe_col = nullptr;
        s.inp_seg = nullptr;
        s.inp_packed = nullptr;
    }
    extern __shared__ float ring_l[];  // [L*4][span], then see row_cap
    __shared__ int go_on[2];  // by the round, as rows_l is: a slot is written again only after a meeting behind all reads of it
    __shared__ unsigned rows_l[2], spikes_l[2], team_l[2], crowd_l[3], done_l, updated_l, listed_l;  // rows of a step, of neurons (the others: of inputs), ..
    __shared__ unsigned fired_n[2];                               // how many fired in this step and the one before
    __shared__ unsigned long long ballot_l[kResBlock / kWave];
    const int tid = threadIdx.x, lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int per_xcd = (int)gridDim.x >> 3;  // an XCD gets consecutive groups, see sim_resident_kernel
    const int g = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (g >= r.n_groups) return;  // (the grid is rounded up; nobody waits for these)
    const int ne = (int)s.n_neurons;
    const int words = (ne + 63) >> 6;
    const int L = s.ring_slots, G = r.n_groups;
    const int span = r.span;
    const int e0 = g * span;
    const int mine = min(span, ne - e0);
    const bool own = tid < mine;
    const int e = e0 + tid;
    unsigned *rows = reinterpret_cast<unsigned *>(ring_l + L * GLIF3_NREC * span);  // [2][row_cap], a place per lane behind
    unsigned short *fired_l = reinterpret_cast<unsigned short *>(rows + 2 * row_cap + kWave);
    float *frac_l = reinterpret_cast<float *>(fired_l + kResBlock);
    unsigned *abort_word = s.res_sync + 1;
    unsigned long long *lists = lists_in(s.res_sync);
    unsigned long long *hist = reinterpret_cast<unsigned long long *>(s.work_bits);
    const unsigned spin_limit = s.res_spin_limit ? s.res_spin_limit : kMaxSpin;
    const bool alone = s.rec_seg == nullptr;  // nobody's spikes arrive anywhere
    // a run before this one gave up and nobody has looked yet: do nothing, so that the failure is still there to see
    if (tid == 0) {
        go_on[0] = load_agent(abort_word) == 0u;
        fired_n[0] = fired_n[1] = rows_l[0] = rows_l[1] = spikes_l[0] = spikes_l[1] = team_l[0] = team_l[1] = done_l = updated_l = listed_l = 0u;
    }
    __syncthreads();
    if (!go_on[0]) return;

    for (int c = tid; c < L * GLIF3_NREC * span; c += kResBlock) {
        const int dr = c / span, i = c - dr * span;
        ring_l[c] = i < mine ? s.ring[(int64_t)dr * ne + e0 + i] : 0.0f;
    }
    Glif3Elem st{};
    Glif3Prop p{};
    float I = 0.0f;
    if (own) {
        const int64_t col = s.class_id ? (int64_t)s.class_id[e] : e;
        p.load(s.prop, s.prop_stride, col);
        glif3_load(st, s.V, s.asc, s.y1, s.y2, s.ref, ne, e);
        I = s.i_ext ? s.i_ext[e] : 0.0f;
    }
    __syncthreads();

    const int n_steps = (int)r.n_steps;
    auto wrap = [](int64_t a, int m) { return (int)(((a % m) + m) % m); };
    int slot_prev = wrap(r.step0 - 1, L), row_t = wrap(r.step0, r.hist);  // ring slot of step t-1, history row of step t
    auto next = [](int a, int m) { return a + 1 == m ? 0 : a + 1; };
    auto row_before = [&]() { return row_t == 0 ? r.hist - 1 : row_t - 1; };
    auto events_at = [&](int k) -> int64_t { return s.in_ptr ? s.in_ptr[r.step0 + k] : 0; };
    auto lists_of = [&](int k) { return ListRow{lists + (k & (kListRows - 1)) * kListRowWords, 0, G}; };

    auto fold = [&](int slot) __attribute__((always_inline)) {
        float *prev = ring_l + slot * GLIF3_NREC * span + tid;
#pragma unroll
        for (int q = 0; q < GLIF3_NREC; ++q) {
            const float a = prev[q * span];
            prev[q * span] = 0.0f;
            st.y1[q] = st.y1[q] + a * p.psc0[q];
        }
    };
    const int probe_col = (own && s.probe_col) ? s.probe_col[e] : -1;
    int probe_phase = s.probe_col ? (int)((r.step0 + 1) % s.probe_every) : 1;  // 0: sample after this step
    int64_t probe_row = 0;
    const float zero[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f};
    // fold and update of step step0 + k; what fired stays in LDS
    auto update = [&](int k) __attribute__((always_inline)) {
        bool spike = false;
        float frac = 0.0f;
        if (own) {
            if (k > 0) fold(slot_prev);
            spike = glif3_update(st, p, s.h, zero, I, &frac);
        }
        if (s.probe_col) {
            if (probe_phase == 0) {
                if (probe_col >= 0) s.probe_v[probe_row * s.probe_stride + probe_col] = st.V;
                ++probe_row;
            }
            probe_phase = probe_phase + 1 == s.probe_every ? 0 : probe_phase + 1;
        }
        const unsigned long long m = __ballot(spike);
        if (lane == 0) ballot_l[wave] = m;
        if (m != 0ull && spike) {
            const unsigned at = atomicAdd(&fired_n[k & 1], 1u);  // (at most span)
            fired_l[at] = (unsigned short)tid;
            if (kRecord) frac_l[at] = frac;
        }
    };
    auto row_bounds = [&](unsigned row) __attribute__((always_inline)) -> SegBounds {
        if (kUnified)  // rows * (n_groups + 1) stays below 2^32 (checked before the launch)
            return *reinterpret_cast<const SegBounds *>(s.rec_seg + mul_u24(row, (unsigned)(G + 1)) + g);
        const uint32_t *seg = row & kInputTag ? s.inp_seg : s.rec_seg;
        return *reinterpret_cast<const SegBounds *>(seg + (int64_t)(row & ~kInputTag) * (G + 1) + g);
    };
    auto input_row = [&](int32_t source) { return kUnified ? (unsigned)source + (unsigned)s.n_neurons : (unsigned)source | kInputTag; };
    auto add_bounds = [&](SegBounds b, bool of_input, unsigned part, unsigned team) __attribute__((always_inline)) {
        const bmtk_synapse *tab = !kUnified && of_input ? s.inp_packed : s.rec_packed;
        pull_bounds(b.lo, b.hi - b.lo, part, team, tab, RingSlice(ring_l, span, e0, L, slot_prev));  // the offsets never decrease
    };
    // The rows of step k-1 into the ring slice.  Where they are listed before the update of step k already (`ask` ahead of it),
    // the bounds of a thread's first row are on their way meanwhile.
    // What the reader has no lanes for, input events from the kReaderEvents * kWave-th on, follows the listed rows, straight from the input
    // lists.  (Put into the rows by the reader, 64 at a time, they made it the one all waited for: 60,000 neurons, 800 / 2,000 / 3,600
    // events a step 4.5 / 10.0 / 17.1 us, with ballots 4.0 / 7.5 / 12.9, so 3.7 / 5.6 / 7.6; eight of a lane under way at a time 3.8 / 5.9 / 8.3.)
    unsigned listed = 0u, n_rows = 0u, team = 0u, at_row = 0u, n_more = 0u;
    const int32_t *more_events = nullptr;
    int32_t next_source = 0;
    SegBounds first_row{0u, 0u};
    auto ask = [&](int k) __attribute__((always_inline)) {
        unsigned me = (unsigned)tid;
        asm volatile("" : "+v"(me));
        const int buf = (k - 1) & 1;
        listed = (unsigned)__builtin_amdgcn_readfirstlane((int)rows_l[buf]);
        team = (unsigned)__builtin_amdgcn_readfirstlane((int)team_l[buf]);
        const bool pulls = listed != kCrowded && wave != kWriter;
        n_rows = pulls ? listed & ~kMoreEvents : 0u;
        at_row = me >> team;
        if (at_row < n_rows) first_row = row_bounds(rows[buf * row_cap + at_row]);
        n_more = 0u;
        if (pulls && (listed & kMoreEvents)) {
            const int64_t from = events_at(k - 1) + kReaderEvents * kWave;
            n_more = (unsigned)(events_at(k) - from);
            more_events = s.in_events + from;
            if (at_row >= n_rows && at_row - n_rows < n_more) next_source = more_events[at_row - n_rows];
        }
    };
    auto pull = [&](int k) __attribute__((always_inline)) {
        const int buf = (k - 1) & 1;
        const unsigned part = (unsigned)lane & ((1u << team) - 1u), step = (unsigned)kPullThreads >> team, n_spikes = spikes_l[buf];
        const bool at_hand = at_row >= n_rows;
        while (at_row < n_rows) {
            const SegBounds b = first_row;
            const bool of_input = at_row >= n_spikes;
            at_row += step;
            if (at_row < n_rows) first_row = row_bounds(rows[buf * row_cap + at_row]);
            add_bounds(b, of_input, part, 1u << team);
        }
        if (n_more != 0u) {
            unsigned a = at_row - n_rows;
            if (!at_hand && a < n_more) next_source = more_events[a];
            while (a < n_more) {
                const int32_t source = next_source;
                a += step;
                if (a < n_more) next_source = more_events[a];
                add_bounds(row_bounds(input_row(source)), true, part, 1u << team);
            }
        }
    };
    // A crowded step, by all threads: lists (row `row` of the history), ballots where a list did not suffice, a thread's input event.
    // Further events are left to pull.
    auto pull_crowded = [&](int k) __attribute__((always_inline)) {
        const int64_t lo = events_at(k - 1);
        const unsigned n_ev = (unsigned)(events_at(k) - lo);  // (a step's events are below 2^31)
        const int32_t *const events = s.in_events + lo;
        const unsigned n_first = alone ? 0u : min(n_ev, min((unsigned)kResBlock, 2u * row_cap));
        if (!alone)
            crowded_rows<kResBlock / kWave>(
                lists_of(k - 1), list_tag(k - 1), span, hist + (int64_t)row_before() * (words + 1), words, n_first,
                [&](unsigned i) { return input_row(events[i]); }, rows, 2u * row_cap, crowd_l, abort_word, spin_limit,
                [&](unsigned total) __attribute__((always_inline)) {
                    for (unsigned a = (unsigned)tid; a < total; a += kResBlock) {
                        const unsigned row = rows[a];
                        add_bounds(row_bounds(row), (row & kInputTag) != 0u, 0u, 1u);
                    }
                });
        n_more = wave < kWriter ? n_ev - n_first : 0u;
        more_events = events + n_first;
        if (at_row < n_more) next_source = more_events[at_row];  // (n_rows is 0, and a team one lane)
    };
    // The writer's part of a step: the list (the others wait for it), ballots, record.
    const unsigned rec_ways = s.spike_ways > 1 ? (unsigned)s.spike_ways : 1u;
    const unsigned long long rec_way = blockIdx.x & (rec_ways - 1u), rec_cap = (unsigned long long)s.spike_cap / rec_ways;
    // with as many lists of the record as workgroups this one appends to its own alone and keeps the count in a register
    const bool own_record = kRecord && s.spike_count != nullptr && rec_ways >= gridDim.x;
    unsigned long long rec_count = own_record ? s.spike_count[rec_way * BMTK_RECORD_COUNT_STRIDE] : 0ull;
    auto write = [&](int k) __attribute__((always_inline)) {
        const int w = lane_here();
        ListWrite list;
        list.read(fired_l);
        const unsigned n = fired_n[k & 1];
        const unsigned long long m = ballot_l[w & (kResBlock / kWave - 1)];
        const bool has = w < (span >> 6) && (e0 >> 6) + w < words;
        auto ballots = [&]() {
            if (has) __hip_atomic_store(hist + (int64_t)row_t * (words + 1) + (e0 >> 6) + w, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        if (n > kListMax) {  // the ballots will be read: they have to have arrived before the list says so
            ballots();
            wait_vector_memory();
        }
        list.publish(lists_of(k), g, list_tag(k), n);
        if (n <= kListMax) ballots();
        if (s.spike_bits && has) s.spike_bits[k * s.spike_bits_stride + (e0 >> 6) + w] = m;
        if (lane == 0) fired_n[(k + 1) & 1] = 0u;
        if (kRecord && s.spike_count && n > 0u) {
            unsigned long long base = rec_count;
            if (!own_record) {
                if (lane == 0) base = atomicAdd(s.spike_count + rec_way * BMTK_RECORD_COUNT_STRIDE, (unsigned long long)n);
                base = bcast_u64(base, 0);
            }
            for (unsigned i = (unsigned)lane; i < n; i += kWave) {
                if (base + i >= rec_cap) break;
                const unsigned long long to = rec_way * rec_cap + base + i;
                s.spike_step[to] = (int32_t)(r.step0 + k);
                s.spike_elem[to] = e0 + (int)fired_l[i];
                if (s.spike_frac) s.spike_frac[to] = frac_l[i];
            }
            rec_count += n;
        }
    };

    // the pulls of round k are complete
    auto pulled = [&](int k) __attribute__((always_inline)) {
        while ((int)(load_lds(&done_l) - (unsigned)(k + 1) * kWriter) < 0) {}
    };

    bool aborted = false;
    if (wave != kReader) {
        for (int k = 0; k <= n_steps; ++k) {  // (one round more than steps: the closing pull)
            const bool asked = k > 0 && load_lds(&listed_l) == (unsigned)k;
            if (asked) ask(k);
            if (k < n_steps) {
                update(k);
                if (wave != kWriter) {
                    count_lds(&updated_l);
                } else {
                    const unsigned all = (unsigned)(k + 1) * (kReaderOwns ? kReader : kWriter);
                    while ((int)(load_lds(&updated_l) - all) < 0) {}
                    write(k);
                }
            }
            __syncthreads();  // X
            if (k > 0 && !go_on[k & 1]) {
                aborted = true;
                break;
            }
            if (k > 0) {
                if (!asked) ask(k);
                if (listed == kCrowded) pull_crowded(k);
                pull(k);
            }
            if (k < n_steps) {
                slot_prev = next(slot_prev, L);
                row_t = next(row_t, r.hist);
            }
            if (wave != kWriter) count_lds(&done_l);
            pulled(k);  // Y
        }
    } else {
        ListLook seen;
        seen.none();
        bool have = false, lost = false;  // the step in hand: its rows are in LDS; given up
        unsigned failed = 0u;
        int opaque_zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(opaque_zero));
        // lanes to a segment at most: its synapses on average, rounded up to a power of two
        unsigned max_team = 0u;
        {
            float synapses = 0.0f, segments = 0.0f;
            if (!alone) synapses += (float)s.rec_indptr[s.n_neurons], segments += (float)s.n_neurons;
            if (s.in_ptr) synapses += (float)s.inp_indptr[s.n_inputs], segments += (float)s.n_inputs;
            segments *= (float)G;
            while (max_team < 6u && segments * (float)(1u << max_team) < synapses) ++max_team;
        }
        // the input events of the step in hand, the first of them on their way
        int64_t ev_lo = events_at(0), ev_hi = events_at(1);
        long long ev_next = 0;
        int32_t ev[kReaderEvents] = {};
        // one more look in vain: false when it is time to give up
        auto again = [&]() __attribute__((always_inline)) -> bool {
            if (++failed > spin_limit) __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return failed <= spin_limit && load_agent(abort_word) == 0u;
        };
        // the rows of step k, whose lists have been seen, into LDS
        auto take = [&](int k) __attribute__((always_inline)) {
            const int buf = k & 1;
            const unsigned n_ev = (unsigned)(ev_hi - ev_lo), n_listed = min(n_ev, (unsigned)(kReaderEvents * kWave));
            const unsigned me = (unsigned)lane_here(), spare = 2u * row_cap + me, at_buf = (unsigned)buf * row_cap;
            have = true;
            const unsigned total = rows_from_lists(seen, lists_of(k), list_tag(k), span, rows, at_buf, row_cap, spare, n_listed, again, lost);
            unsigned n = kCrowded;
            if (total != kCrowded) {
                n = total + n_listed;
#pragma unroll
                for (int i = 0; i < kReaderEvents; ++i) {
                    if ((unsigned)(i * kWave) >= n_ev) break;
                    const unsigned a = i * kWave + me;
                    int32_t source = ev[i];
                    asm volatile("" : "+v"(source));  // (not looked at ahead of the lists)
                    rows[a < n_ev ? at_buf + total + a : spare] = input_row(source);
                }
            }
            unsigned ts = 0u;
            if (n != kCrowded)
                while (ts < max_team && ((n + n_ev - n_listed) << (ts + 1u)) <= (unsigned)kPullThreads) ++ts;
            if (lane == 0) {
                rows_l[buf] = n == kCrowded || n_ev == n_listed ? n : n | kMoreEvents;
                spikes_l[buf] = total;
                team_l[buf] = ts;
                store_lds(&listed_l, lost ? 0u : (unsigned)k + 1u);
            }
        };
        for (int k = 0; k <= n_steps; ++k) {
            if (kReaderOwns && k < n_steps) {
                if (k > 0) pulled(k - 1);
                update(k);
                count_lds(&updated_l);
            }
            if (k > 0) {
                if (!alone) __builtin_amdgcn_s_sleep(8);
                while (!have && !lost) {
                    if (alone || seen.look(lists_of(k - 1), list_tag(k - 1)))
                        take(k - 1);
                    else
                        lost = !again();
                }
                if (lane == 0) go_on[k & 1] = !lost;
            }
            // vmcnt(0): nothing is on its way here, and with that said the compiler does not wait for loads below before it
            // uses their registers again (a trip to memory at the busiest time)
            __builtin_amdgcn_s_waitcnt(0x0F70);
            const int64_t ev_end = ((int64_t)__builtin_amdgcn_readfirstlane((int)(ev_next >> 32)) << 32) |
                                   (int64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)ev_next);
            __syncthreads();  // X
            if (k > 0 && !go_on[k & 1]) {
                aborted = true;
                break;
            }
            // (as vector loads: a scalar load's answer would be waited for at the next LDS access)
            if (s.in_ptr) ev_next = s.in_ptr[r.step0 + min(k + 2, n_steps) + opaque_zero];
            if (k > 0 && k < n_steps) {  // the events of step k are next: their end was asked for a step ago
                ev_lo = ev_hi;
                ev_hi = ev_end;
            }
            if (k < n_steps) {
                const unsigned n_ev = (unsigned)(ev_hi - ev_lo);
                const int32_t *const from = s.in_events + ev_lo;
                const unsigned me = (unsigned)lane_here();
#pragma unroll
                for (int i = 0; i < kReaderEvents; ++i) {
                    if ((unsigned)(i * kWave) >= n_ev) break;
                    if (i * kWave + me < n_ev) ev[i] = from[i * kWave + me];
                }
            }
            have = false;
            failed = 0u;
            if (k > 0 && rows_l[(k - 1) & 1] == kCrowded) pull_crowded(k);
            if (k < n_steps) {
                slot_prev = next(slot_prev, L);
                row_t = next(row_t, r.hist);
            }
        }
        if (kReaderOwns && !aborted) pulled(n_steps);
    }
    if (wave != kReader || kReaderOwns) {
        if (own && !aborted) fold(slot_prev);
        if (own) glif3_store(st, s.V, s.asc, s.y1, s.y2, s.ref, ne, e);
    }
    if (own_record && wave == kWriter && lane == 0) s.spike_count[rec_way * BMTK_RECORD_COUNT_STRIDE] = rec_count;
    __syncthreads();
    for (int c = tid; c < L * GLIF3_NREC * span; c += kResBlock) {
        const int dr = c / span, i = c - dr * span;
        if (i < mine) s.ring[(int64_t)dr * ne + e0 + i] = ring_l[c];
    }
}


// the lists of a run back to no step's
__global__ __launch_bounds__(kBlock) void zero_words_kernel(unsigned *w, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) w[i] = 0u;
}

// abort flag and arrival counters of a resident run
__global__ void zero_sync_kernel(unsigned *sync)
{
    // word 1, the abort flag, is left alone: it stays set until the host has read and cleared it
    if (threadIdx.x == 0) sync[0] = 0u;
    for (int c = threadIdx.x; c < kWays * kBarrierWords; c += blockDim.x) sync[(1 + c) * kBarrierStride] = 0u;
}

// A wavefront a row, one read of the row: where the group of a synapse's target is not that of the one before it, the groups up
// to it begin there.  One read of the indices and one write of the offsets; a binary search per offset, and a thread per row that
// looked whether it is in order, took 560 us for 30,011 rows of 300 in 256 groups and 2.8 ms for 100,000 of 500, this takes 65 and 190 (with the look at the flag).
__global__ __launch_bounds__(kBlock) void segment_offsets_kernel(int64_t n_rows, const int32_t *__restrict__ indptr,
                                                                 const int32_t *__restrict__ indices, int span,
                                                                 int n_groups, uint32_t *__restrict__ seg,
                                                                 int32_t *__restrict__ unsorted)
{
    const int lane = lane_id();
    const int64_t row = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (row >= n_rows) return;
    uint32_t *__restrict__ to = seg + row * (n_groups + 1);
    const int lo = indptr[row], hi = indptr[row + 1];
    int begun = 0;  // groups that have begun before the chunk at hand
    for (int64_t base = lo; base < hi; base += kWave) {
        const int64_t p = base + lane;
        const int mine = p < hi ? indices[p] : 0x7FFFFFFF;
        int before = __shfl_up(mine, 1, kWave);
        if (lane == 0) before = base > lo ? indices[base - 1] : mine;
        if (p < hi && mine < before) *unsorted = 1;
        // groups 0 .. mine / span have begun with this synapse
        const int upto = p < hi ? min((mine < 0 ? -1 : mine / span) + 1, n_groups + 1) : 0;
        int from = __shfl_up(upto, 1, kWave);
        if (lane == 0) from = begun;
        for (int g = from; g < upto; ++g) to[g] = (uint32_t)p;
        const int last = (int)min((int64_t)hi - base, (int64_t)kWave) - 1;
        begun = max(begun, __shfl(upto, last, kWave));
    }
    for (int g = begun + lane; g <= n_groups; g += kWave) to[g] = (uint32_t)hi;
}

int simulate_resident(const bmtk_glif3_sim &s, int64_t step0, int64_t n_steps, hipStream_t stream)
{
    if (s.res_groups == 1) return simulate_resident_solo(s, step0, n_steps, stream);  // the whole network in one workgroup
    if (n_steps >= (1ll << 31)) {
        set_error("glif3_simulate_fwd: a resident call covers fewer than 2^31 steps");
        return BMTK_E_ARG;
    }
    const int hist = s.hist_slots ? s.hist_slots : 3;
    int slack = s.delay_offset < hist - 3 - s.delay_offset ? s.delay_offset : hist - 3 - s.delay_offset;
    slack = slack < kMaxSlack ? slack : kMaxSlack;
    Resident r{step0, n_steps, s.res_span, s.res_groups, s.delay_offset, hist, slack, slack / 2 + 1, 0};
    const size_t ring_bytes = (size_t)s.ring_slots * GLIF3_NREC * s.res_span * sizeof(float);
    size_t lds = ring_bytes + kActCap * sizeof(int);
    // one table for recurrent and input rows lets the kernel drop the second set of pointers
    const bool has_inputs = s.in_ptr != nullptr;
    const int64_t rows = s.n_neurons + (has_inputs ? s.n_inputs : 0);
    const bool unified = s.rec_seg != nullptr && rows < (1ll << 24) && rows * (s.res_groups + 1) < (1ll << 32) &&
                         (!has_inputs || (s.inp_packed == s.rec_packed &&
                                          s.inp_seg == s.rec_seg + s.n_neurons * (int64_t)(s.res_groups + 1)));
    const int form = !unified || s.probe_col != nullptr ? kFormAny : (s.spike_count != nullptr ? kFormRecord : kFormLean);
    // without slack the workgroups exchange lists (a history of four rows: see sim_resident_lists_kernel)
    const bool lists = slack == 0 && s.delay_offset == 0 && s.res_fired != nullptr && s.res_groups <= kListGroups && hist >= 4;
    if (lists) {
        const size_t most = 4 * kActCap * sizeof(int), rest = kResLdsBytes - 256u - ring_bytes;
        lds = ring_bytes + (rest < most ? rest : most) / 16 * 16;
        r.row_cap = row_cap(lds - ring_bytes, form != kFormLean);
    }
    const bool reader_owns = s.res_span > kReader * kWave;
    const void *const kernels[4][3] = {
        {reinterpret_cast<const void *>(sim_resident_kernel<false, kFormAny>),
         reinterpret_cast<const void *>(sim_resident_kernel<false, kFormRecord>),
         reinterpret_cast<const void *>(sim_resident_kernel<false, kFormLean>)},
        {reinterpret_cast<const void *>(sim_resident_kernel<true, kFormAny>),
         reinterpret_cast<const void *>(sim_resident_kernel<true, kFormRecord>),
         reinterpret_cast<const void *>(sim_resident_kernel<true, kFormLean>)},
        {reinterpret_cast<const void *>(sim_resident_lists_kernel<kFormAny, false>),
         reinterpret_cast<const void *>(sim_resident_lists_kernel<kFormRecord, false>),
         reinterpret_cast<const void *>(sim_resident_lists_kernel<kFormLean, false>)},
        {reinterpret_cast<const void *>(sim_resident_lists_kernel<kFormAny, true>),
         reinterpret_cast<const void *>(sim_resident_lists_kernel<kFormRecord, true>),
         reinterpret_cast<const void *>(sim_resident_lists_kernel<kFormLean, true>)}};
    const void *kernel = kernels[lists ? (reader_owns ? 3 : 2) : (slack > 0 ? 1 : 0)][form];
    hipError_t err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) {
        set_error("glif3_simulate_fwd: resident mode needs %zu bytes of LDS: %s", lds, hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    const unsigned grid = 8u * (unsigned)((s.res_groups + 7) / 8);
    // every workgroup must be on the device at once: the grid barrier has no other way to fill
    int dev = 0, n_cu = 0, per_cu = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kResBlock, lds);
    if ((int64_t)per_cu * n_cu < (int64_t)grid) {
        set_error("glif3_simulate_fwd: %u resident workgroups do not fit the device (%d compute units x %d)", grid,
                  n_cu, per_cu);
        return BMTK_E_LAUNCH;
    }
    const int64_t list_words = 2 * kListRows * kListRowWords;  // (32-bit ones)
    if (lists)
        hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((list_words + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream,
                           reinterpret_cast<unsigned *>(lists_in(s.res_sync)), list_words);
    else
        hipLaunchKernelGGL(zero_sync_kernel, dim3(1), dim3(kBlock), 0, stream, s.res_sync);
    bmtk_glif3_sim s_copy = s;
    // BMTK_AMD_PLAIN_LAUNCH=1 uses an ordinary launch (co-residency then rests on the occupancy check
    // above and an otherwise idle device); for tools that cannot follow cooperative launches.
    const char *plain = getenv("BMTK_AMD_PLAIN_LAUNCH");
    void *args[] = {&s_copy, &r};
    if (plain && plain[0] == '1')
        err = hipLaunchKernel(kernel, dim3(grid), dim3(kResBlock), args, lds, stream);
    else
        err = hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(kResBlock), args, lds, stream);
    if (err != hipSuccess) {
        set_error("glif3_simulate_fwd: launch of %u resident workgroups failed: %s", grid, hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    return BMTK_OK;
}

}  // namespace bmtk

using namespace bmtk;

#ifdef BMTK_RES_PROFILE
extern "C" void bmtk_debug_read_prof(unsigned long long *out)
{
    (void)hipMemcpyFromSymbol(out, HIP_SYMBOL(g_prof), sizeof(g_prof));
}
extern "C" void bmtk_debug_read_prof_blocks(unsigned long long *out)
{
    (void)hipMemcpyFromSymbol(out, HIP_SYMBOL(g_prof_blk), sizeof(g_prof_blk));
}
#endif

extern "C" int bmtk_csr_segment_offsets(int64_t n_rows, const int32_t *indptr, const int32_t *indices, int32_t span,
                                        int32_t n_groups, uint32_t *seg, int32_t *unsorted, void *stream)
{
    BMTK_REQUIRE(n_rows > 0 && indptr && indices && seg && unsorted, "csr_segment_offsets: bad sizes or null pointers");
    BMTK_REQUIRE(span > 0 && n_groups > 0, "csr_segment_offsets: span and n_groups must be positive");
    const int64_t total = n_rows * (int64_t)(n_groups + 1);
    BMTK_REQUIRE(total < (1ll << 40), "csr_segment_offsets: table too large");
    hipLaunchKernelGGL(segment_offsets_kernel, dim3((unsigned)((n_rows + kBlock / kWave - 1) / (kBlock / kWave))), dim3(kBlock), 0,
                       (hipStream_t)stream, n_rows, indptr, indices, span, n_groups, seg, unsorted);
    BMTK_CHECK_LAUNCH("csr_segment_offsets");
    return BMTK_OK;
}
