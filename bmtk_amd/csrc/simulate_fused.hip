// Batched forward simulation: pull and update fused, TWO steps per pass over
// the synapse table.
//
// A wavefront advances a group of R = 64 / batch neurons (rounded down; batches of
// 8 to 64) at a time with all their trials, lane = (neuron of the group, trial);
// a batch that does not divide 64 leaves the last lanes idle (12 % at worst up to 21
// trials, 33 % at 43).  In the launch for steps t and t+1 it
//   1. streams the run of the group's rows in the joint target-major table
//      (recurrent synapses and input synapses, lane = synapse) ONCE and asks of
//      every synapse two things: did its source fire in some trial of step
//      t-1-delay (then it contributes to what arrives in step t-1) and of step
//      t-delay (arrival in step t) -- a map of the last steps' activity in LDS.
//      The synapses that pass fetch their sources' trial masks from the joint
//      history and add their weights into 64-bit fixed-point sums in LDS, one
//      per (arrival step, receptor, neuron of the group, trial): exact and
//      independent of the order of the additions.  Both questions only concern
//      spikes of steps <= t-1, which earlier launches left complete: delays are
//      at least one step, so nothing that fires in step t can arrive before
//      step t+1, whose arrivals the NEXT launch sums.  The table -- three
//      quarters of all bytes a step moves -- is thus read once per two steps;
//   2. folds the first sums into y1 and advances the elements through step
//      t, folds the second sums and advances them through step t+1, state in
//      registers in between (NEST adds the arrivals of a step at the end of
//      that step and nothing reads y1 before the next update, so adding them at
//      the top of that update performs the same two rounded operations);
//   3. writes the spike bits of both steps -- one 64-bit word each -- into rows
//      t and t+1 of the history, where later launches find them.
// No arrival sum passes through device memory.  A workgroup owns a run of
// consecutive groups and its wavefronts take them one by one from a counter in
// LDS; two of them first turn the workgroup's share of the input events of
// steps t and t+1 into bits of the same history rows, and deliver the few ids
// that occur twice within a step (bits hold an id once) as events into the
// ring, which the update folds along.
//
// What bounds it: half of a quiet launch's time is waiting for the table (51,978 neurons x 32 trials, 60 M synapses:
// 71 us per step at rest, 4.5 TB/s), the rest the events' mask fetches (one L2 line each) and additions.  Per-row
// blocks, a stage per arrival step and a map of bits took 113 us per step at 2.4 Hz; runs of rows as blocks (no block
// cut short at a row's end), one stage for both steps that is worked off when it is full, and a byte per source: 95.
// Any batch from 8 on: 20,011 x 20 trials, 16 M synapses: 36 us per step against 68 as separate pull and update launches.
// Small networks wait for chains of loads and instructions: 3,001 x 12 12.9 us a launch, 14.6 before the input events were looked up by a whole
// wavefront (input_words) and the host divided by history and ring length.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "glif3_update.hpp"
#include "propagate.hpp"
#include "pull_common.hpp"
#include "sim_internal.hpp"

namespace bmtk {

constexpr int kFuseBlock = 1024;
constexpr int kFuseWaves = kFuseBlock / kWave;
constexpr int kFuseAhead = 2;     // table blocks of 2 KB per wavefront, in flight or at hand (4 and 5: no faster)
constexpr int kFuseStage = 128;   // entries of a wavefront's stage: fewer than 64 left over and up to 64 new ones
constexpr int kFuseAccWave = 2 * GLIF3_NREC * kWave;  // sums of a wavefront: [arrival step][receptor][64]
// accumulators and stages (8 + 4 bytes per entry), then the activity map
constexpr size_t kFuseLdsFixed = (size_t)kFuseWaves * (kFuseAccWave * 8 + kFuseStage * 12);
constexpr size_t kFuseLdsMax = 160u * 1024u - 512u;  // one workgroup per compute unit

struct FusedLaunch {
    int64_t t0;          // first step of the launch (closing launch: one past the last step)
    int64_t out_row;     // row of spike_bits / save_v / save_flags of the first step (the second: one further)
    int64_t probe_row0, probe_row1;  // rows of probe_v, -1: not a sampled step
    int n_in_words;      // 64-bit words of the input part of a history row
    int n_main;          // workgroups
    int n_sub;           // steps the launch advances: 2, 1 (the odd one of a call), 0 (closing launch: fold only)
    int fold0;           // the arrivals of step t0-1 are pulled and folded first (every launch but a call's first)
    int use_ring;        // ring slots may hold arrivals (ids repeated within a step, of this call's lists or of earlier ones)
    int in_bits;         // the input events of the launch's steps become bits of their history rows
    int repeats;         // the repeated ids of the launch's steps are delivered as events
    int H;               // rows of the history (L + 4)
    int Lr;              // slots of the ring (L + 2)
    // (divisions are the host's: a 64-bit remainder is 150 scalar instructions, and a group's closing work needed four)
    int hist_row[3];     // history rows of steps t0-1, t0, t0+1
    int ring_slot[3];    // ring slots of steps t0-1, t0, t0+1
    int n_w32;           // words per row of the activity map of bits; words of one map of bytes
    int shift;           // sources per bit of the activity map: 2^shift
    int team;            // wavefronts that share a group (1: every wavefront takes groups of its own from the workgroup's counter)
    int pending;         // bit 0 / 1: the resident form left arrivals of step t0-1 / t0 in rb_ring
    int pend_slot[2];    // their slots of rb_ring
    int map_read, map_write;  // which of the two maps of bytes the launch reads and leaves behind (-1: none)
    double unit;         // of the fixed-point sums
};

// One block of the synapse stream a wavefront works through: `left` synapses (up to 256 count) of a group's run, which
// begin at position `base` of the packed table and `at` synapses into the run.
struct FuseBlockDesc {
    int grp;       // -1: past the end (an empty block of no group)
    int base, at, left;
    bool first;    // first block of its group: the group's state is asked for
    bool closes;   // last block of its group: the group is closed after it
};

// The groups a wavefront takes from its workgroup's counter, as a stream of blocks: the rows of a group follow one another
// in the table, so that its synapses are one run.  A group's row bounds sit in the lanes of one register (lane i: where
// row i of the group begins) and are fetched a group ahead, like the group itself.  A wavefront of a team has one group,
// which it shares with the others: it takes every team-th block.
template <int kRows>
struct GroupCursor {
    const int32_t *__restrict__ indptr;
    int *counter;
    int n, g_end;
    int grp, base, end;   // group at hand (-1: none), what is left of its run
    int run;              // where its run begins
    int bounds;           // row bounds of the group at hand
    int ngrp, nbounds;    // the group after (>= g_end: none)
    int stride;           // synapses from one block of the wavefront to its next
    bool at_start;

    __device__ __forceinline__ int grab()
    {
        int g = 0;
        if (lane_id() == 0) g = atomicAdd(counter, 1);
        return __builtin_amdgcn_readfirstlane(g);
    }
    __device__ __forceinline__ void look_ahead(int g)
    {
        ngrp = g;
        nbounds = indptr[min(min(ngrp, g_end) * kRows + min(lane_id(), kRows), n)];
    }
    __device__ __forceinline__ void advance()
    {
        if (ngrp >= g_end) {
            grp = -1;
            return;
        }
        grp = ngrp;
        bounds = nbounds;
        run = base = __builtin_amdgcn_readlane(bounds, 0);
        end = __builtin_amdgcn_readlane(bounds, kRows);
        at_start = true;
        look_ahead(stride == kPullChunks * kWave ? grab() : g_end);
    }
    // team == 1: groups from the counter; otherwise group `group` alone, as member `member` of a team
    __device__ __forceinline__ void start(const int32_t *ip, int n_rows, int groups_end, int *ctr, int team, int group, int member)
    {
        indptr = ip;
        counter = ctr;
        n = n_rows;
        g_end = groups_end;
        base = end = run = bounds = 0;
        stride = team * kPullChunks * kWave;
        look_ahead(team == 1 ? grab() : group);
        advance();
        if (grp >= 0) base += member * kPullChunks * kWave;
    }
    __device__ __forceinline__ FuseBlockDesc next()
    {
        if (grp < 0) return FuseBlockDesc{-1, 0, 0, 0, false, false};
        FuseBlockDesc b{grp, min(base, end), base - run, end - base, at_start, false};
        at_start = false;
        base += stride;
        if (base >= end) {
            b.closes = true;
            advance();
        }
        return b;
    }
};

// The kernel's argument block as the constant memory it lies in.  What only a group's load and closing work need of it --
// some twenty pointers -- is read from there each time (fresh_args hides where the address comes from): kept in scalar
// registers for the whole kernel, those pointers did not fit and were spilled to vector lanes and back in every turn.
using FuseArgs = const __attribute__((address_space(4))) bmtk_glif3_sim *;
__device__ __forceinline__ FuseArgs fresh_args()
{
    FuseArgs p = (FuseArgs)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}
// likewise the launch's own block, which follows it
using FuseLaunchArgs = const __attribute__((address_space(4))) FusedLaunch *;
__device__ __forceinline__ FuseLaunchArgs fresh_launch()
{
    static_assert(sizeof(bmtk_glif3_sim) % alignof(FusedLaunch) == 0, "the second argument follows the first");
    auto p = (const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr() + sizeof(bmtk_glif3_sim);
    asm volatile("" : "+s"(p));
    return (FuseLaunchArgs)p;
}
// a pointer read from there, known to point into device memory
template <typename T>
__device__ __forceinline__ T *in_memory(T *p)
{
    return (T *)(__attribute__((address_space(1))) T *)p;
}

// the input events of step t that belong to word w of the input part of a history row (`per_word` event ids a word), as bits
__device__ __forceinline__ unsigned long long input_word(const int64_t *__restrict__ in_ptr, const int32_t *__restrict__ in_events,
                                                         int64_t t, int w, int per_word)
{
    const int64_t k1 = in_ptr[t + 1];
    const int64_t lo = (int64_t)w * per_word;
    int64_t a = in_ptr[t], b = k1;
    while (a < b) {
        const int64_t mid = (a + b) >> 1;
        if ((int64_t)in_events[mid] < lo)
            a = mid + 1;
        else
            b = mid;
    }
    unsigned long long m = 0ull;
    for (; a < k1; ++a) {
        const int64_t ev = in_events[a];
        if (ev >= lo + per_word) break;
        m |= 1ull << (ev - lo);
    }
    return m;
}

// The same for steps t .. t + n_sub - 1 (at most two) and the 64 words from `w0` on, by a whole wavefront: lane l gets word w0 + l
// of either step.  `words`: 128 words of LDS of the wavefront's own.  What it costs is trips to memory, on a wavefront whose group
// waits for it: where the words' events begin is looked for with 64 probes a round, in both steps at once, and the events
// themselves come 64 at a time.  A bisection per lane and step was up to twice twelve trips, one after
// the other: 3,001 neurons x 12 trials, 1,000 inputs 14.6 -> 13.9 us a launch (12.2 without input events); 51,978 x 32 the same 187.
__device__ __forceinline__ void input_words(const int64_t *__restrict__ in_ptr, const int32_t *__restrict__ in_events, int64_t t, int n_sub,
                                            int w0, int per_word, unsigned long long *words, unsigned long long (&m)[2])
{
    const int lane = lane_id();
    const int64_t id0 = (int64_t)w0 * per_word, id1 = id0 + (int64_t)kWave * per_word;
    int64_t at[2], to[2], end[2];  // where the words' events begin lies in at .. to
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
        at[sub] = in_ptr[sub < n_sub ? t + sub : t];
        end[sub] = to[sub] = sub < n_sub ? in_ptr[t + sub + 1] : at[sub];
        words[sub * kWave + lane] = 0ull;
    }
    while (at[0] < to[0] || at[1] < to[1]) {
        int64_t step[2];
        bool before[2];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            step[sub] = (to[sub] - at[sub] + kWave - 1) / kWave;
            const int64_t r = at[sub] + lane * step[sub];
            before[sub] = r < to[sub] && (int64_t)in_events[r] < id0;
        }
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const int n = __popcll(__ballot(before[sub]));
            if (n == 0) {
                to[sub] = at[sub];
            } else {
                to[sub] = min(to[sub], at[sub] + n * step[sub]);
                at[sub] += (n - 1) * step[sub] + 1;
            }
        }
    }
    bool more[2] = {true, true};
    while (more[0] || more[1]) {
        int64_t ev[2];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) ev[sub] = more[sub] && at[sub] + lane < end[sub] ? (int64_t)in_events[at[sub] + lane] : id1;
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const bool here = ev[sub] >= id0 && ev[sub] < id1;
            if (here) {
                const unsigned in = (unsigned)(ev[sub] - id0), w = in / (unsigned)per_word;
                atomicOr(words + sub * kWave + w, 1ull << (in - w * (unsigned)per_word));
            }
            more[sub] = __ballot(here) == ~0ull;
            at[sub] += kWave;
        }
    }
    __builtin_amdgcn_wave_barrier();
    m[0] = words[lane];
    m[1] = words[kWave + lane];
    asm volatile("" : : : "memory");  // (the room is used for something else next)
}

// kRows: neurons of a group, 64 / batch.  kBytes: the activity map holds one byte per source, bit (t mod 8) = the source
// fired in some trial of step t -- one LDS read then answers both questions a synapse asks -- which takes histories of
// at most 8 rows and as many bytes of LDS as there are sources.  Otherwise it holds one bit per 2^shift sources and history row.
template <int kRows, bool kBytes>
__global__ __launch_bounds__(kFuseBlock) void sim_fused_kernel(bmtk_glif3_sim s, FusedLaunch q)
{
    extern __shared__ unsigned long long fuse_lds[];
    __shared__ int next_group;
    __shared__ int team_done[kFuseWaves];  // wavefronts of a team that are through with their blocks
    using Mask = typename std::conditional<kRows == 1, unsigned long long, unsigned>::type;  // trials of one neuron
    const int bid = (int)blockIdx.x;
    const int n = (int)s.n_neurons, batch = s.batch;
    const int64_t ne = (int64_t)n * batch;
    const int L = s.ring_slots, H = q.H;
    const unsigned lane = (unsigned)lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const bool pull_a = q.fold0 != 0, pull_b = q.n_sub == 2;  // what arrives in step t0-1 / in step t0 is summed
    const int team = q.team, team_in_wg = wave / team;
    unsigned long long *acc = fuse_lds + team_in_wg * team * kFuseAccWave;  // (a team adds into its first member's sums)
    uint2 *stage = reinterpret_cast<uint2 *>(fuse_lds + kFuseWaves * kFuseAccWave) + wave * kFuseStage;
    unsigned *stage_at = reinterpret_cast<unsigned *>(fuse_lds + kFuseWaves * (kFuseAccWave + kFuseStage)) + wave * kFuseStage;
    uint32_t *any_l = reinterpret_cast<uint32_t *>(fuse_lds + kFuseWaves * (kFuseAccWave + kFuseStage)) + kFuseWaves * kFuseStage;
    const uint8_t *any_b = reinterpret_cast<const uint8_t *>(any_l);
    const uint8_t *map_old = reinterpret_cast<const uint8_t *>(s.fuse_any + (int64_t)max(q.map_read, 0) * q.n_w32);

    // the workgroup's run of groups, and the counter its wavefronts take them from
    const int n_groups = (n + kRows - 1) / kRows;
    const int per_wg = (n_groups + q.n_main - 1) / q.n_main;
    const int g_first = bid * per_wg, g_end = min(n_groups, g_first + per_wg);
    if (threadIdx.x == 0) next_group = g_first;
    if (threadIdx.x < kFuseWaves) team_done[threadIdx.x] = 0;
    for (int r = 0; r < 2 * GLIF3_NREC; ++r) fuse_lds[wave * kFuseAccWave + r * kWave + lane] = 0ull;
    if (!kBytes) {
        // the activity rows of the steps the NEXT launch writes start empty (no launch reads them before)
        for (int k = 0; k < 2; ++k) {
            int row = q.hist_row[1] + q.n_sub + k;
            row = row >= H ? row - H : row;
            uint32_t *__restrict__ next = s.fuse_any + (int64_t)row * q.n_w32;
            for (int i = bid * kFuseBlock + (int)threadIdx.x; i < q.n_w32; i += q.n_main * kFuseBlock) next[i] = 0u;
        }
    }
    if (pull_a || pull_b) {
        if (kBytes) {
            // every byte turned so that step t0-1 is bit 7, t0-2 bit 6, ...
            const unsigned turn = 7u - (unsigned)((q.t0 - 1) & 7);
            const uint32_t up = ((0xFFu << turn) & 0xFFu) * 0x01010101u;
            const uint32_t *__restrict__ src = reinterpret_cast<const uint32_t *>(map_old);
            for (int i = threadIdx.x; i < q.n_w32; i += kFuseBlock) {
                const uint32_t x = src[i];
                any_l[i] = ((x << turn) & up) | ((x >> (8u - turn)) & ~up);
            }
        } else {
            // the activity maps of the steps t0-1 .. t0-L, one after the other
            for (int k = 0; k < L; ++k) {
                const int row = q.hist_row[0] - k;
                const uint32_t *__restrict__ src = s.fuse_any + (int64_t)(row < 0 ? row + H : row) * q.n_w32;
                for (int i = threadIdx.x; i < q.n_w32; i += kFuseBlock) any_l[k * q.n_w32 + i] = src[i];
            }
        }
    }
    __syncthreads();

    const unsigned long long field = batch == 64 ? ~0ull : ((1ull << batch) - 1ull);
    if (wave == kFuseWaves - 1 && (q.in_bits || q.map_write >= 0)) {
        // ---- the workgroup's share of the input events of the launch's steps as bits of their history rows: a
        //      lane per 64-bit word, which holds the trials of kRows sources.  (Read by later launches.)  The wavefront
        //      then takes groups like the others, which have taken a few more meanwhile. ----
        uint8_t *map_new = reinterpret_cast<uint8_t *>(s.fuse_any + (int64_t)max(q.map_write, 0) * q.n_w32);
        // the bits of the map's bytes that belong to the launch's steps
        const unsigned step_bit0 = 1u << (unsigned)(q.t0 & 7), step_bit1 = 1u << (unsigned)((q.t0 + 1) & 7);
        const unsigned step_bits = (q.n_sub > 0 ? step_bit0 : 0u) | (q.n_sub > 1 ? step_bit1 : 0u);
        const int in_word0 = (int)(s.fuse_in_base / kRows);
        const int per_word = kRows * batch;
        for (int w0 = bid * kWave; w0 < q.n_in_words; w0 += q.n_main * kWave) {
            unsigned long long bits[2] = {0ull, 0ull};
            const int w = w0 + (int)lane;
            if (q.in_bits) input_words(s.in_ptr, s.in_events, q.t0, q.n_sub, w0, per_word, reinterpret_cast<unsigned long long *>(stage), bits);
            if (w >= q.n_in_words) break;
            if (q.in_bits) {
#pragma unroll
                for (int sub = 0; sub < 2; ++sub)
                    if (sub < q.n_sub) s.work_bits[(int64_t)q.hist_row[1 + sub] * s.fuse_hist_stride + in_word0 + w] = bits[sub];
            }
#pragma unroll
            for (int f = 0; f < kRows; ++f) {
                const int source = (int)s.fuse_in_base + w * kRows + f;
                const bool on0 = ((bits[0] >> (f * batch)) & field) != 0ull, on1 = ((bits[1] >> (f * batch)) & field) != 0ull;
                if (kBytes) {
                    if (q.map_write >= 0)
                        map_new[source] = (uint8_t)((map_old[source] & ~step_bits) | (on0 ? step_bit0 : 0u) | (on1 ? step_bit1 : 0u));
                } else {
                    const unsigned g = (unsigned)source >> q.shift;
                    if (on0) atomicOr(s.fuse_any + (int64_t)q.hist_row[1] * q.n_w32 + (g >> 5), 1u << (g & 31u));
                    if (on1) atomicOr(s.fuse_any + (int64_t)q.hist_row[2] * q.n_w32 + (g >> 5), 1u << (g & 31u));
                }
            }
        }
    }
    if (wave == kFuseWaves - 2 && q.repeats) {
        // ---- ids that occur more than once among the input events of the launch's steps: the occurrences after
        //      the first, as events into the ring.  Those of step u land in slots u+1 .. u+L-1; this launch takes
        //      slots t0-1 and t0 along, which the launches before it completed (the ring has L+2 slots, so that
        //      slot t0+L is neither of the two) ----
        const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(s.inp_packed);
        const int ring_map_words = (n + 31) >> 5;
        uint32_t *__restrict__ ring_map = s.fuse_any + (kBytes ? 2 : (int64_t)H) * q.n_w32;
        for (int sub = 0; sub < q.n_sub; ++sub) {
            const int64_t t = q.t0 + sub;
            const int64_t k0 = s.in_repeat_ptr[t], k1 = s.in_repeat_ptr[t + 1];
            for (int64_t k = k0 + bid; k < k1; k += q.n_main) {
                const int e = s.in_repeat_events[k];
                const int j = (int)((uint32_t)e / (uint32_t)batch), b = e - j * batch;
                const int p1 = s.inp_indptr[j + 1];
                for (int p = s.inp_indptr[j] + (int)lane; p < p1; p += kWave) {
                    const uint2 sy = rows[p];
                    int slot = q.ring_slot[1 + sub] + (int)(sy.x >> 26);  // (delays are below L, Lr is L + 2)
                    slot = slot >= q.Lr ? slot - q.Lr : slot;
                    const int64_t i = sy.x & 0xFFFFFFu;
                    atomicAdd(s.ring + ((int64_t)(slot * GLIF3_NREC + (int)((sy.x >> 24) & 3u)) * ne + i * batch + b),
                              __uint_as_float(sy.y));
                    atomicOr(ring_map + (int64_t)slot * ring_map_words + (i >> 5), 1u << (i & 31));
                }
            }
        }
    }

    // ---- a group at a time: pull, fold, update, fold, update ----
    const unsigned uw32 = (unsigned)q.n_w32, ushift = (unsigned)q.shift, umax_dd = (unsigned)(L - 2);
    const unsigned sub_lane = lane / (unsigned)batch;            // this lane's neuron within a group
    const unsigned sub_bit = sub_lane * (unsigned)batch;         // where the neuron's trials begin in the group's 64 bits
    const bool first_trial = lane == sub_bit, in_group = sub_lane < (unsigned)kRows;
    // Asked for when a group's first block turns up, used when the group is closed: the state of its elements,
    // their propagators (every lane its neuron's column), the words of the ring map that hold the group's bits, and the
    // neuron's byte of the activity map.
    Glif3Elem st;
    Glif3Prop pr;
    unsigned ring_word0 = 0u, ring_word1 = 0u, byte_old = 0u;

    // Element accesses: a scalar base (array + plane k of ne elements) and this lane's 32-bit byte offset
    // (n_neurons * batch < 2^30, checked by the caller), the address form that needs no 64-bit lane arithmetic.
    const size_t plane = (size_t)ne * sizeof(float);
    auto ldf = [&](const float *base, int k, unsigned boff) {
        return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(in_memory(base)) + k * plane + boff);
    };
    auto stf = [&](float *base, int k, unsigned boff, float v) {
        *reinterpret_cast<float *>(reinterpret_cast<char *>(in_memory(base)) + k * plane + boff) = v;
    };
    // All lanes load, whatever they hold (the lanes past the last neuron of the network or past the group's elements load
    // the last element's values and keep them to themselves): a load under a condition would have to be waited for at
    // once, where the two ways meet again.
    // ring map: bit i of row (u % Lr) = some ring cell of neuron i in slot u % Lr holds an arrival (set where
    // repeated ids are delivered, cleared by the neuron's owner when it takes the cells along); behind the activity map
    auto ring_row = [&](FuseArgs sp, FuseLaunchArgs qp, int slot) -> uint32_t * {
        return in_memory(sp->fuse_any) + (kBytes ? 2 : (int64_t)qp->H) * qp->n_w32 + (int64_t)slot * ((n + 31) >> 5);
    };
    auto load_group = [&](int grp) {
        const FuseArgs sp = fresh_args();
        const FuseLaunchArgs qp = fresh_launch();
        const int row = min(grp * kRows + (int)min(sub_lane, (unsigned)kRows - 1u), n - 1);
        const unsigned e = min((unsigned)(grp * kRows) * (unsigned)batch + lane, (unsigned)ne - 1u);
        const unsigned boff = e * 4u;
        const int64_t col = sp->class_id ? (int64_t)in_memory(sp->class_id)[row] : (int64_t)row;
        pr.load(in_memory(sp->prop), sp->prop_stride, col);
        if (qp->use_ring) {
            ring_word0 = ring_row(sp, qp, qp->ring_slot[0])[row >> 5];
            ring_word1 = ring_row(sp, qp, qp->ring_slot[1])[row >> 5];
        }
        if (kBytes) byte_old = reinterpret_cast<const uint8_t *>(in_memory(sp->fuse_any) + (int64_t)max(qp->map_read, 0) * qp->n_w32)[row];
        if (qp->n_sub > 0) {
            st.V = ldf(sp->V, 0, boff);
            st.ref = *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(in_memory(sp->ref)) + boff);
#pragma unroll
            for (int k = 0; k < GLIF3_NASC; ++k) st.asc[k] = ldf(sp->asc, k, boff);
#pragma unroll
            for (int k = 0; k < GLIF3_NREC; ++k) {
                st.y1[k] = ldf(sp->y1, k, boff);
                st.y2[k] = ldf(sp->y2, k, boff);
            }
        }
    };
    // what is left to do for a group once its arrival sums are known: a0 what arrived in step t0-1, a1 in step t0
    auto finish_group = [&](int grp, float (&a0)[GLIF3_NREC], float (&a1)[GLIF3_NREC]) {
        const FuseArgs sp = fresh_args();
        const FuseLaunchArgs qp = fresh_launch();
        const int row = grp * kRows + (int)sub_lane;
        const bool on = in_group && row < n;  // this lane holds an element
        const unsigned e0 = (unsigned)(grp * kRows) * (unsigned)batch, e = e0 + lane, boff = e * 4u;
        // the ring cells of one slot, where an id repeated within a step reached this neuron (rare)
        auto take_ring = [&](int slot, unsigned word, float (&a)[GLIF3_NREC]) {
            if (qp->use_ring && on && ((word >> ((unsigned)row & 31u)) & 1u)) {
                float *cells = in_memory(sp->ring) + (int64_t)slot * GLIF3_NREC * ne;
                float v[GLIF3_NREC];
#pragma unroll
                for (int k = 0; k < GLIF3_NREC; ++k) v[k] = ldf(cells, k, boff);
#pragma unroll
                for (int k = 0; k < GLIF3_NREC; ++k) {
                    stf(cells, k, boff, 0.0f);
                    a[k] = v[k] + a[k];
                }
                if (first_trial) atomicAnd(ring_row(sp, qp, slot) + (row >> 5), ~(1u << ((unsigned)row & 31u)));
            }
        };
        if (qp->fold0) take_ring(qp->ring_slot[0], ring_word0, a0);
        if (qp->n_sub == 0) {
            // closing launch: what arrived in the last step enters y1, as at the end of that step
            if (on) {
#pragma unroll
                for (int k = 0; k < GLIF3_NREC; ++k) stf(sp->y1, k, boff, ldf(sp->y1, k, boff) + a0[k] * pr.psc0[k]);
                if (kBytes && first_trial && qp->map_write >= 0) reinterpret_cast<uint8_t *>(in_memory(sp->fuse_any) + (int64_t)qp->map_write * qp->n_w32)[row] = (uint8_t)byte_old;
            }
            return;
        }
        const unsigned step_bit0 = 1u << (unsigned)(qp->t0 & 7), step_bit1 = 1u << (unsigned)((qp->t0 + 1) & 7);
        unsigned fired_bits = 0u;  // of the neuron's byte of the activity map
        // one step: fold, update, the step's outputs
        auto one_step = [&](int sub, bool fold, const float (&a)[GLIF3_NREC], int64_t probe_row) {
            const int64_t t = qp->t0 + sub, out_row = qp->out_row + sub;
            bool spike = false;
            float frac = 0.0f;
            if (on) {
                if (fold) {
#pragma unroll
                    for (int k = 0; k < GLIF3_NREC; ++k) st.y1[k] = st.y1[k] + a[k] * pr.psc0[k];
                }
                const float zero[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f};
                const float I = sp->i_ext ? ldf(sp->i_ext, 0, boff) : 0.0f;
                const int ref_before = st.ref;
                spike = glif3_update(st, pr, sp->h, zero, I, &frac);
                if (probe_row >= 0) {
                    const int pc = *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(in_memory(sp->probe_col)) + boff);
                    if (pc >= 0) in_memory(sp->probe_v)[probe_row * sp->probe_stride + pc] = st.V;
                }
                if (sp->save_v) {
                    stf(sp->save_v + out_row * ne, 0, boff, st.V);
                    in_memory(sp->save_flags)[out_row * ne + e] = (uint8_t)((spike ? BMTK_F_SPIKE : 0) |
                                                                  (ref_before == 0 ? BMTK_F_INTEGRATING : 0) |
                                                                  (ref_before > 0 && st.ref == 0 ? BMTK_F_RESET : 0));
                }
            }
            // the group's elements are one word of spike bits
            const unsigned long long m = __ballot(spike);
            if (lane == 0) in_memory(sp->work_bits)[qp->hist_row[1 + sub] * sp->fuse_hist_stride + grp] = m;
            if (sp->spike_bits) {
                // the same bits in the run's output, element after element: where a group fills its 64 bits a word of
                // its own, otherwise pieces of one or two words (cleared by the driver)
                uint64_t *out = in_memory(sp->spike_bits) + out_row * sp->spike_bits_stride;
                if (kRows * batch == 64) {
                    if (lane == 0) out[grp] = m;
                } else if (m != 0ull) {
                    const unsigned sh = e0 & 63u;
                    const unsigned long long part = lane == 0 ? m << sh : sh != 0u ? m >> (64u - sh) : 0ull;
                    if (lane < 2u && part != 0ull) atomicOr(reinterpret_cast<unsigned long long *>(out) + (e0 >> 6) + lane, part);
                }
            }
            const bool row_fired = ((m >> (sub_bit & 63u)) & field) != 0ull;
            if (kBytes) {
                fired_bits |= row_fired ? (sub == 0 ? step_bit0 : step_bit1) : 0u;
            } else if (m != 0ull && on && first_trial && row_fired) {
                const unsigned g = (unsigned)row >> qp->shift;
                atomicOr(in_memory(sp->fuse_any) + (int64_t)qp->hist_row[1 + sub] * qp->n_w32 + (g >> 5), 1u << (g & 31u));
            }
            if (sp->spike_count && m != 0ull) {
                // one counter bump per wavefront, record slots handed out in lane order
                const int leader = __ffsll((long long)m) - 1;
                unsigned long long base = 0ull;
                const unsigned ways = sp->spike_ways > 1 ? (unsigned)sp->spike_ways : 1u;
                const unsigned long long way = (unsigned)bid & (ways - 1u), way_cap = (unsigned long long)sp->spike_cap / ways;
                if ((int)lane == leader)
                    base = atomicAdd(in_memory(sp->spike_count) + way * BMTK_RECORD_COUNT_STRIDE, (unsigned long long)__popcll(m));
                base = bcast_u64(base, leader);
                unsigned long long idx = base + (unsigned long long)lane_prefix(m);
                if (spike && idx < way_cap) {
                    idx += way * way_cap;
                    in_memory(sp->spike_step)[idx] = (int32_t)t;
                    in_memory(sp->spike_elem)[idx] = (int32_t)e;
                    if (sp->spike_frac) in_memory(sp->spike_frac)[idx] = frac;
                }
            }
        };
        one_step(0, qp->fold0 != 0, a0, qp->probe_row0);
        if (qp->n_sub == 2) {
            take_ring(qp->ring_slot[1], ring_word1, a1);
            one_step(1, true, a1, qp->probe_row1);
        }
        if (on) {
            if (kBytes && first_trial && qp->map_write >= 0) reinterpret_cast<uint8_t *>(in_memory(sp->fuse_any) + (int64_t)qp->map_write * qp->n_w32)[row] = (uint8_t)((byte_old & ~(step_bit0 | (qp->n_sub > 1 ? step_bit1 : 0u))) | fired_bits);
            stf(sp->V, 0, boff, st.V);
            *reinterpret_cast<int32_t *>(reinterpret_cast<char *>(in_memory(sp->ref)) + boff) = st.ref;
#pragma unroll
            for (int k = 0; k < GLIF3_NASC; ++k) stf(sp->asc, k, boff, st.asc[k]);
#pragma unroll
            for (int k = 0; k < GLIF3_NREC; ++k) {
                stf(sp->y1, k, boff, st.y1[k]);
                stf(sp->y2, k, boff, st.y2[k]);
            }
        }
    };

    if (!pull_a && !pull_b) {
        // one step as a call's first launch: the closing launch of the call before it has folded everything that
        // arrived, and nothing is summed here
        if (team > 1) {
            const int grp = bid * (kFuseWaves / team) + team_in_wg;
            if (grp >= n_groups || wave != team_in_wg * team) return;
            float a0[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f}, a1[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f};
            load_group(grp);
            finish_group(grp, a0, a1);
            return;
        }
        for (int grp = 0;;) {
            if (lane == 0) grp = atomicAdd(&next_group, 1);
            grp = __builtin_amdgcn_readfirstlane(grp);
            if (grp >= g_end) break;
            float a0[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f}, a1[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f};
            load_group(grp);
            finish_group(grp, a0, a1);
        }
        return;
    }

    const unsigned hrow_bytes = (unsigned)s.fuse_hist_stride * 8u;  // H * stride * 8 < 2^32 (checked by the caller)
    const unsigned uH = (unsigned)H;
    const char *__restrict__ hist_bytes = reinterpret_cast<const char *>(s.work_bits);
    const char *__restrict__ packed = reinterpret_cast<const char *>(s.fuse_packed);
    // Block of the table: 64-bit words at a scalar base, 8 * lane bytes on.  A chunk that lies wholly past the end of the
    // group's run reads the run's last chunk again, one that lies partly past it the synapses behind (the table is
    // followed by a chunk of any content): no lane arithmetic and no branch, every call issues exactly four loads, which
    // is what lets a turn wait for ITS block only and leave the younger ones in flight (the wait is a count of loads
    // still out, fixed at compile time).
    auto fetch = [&](unsigned long long *dst, const FuseBlockDesc &blk) {
        const char *__restrict__ src = packed + (size_t)(unsigned)blk.base * 8u;
        const int last = (max(blk.left, 1) - 1) >> 6;
#pragma unroll
        for (int u = 0; u < kPullChunks; ++u)
            dst[u] = __builtin_nontemporal_load(
                reinterpret_cast<const unsigned long long *>(src + (size_t)(unsigned)min(u, last) * (kWave * 8u) + lane * 8u));
    };
    // kFuseAhead table blocks per wavefront: the one at hand and the ones after it, whose loads stay in flight
    // while the wavefront works (a buffer is refilled, with the block kFuseAhead ahead, as soon as its turn is
    // over).  The buffers take turns in place -- a register copy of a block still on its way would wait for it --
    // (and a buffer chosen at run time would leave the compiler no way to tell which loads a turn may leave in
    // flight: it then waits for all of them), so the loop body holds one turn per buffer.
    GroupCursor<kRows> cursor;
    cursor.start(s.fuse_indptr, n, team == 1 ? g_end : n_groups, &next_group, team, bid * (kFuseWaves / team) + team_in_wg, wave - team_in_wg * team);
    FuseBlockDesc dq[kFuseAhead];
    unsigned long long d[kFuseAhead][kPullChunks];
    int row_bounds = 0;  // of the group whose synapses are being staged
    int bounds_of[kFuseAhead];
#pragma unroll
    for (int k = 0; k < kFuseAhead; ++k) {
        bounds_of[k] = cursor.bounds;
        dq[k] = cursor.next();
        fetch(d[k], dq[k]);
    }
    if (dq[0].grp < 0) return;
    // Synapses whose source was active, of either arrival step, are parked in one stage: {source | receptor << 24 | how
    // many steps before step t0-1 the source fired << 26, weight} and {place in the group's run | arrival step << 31}.  As soon as it
    // holds 64 of them they are worked off, in two halves a turn apart, so that the masks travel while the wavefront
    // works on the next block: the first takes them into registers and asks for their sources' trial masks, the
    // second adds the weights.  A group's closing work waits for its last masks the same way and is done in the turn
    // after the group's last block.
    unsigned head = 0u, tail = 0u;   // entries head .. tail-1 (mod kFuseStage) are parked; same in all lanes
    const unsigned arrive = (unsigned)q.hist_row[0];
    unsigned pend_acc = 0u, pend_shift = 0u;
    unsigned long long pend_w = 0ull, pend_m = 0ull;
    bool pend_any = false;           // masks are on their way (same in all lanes)
    int fin_grp = -1;                // the group whose closing work is due
    auto flush_issue = [&](unsigned count) {
        const unsigned at = (head + lane) & (unsigned)(kFuseStage - 1);
        const bool some = lane < count;
        const uint2 e = stage[at];
        const unsigned pos = stage_at[at];
        // (every lane loads: the lanes without a synapse the mask of source 0 in the row of step t0-1, and ignore it)
        const unsigned tdr = some ? e.x : 0u;
        const unsigned src = tdr & 0xFFFFFFu;
        const unsigned word = src / (unsigned)kRows;
        const unsigned back = arrive - (tdr >> 26);  // history row of the emitting step, by unsigned wrap-around
        const unsigned hrow = min(back, back + uH);
        pend_m = *reinterpret_cast<const unsigned long long *>(hist_bytes + (hrow * hrow_bytes + word * 8u));
        pend_shift = some ? (src - word * (unsigned)kRows) * (unsigned)batch : 64u;
        unsigned row = 0u;
        const int run = __builtin_amdgcn_readlane(row_bounds, 0);
#pragma unroll
        for (int r = 1; r < kRows; ++r)
            row += (pos & 0x7FFFFFFFu) >= (unsigned)(__builtin_amdgcn_readlane(row_bounds, r) - run) ? 1u : 0u;
        pend_acc = (((pos >> 31) * GLIF3_NREC + ((tdr >> 24) & 3u)) * kWave + row * (unsigned)batch);
        pend_w = to_fixed(__uint_as_float(e.y));
        pend_any = true;
        head += count;
    };
    auto flush_complete = [&]() {
        if (!pend_any) return;
        Mask m = pend_shift < 64u ? (Mask)((pend_m >> (pend_shift & 63u)) & field) : (Mask)0;
        unsigned long long *a = acc + pend_acc;
        while (m) {
            const int b = kRows == 1 ? __ffsll((long long)m) - 1 : __ffs((int)m) - 1;
            m &= m - 1;
            atomicAdd(a + b, pend_w);
        }
        pend_any = false;
    };
    // the masks under way, then the closing work of the group they belonged to
    auto resolve = [&]() {
        flush_complete();
        if (team > 1) {
            // the member that is through last closes the group: its look at the counter comes after everybody's additions
            int before = 0;
            if (lane == 0) before = __hip_atomic_fetch_add(&team_done[team_in_wg], 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (__builtin_amdgcn_readfirstlane(before) != team - 1) {
                fin_grp = -1;
                return;
            }
        }
        float a0[GLIF3_NREC], a1[GLIF3_NREC];
        const FuseLaunchArgs qp = fresh_launch();
        if (qp->pending) {
            // the first steps after a call in the resident form: what that call's spikes still send joins the sums (and is cleared
            // behind the launches, see clear_taken_kernel)
            const FuseArgs sp = fresh_args();
            const int row = fin_grp * kRows + (int)sub_lane;
            if (in_group && row < n) {
                uint64_t *left = in_memory(sp->rb_ring) + (int64_t)(lane - sub_bit) * (L - 1) * GLIF3_NREC * n + row;
                // (a cell at a time: 16 of them at once spill registers that every turn of a launch without any needs)
#pragma unroll
                for (int r = 0; r < GLIF3_NREC; ++r) {
                    if (qp->pending & 1) acc[r * kWave + lane] += left[(int64_t)(qp->pend_slot[0] * GLIF3_NREC + r) * n];
                    if (qp->pending & 2) acc[(GLIF3_NREC + r) * kWave + lane] += left[(int64_t)(qp->pend_slot[1] * GLIF3_NREC + r) * n];
                }
            }
        }
#pragma unroll
        for (int r = 0; r < GLIF3_NREC; ++r) {
            a0[r] = from_fixed(acc[r * kWave + lane], qp->unit);
            a1[r] = from_fixed(acc[(GLIF3_NREC + r) * kWave + lane], qp->unit);
            acc[r * kWave + lane] = 0ull;
            acc[(GLIF3_NREC + r) * kWave + lane] = 0ull;
        }
        finish_group(fin_grp, a0, a1);
        fin_grp = -1;
    };
    auto park = [&](unsigned long long who, unsigned long long syn, unsigned pos, bool later) {
        const unsigned count = (unsigned)__popcll(who);
        if (count == 0u) return;
        const unsigned at = (tail + (unsigned)lane_prefix(who)) & (unsigned)(kFuseStage - 1);
        if ((who >> lane) & 1ull) {
            stage[at] = make_uint2((unsigned)syn - (later ? 1u << 26 : 0u), (unsigned)(syn >> 32));
            stage_at[at] = pos + (later ? 0x80000000u : 0u);
        }
        tail += count;
        if (tail - head >= (unsigned)kWave) {
            flush_complete();
            flush_issue(kWave);
        }
    };
    // one turn: the block `cb` with its table words `cd`; afterwards the buffer takes the block kFuseAhead ahead
    auto turn = [&](FuseBlockDesc &cb, unsigned long long *cd, int &cb_bounds) {
        // activity of the four chunks' sources, for both arrival steps (LDS reads, no branch between them): a synapse of
        // delay d sends what its source fired in step t0-1-d to arrival step t0-1 and what it fired in step t0-d to
        // arrival step t0
        unsigned long long who_a[kPullChunks], who_b[kPullChunks];
        if (kBytes) {
            unsigned byte[kPullChunks];
#pragma unroll
            for (int u = 0; u < kPullChunks; ++u) byte[u] = any_b[(unsigned)cd[u] & 0xFFFFFFu];
#pragma unroll
            for (int u = 0; u < kPullChunks; ++u) {
                const bool valid = (int)lane + u * kWave < cb.left;
                // (bit 7: step t0-1; the synapse's delay moves step t0-1-delay there, and step t0-delay to bit 8)
                const unsigned x = byte[u] << ((unsigned)cd[u] >> 26);
                who_a[u] = __ballot(valid && pull_a && (x & 0x80u));
                who_b[u] = __ballot(valid && pull_b && (x & 0x100u));
            }
        } else {
            unsigned word_a[kPullChunks], word_b[kPullChunks], bit[kPullChunks];
#pragma unroll
            for (int u = 0; u < kPullChunks; ++u) {
                const unsigned tdr = (unsigned)cd[u];
                const unsigned g = (tdr & 0xFFFFFFu) >> ushift;
                bit[u] = g & 31u;
                // the map of step t0-1-k is row k; delays are 1 .. L-1 (the records behind the table may hold delay 0: kept
                // inside the map, ignored below)
                const unsigned at = __umul24(min((tdr >> 26) - 1u, umax_dd), uw32) + (g >> 5);
                word_b[u] = any_l[at];
                word_a[u] = any_l[at + uw32];
            }
#pragma unroll
            for (int u = 0; u < kPullChunks; ++u) {
                const bool valid = (int)lane + u * kWave < cb.left;
                who_a[u] = __ballot(valid && pull_a && ((word_a[u] >> bit[u]) & 1u));
                who_b[u] = __ballot(valid && pull_b && ((word_b[u] >> bit[u]) & 1u));
            }
        }
        // the group before: its last masks were asked for a turn ago, its closing work comes before any synapse of
        // this group is added (the one place of a turn where a group is closed)
        if (fin_grp >= 0) resolve();
        if (cb.first) {
            row_bounds = cb_bounds;
            load_group(cb.grp);  // (after that group's closing work, which used the same registers)
        }
#pragma unroll
        for (int u = 0; u < kPullChunks; ++u) {
            const unsigned pos = (unsigned)cb.at + u * kWave + lane;
            park(who_a[u], cd[u], pos, false);
            park(who_b[u], cd[u], pos, true);
        }
        if (cb.closes) {
            flush_complete();
            if (tail != head) flush_issue(tail - head);
            fin_grp = cb.grp;
        }
        cb_bounds = cursor.bounds;
        cb = cursor.next();
        fetch(cd, cb);
    };
    // One way out of the loop, after a whole round of the buffers: with a way out after every turn the compiler
    // joins them in one block before the loop's head, and from there it looks as if a turn could follow directly
    // on the fetch of its own buffer -- every turn would then wait for all loads in flight.  The turns past a
    // wavefront's last block (at most kFuseAhead - 1) see empty blocks of no group.
    do {
#pragma unroll
        for (int k = 0; k < kFuseAhead; ++k) turn(dq[k], d[k], bounds_of[k]);
    } while (dq[0].grp >= 0);
    if (fin_grp >= 0) resolve();
}

// the launch-per-two-steps variant for `rows` neurons per group
const void *fused_variant(int rows, bool bytes)
{
#define BMTK_FUSE(r) case r: return bytes ? reinterpret_cast<const void *>(sim_fused_kernel<r, true>) : reinterpret_cast<const void *>(sim_fused_kernel<r, false>)
    switch (rows) {
        BMTK_FUSE(1);
        BMTK_FUSE(2);
        BMTK_FUSE(3);
        BMTK_FUSE(4);
        BMTK_FUSE(5);
        BMTK_FUSE(6);
        BMTK_FUSE(7);
        BMTK_FUSE(8);
    default: return nullptr;
    }
#undef BMTK_FUSE
}

// The input part of the history row of step t once more, from the lists in force, before a call's first launch
// (bmtk_glif3_sim.in_again): its words, and the sources' bits in the activity map (a map of bits only gains some: a bit
// too many costs a mask fetch).
template <bool kBytes>
__global__ __launch_bounds__(kBlock) void input_again_kernel(bmtk_glif3_sim s, FusedLaunch q, int64_t t, int rows)
{
    const int w = (int)blockIdx.x * kBlock + (int)threadIdx.x;
    if (w >= q.n_in_words) return;
    const unsigned long long m = input_word(s.in_ptr, s.in_events, t, w, rows * s.batch);
    s.work_bits[(t % q.H) * s.fuse_hist_stride + s.fuse_in_base / rows + w] = m;
    const unsigned long long field = s.batch == 64 ? ~0ull : ((1ull << s.batch) - 1ull);
    for (int f = 0; f < rows; ++f) {
        const int source = (int)s.fuse_in_base + w * rows + f;
        const bool on = ((m >> (f * s.batch)) & field) != 0ull;
        if (kBytes) {
            uint8_t *map = reinterpret_cast<uint8_t *>(s.fuse_any);
            map[source] = (uint8_t)((map[source] & ~(1u << (unsigned)(t & 7))) | (on ? 1u << (unsigned)(t & 7) : 0u));
        } else if (on) {
            const unsigned g = (unsigned)source >> q.shift;
            atomicOr(s.fuse_any + (t % q.H) * q.n_w32 + (g >> 5), 1u << (g & 31u));
        }
    }
}

__global__ __launch_bounds__(kBlock) void zero_bits_kernel(uint64_t *__restrict__ bits, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) bits[i] = 0ull;
}

// What a call took from rb_ring, [trial][slot][receptor][neuron], cleared behind its launches: `count` slots from `slot0` on.  A
// call that is captured into a graph thereby takes it over in the first replay only.  (Cleared by the launches themselves,
// each cell as it was read, it cost all of them two spilled registers and 12 bytes of scratch: 1 % of a training step of
// 3,001 neurons x 12 trials, which never leaves anything there.)
__global__ __launch_bounds__(kBlock) void clear_taken_kernel(uint64_t *__restrict__ ring, int64_t words, int slot_words, int slots, int slot0, int count)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < words; i += (int64_t)gridDim.x * kBlock) {
        const int64_t row = i / slot_words, trial = row / count;
        const int slot = (slot0 + (int)(row - trial * count)) % slots;
        ring[(trial * slots + slot) * slot_words + (i - row * slot_words)] = 0ull;
    }
}

int simulate_fused(const bmtk_glif3_sim &s, int64_t step0, int64_t n_steps, hipStream_t stream)
{
    const int batch = s.batch, L = s.ring_slots;
    BMTK_REQUIRE(batch >= 8 && batch <= kWave, "glif3_simulate_fwd: the fused form runs batches of 8 to 64");
    BMTK_REQUIRE(s.fuse_indptr && s.fuse_any, "glif3_simulate_fwd: the fused form needs fuse_indptr and fuse_any");
    BMTK_REQUIRE(s.n_neurons * (int64_t)batch < (1ll << 30),
                 "glif3_simulate_fwd: the fused form addresses fewer than 2^30 elements");
    BMTK_REQUIRE(s.delay_offset == 0 && (s.delay_bits == 0 || s.delay_bits == 6) && s.hist_slots == L + 4,
                 "glif3_simulate_fwd: the fused form needs delay_offset 0, the standard packing and hist_slots == ring_slots + 4");
    BMTK_REQUIRE(s.sum_shift >= 0 && s.sum_shift <= BMTK_SUM_SHIFT_MAX, "glif3_simulate_fwd: sum_shift must lie in 0..BMTK_SUM_SHIFT_MAX");
    BMTK_REQUIRE(s.fuse_shift >= 0 && s.fuse_shift <= 16, "glif3_simulate_fwd: fuse_shift must lie in 0..16");
    const int rows = kWave / batch;  // neurons of a group: one 64-bit word of a history row
    const int64_t n_groups = (s.n_neurons + rows - 1) / rows;
    const int64_t in_base = n_groups * rows;
    BMTK_REQUIRE(s.fuse_in_base == in_base, "glif3_simulate_fwd: fuse_in_base must be n_neurons rounded up to a multiple of 64 / batch");
    const bool has_inp = s.in_ptr != nullptr;
    BMTK_REQUIRE(s.n_inputs >= 0, "glif3_simulate_fwd: n_inputs must not be negative");
    const int64_t n_in = s.n_inputs;  // input sources of the joint space, with or without events in this call
    BMTK_REQUIRE(in_base + n_in + rows < (1ll << 24),
                 "glif3_simulate_fwd: the fused form indexes fewer than 2^24 sources (neurons and inputs together)");
    const int64_t n_in_words = (n_in + rows - 1) / rows;
    BMTK_REQUIRE(s.fuse_hist_stride == n_groups + n_in_words + 1,
                 "glif3_simulate_fwd: fuse_hist_stride must be the words of both parts of a history row plus one");
    BMTK_REQUIRE((int64_t)(L + 4) * s.fuse_hist_stride < (1ll << 29), "glif3_simulate_fwd: joint history beyond 4 GiB");
    // the activity map: one byte per source where steps and sources allow it, else a bit per 2^shift sources and row
    const int64_t byte_words = ((n_groups + n_in_words) * rows + 3) / 4;
    const bool bytes = s.fuse_shift == 0 && L <= 8 && kFuseLdsFixed + (size_t)byte_words * 4u <= kFuseLdsMax;
    const int64_t groups = (in_base + n_in + (1ll << s.fuse_shift) - 1) >> s.fuse_shift;
    const int n_w32 = bytes ? (int)byte_words : (int)((groups + 31) / 32);
    const size_t lds = kFuseLdsFixed + (size_t)n_w32 * 4u * (bytes ? 1u : (unsigned)L);
    BMTK_REQUIRE(lds <= kFuseLdsMax, "glif3_simulate_fwd: the activity map does not fit in LDS; use a larger fuse_shift");
    BMTK_REQUIRE(s.rb_pend_until == 0 || s.rb_ring, "glif3_simulate_fwd: rb_pend_until needs rb_ring");
    BMTK_REQUIRE(!s.in_repeat_ptr || (s.in_repeat_events && s.inp_indptr && s.inp_packed),
                 "glif3_simulate_fwd: repeat lists need in_repeat_events and the source-major input table");
    BMTK_REQUIRE(!s.probe_col || (s.probe_v && s.probe_every >= 1 && s.probe_stride >= 1),
                 "glif3_simulate_fwd: probes need probe_v, probe_stride and probe_every >= 1");
    int dev = 0;
    (void)hipGetDevice(&dev);
    static int cu_count[64];  // compute units of every device seen so far
    int n_cu = (dev >= 0 && dev < 64) ? cu_count[dev] : 0;
    if (n_cu <= 0) {
        n_cu = 256;
        (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
        if (dev >= 0 && dev < 64) cu_count[dev] = n_cu;
    }
    const void *kernel = fused_variant(rows, bytes);
    static bool asked[2][9][64];
    if (dev >= 0 && dev < 64 && !asked[bytes][rows][dev]) {
        const hipError_t err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFuseLdsMax);
        if (err != hipSuccess) {
            set_error("glif3_simulate_fwd: cannot reserve %zu bytes of LDS: %s", kFuseLdsMax, hipGetErrorString(err));
            return BMTK_E_LAUNCH;
        }
        asked[bytes][rows][dev] = true;
    }
    FusedLaunch q{};
    const int per_cu = s.fuse_wg_per_cu > 0 ? s.fuse_wg_per_cu : 1;
    const int64_t cap = (int64_t)n_cu * per_cu;
    // A network with fewer groups than the chip has wavefronts: several share a group, so that its run of synapses is not
    // one wavefront's chain of dependent turns (1,500 neurons x 8 trials, 188 groups of 3,200 synapses: 14.9 -> 7.2 us per
    // step; no more of them than the run has blocks: 2,000 x 32, two blocks a group: 6.3 us alone, 8.3 with four)
    const int max_team = s.fuse_max_team > 0 ? s.fuse_max_team : kFuseWaves;
    q.team = 1;
    while (q.team < kFuseWaves && q.team * 2 <= max_team && n_groups * q.team * 2 <= cap * kFuseWaves) q.team *= 2;
    const int64_t teams = kFuseWaves / q.team;  // of a workgroup
    q.n_main = (int)(q.team > 1 ? (n_groups + teams - 1) / teams : n_groups < cap ? n_groups : cap);
    q.H = L + 4;
    q.Lr = L + 2;
    q.n_w32 = n_w32;
    q.unit = ldexp(1.0, -32 - s.sum_shift);
    q.shift = s.fuse_shift;
    q.n_in_words = (int)n_in_words;
    // (whatever this call's lists hold: repeats of an earlier call's lists may still be under way)
    q.use_ring = n_in > 0 ? 1 : 0;
    if (s.spike_bits && rows * batch != kWave) {
        // (groups that do not fill a word add their bits to words they share)
        const int64_t words = n_steps * s.spike_bits_stride;
        const int64_t blocks = (words + kBlock - 1) / kBlock;
        hipLaunchKernelGGL(zero_bits_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0, stream, s.spike_bits, words);
    }
    if (s.in_again && has_inp && step0 >= 1 && n_in_words > 0) {
        const dim3 grid((unsigned)((n_in_words + kBlock - 1) / kBlock));
        if (bytes)
            hipLaunchKernelGGL(input_again_kernel<true>, grid, dim3(kBlock), 0, stream, s, q, step0 - 1, rows);
        else
            hipLaunchKernelGGL(input_again_kernel<false>, grid, dim3(kBlock), 0, stream, s, q, step0 - 1, rows);
    }
    // sampled steps: (t + 1) % every == 0; row = how many of them the call has seen before
    auto probe_row = [&](int64_t t) -> int64_t {
        if (!s.probe_col || (t + 1) % s.probe_every != 0) return -1;
        return (t + 1) / s.probe_every - step0 / s.probe_every - 1;
    };
    // two steps per launch; a call's first launch folds nothing (the closing launch of the call before it did), an
    // odd step count leaves one step for the last regular launch, the closing launch folds what arrived in the
    // last step.  The maps of bytes alternate from launch to launch; a call begins and ends with map 0.
    int map = 0;
    for (int64_t k = 0; k <= n_steps;) {
        const bool closing = k == n_steps;
        q.n_sub = closing ? 0 : (int)(n_steps - k < 2 ? n_steps - k : 2);
        q.t0 = step0 + k;
        q.out_row = k;
        for (int i = 0; i < 3; ++i) {
            q.hist_row[i] = (int)((q.t0 + i - 1 + q.H) % q.H);
            q.ring_slot[i] = (int)((q.t0 + i - 1 + q.Lr) % q.Lr);
        }
        q.probe_row0 = closing ? -1 : probe_row(q.t0);
        q.probe_row1 = q.n_sub == 2 ? probe_row(q.t0 + 1) : -1;
        q.fold0 = k > 0 ? 1 : 0;
        q.in_bits = (has_inp && !closing && n_in_words > 0) ? 1 : 0;
        q.repeats = (s.in_repeat_ptr && !closing) ? 1 : 0;
        q.pending = (q.fold0 && q.t0 - 1 < s.rb_pend_until ? 1 : 0) | (q.n_sub == 2 && q.t0 < s.rb_pend_until ? 2 : 0);
        for (int i = 0; i < 2; ++i) q.pend_slot[i] = (int)((q.t0 + (L - 1) + i - 1) % (L - 1));
        q.map_read = map;
        q.map_write = bytes && (!closing || map == 1) ? 1 - map : -1;
        if (q.map_write >= 0) map = q.map_write;
        k += closing ? 1 : q.n_sub;
        bmtk_glif3_sim args = s;
        FusedLaunch launch = q;
        void *params[] = {&args, &launch};
        const hipError_t err = hipLaunchKernel(kernel, dim3((unsigned)q.n_main), dim3(kFuseBlock),
                                               params, lds, stream);
        if (err != hipSuccess) {
            set_error("glif3_simulate_fwd: launch failed: %s", hipGetErrorString(err));
            return BMTK_E_LAUNCH;
        }
    }
    if (n_steps > 0 && step0 < s.rb_pend_until) {
        const int64_t left = s.rb_pend_until - step0;
        const int slots = L - 1, slot_words = GLIF3_NREC * (int)s.n_neurons;
        const int count = (int)std::min<int64_t>(std::min<int64_t>(n_steps, left), slots);
        const int64_t words = (int64_t)batch * count * slot_words, blocks = (words + kBlock - 1) / kBlock;
        hipLaunchKernelGGL(clear_taken_kernel, dim3((unsigned)std::min<int64_t>(blocks, 4096)), dim3(kBlock), 0, stream, s.rb_ring, words, slot_words,
                           slots, (int)(step0 % slots), count);
    }
    BMTK_CHECK_LAUNCH("glif3_simulate_fwd");
    return BMTK_OK;
}

}  // namespace bmtk
