// Resident simulation of the trials of a batch: state in registers and the ring in LDS for the length of a call, as in
// resident.hip, with the workgroups of the chip divided among several trials.
//
// The trials of a batch do not touch one another.  `ways` of them run side by side in one cooperative launch, each on
// `groups` workgroups that exchange lists of the neurons that fired (fired_lists.hpp); launches follow one another until
// every trial has had its turn.  A workgroup owns `span` neurons of its trial, and its wavefronts divide the work as those of
// sim_resident_lists_kernel (resident.hip) do: a reader, a writer, the others pull; all but the reader update.  Round k
//   1. folds the arrivals of slot k-1 (LDS) into y1 and updates from registers; the writer publishes who fired, the reader
//      makes the lists of step k-1 and the trial's input events into a list of rows;
//   2. behind the workgroup's meeting, adds its own segment of every listed row (rows sorted by target, segment bounds in a
//      table) to its ring slice.  A row's segment is read by `1 << team_shift` neighbouring lanes: with few workgroups to a
//      trial a segment holds tens of synapses, which one lane would take one after the other.
// Neither state nor arrival sums cross the memory system, and of the table only the segments of rows that fired.
//
// Sums are exact and independent of the order: 64-bit fixed point as in the fused batched driver, or 32-bit whole numbers where the
// weights allow them (rb_whole, half the room; an integer addition in LDS costs 28 clocks per wavefront where a float's costs 194).  Slot t-1 is folded and cleared before the
// spikes of step t-1 are added, so that ring_slots - 1 slots suffice: 160 bytes of LDS per neuron and trial at delays of
// up to five steps with 64-bit sums for all four receptors.  Behind a call the arrivals still ahead wait in rb_ring, trial by trial.
//
// Where that saves launches a neuron has sums only for the receptors that some synapse of it ends on (rb_cells): of four ports the cells
// of a population mostly use two, which is 80 bytes, and with two neurons to a thread (1088 to 1920 a workgroup) twice the
// trials run side by side.  The first two sums of every neuron are planes over the span (the fold reads them without bank
// conflicts), the rarer third and fourth stand behind; a record names its cell, so that the pull asks nothing.  A step then takes 1.2 to 1.4
// times as long: update 0.7 -> 1.4 us (the issue of two neurons' instructions), the pull's chain as before with twice the
// synapses in a segment.  At 2.2 sums a neuron, 200 steps: 51,978 x 32 in 4 launches of 32 workgroups a trial 5.85 ms, in 8 of 63 8.03;
// 20,011 x 20 in one launch 1.47, in two 1.74.  230,924 x 8 have room for two trials with 32-bit sums only.
//
// What bounds it: a step is a chain of dependent loads (lists, segment bounds, synapses), 2.5 us at the smallest sizes,
// whatever the number of trials side by side; then the table's segments, which every trial reads for itself.  Per step and
// launch, ballots and a grid barrier per trial -> lists, in turn in one process: 230,924 neurons x 4 6.0 -> 5.6 us, 20,011 x 20 4.5 ->
// 4.3, 3,001 x 12 3.0 -> 2.8, 400,123 x 1 with 1,024 spikes a step 10.5 -> 7.6; 51,978 x 32, which reads 18 synapses a segment for 243
// rows of each of four trials, as before.
// At tens of Hz, where steps are crowded (see resident.hip), the ballots were the faster exchange still: 60,000 x 4 at 24 / 45 Hz 12.3 /
// 20.3 us a step against 14.9 / 24.8 (15.1 / 35.7 with every list of more than 19 neurons crowded), 230,924 x 2 at 28 Hz 56 against 62;
// at 19 Hz 60,000 x 4 take 5.4 against 10.0.
//
// One trial of more neurons than the compute units have threads (resident.hip ends at 1024 to a workgroup) runs here with two
// neurons to a thread and its ring in floats, 80 bytes a neuron: 400,123 neurons, 72 M synapses, 23 -> 6.6 us per step against
// a launch per step with an atomic per event.  What it is short of are the 128 vector
// registers a thread has: 84 hold two neurons.  Addresses and products worked out once for all steps spill
// half of them to memory, hence the opaque thread numbers below.
#include <math.h>
#include <stdlib.h>

#include <type_traits>

#include "fired_lists.hpp"
#include "glif3_update.hpp"
#include "pull_common.hpp"
#include "sim_internal.hpp"

namespace bmtk {

constexpr int kRbBlock = 1024;
constexpr int kRbWaves = kRbBlock / kWave;
constexpr int kRbReader = kRbWaves - 1, kRbWriter = kRbReader - 1;  // wavefronts with a part of their own, see resident.hip
constexpr int kRbPullThreads = kRbWriter * kWave;
constexpr unsigned kRbMaxSpin = 4000000u; // looks in vain before giving up (seconds)
// (two neurons to a thread and their sums leave registers for four: with six the compiler spills)
constexpr int kRbTogether = 6;            // synapses a lane has in flight (20,011 x 20, 8 lanes to 33: 4 of them 9.6 us per step, 6 9.3)
constexpr int kRbEvents = 8;              // input events a lane of the reader asks for ahead

struct RbLaunch {
    int64_t step0;
    int n_steps;
    int trial0, trials;   // trials of this launch
    int slots;            // of the ring slice: ring_slots - 1
    int words;            // ballot words of a trial
    int has_events;
    double unit;          // of the sums
    int down;             // whole numbers: bits that a kept sum is shifted by (Kept)
};

__device__ __forceinline__ unsigned rb_load(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Where the sums of a neuron's receptor r stand within a slot of its workgroup's slice.  `word` is rb_cells': bits 0..3 the
// receptors that some synapse of the neuron ends on, above them where its third sum stands among the workgroup's.
__host__ __device__ inline int rb_cell(unsigned word, int r, int place, int span)
{
    const unsigned below = word & ((1u << r) - 1u);
    const int j = (int)((below & 1u) + (below >> 1 & 1u) + (below >> 2 & 1u));
    return j < 2 ? j * span + place : 2 * span + (int)(word >> GLIF3_NREC) + j - 2;
}

struct __attribute__((packed, aligned(4))) RbBounds {
    uint32_t lo, hi;
};

// kPer: neurons per thread; with two, the threads of the reader own none.  Sum: what the ring holds, 64-bit fixed point
// (from_fixed), or floats where a workgroup's neurons are too many for that (batch 1): fp32 atomics into device memory are what
// it then takes the place of, or 32-bit whole numbers where every weight is a whole multiple of one power of two and all that
// reaches a neuron in a step stays below 2^31 of it (rb_whole): the same sums, bit for bit, in half the room, which is what decides how
// many trials share a launch (230,924 x 8, 100 steps: 5.38 -> 3.40 ms; 10,000 x 8, 200 steps in one launch either way: 0.74 -> 0.59).  kAllSums: every neuron has all four sums, in planes (no rb_cells); at 1,000 neurons and less to a
// workgroup the fold's selections cost 0.1 us a step, so that few sums are for where they save launches.  kSave: potentials and step flags of every step go to rb_save_*, trial by trial; by_step_kernel
// puts them in their order.  kReaderOwns: spans above 960 with a neuron to a thread.
template <int kPer, typename Sum, bool kAllSums, bool kSave, bool kReaderOwns>
__global__ __launch_bounds__(kRbBlock) void sim_resident_batch_kernel(bmtk_glif3_sim s, RbLaunch q)
{
    constexpr bool kFixed = sizeof(Sum) == 8, kWhole = std::is_same<Sum, unsigned>::value;
    using Kept = typename std::conditional<std::is_same<Sum, float>::value, float, unsigned long long>::type;   // of rb_ring
    constexpr int kTogether = kPer > 1 ? 4 : kRbTogether;
    constexpr int kOwners = kRbReader * kWave;  // with two neurons to a thread: threads that own tid, tid + kOwners
    extern __shared__ unsigned long long rb_lds[];  // ring slice [slots][cells], then rb_list words for rows
    __shared__ int go_on[2];  // by the round, as rows_l is: a slot is written again only after a meeting behind all reads of it
    __shared__ unsigned rows_l[2], crowd_l[3], done_l, updated_l, listed_l;  // rows of a round, ..
    __shared__ unsigned fired_n[2];                  // how many fired in this step and the one before
    __shared__ unsigned short fired_l[kListMax + 1]; // the first of them, counted within the span
    const int tid = threadIdx.x, lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int span = s.rb_span, G = s.rb_groups;
    // an XCD (block number mod 8) gets consecutive workgroups, hence a trial as few XCDs as hold it
    const int per_xcd = (int)gridDim.x >> 3;
    const int at = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (at >= q.trials * G) return;
    const int way = at / G, g = at - way * G;
    const int trial = q.trial0 + way;
    const int n = (int)s.n_neurons, batch = s.batch, S = q.slots;
    const int e0 = g * span;
    const int mine = min(span, n - e0);
    const int64_t ne = (int64_t)n * batch;
    auto place = [&](int u) __attribute__((always_inline)) {
        int me = tid;
        if (kPer > 1) asm volatile("" : "+v"(me));  // (addresses and products of it, kept for all steps, would push the state out)
        return kPer == 1 ? me : (me < kOwners ? u * kOwners + me : span);
    };  // in the workgroup's span
    auto owns = [&](int u) __attribute__((always_inline)) { return place(u) < mine; };
    auto element = [&](int u) { return (int64_t)(e0 + (owns(u) ? place(u) : 0)) * batch + trial; };
    // cells of a slot: two planes of the workgroup's neurons, then the third and fourth sums of those that have any
    const int cells = kAllSums ? GLIF3_NREC * span : 2 * span + s.rb_extra;
    Sum *ring_l = reinterpret_cast<Sum *>(rb_lds);
    unsigned *rows = reinterpret_cast<unsigned *>(ring_l + (size_t)S * cells);  // [2][row_cap], a place per lane behind
    const unsigned row_cap = ((unsigned)s.rb_list - kWave) / 2u;
    unsigned *abort_word = s.res_sync + 1;
    const unsigned spin_limit = s.res_spin_limit ? s.res_spin_limit : kRbMaxSpin;
    unsigned long long *lists = lists_in(s.res_sync);
    unsigned long long *hist = reinterpret_cast<unsigned long long *>(s.rb_hist) + (int64_t)way * kListRows * (q.words + 1);
    auto lists_of = [&](int k) { return ListRow{lists + (k & (kListRows - 1)) * kListRowWords, way * G, G}; };
    auto ballots_of = [&](int k) { return hist + (int64_t)(k & (kListRows - 1)) * (q.words + 1); };
    if (tid == 0) {
        go_on[0] = rb_load(abort_word) == 0u;
        rows_l[0] = rows_l[1] = done_l = updated_l = listed_l = fired_n[0] = fired_n[1] = 0u;
    }
    __syncthreads();
    if (!go_on[0]) return;

    // the arrivals that the call before left; some slots' are asked for together, before the state takes the registers
    auto cell_of = [&](unsigned word, int r, int at) __attribute__((always_inline)) { return kAllSums ? r * span + at : rb_cell(word, r, at, span); };
    auto from_kept = [&](Kept v) __attribute__((always_inline)) -> Sum {
        if constexpr (kWhole)
            return (Sum)((long long)v >> q.down);
        else
            return v;
    };
    auto to_kept = [&](Sum v) __attribute__((always_inline)) -> Kept {
        if constexpr (kWhole)
            return (Kept)((long long)(int)v << q.down);
        else
            return v;
    };
    Kept *const ring_g = reinterpret_cast<Kept *>(s.rb_ring) + (int64_t)trial * S * GLIF3_NREC * n + e0;  // (all receptors' planes)
    unsigned sums[kPer]{};  // a neuron's word of rb_cells
#pragma unroll
    for (int u = 0; u < kPer; ++u)
        if (owns(u)) sums[u] = kAllSums ? 15u : s.rb_cells[e0 + place(u)];
    for (int c = tid; c < S * cells; c += kRbBlock) ring_l[c] = (Sum)0;
    __syncthreads();
    constexpr int kSlots = kPer > 1 ? 2 : 4;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        if (!owns(u)) continue;
#pragma unroll 1
        for (int k = 0; k < S; k += kSlots) {
            Kept v[kSlots * GLIF3_NREC];
#pragma unroll
            for (int j = 0; j < kSlots * GLIF3_NREC; ++j)
                if (k + j / GLIF3_NREC < S && (sums[u] >> j % GLIF3_NREC & 1u)) v[j] = ring_g[((int64_t)k * GLIF3_NREC + j) * n + place(u)];
#pragma unroll
            for (int j = 0; j < kSlots * GLIF3_NREC; ++j)
                if (k + j / GLIF3_NREC < S && (sums[u] >> j % GLIF3_NREC & 1u))
                    ring_l[(k + j / GLIF3_NREC) * cells + cell_of(sums[u], j % GLIF3_NREC, place(u))] = from_kept(v[j]);
        }
    }
    Glif3Elem st[kPer]{};
    Glif3Prop p[kPer]{};
    float I[kPer]{};
#pragma unroll
    for (int u = 0; u < kPer; ++u)
        if (owns(u)) {
            const int i = e0 + place(u);
            const int64_t col = s.class_id ? (int64_t)s.class_id[i] : (int64_t)i;
            p[u].load(s.prop, s.prop_stride, col);
            glif3_load(st[u], s.V, s.asc, s.y1, s.y2, s.ref, ne, element(u));
            I[u] = s.i_ext ? s.i_ext[element(u)] : 0.0f;
        }
    __syncthreads();  // (the ring slice is there, and go_on is written again below)

    const int n_steps = q.n_steps;
    int slot = (int)((q.step0 - 1 + S) % S);  // of step k-1
    const float zero[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto fold = [&](int at_slot) __attribute__((always_inline)) {
        if (kPer > 1) asm volatile("" : "+s"(at_slot));
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            if (!owns(u)) continue;
            Sum *const row = ring_l + (size_t)at_slot * cells;
            auto take = [&](int cell) __attribute__((always_inline)) {
                const Sum v = row[cell];
                row[cell] = (Sum)0;
                if constexpr (kFixed)
                    return from_fixed(v, q.unit);
                else if constexpr (kWhole)
                    return (float)(int)v * (float)q.unit;
                else
                    return v;
            };
            if constexpr (kAllSums) {
#pragma unroll
                for (int r = 0; r < GLIF3_NREC; ++r) st[u].y1[r] = st[u].y1[r] + take(r * span + place(u)) * p[u].psc0[r];
                continue;
            }
            unsigned word = sums[u];
            if (kPer > 1) asm volatile("" : "+v"(word));
            float a[GLIF3_NREC];
            a[0] = take(place(u));
            a[1] = take(span + place(u));
            a[2] = a[3] = 0.0f;
            const int third = 2 * span + (int)(word >> GLIF3_NREC);
            if (__popc(word & 15u) > 2) a[2] = take(third);
            if ((word & 15u) == 15u) a[3] = take(third + 1);
            // (a sum for every receptor used, in their order: receptor r has as many before it as bits are set below bit r)
#pragma unroll
            for (int r = 0; r < GLIF3_NREC; ++r) {
                const unsigned below = word & ((1u << r) - 1u);
                float x = a[0];
                if (r > 0) x = below ? a[1] : x;
                if (r > 1) x = (below & (below - 1u)) ? a[2] : x;
                if (r > 2) x = below == 7u ? a[3] : x;
                x = (word >> r & 1u) ? x : 0.0f;
                st[u].y1[r] = st[u].y1[r] + x * p[u].psc0[r];
            }
        }
    };
    auto spike_bit = [&](int k, int i) {  // (a word of the output holds several trials)
        const int64_t e = (int64_t)i * batch + trial;
        __hip_atomic_fetch_or(reinterpret_cast<unsigned long long *>(s.spike_bits) + (int64_t)k * s.spike_bits_stride + (e >> 6),
                              1ull << (e & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // fold and update of step step0 + k (the fold alone behind the last step)
    unsigned fired = 0u;  // bit u: this thread's u-th neuron
    float potential[kPer]{};
    auto save = [&](int k, int u, bool spike, int ref_before) __attribute__((always_inline)) {
        if (!kSave) return;
        const int64_t to = ((int64_t)trial * n_steps + k) * n + e0 + place(u);
        s.rb_save_v[to] = st[u].V;
        s.rb_save_flags[to] = (uint8_t)((spike ? BMTK_F_SPIKE : 0) | (ref_before == 0 ? BMTK_F_INTEGRATING : 0) |
                                        (ref_before > 0 && st[u].ref == 0 ? BMTK_F_RESET : 0));
    };
    auto update = [&](int k) __attribute__((always_inline)) {
        if (k > 0) fold(slot);
        if (k == n_steps) return;
        float h = s.h;
        if (kPer > 1) asm volatile("" : "+s"(h));  // (h times a neuron's propagators: not to be worked out once for all steps)
        fired = 0u;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            if (!owns(u)) continue;
            bool spike;
            if constexpr (kPer > 1) {
                potential[u] = glif3_potential(st[u], p[u], I[u]);
                spike = glif3_fires(st[u], p[u], potential[u]);
            } else {
                float frac;
                const int ref_before = st[u].ref;
                spike = glif3_update(st[u], p[u], h, zero, I[u], &frac);
                save(k, u, spike, ref_before);
            }
            if (spike) {
                fired |= 1u << u;
                const unsigned to = atomicAdd(&fired_n[k & 1], 1u);
                if (to < kListMax) fired_l[to] = (unsigned short)place(u);
            }
        }
    };
    // Two neurons to a thread: the second half of their update, which nobody waits for, while the bounds of a thread's first row are on their
    // way (with one, the whole update hides them): 51,978 x 32 5.61 -> 5.46 ms for 200 steps, 20,011 x 20 1.61 -> 1.58, 400,123 x 1 2.03 -> 2.00 for 300.
    auto finish = [&](int k) __attribute__((always_inline)) {
        float h = s.h;
        asm volatile("" : "+s"(h));
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            if (!owns(u)) continue;
            const int ref_before = st[u].ref;
            const bool spike = (fired >> u) & 1u;
            glif3_finish(st[u], p[u], h, zero, potential[u], spike);
            save(k, u, spike, ref_before);
        }
    };
    // Writer, before the workgroup meets: the list, where it holds the neurons, then their bits in the output.
    auto write = [&](int k) __attribute__((always_inline)) {
        ListWrite list;
        list.read(fired_l);
        const unsigned m = fired_n[k & 1];
        const int i = lane_here();
        const int id = fired_l[min((unsigned)i, kListMax)];
        if (m <= kListMax) {
            list.publish(lists_of(k), g, list_tag(k), m);
            if (s.spike_bits && (unsigned)i < m) spike_bit(k, e0 + id);
        }
        if (lane == 0) fired_n[(k + 1) & 1] = 0u;
    };
    // All, behind the meeting: a volley's ballots, which have to have arrived before the list says that they are to be read.
    auto volley = [&](int k) __attribute__((always_inline)) {
        if (fired_n[k & 1] <= kListMax) return;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const bool spike = (fired >> u) & 1u;
            const unsigned long long m = __ballot(spike);
            const int i = e0 + place(u);
            if (lane == 0 && place(u) < span && i < n)
                __hip_atomic_store(ballots_of(k) + (i >> 6), m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (spike && s.spike_bits) spike_bit(k, i);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (wave == kRbWriter) {
            ListWrite list;
            list.read(fired_l);
            list.publish(lists_of(k), g, list_tag(k), fired_n[k & 1]);
        }
    };

    // this workgroup's segment of a row into the slots behind `slot`, lane `part` of `step`
    const int ts = s.rb_team_shift;
    const uint32_t *__restrict__ seg = s.rb_seg + g;
    const uint2 *__restrict__ table = reinterpret_cast<const uint2 *>(s.rb_packed);
    const unsigned seg_stride = (unsigned)G + 1u;
    auto row_bounds = [&](unsigned row) __attribute__((always_inline)) { return *reinterpret_cast<const RbBounds *>(seg + (size_t)row * seg_stride); };
    auto add_segment = [&](RbBounds b, unsigned part, unsigned step) __attribute__((always_inline)) {
        const unsigned q_lo = (unsigned)slot, q_wrap = q_lo - (unsigned)S;
        // (slot + delay) % slots = min(u, u - slots), u = slot + the record's upper byte; below it the cell
        auto add = [&](const uint2 sy, bool crowded) {
            const unsigned dq = sy.x >> 24;
            Sum *cell = ring_l + mad_u24(min(dq + q_lo, dq + q_wrap), (unsigned)cells, sy.x & 0xFFFFFFu);
            if constexpr (kFixed)
                atomicAdd(cell, to_fixed(__uint_as_float(sy.y)));
            else if constexpr (kWhole)
                atomicAdd(cell, sy.y);
            else if (!crowded)
                atomicAdd(cell, __uint_as_float(sy.y));
            else {
                // (where most lanes take part: a float atomic is worked off lane by lane, see resident.hip)
                unsigned *bits = reinterpret_cast<unsigned *>(cell);
                unsigned old = *bits;
                while (true) {
                    const unsigned seen = atomicCAS(bits, old, __float_as_uint(__uint_as_float(old) + __uint_as_float(sy.y)));
                    if (seen == old) break;
                    old = seen;
                }
            }
        };
        for (uint32_t at_p = b.lo + part; at_p < b.hi; at_p += kTogether * step) {
            uint2 sy[kTogether];
#pragma unroll
            for (int u = 0; u < kTogether; ++u)
                if (at_p + u * step < b.hi) sy[u] = table[at_p + u * step];
#pragma unroll
            for (int u = 0; u < kTogether; ++u)
                if (at_p + u * step < b.hi) add(sy[u], u == 0);
        }
    };
    // the input events of round k: rb_in_events[in_ptr[k] .. in_ptr[k + 1])
    const int64_t *in_ptr = q.has_events ? s.rb_in_ptr + (int64_t)trial * (n_steps + 1) : nullptr;
    // (a call's first step: the spikes of the step before were added by the call before it, and so were its events unless
    //  they are to be taken from this call's lists)
    auto with_events = [&](int k) { return in_ptr && (k > 0 || s.rb_late_events); };
    // The rows of round k: what fired in step k-1, and the input events handed over with it.  Where they are listed before the
    // update of step k (`ask` ahead of it), the bounds of a thread's first row are on their way meanwhile.
    // Events that the reader has no lanes for follow the listed rows (see resident.hip).
    unsigned listed = 0u, n_rows = 0u, at_row = 0u, n_more = 0u;
    const int32_t *more_events = nullptr;
    int32_t next_source = 0;
    RbBounds first_row{0u, 0u};
    auto ask = [&](int k) __attribute__((always_inline)) {
        unsigned me = (unsigned)tid;
        asm volatile("" : "+v"(me));
        listed = (unsigned)__builtin_amdgcn_readfirstlane((int)rows_l[k & 1]);
        const bool pulls = listed != kCrowded && wave != kRbWriter;
        n_rows = pulls ? listed & ~kMoreEvents : 0u;
        at_row = me >> ts;
        if (at_row < n_rows) first_row = row_bounds(rows[(k & 1) * row_cap + at_row]);
        n_more = 0u;
        if (pulls && (listed & kMoreEvents)) {
            const unsigned from = (unsigned)in_ptr[k] + kRbEvents * kWave;
            n_more = (unsigned)in_ptr[k + 1] - from;
            more_events = s.rb_in_events + from;
            if (at_row >= n_rows && at_row - n_rows < n_more) next_source = more_events[at_row - n_rows];
        }
    };
    auto pull = [&](int k) __attribute__((always_inline)) {
        const unsigned part = (unsigned)lane & ((1u << ts) - 1u), step = (unsigned)kRbPullThreads >> ts;
        const bool at_hand = at_row >= n_rows;
        while (at_row < n_rows) {
            const RbBounds b = first_row;
            at_row += step;
            if (at_row < n_rows) first_row = row_bounds(rows[(k & 1) * row_cap + at_row]);
            add_segment(b, part, 1u << ts);
        }
        if (n_more != 0u) {
            unsigned a = at_row - n_rows;
            if (!at_hand && a < n_more) next_source = more_events[a];
            while (a < n_more) {
                const int32_t source = next_source;
                a += step;
                if (a < n_more) next_source = more_events[a];
                add_segment(row_bounds((unsigned)n + (unsigned)source), part, 1u << ts);
            }
        }
    };
    auto pull_crowded = [&](int k) __attribute__((always_inline)) {
        const unsigned lo = with_events(k) ? (unsigned)in_ptr[k] : 0u, n_ev = with_events(k) ? (unsigned)in_ptr[k + 1] - lo : 0u;
        const int32_t *const events = s.rb_in_events + lo;
        const unsigned n_first = k > 0 ? min(n_ev, min((unsigned)kRbBlock, (unsigned)s.rb_list)) : 0u;
        if (k > 0)
            crowded_rows<kPer * kRbWaves>(
                lists_of(k - 1), list_tag(k - 1), span, ballots_of(k - 1), q.words, n_first,
                [&](unsigned i) { return (unsigned)n + (unsigned)events[i]; }, rows, (unsigned)s.rb_list, crowd_l, abort_word, spin_limit,
                [&](unsigned total) __attribute__((always_inline)) {
                    for (unsigned a = (unsigned)tid >> ts; a < total; a += (unsigned)kRbBlock >> ts)
                        add_segment(row_bounds(rows[a]), (unsigned)lane & ((1u << ts) - 1u), 1u << ts);
                });
        // (further events are left to pull; n_rows is 0)
        n_more = wave < kRbWriter ? n_ev - n_first : 0u;
        more_events = events + n_first;
        if (at_row < n_more) next_source = more_events[at_row];
    };
    // the pulls of round k are complete
    auto pulled = [&](int k) __attribute__((always_inline)) {
        while ((int)(load_lds(&done_l) - (unsigned)(k + 1) * kRbWriter) < 0) {}
    };

    auto store = [&]() __attribute__((always_inline)) {
        int64_t all = ne;
        asm volatile("" : "+s"(all));  // (its addresses are not those of the loads, kept all along)
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            if (owns(u)) glif3_store(st[u], s.V, s.asc, s.y1, s.y2, s.ref, all, element(u));
    };

    bool aborted = false;
    if (wave != kRbReader) {
        for (int k = 0; k <= n_steps; ++k) {  // (one round more than steps: the closing pull)
            const bool asked = kPer == 1 && load_lds(&listed_l) == (unsigned)k + 1u;  // (two neurons leave no registers for it)
            if (asked) ask(k);
            update(k);
            if (wave != kRbWriter) {
                count_lds(&updated_l);
            } else if (k < n_steps) {
                const unsigned all = (unsigned)(k + 1) * (kReaderOwns ? kRbReader : kRbWriter);
                while ((int)(load_lds(&updated_l) - all) < 0) {}
                write(k);
            }
            __syncthreads();  // the workgroup meets: every slot k-1 is folded, the rows of the round are there
            if (!go_on[k & 1]) {
                aborted = true;
                break;
            }
            if (k < n_steps) volley(k);
            if (!asked) ask(k);
            if (kPer > 1 && k < n_steps) finish(k);
            if (listed == kCrowded) pull_crowded(k);
            pull(k);
            slot = slot + 1 == S ? 0 : slot + 1;
            if (wave != kRbWriter) count_lds(&done_l);
            pulled(k);
        }
        store();
    } else {
        ListLook seen;
        bool lost = false;  // given up
        unsigned failed = 0u;
        int opaque_zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(opaque_zero));
        // the input events of the round in hand, the first of them on their way
        unsigned ev_lo = with_events(0) ? (unsigned)in_ptr[0] : 0u, ev_hi = with_events(0) ? (unsigned)in_ptr[1] : 0u;
        unsigned next_lo = 0u, next_hi = 0u;
        if (in_ptr) next_lo = (unsigned)in_ptr[1], next_hi = (unsigned)in_ptr[min(2, n_steps + 1)];
        int32_t ev[kRbEvents] = {};
        auto ask_events = [&]() __attribute__((always_inline)) {
            const unsigned n_ev = ev_hi - ev_lo, me = (unsigned)lane_here();
            const int32_t *const from = s.rb_in_events + ev_lo;
#pragma unroll
            for (int i = 0; i < kRbEvents; ++i) {
                if ((unsigned)(i * kWave) >= n_ev) break;
                if (i * kWave + me < n_ev) ev[i] = from[i * kWave + me];
            }
        };
        ask_events();
        // one more look in vain: false when it is time to give up
        auto again = [&]() __attribute__((always_inline)) -> bool {
            if (++failed > spin_limit) __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return failed <= spin_limit && rb_load(abort_word) == 0u;
        };
        for (int k = 0; k <= n_steps; ++k) {
            if (kReaderOwns) {
                if (k > 0) pulled(k - 1);
                update(k);
                count_lds(&updated_l);
            }
            seen.none();
            failed = 0u;
            if (k > 0) {
                __builtin_amdgcn_s_sleep(8);  // (see resident.hip)
                while (!lost && !seen.look(lists_of(k - 1), list_tag(k - 1))) lost = !again();
            }
            if (!lost) {
                const unsigned me = (unsigned)lane_here(), spare = 2u * row_cap + me, to = (unsigned)(k & 1) * row_cap, n_ev = ev_hi - ev_lo;
                const unsigned n_listed = min(n_ev, (unsigned)(kRbEvents * kWave));
                const unsigned total = rows_from_lists(seen, lists_of(k - 1), list_tag(k - 1), span, rows, to, row_cap, spare, n_listed, again, lost);
                if (total != kCrowded) {
#pragma unroll
                    for (int i = 0; i < kRbEvents; ++i) {
                        if ((unsigned)(i * kWave) >= n_ev) break;
                        const unsigned a = i * kWave + me;
                        int32_t source = ev[i];
                        asm volatile("" : "+v"(source));  // (not looked at ahead of the lists)
                        rows[a < n_ev ? to + total + a : spare] = (unsigned)n + (unsigned)source;
                    }
                }
                if (lane == 0) {
                    rows_l[k & 1] = total == kCrowded ? kCrowded : (total + n_listed) | (n_ev > n_listed ? kMoreEvents : 0u);
                    if (!lost) store_lds(&listed_l, (unsigned)k + 1u);
                }
            }
            if (lane == 0) go_on[k & 1] = !lost;
            // vmcnt(0): nothing is on its way here, and with that said the compiler does not wait for loads below before it
            // uses their registers again
            __builtin_amdgcn_s_waitcnt(0x0F70);
            ev_lo = next_lo;
            ev_hi = (unsigned)__builtin_amdgcn_readfirstlane((int)next_hi);
            __syncthreads();
            if (!go_on[k & 1]) {
                aborted = true;
                break;
            }
            if (in_ptr) {
                next_lo = ev_hi;
                next_hi = (unsigned)in_ptr[min(k + 3, n_steps + 1) + opaque_zero];
                if (k < n_steps) ask_events();
            }
            if (k < n_steps) volley(k);
            if (rows_l[k & 1] == kCrowded) pull_crowded(k);
            slot = slot + 1 == S ? 0 : slot + 1;
        }
        if (kReaderOwns && !aborted) pulled(n_steps);
        if (kReaderOwns) store();
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        if (!owns(u)) continue;
        unsigned word = sums[u];
        asm volatile("" : "+v"(word));  // (what the reads of the ring worked out from it is not kept for this)
#pragma unroll 1
        for (int k = 0; k < S; ++k)
#pragma unroll
            for (int r = 0; r < GLIF3_NREC; ++r)
                if (word >> r & 1u) ring_g[(int64_t)(k * GLIF3_NREC + r) * n + place(u)] = to_kept(ring_l[k * cells + cell_of(word, r, place(u))]);
    }
}

// Potentials and flags of 64 neurons and one step from the trials' own rows to the order of the record, [step][neuron][trial].
// A trial's lane writing its place there itself would store 4 bytes of every 4 * batch, each trial from another XCD: the
// detour is one more read and write of the record, 0.17 ms for 40 steps of 51,978 x 32 (332 MB).
constexpr int kByStepPitch = kWave + 1;
__global__ __launch_bounds__(kBlock) void by_step_kernel(const float *__restrict__ v, const uint8_t *__restrict__ flags, int batch,
                                                         int n_steps, int n, float *__restrict__ out_v, uint8_t *__restrict__ out_flags)
{
    __shared__ float v_l[kWave * kByStepPitch];
    __shared__ uint8_t flags_l[kWave * kByStepPitch];
    const int n0 = (int)blockIdx.x * kWave, k = (int)blockIdx.y, mine = min(kWave, n - n0);
    for (int c = (int)threadIdx.x; c < batch * kWave; c += kBlock) {
        const int b = c / kWave, j = c % kWave;
        if (j >= mine) continue;
        const int64_t from = ((int64_t)b * n_steps + k) * n + n0 + j;
        v_l[b * kByStepPitch + j] = v[from];
        flags_l[b * kByStepPitch + j] = flags[from];
    }
    __syncthreads();
    const int64_t to = ((int64_t)k * n + n0) * batch;
    for (int c = (int)threadIdx.x; c < mine * batch; c += kBlock) {
        const int j = (int)((unsigned)c / (unsigned)batch), b = c - j * batch;
        out_v[to + c] = v_l[b * kByStepPitch + j];
        out_flags[to + c] = flags_l[b * kByStepPitch + j];
    }
}

__global__ __launch_bounds__(kBlock) void rb_zero_bits_kernel(uint64_t *__restrict__ bits, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) bits[i] = 0ull;
}

// The input events of a run of steps, apart by trial: one workgroup per step counts the step's events of every trial, a
// second pass puts their sources where the running sums of those counts say.
template <bool kFill>
__global__ __launch_bounds__(kBlock) void events_by_trial_kernel(int batch, int64_t step0, int64_t n_steps, int late,
                                                                 const int64_t *__restrict__ in_ptr, const int32_t *__restrict__ in_events,
                                                                 int32_t *__restrict__ counts, const int64_t *__restrict__ first,
                                                                 int32_t *__restrict__ sources)
{
    __shared__ unsigned next[kWave];
    const int64_t k = blockIdx.x, t = step0 + k;
    if (threadIdx.x < (unsigned)batch) next[threadIdx.x] = kFill ? (unsigned)first[threadIdx.x * n_steps + k] : 0u;
    __syncthreads();
    const int64_t p0 = t >= 0 ? in_ptr[t] : 0, p1 = t >= 0 ? in_ptr[t + 1] : 0;
    for (int64_t p = p0 + threadIdx.x; p < p1; p += kBlock) {
        const unsigned ev = (unsigned)in_events[p], source = ev / (unsigned)batch;
        // (late: of the step before the call an id once, of the call's last step its occurrences after the first)
        const bool again = p > p0 && (unsigned)in_events[p - 1] == ev;
        if (late && (k == 0 ? again : k == n_steps - 1 && !again)) continue;
        const unsigned at = atomicAdd(&next[ev - source * (unsigned)batch], 1u);
        if (kFill) sources[at] = (int32_t)source;
    }
    __syncthreads();
    if (!kFill && threadIdx.x < (unsigned)batch) counts[threadIdx.x * n_steps + k] = (int32_t)next[threadIdx.x];
}

int simulate_resident_batch(const bmtk_glif3_sim &s, int64_t step0, int64_t n_steps, hipStream_t stream)
{
    const int batch = s.batch, S = s.ring_slots - 1, span = s.rb_span, G = s.rb_groups, W = s.rb_ways;
    const int64_t n = s.n_neurons;
    BMTK_REQUIRE(batch >= 1 && batch <= kWave, "glif3_simulate_fwd: resident trials come in batches of 1 to 64");
    const bool wide = span > kRbBlock;
    BMTK_REQUIRE(span >= kWave && span % kWave == 0 && span <= 2 * kRbReader * kWave && G == (n + span - 1) / span,
                 "glif3_simulate_fwd: rb_span must be a multiple of 64 up to 1920 and rb_groups ceil(n_neurons / rb_span)");
    BMTK_REQUIRE(wide || batch > 1, "glif3_simulate_fwd: a single trial is resident in spans above 1024 here, in shorter ones by res_span");
    BMTK_REQUIRE(s.rb_cells ? batch > 1 && s.rb_extra >= 0 && s.rb_extra <= 2 * span : s.rb_extra == 2 * span && (batch == 1 || !wide || s.rb_whole),
                 "glif3_simulate_fwd: rb_extra must lie in 0..2 * rb_span with rb_cells (batches; spans above 1024 need it or rb_whole) and be 2 * rb_span without");
    BMTK_REQUIRE(s.sum_shift >= 0 && s.sum_shift <= BMTK_SUM_SHIFT_MAX, "glif3_simulate_fwd: sum_shift must lie in 0..BMTK_SUM_SHIFT_MAX");
    const bool whole = s.rb_whole != 0;
    // (a kept sum is 33 + sum_shift - rb_whole bits further up than a 32-bit one, which 64 bits hold up to 32)
    BMTK_REQUIRE(!whole || (s.rb_whole > s.sum_shift && s.rb_whole <= 33 + s.sum_shift && batch > 1 && !s.rb_cells),
                 "glif3_simulate_fwd: rb_whole must be 0 or lie in sum_shift + 1..sum_shift + 33 and is for batches without rb_cells");
    BMTK_REQUIRE(W >= 1 && W <= batch && s.rb_team_shift >= 0 && s.rb_team_shift <= 6 && s.rb_list >= kWave,
                 "glif3_simulate_fwd: rb_ways must lie in 1..batch, rb_team_shift in 0..6, rb_list from 64 on");
    BMTK_REQUIRE(s.rb_seg && s.rb_packed && s.rb_ring && s.rb_hist && s.res_sync, "glif3_simulate_fwd: resident trials need rb_* and res_sync");
    BMTK_REQUIRE(s.delay_offset == 0 && (s.delay_bits == 0 || s.delay_bits == 6), "glif3_simulate_fwd: resident trials need delay_offset 0 and the standard packing");
    const bool save = s.save_v != nullptr;
    BMTK_REQUIRE(!s.probe_col && !s.spike_count, "glif3_simulate_fwd: resident trials take no probes and keep no spike record");
    BMTK_REQUIRE(!save || (batch > 1 && s.rb_save_v && s.rb_save_flags && n_steps <= 65535),
                 "glif3_simulate_fwd: resident trials keep the per-step record of batches, up to 65535 steps a call, with rb_save_v and rb_save_flags");
    BMTK_REQUIRE((s.rb_in_ptr == nullptr) == (s.rb_in_events == nullptr), "glif3_simulate_fwd: rb_in_ptr and rb_in_events go together");
    BMTK_REQUIRE(n_steps < (1ll << 30) && n + s.n_inputs < (1ll << 24), "glif3_simulate_fwd: too many steps or sources for resident trials");
    const size_t lds = (size_t)S * (2 * span + s.rb_extra) * (batch == 1 || whole ? sizeof(float) : sizeof(unsigned long long)) + (size_t)s.rb_list * sizeof(unsigned);
    BMTK_REQUIRE(lds + 256u <= kResLdsBytes, "glif3_simulate_fwd: the ring slice of resident trials does not fit in LDS");
    RbLaunch q{};
    q.step0 = step0;
    q.n_steps = (int)n_steps;
    q.slots = S;
    q.words = (int)((n + kWave - 1) / kWave);
    q.has_events = s.rb_in_ptr != nullptr;
    q.unit = ldexp(1.0, whole ? 1 - s.rb_whole : -32 - s.sum_shift);
    q.down = whole ? 33 + s.sum_shift - s.rb_whole : 0;
    BMTK_REQUIRE((wide ? 2 * kRbReader * kWave : kRbBlock) * (int64_t)kListGroups >= n, "glif3_simulate_fwd: more neurons than resident trials can hold");
    using Fixed = unsigned long long;
    auto address = [](auto *k) { return reinterpret_cast<const void *>(k); };
    const bool owns = span > kRbReader * kWave, few = s.rb_cells != nullptr;
    const void *const kernels[2][2][2] = {  // one neuron to a thread: few sums, record, neurons of the reader's
        {{address(sim_resident_batch_kernel<1, Fixed, true, false, false>), address(sim_resident_batch_kernel<1, Fixed, true, false, true>)},
         {address(sim_resident_batch_kernel<1, Fixed, true, true, false>), address(sim_resident_batch_kernel<1, Fixed, true, true, true>)}},
        {{address(sim_resident_batch_kernel<1, Fixed, false, false, false>), address(sim_resident_batch_kernel<1, Fixed, false, false, true>)},
         {address(sim_resident_batch_kernel<1, Fixed, false, true, false>), address(sim_resident_batch_kernel<1, Fixed, false, true, true>)}}};
    const void *const whole_kernels[2][2] = {  // record, neurons of the reader's
        {address(sim_resident_batch_kernel<1, unsigned, true, false, false>), address(sim_resident_batch_kernel<1, unsigned, true, false, true>)},
        {address(sim_resident_batch_kernel<1, unsigned, true, true, false>), address(sim_resident_batch_kernel<1, unsigned, true, true, true>)}};
    const void *kernel = whole && !wide ? whole_kernels[save][owns]
                         : whole        ? (save ? address(sim_resident_batch_kernel<2, unsigned, true, true, false>)
                                                : address(sim_resident_batch_kernel<2, unsigned, true, false, false>))
                         : batch == 1   ? address(sim_resident_batch_kernel<2, float, true, false, false>)
                         : !wide    ? kernels[few][save][owns]
                         : save     ? address(sim_resident_batch_kernel<2, Fixed, false, true, false>)
                                    : address(sim_resident_batch_kernel<2, Fixed, false, false, false>);
    hipError_t err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) {
        set_error("glif3_simulate_fwd: resident trials need %zu bytes of LDS: %s", lds, hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    const unsigned grid = 8u * (unsigned)((W * G + 7) / 8);
    int dev = 0, n_cu = 0, per_cu = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kRbBlock, lds);
    if ((int64_t)per_cu * n_cu < (int64_t)grid) {
        set_error("glif3_simulate_fwd: %u resident workgroups do not fit the device (%d compute units x %d)", grid, n_cu, per_cu);
        return BMTK_E_LAUNCH;
    }
    BMTK_REQUIRE(W * G <= kListGroups, "glif3_simulate_fwd: a launch of resident trials has at most 256 workgroups");
    if (s.spike_bits) {
        // (a spike is one bit in a word its trials share)
        const int64_t words = n_steps * s.spike_bits_stride, blocks = (words + kBlock - 1) / kBlock;
        hipLaunchKernelGGL(rb_zero_bits_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0, stream, s.spike_bits, words);
    }
    const char *plain = getenv("BMTK_AMD_PLAIN_LAUNCH");  // see simulate_resident
    for (int trial0 = 0; trial0 < batch; trial0 += W) {
        q.trial0 = trial0;
        q.trials = batch - trial0 < W ? batch - trial0 : W;
        // the lists of the launch before back to no step's
        const int64_t list_words = (int64_t)kListRows * kListRowWords;
        hipLaunchKernelGGL(rb_zero_bits_kernel, dim3((unsigned)((list_words + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream,
                           reinterpret_cast<uint64_t *>(lists_in(s.res_sync)), list_words);
        bmtk_glif3_sim copy = s;
        RbLaunch launch = q;
        void *args[] = {&copy, &launch};
        err = plain && plain[0] == '1' ? hipLaunchKernel(kernel, dim3(grid), dim3(kRbBlock), args, lds, stream)
                                       : hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(kRbBlock), args, (unsigned)lds, stream);
        if (err != hipSuccess) {
            set_error("glif3_simulate_fwd: launch of %u resident workgroups failed: %s", grid, hipGetErrorString(err));
            return BMTK_E_LAUNCH;
        }
    }
    if (save)
        hipLaunchKernelGGL(by_step_kernel, dim3((unsigned)((n + kWave - 1) / kWave), (unsigned)n_steps), dim3(kBlock), 0, stream,
                           s.rb_save_v, s.rb_save_flags, batch, (int)n_steps, (int)n, s.save_v, s.save_flags);
    BMTK_CHECK_LAUNCH("glif3_simulate_fwd");
    return BMTK_OK;
}

}  // namespace bmtk

namespace bmtk {

__global__ __launch_bounds__(kBlock) void receptors_used_kernel(int64_t nnz, const int32_t *__restrict__ indices, const uint8_t *__restrict__ receptors,
                                                                uint32_t *__restrict__ used)
{
    for (int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x; p < nnz; p += (int64_t)gridDim.x * kBlock) {
        const unsigned bit = 1u << (receptors[p] & 3u);
        uint32_t *const word = used + indices[p];
        // (nearly always there already: a look costs less than an atomic)
        if (!(__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit)) atomicOr(word, bit);
    }
}

__global__ __launch_bounds__(kBlock) void pack_cells_kernel(int64_t nnz, int span, const uint32_t *__restrict__ words, uint2 *__restrict__ packed)
{
    for (int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x; p < nnz; p += (int64_t)gridDim.x * kBlock) {
        const unsigned x = packed[p].x, i = x & 0xFFFFFFu;
        const int r = (int)(x >> 24 & 3u), place = (int)(i % (unsigned)span);
        packed[p].x = (x >> 26) << 24 | (unsigned)(words ? rb_cell(words[i], r, place, span) : r * span + place);
    }
}

}  // namespace bmtk

using namespace bmtk;

extern "C" int bmtk_csr_receptors_used(int64_t nnz, const int32_t *indices, const uint8_t *receptors, uint32_t *used, void *stream)
{
    BMTK_REQUIRE(nnz >= 0 && (nnz == 0 || (indices && receptors && used)), "csr_receptors_used: bad arguments");
    if (nnz == 0) return BMTK_OK;
    const int64_t blocks = (nnz + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(receptors_used_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0, (hipStream_t)stream, nnz, indices, receptors, used);
    BMTK_CHECK_LAUNCH("csr_receptors_used");
    return BMTK_OK;
}

extern "C" int bmtk_csr_pack_cells(int64_t nnz, int32_t span, const uint32_t *cells, bmtk_synapse *packed, void *stream)
{
    BMTK_REQUIRE(nnz >= 0 && span > 0 && (nnz == 0 || packed), "csr_pack_cells: bad arguments");
    if (nnz == 0) return BMTK_OK;
    const int64_t blocks = (nnz + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(pack_cells_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0, (hipStream_t)stream, nnz, span, cells,
                       reinterpret_cast<uint2 *>(packed));
    BMTK_CHECK_LAUNCH("csr_pack_cells");
    return BMTK_OK;
}

extern "C" int bmtk_events_by_trial(int32_t batch, int64_t step0, int64_t n_steps, int32_t late, const int64_t *in_ptr,
                                    const int32_t *in_events, int32_t *counts, const int64_t *first, int32_t *sources, void *stream)
{
    BMTK_REQUIRE(batch >= 1 && batch <= kWave, "events_by_trial: batch must lie in 1..64");
    BMTK_REQUIRE(step0 >= -1 && n_steps > 0 && n_steps < (1ll << 31), "events_by_trial: bad steps");
    BMTK_REQUIRE(in_ptr && in_events && (counts != nullptr) != (first != nullptr) && (first != nullptr) == (sources != nullptr),
                 "events_by_trial: null pointers, or counts and first together");
    if (counts)
        hipLaunchKernelGGL(events_by_trial_kernel<false>, dim3((unsigned)n_steps), dim3(kBlock), 0, (hipStream_t)stream, batch, step0, n_steps, late,
                           in_ptr, in_events, counts, first, sources);
    else
        hipLaunchKernelGGL(events_by_trial_kernel<true>, dim3((unsigned)n_steps), dim3(kBlock), 0, (hipStream_t)stream, batch, step0, n_steps, late,
                           in_ptr, in_events, counts, first, sources);
    BMTK_CHECK_LAUNCH("events_by_trial");
    return BMTK_OK;
}
