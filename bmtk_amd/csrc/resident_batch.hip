// Resident simulation of the trials of a batch: state in registers and the ring in LDS for the length of a call, as in
// resident.hip, with the workgroups of the chip divided among several trials.
//
// The trials of a batch do not touch one another.  `ways` of them run side by side in one cooperative launch, each on
// `groups` workgroups with a grid barrier of its own; launches follow one another until every trial has had its turn.
// A workgroup owns `span` neurons of its trial.  Per step it
//   1. folds the arrivals of slot t-1 (LDS) into y1, updates its neurons from registers and publishes their ballots;
//   2. reads the ballots that its trial's workgroups published a step ago, packs the neurons that fired and the trial's
//      input events into a list of rows, signals the barrier of step t on the way, and adds its own segment of every
//      listed row (rows sorted by target, segment bounds in a table) to its ring slice.  A row's segment is read by
//      `1 << team_shift` neighbouring lanes: with few workgroups to a trial a segment holds tens of synapses, which one
//      lane would take one after the other.
// Neither state nor arrival sums cross the memory system, and of the table only the segments of rows that fired.
//
// Sums are 64-bit fixed point, exact and independent of the order, as in the fused batched driver (and an integer
// addition in LDS costs 28 clocks per wavefront where a float's costs 194).  Slot t-1 is folded and cleared before the
// spikes of step t-1 are added, so that ring_slots - 1 slots suffice: 160 bytes of LDS per neuron and trial at delays of
// up to five steps.  Behind a call the arrivals still ahead wait in rb_ring, trial by trial.
//
// What bounds it: a step is a chain of dependent loads (ballots, segment bounds, synapses) and the barrier, 3 us at the
// smallest sizes, whatever the number of trials side by side; then the table's segments, which every trial reads for itself.
//
// One trial of more neurons than the compute units have threads (resident.hip ends at 1024 to a workgroup) runs here with two
// neurons to a thread and its ring in floats, 80 bytes a neuron: 400,123 neurons, 72 M synapses, 23 -> 9 us per step against a
// launch per step with an atomic per event (call and set-up included: 25.4 -> 9.8).  What it is short of are the 128 vector
// registers a thread has: 84 hold two neurons.  Ballots kept over the prefix sum, addresses and products worked out once
// for all steps spilled 81 of them to memory (13.3 us per step).
#include <math.h>
#include <stdlib.h>

#include "glif3_update.hpp"
#include "pull_common.hpp"
#include "sim_internal.hpp"

namespace bmtk {

constexpr int kRbBlock = 1024;
constexpr int kRbWaves = kRbBlock / kWave;
constexpr int kRbHist = 4;                // rows of the ballot history
constexpr unsigned kRbMaxSpin = 4000000u; // polls of the barrier before giving up (seconds)
constexpr int kRbCounters = 64;           // arrival counters per way of res_sync, dealt out to the trials of a launch
constexpr int kRbWideWords = 8;           // ballot words per thread with two neurons to a thread
constexpr int kRbTogether = 4;            // synapses a lane has in flight

struct RbLaunch {
    int64_t step0;
    int n_steps;
    int trial0, trials;   // trials of this launch
    int slots;            // of the ring slice: ring_slots - 1
    int sync_slots;       // arrival counters of a trial, used in turn (a power of two)
    int words;            // ballot words of a trial
    int has_events;
    double unit;          // of the fixed-point sums
};

__device__ __forceinline__ unsigned rb_load(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct __attribute__((packed, aligned(4))) RbBounds {
    uint32_t lo, hi;
};

// The barrier's contract is that of resident.hip: ballots are stored and read with agent-scope accesses, every wavefront
// waits until its stores have been acknowledged (s_waitcnt vmcnt(0)) before its workgroup meets and one thread arrives,
// and a reader has counted all arrivals of the step before.  A trial's workgroups only count one another.  A workgroup
// arrives for step t after it has seen everybody arrive for step t-1, so that the arrivals of two steps never mix and one
// counter per trial would do; several used in turn keep a look at step t-1 apart from the arrivals of step t.  A workgroup
// that writes ballot row t%4 is at most two steps ahead of one that still reads row (t-3)%4.
// kWords: ballot words per thread.  kPer: neurons per thread; with two, the threads of the last wavefront (the looker) own
// none.  Sum: what the ring holds, 64-bit fixed point (from_fixed), or floats where a workgroup's neurons are too many for
// that (batch 1): fp32 atomics into device memory are what it then takes the place of.
// kSave: potentials and step flags of every step go to rb_save_*, trial by trial; by_step_kernel puts them in their order.
template <int kWords, int kPer, typename Sum, bool kSave>
__global__ __launch_bounds__(kRbBlock) void sim_resident_batch_kernel(bmtk_glif3_sim s, RbLaunch q)
{
    constexpr bool kFixed = sizeof(Sum) == 8;
    constexpr int kOwners = kPer == 1 ? kRbBlock : kRbBlock - kWave;  // threads that own neurons tid, tid + kOwners, ..
    extern __shared__ unsigned long long rb_lds[];  // ring slice [slots * 4][span], then the list of rows
    __shared__ int go_on;
    __shared__ unsigned scan_l[kRbWaves];
    __shared__ unsigned listed[2];  // rows in the list of this step and the next (one wide trial)
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
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
    auto place = [&](int u) { return kPer == 1 ? tid : (tid < kOwners ? u * kOwners + tid : span); };  // in the workgroup's span
    auto owns = [&](int u) { return place(u) < mine; };
    auto element = [&](int u) { return (int64_t)(e0 + (owns(u) ? place(u) : 0)) * batch + trial; };
    Sum *ring_l = reinterpret_cast<Sum *>(rb_lds);
    unsigned *act = reinterpret_cast<unsigned *>(ring_l + (size_t)S * GLIF3_NREC * span);
    unsigned *abort_word = s.res_sync + 1;
    unsigned *arrivals = s.res_sync + BMTK_RES_SYNC_STRIDE + way * q.sync_slots * BMTK_RES_SYNC_STRIDE;
    constexpr int kWayStride = kRbCounters * BMTK_RES_SYNC_STRIDE;
    unsigned long long *hist = reinterpret_cast<unsigned long long *>(s.rb_hist) + (int64_t)way * kRbHist * (q.words + 1);
    if (tid == 0) {
        go_on = rb_load(abort_word) == 0u;
        listed[0] = listed[1] = 0u;
    }
    __syncthreads();
    if (!go_on) return;

    Sum *ring_g = reinterpret_cast<Sum *>(s.rb_ring) + (int64_t)trial * S * GLIF3_NREC * n + e0;
    for (int c = tid; c < S * GLIF3_NREC * span; c += kRbBlock) {
        const int plane = c / span, k = c - plane * span;
        ring_l[c] = k < mine ? ring_g[(int64_t)plane * n + k] : (Sum)0;
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

    auto counter_of = [&](int j) { return arrivals + (j & (q.sync_slots - 1)) * BMTK_RES_SYNC_STRIDE; };
    auto poll = [&](int j) -> int {  // one thread: 1 = the trial's workgroups have all arrived at step j, 0 = given up
        const unsigned *word = counter_of(j);
        const unsigned target = (unsigned)G * ((unsigned)j / (unsigned)q.sync_slots + 1u);
        unsigned spins = 0;
        auto arrived = [&]() {
            unsigned v[BMTK_RES_SYNC_WAYS], sum = 0;
#pragma unroll
            for (int x = 0; x < BMTK_RES_SYNC_WAYS; ++x) v[x] = rb_load(word + x * kWayStride);
#pragma unroll
            for (int x = 0; x < BMTK_RES_SYNC_WAYS; ++x) sum += v[x];
            return sum;
        };
        while (arrived() < target) {
            if (rb_load(abort_word) != 0u) return 0;
            if (++spins > (s.res_spin_limit ? s.res_spin_limit : kRbMaxSpin)) {
                __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return 0;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        return 1;
    };

    // this workgroup's segment of one row, `part` of 1 << team_shift lanes, into the slots behind slot0
    const int ts = s.rb_team_shift;
    const unsigned part = (unsigned)tid & ((1u << ts) - 1u), step = 1u << ts;
    const uint32_t *__restrict__ seg = s.rb_seg + g;
    const uint2 *__restrict__ table = reinterpret_cast<const uint2 *>(s.rb_packed);
    const unsigned seg_stride = (unsigned)G + 1u;
    auto pull_row = [&](unsigned row, unsigned q_lo, unsigned q_wrap) {
        const RbBounds b = *reinterpret_cast<const RbBounds *>(seg + (size_t)row * seg_stride);
        // (slot0 + delay) % slots * 4 + receptor = min(u, u - 4 * slots), u = slot0 * 4 + the record's upper byte
        auto add = [&](const uint2 sy, bool crowded) {
            const unsigned dq = sy.x >> 24;
            const unsigned plane = min(dq + q_lo, dq + q_wrap);
            Sum *cell = ring_l + (mad_u24(plane, (unsigned)span, sy.x & 0xFFFFFFu) - (unsigned)e0);
            if constexpr (kFixed)
                atomicAdd(cell, to_fixed(__uint_as_float(sy.y)));
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
        for (uint32_t at_p = b.lo + part; at_p < b.hi; at_p += kRbTogether * step) {
            uint2 sy[kRbTogether];
#pragma unroll
            for (int u = 0; u < kRbTogether; ++u)
                if (at_p + u * step < b.hi) sy[u] = table[at_p + u * step];
#pragma unroll
            for (int u = 0; u < kRbTogether; ++u)
                if (at_p + u * step < b.hi) add(sy[u], u == 0);
        }
    };
    // Spikes in row `hist_row` of the ballot history (-1: none) and the input events [ka, kb) of the same step, whose ring
    // slot is slot0, into the ring slice.  All threads of the workgroup call it.  `arrival`: the counter to signal once
    // every wavefront's ballot store has been acknowledged.
    const int cap = s.rb_list;
    // The same for a single wide trial, whose many ballot words would not stay in registers beside two neurons' state: each
    // wavefront reads them kWideScan per thread at a time and takes its places in the list from a counter in LDS (`turn` tells
    // which of two: the other is cleared on the way), so that no word outlives its turn and the workgroup meets once less.
    constexpr int kWideScan = 4, kWideTurns = (kWords + kWideScan - 1) / kWideScan;
    auto pull_wide = [&](int hist_row, int slot0, unsigned ka, unsigned kb, unsigned *arrival, int turn) {
        const unsigned q_lo = (unsigned)slot0 * 4u, q_wrap = q_lo - 4u * (unsigned)S;
        const unsigned n_ev = kb - ka;
        unsigned base[kWideTurns];
        // the places from `base` on of the list's window [c0, c0 + cap); the first look takes the places
        auto list_words = [&](bool first, unsigned c0) {
            // (not to be worked out once for all steps: that many addresses would push the state out of the registers)
            int me = tid;
            asm volatile("" : "+v"(me));
#pragma unroll
            for (int b = 0; b < kWideTurns; ++b) {
                unsigned long long v[kWideScan];
                unsigned cnt = 0u;
#pragma unroll
                for (int u = 0; u < kWideScan; ++u) {
                    const int w = min((b * kWideScan + u) * kRbBlock + me, q.words);  // (a row's last word stays zero)
                    v[u] = hist_row >= 0 ? __hip_atomic_load(hist + (int64_t)hist_row * (q.words + 1) + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
                }
#pragma unroll
                for (int u = 0; u < kWideScan; ++u) cnt += (unsigned)__popcll(v[u]);
                const unsigned inc = wave_inclusive_scan(cnt);
                if (first) {
                    unsigned to = 0u;
                    if (lane == kWave - 1) to = inc ? atomicAdd(&listed[turn], inc) : 0u;
                    base[b] = (unsigned)bcast_i((int)to, kWave - 1);
                }
                unsigned pos = base[b] + inc - cnt - c0;  // (wraps below zero for places of an earlier window)
#pragma unroll
                for (int u = 0; u < kWideScan; ++u) {
                    unsigned long long x = v[u];
                    const unsigned j0 = (unsigned)((b * kWideScan + u) * kRbBlock + me) << 6;
                    while (x) {
                        const unsigned bit = (unsigned)__ffsll((long long)x) - 1u;
                        x &= x - 1ull;
                        if (pos < (unsigned)cap) act[pos] = j0 + bit;
                        ++pos;
                    }
                }
            }
        };
        // (the events first: their places are known)
        for (unsigned k = (unsigned)tid; k < n_ev && k < (unsigned)cap; k += kRbBlock) act[k] = (unsigned)n + (unsigned)s.rb_in_events[ka + k];
        if (tid == 0) listed[turn ^ 1] = 0u;
#pragma unroll
        for (int b = 0; b < kWideTurns; ++b) base[b] = 0u;
        list_words(true, 0u - n_ev);
        if (arrival) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (arrival && tid == 0) __hip_atomic_fetch_add(arrival, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned total = listed[turn] + n_ev;
        for (unsigned c0 = 0;;) {
            const unsigned here = min(total - c0, (unsigned)cap);
            for (unsigned a = (unsigned)tid >> ts; a < here; a += (unsigned)kRbBlock >> ts) pull_row(act[a], q_lo, q_wrap);
            __syncthreads();
            c0 += (unsigned)cap;
            if (c0 >= total) break;
            // (a volley outgrows the list: the next window of it)
            for (unsigned k = (unsigned)tid; k < n_ev; k += kRbBlock)
                if (k - c0 < (unsigned)cap) act[k - c0] = (unsigned)n + (unsigned)s.rb_in_events[ka + k];
            list_words(false, c0 - n_ev);
            __syncthreads();
        }
    };
    auto pull = [&](int hist_row, int slot0, unsigned ka, unsigned kb, unsigned *arrival) {
        const unsigned q_lo = (unsigned)slot0 * 4u, q_wrap = q_lo - 4u * (unsigned)S;
        unsigned long long v[kWords];
        unsigned cnt = 0u;
#pragma unroll
        for (int u = 0; u < kWords; ++u) {
            // (the last word of a row is never written: it stays zero)
            const int w = min(u * kRbBlock + tid, q.words);
            v[u] = hist_row >= 0 ? __hip_atomic_load(hist + (int64_t)hist_row * (q.words + 1) + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        }
        const unsigned n_ev = kb - ka;
        const unsigned ev = (unsigned)tid < n_ev ? (unsigned)s.rb_in_events[ka + tid] : 0u;
#pragma unroll
        for (int u = 0; u < kWords; ++u) cnt += (unsigned)__popcll(v[u]);
        const unsigned inc = wave_inclusive_scan(cnt);
        if (lane == kWave - 1) scan_l[wave] = inc;
        if (arrival) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (arrival && tid == 0) __hip_atomic_fetch_add(arrival, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned parts = wave_inclusive_scan(lane < kRbWaves ? scan_l[lane] : 0u);
        const unsigned n_spk = (unsigned)bcast_i((int)parts, kRbWaves - 1);
        const unsigned base = wave > 0 ? (unsigned)__shfl((int)parts, wave - 1, kWave) : 0u;
        const unsigned total = n_spk + n_ev;
        for (unsigned c0 = 0; c0 < total; c0 += (unsigned)cap) {  // (one round unless a volley outgrows the list)
            unsigned pos = base + inc - cnt - c0;  // (wraps below zero for places of an earlier round)
#pragma unroll
            for (int u = 0; u < kWords; ++u) {
                unsigned long long x = v[u];
                const unsigned j0 = (unsigned)(u * kRbBlock + tid) << 6;
                while (x) {
                    const unsigned bit = (unsigned)__ffsll((long long)x) - 1u;
                    x &= x - 1ull;
                    if (pos < (unsigned)cap) act[pos] = j0 + bit;
                    ++pos;
                }
            }
            for (unsigned k = (unsigned)tid; k < n_ev; k += kRbBlock) {
                const unsigned to = n_spk + k - c0;
                if (to < (unsigned)cap) act[to] = (unsigned)n + (k == (unsigned)tid ? ev : (unsigned)s.rb_in_events[ka + k]);
            }
            __syncthreads();
            const unsigned here = min(total - c0, (unsigned)cap);
            for (unsigned a = (unsigned)tid >> ts; a < here; a += (unsigned)kRbBlock >> ts) pull_row(act[a], q_lo, q_wrap);
            __syncthreads();
        }
    };
    auto fold = [&](int slot) {
        if (kPer > 1) asm volatile("" : "+s"(slot));
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            if (!owns(u)) continue;
            Sum *cell = ring_l + (size_t)slot * GLIF3_NREC * span + place(u);
#pragma unroll
            for (int r = 0; r < GLIF3_NREC; ++r) {
                float a;
                if constexpr (kFixed)
                    a = from_fixed(cell[r * span], q.unit);
                else
                    a = cell[r * span];
                cell[r * span] = (Sum)0;
                st[u].y1[r] = st[u].y1[r] + a * p[u].psc0[r];
            }
        }
    };

    // the input events of the call's steps, trial by trial: those of step step0 - 1 + k are rb_in_events[in_ptr[k], in_ptr[k+1])
    const int64_t *in_ptr = q.has_events ? s.rb_in_ptr + (int64_t)trial * (q.n_steps + 1) : nullptr;
    int opaque_zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(opaque_zero));
    constexpr int kLooker = kRbBlock - kWave;  // its wavefront owns no neurons at spans up to 960, or with two to a thread
    const float zero[GLIF3_NREC] = {0.0f, 0.0f, 0.0f, 0.0f};
    unsigned ka = 0u, kb = 0u;
    if (in_ptr) {
        ka = (unsigned)in_ptr[0];
        kb = (unsigned)in_ptr[1];
    }
    int slot = (int)((q.step0 - 1 + S) % S);  // of step t-1
    const int n_steps = q.n_steps;
    bool aborted = false;
    for (int k = 0; k < n_steps; ++k) {
        // the bound of the next step's events: asked for here, looked at after the pull (see resident.hip)
        unsigned kn = 0u;
        if (in_ptr) kn = (unsigned)in_ptr[k + 2 + opaque_zero];
        if (k > 0 && tid == kLooker) go_on = poll(k - 1);
        if (k > 0) fold(slot);
        float h = s.h;
        if (kPer > 1) asm volatile("" : "+s"(h));  // (nor h times a neuron's propagators)
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            bool spike = false;
            float frac;
            const int ref_before = st[u].ref;
            if (owns(u)) spike = glif3_update(st[u], p[u], h, zero, I[u], &frac);
            const unsigned long long m = __ballot(spike);
            const int i = e0 + place(u);
            if (lane == 0 && place(u) < span && i < n)
                __hip_atomic_store(hist + (int64_t)(k & (kRbHist - 1)) * (q.words + 1) + (i >> 6), m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (kSave && owns(u)) {
                const int64_t to = ((int64_t)trial * n_steps + k) * n + i;
                s.rb_save_v[to] = st[u].V;
                s.rb_save_flags[to] = (uint8_t)((spike ? BMTK_F_SPIKE : 0) | (ref_before == 0 ? BMTK_F_INTEGRATING : 0) |
                                                (ref_before > 0 && st[u].ref == 0 ? BMTK_F_RESET : 0));
            }
            if (spike && s.spike_bits) {
                const int64_t e = element(u);
                __hip_atomic_fetch_or(reinterpret_cast<unsigned long long *>(s.spike_bits) + (int64_t)k * s.spike_bits_stride + (e >> 6),
                                      1ull << (e & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();
        if (k > 0 && !go_on) {
            aborted = true;
            break;
        }
        // (a call's first step: the spikes of the step before were added by the call before it, and so were its events unless
        //  they are to be taken from this call's lists)
        const bool with_events = k > 0 || s.rb_late_events;
        unsigned *const arrival = counter_of(k) + (g & (BMTK_RES_SYNC_WAYS - 1)) * kWayStride;
        if constexpr (kPer > 1)
            pull_wide(k > 0 ? (k - 1) & (kRbHist - 1) : -1, slot, ka, with_events ? kb : ka, arrival, k & 1);
        else
            pull(k > 0 ? (k - 1) & (kRbHist - 1) : -1, slot, ka, with_events ? kb : ka, arrival);
        ka = kb;
        kb = (unsigned)__builtin_amdgcn_readfirstlane((int)kn);
        slot = slot + 1 == S ? 0 : slot + 1;
    }
    if (!aborted) {
        if (tid == 0) go_on = poll(n_steps - 1);
        __syncthreads();
        aborted = go_on == 0;
    }
    if (!aborted) {
        // closing: what arrived in the last step, then the spikes (and events) of the last step
        fold(slot);
        __syncthreads();
        if constexpr (kPer > 1)
            pull_wide((n_steps - 1) & (kRbHist - 1), slot, ka, kb, nullptr, n_steps & 1);
        else
            pull((n_steps - 1) & (kRbHist - 1), slot, ka, kb, nullptr);
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u)
        if (owns(u)) glif3_store(st[u], s.V, s.asc, s.y1, s.y2, s.ref, ne, element(u));
    for (int c = tid; c < S * GLIF3_NREC * span; c += kRbBlock) {
        const int plane = c / span, k = c - plane * span;
        if (k < mine) ring_g[(int64_t)plane * n + k] = ring_l[c];
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

// arrival counters of a launch back to zero (the abort word stays until the host has seen it)
__global__ void rb_zero_sync_kernel(unsigned *sync)
{
    for (int c = threadIdx.x; c < BMTK_RES_SYNC_WAYS * kRbCounters; c += blockDim.x) sync[(1 + c) * BMTK_RES_SYNC_STRIDE] = 0u;
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
    BMTK_REQUIRE(span >= kWave && span % kWave == 0 && span <= (batch == 1 ? 2 * (kRbBlock - kWave) : kRbBlock) && G == (n + span - 1) / span,
                 "glif3_simulate_fwd: rb_span must be a multiple of 64 up to 1024 (one trial: 1920) and rb_groups ceil(n_neurons / rb_span)");
    BMTK_REQUIRE(wide == (batch == 1), "glif3_simulate_fwd: a single trial is resident in spans above 1024 here, in shorter ones by res_span");
    BMTK_REQUIRE(W >= 1 && W <= batch && s.rb_team_shift >= 0 && s.rb_team_shift <= 6 && s.rb_list >= kWave,
                 "glif3_simulate_fwd: rb_ways must lie in 1..batch, rb_team_shift in 0..6, rb_list from 64 on");
    BMTK_REQUIRE(s.rb_seg && s.rb_packed && s.rb_ring && s.rb_hist && s.res_sync, "glif3_simulate_fwd: resident trials need rb_* and res_sync");
    BMTK_REQUIRE(s.delay_offset == 0 && (s.delay_bits == 0 || s.delay_bits == 6), "glif3_simulate_fwd: resident trials need delay_offset 0 and the standard packing");
    const bool save = s.save_v != nullptr;
    BMTK_REQUIRE(!s.probe_col && !s.spike_count, "glif3_simulate_fwd: resident trials take no probes and keep no spike record");
    BMTK_REQUIRE(!save || (batch > 1 && s.rb_save_v && s.rb_save_flags && n_steps <= 65535),
                 "glif3_simulate_fwd: resident trials keep the per-step record of batches, up to 65535 steps a call, with rb_save_v and rb_save_flags");
    BMTK_REQUIRE(s.sum_shift >= 0 && s.sum_shift <= BMTK_SUM_SHIFT_MAX, "glif3_simulate_fwd: sum_shift must lie in 0..BMTK_SUM_SHIFT_MAX");
    BMTK_REQUIRE((s.rb_in_ptr == nullptr) == (s.rb_in_events == nullptr), "glif3_simulate_fwd: rb_in_ptr and rb_in_events go together");
    BMTK_REQUIRE(n_steps < (1ll << 30) && n + s.n_inputs < (1ll << 24), "glif3_simulate_fwd: too many steps or sources for resident trials");
    const size_t lds = (size_t)S * GLIF3_NREC * span * (wide ? sizeof(float) : sizeof(unsigned long long)) + (size_t)s.rb_list * sizeof(unsigned);
    BMTK_REQUIRE(lds + 256u <= kResLdsBytes, "glif3_simulate_fwd: the ring slice of resident trials does not fit in LDS");
    RbLaunch q{};
    q.step0 = step0;
    q.n_steps = (int)n_steps;
    q.slots = S;
    q.words = (int)((n + kWave - 1) / kWave);
    q.has_events = s.rb_in_ptr != nullptr;
    q.unit = ldexp(1.0, -32 - s.sum_shift);
    q.sync_slots = kRbCounters;
    while (q.sync_slots * W > kRbCounters) q.sync_slots /= 2;
    BMTK_REQUIRE(q.words <= (wide ? kRbWideWords : 4) * kRbBlock, "glif3_simulate_fwd: more neurons than resident trials can hold");
    const bool few = q.words <= kRbBlock;
    const void *kernel = wide ? reinterpret_cast<const void *>(sim_resident_batch_kernel<kRbWideWords, 2, float, false>)
        : few ? (save ? reinterpret_cast<const void *>(sim_resident_batch_kernel<1, 1, unsigned long long, true>)
                      : reinterpret_cast<const void *>(sim_resident_batch_kernel<1, 1, unsigned long long, false>))
              : (save ? reinterpret_cast<const void *>(sim_resident_batch_kernel<4, 1, unsigned long long, true>)
                      : reinterpret_cast<const void *>(sim_resident_batch_kernel<4, 1, unsigned long long, false>));
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
    if (s.spike_bits) {
        // (a spike is one bit in a word its trials share)
        const int64_t words = n_steps * s.spike_bits_stride, blocks = (words + kBlock - 1) / kBlock;
        hipLaunchKernelGGL(rb_zero_bits_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0, stream, s.spike_bits, words);
    }
    const char *plain = getenv("BMTK_AMD_PLAIN_LAUNCH");  // see simulate_resident
    for (int trial0 = 0; trial0 < batch; trial0 += W) {
        q.trial0 = trial0;
        q.trials = batch - trial0 < W ? batch - trial0 : W;
        hipLaunchKernelGGL(rb_zero_sync_kernel, dim3(1), dim3(kBlock), 0, stream, s.res_sync);
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

using namespace bmtk;

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
