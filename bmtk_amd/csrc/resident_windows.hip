// Resident forward simulation of a SMALL network whose delays leave several steps between a spike and its first arrival.
//
// resident_solo.hip keeps a network of up to 1024 neurons on one compute unit, at one workgroup barrier per step and one
// trip to memory for the step's rows.  bmtk's example networks run at a resolution of 0.1 ms or finer with delays of 1 to 2 ms:
// what fires in a step arrives ten to some thousand steps later.  Here the wavefronts that hold neurons run a WINDOW of up
// to eight steps from registers with no barrier in between; meanwhile the others walk the rows of spikes and input events that
// arrive from the next window on.  One barrier ends a window.
//
// A spike of step u arrives from step u + E + 1 on, E = delay offset + smallest residual delay - 1.  Let a window be the
// steps [T, T+S).  Its updates use up the ring slots [T, T+S), which earlier windows have completed.  Delivered beside them are
// the spikes and events of the steps u in [T+S-1-E, T+2S-2-E]: their first arrivals lie in the next window, their last at
// most 2S-1 + (largest - smallest delay) steps from T: a ring of one slot more.  Their rows are listed a window ahead, from
// ballots of steps before T-S: 3S-1 <= E.  In front of the first window its own share is delivered, behind the last one what
// the call still owes, so that state and ring are left exactly as the other drivers leave them.
//
// What a wavefront does beside its neurons, in a window: the event wavefront and the fired wavefront turn the next window's input
// events and spikes into items (first synapse, length, step) in LDS; the store wavefront writes the window before out: ballots,
// record; the others take rows, one trip to memory for four of them.  Those without neurons come first; where a window has many
// rows, all take some; where it has more than the lists hold, all look them up for themselves.
//
// What sets the pace is the chain of instructions of the wavefronts that hold neurons: 650 clocks a step whether a SIMD has one
// of them or two (issue, at four clocks an instruction, is used up by two), 1,000 clocks a window for the barrier and what surrounds it.  A ring
// cell holds its four receptors side by side, so that an update takes them with one read and clears them with one write, and an
// update folds the arrivals of its own step (the sum that the other forms leave to the step after: the same roundings).  A wavefront's
// roles are compiled apart: with one loop for all, spilled registers, whose reloads wait for every load and store under way,
// made it 0.52 us a step, and lists made by the wavefronts that take the rows 0.46.  One loop spills still, that of wavefronts with neurons
// where fewer than three others are left to take rows (more than 640 cells), which holds every role: 56 of the kernel's 108 scratch
// instructions, once a window each, none within a step or a row; the others stand before and behind the loops.
//   450 cells at 0.1 ms, delays of 20 steps, 5 Hz of 1,000 inputs, with record: 0.34 us a step (single steps: 1.03); 900 cells: 1.05 (1.5);
//   450 cells at 0.001 ms, delays of 2,000 steps: 0.31 (0.74).
#include <type_traits>

#include "glif3_update.hpp"
#include "sim_internal.hpp"

namespace bmtk {

constexpr int kWinBlock = 1024;
constexpr int kWinWaves = kWinBlock / kWave;
constexpr int kWinSteps = 8;       // steps of a window at most (a lane holds two of a window's 8 x 16 ballots)
constexpr int kWinNear = 64;       // steps whose ballots stay in LDS
constexpr int kWinFar = kWinNear - 2;   // beyond this distance ballots come from the history in device memory
constexpr int kWinItems = 4 * kWave;    // rows of input events, and of neurons that fired, that a window's lists hold
constexpr int kWinStoreWave = kWinWaves - 1, kWinEventWave = kWinWaves - 2, kWinFiredWave = kWinWaves - 3;
constexpr int kWinAhead = 2 * kWinSteps;   // with those, from this row on, the ballots of the window at hand and of the next

constexpr int kTakeRole = 0, kEventRole = 1, kFiredRole = 2, kStoreRole = 3;   // what a wavefront does beside its neurons, see below

struct Window {
    int64_t step0;
    int n_steps, span;
    int offset, hist;        // delay offset B, rows of the ballot history
    int steps, slots;        // S, ring slots in LDS
    int lead;                // E
    int inp_lds, rec_lds;    // the row bounds of the input and of the recurrent table have room in LDS
    int record;              // spike offsets are kept
};

// dynamic LDS: the ring, the spike offsets of two windows
static size_t window_lds_bytes(int slots, int steps, int span, bool record)
{
    return (size_t)slots * span * sizeof(float4) + (record ? (size_t)2 * steps * span * sizeof(float) : 0);
}
constexpr size_t kWinStaticLds = kWinNear * kWinWaves * 8 + kWinWaves * kWave * 2 + 4 * kWinItems * 16 + 2 * (kWinSteps + 1) * 8 + 256;   // with the compiler's padding

__global__ __launch_bounds__(kWinBlock) void sim_window_kernel(bmtk_glif3_sim s, Window r)
{
    extern __shared__ float4 cells_l[];                                  // [slots][span], then as window_lds_bytes says
    __shared__ unsigned long long near_l[kWinNear][kWinWaves];           // ballots of the last steps
    __shared__ unsigned short ids_l[kWinWaves][kWave];                   // per wavefront: neurons whose rows it takes next
    __shared__ int4 items_l[2][2][kWinItems];                            // rows delivered beside this and the next window: events, fired
    __shared__ int2 counts_l[2];                                         // ... how many (with those that the lists do not hold)
    __shared__ int64_t begins_l[2][kWinSteps + 1];                       // where their steps' events begin
    __shared__ int go_on;
    const int tid = threadIdx.x, lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int ne = (int)s.n_neurons, words = (ne + 63) >> 6;
    const int L = s.ring_slots, span = r.span, B = r.offset, S = r.steps, R = r.slots, n = r.n_steps;
    const bool own = tid < ne;
    const bool far = B > kWinFar;
    // (with ballots from the history only those of two windows are kept)
    const int near_mask = far ? 2 * kWinSteps - 1 : kWinNear - 1;
    float *frac_l = reinterpret_cast<float *>(cells_l + R * span);       // [2][S][span]
    int *inp_ip_l = reinterpret_cast<int *>(frac_l + (r.record ? 2 * S * span : 0));
    int *rec_ip_l = inp_ip_l + (r.inp_lds ? (int)s.n_inputs + 1 : 0);
    unsigned long long *hist = reinterpret_cast<unsigned long long *>(s.work_bits);
    // an earlier resident run on this simulator gave up and nobody has looked yet: do nothing (the word is sticky)
    if (tid == 0)
        go_on = (s.res_sync == nullptr || __hip_atomic_load(s.res_sync + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) ? 1 : 0;
    __syncthreads();
    if (!go_on) return;

    // steps, ring slots and arrivals count from step0 in what follows
    for (int c = tid; c < R * span; c += kWinBlock) {
        const int a = c / span, i = c - a * span;
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (a < L - 1 && i < ne) {
            const float *cell = s.ring + (r.step0 + a) % L * GLIF3_NREC * ne + i;
            v = make_float4(cell[0], cell[ne], cell[2 * ne], cell[3 * ne]);
        }
        cells_l[c] = v;
    }
    if (r.inp_lds)
        for (int c = tid; c <= (int)s.n_inputs; c += kWinBlock) inp_ip_l[c] = s.inp_indptr[c];
    if (r.rec_lds)
        for (int c = tid; c <= ne; c += kWinBlock) rec_ip_l[c] = s.rec_indptr[c];
    if (!far)
        for (int c = tid; c < B * kWinWaves; c += kWinBlock) {
            // the ballots of the B steps before this call
            const int64_t u = r.step0 - 1 - c / kWinWaves;
            const int w = c % kWinWaves;
            near_l[u & near_mask][w] = (u >= 0 && w < words) ? hist[u % r.hist * (words + 1) + w] : 0ull;
        }
    Glif3Elem st{};
    Glif3Prop p{};
    float I = 0.0f;
    if (own) {
        const int64_t col = s.class_id ? (int64_t)s.class_id[tid] : tid;
        p.load(s.prop, s.prop_stride, col);
        glif3_load(st, s.V, s.asc, s.y1, s.y2, s.ref, ne, tid);
        I = s.i_ext ? s.i_ext[tid] : 0.0f;
    }
    const int probe_col = (own && s.probe_col) ? s.probe_col[tid] : -1;
    int probe_phase = s.probe_col ? (int)((r.step0 + 1) % s.probe_every) : 1;   // 0: sample after this step
    float *probe_out = s.probe_v;                                               // the row of the next sample
    const unsigned long long rec_cap = (unsigned long long)s.spike_cap / (s.spike_ways > 1 ? (unsigned)s.spike_ways : 1u);
    unsigned long long rec_count = (wave == kWinStoreWave && s.spike_count) ? s.spike_count[0] : 0ull;
    __syncthreads();

    const uint2 *__restrict__ rec_tab = reinterpret_cast<const uint2 *>(s.rec_packed);
    const uint2 *__restrict__ inp_tab = reinterpret_cast<const uint2 *>(s.inp_packed);
    const bool has_rec = s.rec_indptr != nullptr, has_in = s.in_ptr != nullptr && s.inp_indptr != nullptr;
    // Ring slot of a synapse of delay d (as the packed record has it) for the j-th step of spikes delivered beside a window:
    // (slot0 + j + d - (E - B)) % R, where no d is below E - B + 1: the sum lies in [0, 2R).
    const int less = r.lead - B;
    int slot0 = R - 1;
    auto add = [&](const uint2 sy, int first) {
        const unsigned x = (unsigned)first + (sy.x >> 26);
        const unsigned slot = min(x, x - (unsigned)R);
        // (a compare-and-swap loop: the LDS unit works a float atomic off lane by lane, see resident_solo.hip)
        unsigned *cell = reinterpret_cast<unsigned *>(cells_l) + (((slot * (unsigned)span + (sy.x & 0xFFFFFFu)) << 2) + ((sy.x >> 24) & 3u));
        const float w = __uint_as_float(sy.y);
        unsigned old = *cell;   // only seeds the loop
        while (true) {
            const unsigned seen = atomicCAS(cell, old, __float_as_uint(__uint_as_float(old) + w));
            if (seen == old) break;
            old = seen;
        }
    };
    // Rows that this wavefront takes, a lane each: first synapse, length, which of the window's steps of spikes.  Lanes below n_ev
    // hold rows of the input table, lanes below n_have rows at all.
    int p0_v = 0, len_v = 0, j_v = 0, n_ev = 0, n_have = 0;
    constexpr int kAhead = 4;      // rows whose first 64 synapses are asked for before any is added
    uint2 head[kAhead];
    auto ask = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kAhead; ++q)
            if (i + q < n_have) {      // (at most 64)
                const uint2 *__restrict__ tab = i + q < n_ev ? inp_tab : rec_tab;
                if (lane < bcast_i(len_v, i + q)) head[q] = tab[bcast_i(p0_v, i + q) + lane];
            }
    };
    auto put = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kAhead; ++q)
            if (i + q < n_have) {
                const uint2 *__restrict__ tab = i + q < n_ev ? inp_tab : rec_tab;
                const int first = slot0 - less + bcast_i(j_v, i + q), len = bcast_i(len_v, i + q);
                if (lane < len) add(head[q], first);
                for (int k = lane + kWave; k < len; k += kWave) add(tab[bcast_i(p0_v, i + q) + k], first);
            }
    };
    // (what LDS holds is pinned to a register: the compiler would make one generic load, which waits for everything, of the two)
    auto pin = [](int v) -> int {
        asm volatile("" : "+v"(v));
        return v;
    };
    auto bounds = [&](int in_lds, const int *lds, const int32_t *__restrict__ mem, int row) __attribute__((always_inline)) {
        if (in_lds) {
            p0_v = pin(lds[row]);
            len_v = pin(lds[row + 1]) - p0_v;
        } else {
            p0_v = mem[row];
            len_v = mem[row + 1] - p0_v;
        }
    };
    // A lane holds the ballots lane and lane + 64 of a window's S x words: word w of its j-th step.
    const int j0 = lane / words, w0 = lane - j0 * words;
    const int j1 = (lane + kWave) / words, w1 = lane + kWave - j1 * words;
    // The spikes and events delivered beside the window at hand are those of the steps u0 .. u0+S-1 that this call owes.
    const int u_first = -B, u_last = n - 1 - B;
    int u0 = -1 - r.lead;
    int half = 0;           // of what has been left in LDS for the window at hand; the other half is the next window's
    auto owed = [&](int u, int j) -> bool { return j < S && u + j >= u_first && u + j <= u_last; };
    // the ballots of the neurons that fired in the steps from u on: those of recent steps
    unsigned long long x0 = 0ull, x1 = 0ull;
    auto near_ballots = [&](int u) __attribute__((always_inline)) {
        x0 = owed(u, j0) ? near_l[(r.step0 + u + j0) & near_mask][w0] : 0ull;
        x1 = owed(u, j1) ? near_l[(r.step0 + u + j1) & near_mask][w1] : 0ull;
    };
    // Neurons `base` .. `base` + 63 of the marked ones: lane i's, from lane `from` on, and their rows.
    unsigned rank = 0;      // of this lane's first
    auto ranks = [&]() __attribute__((always_inline)) -> int {
        const unsigned cnt = (unsigned)__popcll(x0) + (unsigned)__popcll(x1);
        if (__ballot(cnt != 0u) == 0ull) return 0;
        const unsigned upto = wave_inclusive_scan(cnt);
        rank = upto - cnt;
        return bcast_i((int)upto, kWave - 1);
    };
    auto fired_rows = [&](int base, int from, int n_fired) __attribute__((always_inline)) {
        int at = (int)rank - base + from;
        for (unsigned long long x = x0; x; x &= x - 1ull, ++at)
            if ((unsigned)at < (unsigned)kWave) ids_l[wave][at] = (unsigned short)(w0 * kWave + __ffsll((long long)x) - 1 + (j0 << 10));
        for (unsigned long long x = x1; x; x &= x - 1ull, ++at)
            if ((unsigned)at < (unsigned)kWave) ids_l[wave][at] = (unsigned short)(w1 * kWave + __ffsll((long long)x) - 1 + (j1 << 10));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane >= from && lane - from < n_fired - base) {
            const unsigned v = ids_l[wave][lane];
            const int id = (int)(v & 1023u);
            j_v = (int)(v >> 10);
            bounds(r.rec_lds, rec_ip_l, s.rec_indptr, id);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };

    // Event wavefront: the rows of a window's input events, as items in LDS a window ahead; the events are asked for another window
    // ahead, and the places where they stand (lane j: those of its j-th step begin; lane S: the end) a third.
    int ahead[kWinItems / kWave];
    int64_t ev1 = 0, ev2 = 0;
    auto ask_begins = [&](int u) -> int64_t {
        const int64_t i = r.step0 + min(max(u + min(lane, S), u_first), u_last + 1);
        return has_in && i > 0 ? s.in_ptr[i] : 0;    // (steps before 0 have no events)
    };
    auto ask_events = [&]() __attribute__((always_inline)) {
        const int64_t lo = (int64_t)bcast_u64((unsigned long long)ev1, 0);
        const int count = bcast_i((int)(ev1 - lo), S);
#pragma unroll
        for (int q = 0; q < kWinItems / kWave; ++q)
            if (q * kWave + lane < count) ahead[q] = s.in_events[lo + q * kWave + lane];
    };
    auto leave_events = [&](int h) __attribute__((always_inline)) {
        const int64_t lo = (int64_t)bcast_u64((unsigned long long)ev1, 0);
        const int begins = (int)(ev1 - lo), count = bcast_i(begins, S);
        if (lane <= S) begins_l[h][lane] = ev1;
        if (lane == 0) counts_l[h].x = count;
        if (count == 0 || count > kWinItems) return;
#pragma unroll
        for (int k = 0; k < kWinItems / kWave; ++k) {
            const int i = k * kWave + lane;
            if (k * kWave >= count) break;
            int j = 0;
            for (int q = 1; q < S; ++q) j += i >= bcast_i(begins, q) ? 1 : 0;
            if (i < count) {
                bounds(r.inp_lds, inp_ip_l, s.inp_indptr, ahead[k]);
                items_l[h][0][i] = make_int4(p0_v, len_v, j, 0);
            }
        }
    };
    // Fired wavefront: the same of the neurons that fired; a distant step's ballots are asked for two windows ahead.
    unsigned long long ahead_x0 = 0ull, ahead_x1 = 0ull;
    auto ask_far = [&](int u) __attribute__((always_inline)) {
        auto row = [&](int j, int w) -> unsigned long long {
            const int64_t at = r.step0 + u + j;
            if (!has_rec || at < 0 || !owed(u, j)) return 0ull;
            return __hip_atomic_load(hist + at % r.hist * (words + 1) + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        ahead_x0 = row(j0, w0);
        ahead_x1 = row(j1, w1);
    };
    auto leave_fired = [&](int u, int h) __attribute__((always_inline)) {
        if (far) {
            x0 = ahead_x0;
            x1 = ahead_x1;
            // (for a crowded window)
            if (j0 < S) near_l[kWinAhead + h * kWinSteps + j0][w0] = x0;
            if (j1 < S) near_l[kWinAhead + h * kWinSteps + j1][w1] = x1;
        } else if (has_rec) {
            near_ballots(u);
        }
        const int count = ranks();
        if (lane == 0) counts_l[h].y = count;
        if (count > kWinItems) return;
        for (int base = 0; base < count; base += kWave) {
            fired_rows(base, 0, count);
            if (base + lane < count) items_l[h][1][base + lane] = make_int4(p0_v, len_v, j_v, 0);
        }
    };
    if (wave == kWinEventWave) {
        ev1 = ask_begins(u0);
        ask_events();
        leave_events(half);
        ev1 = ask_begins(u0 + S);
        ask_events();
        ev2 = ask_begins(u0 + 2 * S);
    }
    if (wave == kWinFiredWave) {
        if (far) ask_far(u0);
        leave_fired(u0, half);
        if (far) ask_far(u0 + S);
    }
    __syncthreads();
    // Who takes rows: the wavefronts without neurons or another role first (`few` of them); not the store wavefront, whose loads
    // would wait for its stores.
    const int takers_most = kWinWaves - 1, few = kWinFiredWave - words;
    const int turn = wave == kWinStoreWave ? takers_most : (wave + max(takers_most - words, 0)) % takers_most;
    // A crowded window has more rows than the lists of items hold: every wavefront takes events turn, turn + 15, ... (ev_mine of
    // them) from where they are and the neurons of every 15th ballot (fired_mine of them), counted from the other end.
    int ev_mine = 0, fired_mine = 0;
    int64_t ev_lo = 0;
    int begins = 0;
    auto deal = [&](int events) __attribute__((always_inline)) {
        const int64_t ev = begins_l[half][min(lane, S)];
        ev_lo = (int64_t)bcast_u64((unsigned long long)ev, 0);
        begins = (int)(ev - ev_lo);
        ev_mine = turn < events ? (events - 1 - turn) / takers_most + 1 : 0;
        if (far) {
            x0 = j0 < S ? near_l[kWinAhead + half * kWinSteps + j0][w0] : 0ull;
            x1 = j1 < S ? near_l[kWinAhead + half * kWinSteps + j1][w1] : 0ull;
        } else if (has_rec) {
            near_ballots(u0);
        }
        if (lane % takers_most != takers_most - 1 - turn) x0 = 0ull;
        if ((lane + kWave) % takers_most != takers_most - 1 - turn) x1 = 0ull;
        fired_mine = ranks();
    };
    auto look_up = [&](int base) __attribute__((always_inline)) {
        n_ev = min(max(ev_mine - base, 0), kWave);
        n_have = min(max(ev_mine + fired_mine - base, 0), kWave);
        p0_v = len_v = j_v = 0;
        if (n_have > n_ev) fired_rows(max(base - ev_mine, 0), n_ev, fired_mine);
        if (n_ev == 0) return;
        const int i = turn + takers_most * (base + lane);
        int j = 0;
        for (int q = 1; q < S; ++q) j += i >= bcast_i(begins, q) ? 1 : 0;
        if (lane < n_ev) {
            bounds(r.inp_lds, inp_ip_l, s.inp_indptr, s.in_events[ev_lo + i]);
            j_v = j;
        }
    };
    // The rows base .. base + 63 of this wavefront: those of a crowded window (takers = 0), or turn, turn + takers, ... of the lists.
    auto refill = [&](int base, int takers, int2 count) __attribute__((always_inline)) {
        if (takers == 0) {
            look_up(base);
            return;
        }
        const int g = turn + takers * (base + lane);
        const bool ev = g < count.x, in = g < count.x + count.y;
        int4 item = make_int4(0, 0, 0, 0);
        if (in) item = *(ev ? &items_l[half][0][g] : &items_l[half][1][g - count.x]);
        p0_v = item.x;
        len_v = item.y;
        j_v = item.z;
        n_ev = (int)__popcll(__ballot(ev));
        n_have = (int)__popcll(__ballot(in));
    };

    // Store wavefront: ballots to the history and the output rows, the spike record, `c` steps from step `stored` on.
    int stored = 0, stored_buf = 0;
    int hist_row = (int)(r.step0 % r.hist);
    uint64_t *bits_out = s.spike_bits;
    auto write_out = [&](int c) __attribute__((always_inline)) {
        auto put = [&](int j, int w) -> unsigned long long {
            if (j >= c) return 0ull;
            const unsigned long long v = near_l[(r.step0 + stored + j) & near_mask][w];
            // (of rows that share a place in a short history the last one stays)
            if (j >= c - r.hist) __hip_atomic_store(hist + (int64_t)((hist_row + j) % r.hist) * (words + 1) + w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (bits_out) bits_out[(int64_t)j * s.spike_bits_stride + w] = v;
            return v;
        };
        auto record = [&](unsigned long long v, int j, int w) {
            if (__ballot(v != 0ull) == 0ull) return;
            const unsigned cnt = (unsigned)__popcll(v);
            const unsigned inc = wave_inclusive_scan(cnt);
            unsigned long long idx = rec_count + (inc - cnt);
            for (; v; v &= v - 1ull, ++idx) {
                const int elem = w * kWave + __ffsll((long long)v) - 1;
                if (idx < rec_cap) {
                    s.spike_step[idx] = (int32_t)(unsigned)(r.step0 + stored + j);
                    s.spike_elem[idx] = (int32_t)elem;
                    if (s.spike_frac) s.spike_frac[idx] = frac_l[(stored_buf * S + j) * span + elem];
                }
            }
            rec_count += (unsigned long long)(unsigned)bcast_i((int)inc, kWave - 1);
        };
        const unsigned long long v0 = put(j0, w0), v1 = put(j1, w1);
        if (s.spike_count) {
            record(v0, j0, w0);
            record(v1, j1, w1);
        }
        stored += c;
        stored_buf ^= 1;
        hist_row = (hist_row + c) % r.hist;
        if (bits_out) bits_out += c * s.spike_bits_stride;
    };

    int t = -S;              // the window's first step; the first round has none and delivers in front of step 0
    int take = 0, buf = 1;   // ring slot of step t, half of frac_l
    // The loop over the windows, compiled once per role of a wavefront, so that none keeps the registers of the others (what does
    // not fit is spilled to memory, and a reload there waits for every load and store under way).
    auto windows = [&](auto neuron, auto what, auto late) __attribute__((always_inline)) {
        constexpr bool kNeuron = decltype(neuron)::value, kLate = decltype(late)::value;
        constexpr int kRole = decltype(what)::value;
        // (of wavefronts with neurons only some have a second role, and only where nearly all have neurons)
        constexpr bool kAny = kNeuron && !kLate;
        const bool is_event = kAny ? wave == kWinEventWave : kRole == kEventRole, is_fired = kAny ? wave == kWinFiredWave : kRole == kFiredRole;
        const bool stores = kAny ? wave == kWinStoreWave : kRole == kStoreRole, takes = !stores;
        while (true) {
            // what the next window needs
            if (is_event) {
                leave_events(half ^ 1);
                ev1 = ev2;
                ask_events();
                ev2 = ask_begins(u0 + 3 * S);
            }
            if (is_fired) {
                leave_fired(u0 + S, half ^ 1);
                if (far) ask_far(u0 + 2 * S);
            }
            int2 count = make_int2(0, 0);
            int takers = 0, base = 0;
            n_have = 0;
            // The rows delivered beside this window: few of them are the business of the wavefronts without neurons, many (it pays from
            // some four to each of those on) everybody's.
            auto begin = [&]() __attribute__((always_inline)) {
                count = counts_l[half];
                count = make_int2(__builtin_amdgcn_readfirstlane(count.x), __builtin_amdgcn_readfirstlane(count.y));
                const bool crowded = count.x > kWinItems || count.y > kWinItems;
                takers = crowded ? 0 : few < 3 || count.x + count.y > 4 * few ? takers_most : few;
                if (crowded) deal(count.x);
                if (crowded || turn < min(takers, count.x + count.y)) {
                    refill(0, takers, count);
                    ask(0);
                }
            };
            // (a wavefront with neurons seldom has a row where there are others without: after its update is soon enough)
            if (takes && !kLate) begin();
            if (kNeuron && t >= 0 && t < n) {
                const int c = min(S, n - t);
                int at = take * span + tid;
                int slot = take;
                float4 next = cells_l[at];
                unsigned long long mine = 0ull;   // lane j: the ballot of the window's j-th step
                for (int j = 0; j < c; ++j) {
                    const float arrived[GLIF3_NREC] = {next.x, next.y, next.z, next.w};
                    cells_l[at] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    ++slot;
                    at += span;
                    if (slot == R) {
                        slot = 0;
                        at = tid;
                    }
                    next = cells_l[at];      // (behind the window's last step: not used)
                    float frac = 0.0f;
                    unsigned long long m;
                    glif3_update_wave(st, p, s.h, arrived, I, own, &m, &frac);
                    if (lane == j) mine = m;
                    // (any of the wavefront's cells: only those of neurons that fired are read)
                    if (m != 0ull && r.record) frac_l[(buf * S + j) * span + tid] = frac;
                    if (s.probe_col) {
                        if (probe_phase == 0) {
                            if (probe_col >= 0) probe_out[probe_col] = st.V;
                            probe_out += s.probe_stride;
                        }
                        probe_phase = probe_phase + 1 == s.probe_every ? 0 : probe_phase + 1;
                    }
                }
                if (lane < c) near_l[(r.step0 + t + lane) & near_mask][wave] = mine;
                take = slot;
            }
            if (stores) {
                const int c = min(t, n) - stored;      // the window before (its last steps, if it was cut short)
                if (c > 0) write_out(c);
            }
            if (takes && kLate) begin();
            for (int i = 0; i < n_have;) {
                put(i);
                i += kAhead;
                if (i >= n_have) {
                    base += kWave;
                    i = 0;
                    refill(base, takers, count);
                }
                ask(i);
            }
            // (a history row that ask_far reads is 30 steps old at least: written, and acknowledged windows ago)
            if (stores && far) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            t += S;
            u0 += S;
            slot0 += S;
            if (slot0 >= R) slot0 -= R;
            buf ^= 1;
            half ^= 1;
            if (t >= n && u0 > u_last) break;
        }
    };
    if (wave < words && few >= 3)
        windows(std::true_type{}, std::integral_constant<int, kTakeRole>{}, std::true_type{});
    else if (wave < words)
        windows(std::true_type{}, std::integral_constant<int, kTakeRole>{}, std::false_type{});
    else if (wave == kWinEventWave)
        windows(std::false_type{}, std::integral_constant<int, kEventRole>{}, std::false_type{});
    else if (wave == kWinFiredWave)
        windows(std::false_type{}, std::integral_constant<int, kFiredRole>{}, std::false_type{});
    else if (wave == kWinStoreWave)
        windows(std::false_type{}, std::integral_constant<int, kStoreRole>{}, std::false_type{});
    else
        windows(std::false_type{}, std::integral_constant<int, kTakeRole>{}, std::false_type{});
    if (wave == kWinStoreWave && stored < n) write_out(n - stored);
    if (own) glif3_store(st, s.V, s.asc, s.y1, s.y2, s.ref, ne, tid);
    if (wave == kWinStoreWave && lane == 0 && s.spike_count) s.spike_count[0] = rec_count;
    for (int c = tid; c < L * span; c += kWinBlock) {
        const int a = c / span, i = c - a * span;
        if (i >= ne) continue;
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (a < L - 1) v = cells_l[(n + a) % R * span + i];
        float *cell = s.ring + (r.step0 + n + a) % L * GLIF3_NREC * ne + i;
        cell[0] = v.x;
        cell[ne] = v.y;
        cell[2 * ne] = v.z;
        cell[3 * ne] = v.w;
    }
}

// Steps of a window, ring slots and all; false where the form by single steps is the faster one: the spikes arrive too early for
// windows of several steps, or the ring has no room.  A window of two steps pays while three wavefronts hold no neurons (us per step,
// windows / single steps, delays of 8 steps: 450 cells 0.77 / 0.97, 640 1.07 / 1.16, 780 1.21 / 1.28, 900 1.6 / 1.57), one of three always (900
// cells, 10 steps 1.25 / 1.55).  Where nearly all wavefronts hold neurons, windows of more input events than their lists hold are not
// for them (all rows are looked up by wavefronts that have an update to do; us per step, windows of three steps / single steps, 1,000 inputs
// of 110 synapses a cell: 900 cells 58 events a step 4.66 / 4.71, 72 5.48 / 5.48, 91 6.69 / 6.50, 113 7.95 / 7.60, 139 9.29 / 9.11; 840 cells 72 5.02 / 5.35, 91
// 6.34 / 6.35, 113 7.59 / 7.42; with three wavefronts free windows stay ahead, 832 cells 91 6.09 / 6.30, 139 8.54 / 8.90).  With ballots from the history (a delay offset beyond what LDS keeps) the offset is all that counts.
static bool plan_windows(const bmtk_glif3_sim &s, int hist, Window &w, size_t &lds)
{
    const int longest = s.ring_slots - 1, B = s.delay_offset;
    int less = 0;
    if (B <= kWinFar) {
        less = s.res_min_delay - 1;
        if (less > longest - 1) less = longest - 1;
        if (less > kWinFar - B) less = kWinFar - B;
        if (less < 0) less = 0;
    }
    w.offset = B;
    w.hist = hist;
    w.span = s.res_span;
    w.lead = B + less;
    w.record = s.spike_count != nullptr && s.spike_frac != nullptr;
    const int least = w.span / kWave <= kWinFiredWave ? 2 : 3;
    const size_t bounds = s.inp_indptr ? (size_t)(s.n_inputs + 1) * sizeof(int) : 0;
    for (w.steps = (w.lead + 1) / 3 < kWinSteps ? (w.lead + 1) / 3 : kWinSteps; w.steps >= least; --w.steps) {
        w.slots = 2 * w.steps - 1 + longest - less;
        if (w.slots < s.ring_slots) w.slots = s.ring_slots;
        lds = window_lds_bytes(w.slots, w.steps, w.span, w.record);
        if (lds + kWinStaticLds > kResLdsBytes) continue;
        if (least == 3 && (int64_t)s.res_step_events * w.steps > kWinItems) continue;
        w.inp_lds = bounds > 0 && lds + bounds + kWinStaticLds <= kResLdsBytes;
        if (w.inp_lds) lds += bounds;
        const size_t own = s.rec_indptr ? (size_t)(s.n_neurons + 1) * sizeof(int) : 0;
        w.rec_lds = own > 0 && lds + own + kWinStaticLds <= kResLdsBytes;
        if (w.rec_lds) lds += own;
        return true;
    }
    return false;
}

int simulate_resident_windows(const bmtk_glif3_sim &s, int64_t step0, int64_t n_steps, hipStream_t stream, bool *taken)
{
    Window w{};
    size_t lds = 0;
    *taken = n_steps < (1ll << 30) && plan_windows(s, s.hist_slots ? s.hist_slots : 3, w, lds);
    if (!*taken) return BMTK_OK;
    w.step0 = step0;
    w.n_steps = (int)n_steps;
    const void *kernel = reinterpret_cast<const void *>(sim_window_kernel);
    hipError_t err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) {
        set_error("glif3_simulate_fwd: the form by windows needs %zu bytes of LDS: %s", lds, hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    hipLaunchKernelGGL(sim_window_kernel, dim3(1), dim3(kWinBlock), lds, stream, s, w);
    err = hipGetLastError();
    if (err != hipSuccess) {
        set_error("glif3_simulate_fwd: launch of the form by windows failed: %s", hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    return BMTK_OK;
}

}  // namespace bmtk

extern "C" int bmtk_resident_window_steps(const bmtk_glif3_sim *s)
{
    bmtk::Window w{};
    size_t lds = 0;
    return s && s->res_groups == 1 && bmtk::plan_windows(*s, s->hist_slots ? s->hist_slots : 3, w, lds) ? w.steps : 0;
}
