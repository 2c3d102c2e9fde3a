// How the workgroups of a resident run tell one another which neurons fired: lists whose words say themselves which step
// they belong to.
//
// A list is eight 64-bit words per workgroup and step.  Every word carries a tag of its step in its upper nine bits, is
// stored with ONE agent-scope store and read with agent-scope loads: a reader that finds the tag it wants has the word,
// one that does not asks again.  Nothing has to be ordered between two words, so the writer waits for no acknowledgement
// and signals no counter, and a step needs no grid barrier: whoever has read the lists of step t of all workgroups knows
// that all have finished step t.  (With ballots and arrival counters three trips to memory followed one another -- the
// stores' acknowledgement, the arrivals, the look at the counters -- before the ballots could be asked for.)
//
//   word 0       tag | number that fired (11 bits) | 4 neurons (11 bits each, counted within the workgroup's span)
//   words 1..7   tag | 5 neurons
//
// A step in which more than 39 neurons of a workgroup fired says so in the number (kListMany): its ballots are read then,
// which the writer has waited for before it published the word.  All eight words are written in every step: the word a
// reader meets in place of the one it wants is then that row's last user's, `rows` steps ago, and nothing older, which
// is what makes eight bits of step number enough.  The rows are cleared before a launch, and a tag is never zero.
#pragma once

#include "common.hpp"

namespace bmtk {

constexpr int kListWords = BMTK_RES_FIRED_SLOTS / 2;
constexpr int kListQuickWords = 2;          // these of all workgroups side by side: what a reader asks for first
constexpr unsigned kListQuick = 9, kListMax = 39;  // neurons in words 0..1, 0..7
constexpr unsigned kListMany = 2047;        // in place of the number: more than kListMax, see the ballots
constexpr int kListRounds = 4;              // workgroups a lane of the reading wavefront looks after
constexpr int kListGroups = kListRounds * kWave;
constexpr int kListIdBits = 11, kListCountAt = 44, kListTagAt = 55;
static_assert(kListWords == 8 && kListCountAt == 4 * kListIdBits && kListTagAt == 5 * kListIdBits, "list layout");

__device__ __forceinline__ unsigned list_tag(int k) { return 256u | ((unsigned)k & 255u); }

__device__ __forceinline__ unsigned long long load_agent64(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The lists of one step: words 0 and 1 of every list, then words 2..7 of every list (a writer's stores and a reader's loads meet
// as few lines as that allows).
constexpr int kListRows = 4;   // lists of so many steps are kept
constexpr int kListRowWords = kListWords * kListGroups;
// They begin behind the first line of res_sync, at the next whole 64-bit word: that is scratch of 32-bit words, and as long as
// they were all that it held a caller's could lie on any of them.
constexpr size_t kListSyncWords = BMTK_RES_SYNC_STRIDE + 1 + (size_t)2 * kListRows * kListRowWords;  // of res_sync
static_assert(BMTK_RES_SYNC_WORDS >= kListSyncWords, "res_sync holds the lists");
__host__ __device__ inline unsigned long long *lists_in(unsigned *res_sync)
{
    return reinterpret_cast<unsigned long long *>((reinterpret_cast<uintptr_t>(res_sync + BMTK_RES_SYNC_STRIDE) + 7u) & ~(uintptr_t)7u);
}
struct ListRow {
    unsigned long long *w;
    int first, G;  // the lists that belong together: first .. first + G - 1
    __device__ __forceinline__ unsigned long long *at(int g, int j) const
    {
        g += first;
        return w + (j < kListQuickWords ? kListQuickWords * g + j
                                        : kListQuickWords * kListGroups + (kListWords - kListQuickWords) * g + j - kListQuickWords);
    }
};

// The lane's number, worked out where it is used: addresses and products of it, hoisted out of a loop over the steps, would
// push a neuron's state out of the registers.
__device__ __forceinline__ int lane_here()
{
    int l = lane_id();
    asm volatile("" : "+v"(l));
    return l;
}

// One wavefront: the list of workgroup g, of n neurons that stand in fired_l.  In two parts, so that its reads of LDS go out
// beside others of the caller.
struct ListWrite {
    unsigned first, id[5];

    __device__ __forceinline__ void read(const unsigned short *fired_l)
    {
        const unsigned j = (unsigned)lane_here() & (kListWords - 1u);
        first = max(5u * j, 1u) - 1u;  // (39 entries are looked at, whatever their number)
#pragma unroll
        for (unsigned i = 0; i < 5u; ++i) id[i] = fired_l[first + i];
    }
    __device__ __forceinline__ void publish(const ListRow &row, int g, unsigned tag, unsigned n) const
    {
        const int j = lane_here();
        unsigned long long word = (unsigned long long)tag << kListTagAt;
#pragma unroll
        for (unsigned i = 0; i < 4u; ++i) word |= (unsigned long long)(first + i < n ? id[i] : 0u) << (kListIdBits * i);
        // (word 0: the number stands where the others have their fifth neuron)
        const unsigned fifth = first + 4u < n ? id[4] : 0u;
        word |= (unsigned long long)(j > 0 ? fifth : n > kListMax ? kListMany : n) << kListCountAt;
        if (j < kListWords) __hip_atomic_store(row.at(g, j), word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};
// What the reading wavefront holds of a step's lists: words 0 and 1, lane l those of workgroups l, l + 64, ..
struct ListLook {
    unsigned long long v[kListRounds][kListQuickWords];

    __device__ __forceinline__ void none()
    {
#pragma unroll
        for (int u = 0; u < kListRounds; ++u) v[u][0] = v[u][1] = 0ull;
    }
    // asks once for words `from`, `from` + 1 of all G lists; true when every workgroup has published them in the wanted step
    // (beyond the G-th the last list over again: with a branch past those, 16 to 256 lists took the same time within 2 %)
    __device__ __forceinline__ bool look(const ListRow &row, unsigned tag, int from = 0)
    {
        const unsigned lane = (unsigned)lane_here();
        const char *base = reinterpret_cast<const char *>(row.at(0, from));
        const unsigned stride = 8u * (from ? kListWords - kListQuickWords : kListQuickWords);
#pragma unroll
        for (int u = 0; u < kListRounds; ++u) {
            const unsigned long long *p = reinterpret_cast<const unsigned long long *>(base + min(u * kWave + lane, (unsigned)row.G - 1u) * stride);
            v[u][0] = load_agent64(p);
            v[u][1] = load_agent64(p + 1);
        }
        unsigned differs = 0u;
#pragma unroll
        for (int u = 0; u < kListRounds; ++u)
            differs |= ((unsigned)(v[u][0] >> 32) ^ (tag << (kListTagAt - 32))) | ((unsigned)(v[u][1] >> 32) ^ (tag << (kListTagAt - 32)));
        return __ballot((differs >> (kListTagAt - 32)) != 0u) == 0ull;
    }
    __device__ __forceinline__ unsigned count(int u, int G) const
    {
        return u * kWave + lane_id() < G ? (unsigned)(v[u][0] >> kListCountAt) & kListMany : 0u;
    }
};

// the i-th neuron of a word
__device__ __forceinline__ unsigned list_id(unsigned long long word, int i)
{
    const unsigned lo = (unsigned)word, hi = (unsigned)(word >> 32);
    const int at = kListIdBits * i;
    const unsigned bits = at + kListIdBits <= 32 ? lo >> at : at >= 32 ? hi >> (at - 32) : __builtin_amdgcn_alignbit(hi, lo, at);
    return bits & ((1u << kListIdBits) - 1u);
}

// One wavefront: the neurons in the lists `seen`, whose workgroups own `span` neurons each, to rows[to ..] in LDS.  Returns their
// number, or kCrowded where a list holds too many for this or there is no room for them and `more` rows in `cap` places; false
// of `again` (called with every look in vain) gives up.  rows[spare] is the lane's own place for what is no row.
// Every instruction here is one of a single wavefront, four clocks each and more beside three others on its SIMD: what no
// list holds is not stepped through, and a store too many is cheaper than a branch of lanes.
constexpr unsigned kCrowded = 0xFFFFFFFFu;  // in place of a number of rows
constexpr unsigned kMoreEvents = 1u << 30;  // beside it: the step has more input events than the reader has listed
template <typename Again>
__device__ __forceinline__ unsigned rows_from_lists(ListLook &seen, const ListRow &lists, unsigned tag, int span, unsigned *rows,
                                                    unsigned to, unsigned cap, unsigned spare, unsigned more, Again again, bool &lost)
{
    unsigned c[kListRounds], sum = 0u;
#pragma unroll
    for (int u = 0; u < kListRounds; ++u) {
        c[u] = seen.count(u, lists.G);
        sum += c[u];
    }
    const unsigned inc = wave_inclusive_scan(sum);
    const unsigned total = (unsigned)bcast_i((int)inc, kWave - 1);
    const unsigned most = max(max(c[0], c[1]), max(c[2], c[3]));
    if (__any(most > kListMax) || more > cap || total + more > cap) return kCrowded;
    const unsigned me = (unsigned)lane_here();
    // the neurons in the words of `seen`, from the j0-th of a list on
    auto emit = [&](unsigned j0, bool first) __attribute__((always_inline)) {
        unsigned pos = to + inc - sum + j0;
#pragma unroll
        for (int u = 0; u < kListRounds; ++u) {
            if (u * kWave >= lists.G) break;
            const unsigned base = (u * kWave + me) * (unsigned)span;
#pragma unroll
            for (int i = 0; i < (first ? 9 : 10); ++i) {
                const bool is = c[u] > j0 + (unsigned)i;
                if (__ballot(is) == 0ull) break;
                const int at = first && i > 3 ? i + 1 : i;  // (word 0 holds four)
                rows[is ? pos + (unsigned)i : spare] = base + list_id(seen.v[u][at / 5], at % 5);
            }
            pos += c[u];
        }
    };
    emit(0u, true);
    // (two more words of all lists at a time)
#pragma unroll
    for (int from = kListQuickWords; from < kListWords; from += 2) {
        const unsigned j0 = 5u * from - 1u;
        if (!__any(most > j0)) break;
        while (!seen.look(lists, tag, from)) {
            if (!again()) {
                lost = true;
                return kCrowded;
            }
        }
        emit(j0, false);
    }
    return total;
}

// All 1024 threads: the rows of a crowded step -- n_first rows first(i), at most one to a thread and cap, and the neurons in `lists`,
// ballots where a list did not suffice (`words` in all) -- to act[0 .. cap), as many at a time as there is room for; pull(n) works act[0 .. n) off.  count: three words of LDS.  A word is
// looked for max_spin times in vain at most.  kBallotWords: of a workgroup, at most.
// A thread holds two words a round, and as many threads share a list as let all lists have theirs: eight words of every
// list are one round, sixteen ballots of every workgroup one or two.
template <int kBallotWords, typename First, typename Pull>
__device__ __forceinline__ void crowded_rows(const ListRow &lists, unsigned tag, int span, const unsigned long long *ballots, int words,
                                             unsigned n_first, First first_row, unsigned *act, unsigned cap, unsigned *count, unsigned *abort_word,
                                             unsigned max_spin, Pull pull)
{
    constexpr unsigned kManyAt = 24u;  // upper bits of a counter: wavefronts that met a list that did not suffice
    // (worked out where it is used: beside a neuron's state there are no registers for it)
    auto here = []() __attribute__((always_inline)) {
        int me = (int)threadIdx.x;
        asm volatile("" : "+v"(me));
        return me;
    };
    if (here() < 3) count[here()] = 0u;
    __syncthreads();
    const int sharing = lists.G <= 64 ? 4 : lists.G <= 128 ? 3 : 2;  // 1 << sharing threads to a list
    unsigned filled = n_first;  // places taken
    int turn = 0;          // a counter for every handing out of places: the one before may still be read, the one after is cleared
    bool ballots_too = false, last = false;
    bool bits = false;     // this thread's words are ballots
    for (int round = 0; !last; ++round) {
        unsigned long long v[2] = {0ull, 0ull};
        auto word = [&](int i) __attribute__((always_inline)) { return ((2 * round + i) << sharing) + (here() & ((1 << sharing) - 1)); };
        const int of = here() >> sharing;
        const unsigned first_one = round == 0 && (unsigned)here() < n_first ? first_row((unsigned)here()) : 0u;
        if (of < lists.G && (round == 0 || bits)) {
            // (the reader has seen all lists, so their ballots are there: both are asked for at once.  A list's words end in the first round)
            unsigned long long ballot[2] = {0ull, 0ull}, head = 0ull;
            if (round == 0) head = load_agent64(lists.at(of, 0));
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int w = of * (span >> 6) + word(i);
                if (round == 0 && word(i) < kListWords) v[i] = load_agent64(lists.at(of, word(i)));
                if (word(i) < (span >> 6) && w < words) ballot[i] = load_agent64(ballots + w);
            }
            const unsigned n = (unsigned)(head >> kListCountAt) & kListMany;
            bits = bits || n == kListMany;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (bits) {
                    v[i] = ballot[i];
                    continue;
                }
                const int j = word(i);
                const unsigned first = j == 0 ? 0u : 5u * (unsigned)j - 1u;
                unsigned left = 0u;
                if (j < kListWords && n > first) {
                    // (words 0 and 1 have been seen; the others left with them)
                    left = min(n - first, j == 0 ? 4u : 5u);
                    for (unsigned spins = 0u; (unsigned)(v[i] >> kListTagAt) != tag; v[i] = load_agent64(lists.at(of, j))) {
                        // (given up, here or elsewhere: nothing of the run is valid, and check() will say so)
                        if (++spins > max_spin) __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (spins > max_spin || __hip_atomic_load(abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
                            left = 0u;
                            break;
                        }
                    }
                }
                // (in place of the tag: the neurons left in the word)
                v[i] = (v[i] & ((1ull << kListTagAt) - 1ull)) | (unsigned long long)left << kListTagAt;
            }
        }
        if (round == 0 && (unsigned)here() < n_first) act[here()] = first_one;
        while (true) {
            unsigned mine = 0u;
#pragma unroll
            for (int i = 0; i < 2; ++i) mine += bits ? (unsigned)__popcll(v[i]) : (unsigned)(v[i] >> kListTagAt);
            const unsigned inc = wave_inclusive_scan(mine);
            const unsigned flag = __any(bits) ? 1u << kManyAt : 0u;
            unsigned at = 0u;
            if (lane_id() == kWave - 1 && (inc | flag)) at = atomicAdd(&count[turn], inc + flag);
            at = filled + ((unsigned)bcast_i((int)at, kWave - 1) & ((1u << kManyAt) - 1u)) + inc - mine;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const unsigned base = (unsigned)((here() >> sharing) * span + (bits ? 64 * word(i) : 0));
                while (at < cap && (bits ? v[i] : v[i] >> kListTagAt)) {
                    unsigned id = (unsigned)v[i];
                    if (bits) {
                        id = (unsigned)__ffsll((long long)v[i]) - 1u;
                        v[i] &= v[i] - 1ull;
                    } else {
                        id &= (1u << kListIdBits) - 1u;
                        const unsigned long long left = (v[i] >> kListTagAt) - 1ull;
                        v[i] = ((v[i] & ((1ull << kListTagAt) - 1ull)) >> kListIdBits) | left << kListTagAt;
                    }
                    act[at++] = base + id;
                }
            }
            __syncthreads();
            const unsigned handed = count[turn];
            turn = turn == 2 ? 0 : turn + 1;
            if (here() == 0) count[turn == 2 ? 0 : turn + 1] = 0u;
            ballots_too = ballots_too || (handed >> kManyAt) != 0u;
            const unsigned total = filled + (handed & ((1u << kManyAt) - 1u));
            last = total <= cap && (2 * (round + 1)) << sharing >= (ballots_too ? kBallotWords : kListWords);
            filled = total;
            if (total <= cap && !last) break;
            pull(min(total, cap));
            __syncthreads();
            filled = 0u;
            if (last) break;
        }
    }
}

// Words of LDS that wavefronts of the workgroup tell one another how far they are by.  A wavefront's accesses to LDS are worked
// off in the order it issues them; only the compiler has to be kept from another order.
__device__ __forceinline__ unsigned load_lds(unsigned *p)
{
    const unsigned v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    asm volatile("" ::: "memory");
    return v;
}
__device__ __forceinline__ void store_lds(unsigned *p, unsigned v)
{
    asm volatile("" ::: "memory");
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void count_lds(unsigned *p)
{
    asm volatile("" ::: "memory");
    if (lane_id() == 0) __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

}  // namespace bmtk
