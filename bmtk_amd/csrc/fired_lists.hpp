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
constexpr unsigned kListQuick = 9, kListHalf = 19, kListMax = 39;  // neurons in words 0..1, 0..3, 0..7
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
    // (kFew: lists are seldom more than a wavefront's lanes, and a branch past the rest is worth it)
    template <bool kFew>
    __device__ __forceinline__ bool look(const ListRow &row, unsigned tag, int from = 0)
    {
        const unsigned lane = (unsigned)lane_here();
        const char *base = reinterpret_cast<const char *>(row.at(0, from));
        const unsigned stride = 8u * (from ? kListWords - kListQuickWords : kListQuickWords);
#pragma unroll
        for (int u = 0; u < kListRounds; ++u) {
            if (kFew && u * kWave >= row.G) break;
            const unsigned long long *p = reinterpret_cast<const unsigned long long *>(base + min(u * kWave + lane, (unsigned)row.G - 1u) * stride);
            v[u][0] = load_agent64(p);
            v[u][1] = load_agent64(p + 1);
        }
        unsigned differs = 0u;
#pragma unroll
        for (int u = 0; u < kListRounds; ++u) {
            if (kFew && u * kWave >= row.G) break;
            differs |= ((unsigned)(v[u][0] >> 32) ^ (tag << (kListTagAt - 32))) | ((unsigned)(v[u][1] >> 32) ^ (tag << (kListTagAt - 32)));
        }
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
template <bool kFew, typename Again>
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
    if (__any(most > kListHalf) || more > cap || total + more > cap) return kCrowded;
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
    if (__any(most > kListQuick)) {
        while (!seen.template look<kFew>(lists, tag, kListQuickWords)) {
            if (!again()) {
                lost = true;
                return kCrowded;
            }
        }
        emit(kListQuick, false);
    }
    return total;
}

// All 1024 threads: the rows of a crowded step -- the neurons in `lists` (ballots where a list did not suffice, `ballot_words` to a
// workgroup, `words` in all) and n_ev rows event(i) -- to act[0 .. cap), their number to *count, which was zero.  What finds no
// room goes to spot(row) at once.  A word is looked for max_spin times in vain at most.  kWordRounds: 4 * kWordRounds words cover a list or a workgroup's ballots.
template <int kWordRounds, typename Event, typename Spot>
__device__ __forceinline__ void crowded_rows(const ListRow &lists, bool any, int span, const unsigned long long *ballots, int words,
                                             unsigned n_ev, unsigned *act, unsigned cap, unsigned *count, unsigned *abort_word,
                                             unsigned max_spin, Event event, Spot spot)
{
    constexpr unsigned kThreads = 1024u;
    int me = (int)threadIdx.x;
    asm volatile("" : "+v"(me));
    const int of = me >> 2, sub = me & 3;  // four threads to a list
    unsigned long long head = 0ull;
    if (any && of < lists.G) head = load_agent64(lists.at(of, 0));
    const unsigned n = (unsigned)(head >> kListCountAt) & kListMany;
    const bool many = n == kListMany;
    const int event_rounds = (int)((n_ev + kThreads - 1u) / kThreads);
    for (int round = -event_rounds; round < kWordRounds; ++round) {
        unsigned long long v = 0ull;
        unsigned cnt = 0u, base = (unsigned)(of * span);
        bool bits = false;
        if (round < 0) {
            const unsigned at = (unsigned)(round + event_rounds) * kThreads + (unsigned)me;
            if (at < n_ev) base = event(at), cnt = 1u;
        } else {
            const int j = round * 4 + sub;  // word of the list, or of the workgroup's ballots
            const unsigned first = j == 0 ? 0u : 5u * (unsigned)j - 1u;
            if (many) {
                const int w = of * (span >> 6) + j;
                if (j < (span >> 6) && w < words) v = load_agent64(ballots + w);
                cnt = (unsigned)__popcll(v);
                base += 64u * (unsigned)j;
                bits = true;
            } else if (j < kListWords && n > first) {
                // (words 0 and 1 have been seen; the others left with them)
                cnt = min(n - first, j == 0 ? 4u : 5u);
                unsigned spins = 0u;
                while (((v = load_agent64(lists.at(of, j))) ^ head) >> kListTagAt) {
                    // (given up, here or elsewhere: nothing of the run is valid, and check() will say so)
                    if (++spins > max_spin) __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (spins > max_spin || __hip_atomic_load(abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
                        cnt = 0u;
                        break;
                    }
                }
            }
        }
        const unsigned inc = wave_inclusive_scan(cnt);
        unsigned at = 0u;
        if (lane_id() == kWave - 1 && inc) at = atomicAdd(count, inc);
        at = (unsigned)bcast_i((int)at, kWave - 1) + inc - cnt;
        for (; cnt > 0u; --cnt, ++at) {
            unsigned id = base;
            if (bits) {
                id += (unsigned)(__ffsll((long long)v) - 1);
                v &= v - 1ull;
            } else if (round >= 0) {
                id += (unsigned)v & ((1u << kListIdBits) - 1u);
                v >>= kListIdBits;
            }
            if (at < cap)
                act[at] = id;
            else
                spot(id);
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
