// HIP kernels and C entry points of the per-step operations: propagator
// precompute, fused GLIF3 state update, spike compaction, event-driven scatter
// and row-wise gather into the delay ring buffer.  gfx950 only.
#include <math.h>
#include <stdarg.h>

#include <mutex>

#include "common.hpp"
#include "glif3_update.hpp"
#include "propagate.hpp"

namespace bmtk {

static thread_local char g_error[512] = "";

void set_error(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
}

// ---------------------------------------------------------------------------
// Propagators (NEST glif_psc::pre_run_hook + libnestutil/propagator_stability)
// ---------------------------------------------------------------------------

__device__ double propagator_32(double tau_syn, double tau, double C, double h)
{
    const double lin = 1.0 / (2.0 * C * tau * tau) * h * h * (tau_syn - tau) * exp(-h / tau);
    const double sing = h / C * exp(-h / tau);
    const double P32 = -tau / (C * (1.0 - tau / tau_syn)) * exp(-h / tau_syn) * expm1(h * (1.0 / tau_syn - 1.0 / tau));
    const double dev = fabs(P32 - sing);
    if (tau == tau_syn || (fabs(tau - tau_syn) < 0.1 && dev > 2.0 * fabs(lin))) return sing;
    return P32;
}

__device__ double propagator_31(double tau_syn, double tau, double C, double h)
{
    const double lin = 1.0 / (3.0 * C * tau * tau) * h * h * h * (tau_syn - tau) * exp(-h / tau);
    const double P31 = 1.0 / C *
                       (exp(-h / tau_syn) * expm1(-h / tau + h / tau_syn) / (tau / tau_syn - 1.0) * tau -
                        h * exp(-h / tau_syn)) /
                       (-1.0 - -tau / tau_syn) * tau;
    const double sing = h * h / 2.0 / C * exp(-h / tau);
    const double dev = fabs(P31 - sing);
    if (tau == tau_syn || (fabs(tau - tau_syn) < 0.1 && dev > 2.0 * fabs(lin))) return sing;
    return P31;
}

__global__ __launch_bounds__(kBlock) void precompute_kernel(int64_t n, const double *__restrict__ par, double h,
                                                            float *__restrict__ prop)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
#define PA(k) par[(int64_t)(k) * n + i]
#define PO(k) prop[(int64_t)(k) * n + i]
    const double C = PA(GLIF3_PAR_C_M), g = PA(GLIF3_PAR_G);
    const double tau = C / g;
    const double P33 = exp(-h / tau);
    PO(GLIF3_P33) = (float)P33;
    PO(GLIF3_P30) = (float)(1.0 / C * (1.0 - P33) * tau);
    PO(GLIF3_TH) = (float)(PA(GLIF3_PAR_V_TH) - PA(GLIF3_PAR_E_L));
    PO(GLIF3_UR) = (float)(PA(GLIF3_PAR_V_RESET) - PA(GLIF3_PAR_E_L));
    // NEST counts the refractory period down in floating point, one resolution per step
    const double t_ref = PA(GLIF3_PAR_T_REF);
    double rem = t_ref;
    int nref = 0;
    while (rem > 0.0 && nref < (1 << 24)) {
        rem -= h;
        ++nref;
    }
    PO(GLIF3_NREF) = (float)nref;
    for (int a = 0; a < GLIF3_NASC; ++a) {
        const double k = PA(GLIF3_PAR_ASC_DECAY0 + a);
        const double d = exp(-k * h);
        PO(GLIF3_D0 + a) = (float)d;
        PO(GLIF3_C0 + a) = (float)(((1.0 / k) / h) * (1.0 - d));
        PO(GLIF3_R0 + a) = (float)(PA(GLIF3_PAR_ASC_R0 + a) * exp(-k * t_ref));
        PO(GLIF3_AMP0 + a) = (float)PA(GLIF3_PAR_ASC_AMPS0 + a);
    }
    for (int r = 0; r < GLIF3_NREC; ++r) {
        const double ts = PA(GLIF3_PAR_TAU_SYN0 + r);
        PO(GLIF3_P11_0 + r) = (float)exp(-h / ts);
        PO(GLIF3_P31_0 + r) = (float)propagator_31(ts, tau, C, h);
        PO(GLIF3_P32_0 + r) = (float)propagator_32(ts, tau, C, h);
        PO(GLIF3_PSC0_0 + r) = (float)(2.718281828459045235360287 / ts);
    }
#undef PA
#undef PO
}

// ---------------------------------------------------------------------------
// Fused state update: one thread per element, every array access is a
// contiguous 256-byte row per wavefront.
// ---------------------------------------------------------------------------

struct StepArgs {
    int64_t ne;
    int32_t batch;
    float *V, *asc, *y1, *y2;
    int32_t *ref;
    const float *prop;
    int64_t stride;
    const int32_t *class_id;
    float h;
    float *syn;
    int32_t clear_syn;
    const float *i_ext;
    uint8_t *z;
    uint64_t *zbits;
    float *frac;
};

// kLdsTable: the propagators come from a class table small enough for LDS; the workgroup copies it there once
// and every thread reads its class's 29 values from there.  Read from device memory instead, those 29 scattered
// loads per thread, not the state traffic, set the pace (4.3 TB/s of algorithmic traffic against 6.1 with one
// parameter column per neuron).  At N = 2^20 with 111 classes, on two machines: 18.3 / 18.5 us with four tiles
// per workgroup, 18.1 / 19.5 with two, 24.4 with one; transposing the table on its way into LDS (an integer
// division per word, one word per load) took 19.8 / 20.2 with four tiles.  By measured bytes the launch then moves
// 5.95 TB/s where the form with a column per neuron moved 6.15 TB/s on the same machine.
//
// While all workgroups of one tile are resident at once there is nothing to share the staging with, and four tiles a workgroup leave compute
// units idle: 30,011 elements are 30 workgroups.  Seven of them fit a compute unit by their 72 registers a thread, fewer by the table: five
// of 250 classes (29 KB), three of 423 (49 KB).  One tile / four, us a call (of a loop of calls: not below 5.2 on the host), by classes:
//   37: 200,000 elements 5.4 / 6.2, 440,000 7.1 / 7.4, 524,288 7.9 / 7.8     111: 5.3 / 6.4, 7.2 / 7.7, 8.4 / 7.9     176: 5.2 / 6.9, 7.7 / 8.0, 8.9 / 8.4
//   200 (six): 350,000 7.0 / 7.9, 400,000 8.1 / 8.0          250 (five): 327,680 6.6 / 7.9, 350,000 8.8 / 8.2
//   300 (four): 262,144 6.2 / 7.5, 327,680 8.5 / 8.2         423 (three): 196,608 5.7 / 7.6, 230,924 8.9 / 8.1, 524,288 13.0 / 9.8
// (kernels alone at 5,000, 30,011 and 100,000 elements: 111 classes 3.7 / 5.6, 3.8 / 6.1, 4.2 / 6.3; 423 classes 4.8 / 6.8, 4.9 / 7.4, 5.5 / 7.6.)
constexpr int kStepTiles = 4;
constexpr int kStepPerCu = 7;                 // workgroups of one tile on a compute unit
constexpr size_t kLdsPerCu = 160u * 1024u, kLdsUnit = 1280u;  // LDS of a compute unit, and what it is given out in

// kTilesOrNone: tiles of a workgroup that stages the class table in LDS; 0: the table is not staged
template <int kTilesOrNone>
__global__ __launch_bounds__(kBlock) void glif3_step_kernel(StepArgs a)
{
    extern __shared__ __align__(16) float step_table[];  // [GLIF3_NPROP][columns] when kLdsTable
    // with the table in LDS a workgroup of a large launch takes kStepTiles tiles of 256 elements, so that staging the table is
    // shared by several tiles.  The state of all tiles is asked for first, before the table is staged: the loads
    // of the tiles travel together, and the staging runs while they are on their way.
    constexpr bool kLdsTable = kTilesOrNone > 0;
    constexpr int kTiles = kLdsTable ? kTilesOrNone : 1;
    Glif3Elem s[kTiles];
    float syn[kTiles][GLIF3_NREC], I[kTiles];
    int64_t e[kTiles], col[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        e[t] = ((int64_t)blockIdx.x * kTiles + t) * kBlock + threadIdx.x;
        col[t] = 0;
        I[t] = 0.0f;
        if (e[t] < a.ne) {
            const int64_t n = (a.batch == 1) ? e[t] : (int64_t)((uint32_t)e[t] / (uint32_t)a.batch);
            col[t] = a.class_id ? (int64_t)a.class_id[n] : n;
            glif3_load(s[t], a.V, a.asc, a.y1, a.y2, a.ref, a.ne, e[t]);
#pragma unroll
            for (int k = 0; k < GLIF3_NREC; ++k) syn[t][k] = a.syn ? a.syn[k * a.ne + e[t]] : 0.0f;
            I[t] = a.i_ext ? a.i_ext[e[t]] : 0.0f;
        }
    }
    if (kLdsTable) {
        stage_class_table<kBlock>(step_table, a.prop, (int)a.stride * GLIF3_NPROP);
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        bool spike = false;
        if (e[t] < a.ne) {
            Glif3Prop p;
            if (kLdsTable)
                p.load(step_table, a.stride, col[t]);
            else
                p.load(a.prop, a.stride, col[t]);
            float frac = 0.0f;
            spike = glif3_update(s[t], p, a.h, syn[t], I[t], &frac);
            glif3_store(s[t], a.V, a.asc, a.y1, a.y2, a.ref, a.ne, e[t]);
            if (a.syn && a.clear_syn) {
#pragma unroll
                for (int k = 0; k < GLIF3_NREC; ++k) a.syn[k * a.ne + e[t]] = 0.0f;
            }
            if (a.z) a.z[e[t]] = spike ? 1 : 0;
            if (a.frac && spike) a.frac[e[t]] = frac;
        }
        if (a.zbits) {
            const unsigned long long m = __ballot(spike);
            if (lane_id() == 0 && (e[t] & ~(int64_t)(kWave - 1)) < a.ne) a.zbits[e[t] >> 6] = m;
        }
    }
}

// ---------------------------------------------------------------------------
// Compaction: flags -> bits -> per-block popcounts -> scan -> ordered ids
// ---------------------------------------------------------------------------

constexpr int kWordsPerBlock = kBlock;  // one 64-element word per thread

__global__ __launch_bounds__(kBlock) void pack_bits_kernel(const uint8_t *__restrict__ z, int64_t n,
                                                           uint64_t *__restrict__ bits)
{
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const bool on = e < n && z[e] != 0;
    const unsigned long long m = __ballot(on);
    if (lane_id() == 0 && (e & ~(int64_t)(kWave - 1)) < n) bits[e >> 6] = m;
}

__device__ __forceinline__ unsigned long long load_word(const uint64_t *bits, int64_t w, int64_t n_words, int64_t n)
{
    if (w >= n_words) return 0ull;
    unsigned long long v = bits[w];
    const int tail = (int)(n & 63);
    if (w == n_words - 1 && tail) v &= (1ull << tail) - 1ull;
    return v;
}

__global__ __launch_bounds__(kBlock) void compact_count_kernel(const uint64_t *__restrict__ bits, int64_t n_words,
                                                               int64_t n, uint32_t *__restrict__ block_count)
{
    const int64_t w = (int64_t)blockIdx.x * kWordsPerBlock + threadIdx.x;
    unsigned total;
    block_exclusive_scan((unsigned)__popcll(load_word(bits, w, n_words, n)), &total);
    if (threadIdx.x == 0) block_count[blockIdx.x] = total;
}

// one workgroup: exclusive scan of block_count in place, total -> *count
__global__ __launch_bounds__(kBlock) void compact_scan_kernel(uint32_t *__restrict__ block_count, int n_blocks,
                                                              int32_t *__restrict__ count)
{
    const int per = (n_blocks + kBlock - 1) / kBlock;
    const int lo = threadIdx.x * per;
    const int hi = min(lo + per, n_blocks);
    unsigned sum = 0;
    for (int i = lo; i < hi; ++i) sum += block_count[i];
    unsigned total;
    unsigned run = block_exclusive_scan(sum, &total);
    for (int i = lo; i < hi; ++i) {
        const unsigned c = block_count[i];
        block_count[i] = run;
        run += c;
    }
    if (threadIdx.x == 0) *count = (int32_t)total;
}

__global__ __launch_bounds__(kBlock) void compact_write_kernel(const uint64_t *__restrict__ bits, int64_t n_words,
                                                               int64_t n, const uint32_t *__restrict__ block_offset,
                                                               int32_t *__restrict__ ids)
{
    const int64_t w = (int64_t)blockIdx.x * kWordsPerBlock + threadIdx.x;
    unsigned long long v = load_word(bits, w, n_words, n);
    unsigned total;
    unsigned pos = block_offset[blockIdx.x] + block_exclusive_scan((unsigned)__popcll(v), &total);
    const int32_t base = (int32_t)(w << 6);
    while (v) {
        const int b = __ffsll((long long)v) - 1;
        v &= v - 1ull;
        ids[pos++] = base + b;
    }
}

// Two launches instead of three or four, for up to kMaxFused blocks: the first counts (from flags it also packs
// the bits, 64 flags per thread), the second has every workgroup add up the counts of the workgroups before
// it by itself -- a few KB from L2 -- instead of waiting for a scan launch in between.
constexpr int kMaxFused = 4096;

// bits 0..3 = which of the four bytes of x are non-zero
__device__ __forceinline__ unsigned nonzero_bytes(unsigned x)
{
    const unsigned high = (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u;  // bit 7 of every non-zero byte
    return (((high >> 7) * 0x00204081u) >> 21) & 0xFu;                             // bits 0, 8, 16, 24 -> 0..3
}

__global__ __launch_bounds__(kBlock) void compact_count_flags_kernel(const uint8_t *__restrict__ z, int64_t n,
                                                                     int64_t n_words, uint64_t *__restrict__ bits,
                                                                     uint32_t *__restrict__ block_count)
{
    const int64_t w = (int64_t)blockIdx.x * kWordsPerBlock + threadIdx.x;
    unsigned long long v = 0ull;
    if (w < n_words) {
        const int64_t e0 = w << 6;
        if (e0 + 64 <= n) {
            const uint4 *q = reinterpret_cast<const uint4 *>(z + e0);  // z is 16-byte aligned (checked by the caller)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4 x = q[i];
                const unsigned long long part = nonzero_bytes(x.x) | (nonzero_bytes(x.y) << 4) |
                                                (nonzero_bytes(x.z) << 8) | (nonzero_bytes(x.w) << 12);
                v |= part << (16 * i);
            }
        } else {
            for (int64_t e = e0; e < n; ++e) v |= (unsigned long long)(z[e] != 0) << (e - e0);
        }
        bits[w] = v;
    }
    unsigned total;
    block_exclusive_scan((unsigned)__popcll(v), &total);
    if (threadIdx.x == 0) block_count[blockIdx.x] = total;
}

// block_count holds the plain per-block counts here
__global__ __launch_bounds__(kBlock) void compact_write_fused_kernel(const uint64_t *__restrict__ bits, int64_t n_words,
                                                                     int64_t n, const uint32_t *__restrict__ block_count,
                                                                     int32_t *__restrict__ ids,
                                                                     int32_t *__restrict__ count)
{
    unsigned before = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += kBlock) before += block_count[b];
    unsigned offset;
    block_exclusive_scan(before, &offset);  // the block sum is what is wanted
    const int64_t w = (int64_t)blockIdx.x * kWordsPerBlock + threadIdx.x;
    unsigned long long v = load_word(bits, w, n_words, n);
    unsigned total;
    unsigned pos = offset + block_exclusive_scan((unsigned)__popcll(v), &total);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *count = (int32_t)(offset + total);
    const int32_t base = (int32_t)(w << 6);
    while (v) {
        const int b = __ffsll((long long)v) - 1;
        v &= v - 1ull;
        ids[pos++] = base + b;
    }
}

// The bits of up to kOneLaunchWords words in ONE launch of one workgroup: a thread holds a word, a wavefront counts its 64 and writes
// its ids behind those of the wavefronts before it.  What bounds it with few of them on is the launch and three trips, with many the
// instructions of one compute unit.  One launch / two, us in a captured graph, 4.6 % on: 5,000 elements 1.9 / 3.4, 30,011 2.1 / 3.9, 65,536 2.4 / 3.9
// (in a loop of calls 4.0 / 6.9, the host's time); three in ten on: 30,011 5.1 / 5.6, 49,152 5.9 / 6.0, 65,536 6.8 / 5.9 (loop 6.9 / 6.9); all on: 65,536 6.9 / 11.6.
// It ends at a word a thread: with two words a thread 131,072 elements took 3.4 / 4.0 at 4.6 % on, but 15.2 / 6.4 at three in ten.  The scalar base and
// mask of the dense way: 8.3 -> 6.8 at 65,536 with three in ten on.
constexpr int kOneLaunchWords = 1024;
__global__ __launch_bounds__(kOneLaunchWords) void compact_one_kernel(const uint64_t *__restrict__ bits, int64_t n_words, int64_t n,
                                                                      int32_t *__restrict__ ids, int32_t *__restrict__ count)
{
    constexpr int kWaves = kOneLaunchWords / kWave;
    __shared__ unsigned total_l[kWaves];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const unsigned long long v = load_word(bits, threadIdx.x, n_words, n);
    const unsigned in = wave_inclusive_scan((unsigned)__popcll(v));
    const unsigned here = (unsigned)__builtin_amdgcn_readlane((int)in, kWave - 1);
    if (lane == 0) total_l[wave] = here;
    __syncthreads();
    unsigned at = 0u, total = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        if (w < wave) at += total_l[w];
        total += total_l[w];
    }
    if (threadIdx.x == 0) *count = (int32_t)total;
    if (here > 8 * kWave) {
        // many of them: word by word, so that a store's ids lie side by side
        const int32_t first = wave * kWave * 64 + lane;
        at = (unsigned)__builtin_amdgcn_readfirstlane((int)at);
#pragma unroll 16
        for (int l = 0; l < kWave; ++l) {
            const unsigned long long m = bcast_u64(v, l);
            int32_t *__restrict__ to = ids + at;  // (a scalar base: the lanes' part is their place in the word)
            if (__builtin_amdgcn_inverse_ballot_w64(m)) to[lane_prefix(m)] = first + 64 * l;
            at += (unsigned)__popcll(m);
        }
        return;
    }
    unsigned pos = at + in - (unsigned)__popcll(v);
    const int32_t base = (int32_t)(threadIdx.x << 6);
    unsigned long long m = v;
    while (m) {
        const int b = __ffsll((long long)m) - 1;
        m &= m - 1ull;
        ids[pos++] = base + b;
    }
}

// By which the weights of a table are known again, whatever their order: the sum of a synapse's target and weight, mixed (the finaliser
// of splitmix64, Steele, Lea and Flood 2014).
__device__ __forceinline__ unsigned long long synapse_mark(unsigned target, unsigned weight_bits)
{
    unsigned long long z = ((unsigned long long)weight_bits << 32 | target) + 0x9E3779B97F4A7C15ull;
    z = (z ^ z >> 30) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ z >> 27) * 0x94D049BB133111EBull;
    return z ^ z >> 31;
}
// One addition to device memory a workgroup, and no more workgroups than run at once: all go to one address, and take their turns there
// (one a wavefront and up to twice the workgroups: a simulator of 20,000 x 8 with 8 M synapses 2.55 ms, 1.76 so).  All threads take part.
constexpr int64_t kMarkBlocks = 2048;
__device__ __forceinline__ void add_mark(unsigned long long *mark, unsigned long long own)
{
    __shared__ unsigned long long part[kBlock / kWave];
#pragma unroll
    for (int step = kWave / 2; step > 0; step >>= 1) own += __shfl_xor(own, step, kWave);
    if (lane_id() == 0) part[threadIdx.x / kWave] = own;
    __syncthreads();
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int w = 1; w < kBlock / kWave; ++w) own += part[w];
    atomicAdd(mark, own);
}

// What 32-bit sums of arrivals have to know of a table's weights, in one pass: the lowest power of two that a set bit of some weight
// stands for, the largest size (both reduced per workgroup first), and how much could reach each target at once, in multiples of 2^-10
// rounded up.  Bounded by the additions, 44 ps each: 3.4 ms for 77 M synapses, where a count in doubles and ten array
// operations took 9 for 62 M.
__global__ __launch_bounds__(kBlock) void weight_reach_kernel(int64_t nnz, const int32_t *__restrict__ indices, const float *__restrict__ weights,
                                                              unsigned long long *__restrict__ reach, int32_t *__restrict__ found,
                                                              unsigned long long *__restrict__ mark)
{
    __shared__ int lowest_l[kBlock / kWave], largest_l[kBlock / kWave];
    int lowest = 0, largest = 0;
    unsigned long long own = 0ull;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nnz; i += (int64_t)gridDim.x * kBlock) {
        const unsigned bits = __float_as_uint(weights[i]) & 0x7FFFFFFFu, exponent = bits >> 23;
        const unsigned mantissa = (bits & 0x7FFFFFu) | (exponent ? 0x800000u : 0u);
        largest = max(largest, (int)bits);
        own += synapse_mark((unsigned)indices[i], __float_as_uint(weights[i]));
        if (mantissa == 0u) continue;
        lowest = min(lowest, (int)max(exponent, 1u) - 150 + __ffs((int)mantissa) - 1);
        // (sizes of 2^30 and more, infinities and NaN are told by found[1])
        if (bits < 0x4E800000u) atomicAdd(reach + indices[i], (unsigned long long)ceilf(__uint_as_float(bits) * 1024.0f));
    }
#pragma unroll
    for (int step = kWave / 2; step > 0; step >>= 1) {
        lowest = min(lowest, __shfl_xor(lowest, step, kWave));
        largest = max(largest, __shfl_xor(largest, step, kWave));
    }
    if (lane_id() == 0) {
        lowest_l[threadIdx.x / kWave] = lowest;
        largest_l[threadIdx.x / kWave] = largest;
    }
    add_mark(mark, own);    // (the workgroup meets there)
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int w = 1; w < kBlock / kWave; ++w) {
        lowest = min(lowest, lowest_l[w]);
        largest = max(largest, largest_l[w]);
    }
    atomicMin(found, lowest);
    atomicMax(found + 1, largest);
}

// The weights of packed records as whole numbers of 2^-k (scale = 2^k).  One read and one write of the records.
__global__ __launch_bounds__(kBlock) void pack_whole_kernel(int64_t nnz, float scale, uint2 *__restrict__ packed, unsigned long long *__restrict__ mark)
{
    unsigned long long own = 0ull;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nnz; i += (int64_t)gridDim.x * kBlock) {
        const uint2 sy = packed[i];
        own += synapse_mark(sy.x & 0xFFFFFFu, sy.y);
        packed[i].y = (unsigned)(int)(__uint_as_float(sy.y) * scale);
    }
    add_mark(mark, own);
}

// Input event lists looked over, a wavefront per step.  Bounded by launches and the one look at `found` that follows: the same in
// array operations (marks at every step's start, differences, comparisons, reductions, four of them waited for) took 270 us a
// call, 350 with repeats to list, beside runs of 1.5 to 2.3 ms; this takes 55, and 60 with repeats, 67 where a step has 2,800 events.
// 1 to 2 of those are for how often a step repeats one id.
__global__ __launch_bounds__(kBlock) void events_check_kernel(int64_t n_steps, const int64_t *__restrict__ in_ptr, int64_t n_events,
                                                              const int32_t *__restrict__ in_events, int64_t n_ids, int32_t *__restrict__ repeats,
                                                              int32_t *__restrict__ longest, unsigned *__restrict__ found)
{
    const int lane = lane_id();
    const int64_t wave = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave, n_waves = (int64_t)gridDim.x * (kBlock / kWave);
    constexpr int kTogether = 4;
    unsigned bad = 0u, total = 0u, most = 0u;
    if (wave == 0 && (in_ptr[0] != 0 || in_ptr[n_steps] != n_events)) bad = BMTK_EVENTS_INCONSISTENT;
    for (int64_t t = wave; t < n_steps; t += n_waves) {
        const int64_t p0 = in_ptr[t], p1 = in_ptr[t + 1];
        unsigned again = 0u, run = 0u, of_one = 0u;   // run: repeats of one id on end up to here
        if (p0 < 0 || p1 < p0 || p1 > n_events)
            bad |= BMTK_EVENTS_INCONSISTENT;    // (nothing is read through them)
        else
            for (int64_t base = p0; base < p1; base += kTogether * kWave) {
                int32_t id[kTogether], before[kTogether];
                unsigned long long same[kTogether], any = 0ull;
#pragma unroll
                for (int u = 0; u < kTogether; ++u) {
                    const int64_t p = min(base + u * kWave + lane, p1 - 1);
                    id[u] = in_events[p];
                    before[u] = in_events[max(p - 1, p0)];
                }
#pragma unroll
                for (int u = 0; u < kTogether; ++u) {
                    const int64_t p = base + u * kWave + lane;
                    if (p < p1 && (id[u] < 0 || id[u] >= n_ids)) bad |= BMTK_EVENTS_INCONSISTENT;
                    if (p < p1 && id[u] < before[u]) bad |= BMTK_EVENTS_UNORDERED;
                    same[u] = __ballot(p > p0 && p < p1 && id[u] == before[u]);
                    any |= same[u];
                }
                // (one branch for what is usual: a branch each made a hand-over of 2,784 events a step, 1 in 200 a repeat, 2.5 us longer)
                if (any == 0ull) {
                    run = 0u;
                    continue;
                }
#pragma unroll
                for (int u = 0; u < kTogether; ++u) {
                    unsigned long long on = same[u];
                    if (on == 0ull) {
                        run = 0u;
                        continue;
                    }
                    again += (unsigned)__popcll(on);
                    if (on == ~0ull) {
                        run += kWave;
                        of_one = max(of_one, run);
                        continue;
                    }
                    of_one = max(of_one, run + (unsigned)__ffsll((long long)~on) - 1u);
                    run = (unsigned)__clzll((long long)~on);
                    unsigned on_end = 0u;
                    for (; on; on &= on << 1) ++on_end;
                    of_one = max(of_one, on_end);
                }
            }
        if (lane == 0) {
            repeats[t] = (int32_t)again;
            longest[t] = (int32_t)of_one;
        }
        total += again;
        most = max(most, of_one);
    }
    if (bad) atomicOr(found, bad);
    if (lane == 0 && total) {
        atomicAdd(found + 1, total);
        atomicMax(found + 2, most);
    }
}

// The second and later occurrences of an id in its step, in order: those of step t from to[first[t]] on.
__global__ __launch_bounds__(kBlock) void events_repeated_kernel(int64_t n_steps, const int64_t *__restrict__ in_ptr,
                                                                 const int32_t *__restrict__ in_events, const int64_t *__restrict__ first,
                                                                 int32_t *__restrict__ to)
{
    const int lane = lane_id();
    const int64_t wave = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave, n_waves = (int64_t)gridDim.x * (kBlock / kWave);
    for (int64_t t = wave; t < n_steps; t += n_waves) {
        int64_t at = first[t];
        if (first[t + 1] == at) continue;
        const int64_t p0 = in_ptr[t], p1 = in_ptr[t + 1];
        for (int64_t base = p0; base < p1; base += kWave) {
            const int64_t p = base + lane;
            const bool same = p > p0 && p < p1 && in_events[p] == in_events[p - 1];
            const unsigned long long m = __ballot(same);
            if (same) to[at + lane_prefix(m)] = in_events[p];
            at += __popcll(m);
        }
    }
}

// ---------------------------------------------------------------------------
// Event-driven scatter: wavefronts walk the out-going synapses of the active
// elements 64 at a time (coalesced table reads), fp32 atomics into the ring.
//
// What bounds it is the chain count -> element -> row bounds -> synapses ->
// atomics; the grid is sized for every element being active, the count only
// known here.  With few active elements several wavefronts share a row (a power
// of two of them, as many as the grid holds per active element), so that a row
// of 2000 synapses is two passes of loads instead of 32 in a row.  Measured per
// call, one wavefront a row / shared (elements x synapses): 10 x 2000 17.3 / 7.7
// us, 90 x 2000 22.1 / 10.6, 400 x 2000 48 / 40, 1100 x 300 20.2 / 18.8; from some
// 300,000 events on the atomics' rate, 48 ps each, is what counts: 12000 x 300 184.
// ---------------------------------------------------------------------------

constexpr int kScatterMaxParts = 64;

// the rows of wavefront `wave` of `n_waves`
__device__ __forceinline__ void scatter_rows(const int32_t *__restrict__ active, int cnt, int batch, const Table &t, float *__restrict__ ring, int L,
                                             int64_t ne, int slot0, int n_waves, int wave)
{
    int shift = 0;
    while ((2 << shift) <= kScatterMaxParts && (int64_t)cnt * (2 << shift) <= n_waves) ++shift;
    const int parts = 1 << shift;
    for (int k = wave >> shift; k < cnt; k += n_waves >> shift) {
        const int e = active[k];
        const int j = batch == 1 ? e : (int)((uint32_t)e / (uint32_t)batch);
        deliver_row(t, j, e - j * batch, batch, ring, L, slot0, ne, wave & (parts - 1), parts);
    }
}

__global__ __launch_bounds__(kBlock) void scatter_kernel(const int32_t *__restrict__ active,
                                                         const int32_t *__restrict__ n_active, int batch, Table t,
                                                         float *__restrict__ ring, int L, int64_t ne, int slot0)
{
    scatter_rows(active, *n_active, batch, t, ring, L, ne, slot0, (int)gridDim.x * (kBlock / kWave),
                 (int)blockIdx.x * (kBlock / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave));
}

// The same sums by owners of target ranges, for steps with many events: workgroup g takes what the active rows send to targets
// g * span .. (g + 1) * span - 1, adds it up in LDS, and adds its cells to the ring at the end, sixteen neighbours to a line, where
// an atomic per event is a line per event.  `seg` (bmtk_csr_segment_offsets) only proposes where to cut a row among the workgroups: the
// cuts are held within the row's bounds as the table has them now, the first and last piece begin and end there, and a synapse whose target
// is not in its range goes to the ring by itself.  Whatever was written to the table since, every synapse of a row is delivered once.
//
// What bounds it: lines asked for by a compute unit (a piece's cuts, its row's bounds and its four arrays, 2.3 clocks each) and the chain
// count -> elements -> cuts -> synapses.  Neighbouring ranges share the lines of a row and go to one XCD: dealt out in turn, every XCD
// read every active row (16.4 us instead of 12.0 at 1,380 rows of 300 into 30,011 targets, 64 instead of 54 at 4,600 x 500 into 100,000, both
// before the row bounds were read, which costs 5 %; without them a rewritten indptr would be delivered by the rows it had before).
// us per call, an atomic per event / by ranges: 5,000 targets, 115,000 events 8.2 / 6.2; 12,000, 110,000 7.4 / 6.4; 30,011, 90,000
// 6.4 / 6.6, 414,000 22.5 / 13.2; 60,000, 90,000 6.5 / 7.4, 414,000 22.2 / 15.8; 100,000, 150,000 9.4 / 10.9, 2.3 M 114 / 56; 200,000, 150,000 9.3 / 14.2,
// 500,000 26.6 / 26.0, 2.3 M 113 / 66: below rows_min active elements it is the walk above.
constexpr int kRangeThreads = 1024;
constexpr size_t kRangeLdsMax = 150u * 1024u;
__global__ __launch_bounds__(kRangeThreads) void scatter_ranges_kernel(const int32_t *__restrict__ active, const int32_t *__restrict__ n_active,
                                                                       int batch, Table t, const uint32_t *__restrict__ seg, int span, int rows_min,
                                                                       float *__restrict__ ring, int L, int64_t n_tgt, int64_t ne, int slot0)
{
    extern __shared__ float range_l[];  // [L][4][span * batch]
    const int cnt = *n_active;
    if (cnt < rows_min) {
        scatter_rows(active, cnt, batch, t, ring, L, ne, slot0, (int)gridDim.x * (kRangeThreads / kWave),
                     (int)blockIdx.x * (kRangeThreads / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave));
        return;
    }
    // (workgroups are dealt to the eight XCDs in turn)
    const int g = (gridDim.x & 7) == 0 ? (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) : (int)blockIdx.x;
    const int n_seg = (int)gridDim.x + 1, cells = span * batch;
    const int64_t t0 = (int64_t)g * span;
    const unsigned n_here = (unsigned)max((int64_t)0, min((int64_t)span, n_tgt - t0));
    constexpr int kAhead = 4;  // synapses of a segment in flight
    struct Row {
        int b;
        unsigned p, p1;  // (unsigned: a step past the end of 2^31 - 1 synapses stays behind it)
    };
    struct __attribute__((packed, aligned(4))) Two {
        int at, to;
    };
    const int inner = g == 0 ? 0 : -1, end = g == (int)gridDim.x - 1 ? 0x7FFFFFFF : 0;  // (the first piece begins with its row, the last ends with it)
    auto look = [&](int k) {
        Row r{0, 0u, 0u};
        if (k < cnt) {
            const int e = active[k], j = batch == 1 ? e : (int)((uint32_t)e / (uint32_t)batch);
            const Two cut = *reinterpret_cast<const Two *>(seg + (int64_t)j * n_seg + g), now = *reinterpret_cast<const Two *>(t.indptr + j);
            r.b = e - j * batch;
            r.p = (unsigned)max(now.at, min(cut.at & inner, now.to));
            r.p1 = (unsigned)max(now.at, min(cut.to | end, now.to));
        }
        return r;
    };
    Row row = look(threadIdx.x);
    for (int i = threadIdx.x; i < L * GLIF3_NREC * cells; i += kRangeThreads) range_l[i] = 0.0f;
    __syncthreads();
    for (int k = threadIdx.x; k < cnt; k += kRangeThreads) {
        const Row next = look(k + kRangeThreads);
        for (unsigned p = row.p; p < row.p1; p += kAhead) {
            int i[kAhead], d[kAhead], r[kAhead];
            float w[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (p + u < row.p1) {
                    i[u] = t.indices[p + u];
                    w[u] = t.weights[p + u];
                    d[u] = t.delays[p + u];
                    r[u] = t.receptors[p + u];
                }
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (p + u >= row.p1) break;
                const int64_t in = i[u] - t0;
                int to = slot0 + d[u];
                to = to >= L ? to - L : to;
                if (in >= 0 && in < (int64_t)n_here && d[u] < L && r[u] < GLIF3_NREC)
                    atomicAdd(range_l + (to * GLIF3_NREC + r[u]) * cells + (int)in * batch + row.b, w[u]);
                else
                    atomicAdd(ring + ((int64_t)(to * GLIF3_NREC + r[u]) * ne + (int64_t)i[u] * batch + row.b), w[u]);
            }
        }
        row = next;
    }
    __syncthreads();
    // (atomically: the ring may be added to by others at the same time)
    for (int i = threadIdx.x; i < L * GLIF3_NREC * cells; i += kRangeThreads) {
        const float v = range_l[i];
        const int plane = i / cells;
        if (v != 0.0f) atomicAdd(ring + (int64_t)plane * ne + t0 * batch + (i - plane * cells), v);
    }
}

// ---------------------------------------------------------------------------
// Row-wise gather: one wavefront per target row, lane = trial.  The spike
// bits of a source over 64 trials are a native lane mask: a synapse whose
// source fired in any trial is broadcast to the wavefront and every lane whose
// trial fired adds the weight to its own accumulator (LDS, one column per
// lane, one row per (slot, receptor)).  Accumulators start from the ring cell
// on first touch and are stored back once, so every cell sees its additions
// in stored synapse order: deterministic and equal to a scalar loop.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void gather_kernel(const uint64_t *__restrict__ zbits, int batch, Table t,
                                                        float *__restrict__ ring, int L, int64_t n_tgt, int64_t ne,
                                                        int slot0)
{
    extern __shared__ float lds[];
    const int lane = lane_id();
    const int wave_in_block = threadIdx.x / kWave;
    float *acc = lds + (size_t)wave_in_block * L * GLIF3_NREC * kWave;
    const int64_t row = (int64_t)blockIdx.x * (kBlock / kWave) + wave_in_block;
    if (row >= n_tgt) return;
    const int tile0 = blockIdx.y * kWave;
    const int width = min(kWave, batch - tile0);
    const bool lane_on = lane < width;
    const int64_t cell0 = row * batch + tile0 + lane;
    unsigned long long touched = 0ull;  // bit (slot*4+r): accumulator row is live
    const int p0 = t.indptr[row], p1 = t.indptr[row + 1];
    for (int base = p0; base < p1; base += kWave) {
        const int p = base + lane;
        const bool valid = p < p1;
        float w = 0.0f;
        int dr = 0;
        unsigned long long m = 0ull;
        if (valid) {
            const int src = t.indices[p];
            w = t.weights[p];
            int slot = slot0 + (int)t.delays[p];
            slot = slot >= L ? slot - L : slot;
            dr = slot * GLIF3_NREC + (int)t.receptors[p];
            m = source_mask(zbits, src, batch, tile0, width);
        }
        unsigned long long act = __ballot(m != 0ull);
        while (act) {
            const int l = __ffsll((long long)act) - 1;
            act &= act - 1ull;
            const float wl = bcast_f(w, l);
            const int drl = bcast_i(dr, l);
            const unsigned long long ml = bcast_u64(m, l);
            float *a = acc + drl * kWave + lane;
            if (!((touched >> drl) & 1ull)) {
                touched |= 1ull << drl;
                *a = lane_on ? ring[(int64_t)drl * ne + cell0] : 0.0f;
            }
            if ((ml >> lane) & 1ull) *a += wl;
        }
    }
    while (touched) {
        const int drl = __ffsll((long long)touched) - 1;
        touched &= touched - 1ull;
        if (lane_on) ring[(int64_t)drl * ne + cell0] = acc[drl * kWave + lane];
    }
}

}  // namespace bmtk

// ===========================================================================
// C entry points
// ===========================================================================

using namespace bmtk;

// of the current device (asked for once)
static unsigned compute_units()
{
    static int count[64];
    int dev = 0;
    (void)hipGetDevice(&dev);
    int n = dev >= 0 && dev < 64 ? count[dev] : 0;
    if (n <= 0) {
        n = 256;
        (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        if (dev >= 0 && dev < 64) count[dev] = n;
    }
    return (unsigned)n;
}

extern "C" {

int bmtk_amd_abi_version(void) { return BMTK_AMD_ABI_VERSION; }

const char *bmtk_amd_last_error(void) { return g_error; }

int64_t bmtk_glif3_sim_sizeof(void) { return (int64_t)sizeof(bmtk_glif3_sim); }

int64_t bmtk_glif3_bwd_sizeof(void) { return (int64_t)sizeof(bmtk_glif3_bwd); }

int bmtk_glif3_precompute(int64_t n, const double *par, double h, float *prop, void *stream)
{
    BMTK_REQUIRE(n > 0 && par && prop, "glif3_precompute: n must be positive and pointers non-null");
    BMTK_REQUIRE(h > 0.0, "glif3_precompute: resolution h must be positive");
    const unsigned grid = (unsigned)((n + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(precompute_kernel, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, n, par, h, prop);
    BMTK_CHECK_LAUNCH("glif3_precompute");
    return BMTK_OK;
}

int bmtk_glif3_step_fwd(int64_t n_neurons, int32_t batch, float *V, float *asc, float *y1, float *y2, int32_t *ref,
                        const float *prop, int64_t prop_stride, const int32_t *class_id, float h, float *syn,
                        int32_t clear_syn, const float *i_ext, uint8_t *z, uint64_t *zbits, float *frac,
                        void *stream)
{
    BMTK_REQUIRE(n_neurons > 0 && batch > 0, "glif3_step_fwd: n_neurons and batch must be positive");
    BMTK_REQUIRE(V && asc && y1 && y2 && ref && prop, "glif3_step_fwd: state and prop pointers must be non-null");
    BMTK_REQUIRE(class_id || prop_stride >= n_neurons, "glif3_step_fwd: prop_stride smaller than n_neurons");
    BMTK_REQUIRE(prop_stride > 0, "glif3_step_fwd: prop_stride must be positive");
    BMTK_REQUIRE(h > 0.0f, "glif3_step_fwd: resolution h must be positive");
    const int64_t ne = n_neurons * (int64_t)batch;
    BMTK_REQUIRE(ne < (1ll << 31), "glif3_step_fwd: n_neurons*batch must stay below 2^31");
    StepArgs a{ne, batch, V, asc, y1, y2, ref, prop, prop_stride, class_id, h, syn, clear_syn, i_ext, z, zbits, frac};
    const unsigned grid = (unsigned)((ne + kBlock - 1) / kBlock);
    // a class table of up to 48 KB (423 classes) is staged in LDS by every workgroup (sixteen bytes per load: a
    // table that is not 16-byte aligned is read through the caches instead)
    const size_t table_bytes = (size_t)prop_stride * GLIF3_NPROP * sizeof(float);
    if (class_id && table_bytes <= 48u * 1024u && ((uintptr_t)prop & 15u) == 0) {
        const size_t fit = kLdsPerCu / ((table_bytes + kLdsUnit - 1) / kLdsUnit * kLdsUnit);
        const unsigned per_cu = fit < (size_t)kStepPerCu ? (unsigned)fit : (unsigned)kStepPerCu;
        if (grid <= per_cu * compute_units())
            hipLaunchKernelGGL(glif3_step_kernel<1>, dim3(grid), dim3(kBlock), table_bytes, (hipStream_t)stream, a);
        else
            hipLaunchKernelGGL(glif3_step_kernel<kStepTiles>, dim3((grid + kStepTiles - 1) / kStepTiles), dim3(kBlock), table_bytes,
                               (hipStream_t)stream, a);
    } else
        hipLaunchKernelGGL(glif3_step_kernel<0>, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, a);
    BMTK_CHECK_LAUNCH("glif3_step_fwd");
    return BMTK_OK;
}

static int64_t n_words_of(int64_t n) { return (n + 63) / 64; }
static int64_t n_blocks_of(int64_t n) { return (n_words_of(n) + kWordsPerBlock - 1) / kWordsPerBlock; }

int64_t bmtk_spikes_compact_workspace_bytes(int64_t n)
{
    if (n <= 0) return 0;
    // bit words (+1 padding) followed by the per-block counters
    return 8 * (n_words_of(n) + 1) + 4 * (n_blocks_of(n) + 1);
}

static int compact_from_bits(const uint64_t *bits, int64_t n, int32_t *ids, int32_t *count, uint32_t *block_count,
                             hipStream_t stream)
{
    const int64_t n_words = n_words_of(n);
    const int n_blocks = (int)n_blocks_of(n);
    if (n_words <= kOneLaunchWords) {
        hipLaunchKernelGGL(compact_one_kernel, dim3(1), dim3(kOneLaunchWords), 0, stream, bits, n_words, n, ids, count);
        BMTK_CHECK_LAUNCH("spikes_compact");
        return BMTK_OK;
    }
    if (n_blocks <= kMaxFused) {
        hipLaunchKernelGGL(compact_count_kernel, dim3(n_blocks), dim3(kBlock), 0, stream, bits, n_words, n, block_count);
        hipLaunchKernelGGL(compact_write_fused_kernel, dim3(n_blocks), dim3(kBlock), 0, stream, bits, n_words, n,
                           (const uint32_t *)block_count, ids, count);
        BMTK_CHECK_LAUNCH("spikes_compact");
        return BMTK_OK;
    }
    hipLaunchKernelGGL(compact_count_kernel, dim3(n_blocks), dim3(kBlock), 0, stream, bits, n_words, n, block_count);
    hipLaunchKernelGGL(compact_scan_kernel, dim3(1), dim3(kBlock), 0, stream, block_count, n_blocks, count);
    hipLaunchKernelGGL(compact_write_kernel, dim3(n_blocks), dim3(kBlock), 0, stream, bits, n_words, n,
                       (const uint32_t *)block_count, ids);
    BMTK_CHECK_LAUNCH("spikes_compact");
    return BMTK_OK;
}

int bmtk_spikes_compact(const uint8_t *z, int64_t n, int32_t *ids, int32_t *count, void *workspace, void *stream)
{
    BMTK_REQUIRE(n > 0 && n < (1ll << 31), "spikes_compact: n must lie in 1..2^31-1");
    BMTK_REQUIRE(z && ids && count && workspace, "spikes_compact: pointers must be non-null");
    uint64_t *bits = (uint64_t *)workspace;
    uint32_t *block_count = (uint32_t *)(bits + n_words_of(n) + 1);
    const int n_blocks = (int)n_blocks_of(n);
    if (n_blocks <= kMaxFused && (reinterpret_cast<uintptr_t>(z) & 15u) == 0) {
        hipLaunchKernelGGL(compact_count_flags_kernel, dim3(n_blocks), dim3(kBlock), 0, (hipStream_t)stream, z, n,
                           n_words_of(n), bits, block_count);
        hipLaunchKernelGGL(compact_write_fused_kernel, dim3(n_blocks), dim3(kBlock), 0, (hipStream_t)stream,
                           (const uint64_t *)bits, n_words_of(n), n, (const uint32_t *)block_count, ids, count);
        BMTK_CHECK_LAUNCH("spikes_compact");
        return BMTK_OK;
    }
    const unsigned grid = (unsigned)((n + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(pack_bits_kernel, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, z, n, bits);
    return compact_from_bits(bits, n, ids, count, block_count, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// The same compaction with the workspace inside the library: a file-scope
// device array, so that the call allocates nothing.  In host code the array's
// name is only a handle; its device address is asked for once per device, with
// that device current, and kept.
// ---------------------------------------------------------------------------

constexpr int64_t kNoAllocBytes = 8 * (BMTK_COMPACT_NOALLOC_MAX_N / 64 + 1) +
                                  4 * (BMTK_COMPACT_NOALLOC_MAX_N / 64 / kWordsPerBlock + 2);
static __device__ __align__(256) unsigned char scratch[(kNoAllocBytes + 255) / 256 * 256];

constexpr int kMaxDevices = 64;
static void *g_scratch_ptr[kMaxDevices];  // device address of `scratch` on every device seen so far
static std::mutex g_scratch_mutex;

// device address of this device's copy of `scratch`, or nullptr with the error message set
static void *scratch_of_current_device()
{
    int dev = -1;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("spikes_compact_noalloc: cannot tell the current device (%s)", hipGetErrorString(err));
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !ptr) {
            set_error("spikes_compact_noalloc: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(err));
            return nullptr;
        }
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

int bmtk_spikes_compact_noalloc(const uint8_t *z, int64_t n, int32_t *ids, int32_t *count, void *stream)
{
    BMTK_REQUIRE(n > 0, "spikes_compact_noalloc: n must be positive");
    BMTK_REQUIRE(n <= BMTK_COMPACT_NOALLOC_MAX_N,
                 "spikes_compact_noalloc: n = %lld exceeds the %lld elements the built-in workspace holds; use "
                 "bmtk_spikes_compact with a workspace of the caller's", (long long)n,
                 (long long)BMTK_COMPACT_NOALLOC_MAX_N);
    BMTK_REQUIRE(z && ids && count, "spikes_compact_noalloc: pointers must be non-null");
    static_assert(kNoAllocBytes >= 8 * ((BMTK_COMPACT_NOALLOC_MAX_N + 63) / 64 + 1) +
                                       4 * (((BMTK_COMPACT_NOALLOC_MAX_N + 63) / 64 + kWordsPerBlock - 1) / kWordsPerBlock + 1),
                  "scratch smaller than bmtk_spikes_compact_workspace_bytes(BMTK_COMPACT_NOALLOC_MAX_N)");
    void *ws = scratch_of_current_device();
    if (!ws) return BMTK_E_DEVICE;
    // every word of the workspace a kernel reads is written earlier in the same call, so what the call before
    // left behind does not matter and nothing has to be cleared
    return bmtk_spikes_compact(z, n, ids, count, ws, stream);
}

int bmtk_spikes_compact_bits(const uint64_t *zbits, int64_t n, int32_t *ids, int32_t *count, void *workspace,
                             void *stream)
{
    BMTK_REQUIRE(n > 0 && n < (1ll << 31), "spikes_compact_bits: n must lie in 1..2^31-1");
    BMTK_REQUIRE(zbits && ids && count && workspace, "spikes_compact_bits: pointers must be non-null");
    uint32_t *block_count = (uint32_t *)((uint64_t *)workspace + n_words_of(n) + 1);
    return compact_from_bits(zbits, n, ids, count, block_count, (hipStream_t)stream);
}

int bmtk_csr_weight_reach(int64_t nnz, const int32_t *indices, const float *weights, uint64_t *reach, int32_t *found, uint64_t *mark, void *stream)
{
    BMTK_REQUIRE(nnz >= 0 && found && reach && mark && (nnz == 0 || (indices && weights)), "csr_weight_reach: bad sizes or null pointers");
    if (nnz == 0) return BMTK_OK;
    const int64_t blocks = (nnz + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(weight_reach_kernel, dim3((unsigned)(blocks < kMarkBlocks ? blocks : kMarkBlocks)), dim3(kBlock), 0, (hipStream_t)stream, nnz, indices,
                       weights, reinterpret_cast<unsigned long long *>(reach), found, reinterpret_cast<unsigned long long *>(mark));
    BMTK_CHECK_LAUNCH("csr_weight_reach");
    return BMTK_OK;
}

int bmtk_csr_pack_whole(int64_t nnz, int32_t k, bmtk_synapse *packed, uint64_t *mark, void *stream)
{
    BMTK_REQUIRE(nnz >= 0 && k >= 0 && k <= 30 && mark && (nnz == 0 || packed), "csr_pack_whole: bad sizes or null pointers");
    if (nnz == 0) return BMTK_OK;
    const int64_t blocks = (nnz + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(pack_whole_kernel, dim3((unsigned)(blocks < kMarkBlocks ? blocks : kMarkBlocks)), dim3(kBlock), 0, (hipStream_t)stream, nnz, ldexpf(1.0f, k),
                       reinterpret_cast<uint2 *>(packed), reinterpret_cast<unsigned long long *>(mark));
    BMTK_CHECK_LAUNCH("csr_pack_whole");
    return BMTK_OK;
}

int bmtk_events_check(int64_t n_steps, const int64_t *in_ptr, int64_t n_events, const int32_t *in_events, int64_t n_ids, int32_t *repeats,
                      int32_t *longest, uint32_t *found, void *stream)
{
    BMTK_REQUIRE(n_steps >= 0 && n_events >= 0 && n_ids >= 0, "events_check: bad sizes");
    BMTK_REQUIRE(in_ptr && (in_events || n_events == 0) && ((repeats && longest) || n_steps == 0) && found, "events_check: pointers must be non-null");
    const int64_t blocks = (n_steps + kBlock / kWave - 1) / (kBlock / kWave);
    hipLaunchKernelGGL(events_check_kernel, dim3((unsigned)(blocks < 1 ? 1 : blocks < 8192 ? blocks : 8192)), dim3(kBlock), 0, (hipStream_t)stream,
                       n_steps, in_ptr, n_events, in_events, n_ids, repeats, longest, found);
    BMTK_CHECK_LAUNCH("events_check");
    return BMTK_OK;
}

int bmtk_events_repeated(int64_t n_steps, const int64_t *in_ptr, const int32_t *in_events, const int64_t *first, int32_t *to, void *stream)
{
    BMTK_REQUIRE(n_steps > 0, "events_repeated: bad sizes");
    BMTK_REQUIRE(in_ptr && in_events && first && to, "events_repeated: pointers must be non-null");
    const int64_t blocks = (n_steps + kBlock / kWave - 1) / (kBlock / kWave);
    hipLaunchKernelGGL(events_repeated_kernel, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(kBlock), 0, (hipStream_t)stream, n_steps,
                       in_ptr, in_events, first, to);
    BMTK_CHECK_LAUNCH("events_repeated");
    return BMTK_OK;
}

int bmtk_csr_propagate_scatter(const int32_t *active, const int32_t *n_active, int64_t max_active, int32_t batch,
                               const int32_t *indptr, const int32_t *indices, const float *weights,
                               const uint8_t *delays, const uint8_t *receptors, float *ring, int32_t L,
                               int64_t n_tgt, int64_t step, void *stream)
{
    BMTK_REQUIRE(active && n_active && indptr && indices && weights && delays && receptors && ring,
                 "csr_propagate_scatter: pointers must be non-null");
    BMTK_REQUIRE(batch > 0 && n_tgt > 0 && L > 1 && step >= 0, "csr_propagate_scatter: bad batch, n_tgt, L or step");
    BMTK_REQUIRE(n_tgt * (int64_t)batch < (1ll << 31), "csr_propagate_scatter: n_tgt*batch must stay below 2^31");
    if (max_active <= 0) return BMTK_OK;
    // (a short list gets wavefronts to share its rows among, too)
    const int64_t waves = max_active < 8192 / 16 ? max_active * 16 : 8192;
    const unsigned grid = (unsigned)((waves + kBlock / kWave - 1) / (kBlock / kWave));
    Table t{indptr, indices, weights, delays, receptors};
    hipLaunchKernelGGL(scatter_kernel, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, active, n_active, batch, t,
                       ring, L, n_tgt * (int64_t)batch, (int)(step % L));
    BMTK_CHECK_LAUNCH("csr_propagate_scatter");
    return BMTK_OK;
}

int bmtk_csr_propagate_scatter_ranges(const int32_t *active, const int32_t *n_active, int32_t batch, const int32_t *indptr, const int32_t *indices,
                                      const float *weights, const uint8_t *delays, const uint8_t *receptors, const uint32_t *seg, int32_t span,
                                      int32_t n_ranges, int32_t rows_min, float *ring, int32_t L, int64_t n_tgt, int64_t step, void *stream)
{
    BMTK_REQUIRE(active && n_active && indptr && indices && weights && delays && receptors && seg && ring,
                 "csr_propagate_scatter_ranges: pointers must be non-null");
    BMTK_REQUIRE(batch > 0 && n_tgt > 0 && L > 1 && step >= 0, "csr_propagate_scatter_ranges: bad batch, n_tgt, L or step");
    BMTK_REQUIRE(n_tgt * (int64_t)batch < (1ll << 31), "csr_propagate_scatter_ranges: n_tgt*batch must stay below 2^31");
    BMTK_REQUIRE(span > 0 && n_ranges > 0 && n_ranges <= 65536 && (int64_t)span * n_ranges >= n_tgt && rows_min >= 0,
                 "csr_propagate_scatter_ranges: the ranges must cover the targets, rows_min must not be negative");
    BMTK_REQUIRE((int64_t)L * GLIF3_NREC * span * batch * 4 <= (int64_t)kRangeLdsMax,
                 "csr_propagate_scatter_ranges: the cells of a range (L * 4 * span * batch * 4 bytes) must fit %zu bytes of LDS", kRangeLdsMax);
    static bool asked[kMaxDevices];
    int dev = -1;
    (void)hipGetDevice(&dev);
    if (dev < 0 || dev >= kMaxDevices || !asked[dev]) {
        const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void *>(scatter_ranges_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)kRangeLdsMax);
        if (err != hipSuccess) {
            set_error("csr_propagate_scatter_ranges: cannot reserve LDS: %s", hipGetErrorString(err));
            return BMTK_E_LAUNCH;
        }
        if (dev >= 0 && dev < kMaxDevices) asked[dev] = true;
    }
    Table t{indptr, indices, weights, delays, receptors};
    hipLaunchKernelGGL(scatter_ranges_kernel, dim3((unsigned)n_ranges), dim3(kRangeThreads), (size_t)L * GLIF3_NREC * span * batch * sizeof(float),
                       (hipStream_t)stream, active, n_active, batch, t, seg, span, rows_min, ring, L, n_tgt, n_tgt * (int64_t)batch, (int)(step % L));
    BMTK_CHECK_LAUNCH("csr_propagate_scatter_ranges");
    return BMTK_OK;
}

int bmtk_csr_propagate_gather(const uint64_t *zbits, int64_t n_src, int32_t batch, const int32_t *indptr,
                              const int32_t *indices, const float *weights, const uint8_t *delays,
                              const uint8_t *receptors, float *ring, int32_t L, int64_t n_tgt, int64_t step,
                              void *stream)
{
    BMTK_REQUIRE(zbits && indptr && indices && weights && delays && receptors && ring,
                 "csr_propagate_gather: pointers must be non-null");
    BMTK_REQUIRE(batch > 0 && n_tgt > 0 && n_src > 0 && step >= 0, "csr_propagate_gather: bad batch, sizes or step");
    BMTK_REQUIRE(L > 1 && L <= 16, "csr_propagate_gather: ring_slots must lie in 2..16");
    BMTK_REQUIRE(n_tgt * (int64_t)batch < (1ll << 31), "csr_propagate_gather: n_tgt*batch must stay below 2^31");
    const unsigned rows_per_block = kBlock / kWave;
    const dim3 grid((unsigned)((n_tgt + rows_per_block - 1) / rows_per_block), (unsigned)((batch + kWave - 1) / kWave));
    BMTK_REQUIRE(grid.y <= 65535, "csr_propagate_gather: batch too large");
    const size_t lds = (size_t)rows_per_block * L * GLIF3_NREC * kWave * sizeof(float);
    Table t{indptr, indices, weights, delays, receptors};
    hipLaunchKernelGGL(gather_kernel, grid, dim3(kBlock), lds, (hipStream_t)stream, zbits, batch, t, ring, L, n_tgt,
                       n_tgt * (int64_t)batch, (int)(step % L));
    BMTK_CHECK_LAUNCH("csr_propagate_gather");
    return BMTK_OK;
}

}  // extern "C"
