// Reverse-time adjoint of the forward simulation: transposed propagation,
// state adjoint, event-driven weight gradients.  The differentiable model
// these kernels transpose is stated in include/bmtk_amd.h (bmtk_glif3_bwd).
#include <type_traits>

#include "common.hpp"
#include "glif3_update.hpp"

namespace bmtk {

struct BwdStep {
    int64_t t;    // absolute step being differentiated
    int64_t row;  // its row in the forward record
    int parts;    // partial sums gz[parts][ne] that the transposed propagation left (1, or 8 from the blocked form)
    int slot;     // t % ring_slots (divided on the host: a 64-bit remainder is 150 scalar instructions, one after the other)
};

__device__ __forceinline__ float surrogate(float U, float th, float dampening)
{
    const float vhat = (U - th) / th;
    return dampening * fmaxf(0.0f, 1.0f - fabsf(vhat)) / th;
}

__device__ __forceinline__ unsigned long long trial_mask(const uint64_t *__restrict__ bits, int64_t j, int batch,
                                                         int tile0, int width)
{
    const int64_t bit = j * batch + tile0;
    const int64_t w = bit >> 6;
    const int sh = (int)(bit & 63);
    unsigned long long m = bits[w] >> sh;
    if (sh + width > 64) m |= bits[w + 1] << (64 - sh);
    if (width < 64) m &= (1ull << width) - 1ull;
    return m;
}

// gz[j*B+b] = sum over out-going synapses (j -> i, w, d, r) of w * lam_ring[(t+d)%L][r][i*B+b]:
// one wavefront per source neuron and trial tile.  A tile is `bp` trials wide
// (the batch rounded up to a power of two, at most 64) and the wavefront's 64
// lanes hold 64/bp synapses side by side, each lane reading one trial of one
// synapse's adjoint row (bp*4 contiguous bytes per synapse); four such groups
// are in flight before their products are added.  Rows whose every trial has
// a zero surrogate derivative in this step are skipped.
// kGrad (batches of one tile only): the recurrent weight gradient of the step rides along.  The wavefront has a
// synapse's adjoint row in registers anyway; where the source fired in some trial of this step, the entries of
// those trials are summed over the row's lanes and added to d_rec_w[p] -- this wavefront is the only writer of
// its row.  A separate kernel would fetch every such adjoint row a second time to use one or two words of it.
template <bool kGrad>
__global__ __launch_bounds__(kBlock) void bwd_gather_kernel(bmtk_glif3_bwd a, BwdStep q, int bp)
{
    const int batch = a.batch;
    const int64_t ne = a.n_neurons * (int64_t)batch;
    const int L = a.ring_slots;
    const int lane = lane_id();
    const int64_t j = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (j >= a.n_neurons) return;
    const int per = kWave / bp;  // synapses per wavefront instruction
    const int sub = lane / bp, b = lane - sub * bp;
    const int tile0 = blockIdx.y * kWave;
    const bool lane_on = tile0 + b < batch;
    const int64_t e = j * batch + tile0 + b;
    bool active = lane_on && a.save_flags == nullptr;  // without a forward record every element counts
    if (lane_on && a.save_flags) {
        const uint8_t f = a.save_flags[q.row * ne + e];
        if (f & BMTK_F_INTEGRATING) {
            const int64_t col = a.class_id ? (int64_t)a.class_id[j] : j;
            const float th = a.prop[GLIF3_TH * a.prop_stride + col];
            active = fabsf((a.save_v[q.row * ne + e] - th) / th) < 1.0f;
        }
    }
    // trials in which source j fired in this step (the same in all lanes)
    const unsigned long long fired = kGrad ? trial_mask(a.spike_bits + q.row * a.spike_bits_stride, j, batch, 0, batch) : 0ull;
    const bool mine = lane_on && ((fired >> b) & 1ull);
    if (__ballot(active) == 0ull && fired == 0ull) {
        if (lane_on && sub == 0) a.gz[e] = 0.0f;
        return;
    }
    const int slot0 = q.slot;
    const int p0 = a.rec_indptr[j], p1 = a.rec_indptr[j + 1];
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(a.rec_packed);
    const float *__restrict__ ring = a.lam_ring + tile0 + b;
    constexpr int kInFlight = 4;
    float acc = 0.0f;
    for (int base = p0; base < p1; base += kWave) {
        const int p = base + lane;
        uint2 sy = make_uint2(0u, 0u);
        if (p < p1) sy = rows[p];
        const int n_here = min(kWave, p1 - base);
        for (int l0 = 0; l0 < n_here; l0 += per * kInFlight) {
            float w[kInFlight], v[kInFlight];
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                const int idx = l0 + u * per + sub;
                const unsigned tdr = (unsigned)__shfl((int)sy.x, idx & (kWave - 1), kWave);
                w[u] = __uint_as_float((unsigned)__shfl((int)sy.y, idx & (kWave - 1), kWave));
                int slot = slot0 + (int)(tdr >> 26);
                slot = slot >= L ? slot - L : slot;
                const int r = (tdr >> 24) & 3;
                const int64_t i = tdr & 0xFFFFFFu;
                v[u] = ((active || mine) && idx < n_here) ? ring[(int64_t)(slot * GLIF3_NREC + r) * ne + i * batch] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) acc += active ? w[u] * v[u] : 0.0f;
            if (kGrad && fired != 0ull) {
#pragma unroll
                for (int u = 0; u < kInFlight; ++u) {
                    float g = mine ? v[u] : 0.0f;
                    for (int off = 1; off < bp; off <<= 1) g += __shfl_xor(g, off, kWave);
                    const int idx = l0 + u * per + sub;
                    if (b == 0 && idx < n_here) a.d_rec_w[base + idx] += g;
                }
            }
        }
    }
    for (int off = bp; off < kWave; off <<= 1) acc += __shfl_xor(acc, off, kWave);
    if (lane_on && sub == 0) a.gz[e] = acc;
}

// The same sums with four trials per lane, for batches that are a multiple of 4 and at most 64: a synapse's
// adjoint row (batch*4 contiguous bytes) is read by lp = bp/4 lanes as 16-byte pieces, so one wavefront
// instruction covers 64/lp synapses (8 at batch 32) and the address arithmetic and lane exchanges per synapse
// shrink fourfold.  Partial sums of the 64/lp synapse lanes are folded at the end.
template <bool kGrad>
__global__ __launch_bounds__(kBlock) void bwd_gather4_kernel(bmtk_glif3_bwd a, BwdStep q, int lp)
{
    const int batch = a.batch;
    const int64_t ne = a.n_neurons * (int64_t)batch;
    const int L = a.ring_slots;
    const int lane = lane_id();
    const int64_t j = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (j >= a.n_neurons) return;
    const int per = kWave / lp;  // synapses per wavefront instruction
    const int sub = lane / lp, b4 = (lane - sub * lp) * 4;
    const bool lane_on = b4 < batch;
    const int64_t e = j * batch + b4;
    unsigned act = (lane_on && a.save_flags == nullptr) ? 0xFu : 0u;  // bit c: trial b4+c has a non-zero surrogate derivative in this step
    if (lane_on && a.save_flags) {
        const uint32_t f4 = *reinterpret_cast<const uint32_t *>(a.save_flags + q.row * ne + e);
        const float4 v4 = *reinterpret_cast<const float4 *>(a.save_v + q.row * ne + e);
        const int64_t col = a.class_id ? (int64_t)a.class_id[j] : j;
        const float th = a.prop[GLIF3_TH * a.prop_stride + col];
        const float v[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (((f4 >> (8 * c)) & BMTK_F_INTEGRATING) && fabsf((v[c] - th) / th) < 1.0f) act |= 1u << c;
    }
    // trials in which source j fired in this step (the same in all lanes), and this lane's four of them
    const unsigned long long fired = kGrad ? trial_mask(a.spike_bits + q.row * a.spike_bits_stride, j, batch, 0, batch) : 0ull;
    const unsigned mine = lane_on ? (unsigned)(fired >> b4) & 0xFu : 0u;
    if (__ballot(act != 0u) == 0ull && fired == 0ull) {
        if (lane_on && sub == 0) *reinterpret_cast<float4 *>(a.gz + e) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const int slot0 = q.slot;
    const int p0 = a.rec_indptr[j], p1 = a.rec_indptr[j + 1];
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(a.rec_packed);
    const float *__restrict__ ring = a.lam_ring + b4;
    constexpr int kInFlight = 4;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int base = p0; base < p1; base += kWave) {
        const int p = base + lane;
        uint2 sy = make_uint2(0u, 0u);
        if (p < p1) sy = rows[p];
        const int n_here = min(kWave, p1 - base);
        for (int l0 = 0; l0 < n_here; l0 += per * kInFlight) {
            float w[kInFlight];
            float4 v[kInFlight];
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                const int idx = l0 + u * per + sub;
                const unsigned tdr = (unsigned)__shfl((int)sy.x, idx & (kWave - 1), kWave);
                w[u] = __uint_as_float((unsigned)__shfl((int)sy.y, idx & (kWave - 1), kWave));
                int slot = slot0 + (int)(tdr >> 26);
                slot = slot >= L ? slot - L : slot;
                const int r = (tdr >> 24) & 3;
                const int64_t i = tdr & 0xFFFFFFu;
                v[u] = ((act | mine) != 0u && idx < n_here)
                           ? *reinterpret_cast<const float4 *>(ring + (int64_t)(slot * GLIF3_NREC + r) * ne + i * batch)
                           : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                acc[0] += w[u] * v[u].x;
                acc[1] += w[u] * v[u].y;
                acc[2] += w[u] * v[u].z;
                acc[3] += w[u] * v[u].w;
            }
            if (kGrad && fired != 0ull) {
#pragma unroll
                for (int u = 0; u < kInFlight; ++u) {
                    float g = ((mine & 1u) ? v[u].x : 0.0f) + ((mine & 2u) ? v[u].y : 0.0f) +
                              ((mine & 4u) ? v[u].z : 0.0f) + ((mine & 8u) ? v[u].w : 0.0f);
                    for (int off = 1; off < lp; off <<= 1) g += __shfl_xor(g, off, kWave);
                    const int idx = l0 + u * per + sub;
                    if (b4 == 0 && idx < n_here) a.d_rec_w[base + idx] += g;
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        for (int off = lp; off < kWave; off <<= 1) acc[c] += __shfl_xor(acc[c], off, kWave);
    if (lane_on && sub == 0)
        *reinterpret_cast<float4 *>(a.gz + e) = make_float4((act & 1u) ? acc[0] : 0.0f, (act & 2u) ? acc[1] : 0.0f,
                                                            (act & 4u) ? acc[2] : 0.0f, (act & 8u) ? acc[3] : 0.0f);
}

// The same sums through the table regrouped by target range, for networks whose adjoint ring is far larger than an
// L2.  bwd_gather4_kernel visits the adjoint rows of a source's targets all over the ring: at 52k neurons x 32
// trials the ring is 133 MB, every 128-byte row misses the 4 MB L2 of its XCD and the kernel runs at the rate the
// fabric fills L2 lines (6.4 GB per step).  Here the targets are cut into blk_count ranges whose slice of the ring
// (all slots and receptors) fits an L2, and the table holds, range after range, a CSR over the sources of the
// synapses into that range.  Workgroup b runs on XCD b % 8 (workgroups are dealt to the XCDs in turn) and takes
// the ranges x*P .. x*P+P-1, one after the other, over a fixed share of the source rows, so that while an XCD
// works through a range its L2 holds that slice and each adjoint row is fetched from memory once per sweep
// instead of once per synapse.  A lane group of lp lanes (4 trials each) owns one source row; its partial sum
// over the ranges seen so far waits in LDS (16 bytes per lane and row, lane-private, so no barriers), which is
// what bounds the rows of a sweep: 16 wavefronts x gpw row groups x 64/lp rows.  The eight XCDs each see every
// row for their own ranges and write a partial sum of their own, gz[x][ne]; the state adjoint adds the eight.
__device__ __forceinline__ void bwd_inp_grad_waves(const bmtk_glif3_bwd &a, const BwdStep &q, int wave, int n_waves);
__device__ __forceinline__ void bwd_inp_grad2_waves(const bmtk_glif3_bwd &a, const BwdStep &q, int wave, int n_waves);
constexpr int kBlkThreads = 1024;
constexpr int kBlkWaves = kBlkThreads / kWave;
constexpr int kBlkMaxGroups = 8;  // row groups per wavefront and sweep: one byte of trial masks each in a 64-bit register
constexpr int kBlkInFlight = 8;   // synapses of a row in flight
static_assert(kBlkInFlight % 8 == 0 && 2 * kBlkInFlight <= BMTK_BLOCKED_PAD, "the kernel reads up to 2*kBlkInFlight - 1 records past a row's end");

// the value of `x` in the lane a data-parallel-primitive control word names (all of the ones used here have a source)
template <int kCtrl>
__device__ __forceinline__ float dpp_move(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xF, 0xF, false));
}

// kNe24: n_neurons*batch < 2^24, so that the cell arithmetic can use 24-bit multiplies; kWide: lp >= 8
template <bool kGrad, bool kNe24, bool kWide>
__global__ __launch_bounds__(kBlkThreads) void bwd_gather_blocked_kernel(bmtk_glif3_bwd a, BwdStep q, int lp, int rows_cu,
                                                                         int sweeps, int gpw, int use_order, int do_inp)
{
    extern __shared__ float4 blk_acc[];  // [kBlkWaves][gpw][kWave], then the row order (uint16 per place)
    constexpr int kF = kBlkInFlight;
    const int batch = a.batch;
    const int64_t n = a.n_neurons, ne = n * batch;
    const int L = a.ring_slots;
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const int x = blockIdx.x & 7;
    const int P = a.blk_count >> 3;
    const int per = kWave / lp;  // rows a wavefront works on side by side
    const int grp = lane / lp, b4 = (lane - grp * lp) * 4;
    const bool lane_on = b4 < batch;
    const unsigned long long grp_lanes = (lp == kWave ? ~0ull : ((1ull << lp) - 1ull)) << (grp * lp);
    const int64_t row_lo = (int64_t)(blockIdx.x >> 3) * rows_cu;
    const int64_t row_hi = row_lo + rows_cu < n ? row_lo + rows_cu : n;
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(a.blk_packed);
    // byte offset of a synapse's adjoint cell from the start of the ring, in 32 bits: the record's upper byte is
    // delay*4 + receptor, so (slot0 + delay) % L * 4 + receptor = min(u, u - 4L) with u = slot0*4 + that byte
    const char *__restrict__ ring = reinterpret_cast<const char *>(a.lam_ring);
    const unsigned lane_off = (unsigned)b4 * 4u;
    const unsigned q_lo = (unsigned)q.slot * 4u, q_wrap = q_lo - 4u * (unsigned)L;
    const unsigned ne32 = (unsigned)ne, batch32 = (unsigned)batch;
    auto cell_off = [&](unsigned tdr) -> unsigned {
        const unsigned dq = tdr >> 24;
        const unsigned plane = min(dq + q_lo, dq + q_wrap);
        const unsigned elem = mad_u24(tdr, batch32, kNe24 ? mul_u24(plane, ne32) : plane * ne32);  // bits 24-31 of tdr do not count
        return (elem << 2) + lane_off;
    };
    float4 *acc = blk_acc + (size_t)wave * gpw * kWave + lane;
    // Which row a lane group works on.  The workgroup's rows are taken in groups of `per` (a wavefront's lane groups
    // side by side), group g by wavefront g % 16 as its (g / 16)-th.  With the gradient riding along, the rows
    // whose source fired in this step come first in that order (a list in LDS, built once per launch): a wavefront
    // runs the gradient's extra work whenever ONE of its rows fired, so with a tenth of the rows firing and eight
    // rows side by side more than half of all visits ran it, seven eighths idle; gathered into the first groups
    // the fired rows fill a tenth of the visits, dealt out evenly over the wavefronts.
    uint16_t *order = reinterpret_cast<uint16_t *>(blk_acc + (size_t)kBlkWaves * gpw * kWave);
    const int places = sweeps * kBlkWaves * gpw * per;
    if (kGrad && use_order) {
        __shared__ unsigned scan_l[2][kBlkWaves];
        const uint64_t *__restrict__ bits = a.spike_bits + q.row * a.spike_bits_stride;
        // a thread looks at rows threadIdx.x, threadIdx.x + 1024, ... (at most 16): fired or not, one bit each
        unsigned fm = 0u, n_mine = 0u;
        for (int i = 0; (int)threadIdx.x + i * kBlkThreads < rows_cu; ++i) {
            const int64_t j = row_lo + threadIdx.x + i * kBlkThreads;
            if (j < row_hi && trial_mask(bits, j, batch, 0, batch) != 0ull) fm |= 1u << i;
            ++n_mine;
        }
        const unsigned c1 = (unsigned)__popc(fm), c0 = n_mine - c1;
        const unsigned in1 = wave_inclusive_scan(c1), in0 = wave_inclusive_scan(c0);
        if (lane == kWave - 1) {
            scan_l[0][wave] = in0;
            scan_l[1][wave] = in1;
        }
        __syncthreads();
        unsigned base0 = 0u, base1 = 0u, total1 = 0u;
#pragma unroll
        for (int w = 0; w < kBlkWaves; ++w) {
            if (w < wave) {
                base0 += scan_l[0][w];
                base1 += scan_l[1][w];
            }
            total1 += scan_l[1][w];
        }
        unsigned p1 = base1 + in1 - c1, p0 = total1 + base0 + in0 - c0;  // next place among the fired / the others
        for (unsigned i = 0; i < n_mine; ++i) {
            const unsigned local = threadIdx.x + i * kBlkThreads;
            if ((fm >> i) & 1u)
                order[p1++] = (uint16_t)local;
            else
                order[p0++] = (uint16_t)local;
        }
        for (int i = rows_cu + (int)threadIdx.x; i < places; i += kBlkThreads) order[i] = 0xFFFFu;  // places without a row
        __syncthreads();
    }
    // row of lane group `grp` in the wavefront's k-th group of sweep sw (row_hi and beyond: none)
    auto row_of = [&](int sw, int k) -> int64_t {
        const int place = ((sw * gpw + k) * kBlkWaves + wave) * per + grp;
        if (kGrad && use_order) {
            const unsigned local = order[place];
            return local == 0xFFFFu ? row_hi : row_lo + local;
        }
        return place < rows_cu ? row_lo + place : row_hi;
    };
    for (int sw = 0; sw < sweeps; ++sw) {
        // per row group one byte: bits 0-3 the lane's trials with a non-zero surrogate derivative in this step,
        // bits 4-7 those in which the source fired (kGrad)
        unsigned long long masks = 0ull;
        for (int k = 0; k < gpw; ++k) {
            const int64_t j = row_of(sw, k);
            unsigned act = 0u, mine = 0u;
            if (j < row_hi && lane_on) {
                const int64_t e = j * batch + b4;
                if (a.save_flags) {
                    const uint32_t f4 = *reinterpret_cast<const uint32_t *>(a.save_flags + q.row * ne + e);
                    const float4 v4 = *reinterpret_cast<const float4 *>(a.save_v + q.row * ne + e);
                    const int64_t col = a.class_id ? (int64_t)a.class_id[j] : j;
                    const float th = a.prop[GLIF3_TH * a.prop_stride + col];
                    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (((f4 >> (8 * c)) & BMTK_F_INTEGRATING) && fabsf((v[c] - th) / th) < 1.0f) act |= 1u << c;
                } else {
                    act = 0xFu;
                }
                if (kGrad)
                    mine = (unsigned)(trial_mask(a.spike_bits + q.row * a.spike_bits_stride, j, batch, 0, batch) >> b4) & 0xFu;
            }
            masks |= (unsigned long long)(act | (mine << 4)) << (8 * k);
            acc[k * kWave] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        // the synapses this lane's row of group k sends into range ph: [p, p1); empty for rows none of whose
        // trials needs them, and for rows past the end
        auto row_range = [&](int ph, int k, int &p, int &p1) {
            p = p1 = 0;
            if (ph >= P) return;
            const bool want = ((masks >> (8 * k)) & 0xFFull) != 0ull;
            const int64_t j = row_of(sw, k);
            if ((__ballot(want) & grp_lanes) != 0ull && j < row_hi) {
                const int32_t *__restrict__ ip = a.blk_indptr + (int64_t)(x * P + ph) * n + j;
                p = ip[0];
                p1 = ip[1];
            }
        };
        int p_next, p1_next;
        row_range(0, 0, p_next, p1_next);
        for (int ph = 0; ph < P; ++ph) {
            for (int k = 0; k < gpw; ++k) {
                int p = p_next;
                const int p1 = p1_next;
                row_range(k + 1 < gpw ? ph : ph + 1, k + 1 < gpw ? k + 1 : 0, p_next, p1_next);  // asked for a visit ahead
                if (__ballot(p < p1) == 0ull) continue;
                const unsigned mine = (unsigned)(masks >> (8 * k + 4)) & 0xFu;
                const int p1_lane = ((masks >> (8 * k)) & 0xFFull) != 0ull ? p1 : 0;  // lanes none of whose trials counts stay idle
                const bool row_fired = kGrad && (__ballot(mine != 0u) & grp_lanes) != 0ull;
                const float fired_f[4] = {(mine & 1u) ? 1.0f : 0.0f, (mine & 2u) ? 1.0f : 0.0f, (mine & 4u) ? 1.0f : 0.0f,
                                          (mine & 8u) ? 1.0f : 0.0f};
                const int in_row = lane - grp * lp;  // this lane's place among its row's lanes
                float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                // kF synapses of the row at a time: their adjoint rows are asked for, then the row's next kF
                // records (which arrive while the adjoint rows are on their way), then the products are added.
                // Lanes past the row's end read the ring's first cell with weight 0 -- no branches around loads.
                auto visit = [&](auto fetch, auto record) {
                    auto cur = fetch(0), nxt = cur;
                    auto work = [&](const decltype(cur) &have, decltype(cur) &ahead) {
                        float4 v[kF];
                        float w[kF];
#pragma unroll
                        for (int u = 0; u < kF; ++u) {
                            const uint2 sy = record(have, u);
                            const bool valid = p + u < p1_lane;
                            const unsigned off = valid ? cell_off(sy.x) : lane_off;
                            w[u] = valid ? __uint_as_float(sy.y) : 0.0f;
                            v[u] = *reinterpret_cast<const float4 *>(ring + off);
                        }
                        ahead = fetch(kF);
#pragma unroll
                        for (int u = 0; u < kF; ++u) {
                            s.x = fmaf(w[u], v[u].x, s.x);
                            s.y = fmaf(w[u], v[u].y, s.y);
                            s.z = fmaf(w[u], v[u].z, s.z);
                            s.w = fmaf(w[u], v[u].w, s.w);
                        }
                        if (kGrad && __ballot(row_fired && p < p1) != 0ull) {
                            if (kWide) {
                                // the gradient of record u is the sum, over the row's lanes, of the adjoint entries of
                                // the trials in which the source fired; every lane gets every sum (data-parallel
                                // moves within quads, half rows and rows of 16 lanes) and keeps the one of the
                                // record it then updates: one read-modify-write for the kF records of all rows
                                float keep = 0.0f;
#pragma unroll
                                for (int u = 0; u < kF; ++u) {
                                    float g = fmaf(fired_f[3], v[u].w, fmaf(fired_f[2], v[u].z, fmaf(fired_f[1], v[u].y, fired_f[0] * v[u].x)));
                                    g += dpp_move<0xB1>(g);   // quad_perm [1,0,3,2]
                                    g += dpp_move<0x4E>(g);   // quad_perm [2,3,0,1]
                                    g += dpp_move<0x141>(g);  // row_half_mirror: the other quad of these eight lanes
                                    if (lp > 8) g += dpp_move<0x140>(g);  // row_mirror: the other eight of these sixteen
                                    keep = in_row == u ? g : keep;
                                }
                                if (row_fired && in_row < kF && p + in_row < p1) a.d_blk_w[p + in_row] += keep;
                            } else {
#pragma unroll
                                for (int u = 0; u < kF; ++u) {
                                    float g = ((mine & 1u) ? v[u].x : 0.0f) + ((mine & 2u) ? v[u].y : 0.0f) +
                                              ((mine & 4u) ? v[u].z : 0.0f) + ((mine & 8u) ? v[u].w : 0.0f);
                                    for (int off = 1; off < lp; off <<= 1) g += __shfl_xor(g, off, kWave);
                                    if (row_fired && b4 == 0 && p + u < p1) a.d_blk_w[p + u] += g;
                                }
                            }
                        }
                        // a lane whose row segment has ended stays at its end: with p <= p1 at every fetch no lane
                        // reads a record at or beyond p1 + 2*kF, which is what BMTK_BLOCKED_PAD covers, however much
                        // longer the other rows of the visit are
                        p = min(p + kF, p1);
                    };
                    while (true) {
                        work(cur, nxt);
                        if (__ballot(p < p1) == 0ull) break;
                        work(nxt, cur);
                        if (__ballot(p < p1) == 0ull) break;
                    }
                };
                if (kWide) {
                    // a row's first eight lanes fetch one record in eight each (one wavefront instruction for eight
                    // records of every row) and pass them round; eight lanes fetching the same record eight times
                    // over kept the address unit busier than the adjoint rows did
                    struct Shared {
                        uint2 r[kF / 8];
                    };
                    const int c = (lane - grp * lp) & 7, first = grp * lp;
                    visit(
                        [&](int ahead) {
                            Shared f;
#pragma unroll
                            for (int i = 0; i < kF / 8; ++i) f.r[i] = rows[p + ahead + 8 * i + c];
                            return f;
                        },
                        [&](const Shared &have, int u) {
                            return make_uint2((unsigned)__shfl((int)have.r[u / 8].x, first + (u & 7), kWave),
                                              (unsigned)__shfl((int)have.r[u / 8].y, first + (u & 7), kWave));
                        });
                } else {
                    struct Records {
                        uint2 r[kF];
                    };
                    visit(
                        [&](int ahead) {
                            Records f;
#pragma unroll
                            for (int u = 0; u < kF; ++u) f.r[u] = rows[p + ahead + u];
                            return f;
                        },
                        [&](const Records &have, int u) { return have.r[u]; });
                }
                float4 t = acc[k * kWave];
                t.x += s.x;
                t.y += s.y;
                t.z += s.z;
                t.w += s.w;
                acc[k * kWave] = t;
            }
        }
        for (int k = 0; k < gpw; ++k) {
            const int64_t j = row_of(sw, k);
            if (j < row_hi && lane_on) {
                const unsigned act = (unsigned)(masks >> (8 * k)) & 0xFu;
                const float4 t = acc[k * kWave];
                *reinterpret_cast<float4 *>(a.gz + (int64_t)x * ne + j * batch + b4) =
                    make_float4((act & 1u) ? t.x : 0.0f, (act & 2u) ? t.y : 0.0f, (act & 4u) ? t.z : 0.0f,
                                (act & 8u) ? t.w : 0.0f);
            }
        }
    }
    // The input-weight gradient of the same step (it reads the same adjoint slots): a few thousand runs of events,
    // each a chain of dependent reads for one wavefront.  Done here by whichever wavefronts are through with their
    // rows, it disappears in this kernel's tail; beside the state adjoint it lengthened that launch by 20 us.
    if (do_inp) bwd_inp_grad_waves(a, q, (int)blockIdx.x * kBlkWaves + wave, (int)gridDim.x * kBlkWaves);
}

// `x` of lane kU of the lane's own group of kLp (8 or 16) lanes
template <int kLp, int kU>
__device__ __forceinline__ unsigned of_row(unsigned x)
{
    static_assert(kLp == 8 || kLp == 16, "lane groups of half a 32-lane swizzle or less");
    return (unsigned)__builtin_amdgcn_ds_swizzle((int)x, (kU << 5) | (32 - kLp));
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kBlkBurst = 3;         // batches of sixteen records a row that are asked for at once
constexpr int kBlkLengthKeys = 128;  // rows of a sweep are sorted by the length of their segment, up to this

// records `at` and `at + 1` (any `at`: sixteen bytes on a boundary of eight)
__device__ __forceinline__ uint4 pair_at(const uint2 *__restrict__ rows, int at)
{
    struct __attribute__((packed, aligned(8))) Pair {
        unsigned x, y, z, w;
    };
    const Pair r = *reinterpret_cast<const Pair *>(rows + at);
    return make_uint4(r.x, r.y, r.z, r.w);
}

// LDS of bwd_gather_blocked2_kernel behind the partial sums, by rows of a sweep
constexpr size_t blk2_sort_bytes(size_t rows_sweep)
{
    return rows_sweep * (2 * sizeof(unsigned long long) + 2 * sizeof(int2) + 3 * sizeof(uint16_t)) + 2 * kBlkLengthKeys * sizeof(unsigned);
}

// TWO steps, t = q.t and t-1, in one pass over the blocked table (batches above 16: lp >= 8).  gz of step t reads
// the adjoint slots t+1 .. t+L-1, gz of step t-1 the slots t .. t+L-2, and slot t only depends on what the state
// adjoint of step t+1 left behind (it is psc0 times the adjoint of y1 BEFORE step t is undone): both sums can be taken
// before the state adjoint of step t runs.  Per synapse the record, its weight, the trip round the row's lanes, the
// row's bounds and the loop around them are paid once for two steps; the two adjoint rows (same target and
// receptor, neighbouring slots) are fetched side by side.  The weight gradient rides along for both steps with ONE
// read-modify-write per record.  Partial sums: gz[x] for step t, gz[8 + x] for step t-1.  A row's two partial sums take
// 32 bytes of LDS per lane (half as many rows per sweep as in bwd_gather_blocked_kernel).
//
// What bounds it: a compute unit gets its loads back in the order in which it asked for them.  Adjoint rows that the L2 holds
// come at one 128-byte row per 2.3 clocks (33 TB/s over the chip), but every record that has to come from memory holds up
// the rows asked for behind it: 100 M rows beside a 400 MB stream of records take 420 us without the stream, 614 with a
// piece of it fetched now and then, 457 with eight pieces at once, all wavefronts of a workgroup together.  So the records
// (and bounds) of a whole visit are asked for at once, a visit ahead, behind a barrier; the barriers also keep the
// wavefronts within a range, so that its adjoint rows stay in the L2 (misses 46 M -> 12 M lines of 107 M).  And a wavefront's
// eight rows take as long as the longest of them: 30 % of the lanes' work at 42 records a segment, which is why a sweep's rows
// are sorted by the length of their segment before every range (and by whether they fired: the gradient's work).  Rows that fired are not gathered into
// sweeps of their own, as bwd_gather_blocked_kernel gathers them: within a sweep the sort does it, and sweeps of like work are no slower (us per step with a list
// of all rows / without, one row in five fired: 51978 x 32, in-degree 1000: 416 / 413; 100000 x 32, 300: 470 / 455; 30000 x 64, 600: 317 / 310).
// 51978 neurons x 32 trials, in-degree 1000, us per launch: as before 1025, with bursts and barriers 880, rows sorted 787, a visit
// ahead and two records a lane 750; of these 35 are the gradients' read-modify-writes and 50 the input gradients in the tail.
// Tried: records without a place in the caches (nontemporal, 3 % slower), gradients as atomic additions (1 %), their
// old values fetched with the records (spills, 2 %).
template <int kLp, bool kGrad, bool kNe24>
__global__ __launch_bounds__(kBlkThreads) void bwd_gather_blocked2_kernel(bmtk_glif3_bwd a, BwdStep q, int rows_cu, int sweeps,
                                                                          int gpw, int do_inp)
{
    // partial sums [rows of a sweep][2][kLp], the sweep's fired trials, segment bounds, the counters of the sort, places in the
    // order of the visits
    extern __shared__ float4 blk_acc[];
    constexpr int kBurst = kBlkBurst;
    constexpr int per = kWave / kLp;
    const int batch = a.batch;
    const int64_t n = a.n_neurons, ne = n * batch;
    const int L = a.ring_slots;
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int x = blockIdx.x & 7;
    const int P = a.blk_count >> 3;
    const int grp = lane / kLp, in_row = lane & (kLp - 1), b4 = in_row * 4, c8 = in_row & 7;
    const bool lane_on = b4 < batch;
    const unsigned long long grp_lanes = ((1ull << kLp) - 1ull) << (grp * kLp);
    const int64_t row_lo = (int64_t)(blockIdx.x >> 3) * rows_cu;
    const int64_t row_hi = row_lo + rows_cu < n ? row_lo + rows_cu : n;
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(a.blk_packed);
    const char *__restrict__ ring = reinterpret_cast<const char *>(a.lam_ring);
    const unsigned lane_off = (unsigned)(lane_on ? b4 : 0) * 4u;  // (lanes without a trial read what the row's first lane reads)
    const unsigned q_lo = (unsigned)q.slot * 4u, q_wrap = q_lo - 4u * (unsigned)L;
    const unsigned ne32 = (unsigned)ne, batch32 = (unsigned)batch;
    // from a synapse's cell for step t to its cell for step t-1: one slot down, or L-1 slots up from slot 0 (bytes)
    const unsigned slot_down = 0u - 16u * ne32, slot_up = 16u * ne32 * (unsigned)(L - 1);
    auto cell_offs = [&](unsigned tdr, unsigned &off_t, unsigned &off_p) {
        const unsigned dq = tdr >> 24;
        const unsigned plane = min(dq + q_lo, dq + q_wrap);  // (slot of step t + delay) * 4 + receptor
        const unsigned elem = mad_u24(tdr, batch32, kNe24 ? mul_u24(plane, ne32) : plane * ne32);
        off_t = elem << 2;
        off_p = off_t + (plane < 4u ? slot_up : slot_down);
    };
    const int rows_sweep = kBlkWaves * gpw * per;
    unsigned long long *fired_l = reinterpret_cast<unsigned long long *>(blk_acc + (size_t)rows_sweep * 2 * kLp);  // [2][rows_sweep]
    int2 *bounds_l = reinterpret_cast<int2 *>(fired_l + 2 * rows_sweep);             // [2][rows_sweep], by visit of even and odd ranges
    unsigned *count_l = reinterpret_cast<unsigned *>(bounds_l + 2 * rows_sweep);     // [2 * kBlkLengthKeys]
    uint16_t *visit_l = reinterpret_cast<uint16_t *>(count_l + 2 * kBlkLengthKeys);  // [2][rows_sweep]: place of a visit's row
    uint16_t *wanted_l = visit_l + 2 * rows_sweep;                                   // by place: whether its row has visits
    const uint64_t *__restrict__ bits_t = a.spike_bits + q.row * a.spike_bits_stride;
    const uint64_t *__restrict__ bits_p = a.spike_bits + (q.row - 1) * a.spike_bits_stride;
    // the row at a place of sweep sw, counted from the workgroup's first (0xFFFFFFFF: none)
    auto row_at = [&](int sw, int place) -> unsigned {
        place += sw * rows_sweep;
        return place < rows_cu && row_lo + place < row_hi ? (unsigned)place : ~0u;
    };
    for (int i = threadIdx.x; i < 2 * kBlkLengthKeys; i += kBlkThreads) count_l[i] = 0u;
    for (int sw = 0; sw < sweeps; ++sw) {
        // The places of a lane group, k = 0 .. gpw-1: what belongs to their rows for the whole sweep.
        // active: four bits a place, the lane's trials with a non-zero surrogate derivative; of step t, and 16 up of step t-1
        unsigned active = 0u;
        {
            constexpr int kPlaces = kBlkMaxGroups / 2;
            // (no branches around the loads: those of all places travel together, where there is no row the last one's)
            uint32_t f4[kPlaces][2];
            float4 v4[kPlaces][2];
            float th[kPlaces];
            unsigned long long fired[kPlaces][2];
            bool have[kPlaces];
#pragma unroll
            for (int k = 0; k < kPlaces; ++k) {
                const unsigned local = k < gpw ? row_at(sw, (k * kBlkWaves + wave) * per + grp) : ~0u;
                have[k] = local != ~0u && row_lo + local < row_hi;
                const int64_t j = have[k] ? row_lo + local : n - 1, e = j * batch + (lane_on ? b4 : 0);
                th[k] = a.prop[GLIF3_TH * a.prop_stride + (a.class_id ? (int64_t)a.class_id[j] : j)];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    f4[k][s] = *reinterpret_cast<const uint32_t *>(a.save_flags + (q.row - s) * ne + e);
                    v4[k][s] = *reinterpret_cast<const float4 *>(a.save_v + (q.row - s) * ne + e);
                    if (kGrad) {
                        const uint64_t *bits = s == 0 ? bits_t : bits_p;
                        const int64_t bit = j * batch;
                        const int sh = (int)(bit & 63);
                        const bool two = sh + batch > 64;
                        const unsigned long long lo = bits[bit >> 6], hi = bits[(bit >> 6) + (two ? 1 : 0)];
                        fired[k][s] = lo >> sh | (two ? hi << (64 - sh) : 0ull);
                        if (batch < 64) fired[k][s] &= (1ull << batch) - 1ull;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < kPlaces; ++k) {
                if (k >= gpw) break;
                const int place = (k * kBlkWaves + wave) * per + grp;
                unsigned act = 0u;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const float v[4] = {v4[k][s].x, v4[k][s].y, v4[k][s].z, v4[k][s].w};
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (((f4[k][s] >> (8 * c)) & BMTK_F_INTEGRATING) && fabsf((v[c] - th[k]) / th[k]) < 1.0f) act |= 1u << (16 * s + c);
                }
                if (!have[k] || !lane_on) act = 0u;
                active |= act << (4 * k);
                const bool spiked = kGrad && have[k] && (fired[k][0] | fired[k][1]) != 0ull;
                // (rows none of whose trials needs a sum, and whose source did not fire, have no visits)
                const bool wanted = (__ballot(act != 0u) & grp_lanes) != 0ull || spiked;
                if (in_row == 0) {
                    wanted_l[place] = wanted ? 1u : 0u;
                    if (kGrad) {
                        fired_l[place] = spiked ? fired[k][0] : 0ull;
                        fired_l[rows_sweep + place] = spiked ? fired[k][1] : 0ull;
                    }
                }
                blk_acc[(size_t)place * 2 * kLp + in_row] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                blk_acc[(size_t)place * 2 * kLp + kLp + in_row] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
        __syncthreads();
        // thread i keeps the segment bounds of the row at place i for the range ahead
        const bool sorts = (int)threadIdx.x < rows_sweep;
        const unsigned my_row = sorts && wanted_l[threadIdx.x] ? row_at(sw, (int)threadIdx.x) : ~0u;
        const bool my_fired = kGrad && sorts && (fired_l[threadIdx.x] | fired_l[rows_sweep + threadIdx.x]) != 0ull;
        int2 ahead = make_int2(0, 0);
        auto ask_bounds = [&](int ph) {
            ahead = make_int2(0, 0);
            if (ph < P && my_row != ~0u) {
                const int32_t *__restrict__ ip = a.blk_indptr + (int64_t)(x * P + ph) * n + row_lo + my_row;
                ahead = make_int2(ip[0], ip[1]);
            }
        };
        // The rows in the order of their visits to a range: those whose source fired first, the longer segments before the
        // shorter (a wavefront takes as long as the longest of its eight rows), by counting.  Which of two equal ones
        // comes first does not matter: a row's sum is its own.
        auto sort_visits = [&](int ph) {
            int key = 0;
            unsigned rank = 0u;
            if (sorts) {
                key = kBlkLengthKeys - 1 - min(ahead.y - ahead.x, kBlkLengthKeys - 1) + (my_fired ? 0 : kBlkLengthKeys);
                rank = atomicAdd(count_l + key, 1u);
            }
            __syncthreads();
            if (wave == 0) {
                unsigned c[2 * kBlkLengthKeys / kWave], sum = 0u;
#pragma unroll
                for (int i = 0; i < 2 * kBlkLengthKeys / kWave; ++i) {
                    c[i] = count_l[lane * (2 * kBlkLengthKeys / kWave) + i];
                    sum += c[i];
                }
                unsigned at = wave_inclusive_scan(sum) - sum;
#pragma unroll
                for (int i = 0; i < 2 * kBlkLengthKeys / kWave; ++i) {
                    count_l[lane * (2 * kBlkLengthKeys / kWave) + i] = at;
                    at += c[i];
                }
            }
            __syncthreads();
            if (sorts) {
                const unsigned at = (ph & 1) * rows_sweep + count_l[key] + rank;
                visit_l[at] = (uint16_t)threadIdx.x;
                bounds_l[at] = ahead;
            }
            ask_bounds(ph + 1);
            __syncthreads();
            if (threadIdx.x < 2 * kBlkLengthKeys) count_l[threadIdx.x] = 0u;  // (there is a barrier before the next count)
        };
        ask_bounds(0);
        sort_visits(0);
        // A visit's records, kBurst batches of sixteen a row (lane c8 of a row takes records 2 c8 and 2 c8 + 1 of each), are
        // asked for a visit ahead and by all wavefronts together.
        uint4 rec[kBurst];
        int p = 0, p1 = 0, place = 0;
        auto burst = [&](uint4 (&r)[kBurst], int from, int end) {
            const int last = max(end, 2) - 2;  // (a pair past the row's end is the last two records before it)
#pragma unroll
            for (int m = 0; m < kBurst; ++m) r[m] = pair_at(rows, min(from + 16 * m + 2 * c8, last));
        };
        auto visit_at = [&](int ph, int k, int &from, int &end, int &of) {
            const int at = (ph & 1) * rows_sweep + (k * kBlkWaves + wave) * per + grp;
            from = bounds_l[at].x;
            end = bounds_l[at].y;
            of = visit_l[at];
        };
        visit_at(0, 0, p, p1, place);
        burst(rec, p, p1);
        for (int ph = 0; ph < P; ++ph) {
            for (int k = 0; k < gpw; ++k) {
                const bool more = k + 1 < gpw || ph + 1 < P;
                int p_next = 0, p1_next = 0, place_next = place;
                uint4 rec_next[kBurst];
                __syncthreads();
                if (k + 1 == gpw && ph + 1 < P) sort_visits(ph + 1);
                if (more) visit_at(k + 1 < gpw ? ph : ph + 1, k + 1 < gpw ? k + 1 : 0, p_next, p1_next, place_next);
                burst(rec_next, p_next, p1_next);
                auto on = [&]() {
                    p = p_next;
                    p1 = p1_next;
                    place = place_next;
#pragma unroll
                    for (int m = 0; m < kBurst; ++m) rec[m] = rec_next[m];
                };
                if (__ballot(p < p1) == 0ull) {
                    on();
                    continue;
                }
                const unsigned mine_t = kGrad ? (unsigned)(fired_l[place] >> b4) & 0xFu : 0u;
                const unsigned mine_p = kGrad ? (unsigned)(fired_l[rows_sweep + place] >> b4) & 0xFu : 0u;
                const unsigned long long fired_lanes = kGrad ? __ballot((mine_t | mine_p) != 0u) : 0ull;
                const bool row_fired = (fired_lanes & grp_lanes) != 0ull;
                float4 s_t = make_float4(0.0f, 0.0f, 0.0f, 0.0f), s_p = s_t;
                auto sixteen = [&](uint4 own) {
                    // the lane's own two records first: past the row's end they are record 0 with weight 0 (the same arithmetic and
                    // the same loads for every lane); their cells are worked out once and passed round with the weights.
                    // (A pair that begins with the row's last record was fetched one record early.)
                    const int left = p1 - p - 2 * c8;
                    const bool some = left > 0, both = left > 1, shifted = left == 1 && p1 > 1;
                    unsigned own_t[2], own_p[2];
                    cell_offs(shifted ? own.z : some ? own.x : 0u, own_t[0], own_p[0]);
                    cell_offs(both ? own.z : 0u, own_t[1], own_p[1]);
                    const unsigned own_w[2] = {shifted ? own.w : some ? own.y : 0u, both ? own.w : 0u};
                    auto eight = [&](auto second) {
                        constexpr int kSecond = decltype(second)::value;
                        const bool grad_now = kGrad && (fired_lanes & __ballot(p < p1)) != 0ull;
                        float keep = 0.0f;
                        auto four = [&](auto which) {
                            constexpr int h = 4 * decltype(which)::value, l = 4 * kSecond + h / 2;  // (two records a lane)
                            const unsigned off_t[4] = {of_row<kLp, l>(own_t[0]), of_row<kLp, l>(own_t[1]), of_row<kLp, l + 1>(own_t[0]), of_row<kLp, l + 1>(own_t[1])};
                            const unsigned off_p[4] = {of_row<kLp, l>(own_p[0]), of_row<kLp, l>(own_p[1]), of_row<kLp, l + 1>(own_p[0]), of_row<kLp, l + 1>(own_p[1])};
                            float4 vt[4], vp[4];
#pragma unroll
                            for (int u = 0; u < 4; ++u) {
                                vt[u] = *reinterpret_cast<const float4 *>(ring + (off_t[u] + lane_off));
                                vp[u] = *reinterpret_cast<const float4 *>(ring + (off_p[u] + lane_off));
                            }
                            const unsigned w[4] = {of_row<kLp, l>(own_w[0]), of_row<kLp, l>(own_w[1]), of_row<kLp, l + 1>(own_w[0]), of_row<kLp, l + 1>(own_w[1])};
#pragma unroll
                            for (int u = 0; u < 4; ++u) {
                                const float wu = __uint_as_float(w[u]);
                                s_t.x = fmaf(wu, vt[u].x, s_t.x);
                                s_t.y = fmaf(wu, vt[u].y, s_t.y);
                                s_t.z = fmaf(wu, vt[u].z, s_t.z);
                                s_t.w = fmaf(wu, vt[u].w, s_t.w);
                                s_p.x = fmaf(wu, vp[u].x, s_p.x);
                                s_p.y = fmaf(wu, vp[u].y, s_p.y);
                                s_p.z = fmaf(wu, vp[u].z, s_p.z);
                                s_p.w = fmaf(wu, vp[u].w, s_p.w);
                            }
                            if (grad_now) {
                                // gradient of a record: over the row's lanes, the adjoint entries of the trials in which the
                                // source fired, of step t and of step t-1 (see bwd_gather_blocked_kernel)
#pragma unroll
                                for (int u = 0; u < 4; ++u) {
                                    float g = ((mine_t & 1u) ? vt[u].x : 0.0f) + ((mine_t & 2u) ? vt[u].y : 0.0f) +
                                              ((mine_t & 4u) ? vt[u].z : 0.0f) + ((mine_t & 8u) ? vt[u].w : 0.0f);
                                    g += ((mine_p & 1u) ? vp[u].x : 0.0f) + ((mine_p & 2u) ? vp[u].y : 0.0f) +
                                         ((mine_p & 4u) ? vp[u].z : 0.0f) + ((mine_p & 8u) ? vp[u].w : 0.0f);
                                    g += dpp_move<0xB1>(g);
                                    g += dpp_move<0x4E>(g);
                                    g += dpp_move<0x141>(g);
                                    if (kLp > 8) g += dpp_move<0x140>(g);
                                    keep = in_row == h + u ? g : keep;
                                }
                            }
                        };
                        four(std::integral_constant<int, 0>{});
                        if (__ballot(p + 4 < p1) != 0ull) four(std::integral_constant<int, 1>{});
                        if (grad_now && row_fired && in_row < 8 && p + in_row < p1) a.d_blk_w[p + in_row] += keep;
                        p = min(p + 8, p1);
                    };
                    eight(std::integral_constant<int, 0>{});
                    if (__ballot(p < p1) != 0ull) eight(std::integral_constant<int, 1>{});
                };
                while (true) {
#pragma unroll
                    for (int m = 0; m < kBurst; ++m) {
                        if (__ballot(p < p1) == 0ull) break;
                        sixteen(rec[m]);
                    }
                    if (__ballot(p < p1) == 0ull) break;
                    burst(rec, p, p1);  // (segments longer than a burst)
                }
                float4 *acc = blk_acc + (size_t)place * 2 * kLp + in_row;
                float4 t = acc[0];
                t.x += s_t.x;
                t.y += s_t.y;
                t.z += s_t.z;
                t.w += s_t.w;
                acc[0] = t;
                t = acc[kLp];
                t.x += s_p.x;
                t.y += s_p.y;
                t.z += s_p.z;
                t.w += s_p.w;
                acc[kLp] = t;
                on();
            }
        }
        __syncthreads();  // (a row's sums were last added to by whichever wavefront its last visit fell to)
        for (int k = 0; k < gpw; ++k) {
            const int place = (k * kBlkWaves + wave) * per + grp;
            const unsigned local = row_at(sw, place);
            if (local == ~0u || row_lo + local >= row_hi || !lane_on) continue;
            const int64_t j = row_lo + local;
            const unsigned at = active >> (4 * k), ap = active >> (16 + 4 * k);
            // (written once, read by the next launch: not kept in the L2 that the adjoint rows are to stay in)
            const f32x4 *sums = reinterpret_cast<const f32x4 *>(blk_acc) + (size_t)place * 2 * kLp + in_row;
            const f32x4 st = sums[0], sp = sums[kLp];
            __builtin_nontemporal_store(f32x4{(at & 1u) ? st.x : 0.0f, (at & 2u) ? st.y : 0.0f, (at & 4u) ? st.z : 0.0f, (at & 8u) ? st.w : 0.0f},
                                        reinterpret_cast<f32x4 *>(a.gz + (int64_t)x * ne + j * batch + b4));
            __builtin_nontemporal_store(f32x4{(ap & 1u) ? sp.x : 0.0f, (ap & 2u) ? sp.y : 0.0f, (ap & 4u) ? sp.z : 0.0f, (ap & 8u) ? sp.w : 0.0f},
                                        reinterpret_cast<f32x4 *>(a.gz + (int64_t)(8 + x) * ne + j * batch + b4));
        }
    }
    // the input-weight gradients of both steps, in the kernel's tail
    if (do_inp) bwd_inp_grad2_waves(a, q, (int)blockIdx.x * kBlkWaves + wave, (int)gridDim.x * kBlkWaves);
}

// One step of the state adjoint on registers: the adjoint of the state after the step comes in, that of the state
// before it goes out.  sg = surrogate derivative times the adjoint of the step's spike (only read where the
// element was integrating).
__device__ __forceinline__ void state_adjoint_step(float &lV, float (&lA)[GLIF3_NASC], float (&l1)[GLIF3_NREC],
                                                   float (&l2)[GLIF3_NREC], const Glif3Prop &p, float h, uint8_t f, float sg)
{
    // y1' = P11*y1 + psc0*s ; y2' = P21*y1 + P11*y2
    float n1[GLIF3_NREC], n2[GLIF3_NREC];
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) {
        n1[k] = p.P11[k] * l1[k] + (h * p.P11[k]) * l2[k];
        n2[k] = p.P11[k] * l2[k];
    }
    float nV, nA[GLIF3_NASC];
    if (f & BMTK_F_INTEGRATING) {
        const float lU = lV + sg;
        nV = p.P33 * lU;
        const float lS = p.P30 * lU;
#pragma unroll
        for (int k = 0; k < GLIF3_NASC; ++k) nA[k] = p.c[k] * lS + p.d[k] * lA[k];
#pragma unroll
        for (int k = 0; k < GLIF3_NREC; ++k) {
            n1[k] += p.P31[k] * lU;
            n2[k] += p.P32[k] * lU;
        }
    } else if (f & BMTK_F_RESET) {
        nV = 0.0f;
#pragma unroll
        for (int k = 0; k < GLIF3_NASC; ++k) nA[k] = p.r[k] * lA[k];
    } else {
        nV = lV;
#pragma unroll
        for (int k = 0; k < GLIF3_NASC; ++k) nA[k] = lA[k];
    }
    lV = nV;
#pragma unroll
    for (int k = 0; k < GLIF3_NASC; ++k) lA[k] = nA[k];
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) {
        l1[k] = n1[k];
        l2[k] = n2[k];
    }
}

// surrogate derivative times the adjoint of the spike of element e in the step of record row `row`: what comes back
// through the synapses (`parts` partial sums from plane `first` of gz on) plus the loss derivative
__device__ __forceinline__ float spike_adjoint(const bmtk_glif3_bwd &a, const Glif3Prop &p, int64_t row, int64_t e, int64_t ne,
                                               int first, int parts)
{
    float g = a.gz[(int64_t)first * ne + e];
    for (int x = 1; x < parts; ++x) g += a.gz[(int64_t)(first + x) * ne + e];
    if (a.dl_dz) g += a.dl_dz[row * ne + e];
    if (a.dl_dz_const) g += a.dl_dz_const[e];
    return surrogate(a.save_v[row * ne + e], p.th, a.dampening) * g;
}

// state adjoint of one step, one thread per element; writes the adjoint of
// this step's arrivals into ring slot t
__device__ __forceinline__ void bwd_state_block(const bmtk_glif3_bwd &a, const BwdStep &q, int64_t block)
{
    const int64_t ne = a.n_neurons * (int64_t)a.batch;
    const int64_t e = block * kBlock + threadIdx.x;
    if (e >= ne) return;
    const int64_t n = a.batch == 1 ? e : (int64_t)((uint32_t)e / (uint32_t)a.batch);
    const int64_t col = a.class_id ? (int64_t)a.class_id[n] : n;
    Glif3Prop p;
    p.load(a.prop, a.prop_stride, col);
    const uint8_t f = a.save_flags[q.row * ne + e];
    float lV = a.lam_V[e];
    float lA[GLIF3_NASC], l1[GLIF3_NREC], l2[GLIF3_NREC];
#pragma unroll
    for (int k = 0; k < GLIF3_NASC; ++k) lA[k] = a.lam_asc[k * ne + e];
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) {
        l1[k] = a.lam_y1[k * ne + e];
        l2[k] = a.lam_y2[k * ne + e];
    }
    float *slot = a.lam_ring + (int64_t)q.slot * GLIF3_NREC * ne + e;
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) slot[k * ne] = p.psc0[k] * l1[k];
    const float sg = (f & BMTK_F_INTEGRATING) ? spike_adjoint(a, p, q.row, e, ne, 0, q.parts) : 0.0f;
    state_adjoint_step(lV, lA, l1, l2, p, a.h, f, sg);
    a.lam_V[e] = lV;
#pragma unroll
    for (int k = 0; k < GLIF3_NASC; ++k) a.lam_asc[k * ne + e] = lA[k];
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) {
        a.lam_y1[k * ne + e] = l1[k];
        a.lam_y2[k * ne + e] = l2[k];
    }
}

// The state adjoints of steps t = q.t and t-1 in one launch, the adjoint state in registers in between: the partial
// sums of step t are planes 0-7 of gz, those of step t-1 planes 8-15 (bwd_gather_blocked2_kernel).  Ring slots
// follow the rule of that kernel: slot s holds psc0 times the adjoint of y1 before step s is undone, so this launch
// writes slot t-1 between its two steps and, with write_after, slot t-2 from what it leaves (for the pair of steps
// that follows); slot t was written by the launch before, or by bwd_seed_slot_kernel at the start of a call.
__global__ __launch_bounds__(kBlock) void bwd_state2_kernel(bmtk_glif3_bwd a, BwdStep q, int write_after)
{
    const int64_t ne = a.n_neurons * (int64_t)a.batch;
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= ne) return;
    const int64_t n = a.batch == 1 ? e : (int64_t)((uint32_t)e / (uint32_t)a.batch);
    const int64_t col = a.class_id ? (int64_t)a.class_id[n] : n;
    Glif3Prop p;
    p.load(a.prop, a.prop_stride, col);
    const int L = a.ring_slots;
    float lV = a.lam_V[e];
    float lA[GLIF3_NASC], l1[GLIF3_NREC], l2[GLIF3_NREC];
#pragma unroll
    for (int k = 0; k < GLIF3_NASC; ++k) lA[k] = a.lam_asc[k * ne + e];
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) {
        l1[k] = a.lam_y1[k * ne + e];
        l2[k] = a.lam_y2[k * ne + e];
    }
    const uint8_t f_t = a.save_flags[q.row * ne + e], f_p = a.save_flags[(q.row - 1) * ne + e];
    const float sg_t = (f_t & BMTK_F_INTEGRATING) ? spike_adjoint(a, p, q.row, e, ne, 0, 8) : 0.0f;
    const float sg_p = (f_p & BMTK_F_INTEGRATING) ? spike_adjoint(a, p, q.row - 1, e, ne, 8, 8) : 0.0f;
    state_adjoint_step(lV, lA, l1, l2, p, a.h, f_t, sg_t);
    const int before = q.slot == 0 ? L - 1 : q.slot - 1;
    float *slot = a.lam_ring + (int64_t)before * GLIF3_NREC * ne + e;
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) slot[k * ne] = p.psc0[k] * l1[k];
    state_adjoint_step(lV, lA, l1, l2, p, a.h, f_p, sg_p);
    if (write_after) {
        slot = a.lam_ring + (int64_t)(before == 0 ? L - 1 : before - 1) * GLIF3_NREC * ne + e;
#pragma unroll
        for (int k = 0; k < GLIF3_NREC; ++k) slot[k * ne] = p.psc0[k] * l1[k];
    }
    a.lam_V[e] = lV;
#pragma unroll
    for (int k = 0; k < GLIF3_NASC; ++k) a.lam_asc[k * ne + e] = lA[k];
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k) {
        a.lam_y1[k * ne + e] = l1[k];
        a.lam_y2[k * ne + e] = l2[k];
    }
}

// The adjoint state of one element, its loss derivative and what of the forward record the swept form needs of it.
template <bool kTwo>
struct SweepElem {
    float lV, lA[GLIF3_NASC], l1[GLIF3_NREC], l2[GLIF3_NREC], dl[kTwo ? 2 : 1], dl_const;

    __device__ __forceinline__ void load(const bmtk_glif3_bwd &a, const BwdStep &q, int64_t e, int64_t ne)
    {
        lV = a.lam_V[e];
#pragma unroll
        for (int k = 0; k < GLIF3_NASC; ++k) lA[k] = a.lam_asc[k * ne + e];
#pragma unroll
        for (int k = 0; k < GLIF3_NREC; ++k) {
            l1[k] = a.lam_y1[k * ne + e];
            l2[k] = a.lam_y2[k * ne + e];
        }
        dl_const = a.dl_dz_const ? a.dl_dz_const[e] : 0.0f;
#pragma unroll
        for (int s = 0; s < (kTwo ? 2 : 1); ++s) dl[s] = a.dl_dz ? a.dl_dz[(q.row - s) * ne + e] : 0.0f;
    }
    // steps t and (kTwo) t-1 undone: g[s] = what comes back through the synapses, v[s], f[s] = potential and flags
    __device__ __forceinline__ void undo(const bmtk_glif3_bwd &a, const BwdStep &q, const Glif3Prop &p, int64_t e, int64_t ne,
                                         const float (&g)[2], const float (&v)[2], const unsigned (&f)[2])
    {
        const int L = a.ring_slots;
        int slot = q.slot;
#pragma unroll
        for (int s = 0; s < (kTwo ? 2 : 1); ++s) {
            float gs = g[s];
            if (a.dl_dz) gs += dl[s];
            if (a.dl_dz_const) gs += dl_const;
            const float sg = (f[s] & BMTK_F_INTEGRATING) ? surrogate(v[s], p.th, a.dampening) * gs : 0.0f;
            state_adjoint_step(lV, lA, l1, l2, p, a.h, (uint8_t)f[s], sg);
            // slot t-1 (t-2): what the launches ahead read of the step before
            slot = slot == 0 ? L - 1 : slot - 1;
            float *cells = a.lam_ring + (int64_t)slot * GLIF3_NREC * ne + e;
#pragma unroll
            for (int k = 0; k < GLIF3_NREC; ++k) cells[k * ne] = p.psc0[k] * l1[k];
        }
        a.lam_V[e] = lV;
#pragma unroll
        for (int k = 0; k < GLIF3_NASC; ++k) a.lam_asc[k * ne + e] = lA[k];
#pragma unroll
        for (int k = 0; k < GLIF3_NREC; ++k) {
            a.lam_y1[k * ne + e] = l1[k];
            a.lam_y2[k * ne + e] = l2[k];
        }
    }
};

// The swept form of a backward step, for networks whose adjoint ring the L2s hold (batches that are a multiple of 4 up to
// 64): transposed propagation, weight gradients and state adjoint of step t -- with kTwo of steps t and t-1 -- in ONE
// launch through the plain source-major table.  At these sizes a step's launches are short chains of dependent loads,
// not traffic: what counts is how many launches a step takes and how long the chain in each is.
//
// A row's synapses are shared by `splits` neighbouring lane groups of LP lanes (four trials each), as many as the chip
// has room for (3001 rows x batch 12: 33 / 19 / 12 / 10 us per step with 1 / 2 / 4 / 16 groups a row; 14461 rows: 32 / 32 / 42
// / 55); they take the row's batches of kF synapses in turn and fold their sums at the end.  A row's sum is then
// complete in one wavefront and the state adjoint of its elements follows in the same launch.  For that the adjoint
// ring has two slots more than the table's delays need (ring_slots >= largest delay + 3): while some wavefronts still
// read the slots t .. t+L-1, others write slots t-1 and t-2.  Slot s holds psc0 times the adjoint of y1 before step s is
// undone; slot t was written by the launch before (bwd_seed_slot_kernel at the start of a call).
//
// No array of the kernel is indexed at run time: a choice of one of four trials' values by the lane's place made the sums and potentials an array
// in scratch memory, whose stores waited for the loads (and the records asked for before them) ahead of the first turn.  us per two
// steps, with scratch / without: 3001 x 12, in-degree 200: 19.6 / 16.2 (15.2 since the host divides by the ring's length); 3001 x 32, 100: 25.1 / 18.0; 20000 x 16, 150: 114.5 / 92.6; 12000 x 32, 120: 85.3 / 66.7;
// 12000 x 12, 400: 92.5 / 89.0; 14000 x 16, 200: 71.3 / 71.7.  Tried: eight synapses in flight for rows of a wavefront's own (1800 x 32, 600: 29.8 -> 26.5, but
// 3001 x 4, 200: 12.5 -> 15.2, spilled registers), two turns in flight (spilled registers: 17 to 18.5 against 16.2).
//
// Per step, gather and state adjoint as launches of their own against this form: 3001 neurons x batch 12, in-degree 200:
// 21.8 -> 10.2 us; 6920 x 16, in-degree 525: 56 -> 33; 30000 x 16, in-degree 300: 194 -> 124.  What bounds it: at the smallest sizes the chain
// row bounds -> records -> adjoint rows -> state (a launch starts with cold L2s, 1 to 2.5 us a link), above some 5,000 rows
// the rate at which the L2s hand out adjoint rows (2.6e11 lines of 64 bytes per second).  Rings that the L2s do not
// hold make it pay fabric latency per row, and the blocked table wins (51978 x 32, in-degree 1000: 546 against 740 us).
struct SweepLaunch {
    int splits;      // lane groups that share a row, a power of two
    int n_row_wg;    // workgroups that hold rows; the ones behind them take the input-weight gradients
    int n_sets;      // sets of rows (what a wavefront holds at a time)
    int do_grad;
};
constexpr int kSweepThreads = 256;
constexpr int kSweepWaves = kSweepThreads / kWave;
constexpr int kSweepPerCu = 3;  // workgroups a compute unit holds: 168 vector registers per lane

// kOne: a wavefront holds one row.  What belongs to the row is then the same in all lanes (scalar loads, which leave the
// vector memory path to the adjoint rows), a lane has at most one element of it to undo, and its state is asked for before
// the sums are taken.
template <int LP, bool kOne, bool kTwo>
__global__ __launch_bounds__(kSweepThreads, kSweepPerCu) void bwd_sweep_kernel(bmtk_glif3_bwd a, BwdStep q, SweepLaunch sw)
{
    constexpr int kF = kOne ? 4 : 8;                         // synapses of a row in flight per lane group
    constexpr int kRecs = kF / LP > 1 ? kF / LP : 1;         // records a lane fetches of them
    constexpr int kPer = kWave / LP;
    constexpr int kSteps = kTwo ? 2 : 1;
    const int batch = a.batch;
    const int64_t n = a.n_neurons, ne = n * batch;
    const int L = a.ring_slots;
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    if ((int)blockIdx.x >= sw.n_row_wg) {
        const int w = ((int)blockIdx.x - sw.n_row_wg) * kSweepWaves + wave, nw = ((int)gridDim.x - sw.n_row_wg) * kSweepWaves;
        if (kTwo)
            bwd_inp_grad2_waves(a, q, w, nw);
        else
            bwd_inp_grad_waves(a, q, w, nw);
        return;
    }
    const int grp = lane / LP, in_row = lane & (LP - 1), b4 = in_row * 4;
    const int S = kOne ? kPer : sw.splits, part = grp & (S - 1);
    const int rows_set = kPer / S;
    const bool lane_on = b4 < batch;
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(a.rec_packed);
    const char *__restrict__ ring = reinterpret_cast<const char *>(a.lam_ring);
    const unsigned lane_off = (unsigned)(lane_on ? b4 : 0) * 4u;
    const unsigned q_lo = (unsigned)q.slot * 4u, q_wrap = q_lo - 4u * (unsigned)L;
    const unsigned ne32 = (unsigned)ne, batch32 = (unsigned)batch;
    // from a synapse's cell for step t to its cell for step t-1: one slot down, or L-1 slots up from slot 0 (bytes)
    const unsigned slot_down = 0u - 16u * ne32, slot_up = 16u * ne32 * (unsigned)(L - 1);
    const unsigned long long grp_lanes = (LP == kWave ? ~0ull : ((1ull << LP) - 1ull)) << (grp * LP);

    for (int set = (int)blockIdx.x * kSweepWaves + wave; set < sw.n_sets; set += sw.n_row_wg * kSweepWaves) {
        const int64_t row_set = kOne ? (int64_t)set : (int64_t)set * rows_set + grp / S;
        const bool have = row_set < n;
        const int64_t row = have ? row_set : n - 1;  // (lanes past the last row load what the last one loads)
        int p = a.rec_indptr[row];
        const int p1 = have ? a.rec_indptr[row + 1] : p;
        const int64_t col = a.class_id ? (int64_t)a.class_id[row] : row;
        const int64_t e4 = row * batch + (lane_on ? b4 : 0);
        p = min(p + part * kF, p1);
        // records p .. p+kF-1 of the row, one (kRecs) per lane; places past the row's end repeat its last record
        uint2 rec[kRecs];
        const int last = max(p1, 1) - 1;
        auto fetch = [&](int from) {
#pragma unroll
            for (int i = 0; i < kRecs; ++i) rec[i] = rows[min(from + i * LP + in_row, last)];
        };
        bool busy = __ballot(p < p1) != 0ull;
        if (busy) fetch(p);
        float4 v4[kSteps];
        uint32_t f4[kSteps];
        unsigned fire = 0u;  // bits 0-3: the lane's trials in which the source fired in step t, 4-7: in step t-1
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            f4[s] = *reinterpret_cast<const uint32_t *>(a.save_flags + (q.row - s) * ne + e4);
            v4[s] = *reinterpret_cast<const float4 *>(a.save_v + (q.row - s) * ne + e4);
            if (sw.do_grad && have && lane_on)
                fire |= ((unsigned)(trial_mask(a.spike_bits + (q.row - s) * a.spike_bits_stride, row, batch, 0, batch) >> b4) & 0xFu) << (4 * s);
        }
        Glif3Prop pr;
        SweepElem<kTwo> el;
        if (kOne) {
            pr.load(a.prop, a.prop_stride, col);
            if (kPer >= 4) el.load(a, q, e4 + (part & 3), ne);
        }
        const bool grad = sw.do_grad && __ballot(fire != 0u) != 0ull;
        const bool row_fired = (__ballot(fire != 0u) & grp_lanes) != 0ull;
        if (!kOne) {
            // a row none of whose trials has a surrogate derivative, and whose source did not fire, needs no sum
            const float th = a.prop[GLIF3_TH * a.prop_stride + col];
            bool want = fire != 0u;
#pragma unroll
            for (int s = 0; s < kSteps; ++s)
                want = want || ((f4[s] & (BMTK_F_INTEGRATING << 0)) && fabsf((v4[s].x - th) / th) < 1.0f) ||
                       ((f4[s] & (BMTK_F_INTEGRATING << 8)) && fabsf((v4[s].y - th) / th) < 1.0f) ||
                       ((f4[s] & (BMTK_F_INTEGRATING << 16)) && fabsf((v4[s].z - th) / th) < 1.0f) ||
                       ((f4[s] & (BMTK_F_INTEGRATING << 24)) && fabsf((v4[s].w - th) / th) < 1.0f);
            if ((__ballot(want && lane_on) & grp_lanes) == 0ull) p = p1;
            busy = __ballot(p < p1) != 0ull;
        }
        float4 sum[kSteps];
#pragma unroll
        for (int s = 0; s < kSteps; ++s) sum[s] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        // record u of the batch, from the lane that fetched it
        auto record = [&](int u) {
            const uint2 r = rec[kRecs > 1 ? u / LP : 0];
            if (LP == 1) return r;
            const int src = (lane & ~(LP - 1)) + (u & (LP - 1));
            return make_uint2((unsigned)__shfl((int)r.x, src, kWave), (unsigned)__shfl((int)r.y, src, kWave));
        };
        auto turn = [&](auto with_grad) {
            constexpr bool kG = decltype(with_grad)::value;
            float4 x[kSteps][kF];
            float w[kF];
#pragma unroll
            for (int u = 0; u < kF; ++u) {
                const uint2 sy = record(u);
                const unsigned dq = sy.x >> 24;
                const unsigned plane = min(dq + q_lo, dq + q_wrap);  // (slot of step t + delay) * 4 + receptor
                const unsigned off_t = (mad_u24(sy.x, batch32, mul_u24(plane, ne32)) << 2) + lane_off;
                w[u] = p + u < p1 ? __uint_as_float(sy.y) : 0.0f;  // (past the row's end: its last record with weight 0)
                x[0][u] = *reinterpret_cast<const float4 *>(ring + off_t);
                if (kTwo) x[kSteps - 1][u] = *reinterpret_cast<const float4 *>(ring + (off_t + (plane < 4u ? slot_up : slot_down)));
            }
            float old[kRecs];
            if (kG) {
#pragma unroll
                for (int i = 0; i < kRecs; ++i) old[i] = a.d_rec_w[min(p + i * LP + in_row, last)];
            }
            const int next = min(p + S * kF, p1);
            fetch(next);
#pragma unroll
            for (int u = 0; u < kF; ++u) {
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    sum[s].x = fmaf(w[u], x[s][u].x, sum[s].x);
                    sum[s].y = fmaf(w[u], x[s][u].y, sum[s].y);
                    sum[s].z = fmaf(w[u], x[s][u].z, sum[s].z);
                    sum[s].w = fmaf(w[u], x[s][u].w, sum[s].w);
                }
            }
            if (kG) {
                // gradient of a record: over the row's lanes, the adjoint entries of the trials in which the source
                // fired; every lane gets every sum and keeps those of the records it fetched
                float keep[kRecs];
#pragma unroll
                for (int i = 0; i < kRecs; ++i) keep[i] = 0.0f;
#pragma unroll
                for (int u = 0; u < kF; ++u) {
                    float g = 0.0f;
#pragma unroll
                    for (int s = 0; s < kSteps; ++s) {
                        const unsigned m = fire >> (4 * s);
                        g += ((m & 1u) ? x[s][u].x : 0.0f) + ((m & 2u) ? x[s][u].y : 0.0f) + ((m & 4u) ? x[s][u].z : 0.0f) +
                             ((m & 8u) ? x[s][u].w : 0.0f);
                    }
                    if (LP > 1) g += dpp_move<0xB1>(g);   // quad_perm [1,0,3,2]
                    if (LP > 2) g += dpp_move<0x4E>(g);   // quad_perm [2,3,0,1]
                    if (LP > 4) g += dpp_move<0x141>(g);  // row_half_mirror: the other quad of these eight lanes
                    if (LP > 8) g += dpp_move<0x140>(g);  // row_mirror: the other eight of these sixteen
                    if (in_row == (kRecs > 1 ? (u & (LP - 1)) : u)) keep[kRecs > 1 ? u / LP : 0] = g;
                }
#pragma unroll
                for (int i = 0; i < kRecs; ++i) {
                    const int at = p + i * LP + in_row;
                    if (row_fired && i * LP + in_row < kF && at < p1) a.d_rec_w[at] = old[i] + keep[i];
                }
            }
            p = next;
        };
        while (busy) {
            if (grad)
                turn(std::true_type{});
            else
                turn(std::false_type{});
            busy = __ballot(p < p1) != 0ull;
        }
        // ---- the row's sum is complete: the state adjoint of its elements ----
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
            for (int off = LP; off < S * LP; off <<= 1) {
                sum[s].x += __shfl_xor(sum[s].x, off, kWave);
                sum[s].y += __shfl_xor(sum[s].y, off, kWave);
                sum[s].z += __shfl_xor(sum[s].z, off, kWave);
                sum[s].w += __shfl_xor(sum[s].w, off, kWave);
            }
        auto undo = [&](int c) {
            // (of values: a choice between members of a struct became a place in scratch memory, whose stores waited for the loads)
            auto pick = [c](float x0, float x1, float x2, float x3) { return c == 0 ? x0 : c == 1 ? x1 : c == 2 ? x2 : x3; };
            float g[2] = {0.0f, 0.0f}, v[2] = {0.0f, 0.0f};
            unsigned f[2] = {0u, 0u};
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                g[s] = pick(sum[s].x, sum[s].y, sum[s].z, sum[s].w);
                v[s] = pick(v4[s].x, v4[s].y, v4[s].z, v4[s].w);
                f[s] = (f4[s] >> (8 * c)) & 0xFFu;
            }
            el.undo(a, q, pr, e4 + c, ne, g, v, f);
        };
        if (have && lane_on && part < 4) {
            if (kOne && kPer >= 4) {
                undo(part);
            } else {
                if (!kOne) pr.load(a.prop, a.prop_stride, col);
                for (int c = part; c < 4; c += S) {
                    el.load(a, q, e4 + c, ne);
                    undo(c);
                }
            }
        }
    }
}

// ring slot `slot` = psc0 times the present adjoint of y1: what the state adjoint of the step the slot belongs to
// would write first, done ahead for the two-step form, whose transposed propagation reads it before that
__global__ __launch_bounds__(kBlock) void bwd_seed_slot_kernel(bmtk_glif3_bwd a, int slot)
{
    const int64_t ne = a.n_neurons * (int64_t)a.batch;
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= ne) return;
    const int64_t n = a.batch == 1 ? e : (int64_t)((uint32_t)e / (uint32_t)a.batch);
    const int64_t col = a.class_id ? (int64_t)a.class_id[n] : n;
#pragma unroll
    for (int k = 0; k < GLIF3_NREC; ++k)
        a.lam_ring[((int64_t)slot * GLIF3_NREC + k) * ne + e] =
            a.prop[(GLIF3_PSC0_0 + k) * a.prop_stride + col] * a.lam_y1[k * ne + e];
}

// d_rec_w[p] += sum over trials b in which source j spiked in step t of
// lam_ring[(t+d)%L][r][i*B+b]: one wavefront owns the whole row of a source, so
// the accumulation needs no atomics; lane = synapse.
__global__ __launch_bounds__(kBlock) void bwd_rec_grad_kernel(bmtk_glif3_bwd a, BwdStep q)
{
    const int batch = a.batch;
    const int64_t ne = a.n_neurons * (int64_t)batch;
    const int L = a.ring_slots;
    const int64_t j = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (j >= a.n_neurons) return;
    const uint64_t *__restrict__ bits = a.spike_bits + q.row * a.spike_bits_stride;
    const int slot0 = q.slot;
    const int p0 = a.rec_indptr[j], p1 = a.rec_indptr[j + 1];
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(a.rec_packed);
    for (int tile0 = 0; tile0 < batch; tile0 += kWave) {
        const unsigned long long m = trial_mask(bits, j, batch, tile0, min(kWave, batch - tile0));
        if (m == 0ull) continue;
        for (int p = p0 + lane_id(); p < p1; p += kWave) {
            const uint2 sy = rows[p];
            int slot = slot0 + (int)(sy.x >> 26);
            slot = slot >= L ? slot - L : slot;
            const int r = (sy.x >> 24) & 3;
            const int64_t i = sy.x & 0xFFFFFFu;
            const float *cell = a.lam_ring + (int64_t)(slot * GLIF3_NREC + r) * ne + i * batch + tile0;
            float acc = 0.0f;
            unsigned long long mm = m;
            while (mm) {
                const int b = __ffsll((long long)mm) - 1;
                mm &= mm - 1ull;
                acc += cell[b];
            }
            a.d_rec_w[p] += acc;
        }
    }
}

// Input weights.  The events of a step are ascending in source*batch+trial, so the trials in
// which one source fired are adjacent: the wavefront that holds the first event of such a run
// takes the whole run, which makes it the only writer of that source's row -- no atomics.
constexpr int kInpGradGrid = 1024;  // workgroups of the input-gradient part of a launch
// (a workgroup of any size: wavefront `wave` of `n_waves`)
__device__ __forceinline__ void bwd_inp_grad_waves(const bmtk_glif3_bwd &a, const BwdStep &q, int wave, int n_waves);
__device__ __forceinline__ void bwd_inp_grad_block(const bmtk_glif3_bwd &a, const BwdStep &q, int block, int n_blocks)
{
    bwd_inp_grad_waves(a, q, block * (kBlock / kWave) + threadIdx.x / kWave, n_blocks * (kBlock / kWave));
}
// source of an input event
__device__ __forceinline__ int event_source(int ev, int batch)
{
    return batch == 1 ? ev : (int)((uint32_t)ev / (uint32_t)batch);
}

// d_inp_w of source j's row += the adjoint cells of the trials of two runs of events: [k, k_end) of a step whose
// adjoint slots start at slot0, and [m, m_end) of the step before it (slots start one lower); either may be empty
__device__ __forceinline__ void inp_grad_row(const bmtk_glif3_bwd &a, int j, int slot0, int64_t k, int64_t k_end,
                                             int slot0_before, int64_t m, int64_t m_end)
{
    const int batch = a.batch;
    const int64_t ne = a.n_neurons * (int64_t)batch;
    const int L = a.ring_slots;
    const uint2 *__restrict__ rows = reinterpret_cast<const uint2 *>(a.inp_packed);
    const int p0 = a.inp_indptr[j], p1 = a.inp_indptr[j + 1];
    // four synapses per lane at a time: their records, then their adjoint cells, travel together
    constexpr int kUnroll = 4;
    for (int base = p0 + lane_id(); base < p1; base += kUnroll * kWave) {
        uint2 sy[kUnroll];
        float old[kUnroll], acc[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int p = base + u * kWave;
            if (p < p1) {
                sy[u] = rows[p];
                old[u] = a.d_inp_w[p];
            }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            acc[u] = 0.0f;
            if (base + u * kWave < p1) {
                const int d = (int)(sy[u].x >> 26), r = (sy[u].x >> 24) & 3;
                const int64_t i = sy[u].x & 0xFFFFFFu;
                int slot = slot0 + d;
                slot = slot >= L ? slot - L : slot;
                const float *cell = a.lam_ring + (int64_t)(slot * GLIF3_NREC + r) * ne + i * batch;
                for (int64_t kk = k; kk < k_end; ++kk) acc[u] += cell[a.in_events[kk] - j * batch];
                if (m < m_end) {
                    slot = slot0_before + d;
                    slot = slot >= L ? slot - L : slot;
                    cell = a.lam_ring + (int64_t)(slot * GLIF3_NREC + r) * ne + i * batch;
                    for (int64_t kk = m; kk < m_end; ++kk) acc[u] += cell[a.in_events[kk] - j * batch];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
            if (base + u * kWave < p1) a.d_inp_w[base + u * kWave] = old[u] + acc[u];
    }
}

__device__ __forceinline__ void bwd_inp_grad_waves(const bmtk_glif3_bwd &a, const BwdStep &q, int wave, int n_waves)
{
    const int batch = a.batch;
    const int slot0 = q.slot;
    const int64_t k0 = a.in_ptr[q.t], k1 = a.in_ptr[q.t + 1];
    for (int64_t k = k0 + wave; k < k1; k += n_waves) {
        const int j = event_source(a.in_events[k], batch);
        if (k > k0 && event_source(a.in_events[k - 1], batch) == j) continue;  // not the first event of its source's run
        int64_t k_end = k + 1;
        while (k_end < k1 && event_source(a.in_events[k_end], batch) == j) ++k_end;
        inp_grad_row(a, j, slot0, k, k_end, 0, 0, 0);
    }
}

// first event of [lo, hi) (ascending in source*batch+trial) whose source is at least j; called by a whole wavefront
// with the same arguments in every lane: 64 probes a round instead of one, two rounds for a step's few thousand
// events where a binary search is a chain of twelve dependent loads
__device__ __forceinline__ int64_t first_event_of(const int32_t *__restrict__ events, int64_t lo, int64_t hi, int j, int batch)
{
    const int lane = lane_id();
    while (hi - lo > kWave) {
        const int64_t stride = (hi - lo + kWave - 1) / kWave;
        const int64_t at = lo + lane * stride;
        const bool below = at < hi && event_source(events[at], batch) < j;  // ascending: the lanes below j are a prefix
        const int c = __popcll(__ballot(below));
        if (c == 0) return lo;
        const int64_t upto = lo + c * stride;
        lo = lo + (c - 1) * stride + 1;
        hi = upto < hi ? upto : hi;
    }
    const int64_t at = lo + lane;
    const unsigned long long at_least = __ballot(at < hi && event_source(events[at], batch) >= j);
    return at_least ? lo + (__ffsll((long long)at_least) - 1) : hi;
}

// The run of events of one source that begins at `at` (lo <= at < hi, the events of a step): its source and its end, which
// is `at` where the event before is of the same source.  Called by a whole wavefront with the same arguments in every lane:
// one load answers all of it for runs of up to 62 events.
__device__ __forceinline__ int64_t run_at(const int32_t *__restrict__ events, int64_t lo, int64_t at, int64_t hi, int batch, int &j)
{
    const int64_t mine = at - 1 + lane_id();  // (lane 0: the event before)
    const int source = event_source(events[mine < lo ? lo : mine < hi ? mine : hi - 1], batch);
    j = __builtin_amdgcn_readlane(source, 1);
    const unsigned long long same = __ballot(mine >= lo && mine < hi && source == j);
    if (same & 1ull) return at;
    const unsigned long long other = ~(same >> 1);  // (bit 63 is set: the shift brings in a zero)
    int64_t end = at + __ffsll((long long)other) - 1;
    while (end == at + 63 && end < hi && event_source(events[end], batch) == j) ++at, ++end;
    return end;
}

// The same for steps t = q.t and t-1 in ONE launch.  Two wavefronts must never update one source's row at a time, so
// a source with events in both steps belongs to the wavefront that holds the first event of its run in step t,
// which looks its run of step t-1 up (the events of a step are sorted) and adds both with one read-modify-write;
// runs of step t-1 whose source has no event in step t are taken by the holder of their first event.  The two steps'
// events are dealt out from the two ends of the wavefronts: with fewer events than wavefronts few get a chain of each.
__device__ __forceinline__ void bwd_inp_grad2_waves(const bmtk_glif3_bwd &a, const BwdStep &q, int wave, int n_waves)
{
    const int batch = a.batch;
    const int L = a.ring_slots;
    const int slot_t = q.slot, slot_p = q.slot == 0 ? L - 1 : q.slot - 1;
    const int64_t k0 = a.in_ptr[q.t], k1 = a.in_ptr[q.t + 1];
    const int64_t m0 = a.in_ptr[q.t - 1], m1 = k0;  // (in_ptr[t-1] .. in_ptr[t]: the events of step t-1)
    for (int64_t k = k0 + wave; k < k1; k += n_waves) {
        int j, same;
        const int64_t k_end = run_at(a.in_events, k0, k, k1, batch, j);
        if (k_end == k) continue;
        const int64_t m = first_event_of(a.in_events, m0, m1, j, batch);
        int64_t m_end = m;
        if (m < m1) {
            m_end = run_at(a.in_events, m0, m, m1, batch, same);
            if (same != j) m_end = m;
        }
        inp_grad_row(a, j, slot_t, k, k_end, slot_p, m, m_end);
    }
    for (int64_t m = m0 + (n_waves - 1 - wave); m < m1; m += n_waves) {
        int j;
        const int64_t m_end = run_at(a.in_events, m0, m, m1, batch, j);
        if (m_end == m) continue;
        const int64_t k = first_event_of(a.in_events, k0, k1, j, batch);
        if (k < k1 && event_source(a.in_events[k], batch) == j) continue;  // the source's run of step t takes it along
        inp_grad_row(a, j, slot_p, m, m_end, 0, 0, 0);
    }
}

// The state adjoint of step t and the input-weight gradient of the same step in one launch, side by side: the
// gradient reads the adjoint slots t+1 .. t+L-1 and the step's events, the state adjoint writes slot t -- neither
// needs the other.  The gradient's workgroups (a chain of dependent reads per event run, few wavefronts) take the
// lowest block ids so that they start first and run under the streaming state adjoint instead of after it.
__global__ __launch_bounds__(kBlock) void bwd_state_kernel(bmtk_glif3_bwd a, BwdStep q, int n_inp_blocks)
{
    if ((int)blockIdx.x < n_inp_blocks)
        bwd_inp_grad_block(a, q, (int)blockIdx.x, n_inp_blocks);
    else
        bwd_state_block(a, q, (int64_t)blockIdx.x - n_inp_blocks);
}

__global__ __launch_bounds__(kBlock) void fill_zero_kernel(float *x, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) x[i] = 0.0f;
}

// A wavefront a word of the bits: lane k fetches the word of step k, 64 steps with one load, the words then go round through
// scalar registers and lane e adds bit e.  What bounds it are trips to memory and lines: a word a load, one at a time, took 25.6 us for 36,012
// elements x 100 steps and 55 for 1.66 M x 40, scalar loads sixteen at a time 13.3 and 30.3, this takes 4.5 and 14.6.
__global__ __launch_bounds__(kBlock) void spike_counts_kernel(const uint64_t *__restrict__ bits, int64_t stride,
                                                              int64_t n_steps, int64_t ne,
                                                              int32_t *__restrict__ counts)
{
    const int lane = lane_id();
    const int64_t w = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave, e = w * kWave + lane;
    if (w * kWave >= ne) return;
    int c = 0;
    for (int64_t k = 0; k < n_steps; k += kWave) {
        const int here = (int)min(n_steps - k, (int64_t)kWave);
        const uint64_t v = lane < here ? bits[(k + lane) * stride + w] : 0ull;
        for (int u0 = 0; u0 < here; u0 += 8) {
#pragma unroll
            for (int u = u0; u < u0 + 8; ++u) {  // (words past the last step are 0)
                const uint64_t m = (uint64_t)(unsigned)__builtin_amdgcn_readlane((int)(v >> 32), u) << 32 | (unsigned)__builtin_amdgcn_readlane((int)v, u);
                c += __builtin_amdgcn_inverse_ballot_w64(m) ? 1 : 0;
            }
        }
    }
    if (e < ne) counts[e] = c;
}

// The loss of population rates and its derivative per spike (bmtk_rate_mse), in two launches.  work: [n_pops][batch] spikes of a
// population in a trial, [n_pops] its neurons, then a flag that some neuron's population does not exist.
//
// Spikes of a population: every workgroup adds its neurons' in LDS, where the cells fit, and its cells to the sums (a whole number
// whatever the order).  What bounds them are the launches: as some 25 array operations with three looks at the device in between the loss
// held up a training step by 200 to 250 us; 3,001 neurons x 12 trials, 17 populations: 7.7 and 3.8 us, 51,978 x 32: 18.5 and 8.1.
// A training step of 100 steps of the former 1.98 -> 1.80 ms (with the counts above).
constexpr int kRateCellsMax = 4096;
__global__ __launch_bounds__(kBlock) void rate_sums_kernel(const int32_t *__restrict__ counts, int64_t ne, int batch, const int64_t *__restrict__ pop_id,
                                                           int64_t n_pops, unsigned long long *__restrict__ work)
{
    __shared__ unsigned long long cells_l[kRateCellsMax];
    const int64_t cells = n_pops * batch, all = cells + n_pops;
    const bool in_lds = all <= kRateCellsMax;
    if (in_lds) {
        for (int i = threadIdx.x; i < (int)all; i += kBlock) cells_l[i] = 0ull;
        __syncthreads();
    }
    unsigned long long *to = in_lds ? cells_l : work;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < ne; e += (int64_t)gridDim.x * kBlock) {
        const int64_t i = e / batch;
        const int b = (int)(e - i * batch);
        const int64_t p = pop_id[i];
        if (p < 0 || p >= n_pops) {
            work[all] = 1ull;
            continue;
        }
        const int c = counts[e];
        if (c != 0) atomicAdd(to + p * batch + b, (unsigned long long)(long long)c);
        if (b == 0) atomicAdd(to + cells + p, 1ull);
    }
    if (in_lds) {
        __syncthreads();
        for (int i = threadIdx.x; i < (int)all; i += kBlock)
            if (cells_l[i] != 0ull) atomicAdd(work + i, cells_l[i]);
    }
}

// per_spike[e] for every element; the first workgroup's also the loss
__global__ __launch_bounds__(kBlock) void rate_mse_kernel(const unsigned long long *__restrict__ work, int64_t ne, int batch, const int64_t *__restrict__ pop_id,
                                                          int64_t n_pops, float n_steps, const float *__restrict__ targets, float *__restrict__ loss,
                                                          float *__restrict__ per_spike)
{
    const int64_t cells = n_pops * batch;
    const float n_rates = (float)cells;
    // rate of population p in trial b less its target, and what the rate is spikes over
    auto error = [&](int64_t p, int b, float &over) {
        over = (float)work[cells + p] * n_steps;
        return (float)(long long)work[p * batch + b] / over - targets[b * n_pops + p];
    };
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e < ne) {
        const int64_t i = e / batch, p = pop_id[i];
        float g = 0.0f, over;
        if (p >= 0 && p < n_pops) {
            const float err = error(p, (int)(e - i * batch), over);
            g = 2.0f * err / n_rates / over;
        }
        per_spike[e] = g;
    }
    if (blockIdx.x == 0) {
        __shared__ double part_l[kBlock / kWave];
        double sum = 0.0;
        for (int64_t c = threadIdx.x; c < cells; c += kBlock) {
            float over;
            const float err = error(c / batch, (int)(c % batch), over);
            sum += (double)(err * err);
        }
        for (int off = 1; off < kWave; off <<= 1) sum += __shfl_xor(sum, off, kWave);
        if (lane_id() == 0) part_l[threadIdx.x / kWave] = sum;
        __syncthreads();
        if (threadIdx.x == 0) {
            double total = 0.0;
            for (int w = 0; w < kBlock / kWave; ++w) total += part_l[w];
            *loss = (float)(total / (double)cells);
        }
    }
}

}  // namespace bmtk

using namespace bmtk;

namespace {

const void *blocked_variant(bool grad, bool ne24, bool wide)
{
#define BMTK_BLK(g, n, w) reinterpret_cast<const void *>(bwd_gather_blocked_kernel<g, n, w>)
    if (grad) {
        if (ne24) return wide ? BMTK_BLK(true, true, true) : BMTK_BLK(true, true, false);
        return wide ? BMTK_BLK(true, false, true) : BMTK_BLK(true, false, false);
    }
    if (ne24) return wide ? BMTK_BLK(false, true, true) : BMTK_BLK(false, true, false);
    return wide ? BMTK_BLK(false, false, true) : BMTK_BLK(false, false, false);
#undef BMTK_BLK
}

const void *blocked2_variant(bool lp16, bool grad, bool ne24)
{
#define BMTK_BLK2(l, g) (ne24 ? reinterpret_cast<const void *>(bwd_gather_blocked2_kernel<l, g, true>) \
                              : reinterpret_cast<const void *>(bwd_gather_blocked2_kernel<l, g, false>))
    if (lp16) return grad ? BMTK_BLK2(16, true) : BMTK_BLK2(16, false);
    return grad ? BMTK_BLK2(8, true) : BMTK_BLK2(8, false);
#undef BMTK_BLK2
}

// launch geometry of bwd_gather_blocked_kernel for a network on the current device
struct BlockedPlan {
    unsigned grid;
    int lp, rows_cu, sweeps, gpw, use_order;
    size_t lds;
    // the two-step kernel: twice the LDS per row, hence half as many row groups per wavefront and sweep
    int sweeps2, gpw2;
    size_t lds2;
};
constexpr size_t kBlkLdsMax = 160u * 1024u - 256u;  // a compute unit's LDS less the kernel's static part

int blocked_plan(const bmtk_glif3_bwd &a, BlockedPlan &pl)
{
    int dev = 0;
    (void)hipGetDevice(&dev);
    static int cu_count[64];
    int n_cu = (dev >= 0 && dev < 64) ? cu_count[dev] : 0;
    if (n_cu <= 0) {
        n_cu = 256;
        (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
        if (dev >= 0 && dev < 64) cu_count[dev] = n_cu;
    }
    const int cus = n_cu >= 8 ? n_cu / 8 : 1;  // workgroups per XCD, one per compute unit
    int bp = 4;
    while (bp < a.batch) bp <<= 1;
    pl.lp = bp / 4;
    const int per = kWave / pl.lp;
    int64_t rows_cu = (a.n_neurons + cus - 1) / cus;
    rows_cu = (rows_cu + per - 1) / per * per;
    const int64_t cap = (int64_t)kBlkWaves * kBlkMaxGroups * per;  // rows of one sweep
    pl.sweeps = (int)((rows_cu + cap - 1) / cap);
    pl.gpw = (int)((rows_cu + (int64_t)pl.sweeps * kBlkWaves * per - 1) / ((int64_t)pl.sweeps * kBlkWaves * per));
    pl.rows_cu = (int)rows_cu;
    pl.grid = (unsigned)cus * 8u;
    pl.lds = (size_t)kBlkWaves * pl.gpw * kWave * sizeof(float4);
    // the row order list (gradient riding along): two bytes per place, where it fits (up to 16 rows per thread)
    const size_t order_bytes = (size_t)pl.sweeps * kBlkWaves * pl.gpw * per * sizeof(uint16_t);
    pl.use_order = (pl.lds + order_bytes <= kBlkLdsMax && rows_cu <= 16 * kBlkThreads && rows_cu < 0xFFFF) ? 1 : 0;
    if (pl.use_order) pl.lds += order_bytes;
    const int64_t cap2 = (int64_t)kBlkWaves * (kBlkMaxGroups / 2) * per;
    pl.sweeps2 = (int)((rows_cu + cap2 - 1) / cap2);
    pl.gpw2 = (int)((rows_cu + (int64_t)pl.sweeps2 * kBlkWaves * per - 1) / ((int64_t)pl.sweeps2 * kBlkWaves * per));
    pl.lds2 = (size_t)kBlkWaves * pl.gpw2 * 2 * kWave * sizeof(float4) + blk2_sort_bytes((size_t)kBlkWaves * pl.gpw2 * per);
    static bool asked[8][64];
    const void *variants[8];
    for (int g = 0; g < 8; ++g) variants[g] = blocked_variant(g & 4, g & 2, g & 1);
    for (int g = 0; g < 8; ++g) {
        if (dev < 0 || dev >= 64 || asked[g][dev]) continue;
        const hipError_t err = hipFuncSetAttribute(
            variants[g], hipFuncAttributeMaxDynamicSharedMemorySize, (int)kBlkLdsMax);
        if (err != hipSuccess) {
            set_error("transposed propagation: cannot reserve LDS: %s", hipGetErrorString(err));
            return BMTK_E_LAUNCH;
        }
        asked[g][dev] = true;
    }
    static bool asked2[64];
    if (dev >= 0 && dev < 64 && !asked2[dev]) {
        for (int g = 0; g < 8; ++g) {
            const hipError_t err = hipFuncSetAttribute(blocked2_variant(g & 4, g & 2, g & 1), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kBlkLdsMax);
            if (err != hipSuccess) {
                set_error("transposed propagation: cannot reserve LDS: %s", hipGetErrorString(err));
                return BMTK_E_LAUNCH;
            }
        }
        asked2[dev] = true;
    }
    return BMTK_OK;
}

// what the blocked form of the table must satisfy
int blocked_check(const bmtk_glif3_bwd &a, const char *who)
{
    BMTK_REQUIRE(a.blk_count > 0 && a.blk_count % 8 == 0 && a.blk_indptr && a.blk_packed,
                 "%s: the blocked table needs blk_count (a multiple of 8), blk_indptr and blk_packed", who);
    BMTK_REQUIRE(a.batch % 4 == 0 && a.batch <= kWave, "%s: the blocked table serves batches that are a multiple of 4 up to 64",
                 who);
    BMTK_REQUIRE((int64_t)a.ring_slots * GLIF3_NREC * a.n_neurons * a.batch < (1ll << 30),
                 "%s: the adjoint ring must stay below 4 GB for the blocked table", who);
    return BMTK_OK;
}

int blocked_launch(const bmtk_glif3_bwd &a, const BwdStep &q, const BlockedPlan &pl, bool grad, bool inp_grad,
                   hipStream_t st)
{
    const bool ne24 = a.n_neurons * (int64_t)a.batch < (1ll << 24);
    bmtk_glif3_bwd args = a;
    BwdStep step = q;
    int lp = pl.lp, rows_cu = pl.rows_cu, sweeps = pl.sweeps, gpw = pl.gpw, use_order = pl.use_order;
    int do_inp = inp_grad ? 1 : 0;
    void *params[] = {&args, &step, &lp, &rows_cu, &sweeps, &gpw, &use_order, &do_inp};
    const hipError_t err = hipLaunchKernel(blocked_variant(grad, ne24, pl.lp >= 8), dim3(pl.grid), dim3(kBlkThreads),
                                           params, pl.lds, st);
    if (err != hipSuccess) {
        set_error("transposed propagation: launch failed: %s", hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    return BMTK_OK;
}

// the two-step kernel for steps q.t and q.t - 1
int blocked2_launch(const bmtk_glif3_bwd &a, const BwdStep &q, const BlockedPlan &pl, bool grad, bool inp_grad, hipStream_t st)
{
    const bool ne24 = a.n_neurons * (int64_t)a.batch < (1ll << 24);
    bmtk_glif3_bwd args = a;
    BwdStep step = q;
    int rows_cu = pl.rows_cu, sweeps = pl.sweeps2, gpw = pl.gpw2;
    int do_inp = inp_grad ? 1 : 0;
    void *params[] = {&args, &step, &rows_cu, &sweeps, &gpw, &do_inp};
    const hipError_t err = hipLaunchKernel(blocked2_variant(pl.lp > 8, grad, ne24), dim3(pl.grid), dim3(kBlkThreads), params, pl.lds2, st);
    if (err != hipSuccess) {
        set_error("transposed propagation (two steps): launch failed: %s", hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    return BMTK_OK;
}


// ---- the swept form ----
template <int LP>
const void *sweep_variant(bool one, bool two)
{
    if (one)
        return two ? reinterpret_cast<const void *>(bwd_sweep_kernel<LP, true, true>)
                   : reinterpret_cast<const void *>(bwd_sweep_kernel<LP, true, false>);
    return two ? reinterpret_cast<const void *>(bwd_sweep_kernel<LP, false, true>)
               : reinterpret_cast<const void *>(bwd_sweep_kernel<LP, false, false>);
}

struct SweepPlan {
    int lp;
    SweepLaunch launch;
    unsigned grid;
};

int sweep_plan(const bmtk_glif3_bwd &a, SweepPlan &pl)
{
    BMTK_REQUIRE(a.batch % 4 == 0 && a.batch <= kWave, "glif3_simulate_bwd: the swept form serves batches that are a multiple of 4 up to 64");
    const int64_t ne = a.n_neurons * a.batch;
    BMTK_REQUIRE(ne < (1ll << 24) && (int64_t)a.ring_slots * GLIF3_NREC * ne < (1ll << 30),
                 "glif3_simulate_bwd: the swept form needs fewer than 2^24 elements and an adjoint ring below 4 GB");
    BMTK_REQUIRE(a.rec_indptr && a.rec_packed && a.ring_slots >= 4,
                 "glif3_simulate_bwd: the swept form needs the recurrent table and ring_slots >= largest delay + 3");
    int dev = 0, n_cu = 256;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    pl.lp = 1;
    while (pl.lp * 4 < a.batch) pl.lp <<= 1;
    const int per = kWave / pl.lp;
    const int64_t groups = (int64_t)n_cu * kSweepPerCu * kSweepWaves * per;  // lane groups the chip holds
    pl.launch.splits = 1;
    while (pl.launch.splits < per && a.n_neurons * pl.launch.splits * 2 <= groups) pl.launch.splits *= 2;
    const int rows_set = per / pl.launch.splits;
    pl.launch.n_sets = (int)((a.n_neurons + rows_set - 1) / rows_set);
    pl.launch.n_row_wg = (pl.launch.n_sets + kSweepWaves - 1) / kSweepWaves;
    pl.launch.do_grad = a.d_rec_w != nullptr ? 1 : 0;
    pl.grid = (unsigned)(pl.launch.n_row_wg + (a.d_inp_w ? n_cu : 0));
    return BMTK_OK;
}

int sweep_launch(const bmtk_glif3_bwd &a, const SweepPlan &pl, const BwdStep &q, bool two, hipStream_t st)
{
    bmtk_glif3_bwd args = a;
    BwdStep step = q;
    SweepLaunch launch = pl.launch;
    void *params[] = {&args, &step, &launch};
    const bool one = launch.splits == kWave / pl.lp;
    const void *fn = pl.lp == 1 ? sweep_variant<1>(one, two) : pl.lp == 2 ? sweep_variant<2>(one, two)
                   : pl.lp == 4 ? sweep_variant<4>(one, two) : pl.lp == 8 ? sweep_variant<8>(one, two) : sweep_variant<16>(one, two);
    const hipError_t err = hipLaunchKernel(fn, dim3(pl.grid), dim3(kSweepThreads), params, 0, st);
    if (err != hipSuccess) {
        set_error("glif3_simulate_bwd: launch failed: %s", hipGetErrorString(err));
        return BMTK_E_LAUNCH;
    }
    return BMTK_OK;
}

}  // namespace

namespace {

// what every entry point that takes the whole bmtk_glif3_bwd requires of it
int bwd_check(const bmtk_glif3_bwd *bwd, const char *who)
{
    BMTK_REQUIRE(bwd != nullptr, "%s: bwd is null", who);
    const bmtk_glif3_bwd &a = *bwd;
    BMTK_REQUIRE(a.n_neurons > 0 && a.batch > 0, "%s: n_neurons and batch must be positive", who);
    const int64_t ne = a.n_neurons * (int64_t)a.batch;
    BMTK_REQUIRE(ne < (1ll << 31) && a.n_neurons < (1ll << 24), "%s: network too large", who);
    BMTK_REQUIRE(a.ring_slots > 1 && a.ring_slots <= 64, "%s: ring_slots must lie in 2..64", who);
    BMTK_REQUIRE(a.h > 0.0f && a.dampening >= 0.0f, "%s: h must be positive, dampening non-negative", who);
    BMTK_REQUIRE(a.prop && a.prop_stride > 0 && (a.class_id || a.prop_stride >= a.n_neurons),
                 "%s: prop table missing or too small", who);
    BMTK_REQUIRE(a.save_v && a.save_flags && a.spike_bits, "%s: the forward record is incomplete", who);
    BMTK_REQUIRE(a.spike_bits_stride >= (ne + 63) / 64, "%s: spike_bits_stride too small", who);
    BMTK_REQUIRE(a.lam_V && a.lam_asc && a.lam_y1 && a.lam_y2 && a.lam_ring && a.gz,
                 "%s: adjoint state pointers must be non-null", who);
    BMTK_REQUIRE(!(a.dl_dz && a.dl_dz_const), "%s: give dl_dz or dl_dz_const, not both", who);
    const bool has_rec = a.rec_indptr != nullptr;
    BMTK_REQUIRE(!has_rec || a.rec_packed, "%s: recurrent table needs rec_packed", who);
    BMTK_REQUIRE(!a.d_rec_w || has_rec, "%s: d_rec_w without a recurrent table", who);
    BMTK_REQUIRE(!a.d_blk_w || a.blk_count != 0, "%s: d_blk_w without the blocked table", who);
    BMTK_REQUIRE(!a.d_inp_w || (a.in_ptr && a.in_events && a.inp_indptr && a.inp_packed),
                 "%s: d_inp_w needs the input events and the input table", who);
    return BMTK_OK;
}

}  // namespace

extern "C" int bmtk_glif3_simulate_bwd(const bmtk_glif3_bwd *bwd, int64_t step0, int64_t n_steps, void *stream)
{
    {
        const int rc = bwd_check(bwd, "glif3_simulate_bwd");
        if (rc != BMTK_OK) return rc;
    }
    const bmtk_glif3_bwd &a = *bwd;
    const int64_t ne = a.n_neurons * (int64_t)a.batch;
    const bool blocked = a.blk_count != 0;
    BlockedPlan pl{};
    if (blocked) {
        int rc = blocked_check(a, "glif3_simulate_bwd");
        if (rc == BMTK_OK) rc = blocked_plan(a, pl);
        if (rc != BMTK_OK) return rc;
    }
    const bool has_rec = a.rec_indptr != nullptr;
    const bool inp_grad = a.d_inp_w != nullptr;
    BMTK_REQUIRE(step0 >= 0 && n_steps >= 0, "glif3_simulate_bwd: step0 and n_steps must be non-negative");
    hipStream_t st = (hipStream_t)stream;
    const unsigned rows_grid = (unsigned)((a.n_neurons + kBlock / kWave - 1) / (kBlock / kWave));
    const unsigned tiles = (unsigned)((a.batch + kWave - 1) / kWave);
    const unsigned elem_grid = (unsigned)((ne + kBlock - 1) / kBlock);
    int bp = 1;  // trial-tile width: the batch rounded up to a power of two, at most one wavefront
    while (bp < a.batch && bp < kWave) bp <<= 1;
    int64_t k_top = n_steps - 1;
    if (a.swept) {
        BMTK_REQUIRE(!blocked, "glif3_simulate_bwd: give the blocked table or ask for the swept form, not both");
        SweepPlan sp{};
        int rc = sweep_plan(a, sp);
        if (rc != BMTK_OK) return rc;
        if (n_steps > 0)
            hipLaunchKernelGGL(bwd_seed_slot_kernel, dim3(elem_grid), dim3(kBlock), 0, st, a, (int)((step0 + k_top) % a.ring_slots));
        while (k_top >= 0) {
            const bool two = k_top >= 1;
            rc = sweep_launch(a, sp, BwdStep{step0 + k_top, k_top, 1, (int)((step0 + k_top) % a.ring_slots)}, two, st);
            if (rc != BMTK_OK) return rc;
            k_top -= two ? 2 : 1;
        }
        BMTK_CHECK_LAUNCH("glif3_simulate_bwd");
        return BMTK_OK;
    }
    // Two steps per pass over the blocked table where gz has room for both steps' partial sums and a lane holds
    // whole adjoint rows of eight lanes (batches above 16): pairs (k, k-1) from the top, a step left over at the
    // end goes the one-step way.
    if (blocked && a.gz_planes >= 16 && pl.lp >= 8 && n_steps >= 2) {
        hipLaunchKernelGGL(bwd_seed_slot_kernel, dim3(elem_grid), dim3(kBlock), 0, st, a, (int)((step0 + k_top) % a.ring_slots));
        for (; k_top >= 1; k_top -= 2) {
            BwdStep q{step0 + k_top, k_top, 8, (int)((step0 + k_top) % a.ring_slots)};
            const int rc = blocked2_launch(a, q, pl, a.d_blk_w != nullptr, inp_grad, st);
            if (rc != BMTK_OK) return rc;
            if (a.d_rec_w && !a.d_blk_w) {  // (before the state adjoint, which overwrites a slot step t-1's gradient reads)
                const BwdStep before{q.t - 1, q.row - 1, 8, (int)((q.t - 1) % a.ring_slots)};
                hipLaunchKernelGGL(bwd_rec_grad_kernel, dim3(rows_grid), dim3(kBlock), 0, st, a, q);
                hipLaunchKernelGGL(bwd_rec_grad_kernel, dim3(rows_grid), dim3(kBlock), 0, st, a, before);
            }
            hipLaunchKernelGGL(bwd_state2_kernel, dim3(elem_grid), dim3(kBlock), 0, st, a, q, k_top - 1 > 0 ? 1 : 0);
        }
    }
    for (int64_t k = k_top; k >= 0; --k) {
        BwdStep q{step0 + k, k, blocked ? 8 : 1, (int)((step0 + k) % a.ring_slots)};
        // The recurrent weight gradient of step t reads the adjoint slots t+1 .. t+L-1, which the state adjoint of
        // this step (it writes slot t) leaves alone: it can ride along with the transposed propagation, which
        // reads the same slots before the state adjoint runs.  Batches of more than one tile keep the kernel of
        // their own (several wavefronts would share a row).
        const bool fused = blocked ? a.d_blk_w != nullptr : (a.d_rec_w && tiles == 1);
        if (blocked) {
            const int rc = blocked_launch(a, q, pl, fused, inp_grad, st);
            if (rc != BMTK_OK) return rc;
        } else if (has_rec && a.batch % 4 == 0 && a.batch <= kWave) {
            if (fused)
                hipLaunchKernelGGL(bwd_gather4_kernel<true>, dim3(rows_grid), dim3(kBlock), 0, st, a, q, bp / 4);
            else
                hipLaunchKernelGGL(bwd_gather4_kernel<false>, dim3(rows_grid), dim3(kBlock), 0, st, a, q, bp / 4);
        } else if (has_rec) {
            if (fused)
                hipLaunchKernelGGL(bwd_gather_kernel<true>, dim3(rows_grid, tiles), dim3(kBlock), 0, st, a, q, bp);
            else
                hipLaunchKernelGGL(bwd_gather_kernel<false>, dim3(rows_grid, tiles), dim3(kBlock), 0, st, a, q, bp);
        } else {
            hipLaunchKernelGGL(fill_zero_kernel, dim3(elem_grid), dim3(kBlock), 0, st, a.gz, ne);
        }
        const int n_inp_blocks = (inp_grad && !blocked) ? kInpGradGrid : 0;  // (the blocked kernel took it along)
        hipLaunchKernelGGL(bwd_state_kernel, dim3(elem_grid + n_inp_blocks), dim3(kBlock), 0, st, a, q, n_inp_blocks);
        if (a.d_rec_w && !fused) hipLaunchKernelGGL(bwd_rec_grad_kernel, dim3(rows_grid), dim3(kBlock), 0, st, a, q);
    }
    BMTK_CHECK_LAUNCH("glif3_simulate_bwd");
    return BMTK_OK;
}

extern "C" int bmtk_glif3_step_bwd(const bmtk_glif3_bwd *bwd, int64_t step0, int64_t k, int32_t gz_parts, void *stream)
{
    const int rc = bwd_check(bwd, "glif3_step_bwd");
    if (rc != BMTK_OK) return rc;
    BMTK_REQUIRE(step0 >= 0 && k >= 0, "glif3_step_bwd: step0 and k must be non-negative");
    BMTK_REQUIRE(gz_parts == 1 || gz_parts == 8, "glif3_step_bwd: gz holds 1 sum or 8 partial sums per element");
    const bmtk_glif3_bwd &a = *bwd;
    const int64_t ne = a.n_neurons * (int64_t)a.batch;
    BwdStep q{step0 + k, k, gz_parts, (int)((step0 + k) % a.ring_slots)};
    hipLaunchKernelGGL(bwd_state_kernel, dim3((unsigned)((ne + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       (hipStream_t)stream, a, q, 0);
    BMTK_CHECK_LAUNCH("glif3_step_bwd");
    return BMTK_OK;
}

extern "C" int bmtk_csr_weight_grad(const bmtk_glif3_bwd *bwd, int64_t step0, int64_t k, void *stream)
{
    const int rc = bwd_check(bwd, "csr_weight_grad");
    if (rc != BMTK_OK) return rc;
    BMTK_REQUIRE(step0 >= 0 && k >= 0, "csr_weight_grad: step0 and k must be non-negative");
    const bmtk_glif3_bwd &a = *bwd;
    BMTK_REQUIRE(a.d_rec_w || a.d_inp_w, "csr_weight_grad: neither d_rec_w nor d_inp_w is given");
    BwdStep q{step0 + k, k, 1, (int)((step0 + k) % a.ring_slots)};
    if (a.d_rec_w)
        hipLaunchKernelGGL(bwd_rec_grad_kernel, dim3((unsigned)((a.n_neurons + kBlock / kWave - 1) / (kBlock / kWave))),
                           dim3(kBlock), 0, (hipStream_t)stream, a, q);
    if (a.d_inp_w)  // (bwd_state_kernel with nothing but gradient workgroups)
        hipLaunchKernelGGL(bwd_state_kernel, dim3(kInpGradGrid), dim3(kBlock), 0, (hipStream_t)stream, a, q, kInpGradGrid);
    BMTK_CHECK_LAUNCH("csr_weight_grad");
    return BMTK_OK;
}

extern "C" int bmtk_csr_propagate_bwd(const int32_t *indptr, const bmtk_synapse *packed, int64_t n_neurons,
                                      int32_t batch, const float *lam_ring, int32_t L, int64_t step, float *gz,
                                      int32_t trials_per_lane, void *stream)
{
    BMTK_REQUIRE(indptr && packed && lam_ring && gz, "csr_propagate_bwd: pointers must be non-null");
    BMTK_REQUIRE(n_neurons > 0 && batch > 0 && step >= 0, "csr_propagate_bwd: bad sizes or step");
    BMTK_REQUIRE(n_neurons * (int64_t)batch < (1ll << 31) && n_neurons < (1ll << 24), "csr_propagate_bwd: network too large");
    BMTK_REQUIRE(L > 1 && L <= 64, "csr_propagate_bwd: L must lie in 2..64");
    const bool can4 = batch % 4 == 0 && batch <= kWave;
    BMTK_REQUIRE(trials_per_lane == 0 || trials_per_lane == 1 || (trials_per_lane == 4 && can4),
                 "csr_propagate_bwd: trials_per_lane must be 0 (choose), 1, or 4 for batches that are a multiple of 4 up to 64");
    bmtk_glif3_bwd a{};
    a.n_neurons = n_neurons;
    a.batch = batch;
    a.ring_slots = L;
    a.rec_indptr = indptr;
    a.rec_packed = packed;
    a.lam_ring = const_cast<float *>(lam_ring);
    a.gz = gz;
    BwdStep q{step, 0, 1, (int)(step % L)};
    const unsigned rows_grid = (unsigned)((n_neurons + kBlock / kWave - 1) / (kBlock / kWave));
    int bp = 1;
    while (bp < batch && bp < kWave) bp <<= 1;
    if (trials_per_lane == 4 || (trials_per_lane == 0 && can4))
        hipLaunchKernelGGL(bwd_gather4_kernel<false>, dim3(rows_grid), dim3(kBlock), 0, (hipStream_t)stream, a, q, bp / 4);
    else
        hipLaunchKernelGGL(bwd_gather_kernel<false>, dim3(rows_grid, (unsigned)((batch + kWave - 1) / kWave)), dim3(kBlock), 0,
                           (hipStream_t)stream, a, q, bp);
    BMTK_CHECK_LAUNCH("csr_propagate_bwd");
    return BMTK_OK;
}

extern "C" int bmtk_csr_propagate_bwd_blocked(const int32_t *blk_indptr, const bmtk_synapse *blk_packed, int32_t blk_count,
                                              int64_t n_neurons, int32_t batch, const float *lam_ring, int32_t L,
                                              int64_t step, float *gz_parts, void *stream)
{
    BMTK_REQUIRE(lam_ring && gz_parts, "csr_propagate_bwd_blocked: pointers must be non-null");
    BMTK_REQUIRE(n_neurons > 0 && batch > 0 && step >= 0, "csr_propagate_bwd_blocked: bad sizes or step");
    BMTK_REQUIRE(n_neurons * (int64_t)batch < (1ll << 31) && n_neurons < (1ll << 24),
                 "csr_propagate_bwd_blocked: network too large");
    BMTK_REQUIRE(L > 1 && L <= 64, "csr_propagate_bwd_blocked: L must lie in 2..64");
    bmtk_glif3_bwd a{};
    a.n_neurons = n_neurons;
    a.batch = batch;
    a.ring_slots = L;
    a.blk_count = blk_count;
    a.blk_indptr = blk_indptr;
    a.blk_packed = blk_packed;
    a.lam_ring = const_cast<float *>(lam_ring);
    a.gz = gz_parts;
    BlockedPlan pl{};
    int rc = blocked_check(a, "csr_propagate_bwd_blocked");
    if (rc == BMTK_OK) rc = blocked_plan(a, pl);
    if (rc != BMTK_OK) return rc;
    BwdStep q{step, 0, 8, (int)(step % a.ring_slots)};
    rc = blocked_launch(a, q, pl, false, false, (hipStream_t)stream);
    if (rc != BMTK_OK) return rc;
    BMTK_CHECK_LAUNCH("csr_propagate_bwd_blocked");
    return BMTK_OK;
}

extern "C" int bmtk_csr_propagate_bwd_blocked_plan(int64_t n_neurons, int32_t batch, int32_t *plan_host)
{
    BMTK_REQUIRE(plan_host != nullptr, "csr_propagate_bwd_blocked_plan: plan_host is null");
    BMTK_REQUIRE(n_neurons > 0 && n_neurons < (1ll << 24) && batch > 0 && batch % 4 == 0 && batch <= kWave,
                 "csr_propagate_bwd_blocked_plan: n_neurons must lie in 1..2^24-1, batch be a multiple of 4 up to 64");
    bmtk_glif3_bwd a{};
    a.n_neurons = n_neurons;
    a.batch = batch;
    BlockedPlan pl{};
    const int rc = blocked_plan(a, pl);
    if (rc != BMTK_OK) return rc;
    plan_host[0] = (int32_t)pl.grid;
    plan_host[1] = pl.rows_cu;
    plan_host[2] = pl.sweeps;
    plan_host[3] = pl.gpw;
    return BMTK_OK;
}

extern "C" int bmtk_spike_counts(const uint64_t *spike_bits, int64_t stride, int64_t n_steps, int64_t ne,
                                 int32_t *counts, void *stream)
{
    BMTK_REQUIRE(spike_bits && counts && ne > 0 && n_steps >= 0 && stride >= (ne + 63) / 64,
                 "spike_counts: bad sizes or null pointers");
    hipLaunchKernelGGL(spike_counts_kernel, dim3((unsigned)((ne + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       (hipStream_t)stream, spike_bits, stride, n_steps, ne, counts);
    BMTK_CHECK_LAUNCH("spike_counts");
    return BMTK_OK;
}

extern "C" int bmtk_rate_mse(const int32_t *counts, int64_t n_neurons, int32_t batch, int64_t n_steps, const int64_t *pop_id, int64_t n_pops,
                             const float *targets, int64_t *work, float *loss, float *per_spike, void *stream)
{
    BMTK_REQUIRE(counts && pop_id && targets && work && loss && per_spike, "rate_mse: pointers must be non-null");
    BMTK_REQUIRE(n_neurons > 0 && batch > 0 && n_pops > 0 && n_steps > 0, "rate_mse: sizes must be positive");
    const int64_t ne = n_neurons * batch;
    const int64_t blocks = (ne + kBlock - 1) / kBlock;
    BMTK_REQUIRE(blocks < (1ll << 31) && n_pops < (1ll << 31), "rate_mse: too many elements or populations");
    const hipStream_t st = (hipStream_t)stream;
    // (eight elements a thread: a workgroup's cells are added to the sums one by one)
    const int64_t sums = (blocks + 7) / 8 < 512 ? (blocks + 7) / 8 : 512;
    hipLaunchKernelGGL(rate_sums_kernel, dim3((unsigned)sums), dim3(kBlock), 0, st, counts, ne, batch, pop_id, n_pops, (unsigned long long *)work);
    hipLaunchKernelGGL(rate_mse_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, st, (const unsigned long long *)work, ne, batch, pop_id, n_pops,
                       (float)n_steps, targets, loss, per_spike);
    BMTK_CHECK_LAUNCH("rate_mse");
    return BMTK_OK;
}
