// kernels.hpp — gfx950 device code of libttperf_hip.
//
// One optimizer step over a small tensor set is one launch (see adam_small_kernel); over any
// other, at most three on one stream (an update of more than 2^32 work-items is split, and
// mark_mom_init_kernel follows a momentum step whose decisions did not set the marks: of more
// than 4096 tensors, or without decisions on the device):
//   norm_partials_kernel  reads only the gradients (2 B/param bf16, 4 B/param fp32) in 16 KiB
//                         tiles: fp64 sum of squares of the unscaled grads, one partial per
//                         block; the last block to finish sums the partials in index order
//                         (deterministic), decides found_inf / skip and the clip coefficient,
//                         advances the step count and the loss scale.  Two launches above
//                         256 MiB of gradients: non-temporal loads, then cached loads for the
//                         last 256 MiB;
//   adam_lane_kernel /    one fused pass per element: grad transform (unscale, clip), weight
//   sgd_lane_kernel       decay, the optimizer update and the bf16 copy, one or two elements
//                         per lane; sgd_kernel does the same with four elements per lane
//                         (16-byte fp32 and 8-byte bf16 vectors) for MIXED SGD momentum
//                         updates whose gradients fit the Infinity Cache.  Each element is touched once.
// Optimizer state is stored in records (see kRec): in MIXED mode each 64-element group of the
// flat store keeps its fp32 master, m and v side by side in one 768-byte record; in FP32 mode
// (where the fp32 master is the model-facing weight and stays contiguous) m and v share
// 512-byte records.  The update then streams grad, state records and the bf16 copy instead of
// nine separate arrays: the state read and write of a group hit the same DRAM pages, and the
// step no longer depends on where the allocator happened to place five large buffers
// relative to each other (GPT-2 124M, fresh allocations, 6 rounds: 571-617 us per step with
// separate buffers, 570-580 us with records).
// Work is a table of chunks of kChunk elements (the last chunk of a tensor is shorter; every
// chunk starts on a 64-element boundary).  Update blocks are dispatched in (reverse) chunk
// order, so the resident blocks sweep a narrow window of each buffer, which keeps DRAM pages
// open.  The four-element update (MIXED SGD momentum, cached gradients) runs one 256-thread block
// per chunk, one vector per lane, at most kUpdBlocksPerCU blocks per CU; for it 16K-element
// chunks, a persistent grid, two or four vectors per lane, 512-thread blocks and unlimited
// occupancy each measured 3-12% slower (as a four-element Adam update, which the lane forms
// have replaced).  No MFMA: nothing here is a contraction.
//
// Arithmetic matches the oracle bit for bit: no contraction (-ffp-contract=off), IEEE
// division and square root (HIP's correctly rounded fp32 div/sqrt), denormals kept.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ttp {

constexpr int kBlock = 256;     // 4 wave64s: norm pass, its decisions and helper kernels
constexpr int kUpdBlock = 256;  // 4 wave64s: the four-element update
constexpr int kVec = 4;         // elements per lane per vector
constexpr uint32_t kChunk = kUpdBlock * kVec;  // 1024 elements: one vector per lane
// Resident blocks per CU of the four-element update.  The host reserves LDS_per_CU /
// kUpdBlocksPerCU bytes of (unused) dynamic LDS per block so that no more than this many are
// resident: 16 waves per CU sweep the HBM pages of the streams with fewer row conflicts than
// the 32+ waves that registers alone would allow (measured on the four-element Adam update
// that the lane forms have replaced: separate state arrays, GPT-2 124M, same box,
// interleaved repeats: 568 us vs 588 us for 512-thread blocks at 3 per CU, 622 us uncapped;
// GPT-2 XL fp32: 7.36 ms vs 7.63 ms).  With state records, 4, 5, 6 and 8 blocks per CU
// measure alike and 3 is 27% slower.
constexpr int kUpdBlocksPerCU = 4;
constexpr uint32_t kChunkDecay = 1u;

// State records.  Element i of a record-stored buffer sits at
//   slot_base + (i / kRec) * stride + i % kRec
// where slot_base is the record array's base plus slot * kRec.  Tensors start on kRec
// boundaries, so a tensor's state is whole records and a lane's 4-element vector never
// straddles two.  A contiguous buffer is the case stride == kRec.
constexpr uint32_t kRec = 64;
constexpr uint32_t kStrideMixed = 3 * kRec;  // MIXED: [master | m | v]
constexpr uint32_t kStrideMV = 2 * kRec;     // FP32:  [m | v]

__host__ __device__ __forceinline__ uint64_t rec_index(uint64_t i, uint32_t stride) {
    return (i / kRec) * stride + (i % kRec);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Chunk {
    uint64_t begin;  // first element (flat index)
    uint32_t count;  // elements in this chunk (exact, not padded)
    uint32_t meta;   // bit 0: decay; bits 8..31: tensor index
};

// chunk k of a table as one 16-byte load (a field-wise read compiles to two dependent loads:
// the count first, then begin and meta)
__device__ __forceinline__ Chunk load_chunk(const Chunk* t, uint64_t k) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(t + k);
    return Chunk{(uint64_t)w.x | ((uint64_t)w.y << 32), w.z, w.w};
}

// Device-resident step state.  Written only by the block that decides (write_state), by
// scaler_update_kernel and by swap_step_kernel (and by the host between
// steps); read by the update pass that follows it on the same stream.
struct DevState {
    float scale;             // loss scale (persistent)
    int32_t growth_tracker;  // clean steps since the last scale change (persistent)
    uint64_t t;              // applied steps while loss scaling is on (persistent)
    double sumsq;            // last pass: sum of squares of the unscaled grads
    double norm;             // last pass: sqrt(sumsq)
    float inv_scale;         // last pass: 1/scale used to unscale
    float clip_coef;         // last pass: clip multiplier (1 when not clipping)
    float bias1, bias2;      // last pass: Adam bias corrections for the new t
    int32_t found_inf;       // last pass: a non-finite gradient was seen
    int32_t skip;            // last pass: the update must not run
    // steps that deferred the scale update since the last one (several optimizers over one
    // store: torch's GradScaler.step per optimizer, then one update): kPendingStep once such a
    // step ran, | kPendingInf if one of them saw an overflow.  The next scale update combines
    // it with its own and clears it (persistent).
    int32_t pending;
    int32_t reserved;
};
static_assert(sizeof(DevState) == 64, "DevState is one 64-byte block");
constexpr int32_t kPendingInf = 1, kPendingStep = 2;

// ------------------------------------------------------------------------------------
// bf16
// ------------------------------------------------------------------------------------
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// round-to-nearest-even; NaN -> canonical 0x7FC0
__device__ __forceinline__ uint32_t bf16_rne(float x) {
    const uint32_t u = __float_as_uint(x);
    const uint32_t r = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
    return ((u & 0x7FFFFFFFu) > 0x7F800000u) ? 0x7FC0u : r;
}

__device__ __forceinline__ uint32_t bf16_pack(float a, float b) {
    return bf16_rne(a) | (bf16_rne(b) << 16);
}

// ------------------------------------------------------------------------------------
// vector memory helpers (all addresses 16-byte / 8-byte aligned by construction)
// ------------------------------------------------------------------------------------
__device__ __forceinline__ f32x4 ld4(const float* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
}
__device__ __forceinline__ void st4(float* p, f32x4 v) {
    __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(p));
}

// 4 gradients as fp32 from either storage type, with ordinary (temporal) loads: the
// four-element update runs only on gradients that fit the 256 MB Infinity Cache, where the
// norm pass or the backward left them
__device__ __forceinline__ f32x4 ld_grad4(const float* g, uint64_t i) {
    return *reinterpret_cast<const f32x4*>(g + i);
}
__device__ __forceinline__ f32x4 ld_grad4(const uint16_t* g, uint64_t i) {
    const u32x2 w = *reinterpret_cast<const u32x2*>(g + i);
    f32x4 r;
    r.x = bf16_lo(w.x);
    r.y = bf16_hi(w.x);
    r.z = bf16_lo(w.y);
    r.w = bf16_hi(w.y);
    return r;
}

__device__ __forceinline__ void st_bf16x4(uint16_t* p, uint64_t i, f32x4 v) {
    u32x2 w;
    w.x = bf16_pack(v.x, v.y);
    w.y = bf16_pack(v.z, v.w);
    __builtin_nontemporal_store(w, reinterpret_cast<u32x2*>(p + i));
}

// partial vector (the last one of a tensor): element-wise stores of the first n lanes
__device__ __forceinline__ void st4_partial(float* p, f32x4 v, int n) {
    p[0] = v.x;
    if (n > 1) p[1] = v.y;
    if (n > 2) p[2] = v.z;
}
__device__ __forceinline__ void st_bf16x4_partial(uint16_t* p, f32x4 v, int n) {
    p[0] = (uint16_t)bf16_rne(v.x);
    if (n > 1) p[1] = (uint16_t)bf16_rne(v.y);
    if (n > 2) p[2] = (uint16_t)bf16_rne(v.z);
}

// ------------------------------------------------------------------------------------
// block reduction of a double (fixed shape: deterministic)
// ------------------------------------------------------------------------------------
// x of the lane that a DPP control names (both 32-bit halves)
template <int kCtrl>
__device__ __forceinline__ double dpp(double x) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, kCtrl, 0xF, 0xF, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), kCtrl, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

// The wave's sum in every lane, as the butterfly x += x[lane ^ off] for off = 32, 16, 8, 4, 2, 1
// gives it (bit for bit), without LDS permutes: a swap of the wave's halves, then of its 16-lane
// rows; within a row a rotation by 8, then by 4 (the values repeat every 8 lanes by then, so lane
// + 4 holds what lane ^ 4 does), then quad permutes.  Each LDS permute waited ~100 cycles, twelve
// of them in a chain at the end of every block: nanoGPT-char's AdamW step took 53.6 us with them
// and takes 53.2, the last of 8 GPT-2 124M shards 74.3 and 74.0.
__device__ __forceinline__ double wave_sum(double x) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    {
        const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)u, false, false);
        const auto hi =
            __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
        x = __builtin_bit_cast(double, (uint64_t)lo[0] | ((uint64_t)hi[0] << 32)) +
            __builtin_bit_cast(double, (uint64_t)lo[1] | ((uint64_t)hi[1] << 32));
    }
    {
        const uint64_t w = __builtin_bit_cast(uint64_t, x);
        const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)w, (uint32_t)w, false, false);
        const auto hi =
            __builtin_amdgcn_permlane16_swap((uint32_t)(w >> 32), (uint32_t)(w >> 32), false, false);
        x = __builtin_bit_cast(double, (uint64_t)lo[0] | ((uint64_t)hi[0] << 32)) +
            __builtin_bit_cast(double, (uint64_t)lo[1] | ((uint64_t)hi[1] << 32));
    }
    x += dpp<0x128>(x);  // row_ror:8
    x += dpp<0x124>(x);  // row_ror:4
    x += dpp<0x4E>(x);   // quad_perm:[2,3,0,1]
    x += dpp<0xB1>(x);   // quad_perm:[1,0,3,2]
    return x;
}

__device__ __forceinline__ double block_sum(double x, double* lds) {
    x = wave_sum(x);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) lds[wave] = x;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 0; w < kBlock / 64; ++w) r += lds[w];
    }
    __syncthreads();
    return r;  // valid in thread 0
}

// ------------------------------------------------------------------------------------
// the step's decisions: found_inf / skip, the clip coefficient, the step count, the loss scale
// ------------------------------------------------------------------------------------
struct FinalizeArgs {
    const double* partials;
    const uint32_t* idx;    // non-null: partial k is partials[idx[k]] (per-tensor sums)
    uint32_t npartials;     // 0: no norm pass ran (step counting only)
    int32_t scaler_on;      // unscale by 1/scale, skip on inf, update the scale
    int32_t defer_scale;    // with scaler_on: note the step and its overflow in `pending`;
                            // leave the scale as it is
    int32_t count_t;        // the step count lives on the device: advance it (unless skipped)
    int32_t probe;          // only compute sumsq/norm (ttp_grad_norm); touch nothing else
    int32_t growth_interval;
    double growth_factor;
    double backoff_factor;
    double max_norm;        // > 0: clip
    const float* bias_tab;  // [2*bias_len]: (1-beta1^t, 1-beta2^t) for t = 1..bias_len
    uint32_t bias_len;      // t > bias_len: both corrections are exactly 1.0f
    int32_t want_bias;
    DevState* st;
    uint32_t* mom_init;       // momentum marks (see kMomNew) of the n_mom stepped tensors
    const uint32_t* mom_ids;  // (n_mom 0: none to set)
    uint32_t n_mom;
};

// A tensor's momentum mark: 0 while its buffer holds no value, kMomNew in the step that gives it
// its first one where the decisions mark it (the update that follows must still see that it is
// the first), 1 from then on.  Any mark but 0 means a buffer that holds a value to every step
// that does not stage its marks.  (Marked in a launch after the update, a loss-scaled SGD momentum
// step took 13.1 us at 1.0M parameters and takes 10.4; nanoGPT-char 44.5 and 43.1; at GPT-2 124M,
// 414 us, the two do not differ beyond noise.)
constexpr uint32_t kMomNew = 2u;

// torch _amp_update_scale_ semantics, over this step's overflow and the pending overflow of
// the steps that deferred their update since the last one (found_inf summed over optimizers,
// as GradScaler.update does): the new scale and growth tracker (the pending flag is cleared)
struct ScaleUpdate {
    float scale;
    int32_t tracker;
};
__device__ __forceinline__ ScaleUpdate next_scale(float scale, int32_t tracker, int32_t pending,
                                                  int32_t found, int32_t growth_interval,
                                                  double growth_factor, double backoff_factor) {
    if (found || (pending & kPendingInf)) return {(float)((double)scale * backoff_factor), 0};
    const int32_t ok = tracker + 1;
    if (ok == growth_interval) {
        const float ns = (float)((double)scale * growth_factor);
        return {ns - ns == 0.0f ? ns : scale, 0};  // grows only to a finite scale
    }
    return {scale, ok};
}

// (float)(1 - beta^t) for t = 1 .. bias_len from the host-built table; 1.0f beyond (and for
// t = 0, which no applied step has)
__device__ __forceinline__ float bias_entry(const float* tab, uint32_t len, uint64_t t, int j) {
    return (t >= 1 && t <= len) ? tab[2 * (t - 1) + j] : 1.0f;
}

// the bias corrections of both outcomes: of t + 1 if the step applies, of t if it is skipped
struct BiasPair {
    float next1, next2, same1, same2;
};
__device__ __forceinline__ BiasPair load_bias(const FinalizeArgs& a, uint64_t t) {
    if (!(a.count_t && a.want_bias)) return {1.0f, 1.0f, 1.0f, 1.0f};
    return {bias_entry(a.bias_tab, a.bias_len, t + 1, 0), bias_entry(a.bias_tab, a.bias_len, t + 1, 1),
            bias_entry(a.bias_tab, a.bias_len, t, 0), bias_entry(a.bias_tab, a.bias_len, t, 1)};
}

// what a step does, from the sum of squares of its unscaled gradients
struct Decision {
    double norm;
    float inv, coef;
    int32_t found, skip;
};
__device__ __forceinline__ float unscale_factor(const FinalizeArgs& a, float scale) {
    return a.scaler_on ? (float)(1.0 / (double)scale) : 1.0f;
}
__device__ __forceinline__ Decision decide(const FinalizeArgs& a, float scale, double sumsq) {
    Decision d;
    d.inv = unscale_factor(a, scale);
    d.norm = sqrt(sumsq);
    d.found = !(sumsq <= 1.7976931348623157e308);  // inf or NaN
    d.skip = a.scaler_on && d.found;
    d.coef = 1.0f;
    if (a.max_norm > 0.0) {
        double cd = a.max_norm / (d.norm + 1e-6);
        if (cd > 1.0) cd = 1.0;
        d.coef = (float)cd;
    }
    return d;
}

// the step state after the step (one thread): s0 is the state before it
__device__ __forceinline__ void write_state(const FinalizeArgs& a, const DevState& s0,
                                            const BiasPair& b, double sumsq, const Decision& d) {
    DevState* st = a.st;
    st->sumsq = sumsq;
    st->norm = d.norm;
    if (a.probe) return;
    st->found_inf = d.found;
    st->skip = d.skip;
    st->inv_scale = d.inv;
    st->clip_coef = d.coef;
    if (a.count_t) {
        st->t = d.skip ? s0.t : s0.t + 1;
        if (a.want_bias) {
            st->bias1 = d.skip ? b.same1 : b.next1;
            st->bias2 = d.skip ? b.same2 : b.next2;
        }
    }
    if (a.scaler_on) {
        if (a.defer_scale) {
            st->pending = s0.pending | kPendingStep | (d.found ? kPendingInf : 0);
        } else {
            const ScaleUpdate u = next_scale(s0.scale, s0.growth_tracker, s0.pending, d.found,
                                             a.growth_interval, a.growth_factor,
                                             a.backoff_factor);
            st->scale = u.scale;
            st->growth_tracker = u.tracker;
            st->pending = 0;
        }
    }
}

// ------------------------------------------------------------------------------------
// the last block of a launch
// ------------------------------------------------------------------------------------
// A value that the launch's last block reads: stored and loaded as a relaxed atomic of device
// scope, past the caches that other XCDs do not share.
__device__ __forceinline__ void st_device(double* p, double x) {
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_device(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Tickets: kTicketGroups counters 128 B apart, which block b takes from counter b modulo
// kTicketGroups, and one more that the last block of each group takes from.  One counter for a
// whole launch made 2,048 blocks wait in line for the same word.  All are zero between
// launches: the block that takes a counter's last ticket sets it back.
constexpr uint32_t kTicketGroups = 32, kTicketPitch = 32;
constexpr uint32_t kTicketWords = (kTicketGroups + 1) * kTicketPitch;
__device__ __forceinline__ bool last_ticket(uint32_t* p, uint32_t of) {
    const bool last =
        __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == of - 1;
    if (last) __hip_atomic_store(p, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return last;
}

// Whether this block is the launch's last to get here; every block of the launch calls it, with
// all its lanes, after thread 0's st_device() stores, which the last block may then read with
// ld_device().  Thread 0 waits until its stores have been acknowledged (device-scope stores
// write through, so that is at memory) before it takes its ticket.  That wait takes the place of
// a release fence: a device-scope fence per block also writes the XCD's L2 back and costs
// ~50 ns per block, one block after another.
// Measured (MLP AdamW with clipping, fp32): the step 9.0-9.5 us in two launches against 12.7 with
// a launch of one block for the decisions; the norm kernel's tail takes about as long as that
// launch did where the GPU is the bound (nanoGPT-char 53.7 against 53.6 us).
__device__ __forceinline__ bool is_last_block(uint32_t* tickets, uint32_t* lds_flag) {
    if (threadIdx.x == 0) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0);
        asm volatile("" ::: "memory");
        const uint32_t g = blockIdx.x % kTicketGroups;
        const uint32_t size = (gridDim.x - g + kTicketGroups - 1) / kTicketGroups;
        const uint32_t groups = min(gridDim.x, kTicketGroups);
        *lds_flag = last_ticket(tickets + g * kTicketPitch, size) &&
                    last_ticket(tickets + kTicketGroups * kTicketPitch, groups);
    }
    __syncthreads();
    return *lds_flag != 0;
}

// One block of kBlock lanes combines the partials in index order (deterministic) and decides.
// kLast: in the last block of the launch that stored the partials (see is_last_block).
// Partials: all loads of a round issued before the adds, each thread's order fixed
// (deterministic); with an index list (per-tensor sums), a round's indices load first.
// Loads past the end read the last entry and count as 0 in the adds (a branch or a select
// at each load made the compiler wait for it there).  s0 is the step state before the step,
// which the caller loaded first; the bias corrections of both outcomes load beside the partials.
template <bool kLast>
__device__ __forceinline__ void finalize_block(const FinalizeArgs& a, const DevState& s0,
                                               double* lds) {
    constexpr int kPer = 8;
    const uint32_t n = a.npartials;
    const BiasPair bias = load_bias(a, s0.t);
    double s = 0.0;
    for (uint32_t base = 0; base < n; base += kBlock * kPer) {
        uint32_t at[kPer];
        double v[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) at[k] = min(base + (uint32_t)k * kBlock + threadIdx.x, n - 1);
        if (a.idx) {
#pragma unroll
            for (int k = 0; k < kPer; ++k) at[k] = a.idx[at[k]];
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            v[k] = kLast ? ld_device(a.partials + at[k]) : a.partials[at[k]];
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            s += base + (uint32_t)k * kBlock + threadIdx.x < n ? v[k] : 0.0;
    }
    s = block_sum(s, lds);
    if (threadIdx.x == 0) write_state(a, s0, bias, s, decide(a, s0.scale, s));
    if (a.n_mom) {
        if (threadIdx.x == 0) lds[0] = s;
        __syncthreads();
        if (decide(a, s0.scale, lds[0]).skip) return;
        for (uint32_t k = threadIdx.x; k < a.n_mom; k += kBlock) {
            uint32_t* m = a.mom_init + a.mom_ids[k];
            *m = *m == 0u ? kMomNew : 1u;
        }
    }
}

// the decisions alone, in a launch of one block: without a norm pass (step counting), or over
// per-tensor sums
__global__ __launch_bounds__(kBlock) void norm_finalize_kernel(FinalizeArgs a) {
    __shared__ double lds[kBlock / 64];
    const DevState s0 = *a.st;
    finalize_block<false>(a, s0, lds);
}

// ------------------------------------------------------------------------------------
// norm pass: per-block partial sums of squares of the unscaled gradients, and the decisions
// ------------------------------------------------------------------------------------
// 16-byte loads: 8 bf16 or 4 fp32 gradients per lane
template <typename GradT>
struct GradVec;
template <>
struct GradVec<uint16_t> {
    static constexpr int kElems = 8;
    typedef uint32_t raw __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ float at(const raw& w, int j) {
        return (j & 1) ? bf16_hi(w[j >> 1]) : bf16_lo(w[j >> 1]);
    }
    // element j of a vector that starts as zeros
    static __device__ __forceinline__ void put(raw& w, int j, uint16_t h) {
        w[j >> 1] |= (j & 1) ? ((uint32_t)h << 16) : (uint32_t)h;
    }
};
template <>
struct GradVec<float> {
    static constexpr int kElems = 4;
    typedef f32x4 raw;
    static __device__ __forceinline__ float at(const raw& w, int j) { return w[j]; }
    static __device__ __forceinline__ void put(raw& w, int j, float x) { w[j] = x; }
};

// Norm tiles: kNormLoads 16-byte loads per lane, so a tile is 16 KiB of gradients (8192 bf16
// or 4096 fp32); the pass has its own tile table (same tensors, bigger pieces than the update's
// chunks) so each descriptor fetch is amortised over 4 loads per lane.
constexpr int kNormLoads = 4;
template <typename GradT>
constexpr uint32_t norm_tile_elems() {
    return (uint32_t)(kBlock * kNormLoads * 16 / sizeof(GradT));
}

// Grid-stride over the norm tiles t0 .. t1-1, one partial per block.  A whole tile (every tile
// but a tensor's last) is four unconditional 16-byte loads per lane, all issued before the
// arithmetic (the scheduling barrier keeps the compiler from interleaving them with it, which
// left one or two loads in flight: 6.0-6.3 TB/s against 6.7-6.9 at GPT-2 774M / 1558M).
// kNT selects non-temporal loads.  The host runs the pass as two launches: non-temporal over
// all but the last kCachedGradBytes of gradients, then cached loads over those, which the
// update, walking the chunks in reverse, reads first and so finds in the 256 MB Infinity
// Cache (measured on GPT-2 124M: update 531 us after this pass vs 559 us alone; at 774M and
// 1558M fp32 the split pass runs 232 and 931 us against 246-260 and 978-1030 us with cached
// loads throughout, the update unchanged).  Each block writes one partial, and with kDecide the
// launch's last block combines all of them (an earlier launch's included) and decides.  Squares
// of fp32 values are exact in fp64, and any inf/NaN gradient makes the sum non-finite.
// st and partials are not __restrict__: the deciding block writes the one and reads the other
// through fin.
template <typename GradT, bool kNT, bool kDecide>
__global__ __launch_bounds__(kBlock) void norm_partials_kernel(const GradT* __restrict__ g,
                                                               const Chunk* __restrict__ tiles,
                                                               uint32_t t0, uint32_t t1,
                                                               const DevState* st,
                                                               int32_t scaler_on,
                                                               double* partials,
                                                               FinalizeArgs fin,
                                                               uint32_t* __restrict__ tickets) {
    typedef GradVec<GradT> GV;
    typedef typename GV::raw R;
    constexpr int E = GV::kElems;
    constexpr uint32_t kTile = norm_tile_elems<GradT>();
    __shared__ double lds[kBlock / 64];
    // The first tile's descriptor and the step state load together, ahead of the arithmetic on
    // the scale, and each further descriptor beside the tile before it: one round trip less
    // before each tile's data than with the loads where their values are used.
    uint32_t c = t0 + blockIdx.x;
    Chunk ch = load_chunk(tiles, c < t1 ? c : t0);
    const DevState s0 = *st;  // whole, since any block may be the launch's last
    // both are here from this point on (left to itself, the compiler loads the descriptor after
    // the division)
    asm volatile("" ::"s"(ch.count), "s"(s0.scale) : "memory");
    const float inv = scaler_on ? (float)(1.0 / (double)s0.scale) : 1.0f;
    // two accumulators (element j of a vector goes to acc[j & 1]): a fixed order, so the
    // sum stays deterministic, with half the dependent-add chain.  The square of an fp32 value
    // is exact in fp64, so fma(x, x, acc) rounds exactly as acc + x*x does (one rounding, of
    // the add) with one instruction instead of two.
    double acc[2] = {0.0, 0.0};
    for (; c < t1; c += gridDim.x) {
        const R* q = reinterpret_cast<const R*>(g + ch.begin) + threadIdx.x;
        const uint32_t count = ch.count;
        const uint32_t next = c + gridDim.x;  // (below 2^28 tiles, 2^24 blocks: no wrap)
        ch = load_chunk(tiles, next < t1 ? next : c);
        if (count == kTile) {
            R w[kNormLoads];
#pragma unroll
            for (int l = 0; l < kNormLoads; ++l)
                w[l] = kNT ? __builtin_nontemporal_load(q + l * kBlock) : q[l * kBlock];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int l = 0; l < kNormLoads; ++l) {
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    const double x = (double)(GV::at(w[l], j) * inv);
                    acc[j & 1] = __builtin_fma(x, x, acc[j & 1]);
                }
            }
        } else {  // a tensor's last tile: only the vectors (and elements) below its count
#pragma unroll
            for (int l = 0; l < kNormLoads; ++l) {
                const uint32_t off = (uint32_t)(l * kBlock + threadIdx.x) * E;
                const uint32_t nv = off < count ? min(count - off, (uint32_t)E) : 0u;
                if (nv) {
                    const R w = q[l * kBlock];
#pragma unroll
                    for (int j = 0; j < E; ++j) {
                        const double x = (uint32_t)j < nv ? (double)(GV::at(w, j) * inv) : 0.0;
                        acc[j & 1] = __builtin_fma(x, x, acc[j & 1]);
                    }
                }
            }
        }
    }
    const double b = block_sum(acc[0] + acc[1], lds);
    if constexpr (kDecide) {
        __shared__ uint32_t last;
        if (threadIdx.x == 0) st_device(partials + blockIdx.x, b);
        if (is_last_block(tickets, &last)) finalize_block<true>(fin, s0, lds);
    } else {
        if (threadIdx.x == 0) partials[blockIdx.x] = b;
    }
}

// ttp_scaler_update: the scale update of an iteration whose steps all deferred it; nothing
// when no step deferred it since the last update, so an iteration's scale never moves twice
__global__ void scaler_update_kernel(DevState* st, int32_t growth_interval, double growth_factor,
                                     double backoff_factor) {
    if (threadIdx.x == 0 && blockIdx.x == 0 && (st->pending & kPendingStep)) {
        const ScaleUpdate u = next_scale(st->scale, st->growth_tracker, st->pending, 0,
                                         growth_interval, growth_factor, backoff_factor);
        st->scale = u.scale;
        st->growth_tracker = u.tracker;
        st->pending = 0;
    }
}

// ttp_swap_step: one optimizer's step count into slot `save` (none: -1), another's from slot
// `load` (0: -1).  A launch of a few microseconds where the host read the count back and wrote the
// other one, each behind everything queued: two optimizers over 300 small tensors took 95 us an
// iteration that way and take 30.
__global__ void swap_step_kernel(DevState* st, uint64_t* slots, int32_t save, int32_t load) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        const uint64_t next = load >= 0 ? slots[load] : 0;
        if (save >= 0) slots[save] = st->t;
        st->t = next;
    }
}

// Per-tensor sums of squares (ttp_grad_sumsq_tensors), from one norm_partials_kernel block per
// tile: block t adds the tile sums of the t-th listed tensor, tiles tile_start[t] ..
// tile_start[t+1]-1, each lane in tile order, then the fixed block reduction, into
// sums[tensor_ids[t]].
// the sum of tile_sums[b .. e-1] in a fixed order (valid in thread 0): lane l adds tiles
// b + l, b + l + kBlock, b + l + 2 kBlock, ... in that order, a round of kSumRound of them
// loaded before their adds (as finalize_block), then the fixed block reduction.  One
// order for every caller, so a tensor's sum does not depend on which call computed its tiles.
// The round size sets only how many loads are in flight, not the order (tiles past the end
// add +0.0 to a sum of squares, which leaves it as it is).  A round's loads are unconditional
// (an index past the end reads tile e-1, whose value the add then replaces by +0.0), so all of
// them are in flight at once: with a bounds check at each load, the compiler waited for each
// one before the next (GPT-2 124M's largest tensor, 4,712 tiles of four wave partials,
// combined in 8.6 us).
constexpr int kSumRound = 16;
__device__ __forceinline__ double sum_tiles(const double* __restrict__ tile_sums, uint32_t b,
                                            uint32_t e, double* lds) {
    constexpr int kPer = kSumRound;
    double s = 0.0;
    for (uint32_t base = b; base < e; base += kBlock * kPer) {
        double v[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            v[k] = tile_sums[min(base + (uint32_t)k * kBlock + threadIdx.x, e - 1)];
#pragma unroll
        for (int k = 0; k < kPer; ++k) s += base + (uint32_t)k * kBlock + threadIdx.x < e ? v[k] : 0.0;
    }
    return block_sum(s, lds);
}

// A tensor's sum supersedes tile sums an earlier accumulate with sums left pending for it.
__global__ __launch_bounds__(kBlock) void tensor_sums_kernel(const double* __restrict__ tile_sums,
                                                             const uint32_t* __restrict__ tile_start,
                                                             const uint32_t* __restrict__ tensor_ids,
                                                             double* __restrict__ sums,
                                                             uint32_t* __restrict__ pending) {
    __shared__ double lds[kBlock / 64];
    const uint32_t t = blockIdx.x;
    const double s = sum_tiles(tile_sums, tile_start[t], tile_start[t + 1], lds);
    if (threadIdx.x == 0) {
        sums[tensor_ids[t]] = s;
        pending[tensor_ids[t]] = 0u;
    }
}

// The wave partials an accumulate with sums leaves per 16 KiB tile (kWaves of them, in wave
// order; see accumulate_grad_tiles_kernel): tile k's sum is their total added as block_sum
// adds its waves' sums, (((0 + w0) + w1) + w2) + w3, so it equals the norm pass's partial of
// that tile bit for bit.
constexpr int kWaves = kBlock / 64;
__device__ __forceinline__ double tile_from_waves(const double* __restrict__ w, uint32_t k) {
    double r = 0.0;
#pragma unroll
    for (int j = 0; j < kWaves; ++j) r += w[(uint64_t)k * kWaves + j];
    return r;
}

// Before a step that takes its norm from per-tensor sums: block t combines the t-th stepped
// tensor's tile sums that accumulates with their sums left in the store-wide array (the wave
// partials of its tiles, from kWaves x tile_base[tensor]), if it has any pending: each tile
// from its waves, then the tiles in sum_tiles' order, so the tensor's sum equals what
// ttp_grad_sumsq_tensors gives for the same gradients.  One launch per step instead of one
// per accumulate; its last block combines the sums of all stepped tensors and decides (it reads
// them through fin, so sums is not __restrict__).
__global__ __launch_bounds__(kBlock) void combine_pending_sums_kernel(
    const double* __restrict__ acc_waves, const uint32_t* __restrict__ tile_base,
    const uint32_t* __restrict__ tile_start, const uint32_t* __restrict__ tensor_ids,
    uint32_t* __restrict__ pending, double* sums, FinalizeArgs fin,
    uint32_t* __restrict__ tickets) {
    __shared__ double lds[kBlock / 64];
    __shared__ uint32_t last;
    const DevState s0 = *fin.st;  // any block may be the last
    asm volatile("" ::: "memory");
    const uint32_t t = blockIdx.x, i = tensor_ids[t];
    const double* w = acc_waves + (uint64_t)tile_base[i] * kWaves;
    // nothing pending (uniform over the block): the sum is there already
    const uint32_t e = pending[i] ? tile_start[t + 1] - tile_start[t] : 0u;
    // sum_tiles' order, rounds and unconditional loads, over tile values formed from the wave
    // partials
    constexpr int kPer = kSumRound;
    double s = 0.0;
    for (uint32_t base = 0; base < e; base += kBlock * kPer) {
        double v[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            v[k] = tile_from_waves(w, min(base + (uint32_t)k * kBlock + threadIdx.x, e - 1));
#pragma unroll
        for (int k = 0; k < kPer; ++k) s += base + (uint32_t)k * kBlock + threadIdx.x < e ? v[k] : 0.0;
    }
    if (e) {
        s = block_sum(s, lds);
        if (threadIdx.x == 0) {
            st_device(sums + i, s);
            pending[i] = 0u;
        }
    }
    if (is_last_block(tickets, &last)) finalize_block<true>(fin, s0, lds);
}

// ------------------------------------------------------------------------------------
// fused Adam / AdamW update
// ------------------------------------------------------------------------------------
constexpr uint32_t kUseInv = 1u;    // multiply grads by st->inv_scale
constexpr uint32_t kUseClip = 2u;   // multiply grads by st->clip_coef
constexpr uint32_t kDevBias = 4u;   // take bias1/bias2 from st (step count on device)
constexpr uint32_t kCheckSkip = 8u; // return if st->skip
constexpr uint32_t kDecoupled = 16u;
constexpr uint32_t kWdOn = 32u;

struct AdamArgs {
    const Chunk* chunks;
    uint32_t nchunks;
    uint32_t flags;
    float lr, b1, omb1, b2, omb2, eps, bias1, bias2, decay_mul, wd;
    const DevState* st;
};

struct Coefs {
    float inv, clip, bias1, bias2;
};

// One element in the op order of py/optim.py:76-86 after the grad transforms and decay.
__device__ __forceinline__ void adam_elem(float& p, float g, float& m, float& v,
                                          const AdamArgs& a, const Coefs& k, bool use_inv,
                                          bool use_clip, bool decay) {
    if (use_inv) g = g * k.inv;
    if (use_clip) g = g * k.clip;
    if (decay) {
        if (a.flags & kDecoupled) p = p * a.decay_mul;
        else g = g + a.wd * p;
    }
    m = a.b1 * m + a.omb1 * g;
    const float gsq = g * g;
    v = a.b2 * v + a.omb2 * gsq;
    const float m_hat = m / k.bias1;
    const float v_hat = v / k.bias2;
    const float denom = __builtin_sqrtf(v_hat) + a.eps;
    const float step = a.lr * (m_hat / denom);
    p = p - step;
}

// Stores of one vector: whole (16 B / 8 B) or the first n elements (a tensor's last vector).
// a, b, c point at the vector's first element in their buffers; the bf16 copy of va goes to
// p16[i].
template <bool kMixed>
__device__ __forceinline__ void store_vec(float* a, float* b, float* c, uint16_t* p16, uint64_t i,
                                          const f32x4& va, const f32x4& vb, const f32x4& vc,
                                          int n) {
    if (n >= kVec) {
        st4(a, va);
        if (b) st4(b, vb);
        if (c) st4(c, vc);
        if (kMixed) st_bf16x4(p16, i, va);
    } else {
        st4_partial(a, va, n);
        if (b) st4_partial(b, vb, n);
        if (c) st4_partial(c, vc, n);
        if (kMixed) st_bf16x4_partial(p16 + i, va, n);
    }
}

// ------------------------------------------------------------------------------------
// lane forms: one or two elements per lane, for stores whose gradients exceed the Infinity
// Cache
// ------------------------------------------------------------------------------------
// Each block of kLanes lanes takes 1/lane_parts<kE, kLanes, kIt>() of a chunk (the last chunks
// first): kIt consecutive pieces of kLanes x kE elements, each lane kE consecutive elements of
// each piece, with no occupancy cap.  A lane holds 14-32 B of loads in flight instead of the
// four-element form's 56-64 B (one 4-element vector per stream), and full occupancy
// (registers allow 32 waves per CU) hides the
// arithmetic.  The state is addressed from the record base alone (one 64-bit address per
// lane, the other slots at immediate offsets), and the chunk descriptor is one 16-byte scalar
// load issued together with the device-state loads, so two dependent scalar round trips
// (arguments, then descriptor and state) precede the data loads.  The host picks the shape
// per optimizer and mode (see kLaneAdamMixed in ttperf.hip).  Measured (interleaved rounds,
// x a plain 256-lane non-temporal copy of the same bytes): GPT-2 774M mixed AdamW, one element
// per lane, 256 lanes, two pieces: 1.014-1.018 against 0.96-0.98 with one piece and
// 0.91-0.93 for a four-element Adam form; GPT-2 1558M fp32 AdamW, one element, 128 lanes, two
// pieces: 1.018-1.027 against 0.977 for two elements in one piece and 0.905-0.927.  Below
// the Infinity Cache bound, GPT-2 124M mixed AdamW with 128-lane blocks of two pieces runs its
// update in 0.512-0.514 ms against 0.522 ms for the four-element Adam form, and 5% faster when
// a backward has just rewritten the gradients; FP32 AdamW and SGD momentum at 57.5M params run
// their steps 2-3% faster than in four-element forms.  A four-element form dispatched half the
// grid for a skipped step's early exit.
template <int kE, int kLanes, int kIt>
constexpr uint32_t lane_parts() {
    return kChunk / (kLanes * kE * kIt);
}

// kE (1, 2 or 4) gradients as fp32 (ordinary loads: faster here than non-temporal ones at
// 774M).  A lane's kE elements start at a multiple of kE and tensors start on 64-element
// boundaries, so a lane whose tensor ends inside it still reads inside the tensor's footprint.
template <int kE>
__device__ __forceinline__ void ld_grad_lane(const uint16_t* g, uint64_t i, float* out) {
    static_assert(kE == 1 || kE == 2 || kE == 4, "1, 2 or 4 elements per lane");
    if constexpr (kE == 1) {
        out[0] = __uint_as_float((uint32_t)g[i] << 16);
    } else if constexpr (kE == 2) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(g + i);
        out[0] = bf16_lo(w);
        out[1] = bf16_hi(w);
    } else {
        const u32x2 w = *reinterpret_cast<const u32x2*>(g + i);
        out[0] = bf16_lo(w.x);
        out[1] = bf16_hi(w.x);
        out[2] = bf16_lo(w.y);
        out[3] = bf16_hi(w.y);
    }
}
template <int kE>
__device__ __forceinline__ void ld_grad_lane(const float* g, uint64_t i, float* out) {
    static_assert(kE == 1 || kE == 2 || kE == 4, "1, 2 or 4 elements per lane");
    if constexpr (kE == 1) {
        out[0] = g[i];
    } else if constexpr (kE == 2) {
        const f32x2 w = *reinterpret_cast<const f32x2*>(g + i);
        out[0] = w.x;
        out[1] = w.y;
    } else {
        const f32x4 w = *reinterpret_cast<const f32x4*>(g + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = w[j];
    }
}
// kE fp32 values, non-temporal
template <int kE>
__device__ __forceinline__ void ld_lane(const float* p, float* out) {
    if constexpr (kE == 1) {
        out[0] = __builtin_nontemporal_load(p);
    } else if constexpr (kE == 2) {
        const f32x2 w = __builtin_nontemporal_load(reinterpret_cast<const f32x2*>(p));
        out[0] = w.x;
        out[1] = w.y;
    } else {
        const f32x4 w = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = w[j];
    }
}
// the first n (1..kE) of kE fp32 values, non-temporal: one vector store when n == kE
template <int kE>
__device__ __forceinline__ void st_lane(float* p, const float* v, int n) {
    if constexpr (kE == 1) {
        __builtin_nontemporal_store(v[0], p);
    } else if constexpr (kE == 2) {
        if (n == 2)
            __builtin_nontemporal_store(f32x2{v[0], v[1]}, reinterpret_cast<f32x2*>(p));
        else
            __builtin_nontemporal_store(v[0], p);
    } else {
        if (n == 4) {
            __builtin_nontemporal_store(f32x4{v[0], v[1], v[2], v[3]},
                                        reinterpret_cast<f32x4*>(p));
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (j < n) __builtin_nontemporal_store(v[j], p + j);
        }
    }
}
// the bf16 copies of the first n (1..kE) of kE values, non-temporal or (kNT false) ordinary
template <bool kNT, typename T>
__device__ __forceinline__ void st_word(T* p, T w) {
    if constexpr (kNT) __builtin_nontemporal_store(w, p);
    else *p = w;
}
template <int kE, bool kNT = true>
__device__ __forceinline__ void st_bf16_lane(uint16_t* p, const float* v, int n) {
    if constexpr (kE == 1) {
        st_word<kNT>(p, (uint16_t)bf16_rne(v[0]));
    } else if constexpr (kE == 2) {
        if (n == 2)
            st_word<kNT>(reinterpret_cast<uint32_t*>(p), bf16_pack(v[0], v[1]));
        else
            st_word<kNT>(p, (uint16_t)bf16_rne(v[0]));
    } else {
        if (n == 4) {
            st_word<kNT>(reinterpret_cast<u32x2*>(p),
                         u32x2{bf16_pack(v[0], v[1]), bf16_pack(v[2], v[3])});
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (j < n) st_word<kNT>(p + j, (uint16_t)bf16_rne(v[j]));
        }
    }
}

// One piece of the lane-form Adam update: this lane's kE elements at flat index i (the first
// n of them stored: a tensor's last piece may end inside the lane).
template <typename GradT, bool kMixed, int kE, bool kCopyNT>
__device__ __forceinline__ void adam_piece(const GradT* __restrict__ grad,
                                           float* __restrict__ records, float* __restrict__ master,
                                           uint16_t* __restrict__ param16, const AdamArgs& a,
                                           const Coefs& k, bool use_inv, bool use_clip,
                                           bool decay, uint64_t i, int n) {
    constexpr uint32_t kStateStride = kMixed ? kStrideMixed : kStrideMV;
    const uint64_t s = rec_index(i, kStateStride);
    float* pp = kMixed ? records + s : master + i;
    float* mp = kMixed ? records + s + kRec : records + s;
    float* vp = mp + kRec;
    float g[kE], p[kE], m[kE], v[kE];
    ld_grad_lane<kE>(grad, i, g);
    ld_lane<kE>(pp, p);
    ld_lane<kE>(mp, m);
    ld_lane<kE>(vp, v);
#pragma unroll
    for (int j = 0; j < kE; ++j) adam_elem(p[j], g[j], m[j], v[j], a, k, use_inv, use_clip, decay);
    st_lane<kE>(pp, p, n);
    st_lane<kE>(mp, m, n);
    st_lane<kE>(vp, v, n);
    if (kMixed) st_bf16_lane<kE, kCopyNT>(param16 + i, p, n);
}

// The lane-form Adam update: one block per part of kIt consecutive pieces of kLanes x kE
// elements, r = nparts - 1 - (part0 + blockIdx.x) (the last chunks first, as the norm pass);
// the host splits stores beyond one launch's 2^32 - 1 work-items into launches at increasing
// part0.  With kIt = 2 each lane walks its two pieces in turn (a loop the compiler keeps
// rolled): at GPT-2 774M mixed that measured 1.01x the copy against 0.96-0.98x for one piece
// per block, and halves the grid a skipped step dispatches.  records is the record array's
// base ([master|m|v] in MIXED, [m|v] in FP32), master the contiguous FP32 weights (unused in
// MIXED).  a.st must be valid: its fields are read unconditionally and used as a.flags say.
// The arithmetic is adam_elem's, so every shape gives the same results bit for bit.  kCopyNT: the
// bf16 copy is stored non-temporally (see kCachedCopyElems in ttperf.hip).
template <typename GradT, bool kMixed, int kE, int kLanes, int kIt, bool kCopyNT = true>
__global__ __launch_bounds__(kLanes) void adam_lane_kernel(const GradT* __restrict__ grad,
                                                           float* __restrict__ records,
                                                           float* __restrict__ master,
                                                           uint16_t* __restrict__ param16,
                                                           AdamArgs a, uint64_t part0) {
    constexpr uint32_t kPiece = kLanes * kE;
    constexpr uint32_t kP = lane_parts<kE, kLanes, kIt>();
    const uint64_t r = (uint64_t)a.nchunks * kP - 1 - (part0 + blockIdx.x);
    const Chunk ch = load_chunk(a.chunks, r / kP);
    const DevState* st = a.st;
    // `|` and `&`, not `||` and `&&`: the skip flag and the descriptor are both needed before
    // the first branch, so their loads issue together
    const bool run = ((a.flags & kCheckSkip) == 0) | (st->skip == 0);
    const uint32_t off = (uint32_t)(r % kP) * (kPiece * kIt) + threadIdx.x * kE;
    if (!(run & (off < ch.count))) return;
    const bool dev_bias = a.flags & kDevBias;
    const Coefs k{st->inv_scale, st->clip_coef, dev_bias ? st->bias1 : a.bias1,
                  dev_bias ? st->bias2 : a.bias2};
    const bool use_inv = a.flags & kUseInv, use_clip = a.flags & kUseClip;
    const bool decay = (ch.meta & kChunkDecay) && (a.flags & kWdOn);
    if constexpr (kIt == 1) {
        adam_piece<GradT, kMixed, kE, kCopyNT>(grad, records, master, param16, a, k, use_inv,
                                               use_clip, decay, ch.begin + off,
                                               (int)min(ch.count - off, (uint32_t)kE));
    } else {
#pragma unroll 1
        for (int q = 0; q < kIt; ++q) {
            const uint32_t o = off + q * kPiece;
            if (o >= ch.count) break;
            adam_piece<GradT, kMixed, kE, kCopyNT>(grad, records, master, param16, a, k, use_inv,
                                                   use_clip, decay, ch.begin + o,
                                                   (int)min(ch.count - o, (uint32_t)kE));
        }
    }
}

// ------------------------------------------------------------------------------------
// fused SGD (+ momentum / dampening / nesterov / L2)
// ------------------------------------------------------------------------------------
constexpr uint32_t kMomOn = 64u;
constexpr uint32_t kNesterov = 128u;
constexpr uint32_t kMomStaged = 256u;  // the decisions marked this step's first buffers kMomNew

struct SgdArgs {
    const Chunk* chunks;
    uint32_t nchunks;
    uint32_t flags;
    float lr, mu, omd, wd;
    const uint32_t* mom_init;  // per tensor: its momentum mark (see kMomNew)
    const DevState* st;
};

// whether the chunk's tensor gets its first momentum value in this step
__device__ __forceinline__ bool first_momentum(const SgdArgs& a, const Chunk& ch) {
    return (a.flags & kMomOn) &&
           a.mom_init[ch.meta >> 8] == ((a.flags & kMomStaged) ? kMomNew : 0u);
}

// One element of SGD: grad transforms, L2 decay, momentum / dampening / nesterov, then
// `p - g*lr` rounded after the multiply and after the subtract.
__device__ __forceinline__ void sgd_elem(float& p, float g, float& b, const SgdArgs& a, float inv,
                                         float clip, bool use_inv, bool use_clip, bool decay,
                                         bool mom_on, bool first, bool nesterov) {
    if (use_inv) g = g * inv;
    if (use_clip) g = g * clip;
    if (decay) g = g + a.wd * p;
    if (mom_on) {
        const float bj = first ? g : a.mu * b + a.omd * g;
        b = bj;
        g = nesterov ? g + a.mu * bj : bj;
    }
    const float update = g * a.lr;  // autograd/dynamic/optim.hpp:24
    p = p - update;                 // autograd/dynamic/optim.hpp:25
}

// Flat element i of a master slot with kMStride elements per record: kRec is a contiguous
// master (FP32 mode, and the SGD layout of a MIXED store), kStrideMixed slot 0 of the
// [master|m|v] records.
template <uint32_t kMStride>
__device__ __forceinline__ uint64_t master_index(uint64_t i) {
    if constexpr (kMStride == kRec) return i;
    else return rec_index(i, kMStride);
}

// The four-element SGD update: one block per chunk (grid == nchunks), blocks in reverse chunk
// order, one 4-element vector per lane, for MIXED momentum steps whose gradients fit the
// Infinity Cache (at most 2^17 chunks), at most kUpdBlocksPerCU blocks per CU.  master is
// the master slot base (see master_index); momentum is contiguous.
template <typename GradT, bool kMixed, uint32_t kMStride>
__global__ __launch_bounds__(kUpdBlock) void sgd_kernel(const GradT* __restrict__ grad,
                                                        float* __restrict__ master,
                                                        float* __restrict__ momentum,
                                                        uint16_t* __restrict__ param16,
                                                        SgdArgs a) {
    float inv = 1.0f, clip = 1.0f;
    if (a.st) {
        if ((a.flags & kCheckSkip) && a.st->skip) return;
        inv = a.st->inv_scale;
        clip = a.st->clip_coef;
    }
    const bool use_inv = a.flags & kUseInv, use_clip = a.flags & kUseClip;
    const bool mom_on = a.flags & kMomOn, nesterov = a.flags & kNesterov;
    const Chunk ch = a.chunks[a.nchunks - 1 - blockIdx.x];  // last chunks first (see norm pass)
    const uint32_t off = threadIdx.x * kVec;
    if (off >= ch.count) return;
    const int n = (int)min(ch.count - off, (uint32_t)kVec);
    const bool decay = (ch.meta & kChunkDecay) && (a.flags & kWdOn);
    const bool first = first_momentum(a, ch);
    const uint64_t i = ch.begin + off;
    float* pp = master + master_index<kMStride>(i);
    f32x4 g = ld_grad4(grad, i);
    f32x4 p = ld4(pp);
    f32x4 b = {0.0f, 0.0f, 0.0f, 0.0f};
    if (mom_on && !first) b = ld4(momentum + i);
#pragma unroll
    for (int j = 0; j < kVec; ++j) {
        float pj = p[j], bj = b[j];
        sgd_elem(pj, g[j], bj, a, inv, clip, use_inv, use_clip, decay, mom_on, first, nesterov);
        p[j] = pj;
        b[j] = bj;
    }
    store_vec<kMixed>(pp, mom_on ? momentum + i : nullptr, nullptr, param16, i, p, b, b, n);
}

// One piece of the lane-form SGD update (see adam_piece).
template <typename GradT, bool kMixed, uint32_t kMStride, int kE>
__device__ __forceinline__ void sgd_piece(const GradT* __restrict__ grad,
                                          float* __restrict__ master,
                                          float* __restrict__ momentum,
                                          uint16_t* __restrict__ param16, const SgdArgs& a,
                                          float inv, float clip, bool use_inv, bool use_clip,
                                          bool decay, bool mom_on, bool first, bool nesterov,
                                          uint64_t i, int n) {
    float* pp = master + master_index<kMStride>(i);
    float g[kE], p[kE], bm[kE];
    ld_grad_lane<kE>(grad, i, g);
    ld_lane<kE>(pp, p);
    if (mom_on && !first) {
        ld_lane<kE>(momentum + i, bm);
    } else {
#pragma unroll
        for (int j = 0; j < kE; ++j) bm[j] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < kE; ++j)
        sgd_elem(p[j], g[j], bm[j], a, inv, clip, use_inv, use_clip, decay, mom_on, first,
                 nesterov);
    st_lane<kE>(pp, p, n);
    if (mom_on) st_lane<kE>(momentum + i, bm, n);
    if (kMixed) st_bf16_lane<kE>(param16 + i, p, n);
}

// The lane-form SGD update, launched and shaped as adam_lane_kernel.  master is the master
// slot base (see master_index); momentum is contiguous.  a.st must be valid.
template <typename GradT, bool kMixed, uint32_t kMStride, int kE, int kLanes, int kIt>
__global__ __launch_bounds__(kLanes) void sgd_lane_kernel(const GradT* __restrict__ grad,
                                                          float* __restrict__ master,
                                                          float* __restrict__ momentum,
                                                          uint16_t* __restrict__ param16,
                                                          SgdArgs a, uint64_t part0) {
    constexpr uint32_t kPiece = kLanes * kE;
    constexpr uint32_t kP = lane_parts<kE, kLanes, kIt>();
    const uint64_t r = (uint64_t)a.nchunks * kP - 1 - (part0 + blockIdx.x);
    const Chunk ch = load_chunk(a.chunks, r / kP);
    const DevState* st = a.st;
    const bool run = ((a.flags & kCheckSkip) == 0) | (st->skip == 0);  // see adam_lane_kernel
    const uint32_t off = (uint32_t)(r % kP) * (kPiece * kIt) + threadIdx.x * kE;
    if (!(run & (off < ch.count))) return;
    const bool use_inv = a.flags & kUseInv, use_clip = a.flags & kUseClip;
    const bool mom_on = a.flags & kMomOn, nesterov = a.flags & kNesterov;
    const bool decay = (ch.meta & kChunkDecay) && (a.flags & kWdOn);
    const bool first = first_momentum(a, ch);
    const float inv = st->inv_scale, clip = st->clip_coef;
    if constexpr (kIt == 1) {
        sgd_piece<GradT, kMixed, kMStride, kE>(grad, master, momentum, param16, a, inv, clip,
                                               use_inv, use_clip, decay, mom_on, first, nesterov,
                                               ch.begin + off,
                                               (int)min(ch.count - off, (uint32_t)kE));
    } else {
#pragma unroll 1
        for (int q = 0; q < kIt; ++q) {
            const uint32_t o = off + q * kPiece;
            if (o >= ch.count) break;
            sgd_piece<GradT, kMixed, kMStride, kE>(grad, master, momentum, param16, a, inv, clip,
                                                   use_inv, use_clip, decay, mom_on, first,
                                                   nesterov, ch.begin + o,
                                                   (int)min(ch.count - o, (uint32_t)kE));
        }
    }
}

// ------------------------------------------------------------------------------------
// plain SGD of a TTP_MODE_BF16 store: bf16 weights updated in place, no fp32 state
// ------------------------------------------------------------------------------------
// The value of x rounded to bf16 (round to nearest even; NaN -> the quiet NaN 0x7FC0).
__device__ __forceinline__ float bf16_round(float x) {
    return __uint_as_float(bf16_rne(x) << 16);
}

// One element: the grad transforms, then autograd/dynamic/optim.hpp:24-25 on bf16 tensors,
// each ttnn op's result rounded to bf16: update = multiply(grad, lr), data = subtract(data,
// update).  Product and difference are formed in fp32 and rounded from there.
__device__ __forceinline__ float sgd_bf16_elem(float p, float g, float lr, float inv, float clip,
                                               bool use_inv, bool use_clip) {
    if (use_inv) g = g * inv;
    if (use_clip) g = g * clip;
    const float update = bf16_round(g * lr);  // autograd/dynamic/optim.hpp:24
    return bf16_round(p - update);            // autograd/dynamic/optim.hpp:25
}

// kE (2, 4 or 8) bf16 values at p as fp32: one 4-, 8- or 16-byte word (non-temporal: the
// weights are read once and rewritten)
template <int kE>
__device__ __forceinline__ void ld_bf16_lane(const uint16_t* p, float* out) {
    static_assert(kE == 2 || kE == 4 || kE == 8, "2, 4 or 8 elements per lane");
    if constexpr (kE == 2) {
        const uint32_t w = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p));
        out[0] = bf16_lo(w);
        out[1] = bf16_hi(w);
    } else if constexpr (kE == 4) {
        const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
        out[0] = bf16_lo(w.x);
        out[1] = bf16_hi(w.x);
        out[2] = bf16_lo(w.y);
        out[3] = bf16_hi(w.y);
    } else {
        const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            out[2 * j] = bf16_lo(w[j]);
            out[2 * j + 1] = bf16_hi(w[j]);
        }
    }
}
// kE gradients as fp32 (ordinary loads, as ld_grad_lane)
template <int kE>
__device__ __forceinline__ void ld_grad_bf16_lane(const uint16_t* g, float* out) {
    if constexpr (kE <= 4) {
        ld_grad_lane<kE>(g, 0, out);
    } else {
        const u32x4 w = *reinterpret_cast<const u32x4*>(g);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            out[2 * j] = bf16_lo(w[j]);
            out[2 * j + 1] = bf16_hi(w[j]);
        }
    }
}
// the first n (1..kE) of kE values already rounded to bf16: one word when n == kE
template <int kE>
__device__ __forceinline__ void st_bf16_rounded_lane(uint16_t* p, const float* v, int n) {
    if (n == kE) {
        if constexpr (kE == 2) {
            __builtin_nontemporal_store(bf16_pack(v[0], v[1]), reinterpret_cast<uint32_t*>(p));
        } else if constexpr (kE == 4) {
            __builtin_nontemporal_store(u32x2{bf16_pack(v[0], v[1]), bf16_pack(v[2], v[3])},
                                        reinterpret_cast<u32x2*>(p));
        } else {
            __builtin_nontemporal_store(u32x4{bf16_pack(v[0], v[1]), bf16_pack(v[2], v[3]),
                                              bf16_pack(v[4], v[5]), bf16_pack(v[6], v[7])},
                                        reinterpret_cast<u32x4*>(p));
        }
    } else {
#pragma unroll
        for (int j = 0; j < kE - 1; ++j)
            if (j < n) p[j] = (uint16_t)bf16_rne(v[j]);
    }
}

// The plain SGD update of a BF16 store, launched and shaped as the other lane forms (one
// block per 1/lane_parts of a chunk, the last chunks first): 6 B per element (gradient and
// weight read, weight written).  A lane's kE elements start at a multiple of kE and tensors
// start on 64-element boundaries, so the whole-word loads of a tensor's last lane stay inside
// its footprint; only its first n values are stored.  a.st must be valid.
template <int kE, int kLanes, int kIt>
__global__ __launch_bounds__(kLanes) void sgd_bf16_lane_kernel(const uint16_t* __restrict__ grad,
                                                               uint16_t* __restrict__ param,
                                                               SgdArgs a, uint64_t part0) {
    constexpr uint32_t kPiece = kLanes * kE;
    constexpr uint32_t kP = lane_parts<kE, kLanes, kIt>();
    const uint64_t r = (uint64_t)a.nchunks * kP - 1 - (part0 + blockIdx.x);
    const Chunk ch = load_chunk(a.chunks, r / kP);
    const DevState* st = a.st;
    const bool run = ((a.flags & kCheckSkip) == 0) | (st->skip == 0);  // see adam_lane_kernel
    const uint32_t off = (uint32_t)(r % kP) * (kPiece * kIt) + threadIdx.x * kE;
    if (!(run & (off < ch.count))) return;
    const bool use_inv = a.flags & kUseInv, use_clip = a.flags & kUseClip;
    const float inv = st->inv_scale, clip = st->clip_coef;
#pragma unroll 1
    for (int q = 0; q < kIt; ++q) {
        const uint32_t o = off + q * kPiece;
        if (o >= ch.count) break;
        const uint64_t i = ch.begin + o;
        float g[kE], p[kE];
        ld_grad_bf16_lane<kE>(grad + i, g);
        ld_bf16_lane<kE>(param + i, p);
#pragma unroll
        for (int j = 0; j < kE; ++j)
            p[j] = sgd_bf16_elem(p[j], g[j], a.lr, inv, clip, use_inv, use_clip);
        st_bf16_rounded_lane<kE>(param + i, p, (int)min(ch.count - o, (uint32_t)kE));
    }
}

// ------------------------------------------------------------------------------------
// the whole step of a small tensor set in one launch
// ------------------------------------------------------------------------------------
// One 1024-lane block per chunk, one element per lane.  Every block sums the squares of all the
// set's gradients itself and takes the same decisions, so no block waits for another; the last
// block to finish (see is_last_block) writes the step state, which all blocks have read by then.
// The sum is the norm pass's bit for bit: each tile's four waves, the tile from its waves, then
// the tiles in the order of finalize_block.  A step this small
// is bound by launches and by the chain of round trips in each: at the MLP's 9,610 parameters
// (fp32 AdamW with clipping, four tiles) it took 9.3 us in two launches and takes 5.7.
constexpr int kSmallBlock = 1024;
constexpr uint32_t kSmallTiles = 64;  // at most: one lane of a wave per tile

struct SmallArgs {
    FinalizeArgs fin;
    const Chunk* tiles;
    uint32_t ntiles;          // 0: no norm (step counting only)
    uint32_t n_mom;           // tensors to mark as holding a momentum buffer (0: none)
    uint32_t* mom_init;
    const uint32_t* mom_ids;
    uint32_t* tickets;
};

// Every tile descriptor in one load, a lane each (there are at most 64): a wave reads the ones it
// needs from there.  A kernel's first load: it waits for nothing but the arguments.
__device__ __forceinline__ u32x4 small_descs(const SmallArgs& s) {
    const uint32_t lane = threadIdx.x & 63u;
    return *reinterpret_cast<const u32x4*>(s.tiles + min(lane, max(s.ntiles, 1u) - 1));
}

template <typename GradT>
__device__ __forceinline__ double small_sumsq(const GradT* __restrict__ g, const SmallArgs& s,
                                              const u32x4& desc, float inv, double* lds) {
    typedef GradVec<GradT> GV;
    typedef typename GV::raw R;
    constexpr int E = GV::kElems;
    constexpr uint32_t kTilesAtOnce = kSmallBlock / kBlock;  // four waves a tile
    constexpr int kRound = 2;                                // tiles in flight per wave
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    // Goes to the wave's next tile, from the j-th on, that has elements in the wave's part
    // (uniform; the sums of parts without are 0).  The part moves on with each tile, so that the
    // first parts, all that short tensors have, are spread over the four waves.
    uint32_t j = 0;
    auto next = [&](uint32_t& tile, uint32_t& part, uint32_t& count, uint64_t& begin) {
        for (;; ++j) {
            tile = wave / kWaves + j * kTilesAtOnce;
            part = (wave + j) % kWaves;
            count = 0;
            if (tile >= s.ntiles) return false;
            count = (uint32_t)__builtin_amdgcn_readlane(desc.z, tile);
            if (part * 64 * E < count) break;
            if (lane == 0) lds[tile * kWaves + part] = 0.0;
        }
        begin = (uint32_t)__builtin_amdgcn_readlane(desc.x, tile) |
                ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(desc.y, tile) << 32);
        ++j;
        return true;
    };
    uint32_t tile[kRound], part[kRound], count[kRound];
    uint64_t begin[kRound];
    while (next(tile[0], part[0], count[0], begin[0])) {
        R w[kRound][kNormLoads];
        begin[1] = begin[0];  // no second tile: its loads read this one's start, and count as 0
        next(tile[1], part[1], count[1], begin[1]);
#pragma unroll
        for (int u = 0; u < kRound; ++u) {
#pragma unroll
            for (int l = 0; l < kNormLoads; ++l) {
                // a lane's vector past the count reads the tile's first one, and counts as 0
                const uint32_t off = (uint32_t)(l * kBlock + part[u] * 64 + lane) * E;
                w[u][l] =
                    *reinterpret_cast<const R*>(g + begin[u] + (off < count[u] ? off : 0u));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kRound; ++u) {
            if (!count[u]) break;
            double acc[2] = {0.0, 0.0};  // as norm_partials_kernel
#pragma unroll
            for (int l = 0; l < kNormLoads; ++l) {
                // What is left out here would add zeros, which change no sum.  (All of it for
                // every part, with no branch, took 11.7-13.8 us where this takes 9.5: 60
                // tensors of 300 elements, whose one wave part each is all there is.)
                if ((uint32_t)(l * kBlock + part[u] * 64) * E >= count[u]) break;
                const uint32_t off = (uint32_t)(l * kBlock + part[u] * 64 + lane) * E;
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    const double x = off + j < count[u] ? (double)(GV::at(w[u][l], j) * inv) : 0.0;
                    acc[j & 1] = __builtin_fma(x, x, acc[j & 1]);
                }
            }
            const double sum = wave_sum(acc[0] + acc[1]);
            if (lane == 0) lds[tile[u] * kWaves + part[u]] = sum;
        }
    }
    __syncthreads();
    return wave_sum(lane < s.ntiles ? tile_from_waves(lds, lane) : 0.0);
}

// what a block knows before its update
struct SmallStep {
    DevState s0;
    BiasPair bias;
    double sumsq;
    Decision d;
};
template <typename GradT>
__device__ __forceinline__ SmallStep small_step(const GradT* __restrict__ g, const SmallArgs& s,
                                                const u32x4& desc, double* lds) {
    SmallStep r;
    r.s0 = *s.fin.st;
    r.bias = load_bias(s.fin, r.s0.t);
    r.sumsq = s.ntiles ? small_sumsq(g, s, desc, unscale_factor(s.fin, r.s0.scale), lds) : 0.0;
    r.d = decide(s.fin, r.s0.scale, r.sumsq);
    return r;
}
// after every block's update: the state and the momentum marks, by the last block
__device__ __forceinline__ void small_finish(const SmallArgs& s, const SmallStep& r,
                                             uint32_t* lds_flag) {
    __syncthreads();  // every wave of the block has read the state and its marks
    if (!is_last_block(s.tickets, lds_flag)) return;
    if (threadIdx.x == 0) write_state(s.fin, r.s0, r.bias, r.sumsq, r.d);
    if (!r.d.skip)
        for (uint32_t k = threadIdx.x; k < s.n_mom; k += kSmallBlock) s.mom_init[s.mom_ids[k]] = 1u;
}

template <typename GradT, bool kMixed>
__global__ __launch_bounds__(kSmallBlock) void adam_small_kernel(const GradT* __restrict__ grad,
                                                                 float* __restrict__ records,
                                                                 float* __restrict__ master,
                                                                 uint16_t* __restrict__ param16,
                                                                 AdamArgs a, SmallArgs s) {
    __shared__ double lds[kSmallTiles * kWaves];
    __shared__ uint32_t last;
    const u32x4 desc = small_descs(s);
    const Chunk ch = load_chunk(a.chunks, blockIdx.x);
    const bool live = threadIdx.x < ch.count;
    const uint64_t i = ch.begin + threadIdx.x;
    const uint64_t e = rec_index(i, kMixed ? kStrideMixed : kStrideMV);
    float* pp = kMixed ? records + e : master + i;
    float* mp = kMixed ? records + e + kRec : records + e;
    float g = 0.0f, p = 0.0f, m = 0.0f, v = 0.0f;
    if (live) {  // in flight during the norm
        ld_grad_lane<1>(grad, i, &g);
        p = *pp;
        m = *mp;
        v = mp[kRec];
    }
    const SmallStep r = small_step(grad, s, desc, lds);
    if (live && !r.d.skip) {
        const bool dev_bias = a.flags & kDevBias;
        const Coefs k{r.d.inv, r.d.coef, dev_bias ? r.bias.next1 : a.bias1,
                      dev_bias ? r.bias.next2 : a.bias2};
        adam_elem(p, g, m, v, a, k, a.flags & kUseInv, a.flags & kUseClip,
                  (ch.meta & kChunkDecay) && (a.flags & kWdOn));
        *pp = p;
        *mp = m;
        mp[kRec] = v;
        if (kMixed) param16[i] = (uint16_t)bf16_rne(p);
    }
    small_finish(s, r, &last);
}

template <typename GradT, bool kMixed, uint32_t kMStride>
__global__ __launch_bounds__(kSmallBlock) void sgd_small_kernel(const GradT* __restrict__ grad,
                                                                float* __restrict__ master,
                                                                float* __restrict__ momentum,
                                                                uint16_t* __restrict__ param16,
                                                                SgdArgs a, SmallArgs s) {
    __shared__ double lds[kSmallTiles * kWaves];
    __shared__ uint32_t last;
    const u32x4 desc = small_descs(s);
    const Chunk ch = load_chunk(a.chunks, blockIdx.x);
    const bool live = threadIdx.x < ch.count;
    const bool mom_on = a.flags & kMomOn;
    const bool first = mom_on && a.mom_init[ch.meta >> 8] == 0u;
    const uint64_t i = ch.begin + threadIdx.x;
    float* pp = master + master_index<kMStride>(i);
    float g = 0.0f, p = 0.0f, b = 0.0f;
    if (live) {
        ld_grad_lane<1>(grad, i, &g);
        p = *pp;
        if (mom_on && !first) b = momentum[i];
    }
    const SmallStep r = small_step(grad, s, desc, lds);
    if (live && !r.d.skip) {
        sgd_elem(p, g, b, a, r.d.inv, r.d.coef, a.flags & kUseInv, a.flags & kUseClip,
                 (ch.meta & kChunkDecay) && (a.flags & kWdOn), mom_on, first,
                 a.flags & kNesterov);
        *pp = p;
        if (mom_on) momentum[i] = b;
        if (kMixed) param16[i] = (uint16_t)bf16_rne(p);
    }
    small_finish(s, r, &last);
}

__global__ __launch_bounds__(kSmallBlock) void sgd_bf16_small_kernel(
    const uint16_t* __restrict__ grad, uint16_t* __restrict__ param, SgdArgs a, SmallArgs s) {
    __shared__ double lds[kSmallTiles * kWaves];
    __shared__ uint32_t last;
    const u32x4 desc = small_descs(s);
    const Chunk ch = load_chunk(a.chunks, blockIdx.x);
    const bool live = threadIdx.x < ch.count;
    const uint64_t i = ch.begin + threadIdx.x;
    float g = 0.0f, p = 0.0f;
    if (live) {
        ld_grad_lane<1>(grad, i, &g);
        ld_grad_lane<1>(param, i, &p);
    }
    const SmallStep r = small_step(grad, s, desc, lds);
    if (live && !r.d.skip)
        param[i] = (uint16_t)bf16_rne(sgd_bf16_elem(p, g, a.lr, r.d.inv, r.d.coef,
                                                    a.flags & kUseInv, a.flags & kUseClip));
    small_finish(s, r, &last);
}

// after a momentum step whose decisions did not mark the stepped tensors' buffers: mark them
// (unless skipped)
__global__ __launch_bounds__(kBlock) void mark_mom_init_kernel(const Chunk* chunks, uint32_t n,
                                                               uint32_t* mom_init,
                                                               const DevState* st,
                                                               int check_skip) {
    if (check_skip && st->skip) return;
    for (uint32_t c = blockIdx.x * kBlock + threadIdx.x; c < n; c += gridDim.x * kBlock)
        mom_init[chunks[c].meta >> 8] = 1u;
}

// ------------------------------------------------------------------------------------
// gradient accumulation into the flat grad buffer (the backward side of the store)
// ------------------------------------------------------------------------------------
__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ void from_f32(float x, float* out) { *out = x; }
__device__ __forceinline__ void from_f32(float x, uint16_t* out) { *out = (uint16_t)bf16_rne(x); }

// first: grad = incoming (converted); else grad = grad + incoming (fp32 add, one rounding)
template <typename SrcT, typename GradT>
__global__ __launch_bounds__(kBlock) void accumulate_grad_kernel(GradT* __restrict__ grad,
                                                                 const SrcT* __restrict__ src,
                                                                 uint64_t n, int first) {
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * kBlock) {
        const float in = to_f32(src[i]);
        const float r = first ? in : to_f32(grad[i]) + in;
        from_f32(r, grad + i);
    }
}

// zero the grads of the chunks' tensors (a module's zero_grad): one vector per lane
__device__ __forceinline__ void zero_vec(float* g, uint64_t i, int n) {
    if (n >= kVec) {
        st4(g + i, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
    } else {
        for (int j = 0; j < n; ++j) g[i + j] = 0.0f;
    }
}
__device__ __forceinline__ void zero_vec(uint16_t* g, uint64_t i, int n) {
    if (n >= kVec) {
        __builtin_nontemporal_store(u32x2{0u, 0u}, reinterpret_cast<u32x2*>(g + i));
    } else {
        for (int j = 0; j < n; ++j) g[i + j] = 0;
    }
}

// The same accumulation over one tensor of n elements in 16 KiB norm tiles, one 64-lane block
// per wave-share of a tile (kAccBlocksPerTile blocks per tile), all of a lane's loads of a whole
// tile issued before its arithmetic (the grid-stride kernel above, one element per lane per
// iteration, serves tensors of 2^24 or more tiles only).
// kSums: it also computes the sum of squares of the resulting (stored) gradients, unscaled by
// 1/scale when scaler_on: tile t of the tensor (tiles start at its first element, as the norm
// pass's tiles do) is split over kAccBlocksPerTile one-wave blocks, and each lane takes the
// elements that lane `lane` (0..kBlock-1) of the norm pass takes in that tile (kNormLoads
// vectors of GradVec<GradT>::kElems); the squares go into the two accumulators in the norm
// pass's order, and each wave's total (wave_sum, block_sum's first stage) is stored as that
// tile's partial of that wave.  tile_from_waves then adds a tile's wave partials as block_sum
// does, so the tile sums are bit-identical to norm_partials_kernel's over the same gradients.
// A wave's partial needs no LDS and no barrier (a block reduction lengthened each launch by
// 0.6-2.4 us).  The first wave of tile 0 marks the tensor's partials pending.  The squares come
// from values already in registers, so the sums add no memory traffic.
// Measured on MI355X over GPT-2 124M's seven 25 MB buckets of bf16 gradients (assigned; each
// source written just before its call, as a backward leaves it, or long before): one-wave
// blocks against 256-lane ones 92-101 against 98-108 us with the sums (within 2% without);
// non-temporal source loads against cached ones 83-97 against 94-110 us without the sums
// (added onto the stored gradients: 126 against 132-154 us).  The source is read once.
// kVecSrc: the source is 16-byte aligned and read in non-temporal vectors (else element by
// element).
constexpr uint32_t kAccLanes = 64;
constexpr uint32_t kAccBlocksPerTile = kBlock / kAccLanes;
template <int E, bool kVecSrc>
__device__ __forceinline__ void ld_src(const uint16_t* p, float* out) {
    if constexpr (kVecSrc && E == 8) {
        const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            out[2 * j] = bf16_lo(w[j]);
            out[2 * j + 1] = bf16_hi(w[j]);
        }
    } else if constexpr (kVecSrc && E == 4) {
        const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
        out[0] = bf16_lo(w.x);
        out[1] = bf16_hi(w.x);
        out[2] = bf16_lo(w.y);
        out[3] = bf16_hi(w.y);
    } else {
#pragma unroll
        for (int j = 0; j < E; ++j) out[j] = to_f32(p[j]);
    }
}
template <int E, bool kVecSrc>
__device__ __forceinline__ void ld_src(const float* p, float* out) {
    if constexpr (kVecSrc) {
#pragma unroll
        for (int h = 0; h < E / 4; ++h) {
            const f32x4 w = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p + 4 * h));
#pragma unroll
            for (int j = 0; j < 4; ++j) out[4 * h + j] = w[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < E; ++j) out[j] = p[j];
    }
}

// Tile `tile` of one tensor's gradients (grad, n elements) from src, as the lanes
// wave * 64 .. wave * 64 + 63 of a 256-lane tile: a one-wave block's work in both accumulate
// kernels.  inv: 1/scale for the sums; wave_sums: the tensor's run of the store-wide wave
// partials; pending: its flag, which the first wave of its first tile sets.
template <typename SrcT, typename GradT, bool kVecSrc, bool kSums>
__device__ __forceinline__ void accumulate_tile(GradT* __restrict__ grad,
                                                const SrcT* __restrict__ src, uint64_t n,
                                                int first, float inv, uint32_t tile,
                                                uint32_t wave, double* __restrict__ wave_sums,
                                                uint32_t* __restrict__ pending) {
    const uint32_t lane = wave * kAccLanes + threadIdx.x;  // the lane of a 256-lane tile
    typedef GradVec<GradT> GV;
    typedef typename GV::raw R;
    constexpr int E = GV::kElems;
    constexpr uint32_t kTile = norm_tile_elems<GradT>();
    const uint64_t t0 = (uint64_t)tile * kTile;
    // Elements from this tile's start to the tensor's end; below kTile, the last tile's count.
    // No min() of the two ahead of the branch: hipcc (ROCm 7.2, gfx950) has built such a
    // min as a scalar select at the top of the last-tile branch that read the condition code
    // of another compare (of `first`), so that an assign into a last tile took the whole tile
    // and wrote past the tensor's end (tests/test_isa_cpu.py scans for that form).
    const uint64_t left = n - t0;
    double acc[2] = {0.0, 0.0};
    // the squares of a vector's stored values, in the norm pass's order
    auto add_squares = [&](const float* v, uint32_t nv) {
        if constexpr (kSums) {
#pragma unroll
            for (int j = 0; j < E; ++j) {
                const double x = (uint32_t)j < nv ? (double)(v[j] * inv) : 0.0;
                acc[j & 1] = __builtin_fma(x, x, acc[j & 1]);
            }
        }
    };
    // a whole vector's new values from the incoming ones (and the old gradient vector w),
    // stored as one 16-byte word; v receives the stored values
    auto store_vec = [&](uint64_t i, const float* in, const R& w, float* v) {
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const float r = first ? in[j] : GV::at(w, j) + in[j];
            GradT h;
            from_f32(r, &h);
            v[j] = to_f32(h);
        }
        if constexpr (E == 8) {
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = bf16_pack(v[2 * j], v[2 * j + 1]);
            *reinterpret_cast<u32x4*>(grad + i) = o;
        } else {
            *reinterpret_cast<f32x4*>(grad + i) = f32x4{v[0], v[1], v[2], v[3]};
        }
    };
    if (left >= kTile) {
        // a whole tile: every load of the lane issued before the arithmetic (the scheduling
        // barrier keeps them ahead of it, as in the norm pass: with one vector in flight at a
        // time the call ran at a fraction of the copy rate)
        float in[kNormLoads][E];
        R w[kNormLoads];
#pragma unroll
        for (int l = 0; l < kNormLoads; ++l) {
            const uint64_t i = t0 + (uint32_t)(l * kBlock + lane) * E;
            ld_src<E, kVecSrc>(src + i, in[l]);
            if (!first) w[l] = *reinterpret_cast<const R*>(grad + i);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int l = 0; l < kNormLoads; ++l) {
            float v[E];
            store_vec(t0 + (uint32_t)(l * kBlock + lane) * E, in[l], w[l], v);
            add_squares(v, (uint32_t)E);
        }
    } else {  // a tensor's last tile: the vectors (and elements) below its count
        const uint32_t count = (uint32_t)left;
#pragma unroll
        for (int l = 0; l < kNormLoads; ++l) {
            const uint32_t off = (uint32_t)(l * kBlock + lane) * E;
            const uint32_t nv = off < count ? min(count - off, (uint32_t)E) : 0u;
            if (!nv) continue;
            const uint64_t i = t0 + off;
            float v[E];
            if (nv == (uint32_t)E) {
                float in[E];
                ld_src<E, kVecSrc>(src + i, in);
                R w;
                if (!first) w = *reinterpret_cast<const R*>(grad + i);
                store_vec(i, in, w, v);
            } else {  // the tensor's last, partial vector
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    v[j] = 0.0f;
                    if ((uint32_t)j < nv) {
                        const float x = to_f32(src[i + j]);
                        const float r = first ? x : to_f32(grad[i + j]) + x;
                        GradT h;
                        from_f32(r, &h);
                        grad[i + j] = h;
                        v[j] = to_f32(h);
                    }
                }
            }
            add_squares(v, nv);
        }
    }
    if constexpr (kSums) {
        // each wave's total, the first stage of block_sum, with no LDS or barrier after it
        const double part = wave_sum(acc[0] + acc[1]);
        if (threadIdx.x == 0) wave_sums[(uint64_t)tile * kWaves + wave] = part;
        if (tile == 0 && lane == 0) *pending = 1u;
    }
}

// one tensor per launch, kAccBlocksPerTile one-wave blocks per tile
template <typename SrcT, typename GradT, bool kVecSrc, bool kSums>
__global__ __launch_bounds__(kAccLanes) void accumulate_grad_tiles_kernel(
    GradT* __restrict__ grad, const SrcT* __restrict__ src, uint64_t n, int first,
    const DevState* __restrict__ st, int32_t scaler_on, double* __restrict__ wave_sums,
    uint32_t* __restrict__ pending) {
    const float inv = (kSums && scaler_on) ? (float)(1.0 / (double)st->scale) : 1.0f;
    accumulate_tile<SrcT, GradT, kVecSrc, kSums>(grad, src, n, first, inv,
                                                 blockIdx.x / kAccBlocksPerTile,
                                                 blockIdx.x % kAccBlocksPerTile, wave_sums,
                                                 pending);
}

// Several tensors per launch (a backward's bucket): the table travels in the kernel
// arguments, so a call allocates and copies nothing and can be captured.  Tensor k takes
// tiles [tile_end[k-1], tile_end[k]) of the launch, kAccBlocksPerTile one-wave blocks each;
// its fields as in accumulate_grad_tiles_kernel.
constexpr uint32_t kMultiMax = 64;
struct MultiAccArgs {
    uint32_t n;                      // tensors in the table (each with at least one element)
    uint32_t first[kMultiMax / 32];  // bit k: tensor k has no grad yet (its values assign)
    uint32_t tile_end[kMultiMax];    // tiles of tensors 0..k
    uint32_t tile_base[kMultiMax];   // its first tile in the store-wide wave partials
    uint32_t tensor[kMultiMax];      // its index in the tensor table (its pending flag)
    uint64_t offset[kMultiMax];      // its first element in the flat grad buffer
    uint64_t numel[kMultiMax];
    const void* src[kMultiMax];
};

template <typename SrcT, typename GradT, bool kVecSrc, bool kSums>
__global__ __launch_bounds__(kAccLanes) void accumulate_grads_multi_kernel(
    GradT* __restrict__ grad, const MultiAccArgs a, const DevState* __restrict__ st,
    int32_t scaler_on, double* __restrict__ wave_sums, uint32_t* __restrict__ pending) {
    // the block's tensor: the first k with its tile g < tile_end[k] (uniform in the block)
    const uint32_t g = blockIdx.x / kAccBlocksPerTile;
    uint32_t lo = 0, hi = a.n - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (g < a.tile_end[mid])
            hi = mid;
        else
            lo = mid + 1;
    }
    const uint32_t k = lo;
    const uint32_t tile = g - (k ? a.tile_end[k - 1] : 0u);
    const float inv = (kSums && scaler_on) ? (float)(1.0 / (double)st->scale) : 1.0f;
    accumulate_tile<SrcT, GradT, kVecSrc, kSums>(
        grad + a.offset[k], static_cast<const SrcT*>(a.src[k]), a.numel[k],
        (int)((a.first[k >> 5] >> (k & 31)) & 1u), inv, tile, blockIdx.x % kAccBlocksPerTile,
        wave_sums + (uint64_t)a.tile_base[k] * kWaves, pending + a.tensor[k]);
}

template <typename GradT>
__global__ __launch_bounds__(kUpdBlock) void zero_chunks_kernel(GradT* __restrict__ grad,
                                                                const Chunk* __restrict__ chunks,
                                                                uint32_t nchunks) {
    for (uint32_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const Chunk ch = chunks[c];
        const uint32_t off = threadIdx.x * kVec;
        if (off >= ch.count) continue;
        zero_vec(grad, ch.begin + off, (int)min(ch.count - off, (uint32_t)kVec));
    }
}

// ------------------------------------------------------------------------------------
// small elementwise helpers
// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void fill_zero_kernel(uint32_t* p, uint64_t n_words) {
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n_words;
         i += (uint64_t)gridDim.x * kBlock)
        p[i] = 0u;
}

// The kernels below address a state slot (base, stride) over the flat elements
// [first, first + n); stride == kRec is a contiguous buffer.

// bf16 copy of the master weights: p16[i] = RNE(master[i])
__global__ __launch_bounds__(kBlock) void master_to_bf16_kernel(const float* master,
                                                                uint32_t stride, uint16_t* p16,
                                                                uint64_t first, uint64_t n) {
    for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < n;
         k += (uint64_t)gridDim.x * kBlock) {
        const uint64_t i = first + k;
        p16[i] = (uint16_t)bf16_rne(master[rec_index(i, stride)]);
    }
}

// master[i] = float(p16[i]) (exact widening)
__global__ __launch_bounds__(kBlock) void bf16_to_master_kernel(const uint16_t* p16,
                                                                float* master, uint32_t stride,
                                                                uint64_t first, uint64_t n) {
    for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < n;
         k += (uint64_t)gridDim.x * kBlock) {
        const uint64_t i = first + k;
        master[rec_index(i, stride)] = __uint_as_float((uint32_t)p16[i] << 16);
    }
}

// dst[k] = slot[first + k]: a slot's elements as one contiguous array (downloads, checkpoints).
// One element per lane: for contiguous arrays that are not 16-byte aligned.
__global__ __launch_bounds__(kBlock) void gather_slot_kernel(const float* slot, uint32_t stride,
                                                             uint64_t first, uint64_t n,
                                                             float* dst) {
    for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < n;
         k += (uint64_t)gridDim.x * kBlock)
        dst[k] = slot[rec_index(first + k, stride)];
}

// slot[first + k] = src[k] (0 when src is null); with p16, also p16[first + k] = RNE(value)
// (an upload of MIXED-mode master weights keeps the bf16 copy consistent).  One element per
// lane: for zeros and for contiguous arrays that are not 16-byte aligned.
__global__ __launch_bounds__(kBlock) void scatter_slot_kernel(float* slot, uint32_t stride,
                                                              uint64_t first, uint64_t n,
                                                              const float* src, uint16_t* p16) {
    for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < n;
         k += (uint64_t)gridDim.x * kBlock) {
        const uint64_t i = first + k;
        const float x = src ? src[k] : 0.0f;
        slot[rec_index(i, stride)] = x;
        if (p16) p16[i] = (uint16_t)bf16_rne(x);
    }
}

// The same two conversions with four elements per lane: one 16-byte word of the contiguous
// array (16-byte aligned) and of the slot (`first` is a multiple of kRec, so a lane's four
// elements never straddle a record).  One straight-line 64-lane block per 256 elements, four
// records, block0 on: the shape of the fastest copy here.  Bound by HBM bandwidth, of which the
// slot's 256-byte pieces of 768- or 512-byte records take a little more than a copy's.
// Measured at 124,439,808 elements (two arrays in turn), us, [master|m|v] / [m|v] records:
//   gather               157 / 145  (6.3 / 6.9 TB/s)   one element per lane: 220 / 217
//   scatter              164 / 150                                          219 / 218
//   scatter + bf16 copy  209 / 192                                          266 / 264
// (128 or 256 lanes 163-172, two pieces per block 165-188, two elements per lane 167-209.)
constexpr int kSlotLanes = 64, kSlotElems = 4;
__global__ __launch_bounds__(kSlotLanes) void gather_slot4_kernel(const float* __restrict__ slot,
                                                                  uint32_t stride, uint64_t first,
                                                                  uint64_t n,
                                                                  float* __restrict__ dst,
                                                                  uint64_t block0) {
    const uint64_t k = ((block0 + blockIdx.x) * kSlotLanes + threadIdx.x) * kSlotElems;
    if (k >= n) return;
    float v[kSlotElems];
    ld_lane<kSlotElems>(slot + rec_index(first + k, stride), v);
    st_lane<kSlotElems>(dst + k, v, (int)min(n - k, (uint64_t)kSlotElems));
}

template <bool kCopy16>
__global__ __launch_bounds__(kSlotLanes) void scatter_slot4_kernel(
    float* __restrict__ slot, uint32_t stride, uint64_t first, uint64_t n,
    const float* __restrict__ src, uint16_t* __restrict__ p16, uint64_t block0) {
    const uint64_t k = ((block0 + blockIdx.x) * kSlotLanes + threadIdx.x) * kSlotElems;
    if (k >= n) return;
    const int m = (int)min(n - k, (uint64_t)kSlotElems);
    float v[kSlotElems];
    if (m == kSlotElems) {
        ld_lane<kSlotElems>(src + k, v);
    } else {  // the source ends inside the lane
#pragma unroll
        for (int j = 0; j < kSlotElems; ++j) v[j] = j < m ? src[k + j] : 0.0f;
    }
    st_lane<kSlotElems>(slot + rec_index(first + k, stride), v, m);
    if (kCopy16) st_bf16_lane<kSlotElems>(p16 + first + k, v, m);
}

}  // namespace ttp
