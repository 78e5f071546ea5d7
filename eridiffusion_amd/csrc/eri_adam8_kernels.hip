/*
 * Dispatch of the step to its two kernels, and the smaller kernels around it: state creation,
 * checkpoint quantisation, the gradient-norm pass, the quantisation-error pass, the 32-bit step and the
 * EMA sweep.
 */
#include "eri_adam8_inline.h"

namespace eri {

/* The one case in which the EMA runs inside the step kernel: the prefetching kernel in mode ERI, on bf16
 * parameters (with bf16 or fp32 gradients).  On tables that its eight waves per compute unit go through in a few rounds
 * the plain kernel and the sweep behind it are faster.  us per step and EMA, prefetching kernel | plain kernel and sweep,
 * 256 units, no two launches on the same data:
 *   blocks               1,025        2,560        4,096        8,192       12,288       16,896       74,784
 *   bf16           13.5 | 13.1  23.7 | 21.2  31.5 | 29.9  49.1 | 51.5  68.1 | 74.6   88.9 | 100    354 | 417
 *   fp32 gradients 14.2 | 14.1  25.7 | 23.0  32.3 | 33.4  50.6 | 57.9  75.5 | 86.5    100 | 111    408 | 467
 * With partial blocks the same: 7,680 and 15,360 tensors of 1,501 elements 74 | 83 and 143 | 130, half as many of 3,075
 * elements 57 | 76 and 101 | 117. */
constexpr uint32_t kFusedEmaBlocksPerCu = 24, kFusedEmaBlocksPerCuGradF32 = 14;
bool step_fuses_ema(const TableShape &t, const EriAdam8Hyper &h, uint32_t compute_units) {
    if ((h.flags & ERI_ADAM8_FLAG_EMA) == 0 || !layout_param_bf16(t.layout) || h.mode != ERI_ADAM8_MODE_ERI) return false;
    if (h.flags & (ERI_ADAM8_FLAG_BSEARCH | ERI_ADAM8_FLAG_NO_PIPELINE)) return false;
    if ((h.flags & ERI_ADAM8_FLAG_ONE_WAVE) != 0) return true;
    return (uint64_t)t.units() > (uint64_t)compute_units * (layout_grad_bf16(t.layout) ? kFusedEmaBlocksPerCu : kFusedEmaBlocksPerCuGradF32);
}

/* Whether a table that qualifies for the prefetching kernel is large enough to gain from it, or has its EMA inside that
 * kernel.  A step whose EMA is a sweep of its own runs as it would without one: on the prefetching kernel all the same,
 * mode BNB took 38.1 us for 4,096 bf16 blocks instead of 29.0, and fp32 parameters 39 for 2,816 instead of 31.5. */
static bool prefetch_pays(const TableShape &t, const EriAdam8Hyper &h, uint32_t compute_units) {
    if ((h.flags & ERI_ADAM8_FLAG_ONE_WAVE) != 0 || step_fuses_ema(t, h, compute_units)) return true;
    return !long_tails_weigh(t) && (uint64_t)t.total_blocks > (uint64_t)compute_units * prefetch_blocks_per_cu(h.mode, t.layout);
}

int launch_step(const DevTensor *rows, uint32_t n_rows, const TableShape &t, const EriAdam8Hyper &h, const void *lds_image,
                const float *dev_scale, uint32_t grid, uint32_t wg, uint32_t compute_units, void *stream) {
    const uint32_t total_blocks = t.total_blocks, n_tails = t.n_tails, units = t.units();
    const int layout = t.layout;
    const bool bf16 = layout_param_bf16(layout);
    const bool mixed = layout == kLayoutBF16GradF32; // F32 gradients for BF16 parameters
    const bool gs = (h.flags & ERI_ADAM8_FLAG_GRAD_SCALE) != 0;
    // Four waves share each block where one wave per block would leave the chip idle: tables of few blocks.
    // The flags that name a kernel (cross-checks) keep their meaning; bf16 parameters with fp32 gradients
    // have no binary-search variant of the one-wave kernel and stay on this one for those flags.
    const bool one_wave = (h.flags & ERI_ADAM8_FLAG_ONE_WAVE) != 0;
    const bool kernel_named = (h.flags & (ERI_ADAM8_FLAG_BSEARCH | ERI_ADAM8_FLAG_NO_PIPELINE)) != 0;
    const bool few = (uint64_t)units <= (uint64_t)compute_units * (uint64_t)kSplitBlocksPerCu;
    if ((mixed && (h.flags & ERI_ADAM8_FLAG_BSEARCH) != 0) || (!kernel_named && !one_wave && few)) {
        const bool bnb = h.mode == ERI_ADAM8_MODE_BNB;
        const bool wd_s = bnb ? h.weight_decay != 1.0f : h.weight_decay > 0.0f;
        const bool exact_s = !bf16 || (h.flags & ERI_ADAM8_FLAG_EXACT_PARAM) != 0;
        // Up to four blocks per workgroup at a time (a team of four waves each), but no more than it takes to
        // give every compute unit a workgroup: 512 blocks on 256 units run as 256 workgroups of two teams.
        uint32_t teams = (units + compute_units - 1) / compute_units;
        teams = teams < 1 ? 1 : teams > 4 ? 4 : teams;
        uint32_t need = (units + teams - 1) / teams;
        if (need > compute_units) need = compute_units;
        if (need == 0) need = 1;
        return launch_step_split(layout, h.mode, exact_s, wd_s, gs, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, need,
                                 teams, stream);
    }
    if (mixed) {
        const bool wd_m = h.mode == ERI_ADAM8_MODE_BNB ? h.weight_decay != 1.0f : h.weight_decay > 0.0f;
        if ((h.flags & ERI_ADAM8_FLAG_NO_PIPELINE) == 0 && prefetch_pays(t, h, compute_units))
            return launch_step_pipelined_grad_f32(h.mode, (h.flags & ERI_ADAM8_FLAG_EXACT_PARAM) != 0, wd_m, gs,
                                                  step_fuses_ema(t, h, compute_units), rows, n_rows,
                                                  total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
        return launch_step_plain_grad_f32(h.mode, (h.flags & ERI_ADAM8_FLAG_EXACT_PARAM) != 0, wd_m, gs, rows, n_rows,
                                          total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
    }
    if (h.mode == ERI_ADAM8_MODE_BNB) { // slot table only; the decay is a factor
        const bool wd = h.weight_decay != 1.0f;
        const bool exact = (h.flags & ERI_ADAM8_FLAG_EXACT_PARAM) != 0;
        if (bf16 && !kernel_named && prefetch_pays(t, h, compute_units))
            return launch_step_pipelined(h.mode, exact, wd, gs, false, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
        if (bf16) return launch_step_plain_bf16(h.mode, exact, wd, gs, true, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
        if (!kernel_named && prefetch_pays(t, h, compute_units))
            return launch_step_pipelined_f32(h.mode, wd, gs, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
        return launch_step_plain_f32(h.mode, wd, gs, true, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
    }
    const bool wd = h.weight_decay > 0.0f;
    const bool exact = (h.flags & ERI_ADAM8_FLAG_EXACT_PARAM) != 0;
    const bool keytab = (h.flags & ERI_ADAM8_FLAG_BSEARCH) == 0;
    if (!bf16 && !kernel_named && prefetch_pays(t, h, compute_units))
        return launch_step_pipelined_f32(h.mode, wd, gs, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
    if (!bf16) return launch_step_plain_f32(h.mode, wd, gs, keytab, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
    if (keytab && (h.flags & ERI_ADAM8_FLAG_NO_PIPELINE) == 0 && prefetch_pays(t, h, compute_units))
        return launch_step_pipelined(h.mode, exact, wd, gs, step_fuses_ema(t, h, compute_units), rows, n_rows,
                                     total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
    return launch_step_plain_bf16(h.mode, exact, wd, gs, keytab, rows, n_rows, total_blocks, n_tails, h, lds_image, dev_scale, grid, wg, stream);
}

// ------------------------------------------------------------------------------------------
// state initialisation and blockwise (de)quantisation for checkpoint traffic
// ------------------------------------------------------------------------------------------

__global__ void state_init_kernel(uint8_t *m, uint8_t *v, float *am, float *av, uint64_t numel, uint64_t nblocks) {
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t n = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = tid; i < numel; i += n) {
        m[i] = 127;
        v[i] = 0;
    }
    for (uint64_t b = tid; b < nblocks; b += n) {
        am[b] = 0.0f;
        av[b] = 0.0f;
    }
}

// ------------------------------------------------------------------------------------------
// diagnostics: the memory traffic of one step over bf16 rows and nothing else
// ------------------------------------------------------------------------------------------

/* Every full block of the table is read and written as the step kernel reads and writes it -- the launch shape
 * of the prefetching kernel (one workgroup of 512 threads per compute unit, rounds of blocks by ticket),
 * 128-bit non-temporal loads of parameters and gradients, 64-bit ones of the two code arrays, the two absmax
 * words, all of a block's loads in flight before its first store -- with no arithmetic between load and store.
 * Parameters, codes and absmax are written back with the bits they had (`zero` is 0 at run time, which the
 * compiler cannot know, so neither the loads of the gradients nor the stores fall away).  What this launch takes
 * is what the memory system gives the step's mix of four read and three written streams in the placement at
 * hand. */
constexpr uint32_t kProbeThreads = 512;
__global__ __launch_bounds__(kProbeThreads) void traffic_probe_kernel(const DevTensor *__restrict__ rows, uint32_t n_rows,
                                                            uint32_t total_blocks, uint32_t zero) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t waves_per_wg = blockDim.x / kWave;
    const uint32_t wave_in_wg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const Tickets tickets(rows, total_blocks, waves_per_wg);
    if (blockIdx.x >= tickets.rounds) return;
    const BlockRowMap map(rows, n_rows);
    __shared__ uint32_t coming[2];
    uint32_t ti = 0, t_end = 0;
    DevTensor t;
    uint32_t round = blockIdx.x;
    for (uint32_t slot = 0; round < tickets.rounds; slot ^= 1) {
        uint32_t answer = 0;
        if (threadIdx.x == 0) answer = tickets.ask();
        const uint32_t blk = round * waves_per_wg + wave_in_wg;
        if (blk >= total_blocks) break; // in the last round, which is a workgroup's last
        map.seek(rows, blk, ti, t, t_end);
        const uint32_t lb = blk - t.full_start;
        const size_t e0 = (size_t)lb * kBlock;
        ERI_GLOBAL u32x4 *pp = as_global(reinterpret_cast<u32x4 *>(static_cast<char *>(t.p) + e0 * 2));
        ERI_GLOBAL const u32x4 *gp = as_global(reinterpret_cast<const u32x4 *>(static_cast<const char *>(t.g) + e0 * 2));
        ERI_GLOBAL u32x2 *mp = as_global(reinterpret_cast<u32x2 *>(t.m + e0));
        ERI_GLOBAL u32x2 *vp = as_global(reinterpret_cast<u32x2 *>(t.v + e0));
        u32x4 p[4], g[4];
        u32x2 m[4], v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            p[c] = __builtin_nontemporal_load(&pp[c * 64 + lane]);
            g[c] = __builtin_nontemporal_load(&gp[c * 64 + lane]);
            m[c] = __builtin_nontemporal_load(&mp[c * 64 + lane]);
            v[c] = __builtin_nontemporal_load(&vp[c * 64 + lane]);
        }
        const uint32_t a_m = f2u(as_global(t.absmax_m)[lb]), a_v = f2u(as_global(t.absmax_v)[lb]);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            __builtin_nontemporal_store(p[c] ^ (g[c] & zero), &pp[c * 64 + lane]);
            __builtin_nontemporal_store(m[c] ^ zero, &mp[c * 64 + lane]);
            __builtin_nontemporal_store(v[c] ^ zero, &vp[c * 64 + lane]);
        }
        if (lane == 0) {
            as_global(t.absmax_m)[lb] = u2f(a_m ^ zero);
            as_global(t.absmax_v)[lb] = u2f(a_v ^ zero);
        }
        if (threadIdx.x == 0) coming[slot] = tickets.round_of(answer);
        lds_barrier();
        round = __builtin_amdgcn_readfirstlane(coming[slot]);
    }
}

int launch_traffic_probe(const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t grid, void *stream) {
    hipLaunchKernelGGL(traffic_probe_kernel, dim3(grid), dim3(kProbeThreads), 0, static_cast<hipStream_t>(stream), rows, n_rows,
                       total_blocks, 0u);
    return (int)hipGetLastError();
}

__global__ void fill_zero_kernel(uint4 *p, uint64_t words) {
    const uint64_t n = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += n) p[i] = uint4{0u, 0u, 0u, 0u};
}

int launch_fill_zero(void *p, size_t bytes, void *stream) {
    if (bytes == 0) return 0;
    if ((((uintptr_t)p) | bytes) & 15u) return (int)hipErrorInvalidValue;
    const uint64_t words = bytes / 16;
    uint64_t grid = (words + 255) / 256;
    if (grid > 8192) grid = 8192;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((uint32_t)grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<uint4 *>(p), words);
    return (int)hipGetLastError();
}

int launch_state_init(uint8_t *m, uint8_t *v, float *absmax_m, float *absmax_v, uint64_t numel, void *stream) {
    const uint64_t nblocks = (numel + kBlock - 1) / kBlock;
    uint64_t grid = (numel + 255) / 256;
    if (grid > 8192) grid = 8192;
    hipLaunchKernelGGL(state_init_kernel, dim3((uint32_t)grid), dim3(256), 0, static_cast<hipStream_t>(stream), m,
                       v, absmax_m, absmax_v, numel, nblocks);
    return (int)hipGetLastError();
}

/* Gradients come at new addresses every step, and so do the outputs of named updates.  A copy of the rows from pinned
 * memory, its event and the wait for the copy before cost the host 16 us a step, a launch with the addresses 5.5: 60 named
 * tensors 88 -> 79 us a step.  256 short tensors in a list, clipped, are level at 75: two tables, two such launches. */
struct AddressArgs { RowAddresses row[kAddressRows]; };
struct GradArgs { const void *g[kGradRows]; };
__global__ void set_addresses_kernel(DevTensor *rows, uint32_t n, AddressArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rows[i].p = a.row[i].p;
    rows[i].p_in = a.row[i].p_in;
    rows[i].g = a.row[i].g;
}
__global__ void set_gradients_kernel(DevTensor *rows, uint32_t n, GradArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) rows[i].g = a.g[i];
}

int launch_set_addresses(DevTensor *rows, const RowAddresses *a, uint32_t n, void *stream) {
    for (uint32_t at = 0; at < n; at += kAddressRows) {
        AddressArgs args;
        const uint32_t k = n - at < kAddressRows ? n - at : kAddressRows;
        for (uint32_t i = 0; i < k; ++i) args.row[i] = a[at + i];
        hipLaunchKernelGGL(set_addresses_kernel, dim3((k + kWave - 1) / kWave), dim3(kWave), 0, static_cast<hipStream_t>(stream), rows + at, k, args);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
    }
    return 0;
}

int launch_set_gradients(DevTensor *rows, const void *const *g, uint32_t n, void *stream) {
    for (uint32_t at = 0; at < n; at += kGradRows) {
        GradArgs args;
        const uint32_t k = n - at < kGradRows ? n - at : kGradRows;
        for (uint32_t i = 0; i < k; ++i) args.g[i] = g[at + i];
        hipLaunchKernelGGL(set_gradients_kernel, dim3((k + kWave - 1) / kWave), dim3(kWave), 0, static_cast<hipStream_t>(stream), rows + at, k, args);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
    }
    return 0;
}

/* Checkpoint traffic: fp32 moments to codes and absmax and back.  HBM is the bound, 5 bytes per element (4 of fp32, 1 of
 * code) each way.  One wave takes a 2048-element block: lane l of pass c holds elements c*256 + 4l .. +3, which is one
 * 128-bit access of fp32 and one 32-bit access of codes per lane, both contiguous over the wave.
 * All moments of a call are one launch, their rows in its arguments, a workgroup per four blocks: the hardware starts these
 * in the order of the list, which keeps the reads and writes of the launch close together.  How close is a matter of how
 * many run at once, which the LDS they ask for sets: 28,000 bytes beside their tables leave four and five to a unit.
 * us, quantise and dequantise, both moments; a launch per tensor with a persistent grid | one launch, no LDS beside the
 * tables | 28,000 bytes | 60,000:
 *   24 tensors, 340 M parameters   683 + 660 | 570 + 643 | 529 + 600 (6.4 and 5.7 TB/s) | 682 + 656
 *   30 tensors of a rank-128 adapter, 27 M   175 + 119 |  48 +  49 |  49 +  48 |  65 +  50
 *   20 tensors of a rank-16 adapter, 2.3 M    97 +  99 |  12 +  13 |  12 +  13 |  13 +  12 */
constexpr uint32_t kMomentThreads = 256;
constexpr uint32_t kMomentLds = 28000;
/* One moment as a launch carries it. */
struct MomentRow {
    float *x;
    uint8_t *codes;
    float *absmax;
    uint64_t numel;
    uint32_t first_wg; // of the launch's workgroups, the first that takes this row
    uint32_t is_signed;
};
constexpr uint32_t kMomentRows = 96; // 3.8 KB of arguments
struct MomentRows {
    MomentRow row[kMomentRows];
    uint32_t n;
};

/* Pass c of a block of n elements: whole = this lane's four elements exist, else the ones below n - o do. */
template <bool VEC>
__device__ __forceinline__ f32x4 moment_load(const float *x, uint32_t o, uint32_t n) {
    f32x4 r = {0.0f, 0.0f, 0.0f, 0.0f};
    if (VEC && o + 4 <= n) return __builtin_nontemporal_load(as_global(reinterpret_cast<const f32x4 *>(x + o)));
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (o + k < n) r[k] = as_global(x)[o + k];
    return r;
}

template <bool SIGNED>
__device__ __forceinline__ uint32_t small_code(float xs, uint32_t half, const unsigned char *lo, const float *mid) {
    const uint32_t base = lo[SIGNED ? half >> kSKeyDrop : (half & 0x7fffu) >> kUKeyDrop];
    return base + (xs > mid[base] ? 1u : 0u);
}

template <bool VEC, bool SIGNED>
__device__ __forceinline__ void quantize_block(const f32x4 (&v)[8], uint8_t *codes, float *absmax, uint32_t n, uint32_t lane,
                                               const unsigned char *lo, const float *mid) {
    float a = 0.0f;
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c)
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) a = fmaxf(a, __builtin_fabsf(v[c][k]));
    a = wave_max(a);
    const BlockDiv d(a, kKeyScale, kKeyScaleInv);
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        const uint32_t o = c * 256 + lane * 4;
        float q[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            q[k] = d.fast ? d.div_fast(v[c][k]) : d.div_slow(v[c][k]);
            if (!SIGNED) q[k] = fmaxf(q[k], 0.0f); // the unsigned map answers code 0 below zero and for NaN
        }
        const uint32_t h01 = half_key2(q[0], q[1]), h23 = half_key2(q[2], q[3]);
        const uint32_t c0 = small_code<SIGNED>(q[0], h01 & 0xffffu, lo, mid), c1 = small_code<SIGNED>(q[1], h01 >> 16, lo, mid);
        const uint32_t c2 = small_code<SIGNED>(q[2], h23 & 0xffffu, lo, mid), c3 = small_code<SIGNED>(q[3], h23 >> 16, lo, mid);
        const uint32_t w = c0 | (c1 << 8) | (c2 << 16) | (c3 << 24);
        if (VEC && o + 4 <= n) {
            __builtin_nontemporal_store(w, as_global(reinterpret_cast<uint32_t *>(codes + o)));
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if (o + k < n) as_global(codes)[o + k] = (uint8_t)(w >> (8 * k));
        }
    }
    if (lane == 0) *as_global(absmax) = a;
}

/* The row of this workgroup and the block of this wave in it. */
struct MomentBlock {
    MomentRow row;
    uint64_t block;
    size_t e0;
    uint32_t n; // elements of the block, 0 past the row's last
    __device__ __forceinline__ explicit MomentBlock(const MomentRows &rows) {
        uint32_t lo = 0, hi = rows.n; // row[lo].first_wg <= blockIdx.x
        while (hi - lo > 1) {
            const uint32_t at = (lo + hi) >> 1;
            if (rows.row[at].first_wg <= blockIdx.x) lo = at; else hi = at;
        }
        row = rows.row[lo];
        block = (uint64_t)(blockIdx.x - row.first_wg) * (kMomentThreads / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
        e0 = block * kBlock;
        n = e0 >= row.numel ? 0u : row.numel - e0 < kBlock ? (uint32_t)(row.numel - e0) : kBlock;
    }
};

template <bool VEC>
__global__ __launch_bounds__(kMomentThreads) void quantize_kernel(MomentRows rows, const unsigned char *__restrict__ image) {
    __shared__ float mid[256];
    __shared__ uint4 lo_words[kSKeyCount / 16]; // bytes, staged in 16-byte words and aligned for them
    const unsigned char *lo = reinterpret_cast<const unsigned char *>(lo_words);
    static_assert(kSKeyCount == kUKeyCount && kSKeyCount == 16 * kMomentThreads, "one 16-byte word per thread");
    const MomentBlock b(rows);
    const uint32_t lane = threadIdx.x & (kWave - 1);
    f32x4 v[8];
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) v[c] = moment_load<VEC>(b.row.x + b.e0, c * 256 + lane * 4, b.n);
    const bool is_signed = b.row.is_signed != 0;
    mid[threadIdx.x] = reinterpret_cast<const float *>(image + (is_signed ? kSmallMidS : kSmallMidU))[threadIdx.x];
    lo_words[threadIdx.x] = reinterpret_cast<const uint4 *>(image + (is_signed ? kSmallLoS : kSmallLoU))[threadIdx.x];
    __syncthreads();
    if (b.n == 0) return;
    if (is_signed) quantize_block<VEC, true>(v, b.row.codes + b.e0, b.row.absmax + b.block, b.n, lane, lo, mid);
    else quantize_block<VEC, false>(v, b.row.codes + b.e0, b.row.absmax + b.block, b.n, lane, lo, mid);
}

template <bool VEC>
__global__ __launch_bounds__(kMomentThreads) void dequantize_kernel(MomentRows rows, const unsigned char *__restrict__ image) {
    __shared__ float map[256];
    const MomentBlock b(rows);
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint8_t *codes = b.row.codes + b.e0;
    uint32_t w[8];
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        const uint32_t o = c * 256 + lane * 4;
        w[c] = 0;
        if (VEC && o + 4 <= b.n) {
            w[c] = __builtin_nontemporal_load(as_global(reinterpret_cast<const uint32_t *>(codes + o)));
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if (o + k < b.n) w[c] |= (uint32_t)as_global(codes)[o + k] << (8 * k);
        }
    }
    map[threadIdx.x] = reinterpret_cast<const float *>(image + (b.row.is_signed ? kSmallMapS : kSmallMapU))[threadIdx.x];
    __syncthreads();
    if (b.n == 0) return;
    const float a = as_global(b.row.absmax)[b.block];
    float *out = b.row.x + b.e0;
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        const uint32_t o = c * 256 + lane * 4;
        const f32x4 r = {map[w[c] & 0xffu] * a, map[(w[c] >> 8) & 0xffu] * a, map[(w[c] >> 16) & 0xffu] * a, map[w[c] >> 24] * a};
        if (VEC && o + 4 <= b.n) {
            __builtin_nontemporal_store(r, as_global(reinterpret_cast<f32x4 *>(out + o)));
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if (o + k < b.n) as_global(out)[o + k] = r[k];
        }
    }
}

/* Whole words need fp32 pointers on 16 bytes and code pointers on 4 (the optimizers' states and every allocator's
 * buffers are); moments at other addresses take the same kernels element by element, in launches of their own: 24 tensors
 * of 340 M parameters loaded with one of them at an odd address 925 -> 578 us, all aligned 566. */
static bool moment_aligned(const Moment &m) { return ((uintptr_t)m.x & 15u) == 0 && ((uintptr_t)m.codes & 3u) == 0; }

/* Rows as far as they fit one launch's arguments and grid, then the rest. */
static int launch_moments(bool quantize, const Moment *moments, uint32_t n, const void *small_image, hipStream_t s) {
    constexpr uint64_t kWgBlocks = kMomentThreads / kWave, kMaxWgs = 0x7fffffffu / kMomentThreads;
    const unsigned char *image = static_cast<const unsigned char *>(small_image);
    for (const bool vec : {true, false}) {
        uint32_t i = 0;
        while (i < n) {
            MomentRows rows;
            rows.n = 0;
            uint64_t wgs = 0;
            for (; i < n && rows.n < kMomentRows; ++i) {
                if (moment_aligned(moments[i]) != vec) continue;
                const uint64_t need = ((moments[i].numel + kBlock - 1) / kBlock + kWgBlocks - 1) / kWgBlocks;
                if (wgs + need > kMaxWgs) {
                    if (rows.n == 0) return (int)hipErrorInvalidValue; // one moment of 2^36 elements and more
                    break;
                }
                rows.row[rows.n++] = {moments[i].x, moments[i].codes, moments[i].absmax, moments[i].numel, (uint32_t)wgs, moments[i].is_signed ? 1u : 0u};
                wgs += need;
            }
            if (rows.n == 0) break;
            const auto k = quantize ? (vec ? quantize_kernel<true> : quantize_kernel<false>) : (vec ? dequantize_kernel<true> : dequantize_kernel<false>);
            hipLaunchKernelGGL(k, dim3((uint32_t)wgs), dim3(kMomentThreads), kMomentLds, s, rows, image);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return (int)e;
        }
    }
    return 0;
}

int launch_dequantize(const Moment *moments, uint32_t n, const void *small_image, void *stream) {
    return launch_moments(false, moments, n, small_image, static_cast<hipStream_t>(stream));
}

int launch_quantize(const Moment *moments, uint32_t n, const void *small_image, void *stream) {
    return launch_moments(true, moments, n, small_image, static_cast<hipStream_t>(stream));
}

// ------------------------------------------------------------------------------------------
// global gradient norm over the launch table (the trainers' clip_gradients,
// src/trainers/pipeline_flux_lora_sequential.rs:1198-1213,1939-1950), without a host round trip:
// pass 1 forms one fp32 sum of squares per block and adds a workgroup's blocks in f64, pass 2 adds the workgroups'
// partials and writes the norm and the clip factor to device memory, where the step kernel reads it.
// ------------------------------------------------------------------------------------------

/* 1.0 for NaN and +-infinity, else 0.0 */
__device__ __forceinline__ float not_finite(float x) { return (__builtin_fabsf(x) <= 3.4028234e38f) ? 0.0f : 1.0f; }

__device__ __forceinline__ float wave_sum(float x) {
    // fixed reduction tree, so the result does not depend on scheduling
    x += dpp_mov<0xB1, 0xf>(x);
    x += dpp_mov<0x4E, 0xf>(x);
    x += dpp_mov<0x141, 0xf>(x);
    x += dpp_mov<0x140, 0xf>(x); // every lane: its row's sum
    float r = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(x), 15));
    r += u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(x), 31));
    r += u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(x), 47));
    r += u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(x), 63));
    return r;
}

__device__ __forceinline__ double wave_sum_f64(double x) {
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

/* One wave's blocks of one group of rows: its partial last blocks, then its full ones from the last to the first, one
 * block's loads ahead.  The order of the additions within a block is part of the result's bits: a lane adds groups of
 * eight of a full block and every 64th element of a partial one. */
template <bool BF16>
__device__ __forceinline__ void grad_sumsq_walk(const NormGroup &g, uint32_t wg, uint32_t wave_in_wg, uint32_t lane,
                                                double &total, double &bad) {
    const BlockRowMap map(g.rows, g.n_rows);
    // dealt from the group's last wave backwards: the waves that have a block less, or none
    const uint32_t waves = g.wgs * kNormWaves;
    for (uint32_t i = waves - 1 - (wg * kNormWaves + wave_in_wg); i < g.n_tails; i += waves) {
        const DevTensor &t = g.rows[map.tail_row(g.total_blocks, i)];
        const uint32_t n = (uint32_t)(t.numel % kBlock);
        const size_t e0 = (size_t)(t.numel / kBlock) * kBlock;
        const void *tail_g = t.g;
        float acc = 0.0f, nf = 0.0f;
        for (uint32_t c = 0; c < n; c += 8 * kWave) { // eight loads in flight
            float x[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                const uint32_t e = c + k * kWave + lane;
                x[k] = e < n ? load1<BF16>(tail_g, e0 + e) : 0.0f;
            }
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                acc += x[k] * x[k];
                nf += not_finite(x[k]);
            }
        }
        total += (double)wave_sum(acc);
        bad += (double)wave_sum(nf);
    }
    const uint32_t per_chunk = (g.total_blocks + g.chunks - 1) / g.chunks;
    const uint32_t lo = (wg % g.chunks) * per_chunk;
    const uint32_t end = lo + per_chunk < g.total_blocks ? lo + per_chunk : g.total_blocks;
    const uint32_t stride = (g.wgs / g.chunks) * kNormWaves;
    const uint32_t first = lo + (wg / g.chunks) * kNormWaves + wave_in_wg;
    if (first >= end) return;
    uint32_t left = (end - first + stride - 1) / stride; // blocks of this wave, counted down
    uint32_t unit = first + (left - 1) * stride;
    // full blocks [row_start, row_start + row_blocks) belong to the row at hand, whose gradients start at row_g
    uint32_t row_start = 0, row_blocks = 0;
    const char *row_g = nullptr;
    Raw8<BF16> raw[4];
    auto request = [&](uint32_t u) {
        if (u - row_start >= row_blocks) {
            const DevTensor &t = g.rows[map.row_of[u]];
            row_g = static_cast<const char *>(t.g);
            row_start = t.full_start;
            row_blocks = (uint32_t)(t.numel / kBlock);
        }
        const char *base = row_g + (size_t)(u - row_start) * kBlock * (BF16 ? 2 : 4);
#pragma unroll
        for (int c = 0; c < 4; ++c) raw[c].load(base, c * 512 + lane * 8);
    };
    request(unit);
    while (true) {
        Raw8<BF16> cur[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) cur[c] = raw[c];
        const bool more = left > 1;
        if (more) {
            unit -= stride;
            request(unit);
        }
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float x[8];
            cur[c].unpack(x);
#pragma unroll
            for (int k = 0; k < 8; ++k) acc += x[k] * x[k];
        }
        const float block_sum = wave_sum(acc);
        total += (double)block_sum;
        if (not_finite(block_sum) != 0.0f) { // rare: count the NaN / infinite elements of this block
            float nf = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float x[8];
                cur[c].unpack(x);
#pragma unroll
                for (int k = 0; k < 8; ++k) nf += not_finite(x[k]);
            }
            bad += (double)wave_sum(nf);
        }
        if (!more) break;
        --left;
    }
}

/* All groups of rows of a pass in one launch: workgroups [first_wg, first_wg + wgs) take a group.  Reading the
 * gradients once is the bound (6.2 TB/s on 10.3 GB); on the tables of an adapter the launches count as much, so there
 * is one whatever the tables hold.  Measured, this pass and the one behind it, before (a launch per group, a pair per
 * wave, partial blocks one load at a time) and after:
 *   256 short tensors in two tables  5.4 + 5.4 + 3.1 -> 5.8 + 2.6 us
 * and both kernels together, over the same arrays:
 *   608 tensors, 306 MB of bf16      52.3 -> 49.9 us, and with the clipped step behind it 334.6 -> 331.5 (it starts on
 *                                    gradients that the last-level cache still holds: the walk goes backwards)
 *   608 tensors, 1.23 GB of bf16     187.8 -> 186.1 us
 *   1,680 tensors, 10.3 GB of fp32   1,721 -> 1,680 us
 * A pass over gradients of one dtype has an instantiation of its own: beside the fp32 walk the bf16 one took 75
 * registers for 57, six waves per SIMD for eight, and 197.6 us on those 1.23 GB. */
enum NormDtypes { kNormF32, kNormBF16, kNormBoth };
template <NormDtypes GRADS>
__global__ __launch_bounds__(kNormWaves * kWave) void grad_sumsq_kernel(NormGroups groups, double *__restrict__ partial) {
    __shared__ double sums[kNormWaves][2];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave_in_wg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    uint32_t gi = 0;
    while (gi + 1 < groups.n && blockIdx.x >= groups.g[gi + 1].first_wg) ++gi;
    const NormGroup &g = groups.g[gi];
    double total = 0.0, bad = 0.0;
    if (GRADS == kNormBF16 || (GRADS == kNormBoth && g.grad_bf16 != 0)) grad_sumsq_walk<true>(g, blockIdx.x - g.first_wg, wave_in_wg, lane, total, bad);
    else grad_sumsq_walk<false>(g, blockIdx.x - g.first_wg, wave_in_wg, lane, total, bad);
    if (lane == 0) {
        sums[wave_in_wg][0] = total;
        sums[wave_in_wg][1] = bad;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double x = 0.0;
        for (uint32_t w = 0; w < kNormWaves; ++w) x += sums[w][threadIdx.x];
        partial[2 * blockIdx.x + threadIdx.x] = x;
    }
}

__global__ __launch_bounds__(1024) void grad_norm_finish_kernel(const double *__restrict__ partial, uint32_t n,
                                                                float max_norm, float denom_eps,
                                                                float *__restrict__ out /* norm, scale, u64 count */) {
    // partial holds, per workgroup of the first pass, the sum of squares and the count of non-finite elements
    __shared__ double sums[16][2];
    double acc = 0.0, bad = 0.0;
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < n; i += 1024) {
        acc += partial[2 * i];
        bad += partial[2 * i + 1];
    }
    acc = wave_sum_f64(acc);
    bad = wave_sum_f64(bad);
    if (threadIdx.x % kWave == 0) {
        sums[threadIdx.x / kWave][0] = acc;
        sums[threadIdx.x / kWave][1] = bad;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        acc = bad = 0.0;
        for (int w = 0; w < 16; ++w) {
            acc += sums[w][0];
            bad += sums[w][1];
        }
        const float norm = (float)sqrt(acc);
        float scale = 1.0f;
        // clip only a finite norm above the limit (crates/training/src/optimizer.rs:79-84)
        if (max_norm > 0.0f && norm > max_norm && norm <= 3.4028234e38f) scale = max_norm / (norm + denom_eps);
        out[0] = norm;
        out[1] = scale;
        *reinterpret_cast<unsigned long long *>(out + 2) = (unsigned long long)bad;
    }
}

int launch_grad_sumsq(const NormGroups &groups, double *partial, void *stream) {
    const NormGroup &last = groups.g[groups.n - 1];
    bool f32 = false, bf16 = false;
    for (uint32_t i = 0; i < groups.n; ++i) (groups.g[i].grad_bf16 ? bf16 : f32) = true;
    const auto k = f32 ? (bf16 ? grad_sumsq_kernel<kNormBoth> : grad_sumsq_kernel<kNormF32>) : grad_sumsq_kernel<kNormBF16>;
    hipLaunchKernelGGL(k, dim3(last.first_wg + last.wgs), dim3(kNormWaves * kWave), 0, static_cast<hipStream_t>(stream),
                       groups, partial);
    return (int)hipGetLastError();
}

int launch_grad_norm_finish(const double *partial, uint32_t n, float max_norm, float denom_eps, float *out,
                            void *stream) {
    hipLaunchKernelGGL(grad_norm_finish_kernel, dim3(1), dim3(1024), 0, static_cast<hipStream_t>(stream), partial, n,
                       max_norm, denom_eps, out);
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// quantisation error of the step that is about to run (quantization_stats,
// src/trainers/adam8bit_enhanced.rs:93-100,318-327): a read-only pass that forms the new moments
// exactly as the step will, quantises them, and adds |value - dequantised value| per row in f64.
// Diagnostics, not tuned: element by element, binary search.
// ------------------------------------------------------------------------------------------

template <bool BF16, int MODE, bool WD, bool GS>
__global__ __launch_bounds__(256) void quant_error_kernel(const DevTensor *__restrict__ rows, uint32_t n_rows,
                                                          uint32_t total_blocks, EriAdam8Hyper h_in,
                                                          const float *__restrict__ lds_image,
                                                          const float *__restrict__ dev_scale,
                                                          double *__restrict__ err /* [2 * n_rows] */, bool grad_f32) {
    const StepHyper h = make_step_hyper<MODE>(h_in);
    __shared__ float tab[1024]; // signed map, unsigned map, signed midpoints, unsigned midpoints
    for (uint32_t i = threadIdx.x; i < 1024; i += blockDim.x) tab[i] = lds_image[i];
    __syncthreads();
    const float *map_s = tab, *map_u = tab + 256, *mid_s = tab + 512, *mid_u = tab + 768;
    const float tscale = (GS && dev_scale) ? *dev_scale : 1.0f;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t waves_per_wg = blockDim.x / kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * waves_per_wg + threadIdx.x / kWave);
    const uint32_t stride = gridDim.x * waves_per_wg;
    const BlockDiv dbc1(h.bc1), dbc2(h.bc2);
    // every block of every row, partial ones included: rows are walked block by block
    uint32_t ti = 0;
    const uint32_t all_blocks = total_blocks + n_rows; // full blocks, then one (possibly empty) tail per row
    for (uint32_t w = wave; w < all_blocks; w += stride) {
        uint32_t lb, n;
        if (w < total_blocks) {
            ti = find_row(rows, n_rows, ti, w);
            lb = w - rows[ti].full_start;
            n = kBlock;
        } else {
            ti = w - total_blocks;
            lb = (uint32_t)(rows[ti].numel / kBlock);
            n = (uint32_t)(rows[ti].numel % kBlock);
            if (n == 0) continue;
        }
        const DevTensor t = rows[ti];
        const float gscale = GS ? (h.grad_scale * t.grad_scale) * tscale : 1.0f;
        const size_t e0 = (size_t)lb * kBlock;
        ERI_GLOBAL const uint8_t *mc = as_global(static_cast<const uint8_t *>(t.m));
        ERI_GLOBAL const uint8_t *vc = as_global(static_cast<const uint8_t *>(t.v));
        const float a_m = as_global(t.absmax_m)[lb];
        const float a_v = as_global(t.absmax_v)[lb];
        float lm = 0.0f, lv = 0.0f;
        for (uint32_t i = lane; i < n; i += kWave) {
            const size_t e = e0 + i;
            float m, v, pn;
            uint64_t unused = 0; // the exact chain never sets it
            const float gr = (BF16 && !grad_f32) ? load1<true>(t.g, e) : load1<false>(t.g, e);
            adam_elem<MODE, true, BF16, WD, GS>(load1<BF16>(t.p_in, e), gr, map_s[mc[e]] * a_m,
                                                map_u[vc[e]] * a_v, h, gscale, dbc1, dbc2, m, v, pn, unused);
            lm = fmaxf(lm, __builtin_fabsf(m));
            lv = fmaxf(lv, __builtin_fabsf(v));
        }
        float nam = lm, nav = lv;
        wave_max2(nam, nav);
        const BlockDiv dm(nam), dv(nav);
        double em = 0.0, ev = 0.0;
        for (uint32_t i = lane; i < n; i += kWave) {
            const size_t e = e0 + i;
            float m, v, pn;
            uint64_t unused = 0; // the exact chain never sets it
            const float gr = (BF16 && !grad_f32) ? load1<true>(t.g, e) : load1<false>(t.g, e);
            adam_elem<MODE, true, BF16, WD, GS>(load1<BF16>(t.p_in, e), gr, map_s[mc[e]] * a_m,
                                                map_u[vc[e]] * a_v, h, gscale, dbc1, dbc2, m, v, pn, unused);
            const float qm = map_s[code_bsearch(dm.div_slow(m), mid_s)] * nam;
            const float qv = map_u[code_bsearch(dv.div_slow(v), mid_u)] * nav;
            em += (double)__builtin_fabsf(m - qm);
            ev += (double)__builtin_fabsf(v - qv);
        }
        em = wave_sum_f64(em);
        ev = wave_sum_f64(ev);
        if (lane == 0) {
            atomicAdd(&err[2 * ti], em);
            atomicAdd(&err[2 * ti + 1], ev);
        }
    }
}

__global__ void zero_f64_kernel(double *x, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) x[i] = 0.0;
}

int launch_quant_error(const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, int layout,
                       const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale, double *err,
                       uint32_t grid, void *stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    const float *img = static_cast<const float *>(lds_image);
    hipLaunchKernelGGL(zero_f64_kernel, dim3(64), dim3(256), 0, s, err, 2 * n_rows);
    const bool bf16 = layout_param_bf16(layout), l2 = h.mode == ERI_ADAM8_MODE_L2;
    const bool grad_f32 = !layout_grad_bf16(layout);
    const bool wd = h.weight_decay > 0.0f, gs = (h.flags & ERI_ADAM8_FLAG_GRAD_SCALE) != 0;
#define ERI_QE(B, M, W, G) hipLaunchKernelGGL((quant_error_kernel<B, M, W, G>), dim3(grid), dim3(256), 0, s, rows, n_rows, total_blocks, h, img, dev_scale, err, grad_f32)
#define ERI_QE2(B, M) do { if (wd) { if (gs) ERI_QE(B, M, true, true); else ERI_QE(B, M, true, false); } else { if (gs) ERI_QE(B, M, false, true); else ERI_QE(B, M, false, false); } } while (0)
    if (bf16) { if (l2) ERI_QE2(true, ERI_ADAM8_MODE_L2); else ERI_QE2(true, ERI_ADAM8_MODE_ERI); }
    else { if (l2) ERI_QE2(false, ERI_ADAM8_MODE_L2); else ERI_QE2(false, ERI_ADAM8_MODE_ERI); }
#undef ERI_QE2
#undef ERI_QE
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// plain element-wise sweeps over a row table: 32-bit AdamW and EMA.  HBM-bound: AdamW bf16 22 B/param (read 2+2+4+4,
// write 2+4+4), fp32 28 B/param; EMA 3 x element size.
//
// The persistent kernels run one workgroup of eight waves per compute unit and take rounds of blocks by ticket (Tickets:
// what HBM gives depends on how close together the launch reads and writes).  A lane holds four consecutive elements per
// pass, so that every access of either dtype is whole cache lines over the wave and nothing is read twice: streamed.
// A round is what keeps the counter's rate low and the window narrow, about 200 KB per workgroup.  us over the same arrays
// side by side, 1.31 G parameters: 64 waves per unit on a static walk, eight elements per lane, fp32 in two half-line
// words | by ticket:
//   32-bit step bf16 5,784 | 4,563 (6.3 TB/s), fp32 7,393 | 5,840 (6.3), with masters 7,322 | 5,992
//   EMA bf16 1,470 | 1,217 (6.5), fp32 3,100 | 2,364 (6.7)
// Traffic of the 32-bit step alone by what a round holds, 8 waves: half a block per wave 4,476, a block 4,783, two 4,817.
// Sweeps of few blocks take a quarter block per wave (kSmallSweepBlocksPerCu): the 32-bit step over the 87 tensors of
// 1,280 to 2,560 elements of a small adapter 14.2 -> 4.1 us with a wave per block before; whole-line words there
// (4,678 blocks): bf16 37.6 -> 33.7, with masters 48.3 -> 42.8, EMA fp32 18.9 -> 16.8.
// ------------------------------------------------------------------------------------------

/* crates/common/optim/src/adamw.rs:34-54, one rounded operation per line */
__device__ __forceinline__ void adamw32_elem(float p, float g, float &m, float &v, const EriAdamW32Hyper &h, float omb1,
                                             float omb2, float neg_lr, float &pn) {
    float ms = m * h.beta1;
    float gs = g * omb1;
    m = ms + gs;
    float vs = v * h.beta2;
    float g2 = g * g;
    float g2s = g2 * omb2;
    v = vs + g2s;
    float denom = sqrtf(v) + h.eps;
    float update = m / denom;
    float wd = h.weight_decay != 0.0f ? p * h.weight_decay : 0.0f;
    float total = update + wd;
    float step = total * neg_lr;
    pn = p + step;
}

/* Four consecutive elements of a lane as they come from memory; `count` of them exist. */
template <bool BF16>
struct Raw4;
template <>
struct Raw4<true> {
    u32x2 w;
    template <bool PARTIAL>
    __device__ __forceinline__ void load(const void *base, uint32_t elem, uint32_t count) {
        ERI_GLOBAL const uint16_t *q = as_global(static_cast<const uint16_t *>(base) + elem);
        if (!PARTIAL || count == 4) {
            w = __builtin_nontemporal_load((ERI_GLOBAL const u32x2 *)q);
            return;
        }
        uint32_t x[3] = {0, 0, 0};
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k)
            if (k < count) x[k] = q[k];
        w = u32x2{x[0] | x[1] << 16, x[2]};
    }
    __device__ __forceinline__ f32x4 unpack() const { return f32x4{bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)}; }
    template <bool PARTIAL>
    static __device__ __forceinline__ void store(void *base, uint32_t elem, const f32x4 &v, uint32_t count) {
        ERI_GLOBAL uint16_t *q = as_global(static_cast<uint16_t *>(base) + elem);
        if (!PARTIAL || count == 4) {
            __builtin_nontemporal_store(u32x2{bf16_pair(v.x, v.y), bf16_pair(v.z, v.w)}, (ERI_GLOBAL u32x2 *)q);
            return;
        }
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k)
            if (k < count) q[k] = (uint16_t)bf16_bits(v[k]);
    }
};
template <>
struct Raw4<false> {
    f32x4 w;
    template <bool PARTIAL>
    __device__ __forceinline__ void load(const void *base, uint32_t elem, uint32_t count) {
        ERI_GLOBAL const float *q = as_global(static_cast<const float *>(base) + elem);
        if (!PARTIAL || count == 4) {
            w = __builtin_nontemporal_load((ERI_GLOBAL const f32x4 *)q);
            return;
        }
        w = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k)
            if (k < count) w[k] = q[k];
    }
    __device__ __forceinline__ f32x4 unpack() const { return w; }
    template <bool PARTIAL>
    static __device__ __forceinline__ void store(void *base, uint32_t elem, const f32x4 &v, uint32_t count) {
        ERI_GLOBAL float *q = as_global(static_cast<float *>(base) + elem);
        if (!PARTIAL || count == 4) {
            __builtin_nontemporal_store(v, (ERI_GLOBAL f32x4 *)q);
            return;
        }
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k)
            if (k < count) q[k] = v[k];
    }
};

constexpr uint32_t kSweepThreads = 512;
constexpr uint32_t kPass = 4 * kWave; // elements of a wave's pass
/* Of the four elements of a lane that begin at o, how many exist in a piece of n. */
__device__ __forceinline__ uint32_t lane_count4(uint32_t o, uint32_t n) { return o + 4 <= n ? 4u : o < n ? n - o : 0u; }

/* Up to PASSES * kPass elements of one tensor from e0 on, n of them; PARTIAL: fewer than that.  Requested whole, then
 * worked off, so that the caller can look up its next row in between. */
template <bool BF16, bool MASTER, bool GS, int PASSES, bool PARTIAL>
struct AdamW32Piece {
    Raw4<BF16> pr[PASSES], gr[PASSES];
    Raw4<false> mr[PASSES], vr[PASSES], wr[PASSES];
    __device__ __forceinline__ void request(const ElemRow &t, size_t e0, uint32_t n, uint32_t lane) {
        const char *p = static_cast<const char *>(t.a) + e0 * (BF16 ? 2 : 4), *g = static_cast<const char *>(t.b) + e0 * (BF16 ? 2 : 4);
        const float *m = static_cast<const float *>(t.c) + e0, *v = static_cast<const float *>(t.d) + e0, *w = static_cast<const float *>(t.e) + (MASTER ? e0 : 0);
#pragma unroll
        for (int c = 0; c < PASSES; ++c) {
            const uint32_t o = c * kPass + lane * 4, count = lane_count4(o, n);
            if (MASTER) wr[c].template load<PARTIAL>(w, o, count);
            else pr[c].template load<PARTIAL>(p, o, count);
            gr[c].template load<PARTIAL>(g, o, count);
            mr[c].template load<PARTIAL>(m, o, count);
            vr[c].template load<PARTIAL>(v, o, count);
        }
    }
    /* MASTER: the parameter value comes from, and goes back to, an fp32 master copy; the tensor itself only receives the
     * rounded result (mixed precision, src/kernels/fused_adam.cu:151-193, with the arithmetic of adamw.rs). */
    __device__ __forceinline__ void step(const ElemRow &t, size_t e0, uint32_t n, uint32_t lane, const EriAdamW32Hyper &h, float omb1,
                                         float omb2, float neg_lr, float gscale) {
        char *p = static_cast<char *>(t.a) + e0 * (BF16 ? 2 : 4);
        float *m = static_cast<float *>(t.c) + e0, *v = static_cast<float *>(t.d) + e0, *w = static_cast<float *>(t.e) + (MASTER ? e0 : 0);
#pragma unroll
        for (int c = 0; c < PASSES; ++c) {
            const uint32_t o = c * kPass + lane * 4, count = lane_count4(o, n);
            const f32x4 pv = MASTER ? wr[c].unpack() : pr[c].unpack(), gv = gr[c].unpack();
            f32x4 mv = mr[c].unpack(), vv = vr[c].unpack(), pn;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float a = mv[k], b = vv[k], x;
                adamw32_elem(pv[k], GS ? gv[k] * gscale : gv[k], a, b, h, omb1, omb2, neg_lr, x);
                mv[k] = a;
                vv[k] = b;
                pn[k] = x;
            }
            Raw4<BF16>::template store<PARTIAL>(p, o, pn, count);
            if (MASTER) Raw4<false>::template store<PARTIAL>(w, o, pn, count);
            Raw4<false>::template store<PARTIAL>(m, o, mv, count);
            Raw4<false>::template store<PARTIAL>(v, o, vv, count);
        }
    }
};

/* A workgroup of the small sweeps: one block, partial or not, a quarter of it per wave (nothing crosses lanes here).
 * The list of blocks rides behind the rows, so a wave finds its row with one load instead of a search. */
struct SweepQuarter {
    ElemRow t;
    size_t e0;
    uint32_t n; // elements of the quarter that exist
    __device__ __forceinline__ SweepQuarter(const ElemRow *rows, const SweepUnit &u) : t(rows[u.row]) {
        constexpr uint32_t kQuarter = kBlock / 4;
        const uint32_t from = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * kQuarter;
        const size_t b0 = (size_t)u.block * kBlock;
        const uint32_t here = t.numel - b0 >= kBlock ? kBlock : (uint32_t)(t.numel - b0);
        e0 = b0 + from;
        n = here <= from ? 0u : here - from < kQuarter ? here - from : kQuarter;
    }
    static constexpr int kPasses = kBlock / 4 / kPass;
    __device__ __forceinline__ bool whole() const { return n == kBlock / 4; }
};

template <bool BF16, bool MASTER, bool GS, bool PARTIAL>
__device__ __forceinline__ void adamw32_quarter(const SweepQuarter &q, uint32_t lane, const EriAdamW32Hyper &h, float omb1, float omb2,
                                                float neg_lr, float gscale) {
    AdamW32Piece<BF16, MASTER, GS, SweepQuarter::kPasses, PARTIAL> x;
    x.request(q.t, q.e0, q.n, lane);
    x.step(q.t, q.e0, q.n, lane, h, omb1, omb2, neg_lr, gscale);
}

template <bool BF16, bool GS>
__global__ __launch_bounds__(256) void adamw32_small_kernel(const ElemRow *__restrict__ rows, const SweepUnit *__restrict__ units,
                                                            EriAdamW32Hyper h, float grad_scale,
                                                            const float *__restrict__ dev_scale) {
    const float tscale = (GS && dev_scale) ? *dev_scale : 1.0f;
    const float omb1 = 1.0f - h.beta1, omb2 = 1.0f - h.beta2, neg_lr = -h.lr; // adamw.rs:36,42,53
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const SweepQuarter q(rows, units[blockIdx.x]);
    if (q.n == 0) return;
    const float gscale = GS ? (grad_scale * q.t.scale) * tscale : 1.0f;
    if (q.t.e) {
        if (q.whole()) adamw32_quarter<BF16, true, GS, false>(q, lane, h, omb1, omb2, neg_lr, gscale);
        else adamw32_quarter<BF16, true, GS, true>(q, lane, h, omb1, omb2, neg_lr, gscale);
    } else {
        if (q.whole()) adamw32_quarter<BF16, false, GS, false>(q, lane, h, omb1, omb2, neg_lr, gscale);
        else adamw32_quarter<BF16, false, GS, true>(q, lane, h, omb1, omb2, neg_lr, gscale);
    }
}

/* A wave's way through a list of `units`, SUB of them per wave and round, `per_block` units to a block: at(row, unit,
 * ahead) is called for each with the row that owns its block, and calls ahead() once its loads are on the way, which
 * looks up the row of the unit after it. */
template <uint32_t SUB, uint32_t PER_BLOCK, typename At>
__device__ __forceinline__ void sweep_by_ticket(const ElemRow *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t *coming, At at) {
    const uint32_t units = total_blocks * PER_BLOCK, waves = blockDim.x / kWave;
    const uint32_t wave_in_wg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const Tickets tickets(rows, units, waves * SUB);
    uint32_t round = blockIdx.x;
    if (round >= tickets.rounds) return;
    if (threadIdx.x == 0) coming[0] = tickets.round_of(tickets.ask());
    auto unit_of = [&](uint32_t r, uint32_t sub) { return (r * SUB + sub) * waves + wave_in_wg; };
    uint32_t ti = 0, t_end = 0;
    ElemRow t;
    if (unit_of(round, 0) < units) seek_row(rows, n_rows, unit_of(round, 0) / PER_BLOCK, ti, t, t_end);
    lds_barrier();
    uint32_t next = __builtin_amdgcn_readfirstlane(coming[0]);
    for (uint32_t slot = 1;; slot ^= 1) {
        const bool more = next < tickets.rounds;
        uint32_t answer = 0;
        if (more && threadIdx.x == 0) answer = tickets.ask(); // for the round after next
#pragma unroll
        for (uint32_t sub = 0; sub < SUB; ++sub) {
            const uint32_t unit = unit_of(round, sub);
            if (unit >= units) break; // in the last round
            const uint32_t then = sub + 1 < SUB ? unit + waves : more ? unit_of(next, 0) : units;
            const ElemRow here = t;
            at(here, unit, [&] { if (then < units) seek_row(rows, n_rows, then / PER_BLOCK, ti, t, t_end); });
        }
        if (!more) break;
        if (threadIdx.x == 0) coming[slot] = tickets.round_of(answer);
        lds_barrier();
        round = next;
        next = __builtin_amdgcn_readfirstlane(coming[slot]);
    }
}

template <bool BF16, bool GS>
__global__ __launch_bounds__(kSweepThreads) void adamw32_kernel(const ElemRow *__restrict__ rows, uint32_t n_rows,
                                                                uint32_t total_blocks, EriAdamW32Hyper h, float grad_scale,
                                                                const float *__restrict__ dev_scale) {
    constexpr int kPasses = 4; // half a block per wave
    constexpr uint32_t kPiece = kPasses * kPass;
    __shared__ uint32_t coming[2];
    // the clip factor left on the device by the gradient-norm pass (1.0 when there is none)
    const float tscale = (GS && dev_scale) ? *dev_scale : 1.0f;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const float omb1 = 1.0f - h.beta1, omb2 = 1.0f - h.beta2, neg_lr = -h.lr; // adamw.rs:36,42,53
    auto gscale_of = [&](const ElemRow &t) { return GS ? (grad_scale * t.scale) * tscale : 1.0f; }; // the order of the 8-bit step's factors
    const uint32_t waves = blockDim.x / kWave;
    for (uint32_t i = __builtin_amdgcn_readfirstlane(blockIdx.x * waves + threadIdx.x / kWave); i < 2 * n_rows; i += gridDim.x * waves) {
        const ElemRow t = load_constant(rows + i / 2);
        const uint32_t tail = (uint32_t)(t.numel % kBlock), from = (i & 1) * kPiece;
        if (tail <= from) continue;
        const uint32_t n = tail - from < kPiece ? tail - from : kPiece;
        const size_t e0 = (size_t)(t.numel / kBlock) * kBlock + from;
        if (t.e) {
            AdamW32Piece<BF16, true, GS, kPasses, true> x;
            x.request(t, e0, n, lane);
            x.step(t, e0, n, lane, h, omb1, omb2, neg_lr, gscale_of(t));
        } else {
            AdamW32Piece<BF16, false, GS, kPasses, true> x;
            x.request(t, e0, n, lane);
            x.step(t, e0, n, lane, h, omb1, omb2, neg_lr, gscale_of(t));
        }
    }
    sweep_by_ticket<1, 2>(rows, n_rows, total_blocks, coming, [&](const ElemRow &t, uint32_t unit, auto ahead) {
        const size_t e0 = (size_t)(unit / 2 - t.full_start) * kBlock + (unit & 1) * kPiece;
        if (t.e) {
            AdamW32Piece<BF16, true, GS, kPasses, false> x;
            x.request(t, e0, kPiece, lane);
            ahead();
            x.step(t, e0, kPiece, lane, h, omb1, omb2, neg_lr, gscale_of(t));
        } else {
            AdamW32Piece<BF16, false, GS, kPasses, false> x;
            x.request(t, e0, kPiece, lane);
            ahead();
            x.step(t, e0, kPiece, lane, h, omb1, omb2, neg_lr, gscale_of(t));
        }
    });
}

/* src/trainers/ema_enhanced.rs:91-100 */
__device__ __forceinline__ float ema_elem(float shadow, float p, float decay, float omd) {
    float a = shadow * decay;
    float b = p * omd;
    return a + b;
}

/* Up to PASSES * kPass elements from e0 on, requested whole. */
template <bool BF16, int PASSES, bool PARTIAL>
struct EmaPiece {
    static constexpr int kPasses = PASSES;
    Raw4<BF16> sr[kPasses], pr[kPasses];
    __device__ __forceinline__ void request(const ElemRow &t, size_t e0, uint32_t n, uint32_t lane) {
        const char *s = static_cast<const char *>(t.a) + e0 * (BF16 ? 2 : 4), *p = static_cast<const char *>(t.b) + e0 * (BF16 ? 2 : 4);
#pragma unroll
        for (int c = 0; c < kPasses; ++c) {
            const uint32_t o = c * kPass + lane * 4, count = lane_count4(o, n);
            sr[c].template load<PARTIAL>(s, o, count);
            pr[c].template load<PARTIAL>(p, o, count);
        }
    }
    __device__ __forceinline__ void update(const ElemRow &t, size_t e0, uint32_t n, uint32_t lane, float decay, float omd) {
        char *s = static_cast<char *>(t.a) + e0 * (BF16 ? 2 : 4);
#pragma unroll
        for (int c = 0; c < kPasses; ++c) {
            const uint32_t o = c * kPass + lane * 4;
            const f32x4 sv = sr[c].unpack(), pv = pr[c].unpack();
            f32x4 out;
#pragma unroll
            for (int k = 0; k < 4; ++k) out[k] = ema_elem(sv[k], pv[k], decay, omd);
            Raw4<BF16>::template store<PARTIAL>(s, o, out, lane_count4(o, n));
        }
    }
};

template <bool BF16, bool PARTIAL>
__device__ __forceinline__ void ema_quarter(const SweepQuarter &q, uint32_t lane, float decay, float omd) {
    EmaPiece<BF16, SweepQuarter::kPasses, PARTIAL> x;
    x.request(q.t, q.e0, q.n, lane);
    x.update(q.t, q.e0, q.n, lane, decay, omd);
}

template <bool BF16>
__global__ __launch_bounds__(256) void ema_small_kernel(const ElemRow *__restrict__ rows, const SweepUnit *__restrict__ units,
                                                        float decay) {
    const float omd = 1.0f - decay; // ema_enhanced.rs:96
    const SweepQuarter q(rows, units[blockIdx.x]);
    if (q.n == 0) return;
    if (q.whole()) ema_quarter<BF16, false>(q, threadIdx.x & (kWave - 1), decay, omd);
    else ema_quarter<BF16, true>(q, threadIdx.x & (kWave - 1), decay, omd);
}

template <bool BF16>
__global__ __launch_bounds__(kSweepThreads) void ema_kernel(const ElemRow *__restrict__ rows, uint32_t n_rows,
                                                            uint32_t total_blocks, float decay) {
    __shared__ uint32_t coming[2];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const float omd = 1.0f - decay; // ema_enhanced.rs:96
    const uint32_t waves = blockDim.x / kWave;
    for (uint32_t r = __builtin_amdgcn_readfirstlane(blockIdx.x * waves + threadIdx.x / kWave); r < n_rows; r += gridDim.x * waves) {
        const ElemRow t = load_constant(rows + r);
        const uint32_t n = (uint32_t)(t.numel % kBlock);
        if (n == 0) continue;
        const size_t e0 = (size_t)(t.numel / kBlock) * kBlock;
        EmaPiece<BF16, kBlock / kPass, true> x;
        x.request(t, e0, n, lane);
        x.update(t, e0, n, lane, decay, omd);
    }
    sweep_by_ticket<BF16 ? 2 : 1, 1>(rows, n_rows, total_blocks, coming, [&](const ElemRow &t, uint32_t blk, auto ahead) {
        const size_t e0 = (size_t)(blk - t.full_start) * kBlock;
        EmaPiece<BF16, kBlock / kPass, false> x;
        x.request(t, e0, kBlock, lane);
        ahead();
        x.update(t, e0, kBlock, lane, decay, omd);
    });
}

int launch_adamw32(const ElemRow *rows, uint32_t n_rows, uint32_t total_blocks, const SweepUnit *units, uint32_t n_units,
                   int dtype_tag, const EriAdamW32Hyper &h, bool scaled, float grad_scale, const float *dev_scale, uint32_t grid,
                   void *stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
#define ERI_GO(B, G)                                                                                                     \
    do {                                                                                                                 \
        if (units)                                                                                                       \
            hipLaunchKernelGGL((adamw32_small_kernel<B, G>), dim3(n_units), dim3(256), 0, s, rows, units, h, grad_scale, dev_scale); \
        else                                                                                                             \
            hipLaunchKernelGGL((adamw32_kernel<B, G>), dim3(grid), dim3(kSweepThreads), 0, s, rows, n_rows, total_blocks, h, \
                               grad_scale, dev_scale);                                                                   \
    } while (0)
    if (dtype_tag == ERI_DTYPE_F32) {
        if (scaled) ERI_GO(false, true);
        else ERI_GO(false, false);
    } else {
        if (scaled) ERI_GO(true, true);
        else ERI_GO(true, false);
    }
#undef ERI_GO
    return (int)hipGetLastError();
}

int launch_ema(const ElemRow *rows, uint32_t n_rows, uint32_t total_blocks, const SweepUnit *units, uint32_t n_units,
               int dtype_tag, float decay, uint32_t grid, void *stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (units && dtype_tag == ERI_DTYPE_F32)
        hipLaunchKernelGGL(ema_small_kernel<false>, dim3(n_units), dim3(256), 0, s, rows, units, decay);
    else if (units)
        hipLaunchKernelGGL(ema_small_kernel<true>, dim3(n_units), dim3(256), 0, s, rows, units, decay);
    else if (dtype_tag == ERI_DTYPE_F32)
        hipLaunchKernelGGL(ema_kernel<false>, dim3(grid), dim3(kSweepThreads), 0, s, rows, n_rows, total_blocks, decay);
    else
        hipLaunchKernelGGL(ema_kernel<true>, dim3(grid), dim3(kSweepThreads), 0, s, rows, n_rows, total_blocks, decay);
    return (int)hipGetLastError();
}

} // namespace eri
