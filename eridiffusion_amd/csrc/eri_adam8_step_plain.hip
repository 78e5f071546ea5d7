/*
 * The plain step kernel (one wave per block, no cross-block prefetch): tables of every layout and mode between the
 * four-waves-per-block kernel's (kSplitBlocksPerCu) and the prefetching kernel's (prefetch_blocks_per_cu), and any table
 * with ERI_ADAM8_FLAG_BSEARCH or ERI_ADAM8_FLAG_NO_PIPELINE.  HBM traffic bounds it, with the launch's start and its
 * last round on the smaller tables.  A row's partial last block is one more block of the walk, with the lanes past its
 * end off and one trip less in flight: as a two-sweep chain on one wave each it made 300 odd bf16 tensors with 14 M
 * parameters 32.8 us, 28.3 so; 1,400 LoRA tensors 93.9 -> 92.1 us.  Compiled three times, once per layout of the
 * rows (-DERI_PLAIN_LAYOUT=0: fp32, 1: bf16, 2: bf16 parameters with fp32 gradients), so that they build in parallel.
 */
#include "eri_adam8_inline.h"

#if !defined(ERI_PLAIN_LAYOUT) || ERI_PLAIN_LAYOUT < 0 || ERI_PLAIN_LAYOUT > 2
#error "compile with -DERI_PLAIN_LAYOUT=0, 1 or 2"
#endif

namespace eri {

static_assert(kLayoutF32 == 0 && kLayoutBF16 == 1 && kLayoutBF16GradF32 == 2, "ERI_PLAIN_LAYOUT names a Layout");
constexpr bool kBf16 = ERI_PLAIN_LAYOUT != kLayoutF32;
constexpr bool kGradBf16 = ERI_PLAIN_LAYOUT == kLayoutBF16;

/* Which tables an instantiation is for.  Only the first holds the code for partial blocks: beside it the loop over
 * whole ones took 128 registers and up to 20 bytes of scratch, 109 to 127 and none without (2,816 bf16 blocks 14.1 ->
 * 13.5 us, 15.1 -> 14.2 with fp32 gradients). */
enum Table { kTails, kWhole };

/* Threads per workgroup: sixteen waves per compute unit where the instantiation fits the 128 registers that
 * leaves each lane, twelve (170 registers) where it would spill: the coupled-decay mode with a gradient scale,
 * with fp32 gradients or with the binary search (12-30 spilled registers at sixteen waves).  Instantiations of kWhole
 * use no scratch, kTails of bf16 parameters up to 20 bytes per lane. */
constexpr uint32_t plain_threads(int mode, bool gs, bool keytab, bool gbf16) {
    return (mode == ERI_ADAM8_MODE_L2 && (gs || !keytab || !gbf16)) ? 768 : 1024;
}

template <bool BF16, int MODE, bool EXACT, bool WD, bool GS, bool KEYTAB, bool GBF16, Table TABLE>
__global__ __launch_bounds__(plain_threads(MODE, GS, KEYTAB, GBF16)) void adam8_step_kernel(const DevTensor *__restrict__ rows, uint32_t n_rows,
                                                          uint32_t total_blocks, uint32_t n_tails, EriAdam8Hyper h_in,
                                                          const uint4 *__restrict__ lds_image,
                                                          const float *__restrict__ dev_scale) {
    ERI_LDS_IMAGE;
    __shared__ float decayed[16][2][256]; // per wave: the values its block's state codes stand for, decayed
    const StepHyper h = make_step_hyper<MODE>(h_in);
    // clip factor left on the device by the gradient-norm pass (1.0 when there is none)
    const float tscale = (GS && dev_scale) ? *dev_scale : 1.0f;
    // the binary search needs the maps and midpoints only (4 KB); the slot tables are the other 96 KB
    constexpr uint32_t staged = KEYTAB ? kLdsImageBytes : kOffKeyU;
    stage_begin<staged>(lds_raw, lds_image);
    stage_end();
    const char *base = reinterpret_cast<const char *>(lds_raw);
    Lds L;
    L.map_s = reinterpret_cast<const float *>(base + kOffMapS);
    L.map_u = reinterpret_cast<const float *>(base + kOffMapU);
    L.mid_s = reinterpret_cast<const float *>(base + kOffMidS);
    L.mid_u = reinterpret_cast<const float *>(base + kOffMidU);
    L.key_s = base + kOffKeyS;
    L.key_u = base + kOffKeyU;

    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t waves_per_wg = blockDim.x / kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * waves_per_wg + threadIdx.x / kWave);
    const uint32_t stride = gridDim.x * waves_per_wg;
    const BlockDiv dbc1(h.bc1), dbc2(h.bc2);

    // The blocks, partial last ones behind the full ones: round k gives wave w block k * stride + w, and the blocks
    // left over when the list does not divide (fewer than one per wave) go one to each workgroup in turn -- workgroup
    // i takes left-over blocks i, i + grid, i + 2 grid, ... on its first waves -- so that the short last round runs on
    // every compute unit instead of filling the first few (2-3 % of the launch on tables of 5-20 blocks per wave).
    const uint32_t units = TABLE == kTails ? total_blocks + n_tails : total_blocks;
    const uint32_t wave_in_wg = threadIdx.x / kWave;
    const uint32_t rounds = units / stride;
    const uint32_t left_first = rounds * stride;
    const uint32_t left_mine = wave_in_wg * gridDim.x + blockIdx.x;
    const bool has_left = left_first + left_mine < units;

    // Rows are looked up through ordinary loads.  These wait for the stores of the block before, because one counter holds a
    // wave's loads and stores, and so keep its reads and writes apart: through the scalar cache, 600 LoRA tensors took
    // 28.8 us for 27.4, 1,400 in mode L2 97.0 for 93.5, and tables of few rows the same.
    uint32_t ti = 0, t_end = 0;
    DevTensor t;
    const BlockRowMap map(rows, n_rows);
    const uint32_t trips = rounds + (has_left ? 1u : 0u);
    for (uint32_t k = 0; k < trips; ++k) {
        uint32_t unit = k < rounds ? k * stride + wave : left_first + left_mine;
        unit = __builtin_amdgcn_readfirstlane(unit);
        if (TABLE != kTails || unit < total_blocks) {
            if (unit >= t_end) {
                ti = map.row_of[unit];
                t = rows[ti];
                t_end = t.full_start + (uint32_t)(t.numel / kBlock);
            }
            const float gscale = GS ? (h.grad_scale * t.grad_scale) * tscale : 1.0f;
            full_block<BF16, MODE, EXACT, WD, GS, KEYTAB, GBF16>(t, unit - t.full_start, kBlock, lane, h, gscale, dbc1, dbc2, L,
                                                                 decayed[threadIdx.x / kWave]);
        } else {
            t = rows[map.row_of[unit]];
            const float gscale = GS ? (h.grad_scale * t.grad_scale) * tscale : 1.0f;
            full_block<BF16, MODE, EXACT, WD, GS, KEYTAB, GBF16, true>(t, (uint32_t)(t.numel / kBlock), (uint32_t)(t.numel % kBlock),
                                                                       lane, h, gscale, dbc1, dbc2, L, decayed[threadIdx.x / kWave]);
        }
    }
}

namespace {

template <int MODE, bool EXACT, bool WD, bool GS, bool KEYTAB>
int launch_one(const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h,
               const void *lds_image, const float *dev_scale, uint32_t grid, uint32_t wg, hipStream_t s) {
    auto k = adam8_step_kernel<kBf16, MODE, EXACT, WD, GS, KEYTAB, kGradBf16, kTails>;
    if constexpr (KEYTAB) // the binary search is a cross-check and has the one variant
        if (n_tails == 0) k = adam8_step_kernel<kBf16, MODE, EXACT, WD, GS, KEYTAB, kGradBf16, kWhole>;
    if (wg > plain_threads(MODE, GS, KEYTAB, kGradBf16)) wg = plain_threads(MODE, GS, KEYTAB, kGradBf16);
    // One common window for all dies (a grid-stride walk).
    hipLaunchKernelGGL(k, dim3(grid), dim3(wg), 0, s, rows, n_rows, total_blocks, n_tails, h,
                       static_cast<const uint4 *>(lds_image), dev_scale);
    return (int)hipGetLastError();
}

/* BSEARCH: the layout and mode have the cross-check variants (binary search of the midpoint table); mode BNB and fp32
 * gradients of bf16 parameters have none. */
template <int MODE, bool EXACT, bool BSEARCH>
int launch_flags(bool wd, bool gs, bool keytab, const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails,
                 const EriAdam8Hyper &h, const void *img, const float *dev_scale, uint32_t grid, uint32_t wg, hipStream_t s) {
#define ERI_GO(W, G, K) return launch_one<MODE, EXACT, W, G, K>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s)
    if (BSEARCH && !keytab) {
        if (wd) { if (gs) ERI_GO(true, true, !BSEARCH); ERI_GO(true, false, !BSEARCH); }
        if (gs) ERI_GO(false, true, !BSEARCH);
        ERI_GO(false, false, !BSEARCH);
    }
    if (wd) { if (gs) ERI_GO(true, true, true); ERI_GO(true, false, true); }
    if (gs) ERI_GO(false, true, true);
    ERI_GO(false, false, true);
#undef ERI_GO
}

} // namespace

#define ERI_ARGS wd, gs, keytab, rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, static_cast<hipStream_t>(stream)
#if ERI_PLAIN_LAYOUT == 1
int launch_step_plain_bf16(int mode, bool exact, bool wd, bool gs, bool keytab, const DevTensor *rows,
                           uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *img,
                           const float *dev_scale, uint32_t grid, uint32_t wg, void *stream) {
    if (mode == ERI_ADAM8_MODE_BNB)
        return exact ? launch_flags<ERI_ADAM8_MODE_BNB, true, false>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_BNB, false, false>(ERI_ARGS);
    if (mode == ERI_ADAM8_MODE_L2) return launch_flags<ERI_ADAM8_MODE_L2, true, true>(ERI_ARGS); // always the IEEE chain
    return exact ? launch_flags<ERI_ADAM8_MODE_ERI, true, true>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_ERI, false, true>(ERI_ARGS);
}
#elif ERI_PLAIN_LAYOUT == 2
int launch_step_plain_grad_f32(int mode, bool exact, bool wd, bool gs, const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks,
                               uint32_t n_tails, const EriAdam8Hyper &h, const void *img, const float *dev_scale, uint32_t grid,
                               uint32_t wg, void *stream) {
    constexpr bool keytab = true;
    if (mode == ERI_ADAM8_MODE_BNB)
        return exact ? launch_flags<ERI_ADAM8_MODE_BNB, true, false>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_BNB, false, false>(ERI_ARGS);
    if (mode == ERI_ADAM8_MODE_L2) return launch_flags<ERI_ADAM8_MODE_L2, true, false>(ERI_ARGS);
    return exact ? launch_flags<ERI_ADAM8_MODE_ERI, true, false>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_ERI, false, false>(ERI_ARGS);
}
#else
/* fp32 parameters always take the IEEE square root and division. */
int launch_step_plain_f32(int mode, bool wd, bool gs, bool keytab, const DevTensor *rows, uint32_t n_rows,
                          uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *img, const float *dev_scale,
                          uint32_t grid, uint32_t wg, void *stream) {
    if (mode == ERI_ADAM8_MODE_BNB) return launch_flags<ERI_ADAM8_MODE_BNB, true, false>(ERI_ARGS);
    if (mode == ERI_ADAM8_MODE_L2) return launch_flags<ERI_ADAM8_MODE_L2, true, true>(ERI_ARGS);
    return launch_flags<ERI_ADAM8_MODE_ERI, true, true>(ERI_ARGS);
}
#endif
#undef ERI_ARGS

} // namespace eri
