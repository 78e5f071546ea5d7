/*
 * The step over a table that holds both bf16 and fp32 parameters (norms and embeddings kept in fp32 beside bf16
 * matrices), in one launch: a wave per block as in the plain kernel, over the fp32 blocks and then the bf16 ones of one
 * list.  As a launch per dtype, the second waits for the last wave of the first and stages the table image again, which
 * on the tables of an adapter is up to a third of the time.  Measured, two launches and one, 256 units:
 *   300 bf16 and 100 fp32 tensors of odd sizes, 18 M parameters   28.3 + 15.1 -> 38.2 us
 */
#include "eri_adam8_inline.h"

namespace eri {

/* Sixteen waves per compute unit, twelve in mode L2, whose fp32 chain does not fit the registers of sixteen. */
constexpr uint32_t two_threads(int mode) { return mode == ERI_ADAM8_MODE_L2 ? 768 : 1024; }

template <int MODE, bool EXACT, bool WD, bool GS>
__global__ __launch_bounds__(two_threads(MODE)) void adam8_step_two_kernel(StepGroup f32, StepGroup bf16, EriAdam8Hyper h_in,
                                                                            const uint4 *__restrict__ lds_image,
                                                                            const float *__restrict__ dev_scale) {
    ERI_LDS_IMAGE;
    __shared__ float decayed[16][2][256]; // per wave: the values its block's state codes stand for, decayed
    const StepHyper h = make_step_hyper<MODE>(h_in);
    const float tscale = (GS && dev_scale) ? *dev_scale : 1.0f;
    stage_begin<kLdsImageBytes>(lds_raw, lds_image);
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
    const uint32_t wave_in_wg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t waves_per_wg = blockDim.x / kWave;
    const uint32_t wave = blockIdx.x * waves_per_wg + wave_in_wg;
    const uint32_t stride = gridDim.x * waves_per_wg;
    const BlockDiv dbc1(h.bc1), dbc2(h.bc2);
    float(*const mine)[256] = decayed[wave_in_wg];

    const uint32_t f32_units = f32.total_blocks + f32.n_tails;
    const uint32_t units = f32_units + bf16.total_blocks + bf16.n_tails;
    // the plain kernel's dealing: whole rounds, then the blocks left over one to each workgroup in turn
    const uint32_t rounds = units / stride;
    const uint32_t left = rounds * stride + wave_in_wg * gridDim.x + blockIdx.x;
    const uint32_t trips = rounds + (left < units ? 1u : 0u);
    for (uint32_t k = 0; k < trips; ++k) {
        uint32_t unit = k < rounds ? k * stride + wave : left;
        const bool is_f32 = unit < f32_units;
        const StepGroup &g = is_f32 ? f32 : bf16;
        if (!is_f32) unit -= f32_units;
        // a full block's row or, behind those, the row of a partial one: one list (BlockRowMap)
        const BlockRowMap map(g.rows, g.n_rows);
        const DevTensor t = load_constant(g.rows + load_constant(map.row_of + unit));
        const float gscale = GS ? (h.grad_scale * t.grad_scale) * tscale : 1.0f;
        const bool partial = unit >= g.total_blocks;
        const uint32_t lb = partial ? (uint32_t)(t.numel / kBlock) : unit - t.full_start;
        const uint32_t n = partial ? (uint32_t)(t.numel % kBlock) : kBlock;
        if (is_f32) {
            if (partial) full_block<false, MODE, true, WD, GS, true, false, true>(t, lb, n, lane, h, gscale, dbc1, dbc2, L, mine);
            else full_block<false, MODE, true, WD, GS, true>(t, lb, kBlock, lane, h, gscale, dbc1, dbc2, L, mine);
        } else {
            if (partial) full_block<true, MODE, EXACT, WD, GS, true, true, true>(t, lb, n, lane, h, gscale, dbc1, dbc2, L, mine);
            else full_block<true, MODE, EXACT, WD, GS, true>(t, lb, kBlock, lane, h, gscale, dbc1, dbc2, L, mine);
        }
    }
}

namespace {

template <int MODE, bool EXACT>
int launch_flags(bool wd, bool gs, const StepGroup &f32, const StepGroup &bf16, const EriAdam8Hyper &h, const void *img,
                 const float *dev_scale, uint32_t grid, uint32_t wg, hipStream_t s) {
    if (wg > two_threads(MODE)) wg = two_threads(MODE);
    const auto k = wd ? (gs ? adam8_step_two_kernel<MODE, EXACT, true, true> : adam8_step_two_kernel<MODE, EXACT, true, false>)
                      : (gs ? adam8_step_two_kernel<MODE, EXACT, false, true> : adam8_step_two_kernel<MODE, EXACT, false, false>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(wg), 0, s, f32, bf16, h, static_cast<const uint4 *>(img), dev_scale);
    return (int)hipGetLastError();
}

} // namespace

int launch_step_two(const StepGroup &f32, const StepGroup &bf16, const EriAdam8Hyper &h, const void *img, const float *dev_scale,
                    uint32_t grid, uint32_t wg, void *stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool gs = (h.flags & ERI_ADAM8_FLAG_GRAD_SCALE) != 0;
    const bool exact = (h.flags & ERI_ADAM8_FLAG_EXACT_PARAM) != 0;
    const bool bnb = h.mode == ERI_ADAM8_MODE_BNB;
    const bool wd = bnb ? h.weight_decay != 1.0f : h.weight_decay > 0.0f; // mode BNB carries the factor 1 - lr*wd
#define ERI_ARGS wd, gs, f32, bf16, h, img, dev_scale, grid, wg, s
    if (h.mode == ERI_ADAM8_MODE_L2) return launch_flags<ERI_ADAM8_MODE_L2, true>(ERI_ARGS); // always the IEEE chain's bits
    if (bnb) return exact ? launch_flags<ERI_ADAM8_MODE_BNB, true>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_BNB, false>(ERI_ARGS);
    return exact ? launch_flags<ERI_ADAM8_MODE_ERI, true>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_ERI, false>(ERI_ARGS);
#undef ERI_ARGS
}

} // namespace eri
