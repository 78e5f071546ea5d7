/* The software-pipelined step kernel: the benchmark kernel.  Compiled three times, once per layout of the
 * rows (-DERI_PIPE_LAYOUT=1: bf16 parameters and gradients, 2: bf16 parameters with fp32 gradients, 0: fp32
 * parameters and gradients), so that the three build in parallel. */
#include "eri_adam8_inline.h"

#if !defined(ERI_PIPE_LAYOUT) || ERI_PIPE_LAYOUT < 0 || ERI_PIPE_LAYOUT > 2
#error "compile with -DERI_PIPE_LAYOUT=0, 1 or 2"
#endif

namespace eri {

static_assert(kLayoutF32 == 0 && kLayoutBF16 == 1 && kLayoutBF16GradF32 == 2, "ERI_PIPE_LAYOUT names a Layout");
constexpr bool kParamBf16 = ERI_PIPE_LAYOUT != kLayoutF32;
constexpr bool kGradBf16 = ERI_PIPE_LAYOUT == kLayoutBF16;

// ------------------------------------------------------------------------------------------
// software-pipelined step kernel
//
// Same arithmetic as adam8_step_kernel, but a wave requests its NEXT block quarter by quarter as soon as
// the same quarter of this one has been consumed: the registers of the raw words are free from then on,
// so every load has a whole block's time to arrive and the pipeline costs no copies.
// HBM bounds it, and what HBM gives depends on how close together the launch reads and writes: rounds of
// blocks are handed out by ticket (Tickets), and eight waves per compute unit, two per SIMD with 256
// registers each, are enough to keep the memory busy and few enough for a narrow window.
// us per launch, arrays side by side; twelve waves on a static walk (bf16 gradients; eight for the others)
// | the same by ticket | eight waves by ticket:
//   bf16, 11.9 G parameters                23,506 | 20,236 | 19,225 (6.2 TB/s; six waves 20,265)
//   bf16, 2.57 G                            5,060 |  4,832 |  4,216
//   ... with the EMA                        7,170 |  7,624 |  5,699 (the next block requested quarter by quarter;
//                                                                    5,867 after the update half, as it was)
//   bf16 with fp32 gradients, 2.57 G        5,980 |        |  4,924
//   ... with the EMA                        8,140 |        |  6,627 (6,848 after the update half)
//   fp32, 2.57 G                            8,031 |        |  7,348 (6,785 in whole lines)
// ------------------------------------------------------------------------------------------

constexpr uint32_t kPipeThreads = 512;
#if ERI_PIPE_LAYOUT == 1
#define ERI_PIPE_KERNEL adam8_step_pipelined_kernel
#elif ERI_PIPE_LAYOUT == 2
#define ERI_PIPE_KERNEL adam8_step_pipelined_grad_f32_kernel
#else
#define ERI_PIPE_KERNEL adam8_step_pipelined_f32_kernel
#endif

/* Eight shadow values of a lane: shadow = d*shadow + (1-d)*p', each operation rounded on its own; the store rounds the
 * result to bf16. */
__device__ __forceinline__ void ema_eight(const u32x4 &old, const u32x4 &pnew, float decay, float (&out)[8]) {
    const float omd = 1.0f - decay; // ema_enhanced.rs:96
    Raw8<true> so, pn;
    so.w = old;
    pn.w = pnew;
    float sv[8], pv[8];
    so.unpack(sv);
    pn.unpack(pv);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float a = sv[k] * decay;
        float b = pv[k] * omd;
        out[k] = a + b;
    }
}

/* The shadow of a row's partial last block of n elements.  A lane takes the eight elements that it has just stored as
 * parameters (full_block), so that what it reads back are its own stores: nothing orders them before another lane's
 * loads. */
__device__ __forceinline__ void ema_tail(const DevTensor &t, uint32_t n, uint32_t lane, float decay) {
    const size_t e0 = (size_t)(t.numel / kBlock) * kBlock;
    char *shadow = static_cast<char *>(t.shadow) + e0 * 2;
    const char *p = static_cast<const char *>(t.p) + e0 * 2;
    for (uint32_t o = lane * 8; o < n; o += 8 * kWave) {
        const uint32_t count = lane_count(o, n);
        Raw8<true> so, pn;
        float out[8];
        if (count == 8) {
            so.load(shadow, o);
            pn.load(p, o);
        } else {
            so.load_some(shadow, o, count);
            pn.load_some(p, o, count);
        }
        ema_eight(so.w, pn.w, decay, out);
        if (count == 8) store8<true>(shadow, o, out);
        else store_some<true>(shadow, o, out, count);
    }
}

/* A lane's eight elements of a quarter block (512 elements).  Where everything is bf16 they are consecutive: one 128-bit
 * word each of parameters and gradients, 64 bits of codes.  Beside fp32 they are four of the quarter's first half and four
 * of its second, so that an access of either dtype is whole cache lines over the wave and can be streamed; as two half-line
 * words of eight consecutive fp32 values, every line was asked for twice and had to stay in the caches in between.
 *   fp32, 2.57 G parameters 7,302 -> 6,785 us; bf16 with fp32 gradients 4,979 -> 4,924, with the EMA level */
constexpr bool kHalves = !kGradBf16;
__device__ __forceinline__ u32x4 load_bf16_quarter(const void *block, int c, uint32_t lane) {
    if (kHalves) {
        ERI_GLOBAL const u32x2 *q = as_global(static_cast<const u32x2 *>(block)) + c * 128 + lane;
        const u32x2 a = __builtin_nontemporal_load(q), b = __builtin_nontemporal_load(q + 64);
        return u32x4{a.x, a.y, b.x, b.y};
    }
    return __builtin_nontemporal_load(as_global(static_cast<const u32x4 *>(block)) + c * 64 + lane);
}
__device__ __forceinline__ void store_bf16_quarter(const u32x4 &w, void *block, int c, uint32_t lane) {
    if (kHalves) {
        ERI_GLOBAL u32x2 *q = as_global(static_cast<u32x2 *>(block)) + c * 128 + lane;
        __builtin_nontemporal_store(u32x2{w.x, w.y}, q);
        __builtin_nontemporal_store(u32x2{w.z, w.w}, q + 64);
    } else {
        __builtin_nontemporal_store(w, as_global(static_cast<u32x4 *>(block)) + c * 64 + lane);
    }
}
/* Parameters and gradients by how many words a lane's eight elements take: bf16 one, fp32 two. */
__device__ __forceinline__ void load_quarter(u32x4 (&w)[1], const void *block, int c, uint32_t lane) { w[0] = load_bf16_quarter(block, c, lane); }
__device__ __forceinline__ void load_quarter(u32x4 (&w)[2], const void *block, int c, uint32_t lane) {
    ERI_GLOBAL const u32x4 *q = as_global(static_cast<const u32x4 *>(block)) + c * 128 + lane;
    w[0] = __builtin_nontemporal_load(q);
    w[1] = __builtin_nontemporal_load(q + 64);
}
__device__ __forceinline__ void unpack_quarter(const u32x4 (&w)[1], float (&out)[8]) {
    Raw8<true> r;
    r.w = w[0];
    r.unpack(out);
}
__device__ __forceinline__ void unpack_quarter(const u32x4 (&w)[2], float (&out)[8]) {
    Raw8<false> r;
    r.a = __builtin_bit_cast(f32x4, w[0]);
    r.b = __builtin_bit_cast(f32x4, w[1]);
    r.unpack(out);
}
__device__ __forceinline__ void store_f32_quarter(const float (&v)[8], void *block, int c, uint32_t lane) {
    ERI_GLOBAL f32x4 *q = as_global(static_cast<f32x4 *>(block)) + c * 128 + lane;
    __builtin_nontemporal_store(f32x4{v[0], v[1], v[2], v[3]}, q);
    __builtin_nontemporal_store(f32x4{v[4], v[5], v[6], v[7]}, q + 64);
}
__device__ __forceinline__ u32x2 load_codes_quarter(const uint8_t *block, int c, uint32_t lane) {
    if (kHalves) {
        ERI_GLOBAL const uint32_t *q = as_global(reinterpret_cast<const uint32_t *>(block)) + c * 128 + lane;
        return u32x2{__builtin_nontemporal_load(q), __builtin_nontemporal_load(q + 64)};
    }
    return __builtin_nontemporal_load(as_global(reinterpret_cast<const u32x2 *>(block)) + c * 64 + lane);
}
__device__ __forceinline__ void store_codes_quarter(const u32x2 &w, uint8_t *block, int c, uint32_t lane) {
    if (kHalves) {
        ERI_GLOBAL uint32_t *q = as_global(reinterpret_cast<uint32_t *>(block)) + c * 128 + lane;
        __builtin_nontemporal_store(w.x, q);
        __builtin_nontemporal_store(w.y, q + 64);
    } else {
        __builtin_nontemporal_store(w, as_global(reinterpret_cast<u32x2 *>(block)) + c * 64 + lane);
    }
}

struct RawBlock {
    u32x4 p[4][kParamBf16 ? 1 : 2]; // per quarter block
    u32x4 g[4][kGradBf16 ? 1 : 2];
    u32x2 m[4], v[4];
    float a_m, a_v;
    /* Requests quarter c of block lb; the block's two absmax words ride with quarter 0. */
    __device__ __forceinline__ void issue_quarter(const DevTensor &t, uint32_t lb, int c, uint32_t lane) {
        const size_t e0 = (size_t)lb * kBlock;
        const char *pp = static_cast<const char *>(t.p_in) + e0 * (kParamBf16 ? 2 : 4), *gp = static_cast<const char *>(t.g) + e0 * (kGradBf16 ? 2 : 4);
        load_quarter(p[c], pp, c, lane);
        load_quarter(g[c], gp, c, lane);
        m[c] = load_codes_quarter(t.m + e0, c, lane);
        v[c] = load_codes_quarter(t.v + e0, c, lane);
        if (c == 0) {
            a_m = as_global(t.absmax_m)[lb];
            a_v = as_global(t.absmax_v)[lb];
        }
    }
    __device__ __forceinline__ void issue(const DevTensor &t, uint32_t lb, uint32_t lane) {
#pragma unroll
        for (int c = 0; c < 4; ++c) issue_quarter(t, lb, c, lane);
    }
};

/* EMA: rows that carry a shadow also get shadow = d*shadow + (1-d)*p' (src/trainers/ema_enhanced.rs:91-100),
 * p' being the parameter as it is stored (rounded to bf16). */
template <int MODE, bool EXACT, bool WD, bool GS, bool EMA>
__global__ __launch_bounds__(kPipeThreads) void ERI_PIPE_KERNEL(const DevTensor *__restrict__ rows,
                                                                   uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails,
                                                                   EriAdam8Hyper h_in,
                                                                   const uint4 *__restrict__ lds_image,
                                                                   const float *__restrict__ dev_scale) {
    ERI_LDS_IMAGE;
    const StepHyper h = make_step_hyper<MODE>(h_in);
    // Per wave, the 2 x 256 values a state code of the block at hand can stand for, already multiplied by the
    // block's absmax and by beta: (MAP[c] * absmax) * beta, the first two operations of both moment
    // updates, done once per code (8 per lane) instead of once per element (64 per lane).
    __shared__ float decayed[kPipeThreads / kWave][2][256];
    // clip factor left on the device by the gradient-norm pass (1.0 when there is none)
    const float tscale = (GS && dev_scale) ? *dev_scale : 1.0f;
    const uint32_t waves_per_wg = blockDim.x / kWave;
    const Tickets tickets(rows, total_blocks, waves_per_wg);
    __shared__ uint32_t coming[2];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave_in_wg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const BlockRowMap map(rows, n_rows);
    uint32_t blk = blockIdx.x * waves_per_wg + wave_in_wg;
    stage_begin<kLdsImageBytes>(lds_raw, lds_image);
    if (threadIdx.x == 0 && blockIdx.x < tickets.rounds) coming[0] = tickets.round_of(tickets.ask());
    stage_end();
    const char *base = reinterpret_cast<const char *>(lds_raw);
    Lds L;
    L.map_s = reinterpret_cast<const float *>(base + kOffMapS);
    L.map_u = reinterpret_cast<const float *>(base + kOffMapU);
    L.mid_s = reinterpret_cast<const float *>(base + kOffMidS);
    L.mid_u = reinterpret_cast<const float *>(base + kOffMidU);
    L.key_s = base + kOffKeyS;
    L.key_u = base + kOffKeyU;

    const uint32_t stride = gridDim.x * waves_per_wg;
    const BlockDiv dbc1(h.bc1), dbc2(h.bc2);
    float(*const mine)[256] = decayed[threadIdx.x / kWave];

    // partial last blocks first, handed out from the last wave backwards; their workgroups come to the tickets later
    for (uint32_t i = stride - 1 - blk; i < n_tails; i += stride) {
        const DevTensor t = load_constant(rows + map.tail_row(total_blocks, i));
        const uint32_t n = (uint32_t)(t.numel % kBlock);
        const float gscale = GS ? (h.grad_scale * t.grad_scale) * tscale : 1.0f;
        full_block<kParamBf16, MODE, EXACT, WD, GS, true, kGradBf16, true, true>(t, (uint32_t)(t.numel / kBlock), n, lane, h, gscale, dbc1, dbc2, L, mine);
        if (EMA && t.shadow != nullptr) ema_tail(t, n, lane, h.ema_decay);
    }
    uint32_t next_round = __builtin_amdgcn_readfirstlane(coming[0]);
    // the last round may have fewer blocks than the workgroup has waves, and is a workgroup's last: a wave without one ends
    if (blk >= total_blocks) return;
    const f32x4 base_s = reinterpret_cast<const f32x4 *>(L.map_s)[lane]; // codes 4*lane .. 4*lane + 3
    const f32x4 base_u = reinterpret_cast<const f32x4 *>(L.map_u)[lane];

    uint32_t ti = 0, t_end = 0;
    DevTensor t;
    map.seek(rows, blk, ti, t, t_end);
    RawBlock raw;
    raw.issue(t, blk - t.full_start, lane);
    uint32_t nti = ti, nt_end = t_end;
    DevTensor nt = t;
    for (uint32_t slot = 1;; slot ^= 1) {
        const bool more = next_round < tickets.rounds;
        uint32_t answer = 0;
        if (more && threadIdx.x == 0) answer = tickets.ask(); // for the round after next
        // the block after this one; past the end every wave reads the table's last block, which a cache holds (the loads
        // must stay unconditional so that the raw registers have a single definition in the loop).  When each read its own
        // last block again a launch fetched 25 MB (bf16; 42 MB fp32) for nothing: 16,384 blocks of fp32 102.1 -> 101.3 us,
        // bf16 with fp32 gradients 75.8 -> 74.9, bf16 level; arrays far apart 99.1 -> 97.9, 74.2 -> 73.3, level
        const uint32_t nblk = next_round * waves_per_wg + wave_in_wg;
        const uint32_t pblk = more && nblk < total_blocks ? nblk : total_blocks - 1;
        map.seek(rows, pblk, nti, nt, nt_end);

        const uint32_t lb = blk - t.full_start;
        const float gscale = GS ? (h.grad_scale * t.grad_scale) * tscale : 1.0f;
        const size_t e0 = (size_t)lb * kBlock;
        char *p = static_cast<char *>(t.p) + e0 * (kParamBf16 ? 2 : 4);
        uint8_t *mc = t.m + e0;
        uint8_t *vc = t.v + e0;
        float mf[32], vf[32];
        u32x4 pw[4]; // updated parameters, packed
        float lm = 0.0f, lv = 0.0f;
        const float a_m = raw.a_m, a_v = raw.a_v;
        {
            f32x4 ds, du;
            ds.x = (base_s.x * a_m) * h.beta1; ds.y = (base_s.y * a_m) * h.beta1;
            ds.z = (base_s.z * a_m) * h.beta1; ds.w = (base_s.w * a_m) * h.beta1;
            du.x = (base_u.x * a_v) * h.beta2; du.y = (base_u.y * a_v) * h.beta2;
            du.z = (base_u.z * a_v) * h.beta2; du.w = (base_u.w * a_v) * h.beta2;
            reinterpret_cast<f32x4 *>(mine[0])[lane] = ds;
            reinterpret_cast<f32x4 *>(mine[1])[lane] = du;
        }
        // EMA: the shadow's words are requested first and used quarter by quarter in the update half, where the
        // registers of the moments are still filling up (in the requantisation half, beside the next block's
        // words, they did not fit: 104-152 bytes of scratch per lane)
        u32x4 sh[4];
        const bool with_shadow = EMA && t.shadow != nullptr;
        if (EMA && with_shadow) {
#pragma unroll
            for (int c = 0; c < 4; ++c) sh[c] = load_bf16_quarter(static_cast<const char *>(t.shadow) + e0 * 2, c, lane);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float pv[8], gv[8], pn[8];
            unpack_quarter(raw.p[c], pv);
            unpack_quarter(raw.g[c], gv);
            // one flag per element: flagged elements are put right quarter by quarter (before the shadow uses
            // them), and the exact chain runs for the flagged positions only
            Redo8 redo;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float t1 = lds_float_at(mine[0], code_offset(raw.m[c], k));
                const float t3 = lds_float_at(mine[1], code_offset(raw.v[c], k));
                float m, v;
                uint64_t flagged = 0;
                adam_elem_decayed<MODE, EXACT, kParamBf16, WD, GS>(pv[k], gv[k], t1, t3, h, gscale, dbc1, dbc2, m, v, pn[k], flagged);
                redo.set(k, flagged);
                mf[c * 8 + k] = m;
                vf[c * 8 + k] = v;
                lm = fmaxf(lm, __builtin_fabsf(m));
                lv = fmaxf(lv, __builtin_fabsf(v));
            }
            if (kParamBf16 && MODE == ERI_ADAM8_MODE_L2 && h.l2_all_exact) redo.set_all();
            if (kParamBf16 && redo.any) {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (redo.lanes[k] && redo.mine(k))
                        pn[k] = param_exact<MODE, WD, true>(pv[k], mf[c * 8 + k], vf[c * 8 + k], h, dbc1, dbc2);
            }
            if (kParamBf16) {
                pw[c].x = bf16_pair(pn[0], pn[1]);
                pw[c].y = bf16_pair(pn[2], pn[3]);
                pw[c].z = bf16_pair(pn[4], pn[5]);
                pw[c].w = bf16_pair(pn[6], pn[7]);
            } else { // fp32 parameters are final here (they take the exact chain): stored quarter by quarter
                store_f32_quarter(pn, p, c, lane);
            }
            if (EMA && with_shadow) {
                float out[8];
                ema_eight(sh[c], pw[c], h.ema_decay, out);
                const u32x4 w = {bf16_pair(out[0], out[1]), bf16_pair(out[2], out[3]), bf16_pair(out[4], out[5]), bf16_pair(out[6], out[7])};
                store_bf16_quarter(w, static_cast<char *>(t.shadow) + e0 * 2, c, lane);
            }
            // the quarter's raw words are dead: the next block's quarter takes their registers now
            raw.issue_quarter(nt, pblk - nt.full_start, c, lane);
            if (kParamBf16) store_bf16_quarter(pw[c], p, c, lane);
        }
        float nam = lm, nav = lv;
        wave_max2(nam, nav);
        if (lane == 0) {
            as_global(t.absmax_m)[lb] = nam;
            as_global(t.absmax_v)[lb] = nav;
        }
        const BlockDiv dm(nam, kKeyScale, kKeyScaleInv), dv(nav, kKeyScale, kKeyScaleInv);
        if (dm.fast && dv.fast) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                u32x2 mw, vw;
                requant8<true, true, MODE == ERI_ADAM8_MODE_BNB>(mf + c * 8, vf + c * 8, dm, dv, L, mw, vw);
                store_codes_quarter(mw, mc, c, lane);
                store_codes_quarter(vw, vc, c, lane);
            }
        } else {
            for (int c = 0; c < 4; ++c) {
                u32x2 mw, vw;
                requant8<false, true, MODE == ERI_ADAM8_MODE_BNB>(mf + c * 8, vf + c * 8, dm, dv, L, mw, vw);
                store_codes_quarter(mw, mc, c, lane);
                store_codes_quarter(vw, vc, c, lane);
            }
        }
        if (!more) break;
        if (threadIdx.x == 0) coming[slot] = tickets.round_of(answer);
        lds_barrier();
        next_round = __builtin_amdgcn_readfirstlane(coming[slot]);
        blk = nblk;
        t = nt;
        if (blk >= total_blocks) break;
    }
}

namespace {

template <int MODE, bool EXACT, bool WD, bool GS, bool EMA = false>
int launch_pipelined(const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h,
                     const void *lds_image, const float *dev_scale, uint32_t grid, uint32_t wg, hipStream_t s) {
    if (wg > kPipeThreads) wg = kPipeThreads;
    hipLaunchKernelGGL((ERI_PIPE_KERNEL<MODE, EXACT, WD, GS, EMA>), dim3(grid), dim3(wg), 0, s, rows, n_rows, total_blocks, n_tails, h,
                       static_cast<const uint4 *>(lds_image), dev_scale);
    return (int)hipGetLastError();
}

template <int MODE, bool EXACT>
int launch_flags(bool wd, bool gs, bool ema, const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h,
                 const void *img, const float *dev_scale, uint32_t grid, uint32_t wg, hipStream_t s) {
    if constexpr (MODE == ERI_ADAM8_MODE_ERI && kParamBf16) { // the EMA is built into the reference's own update, on bf16 parameters
        if (ema) {
            if (wd) {
                if (gs) return launch_pipelined<MODE, EXACT, true, true, true>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
                return launch_pipelined<MODE, EXACT, true, false, true>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
            }
            if (gs) return launch_pipelined<MODE, EXACT, false, true, true>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
            return launch_pipelined<MODE, EXACT, false, false, true>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
        }
    }
    if (wd) {
        if (gs) return launch_pipelined<MODE, EXACT, true, true>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
        return launch_pipelined<MODE, EXACT, true, false>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
    }
    if (gs) return launch_pipelined<MODE, EXACT, false, true>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
    return launch_pipelined<MODE, EXACT, false, false>(rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s);
}

} // namespace

/* All three modes, 160-220 registers, no scratch. */
#if ERI_PIPE_LAYOUT == 1
int launch_step_pipelined(int mode, bool exact, bool wd, bool gs, bool ema, const DevTensor *rows, uint32_t n_rows,
                          uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *img, const float *dev_scale,
                          uint32_t grid, uint32_t wg, void *stream) {
#elif ERI_PIPE_LAYOUT == 2
int launch_step_pipelined_grad_f32(int mode, bool exact, bool wd, bool gs, bool ema, const DevTensor *rows, uint32_t n_rows,
                                   uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *img,
                                   const float *dev_scale, uint32_t grid, uint32_t wg, void *stream) {
#else
int launch_step_pipelined_f32(int mode, bool wd, bool gs, const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails,
                              const EriAdam8Hyper &h, const void *img, const float *dev_scale, uint32_t grid,
                              uint32_t wg, void *stream) {
    const bool ema = false;   // fp32 rows get their EMA from the sweep
    constexpr bool exact = true; // fp32 parameters always take the IEEE square root and division
#endif
    hipStream_t s = static_cast<hipStream_t>(stream);
#define ERI_ARGS wd, gs, ema, rows, n_rows, total_blocks, n_tails, h, img, dev_scale, grid, wg, s
#if ERI_PIPE_LAYOUT == 0
    if (mode == ERI_ADAM8_MODE_L2) return launch_flags<ERI_ADAM8_MODE_L2, exact>(ERI_ARGS);
    if (mode == ERI_ADAM8_MODE_BNB) return launch_flags<ERI_ADAM8_MODE_BNB, exact>(ERI_ARGS);
    return launch_flags<ERI_ADAM8_MODE_ERI, exact>(ERI_ARGS);
#else
    if (mode == ERI_ADAM8_MODE_L2) return launch_flags<ERI_ADAM8_MODE_L2, true>(ERI_ARGS); // its fast chain always checks itself
    if (mode == ERI_ADAM8_MODE_BNB)
        return exact ? launch_flags<ERI_ADAM8_MODE_BNB, true>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_BNB, false>(ERI_ARGS);
    return exact ? launch_flags<ERI_ADAM8_MODE_ERI, true>(ERI_ARGS) : launch_flags<ERI_ADAM8_MODE_ERI, false>(ERI_ARGS);
#endif
#undef ERI_ARGS
}

} // namespace eri
