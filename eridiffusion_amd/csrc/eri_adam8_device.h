/*
 * Layouts shared by the host side of the library and its gfx950 kernels: the device row of the
 * launch table and the image of lookup tables every workgroup stages into LDS.
 */
#ifndef ERI_ADAM8_DEVICE_H
#define ERI_ADAM8_DEVICE_H

#include <stdint.h>

#include "../../include/eri_optim8.h"

namespace eri {

constexpr uint32_t kBlock = ERI_ADAM8_BLOCK; /* elements per quantisation block, one wavefront each */
constexpr uint32_t kWave = 64;

/* One tensor as the kernels see it (80 bytes, read through scalar loads). */
struct DevTensor {
    void *p;          /* new parameters are written here */
    const void *p_in; /* old parameters are read from here: p itself for an in-place update */
    const void *g;
    uint8_t *m;
    uint8_t *v;
    float *absmax_m;
    float *absmax_v;
    uint64_t numel;
    uint32_t full_start;  /* number of full 2048-element blocks in the rows before this one (same dtype) */
    float grad_scale;
    void *shadow;     /* EMA shadow of the parameter, or null */
};
static_assert(sizeof(DevTensor) == 80, "DevTensor must stay 80 bytes");
/* In front of the rows of a launch table or a sweep on the device: the counter its launches take their rounds from, zero
 * between launches, alone in its cache line. */
constexpr uint32_t kTableHead = 256;

/* New addresses for rows of a launch table, as a launch carries them in its arguments. */
struct RowAddresses {
    void *p;
    const void *p_in;
    const void *g;
};
constexpr uint32_t kAddressRows = 160, kGradRows = 480; /* 3.8 KB of arguments either way */
int launch_set_addresses(DevTensor *rows, const RowAddresses *a, uint32_t n, void *stream);
int launch_set_gradients(DevTensor *rows, const void *const *g, uint32_t n, void *stream);

/* How the elements of one group of rows are stored: parameters and gradients F32, both BF16, or BF16
 * parameters with F32 gradients (the reference casts every gradient to F32 and never rounds it). */
enum Layout { kLayoutF32 = 0, kLayoutBF16 = 1, kLayoutBF16GradF32 = 2, kLayouts = 3 };
inline bool layout_param_bf16(int layout) { return layout != kLayoutF32; }
inline bool layout_grad_bf16(int layout) { return layout == kLayoutBF16; }

/*
 * Requantisation without a search.  The quotient x = value / absmax in [-1, 1] is produced
 * already multiplied by kKeyScale (a power of two, so nothing is rounded differently), converted
 * to binary16 rounded toward zero (both moments in one v_cvt_pkrtz_f16_f32), and the top bits of that half float -- sign, exponent
 * and the leading mantissa bits -- select a slot.  The slots are narrow enough that at most one
 * midpoint of the map lies inside any of them, so
 *     code(x) = slot.lo + (x * kKeyScale > slot.mid)
 * equals the number of midpoints below x, i.e. the binary search's answer, ties included.
 * Every binary16 pattern has a slot: there is nothing to clamp, NaN lands in slots that answer 0
 * (a search finds every comparison false), and the scale keeps all midpoints in the normal
 * binary16 range, so the result does not depend on how half denormals are treated.
 */
struct KeySlot {
    float mid;   /* the one midpoint inside the slot times kKeyScale, +inf if there is none */
    uint32_t lo; /* number of midpoints below every value of the slot */
};

constexpr float kKeyScale = 4096.0f;
constexpr float kKeyScaleInv = 1.0f / 4096.0f;
constexpr uint32_t kSKeyDrop = 4;   /* signed map: keep 6 mantissa bits of the half float */
constexpr uint32_t kUKeyDrop = 3;   /* unsigned map: keep 7 */
constexpr uint32_t kSKeyStride = 16; /* bytes between signed slots: address = half & 0xfff0 */
constexpr uint32_t kUKeyStride = 8;  /* bytes between unsigned slots: address = half & 0x7ff8 */
constexpr uint32_t kSKeyCount = 1u << (16 - kSKeyDrop); /* 4096, sign included */
constexpr uint32_t kUKeyCount = 1u << (15 - kUKeyDrop); /* 4096, sign masked off */

/* Byte offsets inside the LDS image. */
constexpr uint32_t kOffMapS = 0;                              /* 256 floats: code -> value */
constexpr uint32_t kOffMapU = kOffMapS + 1024;                /* 256 floats */
constexpr uint32_t kOffMidS = kOffMapU + 1024;                /* 255 midpoints + one +inf */
constexpr uint32_t kOffMidU = kOffMidS + 1024;
/* Both slot tables start below 64 KiB so that their offsets fit the 16-bit immediate of ds_read. */
constexpr uint32_t kOffKeyU = kOffMidU + 1024;                /* kUKeyCount slots, kUKeyStride apart */
constexpr uint32_t kOffKeyS = kOffKeyU + kUKeyCount * kUKeyStride; /* kSKeyCount slots */
constexpr uint32_t kLdsImageBytes = kOffKeyS + kSKeyCount * kSKeyStride;
static_assert(kOffKeyS < 65536 && kOffKeyU < 65536, "slot table offsets must fit a ds_read immediate");
static_assert(kLdsImageBytes % 16 == 0, "the image is staged in 16-byte words");

/* The same lookup in 12 KB, for kernels that cannot afford to stage 100 KB per workgroup: a slot keeps only its `lo`,
 * one byte.  Its midpoint need not be stored, because the one midpoint a slot can contain is midpoint number `lo`,
 * and where it contains none, no quotient of the slot lies above midpoint `lo` either:
 *     code(x) = lo[slot] + (x * kKeyScale > scaled_mid[lo[slot]])
 * Two dependent LDS reads instead of one. */
constexpr uint32_t kSmallMapS = 0;                        /* 256 floats: code -> value */
constexpr uint32_t kSmallMapU = kSmallMapS + 1024;
constexpr uint32_t kSmallMidS = kSmallMapU + 1024;        /* 255 midpoints times kKeyScale + one +inf */
constexpr uint32_t kSmallMidU = kSmallMidS + 1024;
constexpr uint32_t kSmallLoS = kSmallMidU + 1024;         /* kSKeyCount bytes */
constexpr uint32_t kSmallLoU = kSmallLoS + kSKeyCount;    /* kUKeyCount bytes */
constexpr uint32_t kSmallImageBytes = kSmallLoU + kUKeyCount;
static_assert(kSmallImageBytes % 1024 == 0, "the image is staged in pieces of 1 KB");

/* What the choice of a step's kernel goes by, of the rows of one layout. */
struct TableShape {
    uint32_t total_blocks; // full ones
    uint32_t n_tails;      // partial last blocks
    uint32_t n_long;       // of these, the ones of more than half a block
    int layout;
    uint32_t units() const { return total_blocks + n_tails; } // a partial block costs about what a full one does
};

/* Launchers implemented in eri_adam8_kernels.hip; `stream` is a hipStream_t.  All return a
 * hipError_t as int.  `lds_image` is the device copy of the kLdsImageBytes table image. */
int launch_step(const DevTensor *rows, uint32_t n_rows, const TableShape &t, const EriAdam8Hyper &h, const void *lds_image,
                const float *dev_scale, uint32_t grid, uint32_t wg, uint32_t compute_units, void *stream);

constexpr uint32_t kChunks = 8;           /* contiguous ranges the gradient-norm pass cuts long block lists into: one per accelerator die */
/* Tables of at most this many blocks per compute unit (partial ones counted) take the four-waves-per-block kernel: one
 * round of its four teams.  Beyond it that kernel pays a barrier and a trip to memory per round, and a wave per block
 * fills the chip by itself.  us per launch on 256 units, four waves per block | one:
 *   blocks      1,024        1,536         2,816         8,192
 *   bf16       7.6 | 8.9  10.6 | 10.5  15.7 | 15.1   38.4 | 33.7
 *   fp32       9.0 | 10.1 14.4 | 12.8  23.9 | 20.8   53.3 | 50.3
 *   bf16, fp32 gradients, functional update
 *              8.2 | 8.9  12.5 | 10.9  17.3 | 15.1   44.0 | 35.3
 * and with partial blocks of 1,027 elements behind the full ones, just past the line and further:
 *   blocks  1,024 + 64   1,024 + 512   1,536 + 64    2,048 + 64    2,816 + 64
 *   bf16   13.2 | 13.3   13.6 | 14.2   13.8 | 14.2   18.0 | 16.1   18.2 | 17.2
 *   fp32   13.4 | 13.6   14.4 | 14.1   15.3 | 14.7   21.0 | 18.2   23.6 | 20.3 */
constexpr uint32_t kSplitBlocksPerCu = 4;
/* Tables of both parameter dtypes with at most this many blocks per compute unit in all take one launch: it saves the
 * start of a second one, and on larger tables the two kernels' code side by side costs as much.  us, two launches of a
 * wave per block | one, half of the blocks fp32, 256 units:
 *   blocks   256         1,024       2,816       8,192       32,768
 *         14.4 | 8.4  16.6 | 10.7  23.4 | 20.6  50.0 | 46.0  160.8 | 163 */
constexpr uint32_t kTwoDtypeBlocksPerCu = 64;
/* Tables take the prefetching kernel above this many full blocks per compute unit.  Its eight waves by ticket get more out
 * of HBM, the plain kernel's sixteen start and end sooner and hide more arithmetic: mode L2's recomputed elements, the
 * IEEE chain of fp32 parameters.  us per launch, prefetching kernel | plain, 256 units, no two launches on the same data:
 *   blocks                 8,192      12,288      16,896      21,997      37,392      74,784     157,651
 *   bf16                 38 | 34     52 | 50     67 | 68     86 | 93   138 | 143   267 | 294   547 | 671
 *   ... fp32 gradients   41 | 39     59 | 60     77 | 83   100 | 111   160 | 176   310 | 351   637 | 775
 *   fp32                 58 | 58     82 | 84   108 | 114   132 | 146   216 | 235   420 | 482  865 | 1,026
 *   bf16, mode L2        43 | 37     56 | 53     71 | 70     96 | 95   146 | 146   274 | 302   561 | 684
 *   ... fp32 gradients   45 | 37     62 | 62     80 | 85   107 | 110   165 | 179   314 | 360   642 | 770
 *   fp32, mode L2        65 | 61     90 | 90                           242 | 256
 *   bf16, mode BNB       42 | 36     58 | 52     73 | 70     98 | 95   148 | 150   280 | 301   573 | 682
 *   ... fp32 gradients   45 | 39     63 | 62     81 | 84   107 | 115   166 | 180   321 | 350   655 | 781
 *   fp32, mode BNB       60 | 58     84 | 84                           220 | 241
 * Arrays side by side, as a caller's allocator places what it has for one model.  In lanes 48 GiB apart the plain kernel's
 * fixed shares lose little, and the two are level to 3 % around the line (bf16, launches on other data each time; one
 * table again and again is up to 2 % better for the plain kernel): 16,896 blocks 65 | 63, 21,997 with partial ones 83 | 83,
 * 37,392 131 | 130, 74,784 257 | 262, 157,651 524 | 547.  The same run side by side: 67 | 69, 85 | 95, 135 | 147,
 * 257 | 307, 533 | 664.  The line stands where the placement that costs more decides it. */
inline uint32_t prefetch_blocks_per_cu(int mode, int layout) {
    if (mode == ERI_ADAM8_MODE_L2) return layout == kLayoutBF16 ? 96 : 48;
    if (mode == ERI_ADAM8_MODE_BNB) return layout == kLayoutBF16 ? 128 : layout == kLayoutBF16GradF32 ? 56 : 48;
    return layout == kLayoutF32 ? 40 : 48;
}
/* Partial blocks run in front of that kernel's tickets, a wave each without a prefetch, at what their length costs; the
 * plain kernel takes them like whole ones.  With bf16 parameters it is the faster one where many of them are long.  us per
 * launch, prefetching kernel | plain, 256 units, tensors of k blocks and a part of 1,501 elements:
 *   blocks, k            16,384, 1   16,384, 2   16,384, 4   37,376, 1   37,376, 2   37,376, 4
 *   bf16                 151 | 138   108 | 104     86 | 87   330 | 307   232 | 227   182 | 190
 *   ... fp32 gradients   168 | 159   119 | 124    97 | 105   360 | 355   252 | 271   203 | 231
 *   fp32                 200 | 215   153 | 163   124 | 139   432 | 478   324 | 363   263 | 308
 *   bf16, mode L2                                            333 | 294   233 | 222   185 | 189
 *   bf16, mode BNB                                           325 | 288   231 | 219   183 | 187
 * and where all are short (952 elements, k = 1) it is not: 16,384 blocks bf16 122 | 137, 35,840 in mode L2 251 | 267. */
inline bool long_tails_weigh(const TableShape &t) {
    if (t.layout == kLayoutF32) return false;
    return (uint64_t)t.n_long * (t.layout == kLayoutBF16 ? 3 : 2) > t.total_blocks;
}
/* Above this many full blocks per compute unit the gradient-norm pass cuts its list into ranges. */
constexpr uint32_t kNormRangesBlocksPerCu = 1024;
constexpr uint32_t kNormWaves = 4;        /* waves per workgroup of the gradient-norm pass */

/* Such a walk needs the same number of workgroups in every range. */
inline uint32_t chunks_for(uint32_t grid) { return grid % kChunks == 0 ? kChunks : 1u; }

/* The step's kernels live in translation units of their own (they build in parallel); launch_step
 * picks one.  wd / gs / keytab / exact select template instances: decay present, gradient scale present,
 * slot-table (rather than binary-search) requantisation, IEEE square root and division on bf16. */
int launch_step_plain_f32(int mode, bool wd, bool gs, bool keytab, const DevTensor *rows, uint32_t n_rows,
                          uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale,
                          uint32_t grid, uint32_t wg, void *stream);
int launch_step_plain_bf16(int mode, bool exact, bool wd, bool gs, bool keytab, const DevTensor *rows, uint32_t n_rows,
                           uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale,
                           uint32_t grid, uint32_t wg, void *stream);
/* bf16 parameters with fp32 gradients: slot tables only. */
int launch_step_plain_grad_f32(int mode, bool exact, bool wd, bool gs, const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks,
                               uint32_t n_tails, const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale, uint32_t grid,
                               uint32_t wg, void *stream);
/* Four waves per block, for tables of few blocks; `grid` workgroups of 1024 threads. */
int launch_step_split(int layout, int mode, bool exact, bool wd, bool gs, const DevTensor *rows, uint32_t n_rows,
                      uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale,
                      uint32_t grid, uint32_t teams, void *stream);
/* One group of rows of a launch. */
struct StepGroup {
    const DevTensor *rows;
    uint32_t n_rows, total_blocks, n_tails;
};
/* The fp32 and the bf16 rows of one table (gradients of the parameters' dtypes) in one launch of a wave per block. */
int launch_step_two(const StepGroup &f32, const StepGroup &bf16, const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale,
                    uint32_t grid, uint32_t wg, void *stream);
/* Whether launch_step would run this group on the prefetching kernel with the EMA update inside it.  units: full blocks
 * and partial ones. */
bool step_fuses_ema(const TableShape &t, const EriAdam8Hyper &h, uint32_t compute_units);
int launch_step_pipelined(int mode, bool exact, bool wd, bool gs, bool ema, const DevTensor *rows, uint32_t n_rows,
                          uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale,
                          uint32_t grid, uint32_t wg, void *stream);
/* The same kernel for bf16 parameters whose gradients are fp32. */
int launch_step_pipelined_grad_f32(int mode, bool exact, bool wd, bool gs, bool ema, const DevTensor *rows, uint32_t n_rows,
                                   uint32_t total_blocks, uint32_t n_tails, const EriAdam8Hyper &h, const void *lds_image,
                                   const float *dev_scale, uint32_t grid, uint32_t wg, void *stream);
/* The same kernel for fp32 parameters (IEEE chain throughout, no EMA inside it). */
int launch_step_pipelined_f32(int mode, bool wd, bool gs, const DevTensor *rows, uint32_t n_rows, uint32_t total_blocks, uint32_t n_tails,
                              const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale, uint32_t grid,
                              uint32_t wg, void *stream);
/* Sum of |moment - dequantised moment| of the coming step, per row: err[2r] first moment, err[2r+1] second. */
int launch_quant_error(const DevTensor *rows, uint32_t n_rows, uint32_t total_full_blocks, int layout,
                       const EriAdam8Hyper &h, const void *lds_image, const float *dev_scale, double *err,
                       uint32_t grid, void *stream);
/* Gradient norm: one f64 pair per workgroup (sum of squares, count of non-finite elements), then norm and clip factor
 * into out[0], out[1].  A pass covers up to two tables, a group per layout each. */
constexpr uint32_t kNormWavesPerCu = 32; // persistent waves of the gradient-norm pass per compute unit
struct NormGroup {
    const DevTensor *rows;
    uint32_t n_rows, total_blocks, n_tails;
    uint32_t first_wg, wgs; // the launch's workgroups that take this group
    uint32_t chunks;        // ranges the block list is cut into
    uint32_t grad_bf16;
};
struct NormGroups {
    NormGroup g[2 * kLayouts];
    uint32_t n;
};
int launch_grad_sumsq(const NormGroups &groups, double *partial, void *stream);
int launch_grad_norm_finish(const double *partial, uint32_t n, float max_norm, float denom_eps, float *out,
                            void *stream);
/* Diagnostics: reads and rewrites (unchanged) every full block of a group of bf16 rows as the step does. */
int launch_traffic_probe(const DevTensor *rows, uint32_t n_rows, uint32_t total_full_blocks, uint32_t grid, void *stream);
/* Clears `bytes` bytes at `p`; both multiples of 16. */
int launch_fill_zero(void *p, size_t bytes, void *stream);
int launch_state_init(uint8_t *m, uint8_t *v, float *absmax_m, float *absmax_v, uint64_t numel, void *stream);
/* fp32 moments <-> codes and absmax, any number of moments in one launch; `small_image` is the device copy of the
 * kSmallImageBytes image. */
struct Moment {
    float *x; /* fp32 values: read by quantize, written by dequantize */
    uint8_t *codes;
    float *absmax;
    uint64_t numel;
    bool is_signed;
};
int launch_dequantize(const Moment *moments, uint32_t n, const void *small_image, void *stream);
int launch_quantize(const Moment *moments, uint32_t n, const void *small_image, void *stream);

/* Row of the plain element-wise sweeps (32-bit AdamW, EMA): up to five streams of one tensor. */
struct ElemRow {
    void *a;        /* AdamW: p      EMA: shadow */
    const void *b;  /* AdamW: g      EMA: p */
    void *c;        /* AdamW: m (fp32) */
    void *d;        /* AdamW: v (fp32) */
    void *e;        /* AdamW: fp32 master copy of p, or null */
    uint64_t numel;
    uint32_t full_start; /* full 2048-element blocks in the rows before this one */
    float scale;         /* AdamW: per-layer multiplier of the gradients (used by the scaled step only) */
};
static_assert(sizeof(ElemRow) == 56, "ElemRow must stay 56 bytes");

/* One block of a small sweep: block `block` of row `row`.  The small kernels take one per workgroup, a quarter per wave:
 * with a wave per block a table of few blocks lasts as long as one wave's chain of a row search, a partial block and a
 * full one. */
struct SweepUnit {
    uint32_t row, block;
};
/* Sweeps of at most this many blocks per compute unit take the small kernels, whose workgroups the hardware starts in the
 * order of the list, many to a unit.  us per call over the same arrays, a quarter block per wave | by ticket, 256 units:
 *   blocks                 2,048     8,192      16,824      23,639      31,398     72,781       639,470
 *   32-bit step, bf16    16 | 24    59 | 70  119 | 137   168 | 189   236 | 269   554 | 564   5,205 | 4,791
 *   ... fp32                                 159 | 164   229 | 226   313 | 309   749 | 673   6,692 | 5,879
 *   ... with masters                         157 | 166   223 | 230               731 | 685   6,784 | 5,992
 *   EMA, bf16           4.5 | 8.5   17 | 24   31 | 41     44 | 53     58 | 71    133 | 147   1,193 | 1,217
 *   ... fp32                                  62 | 71     89 | 96    120 | 126   287 | 277   2,606 | 2,364
 * Above it the list itself (8 bytes per block, uploaded when the rows' sizes change) is no longer small. */
constexpr uint32_t kSmallSweepBlocksPerCu = 128;
/* Nor is it needed there, except for partial blocks, of which the persistent kernels take one piece per wave ahead of
 * their tickets, with eight waves per unit and nothing to hide behind.  Where these are most of a sweep the list is no
 * longer than the rows are.  us per call, the small kernels | by ticket, 20,000 tensors (40,000 and 34,000 of the first two sizes):
 *   elements                   301         1,501         2,148         3,075         5,597         9,693
 *   EMA, bf16              30 |  95     53 | 133      61 |  91      69 | 106     106 | 160     181 | 236
 *   ... fp32               36 |  66     96 | 104     112 | 113     140 | 128     218 | 221     381 | 376
 *   32-bit step, bf16      74 | 270    204 | 311     226 | 275     287 | 319     451 | 478     768 | 776
 *   ... with masters       82 | 273    261 | 309     292 | 326     371 | 352     588 | 577     997 | 954
 *   ... fp32               77 | 180    249 | 257     287 | 281     361 | 304     566 | 530     975 | 903
 * wide: fp32 tensors, or masters beside bf16 ones. */
inline bool small_sweep(uint64_t units, uint64_t partial, bool wide, uint32_t compute_units) {
    if (units <= (uint64_t)compute_units * kSmallSweepBlocksPerCu) return true;
    const uint64_t full = units - partial;
    return units < (1u << 20) && (wide ? partial > full : 2 * partial >= full);
}

/* units: the list of blocks, n_units of them, for the small kernels; null for the persistent ones, which take `grid`
 * workgroups.  scaled: every gradient is first multiplied by (grad_scale * row.scale) * (*dev_scale, 1 if null), as the
 * 8-bit step does with ERI_ADAM8_FLAG_GRAD_SCALE. */
int launch_adamw32(const ElemRow *rows, uint32_t n_rows, uint32_t total_full_blocks, const SweepUnit *units, uint32_t n_units,
                   int dtype_tag, const EriAdamW32Hyper &h, bool scaled, float grad_scale, const float *dev_scale, uint32_t grid,
                   void *stream);
int launch_ema(const ElemRow *rows, uint32_t n_rows, uint32_t total_full_blocks, const SweepUnit *units, uint32_t n_units,
               int dtype_tag, float decay, uint32_t grid, void *stream);

} // namespace eri
#endif
