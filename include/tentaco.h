/*
 * tentaco.h - C ABI of the MI355X (gfx950) CSF MTTKRP / TTV library.
 *
 * Every function here has C linkage, takes plain pointers and sizes, and
 * reports failure through its return code plus tentaco_last_error(); no
 * entry point calls exit(). The reference's boundary (gpu_kernels.cuh:1-73 of
 * zhang677/tenTACO) is reproduced in three layers:
 *
 *  1. Compute-style entry points, host pointers in, A filled on return:
 *     tentaco_mttkrp3/4/5, tentaco_ttv, tentaco_mttkrp (any order).
 *  2. The reference's own symbol names with their void signatures
 *     (mttkrp_gpu_taco, ttv_csf_gpu_taco, the 67 mttkrp_{R}_eb_{sr|pr}_...
 *     tuning variants, get_gpu_timer_result), so a caller that was compiled
 *     against gpu_kernels.cuh relinks against this library unchanged.
 *  3. A device-resident API (upload a CSF once, run many MTTKRP/TTV calls on
 *     device factors, on a caller stream) for CP-ALS-style loops, batching
 *     and graph capture.
 *
 * Operand contract (matches gpu_library.h:780-859 / ds.h:368-436):
 *   B  CSF tensor, order N in 2..5: indices[0] = {pos={0,n0}, crd[n0]},
 *      indices[m] = {pos, crd} for m >= 1, vals = FP32[nnz]. int32 indices.
 *   C, D, E, F  factor matrices for levels 1..N-1: dimensions = {rows, R},
 *      row-major FP32, element [row*R + col] (ds.h:401).
 *   A  MTTKRP output: dimensions = {rows, R}; every row is overwritten
 *      (rows of empty slices become 0). Row of root node x is crd0[x].
 *   A  TTV output: FP32 vector aligned with B's level N-2 positions (the
 *      (i,j) fibers of a 3-mode tensor); its index pattern is B's levels
 *      0..N-2, so only vals are written.
 */
#ifndef TENTACO_H
#define TENTACO_H

#include <stddef.h>
#include <stdint.h>
#include "taco_tensor_t.h"

#ifdef __cplusplus
extern "C" {
#endif

/* ---- status codes ------------------------------------------------------ */
#define TENTACO_OK 0
#define TENTACO_EINVAL 1        /* malformed operand or argument */
#define TENTACO_EHIP 2          /* HIP runtime error */
#define TENTACO_ENOMEM 3        /* device or host allocation failed */
#define TENTACO_EUNSUPPORTED 4  /* valid request this build does not handle */
#define TENTACO_ENOGPU 5        /* no usable gfx950 device */

/* Variant selector for the MTTKRP kernels (tentaco_variant_name lists them).
 * TENTACO_VARIANT_AUTO lets the library choose (autotuned table or learned
 * selector, falling back to the fixed default). */
#define TENTACO_VARIANT_AUTO (-1)
#define TENTACO_VARIANT_DEFAULT (-2)  /* the fixed TACO-schedule default */

/* Message describing the last failure on the calling thread ("" if none). */
const char* tentaco_last_error(void);
/* Library version, major*10000 + minor*100 + patch. */
int tentaco_version(void);
/* 0 when a gfx950 device is usable, else TENTACO_ENOGPU (no kernel runs). */
int tentaco_device_check(void);

/* ---- layer 1: compute-style entry points (host pointers) --------------- */
/* Replace mttkrp3_cpu_taco (tensor_kernels/mttkrp3_csf_cpu_taco.h:7) and the
 * GPU wrappers of gpu_kernels.cuh:5-73 for a 3-mode CSF. Returns 0. */
int tentaco_mttkrp3(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C,
                    taco_tensor_t* D);
/* Replaces mttkrp4_cpu_taco (tensor_kernels/mttkrp4_csf_cpu_taco.h:7). */
int tentaco_mttkrp4(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C,
                    taco_tensor_t* D, taco_tensor_t* E);
/* Replaces mttkrp5_cpu_taco (tensor_kernels/mttkrp5_csf_cpu_taco.h:7). */
int tentaco_mttkrp5(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C,
                    taco_tensor_t* D, taco_tensor_t* E, taco_tensor_t* F);
/* Any order 2..5: factors[m-1] is the factor of level m. variant as above.
 * Same contract as tentaco_mttkrp3 (gpu_kernels.cuh:5). The order is passed
 * explicitly because the reference's to_taco_tensor (ds.h:368-384) leaves
 * taco_tensor_t.order unset. */
int tentaco_mttkrp(int order, taco_tensor_t* A, taco_tensor_t* B,
                   taco_tensor_t* const* factors, int variant);
/* Replaces ttv_csf_cpu_taco (tensor_kernels/ttv_csf_cpu_taco.h:24) and
 * ttv_csf_gpu_taco (gpu_kernels.cuh:6): A[f] = sum_k B(f,k) c(k) over the
 * level N-2 positions f of B. */
int tentaco_ttv(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* c);
/* TTV over the last mode of an order-2..5 CSF (order passed explicitly). */
int tentaco_ttv_n(int order, taco_tensor_t* A, taco_tensor_t* B,
                  taco_tensor_t* c);

/* ---- layer 2: reference symbol names (gpu_kernels.cuh:4-73) ------------ */
/* The library exports every name of this layer twice: with C linkage (the
 * declarations below) and with C++ linkage, as gpu_kernels.cuh declares them,
 * so objects compiled against either header link. The C++ definitions
 * forward to these three helpers: family < 0 is the fixed default, family 0
 * an eb_sr name (block TB, p = run length g), family 1 an eb_pr name (block
 * TB, p = Nnz, the reference's nonzeros per block). */
float tentaco_legacy_timer_ms(void);
void tentaco_legacy_mttkrp3(int family, int block, int p, const char* name,
                            taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C,
                            taco_tensor_t* D);
/* The variant that the reference name `name` (mttkrp_gpu_taco or one of the
 * 66 tuning names) runs for a tensor of this order at rank R. */
int tentaco_legacy_variant(const char* name, int R, int order, int* variant);
void tentaco_legacy_ttv3(const char* name, taco_tensor_t* A, taco_tensor_t* B,
                         taco_tensor_t* C);

/* Milliseconds of the last call's hot region (partition + zero + kernel),
 * hipEvent-timed like GPUTimer (gpu_library.h:949-988); -1 before any call.
 * Structures built once per CSF (the slice-row expansion, the TTV plan) are
 * built before the region starts. */
float get_gpu_timer_result(void);
/* TACO schedule (mttkrp3_csf_gpu_taco.h:73); runs the fixed default variant. */
void mttkrp_gpu_taco(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C,
                     taco_tensor_t* D);
/* ttv_csf_gpu_taco.h:89. */
void ttv_csf_gpu_taco(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C);

/* Tuning variants of gpu_kernels.cuh:7-73. eb_sr_{TB}_{g}_{c} runs the
 * edge-serial kernel at block TB with run length g (c, the columns per
 * thread, is fixed by R in the wave64 lane layout). eb_pr_{TB}_{Nnz}_{gs}
 * runs the edge-parallel tile whose nonzeros per workgroup are nearest to
 * Nnz at the call's rank (gs, the reference's reduction group width, has no
 * counterpart: the reduction spans the workgroup). */
#define TENTACO_DECL_VARIANT(name)                                             \
  void name(taco_tensor_t* A, taco_tensor_t* B, taco_tensor_t* C,            \
            taco_tensor_t* D);
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_4_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_64_32_manual)
TENTACO_DECL_VARIANT(mttkrp_64_eb_pr_256_32_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_32_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_32_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_32_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_32_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_64_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_64_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_64_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_64_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_128_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_128_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_128_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_128_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_256_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_256_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_256_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_256_256_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_64_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_64_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_64_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_64_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_128_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_128_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_128_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_128_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_256_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_256_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_256_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_256_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_512_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_512_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_512_16)
TENTACO_DECL_VARIANT(mttkrp_32_eb_pr_512_512_32)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_4_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_4_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_4_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_4_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_8_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_8_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_8_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_8_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_16_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_16_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_16_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_16_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_32_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_32_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_32_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_256_32_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_4_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_4_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_4_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_8_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_8_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_8_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_8_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_16_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_16_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_16_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_16_8)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_32_1)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_32_2)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_32_4)
TENTACO_DECL_VARIANT(mttkrp_32_eb_sr_512_32_8)
#undef TENTACO_DECL_VARIANT

/* ---- variant table ------------------------------------------------------ */
/* Number of MTTKRP kernel variants (the sweep/selector space). */
int tentaco_num_variants(void);
/* "es_b256_g16"-style name of variant v, or NULL when out of range. */
const char* tentaco_variant_name(int v);
/* Decode variant v: family (0 edge-serial, 1 edge-parallel, 2 slice-row),
 * block size and group size. Returns 0 or TENTACO_EINVAL. */
int tentaco_variant_params(int v, int* family, int* block, int* group);
/* The fixed default variant (the TACO schedule eb_sr 512/g=4). */
int tentaco_default_variant(void);
/* 1 when variant v's tile fits the LDS limit for this order and rank (a
 * launch of a variant that does not fit returns TENTACO_EUNSUPPORTED). */
int tentaco_variant_fits(int order, int R, int v);

/* ---- layer 3: device-resident API -------------------------------------- */
typedef struct tentaco_csf tentaco_csf; /* opaque device-resident CSF */

/* Validate a host CSF of the given order (contract above) and copy it to the
 * device. The handle owns its device memory; free with tentaco_csf_free. Not
 * tied to a stream. Validation rejects pos arrays that decrease or overrun,
 * root coordinates that are not strictly increasing, and coordinates outside
 * B->dimensions, so no kernel can read out of bounds. */
int tentaco_csf_upload(const taco_tensor_t* B, int order, tentaco_csf** out);
/* The validation of tentaco_csf_upload alone, on the host: 0, or the code
 * the upload would return (no device call). */
int tentaco_csf_check(const taco_tensor_t* B, int order);
int tentaco_csf_free(tentaco_csf* h);
/* order, nnz, number of root nodes, and node counts per level (nodes[5]). */
int tentaco_csf_info(const tentaco_csf* h, int* order, int64_t* nnz,
                     int32_t* nodes);
/* Reserve the per-handle workspace a variant needs, so that later calls on
 * this handle with at most dims[0] output rows allocate nothing (required
 * before graph capture). Edge variants need the partition brackets, and for
 * the variant named here (AUTO: the one it resolves to) the call builds the
 * table of the waves' start nodes, which later calls read instead of writing
 * brackets (4(order-1) B per 16 to 1024 nonzeros; without a reserve call, the
 * first call of a run length builds it and synchronizes its stream), and for
 * edge-parallel tiles of 2048 workgroups and more, and AUTO's from 300k nonzeros,
 * the FP64 rows of the slices that workgroups share (16 R B per workgroup, the 8
 * last used kept; calls outside capture use them, each waiting for the one before
 * on this handle; AUTO runs its variant's own tile where it has none). Memory
 * that does not suffice for these leaves calls without them, and only a reserve
 * call tries again; the
 * edge-serial family also accumulates its rows in FP64 (output rows x R
 * doubles), which keeps atomics on giant slices accurate. For 3-mode
 * handles it also builds the slice-row structures: the expansion (4 B per
 * nonzero plus 4 B per root node) and, for short fibres whose slices fit,
 * the padded slice layout (8 B per slot, at most 2 slots per nonzero). */
int tentaco_csf_reserve(tentaco_csf* h, int R, int variant);
/* The same for calls with a_rows output rows (the edge-serial FP64 rows
 * scale with a_rows). A call enqueued on a capturing stream that would need
 * more workspace than is reserved fails with TENTACO_EINVAL instead of
 * allocating; a workspace replaced by a larger one stays allocated until
 * tentaco_csf_free, so graphs captured before remain valid. */
int tentaco_csf_reserve_rows(tentaco_csf* h, int R, int variant, int32_t a_rows);

/* MTTKRP on device buffers: factors_dev[m-1] (rows_m x R, row-major) for
 * levels m = 1..N-1; A_dev has a_rows x R floats and is fully overwritten.
 * Enqueued on `stream` (a hipStream_t; NULL = default stream); returns
 * after enqueueing. */
int tentaco_mttkrp_dev(tentaco_csf* h, int R, const float* const* factors_dev,
                       float* A_dev, int32_t a_rows, int variant,
                       void* stream);
/* tentaco_mttkrp_dev without any allocation. It has no counterpart in the
 * reference; it is for callers that cannot allocate device memory (code
 * under hipGraph capture, tight serving loops, harnesses that forbid
 * hipMalloc). The call's scratch (partition brackets; FP64 rows for the
 * edge-serial family) lives in a static 32 MiB device array, one per device,
 * held until the process ends; a call that needs more returns
 * TENTACO_EUNSUPPORTED. The scratch is cleared by the call's own kernels.
 * Every call on a device shares that device's array, so calls that overlap
 * on one device (two streams, two threads) race: serialise them. AUTO takes
 * the handle's recorded choice or the structural heuristic (never the
 * selector or the sweep); the slice-row family uses the 3-mode structures
 * only if tentaco_csf_reserve built them. */
int tentaco_mttkrp_dev_noalloc(tentaco_csf* h, int R,
                               const float* const* factors_dev, float* A_dev,
                               int32_t a_rows, int variant, void* stream);
/* Sweep (the measurement of codegen.py + the *_tune.sh loops of the
 * reference, ebsr_32_tune.sh:1-16): times every variant on this handle, rank
 * and device factors with hipEvents on `stream`. Each variant gets a warm-up
 * and a one-call probe (the timed warm-up itself when it exceeds 2 ms);
 * every variant whose probe is within `cut` x the
 * fastest probe (all of them when cut <= 0) is then timed `reps` times, each
 * repetition spanning about 100 us of back-to-back calls (at most 32), and
 * its median per-call time kept. times_ms (tentaco_num_variants() entries)
 * receives per-call ms: the median, the probe for variants past the cut, -1
 * for a variant this rank cannot run. Reserves the largest workspace first;
 * changes nothing else on the handle; not for graph capture. */
int tentaco_csf_sweep(tentaco_csf* h, int R, const float* const* factors_dev,
                      float* A_dev, int32_t a_rows, int reps, float cut,
                      void* stream, float* times_ms);
/* Autotuner (replaces codegen.py + the *_tune.sh sweeps of the reference):
 * tentaco_csf_sweep with cut = 4, then records the fastest variant in the
 * handle so TENTACO_VARIANT_AUTO uses it, and returns it in *best. times_ms
 * (optional) receives the sweep's times. Not for graph capture. */
int tentaco_csf_autotune(tentaco_csf* h, int R, const float* const* factors_dev,
                         float* A_dev, int32_t a_rows, int reps, void* stream,
                         int* best, float* times_ms);
/* Record a variant as this handle's choice for rank R (e.g. from a stored
 * sweep or the learned selector). */
int tentaco_csf_set_tuned(tentaco_csf* h, int R, int variant);

/* How a handle's AUTO choice for rank R was made. */
#define TENTACO_TUNED_NONE 0      /* no entry: AUTO uses the selector or heuristic */
#define TENTACO_TUNED_SWEEP 1     /* measured by the sweep (autotune) */
#define TENTACO_TUNED_SELECTOR 2  /* the learned selector's pick */
#define TENTACO_TUNED_SET 3       /* set by tentaco_csf_set_tuned */
#define TENTACO_TUNED_SELECTOR_TIMED 4  /* best of the selector's top-k, timed */
/* The recorded choice for rank R: *variant = -1 and *source = NONE if none. */
int tentaco_csf_tuned(const tentaco_csf* h, int R, int* variant, int* source);
/* The variant a call with `variant` runs at rank R without consulting a
 * selector: AUTO gives the recorded choice, else the structural heuristic
 * (slice-row for many even slices; edge-parallel 256 x 16 below 300k
 * nonzeros and 512 x 64 from there, stepping down to tiles that fit). These
 * are names: a call that AUTO resolves by the heuristic runs the family at a
 * size chosen from nnz and R (about 3000 runs of 32 to 512 nonzeros) or, for
 * 3-mode short fibres, from the mean slice. A variant given by number runs as
 * named. */
int tentaco_csf_resolve_variant(const tentaco_csf* h, int R, int variant, int* out);

/* ---- CP-ALS around the batched MTTKRP ---------------------------------- */
/* The caller splatt_cpd_als stands in for (ds.h:395), for many tensors at
 * once. handles[t*5 + m] is tensor t's device CSF with mode m at its root
 * (NULL for m >= its order); level_modes[(t*5 + m)*5 + l] is the tensor mode
 * held at level l of that CSF (level 0 must be m). Factors start U[0,1) from
 * seed (as gen_factor_matrices, ds.h:386-409), lambda = 1. R in {16,32,64}. */
typedef struct tentaco_cpd tentaco_cpd;
int tentaco_cpd_create(tentaco_csf* const* handles, const int* level_modes, int ntensors,
                       int R, uint64_t seed, tentaco_cpd** out);
/* Autotune the batched MTTKRP of every mode step (not for capture). */
int tentaco_cpd_tune(tentaco_cpd* c, int reps);
/* `sweeps` ALS sweeps. Mode step m = 0..4: one batched MTTKRP over every
 * tensor of order > m (replayed from a hipGraph when use_graphs), then per
 * tensor A_m = M V^-1 with V the Hadamard product of the other Grams
 * (Cholesky in FP64), column normalisation into lambda (2-norm on the first
 * sweep ever, max(1, max |a|) after), and the new Gram. fits (optional,
 * ntensors entries) receives 1 - ||X - model|| / ||X|| after the last sweep.
 * stream NULL with use_graphs: a stream owned by the handle is used. */
int tentaco_cpd_iterate(tentaco_cpd* c, int sweeps, int use_graphs, void* stream,
                        double* fits);
/* Copy factor m of tensor t (dims x R) and its lambda (R) to the host. */
int tentaco_cpd_factor(const tentaco_cpd* c, int t, int m, float* factor, float* lambda);
/* Replace factor m of tensor t (its Gram is recomputed). */
int tentaco_cpd_set_factor(tentaco_cpd* c, int t, int m, const float* factor);
int tentaco_cpd_free(tentaco_cpd* c);

/* ---- learned variant selector ------------------------------------------ */
/* No reference counterpart: it replaces running the exhaustive sweep
 * (codegen.py:44-51 + ebsr_32_tune.sh / ebpr_*_tune.sh) for every tensor with
 * a prediction from the tensor's structure, trained on the sweep's own
 * timings; the sweep stays as the fallback and as the check on its picks. */
#define TENTACO_NUM_FEATURES 24
#define TENTACO_MLP_HIDDEN 64
/* The 24 features of an uploaded CSF at rank R:
 *   [0]      ln nnz
 *   [1..5]   ln dims[m], m = 0..4 (0 past the order)
 *   [6..10]  ln node count of level m, m = 0..4 (0 past the order)
 *   [11..22] for levels m = 1..4, three each: ln(1 + mean), ln(1 + variance),
 *            ln(1 + max) of the children per level m-1 node (0 past the order)
 *   [23]     ln R */
int tentaco_csf_features(const tentaco_csf* h, int R, float* features);

/* An FP32 MLP 24 -> 64 -> 64 -> n_out (ReLU) resident on the current device
 * (n_out <= 64; n_out = tentaco_num_variants() for selection). Outputs are
 * predicted ln(ms) per variant. Parameters (tentaco_mlp_num_params floats)
 * are W1[64][24] b1[64] W2[64][64] b2[64] W3[n_out][64] b3[n_out], row-major
 * [out][in]; create() draws He-normal weights from seed, zero biases.
 * Inputs are standardised as (x - x_mean) / x_std and outputs mapped back as
 * y * y_std + y_mean (set_scaling; identity until set). */
typedef struct tentaco_mlp tentaco_mlp;
int64_t tentaco_mlp_num_params(int n_out);
int tentaco_mlp_create(int n_out, uint64_t seed, tentaco_mlp** out);
int tentaco_mlp_free(tentaco_mlp* m);
int tentaco_mlp_set_scaling(tentaco_mlp* m, const float* x_mean, const float* x_std,
                            float y_mean, float y_std);
int tentaco_mlp_get_scaling(const tentaco_mlp* m, float* x_mean, float* x_std,
                            float* y_mean, float* y_std);
int tentaco_mlp_get_params(const tentaco_mlp* m, float* host, int64_t n);
int tentaco_mlp_set_params(tentaco_mlp* m, const float* host, int64_t n);
/* Gradients of the last loss_grad / training step (host copy). */
int tentaco_mlp_get_grads(const tentaco_mlp* m, float* host, int64_t n);
/* Inference kernel on device rows: x_dev n x 24 raw features -> y_dev
 * n x n_out predicted ln(ms), on `stream`. */
int tentaco_mlp_forward(tentaco_mlp* m, const float* x_dev, int n, float* y_dev,
                        void* stream);
/* Forward + backward kernels on host arrays x (n x 24), t (n x n_out target
 * ln(ms)) and mask (n x n_out, 1 = use): loss = sum mask * (y_s - t_s)^2 /
 * sum mask over the standardised prediction y_s and target t_s; the
 * gradients stay in the model (get_grads). Synchronous. */
int tentaco_mlp_loss_grad(tentaco_mlp* m, const float* x, const float* t,
                          const float* mask, int n, float* loss);
/* One Adam step (beta1, beta2, eps) with the stored gradients. */
int tentaco_mlp_adam(tentaco_mlp* m, float lr, float beta1, float beta2, float eps);
/* Training loop on the device: the set (host arrays as in loss_grad) is
 * uploaded once; each epoch shuffles it (seeded Fisher-Yates) into
 * minibatches of `batch`, each a gather, forward, backward and Adam kernel
 * (beta 0.9 / 0.999, eps 1e-8, step size lr with cosine decay over the run).
 * *final_loss = mean loss over the last epoch. Deterministic for a seed. */
int tentaco_mlp_train(tentaco_mlp* m, const float* x, const float* t, const float* mask,
                      int n, int epochs, int batch, float lr, uint64_t seed,
                      float* final_loss);
/* Pick: the variant with the smallest predicted time among those that fit an
 * order-`order` tensor at rank R; *margin = predicted runner-up / best - 1;
 * pred_ms (optional, n_out entries) = exp of the predictions. */
int tentaco_mlp_select(tentaco_mlp* m, int order, int R, const float* features,
                       int* variant, float* margin, float* pred_ms);
/* The same pick without margin or predictions: the variant-selection entry
 * point of the handle API (features from tentaco_csf_features). */
int tentaco_select_variant(tentaco_mlp* m, const float* features, int order, int R,
                           int* variant);
/* Attach a selector (not owned; NULL detaches) to a handle: AUTO on a rank
 * with no recorded choice then takes the selector's pick when its margin is
 * at least min_margin (0.03 = 3% with the shipped model) and records it
 * (source SELECTOR); below that it runs the fallback below. Under stream
 * capture the structural heuristic is used instead, since both would
 * synchronise. */
int tentaco_csf_set_selector(tentaco_csf* h, tentaco_mlp* m, float min_margin);
/* Fallback when the margin is under min_margin: k > 0 (4 by default) times
 * only the k best-predicted variants that fit and records the fastest
 * (source SELECTOR_TIMED), a fraction of the sweep's cost; 0 runs
 * tentaco_csf_autotune, the full sweep (source SWEEP). */
int tentaco_csf_set_selector_fallback(tentaco_csf* h, int top_k);

/* tentaco_mttkrp_dev issued `count` times back to back from the library's
 * own loop (the reference drivers' trial loop, mttkrp_csf_gpu.h:148, without
 * per-call host-language overhead between launches). */
int tentaco_mttkrp_dev_repeat(tentaco_csf* h, int R, const float* const* factors_dev,
                              float* A_dev, int32_t a_rows, int variant, void* stream,
                              int count);

/* MTTKRP for the mode held at CSF level `level` (1..order-1) of an uploaded
 * CSF, without a CSF rooted at that mode (one CSF for every mode instead of
 * one per mode): A(j,:) = sum over nonzeros whose level-`level` coordinate
 * is j of val * prod_{l != level} factors_dev[l](coordinate at level l, :).
 * factors_dev has order entries (the root level's factor included; the
 * entry for `level` is not read); A_dev has a_rows x R floats, a_rows above
 * the level's largest coordinate. Each level runs through a per-handle
 * transposed index of its nodes sorted by coordinate, built on the level's
 * first call outside stream capture or by tentaco_csf_reserve_level: 4 B
 * per coordinate plus, for the leaf level, 4 order B per nonzero up to order 3
 * and from there 8 B per nonzero and 4(order-1) B per level order-2 node, or,
 * for an inner level, 4 order B per level order-2
 * node. Every row is then written once, without atomics, bitwise
 * reproducible. A call captured before its level's index exists zero-fills
 * A and accumulates with FP32 atomics instead.
 * No reference counterpart: the reference builds one CSF per mode through
 * splatt (CSF_ONEMODE, ds.h:355-356). */
int tentaco_mttkrp_level_dev(tentaco_csf* h, int level, int R,
                             const float* const* factors_dev, float* A_dev,
                             int32_t a_rows, void* stream);
/* Build the transposed index tentaco_mttkrp_level_dev uses for `level`, so
 * that later calls allocate nothing (e.g. before graph capture).
 * Synchronizes the device. */
int tentaco_csf_reserve_level(tentaco_csf* h, int level);

/* TTV on device buffers: c_dev has the last mode's extent, A_dev has one
 * float per level N-2 node (nodes[N-2]). The first call on a handle (outside
 * stream capture) builds its TTV plan (a fibre-start bitmap, about nnz/8
 * bytes, and the window of c to cache in LDS) and synchronizes; later calls
 * allocate nothing and write each entry of A_dev once without atomics
 * (bitwise reproducible; empty fibres are written as zero). A call captured before
 * the plan exists uses the bracket kernel, which zero-fills A_dev and adds
 * the pieces of fibres that cross workgroups atomically. */
int tentaco_ttv_dev(tentaco_csf* h, const float* c_dev, float* A_dev,
                    void* stream);
/* The TTV plan's layout. When the last mode is wider than one LDS window of
 * c (38912 entries) and the best window would serve under 3/4 of the
 * gathers, the plan also builds a banded copy of the leaf level: the
 * nonzeros of each band of ceil(extent / nb) leaf coordinates in CSF order,
 * 6 bytes per nonzero (a 16-bit index in the band's window and the value)
 * plus 4 per (fibre, band) piece, so that every gather of
 * c is an LDS read; a last pass sums each fibre's pieces in band order (no
 * atomics, bitwise reproducible). bands: 0 picks (the default), 1 keeps one
 * window, 2..8 forces that many bands. A change takes effect at the next
 * TTV outside stream capture; the old plan's memory is kept until the
 * handle is freed (a graph captured earlier may read it). No counterpart in
 * the reference, whose TTV gathers c from global memory. */
int tentaco_csf_set_ttv_bands(tentaco_csf* h, int bands);
/* The layout the handle's TTV plan uses: bands = 0 (no plan yet or the
 * bracket kernel), 1 (one window) or the number of bands; device_bytes = the
 * banded copy's size (0 without one). Either pointer may be NULL. */
int tentaco_csf_ttv_layout(const tentaco_csf* h, int* bands, int64_t* device_bytes);

/* ---- batched persistent launch ----------------------------------------- */
/* Many MTTKRP tasks (e.g. every mode of every tensor of a CP-ALS sweep, one
 * CSF per mode ordering) in one persistent kernel: all tasks' nonzeros are cut
 * into equal work items that persistent workgroups pull from a device
 * counter, so uneven tensor sizes do not leave the GPU idle and the whole
 * batch costs two launches (the walk and its shared rows; long batches of
 * several orders one walk per order), or one graph launch. No
 * counterpart in the reference, which launches per tensor-mode
 * (mttkrp_csf_gpu.h:186-217). */
typedef struct tentaco_batch tentaco_batch;
/* tasks: ntasks device-resident CSFs (kept by pointer, must outlive the
 * batch); R in {16, 32, 64}. */
int tentaco_batch_create(tentaco_csf* const* tasks, int ntasks, int R,
                         tentaco_batch** out);
/* factors_dev: ntasks x 4 device pointers, task-major; slot m-1 of task t is
 * the factor of level m (slots past order-1 ignored). outs_dev[t] holds
 * out_rows[t] x R floats and is fully overwritten by each run. Builds each
 * task's row bitmap (one bit per output row: rows that root nodes with
 * nonzeros store, which are not zeroed) on the null
 * stream and synchronizes the device before returning. */
int tentaco_batch_set_operands(tentaco_batch* b, const float* const* factors_dev,
                               float* const* outs_dev, const int32_t* out_rows);
/* Tile configuration of every order group: family 1 (edge-parallel; the
 * batch runs that walk only, and family 0 returns TENTACO_EUNSUPPORTED,
 * since the edge-serial walk's per-group FP32 atomics lose accuracy on giant
 * slices), block in {128, 256, 512}, group = nonzeros per lane group. Drops
 * a captured graph. */
int tentaco_batch_configure(tentaco_batch* b, int family, int block, int group);
/* The tile and schedule (see tentaco_batch_set_schedule) of the tasks of one
 * tensor order (2..5) only; the groups may differ. Drops a captured graph. */
int tentaco_batch_configure_order(tentaco_batch* b, int order, int family, int block,
                                  int group, int schedule);
/* The tile and schedule an order group runs with. */
int tentaco_batch_get_config(const tentaco_batch* b, int order, int* family, int* block,
                             int* group, int* schedule);
/* Enqueue a run on `stream`. */
int tentaco_batch_run(tentaco_batch* b, void* stream);
/* Capture tentaco_batch_run into an instantiated hipGraph (kernels only). */
int tentaco_batch_capture(tentaco_batch* b, void* stream);
/* Launch the captured graph on `stream`. */
int tentaco_batch_launch(tentaco_batch* b, void* stream);
/* Work items, the largest persistent grid and the nonzeros per item of the
 * order group with the most items, in the current configuration. */
int tentaco_batch_items(const tentaco_batch* b, int32_t* items, int32_t* grid,
                        int32_t* nb);
/* Time every tile configuration for all orders at once (2 schedules x 3
 * blocks x 5 groups) and keep the fastest, returned in
 * best_family / best_block / best_group. Then time every tile and schedule of
 * each order group in turn with the other groups held, keeping what is
 * faster (tentaco_batch_get_config reads the result); best_ms is the final
 * time. Not for graph capture. */
int tentaco_batch_autotune(tentaco_batch* b, int reps, void* stream,
                           int* best_family, int* best_block, int* best_group,
                           float* best_ms);
int tentaco_batch_free(tentaco_batch* b);
/* How persistent workgroups take items, for every order group: 0 = from a
 * device work counter in arrival order (the default), 1 = static cyclic
 * assignment (item = block + k * grid, no shared counter). Kept across
 * configure(); autotune searches both, jointly and per order. get_schedule
 * reports the order group with the most items. */
int tentaco_batch_set_schedule(tentaco_batch* b, int schedule);
int tentaco_batch_get_schedule(const tentaco_batch* b, int* schedule);
/* Output rows no root node stores (rows of empty slices) must read zero
 * after every run. WRITTEN (the default): every run zeroes them. RETAINED:
 * they are zeroed once, when this mode is set and by every later
 * set_operands, and runs leave them alone; a run then writes only the rows
 * that nonzeros reach (stored by the walk, or zeroed and accumulated where
 * a slice crosses a work item). The result of every run is the same, as
 * long as nothing else writes the output buffers: after writing one, set
 * the mode again to refill. For outputs the caller owns exclusively (e.g.
 * one buffer per task across a loop of runs). Not a reference feature.
 * Drops a captured graph; synchronizes the device. */
#define TENTACO_BATCH_OUTPUTS_WRITTEN 0
#define TENTACO_BATCH_OUTPUTS_RETAINED 1
int tentaco_batch_set_output_mode(tentaco_batch* b, int mode);
int tentaco_batch_get_output_mode(const tentaco_batch* b, int* mode);

/* ---- stream-ordered host staging -------------------------------------- */
/* The replacement for the per-call cudaMalloc / H2D / kernel / D2H / free
 * round trip of copy_to_device_mttkrp / copy_from_device_mttkrp /
 * free_tensors_mttkrp (gpu_library.h:780-945). Operand arrays in pinned host
 * memory (tentaco_host_alloc) transfer by DMA without a staging copy and
 * overlap with work on other streams. */
int tentaco_host_alloc(void** ptr, size_t bytes);  /* hipHostMalloc, pinned */
int tentaco_host_free(void* ptr);
int tentaco_stream_create(void** stream);          /* default priority */
int tentaco_stream_destroy(void* stream);
int tentaco_stream_synchronize(void* stream);
/* tentaco_csf_upload with the copies enqueued on `stream` (validation runs on
 * the host first). B's arrays must stay valid until the stream has passed
 * the copies. */
int tentaco_csf_upload_async(const taco_tensor_t* B, int order, void* stream,
                             tentaco_csf** out);
/* MTTKRP from host operands into host A on a device-resident CSF: the
 * factors (levels 1..order-1, dimensions {rows, R}) are copied into device
 * buffers kept by the handle, the kernels run, and A is copied back, all
 * enqueued on `stream`; the call returns before they finish. The host arrays
 * must stay valid (and A unread) until the stream is synchronized. AUTO with
 * a selector may run a sweep, which synchronizes. Calls on one handle share
 * its buffers: order them on one stream. */
int tentaco_mttkrp_host_async(tentaco_csf* h, int R, taco_tensor_t* const* factors,
                              taco_tensor_t* A, int variant, void* stream);

/* Device memory helpers for hosts without their own HIP runtime binding. */
int tentaco_dev_malloc(void** ptr, size_t bytes);
int tentaco_dev_free(void* ptr);
int tentaco_memcpy_h2d(void* dst, const void* src, size_t bytes);
int tentaco_memcpy_d2h(void* dst, const void* src, size_t bytes);
int tentaco_dev_synchronize(void);

/* Read a 512 MiB device buffer (filled once, when first allocated) on
 * `stream` so the next kernel starts with cold caches holding only clean
 * lines: the GPU analog of Timer::clear_cache, which reads a large array
 * (timers.h:62-75). */
int tentaco_flush_cache(void* stream);
/* hipEvent timing of a device-API call sequence on `stream`: record start,
 * record stop + synchronize, elapsed ms. */
int tentaco_timer_start(void* stream);
int tentaco_timer_stop(void* stream, float* ms);

/* Kernel timer: while on, every call records a hipEvent pair on its launch
 * stream around its main kernel only (slice_kernel, slice_short_kernel,
 * slice_group_kernel, slice_pair_kernel, slice_pad_kernel, edge_kernel,
 * level_kernel, tleaf_kernel, inner_leaf_kernel, ttv_unit_kernel (both of its
 * forms), ttv_band_kernel, ttv_kernel, batch_kernel or copy_kernel; not the
 * partition/zero pre-pass or the passes that write FP64 rows), at most 4096
 * launches; never inside a stream capture. stop() turns it off and returns
 * the summed duration, the launch count and the last kernel's name. No
 * reference counterpart (GPUTimer, gpu_library.h:949-988, brackets the whole
 * region). */
int tentaco_ktimer_start(void);
int tentaco_ktimer_stop(double* total_ms, int* launches, char* kernel, int kernel_len);

/* Plain device-to-device copy (16-byte aligned, non-overlapping) through a
 * streaming copy kernel on `stream`: the known-size reference workload for
 * calibrating hardware byte counters, and a staging helper. */
int tentaco_dev_copy(void* dst, const void* src, size_t bytes, void* stream);
/* Random factor-row gathers on `stream`: `blocks` workgroups of 256 lanes,
 * each row group of R/4 lanes (16 from R = 64) reading iters x 8 rows of a
 * rows x R FP32 table at hashed indices, 8 in flight. *bytes receives the
 * bytes gathered. The calibration of the rate the MTTKRP walks' factor-row
 * gathers are bound by; R in {16, 32, 64}; out needs 4 bytes. */
int tentaco_dev_gather(const float* table, int64_t rows, int R, int32_t blocks, int iters,
                       float* out, void* stream, double* bytes);

/* ---- host-side CSF construction ---------------------------------------- */
/* An owned host CSF (dense root, int32 indices, FP32 values) with a
 * taco_tensor_t view. Replaces the reference's splatt load path
 * (read_tensor / to_taco_tensor / compress_top_level, ds.h:351-436). */
typedef struct tentaco_host_csf tentaco_host_csf;

/* FROSTT .tns reader (replaces splatt's load path, ds.h:351-366): one
 * nonzero per line, "i_1 ... i_N value", 1-based indices, '#' comment and
 * blank lines skipped; N = columns - 1 (2..5). dims_in (optional, N entries
 * in file mode order) fixes the dimensions, else each is the largest index.
 * Values are parsed as double and rounded to FP32; duplicates are summed in
 * file order. mode_order (optional) maps CSF level l to file mode
 * mode_order[l]; NULL = shortest mode first (ascending dimension, ties by
 * mode number), the splatt-like ordering. *order_out and mode_order_out
 * (N entries) report what was used. Malformed lines fail with EINVAL naming
 * the line. */
int tentaco_tns_read(const char* path, const int32_t* dims_in, const int* mode_order,
                     tentaco_host_csf** out, int* order_out, int* mode_order_out);

/* Lexicographic COO -> CSF: coords is order x nnz (mode-major, coords[m*nnz +
 * q]); duplicate coordinates are summed in input order (FP32); the root is
 * dense (pos = {0, dims[0]}, crd = 0..dims[0]-1). */
int tentaco_coo_to_csf(int order, const int32_t* dims, int64_t nnz,
                       const int32_t* coords, const float* vals,
                       tentaco_host_csf** out);

/* Synthetic CSF generator (deterministic in seed, independent of thread
 * count): root slice ids Zipf(slice_s) drawn without repetition until nnz is
 * reached; level-1 fan-out Zipf(fanout_s) over dims[1]; levels 2..N-2
 * fan-out round(lognormal(mid_mu, mid_sigma)); leaf fiber length
 * round(lognormal(leaf_mu, leaf_sigma)) capped at leaf_cap; distinct sorted
 * uniform children coordinates; values U[-1,1). The last fiber is truncated
 * so the tensor holds exactly nnz nonzeros when reachable. */
typedef struct tentaco_synth_params {
  int order;
  int32_t dims[5];
  int64_t nnz;
  double slice_s;
  double fanout_s;
  double mid_mu, mid_sigma;
  double leaf_mu, leaf_sigma;
  int32_t leaf_cap;
  uint64_t seed;
} tentaco_synth_params;
int tentaco_synth_csf(const tentaco_synth_params* p, tentaco_host_csf** out);

/* CSF of the same tensor with its modes in another order: level m of the
 * result is mode mode_order[m] of B (so mode_order[0] becomes the root and
 * the MTTKRP of that mode). Values travel with their coordinates; the
 * result is lexicographic with a dense root. B needs a valid dimensions
 * array and CSF levels (order given explicitly). */
int tentaco_csf_reorder(const taco_tensor_t* B, int order, const int* mode_order,
                        tentaco_host_csf** out);
/* View valid until tentaco_host_csf_free; order field is set. */
taco_tensor_t* tentaco_host_csf_view(tentaco_host_csf* h);
/* Number of nodes at a level (level order-1 = nonzeros), -1 if invalid. */
int64_t tentaco_host_csf_nodes(const tentaco_host_csf* h, int level);
int tentaco_host_csf_free(tentaco_host_csf* h);

#ifdef __cplusplus
} /* extern "C" */
#endif

#endif /* TENTACO_H */
