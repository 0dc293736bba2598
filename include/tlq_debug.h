/* libtlq -- development interface: host-side self-checks of the kernels' address arithmetic and launch plans
 * (tlq_debug_*), the launch log, and the tuning hooks for benchmark sweeps and the autotuner (tlq_tune_*).
 *
 * None of this belongs to the operator boundary declared in tlq.h and nothing here has a counterpart in the reference's
 * generated `call(...)` interface: the reference's tile addressing is generated by TVM, and its tunables are the
 * block_M / block_N / block_K factory arguments (examples/dequantize_gemm/example_dequant_gemm_fine_grained.py:437,462)
 * and the autotuner's configurations (tilelang/autotuner/tuner.py:102-760), which here select among pre-built tilings.
 * The same shared library exports both sets of symbols; plain C types only, as in tlq.h. */
#ifndef TLQ_DEBUG_H_
#define TLQ_DEBUG_H_

#include "tlq.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Self-checks of the MFMA GEMM kernels' address arithmetic, evaluated on the HOST with the functions the kernels
 * themselves use (no GPU needed; the reference has no counterpart, its tile addressing is generated by TVM).
 * tlq_debug_check_gemm_addressing walks every tile, thread, load instruction and stage of one operand:
 * source_kind 0 = row-major [rows, row_bytes] operand copied global -> LDS directly in tiles of `tile` rows by
 * `threads` threads; 1 = int8 [K = rows, N = row_bytes] weights in tiles of `tile` (128 | 256 | 64) columns; 2 = 16-bit
 * [K = rows, N = row_bytes (the number of columns)] weights in tiles of 128 | 256 | 64 columns (N a multiple of 8; 64 for 512 threads).  It
 * checks global extents, LDS extents and coverage, agreement with the (transposing) operand-fragment reads and, for
 * kind 2, that no half-wavefront read meets a bank twice.
 * tlq_debug_check_slots_schedule simulates the five-slot kernel's issue / wait / barrier order over `stages` stages
 * with `loads_per_tile` load instructions per wavefront and tile (the kernel's waits assume 4).
 * tlq_debug_check_ring_schedule does so for the ring kernel's loads, waits, barriers, fragment reads and products over `stages` whole
 * stages; extra_in_flight is added to every wait's count of loads (0 = the kernel's own; more: to see it fail).
 * tlq_debug_check_quad_schedule does so for the four-wavefront kernel over `tiles` tiles of a work-group, two stages or more each; extra_start is
 * added to the wait ahead of the first tile, extra_stage to those of the stages.
 * All return 0 when everything holds, else 1 with tlq_last_error() naming the first violation. */
/* Launch log of the calling thread: tlq_debug_launch_log(1) clears it and starts recording, (0) stops; while it records,
 * every kernel launch of this thread's calls appends "entry point [kernel and variant]" (a repeated entry once), joined
 * by " + ".  tlq_debug_launch_log_text returns the text (valid until the thread's next call into the library).  For
 * benchmarks and tests that name the kernel they measured; no counterpart in the reference. */
void tlq_debug_launch_log(int on);
const char* tlq_debug_launch_log_text(void);
int tlq_debug_check_gemm_addressing(int source_kind, int64_t rows, int64_t row_bytes, int tile, int threads);
int tlq_debug_check_slots_schedule(int stages, int loads_per_tile);
int tlq_debug_check_ring_schedule(int stages, int loads_per_stage, int extra_in_flight);
int tlq_debug_check_quad_schedule(int stages, int tiles, int extra_start, int extra_stage);
/* The same walk for the streaming W4A16 kernel (TLQ_ALGO_STREAM): packed weights [N, K / 2] and 2-byte activations [M, K]
 * with 16 * activation_tiles rows per work-group (2 | 4 | 8), and its ring of `ring_depth` steps for 1 .. 40 steps. */
int tlq_debug_check_stream_addressing(int64_t M, int64_t N, int64_t K, int activation_tiles, int ring_depth);
/* Its schedule alone over a window of `steps` steps of `loads` load instructions and `units` units (8 with two groups of wavefronts, 4 with
 * four), with the kernel's own counts of loads that its waits leave outstanding (negative arguments) or others (to see them fail). */
int tlq_debug_check_stream_schedule(int steps, int depth, int loads, int units, int wait_scales, int wait_first, int wait_step);
/* Both orders of its work-groups: every block taken once; by XCD, hardly a slice on more XCDs than it needs. */
int tlq_debug_check_stream_order(int64_t n_blocks, int64_t slices, int64_t m_blocks);
/* The order of the GEMM kernels' work-groups by XCD: every place taken once, an XCD's places in a row. */
int tlq_debug_check_xcd_order(int64_t total);
/* The same walk for the panel kernel (TLQ_ALGO_PANEL) with K slices of `slice_steps` steps of 128 values: every direct load of
 * activations, packed weights and scale windows of every work-group, the LDS map and the operand reads; and the plan the
 * library would choose on a device with `cus` compute units: plan_out is a HOST array of four int64 that receives the tiles
 * along M and N, the K slices and the steps per slice; returns 1 when the kernel applies. */
int tlq_debug_check_panel_addressing(int64_t M, int64_t N, int64_t K, int64_t group, int slice_steps);
int tlq_debug_panel_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out);
/* The same two for the 256-row panel kernel (TLQ_ALGO_PANEL256); its walk also covers every scale / zero-point gather and plays the
 * schedule of loads, waits, barriers and LDS reads of a step through on the host. */
int tlq_debug_check_panel256_addressing(int64_t M, int64_t N, int64_t K, int64_t group, int slice_steps);
int tlq_debug_panel256_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out);
/* The schedule alone over `steps` steps, with the kernel's own wait counts (negative arguments) or others (to see them fail). */
int tlq_debug_check_panel256_schedule(int steps, int wait_w, int wait_a);
/* What the streaming kernel would take for a problem on a device with `cus` compute units: plan_out receives int64 activation rows and weight
 * rows per work-group, K slices, steps of 128 values per slice, estimated nanoseconds; returns 1 when it applies. */
int tlq_debug_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out);
/* What the small-tile kernel (one launch, wavefronts split K) would take for a problem: plan_out receives int64 activation rows and weight
 * rows per work-group, wavefronts, estimated nanoseconds; returns 1 when it applies. */
int tlq_debug_small_plan(int64_t M, int64_t N, int64_t K, int64_t group, void* plan_out);
/* The addresses and the ring of both small-tile kernels on the corner tiles of a problem.  kind as for tlq_debug_small_tile, 4 = W4A16 with
 * groups of `group` values (else ignored); row_bytes: bytes of K of an activation row; rows, cols: of a work-group's tile.  extra_in_flight is added to
 * every wait's count of loads (0 = the kernels' own; more: to see the walk fail). */
int tlq_debug_check_small_addressing(int kind, int64_t M, int64_t N, int64_t row_bytes, int64_t group, int rows, int cols, int waves, int extra_in_flight);
/* The middle-M panel kernel (TLQ_ALGO_PANELM): its plan (plan_out: int64 tiles_m, tiles_n, K slices, steps per slice, activation
 * rows per work-group). */
int tlq_debug_panelm_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out);
/* The host walk over every direct load, LDS cell and operand read of a launch with `rows` (64 or 128) activation rows per
 * work-group and K slices of `slice_steps` steps, and the play-through of its schedule of loads, waits, barriers and LDS
 * reads; the schedule alone with the kernel's own wait counts (negative arguments) or others (to see them fail). */
int tlq_debug_check_panelm_addressing(int64_t M, int64_t N, int64_t K, int64_t group, int rows, int slice_steps);
int tlq_debug_check_panelm_schedule(int rows, int steps, int window, int wait_w, int wait_a);

/* The same walk for the decode kernel (TLQ_ALGO_DECODE) launched as grid_x x chunks work-groups of `waves` wavefronts
 * with 16 * activation_tiles activation rows, and its ring for 2 .. 24 items; tlq_debug_decode_plan gives the geometry
 * the library would choose on a device with `cus` compute units: plan_out is a HOST array of five int64 that receives
 * activation tiles, chunks, wavefronts per work-group, grid_x and bytes of dynamic LDS; returns 1 when the kernel applies. */
int tlq_debug_check_decode_addressing(int64_t M, int64_t N, int64_t K, int64_t group, int activation_tiles, int chunks, int waves,
                                      int grid_x);
int tlq_debug_decode_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out);

/* Launch geometry the register-resident decode GEMV (M = 1, K <= 16384, power-of-two group) would use on a device with
 * `cus` compute units, computed on the host: plan_out is a HOST array of four int64 that receives rows per work-group,
 * work-groups, bytes of dynamic LDS and wavefronts per work-group.  Returns 1 when the kernel applies (its LDS stays
 * within the 64 KB a kernel may use without further set-up), 0 when the launcher falls back to the streaming GEMV,
 * -1 for bad arguments.  No counterpart in the reference. */
int tlq_debug_gemv_rows_plan(int64_t batch, int64_t N, int64_t K, int64_t group, int cus, void* plan_out);

/* The same for the ring kernel, which takes a single decode GEMV (M = 1, or 2 with fp16 activations; K <= 4096, a
 * multiple of 8 groups per row, 16-byte aligned scale / zero tensors) with every global read a direct global -> LDS load:
 * plan_out receives six int64:
 * load instructions per row, ring slots per wavefront, wavefronts per work-group, rows per work-group, work-groups and
 * bytes of dynamic LDS.  Returns 1 when the kernel applies, 0 when not, -1 for bad arguments.
 * tlq_debug_check_gemv_ring_addressing walks, on the host, every load of the first, middle and last work-groups of such a
 * launch (bounds of every global read and LDS write, coverage of the staging data and of the rows, ring order against the
 * kernel's wait counts); 0 = consistent.  No counterpart in the reference. */
/* Output tile (128 or 256, square) by machine fill, for `batch` problems of M x N outputs on the current device (256 CUs when there is none).  fused = 0: the
 * rule of the kernels whose weights pass through registers (16-bit [K, N] with N % 8 != 0, W4A8 unpacked into LDS) and of K slices added by atomics; the other
 * plain products go by tlq_debug_gemm_choice.  fused = 1: that of the fused W4A16 tile kernel.  Host only; no counterpart in the reference (its block_M / block_N are arguments,
 * example_dequant_gemm_fine_grained.py:437). */
int tlq_debug_gemm_tile(int64_t batch, int64_t M, int64_t N, int fused);
int tlq_debug_gemv_ring_plan(int64_t M, int64_t N, int64_t K, int64_t group, int cus, void* plan_out);
int tlq_debug_check_gemv_ring_addressing(int64_t M, int64_t N, int64_t K, int64_t group, int rows_per_block, int waves, int depth);

/* Tuning hooks for benchmark sweeps and the autotuner (each sets a value of the CALLING THREAD, read by that thread's
 * later launches; other threads keep the automatic choice; 0 = automatic choice).
 * They play the role of the reference's block_M / block_N / block_K factory arguments
 * (example_dequant_gemm_fine_grained.py:437,462), which here select among pre-built tilings. */
void tlq_tune_gemv(int rows_per_wave, int waves_per_block); /* rows 1|2|4 (negative: never the register-resident
                                                             * M = 1, K <= 4096 kernel), waves 1..4 (that kernel: 1..16) */
void tlq_tune_gemv_unroll(int blocks_per_cu);               /* resident blocks per CU the GEMV grid is sized for */
void tlq_tune_gemv_depth(int steps_in_flight);               /* load steps (1 KB per row each) a GEMV wavefront keeps in flight */
void tlq_tune_gemv_ring(int on);                             /* 1 (default): a single decode GEMV (1 or 2 activation rows) runs on the
                                                              * ring kernel where it applies; 0: on the kernels it replaced (for one
                                                              * activation row the same results, bit for bit) */
void tlq_tune_gemm_groups(int variant);                       /* the ring kernel in the place of 128-row tiles: 0 = automatic, 1 = never, 2 .. 5: its 128x128, 128x64, 64x128, 64x64 tiles */
/* The kernel and tile that a plain product of one launch gets, by its estimate in microseconds (a double, optional): 1 two-stage kernel 128x128, 2 .. 5 ring kernel
 * (tlq_tune_gemm_groups), 6 two-stage 256x256, 7 .. 11 four wavefronts (tlq_tune_gemm_quad), 12 the same 256x256.  kind: 0 16-bit weights [K, N], 1 [N, K], 2 int8
 * [K, N], 3 [N, K].  0: bad arguments. */
int tlq_debug_gemm_choice(int kind, int64_t batch, int64_t M, int64_t N, int64_t K, void* us_out);
void tlq_tune_gemm_quad(int variant);                         /* the kernel on four wavefronts, tiles other than 256x256: 0 = automatic, 1 = never, 7 .. 11: its
                                                              * 192x256, 128x256, 256x128, 192x128, 128x128 tiles wherever they can run */
void tlq_tune_gemm_band(int tile_rows);                       /* tile rows per band of the MFMA kernels' tile order (default 4) */
void tlq_tune_gemm_tile(int tile);                            /* square tile of the plain 16-bit GEMM (and of the second of the two W4A16 passes):
                                                              * 128 | 256, 0 = by the number of output tiles */
void tlq_tune_gemm_slots(int mode);                          /* 256 x 256 tiles of whole 128-byte stages of K: 1 (default) by the number of stages and
                                                              * tiles, 0 the two-stage kernel, 2 the one that cuts LDS into five operand-tile slots
                                                              * (by itself int8, short rows, several batches of up to 2048 rows), 3 the one on four
                                                              * wavefronts (long rows by itself), each wherever it can run */
void tlq_tune_w4a16_decode(int on);                          /* 0: the decode kernel is never picked automatically */
void tlq_tune_w4a16_stream(int on);                          /* 0: tlq_gemm_w4a16_ws never picks the streaming kernel by itself */
void tlq_tune_w4a16_stream_tiles(int tiles);                 /* 16-row activation tiles per work-group of the streaming kernel, 2, 4, 6 or 8, + 16 for four groups of wavefronts over K (128 weight rows per work-group) instead of two (256); 0 = by its estimate */
void tlq_tune_w4a16_stream_slice(int steps);                 /* K slice of the streaming kernel in steps of 128 values (0 = by its estimate) */
void tlq_tune_w4a16_panel(int mode);                         /* tlq_gemm_w4a16_ws, large M: 0 = automatic, otherwise a panel kernel is never picked automatically */
void tlq_tune_w4a16_panelm_rows(int rows);                   /* activation rows per work-group of the middle-M panel kernel: 64, 128, 0 = its plan's */
void tlq_tune_w4a16_panel_slice(int steps);                  /* K slice of the panel kernels in steps of 128 values (0 = their own plan) */
void tlq_tune_w4a16_tile(int block_m);                      /* 16|32|64|128|256 */
void tlq_tune_w4a16_split(int slices);                       /* K slices of the tile kernel, 16 < M < 256 with a workspace */
void tlq_tune_w4a16_skinny(int waves, int row_tiles);       /* wavefronts per group 1..16; 16-row weight tiles per work-group 1|2|4, +100*(1|2|4):
                                                               16-row activation tiles, +10 = never the small-tile kernel, +20 = that
                                                               kernel whenever it applies */
void tlq_tune_small(int waves, int tiles);                  /* the small-tile kernel of the int8, W4A8 and plain 16-bit products: tiles =
                                                               10 * activation tiles + weight tiles (1|2|4 each), < 0 = never; 0, 0 = by estimate */
/* What that kernel would take: kind 0 weights [N, K] (int8), 1 int8 [K, N], 2 16-bit [K, N], 3 packed int4 [N, K / 2]; row_bytes: bytes of K of an
 * activation row; plan_out as in tlq_debug_small_plan. */
int tlq_debug_small_tile(int kind, int64_t batch, int64_t M, int64_t N, int64_t row_bytes, void* plan_out);
void tlq_tune_i8_tile(int block_m);                         /* 32|128|256 */
void tlq_tune_f16_split(int slices);                        /* K slices of tlq_gemm_f16_ws: 0 = automatic, 1 = never, n = up to n */
int tlq_debug_f16_split(int64_t M, int64_t N, int64_t K);  /* K slices tlq_gemm_f16_ws takes for one batch of this shape */
void tlq_tune_w4a8_ws(int mode);                            /* tlq_gemm_w4a8_ws: 0 = automatic, 1 = K slices in the workspace, 2 = unpack + int8 GEMM */
void tlq_tune_i8_split(int slices);                         /* K slices of the one-batch int8 kernels: 0 = automatic, 1 = never, n = up to n */
int tlq_debug_i8_split(int64_t M, int64_t N, int64_t K, int buffers); /* K slices taken for one batch of this shape: with a matrix per
                                                                      * slice (1, tlq_gemm_w8a8_ws) or atomic adds into C (0, tlq_gemm_i8) */

#ifdef __cplusplus
}
#endif
#endif /* TLQ_DEBUG_H_ */
