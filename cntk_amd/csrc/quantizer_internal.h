// Entry points that the shared library exports for its own tests and tuning runs.
// They are not part of the drop-in boundary and may change.
#pragma once

#include "../../include/cntk_amd_quantizer.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Forces kernel choices on a handle:
 *   quantize_path    0 = automatic, 1 = LDS column tile, 2 = tall-column (global re-read),
 *                    3 = one workgroup per column, column in LDS (fp32, rows a multiple of 4 up to 14336),
 *                    4 = one workgroup per column, column in registers, 16-byte accesses (below 32 (fp64: 64) bits; the
 *                        three matrices at the same offset within 16 bytes),
 *                    5 = the same with one element per access: fp32 any alignment, up to 98304 rows; fp64 256 threads per
 *                        column, 1025 to 6144 rows, below 64 bits, the bytes of path 1
 *                    6 = several workgroups per column, a strip of QWords each (below 32 (fp64: 64) bits, any height whose
 *                        strips number at most half of what the device holds of the kernel, any alignment)
 *                    7 = the same in two or three launches, each reading the matrix: any height of two strips or more (the
 *                        bytes of path 6)
 *   tile_gs          0 = automatic, else threads per column in the tile statistics phase (power of two, 8..256)
 *   unq_slots        0 = automatic, else bit positions decoded per thread by the QWord-major unquantize
 *   unq_mode         0 = automatic, 1 = QWord-major decoder with one store per value, 2 = tile decoder wherever it can run,
 *                    3 = automatic without the tile decoder, 4 = row-major decoder (packed column in LDS) wherever it can
 *                    run, 5 = row-major decoder that fetches its QWords itself wherever it can run, 6 = the same for short
 *                    columns (the matrix as one run of 16-byte groups) wherever it can run
 *   tile_stage       -1 = automatic, 0 = tile kernels write the residual straight to memory, 1 = through LDS */
int cntkq_debug_set_tuning(cntkq_quantizer* h, int quantize_path, unsigned tile_gs, unsigned unq_slots,
                           int unq_mode, int tile_stage);

/* How often a lane of a strip kernel (path 6) polls for another workgroup's partial sum before it gives up and raises the
 * error that the next cntkq_wait_quantize_done reports (UINT_MAX: as often as on a new handle). Zero makes every exchange fail at once while every kernel still
 * runs to its end: the way to test that error path. */
int cntkq_debug_set_strip_spin_limit(cntkq_quantizer* h, unsigned limit);

/* The largest scratch buffer of the strip kernels, in bytes, that the handle allocates from now on: a larger one is refused as if the
 * device had no memory left. */
int cntkq_debug_set_strip_scratch_limit(cntkq_quantizer* h, size_t bytes);

/* The most strips per column that the strip kernels (path 6) take on the handle's device at this bit width: half of what
 * the device holds of the kernel, as the runtime's occupancy query tells (a column of more strips than half a die holds
 * has them on all eight dies), never more than 8 x 128 (0: unknown, or no strip kernel for the bit width). A strip is
 * 512 / 1024 / 2048 QWords at 1 / 2 / 4 and more bits; of a double matrix 128 / 256 / 512 / 1024 at 1 / 2 / 4 / 8 and more. */
unsigned cntkq_debug_strip_max_strips(cntkq_quantizer* h, size_t nbits, int zero_threshold_for_1bit);
unsigned cntkq_debug_strip_max_strips_f64(cntkq_quantizer* h, size_t nbits, int zero_threshold_for_1bit);

/* Whether columns of this shape are quantized (workers == 0; _f64) or reduced by one thread each. Need no device. */
int cntkq_debug_short_columns(size_t rows, size_t cols, size_t nbits, size_t workers);
int cntkq_debug_short_columns_f64(size_t rows, size_t cols, size_t nbits);

/* The decoder (UnqKind, quantizer_kernels_batch.h) of an unquantize call on aligned matrices, the packed one in device memory or in
 * host memory that the kernels read themselves. Need no device. */
int cntkq_debug_decoder(size_t rows, size_t cols, size_t nbits, int packed_on_host);
int cntkq_debug_decoder_f64(size_t rows, size_t cols, size_t nbits, int packed_on_host);

/* Whether a short member of a set may be on lanes beside a column staged in memory and this many elements of other members. Needs no device. */
int cntkq_debug_lanes_beside_staged(size_t rows, size_t elements);

/* Whether an aligned stripe of a set is a member of the register grids, and the height up to which few tall columns of a set stay
 * staged in memory rather than have a register grid launched for them. Need no device. */
int cntkq_debug_stripe_shares_register_grid(size_t rows, size_t cols, size_t nbits, size_t workers);
size_t cntkq_debug_staged_max_rows(size_t nbits);

/* Bytes of the handle's device staging buffer: 0 until a packed matrix lay in host memory that the kernels do not write and
 * read themselves. */
size_t cntkq_debug_staging_bytes(const cntkq_quantizer* h);

/* Ties caller-owned hipEvent_t objects (either may be NULL) to the NEXT kernel this handle launches: start_event is
 * set when that kernel begins, stop_event when it has finished, by the dispatch itself. Used to time single kernels
 * without putting extra commands into the stream. The stop event also becomes what the matching Wait call waits on,
 * so it must stay alive until then. With a gradient-set call next: start_event at its first launch, stop_event at its
 * last, and the call's own completion event recorded on the stream behind that. */
int cntkq_debug_attach_events(cntkq_quantizer* h, void* start_event, void* stop_event);

#ifdef __cplusplus
}
#endif
