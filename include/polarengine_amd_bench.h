/*
 * Measurement helpers of libpolarengine_amd.so (no counterpart in the
 * reference): the plain HBM streaming read and copy that bench.py times beside
 * the quantized linear, as the measured bandwidth ceiling of the part, and the
 * form that a product takes.
 * Same conventions as polarengine_amd.h: device pointers, byte sizes, a
 * hipStream_t, int status; nothing is allocated and nothing synchronises.
 */
#ifndef POLARENGINE_AMD_BENCH_H
#define POLARENGINE_AMD_BENCH_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Bytes of the sink buffer pe_stream_read needs for `bytes` of input. */
size_t pe_stream_read_sink_bytes(int64_t bytes);

/*
 * Read `bytes` (a multiple of 16, 16-byte aligned) of device memory with
 * 128-bit non-temporal loads, 8 KB per 256-lane workgroup. A lane writes its
 * folded word to `sink` only if it equals `magic` (pass a value the data does
 * not produce): the loads stay, the writes are (almost) none.
 */
int pe_stream_read(const void* src, int64_t bytes, void* sink, uint32_t magic, void* stream);

/*
 * The form that pe_linear_forward_xtf takes for these arguments (out_f32: that
 * pe_polar_matmul takes at M > 1): form[0] = 0 small-M kernel, 1 eight-wave
 * GEMM, 2 four-wave GEMM, form[1] x form[2] the GEMM's tile rows and columns,
 * form[3] the K groups; all -1 for the decode kernel. Host arithmetic only.
 */
int pe_linear_xtf_form(int64_t M, int in_f_padded, int out_f, int bits, int packed, int out_f32,
                       int* form);

/* dst[0:bytes] = src[0:bytes] (a multiple of 16; both 16-byte aligned). */
int pe_copy(void* dst, const void* src, int64_t bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif
