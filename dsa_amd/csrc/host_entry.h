// Entry points that only this package's Python layer calls (dsa_amd/_lib.py:
// PRIVATE_SIGNATURES).  Same conventions as include/dsa_mi355x.h (device
// pointers, a stream, 0 / < 0 / > 0 status with dsa_last_error), but not part
// of the installed C ABI: they may change with the package.
#pragma once
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

// fp8 cache rows (656 bytes, see dsa_fwd_options.kv_format) of `rows` bf16
// rows: kv [rows, 512] (16-byte aligned), k_rope [rows, 64] (4-byte aligned),
// out [rows, 656] (16-byte aligned).  pow2 != 0: each 128-wide block's scale
// is the least power of two >= amax / 448, else amax / 448, both as tensor code
// computes them on the GPU: the quotient as a product with the rounded
// reciprocal, 2^k beyond |k| = 15 as powf gives it (some units in the last
// place off for some k).  A block whose amax is 0 or NaN keeps scale 1.
int dsa_kv_quantize_rows(const uint16_t* kv, const uint16_t* k_rope, uint8_t* out, int64_t rows, int pow2,
                         void* stream);

// The bf16 rows of an fp8 cache: in [B * L, 656] or, with a block table (int32
// [B, max_blocks], L = max_blocks * block_size), a pool of num_blocks *
// block_size rows; kv [B * L, 512] (16-byte aligned), k_rope [B * L, 64].
// Rows behind an entry outside [0, num_blocks) become zeros.
int dsa_kv_expand_rows(const uint8_t* in, uint16_t* kv, uint16_t* k_rope, int B, int L, const int32_t* block_table,
                       int max_blocks, int block_size, int num_blocks, void* stream);

// dsa_bucket_indices for a paged cache whose rows are about to be addressed
// without the block table: the same partition of idx [B * SQ, TOPK], with
// every slot whose block entry lies outside [0, num_blocks) masked (-1).
int dsa_bucket_indices_paged(const int32_t* idx, int32_t* out, int B, int SQ, int TOPK, int L,
                             const int32_t* block_table, int max_blocks, int block_size, int num_blocks,
                             void* stream);

#ifdef __cplusplus
}
#endif
