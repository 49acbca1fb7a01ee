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
// is the least power of two >= amax / 448, else amax / 448 itself; a block
// whose amax is 0 or NaN keeps scale 1.
int dsa_kv_quantize_rows(const uint16_t* kv, const uint16_t* k_rope, uint8_t* out, int64_t rows, int pow2,
                         void* stream);

#ifdef __cplusplus
}
#endif
