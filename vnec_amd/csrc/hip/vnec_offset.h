// vnec_offset.h — byte offsets into x that a kernel adds to its base address
// as 32 bits.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define VNEC_HD __host__ __device__ __forceinline__
#else
#define VNEC_HD static inline
#endif

// Part q (of part_bytes each) of row c of x, rows of row_bytes; x below 4 GiB.
// Unsigned throughout: from 2 GiB on the product does not fit an int.
VNEC_HD uint32_t vnec_x_offset(int32_t c, uint32_t row_bytes, int32_t q, uint32_t part_bytes)
{
    return (uint32_t)c * row_bytes + (uint32_t)q * part_bytes;
}
