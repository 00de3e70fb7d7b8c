// rf_packed.h -- device helpers of the packed mtask kernels (emit_packed.py):
// four lanes per thread, a single-bit variable's four bytes (0 or 1 each, one
// per lane) as one 32-bit word.
#pragma once
#include <stdint.h>

#define RF_PK_ONE 0x01010101u

// Bytes 0xff for the lanes of [lane, lane + 4) that exist and are not done.
__device__ __forceinline__ uint32_t rf_pk_active(const uint8_t* done, uint32_t lane, uint32_t nlanes) {
    const uint32_t d = *reinterpret_cast<const uint32_t*>(done + lane);
    uint32_t m = 0;
    for (uint32_t j = 0; j < 4u; ++j)
        if (lane + j < nlanes && !((d >> (8u * j)) & 0xffu)) m |= 0xffu << (8u * j);
    return m;
}
// Bytes of b where m is 0xff, of a elsewhere.
__device__ __forceinline__ uint32_t rf_pk_sel(uint32_t m, uint32_t a, uint32_t b) { return (a & ~m) | (b & m); }
__device__ __forceinline__ uint32_t rf_pk_ld(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }
// FULL: every lane stores.
template <bool FULL>
__device__ __forceinline__ void rf_pk_st(uint8_t* p, uint32_t v, uint32_t m) {
    uint32_t* q = reinterpret_cast<uint32_t*>(p);
    *q = FULL ? v : rf_pk_sel(m, *q, v);
}
// Bit k of four lanes' words as bytes.
__device__ __forceinline__ uint32_t rf_pk_bit(const uint32_t (&w)[4], uint32_t k) {
    return ((w[0] >> k) & 1u) | ((w[1] >> k) & 1u) << 8 | ((w[2] >> k) & 1u) << 16 | ((w[3] >> k) & 1u) << 24;
}
// Four lanes' elements as 32-bit words: word h (0, 1) of 64-bit ones.
template <typename T>
__device__ __forceinline__ void rf_pk_words(const T* p, uint32_t h, uint32_t (&w)[4]) {
    for (uint32_t j = 0; j < 4u; ++j) w[j] = (uint32_t)((uint64_t)p[j] >> (32u * h));
}
// Element of lane j from packed single bits (bit k of it is byte j of b[k]).
template <typename T, int N>
__device__ __forceinline__ T rf_pk_gather(const uint32_t (&b)[N], uint32_t j) {
    T v = 0;
    for (int k = 0; k < N; ++k) v |= (T)((b[k] >> (8u * j)) & 1u) << k;
    return v;
}
