// Coalesced dequantization: raw GGUF blocks -> f32 or f16.
//
// Every value is computed with the reference's own expression and rounding
// order (src/dequant.rs:339-367 Q4_K `d1 * q - m1`, :414-444 Q6_K `d * sc * q`,
// :220-226 Q8_0 `q * d`), with FP contraction disabled, so the f32 output is
// bit-identical to the host dequantizer; the f16 output is the RNE rounding of
// that f32 value. Replaces `dequantize_{q4k,q6k}_coalesced{,_f16}_kernel`
// (src/kernels_cuda/gemv_q4k.cu:359-448) and `dequantize_q8_0_coalesced{,_f16}`
// (src/kernels_cuda/gemv_q8_0.cu:253-282).
//
// Bound: HBM, most of it the output. A lane takes a piece of P code bytes
// (P = 8 for f16, 4 for f32), so that each run of values it stores is 16 bytes
// and eight lanes write one 128-byte line. A K-quant byte holds two codes, so
// a piece gives two runs. A Q6_K table of 151936 x 1024 (439 MB with its f16
// output): 75 us = 5.85 TB/s, against 229 us for a lane per element, whose byte
// loads and 2-byte stores left the memory idle; as f32 109-149 us (750 MB).
// Non-temporal stores: the output does not fit the caches.
#pragma once
#include "common.hpp"

template <typename T>
RFXQ_DEV T store_cvt(float v);
template <> __device__ __forceinline__ float store_cvt<float>(float v) { return v; }
// The empty asm keeps the f32 value opaque so the narrowing is a plain RNE
// conversion: fusing the producing multiply into a mixed-precision mad with a
// +0 addend would turn -0.0 (a Q6_K block with d = 0) into +0.0.
template <> __device__ __forceinline__ half_t store_cvt<half_t>(float v) {
    asm volatile("" : "+v"(v));
    return (half_t)v;
}

// loads of blocks that are only 2-byte aligned, and stores of runs that are
// only aligned to their element (the unaligned access mode splits nothing on
// aligned addresses)
typedef uint32_t u1a2_t __attribute__((aligned(2)));
typedef uint32_t u2a2_t __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u4a2_t __attribute__((ext_vector_type(4), aligned(2)));
typedef _Float16 h8a2_t __attribute__((ext_vector_type(8), aligned(2)));
typedef float f4a4_t __attribute__((ext_vector_type(4), aligned(4)));

// code bytes per piece: the values of a 16-byte store
template <typename T>
constexpr uint32_t dq_piece() { return 16u / sizeof(T); }

// P code bytes (4 or 8) from a 2-byte-aligned address
template <uint32_t P>
RFXQ_DEV u2_t dq_load(const uint8_t* p) {
    if constexpr (P == 8u) return *(const RFXQ_GLOBAL u2a2_t*)p;
    else return u2_t{*(const RFXQ_GLOBAL u1a2_t*)p, 0u};
}
RFXQ_DEV uint32_t dq_byte(u2_t v, uint32_t i) { return (v[i >> 2] >> (8u * (i & 3u))) & 0xFFu; }

RFXQ_DEV void dq_store(half_t* y, const float (&v)[8]) {
    h8a2_t r;
#pragma unroll
    for (int i = 0; i < 8; i++) r[i] = store_cvt<half_t>(v[i]);
    __builtin_nontemporal_store(r, (RFXQ_GLOBAL h8a2_t*)y);
}
RFXQ_DEV void dq_store(float* y, const float (&v)[4]) {
    const f4a4_t r = {v[0], v[1], v[2], v[3]};
    __builtin_nontemporal_store(r, (RFXQ_GLOBAL f4a4_t*)y);
}

// Code bytes [o, o + P) of a Q4_K block's 128: the low nibbles are elements
// [0, P) from 64 (o / 32) + o % 32, the high ones 32 further on.
template <typename T>
RFXQ_DEV void dq_q4k_piece(const uint8_t* blk, uint32_t o, T* y) {
#pragma clang fp contract(off)
    constexpr uint32_t P = dq_piece<T>();
    const u2_t q = dq_load<P>(blk + 16u + o);
    const u4_t h = *(const RFXQ_GLOBAL u4a2_t*)blk;  // d, dmin, 12 scale bytes
    const uint32_t g = o >> 5, s = 8u * ((2u * g) & 3u);  // sub-blocks 2g, 2g + 1: bytes s/8, s/8 + 1
    // get_scale_min_k4 (src/dequant.rs:39-47) of both sub-blocks
    const uint32_t ys = h.y >> s, zs = h.z >> s, ws = h.w >> s;
    const bool up = g >= 2u;
    const uint32_t sc0 = up ? (ws & 0xFu) | (((ys >> 6) & 3u) << 4) : ys & 63u;
    const uint32_t mn0 = up ? ((ws >> 4) & 0xFu) | (((zs >> 6) & 3u) << 4) : zs & 63u;
    const uint32_t sc1 = up ? ((ws >> 8) & 0xFu) | (((ys >> 14) & 3u) << 4) : (ys >> 8) & 63u;
    const uint32_t mn1 = up ? ((ws >> 12) & 0xFu) | (((zs >> 14) & 3u) << 4) : (zs >> 8) & 63u;
    const float d = f16_bits_to_f32(h.x), dmin = f16_bits_to_f32(h.x >> 16);
    const float d0 = d * (float)sc0, m0 = dmin * (float)mn0, d1 = d * (float)sc1, m1 = dmin * (float)mn1;
    const u2_t lo = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
    float v0[P], v1[P];
#pragma unroll
    for (uint32_t i = 0; i < P; i++) {
        const float t0 = d0 * (float)dq_byte(lo, i), t1 = d1 * (float)dq_byte(hi, i);
        v0[i] = t0 - m0;
        v1[i] = t1 - m1;
    }
    y += 64u * g + (o & 31u);
    dq_store(y, v0);
    dq_store(y + 32, v1);
}

// ql bytes [o, o + P) of a Q6_K block's 128 (half n = o / 64, group t = o / 32
// % 2): the low nibbles are elements of group t, the high ones of group t + 2.
template <typename T>
RFXQ_DEV void dq_q6k_piece(const uint8_t* blk, uint32_t o, T* y) {
#pragma clang fp contract(off)
    constexpr uint32_t P = dq_piece<T>();
    const uint32_t n = o >> 6, t = (o >> 5) & 1u, l = o & 31u;
    const u2_t ql = dq_load<P>(blk + o), qh = dq_load<P>(blk + 128u + 32u * n + l);
    const uint8_t* sc = blk + 192u + 8u * n + (l >> 4) + 2u * t;
    const float d = f16_bits_to_f32(ld2(blk + 208));
    const float s0 = d * (float)(int8_t)sc[0], s1 = d * (float)(int8_t)sc[4];
    const u2_t c0 = (ql & 0x0F0F0F0Fu) | (((qh >> (2u * t)) & 0x03030303u) << 4);
    const u2_t c1 = ((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (2u * t + 4u)) & 0x03030303u) << 4);
    float v0[P], v1[P];
#pragma unroll
    for (uint32_t i = 0; i < P; i++) {
        v0[i] = s0 * (float)((int)dq_byte(c0, i) - 32);
        v1[i] = s1 * (float)((int)dq_byte(c1, i) - 32);
    }
    y += 128u * n + 32u * t + l;
    dq_store(y, v0);
    dq_store(y + 64, v1);
}

// codes [o, o + P) of a Q8_0 block's 32
template <typename T>
RFXQ_DEV void dq_q8_0_piece(const uint8_t* blk, uint32_t o, T* y) {
#pragma clang fp contract(off)
    constexpr uint32_t P = dq_piece<T>();
    const u2_t q = dq_load<P>(blk + 2u + o);
    const float d = f16_bits_to_f32(ld2(blk));
    float v[P];
#pragma unroll
    for (uint32_t i = 0; i < P; i++) v[i] = (float)(int8_t)dq_byte(q, i) * d;
    dq_store(y + o, v);
}

// grid-stride over pieces: 128 / P lanes per super-block, 32 / P per Q8_0 block
template <typename T, uint32_t TY>
RFXQ_DEV void dequant_body(const uint8_t* __restrict__ blocks, T* __restrict__ y, uint32_t num_blocks) {
    constexpr uint32_t P = dq_piece<T>();
    constexpr uint32_t per = (TY == TY_Q8_0 ? 32u : 128u) / P;
    const uint64_t total = (uint64_t)num_blocks * per;
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < total; i += (uint64_t)gridDim.x * 256u) {
        const uint64_t b = i / per;
        const uint32_t o = (uint32_t)(i % per) * P;
        if constexpr (TY == TY_Q4K) dq_q4k_piece(blocks + b * 144u, o, y + b * 256u);
        else if constexpr (TY == TY_Q6K) dq_q6k_piece(blocks + b * 210u, o, y + b * 256u);
        else dq_q8_0_piece(blocks + b * 34u, o, y + b * 32u);
    }
}

#define RFXQ_DEQUANT_ENTRY(NAME, T, TY) \
    extern "C" __global__ __launch_bounds__(256) void NAME(const uint8_t* b, T* y, uint32_t n) { dequant_body<T, TY>(b, y, n); }
RFXQ_DEQUANT_ENTRY(rfxq_dequant_q4k_f32, float, TY_Q4K)
RFXQ_DEQUANT_ENTRY(rfxq_dequant_q4k_f16, half_t, TY_Q4K)
RFXQ_DEQUANT_ENTRY(rfxq_dequant_q6k_f32, float, TY_Q6K)
RFXQ_DEQUANT_ENTRY(rfxq_dequant_q6k_f16, half_t, TY_Q6K)
RFXQ_DEQUANT_ENTRY(rfxq_dequant_q8_0_f32, float, TY_Q8_0)
RFXQ_DEQUANT_ENTRY(rfxq_dequant_q8_0_f16, half_t, TY_Q8_0)
