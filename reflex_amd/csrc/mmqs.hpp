// Few-row GEMM Y = X . W^T (up to 32 rows) on f16 MFMAs: the fused few-row
// form (the reference stages up to 16 rows in its GEMV kernels,
// src/kernels_cuda/gemv_q4k.cu:64-138, gemv_q8_0.cu:74-170), with each weight
// read once for all rows.
//
// Bound: the weight stream from HBM. A workgroup takes 256 weight columns (64
// per wave) and a range of at most kMaxSb super-blocks of K, whose activations
// (all rows of the range) it holds in LDS as f16, so the loop over the range
// has no barrier and no activation copies: each wave streams its own columns'
// raw blocks into registers a whole super-block (9-17 KB a wave) ahead of
// their use (ranges of one super-block, which a narrow matrix is cut into, ask
// for theirs once and wait). The activations come straight from f32 (each workgroup converts
// its range: no activation launch; a row's power-of-two scale is then the
// range's, under which no value keeps fewer bits, and those that the row's scale
// would make f16-subnormal keep more) or from the f16 layout (quant.hpp).
// Operands and the order of additions are the tile kernels' (mmqh.hpp), so for
// the same split of K the results are theirs where the row's scale leaves every
// value f16-normal (or zero).
#pragma once
#include "common.hpp"
#include "mmq.hpp"
#include "mmqh.hpp"
#include "quant.hpp"

#define RFXQ_MEMBER __device__ __forceinline__

namespace mmqs {
constexpr uint32_t kMaxSb = 8;  // super-blocks of a workgroup's range

// LDS: activations [rows][nsb * 256] f16 (rows 16 bytes further apart: the
// operand reads of 16 rows cover all banks), Sx records [rows][nsb][16] f16,
// 32 row scales. The rows' results pass through the front of it at the end.
typedef float f2v_t __attribute__((ext_vector_type(2)));
struct Lds {
    uint8_t* x;
    uint8_t* sx;
    float* sc;
    uint32_t xs;  // bytes of an activation row
};
RFXQ_DEV Lds lds_of(uint8_t* base, uint32_t rows, uint32_t nsb) {
    const uint32_t xs = nsb * 512u + 16u;
    return {base + 128u, base + 128u + rows * xs, reinterpret_cast<float*>(base), xs};
}

// f32 rows [m][k] of super-blocks [sb0, sb0 + nsb) -> LDS. Wave w takes rows
// w + 4i, i < 4, of up to eight super-blocks or, in ranges of up to four, i < 8
// (the second four in the upper half of v), four values a lane and super-block,
// all loads in flight together. The arithmetic is rfxq_act_f16's with the
// scale of the range's maximum.
struct StageF32 {
    float4 v[4][kMaxSb];
    // row and super-block (of the range) of v[i][s]
    RFXQ_MEMBER static uint32_t row(uint32_t w, uint32_t i, uint32_t s, uint32_t nsb) { return w + 4u * i + (s >= 4u && nsb <= 4u ? 16u : 0u); }
    RFXQ_MEMBER static uint32_t sb(uint32_t s, uint32_t nsb) { return nsb <= 4u ? s & 3u : s; }
    RFXQ_MEMBER void load(const MmqDesc& ds, uint32_t w, uint32_t sb0, uint32_t nsb) {
        const float* x = reinterpret_cast<const float*>(ds.xq) + 256u * sb0 + 4u * (threadIdx.x & 63u);
#pragma unroll
        for (uint32_t s = 0; s < kMaxSb; s++)
            if (sb(s, nsb) < nsb)
#pragma unroll
                for (uint32_t i = 0; i < 4u; i++)
                    if (row(w, i, s, nsb) < ds.m) v[i][s] = ldf4(x + (uint64_t)row(w, i, s, nsb) * ds.k + 256u * sb(s, nsb));
    }
    RFXQ_MEMBER void put(const MmqDesc& ds, uint32_t w, uint32_t nsb, const Lds& L) const {
        const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            float mx[2] = {0.0f, 0.0f};
#pragma unroll
            for (uint32_t s = 0; s < kMaxSb; s++)
                if (sb(s, nsb) < nsb && row(w, i, s, nsb) < ds.m) mx[s >> 2] = fmaxf(mx[s >> 2], absmax4(v[i][s]));
            if (nsb > 4u) mx[0] = mx[1] = fmaxf(mx[0], mx[1]);
#pragma unroll
            for (uint32_t hf = 0; hf < 2u; hf++) {
                const uint32_t r = row(w, i, 4u * hf, nsb);
                if (r >= ds.m || sb(4u * hf, nsb) >= nsb) continue;
                const int e = act_f16_exp(mx[hf]);
                const float scale = ldexpf(1.0f, -e);
                if (lane == 0u) L.sc[r] = ldexpf(1.0f, e);
#pragma unroll
                for (uint32_t s = 4u * hf; s < 4u * hf + 4u; s++) {
                    const uint32_t b = sb(s, nsb);
                    if (b >= nsb) continue;
                    const h2_t ac = __builtin_convertvector(f2v_t{v[i][s].x * scale, v[i][s].z * scale}, h2_t);
                    const h2_t bd = __builtin_convertvector(f2v_t{v[i][s].y * scale, v[i][s].w * scale}, h2_t);
                    *reinterpret_cast<u2_t*>(L.x + r * L.xs + 512u * b + 8u * lane) = u2_t{h2_bits(ac), h2_bits(bd)};
                    const float t = group_sum<8>((((float)ac.x + (float)bd.x) + (float)ac.y) + (float)bd.y);
                    if ((lane & 7u) == 0u) {
                        half_t* rec = reinterpret_cast<half_t*>(L.sx + 32u * (r * nsb + b)) + (lane >> 3);
                        const half_t hi = (half_t)t, lo = (half_t)(t - (float)hi);
                        rec[0] = hi;
                        rec[8] = lo;
                    }
                }
            }
        }
    }
};

// the f16 layout's rows (gathered through ds.rows when set) -> LDS
RFXQ_DEV void stage_f16(const MmqDesc& ds, uint32_t sb0, uint32_t nsb, const Lds& L) {
    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63u;
    for (uint32_t r = w; r < ds.m; r += 4u) {
        const uint32_t sr = mmqh::act_row(ds, r);
        const uint8_t* x = reinterpret_cast<const uint8_t*>(ds.xq) + (uint64_t)sr * ds.ldq + 512u * sb0;
        const uint8_t* sx = reinterpret_cast<const uint8_t*>(ds.xds) + (uint64_t)sr * (ds.k / 8u) + 32u * sb0;
        for (uint32_t c = lane; c < 32u * nsb; c += 64u) *reinterpret_cast<u4_t*>(L.x + r * L.xs + 16u * c) = ld16(x + 16u * c);
        if (lane < 2u * nsb) *reinterpret_cast<u4_t*>(L.sx + 32u * r * nsb + 16u * lane) = ld16(sx + 16u * lane);
        if (lane == 0u) L.sc[r] = ds.xrs[sr];
    }
}

// ---------------------------------------------------------------- weights
//
// A wave's 64 columns (two 32-column n-tiles j) of one super-block, raw, in
// registers, and the weight operands built from them (mmqh.hpp's). op(g, t, j)
// is step t = 2e + s2 of stage g; xofs(g, t) the byte offset of that step's
// activations in the super-block's 512 bytes (the lane half's 32h included by
// the caller).

struct W4 {  // Q4_K
    static constexpr uint32_t kBytes = 144;
    u4_t q[2][2][2], h[2];  // raw: [stage pair][j][load A, B], headers
    u4_t dsc[2], cop[2];
    u4_t cur[2][4];  // the stages' operands bytes (after the lane swap)
    uint32_t mlo, mhi, mg;
    RFXQ_MEMBER void init() {
        mlo = 0x000F000Fu, mhi = 0x00F000F0u, mg = 0x64006400u;
        asm("" : "+v"(mlo), "+v"(mhi), "+v"(mg));
    }
    // lane offsets: mmqh_q4k_rows' (load A: 16 columns x 64 bytes, B 16 columns on)
    uint32_t g_q[2], g_h[2], g_b;
    RFXQ_MEMBER void place(uint32_t w, uint32_t row_bytes, uint32_t) {
        const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u, hh = lane >> 5;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            g_h[j] = (64u * w + 32u * j + l32) * row_bytes;
            g_q[j] = (64u * w + 32u * j + (l32 & 15u)) * row_bytes + 16u + 32u * (l32 >> 4) + 16u * hh;
        }
        g_b = 16u * row_bytes;
    }
    RFXQ_MEMBER void load(rsrc_t r, uint32_t sb) {
#pragma unroll
        for (int j = 0; j < 2; j++) h[j] = __builtin_amdgcn_raw_buffer_load_b128(r, g_h[j], 144u * sb, 0);
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                q[p][j][0] = __builtin_amdgcn_raw_buffer_load_b128(r, g_q[j], 144u * sb + 64u * p, 0);
                q[p][j][1] = __builtin_amdgcn_raw_buffer_load_b128(r, g_q[j] + g_b, 144u * sb + 64u * p, 0);
            }
    }
    RFXQ_MEMBER void take() {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            mmqh::q4k_sb_operands(h[j], cop[j], dsc[j]);
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const auto r = __builtin_amdgcn_permlane16_swap(q[p][j][0][d], q[p][j][1][d], false, false);
                    cur[j][2 * p][d] = r[0];
                    cur[j][2 * p + 1][d] = r[1];
                }
        }
    }
    static constexpr uint32_t xofs(int g, int t) { return 128u * g + 64u * (t >> 1) + 16u * (t & 1); }
    RFXQ_MEMBER u4_t op(int g, int t, int j) const {
        const int u = 2 * (t & 1);
        const uint32_t a = cur[j][g][u], b = cur[j][g][u + 1];
        if (t >> 1) return mmqh::q4k_codes_f16<1>(a, b, a >> 8, b >> 8, mmqh::splat16<1>(dsc[j][g]), mhi, mg);
        return mmqh::q4k_codes_f16<0>(a, b, a >> 8, b >> 8, mmqh::splat16<0>(dsc[j][g]), mlo, mg);
    }
};

struct W6 {  // Q6_K
    u4_t ql[4][2], qh[2][2], s[2];
    uint32_t d[2];
    u4_t cl[4][2], ch[2][2], mult[2];
    uint32_t mla, mqa, mlb, mqb, mg, g_c[2], hh, sh;
    RFXQ_MEMBER void init() {
        mla = 0x000F000Fu, mqa = 0x00300030u, mlb = 0x00F000F0u, mqb = 0x03000300u, mg = 0x64006400u;
        asm("" : "+v"(mla), "+v"(mqa), "+v"(mlb), "+v"(mqb), "+v"(mg));
    }
    RFXQ_MEMBER void place(uint32_t w, uint32_t row_bytes, uint32_t sh0) {
        const uint32_t lane = threadIdx.x & 63u;
        hh = lane >> 5;
        sh = sh0;
#pragma unroll
        for (int j = 0; j < 2; j++) g_c[j] = (64u * w + 32u * j + (lane & 31u)) * row_bytes + 16u * hh;
    }
    RFXQ_MEMBER void load(rsrc_t r, uint32_t sb) {
        const uint32_t base = 210u * sb + sh;
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int g = 0; g < 4; g++) ql[g][j] = __builtin_amdgcn_raw_buffer_load_b128(r, g_c[j], base + 32u * g, 0);
#pragma unroll
            for (int n = 0; n < 2; n++) qh[n][j] = __builtin_amdgcn_raw_buffer_load_b128(r, g_c[j], base + 128u + 32u * n, 0);
            s[j] = __builtin_amdgcn_raw_buffer_load_b128(r, g_c[j] - 16u * hh, base + 192u, 0);
            d[j] = __builtin_amdgcn_raw_buffer_load_b16(r, g_c[j] - 16u * hh, base + 208u, 0);
        }
    }
    RFXQ_MEMBER void take() {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            mult[j] = mmqh::q6k_multipliers(s[j], d[j], hh);
#pragma unroll
            for (int g = 0; g < 4; g++) cl[g][j] = ql[g][j];
#pragma unroll
            for (int n = 0; n < 2; n++) ch[n][j] = qh[n][j];
        }
    }
    static constexpr uint32_t xofs(int g, int t) { return 256u * (g >> 1) + 64u * (g & 1) + 128u * (t >> 1) + 16u * (t & 1); }
    RFXQ_MEMBER u4_t op(int g, int t, int j) const {
        const int n = g >> 1, b = g & 1, u = 2 * (t & 1);
        const uint32_t l0 = cl[g][j][u], l1 = cl[g][j][u + 1], h0 = ch[n][j][u], h1 = ch[n][j][u + 1];
        const uint32_t m = mult[j][2 * n + (t >> 1)];
        const uint32_t sm = b ? mmqh::splat16<1>(m) : mmqh::splat16<0>(m);
        const uint32_t qa0 = b ? h0 << 2 : h0 << 4, qa1 = b ? h1 << 2 : h1 << 4;
        const uint32_t qb0 = b ? h0 >> 6 : h0 >> 4, qb1 = b ? h1 >> 6 : h1 >> 4;
        if (t >> 1) return mmqh::q6k_codes_f16<1>(l0, l1, l0 >> 8, l1 >> 8, qa0, qa1, qb0, qb1, sm, mlb, mqb, mg);
        return mmqh::q6k_codes_f16<0>(l0, l1, l0 >> 8, l1 >> 8, qa0, qa1, qb0, qb1, sm, mla, mqa, mg);
    }
};

struct W8 {  // Q8_0: eight blocks per 256 values
    u4_t q[4][2][2];
    uint32_t d[4][2][2];
    u4_t c[4][2][2];
    uint32_t cd[4][2][2];
    uint32_t mg, sgn, g_c[2], hh, sh;
    bool al;  // the weights start on a dword: a block pair's codes are read with aligned loads
    RFXQ_MEMBER void init() {
        mg = 0x64646464u, sgn = 0x80808080u;
        asm("" : "+v"(mg), "+v"(sgn));
    }
    RFXQ_MEMBER void place(uint32_t w, uint32_t row_bytes, uint32_t sh0) {
        const uint32_t lane = threadIdx.x & 63u;
        hh = lane >> 5;
        sh = sh0;
        al = sh0 == 0u;
#pragma unroll
        for (int j = 0; j < 2; j++) g_c[j] = (64u * w + 32u * j + (lane & 31u)) * row_bytes;
    }
    RFXQ_MEMBER void load(rsrc_t r, uint32_t sb) {
        const uint32_t e_off = hh ? 0u : 32u;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t o = 272u * sb + 68u * g + sh;  // the stage's block pair
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if (al) {
                    q[g][j][0] = __builtin_amdgcn_raw_buffer_load_b128(r, g_c[j] + 16u * hh, o, 0);
                    d[g][j][0] = __builtin_amdgcn_raw_buffer_load_b32(r, g_c[j] + 16u * hh, o + 16u, 0);
                    q[g][j][1] = __builtin_amdgcn_raw_buffer_load_b128(r, g_c[j] + 16u * hh, o + 36u, 0);
                    d[g][j][1] = __builtin_amdgcn_raw_buffer_load_b32(r, g_c[j] + e_off, o, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        q[g][j][e] = __builtin_amdgcn_raw_buffer_load_b128(r, g_c[j] + 2u + 16u * hh, o + 34u * e, 0);
                        d[g][j][e] = __builtin_amdgcn_raw_buffer_load_b16(r, g_c[j], o + 34u * e, 0);
                    }
                }
            }
        }
    }
    RFXQ_MEMBER void take() {
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if (al) {
                    const u4_t a = q[g][j][0];
                    const uint32_t b = d[g][j][0], e = d[g][j][1];
                    c[g][j][0] = u4_t{alignbyte(a.y, a.x, 2u), alignbyte(a.z, a.y, 2u), alignbyte(a.w, a.z, 2u),
                                      alignbyte(b, a.w, 2u)};
                    c[g][j][1] = q[g][j][1];
                    cd[g][j][0] = mmqh::splat16<0>(hh ? e : a.x);
                    cd[g][j][1] = mmqh::splat16<1>(hh ? b : e);
                } else {
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        c[g][j][e] = q[g][j][e];
                        cd[g][j][e] = mmqh::splat16<0>(d[g][j][e]);
                    }
                }
            }
    }
    static constexpr uint32_t xofs(int g, int t) { return 128u * g + 64u * (t >> 1) + 16u * (t & 1); }
    RFXQ_MEMBER u4_t op(int g, int t, int j) const {
        const int e = t >> 1, u = 2 * (t & 1);
        const u2_t lo = mmqh::q80_codes_f16(c[g][j][e][u] ^ sgn, as_h2(cd[g][j][e]), mg);
        const u2_t hi = mmqh::q80_codes_f16(c[g][j][e][u + 1] ^ sgn, as_h2(cd[g][j][e]), mg);
        return u4_t{lo.x, lo.y, hi.x, hi.y};
    }
};

// the range [sb0, sb0 + nsb) of one tile's 256 columns
template <class W, uint32_t TY>
RFXQ_DEV void tile(const MmqDesc& ds, uint32_t n0, uint32_t ks, uint8_t* lds) {
    using namespace mmqh;
    constexpr uint32_t bb = TY == TY_Q4K ? 144u : TY == TY_Q6K ? 210u : 272u;  // bytes per 256 values
    const uint32_t tid = threadIdx.x, lane = tid & 63u, l32 = lane & 31u, h = lane >> 5;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t tot = ds.k / 256u, sb0 = ks * ds.sb_per_split, nsb = min(tot - sb0, ds.sb_per_split);
    const uint32_t row_bytes = tot * bb;
    // weights: the dword at or below the tile's first column; columns past the matrix read zeros
    const uintptr_t wa = reinterpret_cast<uintptr_t>(ds.w + (uint64_t)n0 * row_bytes);
    const uint32_t sh0 = (uint32_t)(wa & 3u);
    const rsrc_t r_w = make_rsrc(reinterpret_cast<const void*>(wa - sh0), min(BN, ds.n - n0) * row_bytes + sh0);
    const Lds L = lds_of(lds, ds.m, nsb);
    W wt;
    wt.init();
    wt.place(w, row_bytes, sh0);
    if (ds.xrs) {
        wt.load(r_w, sb0);
        stage_f16(ds, sb0, nsb, L);
    } else {
        // The activations first, waited for before the weights are asked for:
        // they are short trips to L2 that would otherwise queue behind every
        // wave's weights (8B gate and up, 12 rows: 25.7 -> 24.6 us; two
        // super-blocks of weights in flight instead of one: 28 us).
        StageF32 st;
        st.load(ds, w, sb0, nsb);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        wt.load(r_w, sb0);
        st.put(ds, w, nsb, L);
    }
    lds_barrier();
    v16f_t acc[1][2] = {};
    // rows past the matrix read its last row (their results are not stored)
    const uint32_t xr = min(l32, ds.m - 1u);
    const uint8_t* px = L.x + xr * L.xs + 32u * h;
    const uint8_t* ps = L.sx + 32u * xr * nsb + 16u * h;
    for (uint32_t s = 0; s < nsb; s++, px += 512u, ps += 32u) {
        // a stage's four operand reads are issued a stage ahead of their use
        // (each waited for at its use, they were half of a lone wave's time)
        u4_t xc[4], sxo = {};
        if constexpr (TY == TY_Q4K) sxo = *reinterpret_cast<const u4_t*>(ps);
#pragma unroll
        for (int t = 0; t < 4; t++) xc[t] = *reinterpret_cast<const u4_t*>(px + W::xofs(0, t));
        wt.take();
        if (s + 1u < nsb) wt.load(r_w, sb0 + s + 1u);
        if constexpr (TY == TY_Q4K) {
            acc[0][0] = mfma16(wt.cop[0], sxo, acc[0][0]);
            acc[0][1] = mfma16(wt.cop[1], sxo, acc[0][1]);
        }
        u4_t wc[2] = {wt.op(0, 0, 0), wt.op(0, 0, 1)};
#pragma unroll
        for (int g = 0; g < 4; g++) {
            u4_t xn[4];
            if (g < 3)
#pragma unroll
                for (int t = 0; t < 4; t++) xn[t] = *reinterpret_cast<const u4_t*>(px + W::xofs(g + 1, t));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                // the next step's weight operands are built while this step's MFMAs run
                acc[0][0] = mfma16(wc[0], xc[t], acc[0][0]);
                acc[0][1] = mfma16(wc[1], xc[t], acc[0][1]);
                if (g < 3 || t < 3) {
                    const int u = 4 * g + t + 1;
                    wc[0] = wt.op(u >> 2, u & 3, 0);
                    wc[1] = wt.op(u >> 2, u & 3, 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (g < 3)
#pragma unroll
                for (int t = 0; t < 4; t++) xc[t] = xn[t];
        }
    }
    lds_barrier();  // every wave past its activations: their LDS takes the results
    float* y = ds.y + (uint64_t)ks * ds.m * ds.ldy;
    store_wave<1, 2>(ds, y, 0u, n0 + 64u * w, acc, L.sc, reinterpret_cast<u4_t*>(lds + 128u + 4096u * w));
}
}  // namespace mmqs

// Tiles of any type in one launch (a layer's Q4_K and Q6_K projections
// together); dynamic LDS as the host sizes it for the largest range.
extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void rfxq_mmqs(MmqArgs args) {
    extern __shared__ __attribute__((aligned(16))) uint8_t mmqs_lds[];
    if (blockDim.x != mmqh::kThreads) return;
    const uint32_t tiles = min(gridDim.x, mmq_tile_count(args));
    if (blockIdx.x >= tiles) return;
    const uint32_t b = mmqh::xcd_tile(blockIdx.x, tiles);
    MmqDesc ds = mmq_pick(args, b);
    uint32_t* p = reinterpret_cast<uint32_t*>(&ds);
#pragma unroll
    for (uint32_t i = 0; i < sizeof(MmqDesc) / 4u; i++) p[i] = __builtin_amdgcn_readfirstlane(p[i]);
    const uint32_t t = __builtin_amdgcn_readfirstlane(b - ds.wg_begin);
    if (t >= ds.tiles_n * ds.splits || ds.m > 32u) return;
    const uint32_t ks = t % ds.splits, n0 = (t / ds.splits) * mmqh::BN;
    if (ds.type == TY_Q4K) mmqs::tile<mmqs::W4, TY_Q4K>(ds, n0, ks, mmqs_lds);
    else if (ds.type == TY_Q6K) mmqs::tile<mmqs::W6, TY_Q6K>(ds, n0, ks, mmqs_lds);
    else mmqs::tile<mmqs::W8, TY_Q8_0>(ds, n0, ks, mmqs_lds);
}
