// mmq.hip -- grouped int8 matrix-core matmul for Q4_K / Q6_K (and, from the
// 32-value-block section below, Q8_0 / Q4_0) weights against int8
// activations, bit-identical to the reference CPU kernels
// (src/gguf/ggml.zig:1002-1059 kBlockDot / matvecK256 / matmulK256,
// 1196-1222 matvecQ40Int, 1277-1294 matvecQ80Int) and so to dmmv.hip.
//
// The integer part of every block dot runs on the int8 MFMAs: the activations
// of 16 tokens are the A rows, 16 weight rows the B columns (Q4_K:
// v_mfma_i32_16x16x64_i8 over a 64-value quant span; Q6_K: the same MFMA
// over four 16-value runs, one run per MFMA, or over two int8 digits of
// scale * quant).  Integer dots are exact in any order, so isum = sum sc * dot
// and msum = sum mn * bsum are the reference's integers; the f32 tail per
// (token, row, super-block) is the reference's expression, and each output
// sums its blocks in block order.
//
// Three forms, chosen in launch_mmq by what fills the chip:
//   one-shot (mmq_kernel, mmq_seg_kernel, mmq32_kernel): a row tile's blocks
//     spread over the waves of a work group, summed from LDS -- small matrices;
//   streamed (mmw_kernel, mmw32_kernel): a wave takes a row tile and walks its
//     blocks in order, the sums in registers -- expert groups, large matrices;
//   tiled (mmp_kernel): 64 rows x 128 vectors per work group -- prefill sizes.
//
// Lane l of a wave: weight row l % 16 of its 16-row tile, k-quarter l / 16;
// the result lane l holds tokens 4*(l/16) .. +3 of that row.
#include <type_traits>

#include "device.hpp"
#include "fmt.hpp"
#include "kernels.hpp"

namespace lh {

typedef int mmq_i4 __attribute__((ext_vector_type(4)));

constexpr uint64_t NIB = 0x0F0F0F0F0F0F0F0Full;

// One wave computes one (16-row tile, super-block) for 16*MT tokens.  Every
// global load of the wave (weights, activation rows, activation scales) is
// issued before its first MFMA, so a wave costs one memory round trip.
//
// Q4_K: isum = sum_g sc[g] * dot(q_g, x_g) from one MFMA per 32-value group;
// the mins' integer sum_g mn[g] * sum(x_g) is one chained MFMA per group
// against mn[g] replicated over the group's bytes (mn <= 63 fits int8).
// Q6_K: the weights enter the MFMA as q - 32 (-32..31 fits int8), so
// isum = sum_run sc[run] * dot(q - 32, x) -- the reference's
// sum sc * (dot(q, x) - 32 * sum(x)) as one exact integer.  A 32-value group
// spans two 16-value runs with their own scales: one MFMA per run, the other
// run's lanes zeroed.

// Q4_K on v_mfma_i32_16x16x64_i8: one MFMA spans the 64 values of a 32-byte
// quant span p (groups 2p and 2p+1).  Lane quarter q4 holds 16 contiguous
// values, [64p + 16*q4, +16): quarters 0-1 lie in group 2p (low nibbles of
// the span's bytes), 2-3 in group 2p+1 (high nibbles), so both the
// activation and the weight loads are 16 contiguous bytes per lane.  The
// group sums come from two MFMAs, each with the other group's quarters of
// the weights zeroed; the mins' sum is one chained MFMA per span against
// each quarter's group min replicated.
struct Q4kTile {
    uint4 hdr;
    uint4 qs[4]; // span p's 16 bytes for this lane's quarter
};

__device__ __forceinline__ Q4kTile q4k_load(const uint8_t *blk, int q4) {
    Q4kTile w;
    w.hdr = *(const uint4 *)blk;
#pragma unroll
    for (int p = 0; p < 4; p++)
        w.qs[p] = *(const uint4 *)(blk + 16 + 32 * p + 16 * (q4 & 1));
    return w;
}

template <int MT>
__device__ __forceinline__ void q4k_tile(const Q4kTile &w, int q4, const mmq_i4 (&xa)[MT][4],
                                         const float (&xd)[MT][4], float (&r)[MT][4]) {
    int sc[8], mn[8];
#pragma unroll
    for (int p = 0; p < 4; p++)
        Fmt<LH_Q4_K>::scales(w.hdr, 2 * p, sc[2 * p], mn[2 * p], sc[2 * p + 1], mn[2 * p + 1]);
    const float d = half_bits_to_float(w.hdr.x & 0xffff);
    const float dmin = half_bits_to_float(w.hdr.x >> 16);
    const mmq_i4 z = {0, 0, 0, 0};
    const bool lo = q4 < 2;
    int isum[MT][4];
    mmq_i4 msum[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        msum[mt] = z;
#pragma unroll
        for (int i = 0; i < 4; i++)
            isum[mt][i] = 0;
    }
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const uint4 v = w.qs[p];
        const int sh = lo ? 0 : 4;
        const mmq_i4 wv = {(int)((v.x >> sh) & 0x0F0F0F0Fu), (int)((v.y >> sh) & 0x0F0F0F0Fu),
                           (int)((v.z >> sh) & 0x0F0F0F0Fu), (int)((v.w >> sh) & 0x0F0F0F0Fu)};
        const mmq_i4 wa = lo ? wv : z, wb = lo ? z : wv;
        const int m32 = (int)((uint32_t)(lo ? mn[2 * p] : mn[2 * p + 1]) * 0x01010101u);
        const mmq_i4 mrep = {m32, m32, m32, m32};
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const mmq_i4 da = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[mt][p], wa, z, 0, 0, 0);
            const mmq_i4 db = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[mt][p], wb, z, 0, 0, 0);
            msum[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[mt][p], mrep, msum[mt], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) // 24-bit products (|dot| < 2^16, sc <= 63): full rate, exact
                isum[mt][i] += __mul24(sc[2 * p], da[i]) + __mul24(sc[2 * p + 1], db[i]);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // xb.d * (d * f32(isum) - dmin * f32(min_isum))  (ggml.zig:1016-1017)
            const float a = d * (float)isum[mt][i];
            const float bb = dmin * (float)msum[mt][i];
            r[mt][i] = xd[mt][i] * (a - bb);
        }
}

// Q6_K (device SoA ql[U][128] | qh[U][64] | sc[U][16] | d[U]) on
// v_mfma_i32_16x16x64_i8: MFMA h spans values [64h, 64h + 64) and lane
// quarter q4 holds the 16 values [64h + 16*q4, +16) -- exactly the 16-value
// run 4h + q4 -- so activation and weight loads are 16 contiguous bytes per
// lane.  Each run has its own scale: one MFMA per run, the other quarters'
// weights zeroed.  The weights enter as q - 32 (-32..31 fits int8), so isum =
// sum_run sc[run] * dot(q - 32, x), the reference's sum sc * (dot(q, x) - 32 *
// sum(x)) as one exact integer.
struct Q6kTile {
    uint4 ql[2], qh[2]; // half n's 16 bytes of low bits / high bits for this lane's quarter
    uint4 sc;
    uint16_t d;
};

__device__ __forceinline__ Q6kTile q6k_load(const uint8_t *base, size_t U, size_t unit, int q4) {
    Q6kTile w;
#pragma unroll
    for (int n = 0; n < 2; n++) {
        w.ql[n] = *(const uint4 *)(base + unit * 128 + 64 * n + 16 * q4);
        w.qh[n] = *(const uint4 *)(base + U * 128 + unit * 64 + 32 * n + 16 * (q4 & 1));
    }
    w.sc = *(const uint4 *)(base + U * 192 + unit * 16);
    w.d = *(const uint16_t *)(base + U * 208 + unit * 2);
    return w;
}

// 4 bytes of 6-bit quants (low nibble at shift ls, two high bits at shift hs)
// -> q - 32 as int8: flip bit 5, then sign-extend it into bits 6 and 7
// where it is set (the values below 32)
__device__ __forceinline__ int q6_minus32(uint32_t ql, uint32_t qh, int ls, int hs) {
    const uint32_t v = ((ql >> ls) & 0x0F0F0F0Fu) | (((qh >> hs) & 0x03030303u) << 4);
    const uint32_t y = v ^ 0x20202020u;
    const uint32_t m = y & 0x20202020u;
    return (int)(y | (m << 1) | (m << 2));
}

template <int MT>
__device__ __forceinline__ void q6k_tile(const Q6kTile &w, int q4, const mmq_i4 (&xa)[MT][4],
                                         const float (&xd)[MT][4], float (&r)[MT][4]) {
    const float dw = half_bits_to_float(w.d);
    const mmq_i4 z = {0, 0, 0, 0};
    int isum[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            isum[mt][i] = 0;
#pragma unroll
    for (int h = 0; h < 4; h++) {
        const int n = h >> 1, ls = 4 * (h & 1), hs = 4 * (h & 1) + 2 * (q4 >> 1);
        const mmq_i4 vs = {q6_minus32(w.ql[n].x, w.qh[n].x, ls, hs), q6_minus32(w.ql[n].y, w.qh[n].y, ls, hs),
                           q6_minus32(w.ql[n].z, w.qh[n].z, ls, hs), q6_minus32(w.ql[n].w, w.qh[n].w, ls, hs)};
#pragma unroll
        for (int qq = 0; qq < 4; qq++) {
            const int sc = (int)(int8_t)byte_of(w.sc, 4 * h + qq);
            const mmq_i4 bq = q4 == qq ? vs : z;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const mmq_i4 dq = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[mt][h], bq, z, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) // 24-bit products (|dot| < 2^16, |sc| <= 128): full rate, exact
                    isum[mt][i] += __mul24(sc, dq[i]);
            }
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // xb.d * dec.d * f32(isum)  (ggml.zig:1019)
            const float s = xd[mt][i] * dw;
            r[mt][i] = s * (float)isum[mt][i];
        }
}

// ---- Q4_K with (token, group) rows: up to 16 tokens against unmasked weights -------
// A 64-deep MFMA span holds two Q4_K groups, each with its own scale.
// q4k_tile zeroes the weights outside one group and runs one MFMA per group:
// a masked copy of every weight tile, and a multiply per (token, group) of 16
// tokens however few there are.  Here the A rows of an MFMA are (token, group)
// pairs instead: row m = (t, g) carries token t's activations on the k slots
// of group part g and zeros elsewhere, so one MFMA over the unmasked weights
// returns both groups' integer dots for 8 tokens, and the scales multiply
// those dots with 24-bit multiply-adds (|dot| < 2^16, scale <= 63).  Integer
// dots are exact in any order, so every block's integers -- and the f32 tail
// after them -- are the reference's.
//
// k slots.  MFMA (P, half) covers quant spans 2P and 2P + 1: lane
// quarter q4 holds the 16 bytes 64P + 16*q4 of the block's 128 (span
// 2P + q4/2, bytes 16*(q4&1) + [0, 16)), their low nibbles for half 0 and
// high nibbles for half 1 -- group 4P + 2*(q4/2) + half.  A lane reads each
// weight byte once.  A row r16 = (token r16/2, part r16&1) is nonzero on the
// quarters with q4/2 == r16&1.
struct Q4kTileV {
    uint4 hdr;
    uint4 qs[2]; // quant bytes 64P + 16*q4, P = 0, 1
};

__device__ __forceinline__ Q4kTileV q4kv_load(const uint8_t *blk, int q4) {
    Q4kTileV w;
    w.hdr = *(const uint4 *)blk;
    w.qs[0] = *(const uint4 *)(blk + 16 + 16 * q4);
    w.qs[1] = *(const uint4 *)(blk + 80 + 16 * q4);
    return w;
}

// Offset in the block's 256 activations of lane quarter q4's 16 k slots in
// MFMA j = 2P + half.
__device__ __forceinline__ int q4kv_xoff(int j, int q4) {
    return 128 * (j >> 1) + 64 * (q4 >> 1) + 32 * (j & 1) + 16 * (q4 & 1);
}

// LDS of one work group: the per-block values [FUSED + 1][nb][16*MT][16*RG + 1]
// (the +1 staggers the four token quarters a wave writes across banks).
static size_t mmq_lds_bytes(int cols, int mt, int rg, bool fused) {
    return (size_t)4 * (fused ? 2 : 1) * (cols / 256) * 16 * mt * (16 * rg + 1);
}

constexpr int MMQ_MAX_SBW = 4; // super-blocks per wave (at most): cols <= 8192 (4096 at 32 tokens)

// Waves per work group (at most).  Eight: with sixteen the waves of a group
// finish microseconds apart at the barrier (four per SIMD share its issue).
constexpr int MMQ_WAVES = 8;

// One wave's operands for one super-block: the activations as the MFMA A
// operands (16 bytes per 64-value span and lane quarter).
template <int T, int MT, bool FUSED>
struct MmqOps {
    typename std::conditional<T == LH_Q4_K, Q4kTile, Q6kTile>::type w, w2;
    mmq_i4 xa[MT][4];
    float xd[MT][4];
};

// Work group: RG row tiles of 16 rows x KS super-block slices, one wave per
// (tile, slice); wave (rg, ks) computes super-blocks ks + j*KS (j < SBW) of
// its 16 rows for the group's tokens.  All of a wave's loads are issued,
// weights first, before its first MFMA.  The values meet in LDS; every output
// sums its blocks in block order (the reference's `acc += r`), SwiGLU(gate,
// up) when FUSED, and is stored or added.
// The work group's part of mmq_kernel: row tile bx, group by.
template <int T, int MT, bool FUSED, int SBW>
__device__ __forceinline__ void mmq_body(const DmmvParams &p, int bx, int by, int RG, int KS, float *part) {
    constexpr int TOK = 16 * MT;
    const bool ident = p.ident_n > 0;
    DmmvGroup grp;
    if (ident) {
        grp.plane = 0;
        grp.first = by * TOK;
        grp.n = min(TOK, p.ident_n - grp.first);
    } else {
        const int ng = p.n_groups_dev ? *p.n_groups_dev : p.n_groups;
        if (by >= ng)
            return;
        grp = p.groups[by];
    }
    const int n = grp.n, cols = p.cols, nb = cols / 256;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    const int r16 = ln & 15, q4 = ln >> 4;
    const int rg = wave % RG, ks = wave / RG;
    const int R = 16 * RG, RS = R + 1;
    const int row0 = bx * R;
    const int rl = 16 * rg + r16;
    const int row = min(row0 + rl, p.rows - 1);
    const size_t U = (size_t)p.rows * nb;
    const size_t mat = (size_t)nb * TOK * RS; // floats per matrix in LDS
    const uint8_t *wb = p.w + (size_t)grp.plane * p.plane_bytes;
    const uint8_t *wb2 = FUSED ? p.w2 + (size_t)grp.plane * p.plane_bytes : nullptr;
    MmqOps<T, MT, FUSED> op[SBW];
    int bj[SBW];
    // 1. weights (they depend on the group only)
#pragma unroll
    for (int j = 0; j < SBW; j++) {
        bj[j] = min(ks + j * KS, nb - 1); // past nb: a real block, never stored
        const size_t unit = (size_t)row * nb + bj[j];
        if constexpr (T == LH_Q4_K) {
            op[j].w = q4k_load(wb + unit * 144, q4);
            if constexpr (FUSED)
                op[j].w2 = q4k_load(wb2 + unit * 144, q4);
        } else {
            op[j].w = q6k_load(wb, U, unit, q4);
        }
    }
    // 2. activations: the row of A-row r16 in each token tile (tokens past n
    // repeat the last one; their outputs are never stored), then every
    // super-block's 8-value pieces and the output tokens' block scales
    int vrow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
        vrow[mt] = ident ? grp.first + min(16 * mt + r16, n - 1) : p.pair_src[grp.first + min(16 * mt + r16, n - 1)];
    int vout[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            vout[mt][i] = __shfl(vrow[mt], 4 * q4 + i);
#pragma unroll
    for (int j = 0; j < SBW; j++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int8_t *xr = p.xq + (size_t)vrow[mt] * cols + 256 * bj[j] + 16 * q4;
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++)
                op[j].xa[mt][s4] = *(const mmq_i4 *)(xr + 64 * s4);
#pragma unroll
            for (int i = 0; i < 4; i++)
                op[j].xd[mt][i] = p.xd[(size_t)vout[mt][i] * nb + bj[j]];
        }
    // 3. the first output of this thread (the common case is one per thread):
    // its destination and, for a residual add, the value it adds to
    const int idx0 = threadIdx.x, tk0 = idx0 / R, rr0 = idx0 % R;
    const bool out0 = idx0 < n * R && row0 + rr0 < p.rows;
    const int dst0 = ident ? grp.first + tk0 : p.pair_dst[grp.first + min(tk0, n - 1)];
    const float old0 = out0 && p.accumulate ? p.out[(size_t)dst0 * p.out_stride + row0 + rr0] : 0.0f;
    __builtin_amdgcn_sched_barrier(0); // every load above is in flight before the first MFMA
    // 4. the tiles
#pragma unroll
    for (int j = 0; j < SBW; j++) {
        float r[MT][4], r2[MT][4];
        if constexpr (T == LH_Q4_K) {
            q4k_tile<MT>(op[j].w, q4, op[j].xa, op[j].xd, r);
            if constexpr (FUSED)
                q4k_tile<MT>(op[j].w2, q4, op[j].xa, op[j].xd, r2);
        } else {
            q6k_tile<MT>(op[j].w, q4, op[j].xa, op[j].xd, r);
        }
        if (ks + j * KS < nb) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const size_t o = ((size_t)bj[j] * TOK + 16 * mt + 4 * q4 + i) * RS + rl;
                    part[o] = r[mt][i];
                    if constexpr (FUSED)
                        part[mat + o] = r2[mt][i];
                }
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < n * R; idx += blockDim.x) {
        const int tk = idx / R, rr = idx % R;
        if (row0 + rr >= p.rows)
            continue;
        const float *pv = part + (size_t)tk * RS + rr;
        float acc = 0.0f;
        for (int b = 0; b < nb; b++)
            acc = acc + pv[(size_t)b * TOK * RS];
        float v = acc;
        if constexpr (FUSED) {
            float acc2 = 0.0f;
            for (int b = 0; b < nb; b++)
                acc2 = acc2 + pv[mat + (size_t)b * TOK * RS];
            v = swiglu1(acc, acc2);
        }
        const bool first = idx == idx0;
        const int dst = first ? dst0 : ident ? grp.first + tk : p.pair_dst[grp.first + tk];
        float *o = p.out + (size_t)dst * p.out_stride + row0 + rr;
        if (p.accumulate)
            v = (first ? old0 : *o) + v;
        *o = v;
    }
}

template <int T, int MT, bool FUSED, int SBW>
__global__ __launch_bounds__(64 * MMQ_WAVES) void mmq_kernel(DmmvParams p, int RG, int KS) {
    extern __shared__ __align__(16) float part[];
    mmq_body<T, MT, FUSED, SBW>(p, blockIdx.x, blockIdx.y, RG, KS, part);
}

// Up to DMMV_MAX_SEG matrices (Q4_K or Q6_K, same columns, same lane groups)
// in one launch: the row tiles of the segments one after another along x.
template <int MT, int SBW>
__global__ __launch_bounds__(64 * MMQ_WAVES) void mmq_seg_kernel(DmmvSegParams sp, int RG, int KS) {
    extern __shared__ __align__(16) float part[];
    int tile = blockIdx.x, s = 0;
    while (s + 1 < sp.n_seg && tile >= sp.seg[s].tiles) {
        tile -= sp.seg[s].tiles;
        s++;
    }
    DmmvParams p = sp.base;
    p.w = sp.seg[s].w;
    p.rows = sp.seg[s].rows;
    p.out = sp.seg[s].out;
    p.out_stride = sp.seg[s].rows;
    if (sp.seg[s].t == LH_Q4_K)
        mmq_body<LH_Q4_K, MT, false, SBW>(p, tile, blockIdx.y, RG, KS, part);
    else
        mmq_body<LH_Q6_K, MT, false, SBW>(p, tile, blockIdx.y, RG, KS, part);
}

// ---- streamed in block order --------------------------------------------------------
// The grouped (expert) matmuls, and lane groups over many rows (the head):
// bound by the weights' bytes once nothing else is in the way.  A wave owns a
// 16-row tile for its group's tokens and walks the row's super-blocks in
// order, so each output is one f32 register that takes `acc += r` block by
// block: no LDS sums, no barrier between the first block and the last, and
// the waves of a work group are independent.  Three things decide its speed:
//   - Loads in address order.  A load whose lanes are in MFMA order (16 rows x
//     64 bytes, neighbouring lanes in different rows) takes 65 cycles of the
//     CU's address path per KB, one with neighbouring lanes in one row 18
//     (probe, L2-resident).  So a wave loads its block with lanes in address
//     order and turns it into MFMA order through its own LDS.
//   - Two blocks in registers or in flight while one computes, at 2-4 waves per
//     SIMD; the tokens' rows staged once per work group with all their loads in
//     one round trip (staged token by token they took 7 us of a wave's 16).
//   - Few VALU operations per block: the sets of 8 tokens below, and the mins on
//     one f16 MFMA.  An int8 MFMA of 16 cycles hides little VALU work (beside
//     four ANDs of 2.9 cycles it takes 24).
// Measured (us per launch, rocprof; against the one-shot kernel, the LDS ring
// that served gate/up over 2048 columns, and the streamed head kernel before):
// gate/up 7168 -> 2048 over about 60 experts at 24 tokens 434 -> 166, its down
// 154 -> 84; 2048 -> 768 at 128 tokens 50.6 -> 34.6, down (Q6_K) 51 -> 35; at
// 32 tokens 26.0 -> 24.9 and 26.9 -> 22.1; the 151936-row Q6_K head at 32
// lanes 111 -> 81.
// Q4_K, up to 16 tokens in sets of 8 (token, group part) rows, the arithmetic
// of q4kv_tile with the mins on one f16 MFMA: sum_g mn_g * sum(x_g) over the
// block's sixteen 16-value sums, |sum| <= 2032 and mn <= 63 exact in f16, their
// total below 2^24 exact in f32.  bs: this lane's four sums (A row r16: token
// mmw_bs_token(r16), sums 4*q4 ..), so result i of a lane is token 8*(i/2) +
// 2*q4 + (i&1) of its row: the tokens of sets 0 and 1.
typedef _Float16 mmq_h4 __attribute__((ext_vector_type(4)));
typedef float mmq_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int mmw_bs_token(int r16) { return 8 * ((r16 >> 1) & 1) + 2 * (r16 >> 2) + (r16 & 1); }

__device__ __forceinline__ void q4kw_acc(const Q4kTileV &w, int q4, int ns, const mmq_i4 (&xa)[2][4], mmq_h4 bs,
                                         const float (&xd)[2][2], float (&acc)[2][2]) {
    const uint32_t a = w.hdr.y, b = w.hdr.z, c = w.hdr.w;
    const uint32_t scv[2] = {a & 0x3F3F3F3Fu, (c & 0x0F0F0F0Fu) | ((a >> 2) & 0x30303030u)};
    const uint32_t mnv[2] = {b & 0x3F3F3F3Fu, ((c >> 4) & 0x0F0F0F0Fu) | ((b >> 2) & 0x30303030u)};
    const float d = half_bits_to_float(w.hdr.x & 0xffff);
    const float dmin = half_bits_to_float(w.hdr.x >> 16);
    const mmq_i4 z = {0, 0, 0, 0};
    const uint32_t m2 = (q4 < 2 ? mnv[0] : mnv[1]) >> (16 * (q4 & 1)); // mins of groups 2*q4, 2*q4 + 1
    const _Float16 m0 = (_Float16)(unsigned short)(m2 & 0xFF), m1 = (_Float16)(unsigned short)((m2 >> 8) & 0xFF);
    const mmq_f4 ms = __builtin_amdgcn_mfma_f32_16x16x16f16(bs, mmq_h4{m0, m0, m1, m1}, mmq_f4{0.0f, 0.0f, 0.0f, 0.0f},
                                                            0, 0, 0);
    mmq_i4 wv[4];
    int s0[4], s1[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int P = j >> 1, half = j & 1;
        const uint32_t sh = 4 * half;
        wv[j] = mmq_i4{(int)((w.qs[P].x >> sh) & 0x0F0F0F0Fu), (int)((w.qs[P].y >> sh) & 0x0F0F0F0Fu),
                       (int)((w.qs[P].z >> sh) & 0x0F0F0F0Fu), (int)((w.qs[P].w >> sh) & 0x0F0F0F0Fu)};
        s0[j] = (int)((scv[P] >> (8 * half)) & 0xFF);
        s1[j] = (int)((scv[P] >> (8 * (2 + half))) & 0xFF);
    }
#pragma unroll
    for (int s = 0; s < 2; s++) {
        if (s >= ns)
            break;
        int isum[2] = {0, 0};
        mmq_i4 dq[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            dq[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[s][j], wv[j], z, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) { // 24-bit products (|dot| < 2^16, sc <= 63): exact
            isum[0] = __mul24(s0[j], dq[j][0]) + isum[0];
            isum[1] = __mul24(s0[j], dq[j][2]) + isum[1];
            isum[0] = __mul24(s1[j], dq[j][1]) + isum[0];
            isum[1] = __mul24(s1[j], dq[j][3]) + isum[1];
        }
#pragma unroll
        for (int jj = 0; jj < 2; jj++) {
            // xb.d * (d * f32(isum) - dmin * f32(min_isum))  (ggml.zig:1016-1017)
            const float aa = d * (float)isum[jj];
            const float bb = dmin * ms[2 * s + jj];
            acc[s][jj] = acc[s][jj] + xd[s][jj] * (aa - bb);
        }
    }
}

// Q6_K, 16*MT tokens: a lane's 16 values of MFMA h are one run (4h + q4) with
// one scale, so the scale goes into the weights: v = sc * (q - 32) (14 bits)
// as the digits v = 128 a + b, a = v >> 7 in [-32, 32] and b = v & 127, each
// int8.  Two unmasked MFMA chains over the block then give
// isum = 128 sum(a x) + sum(b x), the reference's integer -- half the MFMAs of
// one masked MFMA per run, and no multiply per (token, run).
typedef short mmq_s2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void q6k_digits(uint32_t q, mmq_s2 sc, mmq_s2 off, int &hi, int &lo) {
    // bytes (0, 2) and (1, 3) of q as 16-bit pairs, scaled: sc * q - 32 sc
    const mmq_s2 e = __builtin_bit_cast(mmq_s2, q & 0x00FF00FFu) * sc + off;
    const mmq_s2 o = __builtin_bit_cast(mmq_s2, (q >> 8) & 0x00FF00FFu) * sc + off;
    const mmq_s2 eh = e >> 7, oh = o >> 7;
    // result byte k = low byte of value k: e.lo, o.lo, e.hi, o.hi
    hi = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, oh), __builtin_bit_cast(uint32_t, eh), 0x06020400u);
    lo = (int)(__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, o), __builtin_bit_cast(uint32_t, e), 0x06020400u) &
               0x7F7F7F7Fu);
}

template <int MT>
__device__ __forceinline__ void q6kw_acc(const Q6kTile &w, int q4, const mmq_i4 (&xa)[MT][4],
                                         const float4 (&xd)[MT], float (&acc)[MT][4]) {
    const float dw = half_bits_to_float(w.d);
    const mmq_i4 z = {0, 0, 0, 0};
    const uint32_t scw[4] = {w.sc.x, w.sc.y, w.sc.z, w.sc.w};
    mmq_i4 ah[MT], al[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
        ah[mt] = al[mt] = z;
#pragma unroll
    for (int h = 0; h < 4; h++) {
        const int n = h >> 1, ls = 4 * (h & 1), hs = 4 * (h & 1) + 2 * (q4 >> 1);
        const short sc = (short)(int8_t)((scw[h] >> (8 * q4)) & 0xFF);
        const mmq_s2 s2 = {sc, sc};
        mmq_s2 off = s2 * (short)-32;
        asm("" : "+v"(off)); // kept a value of its own: one packed multiply-add per pair below
        const uint32_t ql[4] = {w.ql[n].x, w.ql[n].y, w.ql[n].z, w.ql[n].w};
        const uint32_t qh[4] = {w.qh[n].x, w.qh[n].y, w.qh[n].z, w.qh[n].w};
        mmq_i4 whi, wlo;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            int hi, lo;
            q6k_digits(((ql[e] >> ls) & 0x0F0F0F0Fu) | (((qh[e] >> hs) & 0x03030303u) << 4), s2, off, hi, lo);
            whi[e] = hi;
            wlo[e] = lo;
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            ah[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[mt][h], whi, ah[mt], 0, 0, 0);
            al[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[mt][h], wlo, al[mt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const float xs[4] = {xd[mt].x, xd[mt].y, xd[mt].z, xd[mt].w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // xb.d * dec.d * f32(isum)  (ggml.zig:1019)
            const float s = xs[i] * dw;
            acc[mt][i] = acc[mt][i] + s * (float)((ah[mt][i] << 7) + al[mt][i]);
        }
    }
}

// One block of 16 rows, as loaded (lanes in address order) and as kept in LDS.
// LDS holds a row's 16-byte chunks one after another (Q4_K: the 9 of its
// GGML block; Q6_K: 8 of ql, 4 of qh, the scales; d apart): odd chunk
// strides, so the 16 rows a wave reads together sit in different banks.
// Src: the lane's byte offsets in the tile's rows (rows past the last read that
// one).
template <int T> struct MmwBlk;
template <> struct MmwBlk<LH_Q4_K> {
    static constexpr int ROWB = 144, BYTES = 16 * 144;
    using Tile = Q4kTileV;
    mmq_i4 v0, v1;
    uint32_t t; // chunks 128 .. 143 of the 144, a dword per lane
    struct Src {
        const uint8_t *b;
        uint32_t o[3];
    };
    __device__ __forceinline__ static Src src(const uint8_t *wb, size_t, int rows, int nb, int row0, int ln) {
        Src s;
        s.b = wb;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int q = i < 2 ? 64 * i + ln : 128 + (ln >> 2);
            const int r = q / 9, c = q - 9 * r;
            s.o[i] = (uint32_t)min(row0 + r, rows - 1) * (uint32_t)(nb * 144) + 16 * c + (i == 2 ? 4 * (ln & 3) : 0);
        }
        return s;
    }
    __device__ __forceinline__ void load(const Src &s, int b) {
        const uint8_t *p = s.b + (size_t)b * 144;
        v0 = *(const mmq_i4 *)(p + s.o[0]);
        v1 = *(const mmq_i4 *)(p + s.o[1]);
        t = *(const uint32_t *)(p + s.o[2]);
    }
    __device__ __forceinline__ void store(uint8_t *l, int ln) const {
        *(mmq_i4 *)(l + 16 * ln) = v0;
        *(mmq_i4 *)(l + 1024 + 16 * ln) = v1;
        *(uint32_t *)(l + 2048 + 4 * ln) = t;
    }
    __device__ __forceinline__ static Tile tile(const uint8_t *l, int r16, int q4) {
        return q4kv_load(l + r16 * ROWB, q4);
    }
};
template <> struct MmwBlk<LH_Q6_K> {
    static constexpr int ROWB = 208, BYTES = 16 * 208 + 64;
    using Tile = Q6kTile;
    mmq_i4 v0, v1, v2; // ql chunks 0-63, 64-127 of the 16 rows, qh
    uint32_t s, d;
    struct Src {
        const uint8_t *q, *h, *sc, *d;
        uint32_t oq0, oq1, oh, os, od;
    };
    __device__ __forceinline__ static Src src(const uint8_t *wb, size_t U, int rows, int nb, int row0, int ln) {
        Src s;
        s.q = wb;
        s.h = wb + U * 128;
        s.sc = wb + U * 192;
        s.d = wb + U * 208;
        const uint32_t u0 = (uint32_t)min(row0 + (ln >> 3), rows - 1) * nb;
        const uint32_t u1 = (uint32_t)min(row0 + 8 + (ln >> 3), rows - 1) * nb;
        const uint32_t u2 = (uint32_t)min(row0 + (ln >> 2), rows - 1) * nb;
        s.oq0 = u0 * 128 + 16 * (ln & 7);
        s.oq1 = u1 * 128 + 16 * (ln & 7);
        s.oh = u2 * 64 + 16 * (ln & 3);
        s.os = u2 * 16 + 4 * (ln & 3);
        s.od = u2 * 2;
        return s;
    }
    __device__ __forceinline__ void load(const Src &s_, int b) {
        v0 = *(const mmq_i4 *)(s_.q + (size_t)b * 128 + s_.oq0);
        v1 = *(const mmq_i4 *)(s_.q + (size_t)b * 128 + s_.oq1);
        v2 = *(const mmq_i4 *)(s_.h + (size_t)b * 64 + s_.oh);
        s = *(const uint32_t *)(s_.sc + (size_t)b * 16 + s_.os);
        d = *(const uint16_t *)(s_.d + (size_t)b * 2 + s_.od);
    }
    __device__ __forceinline__ void store(uint8_t *l, int ln) const {
        *(mmq_i4 *)(l + (ln >> 3) * ROWB + 16 * (ln & 7)) = v0;
        *(mmq_i4 *)(l + (8 + (ln >> 3)) * ROWB + 16 * (ln & 7)) = v1;
        *(mmq_i4 *)(l + (ln >> 2) * ROWB + 128 + 16 * (ln & 3)) = v2;
        *(uint32_t *)(l + (ln >> 2) * ROWB + 192 + 4 * (ln & 3)) = s;
        *(uint32_t *)(l + 16 * ROWB + 4 * (ln >> 2)) = d;
    }
    __device__ __forceinline__ static Tile tile(const uint8_t *l, int r16, int q4) {
        Tile w;
        const uint8_t *p = l + r16 * ROWB;
#pragma unroll
        for (int n = 0; n < 2; n++) {
            w.ql[n] = *(const uint4 *)(p + 64 * n + 16 * q4);
            w.qh[n] = *(const uint4 *)(p + 128 + 32 * n + 16 * (q4 & 1));
        }
        w.sc = *(const uint4 *)(p + 192);
        w.d = (uint16_t) * (const uint32_t *)(l + 16 * ROWB + 4 * r16);
        return w;
    }
};

// Orders this wave's LDS stores against its own reads by other lanes (the
// LDS serves a wave's accesses in order; this keeps the compiler's order).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

constexpr int MMW_W = 4;          // waves per work group: four neighbouring row tiles, four staged tokens each
constexpr int MMW_XL_COLS = 2048; // the tokens' whole rows are staged in LDS up to here

// LDS of a work group: scales [nb][TOK]; the tokens' rows [TOK][xrow] (Q4_K:
// then 256 zeros and the 16-value sums [TOK][brow]) once (XL) or one block
// of them per wave; per wave a block of 16 weight rows.
template <int T, int MT, bool XL>
__host__ __device__ constexpr int mmw_xbytes(int cols) {
    const int xrow = (XL ? cols : 256) + 16, brow = (XL ? cols / 256 : 1) * 32 + 16;
    return 16 * MT * xrow + (T == LH_Q4_K ? 256 + 16 * MT * brow : 0);
}
template <int T, int MT, bool XL>
static size_t mmw_lds(int cols) {
    const size_t x = mmw_xbytes<T, MT, XL>(cols);
    return (size_t)(cols / 256) * 64 * MT + (XL ? x + MMW_W * MmwBlk<T>::BYTES : MMW_W * (x + MmwBlk<T>::BYTES));
}

// FUSED: gate and up with the SwiGLU epilogue.  XL: the tokens' int8 rows are
// staged in LDS once per work group; else each wave brings a block's columns of
// them along with the block's weights.
template <int T, int MT, bool FUSED, bool XL, int OCC>
__global__ __launch_bounds__(64 * MMW_W, OCC) void mmw_kernel(DmmvParams p) {
    extern __shared__ __align__(16) uint8_t sh[];
    using B = MmwBlk<T>;
    constexpr bool K4 = T == LH_Q4_K;
    static_assert(!K4 || MT == 1, "Q4_K: 16 tokens");
    static_assert(!FUSED || K4, "a fused pair is Q4_K");
    constexpr int TOK = 16 * MT, M = FUSED ? 2 : 1, W = MMW_W, XN = 4 * MT;
    const bool ident = p.ident_n > 0;
    const int cols = p.cols, nb = cols / 256;
    const int gi = blockIdx.y;
    DmmvGroup grp;
    if (ident) {
        grp.plane = 0;
        grp.first = gi * TOK;
        grp.n = min(TOK, p.ident_n - grp.first);
    } else {
        const int ng = p.n_groups_dev ? *p.n_groups_dev : p.n_groups;
        if (gi >= ng)
            return;
        grp = p.groups[gi];
    }
    const int n = grp.n, ns = (n + 7) / 8; // Q4_K: sets of 8 tokens
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    const int r16 = ln & 15, q4 = ln >> 4;
    const int row0 = ((int)blockIdx.x * W + wave) * 16;
    const int xrow = (XL ? cols : 256) + 16, brow = (XL ? nb : 1) * 32 + 16;
    const int xbytes = mmw_xbytes<T, MT, XL>(cols);
    float *xds = (float *)sh;
    uint8_t *wls = sh + (size_t)nb * TOK * 4 + (XL ? xbytes + wave * B::BYTES : wave * (B::BYTES + xbytes));
    uint8_t *xl = XL ? sh + (size_t)nb * TOK * 4 : wls + B::BYTES;
    uint8_t *zl = xl + TOK * xrow, *bl = zl + 256;
    auto halves = [](const mmq_i4 &v) {
        return mmq_h4{(_Float16)(short)v[0], (_Float16)(short)v[1], (_Float16)(short)v[2], (_Float16)(short)v[3]};
    };
    // the vector of the group's t-th token (past n: the last); group_src needs no group
    const int *tab = p.group_src ? p.group_src + (size_t)gi * p.group_stride : p.pair_src + grp.first;
    const int tmax = p.group_src ? TOK - 1 : n - 1;
    auto vec_of = [&](int t) { return tab[min(t, tmax)]; };
    typename B::Src src[M];
    src[0] = B::src(p.w + (size_t)grp.plane * p.plane_bytes, (size_t)p.rows * nb, p.rows, nb, row0, ln);
    if constexpr (FUSED) {
        src[1] = src[0];
        src[1].b = p.w2 + (size_t)grp.plane * p.plane_bytes;
    }
    struct Stage {
        B w[M];
        mmq_i4 x[XL ? 1 : XN], bs; // (not XL) tokens 4 i + ln / 16, chunk ln % 16; sums 4 (ln % 4) .. of token ln / 4
    } st[2];
    const int8_t *xr[XN];
    const int32_t *br;
    if constexpr (!XL) {
#pragma unroll
        for (int i = 0; i < XN; i++)
            xr[i] = p.xq + (size_t)vec_of(4 * i + (ln >> 4)) * cols + 16 * (ln & 15);
        if constexpr (K4)
            br = p.xs + (size_t)vec_of(ln >> 2) * (cols / 16) + 4 * (ln & 3);
    }
    auto load = [&](Stage &s, int b) {
        s.w[0].load(src[0], b);
        if constexpr (FUSED)
            s.w[1].load(src[1], b);
        if constexpr (!XL) {
#pragma unroll
            for (int i = 0; i < XN; i++)
                s.x[i] = *(const mmq_i4 *)(xr[i] + 256 * b);
            if constexpr (K4)
                s.bs = *(const mmq_i4 *)(br + 16 * b);
        }
    };
    auto commit = [&](const Stage &s, int m) { // matrix m's block to this wave's LDS
        wave_lds_sync();
        s.w[m].store(wls, ln);
        if constexpr (!XL)
            if (m == 0) {
#pragma unroll
                for (int i = 0; i < XN; i++)
                    *(mmq_i4 *)(xl + (4 * i + (ln >> 4)) * xrow + 16 * (ln & 15)) = s.x[i];
                if constexpr (K4)
                    *(mmq_h4 *)(bl + (ln >> 2) * brow + 8 * (ln & 3)) = halves(s.bs);
            }
        wave_lds_sync();
    };
    // the block scales: 16 threads per token
    const int xt16 = threadIdx.x >> 4, xb16 = threadIdx.x & 15;
    const float *xdp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
        xdp[mt] = p.xd + (size_t)vec_of(16 * mt + xt16) * nb;
    if constexpr (XL) {
        // nb <= 8: XN token rows per wave, all their loads before the weights' and
        // the stores behind them, so one round trip covers the staging
        int v[XN];
#pragma unroll
        for (int i = 0; i < XN; i++)
            v[i] = vec_of(XN * wave + i);
        const int c0 = min(ln, 16 * nb - 1), c1 = min(64 + ln, 16 * nb - 1);
        mmq_i4 x0[XN], x1[XN], bs[2];
        float xdv[MT];
#pragma unroll
        for (int i = 0; i < XN; i++) {
            x0[i] = *(const mmq_i4 *)(p.xq + (size_t)v[i] * cols + 16 * c0);
            x1[i] = *(const mmq_i4 *)(p.xq + (size_t)v[i] * cols + 16 * c1);
        }
        if constexpr (K4) {
            const int va = ln < 32 ? v[0] : v[1], vb = ln < 32 ? v[2] : v[3], cb = min(ln & 31, 4 * nb - 1);
            bs[0] = *(const mmq_i4 *)(p.xs + (size_t)va * (cols / 16) + 4 * cb);
            bs[1] = *(const mmq_i4 *)(p.xs + (size_t)vb * (cols / 16) + 4 * cb);
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
            xdv[mt] = xdp[mt][min(xb16, nb - 1)];
        __builtin_amdgcn_sched_barrier(0);
        load(st[0], 0);
        load(st[1], min(1, nb - 1));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < XN; i++) {
            uint8_t *l = xl + (size_t)(XN * wave + i) * xrow;
            if (ln < 16 * nb)
                *(mmq_i4 *)(l + 16 * ln) = x0[i];
            if (64 + ln < 16 * nb)
                *(mmq_i4 *)(l + 16 * (64 + ln)) = x1[i];
        }
        if constexpr (K4)
#pragma unroll
            for (int i = 0; i < 2; i++)
                if ((ln & 31) < 4 * nb)
                    *(mmq_h4 *)(bl + (size_t)(4 * wave + 2 * i + (ln >> 5)) * brow + 8 * (ln & 31)) = halves(bs[i]);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
            if (xb16 < nb)
                xds[xb16 * TOK + 16 * mt + xt16] = xdv[mt];
        if (K4 && threadIdx.x < 16)
            *(mmq_i4 *)(zl + 16 * threadIdx.x) = mmq_i4{0, 0, 0, 0};
    } else {
        load(st[0], 0);
        load(st[1], min(1, nb - 1));
        for (int b0 = 0; b0 < nb; b0 += 64) {
            float v[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int u = 0; u < 4; u++)
                    v[mt][u] = xdp[mt][min(b0 + 16 * u + xb16, nb - 1)];
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (b0 + 16 * u + xb16 < nb)
                        xds[(b0 + 16 * u + xb16) * TOK + 16 * mt + xt16] = v[mt][u];
        }
        if (K4 && ln < 16)
            *(mmq_i4 *)(zl + 16 * ln) = mmq_i4{0, 0, 0, 0};
    }
    lds_barrier();
    // Q4_K: A row r16 = (token r16/2 of the set, group part r16&1): live on the
    // quarters of its part, zeros elsewhere; Q6_K: token r16
    const bool live = (q4 >> 1) == (r16 & 1);
    const int xstep = XL && (live || !K4) ? 256 : 0;
    const uint8_t *xt[2], *bt = bl + mmw_bs_token(r16) * brow + 8 * q4;
    if constexpr (K4) {
        xt[0] = live ? xl + (r16 / 2) * xrow : zl;
        xt[1] = live ? xl + (8 + r16 / 2) * xrow : zl;
    } else {
        xt[0] = xl + r16 * xrow + 16 * q4;
        xt[1] = xl + (MT == 2 ? 16 + r16 : r16) * xrow + 16 * q4;
    }
    // accumulators: Q4_K [matrix][set][token pair], Q6_K [0][token tile][4 tokens]
    float acc4[M][2][2] = {}, acc6[MT][4] = {};
    // Block b: its A rows from LDS, then each matrix's MFMAs with the next
    // tile (the other matrix, or the next block) already stored to LDS and
    // read back in MFMA order, so that latency runs under the arithmetic.
    commit(st[0], 0);
    typename B::Tile w0 = B::tile(wls, r16, q4);
    auto step = [&](int b, Stage &cur, const Stage &nxt) {
        if constexpr (K4) {
            mmq_i4 xa[2][4];
            float xd[2][2];
#pragma unroll
            for (int s = 0; s < 2; s++) {
                if (s >= ns)
                    break;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    xa[s][j] = *(const mmq_i4 *)(xt[s] + b * xstep + q4kv_xoff(j, q4));
                const float2 v = *(const float2 *)(xds + b * TOK + 8 * s + 2 * q4);
                xd[s][0] = v.x;
                xd[s][1] = v.y;
            }
            const mmq_h4 bs = *(const mmq_h4 *)(bt + (XL ? 32 * b : 0));
            commit(FUSED ? cur : nxt, FUSED ? 1 : 0);
            const Q4kTileV w1 = B::tile(wls, r16, q4);
            load(cur, min(b + 2, nb - 1)); // past the last block: the last one again, not used
            __builtin_amdgcn_sched_barrier(0);
            q4kw_acc(w0, q4, ns, xa, bs, xd, acc4[0]);
            if constexpr (FUSED) {
                commit(nxt, 0);
                w0 = B::tile(wls, r16, q4);
                q4kw_acc(w1, q4, ns, xa, bs, xd, acc4[M - 1]);
            } else {
                w0 = w1;
            }
        } else {
            float4 xd[MT];
            mmq_i4 xa[MT][4];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                xd[mt] = *(const float4 *)(xds + b * TOK + 16 * mt + 4 * q4);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    xa[mt][j] = *(const mmq_i4 *)(xt[mt] + b * xstep + 64 * j);
            }
            commit(nxt, 0);
            const typename B::Tile w1 = B::tile(wls, r16, q4);
            load(cur, min(b + 2, nb - 1)); // past the last block: the last one again, not used
            __builtin_amdgcn_sched_barrier(0);
            q6kw_acc<MT>(w0, q4, xa, xd, acc6);
            w0 = w1;
        }
    };
    for (int b = 0; b < nb; b += 2) {
        step(b, st[0], st[1]);
        if (b + 1 >= nb)
            break;
        step(b + 1, st[1], st[0]);
    }
    const int row = row0 + r16;
    if (row >= p.rows)
        return;
    auto put = [&](int t, float v) {
        if (t >= n)
            return;
        const int dst = ident || p.pos_ident ? grp.first + t : p.pair_dst[grp.first + t];
        float *o = p.out + (size_t)dst * p.out_stride + row;
        *o = p.accumulate ? *o + v : v;
    };
    if constexpr (K4) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int jj = 0; jj < 2; jj++)
                put(8 * s + 2 * q4 + jj, FUSED ? swiglu1(acc4[0][s][jj], acc4[M - 1][s][jj]) : acc4[0][s][jj]);
    } else {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                put(16 * mt + 4 * q4 + i, acc6[mt][i]);
    }
}

// Waves per SIMD of each form, as its registers allow (3: 168, 2: 256, 4: 128).
template <int T, int MT, bool FUSED, bool XL> constexpr int mmw_occ() {
    return XL ? (FUSED || MT == 2 ? 3 : 4) : (FUSED || MT == 2 ? 2 : 3);
}
template <int T, int MT, bool FUSED>
static void mmw_launch_t(const DmmvParams &p, hipStream_t st) {
    const int groups = p.ident_n > 0 ? (p.ident_n + 16 * MT - 1) / (16 * MT) : p.n_groups;
    const int tiles = (p.rows + 15) / 16;
    const dim3 grid((tiles + MMW_W - 1) / MMW_W, groups), block(64 * MMW_W);
    if (p.cols <= MMW_XL_COLS)
        hipLaunchKernelGGL((mmw_kernel<T, MT, FUSED, true, mmw_occ<T, MT, FUSED, true>()>), grid, block,
                           (mmw_lds<T, MT, true>(p.cols)), st, p);
    else
        hipLaunchKernelGGL((mmw_kernel<T, MT, FUSED, false, mmw_occ<T, MT, FUSED, false>()>), grid, block,
                           (mmw_lds<T, MT, false>(p.cols)), st, p);
}

// Shape of a launch: KS = min(nb, MMQ_WAVES) slices of SBW super-blocks per
// wave, as many row tiles beside them as fit the wave count and 64 KB of LDS,
// but no more than the matrix has.
static bool mmq_shape(int rows, int cols, int mt, bool fused, int &rg, int &ks, int &sbw) {
    const int nb = cols / 256;
    ks = nb < MMQ_WAVES ? nb : MMQ_WAVES;
    sbw = (nb + ks - 1) / ks;
    if (sbw == 3)
        sbw = 4;
    if (sbw > MMQ_MAX_SBW || (mt == 2 && sbw > 2)) // 4 x 32 tokens would not fit the registers
        return false;
    rg = MMQ_WAVES / ks;
    const int tiles = (rows + 15) / 16;
    if (rg > tiles)
        rg = tiles;
    while (rg > 1 && mmq_lds_bytes(cols, mt, rg, fused) > 64 * 1024)
        rg--;
    return mmq_lds_bytes(cols, mt, rg, fused) <= 64 * 1024;
}

// ---- Q8_0 / Q4_0 (32-value blocks) on the int8 matrix cores ----------------------
// Lane groups (consecutive vectors) of matrices that leave the streamed kernel
// too few waves.  A work group of MQ32_W waves per (16-row tile, 16 vectors);
// wave w takes the w-th share of the rows' 64-value spans.  Per span
// (blocks 2s and 2s + 1) lane quarter q4 holds 16 values of block 2s + q4/2
// -- A: token r16's activations, B: row r16's quants (Q4_0 as nibble - 8) --
// and two MFMAs over the span, each with the other block's quarters of the
// weights zeroed, give each block's integer dot for the 16 tokens: Q8_0
// sum w*x; Q4_0 sum (q - 8)*x, which is the reference's sum q*x - 8*sum x as
// one exact integer.  Each block's f32 tail (d * xd) * f32(isum)
// (ggml.zig:1212-1218, 1289-1290) goes to LDS; then every output sums its
// blocks in block order from +0 -- the reference's acc += r -- one thread
// per output.  A wave's loads run MQ32_AHEAD spans ahead; the tokens' block
// scales are staged in LDS once.
constexpr int MQ32_AHEAD = 4;
constexpr int MQ32_W = 8;         // waves per work group (span shares)
constexpr int MQ32_MAXS = 8;      // spans per wave: cols <= 4096
constexpr int MQ32_PART = 32768;  // LDS floats of block values: nb * 256

template <int T>
__global__ __launch_bounds__(64 * MQ32_W) void mmq32_kernel(DmmvParams p) {
    static_assert(T == LH_Q8_0 || T == LH_Q4_0, "32-value blocks");
    constexpr int QB = T == LH_Q8_0 ? 32 : 16; // quant bytes per block
    constexpr int NO = 256;                    // outputs per work group: (token, row)
    constexpr int MAXNB = 64 * MQ32_W * MQ32_MAXS / 32;
    __shared__ __align__(16) float part[MQ32_PART];      // [block][token * 16 + row]
    __shared__ __align__(16) float xds[16][MAXNB];       // the tokens' block scales
    const int ln = threadIdx.x & 63, r16 = ln & 15, q4 = ln >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int first = (int)blockIdx.y * 16; // this group's vectors: first .. first + n - 1
    const int n = min(16, p.ident_n - first), cols = p.cols, nb = cols / 32, ns = cols / 64;
    const int s_lo = wave * ns / MQ32_W, cnt = (wave + 1) * ns / MQ32_W - s_lo; // this wave's spans
    const int row0 = (int)blockIdx.x * 16;
    const int row = min(row0 + r16, p.rows - 1);
    const size_t U = (size_t)p.rows * nb;
    const uint8_t *wb = p.w;
    // A row r16 carries a vector (tokens past n repeat the last; their outputs are
    // never stored); this lane's outputs are tokens 4 q4 + i of row r16
    const int8_t *xr = p.xq + (size_t)(first + min(r16, n - 1)) * cols + 16 * q4;
    // the group's block scales, bound for LDS (row tk of xds: token tk's nb
    // scales; tokens past n repeat the last): thread (tk, part) loads blocks
    // xpart + TPT u of token tk, unconditionally from clamped indices, first;
    // they are stored after the first spans' loads are out, so that store
    // waits for these loads alone
    constexpr int TPT = 64 * MQ32_W / 16;       // threads per token
    constexpr int XU = (MAXNB + TPT - 1) / TPT; // scales per thread (at most)
    const int xtk = (int)threadIdx.x / TPT, xpart = (int)threadIdx.x % TPT;
    const float *xdr = p.xd + (size_t)(first + min(xtk, n - 1)) * nb;
    float xe[XU];
#pragma unroll
    for (int u = 0; u < XU; u++)
        xe[u] = xdr[min(xpart + TPT * u, nb - 1)];
    __builtin_amdgcn_sched_barrier(0);
    // block 2s + q4/2 of the lane's row: its 16 quant bytes (Q8_0: half q4 & 1;
    // Q4_0: all 16, the nibble half picked below) and the (d, d) pair of blocks 2s, 2s + 1
    const uint8_t *wq = wb + ((size_t)row * nb + (q4 >> 1)) * QB + (T == LH_Q8_0 ? 16 * (q4 & 1) : 0);
    const uint32_t *wd = (const uint32_t *)(wb + U * QB + (size_t)row * nb * 2);
    struct Span {
        mmq_i4 a, w;
        uint32_t d;
    };
    // span j of this wave (past its last: the last, loaded and not used)
    auto load = [&](int j, Span &o) {
        const int sc = s_lo + min(j, cnt - 1);
        o.w = *(const mmq_i4 *)(wq + (size_t)2 * sc * QB);
        o.d = wd[sc];
        o.a = *(const mmq_i4 *)(xr + 64 * sc);
    };
    const mmq_i4 z = {0, 0, 0, 0};
    const bool lo = q4 < 2;
    auto span = [&](const Span &o, int sc) {
        mmq_i4 wv = o.w;
        if constexpr (T == LH_Q4_0) {
            // the lane's nibble half, then q - 8 per byte: (q + 0x78) ^ 0x80
            const uint32_t sh = 4 * (q4 & 1);
#pragma unroll
            for (int e = 0; e < 4; e++)
                wv[e] = (int)((((uint32_t)wv[e] >> sh) & 0x0F0F0F0Fu) + 0x78787878u) ^ (int)0x80808080u;
        }
        const mmq_i4 wa = lo ? wv : z, wbk = lo ? z : wv;
        const float dwa = half_bits_to_float(o.d & 0xffffu), dwb = half_bits_to_float(o.d >> 16);
        const mmq_i4 da = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a, wa, z, 0, 0, 0);
        const mmq_i4 db = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a, wbk, z, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int tk = 4 * q4 + i;
            const float2 xd = *(const float2 *)&xds[tk][2 * sc];
            const float sa = dwa * xd.x;
            part[(size_t)(2 * sc) * NO + tk * 16 + r16] = sa * (float)da[i];
            const float sb = dwb * xd.y;
            part[(size_t)(2 * sc + 1) * NO + tk * 16 + r16] = sb * (float)db[i];
        }
    };
    // each span's loads are issued as a unit, in span order (the fences keep
    // them there), so a span's wait leaves the later spans' loads in flight
    Span ring[MQ32_AHEAD];
#pragma unroll
    for (int j = 0; j < MQ32_AHEAD; j++) {
        load(j, ring[j]);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < XU; u++)
        if (xpart + TPT * u < nb)
            xds[xtk][xpart + TPT * u] = xe[u];
    lds_barrier(); // the scales
#pragma unroll
    for (int j = 0; j < MQ32_MAXS; j++) {
        if (j < cnt)
            span(ring[j % MQ32_AHEAD], s_lo + j);
        __builtin_amdgcn_sched_barrier(0);
        if (j + MQ32_AHEAD < MQ32_MAXS)
            load(j + MQ32_AHEAD, ring[j % MQ32_AHEAD]);
        __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier(); // every block's values
    // output o = (token o / 16, row o % 16): its blocks in order from +0
    for (int o = (int)threadIdx.x; o < NO; o += 64 * MQ32_W) {
        const int tk = o >> 4, rr = o & 15;
        float acc = 0.0f;
#pragma unroll 8
        for (int bl = 0; bl < nb; bl++)
            acc = acc + part[(size_t)bl * NO + o];
        if (tk < n && row0 + rr < p.rows) {
            float *out = p.out + (size_t)(first + tk) * p.out_stride + row0 + rr;
            *out = p.accumulate ? *out + acc : acc;
        }
    }
}

static bool mmq32_supported(int t, int cols, bool fused) {
    // the block values of a work group fill (cols / 32) * 256 floats of LDS
    return (t == LH_Q8_0 || t == LH_Q4_0) && !fused && cols % 64 == 0 && cols >= 64 * MQ32_W &&
           cols <= 64 * MQ32_W * MQ32_MAXS && (size_t)(cols / 32) * 256 <= (size_t)MQ32_PART;
}

// p.ident_n vectors in groups of 16.
static void launch_mmq32(int t, const DmmvParams &p, hipStream_t st) {
    const dim3 grid((p.rows + 15) / 16, (p.ident_n + 15) / 16), block(64 * MQ32_W);
    if (t == LH_Q8_0)
        hipLaunchKernelGGL(mmq32_kernel<LH_Q8_0>, grid, block, 0, st, p);
    else
        hipLaunchKernelGGL(mmq32_kernel<LH_Q4_0>, grid, block, 0, st, p);
}

// ---- many vectors: a 64-row x 128-vector tile per work group -----------------------
// Prefill-sized lane groups (Q4_K / Q6_K).  mmw_kernel decodes a row tile's
// weights once per 16 vectors; here eight waves share one decode per 128.  Each
// thread turns 32 weights of a block into two int8 digits of scale * quant
// (128 a + b: Q4_K sc * q <= 945, Q6_K sc * (q - 32) in 14 bits) in LDS, beside
// the vectors' int8 columns, and each wave forms 32 rows x 32 vectors with
// unmasked MFMAs: isum = 128 sum(a x) + sum(b x), exact in any order; Q4_K's mins
// on one f16 MFMA, as in mmw_kernel.  No multiply per (vector, scale group) is
// left.  Blocks are taken in order, each output one f32 register -- the
// reference's `acc += r`.  The LDS (154 KB, one work group per CU) holds two
// blocks: one is decoded while the other is multiplied and the third's loads
// are in flight, one barrier per block; the two waves of a SIMD run decode
// and multiply in opposite order (3% over the same order).
// Bound by issue, ~4800 cycles of a SIMD per block: 2 x (36 MFMAs at 16, 280
// VALU ops at ~4), the rest LDS reads and waits.  Q4_K 4096 x 2048 at 512 vectors
// 30.2 -> 23.5 us, Q6_K 33.8 -> 21.8; 4096 x 8192 at 512 99 -> 71 and 157 -> 64.  A
// 32 x 64 tile (two groups per CU) took 33.2 / 32.2 at 4096 x 2048.
constexpr int MMP_R = 64, MMP_T = 128, MMP_W = 8, MMP_ROW = 256 + 16;
struct MmpLds {
    int8_t wh[MMP_R * MMP_ROW], wl[MMP_R * MMP_ROW]; // digits, value order
    int8_t x[MMP_T * MMP_ROW];
    _Float16 bs[MMP_T * 20]; // 16 sums per vector
    _Float16 mn[MMP_R * 10]; // 8 mins per row
    float d[MMP_R * 2];      // (d, dmin) per row
    float xd[MMP_T];
};

template <int T>
__global__ __launch_bounds__(64 * MMP_W, 2) void mmp_kernel(DmmvParams p) {
    extern __shared__ __align__(16) uint8_t sh[];
    constexpr bool K4 = T == LH_Q4_K;
    MmpLds *buf = (MmpLds *)sh;
    const int n = p.ident_n, cols = p.cols, nb = cols / 256, tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = tid & 63, r16 = ln & 15, q4 = ln >> 4;
    const int row0 = (int)blockIdx.x * MMP_R, tok0 = (int)blockIdx.y * MMP_T;
    // this thread's share of a block: 16 bytes of quants of one row, four 16-byte
    // pieces of the vectors' columns, four sums
    const int wr = tid >> 3, wc = tid & 7;
    const size_t U = (size_t)p.rows * nb, wrow = (size_t)min(row0 + wr, p.rows - 1) * nb;
    const int8_t *xp[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        xp[i] = p.xq + (size_t)p.pair_src[min(tok0 + 32 * i + (tid >> 4), n - 1)] * cols + 16 * (tid & 15);
    const int32_t *sp = p.xs + (size_t)p.pair_src[min(tok0 + (tid >> 2), n - 1)] * (cols / 16) + 4 * (tid & 3);
    const float *dp = p.xd + (size_t)p.pair_src[min(tok0 + (tid & (MMP_T - 1)), n - 1)] * nb;
    struct Raw {
        mmq_i4 q, h, s; // quants; Q4_K the header, Q6_K the high bits; the vector's sums (Q4_K) or the scales (Q6_K)
        mmq_i4 x[4];
        float xd;
        uint32_t d;
    } raw;
    auto fetch = [&](int b) {
        const size_t u = wrow + b;
        if constexpr (K4) {
            raw.q = *(const mmq_i4 *)(p.w + u * 144 + 16 + 16 * wc);
            raw.h = *(const mmq_i4 *)(p.w + u * 144);
            raw.s = *(const mmq_i4 *)(sp + 16 * b);
        } else {
            raw.q = *(const mmq_i4 *)(p.w + u * 128 + 16 * wc);
            raw.h = *(const mmq_i4 *)(p.w + U * 128 + u * 64 + 32 * (wc >> 2) + 16 * (wc & 1));
            raw.s = *(const mmq_i4 *)(p.w + U * 192 + u * 16);
            raw.d = *(const uint16_t *)(p.w + U * 208 + u * 2);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            raw.x[i] = *(const mmq_i4 *)(xp[i] + 256 * b);
        raw.xd = dp[b];
    };
    auto decode = [&](MmpLds &l) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            *(mmq_i4 *)(l.x + (32 * i + (tid >> 4)) * MMP_ROW + 16 * (tid & 15)) = raw.x[i];
        if (tid < MMP_T)
            l.xd[tid] = raw.xd;
        mmq_i4 h0, l0, h1, l1; // the 16 low-nibble values' digits, the 16 high-nibble ones'
        int k0, k1;            // their first value's place in the block
        if constexpr (K4) {
            const uint32_t a = raw.h[1], m = raw.h[2], c = raw.h[3];
            const int p2 = wc >> 1; // groups 2 p2, 2 p2 + 1
            const uint32_t scv = p2 < 2 ? a & 0x3F3F3F3Fu : (c & 0x0F0F0F0Fu) | ((a >> 2) & 0x30303030u);
            const uint32_t scs = scv >> (16 * (p2 & 1));
            const short s0 = (short)(scs & 0xFF), s1 = (short)((scs >> 8) & 0xFF);
            const mmq_s2 z2 = {0, 0};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                int hi, lo;
                q6k_digits((uint32_t)raw.q[e] & 0x0F0F0F0Fu, mmq_s2{s0, s0}, z2, hi, lo);
                h0[e] = hi, l0[e] = lo;
                q6k_digits(((uint32_t)raw.q[e] >> 4) & 0x0F0F0F0Fu, mmq_s2{s1, s1}, z2, hi, lo);
                h1[e] = hi, l1[e] = lo;
            }
            k0 = 64 * p2 + 16 * (wc & 1);
            k1 = k0 + 32;
            // min of group wc, the row's (d, dmin), the vector's sums
            const uint32_t mv = wc < 4 ? m & 0x3F3F3F3Fu : ((c >> 4) & 0x0F0F0F0Fu) | ((m >> 2) & 0x30303030u);
            l.mn[10 * wr + wc] = (_Float16)(unsigned short)((mv >> (8 * (wc & 3))) & 0xFF);
            if (wc == 0) {
                l.d[2 * wr] = half_bits_to_float((uint32_t)raw.h[0] & 0xffff);
                l.d[2 * wr + 1] = half_bits_to_float((uint32_t)raw.h[0] >> 16);
            }
            *(mmq_h4 *)(l.bs + 20 * (tid >> 2) + 4 * (tid & 3)) =
                mmq_h4{(_Float16)(short)raw.s[0], (_Float16)(short)raw.s[1], (_Float16)(short)raw.s[2],
                       (_Float16)(short)raw.s[3]};
        } else {
            const int h = wc >> 2, qa = (wc >> 1) & 1, r = wc & 1; // quarters qa and qa + 2 of half h, run r
            const uint32_t s01 = h ? (uint32_t)raw.s[2] : (uint32_t)raw.s[0]; // scales 8h .. 8h + 3
            const uint32_t s23 = h ? (uint32_t)raw.s[3] : (uint32_t)raw.s[1]; // 8h + 4 .. 8h + 7
            const short s0 = (short)(int8_t)((s01 >> (8 * (2 * qa + r))) & 0xFF);
            const short s1 = (short)(int8_t)((s23 >> (8 * (2 * qa + r))) & 0xFF);
            mmq_s2 o0 = mmq_s2{s0, s0} * (short)-32, o1 = mmq_s2{s1, s1} * (short)-32;
            asm("" : "+v"(o0), "+v"(o1));
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t ql = (uint32_t)raw.q[e], qh = (uint32_t)raw.h[e];
                int hi, lo;
                q6k_digits((ql & 0x0F0F0F0Fu) | (((qh >> (2 * qa)) & 0x03030303u) << 4), mmq_s2{s0, s0}, o0, hi, lo);
                h0[e] = hi, l0[e] = lo;
                q6k_digits(((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (4 + 2 * qa)) & 0x03030303u) << 4), mmq_s2{s1, s1}, o1,
                           hi, lo);
                h1[e] = hi, l1[e] = lo;
            }
            k0 = 128 * h + 32 * qa + 16 * r;
            k1 = k0 + 64;
            if (wc == 0)
                l.d[2 * wr] = half_bits_to_float(raw.d);
        }
        *(mmq_i4 *)(l.wh + wr * MMP_ROW + k0) = h0;
        *(mmq_i4 *)(l.wl + wr * MMP_ROW + k0) = l0;
        *(mmq_i4 *)(l.wh + wr * MMP_ROW + k1) = h1;
        *(mmq_i4 *)(l.wl + wr * MMP_ROW + k1) = l1;
    };
    const int wrow0 = 32 * (wave & 1), wtok0 = 32 * (wave >> 1); // this wave's 32 x 32
    float acc[2][2][4] = {};
    const mmq_i4 z = {0, 0, 0, 0};
    auto multiply = [&](const MmpLds &l) {
        mmq_i4 ah[2][2], al[2][2];
        mmq_f4 ms[2][2];
        if constexpr (K4) {
            mmq_h4 bs[2], mn[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                bs[i] = *(const mmq_h4 *)(l.bs + 20 * (wtok0 + 16 * i + r16) + 4 * q4);
                const _Float16 *m = l.mn + 10 * (wrow0 + 16 * i + r16) + 2 * q4;
                mn[i] = mmq_h4{m[0], m[0], m[1], m[1]};
            }
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 2; r++)
                    ms[t][r] = __builtin_amdgcn_mfma_f32_16x16x16f16(bs[t], mn[r], mmq_f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            mmq_i4 xa[2], bh[2], bl[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                xa[i] = *(const mmq_i4 *)(l.x + (wtok0 + 16 * i + r16) * MMP_ROW + 64 * s + 16 * q4);
                bh[i] = *(const mmq_i4 *)(l.wh + (wrow0 + 16 * i + r16) * MMP_ROW + 64 * s + 16 * q4);
                bl[i] = *(const mmq_i4 *)(l.wl + (wrow0 + 16 * i + r16) * MMP_ROW + 64 * s + 16 * q4);
            }
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    ah[t][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[t], bh[r], s ? ah[t][r] : z, 0, 0, 0);
                    al[t][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[t], bl[r], s ? al[t][r] : z, 0, 0, 0);
                }
        }
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const float2 d = *(const float2 *)(l.d + 2 * (wrow0 + 16 * r + r16));
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const float4 v = *(const float4 *)(l.xd + wtok0 + 16 * t + 4 * q4);
                const float xd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float is = (float)((ah[t][r][i] << 7) + al[t][r][i]);
                    if constexpr (K4) {
                        // xb.d * (d * f32(isum) - dmin * f32(min_isum))  (ggml.zig:1016-1017)
                        const float aa = d.x * is, bb = d.y * ms[t][r][i];
                        acc[t][r][i] = acc[t][r][i] + xd[i] * (aa - bb);
                    } else {
                        // xb.d * dec.d * f32(isum)  (ggml.zig:1019)
                        const float s = xd[i] * d.x;
                        acc[t][r][i] = acc[t][r][i] + s * is;
                    }
                }
            }
        }
    };
    fetch(0);
    decode(buf[0]);
    fetch(min(1, nb - 1));
    lds_barrier();
    for (int b = 0; b < nb; b++) {
        if (wave >= MMP_W / 2)
            multiply(buf[b & 1]);
        if (b + 1 < nb) { // the other buffer's readers passed the last barrier
            decode(buf[(b + 1) & 1]);
            fetch(min(b + 2, nb - 1)); // past the last block: the last one again, not used
        }
        if (wave < MMP_W / 2)
            multiply(buf[b & 1]);
        lds_barrier();
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int tok = tok0 + wtok0 + 16 * t + 4 * q4 + i, row = row0 + wrow0 + 16 * r + r16;
                if (tok >= n || row >= p.rows)
                    continue;
                float *o = p.out + (size_t)tok * p.out_stride + row;
                *o = p.accumulate ? *o + acc[t][r][i] : acc[t][r][i];
            }
}

template <int T>
static void mmp_launch_t(const DmmvParams &p, hipStream_t st) {
    const dim3 grid((p.rows + MMP_R - 1) / MMP_R, (p.ident_n + MMP_T - 1) / MMP_T);
    hipLaunchKernelGGL(mmp_kernel<T>, grid, dim3(64 * MMP_W), 2 * sizeof(MmpLds), st, p);
}

// ---- Q8_0 / Q4_0 streamed in block order ------------------------------------------
// mmw_kernel's shape for 32-value blocks: a wave owns 16 rows for up to 16
// tokens of a group and walks them in units of 8 blocks (256 columns),
// weights loaded in address order and turned through its LDS, two units in
// registers or in flight.  A 64-deep MFMA spans two blocks; its A rows are
// (token, block) pairs (8 tokens a set, zeros on the other block's quarters),
// so one MFMA over the unmasked weights gives both blocks' integer dots of 8
// tokens, and the tails (d * xd) * f32(isum) add in block order.  Q4_0's
// weights enter as nibble - 8, the reference's sum q*x - 8*sum x as one exact
// integer.  Bound by the weights' bytes at few tokens and by the four VALU
// operations of each (token, row, block)'s tail at 16.
// Measured (us per launch, events; dot4 / this): experts 2048 -> 768 fused
// over 64 planes at 4 tokens each Q4_0 65 / 33, Q8_0 76 / 72, at 10 182 / 38
// and 185 / 87; 768 -> 2048 at 10 57 / 22 and 92 / 29; 11008 x 4096 Q8_0 at
// 32 vectors 126 / 31.
template <int T> struct Mmw32Blk {
    static constexpr bool Q8 = T == LH_Q8_0;
    static constexpr int QB = Q8 ? 32 : 16;          // quant bytes per block
    static constexpr int CH = Q8 ? 16 : 8;           // 16-byte chunks per row and unit
    static constexpr int NL = Q8 ? 4 : 2;            // loads: 64 / CH rows each
    static constexpr int ROWB = 16 * CH + 16;        // odd chunk stride in LDS
    static constexpr int BYTES = 16 * ROWB + 256;    // then the scales, f16 [row][8]
    mmq_i4 v[NL];
    uint32_t d0, d1; // blocks 2 * (ln & 3), + 1 of row ln / 4
    struct Src {
        const uint8_t *q, *d;
        uint32_t row[NL], drow; // byte offset of the lane's row per load; block index of row ln / 4
    };
    __device__ __forceinline__ static Src src(const uint8_t *wb, int rows, int nb, int row0, int ln) {
        Src s;
        s.q = wb;
        s.d = wb + (size_t)rows * nb * QB;
#pragma unroll
        for (int i = 0; i < NL; i++)
            s.row[i] = (uint32_t)min(row0 + (64 / CH) * i + ln / CH, rows - 1) * (uint32_t)(nb * QB);
        s.drow = (uint32_t)min(row0 + (ln >> 2), rows - 1) * (uint32_t)nb;
        return s;
    }
    // unit u: chunks and blocks past the row's end read its last ones
    __device__ __forceinline__ void load(const Src &s, int u, int nb, int ln) {
        const uint32_t c = 16u * (uint32_t)min(CH * u + ln % CH, nb * QB / 16 - 1);
#pragma unroll
        for (int i = 0; i < NL; i++)
            v[i] = *(const mmq_i4 *)(s.q + (s.row[i] + c));
        const int b = 8 * u + 2 * (ln & 3);
        d0 = *(const uint16_t *)(s.d + 2u * (s.drow + min(b, nb - 1)));
        d1 = *(const uint16_t *)(s.d + 2u * (s.drow + min(b + 1, nb - 1)));
    }
    __device__ __forceinline__ void store(uint8_t *l, int ln) const {
#pragma unroll
        for (int i = 0; i < NL; i++)
            *(mmq_i4 *)(l + ((64 / CH) * i + ln / CH) * ROWB + 16 * (ln % CH)) = v[i];
        *(uint32_t *)(l + 16 * ROWB + 4 * ln) = d0 | (d1 << 16);
    }
};

template <int T> struct Mmw32Tile {
    mmq_i4 q[4], d; // MFMA s: blocks 2s, 2s + 1; the row's eight f16 scales
    __device__ __forceinline__ static Mmw32Tile read(const uint8_t *l, int r16, int q4) {
        using B = Mmw32Blk<T>;
        Mmw32Tile w;
#pragma unroll
        for (int s = 0; s < 4; s++)
            w.q[s] = *(const mmq_i4 *)(l + r16 * B::ROWB + (B::Q8 ? 64 * s + 16 * q4 : 32 * s + 16 * (q4 >> 1)));
        w.d = *(const mmq_i4 *)(l + 16 * B::ROWB + 16 * r16);
        return w;
    }
};

// One unit (nbu <= 8 blocks): acc[set][token pair] += its blocks' tails in order.
// xs: the unit's scales, [MFMA s][token pair of both sets][token][block].
template <int T>
__device__ __forceinline__ void mmw32_acc(const Mmw32Tile<T> &w, int q4, int ns, int nbu, const mmq_i4 (&xa)[2][4],
                                          const float4 *xs, float (&acc)[2][2]) {
    const mmq_i4 z = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        if (2 * s >= nbu)
            break;
        mmq_i4 wv = w.q[s];
        if constexpr (T == LH_Q4_0) { // the lane's nibble half, then q - 8 per byte: (q + 0x78) ^ 0x80
            const uint32_t sh = 4 * (q4 & 1);
#pragma unroll
            for (int e = 0; e < 4; e++)
                wv[e] = (int)((((uint32_t)wv[e] >> sh) & 0x0F0F0F0Fu) + 0x78787878u) ^ (int)0x80808080u;
        }
        const float da = half_bits_to_float((uint32_t)w.d[s] & 0xffffu), db = half_bits_to_float((uint32_t)w.d[s] >> 16);
        const bool two = 2 * s + 1 < nbu;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if (t >= ns)
                break;
            const mmq_i4 dq = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[t][s], wv, z, 0, 0, 0);
            const float4 xd = xs[8 * s + 4 * t + q4];
            // d * xd * f32(dot)  (ggml.zig:1212-1218, 1289-1290)
            const float a0 = da * xd.x, a1 = da * xd.z;
            acc[t][0] = acc[t][0] + a0 * (float)dq[0];
            acc[t][1] = acc[t][1] + a1 * (float)dq[2];
            if (two) {
                const float b0 = db * xd.y, b1 = db * xd.w;
                acc[t][0] = acc[t][0] + b0 * (float)dq[1];
                acc[t][1] = acc[t][1] + b1 * (float)dq[3];
            }
        }
    }
}

// LDS: (XL: per work group; else per wave) the tokens' rows [16][xrow], 256
// zeros, the scales [units][32] float4; per wave a unit of 16 weight rows.
template <bool XL> __host__ __device__ constexpr int mmw32_xrow(int nb) { return (XL ? 32 * nb : 256) + 16; }
template <bool XL> __host__ __device__ constexpr int mmw32_xbytes(int nb) {
    return 16 * mmw32_xrow<XL>(nb) + 256 + (XL ? (nb + 7) / 8 : 1) * 512;
}

template <int T, bool FUSED, bool XL, int OCC>
__global__ __launch_bounds__(64 * MMW_W, OCC) void mmw32_kernel(DmmvParams p) {
    extern __shared__ __align__(16) uint8_t sh[];
    using B = Mmw32Blk<T>;
    constexpr int TOK = 16, M = FUSED ? 2 : 1, W = MMW_W;
    const bool ident = p.ident_n > 0;
    const int gi = blockIdx.y;
    DmmvGroup grp;
    if (ident) {
        grp.plane = 0;
        grp.first = gi * TOK;
        grp.n = min(TOK, p.ident_n - grp.first);
    } else {
        const int ng = p.n_groups_dev ? *p.n_groups_dev : p.n_groups;
        if (gi >= ng)
            return;
        grp = p.groups[gi];
    }
    const int n = grp.n, ns = (n + 7) / 8; // sets of 8 tokens
    const int cols = p.cols, nb = cols / 32, nu = (nb + 7) / 8;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    const int r16 = ln & 15, q4 = ln >> 4;
    const int row0 = ((int)blockIdx.x * W + wave) * 16;
    const int xrow = mmw32_xrow<XL>(nb), xbytes = mmw32_xbytes<XL>(nb);
    uint8_t *wls = sh + (XL ? xbytes + wave * B::BYTES : wave * (xbytes + B::BYTES));
    uint8_t *xl = XL ? sh : wls + B::BYTES;
    uint8_t *zl = xl + TOK * xrow;
    float *xds = (float *)(zl + 256);
    // where token t's scale of block b goes: float4 (unit, MFMA, set, pair), element (token, block)
    auto xd_at = [&](int t, int b) {
        return (XL ? (b >> 3) * 128 : 0) + ((b >> 1) & 3) * 32 + (t >> 3) * 16 + ((t >> 1) & 3) * 4 + (t & 1) * 2 + (b & 1);
    };
    // the vector of the group's t-th token (past n: the last); group_src needs no group
    const int *tab = p.group_src ? p.group_src + (size_t)gi * p.group_stride : p.pair_src + grp.first;
    const int tmax = p.group_src ? TOK - 1 : n - 1;
    auto vec_of = [&](int t) { return tab[min(t, tmax)]; };
    typename B::Src src[M];
    src[0] = B::src(p.w + (size_t)grp.plane * p.plane_bytes, p.rows, nb, row0, ln);
    if constexpr (FUSED)
        src[1] = B::src(p.w2 + (size_t)grp.plane * p.plane_bytes, p.rows, nb, row0, ln);
    struct Stage {
        B w[M];
        mmq_i4 x[XL ? 1 : 4]; // (not XL) tokens 4 i + ln / 16, chunk ln % 16
        float xd[2];          // tokens ln / 8, 8 + ln / 8, block ln % 8
    } st[2];
    const int8_t *xr[4];
    const float *xdr[2];
    if constexpr (!XL) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            xr[i] = p.xq + (size_t)vec_of(4 * i + (ln >> 4)) * cols;
#pragma unroll
        for (int i = 0; i < 2; i++)
            xdr[i] = p.xd + (size_t)vec_of(8 * i + (ln >> 3)) * nb;
    }
    auto load = [&](Stage &s, int u) {
        s.w[0].load(src[0], u, nb, ln);
        if constexpr (FUSED)
            s.w[1].load(src[1], u, nb, ln);
        if constexpr (!XL) {
            const int c = 16 * min(16 * u + (ln & 15), 2 * nb - 1), b = min(8 * u + (ln & 7), nb - 1);
#pragma unroll
            for (int i = 0; i < 4; i++)
                s.x[i] = *(const mmq_i4 *)(xr[i] + c);
#pragma unroll
            for (int i = 0; i < 2; i++)
                s.xd[i] = xdr[i][b];
        }
    };
    auto commit = [&](const Stage &s, int m) { // matrix m's unit to this wave's LDS
        wave_lds_sync();
        s.w[m].store(wls, ln);
        if constexpr (!XL)
            if (m == 0) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    *(mmq_i4 *)(xl + (4 * i + (ln >> 4)) * xrow + 16 * (ln & 15)) = s.x[i];
#pragma unroll
                for (int i = 0; i < 2; i++)
                    xds[xd_at(8 * i + (ln >> 3), ln & 7)] = s.xd[i];
            }
        wave_lds_sync();
    };
    if constexpr (XL) {
        // nb <= 64: four token rows per wave, all their loads before the weights' and the
        // stores behind them, so one round trip covers the staging
        int v[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            v[i] = vec_of(4 * wave + i);
        const int c0 = min(ln, 2 * nb - 1), c1 = min(64 + ln, 2 * nb - 1), cb = min(ln, nb - 1);
        mmq_i4 x0[4], x1[4];
        float xd[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            x0[i] = *(const mmq_i4 *)(p.xq + (size_t)v[i] * cols + 16 * c0);
            x1[i] = *(const mmq_i4 *)(p.xq + (size_t)v[i] * cols + 16 * c1);
            xd[i] = p.xd[(size_t)v[i] * nb + cb];
        }
        __builtin_amdgcn_sched_barrier(0);
        load(st[0], 0);
        load(st[1], min(1, nu - 1));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint8_t *l = xl + (size_t)(4 * wave + i) * xrow;
            if (ln < 2 * nb)
                *(mmq_i4 *)(l + 16 * ln) = x0[i];
            if (64 + ln < 2 * nb)
                *(mmq_i4 *)(l + 16 * (64 + ln)) = x1[i];
            if (ln < nb)
                xds[xd_at(4 * wave + i, ln)] = xd[i];
        }
        if (threadIdx.x < 16)
            *(mmq_i4 *)(zl + 16 * threadIdx.x) = mmq_i4{0, 0, 0, 0};
    } else {
        load(st[0], 0);
        load(st[1], min(1, nu - 1));
        if (ln < 16)
            *(mmq_i4 *)(zl + 16 * ln) = mmq_i4{0, 0, 0, 0};
    }
    lds_barrier();
    // A row r16 = (token r16/2 of the set, block r16&1 of the span): live on the
    // block's quarters, zeros elsewhere
    const bool live = (q4 >> 1) == (r16 & 1);
    const int xstep = XL && live ? 256 : 0;
    const uint8_t *xt[2] = {live ? xl + (r16 / 2) * xrow + 16 * q4 : zl, live ? xl + (8 + r16 / 2) * xrow + 16 * q4 : zl};
    float acc[M][2][2] = {};
    // as mmw_kernel's step: the next tile is stored to LDS and read back under the arithmetic
    commit(st[0], 0);
    Mmw32Tile<T> w0 = Mmw32Tile<T>::read(wls, r16, q4);
    auto step = [&](int u, Stage &cur, const Stage &nxt) {
        const int nbu = min(8, nb - 8 * u);
        mmq_i4 xa[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if (t >= ns)
                break;
#pragma unroll
            for (int s = 0; s < 4; s++) // (past the row's end: staged bytes of its clamped loads, or LDS never used)
                xa[t][s] = *(const mmq_i4 *)(xt[t] + (2 * s < nbu ? u * xstep + 64 * s : 0));
        }
        Mmw32Tile<T> w1;
        const float4 *xsp = (const float4 *)(xds + (XL ? u * 128 : 0));
        if constexpr (FUSED) {
            commit(cur, 1);
            w1 = Mmw32Tile<T>::read(wls, r16, q4);
            load(cur, min(u + 2, nu - 1)); // past the last unit: the last one again, not used
            __builtin_amdgcn_sched_barrier(0);
            mmw32_acc<T>(w0, q4, ns, nbu, xa, xsp, acc[0]);
            if constexpr (XL) {
                commit(nxt, 0);
                w0 = Mmw32Tile<T>::read(wls, r16, q4);
                mmw32_acc<T>(w1, q4, ns, nbu, xa, xsp, acc[M - 1]);
            } else { // the unit's scales share the commit's LDS: after their last use
                mmw32_acc<T>(w1, q4, ns, nbu, xa, xsp, acc[M - 1]);
                commit(nxt, 0);
                w0 = Mmw32Tile<T>::read(wls, r16, q4);
            }
        } else {
            if constexpr (XL) {
                commit(nxt, 0);
                w1 = Mmw32Tile<T>::read(wls, r16, q4);
                load(cur, min(u + 2, nu - 1));
                __builtin_amdgcn_sched_barrier(0);
                mmw32_acc<T>(w0, q4, ns, nbu, xa, xsp, acc[0]);
                w0 = w1;
            } else {
                load(cur, min(u + 2, nu - 1));
                __builtin_amdgcn_sched_barrier(0);
                mmw32_acc<T>(w0, q4, ns, nbu, xa, xsp, acc[0]);
                commit(nxt, 0);
                w0 = Mmw32Tile<T>::read(wls, r16, q4);
            }
        }
    };
    for (int u = 0; u < nu; u += 2) {
        step(u, st[0], st[1]);
        if (u + 1 >= nu)
            break;
        step(u + 1, st[1], st[0]);
    }
    const int row = row0 + r16;
    if (row >= p.rows)
        return;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int jj = 0; jj < 2; jj++) {
            const int k = 8 * t + 2 * q4 + jj;
            if (k >= n)
                continue;
            const float v = FUSED ? swiglu1(acc[0][t][jj], acc[M - 1][t][jj]) : acc[0][t][jj];
            const int dst = ident || p.pos_ident ? grp.first + k : p.pair_dst[grp.first + k];
            float *o = p.out + (size_t)dst * p.out_stride + row;
            *o = p.accumulate ? *o + v : v;
        }
}

template <int T, bool FUSED>
static void mmw32_launch_t(const DmmvParams &p, hipStream_t st) {
    const int groups = p.ident_n > 0 ? (p.ident_n + 15) / 16 : p.n_groups, nb = p.cols / 32;
    const dim3 grid(((p.rows + 15) / 16 + MMW_W - 1) / MMW_W, groups), block(64 * MMW_W);
    // waves per SIMD as registers (and for Q8_0 gate/up the LDS) allow
    constexpr int OCC_XL = FUSED && T == LH_Q8_0 ? 2 : 3, OCC = FUSED ? 2 : 3;
    if (p.cols <= MMW_XL_COLS)
        hipLaunchKernelGGL((mmw32_kernel<T, FUSED, true, OCC_XL>), grid, block,
                           (mmw32_xbytes<true>(nb) + MMW_W * Mmw32Blk<T>::BYTES), st, p);
    else
        hipLaunchKernelGGL((mmw32_kernel<T, FUSED, false, OCC>), grid, block,
                           (MMW_W * (mmw32_xbytes<false>(nb) + Mmw32Blk<T>::BYTES)), st, p);
}

static bool is_k(int t) { return t == LH_Q4_K || t == LH_Q6_K; }

// The one-shot kernels' shapes: K-quants in MmqOps registers and LDS sums,
// 32-value blocks in mmq32_kernel's.
static bool mmq_oneshot(int t, int cols, int max_tok, bool fused) {
    if (!is_k(t))
        return mmq32_supported(t, cols, fused);
    if (cols % 256 || cols < 256 || max_tok < 1 || max_tok > 32)
        return false;
    if (fused && t != LH_Q4_K) // a fused pair is gate/up: Q4_K only here
        return false;
    int rg, ks, sbw;
    return mmq_shape(16, cols, (max_tok + 15) / 16, fused, rg, ks, sbw);
}

// The streamed kernels' shapes: whole blocks, the K-quants' block scales of 16
// tokens in the CU's LDS (Q4_K to 532480 columns, Q6_K to 531456; groups of 32
// end at 4096, the 32-value blocks hold one unit's), byte offsets in 32 bits.
constexpr size_t MMW_LDS_MAX = 160 * 1024;
static bool mmw_shape(int t, int rows, int cols, bool fused) {
    if ((t != LH_Q4_K && t != LH_Q6_K && t != LH_Q8_0 && t != LH_Q4_0) || cols < block_elems(t) ||
        cols % block_elems(t) || (fused && t == LH_Q6_K))
        return false;
    if (is_k(t) && (t == LH_Q4_K ? mmw_lds<LH_Q4_K, 1, false>(cols) : mmw_lds<LH_Q6_K, 1, false>(cols)) > MMW_LDS_MAX)
        return false;
    return (size_t)rows * (cols / block_elems(t)) * block_bytes(t) < ((size_t)1 << 32);
}

// (row tile, 16 lanes) pairs of a lane-group launch: the waves the streamed kernels run.
static long lane_pairs(int rows, int n) { return (long)((rows + 15) / 16) * ((n + 15) / 16); }

// Lane groups from MMW_MIN_WAVES pairs on (512 for a fused pair, twice the
// bytes per wave) take the streamed kernel, below that the one-shot kernel
// (8 waves to a row tile) where it serves the shape: too few waves stream.
// Measured, us per launch, one-shot / streamed: Q4_K 8192 x 4096 at 16 lanes
// (512 pairs) 14.4 / 15.1, at 32 (1024) 22.6 / 15.8; 7168 x 2048 at 24 (896)
// 13.1 / 9.8; Q6_K 16384 x 4096 at 16 (1024) 32.7 / 20.6; fused 2048 x 7168 at
// 24 (256) 25.6 / 32.1, at 64 (512) 44.8 / 32.6; fused 4096 x 2048 at 24 (512)
// 12.7 / 13.2, at 64 (1024) 20.4 / 14.0.
// The 32-value blocks' one-shot kernel fills a CU's LDS, so it takes one round
// of the chip per 256 pairs; rows of up to 1536 columns stream as fast as two
// rounds, of 2048 as three.  us per call, dot4 / one-shot / streamed: Q4_0 4096
// x 1024 at 24 (512 pairs) 14.1 / 14.5 / 10.1, 2500 x 1536 at 32 (314) 14.2 /
// 15.3 / 12.3, 2500 x 1984 at 32 13.8 / 11.8 / 14.4, at 63 (628) 22.1 / 15.8 /
// 14.6, 4096 x 4096 at 24 (512) 32.3 / 17.6 / 26.1.
constexpr long MMW_MIN_WAVES = 768, MMW_MIN_WAVES_FUSED = 512;
static bool lanes_streamed(int t, int rows, int cols, int n, bool fused) {
    const long pairs = lane_pairs(rows, n);
    if (!mmw_shape(t, rows, cols, fused))
        return false;
    if (!is_k(t) && !fused && ((cols <= 1536 && pairs > 256) || (cols <= MMW_XL_COLS && pairs > 512)))
        return true;
    return pairs >= (fused ? MMW_MIN_WAVES_FUSED : MMW_MIN_WAVES);
}

// Expert groups of K-quants with fewer (group, row tile, matrix) streams than
// this take the one-shot kernel: the groups the launch has room for, a little
// over nine streams per CU.  Measured, us per layer, one-shot / streamed gate/up
// and down: 1024 x 512 x 32 top-4 Q4_K + Q6_K at 16 tokens (2304 streams each)
// 32.3 / 34.4, at 19 33.9 / 35.6, at 24 (2432) 37.2 / 37.0, at 128 (4096) 49.7 /
// 45.9; 1024 x 1024 x 32 top-4 at 16 (4608 and 2304) 36.4 / 37.1; 1024 x 768 x 64 top-6
// at 16 (6720 and 4480) 43.3 / 43.8, at 24 44.8 / 44.5; 1536 x 768 x 64 top-6 at 5
// (2976 and 2976) 45.3 / 41.5; 2048 x 768 x 128 top-8 at 10 (8160 and 10880) 59.5 /
// 51.5.  The 32-value blocks have no grouped one-shot form.
constexpr long MMW_MIN_GROUP_STREAMS = 2400;
static bool groups_few(int t, int rows, int n_groups, bool fused) {
    return is_k(t) && (long)n_groups * ((rows + 15) / 16) * (fused ? 2 : 1) < MMW_MIN_GROUP_STREAMS;
}

// Lane groups that fill mmp_kernel's 64 x 128 tiles and whole rounds of the
// chip's 256 CUs with them: the pairs that the launch holds over those that its
// rounds could (256 tiles of 32).  A round costs mmp_kernel the same however few
// of its CUs work; Q4_K breaks even at ~3/4, Q6_K at ~3/5.  Measured, us, streamed /
// this: Q4_K 4096 x 2048 at 256 (half a round) 18.7 / 21.8, 8192 x 1024 at 256 (one)
// 18.5 / 14.7, 16384 x 2048 at 192 (3/4) 38.4 / 40.6, at 256 (two rounds) 48.0 / 41.1;
// Q6_K 20.1 / 20.0, 20.1 / 13.9, 43.9 / 37.1, 55.2 / 37.6.
static bool lanes_tiled(int t, int rows, int cols, int n) {
    if (!is_k(t) || !mmw_shape(t, rows, cols, false))
        return false;
    const long tiles = (long)((rows + MMP_R - 1) / MMP_R) * ((n + MMP_T - 1) / MMP_T);
    const long room = (tiles + 255) / 256 * 256 * (MMP_R / 16) * (MMP_T / 16);
    return t == LH_Q4_K ? lane_pairs(rows, n) * 5 >= room * 4 : lane_pairs(rows, n) * 3 >= room * 2;
}

// Q8_0 / Q4_0: whether the matrix cores take n vectors against one matrix from
// the dot4 matvec.  us per call (quantization and matmul, back to back in a
// graph, weights from a ring past the caches), dot4 / matrix cores.
// One-shot shapes (whole 64-value spans, 512 to 4096 columns): the kernel costs
// about the same for any matrix of one round, a little less where a row's
// bytes are no multiple of the 128-byte line; the dot4 matvec's time grows
// with the row length, and with n * rows * cols once the chip is full.
//   8 vectors and up, over 2048 columns, or over 1024 for Q8_0 or rows off the
//     line: 300 x 3072 at 8 Q4_0 11.6 / 9.2, Q8_0 12.4 / 9.3; 200 x 4096 at 16
//     12.6 / 10.5 and 15.8 / 10.6; Q8_0 300 x 1088 at 8 7.9 / 6.9, 300 x 1536
//     8.6 / 8.4; Q4_0 300 x 1088 7.2 / 6.9, 300 x 1984 7.4 / 7.0.
//   Narrower, from n * rows * cols of 40 Mi, off the line 20 Mi: 768 x 1024 at
//     32 (24 Mi) Q8_0 8.2 / 9.1, at 63 (47) 9.4 / 9.2; Q4_0 1000 x 1536 at 16
//     (23) 8.0 / 9.1, at 63 (92) 12.8 / 9.7; 2048 x 512 at 8 (8) 6.6 / 8.4;
//     1000 x 960 at 16 (15) 6.8 / 7.2, at 32 (29) 7.7 / 7.2.
//   From 5 vectors at 8 Mi weights: Q4_0 4096 x 2048 9.2 / 8.9, 4096 x 4096
//     13.4 / 10.0; 2048 x 2048 7.9 / 8.8.
// Shapes only the streamed kernel serves: up to 2048 columns (the vectors' rows
// staged whole) its time grows with the columns alone until the chip is
// full, the dot4 matvec's with n * rows too.
//   Under 256 columns from 8 vectors (512 x 160 Q4_0 7.0 / 5.6, Q8_0 5.8 / 5.5);
//   under 512 from n * rows of 32 Ki (Q4_0 4096 x 288 at 8 6.7 / 6.1, Q8_0 1500 x
//     288 at 16 5.8 / 6.6, 3000 x 416 at 16 7.3 / 7.3);
//   to 2048 from 40000 + 12 * cols (6000 x 864 at 8 (48000) Q4_0 8.7 / 8.2, Q8_0
//     8.4 / 8.4; 1500 x 2016 at 16 (24000) 9.1 / 14.4 and 10.3 / 14.3, 6000 x
//     2016 at 12 (72000) 15.1 / 14.5 and 16.2 / 14.6);
//   wider from 512 pairs (Q8_0 4096 x 11008 at 16 vectors, 256 pairs, 60.5 /
//     56.5, Q4_0 47.9 / 58.2; at 32, 512 pairs, 111 / 57 and 84 / 59).
static bool lanes32_on_cores(int t, int rows, int cols, int n) {
    const size_t size = (size_t)rows * cols;
    if (mmq32_supported(t, cols, false)) {
        if (n < 8)
            return n >= 5 && size >= ((size_t)8 << 20);
        const bool line = cols / 32 * (t == LH_Q8_0 ? 32 : 16) % 128 == 0;
        if (cols > 2048 || (cols > 1024 && (t == LH_Q8_0 || !line)))
            return true;
        return n * size >= ((size_t)(line ? 40 : 20) << 20);
    }
    if (!mmw_shape(t, rows, cols, false))
        return false;
    if (cols > MMW_XL_COLS)
        return n >= (size >= ((size_t)8 << 20) ? 5 : 8) && lane_pairs(rows, n) >= 512;
    if (cols < 256)
        return n >= 8;
    return n >= 5 && (long)n * rows >= (cols < 512 ? 32768 : 40000 + 12 * cols);
}

// The same for one K-quant matrix.  Q4_K from 5 vectors, Q6_K from 8 (us per
// launch, dot4 / matrix cores: Q4_K 4096 x 4096 at 5 vectors 11.4 / 9.1, 1024 x
// 2048 6.7 / 6.6; Q6_K at 5 10.8 / 10.4 and 6.6 / 7.1, at 8 12.5 / 10.6 and 7.8 /
// 7.2), but below 16 vectors (us per call)
//   Q6_K rows of one or two blocks (most of the one-shot kernel's waves idle) from
//     n * rows * cols of 14 Mi: 1004 x 512 at 11 6.5 / 6.9, 2500 x 512 at 12 7.3 /
//     6.9, 8192 x 512 at 8 7.8 / 7.3;
//   rows of 20 to 24 blocks, whose waves hold four blocks for three, from 2048
//     rows: Q6_K 900 x 4864 at 9 13.4 / 12.7, 300 x 5120 12.5 / 13.3, 1900 x 6144
//     14.5 / 15.1, 2500 x 6144 at 8 15.9 / 14.9; Q4_K only where the row's bytes are a
//     multiple of the 128-byte line and under 8 vectors: 1000 x 6144 at 5 11.1 / 12.6,
//     at 8 14.6 / 13.2, 1000 x 5632 at 5 11.1 / 11.0.  Wider shapes (only streamed)
//     from 512 pairs.
static bool lanes_k_on_cores(int t, int rows, int cols, int n) {
    const int nb = cols / 256;
    if (n < (t == LH_Q4_K ? 5 : 8))
        return false;
    if (n < 16 && t == LH_Q6_K && nb <= 2 && (size_t)n * rows * cols < ((size_t)14 << 20))
        return false;
    if (n < 16 && nb >= 20 && nb <= 24 && rows < 2048 && (t == LH_Q6_K || (n < 8 && nb * 144 % 128 == 0)))
        return false;
    return mmq_oneshot(t, cols, 16, false) || (mmw_shape(t, rows, cols, false) && lane_pairs(rows, n) >= 512);
}

// n vectors against one [rows][cols] matrix (or a fused pair): whether the
// matrix cores take them from the dot4 matvec.  One matrix: lanes32_on_cores,
// lanes_k_on_cores.  A fused pair: Q4_K from 16 (us per launch, dot4 / matrix
// cores: 2048 x 7168 at 8 vectors 16 / 24, at 24 47 / 25); Q8_0 / Q4_0, streamed
// only, from 512 pairs (us per call: 4096 x 4096 at 8 (256) 31.5 / 31.8 and 27.6 /
// 32.7; 4096 x 2048 at 16 (256) 29.2 / 23.9 and 24.7 / 23.7, at 24 (512) 37.1 / 23.8
// and 33.4 / 23.7; 2048 x 2048 at 32 (256) 27.5 / 22.8 and 24.6 / 23.7, at 64 (512)
// 44.2 / 23.0 and 42.2 / 23.9; 11008 x 4096 at 5 (688) 57.8 / 32.2 and 50.3 / 32.8).
bool mmq_dense(int t, int rows, int cols, int n, bool fused) {
    if (rows < 1 || n < 1)
        return false;
    if (t != LH_Q4_0 && t != LH_Q8_0 && !is_k(t))
        return false;
    if (!fused)
        return is_k(t) ? lanes_k_on_cores(t, rows, cols, n) : lanes32_on_cores(t, rows, cols, n);
    const size_t size = (size_t)rows * cols;
    if (n < (is_k(t) ? 16 : size >= ((size_t)8 << 20) ? 5 : size >= ((size_t)1 << 20) ? 8 : 64))
        return false;
    return mmq_oneshot(t, cols, 16, true) || (mmw_shape(t, rows, cols, true) && lane_pairs(rows, n) >= 512);
}

// The expert matmuls of n tokens, pairs of them with E experts: whether they run
// on the matrix cores in groups of 16.  By type and expert size, us per layer
// with the dot4 / matrix core matmuls, Zipf-skewed router (uniform):
//   K-quants from 5 tokens at 1.5 M weights, else 10: 2048 x 768 x 128 top-8 at
//     5 47.9 / 44.5 (53.8 / 54.5), 1536 x 768 x 64 top-6 at 10 50.3 / 43.3, 1024
//     x 512 x 32 top-4 at 10 33.8 / 31.2;
//   Q8_0 / Q4_0 from 5 at 8 M (4096 x 2048 x 16 top-4 108 / 72 and 87 / 68), 12
//     at 1.5 M (1536 x 1280 x 60 top-6 80 / 62 and 67 / 57, uniform 111 / 89 and
//     79 / 64; 2048 x 768 x 128 89 / 69 and 74 / 61; Q4_0 at 8 54.5 / 53.1,
//     uniform 62 / 69), else 20 (1024 x 768 x 64 top-6 55.3 / 48.9 and 54.3 / 46.6),
//     of under 750000 weights with 100 pairs or more than three pairs per
//     expert (there the dot4 form goes to groups of eight): 1024 x 512 x 32 top-4
//     at 20 37.3 / 41.5 and 38.0 / 40.4, at 24 40.5 / 41.5 and 41.2 / 40.7, at 26 (768 x
//     384) 38.1 / 37.5 and 39.4 / 36.9; x 64 top-8 at 20 52.5 / 49.5 and 53.1 / 47.1; x
//     16 top-4 at 20 44.3 / 41.0 and 42.7 / 39.7.
// Inputs of over 2048 columns (not staged whole) also need row tiles to stream:
// 4096 x 768 x 64 top-4 K-quants at 5 (960 (pair, tile) streams) 44.4 / 49.3, at 7
// (1344) 49.1 / 49.9, with a Q4_K down 48.6 / 45.5; 4096 x 1024 x 32 top-4 at 5 (1280) 45.7 / 49.6, at 7 (1792)
// 55.3 / 53.7; 4096 x 1280 x 32 at 5 (1600) 58.2 / 54.0.
constexpr long EXPERT_MIN_STREAMS = 1300;
static bool experts_take(int t, size_t size, int n, int pairs, int E) {
    if (is_k(t))
        return n >= (size >= 1500000 ? 5 : 10);
    if (size >= 1500000)
        return n >= (size >= 8000000 ? 5 : 12);
    return n >= 20 && (size >= 750000 || pairs >= 100 || pairs > 3 * E);
}
bool mmq_experts(int gate_t, int down_t, int dim, int ffn, int n, int k, int E) {
    const size_t size = (size_t)dim * ffn;
    if (!mmw_shape(gate_t, ffn, dim, true) || !mmw_shape(down_t, dim, ffn, false) ||
        (dim > MMW_XL_COLS && (long)n * k * ((ffn + 15) / 16) < EXPERT_MIN_STREAMS))
        return false;
    return experts_take(gate_t, size, n, n * k, E) && experts_take(down_t, size, n, n * k, E);
}

template <int T, int MT, bool FUSED>
static void mmq_launch_t(const DmmvParams &p, int rg, int ks, int sbw, hipStream_t st) {
    const size_t lds = mmq_lds_bytes(p.cols, MT, rg, FUSED);
    const int groups = p.ident_n > 0 ? (p.ident_n + 16 * MT - 1) / (16 * MT) : p.n_groups;
    const int tiles = (p.rows + 16 * rg - 1) / (16 * rg);
    const dim3 grid(tiles, groups), block(64 * rg * ks);
    if (sbw == 1)
        hipLaunchKernelGGL((mmq_kernel<T, MT, FUSED, 1>), grid, block, lds, st, p, rg, ks);
    else if (sbw == 2)
        hipLaunchKernelGGL((mmq_kernel<T, MT, FUSED, 2>), grid, block, lds, st, p, rg, ks);
    else if constexpr (MT == 1)
        hipLaunchKernelGGL((mmq_kernel<T, MT, FUSED, 4>), grid, block, lds, st, p, rg, ks);
}

// Segments of Q4_K / Q6_K matrices over the same columns, lanes in groups of
// 16 (identity pairs, sp.base.ident_n set: twice the work groups of 32-lane
// groups measured faster for these small matrices at 32 lanes); declined
// (false) when a segment's type or the shape is not served.
bool launch_mmq_seg(DmmvSegParams sp, hipStream_t st) {
    const DmmvParams &p = sp.base;
    if (p.ident_n < 1 || sp.n_seg < 1 || sp.n_seg > DMMV_MAX_SEG)
        return false;
    constexpr int mt = 1;
    int rg = MMQ_WAVES, ks = 0, sbw = 0, tiles = 0;
    for (int i = 0; i < sp.n_seg; i++) {
        if (!is_k(sp.seg[i].t) || !mmq_oneshot(sp.seg[i].t, p.cols, 16 * mt, false))
            return false;
        int r, k, b;
        if (!mmq_shape(sp.seg[i].rows, p.cols, mt, false, r, k, b))
            return false;
        if (r < rg)
            rg = r;
        ks = k;
        sbw = b;
    }
    if (sbw > 2)
        return false;
    for (int i = 0; i < sp.n_seg; i++) {
        sp.seg[i].tiles = (sp.seg[i].rows + 16 * rg - 1) / (16 * rg);
        tiles += sp.seg[i].tiles;
    }
    const size_t lds = mmq_lds_bytes(p.cols, mt, rg, false);
    const dim3 grid(tiles, (p.ident_n + 16 * mt - 1) / (16 * mt)), block(64 * rg * ks);
    auto kern = sbw == 1 ? mmq_seg_kernel<mt, 1> : mmq_seg_kernel<mt, 2>;
    hipLaunchKernelGGL(kern, grid, block, lds, st, sp, rg, ks);
    note_launch();
    return true;
}

// Groups of at most max_tok (<= 32) tokens (with p.ident_n: max_tok sets
// the group size); p.rpw is unused.
bool launch_mmq(int t, int max_tok, bool fused, const DmmvParams &p, hipStream_t st) {
    if (p.rows < 1 || max_tok < 1 || max_tok > 32)
        return false;
    if (p.ident_n > 0 && max_tok > 16 && !mmq_oneshot(t, p.cols, max_tok, fused))
        max_tok = 16; // the one-shot kernel's registers hold 16 tokens of the widest rows
    const bool oneshot = mmq_oneshot(t, p.cols, max_tok, fused);
    const bool stream = p.ident_n > 0 ? lanes_streamed(t, p.rows, p.cols, p.ident_n, fused) ||
                                            (!oneshot && mmw_shape(t, p.rows, p.cols, fused))
                                      : max_tok <= 16 && mmw_shape(t, p.rows, p.cols, fused) &&
                                            !(oneshot && groups_few(t, p.rows, p.n_groups, fused));
    if (!stream && !oneshot)
        return false;
    const int mt = max_tok > 16 ? 2 : 1;
    if (!is_k(t)) {
        if (!stream && p.ident_n <= 0) // mmq32_kernel takes lane groups only
            return false;
        if (!stream)
            launch_mmq32(t, p, st);
        else if (t == LH_Q8_0)
            fused ? mmw32_launch_t<LH_Q8_0, true>(p, st) : mmw32_launch_t<LH_Q8_0, false>(p, st);
        else
            fused ? mmw32_launch_t<LH_Q4_0, true>(p, st) : mmw32_launch_t<LH_Q4_0, false>(p, st);
        note_launch();
        return true;
    }
    if (p.ident_n > 0 && !fused && lanes_tiled(t, p.rows, p.cols, p.ident_n)) {
        t == LH_Q4_K ? mmp_launch_t<LH_Q4_K>(p, st) : mmp_launch_t<LH_Q6_K>(p, st);
        note_launch();
        return true;
    }
    if (stream) {
        if (t == LH_Q4_K)
            fused ? mmw_launch_t<LH_Q4_K, 1, true>(p, st) : mmw_launch_t<LH_Q4_K, 1, false>(p, st);
        else if (mt == 1)
            mmw_launch_t<LH_Q6_K, 1, false>(p, st);
        else
            mmw_launch_t<LH_Q6_K, 2, false>(p, st);
        note_launch();
        return true;
    }
    int rg, ks, sbw;
    if (!mmq_shape(p.rows, p.cols, mt, fused, rg, ks, sbw))
        return false;
    if (t == LH_Q4_K) {
        if (mt == 1)
            fused ? mmq_launch_t<LH_Q4_K, 1, true>(p, rg, ks, sbw, st)
                  : mmq_launch_t<LH_Q4_K, 1, false>(p, rg, ks, sbw, st);
        else
            fused ? mmq_launch_t<LH_Q4_K, 2, true>(p, rg, ks, sbw, st)
                  : mmq_launch_t<LH_Q4_K, 2, false>(p, rg, ks, sbw, st);
    } else if (mt == 1) {
        mmq_launch_t<LH_Q6_K, 1, false>(p, rg, ks, sbw, st);
    } else {
        mmq_launch_t<LH_Q6_K, 2, false>(p, rg, ks, sbw, st);
    }
    note_launch();
    return true;
}

} // namespace lh
