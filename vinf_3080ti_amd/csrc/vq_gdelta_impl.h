// vq_gdelta_impl.h -- the gated delta rule of a prompt pass in chunks of 32 tokens on fp32 MFMA (included by vq_ops.hip).
//
// The rule per token t (k, q normalised, g the decay, b = beta):
//   S <- g_t S;  d_t = b_t (v_t - S^T k_t);  S <- S + k_t d_t^T;  o_t = S^T q_t.
// Over a chunk that starts from state S0, with D(t, i) = g_{i+1} ... g_t (running products) and G_t = D(t, -1):
//   d_t = b_t (v_t - G_t S0^T k_t) - sum_{i<t} L(t, i) d_i,   L(t, i) = b_t D(t, i) (k_i . k_t)
//   o_t = G_t S0^T q_t + sum_{i<=t} P(t, i) d_i,              P(t, i) = D(t, i) (k_i . q_t)
//   S_C = G_C S0 + sum_i D(C - 1, i) k_i d_i^T
// so with T = (I + L)^-1 everything that meets the state is a matrix product:
//   d = T b (V - G K S0),   o = G (Q S0) + P d,   S_C = G_C S0 + (D(C - 1, .) K)^T d.
// The 1 / |k| of the last two's k and the b go into T, so that the walk's products are of the rows as given.
// What meets the state is fp32 (v_mfma_f32_16x16x4_f32, fp32 operands and sums), with care for the roundings in a row: long
// sums in eight chains, the sums over a chunk's tokens from zero. What does not (the pairs' products, decays and factors,
// T) is fp64 on v_mfma_f64_16x16x4_f64 and rounded once into an operand. Rel-L2 error against float64 as a multiple of the
// per-token kernel's, 24 to 512 tokens, independent keys: outputs 0.83-0.90 (1.1-1.6e-7), state 0.8-1.13 (1.0-2.2e-7); with
// the pairs' products in fp32 the outputs stood at 0.9-1.12, and at 1.3-1.4 (now 1.0-1.1) for keys that share a
// direction. Equal keys, beta near one: 1.3-1.6; there each update of the per-token rule corrects the one before it.
//
// Two launches. gd_prep_kernel, one workgroup per (chunk, value head), all chunks at once: T and P into the workspace in
// MFMA operand order, and the tokens' scales. It leaves V alone (the walk reads and checks it), which pays for the fp64
// products: 15.9 us, as with fp32 ones. gd_chunk_kernel, one workgroup per (value head, 32 state columns), walks
// the chunks with its part of the state in accumulators, the chunk's K, Q, V rows and T, P reaching LDS by DMA a chunk
// ahead: 116 MFMAs per wave and two barriers per 32 tokens, instead of 32 serial tokens of two barriers each. What bounds
// it: the serial chunk walk's MFMA issue (33 cycles each, 1.6 us of a chunk's 3.7, on 192 of 256 CUs). Operands prepared
// in full (W = T diag(b G) K, scaled Q and K in operand order, read straight into registers) moved 55 KB per chunk and
// workgroup through L2 twice and took 28 + 56 us. Measured at 16 key and 48 value heads, kd = vd = 128, 512 tokens:
// 15.9 + 59.5 us against 358 us token by token. With four chains (54.5 us), of a chunk's 6800 cycles the K S0 and Q S0
// products took 3500 (their 64 MFMAs 2100; the rest are the copies and LDS reads of the one wave per SIMD), T R 690, the
// state update 1720; eight waves of 32 rows measured 62 us (more operand reads and a four-way exchange), one copy per four
// MFMAs 57 us.
//
// MFMA layouts used below (lane = 16 lk + lr): C/D element q is row 4 lk + q, column lr; the k index of an operand
// element is free as long as A and B agree, so step q of a 16-deep block takes k = 4 lk + q: an accumulator tile is then
// a B operand as it stands, and an A operand is one float4 of a row.
//
// A value that is not finite, given or arising on the way, would meet zeros of T and P in these products and reach tokens
// before its own. Chunks that could hold one are taken token by token: the prep kernel flags those whose sums of squares
// lie past kGcSquare or whose scales past kGcScale, the walk those whose V or S0 lies past kGcHuge; below these bounds no
// product or sum of a chunk leaves the fp32 range. So are chunks whose decays above one multiply to kGcGrow or more: the
// entries of T reach that product (one otherwise), and with it the rounding of d. Equal keys, beta 0.9975, against
// float64: decays of 1.1 1.3e-6 (token by token 1.2e-7), of 1.3 1.4e-4.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace {

constexpr int kGcC = 32, kGcKd = 128, kGcMaxVd = 128, kGcCols = 32;
// Segments of at least this many rows take the chunks. Measured at 48 value heads of 128, us token by token / in chunks:
// one sequence of 16 rows 15.3 / 15.8, 24 rows 22.3 / 17.7, 512 rows 360 / 75; four of 24 rows 33.5 / 29.5; 16 of 24 rows
// 93 / 89, 64 rows 223 / 142, 512 rows 1656 / 895; 64 of 24 rows 335 / 369 (the one loss: 32 rows 418 / 376, 512 rows
// 6113 / 3570). The rule looks at a segment's own rows alone, so that its bits do not depend on the others of a pass.
constexpr int kGcMinRows = 24;
// Chunks of a segment per launch pair, and the bytes of a launch pair's chunk operands, which the segments of a group
// share. With one launch pair for all long segments at 16 / n chunks each, every 32 tokens of nine and more took a pair of
// launches and the state's way through memory: 64 segments of 512 rows 5919 us and 230 MB of workspace, now 3570 and 28;
// 16 of 64 rows 178 -> 142; 64 of 512 rows, four heads of 64, 426 (403 token by token) -> 243.
constexpr int kGcRound = 16;
constexpr size_t kGcGroupBytes = size_t{32} << 20;
static_assert(kGcRound <= 64, "one lane per chunk reads the non-finite flags");

constexpr float kGcHuge = 1e28f, kGcSquare = 1e18f, kGcScale = 1e6f, kGcGrow = 1.0625f;

typedef float gc_f4 __attribute__((ext_vector_type(4)));
typedef double gc_d4 __attribute__((ext_vector_type(4)));

// Workspace of one (chunk, value head), in floats: T and P as A operands [t tile 2][i tile 2][lane][4], then the tokens'
// scales (32 each: G / |k|, D(C - 1, .), G / (|q| sqrt(kd))), G_C and the flag of a chunk to take token by token.
struct GcSlot {
    static constexpr int T = 0, P = 1024, SC = 2048, KG = 0, DC = 32, QG = 64, GC = 96, BAD = 97;
    static constexpr size_t floats = 2304;
};

// The long segments of a pass, and the chunks [c0, c0 + cr) of each that this launch covers; slot ((seg * cr + c - c0)
// * value_heads + head).
struct GcArgs {
    const float *conv, *braw, *araw, *ssm_a, *dt;
    float *ws;
    int key_heads, value_heads, vd, head_order, c0, cr;
    float eps;
};

__device__ __forceinline__ bool gc_bad(float v) { return (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u; }
__device__ __forceinline__ gc_f4 gc_mfma(float a, float b, gc_f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ gc_d4 gc_mfma64(double a, double b, gc_d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ gc_f4 gc_ld(const float *p) { return *reinterpret_cast<const gc_f4 *>(p); }

__global__ __launch_bounds__(256) void gd_prep_kernel(GcArgs A, SegTable T) {
    constexpr int RS = kGcKd + 4;  // LDS row pitch (floats)
    // K and Q until their products are made, then L and T in their place.
    __shared__ __align__(16) float sKQ[2][kGcC][RS];
    static_assert(2 * kGcC * 34 * sizeof(double) <= sizeof(sKQ));
    auto &sK = sKQ[0], &sQ = sKQ[1];
    double(&sL)[kGcC][34] = reinterpret_cast<double(&)[kGcC][34]>(sKQ[0]);
    double(&sT)[kGcC][34] = *(&sL + 1);
    __shared__ double sD[kGcC][kGcC + 1];  // [t][i + 1]: D(t, i); [t][0]: G_t
    __shared__ double sH[3][4][64];  // the second halves of the three tiles of P^T
    __shared__ float sB[kGcC], sG[kGcC], sQs[kGcC], sKs[kGcC];
    __shared__ int s_bad;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, lr = lane & 15, lk = lane >> 4;
    const int h = blockIdx.x, c = A.c0 + blockIdx.y;
    const Seg &s = T.s[blockIdx.z];
    const int t0 = c * kGcC, nt = min(kGcC, s.rows - t0);
    if (nt <= 0) return;
    const int vh = A.value_heads, vd = A.vd;
    const int kh = A.head_order == 0 ? h / (vh / A.key_heads) : h % A.key_heads;
    const size_t cdim = static_cast<size_t>(2) * A.key_heads * kGcKd + static_cast<size_t>(vh) * vd;
    const size_t row0 = static_cast<size_t>(s.row0) + t0;
    float *const ws = A.ws + ((static_cast<size_t>(blockIdx.z) * A.cr + blockIdx.y) * vh + h) * GcSlot::floats;

    // 1. The chunk's q, k rows (zeros past the segment).
    if (tid == 0) s_bad = 0;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = (tid >> 5) + 8 * i, e = 4 * (tid & 31);
        gc_f4 q = {0.f, 0.f, 0.f, 0.f}, k = q;
        if (r < nt) {
            const float *src = A.conv + (row0 + r) * cdim;
            q = gc_ld(src + static_cast<size_t>(kh) * kGcKd + e);
            k = gc_ld(src + static_cast<size_t>(A.key_heads + kh) * kGcKd + e);
        }
        *reinterpret_cast<gc_f4 *>(&sQ[r][e]) = q;
        *reinterpret_cast<gc_f4 *>(&sK[r][e]) = k;
    }
    __syncthreads();
    // 2. Per token (eight threads each): the norm scales; beta and the decay.
    {
        const int t = tid >> 3, j = tid & 7;
        const bool in = t < nt;
        const size_t rr = (row0 + (in ? t : 0)) * vh + h;
        const float xa = A.araw[rr] + A.dt[h], xb = A.braw[rr], sa = A.ssm_a[h];
        float qq = 0.0f, kk = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const gc_f4 q = gc_ld(&sQ[t][4 * (j + 8 * i)]), k = gc_ld(&sK[t][4 * (j + 8 * i)]);
#pragma unroll
            for (int e = 0; e < 4; ++e) qq = fmaf(q[e], q[e], qq), kk = fmaf(k[e], k[e], kk);
        }
        qq = gsum8(qq);
        kk = gsum8(kk);
        if (j == 0) {
            const float rkd = 1.0f / sqrtf(static_cast<float>(kGcKd));
            const float qs = in ? rkd / sqrtf(qq + A.eps) : 0.0f, ks = in ? 1.0f / sqrtf(kk + A.eps) : 0.0f;
            const float g = in ? expf(sa * (xa > 20.0f ? xa : log1pf(expf(xa)))) : 1.0f;
            const float b = in ? sigmoid_ieee(xb) : 0.0f;
            // The sums themselves: one that overflowed leaves a finite scale (zero).
            bad |= !(qq < kGcSquare) || !(kk < kGcSquare) || !(qs < kGcScale) || !(ks < kGcScale) || gc_bad(g) || gc_bad(b);
            sQs[t] = qs, sKs[t] = ks, sG[t] = g, sB[t] = b;
        }
    }
    if (bad) s_bad = 1;
    __syncthreads();
    // 3. Wave 1, which has no tile below, walks the decays of the pairs down their columns: lane 0 those since the chunk's
    // start (G_t), lane i + 1 the D(t, i). The running products and the pairs' factors are fp64, rounded once where they
    // become operands.
    // 4. Wave (jt, ji): the 16 x 16 tiles L (rows t, columns i) and P^T (rows i, columns t); nothing above the diagonal.
    // D element q of the fp64 MFMA: row 4 q + lk, column lr.
    const int jt = wv >> 1, ji = wv & 1;
    gc_d4 kk = {0.0, 0.0, 0.0, 0.0}, kq = kk;
    if (wv == 1) {
        if (lane <= kGcC) {
            double d = 1.0;
            float grow = 1.0f;
#pragma unroll
            for (int t = 0; t < kGcC; ++t) {
                d = t < lane ? 1.0 : d * sG[t];
                sD[t][lane] = t + 1 < lane ? 0.0 : d;
                grow *= fmaxf(sG[t], 1.0f);
            }
            // Decays above one: T's entries grow with their products while the d_t that the sums leave stay as they were.
            if (!(grow < kGcGrow)) s_bad = 1;
        }
        gc_d4 h[3] = {kk, kk, kk};
#pragma unroll
        for (int cc = kGcKd / 32; cc < kGcKd / 16; ++cc) {
            const gc_f4 k0 = gc_ld(&sK[lr][16 * cc + 4 * lk]), k1 = gc_ld(&sK[16 + lr][16 * cc + 4 * lk]),
                        q0 = gc_ld(&sQ[lr][16 * cc + 4 * lk]), q1 = gc_ld(&sQ[16 + lr][16 * cc + 4 * lk]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                h[0] = gc_mfma64(k0[q], q0[q], h[0]);
                h[1] = gc_mfma64(k0[q], q1[q], h[1]);
                h[2] = gc_mfma64(k1[q], q1[q], h[2]);
            }
        }
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) sH[t][q][lane] = h[t][q];
    } else {
#pragma unroll
        for (int cc = 0; cc < kGcKd / 16; ++cc) {
            const gc_f4 kt = gc_ld(&sK[16 * jt + lr][16 * cc + 4 * lk]), ki = gc_ld(&sK[16 * ji + lr][16 * cc + 4 * lk]),
                        qt = gc_ld(&sQ[16 * jt + lr][16 * cc + 4 * lk]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                kk = gc_mfma64(kt[q], ki[q], kk);
                if (cc < kGcKd / 32) kq = gc_mfma64(ki[q], qt[q], kq);
            }
        }
    }
    __syncthreads();
    if (wv != 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) kq[q] += sH[jt + ji][q][lane];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = 4 * q + lk, t = 16 * jt + e, i = 16 * ji + lr;
        const double ks = sKs[t];
        sL[t][i] = i < t ? sB[t] * sD[t][i + 1] * (ks * sKs[i]) * kk[q] : 0.0;
        const int pt = 16 * jt + lr, pi = 16 * ji + e;
        ws[GcSlot::P + ((jt * 2 + ji) * 64 + 16 * q + lr) * 4 + lk] =
            pi <= pt ? static_cast<float>(sD[pt][pi + 1] * sQs[pt] * kq[q]) : 0.0f;
    }
    if (tid < kGcC) {
        float *const sc = ws + GcSlot::SC;
        const float gc = static_cast<float>(sD[kGcC - 1][0]);
        sc[GcSlot::KG + tid] = static_cast<float>(sD[tid][0] * sKs[tid]);
        sc[GcSlot::DC + tid] = static_cast<float>(sD[kGcC - 1][tid + 1]);
        sc[GcSlot::QG + tid] = static_cast<float>(sD[tid][0] * sQs[tid]);
        if (tid == 0) sc[GcSlot::GC] = gc, sc[GcSlot::BAD] = s_bad || gc_bad(gc) ? 1.0f : 0.0f;
    }
    __syncthreads();
    // 5. (I + L)^-1: the two diagonal blocks by forward substitution (lane = column), then T21 = -T22 (L21 T11).
    if (wv < 2 && lane < 16) {
        const int o = 16 * wv;
        double x[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            double v = t == lane ? 1.0 : 0.0;
#pragma unroll
            for (int i = 0; i < t; ++i) v = fma(-sL[o + t][o + i], x[i], v);
            x[t] = v;
            sT[o + t][o + lane] = v;
        }
    }
    __syncthreads();
    if (wv == 0) {
        gc_d4 m = {0.0, 0.0, 0.0, 0.0}, x = m;
#pragma unroll
        for (int q = 0; q < 4; ++q) m = gc_mfma64(sL[16 + lr][4 * q + lk], sT[4 * q + lk][lr], m);
#pragma unroll
        for (int q = 0; q < 4; ++q) x = gc_mfma64(sT[16 + lr][16 + 4 * q + lk], m[q], x);
#pragma unroll
        for (int q = 0; q < 4; ++q) sT[16 + 4 * q + lk][lr] = -x[q];
    }
    __syncthreads();
    if (ji <= jt) {
        const int t = 16 * jt + lr;
        gc_f4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = 16 * ji + 4 * lk + q;
            v[q] = static_cast<float>(sKs[t] * sT[t][i] * sB[i]);
        }
        *reinterpret_cast<gc_f4 *>(ws + GcSlot::T + ((jt * 2 + ji) * 64 + lane) * 4) = v;
    }
}

// The chunk walk. Wave w of a workgroup: column tile n = w & 1 (16 of the 32 columns), state rows 64 kh .. +64 with
// kh = w >> 1. The two waves of a column tile exchange their halves of W S and of the other's 16 output rows through LDS.
// state_in / state_out: the slot's state, or the fp32 copy between two launches of one pass (tmp, [seg][head][kd][vd]).
template <typename ST>
__global__ __launch_bounds__(256, 1) void gd_chunk_kernel(GcArgs A, SegTable T, ST *__restrict__ state,
                                                          float *__restrict__ tmp, float *__restrict__ out,
                                                          int write_state) {
    // One chunk's operands. A K or Q row's 16-byte pieces sit at piece ^ (row & 15): the 16 rows of an A operand and
    // the rows 4 lk + q of a transposed one then fall on distinct banks. V rows: piece ^ 4 on every other four rows.
    struct Buf {
        float k[kGcC * kGcKd], q[kGcC * kGcKd], v[kGcC * kGcCols], t[1024], p[1024], sc[256];
    };
    __shared__ __align__(1024) Buf buf[2];
    __shared__ __align__(16) gc_f4 ex[4][3][64];  // [wave][tile][lane]
    __shared__ float red[2][4][3][16];            // token-by-token chunks: [wave][sum][column]
    __shared__ __align__(16) int huge[4];         // [wave]: its part of the present chunk's V and S0 is out of range
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), n = wv & 1, kh = wv >> 1;
    const int vh = A.value_heads, vd = A.vd, tiles = vd / kGcCols;
    // Workgroup ids go round-robin over the 8 XCDs: the column tiles of one head, which read the same operands, are 8
    // ids apart and share an XCD's L2.
    const int b = blockIdx.x, g8 = (b / (8 * tiles)) * 8, r8 = b - g8 * tiles, wide = min(8, vh - g8);
    const int h = g8 + r8 % wide, c0 = (r8 / wide) * kGcCols;
    const Seg &s = T.s[blockIdx.y];
    const int nch = (s.rows + kGcC - 1) / kGcC, ca = A.c0, cb = min(nch, A.c0 + A.cr);
    if (ca >= cb) return;
    const int col = c0 + 16 * n + lr;
    const size_t hstate = static_cast<size_t>(kGcKd) * vd;
    ST *const S = state + (static_cast<size_t>(s.slot) * vh + h) * hstate;
    float *const Sx = tmp + (static_cast<size_t>(blockIdx.y) * vh + h) * hstate;
    const float *const slot0 = A.ws + (static_cast<size_t>(blockIdx.y) * A.cr * vh + h) * GcSlot::floats;
    const size_t cstep = static_cast<size_t>(vh) * GcSlot::floats;

    gc_f4 st[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t e = static_cast<size_t>(64 * kh + 16 * i + 4 * lk + q) * vd + col;
            st[i][q] = ca == 0 ? ld_state(S + e) : Sx[e];
        }
    const int kx = A.head_order == 0 ? h / (vh / A.key_heads) : h % A.key_heads;
    const size_t cdim = static_cast<size_t>(2) * A.key_heads * kGcKd + static_cast<size_t>(vh) * vd;
    // DMA of chunk c into buffer c & 1, 11 or 12 KB per wave, in three parts between the products of chunk c - 1 (ahead of
    // them all the wave stalls 850 cycles while the copies are taken up); the lane offsets are those of a full chunk (rows
    // past the segment repeat its last one, their scales are zero).
    uint32_t off_k[4], off_v;
    auto offsets = [&](int last) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 2 * (wv + 4 * j) + (lane >> 5);
            off_k[j] = (static_cast<uint32_t>(min(r, last)) * static_cast<uint32_t>(cdim) + 4u * ((lane & 31) ^ (r & 15))) * 4u;
        }
        const int r = 8 * wv + (lane >> 3);
        off_v = (static_cast<uint32_t>(min(r, last)) * static_cast<uint32_t>(cdim) + 4u * ((lane & 7) ^ (r & 4))) * 4u;
    };
    const float *const conv0 = A.conv + static_cast<size_t>(s.row0) * cdim;
    const uint32_t lds0 = vq::lds_addr(buf);
    auto issue = [&](int c, int part) {
        const float *const base = conv0 + static_cast<size_t>(c * kGcC) * cdim;
        const float *const sl = slot0 + static_cast<size_t>(c - ca) * cstep;
        const uint32_t d = lds0 + (c & 1) * static_cast<uint32_t>(sizeof(Buf)) + 1024u * wv;
        if (part == 0) {
            if (s.rows - c * kGcC < kGcC) offsets(s.rows - c * kGcC - 1);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                vq::dma16u(base + static_cast<size_t>(A.key_heads + kx) * kGcKd, off_k[j], d + offsetof(Buf, k) + 4096 * j, buf);
        } else if (part == 1) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                vq::dma16u(base + static_cast<size_t>(kx) * kGcKd, off_k[j], d + offsetof(Buf, q) + 4096 * j, buf);
        } else {
            vq::dma16u(base + static_cast<size_t>(2) * A.key_heads * kGcKd + static_cast<size_t>(h) * vd + c0, off_v,
                       d + offsetof(Buf, v), buf);
            vq::dma16u(sl + GcSlot::T + 256 * wv, 16u * lane, d + offsetof(Buf, t), buf);
            vq::dma16u(sl + GcSlot::P + 256 * wv, 16u * lane, d + offsetof(Buf, p), buf);
            if (wv == 0) vq::dma16u(sl + GcSlot::SC, 16u * lane, d + offsetof(Buf, sc), buf);
        }
    };
    float *const orow = out + (static_cast<size_t>(s.row0) * vh + h) * vd + col;
    const size_t ostep = static_cast<size_t>(vh) * vd;

    auto state_mag = [&] {  // of the lane's state elements; taken where they are made, off the walk's chain
        gc_f4 m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) m[i] += fabsf(st[i][q]);
        return (m[0] + m[1]) + (m[2] + m[3]);
    };
    float st_mag;

    // One chunk from its operands (landed; all waves past the barrier that says so). False (for all waves alike), with
    // the state as it was, when V or S0 is out of range.
    auto chunk = [&](int c) {
        const Buf &f = buf[c & 1];
        auto a_row = [&](const float *m, int t, int i) {  // A operand: rows 16 t + lr, columns 64 kh + 16 i + 4 lk ..
            return gc_ld(m + (16 * t + lr) * kGcKd + 4 * ((16 * kh + 4 * i + lk) ^ lr));
        };
        // One wave per SIMD: nothing else hides an LDS read, so each part's operands are read a part ahead, and the
        // scheduler is kept from sinking the reads back to their uses (without the fences: 57.6 us for 16 chunks).
#define VQ_GC_FENCE() __builtin_amdgcn_sched_barrier(0)
        gc_f4 ka[2][4], qa[2][4], x[2], o[2];
        float kt[2][4][4];
        auto read_kt = [&](int t) {  // K^T operand: column 64 kh + 16 i + lr of rows 16 t + 4 lk + q
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float *const kr = f.k + (16 * t + 4 * lk + q) * kGcKd + (lr & 3);
#pragma unroll
                for (int i = 0; i < 4; ++i) kt[t][q][i] = kr[4 * ((16 * kh + 4 * i + (lr >> 2)) ^ (4 * lk + q))];
            }
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) ka[0][i] = a_row(f.k, 0, i), ka[1][i] = a_row(f.k, 1, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) qa[0][i] = a_row(f.q, 0, i), qa[1][i] = a_row(f.q, 1, i);
        VQ_GC_FENCE();
        // Eight sums of eight terms per tile, added pairwise: twelve roundings in a row, not 64. The first half's are added
        // while the second half's products run.
        gc_f4 xc[2][2][4], oc[2][2][4], xs[2][2], os[2][2];
        auto part_sum = [&](int i) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const gc_f4 *const a = xc[i][t], *const b = oc[i][t];
                xs[t][i] = (a[0] + a[1]) + (a[2] + a[3]);
                os[t][i] = (b[0] + b[1]) + (b[2] + b[3]);
            }
        };
        gc_f4 kg[2], dc[2], vv[2], tt[3], pp[2], qg;
        float gc;
        // K S0 and Q S0: chains of MFMAs (a dependent one waits 8-12 cycles past its 32), in four parts that also
        // read what the second half of the chunk needs and start the next chunk's DMA.
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i < 2) {
                read_kt(i);
            } else {
                const int t = i - 2;
                kg[t] = gc_ld(f.sc + GcSlot::KG + 16 * t + 4 * lk);
                dc[t] = gc_ld(f.sc + GcSlot::DC + 16 * t + 4 * lk);
                pp[t] = gc_ld(f.p + 4 * ((2 * kh + t) * 64 + lane));
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    vv[t][q] = f.v[(16 * t + 4 * lk + q) * kGcCols + ((16 * n + lr) ^ ((lk & 1) << 4))];
                if (t == 0) {
                    tt[0] = gc_ld(f.t + 4 * lane), tt[1] = gc_ld(f.t + 4 * (128 + lane));
                    tt[2] = gc_ld(f.t + 4 * (192 + lane));
                } else {
                    qg = gc_ld(f.sc + GcSlot::QG + 16 * kh + 4 * lk);
                    gc = f.sc[GcSlot::GC];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const gc_f4 z = {0.f, 0.f, 0.f, 0.f};
                    xc[i >> 1][t][q] = gc_mfma(ka[t][i][q], st[i][q], i & 1 ? xc[i >> 1][t][q] : z);
                    oc[i >> 1][t][q] = gc_mfma(qa[t][i][q], st[i][q], i & 1 ? oc[i >> 1][t][q] : z);
                }
            }
            if (i == 2) part_sum(0);
            if (i < 3 && c + 1 < cb) issue(c + 1, i);
            VQ_GC_FENCE();
        }
        part_sum(1);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            x[t] = xs[t][0] + xs[t][1];
            o[t] = os[t][0] + os[t][1];
        }
        ex[wv][0][lane] = x[0];
        ex[wv][1][lane] = x[1];
        ex[wv][2][lane] = kh == 0 ? o[1] : o[0];  // the partner's output rows
        float mag = st_mag;
#pragma unroll
        for (int q = 0; q < 4; ++q) mag += fabsf(vv[0][q]) + fabsf(vv[1][q]);
        const int far = __any(!(mag < kGcHuge));
        if (lane == 0) huge[wv] = far;
        __syncthreads();
        const int pw = wv ^ 2;
        const gc_f4 xp[2] = {ex[pw][0][lane], ex[pw][1][lane]}, op = ex[pw][2][lane];
        const int4 any = *reinterpret_cast<const int4 *>(huge);
        // R = V - G K S0, then d / |k| = T R
        gc_f4 r[2], d[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, d1 = d[0];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) r[t][q] = fmaf(-kg[t][q], x[t][q] + xp[t][q], vv[t][q]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            d[0] = gc_mfma(tt[0][q], r[0][q], d[0]);
            d[1] = gc_mfma(tt[1][q], r[0][q], d[1]);
            d1 = gc_mfma(tt[2][q], r[1][q], d1);
        }
        d[1] += d1;
        // S = G_C S + K^T (D(C - 1, .) d),  o = G (Q S0) + P d (the tile of P above the diagonal is zero)
        // The sums over the chunk's tokens start from zero and meet the larger terms once, in one fma.
        gc_f4 y = {0.f, 0.f, 0.f, 0.f}, up[4] = {y, y, y, y}, next[4];
        const gc_f4 qs0 = (kh == 0 ? o[0] : o[1]) + op;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const gc_f4 kd = d[t] * dc[t];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int i = 0; i < 4; ++i) up[i] = gc_mfma(kt[t][q][i], kd[q], up[i]);
                y = gc_mfma(pp[t][q], d[t][q], y);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            y[q] = fmaf(qs0[q], qg[q], y[q]);
#pragma unroll
            for (int i = 0; i < 4; ++i) next[i][q] = fmaf(st[i][q], gc, up[i][q]);
        }
#undef VQ_GC_FENCE
        vq::wait_vm<0>();  // the next chunk's operands (not the stores that follow)
        // Only now: a branch among the products cost 2.1 us of the walk's 60.
        if (__builtin_amdgcn_readfirstlane(any.x | any.y | any.z | any.w)) return false;
#pragma unroll
        for (int i = 0; i < 4; ++i) st[i] = next[i];
        st_mag = state_mag();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int t = c * kGcC + 16 * kh + 4 * lk + q;
            if (t < s.rows) orow[t * ostep] = y[q];
        }
        return true;
    };
    // One chunk token by token (a value is out of range): the rule as the per-token kernel computes it.
    auto serial = [&](int c) {
        const float rkd = 1.0f / sqrtf(static_cast<float>(kGcKd));
        // Column sums over all rows: the lane groups, then the two waves of the column tile.
        auto total = [&](float v, int k, int par) {
            v = xor32_add(xor16_add(v));
            if (lk == 0) red[par][wv][k][lr] = v;
        };
        for (int t = c * kGcC; t < min((c + 1) * kGcC, s.rows); ++t) {
            const size_t rr = static_cast<size_t>(s.row0) + t;
            const float *qs = A.conv + rr * cdim + static_cast<size_t>(kx) * kGcKd + 64 * kh + 4 * lk;
            gc_f4 qv[4], kv[4];
            float qq = 0.0f, kk = 0.0f, mem = 0.0f, o = 0.0f;
            const float xa = A.araw[rr * vh + h] + A.dt[h];
            const float decay = expf(A.ssm_a[h] * (xa > 20.0f ? xa : log1pf(expf(xa))));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                qv[i] = gc_ld(qs + 16 * i);
                kv[i] = gc_ld(qs + static_cast<size_t>(A.key_heads) * kGcKd + 16 * i);
                st[i] *= decay;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    qq = fmaf(qv[i][q], qv[i][q], qq);
                    kk = fmaf(kv[i][q], kv[i][q], kk);
                    mem = fmaf(st[i][q], kv[i][q], mem);
                }
            }
            total(qq, 0, 0), total(kk, 1, 0), total(mem, 2, 0);
            __syncthreads();
            qq = red[0][n][0][lr] + red[0][n + 2][0][lr];
            kk = red[0][n][1][lr] + red[0][n + 2][1][lr];
            mem = red[0][n][2][lr] + red[0][n + 2][2][lr];
            const float ks = 1.0f / sqrtf(kk + A.eps), beta = sigmoid_ieee(A.braw[rr * vh + h]);
            const float v = A.conv[rr * cdim + static_cast<size_t>(2) * A.key_heads * kGcKd + static_cast<size_t>(h) * vd + col];
            const float upd = (v - mem * ks) * beta * ks;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    st[i][q] = fmaf(kv[i][q], upd, st[i][q]);
                    o = fmaf(st[i][q], qv[i][q], o);
                }
            total(o, 0, 1);
            __syncthreads();
            if (kh == 0 && lk == 0) orow[t * ostep] = (red[1][n][0][lr] + red[1][n + 2][0][lr]) * (rkd / sqrtf(qq + A.eps));
        }
        __syncthreads();
    };

    offsets(kGcC - 1);
#pragma unroll
    for (int part = 0; part < 3; ++part) issue(ca, part);
    const bool flagged = lane < cb - ca && slot0[lane * cstep + GcSlot::SC + GcSlot::BAD] != 0.0f;
    const uint64_t bad = __ballot(flagged);  // chunk ca + i of this launch: bit i
    vq::wait_vm<0>();
    st_mag = state_mag();
    for (int c = ca; c < cb; ++c) {
        __syncthreads();  // chunk c landed for every wave; every wave is done with chunk c - 1's buffer
        bool done = false;
        if ((bad >> (c - ca) & 1) == 0) {
            done = chunk(c);
        } else {
#pragma unroll
            for (int part = 0; part < 3; ++part)
                if (c + 1 < cb) issue(c + 1, part);
        }
        if (!done) {
            serial(c);
            st_mag = state_mag();
            vq::wait_vm<0>();
        }
    }
    if (cb == nch && !write_state) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t e = static_cast<size_t>(64 * kh + 16 * i + 4 * lk + q) * vd + col;
            if (cb == nch) st_state(S + e, st[i][q]);
            else Sx[e] = st[i][q];
        }
}

// The chunked path takes these shapes (every row offset 16-byte aligned) ...
bool gc_shape(int key_heads, int value_heads, int kd, int vd) {
    return kd == kGcKd && vd % kGcCols == 0 && vd <= kGcMaxVd && key_heads >= 1 && value_heads >= key_heads &&
           value_heads % key_heads == 0;
}
// ... for these segments of a pass (the longest first), which run in groups.
int gc_segments(const SegTable &T, SegTable *longs, SegTable *shorts) {
    SegTable L{}, H{};
    for (int i = 0; i < T.n; ++i) {
        SegTable &d = T.s[i].rows >= kGcMinRows ? L : H;
        d.s[d.n++] = T.s[i];
        d.total += T.s[i].rows;
    }
    std::stable_sort(L.s, L.s + L.n, [](const Seg &x, const Seg &y) { return x.rows > y.rows; });
    if (longs) *longs = L;
    if (shorts) *shorts = H;
    return L.n;
}
// The group that starts at segment i: its segments, the chunks of its longest one and those of a launch pair.
struct GcGroup {
    int n, chunks, cr;
    size_t slots(int value_heads) const { return static_cast<size_t>(n) * cr * value_heads * GcSlot::floats; }
};
GcGroup gc_group(const SegTable &L, int i, int value_heads) {
    const size_t budget = std::max<size_t>(1, kGcGroupBytes / (value_heads * GcSlot::floats * sizeof(float)));
    GcGroup g;
    g.chunks = (L.s[i].rows + kGcC - 1) / kGcC;
    g.cr = static_cast<int>(std::min<size_t>(std::min(g.chunks, kGcRound), budget));
    g.n = std::min(std::max(1, static_cast<int>(budget / g.cr)), L.n - i);
    return g;
}
size_t gc_ws_bytes(const SegTable &T, int key_heads, int value_heads, int kd, int vd) {
    if (!gc_shape(key_heads, value_heads, kd, vd)) return 0;
    SegTable L;
    gc_segments(T, &L, nullptr);
    size_t floats = 0;
    for (int i = 0; i < L.n;) {
        const GcGroup g = gc_group(L, i, value_heads);
        const size_t copy = g.chunks > g.cr ? static_cast<size_t>(g.n) * value_heads * kGcKd * vd : 0;
        floats = std::max(floats, g.slots(value_heads) + copy);
        i += g.n;
    }
    return floats * sizeof(float);
}

template <typename ST>
int gc_launch(const SegTable &L, const float *conv, const float *b, const float *a, const float *ssm_a, const float *dt,
              ST *state, float *out, int key_heads, int value_heads, int vd, float eps, int head_order, int write_state,
              float *ws, hipStream_t s) {
    for (int i = 0; i < L.n;) {
        const GcGroup g = gc_group(L, i, value_heads);
        SegTable T{};
        for (T.n = 0; T.n < g.n; ++T.n) T.s[T.n] = L.s[i + T.n];
        i += g.n;
        GcArgs A{conv, b, a, ssm_a, dt, ws, key_heads, value_heads, vd, head_order, 0, g.cr, eps};
        float *const tmp = ws + g.slots(value_heads);
        for (; A.c0 < g.chunks; A.c0 += A.cr) {
            gd_prep_kernel<<<dim3(value_heads, std::min(A.cr, g.chunks - A.c0), T.n), 256, 0, s>>>(A, T);
            gd_chunk_kernel<ST><<<dim3(value_heads * (vd / kGcCols), T.n), 256, 0, s>>>(A, T, state, tmp, out, write_state);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return status_of(e);
        }
    }
    return VQ_OK;
}

}  // namespace
