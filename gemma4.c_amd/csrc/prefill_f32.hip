// prefill_f32.hip -- Y[m x d] = X[m x n] . W[d x n]^T for fp32 activations
// and Q6_K or bf16 weights on the 16-bit matrix cores (g4_mm_batch; the
// reference's mm_quant_rows and mm_bf16 once per token,
// gemma4-4b/cpu-blas/main.c:1539-1556, 1529-1537).
//
// Products.  bf16: an fp32 activation is the exact sum of three bf16 terms
// (8 + 8 + 8 significant bits, by truncation), so three
// v_mfma_f32_16x16x32_bf16 give the fp32 path's products exactly.  Q6_K: over
// 64 elements of a token the activations are scaled by the power of two that
// brings the largest into [2^14, 2^15) and split into two fp16 terms (within
// 2^-22 of an element or 2^-39 of the largest of the 64, whichever is more; the
// product of both low terms, below 2^-22 of its term, is left out), the integer weight sc * (q - 32) exactly into
// Wh + Wl as in mm_batch_q6s_kernel; three v_mfma_f32_16x16x32_f16, then one
// multiplication by the token's scale and one FMA with the block's d.
// Outputs that are not finite are computed again by plain fp32 dots, so
// infinities and NaN in either operand behave as in the fp32 product.  A wave
// takes one dot after the other (Q6_K 2560 x 10240 over 512 tokens: 0.14 ms, with
// one infinite token 0.9, all of them 12; bf16 10752 x 2560 0.13, 0.8, 19; with a
// thread to a dot one token took 42 and 10 ms).
//
// Work split.  The four waves of a workgroup share one output tile and split
// K: wave w takes the Q6_K blocks b = w (mod 4), or of every 256 bf16
// elements those from 64 w, and the four partial tiles are added through LDS
// at the end, (a0 + a1) + (a2 + a3).  A wave thus needs each operand once, reads
// nothing that another wave brought (no barrier in the loop), and splits each
// activation and decodes each weight once per workgroup.  The order of a token's
// sums depends on n alone, so every tile shape gives the same bits.
#include "g4_device.h"
#include "g4_internal.h"
#include "g4_tile.h"

namespace g4 {
namespace {

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));

// thread t of nt's part of the fp32 dot of a weight row and x (four elements in
// nt * 4; nblk: Q6_K blocks of the matrix)
template <bool BF>
__device__ __forceinline__ float row_dot(const void* w, size_t nblk, const float* x, int n, size_t row, int t, int nt) {
    f4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (size_t k = 4 * (size_t)t; k < (size_t)n; k += 4 * (size_t)nt) {
        const float4 xv = *reinterpret_cast<const float4*>(x + k);
        float wv[4];
        if (BF) {
            const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(w) + row * n + k);
            wv[0] = __uint_as_float(u.x << 16);
            wv[1] = __uint_as_float(u.x & 0xffff0000u);
            wv[2] = __uint_as_float(u.y << 16);
            wv[3] = __uint_as_float(u.y & 0xffff0000u);
        } else {
            // as dequant_elem, whose bytes for four elements in a row are a word each
            const size_t blk = row * ((size_t)n >> 8) + (k >> 8);
            const Q6KPlanes P = q6k_planes(nblk);
            const uint8_t* wb = static_cast<const uint8_t*>(w);
            const int e0 = (int)(k & 255), h = e0 >> 7, kk = (e0 & 127) >> 5, l = e0 & 31;
            const uint32_t ql = *reinterpret_cast<const uint32_t*>(wb + P.ql + blk * 128 + 64 * h + 16 * (l >> 3) + (l & 7) + 8 * (kk & 1));
            const uint32_t qh = *reinterpret_cast<const uint32_t*>(wb + P.qh + blk * 64 + 32 * h + l);
            const float sc = (float)(int8_t)wb[P.sc + blk * 16 + 8 * h + (l >> 4) + 2 * kk];
            const float ds = hbits_to_f32(*reinterpret_cast<const uint16_t*>(wb + P.d + blk * 2)) * sc;
            const uint32_t q = ((ql >> (4 * (kk >> 1))) & 0x0f0f0f0fu) | (((qh >> (2 * kk)) & 0x03030303u) << 4);
#pragma unroll
            for (int e = 0; e < 4; e++) wv[e] = ds * (float)((int)byte_of(q, e) - 32);
        }
        s[0] = __builtin_fmaf(wv[0], xv.x, s[0]);
        s[1] = __builtin_fmaf(wv[1], xv.y, s[1]);
        s[2] = __builtin_fmaf(wv[2], xv.z, s[2]);
        s[3] = __builtin_fmaf(wv[3], xv.w, s[3]);
    }
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// the sum over the four waves' partial tiles and the store.  Weights are the
// A operand: lane (g, i) holds weight rows 4g + v of 16-row group rt and token
// i of 16-token group nt.  T: 16x16 tiles per wave; red_tiles(T) of them
// pass through LDS at a time.
constexpr int red_tiles(int t) { return t < 10 ? t : 10; }

template <int NT, int RT, class Dot>
__device__ __forceinline__ void reduce_store(f4_t (&acc)[RT][NT], f4_t* red, int part, float* __restrict__ out, int row0,
                                             int tok0, int d, int m, bool vec, Dot part_dot) {
    constexpr int T = NT * RT, R = red_tiles(T);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
#pragma unroll
    for (int t0 = 0; t0 < T; t0 += R) {
        if (t0) __syncthreads();
#pragma unroll
        for (int t = t0; t < t0 + R; t++)
            if (t < T) red[(part * R + (t - t0)) * 64 + lane] = acc[t / NT][t % NT];
        __syncthreads();
        auto sums = [&](int u, float (&v)[4]) {   // tile t0 + u
            const f4_t* r = red + u * 64 + lane;
            const f4_t a = r[0], b = r[R * 64], c = r[2 * R * 64], e = r[3 * R * 64];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = (a[k] + b[k]) + (c[k] + e[k]);
        };
        uint32_t again = 0;   // the wave's tiles with an output that is not finite
#pragma unroll
        for (int t = t0; t < t0 + R; t++) {
            if (t >= T || (t & 3) != wave) continue;
            float v[4], chk = 0.0f;
            sums(t - t0, v);
#pragma unroll
            for (int k = 0; k < 4; k++) chk = __builtin_fmaf(v[k], 0.0f, chk);
            if (__ballot(chk != 0.0f)) again |= 1u << (t - t0);
            const int row = row0 + 16 * (t / NT) + 4 * g, tok = tok0 + 16 * (t % NT) + i;
            if (tok >= m) continue;
            float* o = out + (size_t)tok * d + row;
            if (vec && row + 3 < d) {
                *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (row + k < d) o[k] = v[k];
            }
        }
        for (; again; again &= again - 1) {
            const int u = __builtin_ctz(again), t = t0 + u;
            const int row = row0 + 16 * (t / NT) + 4 * g, tok = tok0 + 16 * (t % NT) + i;
            float v[4];
            sums(u, v);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                unsigned long long todo = __ballot(tok < m && row + k < d && !(fabsf(v[k]) <= 3.402823466e38f));
                for (; todo; todo &= todo - 1) {
                    const int l = __builtin_ctzll(todo), tl = __builtin_amdgcn_readlane(tok, l), rl = __builtin_amdgcn_readlane(row, l) + k;
                    const float s = wave_sum(part_dot(tl, rl));
                    if (lane == l) out[(size_t)tl * d + rl] = s;
                }
            }
        }
    }
}

// ---- bf16 weights ---------------------------------------------------------
// Activations come by copies of whole lines (below: mm_batch_q6_kernel), a unit of
// 64 elements (two lines a token) ahead; weight rows straight into registers.
// Line (s, token): chunk c of 16 bytes in slot c ^ bf_swz(token).
__device__ __forceinline__ int bf_swz(int t) { return ((t >> 1) & 1) | ((t >> 1) & 4); }

template <int NT, int RT>
__global__ __launch_bounds__(256) void mm_batch_bf16_kernel(const uint16_t* __restrict__ w, const float* __restrict__ x,
                                                            float* __restrict__ out, int n, int d, int m, int vec) {
    constexpr int kUnit = 4096 * NT;      // bytes of a unit of the tile's tokens
    constexpr size_t kRed = sizeof(f4_t) * 4 * red_tiles(NT * RT) * 64, kStages = (size_t)4 * 2 * kUnit;
    __shared__ __align__(16) uint8_t lds[kStages > kRed ? kStages : kRed];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    int bx, by;
    xcd_tile((m + 16 * NT - 1) / (16 * NT), bx, by);
    const int row0 = bx * 16 * RT, tok0 = by * 16 * NT;
    const int nb = n >> 8;
    uint8_t* stages = lds + (size_t)wave * 2 * kUnit;
    uint32_t vx[NT][2], vw[RT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int t = 8 * q + (lane >> 3);
            vx[nt][q] = (uint32_t)(min(tok0 + 16 * nt + t, m - 1) - tok0) * (uint32_t)n * 4u +
                        16u * (uint32_t)((lane & 7) ^ bf_swz(t));
        }
#pragma unroll
    for (int rt = 0; rt < RT; rt++) vw[rt] = (uint32_t)(min(row0 + 16 * rt + i, d - 1) - row0) * (uint32_t)n * 2u + 16u * g;
    // of the wave's 64 elements of a block, step s of two takes 32 s .. + 31, lane
    // group g 8 of them.  (The block's address goes into the descriptors: offsets
    // stay within a tile's rows.)
    uint4 W[2][RT][2];
    auto load = [&](int b, int st) {
        const size_t o = (size_t)b * 256 + 64 * wave;
        const __amdgpu_buffer_rsrc_t rx =
            __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)tok0 * n + o), (short)0, -1, kBufWord3);
        const __amdgpu_buffer_rsrc_t rw =
            __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)row0 * n + o), (short)0, -1, kBufWord3);
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int q = 0; q < 4; q++)   // lines 8 q .. 8 q + 7: step q / 2, tokens 8 (q & 1) ..
                buf_load_lds16(rx, stages + st * kUnit + nt * 4096 + q * 1024, (int)vx[nt][q & 1], 128 * (q >> 1));
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int k = 0; k < 2; k++) W[st][rt][k] = buf_load16(rw, (int)vw[rt], 64 * k);
    };
    f4_t acc[RT][NT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[rt][nt] = f4_t{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int st) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            b8_t xt[3][NT];
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint8_t* line = stages + st * kUnit + nt * 4096 + (16 * s + i) * 128;
                const uint4 f0 = *reinterpret_cast<const uint4*>(line + 16 * ((2 * g) ^ bf_swz(i)));
                const uint4 f1 = *reinterpret_cast<const uint4*>(line + 16 * ((2 * g + 1) ^ bf_swz(i)));
                uint32_t f[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
#pragma unroll
                for (int t = 0; t < 3; t++) {
                    uint32_t p[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) p[k] = __builtin_amdgcn_perm(f[2 * k + 1], f[2 * k], 0x07060302u);
                    xt[t][nt] = __builtin_bit_cast(b8_t, make_uint4(p[0], p[1], p[2], p[3]));
                    if (t == 2) break;
#pragma unroll
                    for (int k = 0; k < 8; k++)   // exact: the bits below the term's
                        f[k] = __float_as_uint(__uint_as_float(f[k]) - __uint_as_float(f[k] & 0xffff0000u));
                }
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                const b8_t a = __builtin_bit_cast(b8_t, W[st][rt][s]);
#pragma unroll
                for (int t = 2; t >= 0; t--)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++)
                        acc[rt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, xt[t][nt], acc[rt][nt], 0, 0, 0);
            }
        }
    };
    // a block's operands, sent a block ago, have landed; the next one's are sent
    // while it is multiplied (past the end the last block again, read by nobody)
    auto block = [&](int b, int st) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        asm volatile("" ::: "memory");
        load(min(b + 1, nb - 1), st ^ 1);
        compute(st);
    };
    load(0, 0);
    for (int b = 0; b < nb; b += 2) {
        block(b, 0);
        if (b + 1 < nb) block(b + 1, 1);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));   // the last copies land before the sums take their place
    __syncthreads();
    f4_t* red = reinterpret_cast<f4_t*>(lds);
    reduce_store<NT, RT>(acc, red, wave, out, row0, tok0, d, m, vec, [&](int tok, int row) {
        return row_dot<true>(w, 0, x + (size_t)tok * n, n, (size_t)row, lane, 64);
    });
}

// ---- bf16 weights on the fp32 matrix cores -----------------------------------
// g4_mm_batch_bf16_f32: fp32 products and one running fp32 sum per output
// (v_mfma_f32_16x16x4_f32).  A prompt's per-layer-embedding projection stays
// on it (0.27 ms of a 511-token E4B prompt against 0.16 ms): its rows end up in
// 8-bit codes, where a sum in another order moves some code by one and the
// model carries that on, so a prompt would no longer give the bits, nor always
// the tokens, it gave before.
//
// The 16 tokens of a tile are the A rows, 16 weight rows the B columns, so a
// lane's results are one weight row of four tokens.  Lane group g supplies K
// index g of every 16x16x4 step; over one 256-long block it walks elements
// 64 g .. 64 g + 63 of its row.  The activations of the workgroup's tokens are
// staged per block in LDS in natural order (260 floats per token:
// conflict-free 16-byte reads).
constexpr int kF32XS = 260;

template <int RW, int NT>
__global__ __launch_bounds__(64 * RW) void mm_batch_f32_kernel(const uint16_t* __restrict__ w,
                                                               const float* __restrict__ x, float* __restrict__ out,
                                                               int n, int d, int m) {
    constexpr int NTHR = 64 * RW;
    constexpr int TOK = 16 * NT;
    constexpr int XV = TOK * 64 / NTHR;             // float4 of activations per thread and block
    static_assert(XV * NTHR == TOK * 64, "token tile must divide among the threads");
    __shared__ __align__(16) float sx[TOK * kF32XS];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * (16 * RW) + wave * 16;
    const int tok0 = blockIdx.y * TOK;
    const int nb = n >> 8;
    const size_t rj = (size_t)min(row0 + i, d - 1);  // this lane's weight row

    struct WRaw {
        uint4 v[8];     // 64 values
    };
    auto load_w = [&](int b, WRaw& r) {
        const uint4* p = reinterpret_cast<const uint4*>(w + rj * n + (size_t)b * 256 + 64 * g);
#pragma unroll
        for (int k = 0; k < 8; k++) r.v[k] = p[k];
    };
    struct XRaw {
        f4_t v[XV];
    };
    // unit u = tid + j * NTHR: token u >> 6, float4 u & 63 of the block
    auto load_x = [&](int b, XRaw& r) {
#pragma unroll
        for (int j = 0; j < XV; j++) {
            const int u = tid + j * NTHR;
            const int t = min(tok0 + (u >> 6), m - 1);
            r.v[j] = reinterpret_cast<const f4_t*>(x + (size_t)t * n + (size_t)b * 256)[u & 63];
        }
    };
    auto stage = [&](const XRaw& r) {
#pragma unroll
        for (int j = 0; j < XV; j++) {
            const int u = tid + j * NTHR;
            *reinterpret_cast<f4_t*>(sx + (u >> 6) * kF32XS + 4 * (u & 63)) = r.v[j];
        }
    };

    f4_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f4_t{0.f, 0.f, 0.f, 0.f};

    WRaw wn;
    XRaw xn;
    load_w(0, wn);
    load_x(0, xn);
    for (int b = 0; b < nb; b++) {
        lds_barrier();   // the previous block's LDS reads are done
        stage(xn);
        const WRaw wc = wn;
        // the next block (the last one again at the end: an unconditional
        // load keeps the prefetch registers out of scratch memory)
        const int bn = min(b + 1, nb - 1);
        load_w(bn, wn);
        load_x(bn, xn);
        lds_barrier();

        const float* xa = sx + i * kF32XS;
#pragma unroll
        for (int t4 = 0; t4 < 16; t4++) {
            const uint32_t lo = t4 & 1 ? wc.v[t4 >> 1].z : wc.v[t4 >> 1].x;
            const uint32_t hi = t4 & 1 ? wc.v[t4 >> 1].w : wc.v[t4 >> 1].y;
            const float wv[4] = {__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u),
                                 __uint_as_float(hi << 16), __uint_as_float(hi & 0xffff0000u)};
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const float4 a = *reinterpret_cast<const float4*>(xa + 16 * t * kF32XS + 64 * g + 4 * t4);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, wv[0], acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, wv[1], acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, wv[2], acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, wv[3], acc[t], 0, 0, 0);
            }
        }
    }
    // lane (g, i) holds tokens 4g + v of each tile, weight row row0 + i
    const int row = row0 + i;
    if (row < d) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int tok = tok0 + 16 * t + 4 * g + v;
                if (tok < m) out[(size_t)tok * d + row] = acc[t][v];
            }
    }
}

// ---- Q6_K weights -----------------------------------------------------------
// A row group's next weights are loaded once its last group has been decoded, into
// the same registers; the other wave of the SIMD covers the wait.
// The activations come by global -> LDS copies of whole 128-byte lines, eight
// lines an instruction: an instruction costs the L1 four cycles for every line
// it touches, and loads straight into operand order (a 16-byte piece of 32 lines)
// had it busy the whole time.  Each wave copies its own groups, NS - 1 of them
// ahead (a group: the 64 elements a token of one scale, two 128-byte lines), and
// no other wave reads them, so there is no barrier in the loop.  Line (h, token):
// chunk c of 16 bytes lies in slot c ^ line_swz(token), which spreads the sixteen
// lanes that LDS serves at once over all banks.
__device__ __forceinline__ int line_swz(int t) { return ((t >> 1) & 1) | ((t >> 2) & 2); }

template <int NT, int RT, int NS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void mm_batch_q6_kernel(
    const uint8_t* __restrict__ w, const float* __restrict__ x, float* __restrict__ out, int n, int d, int m, int vec) {
    static_assert(NS == 2 || NS == 4, "a block's four groups use the stages in turn");
    constexpr int kGroup = 4096 * NT;     // bytes of a group of the tile's tokens
    constexpr size_t kRed = sizeof(f4_t) * 4 * red_tiles(NT * RT) * 64, kStages = (size_t)4 * NS * kGroup;
    __shared__ __align__(16) uint8_t lds[kStages > kRed ? kStages : kRed];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4, h = g >> 1, s = g & 1;
    int bx, by;
    xcd_tile((m + 16 * NT - 1) / (16 * NT), bx, by);
    const int row0 = bx * 16 * RT, tok0 = by * 16 * NT;
    const int nb = n >> 8;
    // the wave's part of K: workgroups that share a CU give their longer parts to different SIMDs
    const int part = (wave + 2 * (blockIdx.x >> 8) + (blockIdx.x >> 9)) & 3;
    const size_t nblk = (size_t)d * nb;
    const Q6KPlanes P = q6k_planes(nblk);

    // copy q of a group and 16-token tile: lines 8 q .. 8 q + 7, line l is half
    // l / 16 of token l % 16
    uint8_t* stages = lds + (size_t)wave * NS * kGroup;
    uint32_t vx[NT][2];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int t = 8 * q + (lane >> 3);
            vx[nt][q] = (uint32_t)(min(tok0 + 16 * nt + t, m - 1) - tok0) * (uint32_t)n * 4u +
                        16u * (uint32_t)((lane & 7) ^ line_swz(t));
        }
    auto copy_x = [&](int b, int k, int st) {
        // (the block's address goes into the descriptor: offsets stay within a tile's rows)
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(x + (size_t)tok0 * n + (size_t)b * 256 + 32 * k), (short)0, -1, kBufWord3);
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                buf_load_lds16(rx, stages + st * kGroup + nt * 4096 + q * 1024, (int)vx[nt][q & 1], 512 * (q >> 1));
    };

    // lane group g's elements of a block: 128 h + 32 k + 16 s + 8 half + t, in
    // step c = 2 k + half (layout.hip); group k of two steps is 16 in a row
    uint32_t rB[RT];                      // first block of the row, from the tile's first row's
#pragma unroll
    for (int rt = 0; rt < RT; rt++) rB[rt] = (uint32_t)(min(row0 + 16 * rt + i, d - 1) - row0) * (uint32_t)nb;
    const size_t b0 = (size_t)row0 * nb;
    auto rsrc = [&](size_t off) { return __builtin_amdgcn_make_buffer_rsrc((void*)(w + off), (short)0, -1, kBufWord3); };
    const __amdgpu_buffer_rsrc_t rql = rsrc(P.ql + b0 * 128), rqh = rsrc(P.qh + b0 * 64), rsc = rsrc(P.sc + b0 * 16),
                                 rd = rsrc(P.d + b0 * 2);
    struct WRaw {
        uint4 ql[RT][2];
        uint4 qh[RT];
        uint2 sc[RT];
        uint32_t dh[RT];
    };
    WRaw wr;
    auto load_w = [&](int b, int rt) {
        wr.ql[rt][0] = buf_load16(rql, (int)(rB[rt] * 128 + 32 * g), b * 128);
        wr.ql[rt][1] = buf_load16(rql, (int)(rB[rt] * 128 + 32 * g + 16), b * 128);
        wr.qh[rt] = buf_load16(rqh, (int)(rB[rt] * 64 + 16 * g), b * 64);
        wr.sc[rt] = buf_load8(rsc, (int)(rB[rt] * 16 + 8 * h), b * 16);
        wr.dh[rt] = __builtin_amdgcn_raw_buffer_load_b16(rd, (int)(rB[rt] * 2), b * 2, 0);
    };

    f4_t acc[RT][NT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[rt][nt] = f4_t{0.f, 0.f, 0.f, 0.f};
    const h2_t m1056 = {(_Float16)-1056.0f, (_Float16)-1056.0f};

    auto group = [&](int st, int k, int bn, const float (&dw)[RT][4]) {
        h8_t Xh[2][NT], Xl[2][NT];
        float ts[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            f4_t f[4];
            float mx = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                f[q] = *reinterpret_cast<const f4_t*>(stages + st * kGroup + nt * 4096 + (16 * h + i) * 128 +
                                                      16 * ((4 * s + q) ^ line_swz(i)));
                mx = max3_abs(f[q][2], f[q][3], max3_abs(f[q][0], f[q][1], mx));
            }
            // the largest of the token's 64 (lanes i, i + 16, i + 32, i + 48)
            const uint32_t u = __float_as_uint(mx);
            const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
            const uint32_t u2 = max(p[0], p[1]);   // (non-negative floats order as their bits)
            const auto q2 = __builtin_amdgcn_permlane16_swap(u2, u2, false, false);
            const int e = (int)(max(q2[0], q2[1]) >> 23);
            const int fe = min(268 - e, 253);      // 2^(fe - 127) * mx in [2^14, 2^15)
            const float sf = __uint_as_float((uint32_t)fe << 23);
            ts[nt] = __uint_as_float((uint32_t)(254 - fe) << 23);
#pragma unroll
            for (int st2 = 0; st2 < 2; st2++) {
                h2v_t hi[4], lo[4];
#pragma unroll
                for (int q = 0; q < 4; q++)
                    split2(f[2 * st2 + (q >> 1)][2 * (q & 1)], f[2 * st2 + (q >> 1)][2 * (q & 1) + 1], sf, hi[q], lo[q]);
                Xh[st2][nt] = __builtin_bit_cast(h8_t, make_uint4(h2_bits(hi[0]), h2_bits(hi[1]), h2_bits(hi[2]), h2_bits(hi[3])));
                Xl[st2][nt] = __builtin_bit_cast(h8_t, make_uint4(h2_bits(lo[0]), h2_bits(lo[1]), h2_bits(lo[2]), h2_bits(lo[3])));
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const int sb = 2 * k + s;   // sub-block 8 h + 2 k + s
            const _Float16 scf = (_Float16)(float)(int)(int8_t)byte_of(sb < 4 ? wr.sc[rt].x : wr.sc[rt].y, sb & 3);
            const h2_t SC = {scf, scf};
            f4_t S[NT];
#pragma unroll
            for (int half = 0; half < 2; half++) {
                // codes of step 2 k + half: ql bytes 16 half + 8 (k & 1) + t, nibble
                // k >> 1; qh bytes 8 half + t, bits 2 k .. 2 k + 1
                const uint4 L = wr.ql[rt][half];
                const uint32_t l0 = (k & 1) ? L.z : L.x, l1 = (k & 1) ? L.w : L.y;
                const uint32_t h0 = half ? wr.qh[rt].z : wr.qh[rt].x, h1 = half ? wr.qh[rt].w : wr.qh[rt].y;
                const uint32_t q0 = ((l0 >> (4 * (k >> 1))) & 0x0f0f0f0fu) | (((h0 >> (2 * k)) & 0x03030303u) << 4);
                const uint32_t q1 = ((l1 >> (4 * (k >> 1))) & 0x0f0f0f0fu) | (((h1 >> (2 * k)) & 0x03030303u) << 4);
                const h2_t v0 = bits_h2(__builtin_amdgcn_perm(kMagic, q0, kSelLo)) + m1056;
                const h2_t v1 = bits_h2(__builtin_amdgcn_perm(kMagic, q0, kSelHi)) + m1056;
                const h2_t v2 = bits_h2(__builtin_amdgcn_perm(kMagic, q1, kSelLo)) + m1056;
                const h2_t v3 = bits_h2(__builtin_amdgcn_perm(kMagic, q1, kSelHi)) + m1056;
                const h2_t w0 = v0 * SC, w1 = v1 * SC, w2 = v2 * SC, w3 = v3 * SC;
                const h8_t Wa = __builtin_bit_cast(h8_t, make_uint4(h2_bits(w0), h2_bits(w1), h2_bits(w2), h2_bits(w3)));
                const h8_t Wb = __builtin_bit_cast(
                    h8_t, make_uint4(h2_bits(__builtin_elementwise_fma(v0, SC, -w0)), h2_bits(__builtin_elementwise_fma(v1, SC, -w1)),
                                     h2_bits(__builtin_elementwise_fma(v2, SC, -w2)), h2_bits(__builtin_elementwise_fma(v3, SC, -w3))));
                const f4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int nt = 0; nt < NT; nt++) S[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Wa, Xh[half][nt], half ? S[nt] : zero, 0, 0, 0);
#pragma unroll
                for (int nt = 0; nt < NT; nt++) S[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Wa, Xl[half][nt], S[nt], 0, 0, 0);
#pragma unroll
                for (int nt = 0; nt < NT; nt++) S[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Wb, Xh[half][nt], S[nt], 0, 0, 0);
            }
            if (k == 3) load_w(bn, rt);   // the row group's next block, into the registers just read
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    acc[rt][nt][v] = __builtin_fmaf(S[nt][v] * ts[nt], dw[rt][v], acc[rt][nt][v]);
        }
    };
    auto block = [&](int b) {
        const int bn = b + 4 < nb ? b + 4 : b;   // (the last block again at the end: no branch around the loads)
        float dw[RT][4];                         // d of rows 4 g + v
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const float dl = hbits_to_f32(wr.dh[rt]);
#pragma unroll
            for (int v = 0; v < 4; v++) dw[rt][v] = __shfl(dl, 4 * g + v, 64);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // this group's copies have landed: at most the ones of the NS - 2
            // groups after it are in flight (weight loads among them only make
            // the wait longer), and the group before it has been read
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(4 * NT * (NS - 2)));
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);   // (a group's operands are not formed ahead of it)
            constexpr int kAhead = NS - 1;
            copy_x(k + kAhead < 4 ? b : bn, (k + kAhead) & 3, (k + kAhead) & (NS - 1));
            group(k & (NS - 1), k, bn, dw);
        }
    };
    if (part < nb) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) load_w(part, rt);
#pragma unroll
        for (int k = 0; k < NS - 1; k++) copy_x(part, k, k);
        for (int b = part; b < nb; b += 4) block(b);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));   // the last copies, read by nobody, land before the sums go there
    __syncthreads();
    f4_t* red = reinterpret_cast<f4_t*>(lds);
    reduce_store<NT, RT>(acc, red, part, out, row0, tok0, d, m, vec, [&](int tok, int row) {
        return row_dot<false>(w, nblk, x + (size_t)tok * n, n, (size_t)row, lane, 64);
    });
}

// Rows of 2^24 elements and more, where a tile's rows leave the 32-bit offsets of
// the kernels above (Q6_K: sixteen rows of 5.7e8): a workgroup per output, every
// address in 64 bits, bound by the loads that a workgroup keeps in flight.  16 rows
// of 2^24, one / eight tokens: Q6_K 8.9 / 8.8 ms (28 / 224 in a launch a token),
// bf16 7.4 / 7.1 (792 / 6490 in a launch an output).
template <bool BF>
__global__ __launch_bounds__(256) void mm_batch_long_kernel(const void* w, const float* __restrict__ x, float* __restrict__ out,
                                                            int n, int d) {
    __shared__ float red[16];
    const size_t row = blockIdx.x, tok = blockIdx.y;
    const float s = block_sum(row_dot<BF>(w, (size_t)d * (n >> 8), x + tok * n, n, row, threadIdx.x, 256), red);
    if (threadIdx.x == 0) out[tok * d + row] = s;
}

// Tile shapes.  The table holds the times in us of one workgroup on a CU and of
// two that share it, with every CU taken (MI355X, 10240 columns, a sweep of all
// shapes over 2..512 tokens); a launch runs in rounds of two a CU and the
// cheapest shape is taken, so small batches get small tiles and more
// workgroups.  Two Q6_K tiles of 32 tokens x 80 rows take less than one of 64 x
// 80 (122 against 130 us): the second wave of a SIMD covers the first one's
// waits, and their shares of K differ (mm_batch_q6_kernel).  us, and in brackets
// the same kernels with rounds of one a CU, where the long-K shapes took tiles of 64
// tokens, and the fp32 matrix cores before:
//   bf16 10752 x 2560, 512 tokens: 64 x 128 tiles 128 (128, 307); 2560 x 10240, 256
//     tokens, 32 x 80 69 (82), 512 tokens, 64 x 96 107 (116); 10240 x 2560, 37 tokens,
//     64 x 64 22 (25)
//   Q6_K 2560 x 10240, 512 tokens: 32 x 80 tiles 122 (127 -- 137, 344); 10240 x 2560,
//     512 tokens 131 -- 140 (180), 256 tokens 70 (91), 100 tokens 39 (45); 37 tokens, 16 x
//     32 30 (31, 94); 2560 x 256, 512 tokens 10.8 (17).
//     VALU issue (splits and decode) and the products share the SIMDs.
struct Tile {
    int nt, rt, one, two;
    void (*launch)(const void* w, const float* x, float* o, int n, int d, int m);
};

template <int NT, int RT>
void launch_bf16(const void* w, const float* x, float* o, int n, int d, int m) {
    const int gx = (d + 16 * RT - 1) / (16 * RT), gy = (m + 16 * NT - 1) / (16 * NT);
    hipLaunchKernelGGL((mm_batch_bf16_kernel<NT, RT>), dim3(gx * gy), dim3(256), 0, g4_stream(), (const uint16_t*)w, x, o, n,
                       d, m, (int)(d % 4 == 0 && al16(o)));
}
template <int NT, int RT, int NS>
void launch_q6(const void* w, const float* x, float* o, int n, int d, int m) {
    const int gx = (d + 16 * RT - 1) / (16 * RT), gy = (m + 16 * NT - 1) / (16 * NT);
    hipLaunchKernelGGL((mm_batch_q6_kernel<NT, RT, NS>), dim3(gx * gy), dim3(256), 0, g4_stream(), (const uint8_t*)w, x, o, n, d,
                       m, (int)(d % 4 == 0 && al16(o)));
}

const Tile kTilesBf16[] = {{1, 1, 37, 44, launch_bf16<1, 1>},  {1, 2, 42, 50, launch_bf16<1, 2>},
                           {2, 2, 50, 66, launch_bf16<2, 2>},  {2, 4, 67, 101, launch_bf16<2, 4>},
                           {2, 5, 74, 122, launch_bf16<2, 5>}, {4, 4, 89, 178, launch_bf16<4, 4>},
                           {4, 6, 112, 224, launch_bf16<4, 6>}, {4, 8, 141, 282, launch_bf16<4, 8>}};
const Tile kTilesQ6[] = {{1, 1, 20, 32, launch_q6<1, 1, 4>},  {1, 2, 28, 47, launch_q6<1, 2, 4>}, {2, 2, 42, 67, launch_q6<2, 2, 2>},
                         {2, 4, 62, 100, launch_q6<2, 4, 2>}, {2, 5, 75, 122, launch_q6<2, 5, 2>}};

template <int N>
const Tile& pick_tile(const Tile (&tiles)[N], int d, int m) {
    const long long cus = g4_num_cus();
    long long best = 0;
    int at = -1;
    for (int k = 0; k < N; k++) {
        const Tile& t = tiles[k];
        const long long wgs = (long long)((d + 16 * t.rt - 1) / (16 * t.rt)) * ((m + 16 * t.nt - 1) / (16 * t.nt));
        const long long rest = wgs % (2 * cus);
        const long long c = wgs / (2 * cus) * t.two + (rest > cus ? t.two : rest > 0 ? t.one : 0);
        if (at < 0 || c < best) best = c, at = k;
    }
    return tiles[at];
}

}  // namespace
}  // namespace g4

using namespace g4;

extern "C" int g4_mm_batch_bf16_f32(float* o, const float* x, const void* w, int n, int d, int m) {
    G4_CHECK_ARG(o && x && w, "g4_mm_batch_bf16_f32: null pointer");
    G4_CHECK_ARG(n > 0 && n % 256 == 0 && d > 0 && m > 0 && (m + 31) / 32 <= 65535, "g4_mm_batch_bf16_f32: n=%d d=%d m=%d", n,
                 d, m);
    G4_CHECK_ARG(al16(x) && al16(w), "g4_mm_batch_bf16_f32: x and w must be 16-byte aligned");
    // 64 rows x 32 tokens a workgroup (a sweep at the prompt's shape: 302 against 325 us at 64 x 16)
    hipLaunchKernelGGL((mm_batch_f32_kernel<4, 2>), dim3((d + 63) / 64, (m + 31) / 32), dim3(256), 0, g4_stream(),
                       (const uint16_t*)w, x, o, n, d, m);
    return g4_check_launch("mm_batch_f32_kernel");
}

int g4_mm_batch_f32(float* o, const float* x, const void* w, int n, int d, int m, int type) {
    if (n >= 1 << 24) {
        if (type == G4_BF16) hipLaunchKernelGGL(mm_batch_long_kernel<true>, dim3(d, m), dim3(256), 0, g4_stream(), w, x, o, n, d);
        else hipLaunchKernelGGL(mm_batch_long_kernel<false>, dim3(d, m), dim3(256), 0, g4_stream(), w, x, o, n, d);
        return g4_check_launch("mm_batch_long_kernel");
    }
    const Tile& t = type == G4_BF16 ? pick_tile(kTilesBf16, d, m) : pick_tile(kTilesQ6, d, m);
    // a grid holds fewer than 2^32 threads: outputs past 172 GB take several launches
    const int gx = (d + 16 * t.rt - 1) / (16 * t.rt), step = max(1, (1 << 23) / gx) * 16 * t.nt;
    for (int t0 = 0; t0 < m; t0 += step) t.launch(w, x + (size_t)t0 * n, o + (size_t)t0 * d, n, d, min(step, m - t0));
    return g4_check_launch(type == G4_BF16 ? "mm_batch_bf16_kernel" : "mm_batch_q6_kernel");
}
