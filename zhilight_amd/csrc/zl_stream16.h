// zl_stream16.h -- y (m, n) = x (m, k) . w (n, k)^T for up to 32 rows of 16-bit numbers (decode batches): the weights are the traffic, each is
// read once.
//
// A workgroup of W waves owns tiles of 16 columns, its waves share k: wave v takes the 64-k slices v, v + W, ...  Slices go global -> LDS by
// LDS-DMA into a ring of D that belongs to the wave alone -- no barrier in the stream, whole 128-byte lines per row (loads straight into
// MFMA operands take 64-byte runs), and the ring runs on into the next tile, so a tile's end drains nothing.  The matrix cores do the
// multiplying (weights: A operand, rows of x: B operand): the VALU dot products of one wave per row cost 80 instructions per KiB at 4 rows
// and six lane exchanges per row and column.  The waves' partial sums meet in LDS once per tile, added in wave order.
// x: its slices ride in the ring (XS = false), or all of it lies in LDS, optionally RMS-normalised on the way (XS = true, up to 4 rows).
// Measured (cold weights, us; before: k_dense_gemv at 4 rows, the packed k_dense_gemm or k_seq_gemv_mfma at 8): 4 x 6912 x 2304 15.7 -> 8.0, 4 x 2304 x
// 5760 15.1 -> 8.2, 4 x 122753 x 2304 176 -> 100 (5.7 TB/s); 8 x 4096 x 21504 53 -> 35 (5.0 TB/s), 8 x 2304 x 5760 50 -> 9, 8 x 128256 x 4096 196 -> 187.
#pragma once
#include "zl_gemm16.h"

struct Stream16P {
    const uint16_t* x; const uint16_t* w;
    int64_t ldx;
    int m, n, k;                                               // k % 64 == 0, rows of w are k numbers
    const uint16_t* norm_w; float norm_eps;                    // XS: nullable
    const uint16_t* w2;                                        // DUAL: a second matrix of n rows (gate and up rows of the same outputs)
};

constexpr int s16_xrow(int k) { return k * 2 + 64; }           // bytes of a row of x in LDS (XS): rows start 16 banks apart

// DUAL: a tile is 8 rows of w and the same 8 of w2, one load each; the two results of an output meet by a lane exchange
template <int DT, int MR, int W, int D, bool XS, bool DUAL, class Epi>
__global__ __launch_bounds__(64 * W) void k_stream16(const Stream16P p, Epi epi) {
    constexpr int kSlot = 2048 + (XS ? 0 : MR * 128), NL = 2 + (XS ? 0 : MR / 8), NB = (MR + 15) / 16;      // a slice's bytes and loads; blocks of 16 rows of x
    static_assert(XS ? MR <= 16 : MR % 8 == 0, "a load fills 8 rows");
    extern __shared__ __attribute__((aligned(1024))) unsigned char s16_smem[];
    float* red = reinterpret_cast<float*>(s16_smem + W * D * kSlot);                                        // [2][W][MR rows of x, whole 16s][17]
    unsigned char* xs = s16_smem + W * D * kSlot + 2 * W * NB * 16 * 17 * 4;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nrow = lane & 15, kq = lane >> 4;
    constexpr int TC = DUAL ? 8 : 16;                          // outputs of a tile
    const int tiles = (p.n + TC - 1) / TC, S = p.k >> 6, Sw = (S - wave + W - 1) / W;                           // slices of this wave per tile
    const int first = blockIdx.x, step = gridDim.x, mine = (tiles - first + step - 1) / step;
    const int total = mine * Sw;                                                                            // this wave's slices, all tiles
    // a load fills 8 rows of 128 bytes: lane l -> row l / 8, unit l % 8, which holds unit (l % 8) ^ (row / 2 % 8) of the slice
    const int lr = lane >> 3, lu = lane & 7;
    const uint32_t lds0 = (uint32_t)(size_t)(g16_lds)s16_smem + wave * D * kSlot;
    uint32_t xo[MR > 8 ? MR / 8 : 1];
#pragma unroll
    for (int i = 0; i < (MR > 8 ? MR / 8 : 1); ++i) xo[i] = (uint32_t)(min(lr + 8 * i, p.m - 1) * (int)p.ldx * 2 + ((lu ^ (((lr + 8 * i) >> 1) & 7)) * 16));
    const u32x4 rx = g16_rsrc(p.x);
    int i_tile = first, i_s = wave, issued = 0;
    auto issue = [&]() {                                       // the wave's next slice into slot issued % D
        const int c0 = i_tile * TC;
        const u32x4 rw = g16_rsrc(p.w + (size_t)c0 * p.k), rw2 = DUAL ? g16_rsrc(p.w2 + (size_t)c0 * p.k) : rw;
        const uint32_t at = lds0 + (uint32_t)(issued % D) * kSlot;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = lr + 8 * i;
            g16_dma(i ? rw2 : rw, (uint32_t)(min(DUAL ? lr : r, p.n - 1 - c0) * p.k * 2 + ((lu ^ ((r >> 1) & 7)) * 16)), (uint32_t)i_s * 128, at + i * 1024);
        }
        if constexpr (!XS) {
#pragma unroll
            for (int i = 0; i < MR / 8; ++i) g16_dma(rx, xo[i], (uint32_t)i_s * 128, at + 2048 + i * 1024);
        }
        ++issued;
        i_s += W;
        if (i_s >= S) { i_s = wave; i_tile += step; }
    };
    const int ahead = min(D, total);
    for (int i = 0; i < ahead; ++i) issue();
    if constexpr (XS) {
        for (int r = 0; r < MR; ++r) {
            const bool live = r < p.m;
            const uint16_t* xr = p.x + (size_t)r * p.ldx;
            uint16_t* xd = reinterpret_cast<uint16_t*>(xs + (size_t)r * s16_xrow(p.k));
            float ss = 0.f;
            for (int i = threadIdx.x * 8; i < p.k; i += 64 * W * 8) {
                const uint4 v = live ? *reinterpret_cast<const uint4*>(xr + i) : make_uint4(0, 0, 0, 0);
                if (p.norm_w) {
                    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float a = ZT<DT>::to_f32((uint16_t)(u[e] & 0xffffu)), c = ZT<DT>::to_f32((uint16_t)(u[e] >> 16));
                        ss = __builtin_fmaf(a, a, ss);
                        ss = __builtin_fmaf(c, c, ss);
                    }
                }
                *reinterpret_cast<uint4*>(xd + i) = v;
            }
            if (p.norm_w && live) {                            // (workgroup-uniform)
                ss = zl_block_sum(ss, red);
                const float rs = zl_rsqrt_rn(ss / (float)p.k + p.norm_eps);
                for (int i = threadIdx.x * 8; i < p.k; i += 64 * W * 8) {
                    const uint4 v = *reinterpret_cast<const uint4*>(xd + i), wv = *reinterpret_cast<const uint4*>(p.norm_w + i);
                    uint32_t u[4] = {v.x, v.y, v.z, v.w};
                    const uint32_t wu[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float a = ZT<DT>::to_f32((uint16_t)(u[e] & 0xffffu)) * rs * ZT<DT>::to_f32((uint16_t)(wu[e] & 0xffffu));
                        const float c = ZT<DT>::to_f32((uint16_t)(u[e] >> 16)) * rs * ZT<DT>::to_f32((uint16_t)(wu[e] >> 16));
                        u[e] = (uint32_t)ZT<DT>::from_f32(a) | ((uint32_t)ZT<DT>::from_f32(c) << 16);
                    }
                    *reinterpret_cast<uint4*>(xd + i) = make_uint4(u[0], u[1], u[2], u[3]);
                }
            }
        }
        __syncthreads();
    }
    const int sw = (nrow >> 1) & 7, u0 = (kq ^ sw) * 16, u1 = u0 ^ 64;
    const int xrow = NB > 1 ? nrow : nrow & (MR - 1);          // (columns of the MFMA's result past the rows of x are never read)
    int done = 0;
    for (int t = 0; t < mine; ++t) {
        g16_f4 acc[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = (g16_f4){0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < Sw; ++s, ++done) {
            if (issued - done >= D) g16_wait<(D - 1) * NL>();
            else g16_wait<0>();
            const unsigned char* slot = s16_smem + (size_t)(wave * D + done % D) * kSlot;
            const uint4 w0 = *reinterpret_cast<const uint4*>(slot + nrow * 128 + u0), w1 = *reinterpret_cast<const uint4*>(slot + nrow * 128 + u1);
            const unsigned char* x0 = XS ? xs + (size_t)xrow * s16_xrow(p.k) + (size_t)(wave + s * W) * 128 + kq * 16 : slot + 2048 + xrow * 128 + (kq ^ ((xrow >> 1) & 7)) * 16;
            const unsigned char* x1 = XS ? x0 + 64 : slot + 2048 + xrow * 128 + ((4 + kq) ^ ((xrow >> 1) & 7)) * 16;
            uint4 b0[NB], b1[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) { b0[b] = *reinterpret_cast<const uint4*>(x0 + b * 2048); b1[b] = *reinterpret_cast<const uint4*>(x1 + b * 2048); }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the slot is in registers: it may be filled again
            if (issued < total) issue();
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[b] = g16_mfma<DT>(w1, b1[b], g16_mfma<DT>(w0, b0[b], acc[b]));
        }
        float* rd = red + (t & 1) * (W * NB * 16 * 17);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) rd[((wave * NB + b) * 16 + nrow) * 17 + 4 * kq + r] = acc[b][r];      // row 16 b + nrow of x, column 4 kq + r
        __syncthreads();
        const int col = (first + t * step) * TC + (threadIdx.x & (TC - 1));
#pragma unroll
        for (int m = threadIdx.x >> 4; m < MR; m += 4 * W) {
            float v = 0.f;
#pragma unroll
            for (int u = 0; u < W; ++u) v += rd[(u * NB * 16 + m) * 17 + (threadIdx.x & 15)];
            if constexpr (DUAL) {
                const float u = __shfl_xor(v, 8, 64);          // (a wave's rows m are all below MR or none)
                if (m < p.m && col < p.n && !(threadIdx.x & 8)) epi.put2(m, col, v, u);
            } else if (m < p.m && col < p.n) epi.put(m, col, v);
        }
    }
    epi.finish();
}

// Up to 8 rows always.  More rows only for narrow matrices: a tile of 16 columns pulls all rows of x through the ring, which costs more than
// the weights' stream from about 16 k columns on (16 x 128256 x 4096: 214 us against 187 packed; 16 x 21504 x 4096 40 against 37; 16 x 6912 x 2304 9
// against 16; 32 x 2304 x 5760 12 against 35)
static inline bool s16_takes(const void* x, int64_t ldx, const void* w, int64_t m, int64_t n, int64_t k) {
    return m <= 32 && (m <= 8 || n <= 16384) && k % 64 == 0 && k <= (1 << 22) && n < (1 << 30) && ldx % 8 == 0 && ldx <= (1 << 22) &&
           (((uintptr_t)x | (uintptr_t)w) & 15) == 0;
}

template <int DT, int MR, int W, int D, bool XS, bool DUAL, class Epi>
int s16_launch_as(const Stream16P& p, const Epi& e, int grid, hipStream_t s) {
    const int lds = W * D * (2048 + (XS ? 0 : MR * 128)) + 2 * W * ((MR + 15) / 16) * 16 * 17 * 4 + (XS ? MR * s16_xrow(p.k) : 0);
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(&k_stream16<DT, MR, W, D, XS, DUAL, Epi>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return ZL_ELIMIT;
    hipLaunchKernelGGL((k_stream16<DT, MR, W, D, XS, DUAL, Epi>), dim3((unsigned)grid), dim3(64 * W), lds, s, p, e);
    return zl_launch_status();
}

// 8 waves to a tile: with few tiles every wave's ring counts, with many one workgroup per CU walks them (256 workgroups: within 2 % of more)
template <int DT, bool DUAL = false, class Epi>
int s16_launch(const Stream16P& p, const Epi& e, hipStream_t s) {
    const int tiles = DUAL ? (p.n + 7) / 8 : (p.n + 15) / 16, grid = tiles < 256 ? tiles : 256;
    if (p.m <= 8) return s16_launch_as<DT, 8, 8, 3, false, DUAL>(p, e, grid, s);
    if (p.m <= 16) return s16_launch_as<DT, 16, 8, 3, false, DUAL>(p, e, grid, s);
    return s16_launch_as<DT, 32, 8, 2, false, DUAL>(p, e, grid, s);
}
// up to 4 rows, normalised on the way in
template <int DT, bool DUAL = false, class Epi>
int s16_launch_norm(const Stream16P& p, const Epi& e, hipStream_t s) {
    const int tiles = DUAL ? (p.n + 7) / 8 : (p.n + 15) / 16, grid = tiles < 256 ? tiles : 256;
    return s16_launch_as<DT, 4, 8, 3, true, DUAL>(p, e, grid, s);
}
