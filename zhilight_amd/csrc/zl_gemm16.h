// zl_gemm16.h -- the large NT product (prompt portions): y (m, n) = x (m, k) . w (n, k)^T on the matrix cores, 16-bit operands with fp32
// accumulation in k order, or int8 operands with exact int32 sums.  One kernel for dense_gemm.hip (fp16 / bf16 models), int8_ops.hip (INT8
// linears) and csrc_seq/seq_gemm.hip (the ragged-step engine).
//
// What bounds it: the matrix pipe when an operand tile is large, the latency of its slices when it is small.  Both operands go global -> LDS by
// LDS-DMA (no registers, no ds_write) into a ring of ST slices of 64 k (int8: 128; 128 bytes of a row either way); a slice is requested ST - 1 slices ahead, there is one barrier per
// slice, and it sits between the slice's two 32-k halves, so that the second half's MFMAs cover the first LDS reads of the next slice.
// Measured (bf16, fp32 out, weights cold in HBM): 4096^3 1.06 PFLOP/s; 1024 x 28672 x 4096 1.09; 777 x 6912 x 2304 0.65; 777 x 2304 x 5760
// 0.57; the kernels it took the place of (64-row tiles with weights straight into registers; 32-k slices through registers and two barriers)
// ran these at 0.2 .. 0.75.  int8: 1000 x 28672 x
// 4096 with its gated epilogue 142 us, 1.65 POP/s (two products of 216 us and a 28 us pass before).
#pragma once
#include "zl_common.h"

typedef _Float16 g16_h8 __attribute__((ext_vector_type(8)));
typedef __bf16 g16_b8 __attribute__((ext_vector_type(8)));
typedef float g16_f4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* g16_lds;

constexpr int G16_I8 = 64;                                     // operand format beside ZL_F16 / ZL_BF16

struct Gemm16P {
    const void* x; const void* w;
    int64_t ldx, ldw;                                          // elements
    int m, n, k;                                               // k in whole slices
    int gx, gy;                                                // tiles along n and m
    int k_part;                                                // workgroups y = 1, 2, ... take the following k_part numbers of k (whole slices)
    // DUAL: blocks of 16 columns come in turn from w and w2 (gate and up rows of the same outputs); each has w_rows rows, n counts both
    const void* w2;
    int w_rows;
};

typedef int g16_i4 __attribute__((ext_vector_type(4)));
template <int DT> struct G16Acc { typedef g16_f4 type; };
template <> struct G16Acc<G16_I8> { typedef g16_i4 type; };

__device__ __forceinline__ g16_i4 g16_mfma_i8(uint4 a, uint4 b, g16_i4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(g16_i4, a), __builtin_bit_cast(g16_i4, b), c, 0, 0, 0);
}
template <int DT>
__device__ __forceinline__ g16_f4 g16_mfma(uint4 a, uint4 b, g16_f4 c) {
    if constexpr (DT == ZL_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(g16_h8, a), __builtin_bit_cast(g16_h8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(g16_b8, a), __builtin_bit_cast(g16_b8, b), c, 0, 0, 0);
}

// one LDS-DMA load: 64 lanes x 16 bytes from a descriptor + lane offset + scalar offset to 1 KiB at LDS byte address `lds`.  As asm without
// outputs: the compiler knows nothing of it, so it neither waits for it nor keeps other LDS reads from running beside it -- the kernel's
// own waits (g16_wait) order it.
__device__ __forceinline__ void g16_dma(u32x4 rsrc, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %0, %2 offen lds" ::"s"(rsrc), "v"(voff), "s"(soff), "s"(lds) : "m0");
}
template <int N>
__device__ __forceinline__ void g16_wait() {                   // at most N of this wave's loads outstanding, its LDS reads done
    static_assert(N >= 0 && N < 64, "vmcnt has 6 bits");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ u32x4 g16_rsrc(const void* base) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return (u32x4){(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)), 0xffffffffu, 0x00020000u};
}

// BM x BN outputs per workgroup of WM x WN waves; slices of 64 numbers of k in a ring of ST LDS buffers.  The weights are the MFMAs' A operand:
// a lane ends up with four neighbouring columns of one row, which leave in one store.
template <int DT, int BM, int BN, int WM, int WN, int ST, bool DUAL, class Epi>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_gemm16(const Gemm16P p, const Epi epi) {
    constexpr int T = 64 * WM * WN, MI = BM / WM / 16, NI = BN / WN / 16, LX = BM * 8 / T, LW = BN * 8 / T;
    constexpr uint32_t kBuf = (BM + BN) * 128;
    constexpr int ES = DT == G16_I8 ? 1 : 2;                   // bytes of an operand element
    typedef typename G16Acc<DT>::type acc_t;
    static_assert(!DUAL || NI % 2 == 0, "a wave's column blocks pair up");
    extern __shared__ __attribute__((aligned(1024))) unsigned char g16_smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nrow = lane & 15, kq = lane >> 4;
    const int wm = wave % WM, wn = wave / WM;
    // consecutive workgroups go to the 8 XCDs in turn: an XCD gets a contiguous run of tiles, column by column of 8 row tiles
    const int total = p.gx * p.gy, q = total >> 3, rem = total & 7, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int id = xcd * q + min(xcd, rem) + loc;
    const int band = 8 * p.gx, b = id / band, in = id - b * band, hgt = min(8, p.gy - 8 * b);
    const int m0 = (8 * b + in % hgt) * BM, n0 = (in / hgt) * BN;
    const int k0 = blockIdx.y * p.k_part, nt = min(p.k - k0, p.k_part) / (128 / ES);
    const int w0 = DUAL ? n0 >> 1 : n0, wlast = (DUAL ? p.w_rows : p.n) - 1 - w0;                 // the tile's first weight row; rows behind it
    const void* wsrc = DUAL && ((wave >> 1) & 1) ? p.w2 : p.w;                                     // (a wave's loads lie in blocks of one parity)
    const u32x4 rx = g16_rsrc((const char*)p.x + ((size_t)m0 * p.ldx + k0) * ES), rw = g16_rsrc((const char*)wsrc + ((size_t)w0 * p.ldw + k0) * ES);
    // a wave's load fills 8 LDS rows of 64 k: lane l -> row l / 8, 16-byte unit l % 8, which holds unit (l % 8) ^ (row / 2 % 8) of the
    // matrix row: a fragment's 16 rows x 16 bytes then lie in 64 different banks.  Rows past the edge read the last row (never stored).
    uint32_t xo[LX], wo[LW];
    const int lr = wave * 8 + (lane >> 3), lu = lane & 7;
#pragma unroll
    for (int i = 0; i < LX; ++i) {
        const int r = lr + i * (T / 8);
        xo[i] = (uint32_t)(min(r, p.m - 1 - m0) * (int)p.ldx * ES + ((lu ^ ((r >> 1) & 7)) * 16));
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int r = lr + i * (T / 8);
        const int src = DUAL ? (r >> 5) * 16 + (r & 15) : r;
        wo[i] = (uint32_t)(min(src, wlast) * (int)p.ldw * ES + ((lu ^ ((r >> 1) & 7)) * 16));
    }
    const uint32_t lds0 = (uint32_t)(size_t)(g16_lds)g16_smem + wave * 1024;
    auto dma = [&](uint32_t buf, int t) {                      // slice t into the buffer at byte buf
#pragma unroll
        for (int i = 0; i < LX; ++i) g16_dma(rx, xo[i], (uint32_t)t * 128, lds0 + buf + i * (T * 16));
#pragma unroll
        for (int i = 0; i < LW; ++i) g16_dma(rw, wo[i], (uint32_t)t * 128, lds0 + buf + BM * 128 + i * (T * 16));
    };
    const int sw = (nrow >> 1) & 7;
    const uint32_t fx = (wm * MI * 16 + nrow) * 128, fw = (BM + wn * NI * 16 + nrow) * 128, u0 = (kq ^ sw) * 16, u1 = u0 ^ 64;
    acc_t acc[NI][MI];
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[j][i] = (acc_t){0, 0, 0, 0};
    uint4 fa[2][MI], fb[2][NI];
    auto rd = [&](int set, uint32_t at) {
#pragma unroll
        for (int j = 0; j < NI; ++j) fb[set][j] = *reinterpret_cast<const uint4*>(g16_smem + fw + at + j * 2048);
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[set][i] = *reinterpret_cast<const uint4*>(g16_smem + fx + at + i * 2048);
    };
    auto mul = [&](int set) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                if constexpr (DT == G16_I8) acc[j][i] = g16_mfma_i8(fb[set][j], fa[set][i], acc[j][i]);
                else acc[j][i] = g16_mfma<DT>(fb[set][j], fa[set][i], acc[j][i]);
            }
    };
#pragma unroll
    for (int u = 0; u < ST; ++u)
        if (u < nt) dma(u * kBuf, u);
    if (nt >= ST) g16_wait<(ST - 1) * (LX + LW)>();
    else g16_wait<0>();
    __builtin_amdgcn_s_barrier();
    rd(0, u0);
    uint32_t cur = 0;
    for (int t = 0; t < nt; ++t) {
        const uint32_t nxt = cur + kBuf == ST * kBuf ? 0 : cur + kBuf;
        rd(1, cur + u1);
        mul(0);
        // slice t + 1 has landed, every wave holds the rest of slice t in registers: its buffer takes slice t + ST
        if (t + ST <= nt) g16_wait<(ST - 2) * (LX + LW)>();
        else g16_wait<0>();
        __builtin_amdgcn_s_barrier();
        if (t + ST < nt) dma(cur, t + ST);
        rd(0, nxt + u0);                                       // (past the last slice: old numbers, never multiplied)
        mul(1);
        cur = nxt;
    }
    // lane: row nrow of a 16-row block, columns 4 kq .. + 3 of a 16-column block
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int row = m0 + wm * MI * 16 + i * 16 + nrow;
        if (row < p.m) epi.template row<NI>(row, n0 + wn * NI * 16 + 4 * kq, p.n, [&](int j) { return acc[j][i]; });
    }
}

// The tile: the shape whose busiest CU is done first.  `cost` is the measured time of one 64-k slice of one tile (hundredths of a us, cold
// weights) with the CU as full as the shape's LDS allows, `alone` with one such workgroup per CU; a launch takes ceil(tiles / CUs) of them.  The big
// tiles win where they come to whole rounds (1024 x 28672: 220 us against 293 with 128 x 128), the deep rings of small tiles where there
// are fewer tiles than CUs (777 x 2304 x 5760: 36 us with 128 x 64, 77 with 128 x 128 in two slices, 122 with 256 x 256).  160- and 192-row tiles
// are for heights that the powers of two miss (777 x 11520 x 2304: 48 us with 160 x 128, 70 with 256 x 256; 565 x 21504 x 4096: 97 with 192 x 128,
// 126 with 256 x 256; 565 x 4096 x 4096: 32 with 160 x 64, 39 with 128 x 128).  The 16-bit tiles of 128 columns that come two to a CU run 4 waves of 64 (80) x 64, a third
// less LDS traffic per product than 8 of 64 x 32 (4096^3 in 128 x 128: 149 -> 138 us); a workgroup alone on its CU is better off with 8 (2048 x 2048 x
// 2048 .. 8192 between other kernels: 52 us against 57).
struct Gemm16Tile { int bm, bn, alone, cost; };
static const Gemm16Tile kGemm16Tiles[9] = {{256, 256, 185, 172}, {256, 128, 100, 100}, {128, 128, 80, 54}, {128, 128, 60, 61}, {128, 64, 42, 40}, {64, 64, 28, 26},
                                           {160, 128, 78, 62}, {192, 128, 104, 74}, {160, 64, 50, 50}};

static inline int g16_pick(int64_t m, int64_t n) {
    int best = 0;
    int64_t least = INT64_MAX;
    for (int i = 0; i < 9; ++i) {
        const Gemm16Tile& t = kGemm16Tiles[i];
        const int64_t tiles = ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn), r = (tiles + 255) / 256;
        const int64_t c = r == 1 ? t.alone : r * t.cost;
        if (c < least) { least = c; best = i; }
    }
    return best;
}

// whether the kernel takes a 16-bit product: whole slices, 16-byte rows, tile offsets that fit 32 bits
static inline bool g16_takes(const void* x, int64_t ldx, const void* w, int64_t ldw, int64_t k) {
    return k % 64 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0 && ldx <= (1 << 22) && ldw <= (1 << 22);
}

template <int DT, int BM, int BN, int WM, int WN, int ST, bool DUAL, class Epi>
int g16_launch_tile(Gemm16P p, const Epi& e, hipStream_t s) {
    const int parts = (p.k + p.k_part - 1) / p.k_part;
    p.gx = (p.n + BN - 1) / BN;
    p.gy = (p.m + BM - 1) / BM;
    if ((int64_t)p.gx * p.gy > INT32_MAX) return ZL_ELIMIT;
    constexpr int lds = (BM + BN) * 128 * ST;
    if (lds > 64 * 1024 &&                                     // (every launch: the attribute is per device, one process may drive several)
        hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm16<DT, BM, BN, WM, WN, ST, DUAL, Epi>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return ZL_ELIMIT;
    hipLaunchKernelGGL((k_gemm16<DT, BM, BN, WM, WN, ST, DUAL, Epi>), dim3((unsigned)(p.gx * p.gy), (unsigned)parts), dim3(64 * WM * WN), lds, s, p, e);
    return zl_launch_status();
}

template <int DT, bool DUAL = false, class Epi>
int g16_launch(const Gemm16P& p, const Epi& e, hipStream_t s) {
    constexpr int W128 = DT == G16_I8 ? 4 : 2;                 // (two workgroups per CU; int8's scale-backs are long, more waves share them)
    switch (p.k_part < p.k ? 5 : g16_pick(p.m, p.n)) {         // (a divided k: the caller counts 64 x 64 tiles)
        case 0: return g16_launch_tile<DT, 256, 256, 2, 4, 2, DUAL>(p, e, s);
        case 1: return g16_launch_tile<DT, 256, 128, 4, 2, 3, DUAL>(p, e, s);
        case 2: return g16_launch_tile<DT, 128, 128, 2, W128, 2, DUAL>(p, e, s);
        case 3: return g16_launch_tile<DT, 128, 128, 2, 4, 3, DUAL>(p, e, s);
        case 4: return g16_launch_tile<DT, 128, 64, 4, 2, 4, DUAL>(p, e, s);
        case 6: return g16_launch_tile<DT, 160, 128, 2, 2, 2, DUAL>(p, e, s);
        case 7: return g16_launch_tile<DT, 192, 128, 4, 2, 2, DUAL>(p, e, s);
        case 8: return g16_launch_tile<DT, 160, 64, 2, 2, 3, DUAL>(p, e, s);
        default: return g16_launch_tile<DT, 64, 64, 2, 2, 4, DUAL>(p, e, s);
    }
}
