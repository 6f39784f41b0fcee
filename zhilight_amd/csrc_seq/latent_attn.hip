// latent_attn.hip -- attention over a PAGED cache of normed low-rank latents, for every token of a ragged step.
//
// Beside csrc/mla_attn.hip (DeepSeek's geometry: 512 + 64 rotated columns, 16-bit, decode rows only, no sink): any rank / head sizes, a
// learned per-head sink in the softmax denominator, a per-head sigmoid output gate, causal portions of prompts at any offset, an optional
// sliding window, and a 32-bit mode.  Only the latent is cached; for single tokens keys and values are never materialised:
//     score_j = (W_uk,h^T q_h) . c_j * scale          o_h = W_uv,h . (sum_j w_j c_j)
// A rotated key part shared by all heads rides in the same cached row behind the latent: the row is [c | k_rot], the up-projections get
// identity columns for it (W_uk) or zeros (W_uv) on the host, and every kernel below sees one longer "latent".
// k_latent_store        RMS norm (plain weight) of the down-projection -> the token's cache row; the rotated key part behind it and the
//                       queries' rotated parts (in place), turned by the token's position
// k_latent_absorb       the query folded through W_uk (and the scale), once per token and head, 8 tokens to a workgroup
// k_latent_split        single tokens (and, in 32-bit serving, every token): the keys split over workgroups, fp32 VALU
// k_latent_decode_mfma  the same split pass for bf16 on the matrix cores
// k_latent_combine_v    merges the splits with the sink (it counts once, unscaled, with no value), applies W_uv and the gate, 8 tokens to a
//                       workgroup; k_latent_combine keeps ranks that are no whole 8s and very many splits
// k_latent_fa           portions of prompts in bf16 on the matrix cores, over keys and values up-projected for the step
#include <type_traits>
#include "seq_common.h"

namespace {

// rot > 0: the down-projection has rot more columns behind the latent, one rotated key part for all heads: pair (2i, 2i + 1) (interleaved)
// or (i, i + rot / 2) is turned by pos * freq[i] and stored behind the normed latent (cache rows hold rank + rot numbers); the last rot
// coordinates of every query head (q_col0, heads x qdim) are turned the same way in place.  A thread owns a whole pair.
template <int DT>
__global__ __launch_bounds__(256) void k_latent_store(float* __restrict__ proj, int64_t ld, int col0, const float* __restrict__ weight,
                                                      float eps, int rank, int rot, const float* __restrict__ freq, int interleaved, int q_col0,
                                                      int heads, int qdim, const zls_batch_t b, void* __restrict__ cache, float rot_gain) {
    __shared__ float red[16];
    const int t = blockIdx.x;
    const int sq = b.tok_seq[t];
    const int pos = b.seq_pos0[sq] + (t - b.seq_start[sq]);
    const int page = b.page_table[(size_t)sq * b.max_pages + pos / b.page_size];
    const size_t dst = ((size_t)page * b.page_size + pos % b.page_size) * (rank + rot);
    float* row = proj + (size_t)t * ld;
    const float* u = row + col0;
    float ss = 0.f;
    for (int i = threadIdx.x; i < rank; i += 256) ss = fmaf(u[i], u[i], ss);
    ss = zl_block_sum(ss, red);
    const float f = 1.0f / sqrtf(ss / (float)rank + eps);
    for (int i = threadIdx.x; i < rank; i += 256) SeqT<DT>::st(cache, dst + i, u[i] * f * weight[i]);
    const int half = rot >> 1;
    for (int w = threadIdx.x; w < (heads + 1) * half; w += 256) {          // vector 0: the key part; 1 ..: the heads' query parts
        const int vec = w / half, i = w % half;
        const int a = interleaved ? 2 * i : i, c = interleaved ? 2 * i + 1 : i + half;
        float sn, cs;
        seq_sincos((float)pos * freq[i], &sn, &cs);
        sn *= rot_gain; cs *= rot_gain;                                    // (rescaled frequencies come with a gain on cos and sin)
        float* src = vec == 0 ? row + col0 + rank : row + q_col0 + (size_t)(vec - 1) * qdim + (qdim - rot);
        const float x = src[a], y = src[c];
        const float xr = x * cs - y * sn, yr = y * cs + x * sn;
        if (vec == 0) { SeqT<DT>::st(cache, dst + rank + a, xr); SeqT<DT>::st(cache, dst + rank + c, yr); }
        else { src[a] = xr; src[c] = yr; }
    }
}

struct AttnP {
    const float* q; const float* gate; const void* w_uk; const void* w_uv; const float* sink; const void* cache; void* out;
    int64_t ldq, ldg;
    int q_col0, g_col0, heads, dim, vdim, rank, single_only, vec;
    int pairs;                                     // W_uk's rows are even and aligned: two columns per load
    float scale;
    int window;                                    // > 0: a token at position p sees the keys p - window < j <= p only
};

// the workspace: the splits' sums (n_tok, heads, n_splits, rank), the folded queries (n_tok, heads, rank), the splits' (maximum, denominator)
struct LatWs {
    float* acc; float2* ml;
    __device__ __forceinline__ LatWs(float* ws, int n_tok, const AttnP& p, int n_splits, int t, int h, int split) {
        const size_t at = ((size_t)t * p.heads + h) * n_splits + split;
        acc = ws + at * p.rank;
        ml = reinterpret_cast<float2*>(ws + (size_t)n_tok * p.heads * (n_splits + 1) * p.rank) + at;
    }
    // (4-byte aligned only when rank is odd)
    __device__ __forceinline__ void store_ml(float m, float l) const { float* f = reinterpret_cast<float*>(ml); f[0] = m; f[1] = l; }
};

// two consecutive numbers as they lie in memory: what is converted only after every load is on its way
template <int DT> struct Raw2;
template <> struct Raw2<ZL_BF16> {
    uint32_t u;
    __device__ __forceinline__ void load(const void* p, size_t i) { u = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint16_t*>(p) + i); }
    __device__ __forceinline__ void load1(const void* p, size_t i, size_t k) {
        const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
        u = h[i] | (uint32_t)h[k] << 16;
    }
    __device__ __forceinline__ float2 get() const { return make_float2(__builtin_bit_cast(float, u << 16), __builtin_bit_cast(float, u & 0xffff0000u)); }
};
template <> struct Raw2<ZL_F32> {
    float2 v;
    __device__ __forceinline__ void load(const void* p, size_t i) { v = *reinterpret_cast<const float2*>(reinterpret_cast<const float*>(p) + i); }
    __device__ __forceinline__ void load1(const void* p, size_t i, size_t k) { const float* f = reinterpret_cast<const float*>(p); v = make_float2(f[i], f[k]); }
    __device__ __forceinline__ float2 get() const { return v; }
};

constexpr int kLatTok = 8;                         // tokens that share a workgroup's weights

// which of the kLatTok tokens from t0 are this kernel's (portions of several tokens go to the prompt kernel); workgroup-uniform
__device__ __forceinline__ uint32_t lat_live(const AttnP& p, const zls_batch_t& b, int t0) {
    const int t = t0 + (threadIdx.x & (kLatTok - 1));           // (a lane each: one chain of loads instead of eight)
    bool live = t < b.n_tok;
    if (live && p.single_only) {
        const int sq = b.tok_seq[t];
        live = b.seq_start[sq + 1] - b.seq_start[sq] <= 1;
    }
    return (uint32_t)__ballot(live) & ((1u << kLatTok) - 1);
}

// q'_h = scale * W_uk,h^T q_h, once per (token, head): workgroup = 64 latent columns (2 per thread) of one head for 8 tokens, its eight half-waves
// take every eighth query dimension, 16 rows' loads in flight each; the partial sums meet in LDS.  qa (n_tok, heads, rank) fp32.  What bounds it is the
// latency of W_uk's loads; with a workgroup per token the matrix also came from L2 once per token (8 tokens x 32 heads x 128 x 512: 18 -> 5.8 us)
template <int DT>
__global__ __launch_bounds__(256) void k_latent_absorb(const AttnP p, const zls_batch_t b, float* __restrict__ qa) {
    __shared__ __attribute__((aligned(16))) float qs[128][kLatTok];
    __shared__ float part[8][kLatTok][64];
    const int t0 = blockIdx.x * kLatTok, h = blockIdx.y, cp = threadIdx.x & 31, grp = threadIdx.x >> 5;
    const uint32_t live = lat_live(p, b, t0);
    if (!live) return;
    const int c = blockIdx.z * 64 + 2 * cp, c0 = min(c, p.rank - 1), c1 = min(c + 1, p.rank - 1);      // (columns past the rank: the last one, never stored)
    float acc[kLatTok][2];
#pragma unroll
    for (int i = 0; i < kLatTok; ++i) acc[i][0] = acc[i][1] = 0.f;
    for (int d0 = 0; d0 < p.dim; d0 += 128) {
        Raw2<DT> w[16];
        if (p.pairs) {
#pragma unroll
            for (int u = 0; u < 16; ++u) w[u].load(p.w_uk, ((size_t)h * p.dim + min(d0 + grp + 8 * u, p.dim - 1)) * p.rank + (c0 & ~1));
        } else {
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const size_t row = ((size_t)h * p.dim + min(d0 + grp + 8 * u, p.dim - 1)) * p.rank;
                w[u].load1(p.w_uk, row + c0, row + c1);
            }
        }
        if (d0) __syncthreads();
        for (int i = threadIdx.x; i < 128 * kLatTok; i += 256) {
            const int d = i & 127, tk = i >> 7;
            qs[d][tk] = (live >> tk & 1) && d0 + d < p.dim ? p.q[(size_t)(t0 + tk) * p.ldq + p.q_col0 + (size_t)h * p.dim + d0 + d] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const float2 wv = w[u].get();
#pragma unroll
            for (int i = 0; i < kLatTok; ++i) {
                const float qv = qs[grp + 8 * u][i];               // (0 past the last dimension)
                acc[i][0] = fmaf(qv, wv.x, acc[i][0]);
                acc[i][1] = fmaf(qv, wv.y, acc[i][1]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < kLatTok; ++i) { part[grp][i][2 * cp] = acc[i][0]; part[grp][i][2 * cp + 1] = acc[i][1]; }
    __syncthreads();
    for (int i = threadIdx.x; i < kLatTok * 64; i += 256) {
        const int tk = i >> 6, cc = i & 63, r = blockIdx.z * 64 + cc;
        if (!(live >> tk & 1) || r >= p.rank) continue;
        float a = 0.f;
#pragma unroll
        for (int g = 0; g < 8; ++g) a += part[g][tk][cc];
        qa[((size_t)(t0 + tk) * p.heads + h) * p.rank + r] = a * p.scale;
    }
}

// Split over keys: workgroup = (token, group of 4 heads, split), a wave per head.  A tile of 16 cached rows is staged once in LDS as fp32
// (row stride rank + 4) and shared by the four heads.  Scores: lane = (key, quarter of the latent columns), two butterflies; weighted sum:
// a lane owns the latent columns lane, lane + 64, ... (RPL of them, in registers).  Every split leaves (max, denominator, sums) in the
// workspace; the combine merges them WITH the sink (m = max(sink, m_i), l = e^(sink - m) + sum l_i e^(m_i - m)), applies W_uv and the
// gate.  LDS: ct[16][rank + 4] | qk[4][rank]
template <int DT, int RPL>
__global__ __launch_bounds__(256) void k_latent_split(const AttnP p, const zls_batch_t b, const float* __restrict__ qa, float* __restrict__ ws,
                                                      int n_splits) {
    extern __shared__ float lds[];
    const int RP = p.rank + 4;                     // rows 16-byte aligned; 4 banks between neighbouring keys
    float* ct = lds;
    float* qk = lds + 16 * RP + (threadIdx.x >> 6) * p.rank;
    const int t = blockIdx.x, split = blockIdx.z, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.y * 4 + wave;
    const bool hvalid = h < p.heads;
    const int sq = b.tok_seq[t];
    if (p.single_only && b.seq_start[sq + 1] - b.seq_start[sq] > 1) return;      // portions go to the prompt kernel (workgroup-uniform)
    const int pos = b.seq_pos0[sq] + (t - b.seq_start[sq]);
    const int key_lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;
    const int nkeys = pos + 1 - key_lo;
    const int chunk = ((nkeys + n_splits - 1) / n_splits + 15) & ~15;
    const int k0 = key_lo + split * chunk, k1 = min(pos + 1, k0 + chunk);
    const int32_t* pages = b.page_table + (size_t)sq * b.max_pages;
    if (hvalid)
        for (int r = lane; r < p.rank; r += 64) qk[r] = qa[((size_t)t * p.heads + h) * p.rank + r];
    float acc[RPL];
#pragma unroll
    for (int i = 0; i < RPL; ++i) acc[i] = 0.f;
    float m = -INFINITY, l = 0.f;
    const int key = lane & 15, quarter = lane >> 4;
    // tile fill: 16 threads per key; with aligned rows the NEXT tile's 16-byte loads are issued into registers before the current tile is
    // worked on and written to LDS after it (8 slots of 16 bytes cover rank <= 1024)
    constexpr int V = DT == ZL_BF16 ? 8 : 4;
    const int fk = threadIdx.x >> 4, fc = threadIdx.x & 15;
    uint4 raw[8];
    auto row_base = [&](int j) { return ((size_t)pages[j / b.page_size] * b.page_size + j % b.page_size) * p.rank; };
    auto prefetch = [&](int j0) {
        const int j = j0 + fk;
        if (!p.vec || j >= k1) return;
        const size_t base = row_base(j);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int r = (fc + 16 * u) * V;
            if (r < p.rank) {
                if constexpr (DT == ZL_BF16) raw[u] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.cache) + base + r);
                else raw[u] = *reinterpret_cast<const uint4*>(reinterpret_cast<const float*>(p.cache) + base + r);
            }
        }
    };
    auto publish = [&](int j0) {
        const int j = j0 + fk;
        float* dst = ct + fk * RP;
        if (j >= k1) {
            for (int r = fc; r < p.rank; r += 16) dst[r] = 0.f;
        } else if (p.vec) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int r = (fc + 16 * u) * V;
                if (r < p.rank) {
                    if constexpr (DT == ZL_BF16) {
                        const uint32_t w4[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
                        float v[8];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            v[2 * e] = __builtin_bit_cast(float, w4[e] << 16);
                            v[2 * e + 1] = __builtin_bit_cast(float, w4[e] & 0xffff0000u);
                        }
                        *reinterpret_cast<float4*>(dst + r) = make_float4(v[0], v[1], v[2], v[3]);
                        *reinterpret_cast<float4*>(dst + r + 4) = make_float4(v[4], v[5], v[6], v[7]);
                    } else {
                        *reinterpret_cast<uint4*>(dst + r) = raw[u];
                    }
                }
            }
        } else {
            const size_t base = row_base(j);
            for (int r = fc; r < p.rank; r += 16) dst[r] = SeqT<DT>::ld(p.cache, base + r);
        }
    };
    prefetch(k0);
    for (int j0 = k0; j0 < k1; j0 += 16) {
        __syncthreads();
        publish(j0);
        __syncthreads();
        if (j0 + 16 < k1) prefetch(j0 + 16);
        if (!hvalid) continue;
        float sc = 0.f;
        for (int r = quarter; r < p.rank; r += 4) sc = fmaf(qk[r], ct[key * RP + r], sc);    // (key, quarter): 32 banks, two lanes each
        sc += __shfl_xor(sc, 16, 64);
        sc += __shfl_xor(sc, 32, 64);
        const bool valid = j0 + key < k1;
        sc = valid ? sc : -INFINITY;
        float mx = sc;
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        const float mnew = fmaxf(m, mx);                               // finite: key j0 is valid
        const float corr = expf(m - mnew);                             // m = -inf at the first tile: 0
        const float pj = valid ? expf(sc - mnew) : 0.f;
        float ps = pj;
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) ps += __shfl_xor(ps, off, 64);
        l = l * corr + ps;
        m = mnew;
        float pk[16];
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) pk[kk] = __shfl(pj, kk, 64);
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
            const int r = lane + 64 * i;
            if (r < p.rank) {
                float a = acc[i] * corr;
#pragma unroll
                for (int kk = 0; kk < 16; ++kk) a = fmaf(pk[kk], ct[kk * RP + r], a);
                acc[i] = a;
            }
        }
    }
    if (!hvalid) return;
    const LatWs o(ws, b.n_tok, p, n_splits, t, h, split);
    if (lane == 0) o.store_ml(m, l);
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
        const int r = lane + 64 * i;
        if (r < p.rank) o.acc[r] = acc[i];
    }
}

// LDS: acc[rank] | wgt[n_splits]
template <int DT>
__global__ __launch_bounds__(256) void k_latent_combine(const AttnP p, const zls_batch_t b, float* __restrict__ ws, int n_splits) {
    extern __shared__ float lds[];
    __shared__ float red[16];
    float* wgt = lds + p.rank;
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sq = b.tok_seq[t];
    if (p.single_only && b.seq_start[sq + 1] - b.seq_start[sq] > 1) return;
    const LatWs part(ws, b.n_tok, p, n_splits, t, h, 0);
    float mloc = p.sink ? p.sink[h] : -INFINITY;                       // threads along the splits: loads in parallel
    for (int s2 = threadIdx.x; s2 < n_splits; s2 += 256) mloc = fmaxf(mloc, reinterpret_cast<const float*>(part.ml)[2 * s2]);
    const float m = zl_block_max(mloc, red);
    float lloc = 0.f;
    for (int s2 = threadIdx.x; s2 < n_splits; s2 += 256) {
        const float ms = reinterpret_cast<const float*>(part.ml)[2 * s2];
        const float w = ms == -INFINITY ? 0.f : expf(ms - m);
        wgt[s2] = w;
        lloc = fmaf(reinterpret_cast<const float*>(part.ml)[2 * s2 + 1], w, lloc);
    }
    const float l = zl_block_sum(lloc, red) + (p.sink ? expf(p.sink[h] - m) : 0.f);      // (its barriers also publish wgt)
    for (int r = threadIdx.x; r < p.rank; r += 256) {
        float a = 0.f;
#pragma unroll 8
        for (int s2 = 0; s2 < n_splits; ++s2) a = fmaf(part.acc[(size_t)s2 * p.rank + r], wgt[s2], a);
        lds[r] = a;
    }
    __syncthreads();
    const float g = p.gate ? seq_sigmoid(p.gate[(size_t)t * p.ldg + p.g_col0 + h]) : 1.0f;
    const float inv = g / l;
    // a wave per output value, lanes along the latent (coalesced W_uv rows), four values per pass so that their loads are in flight
    // together; the workgroups of blockIdx.z share the head's outputs
    for (int d0 = (blockIdx.z * 4 + wave) * 4; d0 < p.vdim; d0 += gridDim.z * 16) {
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        for (int r = lane; r < p.rank; r += 64) {
            const float c = lds[r];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (d0 + u < p.vdim) a[u] = fmaf(SeqT<DT>::ld(p.w_uv, ((size_t)h * p.vdim + d0 + u) * p.rank + r), c, a[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float v = zl_wave_sum(a[u]);
            if (lane == 0 && d0 + u < p.vdim) SeqT<DT>::st(p.out, ((size_t)t * p.heads + h) * p.vdim + d0 + u, v * inv);
        }
    }
}

// the same for ranks of whole 8s: workgroup = 16 outputs of one head for 8 tokens, whose rows of W_uv are on the way while the splits are merged
// (a wave per token's weights, then 16-byte pieces of the sums); a wave = 4 outputs, a lane = 8 latent columns of each row for all the tokens, and
// the 32 sums of a wave are exchanged down to one per pair of lanes.  LDS: lat[8][rank] | wgt[8][n_splits] | inv[8]
// (8 tokens x 32 heads x 128 x 512: 31 -> 9.3 us: W_uv came from L2 once per token, and every wave sum took six exchanges)
template <int DT> struct Raw8;
template <> struct Raw8<ZL_BF16> {
    uint4 r;
    __device__ __forceinline__ void load(const void* p, size_t i) { r = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p) + i); }
    __device__ __forceinline__ void clear() { r = make_uint4(0, 0, 0, 0); }
    __device__ __forceinline__ void get(float* v) const {
        const uint32_t u[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[2 * e] = __builtin_bit_cast(float, u[e] << 16); v[2 * e + 1] = __builtin_bit_cast(float, u[e] & 0xffff0000u); }
    }
};
template <> struct Raw8<ZL_F32> {
    float4 a, c;
    __device__ __forceinline__ void load(const void* p, size_t i) { const float* f = reinterpret_cast<const float*>(p) + i; a = seq_ld4(f); c = seq_ld4(f + 4); }
    __device__ __forceinline__ void clear() { a = c = make_float4(0.f, 0.f, 0.f, 0.f); }
    __device__ __forceinline__ void get(float* v) const { v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = c.x; v[5] = c.y; v[6] = c.z; v[7] = c.w; }
};

// lanes whose numbers differ in bit 2 N swap halves of v[0 .. 2 N): half as many sums per lane, each over twice as many lanes
template <int N>
__device__ __forceinline__ void lat_fold(float* v, int lane) {
    const bool up = lane & (2 * N);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float keep = up ? v[i + N] : v[i], send = up ? v[i] : v[i + N];
        v[i] = keep + __shfl_xor(send, 2 * N, 64);
    }
}

template <int DT>
__global__ __launch_bounds__(256) void k_latent_combine_v(const AttnP p, const zls_batch_t b, float* __restrict__ ws, int n_splits) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* lat = lds;
    float* wgt = lds + kLatTok * p.rank;
    float* inv = wgt + kLatTok * n_splits;
    const int t0 = blockIdx.x * kLatTok, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t live = lat_live(p, b, t0);
    if (!live) return;
    const int d0 = blockIdx.z * 16 + wave * 4;
    Raw8<DT> w[4];
    auto rows = [&](int c) {                                               // 8 columns from c of the wave's 4 rows of W_uv
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (d0 + u < p.vdim && c < p.rank) w[u].load(p.w_uv, ((size_t)h * p.vdim + d0 + u) * p.rank + c);
            else w[u].clear();
        }
    };
    rows(8 * lane);
    const float sink = p.sink ? p.sink[h] : -INFINITY;
    for (int tk = wave; tk < kLatTok; tk += 4) {
        if (!(live >> tk & 1)) continue;
        const LatWs part(ws, b.n_tok, p, n_splits, t0 + tk, h, 0);
        float m = sink;
        for (int s = lane; s < n_splits; s += 64) m = fmaxf(m, part.ml[s].x);
        m = zl_wave_max(m);
        float l = 0.f;
        for (int s = lane; s < n_splits; s += 64) {
            const float2 v = part.ml[s];
            const float e = v.x == -INFINITY ? 0.f : expf(v.x - m);
            wgt[tk * n_splits + s] = e;
            l = fmaf(v.y, e, l);
        }
        l = zl_wave_sum(l) + (p.sink ? expf(sink - m) : 0.f);
        if (lane == 0) inv[tk] = (p.gate ? seq_sigmoid(p.gate[(size_t)(t0 + tk) * p.ldg + p.g_col0 + h]) : 1.0f) / l;
    }
    __syncthreads();
    const int quads = p.rank >> 2;
    const float* acc = LatWs(ws, b.n_tok, p, n_splits, t0, h, 0).acc;
    const size_t tok = (size_t)p.heads * n_splits * p.rank;                // (the next token's sums of this head)
    for (int i0 = threadIdx.x; i0 < kLatTok * quads; i0 += 1024) {         // 4 pieces of 4 splits in flight per thread
        float4 a[4];
        int tk[4], at[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = min(i0 + 256 * u, kLatTok * quads - 1);          // (past the end: the last piece once more)
            tk[u] = i / quads; at[u] = (i - tk[u] * quads) * 4;
            a[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        for (int s0 = 0; s0 < n_splits; s0 += 4) {
            float4 x[4][4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e)                                // (tokens of other kernels: the room is there, the numbers are not used)
                    x[u][e] = seq_ld4(acc + min(tk[u], b.n_tok - 1 - t0) * tok + (size_t)min(s0 + e, n_splits - 1) * p.rank + at[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (s0 + e >= n_splits || !(live >> tk[u] & 1)) continue;
                    const float f = wgt[tk[u] * n_splits + s0 + e];
                    a[u] = make_float4(fmaf(x[u][e].x, f, a[u].x), fmaf(x[u][e].y, f, a[u].y), fmaf(x[u][e].z, f, a[u].z), fmaf(x[u][e].w, f, a[u].w));
                }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<float4*>(lat + (size_t)tk[u] * p.rank + at[u]) = a[u];
    }
    __syncthreads();
    float v[4 * kLatTok];                                                  // [output][token]
#pragma unroll
    for (int i = 0; i < 4 * kLatTok; ++i) v[i] = 0.f;
    for (int c = 8 * lane; c < p.rank; c += 512) {
        if (c >= 512) rows(c);
        float wf[4][8];
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u].get(wf[u]);
#pragma unroll
        for (int tk = 0; tk < kLatTok; ++tk) {
            if (!(live >> tk & 1)) continue;
            const float4 x = seq_ld4(lat + (size_t)tk * p.rank + c), y = seq_ld4(lat + (size_t)tk * p.rank + c + 4);
            const float xv[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[u * kLatTok + tk] = fmaf(wf[u][e], xv[e], v[u * kLatTok + tk]);
        }
    }
    // lanes 2 i and 2 i + 1 end up with the whole sum of v[i]
    lat_fold<16>(v, lane); lat_fold<8>(v, lane); lat_fold<4>(v, lane); lat_fold<2>(v, lane); lat_fold<1>(v, lane);
    const float sum = v[0] + __shfl_xor(v[0], 1, 64);
    const int tk = (lane >> 1) & 7, d = d0 + (lane >> 4);
    if (!(lane & 1) && (live >> tk & 1) && d < p.vdim) SeqT<DT>::st(p.out, ((size_t)(t0 + tk) * p.heads + h) * p.vdim + d, sum * inv[tk]);
}

// ---- prompt portions on the matrix cores (bf16 serving) -----------------------------------------------------------------------------
// Keys and values of a portion's whole context are up-projected once per step into dense K (n_ctx, heads * dim) and V^T (heads * vdim,
// n_ctx) (zls_gemm_nt_gather over the cached rows; each sequence's rows start at a multiple of 64).  A workgroup = 64 queries of one
// sequence x one head, a wave = 16 of them.  Per 64-key tile (K and V^T staged in LDS, shared by the four waves):
//   S^T (16 keys x 16 queries) = K_tile . Q^T on v_mfma_f32_16x16x32_bf16 -- a lane then holds 4 consecutive keys of ONE query; two such
//   blocks side by side are a B operand of the same instruction with the 32 keys in a permuted order, and V^T is read in that order too,
//   so the weights never travel through LDS:
//   O^T (vdim x 16 queries) += V^T_tile . P^T, with P = hi + lo (two bf16 halves: the weights keep 16 bits of mantissa).
// Scores, running maximum / denominator (starting at the sink: m = sink, l = 1) and the output sums are fp32, per lane = per query; the
// exponentials are the hardware's exp2 of the fp32 argument times log2 e (the softmax VALU work, not the MFMAs, bounds this kernel).
typedef __bf16 fa_b8 __attribute__((ext_vector_type(8)));
typedef short fa_s4 __attribute__((ext_vector_type(4)));
typedef float fa_f4 __attribute__((ext_vector_type(4)));

// a non-negative fp32 weight as two bf16 halves, hi + lo = the weight to 2^-16 relative: hi is its upper 16 bits (truncation), lo the upper
// 16 bits of the exact remainder -- three instructions where two round-to-nearest conversions cost a dozen
__device__ __forceinline__ void fa_split(float pv, uint16_t& hb, uint16_t& lb) {
    const uint32_t u = __builtin_bit_cast(uint32_t, pv);
    hb = (uint16_t)(u >> 16);
    lb = (uint16_t)(__builtin_bit_cast(uint32_t, pv - __builtin_bit_cast(float, u & 0xffff0000u)) >> 16);
}

struct FaP {
    const float* q; const float* gate; const uint16_t* k; const uint16_t* vt; const float* sink; const int32_t* ctx_start; uint16_t* out;
    int64_t ldq, ldg, ldk, ldv;
    int q_col0, g_col0, heads, dim, vdim, tiles_per_seq;
    float scale;
    int window; const int32_t* ctx_pos0;           // window > 0: keys p - window < j <= p; ctx_pos0 (nullable: 0): the position of a sequence's
};                                                 // first up-projected row (a windowed step does not bring its whole context)

// NG groups of four waves take a workgroup's key tiles in turn, each with tiles of its own in LDS, and meet at the end: with as many query tiles as a
// prompt of a few thousand tokens has, the chip holds two workgroups per CU, and a tile's chain of LDS writes, barriers, products and exponentials
// is what the time goes into (2048 tokens x 16 heads of 128: 123 -> 67 us; masks only where a tile has keys that some query must not see).
// VEC: heads in whole 8s, rows aligned (others read K and the queries number by number).
template <int DK, int DV, int NG, bool VEC>
__global__ __launch_bounds__(256 * NG, NG == 2 && DK <= 4 ? 4 : 1) void k_latent_fa(const FaP p, const zls_batch_t b) {
    constexpr int KR = DK * 32 + 8, VR = 64 + 8, kGroup = 64 * KR + DV * 16 * VR;
    static_assert(NG == 1 || 4 * 64 * (DV * 4 + 2) * 4 <= NG * kGroup * 2, "the second group's sums fit");
    __shared__ __attribute__((aligned(16))) uint16_t smem[NG * kGroup];
    // The last query tiles see the most keys: they are dispatched first, so the launch does not end on its longest workgroups.  A launch that the
    // chip holds at once, two workgroups to a CU, is done when its busiest CU is: the second half goes the other way round, the shortest
    // beside the longest.  (Heads vary fastest: with 8 or 16 of them a head's keys and values stay in one XCD's cache.)
    const int total = gridDim.x, id = total <= 512 && blockIdx.x >= 256 ? 256 + total - 1 - (int)blockIdx.x : blockIdx.x, per = b.n_seq * p.heads;
    const int tile = p.tiles_per_seq - 1 - id / per, sq = id % per / p.heads, h = id % p.heads;
    const int first = b.seq_start[sq], count = b.seq_start[sq + 1] - first;
    const int cs = p.ctx_start[sq];
    if (cs < 0 || tile * 64 >= count) return;
    // positions below are counted from the sequence's first up-projected row (position c0): a key's index there is its row in K / V^T
    const int c0 = p.ctx_pos0 ? p.ctx_pos0[sq] : 0;
    const int pos0 = b.seq_pos0[sq] - c0;
    const int tid = threadIdx.x & 255, lane = tid & 63, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nrow = lane & 15, kq = lane >> 4;
    uint16_t* Ks = smem + grp * kGroup;
    uint16_t* Vs = Ks + 64 * KR;
    const int qi = tile * 64 + wave * 16 + nrow;
    const bool qvalid = qi < count;
    const int qpos = pos0 + qi;
    const int j_first = p.window > 0 ? max(0, pos0 + tile * 64 - p.window + 1) & ~63 : 0;     // the tile of the oldest key the first query sees
    const int wave_first = pos0 + tile * 64 + wave * 16;                           // the wave's first query
    const int wave_last = pos0 + min(count, tile * 64 + wave * 16 + 16) - 1;       // the last key any query of this wave sees
    const int block_last = pos0 + min(count, tile * 64 + 64) - 1;

    // K and V^T tiles: the NEXT tile's 16-byte loads are issued into registers before the current tile's MFMAs and written to LDS after them
    constexpr int KU = DK, VU = (DV + 1) / 2;                                      // 16-byte units per thread: 64 DK 4 / 256 and DV 16 8 / 256
    uint4 kreg[KU], vreg[VU];
    constexpr bool kRows = 256 % (DK * 4) == 0;                                    // a thread's units of K lie in one column
    using offs_t = typename std::conditional<VEC, uint32_t, size_t>::type;          // (VEC: strides below 2^24)
    const offs_t k_off = (offs_t)(tid / (DK * 4)) * (offs_t)p.ldk + (tid % (DK * 4)) * 8, v_off = (offs_t)(tid >> 3) * (offs_t)p.ldv + (tid & 7) * 8;
    auto fetch_tiles = [&](int j0) {
        const uint16_t* kb = p.k + (size_t)(cs + j0) * p.ldk + (size_t)h * p.dim;
        const uint16_t* vb = p.vt + (size_t)h * p.vdim * p.ldv + cs + j0;
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int idx = tid + 256 * u;
            const int key = idx / (DK * 4), d = (idx % (DK * 4)) * 8;
            uint4 v = make_uint4(0, 0, 0, 0);
            if constexpr (VEC && kRows) {
                if (d < p.dim) v = *reinterpret_cast<const uint4*>(kb + (size_t)(u * (256 / (DK * 4))) * p.ldk + k_off);
            } else if constexpr (VEC) {
                if (d < p.dim) v = *reinterpret_cast<const uint4*>(kb + (size_t)key * p.ldk + d);
            } else if (d < p.dim) {
                const uint16_t* src = kb + (size_t)key * p.ldk + d;
                uint16_t e[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) e[i] = d + i < p.dim ? src[i] : (uint16_t)0;
                v = make_uint4(e[0] | (uint32_t)e[1] << 16, e[2] | (uint32_t)e[3] << 16, e[4] | (uint32_t)e[5] << 16, e[6] | (uint32_t)e[7] << 16);
            }
            kreg[u] = v;
        }
#pragma unroll
        for (int u = 0; u < VU; ++u) {
            const int idx = tid + 256 * u;
            uint4 v = make_uint4(0, 0, 0, 0);
            if ((DV % 2 == 0 || idx < DV * 16 * 8) && (idx >> 3) < p.vdim) v = *reinterpret_cast<const uint4*>(vb + (size_t)(u * 32) * p.ldv + v_off);
            vreg[u] = v;
        }
    };
    uint16_t* const k_to = Ks + (tid / (DK * 4)) * KR + (tid % (DK * 4)) * 8;
    uint16_t* const v_to = Vs + (tid >> 3) * VR + (tid & 7) * 8;
    auto publish_tiles = [&]() {
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int idx = tid + 256 * u;
            *reinterpret_cast<uint4*>(kRows ? k_to + u * (256 / (DK * 4)) * KR : Ks + (idx / (DK * 4)) * KR + (idx % (DK * 4)) * 8) = kreg[u];
        }
#pragma unroll
        for (int u = 0; u < VU; ++u)
            if (DV % 2 == 0 || tid + 256 * u < DV * 16 * 8) *reinterpret_cast<uint4*>(v_to + u * 32 * VR) = vreg[u];
    };
    if (j_first + 64 * grp <= block_last) fetch_tiles(j_first + 64 * grp);
    uint4 qf[DK];
    {
        const float* qr = p.q + (size_t)(first + (qvalid ? qi : 0)) * p.ldq + p.q_col0 + (size_t)h * p.dim;
#pragma unroll
        for (int kk = 0; kk < DK; ++kk) {
            const int d = 32 * kk + 8 * kq;
            float v[8];
            if constexpr (VEC) {                                                         // (dim in whole 8s: a lane's 8 numbers are there or not)
                const float4 x = seq_ld4(qr + (d < p.dim ? d : 0)), y = seq_ld4(qr + (d < p.dim ? d + 4 : 4));
                v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w; v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = qr[d + i < p.dim ? d + i : 0];
            }
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = (qvalid && d + 2 * i < p.dim ? ZT<ZL_BF16>::from_f32(v[2 * i]) : 0) | (uint32_t)(qvalid && d + 2 * i + 1 < p.dim ? ZT<ZL_BF16>::from_f32(v[2 * i + 1]) : 0) << 16;
            qf[kk] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
    fa_f4 o[DV];
#pragma unroll
    for (int dt = 0; dt < DV; ++dt) o[dt] = (fa_f4){0.f, 0.f, 0.f, 0.f};
    // scores, maximum and sink in powers of two
    constexpr float kL2e = 1.4426950408889634f;
    const float scale2 = p.scale * kL2e;
    float m = p.sink && grp == 0 ? p.sink[h] * kL2e : -INFINITY, l = p.sink && grp == 0 ? 1.0f : 0.0f;

    for (int jb = j_first; jb <= block_last; jb += 64 * NG) {
        const int j0 = jb + 64 * grp;                                              // this group's tile
        __syncthreads();                                                           // the previous tiles are consumed
        if (j0 <= block_last) publish_tiles();
        __syncthreads();
        if (j0 + 64 * NG <= block_last) fetch_tiles(j0 + 64 * NG);                 // in flight during this tile's MFMAs
        if (j0 > wave_last) continue;                                              // wave-uniform; the barriers above stay in step
        const bool whole = j0 + 63 <= wave_first && (p.window <= 0 || wave_last - j0 < p.window);      // every query of the wave sees every key
        fa_f4 sc[4];
        float mx = -INFINITY;
#pragma unroll
        for (int c = 0; c < 4; ++c) sc[c] = (fa_f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < DK; ++kk)                                            // (four chains of products side by side)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint4 a = *reinterpret_cast<const uint4*>(Ks + (16 * c + nrow) * KR + 32 * kk + 8 * kq);
                sc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(fa_b8, a), __builtin_bit_cast(fa_b8, qf[kk]), sc[c], 0, 0, 0);
            }
        if (whole) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                sc[c] *= scale2;
                mx = fmaxf(fmaxf(fmaxf(mx, sc[c][0]), fmaxf(sc[c][1], sc[c][2])), sc[c][3]);
            }
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = j0 + 16 * c + 4 * kq + r;
                    const float v = (qvalid && key <= qpos && (p.window <= 0 || qpos - key < p.window)) ? sc[c][r] * scale2 : -INFINITY;
                    sc[c][r] = v;
                    mx = fmaxf(mx, v);
                }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mnew = fmaxf(m, mx), mref = mnew == -INFINITY ? 0.f : mnew;    // (nothing seen yet and no sink: all weights are 2^-inf = 0)
        const float corr = __builtin_amdgcn_exp2f(m - mref);
        float ps = 0.f;
        // the 32-key contraction of v_mfma_f32_16x16x32_bf16 may run over the keys in ANY order as long as both operands use the same one:
        // slot s of lane group kq stands for key 16 (s / 4) + 4 kq + s % 4 of the pair of 16-key blocks, which is how the scores lie here
        uint32_t hi[2][4], lo[2][4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                uint32_t u[2], rest[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {                                      // fa_split, two at a time
                    const float pv = __builtin_amdgcn_exp2f(sc[c][r + e] - mref);
                    ps += pv;
                    u[e] = __builtin_bit_cast(uint32_t, pv);
                    rest[e] = __builtin_bit_cast(uint32_t, pv - __builtin_bit_cast(float, u[e] & 0xffff0000u));
                }
                hi[c >> 1][2 * (c & 1) + (r >> 1)] = __builtin_amdgcn_perm(u[1], u[0], 0x07060302u);
                lo[c >> 1][2 * (c & 1) + (r >> 1)] = __builtin_amdgcn_perm(rest[1], rest[0], 0x07060302u);
            }
        }
        ps += __shfl_xor(ps, 16, 64);
        ps += __shfl_xor(ps, 32, 64);
        l = l * corr + ps;
        m = mnew;
#pragma unroll
        for (int dt = 0; dt < DV; ++dt) o[dt] *= corr;
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {                                           // (two outputs side by side)
            const fa_b8 ph = __builtin_bit_cast(fa_b8, make_uint4(hi[c2][0], hi[c2][1], hi[c2][2], hi[c2][3]));
            const fa_b8 pl = __builtin_bit_cast(fa_b8, make_uint4(lo[c2][0], lo[c2][1], lo[c2][2], lo[c2][3]));
#pragma unroll
            for (int d4 = 0; d4 < DV; d4 += 2) {
                fa_b8 a[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint16_t* vr = Vs + (16 * (d4 + e) + nrow) * VR + 32 * c2 + 4 * kq;
                    const uint2 a0 = *reinterpret_cast<const uint2*>(vr), a1 = *reinterpret_cast<const uint2*>(vr + 16);
                    a[e] = __builtin_bit_cast(fa_b8, make_uint4(a0.x, a0.y, a1.x, a1.y));
                }
#pragma unroll
                for (int e = 0; e < 2; ++e) o[d4 + e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[e], ph, o[d4 + e], 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 2; ++e) o[d4 + e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[e], pl, o[d4 + e], 0, 0, 0);
            }
        }
    }
    if constexpr (NG > 1) {                                                        // the second group hands its sums over, lane by lane
        float* meet = reinterpret_cast<float*>(smem) + (size_t)wave * 64 * (DV * 4 + 2) + lane;
        __syncthreads();
        if (grp) {
            meet[0] = m; meet[64] = l;
#pragma unroll
            for (int dt = 0; dt < DV; ++dt)
#pragma unroll
                for (int r = 0; r < 4; ++r) meet[64 * (2 + 4 * dt + r)] = o[dt][r];
        }
        __syncthreads();
        if (grp) return;
        const float m1 = meet[0], mm = fmaxf(m, m1), mref = mm == -INFINITY ? 0.f : mm;
        const float f0 = __builtin_amdgcn_exp2f(m - mref), f1 = __builtin_amdgcn_exp2f(m1 - mref);
        l = l * f0 + meet[64] * f1;
#pragma unroll
        for (int dt = 0; dt < DV; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[dt][r] = o[dt][r] * f0 + meet[64 * (2 + 4 * dt + r)] * f1;
    }
    if (!qvalid) return;
    const float g = p.gate ? seq_sigmoid(p.gate[(size_t)(first + qi) * p.ldg + p.g_col0 + h]) : 1.0f;
    const float inv = l > 0.f ? g / l : 0.f;
    uint16_t* orow = p.out + ((size_t)(first + qi) * p.heads + h) * p.vdim;
#pragma unroll
    for (int dt = 0; dt < DV; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 16 * dt + 4 * kq + r;
            if (d < p.vdim) orow[d] = ZT<ZL_BF16>::from_f32(o[dt][r] * inv);
        }
}

// ---- single tokens in bf16 on the matrix cores --------------------------------------------------------------------------------------
// Workgroup = one token x 16 heads x one split of the keys; its NW waves divide the latent's columns, RW blocks of 32 each.  Per 32 keys a wave's
// columns go from the pages straight into A operands (lane = key, 8 consecutive columns per 16-byte load, the next block's on the way), S^T
// (16 keys x 16 heads) += C . Q'^T with the folded queries as B operands held in registers; the waves' partial scores meet in LDS, every wave
// does the softmax per lane (= per head) as in the prompt kernel; the columns are parked in LDS by the wave that owns them and read back
// column-wise for O^T (latent x 16 heads) += C^T . P^T (the contraction runs over the 32 keys in the order the scores lie in the lanes; two bf16
// halves per weight).  What bounds it is this chain per block: one wave did all columns before, 32 waves in all for 8 tokens of 130 keys (35 -> 11 us).
// Leaves (max, denominator, sums) per split in the workspace as k_latent_split does.
template <int RW, int NW>                                                          // rank <= 32 RW NW
__global__ __launch_bounds__(64 * NW) void k_latent_decode_mfma(const AttnP p, const zls_batch_t b, const float* __restrict__ qa,
                                                                float* __restrict__ ws, int n_splits) {
    constexpr int CR = RW * 32 + 8;
    __shared__ __attribute__((aligned(16))) uint16_t ct_all[NW][32 * CR];
    __shared__ __attribute__((aligned(16))) float4 part[2][NW][2][64];
    const int t = blockIdx.x, split = blockIdx.z, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nrow = lane & 15, kq = lane >> 4;
    const int head = blockIdx.y * 16 + nrow, r0 = wave * RW * 32;
    const bool hvalid = head < p.heads;
    const int sq = b.tok_seq[t];
    if (p.single_only && b.seq_start[sq + 1] - b.seq_start[sq] > 1) return;
    const int pos = b.seq_pos0[sq] + (t - b.seq_start[sq]);
    const int key_lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;
    const int nkeys = pos + 1 - key_lo;
    const int chunk = ((nkeys + n_splits - 1) / n_splits + 31) & ~31;
    const int k0 = key_lo + split * chunk, k1 = min(pos + 1, k0 + chunk);
    const int32_t* pages = b.page_table + (size_t)sq * b.max_pages;
    const uint16_t* cache = reinterpret_cast<const uint16_t*>(p.cache);
    uint16_t* ct = ct_all[wave];

    uint4 cr[2][RW];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int j = j0 + 16 * c + nrow;
            const bool valid = j < k1;
            const size_t base = valid ? ((size_t)pages[j / b.page_size] * b.page_size + j % b.page_size) * p.rank : 0;
#pragma unroll
            for (int kk = 0; kk < RW; ++kk) {
                const int r = r0 + 32 * kk + 8 * kq;
                cr[c][kk] = (valid && r < p.rank) ? *reinterpret_cast<const uint4*>(cache + base + r) : make_uint4(0, 0, 0, 0);
            }
        }
    };
    if (k0 < k1) fetch(k0);
    uint4 qf[RW];
    {
        const float* qr = qa + ((size_t)t * p.heads + (hvalid ? head : 0)) * p.rank;
#pragma unroll
        for (int kk = 0; kk < RW; ++kk) {
            const int r = r0 + 32 * kk + 8 * kq;
            const bool in = hvalid && r < p.rank;                                  // (rank comes in whole 8s)
            const float4 a = in ? seq_ld4(qr + r) : make_float4(0.f, 0.f, 0.f, 0.f), c = in ? seq_ld4(qr + r + 4) : make_float4(0.f, 0.f, 0.f, 0.f);
            qf[kk] = make_uint4(ZT<ZL_BF16>::from_f32(a.x) | (uint32_t)ZT<ZL_BF16>::from_f32(a.y) << 16, ZT<ZL_BF16>::from_f32(a.z) | (uint32_t)ZT<ZL_BF16>::from_f32(a.w) << 16,
                                ZT<ZL_BF16>::from_f32(c.x) | (uint32_t)ZT<ZL_BF16>::from_f32(c.y) << 16, ZT<ZL_BF16>::from_f32(c.z) | (uint32_t)ZT<ZL_BF16>::from_f32(c.w) << 16);
        }
    }
    fa_f4 o[2 * RW];
#pragma unroll
    for (int rt = 0; rt < 2 * RW; ++rt) o[rt] = (fa_f4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    int turn = 0;
    for (int j0 = k0; j0 < k1; j0 += 32, turn ^= 1) {
        fa_f4 sc[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            sc[c] = (fa_f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < RW; ++kk)
                sc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(fa_b8, cr[c][kk]), __builtin_bit_cast(fa_b8, qf[kk]), sc[c], 0, 0, 0);
            if (NW > 1) part[turn][wave][c][lane] = make_float4(sc[c][0], sc[c][1], sc[c][2], sc[c][3]);
        }
        // (the wave's own reads of the last block's columns came before these writes, LDS keeps a wave's order)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int kk = 0; kk < RW; ++kk) *reinterpret_cast<uint4*>(ct + (16 * c + nrow) * CR + 32 * kk + 8 * kq) = cr[c][kk];
        if (j0 + 32 < k1) fetch(j0 + 32);
        __syncthreads();                                                           // (one per block: the partial scores alternate between two places)
        float mx = -INFINITY;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (NW > 1) {
                float4 a = part[turn][0][c][lane];
#pragma unroll
                for (int w = 1; w < NW; ++w) {
                    const float4 v = part[turn][w][c][lane];
                    a = make_float4(a.x + v.x, a.y + v.y, a.z + v.z, a.w + v.w);
                }
                sc[c] = (fa_f4){a.x, a.y, a.z, a.w};
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = (j0 + 16 * c + 4 * kq + r < k1) ? sc[c][r] : -INFINITY;        // (the folded query carries the scale)
                sc[c][r] = v;
                mx = fmaxf(mx, v);
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mnew = fmaxf(m, mx);                                           // finite: key j0 is valid
        const float corr = __expf(m - mnew);                                       // m = -inf at the first block: 0
        float ps = 0.f;
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                uint16_t hb[2], lb[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float pv = sc[c][r + e] == -INFINITY ? 0.f : __expf(sc[c][r + e] - mnew);
                    ps += pv;
                    fa_split(pv, hb[e], lb[e]);
                }
                hi[2 * c + (r >> 1)] = hb[0] | (uint32_t)hb[1] << 16;
                lo[2 * c + (r >> 1)] = lb[0] | (uint32_t)lb[1] << 16;
            }
        }
        ps += __shfl_xor(ps, 16, 64);
        ps += __shfl_xor(ps, 32, 64);
        l = l * corr + ps;
        m = mnew;
        const fa_b8 ph = __builtin_bit_cast(fa_b8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
        const fa_b8 pl = __builtin_bit_cast(fa_b8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
#pragma unroll
        for (int rt = 0; rt < 2 * RW; ++rt) {
            // slot s of lane group kq <-> key 16 (s / 4) + 4 kq + s % 4 of the block; this lane's column of the wave's part: 16 rt + nrow
            uint32_t w[4];
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) {
                const int ka = 16 * (s2 >> 1) + 4 * kq + 2 * (s2 & 1);
                w[s2] = ct[ka * CR + 16 * rt + nrow] | (uint32_t)ct[(ka + 1) * CR + 16 * rt + nrow] << 16;
            }
            const fa_b8 a = __builtin_bit_cast(fa_b8, make_uint4(w[0], w[1], w[2], w[3]));
            o[rt] *= corr;
            o[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ph, o[rt], 0, 0, 0);
            o[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pl, o[rt], 0, 0, 0);
        }
    }
    if (!hvalid) return;
    const LatWs out(ws, b.n_tok, p, n_splits, t, head, split);
    if (wave == 0 && kq == 0) *out.ml = make_float2(m, l);
#pragma unroll
    for (int rt = 0; rt < 2 * RW; ++rt) {
        const int r = r0 + 16 * rt + 4 * kq;
        if (r < p.rank) *reinterpret_cast<float4*>(out.acc + r) = make_float4(o[rt][0], o[rt][1], o[rt][2], o[rt][3]);
    }
}

}  // namespace

extern "C" int zls_latent_rope_store(float* proj, int64_t ld, int64_t col0, const float* weight, float eps, int64_t rank, int64_t rot,
                                     const float* freq, int interleaved, int64_t q_col0, int64_t heads, int64_t qdim, float rot_gain,
                                     const zls_batch_t* b, void* cache, int dtype, zl_stream_t s) {
    ZL_CHECK_ARG(proj && weight && cache && seq_batch_ok(b) && b->page_table && b->page_size > 0 && b->max_pages > 0 && rank > 0 && rot >= 0, ZL_EINVAL);
    ZL_CHECK_ARG(col0 >= 0 && col0 + rank + rot <= ld && rot % 2 == 0, ZL_ESHAPE);
    ZL_CHECK_ARG(rot == 0 || (freq && heads > 0 && qdim >= rot && q_col0 >= 0 && q_col0 + heads * qdim <= ld), ZL_ESHAPE);
#define CALL(DT) hipLaunchKernelGGL((k_latent_store<DT>), dim3(b->n_tok), dim3(256), 0, (hipStream_t)s, proj, ld, (int)col0, weight, eps, (int)rank, \
                                    (int)rot, freq, interleaved ? 1 : 0, (int)q_col0, (int)(rot ? heads : 0), (int)qdim, *b, cache, rot_gain);
    ZLS_DISPATCH(dtype, CALL)
#undef CALL
    return zl_launch_status();
}

extern "C" int zls_latent_store(const float* proj, int64_t ld, int64_t col0, const float* weight, float eps, int64_t rank, const zls_batch_t* b,
                                void* cache, int dtype, zl_stream_t s) {
    return zls_latent_rope_store(const_cast<float*>(proj), ld, col0, weight, eps, rank, 0, nullptr, 0, 0, 0, 0, 1.0f, b, cache, dtype, s);
}

extern "C" int64_t zls_latent_attention_workspace_bytes(int64_t n_tok, int64_t heads, int64_t rank, int64_t n_splits) {
    if (n_tok <= 0 || heads <= 0 || rank <= 0 || n_splits <= 0) return ZL_EINVAL;
    return (n_tok * heads * n_splits * (rank + 2) + n_tok * heads * rank) * (int64_t)sizeof(float);    /* sums, (maximum, denominator) | folded queries */
}

extern "C" int zls_latent_attention(const float* q, int64_t ldq, int64_t q_col0, const float* gate, int64_t ldg, int64_t g_col0, const void* w_uk,
                                    const void* w_uv, const float* sink, const void* cache, const zls_batch_t* b, float scale, int64_t heads,
                                    int64_t dim, int64_t vdim, int64_t rank, void* out, int dtype, int single_only, void* workspace,
                                    int64_t n_splits, int no_mfma, int64_t window, zl_stream_t s) {
    ZL_CHECK_ARG(q && w_uk && w_uv && cache && out && workspace && seq_batch_ok(b) && b->page_table && b->page_size > 0 && b->max_pages > 0, ZL_EINVAL);
    ZL_CHECK_ARG(heads > 0 && dim > 0 && vdim > 0 && rank > 0 && heads <= 65535 && n_splits > 0 && n_splits <= 65535, ZL_EINVAL);
    ZL_CHECK_ARG(q_col0 >= 0 && q_col0 + heads * dim <= ldq && (!gate || (g_col0 >= 0 && g_col0 + heads <= ldg)), ZL_ESHAPE);
    const size_t lds = (16 * ((size_t)rank + 4) + 4 * (size_t)rank) * sizeof(float);
    ZL_CHECK_ARG(rank <= 1024 && lds <= 64 * 1024, ZL_ELIMIT);
    AttnP p;
    p.q = q; p.gate = gate; p.w_uk = w_uk; p.w_uv = w_uv; p.sink = sink; p.cache = cache; p.out = out;
    p.ldq = ldq; p.ldg = ldg; p.q_col0 = (int)q_col0; p.g_col0 = (int)g_col0;
    p.heads = (int)heads; p.dim = (int)dim; p.vdim = (int)vdim; p.rank = (int)rank; p.scale = scale; p.single_only = single_only;
    ZL_CHECK_ARG(window < (1 << 30), ZL_ESHAPE);
    p.window = window > 0 ? (int)window : 0;
    // (the split kernel's eight 16-byte slots per thread cover 1024 bf16 or 512 fp32 columns of a row; longer fp32 rows are read singly)
    p.vec = (rank % (dtype == ZL_BF16 ? 8 : 4) == 0 && ((uintptr_t)cache & 15) == 0 && (dtype == ZL_BF16 || rank <= 512)) ? 1 : 0;
    const dim3 grid(b->n_tok, (unsigned)((heads + 3) / 4), (unsigned)n_splits);
    hipStream_t hs = (hipStream_t)s;
    float* ws = (float*)workspace;
    float* qa = ws + (size_t)b->n_tok * heads * n_splits * rank;
    const int ns = (int)n_splits;
    // bf16 with aligned rows of at most 640 latent columns (512 + a rotated part): the split pass on the matrix cores (absorb and combine
    // are shared)
    const bool ws16 = ((uintptr_t)workspace & 15) == 0;
    const bool mfma = dtype == ZL_BF16 && p.vec && ws16 && rank <= 640 && !no_mfma;
    p.pairs = rank % 2 == 0 && ((uintptr_t)w_uk & 7) == 0;
    const unsigned tgrid = (unsigned)((b->n_tok + kLatTok - 1) / kLatTok);
    const size_t lds_v = (size_t)(kLatTok * (rank + n_splits) + kLatTok) * sizeof(float);
    const bool rows8 = rank % 8 == 0 && ws16 && ((uintptr_t)w_uv & 15) == 0 && lds_v <= 64 * 1024;
    const dim3 mgrid(b->n_tok, (unsigned)((heads + 15) / 16), (unsigned)n_splits);
#define MSPLIT(RW, NW) hipLaunchKernelGGL((k_latent_decode_mfma<RW, NW>), mgrid, dim3(64 * NW), 0, hs, p, *b, qa, ws, ns)
#define SPLIT(DT, RPL) hipLaunchKernelGGL((k_latent_split<DT, RPL>), grid, dim3(256), lds, hs, p, *b, qa, ws, ns)
#define CALL(DT)                                  \
    hipLaunchKernelGGL((k_latent_absorb<DT>), dim3(tgrid, (unsigned)heads, (unsigned)((rank + 63) / 64)), dim3(256), 0, hs, p, *b, qa); \
    if (mfma) {                                   \
        if (rank <= 64) MSPLIT(1, 2);             \
        else if (rank <= 128) MSPLIT(1, 4);       \
        else if (rank <= 256) MSPLIT(2, 4);       \
        else if (rank <= 512) MSPLIT(4, 4);       \
        else MSPLIT(5, 4);                        \
    } else if (rank <= 64) SPLIT(DT, 1);          \
    else if (rank <= 128) SPLIT(DT, 2);           \
    else if (rank <= 256) SPLIT(DT, 4);           \
    else if (rank <= 512) SPLIT(DT, 8);           \
    else SPLIT(DT, 16);                           \
    if (rows8) hipLaunchKernelGGL((k_latent_combine_v<DT>), dim3(tgrid, (unsigned)heads, (unsigned)((vdim + 15) / 16)), dim3(256), lds_v, hs, p, *b, ws, ns); \
    else hipLaunchKernelGGL((k_latent_combine<DT>), dim3(b->n_tok, (unsigned)heads, (unsigned)((vdim + 31) / 32 > 4 ? 4 : (vdim + 31) / 32)), dim3(256), (size_t)(rank + n_splits) * sizeof(float), hs, p, *b, ws, ns);
    ZLS_DISPATCH(dtype, CALL)
#undef CALL
#undef SPLIT
#undef MSPLIT
    return zl_launch_status();
}

extern "C" int zls_latent_attention_prompt(const float* q, int64_t ldq, int64_t q_col0, const float* gate, int64_t ldg, int64_t g_col0,
                                           const void* k, int64_t ldk, const void* vt, int64_t ldv, const float* sink, const int32_t* ctx_start,
                                           const zls_batch_t* b, float scale, int64_t heads, int64_t dim, int64_t vdim, void* out, int dtype,
                                           int64_t window, const int32_t* ctx_pos0, zl_stream_t s) {
    ZL_CHECK_ARG(q && k && vt && ctx_start && out && seq_batch_ok(b) && window < (1 << 30), ZL_EINVAL);
    ZL_CHECK_ARG(dtype == ZL_BF16, ZL_EDTYPE);
    ZL_CHECK_ARG(heads > 0 && heads <= 65535 && dim > 0 && vdim > 0 && dim <= 256 && vdim <= 256, ZL_ESHAPE);
    ZL_CHECK_ARG(q_col0 >= 0 && q_col0 + heads * dim <= ldq && (!gate || (g_col0 >= 0 && g_col0 + heads <= ldg)), ZL_ESHAPE);
    ZL_CHECK_ARG(ldk >= heads * dim && ldv % 8 == 0 && ((uintptr_t)vt & 15) == 0, ZL_ESHAPE);
    FaP p;
    p.q = q; p.gate = gate; p.k = (const uint16_t*)k; p.vt = (const uint16_t*)vt; p.sink = sink; p.ctx_start = ctx_start; p.out = (uint16_t*)out;
    p.ldq = ldq; p.ldg = ldg; p.ldk = ldk; p.ldv = ldv; p.q_col0 = (int)q_col0; p.g_col0 = (int)g_col0;
    p.heads = (int)heads; p.dim = (int)dim; p.vdim = (int)vdim; p.scale = scale; p.window = window > 0 ? (int)window : 0; p.ctx_pos0 = ctx_pos0;
    p.tiles_per_seq = (b->max_count + 63) / 64;
    const bool vec = dim % 8 == 0 && ldk % 8 == 0 && ldk < (1 << 24) && ldv < (1 << 24) && seq_aligned(k) && ldq % 4 == 0 && q_col0 % 4 == 0 && seq_aligned(q);
    ZL_CHECK_ARG((int64_t)b->n_seq * p.tiles_per_seq * heads <= INT32_MAX, ZL_ELIMIT);
    const dim3 grid((unsigned)(b->n_seq * p.tiles_per_seq * heads));
    hipStream_t hs = (hipStream_t)s;
    // two groups where some query has more than four key tiles and the workgroups are few to a CU (two groups of long heads: 88 KB of LDS)
    const bool pair = b->max_count > 128 && grid.x <= 1024;
    // the smallest instantiation that holds both the key size (32 DK) and the value size (16 DV): heads with a rotated part have keys
    // longer than their values
#define FA(DK, DV, NG, VEC) if (dim <= 32 * DK && vdim <= 16 * DV) { hipLaunchKernelGGL((k_latent_fa<DK, DV, NG, VEC>), grid, dim3(256 * NG), 0, hs, p, *b); return zl_launch_status(); }
    if (vec && pair) { FA(2, 2, 2, true) FA(2, 4, 2, true) FA(4, 4, 2, true) FA(4, 8, 2, true) FA(6, 8, 2, true) }
    if (vec) { FA(1, 2, 1, true) FA(2, 2, 1, true) FA(2, 4, 1, true) FA(4, 4, 1, true) FA(4, 8, 1, true) FA(6, 8, 1, true) FA(8, 8, 1, true) FA(8, 16, 1, true) }
    FA(1, 2, 1, false) FA(2, 2, 1, false) FA(2, 4, 1, false) FA(4, 4, 1, false) FA(4, 8, 1, false) FA(6, 8, 1, false) FA(8, 8, 1, false) FA(8, 16, 1, false)
#undef FA
    return ZL_ESHAPE;
}
