// arc_prefill.hip -- the batched prompt pass on gfx950 MFMA (the reference's
// build_prefill, src/arcllm_v1_runtime.cpp:340-369, which runs dequant-in-LDS
// fp32 tiles).
//
// A prompt of M <= 256 tokens at positions pos0 .. pos0+M-1 is processed as
// matrices: per layer (8 launches)
//   [q|k|v] = X [Wq|Wk|Wv]^T  (split-K partials, one launch)   k_mm_qkv
//   + bias, RoPE on q and k, q -> fp32, k and v -> fp16 cache  k_pf_qkv_epi
//   causal GQA over the cache (positions <= own) -> X (fp16)    k_pf_attn
//   H += X Wo^T, X = RMSNorm(H) (ffn norm)                      k_mm, k_pf_res_norm
//   s = silu(X Wg^T) * (X Wu^T) -> fp16                         k_mm<SWIGLU>
//   H += s Wd^T, X = RMSNorm(H) (next layer's attention norm)   k_mm, k_pf_res_norm
// after the embedding and the first layer's attention norm (k_pf_embed,
// k_pf_rmsnorm), then the output RMSNorm + LM head + argmax on the last row
// only (the decode step's kernels), leaving the argmax as the next token.
//
// GEMM: arc_pf_gemm.hpp (packed weights decoded in registers, X through LDS).  Operands are fp16, accumulation fp32.
#include "arc_session.hpp"
#include "arc_pf_gemm.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>

namespace arc {

// --------------------------------------------------------- small kernels
// H[m] = dequant(token_embd[tokens[m]]); grid (nb, M), element formula of
// the decode embedding.
__global__ __launch_bounds__(256) void k_pf_embed(const uint8_t* __restrict__ emb, uint32_t nb,
                                                  const uint32_t* __restrict__ tokens, float* __restrict__ h)
{
#pragma clang fp contract(off)
    const uint32_t m = blockIdx.y, e = blockIdx.x * kQK + threadIdx.x;
    const uint8_t* b = emb + (uint64_t(tokens[m]) * nb + blockIdx.x) * kQ4Bytes;
    const uint32_t k = threadIdx.x, j = k >> 5;
    const float d = f16_bits_to_f32(uint32_t(b[0]) | (uint32_t(b[1]) << 8));
    const float dm = f16_bits_to_f32(uint32_t(b[2]) | (uint32_t(b[3]) << 8));
    const uint8_t* s = b + 4;
    uint32_t sc, mn;
    if (j < 4) {
        sc = s[j] & 63u;
        mn = s[j + 4] & 63u;
    } else {
        sc = (s[j + 4] & 15u) | (uint32_t(s[j - 4] >> 6) << 4);
        mn = (s[j + 4] >> 4) | (uint32_t(s[j] >> 6) << 4);
    }
    const uint32_t l64 = k & 63u;
    const uint8_t qb = b[16 + (k >> 6) * 32 + (l64 & 31u)];
    const uint32_t q = l64 < 32u ? (qb & 15u) : (qb >> 4);
    const float t0 = d * float(sc);
    const float t1 = t0 * float(q);
    const float t2 = dm * float(mn);
    h[uint64_t(m) * nb * kQK + e] = t1 - t2;
}

// X[m] = fp16((H[m] * inv) * w), inv = 1/sqrt(mean(H[m]^2) + eps); grid M.
__global__ __launch_bounds__(256) void k_pf_rmsnorm(const float* __restrict__ h, uint32_t n, const float* __restrict__ w,
                                                    float eps, _Float16* __restrict__ x, uint32_t ldx)
{
    __shared__ float red[4];
    const float* r = h + uint64_t(blockIdx.x) * n;
    float ss = 0.0f;
    for (uint32_t i = threadIdx.x; i < n; i += 256) ss = __builtin_fmaf(r[i], r[i], ss);
    ss = block_sum<256>(ss, red);
    const float inv = 1.0f / sqrtf(ss / float(n) + eps);
    _Float16* o = x + uint64_t(blockIdx.x) * ldx;
    for (uint32_t i = threadIdx.x; i < n; i += 256) o[i] = _Float16((r[i] * inv) * w[i]);
}

// q|k|v epilogue, per (m, column pair) of the [hidden | kv_dim | kv_dim]
// partials: fixed-order sum over the splits + bias; q and k pairs are
// rotated (RoPE at position pos0 + m), q -> fp32, k and v -> fp16 cache row
// pos0 + m.
__global__ __launch_bounds__(256) void k_pf_qkv_epi(const float* __restrict__ part, uint32_t splits, uint32_t mpad,
                                                    uint32_t hidden, uint32_t kv_dim, const float* __restrict__ qb,
                                                    const float* __restrict__ kb, const float* __restrict__ vb,
                                                    const float2* __restrict__ rope, uint32_t pos0,
                                                    float* __restrict__ q, _Float16* __restrict__ kc,
                                                    _Float16* __restrict__ vc)
{
    const uint32_t N = hidden + 2 * kv_dim, m = blockIdx.y;
    const uint32_t c = 2 * (blockIdx.x * 256 + threadIdx.x);
    if (c >= N) return;
    float a = 0.0f, b = 0.0f;
    for (uint32_t s0 = 0; s0 < splits; s0 += 8) {  // 8 splits' loads in flight, added in split order
        float2 v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
            v[u] = s0 + u < splits ? *reinterpret_cast<const float2*>(part + (uint64_t(s0 + u) * mpad + m) * N + c)
                                   : float2{0.0f, 0.0f};
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
            if (s0 + u < splits) {
                a += v[u].x;
                b += v[u].y;
            }
    }
    if (c >= hidden + kv_dim) {
        const uint32_t lc = c - hidden - kv_dim;
        _Float16* dst = vc + uint64_t(pos0 + m) * kv_dim + lc;
        dst[0] = _Float16(a + vb[lc]);
        dst[1] = _Float16(b + vb[lc + 1]);
        return;
    }
    const bool isq = c < hidden;
    const uint32_t lc = isq ? c : c - hidden;
    const float* bias = isq ? qb : kb;
    a = a + bias[lc];
    b = b + bias[lc + 1];
    const float2 cs = rope[uint64_t(pos0 + m) * 64 + ((lc & 127u) >> 1)];
    const float ra = a * cs.x - b * cs.y, rb = a * cs.y + b * cs.x;
    if (isq) {
        q[uint64_t(m) * hidden + lc] = ra;
        q[uint64_t(m) * hidden + lc + 1] = rb;
    } else {
        _Float16* dst = kc + uint64_t(pos0 + m) * kv_dim + lc;
        dst[0] = _Float16(ra);
        dst[1] = _Float16(rb);
    }
}

// Fixed-order second pass of a split-K projection with the residual (when
// `res` is set, which may be h) and (NORM) the next RMSNorm: H[m][c] = res[m][c]
// + sum_s part[s][m][c] (s in order), X[m] = fp16((H[m] * inv) * w),
// inv = 1/sqrt(mean(H[m]^2) + eps).  Grid M, one row
// per workgroup of 1024 threads; thread t owns columns t + 1024*k (k < KC,
// n <= 1024*KC), and loads the partials of 8 splits at a time, all in flight,
// before adding them in split order.
constexpr int kResCols = 20;  // n <= 20480, the model limit on hidden
template <bool NORM, int KC>
__global__ __launch_bounds__(1024) void k_pf_res_norm(const float* __restrict__ part, uint32_t splits, uint32_t mpad,
                                                      uint32_t n, const float* res, float* h,
                                                      const float* __restrict__ w, float eps, _Float16* __restrict__ x,
                                                      uint32_t ldx)
{
    static_assert(KC >= 1 && KC <= kResCols, "columns per thread");
    constexpr uint32_t kBatch = 8;
    __shared__ float red[16];
    const uint32_t m = blockIdx.x, t = threadIdx.x;
    float* r = h + uint64_t(m) * n;
    const float* pm = part + uint64_t(m) * n;
    const uint64_t sstride = uint64_t(mpad) * n;
    float a[KC];
#pragma unroll
    for (int k = 0; k < KC; ++k) a[k] = 0.0f;
    for (uint32_t s0 = 0; s0 < splits; s0 += kBatch) {
        float v[kBatch][KC];
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u)
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                const uint32_t c = t + 1024u * k;
                v[u][k] = (s0 + u < splits && c < n) ? pm[(s0 + u) * sstride + c] : 0.0f;
            }
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u)
#pragma unroll
            for (int k = 0; k < KC; ++k)
                if (s0 + u < splits) a[k] += v[u][k];
    }
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < KC; ++k) {
        const uint32_t c = t + 1024u * k;
        if (c < n) {
            if (res) a[k] = res[uint64_t(m) * n + c] + a[k];
            r[c] = a[k];
            if constexpr (NORM) ss = __builtin_fmaf(a[k], a[k], ss);
        }
    }
    if constexpr (NORM) {
        ss = block_sum<1024>(ss, red);
        const float inv = 1.0f / sqrtf(ss / float(n) + eps);
        _Float16* o = x + uint64_t(m) * ldx;
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const uint32_t c = t + 1024u * k;
            if (c < n) o[c] = _Float16((a[k] * inv) * w[c]);
        }
    }
}

template <bool NORM>
void launch_res_norm(uint32_t M, hipStream_t st, const float* part, uint32_t splits, uint32_t mpad, uint32_t n,
                     const float* res, float* h, const float* w, float eps, _Float16* x, uint32_t ldx)
{
    const uint32_t kc = (n + 1023u) / 1024u;
    if (kc <= 4)
        hipLaunchKernelGGL((k_pf_res_norm<NORM, 4>), dim3(M), dim3(1024), 0, st, part, splits, mpad, n, res, h, w, eps, x,
                           ldx);
    else if (kc <= 8)
        hipLaunchKernelGGL((k_pf_res_norm<NORM, 8>), dim3(M), dim3(1024), 0, st, part, splits, mpad, n, res, h, w, eps, x,
                           ldx);
    else
        hipLaunchKernelGGL((k_pf_res_norm<NORM, kResCols>), dim3(M), dim3(1024), 0, st, part, splits, mpad, n, res, h, w,
                           eps, x, ldx);
}

// Causal GQA for query row m (position pos0 + m) and kv head g: the HPK q
// heads of g attend to cache positions 0 .. pos0 + m in chunks of 64 with an
// online softmax (running max and sum, rescaled per chunk); output fp16 into
// the GEMM input X[m][head*128 + d].
template <int HPK>
__global__ __launch_bounds__(256) void k_pf_attn(const float* __restrict__ q, const _Float16* __restrict__ kc,
                                                 const _Float16* __restrict__ vc, uint32_t kv_heads, uint32_t pos0,
                                                 float scale, _Float16* __restrict__ x, uint32_t ldx)
{
    const uint32_t m = blockIdx.x, g = blockIdx.y, kvd = kv_heads * kHeadDim;
    const uint32_t hidden = kv_heads * HPK * kHeadDim;
    const uint32_t T = pos0 + m + 1;
    const int tid = threadIdx.x;
    __shared__ float qs[HPK][kHeadDim];
    __shared__ float sc[HPK][kChunk];
    __shared__ float alpha[HPK], lsum[HPK], mrun[HPK];
    __shared__ float ored[4][HPK][kHeadDim];
    for (uint32_t i = tid; i < HPK * kHeadDim; i += 256)
        qs[i >> 7][i & 127u] = q[uint64_t(m) * hidden + g * HPK * kHeadDim + i];
    if (tid < HPK) {
        mrun[tid] = -INFINITY;
        lsum[tid] = 0.0f;
    }
    const uint32_t tk = uint32_t(tid) >> 2, part = tid & 3;
    const int vi = tid & 63, pg = tid >> 6;
    float o[HPK][2];
#pragma unroll
    for (int h = 0; h < HPK; ++h) o[h][0] = o[h][1] = 0.0f;
    __syncthreads();
    for (uint32_t t0 = 0; t0 < T; t0 += kChunk) {
        const uint32_t nt = min(uint32_t(kChunk), T - t0);
        // every K and V load of the chunk is issued here, so the chunk costs
        // one memory round trip
        uint4 kraw[4];
        half2_t vraw[16];
        {
            const uint4* kp = reinterpret_cast<const uint4*>(kc + uint64_t(t0 + min(tk, nt - 1)) * kvd + g * kHeadDim +
                                                             part * 32);
#pragma unroll
            for (int i = 0; i < 4; ++i) kraw[i] = kp[i];
            const _Float16* vb = vc + uint64_t(t0) * kvd + g * kHeadDim + 2 * vi;
#pragma unroll
            for (int tt = 0; tt < 16; ++tt)
                vraw[tt] = *reinterpret_cast<const half2_t*>(vb + uint64_t(min(uint32_t(pg * 16 + tt), nt - 1)) * kvd);
        }
        {   // scores of positions t0 + tk
            float s[HPK];
#pragma unroll
            for (int h = 0; h < HPK; ++h) s[h] = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4 raw = kraw[i];
                const uint32_t w4[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float kv = static_cast<float>(__builtin_bit_cast(half2_t, w4[e >> 1])[e & 1]);
                    const int d = part * 32 + i * 8 + e;
#pragma unroll
                    for (int h = 0; h < HPK; ++h) s[h] = __builtin_fmaf(qs[h][d], kv, s[h]);
                }
            }
#pragma unroll
            for (int h = 0; h < HPK; ++h) s[h] = group_sum<4>(s[h]);
            if (part == 0 && tk < nt)
#pragma unroll
                for (int h = 0; h < HPK; ++h) sc[h][tk] = s[h] * scale;
        }
        __syncthreads();
        {   // online softmax update: wave w handles heads w, w+4
            const int w = tid >> 6, lane = tid & 63;
            for (int h = w; h < HPK; h += 4) {
                const float sv = uint32_t(lane) < nt ? sc[h][lane] : -INFINITY;
                const float cm = wave_max(sv);
                const float mnew = fmaxf(mrun[h], cm);
                const float e = uint32_t(lane) < nt ? expf(sv - mnew) : 0.0f;
                const float l = group_sum<kWave>(e);
                sc[h][lane] = e;
                if (lane == 0) {
                    const float a = expf(mrun[h] - mnew);  // 0 on the first chunk
                    alpha[h] = a;
                    lsum[h] = lsum[h] * a + l;
                    mrun[h] = mnew;
                }
            }
        }
        __syncthreads();
        {   // o = o * alpha + sum_t p_t v_t over this chunk
#pragma unroll
            for (int h = 0; h < HPK; ++h) {
                o[h][0] *= alpha[h];
                o[h][1] *= alpha[h];
            }
#pragma unroll
            for (int tt = 0; tt < 16; ++tt) {
                const uint32_t t = pg * 16 + tt;
                const bool in = t < nt;
                const half2_t vv = vraw[tt];
                const float v0 = in ? static_cast<float>(vv.x) : 0.0f, v1 = in ? static_cast<float>(vv.y) : 0.0f;
#pragma unroll
                for (int h = 0; h < HPK; ++h) {
                    const float pr = sc[h][t];
                    o[h][0] = __builtin_fmaf(pr, v0, o[h][0]);
                    o[h][1] = __builtin_fmaf(pr, v1, o[h][1]);
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int h = 0; h < HPK; ++h) {
        ored[pg][h][2 * vi] = o[h][0];
        ored[pg][h][2 * vi + 1] = o[h][1];
    }
    __syncthreads();
    for (uint32_t idx = tid; idx < HPK * kHeadDim; idx += 256) {
        const uint32_t h = idx >> 7, d = idx & 127u;
        const float v = ((ored[0][h][d] + ored[1][h][d]) + ored[2][h][d]) + ored[3][h][d];
        x[uint64_t(m) * ldx + (g * HPK + h) * kHeadDim + d] = _Float16(v / lsum[h]);
    }
}

// Causal GQA of the prompt pass on MFMA.  Workgroup (query block b of 32
// rows, q head hq of kv head hq / hpk): 4 waves; wave w takes the
// 64-position key chunks w, w + 4, ... of positions 0 .. the block's last,
// with its own online softmax per query; at the end the waves' states are
// combined through LDS in wave order.
//  scores  S^T = K Q^T per 32-key tile on v_mfma_f32_32x32x16_f16: A = K
//          rows straight from the cache (lane -> key lane%32; step s: dims
//          16s + 8(lane/32) .. +7, 16 bytes of the row), B = Q^T (lane ->
//          query lane%32, the same dims) as fp16 hi + lo parts (q = hi + lo
//          to 2^-22 relative; K*hi and K*lo are exact products).  D: lane ->
//          query lane%32, value i -> key 8(i/4) + 4(lane/32) + i%4.
//  softmax the chunk maximum of a query from the lane's 32 scores and its
//          partner half-wave's (lane ^ 32); positions past the query's own
//          are masked.  Weights e^(x - max), rescaling the running sum and
//          the output by e^(max_old - max_new).
//  Bound by vector instructions: one wave per SIMD, 64 weights per lane and
//  chunk, about 10 instructions each for expf.  256 rows at position 768, 28
//  heads: 21.7 us, 24.8 with the mask compared in every chunk; 8 waves per
//  workgroup (half the chunks each) 26.0; the weights' hi and lo parts by
//  v_cvt_pk_f16_f32 and skipping rescalings by 1 changed nothing.  Weights as
//  v_exp_f32 of scores times log2(e) take 20.1 us and are as accurate, but round
//  differently, and a prompt's logits move by 5e-3 with them.
//  values  O^T = V^T P^T: B = P^T straight from the lane's weights (step s of
//          a tile: values 8s .. 8s+7, keys 16s + 8(j/4) + 4(lane/32) + j%4)
//          as fp16 hi + lo; A = V^T from LDS, where the wave stages its chunk
//          transposed with key k at column k with bits 2 and 3 swapped, so a
//          lane's 8 keys of a step are 16 contiguous bytes.  D: lane ->
//          query lane%32, value i of dim tile t -> dim 32t + 8(i/4) +
//          4(lane/32) + i%4.
// Semantics as k_pf_attn (src/arcllm_v1_runtime.cpp:340-369 per row).
constexpr int kVtLd = kChunk + 8;  // halves per V^T row in LDS (padded)

__device__ __forceinline__ uint32_t swap_bits_2_3(uint32_t k)
{
    return (k & ~12u) | ((k & 4u) << 1) | ((k & 8u) >> 1);
}

__global__ __launch_bounds__(256, 2) void k_pf_attn_mf(const float* __restrict__ q, const _Float16* __restrict__ kc,
                                                       const _Float16* __restrict__ vc, uint32_t kv_heads,
                                                       uint32_t hpk, uint32_t pos0, uint32_t M, uint32_t max_ctx,
                                                       float scale, _Float16* __restrict__ x, uint32_t ldx)
{
    __shared__ __align__(16) _Float16 vt[4][kHeadDim][kVtLd];  // per wave: its chunk's V^T; then the outputs
    __shared__ float mw[4][32], lw[4][32];
    const uint32_t b = blockIdx.x, hq = blockIdx.y, g = hq / hpk;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, l32 = lane & 31, h2 = lane >> 5;
    const uint32_t kvd = kv_heads * kHeadDim, hidden = kv_heads * hpk * kHeadDim;
    const uint32_t q0 = b * 32, qlast = min(q0 + 31, M - 1);
    const uint32_t qpos = pos0 + q0 + uint32_t(l32);  // this lane's query position
    const uint32_t nkc = (pos0 + qlast + kChunk) / kChunk;  // chunks holding positions 0 .. pos0 + qlast

    half8 qh[8], ql[8];  // B operand of the scores: query l32, dims 16s + 8 h2 .. +7
    {
        const float* qp = q + uint64_t(min(q0 + uint32_t(l32), M - 1)) * hidden + hq * kHeadDim + 8 * h2;
#pragma unroll
        for (int st = 0; st < 8; ++st) {
            const float4 a = *reinterpret_cast<const float4*>(qp + 16 * st);
            const float4 c = *reinterpret_cast<const float4*>(qp + 16 * st + 4);
            const float f[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const _Float16 hi = static_cast<_Float16>(f[j]);
                qh[st][j] = hi;
                ql[st][j] = static_cast<_Float16>(f[j] - static_cast<float>(hi));
            }
        }
    }
    f32x16 o[4];  // O^T: dim tile t, query l32
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = 0.0f;
    float mrun = -INFINITY, lrun = 0.0f;  // lrun: this half-wave's share
    _Float16(*vw)[kVtLd] = vt[w];

    for (uint32_t c = uint32_t(w); c < nkc; c += 4) {
        const uint32_t kbase = c * kChunk;
        // this chunk's V rows (lane -> key kbase + lane), 16 bytes at a time,
        // and both tiles' K fragments, all issued before any is used
        uint4 vr[16];
        {
            const uint4* vp = reinterpret_cast<const uint4*>(vc + uint64_t(min(kbase + uint32_t(lane), max_ctx - 1)) * kvd +
                                                             g * kHeadDim);
#pragma unroll
            for (int e = 0; e < 16; ++e) vr[e] = vp[e];
        }
        uint4 kf[2][8];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            const uint4* kp = reinterpret_cast<const uint4*>(
                kc + uint64_t(min(kbase + 32u * kt + uint32_t(l32), max_ctx - 1)) * kvd + g * kHeadDim + 8 * h2);
#pragma unroll
            for (int st = 0; st < 8; ++st) kf[kt][st] = kp[2 * st];
        }
        // scores of the two 32-key tiles
        f32x16 sc[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[kt][i] = 0.0f;
#pragma unroll
            for (int st = 0; st < 8; ++st) {
                const half8 kfr = __builtin_bit_cast(half8, kf[kt][st]);
                sc[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kfr, qh[st], sc[kt], 0, 0, 0);
                sc[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kfr, ql[st], sc[kt], 0, 0, 0);
            }
        }
        // V^T of the chunk into the wave's LDS rows (key k -> column swap_bits_2_3(k))
        {
            const uint32_t col = swap_bits_2_3(uint32_t(lane));
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const half8 v8 = __builtin_bit_cast(half8, vr[e]);
#pragma unroll
                for (int j = 0; j < 8; ++j) vw[8 * e + j][col] = v8[j];
            }
        }
        // scaled scores, masked in the chunks that reach past the block's first
        // query; the chunk maximum per query
        float mx = -INFINITY;
        if (kbase + kChunk - 1 <= pos0 + q0) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    sc[kt][i] *= scale;
                    mx = fmaxf(mx, sc[kt][i]);
                }
        } else {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t kpos = kbase + 32u * kt + 8u * (i >> 2) + 4u * h2 + (i & 3);
                    const float v = kpos <= qpos ? sc[kt][i] * scale : -INFINITY;
                    sc[kt][i] = v;
                    mx = fmaxf(mx, v);
                }
        }
        mx = xor_max<32>(mx);
        const float mnew = fmaxf(mrun, mx);
        const float mr = mnew == -INFINITY ? 0.0f : mnew;  // no position <= the query's yet: all weights 0
        const float alpha = expf(mrun - mr);              // mrun = -inf: 0
        float es = 0.0f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float e = expf(sc[kt][i] - mr);
                sc[kt][i] = e;
                es += e;
            }
        lrun = lrun * alpha + es;
        mrun = mnew;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[t][i] *= alpha;
        // the wave's own V^T rows: its LDS writes above complete before these reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                half8 ph, pl;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float pv = sc[kt][8 * st + j];
                    const _Float16 hi = static_cast<_Float16>(pv);
                    ph[j] = hi;
                    pl[j] = static_cast<_Float16>(pv - static_cast<float>(hi));
                }
                const uint32_t k0 = 32u * kt + 16u * st + 8u * h2;  // the lane's 8 keys, contiguous in LDS
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const half8 va = *reinterpret_cast<const half8*>(&vw[32 * t + l32][k0]);
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, ph, o[t], 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, pl, o[t], 0, 0, 0);
                }
            }
        // the next chunk's V^T overwrites these rows
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // the waves' states, combined in wave order: M = max m_w, f_w = e^(m_w - M),
    // out = sum_w f_w o_w / sum_w f_w l_w (waves without a chunk: m = -inf, f = 0)
    const float ltot = xor_sum<32>(lrun);
    __syncthreads();  // every wave is done with its V^T rows
    float* ot = reinterpret_cast<float*>(&vt[0][0][0]);  // [4][128 dims][32 queries]
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t d = 32u * t + 8u * (i >> 2) + 4u * h2 + (i & 3);
            ot[(w * kHeadDim + d) * 32 + l32] = o[t][i];
        }
    if (h2 == 0) {
        mw[w][l32] = mrun;
        lw[w][l32] = ltot;
    }
    __syncthreads();
    const uint32_t qq = uint32_t(tid) & 31u, d0 = (uint32_t(tid) >> 5) * 16u;
    float Mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < 4; ++v) Mx = fmaxf(Mx, mw[v][qq]);  // finite: chunk 0 holds position 0 <= every query's
    float f[4], L = 0.0f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        f[v] = expf(mw[v][qq] - Mx);
        L = __builtin_fmaf(lw[v][qq], f[v], L);
    }
    const float li = 1.0f / L;
    if (q0 + qq < M) {
        _Float16* dst = x + uint64_t(q0 + qq) * ldx + hq * kHeadDim + d0;
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            float acc = 0.0f;
#pragma unroll
            for (int v = 0; v < 4; ++v) acc = __builtin_fmaf(ot[(v * kHeadDim + d0 + d) * 32 + qq], f[v], acc);
            dst[d] = _Float16(acc * li);
        }
    }
}

// ------------------------------------------------------------------ host
namespace {

constexpr uint32_t kPfTargetWgs = 256;
thread_local int g_pf_attn_mfma = 1;  // 0: the VALU attention kernel (k_pf_attn)

// Tile of an M-row pass: every wave takes all of the pass's rows (MF blocks of
// 32) and 32 weight rows, so each weight is decoded once.  Plain products take
// 4 waves (128 weight rows; 256 workgroups of them ran 17 % faster than 128 of
// 8 waves, 3.7 against 4.3 us per super-block at 256 rows), split over K to
// about one workgroup per CU.  The fused gate/up, not split, takes 4 waves (64
// gate and 64 up rows) while that gives no CU a second workgroup, and 8 (128 and
// 128) for more columns and more than 64 rows; us, 4 waves / 8 waves:
//   columns x K     65 rows       100 rows      192 rows      256 rows
//    1024 x 2048  15.2 / 22.0   17.1 / 25.5   23.9 / 36.0   28.6 / 44.6
//    8192 x 3584  23.1 / 33.7   26.0 / 38.9   37.3 / 55.3   44.5 / 69.4
//   14336 x 4096  29.8 / 38.5   35.3 / 44.4   51.5 / 63.1   64.5 / 78.8
//   18944 x 3584  38.2 / 34.7   47.2 / 42.0   81.3 / 60.6  101.2 / 76.0  (64 rows: 32.0 / 30.9)
#define ARC_MM_ROWS(M, CALL) \
    ((M) > 192 ? CALL(8) : (M) > 128 ? CALL(6) : (M) > 96 ? CALL(4) : (M) > 64 ? CALL(3) : (M) > 32 ? CALL(2) : CALL(1))
constexpr uint32_t kMmCols = 128;  // weight rows per workgroup of a plain product

template <int FMT, int MF, int WN, bool SW>
hipError_t launch_mm_t(const PfGemm& p, uint32_t splits, hipStream_t st)
{
    constexpr uint32_t cols = SW ? 16u * WN : 32u * WN;
    hipLaunchKernelGGL((k_mm<FMT, MF, WN, SW>), dim3((p.N + cols - 1) / cols, splits), dim3(64 * WN), 0, st, p);
    return hipGetLastError();
}

hipError_t launch_gateup(const PfGemm& p, hipStream_t st)
{
#define ARC_MM_CALL(MF) (wide ? launch_mm_t<kFmtQ4, MF, (MF >= 3 ? 8 : 4), true>(p, 1, st) : launch_mm_t<kFmtQ4, MF, 4, true>(p, 1, st))
    const bool wide = p.N > 64u * kPfTargetWgs;
    return ARC_MM_ROWS(p.M, ARC_MM_CALL);
#undef ARC_MM_CALL
}

template <int FMT>
hipError_t launch_gemm_f(const PfGemm& p, uint32_t splits, hipStream_t st)
{
#define ARC_MM_CALL(MF) (launch_mm_t<FMT, MF, 4, false>(p, splits, st))
    return ARC_MM_ROWS(p.M, ARC_MM_CALL);
#undef ARC_MM_CALL
}

hipError_t launch_gemm(int qtype, const PfGemm& p, uint32_t splits, hipStream_t st)
{
    return qtype == kFmtQ4 ? launch_gemm_f<kFmtQ4>(p, splits, st) : launch_gemm_f<kFmtQ6P>(p, splits, st);
}

template <int VF, int MF>
hipError_t launch_qkv_t(const PfGemm& q, const PfGemm& k, const PfGemm& v, uint32_t splits, hipStream_t st)
{
    hipLaunchKernelGGL((k_mm_qkv<VF, MF, 4>), dim3(q.tiles + k.tiles + v.tiles, splits), dim3(256), 0, st, q, k, v);
    return hipGetLastError();
}

template <int VF>
hipError_t launch_qkv_f(const PfGemm& q, const PfGemm& k, const PfGemm& v, uint32_t splits, hipStream_t st)
{
#define ARC_MM_CALL(MF) (launch_qkv_t<VF, MF>(q, k, v, splits, st))
    return ARC_MM_ROWS(q.M, ARC_MM_CALL);
#undef ARC_MM_CALL
}

uint32_t mm_tiles(uint32_t N)
{
    return (N + kMmCols - 1) / kMmCols;
}

// The q|k|v launch: operands q, k, v of the columns [0, H), [H, H + kvd),
// [H + kvd, H + 2 kvd) of one partial buffer.
hipError_t launch_qkv(PfGemm q, const uint8_t* wk, const uint8_t* wv, int vtype, uint32_t kvd, uint32_t splits, hipStream_t st)
{
    const uint32_t H = q.N;
    q.tiles = mm_tiles(H);
    PfGemm k = q, v = q;
    k.w0 = wk;
    k.out = q.out + H;
    v.w0 = wv;
    v.out = q.out + H + kvd;
    k.N = v.N = kvd;
    k.tiles = v.tiles = mm_tiles(kvd);
    v.row_bytes = uint64_t(q.nb) * (vtype == kFmtQ4 ? kQ4Bytes : kQ6PBytes);
    return vtype == kFmtQ4 ? launch_qkv_f<kFmtQ4>(q, k, v, splits, st) : launch_qkv_f<kFmtQ6P>(q, k, v, splits, st);
}

// Split-K plan of a PLAIN projection of `gx` column tiles: the split count
// whose super-blocks per workgroup times rounds of workgroups over the CUs
// (one resident workgroup per CU) is smallest, the fewest splits (least
// partial traffic) among equals.
void split_plan(uint32_t gx, uint32_t nb, uint32_t& splits, uint32_t& bps)
{
    uint32_t best = ~0u;
    for (uint32_t want = 1; want <= nb; ++want) {
        const uint32_t b = (nb + want - 1) / want, sp = (nb + b - 1) / b;
        const uint32_t rounds = (gx * sp + kPfTargetWgs - 1) / kPfTargetWgs;
        if (b * rounds < best) {
            best = b * rounds;
            bps = b;
            splits = sp;
        }
    }
}

void gemm_plan(uint32_t N, uint32_t nb, uint32_t& splits, uint32_t& bps)
{
    split_plan(mm_tiles(N), nb, splits, bps);
}

void qkv_plan(uint32_t H, uint32_t kvd, uint32_t nb, uint32_t& splits, uint32_t& bps)
{
    split_plan(mm_tiles(H) + 2 * mm_tiles(kvd), nb, splits, bps);
}

// Partials of an N-column projection: splits x 256 rows x N floats.
uint64_t gemm_part_elems(uint32_t N, uint32_t nb)
{
    uint32_t sp, bps;
    gemm_plan(N, nb, sp, bps);
    return uint64_t(sp) * kPfMaxM * N;
}

template <int H>
void launch_attn_t(dim3 grid, hipStream_t st, const float* q, const _Float16* kc, const _Float16* vc, uint32_t kvh,
                   uint32_t pos0, float scale, _Float16* x, uint32_t ldx)
{
    hipLaunchKernelGGL(k_pf_attn<H>, grid, dim3(256), 0, st, q, kc, vc, kvh, pos0, scale, x, ldx);
}

void launch_attn(uint32_t hpk, dim3 grid, hipStream_t st, const float* q, const _Float16* kc, const _Float16* vc,
                 uint32_t kvh, uint32_t pos0, float scale, _Float16* x, uint32_t ldx)
{
    switch (hpk) {
    case 1: launch_attn_t<1>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    case 2: launch_attn_t<2>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    case 3: launch_attn_t<3>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    case 4: launch_attn_t<4>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    case 5: launch_attn_t<5>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    case 6: launch_attn_t<6>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    case 7: launch_attn_t<7>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    default: launch_attn_t<8>(grid, st, q, kc, vc, kvh, pos0, scale, x, ldx); break;
    }
}

}  // namespace

uint64_t prefill_part_elems(const arc_model_dims& d)
{
    // q|k|v (one launch), o, down: [split][256][columns] partials
    const uint32_t kvd = d.kv_heads * kHeadDim, nb = d.hidden / kQK;
    return std::max({gemm_part_elems(d.hidden + 2 * kvd, nb), gemm_part_elems(d.hidden, nb),
                     gemm_part_elems(d.hidden, d.ffn / kQK)});
}

int run_prefill(arc_session* S, const uint32_t* tokens, uint32_t n, uint32_t pos0, bool logits)
{
    int rc = ARC_OK;
    PrefillBufs* pf = &S->pf;
    const arc_model* Mdl = S->model;
    const arc_model_dims& d = Mdl->dims;
    const uint32_t H = d.hidden, F = d.ffn, kvd = d.kv_heads * kHeadDim, hpk = d.q_heads / d.kv_heads;
    const uint32_t passes = (n + kPfMaxM - 1) / kPfMaxM;
    if (passes > pf->host_slots)  // the caller keeps pos0 + n within max_ctx
        return set_error(ARC_ERR_INVALID_ARGUMENT, "prompt of %u tokens exceeds the session's %u positions", n,
                         S->max_ctx);
    hipStream_t st = S->stream;
    uint32_t nk = 0;
    auto chk = [&](hipError_t e, const char* what) {
        ++nk;
        return check_hip(e, what);
    };
    const float scale = 1.0f / std::sqrt(float(kHeadDim));
    for (uint32_t pass = 0; pass < passes; ++pass) {
        const uint32_t base = pass * kPfMaxM, M = std::min(uint32_t(kPfMaxM), n - base), p0 = pos0 + base;
        uint32_t* ht = pf->host_tokens + size_t(pass) * kPfMaxM;
        std::memcpy(ht, tokens + base, M * sizeof(uint32_t));
        if ((rc = check_hip(hipMemcpyAsync(pf->tokens, ht, M * sizeof(uint32_t), hipMemcpyHostToDevice, st), "tokens")))
            return rc;
        // the LM head of the last row leaves position p0 + M in the control block
        S->host_ctl[1 + pass] = DecodeCtl{p0 + M - 1, 0u, 0u, 0u, 0u};
        if ((rc = check_hip(hipMemcpyAsync(S->ctl, &S->host_ctl[1 + pass], sizeof(DecodeCtl), hipMemcpyHostToDevice, st),
                            "ctl upload")))
            return rc;
        hipLaunchKernelGGL(k_pf_embed, dim3(H / kQK, M), dim3(kQK), 0, st, Mdl->emb, H / kQK, pf->tokens, pf->h);
        if ((rc = chk(hipGetLastError(), "prefill embed"))) return rc;
        for (uint32_t l = 0; l < d.layers; ++l) {
            const Layer& L = Mdl->layers[l];
            _Float16* kc = S->kcache + uint64_t(l) * S->max_ctx * kvd;
            _Float16* vc = S->vcache + uint64_t(l) * S->max_ctx * kvd;
            if (l == 0) {  // later layers: fused into the previous layer's down residual
                hipLaunchKernelGGL(k_pf_rmsnorm, dim3(M), dim3(256), 0, st, pf->h, H, L.attn_norm, d.rms_eps, pf->x, H);
                if ((rc = chk(hipGetLastError(), "attn norm"))) return rc;
            }

            PfGemm g{};
            g.M = M;
            g.mpad = kPfMaxM;
            g.x = pf->x;
            g.ldx = H;
            g.nb = H / kQK;
            g.out = pf->part;
            uint32_t sp, bps;
            // q | k | v in one launch, partials [split][mpad][H | kvd | kvd]
            const uint32_t nqkv = H + 2 * kvd;
            g.w0 = L.q;
            g.row_bytes = uint64_t(g.nb) * kQ4Bytes;
            g.N = H;
            g.ldo = nqkv;
            qkv_plan(H, kvd, g.nb, sp, bps);
            g.bps = bps;
            if ((rc = chk(launch_qkv(g, L.k, L.v, L.v_type, kvd, sp, st), "q/k/v projection"))) return rc;
            hipLaunchKernelGGL(k_pf_qkv_epi, dim3((nqkv / 2 + 255) / 256, M), dim3(256), 0, st, pf->part, sp,
                               uint32_t(kPfMaxM), H, kvd, L.qb, L.kb, L.vb, S->rope, p0, pf->q, kc, vc);
            if ((rc = chk(hipGetLastError(), "q/k/v epilogue"))) return rc;
            // attention -> x
            if (g_pf_attn_mfma)
                hipLaunchKernelGGL(k_pf_attn_mf, dim3((M + 31) / 32, d.q_heads), dim3(256), 0, st, pf->q, kc, vc,
                                   d.kv_heads, hpk, p0, M, S->max_ctx, scale, pf->x, H);
            else
                launch_attn(hpk, dim3(M, d.kv_heads), st, pf->q, kc, vc, d.kv_heads, p0, scale, pf->x, H);
            if ((rc = chk(hipGetLastError(), "prefill attention"))) return rc;
            // o + residual + ffn norm
            g.w0 = L.o;
            g.row_bytes = uint64_t(g.nb) * kQ4Bytes;
            g.N = H;
            g.ldo = H;
            gemm_plan(g.N, g.nb, sp, bps);
            g.bps = bps;
            if ((rc = chk(launch_gemm(kFmtQ4, g, sp, st), "o projection"))) return rc;
            launch_res_norm<true>(M, st, pf->part, sp, uint32_t(kPfMaxM), H, pf->h, pf->h, L.ffn_norm, d.rms_eps, pf->x, H);
            if ((rc = chk(hipGetLastError(), "o residual + ffn norm"))) return rc;
            // gate/up + SwiGLU -> xs
            PfGemm u = g;
            u.w0 = L.gate;
            u.w1 = L.up;
            u.row_bytes = uint64_t(g.nb) * kQ4Bytes;
            u.N = F;
            u.bps = g.nb;
            u.s = pf->xs;
            u.lds_out = F;
            if ((rc = chk(launch_gateup(u, st), "gate/up"))) return rc;
            // down + residual (+ the next layer's attention norm)
            PfGemm dn = g;
            dn.x = pf->xs;
            dn.ldx = F;
            dn.nb = F / kQK;
            dn.w0 = L.down;
            dn.row_bytes = uint64_t(dn.nb) * (L.down_type == kFmtQ4 ? kQ4Bytes : kQ6PBytes);
            dn.N = H;
            dn.ldo = H;
            gemm_plan(dn.N, dn.nb, sp, bps);
            dn.bps = bps;
            rc = chk(launch_gemm(L.down_type == kFmtQ4 ? kFmtQ4 : kFmtQ6P, dn, sp, st), "down projection");
            if (rc) return rc;
            if (l + 1 < d.layers) {
                launch_res_norm<true>(M, st, pf->part, sp, uint32_t(kPfMaxM), H, pf->h, pf->h, Mdl->layers[l + 1].attn_norm,
                                      d.rms_eps, pf->x, H);
            } else {
                launch_res_norm<false>(M, st, pf->part, sp, uint32_t(kPfMaxM), H, pf->h, pf->h, nullptr, 0.0f, nullptr, 0u);
            }
            if ((rc = chk(hipGetLastError(), "down residual"))) return rc;
        }
        if (pass + 1 == passes) {
            if ((rc = launch_lm_head(S, pf->h + uint64_t(M - 1) * H, logits, st))) return rc;
            nk += 1;
        }
    }
    S->prefill_kernels = nk;
    return ARC_OK;
}

}  // namespace arc

// ------------------------------------ standalone prompt-pass projections
namespace arc {
namespace {

struct PfWorkspace {
    size_t x, part, bytes;
};

// X staging (256 rows of K fp16, see pf_stage_x) and the split partials of the N
// x K projection's plan.
PfWorkspace pf_workspace(uint32_t N, uint32_t K)
{
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    PfWorkspace w{};
    w.x = 0;
    w.part = up(size_t(kPfMaxM) * K * sizeof(_Float16));
    w.bytes = w.part + up(size_t(gemm_part_elems(N, K / kQK)) * sizeof(float));
    return w;
}

int pf_check(const void* w, uint32_t N, uint32_t K, const uint16_t* x, uint32_t M, const void* out, const void* ws)
{
    if (!w || !x || !out || !ws) return set_error(ARC_ERR_INVALID_ARGUMENT, "null argument");
    if (N == 0 || K == 0 || K % kQK || M == 0 || M > uint32_t(kPfMaxM))
        return set_error(ARC_ERR_INVALID_ARGUMENT, "bad shape N=%u K=%u M=%u (K a multiple of 256, 1 <= M <= %d)", N, K,
                         M, kPfMaxM);
    if (N > uint32_t(kResCols) * 1024u) return set_error(ARC_ERR_UNSUPPORTED, "N must be <= %d", kResCols * 1024);
    // the tiles' 32-bit offsets: M rows of X (2 M K bytes) and 32 weight rows (212
    // bytes for 256 columns at most)
    if (uint64_t(M) * K >= (uint64_t(1) << 31) || K > (1u << 27))
        return set_error(ARC_ERR_UNSUPPORTED, "K=%u: M * K must be below 2^31 and K at most 2^27", K);
    if (reinterpret_cast<uintptr_t>(w) & 15u) return set_error(ARC_ERR_INVALID_ARGUMENT, "weights not 16-byte aligned");
    if (reinterpret_cast<uintptr_t>(ws) & 255u)
        return set_error(ARC_ERR_INVALID_ARGUMENT, "workspace must be 256-byte aligned");
    return ARC_OK;
}

// The GEMM's X: the given rows, or a copy of them in the workspace where they do
// not start at a 16-byte boundary (the tiles read 16 bytes at a time) or share
// memory with the `out_bytes` at `out` that the GEMM launch writes (a workgroup
// that has finished stores while others still read X).
int pf_stage_x(uint8_t* ws, const PfWorkspace& w, const uint16_t* x, uint32_t M, uint32_t K, const void* out, size_t out_bytes,
               hipStream_t st, PfGemm& g)
{
    const size_t bytes = size_t(M) * K * sizeof(_Float16);
    const uintptr_t xa = reinterpret_cast<uintptr_t>(x), oa = reinterpret_cast<uintptr_t>(out);
    g.ldx = K;
    g.x = reinterpret_cast<const _Float16*>(x);
    if ((xa & 15u) == 0 && (xa + bytes <= oa || oa + out_bytes <= xa)) return ARC_OK;
    g.x = reinterpret_cast<const _Float16*>(ws + w.x);
    return check_hip(hipMemcpyAsync(ws + w.x, x, bytes, hipMemcpyDeviceToDevice, st), "x staging");
}

// y[m][c] = sum over the splits of part[s][m][c], in split order.
int pf_reduce(const float* part, uint32_t splits, uint32_t M, uint32_t N, float* y, hipStream_t st)
{
    launch_res_norm<false>(M, st, part, splits, uint32_t(kPfMaxM), N, nullptr, y, nullptr, 0.0f, nullptr,
                           0u);
    return check_hip(hipGetLastError(), "split reduction");
}

}  // namespace
}  // namespace arc

using namespace arc;

extern "C" {

int arc_tune_prefill_attention(int mfma)
{
    if (mfma != 0 && mfma != 1) return set_error(ARC_ERR_INVALID_ARGUMENT, "prefill attention: 0 (VALU) or 1 (MFMA)");
    g_pf_attn_mfma = mfma;
    return ARC_OK;
}

size_t arc_prefill_gemm_workspace_bytes(uint32_t N, uint32_t K)
{
    if (N == 0 || K == 0 || K % kQK) return 0;
    return pf_workspace(N, K).bytes;
}

int arc_prefill_gemm(int qtype, const void* w, uint32_t N, uint32_t K, const uint16_t* x, uint32_t M, float* y,
                     void* workspace, arc_stream_t stream)
{
    int rc = pf_check(w, N, K, x, M, y, workspace);
    if (rc) return rc;
    if (qtype != kFmtQ4 && qtype != kFmtQ6P)
        return set_error(ARC_ERR_UNSUPPORTED, "the prompt-pass GEMM takes Q4_K or padded Q6_K (qtype %d)", qtype);
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    const PfWorkspace pw = pf_workspace(N, K);
    PfGemm g{};
    if ((rc = pf_stage_x(ws, pw, x, M, K, ws + pw.part, pw.bytes - pw.part, st, g))) return rc;
    g.M = M;
    g.mpad = kPfMaxM;
    g.nb = K / kQK;
    g.out = reinterpret_cast<float*>(ws + pw.part);
    g.w0 = static_cast<const uint8_t*>(w);
    g.row_bytes = uint64_t(g.nb) * (qtype == kFmtQ4 ? kQ4Bytes : kQ6PBytes);
    g.N = N;
    g.ldo = N;
    uint32_t sp;
    gemm_plan(N, g.nb, sp, g.bps);
    if ((rc = check_hip(launch_gemm(qtype, g, sp, st), "prompt-pass GEMM"))) return rc;
    return pf_reduce(g.out, sp, M, N, y, st);
}

int arc_prefill_gateup(const void* w_gate, const void* w_up, uint32_t N, uint32_t K, const uint16_t* x, uint32_t M,
                       uint16_t* s, void* workspace, arc_stream_t stream)
{
    int rc = pf_check(w_gate, N, K, x, M, s, workspace);
    if (rc) return rc;
    if (!w_up || (reinterpret_cast<uintptr_t>(w_up) & 15u))
        return set_error(ARC_ERR_INVALID_ARGUMENT, "up weights null or not 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    const PfWorkspace pw = pf_workspace(N, K);
    PfGemm u{};
    if ((rc = pf_stage_x(ws, pw, x, M, K, s, size_t(M) * N * sizeof(_Float16), st, u))) return rc;
    u.M = M;
    u.mpad = kPfMaxM;
    u.nb = K / kQK;
    u.w0 = static_cast<const uint8_t*>(w_gate);
    u.w1 = static_cast<const uint8_t*>(w_up);
    u.row_bytes = uint64_t(u.nb) * kQ4Bytes;
    u.N = N;
    u.bps = u.nb;
    u.s = reinterpret_cast<_Float16*>(s);
    u.lds_out = N;
    return check_hip(launch_gateup(u, st), "prompt-pass gate/up");
}

int arc_prefill_attention(const float* q, const void* kc, const void* vc, uint32_t kv_heads, uint32_t hpk,
                          uint32_t max_ctx, uint32_t pos0, uint32_t M, uint16_t* x, uint32_t ldx, int mfma,
                          arc_stream_t stream)
{
    if (!q || !kc || !vc || !x) return set_error(ARC_ERR_INVALID_ARGUMENT, "null argument");
    if (kv_heads == 0 || kv_heads > 64 || hpk == 0 || hpk > uint32_t(kMaxHpk))
        return set_error(ARC_ERR_UNSUPPORTED, "prefill attention supports 1..64 kv heads and 1..%d query heads per kv "
                         "head", kMaxHpk);
    if (M == 0 || max_ctx == 0 || max_ctx > uint32_t(kMaxChunks * kChunk) || uint64_t(pos0) + M > max_ctx)
        return set_error(ARC_ERR_INVALID_ARGUMENT, "bad rows: pos0 %u + M %u > max_ctx %u (at most %d)", pos0, M,
                         max_ctx, kMaxChunks * kChunk);
    const uint32_t hidden = kv_heads * hpk * kHeadDim;
    if (ldx < hidden) return set_error(ARC_ERR_INVALID_ARGUMENT, "ldx %u < %u", ldx, hidden);
    const uintptr_t al = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kc) |
                         reinterpret_cast<uintptr_t>(vc);
    if (al & 15u) return set_error(ARC_ERR_INVALID_ARGUMENT, "q, kc and vc must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const _Float16* k16 = static_cast<const _Float16*>(kc);
    const _Float16* v16 = static_cast<const _Float16*>(vc);
    _Float16* x16 = reinterpret_cast<_Float16*>(x);
    const float scale = 1.0f / std::sqrt(float(kHeadDim));
    if (mfma)
        hipLaunchKernelGGL(k_pf_attn_mf, dim3((M + 31) / 32, kv_heads * hpk), dim3(256), 0, st, q, k16, v16, kv_heads,
                           hpk, pos0, M, max_ctx, scale, x16, ldx);
    else
        launch_attn(hpk, dim3(M, kv_heads), st, q, k16, v16, kv_heads, pos0, scale, x16, ldx);
    return check_hip(hipGetLastError(), "prefill attention");
}

int arc_prefill_qkv(const void* wq, const void* wk, const void* wv, int v_qtype, uint32_t H, uint32_t kvd, uint32_t K,
                    const uint16_t* x, uint32_t M, float* y, void* workspace, arc_stream_t stream)
{
    const uint32_t N = H + 2 * kvd;
    int rc = pf_check(wq, N, K, x, M, y, workspace);
    if (rc) return rc;
    if (!wk || !wv || ((reinterpret_cast<uintptr_t>(wk) | reinterpret_cast<uintptr_t>(wv)) & 15u))
        return set_error(ARC_ERR_INVALID_ARGUMENT, "k or v weights null or not 16-byte aligned");
    if (v_qtype != kFmtQ4 && v_qtype != kFmtQ6P)
        return set_error(ARC_ERR_UNSUPPORTED, "v must be Q4_K or padded Q6_K (qtype %d)", v_qtype);
    if (H == 0 || kvd == 0 || H % 128 || kvd % 128)
        return set_error(ARC_ERR_INVALID_ARGUMENT, "H and kvd must be nonzero multiples of 128");
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    const PfWorkspace pw = pf_workspace(N, K);
    // as run_prefill: partials [split][mpad][H | kvd | kvd]
    PfGemm g{};
    if ((rc = pf_stage_x(ws, pw, x, M, K, ws + pw.part, pw.bytes - pw.part, st, g))) return rc;
    g.M = M;
    g.mpad = kPfMaxM;
    g.nb = K / kQK;
    g.out = reinterpret_cast<float*>(ws + pw.part);
    g.w0 = static_cast<const uint8_t*>(wq);
    g.row_bytes = uint64_t(g.nb) * kQ4Bytes;
    g.N = H;
    g.ldo = N;
    uint32_t sp;
    qkv_plan(H, kvd, g.nb, sp, g.bps);
    rc = check_hip(launch_qkv(g, static_cast<const uint8_t*>(wk), static_cast<const uint8_t*>(wv), v_qtype, kvd, sp, st),
                   "prompt-pass q/k/v");
    if (rc) return rc;
    return pf_reduce(g.out, sp, M, N, y, st);
}

}  // extern "C"
