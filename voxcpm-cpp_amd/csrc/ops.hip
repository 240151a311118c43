// ops.hip -- the non-matmul pieces of the MiniCPM4 block on gfx950:
// RMSNorm (+ residual, + Q8_0 activation quantization), NEOX RoPE with the
// f16 KV-cache append, softmax attention over the f16 cache, SwiGLU (+ Q8_0
// quantization).  Every rounding step follows the reference graph
// (src/minicpm4.c) as restated by the oracle; contraction is off, so each
// a*b+c below rounds twice like the reference's scalar code.
#include "vxm_ops.h"

// ---------------------------------------------------------------------------
// block-wide reductions (blockDim.x == 256)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double block_sum_f64(double v, double *sh) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < (int)(blockDim.x >> 6); i++) t += sh[i];
    return t;
}

// The same for sums of squares in a tree order (each row of 16 lanes on DPP: xor 1,
// xor 2, half mirror, mirror; the wave's four rows read back as scalars).  Every lane
// of the block must be active.  The squares of BF16 values have 16 significant
// bits (of fp32 values, 24), so while a row's squares span less than about 2^26
// (values within 2^13; fp32 values within 2^9) every partial sum of up to 2^11 of
// them is exact in double and any order gives ggml's sequential double.  Beyond
// that the tree and the sequential order can round the double differently, and
// (float)(sum / n) can then differ by one ulp.
__device__ __forceinline__ double block_sum_exact_f64(double v, double *sh) {
    auto dpp = [](double x, auto ctrl) {
        const long long b = __double_as_longlong(x);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, decltype(ctrl)::value, 0xF, 0xF, false);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), decltype(ctrl)::value, 0xF, 0xF, false);
        return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
    };
    v = v + dpp(v, std::integral_constant<int, 0xB1>{});
    v = v + dpp(v, std::integral_constant<int, 0x4E>{});
    v = v + dpp(v, std::integral_constant<int, 0x141>{});
    v = v + dpp(v, std::integral_constant<int, 0x140>{});
    const long long b = __double_as_longlong(v);
    double w = 0.0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, 16 * r);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), 16 * r);
        w += __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    }
    const int wv = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[wv] = w;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < (int)(blockDim.x >> 6); i++) t += sh[i];
    return t;
}

__device__ __forceinline__ float block_max_f32(float v, float *sh) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    float t = sh[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); i++) t = fmaxf(t, sh[i]);
    return t;
}

// ---------------------------------------------------------------------------
// [h = bf16(h + scale * bf16(delta))]; y = vcpm_rms_norm(h) (src/minicpm4.c:132-152):
// ggml_rms_norm (sum of fp32 squares in double, mean = (float)(sum/n),
// scale = 1/sqrtf(mean + eps)), BF16, * gain, BF16.  Outputs y (fp32, if
// non-null) and its Q8_0 quantization (xq/xd, if non-null).
// One workgroup per row: 128 threads for n <= 1024, else 256; n % 8 == 0 and
// n <= 8 * 256 * VXM_NORM_CHUNKS.
// ---------------------------------------------------------------------------
#define VXM_NORM_CHUNKS 4
__global__ __launch_bounds__(256) void k_rmsnorm(float *__restrict__ h, const vxm_parts delta, float res_scale,
                                                 const float *__restrict__ gain, int n, float eps,
                                                 float *__restrict__ y, int8_t *__restrict__ xq,
                                                 uint16_t *__restrict__ xd, int variant, int seg_rows,
                                                 int seg_stride) {
    __shared__ double shd[4];
    // output row `row`; its h / delta row: seg_rows rows of every seg_stride (the identity
    // when seg_rows == seg_stride)
    const int row = blockIdx.x;
    const int64_t hrow = (int64_t)(row / seg_rows) * seg_stride + row % seg_rows;
    float *hr = h + hrow * n;
    const float *dr = delta.p ? delta.p + hrow * n : nullptr;
    float v[VXM_NORM_CHUNKS][8];
    // the gain, fetched with the row (it is needed right after the reduction)
    float4 gl[VXM_NORM_CHUNKS][2];
#pragma unroll
    for (int c = 0; c < VXM_NORM_CHUNKS; c++) {
        const int base = (c * (int)blockDim.x + threadIdx.x) * 8;
        if (gain && base < n) {
            gl[c][0] = *(const float4 *)(gain + base);
            gl[c][1] = *(const float4 *)(gain + base + 4);
        } else {
            gl[c][0] = gl[c][1] = make_float4(1, 1, 1, 1);
        }
    }
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < VXM_NORM_CHUNKS; c++) {
        const int base = (c * (int)blockDim.x + threadIdx.x) * 8;
        if (base < n) {
            float4 a = *(const float4 *)(hr + base), b = *(const float4 *)(hr + base + 4);
            v[c][0] = a.x; v[c][1] = a.y; v[c][2] = a.z; v[c][3] = a.w;
            v[c][4] = b.x; v[c][5] = b.y; v[c][6] = b.z; v[c][7] = b.w;
            if (dr) {
                // K-split slices: all loads in flight, then added in order
                float4 ps[VXM_MAX_PARTS], qs[VXM_MAX_PARTS];
#pragma unroll
                for (int z = 0; z < VXM_MAX_PARTS; z++)
                    if (z < delta.n) {
                        ps[z] = *(const float4 *)(dr + z * delta.stride + base);
                        qs[z] = *(const float4 *)(dr + z * delta.stride + base + 4);
                    }
                float4 p = ps[0], q = qs[0];
#pragma unroll
                for (int z = 1; z < VXM_MAX_PARTS; z++)
                    if (z < delta.n) {
                        p.x = p.x + ps[z].x; p.y = p.y + ps[z].y; p.z = p.z + ps[z].z; p.w = p.w + ps[z].w;
                        q.x = q.x + qs[z].x; q.y = q.y + qs[z].y; q.z = q.z + qs[z].z; q.w = q.w + qs[z].w;
                    }
                float dd[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    float o = vxm_bf16(dd[i]);
                    if (res_scale != 1.0f) o = o * res_scale;
                    v[c][i] = vxm_bf16(v[c][i] + o);
                }
                *(float4 *)(hr + base) = make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
                *(float4 *)(hr + base + 4) = make_float4(v[c][4], v[c][5], v[c][6], v[c][7]);
            }
#pragma unroll
            for (int i = 0; i < 8; i++) ss += (double)(v[c][i] * v[c][i]);
        }
    }
    const double tot = block_sum_exact_f64(ss, shd);
    if (!y && !xq) return;
    const float mean = (float)(tot / (double)n);
    const float sc = __fdiv_rn(1.0f, __fsqrt_rn(mean + eps));
#pragma unroll
    for (int c = 0; c < VXM_NORM_CHUNKS; c++) {
        const int base = (c * (int)blockDim.x + threadIdx.x) * 8;
        if (base >= n) continue;   // whole 32-blocks live in 4 consecutive lanes: n % 32 == 0
        float o[8];
        const float4 g0 = gl[c][0], g1 = gl[c][1];
        const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float t = vxm_bf16(v[c][i] * sc);
            o[i] = gain ? vxm_bf16(t * g[i]) : t;
        }
        if (y) {
            float *yr = y + (int64_t)row * n + base;
            *(float4 *)yr = make_float4(o[0], o[1], o[2], o[3]);
            *(float4 *)(yr + 4) = make_float4(o[4], o[5], o[6], o[7]);
        }
        if (xq) {
            const int64_t e = (int64_t)row * n + base;
            quant_block_4lanes(o, variant, xq + e, xd + e / 32, (threadIdx.x & 3) == 0);
        }
    }
}

int vxm_launch_rmsnorm(vxm_ctx *ctx, float *h, vxm_parts delta, float res_scale, const float *gain,
                       int64_t rows, int64_t n, float eps, float *y, int8_t *xq, uint16_t *xd, int variant,
                       int seg_rows, int seg_stride) {
    if (rows <= 0) return VXM_OK;
    if (seg_rows <= 0) seg_rows = seg_stride = (int)rows;
    if (seg_stride < seg_rows) return vxm_fail(ctx, VXM_ERR_INVALID_ARG, "rms_norm: segment stride below its rows");
    if (n % 32 != 0 || n > 8 * 256 * VXM_NORM_CHUNKS)
        return vxm_fail(ctx, VXM_ERR_INVALID_ARG, "rms_norm: n=%lld must be a multiple of 32 and <= %d",
                        (long long)n, 8 * 256 * VXM_NORM_CHUNKS);
    // rows of up to 1024 values fit 128 threads (8 values each): two waves reduce faster than four
    const unsigned threads = n <= 8 * 128 ? 128 : 256;
    hipLaunchKernelGGL(k_rmsnorm, dim3((unsigned)rows), dim3(threads), 0, ctx->stream, h, delta, res_scale, gain,
                       (int)n, eps, y, xq, xd, variant, seg_rows, seg_stride);
    VXM_CHECK_LAUNCH(ctx);
    return VXM_OK;
}

// ---------------------------------------------------------------------------
// Q/K/V post-processing of vcpm_attention (src/minicpm4.c:270-320): BF16 of
// the projections, NEOX RoPE (pair (i, i+hd/2) rotated by the angle of
// ggml_rope_ext, theta_i / ff_i with theta_0 = pos, theta_{i+1} = theta_i *
// theta_scale; BF16), K and V appended to the f16 cache.  cs holds the
// host-computed (cos, sin) of every (position, pair): [position][hd/2].  qkv: raw projections [M][qd + 2*kvd].
// Tokens come in segments of S (one per CFG branch); token t has position
// pos0 + t % S and segment t / S, whose cache starts at seg * seg_stride.
// One thread per pair of neighbouring projection values (a rotary pair of a q or
// k head, which are stored pair-interleaved: row 2i is dim i, row 2i + 1 dim
// i + hd / 2; two neighbouring dims of a v head).  Latency-bound: a thread issues
// the loads of all K-split slices at once and adds them in slice order, and the
// pairs of one token are spread over workgroups.  (One workgroup per token that
// walked its pairs and read the slices one after another took 15.0 us at 5 and
// at 24 tokens of 16 / 2 x 128 heads with 8 slices.)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_rope_kv(const vxm_parts qkv, int nh, int nkv, int hd,
                                                 int pos0, int S, const float2 *__restrict__ cs,
                                                 int no_rope, float *__restrict__ q_out, uint16_t *__restrict__ kc,
                                                 uint16_t *__restrict__ vc, int cap, int64_t seg_stride,
                                                 int cache_pos0) {
    const int t = blockIdx.x, half = hd / 2, idx = blockIdx.y * blockDim.x + threadIdx.x;
    if (idx >= (nh + 2 * nkv) * half) return;
    const int head = idx / half, i = idx % half;   // q heads, then k heads, then v heads
    const int seg = t / S, ti = t % S;
    // (nh + 2 nkv) hd and hd are even: the pair is 8-byte aligned
    const float *src = qkv.p + ((int64_t)t * (nh + 2 * nkv) + head) * hd + 2 * i;
    float2 part[VXM_MAX_PARTS];
#pragma unroll
    for (int z = 0; z < VXM_MAX_PARTS; z++)
        if (z < qkv.n) part[z] = *(const float2 *)(src + z * qkv.stride);
    const bool rot = !no_rope && head < nh + nkv;
    float2 r = make_float2(1.0f, 0.0f);
    if (rot) r = cs[(int64_t)(pos0 + ti) * half + i];
    float2 x = part[0];
#pragma unroll
    for (int z = 1; z < VXM_MAX_PARTS; z++)
        if (z < qkv.n) {
            x.x = x.x + part[z].x;
            x.y = x.y + part[z].y;
        }
    const float x0 = vxm_bf16(x.x), x1 = vxm_bf16(x.y);
    float y0 = x0, y1 = x1;
    if (rot) {
        y0 = vxm_bf16(x0 * r.x - x1 * r.y);
        y1 = vxm_bf16(x0 * r.y + x1 * r.x);
    }
    if (head < nh) {
        float *qo = q_out + ((int64_t)t * nh + head) * hd;
        qo[i] = y0;
        qo[i + half] = y1;
        return;
    }
    const bool is_k = head < nh + nkv;
    const int kh = is_k ? head - nh : head - nh - nkv;
    uint16_t *dst = (is_k ? kc : vc) + seg * seg_stride + ((int64_t)kh * cap + cache_pos0 + ti) * hd;
    if (is_k) {
        dst[i] = vxm_f2h(y0);
        dst[i + half] = vxm_f2h(y1);
    } else {
        *(uint32_t *)(dst + 2 * i) = (uint32_t)vxm_f2h(y0) | ((uint32_t)vxm_f2h(y1) << 16);
    }
}

int vxm_launch_rope_kv(vxm_ctx *ctx, vxm_parts qkv, int64_t M, int nh, int nkv, int hd, int pos0, int S,
                       const float2 *cs, int cs_rows, int no_rope, float *q_out, uint16_t *kc,
                       uint16_t *vc, int cap, int64_t seg_stride, int cache_pos0) {
    if (M <= 0) return VXM_OK;
    if (!no_rope && (!cs || pos0 + std::min<int64_t>(M, S) > cs_rows))
        return vxm_fail(ctx, VXM_ERR_BACKEND, "rope: table holds %d positions, %lld needed", cs_rows,
                        (long long)(pos0 + std::min<int64_t>(M, S)));
    const int pairs = (nh + 2 * nkv) * (hd / 2);
    hipLaunchKernelGGL(k_rope_kv, dim3((unsigned)M, (unsigned)((pairs + 255) / 256)), dim3(256), 0, ctx->stream, qkv,
                       nh, nkv, hd, pos0, S, cs, no_rope, q_out, kc, vc, cap, seg_stride, cache_pos0);
    VXM_CHECK_LAUNCH(ctx);
    return VXM_OK;
}

// ---------------------------------------------------------------------------
// gqa_group_attn (src/minicpm4.c:232-248) for one (token, query head):
// s_j = (k_j . q) * (1/sqrt(hd)); p = softmax (sum in double, scaled by
// (float)(1/sum)); out = sum_j p_j v_j.  Query head h reads kv head
// h / (nh / nkv).  Causal: token t of a segment sees cache rows
// [0, kv_base + t]; non-causal: rows [0, S).  Scores live in LDS (kv_len <= cap).
// Latency-bound (few tokens, 16 heads): a thread forms whole scores, so it loads
// its key row 16 bytes at a time, eight loads in flight (hd % 8 == 0; 2 bytes at a
// time otherwise), and P V keeps eight V loads in flight; the order of every sum
// is the scalar loop's.  xq != nullptr (hd % 32 == 0): the head's output goes out
// as Q8_0 blocks instead of fp32, without a launch of its own.
// ---------------------------------------------------------------------------
template <bool VEC>
__global__ __launch_bounds__(256) void k_attention(const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                                   const uint16_t *__restrict__ vc, float *__restrict__ out, int nh,
                                                   int nkv, int hd, int cap, int64_t seg_stride, int S,
                                                   int kv_base, int causal, int8_t *__restrict__ xq,
                                                   uint16_t *__restrict__ xd, int variant) {
    extern __shared__ __align__(16) float lds[];
    __shared__ float red[8];
    __shared__ double redd[4];
    const int h = blockIdx.x, t = blockIdx.y;
    const int seg = t / S, ti = t % S;
    const int kvh = h / (nh / nkv);
    const int kv_len = causal ? kv_base + ti + 1 : S;
    const uint16_t *kb = kc + seg * seg_stride + (int64_t)kvh * cap * hd;
    const uint16_t *vb = vc + seg * seg_stride + (int64_t)kvh * cap * hd;
    float *sq = lds;              // [hd]
    float *part = lds + hd;       // [256]
    float *sc = part + 256;       // [kv_len]
    const float *qr = q + (int64_t)t * nh * hd + h * hd;
    for (int d = threadIdx.x; d < hd; d += blockDim.x) sq[d] = qr[d];
    __syncthreads();
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn((float)hd));
    float mx = -INFINITY;
    for (int j = threadIdx.x; j < kv_len; j += blockDim.x) {
        const uint16_t *kr = kb + (int64_t)j * hd;
        float s = 0.0f;
        if (VEC) {
            for (int d0 = 0; d0 < hd; d0 += 64) {
                uint4 kv[8];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (d0 + 8 * u < hd) kv[u] = *(const uint4 *)(kr + d0 + 8 * u);
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    if (d0 + 8 * u >= hd) break;
                    const uint32_t w[4] = {kv[u].x, kv[u].y, kv[u].z, kv[u].w};
                    const float4 qa = *(const float4 *)(sq + d0 + 8 * u), qb = *(const float4 *)(sq + d0 + 8 * u + 4);
                    const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        s += vxm_h2f((uint16_t)(e & 1 ? w[e >> 1] >> 16 : w[e >> 1] & 0xffffu)) * qv[e];
                }
            }
        } else {
            for (int d = 0; d < hd; d++) s += vxm_h2f(kr[d]) * sq[d];
        }
        s = s * scale;
        sc[j] = s;
        mx = fmaxf(mx, s);
    }
    mx = block_max_f32(mx, red);
    double sum = 0.0;
    for (int j = threadIdx.x; j < kv_len; j += blockDim.x) {
        const float e = expf(sc[j] - mx);
        sc[j] = e;
        sum += (double)e;
    }
    sum = block_sum_f64(sum, redd);
    const float inv = (float)(1.0 / sum);
    for (int j = threadIdx.x; j < kv_len; j += blockDim.x) sc[j] = sc[j] * inv;
    __syncthreads();
    // out[d] = sum_j v[j][d] * p_j: thread (sl, d) sums a contiguous j-slice,
    // slices are added in order (hd <= 256, checked by the launcher).
    const int slices = blockDim.x / hd;
    const int d = threadIdx.x % hd, sl = threadIdx.x / hd;
    float acc = 0.0f;
    if (sl < slices) {
        const int jper = (kv_len + slices - 1) / slices;
        const int j0 = sl * jper, j1 = min(kv_len, j0 + jper);
        int j = j0;
        for (; j + 8 <= j1; j += 8) {
            uint16_t v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = vb[(int64_t)(j + u) * hd + d];
#pragma unroll
            for (int u = 0; u < 8; u++) acc += vxm_h2f(v[u]) * sc[j + u];
        }
        for (; j < j1; j++) acc += vxm_h2f(vb[(int64_t)j * hd + d]) * sc[j];
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    float tot = 0.0f;
    if (sl == 0) {
        for (int s2 = 0; s2 < slices; s2++) tot += part[s2 * hd + d];
        if (!xq) out[(int64_t)t * nh * hd + h * hd + d] = tot;
    }
    if (!xq) return;
    if (sl == 0) sq[d] = tot;   // the query row is done with
    __syncthreads();
    if ((int)threadIdx.x < hd / 8) {   // 8 values per thread, 4 threads per block (hd % 32 == 0)
        const float4 a = *(const float4 *)(sq + 8 * threadIdx.x), b = *(const float4 *)(sq + 8 * threadIdx.x + 4);
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        const int64_t e = (int64_t)t * nh * hd + h * hd + 8 * threadIdx.x;
        quant_block_4lanes(v, variant, xq + e, xd + e / 32, (threadIdx.x & 3) == 0, true, true);
    }
}

// ---------------------------------------------------------------------------
// The same attention for many queries of one segment (prefill), on f16 MFMA
// (v_mfma_f32_32x32x16_f16: lane l supplies A[l%32][8(l/32)..+8] and
// B[8(l/32)..+8][l%32]; result register v of lane l is row 8(v/4) + 4(l/32)
// + v%4, column l%32).  One workgroup takes a tile of AQ = 32 consecutive tokens
// and NH query heads of one kv head; wave (hh, sp) = (w % NH, w / NH) takes head hh
// and every fourth 32-key block (block 4 r + sp in round r), so a wave runs its
// scores, softmax and P V without another wave's data:
//   scores  S^T = K Q^T * scale: the key rows are the A operands (LDS), the
//           queries the B operands (registers), so a lane holds 16 keys of one
//           query.  The queries are BF16 values and the cache holds f16, both
//           exact in f16, so every product is exact and only the fp32 summation
//           order differs from the reference's;
//   softmax with a running max m per query and wave: e = expf(s - m), the sums of e
//           in double, both in registers (one exchange with lane l ^ 32, the other
//           half of the query's keys); when m rises, O and the sum are rescaled by
//           expf(m_old - m) (skipped while no query's m rises);
//   output  O^T = V^T P^T: the lane's 16 e values are its B operands as they are.
//           A contraction may take its keys in any order that both operands share,
//           so V^T is stored with the 16 keys of a step in the order in which the
//           lane halves hold them (0-3, 8-11 | 4-7, 12-15).  P enters as f16 hi +
//           lo halves (two products, ~22 bits of e).
// Each round's 128 key rows go to LDS by DMA and its V rows through registers,
// transposed as key-pair words, both one round ahead into the other half of the
// LDS, for one barrier per round.  At the end the four waves of a head merge in
// block order: m = max, weights expf(m_i - m), o = sum(w_i O_i) * (float)(1 / sum(w_i
// l_i)), the sums l in double, and the output goes out as Q8_0 or fp32.
// Every row below is at least one cache line and consecutive lanes take consecutive
// pieces of it.  The LDS is swizzled: 16-byte piece p of key row r at p ^ swz(r), 4-word
// piece p of V^T row d at p ^ ((d ^ d >> 3) & 15), so an operand read of 16 lanes and a
// transposing write of 64 fall on (nearly) distinct banks.
//
// Bound by the VALU work per score (max, exp, the double sum, the hi / lo split: ~22
// instructions) and the matrix products next to it, at two waves per SIMD (two heads per
// workgroup; one wave with one head, as the LDS holds one workgroup), and by what a
// wave waits while its loads queue at the address unit.  The tiles with the most keys
// are launched first.  Measured on 16 / 2 heads x 128, causal, back to back: 2048 tokens
// 56.2 us, 1500 tokens 38.3, 512 tokens 15.4, 333 tokens 12.8, 77 tokens 8.3.  (A workgroup
// per head whose eight waves split each 512-key chunk, with the scores' exponentials through
// LDS, two barriers and a drained load queue per chunk, one pass over at most 512 keys:
// 121.9, 75.9, 15.6, 14.1 and 10.4 us.)  Variants: the V loads issued after the scores +6 us at
// 2048 tokens, two chains of score products +1.5, the max followed exactly (a rescale in
// almost every block) with separate masks +15; expf without its range checks -0.3, as 2^(x
// log2 e) at once with the product's rounding error as a factor -2.7, but 1.26 ulp against 0.86.
// ---------------------------------------------------------------------------
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
constexpr int AQ = 32;
// A query's running max follows its scores only when one exceeds it by more than this:
// e then stays below e^8, far inside f16's range and no less precise relative to the
// sum, and the rescale of O is rare instead of due in almost every block (any of a
// wave's 32 queries may have a new max).
constexpr float kMaxSlack = 8.0f;

template <int HD, int NH>
__global__ __launch_bounds__(256 * NH, 1) void k_attention_mfma(
    const float *__restrict__ q, const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc,
    float *__restrict__ out, int M, int nh, int nkv, int cap, int kv_base, int causal, int8_t *__restrict__ xq,
    uint16_t *__restrict__ xd, int variant) {
    constexpr int NS = 4, KB = 32 * NS;        // key splits, keys of a round
    constexpr int NT = 256 * NH, NW = NT / 64;
    constexpr int KSTEPS = HD / 16;            // MFMA steps over the head dimension
    constexpr int DT = HD / 32;                // 32-dim output tiles
    constexpr int R16 = HD / 8;                // 16-byte pieces of a key or value row
    constexpr int KBytes = KB * HD * 2, Slot = 2 * KBytes;
    constexpr int KI = KBytes / 1024 / NW;     // DMA instructions per wave and round
    constexpr int VI = (KB / 2) * R16 / NT;    // (key pair, 8-dim piece) items per thread and round
    __shared__ __align__(1024) int8_t lds[2 * Slot];
    __shared__ float sm[NH][NS][32];
    __shared__ double sl[NH][NS][32];
    static_assert(NW * DT * 16 * 64 * 4 <= 2 * Slot, "the merge reuses the key and value rows");
    static_assert(KI >= 1 && VI >= 1 && (R16 == 8 || R16 == 16), "whole instructions");
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hh = wave % NH, sp = wave / NH, h = blockIdx.x * NH + hh;
    const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * AQ;
    const int kvh = (blockIdx.x * NH) / (nh / nkv);
    const uint16_t *kb = kc + (int64_t)kvh * cap * HD;
    const uint16_t *vb = vc + (int64_t)kvh * cap * HD;
    const int nq = min(AQ, M - t0);
    const int kv_end = causal ? kv_base + t0 + nq : M;
    const int kv_all = causal ? kv_base + t0 + 1 : M;                    // keys that every live query sees
    const int kvl = lr < nq ? (causal ? kv_base + t0 + lr + 1 : M) : 0;  // keys of query t0 + lr
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn((float)HD));
    const int nblk = (kv_end + 31) / 32, nr = (nblk + NS - 1) / NS;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    auto kswz = [](int r) { return R16 == 8 ? (r & 7) ^ ((r >> 3) & 1) : r & 15; };

    uint4 vr[VI][2];
    // round r's key rows into its slot, its value rows into registers; rows past the span
    // read the clamped last row (their scores are masked, their e zero)
    auto load = [&](int r) {
        const int k0 = KB * r;
#pragma unroll
        for (int i = 0; i < KI; i++) {
            const int in = wave * KI + i, row = in * (64 / R16) + lane / R16;
            const int pc = (lane % R16) ^ kswz(row);
            vxm_lds_dma16(lds0 + (r & 1) * Slot + in * 1024, kb + (int64_t)min(k0 + row, kv_end - 1) * HD + 8 * pc);
        }
#pragma unroll
        for (int u = 0; u < VI; u++) {
            const int item = u * NT + tid, c = item % R16, p = item / R16;
#pragma unroll
            for (int e = 0; e < 2; e++)
                vr[u][e] = *(const uint4 *)(vb + (int64_t)min(k0 + 2 * p + e, kv_end - 1) * HD + 8 * c);
        }
    };
    auto put_v = [&](int r) {
        uint32_t *vt = (uint32_t *)(lds + (r & 1) * Slot + KBytes);
#pragma unroll
        for (int u = 0; u < VI; u++) {
            const int item = u * NT + tid, c = item % R16, p = item / R16, pp = p & 7;
            const int w = (p & ~7) | (pp & 1) | ((pp >> 1) & 2) | ((pp << 1) & 4);
            const uint32_t a[4] = {vr[u][0].x, vr[u][0].y, vr[u][0].z, vr[u][0].w};
            const uint32_t b[4] = {vr[u][1].x, vr[u][1].y, vr[u][1].z, vr[u][1].w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int d = 8 * c + e;
                vt[d * (KB / 2) + (w ^ (((d ^ (d >> 3)) & 15) << 2))] =
                    e & 1 ? (a[e >> 1] >> 16) | (b[e >> 1] & 0xffff0000u) : (a[e >> 1] & 0xffffu) | (b[e >> 1] << 16);
            }
        }
    };

    load(0);
    v8h qa[KSTEPS];   // B operands: query t0 + lr, dims 16 kk + 8 lh .. + 8
    {
        const float *qr = q + (int64_t)(t0 + min(lr, nq - 1)) * nh * HD + h * HD + 8 * lh;
#pragma unroll
        for (int kk = 0; kk < KSTEPS; kk++) {
            const float4 x = *(const float4 *)(qr + 16 * kk), y = *(const float4 *)(qr + 16 * kk + 4);
            const float f[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int e = 0; e < 8; e++) qa[kk][e] = (_Float16)(lr < nq ? f[e] : 0.0f);
        }
    }
    float m = -INFINITY;
    double lsum = 0.0;   // this lane's keys (half of the wave's)
    v16f o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = v16f{};
    put_v(0);
    vxm_vm_wait_all();
    vxm_lds_barrier();
    for (int r = 0; r < nr; r++) {
        if (r + 1 < nr) load(r + 1);
        const int b = NS * r + sp;
        if (b < nblk) {
            const int8_t *ks = lds + (r & 1) * Slot, *vs = ks + KBytes;
            v16f s = v16f{};
            const int row = 32 * sp + lr;
#pragma unroll
            for (int kk = 0; kk < KSTEPS; kk++) {
                const v8h ka = *(const v8h *)(ks + row * (HD * 2) + (((2 * kk + lh) ^ kswz(row)) << 4));
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qa[kk], s, 0, 0, 0);
            }
            if (32 * b + 32 > kv_all) {   // some query does not see the whole block
#pragma unroll
                for (int v = 0; v < 16; v++)
                    if (32 * b + 8 * (v >> 2) + 4 * lh + (v & 3) >= kvl) s[v] = -INFINITY;
            }
            float mx = s[0];
#pragma unroll
            for (int v = 1; v < 16; v++) mx = fmaxf(mx, s[v]);
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * scale;   // scale > 0
            if (__any(mx > m + kMaxSlack)) {
                const float mn = fmaxf(m, mx), alpha = mn == -INFINITY ? 1.0f : expf(m - mn);
                m = mn;
                lsum *= (double)alpha;
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) o[dt][v] = o[dt][v] * alpha;
            }
            // a query without a live key so far has m = -inf and only masked scores: e = 0
            const float mneg = m == -INFINITY ? 0.0f : -m;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                s[v] = expf(__builtin_fmaf(s[v], scale, mneg));
                lsum += (double)s[v];
            }
#pragma unroll
            for (int st = 0; st < 2; st++) {
                v8h hi, lo;
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const v2f p = {s[8 * st + e], s[8 * st + e + 1]};
                    const v2h h2 = __builtin_convertvector(p, v2h);
                    const v2f l = {__builtin_fmaf((float)h2[0], -1.0f, p[0]), __builtin_fmaf((float)h2[1], -1.0f, p[1])};
                    const v2h l2 = __builtin_convertvector(l, v2h);
                    hi[e] = h2[0]; hi[e + 1] = h2[1];
                    lo[e] = l2[0]; lo[e + 1] = l2[1];
                }
#pragma unroll
                for (int dt = 0; dt < DT; dt++) {
                    const int d = 32 * dt + lr;
                    const v8h va = *(const v8h *)(vs + d * (KB * 2) +
                                                  (((4 * sp + 2 * st + lh) ^ ((d ^ (d >> 3)) & 15)) << 4));
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, hi, o[dt], 0, 0, 0);
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, lo, o[dt], 0, 0, 0);
                }
            }
        }
        if (r + 1 < nr) put_v(r + 1);
        vxm_vm_wait_all();   // this wave's key rows of the next round
        vxm_lds_barrier();   // every wave's; and this round's slot is free
    }

    // merge the head's four waves in block order
    lsum += __shfl_xor(lsum, 32);
    if (lh == 0) {
        sm[hh][sp][lr] = m;
        sl[hh][sp][lr] = lsum;
    }
    float *red = (float *)lds;   // [head][split][dim tile][16 values][64 lanes]
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) red[(((hh * NS + sp) * DT + dt) * 16 + v) * 64 + lane] = o[dt][v];
    __syncthreads();
    if (sp >= DT) return;
    const int dt = sp;   // this wave's output tile
    static_assert(DT <= NS, "one output tile per wave");
    float mm = sm[hh][0][lr];
#pragma unroll
    for (int i = 1; i < NS; i++) mm = fmaxf(mm, sm[hh][i][lr]);
    float w[NS];
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < NS; i++) {
        const float mi = sm[hh][i][lr];
        w[i] = mi == -INFINITY ? 0.0f : expf(mi - mm);
        sum += sl[hh][i][lr] * (double)w[i];
    }
    const float inv = kvl > 0 ? (float)(1.0 / sum) : 0.0f;
    float ov[16], amax = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        float a = 0.0f;
#pragma unroll
        for (int i = 0; i < NS; i++) a += red[(((hh * NS + i) * DT + dt) * 16 + v) * 64 + lane] * w[i];
        ov[v] = a * inv;
        amax = fmaxf(amax, fabsf(ov[v]));
    }
    // value v of lane (lr, lh): query t0 + lr, dim 32 dt + 8 (v / 4) + 4 lh + v % 4
    const int64_t e0 = (int64_t)(t0 + min(lr, nq - 1)) * nh * HD + h * HD + 32 * dt;
    if (xq) {
        // Q8_0 of the 32 dims (the arithmetic of quant_block_4lanes; two lanes per block)
        amax = fmaxf(amax, __shfl_xor(amax, 32));
        const float d = __fdiv_rn(amax, 127.0f);
        float id;
        if (variant == VXM_QUANT_X86) id = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
        else id = d != 0.0f ? __fdiv_rn(1.0f, d) : 0.0f;
        if (lr >= nq) return;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t b = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = ov[4 * j + e] * id;
                const float qv = fminf(fmaxf(variant == VXM_QUANT_X86 ? rintf(x) : roundf(x), -128.0f), 127.0f);
                b |= (uint32_t)(uint8_t)(int8_t)(int)qv << (8 * e);
            }
            *(uint32_t *)(xq + e0 + 8 * j + 4 * lh) = b;
        }
        if (lh == 0) xd[e0 / 32] = vxm_f2h(d);
    } else if (lr < nq) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            *(float4 *)(out + e0 + 8 * j + 4 * lh) = make_float4(ov[4 * j], ov[4 * j + 1], ov[4 * j + 2], ov[4 * j + 3]);
    }
}

template <int HD>
static void launch_attention_mfma(vxm_ctx *ctx, const float *q, const uint16_t *kc, const uint16_t *vc, float *out,
                                  int64_t M, int nh, int nkv, int cap, int kv_base, int causal, int8_t *xq,
                                  uint16_t *xd, int variant) {
    const unsigned tiles = (unsigned)((M + AQ - 1) / AQ);
    // two heads per workgroup share its key and value rows where that still fills the device
    // (16 / 2 x 128: 1000 tokens 28.2 against 33.6 us, 512 tokens 18.0 against 16.3)
    if (nh / nkv % 2 == 0 && (int64_t)nh / 2 * tiles >= ctx->n_cu)
        hipLaunchKernelGGL((k_attention_mfma<HD, 2>), dim3(nh / 2, tiles), dim3(512), 0, ctx->stream, q, kc, vc, out,
                           (int)M, nh, nkv, cap, kv_base, causal, xq, xd, variant);
    else
        hipLaunchKernelGGL((k_attention_mfma<HD, 1>), dim3(nh, tiles), dim3(256), 0, ctx->stream, q, kc, vc, out,
                           (int)M, nh, nkv, cap, kv_base, causal, xq, xd, variant);
}

// k_attention's dynamic LDS: a workgroup's 160 KB less its static arrays.
constexpr size_t kAttnMaxLds = 160 * 1024 - 64;

int vxm_launch_attention(vxm_ctx *ctx, const float *q, const uint16_t *kc, const uint16_t *vc, float *out,
                         int64_t M, int nh, int nkv, int hd, int cap, int64_t seg_stride, int S, int kv_base,
                         int causal, int8_t *xq, uint16_t *xd, int variant) {
    if (M <= 0) return VXM_OK;
    if (hd > 256 || hd <= 0 || nkv <= 0 || nh % nkv)
        return vxm_fail(ctx, VXM_ERR_INVALID_ARG, "attention: head_dim %d / heads %d,%d unsupported", hd, nh, nkv);
    // the MFMA kernel: the queries of a single segment, from a tile of them.  Fewer keep
    // k_attention although it is slower over a long context (16 heads of 128, 24 queries over
    // 474 keys: 18.6 against 13.0 us): it reads only the keys that a query sees, so a cache row
    // of infinities or NaN reaches no query before it, and its queries and probabilities stay
    // fp32 (a BF16 query past f16's range stays finite).  Its score buffer holds the capacity;
    // in a cache past that limit, the keys of the call, and past those the MFMA kernel runs.
    const int64_t span = causal ? kv_base + M : M;
    const bool tiles = S == M && span <= cap && (hd == 128 || hd == 64);
    const bool few = tiles && M >= 2 && M < AQ && span > 128;
    size_t lds = (size_t)(hd + cap + 256) * sizeof(float);
    if (few && lds > kAttnMaxLds) lds = (size_t)(hd + span + 256) * sizeof(float);
    if (tiles && (M >= AQ || (few && lds > kAttnMaxLds))) {
        if (hd == 128)
            launch_attention_mfma<128>(ctx, q, kc, vc, out, M, nh, nkv, cap, kv_base, causal, xq, xd, variant);
        else
            launch_attention_mfma<64>(ctx, q, kc, vc, out, M, nh, nkv, cap, kv_base, causal, xq, xd, variant);
        VXM_CHECK_LAUNCH(ctx);
        return VXM_OK;
    }
    if (lds > kAttnMaxLds)
        return vxm_fail(ctx, VXM_ERR_INVALID_ARG, "attention: capacity %d exceeds the LDS score buffer", cap);
    // 16-byte key loads need whole 16-byte rows and bases (the caches and the workspace
    // are 16-byte aligned, their heads and segments whole rows apart)
    const bool vec = hd % 8 == 0 && !(((uintptr_t)kc | (uintptr_t)vc) & 15) && seg_stride % 8 == 0;
    int8_t *fq = xq && hd % 32 == 0 ? xq : nullptr;   // a head's columns are whole Q8_0 blocks
    if (vec)
        hipLaunchKernelGGL(k_attention<true>, dim3(nh, (unsigned)M), dim3(256), lds, ctx->stream, q, kc, vc, out, nh,
                           nkv, hd, cap, seg_stride, S, kv_base, causal, fq, xd, variant);
    else
        hipLaunchKernelGGL(k_attention<false>, dim3(nh, (unsigned)M), dim3(256), lds, ctx->stream, q, kc, vc, out, nh,
                           nkv, hd, cap, seg_stride, S, kv_base, causal, fq, xd, variant);
    VXM_CHECK_LAUNCH(ctx);
    return xq && !fq ? vxm_launch_quantize(ctx, out, M, (int64_t)nh * hd, variant, xq, xd) : VXM_OK;
}

// ---------------------------------------------------------------------------
// Non-causal attention within segments of S tokens at positions pos0 ..
// pos0+S-1 with fresh K/V (the LocDiT and LocEnc blocks): k_rope_kv, the
// f16 K/V rounding, k_attention and the Q8_0 quantization of the output in
// one launch, with the same rounding steps and summation orders as those
// kernels.  One workgroup (256 threads) per (query head, segment) keeps the
// segment's q of its head and k, v of its kv head in LDS; qkv may arrive as
// K-split slices.  Output: the Q8_0 rows of the attention output (xq, xd).
// ---------------------------------------------------------------------------
constexpr int kLocalMaxS = 64, kLocalMaxElems = 2048;   // S, and S * hd per operand
constexpr int kLocalRB = 4;                              // query rows per workgroup

bool vxm_attention_local_fits(int S, int hd) {
    return S >= 1 && S <= kLocalMaxS && (hd == 64 || hd == 128) && (int64_t)S * hd <= kLocalMaxElems;
}

template <int HD>
__global__ __launch_bounds__(256) void k_attention_local(const vxm_parts qkv, int nh, int nkv, int S, int pos0,
                                                         const float2 *__restrict__ cs, int no_rope,
                                                         int8_t *__restrict__ xq, uint16_t *__restrict__ xd,
                                                         int variant) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int HALF = HD / 2, HP = HD + 4, RB = kLocalRB;
    const int h = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
    const int q0 = blockIdx.z * RB, nq = min(RB, S - q0);   // this workgroup's query rows
    const int kvh = h / (nh / nkv);
    const int qd = nh * HD, kvd = nkv * HD, ld = qd + 2 * kvd;
    const int SP = S + 1;
    // raw k, v: [S][HD]; raw q (later the output): [RB][HD]; rotated k: [S][HD + 4],
    // rotated q: [RB][HD + 4] (the pad spreads the score loop's 16-byte row reads over
    // the banks); P: [RB][S + 1]; row max and 1/sum: [RB] each
    float *Kr = lds, *V = Kr + S * HD, *Qr = V + S * HD, *Kf = Qr + RB * HD, *Q = Kf + S * HP, *P = Q + RB * HP;
    float *mx = P + RB * SP, *inv = mx + RB;
    // 1. raw q (rows q0 .. q0+nq-1 of head h), k and v (all S rows of kv head kvh),
    //    K-split slices added in order; the loads of up to four slices are in flight together
    constexpr int kRopePer = ((kLocalMaxElems / HD + RB) * HALF + 255) / 256;
    float2 csr[kRopePer];
    {
        constexpr int kMaxPer = (3 * kLocalMaxElems / 4 + 255) / 256;   // float4s per thread
        constexpr int R4 = HD / 4;                                      // float4s per row
        const int nqf = nq * R4, total = nqf + 2 * S * R4;
        int64_t src[kMaxPer];
        float *dst[kMaxPer];
        float4 acc4[kMaxPer];
#pragma unroll
        for (int k = 0; k < kMaxPer; k++) {
            const int f = min(tid + 256 * k, total - 1);   // threads past the end reload the last element
            int row, col;
            if (f < nqf) {
                row = q0 + f / R4;
                col = h * HD;
                dst[k] = Qr + (f / R4) * HD;
            } else {
                const int e = f - nqf, part = e / (S * R4), rr = (e % (S * R4)) / R4;
                row = rr;
                col = part == 0 ? qd + kvh * HD : qd + kvd + kvh * HD;
                dst[k] = (part == 0 ? Kr : V) + rr * HD;
            }
            const int off = 4 * (f % R4);
            src[k] = (int64_t)(g * S + row) * ld + col + off;
            dst[k] += off;
            acc4[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        // the rope table entries of this thread's phase-2 items, fetched with the projections
        if (!no_rope) {
#pragma unroll
            for (int k = 0; k < kRopePer; k++) {
                const int idx = min(tid + 256 * k, (S + nq) * HALF - 1);
                const int rr = idx / HALF, i = idx % HALF;
                const int pos = pos0 + (rr < S ? rr : q0 + rr - S);
                csr[k] = cs[(int64_t)pos * HALF + i];
            }
        }
        for (int z0 = 0; z0 < qkv.n; z0 += 4) {
            float4 b[4][kMaxPer];
#pragma unroll
            for (int zz = 0; zz < 4; zz++)
#pragma unroll
                for (int k = 0; k < kMaxPer; k++)
                    if (z0 + zz < qkv.n) b[zz][k] = *(const float4 *)(qkv.p + (z0 + zz) * qkv.stride + src[k]);
#pragma unroll
            for (int zz = 0; zz < 4; zz++)
#pragma unroll
                for (int k = 0; k < kMaxPer; k++)
                    if (z0 + zz < qkv.n) {
                        if (z0 + zz == 0) {
                            acc4[k] = b[zz][k];
                        } else {
                            acc4[k].x = acc4[k].x + b[zz][k].x; acc4[k].y = acc4[k].y + b[zz][k].y;
                            acc4[k].z = acc4[k].z + b[zz][k].z; acc4[k].w = acc4[k].w + b[zz][k].w;
                        }
                    }
        }
#pragma unroll
        for (int k = 0; k < kMaxPer; k++)
            if (tid + 256 * k < total) *(float4 *)dst[k] = acc4[k];
    }
    __syncthreads();
    // 2. BF16 + RoPE of q and k (pair-interleaved rows: row 2i = dim i, 2i+1 = dim
    //    i + hd/2), the f16 cache rounding of k and v
#pragma unroll
    for (int k = 0; k < kRopePer; k++) {
        const int idx = tid + 256 * k;
        if (idx >= (S + nq) * HALF) break;
        const int rr = idx / HALF, i = idx % HALF;
        const bool isk = rr < S;
        const int lr = isk ? rr : rr - S;
        float c = 1.0f, sn = 0.0f;
        if (!no_rope) {
            c = csr[k].x;
            sn = csr[k].y;
        }
        const float *sp = (isk ? Kr : Qr) + lr * HD;
        const float x0 = vxm_bf16(sp[2 * i]), x1 = vxm_bf16(sp[2 * i + 1]);
        float y0 = x0, y1 = x1;
        if (!no_rope) {
            y0 = vxm_bf16(x0 * c - x1 * sn);
            y1 = vxm_bf16(x0 * sn + x1 * c);
        }
        if (isk) {
            y0 = vxm_h2f(vxm_f2h(y0));
            y1 = vxm_h2f(vxm_f2h(y1));
        }
        float *dp = (isk ? Kf : Q) + lr * HP;
        dp[i] = y0;
        dp[i + HALF] = y1;
    }
    for (int idx = tid; idx < S * HD; idx += 256) V[idx] = vxm_h2f(vxm_f2h(vxm_bf16(V[idx])));
    __syncthreads();
    // 3. scores s_ij = (k_j . q_i) * scale, d in order
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn((float)HD));
    for (int idx = tid; idx < nq * S; idx += 256) {
        const int i = idx / S, j = idx % S;
        const float4 *kr = (const float4 *)(Kf + j * HP), *qr = (const float4 *)(Q + i * HP);
        float sc = 0.0f;
#pragma unroll 8
        for (int d4 = 0; d4 < HD / 4; d4++) {
            const float4 a = kr[d4], b = qr[d4];
            sc += a.x * b.x;
            sc += a.y * b.y;
            sc += a.z * b.z;
            sc += a.w * b.w;
        }
        P[i * SP + j] = sc * scale;
    }
    __syncthreads();
    // 4. softmax: row max, exponentials, the row sum in double and (float)(1/sum); wave i
    //    takes query row i, lane j key j (S <= 64), so the max and the sum are wave
    //    reductions.  The double sum of at most 64 exponentials of one row is exact
    //    unless they span more than 2^29, so its order matches the serial sum's.
    static_assert(kLocalRB <= 4 && kLocalMaxS <= 64, "one wave per query row, one lane per key");
    {
        const int i = tid >> 6, j = tid & 63;
        if (i < nq) {
            // the wave reductions on DPP within rows of 16 lanes, the four rows read back
            // as scalars (no LDS round trip per step)
            const float sj = j < S ? P[i * SP + j] : -INFINITY;
            float m = sj;
            m = fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m), 0xB1, 0xF, 0xF, false)));
            m = fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m), 0x4E, 0xF, 0xF, false)));
            m = fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m), 0x141, 0xF, 0xF, false)));
            m = fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m), 0x140, 0xF, 0xF, false)));
            {
                float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), 0));
#pragma unroll
                for (int r = 1; r < 4; r++) t = fmaxf(t, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), 16 * r)));
                m = t;
            }
            const float e = j < S ? expf(sj - m) : 0.0f;
            if (j < S) P[i * SP + j] = e;
            double sum = (double)e;
            auto dpp_d = [](double x, auto ctrl) {
                const long long b = __double_as_longlong(x);
                const int lo = __builtin_amdgcn_update_dpp(0, (int)b, decltype(ctrl)::value, 0xF, 0xF, false);
                const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), decltype(ctrl)::value, 0xF, 0xF, false);
                return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
            };
            sum = sum + dpp_d(sum, std::integral_constant<int, 0xB1>{});
            sum = sum + dpp_d(sum, std::integral_constant<int, 0x4E>{});
            sum = sum + dpp_d(sum, std::integral_constant<int, 0x141>{});
            sum = sum + dpp_d(sum, std::integral_constant<int, 0x140>{});
            {
                const long long b = __double_as_longlong(sum);
                double t = 0.0;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, 16 * r);
                    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), 16 * r);
                    t += __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
                }
                sum = t;
            }
            if (j == 0) {
                mx[i] = m;
                inv[i] = (float)(1.0 / sum);
            }
        }
    }
    __syncthreads();
    // 5. out[i][d] = sum_j v[j][d] p_ij, p_ij = e_ij * inv_i, over the j-slices of
    //    k_attention (256 / hd of them, each summed in order, then added in order);
    //    thread (row group rg, dim d) owns rows rg, rg + R, ...; rows past nq read row
    //    nq - 1 with a zero weight, so the loop has no divergent reads
    {
        constexpr int R = 256 / HD, MAXR = (RB + R - 1) / R;
        const int d = tid % HD, rg = tid / HD;
        const int slices = 256 / HD, jper = (S + slices - 1) / slices;
        float tot[MAXR], acc[MAXR], iv[MAXR];
        int prow[MAXR];
#pragma unroll
        for (int k = 0; k < MAXR; k++) {
            tot[k] = 0.0f;
            iv[k] = rg + R * k < nq ? inv[rg + R * k] : 0.0f;
            prow[k] = min(rg + R * k, nq - 1) * SP;
        }
        for (int sl = 0; sl < slices; sl++) {
            const int j0 = sl * jper, j1 = min(S, j0 + jper);
#pragma unroll
            for (int k = 0; k < MAXR; k++) acc[k] = 0.0f;
#pragma unroll 4
            for (int j = j0; j < j1; j++) {
                const float v = V[j * HD + d];
#pragma unroll
                for (int k = 0; k < MAXR; k++) acc[k] += v * (P[prow[k] + j] * iv[k]);
            }
#pragma unroll
            for (int k = 0; k < MAXR; k++) tot[k] += acc[k];
        }
#pragma unroll
        for (int k = 0; k < MAXR; k++)
            if (rg + R * k < nq) Qr[(rg + R * k) * HD + d] = tot[k];
    }
    __syncthreads();
    // 6. Q8_0 of the output rows: thread (i, c) holds dims 8c .. 8c+7, four consecutive
    //    threads one 32-block (hd / 8 % 4 == 0: whole 4-lane groups stop together)
    constexpr int CPR = HD / 8;
    for (int idx = tid; idx < nq * CPR; idx += 256) {
        const int i = idx / CPR, c = idx % CPR;
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = Qr[i * HD + 8 * c + e];
        const int64_t el = (int64_t)(g * S + q0 + i) * qd + h * HD + 8 * c;
        quant_block_4lanes(o, variant, xq + el, xd + el / 32, (tid & 3) == 0);
    }
}

int vxm_launch_attention_local(vxm_ctx *ctx, vxm_parts qkv, int64_t M, int nh, int nkv, int hd, int S, int pos0,
                               const float2 *cs, int cs_rows, int no_rope, int8_t *xq, uint16_t *xd, int variant) {
    if (M <= 0) return VXM_OK;
    if (!vxm_attention_local_fits(S, hd) || M % S || nkv <= 0 || nh % nkv)
        return vxm_fail(ctx, VXM_ERR_INVALID_ARG, "local attention: S=%d hd=%d M=%lld unsupported", S, hd,
                        (long long)M);
    if (!no_rope && (!cs || pos0 + S > cs_rows))
        return vxm_fail(ctx, VXM_ERR_BACKEND, "rope: table holds %d positions, %d needed", cs_rows, pos0 + S);
    // query rows per workgroup: blocks of kLocalRB spread a segment's rows over several CUs
    // (each block re-derives the segment's k and v)
    const int RB = kLocalRB, QB = (S + RB - 1) / RB;
    const size_t lds = (size_t)(2 * S * hd + RB * hd + (S + RB) * (hd + 4) + RB * (S + 1) + 2 * RB) * sizeof(float);
    const dim3 grid(nh, (unsigned)(M / S), QB);
    if (hd == 64)
        hipLaunchKernelGGL(k_attention_local<64>, grid, dim3(256), lds, ctx->stream, qkv, nh, nkv, S, pos0, cs,
                           no_rope, xq, xd, variant);
    else
        hipLaunchKernelGGL(k_attention_local<128>, grid, dim3(256), lds, ctx->stream, qkv, nh, nkv, S, pos0, cs,
                           no_rope, xq, xd, variant);
    VXM_CHECK_LAUNCH(ctx);
    return VXM_OK;
}

// ---------------------------------------------------------------------------
// vcpm_mlp activation (src/minicpm4.c:441-456): p = bf16(bf16(silu(bf16(g))) *
// bf16(u)), silu(x) = x / (1 + expf(-x)), then Q8_0 quantization of p.
// Row m of the fused gate/up projection holds 2F values interleaved: gate n at
// gu[m*ld + 2n], up n at gu[m*ld + 2n + 1].  8 outputs per thread.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_swiglu_quant(const vxm_parts gu, int64_t F, int64_t ld,
                                                      int64_t total, int8_t *__restrict__ xq,
                                                      uint16_t *__restrict__ xd, float *__restrict__ p_out,
                                                      int variant) {
    const int64_t e = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
    if (e >= total) return;   // total, F % 32 == 0: 4-lane groups are all live or all dead
    const int64_t m = e / F, j = e % F;
    const float *s = gu.p + m * ld + 2 * j;
    float gv[8], uv[8];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        // K-split slices: up to four loads in flight, added in order
        float4 a = *(const float4 *)(s + 4 * k);
        for (int z0 = 1; z0 < gu.n; z0 += 4) {
            float4 b[4];
#pragma unroll
            for (int zz = 0; zz < 4; zz++)
                if (z0 + zz < gu.n) b[zz] = *(const float4 *)(s + (z0 + zz) * gu.stride + 4 * k);
#pragma unroll
            for (int zz = 0; zz < 4; zz++)
                if (z0 + zz < gu.n) {
                    a.x = a.x + b[zz].x; a.y = a.y + b[zz].y; a.z = a.z + b[zz].z; a.w = a.w + b[zz].w;
                }
        }
        gv[2 * k] = a.x; uv[2 * k] = a.y; gv[2 * k + 1] = a.z; uv[2 * k + 1] = a.w;
    }
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float gb = vxm_bf16(gv[i]);
        const float s = vxm_bf16(__fdiv_rn(gb, 1.0f + expf(-gb)));
        p[i] = vxm_bf16(s * vxm_bf16(uv[i]));
    }
    if (p_out) {
        *(float4 *)(p_out + e) = make_float4(p[0], p[1], p[2], p[3]);
        *(float4 *)(p_out + e + 4) = make_float4(p[4], p[5], p[6], p[7]);
    }
    quant_block_4lanes(p, variant, xq + e, xd + e / 32, (threadIdx.x & 3) == 0);
}

int vxm_launch_swiglu_quant(vxm_ctx *ctx, vxm_parts gu, int64_t M, int64_t F, int64_t ld, int8_t *xq,
                            uint16_t *xd, float *p_out, int variant) {
    const int64_t total = M * F;
    if (total <= 0) return VXM_OK;
    if (F % 32) return vxm_fail(ctx, VXM_ERR_INVALID_ARG, "swiglu: width %lld not a multiple of 32", (long long)F);
    const int64_t threads = total / 8;
    hipLaunchKernelGGL(k_swiglu_quant, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream, gu, F,
                       ld, total, xq, xd, p_out, variant);
    VXM_CHECK_LAUNCH(ctx);
    return VXM_OK;
}

// ---------------------------------------------------------------------------
// h = bf16(h + scale * bf16(delta)) (the residual adds of
// vcpm_minicpm4_block, src/minicpm4.c:496-528), elementwise.
// ---------------------------------------------------------------------------
// Four elements per thread, every K-split slice's load in flight, added in slice order
// (n % 4 == 0: rows of whole 32-value blocks; h and the slices are 16-byte aligned, as
// the norm that reads them requires).
__global__ __launch_bounds__(256) void k_residual(float *__restrict__ h, const vxm_parts delta, float scale,
                                                  int64_t n) {
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= n) return;
    float4 x = *(const float4 *)(h + i), p[VXM_MAX_PARTS];
#pragma unroll
    for (int z = 0; z < VXM_MAX_PARTS; z++)
        if (z < delta.n) p[z] = *(const float4 *)(delta.p + z * delta.stride + i);
    float4 d = p[0];
#pragma unroll
    for (int z = 1; z < VXM_MAX_PARTS; z++)
        if (z < delta.n) {
            d.x = d.x + p[z].x; d.y = d.y + p[z].y; d.z = d.z + p[z].z; d.w = d.w + p[z].w;
        }
    auto add = [&](float a, float b) {
        float o = vxm_bf16(b);
        if (scale != 1.0f) o = o * scale;
        return vxm_bf16(a + o);
    };
    *(float4 *)(h + i) = make_float4(add(x.x, d.x), add(x.y, d.y), add(x.z, d.z), add(x.w, d.w));
}

int vxm_launch_residual(vxm_ctx *ctx, float *h, vxm_parts delta, float scale, int64_t n) {
    if (n <= 0) return VXM_OK;
    if (n % 4) return vxm_fail(ctx, VXM_ERR_INVALID_ARG, "residual: %lld values are not whole blocks", (long long)n);
    hipLaunchKernelGGL(k_residual, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, ctx->stream, h, delta, scale,
                       n);
    VXM_CHECK_LAUNCH(ctx);
    return VXM_OK;
}

// y = bf16(x + bias) per row (ggml_add of a repeated bias then BF16,
// src/locdit.c:190-210 and :118-121); bias may be null (BF16 only).
__global__ void k_bias_bf16(const float *__restrict__ x, const float *__restrict__ bias, float *__restrict__ y,
                            int64_t rows, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * n) return;
    float v = x[i];
    if (bias) v = v + bias[i % n];
    y[i] = vxm_bf16(v);
}

int vxm_launch_bias_bf16(vxm_ctx *ctx, const float *x, const float *bias, float *y, int64_t rows, int64_t n) {
    if (rows * n <= 0) return VXM_OK;
    hipLaunchKernelGGL(k_bias_bf16, dim3((unsigned)((rows * n + 255) / 256)), dim3(256), 0, ctx->stream, x, bias,
                       y, rows, n);
    VXM_CHECK_LAUNCH(ctx);
    return VXM_OK;
}
