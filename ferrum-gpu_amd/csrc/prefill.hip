// The prompt pass of the GPT-2 decoder for gfx950: the key and value cache rows of many prompt tokens
// at once. Replaces a loop of ferrum_ref's Gpt2::feed over the prompt
// (ferrum_gpu_core/src/engine/mod.rs:204-242, ferrum_ref/src/models/gpt2/decode.rs:57-117), which reads
// every weight once per token: the decode step is bound by the latency of its chain of phases (about
// 195 us a token at GPT-2-small), not by its 131 MB of weights, so a prompt of 480 tokens cost 94 ms.
// Here a chunk's rows go through each product together, on the precise MFMA GEMM, and a layer is nine
// launches whatever the row count. Only the caches are wanted: the last layer stops after its k and v,
// and the prompt's last token, whose logits are, runs as a decode step.
//
// Numerics: f32 rows, biases, LayerNorm, softmax and GELU as in the step. The GEMM takes x as two f16
// parts of a fixed exponent range (gemm.hip); prefill_row_kernel therefore puts every row on a
// power-of-two scale first (largest |x| in [2^13, 2^14): 22 bits of it, and elements down to 2^-13 of
// it keep theirs), and the consumer of the product multiplies by the exact inverse, so rows of any
// magnitude keep that. A step carries x in 30 bits of its block's largest value; in the next logits the difference does
// not show (error against float64, 160 models of 256 to 768 wide, 2 to 12 layers and prompts of 30 to 480, pass over
// steps: 0.99 on the mean, to 0.01). Attention runs on the f32 matrix cores.
#include "device_common.hpp"
#include "internal.hpp"

namespace fh {
namespace {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRowThreads = 256;

__device__ __forceinline__ float block_reduce_add(float v, float *red) {
    v = wave_reduce(v, AddOp());
    __syncthreads();  // an earlier use of red is over
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}
__device__ __forceinline__ float block_reduce_max(float v, float *red) {
    v = wave_reduce(v, MaxOp());
    __syncthreads();
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// One row (blockIdx.x) into the next product's split x. The row's k values by mode: EMBED_LN the
// LayerNorm of the embedding, RES_LN of the residual row plus the previous product (both store the
// residual row), GELU of the product plus its bias, PLAIN the row as it is. NV: 4-value groups a thread
// keeps (k <= 1024 NV). Bound by latency (a 480 x 768 row set is 1.5 MB): one workgroup per row, one
// round of loads, the row in registers through the reductions.
template <int KIND, int MODE, int NV>
__global__ __launch_bounds__(kRowThreads) void prefill_row_kernel(PrefillRow a) {
    __shared__ float red[4];
    const uint32_t row = blockIdx.x, groups = a.k / 4, tid = threadIdx.x;
    const size_t at = (size_t)row * a.k;
    f32x4 v[NV];
#pragma unroll
    for (int u = 0; u < NV; u++) {
        const uint32_t g = tid + u * kRowThreads;
        v[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (g >= groups) continue;
        if constexpr (MODE == PREFILL_EMBED_LN) {
            // x = tok[t] + pos[p] (decode.rs:72-74)
            const uint32_t t = (uint32_t)a.tokens[row], nb = a.k / 32, b = g / 8;
            const f32x4 pv = *(const f32x4 *)(a.pos + at + 4 * g);
            const size_t slot = tile_slot(t, b, nb);
            const float d = half_bits_to_float(a.emb_ds[scale_slot(t, b, nb)]);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint32_t j = 4 * (g % 8) + c;
                float q;
                if constexpr (KIND == FH_Q8_0) {
                    q = (float)(int8_t)a.emb_qs[slot * 32 + j];
                } else {
                    const uint32_t byte = a.emb_qs[slot * 16 + j % 16];
                    q = (float)((int32_t)(j < 16 ? byte & 15u : byte >> 4) - 8);
                }
                v[u][c] = d * q + pv[c];
            }
        } else if constexpr (MODE == PREFILL_PLAIN) {
            v[u] = *(const f32x4 *)(a.src + at + 4 * g);
        } else {
            f32x4 s = *(const f32x4 *)(a.src + at + 4 * g);
            for (uint32_t i = 1; i < a.splits; i++) s += *(const f32x4 *)(a.src + i * a.stride + at + 4 * g);
            s = s * a.in_scale[row] + *(const f32x4 *)(a.bias + 4 * g);
            if constexpr (MODE == PREFILL_RES_LN) {
                v[u] = *(const f32x4 *)(a.x + at + 4 * g) + s;
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++) v[u][c] = gelu_act(s[c]);
            }
        }
        if constexpr (MODE == PREFILL_EMBED_LN || MODE == PREFILL_RES_LN) *(f32x4 *)(a.x + at + 4 * g) = v[u];
    }
    if constexpr (MODE == PREFILL_EMBED_LN || MODE == PREFILL_RES_LN) {  // nn.rs:31-44
        float sum = 0.0f;
#pragma unroll
        for (int u = 0; u < NV; u++) sum += (v[u].x + v[u].y) + (v[u].z + v[u].w);
        const float mean = block_reduce_add(sum, red) / (float)a.k;
        float sq = 0.0f;
#pragma unroll
        for (int u = 0; u < NV; u++)
            if (tid + u * kRowThreads < groups)
#pragma unroll
                for (int c = 0; c < 4; c++) sq += (v[u][c] - mean) * (v[u][c] - mean);
        const float rstd = 1.0f / sqrtf(block_reduce_add(sq, red) / (float)a.k + a.eps);
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const uint32_t g = tid + u * kRowThreads;
            if (g >= groups) continue;
            const f32x4 lg = *(const f32x4 *)(a.ln_g + 4 * g), lb = *(const f32x4 *)(a.ln_b + 4 * g);
#pragma unroll
            for (int c = 0; c < 4; c++) v[u][c] = (v[u][c] - mean) * rstd * lg[c] + lb[c];
        }
    }
    float mx = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; u++)
#pragma unroll
        for (int c = 0; c < 4; c++) mx = fmaxf(mx, fabsf(v[u][c]));
    mx = block_reduce_max(mx, red);
    int e = 0;  // 2^e <= mx < 2^(e + 1); rows with an infinity keep their values (hi and lo stay non-finite)
    if (mx <= 3.4028235e38f) e = max((int)(__float_as_uint(mx) >> 23) - 127, -100);
    const float f = __uint_as_float((uint32_t)(127 + 13 - e) << 23);
    if (tid == 0) a.out_scale[row] = __uint_as_float((uint32_t)(127 - 13 + e) << 23);
    _Float16 *xs = a.xs + (size_t)row * a.k * 2;
#pragma unroll
    for (int u = 0; u < NV; u++) {
        const uint32_t g = tid + u * kRowThreads;
        if (g >= groups) continue;
        // the precise GEMM's operand order (split_x_precise_kernel): a group's four elements in the
        // order 0, 2, 1, 3; Q4_0 pairs group i of the block's first half with group i of its second
        const uint32_t b = g / 8, j = g % 8, place = KIND == FH_Q8_0 ? j : 2 * (j % 4) + j / 4;
        const float w[4] = {v[u].x * f, v[u].z * f, v[u].y * f, v[u].w * f};
        f16x4 hi, lo;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            hi[c] = (_Float16)w[c];
            lo[c] = (_Float16)(w[c] - (float)hi[c]);
        }
        *(f16x4 *)(xs + b * 64 + 4 * place) = hi;
        *(f16x4 *)(xs + b * 64 + 32 + 4 * place) = lo;
    }
}

// The QKV product's rows plus bias: q to its rows, k and v to the caches (decode.rs:78-84).
__global__ __launch_bounds__(256) void prefill_qkv_kernel(const float *__restrict__ src, uint32_t splits, size_t stride,
                                                          const float *__restrict__ in_scale,
                                                          const float *__restrict__ bias, float *__restrict__ q,
                                                          float *__restrict__ kc, float *__restrict__ vc, uint32_t d) {
    const uint32_t row = blockIdx.y, i = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (i >= 3 * d) return;
    const size_t at = (size_t)row * 3 * d + i;
    f32x4 s = *(const f32x4 *)(src + at);
    for (uint32_t p = 1; p < splits; p++) s += *(const f32x4 *)(src + p * stride + at);
    s = s * in_scale[row] + *(const f32x4 *)(bias + i);
    float *dst = i < d ? q : i < 2 * d ? kc : vc;
    *(f32x4 *)(dst + (size_t)row * d + i % d) = s;  // (d is a multiple of 32: a group stays in one part)
}

// Causal attention of `m` rows at positions p0 .. p0 + m - 1 over the caches [position][d], f32 on
// v_mfma_f32_32x32x2_f32. One workgroup per head and 32 query rows; its wavefronts take the 32-key tiles
// in turn, each with a running maximum and sum, the next tile's keys and values loaded while the current
// one computes, and merge through LDS. S^T = K Q^T leaves a lane one query and keys in the order of
// its accumulator registers, which is the B operand's order for O^T += V^T P^T. f32 products keep the
// step's precision; at 480 rows a layer's attention is 0.4 GFLOP, so the f16 matrix cores' speed is
// not needed.
template <int HD>
struct PrefillTile {
    static constexpr int M4 = HD / 8, DB = HD >= 32 ? HD / 32 : 1;
    f32x4 k[M4];
    float v[DB][16];
};

template <int HD, int W>
__global__ __launch_bounds__(64 * W) void prefill_attention_kernel(const float *__restrict__ q,
                                                                   const float *__restrict__ kc,
                                                                   const float *__restrict__ vc,
                                                                   float *__restrict__ att, uint32_t p0, uint32_t m,
                                                                   uint32_t d, float scale) {
    using T = PrefillTile<HD>;
    constexpr int DB = T::DB;
    __shared__ float red[W][2 + 16 * DB][64];
    const uint32_t lane = threadIdx.x % 64, w = threadIdx.x / 64, col = lane % 32, slot = lane / 32;
    const uint32_t q0 = (gridDim.y - 1 - blockIdx.y) * 32;  // the longest rows are dispatched first
    const uint32_t off = blockIdx.x * HD, query = q0 + col, keys = p0 + m;
    f32x4 qf[T::M4];
#pragma unroll
    for (int i = 0; i < T::M4; i++)
        qf[i] = query < m ? *(const f32x4 *)(q + (size_t)query * d + off + 4 * slot + 8 * i) : f32x4{0.f, 0.f, 0.f, 0.f};
    auto load = [&](T &t, uint32_t k0) {
        const uint32_t key = min(k0 + col, keys - 1);  // keys past the last are masked below
#pragma unroll
        for (int i = 0; i < T::M4; i++) t.k[i] = *(const f32x4 *)(kc + (size_t)key * d + off + 4 * slot + 8 * i);
#pragma unroll
        for (int b = 0; b < DB; b++)
#pragma unroll
            for (int s = 0; s < 16; s++) {
                const uint32_t kk = min(k0 + 8 * (s / 4) + 4 * slot + s % 4, keys - 1), dim = 32 * b + col;
                t.v[b][s] = HD >= 32 || dim < (uint32_t)HD ? vc[(size_t)kk * d + off + dim] : 0.0f;
            }
    };
    f32x16 o[DB];
#pragma unroll
    for (int b = 0; b < DB; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[b][i] = 0.0f;
    float mrun = -INFINITY, lrun = 0.0f;
    const uint32_t tiles = (p0 + min(q0 + 31u, m - 1u)) / 32 + 1;  // key tiles the block's rows see
    T cur, nxt;
    if (w < tiles) load(cur, 32 * w);
    for (uint32_t kt = w; kt < tiles; kt += W) {
        const uint32_t k0 = 32 * kt;
        if (kt + W < tiles) load(nxt, k0 + 32 * W);
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.0f;
#pragma unroll
        for (int i = 0; i < T::M4; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(cur.k[i][c], qf[i][c], s, 0, 0, 0);
        float mt = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t key = k0 + 8 * (i / 4) + 4 * slot + i % 4;
            s[i] = key <= p0 + query ? s[i] * scale : -INFINITY;
            mt = fmaxf(mt, s[i]);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float mnew = fmaxf(mrun, mt);
        // (the block's first rows may see no key of its last tile: nothing is added then)
        const float base = mnew == -INFINITY ? 0.0f : mnew;
        const float alpha = expf(mrun - base);
        float ls = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            s[i] = expf(s[i] - base);
            ls += s[i];
        }
        lrun = lrun * alpha + ls;
        mrun = mnew;
#pragma unroll
        for (int b = 0; b < DB; b++) {
#pragma unroll
            for (int i = 0; i < 16; i++) o[b][i] *= alpha;
#pragma unroll
            for (int i = 0; i < 16; i++) o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur.v[b][i], s[i], o[b], 0, 0, 0);
        }
        cur = nxt;
    }
    red[w][0][lane] = mrun;
    red[w][1][lane] = lrun;
#pragma unroll
    for (int b = 0; b < DB; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) red[w][2 + 16 * b + i][lane] = o[b][i];
    __syncthreads();
    if (w) return;
    float M = red[0][0][lane];
#pragma unroll
    for (int j = 1; j < W; j++) M = fmaxf(M, red[j][0][lane]);
    float f[W], l = 0.0f;
#pragma unroll
    for (int j = 0; j < W; j++) {
        f[j] = red[j][0][lane] == -INFINITY ? 0.0f : expf(red[j][0][lane] - M);  // (a wavefront without tiles)
        l += red[j][1][lane] * f[j];
    }
    l += __shfl_xor(l, 32);
    if (query >= m) return;
    float *out = att + (size_t)query * d + off;
#pragma unroll
    for (int b = 0; b < DB; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t dim = 32 * b + 8 * (i / 4) + 4 * slot + i % 4;
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < W; j++) acc += red[j][2 + 16 * b + i][lane] * f[j];
            if (dim < (uint32_t)HD) out[dim] = acc / l;
        }
}

template <int KIND, int MODE>
hipError_t launch_row_mode(hipStream_t s, const PrefillRow &a, uint32_t rows) {
    if (a.k <= 1024)
        prefill_row_kernel<KIND, MODE, 1><<<rows, kRowThreads, 0, s>>>(a);
    else if (a.k <= 4096)
        prefill_row_kernel<KIND, MODE, 4><<<rows, kRowThreads, 0, s>>>(a);
    else
        prefill_row_kernel<KIND, MODE, 16><<<rows, kRowThreads, 0, s>>>(a);
    return hipGetLastError();
}

template <int KIND>
hipError_t launch_row_kind(hipStream_t s, int mode, const PrefillRow &a, uint32_t rows) {
    switch (mode) {
    case PREFILL_EMBED_LN: return launch_row_mode<KIND, PREFILL_EMBED_LN>(s, a, rows);
    case PREFILL_RES_LN: return launch_row_mode<KIND, PREFILL_RES_LN>(s, a, rows);
    case PREFILL_GELU: return launch_row_mode<KIND, PREFILL_GELU>(s, a, rows);
    default: return launch_row_mode<KIND, PREFILL_PLAIN>(s, a, rows);
    }
}

}  // namespace

bool prefill_head_supported(size_t hd) { return hd == 8 || hd == 16 || hd == 32 || hd == 64 || hd == 128; }

hipError_t launch_prefill_row(hipStream_t s, fh_kind kind, int mode, const PrefillRow &a, uint32_t rows) {
    if (a.k % 32 || a.k > 16384) return hipErrorInvalidValue;
    return kind == FH_Q8_0 ? launch_row_kind<FH_Q8_0>(s, mode, a, rows) : launch_row_kind<FH_Q4_0>(s, mode, a, rows);
}

hipError_t launch_prefill_qkv(hipStream_t s, const SplitOut &src, const float *in_scale, const float *bias, float *q,
                              float *kc, float *vc, uint32_t rows, uint32_t d) {
    prefill_qkv_kernel<<<dim3((3 * d / 4 + 255) / 256, rows), 256, 0, s>>>(src.part, src.splits, (size_t)rows * 3 * d,
                                                                           in_scale, bias, q, kc, vc, d);
    return hipGetLastError();
}

hipError_t launch_prefill_attention(hipStream_t s, const float *q, const float *kc, const float *vc, float *att,
                                    uint32_t p0, uint32_t rows, uint32_t heads, uint32_t hd, float scale) {
    const dim3 grid(heads, (rows + 31) / 32);
    const uint32_t d = heads * hd;
    switch (hd) {
    case 8: prefill_attention_kernel<8, 4><<<grid, 256, 0, s>>>(q, kc, vc, att, p0, rows, d, scale); break;
    case 16: prefill_attention_kernel<16, 4><<<grid, 256, 0, s>>>(q, kc, vc, att, p0, rows, d, scale); break;
    case 32: prefill_attention_kernel<32, 4><<<grid, 256, 0, s>>>(q, kc, vc, att, p0, rows, d, scale); break;
    case 64: prefill_attention_kernel<64, 4><<<grid, 256, 0, s>>>(q, kc, vc, att, p0, rows, d, scale); break;
    case 128: prefill_attention_kernel<128, 2><<<grid, 128, 0, s>>>(q, kc, vc, att, p0, rows, d, scale); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace fh
