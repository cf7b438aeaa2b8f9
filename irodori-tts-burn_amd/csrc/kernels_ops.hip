// The staging kernel of the isolated joint attention operator (irodori_op_joint_attention): the
// caller's attention operands into the layouts the model's QKV+gate epilogue writes.
#include "common.hpp"
#include "kernels.hpp"

namespace irodori {

namespace {

template <typename T>
__device__ __forceinline__ int vt_pos(int s) {
    return sizeof(T) == 2 ? vt_pos_bf16(s) : vt_pos_f32(s);
}

// Column of the 64-key block that V^T position p holds (the inverse of vt_pos; both key
// orders only permute keys inside aligned groups of 16 (bf16) or 32 (f32)).
template <typename T>
__device__ __forceinline__ int vt_src(int p) {
    if (sizeof(T) == 2) return vt_pos_bf16(p);  // a swap of key bits 2 and 3: its own inverse
    const int pp = p & 31;
    return (p & ~31) | (((pp >> 2) & 1) * 16 + (pp >> 3) * 4 + (pp & 3));
}

// One block per (b, h, 32 tokens): 16 lanes per token, four head dimensions each, so that a
// lane holds whole RoPE pairs and the head norm's sum stays in one 16-lane row; every load of
// the block's two passes goes out first.  The head RMSNorm (norm.rs:60-74) and the
// interleaved half RoPE (rope.rs:82-135) as the QKV epilogue applies them.  V goes through
// LDS so that each V^T row (b, h, d) leaves as one run of 32 keys; keys past S (up to the
// 64-key boundary) are written as zeros.  HBM-bound in principle (2 x 750 tokens of 16 heads:
// 24.6 MB read and 12.3 MB written, 7 us at copy rate, half of it from cache when the caller has just
// written its operands); a lane per dimension with 4-byte loads and 6-step shuffles took 17 us.
template <typename T>
__global__ __launch_bounds__(256) void attn_op_stage_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ gate, const float* __restrict__ q_norm, const float* __restrict__ k_norm,
    const float* __restrict__ rope_cos, const float* __restrict__ rope_sin, int S, int H, float eps,
    float q_scale, int vt_stride, T* __restrict__ Q, T* __restrict__ K, T* __restrict__ Vt, T* __restrict__ G) {
    __shared__ float vs[32][68];
    const int tid = threadIdx.x, d = 4 * (tid & 15);
    const int s0 = blockIdx.x * 32, h = blockIdx.y, b = blockIdx.z;
    const bool rope = h < H / 2;
    float4 xq[2], xk[2], xv[2], xg[2];
    float2 rc[2], rs[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int s = s0 + 16 * u + (tid >> 4), sc = s < S ? s : S - 1;
        const size_t in = (((size_t)b * S + sc) * H + h) * 64 + d;
        xq[u] = load4u(q + in);
        xk[u] = load4u(k + in);
        xv[u] = load4u(v + in);
        if (gate) xg[u] = load4u(gate + in);
        rc[u] = make_float2(1.f, 1.f);
        rs[u] = make_float2(0.f, 0.f);
        if (rope) {
            rc[u] = *reinterpret_cast<const float2*>(rope_cos + (size_t)sc * 32 + d / 2);
            rs[u] = *reinterpret_cast<const float2*>(rope_sin + (size_t)sc * 32 + d / 2);
        }
    }
    // The head norm and the rotation of a token's four dimensions.
    auto head = [&](const float4& x, const float* norm, const float2& c, const float2& sn) {
        float4 y = x;
        if (norm) {
            const float r = rsqrtf(row16_sum(x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w) * (1.f / 64.f) + eps);
            const float4 w = *reinterpret_cast<const float4*>(norm + h * 64 + d);
            y = make_float4(x.x * (r * w.x), x.y * (r * w.y), x.z * (r * w.z), x.w * (r * w.w));
        }
        if (rope)
            y = make_float4(y.x * c.x - y.y * sn.x, y.x * sn.x + y.y * c.x, y.z * c.y - y.w * sn.y,
                            y.z * sn.y + y.w * c.y);
        return y;
    };
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int sl = 16 * u + (tid >> 4), s = s0 + sl;
        const float4 yq = head(xq[u], q_norm, rc[u], rs[u]), yk = head(xk[u], k_norm, rc[u], rs[u]);
        *reinterpret_cast<float4*>(&vs[sl][d]) = s < S ? xv[u] : make_float4(0.f, 0.f, 0.f, 0.f);
        if (s >= S) continue;
        const size_t o = (((size_t)b * H + h) * S + s) * 64 + d;
        store4<T>(Q + o, yq.x * q_scale, yq.y * q_scale, yq.z * q_scale, yq.w * q_scale);
        store4<T>(K + o, yk.x, yk.y, yk.z, yk.w);
        auto sig = [&](float x) { return gate ? 1.f / (1.f + expf(-x)) : 1.f; };
        store4<T>(G + ((size_t)b * S + s) * H * 64 + h * 64 + d, sig(xg[u].x), sig(xg[u].y), sig(xg[u].z),
                  sig(xg[u].w));
    }
    __syncthreads();
    // V^T row (b, h, dd), positions 8 seg .. 8 seg + 7 of this 32-key group.
    const int dd = tid >> 2, seg = tid & 3;
    alignas(16) T row[8];
#pragma unroll
    for (int j = 0; j < 8; j++) row[j] = from_f32<T>(vs[vt_src<T>(8 * seg + j)][dd]);
    T* dst = Vt + (((size_t)b * H + h) * 64 + dd) * vt_stride + s0 + 8 * seg;
    constexpr int PER = 16 / sizeof(T);  // elements per 16-byte store
#pragma unroll
    for (int j = 0; j < 8; j += PER) *reinterpret_cast<uint4*>(dst + j) = *reinterpret_cast<const uint4*>(row + j);
}

}  // namespace

template <typename T>
void launch_attn_op_stage(const float* q, const float* k, const float* v, const float* gate, const float* q_norm,
                          const float* k_norm, const float* rope_cos, const float* rope_sin, int B, int S, int H,
                          float eps, float q_scale, int vt_stride, T* Q, T* K, T* Vt, T* G, hipStream_t st) {
    // vt_stride is S rounded up to 64: every block's V^T columns lie inside it, and the blocks
    // past S clear the rest.
    const dim3 grid(vt_stride / 32, H, B);
    attn_op_stage_kernel<T><<<grid, 256, 0, st>>>(q, k, v, gate, q_norm, k_norm, rope_cos, rope_sin, S, H, eps,
                                                  q_scale, vt_stride, Q, K, Vt, G);
}
template void launch_attn_op_stage<bf16>(const float*, const float*, const float*, const float*, const float*,
                                         const float*, const float*, const float*, int, int, int, float, float, int,
                                         bf16*, bf16*, bf16*, bf16*, hipStream_t);
template void launch_attn_op_stage<float>(const float*, const float*, const float*, const float*, const float*,
                                          const float*, const float*, const float*, int, int, int, float, float, int,
                                          float*, float*, float*, float*, hipStream_t);

}  // namespace irodori
