// The cached context beside its projections: speaker-KV scaling (kv_scaling.rs:10-60), an
// HBM-bound elementwise pass over the device K / V^T copies the attention reads, and the
// device build's state operand, masks and zeroed tails.  (The sampler's per-evaluation
// update runs in the output head, final_kernel.)
#include "common.hpp"
#include "kernels.hpp"

namespace irodori {

namespace {

// One thread per (row, head, key j, 8 dims) of K and the same for V^T.  V^T keys sit at
// vt_pos_bf16 (bf16_order) or vt_pos_f32.
template <typename T>
__global__ __launch_bounds__(256) void scale_ctx_aux_kernel(const T* __restrict__ src_k, const T* __restrict__ src_v,
                                                            T* __restrict__ dst_k, T* __restrict__ dst_v, int rows,
                                                            int rows_scaled, int H, int Dh, bool bf16_order, int T1,
                                                            int vs1, int t_ctx, int aux_start, float factor) {
    const int d8n = Dh / 8;
    const long total = (long)rows * H * T1 * d8n;
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int d8 = (int)(idx % d8n);
    const long rhj = idx / d8n;
    const int j = (int)(rhj % T1);
    const long rh = rhj / T1;
    const int row = (int)(rh / H);
    const bool scale = row < rows_scaled && j >= aux_start && j < t_ctx;
    const bool copy = src_k != dst_k;
    if (!scale && !copy) return;
    const int pos = bf16_order ? vt_pos_bf16(j) : vt_pos_f32(j);
    for (int d = 8 * d8; d < 8 * d8 + 8; d++) {
        const size_t ko = ((size_t)rh * T1 + j) * Dh + d;
        const size_t vo = ((size_t)rh * Dh + d) * vs1 + pos;
        const float kf = static_cast<float>(src_k[ko]), vf = static_cast<float>(src_v[vo]);
        dst_k[ko] = scale ? static_cast<T>(kf * factor) : src_k[ko];
        dst_v[vo] = scale ? static_cast<T>(vf * factor) : src_v[vo];
    }
}

// One thread per operand element: the row is a few KB, so one launch per segment is bound by
// its launch; it replaces a scalar conversion on the host (0.8 M elements at 631 tokens of 1280).
template <typename T>
__global__ __launch_bounds__(256) void ctx_states_kernel(const float* __restrict__ src, long n, int dim, int kpad,
                                                         T* __restrict__ dst) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const long r = i / kpad;
    const int k = (int)(i - r * kpad);
    dst[i] = from_f32<T>(k < dim ? src[r * dim + k] : 0.f);
}

// Block (h, l): the head's K rows and V^T columns past t_ctx; head 0 also the layer's masks,
// one wavefront per 64-key tile at a time.  Every layer of a row in one launch, where each
// layer took two fills of its whole K / V and three uploads with a wait.
template <typename T>
__global__ __launch_bounds__(256) void ctx_finish_kernel(T* __restrict__ K, T* __restrict__ V, size_t nk, size_t nv,
                                                         const uint8_t* __restrict__ mask, float* __restrict__ fmask,
                                                         int* __restrict__ tile_on, unsigned long long* __restrict__ bits,
                                                         size_t mask_layer, size_t tile_layer, int Dh, int t_ctx,
                                                         int T1, int vs1, bool bf16_order) {
    const int h = blockIdx.x, l = blockIdx.y, tid = threadIdx.x;
    T* k = K + l * nk + ((size_t)h * T1 + t_ctx) * Dh;
    for (int i = tid; i < (T1 - t_ctx) * Dh; i += 256) k[i] = from_f32<T>(0.f);
    T* v = V + l * nv + (size_t)h * Dh * vs1;
    const int tail = vs1 - t_ctx;
    for (int i = tid; i < tail * Dh; i += 256) {
        const int d = i / tail, key = t_ctx + i % tail;
        v[(size_t)d * vs1 + (bf16_order ? vt_pos_bf16(key) : vt_pos_f32(key))] = from_f32<T>(0.f);
    }
    if (h != 0) return;
    for (int t = tid >> 6; t < vs1 / 64; t += 4) {
        const int key = 64 * t + (tid & 63);
        const bool ok = key < t_ctx && mask[key] != 0;
        if (key < T1) fmask[l * mask_layer + key] = ok ? 1.f : 0.f;
        const unsigned long long w = __ballot(ok);
        if ((tid & 63) == 0) {
            tile_on[l * tile_layer + t] = w != 0;
            bits[l * tile_layer + t] = w;
        }
    }
}

}  // namespace

template <typename T>
void launch_ctx_states(const float* src, int rows, int dim, int kpad, T* dst, hipStream_t st) {
    const long n = (long)rows * kpad;
    if (n <= 0) return;
    ctx_states_kernel<T><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(src, n, dim, kpad, dst);
}
template void launch_ctx_states<bf16>(const float*, int, int, int, bf16*, hipStream_t);
template void launch_ctx_states<float>(const float*, int, int, int, float*, hipStream_t);

template <typename T>
void launch_ctx_finish(T* K, T* V, size_t nk, size_t nv, const uint8_t* mask, float* fmask, int* tile_on,
                       unsigned long long* bits, size_t mask_layer, size_t tile_layer, int layers, int H, int Dh,
                       int t_ctx, int T1, int vs1, bool bf16_order, hipStream_t st) {
    ctx_finish_kernel<T><<<dim3(H, layers), 256, 0, st>>>(K, V, nk, nv, mask, fmask, tile_on, bits, mask_layer,
                                                          tile_layer, Dh, t_ctx, T1, vs1, bf16_order);
}
template void launch_ctx_finish<bf16>(bf16*, bf16*, size_t, size_t, const uint8_t*, float*, int*, unsigned long long*,
                                      size_t, size_t, int, int, int, int, int, int, bool, hipStream_t);
template void launch_ctx_finish<float>(float*, float*, size_t, size_t, const uint8_t*, float*, int*,
                                       unsigned long long*, size_t, size_t, int, int, int, int, int, int, bool,
                                       hipStream_t);

template <typename T>
void launch_scale_ctx_aux(const T* src_k, const T* src_v, T* dst_k, T* dst_v, int rows, int rows_scaled, int H,
                          int Dh, bool bf16_order, int T1, int vs1, int t_ctx, int aux_start, float factor,
                          hipStream_t st) {
    const long total = (long)rows * H * T1 * (Dh / 8);
    scale_ctx_aux_kernel<T><<<(unsigned)((total + 255) / 256), 256, 0, st>>>(
        src_k, src_v, dst_k, dst_v, rows, rows_scaled, H, Dh, bf16_order, T1, vs1, t_ctx, aux_start, factor);
}

template void launch_scale_ctx_aux<bf16>(const bf16*, const bf16*, bf16*, bf16*, int, int, int, int, bool, int,
                                         int, int, int, float, hipStream_t);
template void launch_scale_ctx_aux<float>(const float*, const float*, float*, float*, int, int, int, int, bool, int,
                                          int, int, int, float, hipStream_t);

}  // namespace irodori
