// The SDPA operator entry points (native_fa_sdpa_wgsl / native_fa_sdpa_f16_in,
// fused_sdpa_native.rs:220-302, fused_sdpa_native_f16.rs:181-200): argument checks and the
// kernel by dtype -- 16-bit operands on the row-major flash kernel (kernels_attn_nv.hip), f32
// on the generic one.  Neither needs device memory of its own, so irodori_op_sdpa and
// irodori_op_sdpa_noalloc run the same launch; the latter keeps its contract's refusals.
#include <atomic>

#include "../../include/irodori_hip.h"
#include "common.hpp"
#include "host.hpp"
#include "kernels.hpp"

using namespace irodori;

namespace {

int check_sdpa_args(int dtype, const void* q, const void* k, const void* v, int B, int H, int Sq, int Skv, int Dh,
                    const float* out) {
    IRO_REQUIRE(q && k && v && out, IRODORI_ERR_INVALID_ARG, "null argument");
    IRO_REQUIRE(B > 0 && H > 0 && Sq > 0 && Skv > 0, IRODORI_ERR_SHAPE, "SDPA dims must be positive");
    IRO_REQUIRE(Dh == 64 || Dh == 128, IRODORI_ERR_SHAPE, "head_dim must be 64 or 128");
    IRO_REQUIRE(dtype == IRODORI_DTYPE_F32 || dtype == IRODORI_DTYPE_BF16 || dtype == IRODORI_DTYPE_F16,
                IRODORI_ERR_DTYPE, "dtype must be F32, BF16 or F16");
    return IRODORI_OK;
}

template <typename T>
int sdpa_t(const void* q, const void* k, const void* v, const float* mask, int B, int H, int Sq, int Skv, int Dh,
           float scale, float* out, hipStream_t st) {
    AttnArgs<T> a{};
    a.Q = static_cast<const T*>(q);
    a.K0 = static_cast<const T*>(k);
    a.V0 = static_cast<const T*>(v);
    a.len0 = Skv; a.stride0 = Skv; a.mask0 = mask;
    a.B = B; a.H = H; a.Sq = Sq; a.scale = scale; a.out_mode = 1; a.Of = out;
    int rc;
    if constexpr (sizeof(T) == 2)
        rc = Dh == 64 ? launch_attention_nv<T, 64>(a, st) : launch_attention_nv<T, 128>(a, st);
    else
        rc = Dh == 64 ? launch_attention<T, 64>(a, st) : launch_attention<T, 128>(a, st);
    IRO_REQUIRE(rc == 0, IRODORI_ERR_SHAPE, "sdpa launch rejected the shape");
    return check_launch("sdpa");
}

int sdpa_run(int dtype, const void* q, const void* k, const void* v, const float* mask, int B, int H, int Sq,
             int Skv, int Dh, float scale, float* out, hipStream_t st) {
    if (dtype == IRODORI_DTYPE_BF16) return sdpa_t<bf16>(q, k, v, mask, B, H, Sq, Skv, Dh, scale, out, st);
    if (dtype == IRODORI_DTYPE_F16) return sdpa_t<f16>(q, k, v, mask, B, H, Sq, Skv, Dh, scale, out, st);
    return sdpa_t<float>(q, k, v, mask, B, H, Sq, Skv, Dh, scale, out, st);
}

// irodori_op_sdpa_noalloc's contract: 16-bit operands with Dh = 64 and at most 16384 keys are
// held to IRODORI_SDPA_SCRATCH_BYTES of Q, V^T and key bits.  (The kernels need no such buffer; callers
// may rely on the refusal.)
bool noalloc_bounded(int dtype, int Dh, int Skv) { return dtype != IRODORI_DTYPE_F32 && Dh == 64 && Skv <= 16384; }
size_t noalloc_bytes(int B, int H, int Sq, int Skv) {
    const size_t vs = (size_t)(Skv + 63) / 64 * 64;
    auto al = [](size_t n) { return (n + 255) / 256 * 256; };
    return al((size_t)B * H * Sq * 64 * 2) + al((size_t)B * H * 64 * vs * 2) + al((size_t)B * (vs / 64) * 8);
}

constexpr int kMaxDevices = 64;
std::atomic<bool> g_prepared[kMaxDevices] = {};

// The stream must be the current device's, and a device's first call must not be captured: it loads
// the code of the row-major kernel's variants and sets their LDS limits, so that no later call, captured or not, does.
int check_noalloc_stream(hipStream_t st) {
    int dev = -1;
    IRO_HIP_CHECK(hipGetDevice(&dev));
    if (st) {
        int sdev = -1;
        IRO_HIP_CHECK(hipStreamGetDevice(st, &sdev));
        IRO_REQUIRE(sdev == dev, IRODORI_ERR_INVALID_ARG,
                    "irodori_op_sdpa_noalloc: the stream belongs to device " + std::to_string(sdev) +
                        " but device " + std::to_string(dev) + " is current; make the stream's device current");
    }
    IRO_REQUIRE(dev >= 0 && dev < kMaxDevices, IRODORI_ERR_INVALID_ARG, "device index beyond the device table");
    if (!g_prepared[dev].load()) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        IRO_HIP_CHECK(hipStreamIsCapturing(st, &cs));
        IRO_REQUIRE(cs == hipStreamCaptureStatusNone, IRODORI_ERR_INVALID_ARG,
                    "irodori_op_sdpa_noalloc: the first call on a device must not be under graph capture; make "
                    "one call outside the capture first");
        IRO_HIP_CHECK(prepare_attention_nv());
        g_prepared[dev].store(true);
    }
    return IRODORI_OK;
}

}  // namespace

extern "C" {

int irodori_op_sdpa(int dtype, const void* q, const void* k, const void* v, const float* mask, int B, int H, int Sq,
                    int Skv, int Dh, float scale, float* out, void* stream) {
    IRO_GUARD_BEGIN
    IRO_TRY(check_sdpa_args(dtype, q, k, v, B, H, Sq, Skv, Dh, out));
    return sdpa_run(dtype, q, k, v, mask, B, H, Sq, Skv, Dh, scale, out, static_cast<hipStream_t>(stream));
    IRO_GUARD_END
}

int irodori_op_sdpa_noalloc(int dtype, const void* q, const void* k, const void* v, const float* mask, int B, int H,
                            int Sq, int Skv, int Dh, float scale, float* out, void* stream) {
    IRO_GUARD_BEGIN
    IRO_TRY(check_sdpa_args(dtype, q, k, v, B, H, Sq, Skv, Dh, out));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (noalloc_bounded(dtype, Dh, Skv)) {
        const size_t bytes = noalloc_bytes(B, H, Sq, Skv);
        IRO_REQUIRE(bytes <= IRODORI_SDPA_SCRATCH_BYTES, IRODORI_ERR_SHAPE,
                    "irodori_op_sdpa_noalloc: the operands of this shape take " + std::to_string(bytes) +
                        " bytes, above the entry point's " + std::to_string((size_t)IRODORI_SDPA_SCRATCH_BYTES) +
                        "; use irodori_op_sdpa");
        IRO_TRY(check_noalloc_stream(st));
    }
    return sdpa_run(dtype, q, k, v, mask, B, H, Sq, Skv, Dh, scale, out, st);
    IRO_GUARD_END
}

}  // extern "C"
