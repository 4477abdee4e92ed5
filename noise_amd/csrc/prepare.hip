// A parameter update's preparation in one launch: every matrix rounded to bf16 (and laid out for the block kernel),
// every table and scalar copied. As separate casts, copies and layout passes it was 99 launches of 1.4 to 5 us for
// the 60 parameters, most of the time a small population takes.
#include "common.hpp"
#include "mfma.hpp"
#include "tile.hpp"

namespace noise {
namespace {

constexpr int kChunk = 256 * 8;  // elements per workgroup

struct PrepareArgs {
    noise_weight_t e[NOISE_WEIGHTS_MAX];
    int start[NOISE_WEIGHTS_MAX + 1];  // first workgroup of each entry
    int count;
};

// Each parameter is read once, 8 elements per thread. Bound by HBM: 151 MB in and 141 MB out for the 60 parameters.
__global__ __launch_bounds__(256) void prepare_kernel(PrepareArgs p) {
    int k = 0;
    while (k + 1 < p.count && p.start[k + 1] <= (int)blockIdx.x) ++k;
    const noise_weight_t &w = p.e[k];
    const int64_t i = ((int64_t)(blockIdx.x - p.start[k]) * 256 + threadIdx.x) * 8;
    if (i >= w.numel) return;
    const bool whole = i + 8 <= w.numel, wide = whole && ((uintptr_t)w.src & 15) == 0;
    float v[8];
    if (w.src_bf16) {
        const __bf16 *s = static_cast<const __bf16 *>(w.src) + i;
        if (wide) {
            const bf16x8 q = load_bf16x8(s);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (float)q[e];
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = i + e < w.numel ? (float)s[e] : 0.f;
        }
    } else {
        const float *s = static_cast<const float *>(w.src) + i;
        if (wide) {
            const float4 a = ld4(s), b = ld4(s + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = i + e < w.numel ? s[e] : 0.f;
        }
    }
    if (w.kind == NOISE_WEIGHT_BF16) {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (__bf16)v[e];
        __bf16 *d = static_cast<__bf16 *>(w.dst) + i;
        if (!w.dst) {
        } else if (whole) {
            store_bf16x8(d, o);
        } else {
            for (int e = 0; i + e < w.numel; ++e) d[e] = o[e];
        }
        if (w.dst_block) {
            // the block kernel's column order (block_layout_kernel): source group s of 4 within every 32 columns goes to
            // group 2 s (s < 4) or 2 (s - 4) + 1
            __bf16 *b = static_cast<__bf16 *>(w.dst_block) + (i & ~(int64_t)31);
            const int s0 = (int)(i & 31) >> 2;
            const int pos = s0 < 4 ? 2 * s0 : 2 * (s0 - 4) + 1;
            store_bf16x4(b + 4 * pos, bf16x4{o[0], o[1], o[2], o[3]});
            store_bf16x4(b + 4 * pos + 8, bf16x4{o[4], o[5], o[6], o[7]});
        }
    } else {
        if (w.kind == NOISE_WEIGHT_FP32_ROUNDED) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = bfr(v[e]);
        }
        float *d = static_cast<float *>(w.dst) + i;
        if (whole) {
            st4(d, float4{v[0], v[1], v[2], v[3]});
            st4(d + 4, float4{v[4], v[5], v[6], v[7]});
        } else {
            for (int e = 0; i + e < w.numel; ++e) d[e] = v[e];
        }
    }
}

}  // namespace
}  // namespace noise

using namespace noise;

extern "C" int noise_weights_prepare(const noise_weight_t *weights, int count, noise_stream_t stream) {
    clear_error();
    const char *fn = "noise_weights_prepare";
    NOISE_CHECK_ARG(weights && count >= 1 && count <= NOISE_WEIGHTS_MAX, "%s: 1 .. %d entries, got %d", fn,
                    NOISE_WEIGHTS_MAX, count);
    PrepareArgs p;
    int64_t groups = 0;
    p.count = count;
    for (int i = 0; i < count; ++i) {
        const noise_weight_t &w = weights[i];
        NOISE_CHECK_ARG(w.src && (w.dst || w.dst_block) && w.numel > 0 && aligned(w.dst, 16) && aligned(w.src, w.src_bf16 ? 2 : 4),
                        "%s: entry %d: NULL, empty or misaligned", fn, i);
        NOISE_CHECK_ARG(w.kind >= NOISE_WEIGHT_BF16 && w.kind <= NOISE_WEIGHT_FP32_ROUNDED, "%s: entry %d: unknown kind %d",
                        fn, i, w.kind);
        NOISE_CHECK_ARG(!w.dst_block || (w.kind == NOISE_WEIGHT_BF16 && w.numel % 32 == 0 && aligned(w.dst_block, 16)),
                        "%s: entry %d: the block layout is for bf16 rows of whole 32 columns", fn, i);
        p.e[i] = w;
        p.start[i] = (int)groups;
        groups += (w.numel + kChunk - 1) / kChunk;
        NOISE_CHECK_ARG(groups <= INT32_MAX, "%s: too many elements", fn);
    }
    p.start[count] = (int)groups;
    hipLaunchKernelGGL(prepare_kernel, dim3((unsigned)groups), dim3(256), 0, (hipStream_t)stream, p);
    return launch_status(fn);
}
