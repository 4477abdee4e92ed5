// The `lowrank` drop-in (eggroll.py:56-58) in autocast's form, for any shape:
//   y[m, t, o] = bf16(x[m, t] . W[o]) + sign[m] * bf16(x[m, t] . bf16(b[dir])) * a[dir, o]
// with bf16 operands and fp32 sums; y fp32 [m][T][out].
//
//   operands   one pass over x, W (and b): bf16 rows padded to whole 64-wide k steps, and the x . b dots
//   product    MFMA tiles over the flattened rows (m, t), the rank-1 term added in the epilogue
//   narrow     a few outputs of a short contraction (the value-embedding gate's [8, 32] weight on h[..., :32],
//              eggroll.py:88): one launch on the caller's tensors as they are
//
// 24 x 1000 rows, 512 -> 2048, fp32 inputs: 20 us for the operands and 94 for the product; one thread per output element
// with a serial dot, which served this shape before, took 93.9 ms. 16 x 256 rows, 32 -> 8: the narrow kernel 4.1 us.
#include "common.hpp"
#include "mfma.hpp"
#include "tile.hpp"

namespace noise {
namespace {

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// elements k .. k + 4 of a row of n, zeros past its end; vec: the row is 4-element aligned and n % 4 == 0
template <bool FP32>
__device__ __forceinline__ void load4(const void *row, int k, int n, bool vec, float (&v)[4]) {
    if constexpr (FP32) {
        const float *p = static_cast<const float *>(row);
        if (vec && k < n) {
            const float4 q = ld4(p + k);
            v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = k + e < n ? p[k + e] : 0.f;
        }
    } else {
        const __bf16 *p = static_cast<const __bf16 *>(row);
        if (vec && k < n) {
            const bf16x4 q = load_bf16x4(p + k);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (float)q[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = k + e < n ? (float)p[k + e] : 0.f;
        }
    }
}

struct OperandArgs {
    const void *x;            // [m][T][n_in], fp32 or bf16, element strides xs_m, xs_t
    int64_t xs_m, xs_t, rows;
    int tokens, n_in, kp, dir_div;
    const void *w;            // [n_out][n_in], fp32 or bf16
    int n_out;
    const float *b;           // direction rows
    int64_t b_stride;
    int b_rows;               // > 0: rows n_out .. of wb
    __bf16 *xb, *wb;          // [rows][kp] (NULL: x is used as it is), [n_out + b_rows][kp]
    float *dots;              // [rows] x . bf16(b[dir]), or NULL
    int x_fp32, w_fp32, x_vec, w_vec, b_vec;
    int64_t x_blocks;         // workgroups of x's rows
    int64_t first;            // this launch's first workgroup
};

// A launch has fewer than 2^32 threads (one of more is cut short without an error): a call of more workgroups than this
// goes in several launches.
constexpr int64_t kLaunchGroups = 1 << 23;

// One wave per row: x rows first, then W's, then b's. Reads each tensor once and writes its bf16 form once;
// bound by those bytes (24,000 x 512 fp32: 49 MB in, 25 MB out).
__global__ __launch_bounds__(256) void lowrank_operands_kernel(OperandArgs p) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const void *src;
    __bf16 *dst;
    const float *br = nullptr;
    float *dot = nullptr;
    bool fp32, vec;
    const int64_t block = p.first + blockIdx.x;
    if (block < p.x_blocks) {
        const int64_t r = block * 4 + wave;
        if (r >= p.rows) return;
        const int64_t m = r / p.tokens, t = r - m * p.tokens;
        fp32 = p.x_fp32;
        vec = p.x_vec;
        src = static_cast<const char *>(p.x) + (m * p.xs_m + t * p.xs_t) * (fp32 ? 4 : 2);
        dst = p.xb ? p.xb + r * p.kp : nullptr;
        if (p.dots) {
            br = p.b + (m / p.dir_div) * p.b_stride;
            dot = p.dots + r;
        }
    } else {
        const int64_t r = (block - p.x_blocks) * 4 + wave;
        if (r >= p.n_out + p.b_rows) return;
        const bool is_w = r < p.n_out;
        fp32 = is_w ? p.w_fp32 : true;
        vec = is_w ? p.w_vec : p.b_vec;
        src = is_w ? static_cast<const char *>(p.w) + r * p.n_in * (fp32 ? 4 : 2)
                   : reinterpret_cast<const char *>(p.b + (r - p.n_out) * p.b_stride);
        dst = p.wb + r * p.kp;
    }
    float acc = 0.f;
    for (int k = lane * 4; k < p.kp; k += 256) {
        float v[4];
        if (fp32) load4<true>(src, k, p.n_in, vec, v);
        else load4<false>(src, k, p.n_in, vec, v);
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (__bf16)v[e];
        if (dst) store_bf16x4(dst + k, o);
        if (br) {
            float bv[4];
            load4<true>(br, k, p.n_in, p.b_vec, bv);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc += (float)o[e] * bfr(bv[e]);
        }
    }
    if (dot) {
        acc = wave_sum(acc);
        if (lane == 0) *dot = acc;
    }
}

struct ProductArgs {
    const __bf16 *x, *w;      // [rows][ldx], [N][K]
    int64_t rows, ldx;
    int K, N, tokens, dir_div, tiles_n, tiles_t;
    const float *a;           // rank-1 rows, or NULL
    int64_t a_stride;
    const float *sign, *dots;
    float *y, *y2;            // features < split to y [rows][split], the others to y2 [rows][ld2]
    int split;
    int64_t ld2;
    int vec;                  // features in whole, 16 B aligned groups of 4
};

// y rows from MFMA tiles of BN features x BM rows (the K loop of tile.hpp, its operand rows clamped to the last
// valid one, whose surplus results are not stored). The rows of all members form one list, so a length that is
// no multiple of the tile leaves no partial tile per member. Each wave passes its tile through LDS so that a
// store instruction covers two rows of 512 contiguous bytes.
template <int NW, int BN, int BM>
__global__ __launch_bounds__(NW * 64) void lowrank_product_kernel(ProductArgs p) {
    using M = Mma<NW, BN, BM, 64, 2>;
    constexpr int kStage = NW * 32 * 512;  // 32 rows x 128 features fp32 per wave
    constexpr int kLds = cmax(M::LDS_BYTES, kStage);
    __shared__ __attribute__((aligned(16))) char lds[kLds];
    __shared__ float s_corr[BM];
    __shared__ int s_dir[BM];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 31, hf = lane >> 5;
    int nt, tt;
    tile_order(blockIdx.x, p.tiles_n, p.tiles_t, tt, nt);
    const int n0 = nt * BN;
    const int64_t r0 = (int64_t)tt * BM;
    const int64_t left = p.rows - r0;
    const int nx = left < BM ? (int)left : BM, nw = p.N - n0 < BN ? p.N - n0 : BN;
    if (p.a) {
        for (int i = tid; i < nx; i += NW * 64) {
            const int64_t m = (r0 + i) / p.tokens;
            s_corr[i] = p.sign[m] * bfr(p.dots[r0 + i]);
            s_dir[i] = (int)(m / p.dir_div);
        }
    }
    const int wn0 = M::wn0(wave), wm0 = M::wm0(wave);
    f32x16 acc[4][2];
    M::template run<true>(p.w + (int64_t)n0 * p.K, p.K, p.x + r0 * p.ldx, p.ldx, p.K, lds, acc, tid, wn0, wm0, NoTail{},
                          nw - 1, nx - 1);
    // the K loop ended with a barrier: its stages hold the waves' output tiles, [32 rows][32 chunks of 4 features],
    // chunk c of row r at c ^ r (both the writes and the reads below cover the banks evenly)
    char *st = lds + wave * (32 * 512);
    const int fl = 4 * j, f = n0 + wn0 + fl;
    int cur = -1;
    float av[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        wave_lds_sync();
#pragma unroll
        for (int fb = 0; fb < 4; ++fb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = 8 * fb + 2 * g + hf;
                const f32x16 &v = acc[fb][tb];
                st4(reinterpret_cast<float *>(st + j * 512 + ((c ^ j) & 31) * 16),
                    float4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]});
            }
        wave_lds_sync();
#pragma unroll 4
        for (int it = 0; it < 16; ++it) {
            const int tl = 2 * it + hf, i = wm0 + 32 * tb + tl;
            if (i >= nx || f >= p.N) continue;
            const float4 v = ld4(reinterpret_cast<const float *>(st + tl * 512 + ((j ^ tl) & 31) * 16));
            float o[4] = {bfr(v.x), bfr(v.y), bfr(v.z), bfr(v.w)};
            if (p.a) {
                const int dir = s_dir[i];
                if (dir != cur) {
                    cur = dir;
                    const float *ar = p.a + dir * p.a_stride + f;
                    if (p.vec) {
                        const float4 q = ld4(ar);
                        av[0] = q.x; av[1] = q.y; av[2] = q.z; av[3] = q.w;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) av[e] = f + e < p.N ? ar[e] : 0.f;
                    }
                }
                const float c = s_corr[i];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] += c * av[e];
            }
            const int64_t r = r0 + i;
            if (p.vec) {
                float *dst = f < p.split ? p.y + r * p.split + f : p.y2 + r * p.ld2 + (f - p.split);
                st4(dst, float4{o[0], o[1], o[2], o[3]});
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (f + e < p.N) p.y[r * p.split + f + e] = o[e];
            }
        }
    }
}

struct NarrowArgs {
    const void *x, *w;
    int64_t xs_m, xs_t, rows;
    int tokens, n_in, n_out, dir_div, x_vec, w_vec, b_vec;
    const float *a, *b;
    int64_t a_stride, b_stride;
    const float *sign;
    float *y;
    unsigned first;           // this launch's first tile
};

// 32 rows x 8 outputs per workgroup, eight lanes per row: each lane takes 4 of every 32 k for the eight products
// and the dot, the weights wait in LDS as rounded floats, and the lane sums meet by shuffles. Any strides and
// widths. At 4096 rows, 32 -> 8 it is bound by its launch.
constexpr int kNarrowK = 256;
template <bool XF, bool WF>
__global__ __launch_bounds__(256) void lowrank_narrow_kernel(NarrowArgs p) {
    __shared__ __attribute__((aligned(16))) float ws[8][kNarrowK];
    const int tid = threadIdx.x, l = tid & 7, groups = (p.n_out + 7) / 8;
    const unsigned tile = p.first + blockIdx.x;
    const int o0 = (int)(tile % groups) * 8;
    const int64_t row = (int64_t)(tile / groups) * 32 + (tid >> 3);
    const bool live = row < p.rows;
    const int64_t m = live ? row / p.tokens : 0, t = live ? row - m * p.tokens : 0, dir = m / p.dir_div;
    const char *xr = static_cast<const char *>(p.x) + (m * p.xs_m + t * p.xs_t) * (XF ? 4 : 2);
    const float *br = p.a ? p.b + dir * p.b_stride : nullptr;
    float acc[8], dot = 0.f;
#pragma unroll
    for (int o = 0; o < 8; ++o) acc[o] = 0.f;
    for (int k0 = 0; k0 < p.n_in; k0 += kNarrowK) {
        const int kn = p.n_in - k0 < kNarrowK ? p.n_in - k0 : kNarrowK;
        if (k0) __syncthreads();
        for (int i = tid; i < 8 * (kNarrowK / 4); i += 256) {
            const int o = i / (kNarrowK / 4), k = (i % (kNarrowK / 4)) * 4;
            if (k >= kn) continue;
            float v[4] = {0.f, 0.f, 0.f, 0.f};
            if (o0 + o < p.n_out)
                load4<WF>(static_cast<const char *>(p.w) + (int64_t)(o0 + o) * p.n_in * (WF ? 4 : 2), k0 + k, p.n_in,
                          p.w_vec, v);
            st4(&ws[o][k], float4{bfr(v[0]), bfr(v[1]), bfr(v[2]), bfr(v[3])});
        }
        __syncthreads();
        for (int k = 4 * l; k < kn; k += 32) {
            float xv[4];
            load4<XF>(xr, k0 + k, p.n_in, p.x_vec, xv);
#pragma unroll
            for (int e = 0; e < 4; ++e) xv[e] = bfr(xv[e]);
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const float4 wv = ld4(&ws[o][k]);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[o] += xv[e] * f4get(wv, e);
            }
            if (br) {
                float bv[4];
                load4<true>(br, k0 + k, p.n_in, p.b_vec, bv);
#pragma unroll
                for (int e = 0; e < 4; ++e) dot += xv[e] * bfr(bv[e]);
            }
        }
    }
    float mine = 0.f;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        float v = acc[o];
#pragma unroll
        for (int s = 1; s < 8; s <<= 1) v += __shfl_xor(v, s, 64);
        mine = o == l ? v : mine;
    }
#pragma unroll
    for (int s = 1; s < 8; s <<= 1) dot += __shfl_xor(dot, s, 64);
    const int o = o0 + l;
    if (!live || o >= p.n_out) return;
    float v = bfr(mine);
    if (p.a) v += p.sign[m] * bfr(dot) * p.a[dir * p.a_stride + o];
    p.y[row * p.n_out + o] = v;
}

// elements 4-aligned for load4's vector form
bool rows_vec(const void *p, bool fp32, int64_t n, int64_t s0, int64_t s1) {
    return aligned(p, fp32 ? 16 : 8) && n % 4 == 0 && s0 % 4 == 0 && s1 % 4 == 0;
}

int narrow_launch(const noise_population_t *pop, noise_view_t x, bool xf, int64_t n_in, const void *w, bool wf,
                  int64_t n_out, const noise_rank1_t *r1, float *y, noise_stream_t stream, const char *fn) {
    NOISE_CHECK_ARG(pop && pop->members > 0 && pop->tokens > 0 && pop->dir_div >= 1, "%s: bad population", fn);
    NOISE_CHECK_ARG(x.ptr && w && y && n_in > 0 && n_out > 0, "%s: NULL pointer or empty shape", fn);
    NOISE_CHECK_ARG(n_in <= INT32_MAX && n_out <= INT32_MAX, "%s: width too large", fn);
    NOISE_CHECK_ARG(pop->members * pop->tokens * n_out < (1ll << 38), "%s: output too large", fn);
    const bool noisy = r1 && r1->a;
    NOISE_CHECK_ARG(!noisy || (pop->sign && r1->b), "%s: noise needs sign and b rows", fn);
    NarrowArgs p;
    p.x = x.ptr; p.w = w; p.xs_m = x.sm; p.xs_t = x.st; p.rows = pop->members * pop->tokens;
    p.tokens = (int)pop->tokens; p.n_in = (int)n_in; p.n_out = (int)n_out; p.dir_div = (int)pop->dir_div;
    p.x_vec = rows_vec(x.ptr, xf, n_in, x.sm, x.st);
    p.w_vec = rows_vec(w, wf, n_in, 0, 0);
    p.a = noisy ? r1->a : nullptr; p.b = noisy ? r1->b : nullptr;
    p.a_stride = noisy ? r1->a_stride : 0; p.b_stride = noisy ? r1->b_stride : 0;
    p.b_vec = noisy && rows_vec(r1->b, true, n_in, r1->b_stride, 0);
    p.sign = pop->sign; p.y = y;
    const int64_t tiles = (p.rows + 31) / 32 * ((n_out + 7) / 8);
    NOISE_CHECK_ARG(tiles <= INT32_MAX, "%s: output too large", fn);
    hipStream_t st = (hipStream_t)stream;
    for (int64_t first = 0; first < tiles; first += kLaunchGroups) {
        const dim3 grid((unsigned)(tiles - first < kLaunchGroups ? tiles - first : kLaunchGroups));
        p.first = (unsigned)first;
        if (xf && wf) hipLaunchKernelGGL((lowrank_narrow_kernel<true, true>), grid, dim3(256), 0, st, p);
        else if (xf) hipLaunchKernelGGL((lowrank_narrow_kernel<true, false>), grid, dim3(256), 0, st, p);
        else if (wf) hipLaunchKernelGGL((lowrank_narrow_kernel<false, true>), grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL((lowrank_narrow_kernel<false, false>), grid, dim3(256), 0, st, p);
    }
    return launch_status(fn);
}

}  // namespace
}  // namespace noise

using namespace noise;

extern "C" int noise_lowrank_rows(const noise_population_t *pop, noise_view_t x, int64_t n_in, const void *w,
                                  int64_t n_out, const noise_rank1_t *r1, float *y, noise_stream_t stream) {
    clear_error();
    return narrow_launch(pop, x, false, n_in, w, false, n_out, r1, y, stream, "noise_lowrank_rows");
}

extern "C" int noise_lowrank_narrow(const noise_population_t *pop, noise_view_t x, int x_fp32, int64_t n_in,
                                    const void *w, int w_fp32, int64_t n_out, const noise_rank1_t *r1, float *y,
                                    noise_stream_t stream) {
    clear_error();
    return narrow_launch(pop, x, x_fp32 != 0, n_in, w, w_fp32 != 0, n_out, r1, y, stream, "noise_lowrank_narrow");
}

extern "C" int noise_lowrank_operands(const noise_population_t *pop, noise_view_t x, int x_fp32, int64_t n_in,
                                      const void *w, int w_fp32, int64_t n_out, const float *b, int64_t b_stride,
                                      int64_t b_rows, int64_t k_pad, void *xb, void *wb, float *dots,
                                      noise_stream_t stream) {
    clear_error();
    const char *fn = "noise_lowrank_operands";
    NOISE_CHECK_ARG(pop && pop->members > 0 && pop->tokens > 0 && pop->dir_div >= 1, "%s: bad population", fn);
    NOISE_CHECK_ARG(x.ptr && w && wb && n_in > 0 && n_out > 0, "%s: NULL pointer or empty shape", fn);
    NOISE_CHECK_ARG(k_pad >= n_in && k_pad % 64 == 0 && k_pad <= (1 << 21), "%s: k_pad must be n_in in whole 64s", fn);
    NOISE_CHECK_ARG(n_out + b_rows <= INT32_MAX && b_rows >= 0 && pop->tokens <= INT32_MAX, "%s: shape too large", fn);
    NOISE_CHECK_ARG((!dots && b_rows == 0) || b, "%s: dots and direction rows need b", fn);
    NOISE_CHECK_ARG(aligned(wb, 16) && (!xb || aligned(xb, 16)), "%s: 16 B alignment", fn);
    OperandArgs p;
    p.x = x.ptr; p.xs_m = x.sm; p.xs_t = x.st; p.rows = pop->members * pop->tokens;
    p.tokens = (int)pop->tokens; p.n_in = (int)n_in; p.kp = (int)k_pad; p.dir_div = (int)pop->dir_div;
    p.w = w; p.n_out = (int)n_out; p.b = b; p.b_stride = b_stride; p.b_rows = (int)b_rows;
    p.xb = (__bf16 *)xb; p.wb = (__bf16 *)wb; p.dots = dots;
    p.x_fp32 = x_fp32 != 0; p.w_fp32 = w_fp32 != 0;
    p.x_vec = rows_vec(x.ptr, x_fp32, n_in, x.sm, x.st);
    p.w_vec = rows_vec(w, w_fp32, n_in, 0, 0);
    p.b_vec = b && rows_vec(b, true, n_in, b_stride, 0);
    p.x_blocks = xb || dots ? (p.rows + 3) / 4 : 0;
    const int64_t blocks = p.x_blocks + (n_out + b_rows + 3) / 4;
    NOISE_CHECK_ARG(blocks <= INT32_MAX, "%s: too many rows", fn);
    for (p.first = 0; p.first < blocks; p.first += kLaunchGroups) {
        const int64_t n = blocks - p.first < kLaunchGroups ? blocks - p.first : kLaunchGroups;
        hipLaunchKernelGGL(lowrank_operands_kernel, dim3((unsigned)n), dim3(256), 0, (hipStream_t)stream, p);
    }
    return launch_status(fn);
}

extern "C" int noise_lowrank_product(const noise_population_t *pop, const void *x, int64_t ldx, int64_t rows,
                                     const void *w, int64_t K, int64_t N, const noise_rank1_t *r1, const float *dots,
                                     float *y, int64_t split, float *y2, int64_t ld2, noise_stream_t stream) {
    clear_error();
    const char *fn = "noise_lowrank_product";
    NOISE_CHECK_ARG(pop && pop->members > 0 && pop->tokens > 0 && pop->dir_div >= 1, "%s: bad population", fn);
    NOISE_CHECK_ARG(x && w && y && rows > 0 && N > 0 && N <= INT32_MAX, "%s: NULL pointer or empty shape", fn);
    NOISE_CHECK_ARG(K > 0 && K % 64 == 0 && K <= (1 << 21), "%s: K must be a multiple of 64", fn);
    NOISE_CHECK_ARG(aligned(x, 16) && aligned(w, 16) && ldx % 8 == 0 && ldx >= 0 && ldx <= (1 << 21), "%s: x or w rows misaligned",
                    fn);
    NOISE_CHECK_ARG(split > 0 && split <= N && (split == N || (y2 && ld2 >= N - split)), "%s: bad output split", fn);
    const bool noisy = r1 && r1->a;
    NOISE_CHECK_ARG(!noisy || (pop->sign && dots && rows == pop->members * pop->tokens && split == N),
                    "%s: the rank-1 term needs sign, dots and every member's rows", fn);
    ProductArgs p;
    p.x = (const __bf16 *)x; p.w = (const __bf16 *)w; p.rows = rows; p.ldx = ldx;
    p.K = (int)K; p.N = (int)N; p.tokens = (int)pop->tokens; p.dir_div = (int)pop->dir_div;
    p.a = noisy ? r1->a : nullptr; p.a_stride = noisy ? r1->a_stride : 0;
    p.sign = pop->sign; p.dots = dots; p.y = y; p.y2 = y2; p.split = (int)split; p.ld2 = ld2;
    // a split output's last group of 4 may run past N into y2's row padding
    p.vec = split % 4 == 0 && aligned(y, 16) &&
            (split == N || (ld2 % 4 == 0 && ld2 >= (N - split + 3) / 4 * 4 && aligned(y2, 16))) &&
            (!noisy || (aligned(r1->a, 16) && r1->a_stride % 4 == 0));
    NOISE_CHECK_ARG(p.vec || split == N, "%s: a split output needs 16 B aligned groups of 4", fn);
    hipStream_t st = (hipStream_t)stream;
    // 256 x 256 tiles (one workgroup per CU) when they fill the chip's 256 CUs, 128 x 128 (two per CU) below
    const int64_t big = ((N + 255) / 256) * ((rows + 255) / 256);
    if (big >= 256) {
        p.tiles_n = (int)((N + 255) / 256);
        NOISE_CHECK_ARG(big < kLaunchGroups, "%s: too many tiles", fn);
        p.tiles_t = (int)((rows + 255) / 256);
        hipLaunchKernelGGL((lowrank_product_kernel<8, 256, 256>), dim3((unsigned)big), dim3(512), 0, st, p);
    } else {
        p.tiles_n = (int)((N + 127) / 128);
        p.tiles_t = (int)((rows + 127) / 128);
        hipLaunchKernelGGL((lowrank_product_kernel<2, 128, 128>), dim3((unsigned)(p.tiles_n * p.tiles_t)), dim3(128), 0, st, p);
    }
    return launch_status(fn);
}
