// The block kernel's work for few token tiles, shared out over the CUs by output features instead of kept in one
// workgroup per 128 tokens: four launches per block,
//
//   split_rows_kernel<NB, false>   x_mid = x + y W_o^T + rank-1, 16 NB of the 512 features per workgroup
//   split_fc_kernel                h = bf16(norm(x_mid)), hid = bf16(relu(h c_fc^T + rank-1)^2), a part of the units
//   split_rows_kernel<NB, true>    x_out = x_mid + hid c_proj^T + rank-1 [, mixing], 16 NB of the 512 features
//   split_qkv_kernel               the next block's gates, q, k, v from norm(x_out), a part of the 24 heads
//   (split_norm_kernel             the last block: the head's rows from norm(x_out))
//
// x_mid (fp32), hid (bf16) and x_out for the last launch pass through a workspace, in the order the lanes hold them: a
// wave's load or store is then 1 KiB in one piece instead of 16 rows of 64 B. A workgroup still holds 128 tokens of one
// member in 8 waves of 16 with the same lanes, products in the same order and the same reductions as block_kernel, and
// every workgroup that needs a row's norm forms it from the whole row: the results are block_kernel's bit for bit, so a
// loss does not depend on how many members are evaluated together. What it costs is the rows read again by each part
// and the launches; what it gives is CUs: 16 tiles (8 members x 256 tokens) take 67 us per block against 187 on 16
// workgroups (split_rows 10 and 17, split_fc 15, split_qkv 25; with rows in memory order 10, 23, 20 and 30). The
// launches are bound by what a CU can load (384 to 640 KiB per workgroup) and their own start (4 us when empty).
#pragma once
#include "common.hpp"
#include "mfma.hpp"
#include "qkv_phase.hpp"
#include "tile.hpp"

namespace noise {
namespace {

constexpr int kSplitRing = 4 * 32768;                // four weight stages of 32 KiB
constexpr int kSplitLds = kSplitRing + kHidden * 4;  // and mlp.c_proj's b

struct SplitRowsArgs {
    int members, tokens, dir_div, parts;
    const float *sign;
    const __bf16 *x;                  // operand: y's rows (strided), or WIDE: hid in lane order
    int64_t xs_m, xs_t;
    const __bf16 *w;                  // [512][K]
    const float *res;                 // fp32 rows the products accumulate onto (WIDE: mid)
    int64_t rs_m, rs_t;
    const float *a, *b;               // rank-1 rows (b: WIDE only) or NULL
    int64_t a_stride, b_stride;
    const float *dots;                // !WIDE: partial sums of y . b_o [rows][ndots]
    int ndots;
    const __bf16 *jit;                // WIDE: bf16 rows of 512 added to the product, or NULL
    float *mid;                       // lane order: x_mid out, or WIDE: x_mid in, x_out out
    float *out;                       // WIDE: [rows][512]
    int mix;
    const float *lam_r, *lam_x, *eps_r, *eps_x;
    int64_t eps_stride;
    const float *x0;
    int64_t x0_m, x0_t;
};

// lane order of 16 rows from row 16 G: [G][block of 16 features][lane][4] fp32, [G][step of 32 units][lane][8] bf16
__device__ __forceinline__ int64_t lane_block(int64_t row, int blocks) { return (row >> 4) * blocks * 64; }

// 16 NB output features of 128 tokens: the weights' rows stream through LDS in chunks of 1024 / NB columns (32 KiB:
// [column tiles of 64][16 NB rows][128 B]), four buffers; a wave's operand fragments come from global memory a chunk ahead.
// WIDE: K = 2048 with hid . b_proj from the fragments; else K = 512 with y . b_o from the attention's partial sums.
template <int NB, bool WIDE>
__global__ __launch_bounds__(kBlkThreads, 1) void split_rows_kernel(SplitRowsArgs p) {
    constexpr int K = WIDE ? kHidden : kModel;
    constexpr int KC = 1024 / NB, JS = KC / 32, NC = K / KC, R = 16 * NB;
    // up to four chunks: all of them are copied at once, and the loop has neither copies nor barriers, so that the
    // compiler counts the fragment loads alone
    constexpr bool kAll = NC <= 4;
    __shared__ __attribute__((aligned(16))) char lds[WIDE ? kSplitLds : kSplitRing];
    const int T = p.tokens, tiles_t = T / kBlkTok;
    int tile, part;
    if (!part_order(blockIdx.x, p.members * tiles_t, p.parts, tile, part)) return;
    const int m = tile / tiles_t, t0 = (tile % tiles_t) * kBlkTok;
    const int tid = threadIdx.x, lane = tid & 63, tl = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int dir = m / p.dir_div;
    const float sgn = p.sign ? p.sign[m] : 0.f;
    const int tok = t0 + 16 * wave + tl;
    const int64_t row = (int64_t)m * T + tok;
    const unsigned lbase = lds_addr(lds);
    const int f0 = R * part;

    // chunk c: 32 copies of 8 rows x 128 B, 4 per wave; chunk of row r at position c ^ ((r >> 1) & 7)
    auto issue = [&](int c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = 4 * wave + i, kt = n / (2 * NB), rg = n % (2 * NB);
            const int r = 8 * rg + (lane >> 3), ch = (lane & 7) ^ ((r >> 1) & 7);
            lds_dma16_at(p.w + (int64_t)(f0 + 8 * rg) * K + KC * c + 64 * kt, (unsigned)((lane >> 3) * K * 2 + ch * 16),
                         lbase + (c & 3) * 32768 + n * 1024);
        }
    };
#pragma unroll
    for (int c = 0; c < (kAll ? 4 : 3); ++c)
        if (c < NC) issue(c);
    if constexpr (WIDE) {
        if (p.a) lds_dma16_at(p.b + dir * p.b_stride + 256 * wave, (unsigned)(16 * lane), lbase + kSplitRing + 1024 * wave);
    }
    constexpr int XS = WIDE ? 512 : 32;  // elements from one k step to the next
    const __bf16 *xr = WIDE ? p.x + (lane_block(row, kHidden / 32) + lane) * 8
                            : p.x + m * p.xs_m + (int64_t)tok * p.xs_t + 8 * g;
    bf16x8 xf[2][JS];
#pragma unroll
    for (int j = 0; j < JS; ++j) xf[0][j] = load_bf16x8(xr + XS * j);
    float *mid = p.mid + (lane_block(row, kModel / 16) + 64 * NB * part + lane) * 4;
    f32x4 out[NB];
    {
        const float *rr = WIDE ? mid : p.res + m * p.rs_m + (int64_t)tok * p.rs_t + f0 + 4 * g;
#pragma unroll
        for (int ob = 0; ob < NB; ++ob) {
            const float4 v = ld4(rr + (WIDE ? 256 : 16) * ob);
            out[ob] = f32x4{v.x, v.y, v.z, v.w};
        }
    }
    float corr = 0.f;
    if constexpr (!WIDE) {
        float osum = 0.f;
        if (p.a)
            for (int k = 0; k < p.ndots; ++k) osum += p.dots[row * p.ndots + k];
        corr = sgn * osum;
    }
    vm_wait<0>();
    __syncthreads();

    const float *bl = reinterpret_cast<const float *>(lds + kSplitRing) + 4 * g;
    float pd = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (!kAll && c + 3 < NC) issue(c + 3);  // into the buffer of chunk c - 1, which every wave has left
        if (c + 1 < NC) {
#pragma unroll
            for (int j = 0; j < JS; ++j) xf[(c + 1) & 1][j] = load_bf16x8(xr + XS * (JS * (c + 1) + j));
        }
        const char *buf = lds + (c & 3) * 32768;
        auto frag = [&](int f) {  // fragment f = NB j + ob: rows 16 ob .. + 16, k block j of the chunk
            const int j = f / NB, r = 16 * (f % NB) + tl, ch = 4 * (j & 1) + g;
            return *reinterpret_cast<const bf16x8 *>(buf + (j >> 1) * (R * 128) + r * 128 + ((ch ^ ((r >> 1) & 7)) << 4));
        };
        bf16x8 a[kAhead + 1];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) a[i] = frag(i);
#pragma unroll
        for (int f = 0; f < NB * JS; ++f) {
            const int j = f / NB, ob = f % NB;
            const bf16x8 hb = xf[c & 1][j];
            if (f + kAhead < NB * JS) a[(f + kAhead) % (kAhead + 1)] = frag(f + kAhead);
            if constexpr (WIDE) {
                if (ob == 0 && p.a) {
                    // hid . b in block_kernel's order: per step of 32 units, four dots of pairs
                    const int js = JS * c + j;
                    const float4 b0 = ld4(bl + 32 * js), b1 = ld4(bl + 32 * js + 16);
#pragma unroll
                    for (int r = 0; r < 4; r += 2) {
                        pd = __builtin_amdgcn_fdot2_f32_bf16(
                            bf16x2{hb[r], hb[r + 1]}, bf16x2{(__bf16)f4get(b0, r), (__bf16)f4get(b0, r + 1)}, pd, false);
                        pd = __builtin_amdgcn_fdot2_f32_bf16(
                            bf16x2{hb[4 + r], hb[5 + r]}, bf16x2{(__bf16)f4get(b1, r), (__bf16)f4get(b1, r + 1)}, pd, false);
                    }
                }
            }
            out[ob] = mfma16x16x32(a[f % (kAhead + 1)], hb, out[ob]);
            BLOCK_PIN();
        }
        if (!kAll && c + 1 < NC) {
            // chunk c + 1 landed (the copies after it may fly; the fragment loads among them only make this stricter)
            vm_wait_groups<4, 2>(NC - 2 - c < 2 ? NC - 2 - c : 2);
            __syncthreads();
        }
    }

    if constexpr (WIDE) corr = p.a ? sgn * token_sum(pd) : 0.f;
    float rl = 0.f, ml = 0.f;
    if (WIDE && p.mix) {
        rl = *p.lam_r;
        ml = *p.lam_x;
        if (p.eps_r) rl += sgn * p.eps_r[dir * p.eps_stride];
        if (p.eps_x) ml += sgn * p.eps_x[dir * p.eps_stride];
    }
    const float *ar = p.a ? p.a + dir * p.a_stride + f0 + 4 * g : nullptr;
    const float *zr = WIDE && p.mix ? p.x0 + m * p.x0_m + (int64_t)tok * p.x0_t + f0 + 4 * g : nullptr;
    const __bf16 *jr = WIDE && p.jit ? p.jit + row * kModel + f0 + 4 * g : nullptr;
    float *dst = WIDE ? p.out + row * kModel + f0 + 4 * g : nullptr;
#pragma unroll
    for (int ob = 0; ob < NB; ++ob) {
        const float4 a4 = ar ? ld4(ar + 16 * ob) : float4{0.f, 0.f, 0.f, 0.f};
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = out[ob][r] + corr * f4get(a4, r);
        if (jr) {
            const bf16x4 j4 = load_bf16x4(jr + 16 * ob);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = out[ob][r] + (float)j4[r];
        }
        if (zr) {
            const float4 z = ld4(zr + 16 * ob);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = rl * v[r] + ml * f4get(z, r);
        }
        st4(mid + 256 * ob, float4{v[0], v[1], v[2], v[3]});
        if constexpr (WIDE) st4(dst + 16 * ob, float4{v[0], v[1], v[2], v[3]});
    }
}

// fp32 rows ([rows][512], or LANES: in lane order) as block_kernel holds them (block ob, register r: feature
// 16 ob + 4 g + r) and 1 / rms
template <bool LANES>
__device__ __forceinline__ float split_load_rows(const float *x, int64_t row, int lane, f32x4 (&out)[32]) {
    const float *xr = LANES ? x + (lane_block(row, kModel / 16) + lane) * 4 : x + row * kModel + 4 * (lane >> 4);
#pragma unroll
    for (int ob = 0; ob < 32; ++ob) {
        const float4 v = ld4(xr + (LANES ? 256 : 16) * ob);
        out[ob] = f32x4{v.x, v.y, v.z, v.w};
    }
    float ssq = 0.f;
#pragma unroll
    for (int ob = 0; ob < 32; ++ob)
#pragma unroll
        for (int r = 0; r < 4; ++r) ssq += out[ob][r] * out[ob][r];
    return rsqrtf(token_sum(ssq) * (1.0f / kModel) + kBlkEps);
}

// the row's dot with b (512 fp32), summed as block_kernel sums it
__device__ __forceinline__ float split_dot(const float *b, int g, const f32x4 (&out)[32]) {
    const float *bf = b + 4 * g;
    float d = 0.f;
#pragma unroll
    for (int ob = 0; ob < 32; ++ob) {
        const float4 b4 = ld4(bf + 16 * ob);
#pragma unroll
        for (int r = 0; r < 4; ++r) d += out[ob][r] * f4get(b4, r);
    }
    return token_sum(d);
}

// h = bf16(norm(row)) in the permuted k order of c_fc and of the next c_q, c_k, c_v
__device__ __forceinline__ void split_pack(const f32x4 (&out)[32], float rstd, bf16x8 (&xf)[16]) {
#pragma unroll
    for (int kb = 0; kb < 16; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            xf[kb][r] = (__bf16)(out[2 * kb][r] * rstd);
            xf[kb][4 + r] = (__bf16)(out[2 * kb + 1][r] * rstd);
        }
}

struct SplitFcArgs {
    int members, tokens, dir_div, parts;
    const float *sign;
    const float *x;                   // x_mid in lane order
    const __bf16 *w;                  // c_fc [2048][512], columns permuted
    const float *a, *b;               // rank-1 a [dirs][2048], b [dirs][512] or NULL
    int64_t a_stride, b_stride;
    const __bf16 *jit;                // bf16 [rows][2048] added before ReLU^2, or NULL
    __bf16 *hid;                      // in lane order
};

// 2048 / parts hidden units of 128 tokens, in chunks of 64 (64 KiB: [8 column tiles][64 rows][128 B], two buffers)
__global__ __launch_bounds__(kBlkThreads, 1) void split_fc_kernel(SplitFcArgs p) {
    __shared__ __attribute__((aligned(16))) char lds[2 * 65536];
    const int T = p.tokens, tiles_t = T / kBlkTok;
    int tile, part;
    if (!part_order(blockIdx.x, p.members * tiles_t, p.parts, tile, part)) return;
    const int m = tile / tiles_t, t0 = (tile % tiles_t) * kBlkTok;
    const int tid = threadIdx.x, lane = tid & 63, tl = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int dir = m / p.dir_div;
    const float sgn = p.sign ? p.sign[m] : 0.f;
    const int64_t row = (int64_t)m * T + t0 + 16 * wave + tl;
    const unsigned lbase = lds_addr(lds);
    const int nc = kHidden / 64 / p.parts, u0 = part * nc;  // chunks, the first one
    auto issue = [&](int c) {  // wave w copies column tile w: 8 copies of 8 rows
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = 8 * i + (lane >> 3), ch = (lane & 7) ^ ((r >> 1) & 7);
            lds_dma16_at(p.w + (int64_t)(64 * (u0 + c) + 8 * i) * kModel + 64 * wave,
                         (unsigned)((lane >> 3) * kModel * 2 + ch * 16), lbase + (c & 1) * 65536 + wave * 8192 + i * 1024);
        }
    };
    issue(0);
    if (nc > 1) issue(1);
    f32x4 out[32];
    const float rstd = split_load_rows<true>(p.x, row, lane, out);
    const float corr = p.a ? sgn * (rstd * split_dot(p.b + dir * p.b_stride, g, out)) : 0.f;
    bf16x8 xf[16];
    split_pack(out, rstd, xf);
    vm_wait<0>();
    __syncthreads();
    __bf16 *dst = p.hid + (lane_block(row, kHidden / 32) + lane) * 8;
    for (int c = 0; c < nc; ++c) {
        const char *buf = lds + (c & 1) * 65536;
#pragma unroll
        for (int s = 0; s < 2; ++s) {  // steps of 32 units
            const int u = 64 * (u0 + c) + 32 * s;
            f32x4 hacc[2] = {f32x4{}, f32x4{}};
            auto frag = [&](int f) {
                const int r = 32 * s + 16 * (f & 1) + tl, kb = f >> 1, ch = 4 * (kb & 1) + g;
                return *reinterpret_cast<const bf16x8 *>(buf + (kb >> 1) * 8192 + r * 128 + ((ch ^ ((r >> 1) & 7)) << 4));
            };
            bf16x8 a[kAhead + 1];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) a[i] = frag(i);
#pragma unroll
            for (int f = 0; f < 32; ++f) {
                if (f + kAhead < 32) a[(f + kAhead) % (kAhead + 1)] = frag(f + kAhead);
                hacc[f & 1] = mfma16x16x32(a[f % (kAhead + 1)], xf[f >> 1], hacc[f & 1]);
                BLOCK_PIN();
            }
            float add[2][4];
            if (p.jit) {
                const __bf16 *jr = p.jit + row * kHidden + u + 4 * g;
                const bf16x4 j0 = load_bf16x4(jr), j1 = load_bf16x4(jr + 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    add[0][r] = hacc[0][r] + (float)j0[r];
                    add[1][r] = hacc[1][r] + (float)j1[r];
                }
            } else {
                float4 a0{0.f, 0.f, 0.f, 0.f}, a1 = a0;
                if (p.a) {
                    const float *ar = p.a + dir * p.a_stride + u + 4 * g;
                    a0 = ld4(ar);
                    a1 = ld4(ar + 16);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    add[0][r] = hacc[0][r] + corr * f4get(a0, r);
                    add[1][r] = hacc[1][r] + corr * f4get(a1, r);
                }
            }
            bf16x8 hb;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v0 = fmaxf(add[0][r], 0.f), v1 = fmaxf(add[1][r], 0.f);
                hb[r] = (__bf16)(v0 * v0);
                hb[4 + r] = (__bf16)(v1 * v1);
            }
            store_bf16x8(dst + 16 * u, hb);
        }
        if (c + 1 < nc) {
            __syncthreads();  // every wave is done with buffer c & 1
            if (c + 2 < nc) issue(c + 2);
            // chunk c + 1 landed: only chunk c + 2's copies were issued after its own
            vm_wait_groups<8, 1>(c + 2 < nc ? 1 : 0);
            __syncthreads();
        }
    }
}

struct SplitQkvArgs {
    QkvRowsArgs q;
    const float *x;                   // x_out
    int lanes;                        // its order: 1 lane order, 0 [rows][512]
    const float *nb[3];
    int64_t nb_stride[3];
    int parts, heads;                 // heads per part (24 / parts)
};

template <int VE>
__global__ __launch_bounds__(kQThreads, 1) void split_qkv_kernel(SplitQkvArgs p) {
    __shared__ __attribute__((aligned(16))) char lds[kQLds];
    const int T = p.q.tokens, tiles_t = T / kQTok;
    int tile, part;
    if (!part_order(blockIdx.x, p.q.members * tiles_t, p.parts, tile, part)) return;
    const int m = tile / tiles_t, t0 = (tile % tiles_t) * kQTok;
    const int tid = threadIdx.x, lane = tid & 63, tl = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    QkvLane L;
    L.m = m; L.t0 = t0; L.tok = t0 + 16 * wave + tl; L.wave = wave; L.lane = lane; L.tid = tid;
    L.dir = m / p.q.dir_div; L.row = (int64_t)m * T + L.tok;
    L.sgn = p.q.sign ? p.q.sign[m] : 0.f;
    const unsigned lbase = lds_addr(lds);
    const int s0 = part * p.heads, s1 = s0 + p.heads;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (2 * s0 + k < 2 * s1) qkv_issue(p.q, lbase, wave, lane, 2 * s0 + k);
    bf16x8 xf[16];
    {
        f32x4 out[32];
        const float rstd = p.lanes ? split_load_rows<true>(p.x, L.row, lane, out)
                                   : split_load_rows<false>(p.x, L.row, lane, out);
        float dq[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (p.q.a[k]) dq[k] = L.sgn * (rstd * split_dot(p.nb[k] + L.dir * p.nb_stride[k], g, out));
        L.dq0 = dq[0]; L.dq1 = dq[1]; L.dq2 = dq[2];
        split_pack(out, rstd, xf);
    }
    qkv_token_scalars<VE>(p.q, L);
    vm_wait<0>();
    __syncthreads();
    qkv_phase<VE, true, true>(p.q, lds, xf, L, s0, s1);
}

struct SplitNormArgs {
    int members, tokens, dir_div, split3;
    const float *x;                   // in lane order
    const float *nb;                  // the head's b rows or NULL
    int64_t nb_stride;
    float *ndots;
    __bf16 *h;
};

// the last block's normed rows (hi, and [hi | lo | hi] for the fp32 head) and the head's dots
__global__ __launch_bounds__(256) void split_norm_kernel(SplitNormArgs p) {
    const int tid = threadIdx.x, lane = tid & 63, tl = lane & 15, g = lane >> 4;
    const int64_t row = (int64_t)blockIdx.x * 64 + 16 * (tid >> 6) + tl;  // (tokens are whole 128s)
    const int dir = (int)(row / p.tokens) / p.dir_div;
    f32x4 out[32];
    const float rstd = split_load_rows<true>(p.x, row, lane, out);
    if (p.ndots) {
        const float d = p.nb ? split_dot(p.nb + dir * p.nb_stride, g, out) : 0.f;
        if (g == 0) p.ndots[row] = rstd * d;
    }
    __bf16 *dst = p.h + row * (p.split3 ? 3 * kModel : kModel) + 4 * g;
#pragma unroll
    for (int ob = 0; ob < 32; ++ob) {
        bf16x4 hi, lo;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float h = out[ob][r] * rstd;
            hi[r] = (__bf16)h;
            lo[r] = (__bf16)__builtin_fmaf(out[ob][r], rstd, -(float)hi[r]);  // as block_kernel's h - hi contracts
        }
        store_bf16x4(dst + 16 * ob, hi);
        if (p.split3) {
            store_bf16x4(dst + kModel + 16 * ob, lo);
            store_bf16x4(dst + 2 * kModel + 16 * ob, hi);
        }
    }
}

// --- launches ---

// parts per token tile: as many workgroups as CUs, a power of two from 2 to 16
int split_parts(int64_t tiles) {
    int p = 16;
    while (p > 2 && tiles * p > 256) p /= 2;
    return p;
}
// up to this many token tiles the split launches are the faster ones: per block 67 against 187 us at 16 tiles, 120 at
// 64, 176 at 96, 208 at 128
constexpr int64_t kSplitTiles = 96;
int64_t split_bytes(int64_t rows) { return rows * (kModel * 4 + kHidden * 2); }

template <bool WIDE>
void split_rows_launch(const SplitRowsArgs &a, int64_t tiles, hipStream_t s) {
    const dim3 grid((unsigned)part_grid(tiles, a.parts)), block(kBlkThreads);
    switch (a.parts) {
        case 16: hipLaunchKernelGGL((split_rows_kernel<2, WIDE>), grid, block, 0, s, a); break;
        case 8: hipLaunchKernelGGL((split_rows_kernel<4, WIDE>), grid, block, 0, s, a); break;
        case 4: hipLaunchKernelGGL((split_rows_kernel<8, WIDE>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((split_rows_kernel<16, WIDE>), grid, block, 0, s, a); break;
    }
}

// x_mid, hid and x_out of the block's arguments; xout: fp32 [rows][512]; x_out in lane order at the workspace's start
void split_tail_launch(const BlockArgs &a, bool mix, float *xout, void *workspace, hipStream_t s) {
    const int64_t rows = (int64_t)a.members * a.tokens, tiles = rows / kBlkTok;
    float *xmid = static_cast<float *>(workspace);
    __bf16 *hid = reinterpret_cast<__bf16 *>(xmid + rows * kModel);
    SplitRowsArgs r{};
    r.members = a.members; r.tokens = a.tokens; r.dir_div = a.dir_div; r.sign = a.sign;
    r.parts = split_parts(tiles);
    r.x = a.y; r.xs_m = a.ys_m; r.xs_t = a.ys_t; r.w = a.wo;
    r.res = a.xres; r.rs_m = a.xr_m; r.rs_t = a.xr_t;
    r.a = a.ao; r.a_stride = a.ao_stride; r.dots = a.odots; r.ndots = a.odots_n;
    r.mid = xmid;
    split_rows_launch<false>(r, tiles, s);
    SplitFcArgs f{};
    f.members = a.members; f.tokens = a.tokens; f.dir_div = a.dir_div; f.sign = a.sign; f.parts = r.parts;
    f.x = xmid; f.w = a.wfc; f.a = a.afc; f.b = a.bfc; f.a_stride = a.afc_stride; f.b_stride = a.bfc_stride;
    f.jit = a.jfc; f.hid = hid;
    hipLaunchKernelGGL(split_fc_kernel, dim3((unsigned)part_grid(tiles, f.parts)), dim3(kBlkThreads), 0, s, f);
    r.x = hid; r.w = a.wpj; r.res = nullptr;
    r.a = a.apj; r.a_stride = a.apj_stride; r.b = a.bpj; r.b_stride = a.bpj_stride; r.dots = nullptr; r.ndots = 0;
    r.jit = a.jmlp_st ? a.jmlp : nullptr;  // (not the zero row)
    r.out = xout;
    r.mix = mix; r.lam_r = a.lam_r; r.lam_x = a.lam_x; r.eps_r = a.eps_r; r.eps_x = a.eps_x; r.eps_stride = a.eps_stride;
    r.x0 = a.x0; r.x0_m = a.x0_m; r.x0_t = a.x0_t;
    split_rows_launch<true>(r, tiles, s);
}

// x: fp32 rows, lanes: in lane order
void split_qkv_launch(const BlockArgs &a, const float *x, bool lanes, int ve, hipStream_t s) {
    const int64_t tiles = (int64_t)a.members * a.tokens / kBlkTok;
    SplitQkvArgs q;
    q.q = a.q; q.x = x; q.lanes = lanes;
    for (int k = 0; k < 3; ++k) {
        q.nb[k] = a.nb[k];
        q.nb_stride[k] = a.nb_stride[k];
    }
    q.parts = qkv_parts(tiles);
    q.heads = 24 / q.parts;
    const dim3 grid((unsigned)part_grid(tiles, q.parts));
    if (ve == 2)
        hipLaunchKernelGGL(split_qkv_kernel<2>, grid, dim3(kQThreads), 0, s, q);
    else if (ve)
        hipLaunchKernelGGL(split_qkv_kernel<1>, grid, dim3(kQThreads), 0, s, q);
    else
        hipLaunchKernelGGL(split_qkv_kernel<0>, grid, dim3(kQThreads), 0, s, q);
}

void split_norm_launch(const BlockArgs &a, const float *x, int nnext, bool split3, hipStream_t s) {
    SplitNormArgs n;
    n.members = a.members; n.tokens = a.tokens; n.dir_div = a.dir_div; n.split3 = split3;
    n.x = x; n.nb = nnext ? a.nb[0] : nullptr; n.nb_stride = a.nb_stride[0]; n.ndots = nnext ? a.ndots : nullptr;
    n.h = a.hout;
    const int64_t rows = (int64_t)a.members * a.tokens;
    hipLaunchKernelGGL(split_norm_kernel, dim3((unsigned)(rows / 64)), dim3(256), 0, s, n);
}

}  // namespace
}  // namespace noise
