// EGGROLL's update reassembly: fitness weights and the rank-1 gradient sum over the noise slices, read from the
// materialised draw or regenerated from the Philox counter a chunk of directions at a time (no 1 GiB buffer).
//
// Replaces eggroll.py:151-163:
//   fitness = losses[1::2] - losses[0::2]; fitness = fitness / (fitness.std() + 1e-8)
//   weight = zeros(pairs).index_add_(0, arange(len(fitness)) % pairs, fitness)
//   gradients[name] -= (w[:, None] * a).t() @ b       per chunk of directions   (2-D parameters)
//   gradients[name] -= w @ eps                                                  (1-D parameters)
//   p.grad = gradients[name] / len(fitness)
// where a = buffer[off_d + 0 .. rows), b = buffer[off_d + rows .. rows + cols) (eggroll.py:122-128).
//
// A 2-D parameter's gradient G = scale * sum_d w_d a_d b_d^T is a GEMM [rows x pairs] x [pairs x cols]. The
// reference runs it in fp32 (TF32 under set_float32_matmul_precision('high'), run.py:676 / eggroll.py main);
// gfx950 has no xf32 MFMA, so the GEMM splits every value into a hi and a lo bf16 half (v = hi + lo to 2^-16; the
// weights folded into a's side) as its fp32 slices land in LDS, and issues the three bf16 products hi_a hi_b,
// hi_a lo_b, lo_a hi_b of each 16 directions from one read of each fragment (split-bf16x3, fp32 accumulation).
// Chunks accumulate into G in order (deterministic). Parameters whose sides are not multiples of 256 (ve_gate
// [8, 32], the 1-D mixing scalars) are small: their entries' sums run on the vector units.
#include <atomic>

#include "common.hpp"
#include "philox.hpp"
#include "slice_copy.hpp"
#include "tile.hpp"

namespace noise {
namespace {

constexpr int kMaxParams = 64;
constexpr int kTile = 256;

// The big parameters of one call (kernel argument, ~2.6 KB).
struct UpdateSet {
    int n;
    const int64_t *offsets[kMaxParams];
    float *slab[kMaxParams];          // [np][rows + cols]: a chunk's slices, where they are not read from a buffer
    float *grad[kMaxParams];          // [rows][cols]
    int rows[kMaxParams], cols[kMaxParams];
    int row_start[kMaxParams + 1];    // prefix sums of rows + cols
    int tile_start[kMaxParams + 1];   // prefix sums of (rows / 256) (cols / 256)
};

// The small parameters of one call.
struct UpdateSmall {
    int n;
    const int64_t *offsets[kMaxParams];
    float *grad[kMaxParams];
    int rows[kMaxParams], cols[kMaxParams];  // cols = 0: a 1-D parameter of rows entries
    int start[kMaxParams + 1];               // prefix sums of the entry counts
};

__device__ inline float noise_at(const DrawLayout &dl, int64_t L, int64_t numel) {
    return (L >= 0 && L < numel) ? draw_normal(dl, (uint64_t)L, 0.0f, 1.0f) : __builtin_nanf("");
}

// eggroll.py:151-154 in one workgroup: the std is the unbiased one (torch.std's default), accumulated in
// double; fitness and its division stay fp32 as in the reference.
__global__ __launch_bounds__(1024) void update_weights_kernel(const float *__restrict__ losses, int64_t F,
                                                              int64_t pairs, float *__restrict__ weight) {
    __shared__ double red[1024];
    const int tid = threadIdx.x;
    auto block_sum = [&](double v) {
        red[tid] = v;
        __syncthreads();
        for (int s = 512; s > 0; s >>= 1) {
            if (tid < s) red[tid] += red[tid + s];
            __syncthreads();
        }
        const double r = red[0];
        __syncthreads();
        return r;
    };
    double s = 0.0;
    for (int64_t i = tid; i < F; i += 1024) s += (double)(losses[2 * i + 1] - losses[2 * i]);
    const double mean = block_sum(s) / (double)F;
    double q = 0.0;
    for (int64_t i = tid; i < F; i += 1024) {
        const double e = (double)(losses[2 * i + 1] - losses[2 * i]) - mean;
        q += e * e;
    }
    const float denom = (float)sqrt(block_sum(q) / (double)(F - 1)) + 1e-8f;
    for (int64_t d = tid; d < pairs; d += 1024) {
        float w = 0.0f;
        for (int64_t i = d; i < F; i += pairs) w += (losses[2 * i + 1] - losses[2 * i]) / denom;
        weight[d] = w;
    }
}

// A chunk's slices: slab[p][k][r] = element off_d + r of the draw, d = d0 + k, from the Philox counter or (BUFFER) a
// materialised buffer too long for the GEMM's own reads; NaN outside the draw. A thread per element, 256 elements of
// one slice per workgroup and step, so the stores are whole lines. Bound by Philox's ten rounds of two 32 x 32 -> 64
// multiplies per element (four elements 2^19 apart share a block, which slices cannot use): 512 directions of the 60
// parameters, 38.4 M normals, 159 us (split bf16 tables, one direction per lane and 2 B stores 2 np apart, took 662).
// grid = (sum of widths / 256, a share of the directions)
template <bool BUFFER>
__global__ __launch_bounds__(256) void update_slices_kernel(UpdateSet s, int64_t d0, int64_t n, DrawLayout dl,
                                                            const float *__restrict__ buf, int64_t numel) {
    const int r0 = blockIdx.x * 256;
    int p = 0;
    while (p + 1 < s.n && s.row_start[p + 1] <= r0) ++p;
    const int rl = r0 - s.row_start[p] + threadIdx.x;  // (every width is a multiple of 256)
    const int64_t width = s.rows[p] + s.cols[p];
    for (int64_t k = blockIdx.y; k < n; k += gridDim.y) {
        const int64_t L = s.offsets[p][d0 + k] + rl;
        float v;
        if constexpr (BUFFER)
            v = L >= 0 && L < numel ? buf[L] : __builtin_nanf("");
        else
            v = noise_at(dl, L, numel);
        s.slab[p][k * width + rl] = v;
    }
}

// G[o][i] (+)= sum_d A[o][d] B[i][d] over the chunk's directions, A = hi_a + lo_a and B = hi_b + lo_b, as
// hi_a hi_b + hi_a lo_b + lo_a hi_b: one 256 x 256 tile of one parameter per workgroup. 8 waves of 128 (A rows)
// x 64 (B rows), four 32 x 32 accumulator blocks by two. Workgroups past the first `full` take part q of `split`
// equal ranges of the chunk's directions for tile full + (wg - full) / split and write that partial tile to part
// (summed in order by update_reduce_kernel): the last, partial round of workgroups then runs `split` times
// shorter. A stage is 16 directions of the tile's 512 rows (34 KiB) in a ring of four; a wave reads its hi and lo
// fragments once for 24 products.
//
// A stage is the 16 directions' fp32 slices themselves, from the materialised draw or a slab, [direction][A rows | B
// rows] at a stride of 2176 B (2 KiB + 128), copied straight from the buffer (16 B per lane; slices start at any
// element). Each wave copies 2 directions and, once its copies have landed, splits them in place: the 16 B
// holding rows 4 c .. 4 c + 3 of a direction become [hi x 4 | lo x 4] (lo first where bit 1 of the direction is
// set), so nothing crosses lanes or waves before the stage's barrier. Fragments are then read with gfx950's
// transposing LDS read (ds_read_b64_tr_b16: in each 16 lanes, lane i takes element i % 4 of the 8 B that lane
// i / 4 + 4 e addresses), which gathers a row's 4 consecutive directions from 4 direction rows. The odd stride
// (128 B apart mod 256) and the hi / lo swap put a read's 4 directions on 4 disjoint sets of banks.
//
// Between two barriers every wave forms stage s's products and splits its share of stage s + 1: waves 0-3 in that
// order, waves 4-7 (the others of each SIMD) the other way round, so that one wave's conversions and LDS round trips
// run under the other's products; copies of stages s + 2 and s + 3 are in flight meanwhile. What a wave does besides
// its products bounds the stage, so that path is kept short: addresses, weights and the test that a slice lies inside
// the buffer are formed for 32 stages at once, one (stage, direction) per lane, and stages of which one slice does
// not (or is padding) take a branch of their own. 8192 directions of the 576 tiles from a 1 GiB draw: 1868 us (0.99
// PFLOP/s of products). With stages of 32 directions, all waves in one order, both directions' addresses and tests
// formed at each stage and the hi / lo halves stored as 8 B each it took 2158 (the matrix cores busy 38% of the time).
// Of the 1868, splitting accounts for about 330 and the slices' distance (HBM against a draw that fits in L2) for 320.
struct UpdateRaw {
    int64_t d0, n;             // the chunk's first direction and its directions (zeros fill the last stage)
    const float *weight;
    float scale;
    const float *buf;          // fp32 [numel]; NULL: the slabs
    int64_t numel;
};
constexpr int kUgDirs = 16;          // directions per stage
constexpr int kUgDir = 2176;         // bytes per direction of a stage (2 KiB of rows, 128 B apart)
constexpr int kSt = kUgDirs * kUgDir;
constexpr int kUgRing = 4;           // stages in LDS
constexpr int kUgOwn = kUgRing * kSt;        // each wave's offsets and weights of 32 stages (lo, hi, weight: 256 B)
constexpr int kUgLds = kUgOwn + 8 * 768;
__global__ __launch_bounds__(512) void update_gemm_kernel(UpdateSet s, int accumulate, int full, int split,
                                                          float *__restrict__ part, UpdateRaw raw) {
    __shared__ __attribute__((aligned(16))) char lds[kUgLds];
    // workgroups are dispatched round-robin over the 8 XCDs: each XCD takes a contiguous range of the full
    // tiles (and of the partial items), so the tiles that share a slice's panel run under one L2
    int wg = blockIdx.x;
    if (wg < full) {
        if ((full & 7) == 0) wg = (wg & 7) * (full >> 3) + (wg >> 3);
    } else {
        const int items = (int)gridDim.x - full, i = wg - full;
        if ((items & 7) == 0) wg = full + (i & 7) * (items >> 3) + (i >> 3);
    }
    const bool partial = wg >= full;
    const int item = wg - full;  // partial workgroups: item = split * (tile - full) + q
    const int tile = partial ? full + item / split : wg;
    int p = 0;
    while (p + 1 < s.n && s.tile_start[p + 1] <= tile) ++p;
    const int t = tile - s.tile_start[p];
    const int rows = s.rows[p], cols = s.cols[p];
    const int ot = t / (cols / kTile), ct = t % (cols / kTile);
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn0 = 128 * (wave & 1), wm0 = 64 * (wave >> 1);
    const unsigned lbase = lds_addr(lds);
    // stages k0 .. k0 + nk - 1 of the chunk's, 16 directions each (a partial workgroup's range may be empty)
    const int stages = (int)((raw.n + kUgDirs - 1) / kUgDirs);
    const int q0 = partial ? item % split : 0, qn = partial ? split : 1;
    const int k0 = (int)((int64_t)stages * q0 / qn), nk = (int)((int64_t)stages * (q0 + 1) / qn) - k0;

    const float *buf = raw.buf ? raw.buf : s.slab[p];
    const int64_t numel = raw.buf ? raw.numel : raw.n * (rows + cols);
    const int64_t side0 = (int64_t)ot * kTile, side1 = (int64_t)rows + ct * kTile;  // first slice element per side

    // this wave's directions of a stage: dir0 and dir0 + 2 (so that bit 1 of a direction is its place i)
    const int dir0 = 4 * (wave >> 1) + (wave & 1);
    // 32 stages at a time, lane l holds direction l % 2 of stage l / 2: the address of its slice's side 0, its weight
    // and whether both sides lie inside the buffer. own() copies the offsets and weights to this wave's LDS area,
    // take() reads them when the copies have landed.
    const int64_t lane_dir = (int64_t)(lane >> 1) * kUgDirs + dir0 + 2 * (lane & 1);
    auto own = [&](int ks) {
        const int64_t e = (int64_t)(k0 + ks) * kUgDirs + lane_dir, last = raw.n - 1;
        const unsigned k = (unsigned)(e < last ? e : last), at = lbase + kUgOwn + 768 * wave;
        if (raw.buf) {
            lds_dma4_at(s.offsets[p] + raw.d0, 8 * k, at);
            lds_dma4_at(s.offsets[p] + raw.d0, 8 * k + 4, at + 256);
        }
        lds_dma4_at(raw.weight + raw.d0, 4 * k, at + 512);
    };
    unsigned a_lo = 0, a_hi = 0;
    float w_own = 0.0f;
    uint64_t inside = 0;
    auto take = [&](int ks) {
        const int64_t k = (int64_t)(k0 + ks) * kUgDirs + lane_dir;
        const char *at = lds + kUgOwn + 768 * wave + 4 * lane;
        const int64_t o = raw.buf ? (int64_t)(((uint64_t)*reinterpret_cast<const uint32_t *>(at + 256) << 32) |
                                              *reinterpret_cast<const uint32_t *>(at))
                                  : k * (rows + cols);
        w_own = k < raw.n ? *reinterpret_cast<const float *>(at + 512) * raw.scale : 0.0f;
        inside = __builtin_amdgcn_ballot_w64(k < raw.n && o >= 0 && o <= numel - side1 - kTile);
        const uint64_t addr = (uint64_t)buf + 4 * (uint64_t)(o + side0);
        a_lo = (unsigned)addr;
        a_hi = (unsigned)(addr >> 32);
    };
    // a side of a direction (256 rows, 1 KiB) in one copy of 16 B per lane (lane l: rows 4 l .. + 4; a slice may
    // start at any element, so a lane's 16 B are 4 B aligned, which multi-dword global loads accept). The weights pass
    // from here to the split in wave-uniform registers; bit `slot` of slow: a direction of the stage is padding or
    // leaves the buffer
    float wt[3][2] = {};  // of stages ks + 1 .. ks + 3
    unsigned slow = 0;
    // (wave-uniform, and read out of its vector registers here: a load left to its first use in the slow branch makes
    // the compiler wait for every copy in flight where the branches meet, 31.0 -> 36.3 ms for 131,072 pairs)
    auto offset = [&](int64_t k) {
        const int64_t o = raw.buf ? s.offsets[p][raw.d0 + k] : k * (rows + cols);
        return (int64_t)(((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(o >> 32)) << 32) |
                         (unsigned)__builtin_amdgcn_readfirstlane((int)o));
    };
    auto issue = [&](int ks, float (&w)[2]) {
        const int slot = ks & (kUgRing - 1), at = 2 * (ks & 31);
        const unsigned st = lbase + slot * kSt + dir0 * kUgDir;
        if (((inside >> at) & 3) == 3) {
            slow &= ~(1u << slot);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint64_t addr = ((uint64_t)(unsigned)__builtin_amdgcn_readlane((int)a_hi, at + i) << 32) |
                                      (unsigned)__builtin_amdgcn_readlane((int)a_lo, at + i);
                w[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w_own), at + i));
                lds_dma16_at((const void *)addr, (unsigned)(16 * lane), st + 2 * i * kUgDir);
                lds_dma16_at((const void *)(addr + 4 * (side1 - side0)), (unsigned)(16 * lane),
                             st + 2 * i * kUgDir + 1024);
            }
        } else {
            // 4 B copies with every lane's element clamped into the buffer (a padding direction reads from element 0)
            slow |= 1u << slot;
#pragma unroll 1
            for (int i = 0; i < 2; ++i) {
                const int64_t k = (int64_t)(k0 + ks) * kUgDirs + dir0 + 2 * i;
                const int64_t o = k < raw.n ? offset(k) : 0;
#pragma unroll 1
                for (int q = 0; q < 8; ++q) {
                    const int64_t first = k < raw.n ? o + (q >= 4 ? side1 : side0) + 64 * (q & 3) : 0;
                    const int64_t base = slice_base(first, numel);
                    lds_dma4_at(buf + base, slice_lane(first, lane, base, numel), st + 2 * i * kUgDir + 256 * q);
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
                w[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w_own), at + i));
        }
    };
    // split this wave's share of a stage in place: lane l takes rows 4 l .. + 4 of each side and direction. a rows:
    // weight * scale; b rows as they are
    auto split_raw = [&](int ks, const float (&w)[2]) {
        const int slot = ks & (kUgRing - 1);
        char *c = lds + slot * kSt + dir0 * kUgDir + 16 * lane;
        float4 v4[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int side = 0; side < 2; ++side)
                v4[i][side] = *reinterpret_cast<const float4 *>(c + 2 * i * kUgDir + 1024 * side);
        if ((slow >> slot) & 1) {
            // zeros for a padding direction, NaN for a slice's elements outside the buffer
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int64_t k = (int64_t)(k0 + ks) * kUgDirs + dir0 + 2 * i;
                const int64_t o = k < raw.n ? offset(k) : 0;
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    const int64_t L = o + (side ? side1 : side0) + 4 * lane;
                    float *f = reinterpret_cast<float *>(&v4[i][side]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool in = L + e >= 0 && L + e < numel;
                        f[e] = k >= raw.n ? 0.0f : in ? f[e] : __builtin_nanf("");
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                // v rounded to fp32 first, then lo = v - hi exactly (no fused multiply-subtract)
#pragma clang fp contract(off)
                const float4 x = v4[i][side];
                const float v[4] = {side ? x.x : x.x * w[i], side ? x.y : x.y * w[i], side ? x.z : x.z * w[i],
                                    side ? x.w : x.w * w[i]};
                bf16x8 hl;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const __bf16 hi = (__bf16)v[e];
                    hl[4 * i + e] = hi;
                    hl[4 * (1 - i) + e] = (__bf16)(v[e] - (float)hi);
                }
                *reinterpret_cast<bf16x8 *>(c + 2 * i * kUgDir + 1024 * side) = hl;
            }
    };

    // lane 16 G + i addresses direction 8 (G / 2) + i / 4 (+ 4 e) and rows 16 (G % 2) + 4 (i % 4)
    // .. + 4 of a 32-row block; bit 1 of that direction (bit 3 of i) swaps hi and lo. tro[lo]
    int tro[2];
    {
        const int G = lane >> 4, i = lane & 15;
#pragma unroll
        for (int lo = 0; lo < 2; ++lo)
            tro[lo] = (8 * (G >> 1) + (i >> 2)) * kUgDir + 64 * (G & 1) + 16 * (i & 3) + 8 * (((i >> 3) & 1) ^ lo);
    }
    // 32 rows from row R (a multiple of 32 within the side), directions 8 hf + 0 .. 7
    auto tr_frag = [&](const char *st, int side, int R, int lo) {
        const char *b = st + tro[lo] + side * 1024 + 4 * R;
        const bf16x4 x = lds_read_tr16(b), y = lds_read_tr16(b + 4 * kUgDir);
        return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
    };

    f32x16 acc[4][2];
#pragma unroll
    for (int fb = 0; fb < 4; ++fb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) acc[fb][tb] = f32x16{};
    // the three products as three passes over the 8 accumulators: dependent products 8 apart
    auto products = [&](int slot) {
        const char *st = lds + slot * kSt;
        bf16x8 ah[4], al[4], bh[2], bl[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) bh[tb] = tr_frag(st, 1, wm0 + 32 * tb, 0);
#pragma unroll
        for (int fb = 0; fb < 4; ++fb) ah[fb] = tr_frag(st, 0, wn0 + 32 * fb, 0);
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) bl[tb] = tr_frag(st, 1, wm0 + 32 * tb, 1);
#pragma unroll
        for (int fb = 0; fb < 4; ++fb) al[fb] = tr_frag(st, 0, wn0 + 32 * fb, 1);
#pragma unroll
        for (int pr = 0; pr < 3; ++pr)
#pragma unroll
            for (int fb = 0; fb < 4; ++fb)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
                    acc[fb][tb] = mfma32x32x16(pr == 2 ? al[fb] : ah[fb], pr == 1 ? bl[tb] : bh[tb], acc[fb][tb]);
    };
    // this wave's copies of stage ks landed: those of at most two later stages (4 or more each) may still fly
    auto landed = [&](int ks) {
        vm_wait_groups<4, 2>(nk - 1 - ks < 2 ? nk - 1 - ks : 2);
        asm volatile("" ::: "memory");
    };
    const bool split_first = wave >= 4;
    if (nk > 0) {
        float w0[2];
        own(0);
        vm_wait<0>();
        asm volatile("" ::: "memory");
        take(0);
        issue(0, w0);
        if (nk > 1) issue(1, wt[0]);
        if (nk > 2) issue(2, wt[1]);
        landed(0);
        split_raw(0, w0);
        __syncthreads();
    }
#pragma unroll 1
    for (int ks = 0; ks < nk; ++ks) {
        if (ks + 3 < nk) {
            // the next 32 stages' offsets are copied 16 stages before they are taken
            if (((ks + 3) & 31) == 16 && ks + 19 < nk) own(ks + 19);
            if (((ks + 3) & 31) == 0) take(ks + 3);
            issue(ks + 3, wt[2]);  // into the slot of stage ks - 1, which every wave has left
        }
        if (split_first && ks + 1 < nk) {
            landed(ks + 1);
            split_raw(ks + 1, wt[0]);
        }
        __builtin_amdgcn_s_setprio(1);  // the matrix cores before the other wave's conversions
        products(ks & (kUgRing - 1));
        __builtin_amdgcn_s_setprio(0);
        if (!split_first && ks + 1 < nk) {
            landed(ks + 1);
            split_raw(ks + 1, wt[0]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            wt[0][i] = wt[1][i];
            wt[1][i] = wt[2][i];
        }
        __syncthreads();  // stage ks + 1 split; every wave has read its fragments of stage ks
    }
    // lane (j, hf), register 4 g + e of block (fb, tb): row o = wn0 + 32 fb + 8 g + 4 hf + e, column
    // i = wm0 + 32 tb + j; the 32 lanes of a half-wave write 128 contiguous bytes of one row (a partial tile:
    // [256][256] of its own)
    float *g = partial ? part + (int64_t)item * kTile * kTile : s.grad[p] + (int64_t)ot * kTile * cols + ct * kTile;
    const int64_t ldg = partial ? kTile : cols;
    const bool add = accumulate && !partial;
#pragma unroll
    for (int fb = 0; fb < 4; ++fb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int o = wn0 + 32 * fb + 8 * (q >> 2) + 4 * hf + (q & 3);
                float *dst = g + (int64_t)o * ldg + wm0 + 32 * tb + j;
                const float v = acc[fb][tb][q];
                *dst = add ? *dst + v : v;
            }
}

// The partial tiles of update_gemm_kernel summed in order (part 0 first) into G (+=): 1024 entries per
// workgroup, 64 workgroups per tile. grid = (tiles - full) * 64.
__global__ __launch_bounds__(256) void update_reduce_kernel(UpdateSet s, int full, int split,
                                                            const float *__restrict__ part, int accumulate) {
    const int tile = full + blockIdx.x / 64, e = (blockIdx.x % 64) * 1024 + 4 * threadIdx.x;
    int p = 0;
    while (p + 1 < s.n && s.tile_start[p + 1] <= tile) ++p;
    const int t = tile - s.tile_start[p], cols = s.cols[p];
    const int ot = t / (cols / kTile), ct = t % (cols / kTile);
    const float *src = part + (int64_t)(tile - full) * split * kTile * kTile + e;
    float4 v = ld4(src);
    for (int q = 1; q < split; ++q) {
        const float4 w = ld4(src + (int64_t)q * kTile * kTile);
        v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
    }
    float *dst = s.grad[p] + (int64_t)(ot * kTile + e / kTile) * cols + ct * kTile + e % kTile;
    if (accumulate) {
        const float4 g = ld4(dst);
        v.x += g.x; v.y += g.y; v.z += g.z; v.w += g.w;
    }
    st4(dst, v);
}

// One gradient entry per workgroup: scale * sum_d weight[d] a_d[o] (b_d[i] or 1), 256 threads striding
// over the directions, then a fixed-order tree.
__global__ __launch_bounds__(256) void update_small_kernel(UpdateSmall s, int64_t pairs,
                                                           const float *__restrict__ weight, float scale,
                                                           DrawLayout dl, int64_t numel) {
    __shared__ float red[256];
    const int e = blockIdx.x, tid = threadIdx.x;
    int p = 0;
    while (p + 1 < s.n && s.start[p + 1] <= e) ++p;
    const int el = e - s.start[p], rows = s.rows[p], cols = s.cols[p];
    const int o = cols ? el / cols : el, i = cols ? el % cols : 0;
    const int64_t *off = s.offsets[p];
    float acc = 0.0f;
    for (int64_t d = tid; d < pairs; d += 256) {
        const float a = noise_at(dl, off[d] + o, numel);
        const float b = cols ? noise_at(dl, off[d] + rows + i, numel) : 1.0f;
        acc += weight[d] * a * b;
    }
    red[tid] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st) red[tid] += red[tid + st];
        __syncthreads();
    }
    if (tid == 0) s.grad[p][el] = scale * red[0];
}

// Small parameters of at most kSmallWidth slice elements and kSmallEntries entries, many directions: a workgroup draws
// each slice of its chunk of directions once into LDS (16 at a time, the weights folded into a's side) and every
// thread adds up to four entries' products; the chunks' sums go to part [chunk][entry] and are summed in order by
// update_small_reduce_kernel. One workgroup per entry (update_small_kernel) draws a and b again for each of the 256
// entries of a gate, 13 times the normals: 131,072 directions of the model's 6 small parameters, 148 + 6 us
// against 923; below kSmallPairs its single launch is the shorter.
constexpr int kSmallWidth = 512, kSmallEntries = 1024, kSmallDirs = 16;
constexpr int64_t kSmallPairs = 4096;
__global__ __launch_bounds__(256) void update_small_partial_kernel(UpdateSmall s, int64_t pairs, int64_t chunk,
                                                                   int entries, const float *__restrict__ weight,
                                                                   DrawLayout dl, int64_t numel,
                                                                   float *__restrict__ part) {
    __shared__ float sm[kSmallDirs * kSmallWidth];
    const int p = blockIdx.y, tid = threadIdx.x;
    const int rows = s.rows[p], cols = s.cols[p], width = rows + cols, n = rows * (cols ? cols : 1);
    const int64_t *off = s.offsets[p];
    const int64_t d0 = blockIdx.x * chunk, d1 = d0 + chunk < pairs ? d0 + chunk : pairs;
    float acc[kSmallEntries / 256];
#pragma unroll
    for (int q = 0; q < kSmallEntries / 256; ++q) acc[q] = 0.0f;
    for (int64_t d = d0; d < d1; d += kSmallDirs) {
        const int m = d1 - d < kSmallDirs ? (int)(d1 - d) : kSmallDirs;
        for (int i = tid; i < m * width; i += 256) {
            const int k = i / width, r = i - k * width;
            const float v = noise_at(dl, off[d + k] + r, numel);
            sm[k * width + r] = r < rows ? weight[d + k] * v : v;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kSmallEntries / 256; ++q) {
            const int e = 256 * q + tid;
            if (e < n) {
                const int o = cols ? e / cols : e, i = cols ? rows + e % cols : 0;
                for (int k = 0; k < m; ++k) acc[q] += sm[k * width + o] * (cols ? sm[k * width + i] : 1.0f);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kSmallEntries / 256; ++q)
        if (256 * q + tid < n) part[(int64_t)blockIdx.x * entries + s.start[p] + 256 * q + tid] = acc[q];
}

// scale * the chunks' sums of one entry per workgroup, a fixed-order tree
__global__ __launch_bounds__(256) void update_small_reduce_kernel(UpdateSmall s, int chunks, int entries, float scale,
                                                                  const float *__restrict__ part) {
    __shared__ float red[256];
    const int e = blockIdx.x, tid = threadIdx.x;
    int p = 0;
    while (p + 1 < s.n && s.start[p + 1] <= e) ++p;
    float acc = 0.0f;
    for (int c = tid; c < chunks; c += 256) acc += part[(int64_t)c * entries + e];
    red[tid] = acc;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st) red[tid] += red[tid + st];
        __syncthreads();
    }
    if (tid == 0) s.grad[p][e - s.start[p]] = scale * red[0];
}

bool is_big(const noise_update_param_t &q) {
    return q.cols > 0 && q.rows % kTile == 0 && q.cols % kTile == 0;
}

int64_t padded_chunk(int64_t chunk, int64_t pairs) {
    const int64_t c = chunk < pairs ? chunk : pairs;
    return (c + 255) / 256 * 256;
}

// The GEMM's last, partial round of workgroups (one per CU) over `cus` compute units: tiles full .. tiles - 1
// run as `split` shorter partial workgroups each, so that round fills the device; split 1: no partials.
void gemm_split(int64_t tiles, int64_t cus, int64_t &full, int &split) {
    const int64_t r = cus > 0 ? tiles % cus : 0;
    const int64_t sp = r ? cus / r : 1;
    split = sp >= 4 ? 4 : sp >= 2 ? 2 : 1;
    full = split > 1 ? tiles - r : tiles;
}

int64_t partial_bytes(int64_t tiles, int64_t full, int split) {
    return split > 1 ? (tiles - full) * split * kTile * kTile * (int64_t)sizeof(float) : 0;
}

// compute units of the current device (gfx950 parts have 256), cached per device (any host thread may ask)
int64_t device_cus() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int c = cached[dev].load(std::memory_order_relaxed);
    if (!c) {
        int n = 0;
        c = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
        cached[dev].store(c, std::memory_order_relaxed);
    }
    return c;
}

}  // namespace
}  // namespace noise

using namespace noise;

extern "C" int noise_update_weights(const float *losses, int64_t members, int64_t pairs, float *weight,
                                    noise_stream_t stream) {
    clear_error();
    NOISE_CHECK_ARG(members >= 4 && members % 2 == 0,
                    "noise_update_weights: members must be even and >= 4 (two fitness values for a std), got %lld",
                    (long long)members);
    NOISE_CHECK_ARG(pairs >= 1, "noise_update_weights: pairs must be >= 1");
    NOISE_CHECK_ARG(losses != nullptr && weight != nullptr, "noise_update_weights: losses and weight must be non-NULL");
    hipLaunchKernelGGL(update_weights_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, losses, members / 2,
                       pairs, weight);
    return launch_status("noise_update_weights");
}

extern "C" int64_t noise_update_workspace_bytes(const noise_update_param_t *params, int nparams, int64_t pairs,
                                                int64_t chunk) {
    if (params == nullptr || nparams < 0 || pairs < 1 || chunk < 1) return -1;
    const int64_t np = padded_chunk(chunk, pairs);
    int64_t bytes = 0, tiles = 0;
    for (int i = 0; i < nparams; ++i)
        if (is_big(params[i])) {
            bytes += (params[i].rows + params[i].cols) * 2 * np * 2;
            tiles += (params[i].rows / kTile) * (params[i].cols / kTile);
        }
    // the slabs, then the GEMM's partial tiles for a device of 256 compute units
    int64_t full;
    int split;
    gemm_split(tiles, 256, full, split);
    return bytes + partial_bytes(tiles, full, split);
}

extern "C" int noise_update_gradients(const noise_update_param_t *params, int nparams, int64_t pairs,
                                      const float *weight, float scale, int64_t chunk, int64_t numel, uint64_t seed,
                                      uint64_t offset, int64_t threads, const float *buffer, void *workspace,
                                      int64_t workspace_bytes, noise_stream_t stream) {
    clear_error();
    NOISE_CHECK_ARG(params != nullptr && nparams >= 0 && nparams <= kMaxParams,
                    "noise_update_gradients: 0 .. %d parameters per call, got %d", kMaxParams, nparams);
    NOISE_CHECK_ARG(pairs >= 1 && chunk >= 1, "noise_update_gradients: pairs and chunk must be >= 1");
    NOISE_CHECK_ARG(weight != nullptr, "noise_update_gradients: weight must be non-NULL");
    NOISE_CHECK_ARG(threads > 0 && threads % 256 == 0,
                    "noise_update_gradients: threads must be a positive multiple of 256");
    NOISE_CHECK_ARG(offset % 4 == 0, "noise_update_gradients: generator offset must be a multiple of 4");
    NOISE_CHECK_ARG(numel > 0, "noise_update_gradients: numel must be positive");
    NOISE_CHECK_ARG(buffer == nullptr || aligned(buffer, 4), "noise_update_gradients: buffer must be 4-byte aligned");
    const int64_t np = padded_chunk(chunk, pairs);
    NOISE_CHECK_ARG(np <= (1 << 22), "noise_update_gradients: chunk too large (at most 4194304 directions)");
    UpdateSet big{};
    UpdateSmall small{};
    int64_t rows_total = 0, tiles_total = 0, entries_total = 0, need = 0;
    char *ws = static_cast<char *>(workspace);
    for (int i = 0; i < nparams; ++i) {
        const noise_update_param_t &q = params[i];
        NOISE_CHECK_ARG(q.offsets != nullptr && q.grad != nullptr && aligned(q.offsets, 8) && aligned(q.grad, 4),
                        "noise_update_gradients: parameter %d: offsets and grad must be non-NULL and aligned", i);
        NOISE_CHECK_ARG(q.rows >= 1 && q.cols >= 0, "noise_update_gradients: parameter %d: bad shape", i);
        if (is_big(q)) {
            NOISE_CHECK_ARG(q.rows + q.cols <= 65536 && q.rows / kTile * (q.cols / kTile) <= 65536,
                            "noise_update_gradients: parameter %d: %lld x %lld is too large", i, (long long)q.rows,
                            (long long)q.cols);
            const int b = big.n++;
            big.offsets[b] = q.offsets;
            big.grad[b] = q.grad;
            big.rows[b] = (int)q.rows;
            big.cols[b] = (int)q.cols;
            big.row_start[b] = (int)rows_total;
            big.tile_start[b] = (int)tiles_total;
            big.slab[b] = reinterpret_cast<float *>(ws + need);
            rows_total += q.rows + q.cols;
            tiles_total += (q.rows / kTile) * (q.cols / kTile);
            need += (q.rows + q.cols) * 2 * np * 2;
        } else {
            const int64_t entries = q.rows * (q.cols ? q.cols : 1);
            NOISE_CHECK_ARG(entries <= 65536,
                            "noise_update_gradients: parameter %d: %lld x %lld is neither a multiple of 256 on both "
                            "sides nor small (<= 65536 entries)", i, (long long)q.rows, (long long)q.cols);
            const int sm = small.n++;
            small.offsets[sm] = q.offsets;
            small.grad[sm] = q.grad;
            small.rows[sm] = (int)q.rows;
            small.cols[sm] = (int)q.cols;
            small.start[sm] = (int)entries_total;
            entries_total += entries;
        }
    }
    big.row_start[big.n] = (int)rows_total;
    big.tile_start[big.n] = (int)tiles_total;
    small.start[small.n] = (int)entries_total;
    NOISE_CHECK_ARG(rows_total < (1ll << 31) && tiles_total < (1ll << 31) && entries_total < (1ll << 31),
                    "noise_update_gradients: too many rows");
    NOISE_CHECK_ARG(need == 0 || (workspace != nullptr && aligned(workspace, 16) && workspace_bytes >= need),
                    "noise_update_gradients: workspace must be 16-byte aligned and hold %lld bytes (got %lld); "
                    "see noise_update_workspace_bytes", (long long)need, (long long)workspace_bytes);
    DrawLayout dl{seed, offset, (uint64_t)threads};
    hipStream_t s = (hipStream_t)stream;
    // the GEMM's partial tiles after the slabs, when the workspace holds them (else whole tiles only)
    int64_t full;
    int split;
    gemm_split(tiles_total, device_cus(), full, split);
    while (split > 1 && (workspace == nullptr || workspace_bytes - need < partial_bytes(tiles_total, full, split))) {
        split /= 2;
        if (split == 1) full = tiles_total;
    }
    float *part = split > 1 ? reinterpret_cast<float *>(ws + need) : nullptr;
    bool shared_slices = pairs >= kSmallPairs;
    for (int i = 0; i < small.n; ++i) {
        const int64_t cols = small.cols[i], n = small.rows[i] * (cols ? cols : 1);
        shared_slices = shared_slices && small.rows[i] + cols <= kSmallWidth && n <= kSmallEntries;
    }
    // 512 chunks of directions (whole steps of kSmallDirs); their sums use the slabs' area, which is written later
    const int64_t chunk_small = ((pairs + 511) / 512 + kSmallDirs - 1) / kSmallDirs * kSmallDirs;
    const int64_t chunks_small = (pairs + chunk_small - 1) / chunk_small;
    if (small.n && shared_slices && chunks_small * entries_total * (int64_t)sizeof(float) <= need) {
        hipLaunchKernelGGL(update_small_partial_kernel, dim3((unsigned)chunks_small, (unsigned)small.n), dim3(256), 0, s,
                           small, pairs, chunk_small, (int)entries_total, weight, dl, numel, reinterpret_cast<float *>(ws));
        hipLaunchKernelGGL(update_small_reduce_kernel, dim3((unsigned)entries_total), dim3(256), 0, s, small,
                           (int)chunks_small, (int)entries_total, scale, reinterpret_cast<const float *>(ws));
        int st = launch_status("noise_update_gradients (small parameters)");
        if (st) return st;
    } else if (small.n) {
        hipLaunchKernelGGL(update_small_kernel, dim3((unsigned)entries_total), dim3(256), 0, s, small, pairs, weight,
                           scale, dl, numel);
        int st = launch_status("noise_update_gradients (small parameters)");
        if (st) return st;
    }
    if (big.n) {
        // with a buffer of at most 2^30 elements the GEMM reads the slices itself; otherwise they are written out first
        const bool direct = buffer != nullptr && numel <= (1ll << 30);
        for (int64_t d0 = 0; d0 < pairs; d0 += np) {
            const int64_t n = pairs - d0 < np ? pairs - d0 : np;
            const int64_t wgs = full + (tiles_total - full) * split;
            int st;
            if (!direct) {
                // the directions shared out so that some 16 K workgroups are in the launch
                const int64_t cols = rows_total / 256, share = 16384 / cols + 1;
                const dim3 grid((unsigned)cols, (unsigned)(n < share ? n : share));
                if (buffer)
                    hipLaunchKernelGGL(update_slices_kernel<true>, grid, dim3(256), 0, s, big, d0, n, dl, buffer, numel);
                else
                    hipLaunchKernelGGL(update_slices_kernel<false>, grid, dim3(256), 0, s, big, d0, n, dl, buffer, numel);
                st = launch_status("noise_update_gradients (slices)");
                if (st) return st;
            }
            const UpdateRaw raw{d0, n, weight, scale, direct ? buffer : nullptr, numel};
            hipLaunchKernelGGL(update_gemm_kernel, dim3((unsigned)wgs), dim3(512), 0, s, big, d0 > 0 ? 1 : 0, (int)full,
                               split, part, raw);
            st = launch_status("noise_update_gradients (gemm)");
            if (st) return st;
            if (split > 1) {
                hipLaunchKernelGGL(update_reduce_kernel, dim3((unsigned)((tiles_total - full) * 64)), dim3(256), 0, s,
                                   big, (int)full, split, part, d0 > 0 ? 1 : 0);
                st = launch_status("noise_update_gradients (partial tiles)");
                if (st) return st;
            }
        }
    }
    return NOISE_OK;
}
