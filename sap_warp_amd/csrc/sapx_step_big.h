// Factor and solves of the 256-thread step kernel for worlds whose matrices exceed its LDS layout.
//
// The Newton matrix H (order npad <= 256, a multiple of 16) is held as the lower triangle of its
// 16 x 16 blocks, 1 KB each, in LDS when the world's vectors leave room for it and in the world's
// block of device memory otherwise.  Inside a block the four-float groups of row r are stored at
// group ^ (r / 4): 16 rows read with 16-byte loads then hit every LDS bank once.  Row masks (bit jb
// of hm[ib]: block (ib, jb) is nonzero in the factor) skip the blocks that no tree of the dynamics
// matrix, no contact and no fill touches.
//
// Both are chains of npad / 16 block steps whose latency is what they cost.  Measured on a world of 16
// and of 32 bodies (6 and 12 blocks): factor 16 and 31 us.  The solve keeps a row per thread and all
// waves step together, one barrier a block; the same chain on one wave, its rows in turn, took 12 and
// 21 us.
#ifndef SAPX_STEP_BIG_H
#define SAPX_STEP_BIG_H

#include "sapx_kcommon.h"

namespace sapx {
namespace big {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kB = 16;           // block order
constexpr int kMaxBlocks = 16;   // npad / 16 at most

__device__ __forceinline__ float* block(float* H, int ib, int jb) { return H + (ib * (ib + 1) / 2 + jb) * (kB * kB); }
// four columns 4 g .. 4 g + 3 of row r
__device__ __forceinline__ f4* group(float* b, int r, int g) { return reinterpret_cast<f4*>(b + r * kB + 4 * (g ^ (r >> 2))); }
__device__ __forceinline__ float* entry(float* b, int r, int c) { return b + r * kB + 4 * ((c >> 2) ^ (r >> 2)) + (c & 3); }

// fill of the block elimination on one wave: lane i holds row i of the mask
__device__ __forceinline__ void symbolic(unsigned* hm, int nblk) {
    const int i = threadIdx.x & 63;
    unsigned m = i < nblk ? hm[i] : 0u;
    for (int k = 0; k < nblk; ++k) {
        const bool below = i > k && ((m >> k) & 1u);
        const unsigned rows = (unsigned)__ballot(below);
        if (below) m |= rows & ((1u << i) - 1u);
    }
    if (i < nblk) hm[i] = m | (1u << i);
}

// Cholesky of the diagonal block on one wave (lane r = row r, the other lanes repeat it): L replaces the
// lower triangle, zeros the upper one; pivots are clamped to 1e-30
__device__ __forceinline__ void factor_diag(float* b, float* dinv) {
    const int lane = threadIdx.x & 63, r = lane & 15;
    float a[kB];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const f4 v = *group(b, r, g);
#pragma unroll
        for (int u = 0; u < 4; ++u) a[4 * g + u] = v[u];
    }
    float mine = 1.0f, diag = 1.0f;
#pragma unroll
    for (int j = 0; j < kB; ++j) {
        // rows above the pivot hold no entries of L: they compute along and are cleared below
        const float d = fmaxf(rl(a[j], j), 1.0e-30f);
        float inv = __builtin_amdgcn_rsqf(d);
        inv = fmaf(0.5f * inv, fmaf(-d * inv, inv, 1.0f), inv);
        a[j] *= inv;
#pragma unroll
        for (int c = j + 1; c < kB; ++c) a[c] = fmaf(-a[j], rl(a[j], c), a[c]);
        mine = r == j ? inv : mine;
        diag = r == j ? d * inv : diag;
    }
#pragma unroll
    for (int c = 0; c < kB; ++c) a[c] = r == c ? diag : (r > c ? a[c] : 0.0f);
    if (lane < kB) {
#pragma unroll
        for (int g = 0; g < 4; ++g) *group(b, r, g) = f4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
        dinv[r] = mine;
    }
}

// Calls f(count, ib[], jb[]) with the masked blocks (ib, jb), jb <= ib, whose row and column are both in
// `rows`, up to four at a time: the blocks number `part`, part + parts, ... of them.  hm_lane: lane i
// holds the row mask hm[i].
template <typename F>
__device__ __forceinline__ void tiles(unsigned hm_lane, unsigned rows, int nblk, int part, int parts, F&& f) {
    int ib[4], jb[4], have = 0, t = part;
    for (int i = 0; i < nblk; ++i) {
        if (!((rows >> i) & 1u)) continue;
        unsigned cols = rows & ((2u << i) - 1u) & (unsigned)__builtin_amdgcn_readlane((int)hm_lane, i);
        for (; cols; cols &= cols - 1) {
            if (t--) continue;
            t = parts - 1;
            const int j = __builtin_ctz(cols);
            if (have == 0) { ib[0] = i; jb[0] = j; }
            else if (have == 1) { ib[1] = i; jb[1] = j; }
            else if (have == 2) { ib[2] = i; jb[2] = j; }
            else { ib[3] = i; jb[3] = j; }
            if (++have == 4) {
                f(4, ib, jb);
                have = 0;
            }
        }
    }
    if (have) f(have, ib, jb);
}

// H = L L^T in place, then the diagonal blocks are replaced by their inverses.  Per block column: the
// rows below by substitution (a row per thread), then wave 0 updates and factors the next diagonal
// block while the other waves apply the column to the trailing blocks by MFMA, four blocks at a time
// (two barriers a column).  dinv: npad floats.
template <int NT>
__device__ __forceinline__ void factor(float* H, int npad, const unsigned* hm, float* dinv) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nblk = npad >> 4;
    const unsigned hm_lane = lane < nblk ? hm[lane] : 0u;
    if (wave == 0) factor_diag(block(H, 0, 0), dinv);
    __syncthreads();
    // transposed products: a lane holds four columns of one row of the block
    auto update = [&](int count, const int (&ib)[4], const int (&jb)[4], int kb) {
        f4 a[4], b[4], h[4], acc[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = u < count ? ib[u] : ib[0], j = u < count ? jb[u] : jb[0];
            a[u] = *group(block(H, j, kb), lane & 15, lane >> 4);
            b[u] = *group(block(H, i, kb), lane & 15, lane >> 4);
            h[u] = *group(block(H, i, j), lane & 15, lane >> 4);
            acc[u] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][k], b[u][k], acc[u], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (u < count) *group(block(H, ib[u], jb[u]), lane & 15, lane >> 4) = h[u] - acc[u];
    };
    for (int kb = 0; kb + 1 < nblk; ++kb) {
        for (int i = kB * (kb + 1) + tid; i < npad; i += NT) {
            const int ib = i >> 4, r = i & 15;
            if (!((hm[ib] >> kb) & 1u)) continue;
            float* p = block(H, ib, kb);
            float* Lk = block(H, kb, kb);
            float x[kB], di[kB];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f4 v = *group(p, r, g), d = *reinterpret_cast<const f4*>(dinv + kB * kb + 4 * g);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    x[4 * g + u] = v[u];
                    di[4 * g + u] = d[u];
                }
            }
#pragma unroll
            for (int c = 0; c < kB; ++c) {
                float s = x[c];
#pragma unroll
                for (int g = 0; 4 * g < c; ++g) {
                    const f4 l = *group(Lk, c, g);
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (4 * g + u < c) s = fmaf(-x[4 * g + u], l[u], s);
                }
                x[c] = s * di[c];
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) *group(p, r, g) = f4{x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
        }
        __syncthreads();
        // the block rows that column kb reaches
        const unsigned rows = (unsigned)__ballot(lane > kb && ((hm_lane >> kb) & 1u));
        if (wave == 0) {
            const int next[4] = {kb + 1, 0, 0, 0};
            if ((rows >> (kb + 1)) & 1u) update(1, next, next, kb);
            wave_sync();
            factor_diag(block(H, kb + 1, kb + 1), dinv + kB * (kb + 1));
        } else {
            tiles(hm_lane, rows, nblk, wave - 1, NT / 64 - 1, [&](int count, const int (&ib)[4], const int (&jb)[4]) {
                // the next diagonal block is wave 0's
                if (ib[0] == kb + 1) {
                    const int i2[4] = {ib[1], ib[2], ib[3], 0}, j2[4] = {jb[1], jb[2], jb[3], 0};
                    if (count > 1) update(count - 1, i2, j2, kb);
                } else {
                    update(count, ib, jb, kb);
                }
            });
        }
        __syncthreads();
    }
    // inverses of the diagonal blocks: 16 lanes a block, lane c forward-substitutes column c
    for (int kb = tid >> 4; kb < nblk; kb += NT / 16) {
        const int c = tid & 15;
        float* b = block(H, kb, kb);
        float x[kB];
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            float acc = 0.0f;
#pragma unroll
            for (int g = 0; 4 * g < i; ++g) {
                const f4 l = *group(b, i, g);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (4 * g + u < i) acc = fmaf(l[u], x[4 * g + u], acc);
            }
            x[i] = ((i == c ? 1.0f : 0.0f) - acc) * dinv[kB * kb + i];
        }
        wave_sync();  // every lane of the block has read L
#pragma unroll
        for (int i = 0; i < kB; ++i) *entry(b, i, c) = x[i];
    }
    __syncthreads();
}

// b <- (L L^T)^-1 b (b: npad floats in LDS, zero from n on; xr: npad floats of LDS that nobody else uses).
// Thread i keeps row i (npad <= NT).  A block's right-hand side goes through LDS (one barrier a block);
// every wave multiplies it by the block's inverse and takes the 16 unknowns out of its own rows.  Starts
// after a barrier that follows the writes of b, and ends with one.
template <int NT>
__device__ __forceinline__ void solve(float* H, int npad, const unsigned* hm, float* b, float* xr) {
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, nblk = npad >> 4;
    const int ib = tid >> 4;  // this row's block
    const bool live = tid < npad;
    const unsigned below = live ? hm[ib] : 0u;  // bit kb: block (ib, kb)
    float r = live ? b[tid] : 0.0f;
    if (ib == 0) xr[tid] = r;
    auto sixteen = [&](const float* v, f4 (&o)[4]) {
#pragma unroll
        for (int g = 0; g < 4; ++g) o[g] = *reinterpret_cast<const f4*>(v + 4 * g);
    };
    auto dot = [&](const f4 (&a)[4], const f4 (&x)[4]) {
        const f4 s = (a[0] * x[0] + a[1] * x[1]) + (a[2] * x[2] + a[3] * x[3]);
        return (s[0] + s[1]) + (s[2] + s[3]);
    };
    // r -= sum_t a[t] y_t on the lanes that `use` it, y_t on lane t of every row of 16 lanes; the wave's
    // lanes stay together while they read others' y
    auto take = [&](bool use, const f4 (&a)[4], float y) {
        if (!__any(use)) return;
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int t = 0; t < kB; t += 2) {
            s0 = fmaf(a[t >> 2][t & 3], rl(y, t), s0);
            s1 = fmaf(a[(t + 1) >> 2][(t + 1) & 3], rl(y, t + 1), s1);
        }
        r -= use ? s0 + s1 : 0.0f;
    };
    f4 Y[4], p[4], x[4];
    for (int kb = 0; kb < nblk; ++kb) {
        // inverse and own block are loaded before the wait for the right-hand side
        float* Yb = block(H, kb, kb);
#pragma unroll
        for (int g = 0; g < 4; ++g) Y[g] = *group(Yb, c, g);
        const bool use = ib > kb && ((below >> kb) & 1u);
        float* pb = block(H, use ? ib : kb, kb);
#pragma unroll
        for (int g = 0; g < 4; ++g) p[g] = *group(pb, c, g);
        __syncthreads();
        sixteen(xr + kB * kb, x);
        const float y = dot(Y, x);
        take(use, p, y);
        if (ib == kb) r = y;
        if (ib == kb + 1 && live) xr[tid] = r;
    }
    __syncthreads();
    if (ib == nblk - 1) xr[tid] = r;
    for (int kb = nblk - 1; kb >= 0; --kb) {
        float* Yb = block(H, kb, kb);
        float yt[kB], pt[kB];
#pragma unroll
        for (int t = 0; t < kB; ++t) yt[t] = *entry(Yb, t, c);
        const bool use = ib < kb && ((hm[kb] >> ib) & 1u);
        float* pb = block(H, kb, use ? ib : kb);
#pragma unroll
        for (int t = 0; t < kB; ++t) pt[t] = *entry(pb, t, c);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            Y[g] = f4{yt[4 * g], yt[4 * g + 1], yt[4 * g + 2], yt[4 * g + 3]};
            p[g] = f4{pt[4 * g], pt[4 * g + 1], pt[4 * g + 2], pt[4 * g + 3]};
        }
        __syncthreads();
        sixteen(xr + kB * kb, x);
        const float y = dot(Y, x);
        take(use, p, y);
        if (ib == kb) r = y;
        if (ib == kb - 1) xr[tid] = r;
    }
    if (live) b[tid] = r;
    __syncthreads();
}

}  // namespace big
}  // namespace sapx

#endif  // SAPX_STEP_BIG_H
