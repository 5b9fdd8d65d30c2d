// xg_sea.hpp -- successive elimination for exact integer searches (the
// block-sum bound of Li and Salari, IEEE Trans. Image Processing 4(1), 1995,
// on sub-block sums): over any sub-block, the sum of absolute differences is at
// least the absolute difference of the two sums.  Box-sum images of a
// reference plane give every candidate's sub-block sums, so a candidate is
// bounded with one v_sad_u16 per two sub-blocks; only candidates whose bound
// does not exceed a cost already reached can win, ties included, so the
// winner is that of the exhaustive search.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "xg_device.hpp"

namespace xg {

// Box sums of a plane over positions x0 .. x0 + w - 1, y0 .. y0 + h - 1: the
// sum of the 8x8 (s8) and of the 4x4 samples (s4) from (x, y), at
// [(y - y0) * stride + (x - x0)].  x0, w and stride even, rows of whole dwords.
// 10-bit samples keep 8x8 sums (at most 65,472) in 16 bits.
struct SeaPlane {
    const uint16_t *src;           // sample (0, 0) of the plane
    intptr_t rs;                   // its stride (even)
    uint16_t *s8, *s4;
    int stride;                    // sums per row
    int x0, y0, w, h;              // covered positions; the samples read end at x0 + w + 8, y0 + h + 7
};

struct SeaPlanes {
    SeaPlane p[2];
};

// Both sums, two columns per thread, kBoxRows rows by sliding sums: row sums of
// 4 samples at columns +0 and +4, their 4-row sums V and V', s4 = V and
// s8(y) = (V + V')(y) + (V + V')(y + 4).  Also clears *zero (a counter of the
// launches that follow), when set.  Memory-bound: 2 bytes read and 4 written
// per position.
constexpr int kBoxRows = 32;

__global__ void __launch_bounds__(256) k_box_sums(SeaPlanes pl, int *zero)
{
    const SeaPlane &P = pl.p[blockIdx.z];
    if (zero && threadIdx.x == 0 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) *zero = 0;
    const int j = (int)(blockIdx.x * blockDim.x + threadIdx.x), r0 = (int)blockIdx.y * kBoxRows;
    if (2 * j >= P.w) return;
    const gdword *q = (const gdword *)(P.src + (intptr_t)P.y0 * P.rs + P.x0 + 2 * j);
    const int sp = (int)(P.rs >> 1), op = P.stride >> 1, last = P.h - 1 + 7;
    uint32_t *o8 = reinterpret_cast<uint32_t *>(P.s8) + j, *o4 = reinterpret_cast<uint32_t *>(P.s4) + j;
    v2s va = {0, 0}, vb = {0, 0}, ra[4], rb[4], t[4];
#pragma unroll
    for (int k = 0; k < 4; k++) ra[k] = rb[k] = t[k] = (v2s){0, 0};
    // row y of the samples completes s4 of row y - 3 and s8 of row y - 7
    for (int y = r0; y < r0 + kBoxRows + 7 && y <= last; y += 4) {
        uint32_t D[4][5];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int c = 0; c < 5; c++) D[k][c] = q[(intptr_t)min(y + k, last) * sp + c];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v2s e[4];
#pragma unroll
            for (int c = 0; c < 4; c++) e[c] = as_v2s(D[k][c]) + as_v2s(align16(D[k][c + 1], D[k][c], 16));
            const v2s ha = e[0] + e[1], hb = e[2] + e[3];
            va += ha - ra[k];
            vb += hb - rb[k];
            ra[k] = ha;
            rb[k] = hb;
            const v2s s = va + vb;
            const int y4 = y + k - 3, y8 = y + k - 7;
            if (y4 >= r0 && y4 < r0 + kBoxRows && y4 < P.h) o4[(size_t)y4 * op] = as_u32(va);
            if (y8 >= r0 && y8 < r0 + kBoxRows && y8 < P.h) o8[(size_t)y8 * op] = as_u32(s + t[k]);
            t[k] = s;
        }
    }
}

// One launch over n (1 or 2) planes of one size.
inline void box_sums_enqueue(hipStream_t st, const SeaPlane *p, int n, int *zero)
{
    SeaPlanes a;
    a.p[0] = p[0];
    a.p[1] = p[n - 1];
    k_box_sums<<<dim3((p[0].w / 2 + 255) / 256, (p[0].h + kBoxRows - 1) / kBoxRows, n), 256, 0, st>>>(a, zero);
}

// Minimum over aligned groups of 4 or 16 lanes, in every lane of the group.
__device__ __forceinline__ uint32_t min4(uint32_t v)
{
    v = min(v, (uint32_t)shfl_xor<1>((int)v));
    return min(v, (uint32_t)shfl_xor<2>((int)v));
}

__device__ __forceinline__ uint32_t min16(uint32_t v)
{
    v = min4(v);
    v = min(v, (uint32_t)shfl_xor<4>((int)v));
    return min(v, (uint32_t)shfl_xor<8>((int)v));
}

// Bounds of the candidates of one column pair on rows r, r + K, r + 2K, ..., two
// rows a step.  The sums of a window sit in LDS, rows PITCH dwords apart, a dword
// a column pair (2j, 2j + 1); candidate (dx, dy)'s four K x K sub-blocks are at
// columns dx, dx + K and rows dy, dy + K.  lp / hp carry the packed pair (column,
// column + K) of the two columns from step to step, so a row of sums is read
// once for the two candidate rows it serves; rows past the window read its last
// row.  C: the block's sub-block sums, a packed pair per row.  Each bound starts
// from its row's share of the rate (b0, b1).
template <int K, int PITCH>
struct SeaColumn {
    const uint32_t *q;
    int at, last;                  // dword offsets of the current and the last row
    uint32_t lp, hp;
    __device__ __forceinline__ void pair(int o, uint32_t &l, uint32_t &h) const
    {
        const uint32_t u = q[o], v = q[o + K / 2];
        l = __builtin_amdgcn_perm(v, u, 0x05040100u);
        h = __builtin_amdgcn_perm(v, u, 0x07060302u);
    }
    __device__ __forceinline__ void open(const uint32_t *S, int j, int r, int lastRow)
    {
        q = S + j;
        last = lastRow * PITCH;
        at = min(r * PITCH, last);
        pair(at, lp, hp);
    }
    __device__ __forceinline__ void step(const uint32_t (&C)[2], uint32_t b0, uint32_t b1, uint32_t &l0, uint32_t &h0,
                                         uint32_t &l1, uint32_t &h1)
    {
        const int o0 = min(at + K * PITCH, last), o1 = min(at + 2 * K * PITCH, last);
        uint32_t ln, hn, lq, hq;
        pair(o0, ln, hn);
        pair(o1, lq, hq);
        l0 = __builtin_amdgcn_sad_u16(ln, C[1], __builtin_amdgcn_sad_u16(lp, C[0], b0));
        h0 = __builtin_amdgcn_sad_u16(hn, C[1], __builtin_amdgcn_sad_u16(hp, C[0], b0));
        l1 = __builtin_amdgcn_sad_u16(lq, C[1], __builtin_amdgcn_sad_u16(ln, C[0], b1));
        h1 = __builtin_amdgcn_sad_u16(hq, C[1], __builtin_amdgcn_sad_u16(hn, C[0], b1));
        lp = lq;
        hp = hq;
        at = o1;
    }
};

}  // namespace xg
