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

// |a.lo - b.lo| + |a.hi - b.hi| + acc on packed pairs.
__device__ __forceinline__ uint32_t sad2(uint32_t a, uint32_t b, uint32_t acc)
{
    return __builtin_amdgcn_sad_u16(a, b, acc);
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
// rows a step.  The sums of a window sit in LDS, rows `pitch` dwords apart, a dword
// a column pair (2j, 2j + 1); candidate (dx, dy)'s four K x K sub-blocks are at
// columns dx, dx + K and rows dy, dy + K.  lp / hp carry the packed pair (column,
// column + K) of the two columns from step to step, so a row of sums is read
// once for the two candidate rows it serves; rows past the window read its last
// row.  C: the block's sub-block sums, a packed pair per row.  Each bound starts
// from its row's share of the rate (b0, b1).
template <int K>
struct SeaColumn {
    const uint32_t *q;
    int pitch, at, last;           // dword offsets of the current and the last row
    uint32_t lp, hp;
    __device__ __forceinline__ void pair(int o, uint32_t &l, uint32_t &h) const
    {
        const uint32_t u = q[o], v = q[o + K / 2];
        l = __builtin_amdgcn_perm(v, u, 0x05040100u);
        h = __builtin_amdgcn_perm(v, u, 0x07060302u);
    }
    __device__ __forceinline__ void open(const uint32_t *S, int pitch_, int j, int r, int lastRow)
    {
        q = S + j;
        pitch = pitch_;
        last = lastRow * pitch;
        at = min(r * pitch, last);
        pair(at, lp, hp);
    }
    __device__ __forceinline__ void step(const uint32_t (&C)[2], uint32_t b0, uint32_t b1, uint32_t &l0, uint32_t &h0,
                                         uint32_t &l1, uint32_t &h1)
    {
        const int o0 = min(at + K * pitch, last), o1 = min(at + 2 * K * pitch, last);
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
