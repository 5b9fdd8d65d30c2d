// xg_pipeline.hip -- the full motion-search pipeline of a frame with two
// reference pictures, on a raster grid of 16x16 blocks:
//
//   1. k_pipe_full: integer full search +/-range around (0,0) per block and
//      reference (the closed Xin26xMotionEstFull, h26x_core/include/h26x_motion_est.h:26:
//      window intersected with the CU MV window of h266_enc_init.c:1462-1465,
//      cost (SAD << 8) + bits(mvd) * sadLambda, raster order, earliest wins);
//   2. k_pipe_dia: predictor = component-wise median of the left, top and
//      top-right blocks' full-search MVs; start candidates as
//      Xin266FillMeCand (h266_analyze_inter_cu.c:133-293) from the predictor
//      and the own / left / top / top-right MVs; diamond search (the closed
//      Xin26xMotionEstDia); then the half- and quarter-pel rings of
//      Xin266FullSubPelMe (h266_sub_pel_refine.c:81-212) on 8-tap
//      interpolated SAD;
//   3. k_pipe_select: per block the reference with the lower quarter-pel cost
//      (ties: reference 0), written into the session's block list;
//   4. the session's persistent refinement kernel: 1/16-pel candidates around
//      the quarter-pel MV (SATD + chroma) and the motion compensation of the
//      winner.
// All four run on the session stream; in graph mode they are one captured
// HIP graph per frame shape.
//
// Stage 1 is exact but not exhaustive.  The sum over a sub-block of the absolute
// differences is at least the absolute difference of the sub-block's sums, so
// the four 8x8 sums of a block bound its SAD from below.  k_box_sums forms the
// 8x8 and 4x4 sums at every position of both references; k_pipe_bound bounds
// every candidate with two v_sad_u16 instead of 128 and keeps those whose bound
// does not exceed the cost already reached; k_pipe_left costs them.  Blocks that
// keep too many (flat, noisy content) go to the exhaustive k_pipe_full through a
// device list.  3840x2160, two references, +/-64, textured content: 0.85 ms
// (sums 0.02, bounds 0.71, costs 0.08, exhaustive 0.04 for 1.5% of the blocks)
// against 5.24 ms for k_pipe_full over every block.  A whole frame that is flat with
// noise takes 6.65 ms against 5.93.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string.h>
#include <vector>

#include "xg_device.hpp"
#include "xg_runtime.hpp"
#include "xg_sea.hpp"

namespace xg {

constexpr int kPB = 16;                          // block side of the pipeline grid
constexpr int kPipeMaxRange = 64;
constexpr int kPipeQuads = 3;                              // candidate quads per lane in the full search
// window row: 2 * range + 16 samples plus the over-read of the last lane's quads
constexpr int kPipeWinW = 2 * kPipeMaxRange + kPB + 4 * kPipeQuads + 2;   // 158
constexpr int kPipeWinH = 2 * kPipeMaxRange + kPB + 1;    // 145: a two-row item may read one row past the window

// Box sums of a reference plane over positions x0 .. x0 + w - 1, y0 .. y0 + h - 1:
// the sum of the 8x8 (s8) and of the 4x4 samples (s4) from (x, y), at
// [(y - y0) * stride + (x - x0)].  x0, w and stride even, rows of whole dwords.
// 10-bit samples keep 8x8 sums (at most 65,472) in 16 bits.  The plane itself is
// read through the device picture table, so a captured launch follows the pictures.
struct SeaPlane {
    uint16_t *s8, *s4;
    int stride;                    // sums per row
    int x0, y0, w, h;              // covered positions; the samples read end at x0 + w + 8, y0 + h + 7
};

struct SeaPlanes {
    SeaPlane p[2];
    const xg_picture *pics;
    int slot[2];                   // the planes' pictures (even stride, dword aligned: xg_session_set_picture)
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
    const xg_plane &R = pl.pics[pl.slot[blockIdx.z]].plane[0];
    const intptr_t rs = R.stride;
    const gdword *q = (const gdword *)(R.data + (intptr_t)P.y0 * rs + P.x0 + 2 * j);
    const int sp = (int)(rs >> 1), op = P.stride >> 1, last = P.h - 1 + 7;
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

// One launch over both references.
inline void box_sums_enqueue(hipStream_t st, const SeaPlanes &a, int *zero)
{
    const SeaPlane &p = a.p[0];
    k_box_sums<<<dim3((p.w / 2 + 255) / 256, (p.h + kBoxRows - 1) / kBoxRows, 2), 256, 0, st>>>(a, zero);
}

// The full search of a block and reference: the lowest (cost << 32 | position)
// costed, position (my + 128) << 8 | (mx + 128) (raster order), and how many
// candidates the bounded search's scan left.
struct PipeFound {
    unsigned long long best;
    int n, pad;
};
__device__ __forceinline__ int pos_x(unsigned long long best) { return (int)(best & 255) - 128; }
__device__ __forceinline__ int pos_y(unsigned long long best) { return (int)((best >> 8) & 255) - 128; }

struct PipeArgs {
    const xg_picture *pics;
    int curSlot, refSlot0, refSlot1;
    int fw, fh, nbx, nb, range, ctu;
    uint32_t lambda;
    int16_t *fullMv, *predMv, *intMv, *qMv;    // [nb][2 refs][2]
    uint32_t *intCost, *qCost;                 // [nb][2 refs]
    xg_block *blocks;                          // session block list (refinement input)
    SeaPlane sums[2];                          // box sums of the references (k_box_sums)
    PipeFound *found;                          // [nb][2 refs]
    uint32_t *left;                            // [nb][2 refs][kLeftMax]: candidates left, (bound >> 3) << 16 | dy << 8 | dx
    int *dense;                                // [0]: exhaustive searches, [1..]: block * 2 + reference
};

struct IWin { int mnx, mny, mxx, mxy; };       // CU MV window in integer pel

__device__ __forceinline__ IWin int_window(int x, int y, int fw, int fh, int ctu)
{
    IWin w;
    w.mnx = (int16_t)(-x - ctu - 8);
    w.mny = (int16_t)(-y - ctu - 8);
    w.mxx = (int16_t)(fw + (ctu - kPB + 8) - x);
    w.mxy = (int16_t)(fh + (ctu - kPB + 8) - y);
    return w;
}

__device__ __forceinline__ unsigned long long min_u64(unsigned long long a, unsigned long long b)
{
    return a < b ? a : b;
}

__device__ __forceinline__ unsigned long long wave_min_u64(unsigned long long k)
{
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) k = min_u64(k, (unsigned long long)__shfl_xor((long long)k, m, 64));
    return k;
}

// ---------------------------------------------------------------------------
// 1. Full search, exhaustive form: a workgroup per block and reference; LISTED:
// per entry of the list a.dense, the workgroups past its end leave at once (with 1.5 %
// of 64,800 listed the launch takes 36 us, as a resident grid that shares the entries
// out; with all of them listed that grid took 13 % longer, some of its workgroups
// being late)
// ---------------------------------------------------------------------------
// Each lane costs NQ quads (4 * NQ horizontally adjacent candidates) of one
// search row: the window row's dwords D and their one-sample realignment F are
// shared by all of them, so the loads and v_alignbit per v_sad_u16 fall as NQ
// grows.
template <int NQ, bool LISTED>
__global__ void __launch_bounds__(256) k_pipe_full(PipeArgs a)
{
    __shared__ __align__(16) uint16_t win[kPipeWinH * kPipeWinW];
    __shared__ __align__(16) uint32_t curL[kPB * kPB / 2];     // packed pairs
    __shared__ unsigned long long red[4];
    if (LISTED && (int)blockIdx.x >= a.dense[0]) return;
    const int id = LISTED ? a.dense[1 + blockIdx.x] : (int)blockIdx.x;
    const int b = id >> 1, r = id & 1;
    const int x = (b % a.nbx) * kPB, y = (b / a.nbx) * kPB;
    const IWin w = int_window(x, y, a.fw, a.fh, a.ctu);
    const int x0 = max(-a.range, w.mnx), x1 = min(a.range, w.mxx);
    const int y0 = max(-a.range, w.mny), y1 = min(a.range, w.mxy);
    const int nx = x1 - x0 + 1, ny = y1 - y0 + 1;
    const xg_plane &RP = a.pics[r ? a.refSlot1 : a.refSlot0].plane[0];
    const xg_plane &CP = a.pics[a.curSlot].plane[0];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    {   // window rows (ny + 15) x (nx + 15) samples: a wave per row, lanes along it,
        // 4 rows x 3 columns of loads in flight per lane
        const int rows = ny + kPB - 1, cols = nx + kPB - 1;
        const uint16_t *src = RP.data + (intptr_t)(y + y0) * RP.stride + (x + x0);
        for (int r0 = wave; r0 < rows; r0 += 16) {
            uint16_t v[4][3];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint16_t *sp = src + (intptr_t)min(r0 + 4 * k, rows - 1) * RP.stride;
#pragma unroll
                for (int c = 0; c < 3; c++) v[k][c] = sp[min(lane + 64 * c, cols - 1)];
            }
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (r0 + 4 * k < rows)
#pragma unroll
                    for (int c = 0; c < 3; c++)
                        if (lane + 64 * c < cols) win[(r0 + 4 * k) * kPipeWinW + lane + 64 * c] = v[k][c];
        }
        if (tid < kPB * kPB / 2)
            curL[tid] = *reinterpret_cast<const uint32_t *>(CP.data + (intptr_t)(y + (tid >> 3)) * CP.stride + x +
                                                            2 * (tid & 7));
    }
    __syncthreads();
    constexpr int ND = 2 * NQ + 8;                  // window dwords per row read by one lane
    constexpr int NK = 4 * NQ;
    // an item: NK adjacent candidates of two search rows; window row i serves current row i of the
    // first and current row i - 1 of the second, so each window row is read and realigned once
    const int ng = (nx + NK - 1) / NK, items = ((ny + 1) >> 1) * ng;
    const uint32_t *w32 = reinterpret_cast<const uint32_t *>(win);
    unsigned long long best = ~0ull;
    for (int it = tid; it < items; it += 256) {
        const int p = it / ng, g = it - p * ng, dyi = 2 * p;
        const uint32_t *rp = w32 + ((dyi * kPipeWinW) >> 1) + 2 * NQ * g;
        uint32_t acc0[NK], acc1[NK];
#pragma unroll
        for (int k = 0; k < NK; k++) acc0[k] = acc1[k] = 0;
        uint32_t D[ND], F[ND - 1], C[8], Cp[8];
        auto load_row = [&](int i) {
#pragma unroll
            for (int j = 0; j < ND; j++) D[j] = rp[i * (kPipeWinW / 2) + j];
#pragma unroll
            for (int j = 0; j < ND - 1; j++) F[j] = align16(D[j + 1], D[j], 16);    // pairs starting at odd samples
        };
        auto load_cur = [&](int i) {
            const uint4 *c4 = reinterpret_cast<const uint4 *>(curL + i * (kPB / 2));
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint4 v = c4[j];
                C[4 * j] = v.x;
                C[4 * j + 1] = v.y;
                C[4 * j + 2] = v.z;
                C[4 * j + 3] = v.w;
            }
        };
        auto sads = [&](const uint32_t *Cr, uint32_t *acc) {
#pragma unroll
            for (int t = 0; t < NQ; t++)
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    acc[4 * t] = sad2(D[2 * t + j], Cr[j], acc[4 * t]);
                    acc[4 * t + 1] = sad2(F[2 * t + j], Cr[j], acc[4 * t + 1]);
                    acc[4 * t + 2] = sad2(D[2 * t + j + 1], Cr[j], acc[4 * t + 2]);
                    acc[4 * t + 3] = sad2(F[2 * t + j + 1], Cr[j], acc[4 * t + 3]);
                }
        };
        load_row(0);
        load_cur(0);
        sads(C, acc0);
#pragma unroll 2
        for (int i = 1; i < kPB; i++) {
#pragma unroll
            for (int j = 0; j < 8; j++) Cp[j] = C[j];
            load_row(i);
            load_cur(i);
            sads(C, acc0);
            sads(Cp, acc1);
        }
        load_row(kPB);
        sads(C, acc1);
        // the lane's candidates come in raster order, so a strict < keeps the lowest index
        // among equal costs, as the 64-bit key order does
        uint32_t bc = 0xFFFFFFFFu, bi = 0;
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int dy = dyi + r;
            if (dy < ny) {
                const uint32_t by = eg_bits(4 * (y0 + dy));
#pragma unroll
                for (int k = 0; k < NK; k++) {
                    const int ox = NK * g + k;
                    const uint32_t cost = ((r ? acc1[k] : acc0[k]) << 8) + (eg_bits(4 * (x0 + ox)) + by) * a.lambda;
                    if (x0 + ox <= x1 && cost < bc) {
                        bc = cost;
                        bi = (uint32_t)(dy * nx + ox);
                    }
                }
            }
        }
        if (bc != 0xFFFFFFFFu) best = min_u64(best, ((unsigned long long)bc << 32) | bi);
    }
    best = wave_min_u64(best);
    if (lane == 0) red[wave] = best;
    __syncthreads();
    if (tid == 0) {
        best = min_u64(min_u64(red[0], red[1]), min_u64(red[2], red[3]));
        const int idx = (int)(uint32_t)best;
        a.found[id].best = (uint32_t)((y0 + idx / nx + 128) << 8 | (x0 + idx % nx + 128));
    }
}

// ---------------------------------------------------------------------------
// 2. Predictor, candidates, diamond, half/quarter-pel rings (one wave per
//    block and reference)
// ---------------------------------------------------------------------------
__device__ __forceinline__ int median3(int p, int q, int s)
{
    const int lo = min(p, q), hi = max(p, q);
    return min(max(s, lo), hi);
}

// SAD of the current block's row `row` (packed pairs c[0..7]) against the
// reference row at sample (rx, ry) of plane R (16 samples, any parity).
__device__ __forceinline__ uint32_t row_sad(const xg_plane &R, int rx, int ry, const uint32_t *c)
{
    const uint16_t *p = R.data + (intptr_t)ry * R.stride + rx;
    const uint32_t *q = reinterpret_cast<const uint32_t *>(reinterpret_cast<uintptr_t>(p) & ~(uintptr_t)3);
    const uint32_t sh = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 2) << 3;
    uint32_t D[9];
#pragma unroll
    for (int j = 0; j < 9; j++) D[j] = q[j];
    uint32_t acc = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) acc = sad2(align16(D[j + 1], D[j], sh), c[j], acc);
    return acc;
}

__device__ __forceinline__ uint32_t cost_q(uint32_t sad, int mvqx, int mvqy, int px, int py, uint32_t lambda)
{
    return (sad << 8) + (eg_bits(mvqx - px) + eg_bits(mvqy - py)) * lambda;
}

// ---------------------------------------------------------------------------
// 1. Full search, bounded form: a workgroup per 64x64 CTU and reference, a wave per block
// ---------------------------------------------------------------------------
// Costs of four positions at once: the 16 lanes of group lane / 16 cost that
// group's position (mx, my), a row of the block each (c); every lane of the
// group gets the cost.
__device__ __forceinline__ uint32_t cost_row16(const xg_plane &RP, int x, int y, int mx, int my, const uint32_t *c,
                                               uint32_t lambda)
{
    const int row = threadIdx.x & 15;
    const uint32_t s = row_sum<16>(row_sad(RP, x + mx, y + my + row, c));
    return cost_q(s, 4 * mx, 4 * my, 0, 0, lambda);
}

// Lowest of the four groups' (cost, position) keys, in every lane.
__device__ __forceinline__ unsigned long long min_groups(uint32_t cost, uint32_t pos)
{
    unsigned long long k = ((unsigned long long)cost << 32) | pos;
    k = min_u64(k, (unsigned long long)__shfl_xor((long long)k, 16, 64));
    return min_u64(k, (unsigned long long)__shfl_xor((long long)k, 32, 64));
}

// Bound of a block's SAD at the position whose 4x4 sums start at s: 16
// sub-blocks (C4: the block's sums, a row of sub-blocks as two packed pairs).
__device__ __forceinline__ uint32_t bound4(const gword *s, int stride, const uint32_t (&C4)[8])
{
    uint16_t v[16];
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int j = 0; j < 4; j++) v[4 * i + j] = s[4 * j];
        s += 4 * stride;
    }
    uint32_t e = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) e = sad2((uint32_t)v[2 * i] | ((uint32_t)v[2 * i + 1] << 16), C4[i], e);
    return e;
}

// The lane's row of the block at (x, y) (row lane & 15, c) and the block's 4x4
// sums (C4, in every lane; whole waves).
__device__ __forceinline__ void block_sums(const xg_plane &CP, int x, int y, uint32_t (&c)[8], uint32_t (&C4)[8])
{
    const uint32_t *cp = reinterpret_cast<const uint32_t *>(CP.data + (intptr_t)(y + (threadIdx.x & 15)) * CP.stride + x);
#pragma unroll
    for (int j = 0; j < 8; j++) c[j] = cp[j];
    int s[4];
#pragma unroll
    for (int j = 0; j < 4; j++) s[j] = dot2(c[2 * j + 1], 0x00010001u, dot2(c[2 * j], 0x00010001u, 0));
    uint32_t p0 = (uint32_t)s[0] | ((uint32_t)s[1] << 16), p1 = (uint32_t)s[2] | ((uint32_t)s[3] << 16);
    p0 += (uint32_t)shfl_xor<1>((int)p0);
    p1 += (uint32_t)shfl_xor<1>((int)p1);
    p0 += (uint32_t)shfl_xor<2>((int)p0);
    p1 += (uint32_t)shfl_xor<2>((int)p1);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        C4[2 * k] = (uint32_t)__builtin_amdgcn_readlane((int)p0, 4 * k);
        C4[2 * k + 1] = (uint32_t)__builtin_amdgcn_readlane((int)p1, 4 * k);
    }
}

constexpr int kBoundB = 4;                       // blocks per CTU side
constexpr int kBoundWaves = kBoundB * kBoundB;
constexpr int kBoundRows = 2 * kPipeMaxRange + 1 + (kBoundB - 1) * kPB + 8;        // 185
constexpr int kBoundNd = (kBoundB - 1) * kPB / 2 + kPipeMaxRange + 1 + 4;          // 93, odd: rows spread over the banks
constexpr int kBoundList = 368;                  // list entries of a wave; a step adds up to 256
constexpr int kLeftMax = 256;                    // candidates a block may leave for k_pipe_left
constexpr uint32_t kBoundOver = 1u << 22;        // over any limit (a cost >> 8)

// The windows of a CTU's 16 blocks overlap almost wholly, so their union's 8x8
// sums are staged once in LDS (69 KB; two 16-wave workgroups per CU).  Each wave
// then works alone, with no barrier: (1) a limit: the lowest bounds its 16
// 4-lane groups find on every fourth search row are costed, then the neighbours
// of the best for as long as that lowers it; (2) a scan: every candidate whose
// 8x8 bound is within the limit goes to the wave's list; (3) whenever the list
// fills, and at the end, its candidates with a 4x4 bound still within the limit
// go to memory for k_pipe_left, and the lowest four of each 64 are costed, which
// lowers the limit: costing all of them here would leave the workgroup waiting
// for its longest list.  A block that leaves more than kLeftMax goes to the
// exhaustive search.
// Bounds are compared in units of 256 (one SAD), the two shares of the rate
// rounded down.  Positions are dy << 8 | dx, in raster order.
__global__ void __launch_bounds__(64 * kBoundWaves) __attribute__((amdgpu_waves_per_eu(8))) k_pipe_bound(PipeArgs a, int per)
{
    __shared__ uint32_t S[kBoundRows * kBoundNd];
    __shared__ uint32_t byq[2 * kPipeMaxRange + 1 + 2 * 8];      // rate share of row my + range; past the last: over
    __shared__ uint32_t bxq[2 * kPipeMaxRange + 1 + 3];          // of column mx + range + 1; over at both ends
    __shared__ uint16_t list[kBoundWaves][kBoundList];
    // workgroup g runs on XCD g % 8: each XCD takes a contiguous eighth of the CTUs, whose windows overlap
    const int ncx = (a.nbx + kBoundB - 1) / kBoundB, nby = a.nb / a.nbx, ncy = (nby + kBoundB - 1) / kBoundB;
    const int id = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (id >= 2 * ncx * ncy) return;
    const int r = id & 1, ctu = id >> 1;
    const int bx0 = (ctu % ncx) * kBoundB, by0 = (ctu / ncx) * kBoundB;
    const xg_plane &RP = a.pics[r ? a.refSlot1 : a.refSlot0].plane[0];
    const xg_plane &CP = a.pics[a.curSlot].plane[0];
    const SeaPlane &SP = a.sums[r];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int R = a.range;
    // the union of the windows (their starts and ends grow with the block's position)
    const int xl = bx0 * kPB, yl = by0 * kPB;
    const int xr = min(bx0 + kBoundB, a.nbx) * kPB - kPB, yr = min(by0 + kBoundB, nby) * kPB - kPB;
    const int ux = max(xl - R, -a.ctu - 8), uy = max(yl - R, -a.ctu - 8);
    const int rows = min(yr + R, a.fh + a.ctu - 8) - uy + 1 + 8;
    const int col = (ux - SP.x0) & ~1, row = uy - SP.y0;
    {
        const int nd = min(((min(xr + R, a.fw + a.ctu - 8) - SP.x0 - col + 2) >> 1) + 4, kBoundNd);
        const gdword *g = (const gdword *)(SP.s8 + (size_t)row * SP.stride + col);
        const int sw = SP.stride >> 1;
        for (int r0 = wave; r0 < rows; r0 += 4 * kBoundWaves) {
            uint32_t v[4][2];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const gdword *gr = g + (size_t)min(r0 + k * kBoundWaves, rows - 1) * sw;
                v[k][0] = gr[min(lane, nd - 1)];
                v[k][1] = gr[min(lane + 64, nd - 1)];
            }
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (r0 + k * kBoundWaves < rows) {
                    uint32_t *d = S + (r0 + k * kBoundWaves) * kBoundNd + lane;
                    if (lane < nd) d[0] = v[k][0];
                    if (lane + 64 < nd) d[64] = v[k][1];
                }
        }
        if (tid < 2 * R + 17) byq[tid] = tid <= 2 * R ? (eg_bits(4 * (tid - R)) * a.lambda) >> 8 : kBoundOver;
        if (tid < 2 * R + 4) bxq[tid] = tid >= 1 && tid <= 2 * R + 1 ? (eg_bits(4 * (tid - 1 - R)) * a.lambda) >> 8 : kBoundOver;
    }
    __syncthreads();
    const int bx = bx0 + (wave & (kBoundB - 1)), byb = by0 + wave / kBoundB;
    if (bx >= a.nbx || byb >= nby) return;
    const int x = bx * kPB, y = byb * kPB, b = byb * a.nbx + bx;
    const IWin w = int_window(x, y, a.fw, a.fh, a.ctu);
    const int x0 = max(-R, w.mnx), x1 = min(R, w.mxx), y0 = max(-R, w.mny), y1 = min(R, w.mxy);
    const int nx = x1 - x0 + 1, ny = y1 - y0 + 1;
    uint32_t c[8], C4[8], C8[2];
    block_sums(CP, x, y, c, C4);
#pragma unroll
    for (int k = 0; k < 2; k++) {                    // an 8x8 sum is at most 65,472: no carry between the halves
        const uint32_t l = C4[4 * k] + C4[4 * k + 2], h = C4[4 * k + 1] + C4[4 * k + 3];
        C8[k] = ((l & 0xFFFFu) + (l >> 16)) | (((h & 0xFFFFu) + (h >> 16)) << 16);
    }
    // window position (0, 0) in the sums: column p of dword 0 of W, p = 0 or 1
    const int o = x + x0 - SP.x0 - col, p = o & 1;
    const uint32_t *Sw = S + (y + y0 - uy) * kBoundNd + (o >> 1);
    const int lastRow = rows - 1 - (y + y0 - uy);
    const uint32_t *by = byq + y0 + R, *bc = bxq + x0 + R + 1;
    // an item: column pair it % nc, rows it / nc modulo 8; it / nc by a reciprocal exact for it < 1024
    const int nc = (nx + p + 1) >> 1, steps = (ny + 15) >> 4;
    const uint32_t rcp = (65536u + (uint32_t)nc - 1) / (uint32_t)nc;
    auto item_row = [&](int it) { return (int)(((uint32_t)it * rcp) >> 16); };
    unsigned long long best;                         // lowest (cost, position), wave-uniform
    auto lower = [&](uint32_t cost, int pos) {
        const unsigned long long k = min_groups(cost, (uint32_t)pos);
        const uint32_t kh = (uint32_t)__builtin_amdgcn_readfirstlane((int)(k >> 32)), kl = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)k);
        best = min_u64(best, ((unsigned long long)kh << 32) | kl);
    };
    SeaColumn<8> sc;
    {
        uint32_t key = 0xFFFFFFFFu;
        int kpos = 0;
        const int n2 = 2 * nc;
        for (int i0 = 0; i0 == 0 || i0 + 32 < n2; i0 += 64) {
            const int it = min(i0 + lane, n2 - 1), k0 = item_row(it), j = it - k0 * nc, rr = 4 * k0, dx = 2 * j - p;
            uint32_t kl = 0xFFFFFFFFu, kh = 0xFFFFFFFFu;
            sc.open(Sw, kBoundNd, j, rr, lastRow);
            for (int t = 0, dy = rr; t < steps; t++, dy += 16) {
                uint32_t l0, h0, l1, h1;
                sc.step(C8, by[dy], by[dy + 8], l0, h0, l1, h1);
                kl = min(min(kl, (l0 << 5) | (uint32_t)(2 * t)), (l1 << 5) | (uint32_t)(2 * t + 1));
                kh = min(min(kh, (h0 << 5) | (uint32_t)(2 * t)), (h1 << 5) | (uint32_t)(2 * t + 1));
            }
            kl += bc[dx] << 5;
            kh += bc[dx + 1] << 5;
            const uint32_t k = min(kl, kh);
            const int px = min(max(dx + (kh < kl), 0), nx - 1), py = min(rr + 8 * (int)(k & 31u), ny - 1);
            kpos = k < key ? py << 8 | px : kpos;
            key = min(key, k);
        }
        // the lowest of each 4 lanes, a row of 16 lanes costing four of them one after the other
        const unsigned long long m = __ballot(key == min4(key));
        const int low = __shfl(kpos, (lane & 60) + __ffs((int)((m >> (lane & 60)) & 15)) - 1, 64);
        best = ~0ull;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int pos = __shfl(low, (lane & 48) + 4 * k, 64);
            lower(cost_row16(RP, x, y, x0 + (pos & 255), y0 + (pos >> 8), c, a.lambda), pos);
        }
        // the positions beside the best
        for (int k = 0; k < 8; k++) {
            const int bp = (int)(uint32_t)best, g = lane >> 4;
            const int ox = min(max((bp & 255) + (g == 2) - (g == 3), 0), nx - 1);
            const int oy = min(max((bp >> 8) + (g == 0) - (g == 1), 0), ny - 1);
            lower(cost_row16(RP, x, y, x0 + ox, y0 + oy, c, a.lambda), oy << 8 | ox);
            if ((int)(uint32_t)best == bp) break;
        }
    }

    const gword *s4 = (const gword *)(SP.s4 + (size_t)(y + y0 - SP.y0) * SP.stride + (x + x0 - SP.x0));
    uint16_t *mine = list[wave];
    uint32_t *out = a.left + (size_t)(b * 2 + r) * kLeftMax;
    int n = 0, left = 0;
    auto drain = [&]() {
        __builtin_amdgcn_wave_barrier();
        for (int i = 0; i < n; i += 64) {
            const int pos = mine[min(i + lane, n - 1)], oy = pos >> 8, ox = pos & 255;
            const uint32_t q = bound4(s4 + oy * SP.stride + ox, SP.stride, C4) + bc[ox] + by[oy];
            const bool in = i + lane < n && q <= (uint32_t)(best >> 40);
            const unsigned long long m = __ballot(in);
            if (!m) continue;
            const int at = left + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (in && at < kLeftMax) out[at] = min(q >> 3, 65535u) << 16 | (uint32_t)pos;
            left += __popcll(m);
            const uint32_t k = in ? q << 4 | (uint32_t)(lane & 15) : 0xFFFFFFFFu;
            const int cp = __shfl(pos, (lane & 48) | (int)(min16(k) & 15), 64);     // any entry where none is in
            lower(cost_row16(RP, x, y, x0 + (cp & 255), y0 + (cp >> 8), c, a.lambda), cp);
        }
        __builtin_amdgcn_wave_barrier();
        n = 0;
    };
    // steps [u0, u0 + un) of item it (a lane's own; un the same for all)
    auto scan = [&](bool in, int it, int u0, int un) {
        const int k0 = item_row(it), j = it - k0 * nc, dx = 2 * j - p;
        int dy = k0 + 16 * u0;
        sc.open(Sw, kBoundNd, j, dy, lastRow);
        const uint32_t ql = bc[dx], qh = bc[dx + 1];
        for (int u = 0; u < un; u++, dy += 16) {
            uint32_t l0, h0, l1, h1;
            sc.step(C8, by[dy], by[dy + 8], l0, h0, l1, h1);
            // the column's share of the rate is on the limit's side
            const uint32_t limit = (uint32_t)(best >> 40);
            if (!__any((int)min(l0, l1) <= (int)(limit - ql) || (int)min(h0, h1) <= (int)(limit - qh))) continue;
            // (columns and rows past a clipped window have bounds too, but no candidates)
            auto push = [&](uint32_t q, int ddx, int ddy) {
                const bool ok = in && q <= limit && ddx >= 0 && ddx < nx && ddy < ny;
                const unsigned long long m = __ballot(ok);
                if (!m) return;
                const int at = n + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                if (ok) mine[at] = (uint16_t)(ddy << 8 | ddx);
                n += __popcll(m);
            };
            push(l0 + ql, dx, dy);
            push(h0 + qh, dx + 1, dy);
            push(l1 + ql, dx, dy + 8);
            push(h1 + qh, dx + 1, dy + 8);
            if (n > kBoundList - 256) {
                drain();
                if (left > kLeftMax) return;
            }
        }
    };
    // items in rounds of 64; a short remainder (129 columns leave 8 of 520) is spread over its steps
    const int items = 8 * nc, rem = items & 63;
    const bool spread = 2 * ((rem * steps + 63) >> 6) < steps;
    const int whole = spread ? items - rem : items, tasks = spread ? rem * steps : 0;
    for (int i0 = 0; i0 < whole + tasks && left <= kLeftMax; i0 += 64) {
        const int i = i0 + lane;
        int it, u0 = 0;
        bool in;
        if (i0 < whole) {                            // whole rounds first: whole is a multiple of 64 when tasks follow
            it = min(i, items - 1);
            in = i < whole;
        } else {
            const int t = i - whole, k = min(t / steps, rem - 1);
            it = whole + k;
            u0 = min(t - k * steps, steps - 1);
            in = t < tasks;
        }
        scan(in, it, u0, i0 < whole ? steps : 1);
    }
    drain();
    if (lane == 0) {
        const int id = b * 2 + r, pos = (int)(uint32_t)best;
        const PipeFound f = {(best & ~0xFFFFFFFFull) | (uint32_t)((y0 + (pos >> 8) + 128) << 8 | (x0 + (pos & 255) + 128)),
                             left > kLeftMax ? 0 : left, 0};
        a.found[id] = f;
        if (left > kLeftMax) a.dense[1 + atomicAdd(&a.dense[0], 1)] = id;
    }
}

// Costs of the candidates k_pipe_bound left, four at a time and the lowest
// bounds first, by a wave per block and reference: short independent waves, so
// the few blocks with long lists hold nothing else up.
__global__ void __launch_bounds__(256) k_pipe_left(PipeArgs a, int per)
{
    const int g = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    const int id = __builtin_amdgcn_readfirstlane(4 * g + (int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (id >= 2 * a.nb) return;
    const PipeFound f = a.found[id];
    if (!f.n) return;
    const int b = id >> 1, r = id & 1, x = (b % a.nbx) * kPB, y = (b / a.nbx) * kPB;
    const IWin w = int_window(x, y, a.fw, a.fh, a.ctu);
    const int x0 = max(-a.range, w.mnx), y0 = max(-a.range, w.mny);
    const xg_plane &RP = a.pics[r ? a.refSlot1 : a.refSlot0].plane[0];
    const xg_plane &CP = a.pics[a.curSlot].plane[0];
    uint32_t c[8];
    const uint32_t *cp = reinterpret_cast<const uint32_t *>(CP.data + (intptr_t)(y + (lane & 15)) * CP.stride + x);
#pragma unroll
    for (int j = 0; j < 8; j++) c[j] = cp[j];
    const uint32_t *left = a.left + (size_t)id * kLeftMax;
    unsigned long long best = f.best;
    for (int i = 0; i < f.n; i += 64) {
        const uint32_t e = left[min(i + lane, f.n - 1)];
        const int mine = (y0 + (int)((e >> 8) & 255u) + 128) << 8 | (x0 + (int)(e & 255u) + 128);
        bool open = i + lane < f.n && e >> 16 <= (uint32_t)(best >> 43);
        while (__any(open)) {
            const uint32_t k = open ? (e >> 16) << 4 | (uint32_t)(lane & 15) : 0xFFFFFFFFu, m = min16(k);
            open = open && k != m;
            const int pos = __shfl(mine, (lane & 48) | (int)(m & 15), 64);          // any entry where none is open
            const uint32_t cost = cost_row16(RP, x, y, (pos & 255) - 128, (pos >> 8) - 128, c, a.lambda);
            if (__any(cost <= (uint32_t)(best >> 32))) {
                best = min_u64(best, min_groups(cost, (uint32_t)pos));
                open = open && e >> 16 <= (uint32_t)(best >> 43);
            }
        }
    }
    if (lane == 0) a.found[id].best = best;
}

// Bound by VALU issue.  3840x2160, two references, 64,800 waves: 375 -> 209 us,
// 2,990 -> 1,500 vector instructions a wave (159 us to issue).
// What is the same in every lane (predictor, candidate list, the search's position
// and its decisions) is kept in scalars; a 16-lane group costs its own position
// and no other; and the rings filter a column at one of the three horizontal
// offsets a lane (48 of 64), once, into packed row pairs in registers, from which
// the three vertical offsets are formed with scalar taps.
__global__ void __launch_bounds__(64) k_pipe_dia(PipeArgs a, int per)
{
    const int id = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (id >= 2 * a.nb) return;
    const int b = id >> 1, r = id & 1;
    const int by = b / a.nbx, bx = b - by * a.nbx, x = bx * kPB, y = by * kPB;
    const IWin w = int_window(x, y, a.fw, a.fh, a.ctu);
    const xg_plane &RP = a.pics[r ? a.refSlot1 : a.refSlot0].plane[0];
    const xg_plane &CP = a.pics[a.curSlot].plane[0];
    const int lane = threadIdx.x, grp = lane >> 4, row = lane & 15;

    // predictor and start candidates
    int nqx[4], nqy[4];
    {
        const int nbi[4] = {b, bx > 0 ? b - 1 : -1, by > 0 ? b - a.nbx : -1,
                            (by > 0 && bx + 1 < a.nbx) ? b - a.nbx + 1 : -1};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const unsigned long long f = (uint32_t)uniform((int)(uint32_t)a.found[max(nbi[k], 0) * 2 + r].best);
            nqx[k] = nbi[k] < 0 ? 0 : 4 * pos_x(f);
            nqy[k] = nbi[k] < 0 ? 0 : 4 * pos_y(f);
        }
        if (lane == 0) {
            a.fullMv[id * 2] = (int16_t)(nqx[0] >> 2);
            a.fullMv[id * 2 + 1] = (int16_t)(nqy[0] >> 2);
        }
    }
    const int px = (int16_t)median3(nqx[1], nqx[2], nqx[3]), py = (int16_t)median3(nqy[1], nqy[2], nqy[3]);
    int cx[8], cy[8], nc = 1;
#pragma unroll
    for (int j = 0; j < 8; j++) cx[j] = cy[j] = 0;
#pragma unroll
    for (int i = 0; i < 5; i++) {
        const int vx = i == 0 ? px : nqx[i - 1], vy = i == 0 ? py : nqy[i - 1];
        const int ix = (int16_t)((vx + 2) >> 2), iy = (int16_t)((vy + 2) >> 2);
        bool dup = false;
#pragma unroll
        for (int j = 0; j < 6; j++) dup |= (j < nc) && cx[j] == ix && cy[j] == iy;
        if (!dup) {
#pragma unroll
            for (int j = 0; j < 6; j++)
                if (j == nc) {
                    cx[j] = ix;
                    cy[j] = iy;
                }
            nc++;
        }
    }
    // the lane's current row as packed pairs
    uint32_t c[8];
    {
        const uint32_t *cp = reinterpret_cast<const uint32_t *>(CP.data + (intptr_t)(y + row) * CP.stride + x);
#pragma unroll
        for (int j = 0; j < 8; j++) c[j] = cp[j];
    }
    // costs of the four groups' integer positions; UINT32_MAX where a group has none
    auto eval4 = [&](int mx, int my, bool ok, uint32_t *cost) {
        uint32_t s = 0;
        if (ok) s = row_sad(RP, x + mx, y + my + row, c);
        s = row_sum<16>(s);
        const uint32_t k = ok ? cost_q(s, 4 * mx, 4 * my, px, py, a.lambda) : 0xFFFFFFFFu;
#pragma unroll
        for (int g = 0; g < 4; g++) cost[g] = (uint32_t)__builtin_amdgcn_readlane((int)k, 16 * g);
    };
    // start candidates in list order (clipped to the MV window), strict <
    uint32_t best = 0xFFFFFFFFu;
    int bmx = 0, bmy = 0;
#pragma unroll
    for (int base = 0; base < 8; base += 4) {
        if (base >= nc) break;
        uint32_t cost[4];
        int mx[4], my[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            mx[k] = min(max(cx[base + k], w.mnx), w.mxx);
            my[k] = min(max(cy[base + k], w.mny), w.mxy);
        }
        eval4(grp == 0 ? mx[0] : grp == 1 ? mx[1] : grp == 2 ? mx[2] : mx[3],
              grp == 0 ? my[0] : grp == 1 ? my[1] : grp == 2 ? my[2] : my[3], base + grp < nc, cost);
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (cost[k] < best) {
                best = cost[k];
                bmx = mx[k];
                bmy = my[k];
            }
    }
    // small diamond L, R, T, B around the best, inside the window and +/-range of the rounded predictor
    {
        const int ccx = (px + 2) >> 2, ccy = (py + 2) >> 2;
        const int lx = max(w.mnx, ccx - a.range), hx = min(w.mxx, ccx + a.range);
        const int ly = max(w.mny, ccy - a.range), hy = min(w.mxy, ccy + a.range);
        const int gx = (grp == 1) - (grp == 0), gy = (grp == 3) - (grp == 2);
        for (int step = 0; step < 2 * a.range; step++) {
            const int mx = bmx + gx, my = bmy + gy;
            uint32_t cost[4];
            eval4(mx, my, mx >= lx && mx <= hx && my >= ly && my <= hy, cost);
            uint32_t nb = best;
            int win = -1;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (cost[k] < nb) {
                    nb = cost[k];
                    win = k;
                }
            if (win < 0) break;
            bmx += (win == 1) - (win == 0);
            bmy += (win == 3) - (win == 2);
            best = nb;
        }
    }
    if (lane == 0) {
        a.predMv[id * 2] = (int16_t)px;
        a.predMv[id * 2 + 1] = (int16_t)py;
        a.intMv[id * 2] = (int16_t)bmx;
        a.intMv[id * 2 + 1] = (int16_t)bmy;
        a.intCost[id] = best;
    }

    // half- then quarter-pel rings (L, R, T, B, TL, TR, BL, BR), 8-tap SAD, strict <:
    // lane (i, col) = (lane / 16, lane % 16) takes horizontal offset i - 1 and column col;
    // taps and offsets are scaled as in pack_mid16 and clip_hi16
    int qx = bmx * 4, qy = bmy * 4;
    const bool inside = bmx >= w.mnx && bmx <= w.mxx && bmy >= w.mny && bmy <= w.mxy;   // always: the reference's guard
    const int i = min(grp, 2), col = row;
    uint32_t cv[kPB / 2];                            // the column's rows in pairs
    {
        const gword *cp = (const gword *)(CP.data + (intptr_t)y * CP.stride + x + col);
#pragma unroll
        for (int k = 0; k < kPB / 2; k++) cv[k] = pack16(cp[(intptr_t)(2 * k) * CP.stride], cp[(intptr_t)(2 * k + 1) * CP.stride]);
    }
#pragma unroll 1
    for (int step = inside ? 2 : 0; step > 0; step--) {
        const int m16x = 4 * (qx + (i - 1) * step);
        const int top = (4 * (qy - step)) >> 4, spread = ((4 * (qy + step)) >> 4) - top;    // 0 or 1
        const uint16_t *p = RP.data + (intptr_t)(y + top - 3) * RP.stride + x + col + (m16x >> 4) - 3;
        const bool odd = (uintptr_t)p & 2;               // in every row: strides are even
        const gdword *q = (const gdword *)((uintptr_t)p & ~(uintptr_t)3);
        const intptr_t rsw = RP.stride >> 1;
        uint32_t T[5];                                   // tap pairs against the dwords from the one with the first tap
        {
            const int8_t *hf = c_luma[0][m16x & 15];
            uint32_t A[4];
#pragma unroll
            for (int j = 0; j < 4; j++) A[j] = pack16(64 * hf[2 * j], 64 * hf[2 * j + 1]);
            T[0] = odd ? A[0] << 16 : A[0];
#pragma unroll
            for (int j = 1; j < 4; j++) T[j] = odd ? align16(A[j], A[j - 1], 16) : A[j];
            T[4] = odd ? A[3] >> 16 : 0;
        }
        uint32_t P[kPB + 7];                             // P[k]: first-pass rows k and k + 1
        int last = 0;
#pragma unroll
        for (int k = 0; k < kPB + 8; k++) {
            uint32_t D[5];
#pragma unroll
            for (int j = 0; j < 5; j++) D[j] = q[j];
            if (k + 1 < kPB + 7 || spread) q += rsw;     // the last row again when the offsets share their rows
            int u = dot2_first(D[0], T[0], kHRound64);
#pragma unroll
            for (int j = 1; j < 5; j++) u = dot2(D[j], T[j], u);
            if (k) P[k - 1] = pack_mid16(last, u);
            last = u;
            if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // no more than four rows' loads in flight: registers
        }
        int at = top;
        uint32_t mine = 0;
#pragma unroll 1
        for (int j = 0; j < 3; j++) {
            const int my = 4 * (qy + (j - 1) * step);
            if ((my >> 4) != at) {                       // uniform, at most once
#pragma unroll
                for (int k = 0; k < kPB + 6; k++) P[k] = P[k + 1];
                at++;
                asm volatile("");                        // stays a branch
            }
            const int8_t *vf = c_luma[0][my & 15];
            uint32_t V[4];
#pragma unroll
            for (int k = 0; k < 4; k++) V[k] = ((uint32_t)(64 * vf[2 * k]) & 0xFFFF) | (uint32_t)(64 * vf[2 * k + 1]) << 16;
            uint32_t sad = 0;
#pragma unroll
            for (int k = 0; k < kPB; k += 2) {
                int s0 = dot2_first(P[k], V[0], 0), s1 = dot2_first(P[k + 1], V[0], 0);
#pragma unroll
                for (int m = 1; m < 4; m++) {
                    s0 = dot2(P[k + 2 * m], V[m], s0);
                    s1 = dot2(P[k + 1 + 2 * m], V[m], s1);
                }
                sad = sad2(pack_hi16(clip_hi16(s0), clip_hi16(s1)), cv[k / 2], sad);
            }
            sad = row_sum<16>(sad);
            mine = col == j ? sad : mine;
        }
        // lane (i, j): the position at offsets (i - 1, j - 1); its place in the ring's order
        const int dx = i - 1, dy = col - 1;
        const bool ok = grp < 3 && col < 3 && (dx | dy);
        const uint32_t cost = ok ? cost_q(mine, qx + dx * step, qy + dy * step, px, py, a.lambda) : 0xFFFFFFFFu;
        const int order = dy == 0 ? (dx > 0) : dx == 0 ? 2 + (dy > 0) : 4 + 2 * (dy > 0) + (dx > 0);
        const uint32_t lo = wave_min(cost);
        if (lo < best) {
            best = lo;
            const int o = (int)wave_min(cost == lo ? (uint32_t)order : 8u);
            const int wx = o == 2 || o == 3 ? 0 : (o & 1) ? 1 : -1;
            const int wy = o < 2 ? 0 : o == 2 || o == 4 || o == 5 ? -1 : 1;
            qx += wx * step;
            qy += wy * step;
        }
    }
    if (lane == 0) {
        a.qMv[id * 2] = (int16_t)qx;
        a.qMv[id * 2 + 1] = (int16_t)qy;
        a.qCost[id] = best;
    }
}

// ---------------------------------------------------------------------------
// 3. Reference choice -> refinement block list
// ---------------------------------------------------------------------------
__global__ void k_pipe_select(PipeArgs a)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= a.nb) return;
    const int r = a.qCost[b * 2 + 1] < a.qCost[b * 2] ? 1 : 0;
    xg_block B;
    B.x = (int16_t)((b % a.nbx) * kPB);
    B.y = (int16_t)((b / a.nbx) * kPB);
    B.w = kPB;
    B.h = kPB;
    B.pic = (uint8_t)a.curSlot;
    B.ref = (uint8_t)(r ? a.refSlot1 : a.refSlot0);
    B.mvx = 4 * a.qMv[(b * 2 + r) * 2];
    B.mvy = 4 * a.qMv[(b * 2 + r) * 2 + 1];
    B.mvpx = 4 * a.predMv[(b * 2 + r) * 2];
    B.mvpy = 4 * a.predMv[(b * 2 + r) * 2 + 1];
    a.blocks[b] = B;
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct PipeState {
    int fw = 0, fh = 0, nb = 0, cap = 0;
    uint64_t gridVersion = 0;          // session blocksVersion right after the grid was installed
    int16_t *dMv = nullptr;            // fullMv | predMv | intMv | qMv, 4 x nb x 4 int16
    uint32_t *dCost = nullptr;         // intCost | qCost, 2 x nb x 2
    uint16_t *dSums = nullptr;         // box sums of both references, 8 B a sample (72 MB at 4K)
    size_t sumsCap = 0;
    int *dDense = nullptr;             // list of the exhaustive search
    PipeFound *dFound = nullptr;       // the full search's result per block and reference
    uint32_t *dLeft = nullptr;         // what the bounded search's scans leave, 2 KB a block (66 MB at 4K)
    bool bounded = false;              // the full search takes the bounded form
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    uint64_t key = 0;
    PipeArgs args;
};

void pipe_release(xg_session *s)
{
    PipeState *p = static_cast<PipeState *>(session_pipe(s));
    if (!p) return;
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    (void)hipFree(p->dMv);
    (void)hipFree(p->dCost);
    (void)hipFree(p->dSums);
    (void)hipFree(p->dDense);
    (void)hipFree(p->dFound);
    (void)hipFree(p->dLeft);
    delete p;
    session_pipe(s) = nullptr;
}

static uint64_t hmix(uint64_t h, uint64_t v)
{
    h ^= v + 0x9E3779B97F4A7C15ull + (h << 6) + (h >> 2);
    return h;
}

// Largest sadLambda of the bounded search: (SAD << 8) of 26 bits plus at most 38
// MVD bits times lambda stays below 2^28, so its mark for positions past the
// window (kBoundOver) costs more than any candidate and no sum wraps.  The
// encoder's lambdas are below 2^19; larger ones search exhaustively.
constexpr uint32_t kBoundLambda = 1u << 21;
// Fewest blocks of the bounded search.  Below, the CTUs' workgroups and the short
// waves after them leave most of the chip idle and the three launches show:
// whole frames of 920 blocks take 122 us against 106 exhaustively at +/-24 and
// 390 blocks 147 against 117 at +/-64; 2,040 blocks take 140 against 148 at
// +/-16 and 188 against 398 at +/-64, 3,600 blocks 163 against 217 at +/-8.
constexpr int kBoundBlocks = 1600;

// Sum planes of both references over every position the searches read, and
// the list of the exhaustive search.
static bool sums_prepare(PipeState *p, int range, int ctu, hipStream_t st)
{
    const int reach = std::min(range, ctu + 8), left = (reach + 1) & ~1;
    // 4x4 sums to position + 12 of the last candidate; the 8x8 ones (to + 8, + 9 by pairs) fill the same box
    const int w = (p->fw - kPB + reach + 14 + left + 1) & ~1, h = p->fh - kPB + reach + 13 + left;
    const int stride = (int)align_up((size_t)w, 64);
    const size_t one = (size_t)stride * h, need = 4 * one;
    if (need > p->sumsCap) {
        if (!XG_HIP(hipStreamSynchronize(st))) return false;
        (void)hipFree(p->dSums);
        p->dSums = nullptr;
        p->sumsCap = 0;
        if (!XG_HIP(hipMalloc((void **)&p->dSums, need * sizeof(uint16_t)))) return false;
        p->sumsCap = need;
    }
    for (int k = 0; k < 2; k++)
        p->args.sums[k] = {p->dSums + 2 * k * one, p->dSums + (2 * k + 1) * one, stride, -left, -left, w, h};
    p->args.dense = p->dDense;
    p->args.left = p->dLeft;
    return true;
}

static bool enqueue_pipe(const PipeState *p, hipStream_t st, xg_session *s, bool timed)
{
    int ev[2];
    const bool t3 = timed && session_timer_begin(s, 3, ev);
    if (p->bounded) {
        const int nby = p->nb / p->args.nbx;
        const int per = (2 * ((p->args.nbx + kBoundB - 1) / kBoundB) * ((nby + kBoundB - 1) / kBoundB) + 7) / 8;
        const PipeArgs &A = p->args;
        box_sums_enqueue(st, {{A.sums[0], A.sums[1]}, A.pics, {A.refSlot0, A.refSlot1}}, A.dense);
        k_pipe_bound<<<8 * per, 64 * kBoundWaves, 0, st>>>(p->args, per);
        const int perLeft = ((2 * p->nb + 3) / 4 + 7) / 8;
        k_pipe_left<<<8 * perLeft, 256, 0, st>>>(p->args, perLeft);
        k_pipe_full<kPipeQuads, true><<<2 * p->nb, 256, 0, st>>>(p->args);
    } else {
        k_pipe_full<kPipeQuads, false><<<2 * p->nb, 256, 0, st>>>(p->args);
    }
    if (t3) session_timer_end(s, 3, ev);
    const int perDia = (2 * p->nb + 7) / 8;
    k_pipe_dia<<<8 * perDia, 64, 0, st>>>(p->args, perDia);
    k_pipe_select<<<(p->nb + 255) / 256, 256, 0, st>>>(p->args);
    return XG_HIP(hipGetLastError()) && refine_enqueue_prepared(s);
}

}  // namespace xg

using namespace xg;

extern "C" {

int32_t xg_me_pipeline(xg_session *s, const xg_pipeline_cfg *cfg, const xg_picture *cur, const xg_picture *ref0,
                       const xg_picture *ref1, const xg_picture *pred, int32_t mode)
{
    if (!s || !cfg || !cur || !ref0 || !ref1 || !pred || cfg->range < 0 || cfg->range > kPipeMaxRange ||
        cfg->ctuSize < 16 || cfg->ctuSize > 128 || (mode != XG_MODE_BATCHED && mode != XG_MODE_GRAPH)) {
        set_error(XG_ERR_ARG, "xg_me_pipeline: bad arguments");
        return XG_ERR_ARG;
    }
    const int fw = cur->plane[0].width, fh = cur->plane[0].height;
    if (fw < kPB || fh < kPB || (fw % kPB) || (fh % kPB)) {
        set_error(XG_ERR_ARG, "xg_me_pipeline: the frame must be a whole number of 16x16 blocks");
        return XG_ERR_ARG;
    }
    for (const xg_picture *r : {ref0, ref1})
        if (r->plane[0].width != fw || r->plane[0].height != fh || r->plane[0].pad < cfg->ctuSize + 16 ||
            r->plane[1].pad < cfg->ctuSize / 2 + 8) {
            set_error(XG_ERR_ARG, "xg_me_pipeline: reference size/padding (luma pad >= ctuSize + 16)");
            return XG_ERR_ARG;
        }
    const int nbx = fw / kPB, nb = nbx * (fh / kPB);
    SessionView v;
    session_view(s, &v);
    PipeState *p = static_cast<PipeState *>(session_pipe(s));
    if (!p) {
        p = new PipeState();
        session_pipe(s) = p;
    }
    int32_t rc;
    if ((rc = xg_session_set_picture(s, 0, cur)) != XG_OK || (rc = xg_session_set_picture(s, 1, ref0)) != XG_OK ||
        (rc = xg_session_set_picture(s, 2, ref1)) != XG_OK)
        return rc;
    // (re)install the grid when the frame changed or the caller replaced the session's blocks
    if (p->nb != nb || p->fw != fw || p->fh != fh || p->gridVersion != v.blocksVersion) {
        std::vector<xg_block> grid(nb);
        for (int b = 0; b < nb; b++) {
            xg_block &B = grid[b];
            memset(&B, 0, sizeof(B));
            B.x = (int16_t)((b % nbx) * kPB);
            B.y = (int16_t)((b / nbx) * kPB);
            B.w = kPB;
            B.h = kPB;
            B.pic = 0;
            B.ref = 1;
        }
        if ((rc = xg_session_set_blocks(s, grid.data(), nb)) != XG_OK) return rc;
        if (nb > p->cap) {
            if (!XG_HIP(hipStreamSynchronize(v.stream))) return XG_ERR_HIP;
            (void)hipFree(p->dMv);
            (void)hipFree(p->dCost);
            (void)hipFree(p->dDense);
            (void)hipFree(p->dFound);
            (void)hipFree(p->dLeft);
            p->dFound = nullptr;
            p->dLeft = nullptr;
            p->dMv = nullptr;
            p->dCost = nullptr;
            p->dDense = nullptr;
            p->cap = 0;
            if (!XG_HIP(hipMalloc((void **)&p->dMv, sizeof(int16_t) * 16 * (size_t)nb)) ||
                !XG_HIP(hipMalloc((void **)&p->dCost, sizeof(uint32_t) * 4 * (size_t)nb)) ||
                !XG_HIP(hipMalloc((void **)&p->dDense, sizeof(int) * (1 + 2 * (size_t)nb))) ||
                !XG_HIP(hipMalloc((void **)&p->dFound, sizeof(PipeFound) * 2 * (size_t)nb)) ||
                !XG_HIP(hipMalloc((void **)&p->dLeft, sizeof(uint32_t) * 2 * kLeftMax * (size_t)nb)))
                return XG_ERR_NOMEM;
            p->cap = nb;
        }
        p->nb = nb;
        p->fw = fw;
        p->fh = fh;
        session_view(s, &v);
        p->gridVersion = v.blocksVersion;
    }
    if ((rc = refine_prepare(s, &cfg->refine, pred)) != XG_OK) return rc;
    PipeArgs &A = p->args;
    A.pics = v.dPics;
    A.curSlot = 0;
    A.refSlot0 = 1;
    A.refSlot1 = 2;
    A.fw = fw;
    A.fh = fh;
    A.nbx = nbx;
    A.nb = nb;
    A.range = cfg->range;
    A.ctu = cfg->ctuSize;
    A.lambda = cfg->sadLambda;
    A.fullMv = p->dMv;
    A.predMv = p->dMv + 4 * (size_t)nb;
    A.intMv = p->dMv + 8 * (size_t)nb;
    A.qMv = p->dMv + 12 * (size_t)nb;
    A.intCost = p->dCost;
    A.qCost = p->dCost + 2 * (size_t)nb;
    A.blocks = v.dBlocks;
    A.dense = nullptr;
    A.found = p->dFound;
    A.left = nullptr;
    p->bounded = cfg->sadLambda <= kBoundLambda && nb >= kBoundBlocks;
    if (p->bounded && !sums_prepare(p, cfg->range, cfg->ctuSize, v.stream))
        return XG_ERR_NOMEM;
    int ev[2];
    const bool timed = session_timer_begin(s, 4, ev);
    if (mode == XG_MODE_BATCHED) {
        const bool ok = enqueue_pipe(p, v.stream, s, true);
        if (timed) session_timer_end(s, 4, ev);
        return ok ? XG_OK : XG_ERR_HIP;
    }
    uint64_t key = hmix(hmix((uint64_t)nb, (uint64_t)(uintptr_t)v.dPics), (uint64_t)(uintptr_t)v.dBlocks);
    key = hmix(key, ((uint64_t)cfg->range << 40) | ((uint64_t)cfg->ctuSize << 32) | cfg->sadLambda);
    const uint8_t *rb = reinterpret_cast<const uint8_t *>(&cfg->refine);
    for (size_t i = 0; i < sizeof(xg_refine_cfg); i++) key = hmix(key, rb[i]);
    key = hmix(key, (uint64_t)(uintptr_t)p->dMv);
    key = hmix(key, (uint64_t)(uintptr_t)p->dCost);
    if (p->bounded)
        for (const SeaPlane &S : A.sums) key = hmix(key, (uint64_t)(uintptr_t)S.s8);
    key = hmix(hmix(hmix(key, (uint64_t)(uintptr_t)A.dense), (uint64_t)(uintptr_t)A.found), (uint64_t)(uintptr_t)A.left);
    // the captured refinement launch: grid, task lists, tile table, per-block state
    key = hmix(key, refine_prepared_key(s));
    if (!p->exec || key != p->key) {
        if (p->exec) (void)hipGraphExecDestroy(p->exec);
        if (p->graph) (void)hipGraphDestroy(p->graph);
        p->exec = nullptr;
        p->graph = nullptr;
        if (!XG_HIP(hipStreamBeginCapture(v.stream, hipStreamCaptureModeThreadLocal))) return XG_ERR_HIP;
        const bool ok = enqueue_pipe(p, v.stream, s, false);
        hipGraph_t g = nullptr;
        const bool ended = XG_HIP(hipStreamEndCapture(v.stream, &g));
        if (!ok || !ended) return XG_ERR_HIP;
        p->graph = g;
        if (!XG_HIP(hipGraphInstantiate(&p->exec, g, nullptr, nullptr, 0))) return XG_ERR_HIP;
        p->key = key;
    }
    const bool ok = XG_HIP(hipGraphLaunch(p->exec, v.stream));
    if (timed) session_timer_end(s, 4, ev);
    return ok ? XG_OK : XG_ERR_HIP;
}

int32_t xg_me_pipeline_read(xg_session *s, int16_t *fullMv, int16_t *predMv, int16_t *intMv, uint32_t *intCost,
                            int16_t *qMv, uint32_t *qCost)
{
    PipeState *p = s ? static_cast<PipeState *>(session_pipe(s)) : nullptr;
    if (!p || !p->nb) {
        set_error(XG_ERR_STATE, "xg_me_pipeline_read: no pipeline run on this session");
        return XG_ERR_STATE;
    }
    if (xg_session_sync(s) != XG_OK) return XG_ERR_HIP;
    const size_t n4 = 4 * (size_t)p->nb, n2 = 2 * (size_t)p->nb;
    bool ok = true;
    if (fullMv) ok &= XG_HIP(hipMemcpy(fullMv, p->args.fullMv, n4 * sizeof(int16_t), hipMemcpyDeviceToHost));
    if (predMv) ok &= XG_HIP(hipMemcpy(predMv, p->args.predMv, n4 * sizeof(int16_t), hipMemcpyDeviceToHost));
    if (intMv) ok &= XG_HIP(hipMemcpy(intMv, p->args.intMv, n4 * sizeof(int16_t), hipMemcpyDeviceToHost));
    if (qMv) ok &= XG_HIP(hipMemcpy(qMv, p->args.qMv, n4 * sizeof(int16_t), hipMemcpyDeviceToHost));
    if (intCost) ok &= XG_HIP(hipMemcpy(intCost, p->args.intCost, n2 * sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (qCost) ok &= XG_HIP(hipMemcpy(qCost, p->args.qCost, n2 * sizeof(uint32_t), hipMemcpyDeviceToHost));
    return ok ? XG_OK : XG_ERR_HIP;
}

}  // extern "C"
