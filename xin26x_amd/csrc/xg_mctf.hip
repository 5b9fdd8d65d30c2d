// xg_mctf.hip -- motion estimation of the motion-compensated temporal filter.
//
// The reference's MCTF motion search (Xin26xMctfMotionEstFrame,
// h26x_core/include/h26x_mctf.h:27, called per reference, search level and
// block size, with the subsampling Xin26xMctfSubSample, :35, and the MV
// fields l0Mv / l1Mv / l2Mv / mv of h26x_mctf_struct.h:117-127) is closed, so
// this file is a design of its own in that role, hierarchical as the
// published temporal filter of VVC's reference software is:
//   * subsampling: each sample of a half-resolution level is the rounded mean
//     (a + b + c + d + 2) >> 2 of its 2x2 block; the level is edge-padded;
//   * a level: for every block wholly inside the picture, the MVs of the 3x3
//     lower-level blocks around (bx / 2, by / 2), scaled by the resolution
//     factor, and the zero MV are costed (rows then columns), then the integer
//     positions +/-range around the best (rows then columns), then, at the
//     finest level, 7x7 grids of quarter-pel and of 1/16-pel steps around the
//     best; the first strictly lowest SSD wins each comparison.  Fractional
//     predictions use the standard's 8-tap luma filter (h266_luma_mc.c), so
//     every SSD is of a prediction the rest of the library can reproduce.  A
//     position whose 8-tap reach [pos - 3, pos + bs + 4] leaves the
//     reference's padding is not costed.
//   * the frame: 4x level (16x16 blocks, +/-8), 2x level (16x16, +/-5, lower
//     MVs x 2), full resolution (16x16, +/-5, x 2), then 8x8 blocks at full
//     resolution (range 0, lower MVs x 1, fractional rounds).
//
// Mapping: one 64-lane workgroup per block, templated on the block side.  A
// 3x3-and-zero candidate set of integer MVs is costed with a lane per row (four
// or eight candidates at once, straight from the reference); sets with a
// fractional MV one by one from a staged (bs + 7)^2 window with the two-pass
// filter.  The integer search stages its (2 range + bs)^2 window once and each
// lane costs raster positions; the fractional rounds are described at frac_round.
//
// Bound by VALU issue.  1920x1080, before -> now: the 8x8 level with its two
// fractional rounds 280 -> 93 us (49.5 M vector instructions, which take 81 us to
// issue), the three 16x16 levels 41 -> 23 us on average.
#include <algorithm>
#include <mutex>
#include <vector>

#include "xg_device.hpp"
#include "xg_runtime.hpp"

namespace xg {

constexpr int kMctfMaxRange = 8;
constexpr int kMctfMaxBs = 16;

struct MctfArgs {
    const uint16_t *cur;
    intptr_t cs;
    const uint16_t *ref;
    intptr_t rs;
    int w, h, pad;
    int range, rcp, factor;        // rcp: 65536 / (2 range + 1) rounded up, so (p * rcp) >> 16 divides p <= 288
    const int2 *lower;
    int lowerBw, lowerBh;
    int2 *mv;
    uint32_t *err;
    int nbx;
};

// LDS windows are staged shifted, so that column 0 is their first sample
// whatever its address; rows are an odd number of dwords apart.
constexpr int kWinRows = 2 * kMctfMaxRange + kMctfMaxBs;    // 32, also >= bs + 10 of a fractional round
constexpr int kWinDw = kWinRows / 2;                        // dwords staged of a row at most
constexpr int kWinPitch = 19;

template <int BS>
struct MctfLds {
    uint32_t win[kWinRows * kWinPitch];
    uint32_t blk[BS * BS / 2];                              // the current block, BS / 2 dwords a row
    int16_t tmp[(BS + 7) * BS];
};

// Whether the 8-tap reach of a prediction at MV (mx, my) for the block at
// (x, y) stays inside the reference's padding.
template <int BS>
__device__ __forceinline__ bool mctf_valid(const MctfArgs &a, int x, int y, int mx, int my)
{
    const int px = x + (mx >> 4), py = y + (my >> 4);
    return px - 3 >= -a.pad && py - 3 >= -a.pad && px + BS + 4 <= a.w - 1 + a.pad &&
           py + BS + 4 <= a.h - 1 + a.pad;
}

// A reference sample with its coordinates kept inside the padded plane
// (staging may cover cells only invalid positions would read).
__device__ __forceinline__ uint16_t ref_at(const MctfArgs &a, int x, int y)
{
    x = min(max(x, -a.pad), a.w - 1 + a.pad);
    y = min(max(y, -a.pad), a.h - 1 + a.pad);
    return a.ref[(intptr_t)y * a.rs + x];
}

// Stages the window of 2 wd x rows samples at picture position (px, py); wd <= kWinDw.
template <int BS>
__device__ __forceinline__ void stage_window(const MctfArgs &a, MctfLds<BS> &L, int px, int py, int wd, int rows)
{
    const int lane = threadIdx.x, c = lane & (kWinDw - 1), r0 = lane / kWinDw;
    constexpr int STEP = 64 / kWinDw, N = kWinRows / STEP;
    __syncthreads();
    if (px >= -a.pad && py >= -a.pad && px + 2 * wd <= a.w + a.pad && py + rows <= a.h + a.pad) {
        const uint16_t *g = a.ref + (intptr_t)(py + r0) * a.rs + px + 2 * c;
        uint32_t v[N];
#pragma unroll
        for (int k = 0; k < N; k++) {
            if (c < wd && r0 + k * STEP < rows) v[k] = load_pair(g);
            g += STEP * a.rs;
        }
#pragma unroll
        for (int k = 0; k < N; k++)
            if (c < wd && r0 + k * STEP < rows) L.win[(r0 + k * STEP) * kWinPitch + c] = v[k];
    } else if (c < wd) {
        for (int r = r0; r < rows; r += STEP)
            L.win[r * kWinPitch + c] = pack16(ref_at(a, px + 2 * c, py + r), ref_at(a, px + 2 * c + 1, py + r));
    }
    __syncthreads();
}

// SSD of the block (staged in L.blk) against the prediction at MV (mx, my),
// computed by the whole wave; UINT32_MAX when the position is not costed.
template <int BS>
__device__ __forceinline__ uint32_t mctf_candidate(const MctfArgs &a, MctfLds<BS> &L, int x, int y, int mx, int my)
{
    if (!mctf_valid<BS>(a, x, y, mx, my)) return 0xFFFFFFFFu;
    const int lane = threadIdx.x;
    const int8_t *hf = taps_for<8>(mx & 15, 0), *vf = taps_for<8>(my & 15, 0);
    stage_window(a, L, x + (mx >> 4) - 3, y + (my >> 4) - 3, (BS + 8) / 2, BS + 7);
    const uint16_t *w = reinterpret_cast<const uint16_t *>(L.win), *blk = reinterpret_cast<const uint16_t *>(L.blk);
    for (int i = lane; i < (BS + 7) * BS; i += 64)
        L.tmp[i] = (int16_t)hpass<8>(&w[i / BS * 2 * kWinPitch + i % BS], hf);
    __syncthreads();
    uint32_t e = 0;
    for (int i = lane; i < BS * BS; i += 64) {
        int s = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) s += (int)vf[k] * (int)L.tmp[i + k * BS];
        const int d = (int)blk[i] - vfinal_pix(s);
        e += (uint32_t)(d * d);
    }
    return (uint32_t)group_sum<64>((int)e);
}

// SSD of the staged block against the window at (dx, dy) on packed pairs: the
// window pairs realigned by one sample for odd dx (alignbit by 16 dx & 16; an
// even dx also reads the dword past its last pair, inside the window's pitch,
// and shifts it out), each pair difference squared and summed by one v_dot2.
template <int BS>
__device__ __forceinline__ uint32_t int_ssd(const MctfLds<BS> &L, int dx, int dy)
{
    const uint32_t *w = L.win + dy * kWinPitch + (dx >> 1), *b = L.blk;
    const uint32_t sh = (uint32_t)(dx & 1) << 4;
    int e = 0;
#pragma unroll 4
    for (int r = 0; r < BS; r++) {
#pragma unroll
        for (int j = 0; j < BS / 2; j++) {
            const v2s d = as_v2s(b[r * (BS / 2) + j]) - as_v2s(align16(w[r * kWinPitch + j + 1], w[r * kWinPitch + j], sh));
            e = dot2(as_u32(d), as_u32(d), e);
        }
    }
    return (uint32_t)e;
}

// One fractional round: the 7x7 positions around (ox, oy), step sixteenths
// apart, from the window staged at (x0, y0) (picture coordinates).  Lane
// (i, c) = (lane / 8, lane % 8) takes horizontal offset i and column c (and
// c + 8 of a 16-wide block): it filters its column once into packed row pairs
// in registers, and from these forms the prediction at all seven vertical
// offsets, whose taps and first rows are the same in every lane.  So no
// first-pass value goes through LDS, and 56 lanes of 64 work (a lane per
// position leaves 49, each of which reads every first-pass value again).
// Lane (i, j) ends with position (j, i)'s SSD.  Taps and offsets are scaled as
// in pack_mid16 and clip_hi16.
template <int BS>
__device__ __forceinline__ uint32_t frac_round(const MctfLds<BS> &L, int ox, int oy, int step, int rx, int ry)
{
    const int lane = threadIdx.x, i = min(lane >> 3, 6), c = lane & 7;
    const int mx = ox + (i - 3) * step;
    const int col = (mx >> 4) - 3 - rx + c, top = (oy - 3 * step) >> 4;
    const bool odd = col & 1;
    uint32_t T[5];                                    // tap pairs against the dwords from the one with the first tap
    {
        const int8_t *hf = c_luma[0][mx & 15];
        uint32_t A[4];
#pragma unroll
        for (int j = 0; j < 4; j++) A[j] = pack16(64 * hf[2 * j], 64 * hf[2 * j + 1]);
        T[0] = odd ? A[0] << 16 : A[0];
#pragma unroll
        for (int j = 1; j < 4; j++) T[j] = odd ? align16(A[j], A[j - 1], 16) : A[j];
        T[4] = odd ? A[3] >> 16 : 0;
    }
    const uint16_t *blk = reinterpret_cast<const uint16_t *>(L.blk);
    uint32_t mine = 0;
#pragma unroll 1
    for (int h = 0; h < BS / 8; h++) {
        const uint32_t *q = L.win + (top - 3 - ry) * kWinPitch + (col >> 1) + 4 * h;
        uint32_t P[BS + 8], cur[BS / 2];              // P[r]: first-pass rows r and r + 1
#pragma unroll
        for (int r = 0; r < BS; r += 2) cur[r / 2] = pack16(blk[r * BS + 8 * h + c], blk[(r + 1) * BS + 8 * h + c]);
        int last = 0;
#pragma unroll
        for (int r = 0; r <= BS + 8; r++) {
            int u = dot2_first(q[r * kWinPitch], T[0], kHRound64);
#pragma unroll
            for (int j = 1; j < 5; j++) u = dot2(q[r * kWinPitch + j], T[j], u);
            if (r) P[r - 1] = pack_mid16(last, u);
            last = u;
            if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // no more than four rows' reads in flight: registers
        }
        int at = top;                                 // integer row of P[0]'s first tap, 3 above
#pragma unroll 1                                    // one copy of the shift and of the second pass: registers
        for (int j = 0; j < 7; j++) {
            const int my = oy + (j - 3) * step;
            if ((my >> 4) != at) {                    // uniform, at most twice a round
#pragma unroll
                for (int r = 0; r < BS + 7; r++) P[r] = P[r + 1];
                at++;
                asm volatile("");                     // stays a branch: as selects it would cost every offset
            }
            const int8_t *vf = c_luma[0][my & 15];
            uint32_t V[4];
#pragma unroll
            for (int k = 0; k < 4; k++) V[k] = ((uint32_t)(64 * vf[2 * k]) & 0xFFFF) | (uint32_t)(64 * vf[2 * k + 1]) << 16;   // scalars
            int acc = 0;
#pragma unroll
            for (int r = 0; r < BS; r += 2) {
                int s0 = dot2_first(P[r], V[0], 0), s1 = dot2_first(P[r + 1], V[0], 0);
#pragma unroll
                for (int k = 1; k < 4; k++) {
                    s0 = dot2(P[r + 2 * k], V[k], s0);
                    s1 = dot2(P[r + 1 + 2 * k], V[k], s1);
                }
                const v2s d = as_v2s(cur[r / 2]) - as_v2s(pack_hi16(clip_hi16(s0), clip_hi16(s1)));
                acc = dot2(as_u32(d), as_u32(d), acc);
            }
            const uint32_t sum = row_sum<8>((uint32_t)acc);
            mine += c == j ? sum : 0;
        }
    }
    return mine;
}

// FRAC: the finest level's fractional rounds (a separate instantiation, so the
// integer levels keep the register budget of their own code).
template <int BS, bool FRAC>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(FRAC && BS == 16 ? 4 : FRAC ? 6 : 8)))
k_mctf_level(MctfArgs a)
{
    __shared__ MctfLds<BS> L;
    const int lane = threadIdx.x;
    const int by = (int)blockIdx.x / a.nbx, bx = (int)blockIdx.x - by * a.nbx;
    const int x = bx * BS, y = by * BS;
    constexpr int CPR = 64 / BS, NR = (10 + CPR - 1) / CPR;   // candidates at once, rounds of them
    const int row = lane % BS;
    {
        constexpr int N = (BS * BS / 2 + 63) / 64;
        uint32_t v[N];
#pragma unroll
        for (int k = 0; k < N; k++) {
            const int i = lane + 64 * k, r = i / (BS / 2), c = i % (BS / 2);
            if (i < BS * BS / 2) v[k] = load_pair(a.cur + (intptr_t)(y + r) * a.cs + x + 2 * c);
        }
#pragma unroll
        for (int k = 0; k < N; k++)
            if (lane + 64 * k < BS * BS / 2) L.blk[lane + 64 * k] = v[k];
    }
    uint32_t best = 0xFFFFFFFFu;
    int bmx = 0, bmy = 0;
    // candidates: the 3x3 lower-level MVs (rows then columns), then zero
    if (a.lower) {
        int cx[NR], cy[NR];                                   // the lane's candidate of each round
        bool has[NR], allInt = true;
#pragma unroll
        for (int t = 0; t < NR; t++) {
            const int k = t * CPR + lane / BS, ky = (k * 11) >> 5, kx = k - 3 * ky;   // k / 3 for k < 16
            const int tx = bx / 2 + kx - 1, ty = by / 2 + ky - 1;
            cx[t] = cy[t] = 0;
            has[t] = k == 9 || (k < 9 && tx >= 0 && ty >= 0 && tx < a.lowerBw && ty < a.lowerBh);
            if (has[t] && k < 9) {
                const int2 m = a.lower[(intptr_t)ty * a.lowerBw + tx];
                cx[t] = m.x * a.factor;
                cy[t] = m.y * a.factor;
            }
            allInt = allInt && ((cx[t] | cy[t]) & 15) == 0;
        }
        __syncthreads();
        if (__all(allInt)) {
            // integer positions (the lower levels' MVs, scaled, always are): the prediction is the
            // reference itself; a lane takes one row of one candidate, all loads before the first use.
            // A costed position has 3 samples of margin, so the dwords around its rows are in the plane.
            uint32_t D[NR][BS / 2 + 1], sh[NR], e[NR], lo = 0xFFFFFFFFu;
#pragma unroll
            for (int t = 0; t < NR; t++) {
                has[t] = has[t] && mctf_valid<BS>(a, x, y, cx[t], cy[t]);
                if (has[t]) {
                    const uint16_t *p = a.ref + (intptr_t)(y + (cy[t] >> 4) + row) * a.rs + x + (cx[t] >> 4);
                    const gdword *g = (const gdword *)((uintptr_t)p & ~(uintptr_t)3);
                    sh[t] = ((uint32_t)(uintptr_t)p & 2) << 3;
#pragma unroll
                    for (int j = 0; j <= BS / 2; j++) D[t][j] = g[j];
                }
            }
#pragma unroll
            for (int t = 0; t < NR; t++) {
                int s = 0;
#pragma unroll
                for (int j = 0; j < BS / 2; j++) {
                    const v2s d = as_v2s(L.blk[row * (BS / 2) + j]) - as_v2s(align16(D[t][j + 1], D[t][j], sh[t]));
                    s = dot2(as_u32(d), as_u32(d), s);
                }
                e[t] = row_sum<BS>((uint32_t)s);
                if (!has[t]) e[t] = 0xFFFFFFFFu;
                lo = min(lo, e[t]);
            }
            best = wave_min(lo);
            if (best != 0xFFFFFFFFu) {
                // the first candidate with it
                bool found = false;
#pragma unroll
                for (int t = 0; t < NR; t++) {
                    const unsigned long long m = __ballot(e[t] == best);
                    if (m && !found) {
                        found = true;
                        const int l = __builtin_ctzll(m);
                        bmx = __builtin_amdgcn_readlane(cx[t], l);
                        bmy = __builtin_amdgcn_readlane(cy[t], l);
                    }
                }
            }
        } else {
#pragma unroll 1
            for (int k = 0; k < 10; k++) {
                int sx = cx[0], sy = cy[0];
                bool sh = has[0];
#pragma unroll
                for (int t = 1; t < NR; t++)
                    if (k / CPR == t) {
                        sx = cx[t];
                        sy = cy[t];
                        sh = has[t];
                    }
                const int l = k % CPR * BS;
                if (!__builtin_amdgcn_readlane((int)sh, l)) continue;
                sx = __builtin_amdgcn_readlane(sx, l);
                sy = __builtin_amdgcn_readlane(sy, l);
                const uint32_t e = (uint32_t)uniform((int)mctf_candidate(a, L, x, y, sx, sy));
                if (e < best) {
                    best = e;
                    bmx = sx;
                    bmy = sy;
                }
            }
        }
    }
    // integer search +/-range around the best (C division: toward zero); with range 0 around an
    // integer MV that was costed there is nothing new to cost
    if (a.range > 0 || best == 0xFFFFFFFFu || ((bmx | bmy) & 15)) {
        const int R = a.range, ix = bmx / 16, iy = bmy / 16, n1 = 2 * R + 1;
        stage_window(a, L, x + ix - R, y + iy - R, R + BS / 2, 2 * R + BS);
        uint32_t lo = 0xFFFFFFFFu, lp = 0xFFFFFFFFu;
        for (int p = lane; p < n1 * n1; p += 64) {
            const int dy = (p * a.rcp) >> 16, dx = p - dy * n1;
            if (!mctf_valid<BS>(a, x, y, 16 * (ix - R + dx), 16 * (iy - R + dy))) continue;
            const uint32_t e = int_ssd(L, dx, dy);
            if (e < lo) {
                lo = e;
                lp = (uint32_t)p;
            }
        }
        const uint32_t m = wave_min(lo);
        if (m < best) {
            const int p = (int)wave_min(lo == m ? lp : 0xFFFFFFFFu), dy = (p * a.rcp) >> 16, dx = p - dy * n1;
            best = m;
            bmx = 16 * (ix - R + dx);
            bmy = 16 * (iy - R + dy);
        }
    }
    // fractional rounds: 7x7 at quarter-pel steps, then 7x7 at 1/16 pel
    if constexpr (FRAC) {
        const int rx = ((bmx - 15) >> 4) - 3, ry = ((bmy - 15) >> 4) - 3;   // window covering both rounds
        stage_window(a, L, x + rx, y + ry, (((bmx + 15) >> 4) - ((bmx - 15) >> 4) + BS + 8) / 2,
                     ((bmy + 15) >> 4) - ((bmy - 15) >> 4) + BS + 7);
#pragma unroll 1
        for (int step = 4; step >= 1; step -= 3) {
            const int ox = bmx, oy = bmy, i = lane >> 3, j = lane & 7;
            const uint32_t f = frac_round(L, ox, oy, step, rx, ry);
            const bool ok = i < 7 && j < 7 && mctf_valid<BS>(a, x, y, ox + (i - 3) * step, oy + (j - 3) * step);
            const uint32_t e = ok ? f : 0xFFFFFFFFu, m = wave_min(e);
            if (m < best) {
                const int p = (int)wave_min(e == m ? (uint32_t)(7 * j + i) : 0xFFFFFFFFu), pj = (p * 37) >> 8;   // p / 7
                best = m;
                bmx = ox + (p - 7 * pj - 3) * step;
                bmy = oy + (pj - 3) * step;
            }
        }
    }
    if (lane == 0) {
        a.mv[blockIdx.x] = make_int2(bmx, bmy);
        a.err[blockIdx.x] = best;
    }
}

// Rounded 2x2 means of src into dst (w/2 x h/2) with dst's padding filled by
// edge replication: one thread per padded sample of dst.
__global__ void k_mctf_subsample(const uint16_t *__restrict__ src, intptr_t ss, uint16_t *__restrict__ dst,
                                 intptr_t ds, int hw, int hh, int pad)
{
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x) - pad, y = (int)blockIdx.y - pad;
    if (x >= hw + pad) return;
    const int cx = min(max(x, 0), hw - 1), cy = min(max(y, 0), hh - 1);
    const uint16_t *p = src + (intptr_t)(2 * cy) * ss + 2 * cx;
    dst[(intptr_t)y * ds + x] = (uint16_t)(((int)p[0] + p[1] + p[ss] + p[ss + 1] + 2) >> 2);
}

}  // namespace xg

using namespace xg;

namespace {

bool plane_ok(const xg_plane *p)
{
    return p && p->data && p->width >= 2 && p->height >= 2 && p->pad >= 0 && p->stride >= p->width + 2 * p->pad;
}

int32_t level_launch(hipStream_t st, const xg_plane *cur, const xg_plane *ref, int bs, int range,
                     const int32_t *lower, int lowerBw, int lowerBh, int factor, int frac, int32_t *mv, uint32_t *err)
{
    MctfArgs a;
    a.cur = cur->data;
    a.cs = cur->stride;
    a.ref = ref->data;
    a.rs = ref->stride;
    a.w = cur->width;
    a.h = cur->height;
    a.pad = ref->pad;
    a.range = range;
    a.rcp = (65536 + 2 * range) / (2 * range + 1);
    a.factor = factor;
    a.lower = (const int2 *)lower;
    a.lowerBw = lowerBw;
    a.lowerBh = lowerBh;
    a.mv = (int2 *)mv;
    a.err = err;
    a.nbx = cur->width / bs;
    const int n = a.nbx * (cur->height / bs);
    if (n <= 0) return XG_OK;
    if (bs == 8) {
        if (frac) k_mctf_level<8, true><<<n, 64, 0, st>>>(a);
        else k_mctf_level<8, false><<<n, 64, 0, st>>>(a);
    } else {
        if (frac) k_mctf_level<16, true><<<n, 64, 0, st>>>(a);
        else k_mctf_level<16, false><<<n, 64, 0, st>>>(a);
    }
    return XG_HIP(hipGetLastError()) ? XG_OK : XG_ERR_HIP;
}

bool level_args_ok(const char *who, const xg_plane *cur, const xg_plane *ref, int bs, int range, const int32_t *lower,
                   int lowerBw, int lowerBh, int factor, const int32_t *mv, const uint32_t *err)
{
    if (!plane_ok(cur) || !plane_ok(ref) || ref->width != cur->width || ref->height != cur->height ||
        (bs != 8 && bs != 16) || range < 0 || range > kMctfMaxRange || !mv || !err ||
        (lower && (lowerBw < 1 || lowerBh < 1 || factor < 1 || factor > 4))) {
        set_error(XG_ERR_ARG, "%s: bad arguments (planes, blockSize 8 or 16, range 0..%d, lower grid, factor 1..4, "
                              "outputs)", who, kMctfMaxRange);
        return false;
    }
    return true;
}

// Level pictures and fields of xg_mctf_me, one set per session.
struct MctfBufs {
    uint16_t *pic = nullptr;
    int32_t *mv = nullptr;
    uint32_t *err = nullptr;
    size_t picCap = 0, mvCap = 0, errCap = 0;
};
std::mutex g_mctf_mu;
std::vector<std::pair<xg_session *, MctfBufs>> g_mctf;

template <class T>
bool grow(T *&p, size_t &cap, size_t n, hipStream_t st)
{
    if (n <= cap) return true;
    if (p) {
        (void)hipStreamSynchronize(st);
        (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
    if (!XG_HIP(hipMalloc((void **)&p, n * sizeof(T)))) return false;
    cap = n;
    return true;
}

}  // namespace

namespace xg {
void mctf_release(xg_session *s)
{
    std::lock_guard<std::mutex> g(g_mctf_mu);
    for (size_t i = 0; i < g_mctf.size(); i++)
        if (g_mctf[i].first == s) {
            (void)hipFree(g_mctf[i].second.pic);
            (void)hipFree(g_mctf[i].second.mv);
            (void)hipFree(g_mctf[i].second.err);
            g_mctf.erase(g_mctf.begin() + (long)i);
            return;
        }
}
}  // namespace xg

extern "C" {

int32_t xg_mctf_subsample(xg_session *s, const xg_plane *src, const xg_plane *dst)
{
    SessionView v;
    if (!s || !session_view(s, &v) || !plane_ok(src) || !plane_ok(dst) || dst->width != src->width / 2 ||
        dst->height != src->height / 2) {
        set_error(XG_ERR_ARG, "xg_mctf_subsample: bad arguments (planes; dst must be src / 2 in both sides)");
        return XG_ERR_ARG;
    }
    const int pad = dst->pad, hw = dst->width, hh = dst->height;
    k_mctf_subsample<<<dim3((hw + 2 * pad + 255) / 256, hh + 2 * pad), 256, 0, v.stream>>>(
        src->data, src->stride, dst->data, dst->stride, hw, hh, pad);
    return XG_HIP(hipGetLastError()) ? XG_OK : XG_ERR_HIP;
}

int32_t xg_mctf_me_level(xg_session *s, const xg_plane *cur, const xg_plane *ref, int32_t blockSize, int32_t range,
                         const int32_t *lower, int32_t lowerBw, int32_t lowerBh, int32_t factor, int32_t frac,
                         int32_t *mv, uint32_t *err)
{
    SessionView v;
    if (!s || !session_view(s, &v)) {
        set_error(XG_ERR_ARG, "xg_mctf_me_level: bad arguments (no session)");
        return XG_ERR_ARG;
    }
    if (!level_args_ok("xg_mctf_me_level", cur, ref, blockSize, range, lower, lowerBw, lowerBh, factor, mv, err))
        return XG_ERR_ARG;
    return level_launch(v.stream, cur, ref, blockSize, range, lower, lowerBw, lowerBh, factor, frac ? 1 : 0, mv, err);
}

int32_t xg_mctf_me(xg_session *s, const xg_plane *cur, const xg_plane *ref, int32_t *mv, uint32_t *err)
{
    SessionView v;
    if (!s || !session_view(s, &v) || !plane_ok(cur) || !plane_ok(ref) || ref->width != cur->width ||
        ref->height != cur->height || cur->width < 64 || cur->height < 64 || !mv || !err) {
        set_error(XG_ERR_ARG, "xg_mctf_me: bad arguments (planes of the same size, at least 64x64; outputs)");
        return XG_ERR_ARG;
    }
    const int W = cur->width, H = cur->height;
    const int w2 = W / 2, h2 = H / 2, w4 = w2 / 2, h4 = h2 / 2;
    const int p2 = 32, p4 = 16;
    const size_t n2 = (size_t)(w2 + 2 * p2) * (h2 + 2 * p2), n4 = (size_t)(w4 + 2 * p4) * (h4 + 2 * p4);
    const size_t c2 = (size_t)w2 * h2, c4 = (size_t)w4 * h4;
    const int g4x = w4 / 16, g4y = h4 / 16, g2x = w2 / 16, g2y = h2 / 16, g1x = W / 16, g1y = H / 16;
    const size_t nmv = (size_t)g4x * g4y + (size_t)g2x * g2y + (size_t)g1x * g1y;
    MctfBufs *b = nullptr;
    {
        std::lock_guard<std::mutex> g(g_mctf_mu);
        for (auto &p : g_mctf)
            if (p.first == s) b = &p.second;
        if (!b) {
            g_mctf.push_back({s, MctfBufs()});
            b = &g_mctf.back().second;
        }
        if (!grow(b->pic, b->picCap, n2 + n4 + c2 + c4, v.stream) || !grow(b->mv, b->mvCap, 2 * nmv, v.stream) ||
            !grow(b->err, b->errCap, nmv, v.stream))
            return XG_ERR_NOMEM;
    }
    uint16_t *r2 = b->pic, *r4 = r2 + n2, *q2 = r4 + n4, *q4 = q2 + c2;
    const xg_plane R2{r2 + (size_t)p2 * (w2 + 2 * p2) + p2, w2 + 2 * p2, w2, h2, p2};
    const xg_plane R4{r4 + (size_t)p4 * (w4 + 2 * p4) + p4, w4 + 2 * p4, w4, h4, p4};
    const xg_plane C2{q2, w2, w2, h2, 0}, C4{q4, w4, w4, h4, 0};
    int32_t *m4 = b->mv, *m2 = m4 + 2 * (size_t)g4x * g4y, *m1 = m2 + 2 * (size_t)g2x * g2y;
    uint32_t *e4 = b->err, *e2 = e4 + (size_t)g4x * g4y, *e1 = e2 + (size_t)g2x * g2y;
    int32_t rc = XG_OK;
    int evFrame[2], evLast[2];
    const bool tFrame = session_timer_begin(s, 9, evFrame);
    if (rc == XG_OK) rc = xg_mctf_subsample(s, cur, &C2);
    if (rc == XG_OK) rc = xg_mctf_subsample(s, &C2, &C4);
    if (rc == XG_OK) rc = xg_mctf_subsample(s, ref, &R2);
    if (rc == XG_OK) rc = xg_mctf_subsample(s, &R2, &R4);
    if (rc == XG_OK) rc = level_launch(v.stream, &C4, &R4, 16, 8, nullptr, 0, 0, 1, 0, m4, e4);
    if (rc == XG_OK) rc = level_launch(v.stream, &C2, &R2, 16, 5, m4, g4x, g4y, 2, 0, m2, e2);
    if (rc == XG_OK) rc = level_launch(v.stream, cur, ref, 16, 5, m2, g2x, g2y, 2, 0, m1, e1);
    const bool tLast = session_timer_begin(s, 10, evLast);
    if (rc == XG_OK) rc = level_launch(v.stream, cur, ref, 8, 0, m1, g1x, g1y, 1, 1, mv, err);
    if (tLast) session_timer_end(s, 10, evLast);
    if (tFrame) session_timer_end(s, 9, evFrame);
    return rc;
}

}  // extern "C"
