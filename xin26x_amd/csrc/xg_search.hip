// xg_search.hip -- integer and fractional motion search.
//
//  * k_full_search: exhaustive integer search of one block per workgroup; the
//    block's reference window (every candidate position plus the block
//    extent) and the current block are staged once in LDS; each thread costs
//    a strided subset of candidates; the argmin is a 64-bit min over
//    (cost << 32 | raster index), so ties resolve to the earliest candidate
//    in raster order (dy outer, dx inner) whatever the thread schedule.
//    Cost = (SAD << 8) + (EG(4*dx - pmx) + EG(4*dy - pmy)) * lambda
//    (XIN_COST_FRACTION 8, common/include/h26x_definition.h:88; MVD in
//    quarter pel as CALC_MVD_BIT is used at h266_sub_pel_refine.c:155-156).
//  * Xg26xMotionEstDia: start candidates then small-diamond descent, one
//    workgroup, a position per wave.
//  * Xg266FullSubPelMe: the half-pel and quarter-pel rings of
//    h266_encoder/source/h266_sub_pel_refine.c:81-212 with the 8-tap luma
//    interpolation (filterIndex 0) and SAD.
#include <algorithm>
#include <string.h>

#include "xg_device.hpp"
#include "xg_runtime.hpp"
#include "xg_sea.hpp"

namespace xg {

__device__ __forceinline__ unsigned long long block_min_u64(unsigned long long v, unsigned long long *red)
{
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const unsigned long long o = (unsigned long long)__shfl_xor((long long)v, m, 64);
        v = o < v ? o : v;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) red[wid] = v;
    __syncthreads();
    unsigned long long r = red[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); i++) r = red[i] < r ? red[i] : r;
    __syncthreads();
    return r;
}

// One block's full search over window [x0,x1] x [y0,y1] (integer MVs).
// win: reference samples from (x0, y0) relative to the block, stride ws;
// cur: the block, stride bw.  Both in LDS.  STEP: samples whose reads are in flight
// together (bw is a multiple of it).
template <int STEP>
__device__ unsigned long long full_search_core(const uint16_t *win, int ws, const uint16_t *cur, int bw, int bh,
                                               int x0, int x1, int y0, int y1, uint32_t lambda, int pmx, int pmy,
                                               unsigned long long *red)
{
    const int nx = x1 - x0 + 1, n = nx * (y1 - y0 + 1);
    unsigned long long best = ~0ull;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int ox = i % nx, oy = i / nx;
        const uint16_t *w = win + oy * ws + ox;
        uint32_t sad = 0;
        for (int r = 0; r < bh; r++) {
            const uint16_t *wr = w + r * ws, *cr = cur + r * bw;
            for (int c = 0; c < bw; c += STEP)
#pragma unroll
                for (int k = 0; k < STEP; k++) sad += (uint32_t)abs((int)cr[c + k] - (int)wr[c + k]);
        }
        const int mx = x0 + ox, my = y0 + oy;
        const uint32_t cost = (sad << 8) + (eg_bits(4 * mx - pmx) + eg_bits(4 * my - pmy)) * lambda;
        const unsigned long long key = ((unsigned long long)cost << 32) | (uint32_t)i;
        best = key < best ? key : best;
    }
    return block_min_u64(best, red);
}

struct FsFrameArgs {
    const uint16_t *cur; intptr_t cs;
    const uint16_t *ref; intptr_t rs;
    int fw, fh, bw, bh, range, ctu, nbx;
    uint32_t lambda;
    int16_t *bestMv; uint32_t *bestCost; uint32_t *bestSad;
};

// Frame form: block b of the bw x bh grid, predictor (0,0), window
// [-range, range]^2 clipped to the CU MV window (h266_enc_init.c:1462-1465).
__global__ void __launch_bounds__(256) k_full_search_frame(FsFrameArgs a)
{
    extern __shared__ uint16_t smem[];
    __shared__ unsigned long long red[4];
    const int b = blockIdx.x;
    const int x = (b % a.nbx) * a.bw, y = (b / a.nbx) * a.bh;
    const int mnx = (int16_t)(-x - a.ctu - 8), mny = (int16_t)(-y - a.ctu - 8);
    const int mxx = (int16_t)(a.fw + (a.ctu - a.bw + 8) - x), mxy = (int16_t)(a.fh + (a.ctu - a.bh + 8) - y);
    const int x0 = max(-a.range, mnx), x1 = min(a.range, mxx);
    const int y0 = max(-a.range, mny), y1 = min(a.range, mxy);
    const int ws = x1 - x0 + a.bw, wh = y1 - y0 + a.bh;
    uint16_t *win = smem, *cur = smem + ws * wh;
    const uint16_t *rp = a.ref + (intptr_t)(y + y0) * a.rs + (x + x0);
    for (int i = threadIdx.x; i < ws * wh; i += blockDim.x) win[i] = rp[(intptr_t)(i / ws) * a.rs + (i % ws)];
    const uint16_t *cp = a.cur + (intptr_t)y * a.cs + x;
    for (int i = threadIdx.x; i < a.bw * a.bh; i += blockDim.x) cur[i] = cp[(intptr_t)(i / a.bw) * a.cs + (i % a.bw)];
    __syncthreads();
    const unsigned long long k = full_search_core<1>(win, ws, cur, a.bw, a.bh, x0, x1, y0, y1, a.lambda, 0, 0, red);
    if (threadIdx.x == 0) {
        const int i = (int)(uint32_t)k, nx = x1 - x0 + 1;
        const int mx = x0 + i % nx, my = y0 + i / nx;
        a.bestMv[2 * b] = (int16_t)(4 * mx);
        a.bestMv[2 * b + 1] = (int16_t)(4 * my);
        a.bestCost[b] = (uint32_t)(k >> 32);
        uint32_t sad = 0;
        const uint16_t *w = win + (my - y0) * ws + (mx - x0);
        for (int r = 0; r < a.bh; r++)
            for (int c = 0; c < a.bw; c++) sad += (uint32_t)abs((int)cur[r * a.bw + c] - (int)w[r * ws + c]);
        a.bestSad[b] = sad;
    }
}

// ---------------------------------------------------------------------------
// Packed integer search core (block widths 4..64, powers of two)
//
// Each lane costs K horizontally adjacent candidates (Kq .. Kq + K - 1) of one
// search row dyi: a window row is read as BW/2 + K/2 dwords D (sample pairs
// from an even column), F = D realigned by one sample, and v_sad_u16 takes two
// absolute differences per instruction against the packed current row C.
// Window rows are ws samples (ws even, >= nx + BW + K - 1, so the reads of the
// last item stay inside the row); the block is bh rows of BW/2 dwords at a
// 16-byte boundary.  Cost = (SAD << 8) + (EG(4 mx - pmx) + EG(4 my - pmy)) *
// lambda; key = cost << 32 | raster index, as in full_search_core.
// ---------------------------------------------------------------------------

// rows x cols samples from src (row pitch rs) into win (row pitch ws): a wave
// per row, lanes along it, four rows of loads in flight per lane.
__device__ __forceinline__ void stage_rows(uint16_t *win, int ws, const uint16_t *src, intptr_t rs, int rows, int cols)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int r0 = wave; r0 < rows; r0 += 4 * nw) {
        for (int c0 = lane; c0 < cols; c0 += 64) {
            uint16_t v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = src[(intptr_t)min(r0 + k * nw, rows - 1) * rs + c0];
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (r0 + k * nw < rows) win[(r0 + k * nw) * ws + c0] = v[k];
        }
    }
}

// The block's rows as dword pairs (x even, plane dword aligned).
__device__ __forceinline__ void stage_cur(uint32_t *curL, const uint16_t *cp, intptr_t cs, int bw, int bh)
{
    const int nd = bw >> 1;
    for (int i = threadIdx.x; i < bh * nd; i += blockDim.x)
        curL[i] = *reinterpret_cast<const uint32_t *>(cp + (intptr_t)(i / nd) * cs + 2 * (i % nd));
}

template <int BW, int K = 4>
__device__ __forceinline__ unsigned long long packed_items(const uint32_t *w32, int ws, const uint32_t *curL, int bh,
                                                           int x0, int x1, int y0, int nx, int ny, uint32_t lambda,
                                                           int pmx, int pmy)
{
    constexpr int ND = BW / 2;                      // dword pairs per block row
    constexpr int KD = K / 2;                       // dwords the lane's candidates span beyond the block row
    const int nq = (nx + K - 1) / K, items = ny * nq;
    unsigned long long best = ~0ull;
    for (int it = threadIdx.x; it < items; it += blockDim.x) {
        const int dyi = it / nq, q = it - dyi * nq;
        const uint32_t *rp = w32 + ((dyi * ws) >> 1) + KD * q;
        uint32_t acc[K];
#pragma unroll
        for (int k = 0; k < K; k++) acc[k] = 0;
#pragma unroll 2
        for (int i = 0; i < bh; i++) {
            uint32_t D[ND + KD], F[ND + KD - 1], C[ND];
#pragma unroll
            for (int j = 0; j < ND + KD; j++) D[j] = rp[i * (ws >> 1) + j];
            if constexpr (ND >= 4) {
                const uint4 *c4 = reinterpret_cast<const uint4 *>(curL + i * ND);
#pragma unroll
                for (int j = 0; j < ND / 4; j++) {
                    const uint4 v = c4[j];
                    C[4 * j] = v.x;
                    C[4 * j + 1] = v.y;
                    C[4 * j + 2] = v.z;
                    C[4 * j + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int j = 0; j < ND; j++) C[j] = curL[i * ND + j];
            }
#pragma unroll
            for (int j = 0; j < ND + KD - 1; j++) F[j] = align16(D[j + 1], D[j], 16);    // pairs from odd samples
#pragma unroll
            for (int j = 0; j < ND; j++)
#pragma unroll
                for (int m = 0; m < KD; m++) {
                    acc[2 * m] = __builtin_amdgcn_sad_u16(D[j + m], C[j], acc[2 * m]);          // candidate K q + 2m
                    acc[2 * m + 1] = __builtin_amdgcn_sad_u16(F[j + m], C[j], acc[2 * m + 1]);  // K q + 2m + 1
                }
        }
        const int my = y0 + dyi;
        const uint32_t by = eg_bits(4 * my - pmy);
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int mx = x0 + K * q + k;
            if (mx <= x1) {
                const uint32_t cost = (acc[k] << 8) + (eg_bits(4 * mx - pmx) + by) * lambda;
                const unsigned long long key = ((unsigned long long)cost << 32) | (uint32_t)(dyi * nx + K * q + k);
                best = key < best ? key : best;
            }
        }
    }
    return best;
}

// Minimum over the workgroup (up to 16 waves); every thread gets it.
__device__ __forceinline__ unsigned long long block_min_u64_16(unsigned long long v, unsigned long long *red)
{
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const unsigned long long o = (unsigned long long)__shfl_xor((long long)v, m, 64);
        v = o < v ? o : v;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned long long r = red[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); i++) r = red[i] < r ? red[i] : r;
    __syncthreads();
    return r;
}

// Window rows needed by the packed core for nx candidates per row.
__host__ __device__ inline int packed_ws(int nx, int bw, int k = 4) { return (nx + bw + k + 3) & ~1; }

// Candidates per lane of the frame form.  Eight (each window-row read serving
// twice the SADs) measured slightly slower than four at +/-16 and +/-32.
constexpr int kFrameK = 4;

// Threads for a packed search over an n x n candidate window, k candidates
// per lane: the items (search row x run of k candidates) spread evenly over
// the fewest passes a workgroup of at most 1024 threads needs, so no pass runs
// nearly empty (+/-32, k = 4: 1105 items, two passes of 576 threads rather
// than 1024 + 81).
static inline int packed_threads(int n, int k = 4)
{
    const int items = n * ((n + k - 1) / k);
    const int passes = (items + 1023) / 1024;
    return std::min(1024, std::max(64, ((items + passes - 1) / passes + 63) & ~63));
}

// Packed frame form for block widths 8, 16 and 32; same cost, window and tie
// order as k_full_search_frame.
template <int BW>
__global__ void __launch_bounds__(1024) k_full_search_frame_p(FsFrameArgs a, int ws)
{
    extern __shared__ uint32_t smem32[];
    __shared__ unsigned long long red[16];
    const int b = blockIdx.x;
    const int x = (b % a.nbx) * BW, y = (b / a.nbx) * a.bh;
    const int mnx = (int16_t)(-x - a.ctu - 8), mny = (int16_t)(-y - a.ctu - 8);
    const int mxx = (int16_t)(a.fw + (a.ctu - BW + 8) - x), mxy = (int16_t)(a.fh + (a.ctu - a.bh + 8) - y);
    const int x0 = max(-a.range, mnx), x1 = min(a.range, mxx);
    const int y0 = max(-a.range, mny), y1 = min(a.range, mxy);
    const int nx = x1 - x0 + 1, ny = y1 - y0 + 1;
    const int rows = ny + a.bh - 1;
    uint16_t *win = reinterpret_cast<uint16_t *>(smem32);
    uint32_t *curL = smem32 + (((rows * (ws >> 1)) + 3) & ~3);    // 16-byte aligned
    stage_rows(win, ws, a.ref + (intptr_t)(y + y0) * a.rs + (x + x0), a.rs, rows, nx + BW - 1);
    stage_cur(curL, a.cur + (intptr_t)y * a.cs + x, a.cs, BW, a.bh);
    __syncthreads();
    unsigned long long best = packed_items<BW, kFrameK>(smem32, ws, curL, a.bh, x0, x1, y0, nx, ny, a.lambda, 0, 0);
    best = block_min_u64_16(best, red);
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        const int idx = (int)(uint32_t)best;
        const int mx = x0 + idx % nx, my = y0 + idx / nx;
        // the winner's SAD, recomputed by one wave
        uint32_t sad = 0;
        const uint16_t *wr = win + (my - y0) * ws + (mx - x0);
        const uint16_t *cr = reinterpret_cast<const uint16_t *>(curL);
        for (int e = lane; e < a.bh * BW; e += 64) {
            const int r = e / BW, c = e % BW;
            sad += (uint32_t)abs((int)cr[e] - (int)wr[r * ws + c]);
        }
        sad = (uint32_t)group_sum<64>((int)sad);
        if (lane == 0) {
            a.bestMv[2 * b] = (int16_t)(4 * mx);
            a.bestMv[2 * b + 1] = (int16_t)(4 * my);
            a.bestCost[b] = (uint32_t)(best >> 32);
            a.bestSad[b] = sad;
        }
    }
}

// ---------------------------------------------------------------------------
// Bounded frame form (8x8 and 16x16 grids): the results of k_full_search_frame
// from block-sum bounds (xg_sea.hpp) instead of every SAD
//
// A workgroup of four waves takes 2 x 2 blocks, whose windows overlap almost
// wholly: their union is staged once in LDS, and the sums of K x K samples at
// each of its positions (K half the block side: four sub-blocks a block) are
// formed beside it.  Each wave then searches one block alone: (1) a limit: the
// lowest bounds of its 16 4-lane groups on some of the search rows are costed,
// then the neighbours of the best for as long as that lowers it; (2) a scan:
// every candidate with a bound within the limit goes to the block's list.  Then
// all four waves cost the four lists together, from the window in LDS, so one
// long list does not hold the workgroup; a block whose list overflows (flat
// content) they search exhaustively.
// Bounds are compared in units of 256 (one SAD), the two shares of the rate
// rounded down.  Positions are dy << 8 | dx, in raster order.
//
// Bound by VALU issue (staging and sums about a third, the scan the rest) and,
// on small frames, by the latency of one workgroup's phases: about 20 us for a
// lone 16x16 search at range 16, where the exhaustive form takes 12.  Measured,
// exhaustive then this form, several calls in flight, texture with noise:
//   1920x1080 16x16 range 16: 108 -> 33 us; range 40: 606 -> 125; 12: 54 -> 29
//   1920x1080 8x8 range 16: 168 -> 87; range 12: 100 -> 80; range 6: 43 -> 67
//   832x480 16x16 range 16: 22 -> 17; range 12: 13.5 -> 15
//   640x360 16x16 range 16: 14 -> 15; 8x8 range 16: 21 -> 15; 8x8 range 12: 14 -> 14
//   320x320 8x8 range 16: 11 -> 12; 480x400 8x8 range 16: 18 -> 14
// Where nearly every block is searched exhaustively (flat with noise, or noise of
// sigma 64) the limits and scans come on top, and small frames have too few
// workgroups to hide it: 1920x1080 range 16 16x16 107 -> 106 to 111, 8x8 179 -> 172
// to 181, range 32 380 -> 333; 1280x720 range 16 16x16 50 -> 61, 8x8 83 -> 91;
// 832x480 8x8 39 -> 49.  With noise of sigma 16 nothing of this shows (1280x720
// 16x16 50 -> 30).  A lone 640x360 8x8 call at range 16 takes 34.5 -> 33 us.
// The rule: range 16 and over, and 1,750 blocks of 16x16 or 3,500 of 8x8.
// ---------------------------------------------------------------------------
constexpr int kSeaMinRange = 16;
constexpr int kSeaMinWork = 28000;               // blocks times their side
constexpr int kSeaList = 768;                    // list entries of a block
constexpr int kSeaMaxRange = 48;
constexpr uint32_t kSeaOver = 1u << 22;          // over any limit (a cost >> 8)
constexpr uint32_t kSeaLambda = 1u << 21;        // past it the marks above could be undercut: exhaustive

struct SeaFrameArgs {
    FsFrameArgs f;
    int ngx;                                     // groups per row
    int wp, sp;                                  // LDS pitches of window and sums in dwords (odd)
    int rows;                                    // LDS rows of the window
    int aligned;                                 // reference rows are dword aligned
    int most;                                    // list entries past which every candidate is costed instead
};

// LDS dwords of the window, of the sums and in all for a range
static inline void sea_frame_lds(int bs, int range, int *wp, int *sp, int *rows, size_t *bytes)
{
    const int n = 2 * range + 2 * bs;            // window samples a side
    *wp = (n / 2 + 3) | 1;
    *sp = *wp;
    *rows = n;
    *bytes = ((size_t)(*wp + *sp) * n + 2 * (2 * range + 1 + 2 * bs)) * 4 + 4 * kSeaList * 2 + 4 * (size_t)bs * bs * 2 + 16;
}

template <int BS>
__global__ void __launch_bounds__(256) k_search_bound(SeaFrameArgs a)
{
    constexpr int K = BS / 2, LR = BS;           // lanes that cost one candidate: a row each
    constexpr int ND = BS / 2;
    extern __shared__ uint32_t smem32[];
    __shared__ unsigned long long found[4];      // lowest (cost, position) of each block
    __shared__ int lists[4];                     // entries of each list; over a.most: exhaustive
    const FsFrameArgs &f = a.f;
    const int R = f.range, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t *win = smem32, *S = win + a.wp * a.rows;
    uint32_t *byq = S + a.sp * a.rows, *bxq = byq + 2 * R + 1 + 2 * BS;
    uint32_t *curL = bxq + 2 * R + 1 + 2 * BS;   // the four blocks, BS rows of ND dwords each
    uint16_t *list = reinterpret_cast<uint16_t *>(curL + 4 * BS * ND);
    const int nby = f.fh / BS;
    const int gx = (int)blockIdx.x % a.ngx, gy = (int)blockIdx.x / a.ngx;
    const int xl = 2 * gx * BS, yl = 2 * gy * BS;
    const int xr = min(2 * gx + 1, f.nbx - 1) * BS, yr = min(2 * gy + 1, nby - 1) * BS;
    // the union of the windows: their starts and ends grow with the block's position
    const int ux = max(xl - R, -f.ctu - 8), uy = max(yl - R, -f.ctu - 8);
    const int ue = min(xr + R, f.fw + f.ctu - BS + 8) + BS, ve = min(yr + R, f.fh + f.ctu - BS + 8) + BS;   // exclusive
    const int rows = ve - uy;
    // dword loads start at the even column at or left of ux (it shares ux's dword)
    const int lead = a.aligned ? (int)(((reinterpret_cast<uintptr_t>(f.ref) >> 1) + ux) & 1) : 0, cols = ue - ux + lead;
    const uint16_t *src = f.ref + (intptr_t)uy * f.rs + ux - lead;
    if (a.aligned) {
        const int nd = (cols + 1) >> 1;
        for (int r0 = wave; r0 < rows; r0 += 32)
            for (int c = lane; c < nd; c += 64) {
                uint32_t v[8];
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = *(const gdword *)(src + (intptr_t)min(r0 + 4 * k, rows - 1) * f.rs + 2 * c);
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (r0 + 4 * k < rows) win[(r0 + 4 * k) * a.wp + c] = v[k];
            }
    } else {
        for (int r0 = wave; r0 < rows; r0 += 32)
            for (int c = lane; c < cols; c += 64) {
                uint16_t v[8];
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = src[(intptr_t)min(r0 + 4 * k, rows - 1) * f.rs + c];
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (r0 + 4 * k < rows) reinterpret_cast<uint16_t *>(win + (r0 + 4 * k) * a.wp)[c] = v[k];
            }
    }
    if (tid < 2 * R + 1 + 2 * BS) {
        byq[tid] = tid <= 2 * R ? (eg_bits(4 * (tid - R)) * f.lambda) >> 8 : kSeaOver;
        bxq[tid] = tid >= 1 && tid <= 2 * R + 1 ? (eg_bits(4 * (tid - 1 - R)) * f.lambda) >> 8 : kSeaOver;
    }
    // the wave's block and the lane's row of it
    const int bx = 2 * gx + (wave & 1), byb = 2 * gy + (wave >> 1);
    const bool exists = bx < f.nbx && byb < nby;
    const int x = min(bx, f.nbx - 1) * BS, y = min(byb, nby - 1) * BS;
    uint32_t c[ND];
    {
        const gdword *cp = (const gdword *)(f.cur + (intptr_t)(y + lane % LR) * f.cs + x);
#pragma unroll
        for (int j = 0; j < ND; j++) c[j] = cp[j];
        if (lane < LR) {
#pragma unroll
            for (int j = 0; j < ND; j++) curL[(wave * BS + lane) * ND + j] = c[j];
        }
    }
    __syncthreads();
    // sums of K x K samples: a column pair and a run of rows per thread, sliding
    {
        const int nj = (cols - K + 2) >> 1, ns = rows - K + 1;
        const int runs = max(1, 256 / nj), len = (ns + runs - 1) / runs;
        const int run = tid / nj, j = tid - run * nj, y0 = run * len, y1 = min(ns, y0 + len);
        if (run < runs && y0 < y1) {
            auto hsum = [&](int r) {
                uint32_t D[K / 2 + 1];
#pragma unroll
                for (int k = 0; k <= K / 2; k++) D[k] = win[r * a.wp + j + k];
                v2s h = {0, 0};
#pragma unroll
                for (int k = 0; k < K / 2; k++) h += as_v2s(D[k]) + as_v2s(align16(D[k + 1], D[k], 16));
                return h;
            };
            v2s acc = {0, 0};
            for (int r = y0; r < y0 + K - 1; r++) acc += hsum(r);
            for (int r = y0; r < y1; r++) {
                acc += hsum(r + K - 1);
                S[r * a.sp + j] = as_u32(acc);
                acc -= hsum(r);
            }
        }
    }
    __syncthreads();

    // What a block's search needs to know of its window: candidate (0, 0) is
    // column p of dword 0 of W (window) and S (sums), row 0.
    struct View {
        int x0, y0, nx, ny, p;
        const uint32_t *W, *S;
        int lastRow;
    };
    auto view = [&](int bxv, int byv) {
        View v;
        const int xv = bxv * BS, yv = byv * BS;
        const int mnx = (int16_t)(-xv - f.ctu - 8), mny = (int16_t)(-yv - f.ctu - 8);
        const int mxx = (int16_t)(f.fw + (f.ctu - BS + 8) - xv), mxy = (int16_t)(f.fh + (f.ctu - BS + 8) - yv);
        v.x0 = max(-R, mnx);
        v.y0 = max(-R, mny);
        v.nx = min(R, mxx) - v.x0 + 1;
        v.ny = min(R, mxy) - v.y0 + 1;
        const int o = xv + v.x0 - ux + lead, oy = yv + v.y0 - uy;
        v.p = o & 1;
        v.W = win + oy * a.wp + (o >> 1);
        v.S = S + oy * a.sp + (o >> 1);
        v.lastRow = rows - K - oy;
        return v;
    };
    // SADs of 64 / LR positions at once: the LR lanes of a group cost that group's position against the
    // row c of the block, in every lane of it
    auto cost_of = [&](const View &v, const uint32_t *c, int pos) {
        const int cy = pos >> 8, cx = (pos & 255) + v.p;
        const uint32_t *w = v.W + (cy + lane % LR) * a.wp + (cx >> 1);
        const uint32_t sh = (uint32_t)(cx & 1) << 4;
        uint32_t D[ND + 1], e = 0;
#pragma unroll
        for (int j = 0; j <= ND; j++) D[j] = w[j];
#pragma unroll
        for (int j = 0; j < ND; j++) e = sad2(align16(D[j + 1], D[j], sh), c[j], e);
        e = (uint32_t)group_sum<LR>((int)e);
        return (e << 8) + (eg_bits(4 * (v.x0 + (pos & 255))) + eg_bits(4 * (v.y0 + cy))) * f.lambda;
    };
    // lowest key of the groups, in every lane
    auto lowest = [&](uint32_t cost, int pos) {
        unsigned long long k = ((unsigned long long)cost << 32) | (uint32_t)pos;
#pragma unroll
        for (int m = LR; m < 64; m <<= 1) {
            const unsigned long long q = (unsigned long long)__shfl_xor((long long)k, m, 64);
            k = q < k ? q : k;
        }
        return k;
    };
    if (exists) {
    // the block's four sums, a pair per row of sub-blocks: lanes 0 .. K - 1 hold the upper rows
    uint32_t C[2];
    {
        int l = 0, h = 0;
#pragma unroll
        for (int j = 0; j < ND / 2; j++) {
            l = dot2(c[j], 0x00010001u, l);
            h = dot2(c[ND / 2 + j], 0x00010001u, h);
        }
        uint32_t v = (uint32_t)l | ((uint32_t)h << 16);              // each half at most 65,472 when summed
        v += (uint32_t)shfl_xor<1>((int)v);
        v += (uint32_t)shfl_xor<2>((int)v);
        if (K == 8) v += (uint32_t)shfl_xor<4>((int)v);
        C[0] = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
        C[1] = (uint32_t)__builtin_amdgcn_readlane((int)v, K);
    }
    const View v = view(bx, byb);
    const int nx = v.nx, ny = v.ny, p = v.p;
    const uint32_t *by = byq + v.y0 + R, *bc = bxq + v.x0 + R + 1;
    const int nc = (nx + p + 1) >> 1, steps = (ny + 2 * K - 1) / (2 * K);
    const uint32_t rcp = (65536u + (uint32_t)nc - 1) / (uint32_t)nc;   // it / nc, exact for it < 1024
    auto item_row = [&](int it) { return (int)(((uint32_t)it * rcp) >> 16); };
    unsigned long long best = ~0ull;                 // lowest (cost, position), wave-uniform
    auto lower = [&](uint32_t cost, int pos) {
        const unsigned long long k = lowest(cost, pos);
        const uint32_t kh = (uint32_t)__builtin_amdgcn_readfirstlane((int)(k >> 32)),
                       kl = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)k);
        const unsigned long long u = ((unsigned long long)kh << 32) | kl;
        best = u < best ? u : best;
    };
    SeaColumn<K> sc;
    {
        uint32_t key = 0xFFFFFFFFu;
        int kpos = 0;
        const int n2 = 2 * nc;                       // rows 0 and K / 2 modulo K
        for (int i0 = 0; i0 == 0 || i0 + 32 < n2; i0 += 64) {
            const int it = min(i0 + lane, n2 - 1), k0 = item_row(it), j = it - k0 * nc, rr = (K / 2) * k0, dx = 2 * j - p;
            uint32_t kl = 0xFFFFFFFFu, kh = 0xFFFFFFFFu;
            sc.open(v.S, a.sp, j, rr, v.lastRow);
            for (int t = 0, dy = rr; t < steps; t++, dy += 2 * K) {
                uint32_t l0, h0, l1, h1;
                sc.step(C, by[dy], by[dy + K], l0, h0, l1, h1);
                kl = min(min(kl, (l0 << 5) | (uint32_t)(2 * t)), (l1 << 5) | (uint32_t)(2 * t + 1));
                kh = min(min(kh, (h0 << 5) | (uint32_t)(2 * t)), (h1 << 5) | (uint32_t)(2 * t + 1));
            }
            kl += bc[dx] << 5;
            kh += bc[dx + 1] << 5;
            const uint32_t k = min(kl, kh);
            const int px = min(max(dx + (kh < kl), 0), nx - 1), py = min(rr + K * (int)(k & 31u), ny - 1);
            kpos = k < key ? py << 8 | px : kpos;
            key = min(key, k);
        }
        // the lowest of each 4 lanes, costed 64 / LR at a time
        const unsigned long long m = __ballot(key == min4(key));
        const int low = __shfl(kpos, (lane & 60) + __ffs((int)((m >> (lane & 60)) & 15)) - 1, 64);
#pragma unroll
        for (int k = 0; k < LR / 4; k++) {
            const int pos = __shfl(low, (lane / LR) * LR + 4 * k, 64);
            lower(cost_of(v, c, pos), pos);
        }
        for (int k = 0; k < 8; k++) {
            const int bp = (int)(uint32_t)best, g = (lane / LR) & 3;
            const int ax = min(max((bp & 255) + (g == 2) - (g == 3), 0), nx - 1);
            const int ay = min(max((bp >> 8) + (g == 0) - (g == 1), 0), ny - 1);
            lower(cost_of(v, c, ay << 8 | ax), ay << 8 | ax);
            if ((int)(uint32_t)best == bp) break;
        }
    }

    uint16_t *mine = list + wave * kSeaList;
    const uint32_t limit = (uint32_t)(best >> 40);
    int n = 0;
    const int items = K * nc, rem = items & 63;
    const bool spread = 2 * ((rem * steps + 63) >> 6) < steps;
    const int whole = spread ? items - rem : items, tasks = spread ? rem * steps : 0;
    for (int i0 = 0; i0 < whole + tasks && n <= a.most; i0 += 64) {
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
        const int un = i0 < whole ? steps : 1;
        const int k0 = item_row(it), j = it - k0 * nc, dx = 2 * j - p;
        int dy = k0 + 2 * K * u0;
        sc.open(v.S, a.sp, j, dy, v.lastRow);
        const uint32_t ql = bc[dx], qh = bc[dx + 1];
        for (int u = 0; u < un; u++, dy += 2 * K) {
            uint32_t l0, h0, l1, h1;
            sc.step(C, by[dy], by[dy + K], l0, h0, l1, h1);
            if (!__any((int)min(l0, l1) <= (int)(limit - ql) || (int)min(h0, h1) <= (int)(limit - qh))) continue;
            auto push = [&](uint32_t q, int ddx, int ddy) {
                const bool ok = in && q <= limit && ddx >= 0 && ddx < nx && ddy < ny;
                const unsigned long long m = __ballot(ok);
                if (!m) return;
                const int at = n + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                if (ok && at < kSeaList) mine[at] = (uint16_t)(ddy << 8 | ddx);
                n += __popcll(m);
            };
            push(l0 + ql, dx, dy);
            push(h0 + qh, dx + 1, dy);
            push(l1 + ql, dx, dy + K);
            push(h1 + qh, dx + 1, dy + K);
        }
    }
    if (lane == 0) {
        found[wave] = best;
        lists[wave] = n;
    }
    } else if (lane == 0) {
        lists[wave] = 0;
    }
    __syncthreads();

    // all waves: every block's list, or every candidate of a block whose list overflowed, 64 items
    // (four adjacent candidates of a row) a wave in turn over all such blocks
    int turn = 0;
    for (int q = 0; q < 4; q++) {
        const int n = lists[q];
        if (!n) continue;
        const View v = view(2 * gx + (q & 1), 2 * gy + (q >> 1));
        const uint32_t *cl = curL + q * BS * ND;
        unsigned long long k = ~0ull;
        if (n <= a.most) {
            const uint32_t *cr = cl + (lane % LR) * ND;
#pragma unroll
            for (int j = 0; j < ND; j++) c[j] = cr[j];
            for (int i = wave * (64 / LR); i < n; i += 4 * (64 / LR)) {
                const int pos = list[q * kSeaList + min(i + lane / LR, n - 1)];
                const unsigned long long o = ((unsigned long long)cost_of(v, c, pos) << 32) | (uint32_t)pos;
                k = o < k ? o : k;
            }
        } else {
            // four adjacent candidates of a row a thread, which come in raster order: strict < keeps the earliest
            const int nq = (v.nx + v.p + 3) >> 2, items = v.ny * nq;
            const int first = 64 * ((wave - turn) & 3) + lane;
            turn += (items + 63) >> 6;
            uint32_t bcst = 0xFFFFFFFFu;
            int bpos = 0;
            for (int it = first; it < items; it += 256) {
                const int dy = it / nq, qd = it - dy * nq;
                const uint32_t *w = v.W + dy * a.wp + 2 * qd;
                uint32_t acc[4] = {0, 0, 0, 0};
#pragma unroll 2
                for (int r = 0; r < BS; r++) {
                    uint32_t D[ND + 2];
#pragma unroll
                    for (int j = 0; j < ND + 2; j++) D[j] = w[r * a.wp + j];
#pragma unroll
                    for (int j = 0; j < ND; j++) {
                        const uint32_t cj = cl[r * ND + j];
                        acc[0] = sad2(D[j], cj, acc[0]);
                        acc[1] = sad2(align16(D[j + 1], D[j], 16), cj, acc[1]);
                        acc[2] = sad2(D[j + 1], cj, acc[2]);
                        acc[3] = sad2(align16(D[j + 2], D[j + 1], 16), cj, acc[3]);
                    }
                }
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const int dx = 4 * qd + m - v.p;
                    const uint32_t cost = (acc[m] << 8) + (eg_bits(4 * (v.x0 + dx)) + eg_bits(4 * (v.y0 + dy))) * f.lambda;
                    if (dx >= 0 && dx < v.nx && cost < bcst) {
                        bcst = cost;
                        bpos = dy << 8 | dx;
                    }
                }
            }
            k = ((unsigned long long)bcst << 32) | (uint32_t)bpos;
        }
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const unsigned long long o = (unsigned long long)__shfl_xor((long long)k, m, 64);
            k = o < k ? o : k;
        }
        if (lane == 0) atomicMin(&found[q], k);
    }
    __syncthreads();
    if (exists && lane == 0) {
        const View v = view(bx, byb);
        const unsigned long long best = found[wave];
        const int b = byb * f.nbx + bx, pos = (int)(uint32_t)best, mx = v.x0 + (pos & 255), my = v.y0 + (pos >> 8);
        const uint32_t cost = (uint32_t)(best >> 32);
        f.bestMv[2 * b] = (int16_t)(4 * mx);
        f.bestMv[2 * b + 1] = (int16_t)(4 * my);
        f.bestCost[b] = cost;
        f.bestSad[b] = (cost - (eg_bits(4 * mx) + eg_bits(4 * my)) * f.lambda) >> 8;
    }
}

// Region and block (na and nb packed samples, 16-byte aligned, readable to a
// multiple of 8) into LDS at dst and dst + align8(na), 16 bytes a thread and
// load, every load of a thread issued before its first store: over the bus each
// round trip costs about 2 us.
__host__ __device__ constexpr int align8(int n) { return (n + 7) & ~7; }

__device__ __forceinline__ void stage_packed(uint16_t *dst, const uint16_t *a, int na, const uint16_t *b, int nb)
{
    const int qa = (na + 7) >> 3, n = qa + ((nb + 7) >> 3);
    const uint4 *pa = reinterpret_cast<const uint4 *>(a), *pb = reinterpret_cast<const uint4 *>(b) - qa;
    for (int i0 = threadIdx.x; i0 < n; i0 += 8 * (int)blockDim.x) {
        uint4 v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int i = min(i0 + k * (int)blockDim.x, n - 1);
            v[k] = *(i < qa ? pa + i : pb + i);
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int i = i0 + k * (int)blockDim.x;
            if (i < n) reinterpret_cast<uint4 *>(dst)[i] = v[k];
        }
    }
}

// Per-call form: packed window and block, which may be mapped host memory, are
// read once into LDS.  A sample a load, a round trip per 256 samples: 4x4 at +/-84
// took 256 us, 16x16 at +/-16 90 (177 and 83 with copies to device memory); with
// 16-byte loads 146 and 83.  Costing a sample at a time waits for its two reads,
// and its time moves by 3 % with its place in the code; STEP 4 takes the widths that
// are multiples of 4 (104 and 59; 64x64 at +/-44 6,142 -> 3,610, 5,943 with copies).
template <int STEP>
__global__ void __launch_bounds__(256) k_full_search_one(const uint16_t *gwin, int ws, int wh, const uint16_t *gcur,
                                                         int bw, int bh, int x0, int x1, int y0, int y1,
                                                         uint32_t lambda, int pmx, int pmy, uint32_t *out)
{
    extern __shared__ __align__(16) uint16_t smem[];
    __shared__ unsigned long long red[4];
    const uint16_t *win = smem, *cur = smem + align8(ws * wh);
    stage_packed(smem, gwin, ws * wh, gcur, bw * bh);
    __syncthreads();
    const unsigned long long k = full_search_core<STEP>(win, ws, cur, bw, bh, x0, x1, y0, y1, lambda, pmx, pmy, red);
    if (threadIdx.x == 0) {
        const int i = (int)(uint32_t)k, nx = x1 - x0 + 1;
        const int mx = x0 + i % nx, my = y0 + i / nx;
        uint32_t sad = 0;
        const uint16_t *w = win + (my - y0) * ws + (mx - x0);
        for (int r = 0; r < bh; r++)
            for (int c = 0; c < bw; c++) sad += (uint32_t)abs((int)cur[r * bw + c] - (int)w[r * ws + c]);
        out[0] = (uint32_t)mx;
        out[1] = (uint32_t)my;
        out[2] = (uint32_t)(k >> 32);
        out[3] = sad;
    }
}

// SAD of the block at integer offset (mx, my) inside a packed region whose
// origin is (rx0, ry0) relative to the co-located position, by the calling wave;
// every lane gets it.
__device__ uint32_t wave_sad(const uint16_t *reg, int rstride, int rx0, int ry0, const uint16_t *cur, int bw, int bh,
                             int mx, int my)
{
    const int lane = threadIdx.x & 63, dr = 64 / bw, dc = 64 - dr * bw;
    const uint16_t *w = reg + (my - ry0) * rstride + (mx - rx0);
    int r = lane / bw, c = lane - r * bw;
    uint32_t s = 0;
    for (int i = lane; i < bw * bh; i += 64) {
        s += (uint32_t)abs((int)cur[i] - (int)w[r * rstride + c]);
        r += dr;
        c += dc;
        if (c >= bw) {
            c -= bw;
            r++;
        }
    }
    return (uint32_t)group_sum<64>((int)s);
}

// Diamond search in one workgroup of four waves; the region covers every
// position the search can read.  Each wave costs one of four positions at a time
// (start candidates, then the diamond's four), so a step is one barrier pair.
// STAGE: region and block are read once into LDS (they may be mapped host
// memory).  out: bestX, bestY (integer pel), cost, sad.
struct DiaCands {
    int16_t v[24];                 // (x, y) of up to 12
};

template <bool STAGE>
__global__ void __launch_bounds__(256) k_dia_one(const uint16_t *greg, int rstride, int rrows, int rx0, int ry0,
                                                 const uint16_t *gcur, int bw, int bh, DiaCands cands, int ncand, int mnx, int mny, int mxx, int mxy, int cx, int cy,
                                                 int sw, int sh, uint32_t lambda, int pmx, int pmy, uint32_t *out)
{
    extern __shared__ __align__(16) uint16_t smem[];
    __shared__ uint32_t sads[12];
    __shared__ int16_t cand[24];
    const int wave = threadIdx.x >> 6;
    const uint16_t *reg = greg, *cur = gcur;
    if (STAGE) {
        stage_packed(smem, greg, rstride * rrows, gcur, bw * bh);
        reg = smem;
        cur = smem + align8(rstride * rrows);
    }
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < 24; i++) cand[i] = cands.v[i];
    __syncthreads();
    for (int i = wave; i < ncand; i += 4) {
        const int mx = min(max((int)cand[2 * i], mnx), mxx), my = min(max((int)cand[2 * i + 1], mny), mxy);
        const uint32_t s = wave_sad(reg, rstride, rx0, ry0, cur, bw, bh, mx, my);
        if ((threadIdx.x & 63) == 0) sads[i] = s;
    }
    __syncthreads();
    uint32_t best = 0xFFFFFFFFu, bestSad = 0xFFFFFFFFu;
    int bx = 0, by = 0;
    for (int i = 0; i < ncand; i++) {
        const int mx = min(max((int)cand[2 * i], mnx), mxx), my = min(max((int)cand[2 * i + 1], mny), mxy);
        const uint32_t c = (sads[i] << 8) + (eg_bits(4 * mx - pmx) + eg_bits(4 * my - pmy)) * lambda;
        if (c < best) { best = c; bestSad = sads[i]; bx = mx; by = my; }
    }
    const int dxs[4] = {-1, 1, 0, 0}, dys[4] = {0, 0, -1, 1};
    for (int it = 0; it < sw + sh; it++) {
        bool ok[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int mx = bx + dxs[k], my = by + dys[k];
            ok[k] = mx >= mnx && mx <= mxx && my >= mny && my <= mxy && mx >= cx - sw && mx <= cx + sw &&
                    my >= cy - sh && my <= cy + sh;
        }
        const int ox = wave == 0 ? -1 : wave == 1 ? 1 : 0, oy = wave == 2 ? -1 : wave == 3 ? 1 : 0;
        const bool mine = wave == 0 ? ok[0] : wave == 1 ? ok[1] : wave == 2 ? ok[2] : ok[3];
        __syncthreads();                             // the previous step's readers of sads are done
        if (mine) {
            const uint32_t s = wave_sad(reg, rstride, rx0, ry0, cur, bw, bh, bx + ox, by + oy);
            if ((threadIdx.x & 63) == 0) sads[wave] = s;
        }
        __syncthreads();
        int nx = bx, ny = by;
        uint32_t nb = best, ns = bestSad;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (!ok[k]) continue;
            const int mx = bx + dxs[k], my = by + dys[k];
            const uint32_t c = (sads[k] << 8) + (eg_bits(4 * mx - pmx) + eg_bits(4 * my - pmy)) * lambda;
            if (c < nb) { nb = c; ns = sads[k]; nx = mx; ny = my; }
        }
        if (nx == bx && ny == by) break;
        bx = nx; by = ny; best = nb; bestSad = ns;
    }
    if (threadIdx.x == 0) {
        out[0] = (uint32_t)bx;
        out[1] = (uint32_t)by;
        out[2] = best;
        out[3] = bestSad;
    }
}

// Half-pel then quarter-pel ring around (qx, qy) (quarter pel).  reg: luma
// samples whose first row/column is (rx0, ry0) relative to the co-located
// block position (the host stages integer positions -1..+1 plus 8-tap reach).
// A ring's eight positions have three horizontal and three vertical offsets:
// the first pass runs once per horizontal offset into LDS (strips of up to
// `strip` rows), and each thread forms the eight second passes of its samples
// from there.  STAGE: region and block are read once into LDS (they may be
// mapped host memory).  LDS: 3 (strip + 9) bw first-pass values, then those.
template <bool STAGE>
__global__ void __launch_bounds__(256) k_subpel_one(const uint16_t *greg, int rstride, int rrows, int rx0, int ry0,
                                                    const uint16_t *gcur, int bw, int bh, int strip, int qx, int qy,
                                                    uint32_t bestCost, int pmx, int pmy, uint32_t lambda,
                                                    uint32_t *out)
{
    extern __shared__ __align__(16) uint16_t smem[];
    __shared__ uint32_t part[4][8];
    int16_t *mid = reinterpret_cast<int16_t *>(smem);
    const int mrows = strip + 9;
    const uint16_t *reg = greg, *cur = gcur;
    if (STAGE) {
        uint16_t *s = smem + align8(3 * mrows * bw);
        stage_packed(s, greg, rstride * rrows, gcur, bw * bh);
        reg = s;
        cur = s + align8(rstride * rrows);
    }
    __syncthreads();
    constexpr int ring_x[8] = {-1, 1, 0, 0, -1, 1, -1, 1}, ring_y[8] = {0, 0, -1, 1, -1, -1, 1, 1};
    int mx = qx, my = qy;
    uint32_t best = bestCost;
    for (int pass = 0; pass < 2; pass++) {
        const int step = pass == 0 ? 2 : 1, cx = mx, cy = my;
        // window row of the first tap of the ring's top row, and each vertical offset's rows below it
        const int top = ((4 * (cy - step)) >> 4) - 3 - ry0;
        int dyr[3];
        const int8_t *cv[3];
#pragma unroll
        for (int v = 0; v < 3; v++) {
            const int y16 = 4 * (cy + (v - 1) * step);
            dyr[v] = (y16 >> 4) - 3 - ry0 - top;
            cv[v] = c_luma[0][y16 & 15];
        }
        uint32_t e[8] = {};
        for (int y0 = 0; y0 < bh; y0 += strip) {
            const int rows = min(strip, bh - y0), need = rows + 7 + dyr[2];
            __syncthreads();                         // the previous strip's readers are done
            for (int i = threadIdx.x; i < 3 * need * bw; i += 256) {
                const int hr = i / bw, c = i - hr * bw, u = hr / need, r = hr - u * need;
                const int x16 = 4 * (cx + (u - 1) * step);
                mid[(u * mrows + r) * bw + c] =
                    (int16_t)hpass<8>(reg + (top + y0 + r) * rstride + (x16 >> 4) - 3 - rx0 + c, c_luma[0][x16 & 15]);
            }
            __syncthreads();
            for (int i = threadIdx.x; i < rows * bw; i += 256) {
                const int r = i / bw, c = i - r * bw;
                const int s = (int)cur[(y0 + r) * bw + c];
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const int u = ring_x[k] + 1, v = ring_y[k] + 1;
                    const int16_t *m = mid + (u * mrows + r + dyr[v]) * bw + c;
                    int acc = 0;
#pragma unroll
                    for (int j = 0; j < 8; j++) acc += (int)cv[v][j] * (int)m[j * bw];
                    e[k] += (uint32_t)abs(s - vfinal_pix(acc));
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t t = (uint32_t)group_sum<64>((int)e[k]);
            if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][k] = t;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int tx = cx + ring_x[k] * step, ty = cy + ring_y[k] * step;
            const uint32_t sad = part[0][k] + part[1][k] + part[2][k] + part[3][k];
            const uint32_t cost = (sad << 8) + (eg_bits(tx - pmx) + eg_bits(ty - pmy)) * lambda;
            if (cost < best) { best = cost; mx = tx; my = ty; }
        }
        __syncthreads();                             // the readers of part are done
    }
    if (threadIdx.x == 0) {
        out[0] = (uint32_t)mx;
        out[1] = (uint32_t)my;
        out[2] = best;
    }
}

// The bounded form of the block search from range 16 on, where it can take 3,000
// blocks (bound_block; the others, whatever their number, take as long either way).
// With all its launches (predictors, search, refinement), several calls in flight:
// 1280x720 (8,300 blocks) range 16: 166 -> 114 us, range 24: 281 -> 159, range 12:
// no gain; 960x540 (4,600) range 16: 115 -> 83; 640x360 (2,100) range 16: no gain,
// and 416x240 (900) 43 -> 53.  The search alone at range 16, exhaustive then this
// form: 3,000 blocks of 8x8 36 -> 20 us, of 16x16 62 -> 39, with 1,000 of 64x64
// 263 -> 252; 8,000 of 32x32 stay exhaustive.  With noise of sigma 64, or flat with
// noise, 3,000 blocks of up to 16x16 take 0.64 to 1.06 of the time (of 16x32 up to
// 1.17, flat), 2,000 up to 1.17 of it and 1,000 up to 1.45: the line.
constexpr int kBlkMinRange = 16, kBlkMinBlocks = 3000;
static bool bound_blocks_rule(int n, int range, uint32_t lambda)
{
    return n >= kBlkMinBlocks && range >= kBlkMinRange && lambda <= kSeaLambda;
}

// Dynamic LDS of the per-call searches.
constexpr size_t kCallLds = 60 * 1024;         // of samples (two 16-byte round-ups more at most)

static inline int clampi_h(int v, int lo, int hi) { return std::min(std::max(v, lo), hi); }

// Integer search of one block (its workgroup): the window +/-range around the
// rounded predictor, clipped to the CU MV window, staged in LDS with the block
// (packed core; ws: window row pitch for the widest block).  Every thread
// returns the winner as the block's base MV (1/16 pel) in B.mvx / B.mvy.
__device__ __forceinline__ void search_block(const xg_picture *pics, xg_block &B, int range, uint32_t lambda, int ctu,
                                             int ws)
{
    extern __shared__ uint32_t smem32[];
    __shared__ unsigned long long red[16];
    const xg_picture &P = pics[B.pic], &R = pics[B.ref];
    const int fw = P.plane[0].width, fh = P.plane[0].height;
    const int mnx = (int16_t)(-B.x - ctu - 8), mny = (int16_t)(-B.y - ctu - 8);
    const int mxx = (int16_t)(fw + (ctu - B.w + 8) - B.x), mxy = (int16_t)(fh + (ctu - B.h + 8) - B.y);
    // predictor: 1/16 pel -> quarter pel (>> 2) -> integer rounded as Xin266FillMeCand does
    // ((v + 2) >> 2, h266_analyze_inter_cu.c:271-272), kept inside the MV window
    const int cx = min(max(((B.mvpx >> 2) + 2) >> 2, mnx), mxx), cy = min(max(((B.mvpy >> 2) + 2) >> 2, mny), mxy);
    const int x0 = max(cx - range, mnx), x1 = min(cx + range, mxx);
    const int y0 = max(cy - range, mny), y1 = min(cy + range, mxy);
    const int nx = x1 - x0 + 1, ny = y1 - y0 + 1, rows = ny + B.h - 1;
    uint16_t *win = reinterpret_cast<uint16_t *>(smem32);
    uint32_t *curL = smem32 + (((rows * (ws >> 1)) + 3) & ~3);    // 16-byte aligned
    const intptr_t rs = R.plane[0].stride, cs = P.plane[0].stride;
    stage_rows(win, ws, R.plane[0].data + (intptr_t)(B.y + y0) * rs + (B.x + x0), rs, rows, nx + B.w - 1);
    stage_cur(curL, P.plane[0].data + (intptr_t)B.y * cs + B.x, cs, B.w, B.h);
    __syncthreads();
    const int pmx = B.mvpx >> 2, pmy = B.mvpy >> 2;
    unsigned long long k;
    switch (B.w) {
    case 4: k = packed_items<4>(smem32, ws, curL, B.h, x0, x1, y0, nx, ny, lambda, pmx, pmy); break;
    case 8: k = packed_items<8>(smem32, ws, curL, B.h, x0, x1, y0, nx, ny, lambda, pmx, pmy); break;
    case 16: k = packed_items<16>(smem32, ws, curL, B.h, x0, x1, y0, nx, ny, lambda, pmx, pmy); break;
    case 32: k = packed_items<32>(smem32, ws, curL, B.h, x0, x1, y0, nx, ny, lambda, pmx, pmy); break;
    default: k = packed_items<64>(smem32, ws, curL, B.h, x0, x1, y0, nx, ny, lambda, pmx, pmy); break;
    }
    k = block_min_u64_16(k, red);
    const int i = (int)(uint32_t)k;
    B.mvx = 16 * (x0 + i % nx);
    B.mvy = 16 * (y0 + i / nx);
}

// Session blocks that k_search_blocks_bound takes: the others' windows would leave
// its two waves too few to a CU.  From range 16 on (bound_blocks_rule) no block 64
// wide is among them, and 32-wide ones up to a height of 16.
__host__ __device__ __forceinline__ bool bound_block(int w, int h, int range)
{
    return (w + 2 * range) * (h + 2 * range) <= (16 + 2 * range) * (32 + 2 * range);
}

// Integer search of every session block around its predictor; the result is
// written back as the block's base MV.
__global__ void __launch_bounds__(1024) k_search_blocks(const xg_picture *pics, xg_block *blocks, int range,
                                                        uint32_t lambda, int ctu, int ws)
{
    const int b = blockIdx.x;
    xg_block B = blocks[b];
    search_block(pics, B, range, lambda, ctu, ws);
    if (threadIdx.x == 0) {
        blocks[b].mvx = B.mvx;
        blocks[b].mvy = B.mvy;
    }
}

// The same for the blocks that the bounded form leaves, in one launch whatever
// their number: workgroup k takes the k-th.  Their counts by runs of `per` session
// blocks travel with the arguments, and a workgroup looks its block up in its run.
// (A launch per 480 listed blocks waits for the last of each: 4,100 blocks of 16x16 and
// 2,000 of 64x64 at range 16 took 439 us, and take 383; exhaustively 431.)
constexpr int kRestRuns = 480;
struct RestRuns {
    int n, per;                                  // session blocks, of a run
    int before[kRestRuns];                       // blocks left before the run
};

// Session block of the k-th block left, in every lane; -1 where there is none.
__device__ __forceinline__ int rest_block(const RestRuns &l, const xg_block *blocks, int range, int k)
{
    int run = 0;
#pragma unroll 1
    for (int step = 256; step; step >>= 1)       // the last run with no more than k before it
        if (run + step < kRestRuns && l.before[run + step] <= k) run += step;
    int at = k - l.before[run];
    const int end = min(l.n, (run + 1) * l.per);
    for (int b0 = run * l.per; b0 < end; b0 += 64) {
        const int b = b0 + (int)(threadIdx.x & 63);
        const bool left = b < end && !bound_block(blocks[b].w, blocks[b].h, range);
        const unsigned long long m = __ballot(left);
        const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        const unsigned long long hit = __ballot(left && rank == at);
        if (hit) return b0 + (int)__builtin_ctzll(hit);
        at -= (int)__popcll(m);
    }
    return -1;
}

__global__ void __launch_bounds__(1024) k_search_blocks_rest(const xg_picture *pics, xg_block *blocks, int range,
                                                             uint32_t lambda, int ctu, int ws, RestRuns runs)
{
    const int b = rest_block(runs, blocks, range, (int)blockIdx.x);
    if (b < 0) return;
    xg_block B = blocks[b];
    search_block(pics, B, range, lambda, ctu, ws);
    if (threadIdx.x == 0) {
        blocks[b].mvx = B.mvx;
        blocks[b].mvy = B.mvy;
    }
}

// ---------------------------------------------------------------------------
// Session blocks by bounds (xg_sea.hpp), a workgroup of two waves a block
//
// The window, staged so that candidate (0, 0) is column 0 of row 0, and the sums
// of 4x4 samples at each of its positions, lie in LDS.  (1) Each lane takes the
// lowest bound of its share of the candidates, and the 128 of them are costed, a
// lane each: their lowest cost limits the rest.  (2) Every candidate whose
// bound is within the limit goes to its wave's list, which is costed 64 at a
// time, a lane each, and may lower the wave's limit.  A lane that costs a whole candidate needs no
// reduction.  Where over 48 of the 128 lanes' first candidates lie within the limit
// (flat or noisy content) no list is made and every candidate is costed, four a lane
// at once, which takes 0.44 of a listed candidate's instructions.  Up to three
// waves' worth of candidates are costed without bounds.
//
// 1280x720, 8,300 blocks, range 16: 124 us exhaustively; 68 us here, 21 M vector
// instructions (35 us to issue) at 3 waves a SIMD, which is what 13 KB of window
// and sums a block leave, and 20 us for the 2 % it leaves.  Two waves a
// block: one took 87 us.  32,400 blocks of 16x16 at range 16, exhaustively and here:
// texture 623 and 302 us, noise of sigma 64 625 and 440, flat with noise 624 and 475
// (1,068 by lists); 4,000 of 16x32 at range 32 flat 393 and 442, the worst measured.
// ---------------------------------------------------------------------------
constexpr int kBlkDirect = 192;                  // candidates costed without bounds at most
constexpr int kBlkWaves = 2, kBlkWg = 64 * kBlkWaves;
constexpr int kBlkDense = 48;                    // of the 128 lanes' first candidates within the limit, past which every one is costed
constexpr int kBlkList = 192;                    // of a wave: under 64 when a step adds up to 128

struct BlkLds {
    int wp, sums, cur, csum, rates, list, bytes; // window pitch; dword offsets; all in bytes
};
__host__ __device__ __forceinline__ BlkLds blk_lds(int w, int h, int range)
{
    const int n = 2 * range + 1, rows = n + h;   // a row more than the candidates reach
    BlkLds l;
    l.wp = ((n + w) / 2 + 2) | 1;
    l.sums = rows * l.wp;
    l.cur = 2 * l.sums;
    l.csum = l.cur + w * h / 2;
    l.rates = l.csum + (h / 4) * (w < 8 ? 1 : w / 8);
    l.list = l.rates + 2 * (n + 2);
    l.bytes = 4 * l.list + 2 * kBlkList * kBlkWaves;
    return l;
}

// SAD of the candidate at (cx, cy) of the window, by one lane.
template <int W>
__device__ __forceinline__ uint32_t lane_sad(const uint32_t *win, int wp, const uint32_t *cur, int h, int cx, int cy)
{
    constexpr int CH = W < 16 ? W / 2 : 8;       // dwords of a row at once
    const uint32_t sh = (uint32_t)(cx & 1) << 4;
    uint32_t e = 0;
    const uint32_t *w = win + cy * wp + (cx >> 1);
#pragma unroll 1
    for (int i = 0; i < h; i++, w += wp, cur += W / 2)
#pragma unroll
        for (int k = 0; k < W / 2; k += CH) {
            uint32_t D[CH + 1];
#pragma unroll
            for (int j = 0; j <= CH; j++) D[j] = w[k + j];
#pragma unroll
            for (int j = 0; j < CH; j++) e = sad2(align16(D[j + 1], D[j], sh), cur[k + j], e);
        }
    return e;
}

// SADs of the four candidates from column 4 q of window row cy, by one lane.
template <int W>
__device__ __forceinline__ void lane_sad4(const uint32_t *win, int wp, const uint32_t *cur, int h, int q, int cy,
                                          uint32_t (&e)[4])
{
    constexpr int CH = W < 16 ? W / 2 : 8;
    const uint32_t *w = win + cy * wp + 2 * q;
    e[0] = e[1] = e[2] = e[3] = 0;
#pragma unroll 1
    for (int i = 0; i < h; i++, w += wp, cur += W / 2)
#pragma unroll
        for (int k = 0; k < W / 2; k += CH) {
            uint32_t D[CH + 2], F[CH + 1];
#pragma unroll
            for (int j = 0; j < CH + 2; j++) D[j] = w[k + j];
#pragma unroll
            for (int j = 0; j < CH + 1; j++) F[j] = align16(D[j + 1], D[j], 16);
#pragma unroll
            for (int j = 0; j < CH; j++) {
                const uint32_t c = cur[k + j];
                e[0] = sad2(D[j], c, e[0]);
                e[1] = sad2(F[j], c, e[1]);
                e[2] = sad2(D[j + 1], c, e[2]);
                e[3] = sad2(F[j + 1], c, e[3]);
            }
        }
}

// Bounds of candidates 2 j and 2 j + 1 of a row (q: their dword of the sums) of a
// block W wide with hs rows of sub-blocks, added to l and h.  C: the block's sums,
// a packed pair of adjacent sub-blocks a dword (W = 4: one in the lower half).
template <int W>
__device__ __forceinline__ void lane_bounds(const uint32_t *q, int pitch, const uint32_t *C, int hs, uint32_t &l, uint32_t &h)
{
#pragma unroll 1
    for (int i = 0; i < hs; i++, q += 4 * pitch) {
        if constexpr (W == 4) {
            const uint32_t u = q[0], c = C[i];
            l = sad2(u & 0xFFFFu, c, l);
            h = sad2(u >> 16, c, h);
        } else {
#pragma unroll
            for (int k = 0; k < W / 8; k++) {
                const uint32_t u = q[4 * k], v = q[4 * k + 2], c = C[i * (W / 8) + k];
                l = sad2(__builtin_amdgcn_perm(v, u, 0x05040100u), c, l);
                h = sad2(__builtin_amdgcn_perm(v, u, 0x07060302u), c, h);
            }
        }
    }
}

struct BlkWin {
    int x0, y0, nx, ny, pmx, pmy, h;
    uint32_t lambda;
};

template <int W>
__device__ __forceinline__ unsigned long long bound_search(uint32_t *lds, const BlkLds &o, const BlkWin &v, uint32_t *limits)
{
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));               // nothing computed ahead for the other widths: registers
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wp = o.wp, nx = v.nx, ny = v.ny, hs = v.h / 4;
    const uint32_t *win = lds, *S = lds + o.sums, *cur = lds + o.cur, *C = lds + o.csum, *bxq = lds + o.rates + 1,
                   *byq = bxq + nx + 1;
    uint16_t *list = reinterpret_cast<uint16_t *>(lds + o.list) + wave * kBlkList;
    unsigned long long best = ~0ull;             // the lane's lowest (cost, position)
    auto cost = [&](int pos) {
        const int cx = pos & 255, cy = pos >> 8;
        const uint32_t e = lane_sad<W>(win, wp, cur, v.h, cx, cy);
        const uint32_t k = (e << 8) + (eg_bits(4 * (v.x0 + cx) - v.pmx) + eg_bits(4 * (v.y0 + cy) - v.pmy)) * v.lambda;
        const unsigned long long q = ((unsigned long long)k << 32) | (uint32_t)pos;
        best = q < best ? q : best;
    };
    if (nx * ny <= kBlkDirect) {
        const uint32_t rcp = (65536u + (uint32_t)nx - 1) / (uint32_t)nx;
        for (int i = tid; i < nx * ny; i += kBlkWg) {
            const int cy = (int)(((uint32_t)i * rcp) >> 16);
            cost(cy << 8 | (i - cy * nx));
        }
    } else {
        const int nc = (nx + 1) >> 1, items = ny * nc;
        const uint32_t rcp = (65536u + (uint32_t)nc - 1) / (uint32_t)nc;
        const int dr = (int)(((uint32_t)kBlkWg * rcp) >> 16), dj = kBlkWg - dr * nc;
        const int r0 = (int)(((uint32_t)tid * rcp) >> 16), j0 = tid - r0 * nc;
        uint32_t key = 0xFFFFFFFFu, first = kSeaOver;    // first: the bound of the lane's first candidate
        int kpos = 0;
        for (int i = tid, s = 0, r = r0, j = j0; i < items; i += kBlkWg, s++) {
            uint32_t l = byq[r] + bxq[2 * j], h = byq[r] + bxq[2 * j + 1];
            lane_bounds<W>(S + r * wp + j, wp, C, hs, l, h);
            const uint32_t k = min(l, h);
            first = s ? first : l;
            kpos = k < key ? r << 8 | (2 * j + (h < l)) : kpos;
            key = min(key, k);
            r += dr;
            j += dj;
            if (j >= nc) {
                j -= nc;
                r++;
            }
        }
        cost(kpos);                              // lanes without an item cost candidate 0
        uint32_t limit = wave_min((uint32_t)(best >> 32)) >> 8;
        const int within = (int)__popcll(__ballot(first <= limit));
        if (lane == 0) {
            limits[wave] = limit;
            limits[kBlkWaves + wave] = (uint32_t)within;
        }
        __syncthreads();
        limit = min(limits[0], limits[1]);
        const bool dense = (int)uniform((int)(limits[kBlkWaves] + limits[kBlkWaves + 1])) > kBlkDense;
        int n = 0;
        auto flush = [&]() {                     // cost the first 64 of the list, keep the others
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const int rest = n - 64;
            const uint16_t a = list[64 + lane], b = list[128 + lane];
            if (lane < n) cost(list[lane]);
            limit = min(limit, wave_min((uint32_t)(best >> 32)) >> 8);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (lane < rest) list[lane] = a;
            if (lane + 64 < rest) list[64 + lane] = b;
            n = max(rest, 0);
        };
        for (int i0 = 64 * wave, r = r0, j = j0; i0 < items && !dense; i0 += kBlkWg) {
            const bool in = i0 + lane < items;
            uint32_t l = kSeaOver, h = kSeaOver;
            if (in) {
                l = byq[r] + bxq[2 * j];
                h = byq[r] + bxq[2 * j + 1];
                lane_bounds<W>(S + r * wp + j, wp, C, hs, l, h);
            }
            auto push = [&](uint32_t q, int pos) {
                const bool ok = q <= limit;
                const unsigned long long m = __ballot(ok);
                const int at = n + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                if (ok) list[at] = (uint16_t)pos;
                n += __popcll(m);
            };
            push(l, r << 8 | 2 * j);
            push(h, r << 8 | (2 * j + 1));
            while (n >= 64) flush();
            r += dr;
            j += dj;
            if (j >= nc) {
                j -= nc;
                r++;
            }
        }
        if (dense) {
            const int nq = (nx + 3) >> 2;
            uint32_t bc = 0xFFFFFFFFu;
            int bp = 0;                          // a lane's candidates come in raster order: strict < keeps the earliest
            for (int i = tid; i < ny * nq; i += kBlkWg) {
                const int cy = i / nq, q = i - cy * nq;
                uint32_t e[4];
                lane_sad4<W>(win, wp, cur, v.h, q, cy, e);
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const int cx = 4 * q + m;
                    const uint32_t k = (e[m] << 8) + (eg_bits(4 * (v.x0 + cx) - v.pmx) + eg_bits(4 * (v.y0 + cy) - v.pmy)) * v.lambda;
                    if (cx < nx && k < bc) {
                        bc = k;
                        bp = cy << 8 | cx;
                    }
                }
            }
            const unsigned long long q = ((unsigned long long)bc << 32) | (uint32_t)bp;
            best = q < best ? q : best;
        } else if (n) {
            flush();
        }
    }
    const uint32_t lo = wave_min((uint32_t)(best >> 32));
    const uint32_t pos = wave_min((uint32_t)(best >> 32) == lo ? (uint32_t)best : 0xFFFFFFFFu);
    return ((unsigned long long)lo << 32) | pos;
}

__global__ void __launch_bounds__(kBlkWg) __attribute__((amdgpu_waves_per_eu(6))) k_search_blocks_bound(const xg_picture *pics, xg_block *blocks, int range,
                                                            uint32_t lambda, int ctu)
{
    extern __shared__ uint32_t smem32[];
    __shared__ uint32_t limits[2 * kBlkWaves];   // of the waves: limit, first candidates within it
    __shared__ unsigned long long found[kBlkWaves];
    const int tid = threadIdx.x;
    const xg_block &B = blocks[blockIdx.x];
    const int bw = B.w, bh = B.h;
    if (!bound_block(bw, bh, range)) return;
    const xg_picture &P = pics[B.pic], &Rf = pics[B.ref];
    const int fw = P.plane[0].width, fh = P.plane[0].height;
    const int mnx = (int16_t)(-B.x - ctu - 8), mny = (int16_t)(-B.y - ctu - 8);
    const int mxx = (int16_t)(fw + (ctu - bw + 8) - B.x), mxy = (int16_t)(fh + (ctu - bh + 8) - B.y);
    const int cx = min(max(((B.mvpx >> 2) + 2) >> 2, mnx), mxx), cy = min(max(((B.mvpy >> 2) + 2) >> 2, mny), mxy);
    BlkWin v;
    v.x0 = max(cx - range, mnx);
    v.y0 = max(cy - range, mny);
    v.nx = min(cx + range, mxx) - v.x0 + 1;
    v.ny = min(cy + range, mxy) - v.y0 + 1;
    v.pmx = B.mvpx >> 2;
    v.pmy = B.mvpy >> 2;
    v.h = bh;
    v.lambda = lambda;
    const BlkLds o = blk_lds(bw, bh, range);
    const int rows = v.ny + bh - 1, wd = (v.nx + bw) >> 1, wp = o.wp;     // the window: rows of wd dwords
    // window and current block (its rows are dword aligned)
    {
        const int lg = wd <= 16 ? 4 : 5, c = tid & ((1 << lg) - 1), r0 = tid >> lg, step = kBlkWg >> lg;
        const intptr_t rs = Rf.plane[0].stride;
        const uint16_t *g = Rf.plane[0].data + (intptr_t)(B.y + v.y0 + r0) * rs + B.x + v.x0;
        for (int cc = c; cc < wd; cc += 1 << lg) {
            const uint16_t *p = g + 2 * cc;
            uint32_t *d = smem32 + r0 * wp + cc;
            for (int r = r0; r < rows; r += 4 * step) {
                uint32_t w[4];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (r + k * step < rows) w[k] = load_pair(p + (intptr_t)(k * step) * rs);
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (r + k * step < rows) d[k * step * wp] = w[k];
                p += (intptr_t)(4 * step) * rs;
                d += 4 * step * wp;
            }
        }
        const int lw = 30 - __builtin_clz((unsigned)bw);                  // dwords of a block row, log2
        const intptr_t cs = P.plane[0].stride;
        const uint16_t *q = P.plane[0].data + (intptr_t)B.y * cs + B.x;
        for (int i = tid; i < bh << lw; i += kBlkWg)
            smem32[o.cur + i] = *(const gdword *)(q + (intptr_t)(i >> lw) * cs + 2 * (i & ((1 << lw) - 1)));
    }
    // shares of the rate: columns -1 .. nx (over any limit outside), then rows
    uint32_t *rates = smem32 + o.rates;
    for (int i = tid; i < v.nx + 2 + v.ny; i += kBlkWg) {
        const int k = i - 1, m = k <= v.nx ? 4 * (v.x0 + k) - v.pmx : 4 * (v.y0 + i - v.nx - 2) - v.pmy;
        rates[i] = i == 0 || k == v.nx ? kSeaOver : (eg_bits(m) * lambda) >> 8;
    }
    __syncthreads();
    if (v.nx * v.ny > kBlkDirect) {
        // sums of 4x4 samples: a column pair and a run of rows a lane, sliding
        const uint32_t *win = smem32;
        uint32_t *S = smem32 + o.sums;
        const int nj = (v.nx + bw - 2) >> 1, ns = rows - 3;               // column pairs that hold a candidate's sum
        const int runs = max(1, (int)((uint32_t)kBlkWg / (uint32_t)nj)), len = (ns + runs - 1) / runs;
        for (int i = tid; i < runs * nj; i += kBlkWg) {
            const int run = i / nj, j = i - run * nj, y0 = run * len, y1 = min(ns, y0 + len);
            auto hsum = [&](int r) {
                const uint32_t *w = win + r * wp + j;
                const uint32_t a = w[0], b = w[1], c = w[2];
                return as_v2s(a) + as_v2s(align16(b, a, 16)) + as_v2s(b) + as_v2s(align16(c, b, 16));
            };
            if (y0 < y1) {
                v2s h0 = hsum(y0), h1 = hsum(y0 + 1), h2 = hsum(y0 + 2);
                for (int r = y0; r < y1; r++) {
                    const v2s h3 = hsum(r + 3);
                    S[r * wp + j] = as_u32(h0 + h1 + h2 + h3);
                    h0 = h1;
                    h1 = h2;
                    h2 = h3;
                }
            }
        }
        // the block's own sums
        const int lp = bw < 8 ? 0 : 28 - __builtin_clz((unsigned)bw);     // pairs of sub-blocks a row, log2
        for (int i = tid; i < (bh / 4) << lp; i += kBlkWg) {
            const uint32_t *q = smem32 + o.cur + 4 * (i >> lp) * (bw / 2) + 4 * (i & ((1 << lp) - 1));
            uint32_t a = 0, b = 0;
#pragma unroll
            for (int r = 0; r < 4; r++, q += bw / 2) {
                a = sad2(q[0], 0, sad2(q[1], 0, a));
                if (bw >= 8) b = sad2(q[2], 0, sad2(q[3], 0, b));
            }
            smem32[o.csum + i] = a | b << 16;
        }
        __syncthreads();
    }
    unsigned long long k;
    switch (bw) {
    case 4: k = bound_search<4>(smem32, o, v, limits); break;
    case 8: k = bound_search<8>(smem32, o, v, limits); break;
    case 16: k = bound_search<16>(smem32, o, v, limits); break;
    default: k = bound_search<32>(smem32, o, v, limits); break;      // bound_block: no wider
    }
    if ((tid & 63) == 0) found[tid >> 6] = k;
    __syncthreads();
    if (tid == 0) {
        k = min(found[0], found[1]);
        blocks[blockIdx.x].mvx = 16 * (v.x0 + (int)((uint32_t)k & 255));
        blocks[blockIdx.x].mvy = 16 * (v.y0 + (int)((uint32_t)k >> 8));
    }
}

}  // namespace xg

using namespace xg;

extern "C" {

void Xg26xMotionEstFull(xg_me_struct *me)
{
    if (!me || !me->input || !me->ref || me->width == 0 || me->height == 0 || me->width > 128 || me->height > 128) {
        set_error(XG_ERR_ARG, "Xg26xMotionEstFull: bad arguments");
        return;
    }
    const int bw = (int)me->width, bh = (int)me->height;
    const int cx = (me->predMv.mvX + 2) >> 2, cy = (me->predMv.mvY + 2) >> 2;
    const int x0 = std::max(cx - me->searchWidth, (int)me->minMv.mvX), x1 = std::min(cx + me->searchWidth, (int)me->maxMv.mvX);
    const int y0 = std::max(cy - me->searchHeight, (int)me->minMv.mvY), y1 = std::min(cy + me->searchHeight, (int)me->maxMv.mvY);
    if (x1 < x0 || y1 < y0) {
        set_error(XG_ERR_ARG, "Xg26xMotionEstFull: empty search window");
        return;
    }
    const int ws = x1 - x0 + bw, wh = y1 - y0 + bh;
    if (((size_t)ws * wh + (size_t)bw * bh) * 2 > kCallLds) {
        set_error(XG_ERR_ARG, "Xg26xMotionEstFull: window %dx%d exceeds the LDS budget", ws, wh);
        return;
    }
    const size_t lds = ((size_t)align8(ws * wh) + (size_t)align8(bw * bh)) * 2;
    const size_t wB = align_up((size_t)ws * wh * 2, 256), cB = align_up((size_t)bw * bh * 2, 256);
    CallCtx *c = call_ctx(0, wB + cB + 256);
    if (!c) return;
    pack2d(c->host, me->ref + (intptr_t)y0 * me->refStride + x0, me->refStride, ws, wh, 2);
    pack2d(c->host + wB, me->input, me->inputStride, bw, bh, 2);
    auto *kernel = bw % 4 == 0 ? &k_full_search_one<4> : &k_full_search_one<1>;
    kernel<<<1, 256, lds, c->stream>>>((uint16_t *)c->view, ws, wh, (uint16_t *)(c->view + wB), bw, bh, x0, x1, y0, y1,
                                       me->sadLambda, me->predMv.mvX, me->predMv.mvY,
                                       (uint32_t *)(c->view + wB + cB));
    if (!XG_HIP(hipGetLastError())) return;
    uint32_t *hout = (uint32_t *)(c->host + wB + cB);
    if (!XG_HIP(hipStreamSynchronize(c->stream))) return;
    me->bestMv.mvX = (int16_t)(4 * (int)hout[0]);
    me->bestMv.mvY = (int16_t)(4 * (int)hout[1]);
    me->bestCost = hout[2];
    me->bestSad = hout[3];
}

void Xg26xMotionEstDia(xg_me_struct *me)
{
    if (!me || !me->input || !me->ref || me->width == 0 || me->height == 0 || me->width > 128 ||
        me->height > 128 || me->candNum == 0 || me->candNum > 12) {
        set_error(XG_ERR_ARG, "Xg26xMotionEstDia: bad arguments");
        return;
    }
    const int bw = (int)me->width, bh = (int)me->height;
    const int cx = (me->predMv.mvX + 2) >> 2, cy = (me->predMv.mvY + 2) >> 2;
    const int mnx = me->minMv.mvX, mny = me->minMv.mvY, mxx = me->maxMv.mvX, mxy = me->maxMv.mvY;
    // bounding box of every position the search may read
    int x0 = std::max(cx - me->searchWidth, mnx), x1 = std::min(cx + me->searchWidth, mxx);
    int y0 = std::max(cy - me->searchHeight, mny), y1 = std::min(cy + me->searchHeight, mxy);
    DiaCands cands = {};
    int16_t *cand = cands.v;
    for (uint32_t i = 0; i < me->candNum; i++) {
        const int mx = clampi_h(me->meCand[i].mvX, mnx, mxx), my = clampi_h(me->meCand[i].mvY, mny, mxy);
        cand[2 * i] = me->meCand[i].mvX;
        cand[2 * i + 1] = me->meCand[i].mvY;
        x0 = std::min(x0, mx); x1 = std::max(x1, mx);
        y0 = std::min(y0, my); y1 = std::max(y1, my);
        // a descent step can leave the window only from a candidate inside it
    }
    const int rw = x1 - x0 + bw, rh = y1 - y0 + bh;
    const size_t rB = align_up((size_t)rw * rh * 2, 256), cB = align_up((size_t)bw * bh * 2, 256);
    // what fits is read once into LDS from the mapped staging; a wider region is copied to HBM first
    const size_t lds = ((size_t)align8(rw * rh) + (size_t)align8(bw * bh)) * 2;
    const bool staged = lds <= kCallLds;
    CallCtx *c = call_ctx(staged ? 0 : rB + cB + 512, rB + cB + 512);
    if (!c) return;
    pack2d(c->host, me->ref + (intptr_t)y0 * me->refStride + x0, me->refStride, rw, rh, 2);
    pack2d(c->host + rB, me->input, me->inputStride, bw, bh, 2);
    if (!staged && !XG_HIP(hipMemcpyAsync(c->dev, c->host, rB + cB, hipMemcpyHostToDevice, c->stream))) return;
    char *d = staged ? c->view : c->dev;
    auto *kernel = staged ? &k_dia_one<true> : &k_dia_one<false>;
    kernel<<<1, 256, staged ? lds : 0, c->stream>>>((uint16_t *)d, rw, rh, x0, y0, (uint16_t *)(d + rB), bw, bh,
                                                    cands, (int)me->candNum, mnx, mny, mxx, mxy, cx,
                                                    cy, me->searchWidth, me->searchHeight, me->sadLambda,
                                                    me->predMv.mvX, me->predMv.mvY, (uint32_t *)(c->view + rB + cB + 256));
    if (!XG_HIP(hipGetLastError())) return;
    uint32_t *hout = (uint32_t *)(c->host + rB + cB + 256);
    if (!XG_HIP(hipStreamSynchronize(c->stream))) return;
    me->bestMv.mvX = (int16_t)(4 * (int)hout[0]);
    me->bestMv.mvY = (int16_t)(4 * (int)hout[1]);
    me->bestCost = hout[2];
    me->bestSad = hout[3];
}

void Xg266FullSubPelMe(xg_me_struct *me)
{
    if (!me || !me->input || !me->ref || me->width == 0 || me->height == 0 || me->width > 128 || me->height > 128) {
        set_error(XG_ERR_ARG, "Xg266FullSubPelMe: bad arguments");
        return;
    }
    const int qx = me->bestMv.mvX, qy = me->bestMv.mvY;
    // h266_sub_pel_refine.c:125-128: leave the MV alone when it is out of range
    if ((qx >> 2) < me->minMv.mvX || (qy >> 2) < me->minMv.mvY || (qx >> 2) > me->maxMv.mvX ||
        (qy >> 2) > me->maxMv.mvY)
        return;
    const int bw = (int)me->width, bh = (int)me->height;
    // reads span integer positions (qx>>2)-1 .. (qx>>2)+1 plus the 8-tap reach
    const int rx0 = (qx >> 2) - 1 - 3, ry0 = (qy >> 2) - 1 - 3;
    const int rw = bw + 10, rh = bh + 10;
    const size_t rB = align_up((size_t)rw * rh * 2, 256), cB = align_up((size_t)bw * bh * 2, 256);
    // as above; the first-pass strips take what the samples leave of the LDS (at least 16 rows)
    const size_t row = 3 * (size_t)bw * 2, samples = ((size_t)align8(rw * rh) + (size_t)align8(bw * bh)) * 2;
    const bool staged = samples + row * (std::min(bh, 16) + 9) <= kCallLds;
    const int strip = std::min<int>(bh, (int)((kCallLds - (staged ? samples : 0)) / row) - 9);
    const size_t lds = align_up(row * (strip + 9), 16) + (staged ? samples : 0);
    CallCtx *c = call_ctx(staged ? 0 : rB + cB + 256, rB + cB + 256);
    if (!c) return;
    pack2d(c->host, me->ref + (intptr_t)ry0 * me->refStride + rx0, me->refStride, rw, rh, 2);
    pack2d(c->host + rB, me->input, me->inputStride, bw, bh, 2);
    if (!staged && !XG_HIP(hipMemcpyAsync(c->dev, c->host, rB + cB, hipMemcpyHostToDevice, c->stream))) return;
    char *d = staged ? c->view : c->dev;
    auto *kernel = staged ? &k_subpel_one<true> : &k_subpel_one<false>;
    kernel<<<1, 256, lds, c->stream>>>((uint16_t *)d, rw, rh, rx0, ry0, (uint16_t *)(d + rB), bw, bh, strip, qx, qy,
                                       me->bestCost, me->predMv.mvX, me->predMv.mvY, me->sadLambda,
                                       (uint32_t *)(c->view + rB + cB));
    if (!XG_HIP(hipGetLastError())) return;
    uint32_t *hout = (uint32_t *)(c->host + rB + cB);
    if (!XG_HIP(hipStreamSynchronize(c->stream))) return;
    me->bestMv.mvX = (int16_t)hout[0];
    me->bestMv.mvY = (int16_t)hout[1];
    me->bestCost = hout[2];
}

int32_t xg_search_blocks(xg_session *s, int32_t range, uint32_t sadLambda, int32_t ctuSize)
{
    SessionView v;
    if (!session_view(s, &v) || range < 0 || range > 32 || ctuSize < 4 || ctuSize > 256) {
        set_error(XG_ERR_ARG, "xg_search_blocks: bad arguments");
        return XG_ERR_ARG;
    }
    if (v.nblocks == 0) return XG_OK;
    int maxw = 0, maxh = 0, rest = 0, restw = 0, resth = 0, boundLds = 0;    // rest: those k_search_blocks_bound leaves
    for (int i = 0; i < v.nblocks; i++) {
        const xg_block &B = v.hBlocks[i];
        if (B.pic >= kSessionPicSlots || B.ref >= kSessionPicSlots || !v.picSet[B.pic] || !v.picSet[B.ref]) {
            set_error(XG_ERR_ARG, "xg_search_blocks: block %d picture slot not set", i);
            return XG_ERR_ARG;
        }
        const xg_picture &P = v.hPics[B.pic], &R = v.hPics[B.ref];
        if (B.x < 0 || B.y < 0 || B.x + B.w > P.plane[0].width || B.y + B.h > P.plane[0].height ||
            R.plane[0].width != P.plane[0].width || R.plane[0].height != P.plane[0].height ||
            R.plane[0].pad < ctuSize + 16) {
            set_error(XG_ERR_ARG, "xg_search_blocks: block %d outside its picture or reference under-padded", i);
            return XG_ERR_ARG;
        }
        // the packed core reads the current block as dword pairs
        if ((B.w & (B.w - 1)) || B.w < 4 || B.w > 64 || B.h < 1 || B.h > 64 || (B.x & 1) || (P.plane[0].stride & 1) ||
            ((uintptr_t)P.plane[0].data & 3)) {
            set_error(XG_ERR_ARG, "xg_search_blocks: block %d: width must be 4..64 (a power of two) at an even x "
                      "in a dword-aligned plane", i);
            return XG_ERR_ARG;
        }
        maxw = std::max(maxw, (int)B.w);
        maxh = std::max(maxh, (int)B.h);
        if (bound_block(B.w, B.h, range)) {
            boundLds = std::max(boundLds, blk_lds(B.w, B.h, range).bytes);
        } else {
            rest++;
            restw = std::max(restw, (int)B.w);
            resth = std::max(resth, (int)B.h);
        }
    }
    const int ws = packed_ws(2 * range + 1, maxw);
    const size_t lds = ((size_t)(2 * range + maxh) * ws + (size_t)maxw * maxh) * 2 + 16;
    if (lds > 64 * 1024) {
        set_error(XG_ERR_ARG, "xg_search_blocks: window exceeds the LDS budget");
        return XG_ERR_ARG;
    }
    const bool bounded = bound_blocks_rule(v.nblocks - rest, range, sadLambda);
    int ev[2];
    const bool timed = session_timer_begin(s, 3, ev);
    const int threads = packed_threads(2 * range + 1);
    if (!bounded) {
        k_search_blocks<<<v.nblocks, threads, lds, v.stream>>>(v.dPics, v.dBlocks, range, sadLambda, ctuSize, ws);
    } else {
        if (rest) {
            const int wsr = packed_ws(2 * range + 1, restw);
            const size_t ldsr = ((size_t)(2 * range + resth) * wsr + (size_t)restw * resth) * 2 + 16;
            RestRuns l;
            l.n = v.nblocks;
            l.per = (v.nblocks + kRestRuns - 1) / kRestRuns;
            int left = 0, b = 0;
            for (int r = 0; r < kRestRuns; r++) {
                l.before[r] = left;
                for (const int e = std::min(v.nblocks, (r + 1) * l.per); b < e; b++)
                    left += !bound_block(v.hBlocks[b].w, v.hBlocks[b].h, range);
            }
            k_search_blocks_rest<<<rest, threads, ldsr, v.stream>>>(v.dPics, v.dBlocks, range, sadLambda, ctuSize, wsr, l);
        }
        k_search_blocks_bound<<<v.nblocks, kBlkWg, (size_t)boundLds, v.stream>>>(v.dPics, v.dBlocks, range, sadLambda, ctuSize);
    }
    if (timed) session_timer_end(s, 3, ev);
    return XG_HIP(hipGetLastError()) ? XG_OK : XG_ERR_HIP;
}

int32_t xg_full_search_frame(xg_session *s, const xg_plane *cur, const xg_plane *ref, int32_t bw, int32_t bh,
                             int32_t range, uint32_t sadLambda, int32_t ctuSize, int16_t *bestMv,
                             uint32_t *bestCost, uint32_t *bestSad)
{
    if (!s) {
        set_error(XG_ERR_ARG, "xg_full_search_frame: bad arguments");
        return XG_ERR_ARG;
    }
    return xg::full_search_frame_on((hipStream_t)xg_session_stream(s), s, cur, ref, bw, bh, range, sadLambda,
                                    ctuSize, bestMv, bestCost, bestSad);
}

}  // extern "C"

int32_t xg::full_search_frame_on(hipStream_t st, xg_session *timer, const xg_plane *cur, const xg_plane *ref,
                                 int32_t bw, int32_t bh, int32_t range, uint32_t sadLambda, int32_t ctuSize,
                                 int16_t *bestMv, uint32_t *bestCost, uint32_t *bestSad)
{
    if (!cur || !ref || !bestMv || !bestCost || !bestSad || bw < 4 || bh < 4 || bw > 64 || bh > 64 ||
        range < 0 || range > 64 || cur->width != ref->width || cur->height != ref->height ||
        ref->pad < range + 4) {
        set_error(XG_ERR_ARG, "xg_full_search_frame: bad arguments");
        return XG_ERR_ARG;
    }
    const int nbx = cur->width / bw, nby = cur->height / bh;
    if (nbx <= 0 || nby <= 0) return XG_OK;
    const size_t lds = ((size_t)(2 * range + bw) * (2 * range + bh) + (size_t)bw * bh) * 2;
    if (lds > 64 * 1024) {
        set_error(XG_ERR_ARG, "xg_full_search_frame: window exceeds the LDS budget");
        return XG_ERR_ARG;
    }
    // packed form: widths 8, 16, 32 with a dword-aligned current plane
    const int nxm = 2 * range + 1, wsP = packed_ws(nxm, bw, kFrameK);
    const size_t ldsP = ((size_t)(2 * range + bh) * wsP + (size_t)bw * bh) * 2 + 16;
    const bool packed = (bw == 8 || bw == 16 || bw == 32) && ((uintptr_t)cur->data & 3) == 0 && (cur->stride & 1) == 0 &&
                        ldsP <= 64 * 1024;
    FsFrameArgs a;
    a.cur = cur->data; a.cs = cur->stride;
    a.ref = ref->data; a.rs = ref->stride;
    a.fw = cur->width; a.fh = cur->height; a.bw = bw; a.bh = bh; a.range = range; a.ctu = ctuSize; a.nbx = nbx;
    a.lambda = sadLambda;
    a.bestMv = bestMv; a.bestCost = bestCost; a.bestSad = bestSad;
    SeaFrameArgs b;
    size_t seaLds = 0;
    sea_frame_lds(bw, range, &b.wp, &b.sp, &b.rows, &seaLds);
    const bool bounded = bw == bh && (bw == 8 || bw == 16) && packed && range >= kSeaMinRange && range <= kSeaMaxRange &&
                         (int64_t)nbx * nby * bw >= kSeaMinWork && seaLds <= 64 * 1024 && sadLambda <= kSeaLambda;
    int ev[2];
    const bool timed = timer && session_timer_begin(timer, 3, ev);
    if (bounded) {
        b.f = a;
        b.ngx = (nbx + 1) / 2;
        b.aligned = (a.rs & 1) == 0;
        // costed four a lane at once, a candidate takes about a third of a listed one's instructions
        b.most = std::min(kSeaList, (2 * range + 1) * (2 * range + 1) / 3);
        const int groups = b.ngx * ((nby + 1) / 2);
        if (bw == 8) k_search_bound<8><<<groups, 256, seaLds, st>>>(b);
        else k_search_bound<16><<<groups, 256, seaLds, st>>>(b);
    } else if (packed) {
        const int threads = packed_threads(nxm, kFrameK);
        if (bw == 8)
            k_full_search_frame_p<8><<<nbx * nby, threads, ldsP, st>>>(a, wsP);
        else if (bw == 16)
            k_full_search_frame_p<16><<<nbx * nby, threads, ldsP, st>>>(a, wsP);
        else
            k_full_search_frame_p<32><<<nbx * nby, threads, ldsP, st>>>(a, wsP);
    } else {
        k_full_search_frame<<<nbx * nby, 256, lds, st>>>(a);
    }
    if (timed) session_timer_end(timer, 3, ev);
    return XG_HIP(hipGetLastError()) ? XG_OK : XG_ERR_HIP;
}

// ---------------------------------------------------------------------------
// Serving search by CTU group
//
// A workgroup and a window staging per block would spend most of the time on
// setup at 1080p, where most blocks are 4..16 wide.  Here a workgroup of four
// waves takes a group (up to 64 blocks of one CTU): it takes every block's
// predictor (written by the AMVP stage, k_amvp_multi) and window, stages the
// union of the windows once in LDS (with the CTU's current samples), and
// spreads the blocks' items over its waves, 64 consecutive items of the
// group's list per wave step.  An item is K = 10 candidate columns of two
// candidate rows (blocks up to 16 wide: each window row read serves both) or
// of one row (wider blocks).  Each block's minimum (cost << 32 | raster index
// in its own window) is kept by an LDS 64-bit atomic min, so the winner and
// the tie order are those of search_block.  The LDS window starts at an even
// column; a block whose window starts at an odd one reads from one column to
// the left and skips its first candidate (s = 1).  A group whose union does
// not fit stages one block's window at a time instead.
// ---------------------------------------------------------------------------
namespace xg {

constexpr int kGroupWaves = 4;
constexpr int kGroupCurDw = 64 * 32;             // the group's current samples: 64 rows x 32 dwords
static_assert(kGroupCurDw % (64 * kGroupWaves) == 0, "whole current-sample rounds per thread");
constexpr int kGroupK = 10;                      // candidates per lane (an odd number of dwords apart: LDS banks)

struct GroupBlk {
    int b;                                       // block index in the list
    int x0, y0, nx, ny;                          // window in integer pel
    int ox, oy;                                  // window origin in the LDS window (ox even)
    int s;                                       // 1 when the origin is one column left of x0
    int nq, np, items, w, h;                     // column groups, row groups (of rpi rows), nq * np
    int rpi;                                     // candidate rows per item: 2 up to 16 wide, else 1
    int pmx, pmy;                                // predictor, quarter pel
    int cur;                                     // dword offset of the block in the current samples
};

// Dword offset of row R of an LDS window whose rows are ws2 dwords apart plus
// one dword after every second row: two rows apart is then an odd number of
// dwords, so lanes two candidate rows apart use different banks.
__device__ __forceinline__ int win_row(int R, int ws2) { return R * ws2 + (R >> 1); }

// K SADs (candidates K q .. K q + K - 1 of origin-relative column) of one
// candidate row for a block BW wide, h rows: window rows R .. R + h - 1 from
// dword column col (win_row layout, pitch ws2), current rows 32 dwords apart.
template <int BW>
__device__ __forceinline__ void group_item(const uint32_t *win, int col, int R, int ws2, const uint32_t *cp, int h,
                                           uint32_t acc[kGroupK])
{
    constexpr int ND = BW / 2, KD = kGroupK / 2;
#pragma unroll
    for (int k = 0; k < kGroupK; k++) acc[k] = 0;
    int off = win_row(R, ws2) + col;
#pragma unroll(BW >= 32 ? 1 : 2)
    for (int i = 0; i < h; i++) {
        uint32_t D[ND + KD], F[ND + KD - 1], C[ND];
#pragma unroll
        for (int j = 0; j < ND + KD; j++) D[j] = win[off + j];
#pragma unroll
        for (int j = 0; j < ND; j++) C[j] = cp[i * 32 + j];
#pragma unroll
        for (int j = 0; j < ND + KD - 1; j++) F[j] = align16(D[j + 1], D[j], 16);
#pragma unroll
        for (int j = 0; j < ND; j++)
#pragma unroll
            for (int m = 0; m < KD; m++) {
                acc[2 * m] = __builtin_amdgcn_sad_u16(D[j + m], C[j], acc[2 * m]);
                acc[2 * m + 1] = __builtin_amdgcn_sad_u16(F[j + m], C[j], acc[2 * m + 1]);
            }
        off += ws2 + ((R + i) & 1);
    }
}

// SADs of one window row against one current row, added to acc.
template <int ND>
__device__ __forceinline__ void row_sads(const uint32_t *D, const uint32_t *F, const uint32_t *C, uint32_t *acc)
{
    constexpr int KD = kGroupK / 2;
#pragma unroll
    for (int j = 0; j < ND; j++)
#pragma unroll
        for (int m = 0; m < KD; m++) {
            acc[2 * m] = __builtin_amdgcn_sad_u16(D[j + m], C[j], acc[2 * m]);
            acc[2 * m + 1] = __builtin_amdgcn_sad_u16(F[j + m], C[j], acc[2 * m + 1]);
        }
}

// The K SADs of two candidate rows at once (acc0: window rows R .., acc1: the
// next one): window row R + i serves current row i of the first and current
// row i - 1 of the second, so each window row is read and realigned once for
// both.  Reads window rows R .. R + h.
template <int BW>
__device__ __forceinline__ void group_item2(const uint32_t *win, int col, int R, int ws2, const uint32_t *cp, int h,
                                            uint32_t acc0[kGroupK], uint32_t acc1[kGroupK])
{
    constexpr int ND = BW / 2, KD = kGroupK / 2;
#pragma unroll
    for (int k = 0; k < kGroupK; k++) acc0[k] = acc1[k] = 0;
    uint32_t D[ND + KD], F[ND + KD - 1], C[ND], Cp[ND];
    int off = win_row(R, ws2) + col;
    auto load_row = [&](int i) {
#pragma unroll
        for (int j = 0; j < ND + KD; j++) D[j] = win[off + j];
#pragma unroll
        for (int j = 0; j < ND + KD - 1; j++) F[j] = align16(D[j + 1], D[j], 16);
        off += ws2 + ((R + i) & 1);
    };
    load_row(0);
#pragma unroll
    for (int j = 0; j < ND; j++) C[j] = cp[j];
    row_sads<ND>(D, F, C, acc0);
#pragma unroll 2
    for (int i = 1; i < h; i++) {
#pragma unroll
        for (int j = 0; j < ND; j++) Cp[j] = C[j];
        load_row(i);
#pragma unroll
        for (int j = 0; j < ND; j++) C[j] = cp[i * 32 + j];
        row_sads<ND>(D, F, C, acc0);
        row_sads<ND>(D, F, Cp, acc1);
    }
    load_row(h);
    row_sads<ND>(D, F, C, acc1);
}

// Runs the items of blocks [j0, j1), flattened: block j holds items
// ibeg[j] .. ibeg[j + 1] - 1 of the group, and each wave takes 64
// consecutive items at a time (stride kGroupWaves waves), so a wave may span
// the end of one block and the start of the next (the host orders a group's
// blocks by width, so such a wave mostly runs one width).
__device__ __forceinline__ void group_units(const uint32_t *win, int ws, const uint32_t *cur, const GroupBlk *gb,
                                            const int *ibeg, int j0, int j1, unsigned long long *gkey,
                                            uint32_t lambda)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int first = ibeg[j0], total = ibeg[j1] - first;
    for (int u0 = 64 * wave; u0 < total; u0 += 64 * kGroupWaves) {
        const int ig = first + u0 + lane;
        int lo = j0, hi = j1 - 1;                 // the block whose items hold ig
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (ibeg[mid] <= ig) lo = mid;
            else hi = mid - 1;
        }
        const GroupBlk &G = gb[lo];
        const int it = ig - ibeg[lo];
        unsigned long long key = ~0ull;
        if (ig < first + total) {
            // item: candidate rows rpi p .. rpi p + rpi - 1, columns K q .. K q + K - 1
            // row group fastest: adjacent lanes read window rows rpi apart (win_row: distinct banks)
            const int q = it / G.np, p = it - q * G.np, dyi = G.rpi * p;
            const int R = G.oy + dyi, col = (G.ox >> 1) + (kGroupK / 2) * q;
            const uint32_t *cp = cur + G.cur;
            const int ws2 = ws >> 1;
            uint32_t acc[2][kGroupK];
            switch (G.w) {
            case 4: group_item2<4>(win, col, R, ws2, cp, G.h, acc[0], acc[1]); break;
            case 8: group_item2<8>(win, col, R, ws2, cp, G.h, acc[0], acc[1]); break;
            case 16: group_item2<16>(win, col, R, ws2, cp, G.h, acc[0], acc[1]); break;
            case 32: group_item<32>(win, col, R, ws2, cp, G.h, acc[0]); break;
            default: {                                   // 64 wide: two 32-wide halves
                uint32_t t[kGroupK];
                group_item<32>(win, col, R, ws2, cp, G.h, acc[0]);
                group_item<32>(win, col + 16, R, ws2, cp + 16, G.h, t);
#pragma unroll
                for (int k = 0; k < kGroupK; k++) acc[0][k] += t[k];
                break;
            }
            }
            // the lane's best: its candidates come in raster order (rows, then columns), so a
            // strict < keeps the lowest index among equal costs, as the 64-bit key order does
            uint32_t bc = 0xFFFFFFFFu, bi = 0;
            uint32_t bxl[kGroupK];
            bool vx[kGroupK];
#pragma unroll
            for (int k = 0; k < kGroupK; k++) {
                const int dx = kGroupK * q + k - G.s;
                vx[k] = dx >= 0 && dx < G.nx;
                bxl[k] = eg_bits(4 * (G.x0 + dx) - G.pmx);
            }
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int dy = dyi + r;
                if (r < G.rpi && dy < G.ny) {
                    const uint32_t by = eg_bits(4 * (G.y0 + dy) - G.pmy);
                    const int row0 = dy * G.nx + kGroupK * q - G.s;
#pragma unroll
                    for (int k = 0; k < kGroupK; k++) {
                        const uint32_t cost = (acc[r][k] << 8) + (bxl[k] + by) * lambda;
                        if (vx[k] && cost < bc) {
                            bc = cost;
                            bi = (uint32_t)(row0 + k);
                        }
                    }
                }
            }
            if (bc != 0xFFFFFFFFu) key = ((unsigned long long)bc << 32) | bi;
        }
        if (__builtin_amdgcn_readfirstlane(lo) == __builtin_amdgcn_readlane(lo, 63)) {
            // one block in the wave (blocks are ordered, so lanes 0 and 63 bound it)
#pragma unroll
            for (int m = 1; m < 64; m <<= 1) {
                const unsigned long long o = (unsigned long long)__shfl_xor((long long)key, m, 64);
                key = o < key ? o : key;
            }
            if (lane == 0) atomicMin(&gkey[lo], key);
        } else if (key != ~0ull) {
            atomicMin(&gkey[lo], key);
        }
    }
}

// rows x (ws/2) dwords of the reference luma plane from picture column cx
// (even) and row cy into win, in the win_row layout.  A thread's dwords i,
// i + blockDim, ... go in batches of 8 loads before their stores (a load per
// iteration would wait out each load's latency in turn); its (row, column)
// steps by (blockDim / nd, blockDim % nd) with a carry, with no division per
// dword.
__device__ __forceinline__ void stage_win_dw(uint32_t *win, int ws, const xg_plane &pl, int cx, int cy, int rows)
{
    const int nd = ws >> 1, n = rows * nd, nt = (int)blockDim.x;
    const int dr = nt / nd, dc = nt - dr * nd;
    const uint16_t *base = pl.data + (intptr_t)cy * pl.stride + cx;
    int r = (int)threadIdx.x / nd, c = (int)threadIdx.x - r * nd;
    for (int i0 = threadIdx.x; i0 < n; i0 += 8 * nt) {
        uint32_t v[8];
        int at[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const bool in = i0 + k * nt < n;
            at[k] = in ? win_row(r, nd) + c : -1;
            if (in) v[k] = *(const gdword *)(base + (intptr_t)r * pl.stride + 2 * c);
            r += dr;
            c += dc;
            if (c >= nd) {
                c -= nd;
                r++;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (at[k] >= 0) win[at[k]] = v[k];
    }
}

__global__ void __launch_bounds__(64 * kGroupWaves) __attribute__((amdgpu_waves_per_eu(4))) k_search_groups(const xg_picture *pics,
                                                                    const SearchList *__restrict__ lists, int nLists,
                                                                    int range, uint32_t lambda, int ctu, int winDw)
{
    extern __shared__ uint32_t win[];                        // winDw dwords
    __shared__ uint32_t cur[kGroupCurDw];
    __shared__ GroupBlk gb[kSearchGroupMax];
    __shared__ unsigned long long gkey[kSearchGroupMax];
    __shared__ int ibeg[kSearchGroupMax + 1];
    __shared__ int box[6];                                   // union x0, y0, x1, y1; current x0, y0
    int l = 0;
    while (l + 1 < nLists && (int)blockIdx.x >= lists[l + 1].begin) l++;
    const SearchList &L = lists[l];
    const int2 G = L.groups[(int)blockIdx.x - L.begin];
    const int count = G.y, t = threadIdx.x;
    const xg_picture &P = pics[L.curSlot], &R = pics[L.refSlot];
    const int fw = P.plane[0].width, fh = P.plane[0].height;
    if (t == 0) {
        box[0] = box[1] = INT_MAX;
        box[2] = box[3] = INT_MIN;
        box[4] = box[5] = INT_MAX;
    }
    __syncthreads();
    xg_block B;
    int x0 = 0, y0 = 0, nx = 0, ny = 0;
    if (t < count) {
        const int b = L.gidx[G.x + t];
        B = L.blocks[b];
        B.pic = L.curSlot;
        B.ref = L.refSlot;
        const int mnx = (int16_t)(-B.x - ctu - 8), mny = (int16_t)(-B.y - ctu - 8);
        const int mxx = (int16_t)(fw + (ctu - B.w + 8) - B.x), mxy = (int16_t)(fh + (ctu - B.h + 8) - B.y);
        const int cx = min(max(((B.mvpx >> 2) + 2) >> 2, mnx), mxx), cy = min(max(((B.mvpy >> 2) + 2) >> 2, mny), mxy);
        x0 = max(cx - range, mnx);
        y0 = max(cy - range, mny);
        nx = min(cx + range, mxx) - x0 + 1;
        ny = min(cy + range, mxy) - y0 + 1;
        const int sx = (B.x + x0) & 1;                       // origin one column left when odd
        const int nq = (nx + sx + kGroupK - 1) / kGroupK;
        GroupBlk g;
        g.b = b;
        g.x0 = x0; g.y0 = y0; g.nx = nx; g.ny = ny;
        g.s = sx;
        g.nq = nq;
        g.rpi = B.w <= 16 ? 2 : 1;
        g.np = (ny + g.rpi - 1) / g.rpi;
        g.items = g.np * nq;
        g.w = B.w; g.h = B.h;
        g.pmx = B.mvpx >> 2; g.pmy = B.mvpy >> 2;
        gb[t] = g;
        gkey[t] = ~0ull;
        atomicMin(&box[0], B.x + x0 - sx);
        atomicMin(&box[1], B.y + y0);
        atomicMax(&box[2], B.x + x0 - sx + kGroupK * nq + B.w);   // columns the last item reads, exclusive
        atomicMax(&box[3], B.y + y0 + ny - 1 + B.h);
        atomicMin(&box[4], (int)B.x);
        atomicMin(&box[5], (int)B.y);
    }
    __syncthreads();
    // row pitch: an odd number of dwords, so the lanes' rows spread over the LDS banks
    const int ux0 = box[0], uy0 = box[1], rows = box[3] - box[1];
    const int ws = (((box[2] - box[0]) + 1) & ~1) | 2;
    const int cx0 = box[4], cy0 = box[5];
    if (t < count) {
        gb[t].ox = B.x + x0 - gb[t].s - ux0;
        gb[t].oy = B.y + y0 - uy0;
        gb[t].cur = (B.y - cy0) * 32 + ((B.x - cx0) >> 1);
    }
    if (t == 0) {
        ibeg[0] = 0;
        for (int j = 0; j < count; j++) ibeg[j + 1] = ibeg[j] + gb[j].items;
    }
    // the group's current samples (within 64x64 of (cx0, cy0): checked on the
    // host), every load of a thread issued before its first store
    {
        constexpr int kPer = kGroupCurDw / (64 * kGroupWaves);
        uint32_t v[kPer];
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = t + k * 64 * kGroupWaves, r = i >> 5, c = i & 31;
            const bool in = cy0 + r < fh && cx0 + 2 * c < fw;
            v[k] = in ? *(const gdword *)(P.plane[0].data + (intptr_t)(cy0 + r) * P.plane[0].stride + cx0 + 2 * c)
                      : 0u;
        }
#pragma unroll
        for (int k = 0; k < kPer; k++) cur[t + k * 64 * kGroupWaves] = v[k];
    }
    if (win_row(rows + 1, ws >> 1) <= winDw) {               // an item may read one row past the windows
        stage_win_dw(win, ws, R.plane[0], ux0, uy0, rows);
        __syncthreads();
        group_units(win, ws, cur, gb, ibeg, 0, count, gkey, lambda);
    } else {
        // one block's window at a time
        for (int j = 0; j < count; j++) {
            __syncthreads();                                 // the previous block's readers are done
            const GroupBlk g = gb[j];
            const int bx = ux0 + g.ox, byy = uy0 + g.oy;     // the block's window origin in the picture
            const int wsj = ((kGroupK * g.nq + g.w + 1) & ~1) | 2, rj = g.ny + g.h - 1;   // odd dword pitch
            stage_win_dw(win, wsj, R.plane[0], bx, byy, rj);
            if (t == 0) {
                gb[j].ox = 0;
                gb[j].oy = 0;
            }
            __syncthreads();
            group_units(win, wsj, cur, gb, ibeg, j, j + 1, gkey, lambda);
        }
    }
    __syncthreads();
    if (t < count) {
        const unsigned long long k = gkey[t];
        const int i = (int)(uint32_t)k;
        B.mvx = 16 * (x0 + i % nx);
        B.mvy = 16 * (y0 + i / nx);
        L.blocks[gb[t].b] = B;
    }
}

}  // namespace xg

void xg::search_groups(const xg_block *blocks, int n, std::vector<int> &gidx, std::vector<int2> &groups)
{
    // blocks of each 64x64 CTU (by top-left sample), in list order
    std::vector<std::pair<long, int>> key(n);
    for (int i = 0; i < n; i++) key[i] = {((long)(blocks[i].y >> 6) << 20) | (blocks[i].x >> 6), i};
    std::stable_sort(key.begin(), key.end(), [](const std::pair<long, int> &a, const std::pair<long, int> &b) {
        return a.first < b.first;
    });
    gidx.clear();
    groups.clear();
    for (int a = 0; a < n;) {
        int e = a;
        while (e < n && key[e].first == key[a].first) e++;
        int x0 = INT_MAX, y0 = INT_MAX, x1 = INT_MIN, y1 = INT_MIN;
        for (int k = a; k < e; k++) {
            const xg_block &B = blocks[key[k].second];
            x0 = std::min(x0, (int)B.x);
            y0 = std::min(y0, (int)B.y);
            x1 = std::max(x1, B.x + B.w);
            y1 = std::max(y1, B.y + B.h);
        }
        const bool fits = x1 - x0 <= 64 && y1 - y0 <= 64;
        // narrowest first: the waves of k_search_groups run consecutive items
        std::stable_sort(key.begin() + a, key.begin() + e, [&](const std::pair<long, int> &p, const std::pair<long, int> &q) {
            return blocks[p.second].w < blocks[q.second].w;
        });
        for (int k = a; k < e;) {
            const int c = fits ? std::min(kSearchGroupMax, e - k) : 1;   // blocks past 64x64: one per group
            groups.push_back(make_int2((int)gidx.size(), c));
            for (int m = 0; m < c; m++) gidx.push_back(key[k + m].second);
            k += c;
        }
        a = e;
    }
}

int32_t xg::search_groups_enqueue(hipStream_t st, xg_session *timer, const xg_picture *dPics, const SearchList *dLists,
                                  int nLists, int nGroups, int range, uint32_t lambda, int ctu)
{
    if (nLists <= 0 || nGroups <= 0) return XG_OK;
    // room for one 64x64 block's window at this range (the fallback), and for
    // the union of a CTU's windows when their predictors agree
    const int nqMax = (2 * range + 2 + kGroupK - 1) / kGroupK;
    // row pitches plus one dword per two rows (win_row)
    const int oneRows = 2 * range + 65, oneNd = ((kGroupK * nqMax + 64) + 1) / 2 + 1;
    const int one = oneRows * oneNd + oneRows / 2;
    const int uRows = 2 * range + 64 + 4, uNd = (2 * range + 64 + kGroupK + 8) / 2 + 1;
    const int winDw = std::max(one, uRows * uNd + uRows / 2);
    if (winDw * 4 + (int)(kGroupCurDw * 4 + kSearchGroupMax * (sizeof(GroupBlk) + 12)) > 64 * 1024) {
        set_error(XG_ERR_ARG, "search_groups_enqueue: window exceeds the LDS budget");
        return XG_ERR_ARG;
    }
    int ev[2];
    const bool timed = timer && session_timer_begin(timer, 3, ev);
    k_search_groups<<<nGroups, 64 * kGroupWaves, (size_t)winDw * 4, st>>>(dPics, dLists, nLists, range, lambda, ctu,
                                                                          winDw);
    if (timed) session_timer_end(timer, 3, ev);
    return XG_HIP(hipGetLastError()) ? XG_OK : XG_ERR_HIP;
}
