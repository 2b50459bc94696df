// Upstream motion producer of the KV-arena path, gfx950-native: dense
// Farneback optical flow between consecutive gray frames and the per-tile
// change rates the gating policies rank (reference:
// traces/gen_motion_from_video.py:104-135, which calls OpenCV's
// cv2.calcOpticalFlowFarneback with pyr_scale 0.5, levels 3, winsize 15,
// iterations 3, poly_n 5, poly_sigma 1.2, flags 0).
//
// The algorithm is the one OpenCV 4.x publishes (modules/video/src/
// optflowgf.cpp; Farneback, "Two-frame motion estimation based on
// polynomial expansion", SCIA 2003), laid out for the GPU: a launch covers many
// frames (or consecutive pairs: chunk_pairs) of a clip, the pyramid kernels several levels,
// and each frame's pyramid image and polynomial expansion are computed once per
// level and shared by the two pairs that use it.
//
//   preblur_kernel           Gaussian pre-blur (reflect-101 border) and
//                            bilinear resize (half-pixel centres, clamped
//                            edges) of the reduced levels, uint8 -> fp32.
//   poly_exp_kernel          quadratic fit under a separable Gaussian
//                            applicability (2n+1 taps), replicated border;
//                            64 x 40 tile + halo in LDS, vertical then
//                            horizontal pass; 5 fp32 values per pixel
//                            [b_y, b_x, a_yy, a_xx, a_xy]. The full-size
//                            level's 3-tap pre-blur is part of it.
//   init_flow_kernel         a level's initial flow: zero, or the coarser
//                            level's resized and scaled by 1/pyr_scale.
//   flow_step_kernel         one iteration for winsize 15 (the reference's; 14
//                            has the same window): per pixel, the next frame's
//                            expansion sampled bilinearly at x + flow,
//                            averaged with the previous frame's, border
//                            down-weighting, the 5 values of A^T A and A^T
//                            delta-b; their box average (replicated border,
//                            fp64 running column sums); the regularised 2 x 2
//                            solve in fp64.
//   update_matrices_kernel,  the same in two launches, the matrices in HBM, for
//   update_flow_kernel       other window sizes.
//   flow_cells_kernel        |flow| averaged over grid cells (one workgroup
//                            per cell row), then tile_change_kernel: the mean
//                            of each run of tile_tokens cells in fp64.
//
// Layout in HBM: frames uint8 [n, H, W] (any frame stride); pyramid image
// fp32 [n, h, w]; expansion fp32, per frame [h*w][4] then [h*w]; matrices fp32
// [pairs][5][h*w]; flow fp32 [pairs, h, w, 2] (x, y), the final level written
// straight into the caller's output.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <vector>

#include "kvp_internal.h"
#include "kvp_motion.h"

namespace kvp {
namespace {

constexpr int kMaxBlurTaps = 127;   // pre-blur kernel size (level scale >= 1/26)
constexpr int kMaxPolyN = 8;        // applicability half-width
constexpr int kMaxBoxHalf = 24;     // winsize <= 49
constexpr int kMinLevelSide = 32;   // OpenCV's min_size for a pyramid level
constexpr int kBorder = 5;          // down-weighted border width
constexpr int kMinSide = 2 * kBorder;
constexpr int kMaxSide = 8192;
constexpr int kMaxFrames = 4096;
// expansion: 320 threads as 4 rows of 80 columns (source tile, <= 80 columns
// with its halo), as 4 x 74 column runs of 10 rows and as 5 rows of 64 pixels
constexpr int kPeTileW = 64, kPeTileH = 40, kPeThreads = 320;
constexpr int kPeRun = 10;
constexpr int kPeCols = 80;
constexpr int kPbTileW = 32;                        // pre-blur: level columns per block
constexpr int kPbRows = 32;                         // source rows under a block's level rows
constexpr size_t kPbLdsBytes = 64 << 10;            // rows are cut to what fits this
constexpr int kPyrLevels = 9;                       // 8192 px down to 32 px at scale 0.5
constexpr int kPyrTaps = 512;
constexpr long kStepChunkPixels = 17L * 832 * 480;  // pixels x pairs of a chunk: window 15,
constexpr long kChunkPixels = 32 * kStepChunkPixels;  // and any other
constexpr int kBfBatch = 4;       // box filter: rows parked in LDS at a time
constexpr int kBfRun = 2;         // box filter: output columns per sliding run
constexpr int kBfTargetGroups = 2048;
constexpr int kNumXcd = 8;
// whole-iteration kernel (flow_step_kernel): window half-width it serves
// (winsize 15, the reference's), columns of a strip with its halo, threads,
// strips in flight on the chip (two workgroups per CU)
constexpr int kFsHalf = 7;
constexpr int kFsCols = 100;
constexpr int kFsThreads = 512;
constexpr int kFsSlots = 512;

struct BlurTaps {
    int ksize;
    float k[kMaxBlurTaps];
};

struct PolyTaps {
    int n;
    float g[2 * kMaxPolyN + 1];
    float xg[2 * kMaxPolyN + 1];
    float xxg[2 * kMaxPolyN + 1];
    double ig11, ig03, ig33, ig55;
};

__device__ __forceinline__ int reflect101(int i, int n) {
    if (n == 1) return 0;
    const int period = 2 * n - 2;
    i = i < 0 ? -i : i;
    i %= period;
    return i >= n ? period - i : i;
}

// Contiguous run of blocks per XCD (the hardware hands block b to XCD b % 8).
__device__ __forceinline__ int xcd_contiguous(int b, int n) {
    const int per = n / kNumXcd, rem = n % kNumXcd;
    const int x = b % kNumXcd, i = b / kNumXcd;
    return x < rem ? x * (per + 1) + i : rem * (per + 1) + (x - rem) * per + i;
}

// resize INTER_LINEAR source taps of destination index d: s0, s1 and the
// weight of s1 (OpenCV: fx = (d + 0.5) * scale - 0.5, clamped at both ends).
__device__ __forceinline__ void linear_tap(int d, double scale, int src, int& s0, int& s1,
                                           float& w) {
    float f = (float)((d + 0.5) * scale - 0.5);
    int s = (int)floorf(f);
    f -= (float)s;
    if (s < 0) { f = 0.f; s = 0; }
    if (s >= src - 1) { f = 0.f; s = src - 1; }
    s0 = s;
    s1 = min(s + 1, src - 1);
    w = f;
}

// One pyramid level of a merged pyramid launch (blocks of several levels in
// one grid; block b belongs to the last level whose first_block <= b).
struct PyrLevel {
    int w, h;
    int first_block, tiles_x;
    int tile_h;            // preblur_kernel: level rows per block
    int ksize, tap0;       // its pre-blur taps within PyrArgs::taps
    int stage_at;          // LDS byte offset of the staged source, 0: not staged
    double sx, sy;         // source pixels per level pixel
    long img, R;           // float offsets of the level's planes from the base
                           // (img < 0: the full-size level, blurred on the fly)
    int slots;             // frames the level's R holds: frame f is in slot f % slots
};

struct PyrArgs {
    int levels, frames;
    int W, H;
    int first_frame;       // blockIdx.z = 0 is this frame (expansion)
    const uint8_t* src;
    long frame_stride;
    float* base;           // img / R offsets count from here
    PyrLevel lv[kPyrLevels];
    float taps[kPyrTaps];
};

__device__ __forceinline__ const PyrLevel& pyr_level(const PyrArgs& a, int block) {
    int l = 0;
    for (int i = 1; i < a.levels; ++i)
        if (block >= a.lv[i].first_block) l = i;
    return a.lv[l];
}

// Gaussian pre-blur (reflect-101 border) and bilinear resize of a reduced
// level in one pass: a block of kPbTileW x tile_h level pixels (tile_h so that
// its rows lie over about 32 source rows) stages the source bytes under it in
// LDS, blurs, along x, the two source columns each level column samples, over
// the source rows its level rows reach, again into LDS; then blurs those along
// y at the two rows each level row samples and blends. A pixel's two columns
// (rows) are neighbours and share their taps' reads. Nothing but the uint8
// source is read from HBM and nothing but the level is written: as two launches
// per level with the x-blurred rows in HBM the three reduced levels of a
// 50-frame 832x480 clip took 247 us, and take 148 us in one launch for all of them
// (bound by the taps' byte reads and conversions on the VALU).
template <int kTaps>
__device__ __forceinline__ void preblur_tile(const PyrArgs& a, const PyrLevel& L, float* hb) {
    uint8_t* bytes = reinterpret_cast<uint8_t*>(hb) + L.stage_at;
    const int t = (int)blockIdx.x - L.first_block;
    const int X0 = (t % L.tiles_x) * kPbTileW, Y0 = (t / L.tiles_x) * L.tile_h;
    const int f = a.first_frame + (int)blockIdx.z;
    const uint8_t* src = a.src + (long)f * a.frame_stride;
    const float* tap = a.taps + L.tap0;
    const int ksize = kTaps ? kTaps : L.ksize;
    const int hk = ksize / 2, W = a.W, H = a.H;
    int ya, yb, r_lo, r_hi;
    float wt;
    linear_tap(Y0, L.sy, H, ya, yb, wt);
    r_lo = ya - hk;
    linear_tap(min(Y0 + L.tile_h, L.h) - 1, L.sy, H, ya, yb, wt);
    r_hi = yb + hk;
    const int rows = r_hi - r_lo + 1;
    // mirrored rows only at the top and bottom of the image
    const bool rows_in = r_lo >= 0 && r_hi < H;
    auto src_row = [&](int r) { return rows_in ? r_lo + r : reflect101(r_lo + r, H); };
    const int px = (int)threadIdx.x & (kPbTileW - 1);
    const int first = (int)threadIdx.x / kPbTileW;
    constexpr int kStep = 256 / kPbTileW;
    const int x = X0 + px;
    int xa, xb;
    float wx;
    linear_tap(min(x, L.w - 1), L.sx, W, xa, xb, wx);
    const bool inner = xa >= hk && xa + 1 + hk < W;
    // the x pass of row r from `row` (its column 0)
    auto x_pass = [&](const uint8_t* row, int r) {
        float s0 = 0.f, s1 = 0.f;
        if (inner) {
            const uint8_t* v = row + (xa - hk);
            float cur = (float)v[0];
#pragma unroll
            for (int k = 0; k < (kTaps ? kTaps : ksize); ++k) {
                const float next = (float)v[k + 1];
                s0 += tap[k] * cur;
                s1 += tap[k] * next;
                cur = next;
            }
        } else {
            for (int k = 0; k < ksize; ++k) {
                s0 += tap[k] * (float)row[reflect101(xa - hk + k, W)];
                s1 += tap[k] * (float)row[reflect101(xb - hk + k, W)];
            }
        }
        *reinterpret_cast<float2*>(hb + (r * kPbTileW + px) * 2) = make_float2(s0, s1);
    };
    if (L.stage_at) {
        // source columns [c_lo, c_lo + pitch) of the block's rows as bytes
        int x0, x1;
        linear_tap(X0, L.sx, W, x0, x1, wt);
        const int c_lo = max(x0 - hk, 0) & ~3;
        linear_tap(min(X0 + kPbTileW, L.w) - 1, L.sx, W, x0, x1, wt);
        const int c_hi = min(x1 + hk, W - 1);
        const int pitch = (c_hi - c_lo + 4) & ~3;
        if ((W & 3) == 0 && ((uintptr_t)src & 3) == 0) {
            // a wave per row: W is a multiple of 4, so the last word is whole
            for (int r = (int)threadIdx.x >> 6; r < rows; r += 4) {
                const unsigned* row =
                    reinterpret_cast<const unsigned*>(src + (long)src_row(r) * W + c_lo);
                for (int q = (int)threadIdx.x & 63; q < pitch / 4; q += 64)
                    reinterpret_cast<unsigned*>(bytes + r * pitch)[q] = row[q];
            }
        } else {
            for (int r = (int)threadIdx.x >> 6; r < rows; r += 4) {
                const uint8_t* row = src + (long)src_row(r) * W;
                for (int q = (int)threadIdx.x & 63; q < pitch; q += 64)
                    bytes[r * pitch + q] = row[min(c_lo + q, W - 1)];
            }
        }
        __syncthreads();
        for (int r = first; r < rows; r += kStep) x_pass(bytes + r * pitch - c_lo, r);
    } else {
        for (int r = first; r < rows; r += kStep) x_pass(src + (long)src_row(r) * W, r);
    }
    __syncthreads();
    float* out = a.base + L.img + (long)f * L.w * L.h;
    for (int yy = first; yy < L.tile_h; yy += kStep) {
        const int y = Y0 + yy;
        if (x >= L.w || y >= L.h) continue;
        float wy;
        linear_tap(y, L.sy, H, ya, yb, wy);
        // both blurred rows from one walk down the column (yb is ya + 1, or ya
        // at the bottom edge, where its weight is 0)
        const float2* v = reinterpret_cast<const float2*>(hb) + (ya - hk - r_lo) * kPbTileW + px;
        const int end = min(ksize, rows - 1 - (ya - hk - r_lo));  // last row of the walk
        float2 lo = make_float2(0.f, 0.f), hi = lo, cur = v[0];
#pragma unroll
        for (int k = 0; k < (kTaps ? kTaps : ksize); ++k) {
            const float2 next = v[(k + 1 < ksize ? k + 1 : end) * kPbTileW];
            lo.x += tap[k] * cur.x;
            lo.y += tap[k] * cur.y;
            hi.x += tap[k] * next.x;
            hi.y += tap[k] * next.y;
            cur = next;
        }
        const float r0 = lo.x * (1.f - wx) + lo.y * wx;
        const float r1 = hi.x * (1.f - wx) + hi.y * wx;
        out[(long)y * L.w + x] = r0 * (1.f - wy) + r1 * wy;
    }
}

__global__ __launch_bounds__(256) void preblur_kernel(PyrArgs a) {
    extern __shared__ float hb[];  // [rows][2 * kPbTileW]
    const PyrLevel& L = pyr_level(a, blockIdx.x);
    // tap counts of the halving pyramid's levels: unrolled, so that a pixel's
    // byte loads are in flight together
    switch (L.ksize) {
        case 3: preblur_tile<3>(a, L, hb); break;
        case 9: preblur_tile<9>(a, L, hb); break;
        case 19: preblur_tile<19>(a, L, hb); break;
        default: preblur_tile<0>(a, L, hb);
    }
}

// Quadratic expansion of the blocks' levels. The full-size level (its pre-blur
// is always the 3-tap [1 2 1] / 4) is read as uint8 and blurred in LDS, so its
// blurred image never goes to HBM; reduced levels read preblur_kernel's image.
// The border is replicated. kN is the half-width when it is the reference's 5
// (taps in registers, loops unrolled), 0 for any other.
// Bound by the VALU (about 190 instructions per pixel, halo included): 4.1 us a
// frame of 832x480 (21 B per pixel: 2.0 TB/s); as row blur, column blur and
// expansion, each through HBM, the full-size level took 6.1 us a frame.
template <int kN>
__global__ __launch_bounds__(kPeThreads) void poly_exp_kernel(PyrArgs a, PolyTaps t) {
    constexpr int kNMax = kN ? kN : kMaxPolyN;
    constexpr int MW = kPeTileW + 2 * kNMax;   // src columns
    constexpr int MH = kPeTileH + 2 * kNMax;   // src rows
    constexpr int RW = MW + 2;                 // image columns under them
    constexpr int kRowStep = kPeThreads / kPeCols;
    static_assert(MW <= kPeCols, "a thread per source column");
    __shared__ float src[MH * MW];
    // the 3 y-filtered planes; before that the image and its x-blurred rows
    constexpr int kVp = 3 * kPeTileH * MW, kRows = (MH + 2) * (RW + MW);
    __shared__ float vp[kVp > kRows ? kVp : kRows];
    const int n = kN ? kN : t.n;
    const PyrLevel& L = pyr_level(a, blockIdx.x);
    const int tile = (int)blockIdx.x - L.first_block;
    const int X0 = (tile % L.tiles_x) * kPeTileW, Y0 = (tile / L.tiles_x) * kPeTileH;
    const int f = a.first_frame + (int)blockIdx.z;
    const int w = L.w, h = L.h;
    const long P = (long)w * h;
    const int tw = kPeTileW + 2 * n;
    const int tid = threadIdx.x;
    const int cc = tid % kPeCols, rr = tid / kPeCols;
    if (L.img < 0) {
        // image rows Y0-n-1 .. and columns X0-n-1 .. (clamped into the image)
        // as floats; blurred along x, then along y, at the clamped position of
        // every src value, mirroring at the border. The values are multiples of
        // 1/16 below 256: exact.
        const uint8_t* I = a.src + (long)f * a.frame_stride;
        float* raw = vp;
        float* bx = vp + (MH + 2) * RW;
        const int oy = Y0 - n - 1, ox = X0 - n - 1;
        constexpr int kRaw = (MH + 2 + kRowStep - 1) / kRowStep;
        uint8_t u[kRaw] = {};
        // kPeCols may be one column short of RW: the last ones by row 0's threads
        const int gx = min(max(ox + cc, 0), w - 1);
#pragma unroll
        for (int k = 0; k < kRaw; ++k)
            u[k] = I[(long)min(max(oy + rr + kRowStep * k, 0), h - 1) * w + gx];
#pragma unroll
        for (int k = 0; k < kRaw; ++k) {
            const int r = rr + kRowStep * k;
            if (cc < RW && r < MH + 2) raw[r * RW + cc] = (float)u[k];
        }
        if constexpr (RW > kPeCols) {
            for (int i = tid; i < (MH + 2) * (RW - kPeCols); i += kPeThreads) {
                const int r = i / (RW - kPeCols), c = kPeCols + i % (RW - kPeCols);
                raw[r * RW + c] = (float)I[(long)min(max(oy + r, 0), h - 1) * w +
                                           min(max(ox + c, 0), w - 1)];
            }
        }
        __syncthreads();
        const int x = min(max(X0 - n + cc, 0), w - 1);
        if (cc < MW) {
            const float* lo = raw + (x == 0 ? 1 : x - 1) - ox;
            const float* mid = raw + x - ox;
            const float* hi = raw + (x == w - 1 ? w - 2 : x + 1) - ox;
#pragma unroll
            for (int k = 0; k < kRaw; ++k) {
                const int r = rr + kRowStep * k;
                if (r < MH + 2)
                    bx[r * MW + cc] = 0.25f * lo[r * RW] + 0.5f * mid[r * RW] + 0.25f * hi[r * RW];
            }
        }
        __syncthreads();
        if (cc < MW) {
            const float* col = bx - oy * MW + cc;
            const bool in = Y0 - n > 0 && Y0 - n + MH < h;  // no row is mirrored or clamped
#pragma unroll
            for (int k = 0; k < kRaw; ++k) {
                const int r = rr + kRowStep * k;
                if (r >= MH) break;
                int y = Y0 - n + r, ym = y - 1, yp = y + 1;
                if (!in) {
                    y = min(max(y, 0), h - 1);
                    ym = y == 0 ? 1 : y - 1;
                    yp = y == h - 1 ? h - 2 : y + 1;
                }
                src[r * MW + cc] = 0.25f * col[ym * MW] + 0.5f * col[y * MW] + 0.25f * col[yp * MW];
            }
        }
    } else {
        const float* I = a.base + L.img + (long)f * P;
        constexpr int kSrc = (MH + kRowStep - 1) / kRowStep;
        float u[kSrc];
        const int gx = min(max(X0 - n + cc, 0), w - 1);
#pragma unroll
        for (int k = 0; k < kSrc; ++k)
            u[k] = I[(long)min(max(Y0 - n + rr + kRowStep * k, 0), h - 1) * w + gx];
#pragma unroll
        for (int k = 0; k < kSrc; ++k) {
            const int r = rr + kRowStep * k;
            if (cc < MW && r < MH) src[r * MW + cc] = u[k];
        }
    }
    __syncthreads();
    // y pass: a thread takes kPeRun rows of one column, its 2n + kPeRun source
    // values read once
    static_assert(kPeTileH % kPeRun == 0, "whole runs");
    for (int i = tid; i < kPeTileH / kPeRun * tw; i += kPeThreads) {
        const int r0 = i / tw * kPeRun, c = i % tw;
        float v[kPeRun + 2 * kNMax];
#pragma unroll
        for (int k = 0; k < kPeRun + 2 * kNMax; ++k)
            if (kN || k < kPeRun + 2 * n) v[k] = src[(r0 + k) * MW + c];
#pragma unroll
        for (int r = 0; r < kPeRun; ++r) {
            float s0, s1 = 0.f, s2 = 0.f;
            if constexpr (kN > 0) {
                s0 = v[r + kN] * t.g[kN];
#pragma unroll
                for (int k = 1; k <= kN; ++k) {
                    const float lo = v[r + kN - k], hi = v[r + kN + k];
                    const float p = lo + hi;
                    s0 += t.g[kN + k] * p;
                    s1 += t.xg[kN + k] * (hi - lo);
                    s2 += t.xxg[kN + k] * p;
                }
            } else {
                const float* u = src + (r0 + r + n) * MW + c;
                s0 = u[0] * t.g[n];
                for (int k = 1; k <= n; ++k) {
                    const float lo = u[-k * MW], hi = u[k * MW];
                    const float p = lo + hi;
                    s0 += t.g[n + k] * p;
                    s1 += t.xg[n + k] * (hi - lo);
                    s2 += t.xxg[n + k] * p;
                }
            }
            vp[(r0 + r) * MW + c] = s0;
            vp[(kPeTileH + r0 + r) * MW + c] = s1;
            vp[(2 * kPeTileH + r0 + r) * MW + c] = s2;
        }
    }
    __syncthreads();
    float* Rf = a.base + L.R + (long)(f % L.slots) * 5 * P;
    // x pass: a pixel per thread, so that a wave's stores are contiguous
    const int c = tid % kPeTileW, x = X0 + c;
    if (x >= w) return;
    const bool vec = ((uintptr_t)Rf & 15) == 0;
    for (int r = tid / kPeTileW; r < kPeTileH; r += kPeThreads / kPeTileW) {
        const int y = Y0 + r;
        if (y >= h) break;
        const float* v0 = vp + r * MW + c + n;
        const float* v1 = v0 + kPeTileH * MW;
        const float* v2 = v1 + kPeTileH * MW;
        const float g0 = t.g[n];
        float b1 = v0[0] * g0, b2 = 0.f, b3 = v1[0] * g0, b4 = 0.f, b5 = v2[0] * g0, b6 = 0.f;
#pragma unroll
        for (int k = 1; k <= (kN ? kN : n); ++k) {
            const float gk = t.g[n + k], xgk = t.xg[n + k], xxgk = t.xxg[n + k];
            const float tg = v0[k] + v0[-k];
            b1 += tg * gk;
            b4 += tg * xxgk;
            b2 += (v0[k] - v0[-k]) * xgk;
            b3 += (v1[k] + v1[-k]) * gk;
            b6 += (v1[k] - v1[-k]) * xgk;
            b5 += (v2[k] + v2[-k]) * gk;
        }
        const long o = (long)y * w + x;
        const float4 q = make_float4((float)(b3 * t.ig11), (float)(b2 * t.ig11),
                                     (float)(b1 * t.ig03 + b5 * t.ig33),
                                     (float)(b1 * t.ig03 + b4 * t.ig33));
        if (vec) {
            reinterpret_cast<float4*>(Rf)[o] = q;
        } else {
            Rf[4 * o] = q.x;
            Rf[4 * o + 1] = q.y;
            Rf[4 * o + 2] = q.z;
            Rf[4 * o + 3] = q.w;
        }
        Rf[4 * P + o] = (float)(b6 * t.ig55);
    }
}

__device__ __forceinline__ float border_weight(int i) {
    return i == 0 || i == 1 ? 0.14f : 0.4472f;
}

// weight of position i of n along one axis
__device__ __forceinline__ float axis_weight(int i, int n) {
    return (i < kBorder ? border_weight(i) : 1.f) *
           (i >= n - kBorder ? border_weight(n - i - 1) : 1.f);
}

// Flow of the coarser level (cw x ch) resized bilinearly to a pixel of the next
// one, times mul; (xa, xb, wx) and (ya, yb, wy) are the pixel's taps.
__device__ __forceinline__ float2 coarse_flow(const float2* __restrict__ C, int cw, int xa, int xb,
                                              float wx, int ya, int yb, float wy, float mul) {
    const float2 a = C[(long)ya * cw + xa], b = C[(long)ya * cw + xb];
    const float2 c = C[(long)yb * cw + xa], d = C[(long)yb * cw + xb];
    const float rx0 = a.x * (1.f - wx) + b.x * wx, ry0 = a.y * (1.f - wx) + b.y * wx;
    const float rx1 = c.x * (1.f - wx) + d.x * wx, ry1 = c.y * (1.f - wx) + d.y * wx;
    return make_float2((rx0 * (1.f - wy) + rx1 * wy) * mul, (ry0 * (1.f - wy) + ry1 * wy) * mul);
}

// A frame's expansion (h*w pixels of 4 floats [b_y, b_x, a_yy, a_xx], then h*w
// floats a_xy; below 2^31 bytes: sides are at most 8192) as a buffer: loads take
// a 32-bit byte offset per lane and a scalar one, so that none needs address
// arithmetic of its own on the VALU. A wave's gather of one value per lane
// costs the L1 about as much as one of 4 (it serves 64 bytes a cycle, and a
// group of lanes off the 64-byte grid takes two), which is why 4 of the 5
// values lie together.
struct Expansion {
    __amdgpu_buffer_rsrc_t rs;
    int xy;  // byte offset of the a_xy plane
};

__device__ __forceinline__ Expansion expansion(const float* R, int w, int h) {
    const int plane = w * h * 4;
    return {__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(R), (short)0, 5 * plane,
                                              0x00020000),
            4 * plane};
}

// The values of pixel row * w + px (pixel offsets; `row` uniform).
__device__ __forceinline__ void load_pixel(const Expansion& e, int px, int row, float (&v)[5]) {
    const auto u = __builtin_amdgcn_raw_buffer_load_b128(e.rs, 16 * px, 16 * row, 0);
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = __uint_as_float(u[c]);
    v[4] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(e.rs, 4 * px, e.xy + 4 * row, 0));
}

// The 5 values of A^T A and A^T delta-b at pixel (x, y) with flow (dx, dy), in
// two halves so that a thread can have the loads of several pixels in flight.
struct PixelSamples {
    float q[5];          // the previous frame's expansion at (x, y)
    float s[4][5];       // the next frame's at the 2 x 2 pixels around (x, y) + flow
};

// sampling position: top left pixel, weights, whether it lies in the image
__device__ __forceinline__ bool sample_at(int w, int h, int x, int y, float2 d, int& x1, int& y1,
                                          float& fx, float& fy) {
    fx = (float)x + d.x;
    fy = (float)y + d.y;
    // keep the float -> int conversion defined; anything this far out is outside
    fx = fminf(fmaxf(fx, -1e8f), 1e8f);
    fy = fminf(fmaxf(fy, -1e8f), 1e8f);
    x1 = (int)floorf(fx);
    y1 = (int)floorf(fy);
    fx -= (float)x1;
    fy -= (float)y1;
    return (unsigned)x1 < (unsigned)(w - 1) && (unsigned)y1 < (unsigned)(h - 1);
}

__device__ __forceinline__ void load_samples(const Expansion& R0, const Expansion& R1, int w, int h,
                                             int x, int y, float2 d, PixelSamples& s) {
    load_pixel(R0, y * w + x, 0, s.q);
    int x1, y1;
    float fx, fy;
    // outside the image the samples are loaded from pixel 0 and not used
    const bool inside = sample_at(w, h, x, y, d, x1, y1, fx, fy);
    const int o = inside ? y1 * w + x1 : 0;
    load_pixel(R1, o, 0, s.s[0]);
    load_pixel(R1, o, 1, s.s[1]);
    load_pixel(R1, o, w, s.s[2]);
    load_pixel(R1, o, w + 1, s.s[3]);
}

// sc: the border weight
__device__ __forceinline__ void pixel_matrices(const PixelSamples& p, int w, int h, int x, int y,
                                               float2 d, float sc, float (&m)[5]) {
    int x1, y1;
    float fx, fy;
    const bool inside = sample_at(w, h, x, y, d, x1, y1, fx, fy);
    const float a00 = (1.f - fx) * (1.f - fy), a01 = fx * (1.f - fy);
    const float a10 = (1.f - fx) * fy, a11 = fx * fy;
    float s[5];
#pragma unroll
    for (int c = 0; c < 5; ++c)
        s[c] = a00 * p.s[0][c] + a01 * p.s[1][c] + a10 * p.s[2][c] + a11 * p.s[3][c];
    float r2 = inside ? s[0] : 0.f, r3 = inside ? s[1] : 0.f;
    const float r4 = inside ? (p.q[2] + s[2]) * 0.5f : p.q[2];
    const float r5 = inside ? (p.q[3] + s[3]) * 0.5f : p.q[3];
    const float r6 = inside ? (p.q[4] + s[4]) * 0.25f : p.q[4] * 0.5f;
    r2 = (p.q[0] - r2) * 0.5f;
    r3 = (p.q[1] - r3) * 0.5f;
    r2 += r4 * d.y + r6 * d.x;
    r3 += r6 * d.y + r5 * d.x;
    const float c2 = r2 * sc, c3 = r3 * sc, c4 = r4 * sc, c5 = r5 * sc, c6 = r6 * sc;
    m[0] = c4 * c4 + c6 * c6;
    m[1] = (c4 + c5) * c6;
    m[2] = c5 * c5 + c6 * c6;
    m[3] = c4 * c2 + c6 * c3;
    m[4] = c6 * c2 + c5 * c3;
}

// The regularised 2 x 2 solve of one pixel's box sums.
__device__ __forceinline__ float2 solve_flow(float s0, float s1, float s2, float s3, float s4,
                                             double scale) {
    const double g11 = s0 * scale, g12 = s1 * scale, g22 = s2 * scale;
    const double h1 = s3 * scale, h2 = s4 * scale;
    const double idet = 1.0 / (g11 * g22 - g12 * g12 + 1e-3);
    return make_float2((float)((g11 * h2 - g12 * h1) * idet),
                       (float)((g22 * h1 - g12 * h2) * idet));
}

// Some pairs of a level as the flow kernels see them: pair p of the launch is
// frames first_pair + p and the next; in, out and coarse count from the
// launch's first pair.
struct FlowArgs {
    const float* R;
    int first_pair, slots;  // frame f's expansion is in slot f % slots of R
    int w, h;
    int tiles_x, tiles;    // strips across, strips per pair (flow_step_kernel)
    int tw, rows;          // their columns and rows
    const float2* in;
    const float2* coarse;
    int cw, ch;
    double cx_scale, cy_scale;
    float mul;
    double box_scale;
    float2* out;
};

__device__ __forceinline__ Expansion frame_expansion(const FlowArgs& a, int i) {
    const long P = (long)a.w * a.h;
    return expansion(a.R + (long)((a.first_pair + i) % a.slots) * 5 * P, a.w, a.h);
}

// Initial flow of a level: zero, or the coarser level's flow.
__global__ __launch_bounds__(256) void init_flow_kernel(FlowArgs a) {
    const long P = (long)a.w * a.h;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const int p = blockIdx.y;
    if (i >= P) return;
    float2 d = make_float2(0.f, 0.f);
    if (a.coarse) {
        const int y = (int)(i / a.w), x = (int)(i - (long)y * a.w);
        int xa, xb, ya, yb;
        float wx, wy;
        linear_tap(x, a.cx_scale, a.cw, xa, xb, wx);
        linear_tap(y, a.cy_scale, a.ch, ya, yb, wy);
        d = coarse_flow(a.coarse + (long)p * a.cw * a.ch, a.cw, xa, xb, wx, ya, yb, wy, a.mul);
    }
    a.out[(long)p * P + i] = d;
}

// Matrices to HBM (M fp32 [pairs][5][h*w]) for the window sizes that
// flow_step_kernel does not take.
__global__ __launch_bounds__(256) void update_matrices_kernel(FlowArgs a, float* __restrict__ M) {
    const long P = (long)a.w * a.h;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const int p = blockIdx.y;
    if (i >= P) return;
    const int y = (int)(i / a.w), x = (int)(i - (long)y * a.w);
    const float2 d = a.in[(long)p * P + i];
    PixelSamples s;
    load_samples(frame_expansion(a, p), frame_expansion(a, p + 1), a.w, a.h, x, y, d, s);
    float m[5];
    pixel_matrices(s, a.w, a.h, x, y, d, axis_weight(x, a.w) * axis_weight(y, a.h), m);
    float* Mp = M + (long)p * 5 * P + i;
#pragma unroll
    for (int c = 0; c < 5; ++c) Mp[c * P] = m[c];
}

// One whole iteration for winsize 15: the matrices, their box sums and the
// solve of one strip of columns, without the matrices going to HBM (as separate
// launches they cost 20 B per pixel written and 27 B read back).
//
// A workgroup owns tw (a multiple of 4, <= kFsCols - 14) output columns and
// a.rows = 15 k + 1 output rows, and rolls down them in batches of 15 rows of
// matrices (replicated border):
//   1. samples: the 15 x (tw + 14) matrices of a batch, 3 per thread at the
//      same places of every batch; the next batch's flows are loaded a batch
//      ahead, and two samples' loads are in flight at a time;
//   2. column sums: a thread owns one column of one of the 5 matrix planes for
//      the whole strip, its fp64 running sum and the 15 rows of its window in
//      registers (15 rows a batch make the ring's slots static), and replaces
//      each row's value in LDS by the sum of the 15 rows that end there;
//   3. row sums of 4 neighbouring pixels and their solve, 7 rows behind.
// 8 waves of 128 registers: two workgroups share a CU, one's samples under the
// other's sums (10 waves of 96 registers, which need an uneven 3 + 2 waves on a
// SIMD, ran alone: 64 us instead of 54 us at 10 pairs of 832x480).
// Two LDS buffers, so that a batch's samples need not wait for the last
// batch's solves.
//
// Bound by the L1's gather rate and the VALU rather than by memory: 5.0 us an
// iteration and pair of 832x480 in a 50-frame clip, where matrix update and box
// filter launches took 8.3 us.
// kZero: the current flow is zero (the first iteration of the coarsest level).
template <bool kZero>
__global__ __launch_bounds__(kFsThreads, 4) void flow_step_kernel(FlowArgs a) {
    constexpr int kWin = 2 * kFsHalf + 1;
    constexpr int kPitch = (kFsCols + 3) / 4 * 4;
    static_assert(kWin == 15 && 5 * kFsCols <= kFsThreads && kWin * kFsCols <= 3 * kFsThreads &&
                      32 * kWin <= kFsThreads && kFsCols <= 4 * 32,
                  "3 samples, one plane column and one run of 4 pixels per thread");
    __shared__ __attribute__((aligned(16))) float m[2][5][kWin][kPitch];
    // each XCD takes a contiguous run of strips, so that what neighbouring
    // strips share is fetched into one L2
    int b = xcd_contiguous((int)blockIdx.x, (int)gridDim.x);
    const int p = b / a.tiles;
    b -= p * a.tiles;
    const int X0 = (b % a.tiles_x) * a.tw, Y0 = (b / a.tiles_x) * a.rows;
    const int w = a.w, h = a.h;
    const long P = (long)w * h;
    const Expansion R0 = frame_expansion(a, p), R1 = frame_expansion(a, p + 1);
    const int tid = threadIdx.x;
    const int cols = a.tw + 2 * kFsHalf;
    // this thread's samples: row of the batch and column (the last threads
    // repeat the last sample), and the border weight of the column
    int sr[3], sc[3];
    float sw[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int i = min(tid + u * kFsThreads, kWin * cols - 1);
        sr[u] = i / cols;
        sc[u] = i - sr[u] * cols;
        const int x = min(max(X0 - kFsHalf + sc[u], 0), w - 1);
        sw[u] = axis_weight(x, w);
    }
    const __amdgpu_buffer_rsrc_t in_rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float2*>(kZero ? nullptr : a.in + (long)p * P), (short)0,
        kZero ? 0 : (int)(P * 8), 0x00020000);
    auto col_of = [&](int u) { return min(max(X0 - kFsHalf + sc[u], 0), w - 1); };
    auto row_of = [&](int e0, int u) { return min(max(e0 + sr[u], 0), h - 1); };
    auto load_flow = [&](int x, int y) {
        if constexpr (kZero) return make_float2(0.f, 0.f);
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(in_rs, 8 * (y * w + x), 0, 0);
        return make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
    };
    const int yend = min(Y0 + a.rows, h);
    // sums: window ring and running sum of plane tid / kFsCols, column
    // tid % kFsCols
    float ring[kWin];
#pragma unroll
    for (int r = 0; r < kWin; ++r) ring[r] = 0.f;
    double vs = 0.0;
    float* own = &m[0][0][0][0] + tid / kFsCols * kWin * kPitch + tid % kFsCols;
    float2 d[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) d[u] = load_flow(col_of(u), row_of(Y0 - kFsHalf, u));
    float2* out = a.out + (long)p * P;
    int buf = 0;
    // batch e0: matrix rows e0 .. e0 + 14 enter, output rows e0 - 7 .. e0 + 7
    for (int e0 = Y0 - kFsHalf; e0 - kFsHalf < yend; e0 += kWin, buf ^= 1) {
        // rows within the down-weighted border of the image in this batch
        const bool edge = e0 < kBorder || e0 + kWin > h - kBorder;
        PixelSamples s[2];
        auto start = [&](int u) {
            load_samples(R0, R1, w, h, col_of(u), row_of(e0, u), d[u], s[u & 1]);
        };
        auto finish = [&](int u) {
            const int x = col_of(u), y = row_of(e0, u);
            float v[5];
            pixel_matrices(s[u & 1], w, h, x, y, d[u], edge ? sw[u] * axis_weight(y, h) : sw[u], v);
#pragma unroll
            for (int q = 0; q < 5; ++q) m[buf][q][sr[u]][sc[u]] = v[q];
            d[u] = load_flow(x, row_of(e0 + kWin, u));
        };
        // (the fences keep the compiler from issuing more loads than fit)
        start(0);
        start(1);
        asm volatile("" ::: "memory");
        finish(0);
        start(2);
        asm volatile("" ::: "memory");
        finish(1);
        finish(2);
        __syncthreads();
        if (tid < 5 * kFsCols) {
            float* c = own + buf * 5 * kWin * kPitch;
#pragma unroll
            for (int r = 0; r < kWin; ++r) {
                const float e = c[r * kPitch];
                vs += (double)e - (double)ring[r];
                ring[r] = e;
                c[r * kPitch] = (float)vs;
            }
        }
        __syncthreads();
        const int r = tid >> 5, c0 = 4 * (tid & 31);
        const int y = e0 - kFsHalf + r, xo = X0 + c0;
        if (r < kWin && y >= Y0 && y < yend && c0 < a.tw && xo < w) {
            float s4[5][4];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                float v[20];
#pragma unroll
                for (int q = 0; q < 5; ++q) {
                    const float4 t = *reinterpret_cast<const float4*>(&m[buf][k][r][c0 + 4 * q]);
                    v[4 * q] = t.x;
                    v[4 * q + 1] = t.y;
                    v[4 * q + 2] = t.z;
                    v[4 * q + 3] = t.w;
                }
                // columns 3 .. 14 belong to all four windows
                float mid = v[3];
#pragma unroll
                for (int q = 4; q < kWin; ++q) mid += v[q];
                s4[k][0] = mid + ((v[0] + v[1]) + v[2]);
                s4[k][1] = mid + ((v[1] + v[2]) + v[kWin]);
                s4[k][2] = mid + ((v[2] + v[kWin]) + v[kWin + 1]);
                s4[k][3] = mid + ((v[kWin] + v[kWin + 1]) + v[kWin + 2]);
            }
            float2* o = out + (long)y * w + xo;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (xo + q < w)
                    o[q] = solve_flow(s4[0][q], s4[1][q], s4[2][q], s4[3][q], s4[4][q],
                                      a.box_scale);
        }
    }
}

// One workgroup = a strip of COLS - 2m output columns (COLS loaded columns
// with the halo, one thread each) and `rows` output rows. Each thread keeps
// fp64 running vertical sums of the 5 planes for its column (the entering
// row added, the leaving row subtracted, replicated border) and parks them
// in LDS for kBfBatch rows at a time; then each thread turns a run of
// kBfRun columns of one parked row into box sums with a sliding horizontal
// sum and solves those pixels.
template <int COLS>
__global__ __launch_bounds__(COLS) void update_flow_kernel(const float* __restrict__ M, int w,
                                                           int h, int m, int rows, double scale,
                                                           float2* __restrict__ flow) {
    __shared__ float buf[kBfBatch][5][COLS];
    const int tw = COLS - 2 * m;
    const int X0 = blockIdx.x * tw;
    const int Y0 = blockIdx.y * rows;
    const int p = blockIdx.z;
    const long P = (long)w * h;
    const float* Mp = M + (long)p * 5 * P;
    float2* Fp = flow + (long)p * P;
    const int tid = threadIdx.x;
    const int xc = min(max(X0 - m + tid, 0), w - 1);
    double vs[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int r = Y0 - m; r <= Y0 + m; ++r) {
        const float* q = Mp + (long)min(max(r, 0), h - 1) * w + xc;
#pragma unroll
        for (int c = 0; c < 5; ++c) vs[c] += q[c * P];
    }
    const int yend = min(Y0 + rows, h);
    const int xend = min(tw, w - X0);                 // output columns of this strip
    const int runs = (xend + kBfRun - 1) / kBfRun;
    for (int yb = Y0; yb < yend; yb += kBfBatch) {
        const int nr = min(kBfBatch, yend - yb);
#pragma unroll
        for (int r = 0; r < kBfBatch; ++r) {
            if (r < nr) {
#pragma unroll
                for (int c = 0; c < 5; ++c) buf[r][c][tid] = (float)vs[c];
                const int y = yb + r;
                if (y + 1 < yend) {
                    const float* qa = Mp + (long)min(y + m + 1, h - 1) * w + xc;
                    const float* qs = Mp + (long)max(y - m, 0) * w + xc;
#pragma unroll
                    for (int c = 0; c < 5; ++c) vs[c] += (double)qa[c * P] - (double)qs[c * P];
                }
            }
        }
        __syncthreads();
        for (int j = tid; j < nr * runs; j += COLS) {
            const int r = j / runs;
            const int x0 = (j - r * runs) * kBfRun;
            const int n = min(kBfRun, xend - x0);
            float s[5][kBfRun];
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                const float* v = &buf[r][c][x0];
                float a = 0.f;
                for (int k = 0; k <= 2 * m; ++k) a += v[k];
                s[c][0] = a;
#pragma unroll
                for (int i = 1; i < kBfRun; ++i) {
                    if (i < n) a += v[i + 2 * m] - v[i - 1];
                    s[c][i] = a;
                }
            }
            float2* out = Fp + (long)(yb + r) * w + X0 + x0;
#pragma unroll
            for (int i = 0; i < kBfRun; ++i) {
                if (i < n)
                    out[i] = solve_flow(s[0][i], s[1][i], s[2][i], s[3][i], s[4][i], scale);
            }
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void flow_cells_kernel(const float2* __restrict__ flow, int W,
                                                         int H, int rows, int cols,
                                                         float* __restrict__ cells) {
    __shared__ float colsum[kMaxSide];
    const int r = blockIdx.x, p = blockIdx.y;
    const int ch = H / rows, cw = W / cols;
    const float2* F = flow + (long)p * W * H + (long)r * ch * W;
    if ((W & 1) == 0 && (((uintptr_t)F) & 15) == 0) {
        const float4* F4 = reinterpret_cast<const float4*>(F);   // 2 pixels per load
        const int W2 = W / 2;
        for (int x2 = threadIdx.x; x2 < W2; x2 += 256) {
            float s0 = 0.f, s1 = 0.f;
#pragma unroll 4
            for (int yy = 0; yy < ch; ++yy) {
                const float4 d = F4[(long)yy * W2 + x2];
                s0 += sqrtf(d.x * d.x + d.y * d.y);
                s1 += sqrtf(d.z * d.z + d.w * d.w);
            }
            colsum[2 * x2] = s0;
            colsum[2 * x2 + 1] = s1;
        }
    } else {
        for (int x = threadIdx.x; x < W; x += 256) {
            float s = 0.f;
            for (int yy = 0; yy < ch; ++yy) {
                const float2 d = F[(long)yy * W + x];
                s += sqrtf(d.x * d.x + d.y * d.y);
            }
            colsum[x] = s;
        }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < cols; c += 256) {
        float s = 0.f;
        for (int k = 0; k < cw; ++k) s += colsum[c * cw + k];
        cells[((long)p * rows + r) * cols + c] = s / (float)(ch * cw);
    }
}

__global__ __launch_bounds__(256) void tile_change_kernel(const float* __restrict__ cells,
                                                          int pairs, int tokens, int tile_tokens,
                                                          int tiles, double* __restrict__ change) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long)pairs * tiles) return;
    const int p = (int)(i / tiles), t = (int)(i - (long)p * tiles);
    const int b = t * tile_tokens, e = min(b + tile_tokens, tokens);
    double s = 0.0;
    for (int k = b; k < e; ++k) s += (double)cells[(long)p * tokens + k];
    change[i] = s / (double)(e - b);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

int launch_ok(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return 1;
    }
    return 0;
}

int round_half_even(double v) { return (int)std::nearbyint(v); }

struct Level {
    int k;
    double scale, sigma;
    int ksize, w, h;
};

// Levels from the coarsest to the full size (OpenCV: stop at the first
// scale where a side falls under 32 pixels).
std::vector<Level> level_plan(int W, int H, double pyr_scale, int levels) {
    double scale = 1.0;
    int k = 0;
    while (k < levels) {
        scale *= pyr_scale;
        if (W * scale < kMinLevelSide || H * scale < kMinLevelSide) break;
        ++k;
    }
    std::vector<Level> plan;
    for (int lv = k; lv >= 0; --lv) {
        double s = 1.0;
        for (int i = 0; i < lv; ++i) s *= pyr_scale;
        const double sigma = (1.0 / s - 1.0) * 0.5;
        int ksize = round_half_even(sigma * 5) | 1;
        if (ksize < 3) ksize = 3;
        plan.push_back({lv, s, sigma, ksize, round_half_even(W * s), round_half_even(H * s)});
    }
    return plan;
}

// getGaussianKernel(ksize, sigma) for fp32 images: the fixed binomial-like
// tables for ksize <= 7 and sigma <= 0, else normalised exp(-x^2 / 2 sigma^2).
bool blur_taps(int ksize, double sigma, BlurTaps& t) {
    if (ksize > kMaxBlurTaps) return false;
    t.ksize = ksize;
    static const float small[4][7] = {
        {1.f},
        {0.25f, 0.5f, 0.25f},
        {0.0625f, 0.25f, 0.375f, 0.25f, 0.0625f},
        {0.03125f, 0.109375f, 0.21875f, 0.28125f, 0.21875f, 0.109375f, 0.03125f}};
    if (sigma <= 0 && (ksize & 1) && ksize <= 7) {
        for (int i = 0; i < ksize; ++i) t.k[i] = small[ksize >> 1][i];
        return true;
    }
    if (sigma <= 0) sigma = ((ksize - 1) * 0.5 - 1) * 0.3 + 0.8;
    std::vector<double> v(ksize);
    double sum = 0;
    for (int i = 0; i < ksize; ++i) {
        const double x = i - (ksize - 1) * 0.5;
        v[i] = std::exp(-x * x / (2 * sigma * sigma));
        sum += v[i];
    }
    for (int i = 0; i < ksize; ++i) t.k[i] = (float)(v[i] / sum);
    return true;
}

// 6x6 Gauss-Jordan inverse with partial pivoting (the Gram matrix is SPD).
bool invert6(double a[6][6], double inv[6][6]) {
    for (int i = 0; i < 6; ++i)
        for (int j = 0; j < 6; ++j) inv[i][j] = i == j;
    for (int c = 0; c < 6; ++c) {
        int piv = c;
        for (int r = c + 1; r < 6; ++r)
            if (std::fabs(a[r][c]) > std::fabs(a[piv][c])) piv = r;
        if (a[piv][c] == 0) return false;
        for (int j = 0; j < 6; ++j) {
            std::swap(a[c][j], a[piv][j]);
            std::swap(inv[c][j], inv[piv][j]);
        }
        const double d = a[c][c];
        for (int j = 0; j < 6; ++j) {
            a[c][j] /= d;
            inv[c][j] /= d;
        }
        for (int r = 0; r < 6; ++r) {
            if (r == c) continue;
            const double f = a[r][c];
            for (int j = 0; j < 6; ++j) {
                a[r][j] -= f * a[c][j];
                inv[r][j] -= f * inv[c][j];
            }
        }
    }
    return true;
}

// Applicability taps and the inverse-Gram entries of the basis
// [1, x, y, x^2, y^2, xy] (FarnebackPrepareGaussian).
bool poly_taps(int n, double sigma, PolyTaps& t) {
    if (sigma < FLT_EPSILON) sigma = n * 0.3;
    t.n = n;
    double s = 0;
    for (int k = -n; k <= n; ++k) {
        t.g[k + n] = (float)std::exp(-k * k / (2 * sigma * sigma));
        s += t.g[k + n];
    }
    for (int k = -n; k <= n; ++k) {
        t.g[k + n] = (float)(t.g[k + n] / s);
        t.xg[k + n] = (float)(k * (double)t.g[k + n]);
        t.xxg[k + n] = (float)(k * k * (double)t.g[k + n]);
    }
    double G[6][6] = {};
    for (int y = -n; y <= n; ++y)
        for (int x = -n; x <= n; ++x) {
            const double gg = (double)t.g[y + n] * t.g[x + n];
            const double b[6] = {1.0, (double)x, (double)y, (double)x * x, (double)y * y,
                                 (double)x * y};
            for (int i = 0; i < 6; ++i)
                for (int j = 0; j < 6; ++j) G[i][j] += gg * b[i] * b[j];
        }
    double iG[6][6];
    if (!invert6(G, iG)) return false;
    t.ig11 = iG[1][1];
    t.ig03 = iG[0][3];
    t.ig33 = iG[3][3];
    t.ig55 = iG[5][5];
    return true;
}

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// Strips of flow_step_kernel for a level of w x h and n pairs: as few across as
// its columns allow, of equal width; of the heights 15 k + 1 the one whose
// batches (k + 1 a strip) times rounds of strips are fewest, the lower strips
// on a tie.
void flow_strips(int w, int h, int n, FlowArgs& a) {
    const int most = kFsCols - 2 * kFsHalf - (kFsCols - 2 * kFsHalf) % 4;
    a.tiles_x = (w + most - 1) / most;
    a.tw = ((w + a.tiles_x - 1) / a.tiles_x + 3) / 4 * 4;
    a.tiles_x = (w + a.tw - 1) / a.tw;
    long best = 0;
    for (int k = 1; k == 1 || 15 * (k - 1) + 1 < h; ++k) {
        const int rows = 15 * k + 1;
        const long strips = (long)a.tiles_x * ((h + rows - 1) / rows) * n;
        const long cost = (strips + kFsSlots - 1) / kFsSlots * (k + 1);
        if (k == 1 || cost < best) {
            best = cost;
            a.rows = rows;
            a.tiles = a.tiles_x * ((h + rows - 1) / rows);
        }
    }
}

// Pairs of a level taken at a time, in equal shares.
//
// flow_step_kernel (`step`): 17 x 832 x 480 pixels, whose expansions and two flow
// buffers (36 B per pixel) stay in the 256 MiB Infinity Cache from one iteration to
// the next. A chunk's last round of strips costs what that gains, or more on large
// frames: in chunks and in one launch, 50 frames of 832x480 1511 and 1504 us, 100 of
// 416x240 760 and 809, 100 of 832x480 3003 and 3063, 30 of 1920x1080 4875 and 4757,
// 12 of 3840x2160 7930 and 7080.
//
// Other windows: all pairs, but for clips whose full-size expansions and matrices
// (40 B a pixel and pair) would take more than 8.7 GB. Their matrices do not stay in
// the cache, and in short launches their blocks' rows are few for the window (their
// halo). 30 frames of 1920x1080 in chunks of 17 x 832 x 480 pixels and in one launch:
// window 9 6890 and 6259 us, 49 11753 and 9779; 20 of 832x480, window 33, 1492 and 1343.
int chunk_pairs(long pixels, int pairs, bool step) {
    const long cap = std::max<long>(1, (step ? kStepChunkPixels : kChunkPixels) / pixels);
    const long chunks = (pairs + cap - 1) / cap;
    return (int)((pairs + chunks - 1) / chunks);
}

// Workspace for any window: the reduced levels' images and expansions for all
// frames, the full-size level's expansions for one chunk of pairs, two flow buffers of the
// largest reduced level, and a region that holds either the matrices of a chunk
// or the second flow buffer of its iterations, whichever the window size needs.
struct Layout {
    std::vector<size_t> img, R;  // per plan entry
    size_t fa, fb, M, total;
};

Layout layout(int nf, int W, int H, const std::vector<Level>& plan) {
    const int pairs = nf - 1;
    size_t P1 = 0, most = 0;
    Layout L;
    size_t off = 0;
    auto take = [&](size_t floats) {
        const size_t at = off;
        off += align256(floats * sizeof(float));
        return at;
    };
    for (const Level& l : plan) {
        const size_t P = (size_t)l.w * l.h;
        const int chunk = chunk_pairs((long)P, pairs, false);  // the larger of the two
        L.img.push_back(l.k > 0 ? take(nf * P) : 0);
        L.R.push_back(take((l.k > 0 ? (size_t)nf : chunk + 1) * 5 * P));
        if (l.k > 0) P1 = std::max(P1, P);
        most = std::max(most, chunk * P);
    }
    L.fa = take(pairs * P1 * 2);
    L.fb = take(pairs * P1 * 2);
    L.M = take(5 * most);
    L.total = off;
    return L;
}

// launch kinds reported by kvp_farneback_profile
enum {
    KIND_PREBLUR = 1,
    KIND_POLY_EXP = 2,
    KIND_INIT_FLOW = 3,
    KIND_FLOW = 4,
    KIND_MATRICES = 5,
};

int check_params(int nf, int W, int H, double pyr_scale, int levels, int winsize,
                 int iterations, int poly_n, int flags) {
    if (nf < 2 || nf > kMaxFrames) {
        set_error("farneback: %d frames (2..%d)", nf, kMaxFrames);
        return 1;
    }
    if (W < kMinSide || H < kMinSide || W > kMaxSide || H > kMaxSide) {
        set_error("farneback: frame %dx%d outside %d..%d per side", W, H, kMinSide, kMaxSide);
        return 1;
    }
    if (!(pyr_scale > 0 && pyr_scale < 1)) {
        set_error("farneback: pyr_scale %g must be in (0, 1)", pyr_scale);
        return 1;
    }
    if (levels < 0 || iterations < 0) {
        set_error("farneback: levels and iterations must be >= 0");
        return 1;
    }
    if (winsize < 1 || winsize / 2 > kMaxBoxHalf) {
        set_error("farneback: winsize %d outside 1..%d", winsize, 2 * kMaxBoxHalf + 1);
        return 1;
    }
    if (poly_n < 1 || poly_n > kMaxPolyN) {
        set_error("farneback: poly_n %d outside 1..%d", poly_n, kMaxPolyN);
        return 1;
    }
    if (flags != 0) {
        set_error("farneback: flags %d not supported (only 0: zero initial flow, box window)",
                  flags);
        return 1;
    }
    return 0;
}

// Launch timeline for kvp_farneback_profile: an event after every launch. A step
// is one kernel's work of one level and iteration; a clip taken in chunks makes
// several launches of a step, which share its entry, so that the entries of a
// clip do not grow with its length.
struct Timeline {
    struct Step {
        int kind, level, iteration;
        float ms;
    };
    hipStream_t st;
    std::vector<hipEvent_t> ev;  // the first one before the first launch
    std::vector<size_t> step_of;  // of launch i, between events i and i + 1
    std::vector<Step> steps;
    bool ok = true;
    void record() {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) {
            ok = false;
            return;
        }
        if (hipEventRecord(e, st) != hipSuccess) ok = false;
        ev.push_back(e);
    }
    void launched(int kind, int level, int iteration) {
        record();
        size_t i = 0;
        while (i < steps.size() && !(steps[i].kind == kind && steps[i].level == level &&
                                     steps[i].iteration == iteration))
            ++i;
        if (i == steps.size()) steps.push_back({kind, level, iteration, 0.f});
        step_of.push_back(i);
    }
    // waits for the launches and sums their times; false if an event failed
    bool sum() {
        if (!ok || ev.empty() || hipEventSynchronize(ev.back()) != hipSuccess) return false;
        for (size_t i = 0; i < step_of.size(); ++i) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, ev[i], ev[i + 1]) != hipSuccess) return false;
            steps[step_of[i]].ms += ms;
        }
        return true;
    }
    ~Timeline() {
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
    }
};

int farneback_impl(const uint8_t* frames, long frame_stride, int nf, int W, int H,
                   double pyr_scale, int levels, int winsize, int iterations, int poly_n,
                   double poly_sigma, int flags, void* workspace, long workspace_bytes,
                   float* flows, void* stream_v, Timeline* tl = nullptr) {
    if (check_params(nf, W, H, pyr_scale, levels, winsize, iterations, poly_n, flags)) return 1;
    if (!frames || !flows || !workspace) {
        set_error("farneback: null pointer");
        return 1;
    }
    const std::vector<Level> plan = level_plan(W, H, pyr_scale, levels);
    const Layout L = layout(nf, W, H, plan);
    if (workspace_bytes < 0 || (size_t)workspace_bytes < L.total) {
        set_error("farneback: workspace %ld bytes < %zu needed", workspace_bytes, L.total);
        return 1;
    }
    PolyTaps pt;
    if (!poly_taps(poly_n, poly_sigma, pt)) {
        set_error("farneback: singular applicability (poly_n %d, poly_sigma %g)", poly_n,
                  poly_sigma);
        return 1;
    }
    for (const Level& l : plan) {
        if (l.ksize > kMaxBlurTaps) {
            set_error("farneback: level %d needs a %d-tap pre-blur (max %d)", l.k, l.ksize,
                      kMaxBlurTaps);
            return 1;
        }
    }
    hipStream_t st = (hipStream_t)stream_v;
    char* ws = (char*)workspace;
    float* M = (float*)(ws + L.M);
    float2* fbuf[2] = {(float2*)(ws + L.fa), (float2*)(ws + L.fb)};
    const int pairs = nf - 1;
    const int m = winsize / 2;
    const bool step = m == kFsHalf && iterations > 0;  // flow_step_kernel
    std::vector<int> chunk;  // per plan entry
    for (const Level& l : plan) chunk.push_back(chunk_pairs((long)l.w * l.h, pairs, step));
    const double box_scale = 1.0 / ((double)winsize * winsize);

    auto mark = [&](int kind, int lv, int iteration = 0) {
        if (tl) tl->launched(kind, lv, iteration);
    };
    if (tl) tl->record();

    // Image and expansion of frames [f0, f0 + n) on plan levels [l0, l1), as
    // one launch each (more only past kPyrLevels levels or kPyrTaps taps).
    auto pyramid = [&](size_t l0, size_t l1, int f0, int n) {
        while (l0 < l1) {
            PyrArgs blur = {}, poly = {};
            blur.W = W;
            blur.H = H;
            blur.src = frames;
            blur.frame_stride = frame_stride;
            blur.base = (float*)ws;
            blur.first_frame = f0;
            poly = blur;
            int blur_blocks = 0, poly_blocks = 0, taps = 0;
            size_t lds = 0;
            int blur_level = 0, lo_level = 0;  // the lowest level of each launch
            for (; l0 < l1 && poly.levels < kPyrLevels; ++l0) {
                const Level& l = plan[l0];
                if (l.k > 0 && taps + l.ksize > kPyrTaps) break;
                lo_level = l.k;
                PyrLevel v = {};
                v.w = l.w;
                v.h = l.h;
                if (l.k > 0) {
                    BlurTaps bt;
                    blur_taps(l.ksize, l.sigma, bt);
                    v.sx = 1.0 / ((double)l.w / W);
                    v.sy = 1.0 / ((double)l.h / H);
                    v.ksize = l.ksize;
                    v.tap0 = taps;
                    for (int i = 0; i < l.ksize; ++i) blur.taps[taps++] = bt.k[i];
                    v.img = (long)(L.img[l0] / sizeof(float));
                    // x-blurred rows one block's level rows reach, and the
                    // source bytes under them (staged where both fit)
                    auto reach = [&](int th) {
                        return (size_t)((int)((th - 1) * v.sy) + 3 + l.ksize);
                    };
                    auto bytes = [&](int th) { return reach(th) * 2 * kPbTileW * sizeof(float); };
                    v.tile_h = std::max(1, (int)(kPbRows / v.sy + 0.5));
                    const size_t staged =
                        reach(v.tile_h) * ((size_t)((kPbTileW - 1) * v.sx) + 3 + l.ksize + 8);
                    if (bytes(v.tile_h) + staged <= kPbLdsBytes) {
                        v.stage_at = (int)bytes(v.tile_h);
                        lds = std::max(lds, bytes(v.tile_h) + staged);
                    } else {
                        while (v.tile_h > 1 && bytes(v.tile_h) > kPbLdsBytes) v.tile_h /= 2;
                        lds = std::max(lds, bytes(v.tile_h));
                    }
                    v.tiles_x = (l.w + kPbTileW - 1) / kPbTileW;
                    v.first_block = blur_blocks;
                    blur_blocks += v.tiles_x * ((l.h + v.tile_h - 1) / v.tile_h);
                    blur.lv[blur.levels++] = v;
                    blur_level = l.k;
                } else {
                    v.img = -1;
                }
                v.R = (long)(L.R[l0] / sizeof(float));
                v.slots = l.k > 0 ? nf : chunk[l0] + 1;
                v.tiles_x = (l.w + kPeTileW - 1) / kPeTileW;
                v.first_block = poly_blocks;
                poly_blocks += v.tiles_x * ((l.h + kPeTileH - 1) / kPeTileH);
                poly.lv[poly.levels++] = v;
            }
            if (blur_blocks) {
                preblur_kernel<<<dim3(blur_blocks, 1, n), 256, lds, st>>>(blur);
                mark(KIND_PREBLUR, blur_level);
            }
            if (poly_n == 5)
                poly_exp_kernel<5><<<dim3(poly_blocks, 1, n), kPeThreads, 0, st>>>(poly, pt);
            else
                poly_exp_kernel<0><<<dim3(poly_blocks, 1, n), kPeThreads, 0, st>>>(poly, pt);
            mark(KIND_POLY_EXP, lo_level);
        }
        return launch_ok("farneback pyramid");
    };

    // The full-size level (the last of the plan) is expanded chunk by chunk,
    // or with the others where one chunk holds every pair.
    const size_t last = plan.size() - 1;
    const bool whole = chunk[last] >= pairs;
    if (pyramid(0, whole ? last + 1 : last, 0, nf)) return 1;

    // Iterations of plan level li for pairs [p0, p0 + n).
    auto iterate = [&](size_t li, int p0, int n) {
        const Level& l = plan[li];
        const long P = (long)l.w * l.h;
        float2* fl = (l.k == 0 ? (float2*)flows : fbuf[li & 1]) + p0 * P;
        const float2* prev =
            li > 0 ? fbuf[(li - 1) & 1] + (long)p0 * plan[li - 1].w * plan[li - 1].h : nullptr;
        FlowArgs a = {};
        a.R = (const float*)(ws + L.R[li]);
        a.first_pair = p0;
        a.slots = l.k > 0 ? nf : chunk[li] + 1;
        a.w = l.w;
        a.h = l.h;
        a.box_scale = box_scale;
        a.mul = (float)(1.0 / pyr_scale);
        if (prev) {
            a.coarse = prev;
            a.cw = plan[li - 1].w;
            a.ch = plan[li - 1].h;
            a.cx_scale = 1.0 / ((double)l.w / a.cw);
            a.cy_scale = 1.0 / ((double)l.h / a.ch);
        }
        const dim3 pix((unsigned)((P + 255) / 256), n);
        if (step) {
            // iteration i writes what i + 1 reads: two buffers in turn, the
            // last one fl
            float2* other = (float2*)M;
            flow_strips(l.w, l.h, n, a);
            const dim3 grid((unsigned)(a.tiles * n));
            for (int it = 0; it < iterations; ++it) {
                a.out = (iterations - 1 - it) % 2 ? other : fl;
                float2* in = (iterations - 1 - it) % 2 ? fl : other;
                a.in = in;
                if (it == 0 && prev) {
                    FlowArgs c = a;
                    c.out = in;
                    init_flow_kernel<<<pix, 256, 0, st>>>(c);
                    mark(KIND_INIT_FLOW, l.k);
                }
                if (it == 0 && !prev)
                    flow_step_kernel<true><<<grid, kFsThreads, 0, st>>>(a);
                else
                    flow_step_kernel<false><<<grid, kFsThreads, 0, st>>>(a);
                mark(KIND_FLOW, l.k, it);
            }
            return launch_ok("farneback iterations");
        }
        a.in = fl;
        a.out = fl;
        init_flow_kernel<<<pix, 256, 0, st>>>(a);
        mark(KIND_INIT_FLOW, l.k);
        // narrow levels take 128-column strips; rows per workgroup (a multiple
        // of the LDS batch, 8..32) so that a launch has ~kBfTargetGroups groups
        const bool narrow = l.w + 2 * m <= 128 || l.w < 400;
        const int cols = narrow ? 128 : 256;
        const int strips = (l.w + cols - 2 * m - 1) / (cols - 2 * m);
        const long want = ((long)l.h * strips * n + kBfTargetGroups - 1) / kBfTargetGroups;
        int rows = (int)std::min<long>(32, std::max<long>(kBfBatch, want));
        rows = (rows + kBfBatch - 1) / kBfBatch * kBfBatch;
        const dim3 box_grid(strips, (l.h + rows - 1) / rows, n);
        for (int it = 0; it < iterations; ++it) {
            update_matrices_kernel<<<pix, 256, 0, st>>>(a, M);
            mark(KIND_MATRICES, l.k, it);
            if (narrow)
                update_flow_kernel<128><<<box_grid, 128, 0, st>>>(M, l.w, l.h, m, rows, box_scale,
                                                                   fl);
            else
                update_flow_kernel<256><<<box_grid, 256, 0, st>>>(M, l.w, l.h, m, rows, box_scale,
                                                                   fl);
            mark(KIND_FLOW, l.k, it);
        }
        return launch_ok("farneback iterations");
    };

    for (size_t li = 0; li <= last; ++li) {
        for (int p0 = 0; p0 < pairs; p0 += chunk[li]) {
            const int n = std::min(chunk[li], pairs - p0);
            // a later chunk's first frame is the last of the chunk before it
            const int f0 = p0 == 0 ? 0 : p0 + 1;
            if (li == last && !whole && pyramid(last, last + 1, f0, p0 + n + 1 - f0)) return 1;
            if (iterate(li, p0, n)) return 1;
        }
    }
    return 0;
}

}  // namespace
}  // namespace kvp

extern "C" {

long kvp_farneback_workspace_bytes(int num_frames, int width, int height, double pyr_scale,
                                   int levels) {
    if (num_frames < 2 || width < 1 || height < 1 || !(pyr_scale > 0 && pyr_scale < 1) ||
        levels < 0)
        return -1;
    return (long)kvp::layout(num_frames, width, height,
                             kvp::level_plan(width, height, pyr_scale, levels))
        .total;
}

int kvp_farneback_flows(const unsigned char* frames, int num_frames, int width, int height,
                        double pyr_scale, int levels, int winsize, int iterations, int poly_n,
                        double poly_sigma, int flags, void* workspace, long workspace_bytes,
                        float* flows, void* stream) {
    return kvp::farneback_impl(frames, (long)width * height, num_frames, width, height,
                               pyr_scale, levels, winsize, iterations, poly_n, poly_sigma, flags,
                               workspace, workspace_bytes, flows, stream);
}

int kvp_farneback_flow(const unsigned char* prev, const unsigned char* next, float* flow,
                       int width, int height, double pyr_scale, int levels, int winsize,
                       int iterations, int poly_n, double poly_sigma, int flags, void* workspace,
                       long workspace_bytes, void* stream) {
    if (!prev || !next) {
        kvp::set_error("farneback: null frame");
        return 1;
    }
    const long stride = (long)((intptr_t)next - (intptr_t)prev);
    return kvp::farneback_impl(prev, stride, 2, width, height, pyr_scale, levels, winsize,
                               iterations, poly_n, poly_sigma, flags, workspace, workspace_bytes,
                               flow, stream);
}

int kvp_farneback_profile(const unsigned char* frames, int num_frames, int width, int height,
                          double pyr_scale, int levels, int winsize, int iterations, int poly_n,
                          double poly_sigma, int flags, void* workspace, long workspace_bytes,
                          float* flows, float* launch_ms, int* launch_kind, int* launch_level,
                          int capacity, int* count, void* stream) {
    if (!launch_ms || !launch_kind || !launch_level || !count) {
        kvp::set_error("farneback_profile: null output array");
        return 1;
    }
    kvp::Timeline tl;
    tl.st = (hipStream_t)stream;
    const int rc = kvp::farneback_impl(frames, (long)width * height, num_frames, width, height,
                                       pyr_scale, levels, winsize, iterations, poly_n,
                                       poly_sigma, flags, workspace, workspace_bytes, flows,
                                       stream, &tl);
    if (rc) return rc;
    if (!tl.sum()) {
        kvp::set_error("farneback_profile: event timing failed");
        return 1;
    }
    const int n = (int)tl.steps.size();
    *count = n;
    if (n > capacity) {
        kvp::set_error("farneback_profile: %d steps > capacity %d", n, capacity);
        return 1;
    }
    for (int i = 0; i < n; ++i) {
        launch_ms[i] = tl.steps[i].ms;
        launch_kind[i] = tl.steps[i].kind;
        launch_level[i] = tl.steps[i].level;
    }
    return 0;
}

int kvp_motion_change_rates(const float* flows, int pairs, int width, int height, int grid_rows,
                            int grid_cols, int tile_tokens, float* cell_maps, double* change,
                            void* stream) {
    if (!flows || !cell_maps || !change) {
        kvp::set_error("change_rates: null pointer");
        return 1;
    }
    if (pairs < 1 || grid_rows < 1 || grid_cols < 1 || tile_tokens < 1 || width > kvp::kMaxSide ||
        height > kvp::kMaxSide || pairs > 65535) {
        kvp::set_error("change_rates: bad sizes");
        return 1;
    }
    if (width % grid_cols || height % grid_rows) {
        kvp::set_error("change_rates: grid %dx%d does not divide %dx%d", grid_rows, grid_cols,
                       width, height);
        return 1;
    }
    hipStream_t st = (hipStream_t)stream;
    kvp::flow_cells_kernel<<<dim3(grid_rows, pairs), 256, 0, st>>>(
        (const float2*)flows, width, height, grid_rows, grid_cols, cell_maps);
    const int tokens = grid_rows * grid_cols;
    const int tiles = (tokens + tile_tokens - 1) / tile_tokens;
    const long n = (long)pairs * tiles;
    kvp::tile_change_kernel<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(
        cell_maps, pairs, tokens, tile_tokens, tiles, change);
    return kvp::launch_ok("change_rates");
}

}  // extern "C"
