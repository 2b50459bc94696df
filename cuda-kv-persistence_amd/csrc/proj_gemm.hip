// Grouped projection GEMM for the K/V producer, gfx950 (CDNA4).
//
//   out_g[r, n] = sum_k x[r, k] * w[g*Ng + n, k] + bias[g*Ng + n]  (+ out_g[r, n])
//
// for groups g < G, with x [rows, K] and w [G*Ng, K] bf16 or fp32 row-major
// (both K-contiguous), bias fp32, out_g [rows, Ng] bf16 or fp32 (fp32 may
// accumulate into itself: the residual add of out_proj; fp32 operands give
// fp32 outputs). One launch covers every group, so the three q/k/v projections
// of a DiT block (reference: src/backbone.py:13,18-19) run as one grid written
// straight to three token-major outputs, and out_proj (src/backbone.py:22,
// 32-33) adds into the fp32 residual stream in its epilogue.
//
// Two tilings share the operand layout below: 128 features x 128 tokens (four
// waves, two workgroups per CU), and, for bf16 operands, 256 features x 256 or
// 320 tokens (eight waves, one workgroup per CU). choose_tile says which.
//
// Common structure:
//   wave (wn, wr) of a workgroup owns 64 features x 32 * JR tokens as 2 x JR
//   blocks of 32x32 accumulated by v_mfma_f32_32x32x16_bf16 with A = w rows
//   (features), B = x rows (tokens): lane l holds token (l % 32) of a block
//   and features 8*(v/4) + 4*(l/32) + v%4 in accumulator register v.
//   K advances in chunks of 128 bytes per row: both operand chunks arrive by
//   buffer loads straight into a two-stage LDS ring, 16-byte pieces
//   XOR-swizzled by ((row >> 1) & 7) so that the fragment reads
//   (ds_read_b128, 16 rows per read phase) hit distinct banks. Fragments are
//   read one k-step ahead of their MFMAs.
//   The accumulators start at the bias. Epilogue: each wave stages its
//   outputs (converted to the output type) 32 tokens at a time in LDS as
//   token rows, then writes them (and, when accumulating, reads the
//   residual) as full 16-byte lanes along token rows, so global accesses are
//   row-contiguous.
//   Workgroups are numbered in bands of 4 token tiles x all feature tiles
//   (feature tile fastest within a band column) and remapped so that each XCD
//   receives a contiguous range: the workgroups resident on one XCD share a
//   few token tiles and a run of weight tiles through its L2.
//
// Token rows past `rows` read as zeros (buffer bounds) and are not stored.
// Requirements (checked on the host): K % 64 == 0 (fp32 operands: K % 32),
// Ng % 128 == 0, 16-byte aligned operands.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kvp_internal.h"

namespace kvp {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

constexpr int kPThreads = 256;
constexpr int kPSmall = 128;   // features and tokens per tile (small-tile kernel)
constexpr int kPChunkK = 64;   // K per LDS stage
constexpr int kPRowBytes = kPChunkK * 2;
constexpr int kPBand = 4;      // token tiles per scheduling band
constexpr int kWThreads = 512; // wide-tile kernel: 8 waves
constexpr int kWTileN = 256;   // and its features per tile
constexpr int kPNumXcd = 8;
constexpr int kPCus = 256;
constexpr int kPBufFlags = 0x00020000;

struct ProjArgs {
    const void* x;
    const void* w;
    const float* bias;
    void* out[3];
    long rows;
    int K;
    int Ng;
    int groups;
    int n_tiles;  // groups * Ng / TN
    int r_tiles;
};

#define PJ_LDS __attribute__((address_space(3)))

__device__ __forceinline__ void pj_barrier() { asm volatile("s_barrier" ::: "memory"); }

__device__ __forceinline__ void pj_wait_vm0() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int OFF>
__device__ __forceinline__ u32x4 pj_lds_b128(unsigned addr) {
    u32x4 r;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
    return r;
}

// Waits for every LDS read of the wave; the fragments are in/out operands so
// no use of them is scheduled before the wait.
template <int NF>
__device__ __forceinline__ void pj_lgkm_wait(u32x4 (&f)[NF]) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < NF; ++i) asm volatile("" : "+v"(f[i]));
}

__device__ __forceinline__ int pj_xcd_remap(int bid, int n) {
    const int per = n / kPNumXcd;
    const int rem = n % kPNumXcd;
    const int xcd = bid % kPNumXcd;
    const int idx = bid / kPNumXcd;
    return xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

// Small-tile form: TN features x TR tokens per workgroup (128 x 128), two
// workgroups per CU (64 KiB of LDS each); wave (wn, wr) owns (TN/2) x (TR/2) as
// (TN/64) x (TR/64) blocks. Each chunk's copies are issued right after the
// barrier that frees their stage. With two resident workgroups the one in its
// epilogue or waiting on copies leaves the MFMA pipe to the other, and the many
// tiles even out the rounds over the CUs. Bound by its copies: at full MFMA
// rate its two workgroups would draw 64 bytes per cycle and CU from the L2.
//
// InT is the operands' type. A stage row is 128 bytes of K either way (64 bf16
// or 32 fp32 values), so copies, swizzle and fragment reads are the same
// bytes; a 16-byte fragment holds 8 bf16 values of k (one
// v_mfma_f32_32x32x16_bf16) or 4 fp32 ones (four v_mfma_f32_32x32x2_f32, each
// pairing value e of the lower half-wave's fragment with value e of the upper
// one's, in both operands alike).
//
// fp32 (q/k/v of one frame, 1560 rows, K = 1536, 3 x 1536 features) is bound by
// the fp32 matrix cores (157 TFLOP/s peak): LayerNorm and this launch take
// 187 us, 123 TFLOP/s in the GEMM; three launches of the bounds-checked
// any-shape kernel below took 687-696 us with the same LayerNorm. A chunk's 64
// MFMAs per wave (4,096 cycles) cover its copies many times over. 468
// workgroups on 512 slots leave 9 % of the chip idle. One size for all: a single
// layer of few rows is one wave per SIMD of a few CUs, its time the chain of
// chunks (16 rows x 1536 -> 1536: 101 us; 224 any-shape with the weights from
// HBM, 92 with the same weights in the L2 call after call).
template <typename InT, int TN, int TR, typename OutT, bool kAcc>
__global__ __launch_bounds__(kPThreads, 2) void proj_gemm_small_kernel(ProjArgs a) {
    constexpr int JN = TN / 64, JR = TR / 64;
    constexpr int kWB = TN * kPRowBytes, kXB = TR * kPRowBytes, kSB = kWB + kXB;
    constexpr int kWC = kWB / 4096, kXC = kXB / 4096, kCP = kWC + kXC;  // copies per wave
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kSB];

    const int lid = pj_xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int band_tiles = kPBand * a.n_tiles;
    const int band = lid / band_tiles;
    const int in_band = lid % band_tiles;
    const int band_r0 = band * kPBand;
    int band_h = a.r_tiles - band_r0;
    if (band_h > kPBand) band_h = kPBand;
    const int rt = band_r0 + in_band % band_h;
    const int nt = in_band / band_h;
    const int tiles_per_group = a.Ng / TN;
    const int g = nt / tiles_per_group;
    const int n0 = (nt % tiles_per_group) * TN;
    const long r0 = (long)rt * TR;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int lq = lane & 31;
    const int hh = lane >> 5;
    const int wn = wave & 1;
    const int wr = wave >> 1;

    const unsigned kbytes = (unsigned)a.K * (unsigned)sizeof(InT);
    long xrows = a.rows - r0;
    if (xrows > TR) xrows = TR;
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<InT*>(static_cast<const InT*>(a.w) + ((long)g * a.Ng + n0) * a.K), (short)0,
        (int)(TN * kbytes), kPBufFlags);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<InT*>(static_cast<const InT*>(a.x) + r0 * a.K), (short)0,
        (int)(xrows * (long)kbytes), kPBufFlags);
    const unsigned lds0 = (unsigned)(uintptr_t)lds;
    // copy c of a chunk: 1 KiB block blk of the weight (c < kWC) or token
    // operand, rows 8*blk + lane/8, physical chunk lane % 8
    auto issue_copy = [&](int c, int stage, unsigned kofs) {
        const bool isw = c < kWC;
        const int blk = (isw ? kWC : kXC) * wave + (isw ? c : c - kWC);
        const unsigned row = 8u * (unsigned)blk + (unsigned)(lane >> 3);
        const unsigned lc = (unsigned)(lane & 7) ^ ((row >> 1) & 7u);
        const unsigned dst = lds0 + (unsigned)(stage * kSB) + (isw ? 0u : (unsigned)kWB) +
                             1024u * (unsigned)blk;
        PJ_LDS void* d = (PJ_LDS void*)(uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((int)dst);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(isw ? wrs : xrs, d, 16, row * kbytes + 16u * lc,
                                                 (int)kofs, 0, 0);
    };
    const unsigned fs = (unsigned)((lq >> 1) & 7);
    const unsigned w_row = (unsigned)(wn * (TN / 2) + lq) * kPRowBytes;
    const unsigned x_row = (unsigned)(wr * (TR / 2) + lq) * kPRowBytes;
    constexpr int NF = JN + JR;
    auto read_frags = [&](u32x4 (&f)[NF], int stage, int ks) {
        const unsigned fo = ((unsigned)(2 * ks + hh) ^ fs) << 4;
        const unsigned wa = lds0 + (unsigned)(stage * kSB) + w_row + fo;
        const unsigned xa = lds0 + (unsigned)(stage * kSB + kWB) + x_row + fo;
        f[0] = pj_lds_b128<0>(wa);
        if constexpr (JN > 1) f[1] = pj_lds_b128<32 * kPRowBytes>(wa);
        f[JN] = pj_lds_b128<0>(xa);
        if constexpr (JR > 1) f[JN + 1] = pj_lds_b128<32 * kPRowBytes>(xa);
    };
    static_assert(JN <= 2 && JR <= 2, "fragment reads cover two blocks per operand");

    f32x16 acc[JN][JR];
    {
        const float* bias = a.bias ? a.bias + (long)g * a.Ng + n0 + wn * (TN / 2) : nullptr;
#pragma unroll
        for (int i = 0; i < JN; ++i) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const float4 b4 = bias ? *reinterpret_cast<const float4*>(bias + 32 * i + 8 * q4 +
                                                                          4 * hh)
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int j = 0; j < JR; ++j) {
                    acc[i][j][4 * q4 + 0] = b4.x;
                    acc[i][j][4 * q4 + 1] = b4.y;
                    acc[i][j][4 * q4 + 2] = b4.z;
                    acc[i][j][4 * q4 + 3] = b4.w;
                }
            }
        }
    }

    const int nk = (int)(kbytes / kPRowBytes);
    constexpr int kFeat = TN / 2;
    constexpr int kEs = (int)sizeof(OutT);
    constexpr int kChunks = kFeat * kEs / 16;
    constexpr int kRowsPerPass = 64 / kChunks;
    constexpr int kPasses = 32 / kRowsPerPass;
    OutT* out = static_cast<OutT*>(a.out[g]);
    const int rchunk = lane % kChunks;
    const int rrow = lane / kChunks;
    // Accumulating (out_proj into the fp32 residual stream): every residual
    // value the wave adds in the epilogue, loaded all at once during the last
    // chunk's MFMAs (issued after the copies of that chunk, one chunk ahead),
    // so that their memory latency is not paid at the end of every tile.
    float4 resid[kAcc ? JR : 1][kAcc ? kPasses : 1];
    auto load_resid = [&]() {
#pragma unroll
        for (int j = 0; j < JR; ++j) {
#pragma unroll
            for (int pass = 0; pass < kPasses; ++pass) {
                const long r = r0 + wr * (TR / 2) + 32 * j + pass * kRowsPerPass + rrow;
                // every lane loads (a row past the end reads the last row; the
                // epilogue never writes such rows), so the loop's wait below
                // counts exactly these JR * kPasses loads
                const long rc = r < a.rows ? r : a.rows - 1;
                const float* gp = reinterpret_cast<const float*>(out) + rc * a.Ng + n0 +
                                  wn * kFeat + 4 * rchunk;
                resid[j][pass] = *reinterpret_cast<const float4*>(gp);
            }
        }
    };
#pragma unroll
    for (int c = 0; c < kCP; ++c) issue_copy(c, 0, 0u);
    u32x4 fr[2][NF];
    for (int t = 0; t < nk; ++t) {
        const int st = t & 1;
        // chunk t has landed for every wave after the barrier, and every
        // wave has finished chunk t-1, whose stage the next copies refill.
        // Before the last chunk, the only loads issued after chunk t's copies
        // are the residual loads (a wave's vector-memory operations complete
        // in issue order), which may stay in flight.
        if (kAcc && t == nk - 1 && nk >= 2)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(JR * kPasses) : "memory");
        else
            pj_wait_vm0();
        pj_barrier();
        if (t + 1 < nk) {
#pragma unroll
            for (int c = 0; c < kCP; ++c) issue_copy(c, st ^ 1, (unsigned)(t + 1) * kPRowBytes);
        }
        if constexpr (kAcc) {
            if (t == nk - 2) {
                asm volatile("" ::: "memory");  // the loads go out after the copies
                load_resid();
            }
        }
        read_frags(fr[0], st, 0);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4 (&cur)[NF] = fr[ks & 1];
            pj_lgkm_wait(cur);
            if (ks < 3) read_frags(fr[(ks + 1) & 1], st, ks + 1);
            __builtin_amdgcn_s_setprio(1);
            if constexpr (sizeof(InT) == 2) {
#pragma unroll
                for (int i = 0; i < JN; ++i)
#pragma unroll
                    for (int j = 0; j < JR; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, cur[i]),
                            __builtin_bit_cast(bf16x8, cur[JN + j]), acc[i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < JN; ++i)
#pragma unroll
                        for (int j = 0; j < JR; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                __uint_as_float(cur[i][e]), __uint_as_float(cur[JN + j][e]),
                                acc[i][j], 0, 0, 0);
            }
            __builtin_amdgcn_s_setprio(0);
        }
    }

    // epilogue: 32 tokens at a time
    constexpr int kRowB = kFeat * kEs + 16;
    static_assert(4 * 32 * kRowB <= 2 * kSB, "staging exceeds LDS");
    if constexpr (kAcc) {
        if (nk < 2) load_resid();  // a one-chunk K: no earlier chunk to load under
    }
    pj_barrier();
    unsigned char* sbase = lds + wave * 32 * kRowB;
#pragma unroll
    for (int j = 0; j < JR; ++j) {
        unsigned char* wrow = sbase + lq * kRowB;
#pragma unroll
        for (int i = 0; i < JN; ++i) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const float v0 = acc[i][j][4 * q4 + 0];
                const float v1 = acc[i][j][4 * q4 + 1];
                const float v2 = acc[i][j][4 * q4 + 2];
                const float v3 = acc[i][j][4 * q4 + 3];
                OutT* p = reinterpret_cast<OutT*>(wrow) + 32 * i + 8 * q4 + 4 * hh;
                if constexpr (kEs == 4) {
                    *reinterpret_cast<float4*>(p) = make_float4(v0, v1, v2, v3);
                } else {
                    struct alignas(8) B4 {
                        __bf16 v[4];
                    } o;
                    o.v[0] = (__bf16)v0;
                    o.v[1] = (__bf16)v1;
                    o.v[2] = (__bf16)v2;
                    o.v[3] = (__bf16)v3;
                    *reinterpret_cast<B4*>(p) = o;
                }
            }
        }
#pragma unroll
        for (int pass = 0; pass < 32 / kRowsPerPass; ++pass) {
            const int row = pass * kRowsPerPass + rrow;
            const long r = r0 + wr * (TR / 2) + 32 * j + row;
            const u32x4 vals = *reinterpret_cast<const u32x4*>(sbase + row * kRowB + 16 * rchunk);
            if (r >= a.rows) continue;
            unsigned char* gp = reinterpret_cast<unsigned char*>(out + r * a.Ng + n0 + wn * kFeat) +
                                16 * rchunk;
            if constexpr (kAcc) {
                float4 y = resid[j][pass];
                y.x += __uint_as_float(vals[0]);
                y.y += __uint_as_float(vals[1]);
                y.z += __uint_as_float(vals[2]);
                y.w += __uint_as_float(vals[3]);
                *reinterpret_cast<float4*>(gp) = y;
            } else {
                *reinterpret_cast<u32x4*>(gp) = vals;
            }
        }
    }
}

// Wide-tile form (bf16): 256 features x TR = 64 * JR tokens per workgroup of 8
// waves, one workgroup per CU, two waves per SIMD. Wave (wn, wr) = (wave % 4,
// wave / 4) owns 64 features x TR / 2 tokens as 2 x JR blocks. A tile of
// 256 x 320 draws less than half the L2 bytes per MFMA of a 128 x 128 one. The
// chunk barrier sits between the last k-step's MFMAs, so that the next chunk's
// first fragments arrive under the rest of them, and the copies of a chunk
// (a chunk's MFMAs, 2,560 cycles per SIMD or about 1 us, ahead of their use) are
// spread over the k-steps.
// A tile may hold features of two groups (each wave's 64 lie in one) and reach
// past the last group.
//
// 12,480 tokens, K = 1536, kernel times within a backbone's forward: q/k/v, 3 x
// 1536 features, 145 us (1,217 TFLOP/s; 128 x 128 tiles 169 us on the same card),
// out_proj + residual 68 us (82). Called back to back the card's power sets the
// rate: choose_tile. Beyond the MFMAs a tile's epilogue and first chunk are
// exposed, with one workgroup per CU.
template <int JR, typename OutT, bool kAcc>
__global__ __launch_bounds__(kWThreads, 2) void proj_gemm_wide_kernel(ProjArgs a) {
    constexpr int TN = kWTileN, TR = 64 * JR, JN = 2;
    constexpr int kWB = TN * kPRowBytes, kXB = TR * kPRowBytes, kSB = kWB + kXB;
    constexpr int kWC = kWB / 8192, kXC = kXB / 8192, kCP = kWC + kXC;  // copies per wave
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kSB];

    const int lid = pj_xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int band_tiles = kPBand * a.n_tiles;
    const int band = lid / band_tiles;
    const int in_band = lid % band_tiles;
    const int band_r0 = band * kPBand;
    int band_h = a.r_tiles - band_r0;
    if (band_h > kPBand) band_h = kPBand;
    const int rt = band_r0 + in_band % band_h;
    const int n0 = in_band / band_h * TN;  // first feature, over all groups
    const long r0 = (long)rt * TR;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int lq = lane & 31;
    const int hh = lane >> 5;
    const int wn = wave & 3;
    const int wr = wave >> 2;

    const unsigned kbytes = (unsigned)a.K * 2u;
    const int nall = a.groups * a.Ng;
    const int wrows = min(nall - n0, TN);
    long xrows = a.rows - r0;
    if (xrows > TR) xrows = TR;
    // rows past the features or tokens read as zeros
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<__bf16*>(static_cast<const __bf16*>(a.w) + (long)n0 * a.K), (short)0,
        (int)((unsigned)wrows * kbytes), kPBufFlags);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<__bf16*>(static_cast<const __bf16*>(a.x) + r0 * a.K), (short)0,
        (int)(xrows * (long)kbytes), kPBufFlags);
    const unsigned lds0 = (unsigned)(uintptr_t)lds;
    // copy c of a chunk: 1 KiB block blk of the weight (c < kWC) or token
    // operand, rows 8*blk + lane/8, physical chunk lane % 8. Blocks of a wave
    // are 8 apart, so that (row >> 1) & 7 is the same for all of them.
    const unsigned crow = 8u * (unsigned)wave + (unsigned)(lane >> 3);
    const unsigned cofs = crow * kbytes + 16u * ((unsigned)(lane & 7) ^ ((crow >> 1) & 7u));
    auto issue_copy = [&](int c, int stage, unsigned kofs) {
        const bool isw = c < kWC;
        const unsigned blk = 8u * (unsigned)(isw ? c : c - kWC);
        const unsigned dst = lds0 + (unsigned)(stage * kSB) + (isw ? 0u : (unsigned)kWB) +
                             1024u * (blk + (unsigned)wave);
        PJ_LDS void* d = (PJ_LDS void*)(uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((int)dst);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(isw ? wrs : xrs, d, 16, cofs + blk * 8u * kbytes,
                                                 (int)kofs, 0, 0);
    };
    const unsigned fs = (unsigned)((lq >> 1) & 7);
    const unsigned w_row = (unsigned)(wn * 64 + lq) * kPRowBytes;
    const unsigned x_row = (unsigned)(wr * (TR / 2) + lq) * kPRowBytes;
    constexpr int NF = JN + JR;
    auto read_frags = [&](u32x4 (&f)[NF], int stage, int ks) {
        const unsigned fo = ((unsigned)(2 * ks + hh) ^ fs) << 4;
        const unsigned wa = lds0 + (unsigned)(stage * kSB) + w_row + fo;
        const unsigned xa = lds0 + (unsigned)(stage * kSB + kWB) + x_row + fo;
        f[0] = pj_lds_b128<0>(wa);
        f[1] = pj_lds_b128<32 * kPRowBytes>(wa);
        f[JN] = pj_lds_b128<0>(xa);
        f[JN + 1] = pj_lds_b128<32 * kPRowBytes>(xa);
        f[JN + 2] = pj_lds_b128<64 * kPRowBytes>(xa);
        f[JN + 3] = pj_lds_b128<96 * kPRowBytes>(xa);
        if constexpr (JR > 4) f[JN + 4] = pj_lds_b128<128 * kPRowBytes>(xa);
    };
    static_assert(JR == 4 || JR == 5, "fragment reads cover 4 or 5 token blocks");

    // a wave's 64 features lie in one group (Ng is a multiple of 128)
    const int nw = n0 + wn * 64;
    const int g = min(nw / a.Ng, a.groups - 1);
    const int ng = nw - g * a.Ng;  // feature within the group
    f32x16 acc[JN][JR];
    {
        const float* bias = a.bias && nw < nall ? a.bias + nw : nullptr;
#pragma unroll
        for (int i = 0; i < JN; ++i) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const float4 b4 = bias ? *reinterpret_cast<const float4*>(bias + 32 * i + 8 * q4 +
                                                                          4 * hh)
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int j = 0; j < JR; ++j) {
                    acc[i][j][4 * q4 + 0] = b4.x;
                    acc[i][j][4 * q4 + 1] = b4.y;
                    acc[i][j][4 * q4 + 2] = b4.z;
                    acc[i][j][4 * q4 + 3] = b4.w;
                }
            }
        }
    }
    const int nk = (int)(kbytes / kPRowBytes);
#pragma unroll
    for (int c = 0; c < kCP; ++c) issue_copy(c, 0, 0u);
    pj_wait_vm0();
    pj_barrier();
    u32x4 fr[2][NF];
    read_frags(fr[0], 0, 0);
    auto mfma = [&](const u32x4 (&f)[NF], int j0, int j1) {
#pragma unroll
        for (int j = j0; j < j1; ++j)
#pragma unroll
            for (int i = 0; i < JN; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, f[i]), __builtin_bit_cast(bf16x8, f[JN + j]),
                    acc[i][j], 0, 0, 0);
    };
    for (int t = 0; t < nk; ++t) {
        const int st = t & 1;
        const bool more = t + 1 < nk;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4 (&cur)[NF] = fr[ks & 1];
            u32x4 (&nxt)[NF] = fr[(ks + 1) & 1];
            pj_lgkm_wait(cur);
            if (ks < 3) read_frags(nxt, st, ks + 1);
            // the next chunk's copies, spread over the first k-steps: their
            // stage was last read before the barrier of the previous chunk
            if (ks < 3 && more) {
#pragma unroll
                for (int c = ks * kCP / 3; c < (ks + 1) * kCP / 3; ++c)
                    issue_copy(c, st ^ 1, (unsigned)(t + 1) * kPRowBytes);
            }
            __builtin_amdgcn_s_setprio(1);
            if (ks < 3) {
                mfma(cur, 0, JR);
            } else {
                // the chunk barrier sits between the last k-step's MFMAs: every
                // read of chunk t is complete (waited above), and once all
                // waves pass here chunk t+1 has landed; its first fragments
                // arrive under the remaining MFMAs
                mfma(cur, 0, JR / 2);
                if (more) {
                    pj_wait_vm0();
                    pj_barrier();
                    read_frags(nxt, st ^ 1, 0);
                }
                mfma(cur, JR / 2, JR);
            }
            __builtin_amdgcn_s_setprio(0);
        }
    }

    // epilogue: 32 tokens x 64 features of a wave at a time, staged in LDS as
    // token rows and stored as full 16-byte lanes along rows
    constexpr int kFeat = 64;
    constexpr int kEs = (int)sizeof(OutT);
    constexpr int kChunks = kFeat * kEs / 16;
    constexpr int kRowsPerPass = 64 / kChunks;
    constexpr int kPasses = 32 / kRowsPerPass;
    constexpr int kRowB = kFeat * kEs + 16;
    static_assert(8 * 32 * kRowB <= 2 * kSB, "staging exceeds LDS");
    OutT* out = static_cast<OutT*>(a.out[g]);
    const int rchunk = lane % kChunks;
    const int rrow = lane / kChunks;
    float4 resid[kAcc ? 2 : 1][kAcc ? kPasses : 1];
    auto load_resid = [&](int j) {
#pragma unroll
        for (int pass = 0; pass < kPasses; ++pass) {
            const long r = r0 + wr * (TR / 2) + 32 * j + pass * kRowsPerPass + rrow;
            const long rc = r < a.rows ? r : a.rows - 1;
            if (nw < nall)
                resid[j & 1][pass] = *reinterpret_cast<const float4*>(
                    reinterpret_cast<const float*>(out) + rc * a.Ng + ng + 4 * rchunk);
        }
    };
    if constexpr (kAcc) load_resid(0);
    pj_barrier();  // every wave has finished reading the operand stages
    if (nw >= nall) return;
    unsigned char* sbase = lds + wave * 32 * kRowB;
#pragma unroll
    for (int j = 0; j < JR; ++j) {
        if constexpr (kAcc) {
            if (j + 1 < JR) load_resid(j + 1);
        }
        unsigned char* wrow = sbase + lq * kRowB;
#pragma unroll
        for (int i = 0; i < JN; ++i) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const float v0 = acc[i][j][4 * q4 + 0];
                const float v1 = acc[i][j][4 * q4 + 1];
                const float v2 = acc[i][j][4 * q4 + 2];
                const float v3 = acc[i][j][4 * q4 + 3];
                OutT* p = reinterpret_cast<OutT*>(wrow) + 32 * i + 8 * q4 + 4 * hh;
                if constexpr (kEs == 4) {
                    *reinterpret_cast<float4*>(p) = make_float4(v0, v1, v2, v3);
                } else {
                    struct alignas(8) B4 {
                        __bf16 v[4];
                    } o;
                    o.v[0] = (__bf16)v0;
                    o.v[1] = (__bf16)v1;
                    o.v[2] = (__bf16)v2;
                    o.v[3] = (__bf16)v3;
                    *reinterpret_cast<B4*>(p) = o;
                }
            }
        }
#pragma unroll
        for (int pass = 0; pass < kPasses; ++pass) {
            const int row = pass * kRowsPerPass + rrow;
            const long r = r0 + wr * (TR / 2) + 32 * j + row;
            const u32x4 vals = *reinterpret_cast<const u32x4*>(sbase + row * kRowB + 16 * rchunk);
            if (r >= a.rows) continue;
            unsigned char* gp =
                reinterpret_cast<unsigned char*>(out + r * a.Ng + ng) + 16 * rchunk;
            if constexpr (kAcc) {
                float4 y = resid[j & 1][pass];
                y.x += __uint_as_float(vals[0]);
                y.y += __uint_as_float(vals[1]);
                y.z += __uint_as_float(vals[2]);
                y.w += __uint_as_float(vals[3]);
                *reinterpret_cast<float4*>(gp) = y;
            } else {
                *reinterpret_cast<u32x4*>(gp) = vals;
            }
        }
    }
}

template <int JR, typename OutT, bool kAcc>
void launch_wide(ProjArgs a, hipStream_t st) {
    a.n_tiles = (a.groups * a.Ng + kWTileN - 1) / kWTileN;
    a.r_tiles = (int)((a.rows + 64 * JR - 1) / (64 * JR));
    hipLaunchKernelGGL((proj_gemm_wide_kernel<JR, OutT, kAcc>),
                       dim3((unsigned)(a.n_tiles * a.r_tiles)), dim3(kWThreads), 0, st, a);
}

template <int JR>
void launch_wide(const ProjArgs& a, int out_dtype, bool accumulate, hipStream_t st) {
    if (out_dtype == 1)
        launch_wide<JR, __bf16, false>(a, st);
    else if (accumulate)
        launch_wide<JR, float, true>(a, st);
    else
        launch_wide<JR, float, false>(a, st);
}

// Tile of a bf16 launch: 0 = 128 x 128, else JR of the wide form (4: 256 x 256,
// 5: 256 x 320). Each form's time is its rounds over the chip times the measured
// time of a round (K = 1536): 128 x 128 fills 512 slots in 29 us, and its tiles
// even out beyond the first round; 256 x 256 takes 43.6 us a round of 256, 256 x
// 320 51 us. With few chunks of K a launch is bound by its outputs, which the
// 128 x 128 form writes (and, accumulating, whose residual it reads) under its
// other workgroup's MFMAs; the wide forms' one workgroup a CU does not. So these
// take K from 256, accumulating from 768. All three add the same terms in the
// same order: results are equal bit for bit. Measured, the card kept busy (us;
// 128 x 128, 256 x 256, 256 x 320):
//   K = 1536: 12480 tokens x 4608 features 174, 169, 149; x 1536 accumulating 78,
//   93, 66; 9000 x 3072 91, 84, 92; 3120 x 4608 49, 44, 47; 1560 x 4608 27, 38, 41
//   12480 x 3072, K = 512: 53, 53, 44; K = 256: 34, 36, 30; 12480 x 4608, K = 192:
//   41, 44, 41; K = 128: 33, 37, 35; 9000 x 6144, K = 128: 32, 38, 35
//   12480 x 3072 accumulating, K = 1024: 105, 114, 100; K = 512: 72, 80, 72;
//   K = 256: 56, 67, 58; 28000 x 3072, K = 512: 180, 198, 201
int choose_tile(long rows, int K, int features, bool accumulate) {
    if (K < (accumulate ? 768 : 256)) return 0;
    const double small_tiles =
        (double)((rows + kPSmall - 1) / kPSmall) * ((features + kPSmall - 1) / kPSmall);
    double best = 29.0 * (small_tiles > 2 * kPCus ? small_tiles / (2 * kPCus) : 1.0);
    int jr = 0;
    const double round_us[2] = {43.6, 51.0};
    for (int j = 4; j <= 5; ++j) {
        const long tiles =
            ((rows + 64 * j - 1) / (64 * j)) * ((features + kWTileN - 1) / kWTileN);
        const double t = round_us[j - 4] * (double)((tiles + kPCus - 1) / kPCus);
        if (t < best) {
            best = t;
            jr = j;
        }
    }
    return jr;
}

// Shapes the tiled kernels take: whole 128-byte chunks of K, whole feature tiles,
// operand tiles addressed with 32-bit offsets.
bool tileable(int in_dtype, int K, int N, int tile_n) {
    const long kbytes = (long)K * (in_dtype == 0 ? 4 : 2);
    return kbytes % kPRowBytes == 0 && N % tile_n == 0 && kbytes * kWTileN <= 0x7fffffffL;
}

// Tiled kernel of a launch over features in all groups, as kvp_linear_kernel
// reports it: 2 = 128 x 128, 3 = 256 x 256, 4 = 256 features x 320 tokens.
int tiled_kernel(int in_dtype, long rows, int K, int features, bool accumulate) {
    if (in_dtype == 0) return 2;
    const int jr = choose_tile(rows, K, features, accumulate);
    // (a tile's tokens are addressed with 32-bit offsets)
    return jr == 0 || 128L * jr * K > 0x7fffffffL ? 2 : jr - 1;
}

template <typename InT, typename OutT, bool kAcc>
void launch_small(const ProjArgs& a, hipStream_t st) {
    const int grid = a.n_tiles * a.r_tiles;
    hipLaunchKernelGGL((proj_gemm_small_kernel<InT, kPSmall, kPSmall, OutT, kAcc>),
                       dim3((unsigned)grid), dim3(kPThreads), 0, st, a);
}


// ---------------------------------------------------------------------------
// Generic linear layer (shapes and alignments the grouped kernel does not take):
//
//   y[r, n] = sum_k x[r, k] * w[n, k] + bias[n]  (+ y[r, n])
//
// x [rows, K], w [N, K] row-major (K-contiguous), fp32 or bf16 (widened to
// fp32 in LDS), bias fp32 or null, y fp32 or bf16 (fp32 may accumulate into
// itself). fp32 matrix cores: v_mfma_f32_32x32x2_f32 (full fp32 products,
// fp32 accumulation). Workgroup = 4 waves, output tile 64 features x 64
// rows, wave (w & 1, w >> 1) owns 32 x 32 of it: lane l holds row (l % 32)
// of the block and features 8*(v/4) + 4*(l/32) + v%4 in accumulator v (A =
// w rows, B = x rows, as in the grouped kernel). K advances in chunks of 32;
// each chunk of w and x is staged in LDS as 64 rows of 32 values padded to
// 33, so that the 32 lanes of a half-wave reading one k of 32 rows hit 32
// distinct banks. Every global access is bounds-checked: any rows, K and N.
// The epilogue stages the 64 x 64 tile in the same LDS as rows (pitch 65)
// and stores it row by row, 16 lanes per 64-value row, 4 consecutive values
// per lane (one 16-byte fp32 / 8-byte bf16 store where the row and its
// alignment allow, per-value stores at ragged edges): a row's 256 bytes go
// out together instead of 4-byte pieces of 32 rows per instruction.
// ---------------------------------------------------------------------------
constexpr int kGTile = 64;
constexpr int kGChunk = 32;
constexpr int kGPitch = kGChunk + 1;
constexpr int kGOutPitch = kGTile + 1;
static_assert(kGTile * kGOutPitch <= 2 * kGTile * kGPitch, "output staging exceeds LDS");

struct GenericArgs {
    const void* x;
    const void* w;
    const float* bias;
    void* y;
    long rows;
    int K, N;
    int n_tiles;
};

template <typename T>
__device__ __forceinline__ float to_f32(T v) {
    return (float)v;
}

template <typename InT, typename OutT, bool kAcc>
__global__ __launch_bounds__(256) void gemm_generic_kernel(GenericArgs a) {
    __shared__ float lds[2 * kGTile * kGPitch];
    float* ws = lds;
    float* xs = lds + kGTile * kGPitch;
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const long n0 = (long)(blockIdx.x % a.n_tiles) * kGTile;
    const long r0 = (long)(blockIdx.x / a.n_tiles) * kGTile;
    const InT* W = static_cast<const InT*>(a.w);
    const InT* X = static_cast<const InT*>(a.x);
    const int bn = 32 * (wave & 1);   // the wave's feature block within the tile
    const int br = 32 * (wave >> 1);  // its row block
    const int lr = lane & 31;
    const int lk = lane >> 5;
    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    for (int k0 = 0; k0 < a.K; k0 += kGChunk) {
        // 64 rows x 32 k of each operand: element e = tid + 256 j is row
        // e / 32, k e % 32 (a warp's consecutive lanes read consecutive k)
#pragma unroll
        for (int j = 0; j < kGTile * kGChunk / 256; ++j) {
            const int e = tid + 256 * j;
            const int row = e / kGChunk;
            const int kk = e % kGChunk;
            const long gk = (long)k0 + kk;
            const long gn = n0 + row;
            const long gr = r0 + row;
            ws[row * kGPitch + kk] = gn < a.N && gk < a.K ? to_f32(W[gn * a.K + gk]) : 0.f;
            xs[row * kGPitch + kk] = gr < a.rows && gk < a.K ? to_f32(X[gr * a.K + gk]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kGChunk; kk += 2) {
            const float av = ws[(bn + lr) * kGPitch + kk + lk];
            const float bv = xs[(br + lr) * kGPitch + kk + lk];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    // stage: row br + lr of the tile, columns bn + 8*(v/4) + 4*lk + v%4
    // (the loop's last barrier has freed the operand tiles)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int col = bn + 8 * (v / 4) + 4 * lk + v % 4;
        const long n = n0 + col;
        lds[(br + lr) * kGOutPitch + col] = acc[v] + (a.bias && n < a.N ? a.bias[n] : 0.f);
    }
    __syncthreads();
    // 64 rows x 16 four-value groups, 4 per thread; 16 consecutive threads
    // cover one row
    const bool vec_ok = (a.N % 4) == 0 &&
                        ((uintptr_t)a.y % (4 * sizeof(OutT))) == 0;
#pragma unroll
    for (int j = 0; j < kGTile * kGTile / 4 / 256; ++j) {
        const int c = tid + 256 * j;
        const int row = c / (kGTile / 4);
        const int col = 4 * (c % (kGTile / 4));
        const long r = r0 + row;
        const long n = n0 + col;
        if (r >= a.rows || n >= a.N) continue;
        const float* src = lds + row * kGOutPitch + col;
        OutT* Y = static_cast<OutT*>(a.y) + r * a.N + n;
        if (vec_ok) {
            // n + 3 < N: N and n are multiples of 4
            float v4[4] = {src[0], src[1], src[2], src[3]};
            if constexpr (sizeof(OutT) == 4) {
                if constexpr (kAcc) {
                    const float4 y = *reinterpret_cast<const float4*>(Y);
                    v4[0] += y.x;
                    v4[1] += y.y;
                    v4[2] += y.z;
                    v4[3] += y.w;
                }
                *reinterpret_cast<float4*>(Y) = make_float4(v4[0], v4[1], v4[2], v4[3]);
            } else {
                struct alignas(8) B4 {
                    OutT v[4];
                } o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o.v[i] = (OutT)v4[i];
                *reinterpret_cast<B4*>(Y) = o;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (n + i >= a.N) break;
                float val = src[i];
                if constexpr (kAcc) val += to_f32(Y[i]);
                Y[i] = (OutT)val;
            }
        }
    }
}

// Short inner dimension (K = 4, 8, 12 or 16), fp32: y (+)= x W^T + b.
//
// A lane keeps the K weights of 4 neighbouring features in registers (through
// LDS: loaded directly, 64 lines per load, the kernel took 37 us) and its wave
// walks kThinRows rows, whose values are wave-uniform (scalar loads), so a row
// costs 4 K FMAs and one 16-byte store per lane: bound by writing y. The
// 64 x 64 tiles of gemm_generic_kernel pad K to 32 and stage both operands
// through LDS for one chunk of work. 12480 rows x 16 -> 1536 features, within a
// backbone's forward: 46 -> 28 us (2.8 TB/s written; with 16 rows per wave 32 us,
// 8 rows took 32.6 and 32 rows 38.7).
// short_inner says where it is used.
constexpr int kThinRows = 16;
constexpr int kThinCols = 256;

template <int kK, bool kAcc>
__global__ __launch_bounds__(256) void gemm_thin_kernel(const float* __restrict__ X,
                                                         const float* __restrict__ W,
                                                         const float* __restrict__ bias,
                                                         float* __restrict__ Y, long rows, int N,
                                                         int n_tiles) {
    static_assert(kK % 4 == 0 && kK <= 16, "4 kK weights per lane");
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    constexpr int kPitch = kThinCols + 4;  // 16 columns x 4 k's quads: 64 banks
    __shared__ __attribute__((aligned(16))) float ws[kK * kPitch];
    const int n0 = (int)(blockIdx.x % n_tiles) * kThinCols;
    const long r0 = (long)(blockIdx.x / n_tiles) * (4 * kThinRows) + wave * kThinRows;
    for (int i = (int)threadIdx.x; i < kThinCols * (kK / 4); i += 256) {
        const int c = i / (kK / 4), k = 4 * (i % (kK / 4));
        float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
        if (n0 + c < N) t = *reinterpret_cast<const float4*>(W + (long)(n0 + c) * kK + k);
        ws[k * kPitch + c] = t.x;
        ws[(k + 1) * kPitch + c] = t.y;
        ws[(k + 2) * kPitch + c] = t.z;
        ws[(k + 3) * kPitch + c] = t.w;
    }
    __syncthreads();
    const int c = 4 * ((int)threadIdx.x & 63), n = n0 + c;
    if (n >= N) return;  // N is a multiple of 4: the lane's 4 features exist
    float4 w[kK];
#pragma unroll
    for (int k = 0; k < kK; ++k) w[k] = *reinterpret_cast<const float4*>(ws + k * kPitch + c);
    float4 b = bias ? *reinterpret_cast<const float4*>(bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
    // wait for the bias here: its first use is in the loop, where the wait for it
    // would be one for the store of the row before, too (1560 rows, 16 -> 1536:
    // 7.6 -> 7.2 us)
    asm volatile("" : "+v"(b.x), "+v"(b.y), "+v"(b.z), "+v"(b.w));
    const long end = min(r0 + kThinRows, rows);
    Y += n;
#pragma unroll 4
    for (long r = r0; r < end; ++r) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int k = 0; k < kK; ++k) {
            const float x = X[r * kK + k];
            v.x = fmaf(x, w[k].x, v.x);
            v.y = fmaf(x, w[k].y, v.y);
            v.z = fmaf(x, w[k].z, v.z);
            v.w = fmaf(x, w[k].w, v.w);
        }
        v = make_float4(v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w);
        float4* y = reinterpret_cast<float4*>(Y + r * N);
        if constexpr (kAcc) {
            const float4 o = *y;
            v = make_float4(v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w);
        }
        *y = v;
    }
}

// Whether the kernel above takes an fp32 layer (16-byte aligned operands). Its
// waves write rows one by one: stores of less than 256 bytes (512 for 16 inputs)
// hold them up, also in a last column block of few features, which only the work
// of many other blocks hides; few rows leave no work to gain from. Any-shape
// kernel -> this one, us:
// 12480 rows, 16 -> 1536 36.3 -> 19.2, 16 -> 256 11.2 -> 7.3, 16 -> 64 6.5 -> 6.4
// (60000 rows: 1.2 times as long), 16 -> 4 5.2 -> 11.3; 16 -> 260 at 1560 rows
// 6.3 -> 10.9, at 20000 0.80 of the time; 8 -> 64 at 1560 rows 6.1 -> 5.2; 4 -> 4
// at 12480 rows 5.2 -> 5.2, at 200000 17.3 -> 11.5.
bool short_inner(long rows, int K, int N) {
    if (K > 16 || K % 4 || N % 4 || rows < 64) return false;
    const int last = (N - 1) % kThinCols + 1;  // features of the last column block
    return K == 4 || last >= (K < 16 ? 64 : 128) || (long)(N / kThinCols) * rows >= 16384;
}

template <typename InT, typename OutT, bool kAcc>
void launch_generic(const GenericArgs& a, long grid, hipStream_t st) {
    hipLaunchKernelGGL((gemm_generic_kernel<InT, OutT, kAcc>), dim3((unsigned)grid), dim3(256), 0,
                       st, a);
}

}  // namespace

int launch_gemm_generic(int in_dtype, int out_dtype, const void* x, const void* w,
                        const float* bias, void* y, long rows, int K, int N, bool accumulate,
                        void* stream) {
    if (!((in_dtype == 0 && out_dtype == 0) || (in_dtype == 1 && (out_dtype == 0 || out_dtype == 1)))) {
        set_error("linear: dtype pair (%d, %d) not supported (fp32->fp32, bf16->bf16, "
                  "bf16->fp32)",
                  in_dtype, out_dtype);
        return 1;
    }
    if (rows <= 0 || K <= 0 || N <= 0) {
        set_error("linear: empty shape rows=%ld in=%d out=%d", rows, K, N);
        return 1;
    }
    if (accumulate && out_dtype != 0) {
        set_error("linear: accumulate needs fp32 output");
        return 1;
    }
    if (!x || !w || !y) {
        set_error("linear: null x/w/y pointer");
        return 1;
    }
    GenericArgs a;
    a.x = x;
    a.w = w;
    a.bias = bias;
    a.y = y;
    a.rows = rows;
    a.K = K;
    a.N = N;
    const bool thin = in_dtype == 0 && short_inner(rows, K, N) &&
                      ((uintptr_t)w | (uintptr_t)bias | (uintptr_t)y) % 16 == 0;
    const int cols = thin ? kThinCols : kGTile;
    const int tile_rows = thin ? 4 * kThinRows : kGTile;
    const long n_tiles = ((long)N + cols - 1) / cols;
    const long r_tiles = (rows + tile_rows - 1) / tile_rows;
    if (n_tiles * r_tiles > 0x7fffffffL) {
        set_error("linear: grid too large");
        return 1;
    }
    a.n_tiles = (int)n_tiles;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const long grid = n_tiles * r_tiles;
    if (thin) {
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), 0, st,
                               static_cast<const float*>(x), static_cast<const float*>(w), bias,
                               static_cast<float*>(y), rows, N, a.n_tiles);
        };
        auto pick = [&](auto acc) {
            constexpr bool kAcc = decltype(acc)::value;
            switch (K) {
                case 4: go(gemm_thin_kernel<4, kAcc>); break;
                case 8: go(gemm_thin_kernel<8, kAcc>); break;
                case 12: go(gemm_thin_kernel<12, kAcc>); break;
                default: go(gemm_thin_kernel<16, kAcc>);
            }
        };
        if (accumulate)
            pick(std::true_type{});
        else
            pick(std::false_type{});
    } else if (in_dtype == 0) {
        if (accumulate)
            launch_generic<float, float, true>(a, grid, st);
        else
            launch_generic<float, float, false>(a, grid, st);
    } else if (out_dtype == 1) {
        launch_generic<__bf16, __bf16, false>(a, grid, st);
    } else if (accumulate) {
        launch_generic<__bf16, float, true>(a, grid, st);
    } else {
        launch_generic<__bf16, float, false>(a, grid, st);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("linear launch: %s", hipGetErrorString(e));
        return 1;
    }
    return 0;
}

int launch_proj_gemm(int in_dtype, const void* x, const void* w, const float* bias,
                     void* const* outs, int groups, long rows, int K, int Ng, int out_dtype,
                     bool accumulate, int tile_n, void* stream) {
    if (groups < 1 || groups > 3 || rows <= 0 || K <= 0 || Ng <= 0) {
        set_error("proj_gemm: bad shape groups=%d rows=%ld K=%d N=%d", groups, rows, K, Ng);
        return 1;
    }
    if (tile_n != 128 && tile_n != 256) {
        set_error("proj_gemm: tile_n must be 128 or 256");
        return 1;
    }
    if (in_dtype == 0 && (tile_n != 128 || out_dtype != 0)) {
        set_error("proj_gemm: fp32 operands need tile_n 128 and fp32 output");
        return 1;
    }
    if (!tileable(in_dtype, K, Ng, tile_n)) {
        set_error("proj_gemm: shape K=%d N=%d not supported (K %% %d, N %% %d)", K, Ng,
                  in_dtype == 0 ? kPChunkK / 2 : kPChunkK, tile_n);
        return 2;
    }
    if (accumulate && out_dtype != 0) {
        set_error("proj_gemm: accumulate needs fp32 output");
        return 1;
    }
    if (!x || !w) {
        set_error("proj_gemm: null operand");
        return 1;
    }
    uintptr_t al = (uintptr_t)x | (uintptr_t)w | (uintptr_t)bias;
    for (int g = 0; g < groups; ++g) {
        if (!outs[g]) {
            set_error("proj_gemm: null output %d", g);
            return 1;
        }
        al |= (uintptr_t)outs[g];
    }
    if (al & 15u) {
        set_error("proj_gemm: operands must be 16-byte aligned");
        return 1;
    }
    const long r_tiles = (rows + kPSmall - 1) / kPSmall;
    const long n_tiles = (long)groups * (Ng / kPSmall);
    if (r_tiles * n_tiles > 0x7fffffffL || (long)groups * Ng > 0x7fffffffL) {
        set_error("proj_gemm: grid too large");
        return 1;
    }
    ProjArgs a;
    a.x = x;
    a.w = w;
    a.bias = bias;
    for (int g = 0; g < 3; ++g) a.out[g] = g < groups ? outs[g] : nullptr;
    a.rows = rows;
    a.K = K;
    a.Ng = Ng;
    a.groups = groups;
    a.n_tiles = (int)n_tiles;
    a.r_tiles = (int)r_tiles;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (in_dtype == 0) {
        if (accumulate)
            launch_small<float, float, true>(a, st);
        else
            launch_small<float, float, false>(a, st);
    } else {
        const int kernel =
            tile_n == 256 ? 3 : tiled_kernel(in_dtype, rows, K, groups * Ng, accumulate);
        if (kernel == 4)
            launch_wide<5>(a, out_dtype, accumulate, st);
        else if (kernel == 3)
            launch_wide<4>(a, out_dtype, accumulate, st);
        else if (out_dtype == 1)
            launch_small<__bf16, __bf16, false>(a, st);
        else if (accumulate)
            launch_small<__bf16, float, true>(a, st);
        else
            launch_small<__bf16, float, false>(a, st);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("proj_gemm launch: %s", hipGetErrorString(e));
        return 1;
    }
    return 0;
}

}  // namespace kvp

extern "C" int kvp_linear_kernel(int in_dtype, int out_dtype, long rows, int in_features,
                                 int out_features, int groups, int accumulate) {
    using namespace kvp;
    const int K = in_features, N = out_features;
    const bool types = (in_dtype == 1 && (out_dtype == 0 || out_dtype == 1)) ||
                       (in_dtype == 0 && out_dtype == 0);
    if (!types || (accumulate && out_dtype != 0) || rows <= 0 || K <= 0 || N <= 0 || groups < 1 ||
        groups > 3)
        return -1;
    if (tileable(in_dtype, K, N, kPSmall))
        return tiled_kernel(in_dtype, rows, K, groups * N, accumulate != 0);
    return in_dtype == 0 && short_inner(rows, K, N) ? 1 : 0;
}

extern "C" int kvp_proj_gemm(const void* x, const void* w, const float* bias, void* out0,
                             void* out1, void* out2, int groups, long rows, int K, int N,
                             int out_dtype, int accumulate, int tile_n, void* stream) {
    void* outs[3] = {out0, out1, out2};
    const int rc = kvp::launch_proj_gemm(1, x, w, bias, outs, groups, rows, K, N, out_dtype,
                                         accumulate != 0, tile_n, stream);
    return rc == 0 ? 0 : 1;
}
