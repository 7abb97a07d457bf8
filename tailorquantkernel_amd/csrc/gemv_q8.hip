// gemv_q8.hip — the Q8 weight side of the attention layer on gfx950: the
// weight x Q8-activation matmul (kernel/q8_scalar.c:3-30, kernel/kernel.h:13-20)
// and the projections around attention that use it (project_qkv and
// project_output, model/attention_layer.c:38-46,161-167, and their batched
// forms, :213-218,238-241).
//
// Device weight layout ("tiled Q8"), exactly the byte count of the
// reference's rows x cols/32 block_q8 array:
//   codes  [rows][cols] int8.  A row is cut into groups of up to 64 blocks
//          (2048 codes); a group of n blocks holds the first 16 codes of each
//          of its n blocks (16 B per block, in block order), then the last 16
//          codes of each.  Lane l of a wave reads block 64g+l of a row as two
//          16-byte loads, each wave-wide load one contiguous 1 KiB.
//   scales [rows][cols/32] fp32 at byte offset rows*cols, one coalesced
//          dword per lane per group.
// tq_hip_q8_pack turns the reference's block_q8 rows into this layout on the
// device; tq_hip_q8_unpack turns it back.
//
// "Tiled Q4" (packer/packer.h:9, the reference's 20-byte block_q4), the same
// byte count as its rows x cols/32 block_q4 array:
//   codes  [rows][cols/2]: each block's 16 nibble bytes as the reference
//          stores them (byte j: code j + 8 in the low nibble, code j + 24 in
//          the high nibble), blocks in order, so lane l of a wave reads block
//          64g+l as one 16-byte load and a wave-wide load is 1 KiB.
//   scales [rows][cols/32] fp32 at byte offset rows*cols/2.
// A Q4 dword w is turned into two dwords of signed bytes 16*code with
// x = w ^ 0x88888888 (the nibble n becomes n - 8 in 4-bit two's complement):
// (x << 4) & 0xF0F0F0F0 holds the low codes, x & 0xF0F0F0F0 the high codes.
// The int32 dot of those with the activation codes is 16 times the block's
// exact dot sum_j (n_j - 8) * x_j of kernel/q4_scalar.c:6-11, and an
// arithmetic shift by 4 gives it back exactly.
//
// Matmul: the work is one pass over the weight bytes (HBM-bound).  A
// 256-thread work-group runs 4 waves; a wave owns RW consecutive rows.  The
// work-group first copies the activation rows (up to T tokens of block_q8,
// the reference's activation format) straight into LDS with
// global_load_lds_dwordx4, then every wave issues the loads of its first 8
// (row, group) units, and only then waits: the copies, issued first, are
// complete once no more than those 3*8 weight loads are outstanding, so the
// activation copy hides under the weight latency.
// Per block: int32 dot of the 32 code pairs (8 v_dot4_i32_i8), then
// ((float)s * w_d) * x_d as the scalar reference rounds it; the per-lane sums
// over groups and the 64-lane sum replace the reference's serial block-order
// sum (the reference's own SIMD kernels reorder that sum as well).
//
// The projections (project_qkv: wq, wk and wv in one launch over their
// concatenated rows; project_output) take fp32 input rows.  For one or two
// rows the matmul launch copies them into LDS and quantizes them there
// (bit-exact quantize_row_q8), and work-group 0 leaves the blocks in the
// caller's workspace; for more rows quantize_row_q8 runs into the workspace
// first, as the reference quantizes into xn_q8 / ws->xq, and the matmul
// reads the blocks from there.
#include "tq_common.hpp"

#include <stdlib.h>

#include <algorithm>

namespace {

using namespace tq;

constexpr int kGemvWaves = 4;
constexpr int kGroupBlocks = 64;
constexpr int kGroupBytes = kGroupBlocks * kQK;   // 2048
constexpr int kGroupBytes4 = kGroupBlocks * 16;   // 1024: a Q4 group
constexpr int kBlockBytes4 = 20;                  // sizeof(block_q4)
constexpr int kMaxSegs = 3;
// Activation rows in LDS per work-group: 8 rows of 8192 (73,728 bytes) fit,
// two work-groups per CU's 160 KiB.
constexpr size_t kMaxStageBytes = 80 * 1024;
constexpr size_t kDefaultLdsLimit = 64 * 1024;    // beyond this a kernel must opt in

int herr(hipError_t e) { return e == hipSuccess ? TQ_HIP_OK : TQ_HIP_EHIP_BASE - (int)e; }

// Byte offset inside a tiled row of code j (0..31) of block b.
__host__ __device__ __forceinline__ int tiled_offset(int nb, int b, int j) {
    const int g = b / kGroupBlocks;
    const int rest = nb - g * kGroupBlocks;
    const int n = rest < kGroupBlocks ? rest : kGroupBlocks;
    const int i = b - g * kGroupBlocks;
    return g * kGroupBytes + (j < 16 ? 16 * i + j : 16 * n + 16 * i + (j - 16));
}

// ---------------------------------------------------------------------------
// block_q8 rows <-> tiled layout.  One thread per block.
__global__ __launch_bounds__(256) void pack_kernel(unsigned char *__restrict__ dst,
                                                   const unsigned char *__restrict__ src,
                                                   int rows, int nb) {
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= (long long)rows * nb) return;
    const int r = (int)(k / nb), b = (int)(k - (long long)r * nb);
    const uint32_t *blk = reinterpret_cast<const uint32_t *>(src + (size_t)k * kBlockBytes);
    u32x4 lo, hi;
    lo.x = blk[1]; lo.y = blk[2]; lo.z = blk[3]; lo.w = blk[4];
    hi.x = blk[5]; hi.y = blk[6]; hi.z = blk[7]; hi.w = blk[8];
    const int cols = nb * kQK;
    unsigned char *row = dst + (size_t)r * cols;
    *reinterpret_cast<u32x4 *>(row + tiled_offset(nb, b, 0)) = lo;
    *reinterpret_cast<u32x4 *>(row + tiled_offset(nb, b, 16)) = hi;
    reinterpret_cast<uint32_t *>(dst + (size_t)rows * cols)[k] = blk[0];
}

__global__ __launch_bounds__(256) void unpack_kernel(unsigned char *__restrict__ dst,
                                                     const unsigned char *__restrict__ src,
                                                     int rows, int nb) {
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= (long long)rows * nb) return;
    const int r = (int)(k / nb), b = (int)(k - (long long)r * nb);
    const int cols = nb * kQK;
    const unsigned char *row = src + (size_t)r * cols;
    const u32x4 lo = *reinterpret_cast<const u32x4 *>(row + tiled_offset(nb, b, 0));
    const u32x4 hi = *reinterpret_cast<const u32x4 *>(row + tiled_offset(nb, b, 16));
    uint32_t *blk = reinterpret_cast<uint32_t *>(dst + (size_t)k * kBlockBytes);
    blk[0] = reinterpret_cast<const uint32_t *>(src + (size_t)rows * cols)[k];
    blk[1] = lo.x; blk[2] = lo.y; blk[3] = lo.z; blk[4] = lo.w;
    blk[5] = hi.x; blk[6] = hi.y; blk[7] = hi.z; blk[8] = hi.w;
}

// block_q4 rows <-> tiled Q4.  One thread per block.
__global__ __launch_bounds__(256) void pack4_kernel(unsigned char *__restrict__ dst,
                                                    const unsigned char *__restrict__ src, long long n) {
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const uint32_t *blk = reinterpret_cast<const uint32_t *>(src + (size_t)k * kBlockBytes4);
    u32x4 q;
    q.x = blk[1]; q.y = blk[2]; q.z = blk[3]; q.w = blk[4];
    *reinterpret_cast<u32x4 *>(dst + (size_t)k * 16) = q;
    reinterpret_cast<uint32_t *>(dst + (size_t)n * 16)[k] = blk[0];
}

__global__ __launch_bounds__(256) void unpack4_kernel(unsigned char *__restrict__ dst,
                                                      const unsigned char *__restrict__ src, long long n) {
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const u32x4 q = *reinterpret_cast<const u32x4 *>(src + (size_t)k * 16);
    uint32_t *blk = reinterpret_cast<uint32_t *>(dst + (size_t)k * kBlockBytes4);
    blk[0] = reinterpret_cast<const uint32_t *>(src + (size_t)n * 16)[k];
    blk[1] = q.x; blk[2] = q.y; blk[3] = q.z; blk[4] = q.w;
}

// Signed bytes 16 * code from a dword of Q4 nibbles: low nibbles, high nibbles.
__device__ __forceinline__ uint32_t q4_lo16(uint32_t w) { return ((w ^ 0x88888888u) << 4) & 0xF0F0F0F0u; }
__device__ __forceinline__ uint32_t q4_hi16(uint32_t w) { return (w ^ 0x88888888u) & 0xF0F0F0F0u; }

// ---------------------------------------------------------------------------
// Matmul over up to three row-concatenated matrices sharing one input
// (project_qkv runs wq, wk and wv in one launch).

struct GemvSeg {
    const unsigned char *w;   // tiled matrix
    float *y;                 // y[t * rows + r]
    int rows;
};

struct GemvArgs {
    GemvSeg seg[kMaxSegs];
    int seg_end[kMaxSegs];    // cumulative row ends
    int rows_total;
    int cols, nb, ng;
    const unsigned char *xq;  // block_q8 [n_tok][nb] (when x is null)
    const float *x;           // fp32 [n_tok][cols], 16-byte aligned, quantized in LDS
    unsigned char *xq_out;    // where work-group 0 leaves quantize_row_q8(x), or null
    int n_tok;                // rows of input in this launch (<= T)
    bool q4;                  // the matrices are tiled Q4 (else tiled Q8)
    bool uni_tiles;           // GEMM: every 128-row tile lies in one segment and every
                              // segment's codes and scales are under 2 GiB
    float *part;              // GEMM split-K partial tiles [ksplit][n_tok][rows_total], or null
    size_t part_floats;       // their capacity
    int ksplit;               // GEMM: K splits of this launch (1: none)
    bool xs;                  // GEMM: xq holds the block-major split layout of
                              // tq_launch_quantize_split instead of block_q8 rows
    unsigned char *hq;        // GEMM over the MLP's gate (segment 0) and up (segment 1)
                              // matrices: each tile pairs 64 rows of both, and the
                              // epilogue writes silu_mul + quantize_row_q8 of the
                              // hidden rows in the split layout here instead of y;
                              // with K splits the reduce launch does so beside y,
                              // in the split layout or (hq_xs false) as block_q8 rows
    bool hq_xs;
};

typedef __attribute__((address_space(3))) unsigned char lds_u8;
typedef int v4i __attribute__((ext_vector_type(4)));

// 16 bytes from each active lane's global address into LDS at dst + 16*lane
// (global_load_lds_dwordx4; M0 holds the LDS byte address and is restored;
// dst must be the same for the whole wave).  A scalar write of M0 needs one
// wait state before the copy that reads it, which the compiler does not add
// inside an asm block: the s_nop here and in the copies below.
// The memory clobber keeps every later load after it in program order, which
// the vmcnt arithmetic below relies on.
__device__ __forceinline__ void dma16(const void *src, unsigned char *dst) {
    const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u8 *)dst);
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(src), "s"(lds)
        : "memory");
}

// Wait until at most N vector memory operations of this wave are outstanding.
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt immediate");
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// 4 bytes from each active lane's global address into LDS at dst + 4*lane
// (global_load_lds_dword).
__device__ __forceinline__ void dma4(const void *src, unsigned char *dst) {
    const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u8 *)dst);
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
        "global_load_lds_dword %1, off\n\ts_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(src), "s"(lds)
        : "memory");
}

// The same copies from a uniform base plus a 32-bit lane offset (the saddr
// form) to LDS byte address lds + IMM: no per-lane 64-bit address arithmetic,
// and two scalar instructions with the copy, the s_nop among them (M0 is left
// changed; nothing else in these kernels uses it).  base and lds are uniform.
template <int IMM>
__device__ __forceinline__ void dma16s(const unsigned char *base, uint32_t off, uint32_t lds) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(off), "s"(base), "s"(lds), "n"(IMM)
                 : "m0", "scc", "memory");
}
template <int IMM>
__device__ __forceinline__ void dma4s(const unsigned char *base, uint32_t off, uint32_t lds) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :
                 : "v"(off), "s"(base), "s"(lds), "n"(IMM)
                 : "m0", "scc", "memory");
}

// `bytes` (a multiple of 4) from src into LDS at dst, all by DMA: whole
// 16-byte chunks when src is 16-byte aligned, the rest (and everything
// otherwise) as dwords.  The caller's wait_vm covers the copies.
__device__ __forceinline__ void stage_bytes(const unsigned char *src, int bytes, unsigned char *dst) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int chunks = ((uintptr_t)src & 15) ? 0 : bytes >> 4;
    for (int c0 = wave * 64; c0 < chunks; c0 += kThreads) {
        if (c0 + lane < chunks) dma16(src + 16 * (c0 + lane), dst + 16 * c0);
    }
    const int words = (bytes - (chunks << 4)) >> 2;
    const int base = chunks << 4;
    for (int w0 = wave * 64; w0 < words; w0 += kThreads) {
        if (w0 + lane < words) dma4(src + base + 4 * (w0 + lane), dst + base + 4 * w0);
    }
}

// quantize_row_q8 (kernel/quant_x.c:12-33) of the n_tok fp32 rows staged at
// xf into block_q8 rows at xs: 8 lanes x 4 values per block.  The task count
// and the stride are multiples of 8, so a block's 8 lanes are active
// together.  Work-group 0 also leaves the blocks at a.xq_out.
__device__ __forceinline__ void quantize_lds(const GemvArgs &a, const unsigned char *xf, unsigned char *xs) {
    const int blocks = a.n_tok * a.nb;
    for (int k = threadIdx.x; k < blocks * 8; k += kThreads) {
        const int e = k & 7, tb = k >> 3;
        const float4 v = *reinterpret_cast<const float4 *>(xf + (size_t)(tb * kQK + 4 * e) * 4);
        const float xv[4] = {v.x, v.y, v.z, v.w};
        unsigned char *blk = xs + (size_t)tb * kBlockBytes;
        quantize8x4(xv, reinterpret_cast<float *>(blk), blk + 4 + 4 * e, e == 0);
    }
    if (a.xq_out && blockIdx.x == 0) {
        __syncthreads();
        const uint32_t *src = reinterpret_cast<const uint32_t *>(xs);
        uint32_t *dst = reinterpret_cast<uint32_t *>(a.xq_out);
        for (int w = threadIdx.x; w < blocks * (kBlockBytes / 4); w += kThreads) dst[w] = src[w];
    }
}

// Every load is unconditional (rows past the end and groups past the last
// one are clamped to real data and masked out of the sums), so no load
// result is left unread on any path and the compiler never has to wait for
// one in-flight load before issuing the next.
// XF: the input is fp32 rows, staged raw and quantized in LDS (T <= 2).
// Q4: the matrices are tiled Q4: one 16-byte load per (row, block) instead of
// two, turned into the two code halves before the dot products.
template <int T, int RW, int GC, bool XF, bool Q4>
__global__ __launch_bounds__(256) void gemv_q8_kernel(GemvArgs a) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int row0 = (blockIdx.x * kGemvWaves + wave) * RW;
    const int cols = a.cols, nb = a.nb, ng = a.ng;
    // xs: [T][nb] block_q8, as in global memory; with XF the fp32 rows come
    // first in LDS and the blocks after them.
    unsigned char *xs = XF ? smem + (size_t)T * cols * 4 : smem;
    if (XF) stage_bytes(reinterpret_cast<const unsigned char *>(a.x), a.n_tok * cols * 4, smem);
    else stage_bytes(a.xq, a.n_tok * nb * kBlockBytes, smem);

    const unsigned char *wrow[RW];
    const float *drow[RW];
    float *yrow[RW];
    int ldy[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) {
        const int r = row0 + i < a.rows_total ? row0 + i : a.rows_total - 1;
        // Field-wise selects keep the segment in scalar registers (an indexed
        // a.seg[s] would be a vector load of the kernel arguments).
        const bool s0 = r < a.seg_end[0], s1 = !s0 && r < a.seg_end[1];
        const unsigned char *w = s0 ? a.seg[0].w : (s1 ? a.seg[1].w : a.seg[2].w);
        float *y = s0 ? a.seg[0].y : (s1 ? a.seg[1].y : a.seg[2].y);
        const int rows = s0 ? a.seg[0].rows : (s1 ? a.seg[1].rows : a.seg[2].rows);
        const int lr = r - (s0 ? 0 : (s1 ? a.seg_end[0] : a.seg_end[1]));
        const size_t rowb = Q4 ? (size_t)cols / 2 : (size_t)cols;   // code bytes per row
        wrow[i] = w + (size_t)lr * rowb;
        drow[i] = reinterpret_cast<const float *>(w + (size_t)rows * rowb) + (size_t)lr * nb;
        yrow[i] = y + lr;
        ldy[i] = rows;
    }

    float acc[RW][T];
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
        for (int t = 0; t < T; t++) acc[i][t] = 0.0f;

    for (int g0 = 0; g0 < ng; g0 += GC) {
        u32x4 wlo[GC][RW], whi[GC][RW];
        float wd[GC][RW];
#pragma unroll
        for (int u = 0; u < GC; u++) {
            const int g = g0 + u < ng ? g0 + u : ng - 1;
            const int rest = nb - g * kGroupBlocks;
            const int n = rest < kGroupBlocks ? rest : kGroupBlocks;
            const int bl = lane < n ? lane : n - 1;
#pragma unroll
            for (int i = 0; i < RW; i++) {
                if (Q4) {
                    wlo[u][i] = *reinterpret_cast<const u32x4 *>(wrow[i] + g * kGroupBytes4 + 16 * bl);
                } else {
                    const unsigned char *p = wrow[i] + g * kGroupBytes + 16 * bl;
                    wlo[u][i] = *reinterpret_cast<const u32x4 *>(p);
                    whi[u][i] = *reinterpret_cast<const u32x4 *>(p + 16 * n);
                }
                wd[u][i] = drow[i][g * kGroupBlocks + bl];
            }
        }
        if (g0 == 0) {
            // the activation copies, issued first, have landed once no more
            // than this wave's weight loads (2 or 3 per unit) are in flight
            wait_vm<(Q4 ? 2 : 3) * GC * RW>();
            __syncthreads();
            if (XF) {
                quantize_lds(a, smem, xs);
                __syncthreads();
            }
        }
#pragma unroll
        for (int u = 0; u < GC; u++) {
            const int g = g0 + u < ng ? g0 + u : ng - 1;
            const int rest = nb - g * kGroupBlocks;
            const int n = rest < kGroupBlocks ? rest : kGroupBlocks;
            const bool valid = lane < n && g0 + u < ng;
            const int bl = lane < n ? lane : n - 1;
            if (Q4) {
#pragma unroll
                for (int i = 0; i < RW; i++) {
                    const u32x4 w = wlo[u][i];
                    wlo[u][i] = u32x4{q4_lo16(w.x), q4_lo16(w.y), q4_lo16(w.z), q4_lo16(w.w)};
                    whi[u][i] = u32x4{q4_hi16(w.x), q4_hi16(w.y), q4_hi16(w.z), q4_hi16(w.w)};
                }
            }
            int s[T][RW];
            float xd[T];
#pragma unroll
            for (int t = 0; t < T; t++) {
                // Block 64g+bl of token t: d, then 8 dwords of codes (a 36-byte
                // lane stride is 9 banks apart: conflict-free).
                const uint32_t *xb = reinterpret_cast<const uint32_t *>(
                    xs + (size_t)(t * nb + g * kGroupBlocks + bl) * kBlockBytes);
                xd[t] = __uint_as_float(xb[0]);
#pragma unroll
                for (int i = 0; i < RW; i++) {
                    int d = 0;
                    d = __builtin_amdgcn_sdot4(wlo[u][i].x, xb[1], d, false);
                    d = __builtin_amdgcn_sdot4(wlo[u][i].y, xb[2], d, false);
                    d = __builtin_amdgcn_sdot4(wlo[u][i].z, xb[3], d, false);
                    d = __builtin_amdgcn_sdot4(wlo[u][i].w, xb[4], d, false);
                    d = __builtin_amdgcn_sdot4(whi[u][i].x, xb[5], d, false);
                    d = __builtin_amdgcn_sdot4(whi[u][i].y, xb[6], d, false);
                    d = __builtin_amdgcn_sdot4(whi[u][i].z, xb[7], d, false);
                    d = __builtin_amdgcn_sdot4(whi[u][i].w, xb[8], d, false);
                    s[t][i] = Q4 ? d >> 4 : d;
                }
            }
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int i = 0; i < RW; i++) {
                    const float p = ((float)s[t][i] * wd[u][i]) * xd[t];
                    acc[i][t] += valid ? p : 0.0f;
                }
        }
    }

#pragma unroll
    for (int i = 0; i < RW; i++) {
        if (row0 + i >= a.rows_total) continue;
#pragma unroll
        for (int t = 0; t < T; t++) {
            if (t < a.n_tok) {
                const float v = wave_sum(acc[i][t]);
                if (lane == 0) yrow[i][(size_t)t * ldy[i]] = v;
            }
        }
    }
}

// LDS of a launch: t block_q8 rows, plus the t fp32 rows they are quantized
// from when the input is fp32.
size_t lds_bytes(int t, int nb, bool xf) {
    return (size_t)t * nb * kBlockBytes + (xf ? (size_t)t * nb * kQK * 4 : 0);
}

// ---------------------------------------------------------------------------
// Many tokens: int8 MFMA GEMM.  A work-group of 8 waves computes a 128-row x
// 128-token tile (TT = 128), or 64 where that pads less (gemm_toks); wave w
// owns rows 32(w%4)..+31 of tokens 64(w/4)..+63 (32(w/4)..+31), two 32 x 32
// tiles (one).  The smaller tile halves the products and the token copies
// per weight byte: 28,672 x 4,096 over 64 tokens 49 us against 67 with 128
// tokens' tile.  The K dimension goes 4 blocks (128 codes) per stage through
// two LDS buffers filled by direct-to-LDS copies, one stage ahead of the one
// being multiplied; at 74.8 KB and 128 registers two work-groups share a CU,
// four waves per SIMD.
//
// Per block, v_mfma_i32_32x32x32_i8 (one 32-value block deep, the int8 form
// that runs at the full 2,048 operations per cycle: 32 cycles for what four
// 16x16x32 products take 64) gives the exact int32 block dots with the tokens
// as rows, and each lane folds its 16 with fma(s, w_d * x_d, acc): the
// reference's per-block product (kernel/q8_scalar.c:9-11) with one rounding
// fewer, summed over blocks in order.  The products w_d * x_d of two blocks
// come from one v_mfma_f32_32x32x1_2b_f32, an outer product of depth 1 and
// so each product rounded once, like v_mul_f32: 32 cycles per block for 16
// vector multiplies, and the operands are one scale per lane instead of 17.
//
// What bounds it: per 32 x 32 tile and block the matrix products (32 + 32
// cycles) and 32 vector instructions (about 70 cycles at four waves), which
// overlap little (an fp32 MFMA keeps the vector unit from issuing).  Without
// the copies the loop is at that sum; the copies cost the rest, so their
// shape matters: a wave's weight copy reads 64 contiguous bytes per row (four
// lanes a row; one lane a row, 16 bytes every row pitch, cost 20 % more).
// Against 16 x 16 products, vector scale multiplies and 16-byte row pieces
// and per-stage copy addresses (8B shapes): MLP over 2,048 rows 1,277 -> 964
// us, the attention layer over 2,048 rows 451 -> 352 us, results unchanged bit
// for bit.
//
// Tile order: work-groups are dealt to the 8 XCDs round-robin, so the grid is
// laid out so that every token tile of one row tile runs on the same XCD
// (work-group w: XCD w % 8, row tile 8 (w/8 / n_tt) + w % 8) and the tile's
// 128 weight rows are read from HBM once into that XCD's L2.
//
// LDS per stage (37,376 B; 28,160 with 64 tokens):
//   A   [2 halves][128 rows][4 slots][16 B]   weight codes (Q4: one nibble run
//       instead of two halves), block b of row r in slot gemm_slot(b, r)
//   WD  [128 rows][4 blocks] fp32             weight scales
//   B   [128 tokens][4 blocks x 36 B]         the tokens' block_q8, as stored:
//       with 16-byte aligned rows and a block count that is a multiple of 4,
//       a token's 144 bytes are nine 16-byte copies (rounds of 512, the last
//       one's surplus lanes, whole waves, issue none); otherwise 36 dword
//       copies per token.  Or, from the split layout, codes
//       [4 blocks][2 halves][128 tokens][16 B], then scales
//       [4 blocks][128 + 32 tokens] fp32 (two blocks' rows in other banks).
constexpr int kGemmThreads = 512;
constexpr int kGemmRows = 128, kGemmKB = 4, kGemmBufs = 2;
constexpr int kGemmA = kGemmKB * 2 * kGemmRows * 16;            // 16,384
constexpr int kGemmWD = kGemmKB * kGemmRows * 4;                // 2,048
constexpr int kGemmBRow = kGemmKB * kBlockBytes;                // 144 bytes per token
static_assert(kGemmA / 16 == 2 * kGemmThreads && kGemmKB * kGemmRows == kGemmThreads, "whole weight copy rounds per stage");

// Sizes that depend on a tile's tokens (128 or 64).
template <int TT>
struct GemmTile {
    static constexpr int T2 = TT / 64;                              // 32-token tiles per wave
    static constexpr int ROWS = TT * kGemmBRow;                     // block_q8 rows: 18,432 or 9,216
    static constexpr int CHUNKS = ROWS / 16;                        // 16-byte copies
    static constexpr int ROUNDS = (CHUNKS + kGemmThreads - 1) / kGemmThreads;
    static constexpr int WORDS = ROWS / 4;                          // dword copies
    static constexpr int SROW = TT + 32;                            // floats between two blocks' token scales
    static constexpr int CODES = kGemmKB * kQK * TT;                // split-layout codes, then scales
    static constexpr int B = CODES + kGemmKB * SROW * 4;            // 18,944 or 9,728
    static constexpr int STAGE = kGemmA + kGemmWD + B;              // 37,376 or 28,160
    static_assert(ROWS <= B && STAGE % 16 == 0 && CHUNKS % 64 == 0 && WORDS % 64 == 0, "stage layout, whole waves");
};

// Slot of a stage's block (0..3) in its row's 64 bytes of codes (its own
// inverse): any 16 consecutive rows then hold a block in 16 different 16-byte
// bank groups (a 16-byte read of 64 lanes takes 4 cycles; 8 when two of 16
// rows share one, 16 without the permutation).
__device__ __forceinline__ int gemm_slot(int blk, int row) { return blk ^ ((row >> 2) & 3); }

typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

// BX4: the activation rows are 16-byte aligned and nb % 4 == 0.
// Q4: tiled Q4 matrices.  A holds [128 rows][4 slots][16 B] nibble bytes (one
// copy per thread instead of two); each lane turns its row's 16 bytes of a block
// into 16 x its 16 codes (low nibbles for k < 16, high for k >= 16), and the
// scales are 1/16 of the matrix's.
template <bool BX4, bool Q4, bool UNI, bool XS, int TT>
__global__ __launch_bounds__(512, BX4 ? 4 : 2) void gemm_q8_kernel(GemvArgs a) {
    static_assert(!UNI || BX4, "uniform copies need whole 16-byte stages");
    static_assert(!XS || UNI, "the split layout is copied from uniform bases");
    using G = GemmTile<TT>;
    constexpr int T2 = G::T2;
    // two blocks' weight scales at a time where all four do not fit the
    // registers (128-token Q4 tiles of block_q8 rows spilled 5: 28,672 x 4,096
    // over 2,048 tokens 698 us, now 640)
    constexpr bool kScaleEach = Q4 && UNI && !XS && TT == 128;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hi = lane >> 5;
    const int q4_shift = hi ? 0 : 4;
    const int cols = a.cols, nb = a.nb;
    const int n_tt = (a.n_tok + TT - 1) / TT;
    const int n_rt = (a.rows_total + kGemmRows - 1) / kGemmRows;
    // split ks of ksplit takes the ks-th run of stages; the grid repeats the
    // tile order once per split (a multiple of 8 work-groups each, so the XCD
    // of a tile is the same in every split)
    const int g0 = gridDim.x / a.ksplit;
    const int bx = blockIdx.x % g0, ks = blockIdx.x / g0;
    const int k = bx >> 3;
    const int rt = (k / n_tt) * 8 + (bx & 7), tt = k % n_tt;
    if (rt >= n_rt) return;   // the padding of the last row of XCD groups
    const int row0 = rt * kGemmRows, tok0 = tt * TT;
    const int stages = (nb + kGemmKB - 1) / kGemmKB;
    const int st_begin = ks * stages / a.ksplit, st_end = (ks + 1) * stages / a.ksplit;
    const int wr = 32 * (wave & 3), wt = 32 * T2 * (wave >> 2);
    // this wave's token scales of a stage: block, first token
    const int s_blk = TT == 128 ? wave >> 1 : wave, s_tok = TT == 128 ? 64 * (wave & 1) : 0;

    // A: thread tid copies 16 bytes of row tid / 4 (both halves of the block,
    // slot tid % 4); WD: one row's four scales per lane (dwords: scale tid % 4
    // of row tid / 4).
    const int my_row = tid >> 2;
    const int my_blk = gemm_slot(tid & 3, my_row);
    const unsigned char *wrow;
    const float *drow;
    {
        const int r = row0 + my_row < a.rows_total ? row0 + my_row : a.rows_total - 1;
        const bool s0 = r < a.seg_end[0], s1 = !s0 && r < a.seg_end[1];
        const unsigned char *w = s0 ? a.seg[0].w : (s1 ? a.seg[1].w : a.seg[2].w);
        const int rows = s0 ? a.seg[0].rows : (s1 ? a.seg[1].rows : a.seg[2].rows);
        const int lr = r - (s0 ? 0 : (s1 ? a.seg_end[0] : a.seg_end[1]));
        const size_t rowb = Q4 ? (size_t)cols / 2 : (size_t)cols;
        wrow = w + (size_t)lr * rowb;
        drow = reinterpret_cast<const float *>(w + (size_t)rows * rowb) + (size_t)lr * nb;
    }

    // Copies from uniform bases, when every tile lies in one segment (the
    // host checks that segment ends fall on tile boundaries and that offsets
    // fit 32 bits) and every stage is whole (16-byte token rows, nb % 4 == 0):
    // a stage's four blocks then lie in one 64-block group, the block and
    // half of each copy are the same for the whole wave, and a copy is a
    // scalar base (segment, group, block, half) plus this lane's fixed row
    // offset, with no vector address arithmetic per stage.
    constexpr bool uni = UNI;
    const unsigned char *useg = nullptr;   // the rows' segment: codes, then scales at uscale
    const unsigned char *uwd = nullptr;    // the same for this wave's scale rows
    size_t uscale = 0;
    uint32_t vrow = 0, vdrow = 0, vb[XS ? 2 : G::ROUNDS];
    if constexpr (uni) {
        const bool s0 = row0 < a.seg_end[0], s1 = !s0 && row0 < a.seg_end[1];
        useg = uwd = s0 ? a.seg[0].w : (s1 ? a.seg[1].w : a.seg[2].w);
        int rows = s0 ? a.seg[0].rows : (s1 ? a.seg[1].rows : a.seg[2].rows);
        const int start = s0 ? 0 : (s1 ? a.seg_end[0] : a.seg_end[1]);
        auto clamped = [&](int r) { return (row0 + r < a.rows_total ? row0 + r : a.rows_total - 1) - start; };
        int r = clamped(my_row), rd = clamped(64 * (wave & 1) + lane);
        if (a.hq) {
            // paired tile rt: rows 64 rt.. of the gate matrix, then the same
            // rows of the up matrix.  A wave's code copies (16 rows) and its
            // scale copies (64 rows) each lie in one of them.
            useg = wave < 4 ? a.seg[0].w : a.seg[1].w;
            uwd = (wave & 1) ? a.seg[1].w : a.seg[0].w;
            rows = a.seg[0].rows;
            r = 64 * rt + (my_row & 63);
            rd = 64 * rt + lane;
        }
        const uint32_t rowb = Q4 ? (uint32_t)cols / 2 : (uint32_t)cols;
        uscale = (size_t)rows * rowb;
        vrow = (uint32_t)r * rowb + 16u * (uint32_t)my_blk;
        vdrow = (uint32_t)rd * (uint32_t)nb * 4u;
        if constexpr (XS) {
            // every copy of this lane is for one token of the tile: its
            // 16-byte half-block and its scale in the block-major runs
            const int tk = s_tok + lane;
            const int t = tok0 + tk < a.n_tok ? tok0 + tk : a.n_tok - 1;
            vb[0] = 16u * (uint32_t)t;
            vb[1] = 4u * (uint32_t)t;
        } else {
#pragma unroll
            for (int j = 0; j < G::ROUNDS; j++) {
                const int c = tid + kGemmThreads * j;
                const int cc = c < G::CHUNKS ? c : G::CHUNKS - 1;
                const int tk = cc / 9, piece = cc - 9 * tk;
                const int t = tok0 + tk < a.n_tok ? tok0 + tk : a.n_tok - 1;
                vb[j] = (uint32_t)t * (uint32_t)nb * (uint32_t)kBlockBytes + 16u * (uint32_t)piece;
            }
        }
    }

    // The token rows' sources of this thread's B copies, fixed over the stages
    // (a stage only adds 36 bytes per block to each).
    const unsigned char *bsrc[G::ROUNDS];
    if (BX4) {
#pragma unroll
        for (int j = 0; j < G::ROUNDS; j++) {
            const int c = tid + kGemmThreads * j;
            const int cc = c < G::CHUNKS ? c : G::CHUNKS - 1;
            const int tk = cc / 9, piece = cc - 9 * tk;
            const int t = tok0 + tk < a.n_tok ? tok0 + tk : a.n_tok - 1;
            bsrc[j] = a.xq + (size_t)t * nb * kBlockBytes + 16 * piece;
        }
    }

    // The same copies from uniform bases (whole stages only): each copy of a
    // stage has its own base, which moves on by a fixed step from stage to
    // stage (the weight codes jump at the end of a 64-block group), so a
    // copy costs three or four scalar instructions.  (Recomputing the bases
    // from the stage number took about 100 per stage and wave, issued in order
    // in front of its products: attention layer over 2,048 rows 354 us, now
    // 351; Q4 MLP over 100 rows 104.3, now 103.4.)
    const unsigned char *pw0 = nullptr, *pw1 = nullptr, *pd = nullptr, *px[2] = {nullptr, nullptr}, *pxd = nullptr;
    int in_group = 0;   // blocks of the current group already copied
    int group_left = 0; // blocks of the row from the current group on
    size_t xstep = 0;
    auto start_uni = [&](int st) {
        const int b0 = st * kGemmKB;
        const int g = b0 / kGroupBlocks;
        in_group = b0 - g * kGroupBlocks;
        group_left = nb - g * kGroupBlocks;
        const int n = group_left < kGroupBlocks ? group_left : kGroupBlocks;
        if (Q4) {
            pw0 = useg + 16 * b0;
        } else {
            pw0 = useg + g * kGroupBytes + 16 * in_group;
            pw1 = pw0 + 16 * n;
        }
        pd = uwd + uscale + 4 * b0;
        if constexpr (XS) {
            // codes: 16-byte chunk c -> (block c / 2TT, half (c / TT) & 1,
            // token c % TT), so the wave's one or two copies are of half
            // `half` of block blk (and blk + 2); scales: one block's tokens
            const size_t n16 = 16 * (size_t)a.n_tok;
            const int blk = TT == 128 ? wave >> 2 : wave >> 1, half = TT == 128 ? (wave >> 1) & 1 : wave & 1;
            xstep = 2 * kGemmKB * n16;
            px[0] = a.xq + (size_t)(2 * (b0 + blk) + half) * n16;
            px[1] = px[0] + 4 * n16;
            pxd = a.xq + (size_t)a.n_tok * cols + 4 * (size_t)(b0 + s_blk) * a.n_tok;
        } else {
            px[0] = a.xq + (size_t)b0 * kBlockBytes;
        }
    };
    auto issue_uni = [&](uint32_t buf) {
        const uint32_t at = buf + 16 * 64 * wave;   // the wave's KiB of a round of copies
        dma16s<0>(pw0, vrow, at);
        if (!Q4) dma16s<16 * kGemmThreads>(pw1, vrow, at);
        if (wave < 2) dma16s<kGemmA>(pd, vdrow, at);
        if constexpr (XS) {
            dma16s<kGemmA + kGemmWD>(px[0], vb[0], at);
            if (TT == 128) dma16s<kGemmA + kGemmWD + 16 * kGemmThreads>(px[1], vb[0], at);
            if (TT == 128 || wave < kGemmKB)
                dma4s<kGemmA + kGemmWD + G::CODES>(pxd, vb[1], buf + 4 * (G::SROW * s_blk + s_tok));
            px[0] += xstep;
            px[1] += xstep;
            pxd += xstep / 8;
        } else {
            // whole rounds, then the waves of the last one
            constexpr int REST = G::CHUNKS % kGemmThreads / 64;
            dma16s<kGemmA + kGemmWD>(px[0], vb[0], at);
            if (TT == 128 || wave < REST) dma16s<kGemmA + kGemmWD + 16 * kGemmThreads>(px[0], vb[1], at);
            if constexpr (TT == 128) {
                if (wave < REST) dma16s<kGemmA + kGemmWD + 32 * kGemmThreads>(px[0], vb[2], at);
            }
            static_assert(G::ROUNDS == (TT == 128 ? 3 : 2), "the rounds above");
            px[0] += kGemmKB * kBlockBytes;
        }
        pd += 4 * kGemmKB;
        if (Q4) {
            pw0 += 16 * kGemmKB;
        } else {
            pw0 += 16 * kGemmKB;
            pw1 += 16 * kGemmKB;
            in_group += kGemmKB;
            if (in_group == kGroupBlocks) {
                // the next group starts after this one's last halves
                pw0 += 16 * kGroupBlocks;
                in_group = 0;
                group_left -= kGroupBlocks;
                pw1 = pw0 + 16 * (group_left < kGroupBlocks ? group_left : kGroupBlocks);
            }
        }
    };

    // The same from per-lane addresses; LDS addresses from the wave's number, in
    // scalar registers (from tid - lane they are vector ones, and the 128-token
    // Q8 tile spilled 12 of them: rows of 4,032 / 960 / 960 x 4,096 over 2,048
    // tokens 180 us, now 154)
    const int tid0 = 64 * wave;
    auto issue = [&](int st, unsigned char *buf) {
        const int b0 = st * kGemmKB;
        const int bw = b0 + my_blk < nb ? b0 + my_blk : nb - 1;
        if (Q4) {
            dma16(wrow + 16 * bw, buf + 16 * tid0);
        } else {
#pragma unroll
            for (int half = 0; half < 2; half++)
                dma16(wrow + tiled_offset(nb, bw, 16 * half), buf + 16 * (tid0 + kGemmThreads * half));
        }
        dma4(drow + (b0 + (tid & 3) < nb ? b0 + (tid & 3) : nb - 1), buf + kGemmA + 4 * tid0);
        if (BX4) {
            // the last round's copies past the tile are left out (whole waves)
#pragma unroll
            for (int j = 0; j < G::ROUNDS; j++)
                if (tid + kGemmThreads * j < G::CHUNKS)
                    dma16(bsrc[j] + b0 * kBlockBytes, buf + kGemmA + kGemmWD + 16 * (tid0 + kGemmThreads * j));
        } else {
#pragma unroll
            for (int j = 0; j < (G::WORDS + kGemmThreads - 1) / kGemmThreads; j++) {
                const int c = tid + kGemmThreads * j;
                if (c >= G::WORDS) break;   // whole waves
                const int tk = c / (kGemmBRow / 4), w = c - tk * (kGemmBRow / 4);
                const int blk = w / 9;
                const int t = tok0 + tk < a.n_tok ? tok0 + tk : a.n_tok - 1;
                const int b = b0 + blk < nb ? b0 + blk : nb - 1;
                dma4(a.xq + ((size_t)t * nb + b) * kBlockBytes + 4 * (w - 9 * blk),
                     buf + kGemmA + kGemmWD + 4 * (tid0 + kGemmThreads * j));
            }
        }
    };

    v16f acc[T2];
#pragma unroll
    for (int t2 = 0; t2 < T2; t2++) acc[t2] = v16f(0.0f);

    // Two buffers (74.8 KB, or 56.3 with 64 tokens: two work-groups share a CU): stage st+1 is
    // copied while stage st is multiplied.
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_u8 *)smem;
    if constexpr (uni) {
        start_uni(st_begin);
        issue_uni(lds0);
    } else {
        issue(st_begin, smem);
    }
    for (int st = st_begin; st < st_end; st++) {
        unsigned char *buf = smem + ((st - st_begin) & 1) * G::STAGE;
        wait_vm<0>();      // this wave's copies of stage st have landed
        __syncthreads();   // stage st is in LDS everywhere; stage st-1's buffer is free
        if (st + 1 < st_end) {
            if constexpr (uni)
                issue_uni(lds0 + (((st + 1 - st_begin) & 1) ? G::STAGE : 0));
            else
                issue(st + 1, smem + ((st + 1 - st_begin) & 1) * G::STAGE);
        }
        const unsigned char *A = buf, *WD = buf + kGemmA, *B = buf + kGemmA + kGemmWD;
        // the row's four scales (times 1/16 for the Q4 codes, which come as 16 x code)
        float4 wd4 = float4{};
        if (!kScaleEach) wd4 = *reinterpret_cast<const float4 *>(WD + (wr + l32) * 16);
        if (Q4) wd4 = make_float4(wd4.x * 0.0625f, wd4.y * 0.0625f, wd4.z * 0.0625f, wd4.w * 0.0625f);
#pragma unroll
        for (int b2 = 0; b2 < kGemmKB; b2 += 2) {
            // both blocks' scales: lane (l32, hi) holds those of block b2 + hi
            float wd = b2 == 0 ? (hi ? wd4.y : wd4.x) : (hi ? wd4.w : wd4.z);
            if (kScaleEach) wd = *reinterpret_cast<const float *>(WD + (wr + l32) * 16 + 4 * (b2 + hi)) * 0.0625f;
            float xd[T2];
#pragma unroll
            for (int t2 = 0; t2 < T2; t2++) {
                const int t = wt + 32 * t2 + l32;
                if constexpr (XS) {
                    xd[t2] = *reinterpret_cast<const float *>(B + G::CODES + ((b2 + hi) * G::SROW + t) * 4);
                } else {
                    // (with 16-byte token rows every stage is whole; past nb the
                    // copies repeat block nb - 1: load and select, no branch)
                    const float xv = *reinterpret_cast<const float *>(B + t * kGemmBRow + (b2 + hi) * kBlockBytes);
                    xd[t2] = BX4 || st * kGemmKB + b2 + hi < nb ? xv : 0.0f;
                }
            }
            v4i wv[2], xv[2][T2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int blk = b2 + j;
                if (Q4) {
                    const u32x4 w = *reinterpret_cast<const u32x4 *>(A + ((wr + l32) * kGemmKB + gemm_slot(blk, wr + l32)) * 16);
#pragma unroll
                    for (int i = 0; i < 4; i++) wv[j][i] = (int)(((w[i] ^ 0x88888888u) << q4_shift) & 0xF0F0F0F0u);
                } else {
                    wv[j] = *reinterpret_cast<const v4i *>(
                        A + ((hi * kGemmRows + wr + l32) * kGemmKB + gemm_slot(blk, wr + l32)) * 16);
                }
#pragma unroll
                for (int t2 = 0; t2 < T2; t2++) {
                    const int t = wt + 32 * t2 + l32;
                    if constexpr (XS) {
                        xv[j][t2] = *reinterpret_cast<const v4i *>(B + ((blk * 2 + hi) * TT + t) * 16);
                    } else {
                        const int *x = reinterpret_cast<const int *>(B + t * kGemmBRow + blk * kBlockBytes + 4 + 16 * hi);
                        xv[j][t2] = v4i{x[0], x[1], x[2], x[3]};
                    }
                }
            }
#pragma unroll
            for (int t2 = 0; t2 < T2; t2++) {
                const v32f p = __builtin_amdgcn_mfma_f32_32x32x1f32(xd[t2], wd, v32f(0.0f), 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const v16i c = __builtin_amdgcn_mfma_i32_32x32x32_i8(xv[j][t2], wv[j], v16i(0), 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[t2][i] = fmaf((float)c[i], p[16 * j + i], acc[t2][i]);
                }
            }
        }
    }

    // y[t][r]: lane (l32, hi) holds row l32 of the wave's 32, register i token
    // 8 (i / 4) + 4 hi + i % 4 of each 32-token tile, so a store covers 32
    // consecutive rows of two tokens.  A split writes its partial instead.
    auto tok = [&](int t2, int i) { return wt + 32 * t2 + 8 * (i >> 2) + 4 * hi + (i & 3); };
    if (UNI && XS && a.hq) {
        // the paired tile's gate (rows 0-63) and up (rows 64-127) values meet
        // in LDS as [token][row] with 132-float token rows; then
        // h = silu(g) * u of the tile's two 32-row blocks, quantized as
        // silu_quant8_kernel does, 8 lanes x 4 values per (block, token),
        // written in the split layout (codes of block b, token t at
        // ((2b + half) n + t) 16, scales [b][t] after the n * inter code bytes)
        constexpr int kHs = kGemmRows + 4;
        static_assert(TT * kHs * 4 <= kGemmBufs * G::STAGE, "the fp32 tile fits the stage buffers");
        float *hs = reinterpret_cast<float *>(smem);
        __syncthreads();   // every wave is done with the last stage
#pragma unroll
        for (int t2 = 0; t2 < T2; t2++)
#pragma unroll
            for (int i = 0; i < 16; i++) hs[tok(t2, i) * kHs + wr + l32] = acc[t2][i];
        __syncthreads();
        const int n = a.n_tok, inter = a.seg[0].rows;
        float *scales = reinterpret_cast<float *>(a.hq + (size_t)n * inter);
        // (block, token) units in block-major order: consecutive units are
        // consecutive tokens, so a wave's code stores are 128 contiguous bytes
#pragma unroll
        for (int j = 0; j < 2 * TT * 8 / kGemmThreads; j++) {
            const int q = tid + kGemmThreads * j;
            const int e = q & 7, bl = q / (8 * TT), tk = (q >> 3) & (TT - 1);
            const int t = tok0 + tk;
            if (t >= n) continue;   // whole 8-lane groups share t
            const float4 g4 = *reinterpret_cast<const float4 *>(hs + tk * kHs + 32 * bl + 4 * e);
            const float4 u4 = *reinterpret_cast<const float4 *>(hs + tk * kHs + 64 + 32 * bl + 4 * e);
            const float h[4] = {silu_mul(g4.x, u4.x), silu_mul(g4.y, u4.y), silu_mul(g4.z, u4.z),
                                silu_mul(g4.w, u4.w)};
            const size_t gb = 2 * (size_t)rt + bl;
            quantize8x4(h, scales + gb * n + t, a.hq + ((2 * gb + (e >> 2)) * n + t) * 16 + 4 * (e & 3), e == 0);
        }
        return;
    }
    const int r = row0 + wr + l32;
    if (r >= a.rows_total) return;
    float *y;
    int ldy;
    if (a.ksplit > 1) {
        y = a.part + (size_t)ks * a.n_tok * a.rows_total + r;
        ldy = a.rows_total;
    } else {
        const bool s0 = r < a.seg_end[0], s1 = !s0 && r < a.seg_end[1];
        y = (s0 ? a.seg[0].y : (s1 ? a.seg[1].y : a.seg[2].y)) + (r - (s0 ? 0 : (s1 ? a.seg_end[0] : a.seg_end[1])));
        ldy = s0 ? a.seg[0].rows : (s1 ? a.seg[1].rows : a.seg[2].rows);
    }
#pragma unroll
    for (int t2 = 0; t2 < T2; t2++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = tok0 + tok(t2, i);
            if (t < a.n_tok) y[(size_t)t * ldy] = acc[t2][i];
        }
}

// The split-K sum: y of (token t, row r) is the splits' partials added in
// split order (the same order on every launch).  VEC: four rows per thread
// (every segment's rows a multiple of 4, 16-byte aligned partials and
// outputs); the loads of four splits are in flight together.  Bound by those
// loads' latency: 16 splits of 100 x 4,096 (26 MB) took 7.1 us a row per
// thread, one split after another.
template <bool VEC>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemvArgs a) {
    typedef float vec_t __attribute__((ext_vector_type(VEC ? 4 : 1)));
    constexpr int W = VEC ? 4 : 1;
    const size_t total = (size_t)a.n_tok * a.rows_total;
    for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * W; i < total; i += (size_t)gridDim.x * 256 * W) {
        const float *p = a.part + i;
        vec_t acc = *reinterpret_cast<const vec_t *>(p);
        int s = 1;
        for (; s + 4 <= a.ksplit; s += 4) {
            vec_t v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = *reinterpret_cast<const vec_t *>(p + (size_t)(s + k) * total);
#pragma unroll
            for (int k = 0; k < 4; k++) acc += v[k];
        }
        for (; s < a.ksplit; s++) acc += *reinterpret_cast<const vec_t *>(p + (size_t)s * total);
        const int t = (int)(i / a.rows_total), r = (int)(i - (size_t)t * a.rows_total);
        const bool s0 = r < a.seg_end[0], s1 = !s0 && r < a.seg_end[1];
        float *y = s0 ? a.seg[0].y : (s1 ? a.seg[1].y : a.seg[2].y);
        const int rows = s0 ? a.seg[0].rows : (s1 ? a.seg[1].rows : a.seg[2].rows);
        const int lr = r - (s0 ? 0 : (s1 ? a.seg_end[0] : a.seg_end[1]));
        *reinterpret_cast<vec_t *>(y + (size_t)t * rows + lr) = acc;
    }
}

// The split-K sum of the MLP's gate and up matmul and silu_quant8_kernel's
// work in one launch: thread (token, block, lane of 8) adds four gate and four
// up values' partials in split order, stores them, forms h = silu(g) * u and
// quantizes the block with its 7 neighbours, into the split layout (a.hq_xs)
// or block_q8 rows at a.hq.  The same values as the two launches, without the
// second's launch and read.  seg[0].y and seg[1].y 16-byte aligned.
__global__ __launch_bounds__(256) void gemm_reduce_silu_kernel(GemvArgs a) {
    const int inter = a.seg[0].rows, nbi = inter / kQK, n = a.n_tok;
    const size_t k = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= (size_t)n * nbi * 8) return;   // whole 8-lane groups
    const int e = (int)(k & 7);
    const size_t tb = k >> 3;
    const int t = (int)(tb / nbi), b = (int)(tb - (size_t)t * nbi);
    const size_t total = (size_t)n * a.rows_total;
    const float *pg = a.part + (size_t)t * a.rows_total + kQK * b + 4 * e, *pu = pg + inter;
    v4f g = *reinterpret_cast<const v4f *>(pg), u = *reinterpret_cast<const v4f *>(pu);
    int s = 1;
    for (; s + 2 <= a.ksplit; s += 2) {
        const v4f g0 = *reinterpret_cast<const v4f *>(pg + s * total), u0 = *reinterpret_cast<const v4f *>(pu + s * total);
        const v4f g1 = *reinterpret_cast<const v4f *>(pg + (s + 1) * total);
        const v4f u1 = *reinterpret_cast<const v4f *>(pu + (s + 1) * total);
        g += g0;
        u += u0;
        g += g1;
        u += u1;
    }
    if (s < a.ksplit) {
        g += *reinterpret_cast<const v4f *>(pg + s * total);
        u += *reinterpret_cast<const v4f *>(pu + s * total);
    }
    const size_t at = (size_t)t * inter + kQK * b + 4 * e;
    *reinterpret_cast<v4f *>(a.seg[0].y + at) = g;
    *reinterpret_cast<v4f *>(a.seg[1].y + at) = u;
    const float h[4] = {silu_mul(g.x, u.x), silu_mul(g.y, u.y), silu_mul(g.z, u.z), silu_mul(g.w, u.w)};
    if (a.hq_xs) {
        float *scales = reinterpret_cast<float *>(a.hq + (size_t)n * inter);
        quantize8x4(h, scales + (size_t)b * n + t, a.hq + ((size_t)(2 * b + (e >> 2)) * n + t) * 16 + 4 * (e & 3), e == 0);
    } else {
        unsigned char *blk = a.hq + tb * kBlockBytes;
        quantize8x4(h, reinterpret_cast<float *>(blk), blk + 4 + 4 * e, e == 0);
    }
}

int env_int(const char *name, int dflt) {
    const char *s = getenv(name);
    return (s && *s) ? atoi(s) : dflt;
}

// Rows per wave: enough work-groups to put two on every CU where the row
// count allows (TQ_HIP_GEMV_RW=1|2|4 overrides).  Four rows only where a row
// has 4 or more 64-block groups, or for Q4: Q8 rows of 4096 columns (two
// groups) keep more waves streaming at two rows (8B gate/up, 28672 x 4096:
// model forward 437 -> 449 tokens/s), while 10240 x 8192 is faster at four
// (36.1 against 38.2 us).
int pick_rw(int rows_total, int ng, bool q4) {
    const int forced = env_int("TQ_HIP_GEMV_RW", 0);
    if (forced == 1 || forced == 2 || forced == 4) return forced;
    if (rows_total >= 4 * kGemvWaves * 512 && (q4 || ng >= 4)) return 4;
    if (rows_total >= 2 * kGemvWaves * 512) return 2;
    return 1;
}

// Groups per row per pass: up to 8 (row, group) units in flight per wave (16
// for Q4, whose units are half the bytes), never more groups than a row has
// (TQ_HIP_GEMV_GC=1|2|4 overrides).
int pick_gc(int ng, int rw, bool q4) {
    const int forced = env_int("TQ_HIP_GEMV_GC", 0);
    int gc = (forced == 1 || forced == 2 || forced == 4) ? forced : (q4 ? 16 : 8) / rw;
    if (gc > 4) gc = 4;
    while (gc > 1 && gc / 2 >= ng) gc /= 2;
    return gc;
}

// Largest token count per launch whose staged rows fit the LDS budget
// (fp32 input: 1 or 2 rows, quantized in LDS).
int pick_tokens(int nb, bool xf) {
    for (int t : {8, 4, 2, 1})
        if ((!xf || t <= 2) && lds_bytes(t, nb, xf) <= kMaxStageBytes) return t;
    return 0;
}

template <int T, int RW, int GC, bool XF, bool Q4>
hipError_t launch_t(const GemvArgs &a, hipStream_t s) {
    const int waves = (a.rows_total + RW - 1) / RW;
    const int grid = (waves + kGemvWaves - 1) / kGemvWaves;
    const size_t lds = (lds_bytes(T, a.nb, XF) + 15) & ~(size_t)15;
    if (lds > kDefaultLdsLimit) {
        static bool opted = false;   // once per instantiation (and process)
        if (!opted) {
            const hipError_t e = hipFuncSetAttribute((const void *)gemv_q8_kernel<T, RW, GC, XF, Q4>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     (int)kMaxStageBytes);
            if (e != hipSuccess) return e;
            opted = true;
        }
    }
    hipLaunchKernelGGL((gemv_q8_kernel<T, RW, GC, XF, Q4>), dim3(grid), dim3(kThreads), lds, s, a);
    return hipGetLastError();
}

template <int RW, int GC, bool Q4>
hipError_t launch_tok_f(const GemvArgs &a, int tmax, bool xf, hipStream_t s) {
    if (xf) return tmax == 2 ? launch_t<2, RW, GC, true, Q4>(a, s) : launch_t<1, RW, GC, true, Q4>(a, s);
    switch (tmax) {
        case 8: return launch_t<8, RW, GC, false, Q4>(a, s);
        case 4: return launch_t<4, RW, GC, false, Q4>(a, s);
        case 2: return launch_t<2, RW, GC, false, Q4>(a, s);
        default: return launch_t<1, RW, GC, false, Q4>(a, s);
    }
}

template <int RW, int GC>
hipError_t launch_tok(const GemvArgs &a, int tmax, bool xf, hipStream_t s) {
    return a.q4 ? launch_tok_f<RW, GC, true>(a, tmax, xf, s) : launch_tok_f<RW, GC, false>(a, tmax, xf, s);
}

hipError_t launch_gemv(const GemvArgs &a, int tcap, bool xf, int rw, int gc, hipStream_t s) {
    switch (rw * 16 + gc) {
        case 0x11: return launch_tok<1, 1>(a, tcap, xf, s);
        case 0x12: return launch_tok<1, 2>(a, tcap, xf, s);
        case 0x14: return launch_tok<1, 4>(a, tcap, xf, s);
        case 0x21: return launch_tok<2, 1>(a, tcap, xf, s);
        case 0x22: return launch_tok<2, 2>(a, tcap, xf, s);
        case 0x24: return launch_tok<2, 4>(a, tcap, xf, s);
        case 0x41: return launch_tok<4, 1>(a, tcap, xf, s);
        case 0x44: return launch_tok<4, 4>(a, tcap, xf, s);
        default: return launch_tok<4, 2>(a, tcap, xf, s);
    }
}

// From how many tokens on (block_q8 input) the unsplit MFMA GEMM runs instead
// of GEMV launches of tmax tokens each (TQ_HIP_GEMM_MIN_TOKENS overrides).
// The line is a matter of precision, not of time: a GEMV row is 64 short sums
// in a tree, a GEMM row one chain over its blocks.  Distance from the 64-bit
// product of the same codes, GEMV / GEMM: 4,096 columns 8.0e-8 / 2.05e-7, 8,192
// 8.6e-8 / 2.9e-7, 14,336 9.2e-8 / 3.8e-7.  So it stays where an earlier, slower
// GEMM (0.0183 us per column for its first round of tiles, against 5 TB/s and 2
// us per GEMV launch) crossed the GEMV launches: 6144 x 4096 from 81 tokens,
// 28672 x 4096 from 22, 4096 x 14336 from 70.  The present GEMM is ahead from 33,
// 12 and 30 on (Q4 43), us, GEMM against GEMV:
//   6144 x 4096    16 tokens 33 / 18    32: 33 / 33    64: 34 / 63    96: 58 / 94
//   28672 x 4096   8: 48 / 35    12: 48 / 55    16: 37 / 53    20: 38 / 75
//   4096 x 14336   16: 105 / 58   32: 105 / 116  64: 106 / 231   96: 190 / 345
//   the same, Q4   28: 114 / 75   40: 114 / 106  48: 114 / 126   64: 114 / 164
int gemm_min_tokens(int rows, int cols, int tmax) {
    const int v = env_int("TQ_HIP_GEMM_MIN_TOKENS", 0);
    if (v > 0) return v;
    const double chunk_us = (double)rows * cols * (kBlockBytes / (double)kQK) / 5.0e6 + 2.0;
    const double gemm_us = 0.0183 * cols + 2.0;
    const int n = (int)(tmax * gemm_us / chunk_us) + 1;
    return n < 16 ? 16 : (n > 256 ? 256 : n);   // up to 15 tokens a row's bits are the GEMV's whatever its batch
}

// Every 128-row tile inside one segment (segment ends on tile boundaries) and
// 32-bit copy offsets: the uniform-base copies apply.
bool gemm_uniform(const GemvArgs &a) {
    for (int i = 0; i < kMaxSegs; i++) {
        if (a.seg_end[i] < a.rows_total && a.seg_end[i] % kGemmRows != 0) return false;
        const size_t rowb = a.q4 ? (size_t)a.cols / 2 : (size_t)a.cols;
        if ((size_t)a.seg[i].rows * (rowb + 4 * (size_t)a.nb) >= ((size_t)1 << 31)) return false;
    }
    return (size_t)a.n_tok * a.nb * kBlockBytes < ((size_t)1 << 31);
}

// Work-groups of a launch without K splits (row tiles per XCD rounded up).
long gemm_wgs(int rows, int n_tok, int toks) {
    return ((long)(rows + kGemmRows - 1) / kGemmRows + 7) / 8 * 8 * ((n_tok + toks - 1) / toks);
}

// Tokens per tile of a launch over n_tok: 64 where one such tile holds them,
// and up to 320 tokens where 128-token tiles would be half padding at the end
// (an odd count of 64s; a 64-token tile takes 0.54 of a 128-token one).  No
// bit depends on it: the K splits do not follow the tile (gemm_ksplit).  MLP,
// us with 64 / 128, Q8 then Q4: 4,096 x 14,336 over 129 tokens 124 / 139, 126 / 141,
// 300: 204 / 207, 212 / 210; 8,192 x 28,672, 300: 740 / 823, 722 / 814; 2,048 x 5,632,
// 300: 59 / 73, 61 / 77; 8,192 x 5,120, 300: 164 / 161, 173 / 167 (400 tiles of 10,240
// rows in two splits, 1.6 rounds of the CUs, against 0.9).  Choosing by whole
// rounds lost more than it gained (129 tokens 139 again).  At 420 tokens of 4,096 x
// 14,336 the gain was gone (277 / 282, 283 / 277) and at 550 a loss (371 / 345).
constexpr int kGemmSmallToks = 320;

int gemm_toks(int n_tok) { return n_tok <= 64 || (n_tok <= kGemmSmallToks && (n_tok + 63) / 64 % 2) ? 64 : 128; }

template <int TT>
hipError_t launch_gemm_t(const GemvArgs &u, bool bx4, unsigned grid, hipStream_t s) {
    const size_t lds = (size_t)kGemmBufs * GemmTile<TT>::STAGE;
    if (lds > kDefaultLdsLimit) {
        static bool opted = false;   // once per tile (and process)
        if (!opted) {
            for (const void *f : {(const void *)gemm_q8_kernel<true, false, false, false, TT>,
                                  (const void *)gemm_q8_kernel<false, false, false, false, TT>,
                                  (const void *)gemm_q8_kernel<true, true, false, false, TT>,
                                  (const void *)gemm_q8_kernel<false, true, false, false, TT>,
                                  (const void *)gemm_q8_kernel<true, false, true, false, TT>,
                                  (const void *)gemm_q8_kernel<true, true, true, false, TT>,
                                  (const void *)gemm_q8_kernel<true, false, true, true, TT>,
                                  (const void *)gemm_q8_kernel<true, true, true, true, TT>}) {
                const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                if (e != hipSuccess) return e;
            }
            opted = true;
        }
    }
    const dim3 g(grid), b(kGemmThreads);
    if (u.q4) {
        if (u.xs)
            hipLaunchKernelGGL((gemm_q8_kernel<true, true, true, true, TT>), g, b, lds, s, u);
        else if (bx4 && u.uni_tiles)
            hipLaunchKernelGGL((gemm_q8_kernel<true, true, true, false, TT>), g, b, lds, s, u);
        else if (bx4)
            hipLaunchKernelGGL((gemm_q8_kernel<true, true, false, false, TT>), g, b, lds, s, u);
        else
            hipLaunchKernelGGL((gemm_q8_kernel<false, true, false, false, TT>), g, b, lds, s, u);
    } else {
        if (u.xs)
            hipLaunchKernelGGL((gemm_q8_kernel<true, false, true, true, TT>), g, b, lds, s, u);
        else if (bx4 && u.uni_tiles)
            hipLaunchKernelGGL((gemm_q8_kernel<true, false, true, false, TT>), g, b, lds, s, u);
        else if (bx4)
            hipLaunchKernelGGL((gemm_q8_kernel<true, false, false, false, TT>), g, b, lds, s, u);
        else
            hipLaunchKernelGGL((gemm_q8_kernel<false, false, false, false, TT>), g, b, lds, s, u);
    }
    return hipGetLastError();
}

hipError_t launch_gemm(const GemvArgs &a, int ksplit, hipStream_t s) {
    const int toks = gemm_toks(a.n_tok);
    const long grid = gemm_wgs(a.rows_total, a.n_tok, toks) * ksplit;
    if (grid > INT32_MAX) return hipErrorInvalidValue;
    const bool bx4 = (((uintptr_t)a.xq & 15) == 0) && a.nb % kGemmKB == 0;
    GemvArgs u = a;
    u.ksplit = ksplit;
    u.uni_tiles = gemm_uniform(a);
    if (a.xs && !(bx4 && u.uni_tiles)) return hipErrorInvalidValue;   // the caller's plan and this disagree
    // the hidden rows instead of gate and up: two segments of equal rows; in
    // paired tiles (unsplit) a split-layout GEMM and rows a multiple of 64
    if (a.hq && (a.seg[0].rows != a.seg[1].rows || a.rows_total != 2 * a.seg[0].rows ||
                 (ksplit == 1 ? !a.xs || !a.hq_xs || a.seg[0].rows % 64 != 0 : a.seg[0].rows % kQK != 0)))
        return hipErrorInvalidValue;
    if (ksplit > 1) u.hq = nullptr;   // the reduce launch's
    const hipError_t e = toks == 64 ? launch_gemm_t<64>(u, bx4, (unsigned)grid, s)
                                    : launch_gemm_t<128>(u, bx4, (unsigned)grid, s);
    if (e != hipSuccess || ksplit == 1) return e;
    u.hq = a.hq;
    const size_t total = (size_t)a.n_tok * a.rows_total;
    if (u.hq) {
        const size_t threads = (size_t)a.n_tok * (a.seg[0].rows / kQK) * 8;
        hipLaunchKernelGGL(gemm_reduce_silu_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, u);
        return hipGetLastError();
    }
    bool vec = ((uintptr_t)a.part & 15) == 0;
    for (int i = 0; i < kMaxSegs; i++)
        vec = vec && (((uintptr_t)a.seg[i].y & 15) == 0) && a.seg[i].rows % 4 == 0 && a.seg_end[i] % 4 == 0;
    const size_t per = vec ? 4 : 1;
    const size_t blocks = std::min<size_t>((total / per + 255) / 256, 2048);
    if (vec)
        hipLaunchKernelGGL(gemm_reduce_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, s, u);
    else
        hipLaunchKernelGGL(gemm_reduce_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, s, u);
    return hipGetLastError();
}

// Split-K GEMM while the tiles alone leave CUs of the 256 idle (each tile
// then runs the whole K loop): K is cut into S runs of stages, as many as
// keep a grid of 128-token tiles within one round of 512 work-groups (two per
// CU), each split writing a partial tile that one more launch sums in split
// order.  S is counted in 128-token tiles whatever the tile is, so that a row's
// bits and the length of its sums do not change with the padding.  With S from
// the 64-token tiles (fewer and longer sums; 300 rows of 4,096 x 14,336 203 for 214
// us, of 8,192 x 28,672 816 for 794) an attention layer over 300 tokens was 4.29e-4
// from a 64-bit evaluation over 48 seeds, and is 4.16e-4.  MLP at the 8B shape, us with Q8 / Q4 weights over 16, 64, 100, 256
// rows: 63 / 56, 71 / 63, 94 / 93, 144 / 145; with 16 x 16 products and only
// 128-token tiles 112 / 109, 131 / 126, 144 / 139, 197 / 207.  The least is 16
// tokens, as without a workspace: up to 15 a row's bits are the GEMV's whatever
// its batch.  (Splits from 9 tokens took 62 / 56 for 90 / 75 us of GEMV launches
// there, with other bits.)
constexpr int kSplitWgs = 512;
constexpr int kSplitMinTokens = 16;

int gemm_ksplit(int rows, int cols, int n_tok) {
    if (n_tok < kSplitMinTokens) return 1;
    const long wgs = gemm_wgs(rows, n_tok, 128);
    // once every CU holds a tile, splitting adds occupancy but not CUs, and
    // the partials' traffic outweighs it (4,096 x 14,336 at 1,024 tokens)
    if (wgs >= kSplitWgs / 2) return 1;
    const int stages = (cols / kQK + kGemmKB - 1) / kGemmKB;
    long sp = kSplitWgs / wgs;
    if (sp > stages) sp = stages;
    return sp < 2 ? 1 : (int)sp;
}

// The GEMM launch run_gemv makes over n_tok rows of block_q8 input (its K
// split count), or 0 for GEMV launches.  With a workspace for the partials a
// few tokens take the split-K GEMM; otherwise the cost model decides.
int gemm_plan(const GemvArgs &a, int n_tok) {
    if (a.x != nullptr) return 0;
    const int ksplit = a.part ? gemm_ksplit(a.rows_total, a.cols, n_tok) : 1;
    if (ksplit > 1 && (size_t)ksplit * n_tok * a.rows_total <= a.part_floats && env_int("TQ_HIP_GEMM_SPLIT", 1) != 0)
        return ksplit;
    return n_tok >= gemm_min_tokens(a.rows_total, a.cols, pick_tokens(a.nb, false)) ? 1 : 0;
}

// Whether the matmul's input should be quantized into the split layout:
// internal callers (a partials workspace) whose launch is a GEMM with
// uniform-base copies over whole stages, xq 16-byte aligned
// (TQ_HIP_GEMM_XS=0 keeps block_q8 rows).
bool xs_layout(const GemvArgs &a, int n_tok, const void *xq) {
    if (!a.part || a.x || ((uintptr_t)xq & 15) || a.nb % kGemmKB || env_int("TQ_HIP_GEMM_XS", 1) == 0) return false;
    GemvArgs t = a;
    t.n_tok = n_tok;
    return gemm_plan(a, n_tok) > 0 && gemm_uniform(t);
}

// Runs the matmul over all tokens: one GEMM launch for many block_q8 rows,
// else GEMV launches of up to tmax tokens.  With fp32 input (a.x) each GEMV
// launch quantizes its rows in LDS.
int run_gemv(GemvArgs a, int n_tok, hipStream_t s) {
    const bool xf = a.x != nullptr;
    const int plan = gemm_plan(a, n_tok);
    if (plan > 0) {
        if ((size_t)n_tok * a.nb > (size_t)INT32_MAX / kBlockBytes) return TQ_HIP_EINVAL;
        a.n_tok = n_tok;
        return herr(launch_gemm(a, plan, s));
    }
    if (a.xs) return TQ_HIP_EINVAL;   // the split layout is for the GEMM only
    const int tmax = pick_tokens(a.nb, xf);
    if (tmax == 0) return TQ_HIP_EINVAL;
    const int rw = pick_rw(a.rows_total, a.ng, a.q4);
    const int gc = pick_gc(a.ng, rw, a.q4);
    const unsigned char *xq0 = a.xq;
    const float *x0 = a.x;
    unsigned char *out0 = a.xq_out;
    GemvSeg seg0[kMaxSegs];
    for (int i = 0; i < kMaxSegs; i++) seg0[i] = a.seg[i];
    for (int t0 = 0; t0 < n_tok; t0 += tmax) {
        const int nt = n_tok - t0 < tmax ? n_tok - t0 : tmax;
        int tcap = 1;
        while (tcap < nt) tcap *= 2;
        a.n_tok = nt;
        const size_t blk_off = (size_t)t0 * a.nb * kBlockBytes;
        a.xq = xq0 ? xq0 + blk_off : nullptr;
        a.x = x0 ? x0 + (size_t)t0 * a.cols : nullptr;
        a.xq_out = out0 ? out0 + blk_off : nullptr;
        for (int i = 0; i < kMaxSegs; i++)
            a.seg[i].y = seg0[i].y ? seg0[i].y + (size_t)t0 * seg0[i].rows : nullptr;
        const hipError_t e = launch_gemv(a, tcap, xf, rw, gc, s);
        if (e != hipSuccess) return herr(e);
    }
    return TQ_HIP_OK;
}

// fp32 input is quantized inside the matmul launch for one or two rows (one
// launch instead of two); more rows go through quantize_row_q8 into the
// workspace first, so that a launch still covers up to 8 of them.
bool fuse_quantize(const float *x, int n_tok, int nb) {
    return n_tok <= 2 && ((uintptr_t)x & 15) == 0 && lds_bytes(n_tok, nb, true) <= kMaxStageBytes;
}

bool aligned(const void *p, size_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

bool shape_ok(int rows, int cols) { return rows > 0 && cols > 0 && cols % kQK == 0; }

void init_args(GemvArgs &a, int cols) {
    a = GemvArgs{};
    a.cols = cols;
    a.nb = cols / kQK;
    a.ng = (a.nb + kGroupBlocks - 1) / kGroupBlocks;
}

int matmul_fmt(bool q4, const void *W, const block_q8 *xq, float *y, int rows, int cols, int n_tok,
               void *stream) {
    if (!shape_ok(rows, cols) || n_tok <= 0 || !W || !xq || !y || !aligned(W, 16) || !aligned(xq, 4) ||
        !aligned(y, 4))
        return TQ_HIP_EINVAL;
    GemvArgs a;
    init_args(a, cols);
    a.q4 = q4;
    a.seg[0] = GemvSeg{(const unsigned char *)W, y, rows};
    a.seg_end[0] = a.seg_end[1] = a.seg_end[2] = rows;
    a.rows_total = rows;
    a.xq = (const unsigned char *)xq;
    return run_gemv(a, n_tok, (hipStream_t)stream);
}

}  // namespace

extern "C" {

size_t tq_hip_q8_matrix_bytes(int rows, int cols) {
    if (!shape_ok(rows, cols)) return 0;
    return (size_t)rows * (size_t)(cols / kQK) * kBlockBytes;
}

int tq_hip_q8_pack(void *dst, const block_q8 *src, int rows, int cols, void *stream) {
    if (!shape_ok(rows, cols) || !dst || !src || !aligned(dst, 16) || !aligned(src, 4))
        return TQ_HIP_EINVAL;
    const long long n = (long long)rows * (cols / kQK);
    hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (unsigned char *)dst, (const unsigned char *)src, rows, cols / kQK);
    return herr(hipGetLastError());
}

int tq_hip_q8_unpack(block_q8 *dst, const void *src, int rows, int cols, void *stream) {
    if (!shape_ok(rows, cols) || !dst || !src || !aligned(src, 16) || !aligned(dst, 4))
        return TQ_HIP_EINVAL;
    const long long n = (long long)rows * (cols / kQK);
    hipLaunchKernelGGL(unpack_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (unsigned char *)dst, (const unsigned char *)src, rows, cols / kQK);
    return herr(hipGetLastError());
}

int tq_hip_matmul_q8_batch(const void *W, const block_q8 *xq, float *y, int rows, int cols, int n_tok,
                           void *stream) {
    return matmul_fmt(false, W, xq, y, rows, cols, n_tok, stream);
}

int tq_hip_matmul_q8(const void *W, const block_q8 *xq, float *y, int rows, int cols, void *stream) {
    return matmul_fmt(false, W, xq, y, rows, cols, 1, stream);
}

size_t tq_hip_q4_matrix_bytes(int rows, int cols) {
    if (!shape_ok(rows, cols)) return 0;
    return (size_t)rows * (size_t)(cols / kQK) * kBlockBytes4;
}

int tq_hip_q4_pack(void *dst, const block_q4 *src, int rows, int cols, void *stream) {
    if (!shape_ok(rows, cols) || !dst || !src || !aligned(dst, 16) || !aligned(src, 4)) return TQ_HIP_EINVAL;
    const long long n = (long long)rows * (cols / kQK);
    hipLaunchKernelGGL(pack4_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (unsigned char *)dst, (const unsigned char *)src, n);
    return herr(hipGetLastError());
}

int tq_hip_q4_unpack(block_q4 *dst, const void *src, int rows, int cols, void *stream) {
    if (!shape_ok(rows, cols) || !dst || !src || !aligned(src, 16) || !aligned(dst, 4)) return TQ_HIP_EINVAL;
    const long long n = (long long)rows * (cols / kQK);
    hipLaunchKernelGGL(unpack4_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (unsigned char *)dst, (const unsigned char *)src, n);
    return herr(hipGetLastError());
}

int tq_hip_matmul_q4_batch(const void *W, const block_q8 *xq, float *y, int rows, int cols, int n_tok,
                           void *stream) {
    return matmul_fmt(true, W, xq, y, rows, cols, n_tok, stream);
}

int tq_hip_matmul_q4(const void *W, const block_q8 *xq, float *y, int rows, int cols, void *stream) {
    return matmul_fmt(true, W, xq, y, rows, cols, 1, stream);
}

int tq_hip_project_qkv(const void *wq, const void *wk, const void *wv, int q_rows, int kv_rows,
                       int hidden, const float *xn, int n_tok, block_q8 *xq_ws, float *q, float *k,
                       float *v, void *stream) {
    return tq_project_qkv_fmt(false, wq, wk, wv, q_rows, kv_rows, hidden, xn, n_tok, xq_ws, q, k, v, stream);
}

int tq_hip_project_qkv_q4(const void *wq, const void *wk, const void *wv, int q_rows, int kv_rows,
                          int hidden, const float *xn, int n_tok, block_q8 *xq_ws, float *q, float *k,
                          float *v, void *stream) {
    return tq_project_qkv_fmt(true, wq, wk, wv, q_rows, kv_rows, hidden, xn, n_tok, xq_ws, q, k, v, stream);
}

int tq_hip_project_output(const void *wo, int rows, int cols, const float *attn, int n_tok,
                          block_q8 *xq_ws, float *out, void *stream) {
    return tq_project_output_fmt(false, wo, rows, cols, attn, n_tok, xq_ws, out, stream);
}

int tq_hip_project_output_q4(const void *wo, int rows, int cols, const float *attn, int n_tok,
                             block_q8 *xq_ws, float *out, void *stream) {
    return tq_project_output_fmt(true, wo, rows, cols, attn, n_tok, xq_ws, out, stream);
}

}  // extern "C"

// The matmul input of a (segments, workspace set): one or two rows quantized
// inside the GEMV launch; else quantize_row_q8 of every row into the
// workspace first, as block_q8 rows or, for a GEMM that reads it, in the
// split layout.
int quantize_input(GemvArgs &a, const float *x, int n_tok, int cols, void *xq_ws, hipStream_t s) {
    if (fuse_quantize(x, n_tok, a.nb)) {
        a.x = x;
        a.xq_out = (unsigned char *)xq_ws;
        return TQ_HIP_OK;
    }
    a.xs = aligned(x, 16) && xs_layout(a, n_tok, xq_ws);   // its quantizer loads 16 bytes
    const hipError_t e = a.xs ? tq_launch_quantize_split(x, (unsigned char *)xq_ws, n_tok, cols, s)
                              : tq_launch_quantize(x, (block_q8 *)xq_ws, n_tok * cols, s);
    if (e != hipSuccess) return herr(e);
    a.xq = (const unsigned char *)xq_ws;
    return TQ_HIP_OK;
}

int tq_project_qkv_fmt(bool q4, const void *wq, const void *wk, const void *wv, int q_rows, int kv_rows, int hidden,
                    const float *xn, int n_tok, block_q8 *xq_ws, float *q, float *k, float *v, void *stream,
                    float *part, size_t part_floats) {
    if (!shape_ok(q_rows, hidden) || kv_rows <= 0 || n_tok <= 0 || !wq || !wk || !wv || !xn ||
        !xq_ws || !q || !k || !v || !aligned(wq, 16) || !aligned(wk, 16) || !aligned(wv, 16) ||
        !aligned(xn, 4) || !aligned(xq_ws, 4) || !aligned(q, 4) || !aligned(k, 4) || !aligned(v, 4))
        return TQ_HIP_EINVAL;
    const hipStream_t s = (hipStream_t)stream;
    GemvArgs a;
    init_args(a, hidden);
    a.q4 = q4;
    a.seg[0] = GemvSeg{(const unsigned char *)wq, q, q_rows};
    a.seg[1] = GemvSeg{(const unsigned char *)wk, k, kv_rows};
    a.seg[2] = GemvSeg{(const unsigned char *)wv, v, kv_rows};
    a.seg_end[0] = q_rows;
    a.seg_end[1] = q_rows + kv_rows;
    a.seg_end[2] = q_rows + 2 * kv_rows;
    a.rows_total = a.seg_end[2];
    a.part = part;
    a.part_floats = part_floats;
    const int rc = quantize_input(a, xn, n_tok, hidden, xq_ws, s);
    return rc != TQ_HIP_OK ? rc : run_gemv(a, n_tok, s);
}

int tq_project_output_fmt(bool q4, const void *wo, int rows, int cols, const float *attn, int n_tok,
                       block_q8 *xq_ws, float *out, void *stream, float *part, size_t part_floats) {
    if (!shape_ok(rows, cols) || n_tok <= 0 || !wo || !attn || !xq_ws || !out || !aligned(wo, 16) ||
        !aligned(attn, 4) || !aligned(xq_ws, 4) || !aligned(out, 4))
        return TQ_HIP_EINVAL;
    const hipStream_t s = (hipStream_t)stream;
    GemvArgs a;
    init_args(a, cols);
    a.q4 = q4;
    a.seg[0] = GemvSeg{(const unsigned char *)wo, out, rows};
    a.seg_end[0] = a.seg_end[1] = a.seg_end[2] = rows;
    a.rows_total = rows;
    a.part = part;
    a.part_floats = part_floats;
    const int rc = quantize_input(a, attn, n_tok, cols, xq_ws, s);
    return rc != TQ_HIP_OK ? rc : run_gemv(a, n_tok, s);
}

static void output_args(GemvArgs &a, bool q4, const void *wo, int rows, int cols, float *out, float *part,
                        size_t part_floats) {
    init_args(a, cols);
    a.q4 = q4;
    a.seg[0] = GemvSeg{(const unsigned char *)wo, out, rows};
    a.seg_end[0] = a.seg_end[1] = a.seg_end[2] = rows;
    a.rows_total = rows;
    a.part = part;
    a.part_floats = part_floats;
}

bool tq_project_output_takes_xs(bool q4, const void *wo, int rows, int cols, int n_tok, const void *xq_ws,
                                float *part, size_t part_floats) {
    if (!shape_ok(rows, cols) || n_tok <= 2 || !wo || !xq_ws || !aligned(wo, 16)) return false;
    GemvArgs a;
    output_args(a, q4, wo, rows, cols, nullptr, part, part_floats);
    return xs_layout(a, n_tok, xq_ws);
}

int tq_project_output_xs(bool q4, const void *wo, int rows, int cols, const void *xq_ws, int n_tok, float *out,
                         void *stream, float *part, size_t part_floats) {
    if (!out || !aligned(out, 4) || !tq_project_output_takes_xs(q4, wo, rows, cols, n_tok, xq_ws, part, part_floats))
        return TQ_HIP_EINVAL;
    GemvArgs a;
    output_args(a, q4, wo, rows, cols, out, part, part_floats);
    a.xs = true;
    a.xq = (const unsigned char *)xq_ws;
    return run_gemv(a, n_tok, (hipStream_t)stream);
}

// Partial floats a split-K GEMM of rows x cols needs for any token count up
// to n_cap: the largest S * n over the token-tile counts that still split.
size_t tq_gemm_partial_floats(int rows, int cols, int n_cap) {
    if (rows <= 0 || cols <= 0 || n_cap < kSplitMinTokens) return 0;
    size_t most = 0;
    for (int tiles = 1; (long)(tiles - 1) * 128 < n_cap; tiles++) {
        const int n = n_cap < tiles * 128 ? n_cap : tiles * 128;
        const int sp = gemm_ksplit(rows, cols, n);
        if (sp < 2) break;
        const size_t need = (size_t)sp * n * rows;
        if (need > most) most = need;
    }
    return most;
}

extern "C" {

static size_t mlp_ws(int hidden, int inter, int n, size_t *off_gate, size_t *off_up, size_t *off_xq,
                     size_t *off_part, size_t *part_floats) {
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    size_t o = 0;
    *off_gate = o;
    o += al((size_t)n * inter * 4);
    *off_up = o;
    o += al((size_t)n * inter * 4);
    *off_xq = o;
    o += al((size_t)n * (size_t)(hidden > inter ? hidden : inter) / kQK * kBlockBytes);
    // split-K partials of the gate/up and the down matmuls (one at a time)
    const size_t pg = tq_gemm_partial_floats(2 * inter, hidden, n), pd = tq_gemm_partial_floats(hidden, inter, n);
    *part_floats = pg > pd ? pg : pd;
    *off_part = o;
    o += al(*part_floats * 4);
    return o;
}

static bool mlp_ok(const tq_hip_mlp_weights *w, int n) {
    return w && n > 0 && w->wgate && w->wup && w->wdown && shape_ok(w->inter, w->hidden) &&
           shape_ok(w->hidden, w->inter) && aligned(w->wgate, 16) && aligned(w->wup, 16) &&
           aligned(w->wdown, 16) && (w->format == TQ_HIP_FORMAT_Q8 || w->format == TQ_HIP_FORMAT_Q4);
}

size_t tq_hip_mlp_ws_bytes(const tq_hip_mlp_weights *w, int n) {
    if (!mlp_ok(w, n)) return 0;
    size_t a, b, c, d, e;
    return mlp_ws(w->hidden, w->inter, n, &a, &b, &c, &d, &e);
}

int tq_hip_mlp_layer_async(const tq_hip_mlp_weights *w, int n, const float *d_xn, float *d_out, void *d_ws,
                           size_t ws_bytes, void *stream) {
    if (!mlp_ok(w, n) || !d_xn || !d_out || !d_ws || !aligned(d_ws, 16) || !aligned(d_xn, 4) ||
        !aligned(d_out, 4))
        return TQ_HIP_EINVAL;
    size_t og, ou, ox, op, pf;
    if (ws_bytes < mlp_ws(w->hidden, w->inter, n, &og, &ou, &ox, &op, &pf)) return TQ_HIP_EINVAL;
    unsigned char *ws = (unsigned char *)d_ws;
    float *gate = (float *)(ws + og), *up = (float *)(ws + ou);
    float *part = (float *)(ws + op);
    block_q8 *xq = (block_q8 *)(ws + ox);
    const hipStream_t s = (hipStream_t)stream;
    // model/mlp.c:9-11: quantize xn, then the gate and up matmuls in one launch
    const bool q4 = w->format == TQ_HIP_FORMAT_Q4;
    GemvArgs a;
    init_args(a, w->hidden);
    a.q4 = q4;
    a.seg[0] = GemvSeg{(const unsigned char *)w->wgate, gate, w->inter};
    a.seg[1] = GemvSeg{(const unsigned char *)w->wup, up, w->inter};
    a.seg_end[0] = w->inter;
    a.seg_end[1] = a.seg_end[2] = 2 * w->inter;
    a.rows_total = 2 * w->inter;
    a.part = part;
    a.part_floats = pf;
    int rc = quantize_input(a, d_xn, n, w->hidden, xq, s);
    if (rc != TQ_HIP_OK) return rc;
    // :14 the down matmul, over :12-13 silu_mul with the hidden rows quantized
    GemvArgs d;
    init_args(d, w->inter);
    d.q4 = q4;
    d.seg[0] = GemvSeg{(const unsigned char *)w->wdown, d_out, w->hidden};
    d.seg_end[0] = d.seg_end[1] = d.seg_end[2] = w->hidden;
    d.rows_total = w->hidden;
    d.part = part;
    d.part_floats = pf;
    // Where the gate/up matmul is a GEMM it leaves the quantized hidden rows
    // itself.  Unsplit over the split layout, when the down matmul reads the
    // split layout too: its tiles pair 64 rows of both matrices and their
    // epilogue writes them (into the gate rows' space; no gate and up rows).
    // Split: its reduce launch writes them beside gate and up, in the layout
    // the down matmul reads, over the quantized input.  Otherwise one more
    // launch forms them.  TQ_HIP_MLP_FUSED=0 keeps that launch.
    const int plan = n < kSplitMinTokens ? 0 : gemm_plan(a, n);
    const bool fuse = plan > 0 && env_int("TQ_HIP_MLP_FUSED", 1) != 0;
    const bool fused = fuse && a.xs && plan == 1 && w->inter % 64 == 0 && xs_layout(d, n, gate);
    const bool fused_split = fuse && plan > 1;
    d.xs = fused || xs_layout(d, n, xq);
    if (fused || fused_split) {
        a.hq = fused ? (unsigned char *)gate : (unsigned char *)xq;
        a.hq_xs = d.xs;
    }
    rc = run_gemv(a, n, s);
    if (rc != TQ_HIP_OK) return rc;
    if (fused || fused_split) {
        d.xq = a.hq;
        return run_gemv(d, n, s);
    }
    const hipError_t e = d.xs ? tq_launch_silu_quant_split(gate, up, (unsigned char *)xq, n, w->inter, s)
                              : tq_launch_silu_quant(gate, up, xq, (long)n * w->inter, s);
    if (e != hipSuccess) return herr(e);
    d.xq = (const unsigned char *)xq;
    return run_gemv(d, n, s);
}

}  // extern "C"
