// moa_full_attention.hip -- ops::full_attention_first_page / ops::full_attention_page
// (FO/src/ops.rs:148-174; FO/src/device/full/attention.rs): decode attention of a full-attention
// layer over one 512-slot page of its cache, folded into a running softmax state.
//
// The layer has 16 query heads and one KV head of 512 (FO/src/axes.rs: Gf, Df, Tf). For token row
// m and head h the state after pages 0..p is
//   running_max[h] = the largest score q_h . k_t (scale 1.0) over the valid slots seen so far,
//   running_sum[h] = sum of exp(s_t - running_max[h]) over them,
//   out[h]         = bf16(sum of exp(s_t - running_max[h]) v_t),
// where a slot is valid when its mask value is non-zero. The first page starts the state; each
// later page rescales the old state by exp(old max - new max) and adds its own terms, as
// attend_next_page does. full_attention_output divides out by running_sum. This is the softmax
// of the CPU reference over the valid slots (gemma4.py:180-184, causal SDPA with scale 1.0); the
// RNGD kernel takes its page max over every slot, rounds scores and weights to bf16 and adds 1e-6
// to each page sum, which moves results within rounding.
//
// Two launches per page for up to 16 rows (for more, fattn_rows_kernel below takes the first's place):
//  1. fattn_partial_kernel, grid (8 slot chunks, 4 dim blocks, M): workgroup (c, b, m) scores the
//     64 slots of chunk c against all 16 heads on the matrix cores (v_mfma_f32_16x16x32_bf16: the
//     heads as A rows, K rows as B columns, each wave a quarter of the 512 dims), takes each
//     head's max and the f32 exp weights, and multiplies them into its 128 dims of V (V staged
//     through LDS, where the B operand's slot-major gather is cheap). A weight enters the MFMA as two bf16 parts, high
//     and low (about 16 significant bits; one bf16 part alone would put a 2^-9 relative error on
//     every weight). It writes the chunk's per-head max, sum and partial out (f32).
//  2. fattn_combine_kernel, grid (16 heads, M): merges the 8 chunks with the old state and writes
//     the new one. One workgroup owns a head's state, so no other reads it while it is replaced.
//
// moa_full_attention computes the same state over pages 0 .. P - 1 in two launches instead of 2 P (more where
// the rows' records would not fit the scratch); with few rows times pages:
// the partial pass runs over every page at once -- up to 8 pages with the dim-split kernel (one
// chunk per workgroup), beyond with fattn_span_kernel (a workgroup takes a span of chunks over all
// dims with an online softmax; at most 256 records per row) -- and fattn_merge_kernel merges the
// records with a grid of (16 heads, 8 dim blocks): no old state is read, so the split is free of
// races. With more, fattn_rows_kernel shares every tile of K and V among four token rows.
#include <hip/hip_runtime.h>

#include "moa_device.h"
#include "moa_internal.h"

namespace moa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int kFaBlock = 256;
constexpr int kFaChunk = 64;                  // slots per workgroup
constexpr int kFaDims = kDf / kFaDimBlocks;   // 128 dims of V per workgroup
constexpr int kFaVStride = kFaDims + 4;       // LDS row of the V slice, in elements (8-byte aligned rows)
constexpr int kFaPStride = kFaChunk + 8;      // LDS row of the weights, in elements (16-byte aligned rows)
static_assert(kFaChunks * kFaChunk == kTf && kFaRec == 2 * kGf + kGf * kDf, "full attention tiling");

__device__ __forceinline__ bf16x8 as_bf16x8(const uint4& v) { return __builtin_bit_cast(bf16x8, v); }

// Workgroup (x, b, m) of the partial pass: chunks u = x * cpw .. min(x * cpw + cpw, nchunks) - 1 of
// the row's slots (chunk u = slots 64 (u % 8) .. + 63 of page u / 8; pages lie kTf * kDf apart),
// dims 128 b .. 128 b + 127 of V. Across its chunks it keeps an online softmax per head: the
// running max, the sum of exp and out for its dims, rescaled whenever the max grows. Its record
// of part (record x of row m, kFaRec floats): max[16], sum[16], out[16][512] (its 128 dims).
//
// Scores are split by dims: wave w multiplies dims 128 w .. 128 w + 127 of the chunk's 64 K rows
// (four 16-slot tiles) with the 16 heads, so each wave loads a quarter of q once; the four partial
// score tiles meet in LDS. Two register stages hold a chunk's K rows and V slice: the next chunk's
// loads go out at the top of each step, ahead of the current chunk's work.
__global__ __launch_bounds__(kFaBlock) void fattn_partial_kernel(const uint16_t* __restrict__ q,
                                                                 const uint16_t* __restrict__ kc,
                                                                 const uint16_t* __restrict__ vc,
                                                                 const float* __restrict__ mask, int mask_page_stride,
                                                                 int nchunks, int cpw, float* part) {
    __shared__ __attribute__((aligned(16))) uint16_t vs[kFaChunk * kFaVStride];
    __shared__ __attribute__((aligned(16))) uint16_t ps[2][kGf * kFaPStride];  // exp weights: bf16 high, low parts
    __shared__ float sp[4][kGf * kFaChunk];                                   // per-wave partial scores [head][slot]
    __shared__ float red_m[4][kGf], red_l[4][kGf];
    const int b = blockIdx.y, m = blockIdx.z;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l16 = lane & 15, g = lane >> 4;
    const int u0 = blockIdx.x * cpw, u1 = min(u0 + cpw, nchunks);

    // Lane l feeds head l % 16 and, of tile st, slot 16 st + l % 16, k 128 w + 32 j + 8 (l / 16) .. + 7
    // of step j. The V slice (64 rows x 128 dims = 1024 units of 16 bytes) is spread as units
    // t + 256 i. The lane's softmax slot is 16 w + l % 16 (its mask value rides with the stage).
    uint4 qa[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) qa[j] = ld16(q + (size_t)m * kQf + l16 * kDf + 128 * wave + 32 * j + 8 * g);
    auto issue = [&](int u, uint4 (&kr)[4][4], uint4 (&vr)[4], float& mk) {
        const int page = u / kFaChunks, s0 = (u % kFaChunks) * kFaChunk;
        const uint16_t* kp = kc + ((size_t)page * kTf + s0 + l16) * kDf + 128 * wave + 8 * g;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int j = 0; j < 4; ++j) kr[st][j] = ld16(kp + (size_t)16 * st * kDf + 32 * j);
        const uint16_t* vp = vc + ((size_t)page * kTf + s0) * kDf + b * kFaDims;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int un = t + kFaBlock * i, row = un >> 4, cu = un & 15;
            vr[i] = ld16(vp + (size_t)row * kDf + cu * 8);
        }
        mk = mask[(size_t)page * mask_page_stride + (size_t)m * kTf + s0 + 16 * wave + l16];
    };

    float m_run[4], l_run[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        m_run[r] = -INFINITY;
        l_run[r] = 0.0f;
    }
    f32x4v o[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    auto step = [&](int u, const uint4 (&kr)[4][4], const uint4 (&vr)[4], float mk, uint4 (&kn)[4][4], uint4 (&vn)[4],
                    float& mkn) {
        __syncthreads();                              // the previous chunk's LDS reads are done
        if (u + 1 < u1) issue(u + 1, kn, vn, mkn);    // the next chunk's loads go out first
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            f32x4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(qa[j]), as_bf16x8(kr[st][j]), acc, 0, 0, 0);
            // acc[r]: the wave's part of the score of head 4 (l / 16) + r at slot 16 st + l % 16
#pragma unroll
            for (int r = 0; r < 4; ++r) sp[wave][(4 * g + r) * kFaChunk + 16 * st + l16] = acc[r];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int un = t + kFaBlock * i, row = un >> 4, cu = un & 15;
            uint2* dst = reinterpret_cast<uint2*>(vs + row * kFaVStride + cu * 8);
            dst[0] = make_uint2(vr[i].x, vr[i].y);
            dst[1] = make_uint2(vr[i].z, vr[i].w);
        }
        __syncthreads();
        const bool valid = mk != 0.0f;
        float sc[4], mx[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int at = (4 * g + r) * kFaChunk + 16 * wave + l16;
            const float sv = ((sp[0][at] + sp[1][at]) + sp[2][at]) + sp[3][at];
            sc[r] = valid ? sv : -INFINITY;
            mx[r] = sc[r];
#pragma unroll
            for (int sh = 1; sh < 16; sh <<= 1) mx[r] = fmaxf(mx[r], __shfl_xor(mx[r], sh));
        }
        if (l16 == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) red_m[wave][4 * g + r] = mx[r];
        }
        __syncthreads();
        float scale[4], ls[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int h = 4 * g + r;
            const float mc = fmaxf(fmaxf(red_m[0][h], red_m[1][h]), fmaxf(red_m[2][h], red_m[3][h]));
            const float mn = fmaxf(m_run[r], mc);
            scale[r] = m_run[r] == -INFINITY ? 0.0f : __expf(m_run[r] - mn);
            m_run[r] = mn;
            const float pv = sc[r] == -INFINITY ? 0.0f : __expf(sc[r] - mn);
            const uint32_t hi = f2bf(pv);
            ps[0][h * kFaPStride + 16 * wave + l16] = (uint16_t)hi;
            ps[1][h * kFaPStride + 16 * wave + l16] = (uint16_t)f2bf(pv - bf2f(hi));
            ls[r] = pv;
#pragma unroll
            for (int sh = 1; sh < 16; sh <<= 1) ls[r] += __shfl_xor(ls[r], sh);
        }
        if (l16 == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) red_l[wave][4 * g + r] = ls[r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int h = 4 * g + r;
            l_run[r] = fmaf(l_run[r], scale[r], ((red_l[0][h] + red_l[1][h]) + red_l[2][h]) + red_l[3][h]);
#pragma unroll
            for (int dd = 0; dd < 2; ++dd) o[dd][r] *= scale[r];
        }
        // out[h][d] += sum_s p[h][s] v[s][d]: wave w takes dims 32 w .. 32 w + 31 of the block (two
        // 16-column tiles), the 64 slots as two k steps of 32. A: weights of head l % 16, slots
        // 32 kk + 8 (l / 16) .. + 7; B: V at those slots, dim l % 16 of the tile.
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const uint4 a = *reinterpret_cast<const uint4*>(ps[0] + l16 * kFaPStride + 32 * kk + 8 * g);
            const uint4 al = *reinterpret_cast<const uint4*>(ps[1] + l16 * kFaPStride + 32 * kk + 8 * g);
#pragma unroll
            for (int dd = 0; dd < 2; ++dd) {
                const int col = 32 * wave + 16 * dd + l16;
                const uint16_t* vp = vs + (32 * kk + 8 * g) * kFaVStride + col;
                uint32_t w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    w[i] = (uint32_t)vp[(2 * i) * kFaVStride] | ((uint32_t)vp[(2 * i + 1) * kFaVStride] << 16);
                const bf16x8 bv = as_bf16x8(make_uint4(w[0], w[1], w[2], w[3]));
                o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), bv, o[dd], 0, 0, 0);
                o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(al), bv, o[dd], 0, 0, 0);
            }
        }
    };
    uint4 kA[4][4], vA[4], kB[4][4], vB[4];
    float mA = 0.0f, mB = 0.0f;
    issue(u0, kA, vA, mA);
    for (int u = u0; u < u1; u += 2) {
        step(u, kA, vA, mA, kB, vB, mB);
        if (u + 1 < u1) step(u + 1, kB, vB, mB, kA, vA, mA);
    }
    float* pc = part + ((size_t)m * gridDim.x + blockIdx.x) * kFaRec;
    if (b == 0 && l16 == 0 && wave == 0) {  // every wave holds the same per-head values
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            pc[4 * g + r] = m_run[r];
            pc[kGf + 4 * g + r] = l_run[r];
        }
    }
#pragma unroll
    for (int dd = 0; dd < 2; ++dd)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            pc[2 * kGf + (4 * g + r) * kDf + b * kFaDims + 32 * wave + 16 * dd + l16] = o[dd][r];
}

// The span kernel of moa_full_attention for more than 8 pages: workgroup (x, 0, m) takes chunks
// x * cpw .. of row m over all 512 dims, so every K row and V row is read from memory once (the
// dim-split partial kernel above reads a chunk's K rows in each of its 4 dim-block workgroups).
// The chunk's V rows (64 KB) go straight to LDS (global_load_lds, no registers) in rows of 1040
// bytes; the next chunk's K rows are requested before this chunk's products, its V rows once
// they are done. Scores are split by dims as above. Record x of row m holds all 512 dims.
constexpr int kFsVRow = kDf + 8;  // LDS row of the V chunk, in elements (1040 bytes)
typedef __attribute__((address_space(3))) void fa_lds_void;
typedef __attribute__((address_space(1))) void fa_glb_void;

__global__ __launch_bounds__(kFaBlock) void fattn_span_kernel(const uint16_t* __restrict__ q,
                                                              const uint16_t* __restrict__ kc,
                                                              const uint16_t* __restrict__ vc,
                                                              const float* __restrict__ mask, int mask_page_stride,
                                                              int nchunks, int cpw, float* part) {
    __shared__ __attribute__((aligned(16))) uint16_t vsm[kFaChunk * kFsVRow];
    __shared__ __attribute__((aligned(16))) uint16_t ps[2][kGf * kFaPStride];
    __shared__ float sp[4][kGf * kFaChunk];
    __shared__ float red_m[4][kGf], red_l[4][kGf];
    const int m = blockIdx.z;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l16 = lane & 15, g = lane >> 4;
    const int u0 = blockIdx.x * cpw, u1 = min(u0 + cpw, nchunks);

    uint4 qa[4], kr[4][4];
    float mk = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) qa[j] = ld16(q + (size_t)m * kQf + l16 * kDf + 128 * wave + 32 * j + 8 * g);
    auto issue_k = [&](int u) {
        const int page = u / kFaChunks, s0 = (u % kFaChunks) * kFaChunk;
        const uint16_t* kp = kc + ((size_t)page * kTf + s0 + l16) * kDf + 128 * wave + 8 * g;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int j = 0; j < 4; ++j) kr[st][j] = ld16(kp + (size_t)16 * st * kDf + 32 * j);
        mk = mask[(size_t)page * mask_page_stride + (size_t)m * kTf + s0 + 16 * wave + l16];
    };
    auto issue_v = [&](int u) {  // wave w moves rows 16 w .. 16 w + 15, one 1 KB row per instruction
        const int page = u / kFaChunks, s0 = (u % kFaChunks) * kFaChunk;
        const uint16_t* vp = vc + ((size_t)page * kTf + s0) * kDf;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = 16 * wave + i;
            __builtin_amdgcn_global_load_lds((fa_glb_void*)(vp + (size_t)row * kDf + lane * 8),
                                             (fa_lds_void*)(vsm + row * kFsVRow), 16, 0, 0);
        }
    };
    issue_k(u0);
    issue_v(u0);

    float m_run[4], l_run[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        m_run[r] = -INFINITY;
        l_run[r] = 0.0f;
    }
    f32x4v o[8];
#pragma unroll
    for (int dd = 0; dd < 8; ++dd) o[dd] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
    for (int u = u0; u < u1; ++u) {
        __syncthreads();  // the previous chunk's score and weight reads are done
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            f32x4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(qa[j]), as_bf16x8(kr[st][j]), acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) sp[wave][(4 * g + r) * kFaChunk + 16 * st + l16] = acc[r];
        }
        const bool valid = mk != 0.0f;
        __syncthreads();
        float sc[4], mx[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int at = (4 * g + r) * kFaChunk + 16 * wave + l16;
            const float sv = ((sp[0][at] + sp[1][at]) + sp[2][at]) + sp[3][at];
            sc[r] = valid ? sv : -INFINITY;
            mx[r] = sc[r];
#pragma unroll
            for (int sh = 1; sh < 16; sh <<= 1) mx[r] = fmaxf(mx[r], __shfl_xor(mx[r], sh));
        }
        if (l16 == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) red_m[wave][4 * g + r] = mx[r];
        }
        __syncthreads();
        float scale[4], ls[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int h = 4 * g + r;
            const float mc = fmaxf(fmaxf(red_m[0][h], red_m[1][h]), fmaxf(red_m[2][h], red_m[3][h]));
            const float mn = fmaxf(m_run[r], mc);
            scale[r] = m_run[r] == -INFINITY ? 0.0f : __expf(m_run[r] - mn);
            m_run[r] = mn;
            const float pv = sc[r] == -INFINITY ? 0.0f : __expf(sc[r] - mn);
            const uint32_t hi = f2bf(pv);
            ps[0][h * kFaPStride + 16 * wave + l16] = (uint16_t)hi;
            ps[1][h * kFaPStride + 16 * wave + l16] = (uint16_t)f2bf(pv - bf2f(hi));
            ls[r] = pv;
#pragma unroll
            for (int sh = 1; sh < 16; sh <<= 1) ls[r] += __shfl_xor(ls[r], sh);
        }
        if (l16 == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) red_l[wave][4 * g + r] = ls[r];
        }
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's V rows have landed in LDS
        __syncthreads();                                     // and every other wave's
        if (u + 1 < u1) issue_k(u + 1);                      // K registers are free
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int h = 4 * g + r;
            l_run[r] = fmaf(l_run[r], scale[r], ((red_l[0][h] + red_l[1][h]) + red_l[2][h]) + red_l[3][h]);
#pragma unroll
            for (int dd = 0; dd < 8; ++dd) o[dd][r] *= scale[r];
        }
        // out[h][d] += sum_s p[h][s] v[s][d]: wave w takes dims 128 w .. 128 w + 127 (eight 16-column
        // tiles), the 64 slots as two k steps of 32.
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const uint4 a = *reinterpret_cast<const uint4*>(ps[0] + l16 * kFaPStride + 32 * kk + 8 * g);
            const uint4 al = *reinterpret_cast<const uint4*>(ps[1] + l16 * kFaPStride + 32 * kk + 8 * g);
#pragma unroll
            for (int dd = 0; dd < 8; ++dd) {
                const uint16_t* vp = vsm + (32 * kk + 8 * g) * kFsVRow + 128 * wave + 16 * dd + l16;
                uint32_t w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    w[i] = (uint32_t)vp[(2 * i) * kFsVRow] | ((uint32_t)vp[(2 * i + 1) * kFsVRow] << 16);
                const bf16x8 bv = as_bf16x8(make_uint4(w[0], w[1], w[2], w[3]));
                o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), bv, o[dd], 0, 0, 0);
                o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(al), bv, o[dd], 0, 0, 0);
            }
        }
        __syncthreads();  // the V chunk's reads are done
        if (u + 1 < u1) issue_v(u + 1);
    }
    float* pc = part + ((size_t)m * gridDim.x + blockIdx.x) * kFaRec;
    if (l16 == 0 && wave == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            pc[4 * g + r] = m_run[r];
            pc[kGf + 4 * g + r] = l_run[r];
        }
    }
#pragma unroll
    for (int dd = 0; dd < 8; ++dd)
#pragma unroll
        for (int r = 0; r < 4; ++r) pc[2 * kGf + (4 * g + r) * kDf + 128 * wave + 16 * dd + l16] = o[dd][r];
}

// Several token rows: all their heads share the one KV head, so a tile of 64 slots is read once for
// four rows (64 query rows of 512). Workgroup (x, y): rows 4 y .. 4 y + 3, tiles x * tpw .. (64
// slots; a page holds 8), an online softmax over those of its tiles in which some row has a valid
// slot; record x of each row. Eight waves, two per SIMD, on the matrix cores, transposed, so that a lane
// holds one query row's values:
//   scores^T = K Q^T (16x16x32): wave (sh, r) takes 32 of the slots and the 16 heads of row r, whose 512 dims
//     stay in registers; the slot halves exchange their maxima through LDS, sums stay apart to the end;
//   out^T += V^T P^T (32x32x16): wave w takes dims 64 w .. + 63 of all 64 query rows, over the weights of
//     both slot halves from LDS (bf16 high and low parts, as in the kernels above).
// K and V tiles go straight to LDS (16-byte chunks of a row permuted by fr_swizzle, so that neither
// the K rows' reads nor V's transposing reads meet on banks): the next tile's K beside out's
// products, this tile's V beside its scores. Bound by LDS: 450 KB of fragments a tile, 3500 cycles, beside 3100 of
// MFMAs. 200 rows over 6 pages (18 GFLOP, 34 MB of records): 48 us, and 7-10 for the merge; 4 rows over 64 pages
// (67 MB of K and V): 21-23 and 7. (Four waves of 512 registers instead kept Q and out in accumulation registers and
// copied them around the MFMAs: 60 us.)
constexpr int kFrBlock = 512;
constexpr int kFrRows = 4;                      // token rows per workgroup
constexpr int kFrQ = kFrRows * kGf;             // query rows
constexpr int kFrMaxTiles = 64;                 // tiles per workgroup
constexpr int kFrPStride = kFaChunk + 8;        // LDS row of the weights, in elements
// Weights are exp(score - reference) with a reference at most this far below the row's largest score: out
// (64 accumulators a lane) is rescaled only when the maximum has grown by more. The state is brought to
// the maximum at the end.
constexpr float kFrSlack = 8.0f;
// From these row x pages products of a call over all pages (rows of a one-page call) on this path is used, unless
// the span kernel takes all rows with one workgroup per CU. This path against the one-row kernels on every row
// (us, calls replayed as a graph): M x P = 2 x 8 14.9 / 16.3, 3 x 6 15.8 / 22.4, 4 x 4 15.8 / 17.8, 8 x 2 15.8 / 20.1,
// 16 x 1 15.7 / 25.2, 13 x 3 19.2 / 34.0, 200 x 6 50 / 1200, and host-driven 2 x 4 13.5 / 9.9. Against spans, one
// workgroup per CU: 1 x 16 15.7 / 13.4, 1 x 64 22.5 / 20.7, 2 x 9 16.5 / 13.8, 2 x 16 17.9 / 15.9, 3 x 9 19.3 / 16.3;
// more: 3 x 12 20.3 / 26.9, 2 x 24 19.0 / 28.2, 4 x 10 21.6 / 28.4, 2 x 64 25.0 / 41.0. One page: up to 16 rows one
// launch of the one-row kernel (15 us); more would be several (64 rows 22.0 / 59.2, 200 rows 27 / 191).
constexpr int kFrMinRowPages = 16;
constexpr int kFrMinPageRows = 17;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short fa_s16x4 __attribute__((ext_vector_type(4)));
typedef float fa_f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // mask rows are 4-byte aligned
typedef __attribute__((address_space(3))) fa_s16x4 fa_lds_s16x4;

// The chunk of a K or V row in which its 16-byte chunk c lies in LDS: c ^ fr_swizzle(row). Sixteen
// consecutive rows take every value, four rows differ by multiples of four chunks.
__host__ __device__ constexpr int fr_swizzle(int row) { return (row & 3) << 2 | (row >> 2 & 3); }

// LDS barrier that leaves global loads in flight (loads into LDS are waited for explicitly).
__device__ __forceinline__ void fr_barrier() {
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

__global__ __launch_bounds__(kFrBlock) __attribute__((amdgpu_waves_per_eu(2, 2))) void fattn_rows_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const float* __restrict__ mask, int mask_page_stride, int M, int ntiles, int tpw, float* part) {
    __shared__ __attribute__((aligned(1024))) uint16_t ks[kFaChunk * kDf];
    __shared__ __attribute__((aligned(1024))) uint16_t vs[kFaChunk * kDf];
    __shared__ __attribute__((aligned(16))) uint16_t ps[2][kFrQ * kFrPStride];
    __shared__ uint64_t bits[kFrRows][kFrMaxTiles];   // bit s: slot s of the tile is valid for the row
    __shared__ float red[2][kFrQ], scl[kFrQ];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, hf = lane >> 5, l16 = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.y * kFrRows;
    const int u0 = blockIdx.x * tpw, nt = min(tpw, ntiles - u0);
    const int sh = wave & 1, row = wave >> 1, qr = kGf * row + l16;  // the wave's part of the scores; the lane's query row

    // K or V tile u into LDS: wave w moves rows 8 w .. 8 w + 7 (of those, i0 .. i1 - 1), a row (1 KB) per instruction
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(kc + (size_t)u0 * kFaChunk * kDf), 0, (uint32_t)nt * kFaChunk * kDf * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(vc + (size_t)u0 * kFaChunk * kDf), 0, (uint32_t)nt * kFaChunk * kDf * 2, 0x00020000);
    auto issue = [&](__amdgpu_buffer_rsrc_t rs, uint16_t* dst, int u, int i0, int i1) {
#pragma unroll
        for (int i = i0; i < i1; ++i) {
            const int r = wave * 8 + i;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (fa_lds_void*)(dst + r * kDf), 16, (lane ^ fr_swizzle(r)) * 16,
                                                     (u * kFaChunk + r) * kDf * 2, 0, 0);
        }
    };
    issue(krs, ks, 0, 0, 8);  // most often the first tile it needs (else read again)
    // Q: lane (l16, g) holds dims 32 j + 8 g .. + 7 of its query row (a row past M repeats the last)
    uint4 qf[16];
    {
        const uint16_t* qp = q + ((size_t)min(m0 + row, M - 1) * kGf + l16) * kDf + 8 * g;
#pragma unroll
        for (int j = 0; j < 16; ++j) qf[j] = ld16(qp + 32 * j);
    }
    // valid slots: waves r and r + 4 read row m0 + r, 16 slots per lane, 16 tiles per pass
    {
        const int r = wave & 3, m = m0 + r;
        const float* mr = mask + (size_t)min(m, M - 1) * kTf + (lane & 3) * 16;
        for (int base = 16 * (wave >> 2); base < nt; base += 32) {
            const int u = base + (lane >> 2), a = u0 + min(u, nt - 1);
            const float* mp = mr + (size_t)(a / kFaChunks) * mask_page_stride + a % kFaChunks * kFaChunk;
            fa_f32x4u v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const fa_f32x4u*>(mp + 4 * i);
            uint32_t b = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) b |= v[i >> 2][i & 3] != 0.0f ? 1u << i : 0u;
            if (u < nt) reinterpret_cast<uint16_t*>(&bits[r][u])[lane & 3] = m < M ? (uint16_t)b : 0;
        }
    }
    __syncthreads();
    // the tiles some row has a valid slot in, in order
    uint64_t todo = 0;
    {
        uint64_t any = 0;
        if (lane < nt)
#pragma unroll
            for (int r = 0; r < kFrRows; ++r) any |= bits[r][lane];
        todo = __ballot(any != 0);
    }

    // LDS addresses (bytes). K chunk g of slot 32 sh + l16 (chunk 4 j + g: 64 j flips its bits, j / 4 as 256 bytes
    // each; the second 16 slots as rows). V's first read: slots 8 hf + l16 / 4 (16 kk + 4 y more: rows, and y
    // flips the swizzle's low bit, 16 bytes), dims 64 w + 16 (g % 2) + 4 (l16 % 4) (dim tile dt: 64 dt flips).
    const int krow = 32 * sh + l16, vrow = 8 * hf + (l16 >> 2);
    const int ka = krow * 1024 + (g ^ fr_swizzle(krow)) * 16;
    const int va = vrow * 1024 + ((8 * wave + 2 * (g & 1) + (l16 >> 1 & 1)) ^ fr_swizzle(vrow)) * 16 + (l16 & 1) * 8;

    f32x16 o[2][2];
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][qt][e] = 0.0f;
    // of the lane's query row: the largest score, the score that weights are relative to, and the sum of the
    // weights the lane has computed
    float m_run = -INFINITY, m_ref = -INFINITY, l_run = 0.0f;

    int u = todo ? __builtin_ctzll(todo) : 0;
    if (u || !todo) {  // not the first tile, or none: its load ends before the rows are loaded again or the wave does
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (todo) issue(krs, ks, u, 0, 8);
    }
    while (todo) {
        todo &= todo - 1;
        const int un = todo ? __builtin_ctzll(todo) : 0;
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's K rows are in LDS
        fr_barrier();                                          // and the others'; V's reads of the tile before are done
        // per 16 slots four sums of 4 MFMAs, sum c over dims 128 c .. + 127 and added up in that order, as in the
        // one-row kernels: a row's scores, and its maximum, have the same bits in every kernel (running_sum is off
        // by the rounding of the largest score, 1.5e-6 of it). Step n takes 32 dims of sum n % 4;
        // fragments four ahead of the MFMAs that use them; this tile's V beside them
        f32x4v sc[2][4];
        bf16x8 kf[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) sc[i][c] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
        auto read_k = [&](int n) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                kf[i][n & 3] = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const uint8_t*>(ks) + (ka ^ (64 * (n >> 2))) +
                                                                (n & 3) * 256 + i * 16 * 1024);
        };
#pragma unroll
        for (int n = 0; n < 4; ++n) read_k(n);
#pragma unroll
        for (int n = 0; n < 16; ++n) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                sc[i][n & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i][n & 3], as_bf16x8(qf[4 * (n & 3) + (n >> 2)]),
                                                                       sc[i][n & 3], 0, 0, 0);
            if (n < 12) read_k(n + 4);
            if (n & 1) issue(vrs, vs, u, n >> 1, (n >> 1) + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        // element (i, e): slot 32 sh + 16 i + 4 g + e
        const uint32_t vb = (uint32_t)(bits[row][u] >> (32 * sh + 4 * g));
        float x[2][4], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[i][e] = ((sc[i][0][e] + sc[i][1][e]) + sc[i][2][e]) + sc[i][3][e];
                x[i][e] = (vb >> (16 * i + e) & 1) ? x[i][e] : -INFINITY;
                mx = fmaxf(mx, x[i][e]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (g == 0) red[sh][qr] = mx;
        fr_barrier();  // maxima; K's reads are done
        m_run = fmaxf(m_run, fmaxf(red[0][qr], red[1][qr]));
        float scale = 1.0f;
        if (m_run > m_ref + kFrSlack) {
            scale = m_ref == -INFINITY ? 1.0f : __expf(m_ref - m_run);  // -inf: sum and out are still zero
            m_ref = m_run;
        }
        const float mu = m_ref == -INFINITY ? 0.0f : m_ref;
        float ls = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float p[4], lo[4];
            uint32_t hi[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                p[e] = __expf(x[i][e] - mu);
                ls += p[e];
                hi[e] = f2bf(p[e]);
                lo[e] = p[e] - bf2f(hi[e]);
            }
            const int at = qr * kFrPStride + 32 * sh + 16 * i + 4 * g;
            *reinterpret_cast<uint2*>(&ps[0][at]) = make_uint2(hi[0] | hi[1] << 16, hi[2] | hi[3] << 16);
            *reinterpret_cast<uint2*>(&ps[1][at]) = make_uint2(pk_bf16(lo[0], lo[1]), pk_bf16(lo[2], lo[3]));
        }
        l_run = fmaf(l_run, scale, ls);
        if (sh == 0 && g == 0) scl[qr] = scale;
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // V's rows are in LDS
        fr_barrier();                                          // weights and scales too
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            const float f = scl[32 * qt + l32];
            if (__any(f != 1.0f)) {
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) o[dt][qt][e] *= f;
            }
        }
        // Step n: slots 16 (n / 2) .. + 15, dim tile n % 2. V's fragments are all read first: the compiler waits for
        // every load into LDS before a transposing read, so the next tile's K goes out behind them.
        bf16x8 pb[2][2][2], vf[8];
        auto read_p = [&](bf16x8 (&d)[2][2], int kk) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int qt = 0; qt < 2; ++qt)
                    d[h][qt] = *reinterpret_cast<const bf16x8*>(&ps[h][(32 * qt + l32) * kFrPStride + 16 * kk + 8 * hf]);
        };
        auto read_v = [&](bf16x8& d, int n) {
            fa_s16x4 a[2];
#pragma unroll
            for (int y = 0; y < 2; ++y)
                a[y] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (fa_lds_s16x4*)(reinterpret_cast<uint8_t*>(vs) + (va ^ (64 * (n & 1) + 16 * y)) + ((n >> 1) * 16 + 4 * y) * 1024));
            d = __builtin_bit_cast(bf16x8, __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7));
        };
        read_p(pb[0], 0);
#pragma unroll
        for (int n = 0; n < 8; ++n) read_v(vf[n], n);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            if (todo) issue(krs, ks, un, n, n + 1);
            if (n % 2 == 0 && n < 6) read_p(pb[(n / 2 + 1) & 1], n / 2 + 1);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int qt = 0; qt < 2; ++qt)
                    o[n & 1][qt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[n], pb[n / 2 & 1][h][qt], o[n & 1][qt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        u = un;
    }
    // the sums of the lane groups and slot halves, and the factor that brings the state to the maximum
    fr_barrier();
    const float fin = m_ref == -INFINITY ? 0.0f : __expf(m_ref - m_run);
    l_run += __shfl_xor(l_run, 16);
    l_run += __shfl_xor(l_run, 32);
    if (g == 0) {
        red[sh][qr] = l_run;
        if (sh == 0) scl[qr] = fin;
    }
    fr_barrier();
    if (sh == 0 && g == 0 && m0 + row < M) {
        float* pc = part + ((size_t)(m0 + row) * gridDim.x + blockIdx.x) * kFaRec;
        pc[l16] = m_run;
        pc[kGf + l16] = (red[0][qr] + red[1][qr]) * fin;
    }
    // out through LDS (over K and V: 32 query rows of 2 KB each, 16-byte chunks permuted so that neither
    // side meets on banks), so that a wave stores whole 1 KB runs of a record
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
        uint8_t* os = reinterpret_cast<uint8_t*>(qt ? vs : ks);
        const float f = scl[32 * qt + l32];
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *reinterpret_cast<float4*>(os + l32 * 2048 + ((16 * wave + 8 * dt + 2 * a + hf) ^ (l32 & 15)) * 16) =
                    make_float4(o[dt][qt][4 * a] * f, o[dt][qt][4 * a + 1] * f, o[dt][qt][4 * a + 2] * f,
                                o[dt][qt][4 * a + 3] * f);
    }
    fr_barrier();
#pragma unroll
    for (int i = 0; i < kFrQ / 8; ++i) {
        const int r = 8 * i + wave, m = m0 + r / kGf;
        if (m >= M) continue;
        const uint8_t* os = reinterpret_cast<const uint8_t*>(r >= 32 ? vs : ks) + (r & 31) * 2048;
        float* pc = part + ((size_t)m * gridDim.x + blockIdx.x) * kFaRec + 2 * kGf + r % kGf * kDf;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            *reinterpret_cast<float4*>(pc + 4 * (64 * h + lane)) =
                *reinterpret_cast<const float4*>(os + ((64 * h + lane) ^ (r & 15)) * 16);
    }
}

// Workgroup (h, m) merges head h's nrec (at most 8) records into the row's state; thread t owns dims
// 2 t, 2 t + 1. All: nrec is 8, known to the compiler, so that every load is at a fixed offset of a scalar address.
template <bool All>
__global__ __launch_bounds__(kFaBlock) void fattn_combine_kernel(const float* __restrict__ part, float* rmax,
                                                                 float* rsum, uint16_t* out, int first, int n) {
    const int h = blockIdx.x, m = blockIdx.y, t = threadIdx.x;
    const int nrec = All ? kFaChunks : n;
    const float* pm = part + (size_t)m * nrec * kFaRec;
    float mc[kFaChunks], lc[kFaChunks];
    float2 oc[kFaChunks];
#pragma unroll
    for (int c = 0; c < kFaChunks; ++c) {
        const int at = (All ? c : min(c, nrec - 1)) * kFaRec;
        mc[c] = pm[at + h];
        if (!All && c >= nrec) mc[c] = -INFINITY;
        lc[c] = pm[at + kGf + h];
        oc[c] = *reinterpret_cast<const float2*>(pm + at + 2 * kGf + h * kDf + 2 * t);
    }
    const size_t sh = (size_t)m * kGf + h;
    uint32_t* op = reinterpret_cast<uint32_t*>(out + sh * kDf) + t;
    const float om = first ? -INFINITY : rmax[sh];
    const float os = first ? 0.0f : rsum[sh];
    const uint32_t ob = first ? 0u : *op;
    __syncthreads();  // every wave has read the old state before thread 0 replaces it

    float mp = -INFINITY;
#pragma unroll
    for (int c = 0; c < kFaChunks; ++c) mp = fmaxf(mp, mc[c]);
    const float mn = fmaxf(om, mp);
    float l = 0.0f, o0 = 0.0f, o1 = 0.0f;
    if (mn != -INFINITY) {
        const float ro = om == -INFINITY ? 0.0f : __expf(om - mn);
        l = ro * os;
        o0 = ro * bf2f(ob & 0xffffu);
        o1 = ro * bf2f(ob >> 16);
#pragma unroll
        for (int c = 0; c < kFaChunks; ++c) {
            const float f = mc[c] == -INFINITY ? 0.0f : __expf(mc[c] - mn);
            l = fmaf(f, lc[c], l);
            o0 = fmaf(f, oc[c].x, o0);
            o1 = fmaf(f, oc[c].y, o1);
        }
    }
    *op = pk_bf16(o0, o1);
    if (t == 0) {
        rmax[sh] = mn;
        rsum[sh] = l;
    }
}

// The fused pass (state from scratch): workgroup (h, db, m) merges the nrec records of row m for
// head h, dims 64 db .. 64 db + 63. Thread t takes records t / 32, t / 32 + 8, ... (up to 32) and dims
// 2 (t % 32), + 1 of the block, every load issued before any is used; the 8 record groups meet in
// LDS in a fixed order. Records of chunks with no valid slot hold max -inf and add nothing.
constexpr int kFmGroups = 8;
constexpr int kFmDims = 64;

// RPG: the most records per group (every load of them is issued, those past nrec again for the last).
template <int RPG>
__global__ __launch_bounds__(kFaBlock) void fattn_merge_kernel(const float* __restrict__ part, int nrec, float* rmax,
                                                               float* rsum, uint16_t* out) {
    __shared__ float wm[kFmGroups], wl[kFmGroups];
    __shared__ float2 wo[kFmGroups][kFmDims / 2];
    const int h = blockIdx.x, db = blockIdx.y, m = blockIdx.z;
    const int t = threadIdx.x, rg = t / (kFmDims / 2), dp = t % (kFmDims / 2);
    const float* pm = part + (size_t)m * nrec * kFaRec;
    const int d = db * kFmDims + 2 * dp;
    float mr[RPG], lr[RPG];
    float2 ov[RPG];
#pragma unroll
    for (int i = 0; i < RPG; ++i) {
        const int x = rg + kFmGroups * i;
        const float* rec = pm + (size_t)min(x, nrec - 1) * kFaRec;
        mr[i] = x < nrec ? rec[h] : -INFINITY;
        lr[i] = rec[kGf + h];
        ov[i] = *reinterpret_cast<const float2*>(rec + 2 * kGf + h * kDf + d);
    }
    float mw = -INFINITY;
#pragma unroll
    for (int i = 0; i < RPG; ++i) mw = fmaxf(mw, mr[i]);
    if (dp == 0) wm[rg] = mw;
    __syncthreads();
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < kFmGroups; ++k) mx = fmaxf(mx, wm[k]);
    float l = 0.0f, o0 = 0.0f, o1 = 0.0f;
    if (mx != -INFINITY) {
#pragma unroll
        for (int i = 0; i < RPG; ++i) {
            const float f = mr[i] == -INFINITY ? 0.0f : __expf(mr[i] - mx);
            l = fmaf(f, lr[i], l);
            o0 = fmaf(f, ov[i].x, o0);
            o1 = fmaf(f, ov[i].y, o1);
        }
    }
    if (dp == 0) wl[rg] = l;
    wo[rg][dp] = make_float2(o0, o1);
    __syncthreads();
    if (rg != 0) return;
    float s0 = 0.0f, s1 = 0.0f, sl = 0.0f;
#pragma unroll
    for (int k = 0; k < kFmGroups; ++k) {
        s0 += wo[k][dp].x;
        s1 += wo[k][dp].y;
        sl += wl[k];
    }
    const size_t sh = (size_t)m * kGf + h;
    *reinterpret_cast<uint32_t*>(out + sh * kDf + d) = pk_bf16(s0, s1);
    if (db == 0 && dp == 0) {
        rmax[sh] = mx;
        rsum[sh] = sl;
    }
}

}  // namespace

static hipError_t combine_rows(const float* part, int nrec, float* rmax, float* rsum, uint16_t* out, bool first, int mm,
                               hipStream_t s) {
    const dim3 grid(kGf, mm), block(kFaBlock);
    if (nrec == kFaChunks) hipLaunchKernelGGL(fattn_combine_kernel<true>, grid, block, 0, s, part, rmax, rsum, out, first ? 1 : 0, nrec);
    else hipLaunchKernelGGL(fattn_combine_kernel<false>, grid, block, 0, s, part, rmax, rsum, out, first ? 1 : 0, nrec);
    return hipGetLastError();
}

// Rows m0 .. m0 + mm - 1 of the merge; P pages in nrec records per row.
static hipError_t merge_rows(const float* part, int nrec, float* rmax, float* rsum, uint16_t* out, int mm, hipStream_t s) {
    const dim3 grid(kGf, kDf / kFmDims, mm), block(kFaBlock);
    if (nrec <= kFaChunks) return combine_rows(part, nrec, rmax, rsum, out, true, mm, s);  // few: a workgroup per head
    if (nrec <= 4 * kFmGroups) hipLaunchKernelGGL(fattn_merge_kernel<4>, grid, block, 0, s, part, nrec, rmax, rsum, out);
    else if (nrec <= 8 * kFmGroups) hipLaunchKernelGGL(fattn_merge_kernel<8>, grid, block, 0, s, part, nrec, rmax, rsum, out);
    else hipLaunchKernelGGL(fattn_merge_kernel<kFaMaxRecords / kFmGroups>, grid, block, 0, s, part, nrec, rmax, rsum, out);
    return hipGetLastError();
}

// The split of fattn_rows_kernel for M rows over ntiles tiles: records per row, tiles per record and rows
// per launch. About one workgroup per CU (one fits a CU), at most kFrMaxTiles tiles each, and the
// records of a launch within the scratch.
struct RowsSplit {
    int nrec, tpw, rows;
};
static RowsSplit rows_split(int M, int ntiles, int cus) {
    const int blocks = ((M < kFattnRecords ? M : kFattnRecords) + kFrRows - 1) / kFrRows;
    int n = cus / blocks;
    n = n < 1 ? 1 : (n > kFaMaxRecords ? kFaMaxRecords : n);
    if (n > ntiles) n = ntiles;
    if (n * kFrMaxTiles < ntiles) n = (ntiles + kFrMaxTiles - 1) / kFrMaxTiles;
    RowsSplit r;
    r.tpw = (ntiles + n - 1) / n;
    r.nrec = (ntiles + r.tpw - 1) / r.tpw;
    r.rows = kFattnRecords / r.nrec;  // at least kFrRows: nrec <= kFaMaxRecords
    return r;
}
static_assert(kFattnRecords >= kFrRows * kFaMaxRecords, "a launch of fattn_rows_kernel holds four rows");

hipError_t launch_full_attention(const uint16_t* q, const uint16_t* k_pages, const uint16_t* v_pages,
                                 const float* masks, int P, float* running_max, float* running_sum, uint16_t* out,
                                 int M, hipStream_t s, DevCtx* ctx) {
    const int nchunks = P * kFaChunks;
    // One row, up to kFaSplitPages pages: one chunk per dim-split workgroup (P x 32 workgroups). More:
    // spans of chunks over all dims, at most kFaMaxRecords workgroups per row.
    const bool split = P <= kFaSplitPages;
    RowsSplit r = {0, split ? 1 : (nchunks + kFaMaxRecords - 1) / kFaMaxRecords, 1};
    r.nrec = (nchunks + r.tpw - 1) / r.tpw;
    const bool many = M * P >= kFrMinRowPages && (split || M * r.nrec > ctx->cus);
    if (many) r = rows_split(M, nchunks, ctx->cus);
    else r.rows = kFattnRecords / r.nrec;
    for (int m0 = 0; m0 < M; m0 += r.rows) {
        const int mm = M - m0 < r.rows ? M - m0 : r.rows;
        const uint16_t* qm = q + (size_t)m0 * kQf;
        const float* mk = masks + (size_t)m0 * kTf;
        if (many)
            hipLaunchKernelGGL(fattn_rows_kernel, dim3(r.nrec, (mm + kFrRows - 1) / kFrRows), dim3(kFrBlock), 0, s, qm,
                               k_pages, v_pages, mk, M * kTf, mm, nchunks, r.tpw, ctx->fattn_part);
        else if (split)
            hipLaunchKernelGGL(fattn_partial_kernel, dim3(r.nrec, kFaDimBlocks, mm), dim3(kFaBlock), 0, s, qm, k_pages,
                               v_pages, mk, M * kTf, nchunks, r.tpw, ctx->fattn_part);
        else
            hipLaunchKernelGGL(fattn_span_kernel, dim3(r.nrec, 1, mm), dim3(kFaBlock), 0, s, qm, k_pages, v_pages, mk,
                               M * kTf, nchunks, r.tpw, ctx->fattn_part);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        e = merge_rows(ctx->fattn_part, r.nrec, running_max + (size_t)m0 * kGf, running_sum + (size_t)m0 * kGf,
                       out + (size_t)m0 * kQf, mm, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_full_attention_page(const uint16_t* q, const uint16_t* k_page, const uint16_t* v_page,
                                      const float* mask, float* running_max, float* running_sum, uint16_t* out,
                                      int M, bool first, hipStream_t s, DevCtx* ctx) {
    // Many rows share a pass over the page (kFaChunks tiles, at most as many records per row)
    const bool many = M >= kFrMinPageRows;
    const RowsSplit r = many ? rows_split(M, kFaChunks, ctx->cus) : RowsSplit{kFaChunks, 1, kMaxDecodeM};
    for (int m0 = 0; m0 < M; m0 += r.rows) {
        const int mm = M - m0 < r.rows ? M - m0 : r.rows;
        if (many)
            hipLaunchKernelGGL(fattn_rows_kernel, dim3(r.nrec, (mm + kFrRows - 1) / kFrRows), dim3(kFrBlock), 0, s,
                               q + (size_t)m0 * kQf, k_page, v_page, mask + (size_t)m0 * kTf, 0, mm, kFaChunks, r.tpw,
                               ctx->fattn_part);
        else
            hipLaunchKernelGGL(fattn_partial_kernel, dim3(kFaChunks, kFaDimBlocks, mm), dim3(kFaBlock), 0, s,
                               q + (size_t)m0 * kQf, k_page, v_page, mask + (size_t)m0 * kTf, 0, kFaChunks, 1,
                               ctx->fattn_part);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        e = combine_rows(ctx->fattn_part, r.nrec, running_max + (size_t)m0 * kGf, running_sum + (size_t)m0 * kGf,
                         out + (size_t)m0 * kQf, first, mm, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace moa
