// moa_logits.hip -- ops::final_norm_and_logits (FO/src/ops.rs:241-298): the final RMSNorm, the
// lm_head product over 262144 bf16 vocabulary rows (2.01 GB, the largest byte mover per token), and
// Gemma's logit softcap (gemma4.py:256-261, torch bf16 semantics: one rounding per op).
//
// HBM-bound: the lm_head is streamed once per launch, past up to 32 token rows, through
// v_mfma_f32_16x16x32_bf16 (16 vocabulary rows the A operand, 16 token rows the B operand, f32
// accumulation). The twelve waves of a workgroup split k: wave w keeps its slice, k 320 w ..
// 320 w + 319, of the normalised token rows in registers (40 per 16 rows; 32 rows of all k would not
// fit LDS) and streams those 640 bytes, five whole 128-byte lines, of every vocabulary row past them.
// The partial sums of 16 VT vocabulary rows meet in LDS, where a few waves add them in slice order.
// Everything a logit goes through is the same for any number of rows, so a row has the same bits in
// every call.
#include <hip/hip_runtime.h>

#include "moa_device.h"
#include "moa_internal.h"

namespace moa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kLmSlices = 12;            // waves, and partial sums of a logit
constexpr int kLmBlock = kWave * kLmSlices;
constexpr int kLmK = kH / kLmSlices;     // k of each
constexpr int kLmPairs = kLmK / 64;      // 128-byte lines of a vocabulary row in it (two MFMA k steps each)
constexpr int kLmTileBytes = 16 * kH * (int)sizeof(uint16_t);
constexpr int kLmNt = 2;                 // cache policy of the stream: non-temporal (default: 341 against 296 us, 16 rows)
static_assert(kLmK % 64 == 0, "whole lines per slice");

// LDS barrier that leaves global loads in flight.
__device__ __forceinline__ void lm_barrier() {
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

// A load that moves whole 128-byte lines puts one row's line on 8 lanes, where the MFMA wants a row on
// 4: lane (r, g) = (lane % 16, lane / 16) holds chunk 2 g + r / 8 (16 bytes) of row r % 8 in a and of
// row 8 + r % 8 in b. One exchange between lanes r and r ^ 8 (DPP) gives every lane its own row r:
// f[0] chunk 2 g, f[1] chunk 2 g + 1. (Loads in the MFMA's layout move 64 bytes of 16 rows each, half
// a line per request: 460 us at one row against 291 so, 387 against 290 at 2, 396 against 299 at 24.)
__device__ __forceinline__ void lm_rows(const uint4& a, const uint4& b, bf16x8 (&f)[2]) {
    const uint32_t av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
    uint32_t x[4], y[4];
    constexpr int kRor8 = 0x128;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x[i] = __builtin_amdgcn_update_dpp(av[i], bv[i], kRor8, 0xf, 0xc, false);  // lanes 8..15 of a row: from b
        y[i] = __builtin_amdgcn_update_dpp(bv[i], av[i], kRor8, 0xf, 0x3, false);  // lanes 0..7: from a
    }
    f[0] = __builtin_bit_cast(bf16x8, make_uint4(x[0], x[1], x[2], x[3]));
    f[1] = __builtin_bit_cast(bf16x8, make_uint4(y[0], y[1], y[2], y[3]));
}

// Four logits of one token to LDS: the lm_head linear's output is bf16 (FO/src/ops.rs:252, cast to
// f32 at :264).
__device__ __forceinline__ void lm_put(uint16_t* o, const f32x4& a) {
    *reinterpret_cast<uint2*>(o) = make_uint2(softcap30_bf16(rbf(a[0])) | softcap30_bf16(rbf(a[1])) << 16,
                                              softcap30_bf16(rbf(a[2])) | softcap30_bf16(rbf(a[3])) << 16);
}

// bf16(x * inv * w) of 8 elements.
__device__ __forceinline__ uint4 lm_scale(const uint4& x, float inv, const float (&wv)[8]) {
    float v[8];
    bf16x8_to_f32(x, v);
    uint32_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = pk_bf16((v[2 * e] * inv) * wv[2 * e], (v[2 * e + 1] * inv) * wv[2 * e + 1]);
    return make_uint4(h[0], h[1], h[2], h[3]);
}

// MT: 16-row token tiles; VT: 16-row vocabulary tiles per meeting; DB: two meeting buffers and one
// barrier, or one and two; One: one token row, its normalised slice in LDS instead of registers, so that
// two workgroups fit a CU. Workgroup b takes vocabulary rows RW b .. RW b + RW - 1: one (One: two)
// per CU. Each wave has five pairs of loads in flight, 120 KB (240 KB) per CU. The logits wait in
// LDS and go out at the end, 2 KB per token: written 32 or 128 bytes at a time between the reads,
// 16 rows' logits (8 MB) cost 20 us.
// Measured (2.01 GB; the card's attainable read rate takes 285 us): one row 289-292 us by card (on eight lanes
// per vocabulary row and v_dot2, 16 waves per CU: 294), 2 rows 290-294, 16 rows 292-296 (1667 that way), 24 rows
// 300-311 (2640). What the rows over 16 still pay is waves waiting at the meetings: with VT = 1 one row takes
// 297 us against 289, 2 rows 313 against 294, 16 rows 318 against 296, 24 rows 321 against 310. Whole vocabulary rows per wave against token rows in LDS have no
// meetings, but a CU then reads from 256 rows at once: 326 us at one row.
template <int MT, int VT, bool DB, bool One = false>
__global__ __launch_bounds__(kLmBlock, One ? 6 : 3) void logits_kernel(const uint16_t* __restrict__ input,
                                                                       const uint16_t* __restrict__ rms_w,
                                                                       const uint16_t* __restrict__ w,
                                                                       uint16_t* __restrict__ out, int M) {
    constexpr int RW = One ? 512 : 1024, kRows = One ? 1 : 16 * MT, kUnits = MT * VT * kWave;
    static_assert(kW % RW == 0 && RW % (16 * VT) == 0 && kLmBlock % kUnits == 0, "logits tiling");
    __shared__ f32x4 part[DB ? 2 : 1][kLmSlices][MT][VT][kWave];
    __shared__ __attribute__((aligned(16))) uint16_t os[kRows][RW + 8];
    __shared__ float ssq[kLmSlices][16 * MT];
    __shared__ __attribute__((aligned(16))) uint16_t ws[kH];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int r = lane & 15, g = lane >> 4;
    // k of the lane in unit (p, y), for both operands: 64 p + 16 g + 8 y .. + 7 of the wave's slice
    const int k0 = wave * kLmK + 16 * g;
    const int row0 = blockIdx.x * RW;

    // the token rows' loads, then the stream behind them (a row past M repeats the last; not stored)
    if (t < kH / 8) *reinterpret_cast<uint4*>(ws + t * 8) = ld16(rms_w + t * 8);
    uint4 xf[MT][2 * kLmPairs];
    const uint16_t* xr[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        xr[i] = input + (size_t)min(16 * i + r, M - 1) * kH + k0;
#pragma unroll
        for (int j = 0; j < 2 * kLmPairs; ++j) xf[i][j] = ld16(xr[i] + 64 * (j / 2) + 8 * (j % 2));
    }
    __builtin_amdgcn_sched_barrier(0);
    // Buffer loads, so that one past the workgroup's last row reads nothing. Load y of a pair moves one
    // line of rows 8 y .. 8 y + 7 of the 16-row tile at vo.
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(w + (size_t)row0 * kH), 0, (uint32_t)(RW * kH * sizeof(uint16_t)), 0x00020000);
    int vo = ((r & 7) * kH + k0 + (r & 8)) * (int)sizeof(uint16_t);
    uint4 ring[kLmPairs][2];
    auto issue = [&](int p) {
#pragma unroll
        for (int y = 0; y < 2; ++y)
            ring[p][y] = __builtin_bit_cast(
                uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, vo + 128 * p, y * kLmTileBytes / 2, kLmNt));
    };
    if constexpr (!One) {
#pragma unroll
        for (int p = 0; p < kLmPairs; ++p) issue(p);
        __builtin_amdgcn_sched_barrier(0);
    }
    // RMSNorm (FO/src/device/shared/rmsnorm.rs; gemma4.py:83-89)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < 2 * kLmPairs; ++j) {
            float v[8];
            bf16x8_to_f32(xf[i][j], v);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
        }
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (g == 0) ssq[wave][16 * i + r] = ss;
        // the widened values end here: kept for the scaling below they would not fit the registers
#pragma unroll
        for (int j = 0; j < 2 * kLmPairs; ++j)
            __asm__ volatile("" : "+v"(xf[i][j].x), "+v"(xf[i][j].y), "+v"(xf[i][j].z), "+v"(xf[i][j].w));
    }
    lm_barrier();
    float inv[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        float tot = 0.0f;
#pragma unroll
        for (int k = 0; k < kLmSlices; ++k) tot += ssq[k][16 * i + r];
        inv[i] = rms_inverse(tot, kH);
    }
#pragma unroll
    for (int j = 0; j < 2 * kLmPairs; ++j) {
        const int k = k0 + 64 * (j / 2) + 8 * (j % 2);
        float wv[8];
        bf16x8_to_f32(*reinterpret_cast<const uint4*>(ws + k), wv);
#pragma unroll
        for (int i = 0; i < MT; ++i) xf[i][j] = lm_scale(xf[i][j], inv[i], wv);
        if constexpr (One) *reinterpret_cast<uint4*>(ws + k) = xf[0][j];  // over its weights (the wave's own slice)
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (One) {
#pragma unroll
        for (int p = 0; p < kLmPairs; ++p) issue(p);
        __builtin_amdgcn_sched_barrier(0);
    }

    for (int it = 0; it < RW / (16 * VT); ++it) {
        f32x4 acc[MT][VT];
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            vo += kLmTileBytes;
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i][v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int p = 0; p < kLmPairs; ++p) {
                bf16x8 f[2];
                lm_rows(ring[p][0], ring[p][1], f);
                issue(p);
#pragma unroll
                for (int y = 0; y < 2; ++y)
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        const uint4 x = One ? *reinterpret_cast<const uint4*>(ws + k0 + 64 * p + 8 * y) : xf[i][2 * p + y];
                        acc[i][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[y], __builtin_bit_cast(bf16x8, x), acc[i][v], 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);  // the refill goes out as soon as its registers are free
            }
        }
        if constexpr (!DB) lm_barrier();  // the meeting before has been read
        const int b = DB ? it & 1 : 0;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int v = 0; v < VT; ++v) part[b][wave][i][v][lane] = acc[i][v];
        lm_barrier();
        // unit (token tile, vocabulary tile, lane): four consecutive vocabulary rows of one token
        const int u = t - it % (kLmBlock / kUnits) * kUnits;
        if (u >= 0 && u < kUnits) {
            const int i = u / (VT * kWave), v = u / kWave % VT;
            f32x4 a = part[b][0][i][v][lane];
#pragma unroll 3  // all at once would take 48 registers beside the streams
            for (int k = 1; k < kLmSlices; ++k) a += part[b][k][i][v][lane];
            if (!One || r == 0) lm_put(&os[16 * i + r][(it * VT + v) * 16 + 4 * g], a);
        }
    }
    lm_barrier();
    for (int u = t; u < M * (RW / 8); u += kLmBlock) {
        const int m = u / (RW / 8), c = u % (RW / 8) * 8;
        *reinterpret_cast<uint4*>(out + (size_t)m * kW + row0 + c) = *reinterpret_cast<const uint4*>(&os[m][c]);
    }
}

}  // namespace

hipError_t launch_final_norm_and_logits(const uint16_t* input, const uint16_t* rms_w, const uint16_t* w, uint16_t* out,
                                        int M, hipStream_t s) {
    for (int m0 = 0; m0 < M; m0 += 32) {
        const int mm = M - m0 < 32 ? M - m0 : 32;
        const uint16_t* x = input + (size_t)m0 * kH;
        uint16_t* y = out + (size_t)m0 * kW;
        if (mm == 1) hipLaunchKernelGGL((logits_kernel<1, 4, false, true>), dim3(kW / 512), dim3(kLmBlock), 0, s, x, rms_w, w, y, mm);
        else if (mm <= 16) hipLaunchKernelGGL((logits_kernel<1, 4, true>), dim3(kW / 1024), dim3(kLmBlock), 0, s, x, rms_w, w, y, mm);
        else hipLaunchKernelGGL((logits_kernel<2, 2, false>), dim3(kW / 1024), dim3(kLmBlock), 0, s, x, rms_w, w, y, mm);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace moa
