// moa_attention.hip -- ops::sliding_attention (FO/src/ops.rs:118-128): decode attention of token
// rows over the sliding layer's ring cache.
//
// For KV head n and its query heads g = 0, 1 (FO/src/axes.rs: Ns = 8, Gs = 2, Ds = 256, Ts = 1024):
//   s_t = q_g . k_t (scale 1.0), over the slots t whose mask value is non-zero;
//   out_g = sum_t softmax(s)_t v_t, rounded once to bf16.
// This is the CPU reference (FO/scripts/reference/gemma4.py:163-186: scaled_dot_product_attention
// with scale=1.0 over the window's positions). The runtime builds the mask rows as 1.0 for slots
// <= pos and 0.0 beyond (FO/src/host/runtime.rs:160, 409). The RNGD kernel
// (FO/src/device/sliding/attention.rs) applies the mask as min(exp, mask) after a max taken over
// every slot, and adds 1e-6 to the sum. With 0/1 masks that is the same softmax up to rounding,
// unless masked slots hold scores far above the valid ones. Here the max is taken over the valid
// slots only. A row with no valid slot returns zeros.
//
// Few rows: split over slots ("flash decoding"): workgroup (n, c, m) takes the 32 slots 32 c .. 32 c + 31
// of head n for token row m. It computes its partial (max, sum of exp, sum of exp * v) for both
// query heads and publishes it with agent-scope stores. Then it adds one to the head's ticket
// counter; the workgroup that completes the head's 32 (the counter's old value is 31 mod 32)
// combines the partials. Nothing waits on another workgroup, so residency is not required.
// The head is the grid's x index: workgroups go to the 8 XCDs round-robin by linear index, so all
// 32 of head n run on XCD n and its ticket and partials never cross XCDs (7.10 -> 6.96 us per
// call against the chunk as x index; the results do not depend on the placement). More rows:
// attn_rows_kernel below.
#include <hip/hip_runtime.h>

#include "moa_device.h"
#include "moa_internal.h"

namespace moa {
namespace {

constexpr int kAtBlock = 256;
constexpr int kAtSlots = 32;                     // slots per workgroup
constexpr int kAtChunks = kTs / kAtSlots;        // 32 workgroups per head
constexpr int kAtPartFloats = 4 + kDs;           // max, sum, 2 unused, o[256] (16-byte aligned)
static_assert(kAtChunks == 32, "ticket arithmetic assumes 32 chunks per head");

__device__ __forceinline__ float sc1_load(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void sc1_store(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// part: [M][kNs][kAtChunks][kGs][kAtPartFloats]; tickets: one counter per (row, head).
__global__ __launch_bounds__(kAtBlock) void attn_split_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
                                                              const uint16_t* __restrict__ vc, const float* __restrict__ mask,
                                                              uint16_t* __restrict__ out, float* part, uint32_t* tickets) {
    __shared__ float qs[kGs][kDs];
    __shared__ float sc[kGs][kAtSlots];       // scores, then exp weights
    __shared__ float stat[kGs][2];            // max, sum
    __shared__ float ored[8][kGs][kDs];       // per slot group partial o
    __shared__ uint32_t s_last;
    const int t = threadIdx.x;
    const int n = blockIdx.x, c = blockIdx.y, m = blockIdx.z;
    const int t0 = c * kAtSlots;
    const uint16_t* qrow = q + ((size_t)m * kNs + n) * kGs * kDs;
    // The chunk's K and V rows and its mask values are requested first (none depends on q); q
    // of both query heads (512 bf16 values, two per thread) goes to LDS meanwhile.
    const int sg = t / 32, dg = t % 32;  // PV layout: slots sg, sg + 8, ..; dims 8 dg .. 8 dg + 7
    const int s = t / 8, pt = t % 8;     // score layout: slot s, dims 32 pt .. 32 pt + 31
    const uint16_t* kr = kc + ((size_t)(t0 + s) * kNs + n) * kDs + 32 * pt;
    uint4 kq[4], vq[kAtSlots / 8];
#pragma unroll
    for (int i = 0; i < 4; ++i) kq[i] = ld16(kr + 8 * i);
#pragma unroll
    for (int i = 0; i < kAtSlots / 8; ++i) vq[i] = ld16(vc + ((size_t)(t0 + sg + 8 * i) * kNs + n) * kDs + 8 * dg);
    const bool valid = mask[(size_t)m * kTs + t0 + s] != 0.0f;
    const uint32_t q2 = reinterpret_cast<const uint32_t*>(qrow)[t];
    qs[t / 128][2 * (t % 128)] = bf2f(q2 & 0xffffu);
    qs[t / 128][2 * (t % 128) + 1] = bf2f(q2 >> 16);
    __syncthreads();

    // scores: thread (s, pt) dots 32 dims of slot t0 + s with both query heads
    {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float kv[8];
            bf16x8_to_f32(kq[i], kv);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                a0 = fmaf(qs[0][32 * pt + 8 * i + e], kv[e], a0);
                a1 = fmaf(qs[1][32 * pt + 8 * i + e], kv[e], a1);
            }
        }
#pragma unroll
        for (int o = 4; o >= 1; o >>= 1) {
            a0 += __shfl_xor(a0, o);
            a1 += __shfl_xor(a1, o);
        }
        if (pt == 0) {
            sc[0][s] = valid ? a0 : -INFINITY;
            sc[1][s] = valid ? a1 : -INFINITY;
        }
    }
    __syncthreads();
    // softmax statistics of the chunk: wave 0 (lanes 0-31: head 0, 32-63: head 1)
    if (t < 64) {
        const int g = t / 32, s = t % 32;
        const float v = sc[g][s];
        float mx = v;
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        const float e = v == -INFINITY ? 0.0f : __expf(v - mx);
        float sum = e;
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) sum += __shfl_xor(sum, o);
        sc[g][s] = e;
        if (s == 0) {
            stat[g][0] = mx;
            stat[g][1] = sum;
        }
    }
    __syncthreads();
    // o = sum_s e_s v_s: thread (sg, dg) takes 8 dims of slots sg, sg + 8, ...
    {
        float o0[8], o1[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o0[e] = o1[e] = 0.0f;
#pragma unroll
        for (int i = 0; i < kAtSlots / 8; ++i) {
            const int s = sg + 8 * i;
            float vv[8];
            bf16x8_to_f32(vq[i], vv);
            const float w0 = sc[0][s], w1 = sc[1][s];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                o0[e] = fmaf(w0, vv[e], o0[e]);
                o1[e] = fmaf(w1, vv[e], o1[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            ored[sg][0][8 * dg + e] = o0[e];
            ored[sg][1][8 * dg + e] = o1[e];
        }
    }
    __syncthreads();
    float* mypart = part + (((size_t)m * kNs + n) * kAtChunks + c) * kGs * kAtPartFloats;
#pragma unroll
    for (int g = 0; g < kGs; ++g) {
        float o = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) o += ored[k][g][t];
        sc1_store(mypart + g * kAtPartFloats + 4 + t, o);
        if (t < 2) sc1_store(mypart + g * kAtPartFloats + t, stat[g][t]);
    }
    // publish, then count the head's chunks; the workgroup completing the 32 combines them
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t == 0) {
        const uint32_t old = __hip_atomic_fetch_add(tickets + ((size_t)m * kNs + n) * kTicketStride, 1u,
                                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (old % kAtChunks) == kAtChunks - 1;
    }
    __syncthreads();
    if (!s_last) return;

    // combine. Threads 0-63 read the 32 chunks' max and sum of both heads and turn them into the
    // factors exp(max_c - max) and the head's sum. Every thread reads dims 4 q .. 4 q + 3
    // (q = t % 64) of chunks 8 (t / 64) .. + 7 for both heads as 16-byte loads, all issued before
    // any is used; the four chunk groups then meet in LDS in a fixed order. Partials are read
    // coherently (agent scope: 16-byte buffer loads with sc1, and per-thread one-float atomic loads).
    __shared__ float sf[kGs][kAtChunks], sl[kGs];
    __shared__ float4 so[4][kGs][kDs / 4];
    const float* hp = part + ((size_t)m * kNs + n) * kAtChunks * kGs * kAtPartFloats;
    const int q4 = t & 63, cg = t >> 6;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(hp), 0, (uint32_t)(kAtChunks * kGs * kAtPartFloats * sizeof(float)), 0x00020000);
    float mcv = 0.0f, lcv = 0.0f;
    if (t < 64) {  // first: the factors are computed while the outputs' loads are in flight
        mcv = sc1_load(hp + ((t & 31) * kGs + (t >> 5)) * kAtPartFloats);
        lcv = sc1_load(hp + ((t & 31) * kGs + (t >> 5)) * kAtPartFloats + 1);
    }
    float4 oc[kGs][8];
#pragma unroll
    for (int g = 0; g < kGs; ++g)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            oc[g][i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                      rs, (((cg * 8 + i) * kGs + g) * kAtPartFloats + 4 + 4 * q4) * 4,
                                                      0, 16 /* sc1 */));
    if (t < 64) {
        const int g = t >> 5, cc = t & 31;
        float mx = mcv;
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        const float f = mcv == -INFINITY ? 0.0f : __expf(mcv - mx);
        float l = f * lcv;
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) l += __shfl_xor(l, o);
        sf[g][cc] = f;
        if (cc == 0) sl[g] = l;
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < kGs; ++g) {
        float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float f = sf[g][cg * 8 + i];
            a.x = fmaf(f, oc[g][i].x, a.x);
            a.y = fmaf(f, oc[g][i].y, a.y);
            a.z = fmaf(f, oc[g][i].z, a.z);
            a.w = fmaf(f, oc[g][i].w, a.w);
        }
        so[cg][g][q4] = a;
    }
    __syncthreads();
    if (t < kGs * 64) {
        const int g = t >> 6, q = t & 63;
        const float l = sl[g];
        const float4 a = so[0][g][q], b = so[1][g][q], c2 = so[2][g][q], d = so[3][g][q];
        float v[4] = {((a.x + b.x) + c2.x) + d.x, ((a.y + b.y) + c2.y) + d.y, ((a.z + b.z) + c2.z) + d.z,
                      ((a.w + b.w) + c2.w) + d.w};
        uint32_t h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = f2bf(l > 0.0f ? v[e] / l : 0.0f);
        *reinterpret_cast<uint2*>(out + (((size_t)m * kNs + n) * kGs + g) * kDs + 4 * q) =
            make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    }
}

// ---------------------------------------------------------------- many token rows
// Workgroup (n, y, z): head n, token rows 16 y .. + 15 with both query heads (32 query rows), part z of
// the slots. The four waves take the 32-slot tiles in which some row has a valid slot, dealt by the tile's number,
// so that a row's sums run in one order whichever rows stand beside it: wave w one tile of every four, turned by one
// from four to four, so that masks with a period of 2 or 4 tiles keep all waves busy (tiles w, w + 4, ..: 31.1 us for
// 20.2 with every other tile valid, 512 rows). Each has an online softmax of its own, on
// v_mfma_f32_32x32x16_bf16, transposed: scores^T = K Q^T and out^T += V^T P^T, so that a lane holds one query
// row's values. The weights stay in the registers they are computed in -- step kk of the second product takes slots
// 16 kk + 4 h + {0..3, 8..11} from lane half h, for V (transposing LDS reads) alike -- and enter as three bf16 parts,
// which hold the 24 bits of the f32 weight that attn_split_kernel multiplies by (two parts: 16-17 bits, 1-2 us less at
// 512 rows). K and V tiles are loaded a tile ahead into registers, in whole rows, and pass through the wave's own LDS:
// no barrier in the loop.
// The waves' states meet in LDS at the end; with several parts (few rows: the slots are spread over
// up to 8 workgroups), the parts' in attn_merge_kernel.
// Bound: a workgroup reads every valid slot's K and V of its head once (1 MB of 1024 slots) through the
// CU's L1, as long as the 64 MFMAs per tile and wave take. 512 rows
// (causal, from position 300) 29 us, over all slots 33; 1000 rows 56; 16 rows 12 (a workgroup set per row,
// as above: 693, 694, 1357, 22).
constexpr int kArRows = 16;                     // token rows per workgroup
constexpr int kArQ = kArRows * kGs;             // query rows
constexpr int kArTile = 32;                     // slots per tile
constexpr int kArTiles = kTs / kArTile;
constexpr int kArOStride = kDs + 4;             // LDS row of a wave's state, in floats
constexpr int kArRec = 4 + kDs;                 // record of a query row: reference, sum, 2 unused, out[256]
constexpr int kArMaxBlocks = 32;                // row blocks x slot parts of a launch with several parts
// Weights are exp(score - reference) with a reference at most this far below the row's largest score: out
// (128 accumulators a lane) is rescaled only when the maximum has grown by more.
constexpr float kArSlack = 8.0f;
constexpr int kArMinRows = 6;                   // rows of a call from which this path is used. 6 rows 11.3 us (window just begun) to
                                                // 12.1 (full), 7 rows 11.8-12.4; a workgroup set per row 11.8, 12.7
static_assert((size_t)kNs * kArMaxBlocks * kArQ * kArRec <= kAttnPartFloats, "records fit the scratch");

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short at_s16x4 __attribute__((ext_vector_type(4)));
typedef float at_f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // mask rows are 4-byte aligned
typedef __attribute__((address_space(3))) at_s16x4 at_lds_s16x4;

// A K or V row's 16-byte chunk c lies at c ^ ar_swizzle(row) of its LDS row: sixteen consecutive rows
// take every value, four rows differ by multiples of four chunks.
__device__ __forceinline__ int ar_swizzle(int row) { return (row & 3) << 2 | (row >> 2 & 3); }

__global__ __launch_bounds__(kAtBlock) __attribute__((amdgpu_waves_per_eu(1, 1))) void attn_rows_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const float* __restrict__ mask, uint16_t* __restrict__ out, int M, float* __restrict__ part) {
    __shared__ __attribute__((aligned(1024))) uint8_t smem[4 * kArQ * kArOStride * 4];  // K, V tiles (32 KB a wave); then states
    __shared__ __attribute__((aligned(1024))) uint8_t ql[kArQ * kDs * 2];
    __shared__ uint64_t bits[kArRows][kTs / 64];
    __shared__ float st_m[4][kArQ], st_l[4][kArQ];
    static_assert(sizeof(smem) >= 4 * 2 * kArTile * kDs * 2, "tiles fit");
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l32 = lane & 31, hf = lane >> 5;
    const int n = blockIdx.x, m0 = blockIdx.y * kArRows;
    const int nt = kArTiles / gridDim.z, u0 = blockIdx.z * nt;  // tiles of this part

    // Tile loads: instruction i moves rows 2 i, 2 i + 1 (512 bytes each). Buffer loads at a tile's offset vo; past
    // the last tile they read nothing. They are spread over other work: issued together, a tile's 32 hold
    // the wave for two thousand cycles.
    uint8_t* kl = smem + wave * (2 * kArTile * kDs * 2);
    uint8_t* vl = kl + kArTile * kDs * 2;
    constexpr int kRow = kNs * kDs * 2, kCache = kTs * kRow, kNone = 0x40000000;
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kc), 0, kCache, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vc), 0, kCache, 0x00020000);
    const int vo0 = hf * kRow + n * kDs * 2 + 16 * l32;
    uint4 kr[16], vr[16];
    auto load_k = [&](int vo, int i) { kr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(krs, vo, 2 * i * kRow, 0)); };
    auto load_v = [&](int vo, int i) { vr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(vrs, vo, 2 * i * kRow, 0)); };
    auto load_tile = [&](int u) {
        const int vo = vo0 + (u0 + u) * kArTile * kRow;
#pragma unroll
        for (int i = 0; i < 16; ++i) load_k(vo, i);
#pragma unroll
        for (int i = 0; i < 16; ++i) load_v(vo, i);
    };
    const int guess = min(wave, nt - 1);  // the wave's first tile when all are wanted
    {
        // valid slots of rows 4 w .. 4 w + 3 (16 per lane), Q (query row l32: token row l32 / 2, head l32 % 2; wave w
        // brings rows 8 w .. + 7), then the guessed tile
        at_f32x4u v[4][4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[r][i] = *reinterpret_cast<const at_f32x4u*>(mask + (size_t)min(m0 + 4 * wave + r, M - 1) * kTs + 16 * lane + 4 * i);
        uint4 qv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int qr = 8 * wave + 2 * i + hf;
            qv[i] = ld16(q + (((size_t)min(m0 + qr / kGs, M - 1) * kNs + n) * kGs + qr % kGs) * kDs + 8 * l32);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_tile(guess);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            uint32_t b = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) b |= v[r][i >> 2][i & 3] != 0.0f ? 1u << i : 0u;
            reinterpret_cast<uint16_t*>(bits[4 * wave + r])[lane] = m0 + 4 * wave + r < M ? (uint16_t)b : 0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int qr = 8 * wave + 2 * i + hf;
            *reinterpret_cast<uint4*>(ql + qr * 512 + (l32 ^ ar_swizzle(qr)) * 16) = qv[i];
        }
    }
    __syncthreads();
    uint32_t mine = 0;  // this wave's tiles
    {
        uint32_t any = 0;
        if (lane < nt && ((lane + (lane >> 2)) & 3) == wave)
#pragma unroll
            for (int r = 0; r < kArRows; ++r) any |= (uint32_t)(bits[r][(u0 + lane) / 2] >> (32 * ((u0 + lane) & 1)));
        mine = (uint32_t)__ballot(any != 0);
    }

    // LDS addresses: writes (row 2 i + hf: i % 8 here, i / 8 as 16 rows), K reads (chunk 2 j + hf of row l32:
    // j % 8 here, j / 8 as 256 bytes), V reads (dim tile dt, slots 8 y + 4 hf + (lane % 16) / 4 of step kk)
    int wa[8], ka[8], va[4];
#pragma unroll
    for (int i = 0; i < 8; ++i) wa[i] = (2 * i + hf) * 512 + (l32 ^ ar_swizzle(2 * i + hf)) * 16;
#pragma unroll
    for (int j = 0; j < 8; ++j) ka[j] = l32 * 512 + ((2 * j + hf) ^ ar_swizzle(l32)) * 16;
    const int i16 = lane & 15, vrow = 4 * hf + (i16 >> 2), vch = 2 * (lane >> 4 & 1) + (i16 >> 1 & 1);
    // rows 16 kk + 8 y + vrow: row & 3 = i16 / 4, row >> 2 & 3 = 2 y + hf
#pragma unroll
    for (int d = 0; d < 4; ++d) va[d] = vrow * 512 + ((4 * d + vch) ^ ((i16 >> 2) << 2 | hf)) * 16 + (i16 & 1) * 8;

    f32x16 o[8];
#pragma unroll
    for (int d = 0; d < 8; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[d][e] = 0.0f;
    float m_ref = -INFINITY, l_run = 0.0f;  // the score that the row's weights are relative to, their sum
    int u = mine ? __builtin_ctz(mine) : 0;
    if (mine && u != guess) load_tile(u);
    while (mine) {
        mine &= mine - 1;
        const int un = mine ? __builtin_ctz(mine) : 0;
        const int vo = mine ? vo0 + (u0 + un) * kArTile * kRow : kNone;
#pragma unroll
        for (int i = 0; i < 16; ++i) *reinterpret_cast<uint4*>(kl + wa[i & 7] + (i >> 3) * 16 * 512) = kr[i];
#pragma unroll
        for (int i = 0; i < 16; ++i) *reinterpret_cast<uint4*>(vl + wa[i & 7] + (i >> 3) * 16 * 512) = vr[i];
        f32x16 sc[2];
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[0][e] = sc[1][e] = 0.0f;
        // four K and Q fragments (both of row l32, same chunk) ahead of the MFMAs, the next tile's K beside them
        bf16x8 kf[4], qf[4];
        auto read_k = [&](int j) {
            kf[j & 3] = *reinterpret_cast<const bf16x8*>(kl + ka[j & 7] + (j >> 3) * 256);
            qf[j & 3] = *reinterpret_cast<const bf16x8*>(ql + ka[j & 7] + (j >> 3) * 256);
        };
#pragma unroll
        for (int j = 0; j < 4; ++j) read_k(j);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            sc[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[j & 3], qf[j & 3], sc[j & 1], 0, 0, 0);
            if (j < 12) read_k(j + 4);
            load_k(vo, j);
            __builtin_amdgcn_sched_barrier(0);
        }
        // element e: slot 8 (e / 4) + 4 hf + e % 4 of the tile
        const uint32_t vb = (uint32_t)(bits[l32 >> 1][(u0 + u) / 2] >> (32 * ((u0 + u) & 1) + 4 * hf));
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[0][e] += sc[1][e];
        if (!__all((vb & 0x0f0f0f0fu) == 0x0f0f0f0fu)) {
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[0][e] = (vb >> (8 * (e >> 2) + (e & 3)) & 1) ? sc[0][e] : -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[0][e]);
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        float scale = 1.0f;
        if (mx > m_ref + kArSlack) {
            scale = m_ref == -INFINITY ? 1.0f : __expf(m_ref - mx);  // -inf: sum and out are still zero
            m_ref = mx;
        }
        const float mu = m_ref == -INFINITY ? 0.0f : m_ref;
        float ls = 0.0f;
        uint32_t ph[8], pm[8], pl[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float p0 = __expf(sc[0][2 * i] - mu), p1 = __expf(sc[0][2 * i + 1] - mu);
            ls += p0;
            ls += p1;
            ph[i] = pk_bf16(p0, p1);
            const float r0 = p0 - __uint_as_float(ph[i] << 16), r1 = p1 - __uint_as_float(ph[i] & 0xffff0000u);
            pm[i] = pk_bf16(r0, r1);
            pl[i] = pk_bf16(r0 - __uint_as_float(pm[i] << 16), r1 - __uint_as_float(pm[i] & 0xffff0000u));
        }
        l_run = fmaf(l_run, scale, ls + __shfl_xor(ls, 32));
        if (__any(scale != 1.0f)) {
#pragma unroll
            for (int d = 0; d < 8; ++d)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[d][e] *= scale;
        }
        // step x: slots 16 (x / 8) .. + 15, dim tile x % 8; V two steps ahead, the next tile's V beside them
        bf16x8 vf[3];
        auto read_v = [&](bf16x8& f, int x) {
            at_s16x4 a[2];
#pragma unroll
            for (int y = 0; y < 2; ++y)  // y flips bit 1 of the swizzle: 32 bytes
                a[y] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (at_lds_s16x4*)(vl + (va[x & 3] ^ (32 * y)) + (16 * (x >> 3) + 8 * y) * 512 + (x >> 2 & 1) * 256));
            f = __builtin_bit_cast(bf16x8, __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7));
        };
        read_v(vf[0], 0);
        read_v(vf[1], 1);
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            if (x < 14) read_v(vf[(x + 2) % 3], x + 2);
            load_v(vo, x);
            const int k = 4 * (x >> 3);
            auto add = [&](const uint32_t (&w)[8]) {
                o[x & 7] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    vf[x % 3], __builtin_bit_cast(bf16x8, make_uint4(w[k], w[k + 1], w[k + 2], w[k + 3])), o[x & 7], 0, 0, 0);
            };
            add(ph);
            add(pm);
            add(pl);
            __builtin_amdgcn_sched_barrier(0);
        }
        u = un;
    }
    // the waves' states, brought to the largest reference
    if (hf == 0) {
        st_m[wave][l32] = m_ref;
        st_l[wave][l32] = l_run;
    }
    __syncthreads();
    const float mt = fmaxf(fmaxf(st_m[0][l32], st_m[1][l32]), fmaxf(st_m[2][l32], st_m[3][l32]));
    const float f = m_ref == -INFINITY ? 0.0f : __expf(m_ref - mt);
    float* os = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int d = 0; d < 8; ++d)
#pragma unroll
        for (int a = 0; a < 4; ++a)
            *reinterpret_cast<float4*>(os + (wave * kArQ + l32) * kArOStride + 32 * d + 8 * a + 4 * hf) =
                make_float4(o[d][4 * a] * f, o[d][4 * a + 1] * f, o[d][4 * a + 2] * f, o[d][4 * a + 3] * f);
    __syncthreads();
    // thread t: query row t / 8, dims 8 (t % 8) + 64 i
    const int qr = t >> 3, m = m0 + qr / kGs;
    float mq = -INFINITY, lq = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) mq = fmaxf(mq, st_m[w][qr]);
#pragma unroll
    for (int w = 0; w < 4; ++w) lq += st_m[w][qr] == -INFINITY ? 0.0f : st_l[w][qr] * __expf(st_m[w][qr] - mq);
    if (m >= M) return;
    float* rec = part + ((((size_t)blockIdx.y * kNs + n) * gridDim.z + blockIdx.z) * kArQ + qr) * kArRec;
    if (gridDim.z > 1 && (t & 7) == 0) {
        rec[0] = mq;
        rec[1] = lq;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int d = 8 * (t & 7) + 64 * i;
        float v[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float4 a = *reinterpret_cast<const float4*>(os + qr * kArOStride + d + 4 * h);
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                const float4 b = *reinterpret_cast<const float4*>(os + (w * kArQ + qr) * kArOStride + d + 4 * h);
                a.x += b.x;
                a.y += b.y;
                a.z += b.z;
                a.w += b.w;
            }
            v[4 * h] = a.x;
            v[4 * h + 1] = a.y;
            v[4 * h + 2] = a.z;
            v[4 * h + 3] = a.w;
            if (gridDim.z > 1) *reinterpret_cast<float4*>(rec + 4 + d + 4 * h) = a;
        }
        if (gridDim.z == 1) {
            uint32_t h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = pk_bf16(lq > 0.0f ? v[2 * e] / lq : 0.0f, lq > 0.0f ? v[2 * e + 1] / lq : 0.0f);
            *reinterpret_cast<uint4*>(out + (((size_t)m * kNs + n) * kGs + qr % kGs) * kDs + d) =
                make_uint4(h[0], h[1], h[2], h[3]);
        }
    }
}

// Workgroup (n, m): the nz (at most 8) slot parts of token row m, head n; thread t: query head t / 128,
// dims 2 (t % 128), + 1.
__global__ __launch_bounds__(kAtBlock) void attn_merge_kernel(const float* __restrict__ part, int nz, uint16_t* __restrict__ out) {
    const int n = blockIdx.x, m = blockIdx.y, t = threadIdx.x, g = t >> 7, d = 2 * (t & 127);
    const float* rec = part + ((((size_t)(m / kArRows) * kNs + n) * nz) * kArQ + (m % kArRows) * kGs + g) * kArRec;
    float mz[8], lz[8], mt = -INFINITY;
    float2 oz[8];
#pragma unroll
    for (int z = 0; z < 8; ++z) {
        const float* r = rec + (size_t)min(z, nz - 1) * kArQ * kArRec;
        mz[z] = z < nz ? r[0] : -INFINITY;
        lz[z] = r[1];
        oz[z] = *reinterpret_cast<const float2*>(r + 4 + d);
    }
#pragma unroll
    for (int z = 0; z < 8; ++z) mt = fmaxf(mt, mz[z]);
    float l = 0.0f, a = 0.0f, b = 0.0f;
#pragma unroll
    for (int z = 0; z < 8; ++z) {
        const float f = mz[z] == -INFINITY ? 0.0f : __expf(mz[z] - mt);
        l = fmaf(f, lz[z], l);
        a = fmaf(f, oz[z].x, a);
        b = fmaf(f, oz[z].y, b);
    }
    *reinterpret_cast<uint32_t*>(out + (((size_t)m * kNs + n) * kGs + g) * kDs + d) =
        pk_bf16(l > 0.0f ? a / l : 0.0f, l > 0.0f ? b / l : 0.0f);
}

}  // namespace

hipError_t launch_sliding_attention(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const float* mask,
                                    uint16_t* out, int M, hipStream_t s, DevCtx* ctx) {
    if (M >= kArMinRows) {
        // slot parts: as many (1, 2, 4 or 8; a wave needs a tile) as keep the grid within one workgroup per CU
        const int blocks = (M + kArRows - 1) / kArRows;
        int nz = 1;
        while (nz < 8 && blocks * nz * 2 <= kArMaxBlocks) nz *= 2;
        hipLaunchKernelGGL(attn_rows_kernel, dim3(kNs, blocks, nz), dim3(kAtBlock), 0, s, q, k_cache, v_cache, mask, out, M,
                           ctx->attn_part);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess || nz == 1) return e;
        hipLaunchKernelGGL(attn_merge_kernel, dim3(kNs, M), dim3(kAtBlock), 0, s, (const float*)ctx->attn_part, nz, out);
        return hipGetLastError();
    }
    static_assert(kArMinRows <= kMaxDecodeM + 1, "one launch's partials and tickets");
    hipLaunchKernelGGL(attn_split_kernel, dim3(kNs, kAtChunks, M), dim3(kAtBlock), 0, s, q, k_cache, v_cache, mask, out,
                       ctx->attn_part, ctx->tickets + kTicketAttn * kTicketStride);
    return hipGetLastError();
}

}  // namespace moa
