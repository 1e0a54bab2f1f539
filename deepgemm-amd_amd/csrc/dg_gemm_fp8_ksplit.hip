// Dense FP32-scale FP8 GEMM for launches of at most one round of 128 x 128 tiles
// (gfx950): chunked prefill and large decode batches.
//
// Such a launch leaves one 128 x 128 tile on a CU, and the pipelined kernel runs it
// with four waves, one per SIMD: nothing on the SIMD fills the matrix core while the
// wave promotes, reads fragments or waits for a stage (0.72 us per K block at
// 517 x 4096 x 7168, the MFMAs of one take 0.24). Here eight waves share the tile: waves
// 0-3 multiply the even K blocks and waves 4-7 the odd ones, each group a 2 x 2 grid of
// 64 x 64 wave tiles, so every SIMD has two waves. A stage of the two-slot LDS ring is
// one block of either group, each loaded by the group that reads it.
//
// Per block the arithmetic is the pipelined kernel's (two v_mfma_f32_32x32x64_f8f6f4 into a
// fresh accumulator, fin = fma(sa * sb, acc, fin); reference:
// deep_gemm/include/deep_gemm/impls/sm90_fp8_gemm_1d2d.cuh:281-345); the two groups' sums
// meet in LDS and are added once, even + odd, before the rounding. They are grouped
// differently from the single-chain kernels, so the bits differ: a configuration of its
// own (variant 12).
//
// What bounds it: the chain of a pair of blocks, its one barrier and the latency of the
// loads that it waits for, with two pairs of stages in 160 KB: at 517 x 4096 x 7168 a busy
// CU's LDS reads take 29% of its cycles, its MFMAs 40% (21% and 30% with weights
// from HBM, where those loads take longer). Measured (us, the
// pipelined kernel's 128 x 128 tiles -> this): 517 x 4096 x 7168 40.5 -> 32.0,
// 300 x 2112 x 7168 40.8 -> 31.7, 700 x 4096 x 4096 25.6 -> 20.7, 400 x 4096 x 2048
// 15.3 -> 12.6, 140 x 1536 x 16384 84 -> 64; with weights from HBM 47.3 -> 46.9 (640 rows),
// 45.5 -> 42.8, 28.4 -> 27.0, 15.8 -> 14.6, 90.8 -> 88.7. Scales of four blocks per load
// where SFA is K-major and aligned: one word per row and block is a 64-line gather
// per load, 39.2 -> 34.0 at 517 x 4096 x 7168.
// Requirements (checked by the host): BF16 D without C, K a multiple of 128.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "dg_internal.hpp"
#include "dg_kernel_common.hpp"
#include "dg_epilogue.hpp"
#include "dg_lds_dma.hpp"

namespace dgm {
namespace {

using namespace dev;

constexpr int kBK = 128;
constexpr int kTile = 128;           // rows and columns of a tile
constexpr int kMaxKBlocks = 1024;
constexpr int kBlockBytes = 2 * kTile * kBK + 512;   // A rows, B columns, the rows' SFA
constexpr int kStageBytes = 2 * kBlockBytes;         // one block of either group
constexpr int kGroupBytes = kTile * 16;              // KSA: the rows' SFA of four K blocks

__device__ __forceinline__ int swz_g(int r) { return ((r >> 1) ^ ((r & 1) << 2)) & 7; }

// KSA: SFA rows are contiguous over K, 16-byte aligned, a multiple of four blocks: one
// 16-byte load per row brings the scales of two pairs.
template <int KSA>
__global__ void __launch_bounds__(512, 1)
fp8_gemm_ksplit_kernel(const Fp8GemmArgs p, const int num_m_blocks, const int num_n_blocks, const int raster_gm) {
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kStageBytes];
    __shared__ float s_sfb[kMaxKBlocks];
    __shared__ __attribute__((aligned(16))) uint8_t s_sfa[KSA ? 2 * kGroupBytes : 16];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave >> 2, w4 = wave & 3, wm = w4 >> 1, wn = w4 & 1;
    int mb, nb;
    raster_tile(xcd_remap(blockIdx.x, gridDim.x), num_m_blocks, num_n_blocks, raster_gm, mb, nb);
    const int m0 = mb * kTile, n0 = nb * kTile;
    const int a_rows = min(kTile, p.m - m0), b_rows = min(kTile, p.n - n0);
    const int num_kb = p.k / kBK;
    const uint8_t* __restrict__ a_base = p.a + (int64_t)m0 * p.lda;
    const uint8_t* __restrict__ b_base = p.b + (int64_t)n0 * p.ldb;
    const float* __restrict__ sa_base = p.sfa + (int64_t)m0 * p.sfa_sm;

    // The tile's SFB row straight into LDS, ahead of the stage loads (loads retire in
    // order, so the first stage wait covers it).
    {
        const float* row = p.sfb + (int64_t)(n0 >> 7) * p.sfb_sn;
        const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_address(reinterpret_cast<const uint8_t*>(s_sfb)));
        for (int i = wave; i < (num_kb + 63) / 64; i += 8)
            dma4_vaddr(row + (int64_t)min(i * 64 + lane, num_kb - 1) * p.sfb_sk, lds + i * 256);
    }

    // Stage loads: the group's block of pair `pr` (past the end: the last block again,
    // which is then scaled by 0) into slot pr & 1; wave w4 of the group loads 8-row
    // segments 4 i + w4 of A and B and half of the SFA rows. Rows are clamped to the
    // last valid one (one v_min against a uniform limit): their products are never stored.
    const int rs = lane >> 3, pc = lane & 7;
    const uint32_t chunk_off = (pc ^ swz_g((w4 & 1) * 8 + rs)) << 4;
    const uint32_t vlane_a = (uint32_t)rs * (uint32_t)p.lda + chunk_off;
    const uint32_t vlane_b = (uint32_t)rs * (uint32_t)p.ldb + chunk_off;
    const uint32_t voff_sa = (uint32_t)(min((w4 & 1) * 64 + lane, a_rows - 1) * p.sfa_sm) * 4u;
    const uint32_t smem_lds = __builtin_amdgcn_readfirstlane(lds_address(smem));
    auto seg_load = [&](const uint8_t* base, int seg, int rows, int64_t ld, uint32_t vlane, uint32_t lds) {
        const int rb = min(seg * 8, rows - 1);
        uint32_t lim = (uint32_t)(rows - 1 - rb) * (uint32_t)ld + (kBK - 16);
        asm volatile("" : "+s"(lim));
        dma16_saddr(base + (int64_t)rb * ld, min(vlane, lim), lds);
    };
    // KSA: the scales of blocks 4 g .. 4 g + 3 (past the end: the last four) into slot g & 1,
    // the half of the rows that this wave's parity names (the waves of a parity write the
    // same bytes).
    const uint32_t sfa_lds = __builtin_amdgcn_readfirstlane(lds_address(s_sfa));
    auto issue_sfa = [&](int g) {
        dma16_saddr(reinterpret_cast<const uint8_t*>(sa_base + min(4 * g, num_kb - 4)), voff_sa,
                    sfa_lds + (g & 1) * kGroupBytes + (w4 & 1) * 1024);
    };
    constexpr int kLoads = KSA ? 8 : 9;   // per wave and stage
    auto issue = [&](int pr) {
        if (KSA && (pr & 1) == 0) issue_sfa(pr >> 1);   // (before the stage's own: the waits below cover it)
        const int kb = min(2 * pr + kg, num_kb - 1);
        const uint32_t lds = smem_lds + (pr & 1) * kStageBytes + kg * kBlockBytes;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int seg = 4 * i + w4;
            seg_load(a_base + (int64_t)kb * kBK, seg, a_rows, p.lda, vlane_a, lds + seg * 1024);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int seg = 4 * i + w4;
            seg_load(b_base + (int64_t)kb * kBK, seg, b_rows, p.ldb, vlane_b, lds + kTile * kBK + seg * 1024);
        }
        if constexpr (!KSA)
            dma4_saddr(reinterpret_cast<const uint8_t*>(sa_base + (int64_t)kb * p.sfa_sk), voff_sa,
                       lds + 2 * kTile * kBK + (w4 & 1) * 256);
    };

    const int lrow = lane & 31, lhalf = lane >> 5;
    const int gl = swz_g(lrow);
    uint32_t frag_off[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int h = 0; h < 2; ++h) frag_off[ks][h] = lrow * 128 + (((4 * ks + 2 * lhalf + h) ^ gl) << 4);
    auto frag = [&](const uint8_t* rows, int ks) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(rows + frag_off[ks][0]);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(rows + frag_off[ks][1]);
        return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto block = [&](int pr) { return smem + (pr & 1) * kStageBytes + kg * kBlockBytes; };
    auto a_slab = [&](const uint8_t* b, int i) { return b + (wm * 64 + i * 32) * 128; };
    auto b_slab = [&](const uint8_t* b, int j) { return b + kTile * kBK + (wn * 64 + j * 32) * 128; };
    f32x16 fin[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) fin[i][j][e] = 0.f;

    const int num_pr = (num_kb + 1) / 2;
    if (kg == 0) __builtin_amdgcn_s_setprio(1);   // the groups run apart, not both on the LDS at once (1%)
    issue(0);
    issue(1);
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt_barrier<kLoads>();
    __builtin_amdgcn_sched_barrier(0);
    i32x8 op_a[2][2], op_b[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        op_a[0][ks] = frag(a_slab(block(0), 0), ks);
#pragma unroll
        for (int j = 0; j < 2; ++j) op_b[j][ks] = frag(b_slab(block(0), j), ks);
    }
    f32x16 acc[2];
    for (int pr = 0; pr < num_pr; ++pr) {
        const uint8_t* cur = block(pr);
        const uint8_t* next = block(pr + 1);
        const int kb = 2 * pr + kg;
        const float sb = kb < num_kb ? s_sfb[kb] : 0.f;
        float scale[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = wm * 64 + i * 32 + lrow;
            const float sa = KSA ? *reinterpret_cast<const float*>(s_sfa + ((pr >> 1) & 1) * kGroupBytes + row * 16 + (kb & 3) * 4)
                                 : *reinterpret_cast<const float*>(cur + 2 * kTile * kBK + row * 4);
            scale[i] = kb < num_kb ? sa * sb : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (i == 0) {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) op_a[1][ks] = frag(a_slab(cur, 1), ks);
            } else {
                // Hand-off: the next pair has landed, and every read of this one's
                // slot has returned, so the slot is refilled at once. (Past the end the
                // last blocks are loaded again into a slot that nothing uses.)
                __builtin_amdgcn_sched_barrier(0);
                wait_vmcnt_barrier<0>();
                __builtin_amdgcn_sched_barrier(0);
                issue(pr + 2);
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) op_a[0][ks] = frag(a_slab(next, 0), ks);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const f32x16 c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(op_b[j][0], op_a[i][0], f32x16{}, 0, 0, 0,
                                                                                 0, 0, 0);
                acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(op_b[j][1], op_a[i][1], c, 0, 0, 0, 0, 0, 0);
                // the previous sub-tile is promoted while this one's MFMAs run
                __builtin_amdgcn_sched_barrier(0x7F4);
                if (i > 0 || j > 0) {
                    const int pi = j > 0 ? i : i - 1, pj = 1 - j;
#pragma unroll
                    for (int e = 0; e < 16; ++e) fin[pi][pj][e] = __builtin_fmaf(scale[pi], acc[pj][e], fin[pi][pj][e]);
                }
                __builtin_amdgcn_sched_barrier(0x7F4);
                if (i == 1) {
                    __builtin_amdgcn_sched_barrier(0);   // after the MFMAs that read the old registers
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) op_b[j][ks] = frag(b_slab(next, j), ks);
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) fin[1][1][e] = __builtin_fmaf(scale[1], acc[1][e], fin[1][1][e]);
    }
    // No stage load may still be writing LDS, and every wave is done with the ring.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // Even + odd sums: each group gives one 32-row slice of its wave tile away (the
    // even group slice 1, the odd group slice 0) and finishes the other.
    float* const xch = reinterpret_cast<float*>(smem);   // [group][w4][2 sub-tiles][16][64]
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            xch[(((kg * 4 + w4) * 2 + j) * 16 + e) * 64 + lane] = kg == 0 ? fin[1][j][e] : fin[0][j][e];
    __syncthreads();
    f32x16 out[1][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float other = xch[((((kg ^ 1) * 4 + w4) * 2 + j) * 16 + e) * 64 + lane];
            out[0][j][e] = (kg == 0 ? fin[0][j][e] : fin[1][j][e]) + other;
        }
    Tile t{};
    t.m0 = m0, t.n0 = n0, t.row_end = p.m, t.active = 1;
    using Epi = RowEpilogue<kNormal, 0, 0, 1, 2>;
    static_assert(2 * kStageBytes >= 64 * 1024 + 8 * 32 * Epi::ROW_BYTES, "staging beside the exchange");
    Epi::template run<32>(out, smem + 64 * 1024 + wave * 32 * Epi::ROW_BYTES, lane, t, p.m, nullptr, m0 + wm * 64 + kg * 32,
                          n0 + wn * 64, p.n, m0, m0 + kTile, p.d, nullptr, p.ldd, 0, 0);
}

}  // namespace

bool fp8_ksplit_supported(const Fp8GemmArgs& a) {
    return a.m > 0 && a.n > 0 && a.k > 0 && a.k % kBK == 0 && a.k <= kMaxKBlocks * kBK && !a.out_f32 && a.c == nullptr && a.num_groups == 1 &&
           a.layout == nullptr && lane_offsets_fit(std::min(a.m, kTile), std::max(a.lda, a.sfa_sm * 4)) &&
           lane_offsets_fit(std::min(a.n, kTile), a.ldb);
}

void launch_fp8_gemm_ksplit(const Fp8GemmArgs& a, hipStream_t stream) {
    DG_CHECK(fp8_ksplit_supported(a));
    const int64_t nm = (a.m + kTile - 1) / kTile, nn = (a.n + kTile - 1) / kTile;
    DG_CHECK(nm * nn < (int64_t)1 << 31);
    // all m-blocks of a column on one XCD where they are few (34.0 -> 32.4 us at 517 x 4096 x 7168 against 4)
    const int raster_gm = (int)std::min<int64_t>(nm, 8);
    const dim3 grid((unsigned)(nm * nn)), bdim(512);
    const bool ksa = a.sfa_sk == 1 && a.sfa_sm % 4 == 0 && a.k % (4 * kBK) == 0 && reinterpret_cast<uintptr_t>(a.sfa) % 16 == 0;
    const auto kernel = ksa ? fp8_gemm_ksplit_kernel<1> : fp8_gemm_ksplit_kernel<0>;
    hipLaunchKernelGGL(kernel, grid, bdim, 0, stream, a, (int)nm, (int)nn, raster_gm);
    DG_HIP_CHECK(hipGetLastError());
}

}  // namespace dgm
