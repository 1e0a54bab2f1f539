// Dense UE8M0-scale GEMM (FP8 A, FP8 or FP4 B) for few rows of A (gfx950): decode-sized
// fp8_fp4_gemm_nt calls on the scaled MFMA.
//
// At small M the call is a weight stream, N x K codes of B against M x K of A, and the
// 256 x 256 pipelined tiles give it N / 256 workgroups that each walk all of K (28
// workgroups at N = 7168: 1 to 100 x 7168 x 7168 in 70 us). Here a workgroup owns 32 CG
// columns and 32 RT rows and its eight waves split K:
//  * wave w multiplies one contiguous eighth of the K blocks (a row's FP4 bytes of two
//    blocks share a cache line, so neighbouring blocks stay in one wave) with two
//    v_mfma_scale_f32_32x32x64_f8f6f4 per block and 32 x 32 tile, the same fragments as
//    the pipelined kernel, accumulating in place;
//  * fragments and scale words come straight from global memory into registers, a
//    ring of blocks ahead: no LDS and no barrier in the K loop. A slot is multiplied
//    and refilled in place; past the wave's last block the ring holds that block again,
//    multiplied with zero fragments of A. Four slots at most: a wave has 7 blocks of
//    K = 7168, and six slots' surplus loads cost 16 x 7168 x 7168 15.0 against 11.0 us;
//  * the waves' partial sums meet in LDS and are added in wave order: deterministic, no
//    workspace. The sums are grouped differently from the single-pass kernels, so the
//    bits differ from theirs (variant 11 in the configuration's name).
// Measured (us): 1 x 7168 x 7168 8.6, 48 x 7168 x 7168 17, 100 x 2112 x 7168 16,
// 16 x 7168 x 2048 6.5; the 26 MB of FP4 weights of the first alone take 5.5 at 4.7 TB/s.
// Bound by each workgroup's re-read of its rows of A from L2: (rows x K + columns x K / 2)
// bytes per workgroup, which is why more columns per workgroup pay at more rows.
// Requirements (checked by the host): e4m3 A, packed scale words of both operands, K a
// multiple of 128, BF16 D without C, 16-byte aligned rows.
#include <hip/hip_runtime.h>

#include "dg_internal.hpp"
#include "dg_kernel_common.hpp"

namespace dgm {
namespace {

using namespace dev;

constexpr int kBK = 128;
constexpr int kNW = 8;
constexpr int kFmtE4M3 = 0, kFmtE2M1 = 4;   // MFMA operand formats (cbsz / blgp)

// One operand's fragments of a 32-row tile and K block: 16-byte chunks as the scaled
// MFMA takes them (lane half h: e4m3 chunks h, 2 + h | 4 + h, 6 + h of the 128-byte
// row for its two steps of 64, e2m1 chunks h | 2 + h of the 64-byte row).
template <int FP4>
struct Operand {
    static constexpr int kChunks = FP4 ? 2 : 4;
    static constexpr int kRow = FP4 ? 64 : 128;   // bytes of a row and K block
    i32x4 c[kChunks];
    uint32_t word;   // the row's scale word of the block

    __device__ __forceinline__ void load(const uint8_t* row, const int32_t* words, int kb, int64_t s_k, int gran_k) {
        const uint8_t* p = row + (int64_t)kb * kRow;
#pragma unroll
        for (int i = 0; i < kChunks; ++i) c[i] = *reinterpret_cast<const i32x4*>(p + i * 32);
        word = (uint32_t)words[(int64_t)(gran_k == 32 ? kb : kb >> 2) * s_k];
    }
    __device__ __forceinline__ i32x8 frag(int ks) const {
        if constexpr (FP4) return i32x8{c[ks][0], c[ks][1], c[ks][2], c[ks][3], 0, 0, 0, 0};
        else return i32x8{c[2 * ks][0], c[2 * ks][1], c[2 * ks][2], c[2 * ks][3],
                          c[2 * ks + 1][0], c[2 * ks + 1][1], c[2 * ks + 1][2], c[2 * ks + 1][3]};
    }
    // E8M0 byte of step ks: K elements [64 ks + 32 h, +32) of block kb
    __device__ __forceinline__ int scale(int ks, int h, int kb, int gran_k) const {
        const int byte = gran_k == 32 ? 2 * ks + h : kb & 3;
        return (int)((word >> (8 * byte)) & 0xFFu);
    }
};

template <int RT, int CG, int B_FP4>
__global__ void __launch_bounds__(kNW * 64, 1)
fp8_fp4_gemm_tinym_kernel(const Fp8Fp4GemmArgs p) {
    using OA = Operand<0>;
    using OB = Operand<B_FP4>;
    // K blocks in flight per wave: what fits beside the sums in a wave's 256 registers
    constexpr int kSlot = RT * (4 * OA::kChunks + 1) + CG * (4 * OB::kChunks + 1);
    constexpr int kFit = (200 - 16 * RT * CG) / kSlot;
    constexpr int kPD = kFit < 2 ? 2 : kFit > 4 ? 4 : kFit;
    __shared__ __attribute__((aligned(16))) float red[kNW][RT * CG][4][64][4];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lrow = lane & 31, h = lane >> 5;
    const int n0 = blockIdx.x * (32 * CG), m0 = blockIdx.y * (32 * RT);
    const int num_kb = p.k / kBK;
    const int kb0 = num_kb * wave / kNW;
    const int cnt = num_kb * (wave + 1) / kNW - kb0;

    // Rows past the edge read the last row; their outputs are not stored.
    const uint8_t* a_row[RT];
    const int32_t* a_words[RT];
    const uint8_t* b_row[CG];
    const int32_t* b_words[CG];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int m = min(m0 + 32 * t + lrow, p.m - 1);
        a_row[t] = p.a + (int64_t)m * p.lda + 16 * h;
        a_words[t] = static_cast<const int32_t*>(p.sfa) + (int64_t)m * p.sfa_sm;
    }
#pragma unroll
    for (int c = 0; c < CG; ++c) {
        const int n = min(n0 + 32 * c + lrow, p.n - 1);
        b_row[c] = p.b + (int64_t)n * p.ldb + 16 * h;
        b_words[c] = static_cast<const int32_t*>(p.sfb) + (int64_t)n * p.sfb_sn;
    }

    struct Slot {
        OA a[RT];
        OB b[CG];
    };
    auto load = [&](Slot& s, int i) {
        const int kb = kb0 + min(i, cnt - 1);   // past the end: the last block again
#pragma unroll
        for (int c = 0; c < CG; ++c) s.b[c].load(b_row[c], b_words[c], kb, p.sfb_sk, p.gran_k_b);
#pragma unroll
        for (int t = 0; t < RT; ++t) s.a[t].load(a_row[t], a_words[t], kb, p.sfa_sk, p.gran_k_a);
    };
    f32x16 acc[RT][CG];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < CG; ++c)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][c][e] = 0.f;

    if (cnt > 0) {
        Slot ring[kPD];
#pragma unroll
        for (int s = 0; s < kPD; ++s) {
            load(ring[s], s);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto step = [&](Slot& s, int i, bool last) {
            const int kb = kb0 + min(i, cnt - 1);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    i32x8 af = s.a[t].frag(ks);
                    if (last) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) af[e] = i < cnt ? af[e] : 0;
                    }
                    const int sa = s.a[t].scale(ks, h, kb, p.gran_k_a);
#pragma unroll
                    for (int c = 0; c < CG; ++c)
                        acc[t][c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                            s.b[c].frag(ks), af, acc[t][c], B_FP4 ? kFmtE2M1 : kFmtE4M3, kFmtE4M3, 0,
                            s.b[c].scale(ks, h, kb, p.gran_k_b), 0, sa);
                }
            if (!last) {
                // the slot's registers are read before its refill is issued into them
                __builtin_amdgcn_sched_barrier(0);
                load(s, i + kPD);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        const int rings = (cnt + kPD - 1) / kPD;
        for (int it = 0; it + 1 < rings; ++it) {
#pragma unroll
            for (int s = 0; s < kPD; ++s) step(ring[s], it * kPD + s, false);
        }
#pragma unroll
        for (int s = 0; s < kPD; ++s) step(ring[s], (rings - 1) * kPD + s, true);
    }

    // Partial sums, four columns (a quad) of a lane at a time: unit u is fragment
    // u / 4, quad u % 4, added up in wave order by wave u % kNW.
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < CG; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4*>(&red[wave][t * CG + c][q][lane][0]) =
                    f32x4{acc[t][c][4 * q], acc[t][c][4 * q + 1], acc[t][c][4 * q + 2], acc[t][c][4 * q + 3]};
    __syncthreads();
    for (int u = wave; u < RT * CG * 4; u += kNW) {
        const int f = u >> 2, q = u & 3;
        f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][f][q][lane][0]);
#pragma unroll
        for (int w = 1; w < kNW; ++w) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(&red[w][f][q][lane][0]);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] + x[e];
        }
        if (p.alpha != 1.0f) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __fmul_rn(v[e], p.alpha);
        }
        // lane: row m0 + 32 t + lrow, columns n0 + 32 c + 8 q + 4 h + (0 .. 3)
        const int row = m0 + 32 * (f / CG) + lrow, col = n0 + 32 * (f % CG) + 8 * q + 4 * h;
        if (row < p.m && col < p.n) {
            uint16_t* dp = static_cast<uint16_t*>(p.d) + (int64_t)row * p.ldd + col;
            if (col + 4 <= p.n) {
                *reinterpret_cast<uint2*>(dp) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < p.n) dp[e] = bf16_bits(v[e]);
            }
        }
    }
}

template <int RT, int CG, int B_FP4>
void launch(const Fp8Fp4GemmArgs& a, hipStream_t stream) {
    const int64_t gx = (a.n + 32 * CG - 1) / (32 * CG), gy = (a.m + 32 * RT - 1) / (32 * RT);
    DG_CHECK(gx < (int64_t)1 << 31 && gy <= 65535);
    hipLaunchKernelGGL((fp8_fp4_gemm_tinym_kernel<RT, CG, B_FP4>), dim3((unsigned)gx, (unsigned)gy), dim3(kNW * 64),
                       0, stream, a);
    DG_HIP_CHECK(hipGetLastError());
}

template <int B_FP4>
void launch_fmt(const Fp8Fp4GemmArgs& a, int rows, int cols, hipStream_t stream) {
    switch (rows * 1000 + cols) {
        case 32032: launch<1, 1, B_FP4>(a, stream); break;
        case 32064: launch<1, 2, B_FP4>(a, stream); break;
        case 64032: launch<2, 1, B_FP4>(a, stream); break;
        case 64064: launch<2, 2, B_FP4>(a, stream); break;
        default: DG_UNSUPPORTED("UE8M0 tiny-M kernel: 32 or 64 rows and columns per workgroup");
    }
}

}  // namespace

bool fp8_fp4_tinym_supported(const Fp8Fp4GemmArgs& a) {
    // (row groups on the grid's y axis)
    return fp8_fp4_pipe_supported(a) && !a.a_fp4 && a.layout == nullptr && a.num_groups == 1 && !a.out_f32 &&
           a.c == nullptr && a.m <= 65535 * 32;
}

void launch_fp8_fp4_gemm_tinym(const TileConfig& cfg, const Fp8Fp4GemmArgs& args, hipStream_t stream) {
    DG_CHECK(fp8_fp4_tinym_supported(args));
    if (args.b_fp4) launch_fmt<1>(args, cfg.block_m, cfg.block_n, stream);
    else launch_fmt<0>(args, cfg.block_m, cfg.block_n, stream);
}

}  // namespace dgm
