// Mixture of experts, int4 weights, more routed rows per expert than one pass of the panel kernel: a tiled MFMA kernel over
// the sorted rows, gfx950 (flashnn/triton_kernels/fused_moe_a16w4.py:50-206).
//
// The M dimension is the list of sorted routed rows, padded per expert to blocks of q.block_m rows: tile row r multiplies
// activation row sorted_ids[r] / top_k with the weights, scales and zero points of the expert its block belongs to, and the
// result goes to output row sorted_ids[r], times the routing weight on request.  A tile is a part of one block or a few
// blocks of one expert (MoeTiles), so the block size that the caller sorted for decides the padding and not the speed.
// Padding rows read activation row 0 and store nothing.
//
// A workgroup walks K in slabs of 128 (one scale group): activations and packed weights are copied into LDS by direct
// 16-byte loads (two and three stages), every wave turns its weight rows into MFMA operands (values c + q, exact) and
// multiplies all its activation fragments with them; an MFMA against ones gives the row sums that remove c and the zero
// points.  Activations are the first MFMA operand, so a lane's sums are of one channel per operand and the fold of a group,
// out += s * (acc - (c + zp) * sum a) in fp32, needs one scale and one zero point per operand in registers instead of four.
// The group tables, [expert][channel][group] in memory, are transposed into LDS once per tile.
//
// What bounds it is the issue of vector instructions beside the MFMAs: a SIMD hides two of them under a 16x16x32 MFMA
// (7.7 ns against 7.4 alone), three cost 9.5 ns and four 12.8; a slab of the 128 x 256 tile has 80 MFMAs and about 310 of
// them per wave (conversion 128, fold 128).  Wave tiles of 128 x 32 with the conversion a slab ahead (2.1 per MFMA, but half as
// many MFMAs again against ones) measured the same (773 us below), one wave per SIMD with 128 x 64 was slower (1113: the
// accumulators move between the register files).  The 128 x 256 tile with group tables needs more than its 256 registers: 15 (bf16
// tables) and 29 (fp16) are spilled, to 64 and 112 bytes a lane; per-channel tables (243 registers) and the 64 x 128 tile spill none.
// 8 experts of N=28672 K=4096, groups of 128, bf16, 1024 tokens in blocks of 64: 1266 us on the panel kernel -> 775 (620
// TFLOP/s); 2048 tokens in blocks of 128 1706 (the fold on 128 x 128 tiles) -> 1415; 64 experts N=2816 K=2048, 64 rows per
// expert 922 -> 135; per-channel tables, N=4096 K=14336, 250 rows per expert in blocks of 64 1171 -> 370.
#include <cmath>
#include <type_traits>

#include "wo_common.h"

namespace fnn {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* gbl_ptr_t;

// K / 128 at most, where there are group tables: they lie in LDS whole, 33 KB for 32 groups of 256 channels beside 112 KB of
// stages, and 64 groups do not fit the 160 KB.  Longer rows (K = 4224 to 8192) stay on gemm_wo_tile_kernel and the panel kernel.
constexpr int kGroups = 32;

// One tile: rows m0 .. row_end - 1 (at most BM) of the sorted list, channels n0 .. n0 + BN - 1 of one expert.
template <int ADT, bool GROUPS, int SDT, int BM, int BN, int WGM>
__device__ __forceinline__ void moe_tile(const WoArgs& p, const MoeArgs& q, const int m0, const int n0, const int row_end,
                                         const int expert) {
    typedef MfmaT<ADT> MT;
    constexpr int WROWS = BN / 2;                    // weight rows (two channels each) per workgroup
    constexpr int WGN = 4, NWV = WGM * WGN, NT = NWV * 64;      // waves along the channels, waves, threads
    constexpr int WTM = BM / WGM, WTN = BN / WGN;    // a wave's rows and channels
    constexpr int FB = WTM / 16;                     // activation fragments per wave
    constexpr int NF = WTN / 32;                     // 16-row weight fragments per wave
    constexpr int NA = 2 * NF;                       // weight operands per k-step: even and odd channels of each fragment
    constexpr float c_off = ADT == FNN_F16 ? 1024.f + 8.f : 128.f + 8.f;
    constexpr int ASTG = BM * 256, WSTG = WROWS * 128;
    constexpr int MTAB = BN * 4 + 4;                 // one group's scales, then its zero points (and four bytes, for the banks)
    __shared__ __attribute__((aligned(1024))) char sa0[ASTG];
    __shared__ __attribute__((aligned(1024))) char sa1[ASTG];
    __shared__ __attribute__((aligned(1024))) char sw0[WSTG];
    __shared__ __attribute__((aligned(1024))) char sw1[WSTG];
    __shared__ __attribute__((aligned(1024))) char sw2[WSTG];
    __shared__ __attribute__((aligned(16))) int toks[BM];
    __shared__ __attribute__((aligned(16))) char mtab[GROUPS ? kGroups * MTAB : 16];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WGM, wn = wave / WGM;
    const int row16 = lane & 15, g = lane >> 4;
    const int KT = p.K / 128;
    const bool has_zp = p.zp != nullptr;

    int routed = 0;
    for (int r = threadIdx.x; r < BM; r += NT) {
        const int tok = m0 + r < row_end ? q.sorted_ids[m0 + r] : q.num_valid;
        toks[r] = tok < q.num_valid ? tok : -1;
        routed |= tok < q.num_valid;
    }
    // Blocks taller than the tile: a tile may hold nothing but padding (blocks of 256 with 64 rows per expert, 8 experts N=4096
    // K=14336, per-channel tables, us: 235 -> 130; the 256-row tiles of gemm_wo_tile_kernel 218)
    if (q.block_m > BM && !__syncthreads_or(routed)) return;
    if constexpr (GROUPS) {
        const uint16_t* const sc = (const uint16_t*)p.scale + (int64_t)expert * q.stride_scale_be + (int64_t)n0 * KT;
        const uint16_t* const zp = has_zp ? (const uint16_t*)p.zp + (int64_t)expert * q.stride_zp_be + (int64_t)n0 * KT : nullptr;
        // a thread moves four groups of one channel at a time (KT is even: the last ones two)
        const int quads = (KT + 3) / 4;
        for (int e = threadIdx.x; e < BN * quads; e += NT) {
            const int ch = e % BN, g0 = e / BN * 4;
            const uint16_t* const s4 = sc + (int64_t)ch * KT + g0;
            const uint16_t* const z4 = zp + (int64_t)ch * KT + g0;
            uint16_t v[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int at = min(i, KT - 1 - g0);
                v[i] = s4[at];
                v[4 + i] = has_zp ? z4[at] : (uint16_t)0;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (g0 + i < KT) {
                    *(uint16_t*)(mtab + (g0 + i) * MTAB + ch * 2) = v[i];
                    *(uint16_t*)(mtab + (g0 + i) * MTAB + BN * 2 + ch * 2) = v[4 + i];
                }
        }
    }
    __syncthreads();

    // ---- copies
    constexpr int NCA = BM / (4 * NWV), NCW = WROWS / (8 * NWV);
    uint32_t ga[NCA], gw[NCW];
    {
        const int ar0 = wave * 4 + (lane >> 4);          // (+ a multiple of 16: the same chunk order)
        const uint32_t a_chunk = (((lane & 15) ^ (ar0 & 15)) << 4);
#pragma unroll
        for (int i = 0; i < NCA; ++i) {
            const int tok = toks[ar0 + 4 * NWV * i];
            ga[i] = (uint32_t)(tok < 0 ? 0 : tok / q.top_k) * (uint32_t)(p.lda * 2) + a_chunk;
        }
#pragma unroll
        for (int i = 0; i < NCW; ++i) {
            const int r = (i * NWV + wave) * 8 + (lane >> 3);
            gw[i] = (uint32_t)r * (uint32_t)p.ldw + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
        }
    }
    const char* const w_base = (const char*)p.qw + (int64_t)(n0 / 2) * p.ldw + (int64_t)expert * q.stride_be;
    auto uniform = [](const char* ptr) {
        const uint64_t v = (uint64_t)ptr;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return (const char*)(((uint64_t)hi << 32) | lo);
    };
    auto copy_a = [&](char* stage, int j) {
        const char* src = uniform((const char*)p.act + (int64_t)min(j, KT - 1) * 256);
#pragma unroll
        for (int i = 0; i < NCA; ++i)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(src + ga[i]), (lds_ptr_t)(stage + (i * NWV + wave) * 1024), 16, 0, 0);
    };
    auto copy_w = [&](char* stage, int j) {
        const char* src = uniform(w_base + (int64_t)min(j, KT - 1) * 128);
#pragma unroll
        for (int i = 0; i < NCW; ++i)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(src + gw[i]), (lds_ptr_t)(stage + (i * NWV + wave) * 1024), 16, 0, 0);
    };
    auto wait_barrier = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070 | NCW);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    int w_rd[2], a_rd[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) w_rd[h] = (wn * (WTN / 2) + row16) * 128 + (((4 * h + g) ^ ((row16 >> 1) & 7)) << 4);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int s = 0; s < 2; ++s) a_rd[h][s] = (wm * WTM + row16) * 256 + (((8 * h + 2 * g + s) ^ row16) << 4);

    v4f outv[NA][FB];
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
        for (int a = 0; a < NA; ++a) outv[a][b] = v4f{0, 0, 0, 0};
    float czp[NA];       // per-channel tables: c + zp of the lane's channels
    if constexpr (!GROUPS) {
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const int n = n0 + wn * WTN + (a >> 1) * 32 + 2 * row16 + (a & 1);
            czp[a] = c_off + (has_zp ? load_as_f32(p.zp, (int64_t)expert * q.stride_zp_be + n, p.zp_dtype) : 0.f);
        }
    }
    const v4u ones = v4u{MT::one2, MT::one2, MT::one2, MT::one2};
    const v4f zero4 = v4f{0, 0, 0, 0};

    // One slab: all of its weights are converted first, then one activation fragment at a time is read (a fragment ahead),
    // multiplied, and its sums folded while the MFMAs of the next fragment run.  Per-channel tables: the sums go on over K
    // and the fold only takes the slab's (c + zp) * sum a off them.  Left to the end of K, the offset (1032 times the row sum in
    // fp16) makes the fp32 sums that much longer than the result: relative error beside the output's rounding, fp16,
    // K = 14336, activations of mean 0 / all positive: 1.1e-4 / 2.0e-4 with one fold at the end, 1.3e-5 / 2e-6 with one per
    // slab (panel kernel 4.5e-5 / 2.1e-5; K = 1024: 1.4e-5 / 5e-6, level with it).  It costs 4 to 6 %.
    auto slab = [&](const char* sa, const char* sw, const char* tab) {
        v4u A[4][NA];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const v4u w = *(const v4u*)(sw + w_rd[h] + f * 16 * 128);
                convert_w4_nat<ADT>(w, A[2 * h][2 * f], A[2 * h + 1][2 * f], A[2 * h][2 * f + 1], A[2 * h + 1][2 * f + 1]);
            }
        __builtin_amdgcn_sched_barrier(0);
        v4u B[2][4];
        auto read_b = [&](int b) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) B[b & 1][ks] = *(const v4u*)(sa + a_rd[ks >> 1][ks & 1] + b * 16 * 256);
        };
        read_b(0);
        float sc[NA], zc[NA];
        if constexpr (GROUPS) {
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const int ch = wn * WTN + f * 32 + 2 * row16;
                const uint32_t sv = *(const uint32_t*)(tab + ch * 2), zv = *(const uint32_t*)(tab + BN * 2 + ch * 2);
                sc[2 * f] = bits_to_f32<SDT>(sv & 0xFFFFu);
                sc[2 * f + 1] = bits_to_f32<SDT>(sv >> 16);
                zc[2 * f] = c_off + bits_to_f32<SDT>(zv & 0xFFFFu);
                zc[2 * f + 1] = c_off + bits_to_f32<SDT>(zv >> 16);
            }
        }
        v4f acc[2][NA], as[2];
#pragma unroll
        for (int b = 0; b <= FB; ++b) {
            if (b + 1 < FB) read_b(b + 1);
            if (b < FB) {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const v4u bv = B[b & 1][ks];
                    if constexpr (GROUPS) {
#pragma unroll
                        for (int a = 0; a < NA; ++a) acc[b & 1][a] = MT::mma(bv, A[ks][a], ks == 0 ? zero4 : acc[b & 1][a]);
                    } else {
#pragma unroll
                        for (int a = 0; a < NA; ++a) outv[a][b] = MT::mma(bv, A[ks][a], outv[a][b]);
                    }
                    as[b & 1] = MT::mma(bv, ones, ks == 0 ? zero4 : as[b & 1]);
                }
            }
            if (b > 0) {
#pragma unroll
                for (int a = 0; a < NA; ++a)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float sum = as[(b - 1) & 1][r];
                        if constexpr (GROUPS) outv[a][b - 1][r] += sc[a] * (acc[(b - 1) & 1][a][r] - zc[a] * sum);
                        else outv[a][b - 1][r] = __builtin_fmaf(-czp[a], sum, outv[a][b - 1][r]);
                    }
            }
            if (b < FB) {
                if (b + 1 < FB) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
                for (int i = 0; i < 4 * (NA + 1); ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, GROUPS ? 2 : 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#define FNN_ITER(CA, CW, FA, FW, J)                                       \
    do {                                                                  \
        wait_barrier();                                                   \
        copy_a(FA, (J) + 1);                                              \
        copy_w(FW, (J) + 2);                                              \
        __builtin_amdgcn_sched_barrier(0);                                \
        slab(CA, CW, mtab + (GROUPS ? (J) * MTAB : 0));                   \
        __builtin_amdgcn_sched_barrier(0);                                \
    } while (0)
    // prologue, in the order the loop issues them: slab 0 whole, then the weights of slab 1
    copy_a(sa0, 0);
    copy_w(sw0, 0);
    copy_w(sw1, 1);
    __builtin_amdgcn_sched_barrier(0);
    // the stages rotate with periods 2 and 3: six iterations per round
    int j = 0;
    for (; j + 6 <= KT; j += 6) {
        FNN_ITER(sa0, sw0, sa1, sw2, j);
        FNN_ITER(sa1, sw1, sa0, sw0, j + 1);
        FNN_ITER(sa0, sw2, sa1, sw1, j + 2);
        FNN_ITER(sa1, sw0, sa0, sw2, j + 3);
        FNN_ITER(sa0, sw1, sa1, sw0, j + 4);
        FNN_ITER(sa1, sw2, sa0, sw1, j + 5);
    }
    // the remaining slabs (KT is a multiple of 2: checked on the host)
    if (j < KT) {
        FNN_ITER(sa0, sw0, sa1, sw2, j);
        FNN_ITER(sa1, sw1, sa0, sw0, j + 1);
    }
    if (j + 2 < KT) {
        FNN_ITER(sa0, sw2, sa1, sw1, j + 2);
        FNN_ITER(sa1, sw0, sa0, sw2, j + 3);
    }
#undef FNN_ITER

    if constexpr (!GROUPS) {
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const int n = n0 + wn * WTN + (a >> 1) * 32 + 2 * row16 + (a & 1);
            const float sc = load_as_f32(p.scale, (int64_t)expert * q.stride_scale_be + n, p.scale_dtype);
#pragma unroll
            for (int b = 0; b < FB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) outv[a][b][r] *= sc;
        }
    }

    // lane (row16, g) holds, of fragment b, rows 4 g .. + 3 and of weight fragment f channels 2 row16, + 1
    const bool pairs = (p.ldc % 2) == 0 && ((uintptr_t)p.out % 4) == 0;
#pragma unroll
    for (int b = 0; b < FB; ++b) {
        const v4i tk = *(const v4i*)(toks + wm * WTM + b * 16 + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = tk[r];
            if (m < 0) continue;
            const float un = q.mul_w ? load_as_f32(q.topk_w, m, q.topk_w_dtype) : 1.f;
            uint16_t* dst = (uint16_t*)p.out + (int64_t)m * p.ldc + n0 + wn * WTN + 2 * row16;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const uint32_t b0 = f32_to_bits<ADT>(outv[2 * f][b][r] * un), b1 = f32_to_bits<ADT>(outv[2 * f + 1][b][r] * un);
                if (pairs) {
                    *(uint32_t*)(dst + f * 32) = (b0 & 0xFFFFu) | (b1 << 16);
                } else {
                    dst[f * 32] = (uint16_t)b0;
                    dst[f * 32 + 1] = (uint16_t)b1;
                }
            }
        }
    }
}

template <int ADT, bool GROUPS, int SDT, int BM, int BN, int WGM>
__global__ __launch_bounds__(WGM * 256, 2) void gemm_wo_moe_kernel(const WoArgs p, const MoeArgs q) {
    // workgroups id, id + 8, .. share an XCD and take consecutive tiles, numbered in groups of four channel tiles, the
    // channel tile fastest within a group.  The number of tiles is known on the device only: the grid is the host's estimate
    // of it, and where there are more, workgroups take a second tile.
    const int per_xcd = gridDim.x >> 3, xcd = blockIdx.x & 7;
    const MoeTiles<BM> map(q, threadIdx.x & 63);
    const int cols = p.N / BN, all = map.tiles * cols, mine = (all + 7) / 8;
    for (int slot = blockIdx.x >> 3; slot < mine; slot += per_xcd) {
        const int t = xcd * mine + slot;
        if (t >= all) return;
        constexpr int GN = 4;
        const int grp = t / (GN * map.tiles), rem = t - grp * (GN * map.tiles);
        const int gcols = min(GN, cols - grp * GN);
        int m0, rows, expert;
        map.find(rem / gcols, m0, rows, expert);
        moe_tile<ADT, GROUPS, SDT, BM, BN, WGM>(p, q, m0, (grp * GN + rem % gcols) * BN, m0 + rows, expert);
        __builtin_amdgcn_s_waitcnt(0x0070);     // copies of slabs beyond the last are still on their way into LDS
        __syncthreads();
    }
}

template <int ADT, int BM, int BN, int WGM>
static void launch_t(const WoArgs& p, const MoeArgs& q, hipStream_t st) {
    const dim3 grid((unsigned)((moe_tiles_estimate(q, BM) * (p.N / BN) + 7) / 8 * 8)), block(WGM * 256);
    note_kernel(p.group ? "gemm_wo_moe_kernel(group tables)" : "gemm_wo_moe_kernel", 4, BM, BN);
    if (p.group == 0) gemm_wo_moe_kernel<ADT, false, FNN_F16, BM, BN, WGM><<<grid, block, 0, st>>>(p, q);
    else if (p.scale_dtype == FNN_F16) gemm_wo_moe_kernel<ADT, true, FNN_F16, BM, BN, WGM><<<grid, block, 0, st>>>(p, q);
    else gemm_wo_moe_kernel<ADT, true, FNN_BF16, BM, BN, WGM><<<grid, block, 0, st>>>(p, q);
}

bool launch_wo_moe_tiled(WoArgs& p, const MoeArgs& q, int act_dtype, hipStream_t st) {
    const int64_t rows = (q.num_valid + q.top_k - 1) / q.top_k;          // activation rows
    const int G = p.group ? p.K / 128 : 0;
    // group tables: contiguous [expert][channel][group] of one 16-bit type, at most kGroups of them
    const bool tables_ok = p.group == 0 ? q.stride_scale_n == 1 && (!p.zp || (q.stride_zp_n == 1 && p.zp_dtype != FNN_I8))
                                        : p.group == 128 && G <= kGroups && is16(p.scale_dtype) && q.stride_scale_k == 1 &&
                                              q.stride_scale_n == G &&
                                              (!p.zp || (p.zp_dtype == p.scale_dtype && q.stride_zp_k == 1 && q.stride_zp_n == G));
    const bool ok = tables_ok && q.block_m >= 16 && q.EM % q.block_m == 0 && p.N % 128 == 0 && p.K % 256 == 0 && p.K >= 512 &&
                    p.lda % 8 == 0 && p.ldw % 16 == 0 && q.stride_be % 16 == 0 && ((uintptr_t)p.qw % 16) == 0 &&
                    ((uintptr_t)p.act % 16) == 0 && rows * p.lda * 2 < (1LL << 32) && (int64_t)128 * p.ldw < (1LL << 31) &&
                    moe_tiles_estimate(q, 64) * (p.N / 128) < (1LL << 31);
    if (!ok) return false;
    // The other kernels are preferred only where they take the call: what both refuse (groups of 128 in rows of K / 128 not a
    // multiple of 8, short rows, tables that are not aligned) would end on the kernel of one thread per output.
    const bool panel = wo_panel_moe_takes(p, q), others = panel || wo_tile_moe_takes(p, q);
    // Rows of an expert, and what the panel kernel makes of them: it reads the expert's weights once per 16 or 32 rows.  With
    // one such pass and matrices wide enough for its workgroups it stays ahead (same box, groups of 128, panel kernel /
    // 64-row tiles, us - 8 experts N=28672 K=4096: 4 rows per expert 109 / 203, 12 rows 112 / 205, 24 rows 178 / 210, 40 rows 297 /
    // 209; 16 experts N=12288 K=4096: 4 rows 139 / 158, 12 rows 169 / 162, 24 rows 306 / 171; 64 experts N=2816 K=2048: 3 rows 167 /
    // 90, 24 rows 346 / 96; per-channel tables, 8 experts N=4096 K=14336: 12 rows 86 / 102, 24 rows 153 / 100).
    const int64_t experts = moe_experts_estimate(q), mean = (q.num_valid + experts - 1) / experts;
    const int64_t padded = (mean + q.block_m - 1) / q.block_m * q.block_m;
    if (panel && padded <= 16 && (p.N >= 8192 || p.K >= 8192)) return false;
    if (panel && padded <= 32 && p.N >= 20480) return false;
    // Few experts reached: their tiles leave most CUs without one, and the panel kernel's workgroups own a quarter of the channels.
    // How many tiles that is depends on what else a tile costs, which is K, and on how often the panel kernel reads a block's
    // weights (once per 16 rows here).  Panel kernel / 64-row tiles, us, per-channel tables: 8 experts N=4096 K=7168, blocks of 16, 1
    // token 24.7 / 47.8, 2 tokens 25.8 / 48.6, 4 tokens 46.0 / 48.8, 32 tokens level; K=14336, blocks of 64, 1 token 75.8 / 89, 2
    // tokens 108 / 88; 60 experts N=2816 K=3584, 1 token 21.2 / 26.7, 2 tokens 32.1 / 29.0; K=2048 64 experts N=2816 1 token 26.4 /
    // 18.3, 128 experts N=1536 20.8 / 18.0.
    const double e = (double)experts, reached = e * (1.0 - pow(1.0 - 1.0 / e, (double)q.num_valid));
    const double few = p.K >= 8192 ? 260 : p.K >= 6144 ? 240 : p.K >= 3072 ? 120 : 0;
    if (panel && padded <= 64 && reached * (p.N / 128) * (padded / 16) < few) return false;
    // with fewer narrow tiles than CUs the workgroups of the other kernels are no worse off
    if (others && moe_tiles_estimate(q, 64) * (p.N / 128) < 256) return false;
    // The tile: 128 x 256 where the rows fill it, 64 x 128 (two workgroups per CU) elsewhere.
    // 128 x 256 / 64 x 128 over the three layers above with groups of 128, us: 64 rows per
    // expert 339 / 299 | 270 / 269 | 164 / 135; 100 rows 353 / 395 | 279 / 350 | 170 / 193; 160 rows 621 / 577 | 529 / 498 | 324 / 274;
    // 256 rows 775 / 853 | 690 / 714 | 396 / 395; 512 rows 1415 / 1567 | 1225 / 1326.  N=4096 K=14336, per-channel tables, fewer than
    // 512 wide tiles: 100 rows 207 / 148, 250 rows 421 / 378.
    // Blocks of 128 rows and more, which gemm_wo_tile_kernel's 128 x 128 tiles had, by rounds: the wide tiles run one to a CU in whole
    // rounds, of the narrow ones what is left over of a round runs beside the end of the one before, and a round of the first takes
    // about 1.55 times one of the second (128 x 128 / 128 x 256 / 64 x 128, per-channel tables: N=4096 K=14336, 188 rows, 1.0 rounds of wide
    // tiles 272 / 245 / 290, 512 rows, 2.2 rounds 646 / 683 / 667; 4 experts N=16384 K=5120, 128 rows, 1.4 rounds 152 / 171 / 145).
    auto fits = [&](int bm) { return q.block_m % bm == 0 || bm % q.block_m == 0; };
    bool wide = (mean > 72 && mean < 136) || mean > 208;
    if (q.block_m % 128 == 0)
        wide = moe_rounds(q, p.N, 64, 128, 512) + 0.25 > 1.55 * ceil(moe_rounds(q, p.N, 128, 256, 256) - 0.05);
    else
        wide = wide && moe_tiles_estimate(q, 128) * (p.N / 256) >= 512;
    wide = wide && fits(128) && p.N % 256 == 0;
    if (!wide && !fits(64)) return false;
    auto run = [&](auto adt) {
        constexpr int ADT = decltype(adt)::value;
        if (wide) launch_t<ADT, 128, 256, 2>(p, q, st);
        else launch_t<ADT, 64, 128, 1>(p, q, st);
    };
    if (act_dtype == FNN_F16) run(std::integral_constant<int, FNN_F16>{});
    else run(std::integral_constant<int, FNN_BF16>{});
    return true;
}

}  // namespace fnn
