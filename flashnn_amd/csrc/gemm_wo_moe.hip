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
// 16-byte loads (two and three stages).  Every wave owns 32 channels and all rows: it turns its weights into MFMA operands (whole
// numbers u = q + 8, exact) and multiplies all activation fragments with them.  The activations are the first MFMA operand, so a
// lane's sums are of one channel per operand and the fold of a group, out += s * sum a u - s * (8 + zp) * sum a in fp32, takes one
// scale and one zero point per operand.  The sums of the activations come from MFMAs against ones, which the waves share: each sums
// up one fragment and hands the sums on through LDS; they are used a slab later, so that no barrier is added.  Tables are copied into LDS
// as they lie, once per tile.  A tile whose upper half holds padding alone (the last one of an expert) does half the work.
//
// What bounds it: a slab of the 128 x 256 tile has per wave 68 MFMAs, 217 other vector instructions (fold 128, conversion 56) and 50 LDS
// reads (36 of fragments, 8 of sums, 2 of weights, 4 table entries), of which none alone fills the 1.8 us that it takes: the MFMAs of a
// SIMD's two waves take 1.07 us by themselves, the CU's 304 KB of fragments and weights 0.63 (LDS reads of this pattern run at 480
// bytes/ns, eight waves and nothing else).  In a loop of such instructions on LDS contents, without copies, an MFMA takes 12.3 ns (two
// waves a SIMD; 7.9 alone, 8.7 with the first half of the fold, 10.8 with the whole fold and the conversion, the rest is the fragments'
// way from LDS); the kernel takes 13.2.
// About 20 of a tile's 136 thousand cycles are spent before the first slab and behind the last.  Wave tiles of 64 x 64 read half the fragments
// and convert twice the weights: the same within 2 %; the waves of a SIMD half a slab apart, the conversion a slab ahead, fragments read two
// ahead, copies at the slab's start or spread over it: no difference.
// 8 experts of N=28672 K=4096, groups of 128, bf16, 1024 tokens in blocks of 64, us of a call among others: 741 -> 594 (810 TFLOP/s) on one
// box, 736 -> 580 on another (before: 128 rows x 64 channels of every wave in two rows of waves, sums of the activations in every wave, 136
// or 1032 + q as operands, tables transposed by 2-byte stores); over 716 calls of 11 layers 5 to 30 % less than that form wherever
// this kernel has them.
#include <cmath>
#include <type_traits>

#include "wo_common.h"

namespace fnn {

// K / 128 at most, where there are group tables: they lie in LDS whole, 32 KB for 32 groups of 256 channels beside 112 KB of
// stages, and 64 groups do not fit the 160 KB.  Longer rows (K = 4224 to 8192) stay on gemm_wo_tile_kernel and the panel kernel.
constexpr int kGroups = 32;

// One tile: rows m0 .. row_end - 1 (at most BM) of the sorted list, channels n0 .. n0 + BN - 1 of one expert.
template <int ADT, bool GROUPS, int SDT, int BM, int BN>
__device__ __forceinline__ void moe_tile(const WoArgs& p, const MoeArgs& q, const int m0, const int n0, const int row_end,
                                         const int expert) {
    typedef MfmaT<ADT> MT;
    constexpr int WROWS = BN / 2;                    // weight rows (two channels each) per workgroup
    constexpr int NWV = BN / 32, NT = NWV * 64;      // waves (all rows and 32 channels each), threads
    constexpr int FB = BM / 16;                      // activation fragments
    constexpr int NA = 2;                            // weight operands per k-step: even and odd channels
    constexpr int ASTG = BM * 256, WSTG = WROWS * 128;
    static_assert(FB == NWV, "every wave sums up one activation fragment");
    __shared__ __attribute__((aligned(1024))) char sa0[ASTG];
    __shared__ __attribute__((aligned(1024))) char sa1[ASTG];
    __shared__ __attribute__((aligned(1024))) char sw[3 * WSTG];
    __shared__ __attribute__((aligned(1024))) char tab_s[GROUPS ? kGroups * BN * 2 : 1024], tab_z[GROUPS ? kGroups * BN * 2 : 1024];
    __shared__ __attribute__((aligned(16))) int toks[BM];
    __shared__ __attribute__((aligned(16))) float factors[BM];                       // routing weights
    __shared__ __attribute__((aligned(16))) float sums[(GROUPS ? 2 : 1) * 4 * BM];   // activation sums of a slab's rows (per-channel tables: of eight slabs), four copies

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row16 = lane & 15, g = lane >> 4;
    const int KT = p.K / 128;
    const bool has_zp = p.zp != nullptr;

    int routed = 0, above = 0;
    for (int r = threadIdx.x; r < BM; r += NT) {
        const int tok = m0 + r < row_end ? q.sorted_ids[m0 + r] : q.num_valid;
        toks[r] = tok < q.num_valid ? tok : -1;
        routed |= tok < q.num_valid;
        above |= tok < q.num_valid && r >= BM / 2;
    }
    // Blocks taller than the tile: a tile may hold nothing but padding (blocks of 256 with 64 rows per expert, 8 experts N=4096
    // K=14336, per-channel tables, us: 235 -> 130; the 256-row tiles of gemm_wo_tile_kernel 218)
    if (q.block_m > BM && !__syncthreads_or(routed)) return;
    const bool upper = __syncthreads_or(above);      // whether the upper half of the rows holds a routed one

    // The tile's slice of a group table is contiguous, [channel][group]: copied as it lies, 16 bytes per lane, where it is aligned.
    // 16-byte chunk c of channel ch goes to place c ^ (ch / 4) of the channel's row where that is a power of two of chunks, so that
    // the 16 rows of a read do not meet in two banks.
    const int chunks = KT / 8, swz = KT % 8 == 0 && (chunks & (chunks - 1)) == 0 ? chunks - 1 : 0;
    if constexpr (GROUPS) {
        auto stage_table = [&](const void* table, int64_t stride_be, char* to) {
            const char* const src = (const char*)table + ((int64_t)expert * stride_be + (int64_t)n0 * KT) * 2;
            if (((uintptr_t)src & 15) == 0) {
                for (int i = wave; i < (BN * KT * 2 + 1023) / 1024; i += NWV) {
                    int e = i * 64 + lane;
                    if (swz) {
                        const int ch = e / chunks;
                        e ^= (ch >> 2) & swz;
                    }
                    copy_to_lds_16(src, min(e, BN * KT / 8 - 1) * 16, lds_address(to) + i * 1024);
                }
            } else {
                for (int e = threadIdx.x; e < BN * KT; e += NT) {
                    const int ch = e / KT, k = e % KT;
                    *(uint16_t*)(to + ch * KT * 2 + (((k >> 3) ^ ((ch >> 2) & swz)) << 4) + (k & 7) * 2) = ((const uint16_t*)src)[e];
                }
            }
        };
        stage_table(p.scale, q.stride_scale_be, tab_s);
        if (has_zp) stage_table(p.zp, q.stride_zp_be, tab_z);
    }

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
    // copy number i of the NCA + NCW that fill stage `a` with the activations of slab ja and stage `w` with the weights of slab jw
    auto copy = [&](int i, uint32_t a, int ja, uint32_t w, int jw) {
        if (i < NCA) copy_to_lds_16((const char*)p.act + (int64_t)min(ja, KT - 1) * 256, ga[i], a + (i * NWV + wave) * 1024);
        else copy_to_lds_16(w_base + (int64_t)min(jw, KT - 1) * 128, gw[i - NCA], w + ((i - NCA) * NWV + wave) * 1024);
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
    for (int h = 0; h < 2; ++h) w_rd[h] = (wave * 16 + row16) * 128 + (((4 * h + g) ^ ((row16 >> 1) & 7)) << 4);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int s = 0; s < 2; ++s) a_rd[h][s] = row16 * 256 + (((8 * h + 2 * g + s) ^ row16) << 4);
    // the lane's even channel in a table, and what its chunks are XORed with
    const int t_rd = (wave * 32 + 2 * row16) * KT * 2, t_swz = ((wave * 32 + 2 * row16) >> 2) & swz;

    v4f outv[NA][FB];
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
        for (int a = 0; a < NA; ++a) outv[a][b] = v4f{0, 0, 0, 0};
    const v4u ones = v4u{MT::one2, MT::one2, MT::one2, MT::one2};
    const v4f zero4 = v4f{0, 0, 0, 0};
    // (the lanes of every g keep a copy of their own, so that neither writing nor reading one takes a branch)
    const int s_wr = g * BM + wave * 16 + row16, s_rd = g * BM + 4 * g;
    v4f own = zero4;     // activation sums of the wave's share of the rows: fragment `wave`
    float nz[NA];        // what the sums are taken off with: -s * (8 + zp) of the slab before, per-channel tables -(8 + zp)
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        nz[a] = 0.f;
        if constexpr (!GROUPS) {
            const int n = n0 + wave * 32 + 2 * row16 + a;
            nz[a] = rounded_f32(-8.f - (has_zp ? load_as_f32(p.zp, (int64_t)expert * q.stride_zp_be + n, p.zp_dtype) : 0.f));
        }
    }

    typedef v4u Operands[4][NA];
    auto convert = [&](int at, Operands& A) {
#pragma unroll
        for (int h = 0; h < 2; ++h) convert_w4_u<ADT>(*(const v4u*)(sw + at + w_rd[h]), A[2 * h][0], A[2 * h + 1][0], A[2 * h][1], A[2 * h + 1][1]);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](auto frags, const char* sa, int j, float* sums_now, const float* sums_before, const Operands& A, auto beside) {
        constexpr int F = decltype(frags)::value;
        v4u B[2][4];
        auto read_b = [&](int b, int at) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) B[at][ks] = *(const v4u*)(sa + a_rd[ks >> 1][ks & 1] + b * 16 * 256);
        };
        read_b(0, 0);
        float sc[NA], zc[NA];
        if constexpr (GROUPS) {
            const int at = t_rd + (((j >> 3) ^ t_swz) << 4) + (j & 7) * 2;
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                sc[a] = bits_to_f32<SDT>(*(const uint16_t*)(tab_s + at + a * KT * 2));
                const float z = bits_to_f32<SDT>(*(const uint16_t*)(tab_z + at + a * KT * 2));
                zc[a] = has_zp ? -8.f - z : -8.f;
            }
        }
        v4f acc[2][NA], sm[2];
#pragma unroll
        for (int b = 0; b <= F; ++b) {
            beside(b);
            if (b < F) read_b(b + 1 < F ? b + 1 : min(wave, F - 1), (b + 1) & 1);
            if constexpr (GROUPS)
                if (b < F) sm[b & 1] = *(const v4f*)(sums_before + s_rd + b * 16);
            if (b < F) {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const v4u bv = B[b & 1][ks];
#pragma unroll
                    for (int a = 0; a < NA; ++a) {
                        if constexpr (GROUPS) acc[b & 1][a] = MT::mma(bv, A[ks][a], ks == 0 ? zero4 : acc[b & 1][a]);
                        else outv[a][b] = MT::mma(bv, A[ks][a], outv[a][b]);
                    }
                }
            } else {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) own = MT::mma(ones, B[b & 1][ks], GROUPS && ks == 0 ? zero4 : own);
            }
            if constexpr (GROUPS)
                if (b > 0) {
#pragma unroll
                    for (int a = 0; a < NA; ++a)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float t = __builtin_fmaf(nz[a], sm[(b - 1) & 1][r], outv[a][b - 1][r]);
                            outv[a][b - 1][r] = __builtin_fmaf(sc[a], acc[(b - 1) & 1][a][r], t);
                        }
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (GROUPS) {
#pragma unroll
            for (int a = 0; a < NA; ++a) nz[a] = sc[a] * zc[a];
            sums_now[s_wr] = own[0];
        }
    };

    float* const se = sums;                                       // of slabs 0, 2, ..
    float* const so = sums + (GROUPS ? 4 * BM : 0);
    if constexpr (GROUPS) so[s_wr] = 0.f;
    auto take_off = [&](const float* of) {
#pragma unroll
        for (int b = 0; b < FB; ++b) {
            const v4f sm = *(const v4f*)(of + s_rd + b * 16);
#pragma unroll
            for (int a = 0; a < NA; ++a)
#pragma unroll
                for (int r = 0; r < 4; ++r) outv[a][b][r] = __builtin_fmaf(nz[a], sm[r], outv[a][b][r]);
        }
    };
    // prologue, in the order the loop issues them: slab 0 whole, then the weights of slab 1
#pragma unroll
    for (int i = 0; i < NCA + NCW; ++i) copy(i, lds_address(sa0), 0, lds_address(sw), 0);
#pragma unroll
    for (int i = NCA; i < NCA + NCW; ++i) copy(i, 0, 0, lds_address(sw) + WSTG, 1);
    __builtin_amdgcn_sched_barrier(0);
    for (int r = threadIdx.x; r < BM; r += NT)
        factors[r] = q.mul_w && toks[r] >= 0 ? load_as_f32(q.topk_w, toks[r], q.topk_w_dtype) : 1.f;
    // the walk over K with the first F fragments of the tile's rows
    auto walk = [&](auto frags) {
        constexpr int F = decltype(frags)::value, LOADS = NCA * F / FB + NCW, PER = (LOADS + F - 2) / (F - 1);
        Operands A;
        int w0 = 0, w1 = WSTG, w2 = 2 * WSTG;        // weight stages of this slab, the next and the one after
        auto step = [&](const char* now, char* next, int j, float* sums_now, const float* sums_before) {
            wait_barrier();
            convert(w0, A);
            multiply(frags, now, j, sums_now, sums_before, A, [&](int b) {
#pragma unroll
                for (int i = b * PER; i < min((b + 1) * PER, LOADS); ++i)
                    copy(i < LOADS - NCW ? i : i - LOADS + NCW + NCA, lds_address(next), j + 1, lds_address(sw) + w2, j + 2);
            });
            __builtin_amdgcn_sched_barrier(0);
            const int t = w0;
            w0 = w1, w1 = w2, w2 = t;
        };
        for (int j = 0; j < KT; j += 2) {        // (KT is even: checked on the host)
            step(sa0, sa1, j, se, so);
            step(sa1, sa0, j + 1, so, se);
            // Per-channel tables: the activations' share of the sums comes off every eight slabs, so that they do not grow with K
            // beyond the result (error beside the output's rounding, K = 14336, all-positive activations, fp16 / bf16: 2.2e-6 / 1.6e-6
            // with one correction at the end, 6.6e-7 / 5.7e-7 with these; 1.4e-6 / 6.2e-7 with one per slab and operands of 1032 / 136
            // + q).  It costs 2 to 5 % (N=4096, 64 rows per expert 89 -> 94 us; 128.5 in that form).
            if constexpr (!GROUPS)
                if ((j & 6) == 6 && j + 2 < KT) {
                    se[s_wr] = own[0];
                    own = zero4;
                    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    take_off(se);
                }
        }
    };
    if (BM == 128 && !upper) walk(std::integral_constant<int, FB / 2>{});
    else walk(std::integral_constant<int, FB>{});

    // what is left of the zero points: the last slab's (group tables; KT is even, so its sums lie in `so`) or the last slabs'
    if constexpr (!GROUPS) se[s_wr] = own[0];
    __syncthreads();
    take_off(GROUPS ? so : se);
    if constexpr (!GROUPS) {
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const float sc = load_as_f32(p.scale, (int64_t)expert * q.stride_scale_be + n0 + wave * 32 + 2 * row16 + a, p.scale_dtype);
#pragma unroll
            for (int b = 0; b < FB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) outv[a][b][r] *= sc;
        }
    }

    // lane (row16, g) holds, of fragment b, rows 4 g .. + 3 and channels 2 row16, + 1
    const bool pairs = (p.ldc % 2) == 0 && ((uintptr_t)p.out % 4) == 0;
#pragma unroll
    for (int b = 0; b < FB; ++b) {
        const v4i tk = *(const v4i*)(toks + b * 16 + 4 * g);
        const v4f un = *(const v4f*)(factors + b * 16 + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = tk[r];
            if (m < 0) continue;
            uint16_t* dst = (uint16_t*)p.out + (int64_t)m * p.ldc + n0 + wave * 32 + 2 * row16;
            const uint32_t b0 = f32_to_bits<ADT>(rounded_f32(outv[0][b][r] * un[r])), b1 = f32_to_bits<ADT>(rounded_f32(outv[1][b][r] * un[r]));
            if (pairs) {
                *(uint32_t*)dst = (b0 & 0xFFFFu) | (b1 << 16);
            } else {
                dst[0] = (uint16_t)b0;
                dst[1] = (uint16_t)b1;
            }
        }
    }
}

template <int ADT, bool GROUPS, int SDT, int BM, int BN>
__global__ __launch_bounds__(BN * 2, 2) void gemm_wo_moe_kernel(const WoArgs p, const MoeArgs q) {
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
        moe_tile<ADT, GROUPS, SDT, BM, BN>(p, q, m0, (grp * GN + rem % gcols) * BN, m0 + rows, expert);
        __builtin_amdgcn_s_waitcnt(0x0070);     // copies of slabs beyond the last are still on their way into LDS
        __syncthreads();
    }
}

template <int ADT, int BM, int BN>
static void launch_t(const WoArgs& p, const MoeArgs& q, hipStream_t st) {
    const dim3 grid((unsigned)((moe_tiles_estimate(q, BM) * (p.N / BN) + 7) / 8 * 8)), block(BN * 2);
    note_kernel(p.group ? "gemm_wo_moe_kernel(group tables)" : "gemm_wo_moe_kernel", 4, BM, BN);
    if (p.group == 0) gemm_wo_moe_kernel<ADT, false, FNN_F16, BM, BN><<<grid, block, 0, st>>>(p, q);
    else if (p.scale_dtype == FNN_F16) gemm_wo_moe_kernel<ADT, true, FNN_F16, BM, BN><<<grid, block, 0, st>>>(p, q);
    else gemm_wo_moe_kernel<ADT, true, FNN_BF16, BM, BN><<<grid, block, 0, st>>>(p, q);
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
    // Rows of an expert, and what the panel kernel makes of them: it reads the expert's weights once per block of 16 rows.  With
    // one such block and matrices wide enough for its workgroups it stays ahead (panel kernel / 64-row tiles, us - 8 experts N=28672
    // K=4096, groups of 128: 4 rows per expert 102 / 161, 16 rows 136 / 159, 25 rows 190 / 156; 16 experts N=12288 K=4096: 2 rows 94 /
    // 101, 8 rows 138 / 133, 12 rows 165 / 133; per-channel tables, 8 experts N=4096 K=14336: 8 rows 72 / 76, 16 rows 104 / 77; 16
    // experts N=10752 K=6144: 8 rows 131 / 148, 16 rows 171 / 151).
    const int64_t experts = moe_experts_estimate(q), mean = (q.num_valid + experts - 1) / experts;
    const int64_t padded = (mean + q.block_m - 1) / q.block_m * q.block_m;
    if (panel && padded <= 16 && (p.N >= 20480 || (mean <= 10 && (p.N >= 8192 || p.K >= 8192)))) return false;
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
    // The tile: 128 x 256 where the rows fill half of it and more and its rounds are full, 64 x 128 (two workgroups per CU) elsewhere.
    // 64 x 128 / 128 x 256, us, 8 experts N=28672 K=4096, groups of 128: 100 rows per expert 306 / 283, 175 rows 478 / 464; 16 experts
    // N=12288 K=4096: 32 rows 139 / 144, 88 rows 259 / 219, 256 rows 567 / 494; per-channel tables, 8 experts N=4096 K=14336: 100 rows,
    // 0.5 rounds of wide tiles 116 / 157, 175 rows, 1.0 rounds 207 / 182, 250 rows, 1.2 rounds 287 / 335, 512 rows, 2.2 rounds 515 / 535;
    // 4 experts N=16384 K=5120: 64 rows, 1.0 rounds 75 / 69, 250 rows, 2.3 rounds 199 / 186.
    auto fits = [&](int bm) { return q.block_m % bm == 0 || bm % q.block_m == 0; };
    // Less than three rounds count whole: blocks of 128 and more by what narrow tiles would take (of whose rounds what is left over runs
    // beside the end of the one before), smaller ones by how full the rounds are.  Smaller blocks around one round (0.9 to 1.1) stay on
    // narrow tiles: how many tiles they make is known on the device only, and one more is a second round.  64 x 128 / 128 x 256 there, us, even
    // routing and then uneven (scores of the first expert two standard deviations above the last's), blocks of 64, groups of 128: 16 experts
    // N=4096 K=4096, 80 rows 80 / 66 and 80 / 117; 16 experts N=2048, 200 rows 81 / 66 and 81 / 118; per-channel tables, 8 experts N=4096
    // K=14336, 200 rows 207 / 179 and 210 / 289; 4 experts N=16384 K=5120, 96 rows 84 / 74 and 84 / 92.  Taken wide are only those whose
    // experts nearly fill their tiles (the estimate, which counts a partial tile more for each, comes to two rounds: from 97 rows with
    // 4 experts), which lose less: N=16384 K=5120, 100 rows 84 / 74 and 83 / 90; K=4096 with groups of 128 82 / 69 and 82 / 83.
    const double rounds = moe_rounds(q, p.N, 128, 256, 256), whole = ceil(rounds - 0.05);
    bool wide = mean > 60 && (rounds >= 3 || (q.block_m % 128 == 0 ? moe_rounds(q, p.N, 64, 128, 512) + 0.25 > 1.5 * whole
                                                                   : (rounds >= 1.1 || moe_tiles_estimate(q, 128) * (p.N / 256) >= 512) && whole < 1.34 * rounds));
    wide = wide && fits(128) && p.N % 256 == 0;
    if (!wide && !fits(64)) return false;
    auto run = [&](auto adt) {
        constexpr int ADT = decltype(adt)::value;
        if (wide) launch_t<ADT, 128, 256>(p, q, st);
        else launch_t<ADT, 64, 128>(p, q, st);
    };
    if (act_dtype == FNN_F16) run(std::integral_constant<int, FNN_F16>{});
    else run(std::integral_constant<int, FNN_BF16>{});
    return true;
}

}  // namespace fnn
