// K ping-pong: the 128 x 128 tile with two groups of four waves that take alternate K stages.
//
// One workgroup of 8 waves, two per SIMD (waves w and w + 4 share SIMD w % 4).  Each group of
// four waves holds the whole 128 x 128 tile as 2 x 2 wave tiles of 64 x 64 and sums every
// second 128-byte stage of K: in phase p the group of parity p reads the fragments of stage p
// from LDS into registers while the other group runs the MFMAs of stage p - 1, so on every
// SIMD one wave keeps the matrix core busy while the other feeds itself.  One workgroup
// barrier per stage.  At the end the groups exchange half of their partial sums through LDS.
//
//   phase      2i                    2i+1                  2i+2
//   group 0    read stage 2i         compute stage 2i      read stage 2i+2
//   group 1    compute stage 2i-1    read stage 2i+1       compute stage 2i+1
//
// A ring of four 32 KiB stages: the loads of stage p + 3 go out in phase p into the buffer that
// phase p - 1 read, so three stages (96 KiB per CU) are in flight, and a wave waits at the end of
// a phase only for its own loads of the next stage.
//
// What bounds it: LDS traffic (64 KiB of fragment reads and 32 KiB of loads per stage, 768 of the
// ~900 cycles a stage takes) and, on long runs, the board's power limit.  The interleaved 128 x
// 128 tile (mfma16.hpp) has one wave per SIMD and one stage in flight, and waited for both.
// MI355X, bf16, us, best earlier tile -> K ping-pong (torch.matmul): 2048 x 2048 x 4096 41.5 ->
// 32.7 (38.9), 2048^3 25.4 -> 19.9 (24.2), 1536 x 1536 x 4096 39.0 -> 33 (34.6), 2560^3 42.6 -> 35.9
// (40.2, 256 x 128), 2048 x 4096 x 2048 36.8 -> 34.7 (36.8, 256 x 128).
#pragma once

#include <type_traits>

#include "mfma16.hpp"

namespace mb {
namespace m16 {

// What the two 32-deep halves of a stage hold.  kPlain: the next 64 k.  kSplitReal / kSplitComplex
// (K-contiguous fp16, gemm_split32.hip): the high and the low parts of the same 32 k, complex
// ones as (re, im) pairs along k; the B tile of a complex product is 64 complex columns wide, and
// the two real columns of each, (re, -im) and (im, re) with the signs of the conjugations, are made
// from one fragment in registers.
enum KppMode { kPlain, kSplitReal, kSplitComplex };

template <class T, bool A_KC, bool B_KC, bool KTAIL, KppMode MODE> struct Kpp {
    static constexpr bool SPLIT = MODE != kPlain, CPLX = MODE == kSplitComplex;
    static constexpr int BM = 128, BN = 128, NW = 8, NB = 4, MS = 16;
    static constexpr int TM = 4, TN = 4;   // 16 x 16 blocks of a 64 x 64 wave tile
    static constexpr int ES = sizeof(T), BK = 128 / ES;
    using TA = Tile16<BM, NW, A_KC, ES, MS>;
    using TB = Tile16<CPLX ? BN / 2 : BN, NW, B_KC, ES, MS>;
    using Acc = typename AccT<T, MS>::type;
    static constexpr int STAGE = TA::BYTES + TB::BYTES;
    static constexpr int LPW = TA::PER_WAVE + TB::PER_WAVE;   // loads per wave and stage
    static constexpr int SMEM = NB * STAGE;
    static constexpr int SETS = SPLIT ? 2 : 1;   // accumulator sets
    static_assert(TA::SEGS % NW == 0 && TB::SEGS % NW == 0, "every wave issues the same loads");

    // Sums A[m0.., kbeg..kend) x B[.., n0..) into this wave's half of the tile: on return group 0
    // holds column blocks 0, 1 of its 64 x 64 wave tile in out, group 1 blocks 2, 3.
    // Ab / Bb: element (m0, kbeg) / (kbeg, n0).  Complex: out[0] / out[1] are the real / imaginary
    // parts of the group's 16 complex columns; sign_re / sign_im: sign bits flipped in the (re, im)
    // halves of a pair for the real and (after swapping them) the imaginary column.
    __device__ __forceinline__ static void run(const T *Ab, const T *Bb, int64_t lda, int64_t ldb, int rows_a,
                                               int rows_b, int klen, char *smem, int wave, int lane,
                                               Acc (&out)[2][TM], uint32_t sign_re = 0, uint32_t sign_im = 0) {
        const uint32_t smem_lds = lds_addr(smem);
        const int group = wave >> 2, wm = wave & 1, wn = (wave >> 1) & 1;
        const int nk = cdiv(klen, BK), nfull = klen / BK;
        const int stepa = (int)((A_KC ? (int64_t)BK : (int64_t)BK * lda) * ES);
        const int stepb = (int)((B_KC ? (int64_t)BK : (int64_t)BK * ldb) * ES);
        const i32x4 ra = make_rsrc(Ab), rb = make_rsrc(Bb);
        uint32_t offa[TA::PER_WAVE], offb[TB::PER_WAVE];
#pragma unroll
        for (int i = 0; i < TA::PER_WAVE; ++i) offa[i] = TA::src_offset(wave + i * NW, lane, lda, rows_a, BK);
#pragma unroll
        for (int i = 0; i < TB::PER_WAVE; ++i) offb[i] = TB::src_offset(wave + i * NW, lane, ldb, rows_b, BK);
        int fba[A_KC ? 1 : TM], fbb[B_KC ? 1 : TN];
#pragma unroll
        for (int j = 0; j < (A_KC ? 1 : TM); ++j) fba[j] = TA::frag_base16(wm * 64, lane, j);
#pragma unroll
        for (int j = 0; j < (B_KC ? 1 : TN); ++j) fbb[j] = TB::frag_base16(wn * (CPLX ? 32 : 64), lane, j);

        // load `op` of this wave's share of stage kt (EDGE: the stage that holds the K edge)
        auto load_op = [&](auto edge_tag, int kt, int op) {
            constexpr bool EDGE = decltype(edge_tag)::value;
            const uint32_t base = smem_lds + (kt & (NB - 1)) * STAGE;
            const int kleft = klen - kt * BK;
            if (op < TA::PER_WAVE) {
                const int seg = wave + op * NW;
                dma16(ra, base + seg * 1024, EDGE ? TA::src_offset(seg, lane, lda, rows_a, kleft) : offa[op], kt * stepa);
            } else {
                const int ib = op - TA::PER_WAVE, seg = wave + ib * NW;
                dma16(rb, base + TA::BYTES + seg * 1024, EDGE ? TB::src_offset(seg, lane, ldb, rows_b, kleft) : offb[ib],
                      kt * stepb);
            }
        };
        auto load_stage = [&](int kt) {
            if (!KTAIL || kt < nfull) {
#pragma unroll
                for (int op = 0; op < LPW; ++op) load_op(std::false_type{}, kt, op);
            } else {
#pragma unroll
                for (int op = 0; op < LPW; ++op) load_op(std::true_type{}, kt, op);
            }
        };

        Acc acc[SETS][TN][TM];
#pragma unroll
        for (int t = 0; t < SETS; ++t)
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[t][i][j][r] = 0;

        uint4 fa[2][TM], fb[2][TN];
        auto read_stage = [&](int kt) {
            const char *cur = smem + (kt & (NB - 1)) * STAGE;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int j = 0; j < TM; ++j) fa[s][j] = TA::frag16(cur, fba[A_KC ? 0 : j], lane, s, A_KC ? j : 0);
                if constexpr (CPLX) {
#pragma unroll
                    for (int c = 0; c < TN / 2; ++c) fb[s][2 * c] = TB::frag16(cur + TA::BYTES, fbb[0], lane, s, c);
                } else {
#pragma unroll
                    for (int i = 0; i < TN; ++i)
                        fb[s][i] = TB::frag16(cur + TA::BYTES, fbb[B_KC ? 0 : i], lane, s, B_KC ? i : 0);
                }
            }
            if constexpr (CPLX) {
                auto swap = [](uint32_t v) { return __builtin_amdgcn_alignbit(v, v, 16); };
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int c = 0; c < TN / 2; ++c) {
                        const uint4 v = fb[s][2 * c];
                        fb[s][2 * c + 1] = make_uint4(swap(v.x) ^ sign_im, swap(v.y) ^ sign_im, swap(v.z) ^ sign_im,
                                                      swap(v.w) ^ sign_im);
                        fb[s][2 * c] = make_uint4(v.x ^ sign_re, v.y ^ sign_re, v.z ^ sign_re, v.w ^ sign_re);
                    }
            }
        };
        // The MFMAs of the stage in registers.  Plain: both k halves into one accumulator set.
        // SPLIT: half 0 of the stage holds the high parts and half 1 the low parts of the same
        // k, set 0 sums high x high and set 1 the two cross products.
        // PF: this wave's loads of stage pk issued between the MFMAs (an MFMA, then one load per
        // EVERY MFMAs; no condition between them: a VALU compare would wait for the MFMA ahead).
        constexpr int NMMA = (SPLIT ? 3 : 2) * TM * TN, EVERY = NMMA / LPW;
        auto compute_stage = [&](auto pf_tag, auto edge_tag, int pk) {
            constexpr bool PF = decltype(pf_tag)::value;
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int s = 0; s < (SPLIT ? 3 : 2); ++s)
#pragma unroll
                for (int i = 0; i < TN; ++i)
#pragma unroll
                    for (int j = 0; j < TM; ++j) {
                        if constexpr (SPLIT)
                            mma_blk<T, MS>(acc[s ? 1 : 0][i][j], fb[s == 1][i], fa[s == 2][j]);
                        else
                            mma_blk<T, MS>(acc[0][i][j], fb[s][i], fa[s][j]);
                        const int idx = (s * TN + i) * TM + j;
                        if (PF && idx % EVERY == 0 && idx / EVERY < LPW) {
                            __builtin_amdgcn_sched_barrier(0);
                            load_op(edge_tag, pk, idx / EVERY);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
            __builtin_amdgcn_s_setprio(0);
        };
        auto barrier = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        };
        // end of phase p: this wave's loads of stage p + 1 have landed (those of p + 2 and p + 3,
        // when issued, stay in flight), and every wave is done reading stage p
        auto phase_end = [&](int p) {
            __builtin_amdgcn_sched_barrier(0);
            if (p + 3 < nk) vm_wait_n<2 * LPW>();
            else if (p + 2 < nk) vm_wait_n<LPW>();
            else vm_wait_all();
            barrier();
        };

        // stages 0 .. 2 before the loop; the wait publishes stage 0
#pragma unroll
        for (int s = 0; s < NB - 1; ++s)
            if (s < nk) load_stage(s);
        phase_end(-1);
        const int nph = __builtin_amdgcn_readfirstlane((nk + 1) & ~1);   // phases, rounded up to even
        // phases whose loads (stage p + 3) are full stages need no edge code
        const int pf_full = __builtin_amdgcn_readfirstlane((KTAIL ? nfull : nk) - 3);
        if (group == 1) {   // phase 0 of group 1: only its loads of stage 3
            if (3 < nk) load_stage(3);
            phase_end(0);
        }
        // one group's two phases p0 (read stage p0) and p0 + 1 (compute it)
        int p = group;
        for (; p + 1 < pf_full; p += 2) {
            read_stage(p);
#pragma unroll
            for (int op = 0; op < LPW; ++op) load_op(std::false_type{}, p + 3, op);
            __builtin_amdgcn_sched_barrier(0);
            vm_wait_n<2 * LPW>();
            barrier();
            compute_stage(std::true_type{}, std::false_type{}, p + 4);
            __builtin_amdgcn_sched_barrier(0);
            vm_wait_n<2 * LPW>();
            barrier();
        }
        for (; p < nph; p += 2) {
            const bool on = p < nk;
            if (on) read_stage(p);
            if (p + 3 < nk) load_stage(p + 3);
            phase_end(p);
            if (p + 4 < nk) load_stage(p + 4);
            if (on) compute_stage(std::false_type{}, std::false_type{}, 0);
            phase_end(p + 1);
        }
        if (group == 0) barrier();   // the phase that group 1 starts late

        if constexpr (SPLIT) {   // the low parts carry a factor 2^11
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[0][i][j] += acc[1][i][j] * (1.f / 2048.f);
        }
        // exchange: each group hands the other the half of the column blocks it does not keep
        // (one float4 per block and lane, lane-contiguous; every operand stage has been read)
        auto slot = [&](int grp, int i, int j) {
            return (Acc *)(smem + (((grp * 4 + (wave & 3)) * 2 + i) * TM + j) * 1024 + lane * 16);
        };
        if (group == 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) *slot(1, i, j) = acc[0][2 + i][j];
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) *slot(0, i, j) = acc[0][i][j];
        }
        __syncthreads();
        if (group == 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) out[i][j] = acc[0][i][j] + *slot(0, i, j);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) out[i][j] = acc[0][2 + i][j] + *slot(1, i, j);
        }
    }
    // bytes of the exchange area at the front of smem; what is staged there next starts after it
    static constexpr int XBYTES = 2 * 4 * 2 * TM * 1024;
};

// The 256 x 128 tile of the same idea: each group of four waves holds the whole tile as 2 x 2 wave
// tiles of 128 x 64 and group g sums the 32-deep half g of every stage, so a phase is half a
// stage (32 MFMAs per wave, as above) and only 48 registers of fragments are live beside the 128
// accumulators.  What bounds the 128 x 128 tile is LDS traffic: per 64 x 64 of output a stage
// moves 24 KiB there (reads and the loads' writes) and 18 KiB here, against 26 KiB with the 128
// x 32 wave tiles of the two-group ping-pong at 256 x 128.
//
//   phase      2k                          2k+1                      2k+2
//   group 0    read stage k, half 0        compute it                read stage k+1, half 0
//   group 1    compute stage k-1, half 1   read stage k, half 1      compute it
//
// A ring of three 48 KiB stages: stage k + 2 is loaded in phases 2k and 2k+1 into the buffer of
// stage k - 1, read out in phase 2k - 1; two stages are in flight.
template <class T, bool A_KC, bool B_KC, bool KTAIL> struct KppWide {
    static constexpr int BM = 256, BN = 128, NW = 8, NB = 3, MS = 16;
    static constexpr int TM = 8, TN = 4;   // 16 x 16 blocks of a 128 x 64 wave tile
    static constexpr int ES = sizeof(T), BK = 128 / ES;
    using TA = Tile16<BM, NW, A_KC, ES, MS>;
    using TB = Tile16<BN, NW, B_KC, ES, MS>;
    using Acc = typename AccT<T, MS>::type;
    static constexpr int STAGE = TA::BYTES + TB::BYTES;
    static constexpr int LPW = TA::PER_WAVE + TB::PER_WAVE, HALF = LPW / 2;   // loads per wave: stage, phase
    static constexpr int SMEM = NB * STAGE;
    static_assert(TA::SEGS % NW == 0 && TB::SEGS % NW == 0 && LPW % 2 == 0, "every wave issues the same loads");

    // as Kpp::run; on return smem is free once every wave has passed a barrier
    __device__ __forceinline__ static void run(const T *Ab, const T *Bb, int64_t lda, int64_t ldb, int rows_a,
                                               int rows_b, int klen, char *smem, int wave, int lane, Acc (&out)[2][TM]) {
        const uint32_t smem_lds = lds_addr(smem);
        const int group = wave >> 2, wm = wave & 1, wn = (wave >> 1) & 1;
        const int nk = cdiv(klen, BK), nfull = klen / BK;
        const int stepa = (int)((A_KC ? (int64_t)BK : (int64_t)BK * lda) * ES);
        const int stepb = (int)((B_KC ? (int64_t)BK : (int64_t)BK * ldb) * ES);
        const i32x4 ra = make_rsrc(Ab), rb = make_rsrc(Bb);
        uint32_t offa[TA::PER_WAVE], offb[TB::PER_WAVE];
#pragma unroll
        for (int i = 0; i < TA::PER_WAVE; ++i) offa[i] = TA::src_offset(wave + i * NW, lane, lda, rows_a, BK);
#pragma unroll
        for (int i = 0; i < TB::PER_WAVE; ++i) offb[i] = TB::src_offset(wave + i * NW, lane, ldb, rows_b, BK);
        int fba[A_KC ? 1 : TM], fbb[B_KC ? 1 : TN];
#pragma unroll
        for (int j = 0; j < (A_KC ? 1 : TM); ++j) fba[j] = TA::frag_base16(wm * 128, lane, j);
#pragma unroll
        for (int j = 0; j < (B_KC ? 1 : TN); ++j) fbb[j] = TB::frag_base16(wn * 64, lane, j);

        // load `op` of this wave's share of stage kt into buffer buf
        auto load_op = [&](auto edge_tag, int kt, int buf, int op) {
            constexpr bool EDGE = decltype(edge_tag)::value;
            const uint32_t base = smem_lds + buf * STAGE;
            const int kleft = klen - kt * BK;
            if (op < TA::PER_WAVE) {
                const int seg = wave + op * NW;
                dma16(ra, base + seg * 1024, EDGE ? TA::src_offset(seg, lane, lda, rows_a, kleft) : offa[op], kt * stepa);
            } else {
                const int ib = op - TA::PER_WAVE, seg = wave + ib * NW;
                dma16(rb, base + TA::BYTES + seg * 1024, EDGE ? TB::src_offset(seg, lane, ldb, rows_b, kleft) : offb[ib],
                      kt * stepb);
            }
        };
        // loads first .. first + n - 1 of stage kt, if there is such a stage
        auto load_part = [&](int kt, int buf, auto first_tag, auto n_tag) {
            constexpr int F = decltype(first_tag)::value, N = decltype(n_tag)::value;
            if (kt >= nk) return;
            if (!KTAIL || kt < nfull) {
#pragma unroll
                for (int op = F; op < F + N; ++op) load_op(std::false_type{}, kt, buf, op);
            } else {
#pragma unroll
                for (int op = F; op < F + N; ++op) load_op(std::true_type{}, kt, buf, op);
            }
        };
        using C0 = std::integral_constant<int, 0>;
        using CH = std::integral_constant<int, HALF>;
        using CL = std::integral_constant<int, LPW>;

        Acc acc[TN][TM];
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = 0;

        uint4 fa[TM], fb[TN];
        auto read_half = [&](int buf) {
            const char *cur = smem + buf * STAGE;
#pragma unroll
            for (int i = 0; i < TN; ++i)
                fb[i] = group == 0 ? TB::frag16(cur + TA::BYTES, fbb[B_KC ? 0 : i], lane, 0, B_KC ? i : 0)
                                   : TB::frag16(cur + TA::BYTES, fbb[B_KC ? 0 : i], lane, 1, B_KC ? i : 0);
#pragma unroll
            for (int j = 0; j < TM; ++j)
                fa[j] = group == 0 ? TA::frag16(cur, fba[A_KC ? 0 : j], lane, 0, A_KC ? j : 0)
                                   : TA::frag16(cur, fba[A_KC ? 0 : j], lane, 1, A_KC ? j : 0);
        };
        // the MFMAs of the half stage in registers; PF: loads first .. first + HALF - 1 of stage pk
        // (a full one) between them
        constexpr int NMMA = TM * TN, EVERY = NMMA / HALF;
        auto compute = [&](auto pf_tag, int pk, int buf, auto first_tag) {
            constexpr bool PF = decltype(pf_tag)::value;
            constexpr int F = decltype(first_tag)::value;
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    mma_blk<T, MS>(acc[i][j], fb[i], fa[j]);
                    const int idx = i * TM + j;
                    if (PF && idx % EVERY == 0 && idx / EVERY < HALF) {
                        __builtin_amdgcn_sched_barrier(0);
                        load_op(std::false_type{}, pk, buf, F + idx / EVERY);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            __builtin_amdgcn_s_setprio(0);
        };
        auto barrier = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        };
        // this wave's loads of stage k have landed (those of stage k + 1, if any, may be pending)
        auto wait_stage = [&](int k) {
            __builtin_amdgcn_sched_barrier(0);
            if (k + 1 < nk) vm_wait_n<LPW>();
            else vm_wait_all();
        };
        auto inc = [](int b) { return b == NB - 1 ? 0 : b + 1; };

        load_part(0, 0, C0{}, CL{});
        load_part(1, 1, C0{}, CL{});
        wait_stage(0);
        barrier();
        // iterations whose loads are of full stages
        const int full = __builtin_amdgcn_readfirstlane(KTAIL ? nfull : nk);
        int k = 0, b = 0;   // stage k in buffer b; stage k + 2 goes to buffer b - 1
        if (group == 0) {
            for (; k + 2 < full; ++k, b = inc(b)) {
                const int bl = inc(inc(b));
                read_half(b);
#pragma unroll
                for (int op = 0; op < HALF; ++op) load_op(std::false_type{}, k + 2, bl, op);
                barrier();
                compute(std::true_type{}, k + 2, bl, CH{});
                __builtin_amdgcn_sched_barrier(0);
                vm_wait_n<LPW>();
                barrier();
            }
            for (; k < nk; ++k, b = inc(b)) {
                const int bl = inc(inc(b));
                read_half(b);
                load_part(k + 2, bl, C0{}, CL{});
                barrier();
                compute(std::false_type{}, 0, 0, C0{});
                wait_stage(k + 1);
                barrier();
            }
            barrier();   // the phase that group 1 starts late
        } else {
            load_part(2, 2, C0{}, CH{});
            barrier();
            for (; k + 3 < full; ++k, b = inc(b)) {
                const int bl = inc(inc(b));
                read_half(b);
#pragma unroll
                for (int op = HALF; op < LPW; ++op) load_op(std::false_type{}, k + 2, bl, op);
                __builtin_amdgcn_sched_barrier(0);
                vm_wait_n<LPW>();
                barrier();
                compute(std::true_type{}, k + 3, b, C0{});
                barrier();
            }
            for (; k < nk; ++k, b = inc(b)) {
                const int bl = inc(inc(b));
                read_half(b);
                load_part(k + 2, bl, CH{}, CH{});
                wait_stage(k + 1);
                barrier();
                load_part(k + 3, b, C0{}, CH{});
                compute(std::false_type{}, 0, 0, C0{});
                barrier();
            }
        }

        // exchange of the column blocks that each group does not keep (see Kpp::run)
        auto slot = [&](int grp, int i, int j) {
            return (Acc *)(smem + (((grp * 4 + (wave & 3)) * 2 + i) * TM + j) * 1024 + lane * 16);
        };
        if (group == 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) *slot(1, i, j) = acc[2 + i][j];
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) *slot(0, i, j) = acc[i][j];
        }
        __syncthreads();
        if (group == 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) out[i][j] = acc[i][j] + *slot(0, i, j);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) out[i][j] = acc[2 + i][j] + *slot(1, i, j);
        }
    }
    static constexpr int XBYTES = 0;   // the staged output reuses the exchange area
};

template <class T, int BM, bool A_KC, bool B_KC, bool KTAIL>
__global__ __launch_bounds__(512) void k_gemm_kpp(GemmArgs g) {
    using K = std::conditional_t<BM == 256, KppWide<T, A_KC, B_KC, KTAIL>, Kpp<T, A_KC, B_KC, KTAIL, kPlain>>;
    using CS = CStage<T, K::BM, K::BN, K::MS>;
    static_assert(K::XBYTES + CS::BYTES <= K::SMEM, "staged output behind the exchange area");
    __shared__ __attribute__((aligned(1024))) char smem[K::SMEM];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_m = cdiv(g.M, K::BM), tiles_n = cdiv(g.N, K::BN);
    int tm, tn, ks, bz0;
    work_coords(tiles_m, tiles_n, g.swz, g.xcd_batch, tm, tn, ks, bz0);
    const int m0 = tm * K::BM, n0 = tn * K::BN;
    const int kbeg = ks * g.k_chunk;
    const int klen = min(g.K, kbeg + g.k_chunk) - kbeg;
    const int64_t lda = A_KC ? g.a_rs : g.a_cs;
    const int64_t ldb = B_KC ? g.b_cs : g.b_rs;
    // the wave's part of the tile after the exchange
    const int mw = (wave & 1) * (BM / 2), nw = ((wave >> 1) & 1) * 64 + (wave >> 2) * 32;
    for (int bz = bz0; bz < g.batch; bz += gridDim.z) {
        const T *Ab = (const T *)g.a + bz * g.a_bs + (A_KC ? (int64_t)m0 * lda + kbeg : (int64_t)kbeg * lda + m0);
        const T *Bb = (const T *)g.b + bz * g.b_bs + (B_KC ? (int64_t)n0 * ldb + kbeg : (int64_t)kbeg * ldb + n0);
        typename K::Acc out[2][K::TM];
        K::run(Ab, Bb, lda, ldb, g.M - m0, g.N - n0, klen, smem, wave, lane, out);
        if (staged_store_ok<T>(g)) {
            char *ct = smem + K::XBYTES;
            if constexpr (K::XBYTES == 0) __syncthreads();
            stage_acc<T, K::TM, 2, K::MS, CS>(g, ct, out, mw, nw, m0, n0, bz, lane);
            __syncthreads();
            if (g.c_stream)
                store_staged<T, K::BM, K::BN, K::MS, 512, true>(g, ct, m0, n0, bz, tid);
            else
                store_staged<T, K::BM, K::BN, K::MS, 512, false>(g, ct, m0, n0, bz, tid);
        } else {
            store_tile16<T, K::TM, 2, K::MS>(g, out, m0 + mw, n0 + nw, bz, ks, lane);
        }
        __syncthreads();   // LDS reuse by the next batch iteration
    }
}

template <class T, int BM, bool KTAIL>
hipError_t launch_kpp_t(bool a_kc, bool b_kc, const GemmArgs &g, dim3 grid, hipStream_t st) {
    dim3 block(512);
    if (a_kc && b_kc)
        hipLaunchKernelGGL((k_gemm_kpp<T, BM, true, true, KTAIL>), grid, block, 0, st, g);
    else if (a_kc && !b_kc)
        hipLaunchKernelGGL((k_gemm_kpp<T, BM, true, false, KTAIL>), grid, block, 0, st, g);
    else if (!a_kc && b_kc)
        hipLaunchKernelGGL((k_gemm_kpp<T, BM, false, true, KTAIL>), grid, block, 0, st, g);
    else
        hipLaunchKernelGGL((k_gemm_kpp<T, BM, false, false, KTAIL>), grid, block, 0, st, g);
    return hipGetLastError();
}
// the 128 x 128 or (bm 256) the 256 x 128 tile
template <class T> hipError_t launch_kpp(bool ktail, int bm, bool a_kc, bool b_kc, const GemmArgs &g, dim3 grid, hipStream_t st) {
    if (bm == 256)
        return ktail ? launch_kpp_t<T, 256, true>(a_kc, b_kc, g, grid, st) : launch_kpp_t<T, 256, false>(a_kc, b_kc, g, grid, st);
    return ktail ? launch_kpp_t<T, 128, true>(a_kc, b_kc, g, grid, st) : launch_kpp_t<T, 128, false>(a_kc, b_kc, g, grid, st);
}

}  // namespace m16
}  // namespace mb
