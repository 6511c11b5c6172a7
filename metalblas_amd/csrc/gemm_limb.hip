// Integer GEMM on the 8-bit matrix cores for every integer type and any element strides.
//
// An integer of n bytes is a sum of n signed bytes, a = sum_i d_i 256^i modulo 2^(8n) with d_i in
// [-128, 127]: adding 0x80 to every byte with carries and flipping the top bit of each byte gives
// the d_i in place (two instructions per word).  Then a b = sum_{i+j<n} d_i e_j 256^(i+j) modulo
// 2^(8n), so a product of n-byte integers is n (n + 1) / 2 products of signed 8-bit matrices,
// v_mfma_i32_16x16x64_i8, summed by i + j: exact, because only the low 8n bits of the result are
// kept (metalblas/integer_dispatch.py:13-19: accumulation wraps, the store truncates).  int32 takes
// 10 of them, 503 TOP/s nominal, against a 32-bit multiply-add per lane at a quarter of the
// vector rate.
//
// No LDS on the way in: a lane's fragment is 16 consecutive k of one row of A (column of B), read
// from global memory as four (int32) 16-byte loads where K is contiguous and aligned, else as 16
// element loads, and turned into byte planes with v_perm.  What bounds the small products is one
// pass of load latency, so the 16 x 16 and 32 x 32 tiles split K over the four waves of a
// workgroup (partial sums meet in LDS) and the next step's loads go out before this step's
// products.  MI355X, us, the LDS-tiled VALU kernel before -> now: int32 256^3 9.2 -> 4.3, 128^3 8.5 ->
// 3.9, 512^3 34 -> 9.9, 1024^3 213 -> 49; int16 256^3 9.1 -> 5.3; int64 256^3 11.9 -> 5.9, 1024^3 342 ->
// 113.  (16 waves of 16 x 16 for a 64 x 64 tile spilled: 64^3 14.1 against 7.6 on four of 32 x 32.)
#include "launch.hpp"
#include "tile_order.hpp"

namespace mb {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// 16 consecutive k of one row as 32-bit words in element order.
template <class T> struct Raw {
    static constexpr int W = 4 * sizeof(T);
    uint32_t w[W];
};

// VEC: ks == 1, 16-byte aligned rows, K a multiple of the 16-byte element count.
template <class T, bool VEC>
__device__ __forceinline__ void load16(Raw<T> &o, const T *row, int64_t ks, int k0, int kend, bool ok) {
    constexpr int E = 16 / (int)sizeof(T);
    if constexpr (VEC) {
#pragma unroll
        for (int c = 0; c < 16 / E; ++c) {
            uint4 v = make_uint4(0, 0, 0, 0);
            if (ok && k0 + c * E < kend) v = *(const uint4 *)(row + k0 + c * E);
            o.w[4 * c] = v.x;
            o.w[4 * c + 1] = v.y;
            o.w[4 * c + 2] = v.z;
            o.w[4 * c + 3] = v.w;
        }
    } else {
        T e[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            e[i] = 0;
            if (ok && k0 + i < kend) e[i] = row[(k0 + i) * ks];
        }
        if constexpr (sizeof(T) == 8) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                o.w[2 * i] = (uint32_t)e[i];
                o.w[2 * i + 1] = (uint32_t)((uint64_t)e[i] >> 32);
            }
        } else if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o.w[i] = (uint32_t)e[i];
        } else if constexpr (sizeof(T) == 2) {
#pragma unroll
            for (int i = 0; i < 8; ++i) o.w[i] = (uint16_t)e[2 * i] | (uint32_t)(uint16_t)e[2 * i + 1] << 16;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                o.w[i] = (uint8_t)e[4 * i] | (uint32_t)(uint8_t)e[4 * i + 1] << 8 | (uint32_t)(uint8_t)e[4 * i + 2] << 16 |
                         (uint32_t)(uint8_t)e[4 * i + 3] << 24;
        }
    }
}

// bytes of four words gathered by position: out[j] = byte j of w0, w1, w2, w3
__device__ __forceinline__ void planes4(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t (&out)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(w1, w0, 0x05010400u), b = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
    const uint32_t c = __builtin_amdgcn_perm(w3, w2, 0x05010400u), d = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
    out[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// the signed-byte planes of 16 elements: p[i] = digit i of the 16 k
template <class T> __device__ __forceinline__ void to_planes(const Raw<T> &r, i32x4 (&p)[sizeof(T)]) {
    constexpr uint32_t H = 0x80808080u;
    if constexpr (sizeof(T) == 1) {
        p[0] = i32x4{(int)r.w[0], (int)r.w[1], (int)r.w[2], (int)r.w[3]};
    } else if constexpr (sizeof(T) == 2) {
        uint32_t d[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            d[i] = (((r.w[i] + 0x8080u) & 0xffffu) | ((r.w[i] + 0x80800000u) & 0xffff0000u)) ^ H;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            p[0][q] = (int)__builtin_amdgcn_perm(d[2 * q + 1], d[2 * q], 0x06040200u);
            p[1][q] = (int)__builtin_amdgcn_perm(d[2 * q + 1], d[2 * q], 0x07050301u);
        }
    } else if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t o[4];
            planes4((r.w[4 * q] + H) ^ H, (r.w[4 * q + 1] + H) ^ H, (r.w[4 * q + 2] + H) ^ H, (r.w[4 * q + 3] + H) ^ H, o);
#pragma unroll
            for (int j = 0; j < 4; ++j) p[j][q] = (int)o[j];
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t lo[4], hi[4], o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint64_t v = ((uint64_t)r.w[2 * (4 * q + i) + 1] << 32 | r.w[2 * (4 * q + i)]) + ((uint64_t)H << 32 | H);
                lo[i] = (uint32_t)v ^ H;
                hi[i] = (uint32_t)(v >> 32) ^ H;
            }
            planes4(lo[0], lo[1], lo[2], lo[3], o);
#pragma unroll
            for (int j = 0; j < 4; ++j) p[j][q] = (int)o[j];
            planes4(hi[0], hi[1], hi[2], hi[3], o);
#pragma unroll
            for (int j = 0; j < 4; ++j) p[4 + j][q] = (int)o[j];
        }
    }
}

// Workgroup tile (16 WT WM) x (16 WT WN): a WM x WN grid of waves, each WT x WT blocks of 16 x 16,
// times KS waves that take every KS-th 64-deep step of the K slice.
template <class T, int WT, int WM, int WN, int KS, bool VA, bool VB>
__global__ __launch_bounds__(64 * WM * WN * KS) void k_gemm_limb(GemmArgs g) {
    static_assert(KS == 1 || (WM == 1 && WN == 1), "waves share either the tile or K");
    using A = typename Tr<T>::acc;
    constexpr int NL = sizeof(T), BM = 16 * WT * WM, BN = 16 * WT * WN, NW = WM * WN * KS;
    __shared__ A part[KS > 1 ? KS * WT * WT * 256 : 1];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm, tn, ks, bz0;
    work_coords(cdiv(g.M, BM), cdiv(g.N, BN), 3, g.xcd_batch, tm, tn, ks, bz0);
    const int wm = KS > 1 ? 0 : wave % WM, wn = KS > 1 ? 0 : wave / WM, wk = KS > 1 ? wave : 0;
    const int m0 = tm * BM + wm * 16 * WT, n0 = tn * BN + wn * 16 * WT;
    const int kbeg = ks * g.k_chunk, kend = min(g.K, kbeg + g.k_chunk);
    const int r16 = lane & 15, kg = 16 * (lane >> 4);

    for (int bz = bz0; bz < g.batch; bz += gridDim.z) {
        const T *ap[WT], *bp[WT];
        bool oka[WT], okb[WT];
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            const int m = m0 + 16 * j + r16, n = n0 + 16 * j + r16;
            oka[j] = m < g.M;
            okb[j] = n < g.N;
            ap[j] = (const T *)g.a + bz * g.a_bs + (oka[j] ? m : 0) * g.a_rs;
            bp[j] = (const T *)g.b + bz * g.b_bs + (okb[j] ? n : 0) * g.b_cs;
        }
        Raw<T> ra[WT], rb[WT];
        auto load = [&](int k) {
#pragma unroll
            for (int j = 0; j < WT; ++j) load16<T, VA>(ra[j], ap[j], g.a_cs, k + kg, kend, oka[j]);
#pragma unroll
            for (int j = 0; j < WT; ++j) load16<T, VB>(rb[j], bp[j], g.b_rs, k + kg, kend, okb[j]);
        };
        // tot: element (row r16, column 4 (lane / 16) + r) of block (i, j): C^T = B^T A^T
        A tot[WT][WT][4];
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < WT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) tot[i][j][r] = 0;
        int k = kbeg + 64 * wk;
        if (k < kend) load(k);
        while (k < kend) {
            // the 32-bit sums hold 2^31 / (NL 2^14) products without wrapping, which the 64-bit
            // result needs: add them up every 8192 k (narrower results wrap with them)
            const int kstop = min(kend, k + 8192);
            i32x4 acc[NL][WT][WT];
#pragma unroll
            for (int s = 0; s < NL; ++s)
#pragma unroll
                for (int i = 0; i < WT; ++i)
#pragma unroll
                    for (int j = 0; j < WT; ++j) acc[s][i][j] = i32x4{0, 0, 0, 0};
            for (; k < kstop; k += 64 * KS) {
                i32x4 pa[WT][NL], pb[WT][NL];
#pragma unroll
                for (int j = 0; j < WT; ++j) {
                    to_planes<T>(ra[j], pa[j]);
                    to_planes<T>(rb[j], pb[j]);
                }
                if (k + 64 * KS < kend) load(k + 64 * KS);
#pragma unroll
                for (int s = 0; s < NL; ++s)
#pragma unroll
                    for (int l = 0; l <= s; ++l)
#pragma unroll
                        for (int i = 0; i < WT; ++i)
#pragma unroll
                            for (int j = 0; j < WT; ++j)
                                acc[s][i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pb[i][l], pa[j][s - l], acc[s][i][j],
                                                                                     0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WT; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int s = 0; s < NL; ++s) tot[i][j][r] += (A)(int64_t)acc[s][i][j][r] << (8 * s);
        }
        T *Cb = (T *)g.c + bz * g.c_bs;
        auto put = [&](int m, int n, A v) {
            if (m >= g.M || n >= g.N) return;
            if (g.splits > 1)
                ((A *)g.ws)[(((int64_t)ks * g.batch + bz) * g.M + m) * g.N + n] = v;
            else
                store_out<T>(g, Cb + m * g.c_rs + n * g.c_cs, v, bz * g.bias_bs + m * g.bias_rs + n * g.bias_cs);
        };
        if constexpr (KS == 1) {
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WT; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) put(m0 + 16 * j + r16, n0 + 16 * i + 4 * (lane >> 4) + r, tot[i][j][r]);
        } else {
            // part[wave][block][register][lane]; output quantities spread over all threads
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WT; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) part[(((wk * WT + i) * WT + j) * 4 + r) * 64 + lane] = tot[i][j][r];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < WT * WT * 4 / NW; ++q) {
                const int idx = wave + NW * q;   // (block, register)
                A v = 0;
#pragma unroll
                for (int w = 0; w < KS; ++w) v += part[(w * WT * WT * 4 + idx) * 64 + lane];
                const int r = idx & 3, j = (idx >> 2) % WT, i = (idx >> 2) / WT;
                put(m0 + 16 * j + r16, n0 + 16 * i + 4 * (lane >> 4) + r, v);
            }
            __syncthreads();   // LDS reuse by the next batch iteration
        }
    }
}

template <class T, int WT, int WM, int WN, int KS>
hipError_t launch_tile(bool va, bool vb, const GemmArgs &g, dim3 grid, hipStream_t st) {
    const dim3 block(64 * WM * WN * KS);
    if (va && vb) hipLaunchKernelGGL((k_gemm_limb<T, WT, WM, WN, KS, true, true>), grid, block, 0, st, g);
    else if (va) hipLaunchKernelGGL((k_gemm_limb<T, WT, WM, WN, KS, true, false>), grid, block, 0, st, g);
    else if (vb) hipLaunchKernelGGL((k_gemm_limb<T, WT, WM, WN, KS, false, true>), grid, block, 0, st, g);
    else hipLaunchKernelGGL((k_gemm_limb<T, WT, WM, WN, KS, false, false>), grid, block, 0, st, g);
    return hipGetLastError();
}

template <class T> hipError_t launch_typed(int bt, const GemmArgs &g, dim3 grid, hipStream_t st) {
    constexpr int E = 16 / (int)sizeof(T);
    auto vec = [&](const void *p, int64_t ks, int64_t ld, int64_t bs) {
        return ks == 1 && ld % E == 0 && ((uintptr_t)p & 15) == 0 && (g.batch == 1 || bs % E == 0) && g.K % E == 0;
    };
    const bool va = vec(g.a, g.a_cs, g.a_rs, g.a_bs), vb = vec(g.b, g.b_rs, g.b_cs, g.b_bs);
    if (bt == 16) return launch_tile<T, 1, 1, 1, 4>(va, vb, g, grid, st);
    if (bt == 64) return launch_tile<T, 2, 2, 2, 1>(va, vb, g, grid, st);
    if constexpr (sizeof(T) == 8)   // 16 x 16 per wave: a 32 x 32 one takes 400 registers, one wave per SIMD
        return launch_tile<T, 1, 2, 2, 1>(va, vb, g, grid, st);
    else
        return launch_tile<T, 2, 1, 1, 4>(va, vb, g, grid, st);
}

}  // namespace

hipError_t launch_limb(int dt, int bt, const GemmArgs &g, dim3 grid, hipStream_t st) {
    switch (dt) {
        case I8: return launch_typed<int8_t>(bt, g, grid, st);
        case U8: return launch_typed<uint8_t>(bt, g, grid, st);
        case I16: return launch_typed<int16_t>(bt, g, grid, st);
        case I32: return launch_typed<int32_t>(bt, g, grid, st);
        case I64: return launch_typed<int64_t>(bt, g, grid, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace mb
