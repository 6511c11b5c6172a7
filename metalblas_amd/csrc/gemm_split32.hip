// fp32 and complex64 products on the fp16 matrix cores.
//
// An fp32 value scaled by a power of two into fp16's range is the sum of two fp16 numbers: hi, the
// value rounded to 11 bits, and lo, what the rounding left, at most 2^11 units of the value's
// last place and so exact in 11 bits too.  Then a b = hi hi + (hi lo + lo hi) + lo lo, whose
// last term is at most 2^-24 of the product, the rounding of one fp32 multiplication, and is left
// out: three fp16 products with fp32 accumulation, at 16 times the rate of the fp32 matrix
// instructions (2517 against 157 TFLOP/s nominal).  The products of 11-bit numbers are exact in
// fp32, and a sum over K has K / 32 rounded accumulations instead of K, so the result is closer
// to the exact one than that of the fp32 instructions: relative 2-norm error against 64 bits,
// MI355X, N(0,1): 2048^3 fp32 8.1e-7 -> 2.2e-7, 2048^3 complex64 1.1e-6 -> 3.0e-7.
//
// Range.  Each row of A and column of B is scaled by its own power of two (its largest magnitude
// goes to [2^14, 2^15)) and lo is kept 2^11 times larger, with accumulators of its own, so every
// element down to 2^-26 of its row's largest is exact and one at 2^-t of it loses t - 26 bits.
// A product holding an infinity, a NaN, or a nonzero element smaller than K 2^-25 relative
// accuracy allows (the accuracy of a K-term fp32 sum) is left to the fp32 kernels: the split pass
// raises a flag in the workspace, the split product returns at once, and the fp32 plan, queued
// behind it, runs only if the flag is up.
//
// Three launches: the largest magnitude of every row over slices of K, the split into the layout
// the product streams (K-contiguous whatever the operand's layout, 32 hi then 32 lo per 128-byte
// stage row, K zero-padded), and the product on the K ping-pong tile (mfma_kpp.hpp).  Complex
// operands are split as real ones with (re, im) pairs along k; the product makes the two real
// columns of a complex one in registers, so B is neither written nor read as 2 x 2 blocks.
//
// MI355X, us a call: fp32 2048^3 166 -> 83 (magnitudes 14, split 16.5, product 50, guarded fp32
// kernel 4.6), 4096^3 1081 -> 428; complex64 2048^3 584 -> 229 (17 + 31 + 163 + 18, two panels).  The
// product is bound by the board's power limit (0.55-0.69 matrix-core busy at 1.6-1.7 GHz), the
// split by the operands' three passes through the cache.
#include "mfma_kpp.hpp"

namespace mb {

namespace {

// Element (r, k) of the source as NC floats (NC = 2: complex re, im).
template <int NC> struct Vals {
    float v[NC];
};
template <int NC> __device__ __forceinline__ Vals<NC> load_elem(const float *p) {
    Vals<NC> o;
    if constexpr (NC == 2) {
        const float2 f = *(const float2 *)p;
        o.v[0] = f.x;
        o.v[1] = f.y;
    } else {
        o.v[0] = *p;
    }
    return o;
}
// magnitude bits: ordered like the magnitudes, infinities and NaNs above every finite value
__device__ __forceinline__ uint32_t mag(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// Largest magnitude of each row over one K slice: part[bz][slice][row].  16 loads in flight per
// thread: a K-contiguous source takes a wave per row (lanes along K, 4 rows per block), any other
// puts the lanes along 64 rows and the 4 waves along K.
template <int NC> __device__ __forceinline__ void absmax_block(const SplitOperand &o, int blk, int bz0, int nbz, uint32_t *sh) {
    constexpr int U = 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rows_per = o.k_contig ? 4 : 64;
    const int nrb = (o.R + rows_per - 1) / rows_per;
    const int slice = blk / nrb, r0 = (blk - slice * nrb) * rows_per;
    const int kb = slice * o.k_slice, ke = min(o.K, kb + o.k_slice);
    const int r = r0 + (o.k_contig ? wave : lane), kfirst = kb + (o.k_contig ? lane : wave);
    const int kstep = o.k_contig ? 64 : 4;
    for (int bz = bz0; bz < o.batch; bz += nbz) {
        uint32_t *part = o.part + ((int64_t)bz * o.slices + slice) * o.part_ld;
        uint32_t m = 0;
        if (r < o.R) {
            const float *p = (const float *)o.src + (bz * o.bs + r * o.rs) * NC;
            for (int k = kfirst; k < ke; k += U * kstep) {
                Vals<NC> e[U];
#pragma unroll
                for (int i = 0; i < U; ++i) {
                    e[i] = {};
                    if (k + i * kstep < ke) e[i] = load_elem<NC>(p + (k + i * kstep) * o.ks * NC);
                }
#pragma unroll
                for (int i = 0; i < U; ++i)
#pragma unroll
                    for (int c = 0; c < NC; ++c) m = max(m, mag(e[i].v[c]));
            }
        }
        if (o.k_contig) {
#pragma unroll
            for (int s = 32; s > 0; s >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, s, 64));
            if (lane == 0 && r < o.R) part[r] = m;
        } else {
            sh[wave * 64 + lane] = m;
            __syncthreads();
            if (wave == 0 && r < o.R) part[r] = max(max(sh[lane], sh[64 + lane]), max(sh[128 + lane], sh[192 + lane]));
            __syncthreads();
        }
    }
}

__global__ __launch_bounds__(256) void k_split_absmax(SplitOperand a, SplitOperand b, int nblk_a, int32_t *flag) {
    __shared__ uint32_t sh[256];
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *flag = 0;
    const bool is_a = (int)blockIdx.x < nblk_a;
    const SplitOperand &o = is_a ? a : b;
    const int blk = is_a ? blockIdx.x : blockIdx.x - nblk_a;
    if (o.cplx)
        absmax_block<2>(o, blk, blockIdx.y, gridDim.y, sh);
    else
        absmax_block<1>(o, blk, blockIdx.y, gridDim.y, sh);
}

// binary exponent of a magnitude (0 for a zero row: its elements are all zero)
__device__ __forceinline__ int mag_exp(uint32_t m) { return m < 0x00800000u ? (m ? -126 : 0) : (int)(m >> 23) - 127; }

// 64 rows x 64 real k of one operand: read along whichever dimension is contiguous, turned
// through LDS, written as 16-byte chunks of 8 hi / 8 lo.  The element loads go out first, the
// rows' magnitude partials behind them.
template <int NC> __device__ __forceinline__ void split_block(const SplitOperand &o, int blk, int bz0, int nbz, float *s,
                                                                uint32_t *smax, int *sexp, int32_t *flag) {
    constexpr int KT = 64 / NC, P = 65;   // P: LDS row pitch in floats
    constexpr int NE = 64 * KT / 256;                        // elements per thread
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nrb = (o.R + 63) / 64;
    const int kt = blk / nrb, r0 = (blk - kt * nrb) * 64, k0 = kt * KT;
    // element i of this thread: (r + i * rstep, k + i * kstep)
    const int r = o.k_contig ? tid / KT : lane, rstep = o.k_contig ? 256 / KT : 0;
    const int k = o.k_contig ? tid % KT : wave, kstep = o.k_contig ? 0 : 4;
    bool bad = false;
    for (int bz = bz0; bz < o.batch; bz += nbz) {
        const float *src = (const float *)o.src + bz * o.bs * NC;
        Vals<NC> e[NE];
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const int gr = r0 + r + i * rstep, gk = k0 + k + i * kstep;
            e[i] = {};
            if (gr < o.R && gk < o.K) e[i] = load_elem<NC>(src + (gr * o.rs + gk * o.ks) * NC);
        }
        // magnitudes: wave w takes every 4th partial (at most 32) of the 64 rows
        uint32_t m = 0;
        if (r0 + lane < o.R) {
            const uint32_t *part = o.part + (int64_t)bz * o.slices * o.part_ld + r0 + lane;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (wave + 4 * i < o.slices) m = max(m, part[(int64_t)(wave + 4 * i) * o.part_ld]);
        }
        smax[tid] = m;
#pragma unroll
        for (int i = 0; i < NE; ++i)
#pragma unroll
            for (int c = 0; c < NC; ++c) s[(r + i * rstep) * P + (k + i * kstep) * NC + c] = e[i].v[c];
        __syncthreads();
        if (tid < 64) {
            const uint32_t mm = max(max(smax[tid], smax[64 + tid]), max(smax[128 + tid], smax[192 + tid]));
            bad |= mm >= 0x7f800000u;
            const int ex = mag_exp(mm);
            sexp[tid] = 14 - ex;
            if (kt == 0 && r0 + tid < o.R) o.exps[(int64_t)bz * o.R + r0 + tid] = ex - 14;
        }
        __syncthreads();
        _Float16 *dst = (_Float16 *)o.dst + bz * o.d_bs;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int item = tid + 256 * it;
            const int tr = item >> 3, ch = item & 7;   // row of the tile, chunk of 8 k
            const int kc = kt * 64 + ch * 8;           // real k of the chunk
            if (r0 + tr >= o.R || kc >= o.Kp) continue;
            const int sc = sexp[tr];
            _Float16 hi[8], lo[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float x = ldexpf(s[tr * P + ch * 8 + i], sc);
                bad |= x != 0.f && fabsf(x) < o.min_x;
                const _Float16 h = (_Float16)x;
                hi[i] = h;
                lo[i] = (_Float16)((x - (float)h) * 2048.f);
            }
            _Float16 *q = dst + (int64_t)(r0 + tr) * o.ld + (kc >> 5) * 64 + (kc & 31);
            uint4 u;
            __builtin_memcpy(&u, hi, 16);
            *(uint4 *)q = u;
            __builtin_memcpy(&u, lo, 16);
            *(uint4 *)(q + 32) = u;
        }
        __syncthreads();
    }
    if (bad) *flag = 1;
}

__global__ __launch_bounds__(256) void k_split32(SplitOperand a, SplitOperand b, int nblk_a, int32_t *flag) {
    __shared__ float s[64 * 65];
    __shared__ uint32_t smax[256];
    __shared__ int sexp[64];
    const bool is_a = (int)blockIdx.x < nblk_a;
    const SplitOperand &o = is_a ? a : b;
    const int blk = is_a ? blockIdx.x : blockIdx.x - nblk_a;
    if (o.cplx)
        split_block<2>(o, blk, blockIdx.y, gridDim.y, s, smax, sexp, flag);
    else
        split_block<1>(o, blk, blockIdx.y, gridDim.y, s, smax, sexp, flag);
}

// The product of the split operands: g.a / g.b are the split planes (g.a_rs / g.b_cs their row
// length, g.K their padded length, in halves); M, N and the output and bias strides are those of
// the caller's product, in complex elements for complex64.
template <bool CPLX>
__global__ __launch_bounds__(512) void k_gemm_split32(GemmArgs g, SplitExps x) {
    using K = m16::Kpp<f16_t, true, true, false, CPLX ? m16::kSplitComplex : m16::kSplitReal>;
    using T = std::conditional_t<CPLX, c64_t, float>;
    using A = typename Tr<T>::acc;
    constexpr int BN = CPLX ? K::BN / 2 : K::BN, NB = CPLX ? 1 : 2;   // columns per tile, blocks per wave
    __shared__ __attribute__((aligned(1024))) char smem[K::SMEM];
    if (*x.flag) return;   // left to the fp32 kernels
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_m = cdiv(g.M, K::BM), tiles_n = cdiv(g.N, BN);
    int tm, tn, ks, bz0;
    work_coords(tiles_m, tiles_n, g.swz, g.xcd_batch, tm, tn, ks, bz0);
    const int m0 = tm * K::BM, n0 = tn * BN;
    const int kbeg = ks * g.k_chunk;
    const int klen = min(g.K, kbeg + g.k_chunk) - kbeg;
    // column (re, -im) of conj(A) conj(B): the sign of im is -sa sb; column (im, re): (sb im, sa re)
    const uint32_t sign_re = g.conj_a == g.conj_b ? 0x80000000u : 0u;
    const uint32_t sign_im = (g.conj_b ? 0x8000u : 0u) | (g.conj_a ? 0x80000000u : 0u);
    for (int bz = bz0; bz < g.batch; bz += gridDim.z) {
        const f16_t *Ab = (const f16_t *)g.a + bz * g.a_bs + (int64_t)m0 * g.a_rs + kbeg;
        const f16_t *Bb = (const f16_t *)g.b + bz * g.b_bs + (int64_t)n0 * g.b_cs + kbeg;
        typename K::Acc out[2][K::TM];
        K::run(Ab, Bb, g.a_rs, g.b_cs, g.M - m0, g.N - n0, klen, smem, wave, lane, out, sign_re, sign_im);
        int mw = m0 + (wave & 1) * 64;
        int nw = n0 + ((wave >> 1) & 1) * (BN / 2) + (wave >> 2) * (BN / 4);
        asm volatile("" : "+s"(mw), "+s"(nw));   // store addressing stays below the main loop
        const int32_t *ea = x.ea + bz * x.ea_bs, *eb = x.eb + bz * x.eb_bs;
        T *Cb = (T *)g.c + bz * g.c_bs;
        A *ws = (A *)g.ws + ((int64_t)ks * g.batch + bz) * g.M * (int64_t)g.N;
#pragma unroll
        for (int j = 0; j < K::TM; ++j) {
            const int gm = mw + 16 * j + (lane & 15);
            if (gm >= g.M) continue;
            const int em = ea[gm];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int gn = nw + 16 * i + 4 * (lane >> 4);
                A v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int e = gn + r < g.N ? em + eb[gn + r] : 0;
                    if constexpr (CPLX) v[r] = A{ldexpf(out[0][j][r], e), ldexpf(out[1][j][r], e)};
                    else v[r] = ldexpf(out[i][j][r], e);
                }
                const bool planes = g.splits > 1;
                // 4 consecutive outputs as 16-byte stores (which need only 4-byte alignment)
                if (gn + 3 < g.N && (planes || (g.c_cs == 1 && !g.epilogue))) {
                    typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
                    A *dst = planes ? ws + (int64_t)gm * g.N + gn : (A *)(Cb + gm * g.c_rs + gn);
                    f4 u[sizeof(v) / 16];
                    __builtin_memcpy(u, v, sizeof(v));
#pragma unroll
                    for (int q = 0; q < (int)sizeof(v) / 16; ++q) ((f4 *)dst)[q] = u[q];
                    continue;
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = gn + r;
                    if (n >= g.N) continue;
                    if (planes) ws[(int64_t)gm * g.N + n] = v[r];
                    else store_out<T>(g, Cb + gm * g.c_rs + n * g.c_cs, v[r], bz * g.bias_bs + gm * g.bias_rs + n * g.bias_cs);
                }
            }
        }
        __syncthreads();   // LDS reuse by the next batch iteration
    }
}

}  // namespace

// a grid of two operands' blocks (b may have none)
static dim3 split_grid(const SplitOperand &a, int na, const SplitOperand &b, int nb) {
    const int batch = a.batch > b.batch ? a.batch : b.batch;
    return dim3(na + nb, batch < 65535 ? batch : 65535);
}

hipError_t launch_split_absmax(const SplitOperand &a, const SplitOperand &b, int32_t *flag, hipStream_t st) {
    auto blocks = [](const SplitOperand &o) { return cdiv(o.R, o.k_contig ? 4 : 64) * o.slices; };
    const int na = blocks(a), nb = blocks(b);
    hipLaunchKernelGGL(k_split_absmax, split_grid(a, na, b, nb), dim3(256), 0, st, a, b, na, flag);
    return hipGetLastError();
}

hipError_t launch_split32(const SplitOperand &a, const SplitOperand &b, int32_t *flag, hipStream_t st) {
    auto blocks = [](const SplitOperand &o) { return cdiv(o.R, 64) * cdiv(o.Kp, 64); };
    const int na = blocks(a), nb = blocks(b);
    hipLaunchKernelGGL(k_split32, split_grid(a, na, b, nb), dim3(256), 0, st, a, b, na, flag);
    return hipGetLastError();
}

hipError_t launch_gemm_split32(bool cplx, const GemmArgs &g, const SplitExps &x, hipStream_t st) {
    const dim3 grid(cdiv(g.M, 128) * cdiv(g.N, cplx ? 64 : 128), g.splits, g.batch < 65535 ? g.batch : 65535);
    if (cplx)
        hipLaunchKernelGGL(k_gemm_split32<true>, grid, dim3(512), 0, st, g, x);
    else
        hipLaunchKernelGGL(k_gemm_split32<false>, grid, dim3(512), 0, st, g, x);
    return hipGetLastError();
}

}  // namespace mb
