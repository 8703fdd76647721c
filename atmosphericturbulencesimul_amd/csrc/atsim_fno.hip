// atsim_fno.hip -- kernels of the Fourier-neural-operator surrogate of the
// Fresnel layer loop (no counterpart in the reference).
//
// Every linear map of the network -- the truncated DFTs along x and y, the
// per-mode complex channel mixing, the 1x1 channel maps -- and every product
// of its backward pass is a matrix product on the matrix cores with BF16
// operands and FP32 sums.  At the sizes the network is used at, passes of their
// own make them: k_pointwise and k_tail (channel maps with the inverse x
// transform, bias, activation, and the next forward x transform), k_dft2 /
// k_dft_y, k_mix and k_idft_y (spectral path), k_mix_grad and k_weight_grad.
// Other sizes and alignments take k_gemm_bf16, a strided, batched GEMM
//     C[b] = alpha * A[b] (M x K) * B[b] (K x N) + beta * C[b]
// with arbitrary element strides, so transposes, real/imaginary views and
// channel-major / mode-major layouts cost nothing.  Operands are FP32 in
// memory and rounded to BF16 (round to nearest even) when staged into LDS;
// the products run on v_mfma_f32_16x16x32_bf16 with FP32 accumulation.
//
// Tile: 64 x 64 outputs per 256-thread workgroup (4 waves in 2 x 2, each a
// 32 x 32 block of 2 x 2 MFMA 16x16 tiles), K step 64 (two MFMA k-steps per
// staging).  The epilogue can add a per-row bias, keep the pre-activation and
// apply GELU, so a 1x1 channel map, its bias and its activation are one pass.  MFMA 16x16x32 bf16
// operand layout (one wave): lane l holds A[l % 16][8 (l / 16) .. +7] and
// B[8 (l / 16) .. +7][l % 16]; the accumulator holds D[4 (l / 16) .. +3][l % 16].
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "atsim_kernels.hpp"
#include "atsim_launch.hpp"

namespace atsim {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __bf16 to_bf16(float x) {
    // round to nearest even on the bit pattern (finite inputs)
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    const uint16_t h = (uint16_t)(u >> 16);
    return __builtin_bit_cast(__bf16, h);
}

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// GELU, tanh form: 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))
__device__ __forceinline__ float gelu_t(float x, float* dgelu) {
    const float k0 = 0.7978845608028654f, k1 = 0.044715f;
    const float u = k0 * fmaf(k1 * x * x, x, x);
    const float t = tanhf(u);
    if (dgelu) *dgelu = 0.5f * (1.f + t) + 0.5f * x * (1.f - t * t) * k0 * fmaf(3.f * k1, x * x, 1.f);
    return 0.5f * x * (1.f + t);
}

// Stage an RT (rows) x BK (k) tile of an operand into T[row][k] as BF16.
// mode 1: unit stride along k (float4 loads along k); mode 2: unit stride
// along the rows (float4 loads along rows); 0: scalar loads, consecutive
// threads along k.  Vector modes are chosen on the host only when the
// extents and strides are multiples of 4 and the base is 16-byte aligned.
template <int RT, int BK>
__device__ __forceinline__ void stage_tile(__bf16 (*T)[BK + 8], const float* __restrict__ X, long r0, long R,
                                           long srow, long k0, long K, long sk, int mode, int tid) {
    static_assert((RT * BK) % 1024 == 0, "tile must split into float4 per thread");
    if (mode == 1) {
#pragma unroll
        for (int e = 0; e < RT * BK / 4 / 256; e++) {
            const int idx = tid + e * 256;
            const int r = idx / (BK / 4), kq = (idx % (BK / 4)) * 4;
            const long gr = r0 + r, gk = k0 + kq;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (gr < R && gk < K) v = *reinterpret_cast<const float4*>(X + gr * srow + gk);
            bf16x4 h = {to_bf16(v.x), to_bf16(v.y), to_bf16(v.z), to_bf16(v.w)};
            *reinterpret_cast<bf16x4*>(&T[r][kq]) = h;
        }
    } else if (mode == 2) {
#pragma unroll
        for (int e = 0; e < RT * BK / 4 / 256; e++) {
            const int idx = tid + e * 256;
            const int kk = idx / (RT / 4), rq = (idx % (RT / 4)) * 4;
            const long gr = r0 + rq, gk = k0 + kk;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (gr < R && gk < K) v = *reinterpret_cast<const float4*>(X + gr + gk * sk);
            T[rq + 0][kk] = to_bf16(v.x);
            T[rq + 1][kk] = to_bf16(v.y);
            T[rq + 2][kk] = to_bf16(v.z);
            T[rq + 3][kk] = to_bf16(v.w);
        }
    } else {
#pragma unroll
        for (int e = 0; e < RT * BK / 256; e++) {
            const int idx = tid + e * 256;
            const int r = idx / BK, kk = idx % BK;
            const long gr = r0 + r, gk = k0 + kk;
            T[r][kk] = to_bf16((gr < R && gk < K) ? X[gr * srow + gk * sk] : 0.f);
        }
    }
}

// BM x BN outputs per 256-thread workgroup; the 4 waves form WM x (4 / WM)
// and each holds (BM / WM) x (BN / (4 / WM)) outputs as TI x TJ MFMA 16x16
// tiles.  Shapes: 64 x 64 (general), 32 x 256 (few rows: 1x1 channel maps),
// 256 x 32 (few columns: DFTs onto the retained modes).
template <int BM, int BN, int BK, int WM>
__global__ void __launch_bounds__(256) k_gemm_bf16(GemmArgs g) {
    constexpr int WN = 4 / WM, WTM = BM / WM, WTN = BN / WN, TI = WTM / 16, TJ = WTN / 16;
    __shared__ __bf16 As[BM][BK + 8];
    __shared__ __bf16 Bs[BN][BK + 8];
    const long b = blockIdx.z;
    const long m0 = (long)blockIdx.y * BM, n0 = (long)blockIdx.x * BN;
    const float* A = g.A + b * g.sab;
    const float* B = g.B + b * g.sbb;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / WN) * WTM, wn = (wave % WN) * WTN;
    f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (long k0 = 0; k0 < g.K; k0 += BK) {
        stage_tile<BM, BK>(As, A, m0, g.M, g.sam, k0, g.K, g.sak, g.avec, tid);
        stage_tile<BN, BK>(Bs, B, n0, g.N, g.sbn, k0, g.K, g.sbk, g.bvec, tid);
        __syncthreads();
        const int row = lane & 15, kq = (lane >> 4) * 8;
#pragma unroll
        for (int ks = 0; ks < BK; ks += 32) {
            bf16x8 bv[TJ];
#pragma unroll
            for (int j = 0; j < TJ; j++) bv[j] = *reinterpret_cast<const bf16x8*>(&Bs[wn + j * 16 + row][ks + kq]);
#pragma unroll
            for (int i = 0; i < TI; i++) {
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(&As[wm + i * 16 + row][ks + kq]);
#pragma unroll
                for (int j = 0; j < TJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bv[j], acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // epilogue: v = alpha AB + beta C + bias[m]; pre = v; C = act(v)
    float* C = g.C + b * g.scb;
    float* Pre = g.pre ? g.pre + b * g.scb : nullptr;
    const int col = lane & 15, rq = (lane >> 4) * 4;
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const long gm = m0 + wm + i * 16 + rq + q, gn = n0 + wn + j * 16 + col;
                if (gm < g.M && gn < g.N) {
                    const long o = gm * g.scm + gn * g.scn;
                    float v = g.alpha * acc[i][j][q];
                    if (g.beta != 0.f) v = fmaf(g.beta, C[o], v);
                    if (g.bias) v += g.bias[gm];
                    if (Pre) Pre[o] = v;
                    C[o] = g.act ? gelu_t(v, nullptr) : v;
                }
            }
}

// vector staging mode of an operand (see stage_tile)
static int vec_mode(const float* X, long rows, long srow, long K, long sk, long sbatch) {
    const bool aligned = ((uintptr_t)X & 15) == 0 && (sbatch & 3) == 0;
    if (aligned && sk == 1 && (K & 3) == 0 && (srow & 3) == 0) return 1;
    if (aligned && srow == 1 && (rows & 3) == 0 && (sk & 3) == 0) return 2;
    return 0;
}

template <int BM, int BN, int BK, int WM>
static hipError_t gemm_launch(const GemmArgs& g, hipStream_t st) {
    const long gy = (g.M + BM - 1) / BM, gx = (g.N + BN - 1) / BN;
    if (gy > 65535 || g.batch > 65535 || gx > 0x7FFFFFFFL) return hipErrorInvalidValue;
    dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)g.batch);
    k_gemm_bf16<BM, BN, BK, WM><<<grid, 256, 0, st>>>(g);
    return hipGetLastError();
}

hipError_t launch_gemm_bf16(const GemmArgs& g0, hipStream_t st) {
    if (g0.M <= 0 || g0.N <= 0 || g0.batch <= 0) return hipSuccess;
    GemmArgs g = g0;
    g.avec = vec_mode(g.A, g.M, g.sam, g.K, g.sak, g.sab);
    g.bvec = vec_mode(g.B, g.N, g.sbn, g.K, g.sbk, g.sbb);
    const bool k32 = g.K <= 32;
    if (g.M <= 32 && g.N > 64)
        return k32 ? gemm_launch<32, 256, 32, 1>(g, st) : gemm_launch<32, 256, 64, 1>(g, st);
    if (g.N <= 32 && g.M > 64)
        return k32 ? gemm_launch<256, 32, 32, 4>(g, st) : gemm_launch<256, 32, 64, 4>(g, st);
    return k32 ? gemm_launch<64, 64, 32, 2>(g, st) : gemm_launch<64, 64, 64, 2>(g, st);
}

// ------------------------------------------------------------------ channel maps
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// float pairs to BF16, round to nearest even (v_cvt_pk_bf16_f32; the values
// of to_bf16)
__device__ __forceinline__ bf16x8 to_bf16x8(const float (&x)[8]) {
    bf16x8 h;
#pragma unroll
    for (int j = 0; j < 8; j++) h[j] = (__bf16)x[j];
    return h;
}

// out[c][p] = act( sum_i W[c][i] h[i][p]  (+ sum_k U[c][row(p)][k] F[k][x(p)])  (+ bias[c]) )
// over channel-major images [C][nrows][rowlen]: a 1x1 channel map with, in the
// same pass, the spectral path's inverse transform along x (U: the rows'
// retained spectrum, F: the transform's table).  act 0: none, 1: GELU (pre,
// if given, keeps its argument), 2: times GELU'(pre).
//
// Bound: HBM (h read and out written once, U and pre when given).  A wave
// takes 64 pixels: lane l loads float4s of 8 channels at pixels
// 4 (l % 16) .. + 3, so that pixel t of every lane's four is one MFMA column
// and the operand is made in registers, without LDS; the four tiles' outputs
// of a lane are again four neighbouring pixels, stored as float4.  The
// products of one output are summed by the MFMAs in k_gemm_bf16's order (k
// steps of 32, zero padded), the two sums added last: the same results as
// its passes.
// A block's map at 32 channels, 50 images of 256^2 (839 MB + 52 MB of U):
// 194 us, 4.6 TB/s, where the inverse x transform and the map with its bias and
// GELU took 340 + 1 016 us as two k_gemm_bf16 passes (staging through LDS in
// 2-byte stores, the image written, read and written again).
struct PointArgs {
    const float* W;
    long swm, swk;
    int Cout, Cin;
    const float* h;
    float* out;
    long nrows;
    int rowlen;
    const float* U;  // [Cout][nrows][K2], or null
    int K2;
    const float* F;
    long sfk, sfx;
    const float* bias;
    float* pre;
    int act;
    const float* D;  // table of the transform of out along x (NT > 0): D[x dsk + c dsn], dm modes
    long dsk, dsn;
    int dm;
    __bf16* T;       // its result [Cout][nrows][16 NT]; out may then be null
    const float *L, *Lb;  // h = L x + Lb ([Cin][cl], x in h's place)
    int cl;
};

// F [K2][rowlen] staged as MFMA operands [KU][64-pixel group][t][lane][8]
template <int KU>
__device__ __forceinline__ void stage_xtable(__bf16* Fs, const float* __restrict__ F, long sfk, long sfx, int K2,
                                             int rowlen) {
    const int ngrp = (rowlen + 63) / 64;
    for (int e = threadIdx.x; e < KU * ngrp * 256; e += 256) {
        const int ln = e & 63, t = (e >> 6) & 3, kg = e >> 8;
        const int x = (kg % ngrp) * 64 + 4 * (ln & 15) + t, k = (kg / ngrp) * 32 + (ln >> 4) * 8;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            v[j] = F[min(k + j, K2 - 1) * sfk + min(x, rowlen - 1) * sfx];
            if (k + j >= K2) v[j] = 0.f;
        }
        *reinterpret_cast<bf16x8*>(Fs + (size_t)e * 8) = to_bf16x8(v);
    }
}
// F [x][n] (x sfk + n sfn) staged as MFMA operands [k step][NT][lane][8] by TH threads
template <int NT>
__device__ __forceinline__ void stage_dtable(__bf16* Ds, const float* __restrict__ F, long sfk, long sfn, int N, int M2,
                                             int TH) {
    for (int e = threadIdx.x; e < N / 32 * NT * 64; e += TH) {
        const int ln = e & 63, t = e >> 6, nt = t % NT, ks = t / NT;
        const float* p = F + min(nt * 16 + (ln & 15), M2 - 1) * sfn + (long)(ks * 32 + (ln >> 4) * 8) * sfk;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = p[j * sfk];
        *reinterpret_cast<bf16x8*>(Ds + (size_t)e * 8) = to_bf16x8(v);
    }
}
// orders a wave's own LDS writes before its reads
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// The matrix row that row i of an MFMA row tile rt stands for.  CHAIN: pairs of
// tiles hold 32 rows in the order in which a lane's results of both tiles are
// the 8 values of the next product's operand (4 (l / 16) + q of tile 0 and 1 ->
// 8 (l / 16) + 0 .. 7), so that products follow one another in registers.
template <bool CHAIN>
__device__ __forceinline__ int tile_row(int rt, int i) {
    return CHAIN ? 32 * (rt >> 1) + 8 * (i >> 2) + 4 * (rt & 1) + (i & 3) : rt * 16 + i;
}
// a wave's operands of an M x K matrix (element strides sm, sk)
template <int RT, int KT, bool CHAIN = false>
__device__ __forceinline__ void matrix_operands(bf16x8 (&wa)[RT][KT], const float* __restrict__ W, long sm, long sk,
                                                int M, int K, int lm, int lk) {
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                v[j] = W[min(tile_row<CHAIN>(rt, lm), M - 1) * sm + min(kt * 32 + lk + j, K - 1) * sk];
                if (kt * 32 + lk + j >= K) v[j] = 0.f;
            }
            wa[rt][kt] = to_bf16x8(v);
        }
}
// the spectrum operands of row r of every channel
template <int RT, int KU, bool CHAIN = false>
__device__ __forceinline__ void spectrum_operands(bf16x8 (&ua)[RT][KU], const float* __restrict__ U, long nrows,
                                                  long r, int C, int K2, int lm, int lk) {
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int ku = 0; ku < KU; ku++) {
            const int k = ku * 32 + lk;
            const float* up = U + ((long)min(tile_row<CHAIN>(rt, lm), C - 1) * nrows + r) * K2;
            const float4 a = *reinterpret_cast<const float4*>(up + min(k, K2 - 4));
            const float4 b = *reinterpret_cast<const float4*>(up + min(k + 4, K2 - 4));
            float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (k + j >= K2) v[j] = 0.f;
            ua[rt][ku] = to_bf16x8(v);
        }
}
// the operands of pixel t of a lane's four, from its 8 KT loaded channels
template <int KT>
__device__ __forceinline__ void pixel_operands(bf16x8 (&hb)[KT], const float4 (&hv)[KT][8], int t, int C, int lk) {
#pragma unroll
    for (int kt = 0; kt < KT; kt++) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            v[j] = t == 0 ? hv[kt][j].x : t == 1 ? hv[kt][j].y : t == 2 ? hv[kt][j].z : hv[kt][j].w;
            if (kt * 32 + lk + j >= C) v[j] = 0.f;
        }
        hb[kt] = to_bf16x8(v);
    }
}
// every load unconditional, at a clamped channel and pixel: a load under a
// lane's own condition is waited for before the next one
template <int KT>
__device__ __forceinline__ void load_channels(float4 (&hv)[KT][8], const float* __restrict__ h, long SP, long p,
                                              int C, int lk) {
#pragma unroll
    for (int kt = 0; kt < KT; kt++)
#pragma unroll
        for (int j = 0; j < 8; j++)
            hv[kt][j] = *reinterpret_cast<const float4*>(h + min(kt * 32 + lk + j, C - 1) * SP + p);
}

// waves a SIMD that the registers allow without scratch
constexpr int point_waves(int RT, int KT, int KU) {
    return KT == 1 ? (KU == 0 || RT <= 2 ? 3 : 2) : RT == 4 && KU == 2 ? 1 : 2;
}
// NT > 0: with the transform of out along x that the next spectral path begins
// with (k_dft2's first product, 16 NT columns), so that out is not read again
// for it.  A wave takes whole rows then; 64 pixels of all channels pass through
// its own LDS rows as the BF16 operand of k steps of 32 in k_dft2's order, and
// T keeps what k_dft2 keeps in LDS: the same results.  50 images of 256^2, 32
// channels, 16 modes: 232 us + 19 us for k_dft_y, where the map alone takes 190
// and k_dft2 114 (8 images: 60 + 8 us against 55 + 24).  Bound: VALU (tanhf) and
// HBM about equally; channel tiles one after the other, 16 of them live at a time,
// leave room for 3 waves a SIMD (all tiles at once: 2 waves, 264 us; the
// next pixels loaded ahead: scratch, 254 us).
//
// LIFT: the map's input is itself a channel map of x (at most 32 channels), made
// in registers as the operand (tile_row's order) where the pass that would write
// it only leaves its transform (out null): inference needs the first image of
// a network nowhere else.  The same frames from 14 channels: 69 + 219 us, where
// the lift and the first map took 138 + 231.
template <int RT, int KT, int KU, int NT, bool LIFT>
__global__ void __launch_bounds__(256, point_waves(RT, KT, KU)) k_pointwise(PointArgs g) {
    static_assert(!LIFT || KT == 1, "one step of lifted channels");
    extern __shared__ __attribute__((aligned(16))) __bf16 Fs[];  // F as MFMA operands: [KU][64-pixel group][4][lane][8]
    constexpr int XS = 64 + 8;
    __bf16* Ds = Fs + (size_t)KU * ((g.rowlen + 63) / 64) * 2048;                       // [k step][NT][lane][8]
    __bf16* Xs = Ds + (size_t)(g.rowlen / 32) * NT * 512 + (threadIdx.x >> 6) * RT * 16 * XS;  // [channel][XS]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lm = lane & 15, lk = (lane >> 4) * 8;
    const long SP = g.nrows * g.rowlen;
    const int ngrp = (g.rowlen + 63) / 64;
    if constexpr (KU > 0) {
        stage_xtable<KU>(Fs, g.F, g.sfk, g.sfx, g.K2, g.rowlen);
    }
    if constexpr (NT > 0) stage_dtable<NT>(Ds, g.D, g.dsk, g.dsn, g.rowlen, 2 * g.dm, 256);
    if constexpr (KU > 0 || NT > 0) __syncthreads();
    bf16x8 wa[RT][KT];
    matrix_operands<RT, KT>(wa, g.W, g.swm, g.swk, g.Cout, g.Cin, lm, lk);
    float bias[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int q = 0; q < 4; q++)
            bias[rt][q] = g.bias ? g.bias[min(rt * 16 + (lane >> 4) * 4 + q, g.Cout - 1)] : 0.f;
    bf16x8 la[2][1];
    float lb[8];
    if constexpr (LIFT) {
        matrix_operands<2, 1, true>(la, g.L, g.cl, 1, g.Cin, g.cl, lm, lk);
#pragma unroll
        for (int j = 0; j < 8; j++) lb[j] = g.Lb[min(lk + j, g.Cin - 1)];
    }
    f32x4 tx[RT][NT > 0 ? NT : 1];  // the row's transform: columns 4 (l / 16) .. + 3, channel l % 16
    bf16x8 ua[RT][KU > 0 ? KU : 1];
    const long units = NT > 0 ? g.nrows : g.nrows * ngrp, stride = (long)gridDim.x * 4;
    long u = (long)blockIdx.x * 4 + wave;
    if (u >= units) return;
    auto row_of = [&](long v) { return NT > 0 ? v : v / ngrp; };
    auto x_of = [&](long v, int gr) { return NT > 0 ? gr * 64 : (int)(v - v / ngrp * ngrp) * 64; };
    for (int grp = 0;;) {
        const long r = row_of(u);
        const int x0 = x_of(u, grp);
        const bool in = x0 + 4 * lm < g.rowlen;
        const long p = r * g.rowlen + min(x0 + 4 * lm, g.rowlen - 4);
        float4 hv[KT][8];
        load_channels<KT>(hv, g.h, SP, p, LIFT ? g.cl : g.Cin, lk);
        bf16x8 hb[4][KT];
#pragma unroll
        for (int t = 0; t < 4; t++) pixel_operands<KT>(hb[t], hv, t, LIFT ? g.cl : g.Cin, lk);
        if constexpr (LIFT) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                    const f32x4 a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(la[i][0], hb[t][0], z, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        v[4 * i + q] = a[q] + lb[4 * i + q];
                        if (lk + 4 * i + q >= g.Cin) v[4 * i + q] = 0.f;
                    }
                }
                hb[t][0] = to_bf16x8(v);
            }
        }
        if (NT == 0 || grp == 0) {
            if constexpr (KU > 0) spectrum_operands<RT, KU>(ua, g.U, g.nrows, r, g.Cout, g.K2, lm, lk);
#pragma unroll
            for (int i = 0; i < RT * NT; i++) tx[i / (NT > 0 ? NT : 1)][i % (NT > 0 ? NT : 1)] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const bool last = NT == 0 || grp == ngrp - 1;
        const long un = last ? u + stride : u;
        const int gn = last ? 0 : grp + 1;
        if constexpr (NT > 0) wave_fence();  // the operands of the group before are read
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const int c0 = rt * 16 + (lane >> 4) * 4;
            f32x4 res[4];  // [pixel t]: channels c0 .. + 3
#pragma unroll
            for (int t = 0; t < 4; t++) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[rt][kt], hb[t][kt], acc, 0, 0, 0);
                if constexpr (KU > 0) {
                    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ku = 0; ku < KU; ku++)
                        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            ua[rt][ku],
                            *reinterpret_cast<const bf16x8*>(Fs + ((size_t)((ku * ngrp + (x0 >> 6)) * 4 + t) * 64 + lane) * 8),
                            s, 0, 0, 0);
                    acc += s;
                }
                res[t] = acc;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int c = c0 + q;
                if (c >= g.Cout || !in) continue;
                const long o = c * SP + p;
                const float b = bias[rt][q];
                float4 v;
                v.x = res[0][q];
                v.y = res[1][q];
                v.z = res[2][q];
                v.w = res[3][q];
                if (g.bias) {  // (the sum of a null bias could turn -0 into 0)
                    v.x += b;
                    v.y += b;
                    v.z += b;
                    v.w += b;
                }
                if (g.act == 1) {
                    if (g.pre) *reinterpret_cast<float4*>(g.pre + o) = v;
                    v.x = gelu_t(v.x, nullptr);
                    v.y = gelu_t(v.y, nullptr);
                    v.z = gelu_t(v.z, nullptr);
                    v.w = gelu_t(v.w, nullptr);
                } else if (g.act == 2) {
                    const float4 z = *reinterpret_cast<const float4*>(g.pre + o);
                    float d;
                    gelu_t(z.x, &d);
                    v.x *= d;
                    gelu_t(z.y, &d);
                    v.y *= d;
                    gelu_t(z.z, &d);
                    v.z *= d;
                    gelu_t(z.w, &d);
                    v.w *= d;
                } else if (g.pre) {
                    *reinterpret_cast<float4*>(g.pre + o) = v;
                }
                if (NT == 0 || g.out) *reinterpret_cast<float4*>(g.out + o) = v;
                if constexpr (NT > 0) {
                    const bf16x4 t = {(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
                    *reinterpret_cast<bf16x4*>(Xs + c * XS + 4 * lm) = t;
                }
            }
        }
        if constexpr (NT > 0) {
            wave_fence();
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                if (x0 + ks * 32 >= g.rowlen) break;
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const bf16x8 d = *reinterpret_cast<const bf16x8*>(Ds + ((size_t)((x0 / 32 + ks) * NT + nt) * 64 + lane) * 8);
#pragma unroll
                    for (int rt = 0; rt < RT; rt++)
                        tx[rt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            d, *reinterpret_cast<const bf16x8*>(Xs + (rt * 16 + lm) * XS + ks * 32 + lk), tx[rt][nt], 0, 0, 0);
                }
            }
            if (last)
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) {
                        const f32x4 a = tx[rt][nt];
                        const bf16x4 t = {(__bf16)a[0], (__bf16)a[1], (__bf16)a[2], (__bf16)a[3]};
                        if (rt * 16 + lm < g.Cout)
                            *reinterpret_cast<bf16x4*>(g.T + ((rt * 16 + lm) * g.nrows + r) * (NT * 16) + nt * 16 +
                                                       (lane >> 4) * 4) = t;
                    }
        }
        if (un >= units) break;
        u = un;
        grp = gn;
    }
}

// Workgroups of a launch whose waves walk their units: as many as can be
// resident (each stages the tables once), each with the same number of turns.
static unsigned turns_grid(long wg, long resident) {
    const long turns = (wg + resident - 1) / resident;
    return (unsigned)(turns > 0 ? (wg + turns - 1) / turns : 1);
}
template <int RT, int KT, int KU, int NT, bool LIFT>
static hipError_t point_dft_launch(const PointArgs& g, hipStream_t st) {
    const size_t lds = ((size_t)KU * ((g.rowlen + 63) / 64) * 2048 + (size_t)(g.rowlen / 32) * NT * 512 +
                        4 * RT * 16 * (64 + 8)) * sizeof(__bf16);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)k_pointwise<RT, KT, KU, NT, LIFT>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const long cap = 160 * 1024 / (long)lds, wv = point_waves(RT, KT, KU);
    k_pointwise<RT, KT, KU, NT, LIFT><<<turns_grid((g.nrows + 3) / 4, 256 * (cap < wv ? cap : wv)), 256, lds, st>>>(g);
    return hipGetLastError();
}
template <int RT, int KT, int KU>
static hipError_t point_launch(const PointArgs& g, hipStream_t st) {
    if constexpr (RT <= 2 && KU <= 1) {
        if constexpr (KT == 1 && KU == 1)
            if (g.T && g.L)
                return g.dm <= 8 ? point_dft_launch<RT, 1, 1, 1, true>(g, st) : point_dft_launch<RT, 1, 1, 2, true>(g, st);
        if (g.T)
            return g.dm <= 8 ? point_dft_launch<RT, KT, KU, 1, false>(g, st)
                             : point_dft_launch<RT, KT, KU, 2, false>(g, st);
    }
    const long wg = (g.nrows * ((g.rowlen + 63) / 64) + 3) / 4;
    const unsigned grid = turns_grid(wg, 256 * (RT * KT == 1 ? 4 : point_waves(RT, KT, KU)));
    const size_t lds = (size_t)KU * ((g.rowlen + 63) / 64) * 256 * 8 * sizeof(__bf16);
    k_pointwise<RT, KT, KU, 0, false><<<grid, 256, lds, st>>>(g);
    return hipGetLastError();
}

template <int RT, int KT>
static hipError_t point_ku(const PointArgs& g, hipStream_t st) {
    if (!g.U) return point_launch<RT, KT, 0>(g, st);
    return g.K2 <= 32 ? point_launch<RT, KT, 1>(g, st) : point_launch<RT, KT, 2>(g, st);
}
template <int RT>
static hipError_t point_kt(const PointArgs& g, hipStream_t st) {
    return g.Cin <= 32 ? point_ku<RT, 1>(g, st) : point_ku<RT, 2>(g, st);
}

// The network's tail for inference, in one pass over the pixels: the last
// block's map h' = W h + U F + bias (no activation), q = GELU(Q1 h' + q1b),
// y = Q2 q + q2b, without writing h' and q: their rows are taken in tile_row's
// order, so that each product's results are the next one's operand (BF16) in the
// same lane.  Products, sums and roundings as the three k_pointwise passes: the
// same results.  Bound: VALU (64 GELUs a pixel).  50 images of 256^2, 32 and 64
// channels: 222 us, where operands passed through LDS took 255 and the three
// passes 194 + 276 + 207 us, with 1.3 GB written and read between them.
struct TailArgs {
    PointArgs b;     // the block's map (act 0, no pre; out unused)
    const float *Q1, *q1b, *Q2, *q2b;
    int H, cout;
    float* y;        // [cout][nrows][rowlen]
};
// KT, KH: steps of 32 channels of h and h', and of q
template <int KT, int KH, int KU>
__global__ void __launch_bounds__(256, (KT == 1 ? 2 : 1)) k_tail(TailArgs g) {
    constexpr int RT = 2 * KT, RH = 2 * KH;
    extern __shared__ __attribute__((aligned(16))) __bf16 Fs[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lm = lane & 15, lk = (lane >> 4) * 8, lr = (lane >> 4) * 4;
    const int C = g.b.Cout;
    const long SP = g.b.nrows * g.b.rowlen;
    const int ngrp = (g.b.rowlen + 63) / 64;
    stage_xtable<KU>(Fs, g.b.F, g.b.sfk, g.b.sfx, g.b.K2, g.b.rowlen);
    __syncthreads();
    bf16x8 wa[RT][KT], q1[RH][KT], q2[1][KH];
    matrix_operands<RT, KT, true>(wa, g.b.W, g.b.swm, g.b.swk, C, g.b.Cin, lm, lk);
    matrix_operands<RH, KT, true>(q1, g.Q1, C, 1, g.H, C, lm, lk);
    matrix_operands<1, KH>(q2, g.Q2, g.H, 1, g.cout, g.H, lm, lk);
    float b0[KT][8], b1[KH][8], b2[4];
#pragma unroll
    for (int j = 0; j < 8; j++) {
#pragma unroll
        for (int k = 0; k < KT; k++) b0[k][j] = g.b.bias[min(k * 32 + lk + j, C - 1)];
#pragma unroll
        for (int k = 0; k < KH; k++) b1[k][j] = g.q1b[min(k * 32 + lk + j, g.H - 1)];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) b2[q] = g.q2b[min(lr + q, g.cout - 1)];
    const long units = g.b.nrows * ngrp;
    for (long u = (long)blockIdx.x * 4 + wave; u < units; u += (long)gridDim.x * 4) {
        const long r = u / ngrp;
        const int x0 = (int)(u - r * ngrp) * 64;
        bf16x8 ua[RT][KU];
        spectrum_operands<RT, KU, true>(ua, g.b.U, g.b.nrows, r, C, g.b.K2, lm, lk);
        const bool in = x0 + 4 * lm < g.b.rowlen;
        const long p = r * g.b.rowlen + min(x0 + 4 * lm, g.b.rowlen - 4);
        float4 hv[KT][8];
        load_channels<KT>(hv, g.b.h, SP, p, g.b.Cin, lk);
        float yv[4][4];  // [t][row]
#pragma unroll
        for (int t = 0; t < 4; t++) {
            bf16x8 hb[KT], xb[KT];
            pixel_operands<KT>(hb, hv, t, g.b.Cin, lk);
#pragma unroll
            for (int k = 0; k < KT; k++) {
                float v[8];  // channels 32 k + lk + 0 .. 7, zero past the last
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int rt = 2 * k + i;
                    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, sp = acc;
#pragma unroll
                    for (int kt = 0; kt < KT; kt++)
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[rt][kt], hb[kt], acc, 0, 0, 0);
#pragma unroll
                    for (int ku = 0; ku < KU; ku++)
                        sp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            ua[rt][ku],
                            *reinterpret_cast<const bf16x8*>(Fs + ((size_t)((ku * ngrp + (x0 >> 6)) * 4 + t) * 64 + lane) * 8),
                            sp, 0, 0, 0);
                    acc += sp;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        v[4 * i + q] = acc[q] + b0[k][4 * i + q];
                        if (k * 32 + lk + 4 * i + q >= C) v[4 * i + q] = 0.f;
                    }
                }
                xb[k] = to_bf16x8(v);
            }
            f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KH; k++) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int kt = 0; kt < KT; kt++)
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q1[2 * k + i][kt], xb[kt], acc, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        v[4 * i + q] = gelu_t(acc[q] + b1[k][4 * i + q], nullptr);
                        if (k * 32 + lk + 4 * i + q >= g.H) v[4 * i + q] = 0.f;
                    }
                }
                y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q2[0][k], to_bf16x8(v), y, 0, 0, 0);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) yv[t][q] = y[q] + b2[q];
        }
        if (!in) continue;
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (lr + q < g.cout)
                *reinterpret_cast<float4*>(g.y + (lr + q) * SP + p) =
                    make_float4(yv[0][q], yv[1][q], yv[2][q], yv[3][q]);
    }
}

template <int KT, int KH, int KU>
static hipError_t tail_launch(const TailArgs& g, hipStream_t st) {
    const long wg = (g.b.nrows * ((g.b.rowlen + 63) / 64) + 3) / 4;
    const size_t lds = (size_t)KU * ((g.b.rowlen + 63) / 64) * 256 * 8 * sizeof(__bf16);  // 64 KB at most
    k_tail<KT, KH, KU><<<turns_grid(wg, 256 * (KT == 1 ? 2 : 1)), 256, lds, st>>>(g);
    return hipGetLastError();
}
template <int KT>
static hipError_t tail_kt(const TailArgs& g, hipStream_t st) {
    if (g.b.K2 <= 32) return g.H <= 32 ? tail_launch<KT, 1, 1>(g, st) : tail_launch<KT, 2, 1>(g, st);
    return g.H <= 32 ? tail_launch<KT, 1, 2>(g, st) : tail_launch<KT, 2, 2>(g, st);
}
hipError_t launch_tail(const float* W, int C, const float* h, long nrows, int rowlen, const float* U, int K2,
                       const float* F, long sfk, long sfx, const float* bias, const float* Q1, const float* q1b, int H,
                       const float* Q2, const float* q2b, int cout, float* y, hipStream_t st) {
    TailArgs g{};
    g.b = PointArgs{W, C, 1, C, C, h, nullptr, nrows, rowlen, U, K2, F, sfk, sfx, bias, nullptr, 0};
    g.Q1 = Q1;
    g.q1b = q1b;
    g.Q2 = Q2;
    g.q2b = q2b;
    g.H = H;
    g.cout = cout;
    g.y = y;
    return C <= 32 ? tail_kt<1>(g, st) : tail_kt<2>(g, st);
}

// Channel maps of at most 64 in and out channels over rows of a multiple of 4
// pixels at 16-byte aligned addresses (rows of at most 512 pixels and 64
// spectrum values with U); anything else takes k_gemm_bf16.
bool pointwise_supported(const float* h, const float* out, const float* pre, const float* U, long Cout, long Cin,
                         long nrows, long rowlen, long K2) {
    const uintptr_t a = (uintptr_t)h | (uintptr_t)out | (uintptr_t)pre | (uintptr_t)U;
    return Cout >= 1 && Cout <= 64 && Cin >= 1 && Cin <= 64 && nrows >= 1 && rowlen >= 4 && rowlen % 4 == 0 &&
           (a & 15) == 0 && nrows * (rowlen / 4) < (1L << 40) && rowlen < (1L << 30) &&
           (!U || (rowlen <= 512 && K2 >= 4 && K2 <= 64 && K2 % 4 == 0));
}

// With the transform of out: at most 32 channels and 16 modes (more accumulators
// and LDS rows than a wave has room for beside the map's own) over rows of a
// multiple of 32 pixels that the tables' LDS holds.
bool point_dft_supported(const void* T, long Cout, long rowlen, long dm, long K2) {
    return Cout <= 32 && rowlen % 32 == 0 && rowlen <= 512 && dm >= 1 && dm <= 16 && K2 <= 32 && ((uintptr_t)T & 15) == 0;
}

hipError_t launch_pointwise(const float* W, long swm, long swk, int Cout, int Cin, const float* h, float* out,
                            long nrows, int rowlen, const float* U, int K2, const float* F, long sfk, long sfx,
                            const float* bias, float* pre, int act, hipStream_t st, const float* D, long dsk, long dsn,
                            int dm, void* T, const float* L, const float* Lb, int cl) {
    if (!pointwise_supported(h, out, pre, U, Cout, Cin, nrows, rowlen, K2)) return hipErrorInvalidValue;
    if (T && !point_dft_supported(T, Cout, rowlen, dm, K2)) return hipErrorInvalidValue;
    if (L && (!T || !U || !Lb || Cin > 32 || cl < 1 || cl > 32)) return hipErrorInvalidValue;
    if (!U && !T) {  // no rows to tell apart: the image as rows of 64 pixels
        const long SP = nrows * rowlen;
        if (SP % 64 == 0) {
            nrows = SP / 64;
            rowlen = 64;
        }
    }
    const PointArgs g{W, swm, swk, Cout, Cin, h, out, nrows, rowlen, U, K2, F, sfk, sfx, bias, pre, act,
                      D, dsk, dsn, dm, (__bf16*)T, L, Lb, cl};
    switch ((Cout + 15) / 16) {
        case 1: return point_kt<1>(g, st);
        case 2: return point_kt<2>(g, st);
        case 3: return point_kt<3>(g, st);
        default: return point_kt<4>(g, st);
    }
}

// ------------------------------------------------------------------ spectral path
// The products of a block's spectral path, forward and backward, each complex
// product in one pass: the four real products in accumulators of their own, in
// k_gemm_bf16's order (k steps of 32, zero padded), and added last in the order
// its passes added them (first product kept, second added with its sign): the
// same results.  As k_gemm_bf16 passes a complex product read its operands
// and its half-written output four times over, in 4-byte loads.

// the 8 values X[k + j] (j < 8) of one operand row, zero past K
__device__ __forceinline__ bf16x8 operand8(const float* __restrict__ X, long sk, int k, int K) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        v[j] = X[min(k + j, K - 1) * sk];
        if (k + j >= K) v[j] = 0.f;
    }
    return to_bf16x8(v);
}
// the same from interleaved complex values: real and imaginary operands
__device__ __forceinline__ void operand8c(const float* __restrict__ X, long sk, int k, int K, bf16x8& re, bf16x8& im) {
    float a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float2 z = *reinterpret_cast<const float2*>(X + min(k + j, K - 1) * sk);
        a[j] = z.x;
        b[j] = z.y;
        if (k + j >= K) a[j] = b[j] = 0.f;
    }
    re = to_bf16x8(a);
    im = to_bf16x8(b);
}
#define MFMA16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16((a), (b), (c), 0, 0, 0)

// G [2m][N] staged as MFMA operands [re, im][NT][k step][lane][8] by TH threads
template <int NT>
__device__ __forceinline__ void stage_gtable(__bf16* Gs, const float* __restrict__ Gre, const float* __restrict__ Gim,
                                             int N, int M2, int TH) {
    const int KS = N / 32;
    for (int e = threadIdx.x; e < 2 * NT * KS * 64; e += TH) {
        const int ln = e & 63, t = e >> 6, ks = t % KS, mt = (t / KS) % NT, ri = t / (KS * NT);
        const int r = min(mt * 16 + (ln & 15), M2 - 1), k = ks * 32 + (ln >> 4) * 8;
        const float* p = (ri ? Gim : Gre) + (long)r * N + k;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = p[j];
        *reinterpret_cast<bf16x8*>(Gs + (size_t)e * 8) = to_bf16x8(v);
    }
}
// out[ky][kx] = sum_y G[ky][y] T[y][kx] (complex) of one image, T as columns of
// y in LDS (Tt[2 kx + (re, im)][TS])
template <int NT>
__device__ __forceinline__ void ydft_tasks(const __bf16* Gs, const __bf16* Tt, float* __restrict__ out, int KS, int TS,
                                           int m, int wave, int nwave, int lane) {
    const int lm = lane & 15, lk = (lane >> 4) * 8, M2 = 2 * m, NX = (m + 15) / 16;
    // one (ky tile, kx tile, re or im) per wave
    for (int task = wave; task < NT * NX * 2; task += nwave) {
        const int ri = task & 1, nx = (task >> 1) % NX, mt = (task >> 1) / NX;
        f32x4 p = {0.f, 0.f, 0.f, 0.f}, s = {0.f, 0.f, 0.f, 0.f};
        const __bf16* tr = Tt + (2 * (nx * 16 + lm) + ri) * TS + lk;        // multiplied by Gre
        const __bf16* ti = Tt + (2 * (nx * 16 + lm) + 1 - ri) * TS + lk;    // multiplied by Gim
        for (int ks = 0; ks < KS; ks++) {
            const bf16x8 gr = *reinterpret_cast<const bf16x8*>(Gs + ((size_t)(mt * KS + ks) * 64 + lane) * 8);
            const bf16x8 gi = *reinterpret_cast<const bf16x8*>(Gs + ((size_t)((NT + mt) * KS + ks) * 64 + lane) * 8);
            p = MFMA16(gr, *reinterpret_cast<const bf16x8*>(tr + ks * 32), p);
            s = MFMA16(gi, *reinterpret_cast<const bf16x8*>(ti + ks * 32), s);
        }
        const int kx = nx * 16 + lm;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int ky = mt * 16 + (lane >> 4) * 4 + q;
            if (ky < M2 && kx < m) out[((long)ky * m + kx) * 2 + ri] = ri ? p[q] + s[q] : p[q] - s[q];
        }
    }
}

// Retained spectrum of real N x N images: T = h F along x (F[x sfk + c sfn],
// 2m columns: re and im of m modes), then out[ky][kx] = sum_y G[ky][y] T[y][kx]
// (complex) for 2m ky.  One workgroup takes one image at a time: a wave
// transforms 16 rows from float4 loads, T stays in LDS as the BF16 operand of the
// second product (N + 8 values per column), and F and G are staged once per
// workgroup as MFMA operands.  Bound: HBM (the image read once).  1 600 images
// of 256^2, 16 modes (419 MB): 113 us, 3.7 TB/s, where the x product (292 us)
// and the four real y products (49 us each) took 489 us.
template <int NT, int DFT_T>
__global__ void __launch_bounds__(DFT_T) k_dft2(const float* __restrict__ h, const float* __restrict__ F, long sfk,
                                                long sfn, const float* __restrict__ Gre,
                                                const float* __restrict__ Gim, float* __restrict__ out, long images,
                                                int N, int m) {
    extern __shared__ __attribute__((aligned(16))) __bf16 sm[];
    const int KS = N / 32, M2 = 2 * m, TS = N + 8;
    __bf16* Fs = sm;                                  // [KS][NT][lane][8]
    __bf16* Gs = Fs + (size_t)KS * NT * 512;          // [re, im][NT][KS][lane][8]
    __bf16* Tt = Gs + (size_t)2 * NT * KS * 512;      // [column 2 kx + (re, im)][TS]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lm = lane & 15, lk = (lane >> 4) * 8;
    stage_dtable<NT>(Fs, F, sfk, sfn, N, M2, DFT_T);
    stage_gtable<NT>(Gs, Gre, Gim, N, M2, DFT_T);
    for (long img = blockIdx.x; img < images; img += gridDim.x) {
        __syncthreads();  // the tables are staged / the previous image's T is read
        const float* hi = h + img * N * N;
        for (int y0 = wave * 16; y0 < N; y0 += DFT_T / 64 * 16) {
            const float* row = hi + (long)(y0 + lm) * N + lk;
            f32x4 acc[NT];
#pragma unroll
            for (int nt = 0; nt < NT; nt++) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < KS; k0 += 4) {
                float4 a[4][2];  // the loads of 4 k steps together
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float* p = row + min(k0 + q, KS - 1) * 32;
                    a[q][0] = *reinterpret_cast<const float4*>(p);
                    a[q][1] = *reinterpret_cast<const float4*>(p + 4);
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (k0 + q >= KS) break;
                    const float v[8] = {a[q][0].x, a[q][0].y, a[q][0].z, a[q][0].w,
                                        a[q][1].x, a[q][1].y, a[q][1].z, a[q][1].w};
                    const bf16x8 av = to_bf16x8(v);
#pragma unroll
                    for (int nt = 0; nt < NT; nt++)
                        acc[nt] = MFMA16(av, *reinterpret_cast<const bf16x8*>(Fs + ((size_t)((k0 + q) * NT + nt) * 64 + lane) * 8),
                                         acc[nt]);
                }
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const bf16x4 t = {(__bf16)acc[nt][0], (__bf16)acc[nt][1], (__bf16)acc[nt][2], (__bf16)acc[nt][3]};
                *reinterpret_cast<bf16x4*>(Tt + (nt * 16 + lm) * TS + y0 + (lane >> 4) * 4) = t;
            }
        }
        __syncthreads();
        ydft_tasks<NT>(Gs, Tt, out + img * M2 * m * 2, KS, TS, m, wave, DFT_T / 64, lane);
    }
}

// The retained spectrum from T [images][N][16 NT] (BF16), the images' transform
// along x as k_pointwise leaves it: k_dft2's second half.  Bound: HBM (T read).
template <int NT>
__global__ void __launch_bounds__(256) k_dft_y(const __bf16* __restrict__ T, const float* __restrict__ Gre,
                                               const float* __restrict__ Gim, float* __restrict__ out, long images,
                                               int N, int m) {
    extern __shared__ __attribute__((aligned(16))) __bf16 sm[];
    const int KS = N / 32, M2 = 2 * m, TS = N + 8;
    __bf16* Gs = sm;
    __bf16* Tt = Gs + (size_t)2 * NT * KS * 512;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    stage_gtable<NT>(Gs, Gre, Gim, N, M2, 256);
    for (long img = blockIdx.x; img < images; img += gridDim.x) {
        __syncthreads();  // the tables are staged / the previous image's T is read
        // y on the lanes: a lane's 8 columns of one y go to 8 rows of Tt
        for (int e = threadIdx.x; e < N * NT * 2; e += 256) {
            const int y = e % N, c8 = e / N;
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(T + ((size_t)img * N + y) * (NT * 16) + c8 * 8);
#pragma unroll
            for (int j = 0; j < 8; j++) Tt[(c8 * 8 + j) * TS + y] = v[j];
        }
        __syncthreads();
        ydft_tasks<NT>(Gs, Tt, out + img * M2 * m * 2, KS, TS, m, wave, 4, lane);
    }
}

// U[y][kx] = sum_ky conj(G[ky][y]) O[ky][kx] (complex): the spectra back along
// y.  A workgroup stages G once as MFMA operands; a wave keeps an image's
// spectrum operands and makes its 16-row tiles.  Bound: HBM (U written).
template <int KT>
__global__ void __launch_bounds__(256) k_idft_y(const float* __restrict__ Gre, const float* __restrict__ Gim,
                                                const float* __restrict__ O, float* __restrict__ U, long images,
                                                int N, int m) {
    extern __shared__ __attribute__((aligned(16))) __bf16 sm[];
    const int M2 = 2 * m, YT = N / 16, NX = (m + 15) / 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lm = lane & 15, lk = (lane >> 4) * 8;
    // [re, im][YT][KT][lane][8]: row y, k = ky
    for (int e = threadIdx.x; e < 2 * YT * KT * 64; e += 256) {
        const int ln = e & 63, t = e >> 6, kt = t % KT, yt = (t / KT) % YT, ri = t / (KT * YT);
        *reinterpret_cast<bf16x8*>(sm + (size_t)e * 8) =
            operand8((ri ? Gim : Gre) + yt * 16 + (ln & 15), N, kt * 32 + (ln >> 4) * 8, M2);
    }
    __syncthreads();
    for (long img = blockIdx.x; img < images; img += gridDim.x)
        for (int nx = 0; nx < NX; nx++) {
            const int kx = nx * 16 + lm;
            bf16x8 ore[KT], oim[KT];
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
                operand8c(O + (img * M2 * m + min(kx, m - 1)) * 2, 2 * m, kt * 32 + lk, M2, ore[kt], oim[kt]);
            for (int yt = wave; yt < YT; yt += 4) {
                f32x4 rr = {0.f, 0.f, 0.f, 0.f}, ii = rr, ri = rr, ir = rr;
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
                    const bf16x8 gr = *reinterpret_cast<const bf16x8*>(sm + ((size_t)(yt * KT + kt) * 64 + lane) * 8);
                    const bf16x8 gi =
                        *reinterpret_cast<const bf16x8*>(sm + ((size_t)((YT + yt) * KT + kt) * 64 + lane) * 8);
                    rr = MFMA16(gr, ore[kt], rr);
                    ii = MFMA16(gi, oim[kt], ii);
                    ri = MFMA16(gr, oim[kt], ri);
                    ir = MFMA16(gi, ore[kt], ir);
                }
                if (kx < m)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const long y = img * N + yt * 16 + (lane >> 4) * 4 + q;
                        *reinterpret_cast<float2*>(U + y * M2 + 2 * kx) = make_float2(rr[q] + ii[q], ri[q] - ir[q]);
                    }
            }
        }
}

// Per retained mode (one wave each): out[o][s] = sum_i R[o][i] B[i][s], or with
// ADJ out[i][s] = sum_o conj(R[o][i]) B[o][s].  R [mode][C][C], B and out
// [C][S][mode], complex; the four waves of a workgroup take adjacent modes.
template <int RT, int KT, bool ADJ>
__global__ void __launch_bounds__(256) k_mix(const float* __restrict__ R, const float* __restrict__ B,
                                             float* __restrict__ out, int C, int S, int nm) {
    const int lane = threadIdx.x & 63, lm = lane & 15, lk = (lane >> 4) * 8;
    const int mode = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (mode >= nm) return;
    bf16x8 are[RT][KT], aim[RT][KT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            const int r = min(rt * 16 + lm, C - 1);
            operand8c(R + ((long)mode * C * C + (ADJ ? r : r * C)) * 2, ADJ ? 2 * C : 2, kt * 32 + lk, C, are[rt][kt],
                      aim[rt][kt]);
        }
    for (int s0 = blockIdx.y * 16; s0 < S; s0 += gridDim.y * 16) {
        bf16x8 bre[KT], bim[KT];
#pragma unroll
        for (int kt = 0; kt < KT; kt++)
            operand8c(B + ((long)min(s0 + lm, S - 1) * nm + mode) * 2, 2L * S * nm, kt * 32 + lk, C, bre[kt], bim[kt]);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            f32x4 rr = {0.f, 0.f, 0.f, 0.f}, ii = rr, ri = rr, ir = rr;
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
                rr = MFMA16(are[rt][kt], bre[kt], rr);
                ii = MFMA16(aim[rt][kt], bim[kt], ii);
                ri = MFMA16(are[rt][kt], bim[kt], ri);
                ir = MFMA16(aim[rt][kt], bre[kt], ir);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = rt * 16 + (lane >> 4) * 4 + q;
                if (r < C && s0 + lm < S)
                    *reinterpret_cast<float2*>(out + (((long)r * S + s0 + lm) * nm + mode) * 2) =
                        ADJ ? make_float2(rr[q] + ii[q], ri[q] - ir[q]) : make_float2(rr[q] - ii[q], ri[q] + ir[q]);
            }
        }
    }
}

// Gradient of the mixing matrices, one wave per mode and 16 rows:
// dR[o][i] = sum_s dO[o][s] conj(B[i][s]).
template <int CT>
__global__ void __launch_bounds__(256) k_mix_grad(const float* __restrict__ dO, const float* __restrict__ B,
                                                  float* __restrict__ dR, int C, int S, int nm) {
    const int lane = threadIdx.x & 63, lm = lane & 15, lk = (lane >> 4) * 8;
    const int mode = blockIdx.x * 4 + (threadIdx.x >> 6), rt = blockIdx.y;
    if (mode >= nm) return;
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    f32x4 rr[CT], ii[CT], ri[CT], ir[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) rr[ct] = ii[ct] = ri[ct] = ir[ct] = z;
    for (int k0 = 0; k0 < S; k0 += 32) {
        bf16x8 are, aim;
        operand8c(dO + ((long)min(rt * 16 + lm, C - 1) * S * nm + mode) * 2, 2L * nm, k0 + lk, S, are, aim);
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            bf16x8 bre, bim;
            operand8c(B + ((long)min(ct * 16 + lm, C - 1) * S * nm + mode) * 2, 2L * nm, k0 + lk, S, bre, bim);
            rr[ct] = MFMA16(are, bre, rr[ct]);
            ii[ct] = MFMA16(aim, bim, ii[ct]);
            ir[ct] = MFMA16(aim, bre, ir[ct]);
            ri[ct] = MFMA16(are, bim, ri[ct]);
        }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = rt * 16 + (lane >> 4) * 4 + q, i = ct * 16 + lm;
            if (r < C && i < C)
                *reinterpret_cast<float2*>(dR + (((long)mode * C + r) * C + i) * 2) =
                    make_float2(rr[ct][q] + ii[ct][q], ir[ct][q] - ri[ct][q]);
        }
}

// Weight gradient of a channel map, part[chunk][o][i] = sum over the chunk's
// kc pixels of dy[o][q] h[i][q]: one wave takes a chunk and every 16 x 16 tile of
// (o, i), so that each value is loaded and rounded once, straight from float4 loads
// (both operands are contiguous along the sum), the loads of UN k steps in flight.
// Order and results as k_gemm_bf16.  Bound: HBM.  32 x 32 channels over 524 288
// pixels (134 MB): 34 us, 64 x 32 76 us, against 45 and 92 with one tile a wave
// and 53 through k_gemm_bf16's LDS staging.  With bpart also the chunk's sums of
// dy, bpart[chunk][o], in FP64 from the same loads: a pass of its own reads dy
// again (12 us for 67 MB).
template <int RT, int CT>
__global__ void __launch_bounds__(64) k_weight_grad(const float* __restrict__ dy, const float* __restrict__ h,
                                                    float* __restrict__ part, double* __restrict__ bpart, int Cout,
                                                    int Cin, long SP, int kc) {
    constexpr int UN = RT + CT <= 4 ? 4 : RT + CT <= 6 ? 2 : 1;
    const int lane = threadIdx.x, lm = lane & 15, lk = (lane >> 4) * 8;
    const float *a[RT], *b[CT];
#pragma unroll
    for (int r = 0; r < RT; r++) a[r] = dy + min(r * 16 + lm, Cout - 1) * SP + (long)blockIdx.x * kc + lk;
#pragma unroll
    for (int q = 0; q < CT; q++) b[q] = h + min(q * 16 + lm, Cin - 1) * SP + (long)blockIdx.x * kc + lk;
    f32x4 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int q = 0; q < CT; q++) acc[r][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    double bs[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) bs[r] = 0.0;
    float4 v[UN][RT + CT][2];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int s = 0; s < UN; s++)
#pragma unroll
            for (int t = 0; t < RT + CT; t++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    v[s][t][u] = *reinterpret_cast<const float4*>((t < RT ? a[t < RT ? t : 0] : b[t < RT ? 0 : t - RT]) +
                                                                  k0 + s * 32 + u * 4);
    };
    fetch(0);
    for (int k0 = 0; k0 < kc; k0 += 32 * UN) {  // kc is a multiple of 128
        bf16x8 o[UN][RT + CT];
#pragma unroll
        for (int s = 0; s < UN; s++)
#pragma unroll
            for (int t = 0; t < RT + CT; t++) {
                const float x[8] = {v[s][t][0].x, v[s][t][0].y, v[s][t][0].z, v[s][t][0].w,
                                    v[s][t][1].x, v[s][t][1].y, v[s][t][1].z, v[s][t][1].w};
                o[s][t] = to_bf16x8(x);
                if (t < RT && bpart)
#pragma unroll
                    for (int j = 0; j < 8; j++) bs[t < RT ? t : 0] += (double)x[j];
            }
        fetch(min(k0 + 32 * UN, kc - 32 * UN));  // the next steps' loads beside the products
#pragma unroll
        for (int s = 0; s < UN; s++)
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int q = 0; q < CT; q++) acc[r][q] = MFMA16(o[s][r], o[s][RT + q], acc[r][q]);
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int oo = r * 16 + (lane >> 4) * 4 + q, i = c * 16 + lm;
                if (oo < Cout && i < Cin) part[((long)blockIdx.x * Cout + oo) * Cin + i] = acc[r][c][q];
            }
    if (!bpart) return;
#pragma unroll
    for (int r = 0; r < RT; r++) {
        bs[r] += __shfl_xor(bs[r], 16);
        bs[r] += __shfl_xor(bs[r], 32);
        if (lane < 16 && r * 16 + lm < Cout) bpart[(long)blockIdx.x * Cout + r * 16 + lm] = bs[r];
    }
}

// at most 64 channels each way, chunks of a multiple of 128 pixels, 16-byte
// aligned rows
bool weight_grad_supported(const float* dy, const float* h, long Cout, long Cin, long SP, long kc) {
    return Cout >= 1 && Cout <= 64 && Cin >= 1 && Cin <= 64 && kc >= 128 && kc % 128 == 0 && kc <= (1L << 24) &&
           SP % kc == 0 && SP / kc < (1L << 31) && (((uintptr_t)dy | (uintptr_t)h) & 15) == 0;
}
hipError_t launch_weight_grad(const float* dy, const float* h, float* part, double* bpart, int Cout, int Cin, long SP,
                              int kc, hipStream_t st) {
    const unsigned grid = (unsigned)(SP / kc);
    switch ((Cout + 15) / 16 * 4 + (Cin + 15) / 16 - 5) {
#define X(RT, CT)                                                                       \
    case (RT - 1) * 4 + CT - 1:                                                         \
        k_weight_grad<RT, CT><<<grid, 64, 0, st>>>(dy, h, part, bpart, Cout, Cin, SP, kc);     \
        return hipGetLastError();
        X(1, 1) X(1, 2) X(1, 3) X(1, 4) X(2, 1) X(2, 2) X(2, 3) X(2, 4)
        X(3, 1) X(3, 2) X(3, 3) X(3, 4) X(4, 1) X(4, 2) X(4, 3) X(4, 4)
#undef X
        default: return hipErrorInvalidValue;
    }
}

static size_t dft2_lds(long N, long m) {
    const long nt = (2 * m + 15) / 16, ks = N / 32;
    return (size_t)(3 * nt * ks * 512 + 32 * ((m + 15) / 16) * (N + 8)) * sizeof(__bf16);
}
// images of N x N, N a multiple of 32, at most 32 modes, at 16-byte aligned
// addresses (spectra at 8), channels of at most 64, within the LDS of a CU
bool spectral_supported(const float* h, const float* U, const float* B, const float* O, const float* R, long images,
                        long N, long m, long C, long S) {
    return N >= 32 && N % 32 == 0 && N <= 1024 && m >= 1 && 2 * m <= N && m <= 32 && C >= 1 && C <= 64 && S >= 1 &&
           S <= (1L << 24) && images < (1L << 31) && (((uintptr_t)h | (uintptr_t)U) & 15) == 0 &&
           (((uintptr_t)B | (uintptr_t)O | (uintptr_t)R) & 7) == 0 && dft2_lds(N, m) <= 160 * 1024;
}

template <int NT, int TH>
static hipError_t dft2_launch_t(const float* h, const float* F, long sfk, long sfn, const float* Gre, const float* Gim,
                                float* out, long images, int N, int m, hipStream_t st) {
    const size_t lds = dft2_lds(N, m);
    if (lds > 64 * 1024) {
        hipError_t e =
            hipFuncSetAttribute((const void*)k_dft2<NT, TH>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const long res = 256 * (TH == 512 && lds <= 80 * 1024 ? 2 : 1);  // resident workgroups
    k_dft2<NT, TH><<<(unsigned)(images < res ? images : res), TH, lds, st>>>(h, F, sfk, sfn, Gre, Gim, out, images, N, m);
    return hipGetLastError();
}
template <int NT>
static hipError_t dft2_launch(const float* h, const float* F, long sfk, long sfn, const float* Gre, const float* Gim,
                              float* out, long images, int N, int m, hipStream_t st) {
    // few images: 16 waves on a CU's one image (256 of 256^2: 22 us against 25)
    if (images <= 256) return dft2_launch_t<NT, 1024>(h, F, sfk, sfn, Gre, Gim, out, images, N, m, st);
    return dft2_launch_t<NT, 512>(h, F, sfk, sfn, Gre, Gim, out, images, N, m, st);
}
template <int NT>
static hipError_t dft_y_launch(const __bf16* T, const float* Gre, const float* Gim, float* out, long images, int N, int m,
                               hipStream_t st) {
    const size_t lds = ((size_t)2 * NT * (N / 32) * 512 + (size_t)32 * (N + 8)) * sizeof(__bf16);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)k_dft_y<NT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const long res = 256 * (160 * 1024 / (long)lds < 4 ? 160 * 1024 / (long)lds : 4);
    k_dft_y<NT><<<turns_grid(images, res), 256, lds, st>>>(T, Gre, Gim, out, images, N, m);
    return hipGetLastError();
}
hipError_t launch_dft_y(const void* T, const float* Gre, const float* Gim, float* out, long images, int N, int m,
                        hipStream_t st) {
    if (images <= 0) return hipSuccess;
    return m <= 8 ? dft_y_launch<1>((const __bf16*)T, Gre, Gim, out, images, N, m, st)
                  : dft_y_launch<2>((const __bf16*)T, Gre, Gim, out, images, N, m, st);
}
hipError_t launch_dft2(const float* h, const float* F, long sfk, long sfn, const float* Gre, const float* Gim,
                       float* out, long images, int N, int m, hipStream_t st) {
    if (images <= 0) return hipSuccess;
    switch ((2 * m + 15) / 16) {
        case 1: return dft2_launch<1>(h, F, sfk, sfn, Gre, Gim, out, images, N, m, st);
        case 2: return dft2_launch<2>(h, F, sfk, sfn, Gre, Gim, out, images, N, m, st);
        case 3: return dft2_launch<3>(h, F, sfk, sfn, Gre, Gim, out, images, N, m, st);
        default: return dft2_launch<4>(h, F, sfk, sfn, Gre, Gim, out, images, N, m, st);
    }
}

template <int KT>
static hipError_t idft_y_launch(const float* Gre, const float* Gim, const float* O, float* U, long images, int N,
                                int m, hipStream_t st) {
    const size_t lds = (size_t)2 * (N / 16) * KT * 512 * sizeof(__bf16);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)k_idft_y<KT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const long res = 256 * (lds <= 40 * 1024 ? 4 : lds <= 80 * 1024 ? 2 : 1);
    k_idft_y<KT><<<(unsigned)(images < res ? images : res), 256, lds, st>>>(Gre, Gim, O, U, images, N, m);
    return hipGetLastError();
}
hipError_t launch_idft_y(const float* Gre, const float* Gim, const float* O, float* U, long images, int N, int m,
                         hipStream_t st) {
    if (images <= 0) return hipSuccess;
    return 2 * m <= 32 ? idft_y_launch<1>(Gre, Gim, O, U, images, N, m, st)
                       : idft_y_launch<2>(Gre, Gim, O, U, images, N, m, st);
}

template <int RT, int KT>
static hipError_t mix_launch(const float* R, const float* B, float* out, int C, int S, int nm, bool adj,
                             hipStream_t st) {
    const int gy = (S + 15) / 16;
    dim3 grid((nm + 3) / 4, gy < 64 ? gy : 64);
    if (adj) k_mix<RT, KT, true><<<grid, 256, 0, st>>>(R, B, out, C, S, nm);
    else k_mix<RT, KT, false><<<grid, 256, 0, st>>>(R, B, out, C, S, nm);
    return hipGetLastError();
}
hipError_t launch_mix(const float* R, const float* B, float* out, int C, int S, int nm, bool adj, hipStream_t st) {
    switch ((C + 15) / 16) {
        case 1: return mix_launch<1, 1>(R, B, out, C, S, nm, adj, st);
        case 2: return mix_launch<2, 1>(R, B, out, C, S, nm, adj, st);
        case 3: return mix_launch<3, 2>(R, B, out, C, S, nm, adj, st);
        default: return mix_launch<4, 2>(R, B, out, C, S, nm, adj, st);
    }
}
hipError_t launch_mix_grad(const float* dO, const float* B, float* dR, int C, int S, int nm, hipStream_t st) {
    const int ct = (C + 15) / 16;
    dim3 grid((nm + 3) / 4, ct);
    switch (ct) {
        case 1: k_mix_grad<1><<<grid, 256, 0, st>>>(dO, B, dR, C, S, nm); break;
        case 2: k_mix_grad<2><<<grid, 256, 0, st>>>(dO, B, dR, C, S, nm); break;
        case 3: k_mix_grad<3><<<grid, 256, 0, st>>>(dO, B, dR, C, S, nm); break;
        default: k_mix_grad<4><<<grid, 256, 0, st>>>(dO, B, dR, C, S, nm); break;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------ elementwise

// y = act(a + b + bias[channel]) over [S][C][P]; pre (optional) keeps a + b + bias
__global__ void k_add_bias_act(const float* __restrict__ a, const float* __restrict__ b,
                               const float* __restrict__ bias, float* __restrict__ pre, float* __restrict__ y,
                               long C, long P, long n, int gelu) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
        const long c = (e / P) % C;
        float v = a[e] + (b ? b[e] : 0.f) + (bias ? bias[c] : 0.f);
        if (pre) pre[e] = v;
        y[e] = gelu ? gelu_t(v, nullptr) : v;
    }
}

// dx = dy * gelu'(pre)
__global__ void k_gelu_bwd(const float* __restrict__ pre, const float* __restrict__ dy, float* __restrict__ dx,
                           long n) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
        float d;
        gelu_t(pre[e], &d);
        dx[e] = dy[e] * d;
    }
}

// partial[chunk][c] = sum of dy[s][c][p] over this workgroup's chunk of
// the S * P values of channel c, in FP64 as are the chunks' sums
// (k_reduce_batches)
__global__ void __launch_bounds__(256) k_bias_grad(const float* __restrict__ dy, double* __restrict__ partial, long S,
                                                   long C, long P) {
    const long c = blockIdx.x, nchunk = gridDim.y, chunk = blockIdx.y;
    const long n = S * P, per = (n + nchunk - 1) / nchunk;
    const long e0 = chunk * per, e1 = min(n, e0 + per);
    double acc = 0.0;
    if (S == 1) {  // one plane per channel: 8 loads ahead, no divisions (24 -> 13 us at 32 x 524 288)
        const float* d = dy + c * P;
        long e = e0 + threadIdx.x;
        for (; e + 7 * 256 < e1; e += 8 * 256) {
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = d[e + q * 256];
#pragma unroll
            for (int q = 0; q < 8; q++) acc += v[q];
        }
        for (; e < e1; e += 256) acc += d[e];
    } else {
        for (long e = e0 + threadIdx.x; e < e1; e += 256) {
            const long s = e / P, p = e - s * P;
            acc += dy[(s * C + c) * P + p];
        }
    }
    __shared__ double red[256];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[chunk * C + c] = red[0];
}

// mean squared error over n elements: partial sums of (pred - target)^2 and
// grad = 2 (pred - target) / n
__global__ void __launch_bounds__(256) k_mse(const float* __restrict__ pred, const float* __restrict__ target,
                                             float* __restrict__ grad, long n, double* __restrict__ partial) {
    double acc = 0.0;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n; e += (long)gridDim.x * 256L) {
        const float d = pred[e] - target[e];
        acc += (double)d * d;
        if (grad) grad[e] = 2.f * d / (float)n;
    }
    __shared__ double red[256];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// Adam (Kingma & Ba 2015) with bias correction.  Parameters are kept in FP32;
// the GEMMs round them to BF16 when they stage them
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, long n, float lr, float b1, float b2, float eps, float c1, float c2) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
        const float ge = g[e];
        const float me = fmaf(b1, m[e] - ge, ge);
        const float ve = fmaf(b2, v[e] - ge * ge, ge * ge);
        m[e] = me;
        v[e] = ve;
        w[e] -= lr * (me / c1) / (sqrtf(ve / c2) + eps);
    }
}

// The same step on up to ADAM_MOST tensors (blockIdx.y), one launch for a
// network's parameters: most of its tensors are a few hundred values, and each
// launch of its own costs more than they do.
__global__ void k_adam_many(AdamTensors p, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int k = blockIdx.y;
    float *__restrict__ w = p.w[k], *__restrict__ m = p.m[k], *__restrict__ v = p.v[k];
    const float* __restrict__ g = p.g[k];
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < p.n[k]; e += (long)gridDim.x * blockDim.x) {
        const float ge = g[e];
        const float me = fmaf(b1, m[e] - ge, ge);
        const float ve = fmaf(b2, v[e] - ge * ge, ge * ge);
        m[e] = me;
        v[e] = ve;
        w[e] -= lr * (me / c1) / (sqrtf(ve / c2) + eps);
    }
}

// out[i] (+)= sum_b part[b n + i]: the split-K partial products of the
// weight gradients, summed in a fixed order (b ascending, one accumulator).
// A workgroup takes 64 outputs: all four waves load 128 partials of each ahead
// into LDS, and its first wave adds them, so that the chain of dependent adds
// waits for LDS and not for memory (512 partials of 1 024 outputs: 7 us, against
// 66 with one thread walking each output's partials in memory).  A workgroup past
// those takes one bias gradient bout[c], the sum of bpart[b nbias + c] in FP64.
constexpr int RED_B = 128;
__global__ void __launch_bounds__(256) k_reduce_batches(const float* __restrict__ part, float* __restrict__ out,
                                                        long nb, long n, int accumulate,
                                                        const double* __restrict__ bpart, float* __restrict__ bout,
                                                        long nbias) {
    __shared__ __attribute__((aligned(16))) float P[RED_B][64];
    if (blockIdx.x >= (n + 63) / 64) {
        const long c = blockIdx.x - (n + 63) / 64;
        double acc = 0.0;
        for (long b = threadIdx.x; b < nb; b += 256) acc += bpart[b * nbias + c];
        double* red = reinterpret_cast<double*>(&P[0][0]);
        red[threadIdx.x] = acc;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
            __syncthreads();
        }
        if (threadIdx.x == 0) bout[c] = accumulate ? bout[c] + (float)red[0] : (float)red[0];
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long i = blockIdx.x * 64L + lane, ic = min(i, n - 1);
    float v[RED_B / 4];
    auto fetch = [&](long b0) {
#pragma unroll
        for (int q = 0; q < RED_B / 4; q++) v[q] = part[min(b0 + wave + 4 * q, nb - 1) * n + ic];
    };
    float acc = accumulate ? out[ic] : 0.f;
    fetch(0);
    for (long b0 = 0; b0 < nb; b0 += RED_B) {
        __syncthreads();  // the partials before are added
#pragma unroll
        for (int q = 0; q < RED_B / 4; q++) P[wave + 4 * q][lane] = v[q];
        __syncthreads();
        if (b0 + RED_B < nb) fetch(b0 + RED_B);
        if (wave == 0) {
            const int nr = (int)min((long)RED_B, nb - b0);
            if (nr == RED_B) {
#pragma unroll 16
                for (int q = 0; q < RED_B; q++) acc += P[q][lane];
            } else {
                for (int q = 0; q < nr; q++) acc += P[q][lane];
            }
        }
    }
    if (wave == 0 && i < n) out[i] = acc;
}

// Training / serving pairs of the surrogate from one step of the simulator.
// screens [D][L][N*N] (sampled layer screens), s[L] phase multipliers of the
// wavelength; for sample s0 + d, channel-major over Stot samples:
//   x[l][s][p]     = v_l / xs,  v_l = s_l screen_l            (phase, l < L)
//   x[L + l][s][p] = lap(v_l) / xl                            (5-point Laplacian,
//                                                              edge pixels clamped)
// and, when pha and amp are given, the smooth complex field perturbation
// u = amp e^{i (pha - Phi)}, Phi = sum_l v_l:
//   t[0][s][p] = (Re u - 1) / cs,  t[1][s][p] = Im u / ps.
__global__ void k_nn_pairs(const float* __restrict__ screens, const double* __restrict__ sc,
                           const float* __restrict__ pha, const float* __restrict__ amp, int L, int N, long Stot,
                           long s0, float* __restrict__ x, float* __restrict__ t, double xs, double xl, double cs,
                           double ps) {
    const int d = blockIdx.y;
    const long s = s0 + d, P = (long)N * N;
    for (long p = blockIdx.x * (long)blockDim.x + threadIdx.x; p < P; p += (long)gridDim.x * blockDim.x) {
        const int j = (int)(p / N), i = (int)(p - (long)j * N);
        const long pl = j * (long)N + max(i - 1, 0), pr = j * (long)N + min(i + 1, N - 1);
        const long pu = max(j - 1, 0) * (long)N + i, pd = min(j + 1, N - 1) * (long)N + i;
        double phi = 0.0;
        for (int l = 0; l < L; l++) {
            const float* sl = screens + ((long)d * L + l) * P;
            const double v = sc[l] * (double)sl[p];
            const double lap = sc[l] * ((double)sl[pl] + (double)sl[pr] + (double)sl[pu] + (double)sl[pd]) - 4.0 * v;
            phi += v;
            x[((long)l * Stot + s) * P + p] = (float)(v / xs);
            x[((long)(L + l) * Stot + s) * P + p] = (float)(lap / xl);
        }
        if (t && pha && amp) {
            const double a = (double)amp[(long)d * P + p];
            const double dp = (double)pha[(long)d * P + p] - phi;
            t[s * P + p] = (float)((a * cos(dp) - 1.0) / cs);
            t[(Stot + s) * P + p] = (float)(a * sin(dp) / ps);
        }
    }
}

// network output y [2][S][P] -> u = (1 + cs y0) + i ps y1; amp = |u|,
// pha = xs sum_{l < L} x_l + arg u
__global__ void k_nn_unpack(const float* __restrict__ y, const float* __restrict__ x, int L, long S, long P,
                            double xs, double cs, double ps, float* __restrict__ amp, float* __restrict__ pha) {
    const long n = S * P;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
        double phi = 0.0;
        for (int l = 0; l < L; l++) phi += (double)x[(long)l * n + e];
        const double ur = 1.0 + cs * (double)y[e], ui = ps * (double)y[n + e];
        amp[e] = (float)sqrt(ur * ur + ui * ui);
        pha[e] = (float)(xs * phi + atan2(ui, ur));
    }
}

static unsigned grid_for(long n) {
    long g = (n + 255) / 256;
    return (unsigned)(g < 8192 ? (g > 0 ? g : 1) : 8192);
}

hipError_t launch_add_bias_act(const float* a, const float* b, const float* bias, float* pre, float* y, long C,
                               long P, long n, int gelu, hipStream_t st) {
    k_add_bias_act<<<grid_for(n), 256, 0, st>>>(a, b, bias, pre, y, C, P, n, gelu);
    return hipGetLastError();
}
hipError_t launch_gelu_bwd(const float* pre, const float* dy, float* dx, long n, hipStream_t st) {
    k_gelu_bwd<<<grid_for(n), 256, 0, st>>>(pre, dy, dx, n);
    return hipGetLastError();
}
hipError_t launch_bias_grad(const float* dy, double* partial, long S, long C, long P, int nchunk, hipStream_t st) {
    k_bias_grad<<<dim3((unsigned)C, (unsigned)nchunk), 256, 0, st>>>(dy, partial, S, C, P);
    return hipGetLastError();
}
hipError_t launch_mse(const float* pred, const float* target, float* grad, long n, double* partial, int nblk,
                      hipStream_t st) {
    k_mse<<<nblk, 256, 0, st>>>(pred, target, grad, n, partial);
    return hipGetLastError();
}
hipError_t launch_reduce_batches(const float* part, float* out, long nb, long n, int accumulate, const double* bpart,
                                 float* bout, long nbias, hipStream_t st) {
    k_reduce_batches<<<(unsigned)((n + 63) / 64 + nbias), 256, 0, st>>>(part, out, nb, n, accumulate, bpart, bout, nbias);
    return hipGetLastError();
}
hipError_t launch_nn_pairs(const float* screens, const double* sc, const float* pha, const float* amp, long D, long L,
                           long N, long Stot, long s0, float* x, float* t, double xs, double xl, double cs, double ps,
                           hipStream_t st) {
    long g = (N * N + 255) / 256;
    dim3 grid((unsigned)(g < 2048 ? g : 2048), (unsigned)D);
    k_nn_pairs<<<grid, 256, 0, st>>>(screens, sc, pha, amp, (int)L, (int)N, Stot, s0, x, t, xs, xl, cs, ps);
    return hipGetLastError();
}
hipError_t launch_nn_unpack(const float* y, const float* x, long L, long S, long P, double xs, double cs, double ps,
                            float* amp, float* pha, hipStream_t st) {
    k_nn_unpack<<<grid_for(S * P), 256, 0, st>>>(y, x, (int)L, S, P, xs, cs, ps, amp, pha);
    return hipGetLastError();
}
hipError_t launch_adam_many(const AdamTensors& p, int count, float lr, float b1, float b2, float eps, float c1,
                            float c2, hipStream_t st) {
    long most = 1;
    for (int k = 0; k < count; k++) most = p.n[k] > most ? p.n[k] : most;
    const unsigned gx = grid_for(most) < 1024 ? grid_for(most) : 1024;
    k_adam_many<<<dim3(gx, count), 256, 0, st>>>(p, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}
hipError_t launch_adam(float* w, const float* g, float* m, float* v, long n, float lr, float b1, float b2, float eps,
                       float c1, float c2, hipStream_t st) {
    k_adam<<<grid_for(n), 256, 0, st>>>(w, g, m, v, n, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}

}  // namespace atsim
