// atsim_launch.hpp -- host-side launchers of the HIP kernels (atsim_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "atsim_kernels.hpp"

namespace atsim {

enum { OP_FFT = 0, OP_FRESNEL = 1 };

bool supported_n(long n);

// Row pass over F fields of n x n, from in (field f at in + f istride; istride
// 0: one field for all) to out (may be in): op OP_FRESNEL = FFT_x, x h(kx)
// (table tf + (f % W) n), IFFT_x; OP_FFT = one transform of sign dir.  wcnt > 0
// (Fresnel): F = D * wcnt fields, wavelengths wlo .. of each direction.
hipError_t launch_row(long n, int op, int dir, const float2* in, long istride, float2* out, long F, const float2* tf,
                      int W, const float2* tw, hipStream_t st, int wlo = 0, int wcnt = 0);
// Fresnel x pass of every (direction, wavelength) field with the screen
// phase of the layer group sa.lfirst .. + sa.lcount (sampled once per pixel
// and direction); gen: the incoming field is 1.  Tables tf + w n.
// mw: wavelengths per workgroup (0 = largest that fits).  tfp (not with
// gen): the x factor of the gap before the group is applied first (tables
// tfp + w n).  tw: the n twiddles followed by the per-stage tables
// (tw_tables_size(n) entries, tw_stage_off).
hipError_t launch_row_fresnel(long n, bool gen, float2* data, int D, const float2* tf, const float2* tw,
                              const ScreenArgs& sa, hipStream_t st, int mw = 0, const float2* tfp = nullptr);
// Column pass around a layer group: y factor tfp of the gap before the
// group, the group's screen phase (layers sa.lfirst .. + sa.lcount, their
// sampled phases in planes slot0 .. of vq), y factor tf of the gap after it;
// every field of the wavelength range of sa (tables + w n).  n <= 4096.
// e: elements per thread (0 = by size and fields, 16 or 32 forced where built).
// tw as for launch_row_fresnel (with the per-stage tables).
hipError_t launch_col_screen(long n, float2* data, int D, const float2* tfp, const float2* tf, const float2* tw,
                             const ScreenArgs& sa, const double* vq, int slot0, hipStream_t st, int e = 0);
// The row pass around a layer group whose phases are in planes, as
// launch_col_screen along x; tfp null: the first pass (the incoming field is 1).
hipError_t launch_row_screen(long n, float2* data, int D, const float2* tfp, const float2* tf, const float2* tw,
                             const ScreenArgs& sa, const double* vq, int slot0, hipStream_t st);
// Sampled phase planes (FP64 quarter turns) of layers slot_layer[0 ..
// nslots) for every direction: vq[((slot D + d) n + j) n + i].
hipError_t launch_layer_phase(double* vq, const float* masters, const LayerSample* ls, const int* slot_layer,
                              int nslots, long n, long M, long L, long D, hipStream_t st);
bool col_screen_supported(long n);
// Column pass: same transforms along y; no screen.
// F fields, or (wcnt > 0) F = D * wcnt fields: wavelengths wlo .. wlo + wcnt - 1
// of each direction.  c: columns per workgroup (0 = default for n); e = 32: the Fresnel pass
// holds 32 elements per thread and exchanges through float LDS (256 <= n <= 2048)
hipError_t launch_col(long n, int op, int dir, float2* data, long F, const float2* tf, int W,
                      const float2* tw, hipStream_t st, int c = 0, int e = 0, int wlo = 0, int wcnt = 0);

// Fresnel column pass of F fields (tables tf + f n) that writes their amplitude
// and phase ([F][n][n]) instead of the fields
hipError_t launch_col_amp(long n, float2* data, long F, const float2* tf, const float2* tw, float* amp, float* pha,
                          hipStream_t st);

hipError_t launch_permut(float2* data, long n0, long n1, long nbatch, hipStream_t st);
// mixed-precision row transforms (atsim_fft_mfma.hip): length 2048, radix-16
// stages on the matrix cores (FP16 hi + lo operands, FP32 accumulation);
// nrows a multiple of 2
bool fft_mfma_supported(long n);
hipError_t launch_row_fft_mfma(float2* data, long nrows, int dir, const float2* tw, hipStream_t st);
// out[b][x][y] = in[b][y][x], n a multiple of 32
hipError_t launch_transpose(const float2* in, float2* out, long n, long nbatch, hipStream_t st);
// transforms of any length along one axis (atsim_fft_any.hip): length L through
// transforms of length M, with the chirp and filter of one sign (Bluestein), or
// directly (chirp null, L = M)
struct LinePlan {
    int L, M;
    const float2* chirp;  // [L]
    const float2* filt;   // [M]
    const float2* tw;     // twiddles of M, with the per-stage tables
};
// nrows contiguous rows; in may equal out
hipError_t launch_any_row(const LinePlan& p, int sign, const float2* in, float2* out, long nrows, hipStream_t st);
// the columns of nbatch n0-wide images of p.L rows, in place.  back (the plan
// of sign +1): forward transform, times hx[column] hy[row], inverse transform.
hipError_t launch_any_col(const LinePlan& p, const LinePlan* back, int sign, float2* data, long n0, long nbatch,
                          const double2* hx, const double2* hy, hipStream_t st);
// Fresnel factors of even sides: hx [n0], hy [n1] (with 1 / (n0 n1))
hipError_t launch_any_factor(double2* hx, double2* hy, long n0, long n1, double coeff, hipStream_t st);
// the Fresnel factor between the reference's permut pair, any sides; out != in
hipError_t launch_fresnel_odd(const float2* in, float2* out, long n0, long n1, long nbatch, double coeff,
                              hipStream_t st);
// permut on any sides; out != in
hipError_t launch_permut_any(const float2* in, float2* out, long n0, long n1, long nbatch, hipStream_t st);
hipError_t launch_noise(float2* out, long n, uint64_t seed, uint32_t stream, hipStream_t st);
// the filtered noise spectrum transformed along x (tw with the per-stage tables)
hipError_t launch_synth_row(const float2* noise, float2* out, long size, double f0, double fi, double rlim,
                            const float2* tw, hipStream_t st);
// the structure function's fit of Re and Im: partial holds 8 lag_blocks(size)
// doubles, out receives C1, C2, 1/sqrt(C1), 1/sqrt(C2)
int lag_blocks(long size);
hipError_t launch_lag_fit(const float2* c, long size, double* partial, double* out, hipStream_t st);
// o1 = sc[0] Re c, o2 (may be null) = sc[1] Im c
hipError_t launch_split_scale(const float2* c, float* o1, float* o2, long n, const double* sc, hipStream_t st);
hipError_t launch_strfn(const float* s, long size, long a, long b, int circular, double* partial,
                        int nblocks, hipStream_t st);
hipError_t launch_scale(float* s, long n, double scale, hipStream_t st);
hipError_t launch_cmul(float2* a, const float2* b, long n, long nbatch, hipStream_t st);
hipError_t launch_tf_init(float2* C, long size, double coeff, double fpmaskrad, hipStream_t st);

// the planes a.vr, a.vl of the factored geometric phase, and with vq the
// column passes' phase planes of the nslots layers slot_layer as
// launch_layer_phase makes them; zero_n doubles at zero_p are cleared
hipError_t launch_extract_geometry(const ExtractArgs& a, bool full, hipStream_t st, double* vq = nullptr,
                                   const int* slot_layer = nullptr, int nslots = 0, double* zero_p = nullptr,
                                   long zero_n = 0);
hipError_t launch_extract(const ExtractArgs& a, bool full, hipStream_t st);
// cmax: nfields unsigned, zero on entry (the first round's largest |count|
// per field)
hipError_t launch_block_fix(double* bsum, double* bin, double* ch, unsigned* cmax, const int* field_list,
                            int nfields, int xs, hipStream_t st);
// first-round counts alone (float, per field nb = xs^2), with cmax as above
hipError_t launch_block_counts(const double* bin, float* ch, unsigned* cmax, const int* field_list, int nfields,
                               int xs, hipStream_t st);
hipError_t launch_block_apply(float* pha, const float* dres, const double* bin, const int* field_list,
                              const int* blk, int nfields, int Nout, int xs, hipStream_t st);
// the same update, visiting only the blocks whose largest |r| (rmax, [F][nb]
// float bits from the extraction) lets a count be non-zero, with r from dres
// or made again as rs says; bstart[b]: first output row / column of block b
// (xs + 1 entries)
hipError_t launch_block_apply_sparse(float* pha, const float* dres, const double* bin, const unsigned* rmax,
                                     const int* field_list, const int* bstart, int nfields, int Nout, int xs,
                                     const RemainderSource& rs, hipStream_t st);

hipError_t launch_zero_f64(double* p, long n, hipStream_t st);
// per-field sums of pha, pha^2, amp^2, amp^4 over n pixels of F fields:
// out[F][4]; part holds F * 128 * 4 doubles of partial sums
constexpr long STATS_PART_PER_FIELD = 128 * 4;
hipError_t launch_stats(const float* pha, const float* amp, long F, long n, double* part, double* out,
                        hipStream_t st);
hipError_t launch_layer_screens(const float* masters, const LayerSample* ls, float* out, long N, long M, long L,
                                long D, hipStream_t st);

// surrogate network (atsim_fno.hip)
struct GemmArgs {
    long M, N, K, batch;
    float alpha, beta;
    const float* A;
    long sab, sam, sak;
    const float* B;
    long sbb, sbk, sbn;
    float* C;
    long scb, scm, scn;
    const float* bias;  // per-row bias (or null)
    float* pre;         // pre-activation output with C's strides (or null)
    int act;            // 1: GELU
    int avec, bvec;     // staging modes, set by launch_gemm_bf16
};
hipError_t launch_gemm_bf16(const GemmArgs& g, hipStream_t st);
// 1x1 channel map of [C][nrows][rowlen] images, with (U) the inverse transform
// along x of the rows' retained spectrum added; see k_pointwise
bool pointwise_supported(const float* h, const float* out, const float* pre, const float* U, long Cout, long Cin,
                         long nrows, long rowlen, long K2);
hipError_t launch_pointwise(const float* W, long swm, long swk, int Cout, int Cin, const float* h, float* out,
                            long nrows, int rowlen, const float* U, int K2, const float* F, long sfk, long sfx,
                            const float* bias, float* pre, int act, hipStream_t st, const float* D = nullptr,
                            long dsk = 0, long dsn = 0, int dm = 0, void* T = nullptr,
                            const float* L = nullptr, const float* Lb = nullptr, int cl = 0);
// sizes at which launch_pointwise also transforms out along x (T, BF16
// [Cout][nrows][16 or 32 columns]; table D, dm modes; out may be null), its input
// being L x + Lb of cl channels x in h's place if L is given, and the rest of that
// transform; see k_dft_y
bool point_dft_supported(const void* T, long Cout, long rowlen, long dm, long K2);
hipError_t launch_dft_y(const void* T, const float* Gre, const float* Gim, float* out, long images, int N, int m,
                        hipStream_t st);
// the last block's map and the two projection maps in one pass; see k_tail
// (pointwise_supported sizes for both maps, cout <= 16)
hipError_t launch_tail(const float* W, int C, const float* h, long nrows, int rowlen, const float* U, int K2,
                       const float* F, long sfk, long sfx, const float* bias, const float* Q1, const float* q1b, int H,
                       const float* Q2, const float* q2b, int cout, float* y, hipStream_t st);
// the spectral path: see k_dft2, k_idft_y, k_mix, k_mix_grad (spectral_supported
// sizes only)
bool spectral_supported(const float* h, const float* U, const float* B, const float* O, const float* R, long images,
                        long N, long m, long C, long S);
hipError_t launch_dft2(const float* h, const float* F, long sfk, long sfn, const float* Gre, const float* Gim,
                       float* out, long images, int N, int m, hipStream_t st);
hipError_t launch_idft_y(const float* Gre, const float* Gim, const float* O, float* U, long images, int N, int m,
                         hipStream_t st);
hipError_t launch_mix(const float* R, const float* B, float* out, int C, int S, int nm, bool adj, hipStream_t st);
hipError_t launch_mix_grad(const float* dO, const float* B, float* dR, int C, int S, int nm, hipStream_t st);
bool weight_grad_supported(const float* dy, const float* h, long Cout, long Cin, long SP, long kc);
hipError_t launch_weight_grad(const float* dy, const float* h, float* part, double* bpart, int Cout, int Cin, long SP,
                              int kc, hipStream_t st);
hipError_t launch_add_bias_act(const float* a, const float* b, const float* bias, float* pre, float* y, long C,
                               long P, long n, int gelu, hipStream_t st);
hipError_t launch_gelu_bwd(const float* pre, const float* dy, float* dx, long n, hipStream_t st);
hipError_t launch_bias_grad(const float* dy, double* partial, long S, long C, long P, int nchunk, hipStream_t st);
hipError_t launch_mse(const float* pred, const float* target, float* grad, long n, double* partial, int nblk,
                      hipStream_t st);
hipError_t launch_reduce_batches(const float* part, float* out, long nb, long n, int accumulate, const double* bpart,
                                 float* bout, long nbias, hipStream_t st);
hipError_t launch_nn_pairs(const float* screens, const double* sc, const float* pha, const float* amp, long D, long L,
                           long N, long Stot, long s0, float* x, float* t, double xs, double xl, double cs, double ps,
                           hipStream_t st);
hipError_t launch_nn_unpack(const float* y, const float* x, long L, long S, long P, double xs, double cs, double ps,
                            float* amp, float* pha, hipStream_t st);
constexpr int ADAM_MOST = 32;
struct AdamTensors {
    float* w[ADAM_MOST];
    const float* g[ADAM_MOST];
    float* m[ADAM_MOST];
    float* v[ADAM_MOST];
    long n[ADAM_MOST];
};
hipError_t launch_adam_many(const AdamTensors& p, int count, float lr, float b1, float b2, float eps, float c1,
                            float c2, hipStream_t st);
hipError_t launch_adam(float* w, const float* g, float* m, float* v, long n, float lr, float b1, float b2, float eps,
                       float c1, float c2, hipStream_t st);

}  // namespace atsim
