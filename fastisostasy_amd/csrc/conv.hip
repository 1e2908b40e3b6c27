// conv.hip -- linear convolution with a precomputed Green's-function spectrum
// (precomputed_fftconvolution / precompute_kernel, convolutions.f90:59-108).
//
// The reference zero-pads to (2N-1)^2 and uses FFTW r2c/c2r; any transform
// size >= 2N-1 gives the same linear convolution, so here M = 2N (smooth
// whenever N is).  Three passes per convolution, half-spectrum layout
// [ky = 0..M-1][kx = 0..N]:
//   c_rows_r2c   rows j < N of the input (rows >= N are zero): two real rows per
//                complex FFT of length M, split into their half spectra
//   c_cols       per kx column: FFT over ky (input rows >= N are zero),
//                multiply by the kernel spectrum, inverse FFT, keep only the
//                N output rows of the crop window [N/2-1, 3N/2-1)
//   c_rows_c2r   two cropped rows per inverse FFT, scale 1/M^2, subtract the
//                corner correction of apply_zerobc_at_corners_dp on the full
//                (2N-1)^2 array, keep the crop columns (the +1-cell shift of
//                convolutions.f90:34-39,89 is kept)
// Convolutions of N = 2^a 3^b 5^c 7^d from 48 to 512 run the same three passes
// on the grouped register FFT (conv_mix.hpp); these LDS Stockham kernels serve
// the other lengths and compute the kernel spectra once per domain.
// The four corners of the full linear convolution are exact products of input
// and kernel corners, so the correction needs no extra pass.
#include "fi_device.hpp"
#include "fi_kernels.h"

namespace fi {

// pass 1: input rows -> half spectra.  src real N x N; dst complex N x (N+1)
// TWL: the twiddle table is held in LDS after the L lines.
template <typename T, bool TWL>
__global__ void __launch_bounds__(512) c_rows_r2c(const Member* __restrict__ mem, FftPlan plan,
                                                  const void* __restrict__ twv, int L, int which_src) {
    const Member& M = mem[blockIdx.y];
    extern __shared__ __align__(16) unsigned char smem[];
    cplx<T>* buf = (cplx<T>*)smem;
    const int N = M.n, Mm = 2 * N, r0 = blockIdx.x * 2 * L;
    const cplx<T>* tw = TWL ? stage_twiddles<T>(buf, Mm, L, twv) : (const cplx<T>*)twv;
    const double* __restrict__ src = M.conv_in;
    (void)which_src;
    const int tid = threadIdx.x, nt = blockDim.x;
    T* bf = (T*)buf;
    // zero padding: rows >= N and columns >= N of the (2N)^2 input
    auto inside = [&](int q) { return q % Mm < N && r0 + q / Mm < N; };
    staged_copy<8>(2 * L * Mm,
                   [&](int q) { return inside(q) ? src[(size_t)(r0 + q / Mm) * N + q % Mm] : src[0]; },
                   [&](int q, double v) {
                       const int mr = q / Mm, i = q % Mm;
                       bf[2 * (i * L + mr % L) + mr / L] = inside(q) ? (T)v : (T)0;
                   });
    __syncthreads();
    lds_fft<T>(buf, plan, L, L, tw);
    cplx<T>* dst = (cplx<T>*)M.conv_work;
    const int H = N + 1;
    for (int q = tid; q < 2 * L * H; q += nt) {
        const int mr = q / H, k = q % H;
        const int row = r0 + mr;
        if (row >= N) continue;
        const int l = mr % L, part = mr / L;
        const cplx<T> zk = buf[k * L + l], zm = buf[((Mm - k) % Mm) * L + l];
        cplx<T> v;
        if (part == 0) v = mk<T>((T)0.5 * (zk.x + zm.x), (T)0.5 * (zk.y - zm.y));
        else v = mk<T>((T)0.5 * (zk.y + zm.y), -(T)0.5 * (zk.x - zm.x));
        dst[(size_t)row * H + k] = v;
    }
}

// pass 2: columns.  mode 0 = spectrum of a kernel (write all M rows to spec);
// mode 1 = convolve with spec (which: 0 elastic, 1 sea surface, 2 viscous) and keep crop rows.
template <typename T>
__global__ void __launch_bounds__(512) c_cols(const Member* __restrict__ mem, FftPlan plan,
                                              const void* __restrict__ twv, int C, int mode, int which) {
    const Member& M = mem[blockIdx.y];
    extern __shared__ __align__(16) unsigned char smem[];
    cplx<T>* buf = (cplx<T>*)smem;
    const int N = M.n, Mm = 2 * N, H = N + 1;
    const int k0 = blockIdx.x * C;
    const cplx<T>* tw = stage_twiddles<T>(buf, Mm, C, twv);   // the host sizes C to leave room
    const cplx<T>* __restrict__ w1 = (const cplx<T>*)M.conv_work;
    const int tid = threadIdx.x, nt = blockDim.x;
    auto inside = [&](int q) { return q / C < N && k0 + q % C < H; };
    staged_copy<8>(Mm * C, [&](int q) { return inside(q) ? w1[(size_t)(q / C) * H + k0 + q % C] : w1[0]; },
                   [&](int q, cplx<T> v) { buf[q] = inside(q) ? v : mk<T>((T)0, (T)0); });
    __syncthreads();
    lds_fft<T>(buf, plan, C, C, tw);
    cplx<T>* spec = (cplx<T>*)(which == 0 ? M.FGE : which == 1 ? M.FGN : M.FGV);
    if (mode == 0) {
        for (int q = tid; q < Mm * C; q += nt) {
            const int r = q / C, l = q % C;
            const int kx = k0 + l;
            if (kx < H) spec[(size_t)r * H + kx] = buf[r * C + l];
        }
        return;
    }
    // product with the kernel spectrum, then conjugate for the inverse FFT
    staged_copy<8>(Mm * C,
                   [&](int q) { return k0 + q % C < H ? spec[(size_t)(q / C) * H + k0 + q % C] : spec[0]; },
                   [&](int q, cplx<T> sv) {
                       cplx<T> v = mk<T>((T)0, (T)0);
                       if (k0 + q % C < H) v = cmul(sv, buf[q]);
                       v.y = -v.y;
                       buf[q] = v;
                   });
    __syncthreads();
    lds_fft<T>(buf, plan, C, C, tw);
    cplx<T>* w2 = (cplx<T>*)M.conv_work + (size_t)N * H;
    const int c0 = N / 2 - 1 + (N % 2);   // 0-based crop start (convolutions.f90:34-39)
    for (int q = tid; q < N * C; q += nt) {
        const int jj = q / C, l = q % C;
        const int kx = k0 + l;
        if (kx >= H) continue;
        cplx<T> v = buf[(jj + c0) * C + l];
        v.y = -v.y;
        w2[(size_t)jj * H + kx] = v;
    }
}

// pass 3: cropped rows back to real space, scale, corner correction, crop.
template <typename T, bool TWL>
__global__ void __launch_bounds__(512) c_rows_c2r(const Member* __restrict__ mem, FftPlan plan,
                                                  const void* __restrict__ twv, int L, int which) {
    const Member& M = mem[blockIdx.y];
    // w_equilibrium is only recomputed for domains that step in this update
    if (which == 2 && M.ctl->status != ST_RUN) return;
    extern __shared__ __align__(16) unsigned char smem[];
    cplx<T>* buf = (cplx<T>*)smem;
    __shared__ double corr;
    const int N = M.n, Mm = 2 * N, H = N + 1, r0 = blockIdx.x * 2 * L;
    const cplx<T>* tw = TWL ? stage_twiddles<T>(buf, Mm, L, twv) : (const cplx<T>*)twv;
    const cplx<T>* __restrict__ w2 = (const cplx<T>*)M.conv_work + (size_t)N * H;
    const int tid = threadIdx.x, nt = blockDim.x;
    if (tid == 0) {
        const double* u = M.conv_in;
        const double* kc = (which == 0) ? M.kc_E : (which == 1) ? M.kc_N : M.kc_V;
        const double f00 = u[0] * kc[0];
        const double fee = u[(size_t)N * N - 1] * kc[1];
        const double fe0 = u[(size_t)(N - 1) * N] * kc[2];
        const double f0e = u[N - 1] * kc[3];
        corr = 0.25 * (f00 + fee + fe0 + f0e);
    }
    // Hermitian extension of two half-spectrum rows, conjugated for the inverse
    struct Pair { cplx<T> a, b; };
    staged_copy<4>(L * Mm,
                   [&](int q) {
                       const int l = q / Mm, k = q % Mm, kk = k <= N ? k : Mm - k;
                       return Pair{w2[(size_t)(r0 + l) * H + kk], w2[(size_t)(r0 + L + l) * H + kk]};
                   },
                   [&](int q, Pair p) {
                       const int l = q / Mm, k = q % Mm;
                       cplx<T> xa = p.a, xb = p.b;
                       if (k > N) { xa.y = -xa.y; xb.y = -xb.y; }
                       // z = xa + i xb, conjugated
                       buf[k * L + l] = mk<T>(xa.x - xb.y, -(xa.y + xb.x));
                   });
    __syncthreads();
    lds_fft<T>(buf, plan, L, L, tw);
    const double scale = (double)Mm * (double)Mm;
    const double cc = corr;
    const int c0 = N / 2 - 1 + (N % 2);
    // (the viscous convolution goes to the state buffer that is free until the first attempt, k_weq)
    double* out = (which == 0) ? M.we : (which == 1) ? M.dz_ss : M.X[M.ctl->cur ^ 1];
    for (int q = tid; q < 2 * L * N; q += nt) {
        const int mr = q / N, i = q % N;
        const int l = mr % L, part = mr / L;
        const cplx<T> z = buf[(i + c0) * L + l];
        // conj of the FFT: real part = row a, -(imag) = row b
        const double v = part ? -(double)z.y : (double)z.x;
        out[(size_t)(r0 + mr) * N + i] = v / scale - cc;
    }
}

template <typename T>
static size_t lbytes(int m, int lines) { return (size_t)m * lines * sizeof(cplx<T>); }

template <typename T>
static void rows_r2c(const Member* d_mem, int nmem, const ConvShape& s, int which, hipStream_t st) {
    const dim3 g((s.n + 2 * s.Lr - 1) / (2 * s.Lr), nmem), b(s.threads_row);
    if (s.rows_twl)
        hipLaunchKernelGGL((c_rows_r2c<T, true>), g, b, lbytes<T>(s.m, s.Lr + 1), st, d_mem, s.plan, s.tw, s.Lr, which);
    else
        hipLaunchKernelGGL((c_rows_r2c<T, false>), g, b, lbytes<T>(s.m, s.Lr), st, d_mem, s.plan, s.tw, s.Lr, which);
}

// lengths by translation unit
ConvFn conv_part0(int, bool);
ConvFn conv_part1(int, bool);
ConvFn conv_part2(int, bool);
ConvFn conv_part3(int, bool);
ConvFn conv_part4(int, bool);
ConvFn conv_part5(int, bool);
ConvFn conv_part6(int, bool);
ConvFn conv_part7(int, bool);
ConvFn conv_find(int n, bool fp64) {
    using Part = ConvFn (*)(int, bool);
    constexpr Part parts[] = {conv_part0, conv_part1, conv_part2, conv_part3,
                              conv_part4, conv_part5, conv_part6, conv_part7};
    for (Part p : parts)
        if (ConvFn f = p(n, fp64)) return f;
    return nullptr;
}

template <typename T>
static void conv_t(const Member* d_mem, int nmem, const ConvShape& s, int which, hipStream_t st) {
    const bool grouped = s.mix && s.mix(d_mem, nmem, s.tw, which, s.pair, st);
    prof_conv(grouped ? 1 : 0);
    if (grouped) return;
    const int n = s.n, H = n + 1;
    rows_r2c<T>(d_mem, nmem, s, which, st);
    hipLaunchKernelGGL(c_cols<T>, dim3((H + s.Cc - 1) / s.Cc, nmem), dim3(s.threads_col), lbytes<T>(s.m, s.Cc + 1), st,
                       d_mem, s.plan, s.tw, s.Cc, 1, which);
    const dim3 g(n / (2 * s.Lr), nmem), b(s.threads_row);
    if (s.rows_twl)
        hipLaunchKernelGGL((c_rows_c2r<T, true>), g, b, lbytes<T>(s.m, s.Lr + 1), st, d_mem, s.plan, s.tw, s.Lr, which);
    else
        hipLaunchKernelGGL((c_rows_c2r<T, false>), g, b, lbytes<T>(s.m, s.Lr), st, d_mem, s.plan, s.tw, s.Lr, which);
}

void launch_convolution(const Member* d_mem, int nmem, const ConvShape& s, int which, hipStream_t st) {
    if (s.fp64) conv_t<double>(d_mem, nmem, s, which, st);
    else conv_t<float>(d_mem, nmem, s, which, st);
}

// Kernel spectrum: the kernel must already be in conv_in.
template <typename T>
static void spec_t(const Member* d_mem, int nmem, const ConvShape& s, int which, hipStream_t st) {
    const int n = s.n, H = n + 1;
    rows_r2c<T>(d_mem, nmem, s, which, st);
    hipLaunchKernelGGL(c_cols<T>, dim3((H + s.Cc - 1) / s.Cc, nmem), dim3(s.threads_col),
                       lbytes<T>(s.m, s.Cc + 1), st, d_mem, s.plan, s.tw, s.Cc, 0, which);
}

void launch_kernel_spectrum(const Member* d_mem, int nmem, const ConvShape& s, int which,
                            const double* d_kernel, hipStream_t st) {
    (void)d_kernel;
    if (s.fp64) spec_t<double>(d_mem, nmem, s, which, st);
    else spec_t<float>(d_mem, nmem, s, which, st);
}

}  // namespace fi
