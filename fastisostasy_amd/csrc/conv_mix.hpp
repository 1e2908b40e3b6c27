// conv_mix.hpp -- the convolution's three passes (conv.hip) on the grouped
// register FFT (fft_mix.hpp), for every length M = 2N with N an even
// 2^a 3^b 5^c 7^d from 48 to 512.
//
//   cm_rows_r2c   input rows -> half spectra   (two real rows per complex line)
//   cm_cols       forward, times the kernel spectrum, inverse, crop rows
//   cm_rows_c2r   half spectra -> cropped rows, scale, corner correction
//
// What bounds them: one N = 512 domain moves 25 MB per FP64 convolution, 5 us at
// the copy rate, so launches and each block's own chain of exchanges set the
// time.  The LDS Stockham kernels they replace spent it on run-time divisions,
// two barriers per stage and a twiddle table re-staged by every 2-line block.
// Stages, twiddles and row pairings are those of the kernels they replace, so
// FP32 results are bitwise unchanged.
#pragma once
#include "fft_mix.hpp"
#include "fi_kernels.h"
#include "rhs_common.hpp"

namespace fi {

template <typename T, int M> struct ConvMix {
    using PL = MixPlan<M>;
    static constexpr int N = M / 2, H = N + 1, C0 = N / 2 - 1;   // crop start (convolutions.f90:34-39), N even
    // rows: lines per block for about 256 threads;  columns: measured (us, one
    // domain / 16): FP64 M = 1024 with 4 columns and one exchange buffer 13.1 /
    // 140 (two columns and two buffers: 21.9 / 216, one block per CU); shorter
    // FP64 lines with two columns against four, one buffer: M = 320 5.2 / 5.5 for
    // one domain, 480 6.5 / 7.3, 600 8.5 / 9.5, 768 7.7 / 8.1, 16 of 480 22.5 / 26.0,
    // of 768 39.0 / 47.9 (but 16 of 320 12.4 / 10.6, of 600 37 / 34, and 4 of 768
    // 16.2 / 14.6); FP32 M = 1024 with 8 columns and one buffer 9.3 / 74 (4 and two
    // 9.6 / 110); short FP32 lines with 4 and two buffers 6.2 / 19.3
    static constexpr int LB = PL::TPL >= 128 ? 2 : 256 / PL::TPL > 8 ? 8 : 256 / PL::TPL;
    // (M = 1000 takes 200 threads per line: at most 1024 per block)
    static constexpr int CB = sizeof(T) == 8 ? (M > 768 ? 4 : 2) : M > 512 && 8 * PL::TPL <= 1024 ? 8 : 4;
    static constexpr int TR = (LB * PL::TPL + 63) / 64 * 64, TC = (CB * PL::TPL + 63) / 64 * 64;
    static constexpr size_t lds_rows = ((size_t)M + 2 * (size_t)LB * MixRow<T, M>::PITCH) * sizeof(cplx<T>);
    static constexpr bool ONE = sizeof(T) == 8 || M > 512;
    static constexpr size_t lds_cols = ((size_t)M + (ONE ? 1 : 2) * (size_t)MixCol<T, M, CB>::SIZE) * sizeof(cplx<T>);
    static_assert(TR <= 1024 && TC <= 1024, "threads per block");
    static_assert(PL::R0 % 2 == 0, "the zero half of the input falls on whole elements");
};

// Rows of line j: neighbours (pair = 1), or rows l and l + pair of a block of
// 2 pair rows, as the LDS kernels pair them.
__device__ __forceinline__ void conv_rows(int j, int pair, int& ra, int& rb) {
    ra = (j / pair) * 2 * pair + j % pair;
    rb = ra + pair;
}

template <typename T, int THREADS, int M> __device__ __forceinline__ void conv_twiddles(cplx<T>* tw_l, const void* twv) {
    MixTable<T, M, THREADS>(twv, threadIdx.x).store(tw_l, threadIdx.x);
}

template <typename T, int M>
__global__ void __launch_bounds__((ConvMix<T, M>::TR)) cm_rows_r2c(const Member* __restrict__ mem,
                                                                   const void* __restrict__ twv, int pair) {
    using CM = ConvMix<T, M>;
    using PL = MixPlan<M>;
    constexpr int N = CM::N, H = CM::H, TPL = PL::TPL, R0 = PL::R0, T0 = PL::T0, LB = CM::LB;
    const Member& Mb = mem[blockIdx.y];
    extern __shared__ __align__(16) unsigned char smem[];
    cplx<T>* tw_l = (cplx<T>*)smem;
    const int tid = threadIdx.x, line = tid / TPL, t = tid % TPL, j0 = blockIdx.x * LB;
    const bool on = line < LB && j0 + line < N / 2;
    int ra, rb;
    conv_rows(on ? j0 + line : j0, pair, ra, rb);
    gptr<double> src = gin<double>(Mb.conv_in);
    const int tt = t < T0 ? t : 0;
    // columns >= N of the line are zero: elements R0/2 .. R0-1
    double xa[R0 / 2], xb[R0 / 2];
#pragma unroll
    for (int r = 0; r < R0 / 2; ++r) {
        xa[r] = src[(size_t)ra * N + tt + T0 * r];
        xb[r] = src[(size_t)rb * N + tt + T0 * r];
    }
    conv_twiddles<T, CM::TR, M>(tw_l, twv);
    cplx<T> v[PL::E];
#pragma unroll
    for (int r = 0; r < R0; ++r) v[r] = r < R0 / 2 ? mk<T>((T)xa[r % (R0 / 2)], (T)xb[r % (R0 / 2)]) : mk<T>((T)0, (T)0);
    if constexpr (!PL::PLAIN0) __syncthreads();
    MixRow<T, M> xc(tw_l + M, LB, line < LB ? line : 0);
    mix_fft<T, M>(v, t, on, tw_l, xc);
    // the rows' half spectra k = 0 .. N from Z[k] and Z[M - k]
    gmut<T> dst = gout<T>(Mb.conv_work);
    for (int q = tid; q < LB * H; q += CM::TR) {
        const int l = q / H, k = q - l * H;
        if (j0 + l >= N / 2) break;
        int a, b;
        conv_rows(j0 + l, pair, a, b);
        const cplx<T> zk = xc.at(l, k), zm = xc.at(l, k ? M - k : 0);
        const size_t ia = 2 * ((size_t)a * H + k), ib = 2 * ((size_t)b * H + k);
        dst[ia] = (T)0.5 * (zk.x + zm.x);
        dst[ia + 1] = (T)0.5 * (zk.y - zm.y);
        dst[ib] = (T)0.5 * (zk.y + zm.y);
        dst[ib + 1] = -(T)0.5 * (zk.x - zm.x);
    }
}

template <typename T, int M>
__global__ void __launch_bounds__((ConvMix<T, M>::TC)) cm_cols(const Member* __restrict__ mem,
                                                               const void* __restrict__ twv, int which) {
    using CM = ConvMix<T, M>;
    using PL = MixPlan<M>;
    constexpr int N = CM::N, H = CM::H, R0 = PL::R0, T0 = PL::T0, C = CM::CB;
    // neighbouring columns share 128-byte lines: one XCD's blocks take a run of
    // them (FP64, 16 of 384^2: 1594 -> 1566 us per coupling step; one N = 512 355 ->
    // 342), but blocks fewer than nine per XCD spread over all
    int mi = blockIdx.y, cblk = blockIdx.x;
    if (gridDim.x * gridDim.y >= 72) xcd_order(mi, cblk);
    const Member& Mb = mem[mi];
    extern __shared__ __align__(16) unsigned char smem[];
    cplx<T>* tw_l = (cplx<T>*)smem;
    const int tid = threadIdx.x, line = tid % C, t = tid / C, kx = cblk * C + line;
    const bool on = t < PL::TPL, has = t < T0 && kx < H;
    const int kc = kx < H ? kx : H - 1, tt = t < T0 ? t : 0;
    using V2 = typename vec2<T>::type;
    gptr<V2> w1 = gin<V2>(Mb.conv_work), spec = gin<V2>(which == 0 ? Mb.FGE : which == 1 ? Mb.FGN : Mb.FGV);
    // rows >= N are zero
    V2 x[R0 / 2], sp[R0];
#pragma unroll
    for (int r = 0; r < R0 / 2; ++r) x[r] = w1[(size_t)(tt + T0 * r) * H + kc];
#pragma unroll
    for (int r = 0; r < R0; ++r) sp[r] = spec[(size_t)(tt + T0 * r) * H + kc];
    conv_twiddles<T, CM::TC, M>(tw_l, twv);
    cplx<T> v[PL::E];
#pragma unroll
    for (int r = 0; r < R0; ++r) v[r] = r < R0 / 2 ? mk<T>(x[r % (R0 / 2)].x, x[r % (R0 / 2)].y) : mk<T>((T)0, (T)0);
    if constexpr (!PL::PLAIN0) __syncthreads();
    std::conditional_t<CM::ONE, MixCol1<T, M, C>, MixCol<T, M, C>> xc(tw_l + M, line);
    mix_fft<T, M>(v, t, on, tw_l, xc);
    if (on && t < T0) {
        // times the kernel spectrum, conjugated for the inverse transform
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const cplx<T> p = cmul(mk<T>(sp[r].x, sp[r].y), xc.get(t + T0 * r));
            v[r] = mk<T>(p.x, -p.y);
        }
    }
    xc.flip();
    mix_fft<T, M>(v, t, on, tw_l, xc);
    if (!has) return;
    gmut<V2> w2 = gout<V2>((cplx<T>*)Mb.conv_work + (size_t)N * H);
#pragma unroll
    for (int r = 0; r < R0; ++r) {
        const int k = t + T0 * r, jj = k - CM::C0;
        if (jj >= 0 && jj < N) {
            const cplx<T> z = xc.get(k);
            V2 o;
            o.x = z.x;
            o.y = -z.y;
            w2[(size_t)jj * H + kx] = o;
        }
    }
}

template <typename T, int M>
__global__ void __launch_bounds__((ConvMix<T, M>::TR)) cm_rows_c2r(const Member* __restrict__ mem,
                                                                   const void* __restrict__ twv, int which, int pair) {
    using CM = ConvMix<T, M>;
    using PL = MixPlan<M>;
    constexpr int N = CM::N, H = CM::H, TPL = PL::TPL, R0 = PL::R0, T0 = PL::T0, LB = CM::LB;
    const Member& Mb = mem[blockIdx.y];
    // w_equilibrium is only recomputed for domains that step in this update
    if (which == 2 && Mb.ctl->status != ST_RUN) return;
    extern __shared__ __align__(16) unsigned char smem[];
    cplx<T>* tw_l = (cplx<T>*)smem;
    const int tid = threadIdx.x, line = tid / TPL, t = tid % TPL, j0 = blockIdx.x * LB;
    const bool on = line < LB && j0 + line < N / 2;
    int ra, rb;
    conv_rows(on ? j0 + line : j0, pair, ra, rb);
    using V2 = typename vec2<T>::type;
    gptr<V2> w2 = gin<V2>((const cplx<T>*)Mb.conv_work + (size_t)N * H);
    const int tt = t < T0 ? t : 0;
    V2 xa[R0], xb[R0];
#pragma unroll
    for (int r = 0; r < R0; ++r) {
        const int k = tt + T0 * r, kk = k <= N ? k : M - k;
        xa[r] = w2[(size_t)ra * H + kk];
        xb[r] = w2[(size_t)rb * H + kk];
    }
    // the corner correction of apply_zerobc_at_corners_dp on the full array
    gptr<double> u = gin<double>(Mb.conv_in);
    const double* kc = (which == 0) ? Mb.kc_E : (which == 1) ? Mb.kc_N : Mb.kc_V;
    const double f00 = u[0] * kc[0];
    const double fee = u[(size_t)N * N - 1] * kc[1];
    const double fe0 = u[(size_t)(N - 1) * N] * kc[2];
    const double f0e = u[N - 1] * kc[3];
    const double cc = 0.25 * (f00 + fee + fe0 + f0e);
    conv_twiddles<T, CM::TR, M>(tw_l, twv);
    cplx<T> v[PL::E];
#pragma unroll
    for (int r = 0; r < R0; ++r) {
        const bool up = tt + T0 * r > N;   // Hermitian extension
        const T ya = up ? -xa[r].y : xa[r].y, yb = up ? -xb[r].y : xb[r].y;
        // z = xa + i xb, conjugated
        v[r] = mk<T>(xa[r].x - yb, -(ya + xb[r].x));
    }
    if constexpr (!PL::PLAIN0) __syncthreads();
    MixRow<T, M> xc(tw_l + M, LB, line < LB ? line : 0);
    mix_fft<T, M>(v, t, on, tw_l, xc);
    const double scale = (double)M * (double)M, rscale = 1.0 / scale;
    auto scl = [&](double x) {
        if constexpr ((M & (M - 1)) == 0) return x * rscale;
        else return over_known(x, scale, rscale);
    };
    // (the viscous convolution goes to the state buffer that is free until the first attempt, k_weq)
    gmut<double> out = gout<double>((which == 0) ? Mb.we : (which == 1) ? Mb.dz_ss : Mb.X[Mb.ctl->cur ^ 1]);
    for (int q = tid; q < LB * N; q += CM::TR) {
        const int l = q / N, i = q - l * N;
        if (j0 + l >= N / 2) break;
        int a, b;
        conv_rows(j0 + l, pair, a, b);
        // conj of the FFT: real part = row a, -(imag) = row b
        const cplx<T> z = xc.at(l, i + CM::C0);
        out[(size_t)a * N + i] = scl((double)z.x) - cc;
        out[(size_t)b * N + i] = -scl((double)z.y) - cc;
    }
}

// pair: 1, or the row pairing of the LDS kernels (their lines per block)
template <typename T, int M>
bool conv_mix_m(const Member* d, int nmem, const void* tw, int which, int pair, hipStream_t st) {
    using CM = ConvMix<T, M>;
    constexpr int rb = (CM::N / 2 + CM::LB - 1) / CM::LB, cb = (CM::H + CM::CB - 1) / CM::CB;
    static const bool ok = [] {
        auto one = [](const void* k, size_t lds) {
            return lds <= 65536 || (lds <= 160 * 1024 && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                                            (int)lds) == hipSuccess);
        };
        return one((const void*)cm_rows_r2c<T, M>, CM::lds_rows) && one((const void*)cm_rows_c2r<T, M>, CM::lds_rows) &&
               one((const void*)cm_cols<T, M>, CM::lds_cols);
    }();
    if (!ok) return false;
    hipLaunchKernelGGL((cm_rows_r2c<T, M>), dim3(rb, nmem), dim3(CM::TR), CM::lds_rows, st, d, tw, pair);
    hipLaunchKernelGGL((cm_cols<T, M>), dim3(cb, nmem), dim3(CM::TC), CM::lds_cols, st, d, tw, which);
    hipLaunchKernelGGL((cm_rows_c2r<T, M>), dim3(rb, nmem), dim3(CM::TR), CM::lds_rows, st, d, tw, which, pair);
    return true;
}

template <int... Ns>
ConvFn conv_mix_lookup(int n, bool fp64) {
    ConvFn f = nullptr;
    ((n == Ns ? (void)(f = fp64 ? conv_mix_m<double, 2 * Ns> : conv_mix_m<float, 2 * Ns>) : (void)0), ...);
    return f;
}

}  // namespace fi
