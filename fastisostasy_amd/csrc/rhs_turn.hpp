// rhs_turn.hpp -- the LV-ELVA attempt in two launches instead of three (or
// five), for any even N = 2^a 3^b 5^c 7^d from 48 to 512.
//
//   kt_col    column pass: applies the previous attempt's accept / reject, then
//             Hartley along y, divide by kappa R, Hartley along y   (g2 -> g1)
//   kt_turn   turns one attempt into the next: Hartley along x of its own and
//             its neighbours' rows, /N^2, corner BC, stage sums, error
//             partials (g1 -> x'), and, on the new state while it is still on
//             chip, the flexure stencil and the forward Hartley transform
//             along x of the next attempt                           (x' -> g2)
//
// A round of launches begins with kt_turn(first), which only does the forward
// part on the current state, and then alternates kt_col, kt_turn.
//
// Why: one domain's attempt is bound by its launches, not by bytes -- each
// costs about 2 us before its first load returns, and every pass then waits
// for descriptor, control block and fields in turn.  The stencil needs two
// halo rows of the new state on each side, exactly one complex line (rows
// 2j, 2j+1 share one), so a block of LO line pairs transforms LO + 2 and the
// inverse pass, the stencil and the forward pass become one launch.
//
// The new state is assumed accepted (about 99 of 100 attempts are).  After a
// rejection the right-hand side is unchanged -- it reads now%w -- and g1 still
// holds it: kt_col does nothing and the next kt_turn repeats the stage sums
// with the smaller step, so no attempt is lost.  An attempt that can end the
// update (t + dt >= tf) skips the forward part.
//
// Arithmetic and reduction orders are those of the three-pass kernels
// (rhs_fast.hip) where those exist, so a domain gives the same bits in a
// small group here and in a large one there.
#pragma once
#include "fft_mix.hpp"
#include "fi_kernels.h"
#include "rhs_common.hpp"

namespace fi {

// lengths of the register kernels of rhs_fast.hip, whose error partials these
// kernels reproduce: one per row pair, reduced over N/8 threads of 8 columns
// (the other lengths: one per row, as the mixed-radix LDS kernels of rhs.hip)
constexpr bool turn_reg8(int n) { return (n & (n - 1)) == 0 || n == 192 || n == 384; }

template <typename T, int N, int LO> struct Turn {
    using PL = MixPlan<N>;
    static constexpr int LINES = LO + 2, ROWS = 2 * LO, WR = ROWS + 4;
    static constexpr int need() {
        int t = LINES * PL::TPL;
        if (t < N) t = N;
        return t;
    }
    static constexpr int THREADS = (need() + 63) / 64 * 64;
    static constexpr int NB = (N / 2 + LO - 1) / LO;                        // blocks per domain
    static constexpr size_t tw_bytes = (size_t)N * sizeof(cplx<T>);
    static constexpr size_t x_bytes = (size_t)WR * N * sizeof(double);      // new state; later f
    static constexpr size_t z_bytes = (size_t)2 * LINES * MixRow<T, N>::PITCH * sizeof(cplx<T>);
    static constexpr size_t m_bytes = (size_t)(2 * ROWS + 2) * N * sizeof(double);
    static constexpr size_t d_bytes = (size_t)ROWS * N * sizeof(double);    // squared errors
    static constexpr size_t zm_bytes = z_bytes > m_bytes ? z_bytes : m_bytes;
    static constexpr size_t lds = tw_bytes + x_bytes + zm_bytes + d_bytes;
    static_assert(N % 2 == 0 && N >= ROWS, "domain smaller than a block");
    static_assert(THREADS <= 1024, "threads per block");
};

// Row spectrum between the two kernels (g2): column tiles of four (the last
// one of two where 4 does not divide N), row pairs inside, the two rows of a
// column side by side.  The column pass reads whole lines of its two columns'
// tile -- in row-major order each of a wave's loads touched 32 cache lines --
// and the row pass stores each row pair in one store.  Together with the
// decision in a wave of its own: one 512^2 domain 18.9 -> 17.0 us per attempt,
// 320^2 17.1 -> 16.5, 256^2 14.4 -> 13.8.
template <int N> __device__ __forceinline__ int turn_at(int row, int c) {
    const int w = N % 4 == 0 ? 4 : (c < N - 2 ? 4 : 2);
    return (c & ~3) * N + (row >> 1) * (2 * w) + (c & 3) * 2 + (row & 1);
}

// The arrays of a member: from the Member's own address for a single domain,
// so that its first loads wait for no descriptor (with the kernel's arguments
// preloaded into scalar registers: one 256^2 domain 13.8 -> 13.4 us per
// attempt, 512^2 17.0 -> 16.5), else from the descriptor.
struct TurnPtrs {
    Ctl *ctl, *ctl_next;
    PhysDev* phys;
    void *g1, *g2, *D, *eta, *kR, *cfull;
    double *corners, *partials, *X0, *X1, *W, *dwdt;
};
template <typename T, int N>
__device__ __forceinline__ TurnPtrs turn_ptrs(const Member* mem, int mi, int solo) {
    TurnPtrs p;
    if (solo) {
        constexpr HotLayout L = hot_layout(N, sizeof(T));
        char* b = (char*)mem;
        p.ctl = (Ctl*)(b + L.ctl); p.ctl_next = (Ctl*)(b + L.ctl_next); p.phys = (PhysDev*)(b + L.phys);
        p.g1 = b + L.g1; p.g2 = b + L.g2; p.D = b + L.D; p.eta = b + L.eta; p.kR = b + L.kR; p.cfull = b + L.cfull;
        p.corners = (double*)(b + L.corners); p.partials = (double*)(b + L.partials);
        p.X0 = (double*)(b + L.X0); p.X1 = (double*)(b + L.X1); p.W = (double*)(b + L.W);
        p.dwdt = (double*)(b + L.dwdt);
    } else {
        const Member& M = mem[mi];
        p.ctl = M.ctl; p.ctl_next = M.ctl_next; p.phys = M.phys;
        p.g1 = M.g1; p.g2 = M.g2; p.D = M.D; p.eta = M.eta; p.kR = M.kR; p.cfull = M.cfull;
        p.corners = M.corners; p.partials = M.partials;
        p.X0 = M.X[0]; p.X1 = M.X[1]; p.W = M.W; p.dwdt = M.dwdt;
    }
    return p;
}

template <typename T, int N, int LO, bool UNI>
__global__ void __launch_bounds__((Turn<T, N, LO>::THREADS)) kt_turn(const Member* __restrict__ mem,
                                                                   const void* __restrict__ twv, int first,
                                                                   int nmem, int solo) {
    using TN = Turn<T, N, LO>;
    using PL = MixPlan<N>;
    constexpr int THREADS = TN::THREADS, LINES = TN::LINES, ROWS = TN::ROWS, WR = TN::WR, TPL = PL::TPL, T0 = PL::T0;
    constexpr bool REG8 = turn_reg8(N);
    int mi, blk;
    xcd_order(TN::NB, nmem, mi, blk);
    const Member& M = mem[mi];
    const TurnPtrs P = turn_ptrs<T, N>(mem, mi, solo);
    const Ctl* const p_ctl = first ? P.ctl : P.ctl_next;
    const void *p_src = P.g1, *p_D = P.D, *p_C = P.cfull, *p_E = P.eta;
    const double *p_cor = P.corners, *x0 = P.X0, *x1p = P.X1, *wW = P.W;
    // a group's pointers in one batch of scalar loads
    if (!solo) scalars_ready(p_ctl, p_src, p_D, p_C, p_E, p_cor, x0, x1p, wW);
    // the control block and physics scalars, in flight while the vector loads
    // are issued
    const kptr<Ctl> c = kview(p_ctl);
    const kptr<PhysDev> ph = kview(P.phys);
    const int status = c->status, cur = c->cur, w_is_x = c->w_is_x, meth = ph->dt_method;
    const double c_dt = c->dt, c_t = c->t, c_tf = c->tf, dt_max = ph->dt_max, spy = ph->sec_per_year;
    extern __shared__ __align__(16) unsigned char smem[];
    cplx<T>* tw_l = (cplx<T>*)smem;
    double* xr = (double*)(smem + TN::tw_bytes);
    unsigned char* zreg = smem + TN::tw_bytes + TN::x_bytes;
    double* dd = (double*)(zreg + TN::zm_bytes);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // rows [row0, row0 + ROWS); where the blocks do not divide the domain the
    // last one reaches back over rows of the one before and leaves them to it
    const int row0 = min(blk * ROWS, N - ROWS), own0 = blk * LO - row0 / 2;
    const int col = tid < N ? tid : N - 1;
    const int lane_line = tid / TPL, t = tid % TPL;
    // global line (row pair) of local line li (0: the halo above), clamped
    auto gline = [&](int li) {
        const int g = row0 / 2 - 1 + li;
        return g < 0 ? 0 : (g > N / 2 - 1 ? N / 2 - 1 : g);
    };
    auto crow = [](int r) { return r < 0 ? 0 : (r > N - 1 ? N - 1 : r); };

    // ---- loads that need no control block, in the order of use
    MixTable<T, N, THREADS> twr(twv, tid);
    cplx<T> v[PL::E];
    constexpr int NW = THREADS / 64, QPW = NW >= 4 ? 1 : (4 + NW - 1) / NW, CPL = (N + 63) / 64;
    double cq[QPW][CPL];
    if (!first) {
        gptr<T> src = gin<T>(p_src);
        const int g = gline(lane_line < LINES ? lane_line : 0), tt = t < T0 ? t : 0;
#pragma unroll
        for (int r = 0; r < PL::R0; ++r)
            v[r] = mk<T>(src[(size_t)(2 * g) * N + tt + T0 * r], src[(size_t)(2 * g + 1) * N + tt + T0 * r]);
        // the four corner sums over the column pass's N terms: quantity q by
        // wave q (waves 4.. repeat 0..3; fewer waves take several), lane-strided
        gptr<double> cp = gin<double>(p_cor);
#pragma unroll
        for (int j = 0; j < QPW; ++j) {
            const int qi = NW >= 4 ? (wave & 3) : wave + NW * j;
#pragma unroll
            for (int k = 0; k < CPL; ++k) {
                const int c = lane + 64 * k;
                cq[j][k] = cp[(size_t)(c < N ? c : N - 1) * 4 + (qi & 3)];
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // rheology and load of the thread's column strip (D rows -1 .. ROWS)
    T dv[ROWS + 2], cv[ROWS], ev[ROWS];
    {
        gptr<T> Dg = gin<T>(p_D), Cg = gin<T>(p_C), Eg = gin<T>(p_E);
#pragma unroll
        for (int r = 0; r < ROWS + 2; ++r) dv[r] = (Dg + (size_t)crow(row0 - 1 + r) * N)[col];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            cv[r] = (Cg + (size_t)(row0 + r) * N)[col];
            ev[r] = (Eg + (size_t)(row0 + r) * N)[col];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    const bool run = status == ST_RUN;
    twr.store(tw_l, tid);
    // kt_col left the decided control block in ctl_next; block 0 makes it
    // current (every block reads ctl_next) and marks this attempt's decision
    // as pending, after its last load
    auto commit = [&](bool pending) {
        if (!first && blk == 0 && tid == 0) {
            copy_ctl(P.ctl, c);
            if (pending) P.ctl->pending = 1;
        }
    };
    if (!run) {
        commit(false);
        return;
    }
    bool ends = false;
    __shared__ double qs[4];
    __shared__ double red[NW];        // largest |x1|, |x2| of each wave
    __shared__ double rg[LO][3][2];   // squared errors of a line's two rows, by lane group
    // Error partials of the block's rows from their squares in dd, by the
    // block's last waves, in the order of the other attempt kernels.  At the
    // register kernels' lengths one entry per row pair: 8 columns per thread,
    // a butterfly over groups of lanes, the groups in order; else one per row:
    // lane l sums columns l, l + 64, ..., then a butterfly.  Only the largest
    // of all the maxima is used: the block's stands for each of its entries.
    constexpr int TP8 = REG8 ? N / 8 : 64, NG8 = (TP8 & (TP8 - 1)) == 0 ? 1 : 3, GL = TP8 / NG8;
    auto block_max = [&]() {
        double am = red[0];
        for (int w = 1; w < NW; ++w) am = fmax(am, red[w]);
        return am;
    };
    auto partials_sum = [&]() {   // after the barrier behind the squares
        if constexpr (REG8) {
            constexpr int W0 = NW - (LO * TP8 + 63) / 64;
            const int q = tid - 64 * W0, l = q / TP8, t8 = q - l * TP8;
            if (wave >= W0) {
                const int lr = l < LO ? l : 0;
                double sa[8], sb[8], s2a = 0.0, s2b = 0.0;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    sa[e] = dd[(2 * lr) * N + t8 + TP8 * e];
                    sb[e] = dd[(2 * lr + 1) * N + t8 + TP8 * e];
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) { s2a += sa[e]; s2b += sb[e]; }
                s2a = lanes_sum<GL>(s2a);
                s2b = lanes_sum<GL>(s2b);
                if (l < LO && t8 % GL == 0) { rg[l][t8 / GL][0] = s2a; rg[l][t8 / GL][1] = s2b; }
            }
        } else {
            for (int r = NW - 1 - wave; r < ROWS; r += NW) {
                double q[CPL], sm = 0.0;
#pragma unroll
                for (int k = 0; k < CPL; ++k) q[k] = dd[r * N + min(lane + 64 * k, N - 1)];
#pragma unroll
                for (int k = 0; k < CPL; ++k) sm += lane + 64 * k < N ? q[k] : 0.0;
                sm = wave_sum(sm);
                if (lane == 0 && r >= 2 * own0) {
                    gmut<double> pp = gout<double>(P.partials) + (size_t)(row0 + r) * 4;
                    pp[0] = block_max();
                    pp[1] = sm;
                }
            }
        }
    };
    auto partials_store = [&]() {   // after another barrier
        if constexpr (REG8) {
            const int l = THREADS - 1 - tid;
            if (l < LO && l >= own0) {
                double s2a = rg[l][0][0], s2b = rg[l][0][1];
#pragma unroll
                for (int w = 1; w < NG8; ++w) { s2a += rg[l][w][0]; s2b += rg[l][w][1]; }
                gmut<double> pp = gout<double>(P.partials) + (size_t)(row0 / 2 + l) * 4;
                pp[0] = block_max();
                pp[1] = s2a + s2b;
            }
        }
    };
    if (first) {
        gptr<double> w = gin<double>(w_is_x ? (cur ? x1p : x0) : wW);
        double wl[WR];
#pragma unroll
        for (int r = 0; r < WR; ++r) wl[r] = (w + (size_t)crow(row0 - 2 + r) * N)[col];
        if (tid < N) {
#pragma unroll
            for (int r = 0; r < WR; ++r) xr[r * N + tid] = wl[r];
        }
        __syncthreads();
    } else {
        const double dt = attempt_dt(meth, c_dt, c_t, c_tf, dt_max);
        ends = !(c_t + dt < c_tf);
        gptr<double> X = gin<double>(cur ? x1p : x0);
        gmut<double> Xn = gout<double>((void*)(cur ? x0 : x1p));
        gmut<double> dw = gout<double>(P.dwdt);
        // the state of the thread's column, consumed after the transform
        double xv[WR];
#pragma unroll
        for (int r = 0; r < WR; ++r) xv[r] = (X + (size_t)(2 * gline(r / 2) + (r & 1)) * N)[col];
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!PL::PLAIN0) __syncthreads();
        const bool on = lane_line < LINES;
        MixRow<T, N> xc((cplx<T>*)zreg, LINES, on ? lane_line : 0);
        mix_fft<T, N>(v, t, on, tw_l, xc, [&]() {
#pragma unroll
            for (int j = 0; j < QPW; ++j) {
                const int qi = NW >= 4 ? (wave & 3) : wave + NW * j;
                double q = 0;
#pragma unroll
                for (int k = 0; k < CPL; ++k) q += lane + 64 * k < N ? cq[j][k] : 0.0;
                q = wave_sum(q);
                if (lane == 0 && qi < 4 && wave < 4) qs[qi] = q;
            }
        });
        // /(nx*ny*1.) (lv_elva.f90:117): an exact multiplication for N = 2^k
        const double S = (double)(float)((double)N * (double)N), rS = 1.0 / S;
        auto scl = [&](double x) {
            if constexpr ((N & (N - 1)) == 0) return x * rS;
            else return over_known(x, S, rS);
        };
        // x(1,1) + x(nx,ny) + x(1,ny) + x(nx,1)  (isos_utils.f90:116)
        const double cc = 0.25 * (scl(qs[0]) + scl(qs[3]) + scl(qs[2]) + scl(qs[1]));
        // k, stage sums and statistics of C cells of the new state: all
        // transform values first, then the arithmetic (the integrator's
        // branch outside the cells), then the stores
        //   h, x: transform value and state;  x2, d2: new state, squared error
        auto cells = [&](auto cc_, const T* h, const double* x, double* kk, double* x2, double* d2, double& a) {
            constexpr int C = decltype(cc_)::value;
#pragma unroll
            for (int q = 0; q < C; ++q) kk[q] = (scl((double)h[q]) - cc) * spy;
            auto sums = [&](auto mc) {
#pragma unroll
                for (int q = 0; q < C; ++q) {
                    double x1;
                    if constexpr (decltype(mc)::value == 3) x2[q] = stage_sums_m<3>(x[q], kk[q], dt, x1);
                    else x2[q] = stage_sums(meth, x[q], kk[q], dt, x1);
                    a = fmax(a, fmax(fabs(x1), fabs(x2[q])));
                    const double d = x2[q] - x1;
                    d2[q] = d * d;
                }
            };
            if (meth == 3) sums(std::integral_constant<int, 3>{});
            else sums(std::integral_constant<int, -1>{});
        };
        T h[WR];
        double kk[WR], x2[WR], d2[WR], ah = 0.0, a = 0.0;
#pragma unroll
        for (int l = 0; l < LINES; ++l) dht_pair(xc.at(l, col), xc.at(l, col ? N - col : 0), h[2 * l], h[2 * l + 1]);
        // (the halo rows' maxima are their own blocks')
        cells(std::integral_constant<int, 2>{}, h, xv, kk, x2, d2, ah);
        cells(std::integral_constant<int, ROWS>{}, h + 2, xv + 2, kk + 2, x2 + 2, d2 + 2, a);
        cells(std::integral_constant<int, 2>{}, h + 2 + ROWS, xv + 2 + ROWS, kk + 2 + ROWS, x2 + 2 + ROWS,
              d2 + 2 + ROWS, ah);
        if (tid < N) {
#pragma unroll
            for (int r = 0; r < WR; ++r) xr[r * N + tid] = x2[r];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) dd[r * N + tid] = d2[r + 2];
        }
        a = wave_max(tid < N ? a : 0.0);
        if (lane == 0) red[wave] = a;
        __syncthreads();
        // the block's own rows to memory
        if (tid < N) {
#pragma unroll
            for (int l = 0; l < LO; ++l)
                if (l >= own0) {
                    const size_t at = (size_t)(row0 + 2 * l) * N + tid;
                    Xn[at] = x2[2 + 2 * l];
                    Xn[at + N] = x2[3 + 2 * l];
                    if (ends) {
                        dw[at] = kk[2 + 2 * l];
                        dw[at + N] = kk[3 + 2 * l];
                    }
                }
        }
        if (ends) {   // no next attempt if this one is accepted; after a rejection the next kt_turn comes back here
            partials_sum();
            __syncthreads();
            partials_store();
            commit(true);
            return;
        }
    }

    // ---- stencil on the thread's column strip (formulas and operand order of
    // rhs_fast.hip's march; one-sided windows at the domain edges)
    const double nu = ph->nu, g = ph->g;
    const double invq = ph->inv_dx2, inv1 = ph->inv_dx, inv2 = ph->inv_2dx;
    const bool top = row0 == 0, bottom = row0 + ROWS == N;
    double* sxx = (double*)zreg;                 // Mxx rows 0 .. ROWS-1
    double* sxy = sxx + ROWS * N;                // Mxy rows -1 .. ROWS
    const int ii = tid < 1 ? 1 : (tid > N - 2 ? N - 2 : tid);
    const bool left = tid == 0, right = tid == N - 1;
    double my[ROWS + 2];
    // distortion: spacing of the strip's own column, and of the column the
    // second x-difference divides by (the first one at the right edge,
    // finite_differences.f90)
    double h1[UNI ? 1 : WR], hq[UNI ? 1 : WR];
    if constexpr (!UNI) {
        gptr<double> dxm = gin<double>(M.dxm);
#pragma unroll
        for (int r = 0; r < WR; ++r) {
            h1[r] = (dxm + (size_t)crow(row0 - 2 + r) * N)[col];
            hq[r] = (dxm + (size_t)crow(row0 - 2 + r) * N)[right ? 0 : col];
        }
    }
    // difference quotients of a in strip row r: centred / one-sided first, second
    auto q1 = [&](double a, bool one, int r) {
        if constexpr (UNI) return a * (one ? inv1 : inv2);
        else return a / (one ? h1[r] : 2 * h1[r]);
    };
    auto qx = [&](double a, int r) {
        if constexpr (UNI) return a * invq;
        else return a / (hq[r] * hq[r]);
    };
    auto qy = [&](double a, int r) {
        if constexpr (UNI) return a * invq;
        else return a / (h1[r] * h1[r]);
    };
    if (tid < N) {
        double wv[WR], wx[WR], wxx[WR];
#pragma unroll
        for (int r = 0; r < WR; ++r) {
            const double* row = xr + r * N;
            const double a = row[ii + 1], b = row[ii], d = row[ii - 1];
            wv[r] = left ? d : (right ? a : b);
            wx[r] = q1((left ? b : a) - (right ? b : d), left || right, r);
            wxx[r] = qx(a - 2 * b + d, r);
        }
#pragma unroll
        for (int m = -1; m <= ROWS; ++m) {
            const int r = m + 2;
            double wa = wv[r + 1], wb = wv[r], wc = wv[r - 1];
            double whi = wx[r + 1], wlo = wx[r - 1];
            bool one = false;
            if (m == 0 && top) { wa = wv[4]; wb = wv[3]; wc = wv[2]; wlo = wx[2]; one = true; }
            if (m == ROWS - 1 && bottom) {
                wa = wv[ROWS + 1]; wb = wv[ROWS]; wc = wv[ROWS - 1]; whi = wx[ROWS + 1];
                one = true;
            }
            const double wyy = qy(wa - 2 * wb + wc, r);
            const double wxy = q1(whi - wlo, one, r);
            const double D = (double)dv[m + 1];
            if (m >= 0 && m < ROWS) sxx[m * N + tid] = -(D * (wxx[r] + nu * wyy));
            my[m + 1] = -(D * (wyy + nu * wxx[r]));
            sxy[(m + 1) * N + tid] = -(D * (1.0 - nu) * wxy);
        }
    }
    __syncthreads();
    T* sf = (T*)xr;   // the state rows have been read
    if (tid < N) {
        double mx[ROWS + 2];
#pragma unroll
        for (int r = 0; r < ROWS + 2; ++r) {
            const double* row = sxy + r * N;
            mx[r] = q1(row[right ? tid : tid + 1] - row[left ? tid : tid - 1], left || right, r + 1);
        }
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            const double* xrow = sxx + j * N;
            const double mxx = qx(xrow[ii + 1] - 2 * xrow[ii] + xrow[ii - 1], j + 2);
            double ya = my[j + 2], yb = my[j + 1], yc = my[j];
            double hi = mx[j + 2], lo = mx[j];
            bool one = false;
            if (j == 0 && top) { ya = my[3]; yb = my[2]; yc = my[1]; lo = mx[1]; one = true; }
            if (j == ROWS - 1 && bottom) {
                ya = my[ROWS]; yb = my[ROWS - 1]; yc = my[ROWS - 2]; hi = mx[ROWS];
                one = true;
            }
            const double myy = qy(ya - 2 * yb + yc, j + 2);
            const double mxyxy = q1(hi - lo, one, j + 2);
            const double p = -(g * (double)cv[j]);
            const double num = p + mxx + 2.0 * mxyxy + myy;
            T f;
            if constexpr (sizeof(T) == 8) f = (T)(num / (2.0 * (double)ev[j]));
            else f = (T)(num * (double)ev[j]);   // mixed: eta holds 1/(2 eta)
            sf[j * N + tid] = f;
        }
    }
    __syncthreads();

    // ---- forward row transform of the block's own lines, the error partials
    // beside it in the waves that have no line
    {
        if (!first) partials_sum();
        const bool on = lane_line < LO;
        const int l = on ? lane_line : 0;
        if (on && t < T0) {
#pragma unroll
            for (int r = 0; r < PL::R0; ++r)
                v[r] = mk<T>(sf[2 * l * N + t + T0 * r], sf[(2 * l + 1) * N + t + T0 * r]);
        }
        MixRow<T, N> xc((cplx<T>*)zreg, LINES, l);
        mix_fft<T, N>(v, t, on, tw_l, xc);
        if (!first) partials_store();
        using V2 = typename vec2<T>::type;
        gmut<V2> dst = gout<V2>(P.g2);
        if (tid < N) {
#pragma unroll
            for (int p = 0; p < LO; ++p) {
                T ha, hb;
                dht_pair(xc.at(p, tid), xc.at(p, tid ? N - tid : 0), ha, hb);
                V2 o;
                o.x = ha;
                o.y = hb;
                if (p >= own0) dst[turn_at<N>(row0 + 2 * p, tid) / 2] = o;
            }
        }
    }
    commit(true);
}

// Column pass.  C complex lines (columns 2j, 2j+1) per block; the last block
// of a domain transforms copies of its last line where C does not divide N/2.
template <typename T, int N, int C> struct TurnCol {
    // waves of transforms, and one more that finds out whether they count
    static constexpr int FFT = (C * MixPlan<N>::TPL + 63) / 64 * 64, THREADS = FFT + 64;
    static_assert(THREADS <= 1024, "threads per block");
    // column blocks of a domain, and one more block that only decides
    static constexpr int NB = (N / 2 + C - 1) / C;
    static constexpr size_t lds = ((size_t)N + 2 * (size_t)MixCol<T, N, C>::SIZE) * sizeof(cplx<T>);
};

template <typename T, int N, int C>
__global__ void __launch_bounds__((TurnCol<T, N, C>::THREADS)) kt_col(const Member* __restrict__ mem,
                                                                    const void* __restrict__ twv,
                                                                    const double2* __restrict__ tw64, int nmem,
                                                                    int solo) {
    using PL = MixPlan<N>;
    constexpr int THREADS = TurnCol<T, N, C>::THREADS, R0 = PL::R0, T0 = PL::T0;
    // a domain's column blocks on one XCD: neighbours share 128-byte lines
    int mi, cblk;
    // -- but spread over all of them while there are fewer than nine blocks for
    // each: the few lines then come through eight L2 caches at once (one 512^2
    // domain 16.5 -> 16.3 us per attempt in XCD order, 6 of 300^2 30.7 -> 28.8, 2 of
    // 512^2 23.1 -> 21.4, but one 256^2 domain, 65 blocks, 13.2 -> 13.3)
    mi = blockIdx.y;
    cblk = blockIdx.x;
    if ((TurnCol<T, N, C>::NB + 1) * nmem >= 72) xcd_order(TurnCol<T, N, C>::NB + 1, nmem, mi, cblk);
    const TurnPtrs P = turn_ptrs<T, N>(mem, mi, solo);
    const void *p_src = P.g2, *p_kr = P.kR;
    const double* const p_part = P.partials;
    if (!solo) scalars_ready(p_src, p_kr, P.ctl, p_part);
    const kptr<Ctl> c = kview(P.ctl);
    const kptr<PhysDev> ph = kview(P.phys);
    if (cblk == TurnCol<T, N, C>::NB) {
        // the whole decision, to ctl_next, which kt_turn reads and makes
        // current; the column blocks only find out whether they have to run
        if ((int)threadIdx.x >= 64) return;
        StepState st = load_state(c);
        const bool pending = c->pending != 0;
        double amax, s2;
        reduce_partials(gin<double>(p_part), turn_reg8(N) ? N / 2 : N, amax, s2);
        if (pending) st = decide_step(st, amax, s2, ph, N);
        if (threadIdx.x == 0) {
            copy_ctl(P.ctl_next, c);
            store_state(P.ctl_next, st);
            P.ctl_next->pending = 0;
            P.ctl_next->skip = 0;
        }
        return;
    }
    const int status = c->status, pend = c->pending;
    const double c_dt = c->dt, c_t = c->t, c_tf = c->tf;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int go_s;
    cplx<T>* tw_l = (cplx<T>*)smem;
    const int tid = threadIdx.x, line = tid % C, t = tid / C;
    const bool decider = __builtin_amdgcn_readfirstlane(tid) >= TurnCol<T, N, C>::FFT;
    const bool live = cblk * C + line < N / 2, on = !decider && t < PL::TPL;
    const int ca = 2 * (live ? cblk * C + line : N / 2 - 1), tt = t < T0 ? t : 0;
    // spectrum, twiddles, kappa R; none depends on the control block
    using V2 = typename vec2<T>::type;
    gptr<T> src = gin<T>(p_src);
    gptr<V2> kR = gin<V2>(p_kr);
    // (row, column pair) -> vector index of a row-major field
    auto vec = [&](int row) { return ((unsigned)row * N + ca) / 2; };
    V2 xk[R0];
    cplx<T> v[PL::E];
    double2 wa, wb;
    // Run?  Yes for the first attempt of a round and after an accepted step
    // that did not end the update; a rejected attempt keeps its right-hand
    // side, which g1 holds.  The last wave finds out from the previous
    // attempt's partials while the others transform (in line it was 1280 of
    // 10800 cycles at N = 256).
    if (decider) {
        constexpr int NP = turn_reg8(N) ? N / 2 : N, PJ = (NP + 63) / 64;
        typedef double d2v __attribute__((ext_vector_type(2)));
        d2v pa[PJ];
        gptr<d2v> part = gin<d2v>(p_part);
        const int lane = tid & 63;
#pragma unroll
        for (int j = 0; j < PJ; ++j) pa[j] = part[(size_t)min(lane + 64 * j, NP - 1) * 2];
        if (status != ST_RUN) return;
        bool go = true;
        if (pend) {
            double amax = 0.0, s2 = 0.0;
#pragma unroll
            for (int j = 0; j < PJ; ++j) {
                const bool in = lane + 64 * j < NP;
                amax = fmax(amax, in ? pa[j].x : 0.0);
                s2 += in ? pa[j].y : 0.0;
            }
            amax = wave_max(amax);
            s2 = wave_sum(s2);
            go = step_goes_on(c_dt, c_t, c_tf, amax, s2, ph, N);
        }
        if (lane == 0) go_s = go;
    } else {
        MixTable<T, N, TurnCol<T, N, C>::FFT> twr(twv, tid);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const int at = turn_at<N>(tt + T0 * r, ca);
            v[r] = mk<T>(src[at], src[at + 2]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R0; ++r) xk[r] = kR[vec(tt + T0 * r)];
        wa = tw64[ca];
        wb = tw64[ca + 1];
        __builtin_amdgcn_sched_barrier(0);
        if (status != ST_RUN) return;
        twr.store(tw_l, tid);
    }
    if constexpr (!PL::PLAIN0) __syncthreads();
    MixCol<T, N, C> xc((cplx<T>*)smem + N, line);
    mix_fft<T, N>(v, t, on, tw_l, xc);
    if (!go_s) return;
    const bool has = on && t < T0;
    if (has) {
        // Hartley values and the spectral divide (lv_elva.f90:115)
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const int k = t + T0 * r;
            T ha, hb;
            dht_pair(xc.get(k), xc.get(k ? N - k : 0), ha, hb);
            v[r] = mk<T>(kdiv(ha, xk[r].x), kdiv(hb, xk[r].y));
        }
    }
    xc.flip();
    mix_fft<T, N>(v, t, on, tw_l, xc);
    if (has && live) {
        gmut<V2> dst = gout<V2>(P.g1);
        gmut<double> cor = gout<double>(P.corners);
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const int k = t + T0 * r;
            T ha, hb;
            dht_pair(xc.get(k), xc.get(k ? N - k : 0), ha, hb);
            V2 o;
            o.x = ha;
            o.y = hb;
            dst[vec(k)] = o;
            // per-column terms of the four corners of the inverse transform
            // (rows 0 and N-1, weights 1 and cas(2 pi col (N-1) / N))
            if ((r == 0 && k == 0) || (r == R0 - 1 && k == N - 1)) {
                const int q = (k == 0) ? 0 : 2;
                const double va = (double)ha, vb = (double)hb;
                cor[(size_t)ca * 4 + q] = va;
                cor[(size_t)ca * 4 + q + 1] = va * (wa.x + wa.y);
                cor[(size_t)(ca + 1) * 4 + q] = vb;
                cor[(size_t)(ca + 1) * 4 + q + 1] = vb * (wb.x + wb.y);
            }
        }
    }
}

// ------------------------------------------------------------------ launchers
// LDS of one workgroup on gfx950; above 64 KiB it is declared to the runtime
template <class K> bool turn_lds_ok(K kern, size_t lds) {
    if (lds > 160 * 1024) return false;
    return lds <= 65536 || hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)lds) == hipSuccess;
}

template <typename T, int N, int LO, bool UNI>
bool turn_rows(const Member* d, int nmem, const RhsShape& s, hipStream_t st, int which) {
    using TN = Turn<T, N, LO>;
    static const bool ok = turn_lds_ok(kt_turn<T, N, LO, UNI>, TN::lds);
    if (!ok || which < 0) return ok;
    const bool first = which == 0;
    launch_k(first ? 0 : 3, kt_turn<T, N, LO, UNI>, dim3(TN::NB, nmem), dim3(TN::THREADS), TN::lds, st, d, s.tw,
             first ? 1 : 0, nmem, s.solo ? 1 : 0);
    prof_turn(LO, -1);
    return true;
}
template <typename T, int N, int C>
bool turn_cols(const Member* d, int nmem, const RhsShape& s, hipStream_t st, int which) {
    using TC = TurnCol<T, N, C>;
    static const bool ok = turn_lds_ok(kt_col<T, N, C>, TC::lds);
    if (!ok || which < 0) return ok;
    launch_k(2, kt_col<T, N, C>, dim3(TC::NB + 1, nmem), dim3(TC::THREADS), TC::lds, st, d, s.tw, s.tw64, nmem,
             s.solo ? 1 : 0);
    prof_turn(-1, C);
    return true;
}

template <typename T, int N>
bool turn_n(const Member* d, int nmem, const RhsShape& s, hipStream_t st, int which) {
    const bool cols = which == 1 || which < 0, rows = which != 1;
    bool ok = true;
    constexpr int CW = MixPlan<N>::TPL <= 120 ? 8 : 4;   // (with the deciding wave, at most 1024 threads)
    if (cols) ok = s.turn_C >= 8 ? turn_cols<T, N, CW>(d, nmem, s, st, which) : turn_cols<T, N, 2>(d, nmem, s, st, which);
    if (rows && ok)
        ok = s.uniform ? (s.turn_LO == 1 ? turn_rows<T, N, 1, true>(d, nmem, s, st, which)
                                         : turn_rows<T, N, 2, true>(d, nmem, s, st, which))
                       : turn_rows<T, N, 2, false>(d, nmem, s, st, which);
    return ok;
}

template <int... Ns>
TurnFn turn_lookup(int n, bool fp64) {
    TurnFn f = nullptr;
    ((n == Ns ? (void)(f = fp64 ? turn_n<double, Ns> : turn_n<float, Ns>) : (void)0), ...);
    return f;
}

}  // namespace fi
