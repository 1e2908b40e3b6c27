// fft_mix.hpp -- Stockham FFT of any even length N = 2^a 3^b 5^c 7^d known at
// compile time, with several butterflies per exchange.
//
// The stages are those of the run-time plan (radices 8, 4, 2, 3, 5, 7 in this
// order, the twiddles read from the same table), grouped: a group of
// consecutive stages whose radices multiply to R <= 16 runs in one thread on
// R elements in registers, and only the groups exchange data through LDS.
// Every butterfly, twiddle product and rounding is the plan's, so results are
// bitwise those of the stage-by-stage kernels; N = 320 (8 x 8 x 5) exchanges
// three times, N = 240 (8 x 2, 3 x 5) twice.
//
// Group g of radix R takes element r of thread t from position t + (N/R) r and
// leaves its output o at position (t / Ns) Ns R + t mod Ns + o Ns, Ns being the
// product of the radices before it.  A line is worked on by TPL threads, the
// most any group has butterflies; the others idle.
#pragma once
#include <type_traits>

#include "fft_reg.hpp"
#include "rhs_common.hpp"

namespace fi {

struct MixStages {
    int nf = 0, rad[16] = {};
    int ng = 0, first[17] = {}, prod[16] = {}, ns[16] = {};
};

// The plan's radices, grouped into the fewest groups of product <= 16; among
// those the grouping whose smallest group is largest (fewest threads per line).
constexpr MixStages mix_stages(int n) {
    MixStages s{};
    const int order[] = {8, 4, 2, 3, 5, 7};
    int m = n;
    for (int r : order)
        while (m % r == 0 && s.nf < 16) { s.rad[s.nf++] = r; m /= r; }
    // best[i]: groups needed from stage i on, and the smallest product among them
    int cnt[17] = {}, low[17] = {}, next[17] = {};
    cnt[s.nf] = 0;
    low[s.nf] = 1 << 20;
    for (int i = s.nf - 1; i >= 0; --i) {
        cnt[i] = 1 << 20;
        int p = 1;
        for (int j = i; j < s.nf; ++j) {
            p *= s.rad[j];
            if (p > 16) break;
            const int c = 1 + cnt[j + 1], l = p < low[j + 1] ? p : low[j + 1];
            if (c < cnt[i] || (c == cnt[i] && l > low[i])) { cnt[i] = c; low[i] = l; next[i] = j + 1; }
        }
    }
    int ns = 1;
    for (int i = 0; i < s.nf; i = next[i]) {
        int p = 1;
        for (int j = i; j < next[i]; ++j) p *= s.rad[j];
        s.first[s.ng] = i;
        s.prod[s.ng] = p;
        s.ns[s.ng] = ns;
        ns *= p;
        ++s.ng;
    }
    s.first[s.ng] = s.nf;
    return s;
}

template <int N> struct MixPlan {
    static constexpr MixStages S = mix_stages(N);
    static constexpr int NG = S.ng;
    static constexpr int R0 = S.prod[0];                  // elements per thread of the first group
    static constexpr int T0 = N / R0;                     // its threads per line
    static constexpr int emax() {
        int e = 0;
        for (int g = 0; g < S.ng; ++g) e = S.prod[g] > e ? S.prod[g] : e;
        return e;
    }
    static constexpr int tpl() {
        int t = 0;
        for (int g = 0; g < S.ng; ++g) t = N / S.prod[g] > t ? N / S.prod[g] : t;
        return t;
    }
    static constexpr int E = emax(), TPL = tpl();
    // the first group reads no twiddles (a single stage): the table need not
    // be published before the first exchange's barrier does so
    static constexpr bool PLAIN0 = S.first[1] - S.first[0] == 1 && S.ng > 1;
    static constexpr int product(int a, int b) { return a >= b ? 1 : S.rad[a] * product(a + 1, b); }
};

// The block's copy of the twiddle table, in 16-byte pieces: loaded early,
// stored to LDS once the loads behind it have been issued.
template <typename T, int N, int THREADS> struct MixTable {
    typedef T V __attribute__((ext_vector_type(16 / sizeof(T))));
    static constexpr int U = 2 * N * (int)sizeof(T) / 16, Q = (U + THREADS - 1) / THREADS;
    static_assert(2 * N * sizeof(T) % 16 == 0, "table of whole pieces");
    V r[Q];
    __device__ __forceinline__ MixTable(const void* tw, int tid) {
        gptr<V> g = gin<V>(tw);
#pragma unroll
        for (int k = 0; k < Q; ++k) r[k] = g[min(tid + THREADS * k, U - 1)];
    }
    __device__ __forceinline__ void store(cplx<T>* tw_l, int tid) const {
#pragma unroll
        for (int k = 0; k < Q; ++k)
            if (tid + THREADS * k < U) ((V*)tw_l)[tid + THREADS * k] = r[k];
    }
};

// Radix-3 butterfly of the N = 3 * 2^k register engine (fft_reg.hpp): the same
// sums in its order, so that both engines give the same bits at those lengths.
template <typename T> __device__ __forceinline__ void bfly3_reg(cplx<T>* v) {
    const T s = (T)0.86602540378443864676, h = (T)-0.5;
    const cplx<T> y0 = v[0], a = cadd(v[1], v[2]), b = csub(v[1], v[2]);
    v[0] = cadd(y0, a);
    v[1] = mk<T>(y0.x + (h * a.x + s * b.y), y0.y + (h * a.y - s * b.x));
    v[2] = mk<T>(y0.x + (h * a.x - s * b.y), y0.y + (h * a.y + s * b.x));
}
template <typename T, int N, int R> __device__ __forceinline__ void mix_bfly(cplx<T>* v) {
    if constexpr (R == 3 && (N == 192 || N == 384)) bfly3_reg<T>(v);
    else bfly<T, R>(v);
}

// Stages S .. E-1 of one group on P = their product elements: x[m] enters as
// the element at distance m N/P, output o leaves in x[o].  kb + KC is the
// butterfly's index modulo NS (kb = 0 and known in the first group).
template <typename T, int N, int S, int E, int NS, int KC, bool FIRST>
__device__ __forceinline__ void mix_group(cplx<T>* x, int kb, const cplx<T>* __restrict__ tw) {
    using PL = MixPlan<N>;
    constexpr int R = PL::S.rad[S], P = PL::product(S, E), P2 = P / R, STEP = N / (NS * R);
    cplx<T> y[P];
#pragma unroll
    for (int u = 0; u < P2; ++u) {
        cplx<T> b[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            b[r] = x[u + P2 * r];
            if constexpr (!(FIRST && KC == 0))
                if (r > 0) b[r] = cmul(b[r], tw[(kb + KC) * r * STEP]);
        }
        mix_bfly<T, N, R>(b);
#pragma unroll
        for (int q = 0; q < R; ++q) y[q * P2 + u] = b[q];
    }
    if constexpr (S + 1 == E) {
#pragma unroll
        for (int q = 0; q < P; ++q) x[q] = y[q];
    } else {
        static_for<0, R>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            mix_group<T, N, S + 1, E, NS * R, KC + q * NS, FIRST>(y + q * P2, kb, tw);
#pragma unroll
            for (int o = 0; o < P2; ++o) x[q + R * o] = y[q * P2 + o];
        });
    }
}

// Exchange in two buffers used in turn (one barrier per exchange); position
// pos of line `line`, padded by one element in eight.
//   rows: line-major;  columns: C lines side by side
template <typename T, int N> struct MixRow {
    static constexpr int PITCH = N + N / 8 + 1;
    cplx<T>* base;
    int size, line, cur;
    __device__ __forceinline__ MixRow(cplx<T>* b, int lines, int l) : base(b), size(lines * PITCH), line(l), cur(0) {}
    __device__ __forceinline__ int addr(int l, int pos) const { return cur * size + l * PITCH + pos + (pos >> 3); }
    __device__ __forceinline__ void put(int pos, cplx<T> v) { base[addr(line, pos)] = v; }
    __device__ __forceinline__ cplx<T> get(int pos) const { return base[addr(line, pos)]; }
    __device__ __forceinline__ cplx<T> at(int l, int pos) const { return base[addr(l, pos)]; }
    __device__ __forceinline__ void flip() { cur ^= 1; }
};
template <typename T, int N, int C> struct MixCol {
    static constexpr int SIZE = (N + N / 8 + 1) * C;
    cplx<T>* base;
    int line, cur;
    __device__ __forceinline__ MixCol(cplx<T>* b, int l) : base(b), line(l), cur(0) {}
    __device__ __forceinline__ int addr(int pos) const { return cur * SIZE + (pos + (pos >> 3)) * C + line; }
    __device__ __forceinline__ void put(int pos, cplx<T> v) { base[addr(pos)] = v; }
    __device__ __forceinline__ cplx<T> get(int pos) const { return base[addr(pos)]; }
    __device__ __forceinline__ void flip() { cur ^= 1; }
};

// The column exchange in one buffer: a second barrier per exchange for half
// the LDS, where that lets more blocks share a CU.
template <typename T, int N, int C> struct MixCol1 {
    static constexpr int SIZE = (N + N / 8 + 1) * C;
    cplx<T>* base;
    int line;
    __device__ __forceinline__ MixCol1(cplx<T>* b, int l) : base(b), line(l) {}
    __device__ __forceinline__ int addr(int pos) const { return (pos + (pos >> 3)) * C + line; }
    __device__ __forceinline__ void put(int pos, cplx<T> v) { base[addr(pos)] = v; }
    __device__ __forceinline__ cplx<T> get(int pos) const { return base[addr(pos)]; }
    __device__ __forceinline__ void flip() { __syncthreads(); }
};

// Forward FFT of the thread's line from group G on.  Entry: v[r] holds element
// t + (N/R) r of the group's input (threads t < N/R).  Exit: the transform lies
// in the exchange's current buffer, published by a barrier; the caller reads
// it and flips the buffers before the next use.  Every thread of the block
// must call (on: the thread has a line).  last() runs before the last barrier.
template <typename T, int N, int G, class X, class F>
__device__ __forceinline__ void mix_fft_from(cplx<T>* v, int t, bool on, const cplx<T>* __restrict__ tw, X& xc,
                                             F&& last) {
    using PL = MixPlan<N>;
    constexpr int R = PL::S.prod[G], NS = PL::S.ns[G], TG = N / R;
    if (on && (TG == PL::TPL || t < TG)) {
        const int k = NS == 1 ? 0 : t % NS;
        mix_group<T, N, PL::S.first[G], PL::S.first[G + 1], NS, 0, G == 0>(v, k, tw);
        const int base = (t / NS) * (NS * R) + k;
#pragma unroll
        for (int o = 0; o < R; ++o) xc.put(base + o * NS, v[o]);
    }
    if constexpr (G + 1 == PL::NG) last();
    __syncthreads();
    if constexpr (G + 1 < PL::NG) {
        constexpr int RN = PL::S.prod[G + 1], TN = N / RN;
        if (on && (TN == PL::TPL || t < TN)) {
#pragma unroll
            for (int r = 0; r < RN; ++r) v[r] = xc.get(t + TN * r);
        }
        xc.flip();
        mix_fft_from<T, N, G + 1>(v, t, on, tw, xc, last);
    }
}
template <typename T, int N, class X, class F>
__device__ __forceinline__ void mix_fft(cplx<T>* v, int t, bool on, const cplx<T>* __restrict__ tw, X& xc, F&& last) {
    mix_fft_from<T, N, 0>(v, t, on, tw, xc, last);
}
template <typename T, int N, class X>
__device__ __forceinline__ void mix_fft(cplx<T>* v, int t, bool on, const cplx<T>* __restrict__ tw, X& xc) {
    mix_fft_from<T, N, 0>(v, t, on, tw, xc, [] {});
}

}  // namespace fi
