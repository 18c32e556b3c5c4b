// sse_lines.h -- sum-factorised V, V' and line derivatives with a line of nodes per thread.
//
// A column (one variable of one element) is one LDS array of padded tensor-grid positions
// X(a1, a2[, a3]). Every stage of V, V' and of a derivative along a collapsed direction acts
// on lines of the grid: a thread reads its line's N1 values into registers, applies an
// N1 x N1 matrix and writes the N1 results back in place. With one thread per output point
// instead (SumFact of sse_tensor.h) each multiply-add reads one LDS value, which is what
// bounded those kernels: a CU issues four times as many FP64 multiply-adds as LDS reads.
// Here a line costs 2 N1 LDS accesses for N1^2 multiply-adds, and the matrices come through
// the scalar cache where they are the same for all lanes:
//   stage 3 (A[a1, b1]) and the derivatives D1_l: always;
//   stage 2 (B[a2, b1, b2]): b1 is uniform over a wavefront (the wavefronts share out b1,
//     the lanes are (column, a3));
//   stage 1 (C[a3, b1, b2, b3]): a lane per (column, (b1, b2)) reads its entries of C from an
//     LDS copy with (b1, b2) fastest (lanes of different columns read the same word). The lanes
//     go by falling number of modes, so that the entries of one b3 belong to the first ones
//     and the copy holds no padding.
// R and R' ride on the same lines (FaceTables): the value at the end of a line is one row of N1
// uniform weights.
// In place, the modal position (b1, b2, b3) takes the place of (a1, a2, a3).
// The strides of a column are the ones with the fewest LDS bank conflicts over the lane
// patterns of all stages (counted for each N1 on the 64 banks; a fifth to a quarter fewer
// cycles than the next odd strides).
#pragma once

#include <hip/hip_runtime.h>

#include "sse_tensor.h"

namespace sse {

// a read-only table that no kernel writes: loads with a wave-uniform index go to the scalar unit
typedef const __attribute__((address_space(4))) double* UniformTable;
__device__ __forceinline__ UniformTable uniform_table(const double* p) { return (UniformTable)(uintptr_t)p; }
// the same table, but the compiler does not know it: its entries are loaded again where they are
// used instead of being kept (spilled) in scalar registers from an earlier stage
__device__ __forceinline__ UniformTable reload(UniformTable p) {
    uintptr_t v = (uintptr_t)p;
    asm volatile("" : "+s"(v));
    return (UniformTable)v;
}

template <int ELEM, int P>
struct LineGrid {
    using Sh = Shape<ELEM, P>;
    static constexpr int D = Sh::D, N1 = Sh::N1, NP = Sh::NP, NQ = Sh::NQ;
    static constexpr bool TET = ELEM == ELEM_TET;
    static constexpr int N2 = TET ? N1 * N1 : N1;  // lines per direction
    static constexpr int S2 = !TET ? 1 : N1 == 4 ? 5 : N1;
    static constexpr int S1 = !TET ? (N1 | 1) : N1 == 3 ? 11 : N1 == 4 ? 24 : N1 == 5 ? 26 : 37;
    static constexpr int NX = !TET ? N1 * S1 : N1 == 3 ? 41 : N1 == 4 ? 100 : N1 == 5 ? 153 : 228;  // of one column
    static_assert(NX > (N1 - 1) * (S1 + (TET ? S2 + 1 : 1)), "a column holds its grid");
    // lanes of stage 1: (b1, b2), b1 + b2 <= P, on the Tet; b1 on the Tri
    static constexpr int NM = TET ? (P + 1) * (P + 2) / 2 : N1;

    // line t of direction l: first position and stride in X; first node and stride in the
    // unpadded node numbering (last index fastest)
    template <int L>
    __device__ static int base(int t) {
        if constexpr (!TET) return L == 0 ? t : t * S1;
        const int hi = t / N1, lo = t - hi * N1;
        return L == 0 ? hi * S2 + lo : L == 1 ? hi * S1 + lo : hi * S1 + lo * S2;
    }
    template <int L>
    __host__ __device__ static constexpr int stride() {
        return !TET ? (L == 0 ? S1 : 1) : (L == 0 ? S1 : L == 1 ? S2 : 1);
    }
    template <int L>
    __device__ static int node(int t) {
        if constexpr (!TET) return L == 0 ? t : t * N1;
        const int hi = t / N1, lo = t - hi * N1;
        return L == 0 ? t : L == 1 ? hi * N1 * N1 + lo : t * N1;
    }
    template <int L>
    __host__ __device__ static constexpr int node_stride() {
        return !TET ? (L == 0 ? N1 : 1) : (L == 0 ? N1 * N1 : L == 1 ? N1 : 1);
    }
    __host__ __device__ static constexpr int position(int i) {  // of node i in X
        return TET ? (i / (N1 * N1)) * S1 + ((i / N1) % N1) * S2 + i % N1 : (i / N1) * S1 + i % N1;
    }
};

// y[a] = sum_b M[a N1 + b] x[b] (ROW) or sum_b M[b N1 + a] x[b]; M uniform
template <int N1, bool ROW>
__device__ __forceinline__ void line_apply(UniformTable M, const double* x, double* y) {
#pragma unroll
    for (int a = 0; a < N1; ++a) y[a] = 0.0;
#pragma unroll
    for (int b = 0; b < N1; ++b)
#pragma unroll
        for (int a = 0; a < N1; ++a) y[a] += M[ROW ? a * N1 + b : b * N1 + a] * x[b];
}

template <int N1, int ST>
__device__ __forceinline__ void line_load(const double* X, double* x) {
#pragma unroll
    for (int a = 0; a < N1; ++a) x[a] = X[a * ST];
}
template <int N1, int ST>
__device__ __forceinline__ void line_store(double* X, const double* x) {
#pragma unroll
    for (int a = 0; a < N1; ++a) X[a * ST] = x[a];
}

template <int ELEM, int P>
struct LineFact {
    using G = LineGrid<ELEM, P>;
    static constexpr int N1 = G::N1, NM = G::NM;

    struct Modes {  // of a stage-1 lane
        int off, base, lim;  // first mode number, position of the line in X, last b of the line
    };
    __device__ static Modes modes(const int* mode, int m) {
        const int c = mode[m], b1 = (c >> 16) & 0xff, b2 = c >> 24;
        return G::TET ? Modes{c & 0xffff, b1 * G::S1 + b2 * G::S2, P - b1 - b2} : Modes{c & 0xffff, b1 * G::S1, P - b1};
    }
    // LDS doubles of the stage-1 tables, and their copy (all nt threads; a barrier must follow)
    static constexpr int NT1 = N1 * G::NP;
    __device__ static void stage_tables(const LineTables& lt, double* dst, int t, int nt) {
        for (int i = t; i < NT1; i += nt) dst[i] = lt.F1[i];
    }
    // lanes with a mode b, and the first table entry of b
    __host__ __device__ static constexpr int lanes(int b) {
        return G::TET ? (P - b + 1) * (P - b + 2) / 2 : P - b + 1;
    }
    __host__ __device__ static constexpr int first(int b) {
        int o = 0;
        for (int q = 0; q < b; ++q) o += N1 * lanes(q);
        return o;
    }
    // stage 1 of V for one line: modal values x (zero past lim) to N1 values
    __device__ static void up1(const double* F1, int m, const double* x, double* y) {
#pragma unroll
        for (int a = 0; a < N1; ++a) y[a] = 0.0;
#pragma unroll
        for (int b = 0; b < N1; ++b)
            if (m < lanes(b)) {
#pragma unroll
                for (int a = 0; a < N1; ++a) y[a] += F1[first(b) + a * lanes(b) + m] * x[b];
            }
    }
    // stage 1 of V': N1 values to the line's modal values (zero past its last)
    __device__ static void down1(const double* F1, int m, const double* x, double* y) {
#pragma unroll
        for (int b = 0; b < N1; ++b) {
            y[b] = 0.0;
            if (m < lanes(b)) {
#pragma unroll
                for (int a = 0; a < N1; ++a) y[b] += F1[first(b) + a * lanes(b) + m] * x[a];
            }
        }
    }
    // stage 2 (Tet only) of V and of V' for NCOL columns CS apart, in place; B[a2, b1, b2] =
    // VB[a2 + N1 (b1 + N1 b2)]. All TS threads call; no barrier inside.
    template <int NCOL, int TS, int CS = 1>
    __device__ static void up2(UniformTable B, double* X) {
        if constexpr (G::TET) {
            const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
            // b1 back and forth over the wavefronts: the work of b1 falls with it
            for (int q = 0, b1 = wave; b1 <= P; ++q, b1 = (q & 1) ? (q + 1) * (TS / 64) - 1 - wave : q * (TS / 64) + wave)
                for (int t = lane; t < NCOL * N1; t += 64) {
                    const int col = t / N1, a3 = t - col * N1;
                    double* L = X + col * CS * G::NX + b1 * G::S1 + a3;
                    double y[N1];
#pragma unroll
                    for (int a = 0; a < N1; ++a) y[a] = 0.0;
#pragma unroll
                    for (int b2 = 0; b2 <= P; ++b2) {
                        if (b2 > P - b1) break;
                        const double x = L[b2 * G::S2];
#pragma unroll
                        for (int a = 0; a < N1; ++a) y[a] += B[a + N1 * (b1 + N1 * b2)] * x;
                    }
                    line_store<N1, G::S2>(L, y);
                }
        }
    }
    // NSUM: each input is the sum of NSUM consecutive columns
    template <int NCOL, int TS, int CS = 1, int NSUM = 1>
    __device__ static void down2(UniformTable B, double* X) {
        if constexpr (G::TET) {
            const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
            // b1 back and forth over the wavefronts: the work of b1 falls with it
            for (int q = 0, b1 = wave; b1 <= P; ++q, b1 = (q & 1) ? (q + 1) * (TS / 64) - 1 - wave : q * (TS / 64) + wave)
                for (int t = lane; t < NCOL * N1; t += 64) {
                    const int col = t / N1, a3 = t - col * N1;
                    double* L = X + col * CS * G::NX + b1 * G::S1 + a3;
                    double x[N1];
                    line_load<N1, G::S2>(L, x);
#pragma unroll
                    for (int q = 1; q < NSUM; ++q)
#pragma unroll
                        for (int a = 0; a < N1; ++a) x[a] += L[q * G::NX + a * G::S2];
#pragma unroll
                    for (int b2 = 0; b2 <= P; ++b2) {
                        if (b2 > P - b1) break;
                        double y = 0.0;
#pragma unroll
                        for (int a = 0; a < N1; ++a) y += B[a + N1 * (b1 + N1 * b2)] * x[a];
                        L[b2 * G::S2] = y;
                    }
                }
        }
    }
};

// e[f N2 + line] = end value of this line (x, direction L) on every face of direction L
template <int ELEM, int P, int L>
__device__ __forceinline__ void line_ends(const FaceTables& ft, const double* x, int line, double* e) {
    using G = LineGrid<ELEM, P>;
    constexpr int N1 = G::N1;
    const UniformTable w = uniform_table(ft.w);
#pragma unroll
    for (int f = 0; f < G::Sh::NFAC; ++f) {
        if (ft.dir[f] != L) continue;
        double s = 0.0;
#pragma unroll
        for (int a = 0; a < N1; ++a) s += w[f * N1 + a] * x[a];
        e[f * G::N2 + line] = s;
    }
}

// r[a] += w_f[a] s[f N2 + line] over the faces of direction L (the transpose)
template <int ELEM, int P, int L>
__device__ __forceinline__ void line_ends_t(const FaceTables& ft, const double* s, int line, double* r) {
    using G = LineGrid<ELEM, P>;
    constexpr int N1 = G::N1;
    const UniformTable w = uniform_table(ft.w);
#pragma unroll
    for (int f = 0; f < G::Sh::NFAC; ++f) {
        if (ft.dir[f] != L) continue;
        const double v = s[f * G::N2 + line];
#pragma unroll
        for (int a = 0; a < N1; ++a) r[a] += w[f * N1 + a] * v;
    }
}

// Line j0 of N1 facet values (same first face index) of a face of kind 1, in place: P_f' t
template <int N1>
__device__ __forceinline__ void face_line_t(UniformTable Pf, double* t) {
    double x[N1], y[N1];
    line_load<N1, 1>(t, x);
    line_apply<N1, false>(Pf, x, y);
    line_store<N1, 1>(t, y);
}

// acc[c] += row j of M (TR: of M') times column c of x (columns XS apart). The entries of a row
// are requested together.
template <int ELEM, int P, int NCV, int XS, bool TR>
__device__ __forceinline__ void face_row(const FaceTables& ft, int j, const double* x, double* acc) {
    using G = LineGrid<ELEM, P>;
    constexpr int N1 = G::N1, N2 = G::N2, NF = G::Sh::NF;
    if (ft.general) {
        const int* idx = TR ? ft.mt_idx : ft.m_idx;
        const double* val = TR ? ft.mt_val : ft.m_val;
        const int width = TR ? ft.mt_w : ft.m_w;
        for (int w = 0; w < width; ++w) {
            const int i = idx[w * NF + j];
            if (i < 0) break;
#pragma unroll
            for (int c = 0; c < NCV; ++c) acc[c] += val[w * NF + j] * x[c * XS + i];
        }
        return;
    }
    const int f = j / N2;
    if (G::TET && (f == 0 ? ft.kind[0] : f == 1 ? ft.kind[1] : f == 2 ? ft.kind[2] : ft.kind[3])) {
        const int c2 = j % N1, j0 = j - c2;
        const double* Pf = ft.P + f * N1 * N1 + (TR ? c2 : c2 * N1);
        double pv[N1];
#pragma unroll
        for (int b = 0; b < N1; ++b) pv[b] = Pf[TR ? b * N1 : b];
#pragma unroll
        for (int b = 0; b < N1; ++b)
#pragma unroll
            for (int c = 0; c < NCV; ++c) acc[c] += pv[b] * x[c * XS + j0 + b];
    } else {
#pragma unroll
        for (int c = 0; c < NCV; ++c) acc[c] += x[c * XS + j];
    }
}

// in place, the facet values t of NCOL columns (NF apart) to M' t; the caller's barrier follows.
// tt: the thread among the TS (the whole workgroup calls: general has a barrier inside).
// The lines of the faces of kind 1 go to the last threads of the workgroup (the first ones have
// stage-1 lines of V in the same phase).
template <int ELEM, int P, int NCOL, int TS>
__device__ __forceinline__ void face_transpose(const FaceTables& ft, double* t, int tt) {
    using G = LineGrid<ELEM, P>;
    constexpr int N1 = G::N1, N2 = G::N2, NF = G::Sh::NF;
    if (ft.general) {
        constexpr int IT = (NCOL * NF + TS - 1) / TS;
        double v[IT];
#pragma unroll
        for (int q = 0; q < IT; ++q) {
            const int o = tt + q * TS, c = o / NF;
            v[q] = 0.0;
            if (o < NCOL * NF) face_row<ELEM, P, 1, NF, true>(ft, o - c * NF, t + c * NF, v + q);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < IT; ++q)
            if (tt + q * TS < NCOL * NF) t[tt + q * TS] = v[q];
    } else if constexpr (G::TET) {
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if (ft.kind[f] == 0) continue;
            const UniformTable Pf = uniform_table(ft.P) + f * N1 * N1;
            for (int o = TS - 1 - tt; o < NCOL * N1; o += TS) {
                const int c = o / N1;
                face_line_t<N1>(Pf, t + c * NF + f * N2 + (o - c * N1) * N1);
            }
        }
    }
}

// ends of line `line` of every direction but the first, of one column X
template <int ELEM, int P>
__device__ __forceinline__ void other_line_ends(const FaceTables& ft, const double* X, int line, double* e) {
    using G = LineGrid<ELEM, P>;
    constexpr int N1 = G::N1;
    double x[N1];
    line_load<N1, G::template stride<1>()>(X + G::template base<1>(line), x);
    line_ends<ELEM, P, 1>(ft, x, line, e);
    if constexpr (G::TET) {
        line_load<N1, G::template stride<2>()>(X + G::template base<2>(line), x);
        line_ends<ELEM, P, 2>(ft, x, line, e);
    }
}

// Elements and threads of a workgroup of the Euler kernels that only transform: all lines of E elements in one go with few idle threads, and for the Tet enough
// columns to fill the lanes of stage 2 (E NC N1 of 64)
template <int ELEM, int P>
struct EulerTune;
#define SSE_EULER_TUNE(E_, PP, e, ts) \
    template <>                       \
    struct EulerTune<E_, PP> {        \
        static constexpr int E = e, TS = ts; \
    };
SSE_EULER_TUNE(ELEM_TRI, 2, 5, 64)
SSE_EULER_TUNE(ELEM_TRI, 3, 4, 64)
SSE_EULER_TUNE(ELEM_TRI, 4, 3, 64)
SSE_EULER_TUNE(ELEM_TRI, 5, 2, 64)
SSE_EULER_TUNE(ELEM_TRI, 6, 2, 64)
SSE_EULER_TUNE(ELEM_TET, 2, 4, 192)
SSE_EULER_TUNE(ELEM_TET, 3, 3, 256)
SSE_EULER_TUNE(ELEM_TET, 4, 2, 256)
SSE_EULER_TUNE(ELEM_TET, 5, 2, 384)
#undef SSE_EULER_TUNE

// The columns of the Euler kernels: TS threads hold NC columns of each of E elements (column
// s NC + e); a thread has one line of the first direction and one stage-1 line. Every step works
// on all columns at once and ends with a barrier. t: the thread among the TS (on the Tet the TS
// threads are the workgroup).
template <int ELEM, int P, int E_, int TS_>
struct EulerLines {
    using G = LineGrid<ELEM, P>;
    using LF = LineFact<ELEM, P>;
    static constexpr int E = E_, TS = TS_, NC = G::Sh::NC, NCOL = E * NC, N1 = G::N1, N2 = G::N2, NM = G::NM,
                         NX = G::NX;
    static_assert(NCOL * N2 <= TS && NCOL * NM <= TS, "a line per thread");
    UniformTable A, B;
    const double* F1;
    bool on, on1;
    int col, line, c1, m1;
    typename LF::Modes md1;

    __device__ EulerLines(const TensorParams& tp, const double* F1_, int t)
        : A(uniform_table(tp.VA)), B(uniform_table(tp.VB)), F1(F1_) {
        on = t < NCOL * N2;
        on1 = t < NCOL * NM;
        col = on ? t / N2 : 0;
        line = t % N2;
        c1 = on1 ? t / NM : 0;
        m1 = t % NM;
        md1 = LF::modes(tp.lines.mode, m1);
    }
    // LDS column W / J of each element (all threads; a barrier must follow)
    template <typename Elem>
    __device__ static void stage_woj(const DevParams& p, Elem element, double* woj) {
        constexpr int NQ = G::NQ;
        for (int t = threadIdx.x; t < E * NQ; t += TS) {
            const int s = t / NQ, i = t - s * NQ;
            woj[s * NX + G::position(i)] = p.W[i] / p.Jq[(size_t)element(s) * NQ + i];
        }
    }
    __device__ double* line1(double* X) const { return X + c1 * NX + md1.base; }
    __device__ double* line3(double* X) const { return X + col * NX + G::template base<0>(line); }
    // stage 2 of V, of V'
    __device__ void up2(double* X) const {
        if constexpr (G::TET) {
            LF::template up2<NCOL, TS>(reload(B), X);
            __syncthreads();
        }
    }
    __device__ void down2(double* X) const {
        if constexpr (G::TET) {
            LF::template down2<NCOL, TS>(reload(B), X);
            __syncthreads();
        }
    }
    // stage 3 of V: the nodal values; then(y) sees this thread's line before the barrier
    template <typename F>
    __device__ void up3(double* X, F then) const {
        if (on) {
            double x[N1], y[N1];
            line_load<N1, G::S1>(line3(X), x);
            line_apply<N1, false>(reload(A), x, y);
            line_store<N1, G::S1>(line3(X), y);
            then(y);
        }
        __syncthreads();
    }
    // stage 3 of V'
    __device__ void down3(double* X) const {
        if (on) {
            double x[N1], y[N1];
            line_load<N1, G::S1>(line3(X), x);
            line_apply<N1, true>(reload(A), x, y);
            line_store<N1, G::S1>(line3(X), y);
        }
        __syncthreads();
    }
    // stage 3 of V, W/J (an LDS column per element), stage 3 of V'
    __device__ void scale3(double* X, const double* woj) const {
        if (on) {
            double x[N1], y[N1];
            line_load<N1, G::S1>(line3(X), x);
            line_apply<N1, false>(reload(A), x, y);
            line_load<N1, G::S1>(woj + (col / NC) * NX + G::template base<0>(line), x);
#pragma unroll
            for (int a = 0; a < N1; ++a) y[a] *= x[a];
            line_apply<N1, true>(reload(A), y, x);
            line_store<N1, G::S1>(line3(X), x);
        }
        __syncthreads();
    }
    // stage 1 of V', then stage 1 of V
    __device__ void turn1(double* X) const {
        if (on1) {
            double x[N1], y[N1];
            line_load<N1, 1>(line1(X), x);
            LF::down1(F1, m1, x, y);
            LF::up1(F1, m1, y, x);
            line_store<N1, 1>(line1(X), x);
        }
        __syncthreads();
    }
    // stage 1 of V from modal coefficients x (zero past the last mode)
    __device__ void up1(double* X, const double* x) const {
        if (on1) {
            double y[N1];
            LF::up1(F1, m1, x, y);
            line_store<N1, 1>(line1(X), y);
        }
        __syncthreads();
    }
    // from stage 1 of V to stage 1 of V: V' (W/J V .) between them, i.e. the weight-adjusted
    // mass solve (mass_matrix.jl:59-75) of modal values whose stage 1 of V is done
    __device__ void mass(double* X, const double* woj) const {
        up2(X);
        scale3(X, woj);
        down2(X);
        turn1(X);
    }
};

template <int ELEM, int P>
using EulerGroup = EulerLines<ELEM, P, EulerTune<ELEM, P>::E, EulerTune<ELEM, P>::TS>;

// R' at one node: its weight on each face (line_weights: requested early) and, with S = M' t of
// NC columns of facet values NF apart, r[e] -= sum_f w_f S_e[f, line of the node]
template <int ELEM, int P>
struct NodeLift {
    using G = LineGrid<ELEM, P>;
    static constexpr int N1 = G::N1, N2 = G::N2, NF = G::Sh::NF, NFAC = G::Sh::NFAC;
    double w[NFAC];
    __device__ static void coords(int i, int dir, int& a, int& line) {
        if constexpr (G::TET) {
            const int a1 = i / N2, a2 = (i / N1) % N1, a3 = i % N1;
            a = dir == 0 ? a1 : dir == 1 ? a2 : a3;
            line = dir == 0 ? a2 * N1 + a3 : dir == 1 ? a1 * N1 + a3 : a1 * N1 + a2;
        } else {
            const int a1 = i / N1, a2 = i % N1;
            a = dir == 0 ? a1 : a2;
            line = dir == 0 ? a2 : a1;
        }
    }
    __device__ void request(const FaceTables& ft, int i) {
#pragma unroll
        for (int f = 0; f < NFAC; ++f) {
            int a, line;
            coords(i, ft.dir[f], a, line);
            w[f] = ft.w[f * N1 + a];
        }
    }
    template <int NC>
    __device__ void apply(const FaceTables& ft, int i, const double* S, double* r) const {
#pragma unroll
        for (int f = 0; f < NFAC; ++f) {
            int a, line;
            coords(i, ft.dir[f], a, line);
#pragma unroll
            for (int e = 0; e < NC; ++e) r[e] -= w[f] * S[e * NF + f * N2 + line];
        }
    }
};

}  // namespace sse
