// sse_std_tensor.hip -- StandardForm residual of scalar linear laws (advection,
// advection-diffusion with BR1) on ModalTensor triangles and tetrahedra, with
// compile-time element shapes.
//
// Same algebra as the general StandardForm kernels (the reference's
// src/Solvers/standard_form_first_order.jl:16-94 and
// src/Solvers/standard_form_second_order.jl:3-75 with the operators of
// src/Solvers/operators.jl:83-160), arranged for throughput:
//  * a workgroup advances E "slots" at once. A slot is one element of one
//    problem; with an ensemble of R problems that share the mesh and differ
//    only in the diffusion coefficient, consecutive slots are the members of
//    one element, so they also share its geometric factors;
//  * V, V' and the derivatives along collapsed directions go line by line: a thread holds a
//    line of the tensor grid in registers (sse_lines.h). V is followed and V' preceded on
//    the same lines by the pointwise and line operations next to them: the weight-adjusted
//    mass solve (M^{-1} = I, src/Solvers/mass_matrix.jl:59-75) applies stage 3 of V, W/J and
//    stage 3 of V' to a line at once, and stage 1 of V' and stage 1 of the V after it;
//  * the reference derivative operators are applied along lines: with
//    D_m = sum_l diag(c_lm) D1_l (D1_l the 1D derivative in collapsed direction l
//    on every line of the tensor grid, src/SpatialDiscretizations/
//    SpatialDiscretizations.jl:414-418) and the per-element metric folded with the
//    quadrature weight into Wt_ln = h W sum_m c_lm Lambda_mn once at set-up (h = 1/2 for the
//    skew-symmetric mapping, else 1),
//      h sum_m D_m' (W Lambda_mn x)  = sum_l D1_l' (Wt_ln x),
//      h W sum_m Lambda_mn (D_m x)   = sum_l Wt_ln (D1_l x).
//    Each entry of Wt_ln belongs to one line, so a thread loads its own from global memory
//    (all directions at the start, to be there when they are needed);
//  * between the kernels only modal coefficients and facet values go through memory: u_q and
//    q_q are formed again from u and from the modal q (a quarter of the bytes);
//  * with the skew-symmetric mapping the facet terms combine pointwise (R is linear, so
//    R u_q = u_f and R f_n = a_n u_f - b q_f,n): the gradient needs 1/2 B nJf_n u^+ and the
//    time derivative B (-1/2 nJf.a u^+ - halfl |nJf.a| (u^- - u^+) + 1/2 b nJf.q^+).
//
// What bounds it: with a node per thread every multiply-add read an LDS value, R' and R walked
// long table rows one cache latency per entry, and u_q, q_q went through memory. Tet p = 5,
// 24,576 elements: 807 -> 391 us (1.42 GB of memory traffic, 3.6 TB/s; the gradient and the
// time derivative each spend about half of a workgroup's life waiting for their first loads);
// 16 diffusivities on 1,296 Tet p = 3 elements, five steps: 4,640 -> 2,840 us (all data in the
// caches; the chain of short stages between barriers).
//
// Lanes: lane g = k * R + r is member r of element k. Intermediate arrays
// (u_f, modal q, q_f) are indexed by lane; states and time steps by
// r * N_e + k (each member a reference-layout (N_p, 1, N_e) array).
//
// Tangent pairs: the residual is linear in u and in b (viscous flux -b q,
// BR1 flux -b {q}.n, q linear in u), so v = du/db obeys the semi-discrete system
// v' = R(v; b) + dR/db(u) with dR/db(u) the viscous terms of u at unit b. A
// member pair (u, v) advanced together by the same low-storage RK stages gives
// the exact derivative of the discrete solution; only the time derivative
// kernel knows the pairing (it adds -q(u) to the tangent's viscous flux).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sse_lines.h"

namespace sse {

struct Ensemble {
    int R;              // members per element (1: a single problem)
    const double* b;    // diffusion coefficient of each member, or null for the law's b
    int tangent;        // members come in pairs (u, v = du/db): the odd member's residual
                        // is R(v; b) + dR/db(u), dR/db(u) = -(viscous terms of u at b = 1)
};

// Threads and slots of a workgroup: nodal values (TS1, E1; a line of each slot per thread) and
// the other two (TS, E; a line of each slot and direction component per thread).
template <int ELEM, int P>
struct StdTune;
#define SSE_STD_TUNE(E_, PP, ts1, e1, ts, e) \
    template <>                              \
    struct StdTune<E_, PP> {                 \
        static constexpr int TS1 = ts1, E1 = e1, TS = ts, E = e; \
    };
SSE_STD_TUNE(ELEM_TRI, 2, 64, 21, 64, 10)
SSE_STD_TUNE(ELEM_TRI, 3, 64, 16, 64, 8)
SSE_STD_TUNE(ELEM_TRI, 4, 64, 12, 64, 6)
SSE_STD_TUNE(ELEM_TRI, 5, 64, 10, 64, 5)
SSE_STD_TUNE(ELEM_TRI, 6, 64, 9, 64, 4)
SSE_STD_TUNE(ELEM_TET, 2, 128, 14, 128, 4)
SSE_STD_TUNE(ELEM_TET, 3, 192, 12, 192, 4)
SSE_STD_TUNE(ELEM_TET, 4, 256, 10, 256, 3)
SSE_STD_TUNE(ELEM_TET, 5, 256, 7, 256, 2)
#undef SSE_STD_TUNE

// Waves per SIMD the registers must allow. Lines of six and seven values take 81 to 94 registers,
// which allow 5, on either element; with 6 (80 registers) those kernels spill: Tet p = 5 at 24,576
// elements 395 us with 5, 438 with 6, Tri p = 6 at 28,800 elements 59 us with 5, 74 with 6. Up to
// p = 4 the kernels fit 6.
constexpr int std_waves(int P) { return P >= 5 ? 5 : 6; }

namespace {

// Slot s works on lane g0 + s (past the last lane: on the last one, storing nothing). The element
// and the member of a lane come from those of the first slot: a workgroup has few slots, so one
// subtraction replaces the division when the ensemble has more members than that.
template <int E>
struct Slots {
    unsigned g0, nl, R, k0, r0;
    __device__ bool valid(int s) const { return g0 + (unsigned)s < nl; }
    __device__ unsigned clamp(int s) const { return min((unsigned)s, nl - 1 - g0); }
    __device__ unsigned lane(int s) const { return g0 + clamp(s); }
    __device__ unsigned element(int s) const {
        const unsigned q = r0 + clamp(s);
        return R == 1 ? k0 + q : R >= (unsigned)E ? k0 + (q >= R ? 1u : 0u) : k0 + q / R;
    }
    __device__ unsigned member(int s) const {
        const unsigned q = r0 + clamp(s);
        return R == 1 ? 0u : R >= (unsigned)E ? (q >= R ? q - R : q) : q % R;
    }
    __device__ size_t row(int s, int N_e) const { return (size_t)member(s) * N_e + element(s); }
};

template <int E>
__device__ __forceinline__ Slots<E> slots_of(const TensorParams& tp, const Ensemble& en) {
    const unsigned g0 = (unsigned)element_of_block(blockIdx.x, gridDim.x, tp.xcd_remap) * E, R = (unsigned)en.R;
    const unsigned k0 = R == 1 ? g0 : g0 / R;
    return Slots<E>{g0, (unsigned)tp.base.N_e * R, R, k0, g0 - k0 * R};
}

// lane and facet node of the exterior state of facet node j of slot s
template <int NF, int E>
__device__ __forceinline__ unsigned neighbour(const DevParams& p, const Slots<E>& sl, int s, int j, int& jn) {
    const int gl = p.mapP[j + (size_t)NF * sl.element(s)];
    const int kn = gl / NF;
    jn = gl - kn * NF;
    return (unsigned)kn * sl.R + sl.member(s);
}

template <int V>
using Dir = std::integral_constant<int, V>;

}  // namespace

// ----------------------------------------------------------------------------- phase 1
// u_f = R V u
template <int ELEM, int P>
__global__ void __launch_bounds__((StdTune<ELEM, P>::TS1))
k_std_nodal_tensor(TensorParams tp, Ensemble en, const double* __restrict__ u) {
    using G = LineGrid<ELEM, P>;
    using LF = LineFact<ELEM, P>;
    using T = StdTune<ELEM, P>;
    constexpr int E = T::E1, TS = T::TS1, N1 = G::N1, N2 = G::N2, NM = G::NM, NX = G::NX, NP = G::NP, NF = G::Sh::NF;
    static_assert(E * N2 <= TS, "a line per thread");
    extern __shared__ double sm[];
    double* X = sm;              // E columns
    double* F1 = sm + E * NX;
    const DevParams& p = tp.base;
    const int tl = threadIdx.x;
    const Slots<E> sl = slots_of<E>(tp, en);
    const UniformTable A = uniform_table(tp.VA), B = uniform_table(tp.VB);
    LF::stage_tables(tp.lines, F1, tl, TS);
    __syncthreads();
    for (int t = tl; t < E * NM; t += TS) {
        const int s = t / NM, m = t - s * NM;
        const auto md = LF::modes(tp.lines.mode, m);
        const double* um = u + sl.row(s, p.N_e) * NP + md.off;
        double x[N1], y[N1];
#pragma unroll
        for (int b = 0; b < N1; ++b) x[b] = b <= md.lim ? um[b] : 0.0;
        LF::up1(F1, m, x, y);
        line_store<N1, 1>(X + s * NX + md.base, y);
    }
    __syncthreads();
    if constexpr (G::TET) {
        LF::template up2<E, TS>(reload(B), X);
        __syncthreads();
    }
    double* e = F1 + LF::NT1;  // E x NF line ends
    const int s = tl / N2, line = tl - s * N2;
    if (tl < E * N2) {
        double* L = X + s * NX + G::template base<0>(line);
        double x[N1], y[N1];
        line_load<N1, G::S1>(L, x);
        line_apply<N1, false>(reload(A), x, y);
        line_store<N1, G::S1>(L, y);
        line_ends<ELEM, P, 0>(tp.faces, y, line, e + s * NF);
    }
    __syncthreads();
    if (tl < E * N2) other_line_ends<ELEM, P>(tp.faces, X + s * NX, line, e + s * NF);
    __syncthreads();
    for (int t = tl; t < E * NF; t += TS) {
        const int q = t / NF, j = t - q * NF;
        double acc[1] = {0.0};
        face_row<ELEM, P, 1, NF, false>(tp.faces, j, e + q * NF, acc);
        if (sl.valid(q)) p.uf[(size_t)sl.lane(q) * NF + j] = acc[0];
    }
}

// ----------------------------------------------------------------------------- shared stages
// One direction of the terms of r for the line `line`: SIGN VT of column x, with
// VT = D1_l' (Wt x) - Wt (D1_l x) (skew) or D1_l' (Wt x), plus R' of the facet terms fs = M' t
// (fs null: none) on the faces of that direction; on top of r_col unless it is the first direction
template <int ELEM, int P, int L, bool SKEW, int SIGN>
__device__ __forceinline__ void volume_line(UniformTable D1, const FaceTables& ft, const double* x_col,
                                            const double* wt, const double* fs, int line, const double* r_col,
                                            double* r) {
    using G = LineGrid<ELEM, P>;
    constexpr int N1 = G::N1, ST = G::template stride<L>();
    const int base = G::template base<L>(line);
    const UniformTable M = D1 + L * N1 * N1;
    double x[N1], g[N1];
    line_load<N1, ST>(x_col + base, x);
    if constexpr (L == G::D - 1) {
#pragma unroll
        for (int a = 0; a < N1; ++a) r[a] = 0.0;
    } else {
        line_load<N1, ST>(r_col + base, r);
    }
#pragma unroll
    for (int b = 0; b < N1; ++b) g[b] = wt[b] * x[b];
#pragma unroll
    for (int a = 0; a < N1; ++a) {  // a row and a column of D1_l at a time (few registers)
        double y = 0.0, z = 0.0;
#pragma unroll
        for (int b = 0; b < N1; ++b) {
            y += M[b * N1 + a] * g[b];
            if constexpr (SKEW) z += M[a * N1 + b] * x[b];
        }
        if constexpr (SKEW) y -= wt[a] * z;
        r[a] += SIGN > 0 ? y : -y;
    }
    if (fs) line_ends_t<ELEM, P, L>(ft, fs, line, r);
}

// The middle of the weight-adjusted mass solve for NCOL columns CS apart whose V' has gone
// through stage 2: [stage 1 of V', stage 1 of V], stage 2, [stage 3 of V, W/J, stage 3 of V'],
// stage 2 of V'. NSUM: the columns start as sums of NSUM consecutive ones (Tri; on the Tet
// stage 2 has added them). Ends with a barrier.
// on1, c1, m1, md1: this thread's stage-1 line (column c1, lane m1) of all columns; on, col,
// line, wj: its line along the first direction and W / J there.
template <int ELEM, int P, int TS, int NCOL, int CS, int NSUM>
__device__ __forceinline__ void mass_middle(const TensorParams& tp, const double* F1, double* X, bool on1, int c1,
                                            int m1, const typename LineFact<ELEM, P>::Modes& md1, bool on, int col,
                                            int line, const double* wj) {
    using G = LineGrid<ELEM, P>;
    using LF = LineFact<ELEM, P>;
    constexpr int N1 = G::N1, NX = G::NX;
    const UniformTable A = uniform_table(tp.VA), B = uniform_table(tp.VB);
    if (on1 && c1 % CS == 0) {
        const int m = m1;
        double* L = X + c1 * NX + md1.base;
        double x[N1], y[N1];
        line_load<N1, 1>(L, x);
#pragma unroll
        for (int q = 1; q < NSUM; ++q)
#pragma unroll
            for (int a = 0; a < N1; ++a) x[a] += L[q * NX + a];
        LF::down1(F1, m, x, y);
        LF::up1(F1, m, y, x);
        line_store<N1, 1>(L, x);
    }
    __syncthreads();
    if constexpr (G::TET) {
        LF::template up2<NCOL, TS, CS>(reload(B), X);
        __syncthreads();
    }
    if (on && col % CS == 0) {
        double* L = X + col * NX + G::template base<0>(line);
        double x[N1], y[N1];
        line_load<N1, G::S1>(L, x);
        line_apply<N1, false>(reload(A), x, y);
#pragma unroll
        for (int a = 0; a < N1; ++a) y[a] *= wj[a];
        line_apply<N1, true>(reload(A), y, x);
        line_store<N1, G::S1>(L, x);
    }
    __syncthreads();
    if constexpr (G::TET) {
        LF::template down2<NCOL, TS, CS>(reload(B), X);
        __syncthreads();
    }
}

// ----------------------------------------------------------------------------- BR1 auxiliary variable
// q_n = M^{-1} V' [ -VT_n(u_q) + R' (B J_f u*_n) ],  u*_n = 1/2 (u^- + u^+) n_n,
// VT_n(x) = sum_l D1_l' (Wt_ln x) - Wt_ln (D1_l x) + R' (1/2 B nJf_n R x) (skew-symmetric
// mapping) or sum_l D1_l' (Wt_ln x) (standard mapping). With the skew form the facet terms
// combine to R' (1/2 B nJf_n u^+). Writes the modal q_n and q_f,n = R V q_n.
template <int ELEM, int P>
struct StdAuxLayout {
    using G = LineGrid<ELEM, P>;
    static constexpr int E = StdTune<ELEM, P>::E, D = G::D;
    static constexpr int u = 0, r = u + E * G::NX, tf = r + E * D * G::NX, f1 = r + E * D * G::NX + E * D * G::Sh::NF;
    static constexpr int size = f1 + LineFact<ELEM, P>::NT1;
};

template <int ELEM, int P, bool SKEW>
__global__ void __launch_bounds__((StdTune<ELEM, P>::TS), std_waves(P))
    k_std_aux_tensor(TensorParams tp, Ensemble en, const double* __restrict__ u) {
    using G = LineGrid<ELEM, P>;
    using LF = LineFact<ELEM, P>;
    using T = StdTune<ELEM, P>;
    using L = StdAuxLayout<ELEM, P>;
    constexpr int E = T::E, TS = T::TS, D = G::D, N1 = G::N1, N2 = G::N2, NM = G::NM, NX = G::NX, NP = G::NP,
                  NQ = G::NQ, NF = G::Sh::NF;
    static_assert(E * D * N2 <= TS, "a line per thread");
    extern __shared__ double sm[];
    const DevParams& p = tp.base;
    const int tl = threadIdx.x;
    const Slots<E> sl = slots_of<E>(tp, en);
    const UniformTable A = uniform_table(tp.VA), B = uniform_table(tp.VB), D1 = uniform_table(tp.D1);
    double *xu = sm + L::u, *xr = sm + L::r, *stf = sm + L::tf, *F1 = sm + L::f1;

    // this thread's line (slot, component n, line) and its metric entries of every direction
    const bool on = tl < E * D * N2;
    const int ls = on ? tl / (D * N2) : 0, ln = on ? (tl / N2) % D : 0, line = tl % N2;
    double wt[D][N1];  // requested well before its pass: the last two directions now
    const double* Wk = p.Lam + ((size_t)sl.element(ls) * D * D + D * ln) * NQ;
    auto load_wt = [&](auto l) {
        constexpr int l_ = decltype(l)::value;
#pragma unroll
        for (int a = 0; a < N1; ++a)
            wt[l_][a] = Wk[l_ * NQ + G::template node<l_>(line) + a * G::template node_stride<l_>()];
    };
    // and its stage-1 line (column c1 of E D)
    static_assert(E * D * NM <= TS, "a stage-1 line per thread");
    const bool on1 = tl < E * D * NM;
    const int c1 = tl / NM, m1 = tl % NM;
    const auto md1 = LF::modes(tp.lines.mode, m1);
    // this thread's facet nodes: the neighbours first (their states hang on them)
    constexpr int IT = (E * NF + TS - 1) / TS;
    unsigned gn[IT];
    int jn[IT];
#pragma unroll
    for (int q = 0; q < IT; ++q) {
        const int t = min(tl + q * TS, E * NF - 1), s = t / NF;
        gn[q] = neighbour<NF>(p, sl, s, t - s * NF, jn[q]);
    }
    // everything the prologue reads is requested before the first of it is used: modal u of the
    // stage-1 line (column s1 of the first E), the facet states, the metric entries
    const int s1 = min(c1, E - 1);
    double xm[N1], uo[IT], ui[IT], nJ[IT][D];
    {
        const double* um = u + sl.row(s1, p.N_e) * NP + md1.off;
#pragma unroll
        for (int b = 0; b < N1; ++b) xm[b] = um[min(b, md1.lim)];
    }
#pragma unroll
    for (int q = 0; q < IT; ++q) {
        const int t = min(tl + q * TS, E * NF - 1), s = t / NF, j = t - s * NF;
        const unsigned g = sl.lane(s);
        uo[q] = p.uf[(size_t)gn[q] * NF + jn[q]];
        if (!SKEW) ui[q] = p.uf[(size_t)g * NF + j];
        const double* n = p.nJf + (size_t)sl.element(s) * D * NF + D * j;
#pragma unroll
        for (int m = 0; m < D; ++m) nJ[q][m] = n[m];
    }
    LF::stage_tables(tp.lines, F1, tl, TS);
    load_wt(Dir<D - 1>{});
    if constexpr (D == 3) load_wt(Dir<1>{});
    // facet terms: 1/2 B nJf_n u^+ (skew) or 1/2 B nJf_n (u^- + u^+)
#pragma unroll
    for (int q = 0; q < IT; ++q) {
        const int t = tl + q * TS;
        if (t >= E * NF) break;
        const int s = t / NF, j = t - s * NF;
        const double x = 0.5 * p.B[j] * (SKEW ? uo[q] : ui[q] + uo[q]);
#pragma unroll
        for (int n = 0; n < D; ++n) stf[(s * D + n) * NF + j] = nJ[q][n] * x;
    }
    __syncthreads();
    if (tl < E * NM) {  // stage 1 of V u
        double y[N1];
#pragma unroll
        for (int b = 0; b < N1; ++b) xm[b] = b <= md1.lim ? xm[b] : 0.0;
        LF::up1(F1, m1, xm, y);
        line_store<N1, 1>(xu + s1 * NX + md1.base, y);
    }
    face_transpose<ELEM, P, E * D, TS>(tp.faces, stf, tl);
    __syncthreads();
    if constexpr (G::TET) {
        LF::template up2<E, TS>(reload(B), xu);
        __syncthreads();
    }
    if (tl < E * N2) {
        double* X = xu + (tl / N2) * NX + G::template base<0>(tl % N2);
        double x[N1], y[N1];
        line_load<N1, G::S1>(X, x);
        line_apply<N1, false>(reload(A), x, y);
        line_store<N1, G::S1>(X, y);
    }
    __syncthreads();
    // r_n -= VT_n(u_q), one direction after the other; the last (along a1) goes on with stage
    // 3 of V'
    double wj[N1];  // W / J along this thread's line, for the mass solve
    auto load_woj = [&]() {
        const double* w = tp.WoJ + (size_t)sl.element(ls) * NQ + G::template node<0>(line);
#pragma unroll
        for (int a = 0; a < N1; ++a) wj[a] = w[a * G::template node_stride<0>()];
    };
    const double* xc = xu + ls * NX;
    double* rc = xr + (ls * D + ln) * NX;
    auto pass = [&](auto l) {
        constexpr int l_ = decltype(l)::value;
        if constexpr (l_ == D - 1) load_wt(Dir<0>{});
        if constexpr (l_ == 1) load_woj();
        if (on) {
            double r[N1];
            volume_line<ELEM, P, l_, SKEW, -1>(reload(D1), tp.faces, xc, wt[l_], stf + (ls * D + ln) * NF, line, rc,
                                               r);
            if constexpr (l_ == 0) {
                double w[N1];
                line_apply<N1, true>(reload(A), r, w);
                line_store<N1, G::S1>(rc + G::template base<0>(line), w);
            } else {
                line_store<N1, G::template stride<l_>()>(rc + G::template base<l_>(line), r);
            }
        }
        __syncthreads();
    };
    if constexpr (D == 3) pass(Dir<2>{});
    pass(Dir<1>{});
    pass(Dir<0>{});
    if constexpr (G::TET) {
        LF::template down2<E * D, TS>(reload(B), xr);
        __syncthreads();
    }
    mass_middle<ELEM, P, TS, E * D, 1, 1>(tp, F1, xr, on1, c1, m1, md1, on, ls * D + ln, line, wj);
    // modal q_n out, and V q_n
    if (on1) {
        const int s = c1 / D;
        double* X = xr + c1 * NX + md1.base;
        double x[N1], y[N1];
        line_load<N1, 1>(X, x);
        LF::down1(F1, m1, x, y);
        if (sl.valid(s)) {
            double* q = p.qq + ((size_t)sl.lane(s) * D + (c1 - s * D)) * NP + md1.off;
#pragma unroll
            for (int b = 0; b < N1; ++b)
                if (b <= md1.lim) q[b] = y[b];
        }
        LF::up1(F1, m1, y, x);
        line_store<N1, 1>(X, x);
    }
    __syncthreads();
    if constexpr (G::TET) {
        LF::template up2<E * D, TS>(reload(B), xr);
        __syncthreads();
    }
    // q_f = R q_q: the ends of the lines, then the interpolation on the faces
    double* e = stf + (ls * D + ln) * NF;
    if (on) {
        double* X = rc + G::template base<0>(line);
        double x[N1], y[N1];
        line_load<N1, G::S1>(X, x);
        line_apply<N1, false>(reload(A), x, y);
        line_store<N1, G::S1>(X, y);
        line_ends<ELEM, P, 0>(tp.faces, y, line, e);
    }
    __syncthreads();
    if (on) other_line_ends<ELEM, P>(tp.faces, rc, line, e);
    __syncthreads();
    for (int t = tl; t < E * NF; t += TS) {
        const int s = t / NF, j = t - s * NF;
        double acc[D];
#pragma unroll
        for (int n = 0; n < D; ++n) acc[n] = 0.0;
        face_row<ELEM, P, D, NF, false>(tp.faces, j, stf + s * D * NF, acc);
        if (sl.valid(s)) {
#pragma unroll
            for (int n = 0; n < D; ++n) p.qf[((size_t)sl.lane(s) * D + n) * NF + j] = acc[n];
        }
    }
}

// ----------------------------------------------------------------------------- time derivative
// dudt = M^{-1} V' [ sum_n VT_n(f_n) - R' (B J_f f*) ],  f_n = a_n u - b q_n,
// f* = a.n {u} + halfl |a.n| [u] - b {q}.n (LF; BR1 when second order).
// dudt may be u, and an RK stage updates u: a workgroup reads u of its own slots only, all of it
// before the barriers that precede its stores.
template <int ELEM, int P>
struct StdTdLayout {
    using G = LineGrid<ELEM, P>;
    static constexpr int E = StdTune<ELEM, P>::E, D = G::D;
    static constexpr int f = 0, r = f + E * D * G::NX, t = r + E * D * G::NX, f1 = r + E * D * G::NX + E * G::Sh::NF;
    static constexpr int size = f1 + LineFact<ELEM, P>::NT1;
};

template <int ELEM, int P, bool SKEW, bool SECOND>
__global__ void __launch_bounds__((StdTune<ELEM, P>::TS), std_waves(P))
    k_std_td_tensor(TensorParams tp, Ensemble en, const double* u, double* dudt, RKStage rk) {
    using G = LineGrid<ELEM, P>;
    using LF = LineFact<ELEM, P>;
    using T = StdTune<ELEM, P>;
    using L = StdTdLayout<ELEM, P>;
    constexpr int E = T::E, TS = T::TS, D = G::D, N1 = G::N1, N2 = G::N2, NM = G::NM, NX = G::NX, NP = G::NP,
                  NQ = G::NQ, NF = G::Sh::NF;
    extern __shared__ double sm[];
    const DevParams& p = tp.base;
    const int tl = threadIdx.x;
    const Slots<E> sl = slots_of<E>(tp, en);
    const UniformTable A = uniform_table(tp.VA), B = uniform_table(tp.VB), D1 = uniform_table(tp.D1);
    double *xf = sm + L::f, *xr = sm + L::r, *st = sm + L::t, *F1 = sm + L::f1;
    const bool on = tl < E * D * N2;
    const int ls = on ? tl / (D * N2) : 0, ln = on ? (tl / N2) % D : 0, line = tl % N2;
    double wt[D][N1];  // requested well before its pass: the last two directions now
    const double* Wk = p.Lam + ((size_t)sl.element(ls) * D * D + D * ln) * NQ;
    auto load_wt = [&](auto l) {
        constexpr int l_ = decltype(l)::value;
#pragma unroll
        for (int a = 0; a < N1; ++a)
            wt[l_][a] = Wk[l_ * NQ + G::template node<l_>(line) + a * G::template node_stride<l_>()];
    };
    // and its stage-1 line (column c1 of E D)
    static_assert(E * D * NM <= TS, "a stage-1 line per thread");
    const bool on1 = tl < E * D * NM;
    const int c1 = tl / NM, m1 = tl % NM;
    const auto md1 = LF::modes(tp.lines.mode, m1);
    auto member_b = [&](int s) { return en.b ? en.b[sl.member(s)] : p.b; };
    auto is_tangent = [&](int s) { return SECOND && en.tangent && (sl.member(s) & 1); };
    // this thread's facet nodes: the neighbours first (their states hang on them)
    constexpr int IT = (E * NF + TS - 1) / TS;
    unsigned gns[IT];
    int jns[IT];
#pragma unroll
    for (int q = 0; q < IT; ++q) {
        const int t = min(tl + q * TS, E * NF - 1), s = t / NF;
        gns[q] = neighbour<NF>(p, sl, s, t - s * NF, jns[q]);
    }
    // modal u and q_n of the stage-1 line (slot s1, component n1), used after the facets
    const int cc = min(c1, E * D - 1), s1 = cc / D, n1 = cc - s1 * D;
    double xm[N1], qm[N1];
    {
        const double* um = u + sl.row(s1, p.N_e) * NP + md1.off;
#pragma unroll
        for (int b = 0; b < N1; ++b) xm[b] = um[min(b, md1.lim)];
        if constexpr (SECOND) {
            const double* q = p.qq + ((size_t)sl.lane(s1) * D + n1) * NP + md1.off;
#pragma unroll
            for (int b = 0; b < N1; ++b) qm[b] = q[min(b, md1.lim)];
        }
    }
    // facet values 1/2 B sum_n nJf_n (R f_n) - B J_f f* (the first term with the skew form only)
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int t = tl + it * TS;
        if (t >= E * NF) break;
        const int s = t / NF, j = t - s * NF, jn = jns[it];
        const unsigned g = sl.lane(s), gn = gns[it];
        const double um = p.uf[(size_t)g * NF + j], up = p.uf[(size_t)gn * NF + jn];
        const double* nJ = p.nJf + (size_t)sl.element(s) * D * NF + D * j;
        double an = 0.0;  // J_f a.n
#pragma unroll
        for (int m = 0; m < D; ++m) an += p.law.a[m] * nJ[m];
        double val = -0.5 * an * (SKEW ? up : um + up);
        if (p.law.inviscid_flux == 1) val -= p.law.half_lambda * fabs(an) * (um - up);
        if constexpr (SECOND) {
            const double bm = member_b(s);
            const bool tan = is_tangent(s);
            double qn = 0.0;
#pragma unroll
            for (int m = 0; m < D; ++m) {
                double q = bm * p.qf[((size_t)gn * D + m) * NF + jn];
                if (!SKEW) q += bm * p.qf[((size_t)g * D + m) * NF + j];
                if (tan) {  // + the pair's u at unit b
                    q += p.qf[((size_t)(gn - 1) * D + m) * NF + jn];
                    if (!SKEW) q += p.qf[((size_t)(g - 1) * D + m) * NF + j];
                }
                qn += q * nJ[m];
            }
            val += 0.5 * qn;
        }
        st[t] = p.B[j] * val;
    }
    LF::stage_tables(tp.lines, F1, tl, TS);
    load_wt(Dir<D - 1>{});
    if constexpr (D == 3) load_wt(Dir<1>{});
    {  // modal f_n = a_n u - b q_n
        const double an = n1 == 0 ? p.law.a[0] : n1 == 1 ? p.law.a[1] : p.law.a[2];
        const double bm = SECOND ? member_b(s1) : 0.0;
        const bool tan = is_tangent(s1);
#pragma unroll
        for (int b = 0; b < N1; ++b) {
            xm[b] *= an;
            if constexpr (SECOND) {
                xm[b] -= bm * qm[b];
                if (tan)  // dR/db(u) of the pair's u
                    xm[b] -= p.qq[((size_t)sl.lane(s1) * D + n1 - D) * NP + md1.off + min(b, md1.lim)];
            }
            if (b > md1.lim) xm[b] = 0.0;
        }
    }
    __syncthreads();
    if (on1) {  // stage 1 of V f_n
        double y[N1];
        LF::up1(F1, m1, xm, y);
        line_store<N1, 1>(xf + c1 * NX + md1.base, y);
    }
    face_transpose<ELEM, P, E, TS>(tp.faces, st, tl);
    __syncthreads();
    if constexpr (G::TET) {
        LF::template up2<E * D, TS>(reload(B), xf);
        __syncthreads();
    }
    double wj[N1];  // W / J along this thread's line, for the mass solve
    auto load_woj = [&]() {
        const double* w = tp.WoJ + (size_t)sl.element(ls) * NQ + G::template node<0>(line);
#pragma unroll
        for (int a = 0; a < N1; ++a) wj[a] = w[a * G::template node_stride<0>()];
    };
    const double* xc = xf + (ls * D + ln) * NX;
    double* rc = xr + (ls * D + ln) * NX;
    if (on) {
        double* X = xf + (ls * D + ln) * NX + G::template base<0>(line);
        double x[N1], y[N1];
        line_load<N1, G::S1>(X, x);
        line_apply<N1, false>(reload(A), x, y);
        line_store<N1, G::S1>(X, y);
    }
    __syncthreads();
    auto pass = [&](auto l) {
        constexpr int l_ = decltype(l)::value;
        if constexpr (l_ == D - 1) load_wt(Dir<0>{});
        if constexpr (l_ == 1) load_woj();
        if (on) {
            double r[N1];
            // R' of the facet values joins component 0
            volume_line<ELEM, P, l_, SKEW, 1>(reload(D1), tp.faces, xc, wt[l_], ln == 0 ? st + ls * NF : nullptr,
                                              line, rc, r);
            if constexpr (l_ == 0) {
                double w[N1];
                line_apply<N1, true>(reload(A), r, w);
                line_store<N1, G::S1>(rc + G::template base<0>(line), w);
            } else {
                line_store<N1, G::template stride<l_>()>(rc + G::template base<l_>(line), r);
            }
        }
        __syncthreads();
    };
    if constexpr (D == 3) pass(Dir<2>{});
    pass(Dir<1>{});
    pass(Dir<0>{});
    // the D components add up in the next stage of V'; then the mass solve of one column per slot
    if constexpr (G::TET) {
        LF::template down2<E, TS, D, D>(reload(B), xr);
        __syncthreads();
    }
    mass_middle<ELEM, P, TS, E, D, G::TET ? 1 : D>(tp, F1, xr, on1, c1, m1, md1, on, ls * D + ln, line, wj);
    if (on1 && c1 % D == 0 && sl.valid(c1 / D)) {
        const int s = c1 / D;
        const auto& md = md1;
        const size_t row = sl.row(s, p.N_e), o = row * NP + md.off;
        double x[N1], y[N1];
        line_load<N1, 1>(xr + s * D * NX + md.base, x);
        LF::down1(F1, m1, x, y);
        const double dt = rk.dt_e ? rk.dt_e[row] : rk.dt;
#pragma unroll
        for (int b = 0; b < N1; ++b) {
            if (b > md.lim) continue;
            if (!rk.active) {
                dudt[o + b] = y[b];
            } else {
                const double kt = (rk.A == 0.0 ? 0.0 : rk.A * rk.tmp[o + b]) + dt * y[b];
                rk.tmp[o + b] = kt;
                rk.u[o + b] += rk.B * kt;
            }
        }
    }
}

// ----------------------------------------------------------------------------- set-up
// In place: Lambda_mn -> Wt_ln = h W sum_m c_lm Lambda_mn at every node of every
// element (c: N_q x d x d, c[(i d + l) d + m]); WoJ = W / J.
__global__ void k_collapse_metric(double* __restrict__ Lam, const double* __restrict__ c, const double* __restrict__ W,
                                  const double* __restrict__ Jq, double* __restrict__ WoJ, double h, int NQ, int D,
                                  long long n_nodes) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_nodes) return;
    const long long k = t / NQ;
    const int i = (int)(t - k * NQ);
    double* Lk = Lam + (size_t)k * NQ * D * D;
    double in[9], out[9];
    for (int m = 0; m < D; ++m)
        for (int n = 0; n < D; ++n) in[m + 3 * n] = Lk[i + NQ * (m + D * n)];
    for (int l = 0; l < D; ++l)
        for (int n = 0; n < D; ++n) {
            double s = 0.0;
            for (int m = 0; m < D; ++m) s += c[(i * D + l) * D + m] * in[m + 3 * n];
            out[l + 3 * n] = s * (h * W[i]);
        }
    for (int l = 0; l < D; ++l)
        for (int n = 0; n < D; ++n) Lk[i + NQ * (l + D * n)] = out[l + 3 * n];
    WoJ[t] = W[i] / Jq[t];
}

hipError_t collapse_metric(double* Lam, const double* c, const double* W, const double* Jq, double* WoJ, double h,
                           int NQ, int D, int N_e, hipStream_t s) {
    const long long n = (long long)NQ * N_e;
    hipLaunchKernelGGL(k_collapse_metric, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, Lam, c, W, Jq, WoJ, h, NQ,
                       D, n);
    return hipGetLastError();
}

// ----------------------------------------------------------------------------- launch
template <int ELEM, int P>
size_t std_tensor_lds(int which) {
    if (which == 0) return sizeof(double) * (StdTune<ELEM, P>::E1 * (LineGrid<ELEM, P>::NX + LineGrid<ELEM, P>::Sh::NF) + LineFact<ELEM, P>::NT1);
    if (which == 1) return sizeof(double) * StdAuxLayout<ELEM, P>::size;
    return sizeof(double) * StdTdLayout<ELEM, P>::size;
}

template <int ELEM, int P, bool SKEW, bool SECOND>
hipError_t launch_std_tensor_t(const TensorParams& tp, const Ensemble& en, const double* u, double* dudt,
                               const RKStage& rk, hipStream_t s, int which) {
    using T = StdTune<ELEM, P>;
    static_assert(sizeof(double) * StdTdLayout<ELEM, P>::size <= 64 * 1024 &&
                      sizeof(double) * StdAuxLayout<ELEM, P>::size <= 64 * 1024 &&
                      sizeof(double) * (T::E1 * (LineGrid<ELEM, P>::NX + LineGrid<ELEM, P>::Sh::NF) + LineFact<ELEM, P>::NT1) <= 64 * 1024,
                  "within the default dynamic LDS limit");
    const long long nl = (long long)tp.base.N_e * en.R;
    auto blocks = [&](int e) { return dim3((unsigned)((nl + e - 1) / e)); };
    if (which & 1) {
        hipLaunchKernelGGL((k_std_nodal_tensor<ELEM, P>), blocks(T::E1), dim3(T::TS1), (std_tensor_lds<ELEM, P>(0)), s,
                           tp, en, u);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (which & 2) {
        if (SECOND) {
            hipLaunchKernelGGL((k_std_aux_tensor<ELEM, P, SKEW>), blocks(T::E), dim3(T::TS),
                               (std_tensor_lds<ELEM, P>(1)), s, tp, en, u);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL((k_std_td_tensor<ELEM, P, SKEW, SECOND>), blocks(T::E), dim3(T::TS),
                           (std_tensor_lds<ELEM, P>(2)), s, tp, en, u, dudt, rk);
        return hipGetLastError();
    }
    return hipSuccess;
}

template <int ELEM, int P>
hipError_t launch_std_tensor_p(const TensorParams& tp, const Ensemble& en, const double* u, double* dudt,
                               const RKStage& rk, hipStream_t s, int which) {
    const bool skew = tp.base.skew, second = tp.base.second_order;
    if (skew && second) return launch_std_tensor_t<ELEM, P, true, true>(tp, en, u, dudt, rk, s, which);
    if (skew) return launch_std_tensor_t<ELEM, P, true, false>(tp, en, u, dudt, rk, s, which);
    if (second) return launch_std_tensor_t<ELEM, P, false, true>(tp, en, u, dudt, rk, s, which);
    return launch_std_tensor_t<ELEM, P, false, false>(tp, en, u, dudt, rk, s, which);
}

#define SSE_STD_CASES                                                                               \
    SSE_CASE(ELEM_TRI, 2) SSE_CASE(ELEM_TRI, 3) SSE_CASE(ELEM_TRI, 4) SSE_CASE(ELEM_TRI, 5)          \
    SSE_CASE(ELEM_TRI, 6) SSE_CASE(ELEM_TET, 2) SSE_CASE(ELEM_TET, 3) SSE_CASE(ELEM_TET, 4)          \
    SSE_CASE(ELEM_TET, 5)

// (elem, P) has compiled kernels
bool std_tensor_config(int elem, int P) {
#define SSE_CASE(E_, PP) \
    if (elem == E_ && P == PP) return true;
    SSE_STD_CASES
#undef SSE_CASE
    return false;
}

hipError_t launch_std_tensor(const TensorParams& tp, int R, const double* b_member, int tangent, const double* u,
                             double* dudt, const RKStage& rk, hipStream_t s, int which) {
    if (tangent && ((R & 1) || !tp.base.second_order)) return hipErrorInvalidValue;
    const Ensemble en{R, b_member, tangent};
#define SSE_CASE(E_, PP) \
    if (tp.elem == E_ && tp.P == PP) return launch_std_tensor_p<E_, PP>(tp, en, u, dudt, rk, s, which);
    SSE_STD_CASES
#undef SSE_CASE
    return hipErrorInvalidValue;
}

}  // namespace sse
