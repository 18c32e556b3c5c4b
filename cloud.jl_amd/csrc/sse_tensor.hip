// sse_tensor.hip -- residual kernels for ModalTensor triangles and tetrahedra
// with compile-time shapes (element type and degree P), for the Euler equations
// in FluxDifferencingForm with the entropy-conservative two-point flux.
//
// Same algorithm as the reference (src/Solvers/flux_differencing_form.jl), with
// the work organised for CDNA4:
//   * V and V' are applied sum-factorised (the WarpedTensorProductMap2D/3D
//     algorithm of src/MatrixFreeOperators/warped_product_{2d,3d}.jl): in nodal_values a
//     line of the tensor grid per thread (sse_lines.h), in time_derivative one thread
//     per output point, all variables at once, stages staged in LDS;
//   * the Hadamard sum and the facet correction are one list of unique pairs:
//     each volume pair (i < j) of the union sparsity of S_1..S_d and each
//     nonzero C_ij is evaluated exactly once per element; contributions go to
//     an LDS staging area and are summed into the owning node in a fixed,
//     host-built order (deterministic, no atomics);
//   * per-node quantities (velocity, pressure, log rho, rho/p, log(rho/p)) are
//     computed once, so a pair costs one divide and no logarithm;
//   * the flux tensor is never formed: it is contracted with the metric vector
//     inside the flux (ec_dot).
// A "team" of TS threads owns one element; a block holds EPB teams.
#include <hip/hip_runtime.h>

#include "sse_lines.h"

namespace sse {

// ----------------------------------------------------------------------------- set-up
// The weight-adjusted inverse mass matrix of every element, V' diag(W / J_k) V
// (mass_matrix.jl:150-153 with the orthonormal modal basis: M^{-1} = I), column-major
// and symmetric: the upper triangle is summed, each entry written to both halves.
__global__ void __launch_bounds__(256) k_weight_adjusted_inverse(int N_p, int N_q, const double* __restrict__ V,
                                                                 const double* __restrict__ W,
                                                                 const double* __restrict__ Jq, double* __restrict__ Mw) {
    extern __shared__ double s_w[];  // N_q: W / J_k
    const size_t k = blockIdx.x;
    for (int i = threadIdx.x; i < N_q; i += blockDim.x) s_w[i] = W[i] / Jq[k * N_q + i];
    __syncthreads();
    double* Mk = Mw + k * N_p * N_p;
    for (int t = threadIdx.x; t < N_p * N_p; t += blockDim.x) {
        const int a = t % N_p, b = t / N_p;
        if (a > b) continue;
        double s = 0.0;
        for (int i = 0; i < N_q; ++i) s += V[i + (size_t)N_q * a] * s_w[i] * V[i + (size_t)N_q * b];
        Mk[a + (size_t)N_p * b] = s;
        Mk[b + (size_t)N_p * a] = s;
    }
}

hipError_t launch_weight_adjusted_inverse(const DevParams& p, double* Mw, hipStream_t s) {
    if (!p.has_V || !p.V) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_weight_adjusted_inverse, dim3(p.N_e), dim3(256), sizeof(double) * p.N_q, s, p.N_p, p.N_q,
                       p.V, p.W, p.Jq, Mw);
    return hipGetLastError();
}

// ----------------------------------------------------------------------------- nodal_values
// u_q = V u -> w = V' (WJ c2e(u_q)) -> M^{-1} w -> w_q = V w -> u_q = e2c(w_q), u_f = e2c(R w_q),
// line by line (EulerLines), M^{-1} = V' (W/J V .) by the same transforms from p = 4 on: a kept
// matrix per element would be 38 % of this kernel's memory traffic at Tet p = 4, and a line's
// transform is cheap. Up to p = 3 M^{-1} is the kept matrix where there is one: fewer roundings go
// through e2c (error of the residual against 80-bit arithmetic, rms over 24 perturbed states, with
// the transforms and with the matrix: Tet p = 2 4.4e-14 and 3.1e-14, Tet p = 3 4.4e-14 and 3.8e-14,
// Tri p = 2 3.6e-14 and 2.9e-14; Tri p = 4 8.0e-14 with either form of the earlier kernels) at 2 % of
// the residual's time on 16,464 Tet p = 3 elements (183 and 186 us). R is the ends of the lines and the interpolation on the faces (FaceTables).
// With a node per thread (every multiply-add reading LDS, R in table rows) the whole residual
// took 669 us at 24,576 Tet p = 4 elements and 42.3 us at 8,192 Tri p = 3, now 595 and 27.9 us.
template <int ELEM, int P>
struct K1Layout {
    using L = EulerGroup<ELEM, P>;
    using Sh = Shape<ELEM, P>;
    static constexpr int x = 0, woj = x + L::NCOL * L::NX, f1 = woj + L::E * L::NX, e = f1 + L::LF::NT1;
    static constexpr int size = e + L::NCOL * Sh::NF;
};

template <int ELEM, int P>
__device__ __forceinline__ void nodal_values_body(const TensorParams& tp, const double* __restrict__ u, int block,
                                                  int blocks) {
    using Sh = Shape<ELEM, P>;
    using G = LineGrid<ELEM, P>;
    using EL = EulerGroup<ELEM, P>;
    using L = K1Layout<ELEM, P>;
    constexpr int D = Sh::D, NC = Sh::NC, NP = Sh::NP, NQ = Sh::NQ, NF = Sh::NF, N1 = G::N1, NX = G::NX;
    constexpr int E = EL::E, TS = EL::TS, ITQ = (E * NQ + TS - 1) / TS;
    extern __shared__ double sm[];
    const DevParams& p = tp.base;
    const int tl = threadIdx.x;
    const int k0 = element_of_block(block, blocks, tp.xcd_remap) * E, last = p.N_e - 1;
    auto element = [&](int s) { return min(k0 + s, last); };  // past the last: computed, not stored
    double *X = sm + L::x, *woj = sm + L::woj, *F1 = sm + L::f1, *es = sm + L::e;
    EL::LF::stage_tables(tp.lines, F1, tl, TS);
    const EL el(tp, F1, tl);
    double J[ITQ], um[N1];
    {
        const int s = el.c1 / NC, e = el.c1 - s * NC;
        const double* uk = u + ((size_t)element(s) * NC + e) * NP + el.md1.off;
#pragma unroll
        for (int b = 0; b < N1; ++b) um[b] = b <= el.md1.lim ? uk[b] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < ITQ; ++q) {
        const int t = min(tl + q * TS, E * NQ - 1), s = t / NQ;
        J[q] = p.Jq[(size_t)element(s) * NQ + (t - s * NQ)];
    }
    __syncthreads();
    el.up1(X, um);
    el.up2(X);
    el.up3(X, [](const double*) {});  // u_q = V u
    bool ok = true;
#pragma unroll
    for (int q = 0; q < ITQ; ++q) {  // w_q = WJ c2e(u_q)
        const int t = tl + q * TS;
        if (t >= E * NQ) break;
        const int s = t / NQ, i = t - s * NQ;
        double* x = X + s * NC * NX + G::position(i);
        double ub[NC], wb[NC];
#pragma unroll
        for (int e = 0; e < NC; ++e) ub[e] = x[e * NX];
        ok &= c2e_fast<D>(p.law, ub, wb);
        const double W = p.W[i], wj = W * J[q];
        woj[s * NX + G::position(i)] = W / J[q];
#pragma unroll
        for (int e = 0; e < NC; ++e) x[e * NX] = wb[e] * wj;
    }
    __syncthreads();
    // the kept matrix up to p = 3: a row of one element per PARTS neighbouring threads, requested early
    constexpr bool KEPT = P <= 3;
    constexpr int PARTS = E * NP * 4 <= TS ? 4 : E * NP * 2 <= TS ? 2 : 1, LEN = KEPT ? (NP + PARTS - 1) / PARTS : 1;
    static_assert(!KEPT || (E * NP <= TS && NP <= NF), "a row per thread, the modal values in place of the line ends");
    const int row = tl / PARTS, part = tl % PARTS, sm_ = min(row / NP, E - 1), jm = row % NP;
    double mk[LEN];
    if (KEPT && tp.Mw) {
        const double* Mk = tp.Mw + (size_t)element(sm_) * NP * NP + jm;  // symmetric: row j as a column
#pragma unroll
        for (int q = 0; q < LEN; ++q) mk[q] = part + q * PARTS < NP ? Mk[(size_t)(part + q * PARTS) * NP] : 0.0;
    }
    el.down3(X);
    el.down2(X);
    if (KEPT && tp.Mw) {
        double* y = es;  // NCOL x NP modal values
        if (el.on1) {
            double x[N1], m[N1];
            line_load<N1, 1>(el.line1(X), x);
            EL::LF::down1(F1, el.m1, x, m);
#pragma unroll
            for (int b = 0; b < N1; ++b)
                if (b <= el.md1.lim) y[el.c1 * NP + el.md1.off + b] = m[b];
        }
        __syncthreads();
        double s[NC];
#pragma unroll
        for (int e = 0; e < NC; ++e) {
            s[e] = 0.0;
#pragma unroll
            for (int q = 0; q < LEN; ++q) s[e] += mk[q] * y[(sm_ * NC + e) * NP + min(part + q * PARTS, NP - 1)];
#pragma unroll
            for (int w = 1; w < PARTS; w <<= 1) s[e] += __shfl_xor(s[e], w, 64);
        }
        if (part == 0 && row < E * NP) {
#pragma unroll
            for (int e = 0; e < NC; ++e) X[(sm_ * NC + e) * NX + jm] = s[e];
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < N1; ++b) um[b] = b <= el.md1.lim ? X[el.c1 * NX + el.md1.off + b] : 0.0;
        __syncthreads();
        el.up1(X, um);
    } else {
        el.turn1(X);
        el.mass(X, woj);
    }
    el.up2(X);
    double* ec = es + el.col * NF;
    el.up3(X, [&](const double* y) { line_ends<ELEM, P, 0>(tp.faces, y, el.line, ec); });  // w_q = V w
    if (el.on) other_line_ends<ELEM, P>(tp.faces, X + el.col * NX, el.line, ec);
#pragma unroll
    for (int q = 0; q < ITQ; ++q) {  // u_q = e2c(w_q)
        const int t = tl + q * TS;
        if (t >= E * NQ) break;
        const int s = t / NQ, i = t - s * NQ;
        const double* x = X + s * NC * NX + G::position(i);
        double ub[NC], wb[NC];
#pragma unroll
        for (int e = 0; e < NC; ++e) wb[e] = x[e * NX];
        ok &= e2c_fast<D>(p.law, wb, ub);
        if (k0 + s <= last) {
            double* uqk = p.uq + (size_t)(k0 + s) * NQ * NC;
#pragma unroll
            for (int e = 0; e < NC; ++e) uqk[e * NQ + i] = ub[e];
        }
    }
    __syncthreads();
    for (int t = tl; t < E * NF; t += TS) {  // u_f = e2c(R w_q)
        const int s = t / NF, j = t - s * NF, k = element(s);
        const int g = tp.uf_ext ? p.mapP[j + (size_t)NF * k] : 0;
        double ub[NC], wb[NC];
#pragma unroll
        for (int e = 0; e < NC; ++e) wb[e] = 0.0;
        face_row<ELEM, P, NC, NF, false>(tp.faces, j, es + s * NC * NF, wb);
        ok &= e2c_fast<D>(p.law, wb, ub);
        if (k0 + s > last) continue;
        double* ufk = p.uf + (size_t)k * NF * NC;
#pragma unroll
        for (int e = 0; e < NC; ++e) ufk[e * NF + j] = ub[e];
        if (tp.uf_ext) {  // also the neighbour's exterior state: uf_ext at mapP(j, k) = u_f(j, k)
            const int kn = g / NF, jn = g - kn * NF;
            double* uxn = tp.uf_ext + (size_t)kn * NF * NC;
#pragma unroll
            for (int e = 0; e < NC; ++e) uxn[e * NF + jn] = ub[e];
        }
    }
    if (!ok) atomicOr(p.status, 1);
}

template <int ELEM, int P>
__global__ void __launch_bounds__((EulerTune<ELEM, P>::TS), (ELEM == ELEM_TET ? 6 : 1))
k_nodal_values_tensor(TensorParams tp, const double* __restrict__ u) {
    nodal_values_body<ELEM, P>(tp, u, blockIdx.x, gridDim.x);
}

// Triangles of several degrees in one launch: each degree alone leaves most of the chip idle,
// and branches of a graph overlap only in part (24 problems of degrees 2 to 6, 7,468 triangles:
// 133 us per RK stage one after the other, 72 us in five branches, 55 us in one launch of each
// kernel: 17 us here and 38 us for the time derivative, 1.8 rounds of its 4 wavefronts per SIMD).
__global__ void __launch_bounds__(64) k_nodal_values_tri_groups(TriGroups a) {
    static_assert(K1Layout<ELEM_TRI, 2>::size * 8 <= 65536 && K1Layout<ELEM_TRI, 6>::size * 8 <= 65536,
                  "LDS without an attribute");
    int block = blockIdx.x;
#define SSE_TRI_GROUP(PP)                                                                           \
    if (block < a.g[PP - 2].blocks1)                                                                \
        return nodal_values_body<ELEM_TRI, PP>(a.g[PP - 2].params(), a.g[PP - 2].rk.u, block, a.g[PP - 2].blocks1); \
    block -= a.g[PP - 2].blocks1;
    SSE_TRI_GROUP(6)
    SSE_TRI_GROUP(5)
    SSE_TRI_GROUP(4)
    SSE_TRI_GROUP(3)
    SSE_TRI_GROUP(2)
#undef SSE_TRI_GROUP
}

template <int P>
void tri_k1_config(int N_e, int* blocks, int* lds) {
    using T = EulerTune<ELEM_TRI, P>;
    static_assert(T::TS == 64, "one block size");
    *blocks = (N_e + T::E - 1) / T::E;
    *lds = (int)sizeof(double) * K1Layout<ELEM_TRI, P>::size;
}

void tri_k1_config(int P, int N_e, int* blocks, int* lds) {
    switch (P) {
        case 2: return tri_k1_config<2>(N_e, blocks, lds);
        case 3: return tri_k1_config<3>(N_e, blocks, lds);
        case 4: return tri_k1_config<4>(N_e, blocks, lds);
        case 5: return tri_k1_config<5>(N_e, blocks, lds);
        default: return tri_k1_config<6>(N_e, blocks, lds);
    }
}

int tri_nodal_blocks(int P, int N_e) {
    int blocks, lds;
    tri_k1_config(P, N_e, &blocks, &lds);
    return blocks;
}

hipError_t launch_nodal_values_tri_groups(const TriGroups& a, hipStream_t s) {
    int most = 0, blocks = 0;
    for (int P = 2; P <= 6; ++P) {
        if (!a.g[P - 2].blocks1) continue;
        int b, lds;
        tri_k1_config(P, a.g[P - 2].N_e, &b, &lds);
        most = lds > most ? lds : most;
        blocks += a.g[P - 2].blocks1;
    }
    hipLaunchKernelGGL(k_nodal_values_tri_groups, dim3(blocks), dim3(64), most, s, a);
    return hipGetLastError();
}

// ----------------------------------------------------------------------------- time_derivative
template <int ELEM, int P, int VAR>
struct K2Layout {
    using Sh = Shape<ELEM, P>;
    using T = Tune<ELEM, P, VAR>;
    static constexpr int NC = Sh::NC, D = Sh::D, NH = Sh::NH;
    static constexpr int PS = T::TS * T::R;
    static constexpr int off_h = 0;                          // NH x NQ hoisted volume states
    static constexpr int off_L = off_h + NH * Sh::NQ;        // D*D x NQ metric terms
    static constexpr int off_hf = off_L + D * D * Sh::NQ;    // NH x NF hoisted facet states
    static constexpr int off_nJ = off_hf + NH * Sh::NF;      // D x NF scaled normals
    static constexpr int off_st = off_nJ + D * Sh::NF;       // PS x NC staging
    static constexpr int size = off_st + PS * NC;
    // phase-3 aliases
    static constexpr int off_r = off_h;    // NC x NQ (r_q, then V output)
    static constexpr int off_y = off_L;    // NC x NP
    static constexpr int off_z = off_hf;   // NC x NZ
    static constexpr int off_W = off_z + NC * Sh::NZ;  // NC x NW
    static_assert(NC * Sh::NQ <= NH * Sh::NQ, "r_q alias");
    static_assert(NC * Sh::NP <= D * D * Sh::NQ, "y alias");
    static_assert(off_W + NC * Sh::NW <= size, "sum-factorisation temporaries alias");
    static_assert(Sh::NF <= PS, "facet flux alias in staging");
};

template <int ELEM, int P, int VAR>
__global__ void __launch_bounds__((Tune<ELEM, P, VAR>::TS * Tune<ELEM, P, VAR>::EPB))
k_time_derivative_tensor(TensorParams tp, double* __restrict__ dudt, RKStage rk) {
    using Sh = Shape<ELEM, P>;
    using T = Tune<ELEM, P, VAR>;
    using SF = SumFact<ELEM, P, T::TS>;
    using L = K2Layout<ELEM, P, VAR>;
    constexpr int D = Sh::D, NC = Sh::NC, NH = Sh::NH, NP = Sh::NP, NQ = Sh::NQ, NF = Sh::NF, NPF = Sh::NPF;
    constexpr int TS = T::TS, PS = L::PS, MAXW = TENSOR_MAXW;
    static_assert(NQ <= TS && NF <= TS, "one node per thread");
    extern __shared__ double smem[];
    const DevParams& p = tp.base;
    const int team = threadIdx.x / TS, tl = threadIdx.x - team * TS;
    const int k = element_of_block(blockIdx.x, gridDim.x, tp.xcd_remap) * T::EPB + team;
    const bool valid = k < p.N_e;
    const int kk = valid ? k : 0;
    double* sm = smem + team * L::size;
    double* sh = sm + L::off_h;
    double* sL = sm + L::off_L;
    double* shf = sm + L::off_hf;
    double* snJ = sm + L::off_nJ;
    double* sst = sm + L::off_st;
    using Ph = Physics<D, LAW_EULER>;

    // ---- phase 0: hoist volume and facet states, interface flux
    double r[NC], ff[NC];
#pragma unroll
    for (int e = 0; e < NC; ++e) r[e] = ff[e] = 0.0;
    if (tl < NQ) {
        const double* uqk = p.uq + (size_t)kk * NQ * NC;
        double ub[NC], h[NH];
#pragma unroll
        for (int e = 0; e < NC; ++e) ub[e] = uqk[e * NQ + tl];
        hoist<D>(p.law, ub, h);
#pragma unroll
        for (int v = 0; v < NH; ++v) sh[v * NQ + tl] = h[v];
        const double* Lk = p.Lam + (size_t)kk * NQ * D * D;
#pragma unroll
        for (int mn = 0; mn < D * D; ++mn) sL[mn * NQ + tl] = Lk[mn * NQ + tl];
    }
    if (tl < NF) {
        const int j = tl;
        const double* ufk = p.uf + (size_t)kk * NF * NC;
        double uin[NC], uout[NC], hin[NH], hout[NH], nrm[D], c[NC];
#pragma unroll
        for (int e = 0; e < NC; ++e) uin[e] = ufk[e * NF + j];
        hoist<D>(p.law, uin, hin);
#pragma unroll
        for (int v = 0; v < NH; ++v) shf[v * NF + j] = hin[v];
        const int g = p.mapP[j + (size_t)NF * kk];
        const int kn = g / NF, jn = g - kn * NF;
        const double* ufn = p.uf + (size_t)kn * NF * NC;
#pragma unroll
        for (int e = 0; e < NC; ++e) uout[e] = ufn[e * NF + jn];
        hoist<D>(p.law, uout, hout);
        const double jf = p.Jf[j + (size_t)NF * kk];
        const double inv_jf = 1.0 / jf;
#pragma unroll
        for (int m = 0; m < D; ++m) {
            const double nj = p.nJf[m + D * (j + (size_t)NF * kk)];
            snJ[m * NF + j] = nj;
            nrm[m] = nj * inv_jf;
        }
        ec_dot<D>(p.law, hin, hout, nrm, c);
        const double bj = p.B[j] * jf;
        if (p.law.inviscid_flux == 1) {
            const double a = p.law.half_lambda * wave_speed_h<D>(p.law, hin, hout, nrm);
#pragma unroll
            for (int e = 0; e < NC; ++e) ff[e] = (c[e] + a * (uin[e] - uout[e])) * bj;
        } else {
#pragma unroll
            for (int e = 0; e < NC; ++e) ff[e] = c[e] * bj;
        }
    }
    __syncthreads();

    // ---- phase 1: unique pairs, staged contributions, owner reduction
    const int npairs = tp.n_pairs;
    for (int pass = 0; pass < tp.n_pass; ++pass) {
#pragma unroll
        for (int rr = 0; rr < T::R; ++rr) {
            const int slot = rr * TS + tl;
            const int q = pass * PS + slot;
            if (q < npairs) {
                const int code = tp.pk[q];
                const int i = code & 0xfff, j = (code >> 12) & 0xfff;
                double hi[NH], hj[NH], a[D], c[NC];
#pragma unroll
                for (int v = 0; v < NH; ++v) hi[v] = sh[v * NQ + i];
                if (code >> 24) {  // facet pair: C_ij F(u_i, u_f_j) . (nJf_j + nJq_{f(j), i}) / 2
                    const double cij = tp.cf[q];
                    const int f = j / NPF;
#pragma unroll
                    for (int v = 0; v < NH; ++v) hj[v] = shf[v * NF + j];
#pragma unroll
                    for (int n = 0; n < D; ++n) {
                        double s = snJ[n * NF + j];
#pragma unroll
                        for (int l = 0; l < D; ++l) s += sL[(l + D * n) * NQ + i] * p.fn[l + D * f];
                        a[n] = 0.5 * cij * s;
                    }
                } else {  // volume pair: a_n = sum_m S_m[i,j] (Lambda_i + Lambda_j)[m,n]
#pragma unroll
                    for (int v = 0; v < NH; ++v) hj[v] = sh[v * NQ + j];
                    double sv[D];
#pragma unroll
                    for (int m = 0; m < D; ++m) sv[m] = tp.cf[m * npairs + q];
#pragma unroll
                    for (int n = 0; n < D; ++n) {
                        double s = 0.0;
#pragma unroll
                        for (int m = 0; m < D; ++m)
                            s += sv[m] * (sL[(m + D * n) * NQ + i] + sL[(m + D * n) * NQ + j]);
                        a[n] = s;
                    }
                }
                ec_dot<D>(p.law, hi, hj, a, c);
#pragma unroll
                for (int e = 0; e < NC; ++e) sst[e * PS + slot] = c[e];
            }
        }
        __syncthreads();
        if (tl < NQ) {
            int codes[MAXW];
#pragma unroll
            for (int w = 0; w < MAXW; ++w) codes[w] = w < tp.wv ? tp.vt[(pass * tp.wv + w) * NQ + tl] : -1;
#pragma unroll
            for (int w = 0; w < MAXW; ++w) {
                const int code = codes[w];
                if (code >= 0) {
                    const double sg = (code & 1) ? -1.0 : 1.0;
                    const double* src = sst + (code >> 1);
#pragma unroll
                    for (int e = 0; e < NC; ++e) r[e] += sg * src[e * PS];
                }
            }
        }
        if (tl < NF) {
            int codes[MAXW];
#pragma unroll
            for (int w = 0; w < MAXW; ++w) codes[w] = w < tp.wf ? tp.ft[(pass * tp.wf + w) * NF + tl] : -1;
#pragma unroll
            for (int w = 0; w < MAXW; ++w) {
                const int code = codes[w];
                if (code >= 0) {
                    const double* src = sst + (code >> 1);
#pragma unroll
                    for (int e = 0; e < NC; ++e) ff[e] -= src[e * PS];
                }
            }
        }
        __syncthreads();
    }

    // ---- phase 2: lift r_q -= R' f_f
    double* sff = sst;  // NC x NF
    if (tl < NF) {
#pragma unroll
        for (int e = 0; e < NC; ++e) sff[e * NF + tl] = ff[e];
    }
    __syncthreads();
    double* sr = sm + L::off_r;
    if (tl < NQ) {
        constexpr int MAXR = TENSOR_MAXR;
        int js[MAXR];
        double rvs[MAXR];
#pragma unroll
        for (int w = 0; w < MAXR; ++w) {
            js[w] = w < tp.wrt ? tp.rt_idx[w * NQ + tl] : -1;
            rvs[w] = w < tp.wrt ? tp.rt_val[w * NQ + tl] : 0.0;
        }
#pragma unroll
        for (int w = 0; w < MAXR; ++w) {
            if (js[w] >= 0) {
#pragma unroll
                for (int e = 0; e < NC; ++e) r[e] -= rvs[w] * sff[e * NF + js[w]];
            }
        }
#pragma unroll
        for (int e = 0; e < NC; ++e) sr[e * NQ + tl] = r[e];
    }
    __syncthreads();

    // ---- phase 3: dudt = V' r_q, then the weight-adjusted mass solve
    double* sy = sm + L::off_y;
    double* sZ = sm + L::off_z;
    double* sW = sm + L::off_W;
    SF::Vt(tp, tl, sr, sy, sZ, sW);
    SF::V(tp, tl, sy, sr, sZ, sW);
    const double* Jk = p.Jq + (size_t)kk * NQ;
    for (int i = tl; i < NQ; i += TS) {
        const double jw = p.W[i] / Jk[i];
#pragma unroll
        for (int e = 0; e < NC; ++e) sr[e * NQ + i] *= jw;
    }
    __syncthreads();
    SF::Vt(tp, tl, sr, sy, sZ, sW);
    if (!valid) return;
    const size_t base = (size_t)kk * NP * NC;
    if (!rk.active) {
        for (int t = tl; t < NP * NC; t += TS) dudt[base + t] = sy[t];
    } else {
        for (int t = tl; t < NP * NC; t += TS) {
            const double kt = (rk.A == 0.0 ? 0.0 : rk.A * rk.tmp[base + t]) + rk.dt_of(kk) * sy[t];
            rk.tmp[base + t] = kt;
            rk.u[base + t] += rk.B * kt;
        }
    }
}

// ----------------------------------------------------------------------------- launch
struct TensorConfig {
    int TS, EPB, R, lds1, lds2, NQ, NF, NP;
};

template <int ELEM, int P, int VAR>
TensorConfig tensor_config_of() {
    using Sh = Shape<ELEM, P>;
    using T = Tune<ELEM, P, VAR>;
    return TensorConfig{T::TS, T::EPB, T::R,
                        (int)(sizeof(double) * K1Layout<ELEM, P>::size),
                        (int)(sizeof(double) * K2Layout<ELEM, P, VAR>::size * T::EPB), Sh::NQ, Sh::NF, Sh::NP};
}

template <int ELEM, int P, int VAR>
hipError_t launch_tensor_t(const TensorParams& tp, const double* u, double* dudt, const RKStage& rk, hipStream_t s,
                           int which) {
    using T = Tune<ELEM, P, VAR>;
    const TensorConfig c = tensor_config_of<ELEM, P, VAR>();
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e1 = hipFuncSetAttribute((const void*)k_nodal_values_tensor<ELEM, P>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, c.lds1);
        hipError_t e2 = hipFuncSetAttribute((const void*)k_time_derivative_tensor<ELEM, P, VAR>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, c.lds2);
        if (e1 != hipSuccess) return e1;
        if (e2 != hipSuccess) return e2;
        attr_set = true;
    }
    if (which & 1) {
        using N = EulerTune<ELEM, P>;
        hipLaunchKernelGGL((k_nodal_values_tensor<ELEM, P>), dim3((tp.base.N_e + N::E - 1) / N::E), dim3(N::TS), c.lds1,
                           s, tp, u);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (which & 2) {
        const int nb = (tp.base.N_e + T::EPB - 1) / T::EPB;
        hipLaunchKernelGGL((k_time_derivative_tensor<ELEM, P, VAR>), dim3(nb), dim3(T::TS * T::EPB), c.lds2, s, tp,
                           dudt, rk);
        return hipGetLastError();
    }
    return hipSuccess;
}

#define SSE_ALL_CASES                                                                               \
    SSE_CASE(ELEM_TRI, 2, 0) SSE_CASE(ELEM_TRI, 3, 0) SSE_CASE(ELEM_TRI, 4, 0) SSE_CASE(ELEM_TRI, 5, 0) \
    SSE_CASE(ELEM_TRI, 6, 0) SSE_CASE(ELEM_TET, 2, 0) SSE_CASE(ELEM_TET, 3, 0) SSE_CASE(ELEM_TET, 4, 0) \
    SSE_CASE(ELEM_TET, 4, 1) SSE_CASE(ELEM_TET, 4, 2) SSE_CASE(ELEM_TET, 5, 0) SSE_CASE(ELEM_TET, 3, 1) \
    SSE_CASE(ELEM_TRI, 4, 1)

// returns false if (elem, P, variant) has no compiled kernels
bool tensor_config(int elem, int P, int var, TensorConfig* c) {
#define SSE_CASE(E, PP, VV) \
    if (elem == E && P == PP && var == VV) { *c = tensor_config_of<E, PP, VV>(); return true; }
    SSE_ALL_CASES
#undef SSE_CASE
    return false;
}

hipError_t launch_tensor(const TensorParams& tp, const double* u, double* dudt, const RKStage& rk, hipStream_t s,
                         int which) {
#define SSE_CASE(E, PP, VV) \
    if (tp.elem == E && tp.P == PP && tp.variant == VV) return launch_tensor_t<E, PP, VV>(tp, u, dudt, rk, s, which);
    SSE_ALL_CASES
#undef SSE_CASE
    return hipErrorInvalidValue;
}

}  // namespace sse
