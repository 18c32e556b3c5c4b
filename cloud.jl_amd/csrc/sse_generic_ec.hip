// sse_generic_ec.hip -- time_derivative of the Euler equations with the entropy-conservative
// two-point flux, for any element type, degree and sparsity (FluxDifferencingForm).
//
//   time_derivative  src/Solvers/flux_differencing_form.jl:294-347
//   flux_difference! and facet_correction! (sparse and dense)  :1-168
//   mass solve       src/Solvers/mass_matrix.jl:169-196
//
// One workgroup per element, sizes at run time. What bounds it: the two-point fluxes. A dense
// Tet p = 3 element (ModalMulti) has 2,016 volume and 4,096 facet pairs, and evaluating each
// from conservative states (velocities, pressures, two logarithms and seven divides per pair)
// took 1,158 us traced at 10,368 elements; this kernel takes 392 us (162 G fluxes/s; the whole
// residual 1,207 -> 424 us), and a Dormand-Prince step of 216 Hex p = 4 elements 340 -> 214 us:
//   * the states are hoisted per node (logarithms, pressure and velocity once per node), and a
//     pair is one contracted flux ec_dot_h: one refined reciprocal, no logarithm;
//   * a thread stays at one volume node i: its state and metric terms and the sum of its row
//     are registers, so a pair reads only its partner and adds only the partner's share
//     through LDS atomics (five instead of ten, one state instead of two);
//   * every volume pair belongs to one of its two nodes (host-balanced; consecutive nodes have
//     partners at the same cyclic offset, so that the atomic adds of a wavefront go to
//     different rows); the S threads of a node take every S-th entry of its lists;
//   * nJq (the reference normal of each face in the metric of each volume node) is formed once
//     per node and face, not once per pair (the mean of the two normals and the halved
//     contraction vector are the factor of the table's C_ij / 4);
//   * V' r - V' R' f_f is one product with the stacked operator [V; -R V]' over the volume and
//     facet nodes, and the weight-adjusted mass solve one product with the element's kept
//     V' diag(W/J) V (V, W/J, V' where it is not kept).
// DET: no sum depends on the order of atomics. Each node sums its whole row (and each facet
// node its column of C), the S partial sums of a node added in turn; pairs are evaluated twice.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sse_kernels.h"

namespace sse {

namespace {

// Threads of a workgroup by the element's nodes, volume and facet: 512 above 256 (one node per
// thread in the first phase, at least two threads per volume node in the second), else 256. With
// fewer nodes most of 256 threads have nothing to do; that only matters once the elements are more
// than a round of such workgroups, and with fewer threads a node's lists take longer. ModalMulti, us
// per residual with 256 | 128 | 64 threads:
//   Tri p = 2, 18 nodes:    242 elements 19.9 | 19.6 | 19.8    1,568 35.9 | 32.9 | 32.5   3,200 54.1 | 47.9 | 44.5
//   Tri p = 3, 28 nodes:    450 elements 21.6 | 22.0 | 22.7    1,568 35.6 | 34.3 | 34.7   3,200 53.8 | 49.6 | 47.4
//   Tri p = 4, 40 nodes:    450 elements 24.4 | 25.5 | 28.5      800 25.7 | 25.3 | 30.5   3,200 70.2 | 64.7 | 66.7
//   Tri p = 5, 54 nodes:    450 elements 27.1 | 31.2 | 41.3    1,800 61.3 | 63.9 | 77.7
//   Tet p = 2, 63 nodes:  1,296 elements 48.3 | 49.8 | 52.4    4,374 108  | 101  | 110
//   Tet p = 3, 128 nodes:   162 elements 18.2 | 23.6
// (of residuals that overlap on several streams 800 Tri p = 2 elements 12.2 | 10.1 | 10.1, 3,200 Tri
// p = 4 elements 63.1 | 51.8 | 49.2).
__host__ __device__ constexpr int ec_threads(int nodes, int N_e) {
    if (nodes <= 20) return 64;
    if (nodes <= 40) return N_e > 3 * 256 ? 128 : 256;   // three workgroups per compute unit
    if (nodes <= 64) return N_e > 12 * 256 ? 128 : 256;  // twelve
    return nodes <= 256 ? 256 : 512;
}

// LDS of one element (doubles). The state area is dead after the flux phase and then holds
// the partial sums and the transforms of the mass solve.
struct EcLayout {
    int h, hf, L, nq, acc, part, o, size;
    __host__ __device__ EcLayout(const DevParams& p) {
        const int NH = p.d + 5, NC = p.d + 2, nt = ec_threads(p.N_q + p.N_f, p.N_e);
        const bool corr = p.C_kind != 0;
        h = 0;                                            // NH x N_q hoisted volume states
        hf = h + NH * p.N_q;                              // NH x N_f hoisted facet states and
        L = hf + (corr ? (NH + p.d) * p.N_f : 0);         // d x N_f scaled normals (facet correction)
        nq = L + p.d * p.d * p.N_q;                       // N_fac x d x N_q: nJq (facet correction)
        const int states = nq + (corr ? p.N_fac * p.d * p.N_q : 0);
        part = 0;                                         // partial sums [part][c][mode] of the products,
        const int n_part = nt / p.N_p > 1 ? nt / p.N_p : 1;
        const int t = p.has_V ? (n_part * p.N_p > p.N_q ? n_part * p.N_p : p.N_q) * NC : 0;  // or N_q x NC
        o = part + t;                                     // N_p x NC
        const int tail = o + p.N_p * NC;
        acc = states > tail ? states : tail;              // NC x N_q row sums, NC x N_f facet sums
        size = acc + NC * (p.N_q + p.N_f);
    }
};

}  // namespace

// u: the state when the phase-1 arrays are not used (nodal diag-E schemes: u_q = u, u_f a
// selection of it), or null.
template <int D, int EC_NT, bool DET>
__global__ void __launch_bounds__(EC_NT)
    k_time_derivative_ec(DevParams p, const double* __restrict__ u, double* __restrict__ dudt, RKStage rk, ErkTail tail) {
    using Ph = Physics<D, LAW_EULER>;
    constexpr int NC = D + 2, NH = D + 5;
    extern __shared__ double sm[];
    const EcLayout lay(p);
    const int k = blockIdx.x, tid = threadIdx.x;
    const int N_p = p.N_p, N_q = p.N_q, N_f = p.N_f, npf = p.npf;
    const bool corr = p.C_kind != 0, direct = u != nullptr;
    double* sh = sm + lay.h;
    double* shf = sm + lay.hf;
    double* snJ = shf + NH * N_f;
    double* sL = sm + lay.L;
    double* snq = sm + lay.nq;
    double* srq = sm + lay.acc;       // NC x N_q
    double* sff = srq + NC * N_q;     // NC x N_f
    const double* uqk = (direct ? u : p.uq) + (size_t)k * N_q * NC;
    const double* Lk = p.Lam + (size_t)k * N_q * D * D;
    // All states of this element and its facets in units in which node 0 is near one; the row
    // sums are converted back as they are read. Node 0 is requested here and used once a node's
    // own loads are on their way (opaque: else the compiler waits for it before the loop).
    double u0[NC];
#pragma unroll
    for (int e = 0; e < NC; ++e) u0[e] = uqk[N_q * e];
    ElementUnits<D> units;
    auto set_units = [&]() {
        double x[NC];
#pragma unroll
        for (int e = 0; e < NC; ++e) {
            x[e] = u0[e];
            asm volatile("" : "+v"(x[e]));
        }
        units.set(p.law, x);
    };
    if (tid >= N_q + N_f) set_units();

    // hoisted volume states, metric terms; facet nodes: hoisted states and the interface flux
    for (int t = tid; t < N_q + N_f; t += EC_NT) {
        if (t < N_q) {
            double us[NC], h[NH];
#pragma unroll
            for (int e = 0; e < NC; ++e) us[e] = uqk[t + N_q * e];
            double Li[D * D];
#pragma unroll
            for (int mn = 0; mn < D * D; ++mn) Li[mn] = Lk[t + N_q * mn];
            set_units();
            units.in(us);
            hoist<D>(p.law, us, h);
#pragma unroll
            for (int v = 0; v < NH; ++v) sh[v * N_q + t] = h[v];
#pragma unroll
            for (int e = 0; e < NC; ++e) srq[e * N_q + t] = 0.0;
#pragma unroll
            for (int mn = 0; mn < D * D; ++mn) sL[mn * N_q + t] = Li[mn];
            if (corr) {
                for (int f = 0; f < p.N_fac; ++f) {
#pragma unroll
                    for (int n = 0; n < D; ++n) {
                        double s = 0.0;
#pragma unroll
                        for (int l = 0; l < D; ++l) s += Li[l + D * n] * p.fn[l + D * f];
                        snq[(f * D + n) * N_q + t] = s;
                    }
                }
            }
        } else {
            const int j = t - N_q;
            const int g = p.mapP[j + (size_t)N_f * k];
            const double jf = p.Jf[j + (size_t)N_f * k], bj = p.B[j] * jf;
            double nJ[D];
#pragma unroll
            for (int m = 0; m < D; ++m) nJ[m] = p.nJf[D * (j + (size_t)N_f * k) + m];
            const int kn = g / N_f, jn = g - kn * N_f;
            double uin[NC], uout[NC], hin[NH], hout[NH], nrm[D], c[NC];
            if (direct) {
                const int i = p.sel[j], in = p.sel[jn];
                const double* un = u + (size_t)kn * N_q * NC;
#pragma unroll
                for (int e = 0; e < NC; ++e) {
                    uin[e] = uqk[i + N_q * e];
                    uout[e] = un[in + N_q * e];
                }
            } else {
                const double* ufk = p.uf + (size_t)k * N_f * NC;
                const double* ufn = p.uf + (size_t)kn * N_f * NC;
#pragma unroll
                for (int e = 0; e < NC; ++e) {
                    uin[e] = ufk[j + N_f * e];
                    uout[e] = ufn[jn + N_f * e];
                }
            }
            set_units();
            units.in(uin);
            units.in(uout);
            hoist<D>(p.law, uin, hin);
            hoist<D>(p.law, uout, hout);
            const double inv_jf = 1.0 / jf;
#pragma unroll
            for (int m = 0; m < D; ++m) nrm[m] = nJ[m] * inv_jf;
            if (corr) {
#pragma unroll
                for (int v = 0; v < NH; ++v) shf[v * N_f + j] = hin[v];
#pragma unroll
                for (int m = 0; m < D; ++m) snJ[m * N_f + j] = nJ[m];
            }
            ec_dot<D>(p.law, hin, hout, nrm, c);
            const double al =
                p.law.inviscid_flux == 1 ? p.law.half_lambda * wave_speed_h<D>(p.law, hin, hout, nrm) : 0.0;
#pragma unroll
            for (int e = 0; e < NC; ++e) sff[e * N_f + j] = (c[e] + al * (uin[e] - uout[e])) * bj;
        }
    }
    __syncthreads();

    // a/2 of a volume pair, a_n = sum_m S_m[i,j] (Lambda_i + Lambda_j)[m,n]
    auto volume_flux = [&](const double* hi, const double* Li, int j, const double* sv, double* c) {
        double hj[NH], av[D];
#pragma unroll
        for (int v = 0; v < NH; ++v) hj[v] = sh[v * N_q + j];
#pragma unroll
        for (int n = 0; n < D; ++n) {
            av[n] = 0.0;
#pragma unroll
            for (int m = 0; m < D; ++m) av[n] += sv[m] * (Li[m + D * n] + sL[(m + D * n) * N_q + j]);
        }
        ec_dot_h<D>(p.law, hi, hj, av, c);
    };
    // a/2 of a facet pair, a = C_ij (nJ_f,j + nJq_i of j's face) / 2; cq = C_ij / 4, so the sum
    // of the two normals comes in unscaled
    auto facet_flux = [&](const double* hi, int i, int j, double cq, double* c) {
        double hj[NH], av[D];
        const int f = j / npf;
#pragma unroll
        for (int v = 0; v < NH; ++v) hj[v] = shf[v * N_f + j];
#pragma unroll
        for (int n = 0; n < D; ++n) av[n] = cq * (snJ[n * N_f + j] + snq[(f * D + n) * N_q + i]);
        ec_dot_h<D>(p.law, hi, hj, av, c);
    };
    // S threads per node: thread s N_q + i takes entries s, s + S, ... of node i's lists
    const int S = EC_NT / N_q > 1 ? EC_NT / N_q : 1;
    const PairLists& pl = p.pairs;
    auto node_row = [&](int i, int s, double* acc) {
        double hi[NH], Li[D * D], sv[D];
#pragma unroll
        for (int v = 0; v < NH; ++v) hi[v] = sh[v * N_q + i];
#pragma unroll
        for (int mn = 0; mn < D * D; ++mn) Li[mn] = sL[mn * N_q + i];
        int jn = -1;
        double svn[D];
        auto fetch = [&](int w) {  // one entry ahead: the loads overlap the flux before
            jn = w < pl.vol_w ? pl.vol_j[w * N_q + i] : -1;
#pragma unroll
            for (int m = 0; m < D; ++m) svn[m] = w < pl.vol_w ? pl.vol_s[(w * D + m) * N_q + i] : 0.0;
        };
        fetch(s);
        for (int w = s; w < pl.vol_w; w += S) {
            const int j = jn;
#pragma unroll
            for (int m = 0; m < D; ++m) sv[m] = svn[m];
            fetch(w + S);
            if (j < 0) continue;
            double c[NC];
            volume_flux(hi, Li, j, sv, c);
#pragma unroll
            for (int e = 0; e < NC; ++e) {
                acc[e] -= c[e];
                if constexpr (!DET) atomicAdd(&srq[e * N_q + j], c[e]);
            }
        }
        if (!corr) return;
        double cn = 0.0;
        auto fetch_f = [&](int w) {
            jn = w < pl.fac_w ? pl.fac_j[w * N_q + i] : -1;
            cn = w < pl.fac_w ? pl.fac_c[w * N_q + i] : 0.0;
        };
        fetch_f(s);
        for (int w = s; w < pl.fac_w; w += S) {
            const int j = jn;
            const double cq = cn;
            fetch_f(w + S);
            if (j < 0) continue;
            double c[NC];
            facet_flux(hi, i, j, cq, c);
#pragma unroll
            for (int e = 0; e < NC; ++e) {
                acc[e] -= c[e];
                if constexpr (!DET) atomicAdd(&sff[e * N_f + j], -c[e]);
            }
        }
    };
    if constexpr (!DET) {
        for (int t = tid; t < S * N_q; t += EC_NT) {
            const int s = t / N_q, i = t - s * N_q;
            double acc[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) acc[e] = 0.0;
            node_row(i, s, acc);
#pragma unroll
            for (int e = 0; e < NC; ++e) atomicAdd(&srq[e * N_q + i], acc[e]);
        }
        __syncthreads();
    } else {
        // rows, then the columns of C: the partial sums of a node's S threads in turn
        const int rows = (S * N_q + EC_NT - 1) / EC_NT * EC_NT;
        for (int t = tid; t < rows; t += EC_NT) {
            const int s = t / N_q, i = t - s * N_q;
            const bool on = t < S * N_q;
            double acc[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) acc[e] = 0.0;
            if (on) node_row(i, s, acc);
            for (int q = 0; q < S; ++q) {
                if (on && s == q) {
#pragma unroll
                    for (int e = 0; e < NC; ++e) srq[e * N_q + i] += acc[e];
                }
                __syncthreads();
            }
        }
        if (corr) {
            const int Sf = EC_NT / N_f > 1 ? EC_NT / N_f : 1;
            const int cols = (Sf * N_f + EC_NT - 1) / EC_NT * EC_NT;
            for (int t = tid; t < cols; t += EC_NT) {
                const int s = t / N_f, j = t - s * N_f;
                const bool on = t < Sf * N_f;
                double acc[NC];
#pragma unroll
                for (int e = 0; e < NC; ++e) acc[e] = 0.0;
                if (on) {
                    for (int w = s; w < pl.col_w; w += Sf) {
                        const int i = pl.col_i[w * N_f + j];
                        if (i < 0) continue;
                        double hi[NH], c[NC];
#pragma unroll
                        for (int v = 0; v < NH; ++v) hi[v] = sh[v * N_q + i];
                        facet_flux(hi, i, j, pl.col_c[w * N_f + j], c);
#pragma unroll
                        for (int e = 0; e < NC; ++e) acc[e] -= c[e];
                    }
                }
                for (int q = 0; q < Sf; ++q) {
                    if (on && s == q) {
#pragma unroll
                        for (int e = 0; e < NC; ++e) sff[e * N_f + j] += acc[e];
                    }
                    __syncthreads();
                }
            }
        }
    }

    const double* Jk = p.Jq + (size_t)k * N_q;
    double* so = sm + lay.o;
    if (p.has_V) {
        // V' r_q - (R V)' f_f: thread (mode j, part) sums one part of the N_q + N_f nodes for
        // all components (the operator entry serves NC products; the lanes of a part read one
        // node's value), then the parts are added
        double* sp = sm + lay.part;
        const int n_part = EC_NT / N_p > 1 ? EC_NT / N_p : 1;
        const int N_n = N_q + N_f, len = (N_n + n_part - 1) / n_part;
        for (int t = tid; t < n_part * N_p; t += EC_NT) {
            const int part = t / N_p, j = t - part * N_p;
            const int i1 = min(N_n, (part + 1) * len);
            double a[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) a[e] = 0.0;
#pragma unroll 4
            for (int i = part * len; i < i1; ++i) {
                const double q = p.Q[j + (size_t)N_p * i];
                const double* x = i < N_q ? srq + i : sff + (i - N_q);
                const int stride = i < N_q ? N_q : N_f;
#pragma unroll
                for (int e = 0; e < NC; ++e) a[e] += q * x[e * stride];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) sp[(part * NC + e) * N_p + j] = units.out(e, a[e]);
        }
        __syncthreads();
        for (int t = tid; t < N_p * NC; t += EC_NT) {
            double s = 0.0;
            for (int q = 0; q < n_part; ++q) s += sp[q * NC * N_p + t];
            so[t] = s;
        }
        __syncthreads();
        if (p.Mw) {  // the kept weight-adjusted inverse
            const double* Mk = p.Mw + (size_t)k * N_p * N_p;
            for (int t = tid; t < N_p * NC; t += EC_NT) {
                const int e = t / N_p, j = t - e * N_p;
                double s = 0.0;
#pragma unroll 8
                for (int i = 0; i < N_p; ++i) s += Mk[j + (size_t)N_p * i] * so[i + N_p * e];
                sp[t] = s;
            }
            so = sp;
        } else {
            for (int t = tid; t < N_q * NC; t += EC_NT) {  // J^{-1}W (V rhs)
                const int i = t % N_q, e = t / N_q;
                double s = 0.0;
#pragma unroll 8
                for (int j = 0; j < N_p; ++j) s += p.V[i + (size_t)N_q * j] * so[j + N_p * e];
                sp[t] = s * (p.W[i] / Jk[i]);
            }
            __syncthreads();
            for (int t = tid; t < N_p * NC; t += EC_NT) {
                const int j = t % N_p, e = t / N_p;
                double s = 0.0;
#pragma unroll 8
                for (int i = 0; i < N_q; ++i) s += p.Vt[j + (size_t)N_p * i] * sp[i + N_q * e];
                so[t] = s;
            }
        }
    } else {  // r_q - R' f_f, (W J)^{-1}
        for (int t = tid; t < N_q * NC; t += EC_NT) {
            const int i = t % N_q, e = t / N_q;
            double s = srq[t];
#pragma unroll 4
            for (int c = p.Rt_ptr[i]; c < p.Rt_ptr[i + 1]; ++c) s -= p.Rt_val[c] * sff[p.Rt_idx[c] + N_f * e];
            so[t] = units.out(e, s / (p.W[i] * Jk[i]));
        }
    }
    __syncthreads();
    const size_t base = (size_t)k * N_p * NC;
    if (rk.active) {
        for (int t = tid; t < N_p * NC; t += EC_NT) {
            const double kt = (rk.A == 0.0 ? 0.0 : rk.A * rk.tmp[base + t]) + rk.dt_of(k) * so[t];
            rk.tmp[base + t] = kt;
            rk.u[base + t] += rk.B * kt;
        }
        return;
    }
    for (int t = tid; t < N_p * NC; t += EC_NT) {
        const double r = so[t];
        dudt[base + t] = r;
        if (tail.out) {  // the next stage state: this stage's derivative is the last term
            double acc = 0.0;
#pragma unroll 4
            for (int q = 0; q < tail.terms.count; ++q) {
                const int s = tail.terms.idx[q];
                acc += tail.terms.c[q] * (s == tail.stage ? r : tail.K[(size_t)s * tail.n + base + t]);
            }
            tail.out[base + t] = tail.base[base + t] + acc;
        }
    }
}

size_t lds_time_derivative_ec(const DevParams& p) { return sizeof(double) * (size_t)EcLayout(p).size; }

template <int D, int NT, bool DET>
hipError_t launch_ec(const DevParams& p, const double* u, double* dudt, const RKStage& rk, const ErkTail& tail,
                     hipStream_t s) {
    const size_t lds = lds_time_derivative_ec(p);
    if (lds > 64 * 1024) {  // the same limit from every handle and thread
        const hipError_t e = hipFuncSetAttribute((const void*)k_time_derivative_ec<D, NT, DET>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_time_derivative_ec<D, NT, DET>), dim3(p.N_e), dim3(NT), lds, s, p, u, dudt, rk, tail);
    return hipGetLastError();
}

template <int D>
hipError_t launch_ec_d(const DevParams& p, const double* u, double* dudt, const RKStage& rk, const ErkTail& tail,
                       hipStream_t s) {
    auto run = [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        return p.det ? launch_ec<D, NT, true>(p, u, dudt, rk, tail, s)
                     : launch_ec<D, NT, false>(p, u, dudt, rk, tail, s);
    };
    switch (ec_threads(p.N_q + p.N_f, p.N_e)) {
        case 64: return run(std::integral_constant<int, 64>{});
        case 128: return run(std::integral_constant<int, 128>{});
        case 256: return run(std::integral_constant<int, 256>{});
        default: return run(std::integral_constant<int, 512>{});
    }
}

hipError_t launch_time_derivative_ec(const DevParams& p, const double* u, double* dudt, const RKStage& rk,
                                     const ErkTail& tail, hipStream_t s) {
    switch (p.d) {
        case 1: return launch_ec_d<1>(p, u, dudt, rk, tail, s);
        case 2: return launch_ec_d<2>(p, u, dudt, rk, tail, s);
        case 3: return launch_ec_d<3>(p, u, dudt, rk, tail, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace sse
