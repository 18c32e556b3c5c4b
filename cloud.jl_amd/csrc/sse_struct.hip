// sse_struct.hip -- time_derivative for ModalTensor Tri/Tet (Euler, FluxDifferencingForm,
// entropy-conservative two-point flux) driven by the tensor-line structure of
// the operators instead of pair tables.
//
// The union sparsity of S_1..S_d on collapsed-coordinate tensor elements is a
// set of 1D lines (src/Solvers/operators.jl:182-200 with D_xi of
// src/SpatialDiscretizations/SpatialDiscretizations.jl:414-418): node i pairs
// with every node j that differs from i in exactly one tensor index (family f).
// Each unordered volume pair is evaluated once, by the thread of one of its nodes
// (cyclic offsets along the line), and its term
//   c_e = sum_n a_n F(u_i, u_j)[e,n],  a_n = sum_m S_m[i,j] (Lambda_i + Lambda_j)[m,n]
// enters r_q[i] as -c (in registers) and r_q[j] as +c (S antisymmetric, F
// symmetric; an LDS atomic add): the reference's scatter over i < j,
// src/Solvers/flux_differencing_form.jl:37-75. Each facet-correction pair (C
// nonzero) is evaluated once too, by column chunks balanced across the team: the
// same two-point term enters the volume node's row and the facet node's column,
// both accumulated in LDS with atomic adds. These atomic sums are the only ones
// whose order varies from run to run.
//
// A team of TS threads owns one element. The exterior facet state is read
// contiguously: phase 1 writes each facet state also into the neighbour's
// exterior slot (the reference's u_f[CI[mapP[:,k]], :] gather).
//
// The lift, V' and the mass solve at the end took 37 % of a workgroup's life at Tet p = 4 with a
// node per thread (table rows of R', every multiply-add reading LDS, 9.8 KB of kept matrix). On
// lines (EulerLines, NodeLift) the residual of 24,576 elements went from 595 to 557 us.
#include <hip/hip_runtime.h>

#include "sse_lines.h"

namespace sse {

// team size, elements per block, threads per node (SPLIT threads share a
// node's partner list; their partial sums meet in LDS)
template <int ELEM, int P>
struct StructTune;
// WAVES: waves per SIMD the register allocation must allow (the LDS of Tet p = 4
// allows 4; one more register would drop it to 3)
template <int P> struct StructTune<ELEM_TRI, P> { static constexpr int TS = 64, EPB = 2, SPLIT = 1, WAVES = 1; };
template <> struct StructTune<ELEM_TET, 2> { static constexpr int TS = 64, EPB = 1, SPLIT = 1, WAVES = 1; };
template <> struct StructTune<ELEM_TET, 3> { static constexpr int TS = 128, EPB = 1, SPLIT = 2, WAVES = 4; };
template <> struct StructTune<ELEM_TET, 4> { static constexpr int TS = 256, EPB = 1, SPLIT = 2, WAVES = 4; };
template <> struct StructTune<ELEM_TET, 5> { static constexpr int TS = 256, EPB = 1, SPLIT = 1, WAVES = 1; };

template <int ELEM, int P>
struct StructLayout {
    using Sh = Shape<ELEM, P>;
    using T = StructTune<ELEM, P>;
    static constexpr int NC = Sh::NC, D = Sh::D, NH = Sh::NH;
    // facet column chunks per element (N1 entries each): faces with one volume
    // line per facet node, plus N1 chunks per node of a face coupled to N1^2 nodes
    static constexpr int ITEMS = ELEM == ELEM_TET ? 3 * Sh::N1 * Sh::N1 + Sh::N1 * Sh::N1 * Sh::N1 : 3 * Sh::N1;
    static constexpr int MAXITEM = (ITEMS + T::TS - 1) / T::TS * T::TS;
    static constexpr int off_h = 0;                            // NH x NQ
    static constexpr int off_L = off_h + NH * Sh::NQ;          // D*D x NQ
    static constexpr int off_hf = off_L + D * D * Sh::NQ;      // NH x NF
    static constexpr int off_nJ = off_hf + NH * Sh::NF;        // D x NF
    static constexpr int off_st = off_nJ + D * Sh::NF;         // row and facet accumulators of C
    static constexpr int ST = NC * (Sh::NQ + Sh::NF) > NC * MAXITEM ? NC * (Sh::NQ + Sh::NF) : NC * MAXITEM;
    static constexpr int off_fn = off_st + ST;                 // D x NFAC reference face normals
    static constexpr int size = off_fn + D * Sh::NFAC;
    // after the pair phase, in the space of the states and the metric
    using Lines = EulerLines<ELEM, P, 1, T::TS>;
    static constexpr int off_ff = 0;                           // NC x NF facet fluxes
    static constexpr int off_rb = off_ff + NC * Sh::NF;        // NC x NQ partial rows of split threads
    static constexpr int off_x = off_rb + (T::SPLIT > 1 ? NC * Sh::NQ : 0);  // NC columns of r_q
    static constexpr int off_woj = off_x + NC * Lines::NX;     // W / J
    static constexpr int off_f1 = off_woj + Lines::NX;         // stage-1 tables of V
    // The kept inverse mass matrix: a row of up to 20 entries per thread spares three short
    // stages (ten RK steps of 2,058 Tet p = 3 elements 2,330 -> 2,160 us without it and with it);
    // the 35 of Tet p = 4 cost more in registers and memory than the stages (569 against 621 us
    // at 24,576 elements).
    static constexpr bool KEPT = NC * Sh::NP <= T::TS && Sh::NP <= 20 && Sh::NP <= Sh::NF;
    static_assert(off_f1 + Lines::LF::NT1 <= off_st, "tail of the kernel beside the accumulators");
};


template <int V>
struct IntConst {
    static constexpr int value = V;
};

// DET: the deterministic variant. The partner shares of the volume pairs are added in a
// fixed order (the pairs of one offset at a time, one half-team after the other: the
// targets of one offset are distinct), each volume node evaluates its own row of C, and
// the column sums of C go through per-chunk slots summed in chunk order. The C pairs are
// then evaluated twice (row and column), and no sum depends on the order of atomics.
template <int ELEM, int P, bool DET>
__device__ __forceinline__ void time_derivative_body(const TensorParams& tp, const StructTables& st,
                                                     double* __restrict__ dudt, const RKStage& rk, int block,
                                                     int blocks) {
    using Sh = Shape<ELEM, P>;
    using T = StructTune<ELEM, P>;
    using L = StructLayout<ELEM, P>;
    constexpr int D = Sh::D, NC = Sh::NC, NH = Sh::NH, NP = Sh::NP, NQ = Sh::NQ, NF = Sh::NF, NPF = Sh::NPF;
    constexpr int N1 = Sh::N1, TS = T::TS, MAXITEM = L::MAXITEM, SPLIT = T::SPLIT, NT = TS / SPLIT;
    // volume pairs: on each line node a evaluates its pairs with the nodes at cyclic
    // offsets 1..DH from it, which covers every unordered pair of an odd-length line
    // once; on an even-length line the offset N1/2 pairs nodes both ways and only
    // the node in the lower half of the line evaluates it
    constexpr int DH = (N1 - 1) / 2, EVEN = N1 % 2 == 0 ? 1 : 0, PER_F = DH + EVEN;
    constexpr int NPART = D * PER_F, QH = (NPART + SPLIT - 1) / SPLIT;  // volume pairs per thread
    static_assert(NQ <= NT && NF <= NT, "one node per thread");
    extern __shared__ double smem[];
    const DevParams& p = tp.base;
    const int team = threadIdx.x / TS, tt = threadIdx.x - team * TS;
    const int half = tt / NT, tl = tt - half * NT;  // node index tl, partner share `half`
    double* sm = smem + team * L::size;
    double* sh = sm + L::off_h;
    double* sL = sm + L::off_L;
    double* shf = sm + L::off_hf;
    double* snJ = sm + L::off_nJ;
    double* sst = sm + L::off_st;
    using Ph = Physics<D, LAW_EULER>;

    const double Wi = tl < NQ ? p.W[tl] : 0.0;
    const double Bj = tl < NF ? p.B[tl] : 0.0;

    // ---- prefetch registers. With two threads per node, the first half-team loads and
    // hoists the volume nodes and the second the facet nodes (the interface flux is the
    // longer chain of the two)
    constexpr int FH = SPLIT - 1;
    double pu[NC], pL[D * D], pJ, pf[NC], px[NC], pn[D], pJf;
    auto prefetch = [&](int k) {
        if (half == 0 && tl < NQ) {
            const double* uqk = p.uq + (size_t)k * NQ * NC;
            const double* Lk = p.Lam + (size_t)k * NQ * D * D;
#pragma unroll
            for (int e = 0; e < NC; ++e) pu[e] = uqk[e * NQ + tl];
#pragma unroll
            for (int mn = 0; mn < D * D; ++mn) pL[mn] = Lk[mn * NQ + tl];
            pJ = p.Jq[(size_t)k * NQ + tl];
        }
        if (FH == 0 && tl < NF) {
            const double* ufk = p.uf + (size_t)k * NF * NC;
            const double* uxk = st.uf_ext + (size_t)k * NF * NC;
#pragma unroll
            for (int e = 0; e < NC; ++e) {
                pf[e] = ufk[e * NF + tl];
                px[e] = uxk[e * NF + tl];
            }
#pragma unroll
            for (int m = 0; m < D; ++m) pn[m] = p.nJf[m + D * (tl + (size_t)NF * k)];
            pJf = p.Jf[tl + (size_t)NF * k];
        }
    };

    // one element per team; a team past the last element computes on a valid
    // element (block-wide barriers) and stores nothing
    const int last = p.N_e - 1;
    const int kb = element_of_block(block, blocks, tp.xcd_remap) * T::EPB;
    {
        const int k = min(kb + team, last);
        const bool valid = kb + team < p.N_e;
        prefetch(k);
        // ---- phase A: hoist, interface flux; clear the facet-correction accumulators
        double* srow = sst;            // NC x NQ: C-row sums of the volume nodes
        double* sfac = sst + NC * NQ;  // NC x NF: C-column sums of the facet nodes
        double* sfn = sm + L::off_fn;
        // the row accumulators start at zero; each facet node's column accumulator starts at
        // minus its interface flux (written below by the node's thread), so that phase D reads
        // f_f - (column sums of C) from one place and the flux needs no register meanwhile
        for (int t = tt; t < NC * NQ; t += TS) sst[t] = 0.0;
        if (tt < D * Sh::NFAC) sfn[tt] = p.fn[tt];
        double hi[NH], Li[D * D], r[NC], ff[NC], Ji = 1.0;
#pragma unroll
        for (int e = 0; e < NC; ++e) r[e] = ff[e] = 0.0;
        if (half == 0 && tl < NQ) {
            hoist<D>(p.law, pu, hi);
#pragma unroll
            for (int v = 0; v < NH; ++v) sh[v * NQ + tl] = hi[v];
#pragma unroll
            for (int mn = 0; mn < D * D; ++mn) {
                Li[mn] = pL[mn];
                sL[mn * NQ + tl] = pL[mn];
            }
            Ji = pJ;
        }
        if (half == FH && tl < NF) {
            if constexpr (FH > 0) {  // the facet loads of the second half-team
                const double* ufk = p.uf + (size_t)k * NF * NC;
                const double* uxk = st.uf_ext + (size_t)k * NF * NC;
#pragma unroll
                for (int e = 0; e < NC; ++e) {
                    pf[e] = ufk[e * NF + tl];
                    px[e] = uxk[e * NF + tl];
                }
#pragma unroll
                for (int m = 0; m < D; ++m) pn[m] = p.nJf[m + D * (tl + (size_t)NF * k)];
                pJf = p.Jf[tl + (size_t)NF * k];
            }
            double hin[NH], hout[NH], nrm[D], c[NC];
            hoist<D>(p.law, pf, hin);
            hoist<D>(p.law, px, hout);
#pragma unroll
            for (int v = 0; v < NH; ++v) shf[v * NF + tl] = hin[v];
            const double inv_jf = 1.0 / pJf;
#pragma unroll
            for (int m = 0; m < D; ++m) {
                snJ[m * NF + tl] = pn[m];
                nrm[m] = pn[m] * inv_jf;
            }
            ec_dot<D>(p.law, hin, hout, nrm, c);
            const double bj = Bj * pJf;
            if (p.law.inviscid_flux == 1) {
                const double al = p.law.half_lambda * wave_speed_h<D>(p.law, hin, hout, nrm);
#pragma unroll
                for (int e = 0; e < NC; ++e) ff[e] = (c[e] + al * (pf[e] - px[e])) * bj;
            } else {
#pragma unroll
                for (int e = 0; e < NC; ++e) ff[e] = c[e] * bj;
            }
            if constexpr (!DET) {
#pragma unroll
                for (int e = 0; e < NC; ++e) sfac[e * NF + tl] = -ff[e];
            }
        }
        __syncthreads();

        // ---- phase B: volume Hadamard row of node tl
        if (SPLIT > 1 && half > 0 && tl < NQ) {
#pragma unroll
            for (int v = 0; v < NH; ++v) hi[v] = sh[v * NQ + tl];
#pragma unroll
            for (int mn = 0; mn < D * D; ++mn) Li[mn] = sL[mn * NQ + tl];
        }
        if (tl < NQ) {
            // tensor indices of node tl (last index fastest) and the family strides
            const int a_last = tl % N1, a_mid = (tl / N1) % N1, a_first = tl / (N1 * N1);
            // pair q of this node: family f, partner index b on the line, partner node j;
            // `act` is false for the offset N1/2 of an even line taken by the other node
            auto pair_of = [&](int q, int& f, int& b, int& j, bool& act) {
                f = q / PER_F;
                const int dlt = q - f * PER_F + 1;
                const int stride = D == 3 ? (f == 0 ? N1 * N1 : (f == 1 ? N1 : 1)) : (f == 0 ? N1 : 1);
                const int af = D == 3 ? (f == 0 ? a_first : (f == 1 ? a_mid : a_last)) : (f == 0 ? a_mid : a_last);
                act = !(EVEN && 2 * dlt == N1 && 2 * af >= N1);
                b = af + dlt < N1 ? af + dlt : af + dlt - N1;
                j = tl + (b - af) * stride;
            };
            // S_m[i, j] of pair q (the table holds the zeros of m < f too); requested one
            // pair ahead and unconditionally, so that the loads overlap the flux
            // evaluation of the pair before
            auto load_s = [&](int q, double* sv) {
                int f, b, j;
                bool act;
                pair_of(q, f, b, j, act);
                const double* sg = st.SGh + ((f * N1 + b) * D) * NQ + tl;
#pragma unroll
                for (int m = 0; m < D; ++m) sv[m] = sg[m * NQ];
            };
            auto eval = [&](int q, const double* sv) {
                int f, b, j;
                bool act;
                pair_of(q, f, b, j, act);
                if (!act) return;
                double hj[NH], av[D], c[NC];
#pragma unroll
                for (int v = 0; v < NH; ++v) hj[v] = sh[v * NQ + j];
                // -a_n / 2 = sum_{m >= f} (-S_m[i,j] / 2) (Lambda_i + Lambda_j)[m,n]  (S_m = 0 for
                // m < f): the flux is linear in a, so c comes out negated, as both rows take it
#pragma unroll
                for (int n = 0; n < D; ++n) av[n] = 0.0;
#pragma unroll
                for (int m = 0; m < D; ++m) {  // static indices into Li
                    if (m < f) continue;
#pragma unroll
                    for (int n = 0; n < D; ++n) av[n] += sv[m] * (Li[m + D * n] + sL[(m + D * n) * NQ + j]);
                }
                ec_dot_h<D>(p.law, hi, hj, av, c);
                // S antisymmetric, F symmetric: node j's row receives +c, through
                // the row accumulator that phase D subtracts
#pragma unroll
                for (int e = 0; e < NC; ++e) {
                    r[e] += c[e];
                    atomicAdd(&srow[e * NQ + j], c[e]);
                }
            };
            if constexpr (!DET) {
                // the half-team's pairs with compile-time pair indices (half is uniform over
                // a wavefront): the family of each pair, and with it the S_m that vanish, is
                // then known, and the straight-line code lets the next pair's loads overlap
                auto sweep = [&](auto hc) {
                    constexpr int H = decltype(hc)::value;
                    constexpr int Q0 = H * QH, Q1 = (H + 1) * QH < NPART ? (H + 1) * QH : NPART;
                    double sv[2][D];  // the S values of a pair are requested one pair ahead
                    load_s(Q0, sv[0]);
#pragma unroll
                    for (int q = Q0; q < Q1; ++q) {
                        if (q + 1 < Q1) load_s(q + 1, sv[(q + 1 - Q0) & 1]);
                        eval(q, sv[(q - Q0) & 1]);
                    }
                };
                if (half == 0) {
                    sweep(IntConst<0>{});
                } else if constexpr (SPLIT > 1) {
                    sweep(IntConst<1>{});
                }
            }
        }
        if constexpr (DET) {
            // the same pairs, every thread through QH trips: at each trip the half-teams
            // add their partner shares one after the other (plain read-add-write: within a
            // half-team, the partners of one offset are distinct nodes)
#pragma unroll 1
            for (int t = 0; t < QH; ++t) {
                const int q = half * QH + t;
                const bool has = tl < NQ && q < NPART && q < (half + 1) * QH;
                double c[NC];
                int jd = 0;
                bool act = false;
                if (has) {
                    const int a_last = tl % N1, a_mid = (tl / N1) % N1, a_first = tl / (N1 * N1);
                    const int f = q / PER_F, dlt = q - f * PER_F + 1;
                    const int stride = D == 3 ? (f == 0 ? N1 * N1 : (f == 1 ? N1 : 1)) : (f == 0 ? N1 : 1);
                    const int af = D == 3 ? (f == 0 ? a_first : (f == 1 ? a_mid : a_last)) : (f == 0 ? a_mid : a_last);
                    act = !(EVEN && 2 * dlt == N1 && 2 * af >= N1);
                    const int b = af + dlt < N1 ? af + dlt : af + dlt - N1;
                    jd = tl + (b - af) * stride;
                    if (act) {
                        double hj[NH], av[D];
#pragma unroll
                        for (int v = 0; v < NH; ++v) hj[v] = sh[v * NQ + jd];
#pragma unroll
                        for (int n = 0; n < D; ++n) av[n] = 0.0;
#pragma unroll
                        for (int m = 0; m < D; ++m) {
                            if (m < f) continue;
                            const double sv = st.SGh[((f * N1 + b) * D + m) * NQ + tl];
#pragma unroll
                            for (int n = 0; n < D; ++n) av[n] += sv * (Li[m + D * n] + sL[(m + D * n) * NQ + jd]);
                        }
                        ec_dot_h<D>(p.law, hi, hj, av, c);  // negated, as above
#pragma unroll
                        for (int e = 0; e < NC; ++e) r[e] += c[e];
                    }
                }
#pragma unroll 1
                for (int h = 0; h < SPLIT; ++h) {
                    if (has && act && half == h) {
#pragma unroll
                        for (int e = 0; e < NC; ++e) srow[e * NQ + jd] += c[e];
                    }
                    __syncthreads();
                }
            }
            // the partner shares into the node's row; the accumulator area is then free
            if (half == 0 && tl < NQ) {
#pragma unroll
                for (int e = 0; e < NC; ++e) r[e] -= srow[e * NQ + tl];
            }
            __syncthreads();
            // the node's own row of C (entries split between the half-teams)
            if (tl < NQ) {
#pragma unroll 1
                for (int w = half; w < st.rw; w += SPLIT) {
                    const int j = st.cr_j[w * NQ + tl];
                    if (j < 0) break;
                    const double cv = st.cr_v[w * NQ + tl];
                    const int fc = j / NPF;
                    double hj[NH], av[D], c[NC];
#pragma unroll
                    for (int v = 0; v < NH; ++v) hj[v] = shf[v * NF + j];
#pragma unroll
                    for (int n = 0; n < D; ++n) {
                        double s = snJ[n * NF + j];
#pragma unroll
                        for (int l = 0; l < D; ++l) s += sL[(l + D * n) * NQ + tl] * sfn[l + D * fc];
                        av[n] = 0.25 * cv * s;  // half the contraction vector
                    }
                    ec_dot_h<D>(p.law, hi, hj, av, c);
#pragma unroll
                    for (int e = 0; e < NC; ++e) r[e] -= c[e];
                }
            }
        }
        // ---- phase C: facet-correction pairs by column chunks, both sums by LDS atomics
#pragma unroll 1
        for (int it = 0; it < MAXITEM / TS; ++it) {
            const int item = it * TS + tt;
            if (item >= st.n_items) continue;  // the chunks are packed: items below n_items are real
            // the chunk (facet node, N1 volume nodes and C entries) requested at once
            const int j = st.ci_j[item];
            int ci[N1];
#pragma unroll
            for (int w = 0; w < N1; ++w) ci[w] = st.ci_i[w * MAXITEM + item];
            const int fc = j / NPF;
            double hj[NH], fnl[D], nj[D], part[NC];
#pragma unroll
            for (int l = 0; l < D; ++l) fnl[l] = sfn[l + D * fc];
#pragma unroll
            for (int e = 0; e < NC; ++e) part[e] = 0.0;
#pragma unroll
            for (int v = 0; v < NH; ++v) hj[v] = shf[v * NF + j];
#pragma unroll
            for (int n = 0; n < D; ++n) nj[n] = snJ[n * NF + j];
#pragma unroll
            for (int w = 0; w < N1; ++w) {
                const int i = ci[w];
                if (i < 0) continue;
                const double cvw = st.ci_v[w * MAXITEM + item];
                double hv[NH], av[D], c[NC];
#pragma unroll
                for (int v = 0; v < NH; ++v) hv[v] = sh[v * NQ + i];
#pragma unroll
                for (int n = 0; n < D; ++n) {
                    double s = nj[n];
#pragma unroll
                    for (int l = 0; l < D; ++l) s += sL[(l + D * n) * NQ + i] * fnl[l];
                    av[n] = 0.25 * cvw * s;  // half the contraction vector
                }
                ec_dot_h<D>(p.law, hv, hj, av, c);
#pragma unroll
                for (int e = 0; e < NC; ++e) {
                    part[e] += c[e];
                    if constexpr (!DET) atomicAdd(&srow[e * NQ + i], c[e]);
                }
            }
            if constexpr (DET) {
#pragma unroll
                for (int e = 0; e < NC; ++e) sst[e * MAXITEM + item] = part[e];  // the chunk's slot
            } else {
#pragma unroll
                for (int e = 0; e < NC; ++e) atomicAdd(&sfac[e * NF + j], part[e]);
            }
        }
        // the node's weights of R' and this thread's share of the stage-1 tables, requested here
        // so that their latency passes during phase D
        using LN = typename L::Lines;
        NodeLift<ELEM, P> lift;
        if (half == 0 && tl < NQ) lift.request(tp.faces, tl);
        constexpr int NT1 = LN::LF::NT1, IT1 = (NT1 + TS - 1) / TS;
        double f1v[IT1];
#pragma unroll
        for (int q = 0; q < IT1; ++q) f1v[q] = tp.lines.F1[min(tt + q * TS, NT1 - 1)];
        __syncthreads();
        // ---- phase D: the C sums into r (volume nodes) and f_f (facet nodes); f_f to LDS
        double* sff = sm + L::off_ff;
        double* srb = sm + L::off_rb;
        if (SPLIT > 1 && half == 1 && tl < NQ) {
#pragma unroll
            for (int e = 0; e < NC; ++e) srb[e * NQ + tl] = r[e];
        }
        if constexpr (!DET) {
            if (half == 0 && tl < NQ) {  // C-row sums, read before r_q may overwrite them
#pragma unroll
                for (int e = 0; e < NC; ++e) r[e] -= srow[e * NQ + tl];
            }
            if (half == 0 && tl < NF) {
#pragma unroll
                for (int e = 0; e < NC; ++e) sff[e * NF + tl] = -sfac[e * NF + tl];
            }
        } else if (half == FH && tl < NF) {  // the node's chunk slots, in chunk order
            double col[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) col[e] = 0.0;
            const int c0 = st.ci_first[tl], c1 = st.ci_first[tl + 1];
            for (int c = c0; c < c1; ++c) {
#pragma unroll
                for (int e = 0; e < NC; ++e) col[e] += sst[e * MAXITEM + c];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) sff[e * NF + tl] = ff[e] - col[e];
        }
        __syncthreads();
        // ---- phase E: lift r_q -= R' f_f
        double* sx = sm + L::off_x;
        double* woj = sm + L::off_woj;
        double* F1 = sm + L::off_f1;
#pragma unroll
        for (int q = 0; q < IT1; ++q)
            if (tt + q * TS < NT1) F1[tt + q * TS] = f1v[q];
        face_transpose<ELEM, P, NC, TS>(tp.faces, sff, tt);
        __syncthreads();
        if (half == 0 && tl < NQ) {
            using G = LineGrid<ELEM, P>;
            if (SPLIT > 1) {
#pragma unroll
                for (int e = 0; e < NC; ++e) r[e] += srb[e * NQ + tl];
            }
            lift.template apply<NC>(tp.faces, tl, sff, r);
#pragma unroll
            for (int e = 0; e < NC; ++e) sx[e * G::NX + G::position(tl)] = r[e];
            woj[G::position(tl)] = Wi / Ji;
        }
        __syncthreads();
        // ---- phase F: dudt = M^{-1} V' r_q, line by line. M^{-1} = V' diag(W/J) V: the kept
        // matrix where a thread can hold one of its rows (requested before the transform), else
        // (and without kept matrices) V, W/J and V' again
        const LN ln(tp, F1, tt);
        constexpr bool KEPT = L::KEPT;
        if (KEPT && tp.Mw) {
            const bool out = tt < NC * NP;
            const int e = out ? tt / NP : 0, j = tt % NP;
            const size_t o = ((size_t)k * NC + e) * NP + j;
            double m[NP], u0 = 0.0, k0 = 0.0;
            const double* Mk = tp.Mw + (size_t)k * NP * NP + j;  // symmetric: row j as a column
#pragma unroll
            for (int i = 0; i < NP; ++i) m[i] = Mk[(size_t)i * NP];
            if (rk.active) {
                u0 = rk.u[o];
                if (rk.A != 0.0) k0 = rk.tmp[o];
            }
            ln.down3(sx);
            ln.down2(sx);
            double* sy = sm + L::off_ff;  // NC x NP (the facet fluxes are dead)
            if (ln.on1) {
                double x[N1], y[N1];
                line_load<N1, 1>(ln.line1(sx), x);
                LN::LF::down1(F1, ln.m1, x, y);
#pragma unroll
                for (int b = 0; b < N1; ++b)
                    if (b <= ln.md1.lim) sy[ln.c1 * NP + ln.md1.off + b] = y[b];
            }
            __syncthreads();
            if (!valid || !out) return;  // no barrier follows
            double y0 = 0.0, y1 = 0.0;
#pragma unroll
            for (int i = 0; i + 1 < NP; i += 2) {
                y0 += m[i] * sy[e * NP + i];
                y1 += m[i + 1] * sy[e * NP + i + 1];
            }
            if constexpr (NP % 2 == 1) y0 += m[NP - 1] * sy[e * NP + NP - 1];
            const double y = y0 + y1;
            if (!rk.active) {
                dudt[o] = y;
            } else {
                const double kt = rk.A * k0 + rk.dt_of(k) * y;
                rk.tmp[o] = kt;
                if (rk.keep) rk.keep[o] = u0;
                rk.u[o] = u0 + rk.B * kt;
            }
            return;
        }
        const size_t base = ((size_t)k * NC + ln.c1) * NP + ln.md1.off;
        double u0[N1], k0[N1];  // an RK stage's state and register, requested before the transforms
        if (rk.active) {
#pragma unroll
            for (int b = 0; b < N1; ++b) {
                const size_t t = base + min(b, ln.md1.lim);
                u0[b] = rk.u[t];
                k0[b] = rk.A == 0.0 ? 0.0 : rk.tmp[t];
            }
        }
        ln.down3(sx);
        ln.down2(sx);
        ln.turn1(sx);
        ln.up2(sx);
        ln.scale3(sx, woj);
        ln.down2(sx);
        if (!valid || !ln.on1) return;  // no barrier follows
        double x[N1], y[N1];
        line_load<N1, 1>(ln.line1(sx), x);
        LN::LF::down1(F1, ln.m1, x, y);
#pragma unroll
        for (int b = 0; b < N1; ++b) {
            if (b > ln.md1.lim) continue;
            const size_t t = base + b;
            if (!rk.active) {
                dudt[t] = y[b];
            } else {
                const double kt = rk.A * k0[b] + rk.dt_of(k) * y[b];
                rk.tmp[t] = kt;
                if (rk.keep) rk.keep[t] = u0[b];
                rk.u[t] = u0[b] + rk.B * kt;
            }
        }
    }
}

template <int ELEM, int P, bool DET>
__global__ void __launch_bounds__((StructTune<ELEM, P>::TS * StructTune<ELEM, P>::EPB), (StructTune<ELEM, P>::WAVES))
k_time_derivative_struct(TensorParams tp, StructTables st, double* __restrict__ dudt, RKStage rk) {
    time_derivative_body<ELEM, P, DET>(tp, st, dudt, rk, blockIdx.x, gridDim.x);
}

// One RK stage of triangles of several degrees in one launch (see k_nodal_values_tri_groups).
__global__ void __launch_bounds__(128) k_time_derivative_tri_groups(TriGroups a) {
    static_assert(StructTune<ELEM_TRI, 2>::TS * StructTune<ELEM_TRI, 2>::EPB == 128, "the block of every degree");
    static_assert(StructLayout<ELEM_TRI, 6>::size * 16 <= 65536, "LDS without an attribute");
    int block = blockIdx.x;
#define SSE_TRI_GROUP(PP)                                                                                     \
    if (block < a.g[PP - 2].blocks2)                                                                          \
        return time_derivative_body<ELEM_TRI, PP, false>(a.g[PP - 2].params(), a.g[PP - 2].st, nullptr, a.g[PP - 2].rk, \
                                                         block, a.g[PP - 2].blocks2);                         \
    block -= a.g[PP - 2].blocks2;
    SSE_TRI_GROUP(6)
    SSE_TRI_GROUP(5)
    SSE_TRI_GROUP(4)
    SSE_TRI_GROUP(3)
    SSE_TRI_GROUP(2)
#undef SSE_TRI_GROUP
}

struct StructConfig {
    int TS, EPB, lds, max_item;
};

template <int ELEM, int P>
StructConfig struct_config_of() {
    using T = StructTune<ELEM, P>;
    return StructConfig{T::TS, T::EPB, (int)(sizeof(double) * StructLayout<ELEM, P>::size * T::EPB),
                        StructLayout<ELEM, P>::MAXITEM};
}

template <int ELEM, int P, bool DET>
hipError_t launch_struct_v(const TensorParams& tp, const StructTables& st, double* dudt, const RKStage& rk,
                           hipStream_t s, int n_blocks) {
    using T = StructTune<ELEM, P>;
    const StructConfig c = struct_config_of<ELEM, P>();
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)k_time_derivative_struct<ELEM, P, DET>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, c.lds);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    hipLaunchKernelGGL((k_time_derivative_struct<ELEM, P, DET>), dim3(n_blocks), dim3(T::TS * T::EPB), c.lds, s, tp,
                       st, dudt, rk);
    return hipGetLastError();
}

template <int ELEM, int P>
hipError_t launch_struct_t(const TensorParams& tp, const StructTables& st, double* dudt, const RKStage& rk,
                           hipStream_t s, int n_blocks) {
    return st.det ? launch_struct_v<ELEM, P, true>(tp, st, dudt, rk, s, n_blocks)
                  : launch_struct_v<ELEM, P, false>(tp, st, dudt, rk, s, n_blocks);
}

#define SSE_STRUCT_CASES                                                                       \
    SSE_CASE(ELEM_TRI, 2) SSE_CASE(ELEM_TRI, 3) SSE_CASE(ELEM_TRI, 4) SSE_CASE(ELEM_TRI, 5) \
    SSE_CASE(ELEM_TRI, 6) SSE_CASE(ELEM_TET, 2) SSE_CASE(ELEM_TET, 3) SSE_CASE(ELEM_TET, 4) SSE_CASE(ELEM_TET, 5)

template <int ELEM, int P>
int struct_blocks_per_cu() {
    using T = StructTune<ELEM, P>;
    const StructConfig c = struct_config_of<ELEM, P>();
    (void)hipFuncSetAttribute((const void*)k_time_derivative_struct<ELEM, P, false>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, c.lds);
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_time_derivative_struct<ELEM, P, false>, T::TS * T::EPB,
                                                     c.lds) !=
        hipSuccess)
        return 0;
    return nb;
}

int struct_occupancy(int elem, int P) {
#define SSE_CASE(E, PP) \
    if (elem == E && P == PP) return struct_blocks_per_cu<E, PP>();
    SSE_STRUCT_CASES
#undef SSE_CASE
    return 0;
}

bool struct_config(int elem, int P, StructConfig* c) {
#define SSE_CASE(E, PP) \
    if (elem == E && P == PP) { *c = struct_config_of<E, PP>(); return true; }
    SSE_STRUCT_CASES
#undef SSE_CASE
    return false;
}

// the kernel uses each element's kept inverse mass matrix (TensorParams::Mw)
bool struct_keeps_mass(int elem, int P) {
#define SSE_CASE(E, PP) \
    if (elem == E && P == PP) return StructLayout<E, PP>::KEPT;
    SSE_STRUCT_CASES
#undef SSE_CASE
    return false;
}

hipError_t launch_struct(const TensorParams& tp, const StructTables& st, double* dudt, const RKStage& rk,
                         hipStream_t s, int n_blocks) {
#define SSE_CASE(E, PP) \
    if (tp.elem == E && tp.P == PP) return launch_struct_t<E, PP>(tp, st, dudt, rk, s, n_blocks);
    SSE_STRUCT_CASES
#undef SSE_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_time_derivative_tri_groups(const TriGroups& a, hipStream_t s) {
    int lds = 0, blocks = 0;
    for (int P = 2; P <= 6; ++P) {
        if (!a.g[P - 2].blocks2) continue;
        StructConfig c;
        if (!struct_config(ELEM_TRI, P, &c)) return hipErrorInvalidValue;
        lds = c.lds > lds ? c.lds : lds;
        blocks += a.g[P - 2].blocks2;
    }
    hipLaunchKernelGGL(k_time_derivative_tri_groups, dim3(blocks), dim3(128), lds, s, a);
    return hipGetLastError();
}

}  // namespace sse
