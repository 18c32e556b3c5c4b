// sse_tensor.h -- compile-time element shapes, launch shapes and sum-factorised
// V / V' shared by the tensor-product kernels (ModalTensor Tri/Tet).
#pragma once

#include <hip/hip_runtime.h>

#include "sse_kernels.h"

namespace sse {

enum { ELEM_TRI = 2, ELEM_TET = 3 };

// widest owner-reduction table and R' table the tensor kernels accept (checked on the host)
constexpr int TENSOR_MAXW = 16;
constexpr int TENSOR_MAXR = 10;

template <int ELEM, int P>
struct Shape;

template <int P>
struct Shape<ELEM_TRI, P> {
    static constexpr int D = 2, N1 = P + 1, NQ = N1 * N1, NFAC = 3, NPF = N1, NF = NFAC * NPF;
    static constexpr int NP = (P + 1) * (P + 2) / 2, NC = 4, NH = D + 5;
    static constexpr int NZ = (P + 1) * N1;  // Z[b1][a2]
    static constexpr int NW = 0;
};

template <int P>
struct Shape<ELEM_TET, P> {
    static constexpr int D = 3, N1 = P + 1, NQ = N1 * N1 * N1, NFAC = 4, NPF = N1 * N1, NF = NFAC * NPF;
    static constexpr int NP = (P + 1) * (P + 2) * (P + 3) / 6, NC = 5, NH = D + 5;
    static constexpr int NPAIR12 = (P + 1) * (P + 2) / 2;
    static constexpr int NZ = NPAIR12 * N1;  // Z[q(b1,b2)][a3]
    static constexpr int NW = (P + 1) * N1 * N1;  // W[b1][a2][a3]
};

// Launch shape of the table-driven time_derivative: team size TS, EPB elements per block, R
// pairs per thread per pass.
// V selects among variants of the same (element, degree) compiled for tuning (the other kernels
// have one launch shape each).
template <int ELEM, int P, int V>
struct Tune;
#define SSE_TUNE(E, PP, VV, ts, epb, r)                                                \
    template <>                                                                        \
    struct Tune<E, PP, VV> {                                                           \
        static constexpr int TS = ts, EPB = epb, R = r;                                \
    };
SSE_TUNE(ELEM_TRI, 2, 0, 64, 2, 1)
SSE_TUNE(ELEM_TRI, 3, 0, 64, 2, 2)
SSE_TUNE(ELEM_TRI, 4, 0, 64, 2, 3)
SSE_TUNE(ELEM_TRI, 5, 0, 64, 2, 5)
SSE_TUNE(ELEM_TRI, 6, 0, 64, 2, 7)
SSE_TUNE(ELEM_TET, 2, 0, 64, 2, 3)
SSE_TUNE(ELEM_TET, 3, 0, 128, 1, 3)
SSE_TUNE(ELEM_TET, 4, 0, 128, 1, 2)
SSE_TUNE(ELEM_TET, 4, 1, 128, 2, 2)
SSE_TUNE(ELEM_TET, 4, 2, 128, 1, 1)
SSE_TUNE(ELEM_TET, 5, 0, 256, 1, 2)
SSE_TUNE(ELEM_TET, 3, 1, 64, 2, 3)
SSE_TUNE(ELEM_TRI, 4, 1, 64, 2, 3)
#undef SSE_TUNE

// Line-structured operator tables (host-built from the descriptor's S, C and R).
struct StructTables {
    const double* SG;    // D x N1 x D x NQ: S_m[i, j(i, f, b)], index ((f * N1 + b) * D + m) * NQ + i
    const double* SGh;   // -SG / 2: the forward's volume pairs contract with -a / 2
    const int* ci_i;     // CH x MAXITEM: volume nodes of each column chunk (-1 pad)
    const double* ci_v;  // CH x MAXITEM
    const int* ci_j;     // MAXITEM: facet node of each chunk (-1 = no chunk)
    int ch, n_items;
    const double* uf_ext;  // exterior facet states [k][e][j]
    // deterministic mode: the rows of C (RW x NQ, facet node and entry, -1 pad) and the
    // first chunk of each facet node (NF + 1 prefix offsets into the chunks)
    const int* cr_j;
    const double* cr_v;
    const int* ci_first;
    int rw;
    int det;  // 1: every sum in a fixed order (no atomic accumulation)
};

// Triangles of several degrees in one launch (batched problems): entry P - 2 is the group of
// degree P, if it has elements; the blocks of the higher degrees, whose elements take longer, go
// first. By value, and only what these kernels read (at most 4 KiB of arguments): from a table
// in memory they held every pointer in a spilled scalar register (2,000 register moves).
struct TriGroup {
    int N_e, xcd_remap, blocks1, blocks2;  // blocks of the nodal values and of the time derivative
    LawParams law;
    const double *Jq, *Lam, *nJf, *Jf, *W, *B, *fn;
    const int* mapP;
    double *uq, *uf, *uf_ext;
    int* status;
    const double *VA, *VB, *Mw;
    LineTables lines;
    FaceTables faces;
    StructTables st;
    RKStage rk;

    __host__ void set(const TensorParams& tp, const StructTables& t, const RKStage& r) {
        const DevParams& p = tp.base;
        N_e = p.N_e, xcd_remap = tp.xcd_remap, law = p.law;
        Jq = p.Jq, Lam = p.Lam, nJf = p.nJf, Jf = p.Jf, W = p.W, B = p.B, fn = p.fn, mapP = p.mapP;
        uq = p.uq, uf = p.uf, uf_ext = tp.uf_ext, status = p.status;
        VA = tp.VA, VB = tp.VB, Mw = tp.Mw, lines = tp.lines, faces = tp.faces, st = t, rk = r;
    }
    // the parameters as the kernels of one degree take them (what they do not read stays empty)
    __device__ __forceinline__ TensorParams params() const {
        TensorParams tp = {};
        DevParams& p = tp.base;
        p.N_e = N_e, tp.xcd_remap = xcd_remap, p.law = law;
        p.Jq = Jq, p.Lam = Lam, p.nJf = nJf, p.Jf = Jf, p.W = W, p.B = B, p.fn = fn, p.mapP = mapP;
        p.uq = uq, p.uf = uf, tp.uf_ext = uf_ext, p.status = status;
        tp.VA = VA, tp.VB = VB, tp.Mw = Mw, tp.lines = lines, tp.faces = faces;
        return tp;
    }
};

struct TriGroups {
    TriGroup g[5];
};
static_assert(sizeof(TriGroups) <= 4096, "kernel arguments");

// q index of (b1, b2), b1 + b2 <= P, enumerated with b1 outer: also the mode
// number of (b1, b2) in 2D.
template <int P>
__device__ __forceinline__ constexpr int q_index(int b1, int b2) {
    return b1 * (P + 1) - (b1 * (b1 - 1)) / 2 + b2;
}

// number of 3D modes before (b1, b2, 0)
template <int P>
__device__ __forceinline__ constexpr int mode_offset3(int b1, int b2) {
    int off = 0;
    for (int i = 0; i < b1; ++i) off += (P - i + 1) * (P - i + 2) / 2;
    for (int j = 0; j < b2; ++j) off += P - b1 - j + 1;
    return off;
}

__device__ __forceinline__ int element_of_block(int b, int nb, int remap) {
    if (!remap || (nb & 7)) return b;
    return (b & 7) * (nb >> 3) + (b >> 3);
}

// ----------------------------------------------------------------------------- sum factorisation
// All arrays are component-major LDS arrays: x[e * stride + point]. NCV
// components (conserved variables, or several elements or directions side by
// side) go through together, so each factor entry loaded serves all of them.
template <int ELEM, int P, int TS, int NCV = Shape<ELEM, P>::NC>
struct SumFact;

template <int P, int TS, int NCV>
struct SumFact<ELEM_TRI, P, TS, NCV> {
    using Sh = Shape<ELEM_TRI, P>;
    static constexpr int N1 = Sh::N1, NC = NCV, NP = Sh::NP, NQ = Sh::NQ, NZ = Sh::NZ;

    // y[a1,a2] = sum_b1 A[a1,b1] sum_{b2 <= P-b1} B[a2,b1,b2] x[q(b1,b2)]
    __device__ static void V(const TensorParams& tp, int tl, const double* x, double* y, double* Z, double*) {
        for (int o = tl; o < NZ; o += TS) {
            const int b1 = o / N1, a2 = o - b1 * N1;
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
            const int off = q_index<P>(b1, 0);
            for (int b2 = 0; b2 <= P - b1; ++b2) {
                const double bv = tp.VB[a2 + N1 * (b1 + (P + 1) * b2)];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += bv * x[e * NP + off + b2];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) Z[e * NZ + o] = s[e];
        }
        __syncthreads();
        for (int o = tl; o < NQ; o += TS) {
            const int a1 = o / N1, a2 = o - a1 * N1;
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
#pragma unroll
            for (int b1 = 0; b1 <= P; ++b1) {
                const double av = tp.VA[a1 + N1 * b1];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += av * Z[e * NZ + b1 * N1 + a2];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) y[e * NQ + o] = s[e];
        }
        __syncthreads();
    }

    // y[q(b1,b2)] = sum_a2 B[a2,b1,b2] sum_a1 A[a1,b1] x[a1,a2]
    __device__ static void Vt(const TensorParams& tp, int tl, const double* x, double* y, double* Z, double*) {
        for (int o = tl; o < NZ; o += TS) {
            const int b1 = o / N1, a2 = o - b1 * N1;
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
#pragma unroll
            for (int a1 = 0; a1 < N1; ++a1) {
                const double av = tp.VA[a1 + N1 * b1];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += av * x[e * NQ + a1 * N1 + a2];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) Z[e * NZ + o] = s[e];
        }
        __syncthreads();
        for (int m = tl; m < NP; m += TS) {
            int b1 = 0;
            while (q_index<P>(b1 + 1, 0) <= m && b1 < P) ++b1;
            const int b2 = m - q_index<P>(b1, 0);
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
#pragma unroll
            for (int a2 = 0; a2 < N1; ++a2) {
                const double bv = tp.VB[a2 + N1 * (b1 + (P + 1) * b2)];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += bv * Z[e * NZ + b1 * N1 + a2];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) y[e * NP + m] = s[e];
        }
        __syncthreads();
    }
};

template <int P, int TS, int NCV>
struct SumFact<ELEM_TET, P, TS, NCV> {
    using Sh = Shape<ELEM_TET, P>;
    static constexpr int N1 = Sh::N1, NC = NCV, NP = Sh::NP, NQ = Sh::NQ, NZ = Sh::NZ, NW = Sh::NW;
    static constexpr int NN = N1 * N1;

    __device__ static void decode_q(int q, int& b1, int& b2) {
        b1 = 0;
        while (b1 < P && q_index<P>(b1 + 1, 0) <= q) ++b1;
        b2 = q - q_index<P>(b1, 0);
    }

    // y[a1,a2,a3] = sum A[a1,b1] B[a2,b1,b2] C[a3,b1,b2,b3] x[sigma(b1,b2,b3)]
    __device__ static void V(const TensorParams& tp, int tl, const double* x, double* y, double* Z, double* Wt) {
        for (int o = tl; o < NZ; o += TS) {
            const int q = o / N1, a3 = o - q * N1;
            int b1, b2;
            decode_q(q, b1, b2);
            const int off = mode_offset3<P>(b1, b2);
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
            for (int b3 = 0; b3 <= P - b1 - b2; ++b3) {
                const double cv = tp.VC[a3 + N1 * (b1 + (P + 1) * (b2 + (P + 1) * b3))];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += cv * x[e * NP + off + b3];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) Z[e * NZ + o] = s[e];
        }
        __syncthreads();
        for (int o = tl; o < NW; o += TS) {
            const int b1 = o / NN, a23 = o - b1 * NN, a2 = a23 / N1, a3 = a23 - a2 * N1;
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
            const int q0 = q_index<P>(b1, 0);
            for (int b2 = 0; b2 <= P - b1; ++b2) {
                const double bv = tp.VB[a2 + N1 * (b1 + (P + 1) * b2)];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += bv * Z[e * NZ + (q0 + b2) * N1 + a3];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) Wt[e * NW + o] = s[e];
        }
        __syncthreads();
        for (int o = tl; o < NQ; o += TS) {
            const int a1 = o / NN, a23 = o - a1 * NN;
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
#pragma unroll
            for (int b1 = 0; b1 <= P; ++b1) {
                const double av = tp.VA[a1 + N1 * b1];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += av * Wt[e * NW + b1 * NN + a23];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) y[e * NQ + o] = s[e];
        }
        __syncthreads();
    }

    __device__ static void Vt(const TensorParams& tp, int tl, const double* x, double* y, double* Z, double* Wt) {
        for (int o = tl; o < NW; o += TS) {
            const int b1 = o / NN, a23 = o - b1 * NN;
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
#pragma unroll
            for (int a1 = 0; a1 < N1; ++a1) {
                const double av = tp.VA[a1 + N1 * b1];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += av * x[e * NQ + a1 * NN + a23];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) Wt[e * NW + o] = s[e];
        }
        __syncthreads();
        for (int o = tl; o < NZ; o += TS) {
            const int q = o / N1, a3 = o - q * N1;
            int b1, b2;
            decode_q(q, b1, b2);
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
#pragma unroll
            for (int a2 = 0; a2 < N1; ++a2) {
                const double bv = tp.VB[a2 + N1 * (b1 + (P + 1) * b2)];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += bv * Wt[e * NW + b1 * NN + a2 * N1 + a3];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) Z[e * NZ + o] = s[e];
        }
        __syncthreads();
        for (int m = tl; m < NP; m += TS) {  // one thread per mode (b1, b2, b3)
            int b1, b2, b3;
            decode_mode(m, b1, b2, b3);
            const int q = q_index<P>(b1, b2);
            double s[NC];
#pragma unroll
            for (int e = 0; e < NC; ++e) s[e] = 0.0;
#pragma unroll
            for (int a3 = 0; a3 < N1; ++a3) {
                const double cv = tp.VC[a3 + N1 * (b1 + (P + 1) * (b2 + (P + 1) * b3))];
#pragma unroll
                for (int e = 0; e < NC; ++e) s[e] += cv * Z[e * NZ + q * N1 + a3];
            }
#pragma unroll
            for (int e = 0; e < NC; ++e) y[e * NP + m] = s[e];
        }
        __syncthreads();
    }

    // mode number m -> (b1, b2, b3), modes nested b1, b2, b3 (b3 fastest)
    __device__ static void decode_mode(int m, int& b1, int& b2, int& b3) {
        b1 = 0;
        while (b1 < P && m >= (P - b1 + 1) * (P - b1 + 2) / 2) {
            m -= (P - b1 + 1) * (P - b1 + 2) / 2;
            ++b1;
        }
        b2 = 0;
        while (b2 < P - b1 && m >= P - b1 - b2 + 1) {
            m -= P - b1 - b2 + 1;
            ++b2;
        }
        b3 = m;
    }
};

}  // namespace sse
