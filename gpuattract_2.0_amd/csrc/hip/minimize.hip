// Device-resident minimization of many poses with VA13 (va13.h), driven by
// the adjoint: each round scores the points the running minimizers asked
// for (the adjoint reads the number of requests from device memory), then
// k_min_step resumes every minimizer with its value and gradient and appends
// those still running, with their next point, to the next round's list.
// Minimizer states stay in HBM for the whole run; the host only reads the
// number of running poses every few rounds.
//
// The minimizer's variables are (angles, position, receptor modes, ligand
// modes) in double (apps/em/meta.h:90-170); a requested point is rounded to a
// float DOF record before scoring, as the reference builds DOF_6D<float>
// requests; the gradient is the exact dE/dvariables of the adjoint.
#include "device.h"
#include "internal.h"
#include "va13.h"

namespace att {

namespace {

// LDS through LDS-typed pointers (generic ones would be flat accesses): an array
// with one element per pose, P poses side by side, and a pose's view of its
// minimizer state (VaView).
typedef __attribute__((address_space(3))) double LdsDouble;
template <unsigned P>
struct LdsColumn {
    LdsDouble* p;
    __device__ __forceinline__ LdsDouble& operator[](int k) const { return p[(unsigned)k * P]; }
};
template <unsigned P>
struct VaLdsView {
    LdsDouble* st;
    int nmax;
    __device__ __forceinline__ LdsDouble& v(int vec, int k) const { return st[(unsigned)(vec * nmax + k) * P]; }
    __device__ __forceinline__ LdsDouble& h(int k) const { return st[(unsigned)(kVaNumVec * nmax + k) * P]; }
};

// DOF record (pos, ang, modesRec[10], modesLig[10]; or pos, ang) <-> variables.
__device__ inline void dof_to_vars(const float* d, int Mr, int Ml, double* x) {
    for (int k = 0; k < 3; ++k) {
        x[k] = d[3 + k];
        x[3 + k] = d[k];
    }
    for (int m = 0; m < Mr; ++m) x[6 + m] = d[6 + m];
    for (int m = 0; m < Ml; ++m) x[6 + Mr + m] = d[16 + m];
}

template <class X>
__device__ inline void vars_to_dof(X x, int Mr, int Ml, bool modes, float* d) {
    for (int k = 0; k < 3; ++k) {
        d[3 + k] = (float)x[k];
        d[k] = (float)x[3 + k];
    }
    if (modes) {
        for (int m = 0; m < ATT_MODES_MAX; ++m) {
            d[6 + m] = m < Mr ? (float)x[6 + m] : 0.f;
            d[16 + m] = m < Ml ? (float)x[6 + Mr + m] : 0.f;
        }
    }
}

template <class G>
__device__ inline void result_to_grad(const float* r, int Mr, int Ml, bool modes, G g) {
    for (int k = 0; k < 3; ++k) {
        g[k] = r[4 + k];      // dE/dangles
        g[3 + k] = r[1 + k];  // dE/dposition
    }
    if (modes) {
        for (int m = 0; m < Mr; ++m) g[6 + m] = r[7 + m];
        for (int m = 0; m < Ml; ++m) g[6 + Mr + m] = r[17 + m];
    }
}

}  // namespace

__global__ void k_min_start(MinRun R, const float* __restrict__ dofs) {
    const unsigned p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p == 0) {
        R.count[0] = R.npose;
        R.countNext[0] = 0u;
    }
    if (p >= R.npose) return;
    const VaView V{R.st + p, R.npose, R.dim};
    double x[kVaMaxDim], req[kVaMaxDim];
    dof_to_vars(dofs + (size_t)R.ds * p, R.Mr, R.Ml, x);
    for (int i = 0; i < R.dim; ++i) V.v(kVaX, i) = x[i];
    VaState s{};
    s.pc = kVaFresh;
    va_resume(s, V, R.dim, R.ivmax, 0.0, nullptr, req);
    R.sc[p] = s;
    R.list[p] = p;
    vars_to_dof(req, R.Mr, R.Ml, R.modes, R.req + (size_t)R.ds * p);
}

// One wave per workgroup resumes P poses' minimizers.  A minimizer is a long
// serial chain of reads and writes of its vectors and factors; from HBM every
// link waits a memory round trip (4000 poses of 12 variables: 162 us a round).
// The poses' state is therefore copied to LDS (element-major, P poses side by
// side: consecutive lanes, different banks), advanced there and copied back.
// P = 16 so that a few thousand poses are a wave on every CU (8 where 16 poses'
// state would exceed 60 KB): 57 us a round; minimizing 4000 poses (1000/300, 3 + 3
// modes, 60 evaluations) 26.5 -> 19.9 ms.
template <unsigned P>
__global__ __launch_bounds__(64) void k_min_step(MinRun R, const unsigned* __restrict__ listIn,
                                                 const unsigned* __restrict__ countIn,
                                                 const float* __restrict__ reqIn,
                                                 const float* __restrict__ res, unsigned elements) {
    extern __shared__ double s_st[];  // [element][P]
    const unsigned lane = threadIdx.x, t0 = blockIdx.x * P;
    if (t0 == 0 && lane == 0) R.countAfter[0] = 0u;  // read last in the previous round
    const unsigned n = countIn[0];
    if (t0 >= n) return;
    // lane l copies elements l / P, l / P + 64 / P, ... of pose l % P
    const unsigned mine = min(t0 + lane % P, n - 1);
    const unsigned p = listIn[mine];
    double* st = R.st + p;
    for (unsigned e = lane / P; e < elements; e += 64 / P) s_st[e * P + lane % P] = st[(size_t)e * R.npose];
    __syncthreads();
    const unsigned t = t0 + lane;
    const bool active = lane < P && t < n;
    if (active) {
        LdsDouble* const lds = (LdsDouble*)s_st;
        const VaLdsView<P> V{lds + lane, R.dim};
        const float* r = res + (size_t)R.os * t;
        // the gradient and the next point behind the poses' states
        const LdsColumn<P> g{lds + elements * P + lane}, req{g.p + R.dim * P};
        result_to_grad(r, R.Mr, R.Ml, R.modes, g);
        VaState s = R.sc[p];
        const bool more = va_advance(s, V, R.dim, R.ivmax, (double)r[0], g, req);
        R.sc[p] = s;
        if (more) {
            const unsigned slot = atomicAdd(R.count, 1u);
            R.list[slot] = p;
            vars_to_dof(req, R.Mr, R.Ml, R.modes, R.req + (size_t)R.ds * slot);
        } else {
            // the point just scored is the result (the reference reports its
            // solver's last evaluated state and objective)
            const float* q = reqIn + (size_t)R.ds * t;
            float* o = R.dofsOut + (size_t)R.ds * p;
            for (unsigned k = 0; k < R.ds; ++k) o[k] = q[k];
            R.eLast[p] = r[0];
            if (R.eBest) R.eBest[p] = (float)s.gesa;
            if (R.nfun) R.nfun[p] = s.nfun;
        }
    }
    __syncthreads();
    if (t0 + lane % P < n)
        for (unsigned e = lane / P; e < elements; e += 64 / P) st[(size_t)e * R.npose] = s_st[e * P + lane % P];
}

hipError_t launch_min_start(const MinRun& R, const float* dofs, hipStream_t s) {
    hipLaunchKernelGGL(k_min_start, dim3((R.npose + 127) / 128), dim3(128), 0, s, R, dofs);
    return hipGetLastError();
}

hipError_t launch_min_step(const MinRun& R, const unsigned* listIn, const unsigned* countIn,
                           const float* reqIn, const float* res, hipStream_t s) {
    const unsigned elements = (unsigned)va_elements(R.dim);
    const size_t bytes = sizeof(double) * (elements + 2 * R.dim);
    if (16 * bytes <= 60 * 1024)
        hipLaunchKernelGGL(k_min_step<16>, dim3((R.npose + 15) / 16), dim3(64), 16 * bytes, s, R, listIn,
                           countIn, reqIn, res, elements);
    else
        hipLaunchKernelGGL(k_min_step<8>, dim3((R.npose + 7) / 8), dim3(64), 8 * bytes, s, R, listIn,
                           countIn, reqIn, res, elements);
    return hipGetLastError();
}

}  // namespace att
