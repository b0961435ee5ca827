// tail_util.hpp -- what ends a step: source injection, receivers, energy sums, source trace.
// Shared by the tail kernel of the two-pass schedules and by the whole-grid fused step.
#pragma once

#include "device_util.hpp"

namespace ela3d {

// scale of the data written this step (FP16 storage; 1 otherwise)
template <typename T>
__device__ __forceinline__ float nsc(const TailArgs<T>& A, int q)
{
    if constexpr (std::is_same<T, half_t>::value) return A.scl[54 + q];
    return 1.f;
}
template <typename T>
__device__ __forceinline__ float nisc(const TailArgs<T>& A, int q)
{
    if constexpr (std::is_same<T, half_t>::value) return A.scl[81 + q];
    return 1.f;
}

// source injection into field q at cell o, recording the magnitude written
template <typename T>
__device__ __forceinline__ void inject(const TailArgs<T>& A, int q, int o, typename Arith<T>::R v, float* inj)
{
    stf(A.f[q], o, v, nsc<T>(A, q));
    if constexpr (std::is_same<T, half_t>::value) inj[q] = fabsf((float)v);
}

// stress injection at the source cell: into the side slot where FP16 storage
// keeps the source cell's normal stresses there (see StepArgs::side)
template <typename T>
__device__ __forceinline__ void inject_sigma(const TailArgs<T>& A, int q, int o, typename Arith<T>::R add, float* inj)
{
    if constexpr (std::is_same<T, half_t>::value) {
        if (A.side) {
            A.side[q - 3] = A.side[q - 3] + (float)add;
            return;
        }
    }
    inject(A, q, o, ldf(A.f[q], o, nisc<T>(A, q)) + add, inj);
}

template <typename T>
__device__ __forceinline__ double sigma_at_source(const TailArgs<T>& A, int q, int o)
{
    if constexpr (std::is_same<T, half_t>::value) {
        if (A.side) return (double)A.side[q - 3];
    }
    return (double)ldf(A.f[q], o, nisc<T>(A, q));
}

// Source injection of step `it` (one thread), CPU:604-622
template <typename T>
__device__ __forceinline__ void inject_source(const TailArgs<T>& A, int it, float* inj)
{
    typedef typename Arith<T>::R R;
    if (it - 1 < A.nwavelet) {
        const double st = A.wavelet[it - 1];
        const int o = A.src;
        const R DT = (R)A.dt;
        const R l2m = (R)A.rho[o] * (R)A.cp[o] * (R)A.cp[o];
        switch (A.src_kind) {
        case 0: {  // CPU:620-622
            const R fx = (R)(A.sin_t * st), fy = (R)(A.cos_t * st);
            inject_sigma(A, 3, o, fx * DT * l2m, inj);
            inject_sigma(A, 4, o, fx * DT * l2m, inj);
            inject_sigma(A, 5, o, fy * DT * l2m, inj);
            break;
        }
        case 1: {  // CPU:614-617
            const R fx = (R)(A.sin_t * st), fy = (R)(A.cos_t * st);
            const R rx = ((R)A.rho[o] + (R)A.rho[o - 1]) / (R)2;
            const R ry = ((R)A.rho[o] + (R)A.rho[o + A.nx]) / (R)2;
            inject(A, 0, o, ldf(A.f[0], o, nisc<T>(A, 0)) + fx * DT / rx, inj);
            inject(A, 1, o, ldf(A.f[1], o, nisc<T>(A, 1)) + fy * DT / ry, inj);
            break;
        }
        case 2: {
            const R s = (R)st;
            inject_sigma(A, 3, o, s * DT * l2m, inj);
            inject_sigma(A, 4, o, s * DT * l2m, inj);
            inject_sigma(A, 5, o, s * DT * l2m, inj);
            break;
        }
        default: {  // ZC:451-453
            const R s = (R)st;
            const R rx = ((R)A.rho[o] + (R)A.rho[o - 1]) / (R)2;
            const R ry = ((R)A.rho[o] + (R)A.rho[o + A.nx]) / (R)2;
            const R rz = ((R)A.rho[o] + (R)A.rho[o + A.nxy]) / (R)2;
            inject(A, 0, o, ldf(A.f[0], o, nisc<T>(A, 0)) + s * DT / rx, inj);
            inject(A, 1, o, ldf(A.f[1], o, nisc<T>(A, 1)) + s * DT / ry, inj);
            inject(A, 2, o, ldf(A.f[2], o, nisc<T>(A, 2)) + s * DT / rz, inj);
            break;
        }
        }
    }
}

// The rest of a step's end, for the whole-grid fused step (FP32 and FP64 storage; all threads
// of one workgroup): receiver samples and energy sum of step `it` from the set A.g that holds
// it, the source trace, the instability flag.  The source is already in A.g: a receiver on the
// source cell reads the velocities kept from before (receivers come before the source,
// CPU:593-622).  red: LDS, two doubles per wave.  The order of the energy sum depends on the
// number of threads only.
template <typename T>
__device__ __forceinline__ void record_step(const TailArgs<T>& A, int it, double* red)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    bool bad = false;
    if (A.nrec > 0 && it % A.sample_every == 0) {
        const int s = it / A.sample_every - 1;
        if (s < A.nsamples) {
            for (int r = tid; r < A.nrec; r += nt) {
                const int o = A.rec[3 * r] + A.rec[3 * r + 1] * A.nx + A.rec[3 * r + 2] * A.nxy;
                double* dst = A.seis + (size_t(s) * A.nrec + r) * 3;
                for (int q = 0; q < 3; ++q) {
                    const double v = o == A.src ? A.pre_in[q] : (double)A.g[q][o];
                    dst[q] = v;
                    bad = bad || !isfinite(v);
                }
            }
        }
    }
    if (A.energy_every > 0 && it % A.energy_every == 0 && it / A.energy_every <= A.nenergy) {
        double a = 0.0, b = 0.0;
        for (int q = tid; q < A.nepart; q += 4 * nt) {  // four loads in flight
            double x[4] = {0, 0, 0, 0}, y[4] = {0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (q + u * nt < A.nepart) {
                    x[u] = A.epart[2 * (q + u * nt)];
                    y[u] = A.epart[2 * (q + u * nt) + 1];
                }
            a += (x[0] + x[1]) + (x[2] + x[3]);
            b += (y[0] + y[1]) + (y[2] + y[3]);
        }
        a = wave_sum(a);
        b = wave_sum(b);
        if ((tid & 63) == 0) {
            red[2 * (tid >> 6)] = a;
            red[2 * (tid >> 6) + 1] = b;
        }
        __syncthreads();
        if (tid == 0) {
            a = b = 0.0;
            for (int w = 0; w < nt >> 6; ++w) {
                a += red[2 * w];
                b += red[2 * w + 1];
            }
            const int s = it / A.energy_every - 1;
            A.energy[2 * s] = a * A.evol;
            A.energy[2 * s + 1] = b * A.evol;
            bad = bad || !isfinite(a) || !isfinite(b);
        }
    }
    if (tid == 0)  // as in the two-pass tail: a non-finite source cell marks the shot unstable at every step
        for (int q = 0; q < 6; ++q) {
            const double v = (double)A.g[q][A.src];
            bad = bad || !isfinite(v);
            if (q >= 3 && it < A.nsrctrace) A.srctrace[3 * it + q - 3] = v;
        }
    if (bad) *A.flag = 1;
}

}  // namespace ela3d
