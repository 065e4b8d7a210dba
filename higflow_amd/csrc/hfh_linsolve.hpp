// Device Krylov solvers for the pressure-Poisson and solver-plugin systems.
//
// CSR operator resident in HBM, all scalars resident on the device (no host
// round trip inside an iteration); the host polls the residual every
// `check_every` iterations.  Dot products are two-stage (per-workgroup
// partials, then one workgroup) and therefore deterministic.
//
//   pcg()       Jacobi-preconditioned CG for SPD systems (the pinned
//               pressure system after symmetric elimination).
//   bicgstab()  right Jacobi-preconditioned BiCGStab for nonsymmetric systems
//               (the solver-plugin default, as -ksp_type bcgs of the reference
//               run lines, higtree/src/solver-petsc.c:387).
//   mixed()     FP64 defect correction around an FP32 inner PCG.
#pragma once
#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <stdexcept>
#include <string>
#include <vector>

#include "hfh_kernels.hpp"
#include "hfh_fused.hpp"
#include "hfh_fdm.hpp"
#include "hfh_nd.hpp"

#define HFH_CHECK(x)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (x);                                                                \
        if (e_ != hipSuccess)                                                               \
            throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e_) +    \
                                     " at " + __FILE__ + ":" + std::to_string(__LINE__));   \
    } while (0)

namespace hfh {

// ------------------------------------------------------------ reductions
template <typename T>
__device__ inline T wave_sum(T v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

template <typename T>
__device__ inline T block_sum(T v) {
    __shared__ T sh[BLOCK / 64];
    v = wave_sum(v);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    T r = 0;
    if (w == 0) {
        r = lane < BLOCK / 64 ? sh[lane] : T(0);
        r = wave_sum(r);
    }
    __syncthreads();
    return r;
}

// scalar slots
enum { S_RHO = 0, S_PQ, S_ALPHA, S_BETA, S_RR, S_RHONEW, S_OMEGA, S_TS, S_TT, S_RV, S_BB, S_NSC };

// q = A p, partial p.q
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_spmv_dot(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                                                    const T *__restrict__ v, const T *__restrict__ p, T *__restrict__ q,
                                                    T *__restrict__ part) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    T acc = 0;
    if (i < n) {
        T s = 0;
        for (int k = rp[i]; k < rp[i + 1]; k++) s += v[k] * p[ci[k]];
        q[i] = s;
        acc = p[i] * s;
    }
    acc = block_sum(acc);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// y = A x (no reduction)
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_spmv(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                                                const T *__restrict__ v, const T *__restrict__ x, T *__restrict__ y) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        T s = 0;
        for (int k = rp[i]; k < rp[i + 1]; k++) s += v[k] * x[ci[k]];
        y[i] = s;
    }
}

// sums nb partials of up to 2 arrays into sc[o1], sc[o2]
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_reduce(int nb, const T *__restrict__ p1, const T *__restrict__ p2,
                                                  T *sc, int o1, int o2) {
    T a = 0, b = 0;
    for (int i = threadIdx.x; i < nb; i += BLOCK) {
        a += p1[i];
        if (p2) b += p2[i];
    }
    a = block_sum(a);
    b = block_sum(b);
    if (threadIdx.x == 0) {
        sc[o1] = a;
        if (p2) sc[o2] = b;
    }
}

// CG: alpha = rho / pq
template <typename T>
__global__ void k_cg_alpha(T *sc) {
    if (threadIdx.x == 0) {
        T pq = sc[S_PQ];
        sc[S_ALPHA] = pq != T(0) ? sc[S_RHO] / pq : T(0);
    }
}

// x += a p; r -= a q; z = dinv r; partials r.z and r.r
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_cg_update(int n, T *__restrict__ x, T *__restrict__ r,
                                                     const T *__restrict__ p, const T *__restrict__ q,
                                                     const T *__restrict__ dinv, T *__restrict__ z,
                                                     const T *__restrict__ sc, T *__restrict__ prz,
                                                     T *__restrict__ prr) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    T rz = 0, rr = 0;
    if (i < n) {
        T a = sc[S_ALPHA];
        x[i] = x[i] + a * p[i];
        T ri = r[i] - a * q[i];
        r[i] = ri;
        T zi = dinv[i] * ri;
        z[i] = zi;
        rz = ri * zi;
        rr = ri * ri;
    }
    rz = block_sum(rz);
    rr = block_sum(rr);
    if (threadIdx.x == 0) {
        prz[blockIdx.x] = rz;
        prr[blockIdx.x] = rr;
    }
}

template <typename T>
__global__ void k_cg_beta(T *sc) {
    if (threadIdx.x == 0) {
        T rho = sc[S_RHO], rn = sc[S_RHONEW];
        sc[S_BETA] = rho != T(0) ? rn / rho : T(0);
        sc[S_RHO] = rn;
    }
}

template <typename T>
__global__ void __launch_bounds__(BLOCK) k_cg_p(int n, T *__restrict__ p, const T *__restrict__ z,
                                                const T *__restrict__ sc) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = z[i] + sc[S_BETA] * p[i];
}

// r = b - A x, z = dinv r, p = z, partial r.z, r.r, b.b
template <typename T, typename TB>
__global__ void __launch_bounds__(BLOCK) k_cg_init(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                                                   const T *__restrict__ v, const T *__restrict__ x,
                                                   const TB *__restrict__ b, const T *__restrict__ dinv,
                                                   T *__restrict__ r, T *__restrict__ z, T *__restrict__ p,
                                                   T *__restrict__ prz, T *__restrict__ prr, T *__restrict__ pbb) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    T rz = 0, rr = 0, bb = 0;
    if (i < n) {
        T s = 0;
        for (int k = rp[i]; k < rp[i + 1]; k++) s += v[k] * x[ci[k]];
        T bi = (T)b[i];
        T ri = bi - s;
        r[i] = ri;
        T zi = dinv[i] * ri;
        z[i] = zi;
        p[i] = zi;
        rz = ri * zi;
        rr = ri * ri;
        bb = bi * bi;
    }
    rz = block_sum(rz);
    rr = block_sum(rr);
    bb = block_sum(bb);
    if (threadIdx.x == 0) {
        prz[blockIdx.x] = rz;
        prr[blockIdx.x] = rr;
        pbb[blockIdx.x] = bb;
    }
}

// generic helpers for BiCGStab
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_dot2(int n, const T *__restrict__ a, const T *__restrict__ b,
                                                const T *__restrict__ c, const T *__restrict__ d,
                                                T *__restrict__ p1, T *__restrict__ p2) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    T s1 = 0, s2 = 0;
    if (i < n) {
        s1 = a[i] * b[i];
        if (c) s2 = c[i] * d[i];
    }
    s1 = block_sum(s1);
    s2 = block_sum(s2);
    if (threadIdx.x == 0) {
        p1[blockIdx.x] = s1;
        if (p2) p2[blockIdx.x] = s2;
    }
}

// BiCGStab p = r + beta (p - omega v); ph = dinv p
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_bcg_p(int n, int first, T *__restrict__ p, const T *__restrict__ r,
                                                 const T *__restrict__ vv, const T *__restrict__ dinv,
                                                 T *__restrict__ ph, const T *__restrict__ sc) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        T pi;
        if (first) {
            pi = r[i];
        } else {
            T beta = (sc[S_RHONEW] / sc[S_RHO]) * (sc[S_ALPHA] / sc[S_OMEGA]);
            pi = r[i] + beta * (p[i] - sc[S_OMEGA] * vv[i]);
        }
        p[i] = pi;
        ph[i] = dinv[i] * pi;
    }
}

// s = r - alpha v (alpha = rhonew / rv); sh = dinv s; partial s.s
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_bcg_s(int n, const T *__restrict__ r, const T *__restrict__ vv,
                                                 const T *__restrict__ dinv, T *__restrict__ s, T *__restrict__ sh,
                                                 T *sc, T *__restrict__ pss) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    T alpha = sc[S_RV] != T(0) ? sc[S_RHONEW] / sc[S_RV] : T(0);
    T ss = 0;
    if (i < n) {
        T si = r[i] - alpha * vv[i];
        s[i] = si;
        sh[i] = dinv[i] * si;
        ss = si * si;
    }
    ss = block_sum(ss);
    if (threadIdx.x == 0) pss[blockIdx.x] = ss;
}

template <typename T>
__global__ void k_bcg_alpha(T *sc) {
    if (threadIdx.x == 0) sc[S_ALPHA] = sc[S_RV] != T(0) ? sc[S_RHONEW] / sc[S_RV] : T(0);
}

// x += alpha ph + omega sh; r = s - omega t; partial r.r, rh.r
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_bcg_x(int n, T *__restrict__ x, T *__restrict__ r,
                                                 const T *__restrict__ ph, const T *__restrict__ sh,
                                                 const T *__restrict__ s, const T *__restrict__ t,
                                                 const T *__restrict__ rh, T *sc, T *__restrict__ prr,
                                                 T *__restrict__ prhr) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    T omega = sc[S_TT] > T(0) ? sc[S_TS] / sc[S_TT] : T(0);
    T rr = 0, rhr = 0;
    if (i < n) {
        x[i] = x[i] + sc[S_ALPHA] * ph[i] + omega * sh[i];
        T ri = s[i] - omega * t[i];
        r[i] = ri;
        rr = ri * ri;
        rhr = rh[i] * ri;
    }
    rr = block_sum(rr);
    rhr = block_sum(rhr);
    if (threadIdx.x == 0) {
        prr[blockIdx.x] = rr;
        prhr[blockIdx.x] = rhr;
    }
}

template <typename T>
__global__ void k_bcg_shift(T *sc) {
    if (threadIdx.x == 0) {
        sc[S_OMEGA] = sc[S_TT] > T(0) ? sc[S_TS] / sc[S_TT] : T(0);
        sc[S_RHO] = sc[S_RHONEW];
    }
}

// x += alpha ph (early exit when |s| converged)
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_axpy_sc(int n, T *x, const T *y, const T *sc, int slot) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] + sc[slot] * y[i];
}


template <typename TD, typename TS>
__global__ void __launch_bounds__(BLOCK) k_convert(int n, const TS *a, TD *b) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (TD)a[i];
}

template <typename TD, typename TS>
__global__ void __launch_bounds__(BLOCK) k_add_conv(int n, TD *x, const TS *e) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] + (TD)e[i];
}

// block-diagonal refinement: b32 = s_g r and x += u_g e, with g the segment of
// the BLOCK-row block (segments start on BLOCK boundaries); sc holds s_g for
// g < nseg and u_g at nseg + g
__global__ void __launch_bounds__(BLOCK) k_convert_seg(int n, const double *__restrict__ r, float *__restrict__ b32,
                                                       const int *__restrict__ bseg, const double *__restrict__ sc) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b32[i] = (float)(sc[bseg[blockIdx.x]] * r[i]);
}

__global__ void __launch_bounds__(BLOCK) k_add_conv_seg(int n, double *__restrict__ x, const float *__restrict__ e,
                                                        const int *__restrict__ bseg, const double *__restrict__ sc,
                                                        int nseg) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] + sc[nseg + bseg[blockIdx.x]] * (double)e[i];
}

// r = b - A x (FP64), partial r.r and b.b
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_residual(int n, const int *__restrict__ rp, const int *__restrict__ ci,
                                                    const T *__restrict__ v, const T *__restrict__ x,
                                                    const T *__restrict__ b, T *__restrict__ r, T *__restrict__ prr,
                                                    T *__restrict__ pbb) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    T rr = 0, bb = 0;
    if (i < n) {
        T s = 0;
        for (int k = rp[i]; k < rp[i + 1]; k++) s += v[k] * x[ci[k]];
        T ri = b[i] - s;
        r[i] = ri;
        rr = ri * ri;
        bb = b[i] * b[i];
    }
    rr = block_sum(rr);
    bb = block_sum(bb);
    if (threadIdx.x == 0) {
        prr[blockIdx.x] = rr;
        pbb[blockIdx.x] = bb;
    }
}

// the same with 4 lanes per row: workgroups of 4 BLOCK threads, one per
// BLOCK rows, so the partials have k_residual's layout (one per BLOCK rows);
// prs: the sums of r.  LG = 16 takes the rows in four turns of 16 lanes: the
// least-squares rows of a 3D mesh (30-65 entries on average, up to 200) wait
// for their longest row, 49 us on 4 lanes for 47,592 rows, 36 us on 16.
template <typename T, int LG = 4>
__global__ void __launch_bounds__(4 * BLOCK) k_residual_l4(int n, const int *__restrict__ rp,
                                                           const int *__restrict__ ci, const T *__restrict__ v,
                                                           const T *__restrict__ x, const T *__restrict__ b,
                                                           T *__restrict__ r, T *__restrict__ prr,
                                                           T *__restrict__ pbb, T *__restrict__ prs) {
    const int lane = threadIdx.x % LG;
    T rr = 0, bb = 0, rs = 0;
#pragma unroll
    for (int turn = 0; turn < LG / 4; turn++) {
        const int i = blockIdx.x * BLOCK + turn * (4 * BLOCK / LG) + (int)threadIdx.x / LG;
        T s = 0;
        if (i < n)
            for (int k = rp[i] + lane; k < rp[i + 1]; k += LG) s += v[k] * x[ci[k]];
#pragma unroll
        for (int o = 1; o < LG; o *= 2) s += __shfl_xor(s, o, 64);
        if (i < n && lane == 0) {
            const T bi = b[i], ri = bi - s;
            r[i] = ri;
            rr += ri * ri;
            bb += bi * bi;
            rs += ri;
        }
    }
    rr = wave_sum(rr);
    bb = wave_sum(bb);
    rs = wave_sum(rs);
    __shared__ T srr[4 * BLOCK / 64], sbb[4 * BLOCK / 64], srs[4 * BLOCK / 64];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        srr[w] = rr;
        sbb[w] = bb;
        srs[w] = rs;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        T a = 0, c = 0, e = 0;
        for (int q = 0; q < 4 * BLOCK / 64; q++) {
            a += srr[q];
            c += sbb[q];
            e += srs[q];
        }
        prr[blockIdx.x] = a;
        pbb[blockIdx.x] = c;
        prs[blockIdx.x] = e;
    }
}

// r = b - A x with the matrix in the diagonal form of the Krylov kernels
// (KRows::dblk; rows without a template read CSR), one row per thread in
// 1024-row workgroups; partials r.r, b.b and sum(r) per 256-row block as
// k_residual_l4 writes them (one per BLOCK rows, nb of them).
template <typename T>
__global__ void __launch_bounds__(KNT) k_residual_d(int n, KRows<T> A, const T *__restrict__ x,
                                                    const T *__restrict__ b, T *__restrict__ r, T *__restrict__ prr,
                                                    T *__restrict__ pbb, T *__restrict__ prs, int nb) {
    const int i = blockIdx.x * KNT + (int)threadIdx.x;
    const bool in = i < n;
    const int *db = A.dblk + (size_t)blockIdx.x * (KD_MAX + 1);
    const int nd = db[KD_MAX];
    T xv[KD_MAX];
#pragma unroll
    for (int e = 0; e < KD_MAX; e++) {
        int j = i + db[e];
        j = j < 0 ? 0 : (j >= n ? n - 1 : j);
        xv[e] = (in && e < nd) ? x[j] : T(0);
    }
    const int t = in ? A.code[i] : -1;
    T s = 0;
    if (t >= 0) {
        const unsigned msk = A.dmask[t];
        const T *w = A.dw + (size_t)t * KD_MAX;
#pragma unroll
        for (int e = 0; e < KD_MAX; e++) {
            const T a = w[e];
            if ((msk >> e) & 1u) s += a * xv[e];
        }
    } else if (in) {
        for (int k = A.rp[i]; k < A.rp[i + 1]; k++) s += A.val[k] * x[A.ci[k]];
    }
    T rr = 0, bb = 0, rs = 0;
    if (in) {
        const T bi = b[i], ri = bi - s;
        r[i] = ri;
        rr = ri * ri;
        bb = bi * bi;
        rs = ri;
    }
    rr = wave_sum(rr);
    bb = wave_sum(bb);
    rs = wave_sum(rs);
    __shared__ T srr[KNT / 64], sbb[KNT / 64], srs[KNT / 64];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        srr[w] = rr;
        sbb[w] = bb;
        srs[w] = rs;
    }
    __syncthreads();
    constexpr int WPB = BLOCK / 64;  // waves per 256-row block
    if (threadIdx.x < KNT / BLOCK) {
        const int q = threadIdx.x, pb = blockIdx.x * (KNT / BLOCK) + q;
        T a = 0, c = 0, e = 0;
        for (int k = 0; k < WPB; k++) {
            a += srr[q * WPB + k];
            c += sbb[q * WPB + k];
            e += srs[q * WPB + k];
        }
        if (pb < nb) {
            prr[pb] = a;
            pbb[pb] = c;
            prs[pb] = e;
        }
    }
}

// dst = src in the segments whose flag is set (bseg: segment of each BLOCK
// rows, null for one segment), in the rows that have entries
__global__ void __launch_bounds__(BLOCK) k_seg_copy(int n, const int *__restrict__ rp, const int *__restrict__ bseg,
                                                    const int *flag, const double *__restrict__ src,
                                                    double *__restrict__ dst) {
    const int i = blockIdx.x * BLOCK + (int)threadIdx.x;
    if (i < n && flag[bseg ? bseg[blockIdx.x] : 0] && rp[i + 1] > rp[i]) dst[i] = src[i];
}

// what rounding can leave in the 2-norm of b - A x: partials, per 256-row
// block, of ((len + 2) u |A||x| + u |b|)^2 (len entries of the row, u = 2^-53;
// the sum and the difference as evaluated, and x as rounded), 4 lanes per row
__global__ void __launch_bounds__(4 * BLOCK) k_resid_rounding(int n, const int *__restrict__ rp,
                                                              const int *__restrict__ ci, const double *__restrict__ v,
                                                              const double *__restrict__ x,
                                                              const double *__restrict__ b, double *__restrict__ part) {
    const int lane = threadIdx.x & 3, i = blockIdx.x * BLOCK + (int)threadIdx.x / 4;
    double s = 0;
    if (i < n)
        for (int k = rp[i] + lane; k < rp[i + 1]; k += 4) s += fabs(v[k] * x[ci[k]]);
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    double e = 0;
    if (i < n && lane == 0) {
        e = 0x1p-53 * ((rp[i + 1] - rp[i] + 2) * s + fabs(b[i]));
        e *= e;
    }
    e = wave_sum(e);
    __shared__ double se[4 * BLOCK / 64];
    if ((threadIdx.x & 63) == 0) se[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0;
        for (int q = 0; q < 4 * BLOCK / 64; q++) a += se[q];
        part[blockIdx.x] = a;
    }
}

template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    void alloc(size_t k) {
        free();
        if (k == 0) k = 1;
        HFH_CHECK(hipMalloc((void **)&p, k * sizeof(T)));
        n = k;
    }
    void free() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    void upload(const T *h, size_t k, hipStream_t s) {
        if (k > n) alloc(k);
        if (k) HFH_CHECK(hipMemcpyAsync(p, h, k * sizeof(T), hipMemcpyHostToDevice, s));
    }
    ~DevBuf() { free(); }
};

// Field exchange with host memory through one pinned buffer.  A copy from
// or to pageable memory goes through the runtime's own staging and waits for
// the device each time (15-25 us for a field of a small mesh; the 64-cavity
// sweep exchanges 960 fields of its members between two outputs).  Here a
// write is a memcpy and an enqueued copy, waiting only when the buffer is
// full; a read waits for its own copy.  The copies are kernels on the pinned
// buffer (131 KB: 43 us as an enqueued copy, 12 us so).  One
// buffer per solver, used on its stream only.
struct HostStage {
    static constexpr size_t CAP = 4u << 20;
    char *p = nullptr;
    size_t at = 0;  // bytes of enqueued writes
    HostStage() = default;
    HostStage(const HostStage &) = delete;
    HostStage &operator=(const HostStage &) = delete;
    ~HostStage() {
        if (p) (void)hipHostFree(p);
    }
    void open() {
        if (!p) HFH_CHECK(hipHostMalloc((void **)&p, CAP, hipHostMallocDefault));
    }
    void write(double *dst, const double *src, size_t n, hipStream_t st) {
        open();
        while (n > 0) {
            const size_t k = std::min(n, CAP / 2 / sizeof(double)), b = k * sizeof(double);
            if (at + b > CAP) {
                HFH_CHECK(hipStreamSynchronize(st));
                at = 0;
            }
            std::memcpy(p + at, src, b);
            copy(reinterpret_cast<double *>(p + at), dst, k, st);
            at += (b + 63) / 64 * 64;
            dst += k;
            src += k;
            n -= k;
        }
    }
    // the enqueued writes have left the buffer before the read's copy starts
    void read(double *dst, const double *src, size_t n, hipStream_t st) {
        open();
        while (n > 0) {
            const size_t k = std::min(n, CAP / sizeof(double)), b = k * sizeof(double);
            copy(src, reinterpret_cast<double *>(p), k, st);
            HFH_CHECK(hipStreamSynchronize(st));
            at = 0;
            std::memcpy(dst, p, b);
            dst += k;
            src += k;
            n -= k;
        }
    }

  private:
    // a copy that could not be launched is an error here: the buffer would
    // still hold what an earlier exchange left
    static void copy(const double *src, double *dst, size_t k, hipStream_t st) {
        int n = (int)k;
        void *args[] = {&n, &src, &dst};
        HFH_CHECK(hipLaunchKernel(reinterpret_cast<const void *>(k_copy<double>), dim3(nblocks(n)), dim3(BLOCK), args, 0,
                                  st));
    }
};

struct SolveStats {
    int iters = 0;
    double resid = 0.0;  // ||b - Ax|| / ||b||
    int converged = 0;
    int outer = 0;       // refinement steps (mixed)
    int fallback = 0;    // mixed: the solve finished in FP64
    int restarts = 0;    // fused: restarts on the true residual
};

// A sparse system on one device.
class DeviceSystem {
  public:
    int n = 0, nnz = 0;
    DevBuf<int> rp, ci;
    DevBuf<double> v, dinv;
    DevBuf<float> v32, dinv32;
    DevBuf<double> r, z, p, q, rh, s, sh, t, ph, bb_tmp;
    DevBuf<float> r32, z32, p32, q32, x32, b32;
    DevBuf<double> part1, part2, part3, sc;
    DevBuf<float> fpart1, fpart2, fpart3, fsc;
    int nb = 0;
    int check_every = 8;
    // fused iterations (FP64 solve and FP32 inner solve of the mixed form)
    FusedKrylov<double> k64;
    FusedKrylov<float> k32;
    FdmSolver fdm;  // direct solves of Kronecker-sum matrices
    NdSolver nd;    // and of other matrices whose factors are affordable
    // operations that the set-up may spend on the factors of one matrix (0:
    // none); a 16-core host takes about 2 s for 2e11
    double nd_max_flops = 0;
    // the direct solve wants a coupling of at least this share of the diagonal
    double fdm_min_coupling = 0;
    bool allow_direct = true;
    bool direct() const { return fdm.ready || nd.ready; }
    // work that follows the solve on the stream: a direct solve enqueues it
    // behind its first pass, before the wait; early_done tells whether that
    // was the last word on x (else the caller runs it after the solve)
    std::function<void()> early;
    bool early_done = false;
    bool fused = true;
    int max_restarts = 1;      // fused64: restarts on the true residual
    double t_mixed_ = -1, t_fp64_ = -1;  // mixed form: seconds per solve of each form
    int n32_ = 0, n64_ = 0;              // timed solves of each form
    bool explored_ = false;              // the first six solves are done
    struct Pending {                     // a solve whose time is not booked yet
        bool on = false, use32 = false, ok = false, probing = false, pref32 = false;
    } pend_;
    hipEvent_t tev_[2] = {nullptr, nullptr};
    // the slower form is re-timed every probe_every_ solves; the interval
    // doubles (up to 1600) while the faster form keeps winning, and is 10
    // again after a flip
    int since_probe_ = 0, probe_every_ = 10;
    int nseg = 1;
    std::vector<int> seg_off;
    std::vector<SolveStats> seg_stats;  // last solve, per segment
    std::vector<int> seg_hi_;
    std::vector<double> seg_hs_;
    int off_ks_ = 64, off_sc_ = 256;
    size_t hpin_size_ = 0;
    bool force32_ = false;  // HFH_MIXED_FP32=1: always refine with FP32 solves
    bool mixed_amg32_ = true;  // the mixed form's FP64 solves use the FP32 V-cycle
    int pred32_[3] = {0, 0, 0};  // FP32 iterations of the 1st, 2nd, later corrections
    DevBuf<int> segw_;              // first 256-row block of each segment, and the end
    DevBuf<int> bseg_;              // segment of each BLOCK-row block (nseg > 1)
    DevBuf<double> segsc_;          // per-segment scale s_g and unscale u_g
    std::vector<double> hsegsc_;
    DevBuf<double> xbak;

    DeviceSystem() = default;
    DeviceSystem(const DeviceSystem &) = delete;
    DeviceSystem &operator=(const DeviceSystem &) = delete;
    ~DeviceSystem() {
        clear_graphs();
        if (hpin_) (void)hipHostFree(hpin_);
        for (auto &e : tev_)
            if (e) (void)hipEventDestroy(e);
    }

    // `amg`: precondition the fused BiCGStab with a smoothed-aggregation
    // V-cycle (HFH_AMG=0 turns it off)
    // `segs`: row offsets of independent diagonal blocks (multiples of 1024;
    // see set_blocks), solved together with one stopping test each
    // `amg_max_cx` > 0: the hierarchy is kept only up to that operator
    // complexity (sum over levels of the matrix entries / the fine matrix's)
    void set_matrix(const std::vector<int> &hrp, const std::vector<int> &hci, const std::vector<double> &hv,
                    hipStream_t st, bool amg = false, const std::vector<int> &segs = {}, double amg_max_cx = 0) {
        n = (int)hrp.size() - 1;
        nnz = (int)hci.size();
        rp.upload(hrp.data(), hrp.size(), st);
        ci.upload(hci.data(), hci.size(), st);
        v.upload(hv.data(), hv.size(), st);
        std::vector<double> hd(n, 1.0);
        std::vector<float> hv32(hv.begin(), hv.end());
        for (int i = 0; i < n; i++)
            for (int k = hrp[i]; k < hrp[i + 1]; k++)
                if (hci[k] == i && hv[k] != 0.0) hd[i] = 1.0 / hv[k];
        std::vector<float> hd32(hd.begin(), hd.end());
        dinv.upload(hd.data(), n, st);
        v32.upload(hv32.data(), hv32.size(), st);
        dinv32.upload(hd32.data(), n, st);
        nb = nblocks(n);
        for (auto *b : {&r, &z, &p, &q, &rh, &s, &sh, &t, &ph, &bb_tmp})
            if ((int)b->n < n) b->alloc(n);
        for (auto *b : {&r32, &z32, &p32, &q32, &x32, &b32})
            if ((int)b->n < n) b->alloc(n);
        for (auto *b : {&part1, &part2, &part3})
            if ((int)b->n < nb) b->alloc(nb);
        for (auto *b : {&fpart1, &fpart2, &fpart3})
            if ((int)b->n < nb) b->alloc(nb);
        if (!sc.p) sc.alloc(S_NSC);
        if (!fsc.p) fsc.alloc(S_NSC);
        nseg = segs.empty() ? 1 : (int)segs.size() - 1;
        seg_off = segs.empty() ? std::vector<int>{0, n} : segs;
        off_ks_ = ((nseg * KI_N * (int)sizeof(int) + 63) / 64) * 64;
        off_sc_ = off_ks_ + ((nseg * KS_N * (int)sizeof(double) + 63) / 64) * 64;
        off_rr_ = off_sc_ + 256;
        off_fd_ = off_rr_ + 2 * nb * (int)sizeof(double);
        off_bk_ = off_fd_ + 4 * nseg * (int)sizeof(double);
        const size_t pin = (size_t)off_bk_ + (size_t)nseg * sizeof(int);
        clear_graphs();
        {
            // off by default: on the 64-cavity sweep the graph took the FP64
            // step from 8.87 to 11.84 ms (a launch per node with its own
            // dispatch wait, plus the budget's launches past convergence)
            const char *eg = std::getenv("HFH_GRAPH");
            graph_on_ = eg && std::strcmp(eg, "1") == 0;
            // the budget's launches past convergence cost more than the wait
            // they save (sweep: 7.65 ms per mixed step with two waits per
            // solve, 7.93 ms with one), so one wait is used with graphs only
            const char *ef = std::getenv("HFH_FIRST_PASS");
            first_pass_ = graph_on_ || (ef && std::strcmp(ef, "1") == 0);
            const char *er = std::getenv("HFH_RESID_DIAG");
            resid_diag_ = !(er && std::strcmp(er, "0") == 0);
        }
        if (hpin_ && pin > hpin_size_) {
            (void)hipHostFree(hpin_);
            hpin_ = nullptr;
        }
        if (!hpin_) {
            HFH_CHECK(hipHostMalloc((void **)&hpin_, pin, hipHostMallocDefault));
            hpin_size_ = pin;
        }
        seg_stats.assign(nseg, SolveStats());
        {
            std::vector<int> hw(nseg + 1, (n + 255) / 256);
            for (int g = 0; g < nseg; g++) hw[g] = seg_off[g] / 256;
            segw_.upload(hw.data(), hw.size(), st);
            HFH_CHECK(hipStreamSynchronize(st));  // hw is a local
        }
        if (nseg > 1) {
            std::vector<int> hb(nb, nseg - 1);
            for (int g = 0; g < nseg; g++)
                for (int w = seg_off[g] / BLOCK; w < std::min(nb, (seg_off[g + 1] + BLOCK - 1) / BLOCK); w++) hb[w] = g;
            bseg_.upload(hb.data(), hb.size(), st);
            HFH_CHECK(hipStreamSynchronize(st));  // hb is a local
            segsc_.alloc(2 * nseg);
            hsegsc_.assign(2 * nseg, 0.0);
        }
        if ((int)xbak.n < n) xbak.alloc(n);
        if (const char *er = std::getenv("HFH_RESTARTS")) max_restarts = std::max(0, std::atoi(er));
        {
            const char *ea = std::getenv("HFH_AMG");
            k64.want_amg = k32.want_amg = amg && !(ea && std::strcmp(ea, "0") == 0);
            k64.amg_max_cx = k32.amg_max_cx = amg_max_cx;
        }
        // matrices with a Kronecker form are solved directly; their hierarchy
        // is built when a solve or a probe first needs it
        {
            const char *ep = std::getenv("HFH_DIRECT_PASSES");
            direct_passes_ = ep ? std::max(1, std::atoi(ep)) : 4;
            std::vector<int> so = seg_off;
            const bool on = allow_direct && direct_allowed();
            fdm.ready = on && affordable(fdm, [&] { return fdm.build(hrp, hci, hv, so, st, fdm_min_coupling); });
            // a uniform mesh whose system is left to Jacobi-PCG gets no factors
            nd.ready = on && !fdm.kronecker && nd_max_flops > 0 &&
                       affordable(nd, [&] { return nd.build(hrp, hci, hv, st, nd_max_flops, ND_ENTRIES); });
            if (const char *ev = std::getenv("HFH_VERBOSE"))
                if (std::strcmp(ev, "1") == 0 && (nd_max_flops > 0 || fdm.ready))
                    std::fprintf(stderr, "hfh: system of %d rows: %s (factors %.2g operations, %.2g entries)\n", n,
                                 fdm.ready ? "fast diagonalisation" : nd.ready ? "nested dissection" : "Krylov",
                                 nd.flops, nd.entries);
        }
        if (direct() && (int)segback_.n < nseg) segback_.alloc(nseg);
        if (direct() && nseg > 1 && (int)xkeep_.n < n) xkeep_.alloc(n);
        k64.defer_amg = k32.defer_amg = direct() && k64.want_amg;
        hrp_.clear();
        hci_.clear();
        hv_.clear();
        if (k64.defer_amg) {
            hrp_ = hrp;
            hci_ = hci;
            hv_ = hv;
        }
        t_mixed_ = t_fp64_ = -1;
        n32_ = n64_ = 0;
        explored_ = false;
        pend_ = Pending();
        since_probe_ = 0;
        probe_every_ = 10;
        {
            const char *em = std::getenv("HFH_MIXED_FP32");
            force32_ = em && std::strcmp(em, "1") == 0;
        }
        k64.set(n, rp.p, ci.p, hrp, hci, hv, st, segs);
        k32.set(n, rp.p, ci.p, hrp, hci, hv, st, segs);
        // the mixed form's FP64 candidate preconditions with the FP32
        // hierarchy (HFH_MIXED_AMG32=0: with its own FP64 one)
        k64.amg32 = &k32.amg;
        {
            const char *e = std::getenv("HFH_MIXED_AMG32");
            mixed_amg32_ = !(e && std::strcmp(e, "0") == 0);
        }
        // HFH_KRYLOV=classic selects the one-kernel-per-operation iterations
        const char *e = std::getenv("HFH_KRYLOV");
        fused = !(e && std::strcmp(e, "classic") == 0);
        HFH_CHECK(hipStreamSynchronize(st));
    }

    // ------------------------------------------------- fused iterations
    // Copies the flags and scalars of one fused solve (all segments) to
    // pinned host memory; per-segment values go to seg_hi_ / seg_hs_, hi/hs
    // get the aggregate: done and converged when every segment is, the
    // largest iteration count, the scalars of the segment with the largest
    // relative residual.
    template <typename T>
    void read_status(const FusedKrylov<T> &k, int *hi, double *hs, hipStream_t st) {
        copy_status<T>(k, st);
        HFH_CHECK(hipStreamSynchronize(st));
        parse_status<T>(hi, hs);
    }
    // flags and scalars to pinned memory (no wait; capturable)
    template <typename T>
    void copy_status(const FusedKrylov<T> &k, hipStream_t st) {
        HFH_CHECK(hipMemcpyAsync(hpin_, k.ki.p, (size_t)nseg * KI_N * sizeof(int), hipMemcpyDeviceToHost, st));
        HFH_CHECK(hipMemcpyAsync(hpin_ + off_ks_, k.ks.p, (size_t)nseg * KS_N * sizeof(T), hipMemcpyDeviceToHost, st));
    }
    // reads what copy_status left in pinned memory (after a wait)
    template <typename T>
    void parse_status(int *hi, double *hs) {
        seg_hi_.resize((size_t)nseg * KI_N);
        seg_hs_.resize((size_t)nseg * KS_N);
        std::memcpy(seg_hi_.data(), hpin_, (size_t)nseg * KI_N * sizeof(int));
        const T *t = reinterpret_cast<const T *>(hpin_ + off_ks_);
        for (int q = 0; q < nseg * KS_N; q++) seg_hs_[q] = (double)t[q];
        hi[KI_DONE] = 1;
        hi[KI_CONV] = 1;
        hi[KI_ITERS] = 0;
        double worst = -1;
        for (int g = 0; g < nseg; g++) {
            int *gi = &seg_hi_[(size_t)g * KI_N];
            if (gi[KI_BRK] || gi[KI_BRK + 1]) gi[KI_DONE] = 1;  // breakdown: stopped, not converged
            hi[KI_DONE] &= gi[KI_DONE] ? 1 : 0;
            hi[KI_CONV] &= gi[KI_CONV] ? 1 : 0;
            hi[KI_ITERS] = std::max(hi[KI_ITERS], gi[KI_ITERS]);
            const double *gs = &seg_hs_[(size_t)g * KS_N];
            const double rel = gs[KS_BN] > 0 ? std::sqrt(gs[KS_RR]) / gs[KS_BN] : std::sqrt(gs[KS_RR]);
            if (rel > worst || g == 0) {
                worst = rel;
                for (int q = 0; q < KS_N; q++) hs[q] = gs[q];
            }
        }
    }

    // runs one fused solve to its stopping test: the predicted number of
    // iterations, then host checks every 8; returns the iterations used
    template <typename T>
    int run_fused(FusedKrylov<T> &k, bool cg, int maxit, T rtol, T atol, T *x, int *hi, double *hs, hipStream_t st) {
        int it = 0;
        int chunk = std::min(maxit + 1, std::max(k.pred + 1, 2));
        for (;;) {
            k.iterate(cg, it, chunk, maxit, rtol, atol, x, st);
            it += chunk;
            read_status<T>(k, hi, hs, st);
            if (hi[KI_DONE] || it > maxit) break;
            chunk = std::min(check_every, maxit + 1 - it);
        }
        const int used = hi[KI_DONE] ? hi[KI_ITERS] : it;
        k.pred = used;
        return used;
    }

    // a direct solver's set-up; one that runs out of host or device memory
    // is given back whole and leaves the system to the Krylov solver
    template <typename S, typename F>
    static bool affordable(S &solver, F &&build) {
        try {
            return build();
        } catch (const std::exception &) {
            solver.release();
            (void)hipGetLastError();
            return false;
        }
    }
    // A run that names a form of the Krylov or V-cycle kernels by one of
    // their switches gets these kernels; HFH_DIRECT=0 turns the direct solves off
    static bool direct_allowed() {
        if (const char *e = std::getenv("HFH_DIRECT"))
            if (std::strcmp(e, "0") == 0) return false;
        if (const char *e = std::getenv("HFH_MIXED_FP32"))
            if (std::strcmp(e, "1") == 0) return false;
        for (const char *k : {"HFH_KRYLOV", "HFH_KRYLOV_LANES", "HFH_KRYLOV_ROWS", "HFH_KRYLOV_TIMED_LANES", "HFH_AMG",
                              "HFH_AMG_PCG", "HFH_AMG_FUSE", "HFH_AMG_OMEGA", "HFH_AMG_THETA", "HFH_AMG_LANES",
                              "HFH_AMG_DIAG", "HFH_VEL_AMG", "HFH_MIXED_AMG32", "HFH_TEMPLATES", "HFH_DIAG",
                              "HFH_GRAPH", "HFH_FIRST_PASS", "HFH_RESTARTS"})
            if (std::getenv(k)) return false;
        return true;
    }
    // builds the hierarchies that set_matrix deferred
    void ensure_amg(hipStream_t st) {
        if (hrp_.empty()) return;
        k64.build_amg(hrp_, hci_, hv_, st);
        k32.build_amg(hrp_, hci_, hv_, st);
        hrp_.clear();
        hci_.clear();
        hv_.clear();
    }

    // Direct solve (hfh_fdm.hpp, hfh_nd.hpp): x += M (b - A x) until the true
    // residual passes the stopping test, or no longer halves and is not above
    // its own rounding, where no solver has anything to add.  Every segment is
    // judged by itself: one that has ended keeps its x while the others go
    // on.  False when a segment is left to the Krylov solver (SEG_KRYLOV in
    // seg_state_), from its best x, after at most `limit` passes.  A first
    // residual that is not finite ends its segment with x as it was, as it
    // ends a Krylov solve: the corrections leave entries that are not finite
    // out, so no copy of x is needed before the first pass.
    enum { SEG_OPEN = 0, SEG_FINAL, SEG_KRYLOV };
    bool direct_solve(const double *b, double *x, double rtol, double atol, int limit, int fallback, hipStream_t st,
                      SolveStats &S) {
        double *norms = reinterpret_cast<double *>(hpin_ + off_fd_), *rounding = norms + 2 * nseg;
        int *back = reinterpret_cast<int *>(hpin_ + off_bk_);
        const double *h = norms;
        std::vector<SolveStats> &gs = seg_stats;
        S = SolveStats();
        S.fallback = fallback;
        gs.assign(nseg, S);
        seg_state_.assign(nseg, SEG_OPEN);
        bool open = true, undone = false;
        const bool small = fdm.ready && fdm.small;
        if (!small) true_residual(x, b, st);
        int pass = 0;
        while (open && pass < limit) {
            pass++;
            if (pass > 1)
                HFH_CHECK(hipMemcpyAsync(xbak.p, x, n * sizeof(double), hipMemcpyDeviceToDevice, st));
            if (small) {
                fdm.pass_small(k64.Av, dinv.p, b, x, norms, st);
            } else {
                if (fdm.ready)
                    fdm.correct(r.p, x, part3.p, dinv.p, st);
                else
                    nd.correct(r.p, x, st);
                true_residual(x, b, st);
                k_seg_norms<<<nseg, 256, 0, st>>>(segw_.p, part1.p, part2.p, norms);
            }
            if (pass == 1 && early) early();
            HFH_CHECK(hipStreamSynchronize(st));
            open = false;
            bool undo = false;
            std::vector<int> stalled;
            for (int g = 0; g < nseg; g++) {
                const double rn = std::sqrt(h[2 * g]), bn = std::sqrt(h[2 * g + 1]), tol = std::max(rtol * bn, atol);
                const double resid = bn > 0 ? rn / bn : rn, old = gs[g].resid;
                const bool better = pass == 1 || (seg_state_[g] == SEG_OPEN && resid < old);
                back[g] = !better;
                undo = undo || !better;
                if (better) {
                    gs[g].iters = std::isfinite(rn) ? pass : 0;
                    gs[g].resid = resid;
                    gs[g].converged = std::isfinite(rn) && rn <= tol;
                }
                if (seg_state_[g] != SEG_OPEN) continue;
                if (gs[g].converged || gs[g].iters == 0) {
                    seg_state_[g] = SEG_FINAL;
                } else if (pass > 1 && !(resid < 0.5 * old)) {
                    stalled.push_back(g);
                } else {
                    open = true;
                }
            }
            if (undo) {
                put_back(xbak.p, x, st);
                undone = true;
            }
            if (!stalled.empty()) {
                k_resid_rounding<<<nb, 4 * BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, x, b, part1.p);
                k_seg_norms<<<nseg, 256, 0, st>>>(segw_.p, part1.p, part1.p, rounding);
                HFH_CHECK(hipStreamSynchronize(st));
                for (int g : stalled) {
                    const double bn = std::sqrt(h[2 * g + 1]), kept = gs[g].resid * (bn > 0 ? bn : 1.0);
                    seg_state_[g] = kept <= std::sqrt(rounding[2 * g]) ? SEG_FINAL : SEG_KRYLOV;
                }
            }
        }
        for (int g = 0; g < nseg; g++)
            if (seg_state_[g] == SEG_OPEN) seg_state_[g] = SEG_KRYLOV;
        early_done = early && pass == 1 && !undone;
        S.iters = pass;
        return sum_segments(S);
    }
    // x = from in the segments flagged at off_bk_ of the pinned status (not
    // written again before the next wait on the stream).  The flags go to the
    // device first: read from there by each workgroup, host memory costs more
    // than the copies.
    void put_back(const double *from, double *x, hipStream_t st) {
        HFH_CHECK(hipMemcpyAsync(segback_.p, hpin_ + off_bk_, nseg * sizeof(int), hipMemcpyHostToDevice, st));
        k_seg_copy<<<nb, BLOCK, 0, st>>>(n, rp.p, nseg > 1 ? bseg_.p : nullptr, segback_.p, from, x);
    }
    // S's residual and convergence from the segments'; true when all are final
    bool sum_segments(SolveStats &S) {
        bool fin = true;
        S.resid = 0;
        S.converged = 1;
        for (int g = 0; g < nseg; g++) {
            const double q = seg_stats[g].resid;
            if (!(q <= S.resid) && !std::isnan(S.resid)) S.resid = q;
            S.converged = S.converged && seg_stats[g].converged;
            fin = fin && seg_state_[g] == SEG_FINAL;
        }
        return fin;
    }

    // The direct solve, then krylov(iterations left of maxit) for the segments
    // that it leaves: the others keep their x and statistics.  This solve
    // only: the next one starts with the direct solve again.  `fallback`:
    // SolveStats::fallback of what the direct solve ends.
    template <typename F>
    SolveStats direct_first(const double *b, double *x, double rtol, double atol, int maxit, int fallback,
                            hipStream_t st, F &&krylov) {
        SolveStats S;
        const bool done = direct_solve(b, x, rtol, atol, std::min(direct_passes_, maxit), fallback, st, S);
        if (done || S.iters >= maxit) return S;
        early_done = false;
        const std::vector<SolveStats> gs = seg_stats;
        const std::vector<int> state = seg_state_;
        bool keep = false;
        for (int q : state) keep = keep || q == SEG_FINAL;
        if (keep) {
            HFH_CHECK(hipMemcpyAsync(xkeep_.p, x, n * sizeof(double), hipMemcpyDeviceToDevice, st));
        }
        SolveStats K = krylov(maxit - S.iters);
        K.iters += S.iters;
        if (nseg == 1) return K;
        if (keep) {
            int *back = reinterpret_cast<int *>(hpin_ + off_bk_);
            for (int g = 0; g < nseg; g++) back[g] = state[g] == SEG_FINAL;
            put_back(xkeep_.p, x, st);
        }
        for (int g = 0; g < nseg; g++) {
            if (state[g] == SEG_FINAL)
                seg_stats[g] = gs[g];
            else
                seg_stats[g].iters += S.iters;
        }
        sum_segments(K);
        return K;
    }

    // r = b - A x and the per-256-row partials of r.r and b.b in part1 /
    // part2: the diagonal-form rows when the FP64 solver has them
    // (HFH_RESID_DIAG=0: the CSR launch)
    void true_residual(const double *x, const double *b, hipStream_t st) {
        if (k64.Av.dw && resid_diag_)
            k_residual_d<double><<<(n + KNT - 1) / KNT, KNT, 0, st>>>(n, k64.Av, x, b, r.p, part1.p, part2.p,
                                                                       part3.p, nb);
        else if (nnz > 24L * n)
            k_residual_l4<double, 16><<<nb, 4 * BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, x, b, r.p, part1.p, part2.p, part3.p);
        else
            k_residual_l4<double><<<nb, 4 * BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, x, b, r.p, part1.p, part2.p, part3.p);
    }

    // FP64 fused solve: Jacobi-PCG (spd) or BiCGStab, warm-started from x.
    // The stopping test runs on the recursively updated residual; once it
    // passes, the true residual b - A x is checked and the iteration
    // restarted from x (at most twice) while it misses the tolerance.
    // Systems with a direct solver try that first.
    SolveStats fused64(bool spd, const double *b, double *x, double rtol, double atol, int maxit, hipStream_t st) {
        early_done = false;
        auto krylov = [&](int left) { return krylov64(spd, b, x, rtol, atol, left, st); };
        return direct() && maxit > 0 ? direct_first(b, x, rtol, atol, maxit, 0, st, krylov) : krylov(maxit);
    }
    SolveStats krylov64(bool spd, const double *b, double *x, double rtol, double atol, int maxit, hipStream_t st) {
        ensure_amg(st);
        int hi[KI_N];
        double hs[KS_N];
        SolveStats S;
        double best = -1.0;  // largest true relative residual over segments of the kept x
        std::vector<double> rr(nb), bb(nb);
        for (int restart = 0; restart <= max_restarts; restart++) {
            if (restart > 0)  // keep the current x in case the restart does worse
                HFH_CHECK(hipMemcpyAsync(xbak.p, x, n * sizeof(double), hipMemcpyDeviceToDevice, st));
            if (restart == 0 && first_pass_) {
                S.iters += run_first_pass(spd, b, x, rtol, atol, maxit, hi, hs, rr, bb, st);
            } else {
                k64.init<double>(spd, b, x, st);
                S.iters += run_fused<double>(k64, spd, maxit - S.iters, rtol, atol, x, hi, hs, st);
                // true residual per segment (segments start on 256-row blocks)
                true_residual(x, b, st);
                HFH_CHECK(hipMemcpyAsync(rr.data(), part1.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
                HFH_CHECK(hipMemcpyAsync(bb.data(), part2.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
                HFH_CHECK(hipStreamSynchronize(st));
            }
            bool all_conv = true, worth = false;
            double worst = 0;
            std::vector<SolveStats> gs(nseg);
            for (int g = 0; g < nseg; g++) {
                double sr = 0, sb = 0;
                for (int w = seg_off[g] / BLOCK; w < std::min(nb, (seg_off[g + 1] + BLOCK - 1) / BLOCK); w++) {
                    sr += rr[w];
                    sb += bb[w];
                }
                const double bn = std::sqrt(sb), rn = std::sqrt(sr), tol = std::max(rtol * bn, atol);
                const int *gi = &seg_hi_[(size_t)g * KI_N];
                gs[g].iters = gi[KI_DONE] ? gi[KI_ITERS] : S.iters;
                gs[g].resid = bn > 0 ? rn / bn : rn;
                gs[g].converged = rn <= tol;
                all_conv = all_conv && gs[g].converged;
                worst = std::max(worst, gs[g].resid);
                // restart when the recursion claims convergence the true
                // residual misses by more than a factor 10
                if (!gs[g].converged && gi[KI_DONE] && gi[KI_CONV] && rn > 10.0 * tol) worth = true;
            }
            if (restart > 0 && !(worst < best)) {  // no better: restore
                HFH_CHECK(hipMemcpyAsync(x, xbak.p, n * sizeof(double), hipMemcpyDeviceToDevice, st));
                break;
            }
            best = worst;
            seg_stats = gs;
            S.resid = worst;
            S.converged = all_conv;
            if (all_conv || !worth || S.iters >= maxit) break;
            S.restarts++;
        }
        for (auto &g : seg_stats) g.restarts = S.restarts;
        return S;
    }

    // The first pass of an FP64 fused solve: the initialisation, a budget of
    // iterations (the last solve's count plus a quarter; launches after the
    // stopping test return at once), the true-residual partials and the
    // copies of the flags and partials to pinned memory, then one host wait
    // for both (the host-checked loop waits once for the flags, then once
    // more for the residual).  A solve that needs more iterations continues
    // with host-checked chunks from where the pass stopped, so the iterates
    // are those of the host-checked loop.  HFH_GRAPH=1 captures the pass as
    // a hipGraph (budget rounded up to 8; one graph per matrix form,
    // vectors, budget and tolerances, kept until the matrix is set again);
    // it measured slower than the launches from the host, so it is off by
    // default; so is the single wait without a graph (HFH_FIRST_PASS=1).
    int run_first_pass(bool spd, const double *b, double *x, double rtol, double atol, int maxit, int *hi,
                       double *hs, std::vector<double> &rr, std::vector<double> &bb, hipStream_t st) {
        const int want = k64.pred + 2 + k64.pred / 4;
        double *prr = reinterpret_cast<double *>(hpin_ + off_rr_);
        int budget;
        if (!graph_on_) {
            // the same launches from the host: one wait for the flags and
            // the true residual instead of one for each
            budget = std::min(maxit + 1, std::max(2, want));
            k64.init<double>(spd, b, x, st);
            k64.iterate(spd, 0, budget, maxit, rtol, atol, x, st);
            true_residual(x, b, st);
            copy_status<double>(k64, st);
            HFH_CHECK(hipMemcpyAsync(prr, part1.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipMemcpyAsync(prr + nb, part2.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipStreamSynchronize(st));
        } else {
            budget = std::min(maxit + 1, std::max(8, (want + 7) / 8 * 8));
            launch_graph64(spd, b, x, rtol, atol, maxit, budget, prr, st);
        }
        return finish_first_pass(spd, b, x, rtol, atol, maxit, budget, hi, hs, rr, bb, st);
    }
    void launch_graph64(bool spd, const double *b, double *x, double rtol, double atol, int maxit, int budget,
                        double *prr, hipStream_t st) {
        hipGraphExec_t exec = nullptr;
        for (auto &g : graphs_)
            if (g.spd == spd && g.a32 == k64.use_amg32 && g.b == b && g.x == x && g.budget == budget &&
                g.rtol == rtol && g.atol == atol && g.maxit == maxit)
                exec = g.exec;
        if (!exec) {
            if (graphs_.size() >= 16) clear_graphs();
            hipGraph_t graph = nullptr;
            HFH_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
            k64.init<double>(spd, b, x, st);
            k64.iterate(spd, 0, budget, maxit, rtol, atol, x, st);
            true_residual(x, b, st);
            copy_status<double>(k64, st);
            HFH_CHECK(hipMemcpyAsync(prr, part1.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipMemcpyAsync(prr + nb, part2.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipStreamEndCapture(st, &graph));
            HFH_CHECK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
            (void)hipGraphDestroy(graph);
            graphs_.push_back(GraphEntry{spd, k64.use_amg32, b, x, budget, rtol, atol, maxit, exec});
        }
        HFH_CHECK(hipGraphLaunch(exec, st));
        HFH_CHECK(hipStreamSynchronize(st));
    }
    int finish_first_pass(bool spd, const double *b, double *x, double rtol, double atol, int maxit, int budget,
                          int *hi, double *hs, std::vector<double> &rr, std::vector<double> &bb, hipStream_t st) {
        double *prr = reinterpret_cast<double *>(hpin_ + off_rr_);
        parse_status<double>(hi, hs);
        int it = budget;
        if (!hi[KI_DONE] && it <= maxit) {
            // more iterations than the budget: host-checked chunks
            for (;;) {
                const int chunk = std::min(check_every, maxit + 1 - it);
                k64.iterate(spd, it, chunk, maxit, rtol, atol, x, st);
                it += chunk;
                read_status<double>(k64, hi, hs, st);
                if (hi[KI_DONE] || it > maxit) break;
            }
            true_residual(x, b, st);
            HFH_CHECK(hipMemcpyAsync(prr, part1.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipMemcpyAsync(prr + nb, part2.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipStreamSynchronize(st));
        }
        std::memcpy(rr.data(), prr, nb * sizeof(double));
        std::memcpy(bb.data(), prr + nb, nb * sizeof(double));
        const int used = hi[KI_DONE] ? hi[KI_ITERS] : it;
        k64.pred = used;
        return used;
    }
    void clear_graphs() {
        for (auto &g : graphs_)
            if (g.exec) (void)hipGraphExecDestroy(g.exec);
        graphs_.clear();
    }

    // Mixed form: per system, FP32 refinement or the FP64 solve, whichever
    // took less time on its last solves (timed with events on the stream;
    // each solve ends with a host synchronisation).  The first six
    // solves alternate the forms (the first steps of a run are not typical:
    // the initial guesses improve as the solution history fills); after that
    // the form not in use is re-timed after 10 solves (50 when it was 30%
    // slower), the interval doubling (quadrupling when 30% slower) while the
    // choice holds, up to 1600, and returning to 10 when it flips.
    // A refinement whose FP32 solve fails finishes in FP64,
    // and FP32 is tried again 50 solves later.  Block-diagonal systems refine
    // all segments together, each against its own tolerance.
    SolveStats fused_mixed(bool spd, const double *b, double *x, double rtol, double atol, double inner_rtol,
                           int maxit, hipStream_t st) {
        early_done = false;
        auto krylov = [&](int left) { return krylov_mixed(spd, b, x, rtol, atol, inner_rtol, left, st); };
        // a direct solve is FP64 throughout (fallback 2)
        return direct() && maxit > 0 ? direct_first(b, x, rtol, atol, maxit, 2, st, krylov) : krylov(maxit);
    }
    SolveStats krylov_mixed(bool spd, const double *b, double *x, double rtol, double atol, double inner_rtol,
                            int maxit, hipStream_t st) {
        ensure_amg(st);
        account_pending();
        bool use32, probing = false;
        const bool pref32 = t_mixed_ >= 0 && t_fp64_ >= 0 && t_mixed_ < t_fp64_;
        if (force32_)
            use32 = true;
        else if ((n64_ < 3 || n32_ < 3) && t_mixed_ < 1e30)
            use32 = n32_ < n64_;  // first solves: the forms alternate, FP64 first
        else {
            use32 = pref32;
            if (++since_probe_ >= probe_every_) {
                use32 = !use32;
                since_probe_ = 0;
                probing = true;
            }
        }
        // each form is timed on the stream between two events: the solve's
        // launches and the idle gaps of its host checks, not the tail of
        // work queued before it.  The time is read at the next solve of this
        // system, when the end event has long completed, so no extra host
        // wait is added.
        if (!tev_[0]) {
            HFH_CHECK(hipEventCreate(&tev_[0]));
            HFH_CHECK(hipEventCreate(&tev_[1]));
        }
        HFH_CHECK(hipEventRecord(tev_[0], st));
        SolveStats S;
        if (use32) {
            S = mixed_refine(spd, b, x, rtol, atol, inner_rtol, maxit, st);
            if (!S.converged && S.fallback == 0) {
                // the refinement stalled (FP32 too coarse for this system):
                // finish in FP64 from the current x
                SolveStats F = krylov64(spd, b, x, rtol, atol, maxit, st);
                F.iters += S.iters;
                F.outer = S.outer;
                F.fallback = 1;
                S = F;
            }
        } else {
            // the FP32 V-cycle only under PCG.  Under BiCGStab its rounding
            // (a preconditioner that is not exactly linear) made the 3D
            // wall-layer pressure converge erratically (111 iterations
            // against 36 with the FP64 cycle) and stop on its updated
            // residual with a wrong x.
            k64.use_amg32 = mixed_amg32_ && spd;
            S = krylov64(spd, b, x, rtol, atol, maxit, st);
            k64.use_amg32 = false;
            S.fallback = 2;
            for (auto &g : seg_stats) g.fallback = 2;
        }
        HFH_CHECK(hipEventRecord(tev_[1], st));
        pend_ = Pending{true, use32, S.fallback == 0, probing, pref32};
        return S;
    }

    // books the time of the last mixed-form solve (see fused_mixed)
    void account_pending() {
        if (!pend_.on) return;
        pend_.on = false;
        HFH_CHECK(hipEventSynchronize(tev_[1]));
        float ms = 0;
        HFH_CHECK(hipEventElapsedTime(&ms, tev_[0], tev_[1]));
        const double dt = 1e-3 * ms;
        const bool use32 = pend_.use32, probing = pend_.probing, pref32 = pend_.pref32;
        // the second solve of a form replaces the time of its first (which
        // pays one-time costs: first launches, no iteration prediction yet);
        // a re-timing replaces the form's older time; the form in use keeps
        // a running mean
        if (use32 && pend_.ok)
            t_mixed_ = (n32_++ < 2 || t_mixed_ >= 1e30 || probing) ? dt : 0.5 * (t_mixed_ + dt);
        else if (use32)
            t_mixed_ = 1e30;  // FP32 failed on this system: keep FP64
        else
            t_fp64_ = (n64_++ < 2 || probing) ? dt : 0.5 * (t_fp64_ + dt);
        // a clearly slower form (30% or more) is re-timed less often
        const double ratio = std::max(t_mixed_, t_fp64_) / std::max(1e-30, std::min(t_mixed_, t_fp64_));
        if (probing)
            probe_every_ =
                (t_mixed_ < t_fp64_) == pref32 ? std::min((ratio > 1.3 ? 4 : 2) * probe_every_, 1600) : 10;
        if (!explored_ && n32_ >= 3 && n64_ >= 3) {
            explored_ = true;
            since_probe_ = 0;
            probe_every_ = ratio > 1.3 ? 50 : 10;
        }
        if (use32 && !pend_.ok && !force32_) {
            // FP32 failed: FP64 for the next 50 solves, then FP32 is tried again
            since_probe_ = 0;
            probe_every_ = 50;
        }
    }

    // FP64 defect correction around FP32 solves (see fused_mixed)
    SolveStats mixed_refine(bool spd, const double *b, double *x, double rtol, double atol, double inner_rtol,
                            int maxit, hipStream_t st) {
        SolveStats S;
        double h[S_NSC];
        int hi[KI_N];
        double hs[KS_N];
        int outer = 0, inner_total = 0;
        // stopping test on the FP64 residual: one norm for one system, one
        // per segment for block-diagonal systems (all must pass)
        double worst = 0, need = 1.0;  // need: residual reduction still required
        bool all_conv = false;
        std::vector<double> prr(nseg > 1 ? nb : 0), pbb(nseg > 1 ? nb : 0);
        std::vector<SolveStats> gs(nseg);
        for (;;) {
            true_residual(x, b, st);
            if (nseg == 1) {
                k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, part2.p, sc.p, S_RR, S_BB);
                HFH_CHECK(hipMemcpyAsync(hpin_ + off_sc_, sc.p, sizeof h, hipMemcpyDeviceToHost, st));
                HFH_CHECK(hipStreamSynchronize(st));
                std::memcpy(h, hpin_ + off_sc_, sizeof h);
                const double bn = std::sqrt(h[S_BB]), rn = std::sqrt(h[S_RR]);
                const double tol = std::max(rtol * bn, atol);
                all_conv = rn <= tol;
                worst = bn > 0 ? rn / bn : rn;
                need = rn > 0 ? tol / rn : 1.0;
            } else {
                // segments start on BLOCK-row boundaries
                HFH_CHECK(hipMemcpyAsync(prr.data(), part1.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
                HFH_CHECK(hipMemcpyAsync(pbb.data(), part2.p, nb * sizeof(double), hipMemcpyDeviceToHost, st));
                HFH_CHECK(hipStreamSynchronize(st));
                all_conv = true;
                worst = 0;
                for (int g = 0; g < nseg; g++) {
                    double sr = 0, sb = 0;
                    for (int w = seg_off[g] / BLOCK; w < std::min(nb, (seg_off[g + 1] + BLOCK - 1) / BLOCK); w++) {
                        sr += prr[w];
                        sb += pbb[w];
                    }
                    const double bn = std::sqrt(sb), rn = std::sqrt(sr), tol = std::max(rtol * bn, atol);
                    gs[g].resid = bn > 0 ? rn / bn : rn;
                    gs[g].converged = rn <= tol;
                    // the correction of segment g solves A d = s_g r_g with an
                    // absolute tolerance of 1: its residual ends below half
                    // of tol_g (or inner_rtol of ||r_g||); a converged segment
                    // gets s_g = 0 and no correction
                    const double target = std::max(0.5 * tol, 1e-300);
                    hsegsc_[g] = gs[g].converged ? 0.0 : 1.0 / target;
                    hsegsc_[nseg + g] = gs[g].converged ? 0.0 : target;
                    all_conv = all_conv && gs[g].converged;
                    worst = std::isfinite(gs[g].resid) ? std::max(worst, gs[g].resid) : gs[g].resid;
                    if (!std::isfinite(worst)) break;
                }
            }
            if (all_conv || outer >= 50 || inner_total >= maxit || !std::isfinite(worst)) break;
            if (nseg == 1) {
                k_convert<float, double><<<nb, BLOCK, 0, st>>>(n, r.p, b32.p);
            } else {
                HFH_CHECK(hipMemcpyAsync(segsc_.p, hsegsc_.data(), 2 * nseg * sizeof(double), hipMemcpyHostToDevice,
                                         st));
                k_convert_seg<<<nb, BLOCK, 0, st>>>(n, r.p, b32.p, bseg_.p, segsc_.p);
            }
            k32.init<float>(spd, b32.p, x32.p, st, true);  // x32 = 0, r = b32
            // an inner solve may take at most twice the FP64 solve's count
            const int cap = std::min(maxit - inner_total, std::max(200, 2 * k64.pred + 50));
            // one system: the inner solve reduces its residual by what is
            // still needed (with a factor 2 to spare), never further than
            // inner_rtol, so a last correction with one digit to gain is
            // short; block-diagonal systems get the same per segment from
            // the scaling above and an absolute tolerance of 1
            const double eff = std::min(0.5, std::max(inner_rtol, 0.5 * need));
            // first and later corrections differ in length: each keeps its
            // own iteration prediction
            const int slot = std::min(outer, 2);
            k32.pred = pred32_[slot];
            const int used = nseg == 1 ? run_fused<float>(k32, spd, cap, (float)eff, 0.0f, x32.p, hi, hs, st)
                                       : run_fused<float>(k32, spd, cap, (float)inner_rtol, 1.0f, x32.p, hi, hs, st);
            pred32_[slot] = k32.pred;
            inner_total += std::max(used, 1);
            if (!(hi[KI_DONE] && hi[KI_CONV])) {
                // FP32 Krylov cannot reach inner_rtol on this system (too
                // ill-conditioned for single precision): finish in FP64 from
                // the current x (the caller keeps FP64 for a while)
                SolveStats F = krylov64(spd, b, x, rtol, atol, maxit, st);
                F.iters += inner_total;
                F.outer = outer;
                F.fallback = 1;
                return F;
            }
            if (nseg == 1)
                k_add_conv<double, float><<<nb, BLOCK, 0, st>>>(n, x, x32.p);
            else
                k_add_conv_seg<<<nb, BLOCK, 0, st>>>(n, x, x32.p, bseg_.p, segsc_.p, nseg);
            outer++;
        }
        S.iters = inner_total;
        S.outer = outer;
        S.resid = worst;
        S.converged = all_conv;
        if (nseg > 1) {
            for (auto &g : gs) {
                g.iters = inner_total;
                g.outer = outer;
            }
            seg_stats = gs;
        }
        return S;
    }

    int lanes64() const { return k64.lanes; }
    int lanes32() const { return k32.lanes; }

    // Jacobi-PCG, FP64.  x holds the initial guess (warm start).
    SolveStats pcg(const double *b, double *x, double rtol, double atol, int maxit, hipStream_t st) {
        SolveStats S;
        k_cg_init<double, double><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, x, b, dinv.p, r.p, z.p, p.p, part1.p,
                                                         part2.p, part3.p);
        k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, part2.p, sc.p, S_RHO, S_RR);
        k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part3.p, nullptr, sc.p, S_BB, 0);
        double h[S_NSC];
        HFH_CHECK(hipMemcpyAsync(h, sc.p, sizeof h, hipMemcpyDeviceToHost, st));
        HFH_CHECK(hipStreamSynchronize(st));
        double bn = std::sqrt(h[S_BB]);
        double tol = std::max(rtol * bn, atol);
        double rn = std::sqrt(h[S_RR]);
        int it = 0;
        while (rn > tol && it < maxit) {
            int burst = std::min(check_every, maxit - it);
            for (int k = 0; k < burst; k++) {
                k_spmv_dot<double><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, p.p, q.p, part1.p);
                k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, nullptr, sc.p, S_PQ, 0);
                k_cg_alpha<double><<<1, 64, 0, st>>>(sc.p);
                k_cg_update<double><<<nb, BLOCK, 0, st>>>(n, x, r.p, p.p, q.p, dinv.p, z.p, sc.p, part1.p,
                                                          part2.p);
                k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, part2.p, sc.p, S_RHONEW, S_RR);
                k_cg_beta<double><<<1, 64, 0, st>>>(sc.p);
                k_cg_p<double><<<nb, BLOCK, 0, st>>>(n, p.p, z.p, sc.p);
            }
            it += burst;
            HFH_CHECK(hipMemcpyAsync(h, sc.p, sizeof h, hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipStreamSynchronize(st));
            rn = std::sqrt(h[S_RR]);
            if (!std::isfinite(rn)) break;
        }
        S.iters = it;
        S.resid = bn > 0 ? rn / bn : rn;
        S.converged = rn <= tol;
        return S;
    }

    // FP32 Jacobi-PCG on (A32) e = r, e starts at 0; relative tolerance only.
    int pcg32(double inner_rtol, int maxit, hipStream_t st) {
        k_fill<float><<<nb, BLOCK, 0, st>>>(n, x32.p, 0.0f);
        k_cg_init<float, float><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v32.p, x32.p, b32.p, dinv32.p, r32.p, z32.p,
                                                       p32.p, fpart1.p, fpart2.p, fpart3.p);
        k_reduce<float><<<1, BLOCK, 0, st>>>(nb, fpart1.p, fpart2.p, fsc.p, S_RHO, S_RR);
        float h[S_NSC];
        HFH_CHECK(hipMemcpyAsync(h, fsc.p, sizeof h, hipMemcpyDeviceToHost, st));
        HFH_CHECK(hipStreamSynchronize(st));
        double r0 = std::sqrt((double)h[S_RR]);
        double tol = inner_rtol * r0;
        double rn = r0;
        int it = 0;
        while (rn > tol && it < maxit) {
            int burst = std::min(check_every, maxit - it);
            for (int k = 0; k < burst; k++) {
                k_spmv_dot<float><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v32.p, p32.p, q32.p, fpart1.p);
                k_reduce<float><<<1, BLOCK, 0, st>>>(nb, fpart1.p, nullptr, fsc.p, S_PQ, 0);
                k_cg_alpha<float><<<1, 64, 0, st>>>(fsc.p);
                k_cg_update<float><<<nb, BLOCK, 0, st>>>(n, x32.p, r32.p, p32.p, q32.p, dinv32.p, z32.p, fsc.p,
                                                         fpart1.p, fpart2.p);
                k_reduce<float><<<1, BLOCK, 0, st>>>(nb, fpart1.p, fpart2.p, fsc.p, S_RHONEW, S_RR);
                k_cg_beta<float><<<1, 64, 0, st>>>(fsc.p);
                k_cg_p<float><<<nb, BLOCK, 0, st>>>(n, p32.p, z32.p, fsc.p);
            }
            it += burst;
            HFH_CHECK(hipMemcpyAsync(h, fsc.p, sizeof h, hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipStreamSynchronize(st));
            rn = std::sqrt((double)h[S_RR]);
            if (!std::isfinite(rn)) break;
        }
        return it;
    }

    // FP64 iterative refinement around the FP32 PCG.
    SolveStats mixed(const double *b, double *x, double rtol, double atol, double inner_rtol, int maxit,
                     hipStream_t st) {
        SolveStats S;
        double h[S_NSC];
        int outer = 0, inner_total = 0;
        double bn = 0, rn = 0, tol = 0;
        for (;;) {
            k_residual<double><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, x, b, r.p, part1.p, part2.p);
            k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, part2.p, sc.p, S_RR, S_BB);
            HFH_CHECK(hipMemcpyAsync(h, sc.p, sizeof h, hipMemcpyDeviceToHost, st));
            HFH_CHECK(hipStreamSynchronize(st));
            bn = std::sqrt(h[S_BB]);
            rn = std::sqrt(h[S_RR]);
            tol = std::max(rtol * bn, atol);
            if (rn <= tol || outer >= 50 || inner_total >= maxit || !std::isfinite(rn)) break;
            k_convert<float, double><<<nb, BLOCK, 0, st>>>(n, r.p, b32.p);
            inner_total += pcg32(inner_rtol, maxit - inner_total, st);
            k_add_conv<double, float><<<nb, BLOCK, 0, st>>>(n, x, x32.p);
            outer++;
        }
        S.iters = inner_total;
        S.outer = outer;
        S.resid = bn > 0 ? rn / bn : rn;
        S.converged = rn <= tol;
        return S;
    }

    // Right Jacobi-preconditioned BiCGStab, FP64 (van der Vorst 1992).
    SolveStats bicgstab(const double *b, double *x, double rtol, double atol, int maxit, hipStream_t st) {
        SolveStats S;
        double h[S_NSC];
        k_residual<double><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, x, b, r.p, part1.p, part2.p);
        k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, part2.p, sc.p, S_RR, S_BB);
        HFH_CHECK(hipMemcpyAsync(rh.p, r.p, n * sizeof(double), hipMemcpyDeviceToDevice, st));
        HFH_CHECK(hipMemcpyAsync(h, sc.p, sizeof h, hipMemcpyDeviceToHost, st));
        HFH_CHECK(hipStreamSynchronize(st));
        double bn = std::sqrt(h[S_BB]);
        double tol = std::max(rtol * bn, atol);
        double rn = std::sqrt(h[S_RR]);
        // rho(rh, r) = rr at start
        double init[S_NSC] = {0};
        init[S_RHONEW] = h[S_RR];
        init[S_RHO] = 1.0;
        init[S_ALPHA] = 1.0;
        init[S_OMEGA] = 1.0;
        HFH_CHECK(hipMemcpyAsync(sc.p, init, sizeof init, hipMemcpyHostToDevice, st));
        int it = 0;
        while (rn > tol && it < maxit) {
            k_bcg_p<double><<<nb, BLOCK, 0, st>>>(n, it == 0, p.p, r.p, q.p, dinv.p, ph.p, sc.p);
            k_spmv<double><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, ph.p, q.p);  // v = A ph (q holds v)
            k_dot2<double><<<nb, BLOCK, 0, st>>>(n, rh.p, q.p, nullptr, nullptr, part1.p, nullptr);
            k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, nullptr, sc.p, S_RV, 0);
            k_bcg_alpha<double><<<1, 64, 0, st>>>(sc.p);
            k_bcg_s<double><<<nb, BLOCK, 0, st>>>(n, r.p, q.p, dinv.p, s.p, sh.p, sc.p, part1.p);
            k_spmv<double><<<nb, BLOCK, 0, st>>>(n, rp.p, ci.p, v.p, sh.p, t.p);
            k_dot2<double><<<nb, BLOCK, 0, st>>>(n, t.p, s.p, t.p, t.p, part2.p, part3.p);
            k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part2.p, part3.p, sc.p, S_TS, S_TT);
            k_bcg_x<double><<<nb, BLOCK, 0, st>>>(n, x, r.p, ph.p, sh.p, s.p, t.p, rh.p, sc.p, part1.p, part2.p);
            k_bcg_shift<double><<<1, 64, 0, st>>>(sc.p);
            k_reduce<double><<<1, BLOCK, 0, st>>>(nb, part1.p, part2.p, sc.p, S_RR, S_RHONEW);
            it++;
            if (it % check_every == 0 || it == maxit) {
                HFH_CHECK(hipMemcpyAsync(h, sc.p, sizeof h, hipMemcpyDeviceToHost, st));
                HFH_CHECK(hipStreamSynchronize(st));
                rn = std::sqrt(h[S_RR]);
                if (!std::isfinite(rn) || h[S_RHONEW] == 0.0) break;
            }
        }
        HFH_CHECK(hipMemcpyAsync(h, sc.p, sizeof h, hipMemcpyDeviceToHost, st));
        HFH_CHECK(hipStreamSynchronize(st));
        rn = std::sqrt(h[S_RR]);
        S.iters = it;
        S.resid = bn > 0 ? rn / bn : rn;
        S.converged = rn <= tol;
        return S;
    }

  private:
    char *hpin_ = nullptr;  // pinned status: flags at 0, fused scalars at 64, outer scalars at 256
    int off_rr_ = 512;      // pinned true-residual partials (r.r then b.b, nb each)
    int off_fd_ = 0;        // pinned r.r and b.b, then their rounding, per segment (direct solves)
    int direct_passes_ = 4; // of a direct solve (HFH_DIRECT_PASSES)
    int off_bk_ = 0;        // pinned flag per segment: its x is put back
    DevBuf<int> segback_;         // the same on the device
    std::vector<int> seg_state_;  // of the last direct solve
    DevBuf<double> xkeep_;        // x of the segments that a direct solve has ended, during a Krylov solve of others
    std::vector<int> hrp_, hci_;  // the matrix, while its hierarchy is deferred
    std::vector<double> hv_;
    bool graph_on_ = false;  // first pass of FP64 fused solves as a captured graph (HFH_GRAPH=1)
    bool first_pass_ = false;  // one wait for flags and true residual (HFH_FIRST_PASS=1, or with graphs)
    bool resid_diag_ = true;  // true residuals through the diagonal-form rows (HFH_RESID_DIAG)
    struct GraphEntry {
        bool spd, a32;
        const double *b;
        double *x;
        int budget;
        double rtol, atol;
        int maxit;
        hipGraphExec_t exec;
    };
    std::vector<GraphEntry> graphs_;
};

}  // namespace hfh
