// Direct solves of the uniform-mesh systems by fast diagonalisation (Lynch,
// Rice, Thomas: Direct solution of partial difference equations by tensor
// product methods, Numer. Math. 6, 1964).
//
// On a uniform box the pressure and Helmholtz matrices are Kronecker sums
// A = Tx + Ty (+ Tz) of tridiagonal matrices with constant coefficients and
// one of three end rows per wall.  The eigenvectors of such a T are sines or
// cosines in closed form, so with orthogonal Vx, Vy, Vz
//   A^-1 r = V [ (V^T r) / (lx + ly + lz) ]
// which is 2 D dense products per right-hand side: matrix-core work in place
// of 11-16 latency-bound V-cycles.  The structure is read off the assembled
// matrix (fdm_detect); anything else keeps the Krylov solvers.
//
// One unknown p may be special: eliminated with its column (the pinned
// pressure), eliminated with its column kept (slv_impose_value), or carrying
// an added diagonal.  The tensor matrix T behind it is then singular with the
// constant null vector, and with g = T^+ e_p (kept) and mu = -sum(r)
//   z = T^+ r + mu g + c,   c from the value that z_p must have
// solves the other rows exactly.
//
// A solve is iterative refinement on the true residual b - A x of the
// stored matrix: x += M (b - A x) until the stopping test passes; the first
// correction leaves rounding, so it is normally the only one.
//
// Measured on MI355X, 20 steps between two field exchanges, Krylov with the
// V-cycle against this: cavity 64^2 12.8 -> 1.7 ms, cavity 256^2
// 29.4 -> 2.6 ms, Oldroyd-B cavity 512^2 63 -> 11.4 ms, 64-cavity sweep
// 190 -> 40.5 ms, 3D 15^3 (pressure only) 22.1 -> 8.1 ms; one 256^2 Poisson
// solve of the engine (Jacobi-BiCGStab, 1521 iterations) 27.5 -> 0.17 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <set>
#include <stdexcept>
#include <tuple>
#include <vector>

#include "hfh_krylov.hpp"

namespace hfh {

// ------------------------------------------------------------- detection
// T = a/D I + b S: off-diagonals of S are 1, its first and last diagonal
// entries s0, s1 in {0 (Dirichlet at a node), 1 (Neumann, half cell),
// -1 (Dirichlet, half cell)}
enum { FDM_PIN_NONE = 0, FDM_PIN_ELIM, FDM_PIN_ROW, FDM_PIN_SHIFT };
struct FdmSys {
    int off = 0, len = 0;  // the segment's rows
    int n[3] = {1, 1, 1};
    int s0[3] = {0, 0, 0}, s1[3] = {0, 0, 0};
    double a = 0, b[3] = {0, 0, 0};
    int pin = -1, pinmode = FDM_PIN_NONE;  // pin: row of the segment
    double shift = 0;
    int rows() const { return n[0] * n[1] * n[2]; }
};

// eigenvalues of S, ascending angle, and its orthonormal eigenvectors V
// (V[i * n + k]: entry i of vector k).  The entries are sin(pi m / 2q) with
// integer m, taken from one table of 4 q values.
inline void fdm_eigen(int n, int s0, int s1, std::vector<double> &cs, std::vector<double> &V) {
    // angle k: pi (p0 + dp k) / q for k = 0 .. n-1
    int p0, dp, q;
    if (s0 == 0 && s1 == 0) {
        p0 = 1, dp = 1, q = n + 1;
    } else if (s0 == 1 && s1 == 1) {
        p0 = 0, dp = 1, q = n;
    } else if (s0 == -1 && s1 == -1) {
        p0 = 1, dp = 1, q = n;
    } else if (s0 == -s1) {  // one Neumann, one half-cell Dirichlet end
        p0 = 1, dp = 2, q = 2 * n;
    } else if (s0 == 1 || s1 == 1) {  // one Neumann, one node Dirichlet end
        p0 = 1, dp = 2, q = 2 * n + 1;
    } else {  // one half-cell, one node Dirichlet end
        p0 = 2, dp = 2, q = 2 * n + 1;
    }
    const double pi = 3.14159265358979323846264338327950288;
    // sin(pi m / 2q), m in [0, 4q), from the first quarter
    std::vector<double> sn((size_t)4 * q);
    for (int m = 0; m < 4 * q; m++) {
        int h = m % (2 * q);
        if (h > q) h = 2 * q - h;
        const double v = 2 * h <= q ? std::sin(pi * h / (2.0 * q)) : std::cos(pi * (q - h) / (2.0 * q));
        sn[m] = m < 2 * q ? v : -v;
    }
    cs.resize(n);
    V.resize((size_t)n * n);
    std::vector<double> nn(n, 0.0);
    for (int k = 0; k < n; k++) cs[k] = 2.0 * sn[(size_t)((2L * (p0 + (long)dp * k) + q) % (4L * q))];  // 2 cos(pi p / q)
    for (int i = 0; i < n; i++) {
        // the vector starts from the left end's condition: sin(t (i + 1)),
        // cos(t (i + 1/2)) or sin(t (i + 1/2)), t = pi p / q
        const long f = s0 == 0 ? 2L * (i + 1) : 2L * i + 1, step = dp * f % (4L * q);
        long m = (p0 * f + (s0 == 1 ? q : 0)) % (4L * q);
        for (int k = 0; k < n; k++) {
            const double v = sn[(size_t)m];
            V[(size_t)i * n + k] = v;
            nn[k] += v * v;
            if ((m += step) >= 4L * q) m -= 4L * q;
        }
    }
    for (int k = 0; k < n; k++) nn[k] = 1.0 / std::sqrt(nn[k]);
    for (int i = 0; i < n; i++)
        for (int k = 0; k < n; k++) V[(size_t)i * n + k] *= nn[k];
}

// Reads the Kronecker form of rows [s.off, s.off + s.len) of a CSR matrix;
// rows past the box must be empty or purely diagonal padding.  Entries may
// differ from the constant coefficients by 1e-11 of the diagonal (the rows
// come from least-squares stencils); the refinement works on the stored
// matrix, so such differences only change its rate.
inline bool fdm_detect(const std::vector<int> &rp, const std::vector<int> &ci, const std::vector<double> &v,
                       FdmSys &s) {
    const int o = s.off;
    // strides: the distinct positive column offsets
    int st[3] = {0, 0, 0}, ns = 0, last = -1;
    for (int r = 0; r < s.len; r++)
        for (int k = rp[o + r]; k < rp[o + r + 1]; k++) {
            const int d = std::abs(ci[k] - o - r);
            if (d == 0) continue;
            if (ci[k] < o || ci[k] >= o + s.len) return false;
            last = std::max(last, std::max(r, ci[k] - o));
            int q = 0;
            while (q < ns && st[q] != d) q++;
            if (q == ns) {
                if (ns == 3) return false;
                st[ns++] = d;
            }
        }
    if (ns < 2) return false;
    std::sort(st, st + ns);
    if (st[0] != 1 || (ns == 3 && st[2] % st[1] != 0)) return false;
    s.n[0] = st[1];
    s.n[1] = ns == 3 ? st[2] / st[1] : (last + st[1]) / st[1];
    s.n[2] = ns == 3 ? (last + st[2]) / st[2] : 1;
    const int nd = ns, N = s.rows();
    if (N > s.len) return false;
    for (int d = 0; d < nd; d++)
        if (s.n[d] < 3) return false;
    // only empty rows after the box
    for (int r = N; r < s.len; r++)
        if (rp[o + r + 1] != rp[o + r]) return false;
    // at most one row without couplings: the eliminated unknown
    for (int r = 0; r < N; r++) {
        bool iso = true;
        for (int k = rp[o + r]; k < rp[o + r + 1]; k++) iso = iso && (ci[k] == o + r || v[k] == 0.0);
        if (!iso) continue;
        if (s.pin >= 0) return false;
        s.pin = r;
        s.pinmode = FDM_PIN_ELIM;
    }
    const int stride[3] = {1, s.n[0], s.n[0] * s.n[1]};
    // couplings: every neighbour once, equal along each dimension; those to
    // the eliminated unknown all absent (ELIM) or all present (ROW)
    double sum[3] = {0, 0, 0};
    long cnt[3] = {0, 0, 0};
    int topin = 0, nopin = 0;
    std::vector<double> dg(N, 0.0);
    for (int r = 0; r < N; r++) {
        unsigned seen = 0;
        for (int k = rp[o + r]; k < rp[o + r + 1]; k++) {
            const int c = ci[k] - o, off = c - r;
            if (off == 0) {
                dg[r] += v[k];
                continue;
            }
            if (r == s.pin) continue;
            int d = 0;
            while (d < nd && std::abs(off) != stride[d]) d++;
            if (d == nd) return false;
            const int id = (r / stride[d]) % s.n[d];
            if (off > 0 ? id == s.n[d] - 1 : id == 0) return false;
            const unsigned bit = 1u << (2 * d + (off > 0));
            if (seen & bit) return false;
            seen |= bit;
            if (c == s.pin) topin++;
            sum[d] += v[k];
            cnt[d]++;
        }
        if (r == s.pin) continue;
        for (int d = 0; d < nd; d++) {
            const int id = (r / stride[d]) % s.n[d];
            for (int up = 0; up < 2; up++) {
                if (up ? id == s.n[d] - 1 : id == 0) continue;
                if (seen & (1u << (2 * d + up))) continue;
                if (r + (up ? stride[d] : -stride[d]) != s.pin) return false;
                nopin++;
            }
        }
    }
    if (topin && nopin) return false;
    if (topin) s.pinmode = FDM_PIN_ROW;
    for (int d = 0; d < nd; d++) {
        if (!cnt[d]) return false;
        s.b[d] = sum[d] / (double)cnt[d];
    }
    // the interior diagonal, then the end rows of each dimension, from cells
    // beside the middle that are not the special unknown
    auto cell = [&](const int *id) { return id[0] + s.n[0] * (id[1] + s.n[1] * id[2]); };
    int mid[3] = {0, 0, 0};
    for (int d = 0; d < nd; d++) mid[d] = s.n[d] / 2;
    if (cell(mid) == s.pin) mid[0] = s.n[0] == 3 ? mid[0] : mid[0] > 1 ? mid[0] - 1 : mid[0] + 1;
    if (cell(mid) == s.pin) return false;
    s.a = dg[cell(mid)];
    if (!(s.a > 0)) return false;
    const double tol = 1e-11 * s.a;
    for (int r = 0; r < N; r++) {
        if (r == s.pin) continue;
        for (int k = rp[o + r]; k < rp[o + r + 1]; k++) {
            const int off = std::abs(ci[k] - o - r);
            for (int d = 0; d < nd; d++)
                if (off == stride[d] && !(std::fabs(v[k] - s.b[d]) <= tol)) return false;
        }
    }
    for (int d = 0; d < nd; d++)
        for (int hi = 0; hi < 2; hi++) {
            int id[3] = {mid[0], mid[1], mid[2]};
            id[d] = hi ? s.n[d] - 1 : 0;
            if (cell(id) == s.pin) id[(d + 1) % nd] += id[(d + 1) % nd] > 1 ? -1 : 1;
            if (cell(id) == s.pin || s.b[d] == 0.0) return false;
            const double t = (dg[cell(id)] - s.a) / s.b[d];
            const int w = (int)std::lround(std::max(-2.0, std::min(2.0, t)));
            if (w < -1 || w > 1) return false;
            (hi ? s.s1 : s.s0)[d] = w;
        }
    double asum = 0, rest = 0;
    long na = 0;
    for (int pass = 0; pass < 2; pass++) {
        for (int r = 0; r < N; r++) {
            if (r == s.pin && s.pinmode != FDM_PIN_SHIFT) continue;
            double e = s.a;
            for (int d = 0; d < nd; d++) {
                const int id = (r / stride[d]) % s.n[d];
                if (id == 0) e += s.b[d] * s.s0[d];
                if (id == s.n[d] - 1) e += s.b[d] * s.s1[d];
            }
            const double x = dg[r] - e;
            if (pass == 1) {
                if (r == s.pin) rest = x;
                continue;
            }
            if (std::fabs(x) <= tol) {
                asum += x;
                na++;
            } else {
                if (s.pin >= 0 || !(x > 0)) return false;
                s.pin = r;
                s.pinmode = FDM_PIN_SHIFT;
            }
        }
        if (pass == 0) s.a += asum / (double)std::max(1L, na);
    }
    s.shift = rest;
    // definite, or singular with the constant null vector and a special
    // unknown that makes the matrix regular
    double lo = s.a, hi = s.a;
    bool neumann = true;
    for (int d = 0; d < nd; d++) {
        const bool nn = s.s0[d] == 1 && s.s1[d] == 1;
        neumann = neumann && nn && s.b[d] < 0;
        // the largest eigenvalue of S, or a bound just above it
        const double c0 = nn ? 2.0 : 2.0 * std::cos(3.141592653589793 / (2.0 * s.n[d] + 4.0));
        lo += s.b[d] < 0 ? s.b[d] * c0 : -2.0 * s.b[d];
        hi += std::fabs(s.b[d]) * 2.0;
    }
    const bool singular = std::fabs(lo) <= 1e-10 * hi;
    if (singular) return neumann && s.pin >= 0;
    return lo > 1e-10 * hi && s.pin < 0;
}

// The systems of a matrix, or why there is no plan.  Each distinct line of n
// cells costs 2 n^2 table entries (V and V^T), which a pass also reads, so
// thin boxes lose in the end.  A solve of 65,536 rows, directly and with the
// V-cycle: 0.18 and 1.8 ms as 1024 x 64, 0.31 and 1.8 ms as 4096 x 16, 0.88
// and 1.26 ms as 8192 x 8 (tables 1 GB, set-up 2.1 s against 0.1), 2.3 and
// 1.04 ms as 16384 x 4 (4.3 GB, 12 s): sides up to 8192 are taken.  Square
// boxes gain at any size measured (2048 x 2048 6.6 against 23 ms).  Tables of
// all lines: two of the longest (2 GB) plus 4 entries per row, what square
// boxes of all different sides need.
constexpr int FDM_SIDE = 8192;
constexpr long FDM_TABLES = 1L << 28;
struct FdmPlan {
    std::vector<FdmSys> sys;
    int nd = 0;
    bool kronecker = false;  // the matrix has the form (also when the plan was not wanted)
    bool wanted = false;     // sides, tables and couplings within the limits
    long entries = 0;        // of the tables
};
// segments as DeviceSystem::set_matrix takes them; not wanted when no
// coupling reaches min_coupling of the diagonal
inline FdmPlan fdm_plan(const std::vector<int> &rp, const std::vector<int> &ci, const std::vector<double> &v,
                        const std::vector<int> &seg, double min_coupling) {
    FdmPlan P;
    const int n = (int)rp.size() - 1, nsys = (int)seg.size() - 1;
    if (n <= 0 || nsys <= 0) return P;
    P.sys.resize(nsys);
    double coupling = 0;
    int side = 0;
    std::set<std::tuple<int, int, int>> lines;
    for (int q = 0; q < nsys; q++) {
        FdmSys &s = P.sys[q];
        s.off = seg[q];
        s.len = seg[q + 1] - seg[q];
        if (seg[q] % 256 != 0 || !fdm_detect(rp, ci, v, s)) return P;
        const int d = s.n[2] > 1 ? 3 : 2;
        if (q > 0 && d != P.nd) return P;
        P.nd = d;
        for (int e = 0; e < d; e++) {
            coupling = std::max(coupling, std::fabs(s.b[e]) / s.a);
            side = std::max(side, s.n[e]);
            if (lines.emplace(s.n[e], s.s0[e], s.s1[e]).second) P.entries += 2L * s.n[e] * s.n[e];
        }
    }
    P.kronecker = true;
    P.wanted = coupling >= min_coupling && side <= FDM_SIDE && P.entries <= FDM_TABLES + 4L * n;
    return P;
}

// ---------------------------------------------------------------- device
constexpr int FDM_NT = 256;  // threads per workgroup (4 waves)
constexpr int FDM_T = 32;    // output tile

struct FdmJob {
    int M, N, K;
    int lda, ldb, ldc;
    int voff, coff;   // first row of the vector operand and of the result
    int bstride;      // both, per batch entry (z planes)
    int lx, ly, lz;   // eigenvalue tables of the scaled stage
    int nx, sys;
    long moff;        // the eigenvector matrix
};
struct FdmPin {
    int off = 0, pin = -1, mode = 0;
    int w0 = 0, w1 = 0;  // the segment's 256-row blocks
    int rowp = 0, colp = 0, K = 0;  // row of the last stage's source and column of V that give (T^+ r)_p
    long voff = 0;       // V of the first dimension, row colp
    double shift = 0;
};
enum { FDM_PLAIN = 0, FDM_SCALE, FDM_ADD };

typedef double fdm_d4 __attribute__((ext_vector_type(4)));

// C = A B for one 32 x 32 tile per workgroup, FP64 matrix cores.  One
// operand is an eigenvector matrix, the other a slice of the vector:
// AVEC = true: A is the vector, M x K row-major (products along the first
// dimension), B the matrix, K x N; AVEC = false: A is the matrix, stored
// K x M, and B the vector, K x N.  The four waves split K (k-steps of 4,
// round robin) and each holds the whole tile as 2 x 2 matrix-core tiles, so
// a step of 4 loads feeds 4 MFMAs; the partial tiles meet in LDS.
// FDM_SCALE divides by the eigenvalue sums (zero for the null mode),
// FDM_ADD adds the correction to x, with the special unknown's part; a
// right-hand side that is not finite spreads over the whole system in the
// products, and x stays what it was.
template <bool AVEC>
__global__ void __launch_bounds__(FDM_NT) k_fdm(const int4 *__restrict__ tiles, const FdmJob *__restrict__ jobs,
                                                const double *__restrict__ mats, const double *__restrict__ lam,
                                                const double *__restrict__ src, double *__restrict__ dst, int mode,
                                                const FdmPin *__restrict__ pins, const double *__restrict__ psum,
                                                const double *__restrict__ g, const double *__restrict__ r,
                                                const double *__restrict__ dinv) {
    __shared__ double red[4][FDM_T][FDM_T + 1];
    __shared__ double sh[8];
    const int4 tl = tiles[blockIdx.x];
    const FdmJob &J = jobs[tl.x];
    const int M = J.M, N = J.N, K = J.K, lda = J.lda, ldb = J.ldb;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double *vec = src + J.voff + (size_t)tl.w * J.bstride;
    const double *mat = mats + J.moff;
    const double *A = AVEC ? vec : mat, *B = AVEC ? mat : vec;
    const int li = lane & 15, lk = lane >> 4;
    const int m0 = min(tl.y + li, M - 1), m1 = min(tl.y + 16 + li, M - 1);
    const int n0 = min(tl.z + li, N - 1), n1 = min(tl.z + 16 + li, N - 1);
    fdm_d4 c00 = {0, 0, 0, 0}, c01 = c00, c10 = c00, c11 = c00;
    const size_t as = AVEC ? 1 : lda;  // A's stride along k
    const double *a0p = AVEC ? A + (size_t)m0 * lda : A + m0, *a1p = AVEC ? A + (size_t)m1 * lda : A + m1;
    // four k-steps of loads go out together (512^2 cavity: 27 us per product
    // with one step at a time, 20 us so; 256^2: 14 and 11 us)
    constexpr int U = 4;
#pragma unroll 1
    for (int k0 = 4 * w; k0 < K; k0 += 16 * U) {
        double a0[U], a1[U], b0[U], b1[U];
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int k = k0 + 16 * q + lk, kc = min(k, K - 1);
            a0[q] = a0p[kc * as];
            a1[q] = a1p[kc * as];
            b0[q] = B[(size_t)kc * ldb + n0];
            b1[q] = B[(size_t)kc * ldb + n1];
            if (k >= K) a0[q] = a1[q] = b0[q] = b1[q] = 0.0;
        }
#pragma unroll
        for (int q = 0; q < U; q++) {
            if (k0 + 16 * q >= K) break;  // the same for the whole wave
            c00 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[q], b0[q], c00, 0, 0, 0);
            c01 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[q], b1[q], c01, 0, 0, 0);
            c10 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[q], b0[q], c10, 0, 0, 0);
            c11 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[q], b1[q], c11, 0, 0, 0);
        }
    }
    // lane l holds rows 4 q + l / 16, column l % 16 of each 16 x 16 tile
#pragma unroll
    for (int q = 0; q < 4; q++) {
        red[w][4 * q + lk][li] = c00[q];
        red[w][4 * q + lk][16 + li] = c01[q];
        red[w][16 + 4 * q + lk][li] = c10[q];
        red[w][16 + 4 * q + lk][16 + li] = c11[q];
    }
    double mu = 0, c = 0;
    int pin = -1, pmode = 0;
    double zp = 0;
    if (mode == FDM_ADD && pins[J.sys].pin >= 0) {
        const FdmPin P = pins[J.sys];
        pin = P.off + P.pin;
        pmode = P.mode;
        double s = 0, t = 0;
        for (int i = P.w0 + (int)threadIdx.x; i < P.w1; i += FDM_NT) s += psum[i];
        for (int k = threadIdx.x; k < P.K; k += FDM_NT)
            t += src[P.off + (size_t)P.rowp * P.K + k] * mats[P.voff + (size_t)P.colp * P.K + k];
        for (int o = 32; o > 0; o >>= 1) {
            s += __shfl_down(s, o, 64);
            t += __shfl_down(t, o, 64);
        }
        if (lane == 0) {
            sh[w] = s;
            sh[4 + w] = t;
        }
        __syncthreads();
        mu = -((sh[0] + sh[1]) + (sh[2] + sh[3]));
        t = (sh[4] + sh[5]) + (sh[6] + sh[7]);
        zp = pmode == FDM_PIN_SHIFT ? -mu / P.shift : pmode == FDM_PIN_ROW ? r[pin] * dinv[pin] : 0.0;
        c = zp - t - mu * g[pin];
        if (pmode == FDM_PIN_ELIM) zp = r[pin] * dinv[pin];
    } else {
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < FDM_T * FDM_T / FDM_NT; q++) {
        const int e = q * FDM_NT + (int)threadIdx.x, i = e / FDM_T, j = e % FDM_T;
        const int m = tl.y + i, n = tl.z + j;
        if (m >= M || n >= N) continue;
        double v = (red[0][i][j] + red[1][i][j]) + (red[2][i][j] + red[3][i][j]);
        const size_t o = (size_t)J.coff + (size_t)tl.w * J.bstride + (size_t)m * J.ldc + n;
        if (mode == FDM_SCALE) {
            const int kx = n % J.nx, ky = n / J.nx;
            // 2D: rows are ky; 3D: rows are kz, columns (ky, kx)
            const double l = J.lz >= 0 ? (lam[J.lx + kx] + lam[J.ly + ky]) + lam[J.lz + m] : lam[J.lx + kx] + lam[J.ly + m];
            const bool null = pins[J.sys].pin >= 0 && m == 0 && n == 0;
            dst[o] = null ? 0.0 : v / l;
        } else if (mode == FDM_ADD) {
            if (pin >= 0) {
                const double t = mu * g[o] + c;
                v = (int)o == pin && isfinite(t) ? zp : v + t;
            }
            const double x0 = dst[o];
            dst[o] = isfinite(v) ? x0 + v : x0;
        } else {
            dst[o] = v;
        }
    }
}

// ------------------------------------------------------------ small systems
// The whole pass (residual, the 2 D products, x += z, new residual, norms) of
// a system of up to 2048 rows in one workgroup, in LDS: seven launches and the
// gaps between them are all that a system of this size costs otherwise.  One
// CU catches up with them near 48^2 and 14^3 rows; a time step of an explicit
// cavity takes, with launches and in one workgroup, 80 and 66 us at 32^2,
// 81 and 77 at 44^2, 81 and 95 at 64^2; in 3D 95 and 75 us at 8^3, 99 and 88
// at 12^3, 117 and 131 at 16^3.
struct FdmSmall {
    int off, n[3];
    int ld;        // row stride in LDS: odd, so 16 rows fall on 16 bank pairs
    int l[3];      // eigenvalue tables
    long v[3];     // V of each dimension; V^T follows it
};
constexpr int FDM_SMALL = 2048;
constexpr int FDM_SNT = 1024;

// one product along dimension DIM over the LDS array src, 16 x 16 tiles
// round robin over the waves; out(m, n, tile's z plane, LDS index, value)
template <int DIM, typename Out>
__device__ inline void fdm_small_stage(const FdmSmall &J, const double *__restrict__ mat, const double *src, Out &&out) {
    const int nx = J.n[0], ny = J.n[1], nz = J.n[2], ld = J.ld, lz = ld * ny;
    const int M = DIM == 0 ? ny * nz : DIM == 1 ? ny : nz, N = DIM == 2 ? nx * ny : nx, K = J.n[DIM];
    const int tm = (M + 15) / 16, tn = (N + 15) / 16, planes = DIM == 1 ? nz : 1;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    for (int t = threadIdx.x >> 6; t < tm * tn * planes; t += FDM_SNT / 64) {
        const int z = t / (tm * tn), m0 = (t / tn) % tm * 16, n0 = t % tn * 16;
        const int m = min(m0 + li, M - 1), n = min(n0 + li, N - 1);
        const int nat = DIM == 2 ? n / nx * ld + n % nx : n;
        fdm_d4 c = {0, 0, 0, 0};
        constexpr int U = 4;
        for (int k0 = 0; k0 < K; k0 += 4 * U) {
            double a[U], b[U];
#pragma unroll
            for (int q = 0; q < U; q++) {
                const int k = k0 + 4 * q + lk, kc = min(k, K - 1);
                a[q] = DIM == 0 ? src[m * ld + kc] : mat[kc * K + m];
                b[q] = DIM == 0 ? mat[kc * K + n] : DIM == 1 ? src[z * lz + kc * ld + n] : src[kc * lz + nat];
                if (k >= K) a[q] = b[q] = 0.0;
            }
#pragma unroll
            for (int q = 0; q < U; q++) {
                if (k0 + 4 * q >= K) break;  // the same for the whole wave
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[q], c, 0, 0, 0);
            }
        }
        if (n0 + li >= N) continue;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int row = m0 + 4 * q + lk;
            if (row < M) out(row, n0 + li, z, DIM == 0 ? row * ld + n : DIM == 1 ? z * lz + row * ld + n : row * lz + nat, c[q]);
        }
    }
    __syncthreads();
}

// sums of three values over the workgroup, on every thread
__device__ inline void fdm_small_sums(double (&v)[3], double (*sh)[FDM_SNT / 64]) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
        if ((threadIdx.x & 63) == 0) sh[k][threadIdx.x >> 6] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; k++) {
        v[k] = 0;
        for (int q = 0; q < FDM_SNT / 64; q++) v[k] += sh[k][q];
    }
    __syncthreads();
}

__global__ void __launch_bounds__(FDM_SNT) k_fdm_small(const FdmSmall *__restrict__ jobs, const FdmPin *__restrict__ pins,
                                                       int nd, KRows<double> A, const double *__restrict__ mats,
                                                       const double *__restrict__ lam, const double *__restrict__ g,
                                                       const double *__restrict__ dinv, const double *__restrict__ b,
                                                       double *__restrict__ x, double *norms) {
    extern __shared__ double fdm_lds[];
    __shared__ double sh[3][FDM_SNT / 64];
    __shared__ double s_rp;
    const FdmSmall J = jobs[blockIdx.x];
    const FdmPin P = pins[blockIdx.x];
    const int nx = J.n[0], ny = J.n[1], nz = J.n[2], N = nx * ny * nz, ld = J.ld, size = ld * ny * nz;
    double *u = fdm_lds, *w = fdm_lds + size;
    // b - A x of local row i of the stored matrix; at(j) is x of local row j
    auto residual = [&](int i, auto &&at) {
        const int gi = J.off + i, t = A.code ? A.code[gi] : -1;
        double s = 0;
        if (A.dw && t >= 0) {
            const int *db = A.dblk + (size_t)(gi / KNT) * (KD_MAX + 1);
            const unsigned msk = A.dmask[t];
            for (int e = 0; e < KD_MAX; e++)
                if ((msk >> e) & 1u) s += A.dw[(size_t)t * KD_MAX + e] * at(i + db[e]);
        } else {
            for (int k = A.rp[gi]; k < A.rp[gi + 1]; k++) s += A.val[k] * at(A.ci[k] - J.off);
        }
        return b[gi] - s;
    };
    double v[3] = {0, 0, 0};  // sum r
    for (int i = threadIdx.x; i < N; i += FDM_SNT) {
        const double r = residual(i, [&](int j) { return x[J.off + j]; });
        u[i / nx * ld + i % nx] = r;
        v[0] += r;
        if (i == P.pin) s_rp = r;
    }
    fdm_small_sums(v, sh);
    const double mu = -v[0], rp = P.pin >= 0 ? s_rp : 0.0;
    auto to = [](double *d) { return [d](int, int, int, int at, double c) { d[at] = c; }; };
    // V^T r along every dimension, over the eigenvalue sums, and back
    auto scaled = [&](double *d) {
        return [&, d](int m, int n, int z, int at, double c) {
            // 2D: (ky, kx) = (m, n); 3D: kz = m, n = (ky, kx)
            const double l = nd == 3 ? (lam[J.l[0] + n % nx] + lam[J.l[1] + n / nx]) + lam[J.l[2] + m]
                                     : lam[J.l[0] + n] + lam[J.l[1] + m];
            d[at] = P.pin >= 0 && m == 0 && n == 0 ? 0.0 : c / l;
        };
    };
    const double *V[3], *Z[3];
    for (int d = 0; d < 3; d++) {
        V[d] = mats + J.v[d];
        Z[d] = V[d] + (long)J.n[d] * J.n[d];
    }
    fdm_small_stage<0>(J, V[0], u, to(w));
    if (nd == 3) {
        fdm_small_stage<1>(J, V[1], w, to(u));
        fdm_small_stage<2>(J, V[2], u, scaled(w));
        fdm_small_stage<2>(J, Z[2], w, to(u));
        fdm_small_stage<1>(J, Z[1], u, to(w));
    } else {
        fdm_small_stage<1>(J, V[1], w, scaled(u));
        fdm_small_stage<1>(J, Z[1], u, to(w));
    }
    double c = 0, zp = 0;
    if (P.pin >= 0) {  // as k_fdm
        double t[3] = {0, 0, 0};
        for (int k = threadIdx.x; k < nx; k += FDM_SNT) t[0] += w[P.rowp * ld + k] * V[0][(size_t)P.colp * nx + k];
        fdm_small_sums(t, sh);
        const double own = rp * dinv[J.off + P.pin];
        zp = P.mode == FDM_PIN_SHIFT ? -mu / P.shift : P.mode == FDM_PIN_ROW ? own : 0.0;
        c = zp - t[0] - mu * g[J.off + P.pin];
        if (P.mode == FDM_PIN_ELIM) zp = own;
    }
    // the new x stays in LDS (u, without the padding) for its residual
    fdm_small_stage<0>(J, Z[0], w, [&](int m, int n, int, int, double z) {
        const int i = m * nx + n, gi = J.off + i;
        if (P.pin >= 0) {
            const double t = mu * g[gi] + c;
            z = i == P.pin && isfinite(t) ? zp : z + t;
        }
        const double x0 = x[gi], xn = isfinite(z) ? x0 + z : x0;
        x[gi] = xn;
        u[i] = xn;
    });
    double q[3] = {0, 0, 0};
    for (int i = threadIdx.x; i < N; i += FDM_SNT) {
        const double r = residual(i, [&](int j) { return u[j]; }), bi = b[J.off + i];
        q[0] += r * r;
        q[1] += bi * bi;
    }
    fdm_small_sums(q, sh);
    if (threadIdx.x == 0) {
        norms[2 * blockIdx.x] = q[0];
        norms[2 * blockIdx.x + 1] = q[1];
    }
}

// r.r and b.b of each segment from the 256-row partials, written to pinned
// host memory (one workgroup per segment)
__global__ void __launch_bounds__(256) k_seg_norms(const int *__restrict__ w0, const double *__restrict__ prr,
                                                   const double *__restrict__ pbb, double *out) {
    __shared__ double s1[4], s2[4];
    double a = 0, b = 0;
    for (int i = w0[blockIdx.x] + (int)threadIdx.x; i < w0[blockIdx.x + 1]; i += 256) {
        a += prr[i];
        b += pbb[i];
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_down(a, o, 64);
        b += __shfl_down(b, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        s1[threadIdx.x >> 6] = a;
        s2[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[2 * blockIdx.x] = (s1[0] + s1[1]) + (s1[2] + s1[3]);
        out[2 * blockIdx.x + 1] = (s2[0] + s2[1]) + (s2[2] + s2[3]);
    }
}

__global__ void k_fdm_unit(const FdmPin *__restrict__ pins, int n, double *x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && pins[i].pin >= 0) x[pins[i].off + pins[i].pin] = 1.0;
}

class FdmSolver {
  public:
    bool ready = false;
    bool kronecker = false;  // the matrix has the form (also when the plan was not wanted)
    int n = 0, nd = 0, nsys = 0;
    bool small = false;  // every system fits one workgroup (pass_small)

    // false: no plan (fdm_plan)
    bool build(const std::vector<int> &rp, const std::vector<int> &ci, const std::vector<double> &v,
               const std::vector<int> &seg, hipStream_t st, double min_coupling = 0) {
        ready = false;
        const FdmPlan plan = fdm_plan(rp, ci, v, seg, min_coupling);
        kronecker = plan.kronecker;
        if (!plan.wanted) return false;
        n = (int)rp.size() - 1;
        nsys = (int)plan.sys.size();
        nd = plan.nd;
        const std::vector<FdmSys> &sy = plan.sys;
        // the distinct one-dimensional matrices: V, then V^T
        std::map<std::tuple<int, int, int>, std::pair<long, std::vector<double>>> mat;
        std::vector<double> pool, lam;
        pool.reserve(plan.entries);
        auto matrix = [&](const FdmSys &s, int d) -> std::pair<long, std::vector<double>> & {
            const auto key = std::make_tuple(s.n[d], s.s0[d], s.s1[d]);
            auto it = mat.find(key);
            if (it == mat.end()) {
                const int m = s.n[d];
                std::vector<double> cs, V;
                fdm_eigen(m, s.s0[d], s.s1[d], cs, V);
                const long at = (long)pool.size();
                pool.insert(pool.end(), V.begin(), V.end());
                pool.resize(pool.size() + V.size());
                double *T = pool.data() + at + V.size();
                constexpr int B = 32;  // transposed by blocks
                for (int i0 = 0; i0 < m; i0 += B)
                    for (int k0 = 0; k0 < m; k0 += B)
                        for (int k = k0; k < std::min(m, k0 + B); k++)
                            for (int i = i0; i < std::min(m, i0 + B); i++) T[(size_t)k * m + i] = V[(size_t)i * m + k];
                it = mat.emplace(key, std::make_pair(at, cs)).first;
            }
            return it->second;
        };
        std::vector<FdmJob> jobs;
        std::vector<FdmPin> pins(nsys);
        std::vector<FdmSmall> sm(nsys);
        small = true;
        small_lds_ = 0;
        std::vector<std::vector<int4>> tl(2 * nd);
        bool pinned = false;
        for (int q = 0; q < nsys; q++) {
            const FdmSys &s = sy[q];
            long V[3] = {0, 0, 0}, Z[3] = {0, 0, 0};
            int L[3] = {-1, -1, -1};
            for (int d = 0; d < nd; d++) {
                auto &e = matrix(s, d);
                V[d] = e.first;
                Z[d] = V[d] + (long)s.n[d] * s.n[d];
                L[d] = (int)lam.size();
                for (double c : e.second) lam.push_back(s.a / nd + s.b[d] * c);
            }
            const int nx = s.n[0], ny = s.n[1], nz = s.n[2], nxy = nx * ny;
            FdmSmall &j = sm[q];
            j.off = s.off;
            j.ld = nx | 1;
            for (int d = 0; d < 3; d++) {
                j.n[d] = s.n[d];
                j.l[d] = L[d];
                j.v[d] = V[d];
            }
            small = small && nxy * nz <= FDM_SMALL;
            small_lds_ = std::max(small_lds_, 2 * (size_t)j.ld * ny * nz * sizeof(double));
            auto add = [&](int stage, int M, int N, int K, int lda, int ldb, int ldc, int batch, int bstride, long moff) {
                FdmJob j;
                j.M = M, j.N = N, j.K = K, j.lda = lda, j.ldb = ldb, j.ldc = ldc;
                j.voff = j.coff = s.off;
                j.bstride = bstride;
                j.lx = L[0], j.ly = L[1], j.lz = L[2];
                j.nx = nx, j.sys = q;
                j.moff = moff;
                for (int z = 0; z < batch; z++)
                    for (int m = 0; m < M; m += FDM_T)
                        for (int c = 0; c < N; c += FDM_T) tl[stage].push_back(make_int4((int)jobs.size(), m, c, z));
                jobs.push_back(j);
            };
            // products along the first dimension: rows of the vector times V
            // (forward) or V^T; along the others: V^T or V times the vector,
            // the matrix read K x M
            add(0, ny * nz, nx, nx, nx, nx, nx, 1, 0, V[0]);
            add(1, ny, nx, ny, ny, nx, nx, nz, nxy, V[1]);
            if (nd == 3) {
                add(2, nz, nxy, nz, nz, nxy, nxy, 1, 0, V[2]);
                add(3, nz, nxy, nz, nz, nxy, nxy, 1, 0, Z[2]);
            }
            add(2 * nd - 2, ny, nx, ny, ny, nx, nx, nz, nxy, Z[1]);
            add(2 * nd - 1, ny * nz, nx, nx, nx, nx, nx, 1, 0, Z[0]);
            FdmPin &p = pins[q];
            p.off = s.off;
            p.w0 = s.off / 256;
            p.w1 = (s.off + s.len + 255) / 256;
            if (s.pin >= 0) {
                p.pin = s.pin;
                p.mode = s.pinmode;
                p.rowp = s.pin / nx;
                p.colp = s.pin % nx;
                p.K = nx;
                p.voff = V[0];
                p.shift = s.shift;
                pinned = true;
            }
        }
        for (int q = 0; q < 2 * nd; q++) {
            ntiles_[q] = (int)tl[q].size();
            put(tiles_[q], tl[q], st);
        }
        if (small) {
            put(small_, sm, st);
            if (hipFuncSetAttribute(reinterpret_cast<const void *>(k_fdm_small), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)small_lds_) != hipSuccess)
                small = false;
        }
        put(jobs_, jobs, st);
        put(pins_, pins, st);
        put(mats_, pool, st);
        put(lam_, lam, st);
        t0_.alloc(n);
        t1_.alloc(n);
        g_.alloc(n);
        // rows past a segment's box are never written by the stages
        for (KBuf<double> *b : {&t0_, &t1_, &g_}) k_fill<double><<<nblocks(n), BLOCK, 0, st>>>(n, b->p, 0.0);
        if (hipStreamSynchronize(st) != hipSuccess) throw std::runtime_error("fdm upload failed");
        if (pinned) {  // g = T^+ e_p
            KBuf<double> e;
            e.alloc(n);
            k_fill<double><<<nblocks(n), BLOCK, 0, st>>>(n, e.p, 0.0);
            k_fdm_unit<<<nblocks(nsys), BLOCK, 0, st>>>(pins_.p, nsys, e.p);
            stages(e.p, g_.p, nullptr, nullptr, st, false);
            if (hipStreamSynchronize(st) != hipSuccess) throw std::runtime_error("fdm set-up failed");
        }
        ready = true;
        return true;
    }

    void release() {
        ready = false;
        small_.free();
        for (auto &t : tiles_) t.free();
        jobs_.free();
        pins_.free();
        for (KBuf<double> *b : {&mats_, &lam_, &t0_, &t1_, &g_}) b->free();
    }

    // x += M r; psum: sums of r over each 256-row block
    void correct(const double *r, double *x, const double *psum, const double *dinv, hipStream_t st) {
        stages(r, x, psum, dinv, st, true);
    }

    // x += M (b - A x) and the norms of the new residual and of b, with one
    // workgroup per system
    void pass_small(const KRows<double> &A, const double *dinv, const double *b, double *x, double *norms,
                    hipStream_t st) {
        k_fdm_small<<<nsys, FDM_SNT, small_lds_, st>>>(small_.p, pins_.p, nd, A, mats_.p, lam_.p, g_.p, dinv, b, x, norms);
    }

  private:
    KBuf<FdmSmall> small_;
    size_t small_lds_ = 0;
    KBuf<int4> tiles_[6];
    int ntiles_[6] = {0, 0, 0, 0, 0, 0};
    KBuf<FdmJob> jobs_;
    KBuf<FdmPin> pins_;
    KBuf<double> mats_, lam_, t0_, t1_, g_;

    template <typename T>
    static void put(KBuf<T> &d, const std::vector<T> &h, hipStream_t st) {
        d.alloc(h.size());
        if (!h.empty() && (hipMemcpyAsync(d.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, st) != hipSuccess ||
                           hipStreamSynchronize(st) != hipSuccess))
            throw std::runtime_error("fdm upload failed");
    }
    void stages(const double *r, double *x, const double *psum, const double *dinv, hipStream_t st, bool add) {
        const double *in = r;
        double *t[2] = {t0_.p, t1_.p};
        for (int q = 0; q < 2 * nd; q++) {
            const bool lastq = q == 2 * nd - 1;
            const int mode = q == nd - 1 ? FDM_SCALE : lastq && add ? FDM_ADD : FDM_PLAIN;
            double *out = lastq ? x : t[q & 1];
            if (q == 0 || lastq)
                k_fdm<true><<<ntiles_[q], FDM_NT, 0, st>>>(tiles_[q].p, jobs_.p, mats_.p, lam_.p, in, out, mode, pins_.p,
                                                           psum, g_.p, r, dinv);
            else
                k_fdm<false><<<ntiles_[q], FDM_NT, 0, st>>>(tiles_[q].p, jobs_.p, mats_.p, lam_.p, in, out, mode, pins_.p,
                                                            psum, g_.p, r, dinv);
            in = out;
        }
    }
};

}  // namespace hfh
