// Direct solves of the mesh-refined systems by nested dissection.
//
// The pressure and Helmholtz matrices of a refined 2D mesh do not change
// during a run and their graphs have small separators, so their exact
// factors are cheap to keep: the unknowns are split recursively by
// breadth-first level sets (George, Nested dissection of a regular finite
// element mesh, SIAM J. Numer. Anal. 10, 1973), the fronts are factored on
// the host (multifrontal method, Duff and Reid, ACM TOMS 9, 1983) and a
// solve is one launch per tree height up and one down, each a batch of dense
// matrix-vector products:
//   up    rhs_p = b_p + child updates;  update_q = child updates - W rhs_p
//   down  x_p = inv(F11) rhs_p - U x_q
// with W = F21 inv(F11), U = inv(F11) F12 of each front.
//
// Measured on MI355X (20 steps; 10 in 3D), against AMG-BiCGStab and FP32
// refinement: graded 4-level contraction, mixed form, 229 -> 18.5 ms;
// 12^3 wall-layer cavity 56 -> 7.0 ms, where a solve reads 0.57 GB of factors
// (host factors: 1.5e11 operations, 4 s on 8 cores; on 16, the set-up takes
// 5.3 s with them and 5.1 with the V-cycle hierarchy in their place).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <stdexcept>
#include <vector>

#include "hfh_krylov.hpp"
#include "hfh_domain.hpp"
#include "hfh_parallel.hpp"
#include "hfh_progress.hpp"

namespace hfh {

struct NdNode {
    std::vector<int> piv, border, child;
    int parent = -1, height = 0;
    std::vector<int> cmap;              // border -> position in the parent's front (pivots, then border)
    std::vector<double> W, G, S;        // q x p; p x (p + q) = [inv(F11) | -U]; q x q until the parent took it
};

// C(m x n) += f A(m x k) B(k x n), row-major with leading dimensions
inline void nd_gemm_plain(int m, int n, int k, double f, const double *A, int lda, const double *B, int ldb, double *C,
                          int ldc) {
    for (int i = 0; i < m; i++)
        for (int q = 0; q < k; q++) {
            const double x = f * A[(size_t)i * lda + q];
            const double *b = B + (size_t)q * ldb;
            double *c = C + (size_t)i * ldc;
            for (int j = 0; j < n; j++) c[j] += x * b[j];
        }
}
#if !defined(__HIP_DEVICE_COMPILE__) && defined(__x86_64__)
typedef double nd_v4 __attribute__((vector_size(32), aligned(8)));
// 4 x 8 register tiles over blocks of 128 x 256 of B (a 16-core host factors
// the wall-layer pressure's fronts at 10 GFLOP/s per core, 2 with the plain
// loops)
__attribute__((target("avx2,fma"))) inline void nd_gemm_avx2(int m, int n, int k, double f, const double *A, int lda,
                                                             const double *B, int ldb, double *C, int ldc) {
    constexpr int KB = 128, NB = 256;
    for (int k0 = 0; k0 < k; k0 += KB)
        for (int j0 = 0; j0 < n; j0 += NB) {
            const int k1 = std::min(k, k0 + KB), j1 = std::min(n, j0 + NB), je = j0 + (j1 - j0) / 8 * 8;
            const int ie = m / 4 * 4;
            for (int i = 0; i < ie; i += 4)
                for (int j = j0; j < je; j += 8) {
                    nd_v4 c[4][2] = {};
                    for (int q = k0; q < k1; q++) {
                        const double *b = B + (size_t)q * ldb + j;
                        const nd_v4 b0 = *(const nd_v4 *)b, b1 = *(const nd_v4 *)(b + 4);
                        for (int r = 0; r < 4; r++) {
                            const double x = f * A[(size_t)(i + r) * lda + q];
                            const nd_v4 v = {x, x, x, x};
                            c[r][0] += v * b0;
                            c[r][1] += v * b1;
                        }
                    }
                    for (int r = 0; r < 4; r++) {
                        double *o = C + (size_t)(i + r) * ldc + j;
                        *(nd_v4 *)o += c[r][0];
                        *(nd_v4 *)(o + 4) += c[r][1];
                    }
                }
            if (je < j1) nd_gemm_plain(ie, j1 - je, k1 - k0, f, A + k0, lda, B + (size_t)k0 * ldb + je, ldb, C + je, ldc);
            if (ie < m)
                nd_gemm_plain(m - ie, j1 - j0, k1 - k0, f, A + (size_t)ie * lda + k0, lda, B + (size_t)k0 * ldb + j0, ldb,
                              C + (size_t)ie * ldc + j0, ldc);
        }
}
#endif
// the product on `nt` threads (row blocks)
inline void nd_gemm(int nt, int m, int n, int k, double f, const double *A, int lda, const double *B, int ldb, double *C,
                    int ldc) {
    auto rows = [&](int i0, int i1) {
#if !defined(__HIP_DEVICE_COMPILE__) && defined(__x86_64__)
        static const bool avx = __builtin_cpu_supports("avx2") && __builtin_cpu_supports("fma");
        if (avx) return nd_gemm_avx2(i1 - i0, n, k, f, A + (size_t)i0 * lda, lda, B, ldb, C + (size_t)i0 * ldc, ldc);
#endif
        nd_gemm_plain(i1 - i0, n, k, f, A + (size_t)i0 * lda, lda, B, ldb, C + (size_t)i0 * ldc, ldc);
    };
    if (nt <= 1 || (double)m * n * k < 4e6) return rows(0, m);
    const int step = std::max(16, (m + 4 * nt - 1) / (4 * nt) / 4 * 4);
    std::atomic<int> next{0};
    run_parallel(nt, [&](int) {
        for (int i; (i = next.fetch_add(step)) < m;) rows(i, std::min(m, i + step));
    });
}

// inverse of the p x p matrix M (destroyed) into R; false when a pivot
// vanishes.  Blocks of up to 96 by Gauss-Jordan with partial pivoting,
// larger ones by halves through the Schur complement.
inline bool nd_inverse(int nt, int p, double *M, int ldm, double *R, int ldr) {
    if (p <= 96) {
        double amax = 0;
        for (int i = 0; i < p; i++)
            for (int j = 0; j < p; j++) {
                amax = std::max(amax, std::fabs(M[(size_t)i * ldm + j]));
                R[(size_t)i * ldr + j] = i == j ? 1.0 : 0.0;
            }
        for (int c = 0; c < p; c++) {
            int pr = c;
            for (int r = c + 1; r < p; r++)
                if (std::fabs(M[(size_t)r * ldm + c]) > std::fabs(M[(size_t)pr * ldm + c])) pr = r;
            if (!(std::fabs(M[(size_t)pr * ldm + c]) > 1e-14 * amax)) return false;
            double *mc = M + (size_t)c * ldm, *rc = R + (size_t)c * ldr;
            if (pr != c) {
                std::swap_ranges(mc, mc + p, M + (size_t)pr * ldm);
                std::swap_ranges(rc, rc + p, R + (size_t)pr * ldr);
            }
            const double d = 1.0 / mc[c];
            for (int j = c; j < p; j++) mc[j] *= d;
            for (int j = 0; j < p; j++) rc[j] *= d;
            for (int r = 0; r < p; r++) {
                if (r == c) continue;
                double *mr = M + (size_t)r * ldm, *rr = R + (size_t)r * ldr;
                const double f = mr[c];
                if (f == 0.0) continue;
                for (int j = c; j < p; j++) mr[j] -= f * mc[j];
                for (int j = 0; j < p; j++) rr[j] -= f * rc[j];
            }
        }
        return true;
    }
    const int h = (p / 2 + 3) / 4 * 4, g = p - h;
    double *B = M + h, *C = M + (size_t)h * ldm, *S = C + h;
    double *R12 = R + h, *R21 = R + (size_t)h * ldr, *R22 = R21 + h;
    if (!nd_inverse(nt, h, M, ldm, R, ldr)) return false;
    std::vector<double> X((size_t)h * g, 0.0), Y((size_t)g * h, 0.0);
    nd_gemm(nt, h, g, h, 1.0, R, ldr, B, ldm, X.data(), g);
    nd_gemm(nt, g, h, h, 1.0, C, ldm, R, ldr, Y.data(), h);
    nd_gemm(nt, g, g, h, -1.0, C, ldm, X.data(), g, S, ldm);
    if (!nd_inverse(nt, g, S, ldm, R22, ldr)) return false;
    for (int i = 0; i < h; i++) std::fill(R12 + (size_t)i * ldr, R12 + (size_t)i * ldr + g, 0.0);
    for (int i = 0; i < g; i++) std::fill(R21 + (size_t)i * ldr, R21 + (size_t)i * ldr + h, 0.0);
    nd_gemm(nt, h, g, g, -1.0, X.data(), g, R22, ldr, R12, ldr);
    nd_gemm(nt, g, h, g, -1.0, R22, ldr, Y.data(), h, R21, ldr);
    nd_gemm(nt, h, h, g, -1.0, R12, ldr, Y.data(), h, R, ldr);
    return true;
}

// The dissection tree of a matrix and its factors on the host.
class NdTree {
  public:
    std::vector<NdNode> nodes;  // children before parents
    double flops = 0, entries = 0;
    int height = 0;  // tree heights are 0 .. height - 1

    // the tree and the sizes of its fronts; rows without entries stay out
    void symbolic(const std::vector<int> &rp, const std::vector<int> &ci, int leaf) {
        const int n = (int)rp.size() - 1;
        nodes.clear();
        // graph of A + A^T without the diagonal
        xa_.assign(n + 1, 0);
        for (int i = 0; i < n; i++)
            for (int k = rp[i]; k < rp[i + 1]; k++)
                if (ci[k] != i) {
                    xa_[i + 1]++;
                    xa_[ci[k] + 1]++;
                }
        for (int i = 0; i < n; i++) xa_[i + 1] += xa_[i];
        adj_.resize(xa_[n]);
        std::vector<int> at(xa_.begin(), xa_.end() - 1);
        for (int i = 0; i < n; i++)
            for (int k = rp[i]; k < rp[i + 1]; k++)
                if (ci[k] != i) {
                    adj_[at[i]++] = ci[k];
                    adj_[at[ci[k]]++] = i;
                }
        in_.assign(n, 0);
        lvl_.assign(n, -1);
        sets_ = 0;
        leaf_ = leaf;
        std::vector<int> all;
        for (int i = 0; i < n; i++)
            if (rp[i + 1] > rp[i] || xa_[i + 1] > xa_[i]) all.push_back(i);
        dissect(all);
        // fronts
        std::vector<int> owner(n, -1), mark(n, -1), pos(n, -1);
        flops = entries = 0;
        height = 0;
        for (int q = 0; q < (int)nodes.size(); q++)
            for (int v : nodes[q].piv) owner[v] = q;
        for (int q = 0; q < (int)nodes.size(); q++) {
            NdNode &N = nodes[q];
            auto add = [&](int v) {
                if (owner[v] > q && mark[v] != q) {
                    mark[v] = q;
                    N.border.push_back(v);
                }
            };
            for (int v : N.piv)
                for (int k = xa_[v]; k < xa_[v + 1]; k++) add(adj_[k]);
            for (int c : N.child)
                for (int v : nodes[c].border) add(v);
            std::sort(N.border.begin(), N.border.end(),
                      [&](int a, int b) { return owner[a] != owner[b] ? owner[a] < owner[b] : a < b; });
            for (size_t k = 0; k < N.piv.size(); k++) pos[N.piv[k]] = (int)k;
            for (size_t k = 0; k < N.border.size(); k++) pos[N.border[k]] = (int)(N.piv.size() + k);
            for (int c : N.child) {
                NdNode &C = nodes[c];
                C.cmap.resize(C.border.size());
                for (size_t k = 0; k < C.border.size(); k++) C.cmap[k] = pos[C.border[k]];
                N.height = std::max(N.height, C.height + 1);
            }
            const double p = (double)N.piv.size(), b = (double)N.border.size();
            flops += 2 * p * p * p + 4 * p * p * b + 2 * p * b * b;
            entries += p * p + 2 * p * b;
            height = std::max(height, N.height + 1);
        }
    }

    // whether the factors are within the limits: operations, entries, and
    // the rows and columns of the largest front
    bool affordable(double max_flops, double max_entries, int max_front) const {
        if (flops > max_flops || entries > max_entries) return false;
        for (const NdNode &N : nodes)
            if ((int)(N.piv.size() + N.border.size()) > max_front) return false;
        return true;
    }

    // the factors; false when a front's pivot block is singular
    bool numeric(const std::vector<int> &rp, const std::vector<int> &ci, const std::vector<double> &v) {
        const int n = (int)rp.size() - 1;
        std::vector<int> tp(n + 1, 0), tr(ci.size());
        std::vector<double> tv(ci.size());
        for (int c : ci) tp[c + 1]++;
        for (int i = 0; i < n; i++) tp[i + 1] += tp[i];
        {
            std::vector<int> at(tp.begin(), tp.end() - 1);
            for (int i = 0; i < n; i++)
                for (int k = rp[i]; k < rp[i + 1]; k++) {
                    const int q = at[ci[k]]++;
                    tr[q] = i;
                    tv[q] = v[k];
                }
        }
        std::vector<std::vector<int>> by(height);
        for (int q = 0; q < (int)nodes.size(); q++) by[nodes[q].height].push_back(q);
        std::atomic<bool> ok{true};
        const int nt = setup_threads();
        std::vector<std::vector<int>> pos(nt);
        for (auto &list : by) {
            // the costly fronts first: those above 1e9 operations one by one
            // on all threads, the others one per thread
            std::sort(list.begin(), list.end(), [&](int a, int b) {
                const size_t x = nodes[a].piv.size() + nodes[a].border.size(),
                             y = nodes[b].piv.size() + nodes[b].border.size();
                return x != y ? x > y : a < b;
            });
            size_t big = 0;
            auto ops = [&](const NdNode &N) {
                const double p = (double)N.piv.size(), q = (double)N.border.size();
                return 2 * p * p * p + 4 * p * p * q + 2 * p * q * q;
            };
            if (pos[0].empty()) pos[0].assign(n, -1);
            while (big < list.size() && ops(nodes[list[big]]) > 1e9) {
                progress("direct factors, tree height", nodes[list[big]].height, height);
                if (!front(nodes[list[big++]], rp, ci, v, tp, tr, tv, pos[0], nt)) return false;
            }
            std::atomic<size_t> next{big};
            run_parallel(std::min<int>(nt, (int)list.size()), [&](int t) {
                struct Stop {  // the others end with the first that does not return
                    std::atomic<bool> &ok;
                    bool done = false;
                    ~Stop() {
                        if (!done) ok = false;
                    }
                } stop{ok};
                if (pos[t].empty()) pos[t].assign(n, -1);
                for (size_t i; ok && (i = next++) < list.size();)
                    if (!front(nodes[list[i]], rp, ci, v, tp, tr, tv, pos[t], 1)) ok = false;
                stop.done = true;
            });
            if (!ok) return false;
        }
        return true;
    }

  private:
    std::vector<int> xa_, adj_, in_, lvl_;
    int sets_ = 0, leaf_ = 64;

    int leaf_node(std::vector<int> &c) {
        nodes.emplace_back();
        nodes.back().piv = std::move(c);
        return (int)nodes.size() - 1;
    }
    // breadth-first levels of the vertices with in_ == id from s; the order
    // and the first index of each level
    void levels(int s, int id, std::vector<int> &order, std::vector<int> &first) {
        order.assign(1, s);
        first.assign(1, 0);
        lvl_[s] = 0;
        for (size_t lo = 0; lo < order.size();) {
            const size_t hi = order.size();
            for (size_t k = lo; k < hi; k++)
                for (int e = xa_[order[k]]; e < xa_[order[k] + 1]; e++) {
                    const int w = adj_[e];
                    if (in_[w] == id && lvl_[w] < 0) {
                        lvl_[w] = (int)first.size();
                        order.push_back(w);
                    }
                }
            lo = hi;
            if (order.size() > hi) first.push_back((int)hi);
        }
        first.push_back((int)order.size());
    }
    // nodes of the vertices `set`; returns the roots of their components
    std::vector<int> dissect(const std::vector<int> &set) {
        std::vector<int> roots, order, first;
        const int id = ++sets_;
        for (int v : set) in_[v] = id;
        for (int v : set) {
            if (in_[v] != id) continue;  // its component is done
            // a start far from the rest: the end of a breadth-first search, twice
            int s = v;
            for (int rep = 0; rep < 3; rep++) {
                levels(s, id, order, first);
                for (int w : order) lvl_[w] = -1;
                int best = order.back();
                for (int k = first[first.size() - 2]; k < (int)order.size(); k++)
                    if (xa_[order[k] + 1] - xa_[order[k]] < xa_[best + 1] - xa_[best]) best = order[k];
                if ((int)order.size() <= leaf_) break;
                if (rep < 2) s = best;
            }
            const int m = (int)order.size(), nl = (int)first.size() - 1;
            if (m <= leaf_ || nl < 3) {
                for (int w : order) in_[w] = 0;
                roots.push_back(leaf_node(order));
                continue;
            }
            // the level of the smallest size over f (1 - f), f the share of the
            // vertices before it: even halves keep the tree low
            int j = -1;
            double cost = 0;
            for (int k = 1; k + 1 < nl; k++) {
                const double f = (first[k] + 0.5 * (first[k + 1] - first[k])) / m;
                if (f < 0.25 || f > 0.75) continue;
                const double c = (first[k + 1] - first[k]) / (f * f * (1.0 - f) * (1.0 - f));
                if (j < 0 || c < cost) {
                    j = k;
                    cost = c;
                }
            }
            if (j < 0)
                for (j = 1; j + 2 < nl && first[j + 1] < m / 2;) j++;
            for (int k = 0; k < nl; k++)
                for (int e = first[k]; e < first[k + 1]; e++) lvl_[order[e]] = k;
            std::vector<int> sep, left(order.begin(), order.begin() + first[j]),
                right(order.begin() + first[j + 1], order.end());
            for (int e = first[j]; e < first[j + 1]; e++) {
                bool up = false;
                for (int k = xa_[order[e]]; k < xa_[order[e] + 1] && !up; k++)
                    up = in_[adj_[k]] == id && lvl_[adj_[k]] == j + 1;
                (up ? sep : left).push_back(order[e]);
            }
            for (int w : order) {
                lvl_[w] = -1;
                in_[w] = 0;
            }
            std::vector<int> kids = dissect(left), more = dissect(right);
            kids.insert(kids.end(), more.begin(), more.end());
            const int q = leaf_node(sep);
            for (int c : kids) nodes[c].parent = q;
            nodes[q].child = std::move(kids);
            roots.push_back(q);
        }
        return roots;
    }

    bool front(NdNode &N, const std::vector<int> &rp, const std::vector<int> &ci, const std::vector<double> &v,
               const std::vector<int> &tp, const std::vector<int> &tr, const std::vector<double> &tv,
               std::vector<int> &pos, int nt) {
        const int p = (int)N.piv.size(), q = (int)N.border.size(), m = p + q;
        for (int k = 0; k < p; k++) pos[N.piv[k]] = k;
        for (int k = 0; k < q; k++) pos[N.border[k]] = p + k;
        std::vector<double> F11((size_t)p * p, 0.0), F12((size_t)p * q, 0.0), F21((size_t)q * p, 0.0);
        N.S.assign((size_t)q * q, 0.0);
        auto at = [&](int r, int c) -> double & {
            if (r < p) return c < p ? F11[(size_t)r * p + c] : F12[(size_t)r * q + c - p];
            return c < p ? F21[(size_t)(r - p) * p + c] : N.S[(size_t)(r - p) * q + c - p];
        };
        for (int k = 0; k < p; k++) {
            const int g = N.piv[k];
            for (int e = rp[g]; e < rp[g + 1]; e++)
                if (pos[ci[e]] >= 0) at(k, pos[ci[e]]) += v[e];
            for (int e = tp[g]; e < tp[g + 1]; e++)
                if (pos[tr[e]] >= p) at(pos[tr[e]], k) += tv[e];
        }
        for (int c : N.child) {
            NdNode &C = nodes[c];
            const int qc = (int)C.border.size();
            for (int i = 0; i < qc; i++)
                for (int j = 0; j < qc; j++) at(C.cmap[i], C.cmap[j]) += C.S[(size_t)i * qc + j];
            std::vector<double>().swap(C.S);
        }
        for (int g : N.piv) pos[g] = -1;
        for (int g : N.border) pos[g] = -1;
        N.G.assign((size_t)p * m, 0.0);
        if (!nd_inverse(nt, p, F11.data(), p, N.G.data(), m)) return false;
        nd_gemm(nt, p, q, p, -1.0, N.G.data(), m, F12.data(), q, N.G.data() + p, m);
        N.W.assign((size_t)q * p, 0.0);
        nd_gemm(nt, q, p, p, 1.0, F21.data(), p, N.G.data(), m, N.W.data(), p);
        nd_gemm(nt, q, q, p, 1.0, F21.data(), p, N.G.data() + p, m, N.S.data(), q);
        return true;
    }
};

// ---------------------------------------------------------------- device
// One workgroup's share of a front: rows [row0, row1) of W (up) or of
// G = [inv(F11) | -U] (down), one row per lane group.  Everything that the
// workgroup needs to find its data is here, so it starts its matrix loads
// one memory round trip after the launch.
struct NdTask {
    int row0, row1;
    int p, q;     // pivots, border
    int po, bo;   // first pivot / border entry of the node's lists
    int fo;       // first front entry (gather lists of the up pass)
    int gl;       // lanes per row
    long at;      // W or G in the factor array
};
constexpr int ND_NT = 256;
constexpr int ND_LDS = 8192;  // front entries held in LDS (64 KiB)
constexpr int ND_PRE = 16;    // matrix entries per lane in flight before the gather
constexpr int ND_FRONT = ND_LDS - ND_NT / 8;  // the largest front
constexpr int ND_LEAF = 96;                   // unknowns of a leaf
constexpr double ND_ENTRIES = 2.5e8;          // of all factors (2 GB)
// lanes per row: enough that the whole row is in flight (up to 1024 entries)
inline int nd_lanes(int len) { return len <= 8 * ND_PRE ? 8 : len <= 16 * ND_PRE ? 16 : 64; }

// The rows' matrix loads are issued first, then gather() fills the vector in
// LDS (dependent index loads), then the dot products: the two chains of
// memory round trips overlap.  A height of a few fronts is bound by this
// latency (11-19 us with the loads behind the gather and the rows of a wave
// in turn, 5-8 us so), the leaves by the factor bytes (250 MB in 37 us).
template <int GL, typename Gather, typename Put>
__device__ inline void nd_rows(const NdTask &T, const double *__restrict__ fac, int len, const double *v, Gather &&gather,
                               Put &&put) {
    const int row = T.row0 + (int)threadIdx.x / GL, lane = threadIdx.x % GL;
    const bool in = row < T.row1;
    const double *m = fac + T.at + (size_t)(in ? row : T.row0) * len;
    double a[ND_PRE];
#pragma unroll
    for (int q = 0; q < ND_PRE; q++) a[q] = in && lane + q * GL < len ? m[lane + q * GL] : 0.0;
    gather();
    __syncthreads();
    double s[4] = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < ND_PRE; q++)
        if (lane + q * GL < len) s[q & 3] += a[q] * v[lane + q * GL];
    if (in)
        for (int k = lane + ND_PRE * GL; k < len; k += ND_PRE * GL) {
#pragma unroll
            for (int q = 0; q < ND_PRE; q++) a[q] = k + q * GL < len ? m[k + q * GL] : 0.0;
#pragma unroll
            for (int q = 0; q < ND_PRE; q++)
                if (k + q * GL < len) s[q & 3] += a[q] * v[k + q * GL];
        }
    double t = (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
    for (int o = GL / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if (in && lane == 0) put(row, t);
}
template <typename Gather, typename Put>
__device__ inline void nd_dispatch(const NdTask &T, const double *__restrict__ fac, int len, const double *v,
                                   Gather &&gather, Put &&put) {
    if (T.gl == 8)
        nd_rows<8>(T, fac, len, v, gather, put);
    else if (T.gl == 16)
        nd_rows<16>(T, fac, len, v, gather, put);
    else
        nd_rows<64>(T, fac, len, v, gather, put);
}

// Up: the front's right-hand side (pivots, and the border entries of this
// workgroup's rows) from r and the children's updates, by a list of update
// entries for each front entry; then update = rhs_q - W rhs_p.
__global__ void __launch_bounds__(ND_NT) k_nd_up(const NdTask *__restrict__ tasks, const int *__restrict__ piv,
                                                 const int *__restrict__ sptr, const int *__restrict__ src,
                                                 const double *__restrict__ fac, const double *__restrict__ r,
                                                 double *__restrict__ y, double *upd) {
    extern __shared__ double nd_v[];
    const NdTask T = tasks[blockIdx.x];
    auto gather = [&] {
        const int n = T.p + T.row1 - T.row0;
        for (int i = threadIdx.x; i < n; i += ND_NT) {
            const int f = T.fo + (i < T.p ? i : i + T.row0);
            double x = i < T.p ? r[piv[T.po + i]] : 0.0;
            for (int e = sptr[f]; e < sptr[f + 1]; e++) x += upd[src[e]];
            nd_v[i] = x;
            if (i < T.p && T.row0 == 0) y[T.po + i] = x;
        }
    };
    nd_dispatch(T, fac, T.p, nd_v, gather, [&](int row, double s) { upd[T.bo + row] = nd_v[T.p + row - T.row0] - s; });
}

// Down: x_p = [inv(F11) | -U] [rhs_p ; x_q]; z holds the correction by
// matrix row for the nodes below, x takes it.  A right-hand side that is not
// finite reaches the root of its component and from there every unknown, and
// x stays what it was.
__global__ void __launch_bounds__(ND_NT) k_nd_down(const NdTask *__restrict__ tasks, const int *__restrict__ piv,
                                                   const int *__restrict__ border, const double *__restrict__ fac,
                                                   const double *__restrict__ y, double *z, double *__restrict__ x) {
    extern __shared__ double nd_v[];
    const NdTask T = tasks[blockIdx.x];
    const int m = T.p + T.q;
    auto gather = [&] {
        constexpr int U = 8;
        for (int i0 = threadIdx.x; i0 < m; i0 += U * ND_NT) {
            int g[U];
            double x[U];
#pragma unroll
            for (int q = 0; q < U; q++) {
                const int i = i0 + q * ND_NT;
                g[q] = i >= T.p && i < m ? border[T.bo + i - T.p] : -1;
            }
#pragma unroll
            for (int q = 0; q < U; q++) {
                const int i = i0 + q * ND_NT;
                x[q] = g[q] >= 0 ? z[g[q]] : i < T.p ? y[T.po + i] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < U; q++)
                if (i0 + q * ND_NT < m) nd_v[i0 + q * ND_NT] = x[q];
        }
    };
    nd_dispatch(T, fac, m, nd_v, gather, [&](int row, double s) {
        const int g = piv[T.po + row];
        const double x0 = x[g];
        z[g] = s;
        x[g] = isfinite(s) ? x0 + s : x0;
    });
}

class NdSolver {
  public:
    bool ready = false;
    double flops = 0, entries = 0;

    // false (no plan) when the factors would cost more than max_flops or
    // max_entries, or a front exceeds LDS
    bool build(const std::vector<int> &rp, const std::vector<int> &ci, const std::vector<double> &v, hipStream_t st,
               double max_flops, double max_entries) {
        ready = false;
        const int n = (int)rp.size() - 1;
        if (n <= 0 || ci.empty()) return false;
        NdTree T;
        T.symbolic(rp, ci, ND_LEAF);
        flops = T.flops;
        entries = T.entries;
        if (!T.affordable(max_flops, max_entries, ND_FRONT) || !T.numeric(rp, ci, v)) return false;
        const int nn = (int)T.nodes.size();
        std::vector<int> piv, border, sptr(1, 0), src, bo(nn, 0);
        std::vector<double> fac;
        fac.reserve((size_t)T.entries);
        std::vector<std::vector<NdTask>> up(T.height), down(T.height);
        height_ = T.height;
        ulds_.assign(height_, 0);
        dlds_.assign(height_, 0);
        std::vector<std::vector<int>> from;
        for (int q = 0; q < nn; q++) {
            NdNode &N = T.nodes[q];
            NdTask t;
            t.p = (int)N.piv.size();
            t.q = (int)N.border.size();
            t.po = (int)piv.size();
            t.bo = bo[q] = (int)border.size();
            t.fo = (int)sptr.size() - 1;
            const int m = t.p + t.q;
            // the children's update entries of each front entry, in the
            // children's order
            from.assign(m, {});
            for (int c : N.child)
                for (size_t k = 0; k < T.nodes[c].cmap.size(); k++) from[T.nodes[c].cmap[k]].push_back(bo[c] + (int)k);
            for (auto &f : from) {
                src.insert(src.end(), f.begin(), f.end());
                sptr.push_back((int)src.size());
            }
            piv.insert(piv.end(), N.piv.begin(), N.piv.end());
            border.insert(border.end(), N.border.begin(), N.border.end());
            auto cut = [&](int rows, int len, long at, std::vector<NdTask> &out) {
                t.at = at;
                t.gl = nd_lanes(len);
                const int step = ND_NT / t.gl;
                for (t.row0 = 0; t.row0 < std::max(rows, 1); t.row0 += step) {
                    t.row1 = std::min(rows, t.row0 + step);
                    out.push_back(t);
                }
            };
            if (t.q > 0) {
                cut(t.q, t.p, (long)fac.size(), up[N.height]);
            } else {  // a root only gathers: 256 pivots per workgroup
                NdTask c = t;
                c.row0 = c.row1 = 0;
                c.at = 0;
                c.gl = 64;
                for (int k = 0; k < t.p; k += ND_NT) {
                    c.po = t.po + k;
                    c.fo = t.fo + k;
                    c.p = std::min(ND_NT, t.p - k);
                    up[N.height].push_back(c);
                }
            }
            ulds_[N.height] = std::max(ulds_[N.height], t.p + ND_NT / 8);
            fac.insert(fac.end(), N.W.begin(), N.W.end());
            cut(t.p, m, (long)fac.size(), down[N.height]);
            dlds_[N.height] = std::max(dlds_[N.height], m);
            fac.insert(fac.end(), N.G.begin(), N.G.end());
            std::vector<double>().swap(N.W);
            std::vector<double>().swap(N.G);
        }
        up_.assign(height_ + 1, 0);
        down_.assign(height_ + 1, 0);
        std::vector<NdTask> ut, dt;
        for (int h = 0; h < height_; h++) {
            ut.insert(ut.end(), up[h].begin(), up[h].end());
            dt.insert(dt.end(), down[h].begin(), down[h].end());
            up_[h + 1] = (int)ut.size();
            down_[h + 1] = (int)dt.size();
        }
        put(piv_, piv, st);
        put(border_, border, st);
        put(sptr_, sptr, st);
        put(src_, src, st);
        put(fac_, fac, st);
        put(ut_, ut, st);
        put(dt_, dt, st);
        y_.alloc(piv.size());
        updv_.alloc(border.size());
        z_.alloc(n);
        k_fill<double><<<nblocks(n), BLOCK, 0, st>>>(n, z_.p, 0.0);
        ready = true;
        return true;
    }

    void release() {
        ready = false;
        for (KBuf<int> *b : {&piv_, &border_, &sptr_, &src_}) b->free();
        ut_.free();
        dt_.free();
        for (KBuf<double> *b : {&fac_, &y_, &updv_, &z_}) b->free();
    }

    // x += A^-1 r
    void correct(const double *r, double *x, hipStream_t st) {
        for (int h = 0; h < height_; h++)
            k_nd_up<<<up_[h + 1] - up_[h], ND_NT, ulds_[h] * sizeof(double), st>>>(ut_.p + up_[h], piv_.p, sptr_.p, src_.p,
                                                                                 fac_.p, r, y_.p, updv_.p);
        for (int h = height_ - 1; h >= 0; h--)
            k_nd_down<<<down_[h + 1] - down_[h], ND_NT, dlds_[h] * sizeof(double), st>>>(
                dt_.p + down_[h], piv_.p, border_.p, fac_.p, y_.p, z_.p, x);
    }

  private:
    int height_ = 0;
    std::vector<int> up_, down_, ulds_, dlds_;
    KBuf<int> piv_, border_, sptr_, src_;
    KBuf<NdTask> ut_, dt_;
    KBuf<double> fac_, y_, updv_, z_;

    template <typename T>
    static void put(KBuf<T> &d, const std::vector<T> &h, hipStream_t st) {
        d.alloc(h.size());
        if (!h.empty() && (hipMemcpyAsync(d.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, st) != hipSuccess ||
                           hipStreamSynchronize(st) != hipSuccess))
            throw std::runtime_error("direct factors: upload failed");
    }
};

}  // namespace hfh
