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
// refinement: graded 4-level contraction, mixed form, 226 -> 30 ms;
// 12^3 wall-layer cavity 57 -> 13 ms, where a solve reads 0.57 GB of factors
// (host factors: 1.5e11 operations, 4 s on 8 cores).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <stdexcept>
#include <thread>
#include <vector>

#include "hfh_krylov.hpp"
#include "hfh_domain.hpp"
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
    auto work = [&] {
        for (int i; (i = next.fetch_add(step)) < m;) rows(i, std::min(m, i + step));
    };
    std::vector<std::thread> th;
    for (int t = 1; t < nt; t++) th.emplace_back(work);
    work();
    for (auto &t : th) t.join();
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
            auto work = [&](int t) {
                if (pos[t].empty()) pos[t].assign(n, -1);
                for (size_t i; ok && (i = next++) < list.size();)
                    if (!front(nodes[list[i]], rp, ci, v, tp, tr, tv, pos[t], 1)) ok = false;
            };
            std::vector<std::thread> th;
            for (int t = 1; t < std::min<int>(nt, (int)list.size()); t++) th.emplace_back(work, t);
            work(0);
            for (auto &t : th) t.join();
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
struct NdDev {
    int p, q;        // pivots, border
    int po, bo;      // first pivot / border entry of the node's lists
    int kid0, kid1;  // children
    long w, g;       // W and G in the factor array
};
constexpr int ND_NT = 256;
constexpr int ND_LDS = 8192;  // front entries held in LDS (64 KiB)

// rows [row0, row1) of dot products with the vector v (len entries, LDS),
// GL lanes per row; f(row, sum) on the group's first lane.  Four loads per
// lane are in flight.
template <int GL, typename F>
__device__ inline void nd_rows(const double *__restrict__ M, int len, int row0, int row1, const double *v, F &&f) {
    const int lane = threadIdx.x % GL;
    for (int r = row0 + (int)threadIdx.x / GL; r < row1; r += ND_NT / GL) {
        const double *m = M + (size_t)r * len;
        double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
        int k = lane;
        for (; k + 3 * GL < len; k += 4 * GL) {
            const double a0 = m[k], a1 = m[k + GL], a2 = m[k + 2 * GL], a3 = m[k + 3 * GL];
            s0 += a0 * v[k];
            s1 += a1 * v[k + GL];
            s2 += a2 * v[k + 2 * GL];
            s3 += a3 * v[k + 3 * GL];
        }
        for (; k < len; k += GL) s0 += m[k] * v[k];
        double s = (s0 + s1) + (s2 + s3);
#pragma unroll
        for (int o = GL / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) f(r, s);
    }
}

// Up: one workgroup per (node, rows of W) of a tree height.  The front's
// right-hand side is gathered into LDS (the children in turn, so no two
// lanes add to one entry), then update = rhs_q - W rhs_p.
__global__ void __launch_bounds__(ND_NT) k_nd_up(const int4 *__restrict__ tasks, const NdDev *__restrict__ nodes,
                                                 const int *__restrict__ kids, const int *__restrict__ piv,
                                                 const int *__restrict__ cmap, const double *__restrict__ fac,
                                                 const double *__restrict__ r, double *__restrict__ y, double *upd) {
    extern __shared__ double nd_v[];
    const int4 t = tasks[blockIdx.x];
    const NdDev N = nodes[t.x];
    for (int i = threadIdx.x; i < N.p + N.q; i += ND_NT) nd_v[i] = i < N.p ? r[piv[N.po + i]] : 0.0;
    for (int c = N.kid0; c < N.kid1; c++) {
        const NdDev C = nodes[kids[c]];
        __syncthreads();
        for (int j = threadIdx.x; j < C.q; j += ND_NT) nd_v[cmap[C.bo + j]] += upd[C.bo + j];
    }
    __syncthreads();
    if (t.y == 0)
        for (int i = threadIdx.x; i < N.p; i += ND_NT) y[N.po + i] = nd_v[i];
    auto put = [&](int row, double s) { upd[N.bo + row] = nd_v[N.p + row] - s; };
    if (N.p > 256)
        nd_rows<64>(fac + N.w, N.p, t.y, t.z, nd_v, put);
    else
        nd_rows<16>(fac + N.w, N.p, t.y, t.z, nd_v, put);
}

// Down: x_p = [inv(F11) | -U] [rhs_p ; x_q]; z holds the correction by
// matrix row for the nodes below, x takes it.
__global__ void __launch_bounds__(ND_NT) k_nd_down(const int4 *__restrict__ tasks, const NdDev *__restrict__ nodes,
                                                   const int *__restrict__ piv, const int *__restrict__ border,
                                                   const double *__restrict__ fac, const double *__restrict__ y,
                                                   double *z, double *__restrict__ x) {
    extern __shared__ double nd_v[];
    const int4 t = tasks[blockIdx.x];
    const NdDev N = nodes[t.x];
    const int m = N.p + N.q;
    for (int i = threadIdx.x; i < m; i += ND_NT) nd_v[i] = i < N.p ? y[N.po + i] : z[border[N.bo + i - N.p]];
    __syncthreads();
    auto put = [&](int row, double s) {
        const int g = piv[N.po + row];
        z[g] = s;
        x[g] += s;
    };
    if (m > 256)
        nd_rows<64>(fac + N.g, m, t.y, t.z, nd_v, put);
    else
        nd_rows<16>(fac + N.g, m, t.y, t.z, nd_v, put);
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
        T.symbolic(rp, ci, 96);
        flops = T.flops;
        entries = T.entries;
        if (T.flops > max_flops || T.entries > max_entries) return false;
        for (const NdNode &N : T.nodes)
            if ((int)(N.piv.size() + N.border.size()) > ND_LDS) return false;
        if (!T.numeric(rp, ci, v)) return false;
        const int nn = (int)T.nodes.size();
        std::vector<NdDev> dv(nn);
        std::vector<int> kids, piv, border, cmap;
        std::vector<double> fac;
        fac.reserve((size_t)T.entries);
        std::vector<std::vector<int4>> up(T.height), down(T.height);
        height_ = T.height;
        lds_.assign(height_, 0);
        for (int q = 0; q < nn; q++) {
            NdNode &N = T.nodes[q];
            NdDev &d = dv[q];
            d.p = (int)N.piv.size();
            d.q = (int)N.border.size();
            d.po = (int)piv.size();
            d.bo = (int)border.size();
            d.kid0 = (int)kids.size();
            kids.insert(kids.end(), N.child.begin(), N.child.end());
            d.kid1 = (int)kids.size();
            piv.insert(piv.end(), N.piv.begin(), N.piv.end());
            border.insert(border.end(), N.border.begin(), N.border.end());
            cmap.insert(cmap.end(), N.cmap.begin(), N.cmap.end());
            cmap.resize(border.size(), 0);  // a root's (empty) border has no map
            d.w = (long)fac.size();
            fac.insert(fac.end(), N.W.begin(), N.W.end());
            d.g = (long)fac.size();
            fac.insert(fac.end(), N.G.begin(), N.G.end());
            std::vector<double>().swap(N.W);
            std::vector<double>().swap(N.G);
            const int m = d.p + d.q;
            lds_[N.height] = std::max(lds_[N.height], m);
            // about 8192 factor entries per workgroup, 16 to 64 rows
            auto cut = [&](int rows, int len, std::vector<int4> &out) {
                const int step = std::max(16, std::min(64, 8192 / std::max(len, 1) / 16 * 16));
                for (int r = 0; r < std::max(rows, 1); r += step)
                    out.push_back(make_int4(q, r, std::min(rows, r + step), 0));
            };
            cut(d.q, d.p, up[N.height]);
            cut(d.p, m, down[N.height]);
        }
        up_.assign(height_ + 1, 0);
        down_.assign(height_ + 1, 0);
        std::vector<int4> ut, dt;
        for (int h = 0; h < height_; h++) {
            ut.insert(ut.end(), up[h].begin(), up[h].end());
            dt.insert(dt.end(), down[h].begin(), down[h].end());
            up_[h + 1] = (int)ut.size();
            down_[h + 1] = (int)dt.size();
        }
        put(nodes_, dv, st);
        put(kids_, kids, st);
        put(piv_, piv, st);
        put(border_, border, st);
        put(cmap_, cmap, st);
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

    // x += A^-1 r
    void correct(const double *r, double *x, hipStream_t st) {
        for (int h = 0; h < height_; h++)
            k_nd_up<<<up_[h + 1] - up_[h], ND_NT, lds_[h] * sizeof(double), st>>>(ut_.p + up_[h], nodes_.p, kids_.p, piv_.p,
                                                                                cmap_.p, fac_.p, r, y_.p, updv_.p);
        for (int h = height_ - 1; h >= 0; h--)
            k_nd_down<<<down_[h + 1] - down_[h], ND_NT, lds_[h] * sizeof(double), st>>>(
                dt_.p + down_[h], nodes_.p, piv_.p, border_.p, fac_.p, y_.p, z_.p, x);
    }

  private:
    int height_ = 0;
    std::vector<int> up_, down_, lds_;
    KBuf<NdDev> nodes_;
    KBuf<int> kids_, piv_, border_, cmap_;
    KBuf<int4> ut_, dt_;
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
