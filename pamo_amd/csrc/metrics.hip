// Surface metrics on gfx950 behind pamo_metrics_* of include/pamo_hip.h:
// point-to-mesh squared distances and the two-sided Hausdorff distance
// between triangle meshes, with the semantics of the libigl calls the
// reference makes (simp_cuda/safe_project/src/pamo_safe_project/metrics.py:31-51):
//   igl.point_mesh_squared_distance(P, V, F) -> (sqrD, I, C)
//   igl.hausdorff(VA, FA, VB, FB) = sqrt(max(max_{a in VA} d(a, B)^2,
//                                            max_{b in VB} d(b, A)^2))
// (libigl 2.5.1 hausdorff: vertex-to-surface both ways).
//
// Distances are FP64.  A point's squared distance to a triangle is the one of
// Ericson's closest point (Real-Time Collision Detection 5.1.5, the region
// test libigl's point_simplex_squared_distance uses), evaluated in double
// without contraction.  The nearest triangle is found by branch and bound
// over an LBVH of float boxes rounded outward from the double corners: a
// subtree is skipped only when its box is farther than the best distance so
// far, so the result is the minimum over all triangles up to rounding at
// exact ties, with ties broken by the smaller face index.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>

#include "pamo_hip.h"
#include "lbvh_tree.h"

namespace pamo {
namespace metrics {

using s3::kB;
using s3::Tree;
using s3::TreeView;

struct D3 {
    double x, y, z;
};
__device__ __forceinline__ D3 operator-(D3 a, D3 b) { return D3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ D3 operator+(D3 a, D3 b) { return D3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ D3 operator*(double s, D3 a) { return D3{s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ double ddot(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ D3 load3(const double* __restrict__ p, long long i) {
    return D3{p[3 * i], p[3 * i + 1], p[3 * i + 2]};
}

// Ericson 5.1.5: closest point of triangle abc to p by Voronoi regions.
__device__ inline D3 closest_on_tri_d(D3 p, D3 a, D3 b, D3 c) {
    const D3 ab = b - a, ac = c - a, ap = p - a;
    const double d1 = ddot(ab, ap), d2 = ddot(ac, ap);
    if (d1 <= 0.0 && d2 <= 0.0) return a;
    const D3 bp = p - b;
    const double d3 = ddot(ab, bp), d4 = ddot(ac, bp);
    if (d3 >= 0.0 && d4 <= d3) return b;
    const double vc = d1 * d4 - d3 * d2;
    if (vc <= 0.0 && d1 >= 0.0 && d3 <= 0.0) return a + (d1 / (d1 - d3)) * ab;
    const D3 cp = p - c;
    const double d5 = ddot(ab, cp), d6 = ddot(ac, cp);
    if (d6 >= 0.0 && d5 <= d6) return c;
    const double vb = d5 * d2 - d1 * d6;
    if (vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0) return a + (d2 / (d2 - d6)) * ac;
    const double va = d3 * d6 - d5 * d4;
    if (va <= 0.0 && (d4 - d3) >= 0.0 && (d5 - d6) >= 0.0)
        return b + ((d4 - d3) / ((d4 - d3) + (d5 - d6))) * (c - b);
    const double den = 1.0 / (va + vb + vc);
    const double v = vb * den, w = vc * den;
    return a + v * ab + w * ac;
}

// Largest float <= x and smallest float >= x.
__device__ __forceinline__ float f_down(double x) {
    float f = (float)x;
    return (double)f > x ? nextafterf(f, -__builtin_huge_valf()) : f;
}
__device__ __forceinline__ float f_up(double x) {
    float f = (float)x;
    return (double)f < x ? nextafterf(f, __builtin_huge_valf()) : f;
}

// Number of faces with a corner outside [0, nV).
__global__ void __launch_bounds__(kB) check_faces_k(const int* __restrict__ F, int nF, int nV, int* bad) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nF) return;
    const int a = F[3 * (long long)f], b = F[3 * (long long)f + 1], c = F[3 * (long long)f + 2];
    if (a < 0 || a >= nV || b < 0 || b >= nV || c < 0 || c >= nV) atomicAdd(bad, 1);
}

// Float box of each face, rounded outward from its double corners.
__global__ void __launch_bounds__(kB) face_box_d_k(const double* __restrict__ V, const int* __restrict__ F, int nF,
                                                  float4* __restrict__ item) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nF) return;
    const D3 a = load3(V, F[3 * (long long)f]), b = load3(V, F[3 * (long long)f + 1]),
             c = load3(V, F[3 * (long long)f + 2]);
    item[2 * (long long)f] = make_float4(f_down(fmin(fmin(a.x, b.x), c.x)), f_down(fmin(fmin(a.y, b.y), c.y)),
                                         f_down(fmin(fmin(a.z, b.z), c.z)), 0.0f);
    item[2 * (long long)f + 1] = make_float4(f_up(fmax(fmax(a.x, b.x), c.x)), f_up(fmax(fmax(a.y, b.y), c.y)),
                                             f_up(fmax(fmax(a.z, b.z), c.z)), 0.0f);
}

__device__ __forceinline__ double box_d2(D3 p, float4 lo, float4 hi) {
    const double dx = fmax(fmax((double)lo.x - p.x, 0.0), p.x - (double)hi.x);
    const double dy = fmax(fmax((double)lo.y - p.y, 0.0), p.y - (double)hi.y);
    const double dz = fmax(fmax((double)lo.z - p.z, 0.0), p.z - (double)hi.z);
    return dx * dx + dy * dy + dz * dz;
}

// Morton code (its upper 16 bits) of each point in the tree's whole box, the
// walk order of the queries: the lanes of a wave then walk the same part of the
// tree.  A point outside the box takes the code of its nearest corner or side.
__global__ void __launch_bounds__(kB) point_keys_k(const double* __restrict__ P, int nP,
                                                   const float* __restrict__ whole, uint32_t* __restrict__ key,
                                                   uint32_t* __restrict__ val) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nP) return;
    const D3 p = load3(P, i);
    const float c[3] = {(float)p.x, (float)p.y, (float)p.z};
    float u[3];
    for (int d = 0; d < 3; ++d) {
        const float ext = whole[3 + d] - whole[d];
        u[d] = ext > 0.0f ? fminf(fmaxf((c[d] - whole[d]) / ext, 0.0f), 1.0f) : 0.0f;
    }
    key[i] = morton3(u[0], u[1], u[2]) >> 14;
    val[i] = (uint32_t)i;
}

constexpr int kWaveStack = 1024;  // nodes waiting in a wave's walk of one query (8 KiB)

// Steps after which a lane leaves its query to a whole wave.  Up to
// kWavePoints queries take a wave each in a few turns of the chip (some 5000
// such waves are resident), so a lane only finds a first bound (32 steps: about
// the depth of the tree, twice); beyond that the lanes finish the ordinary
// queries by themselves (128 steps) and leave the long ones.  Measured on
// surface samples against a 200k-face union (ms a call, tree build included),
// with 32 | 64 | 128 | 384 steps: 4,096 points 0.34 | 0.45 | 0.62 | 0.64;
// 20,000: 0.48 | 0.54 | 0.65 | 0.69; 100,003: 1.17 | 1.00 | 0.77 | 0.83;
// 300,000: 2.85 | 2.20 | 0.99 | 1.04.
constexpr long long kWavePoints = 32768;
static int lane_steps(long long nP) { return nP <= kWavePoints ? 32 : 128; }

// A nearest-face query under way: the point, and the best face so far.
struct Near {
    D3 p;
    double best;
    int f;
    D3 c;
};

// Face f as the best, if it is: the smallest distance, and among equal ones
// the smallest face (so the result does not depend on the order of the visits).
__device__ __forceinline__ void near_face(Near& q, const double* __restrict__ V, const int* __restrict__ F, int f) {
    const D3 c = closest_on_tri_d(q.p, load3(V, F[3 * (long long)f]), load3(V, F[3 * (long long)f + 1]),
                                  load3(V, F[3 * (long long)f + 2]));
    const D3 d = c - q.p;
    const double d2 = ddot(d, d);
    if (d2 < q.best || (d2 == q.best && f < q.f)) {
        q.best = d2;
        q.f = f;
        q.c = c;
    }
}

__device__ __forceinline__ void near_store(const Near& q, long long i, double* __restrict__ sqd, int* __restrict__ I,
                                           double* __restrict__ C) {
    sqd[i] = q.best;
    if (I) I[i] = q.f;
    if (C) {
        C[3 * i] = q.c.x;
        C[3 * i + 1] = q.c.y;
        C[3 * i + 2] = q.c.z;
    }
}

// A lower bound in 32 bits of a squared distance: 0 where the relative rounding
// does not hold, the largest number where 32 bits end (distances from 1.8e19
// on, whose waiting nodes are then always opened).
__device__ __forceinline__ float near_bound(double d) {
    return d > 1e-30 ? fminf((float)(d * (1.0 - 1.2e-7)), 3.402823466e38f) : 0.0f;
}

// The whole tree by parent links, with the best so far: for a walk whose
// stack ran out.
__device__ inline void near_by_links(Near& q, TreeView T, const double* __restrict__ V, const int* __restrict__ F,
                                     int* err) {
    const int n = T.n;
    auto bd = [&](int node) {  // (the root, which has no box, is entered)
        if (node == 0) return 0.0;
        return box_d2(q.p, T.box[2 * (long long)T.slot[node]], T.box[2 * (long long)T.slot[node] + 1]);
    };
    int prev = -1, cur = 0;
    const long long max_steps = 3LL * (2LL * n - 1) + 1;
    for (long long steps = 0; cur >= 0; ++steps) {
        if (steps >= max_steps || cur > 2 * n - 2) {
            walk_overrun(err);
            break;
        }
        const int par = cur == 0 ? -1 : T.slot[cur] >> 1;
        int next;
        if (prev == par) {
            if (bd(cur) > q.best) {
                next = par;
            } else if (cur >= n - 1) {
                near_face(q, V, F, (int)T.val[cur - (n - 1)]);
                next = par;
            } else {
                const int l = T.left[cur], r = T.right[cur];
                next = bd(l) <= bd(r) ? l : r;
            }
        } else {
            const int l = T.left[cur], r = T.right[cur];
            const bool left_first = bd(l) <= bd(r);
            const int first = left_first ? l : r, second = left_first ? r : l;
            next = prev == first ? second : par;
        }
        prev = cur;
        cur = next;
    }
}

// Nearest face of each point, a point a lane (lane t takes point order[t], or
// t without an order).  Bound by the latency of the node loads: a step reads
// one child pair (both children's boxes in one round of loads) and
// never climbs.  Near child first, subtrees farther than the best
// skipped.  Writes sqd[i] and, when given, I[i] and the closest point C[i].
// With `rest`, a query not finished after max_steps steps is left to
// point_mesh_wave_k: its point and best face go to rest, *n_rest counts them.
__global__ void __launch_bounds__(kWave) point_mesh_k(const double* __restrict__ P, long long nP,
                                                     const uint32_t* __restrict__ order, TreeView T,
                                                     const double* __restrict__ V, const int* __restrict__ F,
                                                     double* __restrict__ sqd, int* __restrict__ I,
                                                     double* __restrict__ C, int max_steps, int2* __restrict__ rest,
                                                     int* __restrict__ n_rest, int* err) {
    __shared__ int stk_n[s3::kNearStack][kWave];
    __shared__ float stk_d[s3::kNearStack][kWave];
    const int lane = threadIdx.x;
    const long long t = (long long)blockIdx.x * kWave + lane;
    if (t >= nP) return;
    const long long i = order ? (long long)order[t] : t;
    Near q{load3(P, i), __builtin_huge_val(), -1, D3{0.0, 0.0, 0.0}};
    const int n = T.n;
    bool left_over = false;
    if (n == 1) {
        near_face(q, V, F, (int)T.val[0]);
    } else if (n > 1) {
        bool dropped = false;
        int cur = 0, sp = 0;  // cur: internal node, ~face, or n when the stack is to be popped
        for (long long steps = 0;; ++steps) {
            if (rest && steps >= max_steps) {
                left_over = true;
                break;
            }
            if (steps >= 4LL * n) {  // every node, leaf and pop at most once
                walk_overrun(err);
                break;
            }
            if (cur >= n - 1) {
                if (sp == 0) break;
                --sp;
                cur = (double)stk_d[sp][lane] > q.best ? n : stk_n[sp][lane];
                continue;
            }
            if (cur < 0) {
                near_face(q, V, F, ~cur);
                cur = n;
                continue;
            }
            const float4* pair = T.box + 4 * (long long)cur;
            const float4 la = pair[0], lb = pair[1], ra = pair[2], rb = pair[3];
            const double dl = box_d2(q.p, la, lb), dr = box_d2(q.p, ra, rb);
            const bool left_first = dl <= dr;
            const double dn = left_first ? dl : dr, df = left_first ? dr : dl;
            const int cn = __float_as_int(left_first ? la.w : ra.w), cf = __float_as_int(left_first ? ra.w : la.w);
            if (!(df > q.best)) {
                if (sp < s3::kNearStack) {
                    stk_d[sp][lane] = near_bound(df);
                    stk_n[sp][lane] = cf;
                    ++sp;
                } else {
                    dropped = true;
                }
            }
            cur = dn > q.best ? n : cn;
        }
        if (dropped && !left_over) near_by_links(q, T, V, F, err);
    }
    near_store(q, i, sqd, I, C);
    const uint64_t m = __ballot(left_over);
    if (m == 0) return;
    int base = 0;
    if (lane == __ffsll((unsigned long long)m) - 1) base = atomicAdd(n_rest, (int)__popcll(m));
    base = __shfl(base, __ffsll((unsigned long long)m) - 1);
    if (left_over) rest[base + lanes_below(m)] = make_int2((int)i, q.f);
}

// The query of rest entry e, with the best that point_mesh_k found for it.
__device__ __forceinline__ Near near_resume(const double* __restrict__ P, const double* __restrict__ V,
                                            const int* __restrict__ F, int2 e) {
    Near q{load3(P, e.x), __builtin_huge_val(), -1, D3{0.0, 0.0, 0.0}};
    if (e.y >= 0) near_face(q, V, F, e.y);
    return q;
}

// The queries that a lane did not finish, a wave each.  The nodes still to
// visit lie on one LIFO in LDS; each step takes up to 64 of them, a lane each,
// and the lanes share their best after a step that reached faces.  Such a
// query (a point far from the surface, at nearly the same distance from much
// of it) visits thousands of nodes, and alone in its lane waits for one memory
// latency each: 10,242 vertices of a sphere around a 200k-face mesh took 7.1
// ms a call with a lane each over parent links, 3.5 ms with the stack, and
// 0.44 ms with this kernel; the mesh's 97,268 vertices against the 20k-face
// sphere 9.5, 3.6 and 1.5 ms.  (One walk for 64 neighbouring points, nodes
// read at one address, took 2.8 ms there: the union of 64 points' nodes is
// several times one point's.)
__global__ void __launch_bounds__(kWave) point_mesh_wave_k(const double* __restrict__ P, TreeView T,
                                                          const double* __restrict__ V, const int* __restrict__ F,
                                                          double* __restrict__ sqd, int* __restrict__ I,
                                                          double* __restrict__ C, const int2* __restrict__ rest,
                                                          const int* __restrict__ n_rest, int* err) {
    __shared__ int stk_n[kWaveStack];
    __shared__ float stk_d[kWaveStack];
    const int lane = threadIdx.x;
    const int nq = *n_rest, n = T.n;
    for (long long t = blockIdx.x; t < nq; t += gridDim.x) {
        const int2 e = rest[t];
        Near q = near_resume(P, V, F, e);
        bool dropped = false;
        if (lane == 0) {
            stk_n[0] = 0;
            stk_d[0] = 0.0f;
        }
        wave_sync();
        int size = 1;  // wave-uniform
        for (long long steps = 0; size > 0; ++steps) {
            if (steps >= 2LL * n) {  // every step takes a node, every node once
                if (lane == 0) walk_overrun(err);
                break;
            }
            const int take = size < kWave ? size : kWave;
            int x = -1;
            if (lane < take) {
                const int s = size - take + lane;
                if (!((double)stk_d[s] > q.best)) x = stk_n[s];
            }
            size -= take;
            wave_sync();  // every pop has read its entry before pushes reuse the slots
            int cl = -1, cr = -1, fl = -1, fr = -1;
            float bl = 0.0f, br = 0.0f;
            if (x >= 0) {
                const float4* pair = T.box + 4 * (long long)x;
                const float4 la = pair[0], lb = pair[1], ra = pair[2], rb = pair[3];
                const double dl = box_d2(q.p, la, lb), dr = box_d2(q.p, ra, rb);
                if (!(dl > q.best)) {
                    cl = __float_as_int(la.w);
                    bl = near_bound(dl);
                }
                if (!(dr > q.best)) {
                    cr = __float_as_int(ra.w);
                    br = near_bound(dr);
                }
                if (cl < -1 || (cl == -1 && !(dl > q.best))) {
                    fl = ~cl;
                    cl = -1;
                }
                if (cr < -1 || (cr == -1 && !(dr > q.best))) {
                    fr = ~cr;
                    cr = -1;
                }
            }
            const uint64_t ml = __ballot(cl >= 0), mr = __ballot(cr >= 0);
            const int pl = size + lanes_below(ml), pr = size + (int)__popcll(ml) + lanes_below(mr);
            if (cl >= 0) {
                if (pl < kWaveStack) {
                    stk_n[pl] = cl;
                    stk_d[pl] = bl;
                } else {
                    dropped = true;
                }
            }
            if (cr >= 0) {
                if (pr < kWaveStack) {
                    stk_n[pr] = cr;
                    stk_d[pr] = br;
                } else {
                    dropped = true;
                }
            }
            size = min(size + (int)__popcll(ml) + (int)__popcll(mr), kWaveStack);
            if (__ballot(fl >= 0 || fr >= 0)) {
                if (fl >= 0) near_face(q, V, F, fl);
                if (fr >= 0) near_face(q, V, F, fr);
                // the wave's best (distance, then face)
                double b = q.best;
                int f = q.f;
#pragma unroll
                for (int o = kWave / 2; o > 0; o >>= 1) {
                    const double ob = __shfl_xor(b, o);
                    const int of = __shfl_xor(f, o);
                    if (ob < b || (ob == b && of >= 0 && (f < 0 || of < f))) {
                        b = ob;
                        f = of;
                    }
                }
                const uint64_t own = __ballot(q.f == f && q.best == b);
                if (own) {
                    const int src = __ffsll((unsigned long long)own) - 1;
                    q.c = D3{__shfl(q.c.x, src), __shfl(q.c.y, src), __shfl(q.c.z, src)};
                    q.best = b;
                    q.f = f;
                }
            }
            wave_sync();
        }
        if (__ballot(dropped)) near_by_links(q, T, V, F, err);  // every lane alike
        if (lane == 0) near_store(q, e.x, sqd, I, C);
        wave_sync();
    }
}

// Maximum of non-negative doubles (their bit patterns order like the values;
// a NaN orders above every number and propagates).
__global__ void __launch_bounds__(kB) max_bits_k(const double* __restrict__ x, long long n,
                                                unsigned long long* out) {
    __shared__ unsigned long long red[kB];
    unsigned long long m = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        m = max(m, (unsigned long long)__double_as_longlong(x[i]));
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = kB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicMax(out, red[0]);
}

// Device memory of one call: the tree over the mesh's faces, the sort and
// scan workspace, and two flags (faces indexing outside the vertices; a tree
// walk that exceeded its bound).  A metrics context owns one that grows with
// the mesh; pamo_point_mesh_sqdist_noalloc carves one out of a static array.
struct Work {
    Tree tree;
    int* ws = nullptr;
    int* flags = nullptr;  // [3] device: bad faces, walk overrun, queries left over
    int* h_flags = nullptr;  // [2] host
    // walk order of up to kCallPoints queries (null: the points' own order):
    // Morton keys, point numbers, and the sort's second pair of buffers
    uint32_t *qkey = nullptr, *qval = nullptr, *qkey2 = nullptr, *qval2 = nullptr;
    int* qws = nullptr;
    long long cap_q = 0;
    int2* rest = nullptr;  // queries that a lane alone did not finish (null: it goes on)
    long long cap_rest = 0;
};

struct Ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    Work w;
    long long cap_ws = 0;
    double* sqd = nullptr;  // Hausdorff: per-vertex squared distances
    long long cap_sqd = 0;
    unsigned long long* mx = nullptr;   // [1]
    unsigned long long* h_mx = nullptr; // pinned
};

static void ctx_free(Ctx& c) {
    s3::tree_free(c.w.tree);
    void* ptrs[] = {c.w.ws, c.sqd, c.w.flags, c.mx, c.w.qkey, c.w.qval, c.w.qkey2, c.w.qval2, c.w.qws, c.w.rest};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    if (c.w.h_flags) (void)hipHostFree(c.w.h_flags);
    if (c.h_mx) (void)hipHostFree(c.h_mx);
    if (c.stream) (void)hipStreamDestroy(c.stream);
}

// Checks every face index, then builds the tree over the faces of (V, F);
// w's tree and workspace must hold nF faces.
static int build_tree(Work& w, hipStream_t st, const double* V, int nV, const int* F, int nF, const char* who) {
    PAMO_CHECK(V && F && nV > 0 && nF > 0, std::string(who) + ": empty or null mesh");
    PAMO_TRY(fill(w.flags, 0, 1, st));
    hipLaunchKernelGGL(check_faces_k, dim3(grid_for(nF, kB)), dim3(kB), 0, st, F, nF, nV, w.flags);
    PAMO_HIP(hipGetLastError());
    PAMO_HIP(hipMemcpyAsync(w.h_flags, w.flags, sizeof(int), hipMemcpyDeviceToHost, st));
    PAMO_HIP(hipStreamSynchronize(st));
    PAMO_CHECK(w.h_flags[0] == 0,
               std::string(who) + ": " + std::to_string(w.h_flags[0]) + " faces index outside the vertices");
    hipLaunchKernelGGL(face_box_d_k, dim3(grid_for(nF, kB)), dim3(kB), 0, st, V, F, nF, w.tree.item);
    PAMO_HIP(hipGetLastError());
    return s3::tree_build(w.tree, nF, w.ws, st);
}

// Fewer points than this are walked in their own order.
constexpr long long kSortPoints = 4096;
// Points that are walked together: the order and leftover buffers that a
// context keeps hold no more (24 bytes a point: 384 MiB, and the sort's
// histograms).  20M points against 200k faces: 21.4 ms so, 20.9 in one turn,
// 22.9 in turns of 2^22.
constexpr long long kCallPoints = 1LL << 24;

static int query_points(Work& w, hipStream_t st, const double* P, long long nP, const double* V, const int* F,
                        double* sqd, int* I, double* C) {
    const uint32_t* order = nullptr;
    if (nP >= kSortPoints && nP <= w.cap_q && w.tree.n > 1) {
        const float* whole = w.tree.part + 6 * grid_for(w.tree.n, kBlock);
        hipLaunchKernelGGL(point_keys_k, dim3(grid_for(nP, kB)), dim3(kB), 0, st, P, (int)nP, whole, w.qkey, w.qval);
        PAMO_HIP(hipGetLastError());
        PAMO_TRY(radix_sort_pairs(w.qkey, w.qval, w.qkey2, w.qval2, (int)nP, 16, w.qws, st));
        order = w.qval;
    }
    int2* rest = nP <= w.cap_rest ? w.rest : nullptr;
    int* n_rest = rest ? w.flags + 2 : nullptr;
    if (rest) PAMO_TRY(fill(n_rest, 0, 1, st));
    hipLaunchKernelGGL(point_mesh_k, dim3(grid_for(nP, kWave)), dim3(kWave), 0, st, P, nP, order, s3::view(w.tree), V,
                       F, sqd, I, C, lane_steps(nP), rest, n_rest, w.flags + 1);
    if (rest) {
        hipLaunchKernelGGL(point_mesh_wave_k, dim3((unsigned)std::min(nP, 8192LL)), dim3(kWave), 0, st, P,
                           s3::view(w.tree), V, F, sqd, I, C, (const int2*)rest, (const int*)n_rest, w.flags + 1);
    }
    PAMO_HIP(hipGetLastError());
    return 0;
}

static int query(Work& w, hipStream_t st, const double* P, long long nP, const double* V, const int* F, double* sqd,
                 int* I, double* C) {
    for (long long k = 0; k < nP; k += kCallPoints)
        PAMO_TRY(query_points(w, st, P + 3 * k, std::min(nP - k, kCallPoints), V, F, sqd + k, I ? I + k : nullptr,
                              C ? C + 3 * k : nullptr));
    return 0;
}

// Clears the walk flag at the start of a call.
static int begin(Work& w, hipStream_t st) { return fill(w.flags + 1, 0, 1, st); }

// Reads the walk flag after the stream's work and reports an overrun.
static int finish(Work& w, hipStream_t st, const char* who) {
    PAMO_HIP(hipMemcpyAsync(w.h_flags + 1, w.flags + 1, sizeof(int), hipMemcpyDeviceToHost, st));
    PAMO_HIP(hipStreamSynchronize(st));
    PAMO_CHECK(w.h_flags[1] == 0, std::string(who) + ": a tree walk exceeded its bound (corrupted LBVH)");
    return 0;
}

// Sizes the context's tree and workspace for nF faces, and the buffers of the
// query order for nP points (none for few points).
static int reserve(Ctx& c, int nF, long long nP) {
    const long long np = std::min(nP, kCallPoints), cap = std::min(np + np / 4, kCallPoints);
    if (np > c.w.cap_rest) {
        c.w.cap_rest = 0;
        PAMO_TRY(s3::dalloc(&c.w.rest, (size_t)cap, c.stream));
        c.w.cap_rest = cap;
    }
    if (np >= kSortPoints && np > c.w.cap_q) {
        c.w.cap_q = 0;
        uint32_t** q[] = {&c.w.qkey, &c.w.qval, &c.w.qkey2, &c.w.qval2};
        for (uint32_t** x : q) PAMO_TRY(s3::dalloc(x, (size_t)cap, c.stream));
        PAMO_TRY(s3::dalloc(&c.w.qws, (size_t)radix_workspace(cap) + 256, c.stream));
        c.w.cap_q = cap;
    }
    const long long need = std::max(radix_workspace(nF + 64LL), scan_workspace(nF + 65LL)) + 256;
    if (need > c.cap_ws) {
        c.cap_ws = need + need / 4;
        PAMO_TRY(s3::dalloc(&c.w.ws, (size_t)c.cap_ws, c.stream));
    }
    return s3::tree_alloc(c.w.tree, nF, c.stream);
}

// max over sqd of the one-sided distances of (VA -> B), written to c.mx
static int one_side(Ctx& c, const double* VA, int nVA, const double* VB, int nVB, const int* FB, int nFB) {
    PAMO_CHECK(nFB > 0, "pamo_hausdorff: empty or null mesh");
    PAMO_TRY(reserve(c, nFB, nVA));
    PAMO_TRY(build_tree(c.w, c.stream, VB, nVB, FB, nFB, "pamo_hausdorff"));
    if (nVA > c.cap_sqd) {
        c.cap_sqd = nVA + nVA / 4;
        PAMO_TRY(s3::dalloc(&c.sqd, (size_t)c.cap_sqd, c.stream));
    }
    PAMO_TRY(query(c.w, c.stream, VA, nVA, VB, FB, c.sqd, nullptr, nullptr));
    const unsigned nb = std::min<unsigned>(grid_for(nVA, kB), 1024u);
    hipLaunchKernelGGL(max_bits_k, dim3(nb), dim3(kB), 0, c.stream, (const double*)c.sqd, (long long)nVA, c.mx);
    PAMO_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------------------ allocation-free variant
// pamo_point_mesh_sqdist_noalloc keeps everything a call needs beyond its
// inputs and outputs (the tree over at most kNoAllocMaxFaces faces, the sort
// and scan workspace and the two flags) in one static device array, so that
// it calls no allocator.  Host code uses the array only through the address
// hipGetSymbolAddress returns for the current device: in host code the
// symbol's name is a host-side stand-in, not a device address.
constexpr int kNoAllocMaxFaces = 1 << 16;
constexpr size_t kNoAllocBytes = (size_t)16 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocMaxDevices = 64;
struct NoAllocDevice {
    std::mutex mu;          // serialises calls on one device
    unsigned char* base = nullptr;  // device address of this device's scratch
    Work w;                 // views into it
};
static NoAllocDevice g_noalloc[kNoAllocMaxDevices];

// Carves the work buffers for up to max_faces faces out of [base, base +
// bytes) (base may be null to only measure).  Returns the bytes needed.
static size_t noalloc_layout(unsigned char* base, int max_faces, Work& w) {
    size_t off = 0;
    auto take = [&](auto*& ptr, size_t count) {
        using T = std::remove_reference_t<decltype(*ptr)>;
        off = (off + 255) & ~(size_t)255;
        ptr = base ? reinterpret_cast<T*>(base + off) : nullptr;
        off += sizeof(T) * std::max<size_t>(count, 1);
    };
    // the sizes of s3::tree_alloc for a capacity of max_faces + 16 items
    const size_t a = (size_t)max_faces + 16;
    Tree& t = w.tree;
    take(t.item, 2 * a);
    take(t.key, a); take(t.val, a); take(t.key2, a); take(t.val2, a);
    take(t.left, a); take(t.right, a); take(t.slot, 2 * a);
    take(t.range, a);
    take(t.box, 4 * a);
    take(t.pre, 2 * a); take(t.suf, 2 * a);
    const size_t nb = a / kBlock + 2, ns = nb / kBlock + 2;
    take(t.blk, 2 * nb); take(t.blkpre, 2 * nb); take(t.blksuf, 2 * nb);
    take(t.sblk, 2 * ns);
    take(t.blktab, 2 * kTabLevels * nb);
    t.tab_stride = (long long)nb;
    take(t.part, 6 * (a / kBlock + 4));
    take(t.cnt, (size_t)C_COUNT);
    t.cap = (int)a;
    const long long ws = std::max(radix_workspace(max_faces + 64LL), scan_workspace(max_faces + 65LL)) + 256;
    take(w.ws, (size_t)ws);
    take(w.flags, 3);
    return off;
}

// Resolves this device's scratch address once (with the device current) and
// lays the work buffers out in it.
static int noalloc_setup(int device, NoAllocDevice*& out) {
    PAMO_CHECK(device >= 0 && device < kNoAllocMaxDevices, "pamo_point_mesh_sqdist_noalloc: device id out of range");
    NoAllocDevice& d = g_noalloc[device];
    out = &d;
    if (d.base) return 0;
    void* ptr = nullptr;
    PAMO_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    PAMO_CHECK(ptr != nullptr, "pamo_point_mesh_sqdist_noalloc: no device address for the scratch array");
    Work probe;
    PAMO_CHECK(noalloc_layout(nullptr, kNoAllocMaxFaces, probe) <= kNoAllocBytes,
               "pamo_point_mesh_sqdist_noalloc: the scratch array is smaller than its layout");
    noalloc_layout(static_cast<unsigned char*>(ptr), kNoAllocMaxFaces, d.w);
    d.base = static_cast<unsigned char*>(ptr);
    return 0;
}

}  // namespace metrics
}  // namespace pamo

using MCtx = pamo::metrics::Ctx;

extern "C" {

int pamo_metrics_create(pamo_metrics** out, int device) {
    pamo::clear_error();
    PAMO_CHECK(out != nullptr, "pamo_metrics_create: null argument");
    MCtx* c = new MCtx();
    c->device = device;
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc((void**)&c->w.flags, 3 * sizeof(int));
    if (e == hipSuccess) e = hipMalloc((void**)&c->mx, sizeof(unsigned long long));
    if (e == hipSuccess) e = hipHostMalloc((void**)&c->w.h_flags, 2 * sizeof(int), 0);
    if (e == hipSuccess) e = hipHostMalloc((void**)&c->h_mx, sizeof(unsigned long long), 0);
    if (e != hipSuccess) {
        pamo::set_error(std::string("pamo_metrics_create: ") + hipGetErrorString(e));
        pamo::metrics::ctx_free(*c);
        delete c;
        return 1;
    }
    *out = reinterpret_cast<pamo_metrics*>(c);
    return 0;
}

int pamo_metrics_destroy(pamo_metrics* m) {
    pamo::clear_error();
    if (!m) return 0;
    MCtx* c = reinterpret_cast<MCtx*>(m);
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    pamo::metrics::ctx_free(*c);
    delete c;
    return 0;
}

int pamo_point_mesh_sqdist(pamo_metrics* m, const double* P, long long n_points, const double* V, int n_v,
                           const int* F, int n_f, double* sqr_d, int* face_index, double* closest) {
    pamo::clear_error();
    PAMO_CHECK(m != nullptr, "pamo_point_mesh_sqdist: null context");
    PAMO_CHECK(n_points >= 0 && (n_points == 0 || (P && sqr_d)), "pamo_point_mesh_sqdist: null argument");
    MCtx& c = *reinterpret_cast<MCtx*>(m);
    PAMO_HIP(hipSetDevice(c.device));
    PAMO_CHECK(V && F && n_v > 0 && n_f > 0, "pamo_point_mesh_sqdist: empty or null mesh");
    PAMO_TRY(pamo::metrics::reserve(c, n_f, n_points));
    PAMO_TRY(pamo::metrics::begin(c.w, c.stream));
    PAMO_TRY(pamo::metrics::build_tree(c.w, c.stream, V, n_v, F, n_f, "pamo_point_mesh_sqdist"));
    PAMO_TRY(pamo::metrics::query(c.w, c.stream, P, n_points, V, F, sqr_d, face_index, closest));
    return pamo::metrics::finish(c.w, c.stream, "pamo_point_mesh_sqdist");
}

int pamo_hausdorff(pamo_metrics* m, const double* VA, int n_va, const int* FA, int n_fa, const double* VB, int n_vb,
                   const int* FB, int n_fb, double* d_out) {
    pamo::clear_error();
    PAMO_CHECK(m != nullptr && d_out != nullptr, "pamo_hausdorff: null argument");
    MCtx& c = *reinterpret_cast<MCtx*>(m);
    PAMO_HIP(hipSetDevice(c.device));
    PAMO_HIP(hipMemsetAsync(c.mx, 0, sizeof(unsigned long long), c.stream));
    PAMO_TRY(pamo::metrics::begin(c.w, c.stream));
    // vertices of B against the surface of A, then vertices of A against B
    PAMO_TRY(pamo::metrics::one_side(c, VB, n_vb, VA, n_va, FA, n_fa));
    PAMO_TRY(pamo::metrics::one_side(c, VA, n_va, VB, n_vb, FB, n_fb));
    PAMO_HIP(hipMemcpyAsync(c.h_mx, c.mx, sizeof(unsigned long long), hipMemcpyDeviceToHost, c.stream));
    PAMO_TRY(pamo::metrics::finish(c.w, c.stream, "pamo_hausdorff"));
    double d2;
    std::memcpy(&d2, c.h_mx, sizeof(double));
    *d_out = std::sqrt(d2);
    return 0;
}

int pamo_point_mesh_sqdist_noalloc(const double* P, long long n_points, const double* V, int n_v, const int* F,
                                   int n_f, double* sqr_d, int* face_index, double* closest, void* stream_handle) {
    using namespace pamo::metrics;
    hipStream_t stream = static_cast<hipStream_t>(stream_handle);
    pamo::clear_error();
    PAMO_CHECK(n_points >= 0 && (n_points == 0 || (P && sqr_d)), "pamo_point_mesh_sqdist_noalloc: null argument");
    PAMO_CHECK(V && F && n_v > 0 && n_f > 0, "pamo_point_mesh_sqdist_noalloc: empty or null mesh");
    PAMO_CHECK(n_f <= kNoAllocMaxFaces, "pamo_point_mesh_sqdist_noalloc: " + std::to_string(n_f) +
                                           " faces, more than the " + std::to_string(kNoAllocMaxFaces) +
                                           " its static scratch holds (use pamo_point_mesh_sqdist)");
    int device = 0;
    PAMO_HIP(hipGetDevice(&device));
    if (stream) {
        hipDevice_t sdev = 0;
        PAMO_HIP(hipStreamGetDevice(stream, &sdev));
        PAMO_CHECK((int)sdev == device, "pamo_point_mesh_sqdist_noalloc: the stream belongs to another device");
    }
    // the setup and the call hold the device's lock: calls on one device
    // share its scratch and run one at a time, each finishing before the next
    NoAllocDevice* d = nullptr;
    std::unique_lock<std::mutex> lock(g_noalloc[std::max(0, std::min(device, kNoAllocMaxDevices - 1))].mu);
    PAMO_TRY(noalloc_setup(device, d));
    // the flags come back to this call's own host words
    int h_flags[2] = {0, 0};
    Work w = d->w;
    w.h_flags = h_flags;
    PAMO_TRY(begin(w, stream));
    PAMO_TRY(build_tree(w, stream, V, n_v, F, n_f, "pamo_point_mesh_sqdist_noalloc"));
    PAMO_TRY(query(w, stream, P, n_points, V, F, sqr_d, face_index, closest));
    return finish(w, stream, "pamo_point_mesh_sqdist_noalloc");
}

}  // extern "C"
