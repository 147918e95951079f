// Stage-1 remeshing on gfx950: the input triangles become the iso-surface
// of an offset distance field, as PaMO.remesh does (simp_cuda/pamo/
// __init__.py:60-120: normalise the triangles into the unit cube, a
// narrow-band distance field on an R^3 grid, the level 0.9 / R, dual
// marching cubes and quads split into triangles).  The reference takes the
// field from torchcumesh2sdf.get_sdf and the extraction from pdmc.DMC,
// neither of which ships with it; the field, its sign and the extraction
// here are restated from their published methods:
//   - unsigned distance to the triangles (closest point on a triangle,
//     Ericson, Real-Time Collision Detection 5.1.5) at every grid sample
//     within the band, by rasterising each triangle column by column along
//     its dominant normal axis;
//   - sign by a flood fill from the grid border through samples farther
//     than half a cell from the surface (a 6-connected path that crosses
//     the surface passes a sample within half a cell of it), so enclosed
//     regions are inside and open sheets get a closed shell;
//   - marching cubes with one face rule for all 256 corner-sign cases (on a
//     face with alternating corner signs the inside corners are cut off
//     separately): the surface patches of a cell are the cycles of its
//     crossing edges joined face by face, each polygon is fanned into
//     triangles, and the vertices are the crossings on the grid edges,
//     shared by the cells around an edge.  Two cells sharing a face always
//     cut it the same way, so the surface is closed and manifold; the
//     reference's dual extraction (one vertex per patch, quads split by an
//     angle rule) is not manifold where the patches of both cells cross the
//     shared face twice, and is not used.
// Grid sample k of an axis sits at (k + 0.5) / R of the normalised cube.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "hip_common.h"
#include "pamo_hip.h"
#include "prim.h"
#include "stage3_math.h"

namespace pamo {
namespace s1 {
namespace {

using s3::V3;
using s3::mk;
using s3::v3;

constexpr int kB = 256;

// ------------------------------------------------------------ dual marching cubes case table
// Cube corner c = x + 2 y + 4 z; edges 0-3 along x, 4-7 along y, 8-11 along z.
constexpr int kEdgeCorner[12][2] = {{0, 1}, {2, 3}, {4, 5}, {6, 7}, {0, 2}, {1, 3},
                                    {4, 6}, {5, 7}, {0, 4}, {1, 5}, {2, 6}, {3, 7}};
// The six faces, corners in cyclic order.
constexpr int kFaceCorner[6][4] = {{0, 2, 6, 4}, {1, 3, 7, 5}, {0, 1, 5, 4},
                                   {2, 3, 7, 6}, {0, 1, 3, 2}, {4, 5, 7, 6}};

struct CaseTable {
    int8_t cyc[256][12];  // the crossing edges, patch after patch, each patch in cycle order
    int8_t plen[256][4];  // edges of each patch
    int8_t npatch[256];
    int8_t ntri[256];     // fan triangles: sum over the patches of (edges - 2)
};

static int edge_of(int a, int b) {
    for (int e = 0; e < 12; ++e)
        if ((kEdgeCorner[e][0] == a && kEdgeCorner[e][1] == b) || (kEdgeCorner[e][0] == b && kEdgeCorner[e][1] == a))
            return e;
    return -1;
}

// Outward normal of face f (x = 0, x = 1, y = 0, y = 1, z = 0, z = 1).
constexpr int kFaceNormal[6][3] = {{-1, 0, 0}, {1, 0, 0}, {0, -1, 0}, {0, 1, 0}, {0, 0, -1}, {0, 0, 1}};

struct Seg {
    int a, b, face;
    double in[3];  // the inside corner(s) the segment cuts off on its face (centroid)
};

// Bit c of `cs` set: corner c is inside (below the level).  The patches are
// the components of the crossing edges linked by the face segments; each is
// ordered so that, seen from outside the cube across every face it crosses,
// the inside corners lie to the right of its segments, which makes the
// fan triangles' normals point from inside to outside.
static bool build_case(int cs, CaseTable& t) {
    auto in = [&](int c) { return (cs >> c) & 1; };
    auto cpos = [](int c, double p[3]) {
        p[0] = c & 1;
        p[1] = (c >> 1) & 1;
        p[2] = c >> 2;
    };
    std::vector<Seg> segs;
    for (int f = 0; f < 6; ++f) {
        const int* q = kFaceCorner[f];
        int fe[4];
        bool cross[4];
        int ncross = 0;
        for (int i = 0; i < 4; ++i) {
            fe[i] = edge_of(q[i], q[(i + 1) & 3]);
            cross[i] = in(q[i]) != in(q[(i + 1) & 3]);
            ncross += cross[i] ? 1 : 0;
        }
        if (ncross == 2) {
            Seg s{-1, -1, f, {0, 0, 0}};
            for (int i = 0; i < 4; ++i)
                if (cross[i]) (s.a < 0 ? s.a : s.b) = fe[i];
            int nin = 0;
            for (int i = 0; i < 4; ++i)
                if (in(q[i])) {
                    double p[3];
                    cpos(q[i], p);
                    for (int d = 0; d < 3; ++d) s.in[d] += p[d];
                    ++nin;
                }
            for (int d = 0; d < 3; ++d) s.in[d] /= nin;
            segs.push_back(s);
        } else if (ncross == 4) {
            // alternating signs: cut each inside corner off on its own
            for (int i = 0; i < 4; ++i)
                if (in(q[i])) {
                    Seg s{fe[(i + 3) & 3], fe[i], f, {0, 0, 0}};
                    cpos(q[i], s.in);
                    segs.push_back(s);
                }
        }
    }
    // each crossing edge lies on two faces: two segments
    std::vector<std::vector<int>> at(12);
    for (int k = 0; k < (int)segs.size(); ++k) {
        at[segs[k].a].push_back(k);
        at[segs[k].b].push_back(k);
    }
    auto mid = [&](int e, double p[3]) {
        double a[3], b[3];
        cpos(kEdgeCorner[e][0], a);
        cpos(kEdgeCorner[e][1], b);
        for (int d = 0; d < 3; ++d) p[d] = 0.5 * (a[d] + b[d]);
    };
    // does going from edge u to edge v along segment k keep the inside on the right?
    auto forward = [&](int k, int u, int v) {
        double a[3], b[3];
        mid(u, a);
        mid(v, b);
        const int* n = kFaceNormal[segs[k].face];
        const double d[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
        const double c[3] = {d[1] * n[2] - d[2] * n[1], d[2] * n[0] - d[0] * n[2], d[0] * n[1] - d[1] * n[0]};
        double w = 0;
        for (int j = 0; j < 3; ++j) w += c[j] * (segs[k].in[j] - 0.5 * (a[j] + b[j]));
        return w > 0;
    };
    bool used[12] = {false};
    int pos = 0, np = 0, ntri = 0;
    for (int e = 0; e < 12; ++e) {
        const bool crossing = in(kEdgeCorner[e][0]) != in(kEdgeCorner[e][1]);
        if (!crossing || used[e]) continue;
        if (at[e].size() != 2) return false;
        // the direction out of e that keeps the inside on the right
        int k0 = at[e][0];
        int nxt = segs[k0].a == e ? segs[k0].b : segs[k0].a;
        if (!forward(k0, e, nxt)) {
            k0 = at[e][1];
            nxt = segs[k0].a == e ? segs[k0].b : segs[k0].a;
            if (!forward(k0, e, nxt)) return false;
        }
        int len = 0, cur = e, k = k0;
        for (;;) {
            t.cyc[cs][pos + len++] = (int8_t)cur;
            used[cur] = true;
            const int n2 = segs[k].a == cur ? segs[k].b : segs[k].a;
            if (!forward(k, cur, n2)) return false;
            if (n2 == e) break;
            if (used[n2] || at[n2].size() != 2) return false;
            k = at[n2][0] == k ? at[n2][1] : at[n2][0];
            cur = n2;
        }
        if (np >= 4 || len < 3) return false;
        t.plen[cs][np++] = (int8_t)len;
        pos += len;
        ntri += len - 2;
    }
    for (int j = pos; j < 12; ++j) t.cyc[cs][j] = -1;
    for (int j = np; j < 4; ++j) t.plen[cs][j] = 0;
    t.npatch[cs] = (int8_t)np;
    t.ntri[cs] = (int8_t)ntri;
    return true;
}

static const CaseTable* case_table() {
    static CaseTable t;
    static const bool ok = [] {
        for (int cs = 0; cs < 256; ++cs)
            if (!build_case(cs, t)) return false;
        return true;
    }();
    return ok ? &t : nullptr;
}

// ------------------------------------------------------------ normalisation
// preprocess_mesh (pamo/__init__.py:60-72) on the device, in the order of
// the reference's float32 numpy expressions: t1 = p - mean; the per-axis
// minimum of t1 over the corners; the maximum of t1 - min over all; then
// ((t1 - min) / max + band) / margin.
__device__ __forceinline__ unsigned f2ord(float f) {
    const unsigned u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Few blocks, each over a strided share, and one set of six atomics a block:
// with a set a corner the launch waited on six words (1.11M corners: 1.18 ms;
// now 20 us).  (Minima and maxima of the ordered words: the order of the
// visits does not matter.)
constexpr unsigned kBoundsBlocks = 512;
__global__ void __launch_bounds__(kB) bounds_k(const float* __restrict__ p, const int* __restrict__ f, long long n3,
                                               float mx, float my, float mz, unsigned* __restrict__ out6) {
    __shared__ unsigned red[kB / kWave][6];
    unsigned lo[3] = {~0u, ~0u, ~0u}, hi[3] = {0u, 0u, 0u};
    for (long long i = (long long)blockIdx.x * kB + threadIdx.x; i < n3; i += (long long)gridDim.x * kB) {
        const int v = f[i];
        const float t[3] = {p[3 * (long long)v] - mx, p[3 * (long long)v + 1] - my, p[3 * (long long)v + 2] - mz};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const unsigned o = f2ord(t[d]);
            lo[d] = min(lo[d], o);
            hi[d] = max(hi[d], o);
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int m = kWave / 2; m > 0; m >>= 1) {
            lo[d] = min(lo[d], (unsigned)__shfl_xor((int)lo[d], m));
            hi[d] = max(hi[d], (unsigned)__shfl_xor((int)hi[d], m));
        }
    if ((threadIdx.x & (kWave - 1)) == 0)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            red[threadIdx.x / kWave][d] = lo[d];
            red[threadIdx.x / kWave][3 + d] = hi[d];
        }
    __syncthreads();
    if (threadIdx.x < 6) {
        unsigned r = red[0][threadIdx.x];
        for (int w = 1; w < kB / kWave; ++w)
            r = threadIdx.x < 3 ? min(r, red[w][threadIdx.x]) : max(r, red[w][threadIdx.x]);
        if (threadIdx.x < 3) atomicMin(&out6[threadIdx.x], r);
        else atomicMax(&out6[threadIdx.x], r);
    }
}

__global__ void __launch_bounds__(kB) normalize_k(const float* __restrict__ p, const int* __restrict__ f, long long n3,
                                                  float mx, float my, float mz, float lx, float ly, float lz,
                                                  float tmax, float band, float margin, float4* __restrict__ tri) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    const int v = f[i];
    const float t0 = p[3 * (long long)v] - mx, t1 = p[3 * (long long)v + 1] - my, t2 = p[3 * (long long)v + 2] - mz;
    tri[i] = make_float4(((t0 - lx) / tmax + band) / margin, ((t1 - ly) / tmax + band) / margin,
                         ((t2 - lz) / tmax + band) / margin, 0.0f);
}

// ------------------------------------------------------------ unsigned distance in the band
struct Raster {
    int axis;        // dominant normal axis (the column direction)
    int lo[3], hi[3];  // sample index box of the triangle grown by the band
};

__device__ __forceinline__ float comp(V3 a, int d) { return d == 0 ? a.x : (d == 1 ? a.y : a.z); }

__device__ __forceinline__ Raster raster_of(V3 a, V3 b, V3 c, int R, float band) {
    Raster r;
    const V3 n = s3::cross(b - a, c - a);
    const float ax = fabsf(n.x), ay = fabsf(n.y), az = fabsf(n.z);
    r.axis = (ax >= ay && ax >= az) ? 0 : (ay >= az ? 1 : 2);
    for (int d = 0; d < 3; ++d) {
        const float mn = fminf(comp(a, d), fminf(comp(b, d), comp(c, d))) - band;
        const float mxv = fmaxf(comp(a, d), fmaxf(comp(b, d), comp(c, d))) + band;
        r.lo[d] = max(0, (int)ceilf(mn * (float)R - 0.5f));
        r.hi[d] = min(R - 1, (int)floorf(mxv * (float)R - 0.5f));
    }
    return r;
}

__device__ __forceinline__ V3 tri_corner(const float4* __restrict__ tri, long long f, int k) {
    return v3(tri[3 * f + k]);
}

// A column is a sample line along the dominant axis; a row holds the columns of
// one index of the second other axis, and is worked on in segments of at most
// 2^seg_log columns.
__device__ __forceinline__ int row_segments(const Raster& r, int seg_log) {
    const int d1 = r.axis == 0 ? 1 : 0;
    return ((r.hi[d1] - r.lo[d1]) >> seg_log) + 1;
}

// Segments of each triangle's box.
__global__ void __launch_bounds__(kB) columns_k(const float4* __restrict__ tri, int nF, int R, float band, int seg_log,
                                                long long* __restrict__ segs) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f > nF) return;
    if (f == nF) {
        segs[nF] = 0;
        return;
    }
    const Raster r = raster_of(tri_corner(tri, f, 0), tri_corner(tri, f, 1), tri_corner(tri, f, 2), R, band);
    const int d2 = r.axis == 2 ? 1 : 2;
    bool any = true;
    for (int d = 0; d < 3; ++d) any = any && r.hi[d] >= r.lo[d];
    segs[f] = any ? (long long)(r.hi[d2] - r.lo[d2] + 1) * row_segments(r, seg_log) : 0;
}

// Exclusive scan of 64-bit column counts in one workgroup per 2048 items
// and a host-side add of the tile sums (the counts are read once per
// remesh, not per round).
__global__ void __launch_bounds__(kB) scan64_tiles_k(long long* __restrict__ v, long long n,
                                                     long long* __restrict__ sums) {
    __shared__ long long lds[kB];
    const long long base = (long long)blockIdx.x * 2048 + (long long)threadIdx.x * 8;
    long long x[8], s = 0;
    for (int i = 0; i < 8; ++i) {
        x[i] = base + i < n ? v[base + i] : 0;
        s += x[i];
    }
    lds[threadIdx.x] = s;
    __syncthreads();
    for (int d = 1; d < kB; d <<= 1) {
        const long long y = threadIdx.x >= (unsigned)d ? lds[threadIdx.x - d] : 0;
        __syncthreads();
        lds[threadIdx.x] += y;
        __syncthreads();
    }
    long long ex = lds[threadIdx.x] - s;
    for (int i = 0; i < 8; ++i) {
        if (base + i < n) v[base + i] = ex;
        ex += x[i];
    }
    if (threadIdx.x == kB - 1) sums[blockIdx.x] = lds[kB - 1];
}

__global__ void __launch_bounds__(kB) scan64_add_k(long long* __restrict__ v, long long n,
                                                   const long long* __restrict__ offs) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] += offs[i / 2048];
}

// One work item per segment of a row: the samples of each column within the
// band of the triangle's plane, each given min(current, distance) (the distance's
// bits order like the non-negative floats they encode).
// A block finds its first and last item's triangles in `off` and the items
// between search the offsets between, brought to LDS (in `off` where there are
// more than kUdfRange, as triangles without items can make it).  Bound by its
// instructions: a column an item, each with its own search, box, plane and
// region setup, took 1.16 ms on 370k faces at R = 256, a row an item 0.88.
//
// Segments: small triangles' rows have some ten columns, and a dense mesh has
// items enough, so a row is one item (16 columns hold it); the rows of a few
// large triangles have up to R columns and are too few for the chip.  Remeshing
// in ms (with four words of crossings a lane, see CrossVertsOp) with 2 | 4 | 8 |
// 16 columns | whole rows: a cube (12 faces) at R = 64
// .32 | .34 | .35 | .39 | .64, at R = 256 .92 | .93 | .95 | .98 | 2.28; a sphere
// of 5120 faces at R = 256 .78 | .81 | .83 | .87 | .87; a union of 19k faces at
// R = 64 .37 | .35 | .36 | .36 | .36, of 366k faces at R = 256 2.00 | 1.81 |
// 1.75 | 1.74 | 1.75.
constexpr int kUdfRange = 512;
constexpr int kFewFaces = 16384;
static int segment_log(int n_tris) { return n_tris <= kFewFaces ? 1 : 4; }

__device__ __forceinline__ int udf_find(const long long* __restrict__ off, int lo, int hi, long long w) {
    while (lo < hi) {  // the last triangle whose items start at or before w
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= w) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__global__ void __launch_bounds__(kB) udf_k(const float4* __restrict__ tri, int nF, const long long* __restrict__ off,
                                            long long total, int R, float band, int seg_log,
                                            unsigned* __restrict__ grid) {
    __shared__ long long loff[kUdfRange];
    __shared__ int ends[2];
    const long long w0 = (long long)blockIdx.x * kB, w = w0 + threadIdx.x;
    if (threadIdx.x < 2) ends[threadIdx.x] = udf_find(off, 0, nF - 1, threadIdx.x ? min(w0 + kB, total) - 1 : w0);
    __syncthreads();
    const int f0 = ends[0], nr = ends[1] - f0 + 1;
    const bool in_lds = nr <= kUdfRange;
    if (in_lds)
        for (int k = threadIdx.x; k < nr; k += kB) loff[k] = off[f0 + k];
    __syncthreads();
    if (w >= total) return;
    const int f = in_lds ? f0 + udf_find(loff, 0, nr - 1, w) : udf_find(off, f0, ends[1], w);
    const V3 a = tri_corner(tri, f, 0), b = tri_corner(tri, f, 1), c = tri_corner(tri, f, 2);
    const Raster r = raster_of(a, b, c, R, band);
    const int ax = r.axis, d1 = ax == 0 ? 1 : 0, d2 = ax == 2 ? 1 : 2;
    const int ns = row_segments(r, seg_log), k = (int)(w - off[f]), i2 = r.lo[d2] + k / ns;
    const int s0 = r.lo[d1] + ((k % ns) << seg_log), s1 = min(r.hi[d1], s0 + (1 << seg_log) - 1);
    const float inv = 1.0f / (float)R, x2 = ((float)i2 + 0.5f) * inv;
    // the triangle lies in the ball (mid, rad): a sample farther from mid than
    // rad plus the distance that its cell already holds (or the band) cannot
    // change the cell.  (slack: the coordinates are below 2, so the distances'
    // rounding errors are below 1e-6)
    const V3 mid = mk((a.x + b.x + c.x) / 3.0f, (a.y + b.y + c.y) / 3.0f, (a.z + b.z + c.z) / 3.0f);
    const float slack = 4e-6f;
    const float rad = fmaxf(s3::len(a - mid), fmaxf(s3::len(b - mid), s3::len(c - mid))) + slack;
    const float e2 = x2 - comp(mid, d2), reach = band + rad, row2 = reach * reach - e2 * e2;
    if (row2 < 0.0f) return;
    const float half1 = sqrtf(row2) + slack, m1 = comp(mid, d1);
    const int c0 = max(s0, (int)ceilf((m1 - half1) * (float)R - 0.5f));
    const int c1 = min(s1, (int)floorf((m1 + half1) * (float)R - 0.5f));
    const V3 n = s3::cross(b - a, c - a);
    const float na = comp(n, ax), nl = s3::len(n);
    const bool plane = fabsf(na) > 1e-30f && nl > 0.0f;
    const float half = plane ? band * nl / fabsf(na) * 1.0001f + 1e-6f : 0.0f;
    const long long stride = ax == 0 ? 1 : (ax == 1 ? R : (long long)R * R);
    for (int i1 = c0; i1 <= c1; ++i1) {
        const float x1 = ((float)i1 + 0.5f) * inv;
        int k0 = r.lo[ax], k1 = r.hi[ax];
        if (plane) {  // the samples of this column within `band` of the plane
            const float ap =
                comp(a, ax) - (comp(n, d1) * (x1 - comp(a, d1)) + comp(n, d2) * (x2 - comp(a, d2))) / na;
            k0 = max(k0, (int)ceilf((ap - half) * (float)R - 0.5f));
            k1 = min(k1, (int)floorf((ap + half) * (float)R - 0.5f));
        }
        const float e1 = x1 - m1, side2 = e1 * e1 + e2 * e2;
        const long long base = ax == 0 ? ((long long)i2 * R + i1) * R
                             : ax == 1 ? (long long)i2 * R * R + i1
                                       : (long long)i2 * R + i1;
        for (int kb = k0; kb <= k1; kb += 4) {
            // four cells are read before any of them is used
            float held[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) held[u] = __uint_as_float(grid[base + stride * min(kb + u, k1)]);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int ka = kb + u;
                if (ka > k1) break;
                const float xa = ((float)ka + 0.5f) * inv;
                const float ea = xa - comp(mid, ax), lim = fminf(held[u], band) + rad;
                if (side2 + ea * ea > lim * lim) continue;
                V3 p;
                if (ax == 0) p = mk(xa, x1, x2);
                else if (ax == 1) p = mk(x1, xa, x2);
                else p = mk(x1, x2, xa);
                const V3 q = s3::closest_on_tri(p, a, b, c);
                const float dist = s3::len(p - q);
                if (!(dist <= band)) continue;
                const unsigned bits = __float_as_uint(dist);
                if (bits < __float_as_uint(held[u])) atomicMin(grid + base + stride * ka, bits);
            }
        }
    }
}

// ------------------------------------------------------------ sign by flood fill
// A sample is passable when it lies farther than `wall` from the surface;
// the outside is the passable region connected (6-neighbours) to the grid
// border.  The fill runs on bits: a brick is 8x8x8 samples, a byte for each
// row along x, row r = 8 z + y of brick b at 64 b + r, so a wave holds a brick
// with a row a lane and fills it with shifts and shuffles.
constexpr int kBrick = 8;

// Passable samples, and the passable ones on the grid's border (outside).
__global__ void __launch_bounds__(kB) fill_init_k(const unsigned* __restrict__ grid, int R, int nb, unsigned wall_bits,
                                                  uint8_t* __restrict__ pass, uint8_t* __restrict__ rows) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long b = t >> 6;
    if (b >= (long long)nb * nb * nb) return;
    const int r = (int)(t & 63);
    const int x0 = (int)(b % nb) * kBrick, y = (int)((b / nb) % nb) * kBrick + (r & 7),
              z = (int)(b / ((long long)nb * nb)) * kBrick + (r >> 3);
    unsigned p = 0, o = 0;
    if (y < R && z < R) {
        const unsigned* g = grid + ((long long)z * R + y) * R;
        const bool side = y == 0 || z == 0 || y == R - 1 || z == R - 1;
#pragma unroll
        for (int j = 0; j < kBrick; ++j) {
            const int x = x0 + j;
            if (x < R && g[x] > wall_bits) {
                p |= 1u << j;
                if (side || x == 0 || x == R - 1) o |= 1u << j;
            }
        }
    }
    pass[t] = (uint8_t)p;
    rows[t] = (uint8_t)o;
}

// One wave a brick: the outside bits of its six neighbours seed it, and it
// fills until it stops changing.  A launch works on the bricks that a
// neighbour's growth can have changed: a brick is at its fixed point after its
// turn, and one that grew marks its neighbours for the next launch (round + 1
// in `due`) and the launch in *changed.  A neighbour of the same launch may
// mark the brick before it reads its own mark: marks only go up, and the brick
// then takes its turn in the next launch, with all the growth up to then.
// (R = 256, 32,768 bricks: a workgroup a brick, a byte a sample in LDS and a
// barrier a step, took 96 us a launch, about 11 launches; now 7.6 us, 20 launches.)
__global__ void __launch_bounds__(kB) fill_brick_k(int nb, const uint8_t* __restrict__ pass, uint8_t* rows, int* due,
                                                   int round, int* __restrict__ changed) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long b = t >> 6;  // uniform per wave
    if (b >= (long long)nb * nb * nb) return;
    if (round > 1 && due[b] != round) return;
    const int r = (int)(t & 63), y = r & 7, z = r >> 3;
    const int bx = (int)(b % nb), by = (int)((b / nb) % nb), bz = (int)(b / ((long long)nb * nb));
    const long long sy = nb, sz = (long long)nb * nb;
    const unsigned p = pass[t], start = rows[t];
    unsigned o = start;
    if (bx > 0) o |= p & (unsigned)(rows[64 * (b - 1) + r] >> 7);
    if (bx + 1 < nb) o |= p & ((unsigned)(rows[64 * (b + 1) + r] & 1) << 7);
    if (y == 0 && by > 0) o |= p & rows[64 * (b - sy) + r + 7];
    if (y == 7 && by + 1 < nb) o |= p & rows[64 * (b + sy) + r - 7];
    if (z == 0 && bz > 0) o |= p & rows[64 * (b - sz) + r + 56];
    if (z == 7 && bz + 1 < nb) o |= p & rows[64 * (b + sz) + r - 56];
    for (int it = 0; it < kBrick * kBrick * kBrick; ++it) {
        const unsigned ym = __shfl_up(o, 1), yp = __shfl_down(o, 1), zm = __shfl_up(o, 8), zp = __shfl_down(o, 8);
        unsigned n = o | (o << 1) | (o >> 1) | (y > 0 ? ym : 0) | (y < 7 ? yp : 0) | (z > 0 ? zm : 0) | (z < 7 ? zp : 0);
        n &= p;
        const bool grew = n != o;
        o = n;
        if (!__ballot(grew)) break;
    }
    if (!__ballot(o != start)) return;
    rows[t] = (uint8_t)o;
    if (r < 6) {
        const int d = r >> 1, dir = (r & 1) ? 1 : -1;
        const int q[3] = {bx + (d == 0 ? dir : 0), by + (d == 1 ? dir : 0), bz + (d == 2 ? dir : 0)};
        if (q[d] >= 0 && q[d] < nb) due[((long long)q[2] * nb + q[1]) * nb + q[0]] = round + 1;
    }
    if (r == 6) *changed = round;
}

// The outside, a byte a sample.
__global__ void __launch_bounds__(kB) fill_out_k(int R, int nb, const uint8_t* __restrict__ rows,
                                                 uint8_t* __restrict__ out) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)R * R * R) return;
    const int x = (int)(i % R), y = (int)((i / R) % R), z = (int)(i / ((long long)R * R));
    const long long b = ((long long)(z >> 3) * nb + (y >> 3)) * nb + (x >> 3);
    out[i] = (rows[64 * b + 8 * (z & 7) + (y & 7)] >> (x & 7)) & 1;
}

// ------------------------------------------------------------ marching cubes
__device__ __forceinline__ float sdf_at(const unsigned* __restrict__ grid, const uint8_t* __restrict__ out,
                                        long long i) {
    const float u = __uint_as_float(grid[i]);
    return out[i] ? u : -u;
}

// The level's sign structure as bits, 64 samples a word (word k: samples 64 k
// ... 64 k + 63 in x, y, z order): `in` the samples below the level, and for
// each direction d at cross + d * words the grid edges (+x, +y, +z of a
// sample) that cross it, one surface vertex each.  One pass over the field in
// place of a count a grid edge (3 R^3 integers, written, scanned and read
// again: 0.73 ms at R = 256, 0.12 with the vertices now).
__global__ void __launch_bounds__(kB) cross_bits_k(const unsigned* __restrict__ grid, const uint8_t* __restrict__ out,
                                                   int R, float iso, long long words, uint64_t* __restrict__ in,
                                                   uint64_t* __restrict__ cross) {
    const long long n = (long long)R * R * R;
    const long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    bool b = false, c[3] = {false, false, false};
    if (s < n) {
        const int q[3] = {(int)(s % R), (int)((s / R) % R), (int)(s / ((long long)R * R))};
        b = sdf_at(grid, out, s) < iso;
        long long step = 1;
        for (int d = 0; d < 3; ++d) {
            if (q[d] + 1 < R) c[d] = (sdf_at(grid, out, s + step) < iso) != b;
            step *= R;
        }
    }
    const uint64_t mb = __ballot(b), m0 = __ballot(c[0]), m1 = __ballot(c[1]), m2 = __ballot(c[2]);
    const long long w = s >> 6;
    if ((threadIdx.x & (kWave - 1)) == 0 && w < words) {
        in[w] = mb;
        cross[w] = m0;
        cross[words + w] = m1;
        cross[2 * words + w] = m2;
    }
}

// The crossing vertices, direction by direction in sample order: a scan over
// the words' counts; the vertices of a word by linear interpolation, in
// sample index units.  wpos[k] (k <= 3 words): vertices before word k.
// A lane writes its words' few vertices one by one; a word of more than kWide,
// up to 64 where a flat face lies along the grid, is written by its wave, a
// sample a lane, which reads the samples in whole lines.  Remeshing in ms, with
// four words a lane and no wave | two and no wave | four and the wave | two and
// the wave: a cube (12 faces) at R = 64 .32 | .28 | .24 | .24, at R = 128 .41 | .42
// | .43 | .35, at R = 256 .92 | .78 | .80 | .71 (a lane a grid edge: .26, .42 and
// 1.35); a union of 366k faces at R = 256 1.76 | 1.76 | 1.74 | 1.72.
struct CrossVertsOp {
    static constexpr int kIpt = 2, kWide = 12;
    const uint64_t* cross;
    const unsigned* grid;
    const uint8_t* out;
    long long words;
    int R;
    float iso;
    int* wpos;
    float4* verts;
    long long cap;   // room in verts (a first guess; the launch is repeated when it was too small)
    int* total;
    __device__ int count(long long k) const { return __popcll(cross[k]); }
    // the vertex of sample `bit` of word k, at place p of verts
    __device__ void put(long long k, int bit, long long p) const {
        if (p >= cap) return;
        const int dir = (int)(k / words);
        const long long step = dir == 0 ? 1 : (dir == 1 ? R : (long long)R * R);
        const long long s = (k - dir * words) * 64 + bit;
        const float d0 = sdf_at(grid, out, s), d1 = sdf_at(grid, out, s + step);
        const float t = (iso - d0) / (d1 - d0);
        float q[3] = {(float)(s % R), (float)((s / R) % R), (float)(s / ((long long)R * R))};
        q[dir] += t;
        verts[p] = make_float4(q[0], q[1], q[2], 0.0f);
    }
    __device__ void emit(long long k, int v, int pos) const {
        wpos[k] = pos;
        uint64_t m = v ? cross[k] : 0;
        uint64_t wide = __ballot(v > kWide);
        if (wide && __ballot(true) == ~0ull) {  // (the last tile's last wave may hold fewer lanes)
            const int lane = threadIdx.x & (kWave - 1);
            if (v > kWide) m = 0;
            for (; wide; wide &= wide - 1) {
                const int src = __ffsll((unsigned long long)wide) - 1;
                const long long wk = __shfl(k, src);
                const int at = __shfl(pos, src);
                const uint64_t w = cross[wk];
                if ((w >> lane) & 1) put(wk, lane, (long long)at + lanes_below(w));
            }
        }
        for (int j = 0; m; ++j, m &= m - 1) put(k, __ffsll((unsigned long long)m) - 1, (long long)pos + j);
    }
    __device__ void done(int n) const { *total = n; }
};

struct McTable {
    int8_t cyc[256][12];
    int8_t plen[256][4];
    int8_t npatch[256];
    int8_t ntri[256];
};

__device__ __forceinline__ int bit_at(const uint64_t* __restrict__ in, long long s) {
    return (int)((in[s >> 6] >> (s & 63)) & 1);
}

__device__ __forceinline__ int cell_case(const uint64_t* __restrict__ in, int R, int x, int y, int z) {
    int cs = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {  // corner c = x + 2 y + 4 z: a pair along x for each (y, z)
        const long long i = ((long long)(z + (r >> 1)) * R + (y + (r & 1))) * R + x;
        cs |= (bit_at(in, i) | (bit_at(in, i + 1) << 1)) << (2 * r);
    }
    return cs;
}

// Triangles of each group of 64 cells (x, y, z order).
__global__ void __launch_bounds__(kB) cell_count_k(const uint64_t* __restrict__ in, int R,
                                                   const McTable* __restrict__ tab, long long groups,
                                                   int* __restrict__ count) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long m = (long long)(R - 1);
    int c = 0;
    if (i < m * m * m)
        c = tab->ntri[cell_case(in, R, (int)(i % m), (int)((i / m) % m), (int)(i / (m * m)))];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) c += __shfl_xor(c, o);
    const long long g = i >> 6;
    if ((threadIdx.x & (kWave - 1)) == 0 && g <= groups) count[g] = g < groups ? c : 0;
}

// The fan triangles of each patch polygon, vertices by crossing edge; tpos:
// triangles before each group of 64 cells.
__global__ void __launch_bounds__(kB) cell_tris_k(const uint64_t* __restrict__ in, const uint64_t* __restrict__ cross,
                                                  long long words, int R, const McTable* __restrict__ tab,
                                                  const int* __restrict__ tpos, const int* __restrict__ wpos,
                                                  int* __restrict__ tris) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long m = (long long)(R - 1), cells = m * m * m;
    const long long g = i >> 6;  // the wave's group
    if ((g << 6) >= cells || tpos[g + 1] == tpos[g]) return;  // uniform per wave
    const int x = (int)(i % m), y = (int)((i / m) % m), z = (int)(i / (m * m));
    const int cs = i < cells ? cell_case(in, R, x, y, z) : 0;
    const int mine = i < cells ? tab->ntri[cs] : 0;
    int before = mine;  // inclusive scan over the wave
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int up = __shfl_up(before, d);
        if ((threadIdx.x & (kWave - 1)) >= d) before += up;
    }
    if (mine == 0) return;
    auto vid = [&](int e) {
        const int c0 = kEdgeCorner[e][0];
        const long long s = ((long long)(z + (c0 >> 2)) * R + (y + ((c0 >> 1) & 1))) * R + (x + (c0 & 1));
        const long long w = (long long)(e >> 2) * words + (s >> 6);
        return wpos[w] + (int)__popcll(cross[w] & ((1ull << (s & 63)) - 1));
    };
    int* o = tris + 3LL * (tpos[g] + before - mine);
    int base = 0;
    for (int p = 0; p < tab->npatch[cs]; ++p) {
        const int len = tab->plen[cs][p];
        const int v0 = vid(tab->cyc[cs][base]);
        for (int j = 1; j + 1 < len; ++j) {
            o[0] = v0;
            o[1] = vid(tab->cyc[cs][base + j]);
            o[2] = vid(tab->cyc[cs][base + j + 1]);
            o += 3;
        }
        base += len;
    }
}

// Sample index units to the centred frame: ((i + 0.5) / R * margin - band)
// * tmax + min (the inverse of the normalisation).
__global__ void __launch_bounds__(kB) to_frame_k(const float4* __restrict__ v, int n, int R, float band, float margin,
                                                 float tmax, float lx, float ly, float lz, float* __restrict__ outp) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 q = v[i];
    const float inv = 1.0f / (float)R;
    outp[3 * (long long)i] = ((q.x + 0.5f) * inv * margin - band) * tmax + lx;
    outp[3 * (long long)i + 1] = ((q.y + 0.5f) * inv * margin - band) * tmax + ly;
    outp[3 * (long long)i + 2] = ((q.z + 0.5f) * inv * margin - band) * tmax + lz;
}

template <typename T>
__global__ void fill_val_k(T* p, T v, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ------------------------------------------------------------ context
struct Ctx {
    hipStream_t stream = nullptr;
    int device = 0;
    int R = 0;
    float band = 0, margin = 0, iso = 0;
    float mean[3] = {0, 0, 0}, lo[3] = {0, 0, 0}, tmax = 0;
    int n_in = 0, n_verts = 0, n_faces = 0, fill_iters = 0;
    float4* tri = nullptr;
    size_t cap_tri = 0;
    long long* cols = nullptr;
    size_t cap_cols = 0;
    long long* sums = nullptr;
    size_t cap_sums = 0;
    unsigned* grid = nullptr;
    uint8_t* outside = nullptr;
    size_t cap_grid = 0;
    int* cnt = nullptr;       // triangles before each group of 64 cells (+1)
    size_t cap_cnt = 0;
    int* wpos = nullptr;      // vertices before each word of crossing edges
    size_t cap_wpos = 0;
    uint64_t* bits = nullptr;  // samples below the level, then the crossing edges of x, y and z
    size_t cap_bits = 0;
    int* due = nullptr;       // flood fill: the round each brick is due in
    size_t cap_due = 0;
    uint8_t* rows = nullptr;  // flood fill: outside bits, then passable bits, a byte a row of a brick
    size_t cap_rows = 0;
    float4* verts = nullptr;
    size_t cap_verts = 0;
    int* tris = nullptr;
    size_t cap_tris = 0;
    unsigned* b6 = nullptr;
    int* flag = nullptr;
    size_t cap_out = 0;
    int* err = nullptr;    // look-back scan error bits
    LookbackScan lb;
    McTable* tab = nullptr;
    int* h_int = nullptr;  // pinned host words
};

template <typename T>
static int ensure(T** p, size_t& cap, size_t n, hipStream_t st) {
    if (n <= cap) return 0;
    if (*p) PAMO_HIP(hipFree(*p));
    *p = nullptr;
    const size_t a = n + n / 8 + 64;
    PAMO_HIP(hipMalloc((void**)p, sizeof(T) * a));
    cap = a;
    (void)st;
    return 0;
}

static void ctx_free(Ctx& c) {
    void* ptrs[] = {c.tri, c.cols, c.sums, c.grid, c.outside, c.cnt, c.wpos, c.bits, c.due, c.rows, c.verts, c.tris, c.b6, c.flag, c.err,
                    c.tab};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    lookback_free(c.lb);
    if (c.h_int) (void)hipHostFree(c.h_int);
}

static int read_int(Ctx& c, const int* d, int& v) {
    PAMO_HIP(hipMemcpyAsync(c.h_int, d, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    PAMO_HIP(hipStreamSynchronize(c.stream));
    v = c.h_int[0];
    return 0;
}

static int scan_int(Ctx& c, int* v, long long n) {
    PAMO_TRY(lookback_reserve(c.lb, n, c.err, c.stream));
    return scan_exclusive_lb(v, v, n, c.lb, c.stream);
}

// `mean`: the centring offset of PaMO.run (numpy's float32
// tris.mean(axis=1).mean(axis=0), pamo_centroid).
static int remesh(Ctx& c, const float* d_pts, const int* d_tris, int n_tris, const float mean[3], int R) {
    hipStream_t st = c.stream;
    const long long n3 = 3LL * n_tris;
    for (int d = 0; d < 3; ++d) c.mean[d] = mean[d];
    c.n_in = n_tris;
    c.R = R;
    c.band = 3.0f / (float)R;
    c.margin = c.band * 2.0f + 1.0f;
    c.iso = (float)(0.9 / (double)R);
    // per-axis minimum and maximum of t1 = p - mean over the corners
    if (!c.b6) PAMO_HIP(hipMalloc((void**)&c.b6, 6 * sizeof(unsigned)));
    {
        unsigned init[6] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0u, 0u, 0u};
        PAMO_HIP(hipMemcpyAsync(c.b6, init, sizeof(init), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(bounds_k, dim3(std::min(grid_for(n3, kB), kBoundsBlocks)), dim3(kB), 0, st, d_pts, d_tris, n3, c.mean[0], c.mean[1],
                           c.mean[2], c.b6);
        PAMO_HIP(hipGetLastError());
        unsigned h6[6];
        PAMO_HIP(hipMemcpyAsync(h6, c.b6, sizeof(h6), hipMemcpyDeviceToHost, st));
        PAMO_HIP(hipStreamSynchronize(st));
        auto dec = [](unsigned u) {
            const unsigned b = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
            float f;
            std::memcpy(&f, &b, 4);
            return f;
        };
        float mx = -INFINITY;
        for (int d = 0; d < 3; ++d) {
            c.lo[d] = dec(h6[d]);
            // max over the corners of (t1 - min): the subtraction is monotonic
            const float diff = dec(h6[3 + d]) - c.lo[d];
            mx = std::max(mx, diff);
        }
        c.tmax = mx;
    }
    PAMO_CHECK(c.tmax > 0.0f, "pamo_s1_remesh: the triangles span no extent");
    PAMO_TRY(ensure(&c.tri, c.cap_tri, (size_t)n3, st));
    hipLaunchKernelGGL(normalize_k, dim3(grid_for(n3, kB)), dim3(kB), 0, st, d_pts, d_tris, n3, c.mean[0], c.mean[1],
                       c.mean[2], c.lo[0], c.lo[1], c.lo[2], c.tmax, c.band, c.margin, c.tri);
    PAMO_HIP(hipGetLastError());
    // distance field in the band
    const long long ng = (long long)R * R * R;
    PAMO_TRY(ensure(&c.grid, c.cap_grid, (size_t)ng, st));
    PAMO_TRY(ensure(&c.outside, c.cap_out, (size_t)ng, st));
    hipLaunchKernelGGL(fill_val_k<unsigned>, dim3(grid_for(ng, kB)), dim3(kB), 0, st, c.grid, 0x7F800000u, ng);
    PAMO_HIP(hipGetLastError());
    PAMO_TRY(ensure(&c.cols, c.cap_cols, (size_t)n_tris + 1, st));
    const int seg_log = segment_log(n_tris);
    hipLaunchKernelGGL(columns_k, dim3(grid_for(n_tris + 1, kB)), dim3(kB), 0, st, (const float4*)c.tri, n_tris, R,
                       c.band, seg_log, c.cols);
    PAMO_HIP(hipGetLastError());
    const long long nc = n_tris + 1, ntile = (nc + 2047) / 2048;
    PAMO_TRY(ensure(&c.sums, c.cap_sums, (size_t)ntile, st));
    hipLaunchKernelGGL(scan64_tiles_k, dim3((unsigned)ntile), dim3(kB), 0, st, c.cols, nc, c.sums);
    PAMO_HIP(hipGetLastError());
    std::vector<long long> hs(ntile), ho(ntile);
    PAMO_HIP(hipMemcpyAsync(hs.data(), c.sums, sizeof(long long) * ntile, hipMemcpyDeviceToHost, st));
    PAMO_HIP(hipStreamSynchronize(st));
    long long run = 0;
    for (long long t = 0; t < ntile; ++t) {
        ho[t] = run;
        run += hs[t];
    }
    const long long total = run;
    PAMO_HIP(hipMemcpyAsync(c.sums, ho.data(), sizeof(long long) * ntile, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(scan64_add_k, dim3(grid_for(nc, kB)), dim3(kB), 0, st, c.cols, nc, (const long long*)c.sums);
    PAMO_HIP(hipGetLastError());
    if (total > 0)
        hipLaunchKernelGGL(udf_k, dim3(grid_for(total, kB)), dim3(kB), 0, st, (const float4*)c.tri, n_tris,
                           (const long long*)c.cols, total, R, c.band, seg_log, c.grid);
    PAMO_HIP(hipGetLastError());
    // sign: flood fill of the outside from the border
    const float wall = 0.55f / (float)R;
    unsigned wall_bits;
    std::memcpy(&wall_bits, &wall, 4);
    if (!c.flag) PAMO_HIP(hipMalloc((void**)&c.flag, 2 * sizeof(int)));
    const int nb = (R + kBrick - 1) / kBrick;
    const int max_iters = 8 * R + 64;  // the front advances at least one brick per launch
    c.fill_iters = 0;
    const long long nbricks = (long long)nb * nb * nb;
    PAMO_TRY(ensure(&c.due, c.cap_due, (size_t)nbricks, st));
    PAMO_TRY(ensure(&c.rows, c.cap_rows, (size_t)(128 * nbricks), st));
    uint8_t *rows = c.rows, *pass = c.rows + 64 * nbricks;
    hipLaunchKernelGGL(fill_init_k, dim3(grid_for(64 * nbricks, kB)), dim3(kB), 0, st, (const unsigned*)c.grid, R, nb,
                       wall_bits, pass, rows);
    hipLaunchKernelGGL(fill_val_k<int>, dim3(grid_for(nbricks, kB)), dim3(kB), 0, st, c.due, 0, nbricks);
    hipLaunchKernelGGL(fill_val_k<int>, dim3(1), dim3(64), 0, st, c.flag, 0, 2LL);
    PAMO_HIP(hipGetLastError());
    // flag[0]: the last round that grew; the host reads it after every fourth
    // (a round with nothing due is over at once)
    for (;;) {
        PAMO_CHECK(c.fill_iters < max_iters, "pamo_s1_remesh: flood fill did not converge");
        for (int k = 0; k < 4; ++k) {
            ++c.fill_iters;
            hipLaunchKernelGGL(fill_brick_k, dim3(grid_for(64 * nbricks, kB)), dim3(kB), 0, st, nb,
                               (const uint8_t*)pass, rows, c.due, c.fill_iters, c.flag);
        }
        PAMO_HIP(hipGetLastError());
        int last = 0;
        PAMO_TRY(read_int(c, c.flag, last));
        if (last < c.fill_iters) break;
    }
    hipLaunchKernelGGL(fill_out_k, dim3(grid_for(ng, kB)), dim3(kB), 0, st, R, nb, (const uint8_t*)rows, c.outside);
    PAMO_HIP(hipGetLastError());
    // marching cubes at the level iso
    if (!c.tab) {
        const CaseTable* t = case_table();
        PAMO_CHECK(t != nullptr, "pamo_s1_remesh: marching-cubes case table inconsistent");
        PAMO_HIP(hipMalloc((void**)&c.tab, sizeof(McTable)));
        McTable h;
        std::memcpy(h.cyc, t->cyc, sizeof(h.cyc));
        std::memcpy(h.plen, t->plen, sizeof(h.plen));
        std::memcpy(h.npatch, t->npatch, sizeof(h.npatch));
        std::memcpy(h.ntri, t->ntri, sizeof(h.ntri));
        PAMO_HIP(hipMemcpyAsync(c.tab, &h, sizeof(McTable), hipMemcpyHostToDevice, st));
        PAMO_HIP(hipStreamSynchronize(st));
    }
    // vertices: one per crossing grid edge
    const long long words = (ng + 63) / 64;
    PAMO_TRY(ensure(&c.bits, c.cap_bits, (size_t)(4 * words), st));
    PAMO_TRY(ensure(&c.wpos, c.cap_wpos, (size_t)(3 * words), st));
    uint64_t *in = c.bits, *cross = c.bits + words;
    hipLaunchKernelGGL(cross_bits_k, dim3(grid_for(words * 64, kB)), dim3(kB), 0, st, (const unsigned*)c.grid,
                       (const uint8_t*)c.outside, R, c.iso, words, in, cross);
    PAMO_HIP(hipGetLastError());
    // triangles of each group of 64 cells
    const long long m3 = (long long)(R - 1) * (R - 1) * (R - 1), groups = (m3 + 63) / 64;
    PAMO_TRY(ensure(&c.cnt, c.cap_cnt, (size_t)groups + 1, st));
    hipLaunchKernelGGL(cell_count_k, dim3(grid_for((groups + 1) * 64, kB)), dim3(kB), 0, st, (const uint64_t*)in, R,
                       (const McTable*)c.tab, groups, c.cnt);
    PAMO_HIP(hipGetLastError());
    PAMO_TRY(scan_int(c, c.cnt, groups + 1));
    PAMO_TRY(lookback_reserve(c.lb, 3 * words, c.err, st));
    int nv = 0, nt = 0;
    for (;;) {
        PAMO_TRY(scan_op(CrossVertsOp{cross, c.grid, c.outside, words, R, c.iso, c.wpos, c.verts, (long long)c.cap_verts,
                                      c.flag + 1}, 3 * words, c.lb, st));
        PAMO_HIP(hipMemcpyAsync(c.h_int, c.flag + 1, sizeof(int), hipMemcpyDeviceToHost, st));
        PAMO_HIP(hipMemcpyAsync(c.h_int + 1, c.cnt + groups, sizeof(int), hipMemcpyDeviceToHost, st));
        PAMO_HIP(hipStreamSynchronize(st));
        nv = c.h_int[0];
        nt = c.h_int[1];
        if ((size_t)nv <= c.cap_verts) break;
        PAMO_TRY(ensure(&c.verts, c.cap_verts, (size_t)nv, st));  // and once more, into the larger buffer
    }
    PAMO_TRY(ensure(&c.tris, c.cap_tris, (size_t)3 * std::max(nt, 1), st));
    if (nt > 0)
        hipLaunchKernelGGL(cell_tris_k, dim3(grid_for(groups * 64, kB)), dim3(kB), 0, st, (const uint64_t*)in,
                           (const uint64_t*)cross, words, R, (const McTable*)c.tab, (const int*)c.cnt,
                           (const int*)c.wpos, c.tris);
    PAMO_HIP(hipGetLastError());
    PAMO_HIP(hipMemcpyAsync(c.h_int, c.err, sizeof(int), hipMemcpyDeviceToHost, st));
    PAMO_HIP(hipStreamSynchronize(st));
    PAMO_CHECK(c.h_int[0] == 0, "pamo_s1_remesh: a look-back scan wait exceeded its bound");
    c.n_verts = nv;
    c.n_faces = nt;
    return 0;
}

}  // namespace
}  // namespace s1
}  // namespace pamo

// ------------------------------------------------------------ C ABI
struct pamo_s1 {};

extern "C" {

int pamo_s1_create(pamo_s1** out, int device) {
    pamo::clear_error();
    PAMO_CHECK(out != nullptr, "pamo_s1_create: out is null");
    auto* c = new pamo::s1::Ctx();
    c->device = device;
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipHostMalloc((void**)&c->h_int, 4 * sizeof(int), 0);
    if (e == hipSuccess) e = hipMalloc((void**)&c->err, sizeof(int));
    if (e == hipSuccess) e = hipMemsetAsync(c->err, 0, sizeof(int), c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) {
        pamo::set_error(std::string("pamo_s1_create: ") + hipGetErrorString(e));
        pamo::s1::ctx_free(*c);
        if (c->stream) (void)hipStreamDestroy(c->stream);
        delete c;
        return 1;
    }
    *out = reinterpret_cast<pamo_s1*>(c);
    return 0;
}

int pamo_s1_destroy(pamo_s1* s) {
    if (!s) return 0;
    auto* c = reinterpret_cast<pamo::s1::Ctx*>(s);
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    pamo::s1::ctx_free(*c);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return 0;
}

int pamo_s1_remesh(pamo_s1* s, const float* d_points, int n_points, const int* d_faces, int n_faces,
                   const float* mean3, int resolution, int* n_verts_out, int* n_faces_out) {
    pamo::clear_error();
    PAMO_CHECK(s && d_points && d_faces && mean3, "pamo_s1_remesh: null argument");
    PAMO_CHECK(n_points > 0 && n_faces > 0, "pamo_s1_remesh: empty mesh");
    PAMO_CHECK(resolution >= 8 && resolution <= 1024, "pamo_s1_remesh: resolution must be in [8, 1024]");
    auto& c = *reinterpret_cast<pamo::s1::Ctx*>(s);
    PAMO_HIP(hipSetDevice(c.device));
    PAMO_TRY(pamo::s1::remesh(c, d_points, d_faces, n_faces, mean3, resolution));
    if (n_verts_out) *n_verts_out = c.n_verts;
    if (n_faces_out) *n_faces_out = c.n_faces;
    return 0;
}

int pamo_s1_get(pamo_s1* s, float* d_verts, int* d_faces) {
    pamo::clear_error();
    PAMO_CHECK(s && d_verts && d_faces, "pamo_s1_get: null argument");
    auto& c = *reinterpret_cast<pamo::s1::Ctx*>(s);
    PAMO_HIP(hipSetDevice(c.device));
    using namespace pamo::s1;
    if (c.n_verts > 0)
        hipLaunchKernelGGL(to_frame_k, dim3(pamo::grid_for(c.n_verts, kB)), dim3(kB), 0, c.stream,
                           (const float4*)c.verts, c.n_verts, c.R, c.band, c.margin, c.tmax, c.lo[0], c.lo[1], c.lo[2],
                           d_verts);
    PAMO_HIP(hipGetLastError());
    if (c.n_faces > 0)
        PAMO_HIP(hipMemcpyAsync(d_faces, c.tris, sizeof(int) * 3 * (size_t)c.n_faces, hipMemcpyDeviceToDevice,
                                c.stream));
    PAMO_HIP(hipStreamSynchronize(c.stream));
    return 0;
}

int pamo_s1_debug(pamo_s1* s, int what, void* h_out, long long cap, long long* n_out) {
    pamo::clear_error();
    PAMO_CHECK(s && n_out, "pamo_s1_debug: null argument");
    auto& c = *reinterpret_cast<pamo::s1::Ctx*>(s);
    PAMO_HIP(hipSetDevice(c.device));
    using namespace pamo::s1;
    const long long ng = (long long)c.R * c.R * c.R;
    long long n = 0;
    const void* src = nullptr;
    size_t elem = 0;
    std::vector<unsigned char> host;
    switch (what) {
    case PAMO_S1_DBG_FRAME: {
        n = 8;
        PAMO_CHECK(h_out && cap >= n, "pamo_s1_debug: output too small");
        float* o = static_cast<float*>(h_out);
        o[0] = c.mean[0]; o[1] = c.mean[1]; o[2] = c.mean[2];
        o[3] = c.lo[0]; o[4] = c.lo[1]; o[5] = c.lo[2];
        o[6] = c.tmax; o[7] = c.iso;
        *n_out = n;
        return 0;
    }
    case PAMO_S1_DBG_CASES: {
        n = 256 * 18;
        PAMO_CHECK(h_out && cap >= n, "pamo_s1_debug: output too small");
        const CaseTable* t = case_table();
        PAMO_CHECK(t != nullptr, "pamo_s1_debug: marching-cubes case table inconsistent");
        auto* o = static_cast<int8_t*>(h_out);
        for (int cs = 0; cs < 256; ++cs) {
            for (int e = 0; e < 12; ++e) o[18 * cs + e] = t->cyc[cs][e];
            for (int p = 0; p < 4; ++p) o[18 * cs + 12 + p] = t->plen[cs][p];
            o[18 * cs + 16] = t->npatch[cs];
            o[18 * cs + 17] = t->ntri[cs];
        }
        *n_out = n;
        return 0;
    }
    case PAMO_S1_DBG_FIELD: n = ng; src = c.grid; elem = 4; break;
    case PAMO_S1_DBG_OUTSIDE: n = ng; src = c.outside; elem = 1; break;
    case PAMO_S1_DBG_NORMALIZED: n = 12LL * c.n_in; src = c.tri; elem = 4; break;
    case PAMO_S1_DBG_VERTS: n = 4LL * c.n_verts; src = c.verts; elem = 4; break;
    default: PAMO_CHECK(false, "pamo_s1_debug: unknown item");
    }
    PAMO_CHECK(src != nullptr || n == 0, "pamo_s1_debug: nothing computed yet");
    PAMO_CHECK(h_out && cap >= n, "pamo_s1_debug: output too small");
    if (n > 0) {
        PAMO_HIP(hipMemcpyAsync(h_out, src, elem * (size_t)n, hipMemcpyDeviceToHost, c.stream));
        PAMO_HIP(hipStreamSynchronize(c.stream));
    }
    *n_out = n;
    return 0;
}

}  // extern "C"
