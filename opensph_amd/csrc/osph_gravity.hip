// Self-gravity of OpenSPH on gfx950 (MI355X): BarnesHut (core/gravity/BarnesHut.cpp) on a binary radix
// tree, BruteForceGravity (core/gravity/BruteForceGravity.h), and resident LeapFrog steps with the
// gravity-only HardSphereSolver (core/timestepping/TimeStepping.cpp:352-391, core/gravity/NBodySolver.cpp:97-117).
//
// Build (IGravity::build): the particles are sorted by the 63-bit Morton code of their position; the
// binary radix tree of the sorted codes (internal node i, 0 <= i < n-1, with one end of its range at
// sorted position i; particle k is node n-1+k) is built level-free in one pass, then the node moments
// are accumulated bottom-up.  Each node carries its box, centre of mass, opening radius
// r_open = 2/sqrt(3) |r_max| / theta (BarnesHut.cpp:411-414), and the traceless quadrupole and octupole
// about its centre of mass, combined from its two children with the parallel-axis theorem
// (BarnesHut.cpp:433-486, Moments.h:176-280).  A node of at most leaf_size particles is a leaf: it is
// never opened, and its particles are summed exactly when it is not approximated.
//
// Evaluation (IGravity::evalSelfGravity): every leaf (a node of <= leaf_size particles whose parent is
// larger) is a target.  Its interaction lists follow the reference's check-list walk (BarnesHut.cpp:212-312):
// a node whose opening ball does not overlap the target's box goes to the node list; a leaf whose ball
// overlaps goes to the particle list; other nodes are opened.  Nodes containing the target are always
// opened and the target's own pairs are summed separately, as the reference's walk never holds a node
// together with its ancestors.  One wavefront walks for a group of up to 16 neighbouring targets, up to 64 nodes
// at a time from a stack in LDS; the sums run one wavefront (or, for few targets, several) per target.
#include "osph_device.h"
#include "osph_gpu.h"
#include "osph_gravity.h"
#include "osph_transfer.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <string>
#include <type_traits>
#include <vector>

namespace osph {
namespace {

constexpr uint32_t END = 0xffffffffu;
constexpr int LUT_ENTRIES = 40000;  // LutKernel<3>::NEntries (core/sph/kernel/Kernel.h:53)
// Bound on the depth of the radix tree: 63 bits of Morton code plus 31 bits of position tie-break.
constexpr int MAX_DEPTH = 96;

// Words of osph_gravity::small and of its host mirror (the last two only there).
constexpr int SMALL_NEED = 6, SMALL_LEAVES = 7, SMALL_ERROR = 8, SMALL_LEVELS = 16;
constexpr int SMALL_HOST_WORDS = SMALL_LEVELS + MAX_DEPTH + 1;

// Plane indices of the resident state (storage order).
enum GPlane : int { GX, GY, GZ, GH, GVX, GVY, GVZ, GVH, GAX, GAY, GAZ, GM, NGPLANES };

// Traceless moments about the node's centre of mass; q2 = { xx, xy, xz, yy, yz } and
// q3 = { xxx, xxy, xxz, xyy, xyz, yyy, yyz } (the other components follow from the vanishing traces).
struct NodeMom {
    double M;
    double q2[5];
    double q3[7];
    double pad[3];
};
static_assert(sizeof(NodeMom) == 128, "NodeMom is 128 bytes");

// What the walk reads of a node it can visit, in FP32: the centre of mass as an offset from the root box's
// centre and r_open, both divided by the power of two 2^e at or above the root box's extent (so the
// offsets lie within [-1/2, 1/2]); count's top bit marks r_open == 0.  Written with the node's moments.
struct WalkNodeF {
    float4 geo;
    uint32_t first, count, left, right;
};
static_assert(sizeof(WalkNodeF) == 32, "WalkNodeF is 32 bytes");
constexpr uint32_t WALK_ZERO_R = 0x80000000u;

struct Tree {
    uint32_t n;        // particles; internal nodes 0..n-2, particle k is node n-1+k
    uint32_t leaf;     // leaf size
    uint32_t* left;    // [n-1]
    uint32_t* right;   // [n-1]
    uint32_t* parent;  // [2n-1]
    uint32_t* skip;    // [2n-1]: the node after this subtree in depth-first order (evaluation at points)
    uint32_t* first;   // [n-1]
    uint32_t* count;   // [n-1]
    double4* geo;      // [n-1]: centre of mass, r_open
    double4* lo;       // [n-1]: box
    double4* hi;
    NodeMom* mom;      // [n-1]
    WalkNodeF* wnf;    // [n-1]
    double ctr[3];     // the root box's centre and 2^-e, the scale of wnf
    double invL;
    uint32_t* flag;    // [n-1]: node depths while the moments are built
    const double4* pos;  // sorted x, y, z, h
    const double* gm;    // sorted G m
    double thetaInv;
    uint32_t* error;     // bit 0: a climb exceeded MAX_DEPTH; bit 1: a walk exceeded 2n visits
};

struct Planes {
    double* d[NGPLANES];
};

__device__ __forceinline__ bool is_particle(const Tree& t, uint32_t id) { return id >= t.n - 1; }

// ---- build ------------------------------------------------------------------------------------------

__global__ void __launch_bounds__(BLOCK) k_bounds3(Planes s, unsigned long long* acc, size_t n) {
    unsigned long long v[6] = { ~0ull, ~0ull, ~0ull, 0ull, 0ull, 0ull };
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
        for (int k = 0; k < 3; ++k) {
            const unsigned long long b = ord_bits(s.d[GX + k][i]);
            v[k] = b < v[k] ? b : v[k];
            v[3 + k] = b > v[3 + k] ? b : v[3 + k];
        }
    }
    __shared__ unsigned long long red[BLOCK / 64][6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < 6; ++k) {
        const unsigned long long r = k < 3 ? wave_min(v[k]) : wave_max(v[k]);
        if (lane == 0) red[wave][k] = r;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int k = threadIdx.x;
        unsigned long long r = red[0][k];
        for (int w = 1; w < BLOCK / 64; ++w) r = k < 3 ? (red[w][k] < r ? red[w][k] : r) : (red[w][k] > r ? red[w][k] : r);
        if (k < 3) {
            atomicMin(&acc[k], r);
        } else {
            atomicMax(&acc[k], r);
        }
    }
}

__device__ __forceinline__ uint64_t spread21(uint64_t v) {
    v &= 0x1fffffull;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

__global__ void __launch_bounds__(BLOCK) k_morton(Planes s, double lo0, double lo1, double lo2, double scale,
                                                  uint64_t* keys, uint32_t* idx, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double lo[3] = { lo0, lo1, lo2 };
    uint64_t key = 0;
    for (int k = 0; k < 3; ++k) {
        double q = floor((s.d[GX + k][i] - lo[k]) * scale);
        q = q < 0.0 ? 0.0 : (q > 2097151.0 ? 2097151.0 : q);
        key |= spread21(uint64_t(q)) << k;
    }
    keys[i] = key;
    idx[i] = uint32_t(i);
}

// The state moved into the slots of the Morton order: slot k of dst takes every plane of slot order[k]
// of src, and the particle's index in the caller's order (perm_in of that slot, or the slot itself while
// the state is in the caller's order) goes with it, into perm_out and its inverse slot_of.
__global__ void __launch_bounds__(BLOCK) k_permute_planes(Planes src, Planes dst, const uint32_t* __restrict__ order,
                                                          const uint32_t* __restrict__ perm_in,
                                                          uint32_t* __restrict__ perm_out,
                                                          uint32_t* __restrict__ slot_of, size_t n) {
    const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t i = order[k];
    for (int p = 0; p < NGPLANES; ++p) dst.d[p][k] = src.d[p][i];
    const uint32_t u = perm_in ? perm_in[i] : i;
    perm_out[k] = u;
    slot_of[u] = uint32_t(k);
}

__global__ void __launch_bounds__(BLOCK) k_sequence(uint32_t* __restrict__ p, size_t n) {
    const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n) p[k] = uint32_t(k);
}

// Particle indices in the caller's order to the slots that hold them.
__global__ void __launch_bounds__(BLOCK) k_to_slots(uint32_t* __restrict__ idx, const uint32_t* __restrict__ slot_of,
                                                    size_t n) {
    const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n) idx[k] = slot_of[idx[k]];
}

__global__ void __launch_bounds__(BLOCK) k_gather(Planes s, const uint32_t* __restrict__ order, double G,
                                                  double4* __restrict__ pos, double* __restrict__ gm, size_t n) {
    const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t i = order[k];
    pos[k] = make_double4(s.d[GX][i], s.d[GY][i], s.d[GZ][i], s.d[GH][i]);
    gm[k] = G * s.d[GM][i];  // BarnesHut::build premultiplies the masses (BarnesHut.cpp:58-60)
}

// Common-prefix length of sorted codes i and j; equal codes are told apart by their positions.
__device__ __forceinline__ int delta(const uint64_t* __restrict__ keys, long long i, long long j, long long n) {
    if (j < 0 || j >= n) return -1;
    const uint64_t a = keys[i], b = keys[j];
    if (a == b) return 64 + __clz(uint32_t(i) ^ uint32_t(j));
    return __clzll(a ^ b);
}

// Internal node i of the binary radix tree of the sorted codes: its range, split and children.
__global__ void __launch_bounds__(BLOCK) k_radix_tree(Tree t, const uint64_t* __restrict__ keys) {
    const long long n = t.n;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (delta(keys, i, i + 1, n) - delta(keys, i, i - 1, n)) >= 0 ? 1 : -1;
    const int dmin_ = delta(keys, i, i - d, n);
    long long lmax = 2;
    while (delta(keys, i, i + lmax * d, n) > dmin_) lmax <<= 1;
    long long l = 0;
    for (long long s = lmax >> 1; s >= 1; s >>= 1) {
        if (delta(keys, i, i + (l + s) * d, n) > dmin_) l += s;
    }
    const long long j = i + l * d;
    const int dnode = delta(keys, i, j, n);
    long long split = 0;
    for (long long div = 2;; div <<= 1) {
        const long long s = (l + div - 1) / div;
        if (delta(keys, i, i + (split + s) * d, n) > dnode) split += s;
        if (s == 1) break;
    }
    const long long gamma = i + split * d + (d < 0 ? -1 : 0);
    const long long lo = i < j ? i : j, hi = i < j ? j : i;
    const uint32_t lc = uint32_t(lo == gamma ? (n - 1 + gamma) : gamma);
    const uint32_t rc = uint32_t(hi == gamma + 1 ? (n - 1 + gamma + 1) : gamma + 1);
    t.left[i] = lc;
    t.right[i] = rc;
    t.first[i] = uint32_t(lo);
    t.count[i] = uint32_t(hi - lo + 1);
    t.parent[lc] = uint32_t(i);
    t.parent[rc] = uint32_t(i);
    if (i == 0) t.parent[0] = END;
}

// Depth-first successor of each node: the right sibling of the nearest ancestor-or-self that is a left
// child, or END.  Only for the nodes a walk can visit: the root and the children of nodes of more than
// leaf_size particles (the nodes inside a leaf are never visited).
__global__ void __launch_bounds__(BLOCK) k_skip(Tree t) {
    const size_t id = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t total = 2 * size_t(t.n) - 1;
    if (id >= total) return;
    if (id != 0 && t.count[t.parent[id]] <= t.leaf) return;
    uint32_t c = uint32_t(id), next = END;
    for (int level = 0; c != 0u && level < MAX_DEPTH; ++level) {
        const uint32_t p = t.parent[c];
        if (t.left[p] == c) {
            next = t.right[p];
            break;
        }
        c = p;
    }
    t.skip[id] = next;
}

struct Moments {
    double M, c[3], lo[3], hi[3], q2[5], q3[7];
};

__device__ void load_node(const Tree& t, uint32_t id, Moments& m) {
    if (is_particle(t, id)) {
        const double4 p = t.pos[id - (t.n - 1)];
        m.M = t.gm[id - (t.n - 1)];
        m.c[0] = m.lo[0] = m.hi[0] = p.x;
        m.c[1] = m.lo[1] = m.hi[1] = p.y;
        m.c[2] = m.lo[2] = m.hi[2] = p.z;
        for (int k = 0; k < 5; ++k) m.q2[k] = 0.0;
        for (int k = 0; k < 7; ++k) m.q3[k] = 0.0;
        return;
    }
    const double4 g = t.geo[id], lo = t.lo[id], hi = t.hi[id];
    const NodeMom& q = t.mom[id];
    m.M = q.M;
    m.c[0] = g.x;
    m.c[1] = g.y;
    m.c[2] = g.z;
    m.lo[0] = lo.x;
    m.lo[1] = lo.y;
    m.lo[2] = lo.z;
    m.hi[0] = hi.x;
    m.hi[1] = hi.y;
    m.hi[2] = hi.z;
    for (int k = 0; k < 5; ++k) m.q2[k] = q.q2[k];
    for (int k = 0; k < 7; ++k) m.q3[k] = q.q3[k];
}

// Adds the moments of child m (shifted by d = com_child - com_parent) to q2 and q3: the parallel-axis
// theorem for traceless moments (Moments.h:176-186, 262-280).  With t = q2 d:
//   q2 += q2c + M (d d - |d|^2/3 I)
//   q3 += q3c + M (d d d - |d|^2/5 sym(I d)) + sym(q2c d) - 2/5 sym(I t)
// where sym sums the three distinct index placements.
__device__ void add_shifted(const Moments& m, const double d[3], double q2[5], double q3[7]) {
    const double dd = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    const double M = m.M;
    q2[0] += m.q2[0] + M * (d[0] * d[0] - dd / 3.0);
    q2[1] += m.q2[1] + M * (d[0] * d[1]);
    q2[2] += m.q2[2] + M * (d[0] * d[2]);
    q2[3] += m.q2[3] + M * (d[1] * d[1] - dd / 3.0);
    q2[4] += m.q2[4] + M * (d[1] * d[2]);
    // full child quadrupole
    const double cxx = m.q2[0], cxy = m.q2[1], cxz = m.q2[2], cyy = m.q2[3], cyz = m.q2[4], czz = -cxx - cyy;
    const double Q[3][3] = { { cxx, cxy, cxz }, { cxy, cyy, cyz }, { cxz, cyz, czz } };
    double tv[3];
    for (int a = 0; a < 3; ++a) tv[a] = Q[a][0] * d[0] + Q[a][1] * d[1] + Q[a][2] * d[2];
    // independent components (i, j, k) of q3
    const int I3[7][3] = { { 0, 0, 0 }, { 0, 0, 1 }, { 0, 0, 2 }, { 0, 1, 1 }, { 0, 1, 2 }, { 1, 1, 1 }, { 1, 1, 2 } };
#pragma unroll
    for (int c = 0; c < 7; ++c) {
        const int i = I3[c][0], j = I3[c][1], k = I3[c][2];
        const double dij = i == j ? 1.0 : 0.0, dik = i == k ? 1.0 : 0.0, djk = j == k ? 1.0 : 0.0;
        const double red = d[i] * d[j] * d[k] - dd / 5.0 * (dij * d[k] + dik * d[j] + djk * d[i]);
        const double perm = Q[i][j] * d[k] + Q[i][k] * d[j] + Q[j][k] * d[i];
        const double permt = dij * tv[k] + dik * tv[j] + djk * tv[i];
        q3[c] += m.q3[c] + M * red + perm - 0.4 * permt;
    }
}

// The walk's record of a node whose centre c and opening radius are known.
__device__ __forceinline__ void write_walk_record(const Tree& t, uint32_t id, const double c[3], double r_open) {
    WalkNodeF f;
    f.geo = make_float4(float((c[0] - t.ctr[0]) * t.invL), float((c[1] - t.ctr[1]) * t.invL),
                        float((c[2] - t.ctr[2]) * t.invL), float(r_open * t.invL));
    f.first = t.first[id];
    f.count = t.count[id] | (r_open == 0.0 ? WALK_ZERO_R : 0u);
    f.left = t.left[id];
    f.right = t.right[id];
    t.wnf[id] = f;
}

// Node `node` from its two children: box, centre of mass and opening radius (BarnesHut::buildInner,
// BarnesHut.cpp:433-468), moments by the parallel-axis theorem.
__device__ void combine(const Tree& t, uint32_t node) {
    Moments a, b;
    load_node(t, t.left[node], a);
    load_node(t, t.right[node], b);
    const double M = a.M + b.M;
    double c[3], lo[3], hi[3];
    for (int q = 0; q < 3; ++q) {
        lo[q] = dmin(a.lo[q], b.lo[q]);
        hi[q] = dmax(a.hi[q], b.hi[q]);
    }
    NodeMom out{};
    double r_open = 0.0;
    if (M == 0.0) {
        c[0] = c[1] = c[2] = 0.0;
    } else {
        for (int q = 0; q < 3; ++q) c[q] = (a.M * a.c[q] + b.M * b.c[q]) / M;
        double rm[3];
        for (int q = 0; q < 3; ++q) rm[q] = dmax(c[q] - lo[q], hi[q] - c[q]);
        r_open = 2.0 / sqrt(3.0) * t.thetaInv * sqrt(rm[0] * rm[0] + rm[1] * rm[1] + rm[2] * rm[2]);
        out.M = M;
        double da[3], db[3];
        for (int q = 0; q < 3; ++q) {
            da[q] = a.c[q] - c[q];
            db[q] = b.c[q] - c[q];
        }
        add_shifted(a, da, out.q2, out.q3);
        add_shifted(b, db, out.q2, out.q3);
    }
    t.geo[node] = make_double4(c[0], c[1], c[2], r_open);
    write_walk_record(t, node, c, r_open);
    t.lo[node] = make_double4(lo[0], lo[1], lo[2], 0.0);
    t.hi[node] = make_double4(hi[0], hi[1], hi[2], 0.0);
    t.mom[node] = out;
}

// Moments of a leaf (an internal node of at most leaf_size particles whose parent is larger, or the
// root when it is that small) from its particles, as BarnesHut::buildLeaf computes them
// (BarnesHut.cpp:401-437; computeMultipole, Moments.h:167-180): mass, box, centre of mass, r_open, and
// the traceless moments about the centre summed particle by particle.  The centre is accumulated
// relative to the first particle, so that a leaf of coincident particles has its centre on them exactly
// (and r_open 0).
// The internal nodes inside a leaf are never read by the walks or the evaluations and get no moments.
// LEAF_LANES lanes per entry of the leaf list (k_mark_leaves, compacted in Morton order), each summing
// every LEAF_LANES-th particle of the leaf, the partial sums then added across the group in a fixed
// order; single-particle leaves need nothing.
constexpr uint32_t LEAF_LANES = 8;
__device__ __forceinline__ double leaf_sum(double v) {
    for (int o = LEAF_LANES / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o, LEAF_LANES);
    return v;
}
__device__ __forceinline__ double leaf_min(double v) {
    for (int o = LEAF_LANES / 2; o >= 1; o >>= 1) v = dmin(v, __shfl_xor(v, o, LEAF_LANES));
    return v;
}
__device__ __forceinline__ double leaf_max(double v) {
    for (int o = LEAF_LANES / 2; o >= 1; o >>= 1) v = dmax(v, __shfl_xor(v, o, LEAF_LANES));
    return v;
}
__global__ void __launch_bounds__(BLOCK) k_leaf_moments(Tree t, const uint32_t* __restrict__ leaves,
                                                        const uint32_t* __restrict__ nleaves) {
    const size_t gid = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t q = gid / LEAF_LANES;
    const uint32_t sub = uint32_t(gid % LEAF_LANES);
    // uniform over the group of LEAF_LANES lanes, so every shuffle below reads lanes of the same leaf
    if (q >= *nleaves) return;
    const uint32_t i = leaves[q];
    if (is_particle(t, i)) return;
    const uint32_t cnt = t.count[i];
    const uint32_t f = t.first[i];
    const double4 p0 = t.pos[f];
    double lo[3] = { p0.x, p0.y, p0.z }, hi[3] = { p0.x, p0.y, p0.z };
    double M = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
    for (uint32_t j = f + sub; j < f + cnt; j += LEAF_LANES) {
        const double4 p = t.pos[j];
        const double m = t.gm[j];
        lo[0] = dmin(lo[0], p.x);
        lo[1] = dmin(lo[1], p.y);
        lo[2] = dmin(lo[2], p.z);
        hi[0] = dmax(hi[0], p.x);
        hi[1] = dmax(hi[1], p.y);
        hi[2] = dmax(hi[2], p.z);
        M += m;
        sx += m * (p.x - p0.x);
        sy += m * (p.y - p0.y);
        sz += m * (p.z - p0.z);
    }
    for (int k = 0; k < 3; ++k) {
        lo[k] = leaf_min(lo[k]);
        hi[k] = leaf_max(hi[k]);
    }
    M = leaf_sum(M);
    sx = leaf_sum(sx);
    sy = leaf_sum(sy);
    sz = leaf_sum(sz);
    NodeMom out{};
    double c[3] = { 0.0, 0.0, 0.0 }, r_open = 0.0;
    if (M != 0.0) {
        c[0] = p0.x + sx / M;
        c[1] = p0.y + sy / M;
        c[2] = p0.z + sz / M;
        double rm[3];
        for (int k = 0; k < 3; ++k) rm[k] = dmax(c[k] - lo[k], hi[k] - c[k]);
        r_open = 2.0 / sqrt(3.0) * t.thetaInv * sqrt(rm[0] * rm[0] + rm[1] * rm[1] + rm[2] * rm[2]);
        out.M = M;
        Moments pm{};
        for (uint32_t j = f + sub; j < f + cnt; j += LEAF_LANES) {
            const double4 p = t.pos[j];
            pm.M = t.gm[j];
            const double d[3] = { p.x - c[0], p.y - c[1], p.z - c[2] };
            add_shifted(pm, d, out.q2, out.q3);  // a point mass: only the shift terms
        }
        for (int k = 0; k < 5; ++k) out.q2[k] = leaf_sum(out.q2[k]);
        for (int k = 0; k < 7; ++k) out.q3[k] = leaf_sum(out.q3[k]);
    }
    if (sub != 0) return;
    t.geo[i] = make_double4(c[0], c[1], c[2], r_open);
    write_walk_record(t, i, c, r_open);
    t.lo[i] = make_double4(lo[0], lo[1], lo[2], 0.0);
    t.hi[i] = make_double4(hi[0], hi[1], hi[2], 0.0);
    t.mom[i] = out;
}

// Depth of every internal node above the leaves (more than leaf_size particles; the number of its
// ancestors, all of them such nodes too) and the node count per depth; the other nodes get NO_DEPTH.
// Their moments are then built one depth per launch, deepest first, from the leaves' moments: the
// children of a node are complete when the launch of its depth starts, with no fences between
// work-groups.  A bounded grid strides over the nodes, so that few blocks add their per-depth counts
// to the ~100 global counters.
constexpr uint32_t NO_DEPTH = 0xffffffffu;
constexpr unsigned LEVEL_BLOCKS = 1024;
__global__ void __launch_bounds__(BLOCK) k_depth(Tree t, uint32_t* __restrict__ depth, uint32_t* __restrict__ per_level) {
    __shared__ uint32_t hist[MAX_DEPTH + 1];
    for (int d = threadIdx.x; d <= MAX_DEPTH; d += blockDim.x) hist[d] = 0u;
    __syncthreads();
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i + 1 < t.n; i += stride) {
        if (t.count[i] <= t.leaf) {
            depth[i] = NO_DEPTH;
            continue;
        }
        uint32_t c = uint32_t(i), d = 0;
        while (c != 0u && d < uint32_t(MAX_DEPTH)) {
            c = t.parent[c];
            ++d;
        }
        if (c != 0u) {
            atomicOr(t.error, 1u);
            d = 0;
        }
        depth[i] = d;
        atomicAdd(&hist[d], 1u);
    }
    __syncthreads();
    for (int d = threadIdx.x; d <= MAX_DEPTH; d += blockDim.x) {
        if (hist[d]) atomicAdd(&per_level[d], hist[d]);
    }
}

// Scatter of the internal nodes above the leaves into per-depth buckets.  Each block of a bounded grid
// counts its strided share of the nodes per depth in LDS, reserves one range per depth, then places
// its nodes from LDS cursors (the order inside a bucket is free: each node's moments depend only on
// its children).
__global__ void __launch_bounds__(BLOCK) k_bucket(uint32_t n_internal, const uint32_t* __restrict__ depth,
                                                  uint32_t* __restrict__ cursor, uint32_t* __restrict__ nodes) {
    __shared__ uint32_t cnt[MAX_DEPTH + 1];
    __shared__ uint32_t base[MAX_DEPTH + 1];
    for (int d = threadIdx.x; d <= MAX_DEPTH; d += blockDim.x) cnt[d] = 0u;
    __syncthreads();
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    const size_t i0 = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (size_t i = i0; i < n_internal; i += stride) {
        const uint32_t d = depth[i];
        if (d != NO_DEPTH) atomicAdd(&cnt[d], 1u);
    }
    __syncthreads();
    for (int k = threadIdx.x; k <= MAX_DEPTH; k += blockDim.x) {
        base[k] = cnt[k] ? atomicAdd(&cursor[k], cnt[k]) : 0u;
        cnt[k] = 0u;
    }
    __syncthreads();
    for (size_t i = i0; i < n_internal; i += stride) {
        const uint32_t d = depth[i];
        if (d != NO_DEPTH) nodes[base[d] + atomicAdd(&cnt[d], 1u)] = uint32_t(i);
    }
}

// First entries of the depths' buckets (cursor), and the leaf count, the error flags and the depths' node counts to the
// host (words SMALL_LEAVES, SMALL_ERROR and SMALL_LEVELS + d).
__global__ void __launch_bounds__(BLOCK) k_levels(const uint32_t* __restrict__ per_level, uint32_t* __restrict__ cursor,
                                                  const uint32_t* __restrict__ leaves, const uint32_t* __restrict__ error,
                                                  MailboxPost post) {
    __shared__ uint32_t cnt[MAX_DEPTH + 1];
    const int d = threadIdx.x;
    if (d <= MAX_DEPTH) {
        cnt[d] = per_level[d];
        __hip_atomic_store(post.host + SMALL_LEVELS + d, cnt[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    } else if (d == MAX_DEPTH + 1) {
        __hip_atomic_store(post.host + SMALL_LEAVES, *leaves, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(post.host + SMALL_ERROR, *error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __threadfence_system();
    __syncthreads();
    if (d == 0) __hip_atomic_store(post.posts, post.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    if (d <= MAX_DEPTH) {
        uint32_t at = 0;
        for (int e = 0; e < d; ++e) at += cnt[e];
        cursor[d] = at;
    }
}

// A run of depths of at most LEVEL_RUN nodes each (most of them the top of the tree), deepest first, in one block, whose
// barrier costs less than a launch per depth: moments of 20k / 100k / 1M particles 87 / 123 / 231 -> 75 / 110 / 220 us
// (runs of up to 64 nodes: 79 / 116 / 228, of 1024: 79 / 128 / 253).  k_bucket leaves the cursors at the ends of the
// depths.
constexpr uint32_t LEVEL_RUN = 256;
__global__ void __launch_bounds__(LEVEL_RUN) k_moments_run(Tree t, const uint32_t* __restrict__ nodes,
                                                           const uint32_t* __restrict__ ends, int deepest, int top) {
    for (int d = deepest; d >= top; --d) {
        const uint32_t k = (d ? ends[d - 1] : 0u) + threadIdx.x;
        if (k < ends[d]) combine(t, nodes[k]);
        __syncthreads();
    }
}

__global__ void __launch_bounds__(BLOCK) k_moments_level(Tree t, const uint32_t* __restrict__ nodes, uint32_t count) {
    const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= count) return;
    combine(t, nodes[k]);
}

// Leaves (targets): nodes of at most leaf_size particles whose parent is larger, and particles whose
// parent is larger.  leaf_at[first] = node id.
__global__ void __launch_bounds__(BLOCK) k_mark_leaves(Tree t, uint32_t* leaf_at) {
    const size_t id = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t total = 2 * size_t(t.n) - 1;
    if (id >= total) return;
    const uint32_t p = id == 0 ? END : t.parent[id];
    const uint32_t pc = p == END ? 0xffffffffu : t.count[p];
    if (is_particle(t, uint32_t(id))) {
        if (pc > t.leaf) leaf_at[id - (t.n - 1)] = uint32_t(id);
    } else if (t.count[id] <= t.leaf && pc > t.leaf) {
        leaf_at[t.first[id]] = uint32_t(id);
    }
}

struct NotEnd {
    __host__ __device__ bool operator()(uint32_t v) const { return v != END; }
};

// Sphere::overlaps (core/objects/geometry/Sphere.h:73-79): the ball (c, r) and the box share a point.
__device__ __forceinline__ bool ball_overlaps_box(double4 g, const double lo[3], const double hi[3]) {
#pragma clang fp contract(off)
    const double c[3] = { g.x, g.y, g.z };
    double l2 = 0.0, r2 = 0.0;
    double lv[3], rv[3];
    for (int k = 0; k < 3; ++k) {
        lv[k] = dmax(lo[k] - c[k], 0.0);
        rv[k] = dmax(c[k] - hi[k], 0.0);
    }
    l2 = lv[0] * lv[0] + lv[1] * lv[1] + lv[2] * lv[2];
    r2 = rv[0] * rv[0] + rv[1] * rv[1] + rv[2] * rv[2];
    return g.w * g.w - l2 - r2 > 0.0;
}

__device__ __forceinline__ void node_range(const Tree& t, uint32_t id, uint32_t& f, uint32_t& c) {
    if (is_particle(t, id)) {
        f = id - (t.n - 1);
        c = 1;
    } else {
        f = t.first[id];
        c = t.count[id];
    }
}

// The target's box: its leaf's box, or the particle itself.
__device__ __forceinline__ void target_box(const Tree& t, uint32_t T, uint32_t tf, double lo[3], double hi[3]) {
    if (is_particle(t, T)) {
        const double4 p = t.pos[tf];
        lo[0] = hi[0] = p.x;
        lo[1] = hi[1] = p.y;
        lo[2] = hi[2] = p.z;
    } else {
        const double4 a = t.lo[T], b = t.hi[T];
        lo[0] = a.x;
        lo[1] = a.y;
        lo[2] = a.z;
        hi[0] = b.x;
        hi[1] = b.y;
        hi[2] = b.z;
    }
}

// ---- evaluation ---------------------------------------------------------------------------------------

// GravityLutKernel::grad (core/sph/kernel/GravityKernel.h:60-70) times the source mass, added to a.
// grads == nullptr is the point-particle kernel (radius 0).  REF evaluates it as the reference does
// (the direct sum is then bit-identical to it); otherwise the tree sums use the cheaper form below.
template <bool REF>
__device__ __forceinline__ void add_pair(const double* __restrict__ grads, double rx, double ry, double rz, double h,
                                         double m, double a[3]) {
#pragma clang fp contract(off)
    if (!REF) {
        // the same branches, decided on |r|^2 against (4 - EPS) h^2 without dividing by h, and the
        // Newtonian branch with one reciprocal square root
        const double d2 = rx * rx + ry * ry + rz * rz;
        if (grads && d2 < (4.0 - EPS_D) * (h * h)) {
            const double hInv = 1.0 / h;
            const double qSqr = d2 * (hInv * hInv);
            const double fi = double(LUT_ENTRIES / 4) * qSqr;
            const uint32_t i1 = uint32_t(fi);
            const double ratio = fi - double(i1);
            const double gr = grads[i1] * (1.0 - ratio) + grads[i1 + 1] * ratio;
            const double f = m * (hInv * hInv * hInv) * gr;
            a[0] += rx * f;
            a[1] += ry * f;
            a[2] += rz * f;
            return;
        }
        const double il = rsqrt(d2);
        const double f = m * (il * il * il);
        a[0] += rx * f;
        a[1] += ry * f;
        a[2] += rz * f;
        return;
    }
    if (grads) {
        const double hInv = 1.0 / h;
        const double sx = rx * hInv, sy = ry * hInv, sz = rz * hInv;
        const double qSqr = sx * sx + sy * sy + sz * sz;
        if (!(qSqr + EPS_D >= 4.0)) {
            // LutKernel<3>::gradImpl (core/sph/kernel/Kernel.h:129-144)
            const double fi = double(LUT_ENTRIES / 4) * qSqr;
            const uint32_t i1 = uint32_t(fi);
            const double ratio = fi - double(i1);
            const double gr = grads[i1] * (1.0 - ratio) + grads[i1 + 1] * ratio;
            const double h3 = hInv * hInv * hInv;
            a[0] += m * ((h3 * rx) * gr);
            a[1] += m * ((h3 * ry) * gr);
            a[2] += m * ((h3 * rz) * gr);
            return;
        }
    }
    const double l = sqrt(rx * rx + ry * ry + rz * rz);
    const double l3 = l * l * l;
    a[0] += m * (rx / l3);
    a[1] += m * (ry / l3);
    a[2] += m * (rz / l3);
}

// evaluateGravity (core/gravity/Moments.h:318-360) of node moments at dr = r - com, added to a.
__device__ __forceinline__ void add_multipole(const NodeMom& q, double drx, double dry, double drz, int order,
                                              double a[3]) {
    const double il = rsqrt(drx * drx + dry * dry + drz * drz);
    const double inv = il * il;
    const double g0 = -il;
    const double g1 = -1.0 * inv * g0;
    const double g2 = -3.0 * inv * g1;
    const double g3 = -5.0 * inv * g2;
    const double g4 = -7.0 * inv * g3;
    const double d0 = -drx, d1 = -dry, d2 = -drz;
    double ax = 0.0, ay = 0.0, az = 0.0;
    if (order >= 3) {
        const double xxx = q.q3[0], xxy = q.q3[1], xxz = q.q3[2], xyy = q.q3[3], xyz = q.q3[4], yyy = q.q3[5],
                     yyz = q.q3[6];
        const double xzz = -xxx - xyy, yzz = -xxy - yyy, zzz = -xxz - yyz;
        // Q1_i = q_ijk d_j d_k
        const double Q1x = xxx * d0 * d0 + xyy * d1 * d1 + xzz * d2 * d2 + 2.0 * (xxy * d0 * d1 + xxz * d0 * d2 + xyz * d1 * d2);
        const double Q1y = xxy * d0 * d0 + yyy * d1 * d1 + yzz * d2 * d2 + 2.0 * (xyy * d0 * d1 + xyz * d0 * d2 + yyz * d1 * d2);
        const double Q1z = xxz * d0 * d0 + yyz * d1 * d1 + zzz * d2 * d2 + 2.0 * (xyz * d0 * d1 + xzz * d0 * d2 + yzz * d1 * d2);
        const double Q0 = (Q1x * d0 + Q1y * d1 + Q1z * d2) * (1.0 / 6.0);
        ax += g4 * d0 * Q0 + g3 * (0.5 * Q1x);
        ay += g4 * d1 * Q0 + g3 * (0.5 * Q1y);
        az += g4 * d2 * Q0 + g3 * (0.5 * Q1z);
    }
    if (order >= 2) {
        const double xx = q.q2[0], xy = q.q2[1], xz = q.q2[2], yy = q.q2[3], yz = q.q2[4], zz = -xx - yy;
        const double Q1x = xx * d0 + xy * d1 + xz * d2;
        const double Q1y = xy * d0 + yy * d1 + yz * d2;
        const double Q1z = xz * d0 + yz * d1 + zz * d2;
        const double Q0 = 0.5 * (Q1x * d0 + Q1y * d1 + Q1z * d2);
        ax += g3 * d0 * Q0 + g2 * Q1x;
        ay += g3 * d1 * Q0 + g2 * Q1y;
        az += g3 * d2 * Q0 + g2 * Q1z;
    }
    ax += g1 * d0 * q.M;
    ay += g1 * d1 * q.M;
    az += g1 * d2 * q.M;
    a[0] += ax;
    a[1] += ay;
    a[2] += az;
}

// 1 / sqrt(x) for x > 0: the hardware estimate and one third-order step, y (1 + e/2 + 3 e^2 / 8) with e = 1 - x y^2, the
// binomial series of (1 - e)^(-1/2) to second order (Householder 1970, The Numerical Treatment of a Single Nonlinear
// Equation, for the family).  WIDE: an infinite x, a squared distance past the largest number, is taken as that
// number, as its estimate would be 0 and the step 0 * infinity.
template <bool WIDE>
__device__ __forceinline__ double rsqrt_step(double x) {
    if (WIDE) x = __builtin_fmin(x, 1.79769313486231570815e308);
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// A node as the evaluation reads it: centre and mass, then by order q2 (6 components) and q3 (10 components),
// in FP64 with the factors -3 and 7.5 of the expansion; whole 16-byte chunks, so that a lane reads it with
// 16-byte LDS loads.
template <typename T, int ORDER>
struct alignas(16) NodeRow {
    static constexpr int N = ORDER >= 3 ? 20 : (ORDER >= 2 ? 10 : 4);
    T v[sizeof(T) == 4 && ORDER == 2 ? 12 : N];
};

// The components of q2 times f2 and q3 times f3 of a node into its row.
template <typename T, int ORDER>
__device__ __forceinline__ void row_moments(NodeRow<T, ORDER>& r, const NodeMom& q, double f2, double f3) {
    if constexpr (ORDER >= 2) {
        for (int k = 0; k < 5; ++k) r.v[4 + k] = T(q.q2[k] * f2);
        r.v[9] = -r.v[4] - r.v[7];  // zz
    }
    if constexpr (ORDER >= 3) {
        for (int k = 0; k < 7; ++k) r.v[10 + k] = T(q.q3[k] * f3);
        r.v[17] = -r.v[10] - r.v[13];  // xzz
        r.v[18] = -r.v[11] - r.v[15];  // yzz
        r.v[19] = -r.v[12] - r.v[16];  // zzz
    }
}

// q3:dd of a row's octupole, the contraction over two indices with d.
__device__ __forceinline__ void octupole_dd(const NodeRow<double, 3>& r, double dx, double dy, double dz, double w[3]) {
    const double xx = dx * dx, yy = dy * dy, zz = dz * dz;
    const double xy = (dx + dx) * dy, xz = (dx + dx) * dz, yz = (dy + dy) * dz;
    w[0] = r.v[10] * xx + r.v[13] * yy + r.v[17] * zz + r.v[11] * xy + r.v[12] * xz + r.v[14] * yz;
    w[1] = r.v[11] * xx + r.v[15] * yy + r.v[18] * zz + r.v[13] * xy + r.v[14] * xz + r.v[16] * yz;
    w[2] = r.v[12] * xx + r.v[16] * yy + r.v[19] * zz + r.v[14] * xy + r.v[17] * xz + r.v[18] * yz;
}

// evaluateGravity (core/gravity/Moments.h:318-360) of a staged node at the point (x, y, z), added to a.  With
// d from the point to the node's centre and il = 1 / |d|:
//   monopole   il^3 M d
//   quadrupole 7.5 il^7 (d.q2.d) d - 3 il^5 q2.d
//   octupole   7.5 il^7 (q3:dd) - 17.5 il^9 (q3:ddd) d
// The terms along d share one factor and the tensors carry theirs (-3, 7.5) from the staging: 40 FP64
// instructions for a quadrupole, against about 65 in the order the reference writes them.
template <int ORDER, bool WIDE>
__device__ __forceinline__ void expand(const NodeRow<double, ORDER>& r, double x, double y, double z, double a[3]) {
    const double dx = r.v[0] - x, dy = r.v[1] - y, dz = r.v[2] - z;
    const double il = rsqrt_step<WIDE>(dx * dx + dy * dy + dz * dz);
    const double inv = il * il, i3 = inv * il;
    double s = i3 * r.v[3];
    if constexpr (ORDER >= 2) {
        const double i5 = i3 * inv;
        double vx = r.v[4] * dx + r.v[5] * dy + r.v[6] * dz;
        double vy = r.v[5] * dx + r.v[7] * dy + r.v[8] * dz;
        double vz = r.v[6] * dx + r.v[8] * dy + r.v[9] * dz;
        s += (-2.5 * i5) * (inv * (vx * dx + vy * dy + vz * dz));
        if constexpr (ORDER >= 3) {
            double w[3];
            octupole_dd(r, dx, dy, dz, w);
            s += (-7.0 / 3.0 * i5) * ((inv * inv) * (w[0] * dx + w[1] * dy + w[2] * dz));
            vx += inv * w[0];
            vy += inv * w[1];
            vz += inv * w[2];
        }
        a[0] += vx * i5;
        a[1] += vy * i5;
        a[2] += vz * i5;
    }
    a[0] += dx * s;
    a[1] += dy * s;
    a[2] += dz * s;
}

// The multipole expansion in FP32, written so that no intermediate leaves FP32's range: with d the vector from
// the target to the node's centre of mass, il = 1/|d|, u = d il and w = il^2,
//   monopole   il^3 M d                                  = w M u
//   quadrupole il^4 (7.5 u (u.q2.u) - 3 q2.u)            = w^2 t2
//   octupole   il^5 (7.5 (q3:uu) - 17.5 u (q3:uuu))      = w^2 il t3
// and an approximated node has size < theta |d|, so w |q2| < theta^2 M and w il |q3| < theta^3 M.  The row holds
// q2 and q3 themselves, with the components that follow from the vanishing traces.
template <int ORDER>
__device__ __forceinline__ void expand(const NodeRow<float, ORDER>& r, float mx, float my, float mz, float a[3]) {
    const float dx = r.v[0] - mx, dy = r.v[1] - my, dz = r.v[2] - mz, M = r.v[3];
    const float il = __builtin_amdgcn_rsqf(dx * dx + dy * dy + dz * dz);
    const float w = il * il;
    const float u0 = dx * il, u1 = dy * il, u2 = dz * il;
    float hx = 0.f, hy = 0.f, hz = 0.f;
    if constexpr (ORDER >= 2) {
        const float xx = r.v[4], xy = r.v[5], xz = r.v[6], yy = r.v[7], yz = r.v[8], zz = r.v[9];
        const float Q1x = xx * u0 + xy * u1 + xz * u2;
        const float Q1y = xy * u0 + yy * u1 + yz * u2;
        const float Q1z = xz * u0 + yz * u1 + zz * u2;
        const float Q0 = 7.5f * (Q1x * u0 + Q1y * u1 + Q1z * u2);
        hx = Q0 * u0 - 3.f * Q1x;
        hy = Q0 * u1 - 3.f * Q1y;
        hz = Q0 * u2 - 3.f * Q1z;
    }
    if constexpr (ORDER >= 3) {
        const float xxx = r.v[10], xxy = r.v[11], xxz = r.v[12], xyy = r.v[13], xyz = r.v[14], yyy = r.v[15],
                    yyz = r.v[16], xzz = r.v[17], yzz = r.v[18], zzz = r.v[19];
        const float Q1x = xxx * u0 * u0 + xyy * u1 * u1 + xzz * u2 * u2 + 2.f * (xxy * u0 * u1 + xxz * u0 * u2 + xyz * u1 * u2);
        const float Q1y = xxy * u0 * u0 + yyy * u1 * u1 + yzz * u2 * u2 + 2.f * (xyy * u0 * u1 + xyz * u0 * u2 + yyz * u1 * u2);
        const float Q1z = xxz * u0 * u0 + yyz * u1 * u1 + zzz * u2 * u2 + 2.f * (xyz * u0 * u1 + xzz * u0 * u2 + yzz * u1 * u2);
        const float Q0 = 17.5f * (Q1x * u0 + Q1y * u1 + Q1z * u2);
        hx += il * (7.5f * Q1x - Q0 * u0);
        hy += il * (7.5f * Q1y - Q0 * u1);
        hz += il * (7.5f * Q1z - Q0 * u2);
    }
    a[0] += w * (M * u0 + w * hx);
    a[1] += w * (M * u1 + w * hy);
    a[2] += w * (M * u2 + w * hz);
}

// add_pair<false> in FP32 on scaled coordinates (r = source - target with d2 = |r|^2, h and m scaled).
// The LUT index is clamped: an FP32 q^2 may round up to 4 where the FP64 test admitted it.
__device__ __forceinline__ void add_pair_f(const double* __restrict__ grads, float rx, float ry, float rz, float d2,
                                           float h, float m, float a[3]) {
    if (grads && d2 < 4.f * (h * h)) {
        const float hInv = __builtin_amdgcn_rcpf(h);
        const float qSqr = d2 * (hInv * hInv);
        const float fi = float(LUT_ENTRIES / 4) * qSqr;
        const uint32_t i1 = min(uint32_t(fi), uint32_t(LUT_ENTRIES - 1));
        const float ratio = fi - float(i1);
        const float gr = float(grads[i1]) * (1.f - ratio) + float(grads[i1 + 1]) * ratio;
        const float f = m * (hInv * hInv * hInv) * gr;
        a[0] += rx * f;
        a[1] += ry * f;
        a[2] += rz * f;
        return;
    }
    const float il = __builtin_amdgcn_rsqf(d2);
    const float f = m * (il * il * il);
    a[0] += rx * f;
    a[1] += ry * f;
    a[2] += rz * f;
}

// Lanes of a wavefront over m particles (or pairs of particles) of a target leaf: lane = sp * m + p, for p < m
// and split sp < S = 64 / m.  Lanes from S * m on take no entries.  (Splits of a power-of-two width would leave
// up to half the lanes idle for 17 particles; a 25-particle leaf limit makes most leaves 9-25 particles.)
struct LaneSplit {
    uint32_t m, S, p, sp;
    bool used;
};

__device__ __forceinline__ LaneSplit lane_split(uint32_t lane, uint32_t m) {
    LaneSplit l;
    l.m = m;
    l.S = __builtin_amdgcn_readfirstlane(64u / m);
    l.sp = lane / m;
    l.p = lane - l.sp * m;
    l.used = l.sp < l.S;
    return l;
}

// Sums the splits' partial accelerations into the lanes of split 0: split sp adds split sp + d for
// d = 1, 2, 4, ... when sp is a multiple of 2d.
__device__ __forceinline__ void sum_splits(const LaneSplit& l, uint32_t lane, double a[3]) {
    for (uint32_t d = 1; d < l.S; d <<= 1) {
        const int src = int(min(lane + d * l.m, 63u));
        const bool take = l.used && (l.sp & (2 * d - 1)) == 0 && l.sp + d < l.S;
        for (int c = 0; c < 3; ++c) {
            const double v = __shfl(a[c], src, 64);
            if (take) a[c] += v;
        }
    }
}

template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) {
    const int b = __float_as_int(v);
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, false)));
}

// Largest value over the wavefront, all lanes active (row shifts by 1, 2, 4, 8, then the row broadcasts: the
// last lane holds it).
__device__ __forceinline__ float wave_max_f(float v) {
    v = dpp_max<0x111>(v);
    v = dpp_max<0x112>(v);
    v = dpp_max<0x114>(v);
    v = dpp_max<0x118>(v);
    v = dpp_max<0x142>(v);
    v = dpp_max<0x143>(v);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Powers of two that bring lengths and G m into FP32's comfortable range: lengths are divided by
// 2^e with the root box extent in [2^(e-1), 2^e), G m by 2^f with the total G m in [2^(f-1), 2^f).
// Both divisions are exact in FP64; the results are scaled back by 2^(f - 2e).
struct EvalScale {
    double invL, invM, back;
};

// A wave-uniform double kept in scalar registers.
__device__ __forceinline__ double uniform_d(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(b)), hi = __builtin_amdgcn_readfirstlane(uint32_t(b >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

__device__ __forceinline__ EvalScale eval_scale(const Tree& t) {
    EvalScale sc{ 1.0, 1.0, 1.0 };
    if (t.n < 2) return sc;
    const double4 lo = t.lo[0], hi = t.hi[0];
    const double ext = fmax(fmax(hi.x - lo.x, hi.y - lo.y), hi.z - lo.z);
    int e = 0, f = 0;
    if (ext > 0.0) (void)frexp(ext, &e);
    const double M = t.mom[0].M;
    if (M > 0.0) (void)frexp(M, &f);
    sc.invL = uniform_d(ldexp(1.0, -e));
    sc.invM = uniform_d(ldexp(1.0, -f));
    sc.back = uniform_d(ldexp(1.0, f - 2 * e));
    return sc;
}

// The walk (BarnesHut::evalNode, BarnesHut.cpp:212-312) for groups of up to WALK_GROUP neighbouring targets, whose
// lists are mostly the same nodes.  The group's list holds, in depth-first order, the nodes that any of its
// targets takes: .x the node, .y the targets that approximate it (bit g for target g of the group) and, in the
// high half, those that sum its particles.  A target's own list is the entries with its bit.
constexpr uint32_t WALK_GROUP = 16;
// Stack items: a node to be classified for the targets .y, or (WALK_KNOWN) an entry of the list that waits for the
// nodes before it.  Node ids take 31 bits: the tree of 2^30 particles would fill 600 GB.
constexpr uint32_t WALK_KNOWN = 0x80000000u;
// A step takes up to 64 items from the top and puts back at most two more than each; the last WALK_DFS slots are
// for single-item steps only, whose growth is bounded by the depth of the tree.
constexpr uint32_t WALK_STACK = 768, WALK_DFS = 256;
static_assert(WALK_DFS > 2 * (MAX_DEPTH + 1), "a depth-first walk fits the reserve");

struct alignas(16) WalkStage {
    uint2 stack[WALK_STACK];
    float4 box_a[WALK_GROUP];  // lo x, y, z and hi x of the targets' boxes in the records' frame
    float4 box_b[WALK_GROUP];  // hi y, z and the first particle (bits)
};

// The opening test of target id (first particle f) on node `node` in FP64.
__device__ __forceinline__ bool overlaps_exact(const Tree& t, uint32_t id, uint32_t f, uint32_t node) {
    double lo[3], hi[3];
    target_box(t, id, f, lo, hi);
    return ball_overlaps_box(t.geo[node], lo, hi);
}

// One wavefront per group.  Each lane classifies one node for every target of the group: a node that contains
// the target is opened (or, when it is the target itself, dropped: its own pairs are summed apart); a node
// without opening ball (coincident particles) is summed when it is a leaf and opened otherwise, as its expansion
// is singular; a node whose ball does not overlap the target's box is approximated; an overlapping leaf is
// summed; others are opened.  A step takes the next 64 items in depth-first order, emits those before the first
// opened node, and puts the others back with each opened node replaced by its children.
//
// With one lane per target instead (each lane its own chain of dependent node loads, 36 cache lines per load
// instruction) the walk of 8M particles took 5.0 ms and of 20k particles 0.78 ms; this walk takes 1.7 ms
// and 40 us, bound by instruction issue: about 24 instructions per node and target, while the group shares the
// node's load and the stack's bookkeeping.
//
// With `screen` the opening test runs in FP32 on the records: with offsets within [-1/2, 1/2], the rounding of
// the box, the centre and r_open moves S = |box - centre|^2 by at most 7 delta sqrt(S) (delta = 2^-24) and the
// FP32 arithmetic adds a few ulps of Q = r_open^2 + S, so that |r_open^2 - S| > 1e-6 sqrt(Q) + 2e-6 Q (16 delta =
// 9.5e-7) decides.  The band is taken per node as 2e-6 r_open + 8e-6 r_open^2 + 1e-10: for S <= 3 r_open^2 it
// is at least that, and beyond, |r_open^2 - S| > 1e-10 alone implies it.  Within the band, and without
// `screen`, the FP64 test decides, so the lists are those of the FP64 test alone.
__global__ void __launch_bounds__(BLOCK) k_walk(Tree t, const uint32_t* __restrict__ targets, uint32_t ntargets,
                                                uint32_t group, int screen, uint2* __restrict__ list, uint32_t cap,
                                                uint32_t* __restrict__ list_count, uint32_t* need) {
    __shared__ WalkStage stages[BLOCK / 64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    WalkStage& S_ = stages[wave];
    // each XCD takes one contiguous range of the (Morton-ordered) targets, so the nodes that neighbouring
    // groups share stay in its L2
    const uint32_t grp = xcd_block(blockIdx.x, gridDim.x) * (BLOCK / 64) + wave;
    const uint32_t q0 = grp * group;
    if (q0 >= ntargets) return;  // uniform over the wavefront
    const uint32_t gc = min(group, ntargets - q0);
    if (lane < gc) {
        const uint32_t id = targets[q0 + lane];
        uint32_t f, c;
        node_range(t, id, f, c);
        double lo[3], hi[3];
        target_box(t, id, f, lo, hi);
        float b[6];
        for (int k = 0; k < 3; ++k) {
            b[k] = float((lo[k] - t.ctr[k]) * t.invL);
            b[3 + k] = float((hi[k] - t.ctr[k]) * t.invL);
        }
        S_.box_a[lane] = make_float4(b[0], b[1], b[2], b[3]);
        S_.box_b[lane] = make_float4(b[4], b[5], __uint_as_float(f), 0.f);
    }
    if (lane == 0) S_.stack[0] = make_uint2(0u, (1u << gc) - 1u);  // the root: internal node 0, or particle 0
    wave_sync();
    uint2* out = list + size_t(grp) * cap;
    const unsigned long long below = (1ull << lane) - 1ull;
    uint32_t size = 1, cnt = 0;
    for (uint32_t steps = 0; size > 0; ++steps) {
        if (steps > 3u * t.n) {  // every step emits, drops or opens the first of its items
            if (lane == 0) atomicOr(t.error, 2u);
            break;
        }
        const uint32_t room = size + WALK_DFS < WALK_STACK ? (WALK_STACK - WALK_DFS - size) / 2u : 0u;
        const uint32_t take = min(min(64u, size), max(room, 1u));
        uint32_t id = 0, left = 0, right = 0, approx = 0, sum = 0, open = 0;
        if (lane < take) {
            const uint2 item = S_.stack[size - 1u - lane];
            id = item.x & ~WALK_KNOWN;
            const uint32_t active = item.y;
            if (item.x & WALK_KNOWN) {
                approx = active & 0xffffu;
                sum = active >> 16;
            } else {
                WalkNodeF w;
                if (is_particle(t, id)) {
                    // a single particle has r_open = 0: always summed pair by pair (BarnesHut.cpp:237-243)
                    w.geo = make_float4(0.f, 0.f, 0.f, 0.f);
                    w.first = id - (t.n - 1);
                    w.count = 1u | WALK_ZERO_R;
                    w.left = w.right = 0u;
                } else {
                    w = t.wnf[id];
                }
                const uint32_t count = w.count & ~WALK_ZERO_R;
                const float R2 = w.geo.w * w.geo.w;
                const float band = 2e-6f * w.geo.w + 8e-6f * R2 + 1e-10f;
                uint32_t near = 0, unsure = 0, own = 0;
                for (uint32_t g = 0; g < gc; ++g) {
                    const float4 a = S_.box_a[g], b = S_.box_b[g];
                    const float dx = fmaxf(fmaxf(a.x - w.geo.x, w.geo.x - a.w), 0.f);
                    const float dy = fmaxf(fmaxf(a.y - w.geo.y, w.geo.y - b.x), 0.f);
                    const float dz = fmaxf(fmaxf(a.z - w.geo.z, w.geo.z - b.y), 0.f);
                    const float m = R2 - (dx * dx + dy * dy + dz * dz);
                    const uint32_t bit = 1u << g;
                    if (m > 0.f) near |= bit;
                    if (!(fabsf(m) > band)) unsure |= bit;
                    if (__float_as_uint(b.z) - w.first < count) own |= bit;  // the node contains the target
                }
                if (!screen) unsure = ~0u;
                if (w.count & WALK_ZERO_R) {
                    near = ~0u;
                    unsure = 0u;
                }
                for (uint32_t u = unsure & active & ~own; u != 0u; u &= u - 1u) {
                    const uint32_t g = uint32_t(__builtin_ctz(u));
                    const bool o = overlaps_exact(t, targets[q0 + g], __float_as_uint(S_.box_b[g].z), id);
                    near = o ? near | (1u << g) : near & ~(1u << g);
                }
                near |= own;
                approx = active & ~near;
                if (count <= t.leaf) {
                    sum = active & near & ~own;
                } else {
                    open = active & near;
                }
                left = w.left;
                right = w.right;
            }
        }
        const bool entry = (approx | sum) != 0u;
        const unsigned long long om = __ballot(open != 0u), em = __ballot(entry);
        // emitted now: the entries up to and with the first opened node (an entry comes before its children)
        const unsigned long long head = om ? om ^ (om - 1ull) : ~0ull;
        if (((em & head) >> lane) & 1ull) {
            const uint32_t at = cnt + __popcll(em & head & below);
            if (at < cap) out[at] = make_uint2(id, approx | (sum << 16));
        }
        cnt += __popcll(em & head);
        // the others go back in order, the top first
        const unsigned long long back = em & ~head;
        size += __popcll(back) + 2u * __popcll(om) - take;
        uint32_t at = size - 1u - (__popcll(back & below) + 2u * __popcll(om & below));
        if ((back >> lane) & 1ull) S_.stack[at--] = make_uint2(id | WALK_KNOWN, approx | (sum << 16));
        if (open) {
            S_.stack[at] = make_uint2(left, open);
            S_.stack[at - 1u] = make_uint2(right, open);
        }
        wave_sync();
    }
    if (lane == 0) {
        list_count[grp] = cnt;
        if (cnt > cap) atomicMax(need, cnt);
    }
}

// A wavefront's LDS: 64 staged nodes or source particles, and the node ids and particle positions collected so
// far (fewer than 64 from before, and up to 64 more from one step or one leaf).
template <typename T, int ORDER>
struct alignas(16) EvalStage {
    struct alignas(16) Src {
        T x, y, z, m;
    };
    union {
        NodeRow<T, ORDER> row[64];
        struct {
            Src src[64];
            T h[64];
            uint32_t idx[64];
        };
    };
    uint32_t nodes[128];
    uint32_t parts[128];
};

// The lists of the groups of targets (k_walk).
struct WalkLists {
    const uint2* list;
    const uint32_t* count;
    uint32_t cap, group;
};

// Interaction counts per target (null: not wanted).
struct EvalCounts {
    uint32_t *nodes, *leaves, *work;
};

// The wavefronts' sums of a shared target (mine: 3 doubles per particle in the wavefront's own stage), added in
// order by the first wavefront to the accelerations of the target's particles.
template <typename Stage>
__device__ __forceinline__ void add_shared(const Planes& s, const uint32_t* __restrict__ order, const Stage* stages,
                                           uint32_t split, uint32_t wave, uint32_t lane, uint32_t tf, uint32_t tc,
                                           double back) {
    static_assert(sizeof(Stage) >= 64 * 3 * sizeof(double), "the stage holds a leaf's sums");
    __syncthreads();
    if (wave != 0 || lane >= tc) return;
    double v[3] = { 0.0, 0.0, 0.0 };
    for (uint32_t w = 0; w < split; ++w) {
        const double* from = reinterpret_cast<const double*>(stages + w);
        for (int c = 0; c < 3; ++c) v[c] += from[3 * lane + c];
    }
    const uint32_t i = order[tf + lane];
    s.d[GAX][i] += v[0] * back;
    s.d[GAY][i] += v[1] * back;
    s.d[GAZ][i] += v[2] * back;
}

// The sums of a target's list in FP64, one target per wavefront (split = 1) or per block (split = the block's
// wavefronts), added to the accelerations in the state planes.  The group's list is scanned 64 entries at a time;
// the target's nodes and the particles of its leaves are collected in LDS, staged by batches and summed.  With
// split > 1 every wavefront of the block scans alike and evaluates every split-th batch.
//
// A lane holds two particles of the target, p and p + m with m = ceil(tc / 2).  That halves the LDS reads of the
// staged entries, which take as long as the arithmetic of one, and fills the wavefront better (17 particles: 63
// lanes of 9 x 7, against 51 of 17 x 3).  A batch is B = S floor(64 / S) entries, so that each of the S splits of
// the wavefront takes the same number.  One comparison against the batch's largest softening radius sends a pair
// to the branch that handles softening and the particle itself; the others are Newtonian.
// WIDE: the tree's box is so wide that squared distances can overflow; the others save the test of it (2 % of the N-body
// step of 1M particles).
template <int ORDER, bool WIDE>
__global__ void __launch_bounds__(BLOCK) k_eval(Tree t, Planes s, const uint32_t* __restrict__ order,
                                                const uint32_t* __restrict__ targets, uint32_t ntargets, WalkLists wl,
                                                uint32_t split, EvalCounts counts, const double* __restrict__ grads) {
    using Stage = EvalStage<double, ORDER>;
    __shared__ Stage stages[BLOCK / 64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    Stage& S_ = stages[wave];
    const uint32_t block = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t q = split > 1 ? block : block * (BLOCK / 64) + wave;
    const uint32_t part = split > 1 ? wave : 0u;
    if (q >= ntargets) return;  // uniform over the wavefront, and over the block when it shares a target
    uint32_t tf, tc;
    node_range(t, targets[q], tf, tc);
    const LaneSplit ls = lane_split(lane, (tc + 1) / 2);
    const uint32_t S = ls.S, B = __builtin_amdgcn_readfirstlane(S * (64u / S));
    const uint32_t j0 = ls.used ? ls.sp : 64u;  // unused lanes take no entries
    const bool two = ls.p + ls.m < tc;
    const uint32_t k0 = tf + ls.p, k1 = two ? k0 + ls.m : k0;
    const double4 me0 = t.pos[k0], me1 = t.pos[k1];
    const float hmax = wave_max_f(ls.used ? fmaxf(float(me0.w), float(me1.w)) * 1.000001f : 0.f);  // rounded up
    double a0[3] = { 0.0, 0.0, 0.0 }, a1[3] = { 0.0, 0.0, 0.0 };
    const unsigned long long below = (1ull << lane) - 1ull;
    const uint32_t grp = q / wl.group, abit = 1u << (q - grp * wl.group), sbit = abit << 16;
    const uint2* list = wl.list + size_t(grp) * wl.cap;
    const uint32_t entries = wl.count[grp];
    uint32_t at = 0, nfill = 0, pfill = 0;     // scanned entries, collected nodes, collected particles
    uint32_t nbatch = 0, pbatch = 0;           // batches so far
    uint32_t ncnt = 0, xcnt = 0, xsum = 0;
    // leaves whose particles are still to be collected: range (ef, ec) in the lanes of `em`; first the target
    uint32_t ef = tf, ec = tc;
    unsigned long long em = 1ull;
    for (;;) {
        while (em != 0ull && pfill < B) {
            const int l = __builtin_ctzll(em);
            em &= em - 1ull;
            const uint32_t f = __builtin_amdgcn_readlane(ef, l), c = __builtin_amdgcn_readlane(ec, l);
            if (lane < c) S_.parts[pfill + lane] = f + lane;
            pfill += c;
            xsum += c;
        }
        wave_sync();
        if (at < entries && em == 0ull && nfill < B && pfill < B) {
            const uint2 e = at + lane < entries ? list[at + lane] : make_uint2(0u, 0u);
            at += 64u;
            const unsigned long long am = __ballot((e.y & abit) != 0u);
            em = __ballot((e.y & sbit) != 0u);
            if (e.y & abit) S_.nodes[nfill + __popcll(am & below)] = e.x;
            nfill += __popcll(am);
            if (e.y & sbit) node_range(t, e.x, ef, ec);
            ncnt += __popcll(am);
            xcnt += __popcll(em);
            continue;
        }
        if (nfill >= B || (at >= entries && nfill > 0)) {
            const uint32_t cnt = min(nfill, B);
            nfill -= cnt;
            if (nbatch++ % split == part) {
                if (lane < cnt) {
                    const uint32_t id = S_.nodes[nfill + lane];
                    const double4 g = t.geo[id];
                    const NodeMom& mm = t.mom[id];
                    NodeRow<double, ORDER> r;
                    r.v[0] = g.x;
                    r.v[1] = g.y;
                    r.v[2] = g.z;
                    r.v[3] = mm.M;
                    row_moments<double, ORDER>(r, mm, -3.0, 7.5);
                    S_.row[lane] = r;
                }
                wave_sync();
                for (uint32_t j = j0; j < cnt; j += S) {
                    const NodeRow<double, ORDER> r = S_.row[j];
                    expand<ORDER, WIDE>(r, me0.x, me0.y, me0.z, a0);
                    expand<ORDER, WIDE>(r, me1.x, me1.y, me1.z, a1);
                }
                wave_sync();
            }
        }
        const bool last = at >= entries && em == 0ull;
        if (pfill >= B || (last && pfill > 0)) {
            const uint32_t cnt = min(pfill, B);
            pfill -= cnt;
            if (pbatch++ % split == part) {
                float reach = 0.f;
                if (lane < cnt) {
                    const uint32_t src = S_.parts[pfill + lane];
                    const double4 o = t.pos[src];
                    S_.src[lane] = { o.x, o.y, o.z, t.gm[src] };
                    S_.h[lane] = o.w;
                    S_.idx[lane] = src;
                    reach = float(o.w);
                }
                wave_sync();
                // pairs beyond `far` are Newtonian: farther than (h_i + h_j), the support of the softened kernel at
                // the mean h, for the largest h of the batch and of the targets (0 for point particles)
                double far = 0.0;
                if (grads) {
                    const double r = double(wave_max_f(reach) * 1.000001f + hmax);
                    far = r * r;
                }
                auto pair = [&](uint32_t j, uint32_t k, const typename Stage::Src& o, const double4& me, double* a) {
                    const double rx = o.x - me.x, ry = o.y - me.y, rz = o.z - me.z;
                    const double d2 = rx * rx + ry * ry + rz * rz;
                    if (d2 <= far) {
                        if (S_.idx[j] != k) add_pair<false>(grads, rx, ry, rz, 0.5 * (S_.h[j] + me.w), o.m, a);
                    } else {
                        const double il = rsqrt_step<WIDE>(d2);
                        const double f = (o.m * il) * (il * il);
                        a[0] += rx * f;
                        a[1] += ry * f;
                        a[2] += rz * f;
                    }
                };
                for (uint32_t j = j0; j < cnt; j += S) {
                    const typename Stage::Src o = S_.src[j];
                    pair(j, k0, o, me0, a0);
                    pair(j, k1, o, me1, a1);
                }
                wave_sync();
            }
        }
        if (last && nfill == 0 && pfill == 0) break;
    }
    sum_splits(ls, lane, a0);
    sum_splits(ls, lane, a1);
    if (counts.nodes && lane == 0 && part == 0) {
        counts.nodes[q] = ncnt;
        counts.leaves[q] = xcnt;
        counts.work[2 * size_t(q)] = tc * ncnt;            // particle-node expansions
        counts.work[2 * size_t(q) + 1] = tc * (xsum - 1);  // particle pairs (xsum with the target's own)
    }
    const bool writes = ls.used && ls.sp == 0;
    if (split > 1) {
        double* mine = reinterpret_cast<double*>(&S_);
        for (int c = 0; c < 3; ++c) {
            if (writes) mine[3 * ls.p + c] = a0[c];
            if (writes && two) mine[3 * (ls.p + ls.m) + c] = a1[c];
        }
        add_shared(s, order, stages, split, wave, lane, tf, tc, 1.0);
        return;
    }
    if (writes) {
        const uint32_t i = order[k0];
        s.d[GAX][i] += a0[0];
        s.d[GAY][i] += a0[1];
        s.d[GAZ][i] += a0[2];
        if (two) {
            const uint32_t i2 = order[k1];
            s.d[GAX][i2] += a1[0];
            s.d[GAY][i2] += a1[1];
            s.d[GAZ][i2] += a1[2];
        }
    }
}

// The sums with FP32 terms: offsets from the target leaf's first particle R, lengths and G m scaled by
// eval_scale.  A pair separation taken as the difference of two FP32 offsets is off by at most 2^-23 O, with O
// the largest offset among the batch's sources and the wavefront's targets: pairs closer than O / 8 (where that
// is more than 1e-6 of the separation) take theirs in FP64 from the source's FP64 position instead.  Each batch
// of up to 64 entries is summed in FP32 and added to FP64 accumulators; the accelerations are scaled back and
// added to the state planes in FP64.
//
// The FP32 sum of a batch depends on which entries it holds, so the lists are taken in their depth-first order,
// the target's own particles last, and cut at fixed places (64 nodes; 64 leaves, and within them 64 particles),
// whatever the number of wavefronts.  lane = sp tc + p, for particle p < tc of the target and split sp < S = 64 /
// tc, which takes every S-th entry.  One comparison against the batch's softening and close radii sends a pair to
// the branch that handles softening, closeness and the particle itself; the others are Newtonian.
//
// Walk and sums of 8M particles (quadrupole, theta 0.5) take 16.6 + 1.7 ms, of which staging is 6.5 ms; before,
// with lists per target and entries read from LDS a component at a time, 17.9 + 5.1 ms.
template <int ORDER>
__global__ void __launch_bounds__(BLOCK) k_eval_mixed(Tree t, Planes s, const uint32_t* __restrict__ order,
                                                      const uint32_t* __restrict__ targets, uint32_t ntargets,
                                                      WalkLists wl, uint32_t split, EvalCounts counts,
                                                      const double* __restrict__ grads) {
    using Stage = EvalStage<float, ORDER>;
    __shared__ Stage stages[BLOCK / 64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    Stage& S_ = stages[wave];
    const uint32_t block = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t q = split > 1 ? block : block * (BLOCK / 64) + wave;
    const uint32_t part = split > 1 ? wave : 0u;
    if (q >= ntargets) return;  // uniform over the wavefront, and over the block when it shares a target
    const EvalScale sc = eval_scale(t);
    uint32_t tf, tc;
    node_range(t, targets[q], tf, tc);
    const LaneSplit ls = lane_split(lane, tc);
    const uint32_t S = ls.S;
    const uint32_t j0 = ls.used ? ls.sp : 64u;  // unused lanes take no entries
    const uint32_t k = tf + ls.p;
    const double4 R = t.pos[tf];
    float mx, my, mz, mh;
    {
        const double4 me = t.pos[k];
        mx = float((me.x - R.x) * sc.invL);
        my = float((me.y - R.y) * sc.invL);
        mz = float((me.z - R.z) * sc.invL);
        mh = float(me.w * sc.invL);
    }
    const float me2 = wave_max_f(ls.used ? mx * mx + my * my + mz * mz : 0.f);
    const float hmax = wave_max_f(ls.used ? mh * 1.000001f : 0.f);  // rounded up
    double a[3] = { 0.0, 0.0, 0.0 };
    const double s2 = sc.invM * sc.invL * sc.invL, s3 = s2 * sc.invL;
    const unsigned long long below = (1ull << lane) - 1ull;
    const uint32_t grp = q / wl.group, abit = 1u << (q - grp * wl.group), sbit = abit << 16;
    const uint2* list = wl.list + size_t(grp) * wl.cap;
    const uint32_t entries = wl.count[grp];
    uint32_t at = 0, nfill = 0, pfill = 0;  // scanned entries, collected nodes, collected particles
    uint32_t nbatch = 0, pbatch = 0;        // batches so far
    uint32_t ncnt = 0, xcnt = 0, xsum = 0;
    uint32_t leaves = 0;                    // leaves collected since the last cut
    bool own = true;                        // the target's own particles are still to come
    uint32_t ef = 0, ec = 0;                // leaves to collect: range (ef, ec) in the lanes of `em`
    unsigned long long em = 0ull;
    for (;;) {
        if (at >= entries && em == 0ull && own) {
            own = false;
            ef = tf;
            ec = tc;
            em = 1ull;
        }
        // a batch of particles is full at 64, or where 64 leaves end
        while (em != 0ull && pfill < 64u && leaves < 64u) {
            const int l = __builtin_ctzll(em);
            em &= em - 1ull;
            const uint32_t f = __builtin_amdgcn_readlane(ef, l), c = __builtin_amdgcn_readlane(ec, l);
            if (lane < c) S_.parts[pfill + lane] = f + lane;
            pfill += c;
            xsum += c;
            ++leaves;
        }
        wave_sync();
        if (at < entries && em == 0ull && nfill < 64u && pfill < 64u) {
            const uint2 e = at + lane < entries ? list[at + lane] : make_uint2(0u, 0u);
            at += 64u;
            const unsigned long long am = __ballot((e.y & abit) != 0u);
            em = __ballot((e.y & sbit) != 0u);
            if (e.y & abit) S_.nodes[nfill + __popcll(am & below)] = e.x;
            nfill += __popcll(am);
            if (e.y & sbit) node_range(t, e.x, ef, ec);
            ncnt += __popcll(am);
            xcnt += __popcll(em);
            continue;
        }
        if (nfill >= 64u || (at >= entries && nfill > 0)) {
            const uint32_t cnt = min(nfill, 64u);
            if (nbatch++ % split == part) {
                if (lane < cnt) {
                    const uint32_t id = S_.nodes[lane];
                    const double4 g = t.geo[id];
                    const NodeMom& mm = t.mom[id];
                    NodeRow<float, ORDER> r;
                    r.v[0] = float((g.x - R.x) * sc.invL);
                    r.v[1] = float((g.y - R.y) * sc.invL);
                    r.v[2] = float((g.z - R.z) * sc.invL);
                    r.v[3] = float(mm.M * sc.invM);
                    row_moments<float, ORDER>(r, mm, s2, s3);
                    S_.row[lane] = r;
                }
                wave_sync();
                float b[3] = { 0.f, 0.f, 0.f };
                for (uint32_t j = j0; j < cnt; j += S) {
                    const NodeRow<float, ORDER> r = S_.row[j];
                    expand<ORDER>(r, mx, my, mz, b);
                }
                for (int c = 0; c < 3; ++c) a[c] += double(b[c]);
            }
            // the nodes past the batch move to the front
            nfill -= cnt;
            const uint32_t rest = lane < nfill ? S_.nodes[64u + lane] : 0u;
            wave_sync();
            if (lane < nfill) S_.nodes[lane] = rest;
            wave_sync();
        }
        const bool last = at >= entries && em == 0ull && !own;
        if (pfill >= 64u || (pfill > 0 && (leaves == 64u || last))) {
            const uint32_t cnt = min(pfill, 64u);
            if (pbatch++ % split == part) {
                float reach = 0.f, o2 = 0.f;
                if (lane < cnt) {
                    const uint32_t src = S_.parts[lane];
                    const double4 o = t.pos[src];
                    typename Stage::Src v;
                    v.x = float((o.x - R.x) * sc.invL);
                    v.y = float((o.y - R.y) * sc.invL);
                    v.z = float((o.z - R.z) * sc.invL);
                    v.m = float(t.gm[src] * sc.invM);
                    reach = float(o.w * sc.invL);
                    S_.src[lane] = v;
                    S_.h[lane] = reach;
                    S_.idx[lane] = src;
                    o2 = v.x * v.x + v.y * v.y + v.z * v.z;
                }
                wave_sync();
                const float close = fmaxf(wave_max_f(o2), me2) * (1.f / 64.f);  // (O / 8)^2
                // pairs beyond `far` are Newtonian and not close: (h_i + h_j) is the support of the softened
                // kernel at the mean h
                const float rs = grads ? wave_max_f(reach) * 1.000001f + hmax : 0.f;
                const float far = fmaxf(rs * rs, close);
                float b[3] = { 0.f, 0.f, 0.f };
                for (uint32_t j = j0; j < cnt; j += S) {
                    const typename Stage::Src o = S_.src[j];
                    float rx = o.x - mx, ry = o.y - my, rz = o.z - mz;
                    float d2 = rx * rx + ry * ry + rz * rz;
                    if (d2 <= far) {
                        const uint32_t src = S_.idx[j];
                        if (src == k) continue;
                        if (d2 < close || d2 == 0.f) {
                            const double4 od = t.pos[src], me = t.pos[k];
                            rx = float((od.x - me.x) * sc.invL);
                            ry = float((od.y - me.y) * sc.invL);
                            rz = float((od.z - me.z) * sc.invL);
                            d2 = rx * rx + ry * ry + rz * rz;
                        }
                        add_pair_f(grads, rx, ry, rz, d2, 0.5f * (S_.h[j] + mh), o.m, b);
                    } else {
                        const float il = __builtin_amdgcn_rsqf(d2);
                        const float f = o.m * (il * il * il);
                        b[0] += rx * f;
                        b[1] += ry * f;
                        b[2] += rz * f;
                    }
                }
                for (int c = 0; c < 3; ++c) a[c] += double(b[c]);
            }
            // the particles past the batch move to the front
            pfill -= cnt;
            const uint32_t rest = lane < pfill ? S_.parts[64u + lane] : 0u;
            wave_sync();
            if (lane < pfill) S_.parts[lane] = rest;
            wave_sync();
        }
        if (leaves == 64u && pfill == 0) leaves = 0;
        if (last && nfill == 0 && pfill == 0) break;
    }
    sum_splits(ls, lane, a);
    if (counts.nodes && lane == 0 && part == 0) {
        counts.nodes[q] = ncnt;
        counts.leaves[q] = xcnt;
        counts.work[2 * size_t(q)] = tc * ncnt;            // particle-node expansions
        counts.work[2 * size_t(q) + 1] = tc * (xsum - 1);  // particle pairs (xsum with the target's own)
    }
    const bool writes = ls.used && ls.sp == 0;
    if (split > 1) {
        double* mine = reinterpret_cast<double*>(&S_);
        for (int c = 0; c < 3; ++c) {
            if (writes) mine[3 * ls.p + c] = a[c];
        }
        add_shared(s, order, stages, split, wave, lane, tf, tc, sc.back);
        return;
    }
    if (writes) {
        const uint32_t i = order[k];
        s.d[GAX][i] += a[0] * sc.back;
        s.d[GAY][i] += a[1] * sc.back;
        s.d[GAZ][i] += a[2] * sc.back;
    }
}

// BarnesHut::evalImpl (BarnesHut.cpp:136-178) at arbitrary points: a node is approximated when the point
// lies outside its box and size^2 / (distance^2 + EPS) < theta^2; leaves are summed with the unsymmetrised
// kernel of the source particle.
__global__ void __launch_bounds__(BLOCK) k_points(Tree t, const double4* __restrict__ pts, double4* __restrict__ acc,
                                                  size_t np, const double* __restrict__ grads, int order_m) {
    const size_t q = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= np) return;
    const double4 r0 = pts[q];
    double a[3] = { 0.0, 0.0, 0.0 };
    const double th2 = 1.0 / (t.thetaInv * t.thetaInv);
    uint32_t id = 0;
    for (size_t visits = 0; id != END; ++visits) {
        if (visits > 2 * size_t(t.n)) {
            atomicOr(t.error, 2u);
            break;
        }
        uint32_t f, c;
        node_range(t, id, f, c);
        if (!is_particle(t, id)) {
            const double4 lo = t.lo[id], hi = t.hi[id], g = t.geo[id];
            const bool inside = !(r0.x < lo.x || r0.x > hi.x || r0.y < lo.y || r0.y > hi.y || r0.z < lo.z || r0.z > hi.z);
            const double sx = hi.x - lo.x, sy = hi.y - lo.y, sz = hi.z - lo.z;
            const double cx = 0.5 * (lo.x + hi.x) - r0.x, cy = 0.5 * (lo.y + hi.y) - r0.y, cz = 0.5 * (lo.z + hi.z) - r0.z;
            const double size2 = sx * sx + sy * sy + sz * sz;
            const double dist2 = cx * cx + cy * cy + cz * cz;
            if (!inside && size2 > 0.0 && size2 / (dist2 + EPS_D) < th2) {
                add_multipole(t.mom[id], r0.x - g.x, r0.y - g.y, r0.z - g.z, order_m, a);
                id = t.skip[id];
                continue;
            }
            if (c > t.leaf) {
                id = t.left[id];
                continue;
            }
        }
        // BarnesHut::evalExact (BarnesHut.cpp:376-387)
        for (uint32_t j = f; j < f + c; ++j) {
            const double4 o = t.pos[j];
            add_pair<false>(grads, o.x - r0.x, o.y - r0.y, o.z - r0.z, o.w, t.gm[j], a);
        }
        id = t.skip[id];
    }
    acc[q] = make_double4(a[0], a[1], a[2], 0.0);
}

// The term of one source in the direct sum, with the bits of add_pair<true> on a sum of zero.  That form takes 1 / h, a
// square root and three quotients (about 90 instructions).  Most pairs are far outside the softening and of ordinary
// size, and take a form with the same roundings in about 45: the branch decided on |r|^2 against 4 h^2 with room for
// every rounding of the quotient it replaces, the square root and the quotients by Goldschmidt's iteration from one
// reciprocal square root, each corrected by its exact remainder (Markstein 1990).  False where the bounds that keep
// the remainders exact do not hold (also for NaN); t is then not to be used.
template <bool M4>
__device__ __forceinline__ bool far_term(double rx, double ry, double rz, double h, double m, double t[3]) {
#pragma clang fp contract(off)
    const double d2 = rx * rx + ry * ry + rz * rz;
    const double least = fmin(fmin(fabs(rx), fabs(ry)), fabs(rz));
    const double y = __builtin_amdgcn_rsq(d2);
    double l = d2 * y, u = 0.5 * y;
    const double e = fma(-u, l, 0.5);
    l = fma(l, e, l);
    u = fma(u, e, u);
    l = fma(fma(-l, l, d2), u, l);
    l = fma(fma(-l, l, d2), u, l);
    const double l3 = l * l * l;
    const double u2 = u + u;
    double il3 = u2 * u2 * u2;
    il3 = fma(fma(-l3, il3, 1.0), il3, il3);
    const double qx = rx * il3, qy = ry * il3, qz = rz * il3;
    t[0] = m * fma(fma(-l3, qx, rx), il3, qx);
    t[1] = m * fma(fma(-l3, qy, ry), il3, qy);
    t[2] = m * fma(fma(-l3, qz, rz), il3, qz);
    // (bitwise: no branches between the conditions)
    return bool(int(d2 >= 1.e-100) & int(d2 <= 1.e100) & int(least >= 1.e-140) &
                int(!M4 || d2 > (4.0 * (1.0 + 1.e-12)) * (h * h)));
}

// BruteForceGravity::evalImpl (BruteForceGravity.h:112-131) for targets tg[0..nt): sources in storage order, each
// target's sum in source order like the reference's two loops.  One lane per target left most of the chip idle up to
// some 100k targets, so DIRECT_WAVES wavefronts share DIRECT_TARGETS targets: each puts the terms of DIRECT_SUB * 4
// sources of a chunk into LDS, and one lane per target and component adds the chunk in order while the others are at
// the next one (two buffers, one barrier per chunk; that chain has the higher wave priority).  A term of zero (the
// target itself, sources past the end) leaves a sum that started at +0 as it is.  Issue-bound, 75 instructions a
// term; few targets per block keep the last wave of blocks short.  n targets and sources, M4, before -> now:
// 500 174 -> 13 us, 3000 1039 -> 51, 12345 4245 -> 534, 30000 10355 -> 2472 (364 G terms/s).  32 targets per block:
// 17, 81, 539, 2413 us; 64: 26, 131, 547, 2508; 8 sources a wavefront per chunk: 735 us at 12345; sources gathered from
// the planes instead of LDS: 656; the general form for every pair: 612.  These are random places: on a lattice many
// separations have a component that is exactly 0, which far_term leaves to the general form, and wavefronts run both:
// a close-packed sphere of 3182 / 13788 / 31925 takes 85 / 970 / 3933 us, 1.5 times as long for its pairs.
constexpr int DIRECT_TARGETS = 16, DIRECT_WAVES = 8, DIRECT_SUB = 2;

template <bool M4>
__global__ void __launch_bounds__(DIRECT_WAVES * 64) k_direct(Planes s, size_t n, const uint32_t* __restrict__ tg,
                                                               size_t nt, const double* __restrict__ grads, double G,
                                                               double4* __restrict__ out) {
#pragma clang fp contract(off)
    constexpr int T = DIRECT_TARGETS, W = DIRECT_WAVES, SUB = DIRECT_SUB;
    constexpr uint32_t PER = 64 / T;            // sources of a wavefront's instruction
    constexpr uint32_t CHUNK = W * SUB * PER;   // sources of a chunk
    constexpr uint32_t PLANES = M4 ? 5 : 4;
    constexpr uint32_t LOADS = (PLANES * CHUNK + W * 64 - 1) / (W * 64);
    static_assert(3 * T <= W * 64 && T <= W * 64, "a thread for every target and component");
    __shared__ double term[2][CHUNK][3 * T];           // 48 KB
    __shared__ __align__(16) double src[2][CHUNK][6];  // x y z m h
    const uint32_t q = threadIdx.x % T, k0 = threadIdx.x / 64 * (SUB * PER) + threadIdx.x % 64 / T;
    const size_t qt = size_t(blockIdx.x) * T + q;
    const uint32_t i = tg[qt < nt ? qt : nt - 1];
    const double xi = s.d[GX][i], yi = s.d[GY][i], zi = s.d[GZ][i], hi = s.d[GH][i];
    // the planes of a source in the order of src, and this thread's elements of a chunk
    const double* lp[LOADS];
    uint32_t lk[LOADS];
    for (uint32_t v = 0; v < LOADS; ++v) {
        const uint32_t e = threadIdx.x + v * (W * 64), c = e / CHUNK;
        lp[v] = c == 0 ? s.d[GX] : c == 1 ? s.d[GY] : c == 2 ? s.d[GZ] : c == 3 ? s.d[GM] : s.d[GH];
        lk[v] = e % CHUNK;
    }
    auto fetch = [&](size_t base, double (&r)[LOADS]) {
        for (uint32_t v = 0; v < LOADS; ++v) {
            const size_t j = base + lk[v];
            r[v] = lp[v][j < n ? j : n - 1];
        }
    };
    auto place = [&](int buf, const double (&r)[LOADS]) {
        for (uint32_t v = 0; v < LOADS; ++v) {
            const uint32_t e = threadIdx.x + v * (W * 64);
            if (e < PLANES * CHUNK) src[buf][lk[v]][e / CHUNK] = r[v];
        }
    };
    double a = 0.0, next[LOADS];
    fetch(0, next);
    place(0, next);
    __syncthreads();
    int buf = 0;
    for (size_t base = 0; base < n; base += CHUNK, buf ^= 1) {
        const uint32_t left = uint32_t(n - base < CHUNK ? n - base : CHUNK);
        const uint32_t self = i - uint32_t(base);
        fetch(base + CHUNK, next);
        double rx[SUB], ry[SUB], rz[SUB], h[SUB], m[SUB], t[SUB][3];
        bool far[SUB];
#pragma unroll
        for (int v = 0; v < SUB; ++v) {
            const double* o = src[buf][k0 + v * PER];
            rx[v] = o[0] - xi;
            ry[v] = o[1] - yi;
            rz[v] = o[2] - zi;
            m[v] = o[3];
            if (M4) h[v] = 0.5 * (o[4] + hi);
        }
#pragma unroll
        for (int v = 0; v < SUB; ++v) far[v] = far_term<M4>(rx[v], ry[v], rz[v], M4 ? h[v] : 0.0, m[v], t[v]);
#pragma unroll
        for (int v = 0; v < SUB; ++v) {
            const uint32_t k = k0 + v * PER;
            if (!far[v] || k >= left || k == self) {
                for (int c = 0; c < 3; ++c) t[v][c] = 0.0;
                if (k < left && k != self) {
                    add_pair<true>(M4 ? grads : nullptr, rx[v], ry[v], rz[v], M4 ? h[v] : 0.0, m[v], t[v]);
                }
            }
            for (int c = 0; c < 3; ++c) term[buf][k][c * T + q] = t[v][c];
        }
        place(buf ^ 1, next);
        __syncthreads();
        if (threadIdx.x < 3 * T) {
            __builtin_amdgcn_s_setprio(2);  // the chunk's longest chain
            constexpr uint32_t B = 16;
            static_assert(CHUNK % B == 0, "whole batches");
            double now[B];
#pragma unroll
            for (uint32_t k = 0; k < B; ++k) now[k] = term[buf][k][threadIdx.x];
            for (uint32_t b = B; b < CHUNK; b += B) {
                double then[B];
#pragma unroll
                for (uint32_t k = 0; k < B; ++k) then[k] = term[buf][b + k][threadIdx.x];
#pragma unroll
                for (uint32_t k = 0; k < B; ++k) a += now[k];
#pragma unroll
                for (uint32_t k = 0; k < B; ++k) now[k] = then[k];
            }
#pragma unroll
            for (uint32_t k = 0; k < B; ++k) a += now[k];
            __builtin_amdgcn_s_setprio(0);
        }
    }
    // the three components of a target to one lane
    __syncthreads();
    if (threadIdx.x < 3 * T) term[0][0][threadIdx.x] = a;
    __syncthreads();
    if (threadIdx.x < T && qt < nt) {
        out[qt] = make_double4(G * term[0][0][q], G * term[0][0][T + q], G * term[0][0][2 * T + q], 0.0);
    }
}

// BruteForceGravity::evalEnergy (BruteForceGravity.h:103-115): per-particle sums m_i m_j value.
__global__ void __launch_bounds__(BLOCK) k_energy(Planes s, size_t n, const double* __restrict__ values,
                                                  double* __restrict__ e_out) {
#pragma clang fp contract(off)
    __shared__ double4 sp[BLOCK];
    __shared__ double sm[BLOCK];
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const bool active = i < n;
    const size_t ii = active ? i : 0;
    const double xi = s.d[GX][ii], yi = s.d[GY][ii], zi = s.d[GZ][ii], hi = s.d[GH][ii], mi = s.d[GM][ii];
    double e = 0.0;
    for (size_t base = 0; base < n; base += BLOCK) {
        const size_t j = base + threadIdx.x;
        if (j < n) {
            sp[threadIdx.x] = make_double4(s.d[GX][j], s.d[GY][j], s.d[GZ][j], s.d[GH][j]);
            sm[threadIdx.x] = s.d[GM][j];
        }
        __syncthreads();
        const size_t cnt = n - base < size_t(BLOCK) ? n - base : size_t(BLOCK);
        if (active) {
            for (size_t c = 0; c < cnt; ++c) {
                if (base + c == i) continue;
                const double4 o = sp[c];
                const double rx = xi - o.x, ry = yi - o.y, rz = zi - o.z, h = 0.5 * (hi + o.w);
                double v = 0.0;
                bool outer = true;
                if (values) {
                    // GravityLutKernel::value (GravityKernel.h:45-58)
                    const double hInv = 1.0 / h;
                    const double sx = rx * hInv, sy = ry * hInv, sz = rz * hInv;
                    const double qSqr = sx * sx + sy * sy + sz * sz;
                    if (!(qSqr + EPS_D >= 4.0)) {
                        const double fi = double(LUT_ENTRIES / 4) * qSqr;
                        const uint32_t i1 = uint32_t(fi);
                        const double ratio = fi - double(i1);
                        v = hInv * (values[i1] * (1.0 - ratio) + values[i1 + 1] * ratio);
                        outer = false;
                    }
                }
                if (outer) v = -1.0 / sqrt(rx * rx + ry * ry + rz * rz);
                e += mi * sm[c] * v;
            }
        }
        __syncthreads();
    }
    if (active) e_out[i] = e;
}

// Deterministic reductions: per-block partial sums in a fixed tree order.
template <int NV>
__device__ void block_sum(double (&v)[NV], double* __restrict__ out) {
    __shared__ double red[BLOCK / 64][NV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < NV; ++k) {
        double x = v[k];
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        if (lane == 0) red[wave][k] = x;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double x = 0.0;
        for (int w = 0; w < BLOCK / 64; ++w) x += red[w][threadIdx.x];
        out[size_t(blockIdx.x) * NV + threadIdx.x] = x;
    }
}

// Integrals (core/physics/Integrals.cpp:24-180): kinetic energy, momentum, angular momentum about the
// origin, mass-weighted position, total mass.
__global__ void __launch_bounds__(BLOCK) k_integrals(Planes s, size_t n, double* __restrict__ partial) {
    double v[11] = { 0.0 };
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
        const double m = s.d[GM][i];
        const double x = s.d[GX][i], y = s.d[GY][i], z = s.d[GZ][i];
        const double vx = s.d[GVX][i], vy = s.d[GVY][i], vz = s.d[GVZ][i];
        v[0] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
        v[1] += m * vx;
        v[2] += m * vy;
        v[3] += m * vz;
        v[4] += m * (y * vz - z * vy);
        v[5] += m * (z * vx - x * vz);
        v[6] += m * (x * vy - y * vx);
        v[7] += m * x;
        v[8] += m * y;
        v[9] += m * z;
        v[10] += m;
    }
    block_sum<11>(v, partial);
}

__global__ void __launch_bounds__(BLOCK) k_sum_partials(const double* __restrict__ partial, int nblocks, int nv,
                                                        double* __restrict__ out) {
    for (int k = threadIdx.x; k < nv; k += blockDim.x) {
        double x = 0.0;
        for (int b = 0; b < nblocks; ++b) x += partial[size_t(b) * nv + k];
        out[k] = x;
    }
}

__global__ void __launch_bounds__(BLOCK) k_sum_vector(const double* __restrict__ v, size_t n, double* __restrict__ partial) {
    double x[1] = { 0.0 };
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) x[0] += v[i];
    block_sum<1>(x, partial);
}

// LeapFrog drift (TimeStepping.cpp:356-360,382-386): r += v dt / 2 in all four lanes.
__global__ void __launch_bounds__(BLOCK) k_drift(Planes s, double dt, size_t n) {
#pragma clang fp contract(off)
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int k = 0; k < 4; ++k) s.d[GX + k][i] += s.d[GVX + k][i] * 0.5 * dt;
}

__global__ void __launch_bounds__(BLOCK) k_zero_acc(Planes s, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    s.d[GAX][i] = 0.0;
    s.d[GAY][i] = 0.0;
    s.d[GAZ][i] = 0.0;
}

// HardSphereSolver zeroes the h lanes of v and dv (NBodySolver.cpp:110-114); then the kick v += dv dt
// (TimeStepping.cpp:372-376) and the second drift.
__global__ void __launch_bounds__(BLOCK) k_kick_drift(Planes s, double dt, size_t n) {
#pragma clang fp contract(off)
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    s.d[GVH][i] = 0.0;
    for (int k = 0; k < 3; ++k) s.d[GVX + k][i] += s.d[GAX + k][i] * dt;
    for (int k = 0; k < 4; ++k) s.d[GX + k][i] += s.d[GVX + k][i] * 0.5 * dt;
}

__global__ void __launch_bounds__(BLOCK) k_fill_u32g(uint32_t* p, size_t count, uint32_t value) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += size_t(gridDim.x) * blockDim.x) {
        p[i] = value;
    }
}

// small[0..5] bounds, [6] list entries needed, [8] traversal error flags.
__global__ void k_init_bounds(unsigned long long* a) {
    const int t = threadIdx.x;
    if (t < 6) a[t] = t < 3 ? ~0ull : 0ull;
}

// Strided element layouts <-> planes.
// Host rows (the caller's order) into the planes and back; perm (slot -> caller's index) is null while
// the state is in the caller's order.
__global__ void __launch_bounds__(BLOCK) k_unstage(const unsigned char* __restrict__ st, size_t stride, int ncomp,
                                                   Planes s, int plane0, const uint32_t* __restrict__ perm, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* e = reinterpret_cast<const double*>(st + size_t(perm ? perm[i] : i) * stride);
    for (int c = 0; c < ncomp; ++c) s.d[plane0 + c][i] = e[c];
}

__global__ void __launch_bounds__(BLOCK) k_stage(unsigned char* __restrict__ st, size_t stride, int ncomp, Planes s,
                                                 int plane0, const uint32_t* __restrict__ perm, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double* e = reinterpret_cast<double*>(st + size_t(perm ? perm[i] : i) * stride);
    for (int c = 0; c < ncomp; ++c) e[c] = s.d[plane0 + c][i];
}

// ---- host-side gravity LUT ------------------------------------------------------------------------------

// GravityKernel<CubicSpline<3>>::gradImpl / valueImpl (core/sph/kernel/GravityKernel.h:82-107) sampled
// by the LutKernel<3> constructor (core/sph/kernel/Kernel.h:83-101).
#pragma STDC FP_CONTRACT OFF
double gk_value(double qSqr) {
    const double q = std::sqrt(qSqr);
    if (q < 1.0) {
        const double q4 = (q * q) * (q * q), q5 = ((q * q) * (q * q)) * q;
        return 2.0 / 3.0 * qSqr - 3.0 / 10.0 * q4 + 1.0 / 10.0 * q5 - 7.0 / 5.0;
    }
    const double q3 = q * q * q, q5 = ((q * q) * (q * q)) * q;
    return 4.0 / 3.0 * qSqr - q3 + 3.0 / 10.0 * (qSqr * qSqr) - 1.0 / 30.0 * q5 - 8.0 / 5.0 + 1.0 / (15.0 * q);
}

double gk_grad(double qSqr) {
    const double q = std::sqrt(qSqr);
    if (q == 0.0) return 4.0 / 3.0;
    if (q < 1.0) return 1.0 / q * (4.0 / 3.0 * q - 6.0 / 5.0 * (q * q * q) + 1.0 / 2.0 * (qSqr * qSqr));
    return 1.0 / q * (8.0 / 3.0 * q - 3.0 * qSqr + 6.0 / 5.0 * (q * q * q) - 1.0 / 6.0 * (qSqr * qSqr) -
                      1.0 / (15.0 * qSqr));
}

}  // namespace
}  // namespace osph

using namespace osph;

struct osph_gravity {
    osph_gravity_config cfg{};
    const void* owner = nullptr;  // the SPH context it is attached to (osph_attach_gravity), if any
    int precision = OSPH_PRECISION_FP64;  // the tree walk's arithmetic (osph_gravity_set_precision)
    hipStream_t stream = nullptr;
    size_t n = 0, cap = 0;
    double* dblock = nullptr;
    Planes s{};
    // LeapFrog steps move the state into the Morton order of the tree every reorder_period builds, so
    // that the tree's gather and the accelerations' writes run over consecutive slots.  perm maps a
    // slot to the particle's index in the caller's order and slot_of back; identity: no move since the
    // particles were set.
    double* dblock2 = nullptr;
    uint32_t *perm = nullptr, *perm2 = nullptr, *slot_of = nullptr;
    bool identity = true;
    int reorder_period = 10, since_reorder = 0;
    // tree
    uint64_t *keys = nullptr, *keys_sorted = nullptr;
    uint32_t *iota = nullptr, *order = nullptr;
    void* sort_temp = nullptr;
    size_t sort_temp_bytes = 0;
    double4* pos = nullptr;
    double* gm = nullptr;
    uint32_t *left = nullptr, *right = nullptr, *parent = nullptr, *skip = nullptr, *first = nullptr, *count = nullptr,
             *flag = nullptr;
    double4 *geo = nullptr, *lo = nullptr, *hi = nullptr;
    NodeMom* mom = nullptr;
    WalkNodeF* wnf = nullptr;
    bool skip_ready = false;  // the skip links of this tree are built (by the first evaluation at points)
    double ctr[3] = { 0.0, 0.0, 0.0 }, invL = 1.0;
    bool wide = false;  // squared distances within the root box may overflow
    int walk_screen = -1;  // 1, -1: FP32-screened opening tests, 0: FP64 tests (the same lists)
    uint32_t *leaf_at = nullptr, *targets = nullptr, *ntargets_dev = nullptr;
    void* select_temp = nullptr;
    size_t select_temp_bytes = 0;
    uint32_t ntargets = 0;
    uint2* list = nullptr;  // walk lists, list_cap entries per group of targets
    uint32_t* list_count = nullptr;
    uint32_t list_cap = 2048;
    size_t list_groups = 0;
    uint32_t* counts = nullptr;  // interaction counts per target (4 words), when statistics are asked for
    size_t counts_cap = 0;
    uint32_t* levels = nullptr;           // node counts per depth, then the bucket cursors
    unsigned long long* small = nullptr;  // [0..5] bounds, [6] list entries needed, [8] error flags
    Mailbox box;                               // host mirror of small
    unsigned long long* small_host = nullptr;  // its words
    double *lut_grads = nullptr, *lut_values = nullptr;
    double* scratch = nullptr;
    size_t scratch_cap = 0;
    unsigned char* staging = nullptr;
    size_t staging_cap = 0;
    bool built = false;
    // profiling
    bool prof = false;
    struct Ev {
        const char* name;
        hipEvent_t a, b;
    };
    std::vector<Ev> events;
    std::vector<hipEvent_t> pool;
    std::map<std::string, std::pair<double, uint64_t>> acc;
    std::string err;

    int fail(int code, const std::string& m) {
        err = m;
        return code;
    }
};

namespace {

#define GCHK(g, expr)                                                                             \
    do {                                                                                          \
        hipError_t e_ = (expr);                                                                   \
        if (e_ != hipSuccess) return (g)->fail(OSPH_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

constexpr int OK = OSPH_OK, ERR_ARG = OSPH_ERR_ARG, ERR_HIP = OSPH_ERR_HIP, ERR_STATE = OSPH_ERR_STATE;

hipEvent_t take_event(osph_gravity* g) {
    if (!g->pool.empty()) {
        hipEvent_t e = g->pool.back();
        g->pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

template <typename F>
void timed(osph_gravity* g, const char* name, F&& f) {
    if (!g->prof) {
        f();
        return;
    }
    osph_gravity::Ev ev{ name, take_event(g), take_event(g) };
    if (ev.a) (void)hipEventRecord(ev.a, g->stream);
    f();
    if (ev.b) (void)hipEventRecord(ev.b, g->stream);
    g->events.push_back(ev);
}

void resolve(osph_gravity* g) {
    for (auto& e : g->events) {
        float ms = 0.f;
        if (e.a && e.b && hipEventSynchronize(e.b) == hipSuccess && hipEventElapsedTime(&ms, e.a, e.b) == hipSuccess) {
            auto& a = g->acc[e.name];
            a.first += ms;
            a.second += 1;
        }
        if (e.a) g->pool.push_back(e.a);
        if (e.b) g->pool.push_back(e.b);
    }
    g->events.clear();
}

int sync(osph_gravity* g) {
    GCHK(g, hipStreamSynchronize(g->stream));
    GCHK(g, hipGetLastError());
    return OK;
}

// Waits for the words posted to small_host, the error flags among them, and fails if a tree climb or walk ran past its
// bound (a malformed tree) since the last check.
int check_traversal(osph_gravity* g) {
    GCHK(g, hipGetLastError());
    GCHK(g, mailbox_wait(g->stream, g->box));
    if (g->small_host[SMALL_ERROR] != 0) {
        k_fill_u32g<<<1, 64, 0, g->stream>>>(reinterpret_cast<uint32_t*>(g->small + SMALL_ERROR), 2, 0u);
        return g->fail(ERR_STATE, "tree traversal exceeded its bound");
    }
    return OK;
}

void free_particles(osph_gravity* g) {
    void* ptrs[] = { g->dblock, g->dblock2, g->perm, g->perm2, g->slot_of, g->keys, g->keys_sorted, g->iota, g->order, g->sort_temp, g->pos, g->gm, g->left,
                     g->right, g->parent, g->skip, g->first, g->count, g->flag, g->geo, g->lo, g->hi, g->mom, g->wnf,
                     g->leaf_at, g->targets, g->ntargets_dev, g->select_temp };
    for (void* p : ptrs) (void)hipFree(p);
    g->dblock = g->dblock2 = nullptr;
    g->perm = g->perm2 = g->slot_of = nullptr;
    g->identity = true;
    g->keys = g->keys_sorted = nullptr;
    g->iota = g->order = nullptr;
    g->sort_temp = g->select_temp = nullptr;
    g->pos = nullptr;
    g->gm = nullptr;
    g->left = g->right = g->parent = g->skip = g->first = g->count = g->flag = nullptr;
    g->geo = g->lo = g->hi = nullptr;
    g->mom = nullptr;
    g->wnf = nullptr;
    g->skip_ready = false;
    g->leaf_at = g->targets = g->ntargets_dev = nullptr;
    g->cap = 0;
}

int ensure_particles(osph_gravity* g, size_t n) {
    if (n <= g->cap) return OK;
    GCHK(g, hipStreamSynchronize(g->stream));
    free_particles(g);
    const size_t c = n, nodes = c > 1 ? c - 1 : 1, ids = 2 * c;
    GCHK(g, hipMalloc(&g->dblock, sizeof(double) * NGPLANES * c));
    GCHK(g, hipMalloc(&g->dblock2, sizeof(double) * NGPLANES * c));
    GCHK(g, hipMalloc(&g->perm, sizeof(uint32_t) * c));
    GCHK(g, hipMalloc(&g->perm2, sizeof(uint32_t) * c));
    GCHK(g, hipMalloc(&g->slot_of, sizeof(uint32_t) * c));
    GCHK(g, hipMalloc(&g->keys, sizeof(uint64_t) * c));
    GCHK(g, hipMalloc(&g->keys_sorted, sizeof(uint64_t) * c));
    GCHK(g, hipMalloc(&g->iota, sizeof(uint32_t) * c));
    GCHK(g, hipMalloc(&g->order, sizeof(uint32_t) * c));
    GCHK(g, hipMalloc(&g->pos, sizeof(double4) * c));
    GCHK(g, hipMalloc(&g->gm, sizeof(double) * c));
    GCHK(g, hipMalloc(&g->left, sizeof(uint32_t) * nodes));
    GCHK(g, hipMalloc(&g->right, sizeof(uint32_t) * nodes));
    GCHK(g, hipMalloc(&g->first, sizeof(uint32_t) * nodes));
    GCHK(g, hipMalloc(&g->count, sizeof(uint32_t) * nodes));
    GCHK(g, hipMalloc(&g->flag, sizeof(uint32_t) * nodes));
    GCHK(g, hipMalloc(&g->geo, sizeof(double4) * nodes));
    GCHK(g, hipMalloc(&g->lo, sizeof(double4) * nodes));
    GCHK(g, hipMalloc(&g->hi, sizeof(double4) * nodes));
    GCHK(g, hipMalloc(&g->mom, sizeof(NodeMom) * nodes));
    GCHK(g, hipMalloc(&g->wnf, sizeof(WalkNodeF) * nodes));
    GCHK(g, hipMalloc(&g->parent, sizeof(uint32_t) * ids));
    GCHK(g, hipMalloc(&g->skip, sizeof(uint32_t) * ids));
    GCHK(g, hipMalloc(&g->leaf_at, sizeof(uint32_t) * c));
    GCHK(g, hipMalloc(&g->targets, sizeof(uint32_t) * c));
    GCHK(g, hipMalloc(&g->ntargets_dev, sizeof(uint32_t)));
    size_t b1 = 0, b2 = 0;
    GCHK(g, hipcub::DeviceRadixSort::SortPairs(nullptr, b1, g->keys, g->keys_sorted, g->iota, g->order, int(c), 0, 63,
                                               g->stream));
    GCHK(g, hipcub::DeviceSelect::If(nullptr, b2, g->leaf_at, g->targets, g->ntargets_dev, int(c), NotEnd(), g->stream));
    g->sort_temp_bytes = b1;
    g->select_temp_bytes = b2;
    GCHK(g, hipMalloc(&g->sort_temp, b1 > 0 ? b1 : 1));
    GCHK(g, hipMalloc(&g->select_temp, b2 > 0 ? b2 : 1));
    for (int k = 0; k < NGPLANES; ++k) g->s.d[k] = g->dblock + size_t(k) * c;
    g->cap = c;
    return OK;
}

int ensure_staging(osph_gravity* g, size_t bytes) {
    if (bytes <= g->staging_cap) return OK;
    (void)hipFree(g->staging);
    g->staging = nullptr;
    g->staging_cap = 0;
    GCHK(g, hipMalloc(&g->staging, bytes));
    g->staging_cap = bytes;
    return OK;
}

int ensure_scratch(osph_gravity* g, size_t doubles) {
    if (doubles <= g->scratch_cap) return OK;
    (void)hipFree(g->scratch);
    g->scratch = nullptr;
    g->scratch_cap = 0;
    GCHK(g, hipMalloc(&g->scratch, doubles * sizeof(double)));
    g->scratch_cap = doubles;
    return OK;
}

int ensure_lists(osph_gravity* g, size_t groups) {
    if (groups <= g->list_groups) return OK;
    (void)hipFree(g->list);
    (void)hipFree(g->list_count);
    g->list = nullptr;
    g->list_count = nullptr;
    g->list_groups = 0;
    GCHK(g, hipMalloc(&g->list, sizeof(uint2) * groups * g->list_cap));
    GCHK(g, hipMalloc(&g->list_count, sizeof(uint32_t) * groups));
    g->list_groups = groups;
    return OK;
}

int ensure_counts(osph_gravity* g, size_t targets) {
    if (targets <= g->counts_cap) return OK;
    (void)hipFree(g->counts);
    g->counts = nullptr;
    g->counts_cap = 0;
    GCHK(g, hipMalloc(&g->counts, 4 * sizeof(uint32_t) * targets));
    g->counts_cap = targets;
    return OK;
}

Tree tree_of(osph_gravity* g) {
    Tree t{};
    t.n = uint32_t(g->n);
    t.leaf = uint32_t(g->cfg.leaf_size);
    t.left = g->left;
    t.right = g->right;
    t.parent = g->parent;
    t.skip = g->skip;
    t.first = g->first;
    t.count = g->count;
    t.geo = g->geo;
    t.lo = g->lo;
    t.hi = g->hi;
    t.mom = g->mom;
    t.wnf = g->wnf;
    for (int k = 0; k < 3; ++k) t.ctr[k] = g->ctr[k];
    t.invL = g->invL;
    t.flag = g->flag;
    t.pos = g->pos;
    t.gm = g->gm;
    t.thetaInv = 1.0 / g->cfg.theta;
    t.error = reinterpret_cast<uint32_t*>(g->small + SMALL_ERROR);
    return t;
}

double decode(unsigned long long e) { return decode_ord_host(e); }

// Node moments: the leaves' from their particles (k_leaf_moments over the leaf list, which must be
// selected into g->targets first), then the nodes above them, deepest level first (k_depth, k_bucket,
// k_moments_level).  The flag array holds the depths and leaf_at the nodes bucketed by depth; leaf_at
// is free once the leaf list is selected.
int build_moments(osph_gravity* g, const Tree& t) {
    const size_t n = g->n;
    hipStream_t st = g->stream;
    uint32_t* per_level = g->levels;
    uint32_t* cursor = g->levels + MAX_DEPTH + 1;
    timed(g, "depth", [&] {
        k_fill_u32g<<<1, BLOCK, 0, st>>>(per_level, MAX_DEPTH + 1, 0u);
        k_depth<<<std::min<unsigned>(grid_for(n - 1), LEVEL_BLOCKS), BLOCK, 0, st>>>(t, g->flag, per_level);
    });
    if (hipPeekAtLastError() != hipSuccess) return sync(g);  // the moments index by what the launches so far have written
    timed(g, "moments", [&] {
        k_levels<<<1, BLOCK, 0, st>>>(per_level, cursor, g->ntargets_dev, t.error, mailbox_next(g->box));
        k_leaf_moments<<<grid_for(n * size_t(LEAF_LANES)), BLOCK, 0, st>>>(t, g->targets, g->ntargets_dev);
        k_bucket<<<std::min<unsigned>(grid_for(n - 1), LEVEL_BLOCKS), BLOCK, 0, st>>>(uint32_t(n - 1), g->flag, cursor,
                                                                                   g->leaf_at);
    });
    // the host waits while these run
    if (int e = check_traversal(g)) return e;
    const unsigned long long* counts = g->small_host + SMALL_LEVELS;
    int deepest = MAX_DEPTH;
    while (deepest > 0 && counts[deepest] == 0) --deepest;
    size_t end = 0;
    for (int d = 0; d <= deepest; ++d) end += counts[d];
    timed(g, "moments", [&] {
        for (int d = deepest; d >= 0;) {
            int top = d;
            while (top > 0 && counts[d] <= LEVEL_RUN && counts[top - 1] <= LEVEL_RUN) --top;
            if (top < d) {
                k_moments_run<<<1, LEVEL_RUN, 0, st>>>(t, g->leaf_at, cursor, d, top);
            } else if (counts[d]) {
                k_moments_level<<<grid_for(counts[d]), BLOCK, 0, st>>>(t, g->leaf_at + (end - counts[d]), uint32_t(counts[d]));
            }
            for (; d >= top; --d) end -= counts[d];
        }
    });
    return OK;
}

// With reorder (LeapFrog steps only), the state is moved into the Morton order when due.
int build_tree(osph_gravity* g, bool reorder = false) {
    const size_t n = g->n;
    g->built = false;
    if (n == 0) {
        g->built = true;
        g->ntargets = 0;
        return OK;
    }
    hipStream_t st = g->stream;
    timed(g, "bounds", [&] {
        k_init_bounds<<<1, 64, 0, st>>>(g->small);
        unsigned gb = grid_for(n);
        gb = gb > 1024 ? 1024 : gb;
        k_bounds3<<<gb, BLOCK, 0, st>>>(g->s, g->small, n);
    });
    mailbox_post(st, g->box, 0, g->small, SMALL_ERROR + 1);
    if (int e = check_traversal(g)) return e;
    double lo[3], ext = 0.0;
    for (int k = 0; k < 3; ++k) {
        lo[k] = decode(g->small_host[k]);
        const double hi = decode(g->small_host[3 + k]);
        if (!std::isfinite(lo[k]) || !std::isfinite(hi)) return g->fail(ERR_STATE, "non-finite positions");
        ext = std::max(ext, hi - lo[k]);
    }
    const double scale = ext > 0.0 ? 2097151.0 / ext : 0.0;
    // the screened walk's frame: the root box's centre, lengths divided by 2^e >= the extent
    for (int k = 0; k < 3; ++k) g->ctr[k] = lo[k] + 0.5 * (decode(g->small_host[3 + k]) - lo[k]);
    int e = 0;
    if (ext > 0.0) (void)std::frexp(ext, &e);
    g->invL = std::ldexp(1.0, -e);
    g->wide = !(ext < std::ldexp(1.0, 510));  // every distance lies within the root box
    g->skip_ready = false;
    Tree t = tree_of(g);
    timed(g, "morton", [&] { k_morton<<<grid_for(n), BLOCK, 0, st>>>(g->s, lo[0], lo[1], lo[2], scale, g->keys, g->iota, n); });
    // (the library's calls take the last error with them)
    hipError_t err = hipPeekAtLastError();
    timed(g, "sort", [&] {
        if (err == hipSuccess) {
            err = hipcub::DeviceRadixSort::SortPairs(g->sort_temp, g->sort_temp_bytes, g->keys, g->keys_sorted, g->iota,
                                                     g->order, int(n), 0, 63, st);
        }
    });
    if (err != hipSuccess) (void)hipGetLastError();
    GCHK(g, err);
    if (reorder && g->reorder_period > 0 && ++g->since_reorder >= g->reorder_period) {
        g->since_reorder = 0;
        Planes dst{};
        for (int k = 0; k < NGPLANES; ++k) dst.d[k] = g->dblock2 + size_t(k) * g->cap;
        timed(g, "reorder", [&] {
            k_permute_planes<<<grid_for(n), BLOCK, 0, st>>>(g->s, dst, g->order, g->identity ? nullptr : g->perm,
                                                            g->perm2, g->slot_of, n);
            k_sequence<<<grid_for(n), BLOCK, 0, st>>>(g->order, n);
        });
        std::swap(g->dblock, g->dblock2);
        std::swap(g->perm, g->perm2);
        g->s = dst;
        g->identity = false;
    }
    timed(g, "gather", [&] { k_gather<<<grid_for(n), BLOCK, 0, st>>>(g->s, g->order, g->cfg.G, g->pos, g->gm, n); });
    if (n > 1) {
        timed(g, "radix_tree", [&] { k_radix_tree<<<grid_for(n - 1), BLOCK, 0, st>>>(t, g->keys_sorted); });
    }
    timed(g, "leaves", [&] {
        k_fill_u32g<<<std::min<unsigned>(grid_for(n), 4096), BLOCK, 0, st>>>(g->leaf_at, n, END);
        k_mark_leaves<<<grid_for(2 * n - 1), BLOCK, 0, st>>>(t, g->leaf_at);
        err = hipPeekAtLastError();
        if (err == hipSuccess) {
            err = hipcub::DeviceSelect::If(g->select_temp, g->select_temp_bytes, g->leaf_at, g->targets, g->ntargets_dev,
                                           int(n), NotEnd(), st);
        }
    });
    if (err != hipSuccess) (void)hipGetLastError();
    GCHK(g, err);
    g->ntargets = 1;  // a single particle is the tree's one leaf
    if (n > 1) {
        if (int e = build_moments(g, t)) return e;
        g->ntargets = uint32_t(g->small_host[SMALL_LEAVES]);
    }
    g->built = true;
    return OK;
}

// Targets below which a block of four wavefronts shares each target: with a wavefront per target, 6000 of them
// are about six per SIMD; fewer leave SIMDs without the wavefronts that hide the loads.  One wavefront / four in us, quadrupole
// FP64, octupole FP64, quadrupole mixed: 1200 targets 187 / 98, 202 / 114, 199 / 92; 3720 264 / 221, 317 / 273, 210 / 189; 5817
// (100k particles) 423 / 391, 503 / 472, 304 / 312; 7351 445 / 447, 552 / 568, 352 / 365; 11521 699 / 757, 896 / 921, 489 / 563.
constexpr uint32_t EVAL_SHARED_TARGETS = 6000;

// Targets per walk group: the largest group shares the most work, but it takes about four wavefronts per SIMD
// to hide the loads (walk of 16 / 8 / 4 targets: 1.70 / 1.69 / 2.02 ms at 8M particles, 0.32 / 0.28 / 0.27 ms at
// 1M; below 100k particles, where even groups of two leave SIMDs idle, 65-70 us whichever).
uint32_t walk_group(uint32_t ntargets) {
    uint32_t group = WALK_GROUP;
    while (group > 2 && ntargets / group < 4096) group /= 2;
    return group;
}

template <int ORDER>
void launch_eval(osph_gravity* g, const Tree& t, const WalkLists& wl, const EvalCounts& counts, const double* grads) {
    const uint32_t nt = g->ntargets, waves = BLOCK / 64;
    const uint32_t split = nt < EVAL_SHARED_TARGETS ? waves : 1u;
    const unsigned blocks = split > 1 ? nt : (nt + waves - 1) / waves;
    if (g->precision == OSPH_PRECISION_MIXED) {
        k_eval_mixed<ORDER><<<blocks, BLOCK, 0, g->stream>>>(t, g->s, g->order, g->targets, nt, wl, split, counts, grads);
    } else {
        const auto kernel = g->wide ? k_eval<ORDER, true> : k_eval<ORDER, false>;
        kernel<<<blocks, BLOCK, 0, g->stream>>>(t, g->s, g->order, g->targets, nt, wl, split, counts, grads);
    }
}

// Barnes-Hut walk and sums, adding to the state's accelerations.
int eval_bh(osph_gravity* g, osph_gravity_stats* stats) {
    const size_t n = g->n;
    if (!n) return OK;
    hipStream_t st = g->stream;
    const Tree t = tree_of(g);
    const uint32_t nt = g->ntargets;
    const uint32_t group = walk_group(nt), groups = (nt + group - 1) / group;
    uint32_t* need = reinterpret_cast<uint32_t*>(g->small + SMALL_NEED);
    for (int attempt = 0;; ++attempt) {
        if (int e = ensure_lists(g, groups)) return e;
        timed(g, "walk", [&] {
            k_fill_u32g<<<1, 64, 0, st>>>(need, 1, 0u);
            k_walk<<<(groups + BLOCK / 64 - 1) / (BLOCK / 64), BLOCK, 0, st>>>(
                t, g->targets, nt, group, g->walk_screen != 0, g->list, g->list_cap, g->list_count, need);
        });
        mailbox_post(st, g->box, SMALL_NEED, g->small + SMALL_NEED, SMALL_ERROR + 1 - SMALL_NEED);
        if (int e = check_traversal(g)) return e;
        const uint32_t most = uint32_t(g->small_host[SMALL_NEED]);
        if (most == 0) break;
        if (attempt == 3) return g->fail(ERR_STATE, "interaction lists did not fit after growing");
        // grow to the longest list and walk again
        g->list_cap = (most + most / 8 + 63u) & ~63u;
        g->list_groups = 0;
    }
    const WalkLists wl{ g->list, g->list_count, g->list_cap, group };
    EvalCounts counts{};
    if (stats) {
        if (int e = ensure_counts(g, nt)) return e;
        counts = { g->counts, g->counts + nt, g->counts + 2 * size_t(nt) };
    }
    const double* grads = g->cfg.kernel == OSPH_GRAVITY_KERNEL_M4 ? g->lut_grads : nullptr;
    timed(g, g->precision == OSPH_PRECISION_MIXED ? "eval_mixed" : "eval", [&] {
        if (g->cfg.order == 3) {
            launch_eval<3>(g, t, wl, counts, grads);
        } else if (g->cfg.order == 2) {
            launch_eval<2>(g, t, wl, counts, grads);
        } else {
            launch_eval<0>(g, t, wl, counts, grads);
        }
    });
    GCHK(g, hipPeekAtLastError());
    if (stats) {
        std::vector<uint32_t> c(4 * size_t(nt));
        GCHK(g, hipMemcpyAsync(c.data(), g->counts, c.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        if (int e = sync(g)) return e;
        *stats = osph_gravity_stats{};
        for (uint32_t k = 0; k < nt; ++k) {
            stats->nodes_approx += c[k];
            stats->nodes_exact += c[nt + k];
            stats->expansions += c[2 * size_t(nt) + 2 * size_t(k)];
            stats->pairs += c[2 * size_t(nt) + 2 * size_t(k) + 1];
        }
        stats->node_count = 2 * uint64_t(n) - 1;
    }
    return OK;
}

// Direct sum for targets (device indices) into out (double4 per target), G applied.
int eval_direct(osph_gravity* g, const uint32_t* tg_dev, size_t nt, double4* out) {
    if (!nt) return OK;
    const double* grads = g->cfg.kernel == OSPH_GRAVITY_KERNEL_M4 ? g->lut_grads : nullptr;
    timed(g, "direct", [&] {
        const auto kernel = grads ? k_direct<true> : k_direct<false>;
        kernel<<<unsigned((nt + DIRECT_TARGETS - 1) / DIRECT_TARGETS), DIRECT_WAVES * 64, 0, g->stream>>>(
            g->s, g->n, tg_dev, nt, grads, g->cfg.G, out);
    });
    return OK;
}

__global__ void k_add_direct(Planes s, const uint32_t* tg, const double4* a, size_t nt) {
    const size_t q = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= nt) return;
    const uint32_t i = tg[q];
    s.d[GAX][i] += a[q].x;
    s.d[GAY][i] += a[q].y;
    s.d[GAZ][i] += a[q].z;
}

__global__ void k_iota(uint32_t* p, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = uint32_t(i);
}

// Self-gravity of every particle added to the state's accelerations.
int eval_self(osph_gravity* g, osph_gravity_stats* stats) {
    if (g->cfg.solver == OSPH_GRAVITY_BARNES_HUT) {
        if (!g->built) return g->fail(ERR_STATE, "gravity not built");
        return eval_bh(g, stats);
    }
    const size_t n = g->n;
    if (!n) return OK;
    if (int e = ensure_scratch(g, 4 * n + n / 2 + 1)) return e;
    double4* out = reinterpret_cast<double4*>(g->scratch);
    uint32_t* tg = reinterpret_cast<uint32_t*>(g->scratch + 4 * n);
    k_iota<<<grid_for(n), BLOCK, 0, g->stream>>>(tg, n);
    if (int e = eval_direct(g, tg, n, out)) return e;
    k_add_direct<<<grid_for(n), BLOCK, 0, g->stream>>>(g->s, tg, out, n);
    if (stats) {
        *stats = osph_gravity_stats{};
        stats->pairs = uint64_t(n) * (n - 1);
    }
    return OK;
}

int upload_vectors(osph_gravity* g, const double* host, size_t stride, int plane0, int ncomp, size_t n) {
    if (!n) return OK;
    if (int e = ensure_staging(g, n * stride)) return e;
    GCHK(g, hipMemcpyAsync(g->staging, host, n * stride, hipMemcpyHostToDevice, g->stream));
    k_unstage<<<grid_for(n), BLOCK, 0, g->stream>>>(g->staging, stride, ncomp, g->s, plane0,
                                                    g->identity ? nullptr : g->perm, n);
    return OK;
}

int download_vectors(osph_gravity* g, double* host, size_t stride, int plane0, int ncomp, size_t n) {
    if (!n) return OK;
    if (int e = ensure_staging(g, n * stride)) return e;
    if (stride > size_t(ncomp) * sizeof(double)) {
        // keep the caller's other lanes: start from their current values
        GCHK(g, hipMemcpyAsync(g->staging, host, n * stride, hipMemcpyHostToDevice, g->stream));
    }
    k_stage<<<grid_for(n), BLOCK, 0, g->stream>>>(g->staging, stride, ncomp, g->s, plane0,
                                                  g->identity ? nullptr : g->perm, n);
    GCHK(g, copy_to_host(g->stream, host, g->staging, n * stride));
    return sync(g);
}

}  // namespace

namespace {

// Positions, smoothing lengths and masses of another context's particles (device planes, n each) into
// this context's planes; accelerations and velocities start at zero.
__global__ void __launch_bounds__(BLOCK) k_load_planes(Planes s, const double* __restrict__ x,
                                                       const double* __restrict__ y, const double* __restrict__ z,
                                                       const double* __restrict__ h, const double* __restrict__ m,
                                                       size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    s.d[GX][i] = x[i];
    s.d[GY][i] = y[i];
    s.d[GZ][i] = z[i];
    s.d[GH][i] = h[i];
    s.d[GM][i] = m[i];
    for (int k = GVX; k <= GVH; ++k) s.d[k][i] = 0.0;
    for (int k = GAX; k <= GAZ; ++k) s.d[k][i] = 0.0;
}

}  // namespace

const void* gravity_owner(const osph_gravity* g) { return g->owner; }
void gravity_set_owner(osph_gravity* g, const void* owner) { g->owner = owner; }

// GravitySolver::loop's gravity half (core/sph/solvers/GravitySolver.cpp:64-80) for particles held in
// another context's device planes: once `ready` has fired, the planes are copied in on this context's
// stream, the tree is built and the self-gravity evaluated; `done` is recorded after the last kernel and
// accel[0..2] then point to the accelerations (n doubles each, in the order of the source planes).
int gravity_self_from_device(osph_gravity* g, size_t n, const double* const src[5], hipEvent_t ready,
                             hipEvent_t done, const double* accel[3]) {
    if (!g || (n && !src)) return ERR_ARG;
    if (n >= (size_t(1) << 31)) return g->fail(ERR_ARG, "particle count must be below 2^31");
    if (int e = ensure_particles(g, n > 0 ? n : 1)) return e;
    g->n = n;
    g->built = false;
    g->identity = true;  // the planes are loaded in the source order and stay in it
    for (int k = 0; k < 3; ++k) accel[k] = g->s.d[GAX + k];
    GCHK(g, hipStreamWaitEvent(g->stream, ready, 0));
    if (n) {
        k_load_planes<<<grid_for(n), BLOCK, 0, g->stream>>>(g->s, src[0], src[1], src[2], src[3], src[4], n);
        GCHK(g, hipPeekAtLastError());
        if (int e = osph_gravity_build(g)) return e;
        if (int e = eval_self(g, nullptr)) return e;
    }
    GCHK(g, hipEventRecord(done, g->stream));
    return OK;
}

extern "C" {

int osph_gravity_create(osph_gravity** out, const osph_gravity_config* cfg) {
    if (!out || !cfg) return ERR_ARG;
    *out = nullptr;
    if (cfg->solver != OSPH_GRAVITY_BRUTE_FORCE && cfg->solver != OSPH_GRAVITY_BARNES_HUT) return ERR_ARG;
    if (cfg->kernel != OSPH_GRAVITY_KERNEL_POINT && cfg->kernel != OSPH_GRAVITY_KERNEL_M4) return ERR_ARG;
    if (cfg->solver == OSPH_GRAVITY_BARNES_HUT) {
        if (!(cfg->theta > 0.0) || !std::isfinite(cfg->theta)) return ERR_ARG;
        if (cfg->order != 0 && cfg->order != 2 && cfg->order != 3) return ERR_ARG;
        if (cfg->leaf_size < 1 || cfg->leaf_size > 64) return ERR_ARG;
    }
    osph_gravity* g = new osph_gravity();
    transfer_attach();
    g->cfg = *cfg;
    auto bail = [&](int code) {
        osph_gravity_destroy(g);
        return code;
    };
    if (hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess) return bail(ERR_HIP);
    if (hipMalloc(&g->small, 16 * sizeof(unsigned long long)) != hipSuccess) return bail(ERR_HIP);
    if (hipMemset(g->small, 0, 16 * sizeof(unsigned long long)) != hipSuccess) return bail(ERR_HIP);
    if (hipMalloc(&g->levels, 2 * (MAX_DEPTH + 1) * sizeof(uint32_t)) != hipSuccess) return bail(ERR_HIP);
    if (mailbox_create(g->box, SMALL_HOST_WORDS) != hipSuccess) return bail(ERR_HIP);
    g->small_host = g->box.host;
    std::vector<double> grads(LUT_ENTRIES + 1), values(LUT_ENTRIES + 1);
    const double qSqrToIdx = double(LUT_ENTRIES) * (1.0 / (2.0 * 2.0));
    for (int i = 0; i <= LUT_ENTRIES; ++i) {
        const double qSqr = double(i) / qSqrToIdx;
        grads[i] = gk_grad(qSqr);
        values[i] = gk_value(qSqr);
    }
    if (hipMalloc(&g->lut_grads, grads.size() * sizeof(double)) != hipSuccess) return bail(ERR_HIP);
    if (hipMalloc(&g->lut_values, values.size() * sizeof(double)) != hipSuccess) return bail(ERR_HIP);
    if (hipMemcpy(g->lut_grads, grads.data(), grads.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(g->lut_values, values.data(), values.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
        return bail(ERR_HIP);
    }
    *out = g;
    return OK;
}

void osph_gravity_destroy(osph_gravity* g) {
    if (!g) return;
    if (g->stream) (void)hipStreamSynchronize(g->stream);
    resolve(g);
    for (hipEvent_t e : g->pool) (void)hipEventDestroy(e);
    free_particles(g);
    void* ptrs[] = { g->list, g->list_count, g->counts, g->small, g->levels, g->lut_grads, g->lut_values,
                     g->scratch, g->staging };
    for (void* p : ptrs) (void)hipFree(p);
    mailbox_destroy(g->box);
    if (g->stream) (void)hipStreamDestroy(g->stream);
    delete g;
    transfer_detach();
}

const char* osph_gravity_last_error(const osph_gravity* g) { return g ? g->err.c_str() : "null context"; }

int osph_gravity_set_precision(osph_gravity* g, int precision) {
    if (!g) return ERR_ARG;
    if (precision != OSPH_PRECISION_FP64 && precision != OSPH_PRECISION_MIXED) {
        return g->fail(ERR_ARG, "precision must be OSPH_PRECISION_FP64 or OSPH_PRECISION_MIXED");
    }
    g->precision = precision;
    return OK;
}

int osph_gravity_tune(osph_gravity* g, const char* key, long long value) {
    if (!g || !key) return ERR_ARG;
    const std::string k(key);
    if (k == "walk_screen" && (value == -1 || value == 0 || value == 1)) {
        g->walk_screen = int(value);
        return OK;
    }
    if (k == "reorder_period" && value >= 0 && value <= 1000000) {
        g->reorder_period = int(value);
        return OK;
    }
    return g->fail(ERR_ARG, "unknown tuning key or value out of range: " + k);
}

int osph_gravity_set_particles(osph_gravity* g, size_t n, const double* r, const double* v, size_t vec_stride,
                               const double* m) {
    if (!g || (n && (!r || !m))) return ERR_ARG;
    if (n >= (size_t(1) << 31)) return g->fail(ERR_ARG, "particle count must be below 2^31");
    const size_t stride = vec_stride ? vec_stride : 4 * sizeof(double);
    if (stride < 4 * sizeof(double) || stride % sizeof(double)) return g->fail(ERR_ARG, "bad vector stride");
    if (int e = ensure_particles(g, n > 0 ? n : 1)) return e;
    g->n = n;
    g->built = false;
    g->identity = true;
    g->since_reorder = g->reorder_period;  // the first LeapFrog build moves the state into Morton order
    if (!n) return sync(g);
    if (int e = upload_vectors(g, r, stride, GX, 4, n)) return e;
    if (v) {
        if (int e = upload_vectors(g, v, stride, GVX, 4, n)) return e;
        if (int e = sync(g)) return e;  // the staging buffer is reused below
    } else {
        GCHK(g, hipMemsetAsync(g->s.d[GVX], 0, 4 * sizeof(double) * g->cap, g->stream));
    }
    GCHK(g, hipMemsetAsync(g->s.d[GAX], 0, 3 * sizeof(double) * g->cap, g->stream));
    GCHK(g, hipMemcpyAsync(g->s.d[GM], m, n * sizeof(double), hipMemcpyHostToDevice, g->stream));
    return sync(g);
}

int osph_gravity_get(osph_gravity* g, int what, double* out, size_t vec_stride) {
    if (!g || !out || what < 0 || what > 2) return ERR_ARG;
    const size_t stride = vec_stride ? vec_stride : 4 * sizeof(double);
    if (stride < 4 * sizeof(double) || stride % sizeof(double)) return g->fail(ERR_ARG, "bad vector stride");
    const int plane0 = what == 0 ? GX : (what == 1 ? GVX : GAX);
    const int ncomp = what == 2 ? 3 : 4;
    if (what == 2) {
        for (size_t i = 0; i < g->n; ++i) out[i * (stride / sizeof(double)) + 3] = 0.0;
    }
    return download_vectors(g, out, stride, plane0, ncomp, g->n);
}

int osph_gravity_build(osph_gravity* g) {
    if (!g) return ERR_ARG;
    if (g->cfg.solver == OSPH_GRAVITY_BRUTE_FORCE) {
        g->built = true;
        return OK;
    }
    return build_tree(g);
}

int osph_gravity_eval_self(osph_gravity* g, double* dv, size_t vec_stride, osph_gravity_stats* stats) {
    if (!g) return ERR_ARG;
    const size_t stride = vec_stride ? vec_stride : 4 * sizeof(double);
    if (dv) {
        if (stride < 4 * sizeof(double) || stride % sizeof(double)) return g->fail(ERR_ARG, "bad vector stride");
        if (int e = upload_vectors(g, dv, stride, GAX, 3, g->n)) return e;
        if (int e = sync(g)) return e;
    }
    if (int e = eval_self(g, stats)) return e;
    if (dv) return download_vectors(g, dv, stride, GAX, 3, g->n);
    return sync(g);
}

int osph_gravity_eval_points(osph_gravity* g, const double* p, size_t np, double* a, size_t vec_stride) {
    if (!g || (np && (!p || !a))) return ERR_ARG;
    const size_t stride = vec_stride ? vec_stride : 4 * sizeof(double);
    if (stride < 4 * sizeof(double) || stride % sizeof(double)) return g->fail(ERR_ARG, "bad vector stride");
    if (!np) return OK;
    if (g->cfg.solver != OSPH_GRAVITY_BARNES_HUT) {
        return g->fail(ERR_STATE, "point evaluation is provided by the Barnes-Hut solver");
    }
    if (!g->built) return g->fail(ERR_STATE, "gravity not built");
    if (int e = ensure_scratch(g, 8 * np)) return e;
    double4* pts = reinterpret_cast<double4*>(g->scratch);
    double4* acc = pts + np;
    std::vector<double4> hp(np), ha(np);
    for (size_t k = 0; k < np; ++k) {
        const double* e = p + k * (stride / sizeof(double));
        hp[k] = make_double4(e[0], e[1], e[2], e[3]);
    }
    GCHK(g, hipMemcpyAsync(pts, hp.data(), np * sizeof(double4), hipMemcpyHostToDevice, g->stream));
    if (g->n == 0) {
        for (size_t k = 0; k < np; ++k) {
            double* e = a + k * (stride / sizeof(double));
            e[0] = e[1] = e[2] = e[3] = 0.0;
        }
        return sync(g);
    }
    const double* grads = g->cfg.kernel == OSPH_GRAVITY_KERNEL_M4 ? g->lut_grads : nullptr;
    Tree t = tree_of(g);
    if (!g->skip_ready) {
        timed(g, "skip", [&] { k_skip<<<grid_for(2 * g->n - 1), BLOCK, 0, g->stream>>>(t); });
        g->skip_ready = true;
    }
    timed(g, "points", [&] { k_points<<<grid_for(np), BLOCK, 0, g->stream>>>(t, pts, acc, np, grads, g->cfg.order); });
    GCHK(g, hipMemcpyAsync(ha.data(), acc, np * sizeof(double4), hipMemcpyDeviceToHost, g->stream));
    mailbox_post(g->stream, g->box, SMALL_ERROR, g->small + SMALL_ERROR, 1);
    if (int e = sync(g)) return e;
    if (int e = check_traversal(g)) return e;
    for (size_t k = 0; k < np; ++k) {
        double* e = a + k * (stride / sizeof(double));
        e[0] = ha[k].x;
        e[1] = ha[k].y;
        e[2] = ha[k].z;
        e[3] = 0.0;
    }
    return OK;
}

int osph_gravity_direct(osph_gravity* g, const uint32_t* t, size_t nt, double* a, size_t vec_stride) {
    if (!g || (nt && (!t || !a))) return ERR_ARG;
    const size_t stride = vec_stride ? vec_stride : 4 * sizeof(double);
    if (stride < 4 * sizeof(double) || stride % sizeof(double)) return g->fail(ERR_ARG, "bad vector stride");
    for (size_t k = 0; k < nt; ++k) {
        if (t[k] >= g->n) return g->fail(ERR_ARG, "target index out of range");
    }
    if (!nt) return OK;
    if (int e = ensure_scratch(g, 4 * nt + nt / 2 + 1)) return e;
    double4* out = reinterpret_cast<double4*>(g->scratch);
    uint32_t* tg = reinterpret_cast<uint32_t*>(g->scratch + 4 * nt);
    GCHK(g, hipMemcpyAsync(tg, t, nt * sizeof(uint32_t), hipMemcpyHostToDevice, g->stream));
    if (!g->identity) k_to_slots<<<grid_for(nt), BLOCK, 0, g->stream>>>(tg, g->slot_of, nt);
    if (int e = eval_direct(g, tg, nt, out)) return e;
    std::vector<double4> ha(nt);
    GCHK(g, hipMemcpyAsync(ha.data(), out, nt * sizeof(double4), hipMemcpyDeviceToHost, g->stream));
    if (int e = sync(g)) return e;
    for (size_t k = 0; k < nt; ++k) {
        double* e = a + k * (stride / sizeof(double));
        e[0] = ha[k].x;
        e[1] = ha[k].y;
        e[2] = ha[k].z;
        e[3] = 0.0;
    }
    return OK;
}

int osph_gravity_energy(osph_gravity* g, double* energy) {
    if (!g || !energy) return ERR_ARG;
    const size_t n = g->n;
    *energy = 0.0;
    if (!n) return OK;
    const unsigned blocks = std::min<unsigned>(grid_for(n), 1024);
    if (int e = ensure_scratch(g, n + blocks + 1)) return e;
    const double* values = g->cfg.kernel == OSPH_GRAVITY_KERNEL_M4 ? g->lut_values : nullptr;
    timed(g, "energy", [&] {
        k_energy<<<grid_for(n), BLOCK, 0, g->stream>>>(g->s, n, values, g->scratch);
        k_sum_vector<<<blocks, BLOCK, 0, g->stream>>>(g->scratch, n, g->scratch + n);
        k_sum_partials<<<1, 64, 0, g->stream>>>(g->scratch + n, int(blocks), 1, g->scratch + n + blocks);
    });
    double sum = 0.0;
    GCHK(g, hipMemcpyAsync(&sum, g->scratch + n + blocks, sizeof(double), hipMemcpyDeviceToHost, g->stream));
    if (int e = sync(g)) return e;
    *energy = 0.5 * g->cfg.G * sum;
    return OK;
}

int osph_gravity_moments(osph_gravity* g, double out[16]) {
    if (!g || !out) return ERR_ARG;
    if (g->cfg.solver != OSPH_GRAVITY_BARNES_HUT || !g->built) return g->fail(ERR_STATE, "no Barnes-Hut tree built");
    std::memset(out, 0, 16 * sizeof(double));
    if (g->n == 0) return OK;
    if (int e = sync(g)) return e;  // the copies below do not wait for the stream
    if (g->n == 1) {
        double4 p;
        double m;
        GCHK(g, hipMemcpy(&p, g->pos, sizeof(p), hipMemcpyDeviceToHost));
        GCHK(g, hipMemcpy(&m, g->gm, sizeof(m), hipMemcpyDeviceToHost));
        out[0] = m / g->cfg.G;
        out[1] = p.x;
        out[2] = p.y;
        out[3] = p.z;
        return OK;
    }
    double4 geo;
    NodeMom mom;
    GCHK(g, hipMemcpy(&geo, g->geo, sizeof(geo), hipMemcpyDeviceToHost));
    GCHK(g, hipMemcpy(&mom, g->mom, sizeof(mom), hipMemcpyDeviceToHost));
    const double inv = 1.0 / g->cfg.G;  // BarnesHut::getMoments divides the premultiplied moments by G
    out[0] = mom.M * inv;
    out[1] = geo.x;
    out[2] = geo.y;
    out[3] = geo.z;
    for (int k = 0; k < 5; ++k) out[4 + k] = mom.q2[k] * inv;
    for (int k = 0; k < 7; ++k) out[9 + k] = mom.q3[k] * inv;
    return OK;
}

int osph_gravity_step_leapfrog(osph_gravity* g, double dt, int steps) {
    if (!g) return ERR_ARG;
    if (!(dt > 0.0) || !std::isfinite(dt) || steps < 0) return g->fail(ERR_ARG, "bad time step or step count");
    const size_t n = g->n;
    if (!n) return OK;
    for (int s = 0; s < steps; ++s) {
        timed(g, "drift", [&] { k_drift<<<grid_for(n), BLOCK, 0, g->stream>>>(g->s, dt, n); });
        k_zero_acc<<<grid_for(n), BLOCK, 0, g->stream>>>(g->s, n);
        if (g->cfg.solver == OSPH_GRAVITY_BARNES_HUT) {
            if (int e = build_tree(g, true)) return e;
        }
        if (int e = eval_self(g, nullptr)) return e;
        timed(g, "kick_drift", [&] { k_kick_drift<<<grid_for(n), BLOCK, 0, g->stream>>>(g->s, dt, n); });
    }
    return sync(g);
}

int osph_gravity_integrals(osph_gravity* g, double out[11]) {
    if (!g || !out) return ERR_ARG;
    std::memset(out, 0, 11 * sizeof(double));
    const size_t n = g->n;
    if (!n) return OK;
    const unsigned blocks = std::min<unsigned>(grid_for(n), 1024);
    if (int e = ensure_scratch(g, size_t(blocks) * 11 + 11)) return e;
    k_integrals<<<blocks, BLOCK, 0, g->stream>>>(g->s, n, g->scratch);
    k_sum_partials<<<1, 64, 0, g->stream>>>(g->scratch, int(blocks), 11, g->scratch + size_t(blocks) * 11);
    GCHK(g, hipMemcpyAsync(out, g->scratch + size_t(blocks) * 11, 11 * sizeof(double), hipMemcpyDeviceToHost, g->stream));
    if (int e = sync(g)) return e;
    // CenterOfMass::evaluate (Integrals.cpp:155-180): sum m r / sum m
    for (int k = 7; k < 10; ++k) out[k] /= out[10];
    return OK;
}

int osph_gravity_sync(osph_gravity* g) {
    if (!g) return ERR_ARG;
    return sync(g);
}

int osph_gravity_profile_enable(osph_gravity* g, int enable) {
    if (!g) return ERR_ARG;
    GCHK(g, hipStreamSynchronize(g->stream));
    resolve(g);
    g->prof = enable != 0;
    g->acc.clear();
    return OK;
}

int osph_gravity_profile_read(osph_gravity* g, char* names, size_t name_cap, double* ms, uint64_t* launches, int cap,
                              int* count) {
    if (!g || !count) return ERR_ARG;
    GCHK(g, hipStreamSynchronize(g->stream));
    resolve(g);
    int k = 0;
    for (const auto& kv : g->acc) {
        if (k < cap) {
            if (names && name_cap) {
                std::strncpy(names + size_t(k) * name_cap, kv.first.c_str(), name_cap - 1);
                names[size_t(k) * name_cap + name_cap - 1] = '\0';
            }
            if (ms) ms[k] = kv.second.first;
            if (launches) launches[k] = kv.second.second;
        }
        ++k;
    }
    *count = k;
    return OK;
}

}  // extern "C"
