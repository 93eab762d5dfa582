// HIP kernels of the OpenSPH per-timestep hot path for gfx950 (MI355X).
//
// Layout: particle state is SoA in HBM (one plane per component, storage order).  Every evaluation
// sorts the particles by the Morton code of a uniform cell grid (cell edge >= 2 h_max), packs the
// per-neighbour data into 128-byte records in that order, builds neighbour lists with the exact FP64
// pair test of SymmetricSolver<3>::loop, and evaluates all pair sums in gather form: each particle
// sums over its own neighbours, so every sum is written by one thread, in a fixed order, without atomics.
#include "osph_device.h"
#include "osph_internal.h"

#include <algorithm>
#include <type_traits>


namespace osph {

namespace {


// ---- material physics (per particle; compiled without FMA contraction so that branch decisions
// ---- follow the reference's rounding) -------------------------------------------------------------

// TillotsonEos::evaluate (core/physics/Eos.cpp:198-238)
__device__ void tillotson(const osph_material& m, double rho, double u, double& p_out, double& cs_out) {
#pragma clang fp contract(off)
    const double eta = rho / m.rho0;
    const double mu = eta - 1.0;
    const double denom = u / (m.u0 * eta * eta) + 1.0;
    const double pc = (m.a + m.b / denom) * rho * u + m.A * mu + m.B * mu * mu;
    double dpdu = m.a * rho + m.b * rho / (denom * denom);
    double dpdrho = m.a * u + m.b * u * (3.0 * denom - 2.0) / (denom * denom) + m.A / m.rho0 + 2.0 * m.B * mu / m.rho0;
    const double csc = dpdrho + dpdu * pc / (rho * rho);
    const double rhoExp = m.rho0 / rho - 1.0;
    const double betaExp = exp(-dmin(m.beta * rhoExp, 70.0));
    const double alphaExp = exp(-dmin(m.alpha * (rhoExp * rhoExp), 70.0));
    const double pe = m.a * rho * u + (m.b * rho * u / denom + m.A * mu * betaExp) * alphaExp;
    dpdu = m.a * rho + alphaExp * m.b * rho / (denom * denom);
    dpdrho = m.a * u + alphaExp * (m.b * u * (3.0 * denom - 2.0) / (denom * denom)) +
             alphaExp * (m.b * u * rho / denom) * m.rho0 * (2.0 * m.alpha * rhoExp) / (rho * rho) +
             alphaExp * m.A * betaExp * (1.0 / m.rho0 + m.rho0 * mu / (rho * rho) * (2.0 * m.alpha * rhoExp + m.beta));
    double cse = dpdrho + dpdu * pe / (rho * rho);
    cse = dmax(cse, 0.0);
    double p = pc, cs = csc;
    if (rho <= m.rho0 && u > m.ucv) {
        p = pe;
        cs = cse;
    } else if (rho <= m.rho0 && u > m.uiv && u <= m.ucv) {
        p = ((u - m.uiv) * pe + (m.ucv - u) * pc) / (m.ucv - m.uiv);
        cs = ((u - m.uiv) * cse + (m.ucv - u) * csc) / (m.ucv - m.uiv);
    }
    cs = dmax(cs, 0.25 * m.A / m.rho0);
    p_out = p;
    cs_out = sqrt(cs);
}

// sqrtInv / sqrtApprox (core/math/MathUtils.h:44-62): the single-precision bit-trick estimate with one
// Newton step that norm(Vector) uses (core/objects/geometry/Vector.h:681-685).
__device__ double sqrt_approx(double f) {
#pragma clang fp contract(off)
    if (f == 0.0) return 0.0;
    const float x2 = float(f) * 0.5f;
    float y = float(f);
    int i = __float_as_int(y);
    i = 0x5f3759df - (i >> 1);
    y = __int_as_float(i);
    const float r = y * (1.5f - (x2 * y * y));
    return 1.0 / double(r);
}

// findEigenvalues (core/objects/geometry/SymmetricTensor.h:377-398); t = {xx, yy, zz, xy, xz, yz}
__device__ void eigenvalues(const double t[6], double out[3]) {
#pragma clang fp contract(off)
    const double d0 = t[0], d1 = t[1], d2 = t[2], o0 = t[3], o1 = t[4], o2 = t[5];
    const double mx0 = dmax(d0, o0), mx1 = dmax(d1, o1), mx2 = dmax(d2, o2);
    const double n = sqrt_approx(mx0 * mx0 + mx1 * mx1 + mx2 * mx2);
    if (n < 1.e-12) {
        out[0] = out[1] = out[2] = 0.0;
        return;
    }
    const double I1 = d0 * 1.0 + d1 * 1.0 + d2 * 1.0;
    const double I2 = (o0 * o0 + o1 * o1 + o2 * o2) - (d1 * d2 + d2 * d0 + d0 * d1);
    const double I3 = d0 * d1 * d2 + 2.0 * o0 * o1 * o2 - ((o0 * o0) * d2 + (o1 * o1) * d1 + (o2 * o2) * d0);
    const double p = -I1 / n;
    const double q = -I2 / (n * n);
    const double r = -I3 / (n * n * n);
    const double a = q - p * p / 3.0;
    const double b = (2.0 * (p * p * p) - 9.0 * p * q + 27.0 * r) / 27.0;
    const double aCub = (a * a * a) / 27.0;
    if (0.25 * b * b + aCub >= 0.0) {
        out[0] = out[1] = out[2] = 0.0;
        return;
    }
    const double t1 = 2.0 * sqrt(-a / 3.0);
    const double phi = acos(-0.5 * b / sqrt(-aCub));
    const double p3 = p / 3.0;
    out[0] = (t1 * cos(phi / 3.0) - p3) * n;
    out[1] = (t1 * cos((phi + 2.0 * PI_D) / 3.0) - p3) * n;
    out[2] = (t1 * cos((phi + 4.0 * PI_D) / 3.0) - p3) * n;
}

// EosMaterial::initialize (core/sph/Materials.cpp:47-58), VonMisesRheology::initialize
// (core/physics/Rheology.cpp:36-83) or DruckerPragerRheology::initialize (core/physics/Rheology.cpp:119-181,
// without acoustic fluidization) and the h clamp of AdaptiveSmoothingLength::initialize
// (core/sph/equations/EquationTerm.cpp:356-364).
__device__ void material_init_at(DevState& s, const osph_material& m, const Params& prm, size_t i) {
#pragma clang fp contract(off)
    double p, cs;
    tillotson(m, s.d[RHO][i], s.d[U][i], p, cs);
    s.d[CS][i] = cs;
    if (m.yielding == 1) {
        const double dmg = prm.has_damage ? s.d[D][i] : 0.0;
        const double d = prm.has_damage ? dmg * dmg * dmg : 0.0;
        if (p < 0.0) p = (1.0 - d) * p;
        const double u = s.d[U][i];
        const double unorm = u / m.melt_energy;
        double Y = unorm < 1.e-5 ? m.elasticity_limit : m.elasticity_limit * dmax(1.0 - unorm, 0.0);
        Y = (1.0 - d) * Y;
        if (Y < EPS_D) {
            s.d[RED][i] = 0.0;
            s.d[SXX][i] = 0.0;
            s.d[SYY][i] = 0.0;
            s.d[SXY][i] = 0.0;
            s.d[SXZ][i] = 0.0;
            s.d[SYZ][i] = 0.0;
        } else {
            const double xx = s.d[SXX][i], yy = s.d[SYY][i], zz = -xx - yy;
            const double xy = s.d[SXY][i], xz = s.d[SXZ][i], yz = s.d[SYZ][i];
            const double dd = (xx * xx + yy * yy + zz * zz) + 2.0 * (xy * xy + xz * xz + yz * yz);
            const double J2 = 0.5 * dd + 1.e-15;
            const double red = dmin(Y / sqrt(3.0 * J2), 1.0);
            s.d[RED][i] = red;
            s.d[SXX][i] = xx * red;
            s.d[SYY][i] = yy * red;
            s.d[SXY][i] = xy * red;
            s.d[SXZ][i] = xz * red;
            s.d[SYZ][i] = yz * red;
        }
    } else if (m.yielding == 2) {
        const double d = prm.has_damage ? s.d[D][i] * s.d[D][i] * s.d[D][i] : 0.0;
        if (p < 0.0) p = (1.0 - d) * p;
        const double Y0 = m.cohesion, YM = m.elasticity_limit, mui = m.internal_friction, mud = m.dry_friction;
        const double Yi = Y0 + mui * p / (1.0 + mui * dmax(p, 0.0) / (YM - Y0));
        const double Yd = mud * p;
        double Y = Yd > Yi ? Yi : (1.0 - d) * Yi + d * Yd;
        const double u = s.d[U][i];
        Y = u < 1.e-5 * m.melt_energy ? Y : Y * dmax(1.0 - u / m.melt_energy, 0.0);
        if (Y < EPS_D) {
            s.d[RED][i] = 0.0;
            s.d[SXX][i] = 0.0;
            s.d[SYY][i] = 0.0;
            s.d[SXY][i] = 0.0;
            s.d[SXZ][i] = 0.0;
            s.d[SYZ][i] = 0.0;
        } else {
            const double xx = s.d[SXX][i], yy = s.d[SYY][i], zz = -xx - yy;
            const double xy = s.d[SXY][i], xz = s.d[SXZ][i], yz = s.d[SYZ][i];
            const double dd = (xx * xx + yy * yy + zz * zz) + 2.0 * (xy * xy + xz * xz + yz * yz);
            const double J2 = 0.5 * dd + EPS_D;
            const double red = dmin(Y / sqrt(J2), 1.0);
            s.d[RED][i] = red;
            s.d[SXX][i] = xx * red;
            s.d[SYY][i] = yy * red;
            s.d[SXY][i] = xy * red;
            s.d[SXZ][i] = xz * red;
            s.d[SYZ][i] = yz * red;
        }
    }
    s.d[P][i] = p;
    if (prm.adaptive_h) {
        s.d[H][i] = dmax(prm.h_lo, dmin(s.d[H][i], prm.h_hi));
    }
}

// ---- grid ------------------------------------------------------------------------------------------

// Block reduction of NV order-encoded values; is_min[k] selects min or max for value k.
template <int NV>
__device__ void block_reduce_ord(unsigned long long (&v)[NV], const bool (&is_min)[NV], unsigned long long* acc) {
    __shared__ unsigned long long red[BLOCK / 64][NV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const unsigned long long r = is_min[k] ? wave_min(v[k]) : wave_max(v[k]);
        if (lane == 0) red[wave][k] = r;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < NV; k += blockDim.x) {
        unsigned long long r = red[0][k];
        for (int w = 1; w < BLOCK / 64; ++w) {
            const unsigned long long x = red[w][k];
            r = is_min[k] ? (x < r ? x : r) : (x > r ? x : r);
        }
        if (is_min[k]) {
            atomicMin(&acc[k], r);
        } else {
            atomicMax(&acc[k], r);
        }
    }
}

__device__ __forceinline__ void init_small_at(unsigned long long* a, int t) {
    bool is_min;
    if (t >= SMALL_CLASSES && t < SMALL_CLASSES + CLASS_STRIDE * MAX_CLASSES) {
        const int k = (t - SMALL_CLASSES) % CLASS_STRIDE;
        is_min = k < 3 || k == 7;
    } else if (t >= SMALL_CRITERIA && t < SMALL_CRITERIA + 4) {
        is_min = true;
    } else if (t >= SMALL_VEL && t < SMALL_VEL + 6) {
        is_min = t < SMALL_VEL + 3;
    } else {
        is_min = t < SMALL_BOUNDS + 3 || t == SMALL_BOUNDS + 7;
    }
    a[t] = is_min ? ~0ull : 0ull;
}

__global__ void __launch_bounds__(SMALL_WORDS) k_init_small(unsigned long long* a) { init_small_at(a, threadIdx.x); }

// acc[0..2] = min x, y, z; acc[3..5] = max x, y, z; acc[6] = max h; acc[7] = min h (order-encoded).
__global__ void __launch_bounds__(BLOCK) k_bounds(DevState s, unsigned long long* acc, size_t n) {
    unsigned long long v[8] = { ~0ull, ~0ull, ~0ull, 0ull, 0ull, 0ull, 0ull, ~0ull };
    const bool is_min[8] = { true, true, true, false, false, false, false, true };
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
        for (int k = 0; k < 3; ++k) {
            const unsigned long long b = ord_bits(s.d[X + k][i]);
            v[k] = b < v[k] ? b : v[k];
            v[3 + k] = b > v[3 + k] ? b : v[3 + k];
        }
        const unsigned long long hb = ord_bits(s.d[H][i]);
        v[6] = hb > v[6] ? hb : v[6];
        v[7] = hb < v[7] ? hb : v[7];
    }
    block_reduce_ord<8>(v, is_min, acc);
}

__device__ __forceinline__ int h_class(double h, double hmin, int nclass) {
    if (nclass <= 1) return 0;
    const int c = int(floor(log2(h / hmin)));
    return c < 0 ? 0 : (c >= nclass ? nclass - 1 : c);
}

__device__ __forceinline__ int cell_coord(const GridClass& g, double x, int k) {
    return int(floor((x - g.lo[k]) * g.inv_cell));
}

__device__ __forceinline__ void cell_of(const GridClass& g, double x, double y, double z, int c[3]) {
    const double v[3] = { x, y, z };
    for (int k = 0; k < 3; ++k) {
        int ci = cell_coord(g, v[k], k);
        ci = ci < 0 ? 0 : (ci >= g.dim[k] ? g.dim[k] - 1 : ci);
        c[k] = ci;
    }
}

__global__ void __launch_bounds__(BLOCK) k_fill_u32(uint32_t* p, size_t count, uint32_t value) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += size_t(gridDim.x) * blockDim.x) {
        p[i] = value;
    }
}

// Row q of the grid (rows of all non-empty classes numbered in turn): its class, y and z.
__device__ __forceinline__ bool row_of(const Grid& g, size_t q, int& cls, uint32_t& cy, uint32_t& cz) {
    for (int c = 0; c < g.nclass; ++c) {
        const GridClass& G = g.c[c];
        if (G.empty) continue;
        const size_t nr = size_t(G.dim[1]) * size_t(G.dim[2]);
        if (q < nr) {
            cls = c;
            cy = uint32_t(q % size_t(G.dim[1]));
            cz = uint32_t(q / size_t(G.dim[1]));
            return true;
        }
        q -= nr;
    }
    return false;
}

// ---- sort by cell and cell table ------------------------------------------------------------------------
// The order of the particles by (cell, particle), and the cell table, in one of two ways (sort_by_cells).
//
// By rows of cells: a row (slot0(class) + Morton(y, z), the cell index without x) is a bucket, and a row's particles
// are ordered by (x, particle) on their own.  Four launches -- count, scan, scatter, order -- whatever the particle
// count, where a radix sort of the keys took 3 passes over them (onesweep, 84 us at 1M particles) or about ten merge
// launches (below 1M: 120 us at 559k, 40 us at 43k), and two more kernels built the table (30 us at 1M).  Measured
// here: 12 + 8 + 6 + 14 us at 1M, 20 us in all up to 170k particles (launch latency).
//
// By cells, where rows are long: far outliers stretch the cells to 1/250 of the extent, and a compact body then fills a
// few rows of thousands of particles, too much for a wavefront or block each.  The cells themselves are the buckets
// and the cell table holds their counts; a particle's place in its cell is the number of lower particles there, counted
// by a thread each.  A wavefront puts its particles of a cell next to one another, so the count goes by such runs: 64 particles
// each where a cell holds most of them, or where the state is nearly in cell order, down to one each in a random order, and then
// still a fraction of what the list kernel does with the same cell.  No row or cell has to fit anywhere.
//
// The buckets are filled with atomics, in any order; the order within them does not depend on it.

// The valid lanes of the wavefront with this lane's bucket: the first of them, how many lie before this one, and all.
struct WaveRun {
    uint32_t leader, before, total;
};
__device__ __forceinline__ WaveRun wave_run(uint32_t bucket, bool valid) {
    const uint32_t lane = threadIdx.x & 63u;
    WaveRun run{ lane, 0u, 0u };
    for (unsigned long long open = __ballot(valid); open != 0ull;) {
        const int l = __builtin_ctzll(open);
        const unsigned long long same = __ballot(bucket == uint32_t(__builtin_amdgcn_readlane(bucket, l))) & open;
        if ((same >> lane) & 1ull) {
            run.leader = uint32_t(l);
            run.before = uint32_t(__popcll(same & ((1ull << lane) - 1ull)));
            run.total = uint32_t(__popcll(same));
        }
        open &= ~same;
    }
    return run;
}

// Counts the particles of every row: where[i] = (row << 8 | x, rank in the row), or by CELLS of every cell (in `first`)
// and row: where[i] = (cell, rank in the cell).  One atomic per row or cell and wavefront.
template <bool CELLS>
__device__ __forceinline__ void row_count_at(const DevState& s, const Grid& g, uint32_t* __restrict__ row_count,
                                             uint32_t* __restrict__ first, uint2* __restrict__ where, size_t i, size_t n) {
    const bool valid = i < n;
    uint32_t row = 0, key = 0xffffffffu;
    if (valid) {
        const int cls = h_class(s.d[H][i], g.hmin, g.nclass);
        int c[3];
        cell_of(g.c[cls], s.d[X][i], s.d[Y][i], s.d[Z][i], c);
        const uint32_t mor = row_key(0u, uint32_t(c[1]), uint32_t(c[2]), 0);
        row = g.c[cls].slot0 + mor;
        key = CELLS ? g.c[cls].base + (mor << g.c[cls].bits) + uint32_t(c[0]) : (row << 8) | uint32_t(c[0]);
    }
    // the lanes of one bucket: its first lane adds their number, each gets its rank among them
    const WaveRun run = wave_run(CELLS ? key : row, valid);
    uint32_t base = 0;
    if (valid && run.leader == (threadIdx.x & 63u)) {
        base = atomicAdd(CELLS ? &first[key] : &row_count[row], run.total);
        if (CELLS) atomicAdd(&row_count[row], run.total);
    }
    base = uint32_t(__shfl(int(base), int(run.leader), 64));
    if (valid) where[i] = make_uint2(key, base + run.before);
}

template <bool CELLS>
__global__ void __launch_bounds__(BLOCK) k_row_count(DevState s, Grid g, uint32_t* __restrict__ row_count,
                                                     uint32_t* __restrict__ first, uint2* __restrict__ where, size_t n) {
    row_count_at<CELLS>(s, g, row_count, first, where, size_t(blockIdx.x) * blockDim.x + threadIdx.x, n);
}

// row_start = exclusive prefix sums of the counts (slots + 1 entries).  Block b sums the counts before its tile of
// SCAN_TILE itself, and scans its tile: no second pass and no waiting for other blocks (53k slots at the 1M impact:
// 14 blocks, the last reading 230 KB; one block stepping through all of them took 25 us).
constexpr uint32_t SCAN_BLOCK = 1024, SCAN_TILE = 4 * SCAN_BLOCK;
__device__ __forceinline__ void row_scan_tile(const uint32_t* __restrict__ row_count, uint32_t* __restrict__ row_start,
                                              uint32_t block) {
    __shared__ uint32_t wave_sum[2][SCAN_BLOCK / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    // the arrays hold whole tiles, the entries past the last row zero
    const uint4* in = reinterpret_cast<const uint4*>(row_count);
    const uint32_t tile = block * SCAN_BLOCK;  // in quads
    uint32_t prior = 0;
    for (uint32_t t = threadIdx.x; t < tile; t += SCAN_BLOCK) {
        const uint4 q = in[t];
        prior += q.x + q.y + q.z + q.w;
    }
    const uint4 c = in[tile + threadIdx.x];
    const uint32_t sum = c.x + c.y + c.z + c.w;
    uint32_t incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = uint32_t(__shfl_up(int(incl), o, 64));
        if (lane >= uint32_t(o)) incl += u;
    }
    for (int o = 32; o > 0; o >>= 1) prior += uint32_t(__shfl_xor(int(prior), o, 64));
    if (lane == 63u) {
        wave_sum[0][wave] = incl;
        wave_sum[1][wave] = prior;
    }
    __syncthreads();
    uint32_t run = incl - sum;
    for (uint32_t w = 0; w < SCAN_BLOCK / 64; ++w) run += wave_sum[1][w] + (w < wave ? wave_sum[0][w] : 0u);
    uint4 o;
    o.x = run;
    o.y = o.x + c.x;
    o.z = o.y + c.y;
    o.w = o.z + c.z;
    reinterpret_cast<uint4*>(row_start)[tile + threadIdx.x] = o;
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_row_scan(const uint32_t* __restrict__ row_count,
                                                         uint32_t* __restrict__ row_start) {
    row_scan_tile(row_count, row_start, blockIdx.x);
}

// bucket[row_start + rank] = (particle, x), or by CELLS (particle, particles of its wavefront's run) at its cell's first
// position + rank.  The row counts go back to zero for the next search.
template <bool CELLS>
__device__ __forceinline__ void row_scatter_at(const uint2* __restrict__ where, const uint32_t* __restrict__ row_start,
                                               const uint32_t* __restrict__ first, uint32_t* __restrict__ row_count,
                                               uint32_t slots, uint2* __restrict__ bucket, size_t i, size_t threads,
                                               size_t n) {
    for (size_t t = i; t < slots; t += threads) row_count[t] = 0u;
    const bool valid = i < n;
    const uint2 w = valid ? where[i] : make_uint2(0u, 0u);
    if constexpr (CELLS) {
        const uint32_t total = wave_run(w.x, valid).total;
        if (valid) bucket[first[w.x] + w.y] = make_uint2(uint32_t(i), total);
    } else if (valid) {
        bucket[row_start[w.x >> 8] + w.y] = make_uint2(uint32_t(i), w.x & 255u);
    }
}

template <bool CELLS>
__global__ void __launch_bounds__(BLOCK) k_row_scatter(const uint2* __restrict__ where,
                                                       const uint32_t* __restrict__ row_start,
                                                       const uint32_t* __restrict__ first,
                                                       uint32_t* __restrict__ row_count, uint32_t slots,
                                                       uint2* __restrict__ bucket, size_t n) {
    row_scatter_at<CELLS>(where, row_start, first, row_count, slots, bucket, size_t(blockIdx.x) * blockDim.x + threadIdx.x,
                          size_t(gridDim.x) * blockDim.x, n);
}

// One wavefront per row: the counts of its cells in `first` become first sorted positions, with that of the row's end in
// the slot past its last cell.  The cells of rows without particles keep their zeros, equal entries, so that every x-run
// of them reads as empty.
__device__ __forceinline__ void cell_starts_at(const Grid& g, const uint32_t* __restrict__ row_start,
                                               uint32_t* __restrict__ first, size_t rows, size_t q) {
    int cls = 0;
    uint32_t cy = 0, cz = 0;
    if (q >= rows || !row_of(g, q, cls, cy, cz)) return;  // uniform over the wavefront
    const GridClass& G = g.c[cls];
    const uint32_t lane = threadIdx.x & 63u, mor = row_key(0u, cy, cz, 0);
    uint32_t run = row_start[G.slot0 + mor];
    if (row_start[G.slot0 + mor + 1u] == run) return;
    uint32_t* cell = first + G.base + (mor << G.bits);
    for (uint32_t x0 = 0; x0 <= uint32_t(G.dim[0]); x0 += 64u) {
        const uint32_t x = x0 + lane;
        const uint32_t c = x < uint32_t(G.dim[0]) ? cell[x] : 0u;
        uint32_t incl = c;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t u = uint32_t(__shfl_up(int(incl), o, 64));
            if (lane >= uint32_t(o)) incl += u;
        }
        if (x <= uint32_t(G.dim[0])) cell[x] = run + incl - c;
        run += uint32_t(__shfl(int(incl), 63, 64));
    }
}

__global__ void __launch_bounds__(BLOCK) k_cell_starts(Grid g, const uint32_t* __restrict__ row_start,
                                                       uint32_t* __restrict__ first, size_t rows) {
    cell_starts_at(g, row_start, first, rows, size_t(blockIdx.x) * (BLOCK / 64) + (threadIdx.x >> 6));
}

// order[] by CELLS: particle i goes behind the lower particles of its cell, those of lower wavefronts a run at a time.
__device__ __forceinline__ void cell_order_at(const uint2* __restrict__ where, const uint32_t* __restrict__ first,
                                              const uint2* __restrict__ bucket, uint32_t* __restrict__ order, size_t i,
                                              size_t n) {
    if (i >= n) return;
    const uint2 w = where[i];
    const uint32_t a = first[w.x], b = first[w.x + 1u], wave = uint32_t(i >> 6);
    uint32_t r = a;
    for (uint32_t j = a; j < b;) {
        const uint2 run = bucket[j];
        if ((run.x >> 6) < wave) r += run.y;
        if ((run.x >> 6) == wave) r += a + w.y - j;  // its own run: those before it
        j += max(run.y, 1u);
    }
    order[r] = uint32_t(i);
}

__global__ void __launch_bounds__(BLOCK) k_cell_order(const uint2* __restrict__ where, const uint32_t* __restrict__ first,
                                                      const uint2* __restrict__ bucket, uint32_t* __restrict__ order,
                                                      size_t n) {
    cell_order_at(where, first, bucket, order, size_t(blockIdx.x) * blockDim.x + threadIdx.x, n);
}

// One wavefront per row (y < dim_y, z < dim_z of every class): its particles ordered by (x, particle) into order[],
// and first[cell] = the first sorted position whose cell is >= cell, for x in [0, dim_x].  Up to ROW_WAVE
// particles in LDS: counted by x, placed, and each ranked among those of its own cell (0.6 per cell at the
// impact).  Longer rows (rare here, see sort_by_cells) take the block together, one after the other, the same way, and
// beyond ROW_BLOCK particles through the row's part of scratch[] (the particles' rows, used up by the scatter).
constexpr uint32_t ROW_WAVE = 512, ROW_BLOCK = 2048;
struct alignas(16) RowStage {  // start is read 16 bytes at a time
    uint32_t start[256];      // counts by x, then their exclusive prefix sums
    uint32_t idx[ROW_WAVE];   // particles placed by cell
};
struct alignas(16) LongRowStage {
    uint32_t start[256];
    uint32_t next[256];       // the next free place of each cell
    uint2 placed[ROW_BLOCK];
};

// start[0..256) from counts to exclusive prefix sums, by one wavefront.
__device__ __forceinline__ void scan_cells(uint32_t* start) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint4 c = reinterpret_cast<const uint4*>(start)[lane];
    const uint32_t sum = c.x + c.y + c.z + c.w;
    uint32_t incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = uint32_t(__shfl_up(int(incl), o, 64));
        if (lane >= uint32_t(o)) incl += u;
    }
    uint4 st;
    st.x = incl - sum;
    st.y = st.x + c.x;
    st.z = st.y + c.y;
    st.w = st.z + c.z;
    reinterpret_cast<uint4*>(start)[lane] = st;
}

// The block's order of one long row of m particles from sorted position f on.
__device__ __forceinline__ void order_long_row(LongRowStage& S, const uint2* __restrict__ row, uint2* placed,
                                               uint32_t* __restrict__ order, uint32_t* __restrict__ cell, uint32_t dimx,
                                               uint32_t f, uint32_t m) {
    for (uint32_t x = threadIdx.x; x < 256u; x += BLOCK) S.start[x] = 0u;
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < m; p += BLOCK) atomicAdd(&S.start[row[p].y], 1u);
    __syncthreads();
    if (threadIdx.x < 64u) scan_cells(S.start);
    __syncthreads();
    for (uint32_t x = threadIdx.x; x < 256u; x += BLOCK) {
        S.next[x] = S.start[x];
        if (x <= dimx) cell[x] = f + S.start[x];
    }
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < m; p += BLOCK) {
        const uint2 e = row[p];
        placed[atomicAdd(&S.next[e.y], 1u)] = e;
    }
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < m; p += BLOCK) {
        const uint2 e = placed[p];
        const uint32_t a = S.start[e.y], b = S.start[e.y + 1u];  // x <= 250: x + 1 is an entry
        uint32_t r = a;
        for (uint32_t j = a; j < b; ++j) r += placed[j].x < e.x ? 1u : 0u;
        order[f + r] = e.x;
    }
    __syncthreads();
}

__device__ __forceinline__ void row_order_block(const Grid& g, const uint32_t* __restrict__ row_start,
                                                const uint2* __restrict__ bucket, uint2* __restrict__ scratch,
                                                uint32_t* __restrict__ order, uint32_t* __restrict__ first, size_t rows,
                                                size_t block) {
    constexpr int WAVES = BLOCK / 64;
    union Lds {
        RowStage stage[WAVES];
        LongRowStage row;
    };
    static_assert(alignof(Lds) >= 16, "RowStage::start is read 16 bytes at a time");
    __shared__ Lds lds;
    __shared__ uint32_t long_row[WAVES][4];  // first position, particles, cell base and dim_x of a long row
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const size_t q = block * WAVES + wave;
    int cls = 0;
    uint32_t cy = 0, cz = 0;
    const bool valid = q < rows && row_of(g, q, cls, cy, cz);
    const GridClass& G = g.c[cls];
    const uint32_t mor = row_key(0u, cy, cz, 0);
    const uint32_t dimx = uint32_t(G.dim[0]), cell0 = G.base + (mor << G.bits);
    uint32_t s0 = 0, cnt = 0;
    if (valid) {
        s0 = row_start[G.slot0 + mor];
        cnt = row_start[G.slot0 + mor + 1u] - s0;
    }
    s0 = __builtin_amdgcn_readfirstlane(s0);
    cnt = __builtin_amdgcn_readfirstlane(cnt);
    if (lane == 0) long_row[wave][1] = 0u;
    if (valid && cnt == 0) {
        for (uint32_t x = lane; x <= dimx; x += 64u) first[cell0 + x] = s0;
    } else if (valid && cnt <= ROW_WAVE) {
        RowStage& S = lds.stage[wave];
        reinterpret_cast<uint4*>(S.start)[lane] = make_uint4(0u, 0u, 0u, 0u);
        wave_sync();
        uint2 e[ROW_WAVE / 64];
        uint32_t rank[ROW_WAVE / 64];
#pragma unroll
        for (uint32_t k = 0; k < ROW_WAVE / 64; ++k) {
            if (64u * k >= cnt) break;
            if (64u * k + lane < cnt) {
                e[k] = bucket[s0 + 64u * k + lane];
                rank[k] = atomicAdd(&S.start[e[k].y], 1u);
            }
        }
        wave_sync();
        scan_cells(S.start);
        wave_sync();
        for (uint32_t x = lane; x <= dimx; x += 64u) first[cell0 + x] = s0 + S.start[x];
#pragma unroll
        for (uint32_t k = 0; k < ROW_WAVE / 64; ++k) {
            if (64u * k >= cnt) break;
            if (64u * k + lane < cnt) S.idx[S.start[e[k].y] + rank[k]] = e[k].x;
        }
        wave_sync();
#pragma unroll
        for (uint32_t k = 0; k < ROW_WAVE / 64; ++k) {
            if (64u * k >= cnt) break;
            if (64u * k + lane < cnt) {
                const uint32_t a = S.start[e[k].y], b = S.start[e[k].y + 1u];  // x <= 250: x + 1 is an entry
                uint32_t r = a;
                for (uint32_t j = a; j < b; ++j) r += S.idx[j] < e[k].x ? 1u : 0u;
                order[s0 + r] = e[k].x;
            }
        }
    } else if (valid && lane == 0) {
        long_row[wave][0] = s0;
        long_row[wave][1] = cnt;
        long_row[wave][2] = cell0;
        long_row[wave][3] = dimx;
    }
    __syncthreads();
    for (int w = 0; w < WAVES; ++w) {
        const uint32_t f = long_row[w][0], m = long_row[w][1];
        if (m == 0) continue;
        order_long_row(lds.row, bucket + f, m <= ROW_BLOCK ? lds.row.placed : scratch + f, order, first + long_row[w][2],
                       long_row[w][3], f, m);
    }
}

__global__ void __launch_bounds__(BLOCK) k_row_order(Grid g, const uint32_t* __restrict__ row_start,
                                                     const uint2* __restrict__ bucket, uint2* __restrict__ scratch,
                                                     uint32_t* __restrict__ order, uint32_t* __restrict__ first,
                                                     size_t rows) {
    row_order_block(g, row_start, bucket, scratch, order, first, rows, blockIdx.x);
}

// Pack the neighbour-side data of particle order[k] into rec[k].
// Origin-relative FP32 position of the screened neighbour test (one rounding of the FP64 offset).
__device__ __forceinline__ float4 screen_pos(const Screen& sc, double x, double y, double z, double h) {
    return make_float4(float(x - sc.o[0]), float(y - sc.o[1]), float(z - sc.o[2]), float(h));
}

__device__ __forceinline__ void pack_at(const DevState& s, const Params& prm, const uint32_t* __restrict__ order,
                                        PairRec* __restrict__ rec, double4* __restrict__ pos,
                                        float4* __restrict__ posf, const Screen& sc, uint32_t* __restrict__ group,
                                        size_t k) {
#pragma clang fp contract(off)
    const uint32_t i = order[k];
    PairRec r;
    r.x = s.d[X][i];
    r.y = s.d[Y][i];
    r.z = s.d[Z][i];
    r.h = s.d[H][i];
    r.vx = s.d[VX][i];
    r.vy = s.d[VY][i];
    r.vz = s.d[VZ][i];
    r.m = s.d[M][i];
    const double rho = s.d[RHO][i];
    const double rho2 = rho * rho;
    r.rho = rho;
    r.cs = s.d[CS][i];
    r.pr = s.d[P][i] / rho2;  // StandardForceDiscr: p / sqr(rho) (EquationTerm.cpp:20-23)
    if (prm.solid_stress) {
        r.sxx = s.d[SXX][i] / rho2;
        r.syy = s.d[SYY][i] / rho2;
        r.sxy = s.d[SXY][i] / rho2;
        r.sxz = s.d[SXZ][i] / rho2;
        r.syz = s.d[SYZ][i] / rho2;
    } else {
        r.sxx = r.syy = r.sxy = r.sxz = r.syz = 0.0;
    }
    rec[k] = r;
    pos[k] = make_double4(r.x, r.y, r.z, r.h);
    if (sc.on) posf[k] = screen_pos(sc, r.x, r.y, r.z, r.h);
    // DerivativeTemplate / AccelerationTemplate sum filter (DerivativeHelpers.h:132-139,262-269):
    // a pair enters the SUM_ONLY_UNDAMAGED sums iff both flags are equal and both reductions nonzero.
    uint32_t gid = 0;
    if (prm.sum_only_undamaged && prm.has_reduce) {
        gid = (s.d[RED][i] == 0.0) ? NO_GROUP : s.u[FLAG][i];
    }
    group[k] = gid;
}

__global__ void __launch_bounds__(BLOCK) k_pack(DevState s, Params prm, const uint32_t* __restrict__ order,
                                                PairRec* __restrict__ rec, double4* __restrict__ pos,
                                                float4* __restrict__ posf, Screen sc, uint32_t* __restrict__ group,
                                                size_t n) {
    const size_t k = size_t(xcd_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x;
    if (k < n) pack_at(s, prm, order, rec, pos, posf, sc, group, k);
}

// The pair test of SymmetricSolver<3>::loop (core/sph/solvers/SymmetricSolver.cpp:126-131) evaluated
// bit for bit: getSqrLength sums the squares left to right without contraction and
// sqr(2 * 0.5 * (h_i + h_j)) == (h_i + h_j)^2 exactly.
__device__ __forceinline__ bool exact_pair(double xi, double yi, double zi, double hi, double xj, double yj, double zj,
                                           double hj) {
    const double dx = rn_sub(xi, xj), dy = rn_sub(yi, yj), dz = rn_sub(zi, zj);
    const double d2 = rn_add(rn_add(rn_mul(dx, dx), rn_mul(dy, dy)), rn_mul(dz, dz));
    const double hs = rn_add(hi, hj);
    return d2 < rn_mul(hs, hs);
}

// Candidates loaded per batch in the neighbour-list kernel: 4 FP32 positions (16 B each) in the screened
// test, 2 FP64 positions (32 B) in the plain one (measured at the 1M impact: 0.305 / 0.313 ms screened at
// 4 / 2, 0.400 / 0.363 ms plain).
template <bool SCREEN>
constexpr uint32_t LIST_BATCH = SCREEN ? 4u : 2u;

// One thread per particle (sorted position k).  For every smoothing-length class whose bounding box
// lies within h_i + h_max(class), the cells of that class within that radius are scanned with the exact
// pair test.  Neighbour positions are buffered four at a time in registers and stored as one 16-byte
// quad at list_quad(k, j, kmax / 4).
//
// With SCREEN, candidates are first tested in FP32 on origin-relative positions (16 bytes per candidate
// instead of 32).  The FP32 squared distance and radius carry a relative error below sc.band (bounded on
// the host from the domain extent and h_min), so d2 < R2 (1 - band) and d2 > R2 (1 + band) decide the
// exact test; only candidates inside the band are re-tested in FP64, and the pair set is unchanged.
template <bool SCREEN>
__device__ __forceinline__ void neighbor_list_at(const double4* __restrict__ pos, const float4* __restrict__ posf,
                                                 const Screen& sc, const Grid& g, const uint32_t* __restrict__ first,
                                                 uint32_t* __restrict__ list, uint32_t* __restrict__ count,
                                                 uint32_t kmax, uint32_t* overflow, size_t k) {
    const double4 me = pos[k];
    const float4 mf = SCREEN ? posf[k] : make_float4(0.f, 0.f, 0.f, 0.f);
    const double p[3] = { me.x, me.y, me.z };
    uint4* list4 = reinterpret_cast<uint4*>(list);
    // the last four entries, oldest first (shifted in: no register indexed by the count)
    uint32_t b0 = 0, b1 = 0, b2 = 0, b3 = 0;
    uint32_t cnt = 0;
    auto append = [&](uint32_t k2) {
        b0 = b1;
        b1 = b2;
        b2 = b3;
        b3 = k2;
        ++cnt;
        if ((cnt & 3u) == 0 && cnt <= kmax) {
            list4[list_quad(k, (cnt >> 2) - 1, kmax >> 2)] = make_uint4(b0, b1, b2, b3);
        }
    };
    for (int cls = 0; cls < g.nclass; ++cls) {
        const GridClass& G = g.c[cls];
        if (G.empty) continue;
        const double R = me.w + G.hmax;  // h_i + h_j <= R for every member j
        double d2b = 0.0;
        for (int a = 0; a < 3; ++a) {
            const double t = dmax(G.lo[a] - p[a], p[a] - G.hi[a]);
            if (t > 0.0) d2b += t * t;
        }
        if (d2b > R * R * (1.0 + 1e-6)) continue;
        // Rows of cells (cy, cz) whose yz-square lies farther than R hold no neighbour; in the others a
        // neighbour lies within the chord half-width w = sqrt(R^2 - d_yz^2) of the particle along x, and
        // the cells of that x-run are one contiguous range of sorted particles.  The planes cz within R,
        // the rows cy of a plane within R (half-width sqrt(R^2 - d_z^2) in y) and the x-runs are computed
        // directly, so every step of the walk yields a row.  The geometry is evaluated in FP32 in cell
        // units with R widened by 1e-3 cells: the FP32 errors (square roots of about 1 ulp included; below
        // 1e-4 cells for the at most a few thousand cells per axis) then only ever add candidates, and the
        // exact test decides.  The ranges of the next row are loaded before the current row's candidates
        // are tested, so the two loads overlap.
        const float pcx = float((p[0] - G.lo[0]) * G.inv_cell);
        const float pcy = float((p[1] - G.lo[1]) * G.inv_cell);
        const float pcz = float((p[2] - G.lo[2]) * G.inv_cell);
        const float Rc = float(R * G.inv_cell) * (1.0f + 1e-6f) + 1e-3f;
        const float R2c = Rc * Rc;
        const int zlast = min(G.dim[2] - 1, int(floorf(pcz + Rc)));
        int cz = max(0, int(floorf(pcz - Rc))) - 1;  // the plane before the first
        int cy = 0, ylast = -1;                       // the row and the last row of the plane within R
        float tz2 = 0.0f;
        uint32_t zkey = 0, ykey = 0;
        // the next row within R: its first and past-the-end sorted positions (an empty range where the
        // x-run misses the grid)
        auto next_row = [&](uint32_t& b, uint32_t& e) -> bool {
            if (++cy > ylast) {
                for (;;) {
                    if (++cz > zlast) return false;
                    const float fz = float(cz);
                    const float tz = fmaxf(fmaxf(fz - pcz, pcz - (fz + 1.0f)), 0.0f);
                    tz2 = tz * tz;
                    if (tz2 > R2c) continue;
                    const float wy = __builtin_amdgcn_sqrtf(R2c - tz2);
                    cy = max(0, int(floorf(pcy - wy)));
                    ylast = min(G.dim[1] - 1, int(floorf(pcy + wy)));
                    if (cy > ylast) continue;
                    zkey = spread2(uint32_t(cz)) << 1;
                    ykey = spread2(uint32_t(cy));
                    break;
                }
            } else {
                // spread2(cy + 1) from spread2(cy): adding one to the even-bit interleaved value with the odd
                // bits set carries through them
                ykey = ((ykey | 0xaaaaaaaau) + 1u) & 0x55555555u;
            }
            const float fy = float(cy);
            const float ty = fmaxf(fmaxf(fy - pcy, pcy - (fy + 1.0f)), 0.0f);
            const float w = __builtin_amdgcn_sqrtf(fmaxf(R2c - (tz2 + ty * ty), 0.0f));
            const int x0 = max(0, int(floorf(pcx - w)));
            const int x1 = min(G.dim[0] - 1, int(floorf(pcx + w)));
            if (x0 > x1) {
                b = e = 0u;
                return true;
            }
            const uint32_t row = G.base + ((ykey | zkey) << G.bits);
            b = first[row + uint32_t(x0)];
            e = first[row + uint32_t(x1) + 1u];
            return true;
        };
        uint32_t nb = 0, ne = 0;
        bool more = next_row(nb, ne);
        while (more) {
            const uint32_t b = nb, e = ne;
            more = next_row(nb, ne);
            // candidates in batches of LIST_BATCH<SCREEN>: all loads of a batch are issued before the first
            // test; a batch may read up to LIST_BATCH - 1 entries past e, which are never tested (e <= n and
            // the arrays hold POS_SLACK >= LIST_BATCH entries past n)
            for (uint32_t k0 = b; k0 < e; k0 += LIST_BATCH<SCREEN>) {
                if (SCREEN) {
                    float4 o[LIST_BATCH<true>];
#pragma unroll
                    for (uint32_t u = 0; u < LIST_BATCH<true>; ++u) o[u] = posf[k0 + u];  // POS_SLACK past n
#pragma unroll
                    for (uint32_t u = 0; u < LIST_BATCH<true>; ++u) {
                        const uint32_t k2 = k0 + u;
                        if (k2 >= e) break;
                        const float dx = mf.x - o[u].x, dy = mf.y - o[u].y, dz = mf.z - o[u].z;
                        const float d2 = dx * dx + dy * dy + dz * dz;
                        const float hs = mf.w + o[u].w;
                        const float rr = hs * hs;
                        bool hit = d2 < rr * sc.lo;
                        if (!hit && !(d2 > rr * sc.hi)) {
                            const double4 od = pos[k2];
                            hit = exact_pair(me.x, me.y, me.z, me.w, od.x, od.y, od.z, od.w);
                        }
                        if (hit && k2 != k) append(k2);
                    }
                } else {
                    double4 o[LIST_BATCH<false>];
#pragma unroll
                    for (uint32_t u = 0; u < LIST_BATCH<false>; ++u) o[u] = pos[k0 + u];  // POS_SLACK past n
#pragma unroll
                    for (uint32_t u = 0; u < LIST_BATCH<false>; ++u) {
                        const uint32_t k2 = k0 + u;
                        if (k2 >= e) break;
                        const bool hit = exact_pair(me.x, me.y, me.z, me.w, o[u].x, o[u].y, o[u].z, o[u].w);
                        if (hit && k2 != k) append(k2);
                    }
                }
            }
        }
    }
    if ((cnt & 3u) != 0 && cnt < kmax) {
        // the r = cnt % 4 entries of the last quad are b(4-r) .. b3; the rest of the quad is not read
        const uint32_t r = cnt & 3u;
        const uint4 q = r == 1 ? make_uint4(b3, 0u, 0u, 0u) : (r == 2 ? make_uint4(b2, b3, 0u, 0u) : make_uint4(b1, b2, b3, 0u));
        list4[list_quad(k, cnt >> 2, kmax >> 2)] = q;
    }
    count[k] = cnt;
    if (cnt > kmax) atomicOr(overflow, 1u);
}

// The same list, with the same entries in the same order, from LIST_LANES lanes per particle: each lane takes one
// row of cells at a time and counts its hits, a prefix sum over the group places them.  One lane per particle
// walks its ~37 rows one after the other, each row two dependent loads (80 us whatever the particle count, until
// the particles fill the chip); here the group's rows are in flight together.  The rows are numbered over the
// rectangle of planes and rows around the particle; those of its corners yield no candidates.  Measured against single
// lanes (lists_shared); other group sizes were not.
constexpr uint32_t LIST_LANES = 16;
template <bool SCREEN>
__device__ __forceinline__ void neighbor_list_shared_at(const double4* __restrict__ pos,
                                                        const float4* __restrict__ posf, const Screen& sc,
                                                        const Grid& g, const uint32_t* __restrict__ first,
                                                        uint32_t* __restrict__ list, uint32_t* __restrict__ count,
                                                        uint32_t kmax, uint32_t* overflow, size_t k, uint32_t sub) {
    const double4 me = pos[k];
    const float4 mf = SCREEN ? posf[k] : make_float4(0.f, 0.f, 0.f, 0.f);
    const double p[3] = { me.x, me.y, me.z };
    uint32_t cnt = 0;
    auto hits = [&](uint32_t k2) {
        if (SCREEN) {
            const float4 o = posf[k2];
            const float dx = mf.x - o.x, dy = mf.y - o.y, dz = mf.z - o.z;
            const float d2 = dx * dx + dy * dy + dz * dz;
            const float hs = mf.w + o.w;
            const float rr = hs * hs;
            if (d2 < rr * sc.lo) return k2 != k;
            if (d2 > rr * sc.hi) return false;
        }
        const double4 o = pos[k2];
        return exact_pair(me.x, me.y, me.z, me.w, o.x, o.y, o.z, o.w) && k2 != k;
    };
    auto put = [&](uint32_t at, uint32_t k2) {
        if (at < kmax) list[4 * list_quad(k, at >> 2, kmax >> 2) + (at & 3u)] = k2;
    };
    for (int cls = 0; cls < g.nclass; ++cls) {
        const GridClass& G = g.c[cls];
        if (G.empty) continue;
        const double R = me.w + G.hmax;  // h_i + h_j <= R for every member j
        double d2b = 0.0;
        for (int a = 0; a < 3; ++a) {
            const double t = dmax(G.lo[a] - p[a], p[a] - G.hi[a]);
            if (t > 0.0) d2b += t * t;
        }
        if (d2b > R * R * (1.0 + 1e-6)) continue;
        // the geometry of neighbor_list_at: FP32 in cell units, R widened by 1e-3 cells
        const float pcx = float((p[0] - G.lo[0]) * G.inv_cell);
        const float pcy = float((p[1] - G.lo[1]) * G.inv_cell);
        const float pcz = float((p[2] - G.lo[2]) * G.inv_cell);
        const float Rc = float(R * G.inv_cell) * (1.0f + 1e-6f) + 1e-3f;
        const float R2c = Rc * Rc;
        const int z0 = max(0, int(floorf(pcz - Rc))), z1 = min(G.dim[2] - 1, int(floorf(pcz + Rc)));
        const int y0 = max(0, int(floorf(pcy - Rc))), y1 = min(G.dim[1] - 1, int(floorf(pcy + Rc)));
        const int ny = y1 - y0 + 1, rows = z1 < z0 || ny <= 0 ? 0 : (z1 - z0 + 1) * ny;
        for (int r0 = 0; r0 < rows; r0 += int(LIST_LANES)) {  // uniform over the group
            const int r = r0 + int(sub);
            uint32_t b = 0, e = 0;
            if (r < rows) {
                const int dz = r / ny;
                const int cz = z0 + dz, cy = y0 + (r - dz * ny);
                const float fz = float(cz), fy = float(cy);
                const float tz = fmaxf(fmaxf(fz - pcz, pcz - (fz + 1.0f)), 0.0f);
                const float ty = fmaxf(fmaxf(fy - pcy, pcy - (fy + 1.0f)), 0.0f);
                const float t2 = R2c - (tz * tz + ty * ty);
                if (t2 >= 0.0f) {
                    const float w = __builtin_amdgcn_sqrtf(t2);
                    const int x0 = max(0, int(floorf(pcx - w)));
                    const int x1 = min(G.dim[0] - 1, int(floorf(pcx + w)));
                    if (x0 <= x1) {
                        const uint32_t row = G.base + row_key(0u, uint32_t(cy), uint32_t(cz), G.bits);
                        b = first[row + uint32_t(x0)];
                        e = first[row + uint32_t(x1) + 1u];
                    }
                }
            }
            // the hits of the first 64 candidates as a mask; the rest of a longer row is counted here and
            // tested again when its hits are placed
            unsigned long long mask = 0ull;
            uint32_t mine = 0;
            for (uint32_t k2 = b; k2 < e; ++k2) {
                if (hits(k2)) {
                    if (k2 - b < 64u) mask |= 1ull << (k2 - b);
                    ++mine;
                }
            }
            uint32_t incl = mine;
            for (uint32_t o = 1; o < LIST_LANES; o <<= 1) {
                const uint32_t v = __shfl_up(incl, o, int(LIST_LANES));
                if (sub >= o) incl += v;
            }
            uint32_t at = cnt + incl - mine;
            for (unsigned long long m = mask; m != 0ull; m &= m - 1ull) put(at++, b + uint32_t(__builtin_ctzll(m)));
            for (uint32_t k2 = b + 64u; k2 < e; ++k2) {
                if (hits(k2)) put(at++, k2);
            }
            cnt += __shfl(incl, int(LIST_LANES) - 1, int(LIST_LANES));
        }
    }
    if (sub == 0) {
        count[k] = cnt;
        if (cnt > kmax) atomicOr(overflow, 1u);
    }
}

template <bool SCREEN>
__global__ void __launch_bounds__(BLOCK) k_neighbor_lists_shared(const double4* __restrict__ pos,
                                                                 const float4* __restrict__ posf, Screen sc, Grid g,
                                                                 const uint32_t* __restrict__ first,
                                                                 uint32_t* __restrict__ list,
                                                                 uint32_t* __restrict__ count, uint32_t kmax,
                                                                 uint32_t* overflow, size_t n) {
    const size_t t = size_t(xcd_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x;
    const size_t k = t / LIST_LANES;
    if (k < n) {  // uniform over each group of lanes
        neighbor_list_shared_at<SCREEN>(pos, posf, sc, g, first, list, count, kmax, overflow, k, uint32_t(t % LIST_LANES));
    }
}

template <bool SCREEN>
__global__ void __launch_bounds__(BLOCK) k_neighbor_lists(const double4* __restrict__ pos,
                                                          const float4* __restrict__ posf, Screen sc, Grid g,
                                                          const uint32_t* __restrict__ first,
                                                          uint32_t* __restrict__ list, uint32_t* __restrict__ count,
                                                          uint32_t kmax, uint32_t* overflow, size_t n) {
    const size_t k = size_t(xcd_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x;
    if (k < n) neighbor_list_at<SCREEN>(pos, posf, sc, g, first, list, count, kmax, overflow, k);
}

// LutKernel<3>::gradImpl (core/sph/kernel/Kernel.h:129-144), linear interpolation in q^2, in two parts: the table's two
// entries, and what is made of them.  One 16-byte load at 8-byte alignment fetches both.
struct LutPair {
    double a, b, ratio;
    bool inside;
    __device__ __forceinline__ double value() const { return inside ? fma(b, ratio, a * (1.0 - ratio)) : 0.0; }
};

__device__ __forceinline__ LutPair lut_fetch(const double* __restrict__ grads, double q2) {
    typedef double Two __attribute__((ext_vector_type(2), aligned(8)));
    LutPair p;
    p.inside = q2 < 4.0;  // outside the support (also NaN, which must not become an index) the value is 0
    const double fi = double(LUT_ENTRIES / 4) * (p.inside ? q2 : 0.0);
    const uint32_t i1 = uint32_t(fi);
    p.ratio = fi - double(i1);
    const Two v = *reinterpret_cast<const Two*>(grads + i1);
    p.a = v.x;
    p.b = v.y;
    return p;
}

// The pair sums of particle i that the finalize, the corrector and the criteria use: acceleration, du,
// velocity divergence and gradient (xx, yy, zz, xy, xz, yz).  The fused pair kernels hand them over in
// registers; the separate passes read them from the state (sums_of).
struct PairSums {
    double a[3], du, divv, g[6];
};
__device__ __forceinline__ PairSums sums_of(const DevState& s, bool solid, size_t i) {
    PairSums ps;
    for (int k = 0; k < 3; ++k) ps.a[k] = s.d[AX + k][i];
    ps.du = s.d[DU][i];
    ps.divv = s.d[DIVV][i];
    for (int k = 0; k < 6; ++k) ps.g[k] = solid ? s.d[GXX + k][i] : 0.0;
    return ps;
}
__device__ void finalize_at(DevState& s, const osph_material& m, const Params& prm, size_t i, const PairSums& ps);
__device__ void correct_at(DevState& s, const osph_material& m, const Params& prm, double dt, size_t i,
                           const double a[3]);
__device__ void criteria_values(const DevState& s, const osph_material& m, const Params& prm, size_t i,
                                const double a[3], double divv, double out[4]);
__device__ void reduce_criteria(double v[4], unsigned long long* mins);


// Per-wavefront LDS stage of neighbour records: 64 records of CH 16-byte chunks.  Chunk c of lane r's record lies at
// place c ^ swizzle(r) of the record, so that 16 consecutive lanes' reads of one chunk fall on all 64 banks.
template <typename Rec>
struct StageOf {
    static constexpr uint32_t CH = sizeof(Rec) / 16;
    static constexpr uint32_t WORDS = 64 * CH;  // uint4 per wavefront
    static_assert(sizeof(Rec) % 16 == 0 && (CH == 4 || CH == 8), "a power of two of 16-byte chunks");
    static __device__ __forceinline__ uint32_t swizzle(uint32_t r) { return (r / (16u / CH)) % CH; }
};

// The neighbour lists of a wavefront's particles, one on each lane, entry t of every list at step t: x = early(record,
// entry) on all lanes, then f(record, entry, x) on those whose list has the entry (the others hold their own record).
// Every lane of the wavefront must call this.
//
// A lane that loads a whole record by itself touches a cache line of its own in every load instruction, CH times as
// many as when consecutive lanes fetch the chunks of one record.  So the wavefront fetches the 64 records of a step
// together, straight into its LDS stage (no registers in between), while the terms of the step before are evaluated;
// early is where f's own loads go, ahead of the next records'.  The trip count is the wavefront's and the steps of a
// list quad are written out, so that the accumulators and the quad stay where they are (with a condition on each lane
// the compiler moved them about, 40 of 180 instructions a step).  Per step at the 1M impact, direct loads or loads
// staged through registers -> this: mixed 551 -> 488 us, FP64 1035 -> 804, 531k particles FP64 434 -> 378.  Mixed is
// bound by the issue (139 instructions a step, 75 % of the issue slots), FP64 by the L1 cache (168 accesses and 62
// line fills a step, 40 % of them the kernel table's).  Buffer loads with 32-bit offsets in place of the global ones:
// 490 and 777 us, but no record past 4 GB; the table's entries computed instead: 762 us; wavefronts of five to a SIMD
// for the mixed kernel (96 registers): 496 us.
template <typename Rec, typename E, typename F>
__device__ __forceinline__ void for_each_neighbor(const Rec* __restrict__ rec, const uint32_t* __restrict__ list,
                                                  size_t k, uint32_t quads, uint32_t listed, uint4* stage, E&& early,
                                                  F&& f) {
    using S = StageOf<Rec>;
    constexpr uint32_t CH = S::CH, PER = 64u / CH;  // records per load
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t most = listed;
    for (int o = 32; o > 0; o >>= 1) most = max(most, uint32_t(__shfl_xor(int(most), o, 64)));
    most = __builtin_amdgcn_readfirstlane(most);
    if (most == 0) return;
    const uint4* my_list = reinterpret_cast<const uint4*>(list) + list_quad(k, 0, quads);
    const uint32_t last = listed ? (listed - 1) >> 2 : 0u;
    auto row = [&](uint32_t j) { return my_list[min(j, last) * LIST_TILE]; };
    // the records this lane fetches chunks of (its own record stands in for entries past its list)
    struct Fetch {
        uint32_t at[CH];  // in units of 16 bytes
    };
    auto plan = [&](uint32_t t, uint32_t e) {
        const int mine = int((t < listed ? e : uint32_t(k)) * CH);
        Fetch p;
#pragma unroll
        for (uint32_t i = 0; i < CH; ++i) p.at[i] = uint32_t(__shfl(mine, int(i * PER + lane / CH), 64));
        return p;
    };
    auto issue = [&](const Fetch& p) {
#pragma unroll
        for (uint32_t i = 0; i < CH; ++i) {
            const uint32_t c = (lane % CH) ^ S::swizzle(i * PER + lane / CH);
            const auto* g = reinterpret_cast<const __attribute__((address_space(1))) void*>(
                (uint64_t(p.at[i]) << 4) + reinterpret_cast<uintptr_t>(reinterpret_cast<const uint4*>(rec) + c));
            __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)(stage + i * 64u), 16, 0, 0);
        }
    };
    auto step = [&](uint32_t t, uint32_t e, uint32_t enext) {
        Fetch p = plan(t + 1, enext);
#pragma unroll
        for (uint32_t i = 0; i < CH; ++i) asm volatile("" : "+v"(p.at[i]));  // before the wait, not after it
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        union {
            uint4 v[CH];
            Rec r;
        } o;
#pragma unroll
        for (uint32_t c = 0; c < CH; ++c) o.v[c] = stage[lane * CH + (c ^ S::swizzle(lane))];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next records overwrite it
        if (t >= listed) e = uint32_t(k);
        const auto first = early(o.r, e);
        asm volatile("" ::: "memory");
        issue(p);
        if (t < listed) f(o.r, e, first);
    };
    uint4 q = row(0);
    issue(plan(0, q.x));
    for (uint32_t t = 0;; t += 4) {
        const uint4 nq = row((t >> 2) + 1);
        step(t, q.x, q.y);
        if (t + 1 >= most) break;
        step(t + 1, q.y, q.z);
        if (t + 2 >= most) break;
        step(t + 2, q.z, q.w);
        if (t + 3 >= most) break;
        step(t + 3, q.w, nq.x);
        if (t + 4 >= most) break;
        q = nq;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still write into the stage
}

// ---- a group of lanes per particle -------------------------------------------------------------------
// For particles too few to fill the chip with one lane each (pair_lanes), LANES (4 or 16) lanes share a particle: each
// evaluates the terms of one listed neighbour and puts them into the group's LDS rows; lane l of the group then
// adds components l, l + LANES, ... of the rows to its accumulators, in list order.  Every sum is the one a single lane makes, bit
// for bit, so how many lanes a particle gets is a question of speed only.  (With one partial sum per lane the
// sums would depend on it, and a small member of a large ensemble would have to be stepped with the lanes it gets
// alone: 10 % slower for members of 5k to 200k particles.)
// The sums then go through LDS to the first lanes of the block, one particle each, for the stores and the fused
// finalize: with one active lane per group that part would take as long as the pairs.
constexpr int PAIR_SUMS = 11;  // ax, ay, az, du, div v, grad v (xx, yy, zz, xy, xz, yz)
enum PairSum : int { SUM_A = 0, SUM_DU = 3, SUM_DIV = 4, SUM_G = 5 };

// FP64: a component gets up to three products factor * x per neighbour, each one fused multiply-add as on a single
// lane (pressure, stress and viscosity for the accelerations; one product for the others).  A product that the pair does not
// have is factor * 0, which leaves the sum as it is, unless the factor is infinite or not a number.  Such a factor makes a
// sum of its particle infinite or NaN, and then the sums are made again with CAREFUL, which multiplies it into the products
// that the pair has (exact, like the product on a single lane) and replaces it by 1; the others are then -0, which no sum
// notices.  (A factor for every product instead: 176 bytes, 27 -> 46 us for the kernel at 10k particles; CAREFUL
// always: 4 lanes 3 to 7 % slower.)
template <bool CAREFUL>
struct alignas(16) PairTerms64 {
    double m, mr;       // factors: mass for the accelerations and du, m / rho_i for the velocity gradients
    double x[11];       // first product of each component
    double stress[3], visc[3];
    uint32_t has_stress, has_visc;
    __device__ __forceinline__ void clear() {
        m = mr = 0.0;
        const double none = CAREFUL ? -0.0 : 0.0;
        for (int c = 0; c < 11; ++c) x[c] = none;
        for (int c = 0; c < 3; ++c) stress[c] = visc[c] = none;
        if (CAREFUL) has_stress = has_visc = 0u;
    }
    __device__ __forceinline__ void factors(double mj, double mjr) {
        m = mj;
        mr = mjr;
    }
    __device__ __forceinline__ void divergence(double, double v) { x[SUM_DIV] = v; }
    __device__ __forceinline__ void pressure(double, double vx, double vy, double vz) {
        x[0] = -vx;
        x[1] = -vy;
        x[2] = -vz;
    }
    __device__ __forceinline__ void gradient(double, const double v[6]) {
        for (int c = 0; c < 6; ++c) x[SUM_G + c] = v[c];
    }
    __device__ __forceinline__ void stresses(double, double vx, double vy, double vz) {
        if (CAREFUL) has_stress = 1u;
        stress[0] = vx;
        stress[1] = vy;
        stress[2] = vz;
    }
    __device__ __forceinline__ void viscosity(double, double vx, double vy, double vz, double heat) {
        if (CAREFUL) has_visc = 1u;
        visc[0] = -vx;
        visc[1] = -vy;
        visc[2] = -vz;
        x[SUM_DU] = heat;
    }
    // After the terms of a pair (gradients and stresses come together).
    __device__ __forceinline__ void finish() {
        if (!CAREFUL || (__builtin_isfinite(m) && __builtin_isfinite(mr))) return;
        if (!__builtin_isfinite(m)) {
            for (int c = 0; c < 3; ++c) {
                x[c] *= m;
                if (has_stress) stress[c] *= m;
                if (has_visc) visc[c] *= m;
            }
            if (has_visc) x[SUM_DU] *= m;
            m = 1.0;
        }
        if (!__builtin_isfinite(mr)) {
            x[SUM_DIV] *= mr;
            for (int c = 0; c < 6; ++c) {
                if (has_stress) x[SUM_G + c] *= mr;
            }
            mr = 1.0;
        }
    }
    __device__ __forceinline__ double add_to(double acc, int c) const {
        const double f = c < SUM_DIV ? m : mr;
        acc = fma(f, x[c], acc);
        if (c < 3) {
            acc = fma(f, stress[c], acc);
            acc = fma(f, visc[c], acc);
        }
        return acc;
    }
};
static_assert(sizeof(PairTerms64<false>) == 160, "PairTerms64 is 160 bytes");

// The sums of one lane's particle in FP64, the same products accumulated in place.
struct PairAcc64 {
    double ax = 0.0, ay = 0.0, az = 0.0, du = 0.0, divv = 0.0;
    double g[6] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    __device__ __forceinline__ void factors(double, double) {}
    __device__ __forceinline__ void divergence(double mjr, double v) { divv = fma(mjr, v, divv); }
    __device__ __forceinline__ void pressure(double mj, double vx, double vy, double vz) {
        ax = fma(mj, -vx, ax);
        ay = fma(mj, -vy, ay);
        az = fma(mj, -vz, az);
    }
    __device__ __forceinline__ void gradient(double mjr, const double v[6]) {
        for (int c = 0; c < 6; ++c) g[c] = fma(mjr, v[c], g[c]);
    }
    __device__ __forceinline__ void stresses(double mj, double vx, double vy, double vz) {
        ax = fma(mj, vx, ax);
        ay = fma(mj, vy, ay);
        az = fma(mj, vz, az);
    }
    __device__ __forceinline__ void viscosity(double mj, double vx, double vy, double vz, double heat) {
        ax = fma(mj, -vx, ax);
        ay = fma(mj, -vy, ay);
        az = fma(mj, -vz, az);
        du = fma(mj, heat, du);
    }
};

// Mixed precision: one FP32 term per component, widened and added in FP64.
struct alignas(16) PairTermsF {
    float x[12];
    __device__ __forceinline__ void clear() {
        for (int c = 0; c < 12; ++c) x[c] = 0.f;
    }
    __device__ __forceinline__ void divergence(float v) { x[SUM_DIV] = v; }
    __device__ __forceinline__ void gradient(int c, float v) { x[SUM_G + c] = v; }
    __device__ __forceinline__ void heat(float v) { x[SUM_DU] = v; }
    __device__ __forceinline__ void force(float vx, float vy, float vz) {
        x[0] = vx;
        x[1] = vy;
        x[2] = vz;
    }
    __device__ __forceinline__ void finish() {}
    __device__ __forceinline__ double add_to(double acc, int c) const { return acc + double(x[c]); }
};

// FP64 accumulators of FP32 terms: each term is widened exactly and summed in FP64 (on gfx950 an FP64 add
// issues at the rate of an unpacked FP32 add, so this costs two instructions per term).
struct PairAccF {
    double ax = 0.0, ay = 0.0, az = 0.0, du = 0.0, divv = 0.0;
    double g[6] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    __device__ __forceinline__ void divergence(float v) { divv += double(v); }
    __device__ __forceinline__ void gradient(int c, float v) { g[c] += double(v); }
    __device__ __forceinline__ void heat(float v) { du += double(v); }
    __device__ __forceinline__ void force(float vx, float vy, float vz) {
        ax += double(vx);
        ay += double(vy);
        az += double(vz);
    }
};

// The sums of particle k by its group of LANES lanes: acc[i] = component sub + i LANES.  rows: the group's LANES rows.
// Every lane of the wavefront must call this.
template <int LANES>
constexpr int GROUP_SUMS = (PAIR_SUMS + LANES - 1) / LANES;
template <int LANES, typename Terms, typename Rec, typename F>
__device__ __forceinline__ void sum_shared(const Rec* __restrict__ rec, const uint32_t* __restrict__ list, size_t k,
                                           uint32_t quads, uint32_t listed, uint32_t sub, Terms* rows,
                                           double (&acc)[GROUP_SUMS<LANES>], F&& f) {
    auto entry = [&](uint32_t t) { return t < listed ? list[4 * list_quad(k, t >> 2, quads) + (t & 3u)] : uint32_t(k); };
    uint32_t e = entry(sub);
    Rec o = rec[e];
    for (uint32_t t0 = 0; __any(t0 < listed); t0 += LANES) {
        // the next record is loaded before the current one's terms
        const uint32_t en = entry(t0 + LANES + sub);
        const Rec on = rec[en];
        Terms v;
        v.clear();
        if (t0 + sub < listed) {
            f(o, e, v);
            v.finish();
        }
        rows[sub] = v;
        wave_sync();
        const uint32_t cnt = t0 < listed ? min(listed - t0, uint32_t(LANES)) : 0u;
#pragma unroll
        for (int i = 0; i < GROUP_SUMS<LANES>; ++i) {
            const int c = int(sub) + i * LANES;
            if (c >= PAIR_SUMS) continue;
            if (cnt == uint32_t(LANES)) {
#pragma unroll
                for (int r = 0; r < LANES; ++r) acc[i] = rows[r].add_to(acc[i], c);
            } else {
                for (uint32_t r = 0; r < cnt; ++r) acc[i] = rows[r].add_to(acc[i], c);
            }
        }
        wave_sync();
        o = on;
        e = en;
    }
}

// The groups' sums through LDS to one thread per particle: thread p < blockDim.x / LANES gets those of the block's
// particle p.
template <int LANES, typename Acc>
__device__ __forceinline__ void collect_shared(const double (&acc)[GROUP_SUMS<LANES>], uint32_t sub,
                                               double (*all)[PAIR_SUMS], Acc& ps) {
#pragma unroll
    for (int i = 0; i < GROUP_SUMS<LANES>; ++i) {
        const int c = int(sub) + i * LANES;
        if (c < PAIR_SUMS) all[threadIdx.x / LANES][c] = acc[i];
    }
    __syncthreads();
    if (threadIdx.x < blockDim.x / LANES) {
        const double* v = all[threadIdx.x];
        ps.ax = v[0];
        ps.ay = v[1];
        ps.az = v[2];
        ps.du = v[SUM_DU];
        ps.divv = v[SUM_DIV];
        for (int c = 0; c < 6; ++c) ps.g[c] = v[SUM_G + c];
    }
}

// Stores the pair sums of particle order[k] and, FUSED, goes on with its finalize, corrector and criteria.  Every
// thread of the block must call this (threads without a particle: valid false).
template <bool FUSED, typename Acc>
__device__ __forceinline__ void pairs_finish(DevState& s, const Params& prm, const uint32_t* __restrict__ order, size_t k,
                                             bool valid, uint32_t cnt, const Acc& ps, const FuseArgs& fa) {
    const bool solid = prm.solid_stress != 0;
    double cv[4] = { INFINITY, INFINITY, INFINITY, INFINITY };
    if (valid) {
        const uint32_t i = order[k];
        const double ax = prm.add_accel ? ps.ax + s.d[AX][i] : ps.ax;
        const double ay = prm.add_accel ? ps.ay + s.d[AY][i] : ps.ay;
        const double az = prm.add_accel ? ps.az + s.d[AZ][i] : ps.az;
        s.d[AX][i] = ax;
        s.d[AY][i] = ay;
        s.d[AZ][i] = az;
        s.d[DU][i] = ps.du;
        s.d[DIVV][i] = ps.divv;
        if (solid) {
            for (int c = 0; c < 6; ++c) s.d[GXX + c][i] = ps.g[c];
        }
        s.u[NCNT][i] = cnt;
        if (FUSED && !*fa.overflow) {
            const osph_material m = fa.mats[s.u[MAT][i]];
            const PairSums sums{ { ax, ay, az }, ps.du, ps.divv, { ps.g[0], ps.g[1], ps.g[2], ps.g[3], ps.g[4], ps.g[5] } };
            finalize_at(s, m, prm, i, sums);
            correct_at(s, m, prm, fa.dt, i, sums.a);
            criteria_values(s, m, prm, i, sums.a, sums.divv, cv);
        }
    }
    if (FUSED && !*fa.overflow) reduce_criteria(cv, fa.mins);
}

// FP64 pair sums in gather form.  For particle i (sorted position k) and each neighbour j, the kernel
// gradient of SymmetrizeSmoothingLengths<LutKernel<3>> (Kernel.h:32-36,640-643) at hbar, then the
// contributions every derivative of the term set makes to particle i:
//   VelocityDivergence<CenterDensityDiscr>   DerivativeHelpers.h:355-371
//   PressureGradient<StandardForceDiscr>     EquationTerm.cpp:61-66 via AccelerationTemplate :229-242
//   VelocityGradient (SUM_ONLY_UNDAMAGED)    DerivativeHelpers.h:382-388, SymmetricTensor.h:362-368
//   StressDivergence (SUM_ONLY_UNDAMAGED)    EquationTerm.cpp:134-139, TracelessTensor.h:151-155
//   StandardAV                               av/Standard.h:62-83
//   NeighborCountTerm                        HelperTerms.h:38-46
// The accumulated buffers replace the storage buffers (Accumulated::store, Accumulated.cpp:87-100).
// With LANES > 1, a group of lanes shares one particle (sum_shared).
template <int LANES, bool FUSED>
__device__ __forceinline__ void pairs_fp64_body(size_t t, DevState s, const Params& prm,
                                                const PairRec* __restrict__ rec, const uint32_t* __restrict__ group,
                                                const uint32_t* __restrict__ order, const uint32_t* __restrict__ list,
                                                const uint32_t* __restrict__ count, const double* __restrict__ lut,
                                                uint32_t kmax, size_t n, const FuseArgs& fa) {
    const uint32_t sub = uint32_t(t % LANES);
    size_t k = t / LANES;
    bool valid = k < n;  // lanes past the end keep running, with an empty list
    if (!valid) k = n - 1;
    const PairRec me = rec[k];
    const uint32_t gi = group[k];
    const double rhoInv = 1.0 / me.rho;
    uint32_t cnt = valid ? count[k] : 0u;
    const uint32_t listed = cnt < kmax ? cnt : kmax;
    const bool solid = prm.solid_stress != 0;
    struct Early {
        double rx, ry, rz, hbar, hInv, hInv2, d2;
        LutPair lut;
        uint32_t group;
    };
    // the fused multiply-adds are written out: which products fuse must not depend on the instance, as the sums
    // are the same bits with one lane and with a group
    auto early = [&](const PairRec& o, uint32_t k2) {
#pragma clang fp contract(off)
        Early a;
        a.rx = me.x - o.x, a.ry = me.y - o.y, a.rz = me.z - o.z;
        a.hbar = 0.5 * (me.h + o.h);
        a.hInv = 1.0 / a.hbar;
        a.hInv2 = a.hInv * a.hInv;
        a.d2 = fma(a.rz, a.rz, fma(a.rx, a.rx, a.ry * a.ry));
        a.lut = lut_fetch(lut, a.d2 * a.hInv2);
        a.group = solid ? group[k2] : 0u;
        return a;
    };
    auto term = [&](const PairRec& o, const Early& a, auto& sum) {
#pragma clang fp contract(off)
        const double rx = a.rx, ry = a.ry, rz = a.rz, hbar = a.hbar, hInv = a.hInv, hInv2 = a.hInv2, d2 = a.d2;
        const double gk = a.lut.value();
        const double h5g = (hInv2 * hInv2) * hInv * gk;
        const double gx = rx * h5g, gy = ry * h5g, gz = rz * h5g;
        const double wx = o.vx - me.vx, wy = o.vy - me.vy, wz = o.vz - me.vz;  // v_j - v_i
        const double mj = o.m;
        const double mjr = mj * rhoInv;
        sum.factors(mj, mjr);
        const double wg = fma(wz, gz, fma(wx, gx, wy * gy));
        sum.divergence(mjr, wg);
        const double coef = me.pr + o.pr;
        sum.pressure(mj, coef * gx, coef * gy, coef * gz);
        if (solid && gi == a.group && gi != NO_GROUP) {
            const double gv[6] = { wx * gx, wy * gy, wz * gz, 0.5 * fma(wx, gy, wy * gx), 0.5 * fma(wx, gz, wz * gx),
                                   0.5 * fma(wy, gz, wz * gy) };
            sum.gradient(mjr, gv);
            const double xx = me.sxx + o.sxx, yy = me.syy + o.syy, xy = me.sxy + o.sxy;
            const double xz = me.sxz + o.sxz, yz = me.syz + o.syz;
            sum.stresses(mj, fma(xz, gz, fma(xx, gx, xy * gy)), fma(yz, gz, fma(yy, gy, xy * gx)),
                         fma(-xx - yy, gz, fma(xz, gx, yz * gy)));
        }
        // artificial viscosity, only in convergent flow
        const double dvdr = -fma(wz, rz, fma(wx, rx, wy * ry));  // (v_i - v_j) . (r_i - r_j)
        if (dvdr < 0.0) {
            const double rhobar = 0.5 * (me.rho + o.rho);
            const double csbar = 0.5 * (me.cs + o.cs);
            const double mu = hbar * dvdr / fma(1.e-2, hbar * hbar, d2);
            const double av = fma(prm.av_beta, mu * mu, -(prm.av_alpha * csbar * mu)) / rhobar;
            sum.viscosity(mj, av * gx, av * gy, av * gz, 0.5 * av * -wg);
        }
    };
    PairAcc64 ps;
    if constexpr (LANES > 1) {
        union Rows {
            __device__ Rows() {}
            PairTerms64<false> plain[BLOCK];
            PairTerms64<true> careful[BLOCK];
        };
        __shared__ Rows rows;
        __shared__ double all[BLOCK / LANES][PAIR_SUMS];
        double acc[GROUP_SUMS<LANES>] = {};
        auto terms = [&](const PairRec& o, uint32_t k2, auto& sum) { term(o, early(o, k2), sum); };
        const uint32_t first = threadIdx.x / LANES * LANES;
        sum_shared<LANES>(rec, list, k, kmax >> 2, listed, sub, rows.plain + first, acc, terms);
        bool odd = false;
        for (double a : acc) odd = odd || !__builtin_isfinite(a);
        if (__any(odd)) {
            for (double& a : acc) a = 0.0;
            sum_shared<LANES>(rec, list, k, kmax >> 2, listed, sub, rows.careful + first, acc, terms);
        }
        collect_shared<LANES>(acc, sub, all, ps);
        // from here on thread p of the block goes on with its particle p
        k = (t - threadIdx.x) / LANES + threadIdx.x;
        valid = threadIdx.x < blockDim.x / LANES && k < n;
        if (valid) cnt = count[k];
    } else {
        __shared__ uint4 stage[(BLOCK / 64) * StageOf<PairRec>::WORDS];
        uint4* my_stage = stage + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * StageOf<PairRec>::WORDS;
        for_each_neighbor(rec, list, k, kmax >> 2, listed, my_stage,
                          early, [&](const PairRec& o, uint32_t, const Early& a) { term(o, a, ps); });
    }
    pairs_finish<FUSED>(s, prm, order, k, valid, cnt, ps, fa);
}

template <int LANES, bool FUSED>
__global__ void __launch_bounds__(BLOCK) k_pairs_fp64(DevState s, Params prm, const PairRec* __restrict__ rec,
                                                      const uint32_t* __restrict__ group,
                                                      const uint32_t* __restrict__ order,
                                                      const uint32_t* __restrict__ list,
                                                      const uint32_t* __restrict__ count,
                                                      const double* __restrict__ lut, uint32_t kmax, size_t n,
                                                      FuseArgs fa) {
    pairs_fp64_body<LANES, FUSED>(size_t(xcd_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x, s, prm, rec,
                                   group, order, list, count, lut, kmax, n, fa);
}

// ---- mixed precision ---------------------------------------------------------------------------------

// Coordinate v on the fixed-point axis from lo with step 1 / inv (a power of two), rounded to nearest.
__device__ __forceinline__ uint32_t fixed_coord(double v, double lo, double inv) {
    const double t = floor((v - lo) * inv + 0.5);
    return uint32_t(t < 0.0 ? 0.0 : (t > 4294967295.0 ? 4294967295.0 : t));
}

// Packs the mixed-precision neighbour record of particle order[k] (and the exact FP64 position used by
// the neighbour-list build): position and velocity as 32-bit fixed-point coordinates, cs rounded to 20
// bits with the group code in the low 4.
__device__ __forceinline__ void pack_mixed_at(const DevState& s, const Params& prm, const Fixed& F,
                                              const uint32_t* __restrict__ order, PairRecF* __restrict__ rec,
                                              double4* __restrict__ pos, float4* __restrict__ posf, const Screen& sc,
                                              uint32_t* __restrict__ group, size_t k) {
    const uint32_t i = order[k];
    const double x[3] = { s.d[X][i], s.d[Y][i], s.d[Z][i] };
    const double h = s.d[H][i];
    PairRecF r;
    r.x = fixed_coord(x[0], F.lo[0], F.inv_step);
    r.y = fixed_coord(x[1], F.lo[1], F.inv_step);
    r.z = fixed_coord(x[2], F.lo[2], F.inv_step);
    r.vx = fixed_coord(s.d[VX][i], F.vlo[0], F.inv_vstep);
    r.vy = fixed_coord(s.d[VY][i], F.vlo[1], F.inv_vstep);
    r.vz = fixed_coord(s.d[VZ][i], F.vlo[2], F.inv_vstep);
    r.h = float(h);
    r.m = float(s.d[M][i]);
    const double rho = s.d[RHO][i];
    const double rho2 = rho * rho;
    r.rho = float(rho);
    r.pr = float(s.d[P][i] / rho2);
    if (prm.solid_stress) {
        r.sxx = float(s.d[SXX][i] / rho2);
        r.syy = float(s.d[SYY][i] / rho2);
        r.sxy = float(s.d[SXY][i] / rho2);
        r.sxz = float(s.d[SXZ][i] / rho2);
        r.syz = float(s.d[SYZ][i] / rho2);
    } else {
        r.sxx = r.syy = r.sxy = r.sxz = r.syz = 0.f;
    }
    uint32_t gid = 0;
    if (prm.sum_only_undamaged && prm.has_reduce) {
        gid = (s.d[RED][i] == 0.0) ? NO_GROUP : s.u[FLAG][i];
    }
    // cs >= 0: rounded to a multiple of 16 units in the last place (ties up), then the code
    const uint32_t cb = __float_as_uint(float(s.d[CS][i]));
    r.cs = __uint_as_float(((cb + 8u) & ~15u) | group_code(gid));
    rec[k] = r;
    pos[k] = make_double4(x[0], x[1], x[2], h);
    if (sc.on) posf[k] = screen_pos(sc, x[0], x[1], x[2], h);
    group[k] = gid;
}

__global__ void __launch_bounds__(BLOCK) k_pack_mixed(DevState s, Params prm, Fixed F,
                                                      const uint32_t* __restrict__ order, PairRecF* __restrict__ rec,
                                                      double4* __restrict__ pos, float4* __restrict__ posf,
                                                      Screen sc, uint32_t* __restrict__ group,
                                                      size_t n) {
    const size_t k = size_t(xcd_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x;
    if (k < n) pack_mixed_at(s, prm, F, order, rec, pos, posf, sc, group, k);
}

// M4 gradient factor grad W / q of CubicSpline<3> (core/sph/kernel/Kernel.h:172-187) in closed form,
// FP32: for q < 1 the bracket divided by q simplifies to (2.25 q - 3) / pi (finite at q = 0, where the
// reference returns -3 / pi); for 1 <= q < 2 it is -0.75 (2 - q)^2 / (pi q).  The square root and the
// reciprocal are the hardware instructions (about 1 ulp).
__device__ __forceinline__ float m4_grad_f(float q2) {
    constexpr float INV_PI = 0.318309886183790671538f;
    if (!(q2 < 4.0f)) return 0.0f;
    const float q = __builtin_amdgcn_sqrtf(q2);
    if (q < 1.0f) return INV_PI * (2.25f * q - 3.0f);
    const float t = 2.0f - q;
    return (-0.75f * INV_PI) * (t * t) * __builtin_amdgcn_rcpf(q);
}

// Mixed-precision pair sums: the same terms and gather form as k_pairs_fp64, evaluated in FP32 on the
// records' fixed-point positions and velocities and accumulated in FP64; results are written in FP64.  A
// difference of fixed-point coordinates is an exact int32 (each frame spans less than 2^31 steps), rounded
// once by the conversion to FP32 and scaled by the power-of-two step exactly, so it keeps FP32 precision
// whatever the magnitudes of the absolute values.  Divisions are hardware reciprocals
// (about 1 ulp) times the numerator.  Groups (SUM_ONLY_UNDAMAGED) compare by the records' 4-bit codes,
// and through the group array for groups beyond the codes' range.
template <int LANES, bool FUSED>
__device__ __forceinline__ void pairs_mixed_body(size_t t, DevState s, const Params& prm, const Fixed& F,
                                                 const PairRecF* __restrict__ rec, const uint32_t* __restrict__ group,
                                                 const uint32_t* __restrict__ order,
                                                 const uint32_t* __restrict__ list, const uint32_t* __restrict__ count,
                                                 uint32_t kmax, size_t n, const FuseArgs& fa) {
    const uint32_t sub = uint32_t(t % LANES);
    size_t k = t / LANES;
    bool valid = k < n;  // lanes past the end keep running, with an empty list
    if (!valid) k = n - 1;
    const PairRecF me = rec[k];
    const uint32_t gi = group[k];
    const uint32_t gci = __float_as_uint(me.cs) & 15u;
    const float csi = __uint_as_float(__float_as_uint(me.cs) & ~15u);
    const float rhoInv = 1.0f / me.rho;
    const float alpha = float(prm.av_alpha), beta = float(prm.av_beta);
    uint32_t cnt = valid ? count[k] : 0u;
    const uint32_t listed = cnt < kmax ? cnt : kmax;
    const bool solid = prm.solid_stress != 0;
    const bool grouped = solid && gci != GROUP_CODE_NONE;  // stress terms with the particle's own group
    // the fused multiply-adds are written out: which products fuse must not depend on the instance, as the sums
    // are the same bits with one lane and with a group
    auto term = [&](const PairRecF& o, uint32_t e, auto& sum) {
#pragma clang fp contract(off)
        const float rx = float(int32_t(me.x - o.x)) * F.stepf;
        const float ry = float(int32_t(me.y - o.y)) * F.stepf;
        const float rz = float(int32_t(me.z - o.z)) * F.stepf;
        const float hbar = 0.5f * (me.h + o.h);
        const float hInv = __builtin_amdgcn_rcpf(hbar);
        const float hInv2 = hInv * hInv;
        const float d2 = fmaf(rz, rz, fmaf(rx, rx, ry * ry));
        const float gk = m4_grad_f(d2 * hInv2);
        const float h5g = (hInv2 * hInv2) * hInv * gk;
        const float gx = rx * h5g, gy = ry * h5g, gz = rz * h5g;
        const float wx = float(int32_t(o.vx - me.vx)) * F.vstepf;  // v_j - v_i
        const float wy = float(int32_t(o.vy - me.vy)) * F.vstepf;
        const float wz = float(int32_t(o.vz - me.vz)) * F.vstepf;
        const float mj = o.m;
        const float mjr = mj * rhoInv;
        const float wgx = wx * gx, wgy = wy * gy, wgz = wz * gz;
        const float wg = wgx + wgy + wgz;
        sum.divergence(mjr * wg);
        const float coef = me.pr + o.pr;
        float fx = -(coef * gx), fy = -(coef * gy), fz = -(coef * gz);
        bool same = grouped && (__float_as_uint(o.cs) & 15u) == gci;
        if (same && gci == GROUP_CODE_WIDE) same = group[e] == gi;
        if (same) {
            sum.gradient(0, mjr * wgx);
            sum.gradient(1, mjr * wgy);
            sum.gradient(2, mjr * wgz);
            sum.gradient(3, mjr * (0.5f * fmaf(wx, gy, wy * gx)));
            sum.gradient(4, mjr * (0.5f * fmaf(wx, gz, wz * gx)));
            sum.gradient(5, mjr * (0.5f * fmaf(wy, gz, wz * gy)));
            const float xx = me.sxx + o.sxx, yy = me.syy + o.syy, xy = me.sxy + o.sxy;
            const float xz = me.sxz + o.sxz, yz = me.syz + o.syz;
            fx += fmaf(xz, gz, fmaf(xx, gx, xy * gy));
            fy += fmaf(yz, gz, fmaf(yy, gy, xy * gx));
            fz += fmaf(-xx - yy, gz, fmaf(xz, gx, yz * gy));
        }
        const float dvdr = -fmaf(wz, rz, fmaf(wx, rx, wy * ry));
        if (dvdr < 0.0f) {
            const float rhobar = 0.5f * (me.rho + o.rho);
            const float csbar = 0.5f * (csi + __uint_as_float(__float_as_uint(o.cs) & ~15u));
            const float mu = hbar * dvdr * __builtin_amdgcn_rcpf(fmaf(1.e-2f, hbar * hbar, d2));
            const float av = fmaf(beta, mu * mu, -(alpha * csbar * mu)) * __builtin_amdgcn_rcpf(rhobar);
            fx = fmaf(-av, gx, fx);
            fy = fmaf(-av, gy, fy);
            fz = fmaf(-av, gz, fz);
            sum.heat(mj * (0.5f * av * -wg));
        }
        sum.force(mj * fx, mj * fy, mj * fz);
    };
    PairAccF ps;
    if constexpr (LANES > 1) {
        __shared__ PairTermsF rows[BLOCK];
        __shared__ double all[BLOCK / LANES][PAIR_SUMS];
        double acc[GROUP_SUMS<LANES>] = {};
        sum_shared<LANES>(rec, list, k, kmax >> 2, listed, sub, rows + threadIdx.x / LANES * LANES, acc, term);
        collect_shared<LANES>(acc, sub, all, ps);
        // from here on thread p of the block goes on with its particle p
        k = (t - threadIdx.x) / LANES + threadIdx.x;
        valid = threadIdx.x < blockDim.x / LANES && k < n;
        if (valid) cnt = count[k];
    } else {
        __shared__ uint4 stage[(BLOCK / 64) * StageOf<PairRecF>::WORDS];
        uint4* my_stage = stage + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * StageOf<PairRecF>::WORDS;
        for_each_neighbor(rec, list, k, kmax >> 2, listed, my_stage,
                          [](const PairRecF&, uint32_t) { return 0; },
                          [&](const PairRecF& o, uint32_t e, int) { term(o, e, ps); });
    }
    pairs_finish<FUSED>(s, prm, order, k, valid, cnt, ps, fa);
}

template <int LANES, bool FUSED>
__global__ void __launch_bounds__(BLOCK) k_pairs_mixed(DevState s, Params prm, Fixed F,
                                                       const PairRecF* __restrict__ rec,
                                                       const uint32_t* __restrict__ group,
                                                       const uint32_t* __restrict__ order,
                                                       const uint32_t* __restrict__ list,
                                                       const uint32_t* __restrict__ count, uint32_t kmax, size_t n,
                                                       FuseArgs fa) {
    pairs_mixed_body<LANES, FUSED>(size_t(xcd_block(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x, s, prm, F, rec,
                                    group, order, list, count, kmax, n, fa);
}

// ScalarGradyKippModel::integrate (core/physics/Damage.cpp:128-170) for particle i.
__device__ void damage_rate(DevState& s, const osph_material& m, size_t i) {
#pragma clang fp contract(off)
    const double D0 = s.d[D][i];
    if (D0 >= m.d_hi) {
        s.d[DD][i] = LARGE_D;
        return;
    }
    const double pr = s.d[P][i];
    const double sxx = s.d[SXX][i], syy = s.d[SYY][i];
    const double t[6] = { sxx - pr * 1.0, syy - pr * 1.0, (-sxx - syy) - pr * 1.0,
                          s.d[SXY][i] - pr * 0.0, s.d[SXZ][i] - pr * 0.0, s.d[SYZ][i] - pr * 0.0 };
    double sig[3];
    eigenvalues(t, sig);
    const double sigMax = dmax(dmax(sig[0], sig[1]), sig[2]);
    const double young_red = dmax((1.0 - D0 * D0 * D0) * m.young_modulus, 1.e-20);
    const double strain = sigMax / young_red;
    const double ratio = strain / s.d[EPSMIN][i];
    if (ratio <= 1.0) {
        s.d[DD][i] = 0.0;
        return;
    }
    s.d[DD][i] = s.d[GROWTH][i] * cbrt(dmin(pow(ratio, s.d[MZERO][i]), double(s.u[NFLAWS][i])));
}

// EquationHolder::finalize in reverse term order (EquationTerm.h:293-297): AdaptiveSmoothingLength
// (EquationTerm.cpp:366-387) or ConstSmoothingLength (:427-434), ContinuityEquation (:289-299),
// SolidStressForce (:177-203), PressureForce (:90-99); then the material finalize (damage).  Every
// highest derivative the step integrates is assigned here or in the pair sums (the reference zeroes them
// before the evaluation and adds the terms' contributions, which is the same value).
__device__ void finalize_at(DevState& s, const osph_material& m, const Params& prm, size_t i, const PairSums& ps) {
#pragma clang fp contract(off)
    const double rho = s.d[RHO][i], divv = ps.divv;
    const double h = s.d[H][i];
    s.d[VH][i] = (prm.adaptive_h && h > 2.0 * prm.h_lo) ? h / 3.0 * divv : 0.0;
    s.d[DRHO][i] = -rho * divv;
    double du = ps.du;
    if (prm.solid_stress && m.yielding != 0) {
        const double sxx = s.d[SXX][i], syy = s.d[SYY][i], szz = -sxx - syy;
        const double gxx = ps.g[0], gyy = ps.g[1], gzz = ps.g[2];
        const double gxy = ps.g[3], gxz = ps.g[4], gyz = ps.g[5];
        const double dd = (sxx * gxx + syy * gyy + szz * gzz) +
                          2.0 * (s.d[SXY][i] * gxy + s.d[SXZ][i] * gxz + s.d[SYZ][i] * gyz);
        du += 1.0 / rho * dd;
        const double tr3 = (gxx * 1.0 + gyy * 1.0 + gzz * 1.0) / 3.0;
        const double twomu = 2.0 * m.shear_modulus;
        s.d[DSXX][i] = twomu * (gxx - tr3);
        s.d[DSYY][i] = twomu * (gyy - tr3);
        s.d[DSXY][i] = twomu * gxy;
        s.d[DSXZ][i] = twomu * gxz;
        s.d[DSYZ][i] = twomu * gyz;
    } else if (prm.solid_stress) {
        for (int k = 0; k < 5; ++k) s.d[DSXX + k][i] = 0.0;
    }
    du -= s.d[P][i] / rho * divv;
    s.d[DU][i] = du;
    if (prm.has_damage) {
        if (m.damage == 1) {
            damage_rate(s, m, i);
        } else {
            s.d[DD][i] = 0.0;
        }
    }
}

__global__ void __launch_bounds__(BLOCK) k_finalize(DevState s, const osph_material* __restrict__ mats, Params prm,
                                                    size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    finalize_at(s, mats[s.u[MAT][i]], prm, i, sums_of(s, prm.solid_stress != 0, i));
}

// Storage::zeroHighestDerivatives (core/quantities/Storage.cpp:594-602)
__global__ void __launch_bounds__(BLOCK) k_zero_derivatives(DevState s, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int planes[] = { AX, AY, AZ, DRHO, DU, DSXX, DSYY, DSXY, DSXZ, DSYZ, DD };
#pragma unroll
    for (int k = 0; k < 11; ++k) s.d[planes[k]][i] = 0.0;
}

// clampWithDerivative<Float> (core/objects/wrappers/Interval.h:158-162)
__device__ __forceinline__ void clamp_deriv(double& v, double& dv, double lo, double hi) {
    const bool zero = (v >= hi && dv > 0.0) || (v <= lo && dv < 0.0);
    v = dmax(lo, dmin(v, hi));
    if (zero) dv = 0.0;
}

// PredictorCorrector::makePredictions (core/timestepping/TimeStepping.cpp:286-300).  The swap of the
// highest derivatives into the predictions storage and Storage::zeroHighestDerivatives (:331-334) are
// done by the host before this pass, by exchanging the plane pointers of each highest derivative and its
// prediction (AX <-> PAX, DRHO <-> PDRHO, ...): the derivative of the last evaluation is read here from
// the prediction planes, and the derivative planes are left for the next evaluation, which assigns every
// one of them (the pair sums, the finalize).  A derivative zeroed by a clamp is written back to its
// prediction plane, as the reference clamps the derivative it saves.
__device__ void predict_at(DevState& s, const osph_material& m, const Params& prm, double dt, size_t i) {
#pragma clang fp contract(off)
    const double dt2 = 0.5 * (dt * dt);
    for (int k = 0; k < 3; ++k) {
        const double a = s.d[PAX + k][i];
        const double v = s.d[VX + k][i];
        s.d[X + k][i] += v * dt + a * dt2;
        s.d[VX + k][i] = v + a * dt;
    }
    s.d[H][i] += s.d[VH][i] * dt + 0.0 * dt2;
    auto first_order = [&](int q, int pq, double lo, double hi) {
        double x = s.d[q][i];
        const double dx0 = s.d[pq][i];
        double dx = dx0;
        x += dx * dt;
        clamp_deriv(x, dx, lo, hi);
        s.d[q][i] = x;
        if (dx != dx0) s.d[pq][i] = dx;
    };
    first_order(RHO, PDRHO, m.rho_lo, m.rho_hi);
    first_order(U, PDU, m.u_lo, m.u_hi);
    if (prm.solid_stress) {
        for (int k = 0; k < 5; ++k) s.d[SXX + k][i] += s.d[PDSXX + k][i] * dt;
    }
    if (prm.has_damage) first_order(D, PDD, m.d_lo, m.d_hi);
}

__device__ __forceinline__ void atomic_min_pos(unsigned long long* addr, double v) {
    // v >= 0 (or +inf): the IEEE bit patterns of non-negative doubles are ordered like the values
    atomicMin(addr, (unsigned long long)__double_as_longlong(v));
}

// Per-particle values of the four criteria of MultiCriterion (TimeStepCriterion.cpp:315-356 Courant,
// :123-211 DerivativeCriterion with the minimal-step mean, :221-257 Acceleration, :267-305 Divergence),
// reduced to the minimum of each criterion in mins[0..3].
__device__ void criteria_values(const DevState& s, const osph_material& m, const Params& prm, size_t i,
                                const double a[3], double divv, double out[4]) {
#pragma clang fp contract(off)
    out[0] = out[1] = out[2] = out[3] = INFINITY;
    const double h = s.d[H][i];
    if (prm.criteria & 1) {
        const double cs = s.d[CS][i];
        if (cs > 0.0) out[0] = prm.courant * h / cs;
    }
    if (prm.criteria & 2) {
        double mn = INFINITY;
        auto add = [&](double v, double dv, double minValue) {
            const double av = fabs(v), adv = fabs(dv);
            if (av < 2.0 * minValue) return;
            mn = dmin(mn, prm.deriv_factor * (av + minValue) / (adv + EPS_D));
        };
        add(s.d[RHO][i], s.d[DRHO][i], m.rho_min);
        add(s.d[U][i], s.d[DU][i], m.u_min);
        if (prm.solid_stress) {
            const double xx = s.d[SXX][i], yy = s.d[SYY][i];
            const double dxx = s.d[DSXX][i], dyy = s.d[DSYY][i];
            add(xx, dxx, m.s_min);
            add(yy, dyy, m.s_min);
            add(-xx - yy, -dxx - dyy, m.s_min);
            add(s.d[SXY][i], s.d[DSXY][i], m.s_min);
            add(s.d[SXZ][i], s.d[DSXZ][i], m.s_min);
            add(s.d[SYZ][i], s.d[DSYZ][i], m.s_min);
        }
        if (prm.has_damage) add(s.d[D][i], s.d[DD][i], m.d_min);
        out[1] = mn;
    }
    if (prm.criteria & 4) {
        const double ax = a[0], ay = a[1], az = a[2];
        const double dvNorm = ax * ax + ay * ay + az * az;
        if (dvNorm > EPS_D) out[2] = prm.deriv_factor * sqrt(sqrt((h * h) / dvNorm));
    }
    if (prm.criteria & 8) {
        const double dv = fabs(divv);
        if (dv > EPS_D) out[3] = prm.div_factor / dv;
    }
}

__device__ void reduce_criteria(double v[4], unsigned long long* mins) {
    __shared__ double red[BLOCK / 64][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int c = 0; c < 4; ++c) {
        double x = v[c];
        for (int o = 32; o > 0; o >>= 1) x = dmin(x, __shfl_xor(x, o, 64));
        if (lane == 0) red[wave][c] = x;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        // the pair kernels run with blocks of 64, 128 or 256 threads: only the block's own waves hold values
        const int waves = int(blockDim.x >> 6);
        double x = red[0][threadIdx.x];
        for (int w = 1; w < waves; ++w) x = dmin(x, red[w][threadIdx.x]);
        // the atomic only when it would lower the current minimum (a device-coherent read): most blocks
        // then skip it, where thousands of same-address atomics would serialise
        const unsigned long long bits = (unsigned long long)__double_as_longlong(x);
        if (x < INFINITY && bits < __hip_atomic_load(&mins[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            atomic_min_pos(&mins[threadIdx.x], x);
        }
    }
}

// PredictorCorrector::makeCorrections (TimeStepping.cpp:302-322): pdv is the new derivative, cdv the
// saved prediction; the clamp zeroes the new derivative at the bounds.
__device__ void correct_at(DevState& s, const osph_material& m, const Params& prm, double dt, size_t i,
                           const double a[3]) {
#pragma clang fp contract(off)
    {
        const double dt2 = 0.5 * (dt * dt);
        const double ca = 1.0 / 3.0, cb = 0.5;
        for (int k = 0; k < 3; ++k) {
            const double pdv = a[k], cdv = s.d[PAX + k][i];
            s.d[X + k][i] -= ca * (cdv - pdv) * dt2;
            s.d[VX + k][i] -= cb * (cdv - pdv) * dt;
        }
        {
            double x = s.d[RHO][i], px = s.d[DRHO][i];
            x -= 0.5 * (s.d[PDRHO][i] - px) * dt;
            clamp_deriv(x, px, m.rho_lo, m.rho_hi);
            s.d[RHO][i] = x;
            s.d[DRHO][i] = px;
        }
        {
            double x = s.d[U][i], px = s.d[DU][i];
            x -= 0.5 * (s.d[PDU][i] - px) * dt;
            clamp_deriv(x, px, m.u_lo, m.u_hi);
            s.d[U][i] = x;
            s.d[DU][i] = px;
        }
        if (prm.solid_stress) {
            for (int k = 0; k < 5; ++k) {
                s.d[SXX + k][i] -= 0.5 * (s.d[PDSXX + k][i] - s.d[DSXX + k][i]) * dt;
            }
        }
        if (prm.has_damage) {
            double x = s.d[D][i], px = s.d[DD][i];
            x -= 0.5 * (s.d[PDD][i] - px) * dt;
            clamp_deriv(x, px, m.d_lo, m.d_hi);
            s.d[D][i] = x;
            s.d[DD][i] = px;
        }
    }
}

// The end of a predictor-corrector step for particle i: EquationHolder::finalize and the material
// finalize, the corrections, then the criteria of the corrected state, reduced into mins[0..3].  When
// the neighbour lists overflowed (*overflow != 0) the kernel changes nothing: the step is repeated with
// larger lists from the same predicted state.
__device__ __forceinline__ void finalize_correct_body(size_t i, DevState s, const osph_material* __restrict__ mats,
                                                      const Params& prm, double dt, unsigned long long* mins,
                                                      const uint32_t* overflow, size_t n) {
    if (*overflow) return;  // uniform over the grid
    double v[4] = { INFINITY, INFINITY, INFINITY, INFINITY };
    if (i < n) {
        const osph_material m = mats[s.u[MAT][i]];
        const PairSums ps = sums_of(s, prm.solid_stress != 0, i);
        finalize_at(s, m, prm, i, ps);
        correct_at(s, m, prm, dt, i, ps.a);
        criteria_values(s, m, prm, i, ps.a, ps.divv, v);
    }
    reduce_criteria(v, mins);
}

__global__ void __launch_bounds__(BLOCK) k_finalize_correct(DevState s, const osph_material* __restrict__ mats,
                                                            Params prm, double dt, unsigned long long* mins,
                                                            const uint32_t* overflow, size_t n) {
    finalize_correct_body(size_t(blockIdx.x) * blockDim.x + threadIdx.x, s, mats, prm, dt, mins, overflow, n);
}

// Per-block partial grid bounds.  Values v = CLASS_VALUES * c + k for class c (k: 0..2 min x, y, z;
// 3..5 max x, y, z; 6 max h; 7 min h; 8 count, min and max as order-preserving bit patterns), then
// VEL_VALUES velocity bounds (min x, y, z, max x, y, z).  part[v * nblocks + block]; k_bounds_final
// reduces them.  Two levels instead of per-block atomics: same-address atomics from thousands of blocks
// serialise (56 us for 1024 blocks at the impact).
constexpr int CLASS_VALUES = 9;
constexpr int VEL_VALUES = 6;
constexpr int BOUND_VALUES = CLASS_VALUES * MAX_CLASSES + VEL_VALUES;

__device__ __forceinline__ bool bound_is_min(int v) {
    if (v >= CLASS_VALUES * MAX_CLASSES) return v - CLASS_VALUES * MAX_CLASSES < 3;
    const int k = v % CLASS_VALUES;
    return k < 3 || k == 7;
}

__device__ __forceinline__ unsigned long long bound_identity(int v) {
    if (v < CLASS_VALUES * MAX_CLASSES && v % CLASS_VALUES == 8) return 0ull;
    return bound_is_min(v) ? ~0ull : 0ull;
}

__device__ __forceinline__ unsigned long long bound_combine(int v, unsigned long long a, unsigned long long b) {
    if (v < CLASS_VALUES * MAX_CLASSES && v % CLASS_VALUES == 8) return a + b;
    return bound_is_min(v) ? (b < a ? b : a) : (b > a ? b : a);
}

// Block-level partial bounds of one particle per thread (cls < 0: no particle).  Every thread of the
// block must call it.
template <bool VEL>
__device__ void block_bounds(int cls, double x, double y, double z, double h, const double* v,
                             unsigned long long* __restrict__ part, uint32_t nblocks, uint32_t block) {
    __shared__ unsigned long long red[BLOCK / 64][BOUND_VALUES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long b[4] = { ord_bits(x), ord_bits(y), ord_bits(z), ord_bits(h) };
    for (int c = 0; c < MAX_CLASSES; ++c) {
        const bool in = cls == c;
        unsigned long long* r = red[wave] + CLASS_VALUES * c;
        if (__any(in)) {
            for (int k = 0; k < 3; ++k) {
                const unsigned long long lo = wave_min(in ? b[k] : ~0ull);
                const unsigned long long hi = wave_max(in ? b[k] : 0ull);
                if (lane == 0) {
                    r[k] = lo;
                    r[3 + k] = hi;
                }
            }
            const unsigned long long hmax = wave_max(in ? b[3] : 0ull), hmin = wave_min(in ? b[3] : ~0ull);
            const unsigned long long cnt = __popcll(__ballot(in));
            if (lane == 0) {
                r[6] = hmax;
                r[7] = hmin;
                r[8] = cnt;
            }
        } else if (lane == 0) {
            for (int k = 0; k < CLASS_VALUES; ++k) r[k] = bound_identity(CLASS_VALUES * c + k);
        }
    }
    if (VEL) {
        for (int k = 0; k < 3; ++k) {
            const bool ok = cls >= 0;
            const unsigned long long bv = ord_bits(v[k]);
            const unsigned long long lo = wave_min(ok ? bv : ~0ull), hi = wave_max(ok ? bv : 0ull);
            if (lane == 0) {
                red[wave][CLASS_VALUES * MAX_CLASSES + k] = lo;
                red[wave][CLASS_VALUES * MAX_CLASSES + 3 + k] = hi;
            }
        }
    }
    __syncthreads();
    const int nv = VEL ? BOUND_VALUES : CLASS_VALUES * MAX_CLASSES;
    if (int(threadIdx.x) < nv) {
        const int vi = threadIdx.x;
        unsigned long long acc = red[0][vi];
        for (int w = 1; w < int(blockDim.x / 64); ++w) acc = bound_combine(vi, acc, red[w][vi]);
        part[size_t(vi) * nblocks + block] = acc;
    }
}

// One pass before the neighbour search, MODE 2: predictions (predict_at) then the material initialize;
// MODE 1: the material initialize only; MODE 0: neither.  Every mode ends with the per-block partial
// grid bounds of the resulting positions (class of h relative to href) and, with VEL, velocities.
template <int MODE, bool VEL>
__device__ __forceinline__ void advance_body(uint32_t bid, uint32_t nb, DevState s,
                                             const osph_material* __restrict__ mats, const Params& prm, double dt,
                                             double href, unsigned long long* __restrict__ part, size_t n) {
    const size_t i = size_t(bid) * BLOCK + threadIdx.x;
    int cls = -1;
    double x = 0.0, y = 0.0, z = 0.0, h = 0.0, v[3] = { 0.0, 0.0, 0.0 };
    if (i < n) {
        if (MODE > 0) {
            const osph_material m = mats[s.u[MAT][i]];
            if (MODE > 1) predict_at(s, m, prm, dt, i);
            material_init_at(s, m, prm, i);
        }
        x = s.d[X][i];
        y = s.d[Y][i];
        z = s.d[Z][i];
        h = s.d[H][i];
        cls = h_class(h, href, MAX_CLASSES);
        if (VEL) {
            v[0] = s.d[VX][i];
            v[1] = s.d[VY][i];
            v[2] = s.d[VZ][i];
        }
    }
    block_bounds<VEL>(cls, x, y, z, h, v, part, nb, bid);
}

template <int MODE, bool VEL>
__global__ void __launch_bounds__(BLOCK) k_advance(DevState s, const osph_material* __restrict__ mats, Params prm,
                                                   double dt, double href, unsigned long long* __restrict__ part,
                                                   size_t n) {
    advance_body<MODE, VEL>(blockIdx.x, gridDim.x, s, mats, prm, dt, href, part, n);
}

// Second level of the bounds: block v reduces value v over the nblocks partials into acc (the class
// values, at CLASS_STRIDE * c + k) or vel.
__device__ __forceinline__ void bounds_final_at(int vi, const unsigned long long* __restrict__ part,
                                                uint32_t nblocks, unsigned long long* __restrict__ acc,
                                                unsigned long long* __restrict__ vel) {
    __shared__ unsigned long long red[BLOCK / 64];
    unsigned long long r = bound_identity(vi);
    for (uint32_t b = threadIdx.x; b < nblocks; b += blockDim.x) r = bound_combine(vi, r, part[size_t(vi) * nblocks + b]);
    for (int o = 32; o > 0; o >>= 1) r = bound_combine(vi, r, __shfl_xor(r, o, 64));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) red[wave] = r;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < int(blockDim.x / 64); ++w) r = bound_combine(vi, r, red[w]);
        if (vi < CLASS_VALUES * MAX_CLASSES) {
            acc[CLASS_STRIDE * (vi / CLASS_VALUES) + vi % CLASS_VALUES] = r;
        } else {
            vel[vi - CLASS_VALUES * MAX_CLASSES] = r;
        }
    }
}

// Block v reduces bound value v; block 0 also starts the step's other accumulators (global bounds,
// criterion minima, list overflow flag: words 0 .. SMALL_CLASSES - 1, which no earlier pass of the step
// uses), in place of a launch of its own.
__global__ void __launch_bounds__(BLOCK) k_bounds_final(const unsigned long long* __restrict__ part, uint32_t nblocks,
                                                        unsigned long long* __restrict__ small) {
    if (blockIdx.x == 0 && threadIdx.x < SMALL_CLASSES) init_small_at(small, threadIdx.x);
    bounds_final_at(blockIdx.x, part, nblocks, small + SMALL_CLASSES, small + SMALL_VEL);
}

__global__ void __launch_bounds__(BLOCK) k_criteria(DevState s, const osph_material* __restrict__ mats, Params prm,
                                                    unsigned long long* mins, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    double v[4] = { INFINITY, INFINITY, INFINITY, INFINITY };
    if (i < n) {
        const osph_material m = mats[s.u[MAT][i]];
        const double a[3] = { s.d[AX][i], s.d[AY][i], s.d[AZ][i] };
        criteria_values(s, m, prm, i, a, s.d[DIVV][i], v);
    }
    reduce_criteria(v, mins);
}

// Statistics of the neighbour counts (SymmetricSolver.cpp:172-179): a bounded grid and one set of atomics per block, as
// those on the same three words take their turns (559k counts 13 us; with a set per wavefront, 128 blocks 27
// and 512 blocks 76).
constexpr unsigned STATS_BLOCKS = 128;
__global__ void __launch_bounds__(BLOCK) k_count_stats(const uint32_t* __restrict__ counts,
                                                       unsigned long long* __restrict__ stats, size_t n) {
    unsigned long long inv = 0ull, mx = 0ull, sum = 0ull;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
        const uint32_t c = counts[i];
        const unsigned long long comp = uint32_t(~c);
        inv = comp > inv ? comp : inv;
        mx = c > mx ? c : mx;
        sum += c;
    }
    inv = wave_max(inv);
    mx = wave_max(mx);
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    __shared__ unsigned long long red[BLOCK / 64][3];
    if ((threadIdx.x & 63u) == 0) {
        unsigned long long* r = red[threadIdx.x >> 6];
        r[0] = inv;
        r[1] = mx;
        r[2] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BLOCK / 64; ++w) {
            inv = red[w][0] > inv ? red[w][0] : inv;
            mx = red[w][1] > mx ? red[w][1] : mx;
            sum += red[w][2];
        }
        atomicMax(&stats[0], inv);
        atomicMax(&stats[1], mx);
        atomicAdd(&stats[2], sum);
    }
}

struct StageDesc {
    int ncomp;
    int elem;
    int off[8];
    void* p[8];
    const uint32_t* slot;  // storage index -> device slot
};

__global__ void __launch_bounds__(BLOCK) k_stage_to_planes(const unsigned char* __restrict__ st, size_t stride,
                                                           StageDesc d, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const unsigned char* e = st + i * stride;
    const size_t k = d.slot[i];
    for (int c = 0; c < d.ncomp; ++c) {
        if (d.elem == 8) {
            static_cast<double*>(d.p[c])[k] = *reinterpret_cast<const double*>(e + d.off[c]);
        } else {
            static_cast<uint32_t*>(d.p[c])[k] = *reinterpret_cast<const uint32_t*>(e + d.off[c]);
        }
    }
}

__global__ void __launch_bounds__(BLOCK) k_planes_to_stage(unsigned char* __restrict__ st, size_t stride, StageDesc d,
                                                           size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    unsigned char* e = st + i * stride;
    const size_t k = d.slot[i];
    for (int c = 0; c < d.ncomp; ++c) {
        if (d.elem == 8) {
            *reinterpret_cast<double*>(e + d.off[c]) = static_cast<const double*>(d.p[c])[k];
        } else {
            *reinterpret_cast<uint32_t*>(e + d.off[c]) = static_cast<const uint32_t*>(d.p[c])[k];
        }
    }
}

// Moves the state into cell order: slot k of dst receives slot order[k] of src, and the slot <-> storage
// maps follow (perm_out[k] = storage index of slot k, slot_of[storage index] = k).
__device__ __forceinline__ void permute_at(const DevState& src, const DevState& dst, const uint32_t* __restrict__ order,
                                           const uint32_t* __restrict__ perm_in, uint32_t* __restrict__ perm_out,
                                           uint32_t* __restrict__ slot_of, size_t k) {
    const uint32_t i = order[k];
#pragma unroll 4
    for (int p = 0; p < NDPLANES; ++p) dst.d[p][k] = src.d[p][i];
#pragma unroll
    for (int p = 0; p < NIPLANES; ++p) dst.u[p][k] = src.u[p][i];
    const uint32_t g = perm_in[i];
    perm_out[k] = g;
    slot_of[g] = uint32_t(k);
}

__global__ void __launch_bounds__(BLOCK) k_permute_state(DevState src, DevState dst, const uint32_t* __restrict__ order,
                                                         const uint32_t* __restrict__ perm_in,
                                                         uint32_t* __restrict__ perm_out,
                                                         uint32_t* __restrict__ slot_of, size_t n) {
    const size_t k = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n) permute_at(src, dst, order, perm_in, perm_out, slot_of, k);
}

__global__ void __launch_bounds__(BLOCK) k_iota_u32(uint32_t* p, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = uint32_t(i);
}

// STREAM-style copy: b[i] = a[i], 16 bytes per lane per iteration.
__global__ void __launch_bounds__(BLOCK) k_stream_copy(const double2* __restrict__ a, double2* __restrict__ b,
                                                       size_t n2) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n2; i += size_t(gridDim.x) * blockDim.x) {
        b[i] = a[i];
    }
}

// Integrals of the state (core/physics/Integrals.cpp:24-180): per block, in a fixed reduction order, then
// one block over the partials.  v[0] kinetic energy, v[1] internal energy, v[2..4] momentum, v[5..7]
// angular momentum about the origin, v[8..10] sum of m r, v[11] total mass.
constexpr int NINT = 12;

__global__ void __launch_bounds__(BLOCK) k_integrals(DevState s, size_t n, double* __restrict__ partial) {
    double v[NINT] = { 0.0 };
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) {
        const double m = s.d[M][i];
        const double x = s.d[X][i], y = s.d[Y][i], z = s.d[Z][i];
        const double vx = s.d[VX][i], vy = s.d[VY][i], vz = s.d[VZ][i];
        v[0] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
        v[1] += m * s.d[U][i];
        v[2] += m * vx;
        v[3] += m * vy;
        v[4] += m * vz;
        v[5] += m * (y * vz - z * vy);
        v[6] += m * (z * vx - x * vz);
        v[7] += m * (x * vy - y * vx);
        v[8] += m * x;
        v[9] += m * y;
        v[10] += m * z;
        v[11] += m;
    }
    __shared__ double red[BLOCK / 64][NINT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < NINT; ++k) {
        double x = v[k];
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        if (lane == 0) red[wave][k] = x;
    }
    __syncthreads();
    if (threadIdx.x < NINT) {
        double x = 0.0;
        for (int w = 0; w < BLOCK / 64; ++w) x += red[w][threadIdx.x];
        partial[size_t(blockIdx.x) * NINT + threadIdx.x] = x;
    }
}

__global__ void __launch_bounds__(64) k_integrals_final(const double* __restrict__ partial, int nblocks,
                                                        double* __restrict__ out) {
    if (threadIdx.x >= NINT) return;
    double x = 0.0;
    for (int b = 0; b < nblocks; ++b) x += partial[size_t(b) * NINT + threadIdx.x];
    out[threadIdx.x] = x;
}

}  // namespace

size_t integrals_scratch_doubles(size_t n) {
    unsigned g = grid_for(n);
    g = g > 1024 ? 1024 : g;
    return size_t(g) * NINT + NINT;
}

void launch_integrals(const Launch& l, DevState s, double* scratch, size_t n) {
    unsigned g = grid_for(n);
    g = g > 1024 ? 1024 : g;
    k_integrals<<<g, BLOCK, 0, l.stream>>>(s, n, scratch);
    k_integrals_final<<<1, 64, 0, l.stream>>>(scratch, int(g), scratch + size_t(g) * NINT);
}

void launch_stream_copy(hipStream_t stream, const void* a, void* b, size_t bytes) {
    const size_t n2 = bytes / sizeof(double2);
    if (!n2) return;
    unsigned g = grid_for(n2);
    g = g > 8192 ? 8192 : g;
    k_stream_copy<<<g, BLOCK, 0, stream>>>(static_cast<const double2*>(a), static_cast<double2*>(b), n2);
}

// ---- launchers ----------------------------------------------------------------------------------------

void launch_init_small(const Launch& l, unsigned long long* small) {
    k_init_small<<<1, SMALL_WORDS, 0, l.stream>>>(small);
}

void launch_bounds_reduce(const Launch& l, DevState s, unsigned long long* acc, size_t n) {
    if (!n) return;
    unsigned g = grid_for(n);
    g = g > 1024 ? 1024 : g;
    k_bounds<<<g, BLOCK, 0, l.stream>>>(s, acc, n);
}

namespace {

unsigned fill_blocks(size_t count) { return std::min(grid_for(count), 4096u); }

}  // namespace

// Whole scan tiles with an entry past the last row.
size_t row_slots(uint32_t slots) { return (size_t(slots) / SCAN_TILE + 1) * SCAN_TILE; }

void launch_cell_sort(const Launch& l, DevState s, Grid g, uint32_t* row_count, uint32_t* row_start, uint2* where,
                      uint2* bucket, uint32_t* order, uint32_t* first, size_t rows, size_t n) {
    // without particles nothing reads the table
    if (!rows || !n) return;
    const unsigned blocks = grid_for(n), scans = unsigned(row_slots(g.slots) / SCAN_TILE), waves = grid_for(rows, BLOCK / 64);
    // a kernel that does not start leaves the next one values of an older grid as indexes: the chain ends there
    if (g.by_cells) {
        const size_t cells = g.cells;
        (void)(started(l.stream, k_fill_u32, fill_blocks(cells), BLOCK, 0, first, cells, 0u) &&
               started(l.stream, k_row_count<true>, blocks, BLOCK, 0, s, g, row_count, first, where, n) &&
               started(l.stream, k_row_scan, scans, SCAN_BLOCK, 0, row_count, row_start) &&
               started(l.stream, k_cell_starts, waves, BLOCK, 0, g, row_start, first, rows) &&
               started(l.stream, k_row_scatter<true>, blocks, BLOCK, 0, where, row_start, first, row_count, g.slots, bucket, n) &&
               started(l.stream, k_cell_order, blocks, BLOCK, 0, where, first, bucket, order, n));
    } else {
        (void)(started(l.stream, k_row_count<false>, blocks, BLOCK, 0, s, g, row_count, first, where, n) &&
               started(l.stream, k_row_scan, scans, SCAN_BLOCK, 0, row_count, row_start) &&
               started(l.stream, k_row_scatter<false>, blocks, BLOCK, 0, where, row_start, first, row_count, g.slots, bucket, n) &&
               started(l.stream, k_row_order, waves, BLOCK, 0, g, row_start, bucket, where, order, first, rows));
    }
}

void launch_clear_u32(const Launch& l, uint32_t* p, size_t count, uint32_t value) {
    if (!count) return;
    k_fill_u32<<<fill_blocks(count), BLOCK, 0, l.stream>>>(p, count, value);
}

size_t bounds_partials(size_t n) { return size_t(grid_for(n)) * BOUND_VALUES; }
size_t bounds_values() { return BOUND_VALUES; }

void launch_advance(const Launch& l, DevState s, const osph_material* mats, Params prm, int mode, double dt,
                    double href, unsigned long long* small, bool vel, unsigned long long* part, size_t n) {
    if (!n) return;
    const unsigned g = grid_for(n);
    const bool v = vel;
    if (mode == 2) {
        if (v) k_advance<2, true><<<g, BLOCK, 0, l.stream>>>(s, mats, prm, dt, href, part, n);
        else k_advance<2, false><<<g, BLOCK, 0, l.stream>>>(s, mats, prm, dt, href, part, n);
    } else if (mode == 1) {
        if (v) k_advance<1, true><<<g, BLOCK, 0, l.stream>>>(s, mats, prm, dt, href, part, n);
        else k_advance<1, false><<<g, BLOCK, 0, l.stream>>>(s, mats, prm, dt, href, part, n);
    } else {
        if (v) k_advance<0, true><<<g, BLOCK, 0, l.stream>>>(s, mats, prm, dt, href, part, n);
        else k_advance<0, false><<<g, BLOCK, 0, l.stream>>>(s, mats, prm, dt, href, part, n);
    }
    k_bounds_final<<<v ? BOUND_VALUES : CLASS_VALUES * MAX_CLASSES, BLOCK, 0, l.stream>>>(part, g, small);
}

void launch_pack(const Launch& l, DevState s, Params prm, const uint32_t* order, PairRec* rec, double4* pos,
                 float4* posf, Screen sc, uint32_t* group, size_t n) {
    if (!n) return;
    k_pack<<<grid_for(n), BLOCK, 0, l.stream>>>(s, prm, order, rec, pos, posf, sc, group, n);
}

bool launch_neighbor_lists(const Launch& l, const double4* pos, const float4* posf, Screen sc, Grid g,
                           const uint32_t* first, uint32_t* list, uint32_t* count, uint32_t kmax, uint32_t* overflow,
                           size_t n) {
    if (!n) return true;
    const int b = l.tune.lists_block;
    const size_t lds = size_t(l.tune.lists_lds);
    if (lists_shared(g, n)) {
        const auto kernel = sc.on ? k_neighbor_lists_shared<true> : k_neighbor_lists_shared<false>;
        return started(l.stream, kernel, grid_for(n * LIST_LANES, b), unsigned(b), lds, pos, posf, sc, g, first, list, count,
                       kmax, overflow, n);
    }
    const auto kernel = sc.on ? k_neighbor_lists<true> : k_neighbor_lists<false>;
    return started(l.stream, kernel, grid_for(n, b), unsigned(b), lds, pos, posf, sc, g, first, list, count, kmax, overflow, n);
}

void launch_pairs_fp64(const Launch& l, DevState s, Params prm, const PairRec* rec, const uint32_t* group,
                       const uint32_t* order, const uint32_t* list, const uint32_t* count, const double* lut_grads,
                       uint32_t kmax, int nclass, size_t n, const FuseArgs* fuse) {
    if (!n) return;
    const int b = l.tune.pairs_block;
    const int lanes = pair_lanes(l.tune, n, nclass);
    const unsigned grid = grid_for(n * size_t(lanes), b);
    const size_t lds = size_t(l.tune.pairs_lds);
    const FuseArgs fa = fuse ? *fuse : FuseArgs{};
#define OSPH_PAIRS64(P, F) \
    k_pairs_fp64<P, F><<<grid, b, lds, l.stream>>>(s, prm, rec, group, order, list, count, lut_grads, kmax, n, fa)
    if (lanes == 16) {
        if (fuse) OSPH_PAIRS64(16, true); else OSPH_PAIRS64(16, false);
    } else if (lanes == 4) {
        if (fuse) OSPH_PAIRS64(4, true); else OSPH_PAIRS64(4, false);
    } else {
        if (fuse) OSPH_PAIRS64(1, true); else OSPH_PAIRS64(1, false);
    }
#undef OSPH_PAIRS64
}

void launch_pack_mixed(const Launch& l, DevState s, Params prm, Fixed fx, const uint32_t* order, PairRecF* rec,
                       double4* pos, float4* posf, Screen sc, uint32_t* group, size_t n) {
    if (!n) return;
    k_pack_mixed<<<grid_for(n), BLOCK, 0, l.stream>>>(s, prm, fx, order, rec, pos, posf, sc, group, n);
}

void launch_pairs_mixed(const Launch& l, DevState s, Params prm, Fixed fx, const PairRecF* rec, const uint32_t* group,
                        const uint32_t* order, const uint32_t* list, const uint32_t* count, uint32_t kmax, int nclass, size_t n,
                        const FuseArgs* fuse) {
    if (!n) return;
    const int b = l.tune.pairs_block;
    const int lanes = pair_lanes(l.tune, n, nclass);
    const unsigned grid = grid_for(n * size_t(lanes), b);
    const size_t lds = size_t(l.tune.pairs_lds);
    const FuseArgs fa = fuse ? *fuse : FuseArgs{};
#define OSPH_PAIRSMX(P, F) \
    k_pairs_mixed<P, F><<<grid, b, lds, l.stream>>>(s, prm, fx, rec, group, order, list, count, kmax, n, fa)
    if (lanes == 16) {
        if (fuse) OSPH_PAIRSMX(16, true); else OSPH_PAIRSMX(16, false);
    } else if (lanes == 4) {
        if (fuse) OSPH_PAIRSMX(4, true); else OSPH_PAIRSMX(4, false);
    } else {
        if (fuse) OSPH_PAIRSMX(1, true); else OSPH_PAIRSMX(1, false);
    }
#undef OSPH_PAIRSMX
}

void launch_finalize(const Launch& l, DevState s, const osph_material* mats, Params prm, size_t n) {
    if (!n) return;
    k_finalize<<<grid_for(n), BLOCK, 0, l.stream>>>(s, mats, prm, n);
}

void launch_zero_derivatives(const Launch& l, DevState s, size_t n) {
    if (!n) return;
    k_zero_derivatives<<<grid_for(n), BLOCK, 0, l.stream>>>(s, n);
}

void launch_finalize_correct(const Launch& l, DevState s, const osph_material* mats, Params prm, double dt,
                             unsigned long long* mins, const uint32_t* overflow, size_t n) {
    if (!n) return;
    k_finalize_correct<<<grid_for(n), BLOCK, 0, l.stream>>>(s, mats, prm, dt, mins, overflow, n);
}

void launch_count_stats(const Launch& l, const uint32_t* counts, unsigned long long* stats, size_t n) {
    if (!n) return;
    const unsigned g = grid_for(n);
    k_count_stats<<<g < STATS_BLOCKS ? g : STATS_BLOCKS, BLOCK, 0, l.stream>>>(counts, stats, n);
}

void launch_criteria(const Launch& l, DevState s, const osph_material* mats, Params prm, unsigned long long* mins,
                     size_t n) {
    if (!n) return;
    k_criteria<<<grid_for(n), BLOCK, 0, l.stream>>>(s, mats, prm, mins, n);
}

static StageDesc make_desc(int ncomp, const int* off, int elem, void* const* p) {
    StageDesc d{};
    d.ncomp = ncomp;
    d.elem = elem;
    for (int c = 0; c < ncomp && c < 8; ++c) {
        d.off[c] = off[c];
        d.p[c] = p[c];
    }
    return d;
}

void launch_stage_to_planes(const Launch& l, const unsigned char* staging, size_t stride, int ncomp,
                            const int* offsets_bytes, int elem_bytes, void* const* dst, const uint32_t* slot_of,
                            size_t n) {
    if (!n) return;
    StageDesc d = make_desc(ncomp, offsets_bytes, elem_bytes, dst);
    d.slot = slot_of;
    k_stage_to_planes<<<grid_for(n), BLOCK, 0, l.stream>>>(staging, stride, d, n);
}

void launch_planes_to_stage(const Launch& l, unsigned char* staging, size_t stride, int ncomp,
                            const int* offsets_bytes, int elem_bytes, void* const* src, const uint32_t* slot_of,
                            size_t n) {
    if (!n) return;
    StageDesc d = make_desc(ncomp, offsets_bytes, elem_bytes, src);
    d.slot = slot_of;
    k_planes_to_stage<<<grid_for(n), BLOCK, 0, l.stream>>>(staging, stride, d, n);
}

void launch_permute_state(const Launch& l, DevState src, DevState dst, const uint32_t* order, const uint32_t* perm_in,
                          uint32_t* perm_out, uint32_t* slot_of, size_t n) {
    if (!n) return;
    k_permute_state<<<grid_for(n), BLOCK, 0, l.stream>>>(src, dst, order, perm_in, perm_out, slot_of, n);
}

void launch_iota(const Launch& l, uint32_t* p, size_t n) {
    if (!n) return;
    k_iota_u32<<<grid_for(n), BLOCK, 0, l.stream>>>(p, n);
}

// ---- batched stages: one launch for every member of an ensemble ------------------------------------------
// Block b runs the single-run kernel's block bid = b - first[m] of the member m = member[b], out of the
// member's nb = first[m + 1] - first[m] blocks, on that member's buffers and parameters.

namespace {

__device__ __forceinline__ const BatchMember& batch_block(const BatchMember* __restrict__ M, const BatchBlocks& t,
                                                         uint32_t& m, uint32_t& bid, uint32_t& nb) {
    m = t.member[blockIdx.x];
    const uint32_t f = t.first[m];
    bid = blockIdx.x - f;
    nb = t.first[m + 1] - f;
    return M[m];
}

__device__ __forceinline__ uint32_t* overflow_of(const BatchMember& a) {
    return reinterpret_cast<uint32_t*>(a.small + SMALL_OVERFLOW);
}

__global__ void __launch_bounds__(SMALL_WORDS) kb_init_small(const BatchMember* __restrict__ M) {
    init_small_at(M[blockIdx.x].small, threadIdx.x);
}

template <bool VEL>
__global__ void __launch_bounds__(BLOCK) kb_advance(const BatchMember* __restrict__ M, BatchBlocks pb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, pb, m, bid, nb);
    advance_body<2, VEL>(bid, nb, a.s, a.mats, a.prm, a.dt, a.href, a.part, a.n);
}

__global__ void __launch_bounds__(BLOCK) kb_bounds_final(const BatchMember* __restrict__ M, BatchBlocks pb, int nv) {
    const uint32_t m = blockIdx.x / uint32_t(nv);
    const int vi = int(blockIdx.x % uint32_t(nv));
    const BatchMember& a = M[m];
    bounds_final_at(vi, a.part, pb.first[m + 1] - pb.first[m], a.small + SMALL_CLASSES, a.small + SMALL_VEL);
}

// The launches of a member's own sort, on each member's rows: 16 members of 5k to 212k particles 190 -> 45 us,
// against one radix sort of all members' keys and two kernels for the tables, 24 launches.
// (A stretched grid has up to 16.7M cells however few particles the member has, so these two take blocks of their own.)
constexpr unsigned CELL_BLOCKS = 256;  // per member
__global__ void __launch_bounds__(BLOCK) kb_cell_clear(const BatchMember* __restrict__ M) {
    const BatchMember& a = M[blockIdx.x / CELL_BLOCKS];
    if (!a.grid.by_cells) return;
    for (uint32_t t = blockIdx.x % CELL_BLOCKS * BLOCK + threadIdx.x; t < a.grid.cells; t += CELL_BLOCKS * BLOCK) {
        a.cell_first[t] = 0u;
    }
}

__global__ void __launch_bounds__(BLOCK) kb_row_count(const BatchMember* __restrict__ M, BatchBlocks pb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, pb, m, bid, nb);
    const size_t i = size_t(bid) * BLOCK + threadIdx.x;
    if (a.grid.by_cells) {
        row_count_at<true>(a.s, a.grid, a.row_count, a.cell_first, a.where, i, a.n);
    } else {
        row_count_at<false>(a.s, a.grid, a.row_count, a.cell_first, a.where, i, a.n);
    }
}

constexpr unsigned SCAN_BLOCKS = 8;  // per member, over its tiles
__global__ void __launch_bounds__(SCAN_BLOCK) kb_row_scan(const BatchMember* __restrict__ M) {
    const BatchMember& a = M[blockIdx.x / SCAN_BLOCKS];
    for (uint32_t t = blockIdx.x % SCAN_BLOCKS; t < a.grid.slots / SCAN_TILE + 1u; t += SCAN_BLOCKS) {
        row_scan_tile(a.row_count, a.row_start, t);
        __syncthreads();
    }
}

__global__ void __launch_bounds__(BLOCK) kb_cell_starts(const BatchMember* __restrict__ M) {
    const BatchMember& a = M[blockIdx.x / CELL_BLOCKS];
    if (!a.grid.by_cells) return;
    constexpr uint32_t WAVES = BLOCK / 64;
    for (uint32_t q = blockIdx.x % CELL_BLOCKS * WAVES + (threadIdx.x >> 6); q < a.rows; q += CELL_BLOCKS * WAVES) {
        cell_starts_at(a.grid, a.row_start, a.cell_first, a.rows, q);
    }
}

__global__ void __launch_bounds__(BLOCK) kb_row_scatter(const BatchMember* __restrict__ M, BatchBlocks pb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, pb, m, bid, nb);
    const size_t i = size_t(bid) * BLOCK + threadIdx.x, threads = size_t(nb) * BLOCK;
    if (a.grid.by_cells) {
        row_scatter_at<true>(a.where, a.row_start, a.cell_first, a.row_count, a.grid.slots, a.bucket, i, threads, a.n);
    } else {
        row_scatter_at<false>(a.where, a.row_start, a.cell_first, a.row_count, a.grid.slots, a.bucket, i, threads, a.n);
    }
}

__global__ void __launch_bounds__(BLOCK) kb_row_order(const BatchMember* __restrict__ M, BatchBlocks pb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, pb, m, bid, nb);
    if (a.grid.by_cells) {
        cell_order_at(a.where, a.cell_first, a.bucket, a.order, size_t(bid) * BLOCK + threadIdx.x, a.n);
        return;
    }
    for (size_t b = bid; b * (BLOCK / 64) < a.rows; b += nb) {
        row_order_block(a.grid, a.row_start, a.bucket, a.where, a.order, a.cell_first, a.rows, b);
        __syncthreads();
    }
}

// Members whose step reorders: the state into cell order (s -> s2), and the order becomes the identity
// (each thread reads its own order entry before it overwrites it).
__global__ void __launch_bounds__(BLOCK) kb_permute(const BatchMember* __restrict__ M, BatchBlocks pb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, pb, m, bid, nb);
    if (!a.reorder) return;
    const size_t k = size_t(bid) * BLOCK + threadIdx.x;
    if (k >= a.n) return;
    permute_at(a.s, a.s2, a.order, a.perm, a.perm2, a.slot_of, k);
    a.order[k] = uint32_t(k);
}

template <bool MIXED>
__global__ void __launch_bounds__(BLOCK) kb_pack(const BatchMember* __restrict__ M, BatchBlocks pb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, pb, m, bid, nb);
    const size_t k = size_t(xcd_block(bid, nb)) * BLOCK + threadIdx.x;
    if (k >= a.n) return;
    if constexpr (MIXED) {
        pack_mixed_at(a.s2, a.prm, a.fx, a.order, static_cast<PairRecF*>(a.rec), a.pos, a.posf, a.screen, a.group, k);
    } else {
        pack_at(a.s2, a.prm, a.order, static_cast<PairRec*>(a.rec), a.pos, a.posf, a.screen, a.group, k);
    }
}

// (Single lanes whatever the members' sizes: the members' grids, which the choice of groups goes by, are planned in every
// step, and the launch is captured once.)
template <bool SCREEN>
__global__ void __launch_bounds__(BLOCK) kb_lists(const BatchMember* __restrict__ M, BatchBlocks lb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, lb, m, bid, nb);
    if ((a.screen.on != 0) != SCREEN) return;
    const size_t k = size_t(xcd_block(bid, nb)) * blockDim.x + threadIdx.x;
    if (k >= a.n) return;
    neighbor_list_at<SCREEN>(a.pos, a.posf, a.screen, a.grid, a.cell_first, a.list, a.count, a.kmax, overflow_of(a), k);
}

template <bool MIXED, int LANES, bool FUSED>
__global__ void __launch_bounds__(BLOCK) kb_pairs(const BatchMember* __restrict__ M, BatchBlocks qb,
                                                  const double* __restrict__ lut) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, qb, m, bid, nb);
    const size_t t = size_t(xcd_block(bid, nb)) * blockDim.x + threadIdx.x;
    const FuseArgs fa{ a.mats, a.dt, a.small + SMALL_CRITERIA, overflow_of(a) };
    if constexpr (MIXED) {
        pairs_mixed_body<LANES, FUSED>(t, a.s2, a.prm, a.fx, static_cast<const PairRecF*>(a.rec), a.group, a.order,
                                     a.list, a.count, a.kmax, a.n, fa);
    } else {
        pairs_fp64_body<LANES, FUSED>(t, a.s2, a.prm, static_cast<const PairRec*>(a.rec), a.group, a.order, a.list,
                                    a.count, lut, a.kmax, a.n, fa);
    }
}

__global__ void __launch_bounds__(BLOCK) kb_finalize_correct(const BatchMember* __restrict__ M, BatchBlocks pb) {
    uint32_t m, bid, nb;
    const BatchMember& a = batch_block(M, pb, m, bid, nb);
    finalize_correct_body(size_t(bid) * BLOCK + threadIdx.x, a.s2, a.mats, a.prm, a.dt, a.small + SMALL_CRITERIA,
                          overflow_of(a), a.n);
}

}  // namespace

void batch_advance(const Launch& l, const BatchMember* M, int count, BatchBlocks pb, bool vel) {
    if (count <= 0) return;
    kb_init_small<<<count, SMALL_WORDS, 0, l.stream>>>(M);
    if (vel) {
        kb_advance<true><<<pb.total, BLOCK, 0, l.stream>>>(M, pb);
    } else {
        kb_advance<false><<<pb.total, BLOCK, 0, l.stream>>>(M, pb);
    }
    const int nv = vel ? BOUND_VALUES : CLASS_VALUES * MAX_CLASSES;
    kb_bounds_final<<<unsigned(count) * unsigned(nv), BLOCK, 0, l.stream>>>(M, pb, nv);
}

void batch_sort(const Launch& l, const BatchMember* M, int count, BatchBlocks pb, bool cells) {
    // as in launch_cell_sort
    (void)((!cells || started(l.stream, kb_cell_clear, CELL_BLOCKS * unsigned(count), BLOCK, 0, M)) && started(l.stream, kb_row_count, pb.total, BLOCK, 0, M, pb) &&
           started(l.stream, kb_row_scan, SCAN_BLOCKS * unsigned(count), SCAN_BLOCK, 0, M) &&
           (!cells || started(l.stream, kb_cell_starts, CELL_BLOCKS * unsigned(count), BLOCK, 0, M)) &&
           started(l.stream, kb_row_scatter, pb.total, BLOCK, 0, M, pb) && started(l.stream, kb_row_order, pb.total, BLOCK, 0, M, pb));
}

void batch_permute(const Launch& l, const BatchMember* M, BatchBlocks pb) {
    kb_permute<<<pb.total, BLOCK, 0, l.stream>>>(M, pb);
}

void batch_pack(const Launch& l, const BatchMember* M, BatchBlocks pb, bool mixed) {
    if (mixed) {
        kb_pack<true><<<pb.total, BLOCK, 0, l.stream>>>(M, pb);
    } else {
        kb_pack<false><<<pb.total, BLOCK, 0, l.stream>>>(M, pb);
    }
}

void batch_lists(const Launch& l, const BatchMember* M, BatchBlocks lb, bool screened, bool plain) {
    const int b = l.tune.lists_block;
    const size_t lds = size_t(l.tune.lists_lds);
    if (screened) kb_lists<true><<<lb.total, b, lds, l.stream>>>(M, lb);
    if (plain) kb_lists<false><<<lb.total, b, lds, l.stream>>>(M, lb);
}

void batch_pairs(const Launch& l, const BatchMember* M, BatchBlocks qb, bool mixed, bool fuse, int lanes,
                 const double* lut) {
    const int b = l.tune.pairs_block;
    const size_t lds = size_t(l.tune.pairs_lds);
#define OSPH_BPAIRS(MX, P, F) kb_pairs<MX, P, F><<<qb.total, b, lds, l.stream>>>(M, qb, lut)
#define OSPH_BPAIRS_OF(P)                                                       \
    do {                                                                        \
        if (mixed) {                                                            \
            if (fuse) OSPH_BPAIRS(true, P, true); else OSPH_BPAIRS(true, P, false);   \
        } else {                                                                \
            if (fuse) OSPH_BPAIRS(false, P, true); else OSPH_BPAIRS(false, P, false); \
        }                                                                       \
    } while (0)
    if (lanes == 16) OSPH_BPAIRS_OF(16);
    else if (lanes == 4) OSPH_BPAIRS_OF(4);
    else OSPH_BPAIRS_OF(1);
#undef OSPH_BPAIRS_OF
#undef OSPH_BPAIRS
}

void batch_finalize_correct(const Launch& l, const BatchMember* M, BatchBlocks pb) {
    kb_finalize_correct<<<pb.total, BLOCK, 0, l.stream>>>(M, pb);
}

}  // namespace osph

// ---- Grady-Kipp flaws on the device ------------------------------------------------------------------

namespace osph {
namespace {

// Uniform particle index of flaw p (1-based) of a body of nb particles: splitmix64 of seed + p times the
// golden-ratio increment, mapped to [0, nb) by the high word of a 64 x 64-bit product.
__device__ __forceinline__ uint32_t flaw_target(uint64_t seed, uint64_t p, uint32_t nb) {
    uint64_t x = seed + p * 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    x ^= x >> 31;
    return uint32_t(__umul64hi(x, uint64_t(nb)));
}

// Flaws p0 .. p0 + count - 1: the first flaw of each hit particle.
__global__ void __launch_bounds__(BLOCK) k_flaws_first(uint64_t seed, uint64_t p0, uint64_t count, uint32_t nb,
                                                       uint32_t* __restrict__ first) {
    const uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= count) return;
    const uint64_t p = p0 + t;
    atomicMin(&first[flaw_target(seed, p, nb)], uint32_t(p));
}

// Particles without a flaw and the largest first flaw (acc[0], acc[1]); one atomic per wavefront.
__global__ void __launch_bounds__(BLOCK) k_flaws_cover(const uint32_t* __restrict__ first, uint32_t nb,
                                                       uint32_t* __restrict__ acc) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t f = i < nb ? first[i] : 0u;
    const bool open = i < nb && f == 0xffffffffu;
    uint32_t mx = open ? 0u : f;
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, uint32_t(__shfl_xor(int(mx), o, 64)));
    const unsigned long long ballot = __ballot(open);
    if ((threadIdx.x & 63) == 0) {
        const uint32_t c = uint32_t(__popcll(ballot));
        if (c) atomicAdd(&acc[0], c);
        atomicMax(&acc[1], mx);
    }
}

// Flaws 1 .. K: count and last flaw of each particle.
__global__ void __launch_bounds__(BLOCK) k_flaws_count(uint64_t seed, uint32_t K, uint32_t nb,
                                                       uint32_t* __restrict__ cnt, uint32_t* __restrict__ last) {
    const uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= K) return;
    const uint64_t p = t + 1;
    const uint32_t i = flaw_target(seed, p, nb);
    atomicAdd(&cnt[i], 1u);
    atomicMax(&last[i], uint32_t(p));
}

// ScalarGradyKippModel::setFlaws (core/physics/Damage.cpp:17-126), accumulate mode, per particle of the
// body: eps_min / eps_max of its first / last flaw, eps(p) = denom p^(1/m); m_zero = ln n / ln(eps_max /
// eps_min) for n > 1 flaws, else 1; growth = cg / (2 h).
__global__ void __launch_bounds__(BLOCK) k_flaws_finish(DevState s, const uint32_t* __restrict__ slot_of,
                                                        size_t body_first, uint32_t nb,
                                                        const uint32_t* __restrict__ first,
                                                        const uint32_t* __restrict__ last,
                                                        const uint32_t* __restrict__ cnt, double denom,
                                                        double inv_m, double cg) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nb) return;
    const uint32_t slot = slot_of[body_first + i];
    const double emin = denom * pow(double(first[i]), inv_m);
    const double emax = denom * pow(double(last[i]), inv_m);
    const uint32_t n = cnt[i];
    s.d[EPSMIN][slot] = emin;
    s.d[MZERO][slot] = n > 1 ? log(double(n)) / log(emax / emin) : 1.0;
    s.d[GROWTH][slot] = cg / (2.0 * s.d[H][slot]);
    s.u[NFLAWS][slot] = n;
}

}  // namespace

int flaws_first_pass(const Launch& l, uint64_t seed, uint64_t p0, uint64_t count, uint32_t nb, uint32_t* first) {
    if (!count) return 0;
    const uint64_t blocks = (count + BLOCK - 1) / BLOCK;
    k_flaws_first<<<unsigned(blocks), BLOCK, 0, l.stream>>>(seed, p0, count, nb, first);
    return 0;
}

void flaws_cover(const Launch& l, const uint32_t* first, uint32_t nb, uint32_t* acc) {
    k_fill_u32<<<1, 64, 0, l.stream>>>(acc, 2, 0u);
    k_flaws_cover<<<grid_for(nb), BLOCK, 0, l.stream>>>(first, nb, acc);
}

void flaws_count_pass(const Launch& l, uint64_t seed, uint32_t K, uint32_t nb, uint32_t* cnt, uint32_t* last) {
    k_flaws_count<<<unsigned((uint64_t(K) + BLOCK - 1) / BLOCK), BLOCK, 0, l.stream>>>(seed, K, nb, cnt, last);
}

void flaws_finish(const Launch& l, DevState s, const uint32_t* slot_of, size_t body_first, uint32_t nb,
                  const uint32_t* first, const uint32_t* last, const uint32_t* cnt, double denom, double inv_m,
                  double cg) {
    k_flaws_finish<<<grid_for(nb), BLOCK, 0, l.stream>>>(s, slot_of, body_first, nb, first, last, cnt, denom, inv_m,
                                                          cg);
}

}  // namespace osph
