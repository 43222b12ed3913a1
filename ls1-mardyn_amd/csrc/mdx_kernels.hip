// mdx_kernels.hip -- gfx950 kernels of the short-range force path.
//
// Step = leapfrog_pre (half kick, drift, periodic wrap, binning) -> scan ->
//        bin_scatter -> bin_gather (stable counting sort) -> site scan ->
//        build_sites -> pair kernels (one per i-site type) -> leapfrog_post (site
//        sums = calcFM, half kick) -> step_end (the step's sums and record).
// Consecutive steps without a thermostat take leapfrog_post and the next step's
// leapfrog_pre in one pass (leapfrog_post_pre).
// Systems of one-centre LJ molecules only: bin_gather_point (gather + site
// cache) -> LJ pair kernel (writes molecule F, Vi) -> leapfrog_post.
// Called one by one (re-bin, traversal, kicks) the same operations run unfused:
// bin_count and calc_fm are then passes of their own.
//
// Pair kernels (mdx_pairs.hip; small dense boxes: mdx_pairs_block.hip): one
// 64-lane wavefront per cell. Lane = (i-site, j-phase):
// the cell's n sites of the i type occupy n lanes per phase and the
// min(floor(64/n), 8) phases stride over the j sites of the 27 neighbour cells
// (periodic images through shift vectors, no halo copies). Stage A tests the
// molecule-centre cutoff of every candidate and appends hits to a per-lane
// list in LDS; stage B evaluates the site-pair bodies for the dense list, so
// lanes do not idle on the 85% of candidates outside the cutoff. Every site
// accumulates only its own force, virial and torque (owner computes), so no
// atomics and no colouring are needed and results are deterministic; each
// unordered pair is evaluated from both sides and the macroscopic sums are
// halved. Phases are folded through LDS at the end of the cell.
#include "mdx_internal.h"

namespace mdx {

// ------------------------------------------------------------------ helpers
// The quaternion helpers and the Leapfrog updates round every product and sum
// on its own (fp contract off, as the oracle is built), so a fused pass over
// two half steps and the separate passes give the same bits.

// Quaternion::rotate (src/molecules/Quaternion.cpp:43-64)
__device__ __forceinline__ void qrot(const double q[4], const double d[3], double o[3]) {
#pragma clang fp contract(off)
    o[0] = o[1] = o[2] = 0.0;
    if (d[0] == 0.0 && d[1] == 0.0 && d[2] == 0.0) return;
    double ww = q[0] * q[0], xx = q[1] * q[1], yy = q[2] * q[2], zz = q[3] * q[3];
    double wx = q[0] * q[1], wy = q[0] * q[2], wz = q[0] * q[3];
    double xy = q[1] * q[2], xz = q[1] * q[3], yz = q[2] * q[3];
    o[0] = (ww + xx - yy - zz) * d[0] + 2. * (xy - wz) * d[1] + 2. * (wy + xz) * d[2];
    o[1] = 2. * (wz + xy) * d[0] + (ww - xx + yy - zz) * d[1] + 2. * (yz - wx) * d[2];
    o[2] = 2. * (xz - wy) * d[0] + 2. * (wx + yz) * d[1] + (ww - xx - yy + zz) * d[2];
}

// Quaternion::rotateinv (Quaternion.cpp:66-86)
__device__ __forceinline__ void qrotinv(const double q[4], const double d[3], double o[3]) {
#pragma clang fp contract(off)
    o[0] = o[1] = o[2] = 0.0;
    if (d[0] == 0.0 && d[1] == 0.0 && d[2] == 0.0) return;
    double ww = q[0] * q[0], xx = q[1] * q[1], yy = q[2] * q[2], zz = q[3] * q[3];
    double wx = q[0] * q[1], wy = q[0] * q[2], wz = q[0] * q[3];
    double xy = q[1] * q[2], xz = q[1] * q[3], yz = q[2] * q[3];
    o[0] = (ww + xx - yy - zz) * d[0] + 2. * (xy + wz) * d[1] + 2. * (xz - wy) * d[2];
    o[1] = 2. * (xy - wz) * d[0] + (ww - xx + yy - zz) * d[1] + 2. * (yz + wx) * d[2];
    o[2] = 2. * (xz + wy) * d[0] + 2. * (yz - wx) * d[1] + (ww - xx - yy + zz) * d[2];
}

// Quaternion::differentiate (Quaternion.cpp:98-103)
__device__ __forceinline__ void qdiff(const double q[4], const double w[3], double dq[4]) {
#pragma clang fp contract(off)
    dq[0] = .5 * (-q[1] * w[0] - q[2] * w[1] - q[3] * w[2]);
    dq[1] = .5 * (q[0] * w[0] - q[3] * w[1] + q[2] * w[2]);
    dq[2] = .5 * (q[3] * w[0] + q[0] * w[1] - q[1] * w[2]);
    dq[3] = .5 * (-q[2] * w[0] + q[1] * w[1] + q[0] * w[2]);
}

// CellBorderAndFlagManager::getBorder (CellBorderAndFlagManager.h:134-152).
// Contraction off: the cell id must match the reference bit for bit.
__device__ __forceinline__ double cell_border(const Geom &g, int idx, int d) {
#pragma clang fp contract(off)
    if (idx == 0) return g.halo_min[d];
    if (idx == 1) return g.bbmin[d];
    if (idx == g.cpd[d] - 1) return g.bbmax[d];
    if (idx == g.cpd[d]) return g.halo_max[d];
    return idx * g.cl[d] + g.halo_min[d];
}

// LinkedCells::getCellIndexOfPoint (LinkedCells.cpp:870-923): 3-D ls1 index
// (halo layer included).
__device__ __forceinline__ void ls1_cell3(const Geom &g, const double p[3], int ci[3]) {
#pragma clang fp contract(off)
    double lp[3] = {p[0], p[1], p[2]};
    for (int d = 0; d < 3; ++d) {
        if (lp[d] <= g.halo_min[d])
            lp[d] += g.cl[d] * 0.5;
        else if (lp[d] >= g.halo_max[d])
            lp[d] -= g.cl[d] * 0.5;
        int v = (int)floor((lp[d] - g.bbmin[d]) * g.rcl[d]) + 1;
        v = v < 0 ? 0 : v;
        v = v > g.cpd[d] - 1 ? g.cpd[d] - 1 : v;
        ci[d] = v;
    }
    bool inside = true;
    for (int d = 0; d < 3; ++d)
        inside = inside && cell_border(g, ci[d], d) <= lp[d] && lp[d] < cell_border(g, ci[d] + 1, d);
    if (!inside) {
        for (int d = 0; d < 3; ++d) {
            if (lp[d] < cell_border(g, ci[d], d))
                ci[d]--;
            else if (lp[d] >= cell_border(g, ci[d] + 1, d))
                ci[d]++;
        }
    }
}

// Inner cell index from an ls1 3-D index (x fastest, like
// LinkedCells::cellIndexOf3DIndex, LinkedCells.cpp:925-927).
__device__ __forceinline__ int inner_index(const Geom &g, const int ci[3]) {
    int x = min(max(ci[0] - 1, 0), g.n[0] - 1);
    int y = min(max(ci[1] - 1, 0), g.n[1] - 1);
    int z = min(max(ci[2] - 1, 0), g.n[2] - 1);
    return (z * g.n[1] + y) * g.n[0] + x;
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// --------------------------------------------------------------- Leapfrog

// Rotational half of FullMolecule::upd_preF (FullMolecule.cpp:340-360):
// L += dt/2 M, q advanced with the half-step angular velocity, normalised.
// Point molecules skip it: their invI and torque are 0, so L is unchanged and
// q only re-normalised (which k_build_sites does every step, as ls1's
// setupSoACache does).
__device__ __forceinline__ void rotate_pre(MolArrays &s, const double M[3], const Component &c,
                                           double dt, int i) {
#pragma clang fp contract(off)
    const double dt_halve = .5 * dt;
    double q[4] = {s.qw[i], s.qx[i], s.qy[i], s.qz[i]};
    double L[3] = {s.Lx[i], s.Ly[i], s.Lz[i]};
    double w[3], qh[4], qi[4];
    qrotinv(q, L, w);
    for (int d = 0; d < 3; ++d) w[d] *= c.invI[d];
    qdiff(q, w, qh);
    for (int k = 0; k < 4; ++k) qh[k] = qh[k] * dt_halve + q[k];
    double qc = 1. / sqrt(qh[0] * qh[0] + qh[1] * qh[1] + qh[2] * qh[2] + qh[3] * qh[3]);
    for (int k = 0; k < 4; ++k) qh[k] *= qc;
    for (int d = 0; d < 3; ++d) L[d] += dt_halve * M[d];
    qrotinv(qh, L, w);
    for (int d = 0; d < 3; ++d) w[d] *= c.invI[d];
    qdiff(qh, w, qi);
    for (int k = 0; k < 4; ++k) q[k] += qi[k] * dt;
    qc = 1. / sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
    for (int k = 0; k < 4; ++k) q[k] *= qc;
    s.qw[i] = q[0]; s.qx[i] = q[1]; s.qy[i] = q[2]; s.qz[i] = q[3];
    s.Lx[i] = L[0]; s.Ly[i] = L[1]; s.Lz[i] = L[2];
}

// FullMolecule::upd_preF (FullMolecule.cpp:331-361), then the periodic wrap of
// DomainDecompBase::handleDomainLeavingParticles (DomainDecompBase.cpp:199-249),
// for molecule i with its velocity v, force f (null: PositionCellProcessorRMM,
// r += dt v only) and torque M in registers. Writes r (also to r[]) and v.
__device__ __forceinline__ void lf_pre_mol(MolArrays &s, const double M[3], const Component &c,
                                           const Geom &g, double dt, int i, double v[3],
                                           const double *f, double r[3]) {
#pragma clang fp contract(off)
    const double dt_halve = .5 * dt;
    const double dtInv2m = dt_halve / c.m;
    r[0] = s.rx[i], r[1] = s.ry[i], r[2] = s.rz[i];
    if (r[0] != r[0]) return;  // deleted at an outflow wall: no longer moved
    if (f && (g.reflect[0] | g.reflect[1] | g.reflect[2] | g.outflow[0] | g.outflow[1] |
              g.outflow[2])) {
        // BoundaryHandler::processGlobalWallLeavingParticles (BoundaryHandler.cpp:
        // 82-134; called before upd_preF, Simulation.cpp:1114), walls in the
        // order +x, -x, +y, -y, +z, -z: a molecule in the wall's slab of width
        // rc (RegionUtils.cpp:11-45, inBox l <= r < u) whose predicted position
        // r + dt (v + dt/2m F) reaches the wall (RegionUtils.cpp:47-56) gets
        // v = -v - 2 dt/2m F at a reflecting wall, so the coming half kick
        // leaves it moving away at -(v + dt/2m F), and is deleted at an
        // outflow wall (later walls no longer see it)
        bool inside = true;
        for (int d = 0; d < 3; ++d) inside = inside && r[d] >= g.bbmin[d] && r[d] < g.bbmax[d];
        bool dead = false;
        for (int d = 0; d < 3 && inside && !dead; ++d) {
            if (!g.reflect[d] && !g.outflow[d]) continue;
            const double adj = dtInv2m * f[d];
            // +wall: slab [max(max - rc, min), max)
            if (r[d] >= fmax(g.bbmax[d] - g.wall_rc, g.bbmin[d]) &&
                r[d] + dt * (v[d] + adj) >= g.bbmax[d]) {
                if (g.reflect[d])
                    v[d] = -v[d] - adj - adj;
                else
                    dead = true;
            }
            // -wall: slab [min, min(min + rc, max))
            if (!dead && r[d] < fmin(g.bbmin[d] + g.wall_rc, g.bbmax[d]) &&
                r[d] + dt * (v[d] + adj) <= g.bbmin[d]) {
                if (g.reflect[d])
                    v[d] = -v[d] - adj - adj;
                else
                    dead = true;
            }
        }
        if (dead) {
            r[0] = s.rx[i] = s.ry[i] = s.rz[i] = __builtin_nan("");
            return;
        }
    }
    for (int d = 0; d < 3; ++d) {
        if (f) v[d] += dtInv2m * f[d];
        r[d] += dt * v[d];
    }
    if (!c.point) rotate_pre(s, M, c, dt, i);
    for (int d = 0; d < 3; ++d) {
        if (!g.pdim[d]) continue;
        double x = r[d];
        if (x < g.bbmin[d]) {
            x = x + g.L[d];
            if (x >= g.bbmax[d]) x = nextafter(g.bbmax[d], -INFINITY);
        } else if (x >= g.bbmax[d]) {
            x = x - g.L[d];
            if (x <= g.bbmin[d]) x = g.bbmin[d];
        }
        r[d] = x;
    }
    s.rx[i] = r[0]; s.ry[i] = r[1]; s.rz[i] = r[2];
    s.vx[i] = v[0]; s.vy[i] = v[1]; s.vz[i] = v[2];
}

// Cell of molecule i at p (ls1 index -> inner index) and its arrival rank in
// the cell, for every lane of the wave (in: the lane has a molecule; the lanes
// that have one come first). Molecules are stored in cell order, so a wave's
// lanes form a few runs of equal cells: the first lane of each run takes one
// atomic for the whole run, and all runs' atomics go out in the same
// instruction (one round trip per wave; a cell that shows up in two runs gets
// two disjoint rank ranges).
__device__ __forceinline__ void bin_mol(const double p[3], const Reps &R, int i, bool in,
                                        const Bins &b) {
    const int lane = threadIdx.x & 63;
    int c = -1;
    if (in) {
        if (p[0] != p[0] && R.nrep == 1) {
            // deleted at an outflow wall: the bin behind the last cell, which
            // no traversal visits
            c = R.cell_off[1];
            b.ls1id[i] = -1;
        } else {
            const int rep = mol_replica(R, i);
            const Geom &g = R.geom[rep];
            int ci[3];
            ls1_cell3(g, p, ci);
            c = R.cell_off[rep] + inner_index(g, ci);
            b.ls1id[i] = (ci[2] * g.cpd[1] + ci[1]) * g.cpd[0] + ci[0];
        }
        b.cell[i] = c;
    }
    const int cprev = __shfl_up(c, 1, 64);
    const bool head = in && (lane == 0 || cprev != c);
    const unsigned long long heads = __ballot(head);
    const unsigned long long valid = __ballot(in);
    // my run's head: the highest head at or below my lane
    const unsigned long long upto = (2ull << lane) - 1ull;  // lanes 0..lane (all for 63)
    const unsigned long long below = heads & upto;
    const int h = in ? 63 - __clzll((long long)below) : 0;
    int base = 0;
    if (head) {
        // the run ends at the next head or at the last valid lane
        const unsigned long long after = heads & ~upto;
        const int end = after ? __ffsll((long long)after) - 1 : 64 - __clzll((long long)valid);
        base = atomicAdd(&b.count[c], end - lane);
    }
    base = __shfl(base, h, 64);
    if (in) b.rank[i] = base + (lane - h);
}

// bins.count non-null: the moved molecules are also binned (the next re-bin's
// k_bin_count, with r in registers).
__global__ __launch_bounds__(256) void k_leapfrog_pre(MolArrays s, const double *__restrict__ F,
                                                      const double *__restrict__ M,
                                                      const Component *__restrict__ comps, Reps R,
                                                      double dt, int n, Bins bins) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    double r[3] = {0., 0., 0.};
    if (i < n) {
        double v[3] = {s.vx[i], s.vy[i], s.vz[i]};
        double f[3] = {0., 0., 0.}, m[3] = {0., 0., 0.};
        const Component &c = comps[s.cid[i]];
        if (F) f[0] = F[i], f[1] = F[n + i], f[2] = F[2 * n + i];
        if (!c.point) m[0] = M[i], m[1] = M[n + i], m[2] = M[2 * n + i];
        lf_pre_mol(s, m, c, R.geom[mol_replica(R, i)], dt, i, v, F ? f : nullptr, r);
    }
    if (bins.count) bin_mol(r, R, i, i < n, bins);
}

// FullMolecule::upd_postF (FullMolecule.cpp:363-387) for molecule i: v (in
// registers) and L advanced, {m v^2, I w^2} added to the sums.
__device__ __forceinline__ void lf_post_mol(MolArrays &s, const double M[3], const Component &c,
                                            double dt, int i, double v[3], const double f[3],
                                            double &mv2, double &iw2) {
#pragma clang fp contract(off)
    const double dt_halve = 0.5 * dt;
    const double dtInv2m = dt_halve / c.m;
    double v2 = 0.;
    for (int d = 0; d < 3; ++d) {
        v[d] += dtInv2m * f[d];
        v2 += v[d] * v[d];
    }
    mv2 = c.m * v2;
    if (!c.point) {  // point molecules: L unchanged, I w^2 = 0
        double L[3] = {s.Lx[i], s.Ly[i], s.Lz[i]};
        for (int d = 0; d < 3; ++d) L[d] += dt_halve * M[d];
        double q[4] = {s.qw[i], s.qx[i], s.qy[i], s.qz[i]};
        double w[3];
        qrotinv(q, L, w);
        for (int d = 0; d < 3; ++d) {
            w[d] *= c.invI[d];
            iw2 += c.I[d] * w[d] * w[d];
        }
        s.Lx[i] = L[0]; s.Ly[i] = L[1]; s.Lz[i] = L[2];
    }
}

// Block partial sums {sum m v^2, sum I w^2, N, rotDOF} (Leapfrog.cpp:63-147).
__device__ __forceinline__ void lf_block_sums(double mv2, double iw2, double cnt, double rot,
                                              double *partial) {
    __shared__ double red[4][4];
    mv2 = wave_sum(mv2);
    iw2 = wave_sum(iw2);
    cnt = wave_sum(cnt);
    rot = wave_sum(rot);
    int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    if (ln == 0) {
        red[wv][0] = mv2; red[wv][1] = iw2; red[wv][2] = cnt; red[wv][3] = rot;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double a = 0;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) a += red[k][threadIdx.x];
        partial[blockIdx.x * 4 + threadIdx.x] = a;
    }
}

// Fixed-order sums of nblocks rows of gridDim.x values, one block per column
// (the columns one after the other in one block took 54 us for 4096 rows of 16,
// now 9). Deterministic.
__global__ __launch_bounds__(256) void k_reduce_partials(const double *__restrict__ partial,
                                                         int nblocks, double *out) {
    __shared__ double red[256];
    const int w = blockIdx.x, width = gridDim.x;
    double a = 0;
    for (int b = threadIdx.x; b < nblocks; b += 256) a += partial[(size_t)b * width + w];
    red[threadIdx.x] = a;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[w] = red[0];
}

// ---------------------------------------------------------------- binning

__global__ void k_fill_int(int *a, int n, int v) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

__global__ __launch_bounds__(256) void k_bin_count(MolArrays s, Reps R, int n, Bins b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = i < n;
    double p[3] = {0., 0., 0.};
    if (in) p[0] = s.rx[i], p[1] = s.ry[i], p[2] = s.rz[i];
    bin_mol(p, R, i, in, b);
}

__global__ __launch_bounds__(256) void k_bin_scatter(int n, const int *__restrict__ cell,
                                                     const int *__restrict__ rank,
                                                     const int *__restrict__ start, int *perm) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    perm[start[cell[i]] + rank[i]] = i;
}

// Destination of entry p of perm (cells in order, each cell's members in
// arrival order): its cell's start plus its stable rank in the cell, the
// number of members with a smaller previous index (which makes the sort
// deterministic and keeps molecules that stay in their cell in order). The
// block's cells occupy one contiguous range of perm, staged in LDS when it
// fits (the rank loops then read LDS); every thread of the block must call
// this. Returns -1 for p >= n.
constexpr int kGatherWin = 1024;
__device__ __forceinline__ int stable_dest(int p, int n, const int *__restrict__ cell,
                                           const int *__restrict__ perm,
                                           const int *__restrict__ start, int *win, int *src_i,
                                           int *cell_of) {
    const int p0 = blockIdx.x * blockDim.x, p1 = min(p0 + (int)blockDim.x, n);
    const int w0 = start[cell[perm[p0]]], w1 = start[cell[perm[p1 - 1]] + 1];
    const bool staged = w1 - w0 <= kGatherWin;
    if (staged)
        for (int k = w0 + (int)threadIdx.x; k < w1; k += blockDim.x) win[k - w0] = perm[k];
    __syncthreads();
    if (p >= n) return -1;
    const int i = perm[p];
    const int c = cell[i];
    const int b = start[c], e = start[c + 1];
    int r = 0;
    if (staged)
        for (int k = b; k < e; ++k) r += win[k - w0] < i;
    else
        for (int k = b; k < e; ++k) r += perm[k] < i;
    *src_i = i;
    *cell_of = c;
    return b + r;
}

// The permutation of the state into cell order (i -> d); q and L are left to
// the caller.
__device__ __forceinline__ void gather_common(int i, int d, int c, const MolArrays &src,
                                              const MolArrays &dst, int *newcell,
                                              const int *__restrict__ ls1id, int *newls1id) {
    dst.rx[d] = src.rx[i]; dst.ry[d] = src.ry[i]; dst.rz[d] = src.rz[i];
    dst.vx[d] = src.vx[i]; dst.vy[d] = src.vy[i]; dst.vz[d] = src.vz[i];
    dst.cid[d] = src.cid[i];
    dst.orig[d] = src.orig[i];
    newcell[d] = c;
    newls1id[d] = ls1id[i];
}

__global__ __launch_bounds__(256) void k_bin_gather(int n, MolArrays src, MolArrays dst,
                                                    const int *__restrict__ cell,
                                                    const int *__restrict__ perm,
                                                    const int *__restrict__ start, int *newcell,
                                                    const int *__restrict__ ls1id, int *newls1id,
                                                    const Component *__restrict__ comps,
                                                    int *nsite0, int *nsite1, int *nsite2,
                                                    int *nsite3) {
    __shared__ int win[kGatherWin];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    int i, c;
    const int d = stable_dest(p, n, cell, perm, start, win, &i, &c);
    if (d < 0) return;
    gather_common(i, d, c, src, dst, newcell, ls1id, newls1id);
    dst.qw[d] = src.qw[i]; dst.qx[d] = src.qx[i]; dst.qy[d] = src.qy[i]; dst.qz[d] = src.qz[i];
    dst.Lx[d] = src.Lx[i]; dst.Ly[d] = src.Ly[i]; dst.Lz[d] = src.Lz[i];
    const Component &cp = comps[src.cid[i]];
    nsite0[d] = cp.n[0];
    nsite1[d] = cp.n[1];
    nsite2[d] = cp.n[2];
    nsite3[d] = cp.n[3];
}

// The same for systems whose every component is one LJ centre at the
// molecule's centre and nothing else: site j is molecule j, so the gather
// also does the SoA cache build of k_build_sites for them: the FP32 position
// relative to the cell corner and the LJ lookup id. Site FP64 positions,
// forces and virials are the molecule arrays themselves. q and L of such
// molecules never change and stay in upload order (q's normalisation of
// setupSoACache, FullMolecule.cpp:719, is applied by k_normalize_q).
__global__ __launch_bounds__(256) void k_bin_gather_point(
    int n, MolArrays src, MolArrays dst, const int *__restrict__ cell,
    const int *__restrict__ perm, const int *__restrict__ start, int *newcell,
    const int *__restrict__ ls1id, int *newls1id, const Component *__restrict__ comps, Reps R,
    float4 *f, int *ljid) {
    __shared__ int win[kGatherWin];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    int i, c;
    const int d = stable_dest(p, n, cell, perm, start, win, &i, &c);
    if (d < 0) return;
    gather_common(i, d, c, src, dst, newcell, ls1id, newls1id);
    const int rep = c < R.cell_off[R.nrep] ? cell_replica(R, c) : 0;  // deleted: the last bin
    const Geom &g = R.geom[rep];
    const int local = c - R.cell_off[rep];
    const int cx = local % g.n[0], cy = (local / g.n[0]) % g.n[1], cz = local / (g.n[0] * g.n[1]);
    const int id = comps[src.cid[i]].lj_base;
    f[d] = make_float4((float)(src.rx[i] - (g.bbmin[0] + cx * g.cl[0])),
                       (float)(src.ry[i] - (g.bbmin[1] + cy * g.cl[1])),
                       (float)(src.rz[i] - (g.bbmin[2] + cz * g.cl[2])),
                       __int_as_float(4 * id));
    ljid[d] = id;
}

// q <- N^k(q), N = Quaternion::normalize (q scaled by 1/sqrt(|q|^2)), for
// molecules whose q is touched by nothing else (one-centre systems, where ls1
// normalises every molecule at each of the k container updates). N reaches a
// fixed point or a two-cycle after a few applications (|q|^2 is then 1 to
// within an ulp or two); the rest of the k are skipped, or reduced to their
// parity for a two-cycle. The loop is capped at kMaxNormalize applications,
// far beyond where the sequence settles.
constexpr long long kMaxNormalize = 64;
__global__ __launch_bounds__(256) void k_normalize_q(int n, MolArrays s, long long k) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double q[4] = {s.qw[i], s.qx[i], s.qy[i], s.qz[i]}, qp[4] = {0, 0, 0, 0};
    for (long long t = 0; t < k && t < kMaxNormalize; ++t) {
        const double qs = 1. / sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
        double qn[4];
        for (int c = 0; c < 4; ++c) qn[c] = q[c] * qs;
        bool same = true, cyc = t > 0;
        for (int c = 0; c < 4; ++c) {
            same = same && qn[c] == q[c];
            cyc = cyc && qn[c] == qp[c];
        }
        if (same) break;
        if (cyc) {  // q <-> qn: the remaining k - t applications alternate
            if ((k - t) & 1)
                for (int c = 0; c < 4; ++c) q[c] = qn[c];
            break;
        }
        for (int c = 0; c < 4; ++c) {
            qp[c] = q[c];
            q[c] = qn[c];
        }
    }
    s.qw[i] = q[0]; s.qx[i] = q[1]; s.qy[i] = q[2]; s.qz[i] = q[3];
}

// ------------------------------------------------------------- scan (int)

// Inclusive scan over the wave.
__device__ __forceinline__ int wave_incl(int x, int lane) {
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    return x;
}

// Exclusive scan of up to kScanOne ints by one block of 1024 threads: four
// tiles of 4096, all loaded at once, the 64 wave sums (tile-major) scanned by
// every wave for itself. One launch of 4.7 us where block scan, scan of the block
// sums, addition and total were four of about 4 us each (2744 cells).
__global__ __launch_bounds__(1024) void k_scan_one(ScanArgs a) {
    __shared__ int ws[64];
    const int *in = a.in[blockIdx.y];
    int *out = a.out[blockIdx.y];
    const int n = a.n, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int v[4][4], incl[4];
    for (int t = 0; t < 4; ++t) {
        const int base = t * 4096 + threadIdx.x * 4;
        for (int k = 0; k < 4; ++k) v[t][k] = base + k < n ? in[base + k] : 0;
    }
    for (int t = 0; t < 4; ++t) {
        incl[t] = wave_incl(v[t][0] + v[t][1] + v[t][2] + v[t][3], lane);
        if (lane == 63) ws[t * 16 + wv] = incl[t];
    }
    __syncthreads();
    const int w = ws[lane], wi = wave_incl(w, lane);
    for (int t = 0; t < 4; ++t) {
        const int base = t * 4096 + threadIdx.x * 4;
        const int woff = __shfl(wi - w, t * 16 + wv, 64);
        int excl = woff + incl[t] - (v[t][0] + v[t][1] + v[t][2] + v[t][3]);
        for (int k = 0; k < 4; ++k) {
            if (base + k < n) {
                out[base + k] = excl;
                if (a.clear) const_cast<int *>(in)[base + k] = 0;
            }
            excl += v[t][k];
        }
    }
    if (threadIdx.x == 63) out[n] = wi;
}

// Exclusive scan of blocks of 1024 ints (256 threads x 4); block totals out.
__global__ __launch_bounds__(256) void k_scan_block(ScanArgs a) {
    __shared__ int ws[4];
    const int *in = a.in[blockIdx.y];
    int *out = a.out[blockIdx.y];
    const int n = a.n;
    int base = blockIdx.x * 1024 + threadIdx.x * 4;
    int v[4], t = 0;
    for (int k = 0; k < 4; ++k) {
        v[k] = (base + k < n) ? in[base + k] : 0;
        t += v[k];
    }
    // inclusive scan of t across the block
    int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int x = wave_incl(t, lane);
    if (lane == 63) ws[wv] = x;
    __syncthreads();
    int woff = 0;
    for (int k = 0; k < wv; ++k) woff += ws[k];
    int excl = woff + x - t;
    for (int k = 0; k < 4; ++k) {
        if (base + k < n) {
            out[base + k] = excl;
            if (a.clear) const_cast<int *>(in)[base + k] = 0;
        }
        excl += v[k];
    }
    if (threadIdx.x == 255) a.aux[blockIdx.y][blockIdx.x] = woff + x;
}

// Adds what the blocks before sum to: aux holds their scan (scanned), or their
// sums, which the block then adds up itself (a few thousand at most: cheaper
// than a launch of their own). The last block writes the total.
__global__ __launch_bounds__(256) void k_scan_add(ScanArgs a) {
    __shared__ int ws[4];
    const int *aux = a.aux[blockIdx.y];
    int *out = a.out[blockIdx.y];
    const int n = a.n, nb = gridDim.x, b = blockIdx.x;
    int off = 0, own = 0;
    if (a.scanned) {
        off = aux[b];
        own = aux[b + 1] - off;
    } else {
        for (int k = threadIdx.x; k < b; k += 256) off += aux[k];
        off = wave_incl(off, threadIdx.x & 63);
        if ((threadIdx.x & 63) == 63) ws[threadIdx.x >> 6] = off;
        __syncthreads();
        off = ws[0] + ws[1] + ws[2] + ws[3];
        own = aux[b];
    }
    int i = b * 1024 + threadIdx.x;
    for (int k = 0; k < 4; ++k) {
        int j = i + k * 256;
        if (j < n) out[j] += off;
    }
    if (b == nb - 1 && threadIdx.x == 0) out[n] = off + own;
}

// --------------------------------------------------- SoA site cache build

// The block's copy of the component table (ncomp records) in LDS: the site
// loops read offsets, axes and parameters per site, and a component's record
// is then one LDS read away instead of a global load after the cid load.
// Every thread of the block must call it (it synchronises the block).
__device__ __forceinline__ const Component *stage_comps(const Component *__restrict__ comps,
                                                        int ncomp) {
    extern __shared__ double comp_lds[];
    static_assert(sizeof(Component) % sizeof(double) == 0, "component record size");
    const double *src = reinterpret_cast<const double *>(comps);
    const int nw = ncomp * (int)(sizeof(Component) / sizeof(double));
    for (int w = threadIdx.x; w < nw; w += blockDim.x) comp_lds[w] = src[w];
    __syncthreads();
    return reinterpret_cast<const Component *>(comp_lds);
}

// FullMolecule::setupSoACache (FullMolecule.cpp:711-767): normalise q (the
// reference mutates the state here, Quaternion.h:40-42), rotate the body-frame
// sites, record molecule position and parameters; positions also relative to
// the molecule's cell corner in FP32.
// forms: bit 0 the FP64 site records (positions, molecule positions,
// orientations, parameters) the FP64 pair kernels and the adjoint read, bit 1
// the FP32 ones of the FP32-pair form. first: the re-bin's build, which also
// normalises q and writes what both forms read (per-cell site starts, molecule
// index of each site, LJ ids, charge head counts); a later call with first = 0 adds a form the
// re-bin did not build, from the same (normalised) q.
__global__ __launch_bounds__(256) void k_build_sites(int n, MolArrays s, Reps R,
                                                     const int *__restrict__ mcell,
                                                     const Component *__restrict__ gcomps,
                                                     int ncomp, int forms, int first,
                                                     int ncell, const int *__restrict__ start,
                                                     SiteArrays s0, SiteArrays s1,
                                                     SiteArrays s2, SiteArrays s3) {
    const Component *comps = stage_comps(gcomps, ncomp);
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (first) {
        // cstart[c] = mstart[start[c]] for c in [0, ncell] (start[ncell]: the
        // live count), for the types that are present
        for (int c = i; c <= ncell; c += gridDim.x * blockDim.x) {
            const int m = start[c];
            if (s0.Fx) s0.cstart[c] = s0.mstart[m];
            if (s1.Fx) s1.cstart[c] = s1.mstart[m];
            if (s2.Fx) s2.cstart[c] = s2.mstart[m];
            if (s3.Fx) s3.cstart[c] = s3.mstart[m];
        }
    }
    if (i >= n) return;
    double q[4] = {s.qw[i], s.qx[i], s.qy[i], s.qz[i]};
    if (first) {
        double qs = 1. / sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
        for (int k = 0; k < 4; ++k) q[k] *= qs;
        s.qw[i] = q[0]; s.qx[i] = q[1]; s.qy[i] = q[2]; s.qz[i] = q[3];
    }
    const bool f64 = forms & 1, f32 = forms & 2;
    const Component &c = comps[s.cid[i]];
    double r[3] = {s.rx[i], s.ry[i], s.rz[i]};
    const int rep = mol_replica(R, i);
    const Geom &g = R.geom[rep];
    int cell = mcell[i] - R.cell_off[rep];
    int cx = cell % g.n[0], cy = (cell / g.n[0]) % g.n[1], cz = cell / (g.n[0] * g.n[1]);
    double corner[3] = {g.bbmin[0] + cx * g.cl[0], g.bbmin[1] + cy * g.cl[1],
                        g.bbmin[2] + cz * g.cl[2]};
    float mrel[3] = {(float)(r[0] - corner[0]), (float)(r[1] - corner[1]),
                     (float)(r[2] - corner[2])};
    SiteArrays *S[4] = {&s0, &s1, &s2, &s3};
#pragma unroll
    for (int t = 0; t < kTypes; ++t) {
        SiteArrays &A = *S[t];
        int base = A.mstart[i];
        for (int k = 0; k < c.n[t]; ++k) {
            int j = base + k;
            double d[3], pos[3];
            qrot(q, c.body[t][k], d);
            for (int a = 0; a < 3; ++a) pos[a] = d[a] + r[a];
            if (first) {
                A.mol[j] = i;
                if (t == T_LJ) A.ljid[j] = c.lj_base + k;
                if (t == T_C) A.nhead[j] = k == 0 ? c.n[T_C] : 0;
            }
            if (f64) {
                A.x[j] = pos[0]; A.y[j] = pos[1]; A.z[j] = pos[2];
                A.mx[j] = r[0]; A.my[j] = r[1]; A.mz[j] = r[2];
                if (t != T_LJ) A.p[j] = c.param[t][k];
            }
            if (f32) {
                A.f[j] = make_float4((float)(pos[0] - corner[0]), (float)(pos[1] - corner[1]),
                                     (float)(pos[2] - corner[2]),
                                     t == T_LJ ? __int_as_float(4 * (c.lj_base + k))
                                               : (float)c.param[t][k]);
                A.fm[j] = make_float4(mrel[0], mrel[1], mrel[2],
                                      __int_as_float(t == T_C && k == 0 ? c.n[T_C] : 0));
            }
            if (t >= T_D) {
                double e[3];
                qrot(q, c.e[t][k], e);
                if (f64) { A.ex[j] = e[0]; A.ey[j] = e[1]; A.ez[j] = e[2]; }
                if (f32) A.fe[j] = make_float4((float)e[0], (float)e[1], (float)e[2], 0.f);
            }
        }
    }
}

// FullMolecule::calcFM (FullMolecule.cpp:548-631): F = sum F_site,
// M = sum d_site x F_site + sum M_site(D, Q), Vi = 0.5 sum V_site (tv: the sum),
// of molecule i.
__device__ __forceinline__ void calc_fm_mol(const MolArrays &s, const Component &c,
                                            const SiteArrays &s0, const SiteArrays &s1,
                                            const SiteArrays &s2, const SiteArrays &s3, int i,
                                            bool virial, double f[3], double M[3], double tv[3]) {
    // point molecules: every site offset is 0, so no d x F term needs q
    double q[4] = {1, 0, 0, 0};
    if (!c.point) q[0] = s.qw[i], q[1] = s.qx[i], q[2] = s.qy[i], q[3] = s.qz[i];
    double m[3] = {0, 0, 0}, tm[3] = {0, 0, 0};
    for (int d = 0; d < 3; ++d) f[d] = tv[d] = 0;
    const SiteArrays *S[4] = {&s0, &s1, &s2, &s3};
#pragma unroll
    for (int t = 0; t < kTypes; ++t) {
        const SiteArrays &A = *S[t];
        int base = A.mstart[i];
        for (int k = 0; k < c.n[t]; ++k) {
            int j = base + k;
            double d[3];
            qrot(q, c.body[t][k], d);
            double fs[3] = {A.Fx[j], A.Fy[j], A.Fz[j]};
            f[0] += fs[0]; f[1] += fs[1]; f[2] += fs[2];
            m[0] += d[1] * fs[2] - d[2] * fs[1];
            m[1] += d[2] * fs[0] - d[0] * fs[2];
            m[2] += d[0] * fs[1] - d[1] * fs[0];
            if (virial) tv[0] += A.Vx[j], tv[1] += A.Vy[j], tv[2] += A.Vz[j];
            if (t >= T_D) {
                tm[0] += A.Mx[j]; tm[1] += A.My[j]; tm[2] += A.Mz[j];
            }
        }
    }
    for (int d = 0; d < 3; ++d) M[d] = m[d] + tm[d];
}

// Molecule i's F, M and Vi into the arrays.
__device__ __forceinline__ void put_fm(const double f[3], const double M[3], const double tv[3],
                                       const Reps &R, const double *__restrict__ lrc, int n, int i,
                                       double *F, double *Mo, double *Vi) {
    for (int d = 0; d < 3; ++d) {
        F[d * n + i] = f[d];
        Mo[d * n + i] = M[d];
        // Homogeneous::calculateLongRange adds VirialCorr / (3N) to every
        // molecule before calcFM adds its sites (Homogeneous.cpp:139-145)
        Vi[d * n + i] =
            lrc ? __dadd_rn(__dmul_rn(0.5, tv[d]), lrc[kThermoW * mol_replica(R, i) + kThVi])
                : 0.5 * tv[d];
    }
}

__global__ __launch_bounds__(256) void k_calc_fm(int n, MolArrays s,
                                                 const Component *__restrict__ gcomps,
                                                 int ncomp, SiteArrays s0, SiteArrays s1,
                                                 SiteArrays s2, SiteArrays s3, double *F,
                                                 double *M, double *Vi, Reps R,
                                                 const double *__restrict__ lrc) {
    const Component *comps = stage_comps(gcomps, ncomp);
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double f[3], m[3], tv[3];
    calc_fm_mol(s, comps[s.cid[i]], s0, s1, s2, s3, i, true, f, m, tv);
    put_fm(f, m, tv, R, lrc, n, i, F, M, Vi);
}

// The second half kick of every molecule with the step's sums. Block b
// covers molecules [chunk[b], chunk[b] + 256) clipped to chunk_end[b]: chunks
// never straddle two replicas. sites: F, M and Vi are first summed from the
// site arrays and stored (k_calc_fm), with no pass of its own.
template <bool SITES>
__global__ __launch_bounds__(256) void k_leapfrog_post(MolArrays s, double *F, double *M,
                                                       double *Vi,
                                                       const Component *__restrict__ gcomps,
                                                       int ncomp, Reps R, double dt, int n,
                                                       const int *__restrict__ chunk,
                                                       const int *__restrict__ chunk_end,
                                                       double *partial, int rmm, int open,
                                                       SiteArrays s0, SiteArrays s1,
                                                       SiteArrays s2, SiteArrays s3,
                                                       const double *__restrict__ lrc) {
    const Component *comps = gcomps;
    if constexpr (SITES) comps = stage_comps(gcomps, ncomp);
    int i = chunk[blockIdx.x] + threadIdx.x;
    const bool in = i < chunk_end[blockIdx.x];
    double mv2 = 0, iw2 = 0, cnt = 0, rot = 0;
    double f[3] = {0., 0., 0.}, m[3] = {0., 0., 0.};
    if constexpr (SITES) {
        if (in) {
            double tv[3];
            calc_fm_mol(s, comps[s.cid[i]], s0, s1, s2, s3, i, true, f, m, tv);
            put_fm(f, m, tv, R, lrc, n, i, F, M, Vi);
        }
    }
    const bool deleted = open && in && s.rx[i] != s.rx[i];
    if (deleted) {
        // deleted at an outflow wall: not moved, not counted
    } else if (rmm && in) {
        // VelocityCellProcessorRMM (VelocityCellProcessorRMM.h:60-110): the
        // kick happened in the force kernel; sum v^2 (no mass factor, as the
        // reference's reduced-memory mode sums it) and N, no rotation
        const double v[3] = {s.vx[i], s.vy[i], s.vz[i]};
        mv2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
        cnt = 1.0;
    } else if (in) {
        const Component &c = comps[s.cid[i]];
        double v[3] = {s.vx[i], s.vy[i], s.vz[i]};
        if constexpr (!SITES) {
            f[0] = F[i], f[1] = F[n + i], f[2] = F[2 * n + i];
            if (!c.point) m[0] = M[i], m[1] = M[n + i], m[2] = M[2 * n + i];
        }
        lf_post_mol(s, m, c, dt, i, v, f, mv2, iw2);
        cnt = 1.0;
        rot = c.rotdof;
        s.vx[i] = v[0]; s.vy[i] = v[1]; s.vz[i] = v[2];
    }
    lf_block_sums(mv2, iw2, cnt, rot, partial);
}

// Step n's second half kick (with its sums) fused with step n + 1's first
// half kick, drift and binning, for consecutive steps without a thermostat
// between them: the same operations in the same order as k_leapfrog_post
// followed by k_leapfrog_pre, with v and F read once. SITES: F and M come from
// the site arrays and stay in registers (nothing reads such a step's F, M and
// Vi). Bound by memory: 1 M molecules of the 2CLJQ + water mixture, calc_fm 76 +
// this 68 + binning 19 us before, 110 with the sites' virials and the molecules'
// F, M and Vi neither read nor written; 1 M one-centre molecules 30 + 20 -> 46.
template <bool SITES>
__global__ __launch_bounds__(256) void k_leapfrog_post_pre(
    MolArrays s, const double *__restrict__ F, const double *__restrict__ M,
    const Component *__restrict__ gcomps, int ncomp, Reps R, double dt, int n,
    const int *__restrict__ chunk, const int *__restrict__ chunk_end, double *partial, Bins bins,
    SiteArrays s0, SiteArrays s1, SiteArrays s2, SiteArrays s3) {
    const Component *comps = gcomps;
    if constexpr (SITES) comps = stage_comps(gcomps, ncomp);
    int i = chunk[blockIdx.x] + threadIdx.x;
    const bool in = i < chunk_end[blockIdx.x];
    double mv2 = 0, iw2 = 0, cnt = 0, rot = 0;
    double r[3] = {0., 0., 0.};
    if (in) {
        const Component &c = comps[s.cid[i]];
        double v[3] = {s.vx[i], s.vy[i], s.vz[i]};
        double f[3], m[3] = {0., 0., 0.};
        if constexpr (SITES) {
            double tv[3];
            calc_fm_mol(s, c, s0, s1, s2, s3, i, false, f, m, tv);
        } else {
            f[0] = F[i], f[1] = F[n + i], f[2] = F[2 * n + i];
            if (!c.point) m[0] = M[i], m[1] = M[n + i], m[2] = M[2 * n + i];
        }
        lf_post_mol(s, m, c, dt, i, v, f, mv2, iw2);
        cnt = 1.0;
        rot = c.rotdof;
        lf_pre_mol(s, m, c, R.geom[mol_replica(R, i)], dt, i, v, f, r);
    }
    bin_mol(r, R, i, in, bins);
    lf_block_sums(mv2, iw2, cnt, rot, partial);
}

// Macroscopic sums of one traversal (VectorizedCellProcessor::endTraversal,
// VectorizedCellProcessor.cpp:122-155). raw = pair-kernel sums over both
// sides of every pair {u6, uXpoles, virial, rf}; halved here. myRF carries
// the reference's negative sign (VectorizedCellProcessor.cpp:2727).
// Step record: Upot, virial, summv2, sumIw2, Upot_LJ, Upot_rest.
__device__ __forceinline__ void finalize_macro(const double raw[4], double *macro, double *rec,
                                               const double *thermo) {
    double u6 = 0.5 * raw[0], ux = 0.5 * raw[1], vir = 0.5 * raw[2], rf = -0.5 * raw[3];
    macro[0] = u6;
    macro[1] = ux;
    macro[2] = vir;
    macro[3] = rf;
    rec[0] = u6 / 6.0 + ux + rf;
    rec[1] = vir + 3.0 * rf;
    if (thermo) {  // Domain::calculateGlobalValues (Domain.cpp:187-188)
        rec[0] = rec[0] + thermo[kThUcorr];
        rec[1] = rec[1] + thermo[kThWcorr];
    }
    rec[4] = u6 / 6.0;
    rec[5] = ux + rf;
}

__device__ __forceinline__ void finalize_lf(const double sums[4], double *rec, double *th,
                                            int heuristics) {
    rec[2] = sums[0];
    rec[3] = sums[1];
    if (!th) return;
    // Domain::calculateGlobalValues, global thermostat, Tfactor 1
    // (Domain.cpp:219-313): temperature and scaling factors; the explosion
    // heuristic replaces them when one is below MIN_BETA = 0.9 (its error
    // counter never rises above 0 in the reference, so it stays armed)
    const double Ti = th[kThTarget];
    const double summv2 = sums[0], N = sums[2], rot = sums[3];
    const double sumIw2 = rot > 0 ? sums[1] : 0.0;
    th[kThT] = N > 0 ? (summv2 + sumIw2) / (3 * N + rot) : Ti;
    double bt = 1.0, br = 1.0;
    if (Ti > 0.0 && N > 0) {
        bt = pow(3.0 * N * Ti / summv2, 0.4);
        br = sumIw2 == 0.0 ? 1.0 : pow(rot * Ti / sumIw2, 0.4);
    }
    double explode = 0.0;
    if ((bt < 0.9 || br < 0.9) && heuristics) {
        explode = 1.0;
        bt = 1.0;
        br = pow(br, 0.0091);
    }
    th[kThBetaT] = bt;
    th[kThBetaR] = br;
    th[kThExplode] = explode;
}

// The explosion capping (Domain.cpp:263-297: a molecule's translational
// kinetic energy above 10 Ti, or rotational above 3 rotDOF Ti, is scaled down,
// v with F and D with M) when the step's heuristic fired, then
// VelocityScalingThermostat::apply for the global thermostat without a
// directed velocity (VelocityScalingThermostat.cpp:70-90): v *= beta_trans,
// D *= beta_rot, for every molecule of a replica with a target temperature.
__global__ __launch_bounds__(256) void k_velocity_scale(MolArrays s, double *F, double *M,
                                                        const Component *__restrict__ comps,
                                                        Reps R, const double *__restrict__ thermo,
                                                        int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double *th = thermo + kThermoW * mol_replica(R, i);
    const double Ti = th[kThTarget];
    if (!(Ti > 0.0)) return;
    const Component &c = comps[s.cid[i]];
    const double bt = th[kThBetaT], br = th[kThBetaR];
    const bool explode = th[kThExplode] != 0.0;
    double v[3] = {s.vx[i], s.vy[i], s.vz[i]};
    // L is rewritten only where it changes: beta_rot is exactly 1 in systems
    // without rotational degrees of freedom, whose L stays in upload order
    bool rot = br != 1.0 || (explode && c.rotdof > 0);
    double L[3] = {0., 0., 0.};
    if (rot) L[0] = s.Lx[i], L[1] = s.Ly[i], L[2] = s.Lz[i];
    if (explode) {
        const double limit = 10.0 * Ti;
        const double ut = 0.5 * c.m * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        if (ut > limit) {
            const double vc = sqrt(limit / ut);
            for (int d = 0; d < 3; ++d) {
                v[d] *= vc;
                F[d * n + i] *= vc;
            }
        }
        if (c.rotdof > 0) {
            const double lr = 3.0 * c.rotdof * Ti;
            const double q[4] = {s.qw[i], s.qx[i], s.qy[i], s.qz[i]};
            double w[3], Iw2 = 0.;
            qrotinv(q, L, w);
            for (int d = 0; d < 3; ++d) {
                w[d] *= c.invI[d];
                Iw2 += c.I[d] * w[d] * w[d];
            }
            const double ur = 0.5 * Iw2;
            if (ur > lr) {
                const double dc = sqrt(lr / ur);
                for (int d = 0; d < 3; ++d) {
                    L[d] *= dc;
                    M[d * n + i] *= dc;
                }
            }
        }
    }
    s.vx[i] = v[0] * bt; s.vy[i] = v[1] * bt; s.vz[i] = v[2] * bt;
    if (rot) {
        s.Lx[i] = L[0] * br; s.Ly[i] = L[1] * br; s.Lz[i] = L[2] * br;
    }
}

// What a step ends with, in one launch: per replica the fixed-order sums of the
// pair kernels' cell rows and of the leapfrog chunks' rows, the step record, the
// thermostat's factors and the step count (before: two reductions of one or two
// launches, two final kernels and the count, 4 to 5 us each; a batch's two
// segmented sums 17 us each; now 4 us for 27 cells, 6 for 2744, 10 for a batch of
// 64 boxes, 15 for 1 M molecules). Replica r's rows go to min(rows / kStepRows,
// kStepBlocks) blocks (its own rows alone decide, so a replica's sums do not
// depend on the batch); a replica of several blocks is finished by the block
// that takes its last ticket, from the block sums in block order. Thread t of a
// block adds rows t, t + 256, ..., the threads' sums go through one tree.
__global__ __launch_bounds__(256) void k_step_end(StepEnd a) {
    const int r = blockIdx.x, t = threadIdx.x;
    const int m0 = a.cell_off[r], m1 = a.cell_off[r + 1];
    const int nb = max(1, min(kStepBlocks, (m1 - m0 + kStepRows - 1) / kStepRows));
    const int b = blockIdx.y;
    if (b >= nb) return;
    double v[8];
    for (int k = 0; k < 8; ++k) v[k] = 0.0;
    auto rows = [&](const double *in, int b0, int b1, double *x) {
        const int per = (b1 - b0 + nb - 1) / nb;
        const int k0 = b0 + b * per, k1 = min(k0 + per, b1);
        for (int k = k0 + t; k < k1; k += 256) {
            const double2 *p = reinterpret_cast<const double2 *>(in) + 2 * (size_t)k;
            const double2 lo = p[0], hi = p[1];
            x[0] += lo.x;
            x[1] += lo.y;
            x[2] += hi.x;
            x[3] += hi.y;
        }
    };
    if ((a.what & kEndMacro) && a.macro_part) {
        if (a.geom[r].small) {
            for (int p = 0; p < kTypes; ++p)
                if (a.present[p]) rows(a.macro_part + 4 * (size_t)p * a.ncell, m0, m1, v);
        } else {
            rows(a.macro_part, m0, m1, v);
        }
    }
    if (a.what & kEndLeapfrog) rows(a.lf_part, a.lf_off[r], a.lf_off[r + 1], v + 4);
    __shared__ double red[8][192];
    if (t >= 64)
        for (int k = 0; k < 8; ++k) red[k][t - 64] = v[k];
    __syncthreads();
    if (t >= 64) return;
    for (int k = 0; k < 8; ++k) v[k] = (v[k] + red[k][t + 64]) + (red[k][t] + red[k][t + 128]);
    auto tree = [&]() {
        for (int k = 0; k < 8; ++k)
            for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_down(v[k], o, 64);
    };
    tree();
    if (nb > 1) {
        double *part = a.part + (size_t)r * kStepBlocks * 8;
        int last = 0;
        if (t == 0) {
            for (int k = 0; k < 8; ++k)
                __hip_atomic_store(&part[b * 8 + k], v[k], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            last = __hip_atomic_fetch_add(&a.ticket[r], 1, __ATOMIC_ACQ_REL,
                                          __HIP_MEMORY_SCOPE_AGENT) == nb - 1;
        }
        if (!__shfl(last, 0, 64)) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        for (int k = 0; k < 8; ++k)
            v[k] = t < nb ? __hip_atomic_load(&part[t * 8 + k], __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT)
                          : 0.0;
        tree();
    }
    if (t > 0) return;
    if (nb > 1) a.ticket[r] = 0;  // (for the next launch: no block is left to take one)
    const int step = a.step_idx[r];
    double *rec = a.step_out + 6 * ((size_t)step * a.nrep + r);
    if (a.what & kEndMacro)
        finalize_macro(v, a.macro + 4 * r, rec, a.lrc ? a.lrc + kThermoW * r : nullptr);
    if (a.what & kEndLeapfrog) {
        for (int k = 0; k < 4; ++k) a.sums[4 * r + k] = v[4 + k];
        finalize_lf(v + 4, rec, a.thermo ? a.thermo + kThermoW * r : nullptr, a.heuristics);
    }
    if (a.what & kEndAdvance) a.step_idx[r] = step + 1;
}

// (the host code lies in another file)
template __global__ void k_leapfrog_post<false>(MolArrays, double *, double *, double *,
                                                const Component *, int, Reps, double, int,
                                                const int *, const int *, double *, int, int,
                                                SiteArrays, SiteArrays, SiteArrays, SiteArrays,
                                                const double *);
template __global__ void k_leapfrog_post<true>(MolArrays, double *, double *, double *,
                                               const Component *, int, Reps, double, int,
                                               const int *, const int *, double *, int, int,
                                               SiteArrays, SiteArrays, SiteArrays, SiteArrays,
                                               const double *);
template __global__ void k_leapfrog_post_pre<false>(MolArrays, const double *, const double *,
                                                    const Component *, int, Reps, double, int,
                                                    const int *, const int *, double *, Bins,
                                                    SiteArrays, SiteArrays, SiteArrays,
                                                    SiteArrays);
template __global__ void k_leapfrog_post_pre<true>(MolArrays, const double *, const double *,
                                                   const Component *, int, Reps, double, int,
                                                   const int *, const int *, double *, Bins,
                                                   SiteArrays, SiteArrays, SiteArrays,
                                                   SiteArrays);

// Download helper: scatter a current-order array back to upload order.
__global__ void k_scatter_orig(int n, const int *__restrict__ orig, const double *__restrict__ a,
                               double *out, int stride_in, int width) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int o = orig[i];
    for (int w = 0; w < width; ++w) out[o * width + w] = a[w * stride_in + i];
}

// A download's arrays (one per blockIdx.y) as the caller's rows, so the host
// only moves bytes: it transposed 16 columns before (1 M molecules: a third of
// 24.7 ms).
__global__ __launch_bounds__(256) void k_pack(PackArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.n) return;
    const PackPart &p = a.p[blockIdx.y];
    const size_t o = p.plain ? i : a.orig[i];
    double *out = a.out + p.off + o * p.width;
    for (int w = 0; w < p.width; ++w) out[w] = p.a[w][i];
}

// An upload's rows into columns.
__global__ __launch_bounds__(256) void k_unpack(UnpackArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.n) return;
    const UnpackPart &p = a.p[blockIdx.y];
    for (int w = 0; w < p.width; ++w)
        p.a[w][i] = p.off >= 0 ? a.in[p.off + (size_t)i * p.width + w] : w == 0 ? p.first : 0.;
    if (blockIdx.y == 0 && a.orig) a.orig[i] = i;
}

__global__ void k_iota(int *a, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = i;
}

}  // namespace mdx
