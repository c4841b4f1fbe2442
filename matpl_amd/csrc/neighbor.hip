// DP neighbor search on gfx950 (the NeighConst.find_neighbore contract,
// src/pre_data/gen_feature/NeighConst.f90:14-149).
//
// Output layout is the reference's, per frame-packed atom i:
//   list  [Ntot][T][m] int32, 1-based neighbor index within the frame, 0 = empty
//   dR    [Ntot][T][m][3] float64 = r_j - r_i (Cartesian)
// plus, for the fused path and MD,
//   counts[Ntot][T] int32 stored neighbors per bucket
//   shift [Ntot][T][m] int32, packed integer image (s1,s2,s3), each +128 in a byte,
//         such that dR = (f_j - f_i + s) . lattice with f the wrapped fractions.
//
// Membership and dR follow the reference bit for bit: positions are wrapped
// with fmod(x+10,1); a frame is "small" when any lattice vector is shorter than
// 2*rc_m, in which case every image in [-nperiod, nperiod]^3 of every atom is
// tested in (j, i1, i2, i3) order; otherwise each fractional difference takes
// the nearest of d, d+1, d-1. dR and |dR|^2 are evaluated in FP64 in the
// reference's operand order with FMA contraction disabled in this file.
// Buckets list neighbors in the reference's order (ascending j, then image).
//
// Two kernels:
//   brute  : one wavefront per atom, j in 64-wide chunks, integer wave scans to
//            place hits; any number of frames (batched training data).
//   cell   : one large frame; atoms binned into a fractional cell grid with a
//            counting sort, each cell's atoms in ascending index. A block owns
//            a cell: it merges the <=27 neighbor cells into one ascending list
//            of candidates in LDS, and each wavefront runs one of the cell's
//            atoms over it, so hits come in list order. Systems of few or sparse
//            cells, and cells too full for that, are searched atom by atom (hits
//            ranked by index).
#include "common.h"

#pragma clang fp contract(off)

namespace matpl {
namespace {

constexpr int WAVE = 64;

struct Lattice {
    double a[9];   // row i = lattice vector i
};

__device__ __forceinline__ int pack_shift(int s1, int s2, int s3) {
    return (s1 + 128) | ((s2 + 128) << 8) | ((s3 + 128) << 16);
}

__device__ __forceinline__ void frac_to_cart(const double *L, double dx1, double dx2, double dx3,
                                             double &dx, double &dy, double &dz) {
    dx = L[0] * dx1 + L[3] * dx2 + L[6] * dx3;
    dy = L[1] * dx1 + L[4] * dx2 + L[7] * dx3;
    dz = L[2] * dx1 + L[5] * dx2 + L[8] * dx3;
}

// Nearest-of {d, d+1, d-1} as NeighConst.f90:98-108; returns the shift taken.
__device__ __forceinline__ int near_image(double &d) {
    int s = 0;
    if (fabs(d + 1.0) < fabs(d)) { d = d + 1.0; s += 1; }
    if (fabs(d - 1.0) < fabs(d)) { d = d - 1.0; s -= 1; }
    return s;
}

__device__ __forceinline__ int wave_incl_scan(int v) {
    const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
        int u = __shfl_up(v, off, WAVE);
        if (lane >= off) v += u;
    }
    return v;
}

// A non-finite coordinate has no cell and no image: status gets STATUS_NONFINITE (before any
// search kernel can record an overflow) and the coordinate is searched as 0, so that every index
// the search forms stays in range.
constexpr int32_t STATUS_NONFINITE = -4;

__global__ void wrap_kernel(const double *__restrict__ frac, double *__restrict__ frac_w, int64_t n3,
                            int32_t *__restrict__ status) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n3;
         i += (int64_t)gridDim.x * blockDim.x) {
        const double x = frac[i];
        if (!isfinite(x)) {
            atomicCAS(status, 0, STATUS_NONFINITE);
            frac_w[i] = 0.0;
        } else {
            frac_w[i] = fmod(x + 10.0, 1.0);
        }
    }
}

// ----------------------------------------------------------------- brute force
// One wavefront per atom. Frame geometry is read from lattice[frame*9].
__global__ void __launch_bounds__(256)
brute_kernel(const double *__restrict__ lattice, const double *__restrict__ fw,
             const int64_t *__restrict__ frame_start, const int32_t *__restrict__ atom_frame,
             const int32_t *__restrict__ type_map, const double *__restrict__ rc_type, int T, int m,
             double rc_m, int64_t ntot, int32_t *__restrict__ list, double *__restrict__ dR,
             int32_t *__restrict__ counts, int32_t *__restrict__ shift, int32_t *__restrict__ status) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t i = blockIdx.x * (int64_t)(blockDim.x / WAVE) + (threadIdx.x / WAVE);
    if (i >= ntot) return;
    const int f = atom_frame[i];
    const int64_t j0 = frame_start[f], j1 = frame_start[f + 1];
    const double *L = lattice + 9 * (int64_t)f;
    int np[3];
    bool small_box = false;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double len = sqrt(L[3 * d] * L[3 * d] + L[3 * d + 1] * L[3 * d + 1] + L[3 * d + 2] * L[3 * d + 2]);
        np[d] = (int)(rc_m / len) + 1;
        if (len < 2.0 * rc_m) small_box = true;
    }
    if (!small_box) np[0] = np[1] = np[2] = 0;
    const double rc2 = rc_m * rc_m;
    const double rci = rc_type[type_map[i]];
    const double rci2 = rci * rci;
    const double fi0 = fw[3 * i], fi1 = fw[3 * i + 1], fi2 = fw[3 * i + 2];
    const int64_t S = (int64_t)T * m;
    int32_t *li = list + i * S;
    double *di = dR ? dR + i * S * 3 : nullptr;
    int32_t *si = shift ? shift + i * S : nullptr;

    // running stored / counted (rc_m) totals per type; T <= 16
    int base[16], baseM[16];
    for (int t = 0; t < T; t++) base[t] = baseM[t] = 0;
    bool overflow = false;

    for (int64_t jc = j0; jc < j1; jc += WAVE) {
        const int64_t j = jc + lane;
        const bool valid = j < j1;
        const int tj = valid ? type_map[j] : 0;
        double fj0 = 0, fj1 = 0, fj2 = 0;
        if (valid) { fj0 = fw[3 * j]; fj1 = fw[3 * j + 1]; fj2 = fw[3 * j + 2]; }
        // pass 1: counts for this lane's j
        int c = 0, cM = 0;
        if (valid) {
            for (int i1 = -np[0]; i1 <= np[0]; i1++)
            for (int i2 = -np[1]; i2 <= np[1]; i2++)
            for (int i3 = -np[2]; i3 <= np[2]; i3++) {
                double dx1 = fj0 - fi0, dx2 = fj1 - fi1, dx3 = fj2 - fi2;
                if (small_box) { dx1 = dx1 + (double)i1; dx2 = dx2 + (double)i2; dx3 = dx3 + (double)i3; }
                else { near_image(dx1); near_image(dx2); near_image(dx3); }
                double dx, dy, dz;
                frac_to_cart(L, dx1, dx2, dx3, dx, dy, dz);
                const double dd = dx * dx + dy * dy + dz * dz;
                if (dd < rc2 && dd > 1e-8) {
                    cM++;
                    if (dd < rci2) c++;
                }
            }
        }
        // place this chunk's hits after the running totals, type by type
        int off = 0;
        for (int t = 0; t < T; t++) {
            const int v = (tj == t && valid) ? c : 0;
            const int vM = (tj == t && valid) ? cM : 0;
            const int incl = wave_incl_scan(v);
            const int inclM = wave_incl_scan(vM);
            const int tot = __shfl(incl, WAVE - 1, WAVE);
            const int totM = __shfl(inclM, WAVE - 1, WAVE);
            if (tj == t) off = base[t] + incl - v;
            base[t] += tot;
            baseM[t] += totM;
            if (baseM[t] > m) overflow = true;
        }
        if (overflow) break;
        // pass 2: write this lane's hits in image order
        if (valid && c > 0) {
            int k = off;
            for (int i1 = -np[0]; i1 <= np[0]; i1++)
            for (int i2 = -np[1]; i2 <= np[1]; i2++)
            for (int i3 = -np[2]; i3 <= np[2]; i3++) {
                double dx1 = fj0 - fi0, dx2 = fj1 - fi1, dx3 = fj2 - fi2;
                int s1 = i1, s2 = i2, s3 = i3;
                if (small_box) { dx1 = dx1 + (double)i1; dx2 = dx2 + (double)i2; dx3 = dx3 + (double)i3; }
                else { s1 = near_image(dx1); s2 = near_image(dx2); s3 = near_image(dx3); }
                double dx, dy, dz;
                frac_to_cart(L, dx1, dx2, dx3, dx, dy, dz);
                const double dd = dx * dx + dy * dy + dz * dz;
                if (dd < rc2 && dd > 1e-8 && dd < rci2) {
                    const int64_t slot = (int64_t)tj * m + k;
                    li[slot] = (int32_t)(j - j0) + 1;
                    if (di) { di[3 * slot] = dx; di[3 * slot + 1] = dy; di[3 * slot + 2] = dz; }
                    if (si) si[slot] = pack_shift(s1, s2, s3);
                    k++;
                }
            }
        }
    }
    if (overflow) {
        if (lane == 0) atomicCAS(status, 0, (int)(i + 1));
        for (int t = 0; t < T; t++) base[t] = 0;
    }
    // zero the unused tail of every bucket
    for (int t = 0; t < T; t++) {
        for (int k = base[t] + lane; k < m; k += WAVE) {
            const int64_t slot = (int64_t)t * m + k;
            li[slot] = 0;
            if (di) { di[3 * slot] = 0.0; di[3 * slot + 1] = 0.0; di[3 * slot + 2] = 0.0; }
            if (si) si[slot] = pack_shift(0, 0, 0);
        }
        if (counts && lane == 0) counts[i * T + t] = base[t];
    }
}

// ------------------------------------------------------------------ cell list
struct Grid {
    int nc[3];
    int noff[3];       // number of distinct offsets per dim (1..3)
    int off[3][3];     // distinct offsets per dim
};

// A wrapped coordinate in [0, 1): fmod leaves one below -10 negative.
__device__ __forceinline__ double cell_frac(double f) { return f < 0.0 ? f + 1.0 : f; }

__device__ __forceinline__ int cell_of(double f, int nc) {
    const int v = (int)(cell_frac(f) * nc);
    return v < 0 ? 0 : (v >= nc ? nc - 1 : v);
}

__global__ void bin_kernel(const double *__restrict__ fw, int64_t n, Grid g, int32_t *__restrict__ atom_cell,
                           int32_t *__restrict__ cell_count) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        int c[3];
#pragma unroll
        for (int d = 0; d < 3; d++) c[d] = cell_of(fw[3 * i + d], g.nc[d]);
        const int cell = (c[0] * g.nc[1] + c[1]) * g.nc[2] + c[2];
        atom_cell[i] = cell;
        atomicAdd(cell_count + cell, 1);
    }
}

// Exclusive scan of cell_count into cell_start (ncells+1 entries), one block.
__global__ void __launch_bounds__(1024) scan_kernel(const int32_t *__restrict__ cnt, int32_t *__restrict__ start,
                                                    int32_t *__restrict__ cursor, int ncells) {
    __shared__ int32_t part[1024 / WAVE];
    __shared__ int32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    for (int base = 0; base < ncells; base += 1024) {
        const int idx = base + threadIdx.x;
        const int v = idx < ncells ? cnt[idx] : 0;
        const int incl = wave_incl_scan(v);
        if (lane == WAVE - 1) part[wid] = incl;
        __syncthreads();
        int wofs = 0;
        for (int w = 0; w < wid; w++) wofs += part[w];
        const int excl = carry + wofs + incl - v;
        if (idx < ncells) { start[idx] = excl; cursor[idx] = excl; }
        __syncthreads();
        if (threadIdx.x == 1023) carry = excl + v;
        __syncthreads();
    }
    if (threadIdx.x == 0) start[ncells] = carry;
}

__global__ void fill_cells_kernel(const int32_t *__restrict__ atom_cell, int64_t n, int32_t *__restrict__ cursor,
                                  int32_t *__restrict__ cell_atoms) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        cell_atoms[atomicAdd(cursor + atom_cell[i], 1)] = (int32_t)i;
}

// The atoms of each cell and its two neighbors along z (a grid of three or more), in ascending order.
// A cell's list starts where the counts of those before it end: whole columns give three times their
// atoms, and within a column the sums of the cells' counts shifted by -1, 0 and 1 telescope.
struct ZRun { int64_t at; int count; };      // in the sorted array

__device__ __forceinline__ ZRun z_run(const int32_t *__restrict__ cell_start, const Grid &g, int cell) {
    const int nz = g.nc[2], z = cell % nz, c0 = cell - z;
    const int s0 = cell_start[c0];
    auto upto = [&](int x) { return cell_start[c0 + x] - s0; };      // atoms of cells z < x
    auto count = [&](int x) { return cell_start[c0 + x + 1] - cell_start[c0 + x]; };
    const int below = z > 0 ? z - 1 : nz - 1, above = z + 1 < nz ? z + 1 : 0;
    const int64_t at = z == 0 ? 0 : (int64_t)upto(z - 1) + count(nz - 1) + upto(z) + upto(z + 1) - upto(1);
    return {3 * (int64_t)s0 + at, count(below) + count(z) + count(above)};
}

// One wavefront per cell; the rank of an atom is the number of smaller ones. A run longer than
// `longest` is left out (the ranking takes its square): a block that would need it leaves its atoms
// to cell_overfull_kernel.
constexpr int SORT_WAVES = 4;
__global__ void __launch_bounds__(SORT_WAVES * WAVE)
sort_runs_kernel(const int32_t *__restrict__ cell_start, int ncells, Grid g, int longest,
                 const int32_t *__restrict__ cell_atoms, int32_t *__restrict__ sorted) {
    const int lane = threadIdx.x & (WAVE - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    for (int c = blockIdx.x * SORT_WAVES + wid; c < ncells; c += gridDim.x * SORT_WAVES) {
        const ZRun run = z_run(cell_start, g, c);
        if (run.count > longest) continue;
        const int nz = g.nc[2], z = c % nz, c0 = c - z;
        // the run's atoms are those of [s0, s1) and, where the period splits it, of [s2, ..)
        int s0, s1, s2 = 0;
        if (nz == 3) { s0 = cell_start[c0]; s1 = cell_start[c0 + 3]; }
        else if (z == 0) { s0 = cell_start[c0]; s1 = cell_start[c0 + 2]; s2 = cell_start[c0 + nz - 1]; }
        else if (z == nz - 1) { s0 = cell_start[c0 + z - 1]; s1 = cell_start[c0 + nz]; s2 = cell_start[c0]; }
        else { s0 = cell_start[c0 + z - 1]; s1 = cell_start[c0 + z + 2]; }
        const int n0 = s1 - s0;
        auto atom = [&](int e) { return e < run.count ? cell_atoms[e < n0 ? s0 + e : s2 + e - n0] : 0x7fffffff; };
        for (int e0 = 0; e0 < run.count; e0 += WAVE) {
            const int j = atom(e0 + lane);
            int rank = 0;
            for (int q0 = 0; q0 < run.count; q0 += WAVE) {
                const int other = atom(q0 + lane);
                const int nq = run.count - q0 < WAVE ? run.count - q0 : WAVE;
                for (int q = 0; q < nq; q++) rank += __builtin_amdgcn_readlane(other, q) < j;
            }
            if (e0 + lane < run.count) sorted[run.at + rank] = j;
        }
    }
}

struct CellArgs {
    Lattice lat;
    Grid g;
    const double *fw;
    const int32_t *atom_cell, *cell_start, *cell_atoms, *type_map;
    const double *rc_type;
    int T, m;
    double rc_m;
    int64_t n;
    int32_t *list;
    double *dR;
    int32_t *counts, *shift, *status;
    // cell_block_kernel only
    const int32_t *sorted;      // ascending runs along z
    double pitch[3];            // of the cells, in fractions
    int32_t *overfull;          // [0] their number, then the atoms of cells with too many candidates
    float pre2;                 // squared radius of the FP32 preselection
    int cap, ncells, nparts;    // candidates in LDS, cells, blocks per cell
};

// The neighbors of atom i found by one wavefront alone, from the cells around it: hits go to
// per-type LDS buckets ([T][m], then [T] stored and [T] counted at rc_m) and are ranked by index.
__device__ void cell_scan_atom(const CellArgs &A, int64_t i, int32_t *bucket) {
    const int lane = threadIdx.x & (WAVE - 1);
    const Grid &g = A.g;
    const double *__restrict__ fw = A.fw;
    const int T = A.T, m = A.m;
    int32_t *cnt = bucket + T * m;                    // [T] stored
    int32_t *cntM = cnt + T;                          // [T] counted at rc_m
    for (int t = lane; t < 2 * T; t += WAVE) cnt[t] = 0;
    wave_sync();
    const double *L = A.lat.a;
    const double rc2 = A.rc_m * A.rc_m;
    const double fi0 = fw[3 * i], fi1 = fw[3 * i + 1], fi2 = fw[3 * i + 2];
    const double rci = A.rc_type[A.type_map[i]];
    const double rci2 = rci * rci;
    int c = A.atom_cell[i];
    int ci[3];
    ci[2] = c % g.nc[2]; c /= g.nc[2];
    ci[1] = c % g.nc[1]; ci[0] = c / g.nc[1];
    // The z cells of one (x, y) column are contiguous in cell_atoms, so the column's 1-3 z
    // offsets become at most two runs of consecutive cells (the periodic wrap splits one), and
    // the lanes sweep each run in one pass rather than cell by cell (about 90 candidates per
    // run against about 30 per cell: fewer, fuller passes of the FP64 distance test).
    int zr0[3], zr1[3], nzr = 0;
    {
        int zs[3];
        const int nzo = g.noff[2];
        for (int c = 0; c < nzo; c++) zs[c] = (ci[2] + g.off[2][c] + g.nc[2]) % g.nc[2];
        for (int x = 1; x < nzo; x++)
            for (int y = x; y > 0 && zs[y - 1] > zs[y]; y--) {
                const int tmp = zs[y]; zs[y] = zs[y - 1]; zs[y - 1] = tmp;
            }
        for (int c = 0; c < nzo; c++) {
            if (nzr > 0 && zs[c] == zr1[nzr - 1] + 1) zr1[nzr - 1] = zs[c];
            else { zr0[nzr] = zs[c]; zr1[nzr] = zs[c]; nzr++; }
        }
    }
    for (int a = 0; a < g.noff[0]; a++)
    for (int b = 0; b < g.noff[1]; b++)
    for (int c = 0; c < nzr; c++) {
        const int cx = (ci[0] + g.off[0][a] + g.nc[0]) % g.nc[0];
        const int cy = (ci[1] + g.off[1][b] + g.nc[1]) % g.nc[1];
        const int col = (cx * g.nc[1] + cy) * g.nc[2];
        const int s0 = A.cell_start[col + zr0[c]], s1 = A.cell_start[col + zr1[c] + 1];
        // two candidates per lane per pass, both passes' loads issued before either is used
        for (int p0 = s0; p0 < s1; p0 += 2 * WAVE) {
            int jj[2];
            double fj[2][3];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int p = p0 + u * WAVE + lane;
                jj[u] = p < s1 ? A.cell_atoms[p] : -1;
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int j = jj[u] < 0 ? 0 : jj[u];
                fj[u][0] = fw[3 * j]; fj[u][1] = fw[3 * j + 1]; fj[u][2] = fw[3 * j + 2];
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int j = jj[u];
                if (j < 0) continue;
                double dx1 = fj[u][0] - fi0, dx2 = fj[u][1] - fi1, dx3 = fj[u][2] - fi2;
                near_image(dx1); near_image(dx2); near_image(dx3);
                double dx, dy, dz;
                frac_to_cart(L, dx1, dx2, dx3, dx, dy, dz);
                const double dd = dx * dx + dy * dy + dz * dz;
                if (dd < rc2 && dd > 1e-8) {
                    const int tj = A.type_map[j];
                    atomicAdd(cntM + tj, 1);
                    if (dd < rci2) {
                        const int k = atomicAdd(cnt + tj, 1);
                        if (k < m) bucket[tj * m + k] = j;
                    }
                }
            }
        }
    }
    wave_sync();
    bool overflow = false;
    for (int t = 0; t < T; t++) overflow |= cntM[t] > m;
    if (overflow) {
        if (lane == 0) atomicCAS(A.status, 0, (int)(i + 1));
        wave_sync();
        for (int t = lane; t < T; t += WAVE) cnt[t] = 0;
        wave_sync();
    }
    const int64_t S = (int64_t)T * m;
    int32_t *li = A.list + i * S;
    double *di = A.dR ? A.dR + i * S * 3 : nullptr;
    int32_t *si = A.shift ? A.shift + i * S : nullptr;
    for (int t = 0; t < T; t++) {
        const int nt = cnt[t];
        const int32_t *bk = bucket + t * m;
        for (int e = lane; e < nt; e += WAVE) {
            const int j = bk[e];
            int rank = 0;
            for (int q = 0; q < nt; q++) rank += bk[q] < j;
            double dx1 = fw[3 * j] - fi0, dx2 = fw[3 * j + 1] - fi1, dx3 = fw[3 * j + 2] - fi2;
            const int s1 = near_image(dx1), s2 = near_image(dx2), s3 = near_image(dx3);
            const int64_t slot = (int64_t)t * m + rank;
            li[slot] = j + 1;
            if (di) {
                double dx, dy, dz;
                frac_to_cart(L, dx1, dx2, dx3, dx, dy, dz);
                di[3 * slot] = dx; di[3 * slot + 1] = dy; di[3 * slot + 2] = dz;
            }
            if (si) si[slot] = pack_shift(s1, s2, s3);
        }
        for (int k = nt + lane; k < m; k += WAVE) {
            const int64_t slot = (int64_t)t * m + k;
            li[slot] = 0;
            if (di) { di[3 * slot] = 0.0; di[3 * slot + 1] = 0.0; di[3 * slot + 2] = 0.0; }
            if (si) si[slot] = pack_shift(0, 0, 0);
        }
        if (A.counts && lane == 0) A.counts[i * T + t] = nt;
    }
    wave_sync();                                      // the next atom reuses the buckets
}

constexpr int CELL_WAVES = 4;   // wavefronts (atoms) per block

__global__ void __launch_bounds__(CELL_WAVES * WAVE) cell_kernel(CellArgs A) {
    extern __shared__ int32_t smem[];
    // wid is the same on every lane: the atom, its cell and the cells' ranges stay scalar
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int64_t i = blockIdx.x * (int64_t)CELL_WAVES + wid;
    if (i < A.n) cell_scan_atom(A, i, smem + wid * (A.T * A.m + 2 * A.T));
}

// The atoms that cell_block_kernel left, a wavefront each: as many wavefronts as it has work for, whether
// they come from a few crowded cells or from many.
__global__ void __launch_bounds__(CELL_WAVES * WAVE) cell_overfull_kernel(CellArgs A) {
    extern __shared__ int32_t smem[];
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    int32_t *bucket = smem + wid * (A.T * A.m + 2 * A.T);
    const int left = A.overfull[0];
    for (int x = blockIdx.x * CELL_WAVES + wid; x < left; x += gridDim.x * CELL_WAVES)
        cell_scan_atom(A, A.overfull[1 + x], bucket);
}

// One block per cell (or per part of a cell's atoms), on a grid of three or more cells in every
// direction. All atoms of a cell have the same candidates, the atoms of the 27 cells around it, so
// the block puts these in ascending order once: the nine runs along z are sorted already, and two
// rounds of merging (along y, then x; an atom's place is its own rank plus its lower bounds in the
// two sibling runs) leave one list. With it go FP32 Cartesian positions relative to the cell, so that a wavefront rejects 64
// candidates with one 16-byte LDS read and seven FP32 operations; the survivors (about one in
// seven) are queued, and 64 at a time take the exact FP64 test with all lanes busy and are stored
// in list order by ballots: no ranking and no atomics.
//
// The preselection keeps every pair that the exact test can accept: with three or more cells in
// every direction the image that a cell pair implies is the only one within rc. It is cut at
// A.pre2, which covers the rounding of FP32 positions.
//
// Four atoms of a wavefront go over the candidates together, so that an LDS read serves four
// tests (one atom a pass: 240 us; LDS reads were then the bound), and the queue holds places in the
// list, not indices. 80 VGPRs (six wavefronts a SIMD): at 64 the compiler kept the four atoms'
// positions in scalar registers and spilled (201 us).
//
// Bound: VALU issue (about 740 instructions an atom: 135 of the sweep over 807 candidates, 240 of
// the exact tests, 160 of its share of the merging). 178 us, against 496 us of the search atom by
// atom, on the 99,636-atom HfO2 list of 160 slots per type at 6.5 A (105 neighbors an atom, 255 MB
// of list and shift stores).
constexpr int CB_WAVES = 8;
constexpr int CB_ATOMS = 4;     // atoms of a wavefront per pass over the candidates
constexpr int CB_QUEUE = 2 * WAVE;
constexpr int CB_MIN_ATOMS = 6;     // atoms per cell, and atoms, from which on this is the faster search
constexpr int CB_MIN_TOTAL = 5000;
constexpr int CB_MIN_BLOCKS = 512;
constexpr int CB_MAX_CAND = 4096;   // candidates of a block, at most
constexpr int CB_RUN_SHARE = 4;     // of its nine runs, each at most this part (a ninth where the density is even)

__device__ __forceinline__ int lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

__global__ void __launch_bounds__(CB_WAVES * WAVE, 6)
cell_block_kernel(CellArgs A) {
    extern __shared__ __align__(16) int32_t smem[];
    __shared__ int run_start[10];
    __shared__ int64_t run_src[9];
    // blocks go round-robin to the 8 XCDs: give each one a contiguous range of cells
    const int nwork = A.ncells * A.nparts, per = (nwork + 7) >> 3;
    const int work = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || work >= nwork) return;
    const int cell = work / A.nparts, part = work - cell * A.nparts;
    const int lane = threadIdx.x & (WAVE - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int own0 = A.cell_start[cell], nown = A.cell_start[cell + 1] - own0;
    if (part * CB_WAVES >= nown) return;
    const Grid &g = A.g;
    const double *__restrict__ fw = A.fw;
    int ci[3];
    {
        int c = cell;
        ci[2] = c % g.nc[2]; c /= g.nc[2];
        ci[1] = c % g.nc[1]; ci[0] = c / g.nc[1];
    }
    if (wid == 0) {
        int64_t src = 0;
        int cnt = 0;
        if (lane < 9) {
            const int cx = (ci[0] + lane / 3 - 1 + g.nc[0]) % g.nc[0];
            const int cy = (ci[1] + lane % 3 - 1 + g.nc[1]) % g.nc[1];
            const ZRun run = z_run(A.cell_start, g, (cx * g.nc[1] + cy) * g.nc[2] + ci[2]);
            src = run.at;
            cnt = run.count;
        }
        const int incl = wave_incl_scan(cnt);
        const bool crowded = __any(cnt > A.cap / CB_RUN_SHARE);
        if (lane < 9) { run_start[lane + 1] = lane == 8 && crowded ? A.cap + 1 : incl; run_src[lane] = src - (incl - cnt); }
        if (lane == 0) run_start[0] = 0;
    }
    __syncthreads();
    const int total = run_start[9];
    if (total > A.cap) {        // cell_overfull_kernel searches this cell's atoms
        if (part == 0) {
            __shared__ int at;
            if (threadIdx.x == 0) at = atomicAdd(A.overfull, nown);
            __syncthreads();
            for (int e = threadIdx.x; e < nown; e += CB_WAVES * WAVE) A.overfull[1 + at + e] = A.cell_atoms[own0 + e];
        }
        return;
    }
    uint32_t *keyA = reinterpret_cast<uint32_t *>(smem);             // [cap], later the wavefronts' queues
    float4 *pos = reinterpret_cast<float4 *>(smem + A.cap);          // [cap] (x, y, z, index)
    uint32_t *keyB = reinterpret_cast<uint32_t *>(pos);              // [cap], before the positions
    auto run_of = [&](int idx, int stride, int nr) {                 // last run that starts at or before idx
        int lo = 0;
        for (int r = 1; r < nr; r++) lo += run_start[r * stride] <= idx;
        return lo;
    };
    for (int idx = threadIdx.x; idx < total; idx += CB_WAVES * WAVE)
        keyA[idx] = (uint32_t)A.sorted[run_src[run_of(idx, 1, 9)] + idx];
    __syncthreads();
#pragma unroll
    for (int round = 0; round < 2; round++) {       // along y (nine runs), then x (three)
        const uint32_t *in = round ? keyB : keyA;
        uint32_t *out = round ? keyA : keyB;
        const int stride = round ? 3 : 1, nr = round ? 3 : 9;
        int longest = 0;
        for (int r = 0; r < nr; r++) {
            const int len = run_start[(r + 1) * stride] - run_start[r * stride];
            longest = len > longest ? len : longest;
        }
        const int top = longest > 0 ? 1 << (31 - __clz(longest)) : 0;
        for (int idx = threadIdx.x; idx < total; idx += CB_WAVES * WAVE) {
            const uint32_t k = in[idx];
            const int r = run_of(idx, stride, nr);
            const int r0 = (r / 3) * 3;
            const int at = run_start[r0 * stride] + idx - run_start[r * stride];
            // the sibling runs r1, r2
            const int r1 = r + 1 < r0 + 3 ? r + 1 : r0, r2 = r + 2 < r0 + 3 ? r + 2 : r - 1;
            const int lo1 = run_start[r1 * stride], lo2 = run_start[r2 * stride];
            const int hi1 = run_start[(r1 + 1) * stride], hi2 = run_start[(r2 + 1) * stride];
            // both lower bounds bit by bit; reads beyond a run (at most 2 * cap words in) are not used
            int b1 = lo1, b2 = lo2;
            for (int step = top; step > 0; step >>= 1) {
                const uint32_t k1 = in[b1 + step - 1], k2 = in[b2 + step - 1];
                b1 = b1 + step <= hi1 && k1 < k ? b1 + step : b1;
                b2 = b2 + step <= hi2 && k2 < k ? b2 + step : b2;
            }
            out[at + (b1 - lo1) + (b2 - lo2)] = k;
        }
        __syncthreads();
    }
    // FP32 positions relative to the cell's corner, the image taken from the cells' distance
    const double *L = A.lat.a;
    const double corner[3] = {ci[0] * A.pitch[0], ci[1] * A.pitch[1], ci[2] * A.pitch[2]};
    auto rel = [&](double f0, double f1, double f2, float o[3]) {
        const double f[3] = {f0, f1, f2};
        double u[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int dc = cell_of(f[d], g.nc[d]) - ci[d];
            const double s = dc > 1 ? -1.0 : (dc < -1 ? 1.0 : 0.0);
            u[d] = (cell_frac(f[d]) + s) - corner[d];
        }
        double x, y, z;
        frac_to_cart(L, u[0], u[1], u[2], x, y, z);
        o[0] = (float)x; o[1] = (float)y; o[2] = (float)z;
    };
    const int padded = (total + WAVE - 1) & ~(WAVE - 1);             // to whole wavefronts with points at infinity
    for (int idx = threadIdx.x; idx < padded; idx += CB_WAVES * WAVE) {
        float o[3] = {INFINITY, INFINITY, INFINITY};
        int64_t j = 0;
        if (idx < total) {
            j = keyA[idx];
            rel(fw[3 * j], fw[3 * j + 1], fw[3 * j + 2], o);
        }
        pos[idx] = make_float4(o[0], o[1], o[2], __int_as_float((int)j));
    }
    __syncthreads();
    const int T = A.T, m = A.m;
    const double rc2 = A.rc_m * A.rc_m;
    const int64_t S = (int64_t)T * m;
    // [CB_ATOMS][CB_QUEUE] candidates (places in pos) of each atom of the wavefront, over keyA, which is spent
    uint16_t *queue = reinterpret_cast<uint16_t *>(smem) + wid * (CB_ATOMS * CB_QUEUE);
    const float pre2 = A.pre2;
    const int first = part * CB_WAVES + wid, step = CB_WAVES * A.nparts;
    for (int a0 = first; a0 < nown; a0 += step * CB_ATOMS) {
        // lane 16 u + t serves the wavefront's u-th atom of this pass; its type-t entries stored and counted
        const int mine = a0 + (lane >> 4) * step;
        const int64_t my_atom = A.cell_atoms[own0 + (mine < nown ? mine : a0)];
        const double my_f[3] = {fw[3 * my_atom], fw[3 * my_atom + 1], fw[3 * my_atom + 2]};
        float my_pos[3];
        rel(my_f[0], my_f[1], my_f[2], my_pos);
        const double my_rc = A.rc_type[A.type_map[my_atom]];
        const double my_rc2 = my_rc * my_rc;
        int stored = 0, counted = 0;
        float px[CB_ATOMS], py[CB_ATOMS], pz[CB_ATOMS];
        int qn[CB_ATOMS];
#pragma unroll
        for (int u = 0; u < CB_ATOMS; u++) {
            // one that is not there is at infinity: nothing is taken for it
            px[u] = __shfl(mine < nown ? my_pos[0] : INFINITY, 16 * u, WAVE);
            py[u] = __shfl(my_pos[1], 16 * u, WAVE);
            pz[u] = __shfl(my_pos[2], 16 * u, WAVE);
            qn[u] = 0;
        }
        for (int s0 = 0; s0 < padded; s0 += WAVE) {
            const float4 c = pos[s0 + lane];
            bool full = false;
#pragma unroll
            for (int u = 0; u < CB_ATOMS; u++) {
                const float dx = c.x - px[u], dy = c.y - py[u], dz = c.z - pz[u];
                const bool take = fmaf(dx, dx, fmaf(dy, dy, dz * dz)) < pre2;
                const unsigned long long mask = __ballot(take);
                if (take) queue[u * CB_QUEUE + qn[u] + lanes_below(mask)] = (uint16_t)(s0 + lane);
                qn[u] += __popcll(mask);
                full |= qn[u] >= WAVE;
            }
            const bool last = s0 + WAVE >= padded;
            if (!full && !last) continue;
            // the exact test on 64 queued candidates at a time, on what is left after the last ones
            wave_sync();
#pragma unroll 1
            for (int u = 0; u < CB_ATOMS; u++) {
                int left = u == 0 ? qn[0] : u == 1 ? qn[1] : u == 2 ? qn[2] : qn[3];
                while (left >= (last ? 1 : WAVE)) {
                    const int64_t i = __builtin_amdgcn_readlane((int)my_atom, 16 * u);
                    const int q = queue[u * CB_QUEUE + lane], rest = queue[u * CB_QUEUE + WAVE + lane];
                    const bool live = lane < left;
                    const int64_t j = live ? __float_as_int(pos[q].w) : i;
                    const int tj = A.type_map[j];
                    double dx1 = fw[3 * j] - lane_value(my_f[0], 16 * u), dx2 = fw[3 * j + 1] - lane_value(my_f[1], 16 * u),
                           dx3 = fw[3 * j + 2] - lane_value(my_f[2], 16 * u);
                    const int s1 = near_image(dx1), s2 = near_image(dx2), s3 = near_image(dx3);
                    double dx, dy, dz;
                    frac_to_cart(L, dx1, dx2, dx3, dx, dy, dz);
                    const double dd = dx * dx + dy * dy + dz * dz;
                    const bool inM = live && dd < rc2 && dd > 1e-8;
                    const bool in = inM && dd < lane_value(my_rc2, 16 * u);
                    int k = 0;
                    for (int t = 0; t < T; t++) {
                        const unsigned long long mk = __ballot(in && tj == t), mkM = __ballot(inM && tj == t);
                        const int b = __builtin_amdgcn_readlane(stored, 16 * u + t);
                        if (tj == t) k = b + lanes_below(mk);
                        if (lane == 16 * u + t) { stored += __popcll(mk); counted += __popcll(mkM); }
                    }
                    if (in && k < m) {
                        const int64_t slot = i * S + (int64_t)tj * m + k;
                        A.list[slot] = (int32_t)j + 1;
                        if (A.dR) { A.dR[3 * slot] = dx; A.dR[3 * slot + 1] = dy; A.dR[3 * slot + 2] = dz; }
                        if (A.shift) A.shift[slot] = pack_shift(s1, s2, s3);
                    }
                    left -= left < WAVE ? left : WAVE;
                    wave_sync();
                    if (lane < left) queue[u * CB_QUEUE + lane] = (uint16_t)rest;
                    wave_sync();
                }
#pragma unroll
                for (int v = 0; v < CB_ATOMS; v++)
                    if (v == u) qn[v] = left;
            }
        }
#pragma unroll 1
        for (int u = 0; u < CB_ATOMS && a0 + u * step < nown; u++) {
            const int64_t i = __builtin_amdgcn_readlane((int)my_atom, 16 * u);
            if (__any((lane >> 4) == u && counted > m)) {
                if (lane == 0) atomicCAS(A.status, 0, (int)(i + 1));
                if ((lane >> 4) == u) stored = 0;
                __threadfence();            // the zeros below go over entries already stored
            }
            for (int t = 0; t < T; t++) {
                const int nt = __builtin_amdgcn_readlane(stored, 16 * u + t);
                for (int k = nt + lane; k < m; k += WAVE) {
                    const int64_t slot = i * S + (int64_t)t * m + k;
                    A.list[slot] = 0;
                    if (A.dR) { A.dR[3 * slot] = 0.0; A.dR[3 * slot + 1] = 0.0; A.dR[3 * slot + 2] = 0.0; }
                    if (A.shift) A.shift[slot] = pack_shift(0, 0, 0);
                }
            }
            if (A.counts && (lane >> 4) == u && (lane & 15) < T) A.counts[i * T + (lane & 15)] = stored;
        }
    }
}

// Reverse slot of every used bucket entry: for s = (i, t, k) naming
// neighbor j with image shift sh, rev[s] is the entry of j's bucket of type
// t_i that names i with image -sh. The list is symmetric because dR_ji is the
// exact negation of dR_ij in the cutoff test; a missing partner (per-type
// cutoffs that differ, or a tie in the nearest-image rule) sets status.
//
// Every entry searches its partner's bucket (sorted by (j, image)) by itself, four entries to a load. The loads
// touch a different cache line per lane, so what bounds the kernel is their number and where they hit. The
// 8 XCDs take contiguous ranges of atoms: where neighbors in space are near in index, the buckets of a range's
// neighbors share its L2, and bisecting the bucket is cheapest. Where the atoms are in no spatial order
// (scattered_order) every line comes from beyond the L2s; but then the entries of a bucket are spread evenly,
// so that the partner's place follows from its index, and the search starts there: one line, not two or three.
// 99,636 HfO2 atoms (160 slots per type, 105 neighbors an atom) 218 us, shuffled 510 (bisected 651);
// 40,000 atoms of 255 neighbors in random order 367 (675), 30,000 of 104 112 (151). A kernel in which one atom
// of each pair searches and stores both directions, between passes that set all slots to -1 and look for
// those left, takes 307, 479, 422 and 114 us.
constexpr int REV_WAVES = 4;
constexpr int REV_XCDS = 8;

struct __attribute__((packed, aligned(4))) Int4 { int32_t v[4]; };

// The entry of row[0 .. cnt) (ascending) that names `target` with image `want`, or -1. guess >= 0: where it is
// likely to be (the search goes outward from there), else the row is bisected.
__device__ __forceinline__ int find_entry(const int32_t *__restrict__ row, const int32_t *__restrict__ image, int cnt,
                                          int target, int want, int guess) {
    int lo = 0, hi = cnt, at = -1, step = 0;
    int g = guess >= 0 ? guess - 1 : (cnt - 4) >> 1;
    while (hi - lo > 4) {
        const int mid = g < lo ? lo : (g > hi - 4 ? hi - 4 : g);
        const Int4 x = *reinterpret_cast<const Int4 *>(row + mid);
        if (x.v[3] < target) lo = mid + 4;
        else if (x.v[0] > target) hi = mid;
        else {
            lo = mid + (x.v[0] < target) + (x.v[1] < target) + (x.v[2] < target);
            const int32_t there = lo == mid ? x.v[0] : lo == mid + 1 ? x.v[1] : lo == mid + 2 ? x.v[2] : x.v[3];
            at = there == target ? lo : -1;
            hi = -1;
        }
        if (guess >= 0 && (lo == 0 || hi == cnt)) {
            g = lo > 0 ? lo + step : hi - 4 - step;
            step = 2 * step + 4;
        } else {
            g = lo + ((hi - lo - 4) >> 1);
        }
    }
    if (hi >= 0) {
        while (lo < hi && row[lo] < target) lo++;
        if (lo < hi && row[lo] == target) at = lo;
    }
    if (at < 0 || image[at] == want) return at;
    while (at > 0 && row[at - 1] == target) at--;        // several images of one atom
    for (; at < cnt && row[at] == target; at++)
        if (image[at] == want) return at;
    return -1;
}

// Whether neighbors in space are far apart in index (one frame): the buckets of an atom then span most of the
// indices, each on its own (types mixed) or together (atoms sorted by type). Asked of four atoms, since the
// buckets of one at the period's edge span the frame in any order; only the search's start depends on it.
__device__ __forceinline__ bool scattered_order(const int32_t *__restrict__ list, const int32_t *__restrict__ counts,
                                                int T, int m, int64_t n) {
    const int lane = threadIdx.x & (WAVE - 1), t = lane & 15;           // 16 lanes, one per type, to an atom
    const int64_t bucket = (2 * (lane >> 4) + 1) * n / 8 * T + t, row = bucket * m;
    const int c = t < T ? min(counts[bucket], m) : 0;
    int64_t f = n, l = 0, sum = 0;
    if (c > 0) {
        f = list[row];
        l = list[row + c - 1];
        sum = l - f;
    }
    int lo = (int)f, hi = (int)l;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o, WAVE);
        lo = min(lo, __shfl_xor(lo, o, WAVE));
        hi = max(hi, __shfl_xor(hi, o, WAVE));
    }
    const bool wide = 4 * (sum < hi - lo ? sum : hi - lo) > 3 * n;
    return __popcll(__ballot(wide && t == 0)) >= 3;
}

__global__ void __launch_bounds__(REV_WAVES * WAVE)
reverse_kernel(const int32_t *__restrict__ list, const int32_t *__restrict__ shift,
               const int32_t *__restrict__ counts, const int32_t *__restrict__ type_map,
               const int64_t *__restrict__ frame_start, const int32_t *__restrict__ atom_frame, int T, int m,
               int64_t n, int32_t *__restrict__ rev, int32_t *__restrict__ status) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int64_t per = (n + REV_XCDS - 1) / REV_XCDS;
    const int64_t i0 = (blockIdx.x % REV_XCDS) * per, i1 = i0 + per < n ? i0 + per : n;
    const bool wide = !frame_start && scattered_order(list, counts, T, m, n);
    for (int64_t i = i0 + (int64_t)(blockIdx.x / REV_XCDS) * REV_WAVES + wid; i < i1;
         i += (int64_t)(gridDim.x / REV_XCDS) * REV_WAVES) {
        const int64_t fb = frame_start ? frame_start[atom_frame[i]] : 0;
        const int ti = type_map[i];
        const int target = (int)(i - fb) + 1;
        bool bad = false;
        float at = 0.0f;
        if (wide) {
            const int own = min(counts[i * T + ti], m);
            const int64_t row = (i * T + ti) * (int64_t)m;
            const int f = own > 0 ? list[row] : target, l = own > 0 ? list[row + own - 1] : target;
            at = fminf(fmaxf((float)(target - f) / (float)(l - f + 1), 0.0f), 1.0f);
        }
        // the entries of all buckets as one sequence: fuller wavefronts, fewer rounds of waiting
        int total = 0;
        for (int t = 0; t < T; t++) {
            const int c = min(counts[i * T + t], m);
            for (int k = c + lane; k < m; k += WAVE) __builtin_nontemporal_store(-1, rev + (i * T + t) * (int64_t)m + k);
            total += c;
        }
        for (int e = lane; e < total; e += WAVE) {
            int t = 0, k = e;
            for (int u = 0; u + 1 < T; u++) {
                const int c = min(counts[i * T + u], m);
                if (t == u && k >= c) { k -= c; t++; }
            }
            const int64_t s = (i * T + t) * (int64_t)m + k;
            const int64_t j = fb + list[s] - 1;
            const int sh = shift[s];
            const int want = pack_shift(-((sh & 255) - 128), -(((sh >> 8) & 255) - 128), -(((sh >> 16) & 255) - 128));
            const int64_t base = (j * T + ti) * (int64_t)m;
            const int cnt = min(counts[j * T + ti], m);
            const int f = find_entry(list + base, shift + base, cnt, target, want, wide ? (int)(at * cnt) : -1);
            if (f < 0) bad = true;
            const int32_t r = f < 0 ? -1 : (int32_t)(base + f);
            __builtin_nontemporal_store(r, rev + s);
        }
        if (__ballot(bad) != 0ull && lane == 0) atomicCAS(status, 0, (int)(i + 1));
    }
}

// ------------------------------------------------------------------ LAMMPS packing
// PairMATPL::generate_neighdata (src/lmps/lammps-libtorch/MATPL/pair_matpl.cpp:522-616)
// on the device. Input is LAMMPS's full neighbor list as CSR (neighbors of atom i
// are neigh[firstneigh[i] .. firstneigh[i] + numneigh[i]), indices over local +
// ghost atoms) and positions x [nall][3] of local and ghost atoms. For list entry
// ii (centre i = ilist[ii]) every neighbor j with |x_j - x_i|^2 <= rc^2 goes,
// in LAMMPS list order, to bucket t_j = type_to_model[type[j] - 1] of row i:
//   list [inum][T][m] = j + 1 (0 = empty), dR [inum][T][m][4] = [r, dx, dy, dz],
//   imagetype[ii] = t_i, counts [inum][T] = neighbors found (may exceed m).
// Unused slots are zeroed (the reference keeps whatever the buffer held).
// status (zero before the call) receives the first problem: 1 + i for a bucket
// that overflowed m (the reference writes past it), -1 for a centre i outside
// [0, inum), -2 for a neighbor outside [0, nall) or a list range outside
// neigh[0 .. nneigh), -3 for a type with no model
// type. min_rsq (uint64, +inf bits before the call) receives the smallest
// accepted |dR|^2 as double bits (non-negative doubles order like their bits),
// for the reference's "two atoms too close" check (pair_matpl.cpp:605-611).
// One wavefront per list entry, lanes over its neighbors, integer wave scans
// to keep list order inside each bucket.
__global__ void __launch_bounds__(256)
lmp_pack_kernel(const double *__restrict__ x, const int32_t *__restrict__ type,
                const int32_t *__restrict__ type_to_model, int ntypes_lmp, const int32_t *__restrict__ ilist,
                const int32_t *__restrict__ numneigh, const int64_t *__restrict__ firstneigh,
                const int32_t *__restrict__ neigh, int64_t nneigh, int64_t inum, int64_t nall, int T, int m,
                double rc2,
                int32_t *__restrict__ imagetype, int32_t *__restrict__ list, double *__restrict__ dR,
                int32_t *__restrict__ counts, unsigned long long *__restrict__ min_rsq,
                int32_t *__restrict__ status) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t ii = blockIdx.x * (int64_t)(blockDim.x / WAVE) + (threadIdx.x / WAVE);
    if (ii >= inum) return;
    const int64_t i = ilist[ii];
    if (i < 0 || i >= inum) {
        if (lane == 0) atomicCAS(status, 0, -1);
        return;
    }
    auto model_type = [&](int64_t a) -> int {
        const int lt = type[a];
        return (lt >= 1 && lt <= ntypes_lmp) ? type_to_model[lt - 1] : -1;
    };
    const int ti = model_type(i);
    if (ti < 0 || ti >= T) {
        if (lane == 0) atomicCAS(status, 0, -3);
        return;
    }
    if (lane == 0) imagetype[ii] = ti;
    const int64_t S = (int64_t)T * m;
    int32_t *li = list + i * S;
    double *di = dR + i * S * 4;
    const double xi = x[3 * i], yi = x[3 * i + 1], zi = x[3 * i + 2];
    const int jnum = numneigh[i];
    const int64_t j0 = firstneigh[i];
    if (jnum < 0 || j0 < 0 || j0 + jnum > nneigh) {
        if (lane == 0) atomicCAS(status, 0, -2);
        return;
    }
    const int32_t *jl = neigh + j0;
    int base[16];
    for (int t = 0; t < T; t++) base[t] = 0;
    double rmin = __longlong_as_double(0x7ff0000000000000LL);
    bool bad_j = false, bad_t = false;
    for (int jc = 0; jc < jnum; jc += WAVE) {
        const int jj = jc + lane;
        int64_t j = jj < jnum ? (int64_t)jl[jj] : -1;
        if (jj < jnum && (j < 0 || j >= nall)) { bad_j = true; j = -1; }
        int tj = -1;
        double dx = 0.0, dy = 0.0, dz = 0.0, rsq = 0.0;
        if (j >= 0) {
            dx = x[3 * j] - xi;
            dy = x[3 * j + 1] - yi;
            dz = x[3 * j + 2] - zi;
            rsq = dx * dx + dy * dy + dz * dz;
            if (rsq <= rc2) {
                tj = model_type(j);
                if (tj < 0 || tj >= T) { bad_t = true; tj = -1; }
            }
        }
        int pos = 0;
        for (int t = 0; t < T; t++) {
            const int v = tj == t ? 1 : 0;
            const int incl = wave_incl_scan(v);
            if (tj == t) pos = base[t] + incl - 1;
            base[t] += __shfl(incl, WAVE - 1, WAVE);
        }
        if (tj >= 0) {
            rmin = fmin(rmin, rsq);
            if (pos < m) {
                const int64_t slot = (int64_t)tj * m + pos;
                li[slot] = (int32_t)(j + 1);
                di[4 * slot] = sqrt(rsq);
                di[4 * slot + 1] = dx;
                di[4 * slot + 2] = dy;
                di[4 * slot + 3] = dz;
            }
        }
    }
    bool over = false;
    for (int t = 0; t < T; t++) {
        over = over || base[t] > m;
        const int used = base[t] < m ? base[t] : m;
        for (int k = used + lane; k < m; k += WAVE) {
            const int64_t slot = (int64_t)t * m + k;
            li[slot] = 0;
            di[4 * slot] = di[4 * slot + 1] = di[4 * slot + 2] = di[4 * slot + 3] = 0.0;
        }
        if (counts && lane == 0) counts[i * T + t] = base[t];
    }
    // wave minimum of the accepted |dR|^2, one atomic per wave
    for (int off = 32; off > 0; off >>= 1) rmin = fmin(rmin, __shfl_xor(rmin, off, WAVE));
    if (lane == 0 && min_rsq) atomicMin(min_rsq, (unsigned long long)__double_as_longlong(rmin));
    const bool any_bad_j = __any(bad_j), any_bad_t = __any(bad_t);
    if (lane == 0) {
        if (any_bad_j) atomicCAS(status, 0, -2);
        else if (any_bad_t) atomicCAS(status, 0, -3);
        else if (over) atomicCAS(status, 0, (int)(i + 1));
    }
}

bool small_box_host(const double *L, double rc) {
    for (int d = 0; d < 3; d++) {
        const double len = sqrt(L[3 * d] * L[3 * d] + L[3 * d + 1] * L[3 * d + 1] + L[3 * d + 2] * L[3 * d + 2]);
        if (len < 2.0 * rc) return true;
    }
    return false;
}

Grid make_grid(const double *L, double rc) {
    // plane spacing h_d = V / |a_e x a_f|
    const double *a = L, *b = L + 3, *c = L + 6;
    auto cross = [](const double *u, const double *v, double *w) {
        w[0] = u[1] * v[2] - u[2] * v[1];
        w[1] = u[2] * v[0] - u[0] * v[2];
        w[2] = u[0] * v[1] - u[1] * v[0];
    };
    double bc[3], ca[3], ab[3];
    cross(b, c, bc); cross(c, a, ca); cross(a, b, ab);
    const double V = fabs(a[0] * bc[0] + a[1] * bc[1] + a[2] * bc[2]);
    const double *ar[3] = {bc, ca, ab};
    Grid g;
    for (int d = 0; d < 3; d++) {
        const double area = sqrt(ar[d][0] * ar[d][0] + ar[d][1] * ar[d][1] + ar[d][2] * ar[d][2]);
        int nc = (int)floor(V / area / rc);
        if (nc < 1) nc = 1;
        if (nc > 1024) nc = 1024;
        g.nc[d] = nc;
        if (nc >= 3) { g.noff[d] = 3; g.off[d][0] = -1; g.off[d][1] = 0; g.off[d][2] = 1; }
        else if (nc == 2) { g.noff[d] = 2; g.off[d][0] = 0; g.off[d][1] = 1; g.off[d][2] = 0; }
        else { g.noff[d] = 1; g.off[d][0] = 0; g.off[d][1] = 0; g.off[d][2] = 0; }
    }
    return g;
}

}  // namespace
}  // namespace matpl

using namespace matpl;

MATPL_EXPORT int64_t matpl_dp_neighbor_cell_workspace_bytes(const double *lattice_host, double rc_m, int64_t n) {
    Grid g = make_grid(lattice_host, rc_m);
    const int64_t ncells = (int64_t)g.nc[0] * g.nc[1] * g.nc[2];
    // atom_cell[n], cell_atoms[n], sorted[3n], cell_count[ncells], overfull[n+1], cell_start[ncells+1],
    // cursor[ncells]
    return (int64_t)sizeof(int32_t) * (6 * n + 3 * ncells + 2 + 64);
}

MATPL_EXPORT int matpl_dp_neighbor_is_small_box(const double *lattice_host, double rc_m) {
    return small_box_host(lattice_host, rc_m) ? 1 : 0;
}

MATPL_EXPORT int matpl_dp_neighbor_brute(const double *lattice, const double *frac, const int64_t *frame_start,
                                         const int32_t *atom_frame, const int32_t *type_map, const double *rc_type,
                                         int ntypes, int m, double rc_m, int64_t nframes, int64_t ntot,
                                         double *frac_wrapped, int32_t *list, double *dR, int32_t *counts,
                                         int32_t *shift, int32_t *status, void *stream) {
    hipStream_t st = (hipStream_t)stream;
    MATPL_CHECK_ARG(ntypes >= 1 && ntypes <= 16, "dp_neighbor: ntypes must be in [1,16]");
    MATPL_CHECK_ARG(m >= 1 && nframes >= 0 && ntot >= 0 && rc_m > 0, "dp_neighbor: bad sizes");
    if (ntot == 0) return OK;
    MATPL_CHECK_ARG(lattice && frac && frame_start && atom_frame && type_map && rc_type && frac_wrapped &&
                        list && status, "dp_neighbor: null pointer");
    hipLaunchKernelGGL(wrap_kernel, dim3(grid_cap(ntot * 3)), dim3(256), 0, st, frac, frac_wrapped, ntot * 3,
                       status);
    int rc = check_launch("wrap_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(brute_kernel, dim3(ceil_div(ntot, 4)), dim3(256), 0, st, lattice, frac_wrapped, frame_start,
                       atom_frame, type_map, rc_type, ntypes, m, rc_m, ntot, list, dR, counts, shift, status);
    return check_launch("brute_kernel");
}

MATPL_EXPORT int matpl_dp_neighbor_cell(const double *lattice_host, const double *frac, const int32_t *type_map,
                                        const double *rc_type, int ntypes, int m, double rc_m, int64_t n,
                                        double *frac_wrapped, int32_t *list, double *dR, int32_t *counts,
                                        int32_t *shift, int32_t *status, void *workspace, int64_t workspace_bytes,
                                        void *stream) {
    hipStream_t st = (hipStream_t)stream;
    MATPL_CHECK_ARG(ntypes >= 1 && ntypes <= 16, "dp_neighbor_cell: ntypes must be in [1,16]");
    MATPL_CHECK_ARG(m >= 1 && n >= 0 && rc_m > 0, "dp_neighbor_cell: bad sizes");
    MATPL_CHECK_ARG(lattice_host, "dp_neighbor_cell: null lattice");
    MATPL_CHECK_ARG(!small_box_host(lattice_host, rc_m),
                    "dp_neighbor_cell: a lattice vector is shorter than 2*rc; use the brute-force search");
    if (n == 0) return OK;
    MATPL_CHECK_ARG(frac && type_map && rc_type && frac_wrapped && list && status && workspace,
                    "dp_neighbor_cell: null pointer");
    MATPL_CHECK_ARG(n < (int64_t)0x7fffffff, "dp_neighbor_cell: too many atoms");
    const int64_t need = matpl_dp_neighbor_cell_workspace_bytes(lattice_host, rc_m, n);
    MATPL_CHECK_ARG(workspace_bytes >= need, "dp_neighbor_cell: workspace %lld < %lld bytes",
                    (long long)workspace_bytes, (long long)need);
    const size_t lds = sizeof(int32_t) * CELL_WAVES * ((size_t)ntypes * m + 2 * ntypes);
    MATPL_CHECK_ARG(lds <= 64 * 1024, "dp_neighbor_cell: ntypes*m too large for LDS buckets");
    Grid g = make_grid(lattice_host, rc_m);
    const int ncells = g.nc[0] * g.nc[1] * g.nc[2];
    int32_t *ws = (int32_t *)workspace;
    int32_t *atom_cell = ws;
    int32_t *cell_atoms = atom_cell + n;
    int32_t *sorted = cell_atoms + n;
    int32_t *cell_count = sorted + 3 * n;               // zeroed, with the word after it
    int32_t *overfull = cell_count + ncells;
    int32_t *cell_start = overfull + 1 + n;
    int32_t *cursor = cell_start + ncells + 1;
    Lattice lat;
    for (int k = 0; k < 9; k++) lat.a[k] = lattice_host[k];
    int rc;
    hipLaunchKernelGGL(wrap_kernel, dim3(grid_cap(n * 3)), dim3(256), 0, st, frac, frac_wrapped, n * 3, status);
    if ((rc = check_launch("wrap_kernel"))) return rc;
    if ((rc = fill_async<int32_t>(cell_count, 0, ncells + 1, st))) return rc;
    hipLaunchKernelGGL(bin_kernel, dim3(grid_cap(n)), dim3(256), 0, st, frac_wrapped, n, g, atom_cell, cell_count);
    if ((rc = check_launch("bin_kernel"))) return rc;
    hipLaunchKernelGGL(scan_kernel, dim3(1), dim3(1024), 0, st, cell_count, cell_start, cursor, ncells);
    if ((rc = check_launch("scan_kernel"))) return rc;
    hipLaunchKernelGGL(fill_cells_kernel, dim3(grid_cap(n)), dim3(256), 0, st, atom_cell, n, cursor, cell_atoms);
    if ((rc = check_launch("fill_cells_kernel"))) return rc;
    CellArgs A{};
    A.lat = lat; A.g = g; A.fw = frac_wrapped; A.atom_cell = atom_cell; A.cell_start = cell_start;
    A.cell_atoms = cell_atoms; A.type_map = type_map; A.rc_type = rc_type; A.T = ntypes; A.m = m; A.rc_m = rc_m;
    A.n = n; A.list = list; A.dR = dR; A.counts = counts; A.shift = shift; A.status = status;
    // A block per cell shares its candidates among the cell's atoms; with few atoms to a cell (a
    // cluster or a slab in vacuum) its wavefronts idle, and with few atoms in all the chip has too
    // few blocks to hide the merging. Whole searches at a cutoff of 6.5 A, by cells' blocks against
    // atom by atom: 20,000 atoms at 4 a cell 100 and 90 us, at 8 a cell 80 and 95, at 16 a cell 91
    // and 119; at a solid's density (0.09 per A^3) 3,000 atoms 82 and 69 us, 6,000 70 and 79,
    // 12,000 89 and 126, 40,000 136 and 264.
    // With fewer than three cells in a direction nothing can be preselected, and every candidate takes
    // the exact test here as there: 14 x 35 x 49 A, 5,123 atoms 177 and 120 us; 13.2 x 13.2 x 400 A,
    // 6,000 atoms 63 and 48. Candidates in LDS (20 bytes each): 2048, which a cell pitch of 6.5 to 9 A
    // needs at the density of a solid, or 4096 where the average cell is fuller; where even that is too
    // small for the average cell (with 8 % for the spread of random positions, some 5 deviations), every
    // block would only find so.
    const double avg = (double)n / ncells * 27.0;
    const bool grid3 = g.nc[0] >= 3 && g.nc[1] >= 3 && g.nc[2] >= 3;
    if (grid3 && n >= CB_MIN_TOTAL && n >= (int64_t)CB_MIN_ATOMS * ncells && 1.08 * avg <= CB_MAX_CAND) {
        A.cap = 1.5 * avg > 2048.0 ? CB_MAX_CAND : 2048;
        hipLaunchKernelGGL(sort_runs_kernel, dim3(grid_cap(ncells, SORT_WAVES)), dim3(SORT_WAVES * WAVE), 0, st,
                           cell_start, ncells, g, A.cap / CB_RUN_SHARE, cell_atoms, sorted);
        if ((rc = check_launch("sort_runs_kernel"))) return rc;
        A.sorted = sorted;
        A.ncells = ncells;
        // enough blocks for the chip, as long as each wavefront has an atom
        const int most = (int)((n / ncells + CB_WAVES - 1) / CB_WAVES);
        int parts = (CB_MIN_BLOCKS + ncells - 1) / ncells;
        A.nparts = parts < 1 ? 1 : (parts > most ? (most > 0 ? most : 1) : parts);
        // FP32 positions span at most three cells, R; each coordinate of a difference is wrong by
        // at most 4 R 2^-24 (two roundings of positions, one of the difference) and the squared
        // length by 4 of its ulps: |d| by less than 6e-7 R + 3e-7 rc.
        double R = 0.0;
        for (int d = 0; d < 3; d++)
            R += 3.0 / g.nc[d] * sqrt(lattice_host[3 * d] * lattice_host[3 * d] +
                                      lattice_host[3 * d + 1] * lattice_host[3 * d + 1] +
                                      lattice_host[3 * d + 2] * lattice_host[3 * d + 2]);
        const double pre = rc_m + 1e-6 * R + 1e-6 * rc_m;
        A.pre2 = (float)(pre * pre * (1.0 + 1e-6));
        for (int d = 0; d < 3; d++) A.pitch[d] = 1.0 / g.nc[d];
        A.overfull = overfull;
        const int64_t nwork = (int64_t)ncells * A.nparts;
        hipLaunchKernelGGL(cell_block_kernel, dim3((unsigned)(8 * ((nwork + 7) / 8))), dim3(CB_WAVES * WAVE),
                           (size_t)A.cap * 20, st, A);
        if ((rc = check_launch("cell_block_kernel"))) return rc;
        hipLaunchKernelGGL(cell_overfull_kernel, dim3(grid_cap(n, CELL_WAVES)), dim3(CELL_WAVES * WAVE), lds, st, A);
        return check_launch("cell_overfull_kernel");
    }
    hipLaunchKernelGGL(cell_kernel, dim3(ceil_div(n, CELL_WAVES)), dim3(CELL_WAVES * WAVE), lds, st, A);
    return check_launch("cell_kernel");
}

MATPL_EXPORT int matpl_dp_neighbor_reverse(const int32_t *list, const int32_t *shift, const int32_t *counts,
                                           const int32_t *type_map, const int64_t *frame_start,
                                           const int32_t *atom_frame, int ntypes, int m, int64_t n, int32_t *rev,
                                           int32_t *status, void *stream) {
    MATPL_CHECK_ARG(ntypes >= 1 && m >= 1 && n >= 0, "dp_neighbor_reverse: bad sizes");
    MATPL_CHECK_ARG(n * ntypes * (int64_t)m < (int64_t)0x7fffffff, "dp_neighbor_reverse: too many slots for int32");
    if (n == 0) return OK;
    MATPL_CHECK_ARG(list && shift && counts && type_map && rev && status, "dp_neighbor_reverse: null pointer");
    MATPL_CHECK_ARG((frame_start == nullptr) == (atom_frame == nullptr),
                    "dp_neighbor_reverse: frame_start and atom_frame go together");
    hipStream_t st = (hipStream_t)stream;
    // at least one block per XCD, a multiple of them
    const unsigned grid = REV_XCDS * ((grid_cap(n, REV_WAVES) + REV_XCDS - 1) / REV_XCDS);
    hipLaunchKernelGGL(reverse_kernel, dim3(grid), dim3(REV_WAVES * WAVE), 0, st, list, shift, counts, type_map,
                       frame_start, atom_frame, ntypes, m, n, rev, status);
    return check_launch("reverse_kernel");
}

MATPL_EXPORT int matpl_dp_lmp_neighdata(const double *x, const int32_t *type, const int32_t *type_to_model,
                                        int ntypes_lmp, const int32_t *ilist, const int32_t *numneigh,
                                        const int64_t *firstneigh, const int32_t *neigh, int64_t nneigh, int64_t inum,
                                        int64_t nall,
                                        int ntypes, int m, double rcut, int32_t *imagetype, int32_t *list,
                                        double *dR, int32_t *counts, void *min_rsq, int32_t *status,
                                        void *stream) {
    MATPL_CHECK_ARG(ntypes >= 1 && ntypes <= 16 && m >= 1 && inum >= 0 && nall >= inum && ntypes_lmp >= 1,
                    "dp_lmp_neighdata: bad sizes");
    MATPL_CHECK_ARG(inum * ntypes * (int64_t)m < (int64_t)0x7fffffff, "dp_lmp_neighdata: too many slots for int32");
    MATPL_CHECK_ARG(nall < (int64_t)0x7fffffff, "dp_lmp_neighdata: too many atoms for int32 indices");
    MATPL_CHECK_ARG(rcut > 0.0, "dp_lmp_neighdata: rcut must be positive");
    if (inum == 0) return OK;
    MATPL_CHECK_ARG(nneigh >= 0, "dp_lmp_neighdata: bad neighbor array size");
    MATPL_CHECK_ARG(x && type && type_to_model && ilist && numneigh && firstneigh && (neigh || nneigh == 0) &&
                        imagetype && list && dR && status,
                    "dp_lmp_neighdata: null pointer");
    hipLaunchKernelGGL(lmp_pack_kernel, dim3((unsigned)((inum + 3) / 4)), dim3(256), 0, (hipStream_t)stream, x, type,
                       type_to_model, ntypes_lmp, ilist, numneigh, firstneigh, neigh, nneigh, inum, nall, ntypes, m,
                       rcut * rcut, imagetype, list, dR, counts, (unsigned long long *)min_rsq, status);
    return check_launch("lmp_pack_kernel");
}
