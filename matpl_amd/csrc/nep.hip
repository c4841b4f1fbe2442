// NEP neighbor search and force / virial scatter on gfx950, FP64 and FP32 (the descriptor's kernels are in
// nep_feat.hip).
//
//   neighbor  : calculateNepNeighbor.cu:166-281 / cpu_calculate_nepneighbor.cpp:97-203
//               every atom of a frame against every atom of the frame in every
//               replica (ia,ib,ic) < num_cell, self excluded in replica 0,
//               minimum image in the expanded box; lists ordered (n2, ia, ib, ic),
//               global indices, -1 padded; Ri = [r, x, y, z] (or [x, y, z])
// Neighbor loops stop at the first -1 entry as the reference's do.
#include "common.h"

#pragma clang fp contract(off)

namespace matpl {
namespace {

constexpr int WAVE = 64;

// ------------------------------------------------------------------ neighbor search
struct NepGeo {
    const double *box;       // [F][18] expanded box + inverse (column-major)
    const double *box_orig;  // [F][9]
    const int64_t *num_cell; // [F][3]
};

__device__ __forceinline__ void apply_mic(const double *h, double &x, double &y, double &z) {
    double sx = h[9] * x + h[10] * y + h[11] * z;
    double sy = h[12] * x + h[13] * y + h[14] * z;
    double sz = h[15] * x + h[16] * y + h[17] * z;
    sx -= nearbyint(sx);
    sy -= nearbyint(sy);
    sz -= nearbyint(sz);
    x = h[0] * sx + h[1] * sy + h[2] * sz;
    y = h[3] * sx + h[4] * sy + h[5] * sz;
    z = h[6] * sx + h[7] * sy + h[8] * sz;
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

// Displacement of replica (ia, ib, ic) of the atom at (px, py, pz) from n1, minimum image in the
// expanded box h, and its square; the expression order is the reference's (calculateNepNeighbor.cu),
// so that the lists and [r, x, y, z] are bit-identical.
__device__ __forceinline__ double replica_disp(const double *h, const double *bo, double px, double py, double pz,
                                               int ia, int ib, int ic, double x1, double y1, double z1, double &x12,
                                               double &y12, double &z12) {
    const double dx = bo[0] * (double)ia + bo[1] * (double)ib + bo[2] * (double)ic;
    const double dy = bo[3] * (double)ia + bo[4] * (double)ib + bo[5] * (double)ic;
    const double dz = bo[6] * (double)ia + bo[7] * (double)ib + bo[8] * (double)ic;
    x12 = px + dx - x1;
    y12 = py + dy - y1;
    z12 = pz + dz - z1;
    apply_mic(h, x12, y12, z12);
    return x12 * x12 + y12 * y12 + z12 * z12;
}

// (R = float: the FP64 values rounded once, as a cast of the double rows would)
template <typename R>
__device__ __forceinline__ void put_entry(int64_t *NL, R *Ri, int64_t idx, int w, int rij4, int64_t n2, double d2,
                                          double x, double y, double z) {
    NL[idx] = n2;
    R *o = Ri + idx * w;
    if (rij4) { o[0] = (R)sqrt(d2); o[1] = (R)x; o[2] = (R)y; o[3] = (R)z; }
    else { o[0] = (R)x; o[1] = (R)y; o[2] = (R)z; }
}

// The same entry from values already rounded, its row in one store where it has four values.
template <typename R>
struct __attribute__((packed, aligned(sizeof(R)))) RiRow {
    R v[4];
};
template <typename R>
__device__ __forceinline__ void put_row(int64_t *NL, R *Ri, int64_t idx, int w, int64_t n2, R r, R x, R y, R z) {
    NL[idx] = n2;
    if (w == 4) {
        *reinterpret_cast<RiRow<R> *>(Ri + idx * 4) = RiRow<R>{{r, x, y, z}};
    } else {
        R *o = Ri + idx * 3;
        o[0] = x; o[1] = y; o[2] = z;
    }
}

// MODE 0: lists; 1: counts; 2: per-type counts. One wavefront per atom n1, lanes over the frame's
// atoms n2, each with its replicas (ia, ib, ic) in the reference's order; a list holds the hits in
// (n2, replica) order. With one replica (the box is at least 2 rc thick) a lane has at most one hit
// per list: the distance test alone runs over the candidates, two chunks of 64 at a time with the next
// two's positions loading, and queues the hits (about one in nine) in LDS; each 64 of them then take the
// square root and the stores together, so that consecutive lanes write consecutive entries. (With root and
// stores under the test of every chunk the kernel was bound by those instructions, run for a few lanes:
// 62,713-atom float batch 303 -> 182 us, 1,728 atoms 28 -> 17.) Several replicas take a counting
// pass, a scan and a writing pass. The per-type counts of MODE 2 are held by lane t for type t, so that the
// lists and counts modes keep their register count low.
template <int MODE, typename R = double>
__global__ void __launch_bounds__(256)
nep_neighbor_kernel(NepGeo g, const int64_t *__restrict__ frame_start, const int32_t *__restrict__ atom_frame,
                    const int64_t *__restrict__ type_map, const double *__restrict__ pos, double rc_r, double rc_a,
                    int64_t maxr, int64_t maxa, int64_t n, int ntypes, int rij4, int64_t *__restrict__ NN_r,
                    int64_t *__restrict__ NL_r, int64_t *__restrict__ NN_a, int64_t *__restrict__ NL_a,
                    R *__restrict__ Ri_r, R *__restrict__ Ri_a, int32_t *__restrict__ status) {
    const int lane = threadIdx.x & (WAVE - 1);
    // the wave index is uniform: the atom, its frame and the frame's boxes stay in scalar registers
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int64_t n1 = blockIdx.x * (int64_t)(blockDim.x / WAVE) + wid;
    if (n1 >= n) return;
    const int f = atom_frame[n1];
    const int64_t N1 = frame_start[f], N2 = frame_start[f + 1];
    double h[18], bo[9];
#pragma unroll
    for (int q = 0; q < 18; q++) h[q] = g.box[18 * (int64_t)f + q];
#pragma unroll
    for (int q = 0; q < 9; q++) bo[q] = g.box_orig[9 * (int64_t)f + q];
    const int64_t *nc = g.num_cell + 3 * (int64_t)f;
    const int na = (int)nc[0], nb = (int)nc[1], ncc = (int)nc[2];
    const bool one = na == 1 && nb == 1 && ncc == 1;
    const double x1 = pos[3 * n1], y1 = pos[3 * n1 + 1], z1 = pos[3 * n1 + 2];
    const double rr2 = rc_r * rc_r, ra2 = rc_a * rc_a;
    const int w = rij4 ? 4 : 3;
    const uint64_t below = (1ull << lane) - 1ull;
    int64_t baser = 0, basea = 0;
    int64_t mytr = 0, myta = 0;     // MODE 2: the counts of type `lane`
    bool overflow = false;
    if constexpr (MODE == 0) {
        if (one) {
            __shared__ int32_t queue[4][2 * WAVE];
            int32_t *qu = queue[wid];
            int nq = 0;
            // the exact entries of the first cnt (<= 64) queued candidates, in order
            auto emit = [&](int cnt) {
                double x12 = 0.0, y12 = 0.0, z12 = 0.0, d2 = 0.0;
                int64_t n2 = 0;
                bool hr = false, ha = false;
                if (lane < cnt) {
                    n2 = N1 + qu[lane];
                    d2 = replica_disp(h, bo, pos[3 * n2], pos[3 * n2 + 1], pos[3 * n2 + 2], 0, 0, 0, x1, y1, z1, x12, y12,
                                      z12);
                    hr = d2 < rr2;
                    ha = d2 < ra2;
                }
                const uint64_t br = __ballot(hr), ba = __ballot(ha);
                const int64_t kr = baser + __popcll(br & below), ka = basea + __popcll(ba & below);
                baser += __popcll(br);
                basea += __popcll(ba);
                if (baser > maxr || basea > maxa) overflow = true;
                const R r = (R)sqrt(d2), x = (R)x12, y = (R)y12, z = (R)z12;
                if (hr && kr < maxr) put_row(NL_r, Ri_r, n1 * maxr + kr, w, n2, r, x, y, z);
                if (ha && ka < maxa) put_row(NL_a, Ri_a, n1 * maxa + ka, w, n2, r, x, y, z);
            };
            double nx[2], ny[2], nz[2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int64_t m2 = N1 + u * WAVE + lane < N2 ? N1 + u * WAVE + lane : N1;
                nx[u] = pos[3 * m2]; ny[u] = pos[3 * m2 + 1]; nz[u] = pos[3 * m2 + 2];
            }
            for (int64_t c0 = N1; c0 < N2; c0 += 2 * WAVE) {
                bool hit[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int64_t n2 = c0 + u * WAVE + lane;
                    double x12, y12, z12;
                    const double d2 = replica_disp(h, bo, nx[u], ny[u], nz[u], 0, 0, 0, x1, y1, z1, x12, y12, z12);
                    hit[u] = n2 < N2 && n1 != n2 && (d2 < rr2 || d2 < ra2);
                    const int64_t m2 = n2 + 2 * WAVE < N2 ? n2 + 2 * WAVE : N1;
                    nx[u] = pos[3 * m2]; ny[u] = pos[3 * m2 + 1]; nz[u] = pos[3 * m2 + 2];
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const uint64_t m = __ballot(hit[u]);
                    if (hit[u]) qu[nq + __popcll(m & below)] = (int32_t)(c0 + u * WAVE + lane - N1);
                    nq += __popcll(m);
                    wave_sync();
                    if (nq >= WAVE) {
                        emit(WAVE);
                        const int32_t rest = lane < nq - WAVE ? qu[WAVE + lane] : 0;
                        wave_sync();
                        qu[lane] = rest;
                        nq -= WAVE;
                        wave_sync();
                    }
                }
            }
            if (nq > 0) emit(nq);
        }
    }
    double px = 0.0, py = 0.0, pz = 0.0;
    if (N1 + lane < N2) {
        const int64_t n2 = N1 + lane;
        px = pos[3 * n2]; py = pos[3 * n2 + 1]; pz = pos[3 * n2 + 2];
    }
    for (int64_t c0 = N1; c0 < N2 && !(MODE == 0 && one); c0 += WAVE) {
        const int64_t n2 = c0 + lane;
        const bool valid = n2 < N2;
        const double cx = px, cy = py, cz = pz;
        if (n2 + WAVE < N2) {
            const int64_t m2 = n2 + WAVE;
            px = pos[3 * m2]; py = pos[3 * m2 + 1]; pz = pos[3 * m2 + 2];
        }
        int cr = 0, ca = 0;
        // type_map is only given (and only read) for the per-type counts of MODE 2
        const int t2 = (MODE == 2 && valid) ? (int)type_map[n2] : 0;
        if (MODE != 0 && one) {
            // one replica: a candidate is at most one hit
            double x12 = 0.0, y12 = 0.0, z12 = 0.0, d2 = 0.0;
            if (valid && n1 != n2) {
                d2 = replica_disp(h, bo, cx, cy, cz, 0, 0, 0, x1, y1, z1, x12, y12, z12);
                cr = d2 < rr2 ? 1 : 0;
                ca = d2 < ra2 ? 1 : 0;
            }
            if constexpr (MODE == 2) {
                for (int t = 0; t < ntypes; t++) {
                    const int ur = __popcll(__ballot(cr && t2 == t)), ua = __popcll(__ballot(ca && t2 == t));
                    if (lane == t) { mytr += ur; myta += ua; }
                }
            } else {
                baser += __popcll(__ballot(cr));
                basea += __popcll(__ballot(ca));
            }
            continue;
        }
        // pass 1: counts
        if (valid) {
            for (int ia = 0; ia < na; ia++)
                for (int ib = 0; ib < nb; ib++)
                    for (int ic = 0; ic < ncc; ic++) {
                        if (ia == 0 && ib == 0 && ic == 0 && n1 == n2) continue;
                        double x12, y12, z12;
                        const double d2 = replica_disp(h, bo, cx, cy, cz, ia, ib, ic, x1, y1, z1, x12, y12, z12);
                        if (d2 < rr2) cr++;
                        if (d2 < ra2) ca++;
                    }
        }
        if constexpr (MODE == 2) {
            for (int t = 0; t < ntypes; t++) {
                const int vr = (valid && t2 == t) ? cr : 0, va = (valid && t2 == t) ? ca : 0;
                const int sr = wave_incl_scan(vr), sa = wave_incl_scan(va);
                const int ur = __shfl(sr, WAVE - 1, WAVE), ua = __shfl(sa, WAVE - 1, WAVE);
                if (lane == t) { mytr += ur; myta += ua; }
            }
            continue;
        }
        const int ir = wave_incl_scan(cr), ia_ = wave_incl_scan(ca);
        const int sumr = __shfl(ir, WAVE - 1, WAVE), suma = __shfl(ia_, WAVE - 1, WAVE);
        const int64_t offr = baser + ir - cr, offa = basea + ia_ - ca;
        baser += sumr;
        basea += suma;
        if constexpr (MODE == 1) continue;
        if (baser > maxr || basea > maxa) { overflow = true; continue; }
        // pass 2: write in (n2, replica) order
        if (valid && (cr > 0 || ca > 0)) {
            int64_t kr = offr, ka = offa;
            for (int ia = 0; ia < na; ia++)
                for (int ib = 0; ib < nb; ib++)
                    for (int ic = 0; ic < ncc; ic++) {
                        if (ia == 0 && ib == 0 && ic == 0 && n1 == n2) continue;
                        double x12, y12, z12;
                        const double d2 = replica_disp(h, bo, cx, cy, cz, ia, ib, ic, x1, y1, z1, x12, y12, z12);
                        if (d2 < rr2) put_entry(NL_r, Ri_r, n1 * maxr + kr++, w, rij4, n2, d2, x12, y12, z12);
                        if (d2 < ra2) put_entry(NL_a, Ri_a, n1 * maxa + ka++, w, rij4, n2, d2, x12, y12, z12);
                    }
        }
    }
    if constexpr (MODE == 2) {
        if (lane < ntypes) { NN_r[n1 * ntypes + lane] = mytr; NN_a[n1 * ntypes + lane] = myta; }
        return;
    }
    if (lane == 0) {
        NN_r[n1] = baser;
        NN_a[n1] = basea;
        if (overflow) atomicCAS(status, 0, (int)(n1 + 1));
    }
    if constexpr (MODE != 0) return;
    // pad the tails (-1 / 0)
    for (int64_t k = (baser < maxr ? baser : maxr) + lane; k < maxr; k += WAVE) {
        NL_r[n1 * maxr + k] = -1;
        for (int q = 0; q < w; q++) Ri_r[(n1 * maxr + k) * w + q] = R(0);
    }
    for (int64_t k = (basea < maxa ? basea : maxa) + lane; k < maxa; k += WAVE) {
        NL_a[n1 * maxa + k] = -1;
        for (int q = 0; q < w; q++) Ri_a[(n1 * maxa + k) * w + q] = R(0);
    }
}

// ------------------------------------------------------------------ force / virial ops
// Neighbor terms of calculateNepForce (NV = 3: out[j] += f, calculateNepForce.cu:25-70) and of
// calculateNepVirial (NV = 9: out[j][3a+c] += f_a Rij[s][c], calculateNepVirial.cu:19-96), with
// f = sum_w dE[s][w] Ri_d[s][w][:] for every slot s whose NL[s] = j >= 0. dE [N][S][4],
// Ri_d [N][S][4][3], Rij [N][S][3], NL int64 [N][S]; out is accumulated into.
// A block takes SC_CH consecutive atoms: a first pass over their slots finds the range [lo, hi) of
// the atoms they name, the terms are added into an LDS copy of out over that range, and the copy's
// nonzero entries are added to out once per block. Per-slot global atomics, which on this GPU are
// carried out beyond the per-XCD L2 caches, remain only for blocks whose range exceeds the copy.
constexpr int SC_CH = 64;       // atoms per block

template <typename T, int NV>
__global__ void __launch_bounds__(256)
nep_scatter_kernel(const int64_t *__restrict__ NL, const T *__restrict__ dE, const T *__restrict__ Ri_d,
                   const T *__restrict__ Rij, T *__restrict__ out, int64_t N, int S, int64_t rcap) {
    extern __shared__ double sc_smem[];
    T *acc = reinterpret_cast<T *>(sc_smem);
    __shared__ int64_t wlo[4], whi[4];
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    const int64_t i0 = blockIdx.x * (int64_t)SC_CH, i1 = i0 + SC_CH < N ? i0 + SC_CH : N;
    const int64_t s0 = i0 * S, s1 = i1 * S;
    int64_t mn = INT64_MAX, mx = -1;
    for (int64_t s = s0 + threadIdx.x; s < s1; s += blockDim.x) {
        const int64_t j = NL[s];
        if (j >= 0) { mn = j < mn ? j : mn; mx = j > mx ? j : mx; }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int64_t a = __shfl_xor(mn, off, WAVE), b = __shfl_xor(mx, off, WAVE);
        mn = a < mn ? a : mn;
        mx = b > mx ? b : mx;
    }
    if (lane == 0) { wlo[wid] = mn; whi[wid] = mx; }
    __syncthreads();
    mn = wlo[0]; mx = whi[0];
    for (int w = 1; w < 4; w++) { mn = wlo[w] < mn ? wlo[w] : mn; mx = whi[w] > mx ? whi[w] : mx; }
    const int64_t lo = mn, hi = mx + 1;
    const bool lds = mx >= 0 && hi - lo <= rcap;
    if (lds)
        for (int64_t r = threadIdx.x; r < NV * (hi - lo); r += blockDim.x) acc[r] = T(0);
    __syncthreads();
    for (int64_t s = s0 + threadIdx.x; s < s1; s += blockDim.x) {
        const int64_t j = NL[s];
        if (j < 0) continue;
        const T *e = dE + 4 * s, *d = Ri_d + 12 * s;
        T v[NV];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const T f = e[0] * d[a] + e[1] * d[3 + a] + e[2] * d[6 + a] + e[3] * d[9 + a];
            if constexpr (NV == 3) {
                v[a] = f;
            } else {
#pragma unroll
                for (int c = 0; c < 3; c++) v[3 * a + c] = f * Rij[3 * s + c];
            }
        }
#pragma unroll
        for (int c = 0; c < NV; c++) {
            if (lds) atomicAdd(acc + NV * (j - lo) + c, v[c]);
            else atomic_add(out + NV * j + c, v[c]);
        }
    }
    __syncthreads();
    if (lds)
        for (int64_t r = threadIdx.x; r < NV * (hi - lo); r += blockDim.x) {
            const T x = acc[r];
            if (x != T(0)) atomic_add(out + NV * lo + r, x);
        }
}

// Centre term of the NEP force, F[i] = -sum_{k, w} dE[i][k][w] Ri_d[i][k][w][:],
// over all S slots (the product src/model/nep_net.py:608 forms with torch.matmul).
// One wavefront per atom; lanes over slots.
template <typename T>
__global__ void __launch_bounds__(256) nep_centre_kernel(const T *__restrict__ dE, const T *__restrict__ Ri_d,
                                                         int64_t N, int S, T *__restrict__ F) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / WAVE;
    if (i >= N) return;
    T f[3] = {T(0), T(0), T(0)};
    for (int k = lane; k < S; k += WAVE) {
        const int64_t s = i * S + k;
        const T *e = dE + 4 * s, *d = Ri_d + 12 * s;
#pragma unroll
        for (int a = 0; a < 3; a++) f[a] += e[0] * d[a] + e[1] * d[3 + a] + e[2] * d[6 + a] + e[3] * d[9 + a];
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const T v = wave_sum(f[a]);
        if (lane == 0) F[3 * i + a] = -v;
    }
}

// Per-frame virial only: sum over the frame's list entries (j >= 0) of
// (dE . Ri_d)_a Rij_c, the row sum of the per-atom virial without forming it.
// Two passes without atomics (deterministic): one wavefront per atom, lanes
// over slots, writes the atom's centre row rows[i][9]; nep_virial_reduce_kernel
// then sums each frame's rows.
template <typename T>
__global__ void __launch_bounds__(256) nep_centre_virial_kernel(const int64_t *__restrict__ NL,
                                                                const T *__restrict__ dE, const T *__restrict__ Rij,
                                                                const T *__restrict__ Ri_d, int64_t N, int S,
                                                                T *__restrict__ rows) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / WAVE;
    if (i >= N) return;
    T v[9];
#pragma unroll
    for (int c = 0; c < 9; c++) v[c] = T(0);
    for (int k = lane; k < S; k += WAVE) {
        const int64_t s = i * S + k;
        if (NL[s] < 0) continue;
        const T *e = dE + 4 * s, *d = Ri_d + 12 * s, *r = Rij + 3 * s;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const T fa = e[0] * d[a] + e[1] * d[3 + a] + e[2] * d[6 + a] + e[3] * d[9 + a];
#pragma unroll
            for (int c = 0; c < 3; c++) v[3 * a + c] += fa * r[c];
        }
    }
#pragma unroll
    for (int c = 0; c < 9; c++) {
        const T x = wave_sum(v[c]);
        if (lane == 0) rows[9 * i + c] = x;
    }
}

// per-frame sum of atom_virial rows: one block per (frame, component)
template <typename T>
__global__ void __launch_bounds__(256) nep_virial_reduce_kernel(const T *__restrict__ atom_virial,
                                                                const int64_t *__restrict__ frame_start,
                                                                T *__restrict__ virial) {
    const int f = blockIdx.y, v = blockIdx.x;
    __shared__ T red[256];
    T acc = T(0);
    for (int64_t r = frame_start[f] + threadIdx.x; r < frame_start[f + 1]; r += 256) acc += atom_virial[9 * r + v];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) virial[9 * f + v] = red[0];
}

// ------------------------------------------------------------------ fused force + frame virial
// F and the per-frame virial of the NEP model from dE and Ri = [r, x, y, z] directly: the position
// derivative Ri_d (row 0 = (x, y, z)/r, rows 1-3 = identity, zero where |r| <= 1e-5; nep_net.py:440-468)
// is formed in registers, so f(s) = dE[s][0] (x, y, z)/r + dE[s][1:4] per used slot s of atom i.
// calculateNepForce's terms (CalcOps.cpp:75-158): F[i] -= f(s), F[j] += f(s); calculateNepVirial's
// frame sum (calculateNepVirial.cu:19-96): V[frame] += f(s) (x) Rij[s].
// A block takes `ch` consecutive atoms i (one wavefront per atom at a time). With LDS copies
// (rcap > 0) it adds the neighbor terms of their slots into an LDS copy of F over the frames those
// atoms belong to (every j of a slot lies in its atom's frame), then writes that copy to its own row
// of `part`; fv_reduce_kernel adds the rows of the blocks covering each atom. A block whose frames
// exceed the LDS copy adds its terms to F with global atomics instead, as does any entry naming an
// atom outside its block's frames, and so does every block without LDS copies (rcap = 0).
// Unlike per-slot global atomics, which on this GPU are carried out beyond the per-XCD L2 caches, the
// LDS adds stay on the CU; the copies pay when many small frames fill the GPU with blocks (fv_plan).
constexpr int FV_CH = 64;        // atoms per block with LDS copies
constexpr int FV_CH_DIRECT = 16; // atoms per block without
constexpr int FV_WAVES = 16;     // one LDS copy shared by many wavefronts, each with few atoms

template <typename T>
struct V4 { T x, y, z, w; };

template <typename T>
__device__ __forceinline__ V4<T> ld4(const T *p) {
    if constexpr (sizeof(T) == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        return {v.x, v.y, v.z, v.w};
    } else {
        const double2 a = reinterpret_cast<const double2 *>(p)[0], b = reinterpret_cast<const double2 *>(p)[1];
        return {a.x, a.y, b.x, b.y};
    }
}

// the frames of atoms [i0, i1): [lo, hi)
__device__ __forceinline__ void fv_range(const int64_t *frame_start, const int32_t *atom_frame, int64_t N, int64_t b,
                                         int ch, int64_t &lo, int64_t &hi) {
    const int64_t i0 = b * ch, i1 = i0 + ch < N ? i0 + ch : N;
    lo = frame_start[atom_frame[i0]];
    hi = frame_start[atom_frame[i1 - 1] + 1];
}

template <typename T>
__global__ void __launch_bounds__(FV_WAVES * WAVE)
nep_fv_kernel(const int64_t *__restrict__ NL, const T *__restrict__ dE, const T *__restrict__ Ri,
              const int64_t *__restrict__ frame_start, const int32_t *__restrict__ atom_frame, int64_t N, int S,
              int ch, int64_t rcap, T *__restrict__ F, T *__restrict__ part, T *__restrict__ rows) {
    extern __shared__ double fv_smem[];
    T *acc = reinterpret_cast<T *>(fv_smem);
    const int lane = threadIdx.x & (WAVE - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int64_t b = blockIdx.x, i0 = b * ch, i1 = i0 + ch < N ? i0 + ch : N;
    int64_t lo, hi;
    fv_range(frame_start, atom_frame, N, b, ch, lo, hi);
    const bool lds = hi - lo <= rcap;
    if (lds)
        for (int64_t r = threadIdx.x; r < 3 * (hi - lo); r += blockDim.x) acc[r] = T(0);
    __syncthreads();
    for (int64_t i = i0 + wid; i < i1; i += FV_WAVES) {
        T c[3] = {T(0), T(0), T(0)}, v[9];
#pragma unroll
        for (int q = 0; q < 9; q++) v[q] = T(0);
        for (int k0 = 0; k0 < S; k0 += 2 * WAVE) {
            // the loads of two passes are issued before either is used
            int64_t jj[2];
            V4<T> qq[2], ee[2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int k = k0 + u * WAVE + lane;
                jj[u] = -1;
                if (k < S) {
                    const int64_t s = i * S + k;
                    jj[u] = NL[s];
                    qq[u] = ld4(Ri + 4 * s);
                    ee[u] = ld4(dE + 4 * s);
                }
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int64_t j = jj[u];
                const V4<T> q = qq[u], e = ee[u];
                if (j < 0 || !(fabs(q.x) > T(1e-5))) continue;
                const T f[3] = {e.x * (q.y / q.x) + e.y, e.x * (q.z / q.x) + e.z, e.x * (q.w / q.x) + e.w};
                const T x[3] = {q.y, q.z, q.w};
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    c[a] += f[a];
#pragma unroll
                    for (int cc = 0; cc < 3; cc++) v[3 * a + cc] += f[a] * x[cc];
                    if (lds && j >= lo && j < hi) atomicAdd(acc + 3 * (j - lo) + a, f[a]);
                    else atomic_add(F + 3 * j + a, f[a]);
                }
            }
        }
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const T x = wave_sum(c[a]);
            if (lane == 0) {
                if (lds) atomicAdd(acc + 3 * (i - lo) + a, -x);
                else atomic_add(F + 3 * i + a, -x);
            }
        }
#pragma unroll
        for (int q = 0; q < 9; q++) {
            const T x = wave_sum(v[q]);
            if (lane == 0) rows[9 * i + q] = x;
        }
    }
    __syncthreads();
    if (lds)
        for (int64_t r = threadIdx.x; r < 3 * (hi - lo); r += blockDim.x) part[b * 3 * rcap + r] = acc[r];
}

// F[j] += the LDS copies of the blocks whose atoms share j's frame (blocks fv_range-covering it)
template <typename T>
__global__ void __launch_bounds__(256)
nep_fv_reduce_kernel(const int64_t *__restrict__ frame_start, const int32_t *__restrict__ atom_frame, int64_t N,
                     int ch, int64_t rcap, const T *__restrict__ part, T *__restrict__ F) {
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < N; j += (int64_t)gridDim.x * blockDim.x) {
        const int f = atom_frame[j];
        const int64_t fs = frame_start[f], fe = frame_start[f + 1];
        if (fe - fs > rcap) continue;             // no block covering this frame used LDS
        T s[3] = {T(0), T(0), T(0)};
        for (int64_t b = fs / ch; b <= (fe - 1) / ch; b++) {
            int64_t lo, hi;
            fv_range(frame_start, atom_frame, N, b, ch, lo, hi);
            if (hi - lo > rcap) continue;
            const T *p = part + b * 3 * rcap + 3 * (j - lo);
            s[0] += p[0]; s[1] += p[1]; s[2] += p[2];
        }
        F[3 * j] += s[0]; F[3 * j + 1] += s[1]; F[3 * j + 2] += s[2];
    }
}

// Backward of nep_fv_kernel wrt dE: with q = gF[j] - gF[i] + gV[frame(i)] Rij[s] (either upstream
// gradient may be absent), g[s] = [q . (x, y, z)/r, q] on used slots with |r| > 1e-5, else 0
// (calculateNepForce.cu:74-122 and the virial's transpose, in one pass). One wavefront per atom.
template <typename T>
__global__ void __launch_bounds__(256)
nep_fv_grad_kernel(const int64_t *__restrict__ NL, const T *__restrict__ Ri, const T *__restrict__ gF,
                   const T *__restrict__ gV, const int32_t *__restrict__ atom_frame, int64_t N, int S,
                   T *__restrict__ g) {
    const int lane = threadIdx.x & (WAVE - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    for (int64_t i = blockIdx.x * (int64_t)(blockDim.x / WAVE) + wid; i < N;
         i += (int64_t)gridDim.x * (blockDim.x / WAVE)) {
        T fi[3] = {T(0), T(0), T(0)}, gv[9];
        if (gF) { fi[0] = gF[3 * i]; fi[1] = gF[3 * i + 1]; fi[2] = gF[3 * i + 2]; }
#pragma unroll
        for (int q = 0; q < 9; q++) gv[q] = gV ? gV[9 * (int64_t)atom_frame[i] + q] : T(0);
        for (int k = lane; k < S; k += WAVE) {
            const int64_t s = i * S + k;
            const int64_t j = NL[s];
            const V4<T> r = ld4(Ri + 4 * s);
            T o[4] = {T(0), T(0), T(0), T(0)};
            if (j >= 0 && fabs(r.x) > T(1e-5)) {
                const T x[3] = {r.y, r.z, r.w};
                T q[3];
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    q[a] = gv[3 * a] * x[0] + gv[3 * a + 1] * x[1] + gv[3 * a + 2] * x[2];
                    if (gF) q[a] += gF[3 * j + a] - fi[a];
                }
                o[0] = q[0] * (x[0] / r.x) + q[1] * (x[1] / r.x) + q[2] * (x[2] / r.x);
                o[1] = q[0]; o[2] = q[1]; o[3] = q[2];
            }
            if constexpr (sizeof(T) == 4) {
                *reinterpret_cast<float4 *>(g + 4 * s) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
                reinterpret_cast<double2 *>(g + 4 * s)[0] = make_double2(o[0], o[1]);
                reinterpret_cast<double2 *>(g + 4 * s)[1] = make_double2(o[2], o[3]);
            }
        }
    }
}

// backward of calculateNepForce wrt dE (calculateNepForce.cu:74-122): the centre
// term -gF_i . Ri_d[s][w] plus the neighbor term gF_j . Ri_d[s][w] (j >= 0)
template <typename T>
__global__ void nep_force_grad_kernel(const int64_t *__restrict__ NL, const T *__restrict__ Ri_d,
                                      const T *__restrict__ gF, T *__restrict__ g, int S, int64_t nslots) {
    for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s < nslots;
         s += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = s / S;
        const int64_t j = NL[s];
        const T *d = Ri_d + 12 * s;
        T q[3] = {-gF[3 * i], -gF[3 * i + 1], -gF[3 * i + 2]};
        if (j >= 0) { q[0] += gF[3 * j]; q[1] += gF[3 * j + 1]; q[2] += gF[3 * j + 2]; }
#pragma unroll
        for (int w = 0; w < 4; w++) g[4 * s + w] = q[0] * d[3 * w] + q[1] * d[3 * w + 1] + q[2] * d[3 * w + 2];
    }
}

// backward of calculateNepVirial wrt dE: g[s][w] = sum_{a,c} gV[f(i)][3a+c] Rij[s][c] Ri_d[s][w][a]
template <typename T>
__global__ void nep_virial_grad_kernel(const int64_t *__restrict__ NL, const T *__restrict__ Rij,
                                       const T *__restrict__ Ri_d, const T *__restrict__ gV,
                                       const int32_t *__restrict__ atom_frame, int S, T *__restrict__ g,
                                       int64_t nslots) {
    for (int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; s < nslots;
         s += (int64_t)gridDim.x * blockDim.x) {
        T o[4] = {T(0), T(0), T(0), T(0)};
        if (NL[s] >= 0) {
            const T *gv = gV + 9 * (int64_t)atom_frame[s / S];
            T q[3];
#pragma unroll
            for (int a = 0; a < 3; a++) q[a] = gv[3 * a] * Rij[3 * s] + gv[3 * a + 1] * Rij[3 * s + 1] + gv[3 * a + 2] * Rij[3 * s + 2];
            const T *d = Ri_d + 12 * s;
#pragma unroll
            for (int w = 0; w < 4; w++) o[w] = q[0] * d[3 * w] + q[1] * d[3 * w + 1] + q[2] * d[3 * w + 2];
        }
#pragma unroll
        for (int w = 0; w < 4; w++) g[4 * s + w] = o[w];
    }
}

template <typename T, int NV>
int scatter_launch(const int64_t *NL, const T *dE, const T *Ri_d, const T *Rij, T *out, int64_t N, int S,
                   hipStream_t st) {
    if (N * S == 0) return OK;
    // LDS copy of at most 63 KB, so that with the kernel's own 64 bytes the block stays within 64 KB
    // (and of no more atoms than there are)
    int64_t rcap = 64512 / (NV * (int64_t)sizeof(T));
    if (rcap > N) rcap = N;
    hipLaunchKernelGGL((nep_scatter_kernel<T, NV>), dim3(ceil_div(N, SC_CH)), dim3(256), NV * rcap * sizeof(T), st, NL,
                       dE, Ri_d, Rij, out, N, S, rcap);
    return check_launch("nep_scatter_kernel");
}

template <typename T>
int virial_launch(const int64_t *NL, const T *dE, const T *Rij, const T *Ri_d, const int64_t *frame_start,
                  int64_t nframes, int64_t N, int S, T *virial, T *atom_virial, hipStream_t st) {
    int rc = fill_async<T>(atom_virial, T(0), N * 9, st);
    if (rc) return rc;
    if ((rc = scatter_launch<T, 9>(NL, dE, Ri_d, Rij, atom_virial, N, S, st))) return rc;
    if (nframes == 0) return OK;
    hipLaunchKernelGGL(nep_virial_reduce_kernel<T>, dim3(9, (unsigned)nframes), dim3(256), 0, st, atom_virial,
                       frame_start, virial);
    return check_launch("nep_virial_reduce_kernel");
}

template <typename T>
int centre_launch(const T *dE, const T *Ri_d, int64_t N, int S, T *F, hipStream_t st) {
    if (N == 0) return OK;
    if (S == 0) return fill_async<T>(F, T(0), N * 3, st);
    hipLaunchKernelGGL(nep_centre_kernel<T>, dim3((unsigned)ceil_div(N, 4)), dim3(256), 0, st, dE, Ri_d, N, S, F);
    return check_launch("nep_centre_kernel");
}

template <typename T>
int frame_virial_launch(const int64_t *NL, const T *dE, const T *Rij, const T *Ri_d, const int64_t *frame_start,
                        int64_t nframes, int64_t N, int S, T *rows, T *virial, hipStream_t st) {
    if (N == 0 || S == 0) return fill_async<T>(virial, T(0), nframes * 9, st);
    hipLaunchKernelGGL(nep_centre_virial_kernel<T>, dim3((unsigned)ceil_div(N, 4)), dim3(256), 0, st, NL, dE, Rij,
                       Ri_d, N, S, rows);
    int rc = check_launch("nep_centre_virial_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(nep_virial_reduce_kernel<T>, dim3(9, (unsigned)nframes), dim3(256), 0, st, rows, frame_start,
                       virial);
    return check_launch("nep_virial_reduce_kernel");
}

}  // namespace
}  // namespace matpl

using namespace matpl;

MATPL_EXPORT int matpl_nep_centre_force(int f64, const void *dE, const void *Ri_d, int64_t N, int S, void *F,
                                        void *stream) {
    MATPL_CHECK_ARG(N >= 0 && S >= 0, "nep_centre_force: bad sizes");
    if (N == 0) return OK;
    MATPL_CHECK_ARG(F && (S == 0 || (dE && Ri_d)), "nep_centre_force: null pointer");
    hipStream_t st = (hipStream_t)stream;
    return f64 ? centre_launch<double>((const double *)dE, (const double *)Ri_d, N, S, (double *)F, st)
               : centre_launch<float>((const float *)dE, (const float *)Ri_d, N, S, (float *)F, st);
}

MATPL_EXPORT int matpl_nep_frame_virial(int f64, const int64_t *NL, const void *dE, const void *Rij, const void *Ri_d,
                                        const int64_t *frame_start, int64_t nframes, int64_t N, int S, void *rows,
                                        void *virial, void *stream) {
    MATPL_CHECK_ARG(N >= 0 && S >= 0 && nframes >= 0, "nep_frame_virial: bad sizes");
    if (nframes == 0) return OK;
    MATPL_CHECK_ARG(virial && (N == 0 || S == 0 || (NL && dE && Rij && Ri_d && frame_start && rows)),
                    "nep_frame_virial: null pointer");
    hipStream_t st = (hipStream_t)stream;
    return f64 ? frame_virial_launch<double>(NL, (const double *)dE, (const double *)Rij, (const double *)Ri_d,
                                             frame_start, nframes, N, S, (double *)rows, (double *)virial, st)
               : frame_virial_launch<float>(NL, (const float *)dE, (const float *)Rij, (const float *)Ri_d,
                                            frame_start, nframes, N, S, (float *)rows, (float *)virial, st);
}

MATPL_EXPORT int matpl_nep_neighbor(const double *box, const double *box_orig, const int64_t *num_cell,
                                    const int64_t *frame_start, const int32_t *atom_frame, const int64_t *type_map,
                                    const double *pos, double rc_r, double rc_a, int64_t maxr, int64_t maxa,
                                    int64_t n, int mode, int ntypes, int rij4, int64_t *NN_r, int64_t *NL_r,
                                    int64_t *NN_a, int64_t *NL_a, double *Ri_r, double *Ri_a, int32_t *status,
                                    void *stream) {
    MATPL_CHECK_ARG(mode >= 0 && mode <= 2 && n >= 0, "nep_neighbor: bad mode/size");
    MATPL_CHECK_ARG(mode != 2 || (ntypes >= 1 && ntypes <= 16), "nep_neighbor: ntypes in [1,16] for typed counts");
    if (n == 0) return OK;
    MATPL_CHECK_ARG(box && box_orig && num_cell && frame_start && atom_frame && pos && NN_r && NN_a,
                    "nep_neighbor: null pointer");
    MATPL_CHECK_ARG(mode != 0 || (NL_r && NL_a && Ri_r && Ri_a && status), "nep_neighbor: null list output");
    MATPL_CHECK_ARG(mode != 2 || type_map, "nep_neighbor: typed counts need type_map");
    NepGeo g{box, box_orig, num_cell};
    const dim3 grid(ceil_div(n, 4)), block(256);
    hipStream_t st = (hipStream_t)stream;
    if (mode == 0)
        hipLaunchKernelGGL(nep_neighbor_kernel<0>, grid, block, 0, st, g, frame_start, atom_frame, type_map, pos, rc_r,
                           rc_a, maxr, maxa, n, ntypes, rij4, NN_r, NL_r, NN_a, NL_a, Ri_r, Ri_a, status);
    else if (mode == 1)
        hipLaunchKernelGGL(nep_neighbor_kernel<1>, grid, block, 0, st, g, frame_start, atom_frame, type_map, pos, rc_r,
                           rc_a, maxr, maxa, n, ntypes, rij4, NN_r, NL_r, NN_a, NL_a, Ri_r, Ri_a, status);
    else
        hipLaunchKernelGGL(nep_neighbor_kernel<2>, grid, block, 0, st, g, frame_start, atom_frame, type_map, pos, rc_r,
                           rc_a, maxr, maxa, n, ntypes, rij4, NN_r, NL_r, NN_a, NL_a, Ri_r, Ri_a, status);
    return check_launch("nep_neighbor_kernel");
}

// matpl_nep_neighbor's lists (mode 0) with the [r, x, y, z] rows in float: each value the FP64 one
// rounded once, as casting matpl_nep_neighbor's double rows would give (for float models).
MATPL_EXPORT int matpl_nep_neighbor_ri32(const double *box, const double *box_orig, const int64_t *num_cell,
                                         const int64_t *frame_start, const int32_t *atom_frame, const double *pos,
                                         double rc_r, double rc_a, int64_t maxr, int64_t maxa, int64_t n, int rij4,
                                         int64_t *NN_r, int64_t *NL_r, int64_t *NN_a, int64_t *NL_a, float *Ri_r,
                                         float *Ri_a, int32_t *status, void *stream) {
    MATPL_CHECK_ARG(n >= 0, "nep_neighbor_ri32: bad size");
    if (n == 0) return OK;
    MATPL_CHECK_ARG(box && box_orig && num_cell && frame_start && atom_frame && pos && NN_r && NN_a && NL_r && NL_a &&
                        Ri_r && Ri_a && status,
                    "nep_neighbor_ri32: null pointer");
    NepGeo g{box, box_orig, num_cell};
    hipLaunchKernelGGL((nep_neighbor_kernel<0, float>), dim3(ceil_div(n, 4)), dim3(256), 0, (hipStream_t)stream, g,
                       frame_start, atom_frame, nullptr, pos, rc_r, rc_a, maxr, maxa, n, 0, rij4, NN_r, NL_r, NN_a,
                       NL_a, Ri_r, Ri_a, status);
    return check_launch("nep_neighbor_kernel");
}

MATPL_EXPORT int matpl_nep_force(int f64, const int64_t *NL, const void *dE, const void *Ri_d, void *F, int64_t N, int S,
                                 void *stream) {
    MATPL_CHECK_ARG(N == 0 || (NL && dE && Ri_d && F), "nep_force: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (f64)
        return scatter_launch<double, 3>(NL, (const double *)dE, (const double *)Ri_d, nullptr, (double *)F, N, S, st);
    return scatter_launch<float, 3>(NL, (const float *)dE, (const float *)Ri_d, nullptr, (float *)F, N, S, st);
}

MATPL_EXPORT int matpl_nep_virial(int f64, const int64_t *NL, const void *dE, const void *Rij, const void *Ri_d,
                                  const int64_t *frame_start, int64_t nframes, int64_t N, int S, void *virial,
                                  void *atom_virial, void *stream) {
    MATPL_CHECK_ARG(N == 0 || (NL && dE && Rij && Ri_d && frame_start && virial && atom_virial),
                    "nep_virial: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (f64)
        return virial_launch<double>(NL, (const double *)dE, (const double *)Rij, (const double *)Ri_d, frame_start,
                                     nframes, N, S, (double *)virial, (double *)atom_virial, st);
    return virial_launch<float>(NL, (const float *)dE, (const float *)Rij, (const float *)Ri_d, frame_start, nframes,
                                N, S, (float *)virial, (float *)atom_virial, st);
}

MATPL_EXPORT int matpl_nep_force_grad(int f64, const int64_t *NL, const void *Ri_d, const void *gF, void *g, int64_t N,
                                      int S, void *stream) {
    if (N * S == 0) return OK;
    MATPL_CHECK_ARG(NL && Ri_d && gF && g, "nep_force_grad: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (f64)
        hipLaunchKernelGGL(nep_force_grad_kernel<double>, dim3(grid_cap(N * S)), dim3(256), 0, st, NL,
                           (const double *)Ri_d, (const double *)gF, (double *)g, S, N * S);
    else
        hipLaunchKernelGGL(nep_force_grad_kernel<float>, dim3(grid_cap(N * S)), dim3(256), 0, st, NL,
                           (const float *)Ri_d, (const float *)gF, (float *)g, S, N * S);
    return check_launch("nep_force_grad_kernel");
}

// LDS copies of F (blocks of FV_CH atoms) when the blocks fill the GPU and every copy spans at most
// the largest span of frames a block can touch (two partial frames and whole ones in between) within
// 64 KB; otherwise blocks of FV_CH_DIRECT atoms and global atomics (a few large frames: a block's
// slots name few of a frame's atoms, and few blocks would share many copies per atom).
struct FvPlan {
    int ch;
    int64_t rcap;
};
inline FvPlan fv_plan(int64_t N, int64_t max_frame, size_t tsize) {
    const int64_t cap = (int64_t)(65536 / (3 * tsize));
    const int64_t want = 2 * max_frame + FV_CH;
    if (N >= 256 * (int64_t)FV_CH && max_frame <= 2048 && want <= cap) return {FV_CH, want};
    return {FV_CH_DIRECT, 0};
}

MATPL_EXPORT int64_t matpl_nep_force_virial_ri_work(int f64, int64_t N, int64_t max_frame) {
    if (N <= 0) return 0;
    const FvPlan pl = fv_plan(N, max_frame, f64 ? 8 : 4);
    return 9 * N + (int64_t)ceil_div(N, pl.ch) * 3 * pl.rcap;
}

template <typename T>
int fv_launch(const int64_t *NL, const T *dE, const T *Ri, const int64_t *frame_start, const int32_t *atom_frame,
              int64_t nframes, int64_t N, int S, int64_t max_frame, T *F, T *virial, T *work, hipStream_t st) {
    int rc = fill_async<T>(F, T(0), 3 * N, st);
    if (rc) return rc;
    if (N == 0 || S == 0) return fill_async<T>(virial, T(0), 9 * nframes, st);
    const FvPlan pl = fv_plan(N, max_frame, sizeof(T));
    T *rows = work, *part = work + 9 * N;
    const int64_t blocks = ceil_div(N, pl.ch);
    hipLaunchKernelGGL(nep_fv_kernel<T>, dim3((unsigned)blocks), dim3(FV_WAVES * WAVE), 3 * pl.rcap * sizeof(T), st,
                       NL, dE, Ri, frame_start, atom_frame, N, S, pl.ch, pl.rcap, F, part, rows);
    if ((rc = check_launch("nep_fv_kernel"))) return rc;
    if (pl.rcap > 0) {
        hipLaunchKernelGGL(nep_fv_reduce_kernel<T>, dim3(grid_cap(N)), dim3(256), 0, st, frame_start, atom_frame, N,
                           pl.ch, pl.rcap, part, F);
        if ((rc = check_launch("nep_fv_reduce_kernel"))) return rc;
    }
    hipLaunchKernelGGL(nep_virial_reduce_kernel<T>, dim3(9, (unsigned)nframes), dim3(256), 0, st, rows, frame_start,
                       virial);
    return check_launch("nep_virial_reduce_kernel");
}

MATPL_EXPORT int matpl_nep_force_virial_ri(int f64, const int64_t *NL, const void *dE, const void *Ri,
                                           const int64_t *frame_start, const int32_t *atom_frame, int64_t nframes,
                                           int64_t N, int S, int64_t max_frame, void *F, void *virial, void *work,
                                           int64_t work_elems, void *stream) {
    MATPL_CHECK_ARG(N >= 0 && S >= 0 && nframes >= 1 && max_frame >= 1, "nep_force_virial_ri: bad sizes");
    MATPL_CHECK_ARG(frame_start && F && virial, "nep_force_virial_ri: null pointer");
    MATPL_CHECK_ARG(N * S == 0 || (NL && dE && Ri && atom_frame && work), "nep_force_virial_ri: null input");
    MATPL_CHECK_ARG(aligned16(dE) && aligned16(Ri), "nep_force_virial_ri: dE and Ri must be 16-byte aligned");
    MATPL_CHECK_ARG(work_elems >= matpl_nep_force_virial_ri_work(f64, N, max_frame),
                    "nep_force_virial_ri: work buffer too small");
    hipStream_t st = (hipStream_t)stream;
    if (f64)
        return fv_launch<double>(NL, (const double *)dE, (const double *)Ri, frame_start, atom_frame, nframes, N, S,
                                 max_frame, (double *)F, (double *)virial, (double *)work, st);
    return fv_launch<float>(NL, (const float *)dE, (const float *)Ri, frame_start, atom_frame, nframes, N, S,
                            max_frame, (float *)F, (float *)virial, (float *)work, st);
}

MATPL_EXPORT int matpl_nep_force_virial_ri_grad(int f64, const int64_t *NL, const void *Ri, const void *gF,
                                                const void *gV, const int32_t *atom_frame, int64_t N, int S, void *g,
                                                void *stream) {
    if (N * S == 0) return OK;
    MATPL_CHECK_ARG(NL && Ri && g && (gF || gV) && (!gV || atom_frame), "nep_force_virial_ri_grad: null pointer");
    MATPL_CHECK_ARG(aligned16(Ri) && aligned16(g), "nep_force_virial_ri_grad: Ri and g must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const unsigned blocks = (unsigned)(ceil_div(N, 4) < 8192 ? ceil_div(N, 4) : 8192);
    if (f64)
        hipLaunchKernelGGL(nep_fv_grad_kernel<double>, dim3(blocks), dim3(256), 0, st, NL, (const double *)Ri,
                           (const double *)gF, (const double *)gV, atom_frame, N, S, (double *)g);
    else
        hipLaunchKernelGGL(nep_fv_grad_kernel<float>, dim3(blocks), dim3(256), 0, st, NL, (const float *)Ri,
                           (const float *)gF, (const float *)gV, atom_frame, N, S, (float *)g);
    return check_launch("nep_fv_grad_kernel");
}

MATPL_EXPORT int matpl_nep_virial_grad(int f64, const int64_t *NL, const void *Rij, const void *Ri_d, const void *gV,
                                       const int32_t *atom_frame, void *g, int64_t N, int S, void *stream) {
    if (N * S == 0) return OK;
    MATPL_CHECK_ARG(NL && Rij && Ri_d && gV && atom_frame && g, "nep_virial_grad: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (f64)
        hipLaunchKernelGGL(nep_virial_grad_kernel<double>, dim3(grid_cap(N * S)), dim3(256), 0, st, NL,
                           (const double *)Rij, (const double *)Ri_d, (const double *)gV, atom_frame, S, (double *)g,
                           N * S);
    else
        hipLaunchKernelGGL(nep_virial_grad_kernel<float>, dim3(grid_cap(N * S)), dim3(256), 0, st, NL,
                           (const float *)Rij, (const float *)Ri_d, (const float *)gV, atom_frame, S, (float *)g,
                           N * S);
    return check_launch("nep_virial_grad_kernel");
}
