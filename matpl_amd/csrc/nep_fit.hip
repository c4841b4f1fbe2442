// NEP fitting net on gfx950: per-type one-hidden-layer nets
//   x = q_scaler * q,  z = x W0[t] + b0[t],  h = tanh z,  Ei = h . w1[t] + b1[t]
// (src/model/nep_fitting.py:40-163 with network_size [H, 1], dispatched per atom
// type at src/model/nep_net.py:470-501), evaluated for every type in one launch.
//
// The forward also writes g = dEi/dq (the reference obtains it by autograd through
// the net); the backward takes the upstream gradients of Ei and of g and returns
// dL/dq and the parameter gradients, i.e. it is the net's first and second
// derivative in one kernel (the force loss reaches the weights through g):
//   u = w1 (1 - h^2),  g_x = W0 u,  gamma = q_scaler * gg,  v = W0^T gamma,
//   t = gE u - 2 v w1 h (1 - h^2)
//   dL/dq  = q_scaler * (W0 t)
//   dL/dW0 = sum_atoms x t^T + gamma u^T,   dL/db0 = sum t,
//   dL/dw1 = sum gE h + v (1 - h^2),        dL/db1 = sum gE.
//
// Layout: atoms grouped by type (perm) and cut into tiles of at most TA atoms of
// one type; one 256-thread block per tile. The tile's rows of x (and gamma) are
// staged in LDS with coalesced loads; thread (a, group) then runs a strided
// subset of hidden units (or features) for atom a, with the weights read as the
// same address across the atom lanes. Parameter gradients are summed per tile
// over its atoms in LDS (threads over weight entries) and written as one partial
// row per tile; a second kernel adds each type's rows in a fixed order, so results
// do not depend on scheduling.
#include "common.h"

namespace matpl {
namespace {

constexpr int FIT_THREADS = 256;

// Each type's weights: W0 [D][H], b0 [H], w1 [H], b1 [1], from stacked arrays ([T] of them) or, when `tables`,
// from one pointer per type, so that a model's own parameters need no stacking.
constexpr int FIT_TYPES = 16;
struct FitWeights {
    const void *W0[FIT_TYPES], *b0[FIT_TYPES], *w1[FIT_TYPES], *b1[FIT_TYPES];
    int tables;
    template <typename T>
    __device__ __forceinline__ void of(int ty, int D, int H, const T *&w0_, const T *&b0_, const T *&w1_,
                                       const T *&b1_) const {
        const int e = tables ? ty : 0;
        const size_t s = tables ? 0 : (size_t)ty;
        w0_ = reinterpret_cast<const T *>(W0[e]) + s * D * H;
        b0_ = reinterpret_cast<const T *>(b0[e]) + s * H;
        w1_ = reinterpret_cast<const T *>(w1[e]) + s * H;
        b1_ = reinterpret_cast<const T *>(b1[e]) + s;
    }
};

struct FitArgs {
    const void *q;           // [N][D] unscaled features
    const void *qs;          // [D]
    const int32_t *perm;     // [N] atoms grouped by type
    const int32_t *tiles;    // [ntiles][3]: type, first position in perm, count (<= TA)
    FitWeights w;
    void *Ei;                // [N]              forward
    void *g;                 // [N][D] dEi/dq    forward (may be null)
    const void *gE;          // [N]              backward (may be null)
    const void *gg;          // [N][D]           backward (may be null)
    void *dq;                // [N][D]           backward (may be null)
    void *part;              // [ntiles][PW]     backward: per-tile parameter-gradient rows
    int D, H, TA;
    int per;                 // forward: atoms per block (divides TA)
    int part_rows;           // forward: rows of W0 in LDS at a time
};

__host__ __device__ inline int odd(int n) { return n | 1; }     // LDS row stride (odd: fewer bank conflicts)

template <typename T>
__device__ __forceinline__ T tanh_t(T z);
template <>
__device__ __forceinline__ float tanh_t<float>(float z) { return tanhf(z); }
template <>
__device__ __forceinline__ double tanh_t<double>(double z) { return tanh(z); }

// Forward: G lanes per R atoms, 256 R / G atoms of a block at a time; lanes over the hidden units, then over the
// features. The type's W0 sits in LDS (rows of odd stride, read along both axes without conflicts), in parts of
// `part` rows where it is larger than FWD_W_LDS; without that the features' sums would read it from global memory
// across its rows, a cache line per lane.
// What bounds it: at thousands of atoms the serial chain of two D x H products on few wavefronts (a block per 64
// atoms, a thread per atom and strided units: 1,728 atoms 23 us, with a block per 8 atoms 5 us); at tens of
// thousands LDS reads, one of W0 per product, hence R atoms to a read. 60,000 atoms, thread per atom / one atom
// per 32 lanes / now: D 30, H 30 float 38 / 23 / 21 us, double 69 / 40 / 33; D 5, H 10 double 19 / 24 / 13;
// D 56, H 100 float 113 / 118 / 88, double 250 / 370 / 195.
constexpr int FIT_GROUP = 32, FIT_GROUP_FEW = 8;     // lanes per atom; of nets with few hidden units
constexpr int FIT_FEW = 16;
constexpr int FIT_ATOMS = FIT_THREADS / FIT_GROUP;
constexpr size_t FWD_W_LDS = 46 * 1024;      // three blocks in a CU's 160 KB

template <typename T, int G, int R, bool WHOLE>
__global__ void __launch_bounds__(FIT_THREADS) nep_fit_fwd_kernel(FitArgs a) {
    extern __shared__ unsigned char smem_raw[];
    constexpr int NA = FIT_THREADS / G;
    const int D = a.D, H = a.H, nsub = a.TA / a.per, DP = WHOLE ? D : a.part_rows;
    const int sd = odd(D), sh = odd(H);
    const int l = threadIdx.x % G, grp = threadIdx.x / G;
    T *x = reinterpret_cast<T *>(smem_raw) + grp * R * (sd + sh);      // [R][D] these atoms' x
    T *u = x + R * sd;                                                 // [R][H] z, then w1 (1 - h^2)
    T *ws = reinterpret_cast<T *>(smem_raw) + NA * R * (sd + sh);   // [DP][sh]
    const int *tile = a.tiles + 3 * (blockIdx.x / nsub);
    const int ty = tile[0], r0 = (blockIdx.x % nsub) * a.per;
    const int first = tile[1] + r0, cnt = tile[2] - r0 < a.per ? tile[2] - r0 : a.per;
    if (cnt <= 0) return;
    const T *q = reinterpret_cast<const T *>(a.q);
    const T *qs = reinterpret_cast<const T *>(a.qs);
    const T *W0, *b0, *w1, *b1;
    a.w.of<T>(ty, D, H, W0, b0, w1, b1);
    // rows [d0, d1) of W0
    auto stage = [&](int d0, int d1) {
        if (!WHOLE) __syncthreads();
        for (int e = threadIdx.x; e < (d1 - d0) * H; e += FIT_THREADS) ws[(e / H) * sh + e % H] = W0[(size_t)d0 * H + e];
        __syncthreads();
    };
    if (WHOLE) stage(0, D);
    for (int rb = 0; rb < cnt; rb += NA * R) {       // the same rounds in every group: parts have barriers
        size_t at[R];
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int r = rb + k * NA + grp;
            at[k] = (size_t)a.perm[first + (r < cnt ? r : cnt - 1)];
            for (int d = l; d < D; d += G) x[k * sd + d] = q[at[k] * D + d] * qs[d];
        }
        wave_sync();
        T e[R];
#pragma unroll
        for (int k = 0; k < R; k++) e[k] = T(0);
        for (int d0 = 0; d0 < D; d0 += DP) {
            const int nd = D - d0 < DP ? D - d0 : DP;
            if (!WHOLE) stage(d0, d0 + nd);
            for (int j = l; j < H; j += G) {
                T z[R];
#pragma unroll
                for (int k = 0; k < R; k++) z[k] = WHOLE || d0 == 0 ? b0[j] : u[k * sh + j];
#pragma unroll 10
                for (int d = 0; d < nd; d++) {
                    const T w = ws[d * sh + j];
#pragma unroll
                    for (int k = 0; k < R; k++) z[k] += x[k * sd + d0 + d] * w;
                }
                const bool last = WHOLE || d0 + nd == D;
                const T w1j = w1[j];
#pragma unroll
                for (int k = 0; k < R; k++) {
                    if (last) {
                        const T h = tanh_t(z[k]);
                        e[k] += w1j * h;
                        z[k] = w1j * (T(1) - h * h);
                    }
                    u[k * sh + j] = z[k];
                }
            }
        }
        wave_sync();
#pragma unroll
        for (int k = 0; k < R; k++) {
#pragma unroll
            for (int o = G / 2; o > 0; o >>= 1) e[k] += __shfl_xor(e[k], o, 64);
            if (l == 0 && rb + k * NA + grp < cnt) reinterpret_cast<T *>(a.Ei)[at[k]] = e[k] + b1[0];
        }
        if (a.g) {
            T *g = reinterpret_cast<T *>(a.g);
            for (int d0 = 0; d0 < D; d0 += DP) {
                const int nd = D - d0 < DP ? D - d0 : DP;
                if (!WHOLE) stage(d0, d0 + nd);
                for (int d = l; d < nd; d += G) {
                    T s[R];
#pragma unroll
                    for (int k = 0; k < R; k++) s[k] = T(0);
#pragma unroll 10
                    for (int j = 0; j < H; j++) {
                        const T w = ws[d * sh + j];
#pragma unroll
                        for (int k = 0; k < R; k++) s[k] += w * u[k * sh + j];
                    }
#pragma unroll
                    for (int k = 0; k < R; k++)
                        if (rb + k * NA + grp < cnt) g[at[k] * D + d0 + d] = s[k] * qs[d0 + d];
                }
            }
        }
        wave_sync();
    }
}

// One partial row per tile: [D*H] dW0, [H] db0, [H] dw1, [1] db1.
__host__ __device__ inline int part_width(int D, int H) { return D * H + 2 * H + 1; }

template <typename T>
__global__ void __launch_bounds__(FIT_THREADS) nep_fit_bwd_kernel(FitArgs a) {
    extern __shared__ unsigned char smem_raw[];
    const int D = a.D, H = a.H, TA = a.TA;
    const int sd = odd(D), sh = odd(H);
    const int NG = FIT_THREADS / TA;
    T *xs = reinterpret_cast<T *>(smem_raw);              // [TA][sd] x
    T *gs = xs + TA * sd;                                 // [TA][sd] gamma
    T *ts = gs + TA * sd;                                 // [TA][sh] t
    T *us = ts + TA * sh;                                 // [TA][sh] u
    T *rs = us + TA * sh;                                 // [TA][sh] gE h + v (1 - h^2)
    T *es = rs + TA * sh;                                 // [TA]     gE
    const int *tile = a.tiles + 3 * blockIdx.x;
    const int ty = tile[0], first = tile[1], cnt = tile[2];
    const T *q = reinterpret_cast<const T *>(a.q);
    const T *qs = reinterpret_cast<const T *>(a.qs);
    const T *gg = reinterpret_cast<const T *>(a.gg);
    const T *gE = reinterpret_cast<const T *>(a.gE);
    const T *W0, *b0, *w1, *b1;
    a.w.of<T>(ty, D, H, W0, b0, w1, b1);
    for (int e = threadIdx.x; e < cnt * D; e += FIT_THREADS) {
        const int at = e / D, d = e - at * D;
        const size_t src = (size_t)a.perm[first + at] * D + d;
        xs[at * sd + d] = q[src] * qs[d];
        gs[at * sd + d] = gg ? gg[src] * qs[d] : T(0);
    }
    for (int r = threadIdx.x; r < TA; r += FIT_THREADS) es[r] = (gE && r < cnt) ? gE[a.perm[first + r]] : T(0);
    __syncthreads();
    const int at = threadIdx.x % TA, grp = threadIdx.x / TA;
    if (at < cnt) {
        const T *x = xs + at * sd, *gm = gs + at * sd;
        const T ge = es[at];
        for (int j = grp; j < H; j += NG) {
            T z = b0[j], v = T(0);
            for (int d = 0; d < D; d++) {
                const T w = W0[d * H + j];
                z += x[d] * w;
                v += gm[d] * w;
            }
            const T h = tanh_t(z), s = T(1) - h * h;
            const T u = w1[j] * s;
            us[at * sh + j] = u;
            ts[at * sh + j] = ge * u - T(2) * v * w1[j] * h * s;
            rs[at * sh + j] = ge * h + v * s;
        }
    }
    __syncthreads();
    if (a.dq && at < cnt) {
        T *dq = reinterpret_cast<T *>(a.dq);
        const T *t = ts + at * sh;
        for (int d = grp; d < D; d += NG) {
            T s = T(0);
            for (int j = 0; j < H; j++) s += W0[d * H + j] * t[j];
            dq[(size_t)a.perm[first + at] * D + d] = s * qs[d];
        }
    }
    // this tile's parameter-gradient row
    const int PW = part_width(D, H);
    T *row = reinterpret_cast<T *>(a.part) + (size_t)blockIdx.x * PW;
    for (int e = threadIdx.x; e < PW; e += FIT_THREADS) {
        T s = T(0);
        if (e < D * H) {
            const int d = e / H, j = e - d * H;
            for (int r = 0; r < cnt; r++) s += xs[r * sd + d] * ts[r * sh + j] + gs[r * sd + d] * us[r * sh + j];
        } else if (e < D * H + H) {
            const int j = e - D * H;
            for (int r = 0; r < cnt; r++) s += ts[r * sh + j];
        } else if (e < D * H + 2 * H) {
            const int j = e - D * H - H;
            for (int r = 0; r < cnt; r++) s += rs[r * sh + j];
        } else {
            for (int r = 0; r < cnt; r++) s += es[r];
        }
        row[e] = s;
    }
}

// Parameter gradients of type t = sum of its tiles' rows [tstart[t], tstart[t+1]): a block takes 32
// entries, its 8 thread groups sum every 8th tile each, and the 8 partial sums are added in group
// order (deterministic).
constexpr int RED_ENTRIES = 32, RED_GROUPS = 8;
template <typename T>
__global__ void __launch_bounds__(RED_ENTRIES * RED_GROUPS)
nep_fit_reduce_kernel(const T *part, const int32_t *tstart, int PW, int D, int H, T *dW0, T *db0, T *dw1, T *db1) {
    __shared__ T red[RED_GROUPS][RED_ENTRIES];
    const int t = blockIdx.y;
    const int el = threadIdx.x % RED_ENTRIES, g = threadIdx.x / RED_ENTRIES;
    const int e = blockIdx.x * RED_ENTRIES + el;
    T s = T(0);
    if (e < PW)
        for (int k = tstart[t] + g; k < tstart[t + 1]; k += RED_GROUPS) s += part[(size_t)k * PW + e];
    red[g][el] = s;
    __syncthreads();
    if (g != 0 || e >= PW) return;
    s = T(0);
    for (int q = 0; q < RED_GROUPS; q++) s += red[q][el];
    if (e < D * H) dW0[(size_t)t * D * H + e] = s;
    else if (e < D * H + H) db0[(size_t)t * H + e - D * H] = s;
    else if (e < D * H + 2 * H) dw1[(size_t)t * H + e - D * H - H] = s;
    else db1[t] = s;
}

size_t fwd_lds(int D, int H, int rows, int atoms, size_t es) {
    return es * ((size_t)atoms * (odd(D) + odd(H)) + (size_t)rows * odd(H));
}
size_t bwd_lds(int D, int H, int TA, size_t es) {
    return es * (2 * (size_t)TA * odd(D) + 3 * (size_t)TA * odd(H) + (size_t)TA);
}

template <typename T, int G, int R>
int fwd_launch_r(FitArgs &a, int ntiles, hipStream_t st) {
    constexpr size_t LDS_MAX = 64 * 1024;
    constexpr int NA = FIT_THREADS / G * R;
    const size_t row = (size_t)odd(a.H) * sizeof(T);
    a.part_rows = a.D * row <= FWD_W_LDS ? a.D : (int)(FWD_W_LDS / 2 / row);
    if (fwd_lds(a.D, a.H, a.part_rows, NA, sizeof(T)) > LDS_MAX) {
        if constexpr (R > 1) return fwd_launch_r<T, G, R / 2>(a, ntiles, st);
        if constexpr (G != FIT_GROUP) return fwd_launch_r<T, FIT_GROUP, 1>(a, ntiles, st);
        // (the atoms' rows of the widest nets, at most half of it, and what is left for W0)
        a.part_rows = (int)((LDS_MAX - fwd_lds(a.D, a.H, 0, NA, sizeof(T))) / row);
    }
    const size_t lds = fwd_lds(a.D, a.H, a.part_rows, NA, sizeof(T));
    const dim3 grid((unsigned)ntiles * (unsigned)(a.TA / a.per)), block(FIT_THREADS);
    if (a.part_rows == a.D) {
        hipLaunchKernelGGL((nep_fit_fwd_kernel<T, G, R, true>), grid, block, lds, st, a);
    } else if constexpr (G != FIT_GROUP) {
        return fwd_launch_r<T, FIT_GROUP, 1>(a, ntiles, st);
    } else {
        hipLaunchKernelGGL((nep_fit_fwd_kernel<T, G, R, false>), grid, block, lds, st, a);
    }
    return check_launch("nep_fit_fwd_kernel");
}

template <typename T>
int fwd_launch(FitArgs &a, int ntiles, hipStream_t st) {
    // fewer atoms per block while that leaves the chip short of blocks (four per CU), down to one per half-wave
    a.per = a.TA;
    while (a.per > FIT_ATOMS && (int64_t)ntiles * (a.TA / a.per) < 1024) a.per /= 2;
    // 32 lanes per atom leave most idle with few hidden units, where the atoms are enough without
    if (a.H <= FIT_FEW && a.per >= FIT_THREADS / FIT_GROUP_FEW) return fwd_launch_r<T, FIT_GROUP_FEW, 1>(a, ntiles, st);
    if (a.per >= 4 * FIT_ATOMS) return fwd_launch_r<T, FIT_GROUP, 4>(a, ntiles, st);
    if (a.per >= 2 * FIT_ATOMS) return fwd_launch_r<T, FIT_GROUP, 2>(a, ntiles, st);
    return fwd_launch_r<T, FIT_GROUP, 1>(a, ntiles, st);
}

int set_stacked(FitArgs &a, const void *W0, const void *b0, const void *w1, const void *b1) {
    a.w.tables = 0;
    a.w.W0[0] = W0; a.w.b0[0] = b0; a.w.w1[0] = w1; a.w.b1[0] = b1;
    return OK;
}

int set_tables(FitArgs &a, int ntypes, const void *const *W0, const void *const *b0, const void *const *w1,
               const void *const *b1) {
    MATPL_CHECK_ARG(ntypes >= 1 && ntypes <= FIT_TYPES, "nep_fit: ntypes must be in [1,%d]", FIT_TYPES);
    MATPL_CHECK_ARG(W0 && b0 && w1 && b1, "nep_fit: null weight table");
    a.w.tables = 1;
    for (int t = 0; t < ntypes; t++) {
        MATPL_CHECK_ARG(W0[t] && b0[t] && w1[t] && b1[t], "nep_fit: null weights of type %d", t);
        a.w.W0[t] = W0[t]; a.w.b0[t] = b0[t]; a.w.w1[t] = w1[t]; a.w.b1[t] = b1[t];
    }
    return OK;
}

int forward_run(FitArgs &a, int f64, const void *q, const void *qs, const int32_t *perm, const int32_t *tiles, int ntiles,
                int tile_atoms, int D, int H, void *Ei, void *g, hipStream_t st) {
    a.q = q; a.qs = qs; a.perm = perm; a.tiles = tiles; a.Ei = Ei; a.g = g; a.D = D; a.H = H; a.TA = tile_atoms;
    return f64 ? fwd_launch<double>(a, ntiles, st) : fwd_launch<float>(a, ntiles, st);
}

int backward_run(FitArgs &a, int f64, const void *q, const void *qs, const int32_t *perm, const int32_t *tiles,
                 int ntiles, int tile_atoms, const int32_t *tstart, int ntypes, int D, int H, const void *gE,
                 const void *gg, void *dq, void *part, void *dW0, void *db0, void *dw1, void *db1, hipStream_t st) {
    const int PW = part_width(D, H);
    if (ntiles > 0) {
        a.q = q; a.qs = qs; a.perm = perm; a.tiles = tiles;
        a.gE = gE; a.gg = gg; a.dq = dq; a.part = part; a.D = D; a.H = H; a.TA = tile_atoms;
        if (f64)
            hipLaunchKernelGGL(nep_fit_bwd_kernel<double>, dim3(ntiles), dim3(FIT_THREADS), bwd_lds(D, H, a.TA, 8), st,
                               a);
        else
            hipLaunchKernelGGL(nep_fit_bwd_kernel<float>, dim3(ntiles), dim3(FIT_THREADS), bwd_lds(D, H, a.TA, 4), st,
                               a);
        int rc = check_launch("nep_fit_bwd_kernel");
        if (rc) return rc;
    }
    const dim3 grid((PW + RED_ENTRIES - 1) / RED_ENTRIES, ntypes);
    const dim3 block(RED_ENTRIES * RED_GROUPS);
    if (f64)
        hipLaunchKernelGGL(nep_fit_reduce_kernel<double>, grid, block, 0, st, static_cast<const double *>(part),
                           tstart, PW, D, H, static_cast<double *>(dW0), static_cast<double *>(db0),
                           static_cast<double *>(dw1), static_cast<double *>(db1));
    else
        hipLaunchKernelGGL(nep_fit_reduce_kernel<float>, grid, block, 0, st, static_cast<const float *>(part),
                           tstart, PW, D, H, static_cast<float *>(dW0), static_cast<float *>(db0),
                           static_cast<float *>(dw1), static_cast<float *>(db1));
    return check_launch("nep_fit_reduce_kernel");
}

}  // namespace
}  // namespace matpl

using namespace matpl;

// Atoms per tile for a net of D features and H hidden units: the largest power of two in
// [8, 64] whose backward LDS fits 64 KiB (the forward needs less).
MATPL_EXPORT int matpl_nep_fit_tile_atoms(int f64, int D, int H) {
    if (D < 1 || H < 1) return -1;
    const size_t es = f64 ? 8 : 4;
    for (int ta = 64; ta >= 8; ta >>= 1)
        if (bwd_lds(D, H, ta, es) <= 64 * 1024) return ta;
    return -1;
}

MATPL_EXPORT int matpl_nep_fit_part_width(int D, int H) { return part_width(D, H); }

MATPL_EXPORT int matpl_nep_fit_forward(int f64, const void *q, const void *qs, const int32_t *perm,
                                       const int32_t *tiles, int ntiles, int tile_atoms, const void *W0,
                                       const void *b0, const void *w1, const void *b1, int D, int H, void *Ei,
                                       void *g, void *stream) {
    MATPL_CHECK_ARG(D >= 1 && H >= 1 && ntiles >= 0, "nep_fit_forward: bad sizes D=%d H=%d", D, H);
    MATPL_CHECK_ARG(tile_atoms == matpl_nep_fit_tile_atoms(f64, D, H),
                    "nep_fit_forward: tile_atoms %d is not matpl_nep_fit_tile_atoms (%d)", tile_atoms,
                    matpl_nep_fit_tile_atoms(f64, D, H));
    if (ntiles == 0) return OK;
    MATPL_CHECK_ARG(q && qs && perm && tiles && W0 && b0 && w1 && b1 && Ei, "nep_fit_forward: null pointer");
    FitArgs a{};
    set_stacked(a, W0, b0, w1, b1);
    return forward_run(a, f64, q, qs, perm, tiles, ntiles, tile_atoms, D, H, Ei, g, (hipStream_t)stream);
}

// matpl_nep_fit_forward with one weight pointer per type (host tables of ntypes device pointers).
MATPL_EXPORT int matpl_nep_fit_forward_nets(int f64, const void *q, const void *qs, const int32_t *perm,
                                            const int32_t *tiles, int ntiles, int tile_atoms, int ntypes,
                                            const void *const *W0, const void *const *b0, const void *const *w1,
                                            const void *const *b1, int D, int H, void *Ei, void *g, void *stream) {
    MATPL_CHECK_ARG(D >= 1 && H >= 1 && ntiles >= 0, "nep_fit_forward_nets: bad sizes D=%d H=%d", D, H);
    MATPL_CHECK_ARG(tile_atoms == matpl_nep_fit_tile_atoms(f64, D, H),
                    "nep_fit_forward_nets: tile_atoms %d is not matpl_nep_fit_tile_atoms", tile_atoms);
    if (ntiles == 0) return OK;
    MATPL_CHECK_ARG(q && qs && perm && tiles && Ei, "nep_fit_forward_nets: null pointer");
    FitArgs a{};
    const int rc = set_tables(a, ntypes, W0, b0, w1, b1);
    if (rc) return rc;
    return forward_run(a, f64, q, qs, perm, tiles, ntiles, tile_atoms, D, H, Ei, g, (hipStream_t)stream);
}

MATPL_EXPORT int matpl_nep_fit_backward(int f64, const void *q, const void *qs, const int32_t *perm,
                                        const int32_t *tiles, int ntiles, int tile_atoms, const int32_t *tstart,
                                        int ntypes, const void *W0, const void *b0, const void *w1, const void *b1,
                                        int D, int H, const void *gE, const void *gg, void *dq, void *part,
                                        void *dW0, void *db0, void *dw1, void *db1, void *stream) {
    MATPL_CHECK_ARG(D >= 1 && H >= 1 && ntiles >= 0 && ntypes >= 1, "nep_fit_backward: bad sizes D=%d H=%d", D, H);
    MATPL_CHECK_ARG(tile_atoms == matpl_nep_fit_tile_atoms(f64, D, H),
                    "nep_fit_backward: tile_atoms %d is not matpl_nep_fit_tile_atoms (%d)", tile_atoms,
                    matpl_nep_fit_tile_atoms(f64, D, H));
    MATPL_CHECK_ARG(tstart && dW0 && db0 && dw1 && db1, "nep_fit_backward: null pointer");
    MATPL_CHECK_ARG(ntiles == 0 || (q && qs && perm && tiles && W0 && b0 && w1 && b1 && part),
                    "nep_fit_backward: null pointer");
    FitArgs a{};
    set_stacked(a, W0, b0, w1, b1);
    return backward_run(a, f64, q, qs, perm, tiles, ntiles, tile_atoms, tstart, ntypes, D, H, gE, gg, dq, part, dW0, db0,
                        dw1, db1, (hipStream_t)stream);
}

// matpl_nep_fit_backward with one weight pointer per type; the gradients stay stacked.
MATPL_EXPORT int matpl_nep_fit_backward_nets(int f64, const void *q, const void *qs, const int32_t *perm,
                                             const int32_t *tiles, int ntiles, int tile_atoms, const int32_t *tstart,
                                             int ntypes, const void *const *W0, const void *const *b0,
                                             const void *const *w1, const void *const *b1, int D, int H,
                                             const void *gE, const void *gg, void *dq, void *part, void *dW0,
                                             void *db0, void *dw1, void *db1, void *stream) {
    MATPL_CHECK_ARG(D >= 1 && H >= 1 && ntiles >= 0, "nep_fit_backward_nets: bad sizes D=%d H=%d", D, H);
    MATPL_CHECK_ARG(tile_atoms == matpl_nep_fit_tile_atoms(f64, D, H),
                    "nep_fit_backward_nets: tile_atoms %d is not matpl_nep_fit_tile_atoms", tile_atoms);
    MATPL_CHECK_ARG(tstart && dW0 && db0 && dw1 && db1 && (ntiles == 0 || (q && qs && perm && tiles && part)),
                    "nep_fit_backward_nets: null pointer");
    FitArgs a{};
    const int rc = set_tables(a, ntypes, W0, b0, w1, b1);
    if (rc) return rc;
    return backward_run(a, f64, q, qs, perm, tiles, ntiles, tile_atoms, tstart, ntypes, D, H, gE, gg, dq, part, dW0, db0,
                        dw1, db1, (hipStream_t)stream);
}
