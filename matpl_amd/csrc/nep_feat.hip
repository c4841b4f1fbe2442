// NEP descriptor kernels on gfx950: radial and angular (3/4/5-body) features, their first and second
// derivatives, FP64 and FP32.
//
// Semantics (the reference's src/op contract, with the maths restated):
//   f_k(r)    : (T_k(x)+1)/2 fc(r), x = 2(r/rc-1)^2-1, fc = (1+cos(pi r/rc))/2 (r < rc)
//   radial    : q_n = sum_j sum_k c2[ti,tj,n,k] f_k(r_ij)         (calculateNepFeat.cu:5-96)
//   angular   : s_nlm = sum_j g_n(r_ij) b_lm(r_ij/r), g_n = sum_k c3[ti,tj,n,k] f_k
//               q = C3B-weighted s^2 per L, 4-body, 5-body         (nep3_small_box.cuh:68-146)
// Derivatives are taken with r and (x, y, z) as independent inputs, the reference's convention for the
// [N, S, 4] gradient of the descriptor ops. Neighbor loops stop at the first -1 entry as the reference's do.
//
// Every quantity is linear in the basis f_k(r) per neighbor type, which both kernel families use:
//   radial : per atom only F[t][k] = sum_{j of type t} f_k(r_ij) is summed over slots. The features are
//            q_n = sum_{t,k} c[ti,t,n,k] F[t][k], the coefficient gradient g_n F[t][k], and the slot
//            derivative sum_k w[t][k] f'_k with w[t][k] = sum_n g_n c[ti,t,n,k] formed once per atom: nb
//            multiply-adds a slot instead of nm nb, and no coefficient loads per slot.
//   angular: sums over slots are products of small matrices with the slots as the reduction index
//            (s = G^T B, P, dc = Z^T V), so they run on the matrix cores (16x16x4, FP32 or FP64 exact
//            products) from per-slot rows in LDS; several atoms of one type share a 64-lane pass.
// Coefficient gradients go to per-block (or per-wavefront) tables in LDS and to global memory once per block.
#include "common.h"

namespace matpl {
namespace {

constexpr int WAVE = 64;
constexpr int NB_MAX = 20;      // basis functions
constexpr int NM_MAX = 8;       // radial functions per descriptor part
constexpr int NT_MAX = 16;      // atom types
constexpr int NLM = 24;
constexpr double PI_D = 3.14159265358979323846;

// f_k(r) and f_k'(r) for k = 0, 1, 2, ... in order, one per next() call. The Chebyshev recursion starts
// from T_{-1} = T_1 = x and T_0 = 1, so that no k is special.
template <typename T>
struct Basis {
    T x2, hfc, h1, h2, tm, t, pm, p;
    __device__ __forceinline__ Basis(T r, T rc) {
        const T rcinv = T(1) / rc, u = r * rcinv, d = u - T(1);
        const T x = T(2) * d * d - T(1);
        T fc = T(0), fcp = T(0);
        if (r < rc) {
            T s, c;
            if constexpr (sizeof(T) == 4) sincospif(u, &s, &c);
            else sincospi(u, &s, &c);
            fc = T(0.5) * c + T(0.5);
            fcp = -T(0.5 * PI_D) * s * rcinv;
        }
        hfc = T(0.5) * fc;
        h1 = T(2) * d * rcinv * fc;
        h2 = T(0.5) * fcp;
        x2 = T(2) * x;
        tm = x; t = T(1); pm = T(1); p = T(0);
    }
    __device__ __forceinline__ void step() {
        const T pn = x2 * p + (T(2) * t - pm), tn = x2 * t - tm;
        tm = t; t = tn; pm = p; p = pn;
    }
    __device__ __forceinline__ T value() const { return (t + T(1)) * hfc; }
    __device__ __forceinline__ T slope() const { return p * h1 + (t + T(1)) * h2; }
};

// The 24 real harmonics b_k(u) of a unit vector u (accumulate_s order): calls
// fn(k, b_k, db_k/dux, db_k/duy, db_k/duz) for k = 0..23. With r and (x, y, z)
// as independent inputs and u = (x, y, z)/r:
//   db_k/dx_w = (db_k/du_w) / r,   db_k/dr = -(u . db_k/du) / r.
template <typename T, typename Fn>
__device__ __forceinline__ void blm_each(T x, T y, T z, Fn &&fn) {
    const T x2 = x * x, y2 = y * y, z2 = z * z, xy2 = x2 - y2;
    fn(0, z, T(0), T(0), T(1));
    fn(1, x, T(1), T(0), T(0));
    fn(2, y, T(0), T(1), T(0));
    fn(3, T(3) * z2 - T(1), T(0), T(0), T(6) * z);
    fn(4, x * z, z, T(0), x);
    fn(5, y * z, T(0), z, y);
    fn(6, xy2, T(2) * x, -T(2) * y, T(0));
    fn(7, T(2) * x * y, T(2) * y, T(2) * x, T(0));
    fn(8, (T(5) * z2 - T(3)) * z, T(0), T(0), T(15) * z2 - T(3));
    fn(9, (T(5) * z2 - T(1)) * x, T(5) * z2 - T(1), T(0), T(10) * x * z);
    fn(10, (T(5) * z2 - T(1)) * y, T(0), T(5) * z2 - T(1), T(10) * y * z);
    fn(11, xy2 * z, T(2) * x * z, -T(2) * y * z, xy2);
    fn(12, T(2) * x * y * z, T(2) * y * z, T(2) * x * z, T(2) * x * y);
    fn(13, (x2 - T(3) * y2) * x, T(3) * x2 - T(3) * y2, -T(6) * x * y, T(0));
    fn(14, (T(3) * x2 - y2) * y, T(6) * x * y, T(3) * x2 - T(3) * y2, T(0));
    fn(15, (T(35) * z2 - T(30)) * z2 + T(3), T(0), T(0), T(140) * z2 * z - T(60) * z);
    fn(16, (T(7) * z2 - T(3)) * x * z, (T(7) * z2 - T(3)) * z, T(0), T(21) * x * z2 - T(3) * x);
    fn(17, (T(7) * z2 - T(3)) * y * z, T(0), (T(7) * z2 - T(3)) * z, T(21) * y * z2 - T(3) * y);
    fn(18, (T(7) * z2 - T(1)) * xy2, T(2) * x * (T(7) * z2 - T(1)), -T(2) * y * (T(7) * z2 - T(1)),
       T(14) * z * xy2);
    fn(19, (T(7) * z2 - T(1)) * x * y * T(2), T(2) * y * (T(7) * z2 - T(1)), T(2) * x * (T(7) * z2 - T(1)),
       T(28) * x * y * z);
    fn(20, (x2 - T(3) * y2) * x * z, (T(3) * x2 - T(3) * y2) * z, -T(6) * x * y * z, (x2 - T(3) * y2) * x);
    fn(21, (T(3) * x2 - y2) * y * z, T(6) * x * y * z, (T(3) * x2 - T(3) * y2) * z, (T(3) * x2 - y2) * y);
    fn(22, xy2 * xy2 - T(4) * x2 * y2, T(4) * x2 * x - T(12) * x * y2, T(4) * y2 * y - T(12) * x2 * y, T(0));
    fn(23, T(4) * x * y * xy2, T(12) * x2 * y - T(4) * y2 * y, T(4) * x2 * x - T(12) * x * y2, T(0));
}

// ------------------------------------------------------------ q(s) and its gradient
// Weighted C3B (factor 2 on m != 0, nep_cpu.cpp:93-107), C4B, C5B (nep_cpu.h:8-16).
__constant__ double kC3B[NLM] = {
    0.238732414637843, 0.238732414637844, 0.238732414637844, 0.099471839432435, 1.193662073189216,
    1.193662073189216, 0.298415518297304, 0.298415518297304, 0.139260575205408, 0.208890862808112,
    0.208890862808112, 2.088908628081126, 2.088908628081126, 0.348151438013522, 0.348151438013522,
    0.011190581936149, 0.447623277445956, 0.447623277445956, 0.223811638722978, 0.223811638722978,
    3.133362942121690, 3.133362942121690, 0.391670367765212, 0.391670367765212};
__constant__ double kC4B[5] = {-0.007499480826664, -0.134990654879954, 0.067495327439977, 0.404971964639861,
                               -0.809943929279723};
__constant__ double kC5B[3] = {0.026596810706114, 0.053193621412227, 0.026596810706114};

// Forward-mode dual number (value, tangent) for Hessian-vector products.
template <typename T>
struct Dual {
    T v, e;
    __device__ Dual() {}
    __device__ Dual(T a) : v(a), e(T(0)) {}
    __device__ Dual(T a, T b) : v(a), e(b) {}
};
template <typename T> __device__ __forceinline__ Dual<T> operator+(Dual<T> a, Dual<T> b) { return {a.v + b.v, a.e + b.e}; }
template <typename T> __device__ __forceinline__ Dual<T> operator-(Dual<T> a, Dual<T> b) { return {a.v - b.v, a.e - b.e}; }
template <typename T> __device__ __forceinline__ Dual<T> operator*(Dual<T> a, Dual<T> b) { return {a.v * b.v, a.v * b.e + a.e * b.v}; }
template <typename T> __device__ __forceinline__ Dual<T> operator*(T a, Dual<T> b) { return {a * b.v, a * b.e}; }

// q for one radial index: q3[l] (l < l3), then 4-body, then 5-body (nq outputs).
// The 4/5-body terms need l3 = 4, so their slots are q[4] and q[5]. Every index
// below is a compile-time constant once unrolled, keeping s, q and D in registers.
constexpr int LSTART[5] = {0, 3, 8, 15, 24};
template <typename T, typename S>
__device__ __forceinline__ int q_of_s(const S s[NLM], int l3, int l4, int l5, S q[6]) {
#pragma unroll
    for (int l = 0; l < 4; l++) {
        S acc(T(0));
#pragma unroll
        for (int m = LSTART[l]; m < LSTART[l + 1]; m++) acc = acc + T(kC3B[m]) * (s[m] * s[m]);
        q[l] = acc;
    }
    if (l4 > 0) {
        q[4] = T(kC4B[0]) * (s[3] * s[3] * s[3]) + T(kC4B[1]) * (s[3] * (s[4] * s[4] + s[5] * s[5])) +
                  T(kC4B[2]) * (s[3] * (s[6] * s[6] + s[7] * s[7])) + T(kC4B[3]) * (s[6] * (s[5] * s[5] - s[4] * s[4])) +
                  T(kC4B[4]) * (s[4] * s[5] * s[7]);
    }
    if (l5 > 0) {
        const S s0 = s[0] * s[0], s12 = s[1] * s[1] + s[2] * s[2];
        q[5] = T(kC5B[0]) * (s0 * s0) + T(kC5B[1]) * (s0 * s12) + T(kC5B[2]) * (s12 * s12);
    }
    return l3 + (l4 > 0) + (l5 > 0);
}

// D[m] = sum_F gq[F] dq_F/ds_m (gq in q_of_s order).
template <typename T, typename S>
__device__ __forceinline__ void dq_ds(const S s[NLM], const T *gq, int l3, int l4, int l5, S D[NLM]) {
#pragma unroll
    for (int m = 0; m < NLM; m++) D[m] = S(T(0));
#pragma unroll
    for (int l = 0; l < 4; l++)
        if (l < l3)
#pragma unroll
            for (int m = LSTART[l]; m < LSTART[l + 1]; m++) D[m] = D[m] + (T(2) * T(kC3B[m]) * gq[l]) * s[m];
    if (l4 > 0) {
        const T g = gq[4];
        const T c0 = T(kC4B[0]), c1 = T(kC4B[1]), c2 = T(kC4B[2]), c3 = T(kC4B[3]), c4 = T(kC4B[4]);
        D[3] = D[3] + g * (T(3) * c0 * (s[3] * s[3]) + c1 * (s[4] * s[4] + s[5] * s[5]) + c2 * (s[6] * s[6] + s[7] * s[7]));
        D[4] = D[4] + g * (T(2) * c1 * (s[3] * s[4]) - T(2) * c3 * (s[6] * s[4]) + c4 * (s[5] * s[7]));
        D[5] = D[5] + g * (T(2) * c1 * (s[3] * s[5]) + T(2) * c3 * (s[6] * s[5]) + c4 * (s[4] * s[7]));
        D[6] = D[6] + g * (T(2) * c2 * (s[3] * s[6]) + c3 * (s[5] * s[5] - s[4] * s[4]));
        D[7] = D[7] + g * (T(2) * c2 * (s[3] * s[7]) + c4 * (s[4] * s[5]));
    }
    if (l5 > 0) {
        const T g = gq[5];
        const T c0 = T(kC5B[0]), c1 = T(kC5B[1]), c2 = T(kC5B[2]);
        const S s12 = s[1] * s[1] + s[2] * s[2];
        D[0] = D[0] + g * (T(4) * c0 * (s[0] * s[0] * s[0]) + T(2) * c1 * (s[0] * s12));
        D[1] = D[1] + g * (T(2) * c1 * (s[0] * s[0] * s[1]) + T(4) * c2 * (s12 * s[1]));
        D[2] = D[2] + g * (T(2) * c1 * (s[0] * s[0] * s[2]) + T(4) * c2 * (s12 * s[2]));
    }
}

// position of feature (group f, radial index n) in the angular feature vector
__device__ __forceinline__ int aidx(int f, int n, int na) { return f * na + n; }

// ------------------------------------------------------------------ shared pieces
struct FeatArgs {
    const void *c;          // [T][T][nm][nb]
    const void *Ri;         // [N][S][4]
    const int64_t *NL;      // [N][S]
    const int64_t *atom_map;
    void *feats;            // [N][ld] (written at column offset col0)
    void *save;             // angular: [N][nm][24] sums s; radial: [N][T][nb] basis sums F (may be null in mode 0)
    const void *gfeat;      // [N][ld] upstream gradient of feats
    const void *gs;         // angular coefficient gradient: [N][nm][24] upstream gradient of s (may be null)
    const void *gg;         // [N][S][4] upstream gradient of the position gradient (2nd order)
    void *gRi;              // [N][S][4] out
    void *gc;               // [T][T][nm][nb] out (accumulated)
    void *ggfeat;           // [N][ld] out (2nd order)
    void *gsave;            // angular 2nd order: [N][nm][24] gradient of s out (null: its coefficient gradient is taken here)
    const void *gF, *gV;    // 2nd order without gg: upstream gradients of the forces [N][3] and frame virials [F][9]
    const int32_t *atom_frame;
    int64_t N;
    int pw;                 // coefficient-gradient tables per wavefront (plain adds) instead of per block (LDS atomics)
    int S, T, nm, nb, ld, col0, l3, l4, l5;
    double rc;
};

// Rows of four values at the element type's own alignment.
template <typename T>
struct __attribute__((packed, aligned(sizeof(T)))) Row4 {
    T v[4];
};

template <typename T>
__device__ __forceinline__ Row4<T> load4(const T *p) { return *reinterpret_cast<const Row4<T> *>(p); }
template <typename T>
__device__ __forceinline__ void store4(T *p, T a, T b, T c, T d) {
    *reinterpret_cast<Row4<T> *>(p) = Row4<T>{{a, b, c, d}};
}

// The second-order pass's gg of slot s (atom i -> j, row er = [r, x, y, z]): read, or formed from the upstream
// gradients of the model's forces F and frame virials V (either may be null). With f(s) = dE[s][0] u +
// dE[s][1:4], F[j] -= f, F[i] += f and V -= f (x) x, so dL/df = q = gF[i] - gF[j] - gV x and gg = [q . u, q].
template <typename T>
__device__ __forceinline__ Row4<T> slot_gg(const FeatArgs &a, int64_t s, int64_t i, int64_t j, const Row4<T> &er) {
    if (a.gg) return load4(reinterpret_cast<const T *>(a.gg) + s * 4);
    Row4<T> g{{T(0), T(0), T(0), T(0)}};
    if (fabs(er.v[0]) > T(1e-5)) {
        const T *gF = reinterpret_cast<const T *>(a.gF), *gV = reinterpret_cast<const T *>(a.gV);
        T q[3] = {T(0), T(0), T(0)};
        if (gF) {
#pragma unroll
            for (int x = 0; x < 3; x++) q[x] = gF[3 * i + x] - gF[3 * j + x];
        }
        if (gV) {
            const T *v = gV + 9 * (int64_t)a.atom_frame[i];
#pragma unroll
            for (int x = 0; x < 3; x++) q[x] -= v[3 * x] * er.v[1] + v[3 * x + 1] * er.v[2] + v[3 * x + 2] * er.v[3];
        }
        const T ir = T(1) / er.v[0];
        g = Row4<T>{{(q[0] * er.v[1] + q[1] * er.v[2] + q[2] * er.v[3]) * ir, q[0], q[1], q[2]}};
    }
    return g;
}

// NL rows are a valid prefix followed by -1: its length, for rows whose first 64 entries are all valid.
__device__ __forceinline__ int slot_count(const int64_t *NL, int64_t i, int S) {
    int lo = 0, hi = S;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (NL[i * S + mid] >= 0) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// The block's coefficient-gradient tables (ntab of count entries: one per wavefront, or one shared)
// summed and added to global memory, one atomic per entry.
template <typename T>
__device__ __forceinline__ void block_flush_add(T *lds, T *glob, int count, int ntab) {
    __syncthreads();
    for (int x = threadIdx.x; x < count; x += blockDim.x) {
        T v = lds[x];
        for (int w = 1; w < ntab; w++) v += lds[w * count + x];
        if (v != T(0)) atomic_add(glob + x, v);
    }
}

template <typename T>
__device__ __forceinline__ void tab_add(T *p, T v, bool own) {
    if (own) *p += v;
    else atomicAdd(p, v);
}

// Positions of the live lanes sorted by their type (stable): pos of this lane; lane t returns in `start`
// the first position of type t (lane T: the total).
__device__ __forceinline__ int sort_by_type(bool live, int tj, int T, int lane, int &start) {
    const uint64_t below = (1ull << lane) - 1ull;
    int pos = 0, base = 0;
    start = 0;
    for (int t = 0; t < T; t++) {
        const bool mine = live && tj == t;
        const uint64_t m = __ballot(mine);
        if (mine) pos = base + __popcll(m & below);
        if (lane == t) start = base;
        base += __popcll(m);
    }
    if (lane == T) start = base;
    return pos;
}

// ------------------------------------------------------------------ radial kernels
// One wavefront per atom, lanes over slots. WHAT is a set of:
constexpr int R_FEAT = 1;      // feats (and the basis sums F into save, if given)
constexpr int R_1ST = 2;       // first derivatives: gRi, and gc from F summed here
constexpr int R_GCF = 8;       // gc from the F of an earlier pass (save): no slots are read
constexpr int R_2ND = 16;      // ggfeat and gc of the second-order pass (V[t][k] = sum gg f'_k in F's place)
// A slot's basis values go to its row in LDS, at its position sorted by neighbor type; lanes over (type, k)
// then add only their own type's rows. What bounds it: the LDS reads of that sum and, with few atoms, the
// chain list -> type -> basis -> sum. Measured on the 62,713-atom four-type float batch, against nm nb
// multiply-adds a slot with gathered coefficients and a scan of all rows per (type, k): features 190 -> 57 us,
// gRi and gc 357 -> 105, second order 373 -> 109; 1,728 atoms, gRi and gc: 32 -> 15, features 16 -> 8.
constexpr int RAD_WAVES = 4;
constexpr int NPASS = (NT_MAX * NB_MAX + WAVE - 1) / WAVE;   // (type, k) pairs per lane at most

template <int NBC>
__host__ __device__ constexpr int rad_stride(int nb) { return (NBC ? NBC : nb) | 1; }

template <typename T, int NMC, int NBC, int WHAT>
__global__ void __launch_bounds__(RAD_WAVES * WAVE)
nep_radial_kernel(FeatArgs a) {
    extern __shared__ unsigned char smem_raw[];
    constexpr bool TAB = (WHAT & (R_1ST | R_GCF | R_2ND)) != 0, SUM = (WHAT & (R_FEAT | R_1ST | R_2ND)) != 0;
    constexpr bool GRAD = (WHAT & ~R_FEAT) != 0;
    const int nm = NMC ? NMC : a.nm, nb = NBC ? NBC : a.nb;
    const int lane = threadIdx.x & (WAVE - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int ncoef = a.T * a.T * nm * nb, tb = a.T * nb, st = rad_stride<NBC>(nb);
    const int waves = blockDim.x / WAVE, ntab = TAB ? (a.pw ? waves : 1) : 0;
    T *gcl = reinterpret_cast<T *>(smem_raw);
    T *gtab = gcl + (ntab > 1 ? wid : 0) * ncoef;
    T *rows = gcl + (size_t)ntab * ncoef + (size_t)wid * WAVE * st;                               // SUM
    T *wt = gcl + (size_t)ntab * ncoef + (SUM ? (size_t)waves * WAVE * st : 0) + (size_t)wid * tb;   // R_1ST
    if constexpr (TAB) {
        for (int x = threadIdx.x; x < ntab * ncoef; x += blockDim.x) gcl[x] = T(0);
        __syncthreads();
    }
    const T *c = reinterpret_cast<const T *>(a.c);
    const T *Ri = reinterpret_cast<const T *>(a.Ri);
    for (int64_t i = (int64_t)blockIdx.x * waves + wid; i < a.N; i += (int64_t)gridDim.x * waves) {
        const int ti = (int)a.atom_map[i];
        const T *ci = c + (int64_t)ti * a.T * nm * nb;
        T g[NM_MAX];
        if constexpr (GRAD) {
#pragma unroll
            for (int n = 0; n < NM_MAX; n++)
                g[n] = n < nm ? reinterpret_cast<const T *>(a.gfeat)[i * a.ld + a.col0 + n] : T(0);
        }
        T acc[NPASS];
#pragma unroll
        for (int p = 0; p < NPASS; p++) acc[p] = T(0);
        if constexpr ((WHAT & R_1ST) != 0) {
            // w[t][k] = sum_n g_n c[ti][t][n][k]
            for (int o = lane; o < tb; o += WAVE) {
                const int t = o / nb, q = o - t * nb;
                T w = T(0);
#pragma unroll
                for (int n = 0; n < NM_MAX; n++)
                    if (n < nm) w += g[n] * ci[(t * nm + n) * nb + q];
                wt[o] = w;
            }
            wave_sync();
        }
        if constexpr (WHAT == R_GCF) {
#pragma unroll
            for (int p = 0; p < NPASS; p++)
                if (lane + p * WAVE < tb) acc[p] = reinterpret_cast<const T *>(a.save)[i * tb + lane + p * WAVE];
        } else {
            for (int k0 = 0; k0 < a.S; k0 += WAVE) {
                const int k = k0 + lane;
                const int64_t s = i * a.S + k;
                const int64_t j = k < a.S ? a.NL[s] : -1;
                const uint64_t end = __ballot(j < 0);
                const bool live = lane < (end ? __builtin_ctzll(end) : WAVE);
                const int tj = live ? (int)a.atom_map[j] : 0;
                int start = 0, pos = 0;
                if constexpr (SUM) pos = sort_by_type(live, tj, a.T, lane, start);
                if (live) {
                    T gg = T(0);
                    if constexpr ((WHAT & R_2ND) != 0) gg = slot_gg<T>(a, s, i, j, load4(Ri + s * 4)).v[0];
                    Basis<T> bs(Ri[s * 4], (T)a.rc);
                    T d = T(0);
                    T *row = rows + pos * st;
                    const T *w = wt + tj * nb;
#pragma unroll
                    for (int q = 0; q < (NBC ? NBC : NB_MAX); q++) {
                        if (NBC == 0 && q >= nb) continue;
                        if constexpr ((WHAT & (R_FEAT | R_1ST)) != 0) row[q] = bs.value();
                        if constexpr ((WHAT & R_2ND) != 0) row[q] = gg * bs.slope();
                        if constexpr ((WHAT & R_1ST) != 0) d += w[q] * bs.slope();
                        bs.step();
                    }
                    if constexpr ((WHAT & R_1ST) != 0) store4<T>(reinterpret_cast<T *>(a.gRi) + s * 4, d, T(0), T(0), T(0));
                } else if constexpr ((WHAT & R_1ST) != 0) {
                    if (k < a.S) store4<T>(reinterpret_cast<T *>(a.gRi) + s * 4, T(0), T(0), T(0), T(0));
                }
                if constexpr (SUM) {
                    wave_sync();
#pragma unroll
                    for (int p = 0; p < NPASS; p++) {
                        if (p * WAVE >= tb) break;
                        const int o = lane + p * WAVE, t = o < tb ? o / nb : 0, q = o - t * nb;
                        const int s0 = __shfl(start, t, WAVE), s1 = __shfl(start, t + 1, WAVE);
                        if (o < tb)
                            for (int x = s0; x < s1; x++) acc[p] += rows[x * st + q];
                    }
                    wave_sync();
                }
                if (end) {
                    if constexpr ((WHAT & R_1ST) != 0)
                        for (int kk = k + WAVE; kk < a.S; kk += WAVE)
                            store4<T>(reinterpret_cast<T *>(a.gRi) + (i * a.S + kk) * 4, T(0), T(0), T(0), T(0));
                    break;
                }
            }
        }
        if constexpr ((WHAT & (R_FEAT | R_2ND)) != 0) {
            // q_n (or its directional derivative): sum over (t, k) of c times the sums
            T v[NM_MAX];
#pragma unroll
            for (int n = 0; n < NM_MAX; n++) v[n] = T(0);
#pragma unroll
            for (int p = 0; p < NPASS; p++) {
                const int o = lane + p * WAVE;
                if (o < tb) {
                    const int t = o / nb, q = o - t * nb;
#pragma unroll
                    for (int n = 0; n < NM_MAX; n++)
                        if (n < nm) v[n] += ci[(t * nm + n) * nb + q] * acc[p];
                }
            }
            T out = T(0);
#pragma unroll
            for (int n = 0; n < NM_MAX; n++)
                if (n < nm) {
                    const T x = wave_sum(v[n]);
                    if (lane == n) out = x;
                }
            T *o = reinterpret_cast<T *>((WHAT & R_FEAT) ? a.feats : a.ggfeat);
            if (lane < nm) o[i * a.ld + a.col0 + lane] = out;
        }
        if constexpr ((WHAT & R_FEAT) != 0) {
            if (a.save) {
#pragma unroll
                for (int p = 0; p < NPASS; p++)
                    if (lane + p * WAVE < tb) reinterpret_cast<T *>(a.save)[i * tb + lane + p * WAVE] = acc[p];
            }
        }
        if constexpr (TAB) {
            // dc[ti][t][n][k] += g_n F[t][k]: lanes own distinct (t, k)
#pragma unroll
            for (int p = 0; p < NPASS; p++) {
                const int o = lane + p * WAVE;
                if (o < tb && acc[p] != T(0)) {
                    const int t = o / nb, q = o - t * nb;
                    T *e = gtab + (ti * a.T + t) * nm * nb + q;
#pragma unroll
                    for (int n = 0; n < NM_MAX; n++)
                        if (n < nm) tab_add(e + n * nb, g[n] * acc[p], ntab > 1);
                }
            }
        }
    }
    if constexpr (TAB) block_flush_add(gcl, reinterpret_cast<T *>(a.gc), ncoef, ntab);
}

// ------------------------------------------------------------------ angular: matrix-core pieces
// What bounds the angular kernels: VALU work per slot (basis, harmonics, the D contractions) and the LDS
// traffic of the slot sums, which as lanes over outputs read every row from every lane and, for dc, read and
// wrote a table entry per slot; as 16x16x4 products each row is read once per 16 outputs and the table once per
// type and batch. Same batch, float: features 136 -> 63 us, first derivative 375 -> 129, second order 1020 -> 357
// with its coefficient gradient, 263 without (the first derivative's pass, 143, then forms both); double on 16
// frames: 65 -> 31, 96 -> 44, 264 -> 183 (142). The second order in double holds 256 VGPRs and 58 AGPRs (104 at
// the general sizes), which is one wavefront per SIMD.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Acc;
template <> struct Acc<float> { typedef f32x4 type; };
template <> struct Acc<double> { typedef f64x4 type; };

// D[16][16] += A[16][4] B[4][16]: lane l gives A[l % 16][l / 16] and B[l / 16][l % 16]; register r of lane l
// holds D[acc_row(l, r)][l % 16].
__device__ __forceinline__ f32x4 mm4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f64x4 mm4(double a, double b, f64x4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
template <typename T>
__device__ __forceinline__ int acc_row(int lane, int r) {
    return sizeof(T) == 4 ? 4 * (lane >> 4) + r : 4 * r + (lane >> 4);
}

// Up to AB consecutive atoms of one type whose slots fit one chunk of CH lanes (the first atom alone may
// have more: several chunks). off: first slot of each atom in the batch.
constexpr int ANG_AB = 4;
template <int AB>
struct Batch {
    int off[AB + 1], na, tot, ti;
    __device__ __forceinline__ int atom(int e) const {
        int q = 0;
#pragma unroll
        for (int x = 1; x < AB; x++) q += (x < na && e >= off[x]) ? 1 : 0;
        return q;
    }
    // off[q] of a lane's own q (selects: an indexed read would go through scratch)
    __device__ __forceinline__ int first(int q) const {
        int f = 0;
#pragma unroll
        for (int x = 1; x < AB; x++) f = q == x ? off[x] : f;
        return f;
    }
};

template <int AB, int CH>
__device__ __forceinline__ Batch<AB> next_batch(const FeatArgs &a, int64_t i, int64_t i1, int lane) {
    Batch<AB> b;
    int64_t j[AB];
    int t[AB];
#pragma unroll
    for (int q = 0; q < AB; q++) {
        j[q] = (i + q < i1 && lane < a.S) ? a.NL[(i + q) * a.S + lane] : -1;
        t[q] = i + q < i1 ? (int)a.atom_map[i + q] : -1;
    }
    b.off[0] = 0;
    b.na = 0;
    b.ti = t[0];
    bool open = true;
#pragma unroll
    for (int q = 0; q < AB; q++) {
        const uint64_t end = __ballot(j[q] < 0);
        int c = end ? __builtin_ctzll(end) : WAVE;
        if (!end && a.S > WAVE) c = slot_count(a.NL, i + q, a.S);
        open = open && (q == 0 || (i + q < i1 && t[q] == b.ti && b.off[q] + c <= CH));
        if (open) b.na = q + 1;
        b.off[q + 1] = b.off[q] + (open ? c : 0);
    }
    b.tot = b.off[AB];
    return b;
}

// This wavefront's contiguous range of atoms.
__device__ __forceinline__ void atom_range(int64_t N, int wid, int64_t &i0, int64_t &i1) {
    const int waves = blockDim.x / WAVE;
    const int64_t nw = (int64_t)gridDim.x * waves, gw = (int64_t)blockIdx.x * waves + wid;
    i0 = N * gw / nw;
    i1 = N * (gw + 1) / nw;
}

// acc[n][m] += sum over rows [k0, k1) and the NTERM terms of u[row][term][n] w[row][term][m] (m < 24: two
// column tiles); rows of `st` values, u at uo (nm per term), w at wo (24 per term).
template <typename T, int NTERM>
__device__ __forceinline__ void sum_nm(const T *rows, int st, int uo, int wo, int nm, int k0, int k1, int lane,
                                       typename Acc<T>::type acc[2]) {
    const int x = lane & 15, h = lane >> 4;
    for (int s = k0; s < k1; s += 4) {
        const bool live = s + h < k1;
        const T *row = rows + (live ? s + h : k1 - 1) * st;
#pragma unroll
        for (int t = 0; t < NTERM; t++) {
            const T av = (live && x < nm) ? row[uo + t * nm + (x < nm ? x : 0)] : T(0);
            const T b0 = row[wo + t * NLM + x], b1 = x < NLM - 16 ? row[wo + t * NLM + 16 + (x & 7)] : T(0);
            acc[0] = mm4(av, b0, acc[0]);
            acc[1] = mm4(av, b1, acc[1]);
        }
    }
}

// dst[n][m] (nm x 24) from sum_nm's accumulators.
template <typename T, typename Fn>
__device__ __forceinline__ void each_nm(const typename Acc<T>::type acc[2], int nm, int lane, Fn &&fn) {
    const int x = lane & 15;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int n = acc_row<T>(lane, r);
        if (n < nm) {
            fn(n * NLM + x, acc[0][r]);
            if (x < NLM - 16) fn(n * NLM + 16 + x, acc[1][r]);
        }
    }
}

// Coefficient gradient of one batch: tab[t][n][q] += sum over type t's rows and the NTERM terms of
// z[row][term][n] v[row][term][q], rows sorted by type (lane t holds type t's first row in `start`).
template <typename T, int NTERM>
__device__ __forceinline__ void add_dc(const T *rows, int st, int zo, int vo, int nm, int nb, int ntypes, int start,
                                       T *tab, bool own, int lane) {
    typedef typename Acc<T>::type A4;
    const int x = lane & 15, h = lane >> 4;
    for (int t = 0; t < ntypes; t++) {
        const int k0 = __builtin_amdgcn_readlane(start, t), k1 = __builtin_amdgcn_readlane(start, t + 1);
        if (k0 == k1) continue;
        for (int q0 = 0; q0 < nb; q0 += 16) {
            const int q = q0 + x;
            A4 acc = {T(0), T(0), T(0), T(0)};
            for (int s = k0; s < k1; s += 4) {
                const bool live = s + h < k1;
                const T *row = rows + (live ? s + h : k1 - 1) * st;
#pragma unroll
                for (int u = 0; u < NTERM; u++) {
                    const T av = (live && x < nm) ? row[zo + u * nm + (x < nm ? x : 0)] : T(0);
                    const T bv = q < nb ? row[vo + u * nb + (q < nb ? q : 0)] : T(0);
                    acc = mm4(av, bv, acc);
                }
            }
            if (q < nb) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int n = acc_row<T>(lane, r);
                    if (n < nm) tab_add(tab + (t * nm + n) * nb + q, acc[r], own);
                }
            }
        }
    }
}

// D = dE/ds of every (atom, n) of a batch into Bq [AB][nm][24] (lanes over (atom, n)), plus gs if given.
template <typename T, int AB>
__device__ __forceinline__ void batch_dq(const FeatArgs &a, const Batch<AB> &b, int64_t i, int nm, int lane, T *Bq,
                                         const T *gs) {
    if (lane >= b.na * nm) return;
    const int q = lane / nm, n = lane - q * nm, nf = a.l3 + (a.l4 > 0) + (a.l5 > 0);
    const int64_t ia = i + q;
    const T *gfe = reinterpret_cast<const T *>(a.gfeat);
    T gq[6];
#pragma unroll
    for (int f = 0; f < 6; f++) gq[f] = (gfe && f < nf) ? gfe[ia * a.ld + a.col0 + aidx(f, n, nm)] : T(0);
    T D[NLM];
    dq_ds<T, T>(reinterpret_cast<const T *>(a.save) + (ia * nm + n) * NLM, gq, a.l3, a.l4, a.l5, D);
#pragma unroll
    for (int m = 0; m < NLM; m++) Bq[(q * nm + n) * NLM + m] = gs ? D[m] + gs[(ia * nm + n) * NLM + m] : D[m];
}

// g_n and, with SLOPE, g'_n of one slot from its coefficient rows, the basis values (and slopes) handed to
// fn(q, f, f').
template <typename T, int NMC, int NBC, bool SLOPE, typename Fn>
__device__ __forceinline__ void radial_fn(const T *cij, T r, T rc, int nm, int nb, T gn[NM_MAX], T gp[NM_MAX], Fn &&fn) {
    Basis<T> bs(r, rc);
#pragma unroll
    for (int n = 0; n < NM_MAX; n++) { gn[n] = T(0); gp[n] = T(0); }
#pragma unroll
    for (int q = 0; q < (NBC ? NBC : NB_MAX); q++) {
        if (NBC == 0 && q >= nb) continue;
        const T f = bs.value(), fp = SLOPE ? bs.slope() : T(0);
#pragma unroll
        for (int n = 0; n < (NMC ? NMC : NM_MAX); n++)
            if (n < nm) {
                const T cv = cij[n * nb + q];
                gn[n] += cv * f;
                if constexpr (SLOPE) gp[n] += cv * fp;
            }
        fn(q, f, fp);
        bs.step();
    }
}

// The first derivative of one angular slot: (D b)_n for every n and, with GRI, dE/d[r, x, y, z]; B the atom's D
// rows [nm][24], u the slot's unit vector. With (D b)_n at hand the radial part of dE/dr is sum_n g'_n (D b)_n.
template <typename T, int NMC, bool GRI>
__device__ __forceinline__ void angular_slot(const T *B, int nm, T ux, T uy, T uz, T ir, const T gn[NM_MAX],
                                             const T gp[NM_MAX], T Db[NM_MAX], T d[4]) {
    T bm[NLM], Dg[NLM];
    blm_each<T>(ux, uy, uz, [&](int m, T bv, T, T, T) { bm[m] = bv; Dg[m] = T(0); });
#pragma unroll
    for (int n = 0; n < (NMC ? NMC : NM_MAX); n++) {
        Db[n] = T(0);
        if (n < nm) {
#pragma unroll
            for (int m = 0; m < NLM; m++) {
                const T Bv = B[n * NLM + m];
                Db[n] += Bv * bm[m];
                if constexpr (GRI) Dg[m] += Bv * gn[n];
            }
        }
    }
    if constexpr (GRI) {
        T gr = T(0), V0 = T(0), V1 = T(0), V2 = T(0);
#pragma unroll
        for (int n = 0; n < (NMC ? NMC : NM_MAX); n++)
            if (n < nm) gr += gp[n] * Db[n];
        blm_each<T>(ux, uy, uz, [&](int m, T, T d0, T d1, T d2) {
            V0 += Dg[m] * d0; V1 += Dg[m] * d1; V2 += Dg[m] * d2;
        });
        d[0] = gr - (ux * V0 + uy * V1 + uz * V2) * ir;
        d[1] = V0 * ir; d[2] = V1 * ir; d[3] = V2 * ir;
    }
}

// ------------------------------------------------------------------ angular features (mode 0)
constexpr int ANG_WAVES = 2;     // wavefronts per angular block (LDS per wave is large)

__host__ __device__ inline int angf_wave_elems(int nm) { return ANG_AB * nm * NLM + WAVE * ((nm + NLM) | 1); }

template <typename T, int NMC, int NBC>
__global__ void __launch_bounds__(ANG_WAVES * WAVE)
nep_angular_fwd_kernel(FeatArgs a) {
    extern __shared__ unsigned char smem_raw[];
    typedef typename Acc<T>::type A4;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int nm = NMC ? NMC : a.nm, nb = NBC ? NBC : a.nb, per = nm * NLM, st = (nm + NLM) | 1;
    T *Sq = reinterpret_cast<T *>(smem_raw) + (size_t)wid * angf_wave_elems(nm);   // [AB][nm][24]
    T *rows = Sq + ANG_AB * per;                                                     // [WAVE][st]: g_n, b_m
    const T *c = reinterpret_cast<const T *>(a.c);
    const T *Ri = reinterpret_cast<const T *>(a.Ri);
    T *fo = reinterpret_cast<T *>(a.feats);
    T *so = reinterpret_cast<T *>(a.save);
    int64_t i, i1;
    atom_range(a.N, wid, i, i1);
    while (i < i1) {
        const Batch<ANG_AB> b = next_batch<ANG_AB, WAVE>(a, i, i1, lane);
        A4 acc[ANG_AB][2];
#pragma unroll
        for (int q = 0; q < ANG_AB; q++)
#pragma unroll
            for (int u = 0; u < 2; u++) acc[q][u] = A4{T(0), T(0), T(0), T(0)};
        for (int e0 = 0; e0 < b.tot; e0 += WAVE) {
            const int nk = b.tot - e0 < WAVE ? b.tot - e0 : WAVE;
            if (lane < nk) {
                const int e = e0 + lane, q = b.atom(e);
                const int64_t s = (i + q) * a.S + (e - b.first(q));
                const int tj = (int)a.atom_map[a.NL[s]];
                const Row4<T> er = load4(Ri + s * 4);
                const T ir = T(1) / er.v[0];
                T gn[NM_MAX], gp[NM_MAX];
                T *row = rows + lane * st;
                radial_fn<T, NMC, NBC, false>(c + (int64_t)(b.ti * a.T + tj) * nm * nb, er.v[0], (T)a.rc, nm, nb, gn,
                                              gp, [](int, T, T) {});
#pragma unroll
                for (int n = 0; n < (NMC ? NMC : NM_MAX); n++)
                    if (n < nm) row[n] = gn[n];
                blm_each<T>(er.v[1] * ir, er.v[2] * ir, er.v[3] * ir, [&](int m, T bv, T, T, T) { row[nm + m] = bv; });
            }
            wave_sync();
#pragma unroll
            for (int q = 0; q < ANG_AB; q++) {
                if (q >= b.na) continue;
                const int k0 = b.off[q] - e0 > 0 ? b.off[q] - e0 : 0;
                const int k1 = b.off[q + 1] - e0 < nk ? b.off[q + 1] - e0 : nk;
                sum_nm<T, 1>(rows, st, 0, nm, nm, k0, k1, lane, acc[q]);
            }
            wave_sync();
        }
#pragma unroll
        for (int q = 0; q < ANG_AB; q++) {
            if (q < b.na) each_nm<T>(acc[q], nm, lane, [&](int o, T v) {
                Sq[q * per + o] = v;
                so[(i + q) * per + o] = v;
            });
        }
        wave_sync();
        if (lane < b.na * nm) {
            const int q = lane / nm, n = lane - q * nm;
            T qv[6];
            const int nq = q_of_s<T, T>(Sq + q * per + n * NLM, a.l3, a.l4, a.l5, qv);
#pragma unroll
            for (int f = 0; f < 6; f++)
                if (f < nq) fo[(i + q) * a.ld + a.col0 + aidx(f, n, nm)] = qv[f];
        }
        wave_sync();
        i += b.na;
    }
}

// ------------------------------------------------------------------ angular first derivative
// dc[ti][tj][n][q] = f_q (D b)_n, and with GRI gRi = sum_nm D_nm d(g_n b_m)/dRi of every slot (mode 1 of
// matpl_nep_feat; without, the coefficient gradient of a training step with gs, the second-order pass's gradient
// of s, added to D).
__host__ __device__ inline int angb_wave_elems(int nm, int nb) { return ANG_AB * nm * NLM + WAVE * ((nm + nb) | 1); }

template <typename T, int NMC, int NBC, bool GRI>
__global__ void __launch_bounds__(ANG_WAVES * WAVE)
nep_angular_bwd_kernel(FeatArgs a) {
    extern __shared__ unsigned char smem_raw[];
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int nm = NMC ? NMC : a.nm, nb = NBC ? NBC : a.nb, per = nm * NLM, st = (nm + nb) | 1;
    const int ncoef = a.T * a.T * nm * nb;
    const int waves = blockDim.x / WAVE, ntab = a.pw ? waves : 1;
    // the D rows first: their 16-byte alignment lets a slot read them four or two values at a time
    T *Bq = reinterpret_cast<T *>(smem_raw) + (size_t)wid * ANG_AB * per;                   // [AB][nm][24]
    T *rows = reinterpret_cast<T *>(smem_raw) + (size_t)waves * ANG_AB * per + (size_t)wid * WAVE * st;
    T *gcl = reinterpret_cast<T *>(smem_raw) + (size_t)waves * angb_wave_elems(nm, nb);   // [ntab][ncoef]
    T *gtab = gcl + (ntab > 1 ? wid : 0) * ncoef;
    for (int x = threadIdx.x; x < ntab * ncoef; x += blockDim.x) gcl[x] = T(0);
    __syncthreads();
    const T *c = reinterpret_cast<const T *>(a.c);
    const T *Ri = reinterpret_cast<const T *>(a.Ri);
    T *gRiA = reinterpret_cast<T *>(a.gRi);
    int64_t i, i1;
    atom_range(a.N, wid, i, i1);
    while (i < i1) {
        const Batch<ANG_AB> b = next_batch<ANG_AB, WAVE>(a, i, i1, lane);
        if constexpr (GRI) {
            // unused slots of each atom
#pragma unroll
            for (int q = 0; q < ANG_AB; q++)
                if (q < b.na)
                    for (int k = b.off[q + 1] - b.off[q] + lane; k < a.S; k += WAVE)
                        store4<T>(gRiA + ((i + q) * a.S + k) * 4, T(0), T(0), T(0), T(0));
        }
        batch_dq<T, ANG_AB>(a, b, i, nm, lane, Bq, GRI ? nullptr : reinterpret_cast<const T *>(a.gs));
        wave_sync();
        for (int e0 = 0; e0 < b.tot; e0 += WAVE) {
            const int nk = b.tot - e0 < WAVE ? b.tot - e0 : WAVE;
            const bool live = lane < nk;
            const int e = e0 + (live ? lane : 0), q = b.atom(e);
            const int64_t s = (i + q) * a.S + (e - b.first(q));
            const int tj = (int)a.atom_map[a.NL[s]];
            int start;
            const int pos = sort_by_type(live, tj, a.T, lane, start);
            if (live) {
                const Row4<T> er = load4(Ri + s * 4);
                const T ir = T(1) / er.v[0];
                const T ux = er.v[1] * ir, uy = er.v[2] * ir, uz = er.v[3] * ir;
                T *row = rows + pos * st;
                T gn[NM_MAX], gp[NM_MAX];
                if constexpr (GRI) {
                    radial_fn<T, NMC, NBC, true>(c + (int64_t)(b.ti * a.T + tj) * nm * nb, er.v[0], (T)a.rc, nm, nb,
                                                 gn, gp, [&](int qb, T f, T) { row[nm + qb] = f; });
                } else {
                    Basis<T> bs(er.v[0], (T)a.rc);
#pragma unroll
                    for (int qb = 0; qb < (NBC ? NBC : NB_MAX); qb++) {
                        if (NBC == 0 && qb >= nb) continue;
                        row[nm + qb] = bs.value();
                        bs.step();
                    }
                }
                T Db[NM_MAX], d[4];
                angular_slot<T, NMC, GRI>(Bq + q * per, nm, ux, uy, uz, ir, gn, gp, Db, d);
#pragma unroll
                for (int n = 0; n < (NMC ? NMC : NM_MAX); n++)
                    if (n < nm) row[n] = Db[n];
                if constexpr (GRI) store4<T>(gRiA + s * 4, d[0], d[1], d[2], d[3]);
            }
            wave_sync();
            add_dc<T, 1>(rows, st, 0, nm, nm, nb, a.T, start, gtab + b.ti * a.T * nm * nb, ntab > 1, lane);
            wave_sync();
        }
        wave_sync();
        i += b.na;
    }
    block_flush_add(gcl, reinterpret_cast<T *>(a.gc), ncoef, ntab);
}

// ------------------------------------------------------------------ angular second order (mode 2)
// With gg the upstream gradient of gRi, beta_m = gg0 b_m and delta_m = (db_m/du . (gg_xyz - gg0 u)) / r:
//   P_nm = sum_slots g'_n beta_m + g_n delta_m        (the directional derivative of s)
//   ggfeat = J P,  E = H(gfeat) P                     (per atom)
//   dc[ti][tj][n][q] = f'_q (D beta)_n + f_q (D delta)_n, and through s: f_q (E b)_n
// GS: E goes to gsave, the gradient of s, whose coefficient gradient the caller's first-derivative pass adds
// to its own; otherwise a second pass over the slots takes it here. Float takes 64 slots of up to 4 atoms a
// pass, double 32 of up to 2 (its rows are twice as wide in LDS).
template <typename T>
struct Ang2Shape {
    static constexpr int CH = sizeof(T) == 4 ? 64 : 32;
    static constexpr int AB = sizeof(T) == 4 ? 4 : 2;
};

__host__ __device__ inline int ang2_stride(int nm, int nb) {
    const int p = 2 * nm + 2 * NLM, d = 2 * nm + 2 * nb;
    return (p > d ? p : d) | 1;
}

template <typename T>
__host__ __device__ inline int ang2_wave_elems(int nm, int nb) {
    return 2 * Ang2Shape<T>::AB * nm * NLM + Ang2Shape<T>::CH * ang2_stride(nm, nb);
}

template <typename T, int NMC, int NBC, bool GS>
__global__ void __launch_bounds__(ANG_WAVES * WAVE)
nep_angular_bwd2_kernel(FeatArgs a) {
    extern __shared__ unsigned char smem_raw[];
    typedef typename Acc<T>::type A4;
    constexpr int CH = Ang2Shape<T>::CH, AB = Ang2Shape<T>::AB, NBM = NBC ? NBC : NB_MAX, NMM = NMC ? NMC : NM_MAX;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int nm = NMC ? NMC : a.nm, nb = NBC ? NBC : a.nb, per = nm * NLM, st = ang2_stride(nm, nb);
    const int ncoef = a.T * a.T * nm * nb;
    const int waves = blockDim.x / WAVE, ntab = a.pw ? waves : 1;
    T *Bq = reinterpret_cast<T *>(smem_raw) + (size_t)wid * 2 * AB * per;        // [AB][nm][24] D
    T *Cq = Bq + AB * per;                                                      // [AB][nm][24] P, then E
    T *rows = reinterpret_cast<T *>(smem_raw) + (size_t)waves * 2 * AB * per + (size_t)wid * CH * st;
    T *gcl = reinterpret_cast<T *>(smem_raw) + (size_t)waves * ang2_wave_elems<T>(nm, nb);
    T *gtab = gcl + (ntab > 1 ? wid : 0) * ncoef;
    for (int x = threadIdx.x; x < ntab * ncoef; x += blockDim.x) gcl[x] = T(0);
    __syncthreads();
    const T *c = reinterpret_cast<const T *>(a.c);
    const T *Ri = reinterpret_cast<const T *>(a.Ri);
    const T *gfe = reinterpret_cast<const T *>(a.gfeat);
    const T *sv = reinterpret_cast<const T *>(a.save);
    T *go = reinterpret_cast<T *>(a.ggfeat);
    const int nf = a.l3 + (a.l4 > 0) + (a.l5 > 0);
    int64_t i, i1;
    atom_range(a.N, wid, i, i1);
    while (i < i1) {
        const Batch<AB> b = next_batch<AB, CH>(a, i, i1, lane);
        T *tab = gtab + b.ti * a.T * nm * nb;
        batch_dq<T, AB>(a, b, i, nm, lane, Bq, nullptr);
        wave_sync();
        A4 acc[AB][2];
#pragma unroll
        for (int q = 0; q < AB; q++)
#pragma unroll
            for (int u = 0; u < 2; u++) acc[q][u] = A4{T(0), T(0), T(0), T(0)};
        for (int e0 = 0; e0 < b.tot; e0 += CH) {
            const int nk = b.tot - e0 < CH ? b.tot - e0 : CH;
            const bool live = lane < nk;
            const int e = e0 + (live ? lane : 0), q = b.atom(e);
            const int64_t s = (i + q) * a.S + (e - b.first(q));
            const int tj = (int)a.atom_map[a.NL[s]];
            int start;
            const int pos = sort_by_type(live, tj, a.T, lane, start);
            T f[NBM], fp[NBM], zb[NM_MAX], zd[NM_MAX];
            if (live) {
                // rows for P, in the slots' own order: g'_n, g_n | beta_m, delta_m
                const Row4<T> er = load4(Ri + s * 4), gg = slot_gg<T>(a, s, i + q, a.NL[s], er);
                const T ir = T(1) / er.v[0];
                const T ux = er.v[1] * ir, uy = er.v[2] * ir, uz = er.v[3] * ir;
                const T g0 = gg.v[0], gx = (gg.v[1] - g0 * ux) * ir, gy = (gg.v[2] - g0 * uy) * ir,
                        gz = (gg.v[3] - g0 * uz) * ir;
                T gn[NM_MAX], gp[NM_MAX];
                radial_fn<T, NMC, NBC, true>(c + (int64_t)(b.ti * a.T + tj) * nm * nb, er.v[0], (T)a.rc, nm, nb, gn, gp,
                                             [&](int qb, T v, T vp) { f[qb] = v; fp[qb] = vp; });
                T *row = rows + lane * st;
#pragma unroll
                for (int n = 0; n < NMM; n++)
                    if (n < nm) { row[n] = gp[n]; row[nm + n] = gn[n]; }
                const T *B = Bq + q * per;
                T be[NLM], de[NLM];
                blm_each<T>(ux, uy, uz, [&](int m, T bv, T d0, T d1, T d2) {
                    be[m] = g0 * bv;
                    de[m] = d0 * gx + d1 * gy + d2 * gz;
                    row[2 * nm + m] = be[m];
                    row[2 * nm + NLM + m] = de[m];
                });
#pragma unroll
                for (int n = 0; n < NMM; n++) {
                    zb[n] = T(0);
                    zd[n] = T(0);
                    if (n < nm) {
#pragma unroll
                        for (int m = 0; m < NLM; m++) {
                            const T Bv = B[n * NLM + m];
                            zb[n] += Bv * be[m];
                            zd[n] += Bv * de[m];
                        }
                    }
                }
            }
            wave_sync();
#pragma unroll
            for (int x = 0; x < AB; x++) {
                if (x >= b.na) continue;
                const int k0 = b.off[x] - e0 > 0 ? b.off[x] - e0 : 0;
                const int k1 = b.off[x + 1] - e0 < nk ? b.off[x + 1] - e0 : nk;
                sum_nm<T, 2>(rows, st, 0, 2 * nm, nm, k0, k1, lane, acc[x]);
            }
            wave_sync();
            if (live) {
                // rows for dc, sorted by neighbor type: (D beta)_n, (D delta)_n | f'_q, f_q
                T *row = rows + pos * st;
#pragma unroll
                for (int n = 0; n < NMM; n++)
                    if (n < nm) { row[n] = zb[n]; row[nm + n] = zd[n]; }
#pragma unroll
                for (int qb = 0; qb < NBM; qb++)
                    if (qb < nb) { row[2 * nm + qb] = fp[qb]; row[2 * nm + nb + qb] = f[qb]; }
            }
            wave_sync();
            add_dc<T, 2>(rows, st, 0, 2 * nm, nm, nb, a.T, start, tab, ntab > 1, lane);
            wave_sync();
        }
        // per atom: ggfeat = J P (the directional derivative of q along P) and E = H(gfeat) P
#pragma unroll
        for (int q = 0; q < AB; q++) {
            if (q < b.na) each_nm<T>(acc[q], nm, lane, [&](int o, T v) { Cq[q * per + o] = v; });
        }
        wave_sync();
        if (lane < b.na * nm) {
            const int q = lane / nm, n = lane - q * nm;
            const int64_t ia = i + q;
            Dual<T> sd[NLM];
#pragma unroll
            for (int m = 0; m < NLM; m++) sd[m] = Dual<T>(sv[(ia * nm + n) * NLM + m], Cq[(q * nm + n) * NLM + m]);
            Dual<T> qv[6];
            q_of_s<T, Dual<T>>(sd, a.l3, a.l4, a.l5, qv);
            T gq[6];
#pragma unroll
            for (int x = 0; x < 6; x++) {
                gq[x] = x < nf ? gfe[ia * a.ld + a.col0 + aidx(x, n, nm)] : T(0);
                if (x < nf) go[ia * a.ld + a.col0 + aidx(x, n, nm)] = qv[x].e;
            }
            Dual<T> D[NLM];
            dq_ds<T, Dual<T>>(sd, gq, a.l3, a.l4, a.l5, D);
#pragma unroll
            for (int m = 0; m < NLM; m++) {
                if constexpr (GS) reinterpret_cast<T *>(a.gsave)[(ia * nm + n) * NLM + m] = D[m].e;
                else Cq[(q * nm + n) * NLM + m] = D[m].e;
            }
        }
        wave_sync();
        if constexpr (!GS) {
            // the coefficient gradient through s: dc += f_q (E b)_n
            for (int e0 = 0; e0 < b.tot; e0 += CH) {
                const int nk = b.tot - e0 < CH ? b.tot - e0 : CH;
                const bool live = lane < nk;
                const int e = e0 + (live ? lane : 0), q = b.atom(e);
                const int64_t s = (i + q) * a.S + (e - b.first(q));
                const int tj = (int)a.atom_map[a.NL[s]];
                int start;
                const int pos = sort_by_type(live, tj, a.T, lane, start);
                if (live) {
                    const Row4<T> er = load4(Ri + s * 4);
                    const T ir = T(1) / er.v[0];
                    T *row = rows + pos * st;
                    Basis<T> bs(er.v[0], (T)a.rc);
#pragma unroll
                    for (int qb = 0; qb < NBM; qb++) {
                        if (NBC == 0 && qb >= nb) continue;
                        row[nm + qb] = bs.value();
                        bs.step();
                    }
                    T bm[NLM];
                    blm_each<T>(er.v[1] * ir, er.v[2] * ir, er.v[3] * ir, [&](int m, T bv, T, T, T) { bm[m] = bv; });
                    const T *E = Cq + q * per;
#pragma unroll
                    for (int n = 0; n < NMM; n++)
                        if (n < nm) {
                            T Eb = T(0);
#pragma unroll
                            for (int m = 0; m < NLM; m++) Eb += E[n * NLM + m] * bm[m];
                            row[n] = Eb;
                        }
                }
                wave_sync();
                add_dc<T, 1>(rows, st, 0, nm, nm, nb, a.T, start, tab, ntab > 1, lane);
                wave_sync();
            }
        }
        i += b.na;
    }
    block_flush_add(gcl, reinterpret_cast<T *>(a.gc), ncoef, ntab);
}

// ------------------------------------------------------------------ model forces
// F [N][3] and the frame virials V [F][9] of the NEP model straight from dE/dq: the radial and angular slot
// derivatives (nep_radial_kernel R_1ST, nep_angular_bwd_kernel GRI) and the force terms of each slot,
// f = dE[s][0] (x, y, z)/r + dE[s][1:4] (src/model/nep_net.py:440-468 and :608; calculateNepForce,
// CalcOps.cpp:75-158; the frame sum of calculateNepVirial, CalcOps.cpp:239-328), with the model's signs
// (nep_net.py negates both): F[i] += f, F[j] -= f, V[frame] -= f (x) x. No [N][S][4] gradient is written or read.
// A block takes windows of `ch` consecutive atoms, frame by frame (a segment); neighbor terms go to an LDS copy
// of F over the segment's frame (n <= rcap atoms), written once to the segment's row in `part`, since device
// atomics are carried out beyond the per-XCD L2 caches here; nep_force_final_kernel adds the rows. A frame's rows
// (as long as the frame, one per window that it touches, at most force_rows) lie together, from 3 force_rows times
// its first atom on: the buffer grows with the atoms, whatever the sizes of the other frames. The copy is in
// double in both precisions: LDS adds of floats take several times those of doubles here (62,713-atom float
// batch: 276 us with a float copy, 181 with this one; the position gradients, two force kernels and their
// reductions that this kernel stands for took 590 us). Segment
// (window b, frame f) has virial row b + f: consecutive segments advance b or f. Larger frames (rcap = 0), and any
// entry naming an atom of another frame, use global atomics.
struct ForceArgs {
    FeatArgs r, a;                // radial / angular: c, Ri, NL, atom_map, gfeat, save, sizes
    const int64_t *frame_start;   // [F + 1]
    const int32_t *atom_frame;    // [N]
    void *F, *part;               // [N][3] (zeroed), the frames' rows
    double *vpart;                // [segments][9]
    int64_t rcap, rows;           // atoms of the LDS copy, rows kept per frame (force_rows)
    int ch;
};

// Sum over the wavefront of up to 16 values per lane at once: lane l returns the total of v[l % 16]. Each step
// exchanges half of the values still held (17 exchanges, not 6 per value).
template <typename T>
__device__ __forceinline__ T fold16(T v[16], int lane) {
#pragma unroll
    for (int b = 0, n = 8; b < 4; b++, n >>= 1)
#pragma unroll
        for (int k = 0; k < n; k++) {
            const bool hi = (lane >> b) & 1;
            const T keep = hi ? v[2 * k + 1] : v[2 * k], send = hi ? v[2 * k] : v[2 * k + 1];
            v[k] = keep + __shfl_xor(send, 1 << b, WAVE);
        }
    T x = v[0];
    x += __shfl_xor(x, 16, WAVE);
    x += __shfl_xor(x, 32, WAVE);
    return x;
}

// (Atom numbers fit 32 bits wherever they are divided by ch: a grid of a block per window holds fewer.)
// Rows of a frame of at most rcap atoms: the windows of ch that it touches.
inline int64_t force_rows(int64_t rcap, int ch) { return rcap > 0 ? (rcap - 1) / ch + 2 : 0; }

// (153 float and 256 double VGPRs: 3 and 2 wavefronts per SIMD, which blocks of 4 wavefronts fill; of 8, one
// float block fits a CU; in double 4 registers spill, in the general sizes' form 32)
constexpr int FORCE_WAVES = 4;

template <typename T>
inline size_t force_fixed_lds(int T_, int na, int nbr) {
    return (size_t)FORCE_WAVES * (((size_t)ANG_AB * na * NLM + (size_t)T_ * nbr) * sizeof(T) + 9 * sizeof(double));
}

template <typename T, int NMC, int NBC>
__global__ void __launch_bounds__(FORCE_WAVES * WAVE, sizeof(T) == 4 ? 3 : 2)
nep_force_kernel(ForceArgs p) {
    extern __shared__ unsigned char smem_raw[];
    constexpr int W = FORCE_WAVES;
    const FeatArgs &R = p.r, &A = p.a;
    const int lane = threadIdx.x & (WAVE - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int nr = NMC ? NMC : R.nm, nbr = NBC ? NBC : R.nb, na = NMC ? NMC : A.nm, nba = NBC ? NBC : A.nb;
    const int per = A.l3 > 0 ? na * NLM : 0, tb = R.T * nbr;       // as force_fixed_lds counts (na = 0 without angular part)
    double *vred = reinterpret_cast<double *>(smem_raw);                          // [W][9]
    double *acc = vred + W * 9;                                                    // [3 rcap]
    T *wv = reinterpret_cast<T *>(acc + 3 * p.rcap);
    T *Bq = wv + (size_t)wid * ANG_AB * per;                                      // [AB][na][24]
    T *wt = wv + (size_t)W * ANG_AB * per + (size_t)wid * tb;                      // [T][nbr]
    T *F = reinterpret_cast<T *>(p.F);
    const int64_t i0 = (int64_t)blockIdx.x * p.ch, i1 = i0 + p.ch < R.N ? i0 + p.ch : R.N;
    const int f1 = p.atom_frame[i1 - 1];
    for (int f = p.atom_frame[i0]; f <= f1; f++) {
        const int64_t fs = p.frame_start[f], fe = p.frame_start[f + 1];
        const int64_t s0 = i0 > fs ? i0 : fs, s1 = i1 < fe ? i1 : fe;
        if (s0 >= s1) continue;
        const bool lds = fe - fs <= p.rcap;
        if (lds)
            for (int64_t x = threadIdx.x; x < 3 * (fe - fs); x += blockDim.x) acc[x] = 0.0;
        __syncthreads();
        auto add = [&](int64_t j, int c, T v) {
            if (lds && j >= fs && j < fe) atomicAdd(acc + 3 * (j - fs) + c, (double)v);
            else atomic_add(F + 3 * j + c, v);
        };
        T vir[9];
#pragma unroll
        for (int x = 0; x < 9; x++) vir[x] = T(0);
        // radial list: one wavefront per atom, lanes over slots
        const T *Rr = reinterpret_cast<const T *>(R.Ri), *Ra = reinterpret_cast<const T *>(A.Ri);
        for (int64_t i = s0 + wid; i < s1; i += W) {
            const T *ci = reinterpret_cast<const T *>(R.c) + (int64_t)R.atom_map[i] * R.T * nr * nbr;
            const T *gi = reinterpret_cast<const T *>(R.gfeat) + i * R.ld + R.col0;
            for (int o = lane; o < tb; o += WAVE) {
                const int t = o / nbr, q = o - t * nbr;
                T w = T(0);
#pragma unroll
                for (int n = 0; n < (NMC ? NMC : NM_MAX); n++)
                    if (n < nr) w += gi[n] * ci[(t * nr + n) * nbr + q];
                wt[o] = w;
            }
            wave_sync();
            T cen[3] = {T(0), T(0), T(0)};
            for (int k0 = 0; k0 < R.S; k0 += WAVE) {
                const int k = k0 + lane;
                const int64_t s = i * R.S + k;
                const int64_t j = k < R.S ? R.NL[s] : -1;
                const uint64_t end = __ballot(j < 0);
                if (lane < (end ? __builtin_ctzll(end) : WAVE)) {
                    const Row4<T> er = load4(Rr + s * 4);
                    const T *w = wt + (int)R.atom_map[j] * nbr;
                    Basis<T> bs(er.v[0], (T)R.rc);
                    T d = T(0);
#pragma unroll
                    for (int q = 0; q < (NBC ? NBC : NB_MAX); q++) {
                        if (NBC == 0 && q >= nbr) continue;
                        d += w[q] * bs.slope();
                        bs.step();
                    }
                    if (fabs(er.v[0]) > T(1e-5)) {
                        const T dr = d / er.v[0];
#pragma unroll
                        for (int x = 0; x < 3; x++) {
                            const T fx = dr * er.v[1 + x];
                            cen[x] += fx;
                            add(j, x, -fx);
#pragma unroll
                            for (int y = 0; y < 3; y++) vir[3 * x + y] -= fx * er.v[1 + y];
                        }
                    }
                }
                if (end) break;
            }
#pragma unroll
            for (int x = 0; x < 3; x++) {
                const T c = wave_sum(cen[x]);
                if (lane == x) add(i, x, c);
            }
            wave_sync();
        }
        // angular list: a contiguous part of the segment's atoms per wavefront, several atoms to a pass
        if (A.l3 > 0) {
            int64_t i = s0 + (s1 - s0) * wid / W;
            const int64_t e1 = s0 + (s1 - s0) * (wid + 1) / W;
            while (i < e1) {
                const Batch<ANG_AB> b = next_batch<ANG_AB, WAVE>(A, i, e1, lane);
                batch_dq<T, ANG_AB>(A, b, i, na, lane, Bq, nullptr);
                wave_sync();
                T cen[16];
#pragma unroll
                for (int x = 0; x < 16; x++) cen[x] = T(0);
                for (int e0 = 0; e0 < b.tot; e0 += WAVE) {
                    if (lane < b.tot - e0) {
                        const int e = e0 + lane, q = b.atom(e);
                        const int64_t s = (i + q) * A.S + (e - b.first(q)), j = A.NL[s];
                        const Row4<T> er = load4(Ra + s * 4);
                        const T ir = T(1) / er.v[0];
                        const T ux = er.v[1] * ir, uy = er.v[2] * ir, uz = er.v[3] * ir;
                        T gn[NM_MAX], gp[NM_MAX];
                        radial_fn<T, NMC, NBC, true>(
                            reinterpret_cast<const T *>(A.c) + (int64_t)(b.ti * A.T + (int)A.atom_map[j]) * na * nba,
                            er.v[0], (T)A.rc, na, nba, gn, gp, [](int, T, T) {});
                        T Db[NM_MAX], d[4];
                        angular_slot<T, NMC, true>(Bq + q * per, na, ux, uy, uz, ir, gn, gp, Db, d);
                        // (selects, not a branch: the compiler would move the slot's work behind it and spill)
                        const bool far = fabs(er.v[0]) > T(1e-5);
                        const T fx[3] = {far ? d[0] * ux + d[1] : T(0), far ? d[0] * uy + d[2] : T(0),
                                         far ? d[0] * uz + d[3] : T(0)};
#pragma unroll
                        for (int x = 0; x < 3; x++) {
                            add(j, x, -fx[x]);
#pragma unroll
                            for (int y = 0; y < 3; y++) vir[3 * x + y] -= fx[x] * er.v[1 + y];
#pragma unroll
                            for (int u = 0; u < ANG_AB; u++) cen[3 * u + x] += q == u ? fx[x] : T(0);
                        }
                    }
                }
                const T c = fold16<T>(cen, lane);
                if (lane < 3 * b.na) add(i + lane / 3, lane % 3, c);
                wave_sync();
                i += b.na;
            }
        }
        T vf[16];
#pragma unroll
        for (int x = 0; x < 16; x++) vf[x] = x < 9 ? vir[x] : T(0);
        const T vs = fold16<T>(vf, lane);
        if (lane < 9) vred[wid * 9 + lane] = (double)vs;
        __syncthreads();
        const int64_t seg = (int64_t)blockIdx.x + f;
        if (threadIdx.x < 9) {
            double v = 0.0;
            for (int w = 0; w < W; w++) v += vred[w * 9 + threadIdx.x];
            p.vpart[seg * 9 + threadIdx.x] = v;
        }
        if (lds) {
            const unsigned row = blockIdx.x - (unsigned)fs / (unsigned)p.ch;
            T *o = reinterpret_cast<T *>(p.part) + 3 * (fs * p.rows + row * (fe - fs));
            for (int64_t x = threadIdx.x; x < 3 * (fe - fs); x += blockDim.x) o[x] = (T)acc[x];
        }
        __syncthreads();
    }
}

// F += the segments' LDS copies (blocks [0, fblocks): 64 entries, the segments of their frame in 4 groups), and
// each frame's virial from its segments' sums (one block per frame after them).
template <typename T>
__global__ void __launch_bounds__(256)
nep_force_final_kernel(const int64_t *__restrict__ frame_start, const int32_t *__restrict__ atom_frame, int64_t N,
                       int ch, int64_t rcap, int64_t rows, const T *__restrict__ part, const double *__restrict__ vpart,
                       T *__restrict__ F, T *__restrict__ V, int64_t fblocks) {
    __shared__ double red[256];
    if ((int64_t)blockIdx.x >= fblocks) {
        const int64_t f = (int64_t)blockIdx.x - fblocks, fs = frame_start[f], fe = frame_start[f + 1];
        const int c = threadIdx.x % 9, g = threadIdx.x / 9;          // 28 groups of 9 components
        double s = 0.0;
        if (fs < fe && g < 28)
            for (int64_t b = fs / ch + g; b <= (fe - 1) / ch; b += 28) s += vpart[(b + f) * 9 + c];
        red[threadIdx.x] = s;
        __syncthreads();
        if (threadIdx.x < 9) {
            s = 0.0;
            for (int q = 0; q < 28; q++) s += red[9 * q + threadIdx.x];
            V[9 * f + threadIdx.x] = (T)s;
        }
        return;
    }
    T *redT = reinterpret_cast<T *>(red);
    const int el = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int64_t e = (int64_t)blockIdx.x * 64 + el;
    T s = T(0);
    bool any = false;
    if (e < 3 * N) {
        const int64_t j = e / 3;
        const int f = atom_frame[j];
        const int64_t fs = frame_start[f], fe = frame_start[f + 1];
        any = fe - fs <= rcap;
        if (any) {
            const T *q = part + 3 * fs * rows + (e - 3 * fs);
            const unsigned w = (unsigned)ch, nw = (unsigned)(fe - 1) / w - (unsigned)fs / w + 1;
            const unsigned pitch = 3 * (unsigned)(fe - fs);          // nw pitch < 2^22: the LDS copy bounds the frame
#pragma unroll 4
            for (unsigned b = g; b < nw; b += 4) s += q[b * pitch];
        }
    }
    redT[threadIdx.x] = s;
    __syncthreads();
    if (g == 0 && any) F[e] += ((redT[el] + redT[el + 64]) + (redT[el + 128] + redT[el + 192]));
}

// The window, and the LDS copy of F: frames of at most rcap atoms within the block's 64 KB. Windows shrink with
// the atom count, down to 8, so that a small system still fills the chip.
struct ForcePlan {
    int ch;
    int64_t rcap;
    size_t lds;
};
template <typename T>
inline ForcePlan force_plan(int64_t N, int64_t max_frame, int ntypes, int na, int nbr) {
    const size_t fixed = force_fixed_lds<T>(ntypes, na, nbr);
    int64_t ch = (N + 511) / 512;
    ch = ch < 8 ? 8 : (ch > 64 ? 64 : ch);
    const int64_t cap = fixed < 64 * 1024 ? (int64_t)((64 * 1024 - fixed) / (3 * sizeof(double))) : 0;
    const int64_t rcap = max_frame <= cap ? max_frame : 0;
    return {(int)ch, rcap, fixed + 3 * rcap * sizeof(double)};
}

template <typename T, int NMC, int NBC>
int force_launch(ForceArgs &p, const ForcePlan &pl, int64_t nframes, T *V, hipStream_t st) {
    const int64_t N = p.r.N, blocks = ceil_div(N, pl.ch);
    p.ch = pl.ch;
    p.rcap = pl.rcap;
    p.rows = force_rows(pl.rcap, pl.ch);
    hipLaunchKernelGGL((nep_force_kernel<T, NMC, NBC>), dim3((unsigned)blocks), dim3(FORCE_WAVES * WAVE), pl.lds, st,
                       p);
    int rc = check_launch("nep_force_kernel");
    if (rc) return rc;
    const int64_t fblocks = pl.rcap > 0 ? ceil_div(3 * N, 64) : 0;
    hipLaunchKernelGGL(nep_force_final_kernel<T>, dim3((unsigned)(fblocks + nframes)), dim3(256), 0, st, p.frame_start,
                       p.atom_frame, N, pl.ch, pl.rcap, p.rows, reinterpret_cast<const T *>(p.part), p.vpart,
                       reinterpret_cast<T *>(p.F), V, fblocks);
    return check_launch("nep_force_final_kernel");
}

// ------------------------------------------------------------------ launch
enum FeatWhat { W_FEAT, W_1ST, W_GC, W_2ND, W_2ND_GS };

template <typename T, int NMC, int NBC>
int feat_launch(FeatArgs &a, bool angular, FeatWhat what, hipStream_t st) {
    if (!angular && what == W_2ND_GS) what = W_2ND;
    const size_t ncoef = (size_t)a.T * a.T * a.nm * a.nb, tb = (size_t)a.T * a.nb;
    const bool table = what == W_1ST || what == W_GC || what == W_2ND || what == W_2ND_GS;
    int waves = angular ? ANG_WAVES : RAD_WAVES;
    // LDS of a block of w wavefronts with ntab coefficient-gradient tables
    auto lds_of = [&](int w, size_t ntab) -> size_t {
        size_t e = table ? ntab * ncoef : 0;
        if (!angular) {
            const bool sum = what == W_FEAT || what == W_1ST || what == W_2ND;
            e += (size_t)w * ((sum ? WAVE * rad_stride<NBC>(a.nb) : 0) + (what == W_1ST ? tb : 0));
        } else if (what == W_FEAT) {
            e += (size_t)w * angf_wave_elems(a.nm);
        } else if (what == W_2ND || what == W_2ND_GS) {
            e += (size_t)w * ang2_wave_elems<T>(a.nm, a.nb);
        } else {
            e += (size_t)w * angb_wave_elems(a.nm, a.nb);
        }
        return e * sizeof(T);
    };
    // float: a table per wavefront (plain adds) when they fit, else one per block (LDS atomics): float LDS
    // atomic adds keep the LDS busy 3-4x longer than double ones for the same instruction count, while the
    // larger tables of double cost occupancy. Where the table of many types leaves too little room for the
    // wavefronts' rows, the block has fewer wavefronts.
    constexpr size_t LDS_MAX = 64 * 1024;
    a.pw = (table && sizeof(T) == 4 && lds_of(waves, waves) <= LDS_MAX) ? 1 : 0;
    while (!a.pw && waves > 1 && lds_of(waves, 1) > LDS_MAX) waves /= 2;
    const size_t lds = lds_of(waves, a.pw ? waves : 1);
    MATPL_CHECK_ARG(lds <= LDS_MAX, "nep_feat: LDS %zu too large", lds);
    int64_t blocks = (a.N + waves - 1) / waves;
    // with coefficient gradients: a bounded grid (4,096 wavefronts, 16 per CU) keeps the global atomics few
    // (one per table entry and block) while hiding the kernels' memory waits
    const int64_t cap = table ? 4096 / waves : 8192;
    if (blocks > cap) blocks = cap;
    dim3 grid((unsigned)blocks), block(waves * WAVE);
    if (!angular) {
        switch (what) {
        case W_FEAT: hipLaunchKernelGGL((nep_radial_kernel<T, NMC, NBC, R_FEAT>), grid, block, lds, st, a); break;
        case W_1ST: hipLaunchKernelGGL((nep_radial_kernel<T, NMC, NBC, R_1ST>), grid, block, lds, st, a); break;
        case W_GC: hipLaunchKernelGGL((nep_radial_kernel<T, NMC, NBC, R_GCF>), grid, block, lds, st, a); break;
        default: hipLaunchKernelGGL((nep_radial_kernel<T, NMC, NBC, R_2ND>), grid, block, lds, st, a); break;
        }
        return check_launch("nep_radial_kernel");
    }
    switch (what) {
    case W_FEAT: hipLaunchKernelGGL((nep_angular_fwd_kernel<T, NMC, NBC>), grid, block, lds, st, a); break;
    case W_1ST: hipLaunchKernelGGL((nep_angular_bwd_kernel<T, NMC, NBC, true>), grid, block, lds, st, a); break;
    case W_GC: hipLaunchKernelGGL((nep_angular_bwd_kernel<T, NMC, NBC, false>), grid, block, lds, st, a); break;
    case W_2ND: hipLaunchKernelGGL((nep_angular_bwd2_kernel<T, NMC, NBC, false>), grid, block, lds, st, a); break;
    default: hipLaunchKernelGGL((nep_angular_bwd2_kernel<T, NMC, NBC, true>), grid, block, lds, st, a); break;
    }
    return check_launch("nep_angular_kernel");
}

int feat_check(const FeatArgs &a, bool angular) {
    MATPL_CHECK_ARG(a.nb >= 1 && a.nb <= NB_MAX && a.nm >= 1 && a.nm <= NM_MAX, "nep_feat: basis sizes out of range");
    MATPL_CHECK_ARG(a.T >= 1 && a.T <= NT_MAX, "nep_feat: ntypes out of range");
    MATPL_CHECK_ARG(!angular || (a.l3 >= 0 && a.l3 <= 4 && (a.l3 == 4 || (a.l4 == 0 && a.l5 == 0))),
                    "nep_feat: l_max_3 must be 4 when 4/5-body terms are on");
    MATPL_CHECK_ARG(!angular || a.l5 == 0 || a.l4 > 0, "nep_feat: the 5-body term needs the 4-body term");
    return OK;
}

// The reference's default sizes (n_max 4, basis_size 12: nm = 5, nb = 13) have kernels of their own, whose
// loops over n and k unroll and keep their values in registers; other sizes run the general ones. At 5 and 13, these
// against the general ones: 62,713-atom float batch, second order 263 us (434), forces 181 (339), angular features
// 63 (133), radial 57 (106) and its second order 109 (244); double on 16 frames 142 (231), 49 (84), 31 (58),
// 18 (39), 30 (48); 1,728 atoms, float: forces 18 (29). At other sizes the training gradient takes 1.6 to 2.3 times
// less than with nm nb multiply-adds a slot (32 frames, n_max 7, basis_size 12, l_max (4, 2, 1): float
// 2228 -> 1106 us, double 2506 -> 1383; n_max 6, basis_size 8: 1851 -> 1020, 2050 -> 1261).
template <typename T>
int feat_sizes(FeatArgs &a, bool angular, FeatWhat what, hipStream_t st) {
    if (a.nm == 5 && a.nb == 13) return feat_launch<T, 5, 13>(a, angular, what, st);
    return feat_launch<T, 0, 0>(a, angular, what, st);
}

int feat_run(FeatArgs &a, int f64, bool angular, FeatWhat what, hipStream_t st) {
    const int rc = feat_check(a, angular);
    if (rc || a.N == 0) return rc;
    return f64 ? feat_sizes<double>(a, angular, what, st) : feat_sizes<float>(a, angular, what, st);
}

}  // namespace
}  // namespace matpl

using namespace matpl;

MATPL_EXPORT int matpl_nep_feat(int f64, int angular, int mode, const void *c, const void *Ri, const int64_t *NL,
                                const int64_t *atom_map, int64_t N, int S, int T, int nm, int nb, int ld, int col0,
                                int l3, int l4, int l5, double rc, void *feats, void *s_save, const void *gfeat,
                                const void *gg, void *gRi, void *gc, void *ggfeat, void *stream) {
    FeatArgs a{};
    a.c = c; a.Ri = Ri; a.NL = NL; a.atom_map = atom_map; a.feats = feats; a.save = angular ? s_save : nullptr;
    a.gfeat = gfeat; a.gg = gg; a.gRi = gRi; a.gc = gc; a.ggfeat = ggfeat;
    a.N = N; a.S = S; a.T = T; a.nm = nm; a.nb = nb; a.ld = ld; a.col0 = col0; a.l3 = l3; a.l4 = l4; a.l5 = l5;
    a.rc = rc;
    MATPL_CHECK_ARG(mode >= 0 && mode <= 2, "nep_feat: bad mode");
    MATPL_CHECK_ARG(N == 0 || (c && Ri && NL && atom_map), "nep_feat: null input");
    MATPL_CHECK_ARG(mode != 0 || N == 0 || (feats && (!angular || s_save)), "nep_feat: null output");
    MATPL_CHECK_ARG(mode != 1 || N == 0 || (gfeat && gRi && gc && (!angular || s_save)), "nep_feat: null grad io");
    MATPL_CHECK_ARG(mode != 2 || N == 0 || (gfeat && gg && gc && ggfeat && (!angular || s_save)),
                    "nep_feat: null 2nd-order io");
    return feat_run(a, f64, angular != 0, mode == 0 ? W_FEAT : (mode == 1 ? W_1ST : W_2ND), (hipStream_t)stream);
}

MATPL_EXPORT int matpl_nep_descriptor(int f64, int angular, int mode, const void *c, const void *Ri, const int64_t *NL,
                                      const int64_t *atom_map, int64_t N, int S, int T, int nm, int nb, int ld,
                                      int col0, int l3, int l4, int l5, double rc, void *feats, void *save,
                                      const void *gfeat, const void *gs, const void *gF, const void *gV,
                                      const int32_t *atom_frame, void *gc, void *ggfeat, void *gsave, void *stream) {
    FeatArgs a{};
    a.c = c; a.Ri = Ri; a.NL = NL; a.atom_map = atom_map; a.feats = feats; a.save = save;
    a.gfeat = gfeat; a.gs = angular ? gs : nullptr; a.gc = gc; a.ggfeat = ggfeat; a.gsave = gsave;
    a.gF = gF; a.gV = gV; a.atom_frame = atom_frame;
    a.N = N; a.S = S; a.T = T; a.nm = nm; a.nb = nb; a.ld = ld; a.col0 = col0; a.l3 = l3; a.l4 = l4; a.l5 = l5;
    a.rc = rc;
    MATPL_CHECK_ARG(mode >= 0 && mode <= 2, "nep_descriptor: bad mode");
    MATPL_CHECK_ARG(N >= 0 && S >= 0 && ld >= 1 && col0 >= 0, "nep_descriptor: bad sizes");
    MATPL_CHECK_ARG(N == 0 || (c && Ri && NL && atom_map), "nep_descriptor: null input");
    MATPL_CHECK_ARG(mode != 0 || N == 0 || (feats && (!angular || save)), "nep_descriptor: null output");
    MATPL_CHECK_ARG(mode != 1 || N == 0 || (gfeat && gc && ggfeat && (gF || gV) && (!gV || atom_frame) &&
                                            (!angular || (save && gsave))),
                    "nep_descriptor: null 2nd-order io");
    MATPL_CHECK_ARG(mode != 2 || N == 0 || (gc && save && (gfeat || (angular && gs))),
                    "nep_descriptor: null coefficient-gradient io");
    static const FeatWhat what[3] = {W_FEAT, W_2ND_GS, W_GC};
    return feat_run(a, f64, angular != 0, what[mode], (hipStream_t)stream);
}

// Bytes of the work buffer of matpl_nep_model_forces (the segments' virials, then the frames' rows of F).
MATPL_EXPORT int64_t matpl_nep_model_forces_work(int f64, int64_t N, int64_t nframes, int64_t max_frame, int ntypes,
                                                 int na, int nbr) {
    if (N <= 0 || nframes < 1 || max_frame < 1 || ntypes < 1 || na < 0 || nbr < 1) return 0;
    const ForcePlan pl = f64 ? force_plan<double>(N, max_frame, ntypes, na, nbr)
                             : force_plan<float>(N, max_frame, ntypes, na, nbr);
    const int64_t seg = ceil_div(N, pl.ch) + nframes;
    return seg * 9 * (int64_t)sizeof(double) + 3 * N * force_rows(pl.rcap, pl.ch) * (f64 ? 8 : 4);
}

MATPL_EXPORT int matpl_nep_model_forces(int f64, const void *c2, const void *c3, const void *Ri_r, const int64_t *NL_r,
                                        const void *Ri_a, const int64_t *NL_a, const int64_t *atom_map,
                                        const int64_t *frame_start, const int32_t *atom_frame, int64_t nframes,
                                        int64_t max_frame, int64_t N, int S_r, int S_a, int T, int nr, int nbr, int na,
                                        int nba, int ld, int l3, int l4, int l5, double rc_r, double rc_a,
                                        const void *gfeat, const void *s_save, void *F, void *V, void *work,
                                        int64_t work_bytes, void *stream) {
    MATPL_CHECK_ARG(N >= 0 && S_r >= 0 && S_a >= 0 && nframes >= 1 && max_frame >= 1 && ld >= 1,
                    "nep_model_forces: bad sizes");
    MATPL_CHECK_ARG(F && V && frame_start, "nep_model_forces: null output");
    hipStream_t st = (hipStream_t)stream;
    int rc = f64 ? fill_async<double>((double *)F, 0.0, 3 * N, st) : fill_async<float>((float *)F, 0.0f, 3 * N, st);
    if (rc) return rc;
    if (N == 0)
        return f64 ? fill_async<double>((double *)V, 0.0, 9 * nframes, st)
                   : fill_async<float>((float *)V, 0.0f, 9 * nframes, st);
    MATPL_CHECK_ARG(c2 && Ri_r && NL_r && atom_map && atom_frame && gfeat && work, "nep_model_forces: null input");
    MATPL_CHECK_ARG(l3 == 0 || (c3 && Ri_a && NL_a && s_save), "nep_model_forces: null angular input");
    if (l3 == 0) na = 0;
    MATPL_CHECK_ARG(work_bytes >= matpl_nep_model_forces_work(f64, N, nframes, max_frame, T, na, nbr) &&
                        ((uintptr_t)work & 7u) == 0,
                    "nep_model_forces: work buffer too small or not 8-byte aligned");
    ForceArgs p{};
    p.r.c = c2; p.r.Ri = Ri_r; p.r.NL = NL_r; p.r.atom_map = atom_map; p.r.gfeat = gfeat; p.r.N = N; p.r.S = S_r;
    p.r.T = T; p.r.nm = nr; p.r.nb = nbr; p.r.ld = ld; p.r.col0 = 0; p.r.rc = rc_r;
    p.a = p.r;
    p.a.c = c3; p.a.Ri = Ri_a; p.a.NL = NL_a; p.a.S = S_a; p.a.nm = na; p.a.nb = nba; p.a.col0 = nr; p.a.rc = rc_a;
    p.a.l3 = l3; p.a.l4 = l4; p.a.l5 = l5;
    p.a.save = const_cast<void *>(s_save);
    p.frame_start = frame_start; p.atom_frame = atom_frame; p.F = F;
    if ((rc = feat_check(p.r, false)) || (l3 > 0 && (rc = feat_check(p.a, true)))) return rc;
    const ForcePlan pl = f64 ? force_plan<double>(N, max_frame, T, na, nbr) : force_plan<float>(N, max_frame, T, na, nbr);
    MATPL_CHECK_ARG(pl.lds <= 64 * 1024, "nep_model_forces: LDS %zu too large", pl.lds);
    p.vpart = (double *)work;
    p.part = (double *)work + 9 * (ceil_div(N, pl.ch) + nframes);
    const bool std_sizes = nr == 5 && nbr == 13 && (l3 == 0 || (na == 5 && nba == 13));
    if (f64)
        return std_sizes ? force_launch<double, 5, 13>(p, pl, nframes, (double *)V, st)
                         : force_launch<double, 0, 0>(p, pl, nframes, (double *)V, st);
    return std_sizes ? force_launch<float, 5, 13>(p, pl, nframes, (float *)V, st)
                     : force_launch<float, 0, 0>(p, pl, nframes, (float *)V, st);
}
