// Group passes of the fused DP kernels: one wavefront takes up to GA consecutive atoms of one frame and one type
// together, so that their in-cutoff neighbors of each type share 32-lane tiles. A four-type system holds ~2 to 25
// neighbors per bucket (48 of 128 tile lanes filled atom by atom); four atoms together fill ~80 %. Used for
// three types and more (dp_group_wanted): with one or two a bucket fills its tiles by itself (HfO2 27 and 55, Cu 78),
// and the per-lane atom selects below would only cost.
#pragma once
#include "dp_fused_common.h"

namespace matpl {
namespace {

constexpr int GA = 4;                          // atoms per group at most
constexpr int GSEG = MAXT * GA;                // (type, atom) segments
constexpr int DA_STRIDE = 33;                  // float4 rows of dA per atom (odd: atoms' rows hit distinct banks)
constexpr int GT_STRIDE = 33;                  // FP32 G tile [32 neighbors][33]
constexpr int QSHIFT = 24;                     // atom of an entry's packed (bucket slot | atom << 24)
constexpr int JSHIFT = 29;                     // atom of an entry's packed (neighbor | atom << 29)

// Where the passes are taken. The caller says whether buckets are short (DP_GROUP in its precision argument), since
// the lists themselves are on the device: matpl_amd.dp_fused.short_buckets, by the mix of types. us of a whole
// evaluation, an atom per wavefront against groups, four-type models in BF16:
//   60,000 atoms of four types (40, 4, 8 and 48 %) 865 and 660; 55,296 HfO2 atoms 726 and 769, 8,640 191 and 222;
//   of few atoms each wavefront takes one (500 atoms 81 and 84, 4,000 126 and 133; 4,500 143 and 120).
// The backward at E = 32 in BF16 needs all registers for groups (one wavefront per SIMD: 20,000 atoms 204 and 245).
constexpr int DP_GROUP = 0x100;
constexpr int64_t GROUP_ATOMS = 4096;

inline bool dp_group_wanted(const FusedParams &p) {
    return p.group && p.T >= 3 && p.natoms >= GROUP_ATOMS && p.natoms < (1ll << JSHIFT) && p.mnl < (1 << QSHIFT);
}

// Atoms per group and wavefront of a kernel that runs `occ` wavefronts on each of the 1,024 SIMDs: those whose
// rounds of wavefronts take the least, a group of g atoms costing about g + 1 (a last round that is nearly empty costs
// as much as a full one: 8,640 atoms in groups of four are 2,160 wavefronts, of 2,048 that run at once). With
// many rounds, whole groups, and several per wavefront.
inline void dp_group_shape(FusedParams &p, int occ) {
    int64_t best = 0;
    for (int g = GA; g >= 2; g--) {
        const int64_t waves = (p.natoms + g - 1) / g, rounds = (waves + 1024 * occ - 1) / (1024 * occ);
        if (g == GA || rounds * (g + 1) < best) {
            best = rounds * (g + 1);
            p.ga = g;
        }
    }
    const int64_t per = p.natoms / (8192 * (int64_t)p.ga);          // whole groups per wavefront
    p.gchunk = p.ga * (int)(per < 1 ? 1 : per);
}

// Blocks of a group kernel: a multiple of the XCDs, which take contiguous ranges of atoms (logical_block).
inline unsigned dp_group_blocks(const FusedParams &p) {
    const int64_t per = FUSED_WAVES * (int64_t)p.gchunk, blocks = (p.natoms + per - 1) / per;
    return (unsigned)((blocks + NXCD - 1) / NXCD * NXCD);
}

struct Group {
    int na, ti, frame;      // atoms, their type and frame
    int tot;                // used list entries of all their buckets
};

// The group starting at atom i: atoms of its frame and type, at most ga, whose used entries fit nbw. Lane s =
// t * GA + q returns in `first` the start of bucket t of atom q in the group's entries taken bucket by bucket
// (lane T * GA: the total).
__device__ __forceinline__ Group group_at(const FusedParams &p, int64_t i, int64_t i1, int ga, int nbw, int lane,
                                          int &first) {
    const int q = lane & (GA - 1), t = lane / GA;
    const int64_t ia = i + q;
    const bool in = q < ga && ia < i1 && t < p.T;
    const int c = in ? p.counts[ia * p.T + t] : 0;
    const bool at = q < ga && ia < i1;
    const int ty = at ? p.type_map[ia] : -1, fr = at ? (p.atom_frame ? p.atom_frame[ia] : 0) : -1;
    Group g;
    g.ti = __builtin_amdgcn_readfirstlane(ty);
    g.frame = __builtin_amdgcn_readfirstlane(fr);
    g.na = 0;
    g.tot = 0;
#pragma unroll
    for (int x = 0; x < GA; x++) {
        int n = 0;
        for (int u = 0; u < p.T; u++) n += __builtin_amdgcn_readlane(c, u * GA + x);
        const bool same = __builtin_amdgcn_readlane(ty, x) == g.ti && __builtin_amdgcn_readlane(fr, x) == g.frame;
        if (g.na == x && same && (x == 0 || g.tot + n <= nbw)) {
            g.na = x + 1;
            g.tot += n;
        }
    }
    int run = q < g.na ? c : 0, mine = run;
#pragma unroll
    for (int o = 1; o < 2 * GSEG; o <<= 1) {
        const int u = __shfl_up(run, o, WAVE);
        if (lane >= o) run += u;
    }
    first = run - mine;
    return g;
}

// Starts a group: its segment starts in LDS, counts cleared.
__device__ __forceinline__ void group_begin(int T, int first, int lane, int *cnt, int *seg) {
    if (lane < T * GA) cnt[lane] = 0;
    if (lane <= T * GA) seg[lane] = first;
    __builtin_amdgcn_wave_barrier();
}

// The end of the range of types from ta whose entries fit nbw together (at least one type): one range for almost
// every group; only a single atom with more entries than nbw takes several.
__device__ __forceinline__ int group_range(int T, int ta, int nbw, const int *seg) {
    int tb = ta + 1;
    while (tb < T && seg[(tb + 1) * GA] - seg[ta * GA] <= nbw) tb++;
    return __builtin_amdgcn_readfirstlane(tb);
}

// Compacts the group's in-cutoff neighbors of types [ta, tb) into nb, bucket by bucket and within a bucket atom by
// atom: (dx, dy, dz, slot | atom << QSHIFT), with BYJ (neighbor atom | atom << JSHIFT). cnt[t * GA + q] receives the
// neighbors of type t of atom q (at most nbw entries are kept). Listed entries beyond the cutoff get a zero per-slot
// force when fslot is given (as compact()). Returns -1, or an atom of the group with a bucket of more than m.
template <bool BYJ>
__device__ __forceinline__ int compact_group(const FusedParams &p, int64_t i, int ta, int tb, int lane, int nbw,
                                             float4 *nb, int *cnt, const int *seg, float4 *fslot) {
    AtomGeo gl = atom_geo(p, i);
    const uint64_t below = (1ull << lane) - 1ull;
    const int ea = seg[ta * GA], eb = seg[tb * GA];
    int nv = 0;
    for (int e0 = ea; e0 < eb; e0 += WAVE) {
        const int e = e0 + lane;
        bool ok = false;
        int s = ta * GA, q = 0, k = 0, j = 0;
        double dx = 0.0, dy = 0.0, dz = 0.0;
        if (e < eb) {
            for (int x = ta * GA + 1; x < tb * GA; x++) s += e >= seg[x] ? 1 : 0;   // the last segment starting at or before e
            q = s & (GA - 1);
            const int64_t ia = i + q;
            k = e - seg[s];
            const int64_t slot = (ia * p.T + s / GA) * (int64_t)p.mnl + k;
            gl.xi = p.pos[3 * ia]; gl.yi = p.pos[3 * ia + 1]; gl.zi = p.pos[3 * ia + 2];
            j = (int)neighbor_disp(p, gl, slot, dx, dy, dz);
            const double r2 = dx * dx + dy * dy + dz * dz;
            ok = r2 < p.rc2 && r2 > 1e-10;
            if (!ok && fslot) {
                const int r = p.rev[slot];
                if (r >= 0) fslot[r] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
        const uint64_t bal = __ballot(ok);
        const int idx = nv + __popcll(bal & below);
        if (ok) {
            if (idx < nbw)
                nb[idx] = make_float4((float)dx, (float)dy, (float)dz,
                                      __int_as_float(BYJ ? (j | (q << JSHIFT)) : (k | (q << QSHIFT))));
            atomicAdd(cnt + s, 1);
        }
        nv += __popcll(bal);
    }
    __builtin_amdgcn_wave_barrier();
    const uint64_t over = __ballot(lane >= ta * GA && lane < tb * GA && cnt[lane] > p.m);
    return over ? (__builtin_ctzll(over) & (GA - 1)) : -1;
}

// Neighbors of type t of the whole group.
__device__ __forceinline__ int group_type(const int *cnt, int t) {
    int n = 0;
#pragma unroll
    for (int q = 0; q < GA; q++) n += cnt[t * GA + q];
    return __builtin_amdgcn_readfirstlane(n);
}

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

// D[(q, w)][f] += sum over the tile's neighbors of x[n][w] (where n's atom is q) times the feature value of n, in
// FP32 on the matrix cores (16x16x4, two column tiles): rows are (atom, component), so lane l, register r of
// column tile c hold atom l / 16, component r, feature 16 c + l % 16. A lane gives its neighbor's four x and
// features (accumulator layout: register r, half h = feature f(r, h)); xs [32][5] and gt [32][GT_STRIDE] are
// the wave's LDS.
template <int E>
__device__ __forceinline__ void contract_group(const float x[4], int q, const float *G, int lane, float *xs, float *gt,
                                               floatx4 D[2]) {
    constexpr int NR = NReg<E>::value;
    const int h = lane >> 5, n = lane & 31;
    if (h == 0) {
#pragma unroll
        for (int w = 0; w < 4; w++) xs[n * 5 + w] = x[w];
        xs[n * 5 + 4] = __int_as_float(q);
    }
    // (columns of D beyond the features are never read: their rows of gt may hold anything)
#pragma unroll
    for (int r = 0; r < NR; r++) gt[n * GT_STRIDE + feat(r, h)] = G[r];
    __builtin_amdgcn_wave_barrier();
    const int row = lane & 15, kk = lane >> 4, aq = row >> 2, aw = row & 3;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int nn = 4 * s + kk;
        const float v = xs[nn * 5 + aw];
        const float a = __float_as_int(xs[nn * 5 + 4]) == aq ? v : 0.0f;
#pragma unroll
        for (int c = 0; c < 2; c++)
            D[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, gt[nn * GT_STRIDE + 16 * c + row], D[c], 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
}

// Per-wave LDS of a group kernel (bytes): entries, counts and segment starts, then what the kernel adds.
inline __host__ __device__ int group_nbw(const FusedParams &p) { return p.cap > 4 * WAVE ? p.cap : 4 * WAVE; }
inline __host__ __device__ size_t group_base_bytes(int nbw) { return (size_t)nbw * 16 + (2 * GSEG + 4) * 4; }
constexpr size_t GROUP_F32_BYTES = (32 * 5 + 32 * GT_STRIDE) * 4;      // xs and gt of contract_group
constexpr size_t GROUP_BF16_BYTES = (32 * 32 + 32 * 40) * 2;           // Ri^T [16 of 32 rows][32], G^T [32][40] in bf16
constexpr size_t GROUP_DA_BYTES = (size_t)GA * DA_STRIDE * 16 + 16 * 4;  // dA rows, centre sums

struct GroupLds {
    float4 *nb;
    int *cnt, *seg;
    unsigned char *rest;
};
__device__ __forceinline__ GroupLds group_lds(unsigned char *smem, int wid, int nbw, size_t extra) {
    unsigned char *b = smem + (size_t)wid * (group_base_bytes(nbw) + extra);
    GroupLds l;
    l.nb = reinterpret_cast<float4 *>(b);
    l.cnt = reinterpret_cast<int *>(l.nb + nbw);
    l.seg = l.cnt + GSEG;
    l.rest = b + group_base_bytes(nbw);
    return l;
}

}  // namespace
}  // namespace matpl
