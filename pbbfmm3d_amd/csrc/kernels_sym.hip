// kernels_sym.hip -- the FP64 M2L in a reflection-adapted basis.
//
// In a basis whose vectors are even or odd under each axis reflection
// (symm.cpp) the operators of mirrored directions differ by signs only:
// E_{Rd} = D_R K_d D_R.  The far field of a box then runs over the 56 orbits
// (|dx|, |dy|, |dz|) instead of the 189 directions: for one orbit, with K the
// orbit's block and p / q the parity classes of its columns and rows,
//   Pf[q] += sum_p K[q, p] v_{q,p},   v_{q,p} = sum_R chi_{q^p}(R) P_{t+Rd}[p],
// v the Walsh-Hadamard transform of the up to 8 mirrored sources.  A
// component of 1 or 2 covers both its signs with one product, and K is zero
// between classes that differ on an axis of component 0: the products of the
// 189 directions shrink to 39.5 in an open cloud.  Of these 81% fill at rank
// 101 (classes padded to 4 rows and 4 k), 89% at rank 181.
//
// Bound: the latency of the gathered sources and the barriers, beside the FP64
// matrix cores (the Walsh-Hadamard sums share their issue slots).  M2L of one
// matvec, with the set's own factors and here: 1M uniform points, 1/r, order 5,
// 8 columns 281 -> 64 ms, from the orbits (at the deepest level 56 ms, of which
// the matrix cores are busy 48%; its products at 78.6 TFLOP/s 21 ms); 1M
// clustered points, Gaussian, order 6, 32 columns 1410 -> 95 ms, from the orbits
// and, more, from the columns at the rounding level that the bases leave out
// (rank 181: 181, 181, 135, 81 and 53 at levels 2 to 6, at level 6 an eleventh
// of a block; there 59 ms, matrix cores 39% busy, 46% L2 hits, products 13 ms).
// Loading a step's sources under the products of the step before (16 columns a
// wave, two register sets) was slower: 75 -> 89 ms for the first of these calls.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kernels.hpp"

namespace pbb {
namespace dev {

namespace {

__constant__ SymOrbits c_orb;

typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) dbl2 dbl2g;  // (global, so that the loads are not flat ones)
typedef __attribute__((address_space(1))) double dblg;
typedef double dbl4 __attribute__((ext_vector_type(4)));

// Row groups (of 4 rows) of a configuration: class q holds cap(q) groups, by
// the number of its odd axes.
template <int C0, int C1, int C2, int C3>
struct Cfg {
    static constexpr int cap(int q)
    {
        const int c = ((q >> 2) & 1) + ((q >> 1) & 1) + (q & 1);
        return c == 0 ? C0 : c == 1 ? C1 : c == 2 ? C2 : C3;
    }
    static constexpr int goff(int q)
    {
        int s = 0;
        for (int i = 0; i < q; i++) s += cap(i);
        return s;
    }
    static constexpr int NG = goff(8);
    static constexpr int GM = C0 > C1 ? C0 : C1;
    static constexpr int AM = GM / 4 + 3;       // operator values of a class, at most
    static constexpr int CB = NG <= SYM_NG2 ? 2 : 1;  // 16-column blocks of a wave
};

// The sources of one orbit for this lane's columns: loads, and the transform
// over the paired axes PM.  x[cb][i], i within PM, ends as the value of class
// bits i on those axes; two consecutive k of the class per lane (one, at an
// odd last k step: half of the pair).  sg: -1 on an axis where the k class is
// odd, else 1.  tab: the boxes' offsets from base in units of 16 bytes.
template <class C, int PM>
__device__ __forceinline__ void sym_load(const uint32_t *const (&tab)[C::CB], const double *const (&base)[C::CB],
                                         const double (&sg)[3], int nj, bool upper, dbl2 (&x)[C::CB][8])
{
#pragma unroll
    for (int cb = 0; cb < C::CB; cb++) {
        int slot = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if ((i & ~PM) != 0) continue;
            x[cb][i] = *(const dbl2g *)((uint64_t)base[cb] + ((uint64_t)tab[cb][slot] << 4));
            slot++;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (nj == 1) {
#pragma unroll
        for (int cb = 0; cb < C::CB; cb++)
#pragma unroll
            for (int i = 0; i < 8; i++)
                if ((i & ~PM) == 0) x[cb][i].x = upper ? x[cb][i].y : x[cb][i].x;
    }
#pragma unroll
    for (int cb = 0; cb < C::CB; cb++) {
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            const int bit = 4 >> ax;
            if (!(PM & bit)) continue;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if ((i & ~PM) != 0 || (i & bit) != 0) continue;
                const dbl2 lo = x[cb][i], hi = x[cb][i | bit];
                x[cb][i].x = __builtin_fma(sg[ax], hi.x, lo.x);
                x[cb][i].y = __builtin_fma(sg[ax], hi.y, lo.y);
                x[cb][i | bit].x = __builtin_fma(-sg[ax], hi.x, lo.x);
                x[cb][i | bit].y = __builtin_fma(-sg[ax], hi.y, lo.y);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One k of the class per lane (4 per 16 columns): the products of the row
// classes that agree with the k class PZ on the axes ZM of component 0.
// Whole 16 rows of a class run on v_mfma_f64_16x16x4, the rest on
// v_mfma_f64_4x4x4, which holds 4 rows x 4 k x 16 columns as 4 blocks of 4
// columns that share the operator (A[i][k] in lanes i + 4 (any block) +
// 16 k, B[k][c] in lane c + 16 k, D[i][c] in lane c + 16 i): both reach the
// same rate, the second pads a class to 4 rows instead of 16, the first reads
// a quarter of the LDS bytes per row.  e4 / e16: this lane's operator value
// of a group / of 4 groups.  The next class's values are read ahead of a
// class's products; the scheduling barriers keep the compiler from reading
// all of them first, which would spill the sums.
template <class C, int PM, int ZM, int PZ, int J>
__device__ __forceinline__ void sym_products(const double *__restrict__ e4, const double *__restrict__ e16,
                                             const dbl2 (&x)[C::CB][8], double (&acc)[C::CB][C::NG])
{
    double av[2][C::AM];
    auto read = [&](int q, double (&v)[C::AM]) {
        const int at = (J * C::NG + C::goff(q)) * 16;
#pragma unroll
        for (int g = 0; g < C::GM / 4; g++)
            if (4 * g + 4 <= C::cap(q)) v[g] = e16[at + g * 64];
#pragma unroll
        for (int g = 0; g < 3; g++)
            if (g < C::cap(q) % 4) v[C::GM / 4 + g] = e4[at + (C::cap(q) / 4 * 4 + g) * 16];
    };
    int cur = 0;
    bool first = true;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        if (((q ^ PZ) & ZM) != 0) continue;
        if (first) read(q, av[0]);
        first = false;
        __builtin_amdgcn_sched_barrier(0);
        bool ahead = false;
#pragma unroll
        for (int n = q + 1; n < 8; n++)
            if (((n ^ PZ) & ZM) == 0 && !ahead) {
                read(n, av[cur ^ 1]);
                ahead = true;
            }
#pragma unroll
        for (int cb = 0; cb < C::CB; cb++) {
            const double b = J == 0 ? x[cb][q & PM].x : x[cb][q & PM].y;
            double *s = &acc[cb][C::goff(q)];
#pragma unroll
            for (int g = 0; g < C::GM / 4; g++) {
                if (4 * g + 4 > C::cap(q)) continue;
                dbl4 d = {s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
                d = __builtin_amdgcn_mfma_f64_16x16x4f64(av[cur][g], b, d, 0, 0, 0);
                s[4 * g] = d[0];
                s[4 * g + 1] = d[1];
                s[4 * g + 2] = d[2];
                s[4 * g + 3] = d[3];
            }
#pragma unroll
            for (int g = 0; g < 3; g++) {
                if (g >= C::cap(q) % 4) continue;
                const int k = C::cap(q) / 4 * 4 + g;
                s[k] = __builtin_amdgcn_mfma_f64_4x4x4f64(av[cur][C::GM / 4 + g], b, s[k], 0, 0, 0);
            }
        }
        cur ^= 1;
    }
    __builtin_amdgcn_sched_barrier(0);
}

template <class C, int PM, int ZM, int PZ>
__device__ __forceinline__ void sym_step(const uint32_t *const (&tab)[C::CB], const double *const (&base)[C::CB],
                                         const double (&sg)[3], const double *e4, const double *e16, int nj,
                                         bool upper, double (&acc)[C::CB][C::NG])
{
    dbl2 x[C::CB][8];
    __builtin_amdgcn_sched_barrier(0);
    sym_load<C, PM>(tab, base, sg, nj, upper, x);
    sym_products<C, PM, ZM, PZ, 0>(e4, e16, x, acc);
    if (nj > 1) sym_products<C, PM, ZM, PZ, 1>(e4, e16, x, acc);
}

}  // namespace

// A workgroup owns TB boxes of one octant class x cpt columns (at most 64 CB
// columns), each wave 16 CB of them with all rows of the launch's row slice in
// registers.  Steps: class p and 8 k of it (two per lane, 64 bytes of a
// proxy), outermost, so that the workgroups of an XCD read the same slice of
// every proxy and operator at about the same time; then the orbits with a
// source, NB to a barrier.  A batch's operator chunks are copied to a
// double-buffered LDS tile without passing through registers.  Proxies are
// gathered straight from memory as pairs of k, [box][k / 2][column][2], so
// that neighbouring lanes read neighbouring columns; between two barriers one
// wave's gathers run under the products of another.  FP64 matrix instructions
// keep the VALU of their SIMD busy, so the addresses come from a table of box
// offsets (one 64-bit add each; a box that is not there is the level's box of
// zeros).
template <class C>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sym_workgroups(C::NG)))) void m2l_sym_f64(SymArgs a)
{
    constexpr int NT = 256, NG = C::NG, ECH = 2 * NG * 16;  // doubles of an operator chunk
    const int NB = a.NB;
    __shared__ unsigned long long s_mask[56];
    __shared__ int4 s_list[56];  // the orbits of this sum part that have a source: kind, block, table offset, boxes
    __shared__ int s_n;
    __shared__ int s_tgt[SYM_TB];
    __shared__ int s_xyz[SYM_TB];
    extern __shared__ __attribute__((aligned(16))) double sE[];  // [2][NB][ECH], written 16 bytes a lane
    uint32_t *s_off = (uint32_t *)(sE + 2 * NB * ECH);           // [TB][189]: source offsets in units of 16 bytes
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int TB = a.TB;
    const int gyz = (int)(gridDim.y * gridDim.z);
    const int lin = xcd_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x * gyz);
    const int tile = lin / gyz;
    const int rem = lin - tile * gyz, chunk = rem / (int)gridDim.z;
    const int z = rem - chunk * (int)gridDim.z;
    const int part = z / a.nrow, rowp = z - part * a.nrow;  // sum part, row slice
    const int zp = part & (a.npz - 1), zo = part / a.npz;
    // tiles interleave the 8 octant classes, each class's tiles spread evenly
    // over the gridDim.x / 8 rounds: the classes are in Morton order, so the
    // workgroups that run together on an XCD read the sources of one region
    // (class after class they read the whole level once per class)
    const int o = tile & 7, round = tile >> 3, rounds = (int)gridDim.x >> 3;
    const int64_t nt = a.class_tiles[o];
    const int64_t mine = (round * nt + rounds - 1) / rounds;
    if (mine >= nt || mine * rounds / nt != round) return;
    const int64_t first = a.class_start[o] + mine * TB;
    const int64_t cend = a.class_start[o + 1];
    const int c0 = chunk * a.cpt;
    const int cpt = min(a.cpt, a.ncols - c0);
    const int S = a.side;
    if (tid < 56) s_mask[tid] = 0;
    if (tid < TB) {
        const int64_t q = first + tid;
        const int t = q < cend ? a.order[q] : -1;
        s_tgt[tid] = t;
        s_xyz[tid] = t >= 0 ? a.coord[t] : 0;
    }
    __syncthreads();
    const uint32_t box16 = (uint32_t)a.ncols * (uint32_t)a.ldp / 2;
    for (int q = tid; q < 189 * TB; q += NT) {
        const int tb = q / 189, u = q - tb * 189;
        int sid = -1;
        if (s_tgt[tb] >= 0) {
            const SymOrbit &w = c_orb.orbit[c_orb.slot_orbit[u]];
            const int neg = c_orb.slot_sign[u] ^ o;  // (mirrored into the octant whose 3s are positive)
            const uint32_t c = (uint32_t)s_xyz[tb];
            const int x = (int)(c & 1023) + ((neg & 4) ? -w.d[0] : w.d[0]);
            const int y = (int)((c >> 10) & 1023) + ((neg & 2) ? -w.d[1] : w.d[1]);
            const int zz = (int)((c >> 20) & 1023) + ((neg & 1) ? -w.d[2] : w.d[2]);
            if (x >= 0 && y >= 0 && zz >= 0 && x < S && y < S && zz < S) sid = a.map[((int64_t)x * S + y) * S + zz];
            if (sid >= 0) atomicOr(&s_mask[c_orb.slot_orbit[u]], 1ull << tb);
        }
        s_off[q] = (uint32_t)(sid + 1) * box16;  // (the launcher checks that it fits; 0: the box of zeros)
    }
    __syncthreads();
    if (wave == 0) {
        const int w = min(lane, 55);
        const SymOrbit &ob = c_orb.orbit[w];
        const unsigned long long m = s_mask[w];
        const bool live = lane < 56 && m != 0 && lane % a.noz == zo;
        const unsigned long long b0 = __ballot(live), below = (1ull << lane) - 1;
        // per axis: 0 component 3, 1 paired, 2 component 0 (3 with an odd k class)
        auto kind = [&](int bit) { return (ob.pm & bit) ? 1 : (ob.zm & bit) ? 2 : 0; };
        if (live)
            s_list[__popcll(b0 & below)] = int4{(kind(4) * 16 + kind(2) * 4 + kind(1)) | (w << 8), ob.slot,
                                                (int)(unsigned)m, (int)(unsigned)(m >> 32)};
        if (lane == 0) s_n = __popcll(b0);
    }
    __syncthreads();

    // this lane's columns: box and column; one past the tile repeats the first
    // and is not stored
    const int fr = lane & 15, fk = lane >> 4;
    int btb[C::CB], bcl[C::CB];
    bool bok[C::CB];
    const double *col[C::CB];
    const uint32_t *tab0[C::CB];
    int wm0 = 0, wm1 = 0;  // the wave's boxes, which are consecutive
#pragma unroll
    for (int cb = 0; cb < C::CB; cb++) {
        const int w0 = (wave * C::CB + cb) * 16, colx = w0 + fr, tbx = colx / cpt;
        bok[cb] = tbx < TB && s_tgt[min(tbx, SYM_TB - 1)] >= 0;
        btb[cb] = bok[cb] ? tbx : 0;
        bcl[cb] = bok[cb] ? colx - tbx * cpt : 0;
        col[cb] = a.P + 2 * (c0 + bcl[cb]);
        tab0[cb] = s_off + btb[cb] * 189;
        for (int t = w0 / cpt, t1 = min((w0 + 15) / cpt, TB - 1); t <= t1; t++) {
            if (t < 32) wm0 |= 1 << t;
            else wm1 |= 1 << (t - 32);
        }
    }
    const int ai4 = (lane & 3) + 4 * fk, ai16 = ((lane & 15) >> 2) * 16 + (lane & 3) + 4 * fk;
    const int n = __builtin_amdgcn_readfirstlane(s_n);

    double acc[C::CB][NG];
#pragma unroll
    for (int cb = 0; cb < C::CB; cb++)
#pragma unroll
        for (int g = 0; g < NG; g++) acc[cb][g] = 0.0;

    // chunks (p, j0) of the k classes; within a chunk the orbits in batches of
    // NB.  The operator chunk of a step: ECH doubles (the second half unused
    // at an odd last k step) from Ef + (((block * nrow + rowp) * nj + kb + j0)
    // * NG) * 16
    const size_t blk = (size_t)a.nrow * a.nj * (NG * 16);
    auto copy = [&](int p, int j0, int oi, int buf) {
        const double *src = a.Ef + ((size_t)rowp * a.nj + a.kb[p] + j0) * (size_t)(NG * 16);
        constexpr int UNITS = (ECH * 8 + 1023) / 1024;  // wave copies of 1 KB (the last one may overlap the one before)
        for (int b = 0; b < NB && oi + b < n; b++) {
            const double *e = src + (size_t)(__builtin_amdgcn_readfirstlane(s_list[oi + b].x) >> 8) * blk;
#pragma unroll
            for (int u = 0; u < UNITS; u += 4) {
                if (u + wave < UNITS) {
                    const int at = min((u + wave) * 128, ECH - 128);
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(e + at + lane * 2),
                                                     (__attribute__((address_space(3))) void *)(sE + (buf * NB + b) * ECH + at), 16, 0,
                                                     0);
                }
            }
        }
    };
    // the next chunk from (p, j0); false at the end
    auto advance = [&](int &p, int &j0) -> bool {
        j0 += 2;
        while (p < 8) {
            if (j0 < a.mk[p] && (p & (a.npz - 1)) == zp) return true;
            p++;
            j0 = 0;
        }
        return false;
    };
    int p = 0, j0 = -2, oi = 0, buf = 0, neg = 0;
    bool more = n > 0 && advance(p, j0);
    if (more) copy(p, j0, 0, 0);
    while (more) {
        // a batch: this wave's share of it is in LDS; the next one is copied meanwhile
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int np = p, nj0 = j0, noi = oi + NB;
        bool next = true;
        if (noi >= n) {
            noi = 0;
            next = advance(np, nj0);
        }
        if (next) copy(np, nj0, noi, buf ^ 1);
        const int nj = min(2, a.mk[p] - j0);
        const double sg[3] = {(p & 4) ? -1.0 : 1.0, (p & 2) ? -1.0 : 1.0, (p & 1) ? -1.0 : 1.0};
        const double *base[C::CB];  // the pair fk of a chunk of 8 k, or half a pair of one of 4
#pragma unroll
        for (int cb = 0; cb < C::CB; cb++)
            base[cb] = col[cb] + (size_t)(2 * (a.kb[p] + j0) + (nj > 1 ? fk : fk >> 1)) * (2 * a.ncols);
        if ((__popc(p & o) & 1) != neg) {  // the class's sign in the mirrored octant
            neg ^= 1;
#pragma unroll
            for (int cb = 0; cb < C::CB; cb++)
#pragma unroll
                for (int g = 0; g < NG; g++) acc[cb][g] = -acc[cb][g];
        }
        const int odd = ((p & 4) << 2) | ((p & 2) << 1) | (p & 1);  // the kinds' odd k classes
#pragma unroll 1
        for (int b = 0; b < NB && oi + b < n; b++) {
            const int4 le = s_list[oi + b];
            if (!((__builtin_amdgcn_readfirstlane(le.z) & wm0) | (__builtin_amdgcn_readfirstlane(le.w) & wm1)))
                continue;  // a wave without a source skips its products
            const int kk = __builtin_amdgcn_readfirstlane(le.x) & 63;
            const uint32_t *tab[C::CB];
#pragma unroll
            for (int cb = 0; cb < C::CB; cb++) tab[cb] = tab0[cb] + le.y;
            const double *eb = sE + (buf * NB + b) * ECH, *e4 = eb + ai4, *e16 = eb + ai16;
#define PBB_SYM_K(X, Y, Z)                                                                                   \
    case X * 16 + Y * 4 + Z:                                                                                 \
        if constexpr (X < 2 || Y < 2 || Z < 2) {                                                             \
            constexpr int PM = (X == 1) * 4 + (Y == 1) * 2 + (Z == 1);                                       \
            constexpr int ZM = (X > 1) * 4 + (Y > 1) * 2 + (Z > 1);                                          \
            constexpr int PZ = (X == 3) * 4 + (Y == 3) * 2 + (Z == 3);                                       \
            sym_step<C, PM, ZM, PZ>(tab, base, sg, e4, e16, nj, fk & 1, acc);                                \
        }                                                                                                    \
        break;
#define PBB_SYM_KY(X, Y) PBB_SYM_K(X, Y, 0) PBB_SYM_K(X, Y, 1) PBB_SYM_K(X, Y, 2) PBB_SYM_K(X, Y, 3)
#define PBB_SYM_KX(X) PBB_SYM_KY(X, 0) PBB_SYM_KY(X, 1) PBB_SYM_KY(X, 2) PBB_SYM_KY(X, 3)
            // (a kind of 2 becomes 3 on the axes where the k class is odd)
            switch (kk | ((kk >> 1) & odd)) { PBB_SYM_KX(0) PBB_SYM_KX(1) PBB_SYM_KX(2) PBB_SYM_KX(3) }
#undef PBB_SYM_K
#undef PBB_SYM_KY
#undef PBB_SYM_KX
        }
        buf ^= 1;
        p = np;
        j0 = nj0;
        oi = noi;
        more = next;
    }
#pragma unroll
    for (int cb = 0; cb < C::CB; cb++) {
        if (!bok[cb]) continue;
        double *dst = a.out + (size_t)part * a.part_stride +
                      ((size_t)(a.out_off + s_tgt[btb[cb]]) * a.ncols + c0 + bcl[cb]) * a.ldf + (size_t)rowp * NG * 4 + fk;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const bool flip = ((__popc(q & o) & 1) ^ neg) != 0;
#pragma unroll
            for (int g = 0; g < C::GM; g++)
                if (g < C::cap(q)) dst[(C::goff(q) + g) * 4] = flip ? -acc[cb][C::goff(q) + g] : acc[cb][C::goff(q) + g];
        }
    }
}

// The levels' boxes of zeros, n[k] doubles at p[k]
__global__ __launch_bounds__(256) void zero_boxes(ZeroBoxes z)
{
    double *p = z.p[blockIdx.x];
    for (int q = threadIdx.x; q < z.n[blockIdx.x]; q += 256) p[q] = 0.0;
}

// Pf = the sum parts in order (one part per z slice of a small launch)
__global__ __launch_bounds__(256) void m2l_sym_reduce(const double *__restrict__ part, int nparts, int64_t stride,
                                                      int64_t n, double *__restrict__ out)
{
    for (int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x; q < n; q += (int64_t)gridDim.x * 256) {
        double s = 0;
        int k = 0;
        for (; k + 8 <= nparts; k += 8) {  // (8 loads in flight)
            double v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = part[(k + i) * stride + q];
#pragma unroll
            for (int i = 0; i < 8; i++) s += v[i];
        }
        for (; k < nparts; k++) s += part[k * stride + q];
        out[q] = s;
    }
}

// dst_d (c x r) = src_d^T, src_d r x c column-major, d < nd
__global__ __launch_bounds__(256) void transpose_blocks(const double *__restrict__ src, int r, int c, int64_t nd,
                                                        double *__restrict__ dst)
{
    const int64_t len = (int64_t)r * c, total = nd * len;
    for (int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x; q < total; q += (int64_t)gridDim.x * 256) {
        const int64_t d = q / len;
        const int e = (int)(q - d * len), j = e % c, i = e / c;  // dst element (j, i)
        dst[q] = src[d * len + i + (int64_t)j * r];
    }
}

// M_w = avg over the reflections R of D_R Z_{R d_w}^T D_R for the 56 orbits,
// from Z_d (rs x rf) of the 316 directions; cf, cs: class of row and column
__global__ __launch_bounds__(256) void sym_average(const double *__restrict__ Z, const int *__restrict__ cf,
                                                   const int *__restrict__ cs, int rf, int rs,
                                                   const int *__restrict__ dir, double *__restrict__ M)
{
    const int64_t len = (int64_t)rf * rs, total = 56 * len;
    for (int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x; q < total; q += (int64_t)gridDim.x * 256) {
        const int w = (int)(q / len);
        const int e = (int)(q - w * len), i = e % rf, j = e / rf;
        const int c = cf[i] ^ cs[j];
        double s = 0;
        for (int R = 0; R < 8; R++) {
            const double v = Z[(int64_t)dir[w * 8 + R] * len + j + (int64_t)i * rs];
            s += (__popc(c & R) & 1) ? -v : v;
        }
        M[q] = 0.125 * s;
    }
}

// E_d of the 316 directions from the orbits' blocks: D_R K_w D_R
__global__ __launch_bounds__(256) void sym_expand(const double *__restrict__ K, const int *__restrict__ cf,
                                                  const int *__restrict__ cs, int rf, int rs,
                                                  const int *__restrict__ of, const int *__restrict__ refl,
                                                  double *__restrict__ E)
{
    const int64_t len = (int64_t)rf * rs, total = 316 * len;
    for (int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x; q < total; q += (int64_t)gridDim.x * 256) {
        const int d = (int)(q / len);
        const int e = (int)(q - d * len), i = e % rf, j = e / rf;
        const double v = K[of[d] * len + e];
        E[q] = (__popc((cf[i] ^ cs[j]) & refl[d]) & 1) ? -v : v;
    }
}

// ---------------------------------------------------------------------------

namespace {
// row-group capacities by the number of odd axes, in the order of their
// cost; the operators are padded to a configuration's groups.  The list is
// made for order 4, order 5 at eps 1e-7 and order 6 at eps 1e-7 and 1e-8; other
// class counts take the next that holds them, some with much padding (order 5
// at eps 1e-9, 26 or 27 columns in the even class: 48 groups where 33 would do;
// 1/r, order 5, eps 1e-5: 28 where 17 would).
struct SymConf {
    int cap[4];
};
constexpr SymConf CONF[SYM_CONFS] = {
    {{2, 2, 1, 1}}, {{2, 2, 2, 2}}, {{3, 3, 2, 2}}, {{5, 4, 3, 2}}, {{6, 4, 3, 2}},
    {{6, 5, 3, 2}}, {{6, 5, 4, 3}}, {{6, 5, 5, 4}}, {{7, 6, 6, 5}},
};
constexpr size_t SYM_LDS = 160 * 1024;      // of a CU
constexpr size_t SYM_LDS_FIXED = 3328;      // the kernel's other arrays, and the allocation's granularity
int blocks_for(int64_t total) { return (int)std::min<int64_t>((total + 255) / 256, 16384); }
}  // namespace

SymShape sym_shape(const int cnt[8])
{
    SymShape s{};
    for (int k = 0; k < SYM_CONFS; k++) {
        const SymConf &c = CONF[k];
        int need = 1;  // row slices of the configuration's capacity
        int ng = 0;
        for (int q = 0; q < 8; q++) {
            const int cp = c.cap[__builtin_popcount(q)], g = (cnt[q] + 3) / 4;
            ng += cp;
            need = std::max(need, (g + cp - 1) / cp);
        }
        if (need > 1 && k < SYM_CONFS - 1) continue;
        s.conf = k;
        s.ng = ng;
        s.nrow = need;
        break;
    }
    return s;
}

int sym_width(const SymShape &s) { return s.ng <= SYM_NG2 ? 128 : 64; }

int sym_row(const SymShape &s, int q, int i)
{
    const SymConf &c = CONF[s.conf];
    const int g = i / 4, cp = c.cap[__builtin_popcount(q)];
    int off = 0;
    for (int m = 0; m < q; m++) off += c.cap[__builtin_popcount(m)];
    return (g / cp * s.ng + off + g % cp) * 4 + i % 4;
}

void upload_sym_orbits()
{
    SymOrbits o;
    sym_orbits(o);
    check(hipMemcpyToSymbol(HIP_SYMBOL(c_orb), &o, sizeof(o)), "hipMemcpyToSymbol(c_orb)");
}

void launch_m2l_sym(const SymArgs &args, const SymShape &s, int ncolchunks, hipStream_t st)
{
    SymArgs a = args;
    if (a.class_start[8] <= 0) return;
    if (a.TB < 1 || a.TB > SYM_TB || a.TB * a.cpt > sym_width(s) || (a.npz & (a.npz - 1)) != 0)
        fail(PBB_ERR_INTERNAL, "M2L tile does not fit its workgroup");
    if (!sym_level_fits(a.class_start[8], a.ncols, a.ldp)) fail(PBB_ERR_INTERNAL, "M2L level of more than 64 GB of proxies");
    const int most = *std::max_element(a.class_tiles, a.class_tiles + 8);
    dim3 grid((unsigned)most * 8, (unsigned)ncolchunks, (unsigned)(a.nrow * a.npz * a.noz));
    // orbits to a barrier: what LDS holds beside the table at the workgroups
    // per CU that the registers allow (a barrier waits for the slowest wave's
    // gathers).  Two for all and now, one matvec: 1M points, 8 columns (4
    // orbits) 75.4 -> 72.0 ms; 1M clustered, 32 columns (4, with the third
    // workgroup of small configurations) 147 -> 129 ms.  Four at the price of a
    // workgroup (500k points, 4 columns) was slower by a third.
    const size_t table = sizeof(uint32_t) * 189 * a.TB, chunk = 2 * sizeof(double) * 2 * s.ng * 16;
    const size_t room = SYM_LDS / sym_workgroups(s.ng) - SYM_LDS_FIXED;
    a.NB = (int)std::max<size_t>(2, std::min<size_t>(SYM_NB, room > table ? (room - table) / chunk : 0));
    const size_t lds = chunk * a.NB + table;
    switch (s.conf) {
    case 0: m2l_sym_f64<Cfg<2, 2, 1, 1>><<<grid, 256, lds, st>>>(a); break;
    case 1: m2l_sym_f64<Cfg<2, 2, 2, 2>><<<grid, 256, lds, st>>>(a); break;
    case 2: m2l_sym_f64<Cfg<3, 3, 2, 2>><<<grid, 256, lds, st>>>(a); break;
    case 3: m2l_sym_f64<Cfg<5, 4, 3, 2>><<<grid, 256, lds, st>>>(a); break;
    case 4: m2l_sym_f64<Cfg<6, 4, 3, 2>><<<grid, 256, lds, st>>>(a); break;
    case 5: m2l_sym_f64<Cfg<6, 5, 3, 2>><<<grid, 256, lds, st>>>(a); break;
    case 6: m2l_sym_f64<Cfg<6, 5, 4, 3>><<<grid, 256, lds, st>>>(a); break;
    case 7: m2l_sym_f64<Cfg<6, 5, 5, 4>><<<grid, 256, lds, st>>>(a); break;
    case 8: m2l_sym_f64<Cfg<7, 6, 6, 5>><<<grid, 256, lds, st>>>(a); break;
    default: fail(PBB_ERR_INTERNAL, "unknown M2L row configuration");
    }
    check(hipGetLastError(), "m2l_sym_f64");
}

void launch_zero_boxes(const ZeroBoxes &z, int nlevels, hipStream_t st)
{
    if (nlevels <= 0) return;
    zero_boxes<<<nlevels, 256, 0, st>>>(z);
    check(hipGetLastError(), "zero_boxes");
}

void launch_m2l_sym_reduce(const double *part, int nparts, int64_t stride, int64_t n, double *out, hipStream_t st)
{
    if (n <= 0) return;
    m2l_sym_reduce<<<blocks_for(n), 256, 0, st>>>(part, nparts, stride, n, out);
    check(hipGetLastError(), "m2l_sym_reduce");
}

void launch_transpose_blocks(const double *src, int r, int c, int64_t nd, double *dst, hipStream_t st)
{
    transpose_blocks<<<blocks_for(nd * r * c), 256, 0, st>>>(src, r, c, nd, dst);
    check(hipGetLastError(), "transpose_blocks");
}

void launch_sym_average(const double *Z, const int *cf, const int *cs, int rf, int rs, const int *dir, double *M,
                        hipStream_t st)
{
    sym_average<<<blocks_for((int64_t)56 * rf * rs), 256, 0, st>>>(Z, cf, cs, rf, rs, dir, M);
    check(hipGetLastError(), "sym_average");
}

void launch_sym_expand(const double *K, const int *cf, const int *cs, int rf, int rs, const int *of, const int *refl,
                       double *E, hipStream_t st)
{
    sym_expand<<<blocks_for((int64_t)316 * rf * rs), 256, 0, st>>>(K, cf, cs, rf, rs, of, refl, E);
    check(hipGetLastError(), "sym_expand");
}

}  // namespace dev
}  // namespace pbb
