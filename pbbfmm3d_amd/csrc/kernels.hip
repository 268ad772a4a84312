// kernels.hip -- gfx950 kernels of the FP64 black-box FMM matvec.
//
// Data layout in HBM (one plan):
//   points    sorted by leaf (Morton order), re-centred, SoA x[N] y[N] z[N]
//   perm      sorted position -> caller's index (weights/outputs stay in the
//             caller's column-major order w[c*N + i])
//   ws        weights gathered into sorted order, ws[c*N + k]
//   S / F     per box (global id = level offset + compact id) a column-major
//             n3 x ncols block: S[(g*ncols + c)*n3 + l].  The upward pass's
//             S (sourceval) and the downward pass's F (targetval) share it.
//   P         proxies (proxysval) r_s x ncols per box, P[(g*ncols + c)*rs + a]
//   Pf        M2L result r_f x ncols per box
// Operators: VTw = VT diag(Kweights) (r_s x n3), Uw = diag(Kweights) U
// (n3 x r_f), E (316 blocks r_f x r_s), all column-major FP64.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.hpp"

namespace pbb {
namespace dev {

__constant__ int c_dirs[8][189][4];  // far directions of each octant class

typedef double dbl4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// device kernel functors (formulas of pbb_kernel_id); r2 = |s - t|^2 with
// the differences taken as source - target (kernel_Types.cpp:21-23)
//
// 1 / sqrt(x) for x other than 0 and infinity (there a NaN): the hardware's
// estimate (2^-23) and one third-order step, 7 operations in place of a square
// root and a division (about 35), and as close (an error of at most about one
// unit in the last place either way)
__device__ __forceinline__ double rsqrt_inner(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = __builtin_fma(-(x * y), y, 1.0);
    return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double rsqrt_step(double x)
{
    const double z = rsqrt_inner(x);
    return __builtin_amdgcn_class(x, 0x264) ? __builtin_amdgcn_rsq(x) : z;  // (+-0, +-infinity)
}
// a / b for a b that many values share (1 / b is formed once outside the
// loop): the quotient's residual corrects it to the division's rounding
__device__ __forceinline__ double div_shared(double a, double b)
{
    const double inv = 1.0 / b, q = a * inv;
    const double z = __builtin_fma(__builtin_fma(-q, b, a), inv, q);
    return z == z ? z : q;  // (an infinite a)
}
template <int KID>
__device__ __forceinline__ double keval(double dx, double dy, double dz, const KParams &p)
{
    double r2 = dx * dx + dy * dy + dz * dz;
    if constexpr (KID == PBB_KERNEL_LAPLACIAN) return rsqrt_step(r2);
    else if constexpr (KID == PBB_KERNEL_ONEOVERR2) { double ri = rsqrt_step(r2); return ri * ri; }
    else if constexpr (KID == PBB_KERNEL_GAUSSIAN) return exp(-div_shared(r2, p.p[0] * p.p[0]));
    else if constexpr (KID == PBB_KERNEL_EXPONENTIAL) return p.p[1] * exp(-div_shared(sqrt(r2), p.p[0]));
    else if constexpr (KID == PBB_KERNEL_SOFT_LAPLACIAN) return rsqrt_step(r2 + p.p[0]);
    else if constexpr (KID == PBB_KERNEL_QUADRIC) return 1.0 + r2;
    else if constexpr (KID == PBB_KERNEL_INV_QUADRIC) return 1.0 / (1.0 + r2);
    else if constexpr (KID == PBB_KERNEL_LOGARITHM) return r2 == 0 ? 0.0 : 0.5 * log(r2);
    else if constexpr (KID == PBB_KERNEL_THIN_PLATE) return r2 == 0 ? 0.0 : 0.5 * r2 * log(r2);
    else if constexpr (KID == PBB_KERNEL_R2) return r2;
    else if constexpr (KID == PBB_KERNEL_CONSTANT) return 1.0;
    else if constexpr (KID == PBB_KERNEL_EXP_ANISO)
        return p.p[0] * exp(-sqrt(p.p[1] * dx * dx + p.p[2] * dy * dy + p.p[3] * dz * dz));
    else return 0.0;
}

// The values of the near field and the direct sum, 0 in place of an infinity
// (coincident points).  An inverse root needs one select for that: it is 0 at
// an infinite argument as well; a Gaussian is never infinite.
template <int KID>
__device__ __forceinline__ double keval0(double dx, double dy, double dz, const KParams &p)
{
    if constexpr (KID == PBB_KERNEL_LAPLACIAN || KID == PBB_KERNEL_SOFT_LAPLACIAN) {
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double x = KID == PBB_KERNEL_LAPLACIAN ? r2 : r2 + p.p[0];
        const double z = rsqrt_inner(x);
        return __builtin_amdgcn_class(x, 0x264) ? 0.0 : z;  // (+-0, +-infinity)
    } else {
        const double kv = keval<KID>(dx, dy, dz, p);
        return KID != PBB_KERNEL_GAUSSIAN && isinf(kv) ? 0.0 : kv;
    }
}

// The values the operators are made from.  They keep the library's square
// root and division: within a degenerate cluster the singular vectors (and
// with them the subspace a cut through the cluster keeps) turn with the last
// bit of the kernel blocks.
template <int KID>
__device__ __forceinline__ double keval_blocks(double dx, double dy, double dz, const KParams &p)
{
    const double r2 = dx * dx + dy * dy + dz * dz;
    if constexpr (KID == PBB_KERNEL_LAPLACIAN) return 1.0 / sqrt(r2);
    else if constexpr (KID == PBB_KERNEL_ONEOVERR2) { double ri = 1.0 / sqrt(r2); return ri * ri; }
    else if constexpr (KID == PBB_KERNEL_GAUSSIAN) return exp(-r2 / (p.p[0] * p.p[0]));
    else if constexpr (KID == PBB_KERNEL_EXPONENTIAL) return p.p[1] * exp(-sqrt(r2) / p.p[0]);
    else if constexpr (KID == PBB_KERNEL_SOFT_LAPLACIAN) return 1.0 / sqrt(r2 + p.p[0]);
    else return keval<KID>(dx, dy, dz, p);
}

// The same functors with the transcendental part in FP32 (the mixed modes'
// near field): r^2 from the FP64 differences, then the FP32 library
// function; relative error a few 1e-7 per value
template <int KID>
__device__ __forceinline__ double keval_f32(double dx, double dy, double dz, const KParams &p)
{
    const double r2 = dx * dx + dy * dy + dz * dz;
    const float f = (float)r2;
    if constexpr (KID == PBB_KERNEL_LAPLACIAN) return (double)(1.0f / sqrtf(f));
    else if constexpr (KID == PBB_KERNEL_ONEOVERR2) return (double)(1.0f / f);
    else if constexpr (KID == PBB_KERNEL_GAUSSIAN) return (double)expf(-f / (float)(p.p[0] * p.p[0]));
    else if constexpr (KID == PBB_KERNEL_EXPONENTIAL) return p.p[1] * (double)expf(-sqrtf(f) / (float)p.p[0]);
    else if constexpr (KID == PBB_KERNEL_SOFT_LAPLACIAN) return (double)(1.0f / sqrtf(f + (float)p.p[0]));
    else if constexpr (KID == PBB_KERNEL_LOGARITHM) return r2 == 0 ? 0.0 : (double)(0.5f * logf(f));
    else if constexpr (KID == PBB_KERNEL_THIN_PLATE) return r2 == 0 ? 0.0 : r2 * (double)(0.5f * logf(f));
    else if constexpr (KID == PBB_KERNEL_EXP_ANISO)
        return p.p[0] * (double)expf(-sqrtf((float)(p.p[1] * dx * dx + p.p[2] * dy * dy + p.p[3] * dz * dz)));
    else return keval<KID>(dx, dy, dz, p);  // polynomial and rational ones: FP64 is as cheap
}

// S_m(u), m < n: Chebyshev interpolant by Clenshaw (H2_3D_Tree.cpp:830-879)
__device__ __forceinline__ void sn_eval(int n, const double *__restrict__ Tkz, double u, double *S)
{
    const double pfac = 2.0 / n;
    for (int m = 0; m < n; m++) {
        const double *Tk = Tkz + m * n;
        double d0 = 0, d1 = 0;
        for (int j = n - 1; j > 0; j--) {
            double d2 = d0;
            d0 = 2.0 * u * d0 - d1 + Tk[j];
            d1 = d2;
        }
        S[m] = pfac * (u * d0 - d1 + 0.5 * Tk[0]);
    }
}

// S_m(u) for m < n written to dst[m * stride]
__device__ __forceinline__ void sn_eval_to(int n, const double *__restrict__ Tkz, double u, double *dst, int stride)
{
    const double pfac = 2.0 / n;
    for (int m = 0; m < n; m++) {
        const double *Tk = Tkz + m * n;
        double d0 = 0, d1 = 0;
        for (int j = n - 1; j > 0; j--) {
            double d2 = d0;
            d0 = 2.0 * u * d0 - d1 + Tk[j];
            d1 = d2;
        }
        dst[m * stride] = pfac * (u * d0 - d1 + 0.5 * Tk[0]);
    }
}

// ---------------------------------------------------------------------------
// ws[c*N + k] = w[c*w_n + j] with j = perm[k] - w_lo when 0 <= j < w_n,
// else 0: the points that carry no weight (the targets of a plan whose
// sources are not its targets) enter the sums with weight zero
__global__ void gather_weights(const double *__restrict__ w, const int32_t *__restrict__ perm, int64_t N,
                               int ncols, double *__restrict__ ws, int64_t w_lo, int64_t w_n)
{
    int64_t total = N * ncols;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total;
         q += (int64_t)gridDim.x * blockDim.x) {
        int64_t c = q / N, k = q - c * N;
        const int64_t j = perm[k] - w_lo;
        ws[q] = (uint64_t)j < (uint64_t)w_n ? w[c * w_n + j] : 0.0;
    }
}

// wsT[k*ncols + c], the same values point-major (for the near field)
__global__ void gather_weights_t(const double *__restrict__ w, const int32_t *__restrict__ perm, int64_t N,
                                 int ncols, double *__restrict__ wsT, int64_t w_lo, int64_t w_n)
{
    int64_t total = N * ncols;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total;
         q += (int64_t)gridDim.x * blockDim.x) {
        int64_t k = q / ncols, c = q - k * ncols;
        const int64_t j = perm[k] - w_lo;
        wsT[q] = (uint64_t)j < (uint64_t)w_n ? w[c * w_n + j] : 0.0;
    }
}

// The same wsT in two coalesced steps: wT[j*ncols + c] = w[c*w_n + j] (a
// transpose through LDS tiles of 32 points x 32 columns), then whole rows
// wsT[k] = wT[perm[k] - w_lo] (zero rows for points outside the range).
__global__ __launch_bounds__(256) void transpose_weights(const double *__restrict__ w, int64_t w_n, int ncols,
                                                         double *__restrict__ wT)
{
    __shared__ double tile[32][33];
    const int64_t j0 = (int64_t)blockIdx.x * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 8 rows of 32 lanes
    for (int c0 = 0; c0 < ncols; c0 += 32) {
        __syncthreads();
        for (int c = ty; c < 32; c += 8)
            tile[c][tx] = c0 + c < ncols && j0 + tx < w_n ? w[(int64_t)(c0 + c) * w_n + j0 + tx] : 0.0;
        __syncthreads();
        for (int j = ty; j < 32; j += 8)
            if (j0 + j < w_n && c0 + tx < ncols) wT[(j0 + j) * ncols + c0 + tx] = tile[tx][j];
    }
}

__global__ void gather_rows(const double *__restrict__ wT, const int32_t *__restrict__ perm, int64_t N, int ncols,
                            double *__restrict__ wsT, int64_t w_lo, int64_t w_n)
{
    const int64_t total = N * ncols;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total;
         q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k = q / ncols, c = q - k * ncols;
        const int64_t j = perm[k] - w_lo;
        wsT[q] = (uint64_t)j < (uint64_t)w_n ? wT[j * ncols + c] : 0.0;
    }
}

// ---------------------------------------------------------------------------
// P2M, compute.hpp:287-323: one workgroup per non-empty leaf.
// S[(g*ncols + c)*n3 + (l1 n + l2) n + l3] = sum_j w_jc Sx_l1(j) Sy_l2(j) Sz_l3(j)
constexpr int P2M_PTS = 32;
constexpr int P2M_R = 16;

__global__ __launch_bounds__(256) void p2m_fp64(P2MArgs a)
{
    __shared__ double sS[3][16][P2M_PTS];
    __shared__ double sW[64][P2M_PTS];
    const int b = blockIdx.x;
    const int n = a.n, n3 = n * n * n, tid = threadIdx.x;
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0;
    const uint32_t cc = (uint32_t)a.coord[b];
    const double cen[3] = {a.ctab[cc & 1023], a.ctab[(cc >> 10) & 1023], a.ctab[(cc >> 20) & 1023]};
    const double ihalfL = 2.0 / a.len;
    const double *xyz[3] = {a.x, a.y, a.z};
    double *Sout = a.S + (size_t)(a.off + b) * a.ncols * n3;

    for (int c0 = 0; c0 < a.ncols; c0 += a.cc) {
        const int cn = min(a.cc, a.ncols - c0);
        double acc[P2M_R];
#pragma unroll
        for (int r = 0; r < P2M_R; r++) acc[r] = 0;
        for (int j0 = 0; j0 < nt; j0 += P2M_PTS) {
            const int jn = min(P2M_PTS, nt - j0);
            if (tid < 3 * P2M_PTS) {
                int p = tid % P2M_PTS, ax = tid / P2M_PTS;
                double S[16];
                double u = p < jn ? ihalfL * (xyz[ax][t0 + j0 + p] - cen[ax]) : 0.0;
                sn_eval(n, a.Tkz, u, S);
                for (int m = 0; m < n; m++) sS[ax][m][p] = p < jn ? S[m] : 0.0;
            }
            for (int q = tid; q < cn * P2M_PTS; q += 256) {
                int c = q / P2M_PTS, p = q % P2M_PTS;
                sW[c][p] = p < jn ? a.ws[(int64_t)(c0 + c) * a.N + t0 + j0 + p] : 0.0;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < P2M_R; r++) {
                int q = tid + 256 * r;
                if (q < cn * n3) {
                    int c = q / n3, l = q - c * n3;
                    int l1 = l / (n * n), l2 = (l / n) % n, l3 = l % n;
                    double s = 0;
                    for (int p = 0; p < jn; p++) s += sW[c][p] * sS[0][l1][p] * sS[1][l2][p] * sS[2][l3][p];
                    acc[r] += s;
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < P2M_R; r++) {
            int q = tid + 256 * r;
            if (q < cn * n3) Sout[(size_t)c0 * n3 + q] = acc[r];
        }
    }
}

// ---------------------------------------------------------------------------
// M2M, compute.hpp:234-283 + :956-1034: one workgroup per parent box; the
// children's expansions are contracted mode by mode (z, y, x) in LDS.
// TS: the storage type of the expansions (FP64, or FP32 in the mixed modes);
// the transfers run in FP64 either way.
template <typename TS>
__global__ __launch_bounds__(256) void m2m_fp64(M2MArgs a)
{
    extern __shared__ double lds[];
    const int n = a.n, n2 = n * n, n3 = n2 * n, tid = threadIdx.x;
    const int CC = a.cc;
    double *A = lds, *B = lds + CC * n3, *Cw = lds + 2 * CC * n3;
    for (int q = tid; q < 2 * n2; q += 256) Cw[q] = a.Cw[q];
    const int b = blockIdx.x;
    TS *Sp = (TS *)a.Sparent + (size_t)(a.off_parent + b) * a.ncols * n3;
    for (int c0 = 0; c0 < a.ncols; c0 += CC) {
        const int cn = min(CC, a.ncols - c0);
        const int tot = cn * n3;
        double acc[P2M_R];
#pragma unroll
        for (int r = 0; r < P2M_R; r++) acc[r] = 0;
        for (int o = 0; o < 8; o++) {
            const int ch = a.child[(int64_t)b * 8 + o];
            if (ch < 0) continue;
            const TS *Sc = (const TS *)a.Schild + ((size_t)(a.off_child + ch) * a.ncols + c0) * n3;
            const double *Cx = Cw + ((o >> 2) & 1) * n2, *Cy = Cw + ((o >> 1) & 1) * n2, *Cz = Cw + (o & 1) * n2;
            __syncthreads();
            for (int q = tid; q < tot; q += 256) A[q] = Sc[q];
            __syncthreads();
            for (int q = tid; q < tot; q += 256) {  // z: B[ab n + l3] = sum_k A[ab n + k] Cz[l3 n + k]
                int c = q / n3, l = q - c * n3, ab = l / n, l3 = l % n;
                const double *src = A + c * n3 + ab * n;
                double s = 0;
                for (int k = 0; k < n; k++) s += src[k] * Cz[l3 * n + k];
                B[q] = s;
            }
            __syncthreads();
            for (int q = tid; q < tot; q += 256) {  // y: A[l1,l2,l3] = sum_k B[l1,k,l3] Cy[l2 n + k]
                int c = q / n3, l = q - c * n3, l1 = l / n2, l2 = (l / n) % n, l3 = l % n;
                const double *src = B + c * n3 + l1 * n2 + l3;
                double s = 0;
                for (int k = 0; k < n; k++) s += src[k * n] * Cy[l2 * n + k];
                A[q] = s;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < P2M_R; r++) {  // x: acc[l1,l2,l3] += sum_k A[k,l2,l3] Cx[l1 n + k]
                int q = tid + 256 * r;
                if (q < tot) {
                    int c = q / n3, l = q - c * n3, l1 = l / n2, l23 = l % n2;
                    const double *src = A + c * n3 + l23;
                    double s = 0;
                    for (int k = 0; k < n; k++) s += src[k * n2] * Cx[l1 * n + k];
                    acc[r] += s;
                }
            }
        }
#pragma unroll
        for (int r = 0; r < P2M_R; r++) {
            int q = tid + 256 * r;
            if (q < tot) Sp[(size_t)c0 * n3 + q] = (TS)acc[r];
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// L2L, compute.hpp:551-587 + :798-878: one workgroup per parent box, the
// transpose of M2M added into each non-empty child.
template <typename TS>
__global__ __launch_bounds__(256) void l2l_fp64(M2MArgs a)
{
    extern __shared__ double lds[];
    const int n = a.n, n2 = n * n, n3 = n2 * n, tid = threadIdx.x;
    const int CC = a.cc;
    double *Pp = lds, *X = lds + CC * n3, *Y = lds + 2 * CC * n3, *Cw = lds + 3 * CC * n3;
    for (int q = tid; q < 2 * n2; q += 256) Cw[q] = a.Cw[q];
    const int b = blockIdx.x;
    const TS *Fp = (const TS *)a.Sparent + (size_t)(a.off_parent + b) * a.ncols * n3;
    for (int c0 = 0; c0 < a.ncols; c0 += CC) {
        const int cn = min(CC, a.ncols - c0);
        const int tot = cn * n3;
        __syncthreads();
        for (int q = tid; q < tot; q += 256) Pp[q] = Fp[(size_t)c0 * n3 + q];
        for (int o = 0; o < 8; o++) {
            const int ch = a.child[(int64_t)b * 8 + o];
            if (ch < 0) continue;
            TS *Fc = (TS *)a.Schild + ((size_t)(a.off_child + ch) * a.ncols + c0) * n3;
            const double *Cx = Cw + ((o >> 2) & 1) * n2, *Cy = Cw + ((o >> 1) & 1) * n2, *Cz = Cw + (o & 1) * n2;
            __syncthreads();
            for (int q = tid; q < tot; q += 256) {  // x: X[l1,l2,l3] = sum_k P[k,l2,l3] Cx[k n + l1]
                int c = q / n3, l = q - c * n3, l1 = l / n2, l23 = l % n2;
                const double *src = Pp + c * n3 + l23;
                double s = 0;
                for (int k = 0; k < n; k++) s += src[k * n2] * Cx[k * n + l1];
                X[q] = s;
            }
            __syncthreads();
            for (int q = tid; q < tot; q += 256) {  // y: Y[l1,l2,l3] = sum_k X[l1,k,l3] Cy[k n + l2]
                int c = q / n3, l = q - c * n3, l1 = l / n2, l2 = (l / n) % n, l3 = l % n;
                const double *src = X + c * n3 + l1 * n2 + l3;
                double s = 0;
                for (int k = 0; k < n; k++) s += src[k * n] * Cy[k * n + l2];
                Y[q] = s;
            }
            __syncthreads();
            for (int q = tid; q < tot; q += 256) {  // z: Fc[ab n + l3] += sum_k Y[ab n + k] Cz[k n + l3]
                int c = q / n3, l = q - c * n3, ab = l / n, l3 = l % n;
                const double *src = Y + c * n3 + ab * n;
                double s = 0;
                for (int k = 0; k < n; k++) s += src[k] * Cz[k * n + l3];
                Fc[q] = (TS)((double)Fc[q] + s);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// C[:, j] = alpha * A B[:, j] for j < ncol: A (M x K, stride lda, FP64), B
// (K x ncol, ldb >= K), C (ldc >= M; rows M..zrows-1 are written as zeros),
// column-major; B and C may be FP32.  Serves the proxy projection P = VTw S
// (compute.hpp:376-395) and the local expansion F = scale Uw Pf
// (compute.hpp:497-508).
// On the FP64 matrix cores: a workgroup of 4 waves computes all
// RB 16-row blocks of M x 64 columns (one 16-column block per wave), K in
// chunks of 16.  A (small, shared by every workgroup) goes through a
// double-buffered LDS tile; each lane loads its own B fragment straight from
// memory, one chunk ahead, into two register sets used in turn.  Within a
// chunk, lane group fk supplies k = 4 fk + ks at MFMA sub-step ks, so its
// four B values are consecutive in memory.  Loads are branch-free (clamped
// addresses, masked values) so that the waits on loads in flight are exact.
template <typename TB, typename TC, int RB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_mfma_f64(GemmArgs g)
{
    constexpr int NT = 256, W = 64, R = 16 * RB, KC = 16, AS = R + 2;
    constexpr int AR = (KC * R + NT - 1) / NT;
    __shared__ double As[2][KC * AS];
    const TB *B = (const TB *)g.B;
    TC *C = (TC *)g.C;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t n0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * W;
    const int nsteps = (g.K + KC - 1) / KC;
    const int fr = lane % 16, fk = lane / 16;
    const int64_t gc = n0 + wave * 16 + fr;  // this lane's B and C column
    const TB *bcol = B + (gc < g.ncol ? gc : 0) * g.ldb;
    double ra[AR];
    auto loadA = [&](int step) {
        const int k0 = step * KC;
#pragma unroll
        for (int r = 0; r < AR; r++) {
            const int q = tid + r * NT, row = q % R, gk = k0 + q / R;
            const bool ok = q < KC * R && row < g.M && gk < g.K;
            const double v = g.A[ok ? row + (int64_t)gk * g.lda : 0];
            ra[r] = ok ? v : 0.0;
        }
    };
    auto storeA = [&](int buf) {
#pragma unroll
        for (int r = 0; r < AR; r++) {
            const int q = tid + r * NT;
            if (AR * NT == KC * R || q < KC * R) As[buf][(q / R) * AS + q % R] = ra[r];
        }
    };
    auto loadB = [&](int step, double (&b)[4]) {
        const int k = step * KC + 4 * fk;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const double v = (double)bcol[min(k + e, g.K - 1)];
            b[e] = k + e < g.K ? v : 0.0;
        }
    };
    dbl4 acc[RB];
#pragma unroll
    for (int i = 0; i < RB; i++) acc[i] = dbl4{0, 0, 0, 0};
    auto run_step = [&](int step, const double (&bcur)[4], double (&bnext)[4]) {
        const int buf = step & 1;
        storeA(buf ^ 1);  // last read in step - 1, before the barrier
        loadA(min(step + 2, nsteps - 1));
        loadB(min(step + 1, nsteps - 1), bnext);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const double *a = &As[buf][(4 * fk + ks) * AS + fr];
#pragma unroll
            for (int rb_ = 0; rb_ < RB; rb_++)
                acc[rb_] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rb_ * 16], bcur[ks], acc[rb_], 0, 0, 0);
        }
        __syncthreads();
    };
    double bA[4], bB[4];
    loadA(0);
    storeA(0);
    loadA(min(1, nsteps - 1));
    loadB(0, bA);
    __syncthreads();
    for (int step = 0; step < nsteps; step += 2) {
        run_step(step, bA, bB);
        if (step + 1 < nsteps) run_step(step + 1, bB, bA);
    }
    if (gc < g.ncol && g.pairs > 0) {
        const int64_t box = gc / g.pairs;
        TC *c = C + box * g.pairs * g.ldc + 2 * (gc - box * g.pairs);
#pragma unroll
        for (int rb_ = 0; rb_ < RB; rb_++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = rb_ * 16 + fk + 4 * v;
                if (row < g.M) c[(int64_t)((row + g.row0) / 2) * 2 * g.pairs + (row & 1)] = (TC)(g.alpha * acc[rb_][v]);
            }
    } else if (gc < g.ncol) {
#pragma unroll
        for (int rb_ = 0; rb_ < RB; rb_++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = rb_ * 16 + fk + 4 * v;
                if (row < g.M) C[row + gc * g.ldc] = (TC)(g.alpha * acc[rb_][v]);
                else if (row < g.zrows) C[row + gc * g.ldc] = (TC)0;
            }
        for (int row = R; row < g.zrows; row++)  // padding rows beyond the MFMA tile
            if (fk == 0) C[row + gc * g.ldc] = (TC)0;
    }
}

// ---------------------------------------------------------------------------
// M2L, compute.hpp:401-493 + Moment2Local :880-923.  A workgroup owns TB
// target boxes of one octant class (Morton-adjacent) and the same column
// chunk of each: a W-wide output tile Pf (all r_f rows) that stays in
// registers while the 189 far directions of the class stream through:
//   Pf[:, tile] += E_d P[:, tile + d]     (empty source boxes give zeros)
// ---------------------------------------------------------------------------
// On the FP64 matrix cores (v_mfma_f64_16x16x4_f64).  The tile is W = 32*NWC
// columns; its 2*NWC waves form a 2 x NWC grid: wave (wr, wc) holds row
// blocks [wr*RBW, wr*RBW + RBW) x the two 16-column blocks of column group
// wc.  The (direction, 16-deep k chunk) steps form one software pipeline
// with one barrier per step: E chunks go through a double-buffered LDS tile;
// each lane loads the proxies of its own B fragments straight from memory,
// one step ahead, into two register sets used in turn.  Within a chunk, lane
// group fk supplies k = 4 fk + ks at MFMA sub-step ks, so its four proxy
// values are consecutive in memory.  Loads are branch-free (clamped
// addresses, masked values) so that the waits on loads in flight are exact.
// Fragment layout of the 16x16x4 FP64 MFMA (lane l of 64):
//   A[i][k]: i = l % 16, k = l / 16      B[k][j]: j = l % 16, k = l / 16
//   D[i][j]: j = l % 16, i = l / 16 + 4*v     (v = 0..3, one double each)

constexpr int TB_MAX = 16;

template <int RB, int NWC>
__global__ __launch_bounds__(NWC * 128) void m2l_mfma_f64(M2LArgs a)
{
    constexpr int NT = NWC * 128, R = 16 * RB, KC = 16, AS = R + 2, RBW = (RB + 1) / 2;
    constexpr int AR = (KC * R + NT - 1) / NT;
    __shared__ double As[2][KC * AS];
    __shared__ int s_sid[189 * TB_MAX];
    __shared__ short s_dir[189];
    __shared__ int s_nd;
    __shared__ int s_tgt[TB_MAX];
    __shared__ int s_xyz[TB_MAX][3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave & 1, wc = wave >> 1;
    const int rf = a.rf, rs = a.rs, TB = a.TB;
    const int nch = (rs + KC - 1) / KC;
    // gridDim.z row groups of R rows each (ranks above one group's rows).
    // The row groups and column chunks of one tile are adjacent in launch
    // order: they run side by side on one XCD through the same (direction,
    // k-chunk) steps and share each proxy and E chunk through its L2
    const int gyz = (int)(gridDim.y * gridDim.z);
    const int lin = xcd_tile(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x * gyz);
    const int tile = lin / gyz;
    const int rem = lin - tile * gyz, chunk = rem / (int)gridDim.z;
    const int row0 = (rem - chunk * (int)gridDim.z) * R;
    int o = 0;
    while (o < 7 && tile >= a.tile_prefix[o + 1]) o++;
    const int64_t first = a.class_start[o] + (int64_t)(tile - a.tile_prefix[o]) * TB;
    const int64_t cend = a.class_start[o + 1];
    const int c0 = chunk * a.cpt;
    const int cpt = min(a.cpt, a.ncols - c0);
    const int S = a.side;
    if (tid < TB) {
        int64_t q = first + tid;
        int t = q < cend ? a.order[q] : -1;
        s_tgt[tid] = t;
        if (t >= 0) {
            uint32_t c = (uint32_t)a.coord[t];
            s_xyz[tid][0] = c & 1023;
            s_xyz[tid][1] = (c >> 10) & 1023;
            s_xyz[tid][2] = (c >> 20) & 1023;
        }
    }
    __syncthreads();
    for (int q = tid; q < 189 * TB; q += NT) {
        const int k = q / TB, tb = q - k * TB;
        int sid = -1;
        if (s_tgt[tb] >= 0) {
            int sx = s_xyz[tb][0] + c_dirs[o][k][0], sy = s_xyz[tb][1] + c_dirs[o][k][1],
                sz = s_xyz[tb][2] + c_dirs[o][k][2];
            if (sx >= 0 && sy >= 0 && sz >= 0 && sx < S && sy < S && sz < S)
                sid = a.map[((int64_t)sx * S + sy) * S + sz];
        }
        s_sid[k * TB_MAX + tb] = sid;
    }
    __syncthreads();
    for (int k = tid; k < 189; k += NT) {  // does direction k reach any source box?
        bool any = false;
        for (int tb = 0; tb < TB; tb++) any |= s_sid[k * TB_MAX + tb] >= 0;
        s_dir[k] = any ? 1 : 0;
    }
    __syncthreads();
    if (tid == 0) {  // compact the non-empty directions in class order
        int nd = 0;
        for (int k = 0; k < 189; k++)
            if (s_dir[k]) s_dir[nd++] = (short)k;
        s_nd = nd;
    }
    __syncthreads();
    // step order: a.chunk_major (see m2l_step); in chunk-major order
    // consecutive steps gather the same proxy rows of largely the same source
    // boxes (see class_directions)
    const int nd = s_nd, nsteps = nd * nch;

    const int fr = lane % 16, fk = lane / 16;
    int btb[2], bcl[2];  // box slot and column of this lane's B column in each block
#pragma unroll
    for (int cb = 0; cb < 2; cb++) {
        const int col = wc * 32 + cb * 16 + fr;
        const int tb = col / cpt;
        btb[cb] = tb < TB ? tb : -1;
        bcl[cb] = col - tb * cpt;
    }
    double ra[AR];
    auto loadA = [&](int step) {
        int di, ch;
        m2l_step(step, nd, nch, a.chunk_major, di, ch);
        const int k = s_dir[di], k0 = ch * KC;
        const double *Ed = a.E + (size_t)c_dirs[o][k][3] * rf * rs;
#pragma unroll
        for (int r = 0; r < AR; r++) {
            const int q = tid + r * NT, row = row0 + q % R, gk = k0 + q / R;
            const bool ok = q < KC * R && row < rf && gk < rs;
            const double v = Ed[ok ? row + (size_t)gk * rf : 0];
            ra[r] = ok ? v : 0.0;
        }
    };
    auto storeA = [&](int buf) {
#pragma unroll
        for (int r = 0; r < AR; r++) {
            const int q = tid + r * NT;
            if (AR * NT == KC * R || q < KC * R) As[buf][(q / R) * AS + q % R] = ra[r];
        }
    };
    // a column without a source box loads box 0 of the level (always valid)
    // and is zeroed through the mask at its use
    auto loadB = [&](int step, double (&bn)[2][4], int &okm) {
        int di, ch;
        m2l_step(step, nd, nch, a.chunk_major, di, ch);
        const int k = s_dir[di], k0 = ch * KC + 4 * fk;
        okm = 0;
#pragma unroll
        for (int cb = 0; cb < 2; cb++) {
            const int sid0 = btb[cb] >= 0 ? s_sid[k * TB_MAX + btb[cb]] : -1;
            okm |= (sid0 >= 0) << cb;
            const double *col = a.P + ((size_t)(a.off + max(sid0, 0)) * a.ncols + c0 + bcl[cb]) * a.ldp;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const double v = col[min(k0 + e, rs - 1)];
                bn[cb][e] = k0 + e < rs ? v : 0.0;
            }
        }
    };
    dbl4 acc[RBW][2];
#pragma unroll
    for (int i = 0; i < RBW; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = dbl4{0, 0, 0, 0};
    auto run_step = [&](int step, const double (&bcur)[2][4], int okcur, double (&bnext)[2][4], int &oknext) {
        const int buf = step & 1;
        double b[2][4];
#pragma unroll
        for (int cb = 0; cb < 2; cb++) {
            const bool ok = (okcur >> cb) & 1;
#pragma unroll
            for (int e = 0; e < 4; e++) b[cb][e] = ok ? bcur[cb][e] : 0.0;
        }
        storeA(buf ^ 1);  // last read in step - 1, before the barrier
        loadA(min(step + 2, nsteps - 1));
        loadB(min(step + 1, nsteps - 1), bnext, oknext);
        // a wave whose two column blocks have no source box in this direction
        // (zero proxies) skips the step's MFMAs; the sums are unchanged
        if (__ballot(okcur != 0) != 0) {
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const double *ap = &As[buf][(4 * fk + ks) * AS + fr];
#pragma unroll
                for (int i = 0; i < RBW; i++) {
                    const int rb_ = wr * RBW + i;
                    if (rb_ >= RB) break;
                    const double av = ap[rb_ * 16];
#pragma unroll
                    for (int cb = 0; cb < 2; cb++)
                        acc[i][cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b[cb][ks], acc[i][cb], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    };
    double bA[2][4], bB[2][4];
    int okA = 0, okB = 0;
    if (nsteps > 0) {
        loadA(0);
        storeA(0);
        loadA(min(1, nsteps - 1));
        loadB(0, bA, okA);
    }
    __syncthreads();
    for (int step = 0; step < nsteps; step += 2) {
        run_step(step, bA, okA, bB, okB);
        if (step + 1 < nsteps) run_step(step + 1, bB, okB, bA, okA);
    }
#pragma unroll
    for (int cb = 0; cb < 2; cb++) {
        if (btb[cb] < 0) continue;
        const int t = s_tgt[btb[cb]];
        if (t < 0) continue;
        double *dst = a.Pf + ((size_t)(a.off + t) * a.ncols + c0 + bcl[cb]) * a.ldf;
#pragma unroll
        for (int i = 0; i < RBW; i++) {
            const int rb_ = wr * RBW + i;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = row0 + rb_ * 16 + fk + 4 * v;
                if (rb_ < RB && row < rf) dst[row] = acc[i][cb][v];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Near field, compute.hpp:590-751, as a target-owner kernel: one wavefront
// per non-empty leaf computes, for each of its targets, the L2P of the
// leaf's local expansion plus the direct sum over the points of the 27
// neighbour leaves (self included, isinf -> 0), and adds both into the
// caller's output through perm.  No partner writes, no atomics.
// The neighbours' point ranges are concatenated into one index space and
// streamed in 64-point chunks; each chunk's kernel values K(t_i, s_j) are
// evaluated once into LDS (targets in passes of up to 16), then lane
// (i, g) accumulates columns g, g+G, ... of target i (G = 64 / TT).
constexpr int NV_SRC = 32;  // source points per chunk (LDS per wave bounds occupancy)
constexpr int NV_TGT = 16;  // targets per pass
constexpr int NV_COL = 32;  // columns per pass

template <int KID>
__global__ __launch_bounds__(64) void near_fp64(NearArgs a)
{
    __shared__ double sK[NV_TGT][NV_SRC + 1];
    __shared__ double sw[NV_COL][NV_SRC + 1];
    __shared__ double sx[NV_SRC], sy[NV_SRC], sz[NV_SRC];
    __shared__ double tx[NV_TGT], ty[NV_TGT], tz[NV_TGT];
    __shared__ double sS[3][16][NV_TGT];  // S_m of each target coordinate
    __shared__ int s_start[27], s_pre[28];
    const int b = blockIdx.x, lane = threadIdx.x;
    const int n = a.n, n2 = n * n, n3 = n2 * n;
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0;
    const uint32_t cc = (uint32_t)a.coord[b];
    const int ix = cc & 1023, iy = (cc >> 10) & 1023, iz = (cc >> 20) & 1023;
    const int S = a.side;
    const double cen[3] = {a.ctab[ix], a.ctab[iy], a.ctab[iz]};
    const double ihalfL = 2.0 / a.len;
    if (lane < 27) {
        int x = ix + lane / 9 - 1, y = iy + (lane / 3) % 3 - 1, z = iz + lane % 3 - 1;
        int sb = (x >= 0 && y >= 0 && z >= 0 && x < S && y < S && z < S) ? a.map[((int64_t)x * S + y) * S + z] : -1;
        s_start[lane] = sb >= 0 ? a.leaf_start[sb] : 0;
        s_pre[lane + 1] = sb >= 0 ? a.leaf_start[sb + 1] - a.leaf_start[sb] : 0;
    }
    __syncthreads();
    if (lane == 0) {
        s_pre[0] = 0;
        for (int m = 0; m < 27; m++) s_pre[m + 1] += s_pre[m];
    }
    __syncthreads();
    const int ns = s_pre[27];

    for (int c0 = 0; c0 < a.ncols; c0 += NV_COL) {
        const int cn = min(NV_COL, a.ncols - c0);
        for (int i0 = 0; i0 < nt; i0 += NV_TGT) {
            const int tn = min(NV_TGT, nt - i0);
            const int TT = tn <= 1 ? 1 : tn <= 2 ? 2 : tn <= 4 ? 4 : tn <= 8 ? 8 : 16;
            const int G = 64 / TT;
            const int i = lane / G, g = lane % G;
            const bool active = i < tn;
            __syncthreads();
            if (lane < tn) {
                tx[lane] = a.x[t0 + i0 + lane];
                ty[lane] = a.y[t0 + i0 + lane];
                tz[lane] = a.z[t0 + i0 + lane];
            }
            __syncthreads();
            if (a.F != nullptr && lane < 3 * tn) {
                const int ti = lane / 3, ax = lane % 3;
                const double xv = ax == 0 ? tx[ti] : ax == 1 ? ty[ti] : tz[ti];
                sn_eval_to(n, a.Tkz, ihalfL * (xv - cen[ax]), &sS[ax][0][ti], NV_TGT);
            }
            __syncthreads();
            double acc[NV_COL / 4];
#pragma unroll
            for (int k = 0; k < NV_COL / 4; k++) acc[k] = 0;
            // L2P (compute.hpp:594-648)
            if (a.F != nullptr && active) {
                const double *Fb = a.F + ((size_t)(a.off + b) * a.ncols + c0) * n3;
#pragma unroll
                for (int k = 0; k < NV_COL / 4; k++) {
                    const int cl = g + G * k;
                    if (cl >= cn) break;
                    const double *F = Fb + (size_t)cl * n3;
                    double sum = 0;
                    int l = 0;
                    for (int l1 = 0; l1 < n; l1++)
                        for (int l2 = 0; l2 < n; l2++) {
                            const double t2 = sS[0][l1][i] * sS[1][l2][i];
                            for (int l3 = 0; l3 < n; l3++) sum += F[l++] * t2 * sS[2][l3][i];
                        }
                    acc[k] += sum;
                }
            }
            // P2P over the concatenated neighbour points (compute.hpp:650-737)
            for (int j0 = 0; j0 < ns; j0 += NV_SRC) {
                const int jn = min(NV_SRC, ns - j0);
                __syncthreads();
                if (lane < jn) {
                    const int q = j0 + lane;
                    int m = 0;
                    while (s_pre[m + 1] <= q) m++;
                    const int gi = s_start[m] + q - s_pre[m];
                    sx[lane] = a.x[gi];
                    sy[lane] = a.y[gi];
                    sz[lane] = a.z[gi];
                    for (int c = 0; c < cn; c++) sw[c][lane] = a.ws[(int64_t)(c0 + c) * a.N + gi];
                }
                __syncthreads();
                for (int q = lane; q < TT * NV_SRC; q += 64) {
                    const int ii = q / NV_SRC, jj = q % NV_SRC;
                    double kv = 0.0;
                    if (ii < tn && jj < jn) {
                        kv = keval<KID>(sx[jj] - tx[ii], sy[jj] - ty[ii], sz[jj] - tz[ii], a.kp);
                        if (isinf(kv)) kv = 0.0;
                    }
                    sK[ii][jj] = kv;
                }
                __syncthreads();
                if (active) {
                    for (int jj = 0; jj < jn; jj++) {
                        const double kv = sK[i][jj];
#pragma unroll
                        for (int k = 0; k < NV_COL / 4; k++) {
                            const int cl = g + G * k;
                            if (cl < cn) acc[k] += kv * sw[cl][jj];
                        }
                    }
                }
            }
            const int64_t oi = active ? a.perm[t0 + i0 + i] - a.out_lo : -1;
            if ((uint64_t)oi < (uint64_t)a.out_n) {
#pragma unroll
                for (int k = 0; k < NV_COL / 4; k++) {
                    const int cl = g + G * k;
                    if (cl < cn) a.out[(int64_t)(c0 + cl) * a.out_n + oi] += acc[k];
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Near field in two kernels, for Chebyshev orders known at compile time.
//   l2p_fp64  L2P (compute.hpp:594-648): lp[k*ncols + c] = sum_l S_l(x_k)
//             F[c][l] for the targets k of each leaf, point-major, sorted
//             order.  8 columns of the leaf's F at a time are staged in LDS
//             with coalesced loads; lanes (target, column, part) split the
//             n^3 sum and reduce across the parts, so that leaves of one or
//             two points keep every lane busy.
//   p2p_*     P2P + scatter on top of lp (below)

constexpr int L2P_CC = 8;    // columns of F staged per step
constexpr int L2P_TGT = 32;  // targets per pass

// one level of the direct downward pass: one workgroup per segment of at
// most L2P_SEG points of one box; writes (or adds to) lp[k*ncols + c]
template <int N, typename TF>
__global__ __launch_bounds__(256) void l2p_fp64(DownArgs a)
{
    constexpr int N2 = N * N, N3 = N2 * N, FS = N3 + 1;
    __shared__ double Fs[L2P_CC * FS];
    __shared__ double sS[3][N][L2P_TGT];
    const int tid = threadIdx.x;
    const int b = a.seg_box[blockIdx.x], p0 = a.seg_p0[blockIdx.x];
    const int p1 = min(p0 + L2P_SEG, a.pstart[b + 1]);
    const uint32_t cc = (uint32_t)a.coord[b];
    const double ihalfL = 2.0 / a.len;
    const TF *Fb = (const TF *)a.F + (size_t)(a.off + b) * a.ncols * N3;
    for (int c0 = 0; c0 < a.ncols; c0 += L2P_CC) {
        const int cn = min(L2P_CC, a.ncols - c0);
        __syncthreads();  // the previous step's readers of Fs and sS are done
        for (int q = tid; q < cn * N3; q += 256) {
            const int qc = q / N3;
            Fs[qc * FS + q - qc * N3] = (double)Fb[(size_t)c0 * N3 + q];
        }
        for (int i0 = p0; i0 < p1; i0 += L2P_TGT) {
            const int tn = min(L2P_TGT, p1 - i0);
            const int tp = tn <= 1 ? 1 : tn <= 2 ? 2 : tn <= 4 ? 4 : tn <= 8 ? 8 : tn <= 16 ? 16 : 32;
            const int P = 32 / tp;  // parts per (target, column): tp * 8 * P = 256
            const int p = tid % P, c = (tid / P) % L2P_CC, i = tid / (P * L2P_CC);
            if (i0 != p0) __syncthreads();  // the previous chunk's readers of sS are done
            if (tid < 3 * L2P_TGT) {
                const int ti = tid % L2P_TGT, ax = tid / L2P_TGT;
                if (ti < tn) {
                    const double *xa = ax == 0 ? a.x : ax == 1 ? a.y : a.z;
                    const double cen = a.ctab[(cc >> (10 * ax)) & 1023];
                    double S[N];
                    sn_eval_n<N>(a.Tkz, ihalfL * (xa[i0 + ti] - cen), S);
#pragma unroll
                    for (int m = 0; m < N; m++) sS[ax][m][ti] = S[m];
                }
            }
            __syncthreads();
            const bool active = i < tn && c < cn;
            double s = 0.0;
            if (active) {
                double Sz[N];
#pragma unroll
                for (int m = 0; m < N; m++) Sz[m] = sS[2][m][i];
                for (int l12 = p; l12 < N2; l12 += P) {
                    const int l1 = l12 / N, l2 = l12 - l1 * N;
                    const double *f = &Fs[c * FS + l12 * N];
                    double s3 = 0.0;
#pragma unroll
                    for (int l3 = 0; l3 < N; l3++) s3 += f[l3] * Sz[l3];
                    s += sS[0][l1][i] * sS[1][l2][i] * s3;
                }
            }
            for (int o = 1; o < P; o <<= 1) s += __shfl_xor(s, o);
            if (active && p == 0) {
                double *dst = a.lp + (int64_t)(i0 + i) * a.ncols + c0 + c;
                *dst = a.accumulate ? *dst + s : s;
            }
        }
    }
}

// The same evaluation with FP32 local expansions (the mixed modes): all
// columns of a box's F staged at once (32 per step, 16 from order 7), as
// FP32 in LDS, so that a box with few points costs one load of F and two
// barriers; lanes take (target, column) pairs of 8 targets at a time and
// each sums the whole n^3 expansion in FP64.
template <int N>
__global__ __launch_bounds__(256, 5) void l2p_f32(DownArgs a)
{
    constexpr int N2 = N * N, N3 = N2 * N, FS = N3 + 1;
    constexpr int CC = N <= 6 ? 32 : 16, TG = 256 / CC;
    __shared__ float Fs[CC * FS];
    __shared__ double sS[3][N][TG];
    const int tid = threadIdx.x;
    const int b = a.seg_box[blockIdx.x], p0 = a.seg_p0[blockIdx.x];
    const int p1 = min(p0 + L2P_SEG, a.pstart[b + 1]);
    const uint32_t cc = (uint32_t)a.coord[b];
    const double ihalfL = 2.0 / a.len;
    const float *Fb = (const float *)a.F + (size_t)(a.off + b) * a.ncols * N3;
    const int i = tid / CC, c = tid % CC;
    for (int c0 = 0; c0 < a.ncols; c0 += CC) {
        const int cn = min(CC, a.ncols - c0);
        __syncthreads();  // the previous step's readers of Fs and sS are done
        for (int q = tid; q < cn * N3; q += 256) {
            const int qc = q / N3;
            Fs[qc * FS + q - qc * N3] = Fb[(size_t)c0 * N3 + q];
        }
        for (int i0 = p0; i0 < p1; i0 += TG) {
            const int tn = min(TG, p1 - i0);
            if (i0 != p0) __syncthreads();  // the previous chunk's readers of sS are done
            if (tid < 3 * TG) {
                const int ti = tid % TG, ax = tid / TG;
                if (ti < tn) {
                    const double *xa = ax == 0 ? a.x : ax == 1 ? a.y : a.z;
                    const double cen = a.ctab[(cc >> (10 * ax)) & 1023];
                    double S[N];
                    sn_eval_n<N>(a.Tkz, ihalfL * (xa[i0 + ti] - cen), S);
#pragma unroll
                    for (int m = 0; m < N; m++) sS[ax][m][ti] = S[m];
                }
            }
            __syncthreads();
            if (i < tn && c < cn) {
                double Sz[N];
#pragma unroll
                for (int m = 0; m < N; m++) Sz[m] = sS[2][m][i];
                const float *f = &Fs[c * FS];
                double s = 0.0;
                for (int l1 = 0; l1 < N; l1++) {
                    const double s1 = sS[0][l1][i];
                    double s2 = 0.0;
#pragma unroll
                    for (int l2 = 0; l2 < N; l2++) {
                        double s3 = 0.0;
#pragma unroll
                        for (int l3 = 0; l3 < N; l3++) s3 += (double)f[(l1 * N + l2) * N + l3] * Sz[l3];
                        s2 += sS[1][l2][i] * s3;
                    }
                    s += s1 * s2;
                }
                double *dst = a.lp + (int64_t)(i0 + i) * a.ncols + c0 + c;
                *dst = a.accumulate ? *dst + s : s;
            }
        }
    }
}

// Direct upward pass.  P2M at the leaves followed by M2M (compute.hpp:
// 234-333, :956-1034) equals P2M at every level straight from the points:
// the child-to-parent transfer interpolates the parent's Chebyshev
// polynomials S_m, which have degree n-1, at the child's nodes, which is
// exact.  A work item is a box of levels 2..L, or a segment of P2M_SEG points
// of a larger box.
// A box's expansion is the matrix product
//   S[(l2, l3), (c, l1)] = sum_p [Sy_l2(p) Sz_l3(p)] [w_pc Sx_l1(p)],
// n^2 rows and ncols n columns, column-major as S is stored, over its points:
// on the FP64 matrix cores, 16 points to a table of S_m in LDS and 4 to a
// step.  A wave holds all row blocks x CB column blocks (9 tiles at most),
// further columns are other waves.  Columns for three waves and more: a
// workgroup takes an item, its waves a column range each.  Fewer: the first
// nbig items (those of the levels of many points a box) take a workgroup each,
// the points dealt to its 4 waves and their sums added up in LDS; the others
// go by fours, a wave to each, or one after another in the first way where one
// of them is large.
// Bound by the writes of S (one column: by the few waves of the coarse
// levels).  Threads that held (column, l1, l2) pencils, barriers per box, and
// now: 5k points, 1 column, order 4 21.6 -> 5.7 us; 78k points, 3 columns of
// weights on 30k, order 5 568 -> 36 us; 1M points, 8 columns, order 5 3.04 ->
// 1.26 ms; 1M clustered, 32 columns, order 6 6.40 -> 5.76 ms (FP32 expansions,
// one level 1.38 -> 0.82 ms).
template <int N, int CB, typename TS>
__global__ __launch_bounds__(256, (N * N + 15) / 16 * CB > 6 ? 2 : 3) void p2m_levels(UpArgs a)
{
    constexpr int N2 = N * N, N3 = N2 * N, RB = (N2 + 15) / 16, TP = (3 * N) | 1;
    constexpr int SMALL = 32;  // points up to which an item is one wave's
    constexpr int U_T = 4 * 16 * TP, U_ALL = U_T > 2048 ? U_T : 2048;
    __shared__ double smem[U_ALL];  // the waves' point tables, then the sums of two tiles
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fk = lane >> 4;
    const int ncols = a.ncols, J = ncols * N;
    const int j0 = (a.by_columns ? (int)blockIdx.y * 4 + wave : (int)blockIdx.y) * (16 * CB);
    double *T = smem + wave * 16 * TP;
    int r2[RB], r3[RB], cl[CB], ch[CB];  // rows' l2 and l3, columns' l1 and c
#pragma unroll
    for (int r = 0; r < RB; r++) {
        const int row = min(r * 16 + fr, N2 - 1);
        r2[r] = N + row / N;
        r3[r] = 2 * N + row % N;
    }
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
        const int j = min(j0 + cb * 16 + fr, J - 1);
        ch[cb] = j / N;
        cl[cb] = j - ch[cb] * N;
    }
    dbl4 acc[RB][CB];
    // acc += the product over points p0 + 16 (first + k step) ..., below p1
    auto sum = [&](const int4 &it, int p1, int first, int step) __attribute__((always_inline)) {
        const int li = it.x;
        const uint32_t cc = (uint32_t)a.lt.coord[li][it.y];
        const double *ctab = a.lt.ctab[li];
        const int ax = min(lane >> 4, 2);
        const double cen = ctab[(cc >> (10 * ax)) & 1023], ihalfL = 2.0 / a.lt.len[li];
        const double *xa = ax == 0 ? a.x : ax == 1 ? a.y : a.z;
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int cb = 0; cb < CB; cb++) acc[r][cb] = dbl4{0, 0, 0, 0};
        for (int q0 = it.z + 16 * first; q0 < p1; q0 += 16 * step) {
            const int jn = min(16, p1 - q0);
            double wv[4][CB];
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int cb = 0; cb < CB; cb++)
                    wv[s][cb] = 4 * s + fk < jn ? a.wsT[(int64_t)(q0 + 4 * s + fk) * ncols + ch[cb]] : 0.0;
            if (lane < 48) {
                double S[N];
#pragma unroll
                for (int m = 0; m < N; m++) S[m] = 0.0;
                if (fr < jn) sn_eval_n<N>(a.Tkz, ihalfL * (xa[q0 + fr] - cen), S);
#pragma unroll
                for (int m = 0; m < N; m++) T[fr * TP + ax * N + m] = S[m];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (4 * s >= jn) break;
                const double *t = T + (4 * s + fk) * TP;
                double av[RB], bv[CB];
#pragma unroll
                for (int r = 0; r < RB; r++) av[r] = t[r2[r]] * t[r3[r]];
#pragma unroll
                for (int cb = 0; cb < CB; cb++) bv[cb] = wv[s][cb] * t[cl[cb]];
#pragma unroll
                for (int cb = 0; cb < CB; cb++) {
                    if (cb > 0 && j0 + cb * 16 >= J) break;
#pragma unroll
                    for (int r = 0; r < RB; r++)
                        acc[r][cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[r], bv[cb], acc[r][cb], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);  // (read ahead, the tables of all steps would spill)
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
        }
    };
    // element (row, column) of the item's expansion: split boxes write FP64
    // partial sums to scratch slots, others S directly
    auto store = [&](const int4 &it, int row, int j, double v) __attribute__((always_inline)) {
        if (row >= N2 || j >= J) return;
        const size_t at = (size_t)j * N2 + row;
        if (it.w >= 0) a.scratch[(size_t)it.w * ncols * N3 + at] = v;
        else ((TS *)a.S)[(size_t)(a.lt.off[it.x] + it.y) * ncols * N3 + at] = (TS)v;
    };
    auto end = [&](const int4 &it) { return min(it.z + P2M_SEG, a.lt.pstart[it.x][it.y + 1]); };

    auto store_all = [&](const int4 &it) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int cb = 0; cb < CB; cb++)
#pragma unroll
                for (int v = 0; v < 4; v++) store(it, r * 16 + fk + 4 * v, j0 + cb * 16 + fr, acc[r][cb][v]);
    };
    const bool big = (int)blockIdx.x < a.nbig;
    const int k0 = big ? (int)blockIdx.x : a.nbig + 4 * ((int)blockIdx.x - a.nbig);
    const int k1 = big ? k0 + 1 : min(k0 + 4, a.nitems);
    bool together = big;
    for (int k = k0; k < k1 && !big; k++) together |= end(a.items[k]) - a.items[k].z > SMALL;
    if (a.by_columns || !together) {
        const int k = a.by_columns ? k0 : k0 + wave;
        if (k >= k1 || j0 >= J) return;
        const int4 it = a.items[k];
        sum(it, end(it), 0, 1);
        store_all(it);
        return;
    }
    for (int k = k0; k < k1; k++) {
        const int4 it = a.items[k];
        sum(it, end(it), wave, 4);
        // two tiles at a time: [tile][wave][v][lane]
#pragma unroll
        for (int t0 = 0; t0 < RB * CB; t0 += 2) {
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (t0 + u < RB * CB)
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        smem[(u * 4 + wave) * 256 + v * 64 + lane] = acc[(t0 + u) / CB][(t0 + u) % CB][v];
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (t0 + u < RB * CB) {
                    const double *p = smem + u * 1024 + tid;  // (tid: v = wave, and the lane)
                    store(it, (t0 + u) / CB * 16 + fk + 4 * wave, j0 + (t0 + u) % CB * 16 + fr,
                          (p[0] + p[256]) + (p[512] + p[768]));
                }
        }
        __syncthreads();
    }
}

// S of the split boxes: the sum of their segments' partial expansions, in
// segment order
template <typename TS>
__global__ void p2m_reduce(UpReduce r)
{
    const int64_t len = (int64_t)r.ncols * r.n3;
    const int64_t total = (int64_t)r.nred * len;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total;
         q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k = q / len, e = q - k * len;
        const int4 rd = r.reds[k];
        double s = 0.0;
        for (int i = 0; i < rd.z; i++) s += r.scratch[(int64_t)(rd.y + i) * len + e];
        ((TS *)r.S)[(int64_t)rd.x * len + e] = (TS)s;
    }
}

// P2P (compute.hpp:650-737) + scatter (:739-749) on top of the L2P sums lp:
// one wave per leaf (or per pass over a large leaf's targets), the largest
// first.  The neighbours' points form one index
// space, staged in LDS chunk by chunk.  Three ways to share the work, by
// columns and leaf size:
//   p2p_few    up to 8 columns: lane (i, g) takes every G-th source for target
//              i and all columns, so a kernel value is evaluated once and used
//              from a register; the G lanes of a target add up at the end.
//   p2p_small  more columns, leaves of up to 16 targets: each value goes
//              through LDS to the lanes that hold the target's columns.
//   p2p_dense  more columns, larger leaves: the matrix cores sum.
// A launch per leaf class, the passes of a large leaf one after another in one
// workgroup, left a tail of a few waves: 5k points, 1 column 200 us -> 16 us;
// 1M uniform points, 1/r, 8 columns (1e8 pairs) 1.82 -> 0.95 ms (bound by the
// VALU: 24 FP64 operations a pair and the staging of 4 points a leaf); 1M
// clustered points, Gaussian in FP32, 32 columns (1.7e9 pairs) 12.3 -> 6.8 ms
// (bound by kernel values and products, which share the SIMD's issue slots).
struct P2PRange {
    int start[27], pre[28];
};

// The leaf's neighbours: first points and, added up, their counts (wave scan)
template <class Args>
__device__ __forceinline__ void p2p_range(const Args &a, int b, P2PRange &r)
{
    const int lane = threadIdx.x;
    const uint32_t cc = (uint32_t)a.coord[b];
    const int ix = cc & 1023, iy = (cc >> 10) & 1023, iz = (cc >> 20) & 1023;
    const int S = a.side;
    int start = 0, cnt = 0;
    if (lane < 27) {
        const int x = ix + lane / 9 - 1, y = iy + (lane / 3) % 3 - 1, z = iz + lane % 3 - 1;
        const int sb = (x >= 0 && y >= 0 && z >= 0 && x < S && y < S && z < S) ? a.map[((int64_t)x * S + y) * S + z] : -1;
        if (sb >= 0) {
            start = a.leaf_start[sb];
            cnt = a.leaf_start[sb + 1] - start;
        }
        r.start[lane] = start;
    }
    int sum = cnt;
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
        const int v = __shfl_up(sum, o);
        if (lane >= o) sum += v;
    }
    if (lane < 27) r.pre[lane + 1] = sum;
    if (lane == 0) r.pre[0] = 0;
    __syncthreads();
}

// Point q of the neighbours' index space; m: the neighbour found for a
// smaller q before (0 at the start)
__device__ __forceinline__ int p2p_point(const P2PRange &r, int q, int &m)
{
    while (r.pre[m + 1] <= q) m++;
    return r.start[m] + q - r.pre[m];
}

template <int KID, int NC>
__device__ __forceinline__ void p2p_few(const NearArgs &a, const P2PRange &r, double *lds, int t0, int nt, int i0, int lg,
                                        bool f32)
{
    // lds: positions x, y, z and NC weights of 64 sources
    double *sx = lds, *sy = lds + 64, *sz = lds + 128, *sw = lds + 192;
    const int lane = threadIdx.x, G = 64 >> lg, i = lane >> (6 - lg), g = lane & (G - 1);
    const bool active = i0 + i < nt;
    const int64_t ti = t0 + (active ? i0 + i : 0);
    const double tx = a.x[ti], ty = a.y[ti], tz = a.z[ti];
    const int ns = r.pre[27], cn = a.ncols;
    double acc[NC], px = 0, py = 0, pz = 0, pw[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) acc[c] = pw[c] = 0;
    int m = 0;
    auto load = [&](int j0) {
        if (j0 + lane < ns) {
            const int64_t gi = p2p_point(r, j0 + lane, m);
            px = a.x[gi];
            py = a.y[gi];
            pz = a.z[gi];
#pragma unroll
            for (int c = 0; c < NC; c++) pw[c] = c < cn ? a.wsT[gi * cn + c] : 0.0;
        }
    };
    load(0);
    for (int j0 = 0; j0 < ns; j0 += 64) {
        const int jn = min(64, ns - j0);
        __syncthreads();  // the previous chunk is consumed
        sx[lane] = px;
        sy[lane] = py;
        sz[lane] = pz;
#pragma unroll
        for (int c = 0; c < NC; c++) sw[lane * NC + c] = pw[c];
        __syncthreads();
        load(j0 + 64);  // in flight during the sums
        if (f32) {
            for (int j = g; j < jn; j += G) {
                double kv = keval_f32<KID>(sx[j] - tx, sy[j] - ty, sz[j] - tz, a.kp);
                if (isinf(kv)) kv = 0.0;
#pragma unroll
                for (int c = 0; c < NC; c++) acc[c] += kv * sw[j * NC + c];
            }
        } else {
#pragma unroll 2
            for (int j = g; j < jn; j += G) {
                const double kv = keval0<KID>(sx[j] - tx, sy[j] - ty, sz[j] - tz, a.kp);
#pragma unroll
                for (int c = 0; c < NC; c++) acc[c] += kv * sw[j * NC + c];
            }
        }
    }
    for (int o = 1; o < G; o <<= 1) {
#pragma unroll
        for (int c = 0; c < NC; c++) acc[c] += __shfl_xor(acc[c], o);
    }
    const int64_t oi = active && g == 0 ? a.perm[ti] - a.out_lo : -1;
    if ((uint64_t)oi < (uint64_t)a.out_n) {
#pragma unroll
        for (int c = 0; c < NC; c++)
            if (c < cn) a.out[(int64_t)c * a.out_n + oi] += a.lp ? acc[c] + a.lp[ti * cn + c] : acc[c];
    }
}

constexpr int P2P_DENSE = 4;  // first leaf class (17 targets and more) of the matrix cores
constexpr int P2P_SC = 32;  // source points per LDS chunk
constexpr int P2P_NC = 32;  // columns per pass
constexpr int P2P_WS = P2P_NC + 1;

// lds: weights [P2P_SC][P2P_WS], then x, y, z of the sources, then the kernel
// values [16][P2P_SC + 1] and the targets' x, y, z
template <int KID, int TT>
__device__ __forceinline__ void p2p_small(const NearArgs &a, const P2PRange &r, double *lds, int t0, int tn, int c0)
{
    constexpr int G = 64 / TT, CPL = P2P_NC / G, WR = P2P_SC * P2P_NC / 64, KS = P2P_SC + 1;
    double *sw = lds, *sx = lds + P2P_SC * P2P_WS, *sy = sx + P2P_SC, *sz = sy + P2P_SC, *sK = sz + P2P_SC,
           *stx = sK + 16 * KS, *sty = stx + 16, *stz = sty + 16;
    const int lane = threadIdx.x, i = lane / G, g = lane % G;
    const int cn = min(P2P_NC, a.ncols - c0), ns = r.pre[27];
    const bool active = i < tn;
    const int64_t ti = t0 + (active ? i : 0);
    if (lane < tn) {
        stx[lane] = a.x[t0 + lane];
        sty[lane] = a.y[t0 + lane];
        stz[lane] = a.z[t0 + lane];
    }
    double acc[CPL];
#pragma unroll
    for (int k = 0; k < CPL; k++) {
        const int cl = g + G * k;
        acc[k] = (a.lp && active && cl < cn) ? a.lp[ti * a.ncols + c0 + cl] : 0.0;
    }
    double pw[WR], px = 0, py = 0, pz = 0;
    int m = 0;
    auto load = [&](int j0) {
        const int jn = min(P2P_SC, ns - j0);
        int gi = 0;
        if (lane < jn) {
            gi = p2p_point(r, j0 + lane, m);
            px = a.x[gi];
            py = a.y[gi];
            pz = a.z[gi];
        }
#pragma unroll
        for (int k = 0; k < WR; k++) {
            const int u = lane + 64 * k, j = u / P2P_NC, c = u % P2P_NC;
            const int gj = __shfl(gi, j);
            const double v = a.wsT[(int64_t)gj * a.ncols + c0 + min(c, cn - 1)];
            pw[k] = (j < jn && c < cn) ? v : 0.0;
        }
    };
    if (ns > 0) load(0);
    for (int j0 = 0; j0 < ns; j0 += P2P_SC) {
        const int jn = min(P2P_SC, ns - j0);
        __syncthreads();  // the previous chunk is consumed
#pragma unroll
        for (int k = 0; k < WR; k++) {
            const int u = lane + 64 * k;
            sw[(u / P2P_NC) * P2P_WS + u % P2P_NC] = pw[k];
        }
        if (lane < P2P_SC) {
            sx[lane] = px;
            sy[lane] = py;
            sz[lane] = pz;
        }
        __syncthreads();
        if (j0 + P2P_SC < ns) load(j0 + P2P_SC);  // in flight during the sums
        for (int q = lane; q < TT * P2P_SC; q += 64) {
            const int ii = q / P2P_SC, jj = q % P2P_SC;
            double kv = 0.0;
            if (ii < tn && jj < jn) kv = keval0<KID>(sx[jj] - stx[ii], sy[jj] - sty[ii], sz[jj] - stz[ii], a.kp);
            sK[ii * KS + jj] = kv;
        }
        __syncthreads();
        if (active)
            for (int jj = 0; jj < jn; jj++) {
                const double kv = sK[i * KS + jj];
#pragma unroll
                for (int k = 0; k < CPL; k++) acc[k] += kv * sw[jj * P2P_WS + g + G * k];
            }
    }
    const int64_t oi = active ? a.perm[ti] - a.out_lo : -1;
    if ((uint64_t)oi < (uint64_t)a.out_n) {
#pragma unroll
        for (int k = 0; k < CPL; k++) {
            const int cl = g + G * k;
            if (cl < cn) a.out[(int64_t)(c0 + cl) * a.out_n + oi] += acc[k];
        }
    }
}

// K (targets x sources) times W (sources x columns) is a product of 16 x 4
// blocks of K with 4 x 16 blocks of W: the A fragment of
// v_mfma_f64_16x16x4f64 holds one value per lane, so each lane evaluates the
// kernel for its (target, source) entry of every block and the matrix cores
// accumulate 16*TB targets x 16*CB columns in FP64.  FP64 matrix
// instructions keep the VALU of their SIMD busy, so the two add up: 64 pairs
// x 32 columns cost 128 cycles of products and the 64 kernel values.  KF32
// (mixed modes): the kernel values in FP32 (keval_f32), the sums still FP64.
// lds: weights [P2P_SC][P2P_WS], then x, y, z of the sources.
template <int KID, int TB, int CB, bool KF32>
__device__ __forceinline__ void p2p_dense(const NearArgs &a, const P2PRange &r, double *lds, int t0, int nt, int i0, int c0)
{
    double *sw = lds, *sx = lds + P2P_SC * P2P_WS, *sy = sx + P2P_SC, *sz = sy + P2P_SC;
    const int lane = threadIdx.x, fr = lane & 15, fk = lane >> 4;
    const int cn = min(16 * CB, a.ncols - c0), ns = r.pre[27];
    // this lane's target row fr of each 16-target block (rows past the leaf
    // repeat its last target; their sums are not stored)
    double tx[TB], ty[TB], tz[TB];
#pragma unroll
    for (int tb = 0; tb < TB; tb++) {
        const int64_t ti = t0 + min(i0 + tb * 16 + fr, nt - 1);
        tx[tb] = a.x[ti];
        ty[tb] = a.y[ti];
        tz[tb] = a.z[ti];
    }
    // accumulators: D[fk + 4v][fr] of block (tb, cb), with the L2P sums
    dbl4 acc[TB][CB];
#pragma unroll
    for (int tb = 0; tb < TB; tb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int ti = i0 + tb * 16 + fk + 4 * v, col = cb * 16 + fr;
                acc[tb][cb][v] = (a.lp && ti < nt && col < cn) ? a.lp[(int64_t)(t0 + ti) * a.ncols + c0 + col] : 0.0;
            }
    int m = 0;
    for (int j0 = 0; j0 < ns; j0 += P2P_SC) {
        const int jn = min(P2P_SC, ns - j0);
        __syncthreads();  // the previous chunk is consumed
        int gi = 0;
        if (lane < jn) {
            gi = p2p_point(r, j0 + lane, m);
            sx[lane] = a.x[gi];
            sy[lane] = a.y[gi];
            sz[lane] = a.z[gi];
        }
        constexpr int NC = 16 * CB;
#pragma unroll
        for (int k = 0; k < P2P_SC * NC / 64; k++) {
            const int u = lane + 64 * k, j = u / NC, c = u % NC;
            const int gj = __shfl(gi, j);
            const double v = a.wsT[(int64_t)gj * a.ncols + c0 + min(c, cn - 1)];
            sw[j * P2P_WS + c] = (j < jn && c < cn) ? v : 0.0;
        }
        __syncthreads();
#pragma unroll 1
        for (int k0 = 0; k0 < jn; k0 += 4) {
            const int jj = k0 + fk;  // this lane's source of the 4-block (padding sources carry zero weights)
            const int js = min(jj, jn - 1);
            const double px = sx[js], py = sy[js], pz = sz[js];
            double b[CB];
#pragma unroll
            for (int cb = 0; cb < CB; cb++) b[cb] = sw[jj * P2P_WS + cb * 16 + fr];
#pragma unroll
            for (int tb = 0; tb < TB; tb++) {
                double kv = KF32 ? keval_f32<KID>(px - tx[tb], py - ty[tb], pz - tz[tb], a.kp)
                                 : keval0<KID>(px - tx[tb], py - ty[tb], pz - tz[tb], a.kp);
                if ((KF32 && isinf(kv)) || jj >= jn) kv = 0.0;  // (padding sources add nothing)
#pragma unroll
                for (int cb = 0; cb < CB; cb++)
                    acc[tb][cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv, b[cb], acc[tb][cb], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int tb = 0; tb < TB; tb++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int ti = i0 + tb * 16 + fk + 4 * v;
            if (ti >= nt) continue;
            const int64_t oi = a.perm[t0 + ti] - a.out_lo;
            if ((uint64_t)oi >= (uint64_t)a.out_n) continue;
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                const int col = cb * 16 + fr;
                if (col < cn) a.out[(int64_t)(c0 + col) * a.out_n + oi] += acc[tb][cb][v];
            }
        }
}

// Workgroup w of a launch over the classes lo..hi: its leaf class (the largest
// leaves first, then class by class), leaf and pass of 64 targets.  Passes of
// the last class come from a list with as many entries as there are passes:
// the size of one leaf says nothing about the others.  As many for each leaf
// as the largest has, for 4096 leaves of 40 points with 20k more in one of
// them: 1.3M workgroups, nearly all empty, matvec of 1 / 16 columns 9.6 / 17.4
// ms, with the list 2.6 / 5.2 ms, gradients 14.8 / 28.9 -> 2.6 / 5.5 ms.
template <class Args>
__device__ __forceinline__ int p2p_leaf(const Args &a, int lo, int hi, int w, int &c, int &pass)
{
    c = hi;
    pass = 0;
    if (c == NEAR_CLASSES - 1) {
        if (w < a.npass) {
            if (!a.passes) return a.leaf_class[a.leaf_class_off[c] + w];
            const int2 it = a.passes[w];
            pass = it.y;
            return it.x;
        }
        w -= a.npass;
        c--;
    }
    for (; c > lo; c--) {
        const int n = a.leaf_class_off[c + 1] - a.leaf_class_off[c];
        if (w < n) break;
        w -= n;
    }
    return a.leaf_class[a.leaf_class_off[c] + w];
}

template <int KID, int NC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void p2p_few_columns(NearArgs a)
{
    __shared__ double lds[64 * (3 + NC)];
    __shared__ P2PRange r;
    int c, pass;
    const int b = p2p_leaf(a, 0, NEAR_CLASSES - 1, blockIdx.x, c, pass);
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0;
    p2p_range(a, b, r);
    p2p_few<KID, NC>(a, r, lds, t0, nt, pass * 64, c + 1, a.kf32 && c >= P2P_DENSE);
}

template <int KID>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void p2p_small_leaves(NearArgs a)
{
    __shared__ double lds[P2P_SC * (P2P_WS + 3) + 16 * (P2P_SC + 1) + 48];
    __shared__ P2PRange r;
    int c, pass;
    const int b = p2p_leaf(a, 0, P2P_DENSE - 1, blockIdx.x, c, pass);
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0, c0 = blockIdx.y * P2P_NC;
    p2p_range(a, b, r);
    switch (c) {
    case 0: p2p_small<KID, 2>(a, r, lds, t0, nt, c0); break;
    case 1: p2p_small<KID, 4>(a, r, lds, t0, nt, c0); break;
    case 2: p2p_small<KID, 8>(a, r, lds, t0, nt, c0); break;
    default: p2p_small<KID, 16>(a, r, lds, t0, nt, c0);
    }
}

template <int KID, bool KF32>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void p2p_dense_leaves(NearArgs a)
{
    __shared__ double lds[P2P_SC * (P2P_WS + 3)];
    __shared__ P2PRange r;
    int c, pass;
    const int b = p2p_leaf(a, P2P_DENSE, NEAR_CLASSES - 1, blockIdx.x, c, pass);
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0, c0 = blockIdx.y * P2P_NC;
    p2p_range(a, b, r);
    // 32 targets where no more are left, 16 columns where no more are
    const bool half = a.ncols - c0 <= 16;
    if (nt - pass * 64 <= 32) {
        if (half) p2p_dense<KID, 2, 1, KF32>(a, r, lds, t0, nt, pass * 64, c0);
        else p2p_dense<KID, 2, 2, KF32>(a, r, lds, t0, nt, pass * 64, c0);
    } else {
        if (half) p2p_dense<KID, 4, 1, KF32>(a, r, lds, t0, nt, pass * 64, c0);
        else p2p_dense<KID, 4, 2, KF32>(a, r, lds, t0, nt, pass * 64, c0);
    }
}

// ---------------------------------------------------------------------------
// Position gradients of the FMM matvec (no reference counterpart: the
// reference has no derivatives).  For each target i of a leaf:
//   g_i += sum_c v_ic [ sum_l F_c[l] grad S_l(x_i) + sum_{j near} grad_1 K(x_i, x_j) u_jc ]
// where grad S_l is the derivative of the tensor-product Chebyshev
// interpolant (S_m'(u) = (2/n) sum_k T_k(x_m) k U_{k-1}(u), times 2/len) and
// grad_1 K the kernel's gradient in its first (target) argument, summed over
// (v, F, u) = (psi, forward leaf expansions Fs, sigma), the target side, and
// (sigma, transposed-FMM leaf expansions Fp, psi), the source side (symmetric
// kernels: d/dy K(x, y) = grad_1 K(y, x)); sigma the weights, psi dL/dout.
// d = source - target: the gradient with respect to the target position is
// kgrad * d (on the axes scaled by kgrad_axis)
template <int KID>
__device__ __forceinline__ double kgrad(double dx, double dy, double dz, const KParams &p)
{
    const double r2 = dx * dx + dy * dy + dz * dz;
    double s = 0.0;
    if constexpr (KID == PBB_KERNEL_LAPLACIAN) {
        const double ri = rsqrt_inner(r2);
        return __builtin_amdgcn_class(r2, 0x264) ? 0.0 : ri * ri * ri;  // (0, infinity)
    }
    else if constexpr (KID == PBB_KERNEL_ONEOVERR2) { s = 2.0 / (r2 * r2); }
    else if constexpr (KID == PBB_KERNEL_GAUSSIAN) { const double a2 = p.p[0] * p.p[0]; s = 2.0 / a2 * exp(-div_shared(r2, a2)); }
    else if constexpr (KID == PBB_KERNEL_EXPONENTIAL) {
        const double r = sqrt(r2);
        s = p.p[1] * exp(-div_shared(r, p.p[0])) / (p.p[0] * r);
    }
    else if constexpr (KID == PBB_KERNEL_SOFT_LAPLACIAN) { const double q = rsqrt_step(r2 + p.p[0]); s = q * q * q; }
    else if constexpr (KID == PBB_KERNEL_QUADRIC || KID == PBB_KERNEL_R2) { s = -2.0; }
    else if constexpr (KID == PBB_KERNEL_INV_QUADRIC) { const double q = 1.0 / (1.0 + r2); s = 2.0 * q * q; }
    else if constexpr (KID == PBB_KERNEL_LOGARITHM) { s = -1.0 / r2; }
    else if constexpr (KID == PBB_KERNEL_THIN_PLATE) { s = -(log(r2) + 1.0); }
    else if constexpr (KID == PBB_KERNEL_EXP_ANISO) {
        const double rho = sqrt(p.p[1] * dx * dx + p.p[2] * dy * dy + p.p[3] * dz * dz);
        s = rho > 0 ? p.p[0] * exp(-rho) / rho : 0.0;
    }
    return r2 == 0.0 ? 0.0 : s;
}
template <int KID>
__device__ __forceinline__ double kgrad_axis(int axis, const KParams &p)
{
    return KID == PBB_KERNEL_EXP_ANISO ? p.p[1 + axis] : 1.0;
}

// The far part: one wave per leaf (or per pass over 64 targets of a large
// one), the leaf's expansion coefficients l over the lanes.  The columns of
// both sides are summed per coefficient first, t_l = sum_c psi_ic Fs_c[l] +
// sigma_ic Fp_c[l], so the derivative terms run once per (target, l) instead
// of once per column; rows of psi and sigma are the same for all lanes and
// come through the scalar cache.  Bound by the reads of Fs and Fp, once per
// block of FG_TGT targets.  Far and near part of both sides, before (one kernel
// per side, every derivative term per column) and now: 500k uniform points,
// soft 1/r, order 5, 4 columns 21.7 -> 1.43 ms (1.11 far: the leaves hold two
// points each, so F is read once per two targets; 0.31 near); 60k clustered
// points, Gaussian, order 6, 16 columns 16.8 -> 1.1 ms.
constexpr int FG_TGT = 4;
__global__ __launch_bounds__(64) void far_grad(NearGradArgs a)
{
    __shared__ double sS[2][3][16][FG_TGT];  // S_m, S_m' of each target coordinate
    const int lane = threadIdx.x, n = a.n, n3 = n * n * n, C = a.ncols;
    int c, pass;
    const int b = p2p_leaf(a, 0, NEAR_CLASSES - 1, blockIdx.x, c, pass);
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0;
    const uint32_t cc = (uint32_t)a.coord[b];
    const double cen[3] = {a.ctab[cc & 1023], a.ctab[(cc >> 10) & 1023], a.ctab[(cc >> 20) & 1023]};
    const double ihalfL = 2.0 / a.len;
    const double *__restrict__ Fs = a.Fs + (size_t)b * C * n3, *__restrict__ Fp = a.Fp + (size_t)b * C * n3;
    const int end = min(nt, pass * 64 + 64);
    for (int i0 = pass * 64; i0 < end; i0 += FG_TGT) {
        const int tn = min(FG_TGT, end - i0);
        __syncthreads();
        for (int q = lane; q < tn * 3 * n; q += 64) {
            const int m = q % n, ax = q / n % 3, ti = q / (3 * n);
            const double *pos = ax == 0 ? a.x : ax == 1 ? a.y : a.z;
            const double u = ihalfL * (pos[t0 + i0 + ti] - (ax == 0 ? cen[0] : ax == 1 ? cen[1] : cen[2]));
            const double *Tk = a.Tkz + m * n;
            // T_k, U_{k-1} by their recurrences; T_k' = k U_{k-1}
            double tp = 1.0, tc = u, up = 0.0, uc = 1.0, s = 0.5 * Tk[0], d = 0.0;
            for (int k = 1; k < n; k++) {
                s += Tk[k] * tc;
                d += Tk[k] * (k * uc);
                const double tn2 = 2.0 * u * tc - tp, un = 2.0 * u * uc - up;
                tp = tc; tc = tn2;
                up = uc; uc = un;
            }
            sS[0][ax][m][ti] = 2.0 / n * s;
            sS[1][ax][m][ti] = 2.0 / n * d;
        }
        __syncthreads();
        double g[FG_TGT][3];
#pragma unroll
        for (int k = 0; k < FG_TGT; k++) g[k][0] = g[k][1] = g[k][2] = 0;
        // (scalar rows; targets past the leaf repeat its last one and are not stored)
        const double *__restrict__ ps[FG_TGT], *__restrict__ sg[FG_TGT];
#pragma unroll
        for (int k = 0; k < FG_TGT; k++) {
            const int64_t r = (int64_t)(t0 + i0 + min(k, tn - 1)) * C;
            ps[k] = a.psi + r;
            sg[k] = a.sig + r;
        }
        for (int l0 = 0; l0 < n3; l0 += 64) {
            const int l = min(l0 + lane, n3 - 1);
            double t[FG_TGT];
#pragma unroll
            for (int k = 0; k < FG_TGT; k++) t[k] = 0;
#pragma unroll 4
            for (int q = 0; q < C; q++) {
                const double fs = Fs[(size_t)q * n3 + l], fp = Fp[(size_t)q * n3 + l];
#pragma unroll
                for (int k = 0; k < FG_TGT; k++) t[k] += ps[k][q] * fs + sg[k][q] * fp;
            }
            const int l1 = l / (n * n), l2 = l / n % n, l3 = l % n;
#pragma unroll
            for (int k = 0; k < FG_TGT; k++) {
                const double tk = l0 + lane < n3 ? t[k] : 0.0;
                const double sx = sS[0][0][l1][k], sy = sS[0][1][l2][k], sz = sS[0][2][l3][k];
                g[k][0] += tk * sS[1][0][l1][k] * (sy * sz);
                g[k][1] += tk * sS[1][1][l2][k] * (sx * sz);
                g[k][2] += tk * sS[1][2][l3][k] * (sx * sy);
            }
        }
#pragma unroll
        for (int k = 0; k < FG_TGT; k++)
#pragma unroll
            for (int ax = 0; ax < 3; ax++)
                for (int o = 1; o < 64; o <<= 1) g[k][ax] += __shfl_xor(g[k][ax], o);
        double mine = 0;
#pragma unroll
        for (int k = 0; k < FG_TGT; k++)
#pragma unroll
            for (int ax = 0; ax < 3; ax++) mine = lane == 3 * k + ax ? g[k][ax] : mine;
        if (lane < 3 * tn) a.grad[3 * (int64_t)a.perm[t0 + i0 + lane / 3] + lane % 3] += mine * ihalfL;
    }
}

// The near part.  A pair's gradient carries the factor
//   s_ij = sum_c psi_ic sigma_jc + sigma_ic psi_jc
// of both sides, so one evaluation of the kernel's derivative serves them.
// Small leaves (up to 16 targets): lane (i, g) takes every G-th source for
// target i; the target's rows stay in registers, the sources' in LDS.
template <int KID, int NC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void near_grad_small(NearGradArgs a)
{
    constexpr int ST = 2 * NC + 1;  // (odd: the lanes' rows start in different banks)
    __shared__ double sx[64], sy[64], sz[64], sw[64 * ST];
    __shared__ P2PRange r;
    const int lane = threadIdx.x, C = a.ncols;
    int c, pass;
    const int b = p2p_leaf(a, 0, P2P_DENSE - 1, blockIdx.x, c, pass);
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0;
    p2p_range(a, b, r);
    const int lg = c + 1, G = 64 >> lg, i = lane >> (6 - lg), g = lane & (G - 1), ns = r.pre[27];
    const bool active = i < nt;
    const int64_t ti = t0 + (active ? i : 0);
    const double tx = a.x[ti], ty = a.y[ti], tz = a.z[ti];
    double gx = 0, gy = 0, gz = 0;
    for (int c0 = 0; c0 < C; c0 += NC) {
        double vp[NC], vs[NC];
#pragma unroll
        for (int k = 0; k < NC; k++) {
            vp[k] = c0 + k < C ? a.psi[ti * C + c0 + k] : 0.0;
            vs[k] = c0 + k < C ? a.sig[ti * C + c0 + k] : 0.0;
        }
        int m = 0;
        for (int j0 = 0; j0 < ns; j0 += 64) {
            const int jn = min(64, ns - j0);
            __syncthreads();  // the previous chunk is consumed
            if (lane < jn) {
                const int64_t gi = p2p_point(r, j0 + lane, m);
                sx[lane] = a.x[gi];
                sy[lane] = a.y[gi];
                sz[lane] = a.z[gi];
#pragma unroll
                for (int k = 0; k < NC; k++) {
                    sw[lane * ST + k] = c0 + k < C ? a.sig[gi * C + c0 + k] : 0.0;
                    sw[lane * ST + NC + k] = c0 + k < C ? a.psi[gi * C + c0 + k] : 0.0;
                }
            }
            __syncthreads();
            for (int j = g; j < jn; j += G) {
                double s = 0;
#pragma unroll
                for (int k = 0; k < NC; k++) s += vp[k] * sw[j * ST + k] + vs[k] * sw[j * ST + NC + k];
                const double dx = sx[j] - tx, dy = sy[j] - ty, dz = sz[j] - tz;
                s *= kgrad<KID>(dx, dy, dz, a.kp);
                gx += s * dx;
                gy += s * dy;
                gz += s * dz;
            }
        }
    }
    for (int o = 1; o < G; o <<= 1) {
        gx += __shfl_xor(gx, o);
        gy += __shfl_xor(gy, o);
        gz += __shfl_xor(gz, o);
    }
    if (active && g == 0) {
        const int64_t oi = a.perm[ti];
        a.grad[3 * oi] += gx * kgrad_axis<KID>(0, a.kp);
        a.grad[3 * oi + 1] += gy * kgrad_axis<KID>(1, a.kp);
        a.grad[3 * oi + 2] += gz * kgrad_axis<KID>(2, a.kp);
    }
}

// Larger leaves: s is the product of the targets' rows (psi, sigma) with the
// sources' (sigma, psi), 2 NC long, which v_mfma_f64_16x16x4f64 forms for 16
// targets x 16 sources at a time; a lane then evaluates the derivative for
// its 4 pairs of a block and keeps 4 targets' sums.  The k of a fragment are
// assigned so that a lane reads NC / 2 values of one row in a piece.
template <int KID, int NC, int TB>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void near_grad_dense(NearGradArgs a)
{
    constexpr int KF = NC / 2;  // k per lane = fragments
    __shared__ P2PRange r;
    const int lane = threadIdx.x, fr = lane & 15, fk = lane >> 4, C = a.ncols;
    int c, pass;
    const int b = p2p_leaf(a, P2P_DENSE, NEAR_CLASSES - 1, blockIdx.x, c, pass);
    const int t0 = a.leaf_start[b], nt = a.leaf_start[b + 1] - t0, i0 = pass * 64 + blockIdx.y * 16 * TB;
    if (i0 >= nt) return;
    p2p_range(a, b, r);
    const int ns = r.pre[27];
    const double *__restrict__ va = fk < 2 ? a.psi : a.sig, *__restrict__ vb = fk < 2 ? a.sig : a.psi;
    const int ck = (fk & 1) * KF;  // this lane's first column of the chunk
    double tx[TB][4], ty[TB][4], tz[TB][4], gx[TB][4], gy[TB][4], gz[TB][4];
#pragma unroll
    for (int tb = 0; tb < TB; tb++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int64_t ti = t0 + min(i0 + tb * 16 + fk + 4 * v, nt - 1);
            tx[tb][v] = a.x[ti];
            ty[tb][v] = a.y[ti];
            tz[tb][v] = a.z[ti];
            gx[tb][v] = gy[tb][v] = gz[tb][v] = 0;
        }
    for (int c0 = 0; c0 < C; c0 += NC) {
        double A[TB][KF];
#pragma unroll
        for (int tb = 0; tb < TB; tb++) {
            const int64_t row = (int64_t)(t0 + min(i0 + tb * 16 + fr, nt - 1)) * C;
#pragma unroll
            for (int f = 0; f < KF; f++) A[tb][f] = c0 + ck + f < C ? va[row + c0 + ck + f] : 0.0;
        }
        int m = 0;
        double px, py, pz, B[KF];
        auto load = [&](int j0) {
            const int j = min(j0 + fr, ns - 1);
            const int64_t gi = p2p_point(r, j, m);
            px = a.x[gi];
            py = a.y[gi];
            pz = a.z[gi];
            const double *row = vb + gi * C + c0 + ck;
#pragma unroll
            for (int f = 0; f < KF; f++) B[f] = j0 + fr < ns && c0 + ck + f < C ? row[f] : 0.0;
        };
        load(0);
#pragma unroll 1
        for (int j0 = 0; j0 < ns; j0 += 16) {
            const double qx = px, qy = py, qz = pz;
            dbl4 s[TB];
#pragma unroll
            for (int tb = 0; tb < TB; tb++) {
                s[tb] = dbl4{0, 0, 0, 0};
#pragma unroll
                for (int f = 0; f < KF; f++) s[tb] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[tb][f], B[f], s[tb], 0, 0, 0);
            }
            load(j0 + 16);  // in flight during the derivatives
#pragma unroll
            for (int tb = 0; tb < TB; tb++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const double dx = qx - tx[tb][v], dy = qy - ty[tb][v], dz = qz - tz[tb][v];
                    const double w = s[tb][v] * kgrad<KID>(dx, dy, dz, a.kp);
                    gx[tb][v] += w * dx;
                    gy[tb][v] += w * dy;
                    gz[tb][v] += w * dz;
                }
        }
    }
#pragma unroll
    for (int tb = 0; tb < TB; tb++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            for (int o = 1; o < 16; o <<= 1) {
                gx[tb][v] += __shfl_xor(gx[tb][v], o);
                gy[tb][v] += __shfl_xor(gy[tb][v], o);
                gz[tb][v] += __shfl_xor(gz[tb][v], o);
            }
            const int ti = i0 + tb * 16 + fk + 4 * v;
            if (fr == 0 && ti < nt) {
                const int64_t oi = a.perm[t0 + ti];
                a.grad[3 * oi] += gx[tb][v] * kgrad_axis<KID>(0, a.kp);
                a.grad[3 * oi + 1] += gy[tb][v] * kgrad_axis<KID>(1, a.kp);
                a.grad[3 * oi + 2] += gz[tb][v] * kgrad_axis<KID>(2, a.kp);
            }
        }
}

// ---------------------------------------------------------------------------
// Direct sum (DirectCalc3D, test.hpp:18-34, isinf -> 0): a workgroup holds 64
// targets, one per lane, its 16 waves a sixteenth of one slice of the sources
// each.  A wave's source is the same for all its lanes, so positions and
// weights come through the scalar cache and cost no LDS; the VALU evaluates
// each kernel value once for NC columns.  With one slice (enough targets to
// fill the GPU) the sums go straight to out, else to part[(split*ncols + c)*T
// + i], reduced by a second kernel.
// Bound: the VALU, some 16 FP64 operations a pair.  50k x 50k points, 1/r, 1
// column: 14.3 ms with sources in LDS, a slice per wave and the library's root
// and division, 1.43 ms here (1.75e12 pairs/s; its operations alone 1.1 ms).
constexpr int DS_TGT = 64, DS_WAVES = 16;

template <int KID, int NC>
__global__ __launch_bounds__(64 * DS_WAVES) void direct_partial(DirectArgs a, int c0)
{
    __shared__ double sh[DS_WAVES][DS_TGT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t i = a.t0 + (int64_t)blockIdx.x * DS_TGT + lane;
    const int split = blockIdx.y;
    const int64_t per = (a.Ns + a.nsplit - 1) / a.nsplit;
    const int64_t s0 = split * per, s1 = min(a.Ns, s0 + per);
    const int64_t pw = s1 > s0 ? (s1 - s0 + DS_WAVES - 1) / DS_WAVES : 0;
    const int64_t j0 = s0 + wave * pw, j1 = min(s1, j0 + pw);
    const bool active = i < a.T;
    const int64_t it = active ? i : 0;
    const double xi = a.tgt[3 * it], yi = a.tgt[3 * it + 1], zi = a.tgt[3 * it + 2];
    const int cn = min(NC, a.ncols - c0);
    const double *__restrict__ src = a.src;
    const double *__restrict__ w = a.w + (int64_t)c0 * a.Ns;
    double acc[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) acc[k] = 0;
#pragma unroll 4
    for (int64_t j = j0; j < j1; j++) {
        const double kv = keval0<KID>(src[3 * j] - xi, src[3 * j + 1] - yi, src[3 * j + 2] - zi, a.kp);
#pragma unroll
        for (int k = 0; k < NC; k++) acc[k] += kv * w[(int64_t)min(k, cn - 1) * a.Ns + j];
    }
#pragma unroll
    for (int k = 0; k < NC; k++) {
        if (k >= cn) break;
        __syncthreads();
        sh[wave][lane] = acc[k];
        __syncthreads();
        if (wave == 0 && active) {
            double s = 0;
            for (int v = 0; v < DS_WAVES; v++) s += sh[v][lane];
            double *dst = a.nsplit > 1 ? a.part + (int64_t)split * a.ncols * a.T : a.out;
            dst[(int64_t)(c0 + k) * a.T + i] = s;
        }
    }
}

__global__ void direct_reduce(const double *__restrict__ part, int nsplit, int64_t total,
                              double *__restrict__ out)
{
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total;
         q += (int64_t)gridDim.x * blockDim.x) {
        double s = 0;
        for (int k = 0; k < nsplit; k++) s += part[k * total + q];
        out[q] = s;
    }
}

// ---------------------------------------------------------------------------
// launchers

void upload_dirs(const int dirs[8][189][4])
{
    check(hipMemcpyToSymbol(HIP_SYMBOL(c_dirs), dirs, sizeof(int) * 8 * 189 * 4), "hipMemcpyToSymbol(c_dirs)");
}

void launch_gather_weights(const double *w, const int32_t *perm, int64_t N, int ncols, double *ws, int64_t w_lo,
                           int64_t w_n, hipStream_t st)
{
    int64_t total = N * ncols;
    int blocks = (int)std::min<int64_t>((total + 255) / 256, 65536);
    gather_weights<<<blocks, 256, 0, st>>>(w, perm, N, ncols, ws, w_lo, w_n);
    check(hipGetLastError(), "gather_weights");
}

void launch_gather_weights_t(const double *w, const int32_t *perm, int64_t N, int ncols, double *wsT,
                             int64_t w_lo, int64_t w_n, hipStream_t st)
{
    int64_t total = N * ncols;
    if (total <= 0) return;
    int blocks = (int)std::min<int64_t>((total + 255) / 256, 65536);
    gather_weights_t<<<blocks, 256, 0, st>>>(w, perm, N, ncols, wsT, w_lo, w_n);
    check(hipGetLastError(), "gather_weights_t");
}

void launch_gather_rows_t(const double *w, const int32_t *perm, int64_t N, int ncols, double *wT, double *wsT,
                          int64_t w_lo, int64_t w_n, hipStream_t st)
{
    if (N * ncols <= 0 || w_n <= 0) return;
    const int64_t tb = (w_n + 31) / 32;
    if (tb > INT32_MAX) fail(PBB_ERR_UNSUPPORTED, "too many points for the weight transpose");
    transpose_weights<<<(unsigned)tb, 256, 0, st>>>(w, w_n, ncols, wT);
    check(hipGetLastError(), "transpose_weights");
    const int blocks = (int)std::min<int64_t>((N * ncols + 255) / 256, 65536);
    gather_rows<<<blocks, 256, 0, st>>>(wT, perm, N, ncols, wsT, w_lo, w_n);
    check(hipGetLastError(), "gather_rows");
}

void launch_p2m(const P2MArgs &a, int nleaf, hipStream_t st)
{
    if (nleaf <= 0) return;
    p2m_fp64<<<nleaf, 256, 0, st>>>(a);
    check(hipGetLastError(), "p2m_fp64");
}

void launch_m2m(const M2MArgs &a, int nparent, hipStream_t st)
{
    if (nparent <= 0) return;
    size_t lds = sizeof(double) * (2 * (size_t)a.cc * a.n * a.n * a.n + 2 * a.n * a.n);
    if (a.s32) m2m_fp64<float><<<nparent, 256, lds, st>>>(a);
    else m2m_fp64<double><<<nparent, 256, lds, st>>>(a);
    check(hipGetLastError(), "m2m_fp64");
}

void launch_l2l(const M2MArgs &a, int nparent, hipStream_t st)
{
    if (nparent <= 0) return;
    size_t lds = sizeof(double) * (3 * (size_t)a.cc * a.n * a.n * a.n + 2 * a.n * a.n);
    if (a.s32) l2l_fp64<float><<<nparent, 256, lds, st>>>(a);
    else l2l_fp64<double><<<nparent, 256, lds, st>>>(a);
    check(hipGetLastError(), "l2l_fp64");
}

void launch_gemm(const GemmArgs &args, hipStream_t st)
{
    GemmArgs g = args;
    if (g.ncol <= 0) return;
    if (g.ldb < g.K || g.ldc < g.M) fail(PBB_ERR_INTERNAL, "gemm: leading dimension too small");
    if (g.lda == 0) g.lda = g.M;
    if (g.zrows == 0) g.zrows = g.ldc;
    // at most 16 row blocks (256 rows) per launch: larger products run as row
    // ranges of about equal size
    const int rball = (g.M + 15) / 16, nparts = (rball + 15) / 16, rb = (rball + nparts - 1) / nparts;
    dim3 grid((unsigned)((g.ncol + 63) / 64));
    const int M = g.M, zrows = g.zrows;
    for (int part = 0; part < nparts; part++) {
        const int r0 = part * rb * 16;
        g.M = std::min(M - r0, rb * 16);
        g.zrows = part + 1 < nparts ? g.M : zrows - r0;
        g.A = args.A + r0;
        g.row0 = g.pairs > 0 ? r0 : 0;
        const int c0 = g.pairs > 0 ? 0 : r0;
        g.C = g.c_f32 ? (void *)((float *)args.C + c0) : (void *)((double *)args.C + c0);
#define PBB_G(R)                                                                                   \
    case R:                                                                                        \
        if (!g.b_f32 && !g.c_f32) gemm_mfma_f64<double, double, R><<<grid, 256, 0, st>>>(g);       \
        else if (!g.b_f32 && g.c_f32) gemm_mfma_f64<double, float, R><<<grid, 256, 0, st>>>(g);    \
        else if (g.b_f32 && !g.c_f32) gemm_mfma_f64<float, double, R><<<grid, 256, 0, st>>>(g);    \
        else gemm_mfma_f64<float, float, R><<<grid, 256, 0, st>>>(g);                              \
        break;
        switch (rb) {
            PBB_G(1) PBB_G(2) PBB_G(3) PBB_G(4) PBB_G(5) PBB_G(6) PBB_G(7) PBB_G(8) PBB_G(9) PBB_G(10) PBB_G(11)
            PBB_G(12) PBB_G(13) PBB_G(14) PBB_G(15) PBB_G(16)
        }
#undef PBB_G
        check(hipGetLastError(), "gemm_mfma_f64");
    }
}

void launch_m2l(const M2LArgs &a, int ntiles, int ncolchunks, hipStream_t st)
{
    if (ntiles <= 0) return;
    // at most 16 row blocks (256 rows) per workgroup: larger ranks run as
    // row groups of equal size
    const int rball = (a.rf + 15) / 16, ngroups = (rball + 15) / 16, rb = (rball + ngroups - 1) / ngroups;
    dim3 grid((unsigned)ntiles, (unsigned)ncolchunks, (unsigned)ngroups);
    const int w = a.TB * a.cpt;  // tile width chosen by the caller: at most 128 columns
    if (w > 128) fail(PBB_ERR_INTERNAL, "FP64 M2L tile wider than 128 columns");
#define PBB_M2L_CASE(R)                                                        \
    case R:                                                                    \
        if (w > 64) m2l_mfma_f64<R, 4><<<grid, 512, 0, st>>>(a);               \
        else if (w > 32) m2l_mfma_f64<R, 2><<<grid, 256, 0, st>>>(a);          \
        else m2l_mfma_f64<R, 1><<<grid, 128, 0, st>>>(a);                      \
        break;
    switch (rb) {
        PBB_M2L_CASE(1) PBB_M2L_CASE(2) PBB_M2L_CASE(3) PBB_M2L_CASE(4) PBB_M2L_CASE(5) PBB_M2L_CASE(6)
        PBB_M2L_CASE(7) PBB_M2L_CASE(8) PBB_M2L_CASE(9) PBB_M2L_CASE(10) PBB_M2L_CASE(11)
        PBB_M2L_CASE(12) PBB_M2L_CASE(13) PBB_M2L_CASE(14) PBB_M2L_CASE(15) PBB_M2L_CASE(16)
    default: fail(PBB_ERR_INTERNAL, "M2L row group above 256 rows");
    }
#undef PBB_M2L_CASE
    check(hipGetLastError(), "m2l_mfma_f64");
}

void launch_near(const NearArgs &a, int kid, int nleaf, hipStream_t st)
{
    if (nleaf <= 0) return;
#define PBB_NEAR_CASE(K)                                  \
    case K:                                               \
        near_fp64<K><<<nleaf, 64, 0, st>>>(a);            \
        break;
    switch (kid) {
        PBB_NEAR_CASE(PBB_KERNEL_LAPLACIAN) PBB_NEAR_CASE(PBB_KERNEL_ONEOVERR2) PBB_NEAR_CASE(PBB_KERNEL_GAUSSIAN)
        PBB_NEAR_CASE(PBB_KERNEL_EXPONENTIAL) PBB_NEAR_CASE(PBB_KERNEL_SOFT_LAPLACIAN)
        PBB_NEAR_CASE(PBB_KERNEL_QUADRIC) PBB_NEAR_CASE(PBB_KERNEL_INV_QUADRIC)
        PBB_NEAR_CASE(PBB_KERNEL_LOGARITHM) PBB_NEAR_CASE(PBB_KERNEL_THIN_PLATE) PBB_NEAR_CASE(PBB_KERNEL_R2)
        PBB_NEAR_CASE(PBB_KERNEL_CONSTANT) PBB_NEAR_CASE(PBB_KERNEL_EXP_ANISO)
    default: fail(PBB_ERR_UNSUPPORTED, "no device functor for this kernel id");
    }
#undef PBB_NEAR_CASE
    check(hipGetLastError(), "near_fp64");
}

namespace {
// Workgroups of one wave over the dense classes, and the limit of a grid:
// below 2^32 threads (the passes are at most N / 64 and one a leaf).
template <class Args>
int64_t near_dense_passes(const Args &a)
{
    const int64_t dense = (int64_t)a.npass + a.leaf_class_off[NEAR_CLASSES - 1] - a.leaf_class_off[P2P_DENSE];
    if (dense + a.leaf_class_off[P2P_DENSE] > UINT32_MAX / 64) fail(PBB_ERR_UNSUPPORTED, "too many near-field passes");
    return dense;
}
}  // namespace

bool launch_near_split(const NearArgs &args, int kid, int nleaf, hipStream_t st)
{
    NearArgs a = args;
    if (a.n < 4 || a.n > 8) return false;
    if (nleaf <= 0) return true;
    const int few = a.leaf_class_off[P2P_DENSE];
    const int64_t dense = near_dense_passes(a);
    const unsigned cols = (unsigned)((a.ncols + P2P_NC - 1) / P2P_NC);
    // (the whole call's columns choose, so that a chunk of them sums in the same order)
    const dim3 all((unsigned)(dense + few)), gs((unsigned)few, cols), gd((unsigned)dense, cols);
#define PBB_P2P_CASE(K)                                                        \
    case K:                                                                    \
        if (a.all <= 8 && a.ncols <= 1) p2p_few_columns<K, 1><<<all, 64, 0, st>>>(a); \
        else if (a.all <= 8 && a.ncols <= 2) p2p_few_columns<K, 2><<<all, 64, 0, st>>>(a); \
        else if (a.all <= 8 && a.ncols <= 4) p2p_few_columns<K, 4><<<all, 64, 0, st>>>(a); \
        else if (a.all <= 8) p2p_few_columns<K, 8><<<all, 64, 0, st>>>(a);     \
        else {                                                                 \
            if (dense && a.kf32) p2p_dense_leaves<K, true><<<gd, 64, 0, st>>>(a); \
            else if (dense) p2p_dense_leaves<K, false><<<gd, 64, 0, st>>>(a);  \
            if (few) p2p_small_leaves<K><<<gs, 64, 0, st>>>(a);                \
        }                                                                      \
        break;
    switch (kid) {
        PBB_P2P_CASE(PBB_KERNEL_LAPLACIAN) PBB_P2P_CASE(PBB_KERNEL_ONEOVERR2) PBB_P2P_CASE(PBB_KERNEL_GAUSSIAN)
        PBB_P2P_CASE(PBB_KERNEL_EXPONENTIAL) PBB_P2P_CASE(PBB_KERNEL_SOFT_LAPLACIAN)
        PBB_P2P_CASE(PBB_KERNEL_QUADRIC) PBB_P2P_CASE(PBB_KERNEL_INV_QUADRIC)
        PBB_P2P_CASE(PBB_KERNEL_LOGARITHM) PBB_P2P_CASE(PBB_KERNEL_THIN_PLATE) PBB_P2P_CASE(PBB_KERNEL_R2)
        PBB_P2P_CASE(PBB_KERNEL_CONSTANT) PBB_P2P_CASE(PBB_KERNEL_EXP_ANISO)
    default: fail(PBB_ERR_UNSUPPORTED, "no device functor for this kernel id");
    }
#undef PBB_P2P_CASE
    check(hipGetLastError(), "p2p");
    return true;
}

bool launch_p2m_levels(const UpArgs &args, int nitems, const UpReduce &r, hipStream_t st)
{
    UpArgs a = args;
    a.nitems = nitems;
    a.nbig = std::min(a.nbig, nitems);
    if (a.n < 4 || a.n > 8) return false;
    if (nitems <= 0) return true;
    // column blocks of a wave: those of the call, or what 9 tiles hold
    const int blocks = (a.ncols * a.n + 15) / 16;
    // (the whole call's columns choose how the points are summed, so that a
    // chunk of them gives the same bits)
    const int whole = (a.all * a.n + 15) / 16, most = a.n == 4 ? 4 : a.n <= 6 ? 3 : 2;
    a.by_columns = whole > 2 * most;
    if (a.by_columns) a.nbig = nitems;
    auto grid = [&](int cb) {
        const int ways = (blocks + cb - 1) / cb;
        return dim3((unsigned)(a.nbig + (nitems - a.nbig + 3) / 4), (unsigned)(a.by_columns ? (ways + 3) / 4 : ways));
    };
#define PBB_P2M_CB(N, CB, TS)                                                                             \
    do {                                                                                                  \
        const dim3 g = grid(CB);                                                                          \
        p2m_levels<N, CB, TS><<<g, 256, 0, st>>>(a);                                                      \
    } while (0)
#define PBB_P2M_N(N, CB, TS)                                                                              \
    case N:                                                                                               \
        if (blocks <= 1) PBB_P2M_CB(N, 1, TS);                                                            \
        else if (blocks <= 2) PBB_P2M_CB(N, 2, TS);                                                       \
        else PBB_P2M_CB(N, CB, TS);                                                                       \
        break;
#define PBB_P2M(TS)                                                                                       \
    switch (a.n) {                                                                                        \
        PBB_P2M_N(4, 4, TS) PBB_P2M_N(5, 3, TS) PBB_P2M_N(6, 3, TS) PBB_P2M_N(7, 2, TS) PBB_P2M_N(8, 2, TS) \
    }
    if (a.s32) { PBB_P2M(float) } else { PBB_P2M(double) }
#undef PBB_P2M
#undef PBB_P2M_CB
#undef PBB_P2M_N
    check(hipGetLastError(), "p2m_levels");
    if (r.nred > 0) {
        const int64_t total = (int64_t)r.nred * r.ncols * r.n3;
        const int blocks = (int)std::min<int64_t>((total + 255) / 256, 65536);
        if (r.s32) p2m_reduce<float><<<blocks, 256, 0, st>>>(r);
        else p2m_reduce<double><<<blocks, 256, 0, st>>>(r);
        check(hipGetLastError(), "p2m_reduce");
    }
    return true;
}

bool launch_l2p_level(const DownArgs &a, int nseg, hipStream_t st)
{
    if (a.n < 4 || a.n > 8) return false;
    if (nseg <= 0) return true;
    if (a.f32) {
        switch (a.n) {
        case 4: l2p_f32<4><<<nseg, 256, 0, st>>>(a); break;
        case 5: l2p_f32<5><<<nseg, 256, 0, st>>>(a); break;
        case 6: l2p_f32<6><<<nseg, 256, 0, st>>>(a); break;
        case 7: l2p_f32<7><<<nseg, 256, 0, st>>>(a); break;
        default: l2p_f32<8><<<nseg, 256, 0, st>>>(a); break;
        }
        check(hipGetLastError(), "l2p_f32");
        return true;
    }
    switch (a.n) {
    case 4: l2p_fp64<4, double><<<nseg, 256, 0, st>>>(a); break;
    case 5: l2p_fp64<5, double><<<nseg, 256, 0, st>>>(a); break;
    case 6: l2p_fp64<6, double><<<nseg, 256, 0, st>>>(a); break;
    case 7: l2p_fp64<7, double><<<nseg, 256, 0, st>>>(a); break;
    default: l2p_fp64<8, double><<<nseg, 256, 0, st>>>(a); break;
    }
    check(hipGetLastError(), "l2p_fp64");
    return true;
}

void launch_direct(const DirectArgs &args, int kid, hipStream_t st)
{
    DirectArgs a = args;
    if (a.T <= 0) return;
    // ranges of targets: a launch holds fewer than 2^32 threads, 16 a target
    constexpr int64_t RANGE = (int64_t)DS_TGT << 21;
    const int ncg = (a.ncols + 15) / 16;
    for (int64_t k = 0, n = (a.T + RANGE - 1) / RANGE * ncg; k < n; k++) {
        const int c0 = (int)(k % ncg) * 16, cn = a.ncols - c0;
        a.t0 = k / ncg * RANGE;
        dim3 grid((unsigned)((std::min(RANGE, a.T - a.t0) + DS_TGT - 1) / DS_TGT), (unsigned)a.nsplit);
#define PBB_DIRECT_CASE(K)                                                                   \
    case K:                                                                                  \
        if (cn <= 1) direct_partial<K, 1><<<grid, 64 * DS_WAVES, 0, st>>>(a, c0);            \
        else if (cn <= 4) direct_partial<K, 4><<<grid, 64 * DS_WAVES, 0, st>>>(a, c0);       \
        else direct_partial<K, 16><<<grid, 64 * DS_WAVES, 0, st>>>(a, c0);                   \
        break;
        switch (kid) {
            PBB_DIRECT_CASE(PBB_KERNEL_LAPLACIAN) PBB_DIRECT_CASE(PBB_KERNEL_ONEOVERR2)
            PBB_DIRECT_CASE(PBB_KERNEL_GAUSSIAN) PBB_DIRECT_CASE(PBB_KERNEL_EXPONENTIAL)
            PBB_DIRECT_CASE(PBB_KERNEL_SOFT_LAPLACIAN) PBB_DIRECT_CASE(PBB_KERNEL_QUADRIC)
            PBB_DIRECT_CASE(PBB_KERNEL_INV_QUADRIC) PBB_DIRECT_CASE(PBB_KERNEL_LOGARITHM)
            PBB_DIRECT_CASE(PBB_KERNEL_THIN_PLATE) PBB_DIRECT_CASE(PBB_KERNEL_R2)
            PBB_DIRECT_CASE(PBB_KERNEL_CONSTANT) PBB_DIRECT_CASE(PBB_KERNEL_EXP_ANISO)
        default: fail(PBB_ERR_UNSUPPORTED, "no device functor for this kernel id");
        }
#undef PBB_DIRECT_CASE
        check(hipGetLastError(), "direct_partial");
    }
    if (a.nsplit <= 1) return;
    int64_t total = a.T * a.ncols;
    int blocks = (int)std::min<int64_t>((total + 255) / 256, 65536);
    direct_reduce<<<blocks, 256, 0, st>>>(a.part, a.nsplit, total, a.out);
    check(hipGetLastError(), "direct_reduce");
}

void launch_near_grad(const NearGradArgs &args, int kid, int nleaf, hipStream_t st)
{
    if (nleaf <= 0) return;
    NearGradArgs a = args;
    const int few = a.leaf_class_off[P2P_DENSE];
    const int64_t dense = near_dense_passes(a);
    const bool wide = a.ncols > 4;
    if (a.Fs && dense + few) {
        far_grad<<<(unsigned)(dense + few), 64, 0, st>>>(a);
        check(hipGetLastError(), "far_grad");
    }
    // 16 x 2 targets at a time: the 64 targets of a pass in two workgroups
    const dim3 gd((unsigned)dense, 2);
#define PBB_GRAD_CASE(K)                                                          \
    case K:                                                                       \
        if (dense && wide) near_grad_dense<K, 16, 2><<<gd, 64, 0, st>>>(a);       \
        else if (dense) near_grad_dense<K, 4, 2><<<gd, 64, 0, st>>>(a);           \
        if (few && wide) near_grad_small<K, 16><<<few, 64, 0, st>>>(a);           \
        else if (few) near_grad_small<K, 4><<<few, 64, 0, st>>>(a);               \
        break;
    switch (kid) {
        PBB_GRAD_CASE(PBB_KERNEL_LAPLACIAN) PBB_GRAD_CASE(PBB_KERNEL_ONEOVERR2) PBB_GRAD_CASE(PBB_KERNEL_GAUSSIAN)
        PBB_GRAD_CASE(PBB_KERNEL_EXPONENTIAL) PBB_GRAD_CASE(PBB_KERNEL_SOFT_LAPLACIAN)
        PBB_GRAD_CASE(PBB_KERNEL_QUADRIC) PBB_GRAD_CASE(PBB_KERNEL_INV_QUADRIC)
        PBB_GRAD_CASE(PBB_KERNEL_LOGARITHM) PBB_GRAD_CASE(PBB_KERNEL_THIN_PLATE) PBB_GRAD_CASE(PBB_KERNEL_R2)
        PBB_GRAD_CASE(PBB_KERNEL_CONSTANT) PBB_GRAD_CASE(PBB_KERNEL_EXP_ANISO)
    default: fail(PBB_ERR_UNSUPPORTED, "no device functor for this kernel id");
    }
#undef PBB_GRAD_CASE
    check(hipGetLastError(), "near_grad");
}

// out[0..n) = 0, as a kernel so that it can sit in a captured graph
__global__ void fill_zero_f64(double *__restrict__ out, int64_t n)
{
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
        out[q] = 0.0;
}

template <int KID>
__global__ __launch_bounds__(256) void kernel_blocks_dev(KernelBlockArgs a)
{
    const int64_t n6 = (int64_t)a.n3 * a.n3, total = a.symm_num * n6;
    const int n = a.n;
    for (int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x; q < total; q += (int64_t)gridDim.x * 256) {
        const int d = (int)(q / n6);
        const int64_t rem = q - d * n6;
        const int j = (int)(rem / a.n3), i = (int)(rem - (int64_t)j * a.n3);
        const int i1 = i / (n * n), i2 = (i / n) % n, i3 = i % n;
        const int j1 = j / (n * n), j2 = (j / n) % n, j3 = j % n;
        const double t0 = 0.5 * a.nodes[i1] * a.box_len, t1 = 0.5 * a.nodes[i2] * a.box_len,
                     t2 = 0.5 * a.nodes[i3] * a.box_len;
        const double s0 = (a.dirs[3 * d] + 0.5 * a.nodes[j1]) * a.box_len,
                     s1 = (a.dirs[3 * d + 1] + 0.5 * a.nodes[j2]) * a.box_len,
                     s2 = (a.dirs[3 * d + 2] + 0.5 * a.nodes[j3]) * a.box_len;
        a.Kcell[q] = keval_blocks<KID>(s0 - t0, s1 - t1, s2 - t2, a.kp) / (a.Kw[i] * a.Kw[j]);
    }
}

// K_d = symm * K_{315-d}^T for the directions past symm_num
__global__ __launch_bounds__(256) void kernel_blocks_symm(KernelBlockArgs a)
{
    const int64_t n6 = (int64_t)a.n3 * a.n3, total = (316 - a.symm_num) * n6;
    for (int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x; q < total; q += (int64_t)gridDim.x * 256) {
        const int d = a.symm_num + (int)(q / n6);
        const int64_t rem = q - (int64_t)(d - a.symm_num) * n6;
        const int j = (int)(rem / a.n3), i = (int)(rem - (int64_t)j * a.n3);
        a.Kcell[d * n6 + i + (int64_t)j * a.n3] = a.symm * a.Kcell[(315 - d) * n6 + j + (int64_t)i * a.n3];
    }
}

void launch_kernel_blocks(const KernelBlockArgs &a, int kid, hipStream_t st)
{
    const int64_t n6 = (int64_t)a.n3 * a.n3;
    if (a.n3 <= 0 || a.n3 != a.n * a.n * a.n || a.kcell_len < 316 * n6 || a.symm_num < 0 || a.symm_num > 316)
        fail(PBB_ERR_INTERNAL, "kernel block arguments do not fit the buffer");
    const int blocks = (int)std::min<int64_t>((a.symm_num * n6 + 255) / 256, 65536);
#define PBB_KB_CASE(K)                                                  \
    case K:                                                             \
        kernel_blocks_dev<K><<<blocks, 256, 0, st>>>(a);                \
        break;
    switch (kid) {
        PBB_KB_CASE(PBB_KERNEL_LAPLACIAN) PBB_KB_CASE(PBB_KERNEL_ONEOVERR2) PBB_KB_CASE(PBB_KERNEL_GAUSSIAN)
        PBB_KB_CASE(PBB_KERNEL_EXPONENTIAL) PBB_KB_CASE(PBB_KERNEL_SOFT_LAPLACIAN) PBB_KB_CASE(PBB_KERNEL_QUADRIC)
        PBB_KB_CASE(PBB_KERNEL_INV_QUADRIC) PBB_KB_CASE(PBB_KERNEL_LOGARITHM) PBB_KB_CASE(PBB_KERNEL_THIN_PLATE)
        PBB_KB_CASE(PBB_KERNEL_R2) PBB_KB_CASE(PBB_KERNEL_CONSTANT) PBB_KB_CASE(PBB_KERNEL_EXP_ANISO)
    default: fail(PBB_ERR_UNSUPPORTED, "no device functor for this kernel id");
    }
#undef PBB_KB_CASE
    check(hipGetLastError(), "kernel_blocks_dev");
    if (a.symm_num < 316) {
        const int b2 = (int)std::min<int64_t>(((316 - a.symm_num) * n6 + 255) / 256, 65536);
        kernel_blocks_symm<<<b2, 256, 0, st>>>(a);
        check(hipGetLastError(), "kernel_blocks_symm");
    }
}

void launch_fill_zero(double *out, int64_t n, hipStream_t st)
{
    if (n <= 0) return;
    int blocks = (int)std::min<int64_t>((n + 255) / 256, 65536);
    fill_zero_f64<<<blocks, 256, 0, st>>>(out, n);
    check(hipGetLastError(), "fill_zero_f64");
}

// Per-workgroup partial sums of (a - b)^2 and b^2 over n doubles, written to
// part[2*g] and part[2*g + 1]; the host adds the pairs (no atomics, so the
// result does not depend on the schedule).
__global__ __launch_bounds__(256) void diff_norms_f64(const double *__restrict__ a, const double *__restrict__ b,
                                                      int64_t n, double *__restrict__ part)
{
    __shared__ double sd[256], sb[256];
    double d2 = 0, b2 = 0;
    for (int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x; q < n; q += (int64_t)gridDim.x * 256) {
        const double bv = b[q], dv = a[q] - bv;
        d2 += dv * dv;
        b2 += bv * bv;
    }
    sd[threadIdx.x] = d2;
    sb[threadIdx.x] = b2;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            sd[threadIdx.x] += sd[threadIdx.x + s];
            sb[threadIdx.x] += sb[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sd[0];
        part[2 * blockIdx.x + 1] = sb[0];
    }
}

void launch_diff_norms(const double *a, const double *b, int64_t n, double *part, int nblocks, hipStream_t st)
{
    diff_norms_f64<<<nblocks, 256, 0, st>>>(a, b, n, part);
    check(hipGetLastError(), "diff_norms_f64");
}

}  // namespace dev
}  // namespace pbb
