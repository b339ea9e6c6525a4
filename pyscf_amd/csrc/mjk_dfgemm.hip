// FP64 matrix-core (v_mfma_f64_16x16x4) products of the density-fitted
// exchange.  MI355X runs one such instruction per SIMD in 64 cycles (78.6
// TFLOP/s), so operands read straight from memory into registers keep up: a
// wave's 64 x 64 tile takes 16 KB of operands per 4096 matrix-core cycles, and
// no LDS is used.
//
//   k_df_tn  C = A^T B over a long inner dimension (10^5 to 10^6) and a small
//            n x n result (30 to 1500): the 64 x 64 tiles of the result are far
//            fewer than the card's 1024 SIMDs, so the inner dimension is split
//            over waves too, each slice's partial tile goes to a workspace and
//            k_df_tn_sum adds the slices (a fixed order: results do not vary).
//   k_df_y   Y_i = B_i X for every i, B_i read once: bound by the larger of
//            reading B and the matrix cores.
//
// Measured on MI355X.  C18H38 cc-pVDZ (442 AOs, 73 orbitals, 2126 fitting
// functions), library products -> these kernels: K product 25.0 -> 0.65 ms
// (rocBLAS DGEMM ran it on 12 tiles of 128 x 192), half transform 1.94 -> 1.39 ms
// (44 TFLOP/s, 48 with the padding of 73 columns to 80).  C30H62 (730 AOs, 3526
// functions): 121 orbitals 5.7 -> 4.3 and 8.7 -> 8.1 ms, general density 51.3 ->
// 46.5 and 42.2 -> 43.6 ms.
#include "df_gemm.h"

#include <algorithm>

namespace mjk {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
// two doubles at 8-byte alignment: columns of odd length start there
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

// Lane (m = lane % 16, q = lane / 16) of v_mfma_f64_16x16x4 holds A[m][k = q],
// B[k = q][m], and rows 4 v + q of column m of the result in register v.
__device__ __forceinline__ v4d mfma(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Sixteen inner elements k .. k + 15 of four 16-row groups: lane (m, q) takes
// elements k + 4q .. k + 4q + 3 of row m of each group (a whole 128-byte line
// per row over the four q), and MFMA step s multiplies elements k + 4q + s: the
// inner index is permuted alike in both operands.
__device__ __forceinline__ void tn_load(const double* const (&p)[4], long long k, double (&x)[4][4])
{
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const d2u lo = *(const d2u*)(p[g] + k), hi = *(const d2u*)(p[g] + k + 2);
        x[g][0] = lo.x;
        x[g][1] = lo.y;
        x[g][2] = hi.x;
        x[g][3] = hi.y;
    }
}

// The last, partial sixteen of a slice: n elements from k on exist for lane
// quarter q (elements at and beyond n count zero and are not read).
__device__ __forceinline__ void tn_load_tail(const double* const (&p)[4], long long k, int n, double (&x)[4][4])
{
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int s = 0; s < 4; ++s) x[g][s] = s < n ? p[g][k + s] : 0.0;
}

__device__ __forceinline__ void tn_mul(const double (&a)[4][4], const double (&b)[4][4], v4d (&acc)[4][4])
{
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = mfma(a[i][s], b[j][s], acc[i][j]);
}

// Tile t of the list: (row tile, column tile), row >= column when sym.
__device__ __forceinline__ void tn_tile(int t, int nt, bool sym, int& ti, int& tj)
{
    if (!sym) {
        ti = t % nt;
        tj = t / nt;
        return;
    }
    int r = 0;
    while ((r + 1) * (r + 2) / 2 <= t) ++r;
    ti = r;
    tj = t - r * (r + 1) / 2;
}

// One wave per (tile, slice); the tiles of one slice run on one XCD (blocks go
// to the XCDs in turn), whose L2 then serves the slice's rows to all of them.
// Inner element k of row i at (k / np) os + i is + k % np (KLayout).
__global__ void __launch_bounds__(256, 1) k_df_tn(const double* __restrict__ A, const double* __restrict__ B, int n,
                                                 long long kin, KLayout la, TnPlan pl, int sym,
                                                 double* __restrict__ part)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, q = lane >> 4;
    const int idx = (blockIdx.x >> 3) * 4 + wave;
    const int s = (idx / pl.ntile) * 8 + (blockIdx.x & 7), t = idx % pl.ntile;
    if (s >= pl.nsplit) return;
    const long long end = min((s + 1) * pl.kc, kin);
    int ti, tj;
    tn_tile(t, pl.nt, sym != 0, ti, tj);
    long long ra[4], rb[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {   // rows past the last are computed on the last row and dropped
        ra[g] = min(ti * 64 + 16 * g + m, n - 1) * la.is + 4 * q;
        rb[g] = min(tj * 64 + 16 * g + m, n - 1) * la.is + 4 * q;
    }
    v4d acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = v4d{0, 0, 0, 0};
    double a0[4][4], b0[4][4], a1[4][4], b1[4][4];
    for (long long at = s * pl.kc; at < end;) {   // the contiguous runs of the slice
        const long long o = at / la.np;
        long long k = at - o * la.np;
        const long long k1 = min(la.np, k + end - at), kf = k + ((k1 - k) & ~15LL);   // whole sixteens
        at += k1 - k;
        const double *pa[4], *pb[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            pa[g] = A + o * la.os + ra[g];
            pb[g] = B + o * la.os + rb[g];
        }
        if (k + 16 <= kf) {
            tn_load(pa, k, a0);
            tn_load(pb, k, b0);
            for (; k + 48 <= kf; k += 32) {   // the next sixteen in flight behind 64 MFMAs
                tn_load(pa, k + 16, a1);
                tn_load(pb, k + 16, b1);
                tn_mul(a0, b0, acc);
                tn_load(pa, k + 32, a0);
                tn_load(pb, k + 32, b0);
                tn_mul(a1, b1, acc);
            }
            tn_mul(a0, b0, acc);
            k += 16;
            if (k + 16 <= kf) {
                tn_load(pa, k, a0);
                tn_load(pb, k, b0);
                tn_mul(a0, b0, acc);
                k += 16;
            }
        }
        if (k < k1) {
            const int rest = (int)min(4LL, max(0LL, k1 - k - 4 * q));
            tn_load_tail(pa, k, rest, a0);
            tn_load_tail(pb, k, rest, b0);
            tn_mul(a0, b0, acc);
        }
    }
    double* out = part + ((long long)s * pl.ntile + t) * 4096 + lane;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) out[((i * 4 + j) * 4 + v) * 64] = acc[i][j][v];
}

// Sum of the slices into C (and its mirror when sym).
__global__ void __launch_bounds__(256) k_df_tn_sum(const double* __restrict__ part, TnPlan pl, int n, int sym,
                                                  double* __restrict__ C)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int t = e >> 12, r = e & 4095;
    if (t >= pl.ntile) return;
    const double* p = part + e;
    const long long stride = (long long)pl.ntile * 4096;
    double v = 0.0;
#pragma unroll 8
    for (int s = 0; s < pl.nsplit; ++s) v += p[s * stride];
    int ti, tj;
    tn_tile(t, pl.nt, sym != 0, ti, tj);
    const int lane = r & 63, u = r >> 6;   // u = (i 4 + j) 4 + v of k_df_tn
    const int row = ti * 64 + (u >> 4) * 16 + 4 * (u & 3) + (lane >> 4);
    const int col = tj * 64 + ((u >> 2) & 3) * 16 + (lane & 15);
    if (row >= n || col >= n) return;
    C[(long long)col * n + row] = v;
    if (sym && ti != tj) C[(long long)row * n + col] = v;
}

// Y_i = B_i X.  A wave owns 64 fitting functions x (16 NSUB) orbitals of one i;
// lane (m, q) reads four consecutive fitting functions 4m .. 4m + 3 of inner
// element l + q (512 contiguous bytes per element over the 16 m), which are
// row m of the wave's four 16-row groups.  The panels of one (i, row tile) are
// neighbouring waves, so B_i comes from memory once.
//   Every load is unconditional, at a clamped address where there is nothing to
// load (the last functions once more, stored again with the same value; the
// last inner element, times a zero row of X): a load under a condition makes
// the compiler wait for all loads at the join, those of the next step with
// them, and nothing is in flight behind the products.  Eight inner elements a
// step: two waves per SIMD to five groups.  MI355X, ms, conditional loads of
// sixteen elements / these: 442 AOs and 73 orbitals 1.67 / 1.39, 730 and 121
// 10.9 / 8.1, general density of 730 85.9 / 43.6 (63 TFLOP/s; spilled registers
// of six groups had their part in it; the library's DGEMM 42.2).
constexpr int Y_U = 2;   // groups of four inner elements a step
template <int NSUB>
__global__ void __launch_bounds__(256, 1) k_df_y(const double* __restrict__ B, const double* __restrict__ Xp, int nao,
                                             int naux, int ncol, int ldx, int npan, KLayout la, double* __restrict__ Y)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, q = lane >> 4;
    const int ntm = (naux + 63) / 64;
    const long long item = (long long)blockIdx.x * 4 + wave;
    const int pan = (int)(item % npan);
    const int tm = (int)((item / npan) % ntm);
    const long long i = item / ((long long)npan * ntm);
    if (i >= nao) return;
    const double* b = B + i * nao * naux + min(tm * 64 + 4 * m, naux - 4);
    const double* x = Xp + pan * 16 * NSUB + m;
    v4d acc[4][NSUB];
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int j = 0; j < NSUB; ++j) acc[g][j] = v4d{0, 0, 0, 0};
    auto load = [&](int l, double (&ab)[Y_U][4], double (&xb)[Y_U][NSUB]) {
#pragma unroll
        for (int u = 0; u < Y_U; ++u) {
            const int le = l + 4 * u + q;
            const double* bl = b + (long long)min(le, nao - 1) * naux;
            const d2u lo = *(const d2u*)bl, hi = *(const d2u*)(bl + 2);
            ab[u][0] = lo.x;
            ab[u][1] = lo.y;
            ab[u][2] = hi.x;
            ab[u][3] = hi.y;
#pragma unroll
            for (int j = 0; j < NSUB; ++j) xb[u][j] = x[(long long)le * ldx + 16 * j];   // rows padded to sixteens
        }
    };
    auto mul = [&](const double (&ab)[Y_U][4], const double (&xb)[Y_U][NSUB]) {
#pragma unroll
        for (int u = 0; u < Y_U; ++u)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int j = 0; j < NSUB; ++j) acc[g][j] = mfma(ab[u][g], xb[u][j], acc[g][j]);
    };
    double a0[Y_U][4], x0[Y_U][NSUB], a1[Y_U][4], x1[Y_U][NSUB];
    constexpr int STEP = 4 * Y_U;
    const int ns = (nao + STEP - 1) / STEP;
    load(0, a0, x0);
    for (int s = 0; s < ns; s += 2) {   // the next step in flight behind the products (the last one loaded again)
        load(STEP * min(s + 1, ns - 1), a1, x1);
        mul(a0, x0);
        load(STEP * min(s + 2, ns - 1), a0, x0);
        if (s + 1 < ns) mul(a1, x1);
    }
    // lane (m, q): orbital m of sub-panel j, fitting functions 4 (4 v + q) .. + 3
    double* y = Y + i * la.is;
#pragma unroll
    for (int j = 0; j < NSUB; ++j) {
        const int o = (pan * NSUB + j) * 16 + m;
        if (o >= ncol) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            double* d = y + o * la.yo + min(tm * 64 + 4 * (4 * v + q), naux - 4);
            *(d2u*)d = d2u{acc[0][j][v], acc[1][j][v]};
            *(d2u*)(d + 2) = d2u{acc[2][j][v], acc[3][j][v]};
        }
    }
}

// The same for fewer than four fitting functions, an element per thread.
__global__ void __launch_bounds__(256) k_df_y_few(const double* __restrict__ B, const double* __restrict__ Xp, int nao,
                                                 int naux, int ncol, int ldx, KLayout la, double* __restrict__ Y)
{
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)nao * ncol * naux) return;
    const int p = (int)(e % naux), o = (int)(e / naux % ncol);
    const long long i = e / ((long long)naux * ncol);
    double v = 0.0;
    for (int l = 0; l < nao; ++l) v = fma(B[(i * nao + l) * naux + p], Xp[(long long)l * ldx + o], v);
    Y[i * la.is + o * la.yo + p] = v;
}

// Panels of the orbitals, at most five 16-column groups per wave (two waves per
// SIMD): the fewest groups with the padding, a panel counted as 0.4 more for
// its reads of B.  MI355X, 730 AOs, ms: 730 columns in 12 panels of 4 groups
// 43.6, in 8 of 6 49.2; 442 AOs: 73 columns in one of 5 1.38, in two of 3 1.60.
void y_panels(int ncol, int& nsub, int& npan)
{
    const int n = (ncol + 15) / 16;
    double best = 0;
    nsub = 0;
    for (int k = 5; k >= 1; --k) {
        const int np = (n + k - 1) / k;
        if (nsub == 0 || np * (k + 0.4) < best) {
            best = np * (k + 0.4);
            nsub = k;
            npan = np;
        }
    }
}

__global__ void __launch_bounds__(256) k_df_pad_x(const double* __restrict__ src, long long sl, long long so, int nao,
                                                 int ncol, int rows, int ldx, double* __restrict__ Xp)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= rows * ldx) return;
    const int l = e / ldx, o = e - l * ldx;
    Xp[e] = l < nao && o < ncol ? src[l * sl + o * so] : 0.0;
}

// Cholesky, right-looking in blocks of 32 columns.  Panel: a wave holds the
// diagonal block (lane i < 32 its row i, in registers) and 64 rows below it, and
// does for each column the pivot, the scaling and the update of both from one
// broadcast column in LDS; every block factors the diagonal block again for its
// own rows, which costs less than a launch between.  A serial chain of n square
// roots, divisions and LDS round trips bounds it (64 columns a block do not fit
// in registers).  The factored diagonal goes to tmp (the other blocks still read
// the original), and the update puts it back.
// (P|Q) of about 900 auxiliary functions (29 blocks) on MI355X: 1.05 ms, 21 us
// a panel and 16 an update; rocsolver_dpotrf 2.4 ms.
__global__ __launch_bounds__(64) void k_chol_panel(double* A, int n, int k0, double* __restrict__ tmp, int* info)
{
    __shared__ double col[2][CHOL_NB];
    const int i = threadIdx.x, nb = min(CHOL_NB, n - k0);
    const int r = k0 + CHOL_NB + blockIdx.x * 64 + i;   // r < n only under a whole block
    double* const Ad = A + (size_t)k0 * n + k0 + i;
    double* const Ar = A + (size_t)k0 * n + r;
    double a[CHOL_NB], x[CHOL_NB];
#pragma unroll
    for (int j = 0; j < CHOL_NB; ++j) {
        a[j] = i < nb && j < nb ? Ad[(size_t)j * n] : i == j ? 1.0 : 0.0;   // (lanes past 31: zero rows)
        x[j] = r < n ? Ar[(size_t)j * n] : 0.0;
    }
    int bad = 0;
#pragma unroll
    for (int j = 0; j < CHOL_NB; ++j) {
        const double d = __shfl(a[j], j);
        if (!(d > 0.0) && bad == 0) bad = k0 + j + 1;
        const double s = sqrt(d), ri = 1.0 / s;
        a[j] = i > j ? a[j] * ri : i == j ? s : 0.0;
        x[j] *= ri;
        if (i < CHOL_NB) col[j & 1][i] = a[j];
        __syncthreads();
#pragma unroll
        for (int k = j + 1; k < CHOL_NB; ++k) {
            const double c = col[j & 1][k];
            a[k] = fma(-a[j], c, a[k]);
            x[k] = fma(-x[j], c, x[k]);
            // (in this step: deferred updates of x keep every column alive, 800 spilled registers)
            asm volatile("" : "+v"(a[k]), "+v"(x[k]));
        }
    }
    if (blockIdx.x == 0) {
        if (i == 0 && bad && *info == 0) *info = bad;
        if (i < CHOL_NB) {
#pragma unroll
            for (int j = 0; j < CHOL_NB; ++j) tmp[j * CHOL_NB + i] = a[j];
        }
    }
    if (r < n) {
#pragma unroll
        for (int j = 0; j < CHOL_NB; ++j) Ar[(size_t)j * n] = x[j];
    }
}

// Trailing update by the panel at k0, a 64 x 64 tile of the lower triangle per
// block (16 rows a wave); the last block stores the factored diagonal block.
__global__ __launch_bounds__(256) void k_chol_update(double* A, int n, int k0, int ntile,
                                                     const double* __restrict__ tmp)
{
    const int tid = threadIdx.x;
    if ((int)blockIdx.x == ntile) {
        for (int e = tid; e < CHOL_NB * CHOL_NB; e += 256) {
            const int i = e % CHOL_NB, j = e / CHOL_NB;
            if (i >= j && k0 + i < n) A[(size_t)(k0 + j) * n + k0 + i] = tmp[e];
        }
        return;
    }
    int ti, tj;
    tn_tile(blockIdx.x, 0, true, ti, tj);
    const int lane = tid & 63, m = lane & 15, q = lane >> 4;
    const int t0 = k0 + CHOL_NB, c0 = t0 + 64 * tj;
    const int r = t0 + 64 * ti + 16 * (tid >> 6) + m;
    const double* P = A + (size_t)(k0 + q) * n;
    v4d acc[4] = {};
#pragma unroll 4
    for (int kk = 0; kk < CHOL_NB / 4; ++kk, P += (size_t)4 * n) {
        const double pr = r < n ? P[r] : 0.0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int c = c0 + 16 * g + m;
            acc[g] = mfma(c < n ? P[c] : 0.0, pr, acc[g]);   // column m of the result: row r of A
        }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = c0 + 16 * g + 4 * v + q;
            if (r < n && c < n) A[(size_t)c * n + r] -= acc[g][v];
        }
}

}  // namespace

// Slices: waves in whole rounds of the card's 1024 SIMDs (a wave holds a SIMD
// to itself).  Eight at least, one per XCD, however short; more while each keeps
// 256 inner elements and all tiles fit eight rounds: the count with the fullest
// last round, of about equals the smallest, as slices cost workspace traffic.
constexpr long long TN_SLICE = 16384;
TnPlan df_tn_plan(int n, long long kin, bool sym)
{
    TnPlan p;
    p.nt = (n + 63) / 64;
    p.ntile = sym ? p.nt * (p.nt + 1) / 2 : p.nt * p.nt;
    const long long most = std::max(1LL, kin / 256);
    double best = -1;
    for (int s = 8; s <= 1024; s += 8) {
        if (s > 8 && (s > most || (long long)s * p.ntile > 8192)) break;
        const long long waves = (long long)s * p.ntile, rounds = (waves + 1023) / 1024;
        const double fill = (double)waves / (double)(rounds * 1024);
        if (fill > best + 0.02) {
            best = fill;
            p.nsplit = s;
        }
    }
    // tiles of a slice drift apart in a long one and no longer find each other's
    // rows in L2: 730 AOs, general density, 56 slices of 46 000 49.9 ms, 128 46.8
    p.nsplit *= (int)std::max(1LL, (kin / p.nsplit + TN_SLICE - 1) / TN_SLICE);
    p.kc = ((kin + p.nsplit - 1) / p.nsplit + 15) / 16 * 16;
    p.ws = (size_t)p.nsplit * p.ntile * 4096;
    return p;
}

int df_tn(const TnPlan& pl, const double* A, const double* B, int n, long long kin, const KLayout& la, bool sym,
          double* part, double* C, hipStream_t st)
{
    const int per_xcd = pl.nsplit / 8 * pl.ntile;
    k_df_tn<<<(unsigned)((per_xcd + 3) / 4 * 8), 256, 0, st>>>(A, B, n, kin, la, pl, sym, part);
    k_df_tn_sum<<<(unsigned)(pl.ntile * 16), 256, 0, st>>>(part, pl, n, sym, C);
    return (int)hipGetLastError();
}

size_t df_xp_size(int nao, int ncol)
{
    int nsub, npan;
    y_panels(ncol, nsub, npan);
    return (size_t)((nao + 15) / 16 * 16) * (nsub * npan * 16);
}

int df_pad_x(const double* src, long long sl, long long so, int nao, int ncol, double* Xp, hipStream_t st)
{
    int nsub, npan;
    y_panels(ncol, nsub, npan);
    const int ldx = nsub * npan * 16, rows = (nao + 15) / 16 * 16;
    k_df_pad_x<<<(unsigned)(((size_t)rows * ldx + 255) / 256), 256, 0, st>>>(src, sl, so, nao, ncol, rows, ldx, Xp);
    return (int)hipGetLastError();
}

// By row up to 2 MB a row, above by column: the 128 rows that a tile's wave reads
// side by side then lie within a few pages instead of one page each.  MI355X,
// K product, ms, by row / by column: 442 AOs, kin 156 000 0.68 / 0.69, 472 000
// 1.90 / 1.72; 730 AOs, 212 000 2.30 / 2.36, 427 000 4.59 / 4.26, 1.3 million
// 15.7 / 11.8, general density (2.6 million) 68.4 / 49.9.
KLayout df_layout(int nao, int naux, int ncol)
{
    const long long kin = (long long)naux * ncol, col = (long long)nao * naux;
    if (kin * (long long)sizeof(double) < (2LL << 20)) return {kin, kin, 0, naux};
    return {naux, naux, col, col};
}

int df_y(const double* B, const double* Xp, int nao, int naux, int ncol, const KLayout& la, double* Y, hipStream_t st)
{
    int nsub, npan;
    y_panels(ncol, nsub, npan);
    const int ldx = nsub * npan * 16;
    if (naux < 4) {
        const long long n = (long long)nao * ncol * naux;
        k_df_y_few<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(B, Xp, nao, naux, ncol, ldx, la, Y);
        return (int)hipGetLastError();
    }
    const long long items = (long long)nao * ((naux + 63) / 64) * npan;
    const unsigned nb = (unsigned)((items + 3) / 4);
    switch (nsub) {
    case 1: k_df_y<1><<<nb, 256, 0, st>>>(B, Xp, nao, naux, ncol, ldx, npan, la, Y); break;
    case 2: k_df_y<2><<<nb, 256, 0, st>>>(B, Xp, nao, naux, ncol, ldx, npan, la, Y); break;
    case 3: k_df_y<3><<<nb, 256, 0, st>>>(B, Xp, nao, naux, ncol, ldx, npan, la, Y); break;
    case 4: k_df_y<4><<<nb, 256, 0, st>>>(B, Xp, nao, naux, ncol, ldx, npan, la, Y); break;
    default: k_df_y<5><<<nb, 256, 0, st>>>(B, Xp, nao, naux, ncol, ldx, npan, la, Y); break;
    }
    return (int)hipGetLastError();
}

int df_potrf(double* A, int n, double* tmp, int* info, hipStream_t st)
{
    for (int k0 = 0; k0 < n; k0 += CHOL_NB) {
        const int nt = (std::max(0, n - k0 - CHOL_NB) + 63) / 64, ntile = nt * (nt + 1) / 2;
        hipLaunchKernelGGL(k_chol_panel, dim3(std::max(1, nt)), dim3(64), 0, st, A, n, k0, tmp, info);
        hipLaunchKernelGGL(k_chol_update, dim3(ntile + 1), dim3(256), 0, st, A, n, k0, ntile, tmp);
    }
    return (int)hipGetLastError();
}

}  // namespace mjk
