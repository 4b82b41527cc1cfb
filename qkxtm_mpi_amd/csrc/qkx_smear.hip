// qkx_smear.hip -- source preparation on the GPU, FP64 like the reference:
// the SU(3) projection, APE smearing of the spatial links, Gaussian smearing
// of spinors (batches of right-hand sides, optionally one time slice) and the
// plaquette.
//
// Reference: qcd_projectSU33d lib/blas.cpp:6-422, Gauge::APE_smearing
// lib/lattice_util.cpp:950-1078, Vector::Gaussian_smearing :1080-1146,
// Gauge::calculatePlaquette :923-946.
//
// Kernels
//   ape_step_kernel    one thread per spatial link (site, mu < 3): the four
//                      staples, alpha-weighted sum with the link, projection,
//                      store.  Reads 13 links per thread, 3 unique per site
//                      from HBM (neighbours come from L2); FP64 ALU-heavy.
//   gauss_step_kernel  one thread per (site, right-hand side): the 3-D
//                      covariant hop on all four spins; the links of a site
//                      are shared by its right-hand sides (adjacent lanes).
//                      HBM-bound: 432 B of links + 384 B per right-hand side.
//   gauss_march_kernel the same for many units: one thread per (column, spin,
//                      right-hand side), marching along z.
//   plaq_kernel        grid-stride per-site sum of the six plaquettes into
//                      per-workgroup partials, summed in a fixed order.
#include <cmath>
#include <algorithm>
#include <memory>
#include "qkx_internal.h"
#include "qkx_core.h"

namespace {

using C = Cx<double>;
struct Mat {
    C a[9];   // row-major
};

constexpr int kThreads = 256;
constexpr int kPlaqBlocks = 1024;

__device__ __forceinline__ Mat ldm(const double2 *base, int V, int mu, int s)
{
    Mat m;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        double2 d = ld(base + (size_t)(mu * 9 + k) * V, (uint32_t)s);
        m.a[k] = {d.x, d.y};
    }
    return m;
}
__device__ __forceinline__ void stm(double2 *base, int V, int mu, int s, const Mat &m)
{
#pragma unroll
    for (int k = 0; k < 9; k++) st(base + (size_t)(mu * 9 + k) * V, (uint32_t)s, make_double2(m.a[k].re, m.a[k].im));
}
// a b
__device__ __forceinline__ Mat mm(const Mat &a, const Mat &b)
{
    Mat r;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            r.a[3 * i + j] = cmac(cmac(cmul_f(a.a[3 * i], b.a[j]), a.a[3 * i + 1], b.a[3 + j]), a.a[3 * i + 2], b.a[6 + j]);
    return r;
}
// a b^dag
__device__ __forceinline__ Mat mmd(const Mat &a, const Mat &b)
{
    Mat r;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            r.a[3 * i + j] = cjmac(cjmac(cjmul_f(b.a[3 * j], a.a[3 * i]), b.a[3 * j + 1], a.a[3 * i + 1]),
                                   b.a[3 * j + 2], a.a[3 * i + 2]);
    return r;
}
// a^dag b
__device__ __forceinline__ Mat mdm(const Mat &a, const Mat &b)
{
    Mat r;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            r.a[3 * i + j] = cjmac(cjmac(cjmul_f(a.a[i], b.a[j]), a.a[3 + i], b.a[3 + j]), a.a[6 + i], b.a[6 + j]);
    return r;
}

__device__ __forceinline__ C conjc(C a) { return {a.re, -a.im}; }
__device__ __forceinline__ double nrm2c(C a) { return a.re * a.re + a.im * a.im; }

// Constants of the closed-form eigenvalues, formed on the host as the
// reference forms them (pow(18, 1/3) ...).
struct ProjConst {
    double r18, r12, r23, s3;
};

// SU(3) projection of one matrix: U = M (M^dag M)^{-1/2} exp(-i arg(det M)/3)
// by the reference's closed-form eigensystem of H = M^dag M (Cardano roots of
// the traceless part, eigenvectors from two rows of H - e), then Gram-Schmidt
// of columns 1-2 and column 3 = conj(col1 x col2).  If the off-diagonal moduli
// of H sum to at most 1e-8, row i of M is scaled by 1/sqrt(H_ii) instead.
// The steps follow lib/blas.cpp:32-420 so that results agree to rounding.
__device__ void su3_project(Mat &M, const ProjConst &pc)
{
    const C *m = M.a;
    C det = cmul(m[0], cmul(m[4], m[8])) + cmul(m[1], cmul(m[5], m[6])) + cmul(m[2], cmul(m[3], m[7]));
    det = det - (cmul(m[2], cmul(m[4], m[6])) + cmul(m[0], cmul(m[5], m[7])) + cmul(m[1], cmul(m[3], m[8])));
    const double phase = atan2(det.im, det.re) / 3.0;

    C H[9];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) H[3 * i + j] = cjmul(m[i], m[j]) + cjmul(m[3 + i], m[3 + j]) + cjmul(m[6 + i], m[6 + j]);
    // exact Hermiticity of the off-diagonal pairs
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = i + 1; j < 3; j++) {
            C h = {(H[3 * i + j].re + H[3 * j + i].re) * 0.5, (H[3 * i + j].im - H[3 * j + i].im) * 0.5};
            H[3 * i + j] = h;
            H[3 * j + i] = conjc(h);
        }
    const double n01 = nrm2c(H[1]), n02 = nrm2c(H[2]), n12 = nrm2c(H[5]);
    if (sqrt(n01) + sqrt(n02) + sqrt(n12) <= 1e-08) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const double e = 1.0 / sqrt(H[4 * i].re);
#pragma unroll
            for (int j = 0; j < 3; j++) M.a[3 * i + j] = e * M.a[3 * i + j];
        }
        return;
    }
    // eigenvalues: e^3 + a e + b = 0 for the traceless part
    const double tr = (H[0].re + H[4].re + H[8].re) / 3.0;
    const double h00 = H[0].re - tr, h11 = H[4].re - tr, h22 = H[8].re - tr;
    const double a = -(h22 * h22 - h00 * h11 + n01 + n02 + n12);
    const C t1 = cmul(H[1], cmul(H[5], conjc(H[2])));
    const C t2 = cmul(H[2], cmul(conjc(H[1]), conjc(H[5])));
    C b;
    b.re = (-h00 * h11 * h22 + h22 * n01 - t1.re + h11 * n02) + (h00 * n12 - t2.re);
    b.im = -t1.im - t2.im;
    const C bb = cmul(b, b);
    const C disc = {12.0 * a * a * a + 81.0 * bb.re, 81.0 * bb.im};
    // principal square root and cube root through the polar form
    double rr = sqrt(disc.re * disc.re + disc.im * disc.im), th = atan2(disc.im, disc.re);
    double sn, cs;
    sincos(0.5 * th, &sn, &cs);
    const C w = {sqrt(rr) * cs, sqrt(rr) * sn};
    const C z = {-9.0 * b.re + w.re, -9.0 * b.im + w.im};
    rr = sqrt(z.re * z.re + z.im * z.im);
    th = atan2(z.im, z.re);
    sincos(th / 3.0, &sn, &cs);
    const double rc = cbrt(rr);
    const C D = {rc * cs, rc * sn};
    const double dd = D.re * D.re + D.im * D.im;
    double e[3];
    e[0] = D.re / pc.r18 - (a * pc.r23 * D.re) / dd;
    {
        const C Ds = {D.re * pc.r12, D.im * pc.r12};
        e[1] = a * ((Ds.re + pc.s3 * Ds.im) / (Ds.re * Ds.re + Ds.im * Ds.im)) - (D.re + pc.s3 * D.im) / (pc.r18 * 2.0);
    }
    e[2] = -e[0] - e[1];
#pragma unroll
    for (int k = 0; k < 3; k++) e[k] += tr;

    // eigenvectors (stored conjugated, as the reference does) for e0 and e1
    C v[9];
    const double H00 = H[0].re, H11 = H[4].re;
    const C p10_21 = cmul(H[3], H[7]), p20_01 = cmul(H[6], H[1]);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const double ek = e[k];
        v[3 * k + 0] = {-(ek * H[6].re - H[6].re * H11 + p10_21.re), -(ek * H[6].im - H[6].im * H11 + p10_21.im)};
        v[3 * k + 1] = {-(p20_01.re + ek * H[7].re - H00 * H[7].re), -(p20_01.im + ek * H[7].im - H00 * H[7].im)};
        v[3 * k + 2] = {-ek * ek + ek * H00 + n01 + ek * H11 - H00 * H11, 0.0};
    }
    // Gram-Schmidt of v1 against v0, normalise both; v2 = conj(v0 x v1)
    double nr = nrm2c(v[0]) + nrm2c(v[1]) + nrm2c(v[2]);
    {
        C ov = cmul(v[0], conjc(v[3])) + cmul(v[1], conjc(v[4])) + cmul(v[2], conjc(v[5]));
        ov = (1.0 / nr) * ov;
#pragma unroll
        for (int j = 0; j < 3; j++) v[3 + j] = v[3 + j] - cmul(ov, v[j]);
    }
    nr = 1.0 / sqrt(nr);
#pragma unroll
    for (int j = 0; j < 3; j++) v[j] = nr * v[j];
    nr = 1.0 / sqrt(nrm2c(v[3]) + nrm2c(v[4]) + nrm2c(v[5]));
#pragma unroll
    for (int j = 0; j < 3; j++) v[3 + j] = nr * v[3 + j];
    v[6] = conjc(cmul(v[1], v[5]) - cmul(v[2], v[4]));
    v[7] = conjc(cmul(v[2], v[3]) - cmul(v[0], v[5]));
    v[8] = conjc(cmul(v[0], v[4]) - cmul(v[1], v[3]));

    // U = (M conj(v)^T) diag(exp(-i phase)/sqrt(e_k)) v
    double ps, pcs;
    sincos(phase, &ps, &pcs);
    C vr[9];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double de = 1.0 / sqrt(e[k]);
        const C s = {de * pcs, -de * ps};
#pragma unroll
        for (int j = 0; j < 3; j++) vr[3 * k + j] = cmul(s, v[3 * k + j]);
    }
    C U[9];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        C hm[3];
#pragma unroll
        for (int k = 0; k < 3; k++)
            hm[k] = cmul(m[3 * i], conjc(v[3 * k])) + cmul(m[3 * i + 1], conjc(v[3 * k + 1])) +
                    cmul(m[3 * i + 2], conjc(v[3 * k + 2]));
#pragma unroll
        for (int l = 0; l < 3; l++) U[3 * i + l] = cmul(hm[0], vr[l]) + cmul(hm[1], vr[3 + l]) + cmul(hm[2], vr[6 + l]);
    }
    // columns: the reference subtracts (sum_i U_i0 conj U_i1)/|col0|^2 col0
    // from col1, normalises both, and sets col3 = conj(col1 x col2)
    nr = nrm2c(U[0]) + nrm2c(U[3]) + nrm2c(U[6]);
    {
        C ov = cmul(U[0], conjc(U[1])) + cmul(U[3], conjc(U[4])) + cmul(U[6], conjc(U[7]));
        ov = (1.0 / nr) * ov;
#pragma unroll
        for (int i = 0; i < 3; i++) U[3 * i + 1] = U[3 * i + 1] - cmul(ov, U[3 * i]);
    }
    nr = 1.0 / sqrt(nr);
#pragma unroll
    for (int i = 0; i < 3; i++) U[3 * i] = nr * U[3 * i];
    nr = 1.0 / sqrt(nrm2c(U[1]) + nrm2c(U[4]) + nrm2c(U[7]));
#pragma unroll
    for (int i = 0; i < 3; i++) U[3 * i + 1] = nr * U[3 * i + 1];
    U[2] = conjc(cmul(U[3], U[7]) - cmul(U[6], U[4]));
    U[5] = conjc(cmul(U[6], U[1]) - cmul(U[0], U[7]));
    U[8] = conjc(cmul(U[0], U[4]) - cmul(U[3], U[1]));
#pragma unroll
    for (int k = 0; k < 9; k++) M.a[k] = U[k];
}

// ---- site coordinates in the parity-blocked layout ------------------------
struct Site {
    int c[4];
};
__device__ __forceinline__ Site coords(const Geom &g, int p, int cb)
{
    Site r;
    const int rest = fdiv(cb, g.dLh0);
    const int xh = cb - rest * g.Lh0;
    const int zt = fdiv(rest, g.dL1);
    r.c[1] = rest - zt * g.L[1];
    r.c[3] = fdiv(zt, g.dL2);
    r.c[2] = zt - r.c[3] * g.L[2];
    r.c[0] = 2 * xh + ((p + r.c[1] + r.c[2] + r.c[3]) & 1);
    return r;
}
__device__ __forceinline__ int blocked(const Geom &g, const Site &x)
{
    const int lex = ((x.c[3] * g.L[2] + x.c[2]) * g.L[1] + x.c[1]) * g.L[0] + x.c[0];
    return ((x.c[0] + x.c[1] + x.c[2] + x.c[3]) & 1) * g.Vh + (lex >> 1);
}
// x + d mu (d = +-1) with periodic wrap; written over constant indices so a
// run-time mu selects instead of indexing a private array in memory
__device__ __forceinline__ Site step(const Geom &g, Site x, int mu, int d)
{
#pragma unroll
    for (int m = 0; m < 4; m++)
        if (m == mu) {
            const int v = x.c[m] + d;
            x.c[m] = v < 0 ? v + g.L[m] : (v >= g.L[m] ? v - g.L[m] : v);
        }
    return x;
}

// ---- traversal ---------------------------------------------------------------
// A launch covers the sites of both parities (time slices t_lo .. t_lo+nt-1)
// with `ups` threads per site (right-hand sides, or link directions; adjacent
// lanes).  Sites of a parity go x fastest, then yb rows of y, then z, then
// the next block of rows, then t: consecutive z of a block of rows are close
// in this order, so the z-neighbours of the sites in flight are still in L2
// when they are used (whole z-planes of a 12-source FP64 field are not).
// Workgroups are remapped so that XCD k (hardware workgroup b runs on XCD
// b % 8) takes the k-th contiguous slab of both parities and sees the
// neighbour reuse of that slab in its own L2.
struct Trav {
    FastDiv dups, dyb, dnyb;
    int ups, yb, nyb, t_lo;
    int nunits;     // units of one parity
    int nblk8;      // workgroups per XCD and parity when remapped, else 0
};

// blocks: workgroups per parity as a function of the parity's units
template <class F> Trav make_trav(const int L[4], int ups, int t, dim3 &grid, F blocks)
{
    Trav tr;
    tr.ups = ups;
    tr.dups = make_fastdiv(ups);
    tr.yb = 1;   // rows per block: the largest divisor of L[1] up to 8
    for (int d = 2; d <= 8; d++)
        if (L[1] % d == 0) tr.yb = d;
    tr.nyb = L[1] / tr.yb;
    tr.dyb = make_fastdiv(tr.yb);
    tr.dnyb = make_fastdiv(tr.nyb);
    tr.t_lo = t < 0 ? 0 : t;
    tr.nunits = L[0] * L[1] * L[2] / 2 * (t < 0 ? L[3] : 1) * ups;
    int nbh = blocks(tr.nunits);
    tr.nblk8 = 0;
    grid = dim3(nbh, 2);
    if (nbh >= 32) {
        nbh = (nbh + 7) / 8 * 8;
        tr.nblk8 = nbh / 8;
        grid = dim3(2 * nbh, 1);
    }
    return tr;
}

// Site v of a parity in walk order: its coordinates and blocked index.
__device__ __forceinline__ void trav_walk(const Geom &g, const Trav &tr, int p, int v, Site &x, int &s)
{
    const int q1 = fdiv(v, g.dLh0), xh = v - q1 * g.Lh0;
    const int q2 = fdiv(q1, tr.dyb), yi = q1 - q2 * tr.yb;
    const int q3 = fdiv(q2, g.dL2), z = q2 - q3 * g.L[2];
    const int tt = fdiv(q3, tr.dnyb), ybk = q3 - tt * tr.nyb;
    x.c[1] = ybk * tr.yb + yi;
    x.c[2] = z;
    x.c[3] = tr.t_lo + tt;
    x.c[0] = 2 * xh + ((p + x.c[1] + z + x.c[3]) & 1);
    s = p * g.Vh + xh + g.Lh0 * (x.c[1] + g.L[1] * (z + g.L[2] * x.c[3]));
}
// This workgroup's parity and index within it.
__device__ __forceinline__ int trav_block(const Trav &tr, int &p)
{
    if (tr.nblk8 > 0) {
        const int b = blockIdx.x, i = b >> 3;
        p = i & 1;
        return (b & 7) * tr.nblk8 + (i >> 1);
    }
    p = blockIdx.y;
    return blockIdx.x;
}
// This thread's unit: parity p, site x, its blocked index s and sub-index
// (0 .. ups-1).  False past the end.
__device__ __forceinline__ bool trav_unit(const Geom &g, const Trav &tr, int &p, Site &x, int &s, int &sub)
{
    const int u = trav_block(tr, p) * blockDim.x + threadIdx.x;
    if (u >= tr.nunits) return false;
    const int v = fdiv(u, tr.dups);
    sub = u - v * tr.ups;
    trav_walk(g, tr, p, v, x, s);
    return true;
}
// ---- APE ---------------------------------------------------------------------
struct ApeArgs {
    const double2 *in;
    double2 *out;
    Geom g;
    Trav tr;        // units: sites
    FastDiv d3;
    double alpha;
    ProjConst pc;
};

// out_mu(x) = P[ U_mu(x) + alpha (forward staples over nu != mu in ascending
// order, then the backward ones) ].  The three links of 64 sites are three
// consecutive wavefronts, one per direction: they share most of their staples'
// links through the CU's cache, and the 64 lanes of a load read one component
// array at consecutive sites, 16 cache accesses a load.  With the three links
// of a site on adjacent lanes almost every lane was an access of its own (57 a
// load), and the kernel spent its time there.  24^3x48: 330 -> 293 us a step, the
// same bits; now bound by the FP64 ALU at two wavefronts per SIMD (3,390 vector
// instructions a thread, 2,500 of them the projection).  Three wavefronts (168
// registers) spill.
// Four wavefronts per workgroup (of three, two workgroups would leave a
// quarter of a CU's eight register-limited wavefront places empty).
constexpr int kApeWaves = 4;
__global__ __launch_bounds__(64 * kApeWaves) void ape_step_kernel(ApeArgs a)
{
    const Geom &g = a.g;
    int p, s;
    const int q = __builtin_amdgcn_readfirstlane(trav_block(a.tr, p) * kApeWaves + (int)(threadIdx.x >> 6));
    const int group = fdiv(q, a.d3), mu = q - 3 * group, v = group * 64 + (int)(threadIdx.x & 63);
    if (v >= a.tr.nunits) return;
    Site x;
    trav_walk(g, a.tr, p, v, x, s);
    const int V = g.V;
    const int xpm = blocked(g, step(g, x, mu, +1));
    const int nus[2] = {mu == 0 ? 1 : 0, mu == 2 ? 1 : 2};
    Mat S;
#pragma unroll
    for (int k = 0; k < 9; k++) S.a[k] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int nu = nus[j];
        const Mat T = mm(ldm(a.in, V, nu, s), ldm(a.in, V, mu, blocked(g, step(g, x, nu, +1))));
        const Mat F = mmd(T, ldm(a.in, V, nu, xpm));
#pragma unroll
        for (int k = 0; k < 9; k++) S.a[k] = S.a[k] + F.a[k];
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int nu = nus[j];
        const Site xm = step(g, x, nu, -1);
        const int sxm = blocked(g, xm);
        const Mat T = mm(ldm(a.in, V, mu, sxm), ldm(a.in, V, nu, blocked(g, step(g, xm, mu, +1))));
        const Mat B = mdm(ldm(a.in, V, nu, sxm), T);
#pragma unroll
        for (int k = 0; k < 9; k++) S.a[k] = S.a[k] + B.a[k];
    }
    const Mat U = ldm(a.in, V, mu, s);
#pragma unroll
    for (int k = 0; k < 9; k++) S.a[k] = {a.alpha * S.a[k].re + U.a[k].re, a.alpha * S.a[k].im + U.a[k].im};
    su3_project(S, a.pc);
    stm(a.out, V, mu, s, S);
}

__global__ __launch_bounds__(kThreads) void project_kernel(double2 *U, int V, ProjConst pc)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= V) return;
    const int mu = blockIdx.y;
    Mat M = ldm(U, V, mu, s);
    su3_project(M, pc);
    stm(U, V, mu, s, M);
}

// ---- plaquette -----------------------------------------------------------------
// Re tr[U_mu(x) U_nu(x+mu) (U_nu(x) U_mu(x+nu))^dag] over the six planes.
// The time-boundary sign of a gauge field cancels in every plaquette (both
// temporal links of a (mu, t) plaquette sit on the same time slice), so the
// stored links are used as they are.
__global__ __launch_bounds__(kThreads) void plaq_kernel(const double2 *U, Geom g, double *partial)
{
    double acc = 0.0;
    const int V = g.V;
    for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < V; s += gridDim.x * blockDim.x) {
        const int p = s >= g.Vh ? 1 : 0;
        const Site x = coords(g, p, s - p * g.Vh);
        int sp[4];
#pragma unroll
        for (int m = 0; m < 4; m++) sp[m] = blocked(g, step(g, x, m, +1));
#pragma unroll
        for (int mu = 0; mu < 3; mu++)
#pragma unroll
            for (int nu = mu + 1; nu < 4; nu++) {
                const Mat P1 = mm(ldm(U, V, mu, s), ldm(U, V, nu, sp[mu]));
                const Mat P2 = mm(ldm(U, V, nu, s), ldm(U, V, mu, sp[nu]));
#pragma unroll
                for (int k = 0; k < 9; k++) acc += P1.a[k].re * P2.a[k].re + P1.a[k].im * P2.a[k].im;
            }
    }
    __shared__ double lds[kThreads / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < (int)(blockDim.x >> 6); i++) t += lds[i];
        partial[blockIdx.x] = t;
    }
}

// ---- Gaussian smearing -------------------------------------------------------
struct GaussArgs {
    SpinorD in, out;
    const double2 *U;
    Geom g;
    Trav tr;        // nr threads per site
    int nr;
    double alpha, norm;
};

// tot += U psi (forward hop) or U^dag psi (backward hop) on the four spins;
// the link elements come from get(k)
template <bool BWD, class GetU>
__device__ __forceinline__ void gauss_hop(C tot[12], GetU get, const C ps[12])
{
#pragma unroll
    for (int i = 0; i < 3; i++) {
        C u0, u1, u2;   // row i of U, or column i of U for U^dag
        if (BWD) { u0 = get(i); u1 = get(3 + i); u2 = get(6 + i); }
        else { u0 = get(3 * i); u1 = get(3 * i + 1); u2 = get(3 * i + 2); }
#pragma unroll
        for (int sp = 0; sp < 4; sp++) {
            const C h = BWD ? cjmac(cjmac(cjmul_f(u0, ps[3 * sp]), u1, ps[3 * sp + 1]), u2, ps[3 * sp + 2])
                            : cmac(cmac(cmul_f(u0, ps[3 * sp]), u1, ps[3 * sp + 1]), u2, ps[3 * sp + 2]);
            tot[3 * sp + i] = tot[3 * sp + i] + h;
        }
    }
}

// The output is not read again in the launch: streamed stores keep its
// 2.3 KB per site (12 FP64 right-hand sides) out of the L2 that holds the
// neighbour spinors.
__device__ __forceinline__ void gauss_finish(const GaussArgs &a, int e, const C tot[12])
{
    typedef __attribute__((ext_vector_type(4))) unsigned int U4;
    C v[12];
    a.in.load(e, v);
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const double2 o = make_double2(a.norm * (v[k].re + a.alpha * tot[k].re), a.norm * (v[k].im + a.alpha * tot[k].im));
        U4 w;
        __builtin_memcpy(&w, &o, sizeof(o));
        __builtin_nontemporal_store(w, reinterpret_cast<U4 *>(a.out.p + (size_t)k * a.out.stride) + (uint32_t)e);
    }
}

// out(x) = norm (in(x) + alpha sum_{mu<3} [U_mu(x) in(x+mu) + U_mu(x-mu)^dag in(x-mu)])
// One thread per (site, right-hand side); the right-hand sides of a site are
// adjacent lanes and read the same links (one memory transaction).  Staging
// the links in LDS, or ordering the six hops with register fences, measured
// no faster.
__global__ __launch_bounds__(kThreads) void gauss_step_kernel(GaussArgs a)
{
    const Geom &g = a.g;
    int p, s, r;
    Site x;
    if (!trav_unit(g, a.tr, p, x, s, r)) return;
    const int V = g.V, nr = a.nr;
    C tot[12];
#pragma unroll
    for (int k = 0; k < 12; k++) tot[k] = {0.0, 0.0};
#pragma unroll
    for (int h = 0; h < 6; h++) {
        const int mu = h >> 1;
        const bool bwd = h & 1;
        const int sn = blocked(g, step(g, x, mu, bwd ? -1 : +1));
        const Mat U = ldm(a.U, V, mu, bwd ? sn : s);
        C ps[12];
        a.in.load(sn * nr + r, ps);
        auto get = [&](int k) { return U.a[k]; };
        if (bwd) gauss_hop<true>(tot, get, ps);
        else gauss_hop<false>(tot, get, ps);
    }
    gauss_finish(a, s * nr + r, tot);
}

ProjConst proj_const()
{
    return ProjConst{std::pow(18., 1. / 3.), std::pow(12., 1. / 3.), std::pow(2. / 3., 1. / 3.), std::sqrt(3.)};
}

// The same step, marching along z: a workgroup owns 64 (column, right-hand
// side) units of one time slice -- a column is a fixed (x, y) -- and walks z0 ..
// z0 + zlen - 1.  Wavefront w works on spin w (the hop does not mix spins), so a
// unit's spinor is three complex numbers per thread: psi(z) and psi(z + 1) stay
// in registers from one plane to the next, and the backward z hop is formed one
// plane early, where its link and spinor are at hand, and carried.  The five
// links of a site's plane (U_x, U_x(x-1), U_y, U_y(y-1), U_z) go to LDS once
// for the four spins and all right-hand sides.  Per (site, spin, right-hand
// side) that is 15 loads of 16 B, where gauss_step_kernel has 138 / 4; and the
// workgroups of a slice walk the same few z planes at a time, so a plane's x
// and y neighbours are in the XCD's L2 when they are read.  Every sum has
// gauss_step_kernel's order: the same bits.  12 right-hand sides at 24^3x48:
// 1015 -> 910 us a step, 4.9 GB of HBM traffic (3.3 compulsory) at 5.4 TB/s; a
// 48^3 slice 192 -> 172 us.
struct GaussMarch {
    const double2 *in;
    double2 *out;
    const double2 *U;
    Geom g;
    FastDiv dnr, dwpp, dseg;
    size_t stride;    // entries of one component
    int nr, cols;     // units of one slice
    int wpp, nseg;    // workgroups per plane, segments of z
    int zlen, t_lo, nblk, nblk8;
    double alpha, norm;
};
constexpr int kMarchLinks = 5;

// tot += U psi or U^dag psi of one spin, in gauss_hop's order
template <bool BWD> __device__ __forceinline__ void march_hop(C tot[3], const double2 *l, const C ps[3])
{
#pragma unroll
    for (int i = 0; i < 3; i++) {
        C u[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const double2 d = BWD ? l[3 * j + i] : l[3 * i + j];
            u[j] = {d.x, d.y};
        }
        const C h = BWD ? cjmac(cjmac(cjmul_f(u[0], ps[0]), u[1], ps[1]), u[2], ps[2])
                        : cmac(cmac(cmul_f(u[0], ps[0]), u[1], ps[1]), u[2], ps[2]);
        tot[i] = tot[i] + h;
    }
}

__device__ __forceinline__ void pin_vec(C t[3])
{
    asm volatile("" : "+v"(t[0].re), "+v"(t[0].im), "+v"(t[1].re), "+v"(t[1].im), "+v"(t[2].re), "+v"(t[2].im)::"memory");
}

template <int NL> __global__ __launch_bounds__(256) void gauss_march_kernel(GaussMarch a)
{
    extern __shared__ double2 march_links[];
    const Geom &g = a.g;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int b = a.nblk8 > 0 ? ((int)blockIdx.x & 7) * a.nblk8 + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
    if (b >= a.nblk) return;   // uniform over the workgroup
    const int pl = fdiv(b, a.dwpp), pw = b - pl * a.wpp;
    const int tt = fdiv(pl, a.dseg), z0 = (pl - tt * a.nseg) * a.zlen;
    const int t = a.t_lo + tt, n = min(a.zlen, g.L[2] - z0);
    const int V = g.V, plane = g.Lh0 * g.L[1], tbase = plane * g.L[2] * t;
    // column q of a slice: xh fastest, then x's parity, then y
    auto column = [&](int q, int &x, int &y) {
        const int rest = fdiv(q, g.dLh0);
        x = 2 * (q - rest * g.Lh0) + (rest & 1);
        y = rest >> 1;
    };
    const int u0 = pw * 64;
    const bool own = u0 + lane < a.cols;
    const int u = min(u0 + lane, a.cols - 1);
    const int q = fdiv(u, a.dnr), r = u - q * a.nr, q0 = fdiv(u0, a.dnr);
    const int ns = fdiv(min(u0 + 63, a.cols - 1), a.dnr) - q0 + 1;   // sites of this workgroup
    int x, y;
    column(q, x, y);
    const int xy = x + y + t;   // parity of the site at z: (xy + z) & 1
    const int cb = tbase + (x >> 1) + g.Lh0 * y;
    const int cxp = tbase + ((x + 1 == g.L[0] ? 0 : x + 1) >> 1) + g.Lh0 * y;
    const int cxm = tbase + ((x == 0 ? g.L[0] - 1 : x - 1) >> 1) + g.Lh0 * y;
    const int cyp = tbase + (x >> 1) + g.Lh0 * (y + 1 == g.L[1] ? 0 : y + 1);
    const int cym = tbase + (x >> 1) + g.Lh0 * (y == 0 ? g.L[1] - 1 : y - 1);
    const double2 *in = a.in + (size_t)(3 * w) * a.stride + r;
    auto load = [&](int c, int z, int par, C v[3]) __attribute__((always_inline)) {
        const size_t e = (size_t)((par ? g.Vh : 0) + c + plane * z) * a.nr;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double2 d = in[(size_t)k * a.stride + e];
            v[k] = {d.x, d.y};
        }
    };
    // this thread's link elements: (site j, link l, element k), sites fastest
    int lsrc[NL], lpar[NL], ldst[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        // past the last element: the last one again (not stored)
        const int id = min((int)threadIdx.x + 256 * i, ns * 9 * kMarchLinks - 1);
        const int e = id / ns, j = id - e * ns, l = e / 9, k = e - 9 * l;
        int lx, ly;
        column(q0 + j, lx, ly);
        ldst[i] = j * 9 * kMarchLinks + e;
        lpar[i] = lx + ly + t + (l & 1);   // links 1 and 3 sit on the other parity
        if (l == 1) lx = lx == 0 ? g.L[0] - 1 : lx - 1;
        if (l == 3) ly = ly == 0 ? g.L[1] - 1 : ly - 1;
        lsrc[i] = ((l >> 1) * 9 + k) * V + tbase + (lx >> 1) + g.Lh0 * ly;
    }
    double lre[NL], lim[NL];
    auto fetch_links = [&](int z) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const double2 d = a.U[(size_t)lsrc[i] + (((lpar[i] + z) & 1) ? g.Vh : 0) + plane * z];
            lre[i] = d.x;
            lim[i] = d.y;
        }
    };
    auto put_links = [&]() __attribute__((always_inline)) {
        __syncthreads();   // the last plane's links have been read
#pragma unroll
        for (int i = 0; i < NL; i++)
            if ((int)threadIdx.x + 256 * i < ns * 9 * kMarchLinks) march_links[ldst[i]] = make_double2(lre[i], lim[i]);
        __syncthreads();
    };
    const double2 *link = march_links + (q - q0) * 9 * kMarchLinks;
    C pc[3], carry[3] = {{0, 0}, {0, 0}, {0, 0}};
    {
        const int zm = z0 == 0 ? g.L[2] - 1 : z0 - 1;
        C pm[3];
        fetch_links(zm);
        load(cb, zm, (xy + zm) & 1, pm);
        load(cb, z0, (xy + z0) & 1, pc);
        put_links();
        fetch_links(z0);
        march_hop<true>(carry, link + 36, pm);
    }
    for (int i = 0; i < n; i++) {
        const int z = z0 + i, zp = z + 1 == g.L[2] ? 0 : z + 1, par = (xy + z) & 1;
        C pn[3], nb[4][3];
        load(cxp, z, par ^ 1, nb[0]);
        load(cxm, z, par ^ 1, nb[1]);
        load(cyp, z, par ^ 1, nb[2]);
        load(cym, z, par ^ 1, nb[3]);
        load(cb, zp, (xy + zp) & 1, pn);
        put_links();
        if (i + 1 < n) fetch_links(zp);
        C tot[3] = {{0, 0}, {0, 0}, {0, 0}};
        // one link of LDS reads in flight at a time: all five take 180 registers
        march_hop<false>(tot, link, nb[0]);
        pin_vec(tot);
        march_hop<true>(tot, link + 9, nb[1]);
        pin_vec(tot);
        march_hop<false>(tot, link + 18, nb[2]);
        pin_vec(tot);
        march_hop<true>(tot, link + 27, nb[3]);
        pin_vec(tot);
        march_hop<false>(tot, link + 36, pn);
        pin_vec(tot);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            tot[k] = tot[k] + carry[k];
            carry[k] = {0, 0};
        }
        march_hop<true>(carry, link + 36, pc);
        if (own) {
            typedef __attribute__((ext_vector_type(2))) double d2v;
            double2 *o = a.out + (size_t)(3 * w) * a.stride + r + (size_t)((par ? g.Vh : 0) + cb + plane * z) * a.nr;
#pragma unroll
            for (int k = 0; k < 3; k++)
                __builtin_nontemporal_store(d2v{a.norm * (pc[k].re + a.alpha * tot[k].re),
                                                a.norm * (pc[k].im + a.alpha * tot[k].im)},
                                            reinterpret_cast<d2v *>(o + (size_t)k * a.stride));
        }
#pragma unroll
        for (int k = 0; k < 3; k++) pc[k] = pn[k];
    }
}

// Launch shape of the march over the slices of a smearing, `lds` bytes of links
struct MarchGrid {
    dim3 grid;
    size_t lds;
    int loads;   // link elements per thread
};
MarchGrid make_march(GaussMarch &m, const qkx_gauge_s *U, int nr, int t, double alpha)
{
    const int *L = U->L;
    m.U = (const double2 *)U->data;
    m.g = qkx::make_geom(L, U->bc);
    m.nr = nr;
    m.dnr = make_fastdiv(nr);
    m.stride = (size_t)U->V * nr;
    m.cols = L[0] * L[1] * nr;
    m.wpp = (m.cols + 63) / 64;
    m.t_lo = t < 0 ? 0 : t;
    const int nt = t < 0 ? L[3] : 1;
    // z in segments (each re-reads one plane) while the slices alone do not
    // give every CU three rounds of resident workgroups; four planes at least
    constexpr int kMarchFill = 2304;
    m.nseg = std::max(1, std::min((kMarchFill + m.wpp * nt - 1) / (m.wpp * nt), L[2] / 4));
    m.zlen = (L[2] + m.nseg - 1) / m.nseg;
    m.nseg = (L[2] + m.zlen - 1) / m.zlen;
    m.dwpp = make_fastdiv(m.wpp);
    m.dseg = make_fastdiv(m.nseg);
    m.nblk = m.wpp * nt * m.nseg;
    m.nblk8 = m.nblk >= 64 ? (m.nblk + 7) / 8 : 0;
    m.alpha = alpha;
    m.norm = 1.0 / (1 + 6 * alpha);
    const int sites = std::min(64, 63 / nr + 2);   // of a workgroup, at most
    MarchGrid r;
    r.lds = (size_t)sites * 9 * kMarchLinks * sizeof(double2);
    r.loads = (sites * 9 * kMarchLinks + 255) / 256;
    r.grid = dim3(m.nblk8 ? 8 * m.nblk8 : m.nblk);
    return r;
}
void launch_march(const GaussMarch &m, const MarchGrid &r)
{
    if (r.loads <= 2) hipLaunchKernelGGL(gauss_march_kernel<2>, r.grid, dim3(256), r.lds, qkx::g_stream, m);
    else if (r.loads <= 3) hipLaunchKernelGGL(gauss_march_kernel<3>, r.grid, dim3(256), r.lds, qkx::g_stream, m);
    else if (r.loads <= 6) hipLaunchKernelGGL(gauss_march_kernel<6>, r.grid, dim3(256), r.lds, qkx::g_stream, m);
    else hipLaunchKernelGGL(gauss_march_kernel<12>, r.grid, dim3(256), r.lds, qkx::g_stream, m);
}
// A step of at least this many (site, right-hand side) units marches: 24 planes in
// a row are a chain that needs enough workgroups beside it.  The line is where the
// two forms cross on average; a shape near it may be either way by a few percent.
// us a step, per unit / marching:
//   16^3x32, 1 RHS (131,072)  29.6 / 24.8    slice  48^3, 1 RHS (110,592)  23.6 / 25.1
//   14^3x24, 2     (131,712)  29.7 / 23.6           32^3, 4     (131,072)  22.8 / 19.4
//   12^3x20, 4     (138,240)  23.4 / 24.0           28^3, 6     (131,712)  22.4 / 23.3
//   12^3x24, 4     (165,888)  25.0 / 23.9           24^3, 10    (138,240)  22.4 / 23.2
//   8^3x16, 12      (98,304)  26.9 / 29.4           24^3, 13    (179,712)  27.2 / 25.9
constexpr long kMarchUnits = 131072;
// its link elements are indexed with 32 bits
constexpr long kMarchSites = ((1L << 31) - 1) / 27;

bool fp64_links(const qkx_gauge_s *g) { return g && g->prec == QKX_PREC_DOUBLE && g->recon == QKX_RECON_18; }

// Spatial-link workspace of the APE ping-pong, kept between calls (a smearing
// run calls this once per configuration; re-allocating 432 B per site each
// time would cost more than a step).  Grows on demand; work queued on the
// library stream against the old buffer finishes before it is freed.
double2 *g_ape_ws = nullptr;
size_t g_ape_ws_bytes = 0;

double2 *ape_workspace(size_t bytes)
{
    if (bytes <= g_ape_ws_bytes) return g_ape_ws;
    if (g_ape_ws) {
        (void)hipStreamSynchronize(qkx::g_stream);
        (void)hipFree(g_ape_ws);
    }
    g_ape_ws = nullptr;
    g_ape_ws_bytes = 0;
    if (hipMalloc(&g_ape_ws, bytes) != hipSuccess) {
        g_ape_ws = nullptr;
        return nullptr;
    }
    g_ape_ws_bytes = bytes;
    return g_ape_ws;
}

} // namespace

namespace qkx {
void smear_release()
{
    if (g_ape_ws) (void)hipFree(g_ape_ws);
    g_ape_ws = nullptr;
    g_ape_ws_bytes = 0;
}
} // namespace qkx

extern "C" {

int qkx_gauge_project_su3(qkx_gauge *g)
{
    QKX_CHECK_ARG(fp64_links(g), "qkx_gauge_project_su3: the gauge field must be FP64 recon 18");
    hipLaunchKernelGGL(project_kernel, dim3((g->V + kThreads - 1) / kThreads, 3), dim3(kThreads), 0, qkx::g_stream,
                       (double2 *)g->data, g->V, proj_const());
    QKX_HIP(hipGetLastError());
    qkx::gauge_modified(g);
    return QKX_SUCCESS;
}

int qkx_ape_smear(qkx_gauge *out, const qkx_gauge *in, int nsmear, double alpha)
{
    QKX_CHECK_ARG(fp64_links(out) && fp64_links(in), "qkx_ape_smear: both gauge fields must be FP64 recon 18");
    QKX_CHECK_ARG(out != in, "qkx_ape_smear: out and in must be different fields");
    QKX_CHECK_ARG(out->V == in->V && out->L[0] == in->L[0] && out->L[1] == in->L[1] && out->L[2] == in->L[2],
                  "qkx_ape_smear: lattices differ");
    QKX_CHECK_ARG(out->bc == in->bc, "qkx_ape_smear: boundaryT of out and in differ");
    QKX_CHECK_ARG(nsmear >= 0, "qkx_ape_smear: nsmear must be >= 0");
    if (nsmear == 0) return QKX_SUCCESS;   // the reference returns before touching the field
    const int V = in->V;
    double2 *tmp = nullptr;
    if (nsmear > 1 && !(tmp = ape_workspace((size_t)3 * 9 * V * sizeof(double2)))) {
        qkx::set_error("qkx_ape_smear: out of device memory");
        return QKX_ERR_NOMEM;
    }
    ApeArgs a;
    a.g = qkx::make_geom(in->L, in->bc);
    dim3 grid;
    a.tr = make_trav(in->L, 1, -1, grid, [](int n) { return ((n + 63) / 64 * 3 + kApeWaves - 1) / kApeWaves; });
    a.d3 = make_fastdiv(3);
    a.alpha = alpha;
    a.pc = proj_const();
    // ping-pong so that the last step lands in out
    double2 *bufs[2] = {(double2 *)out->data, tmp};
    const double2 *src = (const double2 *)in->data;
    for (int it = 0; it < nsmear; it++) {
        double2 *dst = bufs[(nsmear - 1 - it) & 1];
        a.in = src;
        a.out = dst;
        hipLaunchKernelGGL(ape_step_kernel, grid, dim3(64 * kApeWaves), 0, qkx::g_stream, a);
        src = dst;
    }
    QKX_HIP(hipGetLastError());
    // temporal links: in's
    QKX_HIP(hipMemcpyAsync((double2 *)out->data + (size_t)3 * 9 * V, (const double2 *)in->data + (size_t)3 * 9 * V,
                           (size_t)9 * V * sizeof(double2), hipMemcpyDeviceToDevice, qkx::g_stream));
    qkx::gauge_modified(out);
    return QKX_SUCCESS;
}

int qkx_plaquette(double *plaq, const qkx_gauge *g)
{
    QKX_CHECK_ARG(plaq && fp64_links(g), "qkx_plaquette: the gauge field must be FP64 recon 18");
    const int nb = std::min(kPlaqBlocks, (g->V + kThreads - 1) / kThreads);
    Geom geo = qkx::make_geom(g->L, g->bc);
    hipLaunchKernelGGL(plaq_kernel, dim3(nb), dim3(kThreads), 0, qkx::g_stream, (const double2 *)g->data, geo,
                       qkx::reduce_scratch());
    QKX_HIP(hipGetLastError());
    int rc = qkx::finish_sum_dev(qkx::reduce_scratch(), nb, qkx::reduce_result());
    if (rc) return rc;
    double sum = 0;
    QKX_HIP(hipMemcpyAsync(&sum, qkx::reduce_result(), sizeof(double), hipMemcpyDeviceToHost, qkx::g_stream));
    QKX_HIP(hipStreamSynchronize(qkx::g_stream));
    *plaq = sum / ((double)g->V * 3.0 * 6.0);
    return QKX_SUCCESS;
}

int qkx_gauss_smear(qkx_spinor *out, const qkx_spinor *in, const qkx_gauge *U, int nsmear, double alpha, int t)
{
    QKX_CHECK_ARG(out && in && fp64_links(U), "qkx_gauss_smear: null field or gauge field not FP64 recon 18");
    QKX_CHECK_ARG(out != in, "qkx_gauss_smear: out and in must be different fields");
    QKX_CHECK_ARG(in->prec == QKX_PREC_DOUBLE && out->prec == QKX_PREC_DOUBLE && in->subset == QKX_SUBSET_FULL &&
                      out->subset == QKX_SUBSET_FULL,
                  "qkx_gauss_smear: spinors must be full FP64 fields");
    QKX_CHECK_ARG(in->V == U->V && out->V == in->V && out->nrhs == in->nrhs &&
                      in->L[0] == U->L[0] && in->L[1] == U->L[1] && in->L[2] == U->L[2],
                  "qkx_gauss_smear: fields differ in lattice or number of right-hand sides");
    QKX_CHECK_ARG(nsmear >= 0, "qkx_gauss_smear: nsmear must be >= 0");
    QKX_CHECK_ARG(t >= -1 && t < in->L[3], "qkx_gauss_smear: t must be -1 (all slices) or a time slice");
    if (nsmear == 0) return QKX_SUCCESS;   // the reference returns before touching the field
    const int *L = in->L;
    const int nr = in->nrhs;
    const bool march = (long)L[0] * L[1] * L[2] * (t < 0 ? L[3] : 1) * nr >= kMarchUnits && in->V <= kMarchSites;
    GaussMarch m;
    GaussArgs a;
    MarchGrid mg;
    dim3 grid;
    if (march) {
        mg = make_march(m, U, nr, t, alpha);
    } else {
        a.U = (const double2 *)U->data;
        a.g = qkx::make_geom(L, U->bc);
        a.nr = nr;
        a.tr = make_trav(L, nr, t, grid, [](int n) { return (n + kThreads - 1) / kThreads; });
        a.alpha = alpha;
        a.norm = 1.0 / (1 + 6 * alpha);
    }
    int rc;
    if (t >= 0 && (rc = qkx_spinor_zero(out))) return rc;
    std::unique_ptr<qkx::Temp> tmp;
    if (nsmear > 1) {
        tmp.reset(new qkx::Temp(L, QKX_PREC_DOUBLE, QKX_SUBSET_FULL, nr));
        if (!tmp->f) { qkx::set_error("qkx_gauss_smear: out of device memory"); return QKX_ERR_NOMEM; }
        // a pooled temporary may hold anything outside the smeared slice; it
        // is never read there
    }
    qkx_spinor_s *bufs[2] = {out, tmp ? tmp->f : nullptr};
    const qkx_spinor_s *src = in;
    for (int it = 0; it < nsmear; it++) {
        qkx_spinor_s *dst = bufs[(nsmear - 1 - it) & 1];
        if (march) {
            m.in = (const double2 *)src->data;
            m.out = (double2 *)dst->data;
            launch_march(m, mg);
        } else {
            a.in = make_spinor<SpinorD>(src);
            a.out = make_spinor<SpinorD>(dst);
            hipLaunchKernelGGL(gauss_step_kernel, grid, dim3(kThreads), 0, qkx::g_stream, a);
        }
        src = dst;
    }
    QKX_HIP(hipGetLastError());
    return QKX_SUCCESS;
}

} // extern "C"
