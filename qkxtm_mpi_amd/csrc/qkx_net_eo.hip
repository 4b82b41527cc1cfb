// qkx_net_eo.hip -- the learned preconditioner on even-parity fields, as the
// right preconditioner of the even-odd solvers applies it (qkx_learned.hip
// holds the network, its training and the full-lattice form).
#include "qkx_net.h"

namespace {

// ---------------------------------------------------------------------------
// The network on even-parity fields, N_e = P_e L2 L1 P_e (P_e: restriction to
// the even sites), batched over right-hand sides (RHS innermost).  With the
// input zero on the odd sites, L1's hidden channels are W1[0] in(x) at an even
// site x and sum_{p>0} W1[p] (T_p in)(y) at an odd site y (all neighbours of y
// are even), and L2's output at x is
//   C0 in(x) + sum_{p>0} W2[p] (T_p h)(x),   C0 = W2[0] W1[0]  (4 x 4),
// whose hops read only odd-site hidden channels.  So N_e is two launches:
// eo_hidden_kernel (odd sites) and eo_out_kernel (even sites).  The adjoint
// N_e^dag = P_e L1^dag L2^dag P_e has the same form with the adjoint layers'
// weights, A[p][a][b] = conj(W[rev p][b][a]).
//
// Weight table of one direction (forward or adjoint), complex:
//   [8][CH][4] first-layer hops (p = 1..8), [8][4][CH] second-layer hops,
//   [4][4] C0.
constexpr int eo_table(int ch) { return 8 * ch * 4 * 2 + 16; }

__device__ __forceinline__ float2 net_w(const float2 *w, const uint32_t *wb, int bf, int i)
{
    if (!bf) return w[i];
    const uint32_t h = wb[i];
    return make_float2(bf2f(h & 0xffffu), bf2f(h >> 16));
}

// Both tables from the FP32 master weights or their BF16 copies: thread i
// writes entry i of [forward table][adjoint table].
__global__ void eo_weights_kernel(const float2 *w, const uint32_t *wb, int bf, int ch, float2 *out)
{
    const int T = eo_table(ch), i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * T) return;
    const int adj = i / T, j = i % T, n1 = 9 * ch * 4;
    auto W1 = [&](int p, int a, int b) { return net_w(w, wb, bf, (p * ch + a) * 4 + b); };    // [9][ch][4]
    auto W2 = [&](int p, int a, int b) { return net_w(w, wb, bf, n1 + (p * 4 + a) * ch + b); };   // [9][4][ch]
    auto cj = [](float2 v) { return make_float2(v.x, -v.y); };
    const int h1 = 8 * ch * 4;
    float2 v;
    if (j < h1) {                       // first layer, p = 1..8: [a < ch][b < 4]
        const int p = j / (ch * 4) + 1, a = (j / 4) % ch, b = j % 4;
        v = adj ? cj(W2(rev_path(p), b, a)) : W1(p, a, b);
    } else if (j < 2 * h1) {            // second layer: [a < 4][b < ch]
        const int k = j - h1, p = k / (4 * ch) + 1, a = (k / ch) % 4, b = k % ch;
        v = adj ? cj(W1(rev_path(p), b, a)) : W2(p, a, b);
    } else {                            // C0 = W2[0] W1[0], or its adjoint
        const int k = j - 2 * h1, a = adj ? k % 4 : k / 4, b = adj ? k / 4 : k % 4;
        float re = 0.f, im = 0.f;
        for (int c = 0; c < ch; c++) {
            const float2 x = W2(0, a, c), y = W1(0, c, b);
            re += x.x * y.x - x.y * y.y;
            im += x.x * y.y + x.y * y.x;
        }
        v = adj ? make_float2(re, -im) : make_float2(re, im);
    }
    out[i] = v;
}

// Units of a launch: (site, rhs r0 .. r0 + nc - 1) of a batch of nr, upb per
// workgroup, one thread each.  SHARE: a workgroup holds whole sites (upb a
// multiple of nc); it fetches the 8 links of each of its sites once, one
// thread per (site, direction), into LDS, and the nc threads of a site read
// them from there.  What bounds these kernels is the vector-memory pipe (a
// wavefront's load takes it 16 cycles whatever its width): with every thread
// fetching its own 8 links, 72 of the 112 loads per thread of eo_hidden_kernel
// were link loads.  Sites are walked in blocks (blocked_walk): in checkerboard
// order the t neighbours' 1.2 KB per site (12 RHS) leave the L2 before they
// come round, and the two kernels fetched 0.92 and 2.06 GB, now 0.62 and 1.65.
// 12 RHS, FP16, CH = 4, 24^3x48, forward and adjoint: 1979 us with the mixing on
// the vector ALU, 1491-1531 us on the matrix cores, walked in blocks; now bound
// by the vector and matrix pipes (1,680 vector instructions, 400 MFMAs a thread).
struct EoArgs {
    Geom g;
    HopTrav tr;   // order in which the sites are walked
    FastDiv dnc;
    int nr, r0, nc, upb, units, nblk8;
    const int *skip;
};
// w(p, a, b) of a table [8][A][B], p = 1 .. 8
template <int A, int B> struct EoWeights {
    const float2 *w;
    __device__ __forceinline__ float2 operator()(int p, int a, int b) const { return w[((p - 1) * A + a) * B + b]; }
};
extern __shared__ float4 eo_links[];
// this workgroup's first unit; the thread's unit (clamped into the launch) and whether it is its own
__device__ __forceinline__ int eo_unit(const EoArgs &a, int &u, bool &own)
{
    const int u0 = net_block(a.nblk8) * a.upb, i = min((int)threadIdx.x, a.upb - 1);
    own = (int)threadIdx.x < a.upb && u0 + i < a.units;
    u = min(u0 + i, a.units - 1);
    return u0;
}
// the links of the workgroup's sites (parity p, first unit u0) into LDS
__device__ __forceinline__ void eo_share_links(const EoArgs &a, const GaugeF18 &U, int p, int u0)
{
    const Geom &g = a.g;
    const int v0 = fdiv(u0, a.dnc), ns = fdiv(a.upb, a.dnc);
    float *row = reinterpret_cast<float *>(eo_links);
    for (int t = threadIdx.x; t < 8 * ns; t += blockDim.x) {
        const int j = t >> 3, d = t & 7;
        if (v0 + j >= g.Vh) break;
        int cb;
        const HopSite h = hop_site_walk(g, a.tr, p, v0 + j, cb);
        int nb = h.nb[1];
#pragma unroll
        for (int k = 3; k < 8; k += 2) nb = d == k ? h.nb[k] : nb;
        const int s = (d & 1) ? (1 - p) * g.Vh + nb : p * g.Vh + cb;
        const float sg = (d == 6 && h.tw_p) || (d == 7 && h.tw_m) ? (float)g.bc : 1.0f;
        const GaugeF18::Raw r = U.fetch(d >> 1, s);
        float2 *q = reinterpret_cast<float2 *>(row + j * kSiteStride + d * kLinkStride);
#pragma unroll
        for (int k = 0; k < 9; k++) q[k] = make_float2(sg * r.c[k].x, sg * r.c[k].y);
    }
    __syncthreads();
}
// v: the thread's site in the walk
__device__ __forceinline__ LinkShared eo_shared(const EoArgs &a, int v, int u0)
{
    return LinkShared{reinterpret_cast<const float *>(eo_links) + (v - fdiv(u0, a.dnc)) * kSiteStride};
}

// Hidden channels at the odd sites: h_a(y) = sum_{p>0} sum_b w[p][a][b] (T_p in_b)(y).
// in is an even-parity field.
template <int CH, bool SHARE, class S>
__global__ __launch_bounds__(kT) QKX_NET_REGS void eo_hidden_kernel(S in, GaugeF18 U, EoArgs a, EoWeights<CH, 4> w,
                                                                    Hid hid)
{
    if (a.skip && *a.skip) return;   // uniform over the grid
    int u;
    bool own;
    const int u0 = eo_unit(a, u, own);
    if (u0 >= a.units) return;   // uniform over the workgroup
    if constexpr (SHARE) eo_share_links(a, U, 1, u0);
    const int v = fdiv(u, a.dnc), rc = u - v * a.nc, r = a.r0 + rc;
    int cb;
    const NetSite n = net_site_walk(a.g, a.tr, 1, v, cb);
    f4v re[CH / 4][3], im[CH / 4][3];
#pragma unroll
    for (int h = 0; h < CH / 4; h++) {
        zero3(re[h]);
        zero3(im[h]);
    }
    const int nr = a.nr;
    auto unit = [&](int site) { return site * nr + r; };   // even sites: blocked = checkerboard index
    if constexpr (SHARE) expand<CH, 1, 9>(in, eo_shared(a, v, u0), n, unit, w, re, im);
    else expand<CH, 1, 9>(in, LinkGlobal{U, a.g, n}, n, unit, w, re, im);
    if (own) {
#pragma unroll
        for (int h = 0; h < CH / 4; h++) hid.store(h, cb * a.nc + rc, re[h], im[h]);
    }
}

// Output at the even sites: out(x) = C0 in(x) + sum_{p>0} (T_p m_p)(x) with
// m_p = w[p] h at the odd neighbour (the channels are mixed first, then the
// four colour vectors transported).
template <int CH, bool SHARE, class S>
__global__ __launch_bounds__(kT) QKX_NET_REGS void eo_out_kernel(S in, S out, GaugeF18 U, EoArgs a, EoWeights<4, CH> w,
                                                                 const float2 *__restrict__ c0, Hid hid)
{
    if (a.skip && *a.skip) return;   // uniform over the grid
    int u;
    bool own;
    const int u0 = eo_unit(a, u, own);
    if (u0 >= a.units) return;   // uniform over the workgroup
    if constexpr (SHARE) eo_share_links(a, U, 0, u0);
    const int v = fdiv(u, a.dnc), rc = u - v * a.nc;
    int cb;
    const NetSite n = net_site_walk(a.g, a.tr, 0, v, cb);
    const int e = cb * a.nr + a.r0 + rc;   // the unit's entry in the batch fields
    const int nc = a.nc, Vh = a.g.Vh;
    auto hunit = [&](int site) { return (site - Vh) * nc + rc; };
    Cx<float> acc[12];
    {
        const float wc = mix_weights([&](int i, int b) { return c0[i * 4 + b]; });
        Cx<float> x[12];
        const float f = unpack_spinor(in, in.template fetch<3>(e), x);
        f4v re[3], im[3];
        zero3(re);
        zero3(im);
        mix_tile(wc, x, re, im);
#pragma unroll
        for (int k = 0; k < 12; k++) acc[k] = {f * re[k % 3][k / 3], f * im[k % 3][k / 3]};
    }
    if constexpr (SHARE) contract<CH, 1, 9>(hid, eo_shared(a, v, u0), n, hunit, w, acc);
    else contract<CH, 1, 9>(hid, LinkGlobal{U, a.g, n}, n, hunit, w, acc);
    if (!own) return;
    using R = typename S::Real;
    Cx<R> o[12];
#pragma unroll
    for (int k = 0; k < 12; k++) o[k] = {(R)acc[k].re, (R)acc[k].im};
    out.store(e, o);
}

// Links are shared from this many right-hand sides on.  With 4 hidden channels
// the kernels are light enough to run five wavefronts per SIMD with a thread's own
// links, which few right-hand sides' workgroups, each with the links of many sites
// in LDS, do not reach: 16^3x32 FP16, shared / own: 3 RHS 77 / 53 us, 5 89 / 69,
// 6 95 / 80 (FP64 129 / 117); 24^4 FP16: 3 RHS 148 / 107, 6 202 / 192 (FP64 336 / 325).
// With 8 channels: 16^3x32 4 RHS 121 / 105, 24^4 4 RHS 216 / 225, 20^3x44 (FP32)
// 6 RHS 371 / 394.
constexpr int eo_share_min(int ch) { return ch == 4 ? 7 : 3; }
// threads per workgroup: 64 while larger ones would leave SIMDs without a
// wavefront; 128 for few right-hand sides, whose workgroups hold many sites'
// links (656 B a site; 42 sites of 3 RHS take 28 KB)
int eo_block(int units, int nc) { return units < 512 * kT ? 64 : nc < 6 ? 128 : kT; }

// right-hand sides per launch of the even-odd network: all of them while
// their hidden channels fit the bound (default kEoHiddenCap float2 entries,
// 4 GiB) and the launch's units an index of 30 bits, else fewer
constexpr size_t kEoHiddenCap = size_t(1) << 29;
constexpr size_t kEoUnits = (size_t(1) << 30) - 1;
int eo_chunk(const qkx_net_s *n, const qkx_spinor_s *in)
{
    const size_t per_rhs = (size_t)n->ch * 3 * (size_t)in->Vh;
    const size_t cap = n->ehid_limit ? n->ehid_limit : kEoHiddenCap;
    const size_t most = std::min(cap / per_rhs, kEoUnits / (size_t)in->Vh);
    return (int)std::max<size_t>(1, std::min<size_t>((size_t)in->nrhs, most));
}

template <int CH, class S>
int launch_eo(qkx_net_s *n, qkx_spinor_s *out, const qkx_spinor_s *in, const qkx_gauge_s *U, int adjoint,
              const int *skip)
{
    EoArgs a;
    a.g = qkx::make_geom(U->L, U->bc);
    a.nr = in->nrhs;
    a.skip = skip;
    const int nc = eo_chunk(n, in);
    const GaugeF18 G = make_gauge<GaugeF18>(U);
    const float2 *tab = n->weo + (adjoint ? eo_table(CH) : 0);
    // the right-hand sides in chunks of nc, so that the hidden channels of a
    // chunk fit the buffer (out may be in: each chunk reads only its own
    // columns before writing them)
    for (int r0 = 0; r0 < a.nr; r0 += nc) {
        a.r0 = r0;
        a.nc = std::min(nc, a.nr - r0);
        a.dnc = make_fastdiv(a.nc);
        a.units = a.g.Vh * a.nc;
        const int bs = eo_block(a.units, a.nc);
        const bool share = a.nc >= eo_share_min(CH);
        a.upb = share ? bs / a.nc * a.nc : bs;
        const size_t lds = share ? (size_t)(a.upb / a.nc) * kSiteStride * sizeof(float) : 0;
        int nb = (a.units + a.upb - 1) / a.upb;
        a.nblk8 = net_remap(nb);
        // the hidden channels set the walk, and part of the spinors (48 B of an FP64
        // one, 24 B of the others): with the larger of the two in full, 16 FP64
        // right-hand sides at 32^3x32 get blocks of fewer t slices and take 2,607 us
        // instead of 2,476; other storages are equal
        a.tr = blocked_walk(a.g, (double)a.g.Lh0 * a.nc * (24.0 * CH + sizeof(typename S::Real) * 6));
        const Hid hid{n->ehid, (size_t)a.units};
        const S si = make_spinor<S>(in), so = make_spinor<S>(out);
        const EoWeights<CH, 4> w1{tab};
        const EoWeights<4, CH> w2{tab + 8 * CH * 4};
        const float2 *c0 = tab + 2 * 8 * CH * 4;
        if (share) {
            hipLaunchKernelGGL((eo_hidden_kernel<CH, true, S>), dim3(nb), dim3(bs), lds, qkx::g_stream, si, G, a, w1, hid);
            hipLaunchKernelGGL((eo_out_kernel<CH, true, S>), dim3(nb), dim3(bs), lds, qkx::g_stream, si, so, G, a, w2, c0, hid);
        } else {
            hipLaunchKernelGGL((eo_hidden_kernel<CH, false, S>), dim3(nb), dim3(bs), 0, qkx::g_stream, si, G, a, w1, hid);
            hipLaunchKernelGGL((eo_out_kernel<CH, false, S>), dim3(nb), dim3(bs), 0, qkx::g_stream, si, so, G, a, w2, c0, hid);
        }
    }
    QKX_HIP(hipGetLastError());
    return QKX_SUCCESS;
}

} // namespace

namespace qkx {
// The even-odd weight tables from the current weights (BF16 copies when
// the network runs in BF16); a solve prepares them once.
int net_prep_eo(qkx_net_s *n)
{
    const int T = eo_table(n->ch);
    if (!n->weo) QKX_HIP(hipMalloc(&n->weo, sizeof(float2) * 2 * T));
    hipLaunchKernelGGL(eo_weights_kernel, dim3((2 * T + 255) / 256), dim3(256), 0, qkx::g_stream, n->w, n->wb,
                       n->bf16, n->ch, n->weo);
    QKX_HIP(hipGetLastError());
    return QKX_SUCCESS;
}

// out = N_e in (adjoint: N_e^dag in) on even-parity fields of one precision
// and batch size; net_prep_eo must have run since the weights last changed.
// out may be in.  skip (optional, device): both launches return at once
// while *skip != 0.
int net_apply_eo(qkx_net_s *n, qkx_spinor_s *out, const qkx_spinor_s *in, const qkx_gauge_s *U, int adjoint,
                 const int *skip)
{
    int rc;
    if ((rc = check_net_gauge(U))) return rc;
    if (in->subset != QKX_SUBSET_EVEN || out->subset != QKX_SUBSET_EVEN || in->prec != out->prec ||
        in->nrhs != out->nrhs || in->L[0] != U->L[0] || in->L[1] != U->L[1] || in->L[2] != U->L[2] ||
        in->L[3] != U->L[3] || out->L[0] != U->L[0] || out->L[1] != U->L[1] || out->L[2] != U->L[2] ||
        out->L[3] != U->L[3]) {
        qkx::set_error("net (even-odd): in and out must be even-parity fields of one precision and batch size on "
                       "the gauge's lattice");
        return QKX_ERR_ARG;
    }
    const size_t need = (size_t)n->ch * 3 * (size_t)in->Vh * eo_chunk(n, in);
    if (need > n->ehid_cap) {
        if (n->ehid) (void)hipFree(n->ehid);
        n->ehid = nullptr;
        n->ehid_cap = 0;
        QKX_HIP(hipMalloc(&n->ehid, sizeof(float2) * need));
        n->ehid_cap = need;
    }
    return dispatch_prec(in->prec, [&](auto tag) {
        using S = decltype(tag);
        if (n->ch == 16) return launch_eo<16, S>(n, out, in, U, adjoint, skip);
        if (n->ch == 4) return launch_eo<4, S>(n, out, in, U, adjoint, skip);
        return launch_eo<8, S>(n, out, in, U, adjoint, skip);
    });
}
} // namespace qkx
