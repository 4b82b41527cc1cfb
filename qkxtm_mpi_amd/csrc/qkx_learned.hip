// qkx_learned.hip -- learned preconditioner: a gauge-equivariant
// parallel-transport convolution (PTC) network, its training kernels, and the
// flexible GCR solver that uses it as a right preconditioner.
//
// No reference counterpart.  The layer is the published PTC layer (C. Lehner
// and T. Wettig, Phys. Rev. D 108, 034503 (2023), arXiv:2302.05419) with
// paths of length 0 and 1:
//   out_a(x) = sum_p sum_b W[p][a][b] (T_p in_b)(x),   p = 0..8
//   T_0 = 1,  T_{1+2mu} f(x) = U_mu(x) f(x+mu),  T_{2+2mu} f(x) = U_mu(x-mu)^dag f(x-mu)
// The network is M = L2 L1 with 4 -> ch -> 4 colour-vector channels (a spinor
// is 4 channels, one per spin).  It is linear in its input, so it is a fixed
// linear operator once trained.
//
// Hidden-channel fields: component k = channel*3 + colour, two per float4 (see
// Hid), over the parity-blocked site index of the spinor/gauge layout; the
// 4-channel fields are spinors.  Weights are W[9][cout][cin] complex; the
// master copy is FP32, inference reads a BF16 copy (FP32 accumulation).
#include "qkx_net.h"
#include <chrono>
#include <cmath>
#include <vector>

namespace {

// Weights of a full-lattice layer CIN -> COUT as get(p, a, b): W[9][COUT][CIN],
// or (ADJ) the adjoint of the layer W[9][CIN][COUT], A[p][a][b] = conj(W[rev
// p][b][a]); FP32 or BF16 source.
template <int CIN, int COUT, bool ADJ, bool BF> struct LayerWeights {
    const void *w;
    __device__ __forceinline__ float2 operator()(int p, int a, int b) const
    {
        const int i = ADJ ? (rev_path(p) * CIN + b) * COUT + a : (p * COUT + a) * CIN + b;
        float2 v;
        if (BF) {
            const uint32_t h = ((const uint32_t *)w)[i];
            v = make_float2(bf2f(h & 0xffffu), bf2f(h >> 16));
        } else {
            v = ((const float2 *)w)[i];
        }
        if (ADJ) v.y = -v.y;
        return v;
    }
};

// The full-lattice layers run three wavefronts per 64 sites, each on three of
// the nine paths, whose sums the first one adds up through LDS: at the
// training lattice one wavefront per 64 sites would be two per SIMD, too few
// to cover the gathers.  16^3x32, CH = 16: 4 -> 16 takes 38 us (48 us with the
// mixing on the vector ALU), 16 -> 4 takes 48 us (76 us; 73 us with one
// wavefront per 64 sites).
constexpr int kLayerT = 192;
// this thread's site (clamped to the lattice) and whether it is its own; w its wavefront
__device__ __forceinline__ NetSite layer_site(const Geom &g, int nblk8, bool &own, int &w)
{
    w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int u = net_block(nblk8) * 64 + (int)(threadIdx.x & 63);
    own = u < g.V;
    const int s = min(u, g.V - 1);
    const int p = s >= g.Vh ? 1 : 0;
    return net_site(g, p, s - p * g.Vh);
}

// An FP64 field to be rounded into an FP32 one beside other work, or nothing
// (from.p null).
struct RoundOff {
    SpinorD from;
    SpinorF to;
};

// Full-lattice layer 4 -> CH (or the adjoint of a layer CH -> 4, which takes a
// RoundOff along in a wavefront that is done).
template <int CH, bool ADJ, bool BF, class S>
__global__ __launch_bounds__(kLayerT) QKX_NET_REGS void net_expand_kernel(S in, Hid out, GaugeF18 U, Geom g, int nblk8,
                                                                          LayerWeights<4, CH, ADJ, BF> wt, RoundOff ro)
{
    constexpr int H = CH / 4;
    __shared__ f4v part[2][H * 6][64];
    bool own;
    int w;
    const NetSite n = layer_site(g, nblk8, own, w);
    f4v re[H][3], im[H][3];
#pragma unroll
    for (int h = 0; h < H; h++) {
        zero3(re[h]);
        zero3(im[h]);
    }
    auto unit = [](int site) { return site; };
    const LinkGlobal ls{U, g, n};
    if (w == 0) expand<CH, 0, 3>(in, ls, n, unit, wt, re, im);
    else if (w == 1) expand<CH, 3, 6>(in, ls, n, unit, wt, re, im);
    else expand<CH, 6, 9>(in, ls, n, unit, wt, re, im);
    const int lane = threadIdx.x & 63;
    if (w > 0) {
#pragma unroll
        for (int h = 0; h < H; h++)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                part[w - 1][h * 6 + c][lane] = re[h][c];
                part[w - 1][h * 6 + 3 + c][lane] = im[h][c];
            }
    }
    __syncthreads();
    if constexpr (ADJ) {
        if (w == 1 && own && ro.from.p) {
            Cx<double> d[12];
            Cx<float> f[12];
            ro.from.load(n.s, d);
#pragma unroll
            for (int k = 0; k < 12; k++) f[k] = {(float)d[k].re, (float)d[k].im};
            ro.to.store(n.s, f);
        }
    }
    if (w > 0) return;
#pragma unroll
    for (int h = 0; h < H; h++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            re[h][c] += part[0][h * 6 + c][lane] + part[1][h * 6 + c][lane];
            im[h][c] += part[0][h * 6 + 3 + c][lane] + part[1][h * 6 + 3 + c][lane];
        }
    if (own) {
#pragma unroll
        for (int h = 0; h < H; h++) out.store(h, n.s, re[h], im[h]);
    }
}

// Full-lattice layer CH -> 4.  LOSS: the pair loss of the output o against
// the target e instead: out = 2 (o - e), per-workgroup |o - e|^2.
template <int CH, bool BF, bool LOSS, class S, class E>
__global__ __launch_bounds__(kLayerT) QKX_NET_REGS void net_contract_kernel(Hid in, S out, E e, GaugeF18 U, Geom g,
                                                                            int nblk8, LayerWeights<CH, 4, false, BF> wt,
                                                                            double *lpart)
{
    __shared__ float part[2][24][64];
    bool own;
    int w;
    const NetSite n = layer_site(g, nblk8, own, w);
    Cx<float> acc[12];
#pragma unroll
    for (int k = 0; k < 12; k++) acc[k] = {0.f, 0.f};
    auto unit = [](int site) { return site; };
    const LinkGlobal ls{U, g, n};
    if (w == 0) contract<CH, 0, 3>(in, ls, n, unit, wt, acc);
    else if (w == 1) contract<CH, 3, 6>(in, ls, n, unit, wt, acc);
    else contract<CH, 6, 9>(in, ls, n, unit, wt, acc);
    const int lane = threadIdx.x & 63;
    if (w > 0) {
#pragma unroll
        for (int k = 0; k < 12; k++) {
            part[w - 1][2 * k][lane] = acc[k].re;
            part[w - 1][2 * k + 1][lane] = acc[k].im;
        }
    }
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int k = 0; k < 12; k++) {
        acc[k].re += part[0][2 * k][lane] + part[1][2 * k][lane];
        acc[k].im += part[0][2 * k + 1][lane] + part[1][2 * k + 1][lane];
    }
    double d2 = 0;
    if (own) {
        if constexpr (LOSS) {
            Cx<typename E::Real> t[12];
            e.load(n.s, t);
#pragma unroll
            for (int k = 0; k < 12; k++) {
                const float dx = acc[k].re - (float)t[k].re, dy = acc[k].im - (float)t[k].im;
                acc[k] = {2.f * dx, 2.f * dy};
                d2 += (double)dx * dx + (double)dy * dy;
            }
        }
        Cx<typename S::Real> o[12];
#pragma unroll
        for (int k = 0; k < 12; k++) o[k] = {acc[k].re, acc[k].im};
        out.store(n.s, o);
    }
    if constexpr (LOSS) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) d2 += __shfl_xor(d2, off, 64);
        if (lane == 0) lpart[blockIdx.x] = d2;
    }
}

// ---------------------------------------------------------------------------
// Weight gradients of both layers in one form: for a CH-channel field f and a
// 4-channel field v,
//   Z[p][j][k] = sum_y sum_c f_k(y)_c conj((T_p v_j)(y)_c).
// Layer 1 (f = gh, v = r): dL/dW1[p][a][b] = Z[p][b][a].  Layer 2 (f = h, v =
// gout): a sum over all sites may be taken at the other end of the path, and
// T_p and T_rev(p) are adjoint, so dL/dW2[p][a][b] = conj(Z[rev p][a][b]).
//
// The sum over sites is a contraction on the matrix cores: v_mfma_f32_4x4x1
// adds the 4 x 4 outer product of four lanes' real numbers (rows: channels 4 h
// + i of f, columns: vectors i of T_p v, one site) to each of its 16 blocks'
// own sums.  Lane = site for the loads and transports, so that a load reads
// consecutive sites (16 cache accesses; with the four channels of a site on
// adjacent lanes every lane was an access of its own) and a link is fetched
// once per site; a 4 x 4 transposition within each quad of lanes (8 selects
// with a lane-permuted source per 4 registers) then turns four sites' numbers
// into four rounds of MFMA operands.  blockIdx.y is a group of NP paths; the
// sums stay in registers over the sites.  16^3x32, CH = 16: 70 us a layer
// (125 us on the vector ALU, where f and v were read once per path), bound by
// the gathers' latency at two wavefronts per SIMD; the whole gradient of a pair,
// tm included, 592 -> 306 us.
// Partials: part[(widx * 2 + re/im) * gridDim.x + blockIdx.x] with widx = (p *
// 4 + j) * CH + k, summed in a fixed order.
__device__ __forceinline__ float row_sum(float v)   // sum over lanes of equal l % 4 in 16 lanes
{
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, true));   // row_ror:4
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));   // row_ror:8
    return v;
}
// a[i] of lane j <-> a[j] of lane i within each quad of lanes
template <int CTRL> __device__ __forceinline__ void quad_swap(float &x, float &y, bool upper)
{
    const float px = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
    const float py = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(y), CTRL, 0xf, 0xf, true));
    x = upper ? py : x;
    y = upper ? y : px;
}
__device__ __forceinline__ void quad_transpose(float &a, float &b, float &c, float &d)
{
    const bool u1 = threadIdx.x & 1, u2 = threadIdx.x & 2;
    quad_swap<0xB1>(a, b, u1);   // lanes 1 0 3 2
    quad_swap<0xB1>(c, d, u1);
    quad_swap<0x4E>(a, c, u2);   // lanes 2 3 0 1
    quad_swap<0x4E>(b, d, u2);
}
// four colour vectors of the lane's site -> v[3 r + c]: the lane's vector (lane
// & 3) of the quad's site r; zero for lanes past the end
__device__ __forceinline__ void quad_vectors(Cx<float> v[12], bool live)
{
#pragma unroll
    for (int k = 0; k < 12; k++)
        if (!live) v[k] = {0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 3; c++) {
        quad_transpose(v[c].re, v[3 + c].re, v[6 + c].re, v[9 + c].re);
        quad_transpose(v[c].im, v[3 + c].im, v[6 + c].im, v[9 + c].im);
    }
}
// the operands of one path
struct GradOps {
    SpinorF::Raw psi;
    GaugeF18::Raw link;
};
template <int P>
__device__ __forceinline__ void wgrad_fetch(const SpinorF &v, const GaugeF18 &U, const Geom &g, const NetSite &n, GradOps &o)
{
    o.psi = v.template fetch<3>(path_site<P>(n));
    if constexpr (P > 0) o.link = LinkGlobal{U, g, n}.template fetch<P>();
}
// t = T_P v of the lane's site, as quad_vectors leaves it
template <int P>
__device__ __forceinline__ void wgrad_transport(const SpinorF &v, const GaugeF18 &U, const Geom &g, const NetSite &n,
                                                bool live, const GradOps &o, Cx<float> t[12])
{
    Cx<float> x[12];
    (void)unpack_spinor(v, o.psi, x);
    if constexpr (P == 0) {
#pragma unroll
        for (int k = 0; k < 12; k++) t[k] = x[k];
    } else {
        Cx<float> l[9];
        LinkGlobal{U, g, n}.template get<P, false>(o.link, 1.0f, l);
#pragma unroll
        for (int b = 0; b < 4; b++) transport<P>(l, x + 3 * b, t + 3 * b);
    }
    quad_vectors(t, live);
}
// no later load is issued before this point: the fetches stay one step ahead
__device__ __forceinline__ void wgrad_step() { asm volatile("" ::: "memory"); }
// z[q] += f conj(t[q]) over the quad's four sites, the NP sums interleaved so
// that no MFMA waits for the one before it
template <int NP>
__device__ __forceinline__ void wgrad_tiles(const Cx<float> f[12], const Cx<float> (*t)[12], f4v *zr, f4v *zi, int stride)
{
#pragma unroll
    for (int k = 0; k < 12; k++) {
#pragma unroll
        for (int q = 0; q < NP; q++) zr[q * stride] = __builtin_amdgcn_mfma_f32_4x4x1f32(f[k].re, t[q][k].re, zr[q * stride], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < NP; q++) zi[q * stride] = __builtin_amdgcn_mfma_f32_4x4x1f32(f[k].im, t[q][k].re, zi[q * stride], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < NP; q++) zr[q * stride] = __builtin_amdgcn_mfma_f32_4x4x1f32(f[k].im, t[q][k].im, zr[q * stride], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < NP; q++) zi[q * stride] = __builtin_amdgcn_mfma_f32_4x4x1f32(f[k].re, -t[q][k].im, zi[q * stride], 0, 0, 0);
    }
}
// one tile per path (CH = 4): f stays, the transports come one at a time
template <int P, int P1>
__device__ __forceinline__ void wgrad_each(const SpinorF &v, const GaugeF18 &U, const Geom &g, const NetSite &n, bool live,
                                           const GradOps &o, const Cx<float> f[12], f4v (*zr)[1], f4v (*zi)[1])
{
    GradOps next;
    if constexpr (P + 1 < P1) wgrad_fetch<P + 1>(v, U, g, n, next);
    Cx<float> t[1][12];
    wgrad_transport<P>(v, U, g, n, live, o, t[0]);
    wgrad_tiles<1>(f, t, zr[0], zi[0], 1);
    wgrad_step();
    if constexpr (P + 1 < P1) wgrad_each<P + 1, P1>(v, U, g, n, live, next, f, zr + 1, zi + 1);
}
// the transports of paths P .. P1 - 1, and f's first channels requested
template <int P, int P1>
__device__ __forceinline__ void wgrad_hold(const SpinorF &v, const GaugeF18 &U, const Geom &g, const NetSite &n, bool live,
                                           const GradOps &o, Cx<float> (*t)[12], const Hid &f, Hid::Raw &fr)
{
    GradOps next;
    if constexpr (P + 1 < P1) wgrad_fetch<P + 1>(v, U, g, n, next);
    else fr = f.fetch(0, n.s);
    wgrad_transport<P>(v, U, g, n, live, o, *t);
    wgrad_step();
    if constexpr (P + 1 < P1) wgrad_hold<P + 1, P1>(v, U, g, n, live, next, t + 1, f, fr);
}
// The sums of a workgroup's lanes are FP32 over kGradFlush rounds of its sites at
// most (192 products), then go to FP64 in LDS: without that their length, and
// with it their rounding, grows with the volume.  24^3x48, CH = 8 (16 rounds):
// 801 us without, 832, 822, 818 and 806 after every 1, 2, 4 and 8 rounds.
constexpr int kGradFlush = 8;
// LDS of a workgroup, one buffer for whichever path group it takes (a static one
// in wgrad_group would be there once per group: 78 KB for 17 at CH = 16, and two
// workgroups to a CU where the launch counts on eight of 64 threads): the FP64
// sums of the group's numbers, then a row of their FP32 sums per 16 lanes, padded
// so that the rows start on different banks.
extern __shared__ double wgrad_lds[];
constexpr int wgrad_numbers(int ch, int np) { return np * 4 * ch * 2; }
constexpr int wgrad_row(int numbers) { return numbers + 4; }
inline size_t wgrad_lds_bytes(int ch, int np, int bs)
{
    const int w = wgrad_numbers(ch, np);
    return w * sizeof(double) + (size_t)(bs / 16) * wgrad_row(w) * sizeof(float);
}
template <int CH, int P0, int NP>
__device__ __forceinline__ void wgrad_group(const Hid &f, const SpinorF &v, const GaugeF18 &U, const Geom &g, double *part)
{
    constexpr int H = CH / 4, W = wgrad_numbers(CH, NP);
    double *tot = wgrad_lds;   // each number by its own thread
    float *red = reinterpret_cast<float *>(tot + W);
    const int step = gridDim.x * blockDim.x;
    for (int w = threadIdx.x; w < W; w += blockDim.x) tot[w] = 0;
    // the same number of rounds in every wavefront of the workgroup
    for (int s0 = blockIdx.x * blockDim.x; s0 < g.V;) {
        f4v zr[NP][H], zi[NP][H];
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int h = 0; h < H; h++) zr[p][h] = zi[p][h] = f4v{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < kGradFlush && s0 < g.V; k++, s0 += step) {
            const int s1 = s0 + (int)threadIdx.x;
            const bool live = s1 < g.V;
            const int s = min(s1, g.V - 1);
            const int p = s >= g.Vh ? 1 : 0;
            const NetSite n = net_site(g, p, s - p * g.Vh);
            Cx<float> ff[12];
            GradOps o0;
            wgrad_fetch<P0>(v, U, g, n, o0);
            if constexpr (H == 1) {
                Hid::unpack(f.fetch(0, s), ff);
                quad_vectors(ff, live);
                wgrad_each<P0, P0 + NP>(v, U, g, n, live, o0, ff, zr, zi);
            } else {   // the transports stay, the channels come four at a time
                Cx<float> t[NP][12];
                Hid::Raw fr;
                wgrad_hold<P0, P0 + NP>(v, U, g, n, live, o0, t, f, fr);
#pragma unroll
                for (int h = 0; h < H; h++) {
                    Hid::unpack(fr, ff);
                    if (h + 1 < H) fr = f.fetch(h + 1, s);
                    quad_vectors(ff, live);
                    wgrad_tiles<NP>(ff, t, &zr[0][h], &zi[0][h], H);
                    wgrad_step();
                }
            }
        }
        // sums of 16 lanes' blocks in registers, of the workgroup's 16-lane rows in
        // FP64.  The lane is opaque here: the addresses formed from it would
        // otherwise be kept in registers over the rounds.
        int lane = threadIdx.x;
        asm volatile("" : "+v"(lane));
        const int i = lane & 3, row = lane >> 4, rows = blockDim.x >> 4;
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int h = 0; h < H; h++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    zr[p][h][k] = row_sum(zr[p][h][k]);
                    zi[p][h][k] = row_sum(zi[p][h][k]);
                }
        if ((lane & 12) == 0) {
            float *dst = red + row * wgrad_row(W);
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int h = 0; h < H; h++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const int w = (p * 4 + i) * CH + 4 * h + k;   // row k: channel of f, column i: vector of v
                        dst[2 * w] = zr[p][h][k];
                        dst[2 * w + 1] = zi[p][h][k];
                    }
        }
        __syncthreads();
        for (int w = lane; w < W; w += blockDim.x) {
            double t = tot[w];
#pragma unroll 4
            for (int q = 0; q < rows; q++) t += (double)red[q * wgrad_row(W) + w];
            tot[w] = t;
        }
        __syncthreads();   // red has been read
    }
    for (int w = threadIdx.x; w < W; w += blockDim.x) part[(size_t)(P0 * 4 * CH * 2 + w) * gridDim.x + blockIdx.x] = tot[w];
}
// paths per group: the sums take 2 CH registers per path, the transports held
// beside them 24; one more path per group spills (CH = 16: 83 us with three), and
// so does an FP64 v (134 registers at CH = 8), which is therefore rounded first
constexpr int wgrad_np(int ch) { return ch == 4 ? 9 : ch == 8 ? 3 : 2; }
constexpr int wgrad_groups(int ch) { return (9 + wgrad_np(ch) - 1) / wgrad_np(ch); }
template <int CH, int G>
__device__ __forceinline__ void wgrad_select(const Hid &f, const SpinorF &v, const GaugeF18 &U, const Geom &g, double *part)
{
    constexpr int P0 = G * wgrad_np(CH), NP = P0 + wgrad_np(CH) <= 9 ? wgrad_np(CH) : 9 - P0;
    if constexpr (G + 1 == wgrad_groups(CH)) wgrad_group<CH, P0, NP>(f, v, U, g, part);
    else if ((int)blockIdx.y == G) wgrad_group<CH, P0, NP>(f, v, U, g, part);
    else wgrad_select<CH, G + 1>(f, v, U, g, part);
}
template <int CH>
__global__ __launch_bounds__(kT) QKX_NET_REGS void net_wgrad_kernel(Hid f, SpinorF v, GaugeF18 U, Geom g, double *part)
{
    wgrad_select<CH, 0>(f, v, U, g, part);
}

// The gradient of both layers and the loss from their partials, one wavefront
// per number: workgroup w < nw is complex weight w of layer 1, then of layer
// 2, the last one the loss.
__global__ __launch_bounds__(64) void grad_finish_kernel(const double *z1, const double *z2, int nb, const double *lpart,
                                                         int nl, int ch, double2 *grad, double *loss)
{
    const int w = blockIdx.x, n1 = 9 * 4 * ch;
    auto sum = [&](const double *p, int n) {
        double t = 0;
        for (int i = threadIdx.x; i < n; i += 64) t += p[i];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
        return t;
    };
    if (w == 2 * n1) {
        const double t = sum(lpart, nl);
        if (threadIdx.x == 0) *loss += t;
        return;
    }
    const bool first = w < n1;
    const int i = first ? w : w - n1;
    // weight [p][a][b]: layer 1 [9][ch][4] takes Z[p][b][a], layer 2 [9][4][ch] conj(Z[rev p][a][b])
    const int p = i / (4 * ch), r = i % (4 * ch);
    const int zi = first ? (p * 4 + r % 4) * ch + r / 4 : (rev_path(p) * 4 + r / ch) * ch + r % ch;
    const double *z = first ? z1 : z2;
    const double re = sum(z + (size_t)(2 * zi) * nb, nb), im = sum(z + (size_t)(2 * zi + 1) * nb, nb);
    if (threadIdx.x == 0) {
        grad[w].x += re;
        grad[w].y += first ? im : -im;
    }
}

__global__ void adam_kernel(float2 *w, uint32_t *wb, double2 *grad, float2 *m, float2 *v, int n, float lr,
                            float b1, float b2, float eps, float c1, float c2, float scale)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gx = (float)grad[i].x * scale, gy = (float)grad[i].y * scale;
    float2 mm = m[i], vv = v[i], ww = w[i];
    mm.x = b1 * mm.x + (1.f - b1) * gx;
    mm.y = b1 * mm.y + (1.f - b1) * gy;
    vv.x = b2 * vv.x + (1.f - b2) * gx * gx;
    vv.y = b2 * vv.y + (1.f - b2) * gy * gy;
    ww.x -= lr * (mm.x / c1) / (sqrtf(vv.x / c2) + eps);
    ww.y -= lr * (mm.y / c1) / (sqrtf(vv.y / c2) + eps);
    m[i] = mm;
    v[i] = vv;
    w[i] = ww;
    wb[i] = f2bf(ww.x) | (f2bf(ww.y) << 16);
    grad[i] = make_double2(0.0, 0.0);
}

__global__ void to_bf16_kernel(const float2 *w, uint32_t *wb, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) wb[i] = f2bf(w[i].x) | (f2bf(w[i].y) << 16);
}

int layer_blocks(int V) { return (V + 63) / 64; }
// workgroups of a layer launch after XCD remapping: one loss partial each
int loss_blocks(int V)
{
    int nb = layer_blocks(V);
    (void)net_remap(nb);
    return nb;
}
// workgroup size and count of the weight gradient
// (of each path group): as many as are resident at two wavefronts per SIMD,
// all with the same number of rounds, so that the sums' way through LDS and
// memory is paid once per resident workgroup
constexpr int kGradBlocks = 512;
void grad_grid(int ch, int V, int &bs, int &nb)
{
    const int groups = wgrad_groups(ch);
    bs = V >= kGradBlocks / groups * kT ? kT : 64;
    const int most = kGradBlocks * (kT / bs) / groups, tiles = (V + bs - 1) / bs;
    const int rounds = (tiles + most - 1) / most;
    nb = (tiles + rounds - 1) / rounds;
}

int net_buffers(qkx_net_s *n, const int L[4])
{
    if (n->fh && n->L[0] == L[0] && n->L[1] == L[1] && n->L[2] == L[2] && n->L[3] == L[3]) return QKX_SUCCESS;
    // no lattice until every buffer is there: after a failed allocation the next
    // call starts over
    for (int d = 0; d < 4; d++) n->L[d] = 0;
    float4 **bufs[3] = {&n->fh, &n->gout, &n->gh};
    for (auto b : bufs) {
        if (*b) (void)hipFree(*b);
        *b = nullptr;
    }
    const size_t V = (size_t)L[0] * L[1] * L[2] * L[3];
    const int chans[3] = {n->ch, 4, n->ch};
    for (int i = 0; i < 3; i++) QKX_HIP(hipMalloc(bufs[i], sizeof(float2) * 3 * chans[i] * V));
    // partials: both layers' gradients, then the loss
    int bs, nb;
    grad_grid(n->ch, (int)V, bs, nb);
    const size_t need = (size_t)nb * 2 * 9 * 4 * n->ch * 2 + loss_blocks((int)V);
    if (need > n->part_cap) {
        if (n->part) (void)hipFree(n->part);
        n->part = nullptr;
        n->part_cap = 0;
        QKX_HIP(hipMalloc(&n->part, sizeof(double) * need));
        n->part_cap = need;
    }
    for (int d = 0; d < 4; d++) n->L[d] = L[d];
    return QKX_SUCCESS;
}

int check_spinor(const qkx_spinor_s *f, const qkx_gauge_s *U)
{
    if (f->subset != QKX_SUBSET_FULL || f->nrhs != 1 || (f->prec != QKX_PREC_DOUBLE && f->prec != QKX_PREC_SINGLE) ||
        f->L[0] != U->L[0] || f->L[1] != U->L[1] || f->L[2] != U->L[2] || f->L[3] != U->L[3]) {
        qkx::set_error("net: fields must be single full-lattice FP64/FP32 spinors on the gauge's lattice");
        return QKX_ERR_ARG;
    }
    return QKX_SUCCESS;
}

// fn(accessor) for a full-lattice FP64 or FP32 spinor (check_spinor passed)
template <class F> int with_spinor(const qkx_spinor_s *f, F fn)
{
    if (f->prec == QKX_PREC_DOUBLE) return fn(make_spinor<SpinorD>(f));
    return fn(make_spinor<SpinorF>(f));
}
template <class F> int with_bf(const qkx_net_s *n, F fn)
{
    if (n->bf16) return fn(std::true_type{});
    return fn(std::false_type{});
}
Hid hid_of(float4 *p, int V) { return Hid{p, (size_t)V}; }

// layer 1 of a spinor, or (ADJ) the adjoint of layer 2, into a hidden field
template <bool ADJ>
int launch_expand(qkx_net_s *n, const qkx_spinor_s *in, const SpinorF *inf, Hid out, const qkx_gauge_s *U,
                  const RoundOff &ro = RoundOff{})
{
    const Geom g = qkx::make_geom(U->L, U->bc);
    const GaugeF18 G = make_gauge<GaugeF18>(U);
    int nb = layer_blocks(g.V);
    const int nblk8 = net_remap(nb);
    const int off = ADJ ? n->n1 : 0;
    return with_ch(n, [&](auto CHC) {
        constexpr int CH = decltype(CHC)::value;
        return with_bf(n, [&](auto BFC) {
            constexpr bool BF = decltype(BFC)::value;
            const LayerWeights<4, CH, ADJ, BF> w{BF ? (const void *)(n->wb + off) : (const void *)(n->w + off)};
            auto go = [&](auto S) {
                hipLaunchKernelGGL((net_expand_kernel<CH, ADJ, BF, decltype(S)>), dim3(nb), dim3(kLayerT), 0,
                                   qkx::g_stream, S, out, G, g, nblk8, w, ro);
                QKX_HIP(hipGetLastError());
                return QKX_SUCCESS;
            };
            if constexpr (ADJ) return go(*inf);
            else return with_spinor(in, go);
        });
    });
}

// layer 2 into a spinor, or (e given) the loss gradient 2 (o - e) into gout
// and per-workgroup losses into lpart
int launch_contract(qkx_net_s *n, qkx_spinor_s *out, const qkx_spinor_s *e, const qkx_gauge_s *U, double *lpart)
{
    const Geom g = qkx::make_geom(U->L, U->bc);
    const GaugeF18 G = make_gauge<GaugeF18>(U);
    int nb = layer_blocks(g.V);
    const int nblk8 = net_remap(nb);
    const Hid hid = hid_of(n->fh, g.V);
    return with_ch(n, [&](auto CHC) {
        constexpr int CH = decltype(CHC)::value;
        return with_bf(n, [&](auto BFC) {
            constexpr bool BF = decltype(BFC)::value;
            const LayerWeights<CH, 4, false, BF> w{BF ? (const void *)(n->wb + n->n1) : (const void *)(n->w + n->n1)};
            if (e)
                return with_spinor(e, [&](auto E) {
                    hipLaunchKernelGGL((net_contract_kernel<CH, BF, true, SpinorF, decltype(E)>), dim3(nb),
                                       dim3(kLayerT), 0, qkx::g_stream, hid, SpinorF{n->gout, g.V}, E, G, g, nblk8,
                                       w, lpart);
                    QKX_HIP(hipGetLastError());
                    return QKX_SUCCESS;
                });
            return with_spinor(out, [&](auto S) {
                hipLaunchKernelGGL((net_contract_kernel<CH, BF, false, decltype(S), decltype(S)>), dim3(nb),
                                   dim3(kLayerT), 0, qkx::g_stream, hid, S, S, G, g, nblk8, w, (double *)nullptr);
                QKX_HIP(hipGetLastError());
                return QKX_SUCCESS;
            });
        });
    });
}

// Z of a hidden field f and a spinor v
int launch_wgrad(qkx_net_s *n, Hid f, SpinorF v, const qkx_gauge_s *U, double *part, int bs, int nb)
{
    const Geom g = qkx::make_geom(U->L, U->bc);
    const GaugeF18 G = make_gauge<GaugeF18>(U);
    return with_ch(n, [&](auto CHC) {
        constexpr int CH = decltype(CHC)::value;
        hipLaunchKernelGGL(net_wgrad_kernel<CH>, dim3(nb, wgrad_groups(CH)), dim3(bs),
                           wgrad_lds_bytes(CH, wgrad_np(CH), bs), qkx::g_stream, f, v, G, g, part);
        QKX_HIP(hipGetLastError());
        return QKX_SUCCESS;
    });
}

} // namespace

namespace qkx {
// M in -> out (FP64 or FP32 full spinors); used by the flexible solver
int net_apply(qkx_net_s *n, qkx_spinor_s *out, const qkx_spinor_s *in, const qkx_gauge_s *U)
{
    int rc;
    if ((rc = check_net_gauge(U)) || (rc = check_spinor(in, U)) || (rc = check_spinor(out, U))) return rc;
    if ((rc = net_buffers(n, U->L))) return rc;
    if ((rc = launch_expand<false>(n, in, nullptr, hid_of(n->fh, U->V), U))) return rc;
    return launch_contract(n, out, nullptr, U, nullptr);
}
} // namespace qkx

extern "C" {

int qkx_net_create(qkx_net **out, int ch)
{
    QKX_CHECK_ARG(out && (ch == 4 || ch == 8 || ch == 16), "qkx_net_create: hidden channels must be 4, 8 or 16");
    if (int rc = qkx::ensure_init()) return rc;
    qkx_net_s *n = new qkx_net_s{};
    n->ch = ch;
    n->n1 = 9 * ch * 4;
    n->n2 = 9 * 4 * ch;
    n->bf16 = 1;
    const int nt = n->n1 + n->n2;
    bool ok = hipMalloc(&n->w, sizeof(float2) * nt) == hipSuccess &&
              hipMalloc(&n->wb, sizeof(uint32_t) * nt) == hipSuccess &&
              hipMalloc(&n->grad, sizeof(double2) * nt) == hipSuccess &&
              hipMalloc(&n->m, sizeof(float2) * nt) == hipSuccess &&
              hipMalloc(&n->v, sizeof(float2) * nt) == hipSuccess &&
              hipMalloc(&n->loss, sizeof(double)) == hipSuccess;
    if (!ok) {
        qkx_net_destroy(n);
        qkx::set_error("qkx_net_create: device allocation failed");
        return QKX_ERR_NOMEM;
    }
    QKX_HIP(hipMemsetAsync(n->w, 0, sizeof(float2) * nt, qkx::g_stream));
    QKX_HIP(hipMemsetAsync(n->wb, 0, sizeof(uint32_t) * nt, qkx::g_stream));
    QKX_HIP(hipMemsetAsync(n->grad, 0, sizeof(double2) * nt, qkx::g_stream));
    QKX_HIP(hipMemsetAsync(n->m, 0, sizeof(float2) * nt, qkx::g_stream));
    QKX_HIP(hipMemsetAsync(n->v, 0, sizeof(float2) * nt, qkx::g_stream));
    QKX_HIP(hipMemsetAsync(n->loss, 0, sizeof(double), qkx::g_stream));
    QKX_HIP(hipStreamSynchronize(qkx::g_stream));
    *out = n;
    return QKX_SUCCESS;
}

int qkx_net_destroy(qkx_net *n)
{
    if (!n) return QKX_SUCCESS;
    void *ptrs[] = {n->w,  n->wb,   n->grad, n->m,    n->v,   n->loss,
                    n->fh, n->gout, n->gh,   n->part, n->weo, n->ehid};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    delete n;
    return QKX_SUCCESS;
}

int qkx_net_release_buffers(qkx_net *n)
{
    QKX_CHECK_ARG(n, "qkx_net_release_buffers: null argument");
    QKX_HIP(hipStreamSynchronize(qkx::g_stream));   // no launch may still use them
    float4 **bufs[4] = {&n->fh, &n->gout, &n->gh, &n->ehid};
    for (auto b : bufs) {
        if (*b) (void)hipFree(*b);
        *b = nullptr;
    }
    n->ehid_cap = 0;
    n->L[0] = n->L[1] = n->L[2] = n->L[3] = 0;
    return QKX_SUCCESS;
}

int qkx_net_set_hidden_limit(qkx_net *n, unsigned long long bytes)
{
    QKX_CHECK_ARG(n, "qkx_net_set_hidden_limit: null argument");
    n->ehid_limit = (size_t)(bytes / sizeof(float2));
    return QKX_SUCCESS;
}

int qkx_net_nweights(const qkx_net *n, int *ncomplex)
{
    QKX_CHECK_ARG(n && ncomplex, "qkx_net_nweights: null argument");
    *ncomplex = n->n1 + n->n2;
    return QKX_SUCCESS;
}

int qkx_net_set_weights(qkx_net *n, const float *w)
{
    QKX_CHECK_ARG(n && w, "qkx_net_set_weights: null argument");
    const int nt = n->n1 + n->n2;
    QKX_HIP(hipMemcpyAsync(n->w, w, sizeof(float2) * nt, hipMemcpyHostToDevice, qkx::g_stream));
    hipLaunchKernelGGL(to_bf16_kernel, dim3((nt + 255) / 256), dim3(256), 0, qkx::g_stream, n->w, n->wb, nt);
    QKX_HIP(hipGetLastError());
    // a new parameter vector restarts the optimiser
    QKX_HIP(hipMemsetAsync(n->m, 0, sizeof(float2) * nt, qkx::g_stream));
    QKX_HIP(hipMemsetAsync(n->v, 0, sizeof(float2) * nt, qkx::g_stream));
    n->step = 0;
    QKX_HIP(hipStreamSynchronize(qkx::g_stream));
    return QKX_SUCCESS;
}

int qkx_net_get_weights(const qkx_net *n, float *w)
{
    QKX_CHECK_ARG(n && w, "qkx_net_get_weights: null argument");
    QKX_HIP(hipMemcpyAsync(w, n->w, sizeof(float2) * (n->n1 + n->n2), hipMemcpyDeviceToHost, qkx::g_stream));
    QKX_HIP(hipStreamSynchronize(qkx::g_stream));
    return QKX_SUCCESS;
}

int qkx_net_set_bf16(qkx_net *n, int on)
{
    QKX_CHECK_ARG(n, "qkx_net_set_bf16: null argument");
    n->bf16 = on ? 1 : 0;
    return QKX_SUCCESS;
}

int qkx_net_apply(qkx_net *n, qkx_spinor *out, const qkx_spinor *in, const qkx_gauge *U)
{
    QKX_CHECK_ARG(n && out && in && U, "qkx_net_apply: null argument");
    QKX_CHECK_ARG(out != in, "qkx_net_apply: out must differ from in");
    return qkx::net_apply(n, out, in, U);
}

int qkx_net_apply_eo(qkx_net *n, qkx_spinor *out, const qkx_spinor *in, const qkx_gauge *U, int adjoint)
{
    QKX_CHECK_ARG(n && out && in && U, "qkx_net_apply_eo: null argument");
    int rc = qkx::net_prep_eo(n);
    if (rc) return rc;
    return qkx::net_apply_eo(n, out, in, U, adjoint ? 1 : 0, nullptr);
}

int qkx_net_accumulate_grad(qkx_net *n, const qkx_spinor *r, const qkx_spinor *e, const qkx_gauge *U)
{
    QKX_CHECK_ARG(n && r && e && U, "qkx_net_accumulate_grad: null argument");
    int rc;
    if ((rc = check_net_gauge(U)) || (rc = check_spinor(r, U)) || (rc = check_spinor(e, U))) return rc;
    if ((rc = net_buffers(n, U->L))) return rc;
    const int V = U->V;
    int bs, nb;
    grad_grid(n->ch, V, bs, nb);
    const size_t nz = (size_t)nb * 9 * 4 * n->ch * 2;
    double *z1 = n->part, *z2 = z1 + nz, *lpart = z2 + nz;
    const Hid fh = hid_of(n->fh, V), gh = hid_of(n->gh, V);
    const SpinorF gout{n->gout, V};
    if ((rc = launch_expand<false>(n, r, nullptr, fh, U))) return rc;
    if ((rc = launch_contract(n, nullptr, e, U, lpart))) return rc;
    if ((rc = launch_wgrad(n, fh, gout, U, z2, bs, nb))) return rc;
    // layer 1's gradient gathers r nine times: an FP64 one is rounded once, into
    // the hidden channels of the forward pass, which nothing reads any more
    const SpinorF rf{n->fh, V};
    const bool r64 = r->prec == QKX_PREC_DOUBLE;
    const RoundOff ro{r64 ? make_spinor<SpinorD>(r) : SpinorD{}, rf};
    if ((rc = launch_expand<true>(n, nullptr, &gout, gh, U, ro))) return rc;
    if ((rc = launch_wgrad(n, gh, r64 ? rf : make_spinor<SpinorF>(r), U, z1, bs, nb))) return rc;
    hipLaunchKernelGGL(grad_finish_kernel, dim3(2 * 9 * 4 * n->ch + 1), dim3(64), 0, qkx::g_stream, z1, z2, nb, lpart,
                       loss_blocks(V), n->ch, n->grad, n->loss);
    QKX_HIP(hipGetLastError());
    return QKX_SUCCESS;
}

int qkx_net_read_grad(qkx_net *n, float *g, double *loss)
{
    QKX_CHECK_ARG(n, "qkx_net_read_grad: null argument");
    const int nt = n->n1 + n->n2;
    std::vector<double2> h(nt);
    QKX_HIP(hipMemcpyAsync(h.data(), n->grad, sizeof(double2) * nt, hipMemcpyDeviceToHost, qkx::g_stream));
    if (loss) QKX_HIP(hipMemcpyAsync(loss, n->loss, sizeof(double), hipMemcpyDeviceToHost, qkx::g_stream));
    QKX_HIP(hipStreamSynchronize(qkx::g_stream));
    if (g)
        for (int i = 0; i < nt; i++) {
            g[2 * i] = (float)h[i].x;
            g[2 * i + 1] = (float)h[i].y;
        }
    return QKX_SUCCESS;
}

int qkx_net_zero_grad(qkx_net *n)
{
    QKX_CHECK_ARG(n, "qkx_net_zero_grad: null argument");
    QKX_HIP(hipMemsetAsync(n->grad, 0, sizeof(double2) * (n->n1 + n->n2), qkx::g_stream));
    QKX_HIP(hipMemsetAsync(n->loss, 0, sizeof(double), qkx::g_stream));
    return QKX_SUCCESS;
}

int qkx_net_adam(qkx_net *n, double lr, double beta1, double beta2, double eps, int count)
{
    QKX_CHECK_ARG(n && count > 0 && lr > 0, "qkx_net_adam: bad argument");
    n->step++;
    const float c1 = (float)(1.0 - std::pow(beta1, n->step)), c2 = (float)(1.0 - std::pow(beta2, n->step));
    const int nt = n->n1 + n->n2;
    hipLaunchKernelGGL(adam_kernel, dim3((nt + 255) / 256), dim3(256), 0, qkx::g_stream, n->w, n->wb, n->grad, n->m,
                       n->v, nt, (float)lr, (float)beta1, (float)beta2, (float)eps, c1, c2, 1.0f / (float)count);
    QKX_HIP(hipGetLastError());
    return QKX_SUCCESS;
}

} // extern "C"
