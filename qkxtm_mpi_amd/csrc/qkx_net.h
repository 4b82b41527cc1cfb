// qkx_net.h -- what the full-lattice (qkx_learned.hip) and the even-odd
// (qkx_net_eo.hip) kernels of the learned preconditioner share: the network's
// state, channel mixing on the matrix cores, transports and the two layer
// forms.
#pragma once
#include "qkx_internal.h"
#include "qkx_core.h"
#include <algorithm>
#include <type_traits>

struct qkx_net_s {
    int ch;
    int n1, n2;            // complex weights of layer 1 ([9][ch][4]) and layer 2 ([9][4][ch])
    float2 *w;             // FP32 master weights, W1 then W2
    uint32_t *wb;          // BF16 copies (re in the low half, im in the high half)
    double2 *grad;         // accumulated gradient (dL/dRe + i dL/dIm)
    float2 *m, *v;         // Adam moments
    double *loss;          // accumulated loss
    int step;              // Adam steps taken
    int bf16;              // inference/training forward reads the BF16 copy
    int L[4];              // lattice of the work buffers
    float4 *fh, *gout, *gh;   // work buffers: hidden channels, loss gradient (FP32 spinor), its hidden channels
    double *part;             // per-workgroup gradients and losses
    size_t part_cap;
    float2 *weo;           // even-odd weight tables (forward, then adjoint), see eo_weights_kernel
    float4 *ehid;          // even-odd hidden channels on the odd sites, [3 ch / 2][Vh][nrhs]
    size_t ehid_cap;       // float2 entries of ehid
    size_t ehid_limit;     // bound on ehid (float2 entries); 0: kEoHiddenCap
};

namespace {

constexpr int kT = 256;

__device__ __forceinline__ uint32_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);   // round to nearest even
    return u >> 16;
}
__device__ __forceinline__ float bf2f(uint32_t h) { return __uint_as_float(h << 16); }

__host__ __device__ constexpr int rev_path(int p) { return p == 0 ? 0 : (((p - 1) & 1) == 0 ? p + 1 : p - 1); }

// ---------------------------------------------------------------------------
// Channel mixing on the matrix cores.  v_mfma_f32_4x4x1 works on 16 blocks of
// 4 lanes: lane l supplies one element B[col l % 4] of its block and receives
// the four rows D[0..3][col l % 4].  With CBSZ = 4 every block uses the A
// column (4 rows) that block ABID of the A register holds, so one register
// holds 16 columns of weights for the whole wavefront, and
//   D[a] += A_k[a] B
// adds weight column k times the lane's own real number to the lane's own
// four sums: four FP32 multiply-adds per lane and instruction, at twice the
// vector ALU's rate, on data that stays in the lane.  The arithmetic is FP32
// throughout.  A 4 x 4 complex tile takes 12 columns: Re W, Im W and -Im W
// of each input channel.
//
// MFMA ignores the execution mask, so every lane of a wavefront stays active:
// lanes past the end work on the last unit and do not store.
//
// Two wavefronts per SIMD at least: with at most 256 registers per lane the
// compiler keeps the sums in ordinary registers, where the vector ALU reads
// them without moves from the accumulation registers.
#define QKX_NET_REGS __attribute__((amdgpu_waves_per_eu(2, 8)))
typedef float f4v __attribute__((ext_vector_type(4)));
template <int J> __device__ __forceinline__ f4v mfma_bcast(float a, float b, f4v c)
{
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, J, 0);
}
// the A register of a 4 x 4 complex tile: lane 4 j + i holds row i of column
// j = 3 b + {0: Re, 1: Im, 2: -Im}; get(i, b) is the weight as float2
template <class Get> __device__ __forceinline__ float mix_weights(Get get)
{
    const int l = threadIdx.x & 63, j = l >> 2, b = min(j / 3, 3), part = j % 3;
    const float2 w = get(l & 3, b);
    return part == 0 ? w.x : part == 1 ? w.y : -w.y;
}
// re[c][a] + i im[c][a] += sum_b W[a][b] v[b * 3 + c]
template <int B> __device__ __forceinline__ void mix_column(float w, const Cx<float> v[12], f4v re[3], f4v im[3])
{
#pragma unroll
    for (int c = 0; c < 3; c++) {
        re[c] = mfma_bcast<3 * B>(w, v[B * 3 + c].re, re[c]);
        im[c] = mfma_bcast<3 * B>(w, v[B * 3 + c].im, im[c]);
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
        re[c] = mfma_bcast<3 * B + 2>(w, v[B * 3 + c].im, re[c]);
        im[c] = mfma_bcast<3 * B + 1>(w, v[B * 3 + c].re, im[c]);
    }
}
__device__ __forceinline__ void mix_tile(float w, const Cx<float> v[12], f4v re[3], f4v im[3])
{
    mix_column<0>(w, v, re, im);
    mix_column<1>(w, v, re, im);
    mix_column<2>(w, v, re, im);
    mix_column<3>(w, v, re, im);
}
__device__ __forceinline__ void zero3(f4v a[3])
{
#pragma unroll
    for (int c = 0; c < 3; c++) a[c] = f4v{0.f, 0.f, 0.f, 0.f};
}
// the sums written so far are final before any later load is issued: keeps
// the gathers of later paths from piling up in registers
__device__ __forceinline__ void pin3(f4v re[3], f4v im[3])
{
    asm volatile("" : "+v"(re[0]), "+v"(re[1]), "+v"(re[2]), "+v"(im[0]), "+v"(im[1]), "+v"(im[2])::"memory");
}

// o += T_P v for one colour vector (P = 0: the identity), l the link of the
// path: U_mu(x) for a forward path (odd P), U_mu(x - mu) for a backward one
template <int P> __device__ __forceinline__ void transport_add(const Cx<float> l[9], const Cx<float> v[3], Cx<float> o[3])
{
#pragma unroll
    for (int r = 0; r < 3; r++) {
        if constexpr (P == 0) {
            o[r] = o[r] + v[r];
        } else {
#pragma unroll
            for (int c = 0; c < 3; c++) o[r] = (P & 1) ? cmac(o[r], l[r * 3 + c], v[c]) : cjmac(o[r], l[c * 3 + r], v[c]);
        }
    }
}
// o = T_P v
template <int P> __device__ __forceinline__ void transport(const Cx<float> l[9], const Cx<float> v[3], Cx<float> o[3])
{
#pragma unroll
    for (int r = 0; r < 3; r++) {
        if constexpr (P == 0) {
            o[r] = v[r];
        } else {
            o[r] = (P & 1) ? cmul_f(l[r * 3], v[0]) : cjmul_f(l[r], v[0]);
#pragma unroll
            for (int c = 1; c < 3; c++) o[r] = (P & 1) ? cmac(o[r], l[r * 3 + c], v[c]) : cjmac(o[r], l[c * 3 + r], v[c]);
        }
    }
}

// Geometry of one site (parity p, checkerboard index cb): blocked index of
// its neighbour along path P, the link of the path, its boundary sign.
struct NetSite {
    HopSite h;
    int s;      // blocked index of the site
    int qoff;   // blocked offset of the other parity
};
__device__ __forceinline__ NetSite net_site(const Geom &g, int p, int cb)
{
    return NetSite{hop_site(g, p, cb), p * g.Vh + cb, (1 - p) * g.Vh};
}
// the v-th site of parity p in the walk tr, and its checkerboard index
__device__ __forceinline__ NetSite net_site_walk(const Geom &g, const HopTrav &tr, int p, int v, int &cb)
{
    const HopSite h = hop_site_walk(g, tr, p, v, cb);
    return NetSite{h, p * g.Vh + cb, (1 - p) * g.Vh};
}
template <int P> __device__ __forceinline__ int path_site(const NetSite &n)
{
    if constexpr (P == 0) return n.s;
    else return n.qoff + n.h.nb[P - 1];
}
// Where a thread's links come from.  Each source gives l = f times the link of
// path P, boundary sign included; SCALE false: f is 1.
// Global memory: fetched one path ahead of its use.
struct LinkGlobal {
    const GaugeF18 &U;
    const Geom &g;
    const NetSite &n;
    using Raw = GaugeF18::Raw;
    template <int P> __device__ __forceinline__ Raw fetch() const
    {
        return U.fetch((P - 1) >> 1, (P & 1) ? n.s : path_site<P>(n));
    }
    template <int P, bool SCALE> __device__ __forceinline__ void get(const Raw &r, float f, Cx<float> l[9]) const
    {
        U.unpack(r, l);
        if constexpr (P >= 7) f *= (P == 7 ? n.h.tw_p : n.h.tw_m) ? (float)g.bc : 1.0f;
        if constexpr (SCALE || P >= 7) {
#pragma unroll
            for (int k = 0; k < 9; k++) l[k] = {f * l[k].re, f * l[k].im};
        }
    }
};
// LDS, where the workgroup put the 8 links of each of its sites (kLinkStride
// floats per link, kSiteStride per site: rows stay 16-byte aligned, and the
// sites of a wavefront fall on different banks).
constexpr int kLinkStride = 20, kSiteStride = 8 * kLinkStride + 4;
struct LinkShared {
    const float *row;   // the thread's site
    struct Raw {};
    template <int P> __device__ __forceinline__ Raw fetch() const { return Raw{}; }
    template <int P, bool SCALE> __device__ __forceinline__ void get(const Raw &, float f, Cx<float> l[9]) const
    {
        const float *q = row + (P - 1) * kLinkStride;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float4 t = *reinterpret_cast<const float4 *>(q + 4 * k);
            l[2 * k] = {t.x, t.y};
            l[2 * k + 1] = {t.z, t.w};
        }
        const float2 t = *reinterpret_cast<const float2 *>(q + 16);
        l[8] = {t.x, t.y};
        if constexpr (SCALE) {
#pragma unroll
            for (int k = 0; k < 9; k++) l[k] = {f * l[k].re, f * l[k].im};
        }
    }
};

// The four colour vectors of a stored spinor.  FP16 storage: without the site
// scale, which joins the link of the path (or the path-0 weights' input).
template <class S> __device__ __forceinline__ float unpack_spinor(const S &in, const typename S::Raw &r, Cx<float> v[12])
{
    if constexpr (std::is_same_v<S, SpinorH>) {
        in.template unpack_raw<3>(r, v);
        return in.scale(r);
    } else {
        Cx<typename S::Real> t[12];
        in.template unpack<3>(r, t);
#pragma unroll
        for (int k = 0; k < 12; k++) v[k] = {(float)t[k].re, (float)t[k].im};
        return 1.0f;
    }
}

// Hidden-channel fields: two complex numbers per float4, element (k, u) with
// k = channel * 3 + colour in half k & 1 of base[(k >> 1) * stride + u].
struct Hid {
    float4 *p;
    size_t stride;
    // channels 4 h .. 4 h + 3 of unit u
    struct Raw {
        float4 c[6];
    };
    __device__ __forceinline__ Raw fetch(int h, int u) const
    {
        Raw r;
#pragma unroll
        for (int j = 0; j < 6; j++) r.c[j] = p[(size_t)(6 * h + j) * stride + u];
        return r;
    }
    static __device__ __forceinline__ void unpack(const Raw &r, Cx<float> v[12])
    {
#pragma unroll
        for (int j = 0; j < 6; j++) {
            v[2 * j] = {r.c[j].x, r.c[j].y};
            v[2 * j + 1] = {r.c[j].z, r.c[j].w};
        }
    }
    __device__ __forceinline__ void store(int h, int u, const f4v re[3], const f4v im[3]) const
    {
#pragma unroll
        for (int j = 0; j < 6; j++) {
            const int k0 = 2 * j, k1 = 2 * j + 1;   // channel k / 3, colour k % 3
            p[(size_t)(6 * h + j) * stride + u] = make_float4(re[k0 % 3][k0 / 3], im[k0 % 3][k0 / 3],
                                                              re[k1 % 3][k1 / 3], im[k1 % 3][k1 / 3]);
        }
    }
};

// One layer 4 -> CH for one unit: adds the paths P .. P1 - 1 of the mixed
// transports of the four input vectors.  unit(s) is the input field's entry of
// blocked site s; get(p, a, b) is a weight.  The operands of the next path are
// in flight while one is computed.
template <int CH, class S, class LS> struct ExpandOps {
    typename S::Raw psi;
    typename LS::Raw link;
    float w[CH / 4];
};
template <int CH, int P, class S, class LS, class Unit, class Get>
__device__ __forceinline__ ExpandOps<CH, S, LS> expand_fetch(const S &in, const LS &ls, const NetSite &n, Unit unit,
                                                             Get get)
{
    ExpandOps<CH, S, LS> o;
    o.psi = in.template fetch<3>(unit(path_site<P>(n)));
    if constexpr (P > 0) o.link = ls.template fetch<P>();
#pragma unroll
    for (int h = 0; h < CH / 4; h++) o.w[h] = mix_weights([&](int a, int b) { return get(P, 4 * h + a, b); });
    return o;
}
template <int CH, int P, int P1, class S, class LS, class Unit, class Get>
__device__ __forceinline__ void expand_paths(const S &in, const LS &ls, const NetSite &n, Unit unit, Get get,
                                             const ExpandOps<CH, S, LS> &o, f4v re[CH / 4][3], f4v im[CH / 4][3])
{
    auto apply = [&] {
        Cx<float> v[12], t[12];
        const float f = unpack_spinor(in, o.psi, v);
        if constexpr (P == 0) {
#pragma unroll
            for (int k = 0; k < 12; k++) t[k] = {f * v[k].re, f * v[k].im};
        } else {
            Cx<float> l[9];
            ls.template get<P, std::is_same_v<S, SpinorH>>(o.link, f, l);
#pragma unroll
            for (int b = 0; b < 4; b++) transport<P>(l, v + 3 * b, t + 3 * b);
        }
#pragma unroll
        for (int h = 0; h < CH / 4; h++) mix_tile(o.w[h], t, re[h], im[h]);
    };
    if constexpr (P + 1 < P1) {
        const auto next = expand_fetch<CH, P + 1>(in, ls, n, unit, get);
        apply();
#pragma unroll
        for (int h = 0; h < CH / 4; h++) pin3(re[h], im[h]);
        expand_paths<CH, P + 1, P1>(in, ls, n, unit, get, next, re, im);
    } else {
        apply();
    }
}
template <int CH, int P, int P1, class S, class LS, class Unit, class Get>
__device__ __forceinline__ void expand(const S &in, const LS &ls, const NetSite &n, Unit unit, Get get,
                                       f4v re[CH / 4][3], f4v im[CH / 4][3])
{
    expand_paths<CH, P, P1>(in, ls, n, unit, get, expand_fetch<CH, P>(in, ls, n, unit, get), re, im);
}

// One layer CH -> 4 for one unit: the channels are mixed at the neighbour,
// then the four colour vectors transported; acc[a * 3 + c] += the paths P ..
// P1 - 1.  hunit(s) is the hidden field's entry of blocked site s.  A step is
// one path and four channels.
template <class LS> struct ContractOps {
    Hid::Raw hid;
    typename LS::Raw link;
    float w;
};
template <int CH, int P, int H, class LS, class HUnit, class Get>
__device__ __forceinline__ ContractOps<LS> contract_fetch(const Hid &hid, const LS &ls, const NetSite &n, HUnit hunit,
                                                          Get get)
{
    ContractOps<LS> o;
    o.hid = hid.fetch(H, hunit(path_site<P>(n)));
    if constexpr (P > 0 && H == CH / 4 - 1) o.link = ls.template fetch<P>();
    o.w = mix_weights([&](int a, int b) { return get(P, a, 4 * H + b); });
    return o;
}
template <int CH, int P, int H, int P1, class LS, class HUnit, class Get>
__device__ __forceinline__ void contract_paths(const Hid &hid, const LS &ls, const NetSite &n, HUnit hunit, Get get,
                                               const ContractOps<LS> &o, f4v re[3], f4v im[3], Cx<float> acc[12])
{
    constexpr bool last = H == CH / 4 - 1;
    constexpr int PN = last ? P + 1 : P, HN = last ? 0 : H + 1;
    auto apply = [&] {
        if constexpr (H == 0) {
            zero3(re);
            zero3(im);
        }
        Cx<float> v[12];
        Hid::unpack(o.hid, v);
        mix_tile(o.w, v, re, im);
        if constexpr (last) {
            Cx<float> l[9];
            if constexpr (P > 0) ls.template get<P, false>(o.link, 1.0f, l);
#pragma unroll
            for (int a = 0; a < 4; a++) {
                const Cx<float> m[3] = {{re[0][a], im[0][a]}, {re[1][a], im[1][a]}, {re[2][a], im[2][a]}};
                transport_add<P>(l, m, acc + 3 * a);
            }
        }
    };
    if constexpr (PN < P1) {
        const auto next = contract_fetch<CH, PN, HN>(hid, ls, n, hunit, get);
        apply();
        if constexpr (last) {
#pragma unroll
            for (int k = 0; k < 12; k += 4)
                asm volatile("" : "+v"(acc[k].re), "+v"(acc[k].im), "+v"(acc[k + 1].re), "+v"(acc[k + 1].im),
                                  "+v"(acc[k + 2].re), "+v"(acc[k + 2].im), "+v"(acc[k + 3].re), "+v"(acc[k + 3].im)::"memory");
        } else {
            pin3(re, im);
        }
        contract_paths<CH, PN, HN, P1>(hid, ls, n, hunit, get, next, re, im, acc);
    } else {
        apply();
    }
}
template <int CH, int P, int P1, class LS, class HUnit, class Get>
__device__ __forceinline__ void contract(const Hid &hid, const LS &ls, const NetSite &n, HUnit hunit, Get get,
                                         Cx<float> acc[12])
{
    f4v re[3], im[3];
    contract_paths<CH, P, 0, P1>(hid, ls, n, hunit, get, contract_fetch<CH, P, 0>(hid, ls, n, hunit, get), re, im, acc);
}

// Workgroup b of a launch: each XCD (hardware workgroup b runs on XCD b % 8)
// walks one contiguous range of units, so that the neighbour reuse of that
// range stays in its own L2.  nblk8: workgroups / 8, or 0 (no remapping).
__device__ __forceinline__ int net_block(int nblk8)
{
    const int b = blockIdx.x;
    return nblk8 > 0 ? (b & 7) * nblk8 + (b >> 3) : b;
}

// XCD remapping of nb workgroups, once each XCD gets several of them
int net_remap(int &nb)
{
    if (nb < 64) return 0;
    nb = (nb + 7) / 8 * 8;
    return nb / 8;
}
int check_net_gauge(const qkx_gauge_s *U)
{
    if (U->prec != QKX_PREC_SINGLE || U->recon != QKX_RECON_18) {
        qkx::set_error("net: the gauge field must be FP32 with 18 reals");
        return QKX_ERR_ARG;
    }
    return QKX_SUCCESS;
}

// fn(integral_constant) for the network's hidden channels
template <class F> int with_ch(const qkx_net_s *n, F fn)
{
    if (n->ch == 16) return fn(std::integral_constant<int, 16>{});
    if (n->ch == 4) return fn(std::integral_constant<int, 4>{});
    return fn(std::integral_constant<int, 8>{});
}
} // namespace
