// qcd_flow.hip -- learned global proposal for SU(2) lattices: a
// gauge-equivariant normalising flow of masked coupling layers, evaluated
// with BF16 MFMA convolutions (FP32 accumulation), for an independence
// Metropolis step with the exact Wilson action.  No counterpart in the
// reference (new work); its plain heatbath is the fallback and the judge.
//
// Links: unit quaternions q = (a0, a1, a2, a3), U = a0 + i (a1 s1 + a2 s2 +
// a3 s3) = [[a0 + i a3, a2 + i a1], [-a2 + i a1, a0 - i a3]], stored
// links[(b * 4 + mu) * V + site] (float4), site = y + z N2 + t N2 N3 +
// x N2 N3 N4 (the canonical order of the C ABI).
//
// Coupling layer l (direction mu = l % 4, mask parity m = (l / 4) % 2)
// updates U_mu(x) at the active sites, sum_{nu != mu} x_nu + m even.  The
// staple sum A(x) = sum_nu [U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+ +
// U_nu(x+mu-nu)^+ U_mu(x-nu)^+ U_nu(x-nu)] holds frozen links only (the
// U_mu(x +- nu) sit on inactive sites), A = k V with V in SU(2), and the
// local action is -beta k (U V)_0.  W = U V = exp(i theta n.s) is gauge
// covariant; the layer maps theta in [0, pi] by a monotone rational-quadratic
// spline f whose parameters depend on frozen, gauge-invariant features, and
// sets U' = exp(i f(theta) n.s) V^+.  Haar measure in (theta, n) is
// sin^2(theta) d(theta) d(Omega), so log J = log f'(theta) + 2 log(sin
// f(theta) / sin theta).  log q(U) = -sum_layers log J (Haar prior, density
// 1).
//
// Conditioner per layer: features per site (channels-last, BF16, padded to
// 8): k(x)/6 at active sites (0 elsewhere), (P_nu rho)_0 of the three
// plaquettes in the planes orthogonal to mu, the active mask; then a 3^4
// stencil convolution to 32 channels + bias, tanh; then a 3^4 stencil
// convolution to 16 channels + bias (3K + 1 spline parameters used).
// Stencil point st = ((ox * 3 + oy) * 3 + oz) * 3 + ot, offsets o - 1 along
// x, y, z, t, periodic.  Convolutions are implicit GEMMs on
// v_mfma_f32_16x16x16_bf16: rows = sites, K = (stencil point, input
// channel), N = output channels.
//
// Spline (Durkan et al. 2019, rational-quadratic, K bins on [0, pi]): raw
// outputs r[0..K) widths, r[K..2K) heights, r[2K..3K] derivatives; widths =
// pi (eps + (1 - K eps) softmax), heights likewise, derivatives = eps_d +
// (1 - eps_d) softplus(r) / ln 2 (all-zero outputs give the identity map).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/qcd_hip.h"
#include "qcd_device.hpp"
#include "qcd_internal.h"

namespace {

constexpr int kStencil = 81;
constexpr int kCin0 = 8;     // input feature channels (5 used)
constexpr int kHidden = 32;
constexpr int kOut = 16;     // spline parameter channels (3K + 1 used)
constexpr int kMaxBins = 5;
constexpr float kPi = 3.14159265358979323846f;
constexpr float kMinW = 1e-3f, kMinD = 1e-3f;

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ bf8 as_bf(s8 v) { return __builtin_bit_cast(bf8, v); }

struct FGeom {
    int n1, n2, n3, n4;   // extents along x, y, z, t
    uint32_t V;
    qcd::FastDiv d2, d3, d4, dV;   // division by N2, N3, N4, V
};

__host__ __device__ inline uint16_t f2bf(float f)
{   // round to nearest even
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ inline float bf2f(uint16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

__device__ inline void coords(const FGeom& g, uint32_t s, int c[4])
{
    const uint32_t r = g.d2.div(s), r2 = g.d3.div(r), r3 = g.d4.div(r2);
    c[1] = (int)(s - r * (uint32_t)g.n2);
    c[2] = (int)(r - r2 * (uint32_t)g.n3);
    c[3] = (int)(r2 - r3 * (uint32_t)g.n4);
    c[0] = (int)r3;
}
__device__ inline uint32_t site(const FGeom& g, const int c[4])
{
    return (uint32_t)c[1] + (uint32_t)g.n2 * ((uint32_t)c[2] + (uint32_t)g.n3 * ((uint32_t)c[3] + (uint32_t)g.n4 * (uint32_t)c[0]));
}
__device__ inline int wrap(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }
__device__ inline uint32_t shifted(const FGeom& g, const int c[4], int d, int o)
{
    int e[4] = {c[0], c[1], c[2], c[3]};
    const int n[4] = {g.n1, g.n2, g.n3, g.n4};
    e[d] = wrap(e[d] + o, n[d]);
    return site(g, e);
}

// quaternion algebra for U = a0 + i a.s
__device__ inline float4 qmul(float4 a, float4 b)
{
    return make_float4(a.x * b.x - a.y * b.y - a.z * b.z - a.w * b.w,
                       a.x * b.y + b.x * a.y - (a.z * b.w - a.w * b.z),
                       a.x * b.z + b.x * a.z - (a.w * b.y - a.y * b.w),
                       a.x * b.w + b.x * a.w - (a.y * b.z - a.z * b.y));
}
__device__ inline float4 qdag(float4 a) { return make_float4(a.x, -a.y, -a.z, -a.w); }
__device__ inline float4 qadd(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

__device__ inline float4 link(const float4* L, const FGeom& g, uint32_t b, int mu, uint32_t s)
{
    return L[((size_t)b * 4 + mu) * g.V + s];
}

// staple sum of U_mu(x) (see the file comment).  The direction is a template
// parameter and the 18 links are all asked for first: a previous kernel's
// links come from beyond this XCD's L2, so each round of loads that waits for
// the one before costs a microsecond or two.
struct StapleLinks {
    float4 l[3][6];
};
template <int mu>
__device__ __forceinline__ void load_staple(StapleLinks& sl, const float4* L, const FGeom& g, uint32_t b, const int c[4])
{
    const uint32_t x = site(g, c);
    const uint32_t xp = shifted(g, c, mu, 1);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int nu = k + (k >= mu ? 1 : 0);
        const uint32_t xpn = shifted(g, c, nu, 1), xmn = shifted(g, c, nu, -1);
        int cm[4] = {c[0], c[1], c[2], c[3]};
        const int n[4] = {g.n1, g.n2, g.n3, g.n4};
        cm[nu] = wrap(cm[nu] - 1, n[nu]);
        const uint32_t xpmn = shifted(g, cm, mu, 1);   // x + mu - nu
        sl.l[k][0] = link(L, g, b, nu, xp);
        sl.l[k][1] = link(L, g, b, mu, xpn);
        sl.l[k][2] = link(L, g, b, nu, x);
        sl.l[k][3] = link(L, g, b, nu, xpmn);
        sl.l[k][4] = link(L, g, b, mu, xmn);
        sl.l[k][5] = link(L, g, b, nu, xmn);
    }
}
__device__ __forceinline__ float4 staple_sum(const StapleLinks& sl)
{
    float4 A = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float4* l = sl.l[k];
        const float4 f = qmul(qmul(l[0], qdag(l[1])), qdag(l[2]));
        const float4 r = qmul(qmul(qdag(l[3]), qdag(l[4])), l[5]);
        A = qadd(A, qadd(f, r));
    }
    return A;
}
// Nothing after this line is loaded before it, nothing before it later.
__device__ __forceinline__ void loads_issued() { asm volatile("" ::: "memory"); }

// (U_nu(x) U_rho(x+nu) U_nu(x+rho)^+ U_rho(x)^+)_0
__device__ __forceinline__ float plaq0(const float4* L, const FGeom& g, uint32_t b, int nu, int rho, const int c[4])
{
    const uint32_t x = site(g, c);
    const float4 p = qmul(qmul(link(L, g, b, nu, x), link(L, g, b, rho, shifted(g, c, nu, 1))),
                          qmul(qdag(link(L, g, b, nu, shifted(g, c, rho, 1))), qdag(link(L, g, b, rho, x))));
    return p.x;
}

__device__ inline bool is_active(const int c[4], int mu, int par)
{
    int s = par;
    for (int d = 0; d < 4; ++d)
        if (d != mu) s += c[d];
    return (s & 1) == 0;
}

// ---------------------------------------------------------------- kernels
// splitmix64's output function (a bijection of 64-bit words).
__host__ __device__ inline uint64_t mix64(uint64_t x)
{
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// 2 * n uniforms in (0, 1) (24 bits each) for item `j` of the draw keyed by
// `key`: counter-based, the counter (key, j) hashed before the splitmix64
// sequence starts, so neither neighbouring items nor draws with
// neighbouring keys share numbers.
template <int n>
__device__ inline void uniforms(uint64_t key, uint64_t j, float* u)
{
    uint64_t z = mix64(key ^ mix64(j + 0x632BE59BD9B4E019ull));
    for (int k = 0; k < n; ++k) {
        z += 0x9E3779B97F4A7C15ull;
        const uint64_t x = mix64(z);
        u[2 * k] = ((float)(uint32_t)(x >> 40) + 0.5f) * 5.9604644775390625e-8f;
        u[2 * k + 1] = ((float)(uint32_t)((x >> 8) & 0xffffffu) + 0.5f) * 5.9604644775390625e-8f;
    }
}

__global__ void k_flow_haar(float4* L, uint64_t n, uint64_t seed)
{
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    float u[4];
    uniforms<2>(mix64(seed), j, u);
    // Box-Muller: four Gaussians, normalised: uniform on S^3 = Haar on SU(2)
    const float r1 = sqrtf(-2.f * logf(u[0])), r2 = sqrtf(-2.f * logf(u[2]));
    float s1, c1, s2, c2;
    sincosf(2.f * kPi * u[1], &s1, &c1);
    sincosf(2.f * kPi * u[3], &s2, &c2);
    float4 q = make_float4(r1 * c1, r1 * s1, r2 * c2, r2 * s2);
    const float nrm = rsqrtf(q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w);
    L[j] = make_float4(q.x * nrm, q.y * nrm, q.z * nrm, q.w * nrm);
}

template <int mu>
__global__ __launch_bounds__(256) void k_flow_features(const float4* L, uint16_t* feat, FGeom g, uint32_t B, int par)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= B * g.V) return;
    const uint32_t b = g.dV.div(j), s = j - b * g.V;
    int c[4];
    coords(g, s, c);
    const bool act = is_active(c, mu, par);
    StapleLinks sl;
    load_staple<mu>(sl, L, g, b, c);
    // the three planes orthogonal to mu: U_nu(x), U_rho(x) are among the staple's links
    float4 un[3], ur[3];
    int k = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j2 = i + 1; j2 < 3; ++j2) {
            const int nu = i + (i >= mu ? 1 : 0), rho = j2 + (j2 >= mu ? 1 : 0);
            ur[k] = link(L, g, b, rho, shifted(g, c, nu, 1));
            un[k] = link(L, g, b, nu, shifted(g, c, rho, 1));
            ++k;
        }
    loads_issued();
    float f[kCin0] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (act) {
        const float4 A = staple_sum(sl);
        f[0] = sqrtf(A.x * A.x + A.y * A.y + A.z * A.z + A.w * A.w) * (1.f / 6.f);
        f[4] = 1.f;
    }
    k = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j2 = i + 1; j2 < 3; ++j2) {
            const float4 p = qmul(qmul(sl.l[i][2], ur[k]), qmul(qdag(un[k]), qdag(sl.l[j2][2])));
            f[++k] = p.x;
        }
    uint4 o;   // 8 channels, 16 bytes
    o.x = f2bf(f[0]) | (uint32_t)f2bf(f[1]) << 16;
    o.y = f2bf(f[2]) | (uint32_t)f2bf(f[3]) << 16;
    o.z = f2bf(f[4]) | (uint32_t)f2bf(f[5]) << 16;
    o.w = f2bf(f[6]) | (uint32_t)f2bf(f[7]) << 16;
    reinterpret_cast<uint4*>(feat)[j] = o;
}

// ---------------------------------------------------------------- convolution
// Operand orders of the implicit GEMM.  A k-step is 16 consecutive k =
// st * cin + channel; lane (n, q) = (lane % 16, lane / 16) holds the four k
// at 4 q of row / column n.  Weights are stored in the order the lanes load
// them, whole cache lines per wavefront; with 32 input channels a stencil
// point's two k-steps come in one 16-byte load, so hidden channel c sits at
// hid_pos(c) of its site.
constexpr int kSteps1 = 41;   // conv1: 81 * 8 / 16, the last half empty
constexpr size_t kW1Pack = (size_t)2 * kSteps1 * 64 * 4;
__host__ __device__ constexpr int hid_pos(int c) { return 8 * ((c % 16) / 4) + 4 * (c / 16) + c % 4; }
__host__ __device__ constexpr size_t w1_pos(int n, int k)
{
    return ((size_t)((n / 16) * kSteps1 + k / 16) * 64 + n % 16 + 16 * ((k % 16) / 4)) * 4 + k % 4;
}
__host__ __device__ constexpr size_t w2_pos(int n, int k) { return ((size_t)(k / 32) * 64 + n + 16 * ((k % 16) / 4)) * 8 + 4 * ((k % 32) / 16) + k % 4; }
__host__ __device__ constexpr size_t w2t_pos(int c, int k)   // k = st * 16 + n
{
    return ((size_t)((c / 16) * kStencil + k / 16) * 64 + c % 16 + 16 * ((k % 16) / 4)) * 4 + k % 4;
}

template <int CIN> struct ConvOp {
    static constexpr int loads = CIN == 8 ? kSteps1 : kStencil;   // operand loads along k
    static constexpr int per = CIN == 32 ? 2 : 1;                 // k-steps per load
    static constexpr int ntiles = CIN == 32 ? 1 : 2;              // output tiles of 16 channels
    typedef short V __attribute__((ext_vector_type(4 * per)));
};

// What becomes of output n of a row: the hidden layer (tanh, BF16 at
// hid_pos), the spline parameters (FP32), or, given the hidden layer h, the
// gradient before its tanh (v (1 - h^2), BF16).
enum ConvOut { CONV_TANH, CONV_RAW, CONV_TANH_BACK };
template <int ACT, int COUT>
__device__ __forceinline__ void conv_store(float v, size_t r, int n, const uint16_t* h, uint16_t* out_bf, float* out_f)
{
    if constexpr (ACT == CONV_TANH) {
        out_bf[r * COUT + hid_pos(n)] = f2bf(tanhf(v));
    } else if constexpr (ACT == CONV_RAW) {
        out_f[r * COUT + n] = v;
    } else {
        const float hv = bf2f(h[r * COUT + hid_pos(n)]);
        out_bf[r * COUT + n] = f2bf(v * (1.f - hv * hv));
    }
}

// One wavefront: MT tiles of 16 sites x NT tiles of 16 output channels.
// in[row * CIN + channel] (BF16); outputs as conv_store.  The loads of BS
// operand steps are issued before the matrix instructions of the previous BS,
// which run in k order whatever the shape, so every shape gives the same sums.
template <int CIN, int MT, int NT, int BS, int ACT>
__global__ __launch_bounds__(256) void k_flow_conv(const uint16_t* in, const uint16_t* wt, const float* bias,
                                                   const uint16_t* h, uint16_t* out_bf, float* out_f, FGeom g,
                                                   uint32_t ntile_m)
{
    using Op = ConvOp<CIN>;
    using V = typename Op::V;
    constexpr int COUT = 16 * Op::ntiles, NL = Op::loads, NB = (NL + BS - 1) / BS;
    const uint32_t wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const uint32_t groups = (ntile_m + MT - 1) / MT;
    if (wave >= groups * (Op::ntiles / NT)) return;   // whole wavefront
    const uint32_t tm = wave % groups, tn = (wave / groups) * NT;
    // byte offsets of the 3 neighbour positions along each direction, per tile; the tile's configuration is the base
    const char* base[MT];
    uint32_t xo[MT][3], yo[MT][3], zo[MT][3], to[MT][3];
    const int n[4] = {g.n1, g.n2, g.n3, g.n4};
    constexpr uint32_t B = 2u * CIN;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const uint32_t tile = min(tm * MT + m, ntile_m - 1u);
        const uint32_t b = g.dV.div(tile * 16);   // 16 divides V: a tile is inside one configuration
        base[m] = reinterpret_cast<const char*>(in) + (size_t)b * g.V * B;
        int c[4];
        coords(g, tile * 16 - b * g.V + (uint32_t)(lane & 15), c);
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            // the lane's 4 (or 2 x 4) channels of a point: 8 q bytes on, or 16 q
            // for two k-steps; with 8 channels a k-step is two points
            xo[m][o] = (uint32_t)wrap(c[0] + o - 1, n[0]) * (uint32_t)(n[1] * n[2] * n[3]) * B +
                       (CIN == 8 ? 8u * (q & 1) : 8u * Op::per * (uint32_t)q);
            yo[m][o] = (uint32_t)wrap(c[1] + o - 1, n[1]) * B;
            zo[m][o] = (uint32_t)wrap(c[2] + o - 1, n[2]) * (uint32_t)n[1] * B;
            to[m][o] = (uint32_t)wrap(c[3] + o - 1, n[3]) * (uint32_t)(n[1] * n[2]) * B;
        }
    }
    auto point = [&](int m, int st) { return xo[m][st / 27] + yo[m][(st / 9) % 3] + zo[m][(st / 3) % 3] + to[m][st % 3]; };
    auto offset = [&](int m, int l) -> uint32_t {
        if constexpr (CIN == 8) {
            const uint32_t a = point(m, 2 * l), b = 2 * l + 1 < kStencil ? point(m, 2 * l + 1) : a;
            return q < 2 ? a : b;
        } else {
            return point(m, l);
        }
    };
    const V* wl[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) wl[t] = reinterpret_cast<const V*>(wt) + (size_t)(tn + t) * NL * 64 + lane;
    f4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};
    V av[2][BS][MT], bv[2][BS][NT];
    auto issue = [&](int bt) {
#pragma unroll
        for (int i = 0; i < BS; ++i) {
            const int l = bt * BS + i;
            if (l >= NL) break;
#pragma unroll
            for (int t = 0; t < NT; ++t) bv[bt & 1][i][t] = wl[t][(size_t)l * 64];
#pragma unroll
            for (int m = 0; m < MT; ++m) av[bt & 1][i][m] = *reinterpret_cast<const V*>(base[m] + offset(m, l));
        }
        asm volatile("" ::: "memory");   // these loads before, the next batch's after
    };
    issue(0);
#pragma unroll
    for (int bt = 0; bt < NB; ++bt) {
        if (bt + 1 < NB) issue(bt + 1);
#pragma unroll
        for (int i = 0; i < BS; ++i) {
            if (bt * BS + i >= NL) break;
#pragma unroll
            for (int h = 0; h < Op::per; ++h)
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        s4 a, b;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            a[j] = av[bt & 1][i][m][4 * h + j];
                            b[j] = bv[bt & 1][i][t][4 * h + j];
                        }
                        acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[m][t], 0, 0, 0);
                    }
        }
    }
    // lane holds D[4 * (lane / 16) + i][lane % 16]
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (tm * MT + m >= ntile_m) break;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int ncol = (int)(tn + t) * 16 + (lane & 15);
            const float bs = bias[ncol];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const size_t r = (size_t)(tm * MT + m) * 16 + 4 * q + i;
                const float v = acc[m][t][i] + bs;
                conv_store<ACT, COUT>(v, r, ncol, h, out_bf, out_f);
            }
        }
    }
}

// The same sums with the input in LDS: one workgroup of WV wavefronts per
// x-plane of a configuration stages the plane and its two neighbours (`plane`
// sites each, contiguous) and every one of the 81 gathers of a site reads
// from there.  A wavefront takes MT tiles of 16 sites at a time.
template <int CIN, int MT, int BS, int WV, int ACT>
__global__ __launch_bounds__(64 * WV) void k_flow_conv_plane(const uint16_t* in, const uint16_t* wt, const float* bias,
                                                             const uint16_t* h, uint16_t* out_bf, float* out_f, FGeom g,
                                                             uint32_t plane)
{
    using Op = ConvOp<CIN>;
    using V = typename Op::V;
    constexpr int COUT = 16 * Op::ntiles, NL = Op::loads, NB = (NL + BS - 1) / BS, NT = Op::ntiles;
    constexpr uint32_t B = 2u * CIN;
    extern __shared__ uint4 planes[];
    const uint32_t b = blockIdx.x / (uint32_t)g.n1, x = blockIdx.x % (uint32_t)g.n1;
    const uint32_t pv = plane * B / 16u;   // 16-byte vectors of a plane
#pragma unroll
    for (int o = 0; o < 3; ++o) {
        const uint4* src = reinterpret_cast<const uint4*>(in) +
                           ((size_t)b * (uint32_t)g.n1 + (uint32_t)wrap((int)x + o - 1, g.n1)) * pv;
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < pv; i += 64u * WV) planes[o * pv + i] = src[i];
    }
    __syncthreads();
    const char* sm = reinterpret_cast<const char*>(planes);
    const uint32_t w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), tiles = plane / 16u;
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const int n[4] = {g.n1, g.n2, g.n3, g.n4};
    const V* wl[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) wl[t] = reinterpret_cast<const V*>(wt) + (size_t)t * NL * 64 + lane;
    for (uint32_t t0 = w * MT; t0 < tiles; t0 += WV * MT) {
        uint32_t yo[MT][3], zo[MT][3], to[MT][3];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            int c[4];
            coords(g, min(t0 + m, tiles - 1u) * 16u + (uint32_t)(lane & 15), c);
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                yo[m][o] = (uint32_t)wrap(c[1] + o - 1, n[1]) * B + (CIN == 8 ? 8u * (q & 1) : 8u * Op::per * (uint32_t)q);
                zo[m][o] = (uint32_t)wrap(c[2] + o - 1, n[2]) * (uint32_t)n[1] * B;
                to[m][o] = (uint32_t)wrap(c[3] + o - 1, n[3]) * (uint32_t)(n[1] * n[2]) * B;
            }
        }
        auto point = [&](int m, int st) {
            return (uint32_t)(st / 27) * plane * B + yo[m][(st / 9) % 3] + zo[m][(st / 3) % 3] + to[m][st % 3];
        };
        auto offset = [&](int m, int l) -> uint32_t {
            if constexpr (CIN == 8) {
                const uint32_t a0 = point(m, 2 * l), a1 = 2 * l + 1 < kStencil ? point(m, 2 * l + 1) : a0;
                return q < 2 ? a0 : a1;
            } else {
                return point(m, l);
            }
        };
        f4 acc[MT][NT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[m][t] = f4{0.f, 0.f, 0.f, 0.f};
        V av[2][BS][MT], bv[2][BS][NT];
        auto issue = [&](int bt) {
#pragma unroll
            for (int i = 0; i < BS; ++i) {
                const int l = bt * BS + i;
                if (l >= NL) break;
#pragma unroll
                for (int t = 0; t < NT; ++t) bv[bt & 1][i][t] = wl[t][(size_t)l * 64];
#pragma unroll
                for (int m = 0; m < MT; ++m) av[bt & 1][i][m] = *reinterpret_cast<const V*>(sm + offset(m, l));
            }
            asm volatile("" ::: "memory");
        };
        issue(0);
#pragma unroll
        for (int bt = 0; bt < NB; ++bt) {
            if (bt + 1 < NB) issue(bt + 1);
#pragma unroll
            for (int i = 0; i < BS; ++i) {
                if (bt * BS + i >= NL) break;
#pragma unroll
                for (int h = 0; h < Op::per; ++h)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            s4 av4, bv4;
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                av4[j] = av[bt & 1][i][m][4 * h + j];
                                bv4[j] = bv[bt & 1][i][t][4 * h + j];
                            }
                            acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av4, bv4, acc[m][t], 0, 0, 0);
                        }
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (t0 + m >= tiles) break;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int ncol = t * 16 + (lane & 15);
                const float bs = bias[ncol];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const size_t r = (size_t)blockIdx.x * plane + (size_t)(t0 + m) * 16 + 4 * q + i;
                    const float v = acc[m][t][i] + bs;
                    conv_store<ACT, COUT>(v, r, ncol, h, out_bf, out_f);
                }
            }
        }
    }
}

// Launch for `rows` sites.  Measured for 32 -> 16 channels on 8^3 x 4 sites
// (one wavefront per tile and eight gathers in flight before: 33 us for one
// configuration, 159 us for 64, bound by the gathers' latency and the L1):
//   one configuration (128 tiles)    4.0 us as one tile per wavefront, 14 in planes
//   8 (64 planes)                   10.2                             12.2
//   16 (128 planes)                 16.6                             12.6
//   64 (512 planes)                 45.7 with four tiles             25.1, with 8 wavefronts 29.3
// The matrix instructions of 64 configurations take 8.6 us.
// 16 -> 32 channels (backward) has twice the weights to read per input byte:
// 16 configurations 21.4 us as one tile per wavefront, 46.7 in planes (it has
// no such kernel); 64: 56 with four tiles, 76 with one, 78 in planes.
template <int CIN, int ACT>
void launch_conv(const uint16_t* in, const uint16_t* wt, const float* bias, const uint16_t* h, uint16_t* out_bf, float* out_f,
                 const FGeom& g, uint32_t rows, hipStream_t st)
{
    constexpr int NTT = ConvOp<CIN>::ntiles;
    const uint32_t tiles = rows / 16, plane = g.V / (uint32_t)g.n1, planes = rows / plane, lds = 3u * plane * 2u * CIN;
    if (CIN != 16 && plane % 16 == 0 && lds <= 64u * 1024u && planes >= 96u) {
        if constexpr (CIN != 16) {
            if (planes <= 256u)
                hipLaunchKernelGGL((k_flow_conv_plane<CIN, 2, 6, 8, ACT>), dim3(planes), dim3(512), lds, st, in, wt, bias, h,
                                   out_bf, out_f, g, plane);
            else
                hipLaunchKernelGGL((k_flow_conv_plane<CIN, 2, 6, 4, ACT>), dim3(planes), dim3(256), lds, st, in, wt, bias, h,
                                   out_bf, out_f, g, plane);
        }
    } else if (tiles <= 4096u) {
        hipLaunchKernelGGL((k_flow_conv<CIN, 1, 1, 9, ACT>), dim3(tiles * NTT), dim3(64), 0, st, in, wt, bias, h,
                           out_bf, out_f, g, tiles);
    } else {
        hipLaunchKernelGGL((k_flow_conv<CIN, 4, NTT, 3, ACT>), dim3((tiles + 15) / 16), dim3(256), 0, st, in, wt, bias,
                           h, out_bf, out_f, g, tiles);
    }
}

// The number of bins is a template parameter, so that the knots live in
// registers and a site's 16 raw parameters are four loads (with a run-time
// count every one of them was a load of its own, waited for in turn).
template <int K> struct Spline {
    float xk[K + 1], yk[K + 1], d[K + 1];
};

__device__ inline float softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

__device__ __forceinline__ void load_raw(float (&r)[kOut], const float* prm, size_t row)
{
    const float4* v = reinterpret_cast<const float4*>(prm) + 4 * row;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 a = v[q];
        r[4 * q] = a.x;
        r[4 * q + 1] = a.y;
        r[4 * q + 2] = a.z;
        r[4 * q + 3] = a.w;
    }
}

template <int K> __device__ __forceinline__ void make_spline(const float (&r)[kOut], Spline<K>& sp)
{
    float mw = r[0], mh = r[K];
#pragma unroll
    for (int i = 1; i < K; ++i) {
        mw = fmaxf(mw, r[i]);
        mh = fmaxf(mh, r[K + i]);
    }
    float ew[K], eh[K], sw = 0.f, sh = 0.f;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        ew[i] = expf(r[i] - mw);
        eh[i] = expf(r[K + i] - mh);
        sw += ew[i];
        sh += eh[i];
    }
    sp.xk[0] = sp.yk[0] = 0.f;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        sp.xk[i + 1] = sp.xk[i] + kPi * (kMinW + (1.f - K * kMinW) * ew[i] / sw);
        sp.yk[i + 1] = sp.yk[i] + kPi * (kMinW + (1.f - K * kMinW) * eh[i] / sh);
    }
    sp.xk[K] = sp.yk[K] = kPi;
#pragma unroll
    for (int i = 0; i <= K; ++i) sp.d[i] = kMinD + (1.f - kMinD) * softplus(r[2 * K + i]) * 1.4426950408889634f;
}

// Bin of v among the knots (the first whose upper knot exceeds v) and its corner values.
template <int K> struct Bin {
    float x0, x1, y0, y1, d0, d1;
};
template <int K> __device__ __forceinline__ Bin<K> find_bin(const Spline<K>& sp, const float (&knots)[K + 1], float v)
{
    Bin<K> b{sp.xk[0], sp.xk[1], sp.yk[0], sp.yk[1], sp.d[0], sp.d[1]};
    bool go = true;
#pragma unroll
    for (int i = 1; i < K; ++i) {
        go = go && v >= knots[i];
        if (go) b = Bin<K>{sp.xk[i], sp.xk[i + 1], sp.yk[i], sp.yk[i + 1], sp.d[i], sp.d[i + 1]};
    }
    return b;
}

// forward: y = f(x), dlog = log f'(x)
template <int K> __device__ __forceinline__ float spline_fwd(const Spline<K>& sp, float x, float& dlog)
{
    const Bin<K> b = find_bin<K>(sp, sp.xk, x);
    const float w = b.x1 - b.x0, h = b.y1 - b.y0, s = h / w;
    const float xi = fminf(fmaxf((x - b.x0) / w, 0.f), 1.f), om = 1.f - xi;
    const float den = s + (b.d1 + b.d0 - 2.f * s) * xi * om;
    const float y = b.y0 + h * (s * xi * xi + b.d0 * xi * om) / den;
    const float num = s * s * (b.d1 * xi * xi + 2.f * s * xi * om + b.d0 * om * om);
    dlog = logf(num) - 2.f * logf(den);
    return y;
}

// inverse: x = f^-1(y), dlog = log f'(x)
template <int K> __device__ __forceinline__ float spline_inv(const Spline<K>& sp, float y, float& dlog)
{
    const Bin<K> b = find_bin<K>(sp, sp.yk, y);
    const float w = b.x1 - b.x0, h = b.y1 - b.y0, s = h / w;
    const float dy = y - b.y0, dd = b.d1 + b.d0 - 2.f * s;
    const float a = h * (s - b.d0) + dy * dd;
    const float bq = h * b.d0 - dy * dd;
    const float cq = -s * dy;
    const float disc = fmaxf(bq * bq - 4.f * a * cq, 0.f);
    const float xi = fminf(fmaxf(2.f * cq / (-bq - sqrtf(disc)), 0.f), 1.f), om = 1.f - xi;
    const float den = s + dd * xi * om;
    const float num = s * s * (b.d1 * xi * xi + 2.f * s * xi * om + b.d0 * om * om);
    dlog = logf(num) - 2.f * logf(den);
    return b.x0 + xi * w;
}

// Coupling of layer (mu, par): forward (inverse = 0) maps theta -> f(theta),
// inverse maps theta' -> f^-1(theta'); both add log J = log f'(theta) +
// 2 log(sin f(theta) / sin theta) of the forward map to logj[row].
template <int mu, int K>
__global__ __launch_bounds__(256) void k_flow_couple(float4* L, const float* prm, float* logj, FGeom g, uint32_t B, int par,
                                                     int inverse)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= B * g.V) return;
    const uint32_t b = g.dV.div(j), s = j - b * g.V;
    int c[4];
    coords(g, s, c);
    if (!is_active(c, mu, par)) return;
    StapleLinks sl;
    load_staple<mu>(sl, L, g, b, c);
    float4& U = L[((size_t)b * 4 + mu) * g.V + s];
    const float4 U0 = U;
    float raw[kOut];
    load_raw(raw, prm, j);
    const float lj0 = logj[j];
    loads_issued();
    const float4 A = staple_sum(sl);
    const float k = sqrtf(A.x * A.x + A.y * A.y + A.z * A.z + A.w * A.w);
    if (!(k > 1e-20f)) return;
    const float ik = 1.f / k;
    const float4 Vq = make_float4(A.x * ik, A.y * ik, A.z * ik, A.w * ik);
    const float4 W = qmul(U0, Vq);
    const float sn = sqrtf(W.y * W.y + W.z * W.z + W.w * W.w);
    const float th = atan2f(sn, W.x);
    Spline<K> sp;
    make_spline<K>(raw, sp);
    float dlog, th2;
    if (!inverse) th2 = spline_fwd(sp, th, dlog);
    else th2 = spline_inv(sp, th, dlog);
    const float th_in = inverse ? th2 : th, th_out = inverse ? th : th2;   // theta and f(theta)
    const float si = sinf(th_in), so = sinf(th_out);
    const float ratio = (si > 1e-6f && so > 1e-6f) ? so / si : expf(dlog);   // limit at the poles: f'(theta)
    logj[j] = lj0 + (dlog + 2.f * logf(ratio));
    float4 Wn;
    if (sn > 1e-12f) {
        const float f = sinf(th2) / sn;
        Wn = make_float4(cosf(th2), W.y * f, W.z * f, W.w * f);
    } else {
        Wn = make_float4(cosf(th2) >= 0.f ? 1.f : -1.f, 0.f, 0.f, 0.f);
    }
    U = qmul(Wn, qdag(Vq));
}

// log J = log f'(theta) + 2 log(sin f(theta) / sin theta) of the forward map
// at theta (theta_in) with image theta_out; at the poles the ratio's limit
// f'(theta).
__device__ inline float log_jac(float dlog, float th_in, float th_out)
{
    const float si = sinf(th_in), so = sinf(th_out);
    const float ratio = (si > 1e-6f && so > 1e-6f) ? so / si : expf(dlog);
    return dlog + 2.f * logf(ratio);
}

// Learned Metropolis update of layer (mu, par)'s active links of
// configuration 0 (a Metropolis-within-Gibbs step on each).  The layer's
// spline parameters depend on frozen links only, and no plaquette holds two
// active links, so given the frozen links the target factorises into
// exp(beta k (U V)_0) per active link and the layer's map, applied to a
// Haar draw, proposes each active link independently with density
// q_a(U) = exp(-log J(f^-1(theta(U V)))) (w.r.t. Haar).  Each active link is
// replaced by its proposal U' with probability
// min(1, exp(beta k ((U'V)_0 - (UV)_0)) q_a(U) / q_a(U')): detailed balance
// for every link, so the Wilson-action distribution stays exact.  Counts
// accepted links in *accepted (one atomic per wavefront).
// The sweep's seed: mode 0 sets it, 1 advances it by one and counts a
// sweep (a recorded sweep), 2 sets it and counts a sweep.
__global__ void k_flow_imh_key(unsigned long long* imh, unsigned long long seed, int mode)
{
    if (threadIdx.x == 0) {
        imh[2] = mode == 1 ? imh[2] + 1ull : seed;
        if (mode) imh[1] += 1ull;
    }
}

template <int mu, int K>
__global__ __launch_bounds__(256) void k_flow_imh_couple(float4* L, const float* prm, FGeom g, int par,
                                                         float beta, uint64_t lmix, unsigned long long* imh)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    // the layer's draw key: (sweep seed, layer) hashed
    const uint64_t seed = mix64(mix64((uint64_t)imh[2]) ^ lmix);
    unsigned long long* accepted = imh;
    bool acc = false;
    if (s < g.V) {
        int c[4];
        coords(g, s, c);
        if (is_active(c, mu, par)) {
            StapleLinks sl;
            load_staple<mu>(sl, L, g, 0, c);
            float4& U = L[(size_t)mu * g.V + s];
            const float4 U0 = U;
            float raw[kOut];
            load_raw(raw, prm, s);
            loads_issued();
            const float4 A = staple_sum(sl);
            const float k = sqrtf(A.x * A.x + A.y * A.y + A.z * A.z + A.w * A.w);
            if (k > 1e-20f) {
                const float ik = 1.f / k;
                const float4 Vq = make_float4(A.x * ik, A.y * ik, A.z * ik, A.w * ik);
                const float4 W = qmul(U0, Vq);
                const float th = atan2f(sqrtf(W.y * W.y + W.z * W.z + W.w * W.w), W.x);
                Spline<K> sp;
                make_spline<K>(raw, sp);
                float dlog;
                const float thz = spline_inv(sp, th, dlog);
                const float lj_cur = log_jac(dlog, thz, th);
                // the proposal: a Haar element z = (cos thz', sin thz' n') in the W frame, mapped
                float u[6];
                uniforms<3>(seed, s, u);
                const float r1 = sqrtf(-2.f * logf(u[0])), r2 = sqrtf(-2.f * logf(u[2]));
                float s1, c1, s2, c2;
                sincosf(2.f * kPi * u[1], &s1, &c1);
                sincosf(2.f * kPi * u[3], &s2, &c2);
                const float4 zq = make_float4(r1 * c1, r1 * s1, r2 * c2, r2 * s2);
                const float zs = sqrtf(zq.y * zq.y + zq.z * zq.z + zq.w * zq.w);
                const float thz2 = atan2f(zs, zq.x);
                float dlog2;
                const float th2 = spline_fwd(sp, thz2, dlog2);
                const float lj_prop = log_jac(dlog2, thz2, th2);
                // log a = beta k (cos th2 - cos th) + log q(cur) - log q(prop)
                const float log_a = beta * k * (cosf(th2) - cosf(th)) - lj_cur + lj_prop;
                if (logf(u[4]) < log_a) {
                    float4 Wn;
                    if (zs > 1e-12f) {
                        const float f = sinf(th2) / zs;
                        Wn = make_float4(cosf(th2), zq.y * f, zq.z * f, zq.w * f);
                    } else {
                        Wn = make_float4(cosf(th2) >= 0.f ? 1.f : -1.f, 0.f, 0.f, 0.f);
                    }
                    const float4 Un = qmul(Wn, qdag(Vq));
                    const float nn = rsqrtf(Un.x * Un.x + Un.y * Un.y + Un.z * Un.z + Un.w * Un.w);
                    U = make_float4(Un.x * nn, Un.y * nn, Un.z * nn, Un.w * nn);
                    acc = true;
                }
            }
        }
    }
    const unsigned long long m = __ballot(acc);
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(accepted, (unsigned long long)__popcll(m));
}

// ---------------------------------------------------------------- training
// Layer-local forward KL: for every coupling layer l, the mean over data
// configurations of sum over active links of log J(f^-1(theta)) =
// -log q_a(U_a | frozen links), the density with which the learned
// Metropolis sweep proposes each active link.  The layer's input is the data
// configuration itself, so a layer's loss depends on its own parameters
// only, and the gradient flows back through conv2, tanh and conv1 alone.

// -log q_a of one active link in double precision (the map of make_spline /
// spline_inv / log_jac, written for double) and its gradient gr with respect
// to the 3K + 1 raw spline parameters r, from the formulas of bin `bin`;
// pw, ph: the softmax of the widths and heights, th = angle of U V.  In the bin
// with corners (x0, y0), sizes (w, h), slope s = h / w and end derivatives d0, d1
// the inverse xi solves y0 + h A / den = th, and
//   nll = log f' + 2 log(sin th / sin(x0 + xi w)),  f' = s^2 N / den^2,
// so a parameter p moves it by its direct derivative plus, through xi,
// -(dy/dp) / (w f') times the derivative in xi.  (Differences of nll at r +- h
// were 27 evaluations per link: 231 us for 32768 sites, now 8 to 11 us.)
template <int K>
__device__ __forceinline__ double nll_grad_bin(const float (&rf)[kOut], const double (&pw)[K], const double (&ph)[K], double th,
                                               int bin, float (&gr)[kOut])
{
    const double pi = 3.14159265358979323846, ln2i = 1.4426950408889634;
    const double scale = pi * (1.0 - K * (double)kMinW);
    double x0 = 0.0, y0 = 0.0, w = 0.0, h = 0.0, xa = 0.0, ya = 0.0;
    float r0 = 0.f, r1 = 0.f;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const double xb = i == K - 1 ? pi : xa + pi * (double)kMinW + scale * pw[i];
        const double yb = i == K - 1 ? pi : ya + pi * (double)kMinW + scale * ph[i];
        if (i == bin) {
            x0 = xa;
            y0 = ya;
            w = xb - xa;
            h = yb - ya;
            r0 = rf[2 * K + i];
            r1 = rf[2 * K + i + 1];
        }
        xa = xb;
        ya = yb;
    }
    auto sp = [&](double x) { return x > 30.0 ? x : log1p(exp(x)); };
    auto sg = [&](double x) { return x > 30.0 ? 1.0 : 1.0 / (1.0 + exp(-x)); };
    const double dk = (1.0 - (double)kMinD) * ln2i;
    const double d0 = (double)kMinD + dk * sp((double)r0), d1 = (double)kMinD + dk * sp((double)r1);
    const double s = h / w, dy = th - y0, dd = d1 + d0 - 2.0 * s;
    const double a = h * (s - d0) + dy * dd, bq = h * d0 - dy * dd, cq = -s * dy;
    const double disc = fmax(bq * bq - 4.0 * a * cq, 0.0);
    const double xi = fmin(fmax(2.0 * cq / (-bq - sqrt(disc)), 0.0), 1.0), om = 1.0 - xi;
    const double xo = xi * om;
    const double den = s + dd * xo, N = d1 * xi * xi + 2.0 * s * xo + d0 * om * om, A = s * xi * xi + d0 * xo;
    const double iden = 1.0 / den, iN = 1.0 / N;
    const double dlog = log(s * s * N) - 2.0 * log(den);
    const double thz = x0 + xi * w, si = sin(thz), so = sin(th);
    const bool pole = !(si > 1e-9 && so > 1e-9);   // there the ratio's limit f' stands for sin th / sin thz
    const double nll = pole ? 3.0 * dlog : dlog + 2.0 * log(so / si);
    const double c1 = pole ? 3.0 : 1.0, cot = pole ? 0.0 : cos(thz) / si;
    // direct derivatives of log f' and of y = y0 + h A / den
    const double den_s = 1.0 - 2.0 * xo;
    const double l_s = 2.0 / s + 2.0 * xo * iN - 2.0 * den_s * iden;
    const double l_d0 = om * om * iN - 2.0 * xo * iden, l_d1 = xi * xi * iN - 2.0 * xo * iden;
    const double l_xi = (2.0 * d1 * xi + 2.0 * s * (1.0 - 2.0 * xi) - 2.0 * d0 * om) * iN - 2.0 * dd * (1.0 - 2.0 * xi) * iden;
    const double y_s = h * (xi * xi * den - A * den_s) * iden * iden;
    const double y_d0 = h * xo * (den - A) * iden * iden, y_d1 = -h * A * xo * iden * iden;
    const double y_h = A * iden + y_s / w, y_w = -y_s * s / w;
    // d nll / d xi over dy / d xi = w f'
    const double f1 = s * s * N * iden * iden, q = (c1 * l_xi - 2.0 * cot * w) / (w * f1);
    const double g_x0 = -2.0 * cot, g_w = -c1 * l_s * s / w - 2.0 * cot * xi - q * y_w;
    const double g_y0 = -q, g_h = c1 * l_s / w - q * y_h;
    const double g_d0 = c1 * l_d0 - q * y_d0, g_d1 = c1 * l_d1 - q * y_d1;
    // softmax: x0 is the sum of the widths below the bin
    double mwg = 0.0, mhg = 0.0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        mwg += pw[i] * (i < bin ? g_x0 : (i == bin ? g_w : 0.0));
        mhg += ph[i] * (i < bin ? g_y0 : (i == bin ? g_h : 0.0));
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
        gr[i] = (float)(scale * pw[i] * ((i < bin ? g_x0 : (i == bin ? g_w : 0.0)) - mwg));
        gr[K + i] = (float)(scale * ph[i] * ((i < bin ? g_y0 : (i == bin ? g_h : 0.0)) - mhg));
    }
#pragma unroll
    for (int i = 0; i <= K; ++i)
        gr[2 * K + i] = i == bin ? (float)(g_d0 * dk * sg((double)r0)) : (i == bin + 1 ? (float)(g_d1 * dk * sg((double)r1)) : 0.f);
    return nll;
}

// The same in the bin of th.  At a knot nll has a kink in the heights: the
// gradient is that of the symmetric difference over a step of kKinkStep, the
// mean of both sides' derivatives weighted by the parts of the step in which the
// knot lies above and below th.
constexpr double kKinkStep = 1e-5;
template <int K> __device__ __forceinline__ double nll_grad_link(const float (&rf)[kOut], double th, float (&gr)[kOut])
{
    const double pi = 3.14159265358979323846;
    double mw = rf[0], mh = rf[K];
#pragma unroll
    for (int i = 1; i < K; ++i) {
        mw = fmax(mw, (double)rf[i]);
        mh = fmax(mh, (double)rf[K + i]);
    }
    double pw[K], ph[K], sw = 0.0, sh = 0.0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        pw[i] = exp((double)rf[i] - mw);
        ph[i] = exp((double)rf[K + i] - mh);
        sw += pw[i];
        sh += ph[i];
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
        pw[i] /= sw;
        ph[i] /= sh;
    }
    const double scale = pi * (1.0 - K * (double)kMinW);
    // the bin, and the knot (number edge, at y = ye, heights below it se) within reach of a step
    double ya = 0.0, sa = 0.0, ye = 0.0, se = 0.0;
    int bin = 0, edge = 0;
#pragma unroll
    for (int m = 1; m < K; ++m) {
        ya += pi * (double)kMinW + scale * ph[m - 1];
        sa += ph[m - 1];
        if (th >= ya) bin = m;
        if (fabs(th - ya) < kKinkStep) {   // |d ya / d r| <= scale / 4 < 1
            edge = m;
            ye = ya;
            se = sa;
        }
    }
    const double nll = nll_grad_bin<K>(rf, pw, ph, th, bin, gr);
    if (edge) {
        float go[kOut];
        const bool up = bin == edge;   // th lies in the bin above the knot
        (void)nll_grad_bin<K>(rf, pw, ph, th, up ? edge - 1 : edge, go);
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const double dy = scale * ph[i] * ((i < edge ? 1.0 : 0.0) - se);
            // part of the step with the knot above th, where the lower bin holds
            const double at = (th - ye) / (2.0 * kKinkStep * fabs(dy));
            const double low = fmin(fmax(0.5 - at, 0.0), 1.0), other = up ? low : 1.0 - low;
            if (dy != 0.0) gr[K + i] = (float)(gr[K + i] + other * ((double)go[K + i] - (double)gr[K + i]));
        }
    }
    return nll;
}

// Per site of a batch: at active sites, -log q_a and its gradient with
// respect to the raw spline parameters into g (BF16, [row][16], zero at
// inactive sites and for the unused channels); loss[row] = -log q_a (0 at
// inactive sites).
template <int mu, int K>
__global__ __launch_bounds__(256) void k_flow_nll_grad(const float4* L, const float* prm, uint16_t* g, float* loss, FGeom g4,
                                                       uint32_t B, int par)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= B * g4.V) return;
    const uint32_t b = g4.dV.div(j), s = j - b * g4.V;
    int c[4];
    coords(g4, s, c);
    float gr[kOut];
#pragma unroll
    for (int q = 0; q < kOut; ++q) gr[q] = 0.f;
    float lo = 0.f;
    if (is_active(c, mu, par)) {
        StapleLinks sl;
        load_staple<mu>(sl, L, g4, b, c);
        const float4 U = L[((size_t)b * 4 + mu) * g4.V + s];
        float raw[kOut];
        load_raw(raw, prm, j);
        loads_issued();
        const float4 A = staple_sum(sl);
        const float k = sqrtf(A.x * A.x + A.y * A.y + A.z * A.z + A.w * A.w);
        if (k > 1e-20f) {
            const float ik = 1.f / k;
            const float4 W = qmul(U, make_float4(A.x * ik, A.y * ik, A.z * ik, A.w * ik));
            const double th = atan2((double)sqrtf(W.y * W.y + W.z * W.z + W.w * W.w), (double)W.x);
            lo = (float)nll_grad_link<K>(raw, th, gr);
        }
    }
    loss[j] = lo;
    uint4* o = reinterpret_cast<uint4*>(g) + 2 * (size_t)j;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = f2bf(gr[8 * q + 2 * i]) | (uint32_t)f2bf(gr[8 * q + 2 * i + 1]) << 16;
        o[q] = make_uint4(v[0], v[1], v[2], v[3]);
    }
}

// Weight and bias gradients from x-planes in LDS: dW[n][st * C + ch] = sum over
// rows r of gout[r][n] X[r + st][ch] and db[n] = sum of gout[r][n], as
// v_mfma_f32_16x16x32_bf16 tiles with 32 rows (sites) per step.  Both operands
// run along the rows, so they are read transposed (ds_read_b64_tr_b16: lane l
// of 16 gives the address of columns 4 (l % 4) .. + 3 of row l / 4 and gets
// column l of the four rows), at any stencil offset.  One workgroup of 8
// wavefronts stages three planes of X and its rows of the plane of gout; `segs`
// workgroups share a plane's rows.  Wavefront w takes the offsets (oy, oz, ot) =
// w, w + 8, .. with all three ox, and goes on to further units with the same
// sums; one partial array per workgroup.
// For 16 configurations of 8^3 x 4 (128 planes): 32 -> 16 channels 21 us, 8 ->
// 32 channels 14.5 us, against 240 and 142 us of k_flow_wgrad, whose every operand
// element is a load.  A good half of it is staging (57 kB per workgroup before the
// first read) and the partial arrays (166 kB per workgroup, 42 MB in all, which
// k_flow_sum_parts reads back in 9 us); the matrix instructions take 2.6 us.
constexpr int kGradWaves = 8, kGradOffs = 4;   // 27 offsets over 8 wavefronts
constexpr uint32_t kGradRows = 32;
template <int C, int N>
__global__ __launch_bounds__(64 * kGradWaves) void k_flow_wgrad_plane(const uint16_t* gout, const uint16_t* in, float* part,
                                                                      FGeom g, uint32_t plane, uint32_t segs, uint32_t len,
                                                                      uint32_t units)
{
    constexpr int CT = C == 32 ? 6 : 2, NT = N / 16;   // tiles of 16 columns per offset: 3 x 2 halves, or ox pairs
    constexpr uint32_t BX = 2u * C, BG = 2u * N, K = kStencil * C;
    extern __shared__ uint4 planes[];
    const uint32_t w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const uint32_t row4 = (uint32_t)(lane & 15) >> 2, chunk = (uint32_t)lane & 3u;
    const uint32_t xv = plane * BX / 16u;
    const char* sx = reinterpret_cast<const char*>(planes);
    const char* sg = sx + 3u * plane * BX;
    const int n[4] = {g.n1, g.n2, g.n3, g.n4};
    typedef __attribute__((address_space(3))) s4 ls4;
    auto tr = [&](const char* a) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)a); };
    // rows of 64 bytes: their halves change places every four rows, or the
    // eight rows of half a wavefront would meet in half the banks
    auto swz = [](uint32_t byte, uint32_t stride) { return stride == 64u ? byte ^ ((byte >> 3) & 32u) : byte; };
    auto stage = [&](uint4* dst, const uint4* src, uint32_t nv, uint32_t stride) {
#pragma unroll 2
        for (uint32_t i = threadIdx.x; i < nv; i += 64u * kGradWaves) dst[swz(16u * i, stride) / 16u] = src[i];
    };
    f4 acc[kGradOffs][CT][NT], accb[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        accb[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kGradOffs; ++i)
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[i][c][t] = f4{0.f, 0.f, 0.f, 0.f};
    }
    for (uint32_t un = blockIdx.x; un < units; un += gridDim.x) {
        const uint32_t pl = un / segs, first = (un - pl * segs) * len, last = min(first + len, plane);
        const uint32_t b = pl / (uint32_t)g.n1, x = pl % (uint32_t)g.n1;
        __syncthreads();   // the previous unit has been read
#pragma unroll
        for (int o = 0; o < 3; ++o)
            stage(planes + o * xv, reinterpret_cast<const uint4*>(in) +
                                       ((size_t)b * (uint32_t)g.n1 + (uint32_t)wrap((int)x + o - 1, g.n1)) * xv, xv, BX);
        stage(planes + 3 * xv, reinterpret_cast<const uint4*>(gout + ((size_t)pl * plane + first) * N), (last - first) * BG / 16u,
              BG);
        __syncthreads();
        for (uint32_t r0 = first; r0 < last; r0 += kGradRows) {
            // two groups of 16 rows; a plane of an odd number of them ends in
            // half a step, the other half zero in both operands
            const bool two = r0 + 16u < last;
            uint32_t yo[2][3], zo[2][3], to[2][3];
            s8 a[NT];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t r = r0 + (two ? 16u * h : 0u) + 4u * (uint32_t)q + row4;
                int c[4];
                coords(g, r, c);
#pragma unroll
                for (int o = 0; o < 3; ++o) {
                    yo[h][o] = (uint32_t)wrap(c[1] + o - 1, n[1]) * BX;
                    zo[h][o] = (uint32_t)wrap(c[2] + o - 1, n[2]) * (uint32_t)n[1] * BX;
                    to[h][o] = (uint32_t)wrap(c[3] + o - 1, n[3]) * (uint32_t)(n[1] * n[2]) * BX;
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const s4 v = tr(sg + swz((r - first) * BG + 32u * t + 8u * chunk, BG));
#pragma unroll
                    for (int j = 0; j < 4; ++j) a[t][4 * h + j] = h == 0 || two ? v[j] : (short)0;
                }
            }
            auto pick = [](const uint32_t (&v)[3], uint32_t i) { return i == 0 ? v[0] : (i == 1 ? v[1] : v[2]); };
            s8 bv[2][CT];
            auto issue = [&](int i) {
                const uint32_t m = w + kGradWaves * i;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t row = pick(yo[h], m / 9u) + pick(zo[h], (m / 3u) % 3u) + pick(to[h], m % 3u);
#pragma unroll
                    for (int t = 0; t < CT; ++t) {
                        s4 v;
                        if constexpr (C == 32)
                            v = tr(sx + (uint32_t)(t >> 1) * plane * BX + swz(row + 32u * (t & 1) + 8u * chunk, BX));
                        else
                            v = tr(sx + (uint32_t)(t == 0 ? chunk >> 1 : 2) * plane * BX + row + 8u * (chunk & 1));
#pragma unroll
                        for (int j = 0; j < 4; ++j) bv[i & 1][t][4 * h + j] = h == 0 || two ? v[j] : (short)0;
                    }
                }
            };
            issue(0);
#pragma unroll
            for (int i = 0; i < kGradOffs; ++i) {
                if (i + 1 < kGradOffs && w + kGradWaves * (i + 1) < 27u) issue(i + 1);
                if (w + kGradWaves * i >= 27u) break;   // uniform
#pragma unroll
                for (int t = 0; t < CT; ++t)
#pragma unroll
                    for (int u = 0; u < NT; ++u)
                        acc[i][t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(a[u]), as_bf(bv[i & 1][t]),
                                                                               acc[i][t][u], 0, 0, 0);
            }
            if (w == kGradWaves - 1u) {   // three offsets only: the bias sums, times ones
                s8 one;
#pragma unroll
                for (int j = 0; j < 8; ++j) one[j] = 0x3f80;
#pragma unroll
                for (int u = 0; u < NT; ++u)
                    accb[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(a[u]), as_bf(one), accb[u], 0, 0, 0);
            }
        }
    }
    // lane holds D[4 (lane / 16) + i][lane % 16]: rows are output channels
    float* o = part + (size_t)blockIdx.x * (N * K + N);
#pragma unroll
    for (int i = 0; i < kGradOffs; ++i) {
        const uint32_t m = w + kGradWaves * i;
        if (m >= 27u) break;
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            const int col = lane & 15;
            uint32_t ox, ch;
            if constexpr (C == 32) {
                ox = (uint32_t)t >> 1;
                const int ps = 16 * (t & 1) + col;   // stored position -> channel (hid_pos)
                ch = (uint32_t)(16 * ((ps >> 2) & 1) + 4 * (ps >> 3) + (ps & 3));
            } else {
                ox = t == 0 ? (uint32_t)col >> 3 : 2u;
                ch = (uint32_t)col & 7u;
                if (t == 1 && col >= 8) continue;
            }
            const uint32_t k = (27u * ox + m) * C + ch;
#pragma unroll
            for (int u = 0; u < NT; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[(size_t)(16 * u + 4 * q + e) * K + k] = acc[i][t][u][e];
        }
    }
    if (w == kGradWaves - 1u && (lane & 15) == 0)
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[(size_t)N * K + 16 * u + 4 * q + e] = accb[u][e];
}

// Weight gradient dW[n][k] = sum over rows r of gout[r][n] X[r][k], X the
// stencil (im2col) view of `in` (X[r][st * cin + ch] = in[nbr(r, st)][ch]),
// as v_mfma_f32_16x16x16_bf16 tiles: D[n][k] += A[n][r] B[r][k] with the
// rows r as the reduction dimension.  One wavefront per (16 x 16 tile,
// chunk of `chunk` rows); partial sums to part[chunk_index][n][k].
__global__ __launch_bounds__(256) void k_flow_wgrad(const uint16_t* gout, int cout, const uint16_t* in, int cin,
                                                    float* part, FGeom g, uint32_t B, uint32_t chunk)
{
    const uint32_t wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const int lane = threadIdx.x & 63;
    const int K = kStencil * cin;
    const uint32_t tn = (uint32_t)(K + 15) / 16, tm = (uint32_t)cout / 16;
    const uint32_t R = B * g.V, nchunk = (R + chunk - 1) / chunk;
    if (wave >= tn * tm * nchunk) return;   // whole wavefront
    const uint32_t ch_i = wave / (tn * tm), t = wave % (tn * tm);
    const uint32_t mt = t % tm, nt = t / tm;
    const int m = (int)mt * 16 + (lane & 15);       // A row: output channel
    const int kcol = (int)nt * 16 + (lane & 15);     // B column
    const int st = kcol / cin, ch = kcol % cin;
    const int o[4] = {st / 27 - 1, (st / 9) % 3 - 1, (st / 3) % 3 - 1, st % 3 - 1};
    const int n[4] = {g.n1, g.n2, g.n3, g.n4};
    f4 acc = {0.f, 0.f, 0.f, 0.f};
    const uint32_t r0 = ch_i * chunk, r1 = min(r0 + chunk, R);
    for (uint32_t rb = r0; rb < r1; rb += 16) {
        s4 av = {0, 0, 0, 0}, bv = {0, 0, 0, 0};
        for (int q = 0; q < 4; ++q) {
            const uint32_t r = rb + 4 * (uint32_t)(lane >> 4) + (uint32_t)q;
            if (r >= r1) continue;
            av[q] = (short)gout[(size_t)r * cout + m];
            if (kcol < K) {
                const uint32_t b = r / g.V, s = r % g.V;
                int c[4];
                coords(g, s, c);
                int e[4];
                for (int d = 0; d < 4; ++d) e[d] = wrap(c[d] + o[d], n[d]);
                bv[q] = (short)in[((size_t)b * g.V + site(g, e)) * cin + (cin == kHidden ? hid_pos(ch) : ch)];
            }
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc, 0, 0, 0);
    }
    // lane holds D[4 (lane / 16) + i][lane % 16]: rows are output channels
    for (int i = 0; i < 4; ++i) {
        const int mm = (int)mt * 16 + 4 * (lane >> 4) + i, kk = (int)nt * 16 + (lane & 15);
        if (kk < K) part[((size_t)ch_i * cout + mm) * K + kk] = acc[i];
    }
}

// out[i] = sum over the nchunk partial arrays (fixed order)
__global__ __launch_bounds__(256) void k_flow_sum_parts(const float* __restrict__ part, uint32_t nchunk, uint32_t n,
                                                        float* __restrict__ out)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float a = 0.f;
    uint32_t c = 0;
    for (; c + 16 <= nchunk; c += 16) {
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = part[(size_t)(c + k) * n + i];
#pragma unroll
        for (int k = 0; k < 16; ++k) a += v[k];
    }
    for (; c < nchunk; ++c) a += part[(size_t)c * n + i];
    out[i] = a;
}

// bias gradient: out[c] = sum over rows of gout[r][c] (one workgroup per channel)
__global__ __launch_bounds__(256) void k_flow_colsum(const uint16_t* gout, int cout, uint32_t R, float* out)
{
    __shared__ float red[256];
    float a = 0.f;
    for (uint32_t r = threadIdx.x; r < R; r += 256) a += bf2f(gout[(size_t)r * cout + blockIdx.x]);
    red[threadIdx.x] = a;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

// transposed conv2 weights for the input gradient: entry (c, st * 16 + n) =
// W2[n][(80 - st) * 32 + c] (the stencil point of offset -o)
__global__ void k_flow_w2_transpose(const uint16_t* w2, uint16_t* wt)   // blockIdx.y: the layer
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    w2 += (size_t)blockIdx.y * (kHidden * kStencil * kOut);
    wt += (size_t)blockIdx.y * (kHidden * kStencil * kOut);
    if (i >= (uint32_t)(kHidden * kStencil * kOut)) return;
    const uint32_t c = i / (kStencil * kOut), rest = i % (kStencil * kOut);
    const uint32_t st = rest / kOut, nn = rest % kOut;
    wt[w2t_pos((int)c, (int)rest)] = w2[w2_pos((int)nn, (int)((kStencil - 1 - st) * kHidden + c))];
}

// Adam (Kingma and Ba 2015) on the FP32 parameters, then the device copies
// the flow evaluates with (BF16 weights, FP32 biases) of every layer.
__global__ void k_flow_adam(float* p, const float* gr, float* m, float* v, uint32_t n, float lr, float b1, float b2,
                            float eps, float c1, float c2, float gscale)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = gr[i] * gscale;
    const float mi = b1 * m[i] + (1.f - b1) * gi, vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ void k_flow_unpack_params(const float* p, uint32_t layers, uint16_t* w1, float* b1, uint16_t* w2, float* b2)
{
    const uint64_t per = (uint64_t)kHidden * kStencil * kCin0 + kHidden + (uint64_t)kOut * kStencil * kHidden + kOut;
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= per * layers) return;
    const uint32_t l = (uint32_t)(i / per);
    uint64_t o = i % per;
    const uint64_t n1 = (uint64_t)kHidden * kStencil * kCin0, n2 = (uint64_t)kOut * kStencil * kHidden;
    if (o < n1) { w1[l * kW1Pack + w1_pos((int)(o / (kStencil * kCin0)), (int)(o % (kStencil * kCin0)))] = f2bf(p[i]); return; }
    o -= n1;
    if (o < kHidden) { b1[l * kHidden + o] = p[i]; return; }
    o -= kHidden;
    if (o < n2) { w2[l * n2 + w2_pos((int)(o / (kStencil * kHidden)), (int)(o % (kStencil * kHidden)))] = f2bf(p[i]); return; }
    o -= n2;
    b2[l * kOut + o] = p[i];
}

// per-site sum of (1 - (U_p)_0) over the six plaquettes with corner x
__global__ void k_flow_action_sites(const float4* L, double* out, FGeom g, uint32_t B)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= B * g.V) return;
    const uint32_t b = g.dV.div(j), s = j - b * g.V;
    int c[4];
    coords(g, s, c);
    double acc = 0.0;
    for (int nu = 0; nu < 4; ++nu)
        for (int rho = nu + 1; rho < 4; ++rho) acc += 1.0 - (double)plaq0(L, g, b, nu, rho, c);
    out[j] = acc;
}

// out[b] = sum of in[b * n + i] (one workgroup per row, fixed order)
template <typename T>
__global__ __launch_bounds__(256) void k_flow_rowsum(const T* in, uint32_t n, double* out)
{
    __shared__ double red[256];
    const uint32_t b = blockIdx.x;
    double acc = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += 256) acc += (double)in[(size_t)b * n + i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[b] = red[0];
}

int err(int code, const std::string& m) { return qcdhip::set_error(code, m.c_str()); }

}  // namespace

struct qcd_flow {
    qcd_flow_desc d;
    FGeom g;
    size_t nparam = 0;
    float* staged = nullptr;   // parameters as uploaded, FP32
    std::vector<float> host_params;
    uint16_t* w1 = nullptr;    // [layers][32][81 * 8]
    float* b1 = nullptr;       // [layers][32]
    uint16_t* w2 = nullptr;    // [layers][16][81 * 32]
    float* b2 = nullptr;       // [layers][16]
    float4* links = nullptr;   // [max_batch][4][V]
    uint16_t* feat = nullptr;  // [max_batch * V][8]
    uint16_t* hid = nullptr;   // [max_batch * V][32]
    float* prm = nullptr;      // [max_batch * V][16]
    float* logj = nullptr;     // [max_batch * V]
    double* act = nullptr;     // [max_batch * V]
    double* sums = nullptr;    // [2][max_batch]
    // learned sweeps, on the device so that a recorded graph replays them
    // with successive keys: [0] links accepted, [1] sweeps run, [2] the
    // current sweep's seed
    unsigned long long* imh = nullptr;
    // training (allocated by the first qcd_flow_train_step)
    float* tp = nullptr;        // FP32 parameters, the flat layout of qcd_flow_set_params
    float* tgrad = nullptr;     // their gradient
    float* tm = nullptr;        // Adam moments
    float* tv = nullptr;
    uint16_t* tg = nullptr;     // d loss / d spline parameters [max_batch * V][16] (BF16)
    uint16_t* tdpre = nullptr;  // d loss / d pre-activation (BF16)
    float* tloss = nullptr;     // -log q_a per site
    uint16_t* tw2t = nullptr;   // transposed conv2 weights, every layer
    float* tpart = nullptr;     // weight-gradient partial sums
    float* tzero = nullptr;     // zero bias of the transposed convolution
    double* tsums = nullptr;    // per layer and configuration loss
    int tstep = 0;
    bool host_stale = false;    // host_params behind tp
    hipStream_t stream = nullptr;
};

namespace {

constexpr size_t kW1 = (size_t)kHidden * kStencil * kCin0;
constexpr size_t kW2 = (size_t)kOut * kStencil * kHidden;
constexpr size_t kLayerParams = kW1 + kHidden + kW2 + kOut;

#define FCHK(x)                                                                                         \
    do {                                                                                                \
        hipError_t e_ = (x);                                                                            \
        if (e_ != hipSuccess) return err(QCD_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Calls f with the direction as a compile-time constant.
template <typename Fn> void with_mu(int mu, Fn f)
{
    switch (mu) {
        case 0: f(std::integral_constant<int, 0>{}); break;
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        default: f(std::integral_constant<int, 3>{}); break;
    }
}

// The same with the number of spline bins.
template <typename Fn> void with_mu_bins(int mu, int bins, Fn f)
{
    with_mu(mu, [&](auto m) {
        switch (bins) {
            case 1: f(m, std::integral_constant<int, 1>{}); break;
            case 2: f(m, std::integral_constant<int, 2>{}); break;
            case 3: f(m, std::integral_constant<int, 3>{}); break;
            case 4: f(m, std::integral_constant<int, 4>{}); break;
            default: f(m, std::integral_constant<int, kMaxBins>{}); break;
        }
    });
}

// Workgroup of the one-thread-per-site kernels: few sites go to as many CUs
// as there are wavefronts.
dim3 site_block(uint32_t n) { return dim3(n <= 65536u ? 64u : 256u); }
dim3 site_grid(uint32_t n) { return dim3((n + site_block(n).x - 1) / site_block(n).x); }

// Spline parameters (F->prm) of layer l from the features in F->feat.
void conditioner(qcd_flow* F, int l, uint32_t rows, hipStream_t st)
{
    launch_conv<kCin0, CONV_TANH>(F->feat, F->w1 + l * kW1Pack, F->b1 + l * kHidden, nullptr, F->hid, nullptr, F->g, rows, st);
    launch_conv<kHidden, CONV_RAW>(F->hid, F->w2 + l * kW2, F->b2 + l * kOut, nullptr, nullptr, F->prm, F->g, rows, st);
}

int run_layers(qcd_flow* F, uint32_t B, bool inverse)
{
    const FGeom g = F->g;
    const uint32_t n = B * g.V;
    FCHK(hipMemsetAsync(F->logj, 0, sizeof(float) * n, F->stream));
    for (int step = 0; step < F->d.layers; ++step) {
        const int l = inverse ? F->d.layers - 1 - step : step;
        const int mu = l % 4, par = (l / 4) % 2;
        with_mu(mu, [&](auto m) {
            hipLaunchKernelGGL(k_flow_features<decltype(m)::value>, site_grid(n), site_block(n), 0, F->stream, F->links,
                               F->feat, g, B, par);
        });
        conditioner(F, l, n, F->stream);
        with_mu_bins(mu, F->d.bins, [&](auto m, auto k) {
            hipLaunchKernelGGL((k_flow_couple<decltype(m)::value, decltype(k)::value>), site_grid(n), site_block(n), 0,
                               F->stream, F->links, F->prm, F->logj, g, B, par, inverse ? 1 : 0);
        });
    }
    FCHK(hipGetLastError());
    return QCD_OK;
}

// per-site action terms of the configurations now in F->links
int action_sites(qcd_flow* F, uint32_t B)
{
    const uint32_t n = B * F->g.V, nb = (n + 255) / 256;
    hipLaunchKernelGGL(k_flow_action_sites, dim3(nb), dim3(256), 0, F->stream, F->links, F->act, F->g, B);
    FCHK(hipGetLastError());
    return QCD_OK;
}

// log q from the accumulated log J, the action from the per-site terms
int finish(qcd_flow* F, uint32_t B, double beta, double* logq, double* action)
{
    const FGeom g = F->g;
    hipLaunchKernelGGL((k_flow_rowsum<float>), dim3(B), dim3(256), 0, F->stream, F->logj, g.V, F->sums);
    hipLaunchKernelGGL((k_flow_rowsum<double>), dim3(B), dim3(256), 0, F->stream, F->act, g.V, F->sums + F->d.max_batch);
    FCHK(hipGetLastError());
    std::vector<double> h(2 * (size_t)F->d.max_batch);
    FCHK(hipMemcpyAsync(h.data(), F->sums, sizeof(double) * h.size(), hipMemcpyDeviceToHost, F->stream));
    FCHK(hipStreamSynchronize(F->stream));
    for (uint32_t b = 0; b < B; ++b) {
        if (logq) logq[b] = -h[b];
        if (action) action[b] = beta * h[F->d.max_batch + b];
    }
    return QCD_OK;
}

// The training buffers; all are there or none.
void free_training(qcd_flow* F)
{
    auto drop = [](auto*& q) {
        (void)hipFree(q);
        q = nullptr;
    };
    drop(F->tp);
    drop(F->tgrad);
    drop(F->tm);
    drop(F->tv);
    drop(F->tg);
    drop(F->tdpre);
    drop(F->tloss);
    drop(F->tw2t);
    drop(F->tpart);
    drop(F->tzero);
    drop(F->tsums);
}

int check_batch(const qcd_flow* F, int batch)
{
    if (batch < 1 || batch > F->d.max_batch)
        return err(QCD_E_ARG, "batch " + std::to_string(batch) + " outside 1.." + std::to_string(F->d.max_batch));
    if (F->nparam == 0 || F->host_params.empty()) return err(QCD_E_STATE, "flow parameters not set");
    return QCD_OK;
}

}  // namespace

extern "C" {

int qcd_flow_create(const qcd_flow_desc* desc, qcd_flow** out)
{
    if (!desc || !out) return err(QCD_E_ARG, "null argument");
    const qcd_flow_desc d = *desc;
    for (int k = 0; k < 4; ++k)
        if (d.n[k] < 2) return err(QCD_E_ARG, "flow lattice extents must be >= 2");
    if (d.layers < 1 || d.layers > 64) return err(QCD_E_ARG, "layers must be 1..64");
    if (d.hidden != kHidden) return err(QCD_E_UNSUPPORTED, "hidden channels must be 32");
    if (d.bins < 1 || d.bins > kMaxBins) return err(QCD_E_ARG, "bins must be 1..5");
    if (d.max_batch < 1) return err(QCD_E_ARG, "max_batch must be >= 1");
    const uint64_t V = (uint64_t)d.n[0] * d.n[1] * d.n[2] * d.n[3];
    if (V % 16) return err(QCD_E_ARG, "the flow needs a site count divisible by 16");
    if (V * (uint64_t)d.max_batch > (1ull << 26)) return err(QCD_E_ARG, "max_batch x sites above 2^26");
    qcd_flow* F = new qcd_flow();
    F->d = d;
    F->g = FGeom{d.n[0], d.n[1], d.n[2], d.n[3], (uint32_t)V, qcd::make_fastdiv((uint32_t)d.n[1]),
                 qcd::make_fastdiv((uint32_t)d.n[2]), qcd::make_fastdiv((uint32_t)d.n[3]), qcd::make_fastdiv((uint32_t)V)};
    F->nparam = kLayerParams * (size_t)d.layers;
    const size_t n = V * (size_t)d.max_batch;
    bool ok = hipStreamCreateWithFlags(&F->stream, hipStreamNonBlocking) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->w1, sizeof(uint16_t) * kW1Pack * d.layers) == hipSuccess;
    // Cleared (the padded k, the counts) on the stream that packs the weights, which
    // is not ordered with the null stream; qcd_flow_set_params, which everything else
    // needs first, waits for it.
    ok = ok && hipMemsetAsync(F->w1, 0, sizeof(uint16_t) * kW1Pack * d.layers, F->stream) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->staged, sizeof(float) * F->nparam) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->b1, sizeof(float) * kHidden * d.layers) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->w2, sizeof(uint16_t) * kW2 * d.layers) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->b2, sizeof(float) * kOut * d.layers) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->links, sizeof(float4) * 4 * n) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->feat, sizeof(uint16_t) * kCin0 * n) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->hid, sizeof(uint16_t) * kHidden * n) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->prm, sizeof(float) * kOut * n) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->logj, sizeof(float) * n) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->act, sizeof(double) * n) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->sums, sizeof(double) * 2 * d.max_batch) == hipSuccess;
    ok = ok && hipMalloc((void**)&F->imh, 3 * sizeof(unsigned long long)) == hipSuccess;
    ok = ok && hipMemsetAsync(F->imh, 0, 3 * sizeof(unsigned long long), F->stream) == hipSuccess;
    if (!ok) {
        qcd_flow_destroy(F);
        return err(QCD_E_NOMEM, "flow buffers");
    }
    *out = F;
    return QCD_OK;
}

int qcd_flow_destroy(qcd_flow* F)
{
    if (!F) return QCD_OK;
    if (F->stream) (void)hipStreamSynchronize(F->stream);
    (void)hipFree(F->w1);
    (void)hipFree(F->staged);
    (void)hipFree(F->b1);
    (void)hipFree(F->w2);
    (void)hipFree(F->b2);
    (void)hipFree(F->links);
    (void)hipFree(F->feat);
    (void)hipFree(F->hid);
    (void)hipFree(F->prm);
    (void)hipFree(F->logj);
    (void)hipFree(F->act);
    (void)hipFree(F->sums);
    (void)hipFree(F->imh);
    free_training(F);
    if (F->stream) (void)hipStreamDestroy(F->stream);
    delete F;
    return QCD_OK;
}

int qcd_flow_param_count(const qcd_flow* F, size_t* n)
{
    if (!F || !n) return err(QCD_E_ARG, "null argument");
    *n = F->nparam;
    return QCD_OK;
}

int qcd_flow_set_params(qcd_flow* F, const float* p, size_t n)
{
    if (!F || !p) return err(QCD_E_ARG, "null argument");
    if (n != F->nparam) return err(QCD_E_ARG, "expected " + std::to_string(F->nparam) + " parameters, got " + std::to_string(n));
    // Uploaded as they are; the device makes the BF16 operand orders.  A copy on
    // the flow's own stream takes several times as long where the array is new
    // (among 4 flows of 16 configurations 0.82 ms, so 0.15).
    FCHK(hipMemcpy(F->staged, p, sizeof(float) * n, hipMemcpyHostToDevice));
    FCHK(hipStreamSynchronize(nullptr));   // it is there before the flow's stream, which does not wait for this one
    hipLaunchKernelGGL(k_flow_unpack_params, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, F->stream,
                       (const float*)F->staged, (uint32_t)F->d.layers, F->w1, F->b1, F->w2, F->b2);
    FCHK(hipGetLastError());
    if (F->tp) {   // training continues from these parameters, fresh moments
        FCHK(hipMemcpyAsync(F->tp, F->staged, sizeof(float) * n, hipMemcpyDeviceToDevice, F->stream));
        FCHK(hipMemsetAsync(F->tm, 0, sizeof(float) * n, F->stream));
        FCHK(hipMemsetAsync(F->tv, 0, sizeof(float) * n, F->stream));
        F->tstep = 0;
    }
    FCHK(hipStreamSynchronize(F->stream));
    F->host_params.assign(p, p + n);
    F->host_stale = false;
    return QCD_OK;
}

int qcd_flow_sample(qcd_flow* F, unsigned long long seed, int batch, double beta, float* links, double* logq,
                    double* action)
{
    if (!F || !links) return err(QCD_E_ARG, "null argument");
    int rc = check_batch(F, batch);
    if (rc) return rc;
    const uint64_t n = (uint64_t)batch * 4 * F->g.V;
    hipLaunchKernelGGL(k_flow_haar, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, F->stream, F->links, n,
                       (uint64_t)seed);
    if ((rc = run_layers(F, (uint32_t)batch, false))) return rc;
    if ((rc = action_sites(F, (uint32_t)batch))) return rc;   // of the proposals
    if ((rc = finish(F, (uint32_t)batch, beta, logq, action))) return rc;
    FCHK(hipMemcpy(links, F->links, sizeof(float4) * n, hipMemcpyDeviceToHost));
    return QCD_OK;
}

int qcd_flow_evaluate(qcd_flow* F, const float* links, int batch, double beta, double* logq, double* action)
{
    if (!F || !links) return err(QCD_E_ARG, "null argument");
    int rc = check_batch(F, batch);
    if (rc) return rc;
    const uint64_t n = (uint64_t)batch * 4 * F->g.V;
    FCHK(hipMemcpyAsync(F->links, links, sizeof(float4) * n, hipMemcpyHostToDevice, F->stream));
    if ((rc = action_sites(F, (uint32_t)batch))) return rc;   // of the given configurations, before the inverse
    if ((rc = run_layers(F, (uint32_t)batch, true))) return rc;
    return finish(F, (uint32_t)batch, beta, logq, action);
}

namespace {
int imh_sweep(qcd_flow* F, qcd_lattice* lat, unsigned long long seed, int mode, double beta)
{
    if (!F || !lat) return err(QCD_E_ARG, "null argument");
    if (F->nparam == 0 || F->host_params.empty()) return err(QCD_E_STATE, "flow parameters not set");
    int n[4];
    int rc = qcdhip::lattice_dims(lat, n);
    if (rc) return rc;
    for (int k = 0; k < 4; ++k)
        if (n[k] != F->d.n[k]) return err(QCD_E_ARG, "the lattice and the flow have different extents");
    hipStream_t st = nullptr;
    if ((rc = qcdhip::su2_quats(lat, F->links, true, &st))) return rc;   // the lattice's stream from here on
    hipLaunchKernelGGL(k_flow_imh_key, dim3(1), dim3(64), 0, st, F->imh, seed, mode);
    const FGeom g = F->g;
    for (int l = 0; l < F->d.layers; ++l) {
        const int mu = l % 4, par = (l / 4) % 2;
        with_mu(mu, [&](auto m) {
            hipLaunchKernelGGL(k_flow_features<decltype(m)::value>, site_grid(g.V), site_block(g.V), 0, st, F->links, F->feat,
                               g, 1u, par);
        });
        conditioner(F, l, g.V, st);
        with_mu_bins(mu, F->d.bins, [&](auto m, auto k) {
            hipLaunchKernelGGL((k_flow_imh_couple<decltype(m)::value, decltype(k)::value>), site_grid(g.V), site_block(g.V),
                               0, st, F->links, F->prm, g, par, (float)beta, ((uint64_t)l + 1) * 0xD1B54A32D192ED03ull,
                               F->imh);
        });
    }
    FCHK(hipGetLastError());
    return qcdhip::su2_quats(lat, F->links, false, nullptr);
}
}  // namespace

int qcd_flow_imh_sweep(qcd_flow* F, qcd_lattice* lat, unsigned long long seed, double beta)
{
    return imh_sweep(F, lat, seed, 2, beta);
}

int qcd_flow_imh_sweep_next(qcd_flow* F, qcd_lattice* lat, double beta)
{
    return imh_sweep(F, lat, 0ull, 1, beta);
}

int qcd_flow_imh_seed(qcd_flow* F, unsigned long long seed)
{
    if (!F) return err(QCD_E_ARG, "null flow");
    if (!F->imh) return err(QCD_E_STATE, "flow not set up");
    hipLaunchKernelGGL(k_flow_imh_key, dim3(1), dim3(64), 0, F->stream, F->imh, seed, 0);
    FCHK(hipStreamSynchronize(F->stream));
    return QCD_OK;
}

}  // extern "C"

namespace {

// The layer-local loss of `batch` configurations (uploaded from `links`)
// and its gradient with respect to every parameter, into F->tgrad (sums
// over the batch); *loss = the loss per configuration.
int train_grad(qcd_flow* F, const float* links, int batch, double* loss)
{
    if (!F || !links) return err(QCD_E_ARG, "null argument");
    int rc = check_batch(F, batch);
    if (rc) return rc;
    const FGeom g = F->g;
    const uint32_t B = (uint32_t)batch, R = B * g.V;
    const size_t nmax = (size_t)F->d.max_batch * g.V;
    // weight gradients from x-planes in LDS where those fit, one partial
    // array per workgroup; else from chunks of rows
    constexpr uint32_t kChunk = 512, kGradGroups = 256;   // one workgroup per CU; 128 cost 15 % at 64 configurations
    const uint32_t plane = g.V / (uint32_t)g.n1, lds2 = plane * (3u * 2 * kHidden + 2 * kOut),
                   lds1 = plane * (3u * 2 * kCin0 + 2 * kHidden);
    const bool by_plane = plane % 16 == 0 && lds2 <= 64u * 1024u;
    // segments of a plane, a multiple of kGradRows rows each
    auto seg_len = [&](uint32_t nplanes) {
        const uint32_t steps = (plane + kGradRows - 1) / kGradRows, segs = std::clamp(kGradGroups / nplanes, 1u, steps);
        return (steps + segs - 1) / segs * kGradRows;
    };
    const size_t nchunk_max = by_plane ? std::min<size_t>(kGradGroups, nmax / 16) : (nmax + kChunk - 1) / kChunk;
    const size_t part_max = nchunk_max * (kW2 + kHidden);
    if (!F->tp) {   // first step: training buffers and the FP32 parameters from the host copy
        bool ok = true;
        ok = ok && hipMalloc((void**)&F->tp, sizeof(float) * F->nparam) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tgrad, sizeof(float) * F->nparam) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tm, sizeof(float) * F->nparam) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tv, sizeof(float) * F->nparam) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tg, sizeof(uint16_t) * kOut * nmax) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tdpre, sizeof(uint16_t) * kHidden * nmax) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tloss, sizeof(float) * nmax) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tw2t, sizeof(uint16_t) * kW2 * F->d.layers) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tpart, sizeof(float) * part_max) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tzero, sizeof(float) * kHidden) == hipSuccess;
        ok = ok && hipMalloc((void**)&F->tsums, sizeof(double) * F->d.layers * F->d.max_batch) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            free_training(F);
            return err(QCD_E_NOMEM, "flow training buffers");
        }
        FCHK(hipMemcpyAsync(F->tp, F->host_params.data(), sizeof(float) * F->nparam, hipMemcpyHostToDevice, F->stream));
        FCHK(hipMemsetAsync(F->tm, 0, sizeof(float) * F->nparam, F->stream));
        FCHK(hipMemsetAsync(F->tv, 0, sizeof(float) * F->nparam, F->stream));
        FCHK(hipMemsetAsync(F->tzero, 0, sizeof(float) * kHidden, F->stream));
        F->tstep = 0;
    }
    const uint64_t nl = (uint64_t)B * 4 * g.V;
    FCHK(hipMemcpyAsync(F->links, links, sizeof(float4) * nl, hipMemcpyHostToDevice, F->stream));
    const uint32_t nplanes = R / plane, nchunk = (R + kChunk - 1) / kChunk;
    const uint32_t len = seg_len(nplanes), segs = (plane + len - 1) / len, groups = std::min(nplanes * segs, kGradGroups);
    // dW and db of one convolution, gout [R][N] and its input [R][C], to gw
    // (the bias follows the weights)
    auto weight_grad = [&](auto cc, auto nn, const uint16_t* gout, const uint16_t* in, uint32_t lds, float* gw) {
        constexpr int C = decltype(cc)::value, N = decltype(nn)::value, K = kStencil * C;
        if (by_plane) {
            hipLaunchKernelGGL((k_flow_wgrad_plane<C, N>), dim3(groups), dim3(64 * kGradWaves), lds, F->stream, gout, in,
                               F->tpart, g, plane, segs, len, nplanes * segs);
            const uint32_t n = N * K + N;
            hipLaunchKernelGGL(k_flow_sum_parts, dim3((n + 255) / 256), dim3(256), 0, F->stream, (const float*)F->tpart,
                               groups, n, gw);
            return;
        }
        const uint32_t tiles = (uint32_t)((K + 15) / 16) * (N / 16) * nchunk;
        hipLaunchKernelGGL(k_flow_wgrad, dim3((tiles + 3) / 4), dim3(256), 0, F->stream, gout, N, in, C, F->tpart, g, B,
                           kChunk);
        hipLaunchKernelGGL(k_flow_sum_parts, dim3((N * K + 255) / 256), dim3(256), 0, F->stream, (const float*)F->tpart,
                           nchunk, (uint32_t)(N * K), gw);
        hipLaunchKernelGGL(k_flow_colsum, dim3(N), dim3(256), 0, F->stream, gout, N, R, gw + N * K);
    };
    using Hid = std::integral_constant<int, kHidden>;
    using Out = std::integral_constant<int, kOut>;
    using In0 = std::integral_constant<int, kCin0>;
    hipLaunchKernelGGL(k_flow_w2_transpose, dim3((unsigned)((kW2 + 255) / 256), (unsigned)F->d.layers), dim3(256), 0, F->stream,
                       (const uint16_t*)F->w2, F->tw2t);
    for (int l = 0; l < F->d.layers; ++l) {
        const int mu = l % 4, par = (l / 4) % 2;
        float* gl = F->tgrad + (size_t)l * kLayerParams;   // W1, b1, W2, b2 of layer l
        // forward of the conditioner on the data configurations
        with_mu(mu, [&](auto m) {
            hipLaunchKernelGGL(k_flow_features<decltype(m)::value>, site_grid(R), site_block(R), 0, F->stream, F->links,
                               F->feat, g, B, par);
        });
        conditioner(F, l, R, F->stream);
        // -log q_a and its gradient with respect to the spline parameters
        with_mu_bins(mu, F->d.bins, [&](auto m, auto k) {
            hipLaunchKernelGGL((k_flow_nll_grad<decltype(m)::value, decltype(k)::value>), site_grid(R), site_block(R), 0,
                               F->stream, (const float4*)F->links, F->prm, F->tg, F->tloss, g, B, par);
        });
        hipLaunchKernelGGL((k_flow_rowsum<float>), dim3(B), dim3(256), 0, F->stream, F->tloss, g.V,
                           F->tsums + (size_t)l * F->d.max_batch);
        // conv2: weight and bias gradients, then the gradient before tanh
        // through the transposed convolution
        weight_grad(Hid{}, Out{}, F->tg, F->hid, lds2, gl + kW1 + kHidden);
        launch_conv<kOut, CONV_TANH_BACK>(F->tg, F->tw2t + l * kW2, F->tzero, F->hid, F->tdpre, nullptr, g, R, F->stream);
        // conv1: weight and bias gradients (the features are data: no further gradient)
        weight_grad(In0{}, Hid{}, F->tdpre, F->feat, lds1, gl);
    }
    FCHK(hipGetLastError());
    if (loss) {
        std::vector<double> h((size_t)F->d.layers * F->d.max_batch);
        FCHK(hipMemcpyAsync(h.data(), F->tsums, sizeof(double) * h.size(), hipMemcpyDeviceToHost, F->stream));
        FCHK(hipStreamSynchronize(F->stream));
        double a = 0.0;
        for (int l = 0; l < F->d.layers; ++l)
            for (uint32_t b = 0; b < B; ++b) a += h[(size_t)l * F->d.max_batch + b];
        *loss = a / B;
    }
    return QCD_OK;
}

}  // namespace

extern "C" {

int qcd_flow_train_grad(qcd_flow* F, const float* links, int batch, double* loss, float* grad)
{
    const int rc = train_grad(F, links, batch, loss);
    if (rc) return rc;
    if (grad) {
        FCHK(hipMemcpyAsync(grad, F->tgrad, sizeof(float) * F->nparam, hipMemcpyDeviceToHost, F->stream));
        FCHK(hipStreamSynchronize(F->stream));
    }
    return QCD_OK;
}

int qcd_flow_train_step(qcd_flow* F, const float* links, int batch, float lr, double* loss)
{
    if (!(lr > 0.f)) return err(QCD_E_ARG, "learning rate must be positive");
    const int rc = train_grad(F, links, batch, loss);
    if (rc) return rc;
    const uint32_t B = (uint32_t)batch;
    // Adam on the mean over the batch, then the flow's own copies
    ++F->tstep;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)F->tstep), c2 = 1.f - powf(b2, (float)F->tstep);
    const uint32_t np = (uint32_t)F->nparam;
    hipLaunchKernelGGL(k_flow_adam, dim3((np + 255) / 256), dim3(256), 0, F->stream, F->tp, (const float*)F->tgrad,
                       F->tm, F->tv, np, lr, b1, b2, 1e-8f, c1, c2, 1.f / (float)B);
    hipLaunchKernelGGL(k_flow_unpack_params, dim3((np + 255) / 256), dim3(256), 0, F->stream, (const float*)F->tp,
                       (uint32_t)F->d.layers, F->w1, F->b1, F->w2, F->b2);
    FCHK(hipGetLastError());
    F->host_stale = true;
    return QCD_OK;
}

int qcd_flow_get_params(qcd_flow* F, float* p, size_t n)
{
    if (!F || !p) return err(QCD_E_ARG, "null argument");
    if (n != F->nparam) return err(QCD_E_ARG, "expected " + std::to_string(F->nparam) + " parameters, got " + std::to_string(n));
    if (F->host_stale) {
        FCHK(hipStreamSynchronize(F->stream));
        FCHK(hipMemcpy(F->host_params.data(), F->tp, sizeof(float) * F->nparam, hipMemcpyDeviceToHost));
        F->host_stale = false;
    }
    if (F->host_params.size() != n) return err(QCD_E_STATE, "flow parameters not set");
    memcpy(p, F->host_params.data(), sizeof(float) * n);
    return QCD_OK;
}

int qcd_flow_imh_counts(qcd_flow* F, unsigned long long* accepted, unsigned long long* proposed, int reset)
{
    if (!F) return err(QCD_E_ARG, "null flow");
    FCHK(hipDeviceSynchronize());
    unsigned long long a[2] = {0, 0};
    FCHK(hipMemcpy(a, F->imh, sizeof(a), hipMemcpyDeviceToHost));
    if (accepted) *accepted = a[0];
    if (proposed) *proposed = a[1] * (unsigned long long)F->d.layers * (F->g.V / 2);   // every layer proposes V/2 links
    if (reset) {   // the seed stays
        FCHK(hipMemsetAsync(F->imh, 0, 2 * sizeof(unsigned long long), F->stream));
        FCHK(hipStreamSynchronize(F->stream));
    }
    return QCD_OK;
}

}  // extern "C"
