// qcd_ranlux.hpp -- RANLUX produce() with the blocks of a stream generated in
// parallel.
//
// A stream's numbers come in blocks of 24 with P numbers skipped between two
// blocks (P by luxury level).  Stepping through the skips one number at a
// time is a chain of some 2700 dependent instructions per produce(), 21 us on
// the smallest lattice (k_ranlux_produce).  The recursion x_n = x_{n-10} - x_{n-24} - c_{n-1} (mod b = 2^24, borrow
// c) is a linear congruential generator (Marsaglia and Zaman 1991, Luescher
// 1994): with m = b^24 - b^10 + 1 and
//     X_n = sum_{j<24} x_{n-24+j} b^j - sum_{j<10} x_{n-10+j} b^j + c_{n-1}
// one step is b X_{n+1} = X_n + x_n m, so X_{n+N} = b^-N X_n mod m.  From
// X = X_{n+N-24} the ring (and borrow) after N steps is 24 steps of the same
// recursion on the digits of X with nothing before them:
//     r_j = (j >= 10 ? r_{j-10} : 0) - X_j - borrow.
// So a block's start is one multiplication by a fixed 576-bit constant away,
// and as X is linear in the ring's bytes and the borrow, that product is a
// matrix of 72 signed base-256 digits by 73 bytes per stream: v_mfma_i32 on
// int8 operands, exact in 32 bits (|sum| < 2^22).  One wavefront per block and
// 64 streams: 40 matrix instructions, the carries of the digit sums, 24 steps.
// (Both halves of the product use the 16x16x64 form: a 16x16x32 accumulating
// on its result came out wrong.)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "qcd_device.hpp"

namespace qcd {

constexpr int kRlTasks = 24;       // blocks with a table: four produce() of 33 quads
constexpr int kRlSpan = 12;        // blocks a single produce() may span on this path
constexpr int kRlAhead = 4;        // produce() of one launch of rl_ahead
constexpr int kRlWaves = 8;        // wavefronts of a workgroup: 60 kB of LDS
constexpr int kRlTaskVec = 660;    // 16-byte entries of one block's table: 2 x 320 + 20
constexpr int kRlIn = 28, kRlOut = 26;   // words per stream in LDS

typedef int rl_i4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- host tables
// Integers mod m in 24 limbs of 24 bits.
struct RlBig {
    uint32_t x[24];
};
// x + top 2^576 mod m for limbs that may exceed 24 bits or be negative
// (2^576 = b^10 - 1 mod m), canonical.
inline RlBig rl_norm(const int64_t (&v)[24], int64_t top)
{
    int64_t w[24];
    for (int i = 0; i < 24; ++i) w[i] = v[i];
    while (true) {
        w[10] += top;
        w[0] -= top;
        int64_t c = 0;
        for (int i = 0; i < 24; ++i) {
            const int64_t t = w[i] + c;
            w[i] = t & 0xffffff;
            c = t >> 24;
        }
        top = c;
        if (!top) break;
    }
    bool ge = true;   // >= m = (1, 0 x 9, 0xffffff x 14)
    for (int i = 10; i < 24; ++i) ge = ge && w[i] == 0xffffff;
    bool low = false;
    for (int i = 0; i < 10; ++i) low = low || w[i] != 0;
    if (ge && low) {
        int64_t z[24] = {};
        for (int i = 0; i < 10; ++i) z[i] = w[i];
        z[0] -= 1;
        return rl_norm(z, 0);
    }
    RlBig r;
    for (int i = 0; i < 24; ++i) r.x[i] = (uint32_t)w[i];
    return r;
}
inline RlBig rl_shift(const RlBig& a, int bits)   // a 2^bits, bits <= 24
{
    int64_t v[24];
    for (int i = 0; i < 24; ++i) v[i] = (int64_t)a.x[i] << bits;
    return rl_norm(v, 0);
}
inline RlBig rl_sub(const RlBig& a, const RlBig& b)
{
    int64_t v[24];
    for (int i = 0; i < 24; ++i) v[i] = (int64_t)a.x[i] - (int64_t)b.x[i];
    return rl_norm(v, 0);
}
inline RlBig rl_divb(const RlBig& a)   // a / b: (a + q m) / b with q = -a mod b, as m = 1 mod b
{
    const int64_t q = (0x1000000 - a.x[0]) & 0xffffff;
    int64_t v[24], c = ((int64_t)a.x[0] + q) >> 24;
    for (int i = 1; i < 24; ++i) v[i - 1] = a.x[i];
    v[23] = q;
    v[0] += c;
    v[9] -= q;
    return rl_norm(v, 0);
}

constexpr int rl_skip_count(int lux) { return lux == 0 ? 24 : (lux == 1 ? 48 : (lux == 2 ? 97 : (lux == 3 ? 223 : 389))); }

// The matrices of blocks t = 1 .. kRlTasks after a block's end, in the
// operand order of the kernel: row tile rt, row r holds digit
// e = 4 rt + r % 4 of the six limbs of lane group r / 4 (e = 3 limb + byte).
inline const std::vector<uint32_t>& rl_tables(int lux)
{
    static std::vector<uint32_t> tab[5];
    static std::once_flag once[5];
    std::call_once(once[lux], [lux] {
        const int P = rl_skip_count(lux);
        std::vector<uint32_t>& out = tab[lux];
        out.assign((size_t)kRlTasks * kRlTaskVec * 4, 0u);
        RlBig A{};
        A.x[0] = 1;
        int at = 0;   // A = b^-at
        for (int t = 1; t <= kRlTasks; ++t) {
            const int want = t * P + (t - 1) * 24 - 24;
            for (; at < want; ++at) A = rl_divb(A);
            // col[4 w + e]: signed base-256 digits of the factor of byte e of ring word w (limb 23 - w);
            // byte 3 of word 0 carries the borrow
            std::vector<int8_t> col((size_t)96 * 72, 0);
            auto digits = [&](const RlBig& v, int8_t* d) {
                int z[72];
                for (int i = 0; i < 72; ++i) z[i] = (int)((v.x[i / 3] >> (8 * (i % 3))) & 255u);
                while (true) {
                    int c = 0;
                    for (int i = 0; i < 72; ++i) {
                        const int y = z[i] + c;
                        c = (y + 128) >> 8;
                        z[i] = y - 256 * c;
                    }
                    if (!c) break;
                    z[30] += c;
                    z[0] -= c;
                }
                for (int i = 0; i < 72; ++i) d[i] = (int8_t)z[i];
            };
            RlBig Ab[24];
            Ab[0] = A;
            for (int j = 1; j < 24; ++j) Ab[j] = rl_shift(Ab[j - 1], 24);
            for (int j = 0; j < 24; ++j) {
                RlBig v = j >= 14 ? rl_sub(Ab[j], Ab[j - 14]) : Ab[j];
                for (int e = 0; e < 3; ++e) {
                    digits(v, &col[(size_t)(4 * (23 - j) + e) * 72]);
                    v = rl_shift(v, 8);
                }
            }
            digits(A, &col[(size_t)3 * 72]);
            uint32_t* o = &out[(size_t)(t - 1) * kRlTaskVec * 4];
            auto digit_of = [](int rt, int r) {   // -1: unused row
                const int e = 4 * rt + r % 4;
                return e < 18 ? 18 * (r / 4) + e : -1;
            };
            for (int rt = 0; rt < 5; ++rt)
                for (int lane = 0; lane < 64; ++lane) {
                    const int dg = digit_of(rt, lane % 16), kg = lane / 16;
                    if (dg < 0) continue;
                    for (int b = 0; b < 16; ++b)
                        o[4 * (64 * rt + lane) + b / 4] |= (uint32_t)(uint8_t)col[(size_t)(16 * kg + b) * 72 + dg] << (8 * (b % 4));
                    for (int b = 0; b < 16 && kg < 2; ++b)
                        o[4 * (320 + 64 * rt + lane) + b / 4] |=
                            (uint32_t)(uint8_t)col[(size_t)(64 + 16 * kg + b) * 72 + dg] << (8 * (b % 4));
                }
            // the ring's bytes enter as byte - 128: what that takes off every digit
            for (int rt = 0; rt < 5; ++rt)
                for (int g = 0; g < 4; ++g)
                    for (int i = 0; i < 4; ++i) {
                        const int dg = digit_of(rt, 4 * g + i);
                        int s = 0;
                        if (dg >= 0)
                            for (int k = 0; k < 96; ++k)
                                if (k % 4 < 3) s += col[(size_t)k * 72 + dg];
                        o[4 * 640 + 4 * (4 * rt + g) + i] = (uint32_t)(128 * s);
                    }
        }
    });
    return tab[lux];
}

// ---------------------------------------------------------------- device
// One block's table in this lane's registers.
struct RlTab {
    rl_i4 a0[5], a1[5], corr[5];
};
__device__ __forceinline__ void rl_load(RlTab& t, const uint4* tab)
{
    const int lane = threadIdx.x & 63;
    const rl_i4* v = reinterpret_cast<const rl_i4*>(tab);
#pragma unroll
    for (int rt = 0; rt < 5; ++rt) {
        t.a0[rt] = v[64 * rt + lane];
        t.a1[rt] = v[320 + 64 * rt + lane];
        t.corr[rt] = v[640 + 4 * rt + (lane >> 4)];
    }
}

// Ring and borrow of the wavefront's 64 streams at the start of the block of
// table t.  in: the rings at a block's end as words (kRlIn per stream, bytes
// biased by 128, the borrow in byte 3 of word 0); tmp: kRlOut words per stream
// for this wavefront.
__device__ __forceinline__ void rl_jump(const RlTab& t, const uint32_t* in, uint32_t* tmp, uint32_t (&s)[24],
                                        uint32_t& carry)
{
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
        const uint32_t* src = in + (16 * ct + n) * kRlIn;
        const rl_i4 b0 = *reinterpret_cast<const rl_i4*>(src + 4 * g);
        const rl_i4 b1 = *reinterpret_cast<const rl_i4*>(src + 16 + 4 * (g & 1));   // groups 2, 3: zero factors
        int o[20];
#pragma unroll
        for (int rt = 0; rt < 5; ++rt) {
            rl_i4 acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(t.a0[rt], b0, t.corr[rt], 0, 0, 0);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(t.a1[rt], b1, acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[4 * rt + i] = acc[i];
        }
        // this lane's six limbs (6 g .. 6 g + 5) of stream 16 ct + n
        int limb[6], c = 0;
#pragma unroll
        for (int l = 0; l < 6; ++l) {
            const int u = (o[3 * l + 1] << 8) + (o[3 * l] + c);
            const int w = o[3 * l + 2] + (u >> 16);
            limb[l] = (u & 0xffff) | ((w & 0xff) << 16);
            c = w >> 8;
        }
        // carries between the four lanes of a stream, the top one folded with
        // 2^576 = b^10 - 1 (limb 10 is limb 4 of group 1).  What is left
        // then, -1, 0 or 1 per lane and 0 but for one state in 2^100, goes
        // along with the limbs.
        const int below = __shfl(c, (lane + 48) & 63, 64), top = __shfl(c, n + 48, 64);
        c = g == 0 ? -top : below;
#pragma unroll
        for (int l = 0; l < 6; ++l) {
            const int v = limb[l] + c + ((l == 4 && g == 1) ? top : 0);
            limb[l] = v & 0xffffff;
            c = v >> 24;
        }
        uint32_t* dst = tmp + (16 * ct + n) * kRlOut;
#pragma unroll
        for (int l = 0; l < 6; l += 2)
            *reinterpret_cast<uint2*>(dst + 6 * g + l) = make_uint2((uint32_t)limb[l], (uint32_t)limb[l + 1]);
        reinterpret_cast<int8_t*>(dst + 24)[g] = (int8_t)c;
    }
    // A wavefront's LDS operations run in order; the fences keep the compiler
    // from moving a lane's reads above another lane's writes.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    uint32_t X[24];
#pragma unroll
    for (int l = 0; l < 24; l += 2) {
        const uint2 v = *reinterpret_cast<const uint2*>(tmp + lane * kRlOut + l);
        X[l] = v.x;
        X[l + 1] = v.y;
    }
    const uint32_t left = tmp[lane * kRlOut + 24];
    if (left) {   // one carry at a time: at most two rounds, the top one is 0 after the second
        int in6 = (int8_t)left, in12 = (int8_t)(left >> 8), in18 = (int8_t)(left >> 16), top = (int8_t)(left >> 24);
        for (int round = 0; round < 4 && (in6 | in12 | in18 | top); ++round) {
            int c = -top;
#pragma unroll
            for (int l = 0; l < 24; ++l) {
                const int v = (int)X[l] + c + (l == 6 ? in6 : (l == 10 ? top : (l == 12 ? in12 : (l == 18 ? in18 : 0))));
                X[l] = (uint32_t)v & 0xffffffu;
                c = v >> 24;
            }
            top = c;
            in6 = in12 = in18 = 0;
        }
    }
    if (X[23] == 0xffffffu) {   // X in [m, b^24): canonical X - m (one state in 2^336)
        uint32_t hi = 0xffffffu, lo = 0u;
#pragma unroll
        for (int l = 10; l < 24; ++l) hi &= X[l];
#pragma unroll
        for (int l = 0; l < 10; ++l) lo |= X[l];
        if (hi == 0xffffffu && lo) {
            uint32_t bor = 1u;
#pragma unroll
            for (int l = 0; l < 24; ++l) {
                if (l < 10) {
                    const uint32_t d = X[l] - bor;
                    bor = d >> 31;
                    X[l] = d & 0xffffffu;
                } else {
                    X[l] = 0u;
                }
            }
        }
    }
    // The two states no step leaves: X = 0 is reached from X = 0 and from
    // X = m (every digit b - 1, borrow 1) only.
    uint32_t any = 0u;
#pragma unroll
    for (int l = 0; l < 24; ++l) any |= X[l];
    const bool stuck = any == 0u && (in[lane * kRlIn] & 0xffffffu) != 0x808080u;
    carry = 0u;
    uint32_t r[24];
#pragma unroll
    for (int j = 0; j < 24; ++j) {
        uint32_t bor;
        r[j] = __builtin_subc(j >= 10 ? r[j - 10] : 0u, X[j], carry, &bor) & 0xffffffu;
        carry = bor;
    }
    if (stuck) carry = 1u;
#pragma unroll
    for (int j = 0; j < 24; ++j) s[23 - j] = stuck ? 0xffffffu : r[j];
}

template <int K> __device__ __forceinline__ void rl_quad_at(uint32_t (&s)[24], uint32_t& carry, bool keep, float4* out)
{
    if (keep) {
        const float4 q = rl_quad<K>(s, carry);
        if (out) *out = q;
    } else {
        (void)rl_swb<23 - 4 * K, (33 - 4 * K) % 24>(s, carry);
        (void)rl_swb<22 - 4 * K, (32 - 4 * K) % 24>(s, carry);
        (void)rl_swb<21 - 4 * K, (31 - 4 * K) % 24>(s, carry);
        (void)rl_swb<20 - 4 * K, (30 - 4 * K) % 24>(s, carry);
    }
}
// Quads k0 .. k1 - 1 of a block, numbered m0 + (k - k0) in the produce(); those
// below `keep` are stored.  k0, k1, m0 and keep are uniform.
__device__ __forceinline__ void rl_block(uint32_t (&s)[24], uint32_t& carry, uint32_t k0, uint32_t k1, uint32_t m0,
                                         uint32_t keep, float4* quads, uint32_t n, uint32_t g, bool valid)
{
    auto slot = [&](uint32_t k) { return valid ? quads + (size_t)(m0 + k - k0) * n + g : nullptr; };
    auto run = [&](auto K) {
        constexpr uint32_t k = decltype(K)::value;
        if (k >= k0 && k < k1) {
            const bool st = m0 + k - k0 < keep;
            rl_quad_at<(int)k>(s, carry, st, st ? slot(k) : nullptr);
        }
    };
    run(std::integral_constant<uint32_t, 0>{});
    run(std::integral_constant<uint32_t, 1>{});
    run(std::integral_constant<uint32_t, 2>{});
    run(std::integral_constant<uint32_t, 3>{});
    run(std::integral_constant<uint32_t, 4>{});
    run(std::integral_constant<uint32_t, 5>{});
}

__device__ __forceinline__ void rl_store(float4* state, uint32_t n, uint32_t g, const uint32_t (&s)[24], uint32_t carry,
                                         uint32_t k)
{
#pragma unroll
    for (int q = 0; q < 6; ++q)
        state[(size_t)q * n + g] = make_float4((float)s[4 * q] * kRlTwom24, (float)s[4 * q + 1] * kRlTwom24,
                                               (float)s[4 * q + 2] * kRlTwom24, (float)s[4 * q + 3] * kRlTwom24);
    state[(size_t)6 * n + g] = make_float4(23.0f, 9.0f, (float)k, carry ? kRlTwom24 : 0.0f);
}

// produce() of `samples` quads for streams 64 unit .. 64 unit + 63, the first
// `keep` of them stored, by the W wavefronts of one workgroup: wavefront 0
// finishes the block the streams stand in and publishes the rings at its end;
// wavefront w < W - 1 then makes block w + 1, the last wavefront the last block
// and the new state (all have read the old one before the barrier).
__device__ __forceinline__ void rl_produce(float4* state, uint32_t n, uint32_t samples, uint32_t keep, float4* quads,
                                           uint32_t unit, const uint4* tab, uint32_t* lds, uint32_t W)
{
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63, g0 = unit * 64u + lane;
    const bool valid = g0 < n;
    const uint32_t g = valid ? g0 : n - 1u;
    const float4 c6 = state[(size_t)6 * n + g];
    const uint32_t k = min((uint32_t)__builtin_amdgcn_readfirstlane((int)c6.z), 6u);
    const uint32_t first = 6u - k;   // quads left in the current block
    const uint32_t nb = samples > first ? (samples - first + 5u) / 6u : 0u;
    const bool last = w == W - 1u;
    const uint32_t t = last ? nb : w + 1u;
    const uint32_t m0 = first + 6u * (t - 1u);
    const bool idle = t == 0u || t > nb || (!last && (t == nb || m0 >= keep));
    RlTab table;   // asked for before the barrier, so that it arrives with the states
    if (!idle) rl_load(table, tab + (size_t)(t - 1u) * kRlTaskVec);
    uint32_t s[24], carry;
    if (w == 0) {
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const float4 v = state[(size_t)q * n + g];
            s[4 * q] = (uint32_t)(v.x * 16777216.0f);
            s[4 * q + 1] = (uint32_t)(v.y * 16777216.0f);
            s[4 * q + 2] = (uint32_t)(v.z * 16777216.0f);
            s[4 * q + 3] = (uint32_t)(v.w * 16777216.0f);
        }
        carry = c6.w > 0.0f ? 1u : 0u;
        const uint32_t k1 = samples < first ? k + samples : 6u;
        rl_block(s, carry, k, k1, 0u, keep, quads, n, g, valid);
        if (nb == 0 && valid) rl_store(state, n, g, s, carry, k1);
        uint32_t* o = lds + lane * kRlIn;
#pragma unroll
        for (int q = 0; q < 6; ++q)
            *reinterpret_cast<uint4*>(o + 4 * q) =
                make_uint4((s[4 * q] ^ 0x808080u) | (q == 0 ? carry << 24 : 0u), s[4 * q + 1] ^ 0x808080u,
                           s[4 * q + 2] ^ 0x808080u, s[4 * q + 3] ^ 0x808080u);
    }
    __syncthreads();
    if (idle) return;
    rl_jump(table, lds, lds + 64 * kRlIn + w * 64u * kRlOut, s, carry);
    const uint32_t k1 = t == nb ? samples - m0 : 6u;
    rl_block(s, carry, 0u, k1, m0, keep, quads, n, g, valid);
    if (last && valid) rl_store(state, n, g, s, carry, k1);
}

// produce() number h of kRlAhead that follow each other, `samples` quads each
// with the first `keep` of every one stored ([h][quad][stream]): every
// workgroup starts from the states before the first, and the last one's writes
// those after the last to `next`, a buffer of its own.
__device__ __forceinline__ void rl_ahead(const float4* state, float4* next, uint32_t n, uint32_t samples, uint32_t keep,
                                         float4* quads, uint32_t unit, uint32_t h, const uint4* tab, uint32_t* lds,
                                         uint32_t W)
{
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63, g0 = unit * 64u + lane;
    const bool valid = g0 < n;
    const uint32_t g = valid ? g0 : n - 1u;
    const float4 c6 = state[(size_t)6 * n + g];
    const uint32_t k = min((uint32_t)__builtin_amdgcn_readfirstlane((int)c6.z), 6u);
    const uint32_t first = 6u - k, total = (uint32_t)kRlAhead * samples, start = h * samples, stop = start + keep;
    const uint32_t nb = (total - first + 5u) / 6u;
    // blocks after the current one that hold quads start .. stop - 1
    const uint32_t lo = start < first ? 1u : 1u + (start - first) / 6u, hi = stop <= first ? 0u : 1u + (stop - 1u - first) / 6u;
    const bool end = h == (uint32_t)kRlAhead - 1u && w == W - 1u && hi < nb;   // a last block that is not kept
    const uint32_t t = end ? nb : lo + w;
    const bool idle = !end && t > hi;
    RlTab table;
    if (!idle) rl_load(table, tab + (size_t)(t - 1u) * kRlTaskVec);
    quads += (size_t)h * keep * n;
    uint32_t s[24], carry;
    if (w == 0) {
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const float4 v = state[(size_t)q * n + g];
            s[4 * q] = (uint32_t)(v.x * 16777216.0f);
            s[4 * q + 1] = (uint32_t)(v.y * 16777216.0f);
            s[4 * q + 2] = (uint32_t)(v.z * 16777216.0f);
            s[4 * q + 3] = (uint32_t)(v.w * 16777216.0f);
        }
        carry = c6.w > 0.0f ? 1u : 0u;
        rl_block(s, carry, k, 6u, 0u - start, keep, quads, n, g, valid);   // numbers below 0 wrap: not kept
        uint32_t* o = lds + lane * kRlIn;
#pragma unroll
        for (int q = 0; q < 6; ++q)
            *reinterpret_cast<uint4*>(o + 4 * q) =
                make_uint4((s[4 * q] ^ 0x808080u) | (q == 0 ? carry << 24 : 0u), s[4 * q + 1] ^ 0x808080u,
                           s[4 * q + 2] ^ 0x808080u, s[4 * q + 3] ^ 0x808080u);
    }
    __syncthreads();
    if (idle) return;
    rl_jump(table, lds, lds + 64 * kRlIn + w * 64u * kRlOut, s, carry);
    const uint32_t m = first + 6u * (t - 1u);
    const uint32_t k1 = min(6u, (t == nb ? total : stop) - m);
    rl_block(s, carry, 0u, k1, m - start, keep, quads, n, g, valid);
    if (t == nb && valid) rl_store(next, n, g, s, carry, k1);
}

// The same for the units first_unit, first_unit + step, ..: wavefronts
// 0 .. W - 1 keep the table of their block and make it for one unit after the
// other, wavefront W meanwhile finishes the block that the next unit's streams
// stand in.  LDS: two buffers of rings, then the W wavefronts' own words.
// For produce() that keep all quads, where every wavefront has a block for
// every h: heatbath half-step SU(3) 20 x 12 x 28 x 10 19.9 (a unit per workgroup) /
// 18.7 us, 16^3 x 32 28.2 / 24.7, 24^3 x 12 34.2 / 30.6; SU(2) (11 of 33 kept, a
// wavefront in five idle) 16^4 9.3 / 10.8, 32^3 x 16 32.4 / 38.2.
__device__ __forceinline__ void rl_ahead_turns(const float4* state, float4* next, uint32_t n, uint32_t samples, uint32_t keep,
                                         float4* quads, uint32_t first_unit, uint32_t step, uint32_t h, const uint4* tab,
                                         uint32_t* lds, uint32_t W)
{
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63, units = (n + 63u) / 64u;
    const float4 c0 = state[(size_t)6 * n];   // every stream stands at the same place of its block
    const uint32_t k = min((uint32_t)__builtin_amdgcn_readfirstlane((int)c0.z), 6u);
    const uint32_t first = 6u - k, total = (uint32_t)kRlAhead * samples, start = h * samples, stop = start + keep;
    const uint32_t nb = (total - first + 5u) / 6u;
    quads += (size_t)h * keep * n;
    auto ring = [&](uint32_t it) { return lds + (it & 1u) * 64u * kRlIn; };
    if (w == W) {
        auto finish = [&](uint32_t unit, uint32_t* in) {
            const uint32_t g0 = unit * 64u + lane, g = min(g0, n - 1u);
            uint32_t s[24];
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                const float4 v = state[(size_t)q * n + g];
                s[4 * q] = (uint32_t)(v.x * 16777216.0f);
                s[4 * q + 1] = (uint32_t)(v.y * 16777216.0f);
                s[4 * q + 2] = (uint32_t)(v.z * 16777216.0f);
                s[4 * q + 3] = (uint32_t)(v.w * 16777216.0f);
            }
            uint32_t carry = state[(size_t)6 * n + g].w > 0.0f ? 1u : 0u;
            rl_block(s, carry, k, 6u, 0u - start, keep, quads, n, g, g0 < n);   // numbers below 0 wrap: not kept
            uint32_t* o = in + lane * kRlIn;
#pragma unroll
            for (int q = 0; q < 6; ++q)
                *reinterpret_cast<uint4*>(o + 4 * q) =
                    make_uint4((s[4 * q] ^ 0x808080u) | (q == 0 ? carry << 24 : 0u), s[4 * q + 1] ^ 0x808080u,
                               s[4 * q + 2] ^ 0x808080u, s[4 * q + 3] ^ 0x808080u);
        };
        finish(first_unit, ring(0));
        __syncthreads();
        uint32_t it = 0;
        for (uint32_t u = first_unit; u < units; u += step, ++it) {
            if (u + step < units) finish(u + step, ring(it + 1u));
            __syncthreads();
        }
        return;
    }
    // blocks after the current one that hold quads start .. stop - 1
    const uint32_t lo = start < first ? 1u : 1u + (start - first) / 6u, hi = stop <= first ? 0u : 1u + (stop - 1u - first) / 6u;
    const bool end = h == (uint32_t)kRlAhead - 1u && w == W - 1u && hi < nb;   // a last block that is not kept
    const uint32_t t = end ? nb : lo + w, m = first + 6u * (t - 1u);
    const bool idle = !end && t > hi;
    RlTab table;
    if (!idle) rl_load(table, tab + (size_t)(t - 1u) * kRlTaskVec);
    const uint32_t k1 = idle ? 0u : min(6u, (t == nb ? total : stop) - m);
    __syncthreads();
    uint32_t it = 0;
    for (uint32_t u = first_unit; u < units; u += step, ++it) {
        if (!idle) {
            const uint32_t g0 = u * 64u + lane, g = min(g0, n - 1u);
            uint32_t s[24], carry;
            rl_jump(table, ring(it), lds + 128u * kRlIn + w * 64u * kRlOut, s, carry);
            rl_block(s, carry, 0u, k1, m - start, keep, quads, n, g, g0 < n);
            if (t == nb && g0 < n) rl_store(next, n, g, s, carry, k1);
        }
        __syncthreads();
    }
}

// Wavefronts W that make blocks: the blocks that `keep` quads can touch, and
// one for the last block when the last produce() keeps less than all; 0: not on
// this path.
inline uint32_t rl_ahead_waves(uint32_t samples, uint32_t keep)
{
    const uint32_t W = (keep + 4u) / 6u + 1u + (keep < samples ? 1u : 0u);
    const bool fits = samples >= 6u && keep >= 1u && keep <= samples &&
                      ((uint32_t)kRlAhead * samples + 5u) / 6u <= (uint32_t)kRlTasks && W < (uint32_t)kRlWaves;
    return fits ? W : 0u;
}
// rl_ahead_turns: its LDS, and workgroups per produce(): as many as run at once
// (16 wavefronts per CU), each with the same number of units.
inline uint32_t rl_turns_lds(uint32_t W) { return 4u * 64u * (2u * (uint32_t)kRlIn + W * (uint32_t)kRlOut); }
inline uint32_t rl_turns_groups(uint32_t n, uint32_t W)
{
    const uint32_t units = (n + 63u) / 64u, once = 256u * std::min(16u / (W + 1u), 163840u / rl_turns_lds(W)) / (uint32_t)kRlAhead;
    const uint32_t turns = (units + once - 1u) / once;
    return (units + turns - 1u) / turns;
}

// Wavefronts per 64 streams for a produce() of `samples` quads that keeps
// `keep` of them, for n streams; 0: step through the blocks instead.  That is
// for lengths that the tables or a workgroup do not reach, and for many
// streams of which most quads are kept: both ways then run some 620
// instructions per block and 64 streams, and stepping has no tables to load.
// Heatbath half-step with its produce(), stepping / in parallel, luxury 3:
// SU(2) (11 of 33 quads kept) 8^4 27.1 / 11.4 us, 32^4 98.9 / 60.9 us; SU(3)
// (all 33) 8^4 28.8 / 15.2, 24^3 x 12 45.2 / 40.5, 32^3 x 8 50.4 / 53.7 us;
// luxury 0, SU(3): 20 x 12 x 28 x 10 27.8 / 24.7, 16^3 x 32 32.7 / 36.0 us.
inline uint32_t rl_waves(int lux, uint32_t samples, uint32_t keep, uint64_t n)
{
    const uint32_t nb = (samples + 5u) / 6u, kept = (keep + 5u) / 6u + 1u;
    const uint32_t W = nb < kept ? (nb ? nb : 1u) : kept;
    const uint64_t most = rl_skip_count(lux) >= 223 ? 98304u : 40960u;
    if (nb > (uint32_t)kRlSpan || W > (uint32_t)kRlWaves || (W > 4u && n > most)) return 0u;
    return W;
}
inline uint32_t rl_lds_bytes(uint32_t W) { return 4u * 64u * ((uint32_t)kRlIn + W * (uint32_t)kRlOut); }

}  // namespace qcd
