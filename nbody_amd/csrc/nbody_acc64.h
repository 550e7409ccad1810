// Device code of the FP64-accumulation plans (compensated = 2): the
// symmetric block pairs and the LDS-tiled one-sided sweep with every term
// added in FP64.
//
// Each term's inputs are the FP32 values of the default kernels: d = x_j - x_i,
// w = m (inv inv) inv or m inv (inv inv) with inv = v_rsq_f32(|d|^2 + eps2).
// Their product is exact in FP64 (24 x 24 bits), and a sum of such products
// in FP64 loses about 2^-53 of the running sum per term, so the force keeps
// only the FP32 rounding of each term's own inputs, which does not grow with
// cancellation between terms. The FP32 plans round every partial sum to 24
// bits, which is what costs digits on a body whose force is the small
// remainder of large cancelling terms. Partial sums (slots, slices) stay in
// FP64 until the one final rounding to the FP32 force.
#pragma once

#include "nbody_device.h"
#include "nbody_sym.h"

namespace nbody {

template <int I>
struct Lanes64 {
    double x[I], y[I], z[I];
};

template <int I>
__device__ __forceinline__ void zero(Lanes64<I>& a)
{
#pragma unroll
    for (int u = 0; u < I; ++u) a.x[u] = a.y[u] = a.z[u] = 0.0;
}

template <int I>
__device__ __forceinline__ void scale(Lanes64<I>& a, double m)
{
#pragma unroll
    for (int u = 0; u < I; ++u) {
        a.x[u] *= m;
        a.y[u] *= m;
        a.z[u] *= m;
    }
}

typedef SlotMapT<double> SlotMap64;

// Each interaction is cut in two, the FP32 terms with their conversions at the
// wave's low priority and the FP64 sums at high, and the compiler keeps the
// parts apart. An FP64 FMA or a conversion has a SIMD's issue to itself for
// four clocks; only FP32 instructions of different waves go two at a time, and
// they meet when every wave that has sums to do does them first. Clocks of a
// SIMD per 64 pairs of a block pair, 4 bodies per lane, interleaved by the
// compiler and so: unequal masses 95.0 and 82.9, one mass 81.7 and 75.6; with
// the conversions in the high part 85.5 and 78.3. The same operations on each
// sum in the same order, so the same bits. Two or four pairs to a part measured
// slower in the kernel (N = 65536: 1211, 1262 and 1326 us).
__device__ __forceinline__ void begin_terms()
{
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
}
__device__ __forceinline__ void begin_sums()
{
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
}

// wave_ror1 of a double: both 32-bit halves move one lane.
__device__ __forceinline__ double wave_ror1_f64(double v)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, 0x13C, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), 0x13C, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// The FP32 terms of one interaction, as FP64 factors: the difference d, the
// i side's weight and the j side's (with EQ both leave the common mass out and
// the j side's is not formed).
struct Terms64 {
    double x, y, z, si, sj;
};

template <bool NEWTON, bool EQ>
__device__ __forceinline__ Terms64 terms64(const float4& b, float xi, float yi, float zi, float mi, float eps2)
{
    const float dx = b.x - xi;
    const float dy = b.y - yi;
    const float dz = b.z - zi;
    float d2 = __builtin_fmaf(dx, dx, eps2);
    d2 = __builtin_fmaf(dy, dy, d2);
    d2 = __builtin_fmaf(dz, dz, d2);
    const float inv = rsqrt_f32<NEWTON>(d2);
    const float inv3 = (inv * inv) * inv;
    Terms64 t;
    t.x = dx;
    t.y = dy;
    t.z = dz;
    t.si = EQ ? inv3 : b.w * inv3;
    t.sj = EQ ? 0.0 : (double)(-mi * inv3);
    return t;
}

// Tile `tile` of block Q (64 bodies from jbase on) against this lane's A
// bodies: the rotation of nbody_sym.h (the j body's position, mass and FP64
// reaction move one lane per step), each term accumulated in FP64. The tile's
// reactions go straight from the lanes to their slots. With EQ every body of
// both has mass m0: the term weights leave it out (inv^3 on the i side,
// -inv^3 on the j side: one conversion to FP64 instead of two, no mass
// products, the masses do not rotate) and the reactions are multiplied by m0
// at the store; for m0 = 1 the terms are the general path's bits.
template <int A, bool NEWTON, bool EQ>
__device__ __forceinline__ void sym_tile64(const float4* __restrict__ pm, int n, float eps2, int jbase,
                                           const Lanes<A>& me, const float (&mi)[A], double m0, Lanes64<A>& acc,
                                           double* __restrict__ jdst, size_t plane)
{
    const int lane = threadIdx.x & 63;
    float4 b = lane < n - jbase ? pm[jbase + lane] : make_float4(0.f, 0.f, 0.f, 0.f);
    double rx = 0.0, ry = 0.0, rz = 0.0;
    for (int k = 0; k < 64; ++k) {
#pragma unroll
        for (int u = 0; u < A; ++u) {
            begin_terms();
            const Terms64 t = terms64<NEWTON, EQ>(b, me.x[u], me.y[u], me.z[u], mi[u], eps2);
            begin_sums();
            const double sj = EQ ? -t.si : t.sj;
            acc.x[u] = __builtin_fma(t.x, t.si, acc.x[u]);
            acc.y[u] = __builtin_fma(t.y, t.si, acc.y[u]);
            acc.z[u] = __builtin_fma(t.z, t.si, acc.z[u]);
            rx = __builtin_fma(t.x, sj, rx);
            ry = __builtin_fma(t.y, sj, ry);
            rz = __builtin_fma(t.z, sj, rz);
        }
        b.x = wave_ror1(b.x);
        b.y = wave_ror1(b.y);
        b.z = wave_ror1(b.z);
        if constexpr (!EQ) b.w = wave_ror1(b.w);
        rx = wave_ror1_f64(rx);
        ry = wave_ror1_f64(ry);
        rz = wave_ror1_f64(rz);
    }
    jdst[lane] = EQ ? rx * m0 : rx;
    jdst[plane + lane] = EQ ? ry * m0 : ry;
    jdst[2 * plane + lane] = EQ ? rz * m0 : rz;
}

// Body i (this lane's) against bodies [j0, j0 + len), one-sided, in j order,
// every term added in FP64 into (ax, ay, az). A lane whose i is past n
// computes on a zero body. The bodies of four steps are loaded before the
// first of them is used.
template <bool NEWTON>
__device__ __forceinline__ void row64(const float4* __restrict__ pm, int n, float eps2, int i, int j0, int len,
                                      double& ax, double& ay, double& az)
{
    constexpr int L = 4;
    const float4 q = i < n ? pm[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    ax = ay = az = 0.0;
    int j = 0;
    for (; j + L <= len; j += L) {
        float4 b[L];
#pragma unroll
        for (int l = 0; l < L; ++l) b[l] = pm[j0 + j + l];
#pragma unroll
        for (int l = 0; l < L; ++l) {
            begin_terms();
            const Terms64 t = terms64<NEWTON, false>(b[l], q.x, q.y, q.z, 0.f, eps2);
            begin_sums();
            ax = __builtin_fma(t.x, t.si, ax);
            ay = __builtin_fma(t.y, t.si, ay);
            az = __builtin_fma(t.z, t.si, az);
        }
    }
    for (; j < len; ++j) {
        const Terms64 t = terms64<NEWTON, false>(pm[j0 + j], q.x, q.y, q.z, 0.f, eps2);
        ax = __builtin_fma(t.x, t.si, ax);
        ay = __builtin_fma(t.y, t.si, ay);
        az = __builtin_fma(t.z, t.si, az);
    }
}

constexpr int kWaves64 = 4;

// Block pair (P, Q), P < Q, or the diagonal block P == Q, on a workgroup of 4
// waves, with A bodies of block P per lane (B = 64 A).
//
// Bound by issue: a block pair takes 82.9 clocks of a
// SIMD per 64 pairs (above). Four waves and not one: the time of a small
// system is that of one task. Unequal masses, before and after (interleaved
// terms on one-wave tasks): N = 1024 55.5 and 21.9 us, 4096 55.8 and 22.1, 8192
// 60.4 and 41.4, 16384 105.5 and 97.8, 65536 1318 and 1211, 98304 2928 and 2687;
// one mass 4096 50.8 and 22.2, 65536 1150 and 1144.
//
// Pair: every wave holds block P's bodies and meets every fourth tile of block
// Q, whose reactions it stores; the i sides of the four waves are added in
// LDS, in wave order. Tiles past the end of a ragged last block are skipped:
// their bodies are padding, whose slots no reduction reads. A wave whose tiles
// and block P all have the mass of body P*B (a wave vote; padding has mass 0,
// so a ragged tile never qualifies) runs the mass-free terms.
//
// Diagonal: 64 bodies per wave at a time against the bodies of the block,
// one-sided, in j order, into slot P. Lanes past n compute on a zero body and
// store into padding that no reduction reads.
template <int A, bool NEWTON>
__device__ __forceinline__ void sym_task64(const float4* __restrict__ pm, int n, float eps2, const SlotMap64& slots,
                                           int P, int Q, double (*part)[3][64 * A])
{
    constexpr int B = 64 * A, W = kWaves64;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (P == Q) {
        double* __restrict__ dst = slots.j_side(P, P, B);
        for (int k = wave; k < A && P * B + k * 64 < n; k += W) {
            double ax, ay, az;
            row64<NEWTON>(pm, n, eps2, P * B + k * 64 + lane, P * B, min(n - P * B, B), ax, ay, az);
            dst[k * 64 + lane] = ax;
            dst[slots.bplane + k * 64 + lane] = ay;
            dst[2 * slots.bplane + k * 64 + lane] = az;
        }
        return;
    }
    const float m0 = pm[P * B].w;
    Lanes<A> me;
    float mi[A];
    bool same = true;
#pragma unroll
    for (int u = 0; u < A; ++u) {
        const float4 q = pm[P * B + u * 64 + lane];
        me.x[u] = q.x;
        me.y[u] = q.y;
        me.z[u] = q.z;
        mi[u] = q.w;
        same &= q.w == m0;
    }
    for (int tile = wave; tile < A; tile += W) {
        const int j = Q * B + tile * 64 + lane;
        same &= (j < n) & (pm[min(j, n - 1)].w == m0);
    }
    const bool eq = __builtin_amdgcn_ballot_w64(!same) == 0;
    Lanes64<A> acc;
    zero<A>(acc);
    double* jdst = slots.j_side(P, Q, B);
    for (int tile = wave; tile < A; tile += W) {
        const int jbase = Q * B + tile * 64;  // wave-uniform
        if (jbase >= n) break;
        if (eq)
            sym_tile64<A, NEWTON, true>(pm, n, eps2, jbase, me, mi, (double)m0, acc, jdst + tile * 64, slots.bplane);
        else sym_tile64<A, NEWTON, false>(pm, n, eps2, jbase, me, mi, 1.0, acc, jdst + tile * 64, slots.bplane);
    }
    const double scale = eq ? (double)m0 : 1.0;
#pragma unroll
    for (int u = 0; u < A; ++u) {
        part[wave][0][u * 64 + lane] = acc.x[u] * scale;
        part[wave][1][u * 64 + lane] = acc.y[u] * scale;
        part[wave][2][u * 64 + lane] = acc.z[u] * scale;
    }
    __syncthreads();
    double* __restrict__ idst = slots.i_side(P, Q, B);
    const size_t iplane = slots.i_plane(P);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int k = 0; k < B; k += 64 * W) {
            const int o = k + threadIdx.x;
            double sum = part[0][c][o];
#pragma unroll
            for (int w = 1; w < W; ++w) sum += part[w][c][o];
            idst[c * iplane + o] = sum;
        }
}

}  // namespace nbody
