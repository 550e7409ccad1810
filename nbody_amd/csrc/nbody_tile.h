// The one-launch force kernel for evaluations too small to fill the chip in
// j slices or block pairs: one workgroup of 16 waves owns a few i bodies and
// sums their whole force, so there are no partial sums in memory and no
// second launch.
//
// A workgroup takes TI = LI * I i bodies: a wave's 64 lanes are S = 64 / LI
// groups of LI lanes, every lane holds I of the i bodies, and the groups of
// all 16 waves take different j bodies. The j bodies pass through LDS in
// chunks of kTileChunk (double-buffered, one barrier per chunk; the loads of
// the next chunk are in flight while this one is computed): step k of a chunk
// gives group g = wave * S + s the record k * 16 S + g, so a wave reads S
// consecutive records at once. Groups and waves are added at the end in a
// fixed order, so a result depends on the shape only.
//
// What bounds it: up to N = 2048 the launch and the latency of a first read
// of the bodies (2.8 us at N = 256 and 3.1 at 1000, where one lane's serial
// chain over all j took 11.7 and 42); above, the one-sided chain (11 VALU +
// 1 v_rsq_f32 per interaction on one mass, 12 otherwise) at 4 or 8 waves per
// SIMD, with a ds_read_b128 of the CU's LDS (about 12 clocks) per step of I
// interactions: 7.8 us at N = 4096, 21.0 at 8192 (0.41 of the FP32 peak),
// 31 at 10000.
//
// With FP64 accumulation (F64) every term is added in FP64 and the groups'
// and waves' sums stay FP64 to the end (nbody_acc64.h). There it replaces the
// one serial chain over all j of a system below 1024 bodies or of a small i
// range: N = 256 12.2 and 3.9 us, 1000 44.4 and 3.9, 500 of 2000 87 and 4.2,
// 2048 of 16384 52.6 and 21.7 (two launches with slices), 1000 of 65536 70 and
// 49.
#pragma once

#include "nbody_acc64.h"
#include "nbody_device.h"
#include "nbody_kernels.h"

#include <type_traits>

namespace nbody {

typedef float vec4 __attribute__((ext_vector_type(4)));

constexpr int kTileWaves = 16;
constexpr int kTileThreads = 64 * kTileWaves;
constexpr int kTileChunk = 2048;  // j bodies per LDS buffer (32 KiB; two buffers)

// v of the lane CTRL - 0x120 below in the row of 16, turning around (DPP row_ror).
template <int CTRL>
__device__ __forceinline__ float row_ror(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

template <int CTRL>
__device__ __forceinline__ double row_ror(double v)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// add(partner) for each halving of a wave's groups of LI = 4 or 8 lanes; after
// them every lane holds the sum over the groups.
template <int LI, class Add>
__device__ __forceinline__ void over_groups(const Add& add)
{
    static_assert(LI == 4 || LI == 8, "groups within a row of 16 lanes");
    if constexpr (LI == 4) add([](auto v) { return row_ror<0x124>(v); });  // row_ror:4
    add([](auto v) { return row_ror<0x128>(v); });                         // row_ror:8
    add([](auto v) { return __shfl_xor(v, 16); });
    add([](auto v) { return __shfl_xor(v, 32); });
}

// `steps` records t4[0], t4[stride], ... against the lane's i bodies, two
// records at a time; the next two are read while these are in use.
template <int I, bool EQ, class Acc>
__device__ __forceinline__ void tile_sweep(const vec4* t4, int stride, int steps, float eps2, const Lanes<I>& me,
                                           Acc& acc)
{
    auto meet = [&](const vec4& b) {
#pragma unroll
        for (int u = 0; u < I; ++u) {
            if constexpr (std::is_same<Acc, Lanes64<I>>::value) {
                begin_terms();
                const Terms64 t = terms64<false, EQ>(make_float4(b.x, b.y, b.z, b.w), me.x[u], me.y[u], me.z[u], 0.f,
                                                     eps2);
                begin_sums();
                acc.x[u] = __builtin_fma(t.x, t.si, acc.x[u]);
                acc.y[u] = __builtin_fma(t.y, t.si, acc.y[u]);
                acc.z[u] = __builtin_fma(t.z, t.si, acc.z[u]);
            } else {
                interact<false, false, EQ>(b.x, b.y, b.z, b.w, me.x[u], me.y[u], me.z[u], eps2, acc.x[u], acc.y[u],
                                           acc.z[u]);
            }
        }
    };
    if (steps <= 0) return;
    auto record = [&](int k) { return t4[min(k, steps - 1) * stride]; };
    vec4 a = record(0), b = record(1);
    int k = 0;
    for (; k + 4 <= steps; k += 4) {  // four per turn, so that no record is moved between registers
        const vec4 c = record(k + 2), d = record(k + 3);
        meet(a);
        meet(b);
        a = record(k + 4);
        b = record(k + 5);
        meet(c);
        meet(d);
    }
    if (k < steps) meet(a);
    if (k + 1 < steps) meet(b);
    if (k + 2 < steps) meet(record(k + 2));
}

// Up to 3 bodies per lane the kernel fits 64 VGPRs, two workgroups (8 waves
// per SIMD) on a CU. STEP also integrates the workgroup's bodies, into another
// position buffer: a step of a small system is then one launch.
template <int LI, int I, bool STEP, bool F64>
__global__ __launch_bounds__(kTileThreads, I <= 3 && !F64 ? 8 : 4) void k_force_tile(ForceParams p)
{
    typedef typename std::conditional<F64, double, float>::type Sum;
    typedef typename std::conditional<F64, Lanes64<I>, Lanes<I>>::type Acc;
    constexpr int S = 64 / LI;             // groups per wave
    constexpr int G = kTileWaves * S;      // groups per workgroup
    constexpr int TI = LI * I;             // i bodies per workgroup
    constexpr int R = kTileChunk / kTileThreads;
    static_assert(kTileWaves * 3 * TI * sizeof(Sum) <= sizeof(vec4) * 2 * kTileChunk, "last sum fits the tiles");
    __shared__ vec4 tile[2][kTileChunk];
    __shared__ int uneven[2][kTileWaves];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int group = wave * S + lane / LI;
    const int first = blockIdx.x * TI;

    Lanes<I> me;
    Acc acc;
#pragma unroll
    for (int u = 0; u < I; ++u) {
        const float4 q = p.pm[p.i0 + min(first + u * LI + lane % LI, p.ni - 1)];
        me.x[u] = q.x;
        me.y[u] = q.y;
        me.z[u] = q.z;
    }
    zero<I>(acc);
    const float m0 = p.pm[0].w;
    // (vector types: HIP's float4 keeps an array of records out of registers)
    const vec4* src = reinterpret_cast<const vec4*>(p.pm);
    vec4 next[R];
#pragma unroll
    for (int r = 0; r < R; ++r) next[r] = src[min(r * kTileThreads + t, p.n - 1)];

    // The sums leave the mass out until a chunk with another mass than body
    // 0's comes: then they are multiplied by m0 once, and from there on every
    // term carries its mass. On one mass that is one product per sum; for m0 a
    // power of two the same bits either way.
    bool massless = true;
    for (int c = 0, buf = 0; c < p.n; c += kTileChunk, buf ^= 1) {
        const int len = min(kTileChunk, p.n - c);
        // each wave notes whether its part of the chunk is all of body 0's
        // mass, and after the barrier every wave reads all 16 notes
        bool ok = true;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = r * kTileThreads + t;
            tile[buf][k] = next[r];  // past the chunk's end: a copy of the last body, never read
            ok &= next[r].w == m0;
        }
        const bool all = __builtin_amdgcn_ballot_w64(!ok) == 0;
        if (lane == 0) uneven[buf][wave] = !all;
        __syncthreads();
        if (c + kTileChunk < p.n) {
#pragma unroll
            for (int r = 0; r < R; ++r) next[r] = src[min(c + kTileChunk + r * kTileThreads + t, p.n - 1)];
        }
        const bool eq = __builtin_amdgcn_ballot_w64(uneven[buf][lane % kTileWaves] != 0) == 0;
        const vec4* t4 = tile[buf] + group;
        const int steps = len / G;
        if (massless && !eq) {
            if (c > 0) scale<I>(acc, (Sum)m0);
            massless = false;
        }
        if (massless) tile_sweep<I, true, Acc>(t4, G, steps, p.eps2, me, acc);
        else tile_sweep<I, false, Acc>(t4, G, steps, p.eps2, me, acc);
        if (steps * G + group < len) {  // the chunk's ragged last step
            if (massless) tile_sweep<I, true, Acc>(t4 + steps * G, G, 1, p.eps2, me, acc);
            else tile_sweep<I, false, Acc>(t4 + steps * G, G, 1, p.eps2, me, acc);
        }
    }
    if (massless) scale<I>(acc, (Sum)m0);

    // the wave's groups, then the 16 waves in order
    over_groups<LI>([&](const auto& partner) {
#pragma unroll
        for (int u = 0; u < I; ++u) {
            acc.x[u] += partner(acc.x[u]);
            acc.y[u] += partner(acc.y[u]);
            acc.z[u] += partner(acc.z[u]);
        }
    });
    __syncthreads();  // the last chunk has been read by every wave
    Sum* red = reinterpret_cast<Sum*>(&tile[0][0]);  // [wave][3][TI]
    if (lane < LI) {
        Sum* o = red + wave * 3 * TI + lane;
#pragma unroll
        for (int u = 0; u < I; ++u) {
            o[0 * TI + u * LI] = acc.x[u];
            o[1 * TI + u * LI] = acc.y[u];
            o[2 * TI + u * LI] = acc.z[u];
        }
    }
    __syncthreads();
    const int m = first + t % TI;
    float total = 0.f;
    if (t < 3 * TI && m < p.ni) {
        // in FP64: the 16 roundings of this one sum would outweigh those of all the sums before it
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < kTileWaves; ++w) sum += red[w * 3 * TI + t];
        total = (float)sum;
        p.force[4 * (size_t)m + t / TI] = total;
    }
    if constexpr (STEP) {
        float* of = reinterpret_cast<float*>(red + kTileWaves * 3 * TI);  // [3][TI], behind the waves' sums
        static_assert((kTileWaves + 1) * 3 * TI * sizeof(Sum) <= sizeof(vec4) * 2 * kTileChunk, "fits the tiles");
        if (t < 3 * TI) of[t] = total;
        __syncthreads();
        if (t < TI && m < p.ni) step_body(p.step, m, of[t], of[TI + t], of[2 * TI + t]);
    }
}

}  // namespace nbody
