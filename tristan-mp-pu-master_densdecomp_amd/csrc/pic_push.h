// pic_push.h -- gather and Esirkepov deposit of one particle, written against
// a field source and a current sink so the same arithmetic serves the tiled
// kernel (LDS-staged fields, LDS currents) and the flat kernel (HBM fields,
// global atomics).
//
// Reference: mover_{1,2,3}ord gathers (code/particles_movedeposit.F90:
// 1137-1170 and the order-1/2 equivalents) and densdecomp_{1,2,3}ord
// (code/particles.F90:678-1358).
#pragma once
#include "pic_math.h"

namespace tmpg {

__device__ __forceinline__ int wrap1(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// gather nodes with nonzero weights: order 1 uses nodes 0..1, others -1..2
template <int ORD> struct GatherRange { static constexpr int N0 = (ORD == 1) ? 1 : 0, N1 = (ORD == 1) ? 3 : 4; };

// Field sources.  (i,j,k) are the particle's cell in the source's own
// coordinates; node offsets are -2..+3.
struct GlobalSrc {
    const float* f[6];
    int nx, ny, nz;
    __device__ __forceinline__ int64_t row(int j, int k) const
    {
        return (int64_t)nx * (wrap1(j, ny) + (int64_t)ny * wrap1(k, nz));
    }
    __device__ __forceinline__ int col(int i) const { return wrap1(i, nx); }
    __device__ __forceinline__ float get(int q, int64_t r, int c) const { return f[q][r + c]; }
    __device__ __forceinline__ float2 exby(int i, int j) const { return make_float2(get(0, row(j, 0), col(i)), get(4, row(j, 0), col(i))); }
    __device__ __forceinline__ float2 eybx(int i, int j) const { return make_float2(get(1, row(j, 0), col(i)), get(3, row(j, 0), col(i))); }
    __device__ __forceinline__ float ez(int i, int j) const { return get(2, row(j, 0), col(i)); }
    __device__ __forceinline__ float bz(int i, int j) const { return get(5, row(j, 0), col(i)); }
    __device__ __forceinline__ void get6(int64_t r, int c, float* v) const
    {
#pragma unroll
        for (int q = 0; q < 6; ++q) v[q] = f[q][r + c];
    }
};

// 3D primal fields staged in LDS node-major: the six components of a node are
// adjacent (24 bytes), so one node is three 8-byte LDS reads instead of six
// 4-byte reads from six planes.  All six use the same primal weights.
struct LdsSrc6 {
    const float* s;     // [node][6], node = i + fx*(j + fy*k)
    int fx, fy;
    __device__ __forceinline__ int row(int j, int k) const { return (j + fy * k) * fx; }
    __device__ __forceinline__ int col(int i) const { return i; }
    __device__ __forceinline__ void get6(int r, int c, float* v) const
    {
        const float2* p = reinterpret_cast<const float2*>(s) + 3 * (r + c);
        const float2 a = p[0], b = p[1], d = p[2];
        v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y; v[4] = d.x; v[5] = d.y;
    }
};

struct LdsSrc {
    const float* s;     // 6 component planes of fx*fy*fz floats
    int fx, fy, plane;
    __device__ __forceinline__ int row(int j, int k) const { return (j + fy * k) * fx; }
    __device__ __forceinline__ int col(int i) const { return i; }
    __device__ __forceinline__ float get(int q, int r, int c) const { return s[q * plane + r + c]; }
    __device__ __forceinline__ float2 exby(int i, int j) const { return make_float2(get(0, row(j, 0), col(i)), get(4, row(j, 0), col(i))); }
    __device__ __forceinline__ float2 eybx(int i, int j) const { return make_float2(get(1, row(j, 0), col(i)), get(3, row(j, 0), col(i))); }
    __device__ __forceinline__ float ez(int i, int j) const { return get(2, row(j, 0), col(i)); }
    __device__ __forceinline__ float bz(int i, int j) const { return get(5, row(j, 0), col(i)); }
    __device__ __forceinline__ void get6(int r, int c, float* v) const
    {
#pragma unroll
        for (int q = 0; q < 6; ++q) v[q] = s[q * plane + r + c];
    }
};

struct GlobalSink {
    float* j[3];
    int nx, ny, nz;
    __device__ __forceinline__ int64_t row(int jj, int kk) const
    {
        return (int64_t)nx * (wrap1(jj, ny) + (int64_t)ny * wrap1(kk, nz));
    }
    __device__ __forceinline__ int col(int i) const { return wrap1(i, nx); }
    __device__ __forceinline__ void add(int q, int64_t r, int c, float v) const { atomicAdd(j[q] + r + c, v); }
};

// Tile currents in LDS are accumulated in FP64: on gfx950 ds_add_f64 runs
// about 3x faster than ds_add_f32 (measured on the 3D order-3 push), and the
// tile sum is rounded to FP32 once, at the flush.
struct LdsSink {
    double* s;          // 3 component planes of jx*jy*jz doubles
    int jx, jy, plane;
    __device__ __forceinline__ int row(int jj, int kk) const { return (jj + jy * kk) * jx; }
    __device__ __forceinline__ int col(int i) const { return i; }
    __device__ __forceinline__ void add(int q, int r, int c, double v) const { atomicAdd(s + q * plane + r + c, v); }
};

// ---------------------------------------------------------- 2D gather
// Weights of one axis on fixed nodes: primal P at nodes PF .. PF+NP-1, dual
// (half-cell shifted) D at nodes did+DF .. did+DF+ND-1 relative to the cell;
// the values of gather_weights without its zero slots.  Order 2: the dual
// spline's three nodes are always -1..1, and with the reference's loop range
// (code/particles_movedeposit.F90:709-832) the primal sum keeps only the
// nodes 0 and 1 -- except at an offset of 0, where that range keeps node -1
// as well (at_zero).
template <int ORD, bool QUIRK> struct AxisW;

template <bool QUIRK> struct AxisW<1, QUIRK> {
    static constexpr int PF = 0, NP = 2, DF = 0, ND = 2;
    __device__ __forceinline__ static int w(float o, float* P, float* D)
    {
        P[0] = 1.0f - o;
        P[1] = o;
        const bool hi = o >= 0.5f;
        const float od = hi ? o - 0.5f : o + 0.5f;
        D[0] = 1.0f - od;
        D[1] = od;
        return hi ? 0 : -1;
    }
};

template <bool QUIRK> struct AxisW<2, QUIRK> {
    static constexpr int PF = QUIRK ? 0 : -1, NP = QUIRK ? 2 : 4, DF = -1, ND = 3;
    __device__ __forceinline__ static int w(float o, float* P, float* D)
    {
        if constexpr (QUIRK) {
            const bool up = o >= 0.5f;
            const float xi = up ? o - 1.0f : o;
            const float m = 0.75f - xi * xi;
            const float h = up ? 0.5f - xi : 0.5f + xi;
            const float e = 0.5f * h * h;
            P[0] = up ? e : m;
            P[1] = up ? m : e;
        } else {
            frame_weights<2>(o, P);
        }
        const float od = o >= 0.5f ? o - 0.5f : o + 0.5f;
        Piece<2>::w(o >= 0.5f ? od : od - 1.0f, D);
        return 0;
    }
    // the weight that the reference's loop range gives to the primal node -1:
    // nonzero only at an offset that vanishes beside 1/2
    __device__ __forceinline__ static float at_zero(float o)
    {
        const float l = 0.5f - o;
        return o + 0.5f > 0.5f ? 0.0f : 0.5f * l * l;
    }
};

template <bool QUIRK> struct AxisW<3, QUIRK> {
    static constexpr int PF = -1, NP = 4, DF = -1, ND = 4;
    __device__ __forceinline__ static int w(float o, float* P, float* D)
    {
        Piece<3>::w(o, P);
        const bool hi = o >= 0.5f;
        Piece<3>::w(hi ? o - 0.5f : o + 0.5f, D);
        return hi ? 0 : -1;
    }
};

// E, B at a particle of cell (i, j) from the staggered fields with matching
// primal/dual weights (code/particles_movedeposit.F90:1155-1170 and the lower
// orders).  Orders 1 and 3 sum each y row of nodes along x, then scale it by
// its y weight.  Order 2, whose weights jump at half a cell, keeps the
// products and their order of the plain double sum: there a change of
// rounding shifts single particles across the jump.
template <int ORD, bool QUIRK, class Src>
__device__ __forceinline__ void gather2(const Src& src, int i, int j, float ox, float oy, float* E)
{
    using AW = AxisW<ORD, QUIRK>;
    float Px[AW::NP], Dx[AW::ND], Py[AW::NP], Dy[AW::ND];
    const int id = i + AW::w(ox, Px, Dx), jd = j + AW::w(oy, Py, Dy);
#pragma unroll
    for (int q = 0; q < 6; ++q) E[q] = 0.0f;
    // a row's sum r += v w (orders 1, 3), or E += (v w) wy at once (order 2)
    auto add = [](float v, float w, float wy, float& r, float& e) {
        if constexpr (ORD == 2) e = fmaf(v * w, wy, e);
        else r = fmaf(v, w, r);
    };
    if constexpr (ORD == 2 && QUIRK) {
        // (the y row and the x column of node -1 come first in the sums)
        const float mx = AW::at_zero(ox), my = AW::at_zero(oy);
        if (mx != 0.0f || my != 0.0f) {
            // the general double sums over nodes -1, 0, 1 of both kinds
            const float Qx[3] = {mx, Px[0], Px[1]}, Qy[3] = {my, Py[0], Py[1]};
#pragma unroll
            for (int y = 0; y < 3; ++y)
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    const float2 f = src.exby(i + x - 1, j + y - 1), h = src.eybx(i + x - 1, j + y - 1);
                    E[0] = fmaf(f.x * Dx[x], Qy[y], E[0]);
                    E[4] = fmaf(f.y * Dx[x], Qy[y], E[4]);
                    E[1] = fmaf(h.x * Qx[x], Dy[y], E[1]);
                    E[3] = fmaf(h.y * Qx[x], Dy[y], E[3]);
                    E[2] = fmaf(src.ez(i + x - 1, j + y - 1) * Qx[x], Qy[y], E[2]);
                    E[5] = fmaf(src.bz(i + x - 1, j + y - 1) * Dx[x], Dy[y], E[5]);
                }
            return;
        }
    }
#pragma unroll
    for (int y = 0; y < AW::NP; ++y) {
        const int jp = j + AW::PF + y;
        float r0 = 0.0f, r4 = 0.0f, r2 = 0.0f;
#pragma unroll
        for (int x = 0; x < AW::ND; ++x) {
            const float2 f = src.exby(id + AW::DF + x, jp);
            add(f.x, Dx[x], Py[y], r0, E[0]);
            add(f.y, Dx[x], Py[y], r4, E[4]);
        }
#pragma unroll
        for (int x = 0; x < AW::NP; ++x) add(src.ez(i + AW::PF + x, jp), Px[x], Py[y], r2, E[2]);
        if constexpr (ORD != 2) {
            E[0] = fmaf(r0, Py[y], E[0]);
            E[4] = fmaf(r4, Py[y], E[4]);
            E[2] = fmaf(r2, Py[y], E[2]);
        }
    }
#pragma unroll
    for (int y = 0; y < AW::ND; ++y) {
        const int jn = jd + AW::DF + y;
        float r1 = 0.0f, r3 = 0.0f, r5 = 0.0f;
#pragma unroll
        for (int x = 0; x < AW::NP; ++x) {
            const float2 f = src.eybx(i + AW::PF + x, jn);
            add(f.x, Px[x], Dy[y], r1, E[1]);
            add(f.y, Px[x], Dy[y], r3, E[3]);
        }
#pragma unroll
        for (int x = 0; x < AW::ND; ++x) add(src.bz(id + AW::DF + x, jn), Dx[x], Dy[y], r5, E[5]);
        if constexpr (ORD != 2) {
            E[1] = fmaf(r1, Dy[y], E[1]);
            E[3] = fmaf(r3, Dy[y], E[3]);
            E[5] = fmaf(r5, Dy[y], E[5]);
        }
    }
}

// E, B at the particle; 3D from primal-averaged fields with primal weights
// (code/particles_movedeposit.F90:1137-1153), 2D from the staggered fields
// with matching primal/dual weights (:1155-1170).
template <int DIM, int ORD, class Src>
__device__ __forceinline__ void gather(const Src& src, bool quirk2, int i, int j, int k, float ox, float oy,
                                       float oz, float* E)
{
    if constexpr (DIM == 3) {
        constexpr int N0 = GatherRange<ORD>::N0, N1 = GatherRange<ORD>::N1;
#pragma unroll
        for (int q = 0; q < 6; ++q) E[q] = 0.0f;
        float Spx[4], Sdx[4], Spy[4], Sdy[4], Spz[4], Sdz[4];
        int dix, diy, diz;
        gather_weights<ORD>(ox, quirk2, Spx, Sdx, dix);
        gather_weights<ORD>(oy, quirk2, Spy, Sdy, diy);
        gather_weights<ORD>(oz, quirk2, Spz, Sdz, diz);
        int cx[4];
#pragma unroll
        for (int t = N0; t < N1; ++t) cx[t] = src.col(i - 1 + t);
        // each z plane summed with the x-y weights, then scaled by its z
        // weight (the order of every sum is the one of gather3_lds)
        float wxy[4][4];
#pragma unroll
        for (int b = N0; b < N1; ++b)
#pragma unroll
            for (int t = N0; t < N1; ++t) wxy[b][t] = Spx[t] * Spy[b];
#pragma unroll
        for (int c = N0; c < N1; ++c) {
            float acc[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int b = N0; b < N1; ++b) {
                const auto r = src.row(j - 1 + b, k - 1 + c);
#pragma unroll
                for (int t = N0; t < N1; ++t) {
                    float v[6];
                    src.get6(r, cx[t], v);
#pragma unroll
                    for (int q = 0; q < 6; ++q) acc[q] = fmaf(v[q], wxy[b][t], acc[q]);
                }
            }
#pragma unroll
            for (int q = 0; q < 6; ++q) E[q] = fmaf(acc[q], Spz[c], E[q]);
        }
    } else {
        if (ORD == 2 && quirk2) gather2<ORD, true>(src, i, j, ox, oy, E);
        else gather2<ORD, false>(src, i, j, ox, oy, E);
    }
}

// The 3D gather from node-major primal fields in LDS whose strides FX, FY
// (nodes per row, rows per plane) are compile-time constants.  A node's six
// values sit in two arrays of 16-byte entries: (Ex, Ey, Ez, Bx) in s4, and
// in sp (By, Bz) of the node followed by (By, Bz) of its +x neighbour.  A row
// of the block is NB reads of s4 and NB/2 of sp, all 16-byte reads with a
// 16-bit immediate offset, which covers the particle's whole 4x4x4 node
// block (at most 6.4 KB from its first node for the 8x8x4 tile): one base
// address per array and no per-node address arithmetic.
// (i,j,k) is the particle's cell in staged-node coordinates, at least 1 on
// every axis.  Same arithmetic as gather<3, ORD>.  RB node rows go into each
// batch of reads (two batches in flight): 2 hides LDS latency within the
// wave, 1 keeps the registers for more waves.
template <int ORD, int FX, int FY, int RB = 2>
__device__ __forceinline__ void gather3_lds(const float4* __restrict__ s4, const float4* __restrict__ sp, bool quirk2,
                                            int i, int j, int k, float ox, float oy, float oz, float* E)
{
    float Spx[4], Sdx[4], Spy[4], Sdy[4], Spz[4], Sdz[4];
    int dix, diy, diz;
    gather_weights<ORD>(ox, quirk2, Spx, Sdx, dix);
    gather_weights<ORD>(oy, quirk2, Spy, Sdy, diy);
    gather_weights<ORD>(oz, quirk2, Spz, Sdz, diz);
    constexpr int N0 = GatherRange<ORD>::N0, N1 = GatherRange<ORD>::N1, NB = N1 - N0;
    constexpr int NR = NB * NB;          // node rows (y, z) of the block
    constexpr int NBATCH = NR / RB;
    constexpr int BW = RB * NB;          // nodes per batch
#pragma unroll
    for (int q = 0; q < 6; ++q) E[q] = 0.0f;
    const int n0 = (i - 1) + FX * ((j - 1) + FY * (k - 1));
    static_assert(NB % 2 == 0, "node pairs");
    const float4* p4 = s4 + n0;
    const float4* pp = sp + n0;
    // the reads of batch n + 1 are issued before batch n is summed, so a
    // wave waits for LDS once per batch instead of once per node
    float4 b4[2][BW];
    float4 b2[2][BW / 2];
    auto load = [&](int n, float4* d4, float4* d2) {
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            const int r = n * RB + rr;
            const int b = N0 + r % NB, c = N0 + r / NB;
            const int row = FX * (b + FY * c) + N0;
#pragma unroll
            for (int t = 0; t < NB; ++t) d4[rr * NB + t] = p4[row + t];
#pragma unroll
            for (int t = 0; t < NB; t += 2) d2[(rr * NB + t) / 2] = pp[row + t];
        }
    };
    load(0, b4[0], b2[0]);
    // a z plane of the block is summed with the x-y weights, then scaled by
    // its z weight: NB*NB products plus 6 (NB^3 + NB) multiply-adds
    float wxy[NB][NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int t = 0; t < NB; ++t) wxy[b][t] = Spx[N0 + t] * Spy[N0 + b];
    float acc[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int n = 0; n < NBATCH; ++n) {
        if (n + 1 < NBATCH) load(n + 1, b4[(n + 1) & 1], b2[(n + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        const float4* d4 = b4[n & 1];
        const float4* d2 = b2[n & 1];
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            const int r = n * RB + rr;
            const int b = r % NB, c = r / NB;
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                const float w = wxy[b][t];
                const float4 a = d4[rr * NB + t];
                const float4 pr = d2[(rr * NB + t) / 2];
                const float2 m = (t & 1) ? make_float2(pr.z, pr.w) : make_float2(pr.x, pr.y);
                acc[0] = fmaf(a.x, w, acc[0]);
                acc[1] = fmaf(a.y, w, acc[1]);
                acc[2] = fmaf(a.z, w, acc[2]);
                acc[3] = fmaf(a.w, w, acc[3]);
                acc[4] = fmaf(m.x, w, acc[4]);
                acc[5] = fmaf(m.y, w, acc[5]);
            }
            if (b == NB - 1) {
                const float wz = Spz[N0 + c];
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                    E[q] = fmaf(acc[q], wz, E[q]);
                    acc[q] = 0.0f;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// gather3_lds<2> with the reference's loop range, away from offsets of 0: the
// primal weights then leave only nodes 0 and 1 of each axis, 8 of the 64
// nodes; the same products in the same order
template <int FX, int FY>
__device__ __forceinline__ void gather3_quirk2(const float4* __restrict__ s4, const float4* __restrict__ sp, int i,
                                               int j, int k, float ox, float oy, float oz, float* E)
{
    float Px[2], Py[2], Pz[2], D[3];
    AxisW<2, true>::w(ox, Px, D);
    AxisW<2, true>::w(oy, Py, D);
    AxisW<2, true>::w(oz, Pz, D);
    const int n0 = i + FX * (j + FY * k);
#pragma unroll
    for (int q = 0; q < 6; ++q) E[q] = 0.0f;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        float acc[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int n = n0 + FX * (b + FY * c);
            const float4 f0 = s4[n], f1 = s4[n + 1], m = sp[n];
            const float w0 = Px[0] * Py[b], w1 = Px[1] * Py[b];
            acc[0] = fmaf(f1.x, w1, fmaf(f0.x, w0, acc[0]));
            acc[1] = fmaf(f1.y, w1, fmaf(f0.y, w0, acc[1]));
            acc[2] = fmaf(f1.z, w1, fmaf(f0.z, w0, acc[2]));
            acc[3] = fmaf(f1.w, w1, fmaf(f0.w, w0, acc[3]));
            acc[4] = fmaf(m.z, w1, fmaf(m.x, w0, acc[4]));
            acc[5] = fmaf(m.w, w1, fmaf(m.y, w0, acc[5]));
        }
#pragma unroll
        for (int q = 0; q < 6; ++q) E[q] = fmaf(acc[q], Pz[c], E[q]);
    }
}

// Esirkepov deposit of one particle from old cell (i,j,k) / offsets o*, with
// displacement d*, charge q.  The stored current follows the reference's
// sign (E += cur): x current at node a = q * sum_{a'<=a} dSx(a') *
// (Ay Az + dSy dSz/12), A = S1 + dS/2, which is the reference's
// S1 S1 + dS S1/2 + S1 dS/2 + dS dS/3.  The last node of each prefix sum is
// the telescoped zero and is not written.
template <int DIM, int ORD, class Sink>
__device__ __forceinline__ void deposit(const Sink& snk, int i, int j, int k, float ox, float oy, float oz,
                                        float dx, float dy, float dz, float q)
{
    constexpr int W = Win<ORD>::W;
    float S1x[W], dSx[W], S1y[W], dSy[W];
    const int bx = axis_deposit<ORD>(ox, dx, S1x, dSx);
    const int by = axis_deposit<ORD>(oy, dy, S1y, dSy);
    float Ax[W], Ay[W], Cx[W], Cy[W];
    float run_x = 0.0f, run_y = 0.0f;
#pragma unroll
    for (int t = 0; t < W; ++t) {
        Ax[t] = S1x[t] + 0.5f * dSx[t];
        Ay[t] = S1y[t] + 0.5f * dSy[t];
        run_x += dSx[t];
        run_y += dSy[t];
        Cx[t] = q * run_x;
        Cy[t] = q * run_y;
    }
    const float twelfth = 1.0f / 12.0f;
    int cc[W];
#pragma unroll
    for (int t = 0; t < W; ++t) cc[t] = snk.col(i + bx + t);
    if (DIM == 3) {
        float S1z[W], dSz[W], Az[W], Cz[W];
        const int bz = axis_deposit<ORD>(oz, dz, S1z, dSz);
        float run_z = 0.0f;
#pragma unroll
        for (int t = 0; t < W; ++t) {
            Az[t] = S1z[t] + 0.5f * dSz[t];
            run_z += dSz[t];
            Cz[t] = q * run_z;
        }
#pragma unroll
        for (int c = 0; c < W; ++c) {
#pragma unroll
            for (int b = 0; b < W; ++b) {
                const auto r = snk.row(j + by + b, k + bz + c);
                const float wyz = Ay[b] * Az[c] + twelfth * dSy[b] * dSz[c];
#pragma unroll
                for (int t = 0; t < W; ++t) {
                    if (t < W - 1) {
                        const float v = Cx[t] * wyz;
                        if (v != 0.0f) snk.add(0, r, cc[t], v);
                    }
                    if (b < W - 1) {
                        const float v = Cy[b] * (Ax[t] * Az[c] + twelfth * dSx[t] * dSz[c]);
                        if (v != 0.0f) snk.add(1, r, cc[t], v);
                    }
                    if (c < W - 1) {
                        const float v = Cz[c] * (Ax[t] * Ay[b] + twelfth * dSx[t] * dSy[b]);
                        if (v != 0.0f) snk.add(2, r, cc[t], v);
                    }
                }
            }
        }
    } else {
        // 2D: Jz directly from the z displacement (code/particles.F90:822-848)
        const float qdz = -q * dz;
#pragma unroll
        for (int b = 0; b < W; ++b) {
            const auto r = snk.row(j + by + b, 0);
#pragma unroll
            for (int t = 0; t < W; ++t) {
                if (t < W - 1) {
                    const float v = Cx[t] * Ay[b];
                    if (v != 0.0f) snk.add(0, r, cc[t], v);
                }
                if (b < W - 1) {
                    const float v = Cy[b] * Ax[t];
                    if (v != 0.0f) snk.add(1, r, cc[t], v);
                }
                const float v = qdz * (Ax[t] * Ay[b] + twelfth * dSx[t] * dSy[b]);
                if (v != 0.0f) snk.add(2, r, cc[t], v);
            }
        }
    }
}

// ------------------------------------------------- the original scheme
// The -Dzzag build of the reference: its mover interpolates the staggered
// fields trilinearly with the half-cell staggering folded in
// (code/particles_movedeposit.F90:98-347) and its deposit is the zigzag
// scheme of Umeda et al. 2003 (code/particles.F90:550-669).

// E, B at the particle for the zigzag mover: the staggered component along an
// axis is the two half-cell neighbours' sum plus the offset times their
// difference across two cells, then bilinear in the other axes (E) or
// summed once more over the second staggered axis (B).  In 2D every z offset
// is the particle's own plane.  The sums carry a factor 2 (E) and 4 (B),
// removed here, so E[] is on the scale of gather()'s output.
template <int DIM, class Src>
__device__ __forceinline__ void gather_zz(const Src& src, int i, int j, int k, float dx, float dy, float dz,
                                          float* E)
{
    auto at = [&](int q, int a, int b, int c) {
        return src.get(q, src.row(j + b, DIM == 3 ? k + c : 0), src.col(i + a));
    };
    auto sx = [&](int q, int b, int c) {
        return at(q, 0, b, c) + at(q, -1, b, c) + dx * (at(q, 1, b, c) - at(q, -1, b, c));
    };
    auto sy = [&](int q, int a, int c) {
        return at(q, a, 0, c) + at(q, a, -1, c) + dy * (at(q, a, 1, c) - at(q, a, -1, c));
    };
    auto sz = [&](int q, int a, int b) {
        return at(q, a, b, 0) + at(q, a, b, -1) + dz * (at(q, a, b, 1) - at(q, a, b, -1));
    };
    auto lerp = [](float p, float r, float t) { return p + t * (r - p); };
    const float ex = lerp(lerp(sx(0, 0, 0), sx(0, 1, 0), dy), lerp(sx(0, 0, 1), sx(0, 1, 1), dy), dz);
    const float ey = lerp(lerp(sy(1, 0, 0), sy(1, 0, 1), dz), lerp(sy(1, 1, 0), sy(1, 1, 1), dz), dx);
    const float ez = lerp(lerp(sz(2, 0, 0), sz(2, 1, 0), dx), lerp(sz(2, 0, 1), sz(2, 1, 1), dx), dy);
    // Bx: staggered in y and z; By: in z and x; Bz: in x and y
    float f = sz(3, 0, 0) + sz(3, 0, -1) + dy * (sz(3, 0, 1) - sz(3, 0, -1));
    float g = sz(3, 1, 0) + sz(3, 1, -1) + dy * (sz(3, 1, 1) - sz(3, 1, -1));
    const float bx = lerp(f, g, dx);
    f = sx(4, 0, 0) + sx(4, 0, -1) + dz * (sx(4, 0, 1) - sx(4, 0, -1));
    g = sx(4, 1, 0) + sx(4, 1, -1) + dz * (sx(4, 1, 1) - sx(4, 1, -1));
    const float by = lerp(f, g, dy);
    f = sy(5, 0, 0) + sy(5, -1, 0) + dx * (sy(5, 1, 0) - sy(5, -1, 0));
    g = sy(5, 0, 1) + sy(5, -1, 1) + dx * (sy(5, 1, 1) - sy(5, -1, 1));
    const float bz = lerp(f, g, dz);
    E[0] = 0.5f * ex;
    E[1] = 0.5f * ey;
    E[2] = 0.5f * ez;
    E[3] = 0.25f * bx;
    E[4] = 0.25f * by;
    E[5] = 0.25f * bz;
}

// relay point of one axis (positions relative to the old cell: a1 in [0,1),
// a2 = a1 + displacement, in cell n2 = floor(a2)): the midpoint, clamped to
// the cell boundary the move crosses
__device__ __forceinline__ float zz_relay(float a1, float a2, int n2)
{
    const float lo = (float)((n2 < 0 ? n2 : 0) + 1), hi = (float)(n2 > 0 ? n2 : 0);
    return fminf(lo, fmaxf(hi, 0.5f * (a1 + a2)));
}

// zigzag deposit of one particle from old cell (i,j,k) / offsets o*, with
// displacement d*, charge q: each half of the move (start -> relay, relay ->
// end) deposits its flux with area weights at its centre.  Same stored sign
// as deposit() (E += cur).  In 2D, z only splits the z flux at the relay
// point (the reference tracks z modulo one cell there).
template <int DIM, class Sink>
__device__ __forceinline__ void deposit_zz(const Sink& snk, int i, int j, int k, float ox, float oy, float oz,
                                           float dx, float dy, float dz, float q)
{
    const float x2 = ox + dx, y2 = oy + dy, z2 = oz + dz;
    const int i2 = (int)floorf(x2), j2 = (int)floorf(y2), k2 = (int)floorf(z2);
    const float xr = zz_relay(ox, x2, i2), yr = zz_relay(oy, y2, j2), zr = zz_relay(oz, z2, k2);
    const float fx1 = -q * (xr - ox), fy1 = -q * (yr - oy), fz1 = -q * (zr - oz);
    const float fx2 = -q * (x2 - xr), fy2 = -q * (y2 - yr), fz2 = -q * (z2 - zr);
    const float wx1 = 0.5f * (ox + xr), wy1 = 0.5f * (oy + yr);
    const float wx2 = 0.5f * (x2 + xr) - (float)i2, wy2 = 0.5f * (y2 + yr) - (float)j2;
    const float wz1 = DIM == 3 ? 0.5f * (oz + zr) : 0.0f;
    const float wz2 = DIM == 3 ? 0.5f * (z2 + zr) - (float)k2 : 0.0f;
    // both halves of a move within one cell add to the same 12 (8) nodes: one
    // addition each of the exact sum of the two (80x64x48 cells, 8 per cell:
    // 229 -> 189 us with the tiles in cell order, 180 -> 171 without)
    const bool stays = (i2 | j2 | (DIM == 3 ? k2 : 0)) == 0;
    auto half = [&](int ci, int cj, int ck, auto put) {
        const auto r00 = snk.row(cj, ck), r10 = snk.row(cj + 1, ck);
        const int c0 = snk.col(ci), c1 = snk.col(ci + 1);
        put(0, r00, c0, [](float fx, float, float, float, float wy, float wz) { return fx * (1.0f - wy) * (1.0f - wz); });
        put(0, r10, c0, [](float fx, float, float, float, float wy, float wz) { return fx * wy * (1.0f - wz); });
        put(1, r00, c0, [](float, float fy, float, float wx, float, float wz) { return fy * (1.0f - wx) * (1.0f - wz); });
        put(1, r00, c1, [](float, float fy, float, float wx, float, float wz) { return fy * wx * (1.0f - wz); });
        if (DIM == 3) {
            const auto r01 = snk.row(cj, ck + 1), r11 = snk.row(cj + 1, ck + 1);
            put(0, r01, c0, [](float fx, float, float, float, float wy, float wz) { return fx * (1.0f - wy) * wz; });
            put(0, r11, c0, [](float fx, float, float, float, float wy, float wz) { return fx * wy * wz; });
            put(1, r01, c0, [](float, float fy, float, float wx, float, float wz) { return fy * (1.0f - wx) * wz; });
            put(1, r01, c1, [](float, float fy, float, float wx, float, float wz) { return fy * wx * wz; });
        }
        put(2, r00, c0, [](float, float, float fz, float wx, float wy, float) { return fz * (1.0f - wx) * (1.0f - wy); });
        put(2, r00, c1, [](float, float, float fz, float wx, float wy, float) { return fz * wx * (1.0f - wy); });
        put(2, r10, c0, [](float, float, float fz, float wx, float wy, float) { return fz * (1.0f - wx) * wy; });
        put(2, r10, c1, [](float, float, float fz, float wx, float wy, float) { return fz * wx * wy; });
    };
    half(i, j, DIM == 3 ? k : 0, [&](int q, auto r, int col, auto part) {
        const float v1 = part(fx1, fy1, fz1, wx1, wy1, wz1), v2 = part(fx2, fy2, fz2, wx2, wy2, wz2);
        snk.add(q, r, col, (double)v1 + (double)(stays ? v2 : 0.0f));
    });
    if (stays) return;
    half(i + i2, j + j2, DIM == 3 ? k + k2 : 0, [&](int q, auto r, int col, auto part) {
        snk.add(q, r, col, part(fx2, fy2, fz2, wx2, wy2, wz2));
    });
}

}  // namespace tmpg
