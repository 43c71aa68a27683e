// push_common.h -- what the push kernels share: their arguments, the
// particle's load, store and emit into the tile it lands in, the momentum
// push, and the shape profiles of the per-cell register sums.
#pragma once
#include "pic_push.h"
#include "tmpg_internal.h"

namespace tmpg {

struct SpecArgs {
    float qm, q;
    int32_t tcap;
    int64_t ocap;
    PBuf a, b, ob;
    const int32_t* cnt_a;
    int32_t* cnt_b;
    int32_t* olist;         // entries of ob
    int32_t* lost;
};

struct TiledArgs {
    int nx, ny, nz;
    PackInfo pk;
    Tiling tl;
    int fo;                 // field region origin: tile origin - fo
    int FX, FY, FZ;         // staged field region
    int JX, JY, JZ;         // LDS current region (origin: tile origin - 2)
    float c, cinv;
    int flags;              // PUSH_GATHER2 | PUSH_VAY
    int remap;              // XCD-aware tile order
    const float* f6[6];
    float* j3[3];
    SpecArgs sp[2];
    Stamp st;
};

struct Part {
    int i, j, k;
    float ox, oy, oz, u, v, w, ch;
    int32_t id;
};

template <int DIM, bool HAS_CH, bool HAS_ID>
__device__ __forceinline__ void load_part(const PBuf& b, int64_t s, const PackInfo& pk, Part& p)
{
    unpack_cell(pk, b.cell[s], p.i, p.j, p.k);
    p.ox = b.ox[s];
    p.oy = b.oy[s];
    // 2D keeps a z offset only in the zigzag scheme (b.oz allocated)
    p.oz = (DIM == 3 || b.oz != nullptr) ? b.oz[s] : 0.0f;
    p.u = b.u[s];
    p.v = b.v[s];
    p.w = b.w[s];
    p.ch = HAS_CH ? b.ch[s] : 1.0f;
    p.id = HAS_ID ? b.id[s] : 0;
}

template <int DIM, bool HAS_CH, bool HAS_ID>
__device__ __forceinline__ void store_part(const PBuf& b, int64_t s, const PackInfo& pk, const Part& p)
{
    b.cell[s] = pack_cell(pk, p.i, p.j, p.k);
    b.ox[s] = p.ox;
    b.oy[s] = p.oy;
    if (DIM == 3 || b.oz != nullptr) b.oz[s] = p.oz;
    b.u[s] = p.u;
    b.v[s] = p.v;
    b.w[s] = p.w;
    if (HAS_CH) b.ch[s] = p.ch;
    if (HAS_ID) b.id[s] = p.id;
}

// write a pushed particle to slot `slot` of tile `t` in b, or to the
// overflow list when the segment is full; returns the index used
// (t*tcap+slot, or slots + list index, or -1 when lost)
template <int DIM, bool HAS_CH, bool HAS_ID>
__device__ __forceinline__ int64_t emit(const SpecArgs& s, const PackInfo& pk, int64_t slots, int64_t t,
                                        int32_t slot, const Part& p)
{
    if (slot < s.tcap) {
        const int64_t d = t * s.tcap + slot;
        store_part<DIM, HAS_CH, HAS_ID>(s.b, d, pk, p);
        return d;
    }
    const int oi = atomicAdd(s.olist, 1);
    if (oi < s.ocap) {
        store_part<DIM, HAS_CH, HAS_ID>(s.ob, oi, pk, p);
        return slots + oi;
    }
    atomicAdd(s.lost, 1);
    return -1;
}

// push flags: the 2nd-order gather quirk; the Vay pusher instead of Boris
constexpr int PUSH_GATHER2 = 1, PUSH_VAY = 2;

// field gather and momentum push of p; returns the displacement.
// VAY_OK = false compiles the Boris push only (the Boris instantiations of
// the 3D cell-sum kernel, whose register budget is tight)
template <bool VAY_OK = true>
__device__ __forceinline__ void push_fields(const float* E, int flags, float c, float cinv, float qm, Part& p,
                                            float& dx, float& dy, float& dz)
{
    const float se = 0.5f * qm, sb = 0.5f * qm * cinv;
    if (VAY_OK && (flags & PUSH_VAY))
        vay(c, cinv, se * E[0], se * E[1], se * E[2], sb * E[3], sb * E[4], sb * E[5], p.u, p.v, p.w, dx, dy, dz);
    else
        boris(c, cinv, se * E[0], se * E[1], se * E[2], sb * E[3], sb * E[4], sb * E[5], p.u, p.v, p.w, dx, dy,
              dz);
}

__device__ __forceinline__ void advance(Part& p, int dim, int nx, int ny, int nz, float dx, float dy, float dz,
                                        bool z_offset_2d = false)
{
    p.i = wrap1(p.i + advance_offset(p.ox, dx), nx);
    p.j = wrap1(p.j + advance_offset(p.oy, dy), ny);
    if (dim == 3) p.k = wrap1(p.k + advance_offset(p.oz, dz), nz);
    // the 2D zigzag scheme tracks z modulo one cell, like the reference's
    // wrap of z into its single plane (code/particles_movedeposit.F90:1553-1633)
    else if (z_offset_2d) (void)advance_offset(p.oz, dz);
}

// place the W window values starting at node `base` into an NW-node window
// starting at node `first` (values outside are dropped: callers guarantee
// they are zero)
template <int W, int NW>
__device__ __forceinline__ void place(const float* v, int base, int first, float* out)
{
#pragma unroll
    for (int s = 0; s < NW; ++s) {
        float acc = 0.0f;
#pragma unroll
        for (int t = 0; t < W; ++t) acc = (s == base - first + t) ? v[t] : acc;
        out[s] = acc;
    }
}

// Shape profile of one axis of a cell-summed record on nodes [-2,3] (cell
// crossings included): S = old weights, dS = new - old.  Order 3 writes the
// pieces straight into their slots: the old piece is the particle's own cell
// (m0 = 0), the new one is m1 = floor(o + d) in {-1, 0, 1}, and a crossing
// splits dS at the knot K = max(m0, m1) exactly as axis_deposit does.  Other
// orders go through axis_deposit and place the window.
template <int ORD>
__device__ __forceinline__ void profile6(float o, float d, float* S6, float* dS6)
{
    if constexpr (ORD == 3) {
        using P = Piece<3>;
        float w[4], t0[4], t1[4];
        P::w(o, w);
        const int m1 = (int)floorf(o + d);
        const float K = (m1 > 0) ? 1.0f : 0.0f;
        const float b0 = (m1 == 0) ? o + d : K;
        const float d0 = (m1 == 0) ? d : K - o;
        P::dw(o, b0, d0, t0);
        // second segment on piece m1 (length zero, so all zero, without a crossing)
        const float d2 = d - d0;
        const float a1 = K - (float)m1;
        P::dw(a1, a1 + d2, d2, t1);
#pragma unroll
        for (int u = 0; u < 6; ++u) {
            S6[u] = (u >= 1 && u <= 4) ? w[u - 1] : 0.0f;
            const float v = (u >= 1 && u <= 4) ? t0[u - 1] : 0.0f;
            const float up = (u >= 2) ? t1[u - 2] : 0.0f;    // m1 = +1: nodes 0..3
            const float dn = (u <= 3) ? t1[u] : 0.0f;        // m1 = -1: nodes -2..1
            dS6[u] = v + ((m1 > 0) ? up : dn);
        }
    } else {
        constexpr int W = Win<ORD>::W;
        float S1[W], dS[W];
        const int b = axis_deposit<ORD>(o, d, S1, dS);
        place<W, 6>(S1, b, -2, S6);
        place<W, 6>(dS, b, -2, dS6);
    }
}

// y/z shape window of a move inside nodes [-1,2]?
template <int ORD>
__device__ __forceinline__ bool fits4(float o, float d)
{
    const int m0 = piece_of<ORD>(o), m1 = piece_of<ORD>(o + d);
    const int lo = (m0 < m1 ? m0 : m1) + Piece<ORD>::first;
    const int hi = (m0 > m1 ? m0 : m1) + Piece<ORD>::first + Piece<ORD>::cnt - 1;
    return lo >= -1 && hi <= 2;
}

// Shape profile of one axis (S = old weights, dS = new - old) on nodes
// -1..2: the window of every move of orders 1 (|d| < 1) and 2 (inside
// (-1/2, 3/2), which every move of less than half a cell keeps), and of
// order 3 without a cell crossing.  dS is split at the knot that the move
// crosses, as in axis_deposit.
template <int ORD>
__device__ __forceinline__ void window4(float o, float d, float* S, float* dS)
{
    if constexpr (ORD == 1) {
        const float x1 = o + d;
        const bool up = x1 >= 1.0f, dn = x1 < 0.0f;
        const float d0 = up ? 1.0f - o : (dn ? -o : d);   // to the cell's edge
        const float d2 = d - d0;                          // beyond it (zero without a crossing)
        S[0] = 0.0f;
        S[1] = 1.0f - o;
        S[2] = o;
        S[3] = 0.0f;
        const float u2 = up ? d2 : 0.0f, n2 = dn ? d2 : 0.0f;
        dS[0] = -n2;
        dS[1] = n2 - d0;
        dS[2] = d0 - u2;
        dS[3] = u2;
    } else if constexpr (ORD == 2) {
        using P = Piece<2>;
        const bool p0 = o > 0.5f, p1 = o + d > 0.5f;      // pieces 0 or 1 of the old and the new position
        const float m0 = p0 ? 1.0f : 0.0f, m1 = p1 ? 1.0f : 0.0f;
        const bool same = p0 == p1;
        const float d0 = same ? d : 0.5f - o;
        const float a0 = o - m0, b0 = same ? a0 + d : 0.5f - m0;
        const float d2 = d - d0, a1 = 0.5f - m1;
        float w[3], t0[3], t1[3];
        P::w(a0, w);
        P::dw(a0, b0, d0, t0);
        P::dw(a1, a1 + d2, same ? 0.0f : d2, t1);
        S[0] = p0 ? 0.0f : w[0];
        S[1] = p0 ? w[0] : w[1];
        S[2] = p0 ? w[1] : w[2];
        S[3] = p0 ? w[2] : 0.0f;
        dS[0] = (p0 ? 0.0f : t0[0]) + (p1 ? 0.0f : t1[0]);
        dS[1] = (p0 ? t0[0] : t0[1]) + (p1 ? t1[0] : t1[1]);
        dS[2] = (p0 ? t0[1] : t0[2]) + (p1 ? t1[1] : t1[2]);
        dS[3] = (p0 ? t0[2] : 0.0f) + (p1 ? t1[2] : 0.0f);
    } else {
        Piece<3>::w(o, S);
        Piece<3>::dw(o, o + d, d, dS);
    }
}

// push2d.hip: the 2D push in cell order, for the tilings, slots per species
// and Courant numbers that push2d_serves accepts
bool push2d_serves(const Tiling& tl, int64_t slots, int order, float c);
bool push2d_launch(const TiledArgs& a, int order, bool ch, bool id, hipStream_t st);

}  // namespace tmpg
