// The ring march with two threads per cell column: one advances density and velocity (the flow group),
// the other entropy and the magnetic potential (the field group). The FP64 solve (variant 8).
//
// With one thread per column (ZMarchRing, the FP32 form) FP64 takes all 512 registers of a lane, 88
// values move to accumulation registers and back every plane, and a single wave per SIMD issues a
// vector instruction every 6.5 to 8.7 cycles, where two waves issue one every 4.4 to 5 (measured).
// Half a column fits 256 registers with nothing spilled: two waves per SIMD share the issue slots and
// cover each other's waits. The groups need little of each other, seven values of a cell one way and
// six the other, through LDS at the cost of a second barrier per plane.
//
// LDS holds the fields in pairs, a cell's two values side by side, so that every stencil read is 16
// aligned bytes a lane, half as many reads as values, and one base register serves a whole slot. With
// 8-byte reads LDS was busy for 60 % of a plane's time.
//
// What bounds it: a lone block takes 2.55 us a plane, about 45 % of it VALU issue and 45 % LDS, which the
// barriers keep from overlapping fully (offsetting the groups by half a plane gained 2 % on a full chip
// and cost a four-plane column 15 %). On a full chip the clock drops from 2.4 to 2.0 GHz; at 512^3 a
// launch of substeps 1 and 2 moves 29.5 GB at 4.0 TB/s, 85 % of what a plain copy of 4 GiB reaches, and
// substep 0 20.8 GB at 3.3 TB/s. Per launch, sustained, mean of the three substeps (us), one thread per
// column -> this: 32^3 16.5 -> 12.1, 64^3 26.7 -> 22.0, 150 x 33 x 110 65 -> 42.6, 128^3 140 -> 113, 256^3
// 1020 -> 867, 512^3 8160 -> 7020.
#pragma once
#include "physics.h"

namespace ac {
namespace {

// As in the other march, every multiply-add is written out.
#pragma clang fp contract(off)

// FIRST: the build of substep 0, which has no previous stage.
template <int TX, int TY, bool COMP, bool FIRST> struct ZMarchPair {
    static constexpr int NC = TX * TY, NT = 2 * NC; // cell columns, threads
    static_assert(NC % 64 == 0, "whole waves");
    static constexpr int NG = NF / 2; // fields of a group: a vector and a scalar, in this order
    static constexpr int LX = TX + 6, LY = TY + 6, LN = LX * LY;
    static constexpr int R     = (LN + NC - 1) / NC; // staging rounds per field and plane
    // One tile row, in field pairs. With 16-wide tiles a multiple of 256 bytes, so that 16 lanes of one row
    // and 16 of the next, which a 16-byte read serves together, lie in different banks (88 pairs,
    // unpadded: 64^3 in whole columns 199 us, 96: 180). A wider tile's row fills the banks by itself.
    static constexpr int PITCH = TX % 32 ? (NF / 2 * LX + 15) / 16 * 16 : NF / 2 * LX;

    // Two fields of a cell. A group's pairs: vector x and y; vector z and the scalar.
    typedef AcReal Two __attribute__((ext_vector_type(2)));

    struct Shared {
        Two ring[4][LY * PITCH]; // [slot][row][pair][x]
        AcReal flow[7][NC], field[6][NC];
    };

    struct State {
        AcReal q[NG][3];  // planes z-3..z-1, plane p in slot p mod 3 (counted from the first output)
        AcReal x[3][3];   // cross sums of outputs z..z+2, output o in slot o mod 3
        AcReal pv[NG][R]; // the next plane, on its way from global memory to the ring
        AcReal cur[NG];   // output z: values
        AcReal sg[3], slap; // the scalar's gradient and Laplacian
        AcReal vg[3][3];    // the vector's first derivatives [component][axis]
        // its second derivatives along each component's own axis and along the other two, and the cross
        // derivatives of grad div, which the second derivatives join last: they are the largest terms
        AcReal own[3], rest[3], gd[3];
        AcReal prev[FIRST ? 1 : NG];           // output z: previous stage
        AcReal cin[COMP ? NG : 1];             // rounding errors (compensated integration),
        AcReal cprev[COMP && !FIRST ? NG : 1]; // and those of the previous stage
        int s0, s1, s2, s3; // first element of the ring slots of planes z..z+3 (uniform)
    };

    // The constants of the rates and the update, in vector registers: with the stencils' they exceed
    // the scalar ones, and what spills is read back lane by lane (78 v_readlane a plane; with these 36, in
    // substep 0 24; 256^3 948 -> 917 us).
    struct Constants {
        AcReal nu_visc, eta, inv_mu0, eta_mu0, inv_cp, gamma_inv_cp, gamma_m1, exp_lnT0, lnrho0, zeta, cs2_sound,
            k_thermal, dt, beta, ab;
    };

    const SubstepArgs& a;
    Shared& sh;
    int cofs, ze, lane;
    int group;   // 0: flow, 1: field (uniform in a wave)
    int image;   // ghost planes: n_z where they are read at their periodic images, else 0
    long fs, fv; // field 0 to the group's scalar and to its vector, in cells
    unsigned own;
    bool active;
    unsigned goff[R]; // byte offset in a plane of what this thread stages, per round
    int loff[R];      // its place in a ring slot (the group's first pair)

    __device__ __forceinline__ ZMarchPair(const SubstepArgs& args, Shared& shared) : a(args), sh(shared) {}

    typedef __attribute__((address_space(1))) AcReal GReal;
    typedef __attribute__((address_space(1))) const char GByte;
    typedef const Two __attribute__((address_space(3))) LdsTwo;

    // As in ZMarchRing: keeps LDS reads on their side; keeps a value's arithmetic where it stands.
    static __device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
    static __device__ __forceinline__ void settle_one(AcReal& v) { asm volatile("" : "+v"(v)); }
    template <typename... T> static __device__ __forceinline__ void settle(T&... v) { (settle_one(v), ...); }
    static __device__ __forceinline__ unsigned pin(unsigned off)
    {
        asm volatile("" : "+v"(off));
        return off;
    }
    static __device__ __forceinline__ AcReal ld(const AcReal* base, unsigned byte_off)
    {
        return *(const GReal*)((GByte*)base + byte_off);
    }
    static __device__ __forceinline__ void st_global(AcReal* base, unsigned byte_off, AcReal v)
    {
        *(GReal*)((GByte*)base + byte_off) = v;
    }
    // The group's first pair of the corner (-3, -3) of this thread's window in a ring slot, pinned: all
    // reads of the slot go through this one register with immediate offsets.
    __device__ __forceinline__ const LdsTwo* window(int slot) const
    {
        unsigned addr = (unsigned)(size_t)(const LdsTwo*)(&sh.ring[0][0] + slot + (cofs - 3 * PITCH - 3));
        asm volatile("" : "+v"(addr));
        return (const LdsTwo*)(size_t)addr;
    }
    static __device__ __forceinline__ Two at(const LdsTwo* w, int pair, int dx, int dy)
    {
        return w[(dy + 3) * PITCH + pair * LX + dx + 3];
    }
    static __device__ __forceinline__ AcReal one(const LdsTwo* w, int f, int dx, int dy)
    {
        return ((const AcReal __attribute__((address_space(3)))*)(w + (dy + 3) * PITCH + (f >> 1) * LX + dx + 3))[f & 1];
    }

    // Cells from one field to the next (SubstepArgs::stride). Read anew at every use: left to
    // itself the compiler keeps all sixteen field pointers, 32 scalar registers that the stencil
    // and physics constants then spill for.
    __device__ __forceinline__ long field_stride() const
    {
        long s = a.stride;
        asm volatile("" : "+s"(s));
        return s;
    }

    __device__ __forceinline__ void load(AcReal (&pv)[NG][R], int p) const
    {
        int q = min(p, ze + 2);
        q += q < NGHOST ? image : q >= a.mz - NGHOST ? -image : 0;
        const AcReal* plane = a.in[0] + (long)q * a.mxy;
        unsigned go[R];
#pragma unroll
        for (int r = 0; r < R; ++r)
            go[r] = pin(goff[r]);
        each(plane, [&](int f, const AcReal* src) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                pv[f][r] = ld(src, go[r]);
        });
    }
    // Calls f(n, field) for the group's fields, from a place in field 0.
    template <typename P, typename F> __device__ __forceinline__ void each(P* place, F f) const
    {
        const long stride = field_stride();
        P* v              = place + fv;
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            f(n, v);
            v += stride;
        }
        f(3, place + fs);
    }

    __device__ __forceinline__ void stage(int slot, const AcReal (&pv)[NG][R]) const
    {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                sh.ring[0][slot + loff[r] + p * LX] = Two{pv[2 * p][r], pv[2 * p + 1][r]};
    }

    // A pair of fields along one axis: differences and sums at distance 1..3.
    struct Pairs {
        Two p[3], m[3];
    };
    template <int AXIS> static __device__ __forceinline__ Pairs pairs(const LdsTwo* w, int pair)
    {
        Pairs l;
#pragma unroll
        for (int i = 1; i <= 3; ++i) {
            l.m[i - 1] = AXIS == 0 ? at(w, pair, -i, 0) : at(w, pair, 0, -i);
            l.p[i - 1] = AXIS == 0 ? at(w, pair, i, 0) : at(w, pair, 0, i);
        }
        return l;
    }
    // The diagonal pairs of the x-y cross derivative.
    struct Diag {
        Two pp[3], mm[3], pm[3], mp[3];
    };
    static __device__ __forceinline__ Diag diag(const LdsTwo* w)
    {
        Diag d;
#pragma unroll
        for (int i = 1; i <= 3; ++i) {
            d.mm[i - 1] = at(w, 0, -i, -i);
            d.pm[i - 1] = at(w, 0, i, -i);
            d.mp[i - 1] = at(w, 0, -i, i);
            d.pp[i - 1] = at(w, 0, i, i);
        }
        return d;
    }

    struct Line {
        AcReal d[3], s[3];
    };
    static __device__ __forceinline__ Line line(const Pairs& l, int k)
    {
        Line r;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            r.d[i] = l.p[i][k] - l.m[i][k];
            r.s[i] = l.p[i][k] + l.m[i][k];
        }
        return r;
    }
    // Derivatives, their largest terms last, so that only the last sums are rounded at their size. Near
    // the diffusive limit of the time step this shows in a velocity's error: 1.79e-16 of the field
    // with the largest terms first, 1.72e-16 so (mean of 3 states of noise on a grid of 2 pi / 512, 2 steps).
    static __device__ __forceinline__ AcReal first(const Line& l, const AcReal* c)
    {
        return mad(c[1], l.d[0], mad(c[2], l.d[1], c[3] * l.d[2]));
    }
    static __device__ __forceinline__ AcReal second(const Line& l, AcReal v, const AcReal* c)
    {
        return mad(c[0], v, mad(c[1], l.s[0], mad(c[2], l.s[1], c[3] * l.s[2])));
    }
    static __device__ __forceinline__ AcReal cross(const Diag& d, int k, const AcReal* c)
    {
        AcReal t[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            t[i] = (d.pp[i][k] + d.mm[i][k]) - (d.pm[i][k] + d.mp[i][k]);
        return mad(c[1], t[0], mad(c[2], t[1], c[3] * t[2]));
    }

    // The differences of plane z, scattered with their weights into the cross sum n of the
    // outputs z+1, z+2 and z+3 (whose slot is that of output z, which has taken its sum).
    template <int PH>
    static __device__ __forceinline__ void scatter(State& st, int n, const AcReal* c, const AcReal* d, bool add)
    {
        st.x[n][(PH + 1) % 3] = mad(-c[1], d[0], st.x[n][(PH + 1) % 3]);
        st.x[n][(PH + 2) % 3] = mad(-c[2], d[1], st.x[n][(PH + 2) % 3]);
        if (add)
            st.x[n][PH] = mad(-c[3], d[2], st.x[n][PH]);
        else
            st.x[n][PH] = -(c[3] * d[2]);
        settle(st.x[n][0], st.x[n][1], st.x[n][2]);
    }

    // Planes below the first output: only their differences and values are needed.
    template <int PH> __device__ __forceinline__ void warm(State& st) const
    {
        const PhysParams& P = a.phys;
        const LdsTwo* w     = window(PH * LY * PITCH);
        auto dx             = [&](int f, int n, bool add) {
            AcReal d[3];
#pragma unroll
            for (int i = 1; i <= 3; ++i)
                d[i - 1] = one(w, f, i, 0) - one(w, f, -i, 0);
            scatter<PH>(st, n, P.cxz, d, add);
        };
        auto dy = [&](int f, int n, bool add) {
            AcReal d[3];
#pragma unroll
            for (int i = 1; i <= 3; ++i)
                d[i - 1] = one(w, f, 0, i) - one(w, f, 0, -i);
            scatter<PH>(st, n, P.cyz, d, add);
        };
        dx(2, 0, false);
        dy(2, 1, false);
        dx(0, 2, false);
        dy(1, 2, true);
#pragma unroll
        for (int f = 0; f < NG; ++f)
            st.q[f][PH] = one(w, f, 0, 0);
    }

    // The vector's pairs at distance I in plane z + I, for the cross sums: x and y pairs of component z,
    // x pair of x, y pair of y. Whole field pairs are read: 8-byte reads 16 bytes apart meet in the
    // same banks (64^3 in whole columns 180 us, whole pairs 171).
    struct Ahead {
        Two xz[2], yz[2], xx[2], yy[2];
    };
    template <int I> static __device__ __forceinline__ Ahead ahead(const LdsTwo* w)
    {
        Ahead h;
        h.xz[0] = at(w, 1, -I, 0), h.xz[1] = at(w, 1, I, 0);
        h.yz[0] = at(w, 1, 0, -I), h.yz[1] = at(w, 1, 0, I);
        h.xx[0] = at(w, 0, -I, 0), h.xx[1] = at(w, 0, I, 0);
        h.yy[0] = at(w, 0, 0, -I), h.yy[1] = at(w, 0, 0, I);
        return h;
    }
    static __device__ __forceinline__ AcReal difference(const Two* v, int k)
    {
        asm volatile("" : : "v"(v[0]), "v"(v[1])); // (keeps the reads whole)
        return v[1][k] - v[0][k];
    }
    static __device__ __forceinline__ void add_ahead(AcReal* sum, const Ahead& h, AcReal cx, AcReal cy)
    {
        sum[0] = mad(cx, difference(h.xz, 0), sum[0]);
        sum[1] = mad(cy, difference(h.yz, 0), sum[1]);
        sum[2] = mad(cx, difference(h.xx, 0), sum[2]);
        sum[2] = mad(cy, difference(h.yy, 1), sum[2]);
        settle(sum[0], sum[1], sum[2]);
    }

    // What a plane's work begins with, read at the end of the plane before it.
    struct Start {
        const LdsTwo* w;
        Two v;    // vector z and the scalar
        Pairs lx; // along x
    };
    __device__ __forceinline__ Start start(int slot) const
    {
        Start b;
        b.w  = window(slot);
        b.v  = at(b.w, 1, 0, 0);
        b.lx = pairs<0>(b.w, 1);
        return b;
    }

    // In-plane part of output plane z (ring slot PH; planes z+1, z+2 in the next two slots). The LDS
    // reads of each line are issued before the arithmetic of the line before it.
    template <int PH> __device__ __forceinline__ void in_plane(State& st, const Start& b) const
    {
        const PhysParams& P = a.phys;
        const LdsTwo* w     = b.w;
        const Pairs ly1     = pairs<1>(w, 1);
        fence();
#pragma unroll
        for (int n = 0; n < 3; ++n)
            st.gd[n] = st.x[n][PH];
        settle(st.gd[0], st.gd[1], st.gd[2]);
        {
            const Line lz = line(b.lx, 0), ls = line(b.lx, 1);
            st.cur[2] = b.v[0], st.cur[3] = b.v[1];
            st.vg[2][0] = first(lz, P.d1[0]);
            st.rest[2]  = second(lz, b.v[0], P.d2[0]);
            scatter<PH>(st, 0, P.cxz, lz.d, false);
            st.sg[0] = first(ls, P.d1[0]);
            st.slap  = second(ls, b.v[1], P.d2[0]);
            settle(st.vg[2][0], st.rest[2], st.sg[0], st.slap, st.cur[2], st.cur[3]);
        }
        fence();
        const Ahead h1 = ahead<1>(window(st.s1));
        fence();
        {
            const Line lz = line(ly1, 0), ls = line(ly1, 1);
            st.vg[2][1] = first(lz, P.d1[1]);
            st.rest[2] += second(lz, st.cur[2], P.d2[1]);
            scatter<PH>(st, 1, P.cyz, lz.d, false);
            st.sg[1] = first(ls, P.d1[1]);
            st.slap += second(ls, st.cur[3], P.d2[1]);
            settle(st.vg[2][1], st.rest[2], st.sg[1], st.slap);
        }
        fence();
        const Ahead h2 = ahead<2>(window(st.s2));
        fence();
        add_ahead(st.gd, h1, P.cxz[1], P.cyz[1]);
        fence();
        const Two v0    = at(w, 0, 0, 0);
        const Pairs lx0 = pairs<0>(w, 0);
        fence();
        add_ahead(st.gd, h2, P.cxz[2], P.cyz[2]);
        fence();
        const Pairs ly0 = pairs<1>(w, 0);
        fence();
        {
            const Line lx = line(lx0, 0), ly = line(lx0, 1); // x lines of the vector's x and y
            st.cur[0] = v0[0], st.cur[1] = v0[1];
            st.vg[0][0] = first(lx, P.d1[0]);
            st.own[0]   = second(lx, v0[0], P.d2[0]);
            scatter<PH>(st, 2, P.cxz, lx.d, false);
            st.vg[1][0] = first(ly, P.d1[0]);
            st.rest[1]  = second(ly, v0[1], P.d2[0]);
            settle(st.vg[0][0], st.own[0], st.vg[1][0], st.rest[1], st.cur[0], st.cur[1]);
        }
        fence();
        const Diag d = diag(w);
        fence();
        {
            const Line lx = line(ly0, 0), ly = line(ly0, 1); // y lines
            st.vg[0][1] = first(lx, P.d1[1]);
            st.rest[0]  = second(lx, st.cur[0], P.d2[1]);
            st.vg[1][1] = first(ly, P.d1[1]);
            st.own[1]   = second(ly, st.cur[1], P.d2[1]);
            scatter<PH>(st, 2, P.cyz, ly.d, true);
            settle(st.vg[0][1], st.rest[0], st.vg[1][1], st.own[1]);
        }
        fence();
        st.gd[1] += cross(d, 0, P.cxy);
        st.gd[0] += cross(d, 1, P.cxy);
        settle(st.gd[0], st.gd[1]);
    }

    template <int PH> static __device__ __forceinline__ Line zline(const State& st, int f, const AcReal* c)
    {
        const AcReal m[3] = {st.q[f][(PH + 2) % 3], st.q[f][(PH + 1) % 3], st.q[f][PH]};
        Line l;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            l.d[i] = c[i] - m[i];
            l.s[i] = c[i] + m[i];
        }
        return l;
    }

    // The previous stage at output plane z, a whole step before it is used.
    __device__ __forceinline__ void load_prev(State& st, int z) const
    {
        if (FIRST && !COMP)
            return;
        const unsigned long oz = (unsigned long)min(z, ze - 1) * a.mxy;
        const unsigned ow      = pin(own);
        if (!FIRST)
            each(a.out[0] + oz, [&](int n, const AcReal* p) { st.prev[n] = ld(p, ow); });
        if (COMP)
            each(a.cin[0] + oz, [&](int n, const AcReal* p) { st.cin[n] = ld(p, ow); });
        if (COMP && !FIRST)
            each(a.cout[0] + oz, [&](int n, const AcReal* p) { st.cprev[n] = ld(p, ow); });
    }

    // The groups' rates (mhd_rates_lean in two parts), before and after the barrier that both groups share
    // (in finish): what the other group needs is sent first; `keep` is what a group goes on with.
    // `os` is the other group's scalar, `u` its vector; rate[0..2] of the vector, rate[3] of the scalar.
    __device__ __forceinline__ void flow_send(const State& st, AcReal os, const Constants& K, AcReal (&keep)[9]) const
    {
        const AcReal(&ug)[3][3] = st.vg;
        const AcReal *lg = st.sg, lr = st.cur[3];
        const AcReal divu = ug[0][0] + ug[1][1] + ug[2][2];
        const AcReal t    = AcReal(2. / 3.) * divu;
        const AcReal D00 = mad(AcReal(2), ug[0][0], -t), D11 = mad(AcReal(2), ug[1][1], -t),
                     D22 = mad(AcReal(2), ug[2][2], -t);
        const AcReal D01 = ug[0][1] + ug[1][0], D02 = ug[0][2] + ug[2][0], D12 = ug[1][2] + ug[2][1];
        const AcReal rho     = fast_exp<AcReal>(lr);
        const AcReal inv_rho = fast_rcp<AcReal>(rho);
        const AcReal E       = fast_exp<AcReal>(mad(K.gamma_m1, lr - K.lnrho0, K.gamma_inv_cp * os));
        const AcReal cs2     = K.cs2_sound * E;
        const AcReal inv_pT  = inv_rho * fast_rcp<AcReal>(K.exp_lnT0 * E);
        const AcReal on      = mad(D22, D22, mad(D11, D11, D00 * D00));
        const AcReal off     = mad(D12, D12, mad(D02, D02, D01 * D01));
        const AcReal shear   = mad(K.zeta * divu, divu, K.nu_visc * mad(AcReal(0.5), on, off));
        AcReal* x            = &sh.flow[0][lane];
        x[0] = rho * shear, x[NC] = inv_rho, x[2 * NC] = inv_pT;
        x[3 * NC] = lg[0], x[4 * NC] = lg[1], x[5 * NC] = lg[2], x[6 * NC] = st.slap;
        keep[0] = D00, keep[1] = D11, keep[2] = D22, keep[3] = D01, keep[4] = D02, keep[5] = D12;
        keep[6] = divu, keep[7] = inv_rho, keep[8] = cs2;
    }
    __device__ __forceinline__ void flow_rates(const State& st, const Constants& K, const AcReal (&keep)[9],
                                               AcReal* rate) const
    {
        const AcReal(&ug)[3][3] = st.vg;
        const AcReal *lg = st.sg, *u = st.cur;
        const AcReal D[3][3] = {{keep[0], keep[3], keep[4]}, {keep[3], keep[1], keep[5]}, {keep[4], keep[5], keep[2]}};
        const AcReal divu = keep[6], inv_rho = keep[7], cs2 = keep[8];
        const AcReal* y     = &sh.field[0][lane];
        const AcReal jxB[3] = {y[0], y[NC], y[2 * NC]}, sg[3] = {y[3 * NC], y[4 * NC], y[5 * NC]};
        rate[3]             = -mad(u[2], lg[2], mad(u[1], lg[1], u[0] * lg[0])) - divu;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const AcReal gdu  = st.gd[r] + st.own[r];
            const AcReal visc = mad(AcReal(1. / 3.), gdu, st.own[r] + st.rest[r]) +
                                mad(D[r][2], lg[2], mad(D[r][1], lg[1], D[r][0] * lg[0]));
            AcReal du = -(ug[r][0] * u[0]);
            du        = mad(-ug[r][1], u[1], du);
            du        = mad(-ug[r][2], u[2], du);
            du        = mad(inv_rho, jxB[r], du);
            du        = mad(-cs2, mad(K.inv_cp, sg[r], lg[r]), du);
            du        = mad(K.nu_visc, visc, du);
            rate[r]   = mad(K.zeta, gdu, du);
        }
    }
    __device__ __forceinline__ void field_send(const State& st, const Constants& K, AcReal (&keep)[9]) const
    {
        const AcReal(&ag)[3][3] = st.vg;
        const AcReal* sg        = st.sg;
        const AcReal B[3] = {ag[2][1] - ag[1][2], ag[0][2] - ag[2][0], ag[1][0] - ag[0][1]};
        AcReal j[3];
#pragma unroll
        for (int r = 0; r < 3; ++r)
            j[r] = K.inv_mu0 * (st.gd[r] - st.rest[r]);
        AcReal* x = &sh.field[0][lane];
        x[0]      = mad(j[1], B[2], -(j[2] * B[1]));
        x[NC]     = mad(j[2], B[0], -(j[0] * B[2]));
        x[2 * NC] = mad(j[0], B[1], -(j[1] * B[0]));
        x[3 * NC] = sg[0], x[4 * NC] = sg[1], x[5 * NC] = sg[2];
#pragma unroll
        for (int r = 0; r < 3; ++r)
            keep[r] = B[r], keep[3 + r] = j[r];
    }
    __device__ __forceinline__ void field_rates(const State& st, const AcReal* u, const Constants& K,
                                                const AcReal (&keep)[9], AcReal* rate) const
    {
        const AcReal *sg = st.sg, *B = &keep[0], *j = &keep[3];
        const AcReal* y   = &sh.flow[0][lane];
        const AcReal heat = y[0], inv_rho = y[NC], inv_pT = y[2 * NC], lr_lap = y[6 * NC];
        const AcReal lg[3] = {y[3 * NC], y[4 * NC], y[5 * NC]};
        rate[0] = mad(K.eta, st.own[0] + st.rest[0], mad(u[1], B[2], -(u[2] * B[1])));
        rate[1] = mad(K.eta, st.own[1] + st.rest[1], mad(u[2], B[0], -(u[0] * B[2])));
        rate[2] = mad(K.eta, st.own[2] + st.rest[2], mad(u[0], B[1], -(u[1] * B[0])));
        const AcReal j2      = mad(j[2], j[2], mad(j[1], j[1], j[0] * j[0]));
        const AcReal heating = mad(K.eta_mu0, j2, heat);
        AcReal lnT           = mad(K.gamma_m1, lr_lap, K.gamma_inv_cp * st.slap); // lap lnT + |grad lnT|^2
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const AcReal gl = mad(K.gamma_inv_cp, sg[r], K.gamma_m1 * lg[r]);
            lnT             = mad(gl, gl, lnT);
        }
        const AcReal adv = mad(u[2], sg[2], mad(u[1], sg[1], u[0] * sg[0]));
        rate[3]          = mad(inv_pT, heating, mad(K.k_thermal * inv_rho, lnT, -adv));
    }

    // Output plane z: plane z+3 takes slot PH, then the rest of the derivatives, the rates and the
    // update. Ends with the first line of plane z+1 on its way.
    template <int PH> __device__ __forceinline__ void finish(State& st, int z, Start& b, const Constants& K) const
    {
        const PhysParams& P = a.phys;
        // the slot of plane z-1, which every thread left before the barrier in the rates
        stage(st.s3, st.pv);
        __syncthreads();
        load(st.pv, z + 4);

        const LdsTwo *w1 = window(st.s1), *w2 = window(st.s2), *w3 = window(st.s3);
        Two n[2][3];
#pragma unroll
        for (int p = 0; p < 2; ++p)
            n[p][0] = at(w1, p, 0, 0), n[p][1] = at(w2, p, 0, 0), n[p][2] = at(w3, p, 0, 0);
        const Ahead h3 = ahead<3>(w3);
        // the other group's values at this cell
        const LdsTwo* o = window(st.s0) + (group ? -2 : 2) * LX;
        const Two o0 = at(o, 0, 0, 0), o1 = at(o, 1, 0, 0);
        fence();
#pragma unroll
        for (int f = 0; f < NG; ++f) {
            const AcReal c[3] = {n[f >> 1][0][f & 1], n[f >> 1][1][f & 1], n[f >> 1][2][f & 1]};
            const Line l      = zline<PH>(st, f, c);
            const AcReal d = first(l, P.d1[2]), dd = second(l, st.cur[f], P.d2[2]);
            if (f < 2)
                st.vg[f][2] = d, st.rest[f] += dd;
            else if (f == 2)
                st.vg[2][2] = d, st.own[2] = dd;
            else
                st.sg[2] = d, st.slap += dd;
        }
        add_ahead(st.gd, h3, P.cxz[3], P.cyz[3]);
        settle(st.sg[2], st.slap, st.vg[0][2], st.rest[0], st.vg[1][2], st.rest[1], st.vg[2][2], st.own[2]);
        fence();
        AcReal rate[NG], keep[9];
        const AcReal ou[3] = {o0[0], o0[1], o1[0]};
        if (group == 0)
            flow_send(st, o1[1], K, keep);
        else
            field_send(st, K, keep);
        __syncthreads(); // one barrier of the whole block, which no branch between its waves contains
        if (group == 0)
            flow_rates(st, K, keep, rate);
        else
            field_rates(st, ou, K, keep, rate);
        settle(rate[0], rate[1], rate[2], rate[3]);
        fence();
        b = start(st.s1);
        fence();
        AcReal res[NG], err[COMP ? NG : 1];
#pragma unroll
        for (int f = 0; f < NG; ++f) {
            const AcReal u = st.cur[f];
            if (COMP) { // the pair (u, c), as in ZMarchRing
                const AcReal ci   = st.cin[f];
                const AcReal incr = FIRST ? K.dt * rate[f]
                                          : mad(K.dt, rate[f], K.ab * ((u - st.prev[f]) + (ci - st.cprev[f])));
                const AcReal d    = mad(K.beta, incr, ci);
                const AcReal sum  = u + d;
                const AcReal bb   = sum - u;
                err[f]            = (u - (sum - bb)) + (d - bb);
                res[f]            = sum;
            }
            else // the smaller product is the one that is rounded by itself
                res[f] = mad(K.beta, FIRST ? K.dt * rate[f] : mad(K.dt, rate[f], K.ab * (u - st.prev[f])), u);
            settle(res[f]);
        }
        load_prev(st, z + 1);
        if (active) {
            const unsigned long oz = (unsigned long)z * a.mxy;
            const unsigned ow      = pin(own);
            each(a.out[0] + oz, [&](int f, AcReal* p) { st_global(p, ow, res[f]); });
            if (COMP)
                each(a.cout[0] + oz, [&](int f, AcReal* p) { st_global(p, ow, err[f]); });
        }
#pragma unroll
        for (int f = 0; f < NG; ++f)
            st.q[f][PH] = st.cur[f];
        fence();
        const int s = st.s0;
        st.s0 = st.s1, st.s1 = st.s2, st.s2 = st.s3, st.s3 = s;
    }

    __device__ __forceinline__ void march(int zs) const
    {
        State st;
#pragma unroll
        for (int n = 0; n < 3; ++n)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                st.x[n][j] = 0;
        AcReal below[3][NG][R], ahead[3][NG][R];
#pragma unroll
        for (int j = 0; j < 3; ++j)
            load(below[j], zs - 3 + j);
#pragma unroll
        for (int j = 0; j < 3; ++j)
            load(ahead[j], zs + j);
        __syncthreads(); // the block's previous column is done with the ring
#pragma unroll
        for (int j = 0; j < 3; ++j)
            stage(j * LY * PITCH, below[j]);
        __syncthreads();
        warm<0>(st), warm<1>(st), warm<2>(st);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 3; ++j)
            stage(j * LY * PITCH, ahead[j]);
        load(st.pv, zs + 3);
        load_prev(st, zs);
        __syncthreads();
        st.s0 = 0, st.s1 = LY * PITCH, st.s2 = 2 * LY * PITCH, st.s3 = 3 * LY * PITCH;
        Start b = start(st.s0);
        Constants K{a.phys.nu_visc, a.phys.eta, a.phys.inv_mu0, a.phys.eta_mu0, a.phys.inv_cp, a.phys.gamma_inv_cp,
                    a.phys.gamma_m1, a.phys.exp_lnT0, a.phys.lnrho0, a.phys.zeta, a.phys.cs2_sound,
                    a.phys.k_thermal, a.rk.dt, a.rk.beta, a.rk.ab};
        settle(K.nu_visc, K.eta, K.inv_mu0, K.eta_mu0, K.inv_cp, K.gamma_inv_cp, K.gamma_m1, K.exp_lnT0, K.lnrho0, K.zeta,
               K.cs2_sound, K.k_thermal, K.dt, K.beta, K.ab);
        for (int z = zs;; ++z) { // ring phases 0, 1, 2; every branch is uniform
            in_plane<0>(st, b);
            finish<0>(st, z, b, K);
            if (++z == ze)
                break;
            in_plane<1>(st, b);
            finish<1>(st, z, b, K);
            if (++z == ze)
                break;
            in_plane<2>(st, b);
            finish<2>(st, z, b, K);
            if (z + 1 == ze)
                break;
        }
    }
};

// LATE is an option of the one-thread form.
template <int TX, int TY, bool COMP, bool FIRST, bool LATE = false> using RingColumn = ZMarchPair<TX, TY, COMP, FIRST>;

// One z-march column: tile (btx, bty) of box `a`, output planes [zs, min(zs + zdepth, end.z)).
template <int TX, int TY, bool COMP, bool FIRST, bool LATE = false>
__device__ __forceinline__ void
ring_column(const SubstepArgs& a, typename ZMarchPair<TX, TY, COMP, FIRST>::Shared& sh, const int btx, const int bty,
            const int zs, const int zdepth)
{
    typedef ZMarchPair<TX, TY, COMP, FIRST> K;
    K k(a, sh);
    k.group       = __builtin_amdgcn_readfirstlane((int)threadIdx.x / K::NC);
    const int tid = (int)threadIdx.x - k.group * K::NC;
    k.lane        = tid;
    k.fs          = k.group ? VTXBUF_ENTROPY * a.stride : VTXBUF_LNRHO * a.stride;
    k.fv          = (k.group ? VTXBUF_AX : VTXBUF_UUX) * a.stride;
    const int tx = tid % TX, ty = tid / TX;
    const int x0 = a.start.x + btx * TX, y0 = a.start.y + bty * TY;
    const int gx = x0 + tx, gy = y0 + ty;
    k.ze     = min(zs + zdepth, a.end.z);
    k.image  = a.wrap ? a.mz - 2 * NGHOST : 0;
    k.active = gx < a.end.x && gy < a.end.y;
    k.own    = (unsigned)(k.active ? gx + gy * a.mx : x0 + y0 * a.mx) * sizeof(AcReal);
#pragma unroll
    for (int r = 0; r < K::R; ++r) {
        const int e  = min(tid + r * K::NC, K::LN - 1); // surplus threads repeat the last cell
        const int ex = e % K::LX, ey = e / K::LX;
        int xx = x0 - 3 + ex, yy = y0 - 3 + ey;
        const bool in_box = xx < a.mx && yy < a.my;
        if (a.wrap) { // periodic images of the x and y ghost columns
            const int nx = a.mx - 2 * NGHOST, ny = a.my - 2 * NGHOST;
            xx = xx < NGHOST ? xx + nx : xx >= nx + NGHOST ? xx - nx : xx;
            yy = yy < NGHOST ? yy + ny : yy >= ny + NGHOST ? yy - ny : yy;
        }
        k.goff[r] = (unsigned)(in_box ? xx + yy * a.mx : 0) * sizeof(AcReal);
        k.loff[r] = ey * K::PITCH + ex + k.group * 2 * K::LX;
    }
    k.cofs = (ty + 3) * K::PITCH + (tx + 3) + k.group * 2 * K::LX;
    k.march(zs);
}

#pragma clang fp contract(fast)

} // namespace
} // namespace ac
