// The ring march: the default FP32 solve (variant 19). FP64 runs it with two threads per cell column
// (solve_pair.h).
//
// A block owns a TX x TY column of cells and marches it along z, one thread per cell column, all
// eight fields of four planes in an LDS ring. What it does differently from the lean z-march
// (ZMarchLean in solve.hip), which it replaced as the default:
//
// * Cross derivatives. The x-z derivative of output z is sum_i c_i (D_i(z+i) - D_i(z-i)), D_i the
//   difference of a plane's cells at x + i and x - i (y-z alike). The lower half is scattered when a
//   plane is the output plane, from the differences its first derivatives need anyway; the upper
//   half is gathered from the planes z+1..z+3 in the ring. So three outputs are pending instead of
//   seven, 18 registers per lane instead of 42, and planes below the first output are not marched:
//   they are staged at once and only scattered (a block's prologue costs 1.5-3 planes instead of 6).
// * The output plane is worked on in two halves: its in-plane part (in_plane) before plane z+3 is
//   there, the rest (finish) after. Plane z+3 takes the slot that plane z-1 left, so one barrier
//   per plane suffices.
// * Each field's LDS reads are issued before the arithmetic of the field before it, in an order that
//   scheduling barriers hold. The lean march consumed most of its reads as they were issued: 90 waits
//   a plane for LDS, now 60, most of them satisfied. With registers to spare from the smaller
//   pending state this needs no spill (FP32 204 of 256 registers; the same order cost the lean
//   march more in spills than it saved).
// * The ring rows hold all eight fields of a tile row side by side, so one LDS base register per row
//   serves every field's x window, and rows a tile row apart start 16 banks apart (16-wide tiles).
// * The previous stage is loaded a whole plane ahead, the next plane too (but see LATE).
// * One field pointer and a stride instead of sixteen pointers, which in this march spilled 78 scalar
//   registers to lanes of vector ones (50 v_readlane a plane). The rates are
//   formed with fewer operations (mhd_rates_lean). The vector instruction count is level with the
//   lean march's (630 a plane in FP32): what it gains is in the waits.
//
// What bounds it: the vector pipes are busy 65 to 75 % of the time (LDS 50 to 57 %). At 512^3 a launch of
// substeps 1 and 2 moves 13.9 GB at 3.8 TB/s, 81 % of what a plain copy of 4 GiB reaches on this card; substep
// 0 moves 9.6 GB at 2.9 TB/s and is bound by instruction issue. Per launch, sustained, mean of the three
// substeps (us), lean march -> this: 32^3 27.9 -> 7.6, 97 x 61 x 75 35.8 -> 25.4, 128^3 74.7 -> 56.2, 256^3
// 529 -> 447, 512^3 4020 -> 3540.
#pragma once
#include "physics.h"

namespace ac {
namespace {

// Every multiply-add is written out (mad) and the compiler forms none of its own: it would choose
// differently in the three copies of the plane loop, and a cell's value would depend on where its
// block's column begins.
#pragma clang fp contract(off)

// FIRST: the build of substep 0, which has no previous stage.
//
// LATE: the next plane is loaded at the end of a plane's work instead of in its middle, two thirds of a
// plane ahead of its use instead of a whole one. A block then waits for lines that its neighbours have
// not fetched yet, which keeps the blocks of 16 x 16 tiles at nearly the same z, where they share halo
// lines in L2: ensembles on a full chip gain (100 boxes of 48^3 1605 -> 1430 us per step, 20 of 80^3
// 1300 -> 1184, 256 of 32^3 1088 -> 1046), launches with a block or two per CU are level (4 of 48^3 114
// -> 111, 4 of 80^3 239 -> 241), 512-thread blocks, whose waves march together anyway, lose (32 of 64^3
// 816 -> 870).
template <int TX, int TY, bool COMP, bool FIRST, bool LATE> struct ZMarchRing {
    static constexpr int NT = TX * TY;
    static_assert(NT % 64 == 0, "whole waves");
    static constexpr int LX = TX + 6, LY = TY + 6, LN = LX * LY;
    static constexpr int R     = (LN + NT - 1) / NT; // staging rounds per field and plane
    static constexpr int PITCH = NF * LX;            // one tile row of all eight fields

    struct Shared {
        AcReal ring[4][LY * PITCH]; // [slot][row][field][x]
    };

    struct State {
        AcReal q[NF][3];  // planes z-3..z-1, plane p in slot p mod 3 (counted from the first output)
        AcReal x[6][3];   // cross sums of outputs z..z+2, output o in slot o mod 3
        AcReal pv[NF][R]; // the next plane, on its way from global memory to the ring
        MhdAgg g;         // output z: what its in-plane stencils and the planes z+1, z+2 give
        AcReal cur[NF];   // output z: values
        // Second derivatives that join the cross derivatives of grad div u (its own axis) and of
        // grad div A - lap A (the other two axes) last: they are the largest terms, and what is
        // added to them is rounded at their size.
        AcReal own[3], rest[3];
        AcReal prev[FIRST ? 1 : NF];                   // output z: previous stage
        AcReal cin[COMP ? NF : 1];                     // rounding errors (compensated integration),
        AcReal cprev[COMP && !FIRST ? NF : 1];         // and those of the previous stage
        int s0, s1, s2, s3; // first element of the ring slots of planes z..z+3 (uniform)
    };

    const SubstepArgs& a;
    Shared& sh;
    int cofs, ze;
    int image; // ghost planes: n_z where they are read at their periodic images, else 0
    unsigned own;
    bool active;
    unsigned goff[R]; // byte offset in a plane of what this thread stages, per round
    int loff[R];      // its place in a ring slot (field 0)

    __device__ __forceinline__ ZMarchRing(const SubstepArgs& args, Shared& shared) : a(args), sh(shared) {}

    typedef __attribute__((address_space(1))) AcReal GReal;
    typedef __attribute__((address_space(1))) const char GByte;
    typedef const AcReal __attribute__((address_space(3))) LdsReal;

    // Keeps LDS reads on their side (instruction scheduling only).
    static __device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
    // Values that are to be computed here: nothing else keeps the compiler from putting off a
    // field's arithmetic, with its whole window in registers, to where the results are used (up to
    // 470 spilled registers). The derivatives are settled, the cross sums are not, which leaves it
    // freedom to order the rest (3.58 ms at 512^3 against 3.65 with both).
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
    // Row dy of this thread's window in ring slot SLOT, pinned: all reads of that row (every field's
    // x-3..x+3) through one base register with immediate offsets.
    __device__ __forceinline__ const LdsReal* row(int slot, int dy) const
    {
        unsigned addr = (unsigned)(size_t)(const LdsReal*)(&sh.ring[0][0] + (slot + dy * PITCH) + (cofs - 3));
        asm volatile("" : "+v"(addr));
        return (const LdsReal*)(size_t)addr + 3;
    }
    static __device__ __forceinline__ AcReal at(const LdsReal* r, int f, int dx) { return r[f * LX + dx]; }

    // Cells from one field to the next (SubstepArgs::stride). Read anew at every use: left to
    // itself the compiler keeps all sixteen field pointers, 32 scalar registers that the stencil
    // and physics constants then spill for.
    __device__ __forceinline__ long field_stride() const
    {
        long s = a.stride;
        asm volatile("" : "+s"(s));
        return s;
    }

    __device__ __forceinline__ void load(AcReal (&pv)[NF][R], int p) const
    {
        int q = min(p, ze + 2);
        q += q < NGHOST ? image : q >= a.mz - NGHOST ? -image : 0;
        const long pl = (long)q * a.mxy;
        unsigned go[R];
#pragma unroll
        for (int r = 0; r < R; ++r)
            go[r] = pin(goff[r]);
        const AcReal* src = a.in[0] + pl;
        const long stride = field_stride();
#pragma unroll
        for (int f = 0; f < NF; ++f) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                pv[f][r] = ld(src, go[r]);
            src += stride;
        }
    }

    __device__ __forceinline__ void stage(int slot, const AcReal (&pv)[NF][R]) const
    {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int f = 0; f < NF; ++f)
                sh.ring[0][slot + loff[r] + f * LX] = pv[f][r];
    }

    // One field's window in a plane: its cell and the pairs +-1..+-3 along x and y.
    struct Star {
        AcReal v, xp[3], xm[3], yp[3], ym[3];
    };
    // The diagonal pairs of the x-y cross derivative.
    struct Diag {
        AcReal pp[3], mm[3], pm[3], mp[3];
    };
    struct Rows {
        const LdsReal* r[7];
        __device__ __forceinline__ const LdsReal* operator()(int dy) const { return r[dy + 3]; }
    };

    static __device__ __forceinline__ Star star(const Rows& w, int f)
    {
        Star s;
        s.v = at(w(0), f, 0);
#pragma unroll
        for (int i = 1; i <= 3; ++i) {
            s.xm[i - 1] = at(w(0), f, -i);
            s.xp[i - 1] = at(w(0), f, i);
            s.ym[i - 1] = at(w(-i), f, 0);
            s.yp[i - 1] = at(w(i), f, 0);
        }
        return s;
    }
    static __device__ __forceinline__ Diag diag(const Rows& w, int f)
    {
        Diag d;
#pragma unroll
        for (int i = 1; i <= 3; ++i) {
            d.mm[i - 1] = at(w(-i), f, -i);
            d.pm[i - 1] = at(w(-i), f, i);
            d.mp[i - 1] = at(w(i), f, -i);
            d.pp[i - 1] = at(w(i), f, i);
        }
        return d;
    }

    // The pairs along one axis as differences and sums.
    struct Line {
        AcReal d[3], s[3];
    };
    static __device__ __forceinline__ Line line(const AcReal* p, const AcReal* m)
    {
        Line l;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            l.d[i] = p[i] - m[i];
            l.s[i] = p[i] + m[i];
        }
        return l;
    }
    // Derivatives, their largest terms last, so that only the last sums are rounded at their size. Near
    // the diffusive limit of the time step this shows in a velocity's error: 9.12e-8 of the field
    // with the largest terms first, 8.68e-8 so (mean of 3 states of noise on a grid of 2 pi / 512, 2 steps).
    static __device__ __forceinline__ AcReal first(const Line& l, const AcReal* c)
    {
        return mad(c[1], l.d[0], mad(c[2], l.d[1], c[3] * l.d[2]));
    }
    static __device__ __forceinline__ AcReal second(const Line& l, AcReal v, const AcReal* c)
    {
        return mad(c[0], v, mad(c[1], l.s[0], mad(c[2], l.s[1], c[3] * l.s[2])));
    }
    // The same, added to a sum term by term, so that every term is one multiply-add.
    static __device__ __forceinline__ void add_first(AcReal& sum, const Line& l, const AcReal* c)
    {
#pragma unroll
        for (int i = 2; i >= 0; --i)
            sum = mad(c[i + 1], l.d[i], sum);
    }
    static __device__ __forceinline__ AcReal cross(const Diag& d, const AcReal* c)
    {
        AcReal t[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            t[i] = (d.pp[i] + d.mm[i]) - (d.pm[i] + d.mp[i]);
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
    }

    __device__ __forceinline__ Rows rows(int slot) const
    {
        Rows w;
#pragma unroll
        for (int j = -3; j <= 3; ++j)
            w.r[j + 3] = row(slot, j);
        return w;
    }

    // Planes below the first output: only their differences and values are needed.
    template <int PH> __device__ __forceinline__ void warm(State& st) const
    {
        const PhysParams& P = a.phys;
        const Rows w        = rows(PH * LY * PITCH);
        auto dx             = [&](int f, int n, bool add) {
            AcReal d[3];
#pragma unroll
            for (int i = 1; i <= 3; ++i)
                d[i - 1] = at(w(0), f, i) - at(w(0), f, -i);
            scatter<PH>(st, n, P.cxz, d, add);
        };
        auto dy = [&](int f, int n, bool add) {
            AcReal d[3];
#pragma unroll
            for (int i = 1; i <= 3; ++i)
                d[i - 1] = at(w(i), f, 0) - at(w(-i), f, 0);
            scatter<PH>(st, n, P.cyz, d, add);
        };
        dx(VTXBUF_UUZ, 0, false);
        dy(VTXBUF_UUZ, 1, false);
        dx(VTXBUF_UUX, 2, false);
        dy(VTXBUF_UUY, 2, true);
        dx(VTXBUF_AZ, 3, false);
        dy(VTXBUF_AZ, 4, false);
        dx(VTXBUF_AX, 5, false);
        dy(VTXBUF_AY, 5, true);
#pragma unroll
        for (int f = 0; f < NF; ++f)
            st.q[f][PH] = at(w(0), f, 0);
    }

    // One vector field triple's pairs at distance I in plane z + I, for the cross sums.
    struct Ahead {
        AcReal xz[2], yz[2], xx[2], yy[2]; // x and y pairs of component z; x pair of x; y pair of y
    };
    template <int I>
    static __device__ __forceinline__ Ahead ahead(const LdsReal* r0, const LdsReal* rm, const LdsReal* rp, int fx)
    {
        Ahead h;
        h.xz[0] = at(r0, fx + 2, -I), h.xz[1] = at(r0, fx + 2, I);
        h.yz[0] = at(rm, fx + 2, 0), h.yz[1] = at(rp, fx + 2, 0);
        h.xx[0] = at(r0, fx, -I), h.xx[1] = at(r0, fx, I);
        h.yy[0] = at(rm, fx + 1, 0), h.yy[1] = at(rp, fx + 1, 0);
        return h;
    }
    // Adds them to the three sums of that field.
    static __device__ __forceinline__ void add_ahead(AcReal* sum, const Ahead& h, AcReal cx, AcReal cy)
    {
        sum[0] = mad(cx, h.xz[1] - h.xz[0], sum[0]);
        sum[1] = mad(cy, h.yz[1] - h.yz[0], sum[1]);
        sum[2] = mad(cx, h.xx[1] - h.xx[0], sum[2]);
        sum[2] = mad(cy, h.yy[1] - h.yy[0], sum[2]);
    }

    // In-plane part of output plane z (ring slot PH; planes z+1, z+2 in the next two slots). The LDS
    // reads of each field are issued before the arithmetic of the field before it.
    template <int PH> __device__ __forceinline__ void in_plane(State& st, const Rows& w, const Star& lr) const
    {
        const PhysParams& P = a.phys;
        MhdAgg& g           = st.g;
        AcReal* cur         = st.cur;
        const LdsReal *b0 = row(st.s1, 0), *bm = row(st.s1, -1), *bp = row(st.s1, 1);
        const Star ss = star(w, VTXBUF_ENTROPY);
        fence();
        {
            const Line lx = line(lr.xp, lr.xm), ly = line(lr.yp, lr.ym);
            cur[VTXBUF_LNRHO] = lr.v;
            g.lr_x = first(lx, P.d1[0]), g.lr_y = first(ly, P.d1[1]);
            g.lr_lap = second(lx, lr.v, P.d2[0]) + second(ly, lr.v, P.d2[1]);
            settle(g.lr_x, g.lr_y, g.lr_lap, cur[VTXBUF_LNRHO]);
        }
        fence();
        const Ahead u1 = ahead<1>(b0, bm, bp, VTXBUF_UUX), a1 = ahead<1>(b0, bm, bp, VTXBUF_AX);
        fence();
        {
            const Line lx = line(ss.xp, ss.xm), ly = line(ss.yp, ss.ym);
            cur[VTXBUF_ENTROPY] = ss.v;
            g.s_x = first(lx, P.d1[0]), g.s_y = first(ly, P.d1[1]);
            g.s_lap = second(lx, ss.v, P.d2[0]) + second(ly, ss.v, P.d2[1]);
            settle(g.s_x, g.s_y, g.s_lap, cur[VTXBUF_ENTROPY]);
        }
        fence();
        const LdsReal *c0 = row(st.s2, 0), *cm = row(st.s2, -2), *cp = row(st.s2, 2);
        const Ahead u2 = ahead<2>(c0, cm, cp, VTXBUF_UUX), a2 = ahead<2>(c0, cm, cp, VTXBUF_AX);
        fence();
#pragma unroll
        for (int n = 0; n < 3; ++n)
            g.gdu[n] = st.x[n][PH], g.jj[n] = st.x[3 + n][PH];
        add_ahead(g.gdu, u1, P.cxz[1], P.cyz[1]);
        add_ahead(g.jj, a1, P.cxz[1], P.cyz[1]);
        fence();
        const Star ux  = star(w, VTXBUF_UUX);
        const Diag dux = diag(w, VTXBUF_UUX);
        fence();
        add_ahead(g.gdu, u2, P.cxz[2], P.cyz[2]);
        add_ahead(g.jj, a2, P.cxz[2], P.cyz[2]);
        fence();
        const Star uy  = star(w, VTXBUF_UUY);
        const Diag duy = diag(w, VTXBUF_UUY);
        fence();
        {
            const Line lx = line(ux.xp, ux.xm), ly = line(ux.yp, ux.ym);
            cur[VTXBUF_UUX] = ux.v;
            g.ug[0][0] = first(lx, P.d1[0]), g.ug[0][1] = first(ly, P.d1[1]);
            st.own[0] = second(lx, ux.v, P.d2[0]);
            g.ulap[0] = second(ly, ux.v, P.d2[1]);
            g.gdu[1] += cross(dux, P.cxy);
            scatter<PH>(st, 2, P.cxz, lx.d, false);
            settle(g.ug[0][0], g.ug[0][1], st.own[0], g.ulap[0], g.gdu[1], cur[VTXBUF_UUX]);
        }
        fence();
        const Star uz = star(w, VTXBUF_UUZ);
        fence();
        {
            const Line lx = line(uy.xp, uy.xm), ly = line(uy.yp, uy.ym);
            cur[VTXBUF_UUY] = uy.v;
            g.ug[1][0] = first(lx, P.d1[0]), g.ug[1][1] = first(ly, P.d1[1]);
            st.own[1] = second(ly, uy.v, P.d2[1]);
            g.ulap[1] = second(lx, uy.v, P.d2[0]);
            g.gdu[0] += cross(duy, P.cxy);
            scatter<PH>(st, 2, P.cyz, ly.d, true);
            settle(g.ug[1][0], g.ug[1][1], st.own[1], g.ulap[1], g.gdu[0], cur[VTXBUF_UUY]);
        }
        fence();
        const Star ax  = star(w, VTXBUF_AX);
        const Diag dax = diag(w, VTXBUF_AX);
        fence();
        {
            const Line lx = line(uz.xp, uz.xm), ly = line(uz.yp, uz.ym);
            cur[VTXBUF_UUZ] = uz.v;
            g.ug[2][0] = first(lx, P.d1[0]), g.ug[2][1] = first(ly, P.d1[1]);
            g.ulap[2] = second(lx, uz.v, P.d2[0]) + second(ly, uz.v, P.d2[1]);
            scatter<PH>(st, 0, P.cxz, lx.d, false);
            scatter<PH>(st, 1, P.cyz, ly.d, false);
            settle(g.ug[2][0], g.ug[2][1], g.ulap[2], cur[VTXBUF_UUZ]);
        }
        fence();
        const Star ay  = star(w, VTXBUF_AY);
        const Diag day = diag(w, VTXBUF_AY);
        fence();
        {
            const Line lx = line(ax.xp, ax.xm), ly = line(ax.yp, ax.ym);
            cur[VTXBUF_AX]   = ax.v;
            st.rest[0]       = second(ly, ax.v, P.d2[1]);
            g.alap[0]        = second(lx, ax.v, P.d2[0]);
            g.jj[1] += cross(dax, P.cxy);
            g.B[2] = -first(ly, P.d1[1]);
            scatter<PH>(st, 5, P.cxz, lx.d, false);
            settle(g.alap[0], st.rest[0], g.jj[1], g.B[2], cur[VTXBUF_AX]);
        }
        fence();
        const Star az = star(w, VTXBUF_AZ);
        fence();
        {
            const Line lx = line(ay.xp, ay.xm), ly = line(ay.yp, ay.ym);
            cur[VTXBUF_AY]   = ay.v;
            st.rest[1]       = second(lx, ay.v, P.d2[0]);
            g.alap[1]        = second(ly, ay.v, P.d2[1]);
            g.jj[0] += cross(day, P.cxy);
            add_first(g.B[2], lx, P.d1[0]);
            scatter<PH>(st, 5, P.cyz, ly.d, true);
            settle(g.alap[1], st.rest[1], g.jj[0], g.B[2], cur[VTXBUF_AY]);
        }
        fence();
        {
            const Line lx = line(az.xp, az.xm), ly = line(az.yp, az.ym);
            cur[VTXBUF_AZ] = az.v;
            g.alap[2]      = second(lx, az.v, P.d2[0]) + second(ly, az.v, P.d2[1]);
            g.B[0] = first(ly, P.d1[1]);
            g.B[1] = -first(lx, P.d1[0]);
            scatter<PH>(st, 3, P.cxz, lx.d, false);
            scatter<PH>(st, 4, P.cyz, ly.d, false);
            settle(g.alap[2], g.B[0], g.B[1], cur[VTXBUF_AZ]);
        }
    }

    // Four fields' values at planes z+1..z+3.
    struct Above {
        AcReal c[4][3];
    };
    static __device__ __forceinline__ Above above(const LdsReal* r1, const LdsReal* r2, const LdsReal* r3, int f0, int f1,
                                                  int f2, int f3)
    {
        const int f[4] = {f0, f1, f2, f3};
        Above u;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            u.c[n][0] = at(r1, f[n], 0);
            u.c[n][1] = at(r2, f[n], 0);
            u.c[n][2] = at(r3, f[n], 0);
        }
        return u;
    }
    template <int PH> static __device__ __forceinline__ Line zline(const State& st, int f, const AcReal* c)
    {
        const AcReal m[3] = {st.q[f][(PH + 2) % 3], st.q[f][(PH + 1) % 3], st.q[f][PH]};
        return line(c, m);
    }

    // The previous stage at output plane z, a whole step before it is used.
    __device__ __forceinline__ void load_prev(State& st, int z) const
    {
        if (FIRST && !COMP)
            return;
        const unsigned long oz = (unsigned long)min(z, ze - 1) * a.mxy;
        const long stride      = field_stride();
        const unsigned ow      = pin(own);
        if (!FIRST) {
            const AcReal* src = a.out[0] + oz;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                st.prev[f] = ld(src, ow);
                src += stride;
            }
        }
        if (COMP) {
            const AcReal *ci = a.cin[0] + oz, *cp = a.cout[0] + oz;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                st.cin[f] = ld(ci, ow);
                ci += stride;
                if (!FIRST) {
                    st.cprev[f] = ld(cp, ow);
                    cp += stride;
                }
            }
        }
    }

    // Output plane z: plane z+3 takes slot PH, then the rest of the derivatives, the rates and the
    // update. Ends with the first window of plane z+1 on its way (w, lr).
    template <int PH> __device__ __forceinline__ void finish(State& st, int z, Rows& w, Star& lr) const
    {
        const PhysParams& P = a.phys;
        MhdAgg& g           = st.g;
        stage(st.s3, st.pv); // the slot of plane z-1, which every thread left before the last barrier
        __syncthreads();
        if (!LATE)
            load(st.pv, z + 4);

        const LdsReal *r1 = row(st.s1, 0), *r2 = row(st.s2, 0), *r3 = row(st.s3, 0);
        const Above n0 = above(r1, r2, r3, VTXBUF_LNRHO, VTXBUF_UUX, VTXBUF_UUY, VTXBUF_UUZ);
        fence();
        const Above n1 = above(r1, r2, r3, VTXBUF_AX, VTXBUF_AY, VTXBUF_AZ, VTXBUF_ENTROPY);
        fence();
        const AcReal *d1z = P.d1[2], *d2z = P.d2[2];
        {
            const Line l = zline<PH>(st, VTXBUF_LNRHO, n0.c[0]);
            g.lr_z       = first(l, d1z);
            g.lr_lap += second(l, st.cur[VTXBUF_LNRHO], d2z);
        }
        {
            const Line l = zline<PH>(st, VTXBUF_UUX, n0.c[1]);
            g.ug[0][2]   = first(l, d1z);
            g.ulap[0]    = (st.own[0] + g.ulap[0]) + second(l, st.cur[VTXBUF_UUX], d2z);
        }
        {
            const Line l = zline<PH>(st, VTXBUF_UUY, n0.c[2]);
            g.ug[1][2]   = first(l, d1z);
            g.ulap[1]    = (g.ulap[1] + st.own[1]) + second(l, st.cur[VTXBUF_UUY], d2z);
        }
        {
            const Line l = zline<PH>(st, VTXBUF_UUZ, n0.c[3]);
            st.own[2]    = second(l, st.cur[VTXBUF_UUZ], d2z);
            g.ug[2][2]   = first(l, d1z);
            g.ulap[2] += st.own[2];
        }
        settle(g.lr_z, g.lr_lap, g.ug[0][2], g.ulap[0], g.ug[1][2], g.ulap[1], g.ug[2][2], g.ulap[2], st.own[2]);
        fence();
        const LdsReal *rm = row(st.s3, -3), *rp = row(st.s3, 3);
        const Ahead u3 = ahead<3>(r3, rm, rp, VTXBUF_UUX), a3 = ahead<3>(r3, rm, rp, VTXBUF_AX);
        fence();
        {
            const Line l = zline<PH>(st, VTXBUF_AX, n1.c[0]);
            st.rest[0] += second(l, st.cur[VTXBUF_AX], d2z);
            g.alap[0] += st.rest[0];
            add_first(g.B[1], l, d1z);
        }
        {
            const Line l = zline<PH>(st, VTXBUF_AY, n1.c[1]);
            st.rest[1] += second(l, st.cur[VTXBUF_AY], d2z);
            g.alap[1] += st.rest[1];
            g.B[0] -= first(l, d1z);
        }
        {
            const Line l = zline<PH>(st, VTXBUF_AZ, n1.c[2]);
            st.rest[2]   = g.alap[2];
            g.alap[2] += second(l, st.cur[VTXBUF_AZ], d2z);
        }
        {
            const Line l = zline<PH>(st, VTXBUF_ENTROPY, n1.c[3]);
            g.s_z        = first(l, d1z);
            g.s_lap += second(l, st.cur[VTXBUF_ENTROPY], d2z);
        }
        settle(g.alap[0], st.rest[0], g.B[1], g.alap[1], st.rest[1], g.B[0], g.alap[2], g.s_z, g.s_lap);
        fence();
        w  = rows(st.s1);
        lr = star(w, VTXBUF_LNRHO);
        fence();
        add_ahead(g.gdu, u3, P.cxz[3], P.cyz[3]);
        add_ahead(g.jj, a3, P.cxz[3], P.cyz[3]);
#pragma unroll
        for (int r = 0; r < 3; ++r)
            g.gdu[r] += st.own[r], g.jj[r] -= st.rest[r];

        g.lr_v = st.cur[VTXBUF_LNRHO], g.s_v = st.cur[VTXBUF_ENTROPY];
        g.uv[0] = st.cur[VTXBUF_UUX], g.uv[1] = st.cur[VTXBUF_UUY], g.uv[2] = st.cur[VTXBUF_UUZ];
        AcReal rate[NF];
        mhd_rates_lean(g, P, rate);
        AcReal res[NF], err[COMP ? NF : 1];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const AcReal u = st.cur[f];
            if (COMP) {
                // The state is the pair (u, c), u + c carrying the rounding error of every update
                // before (u in in / out, c in cin / cout). The increment is formed from the pairs,
                //   d = beta (ab ((u_in - u_prev) + (c_in - c_prev)) + dt F) + c_in,
                // and added with an error-free two-sum (Knuth's TwoSum), whose error term is the
                // new compensation: u_out + c_out = u_in + d exactly. The stencils read u only.
                const AcReal ci   = st.cin[f];
                const AcReal incr = FIRST ? a.rk.dt * rate[f]
                                          : mad(a.rk.dt, rate[f], a.rk.ab * ((u - st.prev[f]) + (ci - st.cprev[f])));
                const AcReal d    = mad(a.rk.beta, incr, ci);
                const AcReal sum  = u + d;
                const AcReal bb   = sum - u;
                err[f]            = (u - (sum - bb)) + (d - bb);
                res[f]            = sum;
            }
            else
                // the smaller product is the one that is rounded by itself
                res[f] = mad(a.rk.beta,
                             FIRST ? a.rk.dt * rate[f] : mad(a.rk.dt, rate[f], a.rk.ab * (u - st.prev[f])), u);
            settle(res[f]);
        }
        load_prev(st, z + 1);
        if (active) {
            const unsigned long oz = (unsigned long)z * a.mxy;
            AcReal *dst = a.out[0] + oz, *cdst = COMP ? a.cout[0] + oz : nullptr;
            const long stride = field_stride();
            const unsigned ow = pin(own);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                st_global(dst, ow, res[f]);
                dst += stride;
                if (COMP) {
                    st_global(cdst, ow, err[f]);
                    cdst += stride;
                }
            }
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
            st.q[f][PH] = st.cur[f];
        if (LATE)
            load(st.pv, z + 4);
        fence();
        const int s = st.s0;
        st.s0 = st.s1, st.s1 = st.s2, st.s2 = st.s3, st.s3 = s;
    }

    __device__ __forceinline__ void march(int zs) const
    {
        State st;
#pragma unroll
        for (int n = 0; n < 6; ++n)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                st.x[n][j] = 0;
        AcReal below[3][NF][R], ahead[3][NF][R];
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
        Rows w  = rows(st.s0);
        Star lr = star(w, VTXBUF_LNRHO);
        for (int z = zs;; ++z) { // ring phases 0, 1, 2; every branch is uniform
            in_plane<0>(st, w, lr);
            finish<0>(st, z, w, lr);
            if (++z == ze)
                break;
            in_plane<1>(st, w, lr);
            finish<1>(st, z, w, lr);
            if (++z == ze)
                break;
            in_plane<2>(st, w, lr);
            finish<2>(st, z, w, lr);
            if (z + 1 == ze)
                break;
        }
    }
};

template <int TX, int TY, bool COMP, bool FIRST, bool LATE = false>
using RingColumn = ZMarchRing<TX, TY, COMP, FIRST, LATE>;

// One z-march column: tile (btx, bty) of box `a`, output planes [zs, min(zs + zdepth, end.z)).
template <int TX, int TY, bool COMP, bool FIRST, bool LATE = false>
__device__ __forceinline__ void
ring_column(const SubstepArgs& a, typename ZMarchRing<TX, TY, COMP, FIRST, LATE>::Shared& sh, const int btx,
            const int bty, const int zs, const int zdepth)
{
    typedef ZMarchRing<TX, TY, COMP, FIRST, LATE> K;
    K k(a, sh);
    const int tid = threadIdx.x;
    const int tx = tid % TX, ty = tid / TX;
    const int x0 = a.start.x + btx * TX, y0 = a.start.y + bty * TY;
    const int gx = x0 + tx, gy = y0 + ty;
    k.ze     = min(zs + zdepth, a.end.z);
    k.image  = a.wrap ? a.mz - 2 * NGHOST : 0;
    k.active = gx < a.end.x && gy < a.end.y;
    k.own    = (unsigned)(k.active ? gx + gy * a.mx : x0 + y0 * a.mx) * sizeof(AcReal);
#pragma unroll
    for (int r = 0; r < K::R; ++r) {
        const int e  = min(tid + r * K::NT, K::LN - 1); // surplus threads repeat the last cell
        const int ex = e % K::LX, ey = e / K::LX;
        int xx = x0 - 3 + ex, yy = y0 - 3 + ey;
        const bool in_box = xx < a.mx && yy < a.my;
        if (a.wrap) { // periodic images of the x and y ghost columns
            const int nx = a.mx - 2 * NGHOST, ny = a.my - 2 * NGHOST;
            xx = xx < NGHOST ? xx + nx : xx >= nx + NGHOST ? xx - nx : xx;
            yy = yy < NGHOST ? yy + ny : yy >= ny + NGHOST ? yy - ny : yy;
        }
        k.goff[r] = (unsigned)(in_box ? xx + yy * a.mx : 0) * sizeof(AcReal);
        k.loff[r] = ey * K::PITCH + ex;
    }
    k.cofs = (ty + 3) * K::PITCH + (tx + 3);
    k.march(zs);
}

#pragma clang fp contract(fast)

} // namespace
} // namespace ac
