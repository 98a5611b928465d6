// Band tile of the NEMOLite2D step: the body of the kernels the library runs
// by default, FP64 and mixed precision, single domain, ensemble and in place.
//
// A tile is one strip of one band of rows of one domain, walked by one
// wavefront of 64 lanes, one column each, of which OW are owned (stored) and
// the others neighbours, one below and at least two above. Neighbour columns
// come from the next lane (DPP wave shifts).
//
// What is different from the overlapped-wavefront tile of nemo_wave.h (which
// the explicitly numbered kernel shapes keep):
//
//  * every face quantity is evaluated once. An advective flux, a strain or a
//    shear quotient through a face belongs to the two points on either side;
//    the reference evaluates it at both. Here the east one is shifted in
//    from lane l-1 and the north one is carried from row j-1. The two
//    evaluations of the reference differ at most in the order of one
//    commutative sum or product, so the bits are the same. This takes about
//    a third of the arithmetic (4 of the 17 divisions a point) and most of
//    the window of row j-1 out of the registers.
//  * metrics by row (template argument ROWM): on a grid whose spacings,
//    areas, Coriolis factors and after-ssh faces do not vary along a row (any
//    Cartesian or latitude-longitude grid) those 13 arrays are read as one
//    record a row through the scalar cache instead of 13 arrays: 108 instead
//    of 212 bytes a point in FP64, 61 instead of 113 in FP32. The caller has
//    checked that every element of a row has the same bits
//    (launch_row_metrics), so the values the arithmetic sees are the same.
//  * the Flather faces are part of the tile. A Flather face has one open and
//    one wet cell and reads one neighbour face; a chain along the sweep is at
//    most two faces long (an open, a wet and an open cell in a row). The
//    lane that computes the neighbour's new value also writes the face, so
//    no second launch follows (2.3 us of a 11.4 us step at 128^2).
//
// Offsets, bounds and the 2^32-byte limit are those of nemo_wave.h.
#pragma once

#include "nemo_mixed.h"
#include "nemo_step.h"
#include "nemo_wave.h"

namespace nemo {
namespace band {

using wave::from_above;
using wave::from_below;
using wave::Ssh;

// ---- metrics by row -------------------------------------------------------
// One record of 32 values a row. Sums of two rows or two columns are the
// reference's own sums (x + x for the two columns of a row). The R_ slots are
// reciprocals of the divisors: FP32 the hardware reciprocal that
// divide<float> multiplies by, FP64 the refined one of uniform_quotient().
enum RowSlot {
    M_AT, M_ARU, M_ARV, M_E1U, M_E1V, M_E1V2, M_E1T, M_E2U, M_E2US, M_E2V, M_E2T, M_FCU,
    M_FCV, M_SAU, M_SAV,
    R_AT = 16, R_ARU, R_ARV, R_E1V2, R_E1T, R_E2US, R_E2T, ROW_WIDTH = kRowTableWidth
};

// Quotient by a divisor that a whole row shares: a multiplication by its
// refined reciprocal and one correction with a fused remainder (Markstein,
// IBM J. Res. Dev. 34, 1990), the end of the hardware's own division sequence,
// in four instructions instead of eleven. That sequence differs only where it
// first scales its operands, which it does not when the divisor lies in
// 2^+-100 (kDivisorExp, checked for every row) and the numerator is zero, infinite, NaN or
// in 2^-900 .. 2^600: there the quotients are the same bits. The tile tracks
// the exponents of its numerators and redoes a row outside that range with
// plain divisions. 1024^2: 28.6 against 32.1 us (4-row bands), 25.7 against
// 30.3 us (2 rows); 4096^2 is bound by memory and gains nothing.
constexpr int NUM_EXP_MIN = -900, NUM_EXP_MAX = 600;

__device__ __forceinline__ double refined_reciprocal(double b)
{
    const double r = __builtin_amdgcn_rcp(b);
    const double r1 = fma(r, fma(-b, r, 1.0), r);
    return fma(r1, fma(-b, r1, 1.0), r1);
}
__device__ __forceinline__ double uniform_quotient(double a, double b, double y)
{
    const double q = a * y;
    return __builtin_amdgcn_div_fixup(fma(fma(-b, q, a), y, q), b, a);
}

template <typename T>
struct Types;
template <>
struct Types<double> {
    using In = StepIn<double>;
    using Out = StepOut<double>;
    using Tide = double;
    using NewSsh = double;
};
template <>
struct Types<float> {
    using In = MixedIn;
    using Out = MixedOut;
    using Tide = Ssh;
    using NewSsh = Ssh;
};

__device__ __forceinline__ double high(double s) { return s; }
__device__ __forceinline__ float high(Ssh s) { return s.hi; }
__device__ __forceinline__ const double *ssh_of(const StepIn<double> &f) { return f.sshn_t; }
__device__ __forceinline__ const float *ssh_of(const MixedIn &f) { return f.ssh_hi; }

// What the Flather part reads besides the step's inputs. on: 0 where the domain
// has no Flather face. u_prev / v_prev: the velocities at the
// end of the previous step. cu / cv (FP32): sqrt(g / h) at the faces, rounded
// from FP64 (null in FP64, where the tile evaluates it).
template <typename T>
struct Flather {
    const T *u_prev, *v_prev, *cu, *cv;
    int on;
    T two_omega, d2r;  // in-place form (NEXT = false)
};

// First owned lane of a strip of ow columns: one neighbour lane below and two
// above, so ow <= 61.
__device__ __forceinline__ constexpr int first_lane(int ow) { return (64 - ow) / 2; }

template <bool STREAM, typename T>
__device__ __forceinline__ void store(T *__restrict__ base, unsigned off, T v)
{
    T *const q = reinterpret_cast<T *>(reinterpret_cast<char *>(base) +
                                       (unsigned)(off * (unsigned)sizeof(T)));
    if constexpr (STREAM)
        __builtin_nontemporal_store(v, q);
    else
        *q = v;
}

// The outputs of a point: its new u, its new v, its new ssh with the face ssh
// that follow from it. No part needs another's result.
enum Part { PART_U = 1, PART_V = 2, PART_SSH = 4, ALL_PARTS = 7 };

// Keeps an evaluation where it stands: without it the compiler moves the
// arithmetic of a face under the branch of its store, one branch a face, and
// the faces of a row no longer overlap.
template <typename T>
__device__ __forceinline__ void settle(T &x)
{
    asm volatile("" : "+v"(x));
}

// A face that bc_flather_* writes: one open and one wet cell
// (boundary_conditions_kern.c:282-291).
__device__ __forceinline__ bool is_flather(int m_c, int m_p)
{
    return m_c + m_p > -1 && (m_c < 0 || m_p < 0);
}

// One Flather direction at the point this lane owns. vel: the output velocity;
// c: the point's offset, st: the stride of the sweep (1 or W). m_m, m_c, m_p,
// m_pp: mask at -1, 0, +1, +2 along the sweep; face 0 lies between m_c and
// m_p. lo / at / hi: faces -1, 0, +1 inside the sweep's region. first: face
// -1 lies outside the extent. origin: offset of the domain's element 0 (a
// neighbour before it reads as 0). now(): the new velocity at face 0; prev():
// its velocity at the end of the previous step; s(d), h(d): the old face ssh
// and the depth at face d = -1, 0, 1.
// Each value is a functor, called only where the face exists.
template <typename T, typename Now, typename Prev, typename Sm, typename S0, typename Sp,
          typename Hm, typename H0, typename Hp>
__device__ __forceinline__ void flather_faces(T *vel, const T *ssh, const T *coef, T g,
                                              unsigned c, unsigned st, unsigned origin, int m_m,
                                              int m_c, int m_p, int m_pp, bool lo, bool at,
                                              bool hi, bool first, Now now, Prev prev, Sm s_m,
                                              S0 s_0, Sp s_p, Hm h_m, H0 h_0, Hp h_p)
{
    // sqrt(g / h) at face k (boundary_conditions_kern.c:287)
    auto factor = [&](auto h, unsigned k) -> T {
        if constexpr (sizeof(T) == 8)
            return sqrt(g / h());
        else
            return ld32(coef, k);
    };
    const bool self = at && is_flather(m_c, m_p);
    const bool low = lo && m_m < 0 && is_flather(m_m, m_c);    // face -1 reads face 0
    const bool top = hi && m_p >= 0 && is_flather(m_p, m_pp);  // face +1 reads face 0
    if (self && m_c < 0) return;  // reads face +1: that face's owner writes this one
    if (self && first) {
        const bool in = c >= origin + st;
        const T v_nb = in ? ld32(vel, c - st) : T(0), s_nb = in ? ld32(ssh, c - st) : T(0);
        st32(vel, c, v_nb + factor(h_0, c) * (s_0() - s_nb));
        return;
    }
    if (!low && !(top && !self)) return;
    // self && low: a wet cell between two open ones; face -1 reads face 0
    // before the sweep reaches it, face 0 then reads face -1
    const T v_c = self ? prev() : now();
    if (low) {
        const T x = v_c + factor(h_m, c - st) * (s_m() - s_0());
        st32(vel, c - st, x);
        if (self) st32(vel, c, x + factor(h_0, c) * (s_0() - s_m()));
    }
    if (top && !self) st32(vel, c + st, v_c + factor(h_p, c + st) * (s_p() - s_0()));
}

// The Flather faces next to the points that the lanes of a strip own in rows
// jlo .. jhi-1, from memory, after the rows are stored (the lane's own stores
// are visible to it).
template <typename T>
__device__ __forceinline__ void flather_rows(const typename Types<T>::In &f,
                                             const StepScalars<T> &p,
                                             const typename Types<T>::Out &o,
                                             const Flather<T> &fl, int W, unsigned base,
                                             const Bounds &b, int ow, int strip, int jlo,
                                             int jhi)
{
    const int l0 = first_lane(ow);
    const int xmax = b.xe + 1, ymax = b.ye + 1;
    const int lane = (int)(threadIdx.x & 63), i = b.xs - 1 + strip * ow + lane - l0;
    if (lane < l0 || lane >= l0 + ow || i > xmax) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll 1
    for (int j = jlo; j < jhi; j++) {
        auto at = [&](int di, int dj) {
            return base + (unsigned)(min(max(j + dj, 0), ymax) * W) +
                   (unsigned)min(max(i + di, 0), xmax);
        };
        auto mask = [&](int di, int dj) -> int { return ld32(f.tmask, at(di, dj)); };
        const unsigned c = at(0, 0);
        flather_faces(
            o.u, f.sshn_u, fl.cu, p.g, c, 1u, base, mask(-1, 0), mask(0, 0), mask(1, 0),
            mask(2, 0), i - 1 >= b.xs - 1, i <= b.xe, i + 1 <= b.xe, i == b.xs - 1,
            [&] { return ld32(o.u, c); }, [&] { return ld32(fl.u_prev, c); },
            [&] { return ld32(f.sshn_u, at(-1, 0)); }, [&] { return ld32(f.sshn_u, c); },
            [&] { return ld32(f.sshn_u, at(1, 0)); }, [&] { return ld32(f.hu, at(-1, 0)); },
            [&] { return ld32(f.hu, c); }, [&] { return ld32(f.hu, at(1, 0)); });
        flather_faces(
            o.v, f.sshn_v, fl.cv, p.g, c, (unsigned)W, base, mask(0, -1), mask(0, 0),
            mask(0, 1), mask(0, 2), j - 1 >= b.ys - 1 && j - 1 <= b.ye, j <= b.ye,
            j + 1 <= b.ye, j == b.ys - 1, [&] { return ld32(o.v, c); },
            [&] { return ld32(fl.v_prev, c); }, [&] { return ld32(f.sshn_v, at(0, -1)); },
            [&] { return ld32(f.sshn_v, c); }, [&] { return ld32(f.sshn_v, at(0, 1)); },
            [&] { return ld32(f.hv, at(0, -1)); }, [&] { return ld32(f.hv, c); },
            [&] { return ld32(f.hv, at(0, 1)); });
    }
}

// ---- the tile ---------------------------------------------------------------
// T: double (the reference's bits) or float (mixed form). ROWM: metrics by
// row, `tab` the record of row 0. ow: owned columns of the strip (a constant
// of the launch or of the tile). At most R rows (jlo .. jhi-1), PF rows of
// loads in flight beyond the next (the loop is unrolled, so the window shifts
// are register renaming). NEXT: write the new face ssh (false where the step
// updates the caller's arrays in place and a second kernel follows; there
// f.fcor_u and f.fcor_v are the latitudes, and the tile evaluates the Coriolis
// factors itself). STREAM:
// non-temporal stores. QUICK: uniform_quotient for the row's divisors.
// PARTS: the outputs this wavefront evaluates and writes (enum Part).
// tide_of(): the elevation of open cells; one-row bands read it behind their
// loads.
// Returns the first row that is not done: jhi (or jlo + R), or with QUICK a
// row with a numerator outside its range.
template <typename T, bool ROWM, int R, int PF, bool NEXT, bool STREAM, bool QUICK, int PARTS,
          typename Tide>
__device__ __forceinline__ int rows(const typename Types<T>::In &f, const T *__restrict__ tab,
                                    const StepScalars<T> &p, const typename Types<T>::Out &o,
                                    const Flather<T> &fl, int W, unsigned base,
                                    const Bounds &b, int ow, int strip, int jlo, int jhi,
                                    Tide tide_of)
{
    constexpr bool MIXED = sizeof(T) == 4;
    constexpr bool DO_U = PARTS & PART_U, DO_V = PARTS & PART_V, DO_SSH = PARTS & PART_SSH;
    const int l0 = first_lane(ow);
    typename Types<T>::Tide tide{};
    if constexpr (DO_SSH && R > 1) tide = tide_of();
    constexpr bool SHORT = R <= 2;  // Flather faces from the registers
    static_assert(PF >= 0 && PF <= 2 && R >= 1 && R <= 16, "unrolled band");
    using S = typename Types<T>::NewSsh;
    const int xmax = b.xe + 1, ymax = b.ye + 1;
    const int lane = (int)(threadIdx.x & 63);
    const int i = b.xs - 1 + strip * ow + lane - l0;  // may be < 0 or > xmax
    const unsigned ci = (unsigned)min(max(i, 0), xmax);
    const bool own = lane >= l0 && lane < l0 + ow && i <= xmax;
    auto row = [&](int j) { return min(max(j, 0), ymax); };
    auto at_row = [&](int j) { return base + (unsigned)(row(j) * W) + ci; };
    auto rec = [&](int j) { return tab + row(j) * ROW_WIDTH; };

    // window: slot 0 is row j, slot 1 row j+1, then the rows in flight; hu_s
    // and su_s are row j-1, tm_s its mask
    constexpr int NS = 2 + PF, N1 = 1 + PF;
    T un[NS], vn[NS], hu[NS], su[NS], hv[NS], sv[NS], ht[NS], st[NS];
    T lo[NS];                              // MIXED
    T e2u[NS], e1t[NS], e2t[NS], art[NS];  // !ROWM
    T e1v[N1], e1u[N1], e2v[N1], fcu[N1], fcv[N1], aru[N1], arv[N1], sau[N1], sav[N1];  // !ROWM
    int tm[NS + 1];

    auto load_state = [&](int j, int s) {
        const unsigned c = at_row(j);
        un[s] = ld32(f.un, c);
        vn[s] = ld32(f.vn, c);
        hu[s] = ld32(f.hu, c);
        su[s] = ld32(f.sshn_u, c);
        hv[s] = ld32(f.hv, c);
        sv[s] = ld32(f.sshn_v, c);
        ht[s] = ld32(f.ht, c);
        st[s] = ld32(ssh_of(f), c);
        if constexpr (MIXED) lo[s] = ld32(f.ssh_lo, c);
        if constexpr (!ROWM) {
            e2u[s] = ld32(f.dy_u, c);
            e1t[s] = ld32(f.dx_t, c);
            e2t[s] = ld32(f.dy_t, c);
            art[s] = ld32(f.area_t, c);
        }
    };
    auto load_point = [&](int j, int s) {
        if constexpr (!ROWM) {
            const unsigned c = at_row(j);
            e1v[s] = ld32(f.dx_v, c);
            e1u[s] = ld32(f.dx_u, c);
            e2v[s] = ld32(f.dy_v, c);
            fcu[s] = ld32(f.fcor_u, c);
            fcv[s] = ld32(f.fcor_v, c);
            aru[s] = ld32(f.area_u, c);
            arv[s] = ld32(f.area_v, c);
            sau[s] = ld32(f.ssha_u, c);
            sav[s] = ld32(f.ssha_v, c);
        }
    };
    // quotients: by metric slot m of row record r (ROWM) or by x per lane;
    // e_lo / e_hi: smallest and largest exponent of the numerators
    int e_lo = 0, e_hi = 0;
    auto quick = [&](T a, T d, T y) {
        const int e = __builtin_amdgcn_frexp_exp(a);  // 0 for 0, inf and NaN
        e_lo = min(e_lo, e);
        e_hi = max(e_hi, e);
        return uniform_quotient(a, d, y);
    };
    auto over = [&](T a, const T *__restrict__ r, int m, int recip, T x) {
        if constexpr (ROWM && MIXED)
            return a * r[recip];
        else if constexpr (ROWM && QUICK)
            return quick(a, r[m], r[recip]);
        else if constexpr (ROWM)
            return divide(a, r[m]);
        else
            return divide(a, x);
    };
    auto coriolis = [&](T x) -> T {
        if constexpr (NEXT)
            return x;
        else
            return fl.two_omega * sin(x * fl.d2r);  // momentum_u_kern.c:251
    };
    T y_fric = T(0);
    if constexpr (QUICK) y_fric = refined_reciprocal(p.fric);
    auto over_fric = [&](T a) {
        if constexpr (QUICK)
            return quick(a, p.fric, y_fric);
        else
            return divide(a, p.fric);
    };

    // One-row bands, whose time is their latency, issue the loads of all three
    // rows at once, and touch the lines of the row records so that the reads
    // that follow find them in the scalar cache (FP32 128^2 2.97 -> 2.75 us a
    // step, 256^2 3.61 -> 3.36; FP64 without the table 48^2 3.5 -> 3.3). FP64
    // with the table is better off with the last row's loads behind the first
    // arithmetic (181^2 4.28 against 4.50).
    constexpr bool TOGETHER = PF == 0 && R == 1 && (MIXED || !ROWM);
    constexpr int LINES = ROW_WIDTH * (int)sizeof(T) / 64;  // of a record
    unsigned warm[3 * LINES] = {};
    if constexpr (TOGETHER && ROWM) {
#pragma unroll
        for (int l = 0; l < 3 * LINES; l++)
            warm[l] = reinterpret_cast<const unsigned *>(rec(jlo - 1 + l / LINES))[l % LINES * 16];
    }

    // ---- row jlo-1: what row jlo takes from it, then rows jlo and on ------
    const unsigned cs = at_row(jlo - 1);
    const T un_s = ld32(f.un, cs), vn_s = ld32(f.vn, cs);
    T hu_s = ld32(f.hu, cs), su_s = ld32(f.sshn_u, cs);
    T hv_s = ld32(f.hv, cs), sv_s = ld32(f.sshn_v, cs);
    T e2u_s = T(0), e1v_s = T(0);
    if constexpr (!ROWM) {
        e2u_s = ld32(f.dy_u, cs);
        e1v_s = ld32(f.dx_v, cs);
    }
    int tm_s = ld32(f.tmask, cs);
    load_state(jlo, 0);
    tm[0] = ld32(f.tmask, at_row(jlo));
    tm[1] = ld32(f.tmask, at_row(jlo + 1));
#pragma unroll
    for (int k = 1; k <= PF; k++) {
        load_state(jlo + k, k);
        tm[1 + k] = ld32(f.tmask, at_row(jlo + 1 + k));
        load_point(jlo + k - 1, k - 1);
    }

    if constexpr (TOGETHER) {
        load_state(jlo + 1, 1);
        tm[2] = ld32(f.tmask, at_row(jlo + 2));
        load_point(jlo, 0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (ROWM) {
#pragma unroll
            for (int l = 0; l < 3 * LINES; l++) asm volatile("" ::"s"(warm[l]));
        }
    }
    if constexpr (DO_SSH && R == 1) tide = tide_of();

    // carried from row to row: new ssh, its product with the cell area, the
    // continuity flux north, total depths, and the north face of row j-1:
    // mean velocity, momentum flux, shear quotient (u), flux, strain (v)
    S ssh{};
    T cell = T(0), fn, du, dv, dt, vm_s, us, qs = T(0), gs, ss_v = T(0);
    bool shut_s;   // a dry cell south of U(i, j)
    int open = 0;  // negative once the band has seen an open cell

    // new ssh of the row with record r in slot s (mask of the rows south, at
    // and north of it): east depth d, fluxes through its north and south faces
    auto new_ssh = [&](const T *__restrict__ r, int s, T d, T north, T south, int m_s, int m_c,
                       int m_n) -> S {
        const T fe = d * un[s], fw = from_below(fe);
        const int m_w = from_below(m_c), m_e = from_above(m_c);
        const T inc = over((fw - fe + south - north) * p.rdt, r, M_AT, R_AT,
                           ROWM ? T(0) : art[s]);
        const bool clamp = tide_applies(m_c, m_s, m_n, m_e, m_w);
        if constexpr (MIXED) {
            const Ssh x = wave::split((double)st[s] + (double)lo[s] + (double)inc);
            return Ssh{clamp ? tide.hi : x.hi, clamp ? tide.lo : x.lo};
        } else {
            return clamp ? tide : st[s] + inc;
        }
    };
    {
        const T *r0 = ROWM ? rec(jlo - 1) : nullptr, *r1 = ROWM ? rec(jlo) : nullptr;
        const T vn_e = from_above(vn_s), hv_e = from_above(hv_s), sv_e = from_above(sv_s);
        const T e1v_e = ROWM ? T(0) : from_above(e1v_s);
        const int m_e = from_above(tm_s);
        const T dv_s = hv_s + sv_s;
        vm_s = T(0.5) * (vn_s + vn_e);
        const T v = T(0.5) * vm_s * (ROWM ? r0[M_E1V2] : e1v_s + e1v_e);
        const T dep = T(0.5) * (dv_s + hv_e + sv_e);
        const T part = upwind_lo(v) * un[0];
        const T full = upwind_hi(v) * un_s + part;
        shut_s = tm_s <= 0 || m_e <= 0;
        us = (shut_s ? part : full) * v * dep;
        if constexpr (DO_U)
            qs = over(un[0] - un_s, r0, M_E2US, R_E2US, ROWM ? T(0) : e2u_s + e2u[0]);
        du = hu[0] + su[0];
        dv = hv[0] + sv[0];
        dt = ht[0] + st[0];
        const T w = T(0.5) * (vn_s + vn[0]) * (ROWM ? r1[M_E1T] : e1t[0]);
        gs = (upwind_hi(w) * vn_s + upwind_lo(w) * vn[0]) * w * dt;
        if constexpr (DO_V)
            ss_v = over(vn[0] - vn_s, r1, M_E2T, R_E2T, ROWM ? T(0) : e2t[0]) * dt;
        fn = dv * vn[0];
        if constexpr (DO_SSH) {
            ssh = new_ssh(r1, 0, du, fn, dv_s * vn_s, tm_s, tm[0], tm[1]);
            cell = (ROWM ? r1[M_AT] : art[0]) * high(ssh);
        }
    }

    int done = min(jhi, jlo + R);
    constexpr int UNROLL = ROWM && !MIXED && !QUICK ? 1 : R;  // the redone rows: rolled up
#pragma unroll UNROLL
    for (int jj = 0; jj < R; jj++) {
        const int j = jlo + jj;
        if ((R > 1 || jj > 0) && j >= jhi) break;  // wavefront-uniform
        if constexpr (PF >= 1) {
            if (jj + PF < R && j + PF < jhi) {  // rows the band still needs
                load_state(j + 1 + PF, 1 + PF);
                tm[2 + PF] = ld32(f.tmask, at_row(j + 2 + PF));
                load_point(j + PF, PF);
            }
            __builtin_amdgcn_sched_barrier(0);
        } else if (!TOGETHER || jj > 0) {
            load_state(j + 1, 1);
            tm[2] = ld32(f.tmask, at_row(j + 2));
            load_point(j, 0);
        }
        const T *r0 = ROWM ? rec(j) : nullptr, *r1 = ROWM ? rec(j + 1) : nullptr;
        const unsigned c = at_row(j);
        const bool in_t = j >= b.ys && j <= b.ye;      // rows of T and U points
        const bool in_v = j >= b.ys && j <= b.ye - 1;  // rows of V points

        // ---- row j+1: depths, continuity + bc_ssh ----
        const T du1 = hu[1] + su[1], dv1 = hv[1] + sv[1], dt1 = ht[1] + st[1];
        const T fn1 = dv1 * vn[1];
        S ssh1{};
        T cell1 = T(0);
        if constexpr (DO_SSH && (NEXT || R > 1)) {
            ssh1 = new_ssh(r1, 1, du1, fn1, fn, tm[0], tm[1], tm[2]);
            cell1 = (ROWM ? r1[M_AT] : art[1]) * high(ssh1);
        }

        // ---- corner faces: u through the north side, v through the east ----
        const int m_e = from_above(tm[0]), m_ne = from_above(tm[1]);
        const int m_w = from_below(tm[0]), m_nw = from_below(tm[1]);
        const T un_e = from_above(un[0]), vn_e = from_above(vn[0]);
        const T hv_e = from_above(hv[0]), sv_e = from_above(sv[0]);
        const T dt_e = from_above(dt), st_e = from_above(st[0]);
        const T te = dv + hv_e + sv_e, tn = du + hu[1] + su[1];
        const T vm = T(0.5) * (vn[0] + vn_e), um = T(0.5) * (un[0] + un[1]);
        const T e1v2 = ROWM ? r0[M_E1V2] : e1v[0] + from_above(e1v[0]);
        const T e2us = ROWM ? r0[M_E2US] : e2u[0] + e2u[1];
        // seen from row j a dry cell of row j+1 shuts the face, seen from row
        // j+1 one of row j; likewise the east face and its two columns
        T u_north, u_next, v_east, v_west_e;
        {
            const T v = T(0.5) * vm * e1v2, dep = T(0.5) * te;
            const T a = upwind_hi(v) * un[0], z = upwind_lo(v) * un[1], full = a + z;
            u_north = (tm[1] <= 0 || m_ne <= 0 ? a : full) * v * dep;
            u_next = (tm[0] <= 0 || m_e <= 0 ? z : full) * v * dep;
        }
        {
            const T u = T(0.5) * um * e2us, dep = T(0.50) * tn;
            const T a = upwind_hi(u) * vn[0], z = upwind_lo(u) * vn_e, full = a + z;
            v_east = (m_e <= 0 || m_ne <= 0 ? a : full) * u * dep;
            v_west_e = (tm[0] <= 0 || tm[1] <= 0 ? z : full) * u * dep;
        }
        T qn = T(0), qe = T(0);
        if constexpr (DO_U) qn = over(un[1] - un[0], r0, M_E2US, R_E2US, e2us);
        if constexpr (DO_V) qe = over(vn_e - vn[0], r0, M_E1V2, R_E1V2, e1v2);

        // ---- U(i,j): momentum_u, else bc_solid_u ----
        T u_new = T(0);
        bool u_on = false;
        if constexpr (DO_U) {
            const T u = T(0.5) * (un[0] + un_e) * (ROWM ? r0[M_E2T] : from_above(e2t[0]));
            const T fe = (upwind_hi(u) * un[0] + upwind_lo(u) * un_e) * u * dt_e;
            const T se = over(un_e - un[0], r0, M_E1T, R_E1T,
                              ROWM ? T(0) : from_above(e1t[0])) * dt_e;
            const T fw = from_below(fe), sw = from_below(se);
            const T adv = fw - fe + us - u_north;
            const bool shut_n = tm[1] <= 0 || m_ne <= 0;
            const T shear_s = qs * (du + hu_s + su_s), shear_n = qn * tn;
            const T along = ROWM ? r0[M_E2U] : e2u[0], area = ROWM ? r0[M_ARU] : aru[0];
            T vis = (se - sw) * along + ((shut_n ? T(0) : shear_n) - (shut_s ? T(0) : shear_s)) *
                                            (ROWM ? r0[M_E1U] : e1u[0]) * T(0.5);
            vis = p.visc * vis;
            const T cor = T(0.5) * ((ROWM ? r0[M_FCU] : coriolis(fcu[0])) * (vm_s + vm)) * area * du;
            const T hpg = -p.g * du * along * (st_e - st[0]);
            const T acc = over(p.rdt * (adv + vis + cor + hpg), r0, M_ARU, R_ARU, area);
            T val = over_fric(divide(un[0] * du + acc, hu[0] + (ROWM ? r0[M_SAU] : sau[0])));
            settle(val);
            const bool wet = in_t && i >= b.xs && i <= b.xe - 1 && tm[0] > 0 && m_e > 0;
            const bool solid = j >= b.ys - 1 && j <= b.ye + 1 && i <= b.xe && tm[0] * m_e == 0;
            u_new = wet ? val : T(0);
            u_on = own && (wet || solid);
        }
        // ---- V(i,j): momentum_v, else bc_solid_v ----
        T v_new = T(0), v_flux = T(0), v_strain = T(0);
        bool v_on = false;
        if constexpr (DO_V) {
            const T v = T(0.5) * (vn[0] + vn[1]) * (ROWM ? r1[M_E1T] : e1t[1]);
            v_flux = (upwind_hi(v) * vn[0] + upwind_lo(v) * vn[1]) * v * dt1;
            v_strain = over(vn[1] - vn[0], r1, M_E2T, R_E2T, ROWM ? T(0) : e2t[1]) * dt1;
            const T fw = from_below(v_west_e), qw = from_below(qe), um_w = from_below(um);
            const T hv_w = from_below(hv[0]), sv_w = from_below(sv[0]);
            const T adv = fw - v_east + gs - v_flux;
            const bool shut_w = m_w <= 0 || m_nw <= 0, shut_e = m_e <= 0 || m_ne <= 0;
            const T shear_w = qw * (dv + hv_w + sv_w), shear_e = qe * te;
            const T along = ROWM ? r0[M_E1V] : e1v[0], area = ROWM ? r0[M_ARV] : arv[0];
            T vis = (v_strain - ss_v) * along +
                    ((shut_e ? T(0) : shear_e) - (shut_w ? T(0) : shear_w)) *
                        (ROWM ? r0[M_E2V] : e2v[0]) * T(0.5);
            vis = p.visc * vis;
            const T cor = -T(0.5) * ((ROWM ? r0[M_FCV] : coriolis(fcv[0])) * (um + um_w)) * area * dv;
            const T hpg = -p.g * dv * along * (st[1] - st[0]);
            const T acc = over(p.rdt * (adv + vis + cor + hpg), r0, M_ARV, R_ARV, area);
            T val = over_fric(divide(vn[0] * dv + acc, hv[0] + (ROWM ? r0[M_SAV] : sav[0])));
            settle(val);
            const bool wet = in_v && i >= b.xs && i <= b.xe && tm[0] + m_e > 0 && tm[0] > 0 &&
                             tm[1] > 0;
            const bool solid = j >= b.ys - 1 && j <= b.ye && tm[0] * tm[1] == 0;
            v_new = wet ? val : T(0);
            v_on = own && (wet || solid);
        }
        // ---- next_sshu(i,j), next_sshv(i,j) ----
        T su_new = T(0), sv_new = T(0);
        if constexpr (NEXT && DO_SSH) {
            const T s0 = high(ssh), s_e = from_above(s0), cell_e = from_above(cell);
            T mu = over(T(0.5) * (cell + cell_e), r0, M_ARU, R_ARU, ROWM ? T(0) : aru[0]);
            T mv = over(T(0.5) * (cell + cell1), r0, M_ARV, R_ARV, ROWM ? T(0) : arv[0]);
            settle(mu);
            settle(mv);
            su_new = tm[0] * m_e > 0 ? mu : tm[0] <= 0 ? s_e : s0;
            sv_new = tm[0] * tm[1] > 0 ? mv : tm[0] <= 0 ? high(ssh1) : s0;
        }
        if constexpr (QUICK) {
            if (__any(e_lo < NUM_EXP_MIN || e_hi > NUM_EXP_MAX)) {
                done = j;
                break;
            }
        }

        // ---- stores ----
        const bool col_t = own && i >= b.xs && i <= b.xe;
        if (DO_SSH && col_t && in_t) {
            if constexpr (MIXED) {
                store<STREAM>(o.ssh_hi, c, ssh.hi);
                store<STREAM>(o.ssh_lo, c, ssh.lo);
            } else {
                store<STREAM>(o.ssh, c, ssh);
            }
        }
        if (DO_U && u_on) store<STREAM>(o.u, c, u_new);
        if (DO_V && v_on) store<STREAM>(o.v, c, v_new);
        if constexpr (NEXT && DO_SSH) {
            if (col_t && in_t && i <= b.xe - 1 && tm[0] + m_e > 0)
                store<STREAM>(o.sshu, c, su_new);
            if (col_t && in_v && tm[0] + tm[1] > 0) store<STREAM>(o.sshv, c, sv_new);
        }

        // ---- Flather faces next to the points this lane owns (rare) ----
        const int any_open = tm_s | tm[0] | tm[1] | tm[2];  // negative: an open cell
        if constexpr (SHORT) {
            if ((DO_U || DO_V) && fl.on && __any(any_open < 0)) {
                const int m_ee = from_above(m_e);
                const T hu_w = from_below(hu[0]), hu_e = from_above(hu[0]);
                const T su_w = from_below(su[0]), su_e = from_above(su[0]);
                // by value: the functors must not take addresses
                const T su_c = su[0], hu_c = hu[0], sv_c = sv[0], sv_n = sv[1], hv_c = hv[0],
                        hv_n = hv[1], sv_m = sv_s, hv_m = hv_s;
                T *const ou = o.u, *const ov = o.v;
                const T *const up = fl.u_prev, *const vp = fl.v_prev;
                if (DO_U && own)
                    flather_faces(
                        ou, f.sshn_u, fl.cu, p.g, c, 1u, base, m_w, tm[0], m_e, m_ee,
                        i - 1 >= b.xs - 1, i <= b.xe, i + 1 <= b.xe, i == b.xs - 1,
                        [=]() -> T { return u_on ? u_new : ld32(ou, c); },
                        [=] { return ld32(up, c); }, [=] { return su_w; },
                        [=] { return su_c; }, [=] { return su_e; }, [=] { return hu_w; },
                        [=] { return hu_c; }, [=] { return hu_e; });
                if (DO_V && own)
                    flather_faces(
                        ov, f.sshn_v, fl.cv, p.g, c, (unsigned)W, base, tm_s, tm[0], tm[1],
                        tm[2], j - 1 >= b.ys - 1 && j - 1 <= b.ye, j <= b.ye, j + 1 <= b.ye,
                        j == b.ys - 1, [=]() -> T { return v_on ? v_new : ld32(ov, c); },
                        [=] { return ld32(vp, c); }, [=] { return sv_m; },
                        [=] { return sv_c; }, [=] { return sv_n; }, [=] { return hv_m; },
                        [=] { return hv_c; }, [=] { return hv_n; });
            }
            hv_s = hv[0];
            sv_s = sv[0];
        } else {
            open |= any_open;
        }

        // ---- advance ----
        hu_s = hu[0];
        su_s = su[0];
        tm_s = tm[0];
        shut_s = tm[0] <= 0 || m_e <= 0;
        ssh = ssh1;
        cell = cell1;
        fn = fn1;
        du = du1;
        dv = dv1;
        dt = dt1;
        vm_s = vm;
        us = u_next;
        qs = qn;
        gs = v_flux;
        ss_v = v_strain;
#define NEMO_ADVANCE(a, n) \
    _Pragma("unroll") for (int s = 0; s + 1 < (n); s++) a[s] = a[s + 1];
        NEMO_ADVANCE(un, NS) NEMO_ADVANCE(vn, NS) NEMO_ADVANCE(hu, NS) NEMO_ADVANCE(su, NS)
        NEMO_ADVANCE(hv, NS) NEMO_ADVANCE(sv, NS) NEMO_ADVANCE(ht, NS) NEMO_ADVANCE(st, NS)
        NEMO_ADVANCE(tm, NS + 1)
        if constexpr (MIXED) { NEMO_ADVANCE(lo, NS) }
        if constexpr (!ROWM) {
            NEMO_ADVANCE(e2u, NS) NEMO_ADVANCE(e1t, NS) NEMO_ADVANCE(e2t, NS)
            NEMO_ADVANCE(art, NS)
            NEMO_ADVANCE(e1v, N1) NEMO_ADVANCE(e1u, N1) NEMO_ADVANCE(e2v, N1)
            NEMO_ADVANCE(fcu, N1) NEMO_ADVANCE(fcv, N1) NEMO_ADVANCE(aru, N1)
            NEMO_ADVANCE(arv, N1) NEMO_ADVANCE(sau, N1) NEMO_ADVANCE(sav, N1)
        }
#undef NEMO_ADVANCE
    }
    // longer bands: the Flather faces afterwards, where the band has open cells
    if (!SHORT && fl.on && __any(open < 0))
        flather_rows<T>(f, p, o, fl, W, base, b, ow, strip, jlo, done);
    return done;
}

// Rows jlo .. jhi-1 (at most R) of one strip: the quick form, and plain
// divisions from a row on whose numerators leave its range (a wave front that
// runs into a basin at rest).
template <typename T, bool ROWM, int R, int PF, bool NEXT, bool STREAM, int PARTS, typename Tide>
__device__ __forceinline__ void tile(const typename Types<T>::In &f, const T *__restrict__ tab,
                                     const StepScalars<T> &p, const typename Types<T>::Out &o,
                                     const Flather<T> &fl, int W, unsigned base,
                                     const Bounds &b, int ow, int strip, int jlo, int jhi,
                                     Tide tide_of)
{
    static_assert(PARTS == ALL_PARTS || R <= 2, "the faces of longer bands follow all parts");
    constexpr bool QUICK = ROWM && sizeof(T) == 8;
    const int next = rows<T, ROWM, R, PF, NEXT, STREAM, QUICK, PARTS>(
        f, tab, p, o, fl, W, base, b, ow, strip, jlo, jhi, tide_of);
    if constexpr (QUICK)
        if (next < jhi)
            rows<T, ROWM, R, 0, NEXT, STREAM, false, PARTS>(f, tab, p, o, fl, W, base, b, ow,
                                                            strip, next, jhi, tide_of);
}

}  // namespace band
}  // namespace nemo
