// tile_models.hpp -- the per-pixel models of the tile kernel (init / step /
// finish of numba_iterate and numba_iterate_BS), shared by the translation
// units that instantiate them.
//
// Reference loops restated here:
//   holomorphic: numba_iterate, src/fractalshades/perturbation.py:1065-1400
//   burning ship: numba_iterate_BS, perturbation.py:1468-1791
//   model kernels: models/mandelbrot_M2.py:599-622, mandelbrot_Mn.py:646-729,
//                  burning_ship.py:12-60, 440-859
// The ORB parameter adds calc_orbit (perturbation.py:1096-1101, 1266-1273,
// 1390-1396): the orbit point at exit - backshift, in an extra output field.
#pragma once
#include "models.hpp"
#include "tile_loop.hpp"
#include "xl.hpp"

namespace fsg {

// calc_orbit recorder: the last two full orbit points (Z + z), taken at the
// escape test of plain steps when n reaches the next multiple of backshift
// (perturbation.py:1266-1273; n // backshift > div_shift is n >= next).  A
// step at which nothing is due passes the recorder by with the stop tests; the
// division is for a jump over several multiples.
template <bool ORB> struct OrbitRec {
    __device__ void reset(int32_t) {}
    __device__ bool due(int32_t) const { return false; }
    __device__ void record(int32_t, int32_t, double, double) {}
};
template <> struct OrbitRec<true> {
    int32_t next, i1, i2;
    double x1, y1, x2, y2;
    __device__ void reset(int32_t b) { next = b; i1 = 0; i2 = 0; x1 = y1 = x2 = y2 = 0.; }
    __device__ bool due(int32_t n) const { return n >= next; }
    __device__ void record(int32_t n, int32_t b, double x, double y) {
        if (n >= next) {
            int32_t over = n - next;
            pin(over);
            next += b;
            if (over >= b) { pin(over); next = (n / b + 1) * b; }
            i2 = i1; x2 = x1; y2 = y1;
            i1 = n; x1 = x; y1 = y;
        }
    }
};

// the full recurrence, for the orbit finish: M2_iterate (mandelbrot_M2.py:
// 14-15), Mn_iterate (mandelbrot_Mn.py:13-17) by binary powering, and
// BS_iterate (burning_ship.py:82-123)
template <int KIND, int DEG>
__device__ __forceinline__ cplx zn_full(cplx z, cplx c) {
    if constexpr (KIND == KIND_M2) {
        return z * z + c;
    } else {
        cplx r = mk(1., 0.), p = z;
#pragma unroll
        for (int m = DEG; m > 0; m >>= 1) {
            if (m & 1) r = r * p;
            if (m > 1) p = p * p;
        }
        return r + c;
    }
}
template <int FL>
__device__ __forceinline__ void bs_full(double &x, double &y, double A, double B) {
    const double X = x, Y = y;
    if constexpr (FL == 1) { x = X * X - Y * Y + A; y = 2. * fabs(X * Y) - B; }
    else if constexpr (FL == 2) { x = X * X - Y * Y + A; y = 2. * X * fabs(Y) - B; }
    else if constexpr (FL == 3) { x = X * X - Y * fabs(Y) + A; y = 2. * X * Y - B; }
    else if constexpr (FL == 4) { x = fabs(X * X - Y * Y) + A; y = 2. * X * Y - B; }
    else { x = fabs(X * X - Y * Y) + A; y = 2. * fabs(X * Y) - B; }
}

// orbit finish (perturbation.py:1390-1396): from the last-but-one record to
// n - backshift with c + Zn_path[1]
template <int KIND, int DEG>
__device__ __forceinline__ void orbit_finish_holo(const OrbitRec<true> &o, const KArgs &a, const KArgs &g, int32_t n,
                                                  cplx c, int64_t i) {
    cplx zo = mk(o.x2, o.y2);
    const cplx CC = c + a.t.Zn[1];
    for (int32_t k = o.i2; k < n - a.backshift; k++) zo = zn_full<KIND, DEG>(zo, CC);
    const int64_t fo = 1 + a.calc_dz + a.calc_dc;
    g.Z[2 * (fo * g.ld + i)] = zo.re; g.Z[2 * (fo * g.ld + i) + 1] = zo.im;
}
// the same for the burning ship (perturbation.py:1778-1787); the second
// constant is b + Im Zn_path[1], as the reference has it
template <int FL>
__device__ __forceinline__ void orbit_finish_bs(const OrbitRec<true> &o, const KArgs &a, const KArgs &g, int32_t n,
                                                double ca, double cb, int64_t i) {
    double x = o.x2, y = o.y2;
    const cplx R1 = a.t.Zn[1];
    const double AA = ca + R1.re, BB = cb + R1.im;
    for (int32_t k = o.i2; k < n - a.backshift; k++) bs_full<FL>(x, y, AA, BB);
    const int64_t fo = 2 + (a.calc_dc ? 4 : 0);
    g.Z[fo * g.ld + i] = x; g.Z[(fo + 1) * g.ld + i] = y;
}

// BLA lookup on binary64 |z| (ref_BLA_get, perturbation.py:2116-2170)
__device__ __forceinline__ int32_t bla_lookup(const Tables &t, double zre, double zim,
                                              int32_t w, int32_t &idx) {
    return bla_find(t, hypot_key(zre, zim), w, idx);
}
// The same on an extended-range z: the modulus of its mantissa scaled by
// 2^e against the radii.  Where the binary64 copy of z is a normal number
// this takes the decision hypot2 would (the prescale of hypot2 is the same
// power of two); where that copy is subnormal or zero it keeps |z|'s
// precision.
__device__ __forceinline__ int32_t bla_lookup(const Tables &t, xl z, int32_t w, int32_t &idx) {
    return bla_find(t, modulus_key(z.re * z.re + z.im * z.im, z.e), w, idx);
}

// The z^d + c step with the derivatives the launch computes (dz/dc when dc,
// dz/dz when dz): one pass over the shared partial products
// (p_zn_derivs); Zd / Zh are read only for the derivatives computed.
template <int DEG>
__device__ __forceinline__ cplx mn_step(cplx z, cplx Z, cplx c, bool dc, bool dz, cplx &d, cplx &h, cplx Zd, cplx Zh) {
    if (dc && dz) {
        const cplx v[2] = {d, h}, Zv[2] = {Zd, Zh};
        cplx o[2];
        const cplx r = p_zn_derivs<DEG, 2>(z, Z, c, v, Zv, o);
        d = o[0]; h = o[1];
        return r;
    }
    if (dc || dz) {
        const cplx v[1] = {dc ? d : h}, Zv[1] = {dc ? Zd : Zh};
        cplx o[1];
        const cplx r = p_zn_derivs<DEG, 1>(z, Z, c, v, Zv, o);
        (dc ? d : h) = o[0];
        return r;
    }
    return p_zn_derivs<DEG, 0, cplx>(z, Z, c, nullptr, nullptr, nullptr);
}

// ---- pixel -> c (ref_path_c_from_pix + lin_proj_impl, perturbation.py:2214-2230, 2665-2672)
FSG_HD xc c_from_pix(const KArgs &a, double px, double py) {
    double x1 = a.lin[0] * px + a.lin[1] * py;
    double y1 = a.lin[2] * px + a.lin[3] * py;
    xc cx = renorm_c(a.dx_m * x1, a.dx_m * y1, a.dx_e);
    return cx + mkc(a.drift_m[0], a.drift_m[1], a.drift_e[0]);
}

FSG_HD cplx zc() { return mk(0., 0.); }
FSG_HD xc zx() { return mkc(0., 0., 0); }

__device__ __forceinline__ xl c_from_pix_xl(const KArgs &a, double px, double py) {
    const double x1 = a.lin[0] * px + a.lin[1] * py;
    const double y1 = a.lin[2] * px + a.lin[3] * py;
    return xl_of(a.dx_m * x1, a.dx_m * y1, a.dx_e) + xl_of(a.drift_m[0], a.drift_m[1], a.drift_e[0]);
}

// --------------------------------------------------------------------------
// Holomorphic models, binary64 deltas.  DER >= 0 fixes the derivatives at
// compile time (bit 0: dz/dc, bit 1: dz/dz); DER = -1 reads them from the
// launch arguments.
template <int KIND, int DEG, bool ORB = false, int DER = -1>
struct HoloStd {
    __device__ static bool DC_ON(const KArgs &a) { if constexpr (DER >= 0) return (DER & 1) != 0; else return a.calc_dc != 0; }
    __device__ static bool DZ_ON(const KArgs &a) { if constexpr (DER >= 0) return (DER & 2) != 0; else return a.calc_dz != 0; }
    // A pixel around the critical orbit rebases at every step: FLAT has such a
    // step pass the stop tests by (step).  With dz/dz on only, which waits for
    // more: without it the other form is no slower for a lone pixel.
    static constexpr bool FLAT = KIND == KIND_M2 && DER >= 2;
    // Z, A, Zh: as in HoloXr, for z^2 + c.  FLAT: Zd, the dZndc value of the next
    // step, zero for the first one (of the pixel or after a dynamic rebase); first,
    // the plain steps before that step; keep, -1 or, once dZndz is taken at 0
    // (after a rebase), 0.  The other form has dyn, the next step is a first one,
    // and nul: conditions that live across the step, merged in scalar registers
    // at every join of the tests.
    struct State { cplx z, d, h, c, Z, A, Zh, Zd; int32_t w, n, jl, first, keep; bool dyn, nul; OrbitRec<ORB> orb; };
    static constexpr int32_t NOT_FIRST = -1;

    // the carried values at w = 0: from the launch arguments, since a pixel near
    // the critical orbit rebases at every step, each a wait for these otherwise
    __device__ static void at_start(State &s, const KArgs &a) {
        s.Z = mk(a.zn0[0], a.zn0[1]);
        s.A = s.Z + s.z;
        if (DZ_ON(a)) s.Zh = mk(a.dz0[0], a.dz0[1]);
        if (FLAT && DC_ON(a)) {
            s.Zd = zc();
            if (s.first == NOT_FIRST) s.Zd = a.t.dc[0];
        }
    }

    __device__ static void init(State &s, const KArgs &a, double px, double py) {
        s.c = to_std(c_from_pix(a, px, py));
        s.z = zc(); s.d = zc(); s.h = zc();
        s.w = 0; s.n = 0; s.jl = 0; s.dyn = true; s.nul = false; s.first = 0; s.keep = -1;
        if constexpr (KIND == KIND_M2) at_start(s, a);
        s.orb.reset(a.backshift);
    }

    __device__ static bool step(State &s, const KArgs &a, Counters &k, int &reason, int32_t) {
        const Tables &t = a.t;
        if (t.bla_on && (s.w & 7) == 0) {
            int32_t stage, idx;
            [[maybe_unused]] const int32_t w0 = s.w;
            k.looks++;
            do {
                stage = bla_lookup(t, s.z.re, s.z.im, s.w, idx);
                if (stage >= 0) {
                    const int32_t st = 8 << stage;
                    const double *Mb = t.M + 4 * idx;
                    cplx A = mk(Mb[0], Mb[1]), B = mk(Mb[2], Mb[3]);
                    s.n += st;
                    s.w += st;                      // w + st < first_invalid <= order
                    s.z = A * s.z + B * s.c;
                    if (DC_ON(a)) s.d = A * s.d;
                    if (DZ_ON(a)) s.h = A * s.h;
                    s.jl += st; k.bla++;
                }
                pin(stage);
            } while (stage >= 0);
            if constexpr (KIND == KIND_M2) {
                if (s.w != w0) {
                    s.Z = t.Zn[s.w];
                    if (DZ_ON(a) && (FLAT ? s.keep != 0 : !s.nul)) s.Zh = t.dz[s.w];
                    if (FLAT && DC_ON(a) && s.n - s.jl != s.first) s.Zd = t.dc[s.w];
                    s.A = s.Z + s.z;
                }
            }
        }
        s.n += 1;
        // z^d + c: every table value the step reads is loaded here, before any of
        // it is used: the orbit point and path values at w, the next orbit point
        // (escape and rebase tests) and the dZndz value of the interior test,
        // whose indexes are known at the start of the step.  A pixel whose
        // wave has no other work left (the last, longest pixels of a launch)
        // then waits for one table round trip per step instead of one per
        // test.  z^2 + c carries half of them and loads the others where the
        // registers of the old ones are free (HoloXr).  512x512 at 1e-40: 43.9
        // -> 41.4 us.
        int32_t w1 = s.w + 1, wh = w1;                   // wh: index of the interior test's dZndz value
        const bool edge = w1 >= min(t.order, t.div_iter - 1);
        if (edge) {
            pin(w1);
            if (w1 >= t.order) { w1 = 0; wh = s.n == t.order ? t.L : 0; }
        }
        if (FLAT) wh &= s.keep;
        else if (DZ_ON(a) && s.nul) wh = 0;
        cplx Z1, Zd = zc(), H1 = zc(), D1 = zc();
        if (!FLAT && DC_ON(a)) Zd = t.dc[s.w];
        // after the other loads are out: overwriting Zd waits for its own
        const auto first_step = [&]() {
            if (s.dyn) {
                pin(w1);
                Zd = zc();
            }
        };
        if constexpr (KIND == KIND_MN) {
            const cplx Zr = t.Zn[s.w];
            Z1 = t.Zn[w1];
            cplx Zh = zc();
            if (DZ_ON(a)) { Zh = t.dz[s.nul ? 0 : s.w]; H1 = t.dz[wh]; }
            first_step();
            s.z = mn_step<DEG>(s.z, Zr, s.c, DC_ON(a), DZ_ON(a), s.d, s.h, Zd, Zh);
        } else {
            // mandelbrot_M2.py:607-622: z (z + 2 Z) + c, 2 ((Z + z) d + Zd z)
            const cplx W = mk(__builtin_fma(2., s.Z.re, s.z.re), __builtin_fma(2., s.Z.im, s.z.im));
            pin_after(w1, W.re, W.im);
            Z1 = t.Zn[w1];
            // dZndz's term first: its value is at hand, and the load that
            // follows it is then under way before the wait for dZndc's
            cplx v = zc();
            if (DZ_ON(a)) {
                v = s.Zh * s.z;
                pin_after(wh, v.re, v.im);
                H1 = t.dz[wh];
            }
            if constexpr (FLAT) {
                if (DC_ON(a)) {
                    const cplx u = s.Zd * s.z;
                    pin_after(w1, u.re, u.im);
                    D1 = t.dc[w1];
                    s.d = muls(2., s.A * s.d + u);
                }
            } else {
                first_step();
                if (DC_ON(a)) s.d = muls(2., s.A * s.d + Zd * s.z);
            }
            if (DZ_ON(a)) s.h = muls(2., s.A * s.h + v);
            s.z = s.z * W + s.c;
            // the derivatives before Z + z takes A's registers
            if (FLAT && DC_ON(a)) pin_after(Z1.re, s.d.re, s.d.im);
        }
        s.w = w1;
        // The stop and rebase tests are evaluated together: a step that meets
        // none of them (nearly every step) leaves by one branch, and the
        // tests' own order (max_iter, interior, escape, rebase) is kept on
        // the other path.  (The orbit recorder runs between the tests: a
        // step with a point to record takes that path.)  The first branch takes the
        // interior and escape tests by filters that let every step pass that
        // meets them, one component against a bound, and the other path the
        // tests themselves: nine vector instructions less a step
        // (2048x2048 with extended-range deltas: 1e-300 680 -> 649 us,
        // 1e-2000 880 -> 850, interior-dominated 18.3 -> 17.3 ms).
        bool t_int = false;
        if (DZ_ON(a)) t_int = fabs(s.h.re + H1.re) < a.eps_hi;
        const cplx ZZ = s.z + Z1;
        const bool t_esc = amax(ZZ.re, ZZ.im) > a.esc_lo;
        const bool dyn = (fabs(ZZ.re) <= fabs(s.z.re)) && (fabs(ZZ.im) <= fabs(s.z.im));
        if constexpr (KIND == KIND_M2) { s.Z = Z1; s.A = ZZ; s.Zh = H1; s.Zd = D1; }
        if constexpr (FLAT) {
            // Only a step that meets a stop test, the end of the orbit or the recorder
            // takes these branches; the rebase follows for both, its dZndc value at
            // hand.  A lone pixel that rebases at every step takes 320 ns a step, 514 in
            // the other form (1920x1080 at width 4, 1 million steps: 663 -> 405 ms);
            // 900x900 at 1e-12 with the recorder 122 -> 111 us, 1500x1500 at 1e-12 240 ->
            // 230 us.
            bool reb = dyn;
            if (s.n >= a.max_iter || t_int || t_esc || edge || s.orb.due(s.n)) {
                // with the recorder, some lane of the wave is here on most steps: the
                // bounds are read again rather than held beside its scalar values
                const KArgs &b = ORB ? cold_args() : a;
                int32_t r = -1;
                if (t_esc && ZZ.re * ZZ.re + ZZ.im * ZZ.im > b.M2) r = 1;
                if (t_int) {
                    const cplx q = s.h + H1;
                    if (q.re * q.re + q.im * q.im < b.eps2) r = 2;
                }
                if (s.n >= a.max_iter) r = 0;
                if (r != 0 && r != 2) s.orb.record(s.n, b.backshift, ZZ.re, ZZ.im);
                if (r >= 0) { reason = r; return true; }
                if (edge) {
                    if (s.w >= t.div_iter - 1) {
                        reb = true;
                        if (s.n - 1 - s.jl != s.first) s.first = NOT_FIRST;     // not a first step: dZndc at 0
                    } else if (!dyn && s.keep) {
                        s.Zh = t.dz[s.w];               // not the wrapped value of the test
                    }
                }
            }
            if (reb) {
                s.z = ZZ;
                if (DC_ON(a)) s.d = s.d + D1;
                if (s.keep) s.h = s.h + H1;             // dZndz at w (at L after a full period)
                s.keep = 0;
                s.w = 0;
                at_start(s, a);
                s.first = s.first == NOT_FIRST ? NOT_FIRST - 1 : s.n - s.jl;
                k.reb++;
            }
            return false;
        }
        if (!(s.n >= a.max_iter || t_int || t_esc || edge || dyn || s.orb.due(s.n))) { s.dyn = false; return false; }
        if (s.n >= a.max_iter) { reason = 0; return true; }
        if (t_int) {
            const cplx q = s.h + H1;
            if (q.re * q.re + q.im * q.im < a.eps2) { reason = 2; return true; }
        }
        s.orb.record(s.n, a.backshift, ZZ.re, ZZ.im);
        if (t_esc && ZZ.re * ZZ.re + ZZ.im * ZZ.im > a.M2) { reason = 1; return true; }
        bool reb = s.w >= t.div_iter - 1;
        if (!reb) {
            s.dyn = dyn;
            reb = dyn;
        }
        if (reb) {
            s.z = ZZ;
            if (DC_ON(a)) s.d = s.d + t.dc[s.w];
            if (DZ_ON(a)) {
                if (!s.nul) s.h = s.h + H1;     // dZndz at w (at L after a full period)
                s.nul = true;
            }
            s.w = 0;
            if constexpr (KIND == KIND_M2) at_start(s, a);
            k.reb++;
        } else if (KIND == KIND_M2 && DZ_ON(a) && edge && !s.nul) {
            s.Zh = t.dz[s.w];                   // not the wrapped value of the test
        }
        return false;
    }

    __device__ static void finish(const State &s, const KArgs &a, const KArgs &g, int64_t i, int reason) {
        const int64_t n = g.ld;
        cplx z = s.z + a.t.Zn[s.w];
        g.Z[2 * i] = z.re; g.Z[2 * i + 1] = z.im;
        int f = 1;
        if (DZ_ON(a)) { g.Z[2 * (n + i)] = s.h.re; g.Z[2 * (n + i) + 1] = s.h.im; f = 2; }
        if (DC_ON(a)) {
            cplx d = s.d + a.t.dc[s.w];
            g.Z[2 * (f * n + i)] = d.re; g.Z[2 * (f * n + i) + 1] = d.im;
        }
        if constexpr (ORB) orbit_finish_holo<KIND, DEG>(s.orb, a, g, s.n, s.c, i);
        g.U[i] = s.w; g.stop_iter[i] = s.n; g.stop_reason[i] = (int8_t)reason;
    }
};

// Holomorphic models, Xrange deltas (dx < 1e-300), on mantissas with int32
// exponents (xl.hpp).  Where a value is rescaled by a power of two changes no
// rounding, so every operation rounds exactly like the reference's Xrange
// record.
//
// LAZY: the mantissas of z, dz/dc and dz/dz drift freely between
// renormalisations, which the tile loop asks for every RENORM_TRIPS trips
// (and the BLA jump and the rebase for what they read); each keeps one
// exponent, and a sum shifts its other operand -- c, or the path's term -- to
// that exponent instead of aligning both on the larger one.  z^2 + c: Z + z
// and z + 2 Z are formed in binary64 from z's binary64 copy: |Z| is in range,
// so a z that underflows there is far below the rounding of the sum's modulus.
// (Where one component of Z is zero, that component of the sum is z's copy, zero
// or short of digits below 2^-1022.  A component of a result that is itself below
// 2^-1022 can then lose digits; moduli do not.)
// z^d + c: the same for the factors of every binomial term.  Two exceptions
// leave the straight line: an orbit point below 2^LOW_Z (zero, the Xrange
// register) or above 2^HIGH_Z, with which the factors take the exponent of
// the larger of Z and z; and an operand so much larger than the quantity it
// is added to (shift > FAR: a quantity that is still zero, mostly) that the
// exponent moves to the operand's first.  A mantissa then stays within
// 2^+-700: a step multiplies it by at least 2^(LOW_Z (d - 1)) but for
// cancellation and at most d |Z + z|^(d - 1), and adds no more than 2^FAR
// times the operand's mantissa.
// The loop is bound by vector instruction issue (97 % of the cycles on the
// 2048x2048 frames): a z^2 + c step takes about 80 instructions (dz/dc and
// dz/dz on; 58 are the algorithmic flops) where normalising every result and
// aligning every sum took 174.  2048x2048 frames, with drifting mantissas and
// then with what a step shares with the last one carried and the exponents of
// dz/dc and dz/dz relative to the trips: 1e-300 999 -> 792, 636 -> 596 us,
// 1e-2000 1212 -> 1027, 850 -> 774 us, interior-dominated 24.7 -> 22.3, 17.3 ->
// 16.5 ms; 1920x1080 at 1e-800: z^3 + c 850 -> 729 us, z^6 + c 868 -> 666 us.
// DER >= 0 fixes the derivatives at compile time (bit 0: dz/dc, bit 1:
// dz/dz): the step is then one block of straight-line code, which the
// compiler schedules across the z, dz/dc and dz/dz recurrences; DER = -1
// reads them from the launch arguments.
template <int KIND, int DEG, bool ORB = false, int DER = -1>
struct HoloXr {
    __device__ static bool DC_ON(const KArgs &a) { if constexpr (DER >= 0) return (DER & 1) != 0; else return a.calc_dc != 0; }
    __device__ static bool DZ_ON(const KArgs &a) { if constexpr (DER >= 0) return (DER & 2) != 0; else return a.calc_dz != 0; }
    // z^2 + c carries what a step shares with the one before it: the orbit
    // point Z at w and its code kz, A = Z + z (the value of the escape test) and
    // the dZndz value Zh; they are loaded where w becomes a multiple of 8 (the
    // first step, a jump, a rebase, the end of a period).
    struct State { xl z, d, h, c; cplx zs, Z, A; xz Zh; int32_t kz, w, n, jl; bool dyn, nul; OrbitRec<ORB> orb; };
    static constexpr bool LAZY = true;
    // z^2 + c: each step multiplies dz/dc and dz/dz by 2, so their exponents
    // grow by one a trip.  d.e and h.e then hold t - (exponent), t the trips of
    // the pixel, and a step leaves them as they are.  rel converts both ways.
    static constexpr bool REL = KIND == KIND_M2;
    __device__ static int32_t rel(int32_t e, int32_t t) { return REL ? t - e : e; }
    static constexpr int32_t LOW_Z = (KIND == KIND_M2) ? -20 : -60 / (DEG - 1), HIGH_Z = 60, FAR = 256;

    // The z^d + c derivative recurrence of one quantity: its delta v 2^e, the
    // orbit's value Z 2^eG, and the running term t 2^e (times 2^(q eK)).  The
    // inner sum is in the orbit value's scale, far above the delta's: s1
    // takes v's scale there, s2 the product with z back.
    struct Deriv {
        cplx v, Z, t;
        int32_t e, eG, s1, s2;
        __device__ void set(const xl &d, const xz &Zp, int32_t et) {
            v = mk(d.re, d.im); e = d.e; Z = mk(Zp.re, Zp.im);
            eG = Zp.e;                                     // (a zero value, far below: near() takes v's scale)
            s1 = e - eG; s2 = et - s1;
        }
        // the exponents moved together where a shift is out of range
        __device__ void near(int32_t et) {
            if (s1 > FAR) { Z = mk(ldexp(Z.re, -s1), ldexp(Z.im, -s1)); eG = e; s1 = 0; s2 = et; }
            if (s2 > FAR) { v = mk(ldexp(v.re, -s2), ldexp(v.im, -s2)); e += s2; s1 = e - eG; s2 = et - s1; }
        }
        // t <- v mul + z (t + C dZ), t = v at the first term
        __device__ void term(cplx z, cplx mul, cplx CdZ, bool first) {
            const cplx u = first ? v : t;
            const cplx g = z * (mk(ldexp(u.re, s1), ldexp(u.im, s1)) + CdZ);
            const cplx p = v * mul;
            t = mk(p.re + ldexp(g.re, s2), p.im + ldexp(g.im, s2));
        }
    };

    // after t trips
    __device__ static void renorm(State &s, const KArgs &a, int32_t t) {
        s.z = xl_of(as_z(s.z));
        const int32_t zero = rel(XL_ZERO_E, t);
        if (DC_ON(a)) renorm_deriv(s.d, zero);
        if (DZ_ON(a)) renorm_deriv(s.h, zero);
    }
    __device__ static void renorm_deriv(xl &v, int32_t zero) {
        const double mx = amax(v.re, v.im);
        const int32_t k = dexp(mx) - 1;
        v.re = ldexp(v.re, -k); v.im = ldexp(v.im, -k);
        v.e = mx == 0. ? zero : REL ? v.e - k : v.e + k;
    }

    // derivative path values, unnormalised: the host's Xrange records keep
    // |mantissa| within 2^+-100, and a zero entry carries the zero exponent
    // code (the tables are built so), so a value is used as it is loaded
    __device__ static xz DCz(const Tables &t, int32_t i) { const cplx m = t.dc[i]; xz r; r.re = m.re; r.im = m.im; r.e = t.dc_e[i]; return r; }
    __device__ static xz DZz(const Tables &t, int32_t i) { const cplx m = t.dz[i]; xz r; r.re = m.re; r.im = m.im; r.e = t.dz_e[i]; return r; }
    // an orbit point, normalised, from its code k and binary64 value z: the
    // register's Xrange value where the binary64 orbit underflows, z
    // elsewhere, scaled by the exponent k (xl_of of the point, without its
    // exponent extraction)
    __device__ static xl ZRv(const Tables &t, int32_t k, cplx z) {
        if (k < ZK_REGISTER) {
            const int32_t j = k - INT32_MIN;
            return xl_of(t.xr_m[2 * j], t.xr_m[2 * j + 1], t.xr_e[j]);
        }
        xl r;
        r.re = ldexp(z.re, -k); r.im = ldexp(z.im, -k); r.e = k;
        return r;
    }

    __device__ static void init(State &s, const KArgs &a, double px, double py) {
        s.c = c_from_pix_xl(a, px, py);
        s.z = xl_zero(); s.d = xl_zero(); s.h = xl_zero();
        s.d.e = s.h.e = rel(XL_ZERO_E, 0);
        s.zs = zc();
        s.w = 0; s.n = 0; s.jl = 0; s.dyn = true; s.nul = false;
        s.orb.reset(a.backshift);
    }

    __device__ static bool step(State &s, const KArgs &a, Counters &k, int &reason, int32_t trip) {
        const Tables &t = a.t;
        if ((KIND == KIND_M2 || t.bla_on) && (s.w & 7) == 0) {
            int32_t stage, idx;
            const int32_t w0 = s.w;
            if (t.bla_on) {
                s.z = xl_of(as_z(s.z));                          // as the key takes it
                k.looks++;
                do {
                    stage = bla_lookup(t, s.z, s.w, idx);
                    if (stage >= 0) {
                        const int32_t st = 8 << stage;
                        const double *Mb = t.M + 4 * idx;
                        cplx A = mk(Mb[0], Mb[1]), B = mk(Mb[2], Mb[3]);
                        s.n += st;
                        s.w += st;
                        // A's exponent apart: A can be near the end of the binary64
                        // range, and dz/dc and dz/dz keep drifting mantissas (z alone
                        // is normalised, for the next lookup): 56 vector instructions
                        // instead of 86, with amax the 2048x2048 frames 720 -> 675 us
                        // (1e-300), 946 -> 887 us (1e-2000), 20.4 -> 18.3 ms (interior)
                        const int32_t kA = dexp(amax(A.re, A.im)) - 1;
                        A = mk(ldexp(A.re, -kA), ldexp(A.im, -kA));
                        int32_t ez = s.z.e + kA, sc = s.c.e - ez;
                        pin(sc);
                        if (sc > FAR) {
                            pin(sc);
                            s.z.re = ldexp(s.z.re, -sc); s.z.im = ldexp(s.z.im, -sc); ez += sc; sc = 0;
                        }
                        const cplx u = mk(s.z.re, s.z.im) * A, v = mk(s.c.re, s.c.im) * B;
                        s.z = xl_n(u.re + ldexp(v.re, sc), u.im + ldexp(v.im, sc), ez);
                        if (DC_ON(a)) { const cplx p = mk(s.d.re, s.d.im) * A; s.d.re = p.re; s.d.im = p.im; s.d.e += REL ? -kA : kA; }
                        if (DZ_ON(a)) { const cplx p = mk(s.h.re, s.h.im) * A; s.h.re = p.re; s.h.im = p.im; s.h.e += REL ? -kA : kA; }
                        s.jl += st; k.bla++;
                    }
                    pin(stage);
                } while (stage >= 0);
            }
            if (s.w != w0) {
                int32_t e = s.z.e;
                pin(e);
                s.zs = mk(ldexp(s.z.re, e), ldexp(s.z.im, e));
            }
            if constexpr (KIND == KIND_M2) {
                s.Z = t.Zn[s.w];
                s.kz = t.zn_k[s.w];
                if (DZ_ON(a)) s.Zh = DZz(t, s.nul ? 0 : s.w);
                s.A = s.zs + s.Z;
            }
        }
        s.n += 1;
        // Every table value the step reads is loaded here, as in HoloStd: the
        // orbit point, its code and the path values at w, the next orbit
        // point and its code (escape and rebase tests) and the dZndz value of
        // the interior test (z^d + c: after the step, whose partial products
        // need the registers; loaded first, it spilled at d = 3).  A step at
        // the end of the period or next to the orbit's last point (edge) takes
        // the general tests.
        int32_t w1 = s.w + 1, wh = w1;                   // wh: index of the interior test's dZndz value
        const bool edge = w1 >= min(t.order, t.div_iter - 1);
        if (edge) {
            pin(w1);
            if (w1 >= t.order) { w1 = 0; wh = s.n == t.order ? t.L : 0; }
        }
        if (DZ_ON(a) && s.nul) wh = 0;
        cplx Z0, Z1;
        int32_t k0, k1 = 0;
        xz Zd = xz_zero(), Zh = xz_zero(), H1 = xz_zero();
        if (DC_ON(a)) Zd = DCz(t, s.w);
        if constexpr (KIND == KIND_M2) {
            Z0 = s.Z; k0 = s.kz;
            if (DZ_ON(a)) Zh = s.Zh;
        } else {
            Z0 = t.Zn[s.w]; k0 = t.zn_k[s.w]; Z1 = t.Zn[w1];
            if (DZ_ON(a)) Zh = DZz(t, s.nul ? 0 : s.w);
        }
        if constexpr (KIND == KIND_M2) {
            // mandelbrot_M2.py:607-622: z (z + 2 Z) + c, 2 ((Z + z) d + Zd z)
            cplx A = s.A;                                            // Z + z
            cplx W = mk(__builtin_fma(2., Z0.re, s.zs.re), __builtin_fma(2., Z0.im, s.zs.im));   // z + 2 Z
            int32_t zt = s.z.e - trip;
            pin(zt);
            if (k0 < LOW_Z || s.dyn) {
                if (s.dyn) Zd = xz_zero();
                if (k0 < LOW_Z) {
                    const xl Zr = ZRv(t, k0, Z0);
                    s.z = xl_of(as_z(s.z));
                    zt = s.z.e - trip;
                    int32_t eK = max(Zr.e, s.z.e);               // exponent of A and W
                    if (eK < XL_ZERO_E / 2) eK = 0;              // Z = z = 0
                    const int32_t sZ = shift_of(Zr.e, eK), sz = shift_of(s.z.e, eK);
                    const cplx Zk = mk(ldexp(Zr.re, sZ), ldexp(Zr.im, sZ)), zk = mk(ldexp(s.z.re, sz), ldexp(s.z.im, sz));
                    A = Zk + zk;
                    W = mk(__builtin_fma(2., Zk.re, zk.re), __builtin_fma(2., Zk.im, zk.im));
                    s.z.e += eK; s.d.e -= eK; s.h.e -= eK;
                }
            }
            // the shifts of c and of the paths' terms to the exponents of
            // z W, A d and A h
            int32_t sz = s.c.e - s.z.e;
            int32_t sd = DC_ON(a) ? Zd.e + zt + s.d.e : -1, sh = DZ_ON(a) ? Zh.e + zt + s.h.e : -1;
            pin(sd); pin(sh);
            pin_after(w1, W.re, W.im);
            Z1 = t.Zn[w1]; k1 = t.zn_k[w1];
            cplx vh = zc();
            if (DZ_ON(a)) {                                      // (before dz/dc: HoloStd)
                vh = mk(Zh.re, Zh.im) * mk(s.z.re, s.z.im);
                pin_after(wh, vh.re, vh.im);
                H1 = DZz(t, wh);
            }
            if (max(sz, max(sd, sh)) > FAR) {
                if (sz > FAR) { W = mk(ldexp(W.re, -sz), ldexp(W.im, -sz)); s.z.e += sz; sz = 0; }
                if (sd > FAR) { s.d.re = ldexp(s.d.re, -sd); s.d.im = ldexp(s.d.im, -sd); s.d.e -= sd; sd = 0; }
                if (sh > FAR) { s.h.re = ldexp(s.h.re, -sh); s.h.im = ldexp(s.h.im, -sh); s.h.e -= sh; sh = 0; }
            }
            const cplx z = mk(s.z.re, s.z.im);
            if (DC_ON(a)) {
                const cplx u = A * mk(s.d.re, s.d.im), v = mk(Zd.re, Zd.im) * z;
                s.d.re = u.re + ldexp(v.re, sd); s.d.im = u.im + ldexp(v.im, sd);
            }
            if (DZ_ON(a)) {
                const cplx u = A * mk(s.h.re, s.h.im);
                s.h.re = u.re + ldexp(vh.re, sh); s.h.im = u.im + ldexp(vh.im, sh);
            }
            const cplx u = z * W;
            s.z.re = u.re + ldexp(s.c.re, sz); s.z.im = u.im + ldexp(s.c.im, sz);
            s.zs = mk(ldexp(s.z.re, s.z.e), ldexp(s.z.im, s.z.e));
        } else {
            // mandelbrot_Mn.py:646-729 (p_zn_derivs of models.hpp).  zk, Zk: z
            // and Z in units of 2^eK; the running factor mul of term q is then
            // in units of 2^(q eK), and tmp = z mul on z's mantissa comes back
            // to that scale with the shift et.
            cplx Zk = Z0, zk = s.zs;
            int32_t eK = 0;
            const bool far_z = (uint32_t)(k0 - LOW_Z) > (uint32_t)(HIGH_Z - LOW_Z);
            if (far_z || s.dyn) {
                if (s.dyn) Zd = xz_zero();
                if (far_z) {
                    const xl Zr = ZRv(t, k0, Z0);
                    s.z = xl_of(as_z(s.z));
                    eK = max(Zr.e, s.z.e);
                    if (eK < XL_ZERO_E / 2) eK = 0;              // Z = z = 0
                    const int32_t sZ = shift_of(Zr.e, eK), sz = shift_of(s.z.e, eK);
                    Zk = mk(ldexp(Zr.re, sZ), ldexp(Zr.im, sZ));
                    zk = mk(ldexp(s.z.re, sz), ldexp(s.z.im, sz));
                }
            }
            const int32_t et = s.z.e - eK;
            int32_t ez = s.z.e + (DEG - 1) * eK, sz = s.c.e - ez;
            Deriv D[2];
            if (DC_ON(a)) D[0].set(s.d, Zd, et);
            if (DZ_ON(a)) D[1].set(s.h, Zh, et);
            int32_t far = sz;
            if (DC_ON(a)) far = max(far, max(D[0].s1, D[0].s2));
            if (DZ_ON(a)) far = max(far, max(D[1].s1, D[1].s2));
            int32_t cut = 0;
            if (far > FAR) {
                if (sz > FAR) { cut = -sz; ez += sz; sz = 0; }
                if (DC_ON(a)) D[0].near(et);
                if (DZ_ON(a)) D[1].near(et);
            }
            const cplx z = mk(s.z.re, s.z.im);
            cplx mul = zk + scale(cbinom(DEG, 1), Zk);
            cplx tmp = z * mul;
            if (DC_ON(a)) D[0].term(z, mul, scale(cbinom(DEG, 1), D[0].Z), true);
            if (DZ_ON(a)) D[1].term(z, mul, scale(cbinom(DEG, 1), D[1].Z), true);
            cplx Zpk = Zk;
#pragma unroll
            for (int q = 2; q < DEG; q++) {
                const cplx qZ = scale((double)q, Zpk);
                Zpk = Zpk * Zk;
                mul = mk(ldexp(tmp.re, et), ldexp(tmp.im, et)) + scale(cbinom(DEG, q), Zpk);
                if (DC_ON(a)) D[0].term(z, mul, scale(cbinom(DEG, q), qZ * D[0].Z), false);
                if (DZ_ON(a)) D[1].term(z, mul, scale(cbinom(DEG, q), qZ * D[1].Z), false);
                tmp = z * mul;
            }
            if (cut != 0) {            // a branch: as selects, seven instructions a step (z^3 + c at 1e-800 508 -> 497 us)
                pin(cut);
                tmp = mk(ldexp(tmp.re, cut), ldexp(tmp.im, cut));
            }
            if (DC_ON(a)) { s.d.re = D[0].t.re; s.d.im = D[0].t.im; s.d.e = D[0].e + (DEG - 1) * eK; }
            if (DZ_ON(a)) { s.h.re = D[1].t.re; s.h.im = D[1].t.im; s.h.e = D[1].e + (DEG - 1) * eK; }
            s.z.re = tmp.re + ldexp(s.c.re, sz); s.z.im = tmp.im + ldexp(s.c.im, sz); s.z.e = ez;
            s.zs = mk(ldexp(s.z.re, ez), ldexp(s.z.im, ez));
            if (DZ_ON(a)) H1 = DZz(t, wh);
        }
        s.w = w1;
        // the stop and rebase tests evaluated together, as in HoloStd
        // in binary64: what underflows or overflows there lies far on one side
        // of eps
        bool t_int = false;
        double qre = 0.;
        if (DZ_ON(a)) {
            qre = ldexp(s.h.re, rel(s.h.e, trip + 1)) + ldexp(H1.re, H1.e);
            t_int = fabs(qre) < a.eps_hi;
        }
        const cplx ZZ = s.zs + Z1;
        const bool t_esc = amax(ZZ.re, ZZ.im) > a.esc_lo;
        const bool dyn = (fabs(ZZ.re) <= fabs(s.zs.re)) && (fabs(ZZ.im) <= fabs(s.zs.im));
        if constexpr (KIND == KIND_M2) { s.Z = Z1; s.kz = k1; s.A = ZZ; s.Zh = H1; }
        if (!(s.n >= a.max_iter || t_int || t_esc || edge || dyn || s.orb.due(s.n))) { s.dyn = false; return false; }
        const auto stop = [&](int r) { s.d.e = rel(s.d.e, trip + 1); reason = r; return true; };
        if (s.n >= a.max_iter) return stop(0);
        if (t_int) {
            const double qim = ldexp(s.h.im, rel(s.h.e, trip + 1)) + ldexp(H1.im, H1.e);
            if (qre * qre + qim * qim < a.eps2) return stop(2);
        }
        s.orb.record(s.n, a.backshift, ZZ.re, ZZ.im);
        if (t_esc && ZZ.re * ZZ.re + ZZ.im * ZZ.im > a.M2) return stop(1);
        // both rebases (perturbation.py:1283-1372) share the derivative
        // updates: one block, whichever of them a lane takes
        const bool reb_div = s.w >= t.div_iter - 1;
        bool reb = reb_div, plain = true;                // plain: the new z is ZZ
        xl ZZx;
        if (!reb_div) {
            s.dyn = dyn;
            if (s.dyn) {
                // Decided by |z + Z|^2 <= |z|^2 on extended-range values.  Where
                // no component of ZZ is zero or small (the components of z are
                // then no smaller), ZZ is their sum to the bit, the squares
                // round alike, and components that are no larger have a sum of
                // squares that is no larger: 5 instructions instead of 60
                // (1920x1080 at 1e-800: z^3 + c 541 -> 513 us, z^6 + c 555 -> 520).
                const int32_t kr = KIND == KIND_M2 ? k1 : t.zn_k[w1];
                plain = amax(ZZ.re, ZZ.im) >= 0x1p-480 && amin(ZZ.re, ZZ.im) >= 0x1p-1000 && kr >= ZK_REGISTER;
                reb = true;
                if (!plain) {
                    s.z = xl_of(as_z(s.z));
                    ZZx = s.z + ZRv(t, kr, Z1);
                    reb = le_abs2(ZZx, s.z);
                }
            }
        }
        if (reb) {
            if (plain) { s.zs = ZZ; s.z = xl_of(ZZ); }
            else { s.z = ZZx; s.zs = to_std(ZZx); }
            // Neither term normalised: the sum aligns them by their exponents,
            // and what a drifting mantissa loses there lies far below the other
            // term's last place; the sum's normalisation covers the result.
            if (DC_ON(a)) {
                s.d = add_n(xz{s.d.re, s.d.im, rel(s.d.e, trip + 1)}, DCz(t, s.w));
                s.d.e = rel(s.d.e, trip + 1);
            }
            if (DZ_ON(a) && !s.nul) {
                s.h = add_n(xz{s.h.re, s.h.im, rel(s.h.e, trip + 1)}, H1);   // dZndz at w (at L after a full period)
                s.h.e = rel(s.h.e, trip + 1);
            }
            s.nul = DZ_ON(a);
            s.w = 0;
            k.reb++;
        }
        return false;
    }

    __device__ static void finish(State &s, const KArgs &a, const KArgs &g, int64_t i, int reason) {
        const int64_t n = g.ld;
        s.z = xl_of(as_z(s.z));
        cplx z = to_std(s.z) + a.t.Zn[s.w];
        g.Z[2 * i] = z.re; g.Z[2 * i + 1] = z.im;
        int f = 1;
        // perturbation.py:1377-1380 writes zn and dzndc back only; the
        // standard dzndz field keeps the 0 written by numba_initialize
        if (DZ_ON(a)) { g.Z[2 * (n + i)] = 0.; g.Z[2 * (n + i) + 1] = 0.; f = 2; }
        if (DC_ON(a)) {
            cplx d = to_std(add_n(as_z(xl_of(as_z(s.d))), DCz(a.t, s.w)));
            g.Z[2 * (f * n + i)] = d.re; g.Z[2 * (f * n + i) + 1] = d.im;
        }
        if constexpr (ORB) orbit_finish_holo<KIND, DEG>(s.orb, a, g, s.n, to_std(s.c), i);
        g.U[i] = s.w; g.stop_iter[i] = s.n; g.stop_reason[i] = (int8_t)reason;
    }
};

// --------------------------------------------------------------------------
// Burning-ship family, binary64 deltas
template <int FL, bool ORB = false>
struct BsStd {
    struct State { double x, y, P[4], a, b; int32_t w, n, jl; bool dyn; OrbitRec<ORB> orb; };

    __device__ static void init(State &s, const KArgs &a, double px, double py) {
        xc cx = renorm_c(a.dx_m * (a.lin[0] * px + a.lin[1] * py),
                         a.dx_m * (a.lin[2] * px + a.lin[3] * py), a.dx_e);
        s.a = to_std(mkf(cx.re, cx.e) + mkf(a.drift_m[0], a.drift_e[0]));
        s.b = to_std(mkf(cx.im, cx.e) + mkf(a.drift_m[1], a.drift_e[1]));
        s.x = 0.; s.y = 0.; s.P[0] = s.P[1] = s.P[2] = s.P[3] = 0.;
        s.w = 0; s.n = 0; s.jl = 0; s.dyn = true;
        s.orb.reset(a.backshift);
    }

    __device__ static bool step(State &s, const KArgs &a, Counters &k, int &reason, int32_t) {
        const Tables &t = a.t;
        if (t.bla_on && (s.w & 7) == 0) {
            k.looks++;
            int32_t stage, idx;
            do {
                stage = bla_lookup(t, s.x, s.y, s.w, idx);
                if (stage >= 0) {
                    const int32_t st = 8 << stage;
                    const double *M = t.M + 8 * idx;
                    s.n += st; s.w += st;
                    double nx = M[0] * s.x + M[1] * s.y + M[4] * s.a + M[5] * s.b;
                    double ny = M[2] * s.x + M[3] * s.y + M[6] * s.a + M[7] * s.b;
                    s.x = nx; s.y = ny;
                    if (a.calc_dc) {
                        double p0 = M[0] * s.P[0] + M[1] * s.P[2];
                        double p1 = M[0] * s.P[1] + M[1] * s.P[3];
                        double p2 = M[2] * s.P[0] + M[3] * s.P[2];
                        double p3 = M[2] * s.P[1] + M[3] * s.P[3];
                        s.P[0] = p0; s.P[1] = p1; s.P[2] = p2; s.P[3] = p3;
                    }
                    s.jl += st; k.bla++;
                }
                pin(stage);
            } while (stage >= 0);
        }
        s.n += 1;
        // the step's table reads first, its tests together (as in HoloStd)
        const int32_t w1 = (s.w + 1 >= t.order) ? 0 : s.w + 1;
        const cplx R = t.Zn[s.w];
        const cplx R1 = t.Zn[w1];
        if (a.calc_dc) {
            double Rd[4] = {0., 0., 0., 0.};
            if (!s.dyn) { Rd[0] = t.bs[0][s.w]; Rd[1] = t.bs[1][s.w]; Rd[2] = t.bs[2][s.w]; Rd[3] = t.bs[3][s.w]; }
            bs_hess<FL>(s.x, s.y, s.P, R.re, R.im, Rd);
        }
        bs_zn<FL>(s.x, s.y, R.re, R.im, s.a, s.b);
        const double XX = s.x + R1.re, YY = s.y + R1.im;
        const bool t_esc = amax(XX, YY) > a.esc_lo;
        const bool reb_div = w1 >= t.div_iter - 1;
        const bool dyn = (fabs(XX) <= fabs(s.x)) && (fabs(YY) <= fabs(s.y));
        if (!(s.n >= a.max_iter || t_esc || reb_div || dyn || s.orb.due(s.n))) { s.w = w1; s.dyn = false; return false; }
        if (s.n >= a.max_iter) { reason = 0; return true; }
        s.w = w1;
        s.orb.record(s.n, a.backshift, XX, YY);
        if (t_esc && XX * XX + YY * YY > a.M2) { reason = 1; return true; }
        bool reb = reb_div;
        if (!reb) {
            s.dyn = dyn;
            reb = dyn;
        }
        if (reb) {
            s.x = XX; s.y = YY;
            if (a.calc_dc)
                for (int q = 0; q < 4; q++) s.P[q] += t.bs[q][s.w];
            s.w = 0;
            k.reb++;
        }
        return false;
    }

    __device__ static void finish(const State &s, const KArgs &a, const KArgs &g, int64_t i, int reason) {
        const int64_t n = g.ld;
        const cplx R = a.t.Zn[s.w];
        g.Z[i] = s.x + R.re; g.Z[n + i] = s.y + R.im;
        if (a.calc_dc)
            for (int q = 0; q < 4; q++) g.Z[(2 + q) * n + i] = s.P[q] + a.t.bs[q][s.w];
        if constexpr (ORB) orbit_finish_bs<FL>(s.orb, a, g, s.n, s.a, s.b, i);
        g.U[i] = s.w; g.stop_iter[i] = s.n; g.stop_reason[i] = (int8_t)reason;
    }
};

// Burning-ship family, Xrange deltas, on drifting mantissas as HoloXr: x and y
// share one exponent (e), the four Jacobian deltas another (eP), a and b a
// third; a shared exponent changes no rounding, since the mantissas stay far
// inside the binary64 range.  An orbit point's Jacobian values are brought to
// the scale of the deltas' mantissas divided by z's, R' = R 2^(eR + e - eP),
// so that a product of z's mantissa with one is a delta's mantissa; X, Y and
// their sums with x and y are binary64 values.  The folds' derivative terms
// of the orbit (a pixel on the other side of a fold than the orbit) are formed
// in a branch.  An orbit point whose larger coordinate is below 2^LOW_Z (zero,
// the Xrange register) takes the general step on separate exponents.
// Bound by vector instruction issue; with every real on its own exponent, each
// sum aligned, tested for zero and each result renormalised, a trip took 515
// instructions (1920x1080 at 1e-800: 1831 us, now 840).
template <int FL, bool ORB = false, int DER = -1>
struct BsXr {
    __device__ static bool DC_ON(const KArgs &a) { if constexpr (DER >= 0) return DER != 0; else return a.calc_dc != 0; }
    struct State { double x, y, P[4], a, b, xs, ys; int32_t e, eP, ec, w, n, jl; bool dyn; OrbitRec<ORB> orb; };
    static constexpr bool LAZY = true;
    static constexpr int32_t LOW_Z = -20, FAR = 256;

    // two (four) values on one exponent, the larger normalised
    __device__ static void norm2(double &x, double &y, int32_t &e) {
        const xl v = xl_n(x, y, e);
        x = v.re; y = v.im; e = v.e;
    }
    __device__ static void norm4(double *P, int32_t &e) {
        const double mx = amax(amax(P[0], P[1]), amax(P[2], P[3]));
        const int32_t k = dexp(mx) - 1;
        for (int q = 0; q < 4; q++) P[q] = ldexp(P[q], -k);
        e = (mx == 0.) ? XL_ZERO_E : e + k;
    }
    __device__ static void renorm(State &s, const KArgs &a, int32_t = 0) {
        norm2(s.x, s.y, s.e);
        if (DC_ON(a)) norm4(s.P, s.eP);
    }
    // separate exponents, and back
    __device__ static void join2(xlf u, xlf v, double &x, double &y, int32_t &e) {
        e = max(u.e, v.e);
        x = ldexp(u.m, shift_of(u.e, e)); y = ldexp(v.m, shift_of(v.e, e));
    }
    __device__ static void join4(const xlf *u, double *P, int32_t &e) {
        e = max(max(u[0].e, u[1].e), max(u[2].e, u[3].e));
        for (int q = 0; q < 4; q++) P[q] = ldexp(u[q].m, shift_of(u[q].e, e));
    }
    __device__ static xlf PATH(const Tables &t, int q, int32_t i) { return xlf_of(t.bs[q][i], t.bs_e[q][i]); }
    // orbit point i, normalised per coordinate: the register's Xrange
    // values where the binary64 orbit underflows, the binary64 values
    // elsewhere, scaled by the exponents the tables hold for them
    // (from the point's codes kx, ky and binary64 value R, loaded beforehand)
    __device__ static void ZRv(const Tables &t, int32_t kx, int32_t ky, cplx R, xlf &X, xlf &Y) {
        if (kx < ZK_REGISTER) {
            const int32_t j = kx - INT32_MIN;
            X = xlf_of(t.xr_m[2 * j], t.xr_e[2 * j]); Y = xlf_of(t.xr_m[2 * j + 1], t.xr_e[2 * j + 1]);
        } else {
            X.m = ldexp(R.re, -kx); X.e = kx;
            Y.m = ldexp(R.im, -ky); Y.e = ky;
        }
    }

    __device__ static void init(State &s, const KArgs &a, double px, double py) {
        join2(xlf_of(a.dx_m * (a.lin[0] * px + a.lin[1] * py), a.dx_e) + xlf_of(a.drift_m[0], a.drift_e[0]),
              xlf_of(a.dx_m * (a.lin[2] * px + a.lin[3] * py), a.dx_e) + xlf_of(a.drift_m[1], a.drift_e[1]), s.a, s.b, s.ec);
        s.x = s.y = 0.; s.P[0] = s.P[1] = s.P[2] = s.P[3] = 0.;
        s.e = s.eP = XL_ZERO_E;
        s.xs = 0.; s.ys = 0.;
        s.w = 0; s.n = 0; s.jl = 0; s.dyn = true;
        s.orb.reset(a.backshift);
    }

    // The fold |F + f| - |F| of burning_ship.py:19-60 (diffabs, ddX, ddx), F in
    // the scale of f's mantissa: sg is F's sign, cross whether F + f lies on
    // the other side of zero.
    struct Fold {
        double F, f;              // sg F, sg f
        uint32_t sg;
        bool cross;
        __device__ Fold(double Fv, double fv) {
            sg = Fv < 0. ? 0x80000000u : 0u;
            F = flip(Fv, sg); f = flip(fv, sg);
            cross = !(F + f >= 0.);
        }
        // sign bit of the value F + f (a z that underflows binary64 included)
        __device__ uint32_t sum_sign() const { return flip(F + f, sg) < 0. ? 0x80000000u : 0u; }
        __device__ double diff() const { return cross ? -__builtin_fma(2., F, f) : f; }
    };
    __device__ static double flip(double v, uint32_t sg) { return from_bits(bits(v) ^ ((uint64_t)sg << 32)); }

    // one step on shared exponents (bs_hess and bs_zn of models.hpp, the same
    // operations in the same order); a, b: c's parts in z's scale; R: the
    // orbit's Jacobian as above
    __device__ static void fast_step(State &s, const KArgs &ka, double X, double Y, double a, double b, const double *R) {
        const int32_t e = s.e;
        const double x = s.x, y = s.y, xs = s.xs, ys = s.ys;
        const double Ux = __builtin_fma(2., X, xs), Uy = __builtin_fma(2., Y, ys);     // x + 2 X, y + 2 Y
        const double Xs = X + xs, Ys = Y + ys;
        const double q0 = x * Ux - y * Uy;                                  // Re (z (z + 2 Z))
        constexpr bool FX = FL == 4 || FL == 5, FXY = FL == 1 || FL == 5, FY = FL == 2 || FL == 3;
        const double t0 = FXY ? x * ys + x * Y + y * X : X * y + Y * x + x * ys;
        // the fold of the x part (X^2 - Y^2), of the y part (X Y), of Y
        const double Fx = FX ? X * X - Y * Y : 0., Fy = FXY ? X * Y : FY ? Y : 0.;
        const Fold gx(FX ? ldexp(Fx, -e) : 0., q0), gy(FXY || FY ? ldexp(Fy, -e) : 0., FY ? y : t0);
        const double da = gy.diff(), ab = fabs(Ys);
        const uint32_t sy = FY ? gy.sum_sign() : 0u;
        if (DC_ON(ka)) {
            double P[4];
#pragma unroll
            for (int c = 0; c < 2; c++) {                                   // d/da, d/db
                const double xp = s.P[c], yp = s.P[2 + c], Xp = R[c], Yp = R[2 + c];
                const double xe = ldexp(xp, e), ye = ldexp(yp, e);          // the deltas in R's scale
                if constexpr (FX) {
                    const double o = xp * Ux + x * (xe + 2. * Xp) - yp * Uy - y * (ye + 2. * Yp);
                    P[c] = flip(o, gx.sg);
                    if (gx.cross) P[c] = -flip(2. * ldexp(2. * (X * Xp - Y * Yp), -e) + o, gx.sg);
                } else if constexpr (FL == 3) {
                    const double h = gy.cross ? -flip(2. * ldexp(Yp, -e) + yp, gy.sg) : flip(yp, gy.sg);
                    P[c] = xp * Ux + x * (xe + 2. * Xp) - Yp * da - Y * h - yp * ab - flip(y, sy) * (Yp + ye);
                } else {
                    P[c] = 2. * ((Xs * xp + Xp * x) - (Ys * yp + Yp * y));
                }
                if constexpr (FXY) {
                    const double o = xp * ys + xs * yp + xp * Y + x * Yp + yp * X + y * Xp;
                    P[2 + c] = 2. * flip(o, gy.sg);
                    if (gy.cross) P[2 + c] = -2. * flip(2. * ldexp(Xp * Y + X * Yp, -e) + o, gy.sg);
                } else if constexpr (FL == 2) {
                    const double h = gy.cross ? -flip(2. * ldexp(Yp, -e) + yp, gy.sg) : flip(yp, gy.sg);
                    P[2 + c] = 2. * (Xp * da + X * h + xp * ab + flip(x, sy) * (Yp + ye));
                } else {
                    P[2 + c] = 2. * (Xp * y + X * yp + Yp * x + Y * xp + xp * ys + xs * yp);
                }
            }
            for (int q = 0; q < 4; q++) s.P[q] = P[q];
        }
        if constexpr (FX) s.x = gx.diff() + a;
        else if constexpr (FL == 3) s.x = x * Ux - Y * da - y * ab + a;
        else s.x = q0 + a;
        if constexpr (FXY) s.y = __builtin_fma(2., da, -b);
        else if constexpr (FL == 2) s.y = __builtin_fma(2., X * da + x * ab, -b);
        else s.y = __builtin_fma(2., t0, -b);
    }

    // the same on separate exponents
    __device__ static void general_step(State &s, const KArgs &a, int32_t kx, int32_t ky, cplx R0) {
        const Tables &t = a.t;
        xlf X, Y;
        ZRv(t, kx, ky, R0, X, Y);
        const xzf x = as_zf(xlf_of(s.x, s.e)), y = as_zf(xlf_of(s.y, s.e)), Xz = as_zf(X), Yz = as_zf(Y);
        if (DC_ON(a)) {
            const xzf z0 = as_zf(xlf_zero());
            xzf Rd[4] = {z0, z0, z0, z0};
            // the host's Xrange path records keep |mantissa| within 2^+-100 (a
            // zero entry with the zero exponent code): used as loaded
            if (!s.dyn) for (int q = 0; q < 4; q++) { Rd[q].m = t.bs[q][s.w]; Rd[q].e = t.bs_e[q][s.w]; }
            xzf P[4];
            for (int q = 0; q < 4; q++) P[q] = as_zf(xlf_of(s.P[q], s.eP));
            bs_hess<FL>(x, y, P, Xz, Yz, Rd);
            xlf Pn[4];
            for (int q = 0; q < 4; q++) Pn[q] = xlf_of(P[q]);
            join4(Pn, s.P, s.eP);
        }
        xzf nx = x, ny = y;
        bs_zn<FL>(nx, ny, Xz, Yz, as_zf(xlf_of(s.a, s.ec)), as_zf(xlf_of(s.b, s.ec)));
        join2(xlf_of(nx), xlf_of(ny), s.x, s.y, s.e);
    }

    __device__ static bool step(State &s, const KArgs &a, Counters &k, int &reason, int32_t) {
        const Tables &t = a.t;
        if (t.bla_on && (s.w & 7) == 0) {
            k.looks++;
            int32_t stage, idx;
            do {
                stage = bla_lookup(t, s.xs, s.ys, s.w, idx);
                if (stage >= 0) {
                    const int32_t st = 8 << stage;
                    // A z + B c and A J on shared exponents; the coefficients are
                    // split into mantissas on one exponent each (they reach the
                    // ends of the binary64 range)
                    double M[8];
                    for (int q = 0; q < 8; q++) M[q] = t.M[8 * idx + q];
                    s.n += st; s.w += st;
                    renorm(s, a);
                    int32_t eA = 0, eB = 0;
                    norm4(M, eA);
                    norm4(M + 4, eB);
                    double x = s.x, y = s.y;
                    int32_t e = s.e + eA, sc = s.ec + eB - e;
                    if (sc > FAR) { x = ldexp(x, -sc); y = ldexp(y, -sc); e += sc; sc = 0; }
                    s.x = M[0] * x + M[1] * y + ldexp(M[4] * s.a, sc) + ldexp(M[5] * s.b, sc);
                    s.y = M[2] * x + M[3] * y + ldexp(M[6] * s.a, sc) + ldexp(M[7] * s.b, sc);
                    s.e = e;
                    s.xs = ldexp(s.x, e); s.ys = ldexp(s.y, e);
                    if (DC_ON(a)) {
                        const double P0 = s.P[0], P1 = s.P[1], P2 = s.P[2], P3 = s.P[3];
                        s.P[0] = M[0] * P0 + M[1] * P2;
                        s.P[1] = M[0] * P1 + M[1] * P3;
                        s.P[2] = M[2] * P0 + M[3] * P2;
                        s.P[3] = M[2] * P1 + M[3] * P3;
                        s.eP += eA;
                    }
                    s.jl += st; k.bla++;
                }
                pin(stage);
            } while (stage >= 0);
        }
        s.n += 1;
        // the step's table reads first, its tests together (as in HoloStd)
        const int32_t w1 = (s.w + 1 >= t.order) ? 0 : s.w + 1;
        const int32_t kx0 = t.zn_k[2 * s.w], ky0 = t.zn_k[2 * s.w + 1];
        const cplx R0 = t.Zn[s.w], R1 = t.Zn[w1];
        double R[4] = {0., 0., 0., 0.};
        int32_t Re[4] = {XL_ZERO_E, XL_ZERO_E, XL_ZERO_E, XL_ZERO_E};
        if (DC_ON(a)) for (int q = 0; q < 4; q++) { R[q] = t.bs[q][s.w]; Re[q] = t.bs_e[q][s.w]; }
        if (max(kx0, ky0) < LOW_Z) {
            general_step(s, a, kx0, ky0, R0);
        } else {
            if (s.dyn) for (int q = 0; q < 4; q++) { R[q] = 0.; Re[q] = XL_ZERO_E; }
            int32_t sc = s.ec - s.e, sR[4];
            for (int q = 0; q < 4; q++) sR[q] = Re[q] + s.e - s.eP;
            const int32_t mR = DC_ON(a) ? max(max(sR[0], sR[1]), max(sR[2], sR[3])) : 0;
            if (max(sc, mR) > FAR) {
                int32_t up = 0;
                if (sc > FAR) { s.x = ldexp(s.x, -sc); s.y = ldexp(s.y, -sc); s.e += sc; up = sc; sc = 0; }
                if (DC_ON(a)) {
                    const int32_t m = mR + up;
                    const int32_t dn = m > FAR ? m : 0;
                    for (int q = 0; q < 4; q++) { s.P[q] = ldexp(s.P[q], -dn); sR[q] += up - dn; }
                    s.eP += dn;
                }
            }
            for (int q = 0; q < 4; q++) R[q] = ldexp(R[q], sR[q]);
            fast_step(s, a, R0.re, R0.im, ldexp(s.a, sc), ldexp(s.b, sc), R);
        }
        s.xs = ldexp(s.x, s.e); s.ys = ldexp(s.y, s.e);
        const double XX = s.xs + R1.re, YY = s.ys + R1.im;
        const bool t_esc = amax(XX, YY) > a.esc_lo;
        const bool reb_div = w1 >= t.div_iter - 1;
        const bool dyn = (fabs(XX) <= fabs(s.xs)) && (fabs(YY) <= fabs(s.ys));
        if (!(s.n >= a.max_iter || t_esc || reb_div || dyn || s.orb.due(s.n))) { s.w = w1; s.dyn = false; return false; }
        if (s.n >= a.max_iter) { reason = 0; return true; }
        s.w = w1;
        s.orb.record(s.n, a.backshift, XX, YY);
        if (t_esc && XX * XX + YY * YY > a.M2) { reason = 1; return true; }
        bool reb = reb_div;
        xlf x = xlf_of(s.x, s.e), y = xlf_of(s.y, s.e);
        if (reb_div) {
            x = xlf_of(XX, 0); y = xlf_of(YY, 0);
        } else {
            s.dyn = dyn;
            if (s.dyn) {
                xlf X1, Y1;
                ZRv(t, t.zn_k[2 * w1], t.zn_k[2 * w1 + 1], R1, X1, Y1);
                const xlf XXx = x + X1, YYx = y + Y1;
                reb = le(XXx * XXx + YYx * YYx, x * x + y * y);
                if (reb) { x = XXx; y = YYx; }
            }
        }
        if (reb) {
            s.xs = to_std(x); s.ys = to_std(y);
            join2(x, y, s.x, s.y, s.e);
            if (DC_ON(a)) {
                xlf Pn[4];
                for (int q = 0; q < 4; q++) Pn[q] = xlf_of(s.P[q], s.eP) + PATH(t, q, s.w);
                join4(Pn, s.P, s.eP);
            }
            s.w = 0;
            k.reb++;
        }
        return false;
    }

    __device__ static void finish(const State &s, const KArgs &a, const KArgs &g, int64_t i, int reason) {
        const int64_t n = g.ld;
        const cplx R = a.t.Zn[s.w];
        g.Z[i] = to_std(xlf_of(s.x, s.e) + R.re); g.Z[n + i] = to_std(xlf_of(s.y, s.e) + R.im);
        if (DC_ON(a))
            for (int q = 0; q < 4; q++) g.Z[(2 + q) * n + i] = to_std(xlf_of(s.P[q], s.eP) + PATH(a.t, q, s.w));
        if constexpr (ORB) orbit_finish_bs<FL>(s.orb, a, g, s.n, to_std(xlf_of(s.a, s.ec)), to_std(xlf_of(s.b, s.ec)), i);
        g.U[i] = s.w; g.stop_iter[i] = s.n; g.stop_reason[i] = (int8_t)reason;
    }
};

}  // namespace fsg
