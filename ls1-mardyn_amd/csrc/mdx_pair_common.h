// mdx_pair_common.h -- pieces shared by the pair kernels (mdx_pairs.hip) and
// the adjoint kernel (mdx_adjoint.hip): vector helpers, the seven site-pair
// bodies, site accessors per precision, the neighbour images of a cell and the
// LDS tile of staged neighbour sites.
#pragma once

#include "mdx_internal.h"

namespace mdx {


template <typename R> struct V3 { R x, y, z; };

template <typename R> __device__ __forceinline__ R dot3(V3<R> a, V3<R> b) {
    return a.x * b.x + a.y * b.y + a.z * b.z;
}
template <typename R> __device__ __forceinline__ V3<R> cross3(V3<R> a, V3<R> b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

template <typename R> struct Math;
template <> struct Math<double> {
    // 1/x: v_rcp_f64 refined by two Newton steps (error <= 1 ulp; the
    // reference's AVX2 build likewise refines rcp estimates instead of
    // dividing, RealVecDouble.h:414-467); sqrt(1/r^2) as in the NOVEC build.
    static __device__ __forceinline__ double rcp(double x) {
        double y = __builtin_amdgcn_rcp(x);
        double e = __builtin_fma(-x, y, 1.0);
        y = __builtin_fma(y, e, y);
        e = __builtin_fma(-x, y, 1.0);
        return __builtin_fma(y, e, y);
    }
    static __device__ __forceinline__ double rinv(double r2, double r2inv) { return sqrt(r2inv); }
    // 1/r^2 and 1/r of one distance
    static __device__ __forceinline__ void inv2(double r2, double &r2inv, double &rinv) {
        r2inv = rcp(r2);
        rinv = sqrt(r2inv);
    }
};
template <> struct Math<float> {
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    static __device__ __forceinline__ float rinv(float r2, float) { return __builtin_amdgcn_rsqf(r2); }
    // two hardware approximations (1 ulp each); 1/r^2 as the square of 1/r
    // would save one but doubles the bias of v_rsq_f32 in every force, which
    // the sums of neutral molecules (charges of both signs) amplify
    static __device__ __forceinline__ void inv2(float r2, float &r2inv, float &rinv) {
        r2inv = __builtin_amdgcn_rcpf(r2);
        rinv = __builtin_amdgcn_rsqf(r2);
    }
};

template <typename R> struct PO {
    V3<R> f, M1, M2;
    R u, rf;
};

// _loopBodyCharge (VectorizedCellProcessor.cpp:227-277)
template <typename R> __device__ __forceinline__ void body_cc(V3<R> d, R q1, R q2, PO<R> &o) {
    R r2 = dot3(d, d);
    R r2inv, rinv;
    Math<R>::inv2(r2, r2inv, rinv);
    R upot = q1 * q2 * rinv;
    R fac = upot * r2inv;
    o.f = {d.x * fac, d.y * fac, d.z * fac};
    o.u = upot;
}

// _loopBodyChargeDipole (VectorizedCellProcessor.cpp:279-347): first charge,
// second dipole; M2 = torque on the dipole.
template <typename R>
__device__ __forceinline__ void body_cd(V3<R> d, R q, V3<R> e, R p, PO<R> &o) {
    R r2 = dot3(d, d);
    R r2inv, rinv;
    Math<R>::inv2(r2, r2inv, rinv);
    R re = dot3(d, e);
    R qpr3 = q * p * (r2inv * rinv);
    R fac = r2inv * R(3) * re;
    o.f = {qpr3 * (e.x - d.x * fac), qpr3 * (e.y - d.y * fac), qpr3 * (e.z - d.z * fac)};
    o.u = -(qpr3 * re);
    V3<R> c = cross3(e, d);
    o.M2 = {qpr3 * c.x, qpr3 * c.y, qpr3 * c.z};
}

// _loopBodyDipole (VectorizedCellProcessor.cpp:349-442) incl. reaction field
template <typename R>
__device__ __forceinline__ void body_dd(V3<R> d, V3<R> e1, R p1, V3<R> e2, R p2, R epsRFInvrc3,
                                        PO<R> &o) {
    R r2 = dot3(d, d);
    R r2inv, rinv;
    Math<R>::inv2(r2, r2inv, rinv);
    R r2three = R(3) * r2inv;
    R p1p2 = p1 * p2;
    R rffac = p1p2 * epsRFInvrc3;
    R p1p2r3 = p1p2 * rinv * r2inv;
    R p1p2r5 = p1p2r3 * r2three;
    R e1e2 = dot3(e1, e2), re1 = dot3(d, e1), re2 = dot3(d, e2);
    R re1t = re1 * r2three, re2t = re2 * r2three;
    R re1re2 = r2inv * re1 * re2;
    R gg = e1e2 - R(5) * re1re2;
    o.f = {p1p2r5 * (d.x * gg + e1.x * re2 + e2.x * re1),
           p1p2r5 * (d.y * gg + e1.y * re2 + e2.y * re1),
           p1p2r5 * (d.z * gg + e1.z * re2 + e2.z * re1)};
    o.u = p1p2r3 * (e1e2 - R(3) * re1re2);
    o.rf = rffac * e1e2;
    V3<R> c12 = cross3(e1, e2), e1xd = cross3(e1, d), e2xd = cross3(e2, d);
    o.M1 = {p1p2r3 * (re2t * e1xd.x - c12.x) + rffac * c12.x,
            p1p2r3 * (re2t * e1xd.y - c12.y) + rffac * c12.y,
            p1p2r3 * (re2t * e1xd.z - c12.z) + rffac * c12.z};
    o.M2 = {p1p2r3 * (re1t * e2xd.x + c12.x) - rffac * c12.x,
            p1p2r3 * (re1t * e2xd.y + c12.y) - rffac * c12.y,
            p1p2r3 * (re1t * e2xd.z + c12.z) - rffac * c12.z};
}

// _loopBodyChargeQuadrupole (VectorizedCellProcessor.cpp:444-524): first
// charge, second quadrupole; M2 = torque on the quadrupole.
template <typename R>
__device__ __forceinline__ void body_cq(V3<R> d, R q, V3<R> e, R m, PO<R> &o) {
    R r2 = dot3(d, d);
    R r2inv, rinv;
    Math<R>::inv2(r2, r2inv, rinv);
    R costj = dot3(e, d) * rinv;
    R qQr3 = R(0.5) * q * m * rinv * r2inv;
    R upot = qQr3 * (R(3) * costj * costj - R(1));
    R mpR = R(3) * upot * r2inv;
    R pT = R(6) * costj * qQr3 * rinv;
    R fac = costj * pT * rinv + mpR;
    o.f = {fac * d.x - pT * e.x, fac * d.y - pT * e.y, fac * d.z - pT * e.z};
    o.u = upot;
    V3<R> c = cross3(d, e);
    o.M2 = {pT * c.x, pT * c.y, pT * c.z};
}

// _loopBodyDipoleQuadrupole (VectorizedCellProcessor.cpp:526-648): first
// dipole (ei, p), second quadrupole (ej, m).
template <typename R>
__device__ __forceinline__ void body_dq(V3<R> d, V3<R> ei, R p, V3<R> ej, R m, PO<R> &o) {
    R r2 = dot3(d, d);
    R r2inv, rinv;
    Math<R>::inv2(r2, r2inv, rinv);
    R myqfac = R(1.5) * p * m * r2inv * r2inv;
    R costi = dot3(ei, d) * rinv, costj = dot3(ej, d) * rinv;
    R cosgij = dot3(ei, ej);
    R c5 = R(5) * costj * costj - R(1);
    R upot = myqfac * (R(2) * costj * cosgij - costi * c5);
    R myqfacr = myqfac * rinv;
    R mpR = R(4) * upot * r2inv;
    R mpTi = myqfacr * c5;
    R mpTj = myqfacr * R(2) * (R(5) * costi * costj - cosgij);
    R pG = myqfac * R(2) * costj;
    R fac = mpR - (costi * mpTi + costj * mpTj) * rinv;
    o.f = {fac * d.x + mpTi * ei.x + mpTj * ej.x, fac * d.y + mpTi * ei.y + mpTj * ej.y,
           fac * d.z + mpTi * ei.z + mpTj * ej.z};
    o.u = upot;
    V3<R> c12 = cross3(ei, ej), eixd = cross3(ei, d), ejxd = cross3(ej, d);
    o.M1 = {mpTi * eixd.x - pG * c12.x, mpTi * eixd.y - pG * c12.y, mpTi * eixd.z - pG * c12.z};
    o.M2 = {mpTj * ejxd.x + pG * c12.x, mpTj * ejxd.y + pG * c12.y, mpTj * ejxd.z + pG * c12.z};
}

// _loopBodyQuadrupole (VectorizedCellProcessor.cpp:650-792)
template <typename R>
__device__ __forceinline__ void body_qq(V3<R> d, V3<R> ei, R mi, V3<R> ej, R mj, PO<R> &o) {
    R r2 = dot3(d, d);
    R r2inv, rinv;
    Math<R>::inv2(r2, r2inv, rinv);
    R qfac = R(0.75) * rinv * (mi * mj) * (r2inv * r2inv);
    R costi = dot3(ei, d) * rinv, costj = dot3(ej, d) * rinv;
    R c2i = costi * costi, c2j = costj * costj;
    R cosgij = dot3(ei, ej);
    R term = cosgij - R(5) * (costi * costj);
    R upot = qfac * ((R(1) + R(2) * term * term) - (R(5) * (c2i + c2j) + R(15) * c2i * c2j));
    R mpR = R(5) * upot * r2inv;
    R part1 = qfac * R(10) * rinv;
    R part2 = R(2) * term;
    R mpTi = part1 * (costi + (part2 * costj + R(3) * costi * c2j));
    R mpTj = part1 * (costj + (part2 * costi + R(3) * costj * c2i));
    R pG = qfac * R(4) * term;
    R fac = mpR - (mpTi * costi + mpTj * costj) * rinv;
    o.f = {fac * d.x + mpTi * ei.x + mpTj * ej.x, fac * d.y + mpTi * ei.y + mpTj * ej.y,
           fac * d.z + mpTi * ei.z + mpTj * ej.z};
    o.u = upot;
    V3<R> c12 = cross3(ei, ej), eixd = cross3(ei, d), ejxd = cross3(ej, d);
    o.M1 = {mpTi * eixd.x - pG * c12.x, mpTi * eixd.y - pG * c12.y, mpTi * eixd.z - pG * c12.z};
    o.M2 = {mpTj * ejxd.x + pG * c12.x, mpTj * ejxd.y + pG * c12.y, mpTj * ejxd.z + pG * c12.z};
}

// ------------------------------------------------------------- site access

// a[j] with a 32-bit byte offset (at most 2^27 sites of 16 bytes): one scalar
// base and one vector offset register instead of a 64-bit address per lane.
template <typename T> __device__ __forceinline__ const T &item(const T *a, int j) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(a) +
                                        (unsigned)j * (unsigned)sizeof(T));
}

template <typename R> struct alignas(4 * sizeof(R)) Q4 {
    R x, y, z, w;
};

// Site j of an array: site and molecule position, orientation, parameter
// (charge, moment), LJ column (four times the lookup id), and the molecule's
// charge count at its first charge site, 0 at the others.
template <typename R> struct SiteView;

template <> struct SiteView<double> {
    static __device__ __forceinline__ V3<double> pos(const SiteArrays &A, int j) {
        return {item(A.x, j), item(A.y, j), item(A.z, j)};
    }
    static __device__ __forceinline__ V3<double> mol(const SiteArrays &A, int j) {
        return {item(A.mx, j), item(A.my, j), item(A.mz, j)};
    }
    static __device__ __forceinline__ V3<double> ori(const SiteArrays &A, int j) {
        return {item(A.ex, j), item(A.ey, j), item(A.ez, j)};
    }
    static __device__ __forceinline__ double par(const SiteArrays &A, int j) { return item(A.p, j); }
    static __device__ __forceinline__ int column(const SiteArrays &A, int j) {
        return 4 * item(A.ljid, j);
    }
    static __device__ __forceinline__ int heads(const SiteArrays &A, int j) {
        return item(A.nhead, j);
    }
};

template <> struct SiteView<float> {
    static __device__ __forceinline__ V3<float> pos(const SiteArrays &A, int j) {
        const float4 v = item(A.f, j);
        return {v.x, v.y, v.z};
    }
    static __device__ __forceinline__ V3<float> mol(const SiteArrays &A, int j) {
        const float4 v = item(A.fm, j);
        return {v.x, v.y, v.z};
    }
    static __device__ __forceinline__ V3<float> ori(const SiteArrays &A, int j) {
        const float4 v = item(A.fe, j);
        return {v.x, v.y, v.z};
    }
    static __device__ __forceinline__ float par(const SiteArrays &A, int j) { return item(A.f, j).w; }
    static __device__ __forceinline__ int column(const SiteArrays &A, int j) {
        return __float_as_int(item(A.f, j).w);
    }
    static __device__ __forceinline__ int heads(const SiteArrays &A, int j) {
        return __float_as_int(item(A.fm, j).w);
    }
};

// an LJ column as the integer bits of a record's w (FP64: of its low word)
template <typename R> __device__ __forceinline__ R column_bits(int c);
template <> __device__ __forceinline__ double column_bits<double>(int c) {
    return __hiloint2double(0, c);
}
template <> __device__ __forceinline__ float column_bits<float>(int c) { return __int_as_float(c); }

// Neighbour k (0..26, dz-major) of cell (cx,cy,cz): index of the cell that
// holds the image, the FP64 shift of that image (0 or +-L) and the unwrapped
// cell offset. ok = false for open boundaries outside the domain.
struct Nbr {
    int cell;
    bool ok;
    double s[3];
    int dd[3];
};

// nxs = 4 (two cells side by side in x): x offsets -1 .. 2 from the first.
__device__ __forceinline__ Nbr neighbour(const Geom &g, int cx, int cy, int cz, int k,
                                         int nxs = 3) {
    Nbr b;
    b.dd[0] = k % nxs - 1;
    b.dd[1] = (k / nxs) % 3 - 1;
    b.dd[2] = k / (3 * nxs) - 1;
    int c3[3] = {cx + b.dd[0], cy + b.dd[1], cz + b.dd[2]};
    b.ok = true;
    for (int d = 0; d < 3; ++d) {
        b.s[d] = 0.0;
        if (c3[d] < 0) {
            if (!g.pdim[d]) b.ok = false;
            c3[d] += g.n[d];
            b.s[d] = -g.L[d];
        } else if (c3[d] >= g.n[d]) {
            if (!g.pdim[d]) b.ok = false;
            c3[d] -= g.n[d];
            b.s[d] = g.L[d];
        }
    }
    b.cell = (c3[2] * g.n[1] + c3[1]) * g.n[0] + c3[0];
    return b;
}

// x of the lane that the DPP control names; 0 where there is none and in rows
// of 16 lanes outside the row mask
template <int CTRL, int ROWS> __device__ __forceinline__ int dpp(int x) {
    return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp(double x) {
    return __hiloint2double(dpp<CTRL, ROWS>(__double2hiint(x)), dpp<CTRL, ROWS>(__double2loint(x)));
}
// inclusive prefix sums over the wave (row shifts by 1, 2, 4, 8, then the row
// ends broadcast into the next rows), without LDS round trips
template <typename X> __device__ __forceinline__ X wave_scan(X x) {
    x += dpp<0x111, 0xf>(x);
    x += dpp<0x112, 0xf>(x);
    x += dpp<0x114, 0xf>(x);
    x += dpp<0x118, 0xf>(x);
    x += dpp<0x142, 0xa>(x);
    x += dpp<0x143, 0xc>(x);
    return x;
}
// the same for the maximum of values >= 0
__device__ __forceinline__ int wave_max_scan(int x) {
    x = max(x, dpp<0x111, 0xf>(x));
    x = max(x, dpp<0x112, 0xf>(x));
    x = max(x, dpp<0x114, 0xf>(x));
    x = max(x, dpp<0x118, 0xf>(x));
    x = max(x, dpp<0x142, 0xa>(x));
    x = max(x, dpp<0x143, 0xc>(x));
    return x;
}

// LDS by 32-bit address.
__device__ __forceinline__ unsigned lds_address(const void *p) {
    return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

template <typename T> __device__ __forceinline__ T lds_value(unsigned a) {
    return *(const __attribute__((address_space(3))) T *)a;
}
template <typename R> __device__ __forceinline__ Q4<R> lds_q4(unsigned a) {
    typedef R Vec __attribute__((ext_vector_type(4)));
    const Vec q = lds_value<Vec>(a);
    return {q.x, q.y, q.z, q.w};
}

// Neighbour index of tile entry idx (concatenated neighbour order): the
// largest k < nb with pre[k] <= idx.
__device__ __forceinline__ int tile_k(const int *pre, int idx, int nb = 27) {
    int lo = 0, hi = nb;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (pre[mid] <= idx) lo = mid; else hi = mid;
    }
    return lo;
}

struct Acc {
    double f[3], v[3], m[3];
    double u, rf;
};

// i-site data held in registers for a whole pass
template <typename R> struct ISite {
    V3<R> pos, mol, e;
    R par;
    int ljrow;          // LJ id * nlj * 4: the row of the interleaved LJ table
    int idx;            // site index
};

template <int TI, int TJ> struct Kind;  // 0 LJ,1 CC,2 CD,3 DD,4 CQ,5 DQ,6 QQ
template <> struct Kind<T_LJ, T_LJ> { static constexpr int k = 0; };
template <> struct Kind<T_C, T_C> { static constexpr int k = 1; };
template <> struct Kind<T_C, T_D> { static constexpr int k = 2; };
template <> struct Kind<T_D, T_C> { static constexpr int k = 2; };
template <> struct Kind<T_D, T_D> { static constexpr int k = 3; };
template <> struct Kind<T_C, T_Q> { static constexpr int k = 4; };
template <> struct Kind<T_Q, T_C> { static constexpr int k = 4; };
template <> struct Kind<T_D, T_Q> { static constexpr int k = 5; };
template <> struct Kind<T_Q, T_D> { static constexpr int k = 5; };
template <> struct Kind<T_Q, T_Q> { static constexpr int k = 6; };

// FP32 form: most pair terms a lane of a block kernel sums in FP32 before they
// go to its FP64 accumulators (a cell kernel's lane: one drained hit list).
// Charges: the lane meets a molecule's charges in turn with other molecules' (a
// cell kernel's lane sums whole, neutral molecules), and the unbalanced partial
// sums round more, so each term goes to FP64 (250 rigid water molecules, rc 12:
// force error 5.3e-6 -> 4.8e-6, as the cell kernel's; +1.8 us at 9001
// molecules of the mixture)
constexpr int kPart = 24, kPartCharge = 1;
// LJ parameters of a pair: one LJ id (scalar registers), a table in LDS (at
// most kTableIds ids), a table in global memory
enum { kTableNone = 0, kTableLds = 1, kTableGlobal = 2 };
constexpr int kTableIds = 8;

template <typename R> __device__ __forceinline__ V3<R> v3(const Q4<R> &q) { return {q.x, q.y, q.z}; }

// FP32 form: partial sums of a few pair terms, added to the FP64
// accumulators by flush().
struct Part32 {
    float f[3], v[3], m[3], u, rf;
    __device__ __forceinline__ void clear() {
        for (int k = 0; k < 3; ++k) f[k] = v[k] = m[k] = 0.f;
        u = rf = 0.f;
    }
    __device__ __forceinline__ void flush(Acc &a) const {
        for (int k = 0; k < 3; ++k) {
            a.f[k] += (double)f[k];
            a.v[k] += (double)v[k];
            a.m[k] += (double)m[k];
        }
        a.u += (double)u;
        a.rf += (double)rf;
    }
};

// LJ pair seen from site i, evaluated on every lane of the wave: a lane whose
// entry is not accepted (ok false) runs the body at a huge r^2 (FP32: +inf;
// FP64: 1e300, which keeps the Newton steps of 1/r^2 finite), where force and
// virial come out exactly 0, and adds no energy; u = 6 U_LJ + shift6
// (_loopBodyLJ, VectorizedCellProcessor.cpp:171-224). FP64 form: into acc;
// FP32 form: into the FP32 partial sums pa. tab, par: the interleaved
// parameter table in LDS (few LJ ids) or in global memory.
template <typename R, bool MOLSITE, int MULTI>
__device__ __forceinline__ void eval_lj(const Q4<R> *tab, const R *par, const ISite<R> &I,
                                        const Q4<R> &pj, const Q4<R> &mj, bool ok, R eps24, R sig2,
                                        R shift6, Acc &acc, Part32 &pa) {
    const V3<R> d = {I.pos.x - pj.x, I.pos.y - pj.y, I.pos.z - pj.z};
    V3<R> dm = d;
    if constexpr (!MOLSITE) dm = {I.mol.x - mj.x, I.mol.y - mj.y, I.mol.z - mj.z};
    if constexpr (MULTI != kTableNone) {
        // pj.w carries the partner's column offset (4 * its LJ id) as integer
        // bits in the low word
        int col;
        if constexpr (sizeof(R) == 8)
            col = __double2loint(pj.w);
        else
            col = __float_as_int(pj.w);
        const unsigned at = (unsigned)(I.ljrow + col);
        if constexpr (MULTI == kTableLds) {
            const Q4<R> &t = tab[at >> 2];
            eps24 = t.x;
            sig2 = t.y;
            shift6 = t.z;
        } else if constexpr (sizeof(R) == 8) {
            const double *t = par + at;
            const double2 es = *reinterpret_cast<const double2 *>(t);
            eps24 = es.x;
            sig2 = es.y;
            shift6 = t[2];
        } else {
            const float4 t = *reinterpret_cast<const float4 *>(par + at);
            eps24 = t.x;
            sig2 = t.y;
            shift6 = t.z;
        }
    }
    const R far = sizeof(R) == 4 ? R(__builtin_inff()) : R(1e300);
    const R r2inv = Math<R>::rcp(ok ? dot3(d, d) : far);
    const R lj2 = sig2 * r2inv, lj6 = lj2 * lj2 * lj2, lj12 = lj6 * lj6;
    const R lj12m6 = lj12 - lj6;
    const R s = eps24 * r2inv * (lj12 + lj12m6);
    const R fx = d.x * s, fy = d.y * s, fz = d.z * s;
    const R u = ok ? eps24 * lj12m6 + shift6 : R(0);
    if constexpr (sizeof(R) == 4) {
        pa.f[0] += fx;
        pa.f[1] += fy;
        pa.f[2] += fz;
        pa.v[0] += dm.x * fx;
        pa.v[1] += dm.y * fy;
        pa.v[2] += dm.z * fz;
        pa.u += u;
    } else {
        acc.f[0] += fx;
        acc.f[1] += fy;
        acc.f[2] += fz;
        acc.v[0] += dm.x * fx;
        acc.v[1] += dm.y * fy;
        acc.v[2] += dm.z * fz;
        acc.u += u;
    }
}

// One electrostatic site pair seen from site i: force on i, virial
// (m_i - m_j) * f_i, torque on i; roles swapped where the reference swaps.
// pj, mj, ej: the partner's site, molecule and orientation records (the
// caller reads them from its pass's tile records; ej only for dipole and
// quadrupole partners).
template <int TI, int TJ, typename R, bool MOLSITE>
__device__ __forceinline__ void eval_pair(R epsRFInvrc3, const ISite<R> &I, const Q4<R> &eq,
                                          const Q4<R> &pj, const Q4<R> &mj,
                                          Acc &acc, Part32 &pa) {
    V3<R> d = {I.pos.x - pj.x, I.pos.y - pj.y, I.pos.z - pj.z};
    V3<R> dm = d;
    if constexpr (!MOLSITE) dm = {I.mol.x - mj.x, I.mol.y - mj.y, I.mol.z - mj.z};
    PO<R> o;
    o.rf = R(0);
    R sign = R(1);
    V3<R> tq = {R(0), R(0), R(0)};
    static_assert(TI != T_LJ, "LJ pairs go through eval_lj");
    V3<R> ej = {R(0), R(0), R(0)};
    if constexpr (TJ >= T_D) ej = v3(eq);
    const R qj = pj.w;
    if constexpr (TI == T_C && TJ == T_C) {
        body_cc<R>(d, I.par, qj, o);
    } else if constexpr (TI == T_C && TJ == T_D) {
        body_cd<R>(d, I.par, ej, qj, o);
    } else if constexpr (TI == T_C && TJ == T_Q) {
        body_cq<R>(d, I.par, ej, qj, o);
    } else if constexpr (TI == T_D && TJ == T_C) {
        V3<R> nd = {-d.x, -d.y, -d.z};
        body_cd<R>(nd, qj, I.e, I.par, o);
        sign = R(-1);
        tq = o.M2;
    } else if constexpr (TI == T_D && TJ == T_D) {
        body_dd<R>(d, I.e, I.par, ej, qj, epsRFInvrc3, o);
        tq = o.M1;
    } else if constexpr (TI == T_D && TJ == T_Q) {
        body_dq<R>(d, I.e, I.par, ej, qj, o);
        tq = o.M1;
    } else if constexpr (TI == T_Q && TJ == T_C) {
        V3<R> nd = {-d.x, -d.y, -d.z};
        body_cq<R>(nd, qj, I.e, I.par, o);
        sign = R(-1);
        tq = o.M2;
    } else if constexpr (TI == T_Q && TJ == T_D) {
        V3<R> nd = {-d.x, -d.y, -d.z};
        body_dq<R>(nd, ej, qj, I.e, I.par, o);
        sign = R(-1);
        tq = o.M2;
    } else if constexpr (TI == T_Q && TJ == T_Q) {
        body_qq<R>(d, I.e, I.par, ej, qj, o);
        tq = o.M1;
    }
    V3<R> f = {sign * o.f.x, sign * o.f.y, sign * o.f.z};
    if constexpr (sizeof(R) == 4) {
        pa.f[0] += f.x;
        pa.f[1] += f.y;
        pa.f[2] += f.z;
        pa.v[0] += dm.x * f.x;
        pa.v[1] += dm.y * f.y;
        pa.v[2] += dm.z * f.z;
        pa.u += o.u;
        if constexpr (TI == T_D && TJ == T_D) pa.rf += o.rf;
        if constexpr (TI >= T_D) {
            pa.m[0] += tq.x;
            pa.m[1] += tq.y;
            pa.m[2] += tq.z;
        }
    } else {
        acc.f[0] += f.x;
        acc.f[1] += f.y;
        acc.f[2] += f.z;
        acc.v[0] += dm.x * f.x;
        acc.v[1] += dm.y * f.y;
        acc.v[2] += dm.z * f.z;
        acc.u += o.u;
        if constexpr (TI == T_D && TJ == T_D) acc.rf += o.rf;
        if constexpr (TI >= T_D) {
            acc.m[0] += tq.x;
            acc.m[1] += tq.y;
            acc.m[2] += tq.z;
        }
    }
}

}  // namespace mdx
