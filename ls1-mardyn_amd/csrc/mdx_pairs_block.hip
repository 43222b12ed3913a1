// mdx_pairs_block.hip -- pair kernels of small boxes (gfx950, wave64).
//
// The same site pairs, frames, cutoff rules and sums as the cell kernels of
// mdx_pairs.hip, split differently: a block of four waves takes one cell, whose
// sites the waves share, and stages the sites of its 27 neighbour images in
// LDS once for all four. A wave tests one molecule of its quarter against 64
// candidates at a time (the molecule's centre in scalar registers, the
// candidates' in vector registers), so the centre tests of a molecule are made
// once for all its sites, and appends the hits to one list per molecule; the
// sites then share the list's entries among their lanes evenly. The cell
// kernels test per site and leave a lane the hits of its own candidates.
//
// A small box alone is bound by latency (a few hundred cells leave most of the 1024
// SIMDs one wave or none, and a cell kernel's wave walks its whole
// neighbourhood alone): four waves per cell and lists shared evenly cut that
// chain. Time of all pair kernels, cell -> block: 9001 molecules of the 2CLJQ + water
// mixture (512 cells), FP32: 310 -> 75, FP64: 376 -> 93. A full chip is bound by VALU
// issue instead, and there the cell kernels win unless the cells are dense (the
// rule and both sides' figures stand with kSmallSites in mdx_capi.hip).
#include "mdx_pair_common.h"

namespace mdx {

constexpr int kPairWaves = kPairBlock / 64;  // waves per block of the pair kernels
constexpr int kTileCells = 27;  // a cell and its neighbours
template <int TI, typename R, bool MOLSITE, int MULTI> struct BlockCfg {
    static constexpr bool MOL = !MOLSITE;    // molecule positions differ from sites
    static constexpr bool LJID = TI == T_LJ && MULTI != kTableNone;  // several LJ centre types
    static constexpr bool F32 = sizeof(R) == 4;
    // Tile bytes, list entries per wave and rows of 64 candidates a wave keeps
    // in registers. The register bound is WAVES waves per SIMD, and the LDS of a
    // block (BlockShared) lets as many blocks of four waves share a CU; the FP64
    // kernels with molecule records fit three waves (at four they spill: 842 ->
    // 1017 us on a full chip).
    static constexpr int RAW = MOLSITE ? (F32 ? 10752 : 21504) : 32768;
    static constexpr int LCAP = MOLSITE ? 1280 : 768;
    // i sites per pass (the list entries hold a row of 64 hits for each): 12
    // sites have 5 phases, 60 of the 64 lanes
    static constexpr int SPP = MOLSITE ? 16 : 12;
    static constexpr int RG = F32 ? 5 : 4;
    static constexpr int WAVES = F32 || MOLSITE ? 4 : 3;
};

template <int TI, typename R, bool MOLSITE, int MULTI> struct BlockShared {
    using C = BlockCfg<TI, R, MOLSITE, MULTI>;
    alignas(32) unsigned char raw[C::RAW];            // staged sites (BlockTile)
    alignas(16) unsigned short lst[kPairWaves][C::LCAP];  // hit lists per wave (tile indices)
    int j0[kTileCells], pre[kTileCells], code[kTileCells];
    unsigned short zero;  // 0: the list entry of a lane without a list
    double mac[kPairWaves][3];
    Q4<R> tab[MULTI == kTableLds ? kTableIds * kTableIds : 1];
};
// blocks of LDS size `bytes` (given out in steps of 1280) that share a CU
constexpr int blocks_per_cu(size_t bytes) { return (int)(160 * 1024 / ((bytes + 1279) / 1280 * 1280)); }

// The records of one partner pass (partner type TJ) in a tile's bytes: p site
// position (w = charge / moment or LJ table column), m molecule position, e
// orientation (dipole and quadrupole partners). A pass lays out only the
// records its partner type needs.
template <int TI, int TJ, typename R, bool MOLSITE, int MULTI> struct BlockTile {
    using C = BlockCfg<TI, R, MOLSITE, MULTI>;
    static constexpr bool ORIJ = TI != T_LJ && TJ >= T_D;
    static constexpr int REC = (int)sizeof(R) * (4 + 3 * C::MOL + 3 * ORIJ);
    static constexpr int CAP = C::RAW / REC / 16 * 16;
    static_assert(CAP >= 64 && 4 * CAP < 65536, "tile capacity, 4 * index in 16 bits");
    Q4<R> *p;
    R *mx, *my, *mz, *ex, *ey, *ez;
    __device__ __forceinline__ explicit BlockTile(unsigned char *raw) {
        p = reinterpret_cast<Q4<R> *>(raw);
        mx = reinterpret_cast<R *>(p + CAP);
        my = mx + CAP;
        mz = my + CAP;
        ex = mx + (C::MOL ? 3 * CAP : 0);
        ey = ex + CAP;
        ez = ey + CAP;
    }
};

// Order for a wave's own LDS traffic (list writes before list reads and the
// other way round): the hardware runs one wave's LDS operations in order, the
// fence keeps the compiler from moving them.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The kernel's arguments (its only parameter, at the start of the argument
// segment) behind an address the compiler cannot see through: their pointers
// are loaded again where they are used instead of held in scalar registers
// across the cell and pass loops (which spilled up to 200 of them).
__device__ __forceinline__ const PairArgs &args() {
    typedef const __attribute__((address_space(4))) PairArgs *Ptr;
    Ptr p = (Ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const PairArgs *)p;
}

// Memory no kernel of the launch writes, read through the constant address
// space: loads at wave-uniform addresses become scalar loads.
template <typename T> __device__ __forceinline__ const T &constant(const T *p) {
    return *(const T *)(const __attribute__((address_space(4))) T *)p;
}
template <typename T> __device__ __forceinline__ const T &constant(const T *p, int i) {
    return constant(p + __builtin_amdgcn_readfirstlane(i));
}

__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ int lane_value(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// Site position with its charge, moment or (several LJ ids) table column in w.
template <int TI, typename R, bool LJID>
__device__ __forceinline__ Q4<R> site_record(const SiteArrays &S, int j) {
    const V3<R> p = SiteView<R>::pos(S, j);
    R w = R(0);
    if constexpr (LJID) w = column_bits<R>(SiteView<R>::column(S, j));
    if constexpr (TI != T_LJ) w = SiteView<R>::par(S, j);
    return {p.x, p.y, p.z, w};
}

// A block's cell and one wave's share of it (all wave-uniform).
struct Cell {
    const Geom *g;        // (constant address space)
    int cbase;            // first global cell of the replica
    int cx, cy, cz;
    int ib, ie;           // the wave's i sites
};

// Tile cell of a lane (lane < 27, in the order of neighbour()): the cell that
// holds the image, and a code with the position in the tile (bits 0-1 x, 2-3 y,
// 4-5 z) and the image shift per dimension (bits 6, 8, 10: 0 none, 1 minus the
// box length, 2 plus it).
struct TileCell {
    int cell, code;
    bool ok;
};

__device__ __forceinline__ TileCell tile_cell(const Cell &G, int k) {
    const Geom &g = *G.g;
    const int q = k / 3, t[3] = {k - 3 * q, q % 3, q / 3};
    const int c0[3] = {G.cx, G.cy, G.cz};
    TileCell r;
    r.code = t[0] | t[1] << 2 | t[2] << 4;
    r.ok = k < kTileCells;
    int c[3];
    for (int d = 0; d < 3; ++d) {
        c[d] = c0[d] + t[d] - 1;
        if (c[d] < 0) {
            r.ok = r.ok && g.pdim[d];
            c[d] += g.n[d];
            r.code |= 1 << (6 + 2 * d);
        } else if (c[d] >= g.n[d]) {
            r.ok = r.ok && g.pdim[d];
            c[d] -= g.n[d];
            r.code |= 2 << (6 + 2 * d);
        }
    }
    r.cell = (c[2] * g.n[1] + c[1]) * g.n[0] + c[0];
    return r;
}

// Image shift of a tile cell code (FP64 absolute positions).
__device__ __forceinline__ double code_shift(const Geom &g, int code, int d) {
    const int s = code >> (6 + 2 * d) & 3;
    const double L = g.L[d];  // loaded in any case: no branch around it
    return s == 0 ? 0.0 : s == 1 ? -L : L;
}

// What is added to a staged site's stored position. FP64: the image shift.
// FP32: the offset between the corners of its cell and the block's cell, as in
// the cell kernels (the same bits per pair).
template <typename R>
__device__ __forceinline__ V3<R> tile_offset(const Cell &G, int code);
template <>
__device__ __forceinline__ V3<double> tile_offset<double>(const Cell &G, int code) {
    const Geom &g = *G.g;
    return {code_shift(g, code, 0), code_shift(g, code, 1), code_shift(g, code, 2)};
}
template <>
__device__ __forceinline__ V3<float> tile_offset<float>(const Cell &G, int code) {
    const Geom &g = *G.g;
    return {(float)(((code & 3) - 1) * g.cl[0]), (float)(((code >> 2 & 3) - 1) * g.cl[1]),
            (float)(((code >> 4 & 3) - 1) * g.cl[2])};
}

// The lane's i site and its place in the wave's pass.
template <typename R> struct Pass {
    ISite<R> I;
    int first;                 // first i site of the pass
    int nI, P;                 // sites of the pass, phases (lanes) per site
    int ph;                    // the lane's phase
    bool valid;                // the lane has a site
    unsigned long long heads;  // lanes 0 .. nI - 1 that hold the first site of a molecule
    int hl, ord;               // head lane and ordinal of the lane's molecule
    int LS;                    // list entries per molecule
};

// All pairs of the wave's i sites with the j sites of type TJ around them.
// (1) The block stages the sites of the 27 tile cells in LDS (16 lanes per
// cell, in chunks of at most CAP sites); (2) stage A, per molecule of the
// wave's share: its centre goes to scalar registers and RG rows of 64
// candidates are tested at once, the hits of a row are appended to the
// molecule's list in LDS (ballot + mbcnt positions); (3) stage B: the P lanes
// of each site walk its molecule's list with stride P and evaluate the site
// pairs.
template <int TI, int TJ, typename R, bool MOLSITE, int MULTI, bool COUNT>
__device__ __forceinline__ void partner_pass(const Cell &G, const Pass<R> &S,
                                             const TileCell &tc, int lane, int wv, bool staged,
                                             BlockShared<TI, R, MOLSITE, MULTI> &T, Acc &acc,
                                             R eps24, R sig2, R shift6,
                                             unsigned long long &ntest) {
    using C = BlockCfg<TI, R, MOLSITE, MULTI>;
    using PT = BlockTile<TI, TJ, R, MOLSITE, MULTI>;
    const PairArgs &a = args();
    const Geom &g = *G.g;
    const PT V(T.raw);
    const double rc2 = (TI == T_LJ) ? a.rclj2 : a.rc2;
    unsigned long long nhit = 0;
    // tile cell ranges: one per lane, the prefix by a wave scan (every wave
    // has them all, so no barrier before the staging)
    int j0 = 0, nk = 0;
    if (tc.ok) {
        const int *cstart = a.s[TJ].cstart + G.cbase;
        j0 = cstart[tc.cell];
        nk = cstart[tc.cell + 1] - j0;
    }
    const int incl = wave_scan(nk);
    const int pre = incl - nk;
    const int total = lane_value(incl, 63);
    // equal chunks of at most CAP sites (one in most cases)
    int per = total;
    if (total > PT::CAP) {
        const int chunks = (total + PT::CAP - 1) / PT::CAP;
        per = (total + chunks - 1) / chunks;
    }
    for (int base = 0; base < total; base += per) {
        const int top = min(base + per, total);
        if (!(TI == T_LJ && staged && per == total)) {
            if (base > 0 || staged) __syncthreads();  // the tile is no longer read
            const SiteArrays J = args().s[TJ];
            if (wv == 0 && lane < kTileCells) {  // for the FP64 re-check
                T.j0[lane] = j0;
                T.pre[lane] = pre;
                T.code[lane] = tc.code;
            }
            // 16 lanes per tile cell; a lane's two cells go together, so their
            // loads are in flight at once
            constexpr int NC = (kTileCells + 15) / 16;
            int kj[NC], kn[NC], kp[NC];
            V3<R> off[NC];
            V3<R> own;
            if constexpr (sizeof(R) == 4) own = tile_offset<R>(G, tc.code);
            int most = 0;
#pragma unroll
            for (int r = 0; r < NC; ++r) {
                const int k = wv * 4 + (lane >> 4) + 16 * r;  // (27 .. 31: no sites)
                kj[r] = __shfl(j0, k, 64);
                kn[r] = __shfl(nk, k, 64);
                kp[r] = __shfl(pre, k, 64) - base;
                if constexpr (sizeof(R) == 4)  // one lane computes, 16 take it
                    off[r] = {__shfl(own.x, k, 64), __shfl(own.y, k, 64), __shfl(own.z, k, 64)};
                else
                    off[r] = tile_offset<R>(G, __shfl(tc.code, k, 64));
                most = max(most, kn[r]);
            }
            for (int s = lane & 15; __any(s < most); s += 16) {
                Q4<R> p[NC];
                V3<R> m[NC], e[NC];
                bool in[NC];
#pragma unroll
                for (int r = 0; r < NC; ++r) {
                    const int at = kp[r] + s;
                    in[r] = s < kn[r] && at >= 0 && at < per;
                    const int j = in[r] ? kj[r] + s : 0;
                    p[r] = site_record<TI, R, C::LJID>(J, j);
                    if constexpr (C::MOL) m[r] = SiteView<R>::mol(J, j);
                    if constexpr (PT::ORIJ) e[r] = SiteView<R>::ori(J, j);
                }
#pragma unroll
                for (int r = 0; r < NC; ++r) {
                    const int at = kp[r] + s;
                    if (!in[r]) continue;
                    V.p[at] = Q4<R>{p[r].x + off[r].x, p[r].y + off[r].y, p[r].z + off[r].z, p[r].w};
                    if constexpr (C::MOL) {
                        V.mx[at] = m[r].x + off[r].x;
                        V.my[at] = m[r].y + off[r].y;
                        V.mz[at] = m[r].z + off[r].z;
                    }
                    if constexpr (PT::ORIJ) {
                        V.ex[at] = e[r].x;
                        V.ey[at] = e[r].y;
                        V.ez[at] = e[r].z;
                    }
                }
            }
            __syncthreads();
        }
        if (S.nI == 0) continue;
        const int len = top - base;
        unsigned short *lst = T.lst[wv];
        int vcnt = 0;   // lane h: entries in the list of the molecule with head lane h
        int maxc = 0;   // the longest list
        const R *par = nullptr;
        if constexpr (MULTI == kTableGlobal) {
            if constexpr (sizeof(R) == 8)
                par = args().pp.dpar;
            else
                par = args().pp.fpar;
        }
        const R epsRF = TI == T_D && TJ == T_D ? (R)args().epsRFInvrc3 : R(0);
        auto drain = [&]() {
            wave_fence();
            const int hc = __shfl(vcnt, S.hl, 64), myc = S.valid ? hc : 0;
            // (a lane without entries reads tile index 0, always staged)
            const unsigned short *L = myc > 0 ? lst + S.ord * S.LS : &T.zero;
            // the lane's entries (4 times a tile index) from LDS address `at`
            // on with stride P, the last one again behind the list's end
            const unsigned step = 2 * S.P, last = lds_address(L) + 2 * max(myc - 1, 0);
            unsigned at = lds_address(L) + 2 * S.ph;
            auto entry = [&](unsigned a) { return (int)lds_value<unsigned short>(min(a, last)); };
            auto site = [&](int s4) {
                return lds_q4<R>(lds_address(V.p) + s4 * (int)sizeof(R));
            };
            auto mol = [&](int s4, const Q4<R> &pj) {
                if constexpr (C::MOL) {
                    const unsigned b = lds_address(V.mx) + s4 * (int)(sizeof(R) / 4);
                    constexpr unsigned D = PT::CAP * sizeof(R);
                    return Q4<R>{lds_value<R>(b), lds_value<R>(b + D), lds_value<R>(b + 2 * D), R(0)};
                } else {
                    return pj;
                }
            };
            // entry at + 2 step is read while the pair of entry `at` is
            // computed, and the next entry's records, so their latency overlaps
            // the pair; entry `at` exists while at <= last
            int left = maxc;
            int s0 = entry(at), s1 = entry(at + step);
            if (myc == 0) at = last + 1;
            Q4<R> pn = site(s0), mn = mol(s0, pn);
            while (left > 0) {
                // FP32 form: partial sums of at most kPart (kPartCharge) entries
                Part32 pa;
                pa.clear();
                const int stop = sizeof(R) == 4 ? max(left - (TI == T_C ? kPartCharge : kPart) * S.P, 0) : 0;
                for (; left > stop; left -= S.P, at += step) {
                    const Q4<R> pj = pn, mj = mn;
                    const int sj = s0 >> 2;
                    s0 = s1;
                    pn = site(s0);
                    mn = mol(s0, pn);
                    s1 = entry(at + 2 * step);
                    bool ok = at <= last;
                    if constexpr (sizeof(R) == 4) {
                        // the molecule itself (and one at the very same place,
                        // SingleCellPolicy_) is left out; stage A of the FP64
                        // form does it
                        const V3<R> mi = C::MOL ? S.I.mol : S.I.pos;
                        const int bits = __float_as_int(mi.x - mj.x) | __float_as_int(mi.y - mj.y) |
                                         __float_as_int(mi.z - mj.z);
                        ok = ok && bits != 0;
                    }
                    if constexpr (TI == T_LJ) {
                        eval_lj<R, MOLSITE, MULTI>(T.tab, par, S.I, pj, mj, ok, eps24, sig2, shift6,
                                                   acc, pa);
                        if (COUNT) nhit += ok;
                    } else if (ok) {
                        Q4<R> eq{};
                        if constexpr (PT::ORIJ) eq = Q4<R>{V.ex[sj], V.ey[sj], V.ez[sj], R(0)};
                        eval_pair<TI, TJ, R, MOLSITE>(epsRF, S.I, eq, pj, mj, acc, pa);
                        if (COUNT) ++nhit;
                    }
                }
                if constexpr (sizeof(R) == 4) pa.flush(acc);
            }
            vcnt = 0;
            maxc = 0;
            wave_fence();
        };
        // FP32 form: r^2 = |i|^2 + |j|^2 - 2 i.j, three FMAs per candidate; its
        // rounding stays below 1.5e-5 (cl / rc)^2 rc^2 (coordinates within two
        // cell edges of the cell's corner), and every
        // candidate that close to rc^2 is decided in FP64 from the unrounded
        // positions, so the pair set equals the FP64 one
        R nx, ny, nz, hi, lo;
        {
            const V3<R> mi = C::MOL ? S.I.mol : S.I.pos;
            nx = mi.x;
            ny = mi.y;
            nz = mi.z;
            hi = lo = (R)rc2;
            if constexpr (sizeof(R) == 4) {
                const float rcf = (float)rc2,
                            clm = fmaxf((float)g.cl[0], fmaxf((float)g.cl[1], (float)g.cl[2]));
                const float band = fmaxf(1e-5f * rcf, 1.6e-5f * clm * clm);
                const R i2 = mi.x * mi.x + mi.y * mi.y + mi.z * mi.z;
                hi = (rcf + band) - i2;
                lo = (rcf - band) - i2;
                nx = R(-2) * mi.x;
                ny = R(-2) * mi.y;
                nz = R(-2) * mi.z;
                // (kept in registers: else the factors are multiplied again
                // for every molecule of the loop below)
                asm("" : "+v"(nx), "+v"(ny), "+v"(nz));
            }
        }
        for (int row0 = 0; row0 < len; row0 += 64 * C::RG) {
            V3<R> jm[C::RG];
            R jw[C::RG];
            int jid[C::RG];
#pragma unroll
            for (int r = 0; r < C::RG; ++r) {
                const int t = row0 + 64 * r + lane;
                const int s = t < len ? t : 0;
                jid[r] = 4 * s;
                if constexpr (C::MOL)
                    jm[r] = {V.mx[s], V.my[s], V.mz[s]};
                else
                    jm[r] = {V.p[s].x, V.p[s].y, V.p[s].z};
                if (t >= len) jm[r].x = R(sizeof(R) == 4 ? 1e30 : 1e150);  // no candidate
                jw[r] = R(0);
                if constexpr (sizeof(R) == 4)
                    jw[r] = jm[r].x * jm[r].x + jm[r].y * jm[r].y + jm[r].z * jm[r].z;
            }
            unsigned lb = lds_address(lst);  // LDS address of the molecule's list
            for (unsigned long long hm = S.heads; hm; hm &= hm - 1, lb += 2 * S.LS) {
                const int h = __ffsll((long long)hm) - 1;
                const R ix = lane_value(nx, h), iy = lane_value(ny, h), iz = lane_value(nz, h);
                int cnt = lane_value(vcnt, h);
                if (COUNT && lane == 0) ntest += min(64 * C::RG, len - row0);
                unsigned long long m[C::RG];
                if constexpr (sizeof(R) == 4) {
                    const R ihi = lane_value(hi, h), ilo = lane_value(lo, h);
                    unsigned long long near = 0;
#pragma unroll
                    for (int r = 0; r < C::RG; ++r) {
                        const R d = __builtin_fmaf(
                            ix, jm[r].x, __builtin_fmaf(iy, jm[r].y, __builtin_fmaf(iz, jm[r].z, jw[r])));
                        m[r] = __ballot(d <= ihi);
                        near |= m[r] ^ __ballot(d < ilo);
                        asm("" : "+s"(near));  // two scalar operations per row
                    }
                    if (near) {  // some candidate lies in the band around rc^2
#pragma unroll 1
                        for (int r = 0; r < C::RG; ++r) {
                            unsigned long long mr = m[0];
                            int s = jid[0];
                            R x = jm[0].x, y = jm[0].y, z = jm[0].z, w = jw[0];
#pragma unroll
                            for (int q = 1; q < C::RG; ++q)
                                if (r == q) {
                                    mr = m[q];
                                    s = jid[q];
                                    x = jm[q].x, y = jm[q].y, z = jm[q].z, w = jw[q];
                                }
                            const R d = __builtin_fmaf(
                                ix, x, __builtin_fmaf(iy, y, __builtin_fmaf(iz, z, w)));
                            bool hit = __builtin_amdgcn_inverse_ballot_w64(mr);
                            if (hit && !(d < ilo)) {
                                const PairArgs &b = args();
                                const int idx = base + (s >> 2);
                                const int k = tile_k(T.pre, idx, kTileCells);
                                const int j = T.j0[k] + (idx - T.pre[k]), code = T.code[k];
                                const int mi = b.s[TI].mol[S.first + h], mj = b.s[TJ].mol[j];
                                const double ex = b.mrx[mi] - (b.mrx[mj] + code_shift(g, code, 0));
                                const double ey = b.mry[mi] - (b.mry[mj] + code_shift(g, code, 1));
                                const double ez = b.mrz[mi] - (b.mrz[mj] + code_shift(g, code, 2));
                                hit = ex * ex + ey * ey + ez * ez < rc2;
                            }
                            mr = __ballot(hit);
#pragma unroll
                            for (int q = 0; q < C::RG; ++q)
                                if (r == q) m[q] = mr;
                        }
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < C::RG; ++r) {
                        const R dx = ix - jm[r].x, dy = iy - jm[r].y, dz = iz - jm[r].z;
                        const R r2 = dx * dx + dy * dy + dz * dz;
                        m[r] = __ballot(r2 < R(rc2) && r2 != R(0));
                    }
                }
                auto append = [&](int r, int pop) {
                    const unsigned at = __builtin_amdgcn_mbcnt_hi(
                        (unsigned)(m[r] >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m[r], 0u));
                    unsigned end = lb + 2 * cnt;
                    asm("" : "+s"(end));  // scalar: one vector operation for the address
                    // the row's hits store their entry behind the list's end
                    if (__builtin_amdgcn_inverse_ballot_w64(m[r]))
                        *(__attribute__((address_space(3))) unsigned short *)((at << 1) + end) = (unsigned short)jid[r];
                    cnt += pop;
                };
                int tot = 0, pop[C::RG];
#pragma unroll
                for (int r = 0; r < C::RG; ++r) tot += pop[r] = __popcll(m[r]);
                if (cnt + tot <= S.LS) {
#pragma unroll
                    for (int r = 0; r < C::RG; ++r) append(r, pop[r]);
                } else {  // the list fills up: evaluate what is listed in between
                    for (bool more = true; more;) {
                        more = false;
#pragma unroll
                        for (int r = 0; r < C::RG; ++r)
                            if (!more && m[r] != 0) {
                                if (cnt + pop[r] <= S.LS) {
                                    append(r, pop[r]);
                                    m[r] = 0;
                                } else {
                                    more = true;
                                }
                            }
                        if (more) {
                            vcnt = lane == h ? cnt : vcnt;
                            maxc = max(maxc, cnt);
                            drain();
                            cnt = 0;
                        }
                    }
                }
                vcnt = lane == h ? cnt : vcnt;
                maxc = max(maxc, cnt);
            }
        }
        if (maxc > 0) drain();
    }
    if (COUNT) {
        const PairArgs &b = args();
        for (int o = 32; o > 0; o >>= 1) nhit += __shfl_xor(nhit, o, 64);
        if (lane == 0) atomicAdd(&b.counters[8 * TI + 1 + Kind<TI, TJ>::k], nhit);
    }
}

// The wave's pass from site `first` (of at most SPP sites; nI = 0: none left),
// and the lane's site in it.
template <int TI, typename R, bool MOLSITE, int MULTI>
__device__ __forceinline__ Pass<R> load_pass(const Cell &G, int first, int lane) {
    using C = BlockCfg<TI, R, MOLSITE, MULTI>;
    static_assert(C::SPP <= 64 && C::LCAP / C::SPP >= 64, "list room for a row of hits");
    const SiteArrays S = args().s[TI];
    Pass<R> s;
    s.first = first;
    s.nI = max(min(C::SPP, G.ie - first), 0);
    s.heads = 0;
    s.P = 1;
    s.ph = s.hl = s.ord = 0;
    s.valid = false;
    s.LS = C::LCAP;
    if (s.nI == 0) return s;
    // sites at their molecule's centre have a list each, others one per molecule
    s.heads = ~0ull >> (64 - s.nI);
    if constexpr (!MOLSITE) {
        const int mol = lane < s.nI ? item(S.mol, first + lane) : -1;
        const int prev = __shfl_up(mol, 1, 64);
        s.heads = __ballot(lane < s.nI && (lane == 0 || prev != mol));
    }
    // lane = ph * nI + il: P lanes per site, the 64 - P nI lanes left over
    // idle. LJ kernels cap P at 8 (their sparse cells have few candidates and
    // more phases only lengthen the fold), electrostatic ones at 16
    const float rn = __builtin_amdgcn_rcpf((float)s.nI);
    const int most = __builtin_amdgcn_readfirstlane((int)(64.5f * rn));  // 64 / nI (exact, as below)
    s.P = min(most, TI == T_LJ ? 8 : 16);
    s.LS = __builtin_amdgcn_readfirstlane(
        (int)(((float)C::LCAP + 0.5f) * __builtin_amdgcn_rcpf((float)__popcll(s.heads))));
    // lane / nI through a float reciprocal (exact: lane < 64, nI <= 64, and
    // (lane + 0.5) / nI stays >= 1/128 away from an integer)
    const int ph0 = (int)(((float)lane + 0.5f) * rn);
    s.valid = ph0 < s.P;
    s.ph = s.valid ? ph0 : 0;
    const int il = s.valid ? lane - ph0 * s.nI : 0;
    const unsigned long long upto = s.heads & ((2ull << il) - 1ull);
    s.hl = 63 - __clzll((long long)upto);
    s.ord = __popcll(upto) - 1;
    const int i = first + il;
    ISite<R> &I = s.I;
    const Q4<R> p = site_record<TI, R, C::LJID>(S, i);
    I.pos = v3(p);
    I.mol = MOLSITE ? I.pos : SiteView<R>::mol(S, i);
    I.idx = i;
    if constexpr (TI >= T_D) I.e = SiteView<R>::ori(S, i);
    if constexpr (C::LJID) I.ljrow = SiteView<R>::column(S, i) * args().pp.nlj;
    if constexpr (TI != T_LJ) I.par = p.w;
    return s;
}

// The phases of each site of the pass into its phase-0 lane, in phase order,
// through the wave's list buffer.
template <int TI>
__device__ __forceinline__ void fold_phases(double *fb, int nI, int P, bool own, int lane, Acc &acc) {
    auto fold3 = [&](double (&v)[3]) {
        wave_fence();
        for (int k = 0; k < 3; ++k) fb[k * 64 + lane] = v[k];
        wave_fence();
        if (own)
            for (int q = 1; q < P; ++q)
                for (int k = 0; k < 3; ++k) v[k] += fb[k * 64 + lane + q * nI];
    };
    fold3(acc.f);
    fold3(acc.v);
    if constexpr (TI >= T_D) fold3(acc.m);
    wave_fence();
}

// All i sites of one cell.
template <int TI, typename R, bool COUNT, bool MOLSITE, int MULTI>
__device__ __forceinline__ void pair_cell(BlockShared<TI, R, MOLSITE, MULTI> &T, int cell, int lane,
                                          int wv, unsigned long long &ntest) {
    const PairArgs &a = args();
    const int rep = a.R.cell_rep ? constant(a.R.cell_rep, cell) : 0;
    Cell G;
    G.g = &constant(a.R.geom, rep);
    const Geom &g = *G.g;
    G.cbase = constant(a.R.cell_off, rep);
    // (divisions by a float reciprocal, exact: a small box has at most 512
    // cells, and the half keeps the quotients 1/1024 away from an integer)
    const int local = cell - G.cbase;
    const int q = __builtin_amdgcn_readfirstlane(
        (int)((local + 0.5f) * __builtin_amdgcn_rcpf((float)g.n[0])));
    G.cz = __builtin_amdgcn_readfirstlane((int)((q + 0.5f) * __builtin_amdgcn_rcpf((float)g.n[1])));
    G.cx = local - q * g.n[0];
    G.cy = q - G.cz * g.n[1];
    const SiteArrays &S = a.s[TI];
    double wmac[3] = {0.0, 0.0, 0.0};
    G.ib = constant(S.cstart, cell);
    G.ie = constant(S.cstart, cell + 1);
    const int share = (G.ie - G.ib + kPairWaves - 1) / kPairWaves;  // sites per wave
    if (share > 0) {
        G.ib = min(G.ib + wv * share, G.ie);
        G.ie = min(G.ib + share, G.ie);
        const TileCell tc = tile_cell(G, lane);
        R eps24 = R(0), sig2 = R(0), shift6 = R(0);
        if constexpr (TI == T_LJ) {
            if constexpr (sizeof(R) == 8) {
                eps24 = constant(a.pp.eps24); sig2 = constant(a.pp.sig2); shift6 = constant(a.pp.shift6);
            } else {
                eps24 = constant(a.pp.feps24);
                sig2 = constant(a.pp.fsig2);
                shift6 = constant(a.pp.fshift6);
            }
        }
        // (a wave without sites left helps to stage the tile)
        constexpr int SPP = BlockCfg<TI, R, MOLSITE, MULTI>::SPP;
        for (int first = G.ib, done = 0; done < share; first += SPP, done += SPP) {
            const bool again = done > 0;
            const Pass<R> s = load_pass<TI, R, MOLSITE, MULTI>(G, first, lane);
            Acc acc;
            for (int k = 0; k < 3; ++k) acc.f[k] = acc.v[k] = acc.m[k] = 0.0;
            acc.u = acc.rf = 0.0;
            if constexpr (TI == T_LJ) {
                partner_pass<T_LJ, T_LJ, R, MOLSITE, MULTI, COUNT>(G, s, tc, lane, wv, again, T, acc,
                                                                   eps24, sig2, shift6, ntest);
            } else {
                if (a.present[T_C])
                    partner_pass<TI, T_C, R, MOLSITE, MULTI, COUNT>(G, s, tc, lane, wv, again, T,
                                                                    acc, eps24, sig2, shift6, ntest);
                if (a.present[T_D]) {
                    if (a.present[T_C] || again) __syncthreads();
                    partner_pass<TI, T_D, R, MOLSITE, MULTI, COUNT>(G, s, tc, lane, wv, false, T,
                                                                    acc, eps24, sig2, shift6, ntest);
                }
                if (a.present[T_Q]) {
                    if (a.present[T_C] || a.present[T_D] || again) __syncthreads();
                    partner_pass<TI, T_Q, R, MOLSITE, MULTI, COUNT>(G, s, tc, lane, wv, false, T,
                                                                    acc, eps24, sig2, shift6, ntest);
                }
            }
            if (s.nI > 0) {
                const PairArgs &a = args();
                const SiteArrays &S = a.s[TI];
                wmac[0] += acc.u;
                wmac[1] += acc.v[0] + acc.v[1] + acc.v[2];  // virial = trace of the site tensors
                wmac[2] += acc.rf;
                const bool own = lane < s.nI;  // phase-0 lanes
                if (s.P > 1)
                    fold_phases<TI>(reinterpret_cast<double *>(T.lst[wv]), s.nI, s.P, own, lane, acc);
                const int i = s.I.idx;
                if (own) {
                    S.Fx[i] = acc.f[0]; S.Fy[i] = acc.f[1]; S.Fz[i] = acc.f[2];
                    S.Vx[i] = acc.v[0]; S.Vy[i] = acc.v[1]; S.Vz[i] = acc.v[2];
                    if constexpr (TI >= T_D) {
                        S.Mx[i] = acc.m[0]; S.My[i] = acc.m[1]; S.Mz[i] = acc.m[2];
                    }
                }
            }
        }
        // the reaction-field sum (wmac[2]) is non-zero only for dipole i sites
        constexpr int NM = TI == T_D ? 3 : 2;
        for (int k = 0; k < NM; ++k) wmac[k] = wave_scan(wmac[k]);  // the sum in lane 63
        if (lane == 63)
            for (int k = 0; k < NM; ++k) T.mac[wv][k] = wmac[k];
        __syncthreads();  // (all waves are also done with the tile)
        if (wv == 0 && lane == 0)
            for (int k = 0; k < NM; ++k) {
                wmac[k] = T.mac[0][k];
                for (int w = 1; w < kPairWaves; ++w) wmac[k] += T.mac[w][k];
            }
    }
    if (wv == 0 && lane == 0) {
        const PairArgs &a = args();
        double *o = a.macro_part + 4 * ((size_t)TI * a.ncell + cell);
        o[0] = (TI == T_LJ) ? wmac[0] : 0.0;
        o[1] = (TI == T_LJ) ? 0.0 : wmac[0];
        o[2] = wmac[1];
        o[3] = wmac[2];
    }
}

// One block of four waves per cell of a small box. XCD-aware: hardware block b
// runs on XCD b % 8, and XCD x owns the contiguous cell range [x, x + 1) *
// items_per_xcd, so neighbouring cells share its L2. A grid smaller than 8 *
// items_per_xcd makes the blocks persistent: each walks its XCD's cells with
// stride gridDim.x / 8, and every block leaves after its last cell.
template <int TI, typename R, bool COUNT, bool MOLSITE, int MULTI>
__device__ __forceinline__ void block_cells(const PairArgs &a,
                                            BlockShared<TI, R, MOLSITE, MULTI> &T) {
    if constexpr (MULTI == kTableLds) {  // (read behind the first staging's barrier)
        const Q4<R> *par;
        if constexpr (sizeof(R) == 8)
            par = reinterpret_cast<const Q4<R> *>(a.pp.dpar);
        else
            par = reinterpret_cast<const Q4<R> *>(a.pp.fpar);
        const int k = threadIdx.x;
        if (k < a.pp.nlj * a.pp.nlj) T.tab[k] = par[k];
    }
    if (threadIdx.x == 0) T.zero = 0;  // (as the table)
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int xcd = blockIdx.x & 7, stride = gridDim.x >> 3;
    unsigned long long ntest = 0;
    for (int item = blockIdx.x >> 3; item < a.items_per_xcd; item += stride) {
        const int k = xcd * a.items_per_xcd + item;
        if (k >= a.nsmall) break;
        const int cell = a.R.small_cell ? constant(a.R.small_cell, k) : k;
        pair_cell<TI, R, COUNT, MOLSITE, MULTI>(T, cell, lane, wv, ntest);
    }
    if (COUNT && lane == 0) atomicAdd(&a.counters[8 * TI], ntest);
}

template <typename R, bool COUNT, bool MOLSITE, int MULTI>
__global__ __launch_bounds__(64 * kPairWaves) __attribute__((amdgpu_waves_per_eu(
    BlockCfg<T_LJ, R, MOLSITE, MULTI>::WAVES))) void k_block_lj(PairArgs a) {
    __shared__ BlockShared<T_LJ, R, MOLSITE, MULTI> T;
    static_assert(blocks_per_cu(sizeof(T)) >= BlockCfg<T_LJ, R, MOLSITE, MULTI>::WAVES, "occupancy");
    block_cells<T_LJ, R, COUNT, MOLSITE, MULTI>(a, T);
}

// The electrostatic i-site types in one launch, one per blockIdx.y: each alone
// leaves a chip of 256 CUs with one or two blocks per CU that wait for loads and
// barriers; together they overlap (9001 mixture molecules FP32, charges and
// quadrupoles: 24 + 24 -> 30 us; 3001 of all site types FP64, three types: 62 ->
// 42).
template <typename R, bool COUNT>
__global__ __launch_bounds__(64 * kPairWaves) __attribute__((amdgpu_waves_per_eu(
    BlockCfg<T_C, R, false, kTableNone>::WAVES))) void k_block_es(PairArgs a) {
    typedef BlockShared<T_C, R, false, kTableNone> TC;
    typedef BlockShared<T_D, R, false, kTableNone> TD;
    typedef BlockShared<T_Q, R, false, kTableNone> TQ;
    static_assert(sizeof(TC) == sizeof(TD) && sizeof(TC) == sizeof(TQ), "one LDS buffer");
    static_assert(blocks_per_cu(sizeof(TC)) >= BlockCfg<T_C, R, false, kTableNone>::WAVES, "occupancy");
    __shared__ alignas(alignof(TC)) unsigned char buf[sizeof(TC)];
    const int t = a.es[blockIdx.y];
    if (t == T_C)
        block_cells<T_C, R, COUNT, false, kTableNone>(a, *reinterpret_cast<TC *>(buf));
    else if (t == T_D)
        block_cells<T_D, R, COUNT, false, kTableNone>(a, *reinterpret_cast<TD *>(buf));
    else
        block_cells<T_Q, R, COUNT, false, kTableNone>(a, *reinterpret_cast<TQ *>(buf));
}

template <typename R, bool C> PairKernel pick_lj(bool molsite, int nlj) {
    if (nlj > kTableIds)
        return molsite ? k_block_lj<R, C, true, kTableGlobal> : k_block_lj<R, C, false, kTableGlobal>;
    if (nlj > 1) return molsite ? k_block_lj<R, C, true, kTableLds> : k_block_lj<R, C, false, kTableLds>;
    return molsite ? k_block_lj<R, C, true, kTableNone> : k_block_lj<R, C, false, kTableNone>;
}

PairKernel block_kernel_lj(bool fp32, bool count, bool molsite, int nlj) {
    if (fp32) return count ? pick_lj<float, true>(molsite, nlj) : pick_lj<float, false>(molsite, nlj);
    return count ? pick_lj<double, true>(molsite, nlj) : pick_lj<double, false>(molsite, nlj);
}
PairKernel block_kernel_es(bool fp32, bool count) {
    if (fp32) return count ? k_block_es<float, true> : k_block_es<float, false>;
    return count ? k_block_es<double, true> : k_block_es<double, false>;
}

}  // namespace mdx
