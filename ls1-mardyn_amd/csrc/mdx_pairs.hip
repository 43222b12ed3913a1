// mdx_pairs.hip -- site-pair traversal kernels (gfx950, wave64, no MFMA).
//
// The cell kernels; mdx_pairs_block.hip holds the block kernels of small dense
// boxes.
//
// The ten site-pair loops of VectorizedCellProcessor::_calculatePairs
// (VectorizedCellProcessor.cpp:794-2730) with the seven bodies _loopBodyLJ ..
// _loopBodyQuadrupole (VectorizedCellProcessor.cpp:171-792), evaluated owner-
// computes: kernel k_pairs<TI> runs one wavefront per cell for the sites of
// type TI and accumulates force, virial and torque of those sites only.
// The cutoff is tested on molecule centres (calcDistLookup,
// SIMD_VectorizedCellProcessorHelpers.h:427-472): LJ against rcLJ^2, the
// electrostatic types against rc^2, strictly less; inside the own cell a pair
// at molecule distance 0 (the same molecule) is skipped (SingleCellPolicy_).
//
// Precision forms (template R):
//   double : all arithmetic FP64, absolute positions, j images shifted by +-L
//            exactly as the reference's halo copies are (r + L).
//   float  : pair arithmetic FP32 on positions relative to the owning cell's
//            corner (|x| <= ~cell length, so FP32 keeps ~1e-7 absolute
//            accuracy at any box size); the cutoff decision is re-made in FP64
//            when the FP32 r^2 lies within 1e-5 relative of rc^2 so the pair
//            set equals the FP64 one; the pair terms of one drained hit list
//            (at most a list length of partners per lane) are summed in FP32
//            and added to the site's FP64 accumulators once per drain, so
//            every per-site and per-molecule sum across drains, cells and
//            partner types is FP64 (the reference's MIXED build accumulates
//            in RealAccumVec, RealAccumVecSPDP.h).
#include "mdx_pair_common.h"

namespace mdx {

// What the staged sites of a neighbour take: the offset of their positions (FP64:
// the image shift; FP32: between the cells' corners), and the site of tile entry
// e, e + dj.
template <typename R> struct NbrRec;
template <> struct NbrRec<double> {
    double x, y, z;
    int dj, pad;
};
template <> struct alignas(16) NbrRec<float> {
    float x, y, z;
    int dj;
};

// LDS tile: the j sites of the 27 neighbour images of one cell, positions
// already moved into the i cell's frame (FP64: + image shift, exactly the
// reference's halo copy r + L; FP32: + offset of the neighbour's corner).
template <int TI, typename R, bool MOLSITE, bool MULTI> struct TileCfg {
    static constexpr bool ORI = TI != T_LJ;  // partners may be dipoles / quadrupoles
    static constexpr bool MOL = !MOLSITE;    // molecule positions differ from sites
    static constexpr bool LJID = TI == T_LJ && MULTI;  // several LJ centre types
    // Per-lane hit list entries (LIST) and sites per LDS chunk (CAP). The
    // kernels are bound by VALU issue, so the tile is sized for occupancy
    // first (160 KB of LDS per CU in steps of 1280 bytes, shared by the
    // wavefronts of its 4 SIMDs, next to the register limit of each
    // instantiation) and chunk count second: each chunk ends with a drain of
    // half-empty lists. Values measured best on the 1 M-molecule LJ slab and 64
    // replicas (FP32 one-centre: 414 sites fill the 10240 bytes of 16 blocks per
    // CU, 316 -> 307 us for the replicas against 352) and on the 1 M-molecule
    // mixture (2CLJQ + water). The FP32 quadrupole kernel takes the 12800 bytes
    // of 12 blocks: its 36-cell neighbourhood of charges goes in three chunks
    // instead of five, 618 -> 576 us (114 sites: 618, 160: 682, 184: 618).
    // Chunks of equal length cost more than they level (2234 -> 2288 us for all
    // three). The FP64 tiles that carry molecule positions or orientations keep
    // 16-entry lists for their larger records.
    static constexpr int LIST = (sizeof(R) == 8 && !(TI == T_LJ && MOLSITE)) ? 16 : 24;
    static constexpr int CAP =
        TI == T_LJ ? (MOLSITE ? (sizeof(R) == 4 ? 414 : 192) : (sizeof(R) == 4 ? 192 : 112))
        : TI == T_C ? (sizeof(R) == 4 ? 112 : 72)
        : TI == T_Q ? (sizeof(R) == 4 ? 176 : 104)
                    : (sizeof(R) == 4 ? 192 : 160);
    // Quadrupole i sites are few per cell (one per 2CLJQ molecule) against
    // a neighbourhood of many partner sites, so the kernel takes two cells
    // side by side in x at a time (JOINT): their neighbourhood of 4 x 3 x 3
    // cells is staged once for both, two thirds of what two 27-cell tiles
    // load, at the price of tests against the 9 cells that are beyond the
    // cutoff of one of the two (NB neighbour ranges at most).
    static constexpr bool JOINT = TI == T_Q;
    static constexpr int NB = JOINT ? 36 : 27;
    // Minimum waves per SIMD the kernel's registers are allocated for (1: no
    // bound, the compiler's choice). Tiles of at most 10 KB of LDS (lists
    // included) let 16 blocks share a CU, 4 waves per SIMD, when the
    // registers fit 128: the charge kernels (112 and 72 sites) get the bound,
    // which makes the compiler fit them with a few spilled values outside the
    // pair loops (FP32: 129 registers and 1090 us without, 936 with); so does
    // the FP32 quadrupole kernel, whose larger tile runs 3 waves, for 575 us
    // against 588 without. The FP64 multi-site LJ kernel (112 sites) fits
    // without it, and the FP64 quadrupole kernel's 104-site tile (13 KB) reaches
    // 3 waves per SIMD with its 160 registers.
    static constexpr int WAVES =
        (TI == T_Q && sizeof(R) == 4) || TI == T_C ? 4 : 1;
};

template <int TI, typename R, bool MOLSITE, bool MULTI> struct Tile {
    using C = TileCfg<TI, R, MOLSITE, MULTI>;
    // CAP slots of the largest record set (site, molecule, orientation,
    // head index and site count); each partner pass lays out only the records
    // its partner type needs (PassTile), so a pass with smaller records holds
    // more sites in the same bytes
    static constexpr int SLOT =
        (int)sizeof(Q4<R>) * (1 + C::MOL + C::ORI) + (C::MOL && TI != T_LJ ? 3 : 0);
    alignas(32) unsigned char raw[C::CAP * SLOT];
    // per-lane hit lists (LDS addresses of site records); the staging's marks, which
    // are cleared a word at a time, lie in the same bytes
    alignas(4) unsigned short lst[C::LIST][64];
    int pre[C::NB + 1];               // first tile entry of each neighbour
    NbrRec<R> nbr[C::NB];
};

// The records of one partner pass (partner type TJ) in a tile's slot bytes:
// p site position (w = charge / moment, LJ table column, or |x|^2 in FP32
// one-centre tiles), m molecule position (w = |m|^2 in FP32 tiles), e
// orientation (dipole and quadrupole partners), h addresses of the first sites
// and ns site counts at heads (charge partners, tested per molecule).
template <int TI, int TJ, typename R, bool MOLSITE, bool MULTI> struct PassTile {
    using C = TileCfg<TI, R, MOLSITE, MULTI>;
    using TT = Tile<TI, R, MOLSITE, MULTI>;
    static constexpr bool HEADS = C::MOL && TJ == T_C && TI != T_LJ;
    static constexpr bool ORIJ = TI != T_LJ && TJ >= T_D;
    static constexpr int REC = 1 + C::MOL + ORIJ;
    static constexpr int CAP =
        (C::CAP * TT::SLOT) / ((int)sizeof(Q4<R>) * REC + (HEADS ? 3 : 0));
    static_assert(CAP >= C::CAP && CAP < 65536, "pass capacity");
    Q4<R> *p, *m, *e;
    unsigned short *h;
    unsigned char *ns;
    __device__ __forceinline__ explicit PassTile(TT &t) {
        p = reinterpret_cast<Q4<R> *>(t.raw);
        m = p + (C::MOL ? CAP : 0);
        e = p + CAP * (1 + C::MOL);
        h = reinterpret_cast<unsigned short *>(p + CAP * REC);
        ns = reinterpret_cast<unsigned char *>(h + (HEADS ? CAP : 0));
    }
};

template <typename R>
__device__ __forceinline__ NbrRec<R> nbr_rec(const Geom &g, const Nbr &b, int dj);
template <>
__device__ __forceinline__ NbrRec<double> nbr_rec<double>(const Geom &, const Nbr &b, int dj) {
    return {b.s[0], b.s[1], b.s[2], dj, 0};
}
template <>
__device__ __forceinline__ NbrRec<float> nbr_rec<float>(const Geom &g, const Nbr &b, int dj) {
    return {(float)(b.dd[0] * g.cl[0]), (float)(b.dd[1] * g.cl[1]), (float)(b.dd[2] * g.cl[2]), dj};
}

constexpr int kUnroll = 4;  // stage-A candidates in flight per lane

// All pairs of the lane's i site with the j sites of type TJ in the 27
// neighbour images: (1) lanes 0..26 fetch the neighbour ranges in one round,
// (2) the neighbourhood is staged into LDS in chunks of CAP sites with
// coalesced, independent loads, (3) stage A tests the molecule-centre cutoff
// from LDS (kUnroll candidates per lane in flight) and keeps per-lane hit
// lists, (4) stage B evaluates the bodies for the hits.
template <int TI, int TJ, typename R, bool MOLSITE, bool MULTI, bool COUNT>
__device__ __forceinline__ void partner_pass(const PairArgs &a, const Geom &g, int cbase,
                                             const ISite<R> &I, bool valid,
                                             int cx, int cy, int cz, int nxs, int ph, int P,
                                             int lane,
                                             Tile<TI, R, MOLSITE, MULTI> &T, Acc &acc, R eps24,
                                             R sig2, R shift6, unsigned long long &ntest) {
    using C = TileCfg<TI, R, MOLSITE, MULTI>;
    constexpr int TAB = MULTI ? kTableGlobal : kTableNone;
    const R *par;  // the interleaved LJ table
    if constexpr (sizeof(R) == 8)
        par = a.pp.dpar;
    else
        par = a.pp.fpar;
    const SiteArrays &J = a.s[TJ];
    const double rc2 = (TI == T_LJ) ? a.rclj2 : a.rc2;
    const R rc2r = (R)rc2;
    // FP32 tiles: the test record's w holds |x|^2 and stage A computes
    // r^2 = (|i|^2 + |j|^2) - 2 i.j (4 instead of 6 operations); its rounding
    // stays below 1.5e-5 (cl / rc)^2 rc^2 (coordinates within two cell edges
    // of the i cell's corner), so stage A keeps candidates up to that much
    // above rc^2 and stage B re-decides the band in FP64 as before
    constexpr bool NORM = sizeof(R) == 4 && (C::MOL || (TI == T_LJ && !C::LJID));
    // idle lanes test from far away: r^2 overflows or exceeds any cutoff
    const V3<R> far = {R(1e30), R(1e30), R(1e30)};
    const V3<R> Imol = valid ? I.mol : far, Ipos = valid ? I.pos : far;
    // FP32 re-check band around rc^2 (relative 1e-5, far above FP32 rounding
    // of cell-relative coordinates)
    const R lo = rc2r * R(1 - 1e-5), hi = rc2r * R(1 + 1e-5);
    // stage-A bound: FP64 rc^2; FP32 the top of the re-check band, widened
    // by the rounding bound of the expanded r^2 where that is used
    R cut = sizeof(R) == 4 ? hi : rc2r;
    if constexpr (NORM) {
        // (the bound grows with the square of the frame's extent: nxs - 1
        // cell edges in x when two cells share the tile)
        const double clm = fmax(g.cl[0], fmax(g.cl[1], g.cl[2]));
        const double ext = 0.5 * (nxs - 1);
        const double band = fmax(1e-5, 1.5e-5 * ext * ext * clm * clm / rc2);
        cut = (R)(rc2 * (1.0 + band));
    }
    unsigned long long nhit = 0;
    int nk = 0, j0 = 0;
    const int nb = 9 * nxs;  // neighbour ranges: 27, or 36 for two cells
    Nbr nbr = neighbour(g, cx, cy, cz, lane, nxs);
    if (lane < nb && nbr.ok) {
        j0 = J.cstart[cbase + nbr.cell];
        nk = J.cstart[cbase + nbr.cell + 1] - j0;
    }
    const int incl = wave_scan(nk), pre = incl - nk;
    if (lane < nb) {
        T.pre[lane + 1] = incl;
        T.nbr[lane] = nbr_rec<R>(g, nbr, j0 - pre);
    }
    if (lane == 0) T.pre[0] = 0;
    const int total = __builtin_amdgcn_readlane(incl, 63);
    __syncthreads();
    // Charge partners are tested once per molecule (neutral molecules carry
    // two or more charges): the tile keeps a molecule's sites contiguous, the
    // head list names each molecule's first site, stage A runs over heads and
    // stage B over a hit's sites; chunks then end at molecule boundaries. For
    // LJ, dipole and quadrupole partners (typically one or two per molecule)
    // the indirection costs more than it saves (measured) and every site is a
    // candidate.
    constexpr bool heads = C::MOL && TJ == T_C;
    using PT = PassTile<TI, TJ, R, MOLSITE, MULTI>;
    static_assert(PT::HEADS == heads, "head layout");
    const PT V(T);
    // (a molecule's charges are contiguous, and its first one carries the
    // count: one load per site, no chain through the molecule index)
    for (int base = 0; base < total;) {
        int nst = min(PT::CAP, total - base);
        // heads: a chunk that ends inside a molecule ends at that molecule's
        // first site instead (the last head of the chunk); whether it does is
        // the head count of the site after the chunk, loaded beside the
        // chunk's own sites
        int next_head = 1;
        if constexpr (heads) {
            if (base + nst < total) {
                const int idx = base + nst;
                const int k = tile_k(T.pre, idx, nb);
                next_head = SiteView<R>::heads(J, T.nbr[k].dj + idx);
            }
        }
        int nh = nst;
        int hb = 0, last_head = 0;
        // The neighbour of each tile entry: the neighbours of the chunk leave
        // their number + 1 at their first entry (in the hit lists' bytes, not in
        // use here), and a maximum scan over 64 entries at a time carries it to
        // the others: 6 operations without an LDS round trip, where a binary
        // search of the prefix takes five dependent reads of 7 each. With the
        // neighbours' offsets in one LDS record each, and list lengths and prefix
        // by DPP: 1 M-molecule slab FP32 397 -> 355 us, FP64 496 -> 440; 1 M
        // mixture, LJ 842 -> 800, charges 973 -> 936, quadrupoles 706 -> 653.
        unsigned char *mark = reinterpret_cast<unsigned char *>(T.lst);
        static_assert(PT::CAP + 3 <= sizeof(T.lst), "marks");
        static_assert(sizeof(T) < 65536, "LDS addresses in 16 bits");
        for (int z = 4 * lane; z < nst; z += 256) *reinterpret_cast<unsigned *>(mark + z) = 0u;
        __syncthreads();
        if (nk > 0 && pre < base + nst && incl > base)
            mark[max(pre - base, 0)] = (unsigned char)(lane + 1);
        __syncthreads();
        int carry = 0;
        for (int s0 = 0; s0 < nst; s0 += 64) {
            const int s = s0 + lane;
            bool head = false;
            const int k1 = max(wave_max_scan(s < nst ? mark[s] : 0), carry);
            carry = __builtin_amdgcn_readlane(k1, 63);
            if (s < nst) {
            const NbrRec<R> off = T.nbr[k1 - 1];
            const int j = off.dj + base + s;
            const V3<R> p = SiteView<R>::pos(J, j);
            Q4<R> q;
            q.x = p.x + off.x;
            q.y = p.y + off.y;
            q.z = p.z + off.z;
            q.w = R(0);
            // column offset of the interleaved table, as bits
            if constexpr (C::LJID) q.w = column_bits<R>(SiteView<R>::column(J, j));
            if constexpr (TI != T_LJ) q.w = SiteView<R>::par(J, j);
            if constexpr (NORM && !C::MOL) q.w = q.x * q.x + q.y * q.y + q.z * q.z;
            V.p[s] = q;
            if constexpr (C::MOL) {
                const V3<R> m = SiteView<R>::mol(J, j);
                if constexpr (heads) {
                    const int w = SiteView<R>::heads(J, j);
                    head = w != 0;
                    V.ns[s] = (unsigned char)w;
                }
                Q4<R> mq{m.x + off.x, m.y + off.y, m.z + off.z, R(0)};
                if constexpr (NORM) mq.w = mq.x * mq.x + mq.y * mq.y + mq.z * mq.z;
                V.m[s] = mq;
            }
            if constexpr (TI != T_LJ && TJ >= T_D) {
                const V3<R> e = SiteView<R>::ori(J, j);
                V.e[s] = Q4<R>{e.x, e.y, e.z, R(0)};
            }
            }
            if constexpr (heads) {  // compact the heads in tile order
                const unsigned long long hm = __ballot(head);
                if (head)  // the address of the head's record
                    V.h[hb + __popcll(hm & ((1ull << lane) - 1ull))] =
                        (unsigned short)(lds_address(V.p) + s * (unsigned)sizeof(Q4<R>));
                hb += __popcll(hm);
                if (hm) last_head = s0 + 63 - __clzll((long long)hm);
            }
        }
        if constexpr (heads) {
            nh = hb;
            // the split molecule's sites run from the last head to the chunk
            // end: drop them (and that head), the next chunk starts there
            // (a chunk holds many molecules of at most kMaxSite sites, so
            // last_head > 0)
            if (next_head == 0 && last_head > 0) {
                nst = last_head;
                nh = hb - 1;
            }
        }
        __syncthreads();
        // A listed candidate is the LDS address of its site record; its test
        // record (the molecule's, where that differs) and orientation lie MO
        // and EO bytes behind. la: the end of the lane's list.
        constexpr unsigned REC = sizeof(Q4<R>);
        constexpr unsigned MO = C::MOL ? PT::CAP * REC : 0, EO = PT::CAP * REC * (1 + C::MOL);
        const unsigned pb = lds_address(V.p), l0 = lds_address(&T.lst[0][lane]);
        constexpr unsigned ROW = sizeof(T.lst[0]);  // an entry is a row of the lists
        unsigned la = l0;
        auto index = [&](unsigned at) -> int { return (int)((at - pb) / REC); };
        // Stage B. A listed candidate is final unless its molecule distance
        // is 0 (the molecule itself, SingleCellPolicy_) or, in FP32, lies in
        // the band [lo, hi] around rc^2, where the decision is re-made in FP64
        // from the unrounded positions so the pair set equals the FP64 one.
        auto recheck = [&](int s) -> bool {  // the FP64 decision for tile entry s
            const int idx = base + s;
            const int k = tile_k(T.pre, idx, nb);
            const NbrRec<R> rec = T.nbr[k];
            const int j = rec.dj + idx;
            V3<double> sh;  // the image shift
            if constexpr (sizeof(R) == 8) {
                sh = {rec.x, rec.y, rec.z};
            } else {
                const Nbr b = neighbour(g, cx, cy, cz, k, nxs);
                sh = {b.s[0], b.s[1], b.s[2]};
            }
            // molecule positions through the sites' molecule indices (the
            // FP32 form builds no FP64 per-site copies)
            const int mi = a.s[TI].mol[I.idx], mj = J.mol[j];
            const double ex = a.mrx[mi] - (a.mrx[mj] + sh.x);
            const double ey = a.mry[mi] - (a.mry[mj] + sh.y);
            const double ez = a.mrz[mi] - (a.mrz[mj] + sh.z);
            const double r2d = ex * ex + ey * ey + ez * ez;
            return r2d < rc2 && r2d != 0.0;
        };
        auto accept = [&](unsigned at, const Q4<R> &q) -> bool {
            const V3<R> mi = C::MOL ? I.mol : I.pos;
            const R dx = mi.x - q.x, dy = mi.y - q.y, dz = mi.z - q.z;
            const R r2 = dx * dx + dy * dy + dz * dz;
            if (r2 == R(0)) return false;
            if constexpr (sizeof(R) == 4) {
                if (r2 >= lo) return recheck(index(at));
            }
            return true;
        };
        auto drain = [&]() {
            Part32 pa;
            pa.clear();
            // the longest list: a scalar trip count
            const int emax = __builtin_amdgcn_readlane(wave_max_scan((int)((la - l0) / ROW)), 63);
            if constexpr (TI == T_LJ) {
                // LJ: every lane runs every entry up to the longest list
                // (exhausted lanes on the tile's first record with the pair
                // masked off), so the loop has no branch. FP32: entries in the
                // re-check band around rc^2 are masked off here, and re-decided
                // in FP64 in a second walk (rare: some 2e-5 of the entries)
                unsigned long long near = 0;
                unsigned lp = l0;
                for (int e = 0; e < emax; ++e, lp += ROW) {
                    const bool act = lp < la;
                    unsigned raw = lds_value<unsigned short>(lp);  // e < LIST: in bounds
                    asm("" : "+v"(raw));  // (read by all lanes: no branch around it)
                    const unsigned at = act ? raw : pb;
                    const Q4<R> qj = lds_q4<R>(at + MO);
                    const V3<R> mi = C::MOL ? I.mol : I.pos;
                    const R dx = mi.x - qj.x, dy = mi.y - qj.y, dz = mi.z - qj.z;
                    const R r2 = dx * dx + dy * dy + dz * dz;
                    bool ok = act && r2 != R(0);
                    if constexpr (sizeof(R) == 4) {
                        const bool inner = r2 < lo;
                        near |= __ballot(ok && !inner);
                        ok = ok && inner;
                    }
                    const Q4<R> pj = C::MOL ? lds_q4<R>(at) : qj;
                    eval_lj<R, MOLSITE, TAB>((const Q4<R> *)nullptr, par, I, pj, qj, ok, eps24,
                                                sig2, shift6, acc, pa);
                    if (COUNT) nhit += ok;
                }
                if constexpr (sizeof(R) == 4) {
                    if (near) {
                        lp = l0;
                        for (int e = 0; e < emax; ++e, lp += ROW) {
                            const unsigned at = lp < la ? lds_value<unsigned short>(lp) : pb;
                            const Q4<R> qj = lds_q4<R>(at + MO);
                            const V3<R> mi = C::MOL ? I.mol : I.pos;
                            const R dx = mi.x - qj.x, dy = mi.y - qj.y, dz = mi.z - qj.z;
                            const R r2 = dx * dx + dy * dy + dz * dz;
                            const bool b = lp < la && r2 != R(0) && !(r2 < lo);
                            if (!__any(b)) continue;
                            const bool ok = b && recheck(index(at));
                            const Q4<R> pj = C::MOL ? lds_q4<R>(at) : qj;
                            eval_lj<R, MOLSITE, TAB>((const Q4<R> *)nullptr, par, I, pj, qj, ok,
                                                        eps24, sig2, shift6, acc, pa);
                            if (COUNT) nhit += ok;
                        }
                    }
                }
            } else {
                // the next entry's address and cutoff record are read one
                // iteration ahead, so their LDS latency overlaps the current body
                unsigned an = pb, lp = l0;
                Q4<R> qn{};
                if (lp < la) {
                    an = lds_value<unsigned short>(lp);
                    qn = lds_q4<R>(an + MO);
                }
                for (int e = 0; e < emax; ++e) {
                    const bool act = lp < la;
                    const unsigned at = an;
                    const Q4<R> qj = qn;
                    lp += ROW;
                    if (lp < la) {
                        an = lds_value<unsigned short>(lp);
                        qn = lds_q4<R>(an + MO);
                    }
                    if (act && accept(at, qj)) {
                        if constexpr (heads) {
                            const int ns = (int)V.ns[index(at)];  // the molecule's sites from `at` on
                            for (int t = 0; t < ns; ++t) {
                                const Q4<R> pj = lds_q4<R>(at + t * REC);
                                eval_pair<TI, TJ, R, MOLSITE>((R)a.epsRFInvrc3, I, Q4<R>{}, pj, qj, acc, pa);
                            }
                            if (COUNT) nhit += ns;
                        } else {
                            const Q4<R> pj = C::MOL ? lds_q4<R>(at) : qj;
                            Q4<R> eq{};
                            if constexpr (PT::ORIJ) eq = lds_q4<R>(at + EO);
                            eval_pair<TI, TJ, R, MOLSITE>((R)a.epsRFInvrc3, I, eq, pj, qj, acc, pa);
                            if (COUNT) ++nhit;
                        }
                    }
                }
            }
            if constexpr (sizeof(R) == 4) pa.flush(acc);
            la = l0;
        };
        // Stage A: keep candidates below the cutoff (FP32: up to the top of
        // the re-check band). Row m holds candidates m * P + ph; rows below
        // full are inside [0, nst) for every phase and need no bounds test,
        // and idle lanes carry a far-away position, so the bulk loop is a
        // read, a distance, a compare and a list write per candidate. Its VALU
        // count bounds these kernels (80 to 90 % of the issue slots): lists of
        // addresses instead of indices, a running list address instead of a
        // count and |i|^2 taken from the bound leave 31 operations of 37 per
        // four candidates (1 M mixture, FP32: LJ 800 -> 751 us, charges 936 ->
        // 859, quadrupoles 653 -> 618; 64 replicas 328 -> 316).
        // wave-uniform trip counts (scalar loop control; nh and P are
        // wave-uniform, so the division runs on the scalar unit)
        const int nhs = __builtin_amdgcn_readfirstlane(nh), Ps = __builtin_amdgcn_readfirstlane(P);
        const int per = (nhs + Ps - 1) / Ps, full = per - 1;
        // candidate c of the stage-A sequence -> its record's address
        auto cand = [&](int c) -> unsigned {
            if constexpr (heads) return V.h[c];
            else return pb + (unsigned)c * REC;
        };
        const V3<R> mi = C::MOL ? Imol : Ipos;
        // NORM: -2 i, and |i|^2 taken from the bound (idle lanes: far away,
        // never a hit)
        R nx = R(0), ny = R(0), nz = R(0), bound = cut;
        if constexpr (NORM) {
            bound = cut - (mi.x * mi.x + mi.y * mi.y + mi.z * mi.z);
            nx = R(-2) * mi.x;
            ny = R(-2) * mi.y;
            nz = R(-2) * mi.z;
        }
        auto hit = [&](const Q4<R> &q) -> bool {
            if constexpr (NORM) {
                return __builtin_fmaf(nx, q.x, __builtin_fmaf(ny, q.y, __builtin_fmaf(nz, q.z, q.w))) <= bound;
            } else {
                const R dx = mi.x - q.x, dy = mi.y - q.y, dz = mi.z - q.z;
                const R r2 = dx * dx + dy * dy + dz * dz;
                return sizeof(R) == 4 ? r2 <= bound : r2 < bound;
            }
        };
        // every candidate is written at the end of the list and kept only on a
        // hit (no branch; the drain test keeps the write within the list)
        auto list = [&](unsigned at, bool h) {
            *(__attribute__((address_space(3))) unsigned short *)la = (unsigned short)at;
            la += h ? ROW : 0u;
        };
        int m0 = 0;
        for (; m0 + kUnroll <= full; m0 += kUnroll) {
            // drain when some lane's list could overflow in this group
            if (__any(la > l0 + (C::LIST - kUnroll) * ROW)) drain();
            unsigned at[kUnroll];
            Q4<R> q[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                at[u] = cand(ph + (m0 + u) * P);
                q[u] = lds_q4<R>(at[u] + MO);
            }
            if (COUNT && valid) ntest += kUnroll;
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) list(at[u], hit(q[u]));
        }
        for (; m0 < per; ++m0) {  // the last rows, bounds-tested
            if (__any(la > l0 + (C::LIST - 1) * ROW)) drain();
            const int c = ph + m0 * P;
            const unsigned at = cand(min(c, nh - 1));
            const bool in = valid && c < nh;
            if (COUNT && in) ++ntest;
            list(at, in && hit(lds_q4<R>(at + MO)));
        }
        drain();
        __syncthreads();
        base += nst;
    }
    if (COUNT) {
        for (int o = 32; o > 0; o >>= 1) nhit += __shfl_xor(nhit, o, 64);
        if (lane == 0) atomicAdd(&a.counters[1 + Kind<TI, TJ>::k], nhit);
    }
}

__device__ __forceinline__ double shfl_xor_d(double v, int o) { return __shfl_xor(v, o, 64); }

// All i sites of one cell (global index) with their partners; adds the
// cell's per-lane macroscopic sums to wmac and writes a zero row for the cell
// (flush_macro later stores the sums of a group of cells in one row).
// span = 2: the cell and the next one in x together, over their common
// neighbourhood (the i sites of the second cell move into the first cell's
// FP32 frame). Returns whether the cells have i sites.
template <int TI, typename R, bool COUNT, bool MOLSITE, bool MULTI>
__device__ __forceinline__ bool pair_cell(const PairArgs &a, Tile<TI, R, MOLSITE, MULTI> &T,
                                          int cell, int span, int lane,
                                          unsigned long long &ntest, double (&wmac)[3]) {
    bool empty;
    {
        const int rep = cell_replica(a.R, cell);
        const Geom &g = a.R.geom[rep];
        const int cbase = a.R.cell_off[rep], local = cell - cbase;
        const SiteArrays &S = a.s[TI];
        const int i_begin = S.cstart[cell], i_end = S.cstart[cell + span];
        const int i_mid = span > 1 ? S.cstart[cell + 1] : i_end;  // the second cell's first site
        const int nxs = span + 2;
        empty = i_begin == i_end;
        const int cx = local % g.n[0], cy = (local / g.n[0]) % g.n[1],
                  cz = local / (g.n[0] * g.n[1]);
        R eps24 = R(0), sig2 = R(0), shift6 = R(0);
        if constexpr (TI == T_LJ) {
            if constexpr (sizeof(R) == 8) {
                eps24 = a.pp.eps24[0]; sig2 = a.pp.sig2[0]; shift6 = a.pp.shift6[0];
            } else {
                eps24 = a.pp.feps24[0]; sig2 = a.pp.fsig2[0]; shift6 = a.pp.fshift6[0];
            }
        }
        for (int chunk = i_begin; chunk < i_end; chunk += 64) {
            // lane = ph * nI + il: P = floor(64 / nI) phases of the chunk's nI
            // sites split the partner candidates; the 64 - P * nI lanes left
            // over idle (phase 0, never a hit). LJ kernels cap P at 8: their
            // sparse cells (vapour) have few candidates, and more phases only
            // lengthen the phase fold; electrostatic kernels, whose cells hold
            // a few sites of many candidates, gain from up to 16 (measured)
            const int nI = min(64, i_end - chunk);
            const int P = min(64 / nI, TI == T_LJ ? 8 : 16);
            // lane / nI through a float reciprocal (exact: lane < 64, nI <= 64,
            // and (lane + 0.5) / nI stays >= 1/128 away from an integer)
            const int ph0 = (int)(((float)lane + 0.5f) * __builtin_amdgcn_rcpf((float)nI));
            const int il = lane - ph0 * nI;
            const bool valid = ph0 < P;
            const int ph = valid ? ph0 : 0;
            const int i = chunk + (valid ? il : 0);
            ISite<R> I;
            I.pos = SiteView<R>::pos(S, i);
            I.mol = MOLSITE ? I.pos : SiteView<R>::mol(S, i);
            if constexpr (sizeof(R) == 4) {
                if (i >= i_mid) {  // second cell: one cell edge further in x
                    const float sx = (float)g.cl[0];
                    I.pos.x += sx;
                    I.mol.x += sx;
                }
            }
            I.idx = i;
            if constexpr (TI >= T_D) I.e = SiteView<R>::ori(S, i);
            if constexpr (TI == T_LJ) {
                I.ljrow = MULTI ? a.pp.nlj * SiteView<R>::column(S, i) : 0;
            } else
                I.par = SiteView<R>::par(S, i);
            Acc acc;
            for (int k = 0; k < 3; ++k) acc.f[k] = acc.v[k] = acc.m[k] = 0.0;
            acc.u = acc.rf = 0.0;
            if constexpr (TI == T_LJ) {
                partner_pass<T_LJ, T_LJ, R, MOLSITE, MULTI, COUNT>(a, g, cbase, I, valid, cx, cy, cz, nxs, ph, P,
                                                                   lane, T, acc, eps24, sig2,
                                                                   shift6, ntest);
            } else {
                if (a.present[T_C])
                    partner_pass<TI, T_C, R, MOLSITE, MULTI, COUNT>(a, g, cbase, I, valid, cx, cy, cz, nxs, ph, P,
                                                                    lane, T, acc, eps24, sig2,
                                                                    shift6, ntest);
                if (a.present[T_D])
                    partner_pass<TI, T_D, R, MOLSITE, MULTI, COUNT>(a, g, cbase, I, valid, cx, cy, cz, nxs, ph, P,
                                                                    lane, T, acc, eps24, sig2,
                                                                    shift6, ntest);
                if (a.present[T_Q])
                    partner_pass<TI, T_Q, R, MOLSITE, MULTI, COUNT>(a, g, cbase, I, valid, cx, cy, cz, nxs, ph, P,
                                                                    lane, T, acc, eps24, sig2,
                                                                    shift6, ntest);
            }
            // fold the phases of each site into its phase-0 lane, in phase
            // order (the virial sums below take the per-lane parts before
            // the fold)
            wmac[1] += acc.v[0] + acc.v[1] + acc.v[2];  // virial = trace of the site tensors
            if (P > 1) {
                // through LDS: the tile is free after the partner passes
                constexpr int NA = TI >= T_D ? 9 : 6;
                static_assert(sizeof(T) >= NA * 64 * sizeof(double), "fold scratch");
                double *fb = reinterpret_cast<double *>(&T);
                for (int k = 0; k < 3; ++k) {
                    fb[k * 64 + lane] = acc.f[k];
                    fb[(3 + k) * 64 + lane] = acc.v[k];
                    if constexpr (TI >= T_D) fb[(6 + k) * 64 + lane] = acc.m[k];
                }
                __syncthreads();
                if (valid && ph == 0)
                    for (int q = 1; q < P; ++q) {
                        const int src = lane + q * nI;
                        for (int k = 0; k < 3; ++k) {
                            acc.f[k] += fb[k * 64 + src];
                            acc.v[k] += fb[(3 + k) * 64 + src];
                            if constexpr (TI >= T_D) acc.m[k] += fb[(6 + k) * 64 + src];
                        }
                    }
                __syncthreads();
            }
            if (valid && ph == 0 && a.kvx) {
                // VCP1CLJRMM (VCP1CLJRMM.cpp:300-362): the site's force, times
                // dt/m, goes straight into its molecule's velocity
                a.kvx[i] = __dadd_rn(a.kvx[i], __dmul_rn(acc.f[0], a.kick));
                a.kvy[i] = __dadd_rn(a.kvy[i], __dmul_rn(acc.f[1], a.kick));
                a.kvz[i] = __dadd_rn(a.kvz[i], __dmul_rn(acc.f[2], a.kick));
            } else if (valid && ph == 0) {
                S.Fx[i] = acc.f[0]; S.Fy[i] = acc.f[1]; S.Fz[i] = acc.f[2];
                double vv[3] = {__dmul_rn(a.vscale, acc.v[0]), __dmul_rn(a.vscale, acc.v[1]),
                                __dmul_rn(a.vscale, acc.v[2])};
                if (a.thermo) {  // Homogeneous.cpp:139-145, then calcFM's own sum
                    const double w = a.thermo[kThermoW * cell_replica(a.R, cell) + kThVi];
                    for (int k = 0; k < 3; ++k) vv[k] = __dadd_rn(vv[k], w);
                }
                S.Vx[i] = vv[0];
                S.Vy[i] = vv[1];
                S.Vz[i] = vv[2];
                if constexpr (TI >= T_D) {
                    S.Mx[i] = acc.m[0]; S.My[i] = acc.m[1]; S.Mz[i] = acc.m[2];
                }
            }
            wmac[0] += acc.u;
            wmac[2] += acc.rf;
        }
    }
    // zero rows (the sums of the work item's cells go to one row at the end)
    if (lane == 0 && !a.accumulate)
        for (int k = 0; k < 4 * span; ++k) a.macro_part[4 * (size_t)cell + k] = 0.0;
    return !empty;
}

// The per-lane sums of a group of cells of one replica into the row of the
// group's last non-empty cell.
template <int TI>
__device__ __forceinline__ void flush_macro(const PairArgs &a, double (&wmac)[3], int cell,
                                            int lane) {
    // the reaction-field sum (wmac[2]) is non-zero only for dipole i sites
    for (int k = 0; k < (TI == T_D ? 3 : 2); ++k)
        for (int o = 32; o > 0; o >>= 1) wmac[k] += shfl_xor_d(wmac[k], o);
    if (lane == 0) {
        double *o = a.macro_part + 4 * (size_t)cell;
        const double v[4] = {(TI == T_LJ) ? wmac[0] : 0.0, (TI == T_LJ) ? 0.0 : wmac[0], wmac[1],
                             wmac[2]};
        for (int k = 0; k < 4; ++k) o[k] = a.accumulate ? o[k] + v[k] : v[k];
    }
    wmac[0] = wmac[1] = wmac[2] = 0.0;
}

// One 64-lane block (one wavefront) per work item of cpb consecutive cells.
// XCD-aware: hardware block b runs on XCD b % 8, and XCD x owns the
// contiguous item range [x, x + 1) * items_per_xcd, so neighbouring cells
// share its L2. A grid smaller than 8 * items_per_xcd makes the blocks
// persistent: each walks its XCD's items with stride gridDim.x / 8, and every
// block leaves after its last item.
template <int TI, typename R, bool COUNT, bool MOLSITE, bool MULTI>
__global__ __launch_bounds__(64) __attribute__((
    amdgpu_waves_per_eu(TileCfg<TI, R, MOLSITE, MULTI>::WAVES))) void k_pairs(PairArgs a) {
    __shared__ Tile<TI, R, MOLSITE, MULTI> T;
    const int lane = threadIdx.x;
    const int xcd = blockIdx.x & 7, stride = gridDim.x >> 3;
    unsigned long long ntest = 0;
    for (int item = blockIdx.x >> 3; item < a.items_per_xcd; item += stride) {
        const int c0 = (xcd * a.items_per_xcd + item) * a.cpb;
        const int c1 = min(c0 + a.cpb, a.ncell);
        double wmac[3] = {0.0, 0.0, 0.0};
        int last = -1, rep_prev = -1;
        for (int cell = c0; cell < c1;) {
            const int rep = cell_replica(a.R, cell);
            if (a.others && a.R.geom[rep].small) {  // the block kernels'
                ++cell;
                continue;
            }
            if (rep != rep_prev && last >= 0) {  // rows never mix replicas
                flush_macro<TI>(a, wmac, last, lane);
                last = -1;
            }
            rep_prev = rep;
            int span = 1;
            if constexpr (TileCfg<TI, R, MOLSITE, MULTI>::JOINT) {
                // pairs of cells in one x row of one replica, where the cell
                // edge exceeds the cutoff: the 9 cells of the common
                // neighbourhood that are not neighbours of one of the two are
                // then at least a cell edge, more than rc, from its sites, so
                // testing them adds no pair that ls1's traversal leaves out.
                // The cells 0 and 1, 2 and 3, ... of a row go together wherever
                // the row lies in the launch (the item that holds the first one
                // takes both), so a replica gives the bits that it gives alone
                const Geom &g = a.R.geom[rep];
                const int x = (cell - a.R.cell_off[rep]) % g.n[0];
                const double rc2 = TI == T_LJ ? a.rclj2 : a.rc2;
                if (g.cl[0] * g.cl[0] > rc2 * (1.0 + 1e-9)) {
                    if (x & 1) {
                        ++cell;
                        continue;
                    }
                    if (x + 1 < g.n[0]) span = 2;
                }
            }
            if (pair_cell<TI, R, COUNT, MOLSITE, MULTI>(a, T, cell, span, lane, ntest, wmac))
                last = cell + span - 1;
            cell += span;
        }
        if (last >= 0) flush_macro<TI>(a, wmac, last, lane);
    }
    if (COUNT) {
        for (int o = 32; o > 0; o >>= 1) ntest += __shfl_xor(ntest, o, 64);
        if (lane == 0) atomicAdd(&a.counters[0], ntest);
    }
}

// The cell pairs of the traversal on ls1's halo-extended grid: thread
// (cell, k) emits (ls1 index of cell, ls1 index of its neighbour k), i.e. the
// halo cell when the neighbour is a periodic image; -1 when the neighbour
// does not exist (open boundaries).
__global__ void k_enum_pairs(Geom g, int ncell, int *out) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)ncell * 27) return;
    int c = (int)(t / 27), k = (int)(t % 27);
    int cx = c % g.n[0], cy = (c / g.n[0]) % g.n[1], cz = c / (g.n[0] * g.n[1]);
    Nbr b = neighbour(g, cx, cy, cz, k);
    int e1 = ((cz + 1) * g.cpd[1] + (cy + 1)) * g.cpd[0] + (cx + 1);
    int e2 = ((cz + 1 + b.dd[2]) * g.cpd[1] + (cy + 1 + b.dd[1])) * g.cpd[0] + (cx + 1 + b.dd[0]);
    out[2 * t] = b.ok ? e1 : -1;
    out[2 * t + 1] = b.ok ? e2 : -1;
}

// Host-side launcher table (the molecule-centre and several-type variants are
// LJ's only).
template <int T, typename R, bool C> PairKernel pick(bool molsite, bool multi) {
    if constexpr (T == T_LJ) {
        if (molsite) return multi ? k_pairs<T, R, C, true, true> : k_pairs<T, R, C, true, false>;
        if (multi) return k_pairs<T, R, C, false, true>;
    }
    return k_pairs<T, R, C, false, false>;
}

template <int T> PairKernel pick_t(bool fp32, bool count, bool molsite, bool multi) {
    if (fp32) return count ? pick<T, float, true>(molsite, multi) : pick<T, float, false>(molsite, multi);
    return count ? pick<T, double, true>(molsite, multi) : pick<T, double, false>(molsite, multi);
}

PairKernel pair_kernel(int ti, bool fp32, bool count, bool molsite, bool multi) {
    switch (ti) {
    case T_LJ: return pick_t<T_LJ>(fp32, count, molsite, multi);
    case T_C: return pick_t<T_C>(fp32, count, false, false);
    case T_D: return pick_t<T_D>(fp32, count, false, false);
    case T_Q: return pick_t<T_Q>(fp32, count, false, false);
    }
    return nullptr;
}

}  // namespace mdx
