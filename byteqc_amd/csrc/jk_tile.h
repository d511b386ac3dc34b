// Row kernel with its exchange block in LDS: the FP64 kernel of the classes up
// to 324 components except (ff|ps), the larger ones in parts (tile_parts).
//
// As in jk_rows a wavefront owns 64 pairs (a b) of the P list and walks a
// range of the Q list in lock-step, and the six digestion sums are the same.
// Up to 64 Q pairs are taken at a time; the distinct shells a, b of the lanes
// are the rows and the distinct shells c, d of those Q pairs the columns of a
// dense block of K in LDS, into which the lanes add K(a,d), K(b,d) at every
// step and K(a,c), K(b,c) at the end of a run of equal c.  The block goes to
// global memory once per 64 Q pairs (fewer where the block is full).  J(c,d)
// is summed over the wavefront, kept by the lane that holds the Q pair and
// added with the block.
//
// What this replaces: global FP64 atomics take one request per 64-byte segment
// and instruction, 2.4e10 a second on MI355X, and jk_rows issues 26-35 of them
// per step (64 quartets).  An LDS add of 64 doubles takes 9 cycles of its CU
// when no two of 16 neighbouring lanes hit one bank (44 with four equal
// addresses, hence the order of the lanes below).  Per build, jk_rows ->
// jk_tile (ms): 64 waters cc-pVDZ (ps|ps) 18.4 -> 8.6, (ss|ss) 14.8 -> 8.9,
// (ps|ss) 17.4 -> 14.2, all classes 110.6 -> 86.7; 24 waters cc-pVTZ (ps|ss)
// 7.9 -> 3.0, (fs|ss) 3.2 -> 1.0, all classes 172 -> 138; 12 molecules
// def2-SVP all classes 227 -> 187 (86.7, 138 and 187 are 73.9, 100.6 and 141.8
// with the steps noted below).  What is left of (ps|ss) at 64 waters, from
// variants that skip a part: integrals 4 ms, the block's atomics 2.7, J 1.8,
// density gathers 1.2, item set-up 4.3; in batches of def2-SVP molecules the
// integrals of the contracted shells are 3/4 of the time.
#pragma once
#include "jk_v2.h"

// Parts that the Cartesian components of shell a of class code c are dealt
// into, each part an item of its own (0: no tile kernel).  The blocks of the
// larger classes do not fit the 512 registers of a lane; a part's does, at the
// price of its recurrences being evaluated once per part.  All digestion sums
// are linear in the components of a, so a part is a shell with fewer
// components.  Measured on MI355X (24 waters cc-pVTZ, ms, one block or the
// wavefront kernel -> parts): two parts (dp|pp) 9.9 -> 2.9 (12 molecules
// def2-SVP 21.3 -> 6.3), (dp|ds) 5.8 -> 2.7, (dd|ps) 4.8 -> 1.9, (fp|ps) 2.9 ->
// 1.7, (ff|ss) 2.4 -> 0.8, (fs|fs) 2.3 -> 0.4, (fs|pp) 1.5 -> 1.0, (fd|ss) 1.4
// -> 0.9, (fs|ds) 1.4 -> 1.0; five (fs|dp) 4.1 -> 2.1, (fp|ds) 4.1 -> 1.8,
// (fd|ps) 3.7 -> 1.9, (fp|pp) 3.5 -> 1.9, (fp|fs) 1.8 -> 1.0; six (dp|dp) 7.5 ->
// 4.0, (dd|ds) 3.9 -> 2.4, (dd|pp) 3.3 -> 2.4.  Not so (dd|dp) 4.0 -> 8.0,
// (fd|ds) 2.3 -> 3.5, (fd|pp) 2.1 -> 2.3, and hardly (fp|dp) 4.4 -> 3.6,
// (fs|dd) 1.4 -> 1.2, (ff|ps) 1.4 -> 1.1 (5 waters 0.20 -> 0.28, 0.11 -> 0.24).
constexpr int tile_parts(int c) {
    switch (c) {
        case 2111: case 2120: case 2210: case 3011: case 3110: case 3300: case 3030: case 3020:
        case 3200:
            return 2;
        case 3021: case 3120: case 3210: case 3111: case 3130:
            return 5;
        case 2121: case 2211: case 2220:
            return 6;
    }
    return ncart(c / 1000) * ncart(c / 100 % 10) * ncart(c / 10 % 10) * ncart(c % 10) <= 81 ? 1 : 0;
}
template <int LA, int LB, int LC, int LD>
constexpr int tile_parts() { return tile_parts(LA * 1000 + LB * 100 + LC * 10 + LD); }

template <int LA, int LB, int LC, int LD>
struct TileCls {
    using C = Cls<LA, LB, LC, LD>;
    static constexpr int PARTS = tile_parts<LA, LB, LC, LD>() > 0 ? tile_parts<LA, LB, LC, LD>() : 1;
    static constexpr int NA = C::NFI / PARTS, NB = C::NFJ, NC = C::NFK, ND = C::NFL;
    static constexpr int NF = NA * NB * NC * ND;
    // resident wavefronts per SIMD, and so workgroups per CU: what registers
    // allow with few spills.  (pp|ps) runs 20.3 ms with one and no spills, 15.8
    // with two and 95 spilled registers, 12.6 with what RELOAD and DIRECT below
    // spare (12 molecules def2-SVP); (ps|ss) 27.6 with two, 24.2 with three.
    static constexpr int WAVES = NF <= 3 ? 3 : (NF <= 27 ? 2 : 1);
    // Values a lane holds beside the integrals' temporaries: D and J of (a,b),
    // the accumulators and densities of a c-run, D of d, J(c,d), the block.
    // Where they take over 0.6 of the registers (512 / WAVES of 32 bits), the
    // accumulators and densities were spilled and reloaded around every
    // block, to scratch far beyond the L2: (pp|ps) moved 35 GB in 7.9 ms for
    // 64 waters cc-pVDZ.  RELOAD: the densities D(b,c), D(a,c) are read at
    // every step instead of once per c-run.  DIRECT: K(a,c), K(b,c) are added
    // to the LDS block at every step instead of accumulating over the run,
    // which pays at two waves where the additions are fewer than the
    // components.  Held / RELOAD / DIRECT too (ms, 12 molecules def2-SVP):
    // (pp|ps) 16.0 / 14.4 / 12.6, (dp|ss) 4.9 / 4.4 / 4.1, (ds|ps) 9.3 / 7.9 /
    // 8.4, (pp|pp) 6.4 / 5.9 / 6.6, (dp|ps) 8.3 / 8.1 / 7.9; below the line
    // (ds|pp) 4.7 / 4.9 / 4.8, (ds|ds) 2.1 / 2.1 / 2.3.
    static constexpr int LIVE =
        2 * NA * NB + 2 * (NA + NB) * NC + (NA + NB) * ND + NC * ND + NF;
    static constexpr bool RELOAD = LIVE * WAVES > 153;
    static constexpr bool DIRECT = RELOAD && WAVES == 2 && (NA + NB) * NC < NF;
    // doubles of LDS per wavefront for the block of K: what WAVES workgroups
    // per CU leave of 160 KB after the Rys table and the row and column lists
    static constexpr int CAP = (163840 / WAVES - rys_lds_size(C::NR) * 8 -
                                4 * 64 * (NA + NB + NC + ND) * 2 - 64) / 32 / 2 * 2;
    // lanes with all different a and b and one Q pair fit (odd row length):
    // 64 of them, or in the larger classes 32 (the lanes take turns)
    static constexpr bool ALL_FIT = 64 * (NA + NB) * ((NC + ND) | 1) <= CAP;
    static constexpr bool FITS = 32 * (NA + NB) * ((NC + ND) | 1) <= CAP;
};

// Position of this lane's key among the distinct keys of the lanes in mask,
// in ascending order; n: number of distinct keys.
__device__ __forceinline__ int distinct_rank(int key, unsigned long long mask, int &n) {
    int rank = 0;
    n = 0;
    while (mask) {
        const int v = __builtin_amdgcn_readlane(key, __builtin_ctzll(mask));
        mask &= ~__ballot(key == v);
        rank += v < key;
        ++n;
    }
    return rank;
}

// Lanes of mask whose key no lower lane of mask has.
__device__ __forceinline__ unsigned long long distinct_firsts(int key, unsigned long long mask) {
    unsigned long long firsts = 0;
    while (mask) {
        const int lead = __builtin_ctzll(mask);
        firsts |= 1ull << lead;
        mask &= ~__ballot(key == __builtin_amdgcn_readlane(key, lead));
    }
    return firsts;
}

// f(0), f(1), ... f(N - 1) with compile-time arguments.
template <int N, int I = 0, typename F>
__device__ __forceinline__ void each_part(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        each_part<N, I + 1>(f);
    }
}

__device__ __forceinline__ void lds_add(double *p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(256, (TileCls<LA, LB, LC, LD>::WAVES))
    jk_tile(const TaskDesc *__restrict__ tasks, const int4 *__restrict__ items, int nitems,
            int *ticket) {
    using TC = TileCls<LA, LB, LC, LD>;
    using C = typename TC::C;
    constexpr int NA = TC::NA, NB = TC::NB, NC = TC::NC, ND = TC::ND;
    __shared__ __align__(16) double rys_lds[rys_lds_size(C::NR)];
    __shared__ __align__(16) double tile_all[4 * TC::CAP];
    __shared__ unsigned short row_all[4 * 64 * (NA + NB)], col_all[4 * 64 * (NC + ND)];
    rys_stage<C::NR, 256>(rys_lds);
    __syncthreads();
    const rys_lds_ptr rys_tab = (rys_lds_ptr)rys_lds;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double *const tile = tile_all + wave * TC::CAP;
    unsigned short *const row_ao = row_all + wave * 64 * (NA + NB);
    unsigned short *const col_ao = col_all + wave * 64 * (NC + ND);
    // records of the gathered Q pairs, in the block's memory before it is set
    int *const recs = (int *)tile;

    auto run_item = [&](const int4 it, auto part_c) {
        constexpr int X0 = decltype(part_c)::value * NA;  // first component of a
        const TaskDesc &tk = tasks[__builtin_amdgcn_readfirstlane(it.x)];
        const PairData &pd = tk.pd;
        const int chunk = __builtin_amdgcn_readfirstlane(it.y & BQC_PART_MASK);
        const int q0 = __builtin_amdgcn_readfirstlane(it.z);
        const int qe = __builtin_amdgcn_readfirstlane(it.w);
        // neighbours in the list (which share a) sit 16 lanes apart: one LDS
        // add serves 16 lanes at a time, and equal addresses among them wait
        const int pidx = chunk * 64 + ((lane & 15) << 2 | lane >> 4);
        bool pvalid = pidx < tk.np;
        int qlim = 0, ppos = 0;
        if (pvalid) {
            int s = 0;
            while (s < tk.nbins && pidx >= tk.pbins[s + 1]) ++s;
            qlim = tk.qbins[tk.nbins - s];
            ppos = glb(tk.perm_p)[pidx];
        }
        // Q pairs any lane needs: those below the lanes' largest limit, and in
        // a task of a pair type with itself not beyond the largest own position
        int qlim_max = qlim;
        if (tk.diag) qlim_max = min(qlim, ppos + 1);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) qlim_max = max(qlim_max, __shfl_xor(qlim_max, d, 64));
        qlim_max = __builtin_amdgcn_readfirstlane(qlim_max);
        const int q1 = min(qe, tk.qbins[tk.nbins]);

        const gptr<int> lbra = glb(pd.bra), lket = glb(pd.ket), lao = glb(pd.ao_loc);
        const gptr<double> lbx = glb(pd.bas_x), lby = glb(pd.bas_y), lbz = glb(pd.bas_z);
        const cptr<double> ubx = cst(pd.bas_x), uby = cst(pd.bas_y), ubz = cst(pd.bas_z);
        const int gp = tk.bas_p0 + ppos;
        const int sa = pvalid ? lbra[gp] : -1;
        const int sb = pvalid ? lket[gp] : -1;
        const int pp0 = tk.prim_p0 + ppos * tk.nprim_p;
        int a0 = 0, b0 = 0;
        double ra[3] = {0, 0, 0}, rb[3] = {0, 0, 0};
        double p_first[5] = {1, 0, 0, 0, 0};
        if (pvalid) {
            a0 = lao[sa] + X0;
            b0 = lao[sb];
            ra[0] = lbx[sa]; ra[1] = lby[sa]; ra[2] = lbz[sa];
            rb[0] = lbx[sb]; rb[1] = lby[sb]; rb[2] = lbz[sb];
            if (pd.prec) {
#pragma unroll
                for (int k = 0; k < 5; ++k) p_first[k] = glb(pd.prec)[(size_t)pp0 * BQC_PREC + k];
            } else {
                p_first[0] = glb(pd.a12)[pp0]; p_first[1] = glb(pd.e12)[pp0];
                p_first[2] = glb(pd.x12)[pp0]; p_first[3] = glb(pd.y12)[pp0];
                p_first[4] = glb(pd.z12)[pp0];
            }
        }
        // rows of the block: NA per distinct a, then NB per distinct b.  If
        // they leave no room for the columns of one Q pair, the lanes take
        // turns by halves.
        const unsigned long long pall = __ballot(pvalid);
        int ua, ub;
        int la = distinct_rank(sa, pall, ua), lb = distinct_rank(sb, pall, ub);
        const bool halves = !TC::ALL_FIT && (NA * ua + NB * ub) * ((NC + ND) | 1) > TC::CAP;
        for (int part = 0; part < (halves ? 2 : 1); ++part) {
        if (halves) {
            const unsigned long long half = pall & (part ? ~0ull << 32 : ~0ull >> 32);
            la = distinct_rank(sa, half, ua);
            lb = distinct_rank(sb, half, ub);
            pvalid = half >> lane & 1;
        }
        const int R = NA * ua + NB * ub;
        const int row_a = NA * la, row_b = NA * ua + NB * lb;
        if (pvalid) {
#pragma unroll
            for (int x = 0; x < NA; ++x) row_ao[row_a + x] = a0 + x;
#pragma unroll
            for (int y = 0; y < NB; ++y) row_ao[row_b + y] = b0 + y;
        }

        const int nao = tk.nao;
        const size_t nao2 = (size_t)nao * nao;
        const bool do_j = tk.vj != nullptr, do_k = tk.vk != nullptr;
        for (int idm = 0; idm < tk.n_dm; ++idm) {
            const gptr<double> D = glb(tk.dm + idm * nao2);
            const cptr<double> DU = cst(tk.dm + idm * nao2);
            gdouble *VJ = do_j ? glb_rw(tk.vj + idm * nao2) : nullptr;
            gdouble *VK = do_k ? glb_rw(tk.vk + idm * nao2) : nullptr;
            double dab[NA * NB], jab[NA * NB];
#pragma unroll
            for (int x = 0; x < NA; ++x)
#pragma unroll
                for (int y = 0; y < NB; ++y) {
                    dab[x * NB + y] = pvalid ? D[(a0 + x) * nao + b0 + y] : 0.0;
                    jab[x * NB + y] = 0.0;
                }
            int pos = q0;
            for (;;) {
                // the next (up to 64) Q pairs below the limit, one per lane
                int left = 0;
                while (pos < q1 && left < 64) {
                    int4 r = {0x7fffffff, -1, -1, 0};
                    if (pos + lane < q1) {
                        const gptr<int> g = glb(tk.qrec) + 4 * (pos + lane);
                        r = make_int4(g[0], g[1], g[2], g[3]);
                    }
                    unsigned long long keep = __ballot(r.x < qlim_max);
                    int adv = 64;
                    const int room = 64 - left;
                    if (__popcll(keep) > room) {  // take the first `room` of them
                        const bool over =
                            r.x < qlim_max && __popcll(keep & ((1ull << lane) - 1)) == room;
                        adv = __builtin_ctzll(__ballot(over));
                        keep &= (1ull << adv) - 1;
                    }
                    if (keep >> lane & 1)
                        *(int4 *)(recs + 4 * (left + __popcll(keep & ((1ull << lane) - 1)))) = r;
                    left += __popcll(keep);
                    pos += adv;
                }
                if (!left) break;
                wave_sync();
                const int4 rec4 = *(const int4 *)(recs + 4 * lane);
                wave_sync();
                // plan position, shells, AO offsets (16 bits each)
                const int qp = rec4.x, shells = (rec4.y & 0xffff) | rec4.z << 16, aos = rec4.w;
                // columns of the block, and the Q pairs whose columns fit it
                // (at least one does; the others wait for the next block)
                unsigned long long qmask = ~0ull >> (64 - left);
                int first = 0;
                while (first < left) {
                unsigned long long seg_mask = qmask & (~0ull << first);
                int uc, ud;
                const int key_c = shells & 0xffff, key_d = (int)((unsigned)shells >> 16);
                int lc = distinct_rank(key_c, seg_mask, uc), ld = distinct_rank(key_d, seg_mask, ud);
                int end = left;
                if (R * ((NC * uc + ND * ud) | 1) > TC::CAP) {
                    const unsigned long long fc = distinct_firsts(key_c, seg_mask),
                                             fd = distinct_firsts(key_d, seg_mask);
                    const unsigned long long upto = ~0ull >> (63 - lane);
                    const int cols = NC * __popcll(fc & upto) + ND * __popcll(fd & upto);
                    const unsigned long long over = __ballot(R * (cols | 1) > TC::CAP) & seg_mask;
                    end = __builtin_ctzll(over);
                    seg_mask &= (1ull << end) - 1;
                    lc = distinct_rank(key_c, seg_mask, uc);
                    ld = distinct_rank(key_d, seg_mask, ud);
                }
                const int ncol = NC * uc + ND * ud, ldt = ncol | 1;
                // first columns of c and d (16 bits each)
                const int cols_cd = NC * lc | (NC * uc + ND * ld) << 16;
                if (do_k) {
                    if (seg_mask >> lane & 1) {
                        const int col_c = cols_cd & 0xffff, col_d = (int)((unsigned)cols_cd >> 16);
                        const int c0l = aos & 0xffff, d0l = (int)((unsigned)aos >> 16);
#pragma unroll
                        for (int z = 0; z < NC; ++z) col_ao[col_c + z] = c0l + z;
#pragma unroll
                        for (int w = 0; w < ND; ++w) col_ao[col_d + w] = d0l + w;
                    }
                    for (int e = lane; e < R * ldt; e += 64) tile[e] = 0.0;
                    wave_sync();
                }
                double *const ta = tile + row_a * ldt, *const tb = tile + row_b * ldt;
                double jcd[NC * ND], kac[NA * NC], kbc[NB * NC], dbc[NB * NC], dac[NA * NC];
#pragma unroll
                for (int k = 0; k < NC * ND; ++k) jcd[k] = 0.0;
#pragma unroll
                for (int k = 0; k < NA * NC; ++k) kac[k] = dac[k] = 0.0;
#pragma unroll
                for (int k = 0; k < NB * NC; ++k) kbc[k] = dbc[k] = 0.0;
                auto load_c = [&](int c0) {
#pragma unroll
                    for (int z = 0; z < NC; ++z) {
#pragma unroll
                        for (int y = 0; y < NB; ++y) dbc[y * NC + z] = D[(c0 + z) * nao + b0 + y];
#pragma unroll
                        for (int x = 0; x < NA; ++x) dac[x * NC + z] = D[(c0 + z) * nao + a0 + x];
                    }
                };
                auto flush_c = [&](int col) {
#pragma unroll
                    for (int z = 0; z < NC; ++z) {
#pragma unroll
                        for (int x = 0; x < NA; ++x) {
                            if (pvalid) lds_add(ta + x * ldt + col + z, kac[x * NC + z]);
                            kac[x * NC + z] = 0.0;
                        }
#pragma unroll
                        for (int y = 0; y < NB; ++y) {
                            if (pvalid) lds_add(tb + y * ldt + col + z, kbc[y * NC + z]);
                            kbc[y * NC + z] = 0.0;
                        }
                    }
                };
                int ccol = -1;
                for (int i = first; i < end; ++i) {
                    const int qpos = __builtin_amdgcn_readlane(qp, i);
                    bool active = pvalid && qpos < qlim;
                    double norm = TWO_PI_52;
                    if (tk.diag) {
                        active = active && ppos >= qpos;
                        if (ppos == qpos) norm *= 0.5;
                    }
                    if (!__ballot(active)) continue;
                    const int scd = __builtin_amdgcn_readlane(shells, i);
                    const int sc = scd & 0xffff, sd = (int)((unsigned)scd >> 16);
                    const int cd0 = __builtin_amdgcn_readlane(aos, i);
                    const int c0 = cd0 & 0xffff, d0 = (int)((unsigned)cd0 >> 16);
                    const int ccd = __builtin_amdgcn_readlane(cols_cd, i);
                    const int colc = ccd & 0xffff, cold = (int)((unsigned)ccd >> 16);
                    // densities, in flight while the block is computed
                    double dbd[NB * ND], dad[NA * ND];
                    if (do_k) {
#pragma unroll
                        for (int w = 0; w < ND; ++w) {
#pragma unroll
                            for (int y = 0; y < NB; ++y) dbd[y * ND + w] = D[(d0 + w) * nao + b0 + y];
#pragma unroll
                            for (int x = 0; x < NA; ++x) dad[x * ND + w] = D[(d0 + w) * nao + a0 + x];
                        }
                        if (colc != ccol) {
                            if (!TC::DIRECT && ccol >= 0) flush_c(ccol);
                            ccol = colc;
                            if (!TC::RELOAD) load_c(c0);
                        }
                    }
                    double g[TC::NF];
                    if (active) {
                        const int qq0 =
                            __builtin_amdgcn_readfirstlane(tk.prim_q0 + qpos * tk.nprim_q);
                        const double rc[3] = {ubx[sc], uby[sc], ubz[sc]};
                        const double rd[3] = {ubx[sd], uby[sd], ubz[sd]};
                        eri_block<LA, LB, LC, LD, double, NA, rys_lds_ptr, true>(
                            g, pd, pp0, tk.nprim_p, qq0, tk.nprim_q, norm, ra, rb, rc, rd, X0,
                            rys_tab, p_first);
                    } else {
#pragma unroll
                        for (int k = 0; k < TC::NF; ++k) g[k] = 0.0;
                    }
#define G(x, y, z, w) g[(((x) * NB + (y)) * NC + (z)) * ND + (w)]
                    if (do_j) {
#pragma unroll
                        for (int z = 0; z < NC; ++z)
#pragma unroll
                            for (int w = 0; w < ND; ++w) {
                                const double dcd = DU[(c0 + z) * nao + d0 + w];
                                double s = 0.0;
#pragma unroll
                                for (int x = 0; x < NA; ++x)
#pragma unroll
                                    for (int y = 0; y < NB; ++y) {
                                        jab[x * NB + y] += G(x, y, z, w) * dcd;
                                        s += G(x, y, z, w) * dab[x * NB + y];
                                    }
                                s = wave_sum63(s);
                                // lane i keeps the sum of its Q pair
                                const int lo = __builtin_amdgcn_readlane(__double2loint(s), 63);
                                const int hi = __builtin_amdgcn_readlane(__double2hiint(s), 63);
                                if (lane == i) jcd[z * ND + w] = __hiloint2double(hi, lo);
                            }
                    }
                    if (do_k) {
                        if (TC::RELOAD) load_c(c0);
#pragma unroll
                        for (int x = 0; x < NA; ++x)
#pragma unroll
                            for (int y = 0; y < NB; ++y)
#pragma unroll
                                for (int z = 0; z < NC; ++z)
#pragma unroll
                                    for (int w = 0; w < ND; ++w) {
                                        const double v = G(x, y, z, w);
                                        kac[x * NC + z] += v * dbd[y * ND + w];
                                        kbc[y * NC + z] += v * dad[x * ND + w];
                                    }
                        if (TC::DIRECT) flush_c(colc);
#pragma unroll
                        for (int w = 0; w < ND; ++w) {
#pragma unroll
                            for (int x = 0; x < NA; ++x) {
                                double s = 0.0;
#pragma unroll
                                for (int y = 0; y < NB; ++y)
#pragma unroll
                                    for (int z = 0; z < NC; ++z) s += G(x, y, z, w) * dbc[y * NC + z];
                                if (active) lds_add(ta + x * ldt + cold + w, s);
                            }
#pragma unroll
                            for (int y = 0; y < NB; ++y) {
                                double s = 0.0;
#pragma unroll
                                for (int x = 0; x < NA; ++x)
#pragma unroll
                                    for (int z = 0; z < NC; ++z) s += G(x, y, z, w) * dac[x * NC + z];
                                if (active) lds_add(tb + y * ldt + cold + w, s);
                            }
                        }
                    }
#undef G
                }
                if (do_k) {
                    if (!TC::DIRECT && ccol >= 0) flush_c(ccol);
                    wave_sync();
                    // consecutive rows are often consecutive functions, so an
                    // instruction's lanes share 64-byte segments
                    for (int row = lane; row < R; row += 64) {
                        gdouble *const v = VK + row_ao[row];
                        for (int col = 0; col < ncol; ++col) {
                            const double t = tile[row * ldt + col];
                            if (t != 0.0) atomic_add(v + col_ao[col] * nao, t);
                        }
                    }
                    wave_sync();
                }
                if (do_j && (seg_mask >> lane & 1)) {
                    const int c0l = aos & 0xffff, d0l = (int)((unsigned)aos >> 16);
#pragma unroll
                    for (int z = 0; z < NC; ++z)
#pragma unroll
                        for (int w = 0; w < ND; ++w)
                            if (jcd[z * ND + w] != 0.0)
                                atomic_add(VJ + (c0l + z) * nao + d0l + w, jcd[z * ND + w]);
                }
                first = end;
                }
                wave_sync();
            }
            if (do_j && pvalid) {
#pragma unroll
                for (int x = 0; x < NA; ++x)
#pragma unroll
                    for (int y = 0; y < NB; ++y)
                        if (jab[x * NB + y] != 0.0)
                            atomic_add(VJ + (a0 + x) * nao + b0 + y, jab[x * NB + y]);
            }
        }
        }
    };
    ItemQueue queue(ticket, nitems);
    for (int item = queue.next(); item < nitems; item = queue.next()) {
        const int4 it = items[item];
        const int part = __builtin_amdgcn_readfirstlane((unsigned)it.y >> BQC_PART_SHIFT);
        each_part<TC::PARTS>([&](auto c) {
            if (part == decltype(c)::value) run_item(it, c);
        });
    }
}

// Classes with a tile instance.
template <int LA, int LB, int LC, int LD>
constexpr bool use_tile() {
    if constexpr (tile_parts<LA, LB, LC, LD>() > 0) return TileCls<LA, LB, LC, LD>::FITS;
    return false;
}

template <int LA, int LB, int LC, int LD>
static void reg_row(RowKernelTable &tab) {
    constexpr int pab = LA * (LA + 1) / 2 + LB, pcd = LC * (LC + 1) / 2 + LD;
    static_assert(use_tile<LA, LB, LC, LD>() || Cls<LA, LB, LC, LD>::NF > 81,
                  "the wave kernels start above 81 components");
    if constexpr (use_tile<LA, LB, LC, LD>()) {
        static_assert(ncart(LA) % tile_parts<LA, LB, LC, LD>() == 0, "parts of equal size");
        tab[0][pab][pcd] = jk_tile<LA, LB, LC, LD>;
    }
    if constexpr (row_split_candidate<LA, LB, LC, LD>()) {
        tab[1][pab][pcd] = jk_rows<LA, LB, LC, LD, 1>;
        tab[2][pab][pcd] = jk_rows<LA, LB, LC, LD, 2>;
    }
}
