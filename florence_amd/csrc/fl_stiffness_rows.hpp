// The direct scatter of tensor-product hexes: the factorised stiffness straight into the CSR
// (included by fl_assemble.hip).  Same contraction as stiffness_sf_mfma2_kernel (see
// fl_stiffness_sf.hpp), but one workgroup forms the three blocks (i, 0), (i, 1), (i, 2) of an
// element together and stores each entry's three column components side by side.
//
// The launch covers the elements elist[0, n) of one colour: no two of them share a node, so
// no two workgroups of the launch write one entry, and the launches run in colour order on
// one stream.  scat (sf_scatter_index's order, the order this kernel stores in) holds
// each entry's column block in its row, with the sign bit set where an element of an
// earlier colour holds both nodes: that entry is added to, the others are stored as
// 0.0 + value.  Every CSR entry is the sum of its elements' contributions in colour order.
//
// What bounds it: the writes of scattered parts of cache lines.  With every block (i, k) in a
// workgroup of its own, an entry's 8 B went out alone and the lines were completed, if at
// all, by other workgroups at other times: 1.75 times V's bytes written at p = 3, and each
// block built the tables and read the scatter entries anew.  Three components at once are 24 B
// a store, 1.29 times V's bytes.  With the stores to scattered addresses replaced by
// contiguous ones p = 3, 17^3 takes 496 us instead of 862, with none 462; p = 4, 16^3 takes
// 1864 and 1745 instead of 2613.
// Time of the stiffness phase, blocks apart -> together (us): p = 1, 20^3 202 -> 109; p = 2,
// 25^3 1046 -> 780; p = 3, 10^3 224 -> 193, 17^3 999 -> 862; p = 4, 4^3 221 -> 147,
// 16^3 3003 -> 2613; in FP32 p = 4, 16^3 1980 -> 1548.
#pragma once

namespace fl {

// SW waves share a slice az.  SW = 1 (WAVE): a workgroup of P1 waves, each with a slice and its
// own part of LDS to itself, so that no barrier follows the loads.  SW > 1: the waves share
// out the eta tiles and the column tiles, and the slices follow one another in ng workgroups:
// all of them in one, one in each of P1, or two in each but the last (the caller's rule).
template <int P1, int Q, int SW, int OCC, typename CT, typename VT>
__global__ __launch_bounds__(SW == 1 ? 64 * P1 : 64 * SW, OCC) void stiffness_rows_kernel(
    const double *__restrict__ qp, const int32_t *__restrict__ basis, int64_t n, VT *__restrict__ V,
    const int32_t *__restrict__ elist, const int32_t *__restrict__ elements, const int32_t *__restrict__ indptr,
    const int16_t *__restrict__ scat, int ng) {
    typedef SfLayout<P1, Q> L;
    typedef Mfma16<CT> MF;
    // output rows of the beta product (and the scatter table's order): the FP64 MFMA's, rows
    // lk + 4 r.  CT = float feeds the A rows of each tile permuted, i -> (i >> 2) + 4 (i & 3),
    // so that the FP32 MFMA's rows 4 lk + r come out as the same rows.
    typedef Mfma16<double> MO;
    constexpr bool F64 = sizeof(CT) == 8;
    static_assert(!F64 || sizeof(VT) == 8, "FP64 blocks go to an FP64 CSR");
    constexpr int Q3 = L::Q3, N3 = L::N3, PP = L::PP, QQ = Q * Q;
    constexpr bool WAVE = SW == 1;
    constexpr int NT = WAVE ? 64 * P1 : 64 * SW;
    constexpr int MT = (PP + 15) / 16, NT2 = (P1 * Q + 15) / 16, NT3 = (N3 + 15) / 16;
    constexpr int TW = (NT3 + SW - 1) / SW, KB = (2 * Q + 3) / 4;
    static_assert(MT * NT2 <= SW, "one eta tile per wave");
    // waves enough: a wave takes one of a tile's two types, else both
    constexpr bool ONE = 2 * MT * NT2 <= SW;
    typedef short TV __attribute__((ext_vector_type(MT * 4)));
    typedef VT V2 __attribute__((ext_vector_type(2), aligned(sizeof(VT))));
    // pair products of the 1D bases: zeta [s*2+t][az][bz][qz] = T0^s[az][qz] T0^t[bz][qz], eta
    // [s*2+t][ae*P1+be][qe] likewise; the beta ones live in registers
    __shared__ CT sPz[4][P1][P1][Q];
    __shared__ CT sPe[4][PP][Q];
    __shared__ CT sC[27][Q3];
    __shared__ CT sT1_[WAVE ? P1 : 1][9][P1][QQ];
    __shared__ CT sT2_[WAVE ? P1 : 1][2][PP][P1][Q];
    __shared__ int32_t sRow[N3];
    // tensor point of record point g: needed only before the first eta writes sT2
    int16_t *sTg = reinterpret_cast<int16_t *>(&sT2_[0][0][0][0][0]);
    static_assert(sizeof(int16_t) * Q3 <= sizeof(sT2_), "sTg in sT2's space");

    const int64_t wid = blockIdx.x;
    const int64_t slot = wid >> 3;
    const int sub = (int)(slot % (3 * ng));
    const int64_t idx = (slot / (3 * ng)) * 8 + (wid & 7);   // an element's workgroups on one XCD
    if (idx >= n) return;
    const int64_t e = elist[idx];
    const int pi = sub % 3;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int32_t *g_of_t = basis + 4;
    const double *f1d = reinterpret_cast<const double *>(basis + L::INTS);
    // table entries are clamped into range: a table that does not match the launch shape
    // gives wrong values, never an access outside the arrays
    for (int t = tid; t < Q3; t += NT) sTg[min(max(g_of_t[t], 0), Q3 - 1)] = (int16_t)t;
    {
        const int32_t *loc = basis + 4 + Q3, *conn = elements + e * N3;
        for (int t = tid; t < N3; t += NT) sRow[t] = indptr[3 * (int64_t)conn[min(max(loc[t], 0), N3 - 1)] + pi];
    }
    for (int t = tid; t < 4 * PP * Q; t += NT) {
        const int st = t / (PP * Q), r = t - st * (PP * Q);
        const int a = r / (P1 * Q), b = (r / Q) % P1, q = r % Q;
        const int s0 = st >> 1, t0 = st & 1;
        (&sPz[0][0][0][0])[t] = (CT)(f1d[(s0 * P1 + a) * Q + q] * f1d[(t0 * P1 + b) * Q + q]);
        (&sPe[0][0][0])[t] = (CT)(f1d[((2 + s0) * P1 + a) * Q + q] * f1d[((2 + t0) * P1 + b) * Q + q]);
    }
    // this lane's beta A fragments: phase h, step ks, row tile tm -> T2^h[ab][qb] T2^tl[bb][qb]
    CT afr[2][KB][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int ks = 0; ks < KB; ++ks) {
            const int kk = ks * 4 + lk;
            const bool kv = kk < 2 * Q;
            const int tl = kv ? kk / Q : 0, qb = kv ? kk - (kk / Q) * Q : 0;
#pragma unroll
            for (int tm = 0; tm < MT; ++tm) {
                const int arow = tm * 16 + (F64 ? li : (li >> 2) + 4 * (li & 3));
                const int ab_ = min(arow / P1, P1 - 1), bb_ = arow % P1;
                afr[h][ks][tm] = (kv && arow < PP)
                                     ? (CT)(f1d[((4 + h) * P1 + ab_) * Q + qb] * f1d[((4 + tl) * P1 + bb_) * Q + qb])
                                     : CT(0);
            }
        }
    __syncthreads();
    // the point tensors C^{ik} of the three blocks, read point by point (coalesced), kept in
    // tensor point order; C^{ki} = (C^{ik})^T
    {
        const double *rec = qp + e * (int64_t)Q3 * QS + (int64_t)Q_D * Q3;   // field f of point g at rec[f Q3 + g]
        for (int g = tid; g < Q3; g += NT) {
            const int t = sTg[g];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int sp = pi == k ? pi : (pi + k == 1 ? 3 : (pi + k == 2 ? 4 : 5));
                const bool tr = pi > k;
#pragma unroll
                for (int m = 0; m < 3; ++m)
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        sC[9 * k + 3 * m + c][t] = (CT)rec[(9 * sp + (tr ? 3 * c + m : 3 * m + c)) * Q3 + g];
            }
        }
    }
    __syncthreads();

    // one wave's or the workgroup's stages follow one another
    const auto sync = [] {
        if constexpr (WAVE) {
            // a wave's LDS accesses are in order; the fence keeps the compiler's
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    };
    auto &sT1 = sT1_[WAVE ? wave : 0];
    auto &sT2 = sT2_[WAVE ? wave : 0];
    const int sw = WAVE ? 0 : wave, zid = WAVE ? lane : tid;
    // this wave's eta tile, its row and column
    const int etile = ONE ? sw >> 1 : sw, etm = etile / NT2, etn = etile - etm * NT2;
    const bool eta_wave = etile < MT * NT2;
    const int arow = etm * 16 + li, ecol = etn * 16 + li;
    const bool av = arow < PP, ev = ecol < P1 * Q;
    const int arc = av ? arow : 0, ecc = ev ? ecol : 0;
    const int ebz = ecc / Q, eqb = ecc - ebz * Q;   // bz, qb of the column
    const int nz = WAVE || ng == P1 ? 1 : (ng == 1 ? P1 : 2);   // a workgroup's slices
    const int z0 = WAVE ? wave : sub / 3 * nz, z1 = min(z0 + nz, P1);
    for (int az = z0; az < z1; ++az) {
        // the slice's scatter entries: lane's rows (tm, r) of column tile sw + SW v
        TV tv[TW];
#pragma unroll
        for (int v = 0; v < TW; ++v)
            tv[v] = sw + SW * v < NT3
                        ? *reinterpret_cast<const TV *>(scat + sf_scatter_index(P1, e, az, sw + SW * v, lane, 0, 0))
                        : TV{};
        typename MF::acc_t acc[3][TW][MT];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            // zeta (VALU): task (mn, qe qb) holds its Q tensor values and sweeps bz
            int zt = zid;
            // one round of tasks: without this the compiler keeps the indices of all three blocks over
            // the kernel, and Q = 5 spills six registers instead of two (16^3 2890 -> 2780 us; where
            // there are two rounds, as at Q = 6, or registers to spare it costs 1 to 4 %)
            if constexpr (F64 && MT > 1 && 9 * QQ <= 64 * SW) asm volatile("" : "+v"(zt));
            for (int t = zt; t < 9 * QQ; t += 64 * SW) {
                const int mn = t / QQ, qeb = t - mn * QQ;   // qeb = qb * Q + qe
                const int m = mn / 3, c = mn - 3 * m;
                const int qb = qeb / Q, qe = qeb - qb * Q;
                const CT *cp = sC[9 * k + mn] + qeb * Q;
                const CT *f = sPz[(m == 0) * 2 + (c == 0)][az][0];
                CT cv[Q];
#pragma unroll
                for (int qz = 0; qz < Q; ++qz) cv[qz] = cp[qz];
#pragma unroll
                for (int bz = 0; bz < P1; ++bz) {
                    CT x = CT(0);
#pragma unroll
                    for (int qz = 0; qz < Q; ++qz) x += f[bz * Q + qz] * cv[qz];
                    sT1[mn][bz][qe * Q + qb] = x;
                }
            }
            sync();
#pragma unroll
            for (int v = 0; v < TW; ++v)
#pragma unroll
                for (int tm = 0; tm < MT; ++tm) acc[k][v][tm] = typename MF::acc_t{CT(0), CT(0), CT(0), CT(0)};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // eta (MFMA) for the phase's two types (m's beta factor h, n's tl): rows (ae,be),
                // columns (bz,qb), K = (m, n, qe)
                if (eta_wave) {
                    const CT *t1 = &sT1[0][0][0] + ebz * QQ + eqb;
                    // one type's operands of step ks: clamped loads, zeroed by a select where K or
                    // the tile pads
                    const auto operands = [&](int tl, int ks, CT &a, CT &b) {
                        const int nn = tl ? 1 : 2, ke = (h ? 1 : 2) * nn * Q;
                        const int kk = ks * 4 + lk;
                        const bool kv = ks * 4 + 3 < ke || kk < ke;
                        const int kc = min(kk, ke - 1);
                        const int pr = kc / Q, qe = kc - pr * Q;
                        const int m = h ? 2 : pr / nn, c = tl ? 2 : pr % nn;
                        const CT x = sPe[(m == 1) * 2 + (c == 1)][arc][qe];
                        const CT y = t1[(3 * m + c) * P1 * QQ + qe * Q];
                        a = (kv && av) ? x : CT(0);
                        b = (kv && ev) ? y : CT(0);
                    };
                    const auto store = [&](int tl, const typename MF::acc_t &d) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int row = etm * 16 + MF::row(lk, r);
                            if (row < PP && ev) sT2[tl][row][ebz][eqb] = d[r];
                        }
                    };
                    constexpr int K0[2] = {(4 * Q + 3) / 4, (2 * Q + 3) / 4}, K1[2] = {(2 * Q + 3) / 4, (Q + 3) / 4};
                    typename MF::acc_t d0 = {CT(0), CT(0), CT(0), CT(0)}, d1 = d0;
                    CT a, b;
                    if constexpr (ONE) {
                        if (sw & 1) {
#pragma unroll
                            for (int ks = 0; ks < K1[h]; ++ks) {
                                operands(1, ks, a, b);
                                d1 = MF::step(a, b, d1);
                            }
                            store(1, d1);
                        } else {
#pragma unroll
                            for (int ks = 0; ks < K0[h]; ++ks) {
                                operands(0, ks, a, b);
                                d0 = MF::step(a, b, d0);
                            }
                            store(0, d0);
                        }
                    } else {
#pragma unroll
                        for (int ks = 0; ks < K0[h]; ++ks) {
                            operands(0, ks, a, b);
                            d0 = MF::step(a, b, d0);
                            if (ks < K1[h]) {
                                operands(1, ks, a, b);
                                d1 = MF::step(a, b, d1);
                            }
                        }
                        store(0, d0);
                        store(1, d1);
                    }
                }
                sync();
                // beta (MFMA): rows (ab,bb), columns (ae,be,bz), K = (tl, qb)
#pragma unroll
                for (int ks = 0; ks < KB; ++ks) {
                    const int kk = ks * 4 + lk;
                    const bool kv = ks * 4 + 3 < 2 * Q || kk < 2 * Q;
                    const int kc = min(kk, 2 * Q - 1);
                    const int tl = kc / Q, qb = kc - tl * Q;
                    CT bf[TW];
#pragma unroll
                    for (int v = 0; v < TW; ++v) {
                        const int bcol = (sw + SW * v) * 16 + li, bc = min(bcol, N3 - 1);
                        const CT x = sT2[tl][bc / P1][bc % P1][qb];
                        bf[v] = (kv && bcol < N3) ? x : CT(0);
                    }
#pragma unroll
                    for (int v = 0; v < TW; ++v)
#pragma unroll
                        for (int tm = 0; tm < MT; ++tm)
                            if (sw + SW * v < NT3) acc[k][v][tm] = MF::step(afr[h][ks][tm], bf[v], acc[k][v][tm]);
                }
                // the next phase's eta rewrites sT2; the next block's zeta only rewrites sT1,
                // whose last reads precede the sync after this phase's eta
                if (h == 0 || WAVE) sync();
            }
        }
        // CSR positions and, where an earlier colour has written, the values to add to: every
        // load before the first store (stores count in the same memory counter, and a load
        // issued after one waits for it)
        int32_t off[TW][MT][4];
        VT out[3][TW][MT][4];
#pragma unroll
        for (int v = 0; v < TW; ++v) {
            const int bcol = (sw + SW * v) * 16 + li, ae_ = min(bcol, N3 - 1) / PP;
#pragma unroll
            for (int tm = 0; tm < MT; ++tm)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = min(tm * 16 + MO::row(lk, r), PP - 1);
                    const int ta = ((row / P1) * P1 + ae_) * P1 + az;
                    const int sv = tv[v][tm * 4 + r];
                    off[v][tm][r] = sRow[ta] + 3 * (sv & 0x7fff);
                    const bool live = sw + SW * v < NT3 && bcol < N3 && tm * 16 + MO::row(lk, r) < PP;
                    VT p[3] = {VT(0), VT(0), VT(0)};
                    if (live && sv < 0) {
#pragma unroll
                        for (int k = 0; k < 3; ++k) p[k] = V[off[v][tm][r] + k];
                    }
#pragma unroll
                    for (int k = 0; k < 3; ++k) out[k][v][tm][r] = (VT)(p[k] + acc[k][v][tm][r]);
                }
        }
        // vmcnt(0) on every path (expcnt and lgkmcnt left open): no load is still counted when
        // the next slice starts, so the waits placed there do not also wait for these stores
        __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
        for (int v = 0; v < TW; ++v) {
            const int bcol = (sw + SW * v) * 16 + li;
            if (sw + SW * v < NT3 && bcol < N3) {
#pragma unroll
                for (int tm = 0; tm < MT; ++tm)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int rlo = tm * 16 + 4 * r;
                        const int row = tm * 16 + MO::row(lk, r);
                        if (rlo < PP && (rlo + 3 < PP || row < PP)) {
                            VT *dst = V + off[v][tm][r];
                            *reinterpret_cast<V2 *>(dst) = V2{out[0][v][tm][r], out[1][v][tm][r]};
                            dst[2] = out[2][v][tm][r];
                        }
                    }
            }
        }
    }
}

}  // namespace fl
