// Phase 2 for elements of few nodes (the tets of p <= 4): the dense contraction of
// fl_stiffness.hpp with an element to a workgroup (included by fl_assemble.hip).
//
// One wave per displacement block pair i <= k.  All six share G_{a,(g,j)} = dN_a/dx_j, which is
// built once in LDS for every point (no chunks, one barrier), and each forms its operand
// W^{ik}_{b,(g,j)} = sum_l D^{ik}_{jl}(g) G_{b,(g,l)} on the fly.  A workgroup a pair built G six
// times, in chunks of 8 points with a barrier each.
//
// The npe x npe block is MT x MT tiles of 16 x 16 and, with REM, up to four rows and columns
// more, for which 4 x 4 x 4 MFMAs in four blocks take the places of padded tiles: the
// operand of the 16 columns is the one the full tiles use, the other one is four rows,
// the same in every block.  35 nodes: 4 x 64 + 5 x 16 cycles a step instead of 9 x 64.  A
// diagonal pair's block is symmetric: tiles below the diagonal and the columns beyond MT tiles
// are stored from their mirror.
//
// Time of the stiffness phase, a workgroup a pair -> an element (us; elements): 4 nodes, 1
// point (24,576) 101 -> 58; 10 nodes, 8 points (3,072) 24 -> 23, (24,576) 128 -> 113; 20 nodes,
// 14 points (3,072) 73 -> 39; 35 nodes, 31 points (4,374) 341 -> 202, of which its MFMAs take 73
// at the card's rate and the 386 MB of blocks 80.
#pragma once

namespace fl {

template <int MT, bool REM>
struct ElLayout {
    static constexpr int NR = 16 * MT + (REM ? 4 : 0);
    // row stride of G: the four rows of an operand read start 8 or 16 doubles apart (mod 32)
    static constexpr int LDA = REM ? NR + 4 : NR;
    static constexpr int TT = 16 * 17;   // a wave's transpose tile
    // LDS of one element: G [3 G + 3][LDA], the last point's rows 0, and D [6][K][3], K = 3 G
    // rounded up to 4
    static size_t lds(int G) {
        const size_t K = (3 * (size_t)G + 3) / 4 * 4, n = (3 * (size_t)G + 3) * LDA + 18 * K;
        return sizeof(double) * (n > 6 * TT ? n : 6 * TT);
    }
};

template <int MT, bool REM>
__global__ __launch_bounds__(384, 4) void stiffness_el_kernel(const double *__restrict__ JmT, int NP,
                                                              const double *__restrict__ qp, int npe, int G,
                                                              int64_t nelem, double *__restrict__ Ke) {
    typedef ElLayout<MT, REM> L;
    typedef Mfma16<double> MF;
    constexpr int NR = L::NR, LDA = L::LDA;
    extern __shared__ double dsm[];
    const int K = (3 * G + 3) / 4 * 4;
    double *sA = dsm, *sD = dsm + (3 * G + 3) * LDA;
    const int64_t e = blockIdx.x;
    if (e >= nelem) return;
    const int tid = threadIdx.x;
    const int pair = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const double *qe = qp + e * (int64_t)G * QS;
    for (int t = tid; t < G * NR; t += 384) {
        const int g = t / NR, a = t - g * NR;
        const double *jt = JmT + (int64_t)g * 3 * NP + a;
        const double j0 = jt[0], j1 = jt[NP], j2 = jt[2 * NP];   // 0 for a >= npe
        const double *ix = qe + (int64_t)Q_IX * G + g;
#pragma unroll
        for (int j = 0; j < 3; ++j)
            sA[(3 * g + j) * LDA + a] = ix[(3 * j) * G] * j0 + ix[(3 * j + 1) * G] * j1 + ix[(3 * j + 2) * G] * j2;
    }
    // D[pair][(g, j)][l]
    for (int t = tid; t < 54 * G; t += 384) {
        const int f = t / G, g = t - f * G, p = f / 9, jl = f - 9 * p;
        sD[(p * K + 3 * g) * 3 + jl] = qe[(int64_t)(Q_D + f) * G + g];
    }
    for (int t = tid; t < 3 * LDA; t += 384) sA[3 * G * LDA + t] = 0.0;
    for (int t = tid; t < (K - 3 * G) * 18; t += 384)
        sD[((t / 3 % 6) * K + 3 * G + t / 18) * 3 + t % 3] = 0.0;
    __syncthreads();

    const int pi = c_pair_i[pair], pk = c_pair_k[pair];
    const bool diag = pair < 3;
    typename MF::acc_t acc[MT][MT];
    double rrow[MT], rcol[MT], rcc = 0.0;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        rrow[m] = rcol[m] = 0.0;
#pragma unroll
        for (int n = 0; n < MT; ++n) acc[m][n] = typename MF::acc_t{0, 0, 0, 0};
    }
    const double *D = sD + pair * K * 3;
    const int l4 = 16 * MT + (li & 3);
    const auto contract = [&](auto sym) {
        constexpr bool SYM = decltype(sym)::value;
#pragma unroll 2
        for (int q = lk; q < K; q += 4) {
            const double d0 = D[3 * q], d1 = D[3 * q + 1], d2 = D[3 * q + 2];
            const double *A = sA + q * LDA, *Gb = sA + q / 3 * 3 * LDA;
            double af[MT], bf[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) af[m] = A[m * 16 + li];
#pragma unroll
            for (int n = 0; n < MT; ++n) {
                const int b = n * 16 + li;
                bf[n] = d0 * Gb[b] + d1 * Gb[LDA + b] + d2 * Gb[2 * LDA + b];
            }
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < MT; ++n)
                    if (!SYM || m <= n) acc[m][n] = MF::step(af[m], bf[n], acc[m][n]);
            if constexpr (REM) {
                const double ar = A[l4], br = d0 * Gb[l4] + d1 * Gb[LDA + l4] + d2 * Gb[2 * LDA + l4];
#pragma unroll
                for (int n = 0; n < MT; ++n) {
                    rrow[n] = __builtin_amdgcn_mfma_f64_4x4x4f64(ar, bf[n], rrow[n], 0, 0, 0);
                    if (!SYM) rcol[n] = __builtin_amdgcn_mfma_f64_4x4x4f64(br, af[n], rcol[n], 0, 0, 0);
                }
                rcc = __builtin_amdgcn_mfma_f64_4x4x4f64(ar, br, rcc, 0, 0, 0);
            }
        }
    };
    if (diag) contract(std::true_type());
    else contract(std::false_type());

    // rows a, columns b of block (i, k) and its transpose, block (k, i); a full tile's
    // transpose through LDS, for whole-line stores
    const int64_t npe2 = (int64_t)npe * npe;
    double *Kd = Ke + (e * 9 + pi * 3 + pk) * npe2, *Kt = Ke + (e * 9 + pk * 3 + pi) * npe2;
    __syncthreads();   // sA and sD are read; the transpose tiles take their place
    double *tile = dsm + pair * L::TT;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < MT; ++n) {
            if (diag && m > n) continue;
            const int b = n * 16 + li;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int a = m * 16 + MF::row(lk, r);
                if (a < npe && b < npe) Kd[(int64_t)a * npe + b] = acc[m][n][r];
            }
            if (diag && m == n) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) tile[li * 17 + MF::row(lk, r)] = acc[m][n][r];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int bl = 4 * r + lk, a = m * 16 + li;
                if (a < npe && n * 16 + bl < npe) Kt[(int64_t)(n * 16 + bl) * npe + a] = tile[bl * 17 + li];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    if constexpr (REM) {
        // output of the 4 x 4 x 4 MFMA: row lane / 16 of column lane % 16 (four blocks of four)
        const int a4 = 16 * MT + lk;
#pragma unroll
        for (int n = 0; n < MT; ++n) {
            const int c = n * 16 + li;
            if (a4 < npe) {
                Kd[(int64_t)a4 * npe + c] = rrow[n];
                Kt[(int64_t)c * npe + a4] = rrow[n];
                if (!diag) {
                    Kd[(int64_t)c * npe + a4] = rcol[n];
                    Kt[(int64_t)a4 * npe + c] = rcol[n];
                }
            }
        }
        if (li < 4 && a4 < npe && l4 < npe) {
            Kd[(int64_t)a4 * npe + l4] = rcc;
            if (!diag) Kt[(int64_t)l4 * npe + a4] = rcc;
        }
    }
}

}  // namespace fl
