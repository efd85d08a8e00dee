// The assembled tangent applied element by element from the point records, for the
// multigrid's fine-level smoother (included by fl_assemble.hip, which owns the record
// layout; the per-node sums are in fl_mg.hip).
//
// For a tensor-product hex with the factorised path's records (the C tensors, detJ and
// the point weight included),
//     y_{a,i} = sum_q sum_m dN_a/dxi_m(q) S_{im}(q),
//     S_{im}  = sum_{k,n} C^{ik}_{mn}(q) G_{kn}(q),   G_{kn} = sum_b dN_b/dxi_n(q) x_{b,k},
// contracted one direction at a time with SfLines (gradients of x's three components at the
// points, and back to the nodes).
// About 124 kflop per p = 4 element, and the 54 C values per point read once (K_e itself
// is 140,625 doubles).  Each XCD takes a contiguous range of elements (its L2 then holds the x
// of neighbouring elements).
#pragma once

namespace fl {

// CK: 0 the FP64 records, 1 their FP32 copy, 2 their BF16 copy (c32 [e][54][Q3], c16
// [e][27][Q3], two values a word).  The copy's values are loaded after B: loaded when the
// workgroup starts they delay x (18.7 -> 21.1 us).  Bound by the latency of its eight stages: 1,728
// elements of 125 nodes and 6^3 points, BF16, are 6.75 elements a CU, five at a time, each
// about 10 us; the bytes (40 MB of C, 12 of vectors) take 10 us.  Before SfLines, with the 1D
// basis and both buffers in LDS, 25.0 us; now 18.7.  Two points a thread and twice the
// elements in flight: 21.2.
template <int P1, int Q, int CK>
__global__ __launch_bounds__((SfLines<P1, Q, 3>::NT), CK == 1 ? 4 : 5) void mf_element_kernel(
    const double *__restrict__ qp, const float *__restrict__ c32, const uint32_t *__restrict__ c16,
    const int32_t *__restrict__ basis, const int32_t *__restrict__ elements, int64_t nelem,
    const uint8_t *__restrict__ free_mask, const double *__restrict__ x, double *__restrict__ ye) {
    typedef SfLines<P1, Q, 3> C;
    constexpr int Q3 = C::Q3, N3 = C::N3, EPB = C::EPB, NT = C::NT;
    __shared__ double sFb[2][P1][Q];
    __shared__ double sAP[C::LDS];

    const int64_t chunk = ((nelem + EPB - 1) / EPB + 7) / 8;
    const int64_t k8 = blockIdx.x >> 3;
    const int64_t e0 = ((int64_t)(blockIdx.x & 7) * chunk + k8) * EPB;
    const int ne = (int)min((int64_t)EPB, nelem - e0);
    if (k8 >= chunk || ne <= 0) return;
    const int tid = threadIdx.x;
    const int32_t *g_of_t = basis + 4;
    const int32_t *loc = basis + 4 + Q3;
    const double *f1d = reinterpret_cast<const double *>(basis + SfLayout<P1, Q>::INTS);
    const C c = {f1d, loc, ne, tid, __builtin_amdgcn_readfirstlane(tid >> 6), tid & 63, sAP, sAP};
    // this thread's point: table entries are clamped into range
    const int pel = tid / Q3, u = tid - pel * Q3;
    const bool valid = pel < ne;
    const int cel = valid ? pel : 0;
    const int64_t e = e0 + cel;
    const int g = min(max(g_of_t[C::point(u)], 0), Q3 - 1);
    for (int t = tid; t < 2 * P1 * Q; t += NT) (&sFb[0][0][0])[t] = f1d[4 * P1 * Q + t];
    for (int t = tid; t < ne * N3; t += NT) {
        const int el = EPB == 1 ? 0 : t / N3, tn = t - el * N3;
        const int64_t a = elements[(e0 + el) * N3 + min(max(loc[tn], 0), N3 - 1)];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double xv = x[3 * a + k];   // read either way: one latency, not two
            *c.x(el, k, tn) = free_mask[3 * a + k] ? xv : 0.0;
        }
    }
    __syncthreads();
    c.form_A();
    __syncthreads();
    c.form_B(0);
    // the point's values of a rounded copy, in flight over the gradient
    float cr[CK == 1 ? 54 : 1];
    uint32_t cw[CK == 2 ? 27 : 1];
    if constexpr (CK == 1) {
#pragma unroll
        for (int f = 0; f < 54; ++f) cr[f] = c32[(e * 54 + f) * Q3 + g];
    } else if constexpr (CK == 2) {
#pragma unroll
        for (int f = 0; f < 27; ++f) cw[f] = c16[(e * 27 + f) * Q3 + g];
    }
    __syncthreads();
    double G[9], S[9];   // G[3 n + k], S[3 m + i]
    c.gradient(sFb, cel, u, G);
    __syncthreads();   // B's reads
    // S_im = sum_kn C^{ik}_mn G_kn.  The record holds C^{ik} of the six pairs i <= k (0,0 1,1 2,2 0,1
    // 0,2 1,2); C^{ki}_mn = C^{ik}_nm.
    const double *rec = qp + e * (int64_t)QS * Q3 + (int64_t)Q_D * Q3 + g;
    const auto field = [&](int f) -> double {
        if constexpr (CK == 1) return (double)cr[f];
        else if constexpr (CK == 2) return (double)__uint_as_float(f & 1 ? cw[f >> 1] & 0xFFFF0000u : cw[f >> 1] << 16);
        else return rec[(int64_t)f * Q3];
    };
#pragma unroll
    for (int q = 0; q < 9; ++q) S[q] = 0.0;
#pragma unroll
    for (int p = 0; p < 6; ++p) {
        const int i = p < 3 ? p : (p == 5 ? 1 : 0), k = p < 3 ? p : (p == 3 ? 1 : 2);
        double cv[9];
#pragma unroll
        for (int mn = 0; mn < 9; ++mn) cv[mn] = field(9 * p + mn);
#pragma unroll
        for (int m = 0; m < 3; ++m)
            S[3 * m + i] += cv[3 * m] * G[k] + cv[3 * m + 1] * G[3 + k] + cv[3 * m + 2] * G[6 + k];
        if (i != k) {
#pragma unroll
            for (int m = 0; m < 3; ++m) S[3 * m + k] += cv[m] * G[i] + cv[3 + m] * G[3 + i] + cv[6 + m] * G[6 + i];
        }
    }
    if (valid) c.put_point(pel, C::point(u), S);
    __syncthreads();
    c.to_nodes(e0, ye, elements, nullptr, nullptr);
}

// c32[e][f][g] = (float) records' C field f at point g (f < 54)
__global__ __launch_bounds__(256) void mf_round_kernel(const double *__restrict__ qp, int G, int64_t n,
                                                       float *__restrict__ c32) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t per = (int64_t)54 * G;
    const int64_t e = i / per, r = i - e * per;
    c32[i] = (float)qp[e * (int64_t)QS * G + (int64_t)Q_D * G + r];
}

// c16[e][j][g] = bf16(C field 2j) | bf16(C field 2j+1) << 16, rounded to nearest even
__device__ inline uint32_t to_bf16_bits(double v) {
    const uint32_t u = __float_as_uint((float)v);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__global__ __launch_bounds__(256) void mf_round16_kernel(const double *__restrict__ qp, int G, int64_t n,
                                                         uint32_t *__restrict__ c16) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t per = (int64_t)27 * G;
    const int64_t e = i / per, r = i - e * per;
    const int64_t j = r / G, g = r - j * G;
    const double *rec = qp + e * (int64_t)QS * G + (int64_t)Q_D * G;
    c16[i] = to_bf16_bits(rec[(2 * j) * G + g]) | (to_bf16_bits(rec[(2 * j + 1) * G + g]) << 16);
}

}  // namespace fl
