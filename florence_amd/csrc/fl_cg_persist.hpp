// Block-Jacobi CG of the masked operator as one launch, for matrices small enough to live
// in the registers of the whole chip (included by fl_solve.hip and fl_mg.hip).
//
// A CG step of four launches (product, alpha, update, beta) takes 20 us on the 8^3 tet p=2
// cube (14.7k dofs, 9 MB of values) whatever the arithmetic: 16 us inside kernels that
// mostly wait for memory and 4 us between them, and the host looks in every few steps;
// here a step takes 6.0 us, and the 60 of the multigrid's coarsest level on the 12^3 cube
// 288 us against 640 in two launches each.  What remains is two trips through memory.
// Here every workgroup owns a contiguous range of nodes (about equal numbers of 3x3
// blocks), each thread keeps K of the range's blocks in registers for the whole solve, and
// the range's r, z, p, q, x and block inverses stay in LDS.  A step meets twice:
//
//   A(k)  q = A p on the own rows, partial p.q;       all read every partial: alpha
//   B(k)  x, r, z = P r on the own rows, partial r.z, r.r;  all read: beta, the exit test
//
// Meeting and summing are one memory round trip: each workgroup stores its partial into
// its slot, every workgroup polls all slots until none is empty and adds them in the
// same fixed order, so all hold the same alpha and beta and leave in the same step, and a
// solve is bitwise reproducible.  An empty slot holds a signalling NaN, which no
// arithmetic produces.  Slots alternate between two sets: a workgroup empties its A slot
// of step k once it passed B(k+1) (everyone has read it) and its B slots of step k once it
// passed A(k), and each emptying store is complete before the workgroup stores the
// partial that lets the others go on to poll that slot again.  z travels the same way,
// through two buffers whose values say by themselves that they have arrived, so no store
// is waited for before a partial announces it: z(k) is emptied past A(k), when everyone
// has read it, and that is complete before A(k+1), the last meeting before z(k+2) is
// looked for.  All of it at agent scope: the XCDs' L2s do not see each other's writes.
//
// All workgroups must be resident at once: at most one per CU is launched, a process's
// launches on one device follow one another (PersistentTurn), and every wait is bounded: a
// workgroup that waits longer than wait_ticks raises the abort flag and returns, the others
// follow, and the caller solves with the launch-per-step form.  x is undefined then: where
// the wait that runs out is one for the last meeting, others have passed it and written
// their part.  The caller reads b again, so it must not take this form where b is x.
#pragma once
#include <algorithm>

#include "fl_common.hpp"

namespace fl {
namespace {

constexpr int CGP_T = 512;        // threads per workgroup
constexpr int CGP_MAXW = 256;     // workgroups at most (one per slot thread)
constexpr int CGP_MAXK = 5;       // 3x3 blocks per thread at most (90 registers of FP64 values)
constexpr uint64_t CGP_EMPTY = 0xFFF4DEADBEEF0001ull;
constexpr int CGP_SLOTS = 6 * CGP_MAXW;             // one set: [parity][p.q, r.z, r.r][workgroup]
constexpr long long CGP_WAIT_TICKS = 100000000ll;   // 1 s of the 100 MHz wall clock

struct CgpPlan {
    int nw = 0, K = 0;
    int64_t total = 0;
    size_t lds = 0;
};

template <typename VT>
struct CgpArgs {
    const int32_t *indptr, *nbr_ptr, *nbrs;
    const VT *V;
    int64_t nnode, total;
    const uint8_t *free_mask;
    const double *P, *b;
    double *x, *z[2];
    uint64_t *slots, *slots_next;   // this launch's set (empty), and the set it empties for the next launch
    int32_t *abort;
    double *out;                    // iterations, relative residual (or NULL)
    int nw, maxit, check_every;
    double rtol;
    long long wait_ticks;
};

__device__ __forceinline__ double cgp_load(const double *p) {
    return __longlong_as_double((long long)__hip_atomic_load(reinterpret_cast<const uint64_t *>(p), __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void cgp_store(double *p, double v) {
    __hip_atomic_store(reinterpret_cast<uint64_t *>(p), (uint64_t)__double_as_longlong(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
// this wave's stores have reached the agent's coherence point
__device__ __forceinline__ void cgp_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_moved(double v) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, ROWS, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// sum over the wave, in every lane, by register moves between lanes (a shuffle through
// LDS costs over a hundred cycles a step, six of them four times a CG step)
__device__ __forceinline__ double dpp_wave_sum(double v) {
    v += dpp_moved<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8: lane 15 of each row holds the row's sum
    v += dpp_moved<0x112, 0xf>(v);
    v += dpp_moved<0x114, 0xf>(v);
    v += dpp_moved<0x118, 0xf>(v);
    v += dpp_moved<0x142, 0xa>(v);   // row_bcast 15, 31: lane 63 holds the wave's
    v += dpp_moved<0x143, 0xc>(v);
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)u, 63), hi = __builtin_amdgcn_readlane((int)(u >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// sum over eight consecutive lanes, in every lane
__device__ __forceinline__ double dpp_sum8(double v) {
    v += dpp_moved<0xB1, 0xf>(v);    // quad_perm 1 0 3 2
    v += dpp_moved<0x4E, 0xf>(v);    // quad_perm 2 3 0 1
    v += dpp_moved<0x141, 0xf>(v);   // row_half_mirror
    return v;
}

// o[0] = largest, o[1] = 2^30 - smallest neighbour count, o[2] = total (o zeroed before)
__global__ __launch_bounds__(256) void cgp_degree_kernel(const int32_t *__restrict__ nbr_ptr, int64_t nnode,
                                                         int32_t *__restrict__ o) {
    const int64_t a = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int mx = 0, mn = 0;
    if (a < nnode) {
        const int d = nbr_ptr[a + 1] - nbr_ptr[a];
        mx = d;
        mn = (1 << 30) - d;
        if (a == 0) o[2] = nbr_ptr[nnode];
    }
    for (int off = 32; off > 0; off >>= 1) {
        mx = max(mx, __shfl_xor(mx, off, 64));
        mn = max(mn, __shfl_xor(mn, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(o, mx);
        atomicMax(o + 1, mn);
    }
}

__global__ __launch_bounds__(256) void cgp_empty_kernel(uint64_t *__restrict__ slots, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) slots[i] = CGP_EMPTY;
}

// first node whose list starts at or after block t
__device__ inline int cgp_first_node(const int32_t *__restrict__ nbr_ptr, int64_t nnode, int64_t t) {
    int64_t lo = 0, hi = nnode;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (nbr_ptr[mid] < t) lo = mid + 1; else hi = mid;
    }
    return (int)lo;
}

// LDS of nown nodes and K blocks per thread: products | r z p q x [3] P [9] d [3] | list starts, masks
constexpr int CGP_NODE_DOUBLES = 27;
static size_t cgp_lds(int K, int64_t nown) {
    return 8 * ((size_t)3 * CGP_T * K + (size_t)CGP_NODE_DOUBLES * nown) + 4 * (2 * (size_t)nown + 2);
}

// Polls slot `mine` (lanes without one pass active = false); false when the wait ran out.
__device__ __forceinline__ bool cgp_wait(const uint64_t *mine, bool active, const int32_t *abort, long long ticks,
                                         double &v) {
    v = 0.0;
    if (!active) return true;
    const long long t0 = wall_clock64();
    for (int spin = 1;; ++spin) {
        const uint64_t u = __hip_atomic_load(mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (u != CGP_EMPTY) {
            v = __longlong_as_double((long long)u);
            return ticks >= 0;
        }
        if ((spin & 15) == 0 && (wall_clock64() - t0 > ticks ||
                                 __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
            return false;
    }
}

// As cgp_wait, and with z given also the values of the thread's neighbours in it, asked
// for again with every poll until none is empty.
template <int K>
__device__ __forceinline__ bool cgp_wait_z(const uint64_t *mine, bool active, const double *z, const int32_t (&nb)[K],
                                           const bool (&act)[K], const int32_t *abort, long long ticks, double &v,
                                           double (&xz)[K][3]) {
    const long long t0 = wall_clock64();
    bool missing = z != nullptr;
    for (int spin = 1;; ++spin) {
        const uint64_t u = active ? __hip_atomic_load(mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
        if (missing) {
            bool miss = false;
#pragma unroll
            for (int j = 0; j < K; ++j)
#pragma unroll
                for (int c = 0; c < 3; ++c) xz[j][c] = act[j] ? cgp_load(z + nb[j] + c) : 0.0;
#pragma unroll
            for (int j = 0; j < K; ++j)
#pragma unroll
                for (int c = 0; c < 3; ++c) miss |= (uint64_t)__double_as_longlong(xz[j][c]) == CGP_EMPTY;
            missing = __any(miss);
        }
        if (!missing && __all(u != CGP_EMPTY)) {
            v = __longlong_as_double((long long)u);
            return ticks >= 0;
        }
        if ((spin & 15) == 0 && (wall_clock64() - t0 > ticks ||
                                 __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
            v = 0.0;
            return false;
        }
    }
}

template <typename VT, int K>
__global__ __launch_bounds__(CGP_T) void cg_persistent_kernel(CgpArgs<VT> A) {
    extern __shared__ double sm[];
    __shared__ double sw[CGP_T / 64], sw2[CGP_T / 64];
    __shared__ int srange[2];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, w = blockIdx.x;
    if (lane == 0 && wave < 2) {
        const int64_t t = (A.total * (w + wave) + A.nw - 1) / A.nw;
        srange[wave] = w + wave == A.nw ? (int)A.nnode : cgp_first_node(A.nbr_ptr, A.nnode, t);
    }
    if (tid < 6) A.slots_next[tid * CGP_MAXW + w] = CGP_EMPTY;
    __syncthreads();
    const int a0 = srange[0], nown = srange[1] - a0;
    const int32_t blk0 = A.nbr_ptr[a0];
    double *sr = sm + 3 * CGP_T * K, *sz = sr + 3 * nown, *sp = sz + 3 * nown, *sq = sp + 3 * nown,
           *sx = sq + 3 * nown, *sP = sx + 3 * nown, *sd = sP + 9 * nown;
    int32_t *sptr = reinterpret_cast<int32_t *>(sd + 3 * nown), *smask = sptr + nown + 1;
    for (int i = tid; i <= nown; i += CGP_T) sptr[i] = A.nbr_ptr[a0 + i] - blk0;
    __syncthreads();
    const int nblk = sptr[nown];
    // the range's start vectors: x = 0, r = b (masked), z = P r
    double rz = 0.0, rr = 0.0;
    if (tid < nown) {
        const int64_t a = a0 + tid;
        int m = 0;
        double rv[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const bool fr = !A.free_mask || A.free_mask[3 * a + i] != 0;
            m |= fr ? 1 << i : 0;
            rv[i] = fr ? A.b[3 * a + i] : 0.0;
            sr[3 * tid + i] = rv[i];
            sx[3 * tid + i] = 0.0;
            sp[3 * tid + i] = 0.0;
        }
        smask[tid] = m;
#pragma unroll
        for (int i = 0; i < 9; ++i) sP[9 * tid + i] = A.P[9 * a + i];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double zi = sP[9 * tid + 3 * i] * rv[0] + sP[9 * tid + 3 * i + 1] * rv[1] +
                              sP[9 * tid + 3 * i + 2] * rv[2];
            sz[3 * tid + i] = zi;
            cgp_store(A.z[0] + 3 * a + i, zi);
            cgp_store(A.z[1] + 3 * a + i, __longlong_as_double((long long)CGP_EMPTY));
            rz += rv[i] * zi;
            rr += rv[i] * rv[i];
        }
        sd[tid] = rz;
        sd[nown + tid] = rr;
    }
    // this thread's blocks
    VT v[K][9];
    int32_t nb[K], row[K];
    bool act[K];
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int s = tid + u * CGP_T;
        act[u] = s < nblk;
        nb[u] = row[u] = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) v[u][i] = VT(0);
        if (act[u]) {
            int lo = 0, hi = nown;   // last node whose list starts at or before s
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (sptr[mid] <= s) lo = mid; else hi = mid;
            }
            const int64_t a = a0 + lo;
            const int r = s - sptr[lo];
            row[u] = lo;
            nb[u] = 3 * A.nbrs[blk0 + s];
            // the rows of a node whose three dofs are fixed are not read
            const bool any = !A.free_mask || A.free_mask[3 * a] || A.free_mask[3 * a + 1] || A.free_mask[3 * a + 2];
            act[u] = any;
            if (any) {
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int k = 0; k < 3; ++k) v[u][3 * i + k] = A.V[A.indptr[3 * a + i] + 3 * r + k];
            } else {
#pragma unroll
                for (int i = 0; i < 3; ++i) sm[i * CGP_T * K + s] = 0.0;
            }
        }
    }
    cgp_stores_done();
    __syncthreads();
    // sum of d[0, n) by one wave, stored into a slot by its first lane
    auto publish = [&](const double *d, int n, uint64_t *slot) {
        double s = 0.0;
        for (int i = lane; i < n; i += 64) s += d[i];
        s = dpp_wave_sum(s);
        if (lane == 0) cgp_store(reinterpret_cast<double *>(slot + w), s);
    };
    auto slot_of = [&](int par, int j) { return A.slots + (par * 3 + j) * CGP_MAXW; };
    auto empty_slot = [&](uint64_t *slot) {
        __hip_atomic_store(slot + w, CGP_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if (wave == 0) publish(sd, nown, slot_of(0, 1));
    if (wave == 1) publish(sd + nown, nown, slot_of(0, 2));
    double xp[K][3];
#pragma unroll
    for (int u = 0; u < K; ++u) xp[u][0] = xp[u][1] = xp[u][2] = 0.0;
    double rz_old = 0.0, bnorm = 0.0, rel = 0.0;
    int k = 0;
    bool aborted = false;
    for (;; ++k) {
        const int par = k & 1, ts = tid & (CGP_MAXW - 1);
        // B(k): r.z in the slots of the first half of the threads, r.r in the second's, and the
        // neighbours' z(k), looked for together (z(0) only afterwards: its buffer was not
        // empty before)
        double xz[K][3], s;
        bool ok = cgp_wait_z<K>(slot_of(par, tid < CGP_MAXW ? 1 : 2) + ts, ts < A.nw, k > 0 ? A.z[par] : nullptr, nb,
                                act, A.abort, A.wait_ticks, s, xz);
        s = dpp_wave_sum(s);
        if (lane == 0) sw[wave] = s;
        aborted = !__syncthreads_and(ok);
        if (aborted) break;
        cgp_stores_done();   // the emptied values of the last step (long arrived)
        rz = (sw[0] + sw[1]) + (sw[2] + sw[3]);
        rr = (sw[4] + sw[5]) + (sw[6] + sw[7]);
        if (k == 0) {
            bnorm = sqrt(rr);
            if (bnorm == 0.0) break;
#pragma unroll
            for (int u = 0; u < K; ++u)
#pragma unroll
                for (int c = 0; c < 3; ++c) xz[u][c] = act[u] ? cgp_load(A.z[0] + nb[u] + c) : 0.0;
        } else {
            if (tid == 0) empty_slot(slot_of(par ^ 1, 0));
            if (k % A.check_every == 0 || k == A.maxit) {
                rel = sqrt(rr) / bnorm;
                if (!(rel == rel) || rel <= A.rtol) break;
            }
            if (k == A.maxit) break;
        }
        const double beta = k > 0 && rz_old != 0.0 ? rz / rz_old : 0.0;
        rz_old = rz;
        // q = A p, p = z + beta p of every neighbour: each thread keeps its neighbours' p from
        // step to step (the same fma as the owner's, so the same value), only z travels
        double t = 0.0;
#pragma unroll
        for (int u = 0; u < K; ++u)
            if (act[u]) {
                double *x = xp[u];
#pragma unroll
                for (int c = 0; c < 3; ++c) x[c] = fma(beta, x[c], xz[u][c]);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const double y = (double)v[u][3 * i] * x[0] + (double)v[u][3 * i + 1] * x[1] +
                                     (double)v[u][3 * i + 2] * x[2];
                    sm[i * CGP_T * K + u * CGP_T + tid] = y;
                    const int j = 3 * row[u] + i;
                    if (smask[row[u]] >> i & 1) t += fma(beta, sp[j], sz[j]) * y;
                }
            }
        t = dpp_wave_sum(t);
        if (lane == 0) sw2[wave] = t;
        __syncthreads();
        if (tid == 0) {
            double pq = 0.0;
#pragma unroll
            for (int i = 0; i < CGP_T / 64; ++i) pq += sw2[i];
            cgp_store(reinterpret_cast<double *>(slot_of(par, 0) + w), pq);
        }
        // while the partials travel: the own p, and q by eight lanes per row
        for (int j = tid >> 3; j < 3 * nown; j += CGP_T / 8) {
            const int i = j / 3, c = j - 3 * i;
            double q = 0.0;
            for (int e = sptr[i] + (tid & 7); e < sptr[i + 1]; e += 8) q += sm[c * CGP_T * K + e];
            q = dpp_sum8(q);
            if ((tid & 7) == 0) {
                const bool fr = smask[i] >> c & 1;
                sq[j] = fr ? q : 0.0;
                sp[j] = fr ? fma(beta, sp[j], sz[j]) : 0.0;
            }
        }
        // A(k)
        ok = cgp_wait(slot_of(par, 0) + ts, tid < CGP_MAXW && ts < A.nw, A.abort, A.wait_ticks, s);
        s = dpp_wave_sum(s);
        if (lane == 0) sw[wave] = s;
        aborted = !__syncthreads_and(ok);
        if (aborted) break;
        cgp_stores_done();   // the emptied A slot
        const double pq = (sw[0] + sw[1]) + (sw[2] + sw[3]);
        const double alpha = pq != 0.0 ? rz / pq : 0.0;
        if (tid == 0) {
            empty_slot(slot_of(par, 1));
            empty_slot(slot_of(par, 2));
        }
        if (tid < nown) {
            double rv[3], rzi = 0.0, rri = 0.0;
#pragma unroll
            for (int i = 0; i < 3; ++i) rv[i] = sr[3 * tid + i] - alpha * sq[3 * tid + i];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double zi = sP[9 * tid + 3 * i] * rv[0] + sP[9 * tid + 3 * i + 1] * rv[1] +
                                  sP[9 * tid + 3 * i + 2] * rv[2];
                cgp_store(A.z[par ^ 1] + 3 * (int64_t)(a0 + tid) + i, zi);
                sz[3 * tid + i] = zi;
                rzi += rv[i] * zi;
                rri += rv[i] * rv[i];
            }
            sd[tid] = rzi;
            sd[nown + tid] = rri;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                sr[3 * tid + i] = rv[i];
                sx[3 * tid + i] += alpha * sp[3 * tid + i];
            }
        }
        __syncthreads();
        if (wave == 0) publish(sd, nown, slot_of(par ^ 1, 1));
        if (wave == 1) publish(sd + nown, nown, slot_of(par ^ 1, 2));
        // everyone has read z(k): empty it for z(k+2)
        if (tid < nown)
#pragma unroll
            for (int i = 0; i < 3; ++i)
                cgp_store(A.z[par] + 3 * (int64_t)(a0 + tid) + i, __longlong_as_double((long long)CGP_EMPTY));
    }
    if (aborted) {
        if (tid == 0) __hip_atomic_store(A.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    __syncthreads();
    for (int i = tid; i < 3 * nown; i += CGP_T) A.x[3 * (int64_t)a0 + i] = sx[i];
    if (A.out && w == 0 && tid == 0) {
        A.out[0] = (double)k;
        A.out[1] = rel;
    }
}

// The launch shape for a matrix of `total` blocks with between mindeg and maxdeg blocks per
// node, or nw = 0 where the launch-per-step form is taken: more than CGP_MAXK blocks per
// thread, or more nodes per workgroup than LDS or the node threads hold.  One block per
// thread while that needs no more workgroups than there are CUs; beyond, CGP_PER_WG
// blocks per workgroup, then as many as there are CUs.  Measured, us per step (the
// launch-per-step form in brackets): 18k blocks 4.7 (18), 51k on 106 workgroups 4.8, on 54
// 5.4 (19), 139k on 199 workgroups of two blocks per thread 6.0, on 256 7.5 (20), 275k 7.8
// (20), 389k 8.0 (29).
constexpr int CGP_PER_WG = 740;
static CgpPlan cgp_plan(int64_t nnode, int64_t total, int maxdeg, int mindeg) {
    CgpPlan p;
    const int cus = device_cus();
    if (total <= 0 || mindeg < 1 || cus <= 0 || tuning_value(TUNE_CG, 0) == 1) return p;
    const int most_wg = std::min(cus, CGP_MAXW), per_1 = CGP_T - maxdeg;
    const int per_wg = per_1 > CGP_T / 2 && total <= (int64_t)most_wg * per_1 ? per_1 : CGP_PER_WG;
    const int nw = (int)std::min<int64_t>(most_wg, (total + per_wg - 1) / per_wg);
    const int64_t most = (total + nw - 1) / nw + maxdeg;
    const int64_t nown = std::min<int64_t>(nnode, most / mindeg + 1);
    for (int K : {1, 2, 4, CGP_MAXK})
        if (most <= (int64_t)K * CGP_T) {
            const size_t lds = cgp_lds(K, nown);
            if (nown > CGP_T || lds > 150 * 1024) return p;
            p.nw = nw;
            p.K = K;
            p.total = total;
            p.lds = lds;
            return p;
        }
    return p;
}

template <typename VT, int K>
static int cgp_launch_k(const CgpPlan &p, const CgpArgs<VT> &a, hipStream_t st) {
    if (p.lds > 64 * 1024)
        FL_HIP_CHECK(hipFuncSetAttribute((const void *)cg_persistent_kernel<VT, K>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds));
    PersistentTurn turn;
    const int rc = turn.enter(st);
    if (rc) return rc;
    cg_persistent_kernel<VT, K><<<(unsigned)p.nw, CGP_T, p.lds, st>>>(a);
    FL_LAUNCH_CHECK();
    return turn.leave(st);
}

template <typename VT>
static int cgp_launch(const CgpPlan &p, CgpArgs<VT> a, hipStream_t st) {
    a.nw = p.nw;
    a.total = p.total;
    // FL_TUNE_CG 2: every wait counts as run out (the way back to the launch-per-step form)
    a.wait_ticks = tuning_value(TUNE_CG, 0) == 2 ? -1 : CGP_WAIT_TICKS;
    switch (p.K) {
        case 1: return cgp_launch_k<VT, 1>(p, a, st);
        case 2: return cgp_launch_k<VT, 2>(p, a, st);
        case 4: return cgp_launch_k<VT, 4>(p, a, st);
        default: return cgp_launch_k<VT, CGP_MAXK>(p, a, st);
    }
}

}  // namespace
}  // namespace fl
