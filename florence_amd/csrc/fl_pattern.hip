// Sparsity pattern of the displacement-formulation tangent, built on the device.
//
// Same pattern as ComputeSparsityPattern (Florence/FiniteElements/Assembly/_Assembly_/
// ComputeSparsityPattern.pyx:44-90, ComputeSparsityPattern.h:22-62): for node a the
// sorted unique set of nodes sharing an element with it; its three rows 3a+i list the
// columns 3b+k of every neighbour b in ascending order.  The reference builds this per
// node with std::sort/std::unique on the host; here one wave per node (a workgroup where a
// node has many candidates) gathers the candidate nodes of its incident
// elements into LDS, bitonic-sorts them and compacts.
#include <cstdarg>
#include <climits>
#include <algorithm>
#include <vector>

#include "fl_common.hpp"

namespace fl {

static thread_local std::string g_last_error;

void set_error(const char *fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
}

// ------------------------------------------------------------------ prefix sum
constexpr int SCAN_T = 256;
constexpr int SCAN_I = 8;
constexpr int SCAN_B = SCAN_T * SCAN_I;

__global__ __launch_bounds__(SCAN_T) void scan_blocks_kernel(int64_t *d, int64_t n, int64_t *sums) {
    __shared__ int64_t sh[SCAN_T];
    const int t = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * SCAN_B + (int64_t)t * SCAN_I;
    int64_t v[SCAN_I];
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_I; ++i) {
        const int64_t idx = base + i;
        v[i] = idx < n ? d[idx] : 0;
        s += v[i];
    }
    sh[t] = s;
    __syncthreads();
    for (int off = 1; off < SCAN_T; off <<= 1) {
        int64_t x = t >= off ? sh[t - off] : 0;
        __syncthreads();
        sh[t] += x;
        __syncthreads();
    }
    int64_t run = sh[t] - s;
#pragma unroll
    for (int i = 0; i < SCAN_I; ++i) {
        const int64_t idx = base + i;
        if (idx < n) d[idx] = run;
        run += v[i];
    }
    if (t == SCAN_T - 1 && sums != nullptr) sums[blockIdx.x] = sh[t];
}

__global__ void scan_add_kernel(int64_t *d, int64_t n, const int64_t *sums) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < n) d[idx] += sums[idx / SCAN_B];
}

size_t scan_scratch_count(int64_t n) {
    size_t total = 0;
    int64_t m = n;
    while (m > SCAN_B) {
        m = (m + SCAN_B - 1) / SCAN_B;
        total += (size_t)m + 1;
    }
    return total + 1;
}

int exclusive_scan_i64(int64_t *data, int64_t n, int64_t *scratch, size_t scratch_count, hipStream_t st) {
    if (n <= 0) return 0;
    const int64_t nb = (n + SCAN_B - 1) / SCAN_B;
    if (nb == 1) {
        scan_blocks_kernel<<<1, SCAN_T, 0, st>>>(data, n, nullptr);
        FL_LAUNCH_CHECK();
        return 0;
    }
    if ((size_t)nb + 1 > scratch_count) {
        set_error("scan scratch too small");
        return FL_E_SPACE;
    }
    scan_blocks_kernel<<<(unsigned)nb, SCAN_T, 0, st>>>(data, n, scratch);
    FL_LAUNCH_CHECK();
    int rc = exclusive_scan_i64(scratch, nb, scratch + nb + 1, scratch_count - (size_t)nb - 1, st);
    if (rc) return rc;
    scan_add_kernel<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(data, n, scratch);
    FL_LAUNCH_CHECK();
    return 0;
}

// ------------------------------------------------------- node -> element map
__global__ void count_incidence_kernel(const int32_t *__restrict__ elements, int64_t nentries, int64_t nnode,
                                       int64_t *__restrict__ counts, int32_t *__restrict__ bad) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nentries) return;
    const int32_t nd = elements[t];
    if (nd < 0 || nd >= nnode) {
        atomicOr(bad, 1);
        return;
    }
    atomicAdd(reinterpret_cast<unsigned long long *>(counts + nd), 1ull);
}

__global__ void fill_incidence_kernel(const int32_t *__restrict__ elements, int64_t nentries,
                                      const int64_t *__restrict__ offsets, int32_t *__restrict__ cursor,
                                      int32_t *__restrict__ node_elem) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nentries) return;
    const int32_t nd = elements[t];
    const int32_t slot = atomicAdd(cursor + nd, 1);
    node_elem[offsets[nd] + slot] = (int32_t)t;   // t = e*npe + local
}

// Sort each node's incidence list (ascending element, hence ascending e*npe+local) and emit
// the int32 pointer array: sixteen lanes per node hold the list in registers, and an
// entry's place is the number of smaller ones (in place: a list's reads precede its
// writes in the same wave).  Lists of more than 64 entries: insertion by one lane, the
// only form before, which walked every list through memory (61 us on 24k tet p=2 nodes).
constexpr int SI_L = 16, SI_N = 64;
__global__ __launch_bounds__(256) void sort_incidence_kernel(const int64_t *__restrict__ offsets, int64_t nnode,
                                                             int32_t *__restrict__ node_elem,
                                                             int32_t *__restrict__ node_elem_ptr) {
    const int64_t a = ((int64_t)blockIdx.x * 256 + threadIdx.x) / SI_L;
    const int gl = threadIdx.x % SI_L;
    if (a > nnode) return;
    if (gl == 0) node_elem_ptr[a] = (int32_t)offsets[a];
    if (a == nnode) return;
    const int64_t b = offsets[a];
    const int n = (int)(offsets[a + 1] - b);
    int32_t *list = node_elem + b;
    if (n > SI_N) {
        if (gl != 0) return;
        for (int i = 1; i < n; ++i) {
            const int32_t v = list[i];
            int j = i - 1;
            while (j >= 0 && list[j] > v) {
                list[j + 1] = list[j];
                --j;
            }
            list[j + 1] = v;
        }
        return;
    }
    constexpr int U = SI_N / SI_L;
    int32_t v[U];
    int rank[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        v[u] = gl + SI_L * u < n ? list[gl + SI_L * u] : INT_MAX;
        rank[u] = 0;
    }
#pragma unroll
    for (int w = 0; w < U; ++w)
        if (SI_L * w < n)
            for (int j = 0; j < SI_L; ++j) {
                const int32_t x = __shfl(v[w], j, SI_L);
#pragma unroll
                for (int u = 0; u < U; ++u) rank[u] += x < v[u];
            }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (gl + SI_L * u < n) list[rank[u]] = v[u];
}

// ----------------------------------------------------------- neighbour lists
constexpr int NB_T = 256;
constexpr int NB_MAX = 8192;   // candidate nodes per node (incident elements x npe)

// Gather candidates of node a into LDS, sort, mark uniques.  Returns unique count.
__device__ int gather_sort_unique(const int32_t *__restrict__ elements, int32_t npe,
                                  const int32_t *__restrict__ node_elem_ptr,
                                  const int32_t *__restrict__ node_elem, int64_t a, int32_t *cand,
                                  int32_t *flag_sum, int32_t *overflow) {
    const int t = threadIdx.x;
    const int32_t b0 = node_elem_ptr[a], b1 = node_elem_ptr[a + 1];
    const int ncand = (b1 - b0) * npe;
    if (ncand > NB_MAX) {
        if (t == 0) atomicOr(overflow, 1);
        return -1;
    }
    int S = 64;
    while (S < ncand) S <<= 1;
    for (int i = t; i < S; i += NB_T) {
        int32_t v = INT_MAX;
        if (i < ncand) {
            const int32_t ent = node_elem[b0 + i / npe];
            const int32_t e = ent / npe;
            v = elements[(int64_t)e * npe + i % npe];
        }
        cand[i] = v;
    }
    __syncthreads();
    // bitonic sort, ascending
    for (int k = 2; k <= S; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = t; i < S; i += NB_T) {
                const int p = i ^ j;
                if (p > i) {
                    const int32_t x = cand[i], y = cand[p];
                    const bool up = (i & k) == 0;
                    if ((x > y) == up) {
                        cand[i] = y;
                        cand[p] = x;
                    }
                }
            }
            __syncthreads();
        }
    }
    // per-thread contiguous chunk unique counts, then exclusive scan in flag_sum
    const int per = (S + NB_T - 1) / NB_T;
    const int lo = t * per, hi = min(lo + per, ncand);
    int c = 0;
    for (int i = lo; i < hi; ++i) c += (i == 0 || cand[i] != cand[i - 1]) ? 1 : 0;
    flag_sum[t] = c;
    __syncthreads();
    for (int off = 1; off < NB_T; off <<= 1) {
        int x = t >= off ? flag_sum[t - off] : 0;
        __syncthreads();
        flag_sum[t] += x;
        __syncthreads();
    }
    return flag_sum[NB_T - 1];
}

// Nodes of at most rule.wave_max candidates: one wave per node, its candidates sorted in the
// wave's own 4 KB of LDS without a workgroup barrier (a wave's LDS accesses are in order;
// the fences only keep the compiler's).  The workgroup form below, for the nodes above
// that, sorted every list before: its 33 KB of LDS and two dozen barriers for lists of
// mostly under 64 candidates took 292 + 170 us on 24k tet p=2 nodes; this form
// takes 28 + 33.
constexpr int NW_MAX = 1024;

struct ListRule {
    int wave_max;   // candidates of a node that a wave takes, at most NW_MAX
    int per;        // nodes a workgroup of the other form looks through at a time, at most NB_T
};
// A mesh of few nodes waits for its longest list, which a lone wave sorts more slowly than a
// workgroup, and leaves the chip room for a workgroup a node: both passes of p = 4 tets, 793
// nodes 224 -> 184 us, 5,681 nodes 243 -> 208; p = 4 hexes, 729 nodes 230 -> 186, 4,913 249 -> 225
// (lists above 256 only: 204, 222, 207, 234).  From there on workgroups wait for each other: p = 3
// hexes, 6,859 nodes 189 -> 194, p = 4 hexes, 15,625 nodes 262 -> 404.
static ListRule list_rule(int64_t nnode) { return nnode <= 6144 ? ListRule{128, 1} : ListRule{NW_MAX, NB_T}; }

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// the rows of node a (cnt neighbours in c, list start p0): indptr, and every row's columns
__device__ __forceinline__ void write_rows(const int32_t *c, int cnt, int64_t a, int64_t nnode, int32_t p0,
                                           const int32_t *__restrict__ node_nbr_ptr, int32_t *__restrict__ indptr,
                                           int32_t *__restrict__ indices, int t, int nt) {
    const int rowlen = 3 * cnt;
    if (t < 3) indptr[3 * a + t] = (int32_t)(9 * (int64_t)p0 + t * rowlen);
    // the last entry holds a negative flag as well (fl_pattern_fill): added, not stored
    if (a == nnode - 1 && t == 0) atomicAdd(indptr + 3 * nnode, (int32_t)(9 * (int64_t)node_nbr_ptr[nnode]));
    if (indices == nullptr) return;
    for (int q = t; q < 3 * rowlen; q += nt) {
        const int i = q >= 2 * rowlen ? 2 : (q >= rowlen ? 1 : 0);
        const int col = q - i * rowlen, r = col / 3;
        indices[9 * (int64_t)p0 + q] = 3 * c[r] + (col - 3 * r);
    }
}

constexpr int32_t FILL_BAD = INT32_MIN;   // in indptr[3 nnode]: lists inconsistent with the counts

template <bool FILL>
__global__ __launch_bounds__(256) void wave_neighbours_kernel(
    const int32_t *__restrict__ elements, int32_t npe, const int32_t *__restrict__ node_elem_ptr,
    const int32_t *__restrict__ node_elem, int64_t nnode, ListRule rule, int64_t *__restrict__ nbr_count,
    const int32_t *__restrict__ node_nbr_ptr, int32_t *__restrict__ node_nbrs, int32_t *__restrict__ indptr,
    int32_t *__restrict__ indices) {
    __shared__ int32_t sc[4][NW_MAX];
    const int lane = threadIdx.x & 63;
    int32_t *c = sc[threadIdx.x >> 6];
    const int64_t a = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (a >= nnode) return;
    const int32_t b0 = node_elem_ptr[a];
    const int64_t nc = (int64_t)(node_elem_ptr[a + 1] - b0) * npe;
    if (nc > rule.wave_max) return;
    const int ncand = (int)nc;
    int S = 64;
    while (S < ncand) S <<= 1;
    for (int i = lane; i < S; i += 64) {
        int32_t v = INT_MAX;
        if (i < ncand) {
            const int j = i / npe;
            const uint32_t e = (uint32_t)node_elem[b0 + j] / (uint32_t)npe;
            v = elements[(int64_t)e * npe + (i - j * npe)];
        }
        c[i] = v;
    }
    wave_fence();
    for (int k = 2; k <= S; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = lane; t < S / 2; t += 64) {
                const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), p = i | j;
                const int32_t x = c[i], y = c[p];
                if ((x > y) == ((i & k) == 0)) {
                    c[i] = y;
                    c[p] = x;
                }
            }
            wave_fence();
        }
    // the distinct ones, packed to the front (an entry only moves down, past entries read)
    int cnt = 0;
    for (int i0 = 0; i0 < ncand; i0 += 64) {
        const int i = i0 + lane;
        const int32_t v = i < ncand ? c[i] : 0;
        const bool first = i < ncand && (i == 0 || c[i - 1] != v);
        wave_fence();
        const unsigned long long m = __ballot(first);
        if (first) c[cnt + __popcll(m & ((1ull << lane) - 1))] = v;
        cnt += __popcll(m);
        wave_fence();
    }
    if constexpr (!FILL) {
        if (lane == 0) nbr_count[a] = cnt;
    } else {
        const int32_t p0 = node_nbr_ptr[a];
        if (cnt != node_nbr_ptr[a + 1] - p0) {
            if (lane == 0) atomicOr(indptr + 3 * nnode, FILL_BAD);
            return;
        }
        for (int i = lane; i < cnt; i += 64) node_nbrs[p0 + i] = c[i];
        write_rows(c, cnt, a, nnode, p0, node_nbr_ptr, indptr, indices, lane, 64);
    }
}

// The nodes of more candidates than a wave takes, one workgroup per node: a grid of fixed
// size looks through the nodes rule.per at a time and takes up the large ones.
template <bool FILL>
__global__ __launch_bounds__(NB_T) void group_neighbours_kernel(
    const int32_t *__restrict__ elements, int32_t npe, const int32_t *__restrict__ node_elem_ptr,
    const int32_t *__restrict__ node_elem, int64_t nnode, ListRule rule, int64_t *__restrict__ nbr_count,
    int32_t *__restrict__ overflow, const int32_t *__restrict__ node_nbr_ptr,
    int32_t *__restrict__ node_nbrs, int32_t *__restrict__ indptr, int32_t *__restrict__ indices) {
    __shared__ int32_t cand[NB_MAX];
    __shared__ int32_t flag_sum[NB_T];
    __shared__ unsigned long long large[NB_T / 64];
    const int t = threadIdx.x;
    for (int64_t base = (int64_t)blockIdx.x * rule.per; base < nnode; base += (int64_t)gridDim.x * rule.per) {
        const bool mine = t < rule.per && base + t < nnode &&
                          (int64_t)(node_elem_ptr[base + t + 1] - node_elem_ptr[base + t]) * npe > rule.wave_max;
        const unsigned long long m = __ballot(mine);
        if ((t & 63) == 0) large[t >> 6] = m;
        __syncthreads();
        for (int w = 0; w < NB_T / 64; ++w)
            for (unsigned long long rest = large[w]; rest; rest &= rest - 1) {
                const int64_t a = base + 64 * w + __ffsll((long long)rest) - 1;
                __syncthreads();   // the previous node's last reads of cand and flag_sum
                const int cnt = gather_sort_unique(elements, npe, node_elem_ptr, node_elem, a, cand, flag_sum,
                                                   overflow);
                if constexpr (!FILL) {
                    if (t == 0) nbr_count[a] = cnt < 0 ? 0 : cnt;
                } else {
                    const int32_t p0 = node_nbr_ptr[a];
                    if (cnt < 0 || cnt != node_nbr_ptr[a + 1] - p0) {
                        if (t == 0) atomicOr(indptr + 3 * nnode, FILL_BAD);
                        continue;
                    }
                    const int ncand = (node_elem_ptr[a + 1] - node_elem_ptr[a]) * npe;
                    int S = 64;
                    while (S < ncand) S <<= 1;
                    const int per = (S + NB_T - 1) / NB_T;
                    const int lo = t * per, hi = min(lo + per, ncand);
                    int r = t == 0 ? 0 : flag_sum[t - 1];
                    for (int i = lo; i < hi; ++i)
                        if (i == 0 || cand[i] != cand[i - 1]) node_nbrs[p0 + r++] = cand[i];
                    __syncthreads();
                    write_rows(node_nbrs + p0, cnt, a, nnode, p0, node_nbr_ptr, indptr, indices, t, NB_T);
                }
            }
        __syncthreads();   // before the next nodes' masks
    }
}

// node_nbr_ptr from the scanned counts, and the largest count (one atomic per wave that
// has a larger one than is recorded)
__global__ __launch_bounds__(256) void nbr_ptr_kernel(const int64_t *__restrict__ src, int32_t *__restrict__ dst,
                                                      int64_t nnode, int32_t *__restrict__ max_degree) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t <= nnode) dst[t] = (int32_t)src[t];
    int d = t < nnode ? (int)(src[t + 1] - src[t]) : 0;
    for (int off = 32; off > 0; off >>= 1) d = max(d, __shfl_xor(d, off, 64));
    if ((threadIdx.x & 63) == 0 && d > __hip_atomic_load(max_degree, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(max_degree, d);
}

// ranks[(e npe + la) npe + lb] = position of node elements[e][lb] in the sorted
// neighbour list of node elements[e][la] (the CSR column block of that entry); status
// bit FL_S_PATTERN if a node is missing or a list exceeds the int16 range.
__global__ void rank_table_kernel(const int32_t *__restrict__ elements, int64_t nelem, int npe,
                                  const int32_t *__restrict__ nbr_ptr, const int32_t *__restrict__ nbrs,
                                  int16_t *__restrict__ ranks, int32_t *__restrict__ status) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t npe2 = (int64_t)npe * npe;
    if (t >= nelem * npe2) return;
    const int64_t e = t / npe2;
    const int la = (int)((t - e * npe2) / npe), lb = (int)(t - e * npe2 - (int64_t)la * npe);
    const int32_t a = elements[e * npe + la], b = elements[e * npe + lb];
    const int32_t p0 = nbr_ptr[a], deg = nbr_ptr[a + 1] - p0;
    int lo = 0, hi = deg;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (b < nbrs[p0 + mid]) hi = mid; else lo = mid;
    }
    const bool ok = deg > 0 && deg <= 32767 && nbrs[p0 + lo] == b;
    if (!ok) atomicOr(status, FL_S_PATTERN);
    ranks[t] = ok ? (int16_t)lo : (int16_t)0;
}

// The direct scatter's table, one entry per slot of sf_scatter_index's order for hexes
// of p1^3 nodes: the position of the column node b in the sorted neighbour list of the
// row node a, with the sign bit set when an element of a lower colour holds both a and b
// (that element has already written the entry); unused slots hold 0.  Tensor nodes map
// to the element's local nodes through local_of_t of the tensor basis.  Status bit
// FL_S_PATTERN on a missing node, an oversized list, a basis of another p1, or two
// elements of one colour that share a node.
__global__ void scatter_table_kernel(const int32_t *__restrict__ elements, int64_t nelem, int p1,
                                     const int32_t *__restrict__ node_elem_ptr, const int32_t *__restrict__ node_elem,
                                     const int32_t *__restrict__ nbr_ptr, const int32_t *__restrict__ nbrs,
                                     const int32_t *__restrict__ colour, const int32_t *__restrict__ basis,
                                     int16_t *__restrict__ table, int32_t *__restrict__ status) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t per = sf_scatter_per_element(p1);
    if (t >= nelem * per) return;
    const int64_t e = t / per;
    int64_t u = t - e * per;
    const int mt = sf_row_tiles(p1), nt = sf_col_tiles(p1);
    const int r = (int)(u % 4);
    u /= 4;
    const int tm = (int)(u % mt);
    u /= mt;
    const int lane = (int)(u % 64);
    u /= 64;
    const int s = (int)(u % nt);
    const int az = (int)(u / nt);
    const int pp = p1 * p1, npe = pp * p1;
    const int row = 16 * tm + (lane >> 4) + 4 * r, col = 16 * s + (lane & 15);
    if (row >= pp || col >= npe) {
        table[t] = 0;
        return;
    }
    const int ab = row / p1, bb = row % p1, ae = col / pp, be = (col / p1) % p1, bz = col % p1;
    const int ta = (ab * p1 + ae) * p1 + az, tb = (bb * p1 + be) * p1 + bz;
    const int32_t *loc = basis + 4 + basis[1] * basis[1] * basis[1];
    const int la = min(max(loc[ta], 0), npe - 1), lb = min(max(loc[tb], 0), npe - 1);
    const int32_t a = elements[e * npe + la], b = elements[e * npe + lb];
    const int32_t p0 = nbr_ptr[a], deg = nbr_ptr[a + 1] - p0;
    int lo = 0, hi = deg;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (b < nbrs[p0 + mid]) hi = mid; else lo = mid;
    }
    bool ok = basis[0] == p1 && deg > 0 && deg <= 32767 && nbrs[p0 + lo] == b;
    const int32_t ce = colour[e];
    bool add = false;
    for (int32_t q = node_elem_ptr[a]; q < node_elem_ptr[a + 1]; ++q) {
        const int32_t e2 = node_elem[q] / npe;
        if (e2 != e && colour[e2] == ce) ok = false;
        if (colour[e2] >= ce || add) continue;
        for (int32_t q2 = node_elem_ptr[b]; q2 < node_elem_ptr[b + 1]; ++q2)
            if (node_elem[q2] / npe == e2) add = true;
    }
    if (!ok) atomicOr(status, FL_S_PATTERN);
    table[t] = ok ? (int16_t)(add ? lo - 32768 : lo) : (int16_t)0;
}

static unsigned group_grid(int64_t nnode, int per) {
    return (unsigned)(per == 1 ? nnode : std::min<int64_t>((nnode + per - 1) / per, 1024));
}

// ------------------------------------------------------------------- gather plan
// Node classes by neighbour count: class 0 the smallest count (in meshes with
// element-interior nodes, exactly those: a node of two distinct elements has more
// neighbours than an element has nodes), classes 1.. by at most 128, 256, ... 2048.  The
// nodes are grouped by class in ascending order: counts per chunk of PL_CHUNK nodes,
// their scan per class, and a stable scatter.
constexpr int PL_CHUNK = 1024, PL_C = FL_GATHER_BUCKETS;
// scratch (int32, zeroed): [0] 2^30 - smallest count, [1, 7) largest count per class, [7, 13)
// nodes per class, [13] INT32_MAX - the first node above every class; from 16: [chunk][class]
constexpr int PL_HEAD = 16;
__device__ __forceinline__ int plan_class(int d, int dmin) {
    if (d == dmin) return 0;
    int c = 1;
    while (c < PL_C && d > (64 << c)) ++c;
    return c;
}

__global__ __launch_bounds__(256) void plan_min_kernel(const int32_t *__restrict__ ptr, int64_t nnode,
                                                       int32_t *__restrict__ w) {
    const int64_t a = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int m = a < nnode ? (1 << 30) - (ptr[a + 1] - ptr[a]) : 0;
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0 && m > __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(w, m);
}

// SCATTER = false: counts and largest degrees of a chunk's classes; true: its nodes put in
// their places (the chunk counts scanned before)
template <bool SCATTER>
__global__ __launch_bounds__(256) void plan_chunk_kernel(const int32_t *__restrict__ ptr, int64_t nnode,
                                                         int32_t *__restrict__ w, int32_t *__restrict__ order) {
    __shared__ int32_t cnt[4][PL_C], base[PL_C], deg[PL_C];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int dmin = (1 << 30) - w[0];
    int32_t *hist = w + PL_HEAD + PL_C * (int64_t)blockIdx.x;
    if (t < PL_C) base[t] = SCATTER ? hist[t] : 0;
    if (t < PL_C) deg[t] = 0;
    __syncthreads();
    for (int r = 0; r < PL_CHUNK / 256; ++r) {
        const int64_t a = (int64_t)blockIdx.x * PL_CHUNK + 256 * r + t;
        const int d = a < nnode ? ptr[a + 1] - ptr[a] : 0;
        const int c = a < nnode ? plan_class(d, dmin) : -1;
        if (!SCATTER && c == PL_C) atomicMax(w + 13, INT32_MAX - (int32_t)a);
        if (!SCATTER && c >= 0 && c < PL_C && d > deg[c]) atomicMax(&deg[c], d);
        int before = 0;
#pragma unroll
        for (int k = 0; k < PL_C; ++k) {
            const unsigned long long m = __ballot(c == k);
            if (c == k) before = __popcll(m & ((1ull << lane) - 1));
            if (lane == 0) cnt[wave][k] = __popcll(m);
        }
        __syncthreads();
        if (SCATTER && c >= 0 && c < PL_C) {
            for (int v = 0; v < wave; ++v) before += cnt[v][c];
            order[base[c] + before] = (int32_t)a;
        }
        __syncthreads();
        if (t < PL_C) base[t] += cnt[0][t] + cnt[1][t] + cnt[2][t] + cnt[3][t];
        __syncthreads();
    }
    if (!SCATTER) {
        if (t < PL_C) {
            hist[t] = base[t];
            if (deg[t]) atomicMax(w + 1 + t, deg[t]);
        }
    }
}

// chunk counts -> first places, one wave per class; then the class's own start is added
__global__ __launch_bounds__(64 * PL_C) void plan_scan_kernel(int32_t *__restrict__ w, int64_t nchunk) {
    __shared__ int32_t total[PL_C];
    const int c = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int32_t *h = w + PL_HEAD + c;
    int s = 0;
    for (int64_t b = lane; b < nchunk; b += 64) s += h[PL_C * b];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) {
        total[c] = s;
        w[7 + c] = s;
    }
    __syncthreads();
    int run = 0;
    for (int k = 0; k < c; ++k) run += total[k];
    for (int64_t b0 = 0; b0 < nchunk; b0 += 64) {
        const int64_t b = b0 + lane;
        const int v = b < nchunk ? h[PL_C * b] : 0;
        int x = v;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off, 64);
            if (lane >= off) x += y;
        }
        if (b < nchunk) h[PL_C * b] = run + x - v;
        run += __shfl(x, 63, 64);
    }
}

}  // namespace fl

using namespace fl;

extern "C" {

int fl_version(void) { return 100; }

const char *fl_last_error(void) { return g_last_error.c_str(); }

size_t fl_pattern_workspace_size(int64_t nnode) {
    // counts/offsets (nnode+1) x2 int64, cursor int32, scan scratch, flags
    return align_up((size_t)(nnode + 1) * 8, 256) * 2 + align_up((size_t)(nnode + 1) * 4, 256) +
           align_up(scan_scratch_count(nnode + 1) * 8, 256) + 1024;
}

int fl_pattern_graph(const int32_t *elements, int64_t nelem, int32_t npe, int64_t nnode, int32_t *node_elem_ptr,
                     int32_t *node_elem, int32_t *node_nbr_ptr, int64_t *node_nnz, int32_t *max_degree,
                     void *workspace, size_t workspace_bytes, void *stream) {
    hipStream_t st = as_stream(stream);
    if (nelem <= 0 || npe <= 0 || nnode <= 0 || !elements || !node_elem_ptr || !node_elem || !node_nbr_ptr ||
        !node_nnz || !max_degree) {
        set_error("fl_pattern_graph: invalid argument");
        return FL_E_ARG;
    }
    const int64_t nent = nelem * (int64_t)npe;
    if (nent >= INT32_MAX) {
        set_error("fl_pattern_graph: nelem*npe exceeds int32");
        return FL_E_LIMIT;
    }
    Carve cv(workspace, workspace_bytes);
    int64_t *counts = cv.take<int64_t>(nnode + 1);
    int64_t *nbrc = cv.take<int64_t>(nnode + 1);
    int32_t *cursor = cv.take<int32_t>(nnode + 1);
    const size_t sc = scan_scratch_count(nnode + 1);
    int64_t *scratch = cv.take<int64_t>(sc);
    int32_t *flags = cv.take<int32_t>(4);   // [0] bad node id, [1] overflow, [2] max degree
    if (!cv.ok) {
        set_error("fl_pattern_graph: workspace too small (%zu < %zu)", workspace_bytes, cv.off);
        return FL_E_SPACE;
    }
    FL_HIP_CHECK(hipMemsetAsync(counts, 0, sizeof(int64_t) * (nnode + 1), st));
    FL_HIP_CHECK(hipMemsetAsync(cursor, 0, sizeof(int32_t) * (nnode + 1), st));
    FL_HIP_CHECK(hipMemsetAsync(flags, 0, sizeof(int32_t) * 4, st));
    const unsigned gb = (unsigned)((nent + 255) / 256);
    count_incidence_kernel<<<gb, 256, 0, st>>>(elements, nent, nnode, counts, flags);
    FL_LAUNCH_CHECK();
    int rc = exclusive_scan_i64(counts, nnode + 1, scratch, sc, st);
    if (rc) return rc;
    fill_incidence_kernel<<<gb, 256, 0, st>>>(elements, nent, counts, cursor, node_elem);
    FL_LAUNCH_CHECK();
    sort_incidence_kernel<<<(unsigned)(((nnode + 1) * SI_L + 255) / 256), 256, 0, st>>>(counts, nnode, node_elem,
                                                                                        node_elem_ptr);
    FL_LAUNCH_CHECK();
    FL_HIP_CHECK(hipMemsetAsync(nbrc, 0, sizeof(int64_t) * (nnode + 1), st));
    const ListRule rule = list_rule(nnode);
    wave_neighbours_kernel<false><<<(unsigned)((nnode + 3) / 4), 256, 0, st>>>(
        elements, npe, node_elem_ptr, node_elem, nnode, rule, nbrc, nullptr, nullptr, nullptr, nullptr);
    group_neighbours_kernel<false><<<group_grid(nnode, rule.per), NB_T, 0, st>>>(
        elements, npe, node_elem_ptr, node_elem, nnode, rule, nbrc, flags + 1, nullptr, nullptr, nullptr, nullptr);
    FL_LAUNCH_CHECK();
    rc = exclusive_scan_i64(nbrc, nnode + 1, scratch, sc, st);
    if (rc) return rc;
    nbr_ptr_kernel<<<(unsigned)((nnode + 1 + 255) / 256), 256, 0, st>>>(nbrc, node_nbr_ptr, nnode, flags + 2);
    FL_LAUNCH_CHECK();
    int64_t total = 0;
    int32_t hflags[4] = {0, 0, 0, 0};
    FL_HIP_CHECK(hipMemcpyAsync(&total, nbrc + nnode, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    FL_HIP_CHECK(hipMemcpyAsync(hflags, flags, sizeof(hflags), hipMemcpyDeviceToHost, st));
    FL_HIP_CHECK(hipStreamSynchronize(st));
    if (hflags[0]) {
        set_error("fl_pattern_graph: element connectivity references a node outside [0, nnode)");
        return FL_E_ARG;
    }
    if (hflags[1]) {
        set_error("fl_pattern_graph: a node touches more than %d candidate nodes", NB_MAX);
        return FL_E_LIMIT;
    }
    if (9 * total >= (int64_t)INT32_MAX) {
        set_error("fl_pattern_graph: nnz = %lld exceeds int32 CSR indices", (long long)(9 * total));
        return FL_E_LIMIT;
    }
    *node_nnz = total;
    *max_degree = hflags[2];
    return 0;
}

int fl_pattern_fill(const int32_t *elements, int64_t nelem, int32_t npe, int64_t nnode, const int32_t *node_elem_ptr,
                    const int32_t *node_elem, const int32_t *node_nbr_ptr, int32_t *node_nbrs, int32_t *indptr,
                    int32_t *indices, void *stream) {
    hipStream_t st = as_stream(stream);
    if (nelem <= 0 || npe <= 0 || nnode <= 0 || !elements || !node_elem_ptr || !node_elem || !node_nbr_ptr ||
        !node_nbrs || !indptr) {
        set_error("fl_pattern_fill: invalid argument");
        return FL_E_ARG;
    }
    // the last entry of indptr carries the kernels' flag to the host: FILL_BAD, or the total
    int32_t *last = indptr + 3 * nnode;
    FL_HIP_CHECK(hipMemsetAsync(last, 0, sizeof(int32_t), st));
    const ListRule rule = list_rule(nnode);
    wave_neighbours_kernel<true><<<(unsigned)((nnode + 3) / 4), 256, 0, st>>>(
        elements, npe, node_elem_ptr, node_elem, nnode, rule, nullptr, node_nbr_ptr, node_nbrs, indptr, indices);
    group_neighbours_kernel<true><<<group_grid(nnode, rule.per), NB_T, 0, st>>>(
        elements, npe, node_elem_ptr, node_elem, nnode, rule, nullptr, last, node_nbr_ptr, node_nbrs, indptr, indices);
    FL_LAUNCH_CHECK();
    int32_t h = 0;
    FL_HIP_CHECK(hipMemcpyAsync(&h, last, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    FL_HIP_CHECK(hipStreamSynchronize(st));
    if (h < 0) {
        set_error("fl_pattern_fill: neighbour lists inconsistent with fl_pattern_graph");
        return FL_E_ARG;
    }
    return 0;
}

size_t fl_pattern_rank_table_bytes(int64_t nelem, int32_t npe) {
    return nelem > 0 && npe > 0 ? sizeof(int16_t) * (size_t)nelem * npe * npe : 0;
}

int fl_pattern_rank_table(const int32_t *elements, int64_t nelem, int32_t npe, const int32_t *node_nbr_ptr,
                          const int32_t *node_nbrs, int16_t *ranks, int32_t *status, void *stream) {
    if (!elements || !node_nbr_ptr || !node_nbrs || !ranks || !status || nelem <= 0 || npe <= 0) {
        set_error("fl_pattern_rank_table: invalid argument");
        return FL_E_ARG;
    }
    const int64_t n = nelem * npe * (int64_t)npe;
    rank_table_kernel<<<(unsigned)((n + 255) / 256), 256, 0, as_stream(stream)>>>(elements, nelem, npe, node_nbr_ptr,
                                                                                 node_nbrs, ranks, status);
    FL_LAUNCH_CHECK();
    return 0;
}

int fl_pattern_colour(const int32_t *elements, int64_t nelem, int32_t npe, int64_t nnode, int32_t max_colours,
                      int32_t *colour_of_elem, int32_t *colour_elems, int32_t *colour_offsets, int32_t *ncolour) {
    if (!elements || !colour_of_elem || !colour_elems || !colour_offsets || !ncolour || nelem <= 0 || npe <= 0 ||
        nnode <= 0 || max_colours < 1 || max_colours > 64 || nelem >= INT32_MAX) {
        set_error("fl_pattern_colour: invalid argument");
        return FL_E_ARG;
    }
    // greedy first fit in element order; used[a] = colours already holding node a
    std::vector<uint64_t> used((size_t)nnode, 0);
    std::vector<int64_t> count(64, 0);
    int nc = 0;
    for (int64_t e = 0; e < nelem; ++e) {
        const int32_t *conn = elements + e * npe;
        uint64_t taken = 0;
        for (int a = 0; a < npe; ++a) {
            if (conn[a] < 0 || conn[a] >= nnode) {
                set_error("fl_pattern_colour: element %lld has node %d outside [0, %lld)", (long long)e, conn[a],
                          (long long)nnode);
                return FL_E_ARG;
            }
            taken |= used[conn[a]];
        }
        int c = 0;
        while (c < 64 && ((taken >> c) & 1)) ++c;
        if (c >= max_colours) {
            set_error("fl_pattern_colour: element %lld needs more than %d colours", (long long)e, max_colours);
            return FL_E_LIMIT;
        }
        colour_of_elem[e] = c;
        ++count[c];
        nc = std::max(nc, c + 1);
        for (int a = 0; a < npe; ++a) used[conn[a]] |= 1ull << c;
    }
    colour_offsets[0] = 0;
    for (int c = 0; c < nc; ++c) colour_offsets[c + 1] = colour_offsets[c] + (int32_t)count[c];
    std::vector<int32_t> cur(colour_offsets, colour_offsets + nc);
    for (int64_t e = 0; e < nelem; ++e) colour_elems[cur[colour_of_elem[e]]++] = (int32_t)e;
    *ncolour = nc;
    return 0;
}

// p1 of a hex of npe = p1^3 nodes (0 otherwise)
static int cube_root(int32_t npe) {
    for (int p1 = 1; p1 * p1 * p1 <= npe; ++p1)
        if (p1 * p1 * p1 == npe) return p1;
    return 0;
}

size_t fl_pattern_scatter_table_bytes(int64_t nelem, int32_t npe) {
    const int p1 = npe > 0 ? cube_root(npe) : 0;
    return nelem > 0 && p1 > 0 ? sizeof(int16_t) * (size_t)(nelem * sf_scatter_per_element(p1)) : 0;
}

int fl_pattern_scatter_table(const int32_t *elements, int64_t nelem, int32_t npe, const int32_t *node_elem_ptr,
                             const int32_t *node_elem, const int32_t *node_nbr_ptr, const int32_t *node_nbrs,
                             const int32_t *colour_of_elem, const void *tensor_basis, int16_t *table, int32_t *status,
                             void *stream) {
    const int p1 = npe > 0 ? cube_root(npe) : 0;
    if (!elements || !node_elem_ptr || !node_elem || !node_nbr_ptr || !node_nbrs || !colour_of_elem ||
        !tensor_basis || !table || !status || nelem <= 0 || p1 <= 0) {
        set_error("fl_pattern_scatter_table: invalid argument (hexes of p1^3 nodes and their tensor basis)");
        return FL_E_ARG;
    }
    const int64_t n = nelem * sf_scatter_per_element(p1);
    if ((n + 255) / 256 > (int64_t)UINT32_MAX) {
        set_error("fl_pattern_scatter_table: too many entries for one launch");
        return FL_E_LIMIT;
    }
    scatter_table_kernel<<<(unsigned)((n + 255) / 256), 256, 0, as_stream(stream)>>>(
        elements, nelem, p1, node_elem_ptr, node_elem, node_nbr_ptr, node_nbrs, colour_of_elem,
        static_cast<const int32_t *>(tensor_basis), table, status);
    FL_LAUNCH_CHECK();
    return 0;
}

int fl_pattern_gather_plan(const int32_t *node_nbr_ptr, int64_t nnode, int32_t *node_order, int32_t *bucket_offsets,
                           int32_t *bucket_degree, void *stream) {
    hipStream_t st = as_stream(stream);
    if (!node_nbr_ptr || !node_order || !bucket_offsets || !bucket_degree || nnode <= 0) {
        set_error("fl_pattern_gather_plan: invalid argument");
        return FL_E_ARG;
    }
    const int64_t nchunk = (nnode + PL_CHUNK - 1) / PL_CHUNK;
    const size_t bytes = sizeof(int32_t) * (size_t)(PL_HEAD + PL_C * nchunk);
    int32_t *w = nullptr, h[PL_HEAD];
    FL_HIP_CHECK(hipMallocAsync(reinterpret_cast<void **>(&w), bytes, st));
    hipError_t e = hipMemsetAsync(w, 0, bytes, st);
    if (e == hipSuccess) {
        plan_min_kernel<<<(unsigned)((nnode + 255) / 256), 256, 0, st>>>(node_nbr_ptr, nnode, w);
        plan_chunk_kernel<false><<<(unsigned)nchunk, 256, 0, st>>>(node_nbr_ptr, nnode, w, nullptr);
        plan_scan_kernel<<<1, 64 * PL_C, 0, st>>>(w, nchunk);
        plan_chunk_kernel<true><<<(unsigned)nchunk, 256, 0, st>>>(node_nbr_ptr, nnode, w, node_order);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(h, w, sizeof(h), hipMemcpyDeviceToHost, st);
    (void)hipFreeAsync(w, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    FL_HIP_CHECK(e);
    if (h[13] > 0) {
        const int64_t a = INT32_MAX - h[13];
        int32_t p[2] = {0, 0};
        FL_HIP_CHECK(hipMemcpyAsync(p, node_nbr_ptr + a, sizeof(p), hipMemcpyDeviceToHost, st));
        FL_HIP_CHECK(hipStreamSynchronize(st));
        set_error("fl_pattern_gather_plan: node %lld has %d neighbours (limit %d)", (long long)a, p[1] - p[0],
                  64 << (PL_C - 1));
        return FL_E_LIMIT;
    }
    bucket_offsets[0] = 0;
    for (int b = 0; b < PL_C; ++b) {
        bucket_offsets[b + 1] = bucket_offsets[b] + h[7 + b];
        bucket_degree[b] = h[1 + b];
    }
    return 0;
}

}  // extern "C"
