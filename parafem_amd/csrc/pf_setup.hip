// Problem set-up on the device: the element steering g_g_pp from the node
// freedom table, and the transposed steering (equation -> element slots)
// that the order-preserving scatter walks.
//
// Reference: REARRANGE + FIND_G3 / FIND_G4 (src/modules/shared/
// new_library.f90:3059-3271) give every free freedom of every node an
// equation number in ascending node, then freedom, order; g_g_pp(:,iel) is
// that table gathered through g_num_pp(:,iel) (p121.f90:44-47).  MAKE_GGL
// (src/modules/mpi/gather_scatter.f90:1387-1780) builds the halo maps; at one
// rank the only map left is the transposed steering, built here.
//
// The transposed steering lists, for equation q, the slots k = iel*ntot + i
// with g_g(i,iel) = q in ascending k.  Device construction: count the slots
// per equation (integer atomics: exact), exclusive scan of the counts, place
// every slot with an atomic cursor, then sort each equation's short list, so
// the result does not depend on the order the atomics ran in.
#include "pf_internal.h"

#include <algorithm>
#include <vector>

namespace {

constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_CHUNK = 256 * SCAN_ITEMS;

__global__ __launch_bounds__(256) void k_csr_count(const int *__restrict__ gg, long nslot, int neq,
                                                  int *__restrict__ cnt, int *__restrict__ err)
{
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < nslot; k += (long)gridDim.x * blockDim.x) {
        const int g = gg[k];
        if (g < 0 || g > neq) atomicOr(err, 1);
        else if (g) atomicAdd(&cnt[g - 1], 1);
    }
}

// Block sums of consecutive chunks of SCAN_CHUNK counts.
__global__ __launch_bounds__(256) void k_scan_sums(const int *__restrict__ cnt, int n, int *__restrict__ bsum)
{
    __shared__ int ws[4];
    const long base = (long)blockIdx.x * SCAN_CHUNK + (long)threadIdx.x * SCAN_ITEMS;
    int s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; ++j)
        if (base + j < n) s += cnt[base + j];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

// Exclusive scan of the nb block sums in place (one block); total -> *total.
__global__ __launch_bounds__(1024) void k_scan_top(int *__restrict__ bsum, int nb, int *__restrict__ total)
{
    __shared__ int part[1024];
    const int per = (nb + 1023) / 1024;
    const int a = threadIdx.x * per, b = min(a + per, nb);
    int s = 0;
    for (int i = a; i < b; ++i) s += bsum[i];
    part[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int t = 0; t < 1024; ++t) {
            const int v = part[t];
            part[t] = run;
            run += v;
        }
        *total = run;
    }
    __syncthreads();
    int run = part[threadIdx.x];
    for (int i = a; i < b; ++i) {
        const int v = bsum[i];
        bsum[i] = run;
        run += v;
    }
}

// ptr[q + 1] = sum of cnt[0..q] (ptr[0] = 0 is set by the caller); flags an
// equation that no slot touches (2) or more than PF_SLOT8 do (4).
__global__ __launch_bounds__(256) void k_scan_apply(const int *__restrict__ cnt, int n, const int *__restrict__ boff,
                                                   int *__restrict__ ptr, int *__restrict__ err)
{
    __shared__ int ts[256];
    const long base = (long)blockIdx.x * SCAN_CHUNK + (long)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    int s = 0;
    bool many = false;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; ++j) {
        v[j] = base + j < n ? cnt[base + j] : 0;
        if (base + j < n && v[j] == 0) atomicOr(err, 2);
        if (v[j] > PF_SLOT8) many = true;
        s += v[j];
    }
    ts[threadIdx.x] = s;
    if (__syncthreads_or(many) && threadIdx.x == 0) atomicOr(err, 4);
    // inclusive scan of the 256 thread sums (Hillis-Steele)
    for (int off = 1; off < 256; off <<= 1) {
        const int add = threadIdx.x >= off ? ts[threadIdx.x - off] : 0;
        __syncthreads();
        ts[threadIdx.x] += add;
        __syncthreads();
    }
    int run = boff[blockIdx.x] + ts[threadIdx.x] - s;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; ++j) {
        run += v[j];
        if (base + j < n) ptr[base + j + 1] = run;
    }
}

__global__ __launch_bounds__(256) void k_csr_fill(const int *__restrict__ gg, long nslot, int *__restrict__ cursor,
                                                 int *__restrict__ slot)
{
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < nslot; k += (long)gridDim.x * blockDim.x) {
        const int g = gg[k];
        if (g) slot[atomicAdd(&cursor[g - 1], 1)] = (int)k;
    }
}

// slot[a..b) in ascending order: insertion sort of a short list.
__device__ __forceinline__ void sort_slots(int *__restrict__ slot, int a, int b)
{
    for (int i = a + 1; i < b; ++i) {
        const int v = slot[i];
        int j = i - 1;
        while (j >= a && slot[j] > v) {
            slot[j + 1] = slot[j];
            --j;
        }
        slot[j + 1] = v;
    }
}

// Each equation's slots in ascending order, and, with slot8, their copy in the
// padded table.
__global__ __launch_bounds__(256) void k_csr_sort(const int *__restrict__ ptr, int *__restrict__ slot, int neq,
                                                 int *__restrict__ slot8)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= neq) return;
    const int a = ptr[q], b = ptr[q + 1];
    sort_slots(slot, a, b);
    if (slot8)
        for (int j = 0; j < PF_SLOT8; ++j) slot8[(long)j * neq + q] = a + j < b ? slot[a + j] : -1;
}

// slot_t[s] = i*nels + e for slot[s] = e*ntot + i: where the iteration's
// products of a hex8 mesh keep row i of element e (all elements' row i side
// by side, so the scatter's reads of one slot across consecutive equations
// fall on consecutive words).  The list order is unchanged.
__global__ __launch_bounds__(256) void k_csr_transpose(const int *__restrict__ slot, long nnz, int ntot, int nels,
                                                       int *__restrict__ slot_t)
{
    for (long s = (long)blockIdx.x * blockDim.x + threadIdx.x; s < nnz; s += (long)gridDim.x * blockDim.x) {
        const int v = slot[s], e = v / ntot, i = v - e * ntot;
        slot_t[s] = i * nels + e;
    }
}

// g_g(i, iel) = nf(d, g_num(n, iel)) for element node n, freedom d, i = n*nodof + d.
__global__ __launch_bounds__(256) void k_steer_gather(const int *__restrict__ g_num, const int *__restrict__ nf,
                                                     int *__restrict__ gg, long nslot, int nod, int nodof)
{
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < nslot; k += (long)gridDim.x * blockDim.x) {
        const long e = k / (nod * nodof);
        const int i = (int)(k - e * nod * nodof);
        const int node = g_num[e * nod + i / nodof];
        gg[k] = nf[(long)(node - 1) * nodof + i % nodof];
    }
}

// Slots per node; *many and its copy on the device are set where a node has more
// than the sorts take.
__global__ __launch_bounds__(256) void k_node_count(const int *__restrict__ g_num, int ns, int nn,
                                                   int *__restrict__ cnt, int *__restrict__ many,
                                                   int *__restrict__ dmany)
{
    for (long s = (long)blockIdx.x * blockDim.x + threadIdx.x; s < ns; s += (long)gridDim.x * blockDim.x) {
        const int g = g_num[s];
        if (g >= 1 && g <= nn && atomicAdd(&cnt[g - 1], 1) == PF_NODE_LONG) *many = *dmany = 1;
    }
}

// Every slot into its node's list, the counts used up as cursors.
__global__ __launch_bounds__(256) void k_node_fill(const int *__restrict__ g_num, int ns, int nn,
                                                  const int *__restrict__ ptr, int *__restrict__ cnt,
                                                  int *__restrict__ slot)
{
    for (long s = (long)blockIdx.x * blockDim.x + threadIdx.x; s < ns; s += (long)gridDim.x * blockDim.x) {
        const int g = g_num[s];
        if (g >= 1 && g <= nn) slot[ptr[g - 1] + atomicSub(&cnt[g - 1], 1) - 1] = (int)s;
    }
}

// Ascending order of the short lists, a thread each (quadratic in the length);
// the nodes of the longer ones are noted.
__global__ __launch_bounds__(256) void k_node_sort(const int *__restrict__ ptr, int *__restrict__ slot, int nn,
                                                  int *__restrict__ longs, int *__restrict__ nlong)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nn) return;
    const int a = ptr[n], b = ptr[n + 1];
    if (b - a <= PF_NODE_SORT) sort_slots(slot, a, b);
    else if (b - a <= PF_NODE_LONG) longs[atomicAdd(nlong, 1)] = n;
}

// Ascending order of the longer lists, a workgroup each: every slot to the place
// that the number of smaller ones gives.
constexpr int LONG_T = 1024;
__global__ __launch_bounds__(LONG_T) void k_node_sort_long(const int *__restrict__ ptr, int *__restrict__ slot,
                                                       const int *__restrict__ longs, const int *__restrict__ nlong)
{
    __shared__ int s[PF_NODE_LONG];
    const int nl = *nlong;
    for (int l = blockIdx.x; l < nl; l += gridDim.x) {
        const int a = ptr[longs[l]], n = ptr[longs[l] + 1] - a;
        for (int i = threadIdx.x; i < n; i += LONG_T) s[i] = slot[a + i];
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += LONG_T) {
            const int v = s[i];
            int rank = 0;
#pragma unroll 8
            for (int j = 0; j < n; ++j) rank += s[j] < v;
            slot[a + rank] = v;
        }
        __syncthreads();   // the list is read before the next one is written
    }
}

// *bad is set where an entry of g_num is not a node.
__global__ __launch_bounds__(256) void k_num_check(const int *__restrict__ g_num, long n, int nn, int *__restrict__ bad)
{
    bool b = false;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x)
        b |= g_num[k] < 1 || g_num[k] > nn;
    if (b) *bad = 1;
}

// The last restraint row of every node (row + 1; 0: none), *bad where a row
// names no node.
__global__ __launch_bounds__(256) void k_rest_last(const int *__restrict__ rest, int nr, int nodof, int nn,
                                                  int *__restrict__ last, int *__restrict__ bad)
{
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < nr; r += gridDim.x * blockDim.x) {
        const int node = rest[(long)r * (nodof + 1)];
        if (node < 1 || node > nn) *bad = 1;
        else atomicMax(&last[node - 1], r + 1);
    }
}

// Whether each freedom of each node is free.
__global__ __launch_bounds__(256) void k_nf_free(const int *__restrict__ rest, const int *__restrict__ last, int nn,
                                                int nodof, int *__restrict__ nf)
{
    const long n = (long)nn * nodof;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x) {
        const int node = (int)(k / nodof), d = (int)(k - (long)node * nodof), r = last[node];
        nf[k] = r == 0 || rest[(long)(r - 1) * (nodof + 1) + 1 + d] != 0;
    }
}

// Equation numbers from the free freedoms' scan.
__global__ __launch_bounds__(256) void k_nf_number(const int *__restrict__ ptr, long n, int *__restrict__ nf)
{
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x)
        if (nf[k]) nf[k] = ptr[k + 1];
}

// Freedoms of a node list the same elements: the slots of freedom d are those
// of freedom 0 plus d.  Equations past their node's first (the leader) whose
// slots are the leader's plus k, k <= 2; at equation q: k.
__device__ __forceinline__ int node_follow(const int *__restrict__ ptr, const int *__restrict__ slot, int q)
{
    const int d = slot[ptr[q]] % 3;
    int k = 0;
    while (k < d && q - k > 0) {
        const int a = ptr[q - k - 1], b = ptr[q - k], e = ptr[q - k + 1];
        if (e - b != b - a) break;
        bool same = true;
        for (int j = 0; j < e - b; ++j) same &= slot[b + j] == slot[a + j] + 1;
        if (!same) break;
        ++k;
    }
    return k;
}

// The leaders' list lengths (0 for the others) and every equation's code but for
// the offset; *bad where a list is too long for it.
__global__ __launch_bounds__(256) void k_node_leaders(const int *__restrict__ ptr, const int *__restrict__ slot, int neq,
                                                     int *__restrict__ cnt, unsigned *__restrict__ code,
                                                     int *__restrict__ bad)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= neq) return;
    const int n = ptr[q + 1] - ptr[q], k = node_follow(ptr, slot, q);
    if (n > 15) *bad = 1;
    cnt[q] = k ? 0 : n;
    code[q] = (unsigned)n << 2 | (unsigned)k;
}

// The offsets into the codes (off[q + 1]: the leaders' entries up to q) and the
// leaders' slots into the list.
__global__ __launch_bounds__(256) void k_node_lists(const int *__restrict__ ptr, const int *__restrict__ slot,
                                                   const int *__restrict__ off, int neq, unsigned *__restrict__ code,
                                                   int *__restrict__ list)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= neq) return;
    const unsigned c = code[q];
    const int k = c & 3, n = c >> 2, o = off[q - k];
    code[q] = (unsigned)o << 6 | c;
    if (k == 0)
        for (int j = 0; j < n; ++j) list[o + j] = slot[ptr[q] + j];
}

int grid_for_stride(long n) { return (int)std::max<long>(1, std::min<long>((n + 255) / 256, 16384)); }

}  // namespace

int pf_scan_blocks(long n) { return (int)std::max<long>(1, (n + SCAN_CHUNK - 1) / SCAN_CHUNK); }

void pf_scan_launch(pf_ctx *c, const int *cnt, int n, int *bsum, int *ptr, int *total, int *zero_flag)
{
    const int nb = pf_scan_blocks(n);
    hipLaunchKernelGGL(k_scan_sums, dim3(nb), dim3(256), 0, c->stream, cnt, n, bsum);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, c->stream, bsum, nb, total);
    hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(256), 0, c->stream, cnt, n, bsum, ptr, zero_flag);
}

// work: the device's copy of many, the number of longer lists, nn counts (then
// the nodes of the longer lists), the block sums of the scan, its total and its
// flags (unused)
size_t pf_node_work(int nn) { return 2 + (size_t)nn + pf_scan_blocks(nn) + 2; }

void pf_node_slots(pf_ctx *c, const int *g_num, int ns, int nn, int *work, int *ptr, int *slot, int *many)
{
    int *nlong = work + 1, *cnt = work + 2, *bsum = cnt + nn, *total = bsum + pf_scan_blocks(nn);
    (void)hipMemsetAsync(work, 0, ((size_t)nn + 2) * sizeof(int), c->stream);
    (void)hipMemsetAsync(ptr, 0, sizeof(int), c->stream);
    const dim3 gs(grid_for_stride(ns));
    hipLaunchKernelGGL(k_node_count, gs, dim3(256), 0, c->stream, g_num, ns, nn, cnt, many, work);
    pf_scan_launch(c, cnt, nn, bsum, ptr, total, total + 1);
    hipLaunchKernelGGL(k_node_fill, gs, dim3(256), 0, c->stream, g_num, ns, nn, ptr, cnt, slot);
    hipLaunchKernelGGL(k_node_sort, dim3((nn + 255) / 256), dim3(256), 0, c->stream, ptr, slot, nn, cnt, nlong);
    hipLaunchKernelGGL(k_node_sort_long, dim3(64), dim3(LONG_T), 0, c->stream, ptr, slot, cnt, nlong);
}

// Transposed steering of c->g_g (already on the device, c->neq and c->ntot,
// c->nels set) into c->csr_ptr / c->csr_slot; PF_ERR_ARG when an entry is
// outside 0..neq or an equation has no slot.
int pf_csr_build(pf_ctx *c)
{
    const long nslot = (long)c->ntot * c->nels;
    const int neq = c->neq;
    const int nb = (int)((neq + SCAN_CHUNK - 1) / SCAN_CHUNK);
    int *cnt = nullptr, *bsum = nullptr, *flags = nullptr;
    int rc = pf_alloc(c, (void **)&cnt, (size_t)neq * sizeof(int));
    if (!rc) rc = pf_alloc(c, (void **)&bsum, (size_t)std::max(nb, 1) * sizeof(int));
    if (!rc) rc = pf_alloc(c, (void **)&flags, 4 * sizeof(int));   // err, nnz
    auto release = [&]() {
        (void)hipStreamSynchronize(c->stream);
        pf_free(c, cnt, (size_t)neq * sizeof(int));
        pf_free(c, bsum, (size_t)std::max(nb, 1) * sizeof(int));
        pf_free(c, flags, 4 * sizeof(int));
    };
    if (rc) {
        release();
        return rc;
    }
    int host[2] = {0, 0};
    hipError_t he = hipMemsetAsync(cnt, 0, (size_t)neq * sizeof(int), c->stream);
    if (he == hipSuccess) he = hipMemsetAsync(flags, 0, 4 * sizeof(int), c->stream);
    if (he == hipSuccess) he = hipMemsetAsync(c->csr_ptr, 0, sizeof(int), c->stream);
    if (he == hipSuccess) {
        const int gs = grid_for_stride(nslot);
        hipLaunchKernelGGL(k_csr_count, dim3(gs), dim3(256), 0, c->stream, c->g_g, nslot, neq, cnt, flags);
        pf_scan_launch(c, cnt, neq, bsum, c->csr_ptr, flags + 1, flags);
        he = hipGetLastError();
    }
    if (he == hipSuccess) he = hipMemcpyAsync(host, flags, 2 * sizeof(int), hipMemcpyDeviceToHost, c->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
    if (he != hipSuccess) {
        release();
        return pf_set_hip_error(he, "transposed steering", __FILE__, __LINE__);
    }
    if (host[0] & 3) {
        release();
        return PF_ERR_ARG;
    }
    c->nnz = host[1];
    rc = pf_alloc(c, (void **)&c->csr_slot, (size_t)std::max<int64_t>(c->nnz, 1) * sizeof(int));
    if (!rc && c->ntot == 8)
        rc = pf_alloc(c, (void **)&c->csr_slot_t, (size_t)std::max<int64_t>(c->nnz, 1) * sizeof(int));
    if (!rc && !(host[0] & 4) && pf_grid_for(neq) <= PF_FOLD_MAXG)
        rc = pf_alloc(c, (void **)&c->csr_slot8, (size_t)PF_SLOT8 * neq * sizeof(int));
    if (rc) {
        release();
        return rc;
    }
    // the counts become the placement cursors: cursor[q] = ptr[q]
    he = hipMemcpyAsync(cnt, c->csr_ptr, (size_t)neq * sizeof(int), hipMemcpyDeviceToDevice, c->stream);
    if (he == hipSuccess) {
        hipLaunchKernelGGL(k_csr_fill, dim3(grid_for_stride(nslot)), dim3(256), 0, c->stream, c->g_g, nslot, cnt,
                           c->csr_slot);
        hipLaunchKernelGGL(k_csr_sort, dim3((neq + 255) / 256), dim3(256), 0, c->stream, c->csr_ptr, c->csr_slot,
                           neq, c->csr_slot8);
        if (c->csr_slot_t)
            hipLaunchKernelGGL(k_csr_transpose, dim3(grid_for_stride(c->nnz)), dim3(256), 0, c->stream, c->csr_slot,
                               (long)c->nnz, c->ntot, c->nels, c->csr_slot_t);
        he = hipGetLastError();
    }
    if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
    release();
    if (he != hipSuccess) return pf_set_hip_error(he, "transposed steering", __FILE__, __LINE__);
    return c->ntot != 8 && !c->csr_slot8 ? pf_node_lists_build(c) : PF_OK;
}

// The node freedom table and the check of g_num are made on the device from
// STEER_DEVICE element nodes and node freedoms on, by seven small launches; on
// the host they are serial passes over both.  Whole call, host / device:
// 138,275 entries 322 / 356 us, 458,355 515 / 427, 1,076,803 1,206 / 903,
// 8,500,355 11.7 / 5.7 ms.
constexpr long STEER_DEVICE = 1 << 18;

// Builds the table in *dnf behind the upload of g_num to *dnum; *neq is the
// number of equations.  PF_ERR_ARG as the host's passes; PF_ERR_OOM leaves the
// work to them.
static int nf_device(pf_ctx *c, long nslot, int nodof, const int *g_num, int nn, int nr, const int *rest, int *dnum,
                     int *dnf, long *neq)
{
    const long n = (long)nn * nodof;
    const size_t rsz = (size_t)std::max(nr, 1) * (nodof + 1) * sizeof(int), lsz = (size_t)nn * sizeof(int);
    const size_t psz = ((size_t)n + 1) * sizeof(int), bsz = ((size_t)pf_scan_blocks(n) + 1) * sizeof(int);
    int *drest = nullptr, *last = nullptr, *ptr = nullptr, *bsum = nullptr;
    int rc = pf_alloc(c, (void **)&drest, rsz);
    if (!rc) rc = pf_alloc(c, (void **)&last, lsz);
    if (!rc) rc = pf_alloc(c, (void **)&ptr, psz);
    if (!rc) rc = pf_alloc(c, (void **)&bsum, bsz);
    if (!rc) {
        int *bad = pf_flag_word(c), *total = bad + 1;   // both pinned
        hipError_t he = nr ? hipMemcpyAsync(drest, rest, rsz, hipMemcpyHostToDevice, c->stream) : hipSuccess;
        if (he == hipSuccess) he = hipMemsetAsync(last, 0, lsz, c->stream);
        if (he == hipSuccess) {
            if (nr)
                hipLaunchKernelGGL(k_rest_last, dim3(grid_for_stride(nr)), dim3(256), 0, c->stream, drest, nr, nodof, nn,
                                   last, bad);
            hipLaunchKernelGGL(k_nf_free, dim3(grid_for_stride(n)), dim3(256), 0, c->stream, drest, last, nn, nodof, dnf);
            pf_scan_launch(c, dnf, (int)n, bsum, ptr, total, bsum + pf_scan_blocks(n));   // zero counts: not looked at
            hipLaunchKernelGGL(k_nf_number, dim3(grid_for_stride(n)), dim3(256), 0, c->stream, ptr, n, dnf);
            he = hipMemcpyAsync(dnum, g_num, nslot * sizeof(int), hipMemcpyHostToDevice, c->stream);
        }
        if (he == hipSuccess) {
            hipLaunchKernelGGL(k_num_check, dim3(grid_for_stride(nslot)), dim3(256), 0, c->stream, dnum, nslot, nn, bad);
            he = hipGetLastError();
        }
        if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
        if (he != hipSuccess) rc = pf_set_hip_error(he, "node freedoms", __FILE__, __LINE__);
        else if (*bad) rc = PF_ERR_ARG;
        *neq = *total;
    }
    (void)hipStreamSynchronize(c->stream);
    pf_free(c, drest, rsz);
    pf_free(c, last, lsz);
    pf_free(c, ptr, psz);
    pf_free(c, bsum, bsz);
    return rc;
}

// The slot lists of nodes, for element nodes of three freedoms.  They only save
// reads: without the memory, or where a code does not hold a list, none.
int pf_node_lists_build(pf_ctx *c)
{
    const int neq = c->neq;
    const size_t csz = (size_t)neq * sizeof(int), psz = ((size_t)neq + 1) * sizeof(int);
    const size_t bsz = ((size_t)pf_scan_blocks(neq) + 1) * sizeof(int);
    int *cnt = nullptr, *off = nullptr, *bsum = nullptr, *bad = pf_flag_word(c), *total = bad + 1;   // both pinned
    hipError_t he = hipSuccess;
    const dim3 grid((neq + 255) / 256), blk(256);
    bool ok = !pf_alloc(c, (void **)&c->nl_code, csz) && !pf_alloc(c, (void **)&cnt, csz) &&
              !pf_alloc(c, (void **)&off, psz) && !pf_alloc(c, (void **)&bsum, bsz);
    if (ok) {
        hipLaunchKernelGGL(k_node_leaders, grid, blk, 0, c->stream, c->csr_ptr, c->csr_slot, neq, cnt, c->nl_code, bad);
        he = hipMemsetAsync(off, 0, sizeof(int), c->stream);
        pf_scan_launch(c, cnt, neq, bsum, off, total, bsum + pf_scan_blocks(neq));   // zero counts: not looked at
        if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
        ok = he == hipSuccess && !*bad && *total < 1 << 26;
    }
    if (ok) {
        c->nl_n = *total;
        ok = !pf_alloc(c, (void **)&c->nl_slot, (size_t)c->nl_n * sizeof(int));
    }
    if (ok) {
        hipLaunchKernelGGL(k_node_lists, grid, blk, 0, c->stream, c->csr_ptr, c->csr_slot, off, neq, c->nl_code,
                           c->nl_slot);
        he = hipGetLastError();
    }
    if (!ok || he != hipSuccess) {
        pf_free(c, c->nl_code, csz);
        c->nl_code = nullptr;
    }
    pf_free(c, cnt, csz);   // later users of these blocks follow on the same stream
    pf_free(c, off, psz);
    pf_free(c, bsum, bsz);
    return he == hipSuccess ? PF_OK : pf_set_hip_error(he, "node lists", __FILE__, __LINE__);
}

extern "C" int pf_steer_build(pf_ctx *c, int nod, int nels, int nodof, const int *g_num, int nn, int nr,
                              const int *rest, int *neq_out, int *nf_out)
{
    if (!c || !g_num || !neq_out || nod < 1 || nels < 1 || nodof < 1 || nn < 1 || nr < 0 || (nr && !rest))
        return PF_ERR_ARG;
    const long ne = (long)nod * nels, n = (long)nn * nodof;
    const size_t esz = ne * sizeof(int), nsz = n * sizeof(int);
    int *dnum = nullptr, *dnf = nullptr;
    std::vector<int> nf;
    long neq = 0;
    int rc = PF_OK;
    bool on_device = ne + n >= STEER_DEVICE && n < INT32_MAX;
    if (on_device) {
        PF_HIP(hipSetDevice(c->device));
        rc = pf_alloc(c, (void **)&dnum, esz);
        if (!rc) rc = pf_alloc(c, (void **)&dnf, nsz);
        if (!rc) rc = nf_device(c, ne, nodof, g_num, nn, nr, rest, dnum, dnf, &neq);
        if (!rc && neq < 1) rc = PF_ERR_ARG;
        if (rc) {
            pf_free(c, dnum, esz);
            pf_free(c, dnf, nsz);
            dnum = dnf = nullptr;
            if (rc != PF_ERR_OOM) return rc;
            on_device = false;
        }
    }
    if (!on_device) {
        // node freedom table on the host: ascending node, then freedom; nodes
        // without a rest row are free; a later row for a node overrides an
        // earlier one
        nf.assign((size_t)n, 1);
        for (int r = 0; r < nr; ++r) {
            const int *row = rest + (size_t)r * (nodof + 1);
            if (row[0] < 1 || row[0] > nn) return PF_ERR_ARG;
            for (int d = 0; d < nodof; ++d) nf[(size_t)(row[0] - 1) * nodof + d] = row[1 + d] != 0;
        }
        for (auto &v : nf) v = v ? (int)++neq : 0;
        if (neq < 1 || neq >= INT32_MAX) return PF_ERR_ARG;
        for (long k = 0; k < ne; ++k)
            if (g_num[k] < 1 || g_num[k] > nn) return PF_ERR_ARG;
    }
    rc = pf_steer_install(c, nod * nodof, nels, (int)neq);
    if (rc) {
        pf_free(c, dnum, esz);
        pf_free(c, dnf, nsz);
        return rc;
    }
    // g_g gathered on the device, then the transposed steering
    const long nslot = ne * nodof;
    if (!on_device) rc = pf_alloc(c, (void **)&dnum, esz);
    if (!rc && !on_device) rc = pf_alloc(c, (void **)&dnf, nsz);
    if (!rc) {
        hipError_t he = hipSuccess;
        if (!on_device) he = hipMemcpyAsync(dnum, g_num, esz, hipMemcpyHostToDevice, c->stream);
        if (he == hipSuccess && !on_device) he = hipMemcpyAsync(dnf, nf.data(), nsz, hipMemcpyHostToDevice, c->stream);
        if (he == hipSuccess) {
            hipLaunchKernelGGL(k_steer_gather, dim3(grid_for_stride(nslot)), dim3(256), 0, c->stream, dnum, dnf,
                               c->g_g, nslot, nod, nodof);
            he = hipGetLastError();
        }
        if (he == hipSuccess && !on_device) he = hipStreamSynchronize(c->stream);
        if (he != hipSuccess) rc = pf_set_hip_error(he, "steering", __FILE__, __LINE__);
    }
    // (later users of these blocks follow on the same stream)
    pf_free(c, dnum, esz);
    auto take_nf = [&](int *out) {
        hipError_t he = hipMemcpyAsync(out, dnf, nsz, hipMemcpyDeviceToHost, c->stream);
        if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
        if (he != hipSuccess) rc = pf_set_hip_error(he, "node freedoms", __FILE__, __LINE__);
    };
    if (!on_device) {
        pf_free(c, dnf, nsz);
        dnf = nullptr;
    }
    if (!rc) rc = pf_csr_build(c);
    if (rc == PF_ERR_OOM && on_device) {
        // without the table's memory: it waits on the host
        nf.resize((size_t)n);
        rc = PF_OK;
        take_nf(nf.data());
        pf_free(c, dnf, nsz);
        dnf = nullptr;
        on_device = false;
        pf_csr_drop(c);
        if (!rc) rc = pf_csr_build(c);
    }
    if (!rc && nf_out && on_device) take_nf(nf_out);
    pf_free(c, dnf, nsz);
    if (rc) {
        pf_steer_drop(c);
        return rc;
    }
    *neq_out = (int)neq;
    if (nf_out && !on_device) std::copy(nf.begin(), nf.end(), nf_out);
    return PF_OK;
}

extern "C" int pf_steer_get(pf_ctx *c, int *g_g_pp)
{
    if (!c || !g_g_pp) return PF_ERR_ARG;
    if (!c->g_g) return PF_ERR_STATE;
    PF_HIP(hipMemcpyAsync(g_g_pp, c->g_g, (size_t)c->ntot * c->nels * sizeof(int), hipMemcpyDeviceToHost,
                          c->stream));
    PF_HIP(hipStreamSynchronize(c->stream));
    return PF_OK;
}
