// assemble.hip -- triplet assembly of uploaded subdomain matrices on the
// device (src/module_sm.f90:630-685): entries sorted by row and column,
// duplicates summed in input order, so that the result has the bits of the
// host assembly.  Batched over the subdomains of a flush (blockIdx.y).
//
// A counting sort places (column, input index) keys row by row -- in any
// order within a row, by integer atomics -- and a rank sort orders each row's
// few keys (they are distinct, so the ranks do not depend on that order).
// One wave per row: rows are 30 to 200 entries long; the few that are longer
// than 512 are merge-sorted by a workgroup each.  Eight subdomains of
// 147,456 triplets take 0.33 ms (latency-bound: scattered 8-byte accesses and
// integer atomics), while the host copies the next ones: an upload takes 0.15
// ms of host time where its assembly by 16 host threads took 0.30 ms.
#include "kernels.hpp"

namespace bddc {

constexpr int ASM_THR = 256;    // 4 waves
constexpr int ASM_LDS = 512;    // keys of a row staged in LDS (longer rows: k_asm_sort_long)
constexpr int ASM_DUP = 32;     // duplicates that one lane sums

__global__ void k_asm_zero(const AsmSub *__restrict__ subs) {
  const AsmSub d = subs[blockIdx.y];
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < d.nd; r += gridDim.x * blockDim.x) d.cur[r] = 0;
}

__global__ void k_asm_count(const AsmSub *__restrict__ subs) {
  const AsmSub d = subs[blockIdx.y];
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < d.n; k += gridDim.x * blockDim.x)
    atomicAdd(&d.cur[d.i[k] - d.b], 1);
}

// ptr = exclusive sums of cur over the nd rows (ptr[nd] the total), one
// workgroup of 1024 threads per subdomain; which 0: ptr = rowp and cur is
// set to it (the next free place of each row); 1: ptr = uptr, the total is
// info->nnz; 2: ptr = bptr, the total is info->nbc
__global__ __launch_bounds__(1024) void k_asm_scan(const AsmSub *__restrict__ subs, int which) {
  __shared__ int wsum[16];
  __shared__ int carry;
  const AsmSub d = subs[blockIdx.x];
  int *ptr = which == 0 ? d.rowp : which == 1 ? d.uptr : d.bptr;
  if (!ptr) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (threadIdx.x == 0) carry = 0;
  for (int r0 = 0; r0 < d.nd; r0 += 1024) {
    const int r = r0 + threadIdx.x;
    const int v = r < d.nd ? d.cur[r] : 0;
    int s = v;  // inclusive sum over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(s, o);
      if (lane >= o) s += t;
    }
    if (lane == 63) wsum[w] = s;
    __syncthreads();
    int base = carry;
    for (int q = 0; q < w; q++) base += wsum[q];
    if (r < d.nd) {
      ptr[r] = base + s - v;
      if (which == 0) d.cur[r] = base + s - v;
    }
    __syncthreads();
    if (threadIdx.x == 1023) carry = base + s;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    ptr[d.nd] = carry;
    if (which == 1) d.info->nnz = carry, d.info->hash = 0;
    if (which == 2) d.info->nbc = carry;
  }
}

__global__ void k_asm_place(const AsmSub *__restrict__ subs) {
  const AsmSub d = subs[blockIdx.y];
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < d.n; k += gridDim.x * blockDim.x) {
    const int p = atomicAdd(&d.cur[d.i[k] - d.b], 1);
    d.key[p] = (uint64_t)(uint32_t)(d.j[k] - d.b) << 32 | (uint32_t)k;
  }
}

// the keys of every row of up to ASM_LDS ordered by rank into key2;
// cur[row] = its distinct columns
__global__ __launch_bounds__(ASM_THR) void k_asm_sort(const AsmSub *__restrict__ subs) {
  __shared__ uint64_t sh[ASM_THR / 64][ASM_LDS];
  const AsmSub d = subs[blockIdx.y];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int step = gridDim.x * (ASM_THR / 64);
  // every wave of the workgroup takes the same number of rounds (barriers)
  for (int r0 = blockIdx.x * (ASM_THR / 64); r0 < d.nd; r0 += step) {
    const int r = r0 + w;
    const int p0 = r < d.nd ? d.rowp[r] : 0, n = r < d.nd ? d.rowp[r + 1] - p0 : 0;
    const bool mine = n <= ASM_LDS;
    const int len = mine ? n : 0;
    const uint64_t *K = d.key + p0;
    __syncthreads();
    for (int q = lane; q < len; q += 64) sh[w][q] = K[q];
    __syncthreads();
    int heads = 0;
    for (int q0 = 0; q0 < len; q0 += 64) {
      const int q = q0 + lane;
      const bool live = q < len;
      const uint64_t own = live ? sh[w][q] : ~0ull;
      int rank = 0;
      bool first = true;  // no smaller key of the same column
      for (int t = 0; t < len; t++) {
        const uint64_t k = sh[w][t];
        const bool less = k < own;
        rank += less;
        first = first && !(less && (k >> 32) == (own >> 32));
      }
      if (live) d.key2[p0 + rank] = own;
      heads += __popcll(__ballot(live && first));
    }
    if (r < d.nd && mine && lane == 0) d.cur[r] = heads;
  }
}

// longer rows (dofs coupled to many others, many duplicates): a merge sort by
// one workgroup a row.  Runs of ASM_RUN keys are ordered by rank in LDS, then
// pairs of runs merged, key and key2 in turn: a key's place is its place in its
// own run plus the smaller keys of the other, by binary search.  A row of
// 20,000 triplets added to a small problem cost 590 ms by ranks over the whole
// row, one of 8,000 95 ms; now 3.8 and 1.2 ms with their sums, one of 200,000
// 25 ms.
constexpr int ASM_RUN = 1024;
constexpr int ASM_SCAN = 64;  // rows a workgroup looks through at a time
__global__ __launch_bounds__(ASM_RUN) void k_asm_sort_long(const AsmSub *__restrict__ subs) {
  __shared__ uint64_t sh[ASM_RUN];
  __shared__ int list[ASM_SCAN];
  __shared__ int nlist, heads;
  const AsmSub d = subs[blockIdx.y];
  const int tid = threadIdx.x;
  for (int r0 = blockIdx.x * ASM_SCAN; r0 < d.nd; r0 += gridDim.x * ASM_SCAN) {
    if (tid < 64) {  // one wave: the long ones of these rows
      const int r = r0 + tid;
      const bool is_long = r < d.nd && d.rowp[r + 1] - d.rowp[r] > ASM_LDS;
      const unsigned long long m = __ballot(is_long);
      if (is_long) list[__popcll(m & ((1ull << tid) - 1))] = r;
      if (tid == 0) nlist = __popcll(m);
    }
    __syncthreads();
    const int nl = nlist;
    for (int k = 0; k < nl; k++) {
      const int r = list[k], p0 = d.rowp[r], len = d.rowp[r + 1] - p0;
      int levels = 0;
      while ((int64_t)ASM_RUN << levels < len) levels++;
      uint64_t *src = d.key + p0, *dst = d.key2 + p0;
      if (levels & 1) dst = src;  // the last merge writes key2
      for (int s0 = 0; s0 < len; s0 += ASM_RUN) {
        const int n = min(ASM_RUN, len - s0);
        const uint64_t own = tid < n ? src[s0 + tid] : ~0ull;
        sh[tid] = own;
        __syncthreads();
        int rank = 0;
#pragma unroll 8
        for (int t = 0; t < n; t++) rank += sh[t] < own;
        if (tid < n) dst[s0 + rank] = own;
        __syncthreads();
      }
      for (int l = 0; l < levels; l++) {
        const int w = ASM_RUN << l;  // below len: no overflow
        src = dst;
        dst = src == d.key + p0 ? d.key2 + p0 : d.key + p0;
        __threadfence_block();
        __syncthreads();
        for (int q = tid; q < len; q += ASM_RUN) {
          const uint64_t own = src[q];
          const int run = q & ~(w - 1), first = run & w ? run - w : run;  // of its run, of its pair
          const int64_t o0 = run == first ? (int64_t)run + w : first;
          int lo = (int)min(o0, (int64_t)len), hi = (int)min(o0 + w, (int64_t)len);
          const int o = lo;
          while (lo < hi) {
            const int mid = lo + (hi - lo) / 2;
            if (src[mid] < own) lo = mid + 1;
            else hi = mid;
          }
          dst[first + (q - run) + (lo - o)] = own;
        }
      }
      if (tid == 0) heads = 0;
      __threadfence_block();
      __syncthreads();
      int h = 0;
      for (int q = tid; q < len; q += ASM_RUN) h += q == 0 || dst[q] >> 32 != dst[q - 1] >> 32;
      if (h) atomicAdd(&heads, h);
      __syncthreads();
      if (tid == 0) d.cur[r] = heads;
    }
    __syncthreads();  // list and nlist are read before they are set again
  }
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// the assembled entries: one wave per row, the first lane of each column
// sums its duplicates in input order; info->hash = sum of a hash of every
// (row, column), whatever the order of the rows.  Also diag (0 where a row has
// no diagonal entry: it leads its row in the upper triangle) and, where the
// subdomain has fixed dofs (bptr), the row's entries that touch one: cur
__global__ __launch_bounds__(ASM_THR) void k_asm_sum(const AsmSub *__restrict__ subs) {
  const AsmSub d = subs[blockIdx.y];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint64_t h = 0;
  for (int r = blockIdx.x * (ASM_THR / 64) + w; r < d.nd; r += gridDim.x * (ASM_THR / 64)) {
    const int p0 = d.rowp[r], p1 = d.rowp[r + 1];
    int o = d.uptr[r], nbc = 0;
    const bool fr = d.bptr && d.fix[r] != 0;
    if (p0 == p1 && lane == 0) d.diag[r] = 0.0;
    for (int q0 = p0; q0 < p1; q0 += 64) {
      const int q = q0 + lane;
      const bool live = q < p1;
      const uint64_t k = live ? d.key2[q] : 0;
      const uint32_t j = (uint32_t)(k >> 32);
      const bool head = live && (q == p0 || (uint32_t)(d.key2[q - 1] >> 32) != j);
      const unsigned long long m = __ballot(head);
      double s = 0.0;
      int t = q + 1;
      bool more = false;
      if (head) {
        s = d.a[(uint32_t)k];
        const int e = min(q + ASM_DUP, p1);
        for (; t < e; t++) {
          const uint64_t kt = d.key2[t];
          if ((uint32_t)(kt >> 32) != j) break;
          s += d.a[(uint32_t)kt];
        }
        more = t == q + ASM_DUP && t < p1 && (uint32_t)(d.key2[t] >> 32) == j;
      }
      // longer sums, one after the other: the wave reads 64 values at a time,
      // added in the same order
      for (unsigned long long left = __ballot(more); left; left &= left - 1) {
        const int src = __builtin_ctzll(left);
        const uint32_t js = __shfl(j, src);
        double sum = __shfl(s, src);
        int u0 = __shfl(t, src), n = 64;
        for (; n == 64; u0 += 64) {
          const int u = u0 + lane;
          const uint64_t ku = u < p1 ? d.key2[u] : 0;
          const bool in = u < p1 && (uint32_t)(ku >> 32) == js;
          const double v = in ? d.a[(uint32_t)ku] : 0.0;
          n = __popcll(__ballot(in));  // of sorted keys: the first n lanes
          for (int c = 0; c < n; c++) sum += __shfl(v, c);
        }
        if (lane == src) s = sum;
      }
      if (head) {
        const int e = o + __popcll(m & ((1ull << lane) - 1));
        d.ai[e] = r;
        d.aj[e] = (int)j;
        d.av[e] = s;
        h += mix64((uint64_t)(uint32_t)r << 32 | j);
        if (q == p0) d.diag[r] = (int)j == r ? s : 0.0;
      }
      o += __popcll(m);
      if (d.bptr) nbc += __popcll(__ballot(head && (fr || d.fix[j] != 0)));
    }
    if (d.bptr && lane == 0) d.cur[r] = nbc;
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) h += __shfl_xor((unsigned long long)h, s);
  if (lane == 0 && h) atomicAdd((unsigned long long *)&d.info->hash, (unsigned long long)h);
}

// the entries that touch a fixed dof, in order
__global__ __launch_bounds__(ASM_THR) void k_asm_fixed(const AsmSub *__restrict__ subs) {
  const AsmSub d = subs[blockIdx.y];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int r = blockIdx.x * (ASM_THR / 64) + w; r < d.nd; r += gridDim.x * (ASM_THR / 64)) {
    int o = d.bptr[r];
    if (o == d.bptr[r + 1]) continue;
    const int p0 = d.uptr[r], p1 = d.uptr[r + 1];
    const bool fr = d.fix[r] != 0;
    for (int q0 = p0; q0 < p1; q0 += 64) {
      const int q = q0 + lane;
      const bool in = q < p1 && (fr || d.fix[d.aj[q]] != 0);
      const unsigned long long m = __ballot(in);
      if (in) {
        const int e = o + __popcll(m & ((1ull << lane) - 1));
        d.bi[e] = r;
        d.bj[e] = d.aj[q];
        d.ba[e] = d.av[q];
      }
      o += __popcll(m);
    }
  }
}

__global__ __launch_bounds__(256) void k_gather_ranges(const GatherRange *__restrict__ g,
                                                       char *__restrict__ dst) {
  const GatherRange r = g[blockIdx.y];
  const int *s = static_cast<const int *>(r.src);
  int *d = reinterpret_cast<int *>(dst + r.off);
  for (int64_t k = blockIdx.x * 256 + threadIdx.x; k < r.bytes / 4; k += gridDim.x * 256) d[k] = s[k];
}
void launch_gather_ranges(hipStream_t st, const GatherRange *g, int n, char *dst) {
  for (int k = 0; k < n; k += 65535)
    hipLaunchKernelGGL(k_gather_ranges, dim3(32, std::min(n - k, 65535)), dim3(256), 0, st, g + k, dst);
}

static unsigned row_grid(int maxnd) {
  return (unsigned)std::min((maxnd + 15) / 16, 1024);  // 4 rows a wave or more
}
void launch_sort_triplets(hipStream_t st, const AsmSub *subs, int nsub, int maxn, int maxnd) {
  if (nsub <= 0) return;
  const unsigned gn = (unsigned)std::min((maxn + 1023) / 1024, 256);
  hipLaunchKernelGGL(k_asm_zero, dim3((maxnd + 255) / 256, nsub), dim3(256), 0, st, subs);
  hipLaunchKernelGGL(k_asm_count, dim3(gn, nsub), dim3(256), 0, st, subs);
  hipLaunchKernelGGL(k_asm_scan, dim3(nsub), dim3(1024), 0, st, subs, 0);
  hipLaunchKernelGGL(k_asm_place, dim3(gn, nsub), dim3(256), 0, st, subs);
  hipLaunchKernelGGL(k_asm_sort, dim3(row_grid(maxnd), nsub), dim3(ASM_THR), 0, st, subs);
  hipLaunchKernelGGL(k_asm_sort_long, dim3(std::min((maxnd + ASM_SCAN - 1) / ASM_SCAN, 256), nsub),
                     dim3(ASM_RUN), 0, st, subs);
  hipLaunchKernelGGL(k_asm_scan, dim3(nsub), dim3(1024), 0, st, subs, 1);
}
void launch_sum_triplets(hipStream_t st, const AsmSub *subs, int nsub, int maxnd) {
  if (nsub <= 0) return;
  hipLaunchKernelGGL(k_asm_sum, dim3(row_grid(maxnd), nsub), dim3(ASM_THR), 0, st, subs);
  hipLaunchKernelGGL(k_asm_scan, dim3(nsub), dim3(1024), 0, st, subs, 2);
}
void launch_assembled_fixed(hipStream_t st, const AsmSub *subs, int nsub, int maxnd) {
  if (nsub <= 0) return;
  hipLaunchKernelGGL(k_asm_fixed, dim3(row_grid(maxnd), nsub), dim3(ASM_THR), 0, st, subs);
}

}  // namespace bddc
