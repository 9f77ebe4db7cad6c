// Mesh setup on the device: the block-CSR pattern of the FSILS lhs (what
// lhsa builds, lhsa.cpp:153-380, handed to fsils_lhs_create, lhs.cpp:57-120)
// and the element colouring, colour order and the element entries of each block
// slot that the assembly gathers (do_assem's search, lhsa.cpp:123-134, the other
// way round).
//
// Pattern: every element contributes its 16 node pairs and every node its
// diagonal pair as a 64-bit key row * nNo + col; one radix sort and one
// unique pass leave the keys in CSR order (rows ascending, columns strictly
// increasing in a row) — the same rowPtr/colPtr as the host build.
//
// Colouring: Jones-Plassmann. Each element has a fixed pseudo-random
// priority; in each round an uncoloured element whose priority is the
// largest among the uncoloured elements at all four of its nodes (their
// "head") takes the smallest colour not yet used at its nodes (per-node
// 256-bit masks). Winners of a round share no node, so no two elements of a
// colour share a node, and the result is the sequential greedy colouring in
// decreasing priority order. A round looks only at the nodes whose head
// changed in the round before (k_jp_round). The colour order is a stable radix
// sort of the element ids by colour.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "svg_device.h"

namespace svg {

namespace {

constexpr int CW = 4;  // 64-bit words of a node's used-colour mask (256 colours)

__global__ __launch_bounds__(256) void k_check_ien(long long n, const int* __restrict__ ien, int nNo,
                                                   int* __restrict__ err)
{
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int a = ien[q];
  if (a < 0 || a >= nNo) atomicOr(err, 1);
}

__global__ __launch_bounds__(256) void k_pair_keys(int nEl, int nNo, const int4* __restrict__ ien,
                                                   unsigned long long* __restrict__ keys)
{
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nPair = 16LL * nEl;
  if (t < nPair) {
    const int e = (int)(t >> 4), a = (int)((t >> 2) & 3), b = (int)(t & 3);
    const int4 v = ien[e];
    const int na = a == 0 ? v.x : a == 1 ? v.y : a == 2 ? v.z : v.w;
    const int nb = b == 0 ? v.x : b == 1 ? v.y : b == 2 ? v.z : v.w;
    keys[t] = (unsigned long long)na * (unsigned)nNo + (unsigned)nb;
  } else if (t < nPair + nNo) {
    const unsigned long long a = (unsigned long long)(t - nPair);
    keys[t] = a * (unsigned)nNo + a;
  }
}

// Unique sorted keys -> colPtr, rowPtr (first entry of each row; every row
// holds its diagonal), diagPtr.
__global__ __launch_bounds__(256) void k_csr_from_keys(int nnz, int nNo, const unsigned long long* __restrict__ keys,
                                                       int* __restrict__ rowPtr, int* __restrict__ colPtr,
                                                       int* __restrict__ diagPtr)
{
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const unsigned long long key = keys[k];
  const int r = (int)(key / (unsigned)nNo), c = (int)(key - (unsigned long long)r * (unsigned)nNo);
  colPtr[k] = c;
  if (k == 0 || (int)(keys[k - 1] / (unsigned)nNo) != r) rowPtr[r] = k;
  if (c == r) diagPtr[r] = k;
  if (k == nnz - 1) rowPtr[nNo] = nnz;
}

__device__ __forceinline__ unsigned mix32(unsigned x)
{
  // a 32-bit integer hash (the murmur3 finaliser)
  x ^= x >> 16;
  x *= 0x85ebca6bu;
  x ^= x >> 13;
  x *= 0xc2b2ae35u;
  x ^= x >> 16;
  return x;
}

// An element's priority: a bijection of its id, so no two are equal.
__device__ __forceinline__ unsigned prio(int e) { return mix32((unsigned)e * 2654435761u + 0x9e3779b9u); }

// Heads: per node and round parity, (round the node's head last changed << 32)
// | element, kNoElem when every element of the node is coloured. A node's head
// changes at most once a round, into the slot of the round's parity, so a
// reader in round r finds the head before r in the newer of the two slots
// unless a winner of round r already replaced it (stamp r), and then the node
// is taken.
constexpr unsigned kNoElem = 0xffffffffu;

// The uncoloured element other than `won` of the highest priority among
// entries [c0, c1) of a node's element list (clist: 16 e + 4 a + b), by the
// four lanes of a quad (each every fourth entry, 8 loads in flight).
__device__ __forceinline__ unsigned jp_scan(const int* __restrict__ clist, int c0, int c1, const int* color, int won,
                                            int quad)
{
  unsigned best = kNoElem, bp = 0;
  for (int c = c0 + quad; c < c1; c += 32) {
    int e[8], col[8];
#pragma unroll
    for (int q = 0; q < 8; q++) e[q] = c + 4 * q < c1 ? clist[c + 4 * q] >> 4 : -1;
#pragma unroll
    for (int q = 0; q < 8; q++) col[q] = e[q] >= 0 && e[q] != won ? color[e[q]] : 0;
#pragma unroll
    for (int q = 0; q < 8; q++)
      if (col[q] < 0 && (best == kNoElem || prio(e[q]) > bp)) best = (unsigned)e[q], bp = prio(e[q]);
  }
#pragma unroll
  for (int o = 1; o < 4; o <<= 1) {
    const unsigned ob = __shfl_xor(best, o, 4), op = __shfl_xor(bp, o, 4);
    if (ob != kNoElem && (best == kNoElem || op > bp)) best = ob, bp = op;
  }
  return best;
}

// Every node's first head (round 1) and the first list of changed nodes: all.
__global__ __launch_bounds__(256) void k_jp_heads(int nNo, const int* __restrict__ diagPtr,
                                                  const int* __restrict__ cptr, const int* __restrict__ clist,
                                                  const int* __restrict__ color, unsigned long long* __restrict__ head,
                                                  int* __restrict__ list, int* __restrict__ cnt)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x, v = t >> 2;
  if (v >= nNo) return;
  const int s = diagPtr[v];
  const unsigned e = jp_scan(clist, cptr[s], cptr[s + 1], color, -1, t & 3);
  if ((t & 3) == 0) {
    head[2 * (size_t)v] = kNoElem;
    head[2 * (size_t)v + 1] = (1ull << 32) | e;
    list[v] = v;
    if (v == 0) cnt[0] = 0, cnt[1] = nNo, cnt[2] = 0;
  }
}

// Round r: 16 lanes per node of `list` (the nodes whose head changed in round
// r - 1), four per node of its head element e. e wins when it heads all four
// of its nodes; of the nodes that changed, the first in e's order handles it.
// The winner takes its colour, and its nodes' new heads (slots of parity r) go
// to the next list. Lists' lengths rotate through three counters: read
// (r - 1), written (r), cleared for the next round. The counter is added to
// once per 64 nodes: one atomic per node on the one address, 5 ns each, took
// 148 us per round on the 1.2M-tet pipe. What is left is the chain of
// dependent loads (list, element, heads, masks, colours).
constexpr int JP_G = 64;  // nodes per workgroup and pass

__global__ __launch_bounds__(16 * JP_G) void k_jp_round(int r, const int4* __restrict__ ien,
                                                        const int* __restrict__ diagPtr, const int* __restrict__ cptr,
                                                        const int* __restrict__ clist, int* color,
                                                        unsigned long long* head,
                                                        unsigned long long* __restrict__ used,
                                                        const int* __restrict__ list, int* __restrict__ next,
                                                        int* __restrict__ cnt, int* __restrict__ maxColor,
                                                        int* __restrict__ err)
{
  __shared__ int push[4 * JP_G], nPush, at;
  const int n = cnt[(r - 1) % 3];
  if (blockIdx.x == 0 && threadIdx.x == 0) cnt[(r + 1) % 3] = 0;
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 4, a = (threadIdx.x >> 2) & 3, quad = threadIdx.x & 3;
  const unsigned long long group = 0xffffull << (lane & 48);
  for (int q0 = blockIdx.x * JP_G; q0 < n; q0 += gridDim.x * JP_G) {
    if (threadIdx.x == 0) nPush = 0;
    __syncthreads();
    // whole groups of 16 lanes take part or do not
    const int q = q0 + g;
    const int v = q < n ? list[q] : 0;
    const unsigned e = q < n ? (unsigned)head[2 * (size_t)v + ((r - 1) & 1)] : kNoElem;
    if (e != kNoElem) {
      const int4 w = ien[e];
      const int m = a == 0 ? w.x : a == 1 ? w.y : a == 2 ? w.z : w.w;
      const unsigned long long hp = head[2 * (size_t)m + ((r - 1) & 1)];
      const unsigned long long hc =
          __hip_atomic_load(head + 2 * (size_t)m + (r & 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool changed = (int)(hp >> 32) == r - 1;
      const bool heads = (int)(hc >> 32) != r && (unsigned)(hp > hc ? hp : hc) == e;
      const unsigned long long ch = __ballot(changed) & group;
      // e heads every node, and v is the changed node that handles it
      if ((__ballot(heads) & group) == group && __shfl(m, (int)__builtin_ctzll(ch), 64) == v) {
        unsigned long long mk[CW];
#pragma unroll
        for (int k = 0; k < CW; k++) {
          mk[k] = used[(size_t)CW * m + k];
          mk[k] |= __shfl_xor(mk[k], 4, 16);
          mk[k] |= __shfl_xor(mk[k], 8, 16);
        }
        int c = -1;
#pragma unroll
        for (int k = 0; k < CW; k++)
          if (c < 0 && ~mk[k]) c = 64 * k + __builtin_ctzll(~mk[k]);
        if ((threadIdx.x & 15) == 0) {
          color[e] = c < 0 ? 0x7fffffff : c;  // past 256 colours: reported at the end
          if (c < 0)
            atomicOr(err, 2);
          else if (c > __hip_atomic_load(maxColor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(maxColor, c);
        }
        if (quad == 0 && c >= 0) used[(size_t)CW * m + c / 64] |= 1ull << (c % 64);
        const int s = diagPtr[m];
        const unsigned ne = jp_scan(clist, cptr[s], cptr[s + 1], color, (int)e, quad);
        const int m0 = __shfl(m, 0, 16), m1 = __shfl(m, 4, 16), m2 = __shfl(m, 8, 16);
        const bool twice = (a > 0 && m == m0) || (a > 1 && m == m1) || (a > 2 && m == m2);  // a degenerate element
        if (quad == 0 && !twice) {
          __hip_atomic_store(head + 2 * (size_t)m + (r & 1), ((unsigned long long)r << 32) | ne, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
          if (ne != kNoElem) push[atomicAdd(&nPush, 1)] = m;
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0 && nPush) at = atomicAdd(cnt + r % 3, nPush);
    __syncthreads();
    if ((int)threadIdx.x < nPush) next[at + threadIdx.x] = push[threadIdx.x];
    __syncthreads();
  }
}

// Colour-sorted element q = order[q]: its nodes.
__global__ __launch_bounds__(256) void k_sorted_ien(int nEl, const int* __restrict__ order,
                                                    const int4* __restrict__ ien, int4* __restrict__ ienSorted)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nEl) ienSorted[q] = ien[order[q]];
}

// Elements per colour (256 bins, LDS first).
__global__ __launch_bounds__(256) void k_color_hist(int nEl, const int* __restrict__ color, int* __restrict__ hist)
{
  __shared__ int h[64 * CW];
  h[threadIdx.x] = 0;
  __syncthreads();
  for (int e = blockIdx.x * 256 + threadIdx.x; e < nEl; e += gridDim.x * 256)
    if (color[e] < 64 * CW) atomicAdd(&h[color[e]], 1);
  __syncthreads();
  if (h[threadIdx.x]) atomicAdd(hist + threadIdx.x, h[threadIdx.x]);
}

__global__ __launch_bounds__(256) void k_iota(int n, int* __restrict__ v)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = i;
}

int bits_for(unsigned long long v)
{
  int b = 1;
  while (b < 64 && (v >> b) != 0) b++;
  return b;
}

// Device scratch released on every return path, cut from blocks of at least
// `hint` bytes: an allocation and its free cost about 0.1 ms each, so a set-up
// call whose hint covers its arrays pays for one.
struct Scratch {
  size_t hint, used = 0, cap = 0;
  std::vector<void*> blocks;
  explicit Scratch(size_t h) : hint(h) {}
  template <typename T>
  int get(T** out, size_t n)
  {
    const size_t bytes = (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~(size_t)255;
    if (used + bytes > cap) {
      unsigned char* b = nullptr;
      const size_t want = std::max(bytes, hint);
      int rc = dev_alloc(&b, want);
      if (rc) return rc;
      blocks.push_back(b);
      cap = want;
      used = 0;
    }
    *out = reinterpret_cast<T*>((unsigned char*)blocks.back() + used);
    used += bytes;
    return SVG_OK;
  }
  ~Scratch()
  {
    for (void* q : blocks) (void)hipFree(q);
  }
};

// Element-order assembly map: entry k = 16 e + 4 a + b of element e (caller
// order) adds to the block slot (ien[a], ien[b]); key[k] = that slot.
__global__ __launch_bounds__(256) void k_contrib_keys(int nEl, const int4* __restrict__ ien,
                                                      const int* __restrict__ rowPtr, const int* __restrict__ colPtr,
                                                      int* __restrict__ key, int* __restrict__ val,
                                                      int* __restrict__ err)
{
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= 16LL * nEl) return;
  const int e = (int)(k >> 4), a = (int)((k >> 2) & 3), b = (int)(k & 3);
  const int4 v = ien[e];
  const int nd[4] = {v.x, v.y, v.z, v.w};
  const int row = a == 0 ? nd[0] : a == 1 ? nd[1] : a == 2 ? nd[2] : nd[3];
  const int col = b == 0 ? nd[0] : b == 1 ? nd[1] : b == 2 ? nd[2] : nd[3];
  const int s = rowPtr[row], t = rowPtr[row + 1];
  int lo = s, hi = t;  // first position with colPtr >= col
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (colPtr[mid] < col)
      lo = mid + 1;
    else
      hi = mid;
  }
  if (lo == t || colPtr[lo] != col) {
    atomicOr(err, 4);
    lo = s;
  }
  key[k] = lo;
  val[k] = (int)k;
}

// The gather's chunks (whole slots, at most 64 of them and 64 entries, a slot
// of more entries alone), packed greedily along each window of kGatherRows
// rows, one lane per window: FILL = false counts a window's chunks, true
// writes their first slots from off[window] on. 16 rows (about 1440 entries)
// leave half a chunk of 23 unfilled at a window's end. A chunk's slots all have
// entries or none has: the gather writes every slot of a chunk that has any, and
// the slots without are other meshes' of the same lhs, which another stream may
// be assembling.
constexpr int kGatherRows = 16;
template <bool FILL>
__global__ __launch_bounds__(64) void k_chunks(int nWin, int nNo, int nnz, const int* __restrict__ rowPtr,
                                               const int* __restrict__ cptr, int* __restrict__ off,
                                               int2* __restrict__ chunk)
{
  const int w = blockIdx.x * 64 + threadIdx.x;
  if (w >= nWin) return;
  const int s1 = rowPtr[min(nNo, (w + 1) * kGatherRows)];
  int n = FILL ? off[w] : 0;
  int first = rowPtr[w * kGatherRows], c0 = cptr[first];
  if (FILL && first < s1) chunk[n] = make_int2(first, c0);
  const int open = first < s1 ? 1 : 0;
  int last = c0;  // the first entry of slot s + q
  for (int s = first; s < s1; s += 8) {
    int end[8];
#pragma unroll
    for (int q = 0; q < 8; q++) end[q] = cptr[min(s + q, s1 - 1) + 1];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const bool mixed = (end[q] == last) != (last == c0);
      if (s + q < s1 && s + q > first && (end[q] - c0 > 64 || s + q - first >= 64 || mixed)) {
        // slot s + q opens the next chunk
        n++;
        first = s + q;
        c0 = last;
        if (FILL) chunk[n] = make_int2(first, c0);
      }
      last = end[q];
    }
  }
  if (!FILL) off[w] = n + open;
  if (FILL && w == nWin - 1) chunk[n + open] = make_int2(nnz, cptr[nnz]);
}

// The elements of each chunk's entries, each once in the order they first
// appear, and every entry's place among them; one wavefront per chunk.
__global__ __launch_bounds__(256) void k_chunk_uniq(int nChunk, const int2* __restrict__ chunk,
                                                    const int* __restrict__ clist, int* __restrict__ uniq,
                                                    unsigned char* __restrict__ uniqN,
                                                    unsigned short* __restrict__ lcode)
{
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (w >= nChunk) return;
  const int c0 = chunk[w].y, n = chunk[w + 1].y - c0;
  const int code = lane < n ? clist[c0 + lane] : -1, e = code >> 4;
  int first = -1;
  for (int j = 0; j < min(n, 64); j++)
    if (__shfl(e, j, 64) == e && first < 0) first = j;
  const unsigned long long heads = __ballot(first == lane);
  const int u = __popcll(heads);
  if (n <= 64 && u <= kUniq) {
    const int at = __popcll(heads & ((1ull << max(first, 0)) - 1));
    if (first == lane) uniq[(size_t)kUniq * w + at] = e;
    if (lane < n) lcode[c0 + lane] = (unsigned short)((at << 4) | (code & 15));
    if (lane >= u && lane < kUniq) uniq[(size_t)kUniq * w + lane] = 0;
    if (lane == 0) uniqN[w] = (unsigned char)u;
  } else {
    if (lane < kUniq) uniq[(size_t)kUniq * w + lane] = 0;
    if (lane == 0) uniqN[w] = 0;
  }
}

// cptr[s] = first position of slot s in the sorted keys (lower bound), s in [0, nnz].
__global__ __launch_bounds__(256) void k_contrib_ptr(int nnz, long long n, const int* __restrict__ sorted,
                                                     int* __restrict__ cptr)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s > nnz) return;
  long long lo = 0, hi = n;
  while (lo < hi) {
    const long long mid = (lo + hi) >> 1;
    if (sorted[mid] < s)
      lo = mid + 1;
    else
      hi = mid;
  }
  cptr[s] = (int)lo;
}

int check_ien(long long n, const int* d_ien, int nNo, int* d_err, hipStream_t s, const char* who)
{
  SVG_HIP(hipMemsetAsync(d_err, 0, sizeof(int), s));
  hipLaunchKernelGGL(k_check_ien, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, d_ien, nNo, d_err);
  int h = 0;
  SVG_HIP(hipMemcpyAsync(&h, d_err, sizeof(int), hipMemcpyDeviceToHost, s));
  SVG_HIP(hipStreamSynchronize(s));
  if (h) return set_error(SVG_ERR_ARG, std::string(who) + ": IEN entry out of range");
  return SVG_OK;
}

}  // namespace

// The element-order assembly's map and record storage for M (see svg_msh):
// every (element, a, b) entry keyed by its block slot, sorted stably by slot
// (so each slot's entries stay in element order), and the slot offsets.
int msh_gather_build(svg_msh* M, const int* d_IEN, hipStream_t s)
{
  const svg_lhs* L = M->lhs;
  const int nEl = M->nEl, nnz = L->nnz;
  if (nEl >= (1 << 27)) return set_error(SVG_ERR_ARG, "element-order assembly: more than 2^27 elements");
  if (reinterpret_cast<uintptr_t>(d_IEN) & 15)
    return set_error(SVG_ERR_ARG, "element-order assembly: IEN must be 16-byte aligned (read as int4)");
  const long long n = 16LL * nEl;
  Scratch S(sizeof(int) * 5 * (size_t)n + ((size_t)4 << 20));  // key, sorted, val; the sort's two buffers
  int rc;
  int *key = nullptr, *sorted = nullptr, *val = nullptr, *d_err = nullptr;
  if ((rc = dev_alloc(&M->d_ien0, (size_t)4 * nEl)) || (rc = dev_alloc(&M->d_cptr, (size_t)nnz + 1)) ||
      (rc = dev_alloc(&M->d_clist, (size_t)n)) || (rc = dev_alloc(&M->d_rec, (size_t)kTet4Rec * nEl)))
    return rc;
  if ((rc = S.get(&key, (size_t)n)) || (rc = S.get(&sorted, (size_t)n)) || (rc = S.get(&val, (size_t)n)) ||
      (rc = S.get(&d_err, 1)))
    return rc;
  SVG_HIP(hipMemcpyAsync(M->d_ien0, d_IEN, sizeof(int) * 4 * (size_t)nEl, hipMemcpyDeviceToDevice, s));
  SVG_HIP(hipMemsetAsync(d_err, 0, sizeof(int), s));
  hipLaunchKernelGGL(k_contrib_keys, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, nEl,
                     reinterpret_cast<const int4*>(M->d_ien0), (const int*)L->d_rowPtr, (const int*)L->d_colPtr, key,
                     val, d_err);
  SVG_HIP(hipGetLastError());
  const int endBit = bits_for((unsigned long long)(nnz > 0 ? nnz - 1 : 0));
  size_t tb = 0;
  SVG_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, (const int*)key, sorted, (const int*)val, M->d_clist,
                                             (int)n, 0, endBit, s));
  unsigned char* tmp = nullptr;
  if ((rc = S.get(&tmp, tb))) return rc;
  SVG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, (const int*)key, sorted, (const int*)val, M->d_clist, (int)n,
                                             0, endBit, s));
  hipLaunchKernelGGL(k_contrib_ptr, dim3(blocks_for((size_t)nnz + 1, 256)), dim3(256), 0, s, nnz, n,
                     (const int*)sorted, M->d_cptr);
  SVG_HIP(hipGetLastError());
  const int nWin = (L->nNo + kGatherRows - 1) / kGatherRows;
  int *cnt = nullptr, *off = nullptr;
  if ((rc = S.get(&cnt, (size_t)nWin + 1)) || (rc = S.get(&off, (size_t)nWin + 1))) return rc;
  SVG_HIP(hipMemsetAsync(cnt + nWin, 0, sizeof(int), s));
  hipLaunchKernelGGL(k_chunks<false>, dim3(blocks_for(nWin, 64)), dim3(64), 0, s, nWin, L->nNo, nnz,
                     (const int*)L->d_rowPtr, (const int*)M->d_cptr, cnt, (int2*)nullptr);
  SVG_HIP(hipGetLastError());
  size_t tb2 = 0;
  SVG_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb2, (const int*)cnt, off, nWin + 1, s));
  unsigned char* tmp2 = nullptr;
  if ((rc = S.get(&tmp2, tb2))) return rc;
  SVG_HIP(hipcub::DeviceScan::ExclusiveSum(tmp2, tb2, (const int*)cnt, off, nWin + 1, s));
  SVG_HIP(hipMemcpyAsync(&M->nChunk, off + nWin, sizeof(int), hipMemcpyDeviceToHost, s));
  SVG_HIP(hipStreamSynchronize(s));
  if ((rc = dev_alloc(&M->d_chunk, (size_t)M->nChunk + 1))) return rc;
  hipLaunchKernelGGL(k_chunks<true>, dim3(blocks_for(nWin, 64)), dim3(64), 0, s, nWin, L->nNo, nnz,
                     (const int*)L->d_rowPtr, (const int*)M->d_cptr, off, M->d_chunk);
  SVG_HIP(hipGetLastError());
  if ((rc = dev_alloc(&M->d_uniq, (size_t)kUniq * M->nChunk)) || (rc = dev_alloc(&M->d_uniqN, (size_t)M->nChunk)) ||
      (rc = dev_alloc(&M->d_lcode, (size_t)n)))
    return rc;
  hipLaunchKernelGGL(k_chunk_uniq, dim3(blocks_for(M->nChunk, 4)), dim3(256), 0, s, M->nChunk,
                     (const int2*)M->d_chunk, (const int*)M->d_clist, M->d_uniq, M->d_uniqN,
                     M->d_lcode);
  SVG_HIP(hipGetLastError());
  int herr = 0;
  SVG_HIP(hipMemcpyAsync(&herr, d_err, sizeof(int), hipMemcpyDeviceToHost, s));
  SVG_HIP(hipStreamSynchronize(s));
  if (herr & 4) return set_error(SVG_ERR_ARG, "slot_map: pattern does not contain an element pair");
  return SVG_OK;
}

}  // namespace svg

using namespace svg;

extern "C" {

int svg_lhs_create_dev(int nNo, int nEl, const int* d_IEN, int nFaces, svg_lhs** out, void* stream)
{
  hipStream_t s = (hipStream_t)stream;
  if (!out || !d_IEN || nNo <= 0 || nEl <= 0 || nFaces < 0)
    return set_error(SVG_ERR_ARG, "svg_lhs_create_dev: bad argument");
  if (reinterpret_cast<uintptr_t>(d_IEN) & 15)
    return set_error(SVG_ERR_ARG, "svg_lhs_create_dev: d_IEN must be 16-byte aligned (read as int4)");
  if ((unsigned long long)nNo * (unsigned long long)nNo >= (1ULL << 62))
    return set_error(SVG_ERR_ARG, "svg_lhs_create_dev: nNo too large");
  const long long K = 16LL * nEl + nNo;
  if (K > 0x7fffffffLL) return set_error(SVG_ERR_ARG, "svg_lhs_create_dev: too many node pairs");
  Scratch S(sizeof(unsigned long long) * 4 * (size_t)K + ((size_t)4 << 20));
  int rc;
  int* d_err = nullptr;
  if ((rc = S.get(&d_err, 1))) return rc;
  if ((rc = check_ien(4LL * nEl, d_IEN, nNo, d_err, s, "svg_lhs_create_dev"))) return rc;
  unsigned long long *keys = nullptr, *sorted = nullptr, *uniq = nullptr;
  int* d_nnz = nullptr;
  if ((rc = S.get(&keys, (size_t)K)) || (rc = S.get(&sorted, (size_t)K)) || (rc = S.get(&uniq, (size_t)K)) ||
      (rc = S.get(&d_nnz, 1)))
    return rc;
  hipLaunchKernelGGL(k_pair_keys, dim3((unsigned)((K + 255) / 256)), dim3(256), 0, s, nEl, nNo,
                     reinterpret_cast<const int4*>(d_IEN), keys);
  const int endBit = bits_for((unsigned long long)nNo * (unsigned long long)nNo - 1);
  size_t tb1 = 0, tb2 = 0;
  SVG_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, tb1, keys, sorted, (int)K, 0, endBit, s));
  SVG_HIP(hipcub::DeviceSelect::Unique(nullptr, tb2, sorted, uniq, d_nnz, (int)K, s));
  unsigned char* tmp = nullptr;
  if ((rc = S.get(&tmp, std::max(tb1, tb2)))) return rc;
  SVG_HIP(hipcub::DeviceRadixSort::SortKeys(tmp, tb1, keys, sorted, (int)K, 0, endBit, s));
  SVG_HIP(hipcub::DeviceSelect::Unique(tmp, tb2, sorted, uniq, d_nnz, (int)K, s));
  int nnz = 0;
  SVG_HIP(hipMemcpyAsync(&nnz, d_nnz, sizeof(int), hipMemcpyDeviceToHost, s));
  SVG_HIP(hipStreamSynchronize(s));
  if ((long long)nnz * 16 > 0x7fffffffLL) return set_error(SVG_ERR_ARG, "svg_lhs_create_dev: 16*nnz overflows int");
  auto* L = new svg_lhs();
  L->nNo = nNo;
  L->nnz = nnz;
  L->nFaces = nFaces;
  L->face.resize(nFaces);
  if ((rc = dev_alloc(&L->d_rowPtr, nNo + 1)) || (rc = dev_alloc(&L->d_colPtr, nnz)) ||
      (rc = dev_alloc(&L->d_diagPtr, nNo)) || (rc = dev_alloc(&L->d_mask, (size_t)4 * nNo))) {
    svg_lhs_free(L);
    return rc;
  }
  hipLaunchKernelGGL(k_csr_from_keys, dim3(blocks_for(nnz, 256)), dim3(256), 0, s, nnz, nNo,
                     (const unsigned long long*)uniq, L->d_rowPtr, L->d_colPtr, L->d_diagPtr);
  // host mirrors of the pattern (the lhs keeps them for its host-side users)
  L->rowPtr.resize(nNo + 1);
  L->colPtr.resize(nnz);
  L->diagPtr.resize(nNo);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = hipMemcpyAsync(L->rowPtr.data(), L->d_rowPtr, sizeof(int) * (nNo + 1), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipMemcpyAsync(L->colPtr.data(), L->d_colPtr, sizeof(int) * nnz, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess)
    e = hipMemcpyAsync(L->diagPtr.data(), L->d_diagPtr, sizeof(int) * nNo, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    svg_lhs_free(L);
    return hip_check(e, "svg_lhs_create_dev");
  }
  *out = L;
  return SVG_OK;
}

int svg_lhs_nnz(const svg_lhs* L, int* nnz)
{
  if (!L || !nnz) return set_error(SVG_ERR_ARG, "svg_lhs_nnz: null argument");
  *nnz = L->nnz;
  return SVG_OK;
}

int svg_lhs_pattern(const svg_lhs* L, int* rowPtr, int* colPtr)
{
  if (!L || !rowPtr || !colPtr) return set_error(SVG_ERR_ARG, "svg_lhs_pattern: null argument");
  std::memcpy(rowPtr, L->rowPtr.data(), sizeof(int) * (L->nNo + 1));
  std::memcpy(colPtr, L->colPtr.data(), sizeof(int) * L->nnz);
  return SVG_OK;
}

int svg_msh_create_dev(const svg_lhs* L, int nEl, const int* d_IEN, const double* d_x, svg_msh** out,
                       void* stream)
{
  hipStream_t s = (hipStream_t)stream;
  if (!L || !d_IEN || !d_x || !out || nEl <= 0) return set_error(SVG_ERR_ARG, "svg_msh_create_dev: bad argument");
  if (reinterpret_cast<uintptr_t>(d_IEN) & 15)
    return set_error(SVG_ERR_ARG, "svg_msh_create_dev: d_IEN must be 16-byte aligned (read as int4)");
  const int nNo = L->nNo;
  // per element the colour, order and id arrays and the sort's buffers, per node heads, masks and lists
  Scratch S(sizeof(int) * 6 * (size_t)nEl + (16 + 8 * CW + 8) * (size_t)nNo + ((size_t)4 << 20));
  int rc;
  int *d_err = nullptr, *color = nullptr, *d_cnt = nullptr, *order = nullptr, *ids = nullptr, *colSorted = nullptr,
      *list[2] = {nullptr, nullptr}, *hist = nullptr;
  unsigned long long *head = nullptr, *used = nullptr;
  if ((rc = S.get(&d_err, 1))) return rc;
  if ((rc = check_ien(4LL * nEl, d_IEN, nNo, d_err, s, "svg_msh_create_dev"))) return rc;
  if ((rc = S.get(&color, nEl)) || (rc = S.get(&d_cnt, 4)) || (rc = S.get(&head, (size_t)2 * nNo)) ||
      (rc = S.get(&used, (size_t)CW * nNo)) || (rc = S.get(&order, nEl)) || (rc = S.get(&ids, nEl)) ||
      (rc = S.get(&colSorted, nEl)) || (rc = S.get(&list[0], nNo)) || (rc = S.get(&list[1], nNo)) ||
      (rc = S.get(&hist, 64 * CW)))
    return rc;
  const int4* ien4 = reinterpret_cast<const int4*>(d_IEN);
  auto* M = new svg_msh();
  struct Guard {  // a return before the end frees the mesh
    svg_msh* m;
    ~Guard() { svg_msh_free(m); }
  } guard{M};
  M->lhs = L;
  M->nEl = nEl;
  M->nNo = nNo;
  // the element-order map first: its diagonal slots list each node's elements for the colouring
  if ((rc = msh_gather_build(M, d_IEN, s))) return rc;
  SVG_HIP(hipMemsetAsync(color, 0xff, sizeof(int) * nEl, s));  // -1: uncoloured
  SVG_HIP(hipMemsetAsync(used, 0, sizeof(unsigned long long) * CW * nNo, s));
  SVG_HIP(hipMemsetAsync(d_cnt + 3, 0, sizeof(int), s));  // [0..2] list lengths, [3] largest colour
  SVG_HIP(hipMemsetAsync(hist, 0, sizeof(int) * 64 * CW, s));
  const unsigned gE = blocks_for(nEl, 256);
  hipLaunchKernelGGL(k_jp_heads, dim3(blocks_for((size_t)4 * nNo, 256)), dim3(256), 0, s, nNo,
                     (const int*)L->d_diagPtr, (const int*)M->d_cptr, (const int*)M->d_clist, (const int*)color, head,
                     list[1], d_cnt);
  const unsigned gR = std::min(blocks_for((size_t)nNo, JP_G), 512u);
  int h[4] = {0, 1, 0, 0};
  int r = 1;
  while (h[r % 3] > 0) {
    if (r > 400000) return set_error(SVG_ERR_ARG, "svg_msh_create_dev: colouring did not finish");
    // 32 rounds per host check: a round with an empty list does nothing
    for (int k = 0; k < 32; k++) {
      r++;
      hipLaunchKernelGGL(k_jp_round, dim3(gR), dim3(16 * JP_G), 0, s, r, ien4, (const int*)L->d_diagPtr,
                         (const int*)M->d_cptr, (const int*)M->d_clist, color, head, used,
                         (const int*)list[(r - 1) & 1], list[r & 1], d_cnt, d_cnt + 3, d_err);
    }
    SVG_HIP(hipGetLastError());
    SVG_HIP(hipMemcpyAsync(h, d_cnt, 4 * sizeof(int), hipMemcpyDeviceToHost, s));
    SVG_HIP(hipStreamSynchronize(s));
  }
  int herr = 0;
  SVG_HIP(hipMemcpy(&herr, d_err, sizeof(int), hipMemcpyDeviceToHost));
  if (herr & 2) return set_error(SVG_ERR_ARG, "svg_msh_create_dev: more than 256 colours needed");
  const int nColors = h[3] + 1;
  M->nColors = nColors;
  // colour order: stable radix sort of the element ids by colour
  hipLaunchKernelGGL(k_iota, dim3(gE), dim3(256), 0, s, nEl, ids);
  size_t tb = 0;
  SVG_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, (const int*)color, colSorted, (const int*)ids, order, nEl,
                                             0, 8, s));
  unsigned char* tmp = nullptr;
  if ((rc = S.get(&tmp, tb))) return rc;
  SVG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, (const int*)color, colSorted, (const int*)ids, order, nEl, 0,
                                             8, s));
  hipLaunchKernelGGL(k_color_hist, dim3(std::min(gE, 1024u)), dim3(256), 0, s, nEl, (const int*)color, hist);
  SVG_HIP(hipGetLastError());
  std::vector<int> hc(64 * CW);
  SVG_HIP(hipMemcpyAsync(hc.data(), hist, sizeof(int) * hc.size(), hipMemcpyDeviceToHost, s));
  if ((rc = dev_alloc(&M->d_x, (size_t)3 * nNo)) || (rc = dev_alloc(&M->d_ien, (size_t)4 * nEl)) ||
      (rc = construct_fluid_flag(M)))
    return rc;
  hipLaunchKernelGGL(k_sorted_ien, dim3(gE), dim3(256), 0, s, nEl, (const int*)order, ien4,
                     reinterpret_cast<int4*>(M->d_ien));
  SVG_HIP(hipGetLastError());
  SVG_HIP(hipMemcpyAsync(M->d_x, d_x, sizeof(double) * 3 * nNo, hipMemcpyDeviceToDevice, s));
  SVG_HIP(hipStreamSynchronize(s));
  M->colorOff.assign(nColors + 1, 0);
  for (int c = 0; c < nColors; c++) M->colorOff[c + 1] = M->colorOff[c] + hc[c];
  guard.m = nullptr;
  *out = M;
  return SVG_OK;
}

int svg_msh_colors(const svg_msh* M, int* colorOff)
{
  if (!M || !colorOff) return set_error(SVG_ERR_ARG, "svg_msh_colors: null argument");
  std::memcpy(colorOff, M->colorOff.data(), sizeof(int) * (M->nColors + 1));
  return SVG_OK;
}

int svg_msh_sorted_ien(const svg_msh* M, int* ien)
{
  if (!M || !ien) return set_error(SVG_ERR_ARG, "svg_msh_sorted_ien: null argument");
  SVG_HIP(hipMemcpy(ien, M->d_ien, sizeof(int) * 4 * (size_t)M->nEl, hipMemcpyDeviceToHost));
  return SVG_OK;
}

}  // extern "C"
