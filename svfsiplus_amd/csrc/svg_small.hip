// Iterations of small systems as one cooperative launch each. On a mesh of some
// thousand nodes a Krylov step's kernels take their launch, ramp and drain (4 to
// 5 us each) and little else; here the workgroups stay and meet at barriers
// (1.4 us for 4 workgroups, 2.3 us for 64, 4.7 us for 256, exchange included).
// Every sum keeps the order of the per-launch kernels (svg_fsils.hip), so the
// results are theirs bit for bit.
//
// What workgroups read of each other goes through agent-scope accesses, which
// bypass the caches that are not shared: relaxed atomic stores, completed
// (vmcnt 0) before the barrier's arrival, and loads past the barrier. The
// barrier's wait is bounded: if the workgroups do not meet, each leaves and
// flags it, and the host takes the per-launch path, whose inputs a kernel here
// never overwrites before its last barrier.
#include "svg_device.h"

#include <algorithm>
#include <cmath>

namespace svg {

namespace {

constexpr int SPIN_MAX = 1 << 20;  // polls of about 0.7 us

__device__ __forceinline__ double ld_agent(const double* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(double* p, double v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 16-byte loads at agent scope (the sc1 cache policy of ld_agent's).
typedef int v4i __attribute__((ext_vector_type(4)));
struct AgentBuf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ AgentBuf(const void* p, size_t bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000))
  {
  }
  __device__ __forceinline__ double2 ld2(int byte) const
  {
    return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, byte, 0, 16));
  }
};

// All workgroups of the launch meet; false: they did not within SPIN_MAX polls.
__device__ __forceinline__ bool grid_sync(int* ctr, int& target, int* ok)
{
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  target += gridDim.x;
  if (threadIdx.x == 0) {
    int c = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    for (int n = 0; c < target && n < SPIN_MAX; n++)
      c = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *ok = c >= target;
  }
  __syncthreads();
  return *ok != 0;
}

// Sum over n entries in the order of the per-launch reductions: spans of 1024,
// lane t of 256 adds its entries t, t + 256, .. of the span in order, butterflies,
// the four wavefront sums in order, then the spans (lane b, b + 64, .. in order
// and a butterfly). Every workgroup (256 lanes) computes the whole sum. get(k):
// entry k's term.
constexpr int SUM_SPANS = 32;  // most spans

template <typename Get>
__device__ __forceinline__ double sum_all(int n, double* ws, Get get)
{
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int nb = (n + 1023) >> 10;
  __syncthreads();  // ws may still be read
  for (int b0 = 0; b0 < nb; b0 += 4) {
    double x[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int k = ((b0 + q) << 10) + 256 * r + 64 * wv + lane;
        const double v = get(min(k, n - 1));
        x[q][r] = k < n ? v : 0.0;
      }
    double acc[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      acc[q] = 0.0;
#pragma unroll
      for (int r = 0; r < 4; r++) acc[q] = acc[q] + x[q][r];
    }
    wave_sums<4>(acc);
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (b0 + q < nb) ws[4 * (b0 + q) + wv] = acc[q];
    }
  }
  __syncthreads();
  double s = 0.0;
  if (lane < nb) {
    double v = ws[4 * lane];
    for (int q = 1; q < 4; q++) v = v + ws[4 * lane + q];
    s = s + v;
  }
  return wave_sum(s);
}

// ----------------------------------------------------------- Schur CG ------
// cgrad::schur (cgrad.cpp:50-160) without coupled faces, as k_cg_init ..
// k_cg_p compute it. A workgroup owns `rows` rows; its blocks of G, G^T and L
// stay in LDS for the whole solve, and so does the list of the columns they
// touch, whose entries of the exchanged vectors it loads once a phase (about
// 300 for 128 rows; a load per block went past the caches 13 times a row).
// Three barriers an iteration:
//   1  |R|^2 and the stop test; P = c2 (P + c1 R) of the listed columns, and
//      GP = G P                                          -> gpp = (GP, P)
//   2  SP = L P - G^T GP; P SP                           -> prod
//   3  <P, SP>, alpha; X += alpha P; R -= alpha SP       -> pr = (P, R), rc = R
// On the 15k-tet pipe (3 321 nodes, 26 workgroups) an iteration takes 15 us, 6
// of them at the barriers; as four launches it took 52 us, 31 of them in a
// product of one lane per four rows.
constexpr int CG_BS = 256;
// LDS bytes per block (seven values, the column's place in the list) and per listed column (its place's
// id and up to four values), and of the column bitmap
constexpr int CG_BLK_B = 7 * 8 + 2, CG_COL_B = 4 + 32;

__global__ __launch_bounds__(CG_BS) void k_cg_small(int nNo, const int* __restrict__ rowPtr,
                                                    const int* __restrict__ colPtr, const double* __restrict__ mG,
                                                    const double* __restrict__ Gt, const double* __restrict__ mL,
                                                    const double* __restrict__ R0, double* __restrict__ X, double* pr,
                                                    double* gpp, double* prod, double* rc, CgState* cg, int* ctr,
                                                    int rows, int cap, int capU, int mItr, double absTol,
                                                    double relTol)
{
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  __shared__ double ws[4 * SUM_SPANS];
  __shared__ unsigned bits[32 * SUM_SPANS], before[32 * SUM_SPANS];  // listed columns, and how many lie before
  __shared__ int okf, wsum[4];
  double* val = lds;                                                 // [4][capU]: the listed columns' values
  double* m = lds + 4 * (size_t)capU;                                // [7][cap]: G, G^T, L of the blocks
  int* list = reinterpret_cast<int*>(m + 7 * (size_t)cap);           // [capU]: the listed columns
  unsigned short* loc = reinterpret_cast<unsigned short*>(list + capU);  // [cap]: each block's place in the list
  const int t = threadIdx.x, lane = t & 63, r0 = blockIdx.x * rows, r1 = min(nNo, r0 + rows);
  const int j0 = rowPtr[r0], nblk = rowPtr[r1] - j0;
  for (int q = t; q < 32 * SUM_SPANS; q += CG_BS) bits[q] = 0;
  for (int q = t; q < 3 * nblk; q += CG_BS) {
    m[(q % 3) * cap + q / 3] = mG[3 * (size_t)j0 + q];
    m[(3 + q % 3) * cap + q / 3] = Gt[3 * (size_t)j0 + q];
  }
  __syncthreads();
  for (int q = t; q < nblk; q += CG_BS) {
    m[6 * cap + q] = mL[j0 + q];
    const int c = colPtr[j0 + q];
    atomicOr(&bits[c >> 5], 1u << (c & 31));
  }
  __syncthreads();
  {
    // lane t counts words 4 t .. 4 t + 3, a scan over the lanes and the four wavefronts
    int n4[4], n = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) n4[q] = __popc(bits[4 * t + q]), n += n4[q];
    int inc = n;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc, o, 64);
      if (lane >= o) inc += v;
    }
    if (lane == 63) wsum[t >> 6] = inc;
    __syncthreads();
    int at = inc - n;
    for (int q = 0; q < (t >> 6); q++) at += wsum[q];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      before[4 * t + q] = at;
      for (unsigned b = bits[4 * t + q], k = at; b; b &= b - 1, k++) list[k] = 32 * (4 * t + q) + __builtin_ctz(b);
      at += n4[q];
    }
  }
  __syncthreads();
  const int nu = wsum[0] + wsum[1] + wsum[2] + wsum[3];
  for (int q = t; q < nblk; q += CG_BS) {
    const int c = colPtr[j0 + q];
    loc[q] = (unsigned short)(before[c >> 5] + __popc(bits[c >> 5] & ((1u << (c & 31)) - 1u)));
  }
  const bool own = t < rows && r0 + t < r1;
  const int row = r0 + t;
  const int ja = own ? rowPtr[row] - j0 : 0, jb = own ? rowPtr[row + 1] - j0 : 0;
  const AgentBuf bpr(pr, sizeof(double) * 2 * nNo), bgp(gpp, sizeof(double) * 4 * nNo);
  int target = 0;
  double P = own ? R0[row] : 0.0, R = P, Xr = 0.0;
  if (own) {
    st_agent(pr + 2 * (size_t)row, P);
    st_agent(pr + 2 * (size_t)row + 1, R);
  }
  // iNorm = |R|, eps = max(absTol, relTol iNorm)^2, errO = iNorm^2, stop test
  const double iN = sqrt(sum_all(nNo, ws, [&](int k) {
    const double v = R0[k];
    return v * v;
  }));
  double e = fmax(absTol, relTol * iN);
  const double eps = e * e;
  double errO = iN * iN, errO_last = errO, err = errO;
  int suc = 0, last_i = 0;
  bool stop = false;
  if (err < eps) {
    suc = 1;
    stop = true;
  }
  bool ok = grid_sync(ctr, target, &okf);
  double c1 = 0.0, c2 = 0.0;
  for (int i = 0; ok && !stop && mItr > 0; i++) {
    // 1: the listed columns' P and R (the first two per lane on their way while
    // the sum is taken), |R|^2 of the trip before and its stop test
    const double2 x0 = bpr.ld2(16 * list[min(t, nu - 1)]), x1 = bpr.ld2(16 * list[min(t + CG_BS, nu - 1)]);
    if (i > 0) {
      e = sqrt(sum_all(nNo, ws, [&](int k) {
        const double v = ld_agent(rc + k);
        return v * v;
      }));
      e = e * e;
      c1 = errO / e;
      c2 = e / errO;
      err = e;
      errO_last = errO;
      last_i = i - 1;
      if (i < mItr) {
        last_i = i;
        errO = e;
        if (e < eps) {
          suc = 1;
          stop = true;
        }
      } else {
        stop = true;
      }
      if (stop) break;
      P = c2 * (P + c1 * R);  // the first trip's P is R
    }
    auto newP = [&](const double2& x) { return i > 0 ? c2 * (x.x + c1 * x.y) : x.x; };
    if (t < nu) val[t] = newP(x0);
    if (t + CG_BS < nu) val[t + CG_BS] = newP(x1);
    for (int q = t + 2 * CG_BS; q < nu; q += CG_BS) val[q] = newP(bpr.ld2(16 * list[q]));
    __syncthreads();
    if (own) {
      double g0 = 0.0, g1 = 0.0, g2 = 0.0;
#pragma unroll 4
      for (int j = ja; j < jb; j++) {
        const double p = val[loc[j]];
        g0 = g0 + m[j] * p;
        g1 = g1 + m[cap + j] * p;
        g2 = g2 + m[2 * cap + j] * p;
      }
      double* o = gpp + 4 * (size_t)row;
      st_agent(o, g0);
      st_agent(o + 1, g1);
      st_agent(o + 2, g2);
      st_agent(o + 3, P);
    }
    if (!(ok = grid_sync(ctr, target, &okf))) break;
    // 2: SP = L P - G^T GP
    for (int q = t; q < nu; q += CG_BS) {
      const double2 x = bgp.ld2(32 * list[q]), y = bgp.ld2(32 * list[q] + 16);
      val[q] = x.x;
      val[capU + q] = x.y;
      val[2 * capU + q] = y.x;
      val[3 * capU + q] = y.y;
    }
    __syncthreads();
    double sp = 0.0;
    if (own) {
      double dgp = 0.0;
#pragma unroll 4
      for (int j = ja; j < jb; j++) {
        const double* v = val + loc[j];
        dgp = dgp + m[3 * cap + j] * v[0] + m[4 * cap + j] * v[capU] + m[5 * cap + j] * v[2 * capU];
        sp = sp + m[6 * cap + j] * v[3 * capU];
      }
      sp = sp + (-1.0) * dgp;
      st_agent(prod + row, P * sp);
    }
    if (!(ok = grid_sync(ctr, target, &okf))) break;
    // 3: alpha, X and R
    const double alpha = errO / sum_all(nNo, ws, [&](int k) { return ld_agent(prod + k); });
    if (own) {
      Xr = Xr + alpha * P;
      R = R + (-alpha) * sp;
      st_agent(pr + 2 * (size_t)row, P);
      st_agent(pr + 2 * (size_t)row + 1, R);
      st_agent(rc + row, R);
    }
    ok = grid_sync(ctr, target, &okf);
  }
  if (own) X[row] = Xr;
  if (t == 0) {
    if (!ok) __hip_atomic_store(&cg->pad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (blockIdx.x == 0) {
      cg->stop = 1;
      cg->last_i = last_i;
      cg->suc = suc;
      cg->eps = eps;
      cg->err = err;
      cg->iNorm = iN;
      cg->errO_last = errO_last;
    }
  }
}

int num_cus(int* n)
{
  int dev = 0;
  SVG_HIP(hipGetDevice(&dev));
  SVG_HIP(hipDeviceGetAttribute(n, hipDeviceAttributeMultiprocessorCount, dev));
  return SVG_OK;
}

__global__ void k_clear_small(int* ctr, int* flag)
{
  *ctr = 0;
  *flag = 0;
}

}  // namespace

// The most blocks of a group of `rows` consecutive rows.
static int most_blocks(const svg_lhs* L, int rows)
{
  int most = 0;
  for (int r = 0; r < L->nNo; r += rows)
    most = std::max(most, L->rowPtr[std::min(L->nNo, r + rows)] - L->rowPtr[r]);
  return most;
}

// The Schur CG of w's split system as one launch: *ran = 0 when the system does
// not fit (more workgroups than compute units, or blocks than LDS) or the
// workgroups did not meet; else the result is in w.cgX and w.h_cg (synchronises).
int cg_small(svg_lhs* L, const double* R, int mItr, double absTol, double relTol, hipStream_t s, int* ran)
{
  auto& w = L->ns;
  *ran = 0;
  if (w.smallRows < 0) return SVG_OK;
  const int nNo = L->nNo;
  int rc;
  auto bytes = [&](int cap) {
    return (size_t)CG_BLK_B * cap + (size_t)CG_COL_B * std::min(cap, nNo);
  };
  if (w.smallRows == 0) {
    int cus = 0;
    w.smallRows = -1;
    if ((rc = num_cus(&cus))) return rc;
    if (nNo > 1024 * SUM_SPANS) return SVG_OK;
    for (int rows : {128, 64}) {
      const int cap = most_blocks(L, rows);
      if ((int)blocks_for(nNo, rows) > cus || bytes(cap) > 148 * 1024) continue;
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_cg_small), hipFuncAttributeMaxDynamicSharedMemorySize,
                              148 * 1024) != hipSuccess) {
        (void)hipGetLastError();
        return SVG_OK;
      }
      if ((rc = dev_alloc(&w.cgEx, (size_t)8 * nNo)) || (rc = dev_alloc(&w.ctr, 1))) return rc;
      w.smallRows = rows;
      w.smallCap = cap;
      break;
    }
    if (w.smallRows < 0) return SVG_OK;
  }
  int rows = w.smallRows, cap = w.smallCap, capU = std::min(cap, nNo), n = nNo;
  hipLaunchKernelGGL(k_clear_small, dim3(1), dim3(1), 0, s, w.ctr, &w.cg->pad);
  const int *rp = L->d_rowPtr, *cp = L->d_colPtr;
  const double *mG = w.mG, *Gt = w.Gt, *mL = w.mL;
  double *X = w.cgX, *gpp = w.cgEx, *pr = w.cgEx + (size_t)4 * nNo, *prod = w.cgEx + (size_t)6 * nNo,
         *rcv = w.cgEx + (size_t)7 * nNo;
  void* args[] = {&n,    &rp,   &cp,   &mG,    &Gt,  &mL,   &R,    &X,    &pr,     &gpp,
                  &prod, &rcv,  &w.cg, &w.ctr, &rows, &cap, &capU, &mItr, &absTol, &relTol};
  if (hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&k_cg_small), dim3(blocks_for(nNo, rows)), dim3(CG_BS),
                                 args, (unsigned)bytes(cap), s) != hipSuccess) {
    (void)hipGetLastError();  // not launched: the per-launch path
    return SVG_OK;
  }
  SVG_HIP(hipMemcpyAsync(w.h_cg, w.cg, sizeof(CgState), hipMemcpyDeviceToHost, s));
  SVG_HIP(hipStreamSynchronize(s));
  *ran = w.h_cg->pad ? 0 : 1;
  return SVG_OK;
}

}  // namespace svg
