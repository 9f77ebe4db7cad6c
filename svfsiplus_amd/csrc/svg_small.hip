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
// never overwrites before its last barrier. The lhs's later solves go there
// straight away: a wait that ran out took most of a second.
#include "svg_device.h"

#include <algorithm>
#include <cmath>

namespace svg {

namespace {

// Most polls of a barrier, about 0.7 us each. The kernels' other form does not
// wait at all, so that giving up can be tested; the limit as an argument takes a
// register that k_gmres_small does not have (0.5 % of a Newton iteration).
constexpr int SPIN_MAX = 1 << 20;

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

// All workgroups of the launch meet; false: they did not within SPIN polls.
template <int SPIN>
__device__ __forceinline__ bool grid_sync(int* ctr, int& target, int* ok)
{
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  target += gridDim.x;
  if (threadIdx.x == 0) {
    int c = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    for (int n = 0; c < target && n < SPIN; n++)
      c = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *ok = c >= target;
  }
  __syncthreads();
  return *ok != 0;
}

// Orders a wavefront's LDS accesses across its lanes.
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
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
// touch, whose entries of the exchanged vectors it loads once a phase (300 to
// 470 for 128 rows; a load per block went past the caches 13 times a row).
// Three barriers an iteration:
//   1  |R|^2 and the stop test; P = c2 (P + c1 R) of the listed columns, and
//      GP = G P                                          -> gpp = (GP, P)
//   2  SP = L P - G^T GP; P SP                           -> prod
//   3  <P, SP>, alpha; X += alpha P; R -= alpha SP       -> pr = (P, R), rc = R
// On the 15k-tet pipe (3 321 nodes, 26 workgroups) an iteration takes 13.2 us, 6
// of them at the barriers (14.9 with 64 rows a workgroup); as four launches it
// took 52 us, 31 of them in a product of one lane per four rows. The two sums
// over all rows grow with the system: 44 us at 32 490 nodes (84 as launches,
// 45 of them in the product).
constexpr int CG_BS = 256;
// LDS bytes per block (seven values, the column's place in the list) and per listed column (its place's
// id and up to four values), and of the column bitmap
constexpr int CG_BLK_B = 7 * 8 + 2, CG_COL_B = 4 + 32;

template <int SPIN>
__global__ __launch_bounds__(CG_BS) void k_cg_small(int nNo, const int* __restrict__ rowPtr,
                                                    const int* __restrict__ colPtr, const double* __restrict__ mG,
                                                    const double* __restrict__ Gt, const double* __restrict__ mL,
                                                    const double* __restrict__ R0, double* __restrict__ X, double* pr,
                                                    double* gpp, double* prod, double* rc, CgState* cg, int* ctr,
                                                    int rows, int cap, int capU, int mItr,
                                                    double absTol, double relTol)
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
  bool ok = grid_sync<SPIN>(ctr, target, &okf);
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
    if (!(ok = grid_sync<SPIN>(ctr, target, &okf))) break;
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
    if (!(ok = grid_sync<SPIN>(ctr, target, &okf))) break;
    // 3: alpha, X and R
    const double alpha = errO / sum_all(nNo, ws, [&](int k) { return ld_agent(prod + k); });
    if (own) {
      Xr = Xr + alpha * P;
      R = R + (-alpha) * sp;
      st_agent(pr + 2 * (size_t)row, P);
      st_agent(pr + 2 * (size_t)row + 1, R);
      st_agent(rc + row, R);
    }
    ok = grid_sync<SPIN>(ctr, target, &okf);
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

// ----------------------------------------------------------- GMRES ---------
// gmres_v's restart cycles (gmres.cpp:529-612) on the 4x4 system, as run_cycle
// enqueues them: residual, Arnoldi steps, back substitution and X, up to
// `cycles` restarts in a launch. Workgroup 4 b + s owns, of the reduction span
// b (1024 entries), the entries 256 r + 64 s + l (r < 4, l < 64): one
// wavefront's share of the span's sums, so a step's dots follow its product
// without a barrier between them. Its blocks of the matrix and the list of the
// columns they touch stay in LDS; its part of the Krylov basis is read by no
// other workgroup and stays in the caches. Two barriers a step:
//   1  u_i of the listed columns (exchanged), w = A u_i, the share's dots with
//      u_0 .. u_i and w                                   -> part
//   2  every workgroup finishes the dots, the norm and the coefficients itself;
//      u_{i+1}                                            -> ex (double buffered)
// the Givens rotations and the stop test run beside the update, on a wavefront
// of their own, and the first GM_PF columns of the basis are on their way while
// the product is formed (for the dots) and over barrier 1 (for the update): 24
// is what the registers hold, 28 spill. On the 15k-tet pipe (52 workgroups) a
// step takes 15.3 us; 16 without either, 35 as four launches.
constexpr int GM_BS = 320, GM_MAX = 256;  // four wavefronts of entries, one for the rotations
constexpr int GM_PF = 24;
constexpr int GM_BLK_B = 16 * 8 + 2, GM_COL_B = 4 + 32;  // LDS bytes per block and per listed column

struct GmSmall {
  int nNo, sD, cap, capU, cycles;
  const int *rowPtr, *colPtr;
  const double *K, *R;
  double *X, *u, *ex, *part, *h, *y;
  size_t ld;
  GmState* st;
  int* ctr;
};

template <int SPIN>
__global__ __launch_bounds__(GM_BS) void k_gmres_small(GmSmall A)
{
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  __shared__ double sh[4][GM_MAX];  // sums, h column, cosines, sines; the set-up's bitmap first
  __shared__ double wl[4][64];      // the workgroup's entries of w, [r][l]
  __shared__ double sc[4];          // scale, err_i, err_{i+1}
  __shared__ int okf, stopf, wsum[4];
  double *sums = sh[0], *lh = sh[1], *lcs = sh[2], *lsn = sh[3];
  unsigned *bits = reinterpret_cast<unsigned*>(sh[0]), *before = reinterpret_cast<unsigned*>(sh[1]);  // 512 words each
  double* val = lds;                                                     // [capU][4]
  double* K = lds + 4 * (size_t)A.capU;                                  // [cap][16]
  int* list = reinterpret_cast<int*>(K + 16 * (size_t)A.cap);            // [capU]
  unsigned short* loc = reinterpret_cast<unsigned short*>(list + A.capU);  // [cap]
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int b = blockIdx.x >> 2, s = blockIdx.x & 3, n = 4 * A.nNo, nblk = (n + 1023) >> 10;
  const int k = 1024 * b + 256 * wv + 64 * s + lane;  // this lane's entry, r = its wavefront
  const bool own = wv < 4 && k < n;
  const int row = min(k >> 2, A.nNo - 1), ci = k & 3;
  // the rows of share r: 16 from first(r)
  auto first = [&](int r) { return min(A.nNo, 256 * b + 64 * r + 16 * s); };
  int off = 0, j0 = 0;  // this wavefront's blocks in LDS and in the matrix
  for (int r = 0; r <= wv && r < 4; r++) {
    j0 = A.rowPtr[first(r)];
    if (r < wv) off += A.rowPtr[min(A.nNo, first(r) + 16)] - j0;
  }
  const int nb = wv < 4 ? A.rowPtr[min(A.nNo, first(wv) + 16)] - j0 : 0;
  for (int q = t; q < 512; q += GM_BS) bits[q] = 0;
  __syncthreads();
  for (int q = lane; q < 8 * nb; q += 64)
    reinterpret_cast<double2*>(K + 16 * (size_t)off)[q] = reinterpret_cast<const double2*>(A.K + 16 * (size_t)j0)[q];
  for (int q = lane; q < nb; q += 64) {
    const int c = A.colPtr[j0 + q];
    atomicOr(&bits[c >> 5], 1u << (c & 31));
  }
  __syncthreads();
  {
    int n2[2], m = 0;
#pragma unroll
    for (int q = 0; q < 2; q++) n2[q] = wv < 4 ? __popc(bits[2 * t + q]) : 0, m += n2[q];
    int inc = m;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc, o, 64);
      if (lane >= o) inc += v;
    }
    if (lane == 63 && wv < 4) wsum[wv] = inc;
    __syncthreads();
    int at = inc - m;
    for (int q = 0; q < wv; q++) at += wsum[q];
#pragma unroll
    for (int q = 0; q < 2 && wv < 4; q++) {
      before[2 * t + q] = at;
      for (unsigned w = bits[2 * t + q], e = at; w; w &= w - 1, e++) list[e] = 32 * (2 * t + q) + __builtin_ctz(w);
      at += n2[q];
    }
  }
  __syncthreads();
  const int nu = wsum[0] + wsum[1] + wsum[2] + wsum[3];
  for (int q = lane; q < nb; q += 64) {
    const int c = A.colPtr[j0 + q];
    loc[off + q] = (unsigned short)(before[c >> 5] + __popc(bits[c >> 5] & ((1u << (c & 31)) - 1u)));
  }
  const int ja = own ? A.rowPtr[row] - j0 + off : 0, jb = own ? A.rowPtr[row + 1] - j0 + off : 0;
  __syncthreads();

  const AgentBuf bex0(A.ex, sizeof(double) * n), bex1(A.ex + n, sizeof(double) * n);
  const AgentBuf bpart(A.part, sizeof(double) * 4 * nblk * (A.sD + 1));
  // A v for the exchanged vector v of buffer p: this lane's entry
  auto product = [&](int p) {
    for (int q = t; q < 2 * nu; q += GM_BS) {
      const int byte = 32 * list[q >> 1] + 16 * (q & 1);
      reinterpret_cast<double2*>(val)[q] = p ? bex1.ld2(byte) : bex0.ld2(byte);
    }
    __syncthreads();
    double acc = 0.0;
#pragma unroll 4
    for (int j = ja; j < jb; j++) {
      const double2* kp = reinterpret_cast<const double2*>(K + 16 * (size_t)j + 4 * ci);
      const double2* up = reinterpret_cast<const double2*>(val + 4 * (size_t)loc[j]);
      const double2 k0 = kp[0], k1 = kp[1], u0 = up[0], u1 = up[1];
      double x = acc + k0.x * u0.x;
      x = x + k0.y * u0.y;
      x = x + k1.x * u1.x;
      acc = x + k1.y * u1.y;
    }
    return acc;
  };
  // the share's sums of column j over its wavefront's lanes -> part
  auto put_part = [&](int j, double v) {
    if (lane == 0) st_agent(A.part + (size_t)4 * nblk * j + 4 * b + s, v);
  };
  // the finished sum of column j: lane b adds the span's four shares in order
  auto finish = [&](const double2& x, const double2& y) {
    double v = x.x;
    v = v + x.y;
    v = v + y.x;
    v = v + y.y;
    return wave_sum(lane < nblk ? v : 0.0);
  };
  const double eps = A.st->eps;
  int itr = A.st->itr, suc = 0, divzero = 0, last_i = 0, target = 0, cyc = 0;
  double fNorm = A.st->fNorm, fPrev = fNorm;
  const double rhs = own ? A.R[k] : 0.0;
  double x = own ? A.X[k] : 0.0;
  bool ok = true;
  for (; cyc < A.cycles; cyc++) {
    fPrev = fNorm;
    // u_0 = (R - A X) / |R - A X|
    if (own) st_agent(A.ex + k, x);
    if (!(ok = grid_sync<SPIN>(A.ctr, target, &okf))) break;
    double v = rhs - product(0);
    if (wv < 4) wl[wv][lane] = own ? v : 0.0;
    __syncthreads();
    if (wv == 0) {
      double a = 0.0;
#pragma unroll
      for (int r = 0; r < 4; r++) a = a + wl[r][lane] * wl[r][lane];
      put_part(0, wave_sum(a));
    }
    if (!(ok = grid_sync<SPIN>(A.ctr, target, &okf))) break;
    {
      const int c = 32 * min(lane, nblk - 1);
      const double e0 = sqrt(finish(bpart.ld2(c), bpart.ld2(c + 16)));
      itr++;
      if (e0 == 0.0) {
        divzero = 1;
        break;
      }
      v = v / e0;
      if (t == 0) sc[1] = e0;
    }
    if (own) {
      A.u[k] = v;
      st_agent(A.ex + n + k, v);
    }
    if (t == 0) stopf = 0;
    if (!(ok = grid_sync<SPIN>(A.ctr, target, &okf))) break;
    int i = 0;
    for (;; i++) {
      // the share's entries of u_0 .. u_i for the dots, column wv + 4 q, on their
      // way while the product is formed
      const int kb = 1024 * b + 64 * s + lane;
      double pu[GM_PF / 4][4];
#pragma unroll
      for (int q = 0; q < GM_PF / 4; q++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          pu[q][r] = 0.0;
          if (wv < 4 && wv + 4 * q <= i) pu[q][r] = A.u[(size_t)(wv + 4 * q) * A.ld + min(kb + 256 * r, n - 1)];
        }
      const double w = product((i & 1) ^ 1);
      if (wv < 4) wl[wv][lane] = own ? w : 0.0;
      __syncthreads();
      if (wv < 4) {
        double wr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) wr[r] = wl[r][lane];
        // one column: the four spans' rows in order, then the butterfly
        auto dot = [&](double u0, double u1, double u2, double u3) {
          double a = 0.0 + (kb < n ? u0 : 0.0) * wr[0];
          a = a + (kb + 256 < n ? u1 : 0.0) * wr[1];
          a = a + (kb + 512 < n ? u2 : 0.0) * wr[2];
          a = a + (kb + 768 < n ? u3 : 0.0) * wr[3];
          return wave_sum(a);
        };
#pragma unroll
        for (int q = 0; q < GM_PF / 4; q++)
          if (wv + 4 * q <= i) put_part(wv + 4 * q, dot(pu[q][0], pu[q][1], pu[q][2], pu[q][3]));
        for (int c = GM_PF + wv; c <= i; c += 16) {
          double ub[4][4];
#pragma unroll
          for (int q = 0; q < 4; q++)
#pragma unroll
            for (int r = 0; r < 4; r++)
              ub[q][r] = A.u[(size_t)min(c + 4 * q, i) * A.ld + min(kb + 256 * r, n - 1)];
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (c + 4 * q <= i) put_part(c + 4 * q, dot(ub[q][0], ub[q][1], ub[q][2], ub[q][3]));
        }
        if (((i + 1) & 3) == wv) put_part(i + 1, dot(wr[0], wr[1], wr[2], wr[3]));
      }
      // this lane's entries for the update, on their way over the barrier
      double pv[GM_PF];
#pragma unroll
      for (int q = 0; q < GM_PF; q++) {
        pv[q] = 0.0;
        if (wv < 4 && q <= i) pv[q] = A.u[(size_t)q * A.ld + min(k, n - 1)];
      }
      if (!(ok = grid_sync<SPIN>(A.ctr, target, &okf))) break;
      for (int c = wv; wv < 4 && c <= i + 1; c += 16) {
        double2 p0[4], p1[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int byte = 8 * (4 * nblk * min(c + 4 * q, i + 1) + 4 * min(lane, nblk - 1));
          p0[q] = bpart.ld2(byte);
          p1[q] = bpart.ld2(byte + 16);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const double f = finish(p0[q], p1[q]);
          if (lane == 0 && c + 4 * q <= i + 1) sums[c + 4 * q] = f;
        }
      }
      __syncthreads();
      if (t < 64) {
        // h(i+1, i) by the Pythagorean norm, 1 / h(i+1, i) (gmres.cpp:556-566)
        double hh = sums[i + 1];
#pragma unroll 8
        for (int j = 0; j <= i; j++) hh = hh - sums[j] * sums[j];
        hh = sqrt(fabs(hh));
        if (t == 0) {
          lh[i + 1] = hh;
          sc[0] = 1.0 / hh;
        }
      }
      __syncthreads();
      if (wv == 4) {
        // Givens rotations and the stop test (gmres.cpp:568-592), beside the update
        if (lane == 0) {
          const double hh = lh[i + 1];
          double cur = sums[0];
          for (int j = 0; j < i; j++) {
            const double nx = sums[j + 1];
            const double tmp = lcs[j] * cur + lsn[j] * nx;
            cur = -lsn[j] * cur + lcs[j] * nx;
            lh[j] = tmp;
          }
          const double tmp = sqrt(cur * cur + hh * hh);
          const double c = cur / tmp, sv = hh / tmp;
          lcs[i] = c;
          lsn[i] = sv;
          lh[i] = tmp;
          const double ei = sc[1], e1 = -sv * ei;
          sc[1] = e1;
          sc[2] = c * ei;
          stopf = fabs(e1) < eps ? 1 : 0;
        }
      }
      if (wv < 4) {
        double z = w;
#pragma unroll
        for (int q = 0; q < GM_PF; q++)
          if (q <= i) z = z + (-sums[q]) * pv[q];
        for (int jq = GM_PF; jq <= i; jq += 8) {
          double q8[8];
#pragma unroll
          for (int q = 0; q < 8; q++) q8[q] = A.u[(size_t)min(jq + q, i) * A.ld + min(k, n - 1)];
#pragma unroll
          for (int q = 0; q < 8; q++)
            if (jq + q <= i) z = z + (-sums[jq + q]) * q8[q];
        }
        z = sc[0] * z;
        if (own) {
          if (i + 1 < A.sD) A.u[(size_t)(i + 1) * A.ld + k] = z;
          st_agent(A.ex + (size_t)(i & 1) * n + k, z);
        }
      }
      ok = grid_sync<SPIN>(A.ctr, target, &okf);
      itr++;
      if (blockIdx.x == 0) {
        // column i of the triangle and err(i), for the back substitution
        for (int j = t; j <= i; j += GM_BS) A.h[(size_t)(A.sD + 1) * i + j] = lh[j];
        if (t == 0) {
          A.y[i] = sc[2];
          A.y[i + 1] = sc[1];
        }
      }
      if (!ok || stopf || i + 1 == A.sD) break;
    }
    if (!ok) break;
    last_i = i;
    suc = stopf;
    fNorm = fabs(sc[1]);
    __syncthreads();
    // back substitution (gmres.cpp:595-608) by workgroup 0: a row's products by a
    // wavefront (the next row's entries loaded ahead), their sum in order
    double *y = lcs, *pr = lsn;
    if (blockIdx.x == 0 && wv == 0) {
      auto tri = [&](int j, int c) { return A.h[(size_t)(A.sD + 1) * min(c, last_i) + j]; };
      double h0 = tri(last_i, lane), h1 = tri(last_i, lane + 64), h2 = tri(last_i, lane + 128),
             h3 = tri(last_i, lane + 192);
      for (int j = lane; j <= last_i; j += 64) y[j] = A.y[j];
      wave_sync();
      for (int j = last_i; j >= 0; j--) {
        auto put = [&](int c, double hv) {
          if (c >= j && c <= last_i) pr[c] = c > j ? hv * y[c] : hv;
        };
        put(lane, h0);
        put(lane + 64, h1);
        put(lane + 128, h2);
        put(lane + 192, h3);
        const int nx = max(j - 1, 0);
        h0 = tri(nx, lane);
        if (last_i >= 64) h1 = tri(nx, lane + 64), h2 = tri(nx, lane + 128), h3 = tri(nx, lane + 192);
        wave_sync();
        double a = y[j];
#pragma unroll 8
        for (int c = j + 1; c <= last_i; c++) a = a - pr[c];
        a = a / pr[j];
        wave_sync();
        if (lane == 0) y[j] = a;
        wave_sync();
      }
      for (int j = lane; j <= last_i; j += 64) st_agent(A.y + GM_MAX + j, y[j]);
    }
    if (!(ok = grid_sync<SPIN>(A.ctr, target, &okf))) break;
    for (int j = t; j <= last_i; j += GM_BS) sums[j] = ld_agent(A.y + GM_MAX + j);
    __syncthreads();
    for (int jq = 0; jq <= last_i; jq += 8) {
      double q8[8];
#pragma unroll
      for (int q = 0; q < 8; q++) q8[q] = A.u[(size_t)min(jq + q, last_i) * A.ld + min(k, n - 1)];
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (jq + q <= last_i) x = x + sums[jq + q] * q8[q];
    }
    __syncthreads();
    if (suc) {
      cyc++;
      break;
    }
  }
  if (own) A.X[k] = x;
  if (t == 0) {
    if (!ok) __hip_atomic_store(&A.st->pad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (blockIdx.x == 0) {
      A.st->itr = itr;
      A.st->suc = suc;
      A.st->divzero = divzero;
      A.st->last_i = last_i;
      A.st->cyc = cyc;
      A.st->fNorm = fNorm;
      A.st->fStart = fPrev;
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

// A cooperative launch, timed by events around it (the launch has no event
// arguments of its own: a few microseconds of dispatch are timed with it).
hipError_t launch_cooperative(const char* name, const void* kernel, unsigned grid, unsigned block, void** args,
                              unsigned lds, hipStream_t s)
{
  hipEvent_t a = nullptr, b = nullptr;
  const size_t mark = prof_mark();
  const bool timed = prof_begin(name, s, 0.0, &a, &b) >= 0;
  if (timed) (void)hipEventRecord(a, s);
  const hipError_t e = hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(block), args, lds, s);
  if (timed && e == hipSuccess)
    (void)hipEventRecord(b, s);
  else if (timed)
    prof_drop(mark, mark + 1);
  return e;
}

const void* cg_kernel(bool wait)
{
  return wait ? reinterpret_cast<const void*>(&k_cg_small<SPIN_MAX>) : reinterpret_cast<const void*>(&k_cg_small<0>);
}
const void* gmres_kernel(bool wait)
{
  return wait ? reinterpret_cast<const void*>(&k_gmres_small<SPIN_MAX>)
              : reinterpret_cast<const void*>(&k_gmres_small<0>);
}

// No memory for its buffers, the launch refused, or its workgroups did not meet:
// the per-launch path, for the lhs's later solves too.
int missed(svg_lhs* L)
{
  L->oneLaunch = false;
  L->oneLaunchRuns.missed++;
  return SVG_OK;
}

}  // namespace

// The most blocks of a workgroup and the most different columns they touch:
// workgroup w's rows are the ranges [a, e) that part(w, r, a, e) gives for r < parts.
template <typename Part>
static void most_blocks(const svg_lhs* L, int wgs, int parts, Part part, int* cap, int* capU)
{
  *cap = *capU = 0;
  std::vector<int> seen(L->nNo, -1);
  for (int w = 0; w < wgs; w++) {
    int nb = 0, nu = 0;
    for (int r = 0; r < parts; r++) {
      int a, e;
      part(w, r, a, e);
      nb += L->rowPtr[e] - L->rowPtr[a];
      for (int j = L->rowPtr[a]; j < L->rowPtr[e]; j++)
        if (seen[L->colPtr[j]] != w) seen[L->colPtr[j]] = w, nu++;
    }
    *cap = std::max(*cap, nb);
    *capU = std::max(*capU, nu);
  }
}

// The Schur CG of w's split system as one launch: *ran = 0 when the system does
// not fit (more workgroups than compute units, or blocks than LDS) or the
// workgroups did not meet; else the result is in w.cgX and w.h_cg (synchronises).
int cg_small(svg_lhs* L, const double* R, int mItr, double absTol, double relTol, hipStream_t s, int* ran)
{
  auto& w = L->ns;
  *ran = 0;
  if (!L->oneLaunch || w.smallRows < 0) return SVG_OK;
  const int nNo = L->nNo;
  int rc;
  auto bytes = [](int cap, int capU) { return (size_t)CG_BLK_B * cap + (size_t)CG_COL_B * capU; };
  if (w.smallRows == 0) {
    int cus = 0;
    w.smallRows = -1;
    if ((rc = num_cus(&cus))) return rc;
    if (nNo > 1024 * SUM_SPANS) return SVG_OK;
    for (int rows : {128, 64}) {
      const int wgs = (int)blocks_for(nNo, rows);
      if (wgs > cus) continue;
      int cap, capU;
      auto part = [&](int w, int, int& a, int& e) { a = w * rows, e = std::min(nNo, a + rows); };
      most_blocks(L, wgs, 1, part, &cap, &capU);
      if (bytes(cap, capU) > 148 * 1024) continue;
      for (bool wait : {false, true})
        if (hipFuncSetAttribute(cg_kernel(wait), hipFuncAttributeMaxDynamicSharedMemorySize, 148 * 1024) !=
            hipSuccess) {
          (void)hipGetLastError();
          return SVG_OK;
        }
      if (dev_alloc(&w.cgEx, (size_t)8 * nNo) || dev_alloc(&w.ctr, 1)) {
        dev_free(w.cgEx);
        (void)hipGetLastError();
        return missed(L);
      }
      w.smallRows = rows;
      w.smallCap = cap;
      w.smallCapU = capU;
      break;
    }
    if (w.smallRows < 0) return SVG_OK;
  }
  int rows = w.smallRows, cap = w.smallCap, capU = w.smallCapU, n = nNo;
  hipLaunchKernelGGL(k_clear_small, dim3(1), dim3(1), 0, s, w.ctr, &w.cg->pad);
  const int *rp = L->d_rowPtr, *cp = L->d_colPtr;
  const double *mG = w.mG, *Gt = w.Gt, *mL = w.mL;
  double *X = w.cgX, *gpp = w.cgEx, *pr = w.cgEx + (size_t)4 * nNo, *prod = w.cgEx + (size_t)6 * nNo,
         *rcv = w.cgEx + (size_t)7 * nNo;
  void* args[] = {&n,    &rp,   &cp,   &mG,    &Gt,  &mL,   &R,    &X,    &pr,     &gpp,
                  &prod, &rcv,  &w.cg, &w.ctr, &rows, &cap, &capU, &mItr, &absTol, &relTol};
  if (launch_cooperative("cg_small", cg_kernel(L->oneLaunchWait), blocks_for(nNo, rows), CG_BS, args,
                         (unsigned)bytes(cap, capU), s) != hipSuccess) {
    (void)hipGetLastError();
    return missed(L);
  }
  SVG_HIP(hipMemcpyAsync(w.h_cg, w.cg, sizeof(CgState), hipMemcpyDeviceToHost, s));
  SVG_HIP(hipStreamSynchronize(s));
  if (w.h_cg->pad) return missed(L);
  *ran = 1;
  L->oneLaunchRuns.cg++;
  return SVG_OK;
}

// Restart cycles of gmres_v for the system (Val, R) with X = 0 in L->kw.X and
// the initial state in L->kw.st, in launches of up to GM_CYCLES cycles: *ran = 0
// when the system does not fit (a workgroup per compute unit, its blocks in LDS)
// or the workgroups did not meet, else the state after the last cycle is in
// L->kw.h_st, fStart the residual norm before it (synchronises).
constexpr int GM_CYCLES = 16;
constexpr int GM_LDS = 149 * 1024;  // of 160 KB, 10 KB are the kernel's own arrays

bool gmres_small_fits(svg_lhs* L, int sD)
{
  auto& k = L->kw;
  if (!L->oneLaunch) return false;
  if (k.smallCap == 0) {
    k.smallCap = -1;
    const int nNo = L->nNo, nblk = (4 * nNo + 1023) / 1024;
    int cus = 0, cap = 0, capU = 0;
    if (num_cus(&cus) != SVG_OK || 4 * nblk > cus || nblk > 64) return false;
    auto part = [&](int w, int r, int& a, int& e) {
      a = std::min(nNo, 256 * (w / 4) + 64 * r + 16 * (w % 4)), e = std::min(nNo, a + 16);
    };
    most_blocks(L, 4 * nblk, 4, part, &cap, &capU);
    if ((size_t)GM_BLK_B * cap + (size_t)GM_COL_B * capU > GM_LDS) return false;
    for (bool wait : {false, true})
      if (hipFuncSetAttribute(gmres_kernel(wait), hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
    k.smallCap = cap;
    k.smallCapU = capU;
  }
  return k.smallCap > 0 && sD < GM_MAX - 1;
}

int gmres_small(svg_lhs* L, const svg_subls* ls, const double* Val, const double* R, hipStream_t s, int* ran)
{
  auto& k = L->kw;
  *ran = 0;
  const int n = k.n, nblk = (n + 1023) / 1024;
  const size_t nPart = (size_t)4 * nblk * (k.sD + 1);
  if ((!k.small && dev_alloc(&k.small, nPart + 2 * (size_t)n + 2 * GM_MAX)) || (!k.ctr && dev_alloc(&k.ctr, 1))) {
    (void)hipGetLastError();
    return missed(L);
  }
  GmSmall A{};
  A.nNo = L->nNo;
  A.sD = ls->sD;
  A.cap = k.smallCap;
  A.capU = k.smallCapU;
  A.rowPtr = L->d_rowPtr;
  A.colPtr = L->d_colPtr;
  A.K = Val;
  A.R = R;
  A.X = k.X;
  A.u = k.u;
  A.part = k.small;
  A.ex = k.small + nPart;
  A.y = A.ex + 2 * (size_t)n;
  A.h = k.h;
  A.ld = k.ld;
  A.st = k.st;
  A.ctr = k.ctr;
  const unsigned bytes = (unsigned)(GM_BLK_B * A.cap + GM_COL_B * A.capU);
  for (int done = 0; done < ls->mItr;) {
    A.cycles = std::min(GM_CYCLES, ls->mItr - done);
    hipLaunchKernelGGL(k_clear_small, dim3(1), dim3(1), 0, s, k.ctr, &k.st->pad);
    void* args[] = {&A};
    if (launch_cooperative("gmres_small", gmres_kernel(L->oneLaunchWait), 4 * nblk, GM_BS, args, bytes, s) !=
        hipSuccess) {
      (void)hipGetLastError();
      return missed(L);
    }
    SVG_HIP(hipMemcpyAsync(k.h_st, k.st, sizeof(GmState), hipMemcpyDeviceToHost, s));
    SVG_HIP(hipStreamSynchronize(s));
    if (k.h_st->pad) return missed(L);
    done += A.cycles;
    if (k.h_st->suc || k.h_st->divzero) break;
  }
  *ran = 1;
  L->oneLaunchRuns.gmres++;
  return SVG_OK;
}

}  // namespace svg

using namespace svg;

extern "C" int svg_one_launch_info(const svg_lhs* L, svg_one_launch* info)
{
  if (!L || !info) return set_error(SVG_ERR_ARG, "svg_one_launch_info: null argument");
  *info = L->oneLaunchRuns;
  info->cg_rows = L->ns.smallRows;
  return SVG_OK;
}

extern "C" int svg_one_launch_set(svg_lhs* L, int on, int wait)
{
  if (!L) return set_error(SVG_ERR_ARG, "svg_one_launch_set: null lhs");
  L->oneLaunch = on != 0;
  L->oneLaunchWait = wait != 0;
  return SVG_OK;
}
