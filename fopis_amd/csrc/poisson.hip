// Poisson solve for the ES step: FP64 defect correction around geometric
// multigrid V-cycles (red-black SOR smoother, full-weighting restriction,
// trilinear prolongation) on the vertex-centred node grid.
//
// It solves the reference's discrete problem (RootGridField.cpp:105-264):
// the 7-point operator 6 phi - sum(neighbours) = rho_coeff * rho[0] at nodes
// 2..n-1 of each axis (glue indexing), with the face nodes held at their
// current values (0 on Dirichlet faces), then applies the face conditions
// (Field.cpp:10-96). The reference reaches it by zebra SOR; this build stops
// on ||b - A phi||_2 / ||b||_2 <= tol in FP64.
//
// Launch structure. The host queues cycles in batches without waiting: every
// kernel of a cycle first reads a device flag that the norm kernel sets once
// the tolerance (or the cycle cap) is reached, and returns at once when it is
// set, so a batch that overshoots costs only empty launches. The host reads
// the flag once per batch. The coarse levels whose arrays fit in LDS run as
// one single-workgroup kernel per cycle.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <cstdlib>
#include <type_traits>

#include "fopis_internal.hpp"

#pragma clang fp contract(off)

namespace fopis {

namespace {

struct Lv {
  int n0, n1, n2;
  int64_t sx, sy;
};

// Workgroups are handed to the 8 XCDs round-robin by linear id, and each XCD
// has its own L2. Renumber them so that XCD x runs a contiguous run of the
// logical ids (whole planes of the level), keeping a stencil's neighbour rows
// in the same L2. The map is a bijection for any grid size.
__device__ inline int xcd_block(int p, int n) {
  const int per = n >> 3, rem = n & 7, x = p & 7, slot = p >> 3;
  return x * per + min(x, rem) + slot;
}

// (chunk, row, plane) of the calling workgroup in a 3-D launch, XCD-renumbered.
__device__ inline void block3(int& bx, int& by, int& bz) {
  const int gx = gridDim.x, gy = gridDim.y;
  const int n = gx * gy * gridDim.z;
  const int L = xcd_block(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), n);
  bx = L % gx;
  by = (L / gx) % gy;
  bz = L / (gx * gy);
}

// The level-0 passes below (residuals, update) walk the interior by rows:
// each workgroup takes one contiguous range of (a, b) rows (XCD-renumbered, so
// that neighbouring planes stay in one XCD's L2) and spreads its 256 threads
// over 1, 2 or 4 rows at a time, a row's points over 256, 128 or 64 threads.
// f(g, a, b, c) gets the node index and the coordinates of every interior point once.
template <class F>
__device__ inline void for_interior_rows(const int n0, const int n1, const int n2, const int64_t sx,
                                         const int64_t sy, F&& f) {
  const int nrows = n0 * n1;
  const int per = (nrows + (int)gridDim.x - 1) / (int)gridDim.x;
  const int r0 = xcd_block(blockIdx.x, gridDim.x) * per;
  const int r1 = min(r0 + per, nrows);
  const int tpr = n2 <= 64 ? 64 : (n2 <= 128 ? 128 : 256);  // threads per row
  const int sub = threadIdx.x / tpr, lane = threadIdx.x % tpr;
  for (int row = r0 + sub; row < r1; row += 256 / tpr) {
    const int a = row / n1 + 1, b = row % n1 + 1;
    const int64_t base = a * sx + b * sy;
    for (int c = lane + 1; c <= n2; c += tpr) f(base + c, a, b, c);
  }
}

// b = rc * rho at the level-0 interior; r = b - A phi written as P;
// per-block partial sums of r^2 and b^2 in FP64.
// (r64, when given, receives the FP64 residual that the cycle updates keep;
// with r and r64 both null only the norms are formed: the check at a solve's end.)
template <class P>
__global__ __launch_bounds__(256) void k_resid0(const double* __restrict__ phi, const double* __restrict__ rho,
                                                double rc, P* __restrict__ r, Lv L, double* part,
                                                const int* __restrict__ done, double* __restrict__ r64) {
  if (*done) return;
  __shared__ double s1[256], s2[256];
  double rr = 0.0, bb = 0.0;
  for_interior_rows(L.n0, L.n1, L.n2, L.sx, L.sy, [&](const int64_t g, int, int, int) {
    const double bv = rc * rho[g];
    const double ap = 6.0 * phi[g] - (phi[g - L.sx] + phi[g + L.sx] + phi[g - L.sy] + phi[g + L.sy] + phi[g - 1] +
                                      phi[g + 1]);
    const double rv = bv - ap;
    if (r) r[g] = (P)rv;
    if (r64) r64[g] = rv;
    rr += rv * rv;
    bb += bv * bv;
  });
  s1[threadIdx.x] = rr;
  s2[threadIdx.x] = bb;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = s2[0];
  }
}

// Solve state on the device: st[0] done flag, st[1] cycles applied, st[2] 0
// once the true residual has confirmed the end, st[3] stays 0 (the done flag of
// launches that always run), st[4] the current pair's skip flag, st[5] FP64
// updates applied, st[6] pair residual passes run, st[7] the opposite of st[0]
// (the done flag of launches that run once the cycles are done); dst[0..2] =
// ||r||^2, ||b||^2, relative residual of the last check, dst[3] the relative
// residual the solve started from. The first check of a solve sets them.

// After a V-cycle's correction e: phi += e and the FP64 residual
// r = b - A phi is updated as r -= A e (exact up to FP64 rounding, so no
// stencil over phi is needed), its P copy becomes the next cycle's right-hand
// side, and per-block partial sums of r^2 are written (the b^2 slot is 0).
// Reads e at neighbours and writes phi, r only at the point itself.
template <class P>
__global__ __launch_bounds__(256) void k_update(double* __restrict__ phi, const P* __restrict__ e, double* r64,
                                                P* rp, Lv L, double* part, const int* __restrict__ done) {
  if (*done) return;
  __shared__ double s1[256];
  const bool same = (const void*)rp == (const void*)r64;
  double rr = 0.0;
  for_interior_rows(L.n0, L.n1, L.n2, L.sx, L.sy, [&](const int64_t g, int, int, int) {
    const double eg = (double)e[g];
    const double ae = 6.0 * eg - ((double)e[g - L.sx] + (double)e[g + L.sx] + (double)e[g - L.sy] +
                                  (double)e[g + L.sy] + (double)e[g - 1] + (double)e[g + 1]);
    const double rv = r64[g] - ae;
    r64[g] = rv;
    if (!same) rp[g] = (P)rv;
    phi[g] += eg;
    rr += rv * rv;
  });
  s1[threadIdx.x] = rr;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s1[threadIdx.x] += s1[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = 0.0;
  }
}

// Between the two V-cycles of a pair: per-block partial sums of t^2, t = r - A e
// at the level-0 interior (the cycles' right-hand side and the first cycle's
// correction; t formed in P as the cycles form it, its squares summed in
// FP64; the b^2 slot is 0).
template <class P>
__global__ __launch_bounds__(256) void k_pair_resid(const P* __restrict__ e, const P* __restrict__ r, Lv L,
                                                    double* part, const int* __restrict__ done) {
  if (*done) return;
  __shared__ double s1[256];
  double rr = 0.0;
  for_interior_rows(L.n0, L.n1, L.n2, L.sx, L.sy, [&](const int64_t g, int, int, int) {
    const P t = r[g] - ((P)6 * e[g] - (e[g - L.sx] + e[g + L.sx] + e[g - L.sy] + e[g + L.sy] + e[g - 1] + e[g + 1]));
    rr += (double)t * (double)t;
  });
  s1[threadIdx.x] = rr;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s1[threadIdx.x] += s1[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = 0.0;
  }
}

// The pair's decision (one block, fixed tree): skip[0] = 1, so that every
// kernel of the second V-cycle returns at once, when the solve is already
// done or the first cycle's correction alone reaches the tolerance (against
// ||b||^2 of the solve's start, dst[1]). The residual after the first cycle is
// the cycles' right-hand side minus A e; that right-hand side is the FP64
// residual rounded to P, whose rounding (~1e-7 of it in FP32) is far below
// the ~30x a V-cycle removes, so the test agrees with the FP64 check that
// follows the update except within rounding of the tolerance itself.
__global__ __launch_bounds__(256) void k_pair_check(const double* part, int nb, const double* dst, int* st,
                                                    double tol, int* skip) {
  __shared__ double s1[256];
  double a = 0.0;
  for (int i = threadIdx.x; i < nb; i += 256) a += part[2 * i];
  s1[threadIdx.x] = a;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s1[threadIdx.x] += s1[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double rr = s1[0], bb = dst[1];
    const double rel = bb > 0.0 ? sqrt(rr / bb) : sqrt(rr);
    skip[0] = (st[0] || rel <= tol || (bb == 0.0 && rr < 1e-300)) ? 1 : 0;
    if (!st[0]) st[6] += 1;  // (a pass that ran; k_pair_resid returns at once once done)
  }
}

// Sums of the residual partials over a block (fixed tree: deterministic), in s1[0] and s2[0].
__device__ __forceinline__ void sum_partials(const double* part, int nb, double* s1, double* s2) {
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < nb; i += 256) {
    a += part[2 * i];
    b += part[2 * i + 1];
  }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = b;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
}

// Cycle count and the stopping test of the solve loop. FIRST: of the residual
// the solve starts from, which also sets the solve's state. The others keep
// the ||b||^2 in dst[1] (their partials carry r^2 only); count_cycle V-cycles
// were applied, less one when *skipped (a pair whose second cycle was skipped).
template <bool FIRST>
__global__ __launch_bounds__(256) void k_norm(const double* part, int nb, double* dst, int* st, double tol,
                                              int max_cycles, int count_cycle, const int* skipped) {
  if (!FIRST && st[0]) return;
  __shared__ double s1[256], s2[256];
  sum_partials(part, nb, s1, s2);
  if (threadIdx.x == 0) {
    const double rr = s1[0], bb = FIRST ? s2[0] : dst[1];
    const int cyc = FIRST ? 0 : st[1] + count_cycle - (skipped ? skipped[0] : 0);
    const double rel = bb > 0.0 ? sqrt(rr / bb) : sqrt(rr);
    dst[0] = rr;
    dst[1] = bb;
    dst[2] = rel;
    if (FIRST) dst[3] = rel;
    const int end = (rel <= tol || (bb == 0.0 && rr < 1e-300) || cyc >= max_cycles) ? 1 : 0;
    st[0] = end;
    st[1] = cyc;
    if (FIRST) st[2] = 1;
    st[5] = FIRST ? 0 : st[5] + 1;  // an FP64 update preceded this check
    if (FIRST) st[6] = 0;
    st[7] = 1 - end;
  }
}

// What the host reads after a round of cycles (pinned memory it and the device share).
struct SolveWords {
  int32_t done, confirmed, cycles, updates, pair_passes;
  double relres, relres0;
};

// Once the cycles are done: the true residual's norms, and whether they confirm
// the end. The words go to the host directly; with two
// copies, a second wait and a launch per face a solve took 47 to 70 us more
// (33^3: step 634 us, now 587; 17^3 alone: 379 us, now 310).
__global__ __launch_bounds__(256) void k_norm_final(const double* part, int nb, double* dst, int* st, double tol,
                                                    int max_cycles, SolveWords* out) {
  __shared__ double s1[256], s2[256];
  const int done = st[0];
  if (done) sum_partials(part, nb, s1, s2);
  if (threadIdx.x == 0) {
    int good = 0;
    if (done) {
      const double rr = s1[0], bb = s2[0];
      const double rel = bb > 0.0 ? sqrt(rr / bb) : sqrt(rr);
      dst[0] = rr;
      dst[1] = bb;
      dst[2] = rel;
      good = (rel <= tol || (bb == 0.0 && rr < 1e-300) || st[1] >= max_cycles) ? 1 : 0;
    }
    st[2] = 1 - good;
    out->done = done;
    out->confirmed = good;
    out->cycles = st[1];
    out->updates = st[5];
    out->pair_passes = st[6];
    out->relres = dst[2];
    out->relres0 = dst[3];
  }
}

__global__ void k_reopen(int* st) {
  st[0] = 0;
  st[7] = 1;
}

// Kernels over a level's interior give each thread the same column position
// in kRows consecutive rows (b), issue every load of those rows before the
// first store, and so keep several independent loads in flight per thread.
constexpr int kRows = 4;

// Red-black SOR half-sweep over points with (a+b+c) % 2 == color:
// e = (1-w) e + (w/6) (sum of neighbours + r). A half-sweep reads only points
// of the other colour and writes only its own, so the loads of all rows may
// precede the stores.
template <class P>
__global__ void k_smooth(P* __restrict__ e, const P* __restrict__ r, Lv L, int color, P w1, P w6,
                         const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int m = bx * blockDim.x + threadIdx.x;
  const int a = bz + 1;
  P val[kRows];
  int64_t gg[kRows];
  bool ok[kRows];
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    const int c = (((a + b + 1) & 1) == color ? 1 : 2) + 2 * m;
    ok[q] = b <= L.n1 && c <= L.n2;
    const int64_t g = a * L.sx + (ok[q] ? b : 1) * L.sy + (ok[q] ? c : 1);
    gg[q] = g;
    const P nb = e[g - L.sx] + e[g + L.sx] + e[g - L.sy] + e[g + L.sy] + e[g - 1] + e[g + 1];
    val[q] = w1 * e[g] + w6 * (nb + r[g]);
  }
#pragma unroll
  for (int q = 0; q < kRows; ++q)
    if (ok[q]) e[gg[q]] = val[q];
}

// First full sweep of a cycle from e = 0, both colours in one pass: red
// points get (w/6) r, black points the black half-sweep over those red values
// (formed here from r): the operations of a red half-sweep from zero (red
// points (w/6) r, black points cleared) followed by the black half-sweep, in
// the same order (the compiler's fused multiply-adds may round them
// differently), but r is read once and e written once. Points outside the
// interior have r = 0 and so read as red values of 0, as the untouched level
// borders do.
template <class P>
__global__ void k_smooth_first2(P* __restrict__ e, const P* __restrict__ r, Lv L, P w1, P w6,
                                const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  // two neighbouring points of a row per thread, one of each colour, so the
  // lanes of a wavefront all take the same path; every load of the kRows rows
  // is issued before the first store (rows past the level read row 1 instead)
  const int c0 = 2 * (bx * blockDim.x + threadIdx.x) + 1;
  const int a = bz + 1;
  if (c0 > L.n2) return;
  const bool two = c0 + 1 <= L.n2;
  P vb[kRows], vr[kRows];
  int64_t gbq[kRows], grq[kRows];
  bool okq[kRows], fbq[kRows];
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    okq[q] = b <= L.n1;
    const int bb = okq[q] ? b : 1;
    const int64_t g0 = a * L.sx + bb * L.sy + c0;
    // the black point of the pair is c0 when (a + b + c0) is odd, else c0 + 1
    fbq[q] = ((a + bb + c0) & 1) != 0;
    const int64_t gb = fbq[q] ? g0 : g0 + 1;
    const int64_t gr = fbq[q] ? g0 + 1 : g0;
    gbq[q] = gb;
    grq[q] = gr;
    const P nb = w6 * r[gb - L.sx] + w6 * r[gb + L.sx] + w6 * r[gb - L.sy] + w6 * r[gb + L.sy] + w6 * r[gb - 1] +
                 w6 * r[gb + 1];
    vb[q] = w1 * (P)0 + w6 * (nb + r[gb]);
    vr[q] = w6 * r[gr];
  }
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    if (!okq[q]) continue;
    if (fbq[q] || two) e[gbq[q]] = vb[q];
    if (!fbq[q] || two) e[grq[q]] = vr[q];
  }
}

template <class P>
__device__ inline P fw_weight(int da, int db, int dc) {
  const int nz = (da != 0) + (db != 0) + (dc != 0);
  return nz == 0 ? (P)1 : (nz == 1 ? (P)0.5 : (nz == 2 ? (P)0.25 : (P)0.125));
}

// Full weighting of the fine residual r - A e to the coarse grid, scaled by 4
// for the unscaled 2h operator; the residual of each of the 27 fine points is
// formed on the fly (no residual array is written).
template <class P>
__global__ void k_restrict_resid(P* __restrict__ rc, Lv C, const P* __restrict__ e, const P* __restrict__ r, Lv F,
                                 const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int c = bx * blockDim.x + threadIdx.x + 1;
  const int b = by + 1, a = bz + 1;
  if (c > C.n2) return;
  const int64_t f = (2 * a) * F.sx + (2 * b) * F.sy + 2 * c;
  P acc = 0;
#pragma unroll
  for (int da = -1; da <= 1; ++da)
#pragma unroll
    for (int db = -1; db <= 1; ++db)
#pragma unroll
      for (int dc = -1; dc <= 1; ++dc) {
        const int64_t g = f + da * F.sx + db * F.sy + dc;
        const P t = r[g] - ((P)6 * e[g] - (e[g - F.sx] + e[g + F.sx] + e[g - F.sy] + e[g + F.sy] + e[g - 1] + e[g + 1]));
        acc += fw_weight<P>(da, db, dc) * t;
      }
  rc[a * C.sx + b * C.sy + c] = acc * (P)0.5;  // (4/8) * sum
}

// The residual t = r - A e at every interior point of a level, kRows rows per
// thread (the same expression as the restriction forms on the fly).
template <class P>
__global__ void k_resid_level(P* __restrict__ t, const P* __restrict__ e, const P* __restrict__ r, Lv L,
                              const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int c = bx * blockDim.x + threadIdx.x + 1;
  const int a = bz + 1;
  if (c > L.n2) return;
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    if (b > L.n1) break;
    const int64_t g = a * L.sx + b * L.sy + c;
    t[g] = r[g] - ((P)6 * e[g] - (e[g - L.sx] + e[g + L.sx] + e[g - L.sy] + e[g + L.sy] + e[g - 1] + e[g + 1]));
  }
}

// Full weighting of a residual already formed (k_resid_level), in the same
// order as k_restrict_resid: on large levels every fine residual is then
// computed once instead of once per coarse point that weights it.
template <class P>
__global__ void k_restrict_t(P* __restrict__ rc, Lv C, const P* __restrict__ t, Lv F, const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int c = bx * blockDim.x + threadIdx.x + 1;
  const int b = by + 1, a = bz + 1;
  if (c > C.n2) return;
  const int64_t f = (2 * a) * F.sx + (2 * b) * F.sy + 2 * c;
  P acc = 0;
#pragma unroll
  for (int da = -1; da <= 1; ++da)
#pragma unroll
    for (int db = -1; db <= 1; ++db)
#pragma unroll
      for (int dc = -1; dc <= 1; ++dc) acc += fw_weight<P>(da, db, dc) * t[f + da * F.sx + db * F.sy + dc];
  rc[a * C.sx + b * C.sy + c] = acc * (P)0.5;  // (4/8) * sum
}

// e_fine += trilinear interpolation of e_coarse (coarse node A sits at fine 2A).
template <class P>
__global__ void k_prolong(P* __restrict__ e, Lv F, const P* __restrict__ ec, Lv C, const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int c = bx * blockDim.x + threadIdx.x + 1;
  const int a = bz + 1;
  if (c > F.n2) return;
  const int a0 = a >> 1, a1 = (a + 1) >> 1, c0 = c >> 1, c1 = (c + 1) >> 1;
  auto E = [&](int x, int y, int z) { return ec[x * C.sx + y * C.sy + z]; };
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    if (b > F.n1) break;
    const int b0 = b >> 1, b1 = (b + 1) >> 1;
    const P v = (E(a0, b0, c0) + E(a1, b0, c0) + E(a0, b1, c0) + E(a1, b1, c0) + E(a0, b0, c1) + E(a1, b0, c1) +
                 E(a0, b1, c1) + E(a1, b1, c1)) *
                (P)0.125;
    e[a * F.sx + b * F.sy + c] += v;
  }
}

// ---- the finest FP32 level stored by colour ------------------------------
//
// A red-black half-sweep updates the points of one colour from those of the
// other. With both colours in one array every cache line holds both, so a
// half-sweep reads all of e and r and writes all of e: 201 MB per half-sweep
// at 255^3 where the data it needs is 136 MB. Stored by colour, it reads the
// other colour's e and its own e and r and writes its own e, each half-array
// once. Point (a, b, c) of the padded level (interior 1..n) has colour
// (a + b + c) & 1 and sits at a * sx + b * sy + c / 2 of its colour's array
// (rows of (n2 + 3) / 2); its x neighbours c - 1 and c + 1 are at (c - 1) / 2
// and (c + 1) / 2 of the other colour's row, its y and z neighbours at c / 2
// of the other colour's neighbouring rows. Every kernel here forms the same
// sums in the same order as its one-array counterpart, so a solve gives the
// same result bit for bit either way.
struct Rb {
  float* e;  // colour 0; colour 1 at + cs
  float* r;
  int64_t cs, sx, sy;
  int n0, n1, n2;
};

__device__ inline int64_t rb_at(const Rb& R, int a, int b, int c) {
  return a * R.sx + b * R.sy + (c >> 1) + (((a + b + c) & 1) ? R.cs : 0);
}

// A point's slot i in its colour's array, that array (own) and the other
// colour's (oth), where all six neighbours are: oth[i -+ sx], oth[i -+ sy],
// and oth[i + xm], oth[i + xp] for c - 1 and c + 1.
struct RbPt {
  int64_t i;
  int64_t own, oth;  // offsets of the two colours' arrays
  int xm, xp;
};

__device__ inline RbPt rb_pt(const Rb& R, int a, int b, int c) {
  const bool k = ((a + b + c) & 1) != 0, codd = (c & 1) != 0;
  return RbPt{a * R.sx + b * R.sy + (c >> 1), k ? R.cs : 0, k ? 0 : R.cs, codd ? 0 : -1, codd ? 1 : 0};
}

// A e at the point (6 e - the neighbours, summed in the one-array order:
// -x, +x, -y, +y, -z, +z in the level's a, b, c axes)
template <class T>
__device__ inline T rb_ae(const Rb& R, const RbPt& p) {
  const float* eo = R.e + p.own;
  const float* en = R.e + p.oth;
  return (T)6 * (T)eo[p.i] - ((T)en[p.i - R.sx] + (T)en[p.i + R.sx] + (T)en[p.i - R.sy] + (T)en[p.i + R.sy] +
                              (T)en[p.i + p.xm] + (T)en[p.i + p.xp]);
}

// Red-black half-sweep of colour `color` (k_smooth): thread j takes the j-th
// point of the colour in each of its rows (c = 2j + 1 or 2j + 2).
__global__ void k_smooth_rb(Rb R, int color, float w1, float w6, const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int j = bx * blockDim.x + threadIdx.x;
  const int a = bz + 1;
  float* own = R.e + (color ? R.cs : 0);
  const float* oth = R.e + (color ? 0 : R.cs);
  const float* ro = R.r + (color ? R.cs : 0);
  float val[kRows];
  int64_t ii[kRows];
  bool ok[kRows];
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    const int odd = (a + b + color) & 1;  // the row's points of this colour have odd c
    const int c = 2 * j + (odd ? 1 : 2), h = c >> 1;
    ok[q] = b <= R.n1 && c <= R.n2;
    // (a slot outside the level reads slot 1 of row 1 instead)
    const int64_t i = ok[q] ? a * R.sx + b * R.sy + h : a * R.sx + R.sy + 1;
    const bool codd = ok[q] && (c & 1) != 0;
    ii[q] = i;
    const float nb = oth[i - R.sx] + oth[i + R.sx] + oth[i - R.sy] + oth[i + R.sy] + oth[i + (codd ? 0 : -1)] +
                     oth[i + (codd ? 1 : 0)];
    val[q] = w1 * own[i] + w6 * (nb + ro[i]);
  }
#pragma unroll
  for (int q = 0; q < kRows; ++q)
    if (ok[q]) own[ii[q]] = val[q];
}

// First sweep of a cycle from e = 0 (k_smooth_first2): slot h of a row holds
// one red and one black point.
__global__ void k_smooth_first2_rb(Rb R, float w1, float w6, const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int h = bx * blockDim.x + threadIdx.x;
  const int a = bz + 1;
  const float* r0 = R.r;
  const float* r1 = R.r + R.cs;
  float vr[kRows], vb[kRows];
  int64_t ir[kRows], ib[kRows];
  bool okr[kRows], okb[kRows];
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    const int cr = 2 * h + ((a + b) & 1), cb = 2 * h + ((a + b + 1) & 1);
    okr[q] = b <= R.n1 && cr >= 1 && cr <= R.n2;
    okb[q] = b <= R.n1 && cb >= 1 && cb <= R.n2;
    ir[q] = okr[q] ? a * R.sx + b * R.sy + h : a * R.sx + R.sy + 1;
    ib[q] = okb[q] ? a * R.sx + b * R.sy + h : a * R.sx + R.sy + 1;
    vr[q] = w6 * r0[ir[q]];
    const int64_t i = ib[q];
    const bool codd = okb[q] && (cb & 1) != 0;
    const float nb = w6 * r0[i - R.sx] + w6 * r0[i + R.sx] + w6 * r0[i - R.sy] + w6 * r0[i + R.sy] +
                     w6 * r0[i + (codd ? 0 : -1)] + w6 * r0[i + (codd ? 1 : 0)];
    vb[q] = w1 * 0.0f + w6 * (nb + r1[i]);
  }
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    if (okr[q]) R.e[ir[q]] = vr[q];
    if (okb[q]) R.e[R.cs + ib[q]] = vb[q];
  }
}

// t = r - A e at every interior point, t in the one-array layout (k_resid_level).
// (one thread per row slot h, both colours of the slot: every load of a
// wavefront reads one contiguous run of a colour's array)
__global__ void k_resid_level_rb(float* __restrict__ t, Rb R, Lv L, const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int h = bx * blockDim.x + threadIdx.x;
  const int a = bz + 1;
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    if (b > L.n1) break;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int c = 2 * h + ((a + b + k) & 1);
      if (c < 1 || c > L.n2) continue;
      const RbPt pt = rb_pt(R, a, b, c);
      t[a * L.sx + b * L.sy + c] = R.r[pt.own + pt.i] - rb_ae<float>(R, pt);
    }
  }
}

// e += trilinear interpolation of the coarse correction (k_prolong).
__global__ void k_prolong_rb(Rb R, const float* __restrict__ ec, Lv C, const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int c = bx * blockDim.x + threadIdx.x + 1;
  const int a = bz + 1;
  if (c > R.n2) return;
  const int a0 = a >> 1, a1 = (a + 1) >> 1, c0 = c >> 1, c1 = (c + 1) >> 1;
  auto E = [&](int x, int y, int z) { return ec[x * C.sx + y * C.sy + z]; };
#pragma unroll
  for (int q = 0; q < kRows; ++q) {
    const int b = by * kRows + q + 1;
    if (b > R.n1) break;
    const int b0 = b >> 1, b1 = (b + 1) >> 1;
    const float v = (E(a0, b0, c0) + E(a1, b0, c0) + E(a0, b1, c0) + E(a1, b1, c0) + E(a0, b0, c1) + E(a1, b0, c1) +
                     E(a0, b1, c1) + E(a1, b1, c1)) *
                    0.125f;
    R.e[rb_at(R, a, b, c)] += v;
  }
}

// The colour-split analogue of for_interior_rows: each workgroup takes one
// contiguous range of rows and walks their slots h (both colours of a slot
// in one thread); f(g, a, b, c) gets every interior point once.
template <class F>
__device__ inline void for_interior_slots(const Rb& R, const int64_t sx, const int64_t sy, F&& f) {
  const int nrows = R.n0 * R.n1, nh = (R.n2 >> 1) + 1;
  const int per = (nrows + (int)gridDim.x - 1) / (int)gridDim.x;
  const int r0 = xcd_block(blockIdx.x, gridDim.x) * per;
  const int r1 = min(r0 + per, nrows);
  const int tpr = nh <= 64 ? 64 : (nh <= 128 ? 128 : 256);  // threads per row
  const int sub = threadIdx.x / tpr, lane = threadIdx.x % tpr;
  for (int row = r0 + sub; row < r1; row += 256 / tpr) {
    const int a = row / R.n1 + 1, b = row % R.n1 + 1;
    const int64_t base = a * sx + b * sy;
    for (int h = lane; h < nh; h += tpr) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int c = 2 * h + ((a + b + k) & 1);
        if (c >= 1 && c <= R.n2) f(base + c, a, b, c);
      }
    }
  }
}

// The level-0 passes of the defect correction with e and r stored by colour
// (k_resid0, k_update, k_pair_resid); phi, rho and the FP64 residual keep the
// glue layout. The two that read and write FP64 arrays walk the points in
// row order (a slot walk would touch those arrays with a stride of two);
// the residual pass between the cycles of a pair walks the slots.
__global__ __launch_bounds__(256) void k_resid0_rb(const double* __restrict__ phi, const double* __restrict__ rho,
                                                   double rc, Rb R, bool store, Lv L, double* part,
                                                   const int* __restrict__ done, double* __restrict__ r64) {
  if (*done) return;
  __shared__ double s1[256], s2[256];
  double rr = 0.0, bb = 0.0;
  for_interior_rows(L.n0, L.n1, L.n2, L.sx, L.sy, [&](const int64_t g, int a, int b, int c) {
    const double bv = rc * rho[g];
    const double ap = 6.0 * phi[g] - (phi[g - L.sx] + phi[g + L.sx] + phi[g - L.sy] + phi[g + L.sy] + phi[g - 1] +
                                      phi[g + 1]);
    const double rv = bv - ap;
    if (store) {
      const RbPt pt = rb_pt(R, a, b, c);
      R.r[pt.own + pt.i] = (float)rv;
      r64[g] = rv;
    }
    rr += rv * rv;
    bb += bv * bv;
  });
  s1[threadIdx.x] = rr;
  s2[threadIdx.x] = bb;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = s2[0];
  }
}

__global__ __launch_bounds__(256) void k_update_rb(double* __restrict__ phi, Rb R, double* r64, Lv L, double* part,
                                                   const int* __restrict__ done) {
  if (*done) return;
  __shared__ double s1[256];
  double rr = 0.0;
  const float* e = R.e;
  for_interior_rows(L.n0, L.n1, L.n2, L.sx, L.sy, [&](const int64_t g, int a, int b, int c) {
    const RbPt pt = rb_pt(R, a, b, c);
    const double eg = (double)e[pt.own + pt.i];
    const double ae = rb_ae<double>(R, pt);
    const double rv = r64[g] - ae;
    r64[g] = rv;
    R.r[pt.own + pt.i] = (float)rv;
    phi[g] += eg;
    rr += rv * rv;
  });
  s1[threadIdx.x] = rr;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s1[threadIdx.x] += s1[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = 0.0;
  }
}

__global__ __launch_bounds__(256) void k_pair_resid_rb(Rb R, Lv L, double* part, const int* __restrict__ done) {
  if (*done) return;
  __shared__ double s1[256];
  double rr = 0.0;
  const float* e = R.e;
  for_interior_slots(R, L.sx, L.sy, [&](const int64_t, int a, int b, int c) {
    const RbPt pt = rb_pt(R, a, b, c);
    const float t = R.r[pt.own + pt.i] - rb_ae<float>(R, pt);
    rr += (double)t * (double)t;
  });
  s1[threadIdx.x] = rr;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s1[threadIdx.x] += s1[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = 0.0;
  }
}

// ---- a level's smoothing with its transfer in one launch
//
// One V(2,2) visit of a level was about ten launches of 4-6 us (first sweep,
// half-sweeps, residual, restriction, prolongation), each reading the level
// again. Here a workgroup holds a tile of the level with a halo in LDS and does
// the whole downward half (two sweeps, residual, full weighting) or the whole
// upward half (interpolation, two sweeps) on it, recomputing the halo its
// neighbours also compute: every half-sweep narrows the valid region by one
// point. All sums are those of the separate kernels, in their order, so the
// result is the same bit for bit. The upward half reads its neighbours' points,
// so it writes to the level's second array; the downward half reads nothing
// but the right-hand side when it starts from zero.
//
// Halo points beyond the interior stay 0, as the levels' borders do. Tiles of
// 8^3 points: a launch is a chain of ten phases of latency, which more
// workgroups and fewer points each shorten. In a solve
// the visit of a 31^3 level went from ten launches, 38 us, to two, 13 us, of a
// 63^3 level from 40 to 19 us.
constexpr int kTileEdge = 8;

// q / D for 0 <= q <= MAXQ by one 24-bit product and a shift (the level
// kernels are bound by vector instructions, and the compiler's division by a
// constant takes a high product at a quarter of the rate).
template <int D, int MAXQ>
struct SmallDiv {
  static constexpr bool fits(int s) {
    const uint64_t m = ((1ull << s) + D - 1) / D;
    return m < (1u << 24) && MAXQ < (1 << 24) && (uint64_t)MAXQ * m < (1ull << 32) &&
           (uint64_t)MAXQ * (m * D - (1ull << s)) < (1ull << s);
  }
  static constexpr int shift() {
    int s = 4;
    while (s < 31 && !fits(s)) ++s;
    return s;
  }
  static constexpr int S = shift();
  static_assert(fits(S), "no exact multiplier");
  static constexpr uint32_t M = (uint32_t)(((1ull << S) + D - 1) / D);
  static __device__ inline int div(int q) { return (int)(__umul24((uint32_t)q, M) >> S); }
};

// (a, b, c) of point q of an NA x NB x NC box in row order.
template <int NA, int NB, int NC>
__device__ inline void box_point(int q, int& a, int& b, int& c) {
  const int ab = SmallDiv<NC, NA * NB * NC + 2048>::div(q);
  c = q - ab * NC;
  a = SmallDiv<NB, NA * NB + 2048 / NC + 1>::div(ab);
  b = ab - a * NB;
}

template <class P, bool ZERO>
struct DownDim {
  static constexpr int kLo = ZERO ? 4 : 5;               // halo below the tile's first point
  static constexpr int N = kTileEdge + 2 * kLo + 1;      // points per axis
  static constexpr int SB = N + (N & 1), SA = N * SB;    // row and plane length (SA even: the two colours' lanes
  static constexpr size_t kLds = 2 * (size_t)N * SA * sizeof(P);  // then read different banks)
  static_assert(SA % 2 == 0 && kLds <= 163840, "tile fits the LDS");
};
template <class P>
struct UpDim {
  static constexpr int kLo = 4, N = kTileEdge + 8, SB = N, SA = N * SB;
  static constexpr int NC = N / 2 + 1, SCB = NC, SCA = NC * NC;  // the coarse points they interpolate from
  static constexpr size_t kLds = (2 * (size_t)N * SA + (size_t)NC * SCA) * sizeof(P);
  static_assert(SA % 2 == 0 && kLds <= 163840, "tile fits the LDS");
};
constexpr int kTileThreads = 1024;

// The N^3 points of a tile with origin (oa, ob, oc) from a level array, 0
// outside the level's border; all of a thread's loads are in flight at once
// (a loop of one load and one LDS store an iteration spent the launch waiting:
// the data come from another XCD's writes, past this one's L2).
template <class P, int N, int SA, int SB, int NTHR>
struct TileLoad {
  static constexpr int IT = (N * N * N + NTHR - 1) / NTHR;
  P v[IT];
  __device__ inline void fetch(const P* __restrict__ src, const Lv& L, int oa, int ob, int oc) {
#pragma unroll
    for (int u = 0; u < IT; ++u) {
      const int q = threadIdx.x + u * NTHR;
      int a, b, c;
      box_point<N, N, N>(q, a, b, c);
      const int ga = oa + a, gb = ob + b, gc = oc + c;
      v[u] = 0;
      if ((unsigned)ga <= (unsigned)(L.n0 + 1) && (unsigned)gb <= (unsigned)(L.n1 + 1) &&
          (unsigned)gc <= (unsigned)(L.n2 + 1) && q < N * N * N)
        v[u] = src[ga * L.sx + gb * L.sy + gc];
    }
  }
  __device__ inline void put(P* dst) const {
#pragma unroll
    for (int u = 0; u < IT; ++u) {
      const int q = threadIdx.x + u * NTHR;
      int a, b, c;
      box_point<N, N, N>(q, a, b, c);
      if (q < N * N * N) dst[a * SA + b * SB + c] = v[u];
    }
  }
};

// Red-black half-sweep (k_smooth) of the tile's points at least M from its
// edge: a thread takes two points of the colour of one (b, c) column, their
// reads before either's store.
template <class P, int N, int SA, int SB, int M>
__device__ inline void tile_smooth(P* e, const P* r, const Lv& L, int oa, int ob, int oc, int color, P w1, P w6) {
  constexpr int W = N - 2 * M, PAIRS = (W + 3) / 4;
  for (int q = threadIdx.x; q < PAIRS * W * W; q += kTileThreads) {
    int s, b, c;
    box_point<PAIRS, W, W>(q, s, b, c);
    b += M;
    c += M;
    const int gb = ob + b, gc = oc + c;
    if (gb < 1 || gb > L.n1 || gc < 1 || gc > L.n2) continue;
    const int alo = max(M, 1 - oa), ahi = min(N - 1 - M, L.n0 - oa);
    const int a = alo + ((oa + alo + gb + gc + color) & 1) + 4 * s;  // (ga + gb + gc) % 2 == color
    if (a > ahi) continue;
    P* p = e + a * SA + b * SB + c;
    const P* rp = r + a * SA + b * SB + c;
    const bool two = a + 2 <= ahi;
    const int o = two ? 2 * SA : 0;  // (a lone point is read twice)
    const P mid = p[SA];
    const P n0 = p[-SA] + mid + p[-SB] + p[SB] + p[-1] + p[1];
    const P n1 = mid + p[o + SA] + p[o - SB] + p[o + SB] + p[o - 1] + p[o + 1];
    const P v0 = w1 * p[0] + w6 * (n0 + rp[0]);
    const P v1 = w1 * p[o] + w6 * (n1 + rp[o]);
    p[0] = v0;
    if (two) p[2 * SA] = v1;
  }
}

template <class P, bool ZERO>
__global__ __launch_bounds__(kTileThreads) void k_level_down(P* __restrict__ eo, const P* __restrict__ ei,
                                                                const P* __restrict__ r, Lv F, P* __restrict__ rc,
                                                                Lv C, P w1, P w6, const int* __restrict__ done) {
  if (*done) return;
  using D = DownDim<P, ZERO>;
  constexpr int N = D::N, SA = D::SA, SB = D::SB, T = kTileEdge, NT = kTileThreads, LO = D::kLo, M0 = ZERO ? 0 : 1;
  extern __shared__ __attribute__((aligned(16))) char tile_lds[];
  P* se = reinterpret_cast<P*>(tile_lds);
  P* sr = se + N * SA;
  int bx, by, bz;
  block3(bx, by, bz);
  const int s0 = bz * T + 1, s1 = by * T + 1, s2 = bx * T + 1;  // the tile's first point
  const int oa = s0 - LO, ob = s1 - LO, oc = s2 - LO;
  {
    TileLoad<P, N, SA, SB, NT> lr;
    lr.fetch(r, F, oa, ob, oc);
    if constexpr (!ZERO) {
      TileLoad<P, N, SA, SB, NT> le;
      le.fetch(ei, F, oa, ob, oc);
      le.put(se);
    }
    lr.put(sr);
  }
  __syncthreads();
  if constexpr (ZERO) {
    // red points of the first sweep from e = 0; black ones and the border 0
    for (int q = threadIdx.x; q < N * SA; q += NT) {
      int a, b, c;
      box_point<N, N, SB>(q, a, b, c);
      const bool red = ((oa + a + ob + b + oc + c) & 1) == 0;
      const bool in = c < N && oa + a >= 1 && oa + a <= F.n0 && ob + b >= 1 && ob + b <= F.n1 && oc + c >= 1 &&
                      oc + c <= F.n2;
      se[q] = red && in ? w6 * sr[q] : (P)0;
    }
  } else {
    tile_smooth<P, N, SA, SB, M0>(se, sr, F, oa, ob, oc, 0, w1, w6);
  }
  __syncthreads();
  tile_smooth<P, N, SA, SB, M0 + 1>(se, sr, F, oa, ob, oc, 1, w1, w6);
  __syncthreads();
  tile_smooth<P, N, SA, SB, M0 + 2>(se, sr, F, oa, ob, oc, 0, w1, w6);
  __syncthreads();
  tile_smooth<P, N, SA, SB, M0 + 3>(se, sr, F, oa, ob, oc, 1, w1, w6);
  __syncthreads();
  // the tile's points out; the residual (over r, in place) of the tile and one point above
  for (int q = threadIdx.x; q < (T + 1) * (T + 1) * (T + 1); q += NT) {
    int a, b, c;
    box_point<T + 1, T + 1, T + 1>(q, a, b, c);
    const int g = (a + LO) * SA + (b + LO) * SB + c + LO;
    const bool in = s0 + a <= F.n0 && s1 + b <= F.n1 && s2 + c <= F.n2;
    const P e = se[g];
    if (in) {
      sr[g] = sr[g] - ((P)6 * e - (se[g - SA] + se[g + SA] + se[g - SB] + se[g + SB] + se[g - 1] + se[g + 1]));
      if (a < T && b < T && c < T) eo[(s0 + a) * F.sx + (s1 + b) * F.sy + s2 + c] = e;
    }
  }
  __syncthreads();
  // full weighting (k_restrict_resid) at the coarse points inside the tile
  constexpr int TC = T / 2;
  for (int q = threadIdx.x; q < TC * TC * TC; q += NT) {
    const int a = q / (TC * TC), b = (q / TC) % TC, c = q % TC;
    const int A = s0 / 2 + 1 + a, B = s1 / 2 + 1 + b, Cc = s2 / 2 + 1 + c;  // fine 2A = s0 + 1 + 2a (s0 is odd)
    if (A > C.n0 || B > C.n1 || Cc > C.n2) continue;
    const int f = (2 * a + 1 + LO) * SA + (2 * b + 1 + LO) * SB + 2 * c + 1 + LO;
    P acc = 0;
#pragma unroll
    for (int da = -1; da <= 1; ++da)
#pragma unroll
      for (int db = -1; db <= 1; ++db)
#pragma unroll
        for (int dc = -1; dc <= 1; ++dc) acc += fw_weight<P>(da, db, dc) * sr[f + da * SA + db * SB + dc];
    rc[A * C.sx + B * C.sy + Cc] = acc * (P)0.5;  // (4/8) * sum
  }
}

template <class P>
__global__ __launch_bounds__(kTileThreads) void k_level_up(P* __restrict__ eo, const P* __restrict__ ei,
                                                              const P* __restrict__ r, Lv F,
                                                              const P* __restrict__ ec, Lv C, P w1, P w6,
                                                              const int* __restrict__ done) {
  if (*done) return;
  using D = UpDim<P>;
  constexpr int N = D::N, SA = D::SA, SB = D::SB, T = kTileEdge, NT = kTileThreads, LO = D::kLo;
  extern __shared__ __attribute__((aligned(16))) char tile_lds[];
  P* se = reinterpret_cast<P*>(tile_lds);
  P* sr = se + N * SA;
  P* sc = sr + N * SA;
  int bx, by, bz;
  block3(bx, by, bz);
  const int s0 = bz * T + 1, s1 = by * T + 1, s2 = bx * T + 1;
  const int oa = s0 - LO, ob = s1 - LO, oc = s2 - LO;
  const int ca = oa >> 1, cb = ob >> 1, cc = oc >> 1;  // the first coarse point (floor: oa may be negative)
  {
    TileLoad<P, D::NC, D::SCA, D::SCB, NT> lc;
    TileLoad<P, N, SA, SB, NT> le, lr;
    lc.fetch(ec, C, ca, cb, cc);
    le.fetch(ei, F, oa, ob, oc);
    lr.fetch(r, F, oa, ob, oc);
    lc.put(sc);
    le.put(se);
    lr.put(sr);
  }
  __syncthreads();
  // e += trilinear interpolation of the coarse correction (k_prolong)
  for (int q = threadIdx.x; q < N * N * N; q += NT) {
    int a, b, c;
    box_point<N, N, N>(q, a, b, c);
    const int ga = oa + a, gb = ob + b, gc = oc + c;
    if (ga < 1 || ga > F.n0 || gb < 1 || gb > F.n1 || gc < 1 || gc > F.n2) continue;
    const int a0 = ((ga >> 1) - ca) * D::SCA, a1 = (((ga + 1) >> 1) - ca) * D::SCA;
    const int b0 = ((gb >> 1) - cb) * D::SCB, b1 = (((gb + 1) >> 1) - cb) * D::SCB;
    const int c0 = (gc >> 1) - cc, c1 = ((gc + 1) >> 1) - cc;
    const P v = (sc[a0 + b0 + c0] + sc[a1 + b0 + c0] + sc[a0 + b1 + c0] + sc[a1 + b1 + c0] + sc[a0 + b0 + c1] +
                 sc[a1 + b0 + c1] + sc[a0 + b1 + c1] + sc[a1 + b1 + c1]) *
                (P)0.125;
    se[a * SA + b * SB + c] += v;
  }
  __syncthreads();
  tile_smooth<P, N, SA, SB, 1>(se, sr, F, oa, ob, oc, 0, w1, w6);
  __syncthreads();
  tile_smooth<P, N, SA, SB, 2>(se, sr, F, oa, ob, oc, 1, w1, w6);
  __syncthreads();
  tile_smooth<P, N, SA, SB, 3>(se, sr, F, oa, ob, oc, 0, w1, w6);
  __syncthreads();
  tile_smooth<P, N, SA, SB, 4>(se, sr, F, oa, ob, oc, 1, w1, w6);
  __syncthreads();
  for (int q = threadIdx.x; q < T * T * T; q += NT) {
    const int a = q / (T * T), b = (q / T) % T, c = q % T;
    if (s0 + a <= F.n0 && s1 + b <= F.n1 && s2 + c <= F.n2)
      eo[(s0 + a) * F.sx + (s1 + b) * F.sy + s2 + c] = se[(a + LO) * SA + (b + LO) * SB + c + LO];
  }
}

template <class P>
__global__ void k_zero_level(P* __restrict__ e, Lv L, const int* __restrict__ done) {
  if (*done) return;
  int bx, by, bz;
  block3(bx, by, bz);
  const int c = bx * blockDim.x + threadIdx.x + 1;
  const int b = by + 1, a = bz + 1;
  if (c > L.n2) return;
  e[a * L.sx + b * L.sy + c] = (P)0;
}

// One unknown: A = 6.
template <class P>
__global__ void k_coarse_single(P* e, const P* r, Lv L, const int* __restrict__ done) {
  if (*done) return;
  const int64_t g = L.sx + L.sy + 1;
  e[g] = r[g] / (P)6;
}

// ---- coarse tail: the V-cycle below level Lc in one workgroup, arrays in LDS
//
// A phase (half-sweep, residual, transfer) of these levels is a few hundred to
// a few thousand points between two barriers, so its time is the latency of
// one point's LDS reads and of finding the point. The points of each level are
// listed once per context (array index by colour, index of a coarse point's
// fine node, packed interpolation corner), and the lists go to LDS with the
// right-hand side: a phase then takes one list entry instead of two integer
// divisions. 15^3 -> 1: 17.1 -> 15.2 us, bound by LDS reads on the 15^3 level
// (half of it) and latency below; 11 x 9 x 13 -> 5 x 4 x 6 (32 sweeps there):
// 18.3 us, where with 23 x 19 x 27 on top, walked by columns, it was 47 us.

constexpr int kTailMaxLevels = 8;
constexpr int kTailThreads = 1024;
constexpr int kTailWave = 343;  // 7^3

struct TailLv {
  int sx, sy;       // strides of the padded (n+2)^3 array
  int oe, orr, ot;  // element offsets of e, r, t in LDS
  int count, red;   // points, of which colour 0
  int list;         // offsets in the table: array index of each point (colour 0 first),
  int fine;         // the same points' index in the next finer level,
  int corner;       // and the coarse corner they interpolate from (13 bits) with the steps to the next (3 bits)
};

template <class P>
struct TailArgs {
  int nl;
  TailLv lv[kTailMaxLevels];
  P* ge;                // level-Lc e in global memory
  const P* gr;          // level-Lc r in global memory
  const int32_t* gidx;  // its points' index there, in list order
  const uint16_t* tab;
  int ntab;             // table entries (a multiple of 8), staged behind the arrays
  P w1, w6;
  int pre, post, coarse_sweeps;
  int total;            // LDS elements of the arrays
  const int* done;
};

// Orders a wavefront's LDS accesses in the program's order (they execute in
// order; this keeps the compiler from moving them), or the workgroup's.
template <bool BLOCK>
__device__ inline void tail_sync() {
  if constexpr (BLOCK) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

template <class P>
__device__ inline P tail_new(const P* e, const P* r, const TailLv& L, int g, P w1, P w6) {
  const P nb = e[g - L.sx] + e[g + L.sx] + e[g - L.sy] + e[g + L.sy] + e[g - 1] + e[g + 1];
  return w1 * e[g] + w6 * (nb + r[g]);
}

// Sweeps over a level by NT threads; up to U points of each colour per thread
// keep their index over the sweeps, and are read together (a half-sweep reads
// only the other colour and itself).
template <class P, int NT, int U>
__device__ inline void tail_smooth(P* s, const uint16_t* tab, const TailLv L, int sweeps, P w1, P w6) {
  constexpr bool BLOCK = NT == kTailThreads;
  P* e = s + L.oe;
  const P* r = s + L.orr;
  int g[2][U], n[2] = {L.red, L.count - L.red};
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = (int)threadIdx.x + u * NT;
      g[k][u] = tab[L.list + (k ? L.red : 0) + (q < n[k] ? q : 0)];
    }
  for (int it = 0; it < sweeps; ++it)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      P v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = tail_new<P>(e, r, L, g[k][u], w1, w6);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if ((int)threadIdx.x + u * NT < n[k]) e[g[k][u]] = v[u];
      for (int q = threadIdx.x + U * NT; q < n[k]; q += NT) {  // (a large coarsest level)
        const int gq = tab[L.list + (k ? L.red : 0) + q];
        e[gq] = tail_new<P>(e, r, L, gq, w1, w6);
      }
      tail_sync<BLOCK>();
    }
}

// Levels [l0, nl) by NT threads: pre-smoothing, residual and restriction down,
// the coarsest level, interpolation and post-smoothing up.
template <class P, int NT, int U>
__device__ inline void tail_down(P* s, const uint16_t* tab, const TailArgs<P>& A, const TailLv F, const TailLv C) {
  constexpr bool BLOCK = NT == kTailThreads;
  tail_smooth<P, NT, U>(s, tab, F, A.pre, A.w1, A.w6);
  const P* e = s + F.oe;
  for (int q = threadIdx.x; q < F.count; q += NT) {
    const int g = tab[F.list + q];
    s[F.ot + g] = s[F.orr + g] - ((P)6 * e[g] - (e[g - F.sx] + e[g + F.sx] + e[g - F.sy] + e[g + F.sy] + e[g - 1] +
                                                 e[g + 1]));
  }
  tail_sync<BLOCK>();
  for (int q = threadIdx.x; q < C.count; q += NT) {
    const int f = F.ot + tab[C.fine + q];
    P acc = 0;
#pragma unroll
    for (int da = -1; da <= 1; ++da)
#pragma unroll
      for (int db = -1; db <= 1; ++db)
#pragma unroll
        for (int dc = -1; dc <= 1; ++dc) acc += fw_weight<P>(da, db, dc) * s[f + da * F.sx + db * F.sy + dc];
    s[C.orr + tab[C.list + q]] = acc * (P)0.5;
  }
  tail_sync<BLOCK>();
}

template <class P, int NT, int U>
__device__ inline void tail_bottom(P* s, const uint16_t* tab, const TailArgs<P>& A, const TailLv L) {
  if (L.count == 1) {
    if (threadIdx.x == 0) {
      const int g = tab[L.list];
      s[L.oe + g] = s[L.orr + g] / (P)6;
    }
    tail_sync<NT == kTailThreads>();
  } else {
    tail_smooth<P, NT, U>(s, tab, L, A.coarse_sweeps, (P)0, (P)1 / (P)6);
  }
}

template <class P, int NT, int U>
__device__ inline void tail_up(P* s, const uint16_t* tab, const TailArgs<P>& A, const TailLv F, const TailLv C) {
  const P* ec = s + C.oe;
  for (int q = threadIdx.x; q < F.count; q += NT) {
    const int w = tab[F.corner + q];
    const P* p = ec + (w & 0x1fff);
    const int da = (w >> 13) & 1 ? C.sx : 0, db = (w >> 14) & 1 ? C.sy : 0, dc = w >> 15;
    const P v = (p[0] + p[da] + p[db] + p[da + db] + p[dc] + p[da + dc] + p[db + dc] + p[da + db + dc]) * (P)0.125;
    s[F.oe + tab[F.list + q]] += v;
  }
  tail_sync<NT == kTailThreads>();
  tail_smooth<P, NT, U>(s, tab, F, A.post, A.w1, A.w6);
}

// The levels of the cubic chain 15 -> 7 -> 3 -> 1 (every cubic grid of 2^k + 1
// nodes per axis ends in it), as plan_tail lays them out: with the strides known at
// compile time a point's neighbours are immediates of one address.
constexpr int tail_plane(int n1, int n2) { return ((n1 + 2) * (n2 + 2) + 1) & ~1; }
constexpr TailLv cube15_lv(int q) {
  int n = 15, off = 0, at = 0;
  TailLv L{};
  for (int k = 0;; ++k) {
    const int sx = tail_plane(n, n), size = (n + 2) * sx, pts = n * n * n;
    L = TailLv{sx, n + 2, off, off + size, off + 2 * size, pts, pts / 2, at, k ? at + pts : 0, 0};
    at += k ? 2 * pts : pts;
    if (k < 3) {
      L.corner = at;
      at += pts;
    }
    if (k == q) return L;
    off += 3 * size;
    n = (n - 1) / 2;
  }
}

template <class P, bool CUBE15>
__device__ inline TailLv tail_lv(const TailArgs<P>& A, int q) {
  if constexpr (CUBE15) return q == 0 ? cube15_lv(0) : (q == 1 ? cube15_lv(1) : (q == 2 ? cube15_lv(2) : cube15_lv(3)));
  return A.lv[q];
}

template <class P, bool CUBE15>
__global__ __launch_bounds__(kTailThreads) void k_coarse_tail(TailArgs<P> A) {
  if (*A.done) return;
  extern __shared__ __attribute__((aligned(16))) char tail_lds[];
  P* s = reinterpret_cast<P*>(tail_lds);
  uint16_t* tab = reinterpret_cast<uint16_t*>(s + A.total);
  const TailLv L0 = tail_lv<P, CUBE15>(A, 0);
  {
    constexpr int U = 4;  // right-hand side points in flight while the arrays are cleared
    P v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = threadIdx.x + u * kTailThreads;
      v[u] = q < L0.count ? A.gr[A.gidx[q]] : (P)0;
    }
    for (int q = threadIdx.x; q < A.ntab / 8; q += kTailThreads)
      reinterpret_cast<uint4*>(tab)[q] = reinterpret_cast<const uint4*>(A.tab)[q];
    for (int q = threadIdx.x; q < A.total * (int)sizeof(P) / 16; q += kTailThreads)
      reinterpret_cast<uint4*>(s)[q] = make_uint4(0, 0, 0, 0);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = threadIdx.x + u * kTailThreads;
      if (q < L0.count) s[L0.orr + tab[L0.list + q]] = v[u];
    }
    for (int q = threadIdx.x + U * kTailThreads; q < L0.count; q += kTailThreads)
      s[L0.orr + tab[L0.list + q]] = A.gr[A.gidx[q]];
    __syncthreads();
  }
  // levels of at most kTailWave points go to the first wavefront alone, which
  // needs no barriers between its phases
  auto lv = [&](int q) { return tail_lv<P, CUBE15>(A, q); };
  if constexpr (CUBE15) {
    tail_down<P, kTailThreads, 2>(s, tab, A, lv(0), lv(1));
    if (threadIdx.x < 64) {
      tail_down<P, 64, 3>(s, tab, A, lv(1), lv(2));
      tail_down<P, 64, 1>(s, tab, A, lv(2), lv(3));
      tail_bottom<P, 64, 1>(s, tab, A, lv(3));
      tail_up<P, 64, 1>(s, tab, A, lv(2), lv(3));
      tail_up<P, 64, 3>(s, tab, A, lv(1), lv(2));
    }
    __syncthreads();
    tail_up<P, kTailThreads, 2>(s, tab, A, lv(0), lv(1));
  } else {
    int ls = 0;
    while (ls < A.nl && A.lv[ls].count > kTailWave) ++ls;
    const int top = min(ls, A.nl - 1);  // levels the workgroup descends from
    for (int l = 0; l < top; ++l) tail_down<P, kTailThreads, 2>(s, tab, A, lv(l), lv(l + 1));
    if (ls < A.nl) {
      if (threadIdx.x < 64) {
        for (int l = ls; l + 1 < A.nl; ++l) tail_down<P, 64, 3>(s, tab, A, lv(l), lv(l + 1));
        tail_bottom<P, 64, 3>(s, tab, A, lv(A.nl - 1));
        for (int l = A.nl - 2; l >= ls; --l) tail_up<P, 64, 3>(s, tab, A, lv(l), lv(l + 1));
      }
      __syncthreads();
    } else {
      tail_bottom<P, kTailThreads, 2>(s, tab, A, lv(A.nl - 1));
    }
    for (int l = top - 1; l >= 0; --l) tail_up<P, kTailThreads, 2>(s, tab, A, lv(l), lv(l + 1));
  }
  for (int q = threadIdx.x; q < L0.count; q += kTailThreads) A.ge[A.gidx[q]] = s[L0.oe + tab[L0.list + q]];
}

// Face conditions on phi (Field.cpp:10-96): D -> 0, N -> copy the neighbour,
// in the reference's order (x low and up, y, z), where a later face takes what
// an earlier one left on a shared edge. A thread finds its
// node's final value instead: from the last face down, D gives 0 and N steps
// inwards, to a node that no face writes. So the six (blockIdx.z) take one
// launch, not six in order. unconfirmed: nothing is done while the solve goes on.
struct FaceKinds {
  char k[6];
};
__global__ void k_faces(double* phi, int cx, int cy, int cz, FaceKinds bc, const int* unconfirmed) {
  if (*unconfirmed) return;
  const int f = blockIdx.z, axis = f >> 1;
  const int n[3] = {cx, cy, cz};
  const int ua = axis == 2 ? 1 : 2, va = axis == 0 ? 1 : 0;
  const int u = blockIdx.x * blockDim.x + threadIdx.x, v = blockIdx.y;
  if (u >= n[ua] - 2 || v >= n[va] - 2) return;
  int at[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) at[q] = q == axis ? ((f & 1) ? n[q] - 2 : 1) : (q == ua ? u + 1 : v + 1);
  const int64_t t = ((int64_t)at[0] * cy + at[1]) * cz + at[2];
  bool zero = false;
#pragma unroll
  for (int q = 2; q >= 0; --q) {
    const bool low = at[q] == 1;
    if (!low && at[q] != n[q] - 2) continue;
    zero = zero || bc.k[2 * q + (low ? 0 : 1)] != 'N';
    if (!zero) at[q] += low ? 1 : -1;
  }
  phi[t] = zero ? 0.0 : phi[((int64_t)at[0] * cy + at[1]) * cz + at[2]];
}

Lv lv_of(const MgLevel& m) { return Lv{m.n[0], m.n[1], m.n[2], m.sx, m.sy}; }

template <class P>
P* E_(MgLevel& m);
template <>
double* E_<double>(MgLevel& m) {
  return m.e64.p + m.off;
}
template <>
float* E_<float>(MgLevel& m) {
  return m.e32.p + m.off;
}
template <class P>
P* R_(MgLevel& m);
template <>
double* R_<double>(MgLevel& m) {
  return m.r64.p + m.off;
}
template <>
float* R_<float>(MgLevel& m) {
  return m.r32.p + m.off;
}
template <class P>
P* T_(MgLevel& m);
template <>
double* T_<double>(MgLevel& m) {
  return m.t64.p + m.off;
}
template <>
float* T_<float>(MgLevel& m) {
  return m.t32.p + m.off;
}

dim3 grid_full(const MgLevel& m) { return dim3(div_up(m.n[2], 64), m.n[1], m.n[0]); }
// kRows rows per thread
dim3 grid_full4(const MgLevel& m) { return dim3(div_up(m.n[2], 64), div_up(m.n[1], kRows), m.n[0]); }
dim3 grid_half4(const MgLevel& m) { return dim3(div_up((m.n[2] + 1) / 2, 64), div_up(m.n[1], kRows), m.n[0]); }

constexpr int kResidBlocks = 2048;  // workgroups of the level-0 residual and update passes

// Levels with at least this many unknowns form their residual in a pass of
// its own before restricting it (below, one launch forming it on the fly costs less).
constexpr int64_t kSplitRestrict = (int64_t)1 << 20;

int coarse_sweeps(const MgLevel& m) { return 4 * std::max({m.n[0], m.n[1], m.n[2]}) + 8; }

// First level handled by the LDS tail kernel, its LDS bytes for element size
// `esz`, and its point lists on the device. Every level keeps e and r, all but
// the coarsest t, as padded (n+2)^3 arrays.
void plan_tail(Ctx& c, size_t esz) {
  const int nl = (int)c.mg.size();
  c.mg_tail = nl;  // none
  c.mg_tail_bytes = 0;
  // plane length (even, see the lists' order below) and elements of a level's array
  auto plane = [&](int l) { return tail_plane(c.mg[l].n[1], c.mg[l].n[2]); };
  auto padded = [&](int l) { return (size_t)(c.mg[l].n[0] + 2) * plane(l); };
  size_t arrays = 0, entries = 0;
  for (int l = nl - 1; l >= 0 && nl - l <= kTailMaxLevels; --l) {
    const MgLevel& m = c.mg[l];
    const size_t pts = (size_t)m.n[0] * m.n[1] * m.n[2];
    const bool last = l == nl - 1;
    // (indices are 16 bits, a coarse corner's 13)
    if (padded(l) > 65535 || (!last && padded(l + 1) > 8192)) break;
    arrays += (last ? 2 : 3) * padded(l);
    entries += (last ? 2 : 3) * pts;  // (a first level without a finer one leaves its second list unused)
    const size_t bytes = (arrays * esz + 15) / 16 * 16 + (entries + 8) * sizeof(uint16_t);
    if (bytes > c.lds_max) break;
    // A level the level kernels can take leaves the tail above 15^3 points: one
    // workgroup's phases then last longer than two launches (23 x 19 x 27: 29
    // us here, 13 us there).
    if (c.mg_fused && !last && pts > 3375) break;
    c.mg_tail = l;
    c.mg_tail_bytes = bytes;
  }
  c.mg_tail_plan.clear();
  if (c.mg_tail == nl) return;
  std::vector<uint16_t> tab;
  std::vector<int32_t> gidx;
  int off = 0;
  for (int l = c.mg_tail; l < nl; ++l) {
    const MgLevel& m = c.mg[l];
    const int sy = m.n[2] + 2, sx = plane(l);
    std::vector<uint16_t> list[2], fine[2], corner[2];
    std::vector<int32_t> gi[2];
    const bool first = l == c.mg_tail, last = l == nl - 1;
    const int fy = first ? 0 : c.mg[l - 1].n[2] + 2, fx = first ? 0 : plane(l - 1);
    const int cy = last ? 0 : c.mg[l + 1].n[2] + 2, cx = last ? 0 : plane(l + 1);
    // Each colour's points go along c through two planes at once, so that
    // neighbouring lanes read neighbouring banks: along one plane a colour's
    // points are two elements apart, and every read took two turns (15^3: a
    // half-sweep about 1850 cycles, 1100 so). The planes lie an even distance apart.
    for (int k = 0; k < 2; ++k)
      for (int ap = 1; ap <= m.n[0]; ap += 2)
        for (int b = 1; b <= m.n[1]; ++b)
          for (int q = 1; q <= m.n[2]; ++q) {
            const int a = ap + ((ap + b + q + k) & 1);
            if (a > m.n[0]) continue;
            list[k].push_back((uint16_t)(a * sx + b * sy + q));
            fine[k].push_back((uint16_t)(2 * a * fx + 2 * b * fy + 2 * q));
            corner[k].push_back((uint16_t)(((a >> 1) * cx + (b >> 1) * cy + (q >> 1)) | (a & 1) << 13 | (b & 1) << 14 |
                                           (q & 1) << 15));
            gi[k].push_back((int32_t)(a * m.sx + b * m.sy + q));
          }
    auto add = [&](std::vector<uint16_t>(&v)[2]) {
      const int at = (int)tab.size();
      for (auto& x : v) tab.insert(tab.end(), x.begin(), x.end());
      return at;
    };
    TailPlan t{};
    t.sx = sx;
    t.sy = sy;
    t.oe = off;
    t.orr = off + (int)padded(l);
    t.ot = off + 2 * (int)padded(l);
    off += (last ? 2 : 3) * (int)padded(l);
    t.red = (int)list[0].size();
    t.count = t.red + (int)list[1].size();
    t.list = add(list);
    if (!first) t.fine = add(fine);
    if (!last) t.corner = add(corner);
    if (first)
      for (auto& x : gi) gidx.insert(gidx.end(), x.begin(), x.end());
    c.mg_tail_plan.push_back(t);
  }
  c.mg_tail15 = c.mg_tail_plan.size() == 4;
  for (size_t q = 0; q < c.mg_tail_plan.size() && c.mg_tail15; ++q) {
    const TailPlan& t = c.mg_tail_plan[q];
    const TailLv L = cube15_lv((int)q);
    const MgLevel& m = c.mg[c.mg_tail + q];
    c.mg_tail15 = m.n[0] == m.n[1] && m.n[1] == m.n[2] && t.sx == L.sx && t.sy == L.sy && t.oe == L.oe &&
                  t.orr == L.orr && (q == 3 || t.ot == L.ot) && t.count == L.count && t.red == L.red &&
                  t.list == L.list && (q == 0 || t.fine == L.fine) && (q == 3 || t.corner == L.corner);
  }
  c.mg_tail_elems = (int)(((size_t)off * esz + 15) / 16 * 16 / esz);
  while (tab.size() % 8) tab.push_back(0);
  c.mg_tail_ntab = tab.size();
  tab.resize(tab.size() + 2 * gidx.size());
  std::memcpy(tab.data() + c.mg_tail_ntab, gidx.data(), gidx.size() * sizeof(int32_t));
  c.mg_tail_tab.alloc(tab.size());
  FOPIS_HIP(hipMemcpy(c.mg_tail_tab.p, tab.data(), tab.size() * sizeof(uint16_t), hipMemcpyHostToDevice));
}

template <class P>
TailArgs<P> tail_args(Ctx& c, const int* done) {
  TailArgs<P> A{};
  A.nl = (int)c.mg_tail_plan.size();
  for (int q = 0; q < A.nl; ++q) {
    const TailPlan& t = c.mg_tail_plan[q];
    A.lv[q] = TailLv{t.sx, t.sy, t.oe, t.orr, t.ot, t.count, t.red, t.list, t.fine, t.corner};
  }
  MgLevel& m0 = c.mg[c.mg_tail];
  A.ge = E_<P>(m0);
  A.gr = R_<P>(m0);
  A.gidx = reinterpret_cast<const int32_t*>(c.mg_tail_tab.p + c.mg_tail_ntab);
  A.tab = c.mg_tail_tab.p;
  A.ntab = (int)c.mg_tail_ntab;
  A.w1 = (P)(1.0 - c.d.mg_omega);
  A.w6 = (P)(c.d.mg_omega / 6.0);
  A.pre = c.d.mg_pre;
  A.post = c.d.mg_post;
  A.coarse_sweeps = coarse_sweeps(c.mg.back());
  A.total = c.mg_tail_elems;
  A.done = done;
  return A;
}

Rb rb_of(Ctx& c) {
  const MgLevel& m = c.mg[0];
  return Rb{c.erb.p, c.rrb.p, c.rb_cs, c.rb_sx, c.rb_sy, m.n[0], m.n[1], m.n[2]};
}

// the colour-split finest level, kRows rows per thread: the row slots h that
// hold interior points (0 .. n2 / 2) for the first sweep, which takes both
// colours of a slot; a half-sweep takes one colour's points (grid_half4)
dim3 grid_rb(const Ctx& c) {
  const MgLevel& m = c.mg[0];
  return dim3(div_up((m.n[2] >> 1) + 1, 64), div_up(m.n[1], kRows), m.n[0]);
}

template <class P>
void smooth(Ctx& c, MgLevel& m, int sweeps, double w, bool from_zero, const int* done) {
  const P w1 = (P)(1.0 - w), w6 = (P)(w / 6.0);
  if constexpr (std::is_same<P, float>::value) {
    if (c.mg_rb && &m == &c.mg[0]) {
      const Rb R = rb_of(c);
      for (int s = 0; s < sweeps; ++s) {
        if (from_zero && s == 0) {
          k_smooth_first2_rb<<<grid_rb(c), 64, 0, c.stream>>>(R, w1, w6, done);
          continue;
        }
        for (int col = 0; col < 2; ++col) k_smooth_rb<<<grid_half4(m), 64, 0, c.stream>>>(R, col, w1, w6, done);
      }
      return;
    }
  }
  for (int s = 0; s < sweeps; ++s) {
    if (from_zero && s == 0) {
      k_smooth_first2<P><<<grid_half4(m), 64, 0, c.stream>>>(E_<P>(m), R_<P>(m), lv_of(m), w1, w6, done);
      continue;
    }
    for (int col = 0; col < 2; ++col)
      k_smooth<P><<<grid_half4(m), 64, 0, c.stream>>>(E_<P>(m), R_<P>(m), lv_of(m), col, w1, w6, done);
  }
}

dim3 grid_tiles(const MgLevel& m) {
  return dim3(div_up(m.n[2], kTileEdge), div_up(m.n[1], kTileEdge), div_up(m.n[0], kTileEdge));
}

// The level kernels take levels of up to 2^19 unknowns, 1024 tiles, two rounds
// of the chip: beyond, the halo they load and sweep again costs more than the
// launches they save (per point of an 8^3 tile: k_level_down loads 9.6 of r from
// zero and 13.4 of e and r when it continues, k_level_up 8 of e and r; the first
// half-sweeps cover 9.6 and 5.4. 63^3: 19 us in two launches, 40 us in ten; 95 x
// 79 x 111: 59 and 43 us).
constexpr int64_t kLevelMost = (int64_t)1 << 19;
bool level_fused(const Ctx& c, const MgLevel& m) {
  return c.mg_fused && (int64_t)m.n[0] * m.n[1] * m.n[2] <= kLevelMost;
}

// One V-cycle from level l down; returns the array that holds the level's
// correction. from: the correction the finest level's cycle continues from (a
// second cycle on the same right-hand side), null to start from e = 0 (always
// so below the finest level).
template <class P>
P* vcycle(Ctx& c, int l, const int* done, const P* from = nullptr) {
  MgLevel& m = c.mg[l];
  const bool zero = from == nullptr;
  const double w = c.d.mg_omega;
  if (l == c.mg_tail) {
    if (c.mg_tail15)
      k_coarse_tail<P, true><<<1, kTailThreads, c.mg_tail_bytes, c.stream>>>(tail_args<P>(c, done));
    else
      k_coarse_tail<P, false><<<1, kTailThreads, c.mg_tail_bytes, c.stream>>>(tail_args<P>(c, done));
    return E_<P>(m);
  }
  if (l == (int)c.mg.size() - 1) {
    // coarsest level outside the tail kernel: Gauss-Seidel sweeps from zero
    if (m.n[0] == 1 && m.n[1] == 1 && m.n[2] == 1) {
      k_coarse_single<P><<<1, 1, 0, c.stream>>>(E_<P>(m), R_<P>(m), lv_of(m), done);
    } else {
      smooth<P>(c, m, coarse_sweeps(m), 1.0, true, done);
    }
    return E_<P>(m);
  }
  MgLevel& mc = c.mg[l + 1];
  bool rb = false;
  if constexpr (std::is_same<P, float>::value) rb = c.mg_rb && l == 0;
  if (level_fused(c, m)) {
    const P w1 = (P)(1.0 - w), w6 = (P)(w / 6.0);
    if (from)
      k_level_down<P, false><<<grid_tiles(m), kTileThreads, DownDim<P, false>::kLds, c.stream>>>(
          E_<P>(m), from, R_<P>(m), lv_of(m), R_<P>(mc), lv_of(mc), w1, w6, done);
    else
      k_level_down<P, true><<<grid_tiles(m), kTileThreads, DownDim<P, true>::kLds, c.stream>>>(
          E_<P>(m), nullptr, R_<P>(m), lv_of(m), R_<P>(mc), lv_of(mc), w1, w6, done);
    const P* ec = vcycle<P>(c, l + 1, done);
    k_level_up<P><<<grid_tiles(m), kTileThreads, UpDim<P>::kLds, c.stream>>>(T_<P>(m), E_<P>(m), R_<P>(m), lv_of(m), ec,
                                                                           lv_of(mc), w1, w6, done);
    return T_<P>(m);
  }
  // every level starts its cycle from e = 0 (the correction equation)
  if (zero && c.d.mg_pre == 0) k_zero_level<P><<<grid_full(m), 64, 0, c.stream>>>(E_<P>(m), lv_of(m), done);
  smooth<P>(c, m, c.d.mg_pre, w, zero, done);
  if (rb) {
    if constexpr (std::is_same<P, float>::value) {
      k_resid_level_rb<<<grid_rb(c), 64, 0, c.stream>>>(T_<P>(m), rb_of(c), lv_of(m), done);
      k_restrict_t<P><<<grid_full(mc), 64, 0, c.stream>>>(R_<P>(mc), lv_of(mc), T_<P>(m), lv_of(m), done);
    }
  } else if ((int64_t)m.n[0] * m.n[1] * m.n[2] >= kSplitRestrict) {
    k_resid_level<P><<<grid_full4(m), 64, 0, c.stream>>>(T_<P>(m), E_<P>(m), R_<P>(m), lv_of(m), done);
    k_restrict_t<P><<<grid_full(mc), 64, 0, c.stream>>>(R_<P>(mc), lv_of(mc), T_<P>(m), lv_of(m), done);
  } else {
    k_restrict_resid<P><<<grid_full(mc), 64, 0, c.stream>>>(R_<P>(mc), lv_of(mc), E_<P>(m), R_<P>(m), lv_of(m),
                                                            done);
  }
  const P* ec = vcycle<P>(c, l + 1, done);
  if (rb) {
    if constexpr (std::is_same<P, float>::value)
      k_prolong_rb<<<grid_full4(m), 64, 0, c.stream>>>(rb_of(c), ec, lv_of(mc), done);
  } else {
    k_prolong<P><<<grid_full4(m), 64, 0, c.stream>>>(E_<P>(m), lv_of(m), ec, lv_of(mc), done);
  }
  smooth<P>(c, m, c.d.mg_post, w, false, done);
  return E_<P>(m);
}

// A whole solve of some number of expected cycles is captured once that number
// has been expected kWholeAfter times, if its graph has at most kWholeNodes
// nodes. The chip then does not idle between the graphs of single cycles and
// pairs: a solve takes 157 us instead of 178 at 17^3, 230 for 240 at 33^3, 669
// for 681 at 129^3. Capturing takes 130 us at 17^3, 180 at 33^3, 300 at 129^3, so
// it pays after 7 to 30 solves (0.55 ms at 257^3, after 45). At 101^3, where the coarsest level stays outside
// the tail and a cycle has over 200 nodes, the one graph is slower, 4.02 ms for
// 3.87.
constexpr int kWholeAfter = 16, kWholeMost = 32;
constexpr size_t kWholeNodes = 600;

void drop_whole(Ctx& c) {
  for (auto& w : c.mg_whole)
    if (w.exec) (void)hipGraphExecDestroy(w.exec);
  c.mg_whole.assign(kWholeMost + 1, Ctx::Whole());
}

template <class P>
int solve_impl(Ctx& c, double tol, int max_cycles, double* relres_out, const double* rho0) {
  MgLevel& m0 = c.mg[0];
  const Lv L0 = lv_of(m0);
  // level-0 arrays share the glue layout; the MG origin is glue node (1,1,1)
  const int64_t off = m0.off;
  double* phi = c.phi.p + off;
  const double* rho = rho0 + off;
  P* r0 = R_<P>(m0);
  const double rc = 1.0 / c.d.eps0;  // pow(dx, 2) / eps0 with dx = 1
  const int nb = kResidBlocks;  // workgroups of the level-0 residual passes (8 per CU)
  double* part = c.mg_part.p;
  double* dst = c.mg_part.p + 2 * nb;
  int* st = c.mg_state.p;
  const int* done = st;
  // level-0 FP64 residual kept by the cycle updates (the level's own array when P is double)
  double* r64 = std::is_same<P, double>::value ? reinterpret_cast<double*>(r0) : c.mg_r64.p + off;
  const int* never = st + 3;  // stays 0: the final residual always runs
  // the level-0 passes, on the colour-split arrays when the level has them
  bool rb = false;
  if constexpr (std::is_same<P, float>::value) rb = c.mg_rb;
  auto resid0 = [&](bool store, const int* flag) {
    if constexpr (std::is_same<P, float>::value) {
      if (rb) {
        k_resid0_rb<<<nb, 256, 0, c.stream>>>(phi, rho, rc, rb_of(c), store, L0, part, flag, store ? r64 : nullptr);
        return;
      }
    }
    k_resid0<P><<<nb, 256, 0, c.stream>>>(phi, rho, rc, store ? r0 : (P*)nullptr, L0, part, flag,
                                          store ? r64 : (double*)nullptr);
  };
  auto begin = [&] {
    resid0(true, never);
    k_norm<true><<<1, 256, 0, c.stream>>>(part, nb, dst, st, tol, max_cycles, 0, nullptr);
  };
  // Queue as many cycles as the previous two solves needed, then more. With
  // pairs, two V-cycles share one FP64 update and norm check: the second
  // runs on the same right-hand side, continuing from the first's correction
  // (the residual it restricts is then r - A e, formed in P, whose rounding
  // stays far below the ~30x a V-cycle removes). Between the two, one read of
  // e and r gives the residual the first cycle left (k_pair_resid); when that
  // already meets the tolerance the second cycle's kernels all return at
  // once, so a solve applies exactly the cycles it needs, as with single
  // cycles. A pair saves the FP64 update (reads and writes phi and r in FP64)
  // and a norm check for the price of that one read.
  const int pred = std::max(1, std::min(c.mg_hist[0], c.mg_hist[1]));
  // (a finest level inside the single-workgroup tail, or the coarsest level
  // itself, always solves from zero: no pairs there)
  const bool pairs = c.mg_pairs && c.mg_tail > 0 && (int)c.mg.size() > 1;
  int npair = pairs ? pred / 2 : 0;
  int batch = pred - 2 * npair;
  static_assert(kSolveWords + sizeof(SolveWords) <= kWords, "the context's pinned words hold a solve's");
  SolveWords* const words = reinterpret_cast<SolveWords*>(static_cast<char*>(c.host_words.p) + kSolveWords);
  FaceKinds faces;
  for (int f = 0; f < 6; ++f) faces.k[f] = c.d.boundary[f];
  // (u runs along z, or y on the z faces; v along y or x)
  const dim3 face_grid(div_up(std::max(c.cy, c.cz) - 2, 64), std::max(c.cx, c.cy) - 2, 6);
  int* skip = st + 4;
  // One cycle (or pair): the V-cycle(s), the FP64 update and the norm
  // check. Their ~15 (~30) launches are captured once into a graph of kernel
  // nodes (every pointer and size in them is fixed for the context; the
  // tolerance and the cycle cap are arguments of the norm kernel, so the
  // graphs are rebuilt when they change) and replayed. A number of cycles that
  // is expected often gets a graph of the whole solve.
  auto cycle = [&](int nv) {
    const P* e = vcycle<P>(c, 0, done);
    if (nv == 2) {
      if constexpr (std::is_same<P, float>::value) {
        if (rb)
          k_pair_resid_rb<<<nb, 256, 0, c.stream>>>(rb_of(c), L0, part, done);
        else
          k_pair_resid<P><<<nb, 256, 0, c.stream>>>(e, r0, L0, part, done);
      } else {
        k_pair_resid<P><<<nb, 256, 0, c.stream>>>(e, r0, L0, part, done);
      }
      k_pair_check<<<1, 256, 0, c.stream>>>(part, nb, dst, st, tol, skip);
      e = vcycle<P>(c, 0, skip, e);
    }
    if constexpr (std::is_same<P, float>::value) {
      if (rb)
        k_update_rb<<<nb, 256, 0, c.stream>>>(phi, rb_of(c), r64, L0, part, done);
      else
        k_update<P><<<nb, 256, 0, c.stream>>>(phi, e, r64, r0, L0, part, done);
    } else {
      k_update<P><<<nb, 256, 0, c.stream>>>(phi, e, r64, r0, L0, part, done);
    }
    k_norm<false><<<1, 256, 0, c.stream>>>(part, nb, dst, st, tol, max_cycles, nv, nv == 2 ? skip : nullptr);
  };
  // once done, the true residual b - A phi confirms the end and the face
  // conditions follow, all queued before the one wait of the round
  auto finish = [&] {
    resid0(false, st + 7);
    k_norm_final<<<1, 256, 0, c.stream>>>(part, nb, dst, st, tol, max_cycles, words);
    k_faces<<<face_grid, 64, 0, c.stream>>>(c.phi.p, c.cx, c.cy, c.cz, faces, st + 2);
  };
  auto capture = [&](hipGraphExec_t& exec, size_t* nodes, auto body) {
    if (exec) {
      FOPIS_HIP(hipGraphExecDestroy(exec));
      exec = nullptr;
    }
    hipGraph_t g = nullptr;
    FOPIS_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
    body();
    const hipError_t ec = hipStreamEndCapture(c.stream, &g);
    if (ec != hipSuccess || !g)
      throw Error(FOPIS_E_DEVICE, std::string("V-cycle capture: ") + hipGetErrorString(ec));
    if (nodes) FOPIS_HIP(hipGraphGetNodes(g, nullptr, nodes));
    const hipError_t ei = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ei != hipSuccess) {
      exec = nullptr;
      throw Error(FOPIS_E_DEVICE, std::string("V-cycle graph: ") + hipGetErrorString(ei));
    }
  };
  if (c.mg_use_graph && (!c.mg_graph[0] || c.mg_graph_tol != tol || c.mg_graph_cap != max_cycles)) {
    for (int k = 0; k < 2; ++k) capture(c.mg_graph[k], &c.mg_graph_nodes[k], [&] { cycle(k + 1); });
    c.mg_graph_tol = tol;
    c.mg_graph_cap = max_cycles;
    drop_whole(c);
  }
  hipGraphExec_t whole = nullptr;
  if (c.mg_use_graph && rho0 == c.rho.p && pred <= kWholeMost &&
      npair * c.mg_graph_nodes[1] + batch * c.mg_graph_nodes[0] <= kWholeNodes) {
    Ctx::Whole& w = c.mg_whole[pred];
    if (!w.exec && ++w.seen > kWholeAfter)
      capture(w.exec, nullptr, [&] {
        begin();
        for (int q = 0; q < npair; ++q) cycle(2);
        for (int q = 0; q < batch; ++q) cycle(1);
        finish();
      });
    whole = w.exec;
  }
  auto launch = [&](int nv) {
    if (c.mg_use_graph)
      FOPIS_HIP(hipGraphLaunch(c.mg_graph[nv - 1], c.stream));
    else
      cycle(nv);
  };
  if (!whole) begin();
  for (;;) {
    if (whole) {
      FOPIS_HIP(hipGraphLaunch(whole, c.stream));
      whole = nullptr;
    } else {
      for (int q = 0; q < npair; ++q) launch(2);
      for (int q = 0; q < batch; ++q) launch(1);
      finish();
    }
    if (pairs) {  // later rounds: one pair (up to two cycles) at a time
      npair = 1;
      batch = 0;
    } else {
      npair = 0;
      batch = 2;
    }
    FOPIS_HIP(hipGetLastError());
    FOPIS_HIP(hipStreamSynchronize(c.stream));
    if (!words->done) continue;
    if (words->confirmed) break;
    // the recursively updated residual has drifted from the true one: the
    // further cycles start from the true residual
    resid0(true, never);
    k_reopen<<<1, 1, 0, c.stream>>>(st);
  }
  const int cycles = words->cycles;
  c.mg_updates_last = words->updates;
  c.mg_pair_passes_last = words->pair_passes;
  c.mg_hist[1] = c.mg_hist[0];
  c.mg_hist[0] = cycles;
  *relres_out = words->relres;
  c.relres0_last = words->relres0;
  return cycles;
}

// Plans the tail and lets the level kernels and the tail have the LDS they take.
template <typename P>
void plan_levels(Ctx& c) {
  plan_tail(c, sizeof(P));
  if (c.mg_fused) {
    grant_lds(reinterpret_cast<const void*>(&k_level_down<P, false>), DownDim<P, false>::kLds);
    grant_lds(reinterpret_cast<const void*>(&k_level_down<P, true>), DownDim<P, true>::kLds);
    grant_lds(reinterpret_cast<const void*>(&k_level_up<P>), UpDim<P>::kLds);
  }
  if (c.mg_tail < (int)c.mg.size()) {
    grant_lds(reinterpret_cast<const void*>(&k_coarse_tail<P, false>), c.mg_tail_bytes);
    grant_lds(reinterpret_cast<const void*>(&k_coarse_tail<P, true>), c.mg_tail_bytes);
  }
}

}  // namespace

void poisson_init(Ctx& c) {
  c.mg.clear();
  int n[3] = {c.nx - 2, c.ny - 2, c.nz - 2};
  if (n[0] < 1 || n[1] < 1 || n[2] < 1) throw Error(FOPIS_E_ARG, "grid too small for the Poisson solve");
  const bool f32 = c.d.mg_precision == FOPIS_FP32;
  c.mg.reserve(16);
  for (int l = 0;; ++l) {
    c.mg.emplace_back();
    MgLevel& m = c.mg.back();
    for (int q = 0; q < 3; ++q) m.n[q] = n[q];
    if (l == 0) {
      m.sx = (int64_t)c.cy * c.cz;
      m.sy = c.cz;
      m.size = c.nnode;
      m.off = (int64_t)c.id3(1, 1, 1);
    } else {
      m.sx = (int64_t)(n[1] + 2) * (n[2] + 2);
      m.sy = n[2] + 2;
      m.size = (size_t)(n[0] + 2) * (n[1] + 2) * (n[2] + 2);
    }
    if (f32) {
      m.e32.alloc(m.size);
      m.r32.alloc(m.size);
      m.t32.alloc(m.size);
      FOPIS_HIP(hipMemsetAsync(m.e32.p, 0, m.size * sizeof(float), c.stream));
      FOPIS_HIP(hipMemsetAsync(m.r32.p, 0, m.size * sizeof(float), c.stream));
      FOPIS_HIP(hipMemsetAsync(m.t32.p, 0, m.size * sizeof(float), c.stream));
    } else {
      m.e64.alloc(m.size);
      m.r64.alloc(m.size);
      m.t64.alloc(m.size);
      FOPIS_HIP(hipMemsetAsync(m.e64.p, 0, m.size * sizeof(double), c.stream));
      FOPIS_HIP(hipMemsetAsync(m.r64.p, 0, m.size * sizeof(double), c.stream));
      FOPIS_HIP(hipMemsetAsync(m.t64.p, 0, m.size * sizeof(double), c.stream));
    }
    bool can = true;
    for (int q = 0; q < 3; ++q) can = can && (n[q] >= 3) && (n[q] % 2 == 1);
    if (!can) break;
    for (int q = 0; q < 3; ++q) n[q] = (n[q] - 1) / 2;
  }
  if (f32) {
    c.mg_r64.alloc(c.nnode);
    FOPIS_HIP(hipMemsetAsync(c.mg_r64.p, 0, c.nnode * sizeof(double), c.stream));
  }
  // the finest level stored by colour: FP32 levels, a level large enough to
  // form its residual in a pass of its own (and so never inside the LDS tail),
  // pre-smoothing (its first sweep starts from zero); FOPIS_MG_RB=0 keeps one array
  const char* fu = std::getenv("FOPIS_MG_FUSED");
  c.mg_fused = c.d.mg_pre == 2 && c.d.mg_post == 2 && !(fu && fu[0] == '0');
  const char* rbs = std::getenv("FOPIS_MG_RB");
  const MgLevel& l0 = c.mg[0];
  c.mg_rb = f32 && !(rbs && rbs[0] == '0') && c.mg.size() > 1 && c.d.mg_pre > 0 &&
            (int64_t)l0.n[0] * l0.n[1] * l0.n[2] >= kSplitRestrict;
  if (c.mg_rb) {
    c.rb_sy = (l0.n[2] + 3) / 2;
    c.rb_sx = (int64_t)(l0.n[1] + 2) * c.rb_sy;
    c.rb_cs = (int64_t)(l0.n[0] + 2) * c.rb_sx;
    c.erb.alloc(2 * c.rb_cs);
    c.rrb.alloc(2 * c.rb_cs);
    FOPIS_HIP(hipMemsetAsync(c.erb.p, 0, 2 * c.rb_cs * sizeof(float), c.stream));
    FOPIS_HIP(hipMemsetAsync(c.rrb.p, 0, 2 * c.rb_cs * sizeof(float), c.stream));
  }
  c.mg_state.alloc(8);
  FOPIS_HIP(hipMemsetAsync(c.mg_state.p, 0, 8 * sizeof(int32_t), c.stream));
  c.mg_part.alloc(2 * kResidBlocks + 4);
  const char* g = std::getenv("FOPIS_MG_GRAPH");
  c.mg_use_graph = !(g && g[0] == '0');
  const char* pr2 = std::getenv("FOPIS_MG_PAIRS");
  c.mg_pairs = !(pr2 && pr2[0] == '0');
  const char* cy = std::getenv("FOPIS_CARRY");
  c.carry = !(cy && cy[0] == '0');
  int dev = 0;
  FOPIS_HIP(hipGetDevice(&dev));
  hipDeviceProp_t pr;
  FOPIS_HIP(hipGetDeviceProperties(&pr, dev));
  c.lds_max = pr.sharedMemPerBlock;
  if (f32)
    plan_levels<float>(c);
  else
    plan_levels<double>(c);
  c.mg_hist[0] = c.mg_hist[1] = 1;
  FOPIS_HIP(hipStreamSynchronize(c.stream));
}

void poisson_free(Ctx& c) {
  for (auto& g : c.mg_graph) {
    if (g) (void)hipGraphExecDestroy(g);
    g = nullptr;
  }
  drop_whole(c);
}

int poisson_solve(Ctx& c, double tol, int max_cycles, double* relres, const double* rhs_override) {
  Phase ph(c, "poisson");
  const double* rho0 = rhs_override ? rhs_override : c.rho.p;
  int cyc;
  if (c.d.mg_precision == FOPIS_FP32)
    cyc = solve_impl<float>(c, tol, max_cycles, relres, rho0);
  else
    cyc = solve_impl<double>(c, tol, max_cycles, relres, rho0);
  c.mg_cycles_last = cyc;
  c.mg_cycles_total += cyc;
  c.mg_solves_total += 1;
  c.mg_updates_total += c.mg_updates_last;
  c.mg_pair_passes_total += c.mg_pair_passes_last;
  c.relres_last = *relres;
  return cyc;
}

}  // namespace fopis
