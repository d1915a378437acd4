// Fused selected solve for small blocks (gfx950): one workgroup per energy.
//
// Same algorithm and outputs as rgf_selected_solve in rgf.hip, in the operation
// order of its general sweep (four products per lesser / greater block backward;
// reference src/qttools/greens_function_solver/rgf.py:164-414), for stacks whose blocks
// are all at most kSB = 32 wide and at most kSN = 32 long.  At such sizes every
// block product is a few microseconds of matrix-core work, so the general path
// (one launch per product over the whole stack) is bound by launch latency;
// here the whole sweep of one energy runs in one workgroup of two teams of
// four waves (one wave of each team per SIMD).
//
// - The blocks that one step writes and the next reads stay in LDS; the forward
//   blocks, which the backward sweep reads again, go to a per-energy workspace
//   as well, and their lines and those of A are touched one layer ahead.
// - Block products (sgemm): the four waves of a team each own a 16 x 16
//   quarter of the output and load their MFMA fragments straight from LDS or
//   memory, all k-steps issued before the first v_mfma_f64_16x16x4_f64.
//   4M or 3M split, summed over k in the same order as the batched kernels.
// - The two teams run independent products of one step side by side: the
//   lesser and greater chains of a layer, pairs of retarded products
//   (rgf_small_kernel describes the schedule).
// - Block inverse (sinv): gj_invert (gj_core.h), one factoring and two update
//   waves, the block in matrix-core registers; the other waves wait.
// - Elementwise steps (folds, X - X^H parts, traces) as team loops whose
//   loads are all issued before the first use.
// - A barrier closes every step, which makes its writes visible to the other
//   waves of the workgroup.
//
// Bound by the chain of steps: of about 51 us per layer of 32 (59 with the layer
// current) the inverse takes 17 and each of the 15 product steps 1.5 to 5, for
// under 1 of matrix-core work.  Calls, with all blocks in L2 and 16 blocks at
// most before -> now: 16 energies of 8 blocks of 32 677 -> 540 us, 300 of 11
// blocks of 20 1101 -> 894; against one launch per product: 16 of 32 x 32 2.0 ms
// (4.9), 512 of 32 x 32 4.3 (9.4), 64 of 24 x 16 0.9 (2.6), 1024 of 16 x 32 4.2
// (6.3).
#include <algorithm>
#include <cstdlib>

#include "gj_core.h"
#include "qx_internal.h"

namespace qx {
namespace {

// (the workspace bound of rgf_workspace_bytes in rgf.hip follows these)
constexpr int kSB = 32;   // largest block size
constexpr int kSN = 32;   // largest block count
constexpr int kThreads = 256;       // a team: four waves, one per SIMD
constexpr int kSolveThreads = 512;  // the fused kernels: two teams

typedef double d4 __attribute__((ext_vector_type(4)));

struct SLay {
  int32_t diag[kSN], up[kSN], lo[kSN];  // element offsets, -1: not stored
};

struct SmallArgs {
  int N, flags, NS, split;
  int bmax, slot;  // largest block, elements of a workspace slot (bmax^2)
  int shared;      // G^R in the container of G^< or G^>
  int64_t e0;      // energy of the launch's first workgroup
  int bs[kSN];
  int orb[kSN];  // first orbital of each block (density row offsets)
  int64_t n_orb;
  int64_t sA, sSL, sSG, sXL, sXG, sXR;  // stack strides (elements)
  const z2 *A, *SL, *SG;
  z2 *XL, *XG, *XR;
  SLay lA, lSL, lSG, lXL, lXG, lXR;
  const z2* obc[3][kSN];  // retarded, lesser, greater boundary blocks or null
  z2* ws;                 // per energy NS slots
  int* info;
  z2* current;   // (S, N - 1) or null
  z2* corner;    // (S, b_0, b_{N-1}) or null
  double* density;  // (S, n_orb) or null
};

static_assert(sizeof(SmallArgs) <= 4096, "kernel arguments");

struct M {
  z2* p;
  int ld;
};

__device__ inline M blk(const z2* base, int64_t stride, int64_t e, int32_t off, int ld) {
  if (!base || off < 0) return M{nullptr, ld};
  return M{const_cast<z2*>(base) + e * stride + off, ld};
}

constexpr int kLd = kSB + 1;  // rows of a block in LDS: columns fall into different banks
typedef z2 LdsBlock[kSB * kLd];

struct Shared {
  LdsBlock blk[7];
  union {  // the backward sweep inverts nothing
    GjShared<GjWhole32> winv;
    LdsBlock tail[2];
  };
  double red[2][kSolveThreads / 64];
};
static_assert(sizeof(Shared) <= 160 * 1024, "LDS of a CU");

// Touches the cache lines of a block that a later step reads (threads t of the
// workgroup, each line once); the value is dropped by prefetched().
struct Touch {
  unsigned v = 0;
};
__device__ __forceinline__ void prefetch(Touch& x, int t, int lines0, M A, int elems) {
  const int i = (t - lines0) * 8;  // 128 bytes
  if (A.p && i >= 0 && i < elems) x.v = *reinterpret_cast<const unsigned*>(A.p + i);
}
__device__ __forceinline__ void prefetched(const Touch& x) { asm volatile("" ::"v"(x.v)); }

// Element at a byte offset (32 bits, so that it is an address's lane part).
__device__ __forceinline__ z2& at(z2* p, unsigned byte) {
  return *reinterpret_cast<z2*>(reinterpret_cast<char*>(p) + byte);
}

// C = s op(A) op(B) + D, s = 1 or -1, m, n, k <= 32, by one team of four waves
// (tt: the thread's index in the team), each wave owning a 16 x 16 quarter
// of C; a null A or B is zero.  D is zero, Cin, Cin + Cin2, or (E - E^H) + Cin
// (m == n), null terms zero; C2: a second place for C.  Every load (the fragments of all k-steps
// and the values of D) is issued before the first v_mfma_f64_16x16x4_f64, from
// clamped addresses, with no branch between the loads.  A lane whose row of
// A (column of B) lies outside the block feeds only output rows (columns)
// that are not stored, so its value is left as loaded; only a partial last
// k-step (k not a multiple of 4) has its fragments beyond k zeroed.  No
// barrier.
//
// A step is bound by the instructions around its 32 MFMAs (2048 cycles): with
// clamped indexes per element and general complex factors about 500 of them,
// 6500 cycles a step; one clamp per k-step, byte offsets and signs took 16
// energies of 8 blocks of 32 from 560 to 536 us.
__device__ __forceinline__ void sgemm(int tt, int split, int m, int n, int k, int opa, int opb,
                                      double sign, M A, M B, M Cin, M C, M C2 = M{nullptr, 0},
                                      M Cin2 = M{nullptr, 0}, M E = M{nullptr, 0}) {
  const int w = tt >> 6, lane = tt & 63;
  const int r0 = (w >> 1) * 16, c0 = (w & 1) * 16;
  const int r16 = lane & 15, k4 = lane >> 4;
  if (r0 >= m || c0 >= n) return;
  const int row0 = r0 + k4, col = c0 + r16;  // result element q: row row0 + 4 q
  z2 cin[4];
  const bool use_d = Cin.p || Cin2.p;
  if (use_d) {
    const int cc = min(col, n - 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int rr = min(row0 + 4 * q, m - 1);
      cin[q] = make_double2(0.0, 0.0);
      if (Cin.p) cin[q] = at(Cin.p, 16u * (rr * Cin.ld + cc));
      if (Cin2.p) {
        const z2 v = at(Cin2.p, 16u * (rr * Cin2.ld + cc));
        cin[q] = make_double2(cin[q].x + v.x, cin[q].y + v.y);
      }
      if (E.p) {
        const z2 a = at(E.p, 16u * (rr * E.ld + cc)), b = at(E.p, 16u * (cc * E.ld + rr));
        cin[q] = make_double2((a.x - b.x) + cin[q].x, (a.y + b.y) + cin[q].y);
      }
    }
  }
  d4 a1 = {0, 0, 0, 0}, a2 = {0, 0, 0, 0}, a3 = {0, 0, 0, 0};
  if (A.p && B.p) {
    const unsigned sa = opa == QX_OP_N ? 16u : 16u * A.ld, sb = opb == QX_OP_N ? 16u * B.ld : 16u;
    const unsigned ba = min(r0 + r16, m - 1) * (opa == QX_OP_N ? 16u * A.ld : 16u);
    const unsigned bb = min(col, n - 1) * (opb == QX_OP_N ? 16u : 16u * B.ld);
    z2 fa[kSB / 4], fb[kSB / 4];
#pragma unroll
    for (int s = 0; s < kSB / 4; ++s) {
      const unsigned kk = min(4 * s + k4, k - 1);
      fa[s] = at(A.p, ba + kk * sa);
      fb[s] = at(B.p, bb + kk * sb);
    }
    if (k & 3) {
      const int s = k >> 2;  // the partial k-step
#pragma unroll
      for (int u = 0; u < kSB / 4; ++u) {
        if (u == s && 4 * u + k4 >= k) {
          fa[u] = make_double2(0.0, 0.0);
          fb[u] = make_double2(0.0, 0.0);
        }
      }
    }
    // the conjugations, as the instructions' neg modifiers (bit 0: A, 1: B)
    const bool ca = opa != QX_OP_N, cb = opb != QX_OP_N;
#pragma unroll
    for (int s = 0; s < kSB / 4; ++s) {
      if (4 * s < k) {
        const z2 x = fa[s], y = fb[s];
        if (split == 3) {
          const double xs = ca ? x.x - x.y : x.x + x.y, ys = cb ? y.x - y.y : y.x + y.y;
          a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.x, a1, 0, 0, 0);
          a2 = ca != cb ? __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.y, a2, 0, 0, 1)
                        : __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.y, a2, 0, 0, 0);
          a3 = __builtin_amdgcn_mfma_f64_16x16x4f64(xs, ys, a3, 0, 0, 0);
        } else {
          a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.x, a1, 0, 0, 0);
          a2 = cb ? __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.y, a2, 0, 0, 2)
                  : __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.y, a2, 0, 0, 0);
          a1 = ca == cb ? __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.y, a1, 0, 0, 1)
                        : __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.y, a1, 0, 0, 0);
          a2 = ca ? __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.x, a2, 0, 0, 1)
                  : __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.x, a2, 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = row0 + 4 * q;
    if (row < m && col < n) {
      double vr = a1[q], vi = a2[q];
      if (split == 3) {
        vr = a1[q] - a2[q];
        vi = a3[q] - a1[q] - a2[q];
      }
      if (use_d) {
        vr = sign < 0 ? cin[q].x - vr : cin[q].x + vr;
        vi = sign < 0 ? cin[q].y - vi : cin[q].y + vi;
      } else if (sign < 0) {
        vr = -vr;
        vi = -vi;
      }
      at(C.p, 16u * (row * C.ld + col)) = make_double2(vr, vi);
      if (C2.p) at(C2.p, 16u * (row * C2.ld + col)) = make_double2(vr, vi);
    }
  }
}

// The elementwise steps below run over the threads tt = 0 .. nt - 1 of a
// team (nt a multiple of 64); each thread loads the four elements it owns
// (element t + u nt, u = 0..3, addresses clamped into the block) before it
// uses any of them.  A null operand reads from Y and is not used.  No barrier.

// Y = a A + b B (null operands are zero).
__device__ __forceinline__ void saxpby(int tt, int nt, int m, int n, Cplx a, M A, Cplx b, M B,
                                       M Y) {
  const int mn = m * n;
  const z2* pa = A.p ? A.p : Y.p;
  const z2* pb = B.p ? B.p : Y.p;
  const int la = A.p ? A.ld : Y.ld, lb = B.p ? B.ld : Y.ld;
  for (int t0 = tt; t0 < mn; t0 += 4 * nt) {
    z2 va[4], vb[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = min(t0 + u * nt, mn - 1), r = t / n, c = t - r * n;
      va[u] = pa[r * la + c];
      vb[u] = pb[r * lb + c];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t0 + u * nt;
      if (t < mn) {
        const int r = t / n, c = t - r * n;
        double yr = 0.0, yi = 0.0;
        if (A.p) {
          yr += a.re * va[u].x - a.im * va[u].y;
          yi += a.re * va[u].y + a.im * va[u].x;
        }
        if (B.p) {
          yr += b.re * vb[u].x - b.im * vb[u].y;
          yi += b.re * vb[u].y + b.im * vb[u].x;
        }
        Y.p[r * Y.ld + c] = make_double2(yr, yi);
      }
    }
  }
}

// Y = cy Y + ca A + cb B^H + cc D (real coefficients; Y, m x n, aliases none
// of A, B, D; B is n x m).
__device__ __forceinline__ void sherm(int tt, int nt, int m, int n, double cy, double ca, M A,
                                      double cb, M B, M Y, double cc = 0.0,
                                      M D = M{nullptr, 0}) {
  const int mn = m * n;
  const bool uy = cy != 0.0, ua = ca != 0.0 && A.p, ub = cb != 0.0 && B.p, ud = cc != 0.0 && D.p;
  const z2* pa = ua ? A.p : Y.p;
  const z2* pb = ub ? B.p : Y.p;
  const z2* pd = ud ? D.p : Y.p;
  const int la = ua ? A.ld : Y.ld, ld = ud ? D.ld : Y.ld;
  for (int t0 = tt; t0 < mn; t0 += 4 * nt) {
    z2 vy[4], va[4], vb[4], vd[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = min(t0 + u * nt, mn - 1), r = t / n, c = t - r * n;
      vy[u] = Y.p[r * Y.ld + c];
      va[u] = pa[r * la + c];
      vb[u] = pb[ub ? c * B.ld + r : r * Y.ld + c];
      vd[u] = pd[r * ld + c];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t0 + u * nt;
      if (t < mn) {
        const int r = t / n, c = t - r * n;
        double yr = 0.0, yi = 0.0;
        if (uy) {
          yr = cy * vy[u].x;
          yi = cy * vy[u].y;
        }
        if (ua) {
          yr += ca * va[u].x;
          yi += ca * va[u].y;
        }
        if (ub) {
          yr += cb * vb[u].x;
          yi -= cb * vb[u].y;
        }
        if (ud) {
          yr += cc * vd[u].x;
          yi += cc * vd[u].y;
        }
        Y.p[r * Y.ld + c] = make_double2(yr, yi);
      }
    }
  }
}

__device__ __forceinline__ void sdiag_imag(int tt, int nt, int n, M X, double* out) {
  for (int t = tt; t < n; t += nt) out[t] = X.p[t * X.ld + t].y;
}

// out = Tr(X Y) - Tr(Z W), n x n, by the whole workgroup of nt threads
// (X, Y, Z, W all stored); two barriers.
__device__ __forceinline__ void strace_diff(int nt, int n, M X, M Y, M Z, M W, z2* out,
                                            Shared& sh) {
  double sr = 0.0, si = 0.0;
  for (int t0 = threadIdx.x; t0 < n * n; t0 += 2 * nt) {
    z2 x[2], y[2], z[2], w[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = min(t0 + u * nt, n * n - 1), a = t / n, b = t - a * n;
      x[u] = X.p[a * X.ld + b];
      y[u] = Y.p[b * Y.ld + a];
      z[u] = Z.p[a * Z.ld + b];
      w[u] = W.p[b * W.ld + a];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (t0 + u * nt < n * n) {
        sr += x[u].x * y[u].x - x[u].y * y[u].y;
        si += x[u].x * y[u].y + x[u].y * y[u].x;
        sr -= z[u].x * w[u].x - z[u].y * w[u].y;
        si -= z[u].x * w[u].y + z[u].y * w[u].x;
      }
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sr += __shfl_xor(sr, off, 64);
    si += __shfl_xor(si, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    sh.red[0][threadIdx.x >> 6] = sr;
    sh.red[1][threadIdx.x >> 6] = si;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double tr = 0.0, ti = 0.0;
    for (int u = 0; u < nt / 64; ++u) {
      tr += sh.red[0][u];
      ti += sh.red[1][u];
    }
    *out = make_double2(tr, ti);
  }
  __syncthreads();
}

// In-place inverse of the block X by the workgroup.
__device__ __forceinline__ void sinv(int n, M X, int* info, GjShared<GjWhole32>& sh) {
  gj_invert<GjWhole32>(n, X.p, X.ld, nullptr, 0, X.p, X.ld, info, sh);
  __syncthreads();  // the inverse is visible to the workgroup
}

const Cplx kOneS{1.0, 0.0}, kMinusS{-1.0, 0.0}, kZeroS{0.0, 0.0};

// SP: the complex product split (4 = 4M, 3 = 3M), a template parameter so
// that each inlined block product carries only its own MFMA sequence.
//
// Two teams of four waves share the workgroup.  After the retarded block of
// a layer is known, the lesser (q = 1, team 0) and greater (q = 2, team 1)
// chains have the same shape and run side by side; the retarded products
// that do not depend on each other run one per team (b1 | b2, b3 | b4), and
// the products of the lesser and greater chains that do not need the new
// retarded block (a_ji x^≶_ii, then its product with a_ji^H) run on team 1
// while team 0 forms the retarded block.  Every step ends in one workgroup
// barrier, reached by both teams: a team with nothing to do in a step only
// waits.  Within a step a team may run several products and elementwise
// updates that do not read each other's results.
template <int SP>
__global__ __launch_bounds__(kSolveThreads) void rgf_small_kernel(SmallArgs g) {
  __shared__ Shared sh;
  const int64_t e = g.e0 + blockIdx.x;
  const int N = g.N;
  constexpr int sp = SP;
  const bool want_r = (g.flags & QX_SOLVE_RETARDED) != 0;
  const bool want_r_off = (g.flags & QX_SOLVE_RETARDED_OFFDIAG) != 0;
  const bool want_cur = (g.flags & QX_SOLVE_CURRENT) != 0 && g.current;
  const bool skip_lower[2] = {(g.flags & QX_SOLVE_SKIP_LOWER_L) != 0,
                              (g.flags & QX_SOLVE_SKIP_LOWER_G) != 0};
  int* info = g.info + e;
  z2* W = g.ws + e * (int64_t)g.NS * g.slot;
  const int team = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  const int tt = threadIdx.x & (kThreads - 1);  // thread index in the team
  const int tq = 1 + team;                     // the team's chain: 1 lesser, 2 greater
  auto sync = [] { __syncthreads(); };
  auto slot = [&](int s, int ld) { return M{W + (int64_t)s * g.slot, ld}; };
  auto bs = [&](int i) { return g.bs[i]; };
  // Workspace slots: forward x^R, x^<, x^> (0..3N-1), which the backward sweep
  // reads again, and the temporaries of the optional terms.  Everything else
  // stays in LDS: x^R_jj and x^R_ii in lds(0), lds(1) (swapped every layer),
  // x^< and x^> of the current layer in lds(2), lds(3), where the forward sweep
  // also forms t3 and the backward sweep leaves the full block, further
  // temporaries of the two chains in lds(4), lds(5), and lds(6..8).
  auto F = [&](int q, int i) { return q * N + i; };  // q: 0 r, 1 l, 2 g
  const int R0 = 3 * N;
  auto T4 = [&](int q) { return R0 + q; };
  auto T5 = [&](int q) { return R0 + 2 + q; };
  auto C4 = [&](int q) { return R0 + 4 + q; };
  auto CT = [&](int q) { return R0 + 6 + q; };
  const int PG = R0 + 9, B3 = R0 + 10, C1 = R0 + 11, GC0 = R0 + 12, GC1 = R0 + 13,
            GCT = R0 + 14;  // 3 N + 15 slots
  auto lds = [&](int k) { return M{k < 7 ? sh.blk[k] : sh.tail[k - 7], kLd}; };
  auto XQ = [&](int q) { return lds(1 + q); };
  auto PQ = [&](int q) { return lds(3 + q); };
  auto Ad = [&](int i) { return blk(g.A, g.sA, e, g.lA.diag[i], bs(i)); };
  auto Au = [&](int i) { return blk(g.A, g.sA, e, g.lA.up[i], bs(i + 1)); };   // (i, i+1)
  auto Al = [&](int i) { return blk(g.A, g.sA, e, g.lA.lo[i], bs(i)); };       // (i+1, i)
  auto Sd = [&](int q, int i) {
    return q == 1 ? blk(g.SL, g.sSL, e, g.lSL.diag[i], bs(i)) : blk(g.SG, g.sSG, e, g.lSG.diag[i], bs(i));
  };
  auto Su = [&](int q, int i) {
    return q == 1 ? blk(g.SL, g.sSL, e, g.lSL.up[i], bs(i + 1))
                  : blk(g.SG, g.sSG, e, g.lSG.up[i], bs(i + 1));
  };
  auto Od = [&](int q, int i) {
    return q == 1 ? blk(g.XL, g.sXL, e, g.lXL.diag[i], bs(i)) : blk(g.XG, g.sXG, e, g.lXG.diag[i], bs(i));
  };
  auto Ou = [&](int q, int i) {
    return q == 1 ? blk(g.XL, g.sXL, e, g.lXL.up[i], bs(i + 1)) : blk(g.XG, g.sXG, e, g.lXG.up[i], bs(i + 1));
  };
  auto Ol = [&](int q, int i) {
    return q == 1 ? blk(g.XL, g.sXL, e, g.lXL.lo[i], bs(i)) : blk(g.XG, g.sXG, e, g.lXG.lo[i], bs(i));
  };
  auto obc = [&](int q, int i) {
    const z2* p = g.obc[q][i];
    return M{p ? const_cast<z2*>(p) + e * (int64_t)bs(i) * bs(i) : nullptr, bs(i)};
  };
  const M none{nullptr, 0};
  const int b0 = bs(0), bl = bs(N - 1);
  int gc_cur = GC0, gc_nxt = GC1;

  // ---- block 0 (rgf.py:207-231) ----
  {
    const M X0 = lds(0), t3 = XQ(tq), t6 = PQ(tq);
    saxpby(threadIdx.x, kSolveThreads, b0, b0, kOneS, Ad(0), kMinusS, obc(0, 0), X0);
    sync();
    sinv(b0, X0, info, sh.winv);
    saxpby(tt, kThreads, b0, b0, kOneS, Sd(tq, 0), kOneS, obc(tq, 0), t3);
    if (g.corner && team == 0) saxpby(tt, kThreads, b0, b0, kOneS, X0, kZeroS, none, slot(gc_cur, g.bmax));
    sync();
    sgemm(tt, sp, b0, b0, b0, QX_OP_N, QX_OP_N, 1.0, X0, t3, none, t6);
    saxpby(threadIdx.x, kSolveThreads, b0, b0, kOneS, X0, kZeroS, none, slot(F(0, 0), b0));
    sync();
    sgemm(tt, sp, b0, b0, b0, QX_OP_N, QX_OP_C, 1.0, t6, X0, none, XQ(tq),
          slot(F(tq, 0), b0));
    sync();
  }

  // ---- forward sweep (rgf.py:234-295) ----
  for (int i = 0; i + 1 < N; ++i) {
    const int j = i + 1, bi = bs(i), bj = bs(j);
    const M Xri = lds(i & 1), Xrj = lds(j & 1), t1 = lds(6);
    const bool ob0 = obc(0, j).p != nullptr;
    Touch touch;  // the blocks of A of the next layer
    if (j + 1 < N) {
      prefetch(touch, threadIdx.x, 0, Al(j), bs(j + 1) * bj);
      prefetch(touch, threadIdx.x, 128, Au(j), bj * bs(j + 1));
      prefetch(touch, threadIdx.x, 256, Ad(j + 1), bs(j + 1) * bs(j + 1));
    }
    // team 0: a_ji x^R_ii, then x^R_jj's argument a_jj - a_ji x^R_ii a_ij;
    // team 1 meanwhile: a_ji x^<_ii, then a_ji x^>_ii
#pragma unroll 1
    for (int s = 0; s < 2; ++s) {
      if (team == 0) {
        if (s == 0) {
          sgemm(tt, sp, bj, bi, bi, QX_OP_N, QX_OP_N, 1.0, Al(i), Xri, none, t1);
          if (ob0) saxpby(tt, kThreads, bj, bj, kOneS, Ad(j), kMinusS, obc(0, j), Xrj);
        } else if (ob0) {
          sgemm(tt, sp, bj, bj, bi, QX_OP_N, QX_OP_N, -1.0, t1, Au(i), Xrj, Xrj);
        } else {
          sgemm(tt, sp, bj, bj, bi, QX_OP_N, QX_OP_N, -1.0, t1, Au(i), Ad(j), Xrj);
        }
      } else {
        sgemm(tt, sp, bj, bi, bi, QX_OP_N, QX_OP_N, 1.0, Al(i), XQ(1 + s), none,
              PQ(1 + s));
      }
      sync();
    }
    // each chain: t3 = a_ji x_ii a_ji^H + s_jj (+ boundary); team 0 also the
    // corner's g_c a_ij
    const M t3 = XQ(tq), t5 = PQ(tq), t6 = PQ(tq);
    sgemm(tt, sp, bj, bj, bi, QX_OP_N, QX_OP_C, 1.0, PQ(tq), Al(i), Sd(tq, j), t3, none,
          obc(tq, j));
    if (g.corner && team == 0)
      sgemm(tt, sp, b0, bj, bi, QX_OP_N, QX_OP_N, 1.0, slot(gc_cur, g.bmax), Au(i), none,
            slot(GCT, g.bmax));
    sync();
    if (Su(1, i).p || Su(2, i).p) {
      const M sij = Su(tq, i);
      if (sij.p) sgemm(tt, sp, bj, bj, bi, QX_OP_N, QX_OP_N, 1.0, t1, sij, none, t5);
      sync();
      if (sij.p) sherm(tt, kThreads, bj, bj, 1.0, -1.0, t5, 1.0, t5, t3);  // t3 += t5^H - t5
      sync();
    }
    sinv(bj, Xrj, info, sh.winv);
    sgemm(tt, sp, bj, bj, bj, QX_OP_N, QX_OP_N, 1.0, Xrj, t3, none, t6);
    saxpby(threadIdx.x, kSolveThreads, bj, bj, kOneS, Xrj, kZeroS, none, slot(F(0, j), bj));
    sync();
    sgemm(tt, sp, bj, bj, bj, QX_OP_N, QX_OP_C, 1.0, t6, Xrj, none, XQ(tq),
          slot(F(tq, j), bj));
    if (g.corner && team == 1)
      sgemm(tt, sp, b0, bj, bj, QX_OP_N, QX_OP_N, -1.0, slot(GCT, g.bmax), Xrj, none,
            slot(gc_nxt, g.bmax));
    prefetched(touch);
    sync();
    if (g.corner) {
      const int t = gc_cur;
      gc_cur = gc_nxt;
      gc_nxt = t;
    }
  }

  // ---- last diagonal blocks (rgf.py:297-305), the corner ----
  int rj = (N - 1) & 1;  // LDS block of the full x^R_jj
  {
    const int bn = bs(N - 1);
    const M Xq = XQ(tq), od = Od(tq, N - 1);
    if (g.density && team == 0) sdiag_imag(tt, kThreads, bn, Xq, g.density + e * g.n_orb + g.orb[N - 1]);
    if (od.p) sherm(tt, kThreads, bn, bn, 0.0, 0.5, Xq, -0.5, Xq, od);
    if (g.shared) sync();  // G^R is written last
    if (want_r && team == 0) {
      const M xr = blk(g.XR, g.sXR, e, g.lXR.diag[N - 1], bn);
      if (xr.p) saxpby(tt, kThreads, bn, bn, kOneS, lds(rj), kZeroS, none, xr);
    }
    if (g.corner && team == 1)
      saxpby(tt, kThreads, b0, bl, kOneS, slot(gc_cur, g.bmax), kZeroS, none,
             M{g.corner + e * (int64_t)b0 * bl, bl});
    sync();
  }

  // ---- backward sweep (rgf.py:308-404) ----
  for (int i = N - 2; i >= 0; --i) {
    const int j = i + 1, bi = bs(i), bj = bs(j);
    const bool any_s = Su(1, i).p || Su(2, i).p;
    const M sij = Su(tq, i);
    const M Xri = slot(F(0, i), bi), Xrj = lds(rj), Zr = lds(1 - rj);
    const M Aij = Au(i), Aji = Al(i);
    const M b1 = lds(6), b2 = lds(7), b3 = slot(B3, bj), b4 = lds(8);
    Touch touch, touch2;  // what the next layer reads
    if (i > 0) {
      const int h = i - 1, eh = bs(h) * bs(h);
      prefetch(touch, threadIdx.x, 0, Al(h), bi * bs(h));
      prefetch(touch, threadIdx.x, 128, Au(h), bs(h) * bi);
      prefetch(touch, threadIdx.x, 256, slot(F(0, h), bs(h)), eh);
      prefetch(touch, threadIdx.x, 384, slot(F(1, h), bs(h)), eh);
      prefetch(touch2, threadIdx.x, 0, slot(F(2, h), bs(h)), eh);
    }
    if (team == 0)
      sgemm(tt, sp, bi, bj, bi, QX_OP_N, QX_OP_N, 1.0, Xri, Aij, none, b1);  // xr_ii a_ij
    else
      sgemm(tt, sp, bj, bi, bj, QX_OP_N, QX_OP_N, 1.0, Xrj, Aji, none, b2);  // xr_jj a_ji
    sync();
    if (team == 1)
      sgemm(tt, sp, bi, bi, bj, QX_OP_N, QX_OP_N, 1.0, b1, b2, none, b4);  // b1 b2
    else if (any_s || (want_r && want_r_off))
      sgemm(tt, sp, bi, bj, bj, QX_OP_N, QX_OP_N, 1.0, b1, Xrj, none, b3);  // b1 xr_jj
    sync();

    if (want_cur) {
      // layer current from the forward blocks of layer i and the full blocks
      // of layer j (rgf.py:381-400): tl = a_ji x_ii a_ji^H (+ the Σ_ij terms)
      const M c1 = slot(C1, bi), t4 = slot(T4(tq), bi), tl = slot(CT(tq), bj),
              c4 = slot(C4(tq), bj);
      sgemm(tt, sp, bj, bi, bi, QX_OP_N, QX_OP_N, 1.0, Aji, slot(F(tq, i), bi), none, t4);
      if (any_s && team == 0)
        sgemm(tt, sp, bj, bi, bi, QX_OP_N, QX_OP_N, 1.0, Aji, Xri, none, c1);  // a_ji xr_ii
      sync();
      sgemm(tt, sp, bj, bj, bi, QX_OP_N, QX_OP_C, 1.0, t4, Aji, none, tl);
      sync();
      if (any_s) {
        if (sij.p) sgemm(tt, sp, bj, bj, bi, QX_OP_N, QX_OP_N, 1.0, c1, sij, none, c4);
        sync();
        if (sij.p) sherm(tt, kThreads, bj, bj, 1.0, -1.0, c4, 1.0, c4, tl);
        sync();
      }
      strace_diff(kSolveThreads, bj, slot(CT(2), bj), XQ(1), XQ(2), slot(CT(1), bj),
                  g.current + e * (int64_t)(N - 1) + i, sh);
    }

    // each chain (q = tq): G_ii, G_ij and the outputs
    const int q = tq;
    const M Xi = slot(F(q, i), bi), Xj = XQ(q), t1 = PQ(q), t5 = slot(T5(q), bj), Z = XQ(q);
    // P of the lesser chain replaces b4, P of the greater chain x^R_jj, unless
    // a Σ_ij term needs that below
    const M P = q == 1 ? b4 : any_s ? slot(PG, bj) : Xrj;
    // temp_1x = B4 x_ii; team 0 also G^R_ii = xr_ii + B4 xr_ii
    sgemm(tt, sp, bi, bi, bi, QX_OP_N, QX_OP_N, 1.0, b4, Xi, none, t1);
    if (team == 0) sgemm(tt, sp, bi, bi, bi, QX_OP_N, QX_OP_N, 1.0, b4, Xri, Xri, Zr);
    sync();
    if (any_s) {  // temp_1x -= xr_ii s_ij B3^H
      if (sij.p) sgemm(tt, sp, bi, bj, bi, QX_OP_N, QX_OP_N, 1.0, Xri, sij, none, t5);
      sync();
      if (sij.p) sgemm(tt, sp, bi, bi, bj, QX_OP_N, QX_OP_C, -1.0, t5, b3, t1, t1);
      sync();
    }
    sgemm(tt, sp, bi, bj, bj, QX_OP_N, QX_OP_N, -1.0, b1, Xj, none, P);  // -temp_2x
    sync();
    // x_ii' = x_ii + (temp_1x - temp_1x^H) + temp_2x B1^H;
    // x_ij = -temp_2x - x_ii B2^H (+ xr_ii s_ij xr_jj^H)
    M Oij = Ou(q, i);
    if (!Oij.p) Oij = slot(T4(q), bj);
    sgemm(tt, sp, bi, bi, bj, QX_OP_N, QX_OP_C, -1.0, P, b1, Xi, Z, none, none, t1);
    sgemm(tt, sp, bi, bj, bi, QX_OP_N, QX_OP_C, -1.0, Xi, b2, P, Oij);
    prefetched(touch);
    prefetched(touch2);
    sync();
    if (any_s) {
      if (sij.p) sgemm(tt, sp, bi, bj, bj, QX_OP_N, QX_OP_C, 1.0, t5, Xrj, Oij, Oij);
      sync();
    }
    // outputs: x_ji = -x_ij^H, the diagonal block, the density; team 0 the
    // retarded diagonal block, team 1 its off-diagonal blocks on request
    const M low = Ol(q, i), od = Od(q, i);
    if (!skip_lower[q - 1] && low.p) sherm(tt, kThreads, bj, bi, 0.0, 0.0, none, -1.0, Oij, low);
    if (od.p) sherm(tt, kThreads, bi, bi, 0.0, 0.5, Z, -0.5, Z, od);
    if (g.density && q == 1) sdiag_imag(tt, kThreads, bi, Z, g.density + e * g.n_orb + g.orb[i]);
    if (g.shared) sync();  // G^R is written last
    if (want_r && team == 0) {
      const M xr = blk(g.XR, g.sXR, e, g.lXR.diag[i], bi);
      if (xr.p) saxpby(tt, kThreads, bi, bi, kOneS, Zr, kZeroS, none, xr);
    }
    if (want_r && want_r_off) {
      if (team == 1) {
        const M up = blk(g.XR, g.sXR, e, g.lXR.up[i], bj), lo = blk(g.XR, g.sXR, e, g.lXR.lo[i], bi);
        if (up.p) saxpby(tt, kThreads, bi, bj, kMinusS, b3, kZeroS, none, up);
        if (lo.p) sgemm(tt, sp, bj, bi, bi, QX_OP_N, QX_OP_N, -1.0, b2, Xri, none, lo);
      }
      sync();  // before b2 and b3 are formed again
    }
    // (otherwise the next layer's first products write only b1 and b2, which
    // nobody reads here)
    rj = 1 - rj;
  }
}

// Fused selected inversion (rgf.py:25-113 restated in rgf_selected_inv of
// rgf.hip), one workgroup per energy.
struct SmallInvArgs {
  int N, NS, split;
  int slot;    // elements of a workspace slot
  int64_t e0;  // energy of the launch's first workgroup
  int bs[kSN];
  int64_t sA, sX;
  const z2* A;
  z2* X;
  SLay lA, lX;
  const z2* obc[kSN];
  z2* ws;
  int* info;
};

// Two teams as in rgf_small_kernel: the forward sweep is one chain (team 1
// folds the boundary block while team 0 forms a_ji x_ii); in the backward
// sweep x_ji and x_ij run one per team.
template <int SP>
__global__ __launch_bounds__(kSolveThreads) void rgf_small_inv_kernel(SmallInvArgs g) {
  __shared__ GjShared<GjWhole32> sh;
  const int64_t e = g.e0 + blockIdx.x;
  const int N = g.N;
  constexpr int sp = SP;
  int* info = g.info + e;
  z2* W = g.ws + e * (int64_t)g.NS * g.slot;
  const int team = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
  const int tt = threadIdx.x & (kThreads - 1);
  auto sync = [] { __syncthreads(); };
  auto slot = [&](int s, int ld) { return M{W + (int64_t)s * g.slot, ld}; };
  auto bs = [&](int i) { return g.bs[i]; };
  // slots: forward x_ii (0..N-1), full X_ii from the backward sweep
  // (N..2N-1; block N-1 keeps its forward slot), temporaries
  auto F = [&](int i) { return i; };
  auto full = [&](int i) { return i == N - 1 ? i : N + i; };
  const int T1 = 2 * N, T2 = T1 + 1, T3 = T1 + 2;
  const M none{nullptr, 0};
  auto Ad = [&](int i) { return blk(g.A, g.sA, e, g.lA.diag[i], bs(i)); };
  auto Au = [&](int i) { return blk(g.A, g.sA, e, g.lA.up[i], bs(i + 1)); };
  auto Al = [&](int i) { return blk(g.A, g.sA, e, g.lA.lo[i], bs(i)); };
  auto obc = [&](int i) {
    const z2* p = g.obc[i];
    return M{p ? const_cast<z2*>(p) + e * (int64_t)bs(i) * bs(i) : nullptr, bs(i)};
  };

  // forward sweep (rgf.py:70-92)
  saxpby(threadIdx.x, kSolveThreads, bs(0), bs(0), kOneS, Ad(0), kMinusS, obc(0), slot(F(0), bs(0)));
  sync();
  sinv(bs(0), slot(F(0), bs(0)), info, sh);
  for (int i = 0; i + 1 < N; ++i) {
    const int j = i + 1, bi = bs(i), bj = bs(j);
    const M t1 = slot(T1, bi), Xj = slot(F(j), bj);
    const bool ob = obc(j).p != nullptr;
    if (team == 0)
      sgemm(tt, sp, bj, bi, bi, QX_OP_N, QX_OP_N, 1.0, Al(i), slot(F(i), bi), none, t1);
    else if (ob)
      saxpby(tt, kThreads, bj, bj, kOneS, Ad(j), kMinusS, obc(j), Xj);
    sync();
    if (team == 0)
      sgemm(tt, sp, bj, bj, bi, QX_OP_N, QX_OP_N, -1.0, t1, Au(i), ob ? Xj : Ad(j), Xj);
    sync();
    sinv(bj, Xj, info, sh);
  }
  {
    const M xd = blk(g.X, g.sX, e, g.lX.diag[N - 1], bs(N - 1));
    if (xd.p)
      saxpby(threadIdx.x, kSolveThreads, bs(N - 1), bs(N - 1), kOneS, slot(F(N - 1), bs(N - 1)),
             kZeroS, none, xd);
  }
  // backward sweep (rgf.py:97-110)
  for (int i = N - 2; i >= 0; --i) {
    const int j = i + 1, bi = bs(i), bj = bs(j);
    const M Xii = slot(F(i), bi), Xjj = slot(full(j), bj);
    const M t1 = slot(T1, bi), t2 = slot(T2, bj);
    M Xji = blk(g.X, g.sX, e, g.lX.lo[i], bi);
    if (!Xji.p) Xji = slot(T3, bi);
    const M up = blk(g.X, g.sX, e, g.lX.up[i], bj);
    // x_ji = -(x_jj a_ji) x_ii on team 0, x_ij = -(x_ii a_ij) x_jj on team 1
    if (team == 0)
      sgemm(tt, sp, bj, bi, bj, QX_OP_N, QX_OP_N, 1.0, Xjj, Al(i), none, t1);
    else
      sgemm(tt, sp, bi, bj, bi, QX_OP_N, QX_OP_N, 1.0, Xii, Au(i), none, t2);
    sync();
    if (team == 0)
      sgemm(tt, sp, bj, bi, bi, QX_OP_N, QX_OP_N, -1.0, t1, Xii, none, Xji);
    else if (up.p)
      sgemm(tt, sp, bi, bj, bj, QX_OP_N, QX_OP_N, -1.0, t2, Xjj, none, up);
    sync();
    // x_ii <- x_ii - x_ii a_ij x_ji
    const M Z = slot(full(i), bi);
    if (team == 0)
      sgemm(tt, sp, bi, bi, bj, QX_OP_N, QX_OP_N, -1.0, t2, Xji, Xii, Z);
    sync();
    const M xd = blk(g.X, g.sX, e, g.lX.diag[i], bi);
    if (xd.p) saxpby(threadIdx.x, kSolveThreads, bi, bi, kOneS, Z, kZeroS, none, xd);
  }
}

SLay make_lay(const qx_btd_layout* l, int N) {
  SLay s;
  for (int i = 0; i < kSN; ++i) s.diag[i] = s.up[i] = s.lo[i] = -1;
  if (!l) return s;
  for (int i = 0; i < N; ++i) s.diag[i] = (int32_t)l->diag[i];
  for (int i = 0; i + 1 < N; ++i) {
    s.up[i] = (int32_t)l->upper[i];
    s.lo[i] = (int32_t)l->lower[i];
  }
  return s;
}

bool fits32(const qx_btd_layout* l, int N) {
  if (!l) return true;
  auto ok = [](int64_t v) { return v >= -1 && v < (int64_t(1) << 31); };
  for (int i = 0; i < N; ++i)
    if (!ok(l->diag[i])) return false;
  for (int i = 0; i + 1 < N; ++i)
    if (!ok(l->upper[i]) || !ok(l->lower[i])) return false;
  return true;
}

}  // namespace

// Fused path of rgf_selected_solve for small blocks; returns false (and does
// nothing) when the call is not eligible: complex128 arithmetic (4M or 3M),
// at most 32 blocks of at most 32, offsets below 2^31, and QX_RGF_FUSED not 0.
bool rgf_small_solve(qx_handle* h, hipStream_t st, const qx_btd_layout* la, const void* a,
                     const qx_btd_layout* lsl, const void* sl, const qx_btd_layout* lsg,
                     const void* sg, const void* const* obc_r, const void* const* obc_l,
                     const void* const* obc_g, const qx_btd_layout* lxl, void* xl,
                     const qx_btd_layout* lxg, void* xg, const qx_btd_layout* lxr, void* xr,
                     void* current, void* corner, double* density, double* ldos,
                     uint32_t flags, int prec) {
  const char* env = std::getenv("QX_RGF_FUSED");
  if (env && std::atoi(env) == 0) return false;
  if (ldos) return false;  // the per-product path writes the LDOS
  if (prec != QX_PREC_C128 && prec != QX_PREC_C128_3M) return false;
  const int N = la->n_blocks;
  if (N < 1 || N > kSN) return false;
  for (int i = 0; i < N; ++i)
    if (la->block_sizes[i] < 1 || la->block_sizes[i] > kSB) return false;
  const qx_btd_layout* ls[6] = {la, lsl, lsg, lxl, lxg, lxr};
  for (auto* l : ls)
    if (!fits32(l, N)) return false;
  const int64_t S = la->n_stack;
  if (S <= 0) return true;
  QX_REQUIRE(S < (int64_t(1) << 31), "selected_solve: stack too large");
  SmallArgs g;
  g.N = N;
  g.flags = (int)flags;
  g.NS = 3 * N + 15;
  g.bmax = *std::max_element(la->block_sizes, la->block_sizes + N);
  g.slot = g.bmax * g.bmax;
  g.shared = xr && (xr == xl || xr == xg);
  g.split = prec == QX_PREC_C128_3M ? 3 : 4;
  int off = 0;
  for (int i = 0; i < kSN; ++i) {
    g.bs[i] = i < N ? la->block_sizes[i] : 0;
    g.orb[i] = off;
    if (i < N) off += la->block_sizes[i];
  }
  g.n_orb = off;
  g.sA = la->stack_stride;
  g.sSL = lsl ? lsl->stack_stride : 0;
  g.sSG = lsg ? lsg->stack_stride : 0;
  g.sXL = lxl->stack_stride;
  g.sXG = lxg->stack_stride;
  g.sXR = lxr ? lxr->stack_stride : 0;
  g.A = static_cast<const z2*>(a);
  g.SL = static_cast<const z2*>(sl);
  g.SG = static_cast<const z2*>(sg);
  g.XL = static_cast<z2*>(xl);
  g.XG = static_cast<z2*>(xg);
  g.XR = static_cast<z2*>(xr);
  g.lA = make_lay(la, N);
  g.lSL = make_lay(sl ? lsl : nullptr, N);
  g.lSG = make_lay(sg ? lsg : nullptr, N);
  g.lXL = make_lay(lxl, N);
  g.lXG = make_lay(lxg, N);
  g.lXR = make_lay(xr ? lxr : nullptr, N);
  const void* const* ob[3] = {obc_r, obc_l, obc_g};
  for (int q = 0; q < 3; ++q)
    for (int i = 0; i < kSN; ++i)
      g.obc[q][i] = (ob[q] && i < N) ? static_cast<const z2*>(ob[q][i]) : nullptr;
  g.ws = static_cast<z2*>(h->ensure_ws((size_t)S * g.NS * g.slot * sizeof(z2)));
  g.info = h->ensure_info(S);
  g.current = static_cast<z2*>(current);
  g.corner = static_cast<z2*>(corner);
  g.density = density;
  KernelTimer* timer = active_timer;
  hipEvent_t ev0 = nullptr;
  if (timer) timer->begin(st, &ev0);
  for (g.e0 = 0; g.e0 < S; g.e0 += max_groups(kSolveThreads)) {
    const dim3 grid((unsigned)std::min(S - g.e0, max_groups(kSolveThreads)));
    if (g.split == 3)
      hipLaunchKernelGGL(rgf_small_kernel<3>, grid, dim3(kSolveThreads), 0, st, g);
    else
      hipLaunchKernelGGL(rgf_small_kernel<4>, grid, dim3(kSolveThreads), 0, st, g);
    QX_HIP_CHECK(hipGetLastError());
  }
  if (timer) {
    // matrix flops of the products and inverses the kernel runs when no
    // optional term is present (no current, corner, Σ off-diagonal blocks or
    // off-diagonal G^R): 8 m n k per product, 8 n^3 per inverse; all counted
    // as GEMM work of this one launch
    auto cube = [](double m, double n, double k) { return 8.0 * m * n * k; };
    const double b0 = la->block_sizes[0];
    double fl = 4.0 * cube(b0, b0, b0) + cube(b0, b0, b0);
    for (int i = 0; i + 1 < N; ++i) {
      const double bi = la->block_sizes[i], bj = la->block_sizes[i + 1];
      fl += 3.0 * cube(bj, bi, bi) + 3.0 * cube(bj, bj, bi) + 4.0 * cube(bj, bj, bj)  // forward
            + cube(bj, bj, bj)                                                          // inverse
            + cube(bi, bj, bi) + cube(bj, bi, bj) + cube(bi, bi, bj)  // b1, b2, b4
            + 3.0 * cube(bi, bi, bi) + 2.0 * cube(bi, bj, bj) + 2.0 * cube(bi, bi, bj) +
            2.0 * cube(bi, bj, bi);
    }
    timer->end(st, ev0, KernelTimer::GEMM, fl * (double)S);
  }
  return true;
}

// Fused path of rgf_selected_inv for small blocks (same eligibility as the
// fused solve); returns false, having done nothing, when not eligible.
bool rgf_small_inv(qx_handle* h, hipStream_t st, const qx_btd_layout* la, const void* a,
                   const void* const* obc_r, const qx_btd_layout* lx, void* x, int prec) {
  const char* env = std::getenv("QX_RGF_FUSED");
  if (env && std::atoi(env) == 0) return false;
  if (prec != QX_PREC_C128 && prec != QX_PREC_C128_3M) return false;
  const int N = la->n_blocks;
  if (N < 1 || N > kSN) return false;
  for (int i = 0; i < N; ++i)
    if (la->block_sizes[i] < 1 || la->block_sizes[i] > kSB) return false;
  if (!fits32(la, N) || !fits32(lx, N)) return false;
  const int64_t S = la->n_stack;
  if (S <= 0) return true;
  QX_REQUIRE(S < (int64_t(1) << 31), "selected_inv: stack too large");
  SmallInvArgs g;
  g.N = N;
  g.NS = 2 * N + 3;
  const int bmax = *std::max_element(la->block_sizes, la->block_sizes + N);
  g.slot = bmax * bmax;
  g.split = prec == QX_PREC_C128_3M ? 3 : 4;
  for (int i = 0; i < kSN; ++i) {
    g.bs[i] = i < N ? la->block_sizes[i] : 0;
    g.obc[i] = (obc_r && i < N) ? static_cast<const z2*>(obc_r[i]) : nullptr;
  }
  g.sA = la->stack_stride;
  g.sX = lx->stack_stride;
  g.A = static_cast<const z2*>(a);
  g.X = static_cast<z2*>(x);
  g.lA = make_lay(la, N);
  g.lX = make_lay(lx, N);
  g.ws = static_cast<z2*>(h->ensure_ws((size_t)S * g.NS * g.slot * sizeof(z2)));
  g.info = h->ensure_info(S);
  KernelTimer* timer = active_timer;
  hipEvent_t ev0 = nullptr;
  if (timer) timer->begin(st, &ev0);
  for (g.e0 = 0; g.e0 < S; g.e0 += max_groups(kSolveThreads)) {
    const dim3 grid((unsigned)std::min(S - g.e0, max_groups(kSolveThreads)));
    if (g.split == 3)
      hipLaunchKernelGGL(rgf_small_inv_kernel<3>, grid, dim3(kSolveThreads), 0, st, g);
    else
      hipLaunchKernelGGL(rgf_small_inv_kernel<4>, grid, dim3(kSolveThreads), 0, st, g);
    QX_HIP_CHECK(hipGetLastError());
  }
  if (timer) {
    // matrix flops of its products and inverses (8 m n k, 8 n^3), counted as
    // GEMM work of this one launch
    auto cube = [](double m, double n, double k) { return 8.0 * m * n * k; };
    const double b0 = la->block_sizes[0];
    double fl = cube(b0, b0, b0);
    for (int i = 0; i + 1 < N; ++i) {
      const double bi = la->block_sizes[i], bj = la->block_sizes[i + 1];
      fl += cube(bj, bi, bi) + cube(bj, bj, bi) + cube(bj, bj, bj)  // forward + inverse
            + cube(bj, bi, bj) + cube(bj, bi, bi) + cube(bi, bj, bi) + cube(bi, bj, bj) +
            cube(bi, bi, bj);                                          // backward
    }
    timer->end(st, ev0, KernelTimer::GEMM, fl * (double)S);
  }
  return true;
}

}  // namespace qx
