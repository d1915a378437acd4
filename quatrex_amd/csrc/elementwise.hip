// Elementwise and reduction kernels around the GEMM / inverse workhorses.
//
// The conjugate-transpose forms (X - X^H, T^H - T, -X^H) read the transposed
// operand through a 32 x 32 LDS tile so that both the plain and the
// transposed reads are coalesced.  Reductions (traces, norms) use a fixed
// number of workgroups per matrix and a fixed summation order, so results do not
// depend on how many matrices share a launch.
#include <algorithm>
#include <cmath>

#include "qx_internal.h"

namespace qx {
namespace {

constexpr int TS = 32;    // tile edge
constexpr int NT = 256;   // threads per workgroup

struct AxpbyArgs {
  int m, n;
  double ar, ai, br, bi;
  const z2* A;
  int64_t sA;
  int lda;
  const z2* B;
  int64_t sB;
  int ldb;
  z2* Y;
  int64_t sY;
  int ldy;
};

__global__ __launch_bounds__(NT) void axpby_kernel(AxpbyArgs g, int64_t total) {
  const int64_t mn = (int64_t)g.m * g.n;
  for (int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT) {
    const int64_t e = i / mn;
    const int64_t rc = i - e * mn;
    const int r = (int)(rc / g.n), c = (int)(rc - (int64_t)r * g.n);
    double yr = 0.0, yi = 0.0;
    if (g.A) {
      const z2 a = g.A[e * g.sA + (int64_t)r * g.lda + c];
      yr += g.ar * a.x - g.ai * a.y;
      yi += g.ar * a.y + g.ai * a.x;
    }
    if (g.B) {
      const z2 b = g.B[e * g.sB + (int64_t)r * g.ldb + c];
      yr += g.br * b.x - g.bi * b.y;
      yi += g.br * b.y + g.bi * b.x;
    }
    g.Y[e * g.sY + (int64_t)r * g.ldy + c] = make_double2(yr, yi);
  }
}

__global__ __launch_bounds__(NT) void ident_sub_kernel(z2* Y, int64_t sY, int ldy, int n,
                                                       int64_t total) {
  const int64_t nn = (int64_t)n * n;
  for (int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT) {
    const int64_t e = i / nn;
    const int64_t rc = i - e * nn;
    const int r = (int)(rc / n), c = (int)(rc - (int64_t)r * n);
    z2* y = Y + e * sY + (int64_t)r * ldy + c;
    const z2 v = *y;
    *y = make_double2((r == c ? 1.0 : 0.0) - v.x, -v.y);
  }
}

// Y = cy*Y + ca*A + cb*conj(B^T) + cc*D; Y, A, D are m x n, B is n x m.  Real coefs.
struct HermArgs {
  int m, n;
  double cy, ca, cb;
  const z2* A;
  int64_t sA;
  int lda;
  const z2* B;
  int64_t sB;
  int ldb;
  z2* Y;
  int64_t sY;
  int ldy;
  int tm, tn;
  double cc;
  const z2* D;
  int64_t sD;
  int ldd;
  // Two groups of matrices in one launch: matrices e >= half use the second
  // A, B and Y (index e - half); D is single-group only.  One group sets
  // half = batch and the second set equal to the first.
  int64_t half;
  const z2* A2;
  int64_t sA2;
  int lda2;
  const z2* B2;
  int64_t sB2;
  int ldb2;
  z2* Y2;
  int64_t sY2;
  int ldy2;
};

// Workgroup ids are dealt round-robin over the 8 XCDs; this maps them so
// that each XCD receives one contiguous range of logical ids (the tiles of
// one matrix together).
__device__ inline int tile_xcd_remap(int bid, int nblocks) {
  const int nx = 8;
  const int per = nblocks / nx, rem = nblocks % nx;
  const int x = bid % nx, j = bid / nx;
  return x * per + min(x, rem) + j;
}

// Tiles (r, c) and (c, r) read each other's data: with the tiles of a matrix
// on one XCD the second read comes from its L2.
__global__ __launch_bounds__(NT) void herm_kernel(HermArgs g) {
  __shared__ z2 tile[TS][TS + 1];
  const int tiles = g.tm * g.tn;
  const int id = tile_xcd_remap(blockIdx.x, gridDim.x);
  const int64_t eg = id / tiles;
  const int t = id - (int)(eg * tiles);
  const bool second = eg >= g.half;
  const int64_t e = second ? eg - g.half : eg;
  const z2* A = second ? g.A2 + e * g.sA2 : (g.A ? g.A + e * g.sA : nullptr);
  const z2* B = second ? g.B2 + e * g.sB2 : (g.B ? g.B + e * g.sB : nullptr);
  z2* Y = second ? g.Y2 + e * g.sY2 : g.Y + e * g.sY;
  const int lda = second ? g.lda2 : g.lda, ldb = second ? g.ldb2 : g.ldb,
            ldy = second ? g.ldy2 : g.ldy;
  const int r0 = (t / g.tn) * TS, c0 = (t % g.tn) * TS;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  if (g.B) {
    // tile[j][i] = B[c0 + j][r0 + i]
    for (int j = ty; j < TS; j += 8) {
      const int br = c0 + j, bc = r0 + tx;
      z2 v = make_double2(0.0, 0.0);
      if (br < g.n && bc < g.m) v = B[(int64_t)br * ldb + bc];
      tile[j][tx] = v;
    }
  }
  __syncthreads();
  for (int i = ty; i < TS; i += 8) {
    const int r = r0 + i, c = c0 + tx;
    if (r >= g.m || c >= g.n) continue;
    double yr = 0.0, yi = 0.0;
    z2* y = Y + (int64_t)r * ldy + c;
    if (g.cy != 0.0) {
      const z2 v = *y;
      yr = g.cy * v.x;
      yi = g.cy * v.y;
    }
    if (g.A) {
      const z2 a = A[(int64_t)r * lda + c];
      yr += g.ca * a.x;
      yi += g.ca * a.y;
    }
    if (g.B) {
      const z2 b = tile[tx][i];  // B[c][r]
      yr += g.cb * b.x;
      yi -= g.cb * b.y;
    }
    if (g.D) {
      const z2 d = g.D[e * g.sD + (int64_t)r * g.ldd + c];
      yr += g.cc * d.x;
      yi += g.cc * d.y;
    }
    *y = make_double2(yr, yi);
  }
}

// One launch over batch matrices, or over two groups of batch matrices when
// A2 / B2 / Y2 are given (the second group's operands; D must then be zero).
void herm(hipStream_t s, int64_t batch, int m, int n, double cy, double ca,
          const Mat& A, double cb, const Mat& B, const Mat& Y, double cc = 0.0,
          const Mat& D = Mat(), const Mat* A2 = nullptr, const Mat* B2 = nullptr,
          const Mat* Y2 = nullptr) {
  if (batch <= 0 || m <= 0 || n <= 0) return;
  const bool two = Y2 != nullptr;
  QX_REQUIRE(!two || (D.zero() && A2 && B2 && A2->zero() == A.zero() &&
                      B2->zero() == B.zero() && !Y2->zero()),
             "herm: a two-group launch needs matching operands and no D term");
  const Mat& a2 = two ? *A2 : A;
  const Mat& b2 = two ? *B2 : B;
  const Mat& y2 = two ? *Y2 : Y;
  HermArgs g{m, n, cy, ca, cb, A.p, A.stride, A.ld, B.p, B.stride, B.ld,
             Y.p, Y.stride, Y.ld, (m + TS - 1) / TS, (n + TS - 1) / TS,
             cc, D.p, D.stride, D.ld, batch,
             a2.p, a2.stride, a2.ld, b2.p, b2.stride, b2.ld, y2.p, y2.stride, y2.ld};
  const int64_t blocks = (two ? 2 : 1) * batch * g.tm * g.tn;
  hipLaunchKernelGGL(herm_kernel, dim3(groups(blocks, NT, "herm")), dim3(NT), 0, s, g);
  QX_HIP_CHECK(hipGetLastError());
}

// Tile pair t of the upper triangle of tn x tn tiles: (rt, ct), rt <= ct.
__device__ inline void tile_pair(int t, int tn, int& rt, int& ct) {
  rt = 0;
  while (t >= tn - rt) {
    t -= tn - rt;
    ++rt;
  }
  ct = rt + t;
}

// Y = (X - X^H) / 2 + (P - P^H) = W - W^H with W = X / 2 + P, on the tile pair
// (rt, ct), (ct, rt): every element is read once, and Y is skew-Hermitian to
// the bit.  Streaming: 48 n^2 bytes per matrix (the projection kernel it
// replaces moved 32 n^2 and read each X twice).
struct SkewArgs {
  int n, tn;
  int64_t half;  // matrices per group
  const z2 *X[2], *P[2];
  z2* Y[2];
  int64_t sX[2], sP[2], sY[2];
  int lx[2], lp[2], ly[2];
  double* dens;  // Im diag of group 0's Y, or null
  int64_t sd;
};

__global__ __launch_bounds__(NT) void skew_update_kernel(SkewArgs g) {
  __shared__ z2 wa[TS][TS + 1], wb[TS][TS + 1];
  const int pairs = g.tn * (g.tn + 1) / 2;
  const int id = tile_xcd_remap(blockIdx.x, gridDim.x);
  const int64_t eg = id / pairs;
  int rt, ct;
  tile_pair(id - (int)(eg * pairs), g.tn, rt, ct);
  const int grp = eg >= g.half ? 1 : 0;
  const int64_t e = eg - grp * g.half;
  const z2* X = grp ? g.X[1] + e * g.sX[1] : g.X[0] + e * g.sX[0];
  const z2* P = grp ? g.P[1] + e * g.sP[1] : g.P[0] + e * g.sP[0];
  z2* Y = grp ? g.Y[1] + e * g.sY[1] : g.Y[0] + e * g.sY[0];
  const int lx = grp ? g.lx[1] : g.lx[0], lp = grp ? g.lp[1] : g.lp[0],
            ly = grp ? g.ly[1] : g.ly[0];
  const int n = g.n, r0 = rt * TS, c0 = ct * TS;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  z2 xa[4], pa[4], xb[4], pb[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    // all loads in flight together, from addresses clamped into the block
    const int i = ty + 8 * k;
    const int ra = min(r0 + i, n - 1), ca = min(c0 + tx, n - 1);
    const int rb = min(c0 + i, n - 1), cb = min(r0 + tx, n - 1);
    xa[k] = X[(int64_t)ra * lx + ca];
    pa[k] = P[(int64_t)ra * lp + ca];
    xb[k] = X[(int64_t)rb * lx + cb];
    pb[k] = P[(int64_t)rb * lp + cb];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int i = ty + 8 * k;
    wa[i][tx] = make_double2(fma(0.5, xa[k].x, pa[k].x), fma(0.5, xa[k].y, pa[k].y));
    wb[i][tx] = make_double2(fma(0.5, xb[k].x, pb[k].x), fma(0.5, xb[k].y, pb[k].y));
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int i = ty + 8 * k;
    {
      const int r = r0 + i, c = c0 + tx;
      if (r < n && c < n) {
        const z2 u = wa[i][tx], v = wb[tx][i];
        const z2 y = make_double2(u.x - v.x, u.y + v.y);
        Y[(int64_t)r * ly + c] = y;
        if (g.dens && grp == 0 && r == c) g.dens[e * g.sd + r] = y.y;
      }
    }
    if (rt != ct) {
      const int r = c0 + i, c = r0 + tx;
      if (r < n && c < n) {
        const z2 u = wb[i][tx], v = wa[tx][i];
        Y[(int64_t)r * ly + c] = make_double2(u.x - v.x, u.y + v.y);
      }
    }
  }
}

// Largest |s| and largest |s_rc + conj s_cr| (|re| + |im|) of one matrix of one
// block per workgroup; the flag is raised if the second exceeds 64 eps of the
// first, or if anything is not finite.
constexpr int kSkewBlocks = 64;  // blocks per launch
struct SkewCheckArgs {
  int blocks;
  const z2* p[kSkewBlocks];
  int64_t stride[kSkewBlocks];
  int n[kSkewBlocks];
  int* flag;
};

__global__ __launch_bounds__(NT) void skew_check_kernel(SkewCheckArgs g) {
  __shared__ z2 tile[TS][TS + 1];
  __shared__ double red[2][NT / 64];
  const int blk = blockIdx.x % g.blocks;
  const int64_t e = blockIdx.x / g.blocks;
  if (e > 0 && g.stride[blk] == 0) return;  // one matrix for the whole stack
  const z2* S = g.p[blk] + e * g.stride[blk];
  const int n = g.n[blk], tn = (n + TS - 1) / TS;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  double m = 0.0, d = 0.0;
  bool bad = false;
  for (int rt = 0; rt < tn; ++rt)
    for (int ct = rt; ct < tn; ++ct) {
      const int r0 = rt * TS, c0 = ct * TS;
      z2 a[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = ty + 8 * k;
        const int ra = min(r0 + i, n - 1), ca = min(c0 + tx, n - 1);
        const int rb = min(c0 + i, n - 1), cb = min(r0 + tx, n - 1);
        a[k] = S[(int64_t)ra * n + ca];
        tile[i][tx] = S[(int64_t)rb * n + cb];
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = ty + 8 * k;
        if (r0 + i < n && c0 + tx < n) {
          const z2 b = tile[tx][i];  // S[c0 + tx][r0 + i]
          const double ma = fabs(a[k].x) + fabs(a[k].y), mb = fabs(b.x) + fabs(b.y);
          const double df = fabs(a[k].x + b.x) + fabs(a[k].y - b.y);
          bad = bad || !(ma < INFINITY) || !(mb < INFINITY);
          m = fmax(m, fmax(ma, mb));
          d = fmax(d, df);
        }
      }
      __syncthreads();
    }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    m = fmax(m, __shfl_xor(m, off, 64));
    d = fmax(d, __shfl_xor(d, off, 64));
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][w] = m;
    red[1][w] = d;
  }
  __syncthreads();
  for (int u = 0; u < NT / 64; ++u) {
    m = fmax(m, red[0][u]);
    d = fmax(d, red[1][u]);
  }
  // 2^-46 = 64 eps: above the rounding of a product C C^H, below the error the
  // recursion itself makes
  if (bad || !(d <= 0x1p-46 * m)) *g.flag = 1;
}

// Contact self-energies from Sigma^R (one 32 x 32 tile per workgroup, the
// transposed tile through LDS): D = S - S^H, L = -f D, G = (1 - f) D with
// one occupation f per matrix (i f Gamma and i (f - 1) Gamma for
// Gamma = i (S - S^H)).
__global__ __launch_bounds__(NT) void contact_sigma_kernel(const z2* S, int64_t sS, int n,
                                                           const double* f, z2* L, int64_t sL,
                                                           z2* G, int64_t sG, int tn) {
  __shared__ z2 tile[TS][TS + 1];
  const int tiles = tn * tn;
  const int id = tile_xcd_remap(blockIdx.x, gridDim.x);  // as herm_kernel
  const int64_t e = id / tiles;
  const int t = id - (int)(e * tiles);
  const int r0 = (t / tn) * TS, c0 = (t % tn) * TS;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  const z2* Se = S + e * sS;
  for (int j = ty; j < TS; j += 8) {
    const int sr = c0 + j, sc = r0 + tx;
    z2 v = make_double2(0.0, 0.0);
    if (sr < n && sc < n) v = Se[(int64_t)sr * n + sc];
    tile[j][tx] = v;  // S[c0 + j][r0 + tx]
  }
  __syncthreads();
  const double fe = f[e];
  for (int i = ty; i < TS; i += 8) {
    const int r = r0 + i, c = c0 + tx;
    if (r >= n || c >= n) continue;
    const z2 a = Se[(int64_t)r * n + c];
    const z2 b = tile[tx][i];  // S[c][r]
    const double dr = a.x - b.x, di = a.y + b.y;
    L[e * sL + (int64_t)r * n + c] = make_double2(-fe * dr, -fe * di);
    G[e * sG + (int64_t)r * n + c] = make_double2((1.0 - fe) * dr, (1.0 - fe) * di);
  }
}

__global__ __launch_bounds__(NT) void diag_imag_kernel(const z2* X, int64_t sX, int ldx, int n,
                                                       double* out, int64_t so, int64_t total,
                                                       double scale) {
  for (int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT) {
    const int64_t e = i / n;
    const int r = (int)(i - e * n);
    out[e * so + r] = scale * X[e * sX + (int64_t)r * ldx + r].y;
  }
}

// System matrix on the nnz pattern: A[e, k] = z_e S_k + T_k - Sig[e, k].
// A thread covers one entry of E energies: S and T are read once for them, their
// Sigma loads are in flight together.  The grid is entries by groups of energies,
// flat below kAsmFlat entries, where one 32-bit division finds the thread's place
// (one thread per element of a flat grid: two 64-bit divisions each).
// Streaming, 32 bytes per entry and energy with Sigma, 16 without.
// With Sigma E = 4 and stores past the caches, else E = 8: eight loads and eight
// stores in rows a power of two apart evict each other.  us, one thread per
// element / E = 8 / as it is (a grid of entries by energies at 30 entries: 18):
//   energies x entries   with Sigma           without
//   64 x 262144           98 / 108 /  88       39 /  45
//   64 x 262656          147 / 101 /  96      113 /  49
//   256 x 100000         194 / 159 / 145       91 /  76
//   256 x 866304        1674 /1326 /1258      988 / 624
//   100000 x 30         15.5 /15.4 /16.5     11.0 / 9.7
constexpr int64_t kAsmFlat = 2048;
template <bool SIG, int E>
__global__ __launch_bounds__(NT) void assemble_kernel(const z2* z, const z2* S, const z2* T,
                                                      const z2* Sig, int64_t sSig, z2* A,
                                                      int64_t sA, unsigned nnz, int64_t batch) {
  unsigned k = blockIdx.x * (unsigned)NT + threadIdx.x, grp = blockIdx.y;
  if (nnz < kAsmFlat) {
    grp = k / nnz;
    k -= grp * nnz;
  }
  const int64_t e0 = grp * (int64_t)E;
  if (k >= nnz || e0 >= batch) return;
  const int ne = (int)(batch - e0 < E ? batch - e0 : E);
  z2 sg[E];
  if constexpr (SIG) {
#pragma unroll
    for (int u = 0; u < E; ++u) sg[u] = Sig[(e0 + (u < ne ? u : 0)) * sSig + k];
  }
  const z2 sk = S ? S[k] : make_double2(0.0, 0.0);
  const z2 tk = T ? T[k] : make_double2(0.0, 0.0);
#pragma unroll
  for (int u = 0; u < E; ++u) {
    if (u < ne) {
      double vr = 0.0, vi = 0.0;
      if (S) {
        const z2 ze = z[e0 + u];
        vr = ze.x * sk.x - ze.y * sk.y;
        vi = ze.x * sk.y + ze.y * sk.x;
      }
      if (T) {
        vr += tk.x;
        vi += tk.y;
      }
      if constexpr (SIG) {
        vr -= sg[u].x;
        vi -= sg[u].y;
      }
      double* a = &A[(e0 + u) * sA + k].x;
      if constexpr (SIG) {
        typedef double d2 __attribute__((ext_vector_type(2)));
        __builtin_nontemporal_store(d2{vr, vi}, reinterpret_cast<d2*>(a));
      } else {
        a[0] = vr;
        a[1] = vi;
      }
    }
  }
}

// Block reduction of NT doubles in a fixed order.
__device__ inline double block_sum(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < NT / 64; ++q) s += red[q];
  __syncthreads();
  return s;
}

struct TraceArgs {
  int n;
  const z2 *X, *Y, *Z, *W;
  int64_t sX, sY, sZ, sW;
  int lx, ly, lz, lw;
  z2* out;
  int64_t so;
};

// tr(X Y - Z W) = sum_ab X[a][b] Y[b][a] - Z[a][b] W[b][a].  One workgroup per
// 32 rows a of a matrix; Y and W are read through LDS tiles, so every read is
// coalesced.  The partial sums of a matrix's row tiles go to `part` and are
// added in order by trace_sum_kernel, so a result does not depend on how many
// matrices share the launch.  (One workgroup per matrix with strided reads of
// Y and W: 282 us for 12 matrices of 176; 64 n^2 bytes are streamed.)
__global__ __launch_bounds__(NT) void trace_kernel(TraceArgs g, int tn, z2* part, int64_t sp) {
  __shared__ z2 ty_[TS][TS + 1], tw_[TS][TS + 1];
  __shared__ double red[NT / 64];
  const int64_t e = blockIdx.x / tn;
  const int rt = (int)(blockIdx.x - e * tn), r0 = rt * TS;
  const int n = g.n;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  double sr = 0.0, si = 0.0;
  for (int c0 = 0; c0 < n; c0 += TS) {
    z2 x[4], z[4], y[4], w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // rows a of X and Z, rows b of Y and W, from clamped addresses
      const int i = ty + 8 * k;
      const int ra = min(r0 + i, n - 1), ca = min(c0 + tx, n - 1);
      const int rb = min(c0 + i, n - 1), cb = min(r0 + tx, n - 1);
      if (g.X) {
        x[k] = g.X[e * g.sX + (int64_t)ra * g.lx + ca];
        y[k] = g.Y[e * g.sY + (int64_t)rb * g.ly + cb];
      }
      if (g.Z) {
        z[k] = g.Z[e * g.sZ + (int64_t)ra * g.lz + ca];
        w[k] = g.W[e * g.sW + (int64_t)rb * g.lw + cb];
      }
    }
    __syncthreads();  // the previous tile has been read
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (g.X) ty_[ty + 8 * k][tx] = y[k];
      if (g.Z) tw_[ty + 8 * k][tx] = w[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = ty + 8 * k;
      if (r0 + i < n && c0 + tx < n) {
        if (g.X) {
          const z2 v = ty_[tx][i];
          sr += x[k].x * v.x - x[k].y * v.y;
          si += x[k].x * v.y + x[k].y * v.x;
        }
        if (g.Z) {
          const z2 v = tw_[tx][i];
          sr -= z[k].x * v.x - z[k].y * v.y;
          si -= z[k].x * v.y + z[k].y * v.x;
        }
      }
    }
  }
  sr = block_sum(sr, red);
  si = block_sum(si, red);
  if (threadIdx.x == 0) part[e * sp + rt] = make_double2(sr, si);
}

__global__ __launch_bounds__(NT) void trace_sum_kernel(const z2* part, int64_t sp, int tn, z2* out,
                                                       int64_t so, int64_t batch) {
  const int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x;
  if (e >= batch) return;
  double sr = 0.0, si = 0.0;
  for (int t = 0; t < tn; ++t) {
    const z2 v = part[e * sp + t];
    sr += v.x;
    si += v.y;
  }
  out[e * so] = make_double2(sr, si);
}

// One workgroup of NTN threads per matrix, four elements of both in flight per
// thread (NT threads and one element: 21 us for 32 matrices of 96).
constexpr int NTN = 1024;
__global__ __launch_bounds__(NTN) void absnorm_kernel(int n, const z2* A, int64_t sA, int lda,
                                                      const z2* B, int64_t sB, int ldb,
                                                      double* out) {
  __shared__ double red[NTN / 64];
  const int64_t e = blockIdx.x;
  const int nn = n * n;
  double acc = 0.0;
  for (int i0 = threadIdx.x; i0 < nn; i0 += 4 * NTN) {
    z2 a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int idx = min(i0 + u * NTN, nn - 1);
      const int r = idx / n, c = idx - r * n;
      a[u] = A[e * sA + (int64_t)r * lda + c];
      b[u] = B[e * sB + (int64_t)r * ldb + c];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double v = hypot(a[u].x, a[u].y) + hypot(b[u].x, b[u].y);
      if (i0 + u * NTN < nn) acc += v * v;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int q = 0; q < NTN / 64; ++q) s += red[q];
    out[e] = sqrt(s);
  }
}

__global__ __launch_bounds__(NT) void max_kernel(int64_t n, const double* v, double* out) {
  __shared__ double red[NT / 64];
  double m = -INFINITY;
  for (int64_t i = threadIdx.x; i < n; i += NT) {
    const double x = v[i];
    m = x > m ? x : m;  // a NaN is passed over
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < NT / 64; ++q) m = fmax(m, red[q]);
    *out = v[0] == v[0] ? m : v[0];
  }
}

// Newton-Schulz check of one complex64 block inverse per workgroup (see
// ew_ns_check).  Every thread reads the flag after the block sum, so the
// zeroing pass is uniform over the workgroup.
__global__ __launch_bounds__(NT) void ns_check_kernel(int n, z2* R, int64_t sR, int ldr,
                                                      double tol, int* flagged, int* info) {
  __shared__ double red[NT / 64];
  __shared__ int flag;
  const int64_t e = blockIdx.x;
  z2* Re = R + e * sR;
  double acc = 0.0;
  for (int idx = threadIdx.x; idx < n * n; idx += NT) {
    const int r = idx / n, c = idx - r * n;
    const z2 v = Re[(int64_t)r * ldr + c];
    acc += v.x * v.x + v.y * v.y;
  }
  acc = block_sum(acc, red);
  if (threadIdx.x == 0) {
    // NaN and Inf fail the comparison
    flag = sqrt(acc) < tol ? 0 : 1;
    flagged[e] = flag;
    if (flag) info[e] |= 2;
  }
  __syncthreads();
  if (flag)
    for (int idx = threadIdx.x; idx < n * n; idx += NT) {
      const int r = idx / n, c = idx - r * n;
      Re[(int64_t)r * ldr + c] = make_double2(0.0, 0.0);
    }
}

struct ContourArgs {
  int nq, b;
  const z2 *aji, *aii, *aij;
  int64_t s0, s1, s2;
  int l0, l1, l2;
  const z2* z;
  z2* T;
  int64_t sT;
  int lT;
};

__device__ inline z2 cmul(z2 a, z2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// T[e*nq + q] = aji[e] / z_q + aii[e] + aij[e] z_q  (operator.py:57-110)
__global__ __launch_bounds__(NT) void contour_kernel(ContourArgs g, int64_t total) {
  const int64_t bb = (int64_t)g.b * g.b;
  for (int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT) {
    const int64_t eq = i / bb;
    const int64_t rc = i - eq * bb;
    const int r = (int)(rc / g.b), c = (int)(rc - (int64_t)r * g.b);
    const int64_t e = eq / g.nq;
    const int q = (int)(eq - e * g.nq);
    const z2 z = g.z[q];
    const double den = z.x * z.x + z.y * z.y;
    const z2 zi = make_double2(z.x / den, -z.y / den);
    const z2 a0 = g.aji[e * g.s0 + (int64_t)r * g.l0 + c];
    const z2 a1 = g.aii[e * g.s1 + (int64_t)r * g.l1 + c];
    const z2 a2 = g.aij[e * g.s2 + (int64_t)r * g.l2 + c];
    const z2 t0 = cmul(a0, zi), t2 = cmul(a2, z);
    g.T[eq * g.sT + (int64_t)r * g.lT + c] =
        make_double2(t0.x + a1.x + t2.x, t0.y + a1.y + t2.y);
  }
}

struct OperatorArgs {
  int nq, d, nt;
  const z2* a[kOperatorTerms];
  int64_t s[kOperatorTerms];  // matrix strides, 0: one for the batch
  const z2* w;                // nt x nq
  z2* T;
  int64_t sT;
  int lT;
};

// T[e nq + q] = sum_n w[n, q] a_n[e] (terms in order), QT nodes per thread:
// an element of every a_n is read once for QT matrices written, whole 16-byte
// lanes.  Bound by the writes: 4 x 64 nodes of 256 x 256, 268 MB, 70 us against
// 530 us for the term by term sums and products over the stack.
constexpr int QT = 8;
__global__ __launch_bounds__(NT) void operator_kernel(OperatorArgs g) {
  const int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x;  // element of a matrix
  const int64_t e = blockIdx.z;
  const int q0 = blockIdx.y * QT;
  if (i >= (int64_t)g.d * g.d) return;
  z2 acc[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) acc[u] = make_double2(0.0, 0.0);
  for (int n = 0; n < g.nt; ++n) {
    const z2 a = g.a[n][e * g.s[n] + i];
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const z2 t = cmul(g.w[(int64_t)n * g.nq + min(q0 + u, g.nq - 1)], a);
      acc[u] = make_double2(acc[u].x + t.x, acc[u].y + t.y);
    }
  }
  const int r = (int)(i / g.d), c = (int)(i - (int64_t)r * g.d);
#pragma unroll
  for (int u = 0; u < QT; ++u)
    if (q0 + u < g.nq) g.T[(e * g.nq + q0 + u) * g.sT + (int64_t)r * g.lT + c] = acc[u];
}

struct AccArgs {
  int nq, b;
  const z2* Ti;
  int64_t sT;
  int lT;
  const z2 *w0, *w1;
  z2 *q0, *q1;
  int64_t sq;
  int lq;
};

__global__ __launch_bounds__(NT) void contour_acc_kernel(AccArgs g, int64_t total) {
  const int64_t bb = (int64_t)g.b * g.b;
  for (int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT) {
    const int64_t e = i / bb;
    const int64_t rc = i - e * bb;
    const int r = (int)(rc / g.b), c = (int)(rc - (int64_t)r * g.b);
    z2 s0 = make_double2(0, 0), s1 = make_double2(0, 0);
    for (int q = 0; q < g.nq; ++q) {
      const z2 t = g.Ti[(e * g.nq + q) * g.sT + (int64_t)r * g.lT + c];
      const z2 a = cmul(g.w0[q], t), b = cmul(g.w1[q], t);
      s0.x += a.x;
      s0.y += a.y;
      s1.x += b.x;
      s1.y += b.y;
    }
    z2* p0 = g.q0 + e * g.sq + (int64_t)r * g.lq + c;
    z2* p1 = g.q1 + e * g.sq + (int64_t)r * g.lq + c;
    const z2 o0 = *p0, o1 = *p1;
    *p0 = make_double2(o0.x + s0.x, o0.y + s0.y);
    *p1 = make_double2(o1.x + s1.x, o1.y + s1.y);
  }
}

__global__ void clear_flag_kernel(int* flag) { *flag = 0; }

unsigned grid_for(int64_t total) {
  int64_t b = (total + NT - 1) / NT;
  if (b > 65536 * 4) b = 65536 * 4;
  if (b < 1) b = 1;
  return (unsigned)b;
}

}  // namespace

void ew_axpby(hipStream_t s, int64_t batch, int m, int n, Cplx a, const Mat& A,
              Cplx b, const Mat& B, const Mat& Y) {
  if (batch <= 0 || m <= 0 || n <= 0) return;
  QX_REQUIRE(!Y.zero(), "axpby: null output");
  const bool use_a = !A.zero() && (a.re != 0.0 || a.im != 0.0);
  const bool use_b = !B.zero() && (b.re != 0.0 || b.im != 0.0);
  AxpbyArgs g{m, n, a.re, a.im, b.re, b.im,
              use_a ? A.p : nullptr, A.stride, A.ld,
              use_b ? B.p : nullptr, B.stride, B.ld,
              Y.p, Y.stride, Y.ld};
  const int64_t total = batch * m * (int64_t)n;
  hipLaunchKernelGGL(axpby_kernel, dim3(grid_for(total)), dim3(NT), 0, s, g, total);
  QX_HIP_CHECK(hipGetLastError());
}

void ew_contact_sigma(hipStream_t s, int64_t batch, int n, const Mat& S, const double* f,
                      const Mat& L, const Mat& G) {
  if (batch <= 0 || n <= 0) return;
  QX_REQUIRE(!S.zero() && !L.zero() && !G.zero() && f, "contact_sigma: null argument");
  QX_REQUIRE(S.ld == n && L.ld == n && G.ld == n, "contact_sigma: matrices must be dense n x n");
  const int tn = (n + TS - 1) / TS;
  const int64_t blocks = batch * tn * tn;
  hipLaunchKernelGGL(contact_sigma_kernel, dim3(groups(blocks, NT, "contact_sigma")), dim3(NT), 0, s, S.p, S.stride,
                     n, f, L.p, L.stride, G.p, G.stride, tn);
  QX_HIP_CHECK(hipGetLastError());
}

void ew_diag_imag(hipStream_t s, int64_t batch, int n, const Mat& X, double* out,
                  int64_t out_stride, double scale) {
  if (batch <= 0 || n <= 0) return;
  QX_REQUIRE(!X.zero() && out, "diag_imag: null argument");
  const int64_t total = batch * n;
  hipLaunchKernelGGL(diag_imag_kernel, dim3(grid_for(total)), dim3(NT), 0, s, X.p, X.stride, X.ld,
                     n, out, out_stride, total, scale);
  QX_HIP_CHECK(hipGetLastError());
}

void ew_assemble(hipStream_t s, int64_t batch, int64_t nnz, const z2* z, const z2* S,
                 const z2* T, const z2* Sig, int64_t sSig, z2* A, int64_t sA) {
  if (batch <= 0 || nnz <= 0) return;
  QX_REQUIRE(A && (z || !S), "assemble: null argument");
  constexpr int64_t kMost = int64_t(1) << 28;  // threads of a launch
  for (int64_t k = 0; k < nnz; k += kMost) {
    const int64_t len = std::min(kMost, nnz - k);
    const bool flat = len < kAsmFlat;
    auto launch = [&](auto kernel, int per) {  // energies per thread
      const int64_t rows = std::min<int64_t>(kMost / len, flat ? kMost : 65535);
      for (int64_t e = 0; e < batch; e += rows * per) {
        const int64_t n = std::min(rows * per, batch - e), grp = (n + per - 1) / per;
        const dim3 grid((unsigned)(((flat ? grp * len : len) + NT - 1) / NT),
                        flat ? 1u : (unsigned)grp);
        hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, s, z + (S ? e : 0), S ? S + k : nullptr,
                           T ? T + k : nullptr, Sig ? Sig + e * sSig + k : nullptr, sSig,
                           A + e * sA + k, sA, (unsigned)len, n);
        QX_HIP_CHECK(hipGetLastError());
      }
    };
    if (Sig) launch(assemble_kernel<true, 4>, 4);
    else launch(assemble_kernel<false, 8>, 8);
  }
}

void ew_ident_sub(hipStream_t s, int64_t batch, int n, const Mat& Y) {
  if (batch <= 0 || n <= 0) return;
  QX_REQUIRE(!Y.zero(), "ident_sub: null matrix");
  const int64_t total = batch * n * (int64_t)n;
  hipLaunchKernelGGL(ident_sub_kernel, dim3(grid_for(total)), dim3(NT), 0, s, Y.p, Y.stride, Y.ld,
                     n, total);
  QX_HIP_CHECK(hipGetLastError());
}

void ew_antiherm(hipStream_t s, int64_t batch, int n, double scale,
                 const Mat& X, const Mat& Y) {
  QX_REQUIRE(X.p != Y.p, "antiherm: in-place use is not supported");
  herm(s, batch, n, n, 0.0, scale, X, -scale, X, Y);
}

void ew_antiherm_pair(hipStream_t s, int64_t batch, int n, double scale, const Mat& X0,
                      const Mat& Y0, const Mat& X1, const Mat& Y1) {
  QX_REQUIRE(X0.p != Y0.p && X1.p != Y1.p, "antiherm: in-place use is not supported");
  if (Y0.p == Y1.p || Y0.p == X1.p || Y1.p == X0.p) {
    // one group's output is the other's operand: in order
    ew_antiherm(s, batch, n, scale, X0, Y0);
    ew_antiherm(s, batch, n, scale, X1, Y1);
    return;
  }
  herm(s, batch, n, n, 0.0, scale, X0, -scale, X0, Y0, 0.0, Mat(), &X1, &X1, &Y1);
}

void ew_skew_update(hipStream_t s, int64_t batch, int n, const Mat& X0, const Mat& P0,
                    const Mat& Y0, const Mat* X1, const Mat* P1, const Mat* Y1, double* dens,
                    int64_t dens_stride) {
  if (batch <= 0 || n <= 0) return;
  const bool two = Y1 != nullptr;
  QX_REQUIRE(!X0.zero() && !P0.zero() && !Y0.zero(), "skew_update: null operand");
  QX_REQUIRE(!two || (X1 && P1 && !X1->zero() && !P1->zero() && !Y1->zero()),
             "skew_update: a two-group launch needs all operands");
  const Mat &x1 = two ? *X1 : X0, &p1 = two ? *P1 : P0, &y1 = two ? *Y1 : Y0;
  for (const Mat* y : {&Y0, &y1})
    QX_REQUIRE(y->p != X0.p && y->p != P0.p && y->p != x1.p && y->p != p1.p,
               "skew_update: the output aliases an operand");
  const int tn = (n + TS - 1) / TS;
  SkewArgs g{n, tn, batch, {X0.p, x1.p}, {P0.p, p1.p}, {Y0.p, y1.p},
             {X0.stride, x1.stride}, {P0.stride, p1.stride}, {Y0.stride, y1.stride},
             {X0.ld, x1.ld}, {P0.ld, p1.ld}, {Y0.ld, y1.ld}, dens, dens_stride};
  const int64_t blocks = (two ? 2 : 1) * batch * (tn * (tn + 1) / 2);
  hipLaunchKernelGGL(skew_update_kernel, dim3(groups(blocks, NT, "skew_update")), dim3(NT), 0, s, g);
  QX_HIP_CHECK(hipGetLastError());
}

void skew_check(hipStream_t s, int64_t batch, const std::vector<SkewBlock>& blocks, int* flag) {
  hipLaunchKernelGGL(clear_flag_kernel, dim3(1), dim3(1), 0, s, flag);
  if (batch <= 0) return;
  for (size_t b0 = 0; b0 < blocks.size(); b0 += kSkewBlocks) {
    SkewCheckArgs g;
    g.blocks = (int)std::min<size_t>(kSkewBlocks, blocks.size() - b0);
    for (int k = 0; k < g.blocks; ++k) {
      g.p[k] = blocks[b0 + k].p;
      g.stride[k] = blocks[b0 + k].stride;
      g.n[k] = blocks[b0 + k].n;
    }
    g.flag = flag;
    const int64_t most = max_groups(NT) / kSkewBlocks;  // matrices per launch
    for (int64_t e = 0; e < batch; e += most) {
      const unsigned wgs = (unsigned)(std::min(batch - e, most) * g.blocks);
      hipLaunchKernelGGL(skew_check_kernel, dim3(wgs), dim3(NT), 0, s, g);
      QX_HIP_CHECK(hipGetLastError());
      for (int k = 0; k < g.blocks; ++k) g.p[k] += most * g.stride[k];
    }
  }
}

void ew_herm_add(hipStream_t s, int64_t batch, int n, const Mat& D, double scale,
                 const Mat& X, const Mat& Y) {
  QX_REQUIRE(X.p != Y.p, "herm_add: Y must not alias X");
  herm(s, batch, n, n, 0.0, scale, X, -scale, X, Y, 1.0, D);
}

void ew_add_hdiff(hipStream_t s, int64_t batch, int n, const Mat& T,
                  const Mat& Y) {
  QX_REQUIRE(T.p != Y.p, "add_hdiff: in-place use is not supported");
  herm(s, batch, n, n, 1.0, -1.0, T, 1.0, T, Y);
}

void ew_neg_h(hipStream_t s, int64_t batch, int m, int n, const Mat& X,
              const Mat& Y) {
  // X is m x n, Y = -X^H is n x m.
  QX_REQUIRE(X.p != Y.p, "neg_h: in-place use is not supported");
  herm(s, batch, n, m, 0.0, 0.0, Mat(), -1.0, X, Y);
}

void trace_diff(hipStream_t s, int64_t batch, int n, const Mat& X, const Mat& Y,
                const Mat& Z, const Mat& W, z2* out, int64_t out_stride, const Mat& part) {
  if (batch <= 0) return;
  const int tn = (n + TS - 1) / TS;
  QX_REQUIRE(!part.zero() && part.stride >= tn, "trace_diff: scratch too small");
  TraceArgs g{n, X.p, Y.p, Z.p, W.p, X.stride, Y.stride, Z.stride, W.stride,
              X.ld, Y.ld, Z.ld, W.ld, out, out_stride};
  if (X.zero() || Y.zero()) g.X = nullptr;
  if (Z.zero() || W.zero()) g.Z = nullptr;
  hipLaunchKernelGGL(trace_kernel, dim3(groups(batch * tn, NT, "trace_diff")), dim3(NT), 0, s, g,
                     tn, part.p, part.stride);
  hipLaunchKernelGGL(trace_sum_kernel, dim3((unsigned)((batch + NT - 1) / NT)), dim3(NT), 0, s,
                     part.p, part.stride, tn, out, out_stride, batch);
  QX_HIP_CHECK(hipGetLastError());
}

void absnorm2(hipStream_t s, int64_t batch, int n, const Mat& A, const Mat& B,
              double* out) {
  if (batch <= 0) return;
  for (int64_t e = 0; e < batch; e += max_groups(NTN)) {
    const unsigned wgs = (unsigned)std::min(batch - e, max_groups(NTN));
    hipLaunchKernelGGL(absnorm_kernel, dim3(wgs), dim3(NTN), 0, s, n, A.p + e * A.stride, A.stride,
                       A.ld, B.p + e * B.stride, B.stride, B.ld, out + e);
    QX_HIP_CHECK(hipGetLastError());
  }
}

void max_value(hipStream_t s, int64_t n, const double* v, double* out) {
  QX_REQUIRE(n > 0 && v && out, "max_value: nothing to compare");
  hipLaunchKernelGGL(max_kernel, dim3(1), dim3(NT), 0, s, n, v, out);
  QX_HIP_CHECK(hipGetLastError());
}

void ew_ns_check(hipStream_t s, int64_t batch, int n, const Mat& R, double tol, int* flagged,
                 int* info) {
  if (batch <= 0) return;
  hipLaunchKernelGGL(ns_check_kernel, dim3(groups(batch, NT, "ns_check")), dim3(NT), 0, s, n, R.p, R.stride,
                     R.ld, tol, flagged, info);
  QX_HIP_CHECK(hipGetLastError());
}

void contour_operator(hipStream_t s, int64_t batch, int nq, int b,
                      const Mat& aji, const Mat& aii, const Mat& aij,
                      const z2* z, const Mat& T) {
  ContourArgs g{nq, b, aji.p, aii.p, aij.p, aji.stride, aii.stride, aij.stride,
                aji.ld, aii.ld, aij.ld, z, T.p, T.stride, T.ld};
  const int64_t total = batch * nq * (int64_t)b * b;
  if (total <= 0) return;
  hipLaunchKernelGGL(contour_kernel, dim3(grid_for(total)), dim3(NT), 0, s, g, total);
  QX_HIP_CHECK(hipGetLastError());
}

void operator_stack(hipStream_t s, int64_t batch, int nq, int d, int nt, const void* const* a,
                    const int64_t* stride, const void* w, const Mat& T) {
  QX_REQUIRE(nt >= 1 && nt <= kOperatorTerms, "operator: between 1 and 8 terms");
  OperatorArgs g;
  g.nq = nq;
  g.d = d;
  g.nt = nt;
  for (int n = 0; n < kOperatorTerms; ++n) {
    g.a[n] = static_cast<const z2*>(a[n < nt ? n : 0]);
    g.s[n] = stride[n < nt ? n : 0];
    QX_REQUIRE(g.a[n], "operator: null term");
  }
  g.w = static_cast<const z2*>(w);
  g.T = T.p;
  g.sT = T.stride;
  g.lT = T.ld;
  const int64_t tiles = ((int64_t)d * d + NT - 1) / NT;
  const int rows = (nq + QT - 1) / QT;
  QX_REQUIRE(rows <= 65535, "operator: too many nodes");
  for (int64_t e0 = 0; e0 < batch; e0 += 65535) {  // grid limit in z
    const int64_t m = std::min<int64_t>(65535, batch - e0);
    hipLaunchKernelGGL(operator_kernel, dim3((unsigned)tiles, (unsigned)rows, (unsigned)m),
                       dim3(NT), 0, s, g);
    QX_HIP_CHECK(hipGetLastError());
    for (int n = 0; n < kOperatorTerms; ++n) g.a[n] += m * g.s[n];
    g.T += m * nq * g.sT;
  }
}

void contour_accumulate(hipStream_t s, int64_t batch, int nq, int b,
                        const Mat& Tinv, const z2* w0, const z2* w1,
                        const Mat& q0, const Mat& q1) {
  AccArgs g{nq, b, Tinv.p, Tinv.stride, Tinv.ld, w0, w1, q0.p, q1.p, q0.stride, q0.ld};
  QX_REQUIRE(q0.stride == q1.stride && q0.ld == q1.ld, "contour: q0/q1 layouts differ");
  const int64_t total = batch * (int64_t)b * b;
  if (total <= 0) return;
  hipLaunchKernelGGL(contour_acc_kernel, dim3(grid_for(total)), dim3(NT), 0, s, g, total);
  QX_HIP_CHECK(hipGetLastError());
}

}  // namespace qx
