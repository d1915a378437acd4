// Gauss-Jordan inverse of a matrix held in MFMA result registers (gfx950,
// double precision), for the batched inverse up to 128 and the fused
// small-block solves.
//
// A workgroup of one factoring wave (wave 0) and MW update waves holds a matrix
// of up to 16 RT MW rows and 16 CT columns: update wave u the rows
// 16 RT u .. in RT x CT tiles of the v_mfma_f64_16x16x4_f64 result layout.
// The columns are eliminated in sub-panels of SB = 4 or 8:
//   - the sub-panel's columns go to LDS and the factoring wave eliminates
//     them alone, RL rows per lane, with partial pivoting: no barrier and no
//     LDS round trip inside a column, the pivot row reaches the other lanes by
//     v_readlane (gj_factor);
//   - the pivot rows go to LDS and the update waves apply the rank-SB update
//     on the matrix cores.  The update does not overlap the factorisation: FP64
//     vector instructions wait for every FP64 matrix instruction issued on
//     their SIMD (64 cycles each).
// Rows never move: the row interchanges are tracked as positions.
//
// Why one wave per matrix: a column is a serial chain (pivot search, exchange
// of the pivot row, reciprocal, elimination) of about 110 instructions at one
// row per lane, each 4 cycles of issue.  Eight waves that share the columns
// repeat the exchange in every wave (1850 to 2700 cycles per column at 256
// rows, the owner of the next column one ahead); four waves that share the
// rows pay two dependent LDS round trips and a barrier per column (1600
// cycles).
#pragma once

#include "qx_internal.h"

namespace qx {
namespace {

typedef double gj_acc __attribute__((ext_vector_type(4)));

// Wave-wide unsigned max with DPP only: quad and row butterflies give every
// lane its row's maximum, row_bcast:15 / row_bcast:31 carry the row maxima
// up to lane 63, which is read once.  Every lane of the wave must be active.
__device__ inline unsigned gj_wave_max(unsigned v) {
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false));   // quad xor 1
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false));   // quad xor 2
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false));  // row_ror 4
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false));  // row_ror 8
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Value of v in lane l of the wave (l uniform).
__device__ __forceinline__ double gj_lane_read(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float gj_lane_read(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// MW update waves of RT x CT tiles, RL rows per lane of the factoring wave,
// sub-panels of SB columns.
template <int MW_, int RT_, int CT_, int RL_, int SB_>
struct GjShape {
  static constexpr int MW = MW_, RT = RT_, CT = CT_, RL = RL_, SB = SB_;
  static constexpr int R = 16 * RT * MW, C = 16 * CT;  // rows and columns held
  static constexpr int RF = 64 * RL;                   // rows of the factoring wave
  // column stride: a multiple of 16 rows plus 4, so that the columns of a tile
  // row fall into different LDS banks
  static constexpr int LS = (RF > R ? RF : R) + 4;
  static constexpr int THREADS = 64 * (MW + 1);
};

// Whether products are summed before they are subtracted from the matrix, one
// rounding of the matrix's size per column in the factoring wave and per
// sub-panel in the update, or fused into it, two per column.  Error against the
// kernels before this one, which summed up to 32 rows and fused above; geometric
// means over 400 to 2000 matrices (+- 0.01 to 0.02):
//            fused           update summed   both summed
//   n = 20   1.16            1.06            1.02
//   n = 32   1.15 to 1.20    1.07            1.03 to 1.04
//   n = 48   1.02 to 1.04    0.90 to 0.93
//   n = 64   0.99 to 1.05    0.89 to 0.92
//   n = 128  0.78 to 0.84
// (What is left at 32 are the sub-panels' composite coefficients.)  Up to 32 the
// sums cost 0 to 2 % of an inverse (256 x 32^2 20.7 -> 21.3 us; a solve of 16
// energies, 8 blocks of 32 533 -> 540); at 64 the registers of the update's halve
// the workgroups of a CU (4096 x 64^2 551 -> 751 us).
template <typename G>
constexpr bool kSums = G::CT <= 2;

template <typename G>
struct GjShared {
  z2 sub[2][G::SB][G::LS];  // sub-panel columns, alternating buffers
  z2 prow[G::SB][G::C];     // pivot rows, the B operand of the update
  z2 rcp[G::SB];            // pivot reciprocals of a sub-panel
  int step_of[G::LS];       // sub-panel step of a pivot row, or -1
  int piv[G::C];            // pivot row of a column
  int pos[G::LS];           // final position of a row
};

// One wave factors columns [0, ns) of the sub-panel sub, the columns k, k + 1,
// ... of the matrix: the pivot of column k + c is the row of largest |re| + |im| (pivot_key) among the rows at positions >=
// k + c.  pos[j]: the position of row lane + 64 j, -1 for the rows >= n.
// The scaling of a pivot row by its reciprocal is deferred to the end of the
// sub-panel (its multiplier is taken as zero and its active entry as 1; the
// later steps act on it linearly).  On return sub holds the reduced columns
// and step_of the pivot rows' steps.
template <typename G>
__device__ __forceinline__ void gj_factor(GjShared<G>& sh, z2 (*sub)[G::LS], int n, int k,
                                          int ns, int (&pos)[G::RL], int* info) {
  constexpr int RL = G::RL, SB = G::SB;
  const int lane = threadIdx.x & 63;
  double xr[RL][SB], xi[RL][SB];
#pragma unroll
  for (int j = 0; j < RL; ++j)
#pragma unroll
    for (int c = 0; c < SB; ++c) {
      const z2 v = sub[c][lane + 64 * j];
      xr[j][c] = v.x;
      xi[j][c] = v.y;
    }
  unsigned kmin = 0xFFFFFFFFu;  // smallest pivot key of the sub-panel
#pragma unroll
  for (int c = 0; c < SB; ++c) {
    if (c < ns) {  // uniform
      unsigned key = 0;
#pragma unroll
      for (int j = 0; j < RL; ++j) {
        const unsigned kj = pivot_key(xr[j][c], xi[j][c], lane + 64 * j);
        key = max(key, pos[j] >= k + c ? kj : 0u);
      }
      const unsigned kmax = gj_wave_max(key);
      kmin = min(kmin, kmax);
      // a candidate always exists (n - k - c rows), so p < n; min() keeps
      // every index inside the panel whatever the key holds
      const int p = min(511 - (int)(kmax & 0x1FFu), n - 1);
      const int pl = p & 63, pj = p >> 6;
      const bool prow = lane == pl;  // and row slot pj
      double ar[SB], ai[SB];
      int q = 0;
#pragma unroll
      for (int u = 0; u < SB; ++u) ar[u] = ai[u] = 0.0;
#pragma unroll
      for (int j = 0; j < RL; ++j) {
        if (RL == 1 || j == pj) {  // uniform
#pragma unroll
          for (int u = 0; u < SB; ++u) {
            ar[u] = gj_lane_read(xr[j][u], pl);
            ai[u] = gj_lane_read(xi[j][u], pl);
          }
          q = __builtin_amdgcn_readlane(pos[j], pl);
          // zero multiplier for the pivot row
          xr[j][c] = prow ? 0.0 : xr[j][c];
          xi[j][c] = prow ? 0.0 : xi[j][c];
        }
      }
      double vr, vi;
      complex_recip(ar[c], ai[c], vr, vi);
      if (lane == 0) {
        sh.rcp[c] = make_double2(vr, vi);
        sh.piv[k + c] = p;
      }
#pragma unroll
      for (int j = 0; j < RL; ++j) {
        const double mr = fma(xr[j][c], vr, -(xi[j][c] * vi));
        const double mi = fma(xr[j][c], vi, xi[j][c] * vr);
#pragma unroll
        for (int u = 0; u < SB; ++u) {
          if (u == c) {
            xr[j][u] = -mr;
            xi[j][u] = -mi;
          } else {
            if constexpr (kSums<G>) {
              xr[j][u] -= fma(mr, ar[u], -(mi * ai[u]));
              xi[j][u] -= fma(mr, ai[u], mi * ar[u]);
            } else {
              xr[j][u] = fma(-mr, ar[u], fma(mi, ai[u], xr[j][u]));
              xi[j][u] = fma(-mr, ai[u], fma(-mi, ar[u], xi[j][u]));
            }
          }
        }
        // interchange k + c <-> q: row p moves to position k + c
        pos[j] = pos[j] == k + c ? q : pos[j];
      }
#pragma unroll
      for (int j = 0; j < RL; ++j) {
        if (RL == 1 || j == pj) {  // uniform
          xr[j][c] = prow ? 1.0 : xr[j][c];
          pos[j] = prow ? k + c : pos[j];
        }
      }
    }
  }
  // the reciprocals were written by this wave, in program order
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int j = 0; j < RL; ++j) {
    const int st = pos[j] - k;
    const bool pivot = st >= 0 && st < ns;
    if (pivot) {
      const z2 s = sh.rcp[st];
#pragma unroll
      for (int u = 0; u < SB; ++u) {
        const double a = xr[j][u], b = xi[j][u];
        xr[j][u] = fma(a, s.x, -(b * s.y));
        xi[j][u] = fma(a, s.y, b * s.x);
      }
    }
#pragma unroll
    for (int u = 0; u < SB; ++u) sub[u][lane + 64 * j] = make_double2(xr[j][u], xi[j][u]);
    sh.step_of[lane + 64 * j] = pivot ? st : -1;
  }
  if (lane == 0 && (kmin >> 9) == 0u) *info = 1;  // no nonzero pivot: singular
}

// Update waves: the rank-SB update by sub-panel `sub` of the column tile that
// starts at panel column col.
//
// kSums: the rank-SB sum is formed from zero and then added.
template <typename G>
__device__ __forceinline__ void gj_update(const GjShared<G>& sh, const z2 (*sub)[G::LS], int row0,
                                          int l16, int l4, int col, gj_acc (&cr)[G::RT],
                                          gj_acc (&ci)[G::RT]) {
  constexpr bool SUM = kSums<G>;
  gj_acc sr[G::RT], si[G::RT];
#pragma unroll
  for (int i = 0; i < G::RT; ++i) {
    sr[i] = SUM ? gj_acc{0.0, 0.0, 0.0, 0.0} : cr[i];
    si[i] = SUM ? gj_acc{0.0, 0.0, 0.0, 0.0} : ci[i];
  }
#pragma unroll
  for (int ks = 0; ks < G::SB / 4; ++ks) {
    __builtin_amdgcn_sched_barrier(0);  // operands of one k-step at a time: registers
    const z2 b = sh.prow[4 * ks + l4][col + l16];
    z2 a[G::RT];
#pragma unroll
    for (int i = 0; i < G::RT; ++i) a[i] = sub[4 * ks + l4][row0 + 16 * i + l16];
#pragma unroll
    for (int i = 0; i < G::RT; ++i) {
      sr[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b.x, sr[i], 0, 0, 0);
      si[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b.y, si[i], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < G::RT; ++i) {
      sr[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b.y, sr[i], 0, 0, 1);
      si[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b.x, si[i], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < G::RT; ++i) {
    cr[i] = SUM ? cr[i] + sr[i] : sr[i];
    ci[i] = SUM ? ci[i] + si[i] : si[i];
  }
}

// Eliminates the n columns; called by the factoring wave.  Passes the workgroup
// barriers of gj_update_waves.
template <typename G>
__device__ __forceinline__ void gj_factor_wave(GjShared<G>& sh, int n, int* info) {
  const int lane = threadIdx.x & 63;
  const int nsub = (n + G::SB - 1) / G::SB;
  int pos[G::RL];
#pragma unroll
  for (int j = 0; j < G::RL; ++j) pos[j] = lane + 64 * j < n ? lane + 64 * j : -1;
  for (int r = G::RF + lane; r < G::LS; r += 64) sh.step_of[r] = -1;  // rows beyond the wave's
  __builtin_amdgcn_s_setprio(3);
#pragma unroll 1
  for (int s = 0; s < nsub; ++s) {
    __syncthreads();  // the sub-panel's columns are in LDS
    gj_factor<G>(sh, sh.sub[s & 1], n, s * G::SB, min(G::SB, n - s * G::SB), pos, info);
    __syncthreads();  // the reduced sub-panel is in LDS
    __syncthreads();  // the pivot rows are in LDS
  }
  __builtin_amdgcn_s_setprio(0);
#pragma unroll
  for (int j = 0; j < G::RL; ++j) sh.pos[lane + 64 * j] = pos[j];
  __syncthreads();
}

// The same for update wave u: acr / aci hold its rows of the matrix (rows and
// columns >= n zero).  Ends with a barrier after which sh.piv and sh.pos are
// complete.
//
// The loop over the sub-panels stays rolled: unrolled, the code outgrows the
// instruction cache (128 rows: 185 -> 705 us).  Accumulators are therefore
// never selected by a branch on the run-time tile, which makes the compiler
// copy and spill them: every tile takes part in the update, and the tile of
// the sub-panel's own columns is picked by lane selects.
template <typename G>
__device__ __forceinline__ void gj_update_waves(GjShared<G>& sh, int u,
                                                gj_acc (&acr)[G::CT][G::RT],
                                                gj_acc (&aci)[G::CT][G::RT], int n) {
  constexpr int RT = G::RT, CT = G::CT, SB = G::SB;
  const int lane = threadIdx.x & 63, l16 = lane & 15, l4 = lane >> 4;
  const int row0 = 16 * RT * u;
  const int nsub = (n + SB - 1) / SB;
  // the columns of sub-panel s of the own rows to LDS
  auto extract = [&](int s) {
    auto* sub = sh.sub[s & 1];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const int c = 16 * t + l16 - SB * s;
      if (c >= 0 && c < SB) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sub[c][row0 + 16 * i + 4 * e + l4] = make_double2(acr[t][i][e], aci[t][i][e]);
      }
    }
  };
  extract(0);
#pragma unroll 1
  for (int s = 0; s < nsub; ++s) {
    __syncthreads();  // the sub-panel's columns are in LDS
    __syncthreads();  // the reduced sub-panel is in LDS
    // pivot rows to LDS and out of the accumulators; the sub-panel's own
    // columns are replaced by the reduced ones (zero accumulator, identity in
    // the B operand)
    const int c0 = s * SB, ns = min(SB, n - c0);
    int st[RT][4];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) st[i][e] = sh.step_of[row0 + 16 * i + 4 * e + l4];
    if (ns < SB)  // the missing steps' rows of the B operand
      for (int k = threadIdx.x - 64; k < (SB - ns) * G::C; k += 64 * G::MW)
        sh.prow[ns + k / G::C][k % G::C] = make_double2(0.0, 0.0);
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const int c = 16 * t + l16 - c0;
      const bool own = c >= 0 && c < ns;
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acr[t][i][e] = own ? 0.0 : acr[t][i][e];
          aci[t][i][e] = own ? 0.0 : aci[t][i][e];
        }
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = st[i][e];
        if (__builtin_amdgcn_ballot_w64(c >= 0) != 0) {  // few tile rows hold a pivot
          if (c >= 0) {
#pragma unroll
            for (int t = 0; t < CT; ++t) {
              z2 v = make_double2(acr[t][i][e], aci[t][i][e]);
              if (16 * t + l16 == c0 + c) v.x = 1.0;
              sh.prow[c][16 * t + l16] = v;
            }
          }
#pragma unroll
          for (int t = 0; t < CT; ++t) {
            acr[t][i][e] = c >= 0 ? 0.0 : acr[t][i][e];
            aci[t][i][e] = c >= 0 ? 0.0 : aci[t][i][e];
          }
        }
      }
    __syncthreads();  // the pivot rows are in LDS
#pragma unroll
    for (int t = 0; t < CT; ++t)
      gj_update<G>(sh, sh.sub[s & 1], row0, l16, l4, 16 * t, acr[t], aci[t]);
    if (s + 1 < nsub) extract(s + 1);
  }
  __syncthreads();
}

// X = (A - S)^-1 (S may be null, X may alias A) of an n x n matrix, n <= G::C,
// by the first G::THREADS threads of a workgroup; further waves only pass the
// barriers.  The matrix stays in MFMA result registers from the load to the
// store.  Rows never move: with p_j the pivot row of column j, the reduced row
// p_j is row j of the inverse and its column j is column p_j.  The stores are
// not followed by a barrier.
template <typename G>
__device__ __forceinline__ void gj_invert(int n, const z2* A, int lda, const z2* S, int lds, z2* X,
                                          int ldx, int* info, GjShared<G>& sh) {
  static_assert(G::R >= G::C && G::RF >= G::C, "rows cover the columns");
  constexpr int RT = G::RT, CT = G::CT;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w == 0) {
    gj_factor_wave<G>(sh, n, info);
  } else if (w <= G::MW) {
    const int l16 = lane & 15, l4 = lane >> 4, row0 = 16 * RT * (w - 1);
    gj_acc acr[CT][RT], aci[CT][RT];
    // unconditional loads from clamped addresses; one tile after the other,
    // so that the loads in flight do not push the accumulators out
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      if (CT > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = row0 + 16 * i + 4 * q + l4, c = 16 * t + l16;
          const bool ok = r < n && c < n;
          const z2 v = A[ok ? (int64_t)r * lda + c : 0];
          acr[t][i][q] = ok ? v.x : 0.0;
          aci[t][i][q] = ok ? v.y : 0.0;
        }
      if (S) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int r = row0 + 16 * i + 4 * q + l4, c = 16 * t + l16;
            const bool ok = r < n && c < n;
            const z2 v = S[ok ? (int64_t)r * lds + c : 0];
            acr[t][i][q] -= ok ? v.x : 0.0;
            aci[t][i][q] -= ok ? v.y : 0.0;
          }
      }
    }
    gj_update_waves<G>(sh, w - 1, acr, aci, n);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = row0 + 16 * i + 4 * q + l4;
        if (r < n) {
          z2* out = X + (int64_t)sh.pos[r] * ldx;
#pragma unroll
          for (int t = 0; t < CT; ++t)
            if (16 * t + l16 < n)
              out[sh.piv[16 * t + l16]] = make_double2(acr[t][i][q], aci[t][i][q]);
        }
      }
  } else {
    const int nb = 3 * ((n + G::SB - 1) / G::SB) + 1;
    for (int s = 0; s < nb; ++s) __syncthreads();
  }
}

// Shape of a whole matrix of up to 32 rows (used by the batched inverse and by
// the fused small-block solves, which therefore give the same bits).
typedef GjShape<2, 1, 2, 1, 8> GjWhole32;

}  // namespace
}  // namespace qx
