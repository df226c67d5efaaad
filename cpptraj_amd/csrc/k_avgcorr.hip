// k_avgcorr.hip -- RMS average correlation ('rmsavgcorr').
//
//   k_avgcorr  Analysis_RmsAvgCorr::Analyze (src/Analysis_RmsAvgCorr.cpp:
//              119-276): for one window size per wavefront, the running sum
//              of the selected atoms over the last `w` frames (Frame
//              operator+= / operator-=, FP64, in the reference's order),
//              divided by w (Frame::Divide), fitted to the reference
//              (Frame::RMSD_CenteredRef); mean and standard deviation of the
//              RMSD over the F - w + 1 averaged frames.  The reference is the
//              centred reference frame, or ('first') the window's first
//              averaged frame, centred.
//
// The running sum lives in LDS ([3][nsel] FP64), and so does the reference
// in 'first' mode (a fixed reference is read from global memory: the same
// for every window, it stays in cache).  The fit is the one of the
// frame-to-reference path: single-pass moments of the averaged frame shifted
// by its first atom against the centred reference, one wave reduction, then
// FP64 QCP.  The QCP solves leave the frame loop's critical path: lane
// (step mod 64) keeps that step's reduced moments, and every 64 steps all
// lanes solve their own step at once.  The mean and SD then sum the RMSDs in
// lane order instead of frame order (a difference in the last bits).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "rmsd_device.hpp"
#include "rmsd_kernels.hpp"

namespace {

constexpr int AVG_THREADS = 64;

__device__ __forceinline__ float coord(const FrameSetDev& fs, int64_t f, int k, int c) {
  const int a = fs.sel ? fs.sel[k] : k;
  const float* fr = fs.xyz + frame_of(fs, f) * fs.stride;
  return fs.ld ? fr[c * fs.ld + a] : fr[3 * a + c];
}

// Value j of the 13 moments, summed over the wave, on every lane (read from
// lane 4 j into scalar registers).
__device__ __forceinline__ void wave_moments(const double (&v)[13], double (&out)[13]) {
  double p[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) p[i] = i < 13 ? v[i] : 0.0;
  const double r = rmsd_dev::wave_reduce16(p);  // lane l: total of value l >> 2
  const unsigned long long bits = (unsigned long long)__double_as_longlong(r);
  const unsigned lo = (unsigned)bits, hi = (unsigned)(bits >> 32);
#pragma unroll
  for (int i = 0; i < 13; ++i) {
    const unsigned long long b =
        ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)hi, 4 * i) << 32) |
        (unsigned)__builtin_amdgcn_readlane((int)lo, 4 * i);
    out[i] = __longlong_as_double((long long)b);
  }
}

template <bool FIRST, bool WEIGHTED>
__global__ __launch_bounds__(AVG_THREADS) void k_avgcorr(AvgCorrArgs a) {
  extern __shared__ double lds[];
  const int n = a.fs.nsel;
  const int lane = threadIdx.x;
  const int wi = blockIdx.x;
  const int w = a.windows[wi];
  const double dw = (double)w;
  double* S = lds;  // running sum [3][n]
  // centred reference: LDS in 'first' mode, else the prepared reference
  double* Yl = lds + 3 * n;
  const double* Y = FIRST ? Yl : a.ref;
  const int ly = FIRST ? n : a.ldr;
  for (int k = lane; k < n; k += AVG_THREADS)
    for (int c = 0; c < 3; ++c) S[c * n + k] = 0.0;
  // Reference constants: sum w y (3), sum w |y|^2, W (sequential, as the
  // reference's running total).
  double K[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (!FIRST)
    for (int i = 0; i < 5; ++i) K[i] = a.consts[i];
  double W = 0.0;
  if (WEIGHTED) {
    for (int k = 0; k < n; ++k) W += a.mass[k];
  } else {
    W = (double)n;
  }
  __syncthreads();
  bool need_ref = FIRST;
  double sum_r = 0.0, sum_r2 = 0.0;
  // Deferred solves: lane j holds the moments of pending step j (and the
  // reference constants they go with).
  double pm[13], pK[4];
  int npend = 0;
  auto solve_pending = [&]() {
    if (lane < npend) {
      double r;
      if (W < RMSD_SMALL) {
        r = -1.0;
      } else {
        const double c0 = pm[0] / W, c1 = pm[1] / W, c2 = pm[2] / W;
        double R[9];
        R[0] = pm[3] - c0 * pK[0]; R[1] = pm[4] - c0 * pK[1]; R[2] = pm[5] - c0 * pK[2];
        R[3] = pm[6] - c1 * pK[0]; R[4] = pm[7] - c1 * pK[1]; R[5] = pm[8] - c1 * pK[2];
        R[6] = pm[9] - c2 * pK[0]; R[7] = pm[10] - c2 * pK[1]; R[8] = pm[11] - c2 * pK[2];
        const double sx = pm[12] - W * (c0 * c0 + c1 * c1 + c2 * c2);
        const double E0 = 0.5 * (sx + pK[3]);
        r = rmsd_dev::qcp_rmsd(R, E0, W, 1);
      }
      sum_r += r;
      sum_r2 += r * r;
    }
    npend = 0;
  };
  int64_t sub = 0;
  for (int64_t t = 0; t < a.fs.nframes; ++t) {
    for (int k = lane; k < n; k += AVG_THREADS)
      for (int c = 0; c < 3; ++c) S[c * n + k] += (double)coord(a.fs, t, k, c);
    __syncthreads();
    if (t > w - 2) {
      if (FIRST && need_ref) {
        // The first averaged frame, centred (Frame::CenterOnOrigin): the
        // window's reference.
        double v[4] = {0.0, 0.0, 0.0, 0.0};
        for (int k = lane; k < n; k += AVG_THREADS) {
          const double m = WEIGHTED ? a.mass[k] : 1.0;
          for (int c = 0; c < 3; ++c) v[c] += WEIGHTED ? (S[c * n + k] / dw) * m : S[c * n + k] / dw;
          v[3] += m;
        }
        for (int i = 0; i < 4; ++i) v[i] = rmsd_dev::wave_sum(v[i]);
        double cen[3] = {0.0, 0.0, 0.0};
        const double tot = WEIGHTED ? v[3] : (double)n;
        if (tot != 0.0)
          for (int c = 0; c < 3; ++c) cen[c] = v[c] / tot;
        double h[4] = {0.0, 0.0, 0.0, 0.0};
        for (int k = lane; k < n; k += AVG_THREADS) {
          double y[3];
          for (int c = 0; c < 3; ++c) {
            y[c] = S[c * n + k] / dw - cen[c];
            Yl[c * n + k] = y[c];
          }
          const double m = WEIGHTED ? a.mass[k] : 1.0;
          h[0] += m * y[0];
          h[1] += m * y[1];
          h[2] += m * y[2];
          h[3] += m * (y[0] * y[0] + y[1] * y[1] + y[2] * y[2]);
        }
        for (int i = 0; i < 4; ++i) K[i] = rmsd_dev::wave_sum(h[i]);
        K[4] = W;
        need_ref = false;
        __syncthreads();
      }
      // Moments of the averaged frame (shifted by its first atom) against the
      // reference, then the fit of the frame-to-reference path.
      const double s0 = S[0] / dw, s1 = S[n] / dw, s2 = S[2 * n] / dw;
      double v[13];
#pragma unroll
      for (int i = 0; i < 13; ++i) v[i] = 0.0;
      for (int k = lane; k < n; k += AVG_THREADS) {
        const double x0 = S[k] / dw - s0, x1 = S[n + k] / dw - s1, x2 = S[2 * n + k] / dw - s2;
        const double y0 = Y[k], y1 = Y[ly + k], y2 = Y[2 * ly + k];
        double wx0 = x0, wx1 = x1, wx2 = x2;
        if (WEIGHTED) {
          const double m = a.mass[k];
          wx0 = m * x0;
          wx1 = m * x1;
          wx2 = m * x2;
        }
        v[0] += wx0;
        v[1] += wx1;
        v[2] += wx2;
        v[3] += wx0 * y0; v[4] += wx0 * y1; v[5] += wx0 * y2;
        v[6] += wx1 * y0; v[7] += wx1 * y1; v[8] += wx1 * y2;
        v[9] += wx2 * y0; v[10] += wx2 * y1; v[11] += wx2 * y2;
        v[12] += wx0 * x0 + wx1 * x1 + wx2 * x2;
      }
      double m[13];
      wave_moments(v, m);
      if (lane == npend) {
#pragma unroll
        for (int i = 0; i < 13; ++i) pm[i] = m[i];
#pragma unroll
        for (int i = 0; i < 4; ++i) pK[i] = K[i];
      }
      if (++npend == AVG_THREADS) solve_pending();
      // Drop the oldest frame of the window.
      for (int k = lane; k < n; k += AVG_THREADS)
        for (int c = 0; c < 3; ++c) S[c * n + k] -= (double)coord(a.fs, sub, k, c);
      ++sub;
      __syncthreads();
    }
  }
  solve_pending();
  sum_r = rmsd_dev::wave_sum(sum_r);
  sum_r2 = rmsd_dev::wave_sum(sum_r2);
  if (lane == 0) {
    const double d = 1.0 / ((double)a.fs.nframes - dw + 1.0);
    const double avg = sum_r * d;
    double sd = sum_r2 * d;
    sd -= avg * avg;
    a.ct[wi] = avg;
    a.sd[wi] = sd > 0.0 ? sqrt(sd) : 0.0;
  }
}

}  // namespace

hipError_t rmsd_launch_avgcorr(const AvgCorrArgs& a, bool first, hipStream_t s) {
  if (a.nwin == 0) return hipSuccess;
  const size_t lds = sizeof(double) * (first ? 6 : 3) * (size_t)a.fs.nsel;
  if (lds > AVGCORR_LDS_MAX) return hipErrorInvalidValue;
  const bool wt = a.mass != nullptr;
  const void* fn = first ? (wt ? reinterpret_cast<const void*>(&k_avgcorr<true, true>)
                               : reinterpret_cast<const void*>(&k_avgcorr<true, false>))
                         : (wt ? reinterpret_cast<const void*>(&k_avgcorr<false, true>)
                               : reinterpret_cast<const void*>(&k_avgcorr<false, false>));
  hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  void* args[] = {const_cast<AvgCorrArgs*>(&a)};
  return hipLaunchKernel(fn, dim3(a.nwin), dim3(AVG_THREADS), args, lds, s);
}

// ---- prefix-sum form (fixed reference) --------------------------------------------
// With the selected coordinates x_f and their per-coordinate mean mu, the
// prefix sums P_i = sum_{f < i} (x_f - mu) (i = 0..F, P_0 = 0) give the
// window-w average ending at frame t (i = t + 1, j = i - w) as
// a = (P_i - P_j) / w + mu.  The rows lose their centroids, P~_i = P_i - C_i / W
// with C_i = sum m P_i, so that where molecules diffuse or jump no common
// translation has to cancel later.  With d = P~_i - P~_j, v = mu - mu_c (mu_c
// the weighted centroid of mu) and the fit centroid c:
//   sum m (a - c) y^T = (Q_i - Q_j) / w + sum m v y^T
//   sum m |a - c|^2   = sum m |d|^2 / w^2 + 2 (L_i - L_j) / w + sum m |v|^2
// with per-prefix moments Q_i = sum m P~_i y^T and L_i = sum m v . P~_i ('first'
// keeps P_i and C_i: its references move too).  Only sum m |d|^2 needs all
// coordinates of a pair: it is a squared distance between two prefix rows, in
// 64 x 64 tiles of (i, j) pairs.  Each tile fits the pairs whose i - j is a
// window size and sums their RMSDs per diagonal; a last pass adds the per-tile
// sums of every window in a fixed order.  Subtracting mu first keeps the prefix
// sums, and the digits their differences lose, small.
namespace {

constexpr int AC_CHUNK = 128;  // frames per scan chunk
constexpr int AC_THREADS = 256;
constexpr int AC_TILE = 64;    // prefix rows per tile side
constexpr int AC_KC = 32;      // coordinates per LDS stage
constexpr int AC_LD = AC_TILE + 1;
constexpr int AC_XCDS = 8;

__global__ __launch_bounds__(AC_THREADS) void k_ac_chunksum(AvgPrefixArgs a) {
  const int j = blockIdx.x * AC_THREADS + threadIdx.x;
  const int q = blockIdx.y;
  if (j >= a.k) return;
  const int kk = j / 3, c = j - 3 * kk;
  const int64_t f0 = (int64_t)q * AC_CHUNK;
  const int64_t f1 = f0 + AC_CHUNK < a.fs.nframes ? f0 + AC_CHUNK : a.fs.nframes;
  double s = 0.0;
  for (int64_t f = f0; f < f1; ++f) s += (double)coord(a.fs, f, kk, c);
  a.chunk[(int64_t)q * a.k + j] = s;
}

// Coordinate means, and the chunk sums turned into exclusive prefix sums of
// the mean-subtracted coordinates.
__global__ __launch_bounds__(AC_THREADS) void k_ac_scan(AvgPrefixArgs a) {
  const int j = blockIdx.x * AC_THREADS + threadIdx.x;
  if (j >= a.k) return;
  const int nq = (int)((a.fs.nframes + AC_CHUNK - 1) / AC_CHUNK);
  double tot = 0.0;
  for (int q = 0; q < nq; ++q) tot += a.chunk[(int64_t)q * a.k + j];
  const double mu = tot / (double)a.fs.nframes;
  a.mu[j] = mu;
  double off = 0.0;
  for (int q = 0; q < nq; ++q) {
    const int64_t f0 = (int64_t)q * AC_CHUNK;
    const int64_t cnt = f0 + AC_CHUNK < a.fs.nframes ? AC_CHUNK : a.fs.nframes - f0;
    const double s = a.chunk[(int64_t)q * a.k + j];
    a.chunk[(int64_t)q * a.k + j] = off;
    off += s - (double)cnt * mu;
  }
  a.P[j] = 0.0;  // P_0
}

// P rows 1..F, each coordinate times sqrt(mass) when weighted.
__global__ __launch_bounds__(AC_THREADS) void k_ac_prefix(AvgPrefixArgs a) {
  const int j = blockIdx.x * AC_THREADS + threadIdx.x;
  const int q = blockIdx.y;
  if (j >= a.k) return;
  const int kk = j / 3, c = j - 3 * kk;
  const double mu = a.mu[j];
  const double sw = a.mass ? sqrt(a.mass[kk]) : 1.0;
  double run = a.chunk[(int64_t)q * a.k + j];
  const int64_t f0 = (int64_t)q * AC_CHUNK;
  const int64_t f1 = f0 + AC_CHUNK < a.fs.nframes ? f0 + AC_CHUNK : a.fs.nframes;
  for (int64_t f = f0; f < f1; ++f) {
    run += (double)coord(a.fs, f, kk, c) - mu;
    a.P[(f + 1) * a.k + j] = run * sw;
  }
}

// Constants (row F + 1 of rows): sum m mu (3), sum m v y^T (9),
// sum m |v|^2 (1).  One wave.
__global__ __launch_bounds__(64) void k_ac_consts(AvgPrefixArgs a) {
  const int n = a.fs.nsel;
  const double W = a.consts[4];
  double s[3] = {0.0, 0.0, 0.0};
  for (int kk = threadIdx.x; kk < n; kk += 64) {
    const double m = a.mass ? a.mass[kk] : 1.0;
    for (int c = 0; c < 3; ++c) s[c] += m * a.mu[3 * kk + c];
  }
  double mc[3];
  for (int c = 0; c < 3; ++c) {
    s[c] = rmsd_dev::wave_sum(s[c]);
    mc[c] = W > 0.0 ? s[c] / W : 0.0;
  }
  double v[13];
#pragma unroll
  for (int q = 0; q < 13; ++q) v[q] = 0.0;
  for (int kk = threadIdx.x; kk < n; kk += 64) {
    const double m = a.mass ? a.mass[kk] : 1.0;
    const double y0 = a.ref ? a.ref[kk] : 0.0, y1 = a.ref ? a.ref[a.ldr + kk] : 0.0,
                 y2 = a.ref ? a.ref[2 * a.ldr + kk] : 0.0;
    for (int c = 0; c < 3; ++c) {
      const double vc = a.mu[3 * kk + c] - mc[c];
      const double mm = m * vc;
      v[3 + 3 * c] += mm * y0;
      v[4 + 3 * c] += mm * y1;
      v[5 + 3 * c] += mm * y2;
      v[12] += m * vc * vc;
    }
  }
  double r[13];
  wave_moments(v, r);
  if (threadIdx.x == 0) {
    double* o = a.rows + (a.fs.nframes + 1) * 13;
    for (int c = 0; c < 3; ++c) o[c] = s[c];
    for (int q = 3; q < 13; ++q) o[q] = r[q];
  }
}

// Per prefix row i (0..F): C_i (3), Q_i (9), L_i (1).  One wave per row.  With a
// fixed reference the row loses its centroid first: P~_i = P_i - C_i / W (44 us at
// 10,000 x 300, the rows written once more; 19 without).
__global__ __launch_bounds__(64) void k_ac_rows(AvgPrefixArgs a) {
  const int64_t i = blockIdx.x;
  const int n = a.fs.nsel;
  const double W = a.consts[4];
  const double* cr = a.rows + (a.fs.nframes + 1) * 13;
  double mc[3];
  for (int c = 0; c < 3; ++c) mc[c] = W > 0.0 ? cr[c] / W : 0.0;
  double* Pi = a.P + i * a.k;
  double t[3] = {0.0, 0.0, 0.0};
  if (a.ref) {
    for (int kk = threadIdx.x; kk < n; kk += 64) {
      const double sw = a.mass ? sqrt(a.mass[kk]) : 1.0;
      for (int c = 0; c < 3; ++c) t[c] += sw * Pi[3 * kk + c];
    }
    for (int c = 0; c < 3; ++c) {
      t[c] = rmsd_dev::wave_sum(t[c]);
      t[c] = W > 0.0 ? t[c] / W : 0.0;
    }
  }
  double v[13];
#pragma unroll
  for (int q = 0; q < 13; ++q) v[q] = 0.0;
  for (int kk = threadIdx.x; kk < n; kk += 64) {
    const double sw = a.mass ? sqrt(a.mass[kk]) : 1.0;
    const double y0 = a.ref ? a.ref[kk] : 0.0, y1 = a.ref ? a.ref[a.ldr + kk] : 0.0,
                 y2 = a.ref ? a.ref[2 * a.ldr + kk] : 0.0;
    for (int c = 0; c < 3; ++c) {
      const double p = Pi[3 * kk + c] - sw * t[c];
      if (a.ref) Pi[3 * kk + c] = p;
      const double mp = sw * p;  // m P
      v[c] += mp;
      v[3 + 3 * c] += mp * y0;
      v[4 + 3 * c] += mp * y1;
      v[5 + 3 * c] += mp * y2;
      v[12] += mp * (a.mu[3 * kk + c] - mc[c]);
    }
  }
  double r[13];
  wave_moments(v, r);
  if (threadIdx.x == 0)
    for (int q = 0; q < 13; ++q) a.rows[i * 13 + q] = r[q];
}

// The fit of one averaged frame from the difference form's pieces: d2 = sum
// m |P~_i - P~_j|^2, the row moments ri and rj, the constants
// row cm and the reference constants K.
__device__ __forceinline__ double ac_fit(double d2, const double* ri, const double (&rj)[13],
                                         const double* cm, const double* K, double w) {
  const double W = K[4];
  if (W < RMSD_SMALL) return -1.0;
  // 1 / w: the hardware reciprocal, refined twice (2^-53)
  double iw = __builtin_amdgcn_rcp(w);
  iw = fma(iw, fma(-w, iw, 1.0), iw);
  iw = fma(iw, fma(-w, iw, 1.0), iw);
  double R[9];
#pragma unroll
  for (int e = 0; e < 9; ++e) R[e] = (ri[3 + e] - rj[3 + e]) * iw + cm[3 + e];
  const double sx = d2 * (iw * iw) + 2.0 * (ri[12] - rj[12]) * iw + cm[12];
  return rmsd_dev::qcp_rmsd(R, 0.5 * (sx + K[3]), W, 1);
}

// Fits on local diagonal dd = il - jl of row tile ti: il0 ... il1 - 1.
__device__ __forceinline__ void ac_span(int64_t nrow, int ti, int dd, int& il0, int& il1) {
  const int64_t rows = nrow - (int64_t)ti * AC_TILE;
  il0 = dd > 0 ? dd : 0;
  il1 = dd < 0 ? AC_TILE + dd : AC_TILE;
  if (il1 > rows) il1 = (int)rows;
}

// A tile's RMSDs rr[64][AC_LD] along its diagonals, thread dd + 63 taking local
// diagonal dd: their sum, and their squared deviations from its mean, by way of
// the first RMSD (the mean square less the squared mean leaves the last windows,
// whose few fits hardly differ, up to sqrt(eps) of the RMSD: 10,000 x 300, over
// all windows, 7e-10 of the SDs' norm; so 1e-11).
__device__ __forceinline__ void ac_diagonals(const AvgPrefixArgs& a, const double* rr, int ti,
                                             int tj) {
  const int64_t i0 = (int64_t)ti * AC_TILE, j0 = (int64_t)tj * AC_TILE;
  const int64_t nrow = a.fs.nframes + 1;
  const int t = threadIdx.x;
  if (t >= 2 * AC_TILE - 1) return;
  const int dd = t - (AC_TILE - 1);
  const int64_t w = (i0 - j0) + dd;
  if (!(w >= 1 && w < nrow && a.wmap[w] >= 0)) return;
  double s1 = 0.0, s2 = 0.0;
  int il0, il1;
  ac_span(nrow, ti, dd, il0, il1);
  if (il1 > il0) {
    const double r0 = rr[il0 * AC_LD + il0 - dd];
    double t1 = 0.0;
    for (int il = il0; il < il1; ++il) {
      const double r = rr[il * AC_LD + il - dd], e = r - r0;
      s1 += r;
      t1 += e;
      s2 += e * e;
    }
    s2 -= t1 * t1 / (double)(il1 - il0);
  }
  // Slot of this tile among the two j tiles that diagonal w crosses in row
  // tile ti.
  const int half = tj - (ti - (int)((w + AC_TILE - 1) / AC_TILE));
  double* o = a.part + (((int64_t)a.wmap[w] * a.ntile + ti) * 2 + half) * 2;
  o[0] = s1;
  o[1] = s2;
}

// One 64 x 64 tile of (i, j) prefix-row pairs, distances from the differences.
// Thread (ty, tx) = (t / 16, t % 16) owns rows i0 + ty + 16 a and j0 + tx + 16 b
// (a, b < 4).  For the tiles on and next to the diagonal (ac_gram takes the
// others).
// sm: [2][KC][65] staged coordinates (odd row stride: conflict-free transposed
// stores), later the RMSDs [64][65].
constexpr int AC_LDS = 2 * AC_KC * AC_LD;
static_assert(AC_LDS >= AC_TILE * AC_LD, "RMSD tile does not fit");
__device__ __forceinline__ void ac_direct(const AvgPrefixArgs& a, int ti, int tj, double* sm) {
  double* si = sm;
  double* sj = sm + AC_KC * AC_LD;
  const int64_t i0 = (int64_t)ti * AC_TILE, j0 = (int64_t)tj * AC_TILE;
  const int64_t nrow = a.fs.nframes + 1;
  const int t = threadIdx.x, ty = t >> 4, tx = t & 15;
  double acc[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[p][q] = 0.0;
  // Staging: thread t takes coordinate (t % 32) of rows (t / 32) + 8 r, the next
  // stage's in flight meanwhile.  Rows and coordinates past the end are read from
  // the last row and coordinate 0, so that no load waits behind a branch (with
  // branches and no prefetch these few tiles' latency bound the small calls: 128 x
  // 300 332 -> 241 us, 2,000 x 300, every tenth window, 426 -> 336).
  const int lc = t & (AC_KC - 1), lr = t >> 5;
  const auto bi = gp(a.P + i0 * a.k), bj = gp(a.P + j0 * a.k);
  const int ni = (int)(nrow - i0), nj = (int)(nrow - j0);
  int oi[8], oj[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int row = lr + 8 * r;
    oi[r] = (row < ni ? row : ni - 1) * a.k;
    oj[r] = (row < nj ? row : nj - 1) * a.k;
  }
  double vi[8], vj[8];
  auto fetch = [&](int k0) {
    const int kc = k0 + lc < a.k ? k0 + lc : 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      vi[r] = bi[oi[r] + kc];
      vj[r] = bj[oj[r] + kc];
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < a.k; k0 += AC_KC) {
    const bool in = k0 + lc < a.k;
    __syncthreads();  // the last stage's reads
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      si[lc * AC_LD + lr + 8 * r] = in ? vi[r] : 0.0;
      sj[lc * AC_LD + lr + 8 * r] = in ? vj[r] : 0.0;
    }
    __syncthreads();
    if (k0 + AC_KC < a.k) fetch(k0 + AC_KC);
#pragma unroll 4
    for (int c = 0; c < AC_KC; ++c) {
      double pi[4], pj[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        pi[p] = si[c * AC_LD + ty + 16 * p];
        pj[p] = sj[c * AC_LD + tx + 16 * p];
      }
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double d = pi[p] - pj[q];
          acc[p][q] = fma(d, d, acc[p][q]);
        }
    }
  }
  __syncthreads();
  // Fits of the pairs on window diagonals.
  const double* cm = a.rows + nrow * 13;
  double* rr = sm;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int jl = tx + 16 * q;
    const int64_t j = j0 + jl;
    double rj[13];
#pragma unroll
    for (int e = 0; e < 13; ++e) rj[e] = a.rows[(j < nrow ? j : 0) * 13 + e];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int il = ty + 16 * p;
      const int64_t i = i0 + il, w = i - j;
      double r = 0.0;
      if (w >= 1 && i < nrow && a.wmap[w] >= 0)
        r = ac_fit(acc[p][q], a.rows + i * 13, rj, cm, a.consts, (double)w);
      rr[il * AC_LD + jl] = r;
    }
  }
  __syncthreads();
  ac_diagonals(a, rr, ti, tj);
}

// A tile two or more tiles off the diagonal (windows of at least 65 frames):
// the distances as a Gram product on FP64 MFMA, one multiply-add per coordinate
// and pair instead of a difference and a multiply-add.  Rows are taken about the
// middle row m of the column tile, q_i = P_i - P_m, p_j = P_j - P_m:
//   |P_i - P_j|^2 = |q_i|^2 + |p_j|^2 - 2 q_i . p_j.
// With |q_i| <= |P_i - P_j| + |p_j| its rounding is a few eps of |P_i - P_j|^2, as
// the differences' own, and of |p_j|^2, at most 32 frames' deviations from the
// mean.  The latter, over w^2, has to stay below the reference's sum w |y|^2,
// which the fit adds to it and rounds itself: a tile where it does not (returns
// false, before anything is stored) takes the differences.  Deviations that keep
// one direction for 32 frames have to reach twice the reference's radius of
// gyration for that, and only in the tiles of the shortest windows.
//
// Each of the four waves owns 32 x 32 pairs, four 16 x 16 blocks; a stage of 32
// coordinates of the 128 rows goes to LDS shifted, the next stage's loads in
// flight meanwhile.  Bound by the FP64 matrix rate
// and, after it, the fits' vector FP64.  Tiles come in bands of eight row
// tiles, an XCD's workgroups in one run of that order, so that tiles running
// side by side share rows in its L2.  10,000 frames x 300 atoms, all windows: the
// whole call 2.44 ms against 4.80 with every tile's distances from the
// differences; MFMA pipes 54 % busy and vector issue 27 % at 2.1 GHz, three waves
// per SIMD (four spill: 3.36 ms).  The tiles near the diagonal run in the same
// launch: 314 of 12,400.
typedef __attribute__((ext_vector_type(4))) double f64x4;

__device__ __forceinline__ bool ac_gram(const AvgPrefixArgs& a, int ti, int tj, double* sm,
                                        double (*norm)[2 * AC_TILE]) {
  double* si = sm;
  double* sj = sm + AC_KC * AC_LD;
  const int64_t i0 = (int64_t)ti * AC_TILE, j0 = (int64_t)tj * AC_TILE;
  const int64_t nrow = a.fs.nframes + 1;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int lc = t & (AC_KC - 1), lr = t >> 5;
  const double* mid = a.P + (j0 + AC_TILE / 2) * a.k;  // tj < ti: a whole tile of rows
  // Uniform bases and one 32-bit lane offset for all sixteen rows.
  const double* bi = a.P + i0 * a.k;
  const double* bj = a.P + j0 * a.k;
  const int lo = lr * a.k + lc;
  const int rows = (int)(nrow - i0 < AC_TILE ? nrow - i0 : AC_TILE);
  const int kfull = rows == AC_TILE ? a.k - AC_KC : -1;  // stages before it need no checks
  double vi[8], vj[8], vm;
  auto fetch = [&](int k0) {
    if (k0 <= kfull) {  // uniform
      vm = gp(mid + k0)[lc];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        vi[r] = gp(bi + (int64_t)(8 * r) * a.k + k0)[lo];
        vj[r] = gp(bj + (int64_t)(8 * r) * a.k + k0)[lo];
      }
      return;
    }
    const bool in = k0 + lc < a.k;
    vm = in ? gp(mid + k0)[lc] : 0.0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      vi[r] = in && lr + 8 * r < rows ? gp(bi + (int64_t)(8 * r) * a.k + k0)[lo] : vm;
      vj[r] = in ? gp(bj + (int64_t)(8 * r) * a.k + k0)[lo] : vm;
    }
  };
  // The rows' squares: thread t sums half of each stage's coordinates (t / 128)
  // of row t % 128 of the i rows, then the j rows.
  const double* srow = (t & 64 ? sj : si) + (t & 63) + (t >> 7) * (AC_KC / 2) * AC_LD;
  double sq = 0.0;
  f64x4 acc[2][2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q) acc[p][q] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int ri0 = 32 * (wave >> 1) + (lane & 15), cj0 = 32 * (wave & 1) + (lane & 15);
  fetch(0);
  for (int k0 = 0; k0 < a.k; k0 += AC_KC) {
    __syncthreads();  // the last stage's reads
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      si[lc * AC_LD + lr + 8 * r] = vi[r] - vm;
      sj[lc * AC_LD + lr + 8 * r] = vj[r] - vm;
    }
    __syncthreads();
    if (k0 + AC_KC < a.k) fetch(k0 + AC_KC);
#pragma unroll
    for (int c = 0; c < AC_KC / 2; ++c) sq = fma(srow[c * AC_LD], srow[c * AC_LD], sq);
#pragma unroll
    for (int c = 0; c < AC_KC; c += 4) {
      const int kk = (c + (lane >> 4)) * AC_LD;
      double av[2], bv[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        av[p] = si[kk + ri0 + 16 * p];
        bv[p] = sj[kk + cj0 + 16 * p];
      }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[p], bv[q], acc[p][q], 0, 0, 0);
    }
  }
  norm[t >> 7][t & 127] = sq;
  __syncthreads();  // and the last stage's reads: sm becomes the RMSD tile
  const double far = norm[0][AC_TILE + lane] + norm[1][AC_TILE + lane];  // |p_j|^2, j0 + lane
  const double wmin = (double)(AC_TILE * (ti - tj) - (AC_TILE - 1));
  if (!__all(far <= wmin * wmin * a.consts[3])) return false;  // the same in every wave
  const double* cm = a.rows + nrow * 13;
  // The accumulators hold row lane / 16 + 4 v, column lane % 16, in item v.
#pragma unroll 1
  for (int q = 0; q < 2; ++q) {
    const int jl = cj0 + 16 * q;
    const int64_t j = j0 + jl;
    double rj[13];
#pragma unroll
    for (int e = 0; e < 13; ++e) rj[e] = gp(a.rows)[j * 13 + e];
    const double nj = norm[0][AC_TILE + jl] + norm[1][AC_TILE + jl];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int il = 32 * (wave >> 1) + 16 * p + (lane >> 4) + 4 * v;
        const int64_t i = i0 + il, w = i - j;
        double r = 0.0;
        if (i < nrow && a.wmap[w] >= 0) {
          const double g = q == 0 ? acc[p][0][v] : acc[p][1][v];
          const double d2 = fmax(norm[0][il] + norm[1][il] + nj - 2.0 * g, 0.0);
          r = ac_fit(d2, a.rows + i * 13, rj, cm, a.consts, (double)w);
        }
        sm[il * AC_LD + jl] = r;
      }
  }
  __syncthreads();
  ac_diagonals(a, sm, ti, tj);
  return true;
}

// The tiles near the diagonal first: they take longest.
__global__ __launch_bounds__(AC_THREADS) __attribute__((amdgpu_waves_per_eu(3))) void k_ac_tiles(
    AvgPrefixArgs a) {
  __shared__ double sm[AC_LDS];
  __shared__ double norm[2][2 * AC_TILE];
  const int near = a.ntiles - a.ngram;
  int k = (int)blockIdx.x;
  if (k >= near) {
    const int b = k - near;
    const int w = (b % AC_XCDS) * a.gram_per_xcd + b / AC_XCDS;
    if (w >= a.ngram) return;  // the whole workgroup
    k = near + w;
  }
  const int2 tile = a.tiles[k];
  if (k >= near && ac_gram(a, tile.x, tile.y, sm, norm)) return;
  ac_direct(a, tile.x, tile.y, sm);
}

// Mean and standard deviation per window from the per-tile sums, in a fixed
// order.  One wave per window.
__global__ __launch_bounds__(64) void k_ac_final(AvgPrefixArgs a) {
  const int wi = blockIdx.x;
  const int w = a.windows[wi];
  auto slots = [&](auto&& use) {
    for (int slot = threadIdx.x; slot < 2 * a.ntile; slot += 64) {
      const int ti = slot >> 1, half = slot & 1;
      // The tile (ti, tj) that holds this slot; written when it exists and
      // diagonal w crosses it (a multiple of 64 crosses one tile per row tile).
      const int T = a.tile;
      const int tj = ti - (w + T - 1) / T + half;
      if (tj < 0 || tj > ti) continue;
      const int off = w - T * (ti - tj);
      if (off < 1 - T || off > T - 1) continue;
      use(ti, off, a.part + (((int64_t)wi * a.ntile + ti) * 2 + half) * 2);
    }
  };
  const double d = 1.0 / ((double)a.fs.nframes - (double)w + 1.0);
  double s1 = 0.0, s2 = 0.0;
  slots([&](int, int, const double* o) {
    s1 += o[0];
    s2 += o[1];
  });
  const double avg = rmsd_dev::wave_sum(s1) * d;
  // Fixed reference: the slots' own deviations and those of their means; 'first'
  // has sums of squares.
  if (!a.yref)
    slots([&](int ti, int off, const double* o) {
      int il0, il1;
      ac_span(a.fs.nframes + 1, ti, off, il0, il1);
      if (il1 <= il0) return;
      const double e = o[0] / (double)(il1 - il0) - avg;
      s2 += (double)(il1 - il0) * e * e;
    });
  s2 = rmsd_dev::wave_sum(s2);
  if (threadIdx.x == 0) {
    double sd = s2 * d;
    if (a.yref) sd -= avg * avg;
    a.ct[wi] = avg;
    a.sd[wi] = sd > 0.0 ? sqrt(sd) : 0.0;
  }
}

// ---- prefix form, 'first' reference --------------------------------------------------
// Window w's reference is its first averaged frame, centred:
// y_w = P_w / w + mu - c_w.  An averaged frame's cross moment is then
//   sum m a y_w^T = (1/w) sum m (P_i - P_j) y_w^T + sum m mu y_w^T,
// linear in the prefix difference (its rounding stays relative to the
// difference, as for the fixed reference).  k_ac_firstref writes sqrt(m) y_w
// per window and its constants (sum m y_w, sum m |y_w|^2, sum m mu y_w^T);
// k_ac_tiles_first runs 32 x 32 tiles of prefix-row pairs with the window
// references of the tile's 63 diagonals staged beside the rows, 2 x 2 pairs
// per thread (a squared distance and nine cross sums each).
constexpr int ACF_TILE = 32;
constexpr int ACF_KA = 8;                // atoms per LDS stage
constexpr int ACF_KC = 3 * ACF_KA;       // coordinates per stage
constexpr int ACF_LD = ACF_TILE + 1;
constexpr int ACF_NDIAG = 2 * ACF_TILE - 1;

__global__ __launch_bounds__(64) void k_ac_firstref(AvgPrefixArgs a) {
  const int wi = blockIdx.x;
  const int w = a.windows[wi];
  const double dw = (double)w;
  const int n = a.fs.nsel;
  const double W = a.consts[4];
  const double* cm = a.rows + (a.fs.nframes + 1) * 13;
  const double* Cw = a.rows + (int64_t)w * 13;
  double cw[3];
  for (int e = 0; e < 3; ++e) cw[e] = W > 0.0 ? (Cw[e] / dw + cm[e]) / W : 0.0;
  const double* Pw = a.P + (int64_t)w * a.k;
  double* ys = a.yref + (int64_t)wi * a.k;
  double v[13];
#pragma unroll
  for (int q = 0; q < 13; ++q) v[q] = 0.0;
  for (int kk = threadIdx.x; kk < n; kk += 64) {
    const double m = a.mass ? a.mass[kk] : 1.0;
    const double sw = a.mass ? sqrt(m) : 1.0;
    double y[3];
    for (int e = 0; e < 3; ++e) {
      const double pw = sw > 0.0 ? Pw[3 * kk + e] / sw : 0.0;
      y[e] = pw / dw + a.mu[3 * kk + e] - cw[e];
      ys[3 * kk + e] = sw * y[e];
      v[e] += m * y[e];
      v[3] += m * y[e] * y[e];
    }
    for (int c = 0; c < 3; ++c) {
      const double mm = m * a.mu[3 * kk + c];
      for (int e = 0; e < 3; ++e) v[4 + 3 * c + e] += mm * y[e];
    }
  }
  double r[13];
  wave_moments(v, r);
  if (threadIdx.x == 0)
    for (int q = 0; q < 13; ++q) a.wconst[(int64_t)wi * 13 + q] = r[q];
}

__global__ __launch_bounds__(AC_THREADS) void k_ac_tiles_first(AvgPrefixArgs a) {
  // [2][KC][33] staged rows (later the RMSDs [32][33]) and [63][KC] window
  // references.
  __shared__ double sij[2 * ACF_KC * ACF_LD];
  __shared__ double sy[ACF_NDIAG * ACF_KC];
  static_assert(2 * ACF_KC * ACF_LD >= ACF_TILE * ACF_LD, "RMSD tile does not fit");
  double* si = sij;
  double* sj = sij + ACF_KC * ACF_LD;
  const int2 tile = a.tiles[blockIdx.x];
  const int ti = tile.x, tj = tile.y;
  const int64_t i0 = (int64_t)ti * ACF_TILE, j0 = (int64_t)tj * ACF_TILE;
  const int64_t base = i0 - j0;
  const int64_t nrow = a.fs.nframes + 1;
  const int t = threadIdx.x, ty = t >> 4, tx = t & 15;
  double D[2][2], X[2][2][9];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      D[p][q] = 0.0;
#pragma unroll
      for (int e = 0; e < 9; ++e) X[p][q][e] = 0.0;
    }
  // Diagonal of each of the thread's pairs (index into sy).
  int dg[2][2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q) dg[p][q] = (ty + 16 * p) - (tx + 16 * q) + (ACF_TILE - 1);
  for (int k0 = 0; k0 < a.k; k0 += ACF_KC) {
    // Rows: 32 x 24 coordinates each for i and j.
    for (int e = t; e < ACF_TILE * ACF_KC; e += AC_THREADS) {
      const int row = e / ACF_KC, kc = e - row * ACF_KC;
      const int64_t gi = i0 + row, gj = j0 + row;
      const int kg = k0 + kc;
      si[kc * ACF_LD + row] = (kg < a.k && gi < nrow) ? a.P[gi * a.k + kg] : 0.0;
      sj[kc * ACF_LD + row] = (kg < a.k && gj < nrow) ? a.P[gj * a.k + kg] : 0.0;
    }
    // Window references of the 63 diagonals.
    for (int e = t; e < ACF_NDIAG * ACF_KC; e += AC_THREADS) {
      const int d = e / ACF_KC, kc = e - d * ACF_KC;
      const int64_t w = base + d - (ACF_TILE - 1);
      const int kg = k0 + kc;
      double v = 0.0;
      if (w >= 1 && w < nrow && kg < a.k) {
        const int wi = a.wmap[w];
        if (wi >= 0) v = a.yref[(int64_t)wi * a.k + kg];
      }
      sy[d * ACF_KC + kc] = v;
    }
    __syncthreads();
#pragma unroll
    for (int at = 0; at < ACF_KA; ++at) {
      double pi[2][3], pj[2][3];
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          pi[p][c] = si[(3 * at + c) * ACF_LD + ty + 16 * p];
          pj[p][c] = sj[(3 * at + c) * ACF_LD + tx + 16 * p];
        }
      // The pairs (0, 0) and (1, 1) lie on one diagonal: three references.
      double yv[3][3];
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        const double* y = sy + (dg[0][0] + 16 * (u - 1)) * ACF_KC + 3 * at;
        yv[u][0] = y[0];
        yv[u][1] = y[1];
        yv[u][2] = y[2];
      }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int u = p - q + 1;
          const double y0 = yv[u][0], y1 = yv[u][1], y2 = yv[u][2];
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            const double d = pi[p][c] - pj[q][c];
            D[p][q] = fma(d, d, D[p][q]);
            X[p][q][3 * c] = fma(d, y0, X[p][q][3 * c]);
            X[p][q][3 * c + 1] = fma(d, y1, X[p][q][3 * c + 1]);
            X[p][q][3 * c + 2] = fma(d, y2, X[p][q][3 * c + 2]);
          }
        }
    }
    __syncthreads();
  }
  const double W = a.consts[4];
  const double* cm = a.rows + nrow * 13;
  double* rr = sij;  // [32][33] RMSDs, over the staging
  for (int p = 0; p < 2; ++p)
    for (int q = 0; q < 2; ++q) {
      const int il = ty + 16 * p, jl = tx + 16 * q;
      const int64_t i = i0 + il, j = j0 + jl;
      const int64_t w = i - j;
      double r = 0.0;
      if (w >= 1 && i < nrow && a.wmap[w] >= 0) {
        if (W < RMSD_SMALL) {
          r = -1.0;
        } else {
          const int wi = a.wmap[w];
          const double dw = (double)w;
          const double* ri = a.rows + i * 13;
          const double* rj = a.rows + j * 13;
          const double* K = a.wconst + (int64_t)wi * 13;  // sum m y (3), sum m |y|^2, M (9)
          double dc[3], c[3];
          for (int e = 0; e < 3; ++e) {
            dc[e] = (ri[e] - rj[e]) / (dw * W);
            c[e] = dc[e] + cm[e] / W;
          }
          double R[9];
          for (int e = 0; e < 9; ++e) R[e] = X[p][q][e] / dw + K[4 + e] - c[e / 3] * K[e % 3];
          const double sx = D[p][q] / (dw * dw) + 2.0 * (ri[12] - rj[12]) / dw + cm[12] -
                            W * (dc[0] * dc[0] + dc[1] * dc[1] + dc[2] * dc[2]);
          const double E0 = 0.5 * (sx + K[3]);
          r = rmsd_dev::qcp_rmsd(R, E0, W, 1);
        }
      }
      rr[il * ACF_LD + jl] = r;
    }
  __syncthreads();
  if (t < ACF_NDIAG) {
    const int dd = t - (ACF_TILE - 1);
    const int64_t w = base + dd;
    if (w >= 1 && w < nrow && a.wmap[w] >= 0) {
      double s1 = 0.0, s2 = 0.0;
      const int il0 = dd > 0 ? dd : 0, il1 = dd < 0 ? ACF_TILE + dd : ACF_TILE;
      for (int il = il0; il < il1; ++il) {
        const double r = rr[il * ACF_LD + il - dd];
        s1 += r;
        s2 += r * r;
      }
      const int half = tj - (ti - (int)((w + ACF_TILE - 1) / ACF_TILE));
      double* o = a.part + (((int64_t)a.wmap[w] * a.ntile + ti) * 2 + half) * 2;
      o[0] = s1;
      o[1] = s2;
    }
  }
}

// Total weight for the 'first' form (consts[4]; the rest unused): one wave.
__global__ __launch_bounds__(64) void k_ac_wsum(AvgPrefixArgs a, double* consts) {
  double s = 0.0;
  for (int kk = threadIdx.x; kk < a.fs.nsel; kk += 64) s += a.mass ? a.mass[kk] : 1.0;
  s = rmsd_dev::wave_sum(s);
  if (threadIdx.x == 0) {
    for (int q = 0; q < 4; ++q) consts[q] = 0.0;
    consts[4] = s;
  }
}

}  // namespace

int rmsd_avgcorr_chunks(int64_t nframes) { return (int)((nframes + AC_CHUNK - 1) / AC_CHUNK); }
int rmsd_avgcorr_tile(bool first) { return first ? ACF_TILE : AC_TILE; }

hipError_t rmsd_launch_avgcorr_prefix(const AvgPrefixArgs& a, hipStream_t s) {
  if (a.nwin == 0 || a.ntiles == 0) return hipSuccess;
  const int nq = rmsd_avgcorr_chunks(a.fs.nframes);
  const dim3 gj((a.k + AC_THREADS - 1) / AC_THREADS, nq);
  hipLaunchKernelGGL(k_ac_chunksum, gj, dim3(AC_THREADS), 0, s, a);
  hipLaunchKernelGGL(k_ac_scan, dim3(gj.x), dim3(AC_THREADS), 0, s, a);
  hipLaunchKernelGGL(k_ac_prefix, gj, dim3(AC_THREADS), 0, s, a);
  hipLaunchKernelGGL(k_ac_consts, dim3(1), dim3(64), 0, s, a);
  hipLaunchKernelGGL(k_ac_rows, dim3((unsigned)(a.fs.nframes + 1)), dim3(64), 0, s, a);
  return hipGetLastError();
}

hipError_t rmsd_launch_avgcorr_tiles(const AvgPrefixArgs& a, hipStream_t s) {
  if (a.nwin == 0 || a.ntiles == 0) return hipSuccess;
  if (a.yref) {
    hipLaunchKernelGGL(k_ac_firstref, dim3(a.nwin), dim3(64), 0, s, a);
    hipLaunchKernelGGL(k_ac_tiles_first, dim3(a.ntiles), dim3(AC_THREADS), 0, s, a);
  } else {
    if (a.ngram > a.ntiles || a.gram_per_xcd * AC_XCDS < a.ngram) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_ac_tiles, dim3(a.ntiles - a.ngram + a.gram_per_xcd * AC_XCDS),
                       dim3(AC_THREADS), 0, s, a);
  }
  return hipGetLastError();
}

hipError_t rmsd_launch_avgcorr_wsum(const AvgPrefixArgs& a, double* consts, hipStream_t s) {
  hipLaunchKernelGGL(k_ac_wsum, dim3(1), dim3(64), 0, s, a, consts);
  return hipGetLastError();
}

hipError_t rmsd_launch_avgcorr_final(const AvgPrefixArgs& a, hipStream_t s) {
  if (a.nwin == 0) return hipSuccess;
  hipLaunchKernelGGL(k_ac_final, dim3(a.nwin), dim3(64), 0, s, a);
  return hipGetLastError();
}
