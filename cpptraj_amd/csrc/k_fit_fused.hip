// k_fit_fused.hip -- the fit of every frame to one reference in one launch:
// moments, QCP solve and coordinate update with the frame held in registers.
//
// Replaces the per-frame body of Action_Rmsd::DoAction (src/Action_Rmsd.cpp:
// 361-417) where the separate kernels of k_fit.hip (moments, solve, update)
// would read the frame twice or where launches are what the call costs.
//
// A frame is taken by T threads (one wave, or a workgroup of 256 or 512) with
// up to Q quads of four atoms each: three 16-byte loads per quad, all in flight
// at once, kept in registers until the update stores them, so the update's
// traffic is one read and one write of the frame.  The reference comes from L2
// (24 bytes per atom beside 24 of frame traffic; staging it in LDS would leave
// room for one or two frames per CU).  The frames' moments meet in LDS, and
// lanes of wave 0 solve the workgroup's frames side by side.
//
// Bound by HBM, 24 N bytes per frame, and by how many frames are in flight
// while others are being solved.  100,000 x 3,000 AoS frames, fit and rotate:
// 1.66 ms (4.35 TB/s; a plain copy of that size reaches 4.63) against 2.69 ms
// for moments, solve and update one after another.  At 3,000 atoms, threads x
// quads: 128 x 6 1.89 ms, 192 x 4 1.73, 256 x 3 1.66, 384 x 2 2.01, 512 x 2
// 2.63, 768 x 1 2.84; non-temporal stores 1.85, loads too 2.76.  100 x 66 of
// 223 atoms, a small call: 15.2 us against 25.0, in one launch instead of four.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "fit_device.hpp"

namespace {

using namespace fit_dev;

// The reference prepared inside every workgroup (INREF): up to this many atoms.
constexpr int INREF_ATOMS = 512;

struct InRef {
  double y[3 * INREF_ATOMS];  // centred reference [3][ldr]
  double w[INREF_ATOMS];      // weights (1 when unweighted)
  double part[4][4];
  double out[8];              // h (3), sum w |y|^2, W, centre (3)
};

// k_ref_prep's arithmetic by a workgroup of 256, as its own for so few atoms:
// the same sums in the same order (masses one after another), so a call's
// results do not depend on which of the two prepared its reference.
__device__ __forceinline__ void inref_sum(InRef& s, double (&v)[4]) {
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = rmsd_dev::wave_sum(v[i]);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) s.part[wave][i] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = 0.0;
    for (int w = 0; w < 4; ++w) v[i] += s.part[w][i];
  }
  __syncthreads();
}

template <bool WEIGHTED>
__device__ __forceinline__ void inref_prep(const FitFusedArgs& a, int ldr, InRef& s) {
  const int n = a.fs.nsel;
  float p[2][3];
  double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int k = threadIdx.x + 256 * c;
    if (k < n) {
      load_atom(a.R, a.ref_frame, k, p[c]);
      const double m = a.rmass ? a.rmass[k] : 1.0;
      v[0] += (double)p[c][0] * m;
      v[1] += (double)p[c][1] * m;
      v[2] += (double)p[c][2] * m;
      v[3] += m;
      s.w[k] = WEIGHTED ? a.mass[k] : 1.0;
    } else if (k < ldr) {
      s.w[k] = 0.0;
    }
  }
  inref_sum(s, v);
  double cen[3] = {0.0, 0.0, 0.0};
  const double tot = a.rmass ? v[3] : (double)n;
  if (tot != 0.0) {
    cen[0] = v[0] / tot;
    cen[1] = v[1] / tot;
    cen[2] = v[2] / tot;
  }
  double h[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int k = threadIdx.x + 256 * c;
    double y[3] = {0.0, 0.0, 0.0};
    if (k < n) {
      y[0] = (double)p[c][0] - cen[0];
      y[1] = (double)p[c][1] - cen[1];
      y[2] = (double)p[c][2] - cen[2];
      const double w = s.w[k];
      h[0] += w * y[0];
      h[1] += w * y[1];
      h[2] += w * y[2];
      h[3] += w * (y[0] * y[0] + y[1] * y[1] + y[2] * y[2]);
    }
    if (k < ldr)
#pragma unroll
      for (int d = 0; d < 3; ++d) s.y[d * ldr + k] = y[d];
  }
  inref_sum(s, h);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) s.out[i] = h[i];
    double W = 0.0;
    if (WEIGHTED) {
      for (int k = 0; k < n; ++k) W += s.w[k];
    } else {
      W = (double)n;
    }
    s.out[4] = W;
#pragma unroll
    for (int d = 0; d < 3; ++d) s.out[5 + d] = cen[d];
  }
  __syncthreads();
}

// What follows the solve: the update (or nothing), or the gradient of
// rmsd_fit_backward (every fitted atom, no selection) in FP64 or rounded to FP32.
enum { OP_FIT = 0, OP_GRAD64 = 1, OP_GRAD32 = 2 };

// Gradient of one atom, k_fit_grad's: s w_k (x~_k - U^T y_k).
__device__ __forceinline__ void grad_atom(const double (&X)[16], double w, float px, float py,
                                          float pz, double y0, double y1, double y2,
                                          double (&g)[3]) {
  const double s = X[15] * w;
  const double x0 = (double)px + X[9], x1 = (double)py + X[10], x2 = (double)pz + X[11];
  g[0] = s * (x0 - (X[0] * y0 + X[3] * y1 + X[6] * y2));
  g[1] = s * (x1 - (X[1] * y0 + X[4] * y1 + X[7] * y2));
  g[2] = s * (x2 - (X[2] * y0 + X[5] * y1 + X[8] * y2));
}

typedef double f64x2_a8 __attribute__((ext_vector_type(2), aligned(8)));

// PER consecutive atoms' gradients at atom position `at` of the whole output.
template <int OP, int PER>
__device__ __forceinline__ void store_grad(void* grad, int64_t at, const double (&g)[PER][3]) {
  if constexpr (OP == OP_GRAD64) {
    const auto p = gp(static_cast<double*>(grad)) + 3 * at;
    if constexpr (PER == 4) {
#pragma unroll
      for (int i = 0; i < 6; ++i)
        *(__attribute__((address_space(1))) f64x2_a8*)(p + 2 * i) =
            f64x2_a8{g[2 * i / 3][2 * i % 3], g[(2 * i + 1) / 3][(2 * i + 1) % 3]};
    } else {
#pragma unroll
      for (int d = 0; d < 3; ++d) p[d] = g[0][d];
    }
  } else {
    float x[PER], y[PER], z[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      x[e] = (float)g[e][0];
      y[e] = (float)g[e][1];
      z[e] = (float)g[e][2];
    }
    store_step(static_cast<float*>(grad) + 3 * at, 0, 0, x, y, z);
  }
}

// T threads per frame, NF frames of each group of T threads at once (T = 64
// only), Q steps of PER atoms per thread: quads (PER 4), or single atoms where
// quads would leave most lanes idle.
template <int OP, int T, int NF, int Q, int PER, bool WEIGHTED, bool INREF>
__global__ __launch_bounds__(T < 256 ? 256 : T) void k_fit_fused(FitFusedArgs a, int ldr) {
  constexpr int WG = T < 256 ? 256 : T;
  constexpr int G = WG / T * NF;  // frames per workgroup
  constexpr int NW = T / 64;      // waves per frame
  static_assert(G <= 64 && (NF == 1 || T == 64), "the frames are solved by the lanes of wave 0");
  __shared__ double red[G * NW][16];
  __shared__ double xf[G][17];
  __shared__ std::conditional_t<INREF, InRef, char> inref;
  const int g = threadIdx.x / T * NF, t = threadIdx.x % T;
  const int64_t f0 = (int64_t)blockIdx.x * G;
  const int64_t ld = a.fs.ld;
  const bool sel = a.fs.sel != nullptr;
  const int n = a.fs.nsel, nstep = n / PER;
  // Steps held: of all atoms for the update, of the fitted atoms otherwise.
  const int held = a.mode ? a.natom / PER : (sel ? 0 : nstep);
  // The last natom mod PER atoms, one per lane.
  const int ktail = PER * (a.natom / PER) + t;
  const bool tail = PER > 1 && a.mode && ktail < a.natom;
  float x[NF][Q][PER], y[NF][Q][PER], z[NF][Q][PER], xt[NF], yt[NF], zt[NF], s[NF][3];
  const float* fr[NF];
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    // beyond the last frame: the last frame again, never stored
    const int64_t f = f0 + g + j < a.fs.nframes ? f0 + g + j : a.fs.nframes - 1;
    fr[j] = a.fs.xyz + frame_of(a.fs, f) * a.fs.stride;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (t + q * T < held) load_step(fr[j], ld, t + q * T, x[j][q], y[j][q], z[j][q]);
    xt[j] = yt[j] = zt[j] = 0.0f;
    if (tail) {
      float p[3][1];
      load_step(fr[j], ld, ktail, p[0], p[1], p[2]);
      xt[j] = p[0][0];
      yt[j] = p[1][0];
      zt[j] = p[2][0];
    }
    load_atom(a.fs, f, 0, s[j]);
  }
  if constexpr (INREF) inref_prep<WEIGHTED>(a, ldr, inref);
  auto ref = [&](int d, int k) -> double {
    if constexpr (INREF) return inref.y[d * ldr + k];
    else return gp(a.ref)[d * ldr + k];
  };
  auto wt = [&](int k) -> double {
    if constexpr (!WEIGHTED) return 1.0;
    else if constexpr (INREF) return inref.w[k];
    else return gp(a.mass)[k];
  };
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    const double s0 = s[j][0], s1 = s[j][1], s2 = s[j][2];
    double v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = 0.0;
    double (&m)[13] = *reinterpret_cast<double(*)[13]>(v);
    if (!sel) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int i = t + q * T;
        if (i < nstep) {
#pragma unroll
          for (int e = 0; e < PER; ++e)
            accum<WEIGHTED>(m, x[j][q][e] - s0, y[j][q][e] - s1, z[j][q][e] - s2, wt(PER * i + e),
                            ref(0, PER * i + e), ref(1, PER * i + e), ref(2, PER * i + e));
        }
      }
    }
    // The selected atoms, or the last n mod PER fitted ones.
    if (sel || PER > 1) {
      const int64_t f = f0 + g + j < a.fs.nframes ? f0 + g + j : a.fs.nframes - 1;
      for (int k = (sel ? 0 : PER * nstep) + t; k < n; k += T) {
        float p[3];
        load_atom(a.fs, f, k, p);
        accum<WEIGHTED>(m, (double)p[0] - s0, (double)p[1] - s1, (double)p[2] - s2, wt(k),
                        ref(0, k), ref(1, k), ref(2, k));
      }
    }
    const double tot = rmsd_dev::wave_reduce16(v);
    if ((threadIdx.x & 3) == 0) red[(g + j) * NW + t / 64][(threadIdx.x & 63) >> 2] = tot;
  }
  __syncthreads();
  if (threadIdx.x < G && f0 + threadIdx.x < a.fs.nframes) {
    const int64_t fo = f0 + threadIdx.x;
    double mm[13];
#pragma unroll
    for (int i = 0; i < 13; ++i) {
      double sum = red[threadIdx.x * NW][i];
#pragma unroll
      for (int w = 1; w < NW; ++w) sum += red[threadIdx.x * NW + w][i];
      mm[i] = sum;
    }
    // this lane's frame is not its wave's when G > 1: its shift again
    float so[3] = {s[0][0], s[0][1], s[0][2]};
    if (G > 1) load_atom(a.fs, fo, 0, so);
    const double* K = a.consts;
    const double* ct = a.ref_trans;
    if constexpr (INREF) {
      K = inref.out;
      ct = inref.out + 5;
    }
    double U[9], t1[3];
    const double r = solve(mm, K, so[0], so[1], so[2], a.clamp, U, t1);
    if (OP == OP_FIT) a.rmsd[fo] = r;
    if (OP != OP_FIT) {
      xf[threadIdx.x][15] = a.gout[fo] / (K[4] * r);
      // RMSD = 0 (or a NaN, or no weight): no gradient
      xf[threadIdx.x][16] = r > 1e-12 && !(K[4] < RMSD_SMALL) ? 1.0 : 0.0;
    }
    if (a.U)
#pragma unroll
      for (int k = 0; k < 9; ++k) a.U[9 * fo + k] = U[k];
    if (a.tvec)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        a.tvec[6 * fo + k] = t1[k];
        a.tvec[6 * fo + 3 + k] = ct[k];
      }
#pragma unroll
    for (int k = 0; k < 9; ++k) xf[threadIdx.x][k] = U[k];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      xf[threadIdx.x][9 + k] = t1[k];
      xf[threadIdx.x][12 + k] = ct[k];
    }
  }
  if (OP == OP_FIT && !a.mode) return;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    if (f0 + g + j >= a.fs.nframes) return;  // no barrier follows
    double X[16];
#pragma unroll
    for (int k = 0; k < (OP == OP_FIT ? 15 : 16); ++k) X[k] = xf[g + j][k];
    if constexpr (OP != OP_FIT) {
      const int64_t at = (f0 + g + j) * n;
      const bool flat = xf[g + j][16] == 0.0;
      auto step = [&](auto per, int k, const float* px, const float* py, const float* pz) {
        constexpr int P = decltype(per)::value;
        double gr[P][3];
#pragma unroll
        for (int e = 0; e < P; ++e) {
          grad_atom(X, wt(k + e), px[e], py[e], pz[e], ref(0, k + e), ref(1, k + e), ref(2, k + e),
                    gr[e]);
          if (flat) gr[e][0] = gr[e][1] = gr[e][2] = 0.0;
        }
        store_grad<OP, P>(a.grad, at + k, gr);
      };
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int i = t + q * T;
        if (i < nstep) step(std::integral_constant<int, PER>(), PER * i, x[j][q], y[j][q], z[j][q]);
      }
      if (PER > 1 && PER * nstep + t < n) {
        float p[3];
        load_atom(a.fs, f0 + g + j, PER * nstep + t, p);
        step(std::integral_constant<int, 1>(), PER * nstep + t, p, p + 1, p + 2);
      }
      continue;
    }
    float* fw = const_cast<float*>(fr[j]);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = t + q * T;
      if (i < held) {
#pragma unroll
        for (int e = 0; e < PER; ++e)
          move_atom(X, a.mode, x[j][q][e], y[j][q][e], z[j][q][e]);
        store_step(fw, ld, i, x[j][q], y[j][q], z[j][q]);
      }
    }
    if (tail) {
      float tx[1] = {xt[j]}, ty[1] = {yt[j]}, tz[1] = {zt[j]};
      move_atom(X, a.mode, tx[0], ty[0], tz[0]);
      store_step(fw, ld, ktail, tx, ty, tz);
    }
  }
}

template <int OP, int T, int NF, int Q, int PER, bool INREF = false>
hipError_t launch(const FitFusedArgs& a, int ldr, hipStream_t s) {
  constexpr int WG = T < 256 ? 256 : T, G = WG / T * NF;
  const unsigned grid = (unsigned)((a.fs.nframes + G - 1) / G);
  if (a.mass)
    hipLaunchKernelGGL((k_fit_fused<OP, T, NF, Q, PER, true, INREF>), dim3(grid), dim3(WG), 0, s, a,
                       ldr);
  else
    hipLaunchKernelGGL((k_fit_fused<OP, T, NF, Q, PER, false, INREF>), dim3(grid), dim3(WG), 0, s, a,
                       ldr);
  return hipGetLastError();
}

template <int OP>
hipError_t launch_held(const FitFusedArgs& a, int held, int ldr, hipStream_t s) {
  // As the moment kernels where those take the longer calls.
  const bool single = rmsd_fit_single(held, a.fs.ld > 0, OP != OP_FIT || a.mode != 0);
  if (a.ref == nullptr) {
    if (held <= 64) return launch<OP, 64, 1, 1, 1, true>(a, ldr, s);
    if (single) return launch<OP, 64, 1, 2, 1, true>(a, ldr, s);
    if (held <= 256) return launch<OP, 64, 1, 1, 4, true>(a, ldr, s);
    if (held <= 512) return launch<OP, 64, 1, 2, 4, true>(a, ldr, s);
    return launch<OP, 64, 1, 4, 4, true>(a, ldr, s);
  }
  const bool many = a.fs.nframes >= FIT_MANY_FRAMES;
  if (held <= 64)
    return many ? launch<OP, 64, 8, 1, 1>(a, ldr, s) : launch<OP, 64, 1, 1, 1>(a, ldr, s);
  if (single)
    return many ? launch<OP, 64, 4, 2, 1>(a, ldr, s) : launch<OP, 64, 1, 2, 1>(a, ldr, s);
  if (held <= 256)
    return many ? launch<OP, 64, 2, 1, 4>(a, ldr, s) : launch<OP, 64, 1, 1, 4>(a, ldr, s);
  if (held <= 512) return launch<OP, 64, 1, 2, 4>(a, ldr, s);
  if (held <= 1024) return launch<OP, 64, 1, 4, 4>(a, ldr, s);
  if (held <= 2048) return launch<OP, 256, 1, 2, 4>(a, ldr, s);
  if (held <= 3072) return launch<OP, 256, 1, 3, 4>(a, ldr, s);
  if (held <= 4096) return launch<OP, 256, 1, 4, 4>(a, ldr, s);
  return launch<OP, 512, 1, 4, 4>(a, ldr, s);
}

}  // namespace

// One wave per frame up to 1,024 held atoms: its sums run in the order of the
// wave-per-frame moment kernels (k_fit.hip), bit for bit, so the choice between
// the two by the number of frames changes no result.  Without an update larger
// frames go to those kernels (a frame is read once either way, and their solve
// takes a frame per lane); with one, to workgroups of up to 512 threads, 8,192
// atoms.  Where the lines lie (us, this form against the separate kernels):
// nomod 1,000 x 100 13.3 / 16.0, 4,096 x 300 19.0 / 15.9; rotated 2,000 x 8,000
// and up the two read the frame from the same caches.  Several frames per wave
// (their solves share a wave): 200,000 x 50 rotated 296 us with one, 201 with
// eight; 200,000 x 200 325 with one, two and 345 with four.
bool rmsd_fit_fused_fits(int natom, int nsel, int nframes, int mode) {
  if (mode) return natom <= 8192;
  return nsel <= 1024 && nframes <= FIT_FUSED_FRAMES;
}

bool rmsd_fit_inref_fits(int natom, int nsel, int nframes, int mode) {
  return nsel <= INREF_ATOMS && nframes <= FIT_INREF_FRAMES && (!mode || natom <= 1024);
}

hipError_t rmsd_launch_fit_fused(const FitFusedArgs& a, hipStream_t s) {
  if (a.fs.nframes <= 0) return hipSuccess;
  if (!rmsd_fit_fused_fits(a.natom, a.fs.nsel, a.fs.nframes, a.mode)) return hipErrorInvalidValue;
  if (!a.ref && !rmsd_fit_inref_fits(a.natom, a.fs.nsel, a.fs.nframes, a.mode))
    return hipErrorInvalidValue;
  const int held = a.mode ? a.natom : (a.fs.sel ? 0 : a.fs.nsel);
  return launch_held<OP_FIT>(a, held, (a.fs.nsel + 3) & ~3, s);
}

// The gradient holds the fitted atoms as the update holds all of them: the
// same sizes, and frames without a selection.  4,096 x 2,000 weighted, FP32 out:
// 60 us (3.3 TB/s) in place of moments, solve, gradient in FP64 and a
// conversion (25 + 5 + 51 + 60).  FP64 out, its 24 bytes per atom written in
// strided pieces, only up to FIT_GRAD64_ATOMS atoms in all frames where lanes take
// quads: beyond, the separate kernels store full lines and read the frames from
// the caches a second time.  This form against those, us: 700 x 3,000 40 / 49,
// 6,000 x 300 36 / 38, 1,500 x 1,500 44 / 42, 3,000 x 800 47 / 43, 6,000 x 1,500
// 123 / 90; single atoms 40,000 x 128 64 / 73.
bool rmsd_fit_grad_fits(const FrameSetDev& fs, bool f32) {
  if (fs.sel || !rmsd_fit_fused_fits(fs.nsel, fs.nsel, fs.nframes, 1)) return false;
  return f32 || rmsd_fit_single(fs.nsel, fs.ld > 0, true) ||
         (int64_t)fs.nframes * fs.nsel <= FIT_GRAD64_ATOMS;
}

hipError_t rmsd_launch_fit_grad_fused(const FitFusedArgs& a, bool f32, hipStream_t s) {
  if (a.fs.nframes <= 0) return hipSuccess;
  if (!rmsd_fit_grad_fits(a.fs, f32) || a.mode) return hipErrorInvalidValue;
  if (!a.ref && !rmsd_fit_inref_fits(a.fs.nsel, a.fs.nsel, a.fs.nframes, 0))
    return hipErrorInvalidValue;
  const int ldr = (a.fs.nsel + 3) & ~3;
  return f32 ? launch_held<OP_GRAD32>(a, a.fs.nsel, ldr, s)
             : launch_held<OP_GRAD64>(a, a.fs.nsel, ldr, s);
}
