// k_perres.hip -- per-residue no-fit RMSD of the rmsd action ('perres').
//
//   k_perres  Action_Rmsd::DoAction's per-residue loop (src/Action_Rmsd.cpp:
//             398-413): for every frame and residue, the residue's atoms of the
//             frame (optionally as the fit's coordinate update leaves them, in
//             FP64: Frame::Trans_Rot_Trans, src/Frame.h:572-581, or the
//             translate-only update) against the same residue of the uncentred
//             reference frame, both optionally centred (Frame::CenterOnOrigin,
//             src/Frame.cpp:1043-1055), then Frame::RMSD_NoFit
//             (src/Frame.cpp:1279-1307) with the target masses.
//
// The residue list is cut by the host into pieces of whole residues, up to
// PERRES_ENTRIES atoms and PERRES_RES_PIECE residues (a larger residue is a
// piece of its own, taken PERRES_ENTRIES atoms at a time).  A workgroup owns a
// piece and walks over batches of frames.  Each thread owns one atom of the
// piece: its reference atom, mass and index stay in registers, a batch's loads
// (one of 12 bytes per AoS frame) are all in flight together, and the frame's
// update comes through scalar loads.  Its term m |d|^2 goes to LDS; then one
// thread per (frame, residue) adds the residue's terms one after another, while
// the next batch's loads fly.  Every operation and its order are the
// reference's (FP64, contraction off), only spread over the threads, so the
// results are too.
//
// Bound by HBM (12 B per atom and frame), then by the steps' barriers: 50,000
// AoS frames x 3,000 atoms, 194 residues of 7 to 24, masses and update, 1160 ->
// 545 us (3.3 TB/s); centred, 20,000 x 3,000 in residues of 15, 565 -> 282 us
// with the update and 382 -> 217 without.  One lane per (frame, residue) over frames
// staged in LDS (k_perres_lane.hip) has 1.5 waves per SIMD here, and lanes idle where
// residues are shorter than their wave's longest, so that residues of 700 atoms
// took 1264 us where these take 44.  Workgroups of one
// wave (pieces of 64 atoms, no barriers) give 175 us where 256 threads give 159.
// Tables of few atoms, and centred residues of fewer than 5, are the ones that
// lose (idle threads; two steps and three divides for so few terms): those go to
// k_perres_lane.hip, the former kernel.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "rmsd_kernels.hpp"

namespace {

constexpr double kSmall = 0.00000000000001;  // Constants::SMALL, src/Constants.h:35
constexpr int LD = PERRES_ENTRIES + 1;       // a frame's terms in LDS, padded

// Uniform read-only data through the scalar cache.
template <class T>
__device__ __forceinline__ T scalar(const T* p) {
  return *(const __attribute__((address_space(4))) T*)p;
}

// The atom after the fit's update in FP64 with the reference's operation order.
template <int MOD>
__device__ __forceinline__ void moved(const PerresArgs& a, int64_t f, const float (&p)[3],
                                      double& x, double& y, double& z) {
#pragma clang fp contract(off)
  x = (double)p[0];
  y = (double)p[1];
  z = (double)p[2];
  if (MOD == 0) return;
  const double* U = a.U + 9 * f;
  const double* t = a.tvec + 6 * f;
  if (MOD == 1) {
    const double u = x + scalar(t), v = y + scalar(t + 1), w = z + scalar(t + 2);
    x = u * scalar(U) + v * scalar(U + 1) + w * scalar(U + 2) + scalar(t + 3);
    y = u * scalar(U + 3) + v * scalar(U + 4) + w * scalar(U + 5) + scalar(t + 4);
    z = u * scalar(U + 6) + v * scalar(U + 7) + w * scalar(U + 8) + scalar(t + 5);
  } else {
    x = x + (scalar(t) + scalar(t + 3));
    y = y + (scalar(t + 1) + scalar(t + 4));
    z = z + (scalar(t + 2) + scalar(t + 5));
  }
}

// s + q[0] + ... + q[n - 1], one after another.  The loads of several terms are
// in flight together; a term past the end is +0, which leaves a sum that began
// at +0 as it is.
__device__ __forceinline__ double add_terms(double s, const double* q, int n) {
#pragma clang fp contract(off)
  int k = 0;
  for (; k + 8 <= n; k += 8) {
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = q[k + i];
#pragma unroll
    for (int i = 0; i < 8; ++i) s += v[i];
  }
  for (; k < n; k += 4) {
    double v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = q[k + i];
#pragma unroll
    for (int i = 0; i < 4; ++i) s += k + i < n ? v[i] : 0.0;
  }
  return s;
}

template <int MOD, bool CENTER, bool SOA>
__global__ __launch_bounds__(PERRES_THREADS) void k_perres(PerresArgs a) {
#pragma clang fp contract(off)
  constexpr int FB = CENTER ? 4 : 16;  // frames per batch
  constexpr int NS = CENTER ? 3 : 1;   // values per atom and frame in LDS
  constexpr int RES = CENTER ? PERRES_RES_CENTER : PERRES_RES_PIECE;
  constexpr int CJ = CENTER ? FB : 1, CR = CENTER ? RES : 1;
  static_assert(PERRES_THREADS == PERRES_ENTRIES, "one thread per atom of a piece");
  __shared__ double term[NS * FB * LD + 4];
  __shared__ double total[RES];  // target masses of each residue
  __shared__ double ctr[CJ * CR * 3];         // centres of (frame, residue)
  __shared__ int roff[RES + 1];
  __shared__ unsigned char rof[PERRES_ENTRIES];  // residue of each atom (one-stretch pieces)
  const int4 pc = a.pieces[blockIdx.y];
  const int r0 = pc.x, nr = pc.y - pc.x, e0 = pc.z, ne = pc.w - pc.z, t = threadIdx.x;
  const bool big = ne > PERRES_ENTRIES;  // one residue, in stretches
  const float* rfr = a.ref.xyz + frame_of(a.ref, a.ref_frame) * a.ref.stride;

  // This thread's atom of the stretch: entry base + t.  A thread past the end
  // takes the last entry and a batch past the last frame that frame, so that no
  // load waits behind a branch; what they give is not read.
  int at = 0, res = 0;
  double m = 1.0, rm = 1.0, ry[3] = {0.0, 0.0, 0.0}, cref[3] = {0.0, 0.0, 0.0};
  auto entry = [&](int base) {
    if (ne == 0) return;  // empty residues: nothing read but atom 0
    const int k = e0 + (base + t < ne ? base + t : ne - 1);
    at = a.tgt_atoms[k];
    const int q = a.ref_atoms[k];
    if (a.use_mass) {
      m = a.tmass[k];
      if (CENTER) rm = a.rmass[k];
    }
    for (int c = 0; c < 3; ++c) ry[c] = (double)(a.ref.ld ? rfr[c * a.ref.ld + q] : rfr[3 * q + c]);
  };
  const int64_t last = a.nframes - 1;
  float p[FB][3];
  double q[CJ][3];  // of a centred batch: the atoms as the update leaves them
  auto fetch = [&](int64_t f0) {
    int64_t fs[FB];
    if (a.fidx) {
#pragma unroll
      for (int j = 0; j < FB; ++j) fs[j] = scalar(a.fidx + (f0 + j < last ? f0 + j : last));
    } else {
#pragma unroll
      for (int j = 0; j < FB; ++j) fs[j] = f0 + j < last ? f0 + j : last;
    }
#pragma unroll
    for (int j = 0; j < FB; ++j) {
      const auto fr = gp(a.xyz + fs[j] * a.stride);
      if (SOA) {
        p[j][0] = fr[at];
        p[j][1] = fr[a.ld + at];
        p[j][2] = fr[2 * a.ld + at];
      } else {
        const f32x3_a4 q = *(const __attribute__((address_space(1))) f32x3_a4*)(fr + 3 * at);
        p[j][0] = q.x;
        p[j][1] = q.y;
        p[j][2] = q.z;
      }
    }
  };
  // This thread's items of n per residue: item it = t, t + PERRES_THREADS, ...
  // is (it / nr, it % nr), stepped without a division.
  const int ij = t / nr, ir = t - ij * nr, dj = PERRES_THREADS / nr, dr = PERRES_THREADS - dj * nr;
  auto items = [&](int n, int base, auto&& use) {
    const int left = ne - base < PERRES_ENTRIES ? ne - base : PERRES_ENTRIES;
    for (int j = ij, r = ir; j < n;) {
      const int b = big ? 0 : roff[r];
      use(j, r, b, big ? left : roff[r + 1] - b);
      j += dj;
      r += dr;
      if (r >= nr) {
        r -= nr;
        ++j;
      }
    }
  };

  // Masses and reference centres (CenterOnOrigin with the reference masses).
  int64_t f0 = (int64_t)blockIdx.x * FB;
  entry(0);
  fetch(f0);
  for (int r = t; r <= nr; r += PERRES_THREADS) roff[r] = a.res_off[r0 + r] - e0;
  double sum = 0.0;  // of a residue in stretches: one item per thread
  for (int base = 0; base == 0 || base < ne; base += PERRES_ENTRIES) {
    if (base) entry(base);
    __syncthreads();
    if (!big && t < nr)
      for (int k = roff[t]; k < roff[t + 1]; ++k) rof[k] = (unsigned char)t;
    term[t] = m;
    if (CENTER) {
      term[LD + t] = rm;
      for (int d = 0; d < 3; ++d) term[(NS > 1 ? 2 + d : 0) * LD + t] = a.use_mass ? ry[d] * rm : ry[d];
    }
    __syncthreads();
    items(CENTER ? 5 : 1, base, [&](int j, int r, int b, int n) {
      sum = add_terms(base ? sum : 0.0, term + j * LD + b, n);
      if (j == 0) total[r] = sum;
      else ctr[CENTER ? (j - 1) * CR + r : 0] = sum;  // mass, x, y, z
    });
  }
  __syncthreads();
  res = big || t >= ne ? 0 : rof[t];
  if (CENTER && ne > 0) {
    const double w = a.use_mass ? ctr[CENTER ? res : 0] : (double)(roff[res + 1] - roff[res]);
    for (int d = 0; d < 3; ++d)
      cref[d] = w != 0.0 ? ctr[CENTER ? (d + 1) * CR + res : 0] / w : 0.0;
  }
  if (big) entry(0);

  // Steps: a batch's centre sums (pass 0, when centred), then its RMSD sums
  // (pass 1), each over the stretches.  The next step's loads fly while the
  // terms of this one are added.
  constexpr int FIRST = CENTER ? 0 : 1;
  const int64_t stride = (int64_t)gridDim.x * FB;
  int pass = FIRST, base = 0;
  const bool busy = __builtin_amdgcn_readfirstlane(t) < ne;  // the wave has an atom
  for (;;) {
    const int nf = (int)(a.nframes - f0 < FB ? a.nframes - f0 : FB);
    __syncthreads();  // the last terms are read
#pragma unroll
    for (int j = 0; j < FB; ++j) {
      if (!CENTER && !busy) break;
      double x, y, z;
      if (!CENTER || big || pass == 0) {
        moved<MOD>(a, f0 + j < last ? f0 + j : last, p[j], x, y, z);
        if (CENTER) {  // kept for pass 1
          q[CENTER ? j : 0][0] = x;
          q[CENTER ? j : 0][1] = y;
          q[CENTER ? j : 0][2] = z;
        }
      } else {
        x = q[CENTER ? j : 0][0];
        y = q[CENTER ? j : 0][1];
        z = q[CENTER ? j : 0][2];
      }
      if (CENTER && pass == 0) {
        term[(j * NS) * LD + t] = a.use_mass ? x * m : x;
        term[(j * NS + (NS > 1 ? 1 : 0)) * LD + t] = a.use_mass ? y * m : y;
        term[(j * NS + NS - 1) * LD + t] = a.use_mass ? z * m : z;
      } else {
        if (CENTER) {
          const double* c = ctr + 3 * (j * CR + res);
          x = x - c[0];
          y = y - c[1];
          z = z - c[2];
        }
        const double dx = ry[0] - cref[0] - x, dy = ry[1] - cref[1] - y, dz = ry[2] - cref[2] - z;
        term[j * LD + t] = m * (dx * dx + dy * dy + dz * dz);
      }
      __builtin_amdgcn_sched_barrier(0);  // one frame's update in registers at a time
    }
    int64_t f1 = f0;
    int pass1 = pass, base1 = base + PERRES_ENTRIES;
    if (base1 >= ne) {
      base1 = 0;
      pass1 = pass == 0 ? 1 : FIRST;
      f1 = pass == 0 ? f0 : f0 + stride;
    }
    if (f1 < a.nframes && (big || pass == 1)) {
      if (big) entry(base1);
      fetch(f1);
    }
    __syncthreads();
    if (CENTER && pass == 0) {
      items(nf * NS, base, [&](int jd, int r, int b, int n) {
        sum = add_terms(base ? sum : 0.0, term + jd * LD + b, n);
        const int j = jd / NS;  // a compile-time 3
        const double w = a.use_mass ? total[r] : (double)(roff[r + 1] - roff[r]);
        ctr[CENTER ? 3 * (j * CR + r) + jd - j * NS : 0] = a.use_mass && w == 0.0 ? 0.0 : sum / w;
      });
    } else {
      items(nf, base, [&](int j, int r, int b, int n) {
        sum = add_terms(base ? sum : 0.0, term + j * LD + b, n);
        if (base + PERRES_ENTRIES < ne) return;  // more of the residue
        double val;
        if (total[r] < kSmall) val = -1.0;
        else if (sum < 0.0) val = 0.0;
        else val = sqrt(sum / total[r]);
        a.out[(f0 + j) * a.nres + r0 + r] = val;
      });
    }
    if (f1 >= a.nframes) break;
    f0 = f1;
    pass = pass1;
    base = base1;
  }
}

}  // namespace

size_t rmsd_perres_residue_bytes(int natoms, int span) {
  return sizeof(double) * (2 * 15 + (size_t)natoms + 3) + sizeof(float) * 3 * (size_t)natoms +
         sizeof(int) * (2 * (size_t)natoms + 2) + 2 * sizeof(float) * 3 * (size_t)span;
}

hipError_t rmsd_launch_perres(const PerresArgs& a, int npieces, hipStream_t s) {
  if (a.nframes == 0 || npieces == 0) return hipSuccess;
  if (npieces > 65535) return hipErrorInvalidValue;
  const int fb = a.center ? 4 : 16;  // the kernel's FB
  const int64_t batches = (a.nframes + fb - 1) / fb;
  // Enough workgroups to fill the chip a few times over; each walks batches.
  const int64_t want = (8192 + npieces - 1) / npieces;
  const dim3 grid((unsigned)(batches < want ? batches : want), npieces), block(PERRES_THREADS);
#define PERRES_CASE(M, C, S)                                                              \
  case M * 4 + C * 2 + S:                                                                 \
    hipLaunchKernelGGL((k_perres<M, C != 0, S != 0>), grid, block, 0, s, a);              \
    break
  switch (a.modify * 4 + (a.center ? 2 : 0) + (a.ld ? 1 : 0)) {
    PERRES_CASE(0, 0, 0); PERRES_CASE(0, 0, 1); PERRES_CASE(0, 1, 0); PERRES_CASE(0, 1, 1);
    PERRES_CASE(1, 0, 0); PERRES_CASE(1, 0, 1); PERRES_CASE(1, 1, 0); PERRES_CASE(1, 1, 1);
    PERRES_CASE(2, 0, 0); PERRES_CASE(2, 0, 1); PERRES_CASE(2, 1, 0); PERRES_CASE(2, 1, 1);
    default: return hipErrorInvalidValue;
  }
#undef PERRES_CASE
  return hipGetLastError();
}
