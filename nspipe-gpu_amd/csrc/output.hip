// State conversion and output kernels outside the time step: remesh onto
// another grid (tools/Re_Mesh), physical-space fields and the cross-section
// integrals of the reference's diagnostics files (mod_io_nonlinear.cu).
#include <algorithm>

#include "fft_device.h"
#include "nsp_internal.h"

namespace nsp {

using C = cpx<double>;

// Remesh gather (rmsh_k, tools/Re_Mesh/src/mod_remesh.cu:8-29, then
// modeZZ_k :34-40).  One thread per (new mode, component): a mode present
// on the old grid gets, at every new radial row, the remesh row's weights
// times the old column, summed over the row's nonzero band in increasing
// column order; other modes are zero.  ur, ut take the odd-in-r half for even
// m, uz the even half (parity index |(|m| mod 2) - flag|, flag 1 for ur, ut).
// A thread takes kRemeshRows new rows (blockIdx.z) with the old rows of a band
// loaded eight at a time and the weights through the scalar cache; as one walk
// of all rows with one load at a time the waves of present modes were a serial
// chain while the rest only wrote zeros.  Bound by the stores (0.6 of the 0.72
// GB of 48 x 96 x 513 to 64 x 192 x 1025): calls one after the other 322 us ->
// 258 -> 181 with the new state stored past the caches, which so keep the old
// rows that neighbouring chunks share (eight rows a chunk 194, sixteen 197); the
// kernel 290 -> 205 where the new state is copied out between calls.
constexpr int kRemeshRows = 4;
__global__ __launch_bounds__(256) void remesh_kernel(Geom gn, Geom go, const double* __restrict__ RM,
                                                     const int2* __restrict__ band,
                                                     const double2* __restrict__ uo, double2* __restrict__ un) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (k >= gn.modes) return;
  const int it = k / gn.nz, l = k - it * gn.nz;
  const int m = it < gn.nt / 2 ? it : it - gn.nt;
  const bool src = m >= -go.nt / 2 && m < go.nt / 2 && l < go.nz;
  const int ko = src ? (m >= 0 ? m : m + go.nt) * go.nz + l : 0;
  const int par = abs((abs(m) % 2) - (c < 2 ? 1 : 0));
  const ctab R = ctab(RM);  // scalar loads: both parities' weights, selected per lane
  const size_t odd = (size_t)gn.nr * go.nr;
  const double2* col = uo + (size_t)c * go.n + ko;
  double2* dst = un + (size_t)c * gn.n + k;
  const int i0 = blockIdx.z * kRemeshRows, i1 = min(i0 + kRemeshRows, gn.nr);
  for (int i = i0; i < i1; i++) {
    double2 v = make_double2(0.0, 0.0);
    if (src) {
      const int2 bd = band[i];
      for (int j = bd.x; j <= bd.y; j += 8) {
        double2 a[8];
#pragma unroll
        for (int q = 0; q < 8; q++)
          if (j + q <= bd.y) a[q] = col[(size_t)(j + q) * go.modes];
#pragma unroll
        for (int q = 0; q < 8; q++) {
          if (j + q <= bd.y) {
            const size_t e = (size_t)i * go.nr + j + q;
            const double w = par ? R[odd + e] : R[e];
            v.x += w * a[q].x;
            v.y += w * a[q].y;
          }
        }
      }
    }
    if (k == 0) {  // mode (0,0): no radial velocity, real ut and uz
      if (c == 0) v = make_double2(0.0, 0.0);
      else v.y = 0.0;
    }
    store_nt(dst + (size_t)i * gn.modes, v);
  }
}

void launch_remesh(const Geom& gn, const Geom& go, const double* RM, const int2* band, const double2* uo,
                   double2* un, hipStream_t s) {
  const dim3 grid((gn.modes + 255) / 256, 3, (gn.nr + kRemeshRows - 1) / kRemeshRows);
  remesh_kernel<<<grid, 256, 0, s>>>(gn, go, RM, band, uo, un);
}

// ------------------------------------------------------------------ physical space
// padForward_k (mod_io_nonlinear.cu:173-192) and the theta pass of the 2-D
// inverse transform (mod_fft.cu:43-49) for one spectral component: block
// (l-tile, i) transforms TL axial columns of level i; rows it < NT/2 go to
// padded row it, the others to it + NT/2, rows NT/2..NT-1 stay zero.  As many
// columns as leave two workgroups a CU (launch_physical): 16 make a row's piece
// 256 bytes and a pass's butterflies as many as the threads; 48 levels of
// 96 x 513: 44 us with 4 columns -> 27.
template <int TL>
__global__ __launch_bounds__(256) void phys_theta_kernel(Geom g, FftPlan P, const int* __restrict__ perm,
                                                         const C* __restrict__ tw, const double2* __restrict__ u,
                                                         double2* __restrict__ Wt) {
  extern __shared__ double2 smem[];
  C* buf = reinterpret_cast<C*>(smem);
  const int l0 = blockIdx.x * TL, i = blockIdx.y;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int half = g.nt / 2;
  const double2* src = u + (size_t)i * g.modes;
  for (int e = tid; e < g.ntp * TL; e += nthr) {
    const int j = e / TL, tl = e - j * TL, l = l0 + tl;
    double2 v = make_double2(0.0, 0.0);
    if ((j < half || j >= g.nt) && l < g.nz) v = src[(size_t)(j < half ? j : j - half) * g.nz + l];
    buf[lds_pos<TL>(perm[j] * TL + tl)] = C{v.x, v.y};
  }
  __syncthreads();
  fft_passes<double, TL, +1>(buf, P, tw, tid, nthr);
  double2* dst = Wt + (size_t)i * g.ntp * g.nz;
  for (int e = tid; e < g.ntp * TL; e += nthr) {
    const int j = e / TL, tl = e - j * TL, l = l0 + tl;
    const C w = buf[lds_pos<TL>(e)];
    if (l < g.nz) dst[(size_t)j * g.nz + l] = make_double2(w.x, w.y);
  }
}

// Axial real synthesis of two rows of one level of Wt (the last of an odd
// number is alone) as one complex transform of length NZF: with spectra X, Y
// (imaginary parts of X[0], Y[0] ignored, zero from NZ on),
//   Z[l] = X[l] + i Y[l],  Z[NZF-l] = conj(X[l]) + i conj(Y[l])
// gives the samples of X as real and those of Y as imaginary parts.  Both are
// rounded at the scale of the larger: rows of one level are of one scale,
// while a row of the wall's zeros beside one of the level inside would take
// that row's rounding.  A row of out (pitch doubles) receives the samples, then
// zeros up to the pitch.  Bound by the passes' LDS round trips; 6912 rows of
// 1536: 57 us one row a workgroup (half-length transforms, radices to 5) -> 46.
__global__ __launch_bounds__(512) void phys_z_kernel(Geom g, FftPlan P, const int* __restrict__ perm,
                                                     const C* __restrict__ tw, const double2* __restrict__ Wt,
                                                     double* __restrict__ out, size_t pitch) {
  extern __shared__ double2 smem[];
  C* buf = reinterpret_cast<C*>(smem);
  const int pairs = (g.ntp + 1) / 2, lev = blockIdx.x / pairs, th = 2 * (blockIdx.x - lev * pairs);
  const int row = lev * g.ntp + th;
  const bool two = th + 1 < g.ntp;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int nz = g.nz, nzf = g.nzf;
  const double2* X = Wt + (size_t)row * nz;
  for (int l = tid; l < nz; l += nthr) {
    double2 a = X[l], b = make_double2(0.0, 0.0);
    if (two) b = X[nz + l];
    if (l == 0) a.y = b.y = 0.0;
    buf[lds_pos<kPadCol>(perm[l])] = C{a.x - b.y, a.y + b.x};
    if (l > 0) buf[lds_pos<kPadCol>(perm[nzf - l])] = C{a.x + b.y, b.x - a.y};
  }
  for (int k = nz + tid; k <= nzf - nz; k += nthr) buf[lds_pos<kPadCol>(perm[k])] = C{0.0, 0.0};
  __syncthreads();
  fft_passes<double, kPadCol, +1>(buf, P, tw, tid, nthr);
  double* o = out + (size_t)row * pitch;
  for (int n = tid; n < (int)pitch; n += nthr) {
    C v{0.0, 0.0};
    if (n < nzf) v = buf[lds_pos<kPadCol>(n)];
    o[n] = v.x;
    if (two) o[pitch + n] = v.y;
  }
}

// Cross-section integrals of u^2 (q0kernel_k, u0kernel_k and q1kernel_k,
// mod_io_nonlinear.cu:54-103, intq, mod_cublasflux.cu:119-130).  The sum over
// theta of the reference's periodic three-point rule is the mean over the NTP
// points, and NTP >= 3 NT/2 points take the mean of a square exactly, so it
// follows mode by mode, without the theta transform and the physical field:
//   u(theta, n) = e_0(n) + 2 Re sum_{m>0} e^{i m theta} e_m(n),
//   mean u^2 = |e_0|^2 + 2 sum_{m>0} |e_m|^2,
// where e_m is the complex axial transform of the modes m and -m together,
// S[l] = X_m[l], S[NZF-l] = conj(X_-m[l]), S[0] = (X_m[0] + conj(X_-m[0]))/2
// (m = NT/2: only -m is stored).  A workgroup sums |e_m|^2 with the weights
// rdr over its rows (level, m) in registers, then stores one partial row; the
// next row's modes are in flight during a transform.  About 12 samples a
// thread: a pass of radix 12 or 16 then has a butterfly for most threads.
// Bound by the passes' LDS round trips at two waves a SIMD (228 registers; at
// three, with a few of them in memory, 1.2 to 1.4 times as long).  Both
// integrals of 48 x 96 x 513: 0.42 ms through the physical fields -> 0.096.
template <int MPT>
__global__ __launch_bounds__(512) void cross_kernel(Geom g, FftPlan P, const int* __restrict__ perm,
                                                    const C* __restrict__ tw, const double2* __restrict__ u,
                                                    const double* __restrict__ rdr, double* __restrict__ part) {
  extern __shared__ double2 smem[];
  C* buf = reinterpret_cast<C*>(smem);
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int nz = g.nz, nzf = g.nzf, half = g.nt / 2, nm = half + 1, rows = g.nr * nm;
  const double2* src = u + (size_t)blockIdx.y * g.n;
  constexpr int LP = MPT / 3 + 1;  // LP nthr >= NZ (MPT nthr >= 3(NZ-1))
  double2 A[LP], B[LP];
  int pa[LP], pb[LP], pz[LP];  // LDS positions of l, NZF-l and the zeros between, the same for every row
#pragma unroll
  for (int q = 0; q < LP; q++) {
    const int l = tid + q * nthr, k = nz + l;
    pa[q] = lds_pos<kPadCol>(perm[min(l, nz - 1)]);
    pb[q] = lds_pos<kPadCol>(perm[nzf - max(1, min(l, nz - 1))]);
    pz[q] = k <= nzf - nz ? lds_pos<kPadCol>(perm[k]) : -1;
  }
  auto load = [&](int row) {
    const int i = row / nm, m = row - i * nm;
    const double2* lev = src + (size_t)i * g.modes;
#pragma unroll
    for (int q = 0; q < LP; q++) {
      const int l = tid + q * nthr;
      A[q] = B[q] = make_double2(0.0, 0.0);
      if (l < nz) {
        if (m < half) A[q] = lev[(size_t)m * nz + l];
        B[q] = lev[(size_t)(m ? g.nt - m : 0) * nz + l];
      }
    }
  };
  double acc[MPT] = {};
  int row = blockIdx.x;
  if (row < rows) load(row);
  for (; row < rows; row += gridDim.x) {
    const int i = row / nm;
    const double w = (row == i * nm ? 1.0 : 2.0) * rdr[i];
#pragma unroll
    for (int q = 0; q < LP; q++) {
      const int l = tid + q * nthr;
      const double2 a = A[q], b = B[q];
      if (l == 0) {
        buf[pa[q]] = C{0.5 * (a.x + b.x), 0.5 * (a.y - b.y)};
      } else if (l < nz) {
        buf[pa[q]] = C{a.x, a.y};
        buf[pb[q]] = C{b.x, -b.y};
      }
      if (pz[q] >= 0) buf[pz[q]] = C{0.0, 0.0};
    }
    if (row + (int)gridDim.x < rows) load(row + gridDim.x);
    __syncthreads();
    fft_passes<double, kPadCol, +1>(buf, P, tw, opaque(tid), nthr);
#pragma unroll
    for (int q = 0; q < MPT; q++) {
      const int n = tid + q * nthr;
      if (n < nzf) {
        const C e = buf[lds_pos<kPadCol>(n)];
        acc[q] += w * (e.x * e.x + e.y * e.y);
      }
    }
    __syncthreads();
  }
  double* dst = part + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * nzf;
#pragma unroll
  for (int q = 0; q < MPT; q++) {
    const int n = tid + q * nthr;
    if (n < nzf) dst[n] = acc[q];
  }
}

// Sums of the partial rows: out[n] over the first n0 rows, out[nzf + n] over the
// rows n0 .. n1 (blockIdx.y).  16 samples by 16 rows at a time per workgroup.
__global__ __launch_bounds__(256) void cross_sum_kernel(int nzf, int n0, int n1, const double* __restrict__ part,
                                                        double* __restrict__ out) {
  __shared__ double sm[16][17];
  const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
  const int n = blockIdx.x * 16 + x;
  const int b0 = blockIdx.y ? n0 : 0, b1 = blockIdx.y ? n1 : n0;
  double acc = 0.0;
  if (n < nzf) {
#pragma unroll 4
    for (int b = b0 + y; b < b1; b += 16) acc += part[(size_t)b * nzf + n];
  }
  sm[y][x] = acc;
  __syncthreads();
  if (y == 0 && n < nzf) {
#pragma unroll
    for (int k = 1; k < 16; k++) acc += sm[k][x];
    out[(size_t)blockIdx.y * nzf + n] = acc;
  }
}

// real part of uz at mode (0,0) of every level (wrt_mnp_k)
__global__ __launch_bounds__(256) void profile_kernel(Geom g, const double2* __restrict__ u, double* __restrict__ out) {
  for (int i = threadIdx.x; i < g.nr; i += blockDim.x) out[i] = u[2 * g.n + (size_t)i * g.modes].x;
}

// threads of the full-length axial kernels: about 12 samples each
static int axial_threads(const Geom& g, int mpt) { return 64 * ((g.nzf + 64 * mpt - 1) / (64 * mpt)); }

template <int TL>
static void run_phys_theta(const Geom& g, const NlBufs& nb, const double2* u, double2* Wt, hipStream_t s) {
  const size_t lds = size_t(g.ntp) * TL * sizeof(double2);
  (void)hipFuncSetAttribute((const void*)phys_theta_kernel<TL>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  phys_theta_kernel<TL><<<dim3((g.nz + TL - 1) / TL, g.nr), 256, lds, s>>>(g, nb.pt, nb.perm_t, (const C*)nb.tw_t, u,
                                                                           Wt);
}

void launch_physical(const Geom& g, const NlBufs& nb, const double2* u, double2* Wt, double* out, size_t pitch,
                     hipStream_t s) {
  const size_t col = size_t(g.ntp) * sizeof(double2), lim = 81920;  // two workgroups' LDS a CU
  if (col * 16 <= lim) run_phys_theta<16>(g, nb, u, Wt, s);
  else if (col * 8 <= lim) run_phys_theta<8>(g, nb, u, Wt, s);
  else if (col * 4 <= lim) run_phys_theta<4>(g, nb, u, Wt, s);
  else if (col * 2 <= lim) run_phys_theta<2>(g, nb, u, Wt, s);
  else run_phys_theta<1>(g, nb, u, Wt, s);
  const size_t lz = size_t(lds_pos<kPadCol>(g.nzf)) * sizeof(double2);
  (void)hipFuncSetAttribute((const void*)phys_z_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lz);
  phys_z_kernel<<<g.nr * ((g.ntp + 1) / 2), axial_threads(g, g.nzf > 6144 ? 18 : 12), lz, s>>>(
      g, nb.pf, nb.perm_f, (const C*)nb.tw_f, Wt, out, pitch);
}

template <int MPT>
static void run_cross(const Geom& g, const NlBufs& nb, const double2* u, const double* rdr, double* part, int blocks,
                      int fields, hipStream_t s) {
  const size_t lds = size_t(lds_pos<kPadCol>(g.nzf)) * sizeof(double2);
  (void)hipFuncSetAttribute((const void*)cross_kernel<MPT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  cross_kernel<MPT><<<dim3(blocks, fields), axial_threads(g, MPT), lds, s>>>(g, nb.pf, nb.perm_f, (const C*)nb.tw_f, u,
                                                                             rdr, part);
}

// At most 512 workgroups a field (six a CU for all three), one partial row each.
void launch_cross(const Geom& g, const NlBufs& nb, const double2* u, const double* rdr, double* part, size_t room,
                  double* out, bool q, bool u2, hipStream_t s) {
  const int fields = (q ? 2 : 0) + (u2 ? 1 : 0);
  const int blocks = (int)std::min<size_t>(std::min(512, g.nr * (g.nt / 2 + 1)), room / ((size_t)fields * g.nzf));
  const double2* f = q ? u : u + 2 * g.n;
  if (g.nzf <= 256) run_cross<4>(g, nb, f, rdr, part, blocks, fields, s);
  else if (g.nzf <= 6144) run_cross<12>(g, nb, f, rdr, part, blocks, fields, s);
  else run_cross<18>(g, nb, f, rdr, part, blocks, fields, s);
  const int n0 = q ? 2 * blocks : blocks;
  cross_sum_kernel<<<dim3((g.nzf + 15) / 16, q && u2 ? 2 : 1), 256, 0, s>>>(g.nzf, n0, fields * blocks, part, out);
}

void launch_profile(const Geom& g, const double2* u, double* out, hipStream_t s) {
  profile_kernel<<<1, 256, 0, s>>>(g, u, out);
}

}  // namespace nsp
