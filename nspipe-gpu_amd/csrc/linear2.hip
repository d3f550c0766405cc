// Linear phase, streaming form: one thread per Fourier mode, four passes
// over the radial column with sliding register windows.
//
//   A (up)   rhs = E + d_im N (corrector) or N + CN part of u^n (predictor,
//            which also stores the explicit part E); to r/theta; divergence
//            (div_k, zero wall row); forward elimination of the pressure system
//   B (down) pressure back substitution (p overwrites its eliminated rhs)
//   C (up)   rhs -= grad p three rows behind (addGrad_k); to +/-; zero wall
//            rows (write_bcon_k); forward elimination of the u+, u-, uz systems
//   D (down) back substitution of u+, u-, uz together with the homogeneous
//            wall-unit solutions; the wall divergence of the four wall rows
//            fixes the influence coefficients (corBCon); a second walk from
//            the wall applies them row by row; to r/theta; convergence
//            measure (mcor_k) and output.  Mode (0,0) then takes modeZZ_k
//            and the flux correction (adj_flux).
//
// The banded LU factors of the four operators depend only on (m, kz), dt and
// Re, so they are computed once at setup with the reference's recurrence
// (LUsolve_*_k, mod_linear.cu:55-646) and stored per workgroup, 7 per row
// (fidx): every access of a wavefront is one contiguous line.  (Recomputing the L
// multipliers in the upward passes saves 3 of the 7 but needs the U window of
// three operators in registers, which halves occupancy: slower.)
// Workgroups pair the modes m and -m of one axial chunk: the u- factors at m
// are the u+ factors at -m (bit for bit: the operators differ only in the sign
// of the 2m/r^2 term) and the uz and pressure factors and the pressure
// homogeneous solution depend on |m|, so both waves read the same lines.
// Scratch SR (3 complex per row) and SP (1 complex per row) carry the column
// between passes.  Scratch, E, the factors and PH are stored per workgroup
// (sweep-side layout, nsp_internal.h): a workgroup's column is contiguous.
#include <algorithm>

#include "nsp_internal.h"

namespace nsp {

struct ModeQ {
  int k, it, l, m;
  double kt, kz;
};

__device__ __forceinline__ ModeQ modeq(const Geom& g, int k) {
  ModeQ q;
  q.k = k;
  q.it = k / g.nz;
  q.l = k - q.it * g.nz;
  q.m = q.it < g.nt / 2 ? q.it : q.it - g.nt;
  q.kt = double(q.m);
  q.kz = g.kz0 * double(q.l);
  return q;
}

__device__ __forceinline__ void pm_of(double2& a, double2& b) {  // decoupleForward_k
  const double2 ur = a, ut = b;
  a = make_double2(ur.x - ut.y, ur.y + ut.x);
  b = make_double2(ur.x + ut.y, ur.y - ut.x);
}
__device__ __forceinline__ void rt_of(double2& a, double2& b) {  // decoupleBackward_k
  const double2 up = a, um = b;
  a = make_double2(0.5 * (up.x + um.x), 0.5 * (up.y + um.y));
  b = make_double2(0.5 * (up.y - um.y), -0.5 * (up.x - um.x));
}

// factor slot c of operator `kind` at row i: c 0..2 = L multipliers of
// columns i-3..i-1, 3 = 1/U_ii, 4..6 = U_{i,i+1..i+3}.  Only the factors the
// sweep reads are stored, in the sweep-side layout:
//   u+ (kind 0), every mode:          [workgroup][NR][7][128 lanes]
//   u- (kind 1), azimuthal row NT/2:  [chunk][NR][7][128] (lanes 64..127);
//                elsewhere u- at m is u+ at -m, the other wave of the workgroup
//   uz, p (kinds 2, 3), rows it <= NT/2 (they depend on |m|):
//                                     [workgroup or Nyquist chunk][NR][7][64] each
// Per row the u+/u- sets step by FR_UP = 7*128 doubles and per slot by 128,
// the uz/p sets by FR_ABS = 7*64 and 64.
constexpr int FR_UP = 7 * 128, FR_ABS = 7 * 64;
__host__ __device__ __forceinline__ size_t f_u1(const Geom& g) { return sw_nblk(g) * g.nr * FR_UP; }
__host__ __device__ __forceinline__ size_t f_abs(const Geom& g) {
  return f_u1(g) + (size_t)sw_nch(g) * g.nr * FR_UP;
}
__host__ __device__ __forceinline__ size_t f_absn(const Geom& g) {  // doubles of one |m| set
  return (sw_nblk(g) + sw_nch(g)) * g.nr * FR_ABS;
}
__host__ __device__ __forceinline__ size_t fidx(const Geom& g, int kind, int i, int c, int k) {
  const int it = k / g.nz, l = k - it * g.nz, nth = g.nt / 2;
  if (kind == 0) {
    const int pair = it < nth ? it : (it == nth ? 0 : g.nt - it), w = it < nth ? 0 : 1;
    const size_t lb = (size_t)pair * sw_nch(g) + (l >> 6);
    return ((lb * g.nr + i) * 7 + c) * 128 + w * 64 + (l & 63);
  }
  if (kind == 1) return f_u1(g) + (((size_t)(l >> 6) * g.nr + i) * 7 + c) * 128 + 64 + (l & 63);
  return f_abs(g) + (size_t)(kind - 2) * f_absn(g) + sw_abs_idx(g, 7, i, c, k);
}

// The operator rows of one mode (LUsolve_*_k): kind 0 u+, 1 u-, 2 uz
// (velocity Helmholtz, (1/dt) I - (d_im/Re)(Lu + diag)), 3 pressure (Lp + diag;
// mode (0,0) has the wall row p = 0).
struct OpMode {
  const double* LHS;
  int ip0, kind;
  bool vel, p00;
  double a, idt, kt, kz;
};
__device__ __forceinline__ OpMode op_mode(const Geom& g, const double* Lu, const double* Lp, int kind, int m, int l) {
  OpMode o;
  o.kind = kind;
  o.LHS = (kind == 3) ? Lp : Lu;
  const int fp = (kind <= 1) ? 1 : 0;
  o.ip0 = abs((abs(m) % 2) - fp) * STEN * g.nr;
  o.vel = kind < 3;
  o.p00 = (kind == 3) && (l == 0 && m == 0);
  o.a = g.d_im / g.re;
  o.idt = 1.0 / g.dt;
  o.kt = double(m);
  o.kz = g.kz0 * double(l);
  return o;
}

// Row i of the reference recurrence without the right-hand side.  Uw[s] is
// the U row i-3+s (s = 2: row i-1), diagonal first.  Out: Lc[c] = multiplier
// of column i-3+c (0 where the column is outside the band), Ui = U row i.
// NL = min(i, 3) is the number of columns left of the diagonal; it is a
// template parameter so that every register index is a constant.
// Contraction is off so every caller gets the same bits.
template <int NL>
__device__ __forceinline__ void factor_row_nl(const OpMode& o, int nr, int i, double ri, const double (&Uw)[IW][IW + 1],
                                              double (&Lc)[IW], double (&Ui)[IW + 1]) {
#pragma clang fp contract(off)
  const int right = min(i + IW, nr - 1);
  const int i0 = i + IW - right;
  const double r2 = ri * ri;
  const bool last = (i == nr - 1);
  const double* row = o.LHS + o.ip0 + STEN * i + i0;  // row[j] = entry of column left + j
  double L[IW];
#pragma unroll
  for (int j = 0; j < IW; j++) {
    L[j] = 0.0;
    if (j < NL) {
      double XM = row[j];
      if (!last) {
        if (o.vel) XM = -o.a * XM;
      } else if (o.p00) {
        XM = 0.0;
      }
      double Lj = XM;
      // U row of column left+h lives at Uw[IW - NL + h]
#pragma unroll
      for (int h = 0; h < IW; h++)
        if (h < j) Lj -= L[h] * Uw[IW - NL + h][j - h];
      Lj = Lj / Uw[IW - NL + j][0];
      L[j] = Lj;
    }
  }
#pragma unroll
  for (int j = 0; j <= IW; j++) {
    Ui[j] = 0.0;
    if (j < right - i + 1) {
      double XM = row[NL + j];
      if (!last) {
        if (j == 0) {
          const double kt = o.kt, kz = o.kz;
          if (o.kind == 0) XM += -(1.0 / r2) - (2.0 * kt / r2) - kz * kz - kt * kt / r2;
          else if (o.kind == 1) XM += -(1.0 / r2) + (2.0 * kt / r2) - kz * kz - kt * kt / r2;
          else XM += -kz * kz - kt * kt / r2;
          if (o.vel) XM = o.idt - o.a * XM;
        } else if (o.vel) {
          XM = -o.a * XM;
        }
      } else if (o.p00) {
        XM = (j == 0) ? 1.0 : 0.0;
      }
      const int hleft = (NL + j - IW) > 0 ? (NL + j - IW) : 0;
      double Uij = XM;
#pragma unroll
      for (int h = 0; h < IW; h++)
        if (h >= hleft && h < NL) Uij -= L[h] * Uw[IW - NL + h][j + NL - h];
      Ui[j] = Uij;
    }
  }
#pragma unroll
  for (int c = 0; c < IW; c++) Lc[c] = (c - (IW - NL) >= 0) ? L[(c - (IW - NL)) >= 0 ? c - (IW - NL) : 0] : 0.0;
}

__device__ __forceinline__ void factor_row(const OpMode& o, int nr, int i, double ri, const double (&Uw)[IW][IW + 1],
                                           double (&Lc)[IW], double (&Ui)[IW + 1]) {
  if (i >= IW) factor_row_nl<IW>(o, nr, i, ri, Uw, Lc, Ui);
  else if (i == 2) factor_row_nl<2>(o, nr, i, ri, Uw, Lc, Ui);
  else if (i == 1) factor_row_nl<1>(o, nr, i, ri, Uw, Lc, Ui);
  else factor_row_nl<0>(o, nr, i, ri, Uw, Lc, Ui);
}

__device__ __forceinline__ void shift_u(double (&Uw)[IW][IW + 1], const double (&Ui)[IW + 1]) {
#pragma unroll
  for (int s = 0; s < IW - 1; s++)
#pragma unroll
    for (int j = 0; j <= IW; j++) Uw[s][j] = Uw[s + 1][j];
#pragma unroll
  for (int j = 0; j <= IW; j++) Uw[IW - 1][j] = Ui[j];
}

// ------------------------------------------------------------------ factors
__global__ __launch_bounds__(256) void factor_kernel(Geom g, const double* __restrict__ r,
                                                     const double* __restrict__ Lu,
                                                     const double* __restrict__ Lp, double* __restrict__ F,
                                                     float* __restrict__ F32) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int kind = blockIdx.y;
  if (k >= g.modes) return;
  const ModeQ q = modeq(g, k);
  if (kind == 1 && q.it != g.nt / 2) return;  // stored factor sets only (fidx)
  if (kind >= 2 && q.it > g.nt / 2) return;
  const OpMode o = op_mode(g, Lu, Lp, kind, q.m, q.l);
  double Uw[IW][IW + 1];
#pragma unroll
  for (int s = 0; s < IW; s++)
#pragma unroll
    for (int j = 0; j <= IW; j++) Uw[s][j] = 0.0;
  for (int i = 0; i < g.nr; i++) {
    double Lc[IW], Ui[IW + 1];
    factor_row(o, g.nr, i, r[i], Uw, Lc, Ui);
    double fv[7];
#pragma unroll
    for (int c = 0; c < IW; c++) fv[c] = Lc[c];
    fv[3] = 1.0 / Ui[0];
#pragma unroll
    for (int j = 1; j <= IW; j++) fv[3 + j] = Ui[j];
#pragma unroll
    for (int c = 0; c < 7; c++) {
      F[fidx(g, kind, i, c, k)] = fv[c];
      if (F32 && kind <= 2) F32[fidx(g, kind, i, c, k)] = float(fv[c]);
    }
    shift_u(Uw, Ui);
  }
}

// Column scratch of one workgroup at FP64, or (mixed form, |m| >= m32) as
// FP32 pairs.  Both are indexed with the FP64 sweep-side indices; the FP32
// view is offset by the workgroup region's first FP64 index, so its values
// fill the first half of the workgroup's own region.
// NT: streamed accesses, past the caches' usual replacement (sweep_kernel).
template <bool S32, bool NT>
struct Scr;
template <bool NT>
struct Scr<false, NT> {
  double2* p;
  __device__ static Scr at(double2* base, size_t) { return Scr{base}; }
  using V = double2;
  __device__ V raw(size_t i) const {
    if constexpr (NT) return load_nt(p + i);
    else return p[i];
  }
  __device__ double2 ld(size_t i) const { return raw(i); }
  __device__ void st(size_t i, double2 v) const {
    if constexpr (NT) store_nt(p + i, v);
    else p[i] = v;
  }
};
template <bool NT>
struct Scr<true, NT> {
  float2* p;
  __device__ static Scr at(double2* base, size_t region0) { return Scr{reinterpret_cast<float2*>(base) + region0}; }
  using V = float2;
  __device__ V raw(size_t i) const {
    if constexpr (NT) return load_nt(p + i);
    else return p[i];
  }
  __device__ double2 ld(size_t i) const {
    const float2 v = raw(i);
    return make_double2(v.x, v.y);
  }
  __device__ void st(size_t i, double2 v) const {
    if constexpr (NT) store_nt(p + i, make_float2(float(v.x), float(v.y)));
    else p[i] = make_float2(float(v.x), float(v.y));
  }
};

__device__ __forceinline__ double2 wide(double2 v) { return v; }
__device__ __forceinline__ double2 wide(float2 v) { return make_double2(v.x, v.y); }

constexpr int kLatRing = 3;

// Walks rows t0, t0 + DIR, ... (t1 excluded) whose first PD are loaded in ring.
template <int PD, int DIR, typename Row, typename L, typename F>
__device__ __forceinline__ void walk_ring(Row (&ring)[PD], int t0, int t1, L&& load, F&& work) {
  int t = t0;
  for (; DIR * (t1 - t) >= PD; t += DIR * PD) {
#pragma unroll
    for (int q = 0; q < PD; q++) {
      const Row cur = ring[q];
      load(t + DIR * (q + PD), ring[q]);
      work(t + DIR * q, cur);
    }
  }
#pragma unroll
  for (int q = 0; q < PD - 1; q++)
    if (DIR * (t1 - t) > q) work(t + DIR * q, ring[q]);
}

// Walks rows t0, t0 + DIR, ... (t1 excluded): load(t, row) issues a row's loads
// (it clamps rows beyond the grid), work(t, row) does its arithmetic and
// stores.  PD = 0 loads each row as it is reached; PD > 0 keeps the loads of
// PD rows in flight (a ring of rows in registers).
template <int PD, int DIR, typename Row, typename L, typename F>
__device__ __forceinline__ void walk_rows(int t0, int t1, L&& load, F&& work) {
  if constexpr (PD == 0) {
    for (int t = t0; t != t1; t += DIR) {
      Row r;
      load(t, r);
      work(t, r);
    }
  } else {
    Row ring[PD];
#pragma unroll
    for (int q = 0; q < PD; q++) load(t0 + DIR * q, ring[q]);
    walk_ring<PD, DIR>(ring, t0, t1, load, work);
  }
}
// x / d from d's two-word reciprocal (recip_table): x hi + x lo, rounded once but
// for 2^-104 of it, so the quotient of an IEEE division except where that lies
// within 2^-51 of an ulp of a tie.
__device__ __forceinline__ double times_recip(double x, double2 r) { return __builtin_fma(x, r.x, x * r.y); }

// Rounds a value where it is formed: the compiler does not fuse it with its use.
__device__ __forceinline__ void fix(double& x) { asm volatile("" : "+v"(x)); }

// A radial table: through the scalar cache, or (LAT kernels) from LDS.
template <int LAT>
struct Tab {
  ctab g;
  __device__ double operator[](int i) const { return g[i]; }
  __device__ Tab operator+(int o) const { return Tab{g + o}; }
};
template <>
struct Tab<1> {
  const double* l;
  __device__ double operator[](int i) const { return l[i]; }
  __device__ Tab operator+(int o) const { return Tab{l + o}; }
};

// ------------------------------------------------------------------ sweep
// Workgroup = 2 waves: azimuthal rows it and NT - it (0 with NT/2) over one
// chunk of 64 axial modes.  One kernel per pass (PASS 0..3 = A..D): the
// column moves between passes through SR/SP in any case, and each pass then
// gets its own register allocation (and occupancy).
// B = 1: batched launch, one pipe per blockIdx.y with its arguments from tab
// (the single-pipe form B = 0 reads only its own argument block).
// HOLD (pass D): 1 keeps the four wall rows in registers across the
// coefficient solve, 0 walks them twice (fewer registers, one more wave per
// SIMD). The FP64 form is faster with the first, the mixed form with the
// second. The two compile to different instruction sequences (contraction),
// so a pipe's form fixes which one it runs, batched or not.
// INC = 1 (refined mixed form, single pipes): the velocity solves are for the
// increment delta = u^{k+1} - u^n, whose right-hand side is formed in FP64 from
// small quantities, so the FP32 column storage of |m| >= m32 rounds delta,
// not u (one step of iterative refinement from u^n):
//   A1 (PASS 4, predictor only): E' = (1/Re) L'u^n + (1 - d_im) N(u^n) and
//        Dh = div(H u^n) with H u^n = u^n/dt - (d_im/Re) L'u^n, L' = Lu + diag
//        (addLap_k's operator), for every row;
//   A:   rhs' = E' + d_im N(u^k) = rhs - H u^n; div(rhs) = div(rhs') + Dh;
//   C:   wall rows -u^n (so that u^n + delta vanishes there);
//   D:   back substitution gives delta; u^n + delta takes the place of the
//        solution from there on (wall divergence, correction, output).
// LAT = 1 (grids with few workgroups, kSweepLat): the walk is bound by the
// latency of each row's loads and of its arithmetic, not by bandwidth, and
// registers cost nothing (less than one wave per SIMD).  Each pass then keeps
// the loads of kLatRing rows in flight, reads the radial tables from an LDS
// copy (a first touch of a table row through the scalar cache is another
// memory round trip per row) and multiplies by tabled reciprocals of two words
// (of one word, a rounding more per quotient, 24x64x65 took 92 / 93 instead of 94 /
// 95 us and larger grids the same).  Pass D holds the wall rows
// (as HOLD = 1).  The results are the general kernels', bit for bit.
// General / LAT, us, predictor and corrector: 24x64x65 FP64 118 / 94 and 121 /
// 95, 64x64x385 FP64 400 / 248 and 437 / 293, refined 419 / 271 and 372 / 291,
// 64x128x385 FP64 517 / 427 and 543 / 492, mixed 415 / 328 and 461 / 376 (a
// ring of 2 rows is equal, of 1 or 4 slower; pass B keeps 8 rows in flight).
// LAP: the passes that apply the Laplacian (Lu, 1/r^2).
template <int PASS, int PRED, int INC>
constexpr bool lat_lap() {
  return PASS == 4 || (PASS == 0 && PRED && !INC);
}
// small (B): takes the members whose own grid is small, or the others.  (In an
// argument of its own: read from A, it made every access a flat one.)
template <int PASS, int PRED, int B, int HOLD = 0, int INC = 0, int LAT = 0, int STR = 0>
__global__ __launch_bounds__(128) void sweep_kernel(Lin2Args A, const Lin2Args* tab, int small) {
  // LAT, not pass B: reciprocals of r [nr] and, LAP, of r^2 [nr], D [2][nr][7], LAP: Lu [2][nr][7]
  extern __shared__ double2 lat_tab[];
  constexpr bool LAP = lat_lap<PASS, PRED, INC>();
  if constexpr (B != 0) {
    A = tab[blockIdx.y];
    if (A.small != small) return;  // the other launch's
    A.r = gmem(tab, A.r);
    A.rr = gmem(tab, A.rr);
    A.rdr = gmem(tab, A.rdr);
    A.uc = gmem(tab, A.uc);
    A.qc = gmem(tab, A.qc);
    A.Dc = gmem(tab, A.Dc);
    A.Luc = gmem(tab, A.Luc);
    A.Lu = gmem(tab, A.Lu);
    A.Lp = gmem(tab, A.Lp);
    A.F = gmem(tab, A.F);
    if (A.F32) A.F32 = gmem(tab, A.F32);  // nullable: tested before re-deriving
    A.PH = gmem(tab, A.PH);
    A.invc = gmem(tab, A.invc);
    A.N = gmem(tab, A.N);
    A.E = gmem(tab, A.E);
    A.u = gmem(tab, A.u);
    A.out = gmem(tab, A.out);
    A.SR = gmem(tab, A.SR);
    A.SP = gmem(tab, A.SP);
    A.norm = gmem(tab, A.norm);
    if constexpr (PASS == 3 && !LAT) {  // members of the other form are the other launch's
      // The form is tested on a copy the compiler cannot see through: knowing
      // the form past this test would let it drop the other form's paths
      // and then contract the remaining arithmetic differently from the
      // single-pipe kernel, whose results the batched one must match bit for bit.
      int fp64 = __builtin_amdgcn_readfirstlane(A.form64 ? 1 : 0);
      asm volatile("" : "+s"(fp64));
      if (HOLD != fp64) return;
    }
  }
  const Geom& g = A.g;
  if (step_done(g)) return;
  const int nch = (g.nz + 63) / 64;
  // ord 1: the chunks of one azimuthal row, adjacent in memory, run in one XCD's L2
  const int lb = A.ord ? xcd_block(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const int pair = lb / nch, ch = lb - pair * nch;
  if (pair >= g.nt / 2) return;  // beyond this pipe's extent
  const int nth = g.nt / 2;
  const int it = (threadIdx.x < 64) ? pair : (pair == 0 ? nth : g.nt - pair);
  const int l = ch * 64 + (threadIdx.x & 63);
  if constexpr (LAT && PASS != 1) {
    const int n7 = 2 * STEN * g.nr;
    double* const rows = reinterpret_cast<double*>(lat_tab + (LAP ? 2 : 1) * g.nr);
    for (int e = threadIdx.x; e < (LAP ? 2 : 1) * g.nr; e += 128) lat_tab[e] = A.rr[e];
    for (int e = threadIdx.x; e < n7; e += 128) {
      rows[e] = A.Dc[e];
      if constexpr (LAP) rows[n7 + e] = A.Luc[e];
    }
    __syncthreads();
  }
  if (l >= g.nz) return;
  const int k = it * g.nz + l;
  const ModeQ q = modeq(g, k);
  // sweep-side bases of this lane: factors u+ at this mode; u- = u+ at -m,
  // the other wave's lane (the Nyquist row has its own u- set, row 0 is its
  // own mirror); uz, p and the pressure homogeneous solution at |m|, the
  // wave-0 lane of the workgroup (Nyquist row: its own region)
  const int nr = g.nr;
  const int lane = threadIdx.x & 63;
  const bool nyq = pair == 0 && threadIdx.x >= 64;
  const size_t fb_up = (size_t)lb * nr * FR_UP + threadIdx.x;
  const size_t fb_um = nyq ? f_u1(g) + (size_t)ch * nr * FR_UP + threadIdx.x
                           : (pair == 0 ? fb_up : (size_t)lb * nr * FR_UP + (threadIdx.x ^ 64));
  const size_t ab = nyq ? sw_nblk(g) + ch : (size_t)lb;
  const size_t fb_uz = f_abs(g) + ab * nr * FR_ABS + lane;
  const size_t fb_p = fb_uz + f_absn(g);
  // the mixed form reads the u+, u-, uz factors as FP32 for |m| >= m32 (the
  // velocity Helmholtz operators, diagonally dominant through 1/dt); one |m|
  // per wave: rows pair and NT - pair, or the Nyquist row
  const bool f32w = __builtin_amdgcn_readfirstlane(A.F32 != nullptr && (nyq ? nth : pair) >= A.m32 ? 1 : 0) != 0;
  const size_t phb = ab * nr * 128 + lane;              // PH row i: phb + 128 i (+64: p_h)
  const size_t sb3 = (size_t)lb * nr * 384 + threadIdx.x;  // SR, E row i, component c: sb3 + 384 i + 128 c
  const size_t sb1 = (size_t)lb * nr * 128 + threadIdx.x;  // SP row i: sb1 + 128 i
  // N(u) is tile-major (dr_col): this mode's value of level j at nb0 + j npl,
  // components ncs apart; a wave's 64 modes are one tile row
  const size_t nb0 = (size_t)it * 64 + dr_col(g, l), npl = dr_plane(g), ncs = dr_cs(g);
  const size_t n = g.n;
  const int MS = g.modes;
  const double d_im = g.d_im;
  // Radial tables are read through the scalar cache: the parity of |m| is
  // the same for every lane of a wave (rows pair and NT - pair, or 0 and
  // NT/2), and the row index of a pass is uniform.
  const int par_u = __builtin_amdgcn_readfirstlane(abs((abs(q.m) % 2) - 1));  // parity table of ur, ut (u+, u-)
  const int par_p = 1 - par_u;                                                 // parity table of uz, p
  using TB = Tab<LAT>;
  TB Dt, Lt;
  if constexpr (LAT) {
    Dt.l = reinterpret_cast<const double*>(lat_tab + (LAP ? 2 : 1) * nr);
    Lt.l = Dt.l + 2 * STEN * nr;
  } else {
    Dt.g = ctab(A.Dc);
    Lt.g = ctab(A.Luc);
  }
  // x / r and x / r^2 at row i: the LAT kernels multiply by the tabled
  // reciprocals (an IEEE division is a chain of a dozen dependent instructions)
  auto over_r = [&](double x, int i) -> double {
    if constexpr (LAT) return times_recip(x, lat_tab[i]);
    else return x / ctab(A.r)[i];
  };
  auto over_r2 = [&](double x, int i) -> double {
    if constexpr (LAT) {
      return times_recip(x, lat_tab[nr + i]);
    } else {
      const double r2 = ctab(A.r)[i] * ctab(A.r)[i];
      return x / r2;
    }
  };
  const TB Dcu = Dt + par_u * STEN * nr;
  const TB Dcp = Dt + par_p * STEN * nr;
  const double2 z2 = make_double2(0.0, 0.0);
  // Column scratch precision of this workgroup: the mixed form holds SR, SP
  // and E of |m| >= m32 as FP32 pairs (the rhs, eliminated rows and pressure
  // of the fluctuation modes; the mean flow and low |m| stay FP64).  Both
  // waves have the same |m| (pair 0, rows 0 and NT/2, stays FP64).
  const bool s32b = A.s32 != 0 && pair >= A.m32;
  // The factor precision of this wave (F32W) and the storage of N(u) (N32,
  // FP32 in the mixed form) are compile-time branches too: run-time tests
  // inside the walks made the compiler drain outstanding loads before the
  // loads of each branch (two or three memory round trips per row).
  auto body = [&](auto s32_tag, auto f32_tag, auto n32_tag) {
  constexpr bool S32 = decltype(s32_tag)::value;
  constexpr bool F32W = decltype(f32_tag)::value;
  constexpr bool N32 = decltype(n32_tag)::value;
  // STR (kSweepStream): column scratch, the solution written and the previous
  // iterate go past the caches' usual replacement.  96 x 384 x 1537, FP32 N(u),
  // scratch and factors, us: A (corrector) 1137 -> 1106, B 446 -> 398, C 1039 ->
  // 941, D 1440/2030 -> 1422/1984.  Not the predictor's pass A (1704 -> 1820),
  // and not the factors, which the two waves of a workgroup share (all passes
  // 5-7% longer).
  constexpr bool NT = STR && !(PASS == 0 && PRED);
  using ScrT = Scr<S32, NT>;
  const ScrT SR = ScrT::at(A.SR, (size_t)lb * nr * 384);
  const ScrT SP = ScrT::at(A.SP, (size_t)lb * nr * 128);
  const ScrT E = ScrT::at(A.E, (size_t)lb * nr * 384);
  using SV = typename ScrT::V;
  using NV = std::conditional_t<N32, float2, double2>;
  using FT = std::conditional_t<F32W, float, double>;
  const NV* const Nv = reinterpret_cast<const NV*>(A.N);
  auto row_of = [&](int t) { return t < 0 ? 0 : (t < nr ? t : nr - 1); };

  // ============================== pass A1 (up, INC predictor): E', Dh
  if constexpr (PASS == 4) {
    const ScrT DH = ScrT::at(A.DH, (size_t)lb * nr * 128);
    double2 uw[3][7];      // u^n +/- rows t-6..t
    double2 Hr[7];         // (H u^n)_r rows i-3..i+3
    double2 Ht[4], Hz[4];  // (H u^n)_t, (H u^n)_z rows i..i+3
#pragma unroll
    for (int w = 0; w < 7; w++) {
      Hr[w] = z2;
#pragma unroll
      for (int c = 0; c < 3; c++) uw[c][w] = z2;
    }
#pragma unroll
    for (int w = 0; w < 4; w++) Ht[w] = Hz[w] = z2;
    const double ire = 1.0 / g.re, aim = d_im / g.re, idt = 1.0 / g.dt;
    struct Row1 {
      double2 u[3];  // u^n row t
      NV n[3];       // N(u^n) row t - 3
    };
    auto load1 = [&](int t, Row1& R) {
      const size_t h = (size_t)row_of(t) * MS + k, hn = nb0 + (size_t)row_of(t - 3) * npl;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        R.u[c] = A.u[c * n + h];
        R.n[c] = Nv[c * ncs + hn];
      }
    };
    auto work1 = [&](int t, const Row1& R) {
      double2 a = z2, b = z2, c = z2;
      if (t < nr) {  // zero past the wall
        a = R.u[0];
        b = R.u[1];
        c = R.u[2];
        pm_of(a, b);
      }
#pragma unroll
      for (int w = 0; w < 6; w++) {
        uw[0][w] = uw[0][w + 1];
        uw[1][w] = uw[1][w + 1];
        uw[2][w] = uw[2][w + 1];
      }
      uw[0][6] = a;
      uw[1][6] = b;
      uw[2][6] = c;
      const int j = t - 3;  // row whose 7-point window is complete
      double2 H0 = z2, H1 = z2, H2 = z2;
      if (j >= 0 && j < nr) {
        double2 nn[3] = {wide(R.n[0]), wide(R.n[1]), wide(R.n[2])};
        pm_of(nn[0], nn[1]);
        double2 hu[3];
#pragma unroll
        for (int cc = 0; cc < 3; cc++) {  // L'u^n as in addLap_k (mod_linear.cu:12-51)
          const TB Lc = Lt + (((cc < 2) ? par_u : par_p) * STEN * nr + STEN * j);
          double px = 0.0, py = 0.0;
#pragma unroll
          for (int w = 0; w < 7; w++) {
            px += Lc[w] * uw[cc][w].x;
            py += Lc[w] * uw[cc][w].y;
          }
          const double2 aux = uw[cc][3];
          double de = -q.kz * q.kz - over_r2(q.kt * q.kt, j);
          if (cc == 0) de += -over_r2(1.0, j) - over_r2(2.0 * q.kt, j);
          else if (cc == 1) de += -over_r2(1.0, j) + over_r2(2.0 * q.kt, j);
          px += de * aux.x;
          py += de * aux.y;
          E.st(sb3 + (size_t)j * 384 + cc * 128,
               make_double2(ire * px + (1.0 - d_im) * nn[cc].x, ire * py + (1.0 - d_im) * nn[cc].y));
          hu[cc] = make_double2(idt * aux.x - aim * px, idt * aux.y - aim * py);
        }
        rt_of(hu[0], hu[1]);
        H0 = hu[0];
        H1 = hu[1];
        H2 = hu[2];
      }
#pragma unroll
      for (int w = 0; w < 6; w++) Hr[w] = Hr[w + 1];
      Hr[6] = H0;
#pragma unroll
      for (int w = 0; w < 3; w++) {
        Ht[w] = Ht[w + 1];
        Hz[w] = Hz[w + 1];
      }
      Ht[3] = H1;
      Hz[3] = H2;
      const int i = j - 3;
      if (i >= 0 && i < nr) {  // div_k (mod_radialFD.cu:67-96) of H u^n, wall row zero
        double2 dv = z2;
        if (i < nr - 1) {
          const TB Dr = Dcu + STEN * i;
          double px = 0.0, py = 0.0;
#pragma unroll
          for (int w = 0; w < 7; w++) {
            px += Dr[w] * Hr[w].x;
            py += Dr[w] * Hr[w].y;
          }
          const double2 ur = Hr[3], ut = Ht[0], uz = Hz[0];
          px += over_r(ur.x, i);
          py += over_r(ur.y, i);
          px += over_r(-q.kt * ut.y, i);
          py += over_r(q.kt * ut.x, i);
          px += -q.kz * uz.y;
          py += q.kz * uz.x;
          dv = make_double2(px, py);
        }
        DH.st(sb1 + (size_t)i * 128, dv);
      }
    };
    walk_rows<LAT ? kLatRing : 0, 1, Row1>(0, nr + 6, load1, work1);
  }

  // ============================== pass A (up)
  if constexpr (PASS == 0) {
    constexpr bool XPRED = PRED && !INC;  // INC: the predictor's explicit part comes from A1
    constexpr int LAG = XPRED ? 6 : 3;
    const ScrT DH = ScrT::at(INC ? A.DH : A.SP, (size_t)lb * nr * 128);
    double2 uw[3][7];     // predictor: u^n +/- rows t-6..t
    double2 Rr[7];        // R_r rows i-3..i+3
    double2 Rt[4], Rz[4]; // R_t, R_z rows i..i+3
    double2 yp[3];        // pressure elimination rows i-3..i-1
#pragma unroll
    for (int w = 0; w < 7; w++) {
      Rr[w] = z2;
#pragma unroll
      for (int c = 0; c < 3; c++) uw[c][w] = z2;
    }
#pragma unroll
    for (int w = 0; w < 4; w++) Rt[w] = Rz[w] = z2;
#pragma unroll
    for (int w = 0; w < 3; w++) yp[w] = z2;
    const double cn = (1.0 - d_im) / g.re, idt = 1.0 / g.dt;
    // A row's loads are issued together before its stores, which the compiler
    // would not move loads across (one memory round trip per row)
    struct RowA {
      double2 u[3];  // predictor: u^n row t
      NV n[3];       // N(u) row j
      SV e[3];       // E row j
      double fl[3];  // pressure L factors of row i = j - 3
      SV dh;         // INC: Dh row i
    };
    auto loada = [&](int t, RowA& R) {
      const int j = XPRED ? t - 3 : t;
      const size_t hn = nb0 + (size_t)row_of(j) * npl;  // tile-major N(u)
      if constexpr (XPRED) {
        const size_t h = (size_t)row_of(t) * MS + k;
#pragma unroll
        for (int c = 0; c < 3; c++) R.u[c] = A.u[c * n + h];
      } else {
        const size_t he = sb3 + (size_t)row_of(j) * 384;
#pragma unroll
        for (int c = 0; c < 3; c++) R.e[c] = E.raw(he + c * 128);
      }
      const double* fpi = A.F + fb_p + (size_t)row_of(j - 3) * FR_ABS;
#pragma unroll
      for (int w = 0; w < 3; w++) R.fl[w] = fpi[w * 64];
      if constexpr (INC) R.dh = DH.raw(sb1 + (size_t)row_of(j - 3) * 128);
#pragma unroll
      for (int c = 0; c < 3; c++) R.n[c] = Nv[c * ncs + hn];
    };
    auto worka = [&](int t, const RowA& R) {
      if (XPRED) {
        double2 a = z2, b = z2, c = z2;
        if (t < nr) {  // zero past the wall
          a = R.u[0];
          b = R.u[1];
          c = R.u[2];
          pm_of(a, b);
        }
#pragma unroll
        for (int w = 0; w < 6; w++) {
          uw[0][w] = uw[0][w + 1];
          uw[1][w] = uw[1][w + 1];
          uw[2][w] = uw[2][w + 1];
        }
        uw[0][6] = a;
        uw[1][6] = b;
        uw[2][6] = c;
      }
      // rhs row j
      const int j = XPRED ? t - 3 : t;
      const int i = j - 3;  // pressure elimination row
      double2 R0 = z2, R1 = z2, R2 = z2;
      if (j >= 0 && j < nr) {
        double2 n0 = wide(R.n[0]), n1 = wide(R.n[1]);
        const double2 n2 = wide(R.n[2]);
        pm_of(n0, n1);
        double2 rh[3];
        if (XPRED) {
          // addLap_k (mod_linear.cu:12-51) on u^n, then rhs = N + that
          const double2 nn[3] = {n0, n1, n2};
#pragma unroll
          for (int c = 0; c < 3; c++) {
            const TB Lc = Lt + (((c < 2) ? par_u : par_p) * STEN * nr + STEN * j);
            double px = 0.0, py = 0.0;
#pragma unroll
            for (int w = 0; w < 7; w++) {
              px += Lc[w] * uw[c][w].x;
              py += Lc[w] * uw[c][w].y;
            }
            const double2 aux = uw[c][3];
            double de = -q.kz * q.kz - over_r2(q.kt * q.kt, j);
            if (c == 0) de += -over_r2(1.0, j) - over_r2(2.0 * q.kt, j);
            else if (c == 1) de += -over_r2(1.0, j) + over_r2(2.0 * q.kt, j);
            px += de * aux.x;
            py += de * aux.y;
            px *= cn;
            py *= cn;
            px += idt * aux.x;
            py += idt * aux.y;
            rh[c] = make_double2(nn[c].x + px, nn[c].y + py);
            E.st(sb3 + (size_t)j * 384 + c * 128,
                 make_double2(px + (1.0 - d_im) * nn[c].x, py + (1.0 - d_im) * nn[c].y));
          }
        } else {
          const double2 e0 = wide(R.e[0]), e1 = wide(R.e[1]), e2 = wide(R.e[2]);
          rh[0] = make_double2(e0.x + d_im * n0.x, e0.y + d_im * n0.y);
          rh[1] = make_double2(e1.x + d_im * n1.x, e1.y + d_im * n1.y);
          rh[2] = make_double2(e2.x + d_im * n2.x, e2.y + d_im * n2.y);
        }
        rt_of(rh[0], rh[1]);
        R0 = rh[0];
        R1 = rh[1];
        R2 = rh[2];
        const size_t hs = sb3 + (size_t)j * 384;
        SR.st(hs, R0);
        SR.st(hs + 128, R1);
        SR.st(hs + 256, R2);
      }
#pragma unroll
      for (int w = 0; w < 6; w++) Rr[w] = Rr[w + 1];
      Rr[6] = R0;
#pragma unroll
      for (int w = 0; w < 3; w++) {
        Rt[w] = Rt[w + 1];
        Rz[w] = Rz[w + 1];
      }
      Rt[3] = R1;
      Rz[3] = R2;
      // divergence and pressure elimination at row i = j - 3
      if (i >= 0 && i < nr) {
        double2 dv = z2;
        if (i < nr - 1) {  // div_k (mod_radialFD.cu:67-96), wall row zero
          const TB Dr = Dcu + STEN * i;
          double px = 0.0, py = 0.0;
#pragma unroll
          for (int w = 0; w < 7; w++) {
            px += Dr[w] * Rr[w].x;
            py += Dr[w] * Rr[w].y;
          }
          const double2 ur = Rr[3], ut = Rt[0], uz = Rz[0];
          px += over_r(ur.x, i);
          py += over_r(ur.y, i);
          px += over_r(-q.kt * ut.y, i);
          py += over_r(q.kt * ut.x, i);
          px += -q.kz * uz.y;
          py += q.kz * uz.x;
          dv = make_double2(px, py);
          if constexpr (INC) {  // div(rhs) = div(rhs - H u^n) + div(H u^n)
            const double2 dhi = wide(R.dh);
            dv.x += dhi.x;
            dv.y += dhi.y;
          }
        }
        const double l0 = R.fl[0], l1 = R.fl[1], l2 = R.fl[2];
        dv.x -= l0 * yp[0].x;
        dv.y -= l0 * yp[0].y;
        dv.x -= l1 * yp[1].x;
        dv.y -= l1 * yp[1].y;
        dv.x -= l2 * yp[2].x;
        dv.y -= l2 * yp[2].y;
        SP.st(sb1 + (size_t)i * 128, dv);
        yp[0] = yp[1];
        yp[1] = yp[2];
        yp[2] = dv;
      }
    };
    walk_rows<LAT ? kLatRing : 0, 1, RowA>(0, nr + LAG, loada, worka);
  }

  // ============================== pass B (down)
  if constexpr (PASS == 1) {
    double2 pw[3];  // p rows t+1..t+3
#pragma unroll
    for (int w = 0; w < 3; w++) pw[w] = z2;
    struct RowB {
      double f[4];  // 1/U_ii, U1..U3
      SV x;
    };
    auto loadb = [&](int t, RowB& R) {
      const double* fp = A.F + fb_p + (size_t)row_of(t) * FR_ABS;
#pragma unroll
      for (int w = 0; w < 4; w++) R.f[w] = fp[(3 + w) * 64];
      R.x = SP.raw(sb1 + (size_t)row_of(t) * 128);
    };
    auto workb = [&](int t, const RowB& R) {
      const double ru = R.f[0], u1 = R.f[1], u2 = R.f[2], u3 = R.f[3];
      double2 x = wide(R.x);
      x.x -= u1 * pw[0].x;
      x.y -= u1 * pw[0].y;
      x.x -= u2 * pw[1].x;
      x.y -= u2 * pw[1].y;
      x.x -= u3 * pw[2].x;
      x.y -= u3 * pw[2].y;
      const double2 pn = make_double2(x.x * ru, x.y * ru);
      SP.st(sb1 + (size_t)t * 128, pn);
      pw[2] = pw[1];
      pw[1] = pw[0];
      pw[0] = pn;
    };
    walk_rows<LAT ? 8 : 0, -1, RowB>(nr - 1, -1, loadb, workb);
  }

  // ============================== pass C (up)
  if constexpr (PASS == 2) {
    double2 pw[7];      // p rows j-3..j+3
    double2 yw[3][3];   // eliminated rows j-3..j-1 of u+, u-, uz
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int w = 0; w < 3; w++) yw[c][w] = z2;
#pragma unroll
    for (int w = 0; w < 7; w++) pw[w] = z2;
    // the L factors of the three solves at row j and its rhs are loaded before
    // the row's stores (the compiler does not move loads across them)
    struct RowC {
      SV p;             // p row t
      FT lc[3][IW];     // L factors row j = t - 3
      SV r[3];          // rhs row j
    };
    auto loadc = [&](int t, RowC& R) {
      R.p = SP.raw(sb1 + (size_t)row_of(t) * 128);
      const int j = row_of(t - IW);
#pragma unroll
      for (int c = 0; c < 3; c++) {
        // u+, u-: rows of FR_UP, slots of 128; uz: rows of FR_ABS, slots of 64
        const size_t fo = c == 0 ? fb_up + (size_t)j * FR_UP
                                 : (c == 1 ? fb_um + (size_t)j * FR_UP : fb_uz + (size_t)j * FR_ABS);
        const int fs = c == 2 ? 64 : 128;
#pragma unroll
        for (int w = 0; w < IW; w++) {
          if constexpr (F32W) R.lc[c][w] = A.F32[fo + w * fs];
          else R.lc[c][w] = A.F[fo + w * fs];
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++) R.r[c] = SR.raw(sb3 + (size_t)j * 384 + c * 128);
    };
    auto workc = [&](int t, const RowC& R) {
#pragma unroll
      for (int w = 0; w < 6; w++) pw[w] = pw[w + 1];
      pw[6] = (t < nr) ? wide(R.p) : z2;  // zero past the wall
      const int j = t - IW;
      if (j < 0) return;
      // addGrad_k (mod_radialFD.cu:115-143)
      const size_t h = sb3 + (size_t)j * 384;
      const TB Dr = Dcp + STEN * j;
      double px = 0.0, py = 0.0;
#pragma unroll
      for (int w = 0; w < 7; w++) {
        px += Dr[w] * pw[w].x;
        py += Dr[w] * pw[w].y;
      }
      const double2 ph = pw[3];
      double2 rh[3] = {wide(R.r[0]), wide(R.r[1]), wide(R.r[2])};
      rh[0].x -= px;
      rh[0].y -= py;
      rh[1].x -= over_r(-q.kt * ph.y, j);
      rh[1].y -= over_r(q.kt * ph.x, j);
      rh[2].x -= -q.kz * ph.y;
      rh[2].y -= q.kz * ph.x;
      pm_of(rh[0], rh[1]);
      if (j == nr - 1) {  // write_bcon_k: wall rows zero (INC: delta = -u^n there)
        rh[0] = rh[1] = rh[2] = z2;
        if constexpr (INC) {
          const size_t hw = (size_t)j * MS + k;
          double2 a = A.un[hw], b = A.un[n + hw];
          pm_of(a, b);
          const double2 c = A.un[2 * n + hw];
          rh[0] = make_double2(-a.x, -a.y);
          rh[1] = make_double2(-b.x, -b.y);
          rh[2] = make_double2(-c.x, -c.y);
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++) {  // forward elimination
        const double Lc[IW] = {R.lc[c][0], R.lc[c][1], R.lc[c][2]};
        double2 y = rh[c];
        y.x -= Lc[0] * yw[c][0].x;
        y.y -= Lc[0] * yw[c][0].y;
        y.x -= Lc[1] * yw[c][1].x;
        y.y -= Lc[1] * yw[c][1].y;
        y.x -= Lc[2] * yw[c][2].x;
        y.y -= Lc[2] * yw[c][2].y;
        SR.st(h + c * 128, y);
        yw[c][0] = yw[c][1];
        yw[c][1] = yw[c][2];
        yw[c][2] = y;
      }
    };
    walk_rows<LAT ? kLatRing : 0, 1, RowC>(0, nr + IW, loadc, workc);
  }

  // ============================== pass D (down)
  if constexpr (PASS == 3) {
    double2 xw[3][3];   // x rows i+1..i+3
    double xh[3][3];    // homogeneous wall-unit solutions rows i+1..i+3
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int w = 0; w < 3; w++) {
        xw[c][w] = z2;
        xh[c][w] = 0.0;
      }
    auto load_d = [&](const double2* p) {
      if constexpr (NT) return load_nt(p);
      else return *p;
    };
    auto backsub = [&](int i, double2* xo, double* ho) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const size_t fo = c == 0 ? fb_up + (size_t)i * FR_UP
                                 : (c == 1 ? fb_um + (size_t)i * FR_UP : fb_uz + (size_t)i * FR_ABS);
        const int fs = c == 2 ? 64 : 128;
        double ru, u1, u2, u3;
        // FP32 factors by the body's compile-time flag (a run-time test
        // here made the scheduler serialise the FP32 loads of the mixed
        // form); the HOLD kernels (FP64 form) keep the run-time test, with
        // which they were measured 3-7% faster
        if (HOLD ? f32w : F32W) {
          ru = A.F32[fo + 3 * fs];
          u1 = A.F32[fo + 4 * fs];
          u2 = A.F32[fo + 5 * fs];
          u3 = A.F32[fo + 6 * fs];
        } else {
          ru = A.F[fo + 3 * fs];
          u1 = A.F[fo + 4 * fs];
          u2 = A.F[fo + 5 * fs];
          u3 = A.F[fo + 6 * fs];
        }
        double2 x = SR.ld(sb3 + (size_t)i * 384 + c * 128);
        x.x -= u1 * xw[c][0].x;
        x.y -= u1 * xw[c][0].y;
        x.x -= u2 * xw[c][1].x;
        x.y -= u2 * xw[c][1].y;
        x.x -= u3 * xw[c][2].x;
        x.y -= u3 * xw[c][2].y;
        x = make_double2(x.x * ru, x.y * ru);
        double hh = (i == nr - 1) ? 1.0 : 0.0;
        hh -= u1 * xh[c][0];
        hh -= u2 * xh[c][1];
        hh -= u3 * xh[c][2];
        hh *= ru;
        xw[c][2] = xw[c][1];
        xw[c][1] = xw[c][0];
        xw[c][0] = x;
        xh[c][2] = xh[c][1];
        xh[c][1] = xh[c][0];
        xh[c][0] = hh;
        xo[c] = x;
        ho[c] = hh;
      }
      if constexpr (INC) {  // the solution is u^n + delta (FP64)
        const size_t hu = (size_t)i * MS + k;
        double2 a = A.un[hu], b = A.un[n + hu];
        pm_of(a, b);
        const double2 c = A.un[2 * n + hu];
        xo[0] = make_double2(xo[0].x + a.x, xo[0].y + a.y);
        xo[1] = make_double2(xo[1].x + b.x, xo[1].y + b.y);
        xo[2] = make_double2(xo[2].x + c.x, xo[2].y + c.y);
      }
    };
    struct RowD {
      FT f[3][4];      // ru, u1, u2, u3 of the u+, u-, uz solves
      double2 x[3];    // eliminated column rows
      double pd[2];    // dr p_h, p_h
      double2 uc[3];   // corrector: previous iterate
      double2 un[3];   // INC: u^n (+/- form for the velocity pair)
    };
    auto loadrow = [&](int i, RowD& R) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const size_t fo = c == 0 ? fb_up + (size_t)i * FR_UP
                                 : (c == 1 ? fb_um + (size_t)i * FR_UP : fb_uz + (size_t)i * FR_ABS);
        const int fs = c == 2 ? 64 : 128;
#pragma unroll
        for (int w = 0; w < 4; w++) {
          if constexpr (F32W) R.f[c][w] = A.F32[fo + (3 + w) * fs];
          else R.f[c][w] = A.F[fo + (3 + w) * fs];
        }
        R.x[c] = SR.ld(sb3 + (size_t)i * 384 + c * 128);
      }
      R.pd[0] = A.PH[phb + (size_t)i * 128];
      R.pd[1] = A.PH[phb + (size_t)i * 128 + 64];
      const size_t h = (size_t)i * MS + k;
      if constexpr (!PRED) {
#pragma unroll
        for (int c = 0; c < 3; c++) R.uc[c] = load_d(A.u + c * n + h);
      }
      if constexpr (INC) {
#pragma unroll
        for (int c = 0; c < 3; c++) R.un[c] = A.un[c * n + h];
      }
    };
    // A row's last products x / U_ii.  LAT kernels: rounded, or fused with the
    // sums that follow, as in the general kernels, so that all kinds give the
    // same bits.  In the FP64 form (HOLD) the products of u+ and u-, and of the
    // wall rows held (round_uz), are rounded: a run-time test of backsub, or the
    // rows between, part them from their sums.  In the others all are fused, in
    // the wall rows too, whose products are therefore formed anew (emit_wall).
    auto product = [&](const RowD& R, int c, double2 x, bool round_uz) -> double2 {
      x = make_double2(x.x * R.f[c][0], x.y * R.f[c][0]);
      if constexpr (LAT && !N32) {
        if (c < 2 || round_uz) {
          fix(x.x);
          fix(x.y);
        }
      }
      return x;
    };
    auto add_un = [&](const RowD& R, double2* xo) {
      if constexpr (INC) {  // the solution is u^n + delta (FP64)
        double2 a = R.un[0], b = R.un[1];
        pm_of(a, b);
        const double2 c = R.un[2];
        xo[0] = make_double2(xo[0].x + a.x, xo[0].y + a.y);
        xo[1] = make_double2(xo[1].x + b.x, xo[1].y + b.y);
        xo[2] = make_double2(xo[2].x + c.x, xo[2].y + c.y);
      }
    };
    auto wall_rounds_uz = [&](int s) { return s < 3 || !PRED; };
    // s >= 0: wall row nr - 1 - s, whose eliminated row before the product is kept in xe
    auto solve = [&](int i, const RowD& R, double2* xo, double* ho, int s = -1, double2* xe = nullptr) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const double ru = R.f[c][0], u1 = R.f[c][1], u2 = R.f[c][2], u3 = R.f[c][3];
        double2 x = R.x[c];
        x.x -= u1 * xw[c][0].x;
        x.y -= u1 * xw[c][0].y;
        x.x -= u2 * xw[c][1].x;
        x.y -= u2 * xw[c][1].y;
        x.x -= u3 * xw[c][2].x;
        x.y -= u3 * xw[c][2].y;
        if (s >= 0) xe[c] = x;
        x = product(R, c, x, s >= 0 && wall_rounds_uz(s));
        double hh = (i == nr - 1) ? 1.0 : 0.0;
        hh -= u1 * xh[c][0];
        hh -= u2 * xh[c][1];
        hh -= u3 * xh[c][2];
        hh *= ru;
        xw[c][2] = xw[c][1];
        xw[c][1] = xw[c][0];
        xw[c][0] = x;
        xh[c][2] = xh[c][1];
        xh[c][1] = xh[c][0];
        xh[c][0] = hh;
        xo[c] = x;
        ho[c] = hh;
      }
      add_un(R, xo);
    };
    // wall divergence of the provisional solution (divWall_k on r/theta
    // form) from the four wall rows. Without HOLD the walk that emits the
    // solution repeats their back substitution (same arithmetic, same
    // values), which keeps the pass at 3 waves per SIMD instead of 2.
    double2 urw[4], utw = z2, uzw = z2;
    double2 xs[HOLD || LAT ? 4 : 1][3];  // HOLD, LAT: wall rows NR-1..NR-4 (LAT: before the product)
    double xhs[HOLD || LAT ? 4 : 1][3];
    RowD ring[LAT ? 4 : 1];
    if constexpr (LAT) {
#pragma unroll
      for (int s = 0; s < 4; s++) loadrow(nr - 1 - s, ring[s]);
    }
#pragma unroll
    for (int s = 0; s < 4; s++) {
      double2 xo[3];
      double ho[3];
      if constexpr (LAT) solve(nr - 1 - s, ring[s], xo, ho, s, xs[s]);
      else backsub(nr - 1 - s, xo, ho);
      if constexpr (HOLD || LAT) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          if constexpr (!LAT) xs[s][c] = xo[c];
          xhs[s][c] = ho[c];
        }
      }
      double2 a = xo[0], b = xo[1];
      rt_of(a, b);
      urw[s] = a;
      if (s == 0) {
        utw = b;
        uzw = xo[2];
      }
    }
    if constexpr (!HOLD && !LAT) {
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int w = 0; w < 3; w++) {
          xw[c][w] = z2;
          xh[c][w] = 0.0;
        }
    }
    double2 dv;
    {
      const TB Dr = Dcu + STEN * (nr - 1);
      double px = 0.0, py = 0.0;
#pragma unroll
      for (int w = 0; w < 4; w++) {  // columns NR-4..NR-1 = urw[3..0]
        px += Dr[w] * urw[3 - w].x;
        py += Dr[w] * urw[3 - w].y;
      }
      px += urw[0].x;
      py += urw[0].y;
      px += -q.kt * utw.y;
      py += q.kt * utw.x;
      px += -q.kz * uzw.y;
      py += q.kz * uzw.x;
      dv = make_double2(px, py);
    }
    double2 cf[4];  // compcoef_k
    {
      const double2 nd = make_double2(-dv.x, -dv.y);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const double2 im = A.invc[(size_t)k * 4 + j];
        cf[j] = make_double2(nd.x * im.x - nd.y * im.y, nd.x * im.y + nd.y * im.x);
      }
    }
    double num = 0.0, den = 0.0;
    // emit row i: pd = {dr p_h, p_h} and uc (the corrector's previous
    // iterate) come from a prefetched row, or are loaded here when null
    auto emit = [&](int i, const double2* xo, const double* ho, const double* pd = nullptr,
                    const double2* uc = nullptr) {
      const size_t h = (size_t)i * MS + k;
      // pressure-gradient homogeneous solution: (dr p_h -+ kt p_h / r, 0), (0, kz p_h)
      const double dph = pd ? pd[0] : A.PH[phb + (size_t)i * 128];
      const double ph = pd ? pd[1] : A.PH[phb + (size_t)i * 128 + 64];
      const double tq = over_r(q.kt * ph, i);
      const double2 hp[3] = {make_double2(dph - tq, 0.0), make_double2(dph + tq, 0.0), make_double2(-0.0, q.kz * ph)};
      const double2 hv[3] = {make_double2(ho[0], 0.0), make_double2(ho[1], 0.0), make_double2(0.0, ho[2])};
      double2 o[3] = {xo[0], xo[1], xo[2]};
      rt_of(o[0], o[1]);  // decoupleBackward / decoupleForward round trip of corBCon
      pm_of(o[0], o[1]);
#pragma unroll
      for (int c = 0; c < 3; c++) {  // addBCon_k
        const double ax = cf[c].x * hv[c].x - cf[c].y * hv[c].y + cf[3].x * hp[c].x - cf[3].y * hp[c].y;
        const double ay = cf[c].x * hv[c].y + cf[c].y * hv[c].x + cf[3].x * hp[c].y + cf[3].y * hp[c].x;
        o[c] = make_double2(o[c].x + ax, o[c].y + ay);
      }
      rt_of(o[0], o[1]);
      if (!PRED && k != 0) {  // mcor_k; mode (0,0) is measured after its fix-up
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const double2 u1 = uc ? uc[c] : load_d(A.u + c * n + h);
          const double dx = u1.x - o[c].x, dy = u1.y - o[c].y;
          // fused the same way in every kind of kernel
          const double a1 = N32 && c == 0 ? __builtin_fma(dy, dy, dx * dx) : __builtin_fma(dx, dx, dy * dy);
          const double a2 = __builtin_fma(u1.x, u1.x, u1.y * u1.y);
          num = (a1 > num || a1 != a1) ? a1 : num;
          den = (a2 > den || a2 != a2) ? a2 : den;
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++) {
        if constexpr (NT) store_nt(A.out + c * n + h, o[c]);
        else A.out[c * n + h] = o[c];
      }
    };
    if constexpr (LAT) {
      auto loadd = [&](int i, RowD& R) { loadrow(row_of(i), R); };
      auto emit_wall = [&](int s) {
        double2 xo[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          fix(xs[s][c].x);
          fix(xs[s][c].y);
          xo[c] = product(ring[s], c, xs[s][c], wall_rounds_uz(s));
        }
        add_un(ring[s], xo);
        emit(nr - 1 - s, xo, xhs[s], ring[s].pd, PRED ? nullptr : ring[s].uc);
      };
      RowD nxt[kLatRing];
#pragma unroll
      for (int s = 0; s < 4; s++) {
        if (s < kLatRing) loadd(nr - 5 - s, nxt[s < kLatRing ? s : 0]);
        emit_wall(s);
      }
      walk_ring<kLatRing, -1>(nxt, nr - 5, -1, loadd, [&](int i, const RowD& R) {
        double2 xo[3];
        double ho[3];
        solve(i, R, xo, ho);
        emit(i, xo, ho, R.pd, PRED ? nullptr : R.uc);
      });
    } else if constexpr (HOLD) {
#pragma unroll
      for (int s = 0; s < 4; s++) emit(nr - 1 - s, xs[s], xhs[s]);
      for (int i = nr - 5; i >= 0; i--) {
        double2 xo[3];
        double ho[3];
        backsub(i, xo, ho);
        emit(i, xo, ho);
      }
    } else {
      // The walk that emits the solution, software-pipelined: the loads of
      // row i - 1 (factors, column, p_h, previous iterate) are issued before
      // row i is solved and stored, so each row's memory latency overlaps
      // the previous row's arithmetic (the compiler does not move loads
      // across the stores of a row by itself).  Same arithmetic as backsub.
      RowD cur, nxt;
      loadrow(nr - 1, cur);
      for (int i = nr - 1; i >= 0; i--) {
        loadrow(i > 0 ? i - 1 : 0, nxt);
        double2 xo[3];
        double ho[3];
        solve(i, cur, xo, ho);
        emit(i, xo, ho, cur.pd, PRED ? nullptr : cur.uc);
        cur = nxt;
      }
    }
    if (k == 0) {  // modeZZ_k, adj_flux (mod_integrate.cu:63-68, mod_cublasflux.cu:90-103)
      double qa = 0.0;
      for (int i = 0; i < nr; i++) {
        const size_t h = (size_t)i * MS;
        A.out[h] = z2;
        A.out[n + h].y = 0.0;
        A.out[2 * n + h].y = 0.0;
        qa += A.rdr[i] * A.out[2 * n + h].x;
      }
      const double corr = (g.qdes - qa) / A.qc[0];
      for (int i = 0; i < nr; i++) {
        const size_t h = (size_t)i * MS;
        A.out[2 * n + h].x += corr * A.uc[i];
        if (!PRED) {
#pragma unroll
          for (int c = 0; c < 3; c++) {
            const double2 u1 = A.u[c * n + h], o = A.out[c * n + h];
            const double dx = u1.x - o.x, dy = u1.y - o.y;
            const double a1 = dx * dx + dy * dy, a2 = u1.x * u1.x + u1.y * u1.y;
            num = (a1 > num || a1 != a1) ? a1 : num;
            den = (a2 > den || a2 != a2) ? a2 : den;
          }
        }
      }
    }
    if (!PRED) {
      // num, den are >= 0 or NaN, whose bit patterns order as the values do
      // (NaN above every finite value and +inf). A full wave combines its
      // lanes' maxima and issues one atomic per value; a partly filled wave
      // (the last axial chunk) keeps one per lane.
      unsigned long long a = __double_as_longlong(num), b = __double_as_longlong(den);
      if (__builtin_amdgcn_read_exec() == ~0ull) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          const unsigned long long ao = __shfl_xor(a, o), bo = __shfl_xor(b, o);
          a = ao > a ? ao : a;
          b = bo > b ? bo : b;
        }
        if (lane == 0) {
          atomicMax(&A.norm[0], a);
          atomicMax(&A.norm[1], b);
        }
      } else {
        atomicMax(&A.norm[0], a);
        atomicMax(&A.norm[1], b);
      }
    }
  }
  };
  // the FP64 form has FP64 N(u), scratch and factors (s32b and f32w false)
  using T1 = std::true_type;
  using T0 = std::false_type;
  if (!A.n32) body(T0{}, T0{}, T0{});
  else if (s32b) {
    if (f32w) body(T1{}, T1{}, T1{});
    else body(T1{}, T0{}, T1{});
  } else {
    if (f32w) body(T0{}, T1{}, T1{});
    else body(T0{}, T0{}, T1{});
  }
}

size_t factor_count(const Geom& g) { return f_abs(g) + 2 * f_absn(g); }
size_t factor32_count(const Geom& g) { return f_abs(g) + f_absn(g); }

void launch_factor(const Geom& g, const double* r, const double* Lu, const double* Lp, double* F, float* F32,
                   hipStream_t s) {
  dim3 grid((g.modes + 255) / 256, 4);
  factor_kernel<<<grid, 256, 0, s>>>(g, r, Lu, Lp, F, F32);
}

// Small grids run the LAT kernels: at most kLatBlocks workgroups (two per CU)
// and radial tables that fit the default LDS limit.  Sweeps, general / LAT, us,
// predictor and corrector: at 448 workgroups as above; at 544 to 864 the one or
// the other is up to a tenth faster by form and row count (64x64x1025 FP64 601 /
// 633 and 647 / 654, mixed 496 / 574 and 554 / 535; 64x192x385 FP64 646 / 702 and
// 683 / 723, refined 655 / 623 and 615 / 580).
//
// A batch's small members go in launches of their own (in one launch with the
// larger ones the XCD order, made for the largest, would leave half the chip
// without work of theirs: 32 x 48x96x513 and 32 x 64x128x1025 mixed 142 -> 146 ms)
// and count their modes together, as the last chunks of axial modes are nearly
// empty where NZ is a little above a multiple of 64: LAT up to kLatModes, 400
// full workgroups.  Ensemble steps, general / LAT, ms: 12 x 32x64x65 (50k modes)
// FP64 1.44 / 1.45, mixed 1.10 / 1.07, 2 x 24x64x385 (49k) FP64 1.10 / 1.06, mixed
// 0.73 / 0.69; 2 x 64x64x513 (66k) 3.27 / 3.36 and 2.22 / 2.26, 2 x 48x96x513
// (98k) 3.35 / 3.46 and 2.16 / 2.24, 64 x 32x64x65 6.86 / 7.17 and 4.71 / 4.84, 64
// x 48x96x513 mixed 62.2 / 64.3.  A pipe may so run one kind alone and another
// in an ensemble: the arithmetic, and so every bit of the results, is the same.
//
// Streamed accesses where no array outlives a pass in the caches: states of
// more than 1 GiB, four times the 256 MB memory-side cache.  Steps of one pipe,
// general and streamed in turn, ms: 96 x 384 x 1537 (2.5 GiB) FP64 45.1 -> 44.5,
// mixed 25.9 -> 25.4; 48 x 384 x 1537 (1.3 GiB) 22.7 -> 22.4 and 13.0 -> 12.8; 40 x
// 384 x 1537 (1.06 GiB) mixed 10.9 -> 10.75; of 64 x 128 x 1025 (0.4 GB): FP64 3.85
// -> 3.81 ms but refined mixed 2.63 -> 2.74, as the kernels that follow find less
// of the new state in the caches.  The refined form and batched launches do
// not stream (not measured above the limit).
constexpr size_t kLatBlocks = 512;
constexpr int kLatRows = 256;
constexpr size_t kLatModes = 400 * 128;
bool sweep_kind_exists(const Geom& g, bool inc, int kind) {
  return kind == kSweepPlain || (kind == kSweepLat && g.nr <= kLatRows) || (kind == kSweepStream && !inc);
}
int sweep_small(const Geom& g) { return sw_nblk(g) <= kLatBlocks && g.nr <= kLatRows ? 1 : 0; }
int sweep_kind(const Geom& g, bool inc, int choice) {
  if (choice >= 0 && sweep_kind_exists(g, inc, choice)) return choice;
  if (sweep_small(g)) return kSweepLat;
  return !inc && 3 * g.n * sizeof(double2) > (size_t(1) << 30) ? kSweepStream : kSweepPlain;
}
void SweepExtent::add(const Geom& g, bool mixed_form) {
  max_nr = std::max(max_nr, g.nr);
  max_nt = std::max(max_nt, g.nt);
  max_nz = std::max(max_nz, g.nz);
  modes += g.modes;
  (mixed_form ? mixed : fp64) = true;
}
void SweepBatch::add(const Geom& g, bool mixed_form, int choice) {
  const int small = sweep_small(g);
  SweepExtent& x = part[small];
  x.add(g, mixed_form);
  const bool lat = choice >= 0 ? choice == kSweepLat : small && x.modes <= kLatModes;
  kind[small] = lat && x.max_nr <= kLatRows ? kSweepLat : kSweepPlain;
}
template <int PASS, int PRED, int INC>
static size_t lat_lds(int nr) {
  return PASS == 1 ? 0 : (size_t)nr * (2 + 2 * STEN) * (lat_lap<PASS, PRED, INC>() ? 2 : 1) * sizeof(double);
}

template <int PASS, int PRED, int LAT>
static void sweep_pass_inc(const Lin2Args& a, dim3 grid, hipStream_t s) {
  const size_t lds = LAT ? lat_lds<PASS, PRED, 1>(a.g.nr) : 0;
  sweep_kernel<PASS, PRED, 0, 0, 1, LAT><<<grid, 128, lds, s>>>(a, nullptr, 0);
}
template <int PRED, int LAT>
static void sweep_passes_inc(const Lin2Args& a, dim3 grid, hipStream_t s) {
  if constexpr (PRED) sweep_pass_inc<4, PRED, LAT>(a, grid, s);
  sweep_pass_inc<0, PRED, LAT>(a, grid, s);
  sweep_pass_inc<1, PRED, LAT>(a, grid, s);
  sweep_pass_inc<2, PRED, LAT>(a, grid, s);
  sweep_pass_inc<3, PRED, LAT>(a, grid, s);
}

// pass D runs as HOLD = 1 for the FP64-form pipes and as HOLD = 0 for the
// mixed-form ones (a batched launch of both forms makes both launches)
template <int PRED, int B, int STR = 0>
static void sweep_passes(const Lin2Args& a, const Lin2Args* tab, int small, dim3 grid, bool fp64, bool mixed,
                         hipStream_t s) {
  sweep_kernel<0, PRED, B, 0, 0, 0, PRED ? 0 : STR><<<grid, 128, 0, s>>>(a, tab, small);
  sweep_kernel<1, PRED, B, 0, 0, 0, STR><<<grid, 128, 0, s>>>(a, tab, small);
  sweep_kernel<2, PRED, B, 0, 0, 0, STR><<<grid, 128, 0, s>>>(a, tab, small);
  if (fp64) sweep_kernel<3, PRED, B, 1, 0, 0, STR><<<grid, 128, 0, s>>>(a, tab, small);
  if (mixed) sweep_kernel<3, PRED, B, 0, 0, 0, STR><<<grid, 128, 0, s>>>(a, tab, small);
}
template <int PRED, int B>
static void sweep_passes_lat(const Lin2Args& a, const Lin2Args* tab, int small, dim3 grid, int nr, hipStream_t s) {
  sweep_kernel<0, PRED, B, 0, 0, 1><<<grid, 128, lat_lds<0, PRED, 0>(nr), s>>>(a, tab, small);
  sweep_kernel<1, PRED, B, 0, 0, 1><<<grid, 128, lat_lds<1, PRED, 0>(nr), s>>>(a, tab, small);
  sweep_kernel<2, PRED, B, 0, 0, 1><<<grid, 128, lat_lds<2, PRED, 0>(nr), s>>>(a, tab, small);
  sweep_kernel<3, PRED, B, 0, 0, 1><<<grid, 128, lat_lds<3, PRED, 0>(nr), s>>>(a, tab, small);
}

void launch_sweep2(const Lin2Args& a, hipStream_t s) {
  const dim3 grid((a.g.nt / 2) * ((a.g.nz + 63) / 64));
  const bool lat = a.kind == kSweepLat;
  if (a.inc) {
    if (a.predictor) lat ? sweep_passes_inc<1, 1>(a, grid, s) : sweep_passes_inc<1, 0>(a, grid, s);
    else lat ? sweep_passes_inc<0, 1>(a, grid, s) : sweep_passes_inc<0, 0>(a, grid, s);
    return;
  }
  if (lat) {
    if (a.predictor) sweep_passes_lat<1, 0>(a, nullptr, 0, grid, a.g.nr, s);
    else sweep_passes_lat<0, 0>(a, nullptr, 0, grid, a.g.nr, s);
    return;
  }
  const bool fp64 = a.form64 != 0;
  if (a.kind == kSweepStream) {
    if (a.predictor) sweep_passes<1, 0, 1>(a, nullptr, 0, grid, fp64, !fp64, s);
    else sweep_passes<0, 0, 1>(a, nullptr, 0, grid, fp64, !fp64, s);
    return;
  }
  if (a.predictor) sweep_passes<1, 0>(a, nullptr, 0, grid, fp64, !fp64, s);
  else sweep_passes<0, 0>(a, nullptr, 0, grid, fp64, !fp64, s);
}

void launch_sweep_batch(const Lin2Args* tab, int count, int predictor, const SweepBatch& b, hipStream_t s) {
  Lin2Args dummy{};
  for (const int small : {1, 0}) {
    const SweepExtent& x = b.part[small];
    if (x.modes == 0) continue;
    const dim3 grid((x.max_nt / 2) * ((x.max_nz + 63) / 64), count);
    if (b.kind[small] == kSweepLat) {
      if (predictor) sweep_passes_lat<1, 1>(dummy, tab, small, grid, x.max_nr, s);
      else sweep_passes_lat<0, 1>(dummy, tab, small, grid, x.max_nr, s);
    } else {
      if (predictor) sweep_passes<1, 1>(dummy, tab, small, grid, x.fp64, x.mixed, s);
      else sweep_passes<0, 1>(dummy, tab, small, grid, x.fp64, x.mixed, s);
    }
  }
}

}  // namespace nsp
