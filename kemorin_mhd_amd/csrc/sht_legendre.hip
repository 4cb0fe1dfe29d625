// sht_legendre.hip -- FP64-MFMA Legendre transforms (gfx950).
//
// Per zonal order M = |m| the reference's symmetric_BLAS_big mode
// (SS/leg_b_trans_sym_matmul_big.f90:183-293, SS/leg_f_trans_sym_matmul_big.f90:
// 187-305) does four DGEMMs against hemisphere tables of P and dP/dtheta,
// split by the parity of l-m.  Here both slots +M and -M share the tables,
// so one wave handles both; the backward's pack (SS/set_sp_rlm_for_leg_matmul.f90:
// 281-398) is a pass of its own (k_leg_pack), the forward's
// (SS/set_vr_rtm_for_leg_matmul.f90:369-565) is done in registers, and the
// unpack (SS/cal_vr_rtm_by_matmul.f90:357-540, SS/cal_sp_rlm_by_matmul.f90:
// 365-545) is the accumulators' epilogue.  The 1/r, 1/r^2, m and 1/sin(theta)
// factors are applied in the epilogue rather than to the operands (same
// products, different rounding order).
//
// A wave reads both operands straight into MFMA fragments, one K step of 4
// ahead, and waits for no other wave: an FP64 MFMA holds the matrix unit for
// 64 cycles, so the 8 KB of a step (16 fragments for 20 products) are
// 6.4 bytes per cycle and SIMD, which L1 and L2 deliver; two waves per SIMD.
// Large forward calls share their rows through LDS (k_leg_fwd_lds).  The
// matrix units are busy 78 % of the time in the backward's low orders, which
// have many steps, half of it in its high ones (68 % of a call at L = 511) and
// 67 % in the forward; a loop of such products alone reaches 72.6 of their 78.6
// TF.  L = 511, Nr = 257: backward (8 components) 26.4 ms staged through LDS in
// its own layout, now 2.1 to pack and 12.5 to 13.2; forward (9) 36.0, now 17.1.
// L = 255, Nr = 129: forward (9) 3.14, now 1.45.
//
// MFMA: v_mfma_f64_16x16x4f64.  A(16x4): lane holds A[lane%16][lane/16];
// B(4x16): lane holds B[lane/16][lane%16]; D(16x16): lane holds
// D[4*r + lane/16][lane%16] in element r (measured on gfx950, checked by
// sht_selftest).
#include <vector>

#include "sht_internal.h"

namespace ksht {

__device__ __forceinline__ d4 mfma64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// g3 as packed by the reference: l(l+1), with 1/2 for l = m = 0
// (SP/schmidt_poly_on_rtm_grid.f90:109).
__device__ __forceinline__ double g3_of(int l) { return l == 0 ? 0.5 : (double)(l * (l + 1)); }
// g7, g6 of SH/spherical_harmonics.f90:118-137.
__device__ __forceinline__ double g7_of(int l, int M) {
  if (l == 0) return 1.0;
  return M == 0 ? (double)(2 * l + 1) / (double)(2 * l * (l + 1))
                : (double)(2 * l + 1) / (double)(4 * l * (l + 1));
}
__device__ __forceinline__ double g6_of(int l, int M) {
  if (l == 0 && M == 0) return 0.5;
  return M == 0 ? (double)(2 * l + 1) / 2.0 : (double)(2 * l + 1) / 4.0;
}

// A launch covers orders M0 .. M0+nM-1 (one tile of the P tables).  Columns
// are (vector, radius) pairs, flattened so that a few radii past a multiple
// of 16 are padded once per call instead of once per field, then (scalar,
// radius) pairs: ncv and ncs tiles of 16.
struct LegDims {
  int L, nr, nth, nth_h, nth_hp, nv, ns, ncomp;
  int M0, nM, ncv, ncs;
  int ntv, nts;    // backward: row tiles of 16 (vectors) and 32 (scalars)
  unsigned nbv;    // work-groups of the vectors; the scalars' follow
  int W;           // doubles per packed row
};
// sum over x = 1 .. n of ceil(x / u)
__host__ __device__ inline long long ceil_sum(int n, int u) {
  const long long q = n / u, r = n % u;
  return u * q * (q + 1) / 2 + r * (q + 1);
}

// wave-uniform index of the wave in its launch
__device__ __forceinline__ int wave_of_group() {
  return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
}

// Rows of the packed spectra of orders with n = L - M + 1 degrees: steps of 4
// pair indices i and both parities, 8 rows each.
__host__ __device__ inline long long pack_rows(int n) { return 8LL * ((n + 7) / 8); }
__host__ __device__ inline long long pack_rows_sum(int n) { return 8 * ceil_sum(n, 8); }

// element of a wave-uniform base plus a 32-bit lane offset in bytes
__device__ __forceinline__ double ldu(const double *base, unsigned off) {
  return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + off);
}

// ---------------------------------------------------------------------------
// Spectra of orders M0 .. M0+nM-1 in the row order of the backward's K steps:
// row (step, parity, i % 4), columns [slot +-M][pol g3 | dpol | tor | scalars],
// each the flattened (field, radius) columns; zero past the last degree.
// A work-group moves 16 radii of up to 256 contiguous doubles each through
// LDS: long runs on both sides.  L = 511, Nr = 257, 8 components: 2.3 ms for
// 4.3 GB read and 4.5 GB written.
constexpr int kPackRun = 256, kPackPitch = kPackRun + 4;

__global__ void __launch_bounds__(256) k_leg_pack(LegDims d, int dt, int nz,
                                                  const double *__restrict__ sp, long long s_k,
                                                  const int *__restrict__ jst,
                                                  double *__restrict__ Bp) {
  __shared__ double tile[16 * kPackPitch];
  // the radius tiles of a run on one XCD: their rows share 128-byte lines
  const unsigned nk = (d.nr + 15) / 16;
  unsigned id = (unsigned)xcd_group_order(blockIdx.x, gridDim.x, nk);
  const int k0 = (int)(id % nk) * 16;
  id /= nk;
  const int x0 = (int)(id % nz) * dt, sg = (int)(id / nz) & 1, M = d.M0 + (int)(id / nz / 2);
  const int n = d.L - M + 1;
  if (x0 >= pack_rows(n) || (M == 0 && sg)) return;
  const int tid = threadIdx.x;
  const int run = dt * d.ncomp;
  if (tid < run) {
    const int x = x0 + tid / d.ncomp, nd = tid % d.ncomp;
    const double *src = sp + (long long)(jst[sg ? d.L - M : d.L + M] + x0) * d.ncomp + tid;
    const double g = (nd < 3 * d.nv && nd % 3 == 0) ? g3_of(M + x) : 1.0;
    double r[16];
#pragma unroll
    for (int kk = 0; kk < 16; kk++)
      r[kk] = (x < n && k0 + kk < d.nr) ? src[(long long)(k0 + kk) * s_k] : 0.0;
#pragma unroll
    for (int kk = 0; kk < 16; kk++) tile[kk * kPackPitch + tid] = r[kk] * g;
  }
  __syncthreads();
  const int k = k0 + (tid & 15);
  if (k >= d.nr) return;
  const long long row0 = pack_rows_sum(d.L - d.M0 + 1) - pack_rows_sum(n);
  double *dst = Bp + row0 * d.W + (long long)sg * (d.W / 2) + k;
  for (int e = tid >> 4; e < run; e += 16) {
    const int x = x0 + e / d.ncomp, nd = e % d.ncomp;
    if (x >= pack_rows(n)) break;
    const int row = ((x >> 3) * 2 + (x & 1)) * 4 + ((x >> 1) & 3);
    const int col = nd < 3 * d.nv ? (nd % 3) * 16 * d.ncv + (nd / 3) * d.nr
                                  : 3 * 16 * d.ncv + (nd - 3 * d.nv) * d.nr;
    dst[(long long)row * d.W + col] = tile[(tid & 15) * kPackPitch + e];
  }
}

// Rows of a wave in the P tables of order M: uniform bases of both parities
// and the last step of the odd one, whose block may be shorter (its spectra
// past the end are zero) or, for one degree, missing.
struct PBase {
  const double *e, *o;
  int o_last;
};
__device__ __forceinline__ PBase p_base(const double *P, long long off0, long long off1, int ip1) {
  return PBase{P + off0, P + (ip1 ? off1 : off0), ip1 ? ip1 / 4 - 1 : 0};
}

// Spectra as the backward's B fragments: the packed rows, or (PACK false, for
// calls of few waves, where the packing launch costs more than the scattered
// loads) the caller's buffer itself.
template <bool PACK>
struct SpecRows {
  const double *b;       // PACK: the order's rows, else the spectra
  long long sig[2];      // offsets of the slots
  unsigned v;            // lane offset, bytes
  int W, nc, x2, n, M;   // row pitch; components; 2 (lane / 16); degrees; order
  __device__ __forceinline__ double get(int s, int par, int sg, int c, bool pol) const {
    if constexpr (PACK) {
      return ldu(b + (8LL * s + par * 4) * W + sig[sg] + c, v);
    } else {
      const int x = 8 * s + x2 + par, xc = x < n ? x : n - 1;
      const double z = ldu(b + sig[sg] + c, v + (unsigned)(xc * nc * 8));
      return x < n ? (pol ? z * g3_of(M + x) : z) : 0.0;
    }
  }
};
// col0: first column of the wave's tile among the vectors' (nf = 3) or the
// scalars' (nf = 1, whose columns start at c0) columns
template <bool PACK>
__device__ __forceinline__ SpecRows<PACK> spec_rows(const LegDims &d, const double *B, int M,
                                                    int lane, int f, int k, int col, int c0,
                                                    long long s_k, const int *jst) {
  SpecRows<PACK> r;
  const int n = d.L - M + 1;
  r.W = d.W;
  r.nc = d.ncomp;
  r.x2 = 2 * (lane >> 4);
  r.n = n;
  r.M = M;
  if constexpr (PACK) {
    r.b = B + (pack_rows_sum(d.L - d.M0 + 1) - pack_rows_sum(n)) * d.W + c0;
    r.sig[0] = 0;
    r.sig[1] = M ? d.W / 2 : 0;  // one slot for M = 0: read twice, stored once
    r.v = (unsigned)(((lane >> 4) * d.W + col) * 8);
  } else {
    r.b = B;
    r.sig[0] = (long long)jst[d.L + M] * d.ncomp;
    r.sig[1] = (long long)jst[d.L - M] * d.ncomp;
    r.v = (unsigned)((f + k * s_k) * 8);
  }
  return r;
}

// ---------------------------------------------------------------------------
// Backward, vectors: 16 hemisphere rows by 16 columns, (pol, dpol, tor), both
// slots and parities: 20 products (160 accumulator registers) per K step.
template <bool PACK>
__device__ __forceinline__ void leg_bwd_vec(
    const LegDims &d, long long id, const double *__restrict__ B, long long s_k,
    double *__restrict__ out, const GridAddr &ga, const int *__restrict__ jst,
    const long long *__restrict__ offb, const int *__restrict__ ipad,
    const double *__restrict__ Pb, const double *__restrict__ dPb,
    const double *__restrict__ a_r, const double *__restrict__ asin_t) {
  const int lane = threadIdx.x & 63;
  // id = (order ncv + column tile) ntv + row tile
  const int t0 = (int)(id % d.ntv) * 16;
  id /= d.ntv;
  const int ct = (int)(id % d.ncv), M = d.M0 + (int)(id / d.ncv);
  if (M >= d.M0 + d.nM) return;
  const int L = d.L, nstep = (L - M + 8) / 8;
  const int nsig = (M == 0) ? 1 : 2;
  const int col = ct * 16 + (lane & 15);
  const int colc = col < d.nv * d.nr ? col : d.nv * d.nr - 1;
  const int q = colc / d.nr, k = colc - q * d.nr;
  const SpecRows<PACK> x = spec_rows<PACK>(d, B, M, lane, 3 * q, k, col, 0, s_k, jst);
  const int cs = PACK ? 16 * d.ncv : 1;
  const unsigned vp = (unsigned)(((lane >> 4) * d.nth_hp + t0 + (lane & 15)) * 8);
  const PBase p = p_base(Pb, offb[2 * M], offb[2 * M + 1], ipad[2 * M + 1]);
  const PBase dp = p_base(dPb, offb[2 * M], offb[2 * M + 1], ipad[2 * M + 1]);

  d4 acc[2][2][5];  // P pol g3, P tor, P dpol, dP dpol, dP tor
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int c = 0; c < 5; c++) acc[s][u][c] = d4{0.0, 0.0, 0.0, 0.0};
  struct Step {
    double a[2][2], b[2][2][3];
  };
  auto load = [&](int s, Step &f) {
    const long long pe = 4LL * s * d.nth_hp, po = 4LL * (s < p.o_last ? s : p.o_last) * d.nth_hp;
    f.a[0][0] = ldu(p.e + pe, vp);
    f.a[0][1] = ldu(dp.e + pe, vp);
    f.a[1][0] = ldu(p.o + po, vp);
    f.a[1][1] = ldu(dp.o + po, vp);
#pragma unroll
    for (int par = 0; par < 2; par++)
#pragma unroll
      for (int sg = 0; sg < 2; sg++)
#pragma unroll
        for (int c = 0; c < 3; c++) f.b[par][sg][c] = x.get(s, par, sg, c * cs, c == 0);
  };
  auto mul = [&](const Step &f) {
#pragma unroll
    for (int par = 0; par < 2; par++)
#pragma unroll
      for (int sg = 0; sg < 2; sg++) {
        const double *y = f.b[par][sg];
        acc[sg][par][0] = mfma64(f.a[par][0], y[0], acc[sg][par][0]);
        acc[sg][par][1] = mfma64(f.a[par][0], y[2], acc[sg][par][1]);
        acc[sg][par][2] = mfma64(f.a[par][0], y[1], acc[sg][par][2]);
        acc[sg][par][3] = mfma64(f.a[par][1], y[1], acc[sg][par][3]);
        acc[sg][par][4] = mfma64(f.a[par][1], y[2], acc[sg][par][4]);
      }
  };
  Step f0, f1;
  load(0, f0);
  int s = 0;
  for (; s + 2 <= nstep; s += 2) {
    load(s + 1, f1);
    mul(f0);
    load(s + 2 < nstep ? s + 2 : s + 1, f0);
    mul(f1);
  }
  if (s < nstep) mul(f0);
  // epilogue: N/S recombination, conjugate-slot terms, radial factors
  if (col >= d.nv * d.nr) return;
  const double a1 = a_r[k], a2 = a1 * a1;
  const bool odd_nth = (d.nth & 1) != 0;
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
    if (sg >= nsig) continue;
    const double mc = (sg == 0) ? -(double)M : (double)M;  // m of the conjugate slot
    double *ok = out + ga.slot_off[sg == 0 ? L + M : L - M] * ga.slot_mul + (long long)k * ga.s_k +
                 (long long)(3 * q) * ga.s_nd;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int t = t0 + 4 * r + (lane >> 4);
      if (t >= d.nth_h) continue;
      const bool eq = odd_nth && t == d.nth / 2;
      const double c1 = -asin_t[t] * mc * a1;
      const double E0 = acc[sg][0][0][r], O0 = acc[sg][1][0][r];
      const double E3 = acc[sg][0][3][r], O3 = acc[sg][1][3][r];
      const double E4 = acc[sg][0][4][r], O4 = acc[sg][1][4][r];
      const double Ec1 = acc[1 - sg][0][1][r], Oc1 = acc[1 - sg][1][1][r];
      const double Ec2 = acc[1 - sg][0][2][r], Oc2 = acc[1 - sg][1][2][r];
      double *o = ok + (long long)t * ga.s_t;
      if (eq) {
        o[0] = a2 * E0;
        o[ga.s_nd] = a1 * O3 + c1 * Ec1;
        o[2 * ga.s_nd] = -a1 * O4 + c1 * Ec2;
      } else {
        o[0] = a2 * (E0 + O0);
        o[ga.s_nd] = a1 * (E3 + O3) + c1 * (Ec1 + Oc1);
        o[2 * ga.s_nd] = -a1 * (E4 + O4) + c1 * (Ec2 + Oc2);
        o += (long long)(d.nth - 1 - 2 * t) * ga.s_t;
        o[0] = a2 * (E0 - O0);
        o[ga.s_nd] = a1 * (O3 - E3) + c1 * (Ec1 - Oc1);
        o[2 * ga.s_nd] = -a1 * (O4 - E4) + c1 * (Ec2 - Oc2);
      }
    }
  }
}

// Scalars: 32 hemisphere rows by two tiles of 16 columns, both slots and
// parities: 16 products per K step.
template <bool PACK>
__device__ __forceinline__ void leg_bwd_scl(
    const LegDims &d, long long id, const double *__restrict__ B, long long s_k,
    double *__restrict__ out, const GridAddr &ga, const int *__restrict__ jst,
    const long long *__restrict__ offb, const int *__restrict__ ipad,
    const double *__restrict__ Pb) {
  const int lane = threadIdx.x & 63, nct = (d.ncs + 1) / 2;
  const int t0 = (int)(id % d.nts) * 32;
  id /= d.nts;
  const int ct = (int)(id % nct) * 2, M = d.M0 + (int)(id / nct);
  if (M >= d.M0 + d.nM) return;
  const int L = d.L, nstep = (L - M + 8) / 8, nsig = (M == 0) ? 1 : 2;
  int q[2], k[2], col[2];
  SpecRows<PACK> x[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    col[c] = (ct + c) * 16 + (lane & 15);
    const int cc = col[c] < d.ns * d.nr ? col[c] : d.ns * d.nr - 1;
    q[c] = cc / d.nr;
    k[c] = cc - q[c] * d.nr;
    x[c] = spec_rows<PACK>(d, B, M, lane, 3 * d.nv + q[c], k[c],
                           ct + c < d.ncs ? col[c] : lane & 15, 48 * d.ncv, s_k, jst);
  }
  const unsigned vp = (unsigned)(((lane >> 4) * d.nth_hp + t0 + (lane & 15)) * 8);
  const PBase p = p_base(Pb, offb[2 * M], offb[2 * M + 1], ipad[2 * M + 1]);

  d4 acc[2][2][2][2];  // slot, parity, row tile, column tile
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i >> 3][(i >> 2) & 1][(i >> 1) & 1][i & 1] = d4{0.0, 0.0, 0.0, 0.0};
  struct Step {
    double a[2][2], b[2][2][2];
  };
  auto load = [&](int s, Step &f) {
    const long long pe = 4LL * s * d.nth_hp, po = 4LL * (s < p.o_last ? s : p.o_last) * d.nth_hp;
#pragma unroll
    for (int r = 0; r < 2; r++) {
      f.a[0][r] = ldu(p.e + pe + 16 * r, vp);
      f.a[1][r] = ldu(p.o + po + 16 * r, vp);
    }
#pragma unroll
    for (int par = 0; par < 2; par++)
#pragma unroll
      for (int sg = 0; sg < 2; sg++)
#pragma unroll
        for (int c = 0; c < 2; c++) f.b[par][sg][c] = x[c].get(s, par, sg, 0, false);
  };
  auto mul = [&](const Step &f) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int sg = i >> 3, par = (i >> 2) & 1, r = (i >> 1) & 1, c = i & 1;
      acc[sg][par][r][c] = mfma64(f.a[par][r], f.b[par][sg][c], acc[sg][par][r][c]);
    }
  };
  Step f0, f1;
  load(0, f0);
  int s = 0;
  for (; s + 2 <= nstep; s += 2) {
    load(s + 1, f1);
    mul(f0);
    load(s + 2 < nstep ? s + 2 : s + 1, f0);
    mul(f1);
  }
  if (s < nstep) mul(f0);
  const bool odd_nth = (d.nth & 1) != 0;
#pragma unroll
  for (int c = 0; c < 2; c++) {
    if (col[c] >= d.ns * d.nr) continue;
#pragma unroll
    for (int sg = 0; sg < 2; sg++) {
      if (sg >= nsig) continue;
      double *o = out + (long long)(3 * d.nv + q[c]) * ga.s_nd + (long long)k[c] * ga.s_k +
                  ga.slot_off[sg == 0 ? L + M : L - M] * ga.slot_mul;
#pragma unroll
      for (int r = 0; r < 8; r++) {
        const int t = t0 + 16 * (r >> 2) + 4 * (r & 3) + (lane >> 4);
        if (t >= d.nth_h) continue;
        const double E = acc[sg][0][r >> 2][c][r & 3], O = acc[sg][1][r >> 2][c][r & 3];
        if (odd_nth && t == d.nth / 2) {
          o[(long long)t * ga.s_t] = E;
        } else {
          o[(long long)t * ga.s_t] = E + O;
          o[(long long)(d.nth - 1 - t) * ga.s_t] = E - O;
        }
      }
    }
  }
}

// One launch for all fields of a call: the scalars' work-groups fill the tail
// of the vectors'.  Runs of a whole order per XCD (xcd_group_order): the row
// tiles that read the same spectra are resident together on one L2.
template <bool PACK>
__global__ void __launch_bounds__(256, 2) k_leg_bwd(
    LegDims d, const double *__restrict__ B, long long s_k, double *__restrict__ out, GridAddr ga,
    const int *__restrict__ jst, const long long *__restrict__ offb,
    const int *__restrict__ ipad, const double *__restrict__ Pb,
    const double *__restrict__ dPb, const double *__restrict__ a_r,
    const double *__restrict__ asin_t) {
  const int nw = blockDim.x >> 6;
  if (blockIdx.x < d.nbv) {
    const long long g = ((long long)d.ncv * d.ntv + nw - 1) / nw;
    const long long b = xcd_group_order(blockIdx.x, d.nbv, g);
    leg_bwd_vec<PACK>(d, b * nw + wave_of_group(), B, s_k, out, ga, jst, offb, ipad, Pb, dPb, a_r,
                      asin_t);
  } else {
    const long long g = ((long long)((d.ncs + 1) / 2) * d.nts + nw - 1) / nw;
    const long long b = xcd_group_order(blockIdx.x - d.nbv, gridDim.x - d.nbv, g);
    leg_bwd_scl<PACK>(d, b * nw + wave_of_group(), B, s_k, out, ga, jst, offb, ipad, Pb);
  }
}

// ---------------------------------------------------------------------------
// Forward for radius-fastest input (the plan's own workspace), whose rows are
// MFMA fragments as they are: 4 colatitudes by 16 columns, north and south.
// A wave forms the symmetric / antisymmetric combinations of its rows in
// registers, in the products' order, so that only a few are alive.
//
// Tiles of u pair indices are numbered through the orders, which hold fewer
// with growing M: order and first pair index of tile id.
struct FwdTile {
  int M, i0;
};
__device__ __forceinline__ FwdTile fwd_tile(const LegDims &d, long long id, int u) {
  const long long all = ceil_sum(d.L + 1 - d.M0, 2 * u);
  int lo = d.M0, hi = d.M0 + d.nM - 1;
  while (lo < hi) {  // the last order that starts at or before id
    const int mid = (lo + hi + 1) / 2;
    if (all - ceil_sum(d.L + 1 - mid, 2 * u) <= id)
      lo = mid;
    else
      hi = mid - 1;
  }
  return FwdTile{lo, (int)(id - (all - ceil_sum(d.L + 1 - lo, 2 * u))) * u};
}

// North and south rows of K step s: byte offsets within a component's order
// (rows past the equator repeat the last one; their weight is 0)
struct FwdRows {
  unsigned n, s;
};
__device__ __forceinline__ FwdRows fwd_rows(const LegDims &d, unsigned pitch, int s, int lane) {
  const int i = 4 * s + (lane >> 4), t = i < d.nth_h ? i : d.nth_h - 1;
  return FwdRows{t * pitch, (d.nth - 1 - t) * pitch};
}

// Field and radius of element e of column tile ct among nf fields' columns.
struct FwdCol {
  int q, k;
  bool ok;
};
__device__ __forceinline__ FwdCol fwd_col(const LegDims &d, int ct, int e, int nf) {
  const int i = ct * 16 + e, q = i / d.nr;
  const FwdCol c = {q, i - q * d.nr, i < nf * d.nr};
  return c.ok ? c : FwdCol{nf - 1, d.nr - 1, false};
}

// spectra of a wave's vector tile: conjugate-slot terms, degree and radial factors
__device__ __forceinline__ void fwd_vec_store(const LegDims &d, const d4 (&acc)[2][2][5], int M,
                                              int i0, int ct, int lane, double *__restrict__ sp,
                                              const SpecAddr &sa, const int *__restrict__ jst,
                                              const double *__restrict__ radius) {
  const int L = d.L, nsig = (M == 0) ? 1 : 2;
  const int ii = i0 + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const FwdCol fr = fwd_col(d, ct, 4 * r + (lane >> 4), d.nv);
    if (!fr.ok) continue;
    const int qr = fr.q, kr = fr.k;
    const double r1 = radius[kr], r2 = r1 * r1;
#pragma unroll
    for (int par = 0; par < 2; par++) {
      const int l = M + 2 * ii + par;
      if (l > L) continue;
      const double g7 = g7_of(l, M);
#pragma unroll
      for (int sg = 0; sg < 2; sg++) {
        if (sg >= nsig) continue;
        const double ms = (sg == 0) ? (double)M : -(double)M;
        double *o = sp + (long long)(jst[sg == 0 ? L + M : L - M] + l - M) * sa.s_j +
                    (long long)kr * sa.s_k + (long long)(3 * qr) * sa.s_nd;
        o[0] = r2 * g7 * acc[sg][par][0][r];
        o[sa.s_nd] = r1 * g7 * (acc[sg][par][1][r] - ms * acc[sg][par][2][r]);
        o[2 * sa.s_nd] = r1 * g7 * (-acc[sg][par][3][r] - ms * acc[sg][par][4][r]);
      }
    }
  }
}

// spectra of a wave's scalar tile
__device__ __forceinline__ void fwd_scl_store(const LegDims &d, const d4 (&acc)[2][2][2][2], int M,
                                              int i0, int ct, int lane, double *__restrict__ sp,
                                              const SpecAddr &sa, const int *__restrict__ jst) {
  const int L = d.L, nsig = (M == 0) ? 1 : 2;
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      if (ct + c >= d.ncs) continue;
      const FwdCol fr = fwd_col(d, ct + c, 4 * r + (lane >> 4), d.ns);
      if (!fr.ok) continue;
      const int qr = fr.q, kr = fr.k;
      double *ok = sp + (long long)kr * sa.s_k + (long long)(3 * d.nv + qr) * sa.s_nd;
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int par = 0; par < 2; par++) {
          const int l = M + 2 * (i0 + 16 * u + (lane & 15)) + par;
          if (l > L) continue;
          const double g6 = g6_of(l, M);
          ok[(long long)(jst[L + M] + l - M) * sa.s_j] = g6 * acc[0][par][u][c][r];
          if (nsig == 2) ok[(long long)(jst[L - M] + l - M) * sa.s_j] = g6 * acc[1][par][u][c][r];
        }
    }
}

// vectors: 16 pair indices of both parities, both slots: 20 products
__device__ __forceinline__ void leg_fwd_vec(
    const LegDims &d, long long id, int ct, const double *__restrict__ in, const GridAddr &ga,
    double *__restrict__ sp, const SpecAddr &sa, const int *__restrict__ jst,
    const long long *__restrict__ offf, const int *__restrict__ ipad,
    const double *__restrict__ Pf, const double *__restrict__ dPf,
    const double *__restrict__ radius, const double2 *__restrict__ wt) {
  const int lane = threadIdx.x & 63;
  const FwdTile ft = fwd_tile(d, id, 16);
  const int L = d.L, M = ft.M, i0 = ft.i0;
  const int ip0 = ipad[2 * M], ip1 = ipad[2 * M + 1];
  if (i0 >= ip0) return;
  const int nsig = (M == 0) ? 1 : 2;
  const FwdCol fc = fwd_col(d, ct, lane & 15, d.nv);
  const double *x = in;
  const unsigned vx = (unsigned)((fc.q * 3 * ga.s_nd + fc.k) * 8);
  const unsigned pitch = (unsigned)ga.s_t * 8;
  const long long so[2] = {ga.slot_off[L + M] * ga.slot_mul, ga.slot_off[L - M] * ga.slot_mul};
  // columns of P: an odd block may end before the even one (read the even
  // block there: its products are not stored)
  const bool has_o = i0 < ip1;
  const int ipo = has_o ? ip1 : ip0;
  const long long oe = offf[2 * M], oo = has_o ? offf[2 * M + 1] : oe;
  const unsigned ve = (unsigned)(((lane >> 4) * ip0 + i0 + (lane & 15)) * 8);
  const unsigned vo = (unsigned)(((lane >> 4) * ipo + i0 + (lane & 15)) * 8);

  d4 acc[2][2][5];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int c = 0; c < 5; c++) acc[s][u][c] = d4{0.0, 0.0, 0.0, 0.0};
  struct Step {
    double a[2][2], w, as, n[2][3], s[2][3];
  };
  auto load = [&](int s, Step &f) {
    const double2 z = wt[4 * s + (lane >> 4)];
    f.w = z.x;
    f.as = z.y;
    f.a[0][0] = ldu(Pf + oe + 4LL * s * ip0, ve);
    f.a[0][1] = ldu(dPf + oe + 4LL * s * ip0, ve);
    f.a[1][0] = ldu(Pf + oo + 4LL * s * ipo, vo);
    f.a[1][1] = ldu(dPf + oo + 4LL * s * ipo, vo);
    const FwdRows r = fwd_rows(d, pitch, s, lane);
#pragma unroll
    for (int sg = 0; sg < 2; sg++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        f.n[sg][c] = ldu(x + so[sg] + c * ga.s_nd, vx + r.n);
        f.s[sg][c] = ldu(x + so[sg] + c * ga.s_nd, vx + r.s);
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  // The weight and 1/sin go to the P fragments, which all slots and
  // components share: 6 products a step instead of 20 on the rows (FP64
  // vector operations take the matrix unit's time).  eq: the equator, in the
  // last step only, has no mirror row.
  auto mul = [&](const Step &f, bool eq) {
    double p[2], dp[2], ps[2];
#pragma unroll
    for (int par = 0; par < 2; par++) {
      p[par] = f.a[par][0] * f.w;
      dp[par] = f.a[par][1] * f.w;
      ps[par] = p[par] * f.as;
    }
#pragma unroll
    for (int sg = 0; sg < 2; sg++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const double y = eq ? 0.0 : f.s[sg][c];
        const double u = f.n[sg][c] + y;              // symmetric
        const double v = eq ? 0.0 : f.n[sg][c] - y;  // antisymmetric
        if (c == 0) {
          acc[sg][0][0] = mfma64(u, p[0], acc[sg][0][0]);
          acc[sg][1][0] = mfma64(v, p[1], acc[sg][1][0]);
        } else {
          // v_t: dP own slot (1), P / sin conjugate slot (4); v_p: 3 and 2
          const int o = c == 1 ? 1 : 3, z = c == 1 ? 4 : 2;
          acc[sg][0][o] = mfma64(v, dp[0], acc[sg][0][o]);
          acc[sg][1][o] = mfma64(u, dp[1], acc[sg][1][o]);
          acc[1 - sg][0][z] = mfma64(u, ps[0], acc[1 - sg][0][z]);
          acc[1 - sg][1][z] = mfma64(v, ps[1], acc[1 - sg][1][z]);
        }
        // keep the combinations of one component alive at a time
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  const int last = (d.nth_h + 3) / 4 - 1;
  const bool eq = (d.nth & 1) && 4 * last + (lane >> 4) >= d.nth_h - 1;
  Step f0, f1;
  load(0, f0);
  int s = 0;
  for (; s + 2 <= last; s += 2) {
    load(s + 1, f1);
    mul(f0, false);
    load(s + 2, f0);
    mul(f1, false);
  }
  if (s < last) {
    load(s + 1, f1);
    mul(f0, false);
    f0 = f1;
  }
  mul(f0, eq);
  fwd_vec_store(d, acc, M, i0, ct, lane, sp, sa, jst, radius);
}

// scalars: 32 pair indices by two tiles of 16 columns: 16 products
__device__ __forceinline__ void leg_fwd_scl(
    const LegDims &d, long long id, int ct, const double *__restrict__ in, const GridAddr &ga,
    double *__restrict__ sp, const SpecAddr &sa, const int *__restrict__ jst,
    const long long *__restrict__ offf, const int *__restrict__ ipad,
    const double *__restrict__ Pf, const double2 *__restrict__ wt) {
  const int lane = threadIdx.x & 63;
  const FwdTile ft = fwd_tile(d, id, 32);
  const int L = d.L, M = ft.M, i0 = ft.i0;
  const int ip0 = ipad[2 * M], ip1 = ipad[2 * M + 1];
  if (i0 >= ip0) return;
  const int nsig = (M == 0) ? 1 : 2;
  const double *x[2];
  unsigned vx[2];
  const unsigned pitch = (unsigned)ga.s_t * 8;
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const int cc = ct + c < d.ncs ? ct + c : d.ncs - 1;
    const FwdCol fc = fwd_col(d, cc, lane & 15, d.ns);
    x[c] = in + (long long)(3 * d.nv) * ga.s_nd;
    vx[c] = (unsigned)((fc.q * ga.s_nd + fc.k) * 8);
  }
  const long long so[2] = {ga.slot_off[L + M] * ga.slot_mul, ga.slot_off[L - M] * ga.slot_mul};
  // columns of P, 32 of them: clamped to the block (products not stored)
  const int ipo = ip1 ? ip1 : ip0;
  const double *pe = Pf + offf[2 * M], *po = Pf + (ip1 ? offf[2 * M + 1] : offf[2 * M]);
  unsigned ve[2], vo[2];
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const int ce = i0 + 16 * r < ip0 ? i0 + 16 * r : 0, co = i0 + 16 * r < ipo ? i0 + 16 * r : 0;
    ve[r] = (unsigned)(((lane >> 4) * ip0 + ce + (lane & 15)) * 8);
    vo[r] = (unsigned)(((lane >> 4) * ipo + co + (lane & 15)) * 8);
  }

  d4 acc[2][2][2][2];  // slot, parity, row tile, column tile
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i >> 3][(i >> 2) & 1][(i >> 1) & 1][i & 1] = d4{0.0, 0.0, 0.0, 0.0};
  struct Step {
    double a[2][2], n[2][2], s[2][2], w;
  };
  auto load = [&](int s, Step &f) {
    const FwdRows r = fwd_rows(d, pitch, s, lane);
    f.w = wt[4 * s + (lane >> 4)].x;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      f.a[0][u] = ldu(pe + 4LL * s * ip0, ve[u]);
      f.a[1][u] = ldu(po + 4LL * s * ipo, vo[u]);
    }
#pragma unroll
    for (int sg = 0; sg < 2; sg++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        f.n[sg][c] = ldu(x[c] + so[sg], vx[c] + r.n);
        f.s[sg][c] = ldu(x[c] + so[sg], vx[c] + r.s);
      }
  };
  auto mul = [&](const Step &f, bool eq) {
    double p[2][2];
#pragma unroll
    for (int r = 0; r < 4; r++) p[r >> 1][r & 1] = f.a[r >> 1][r & 1] * f.w;
#pragma unroll
    for (int sg = 0; sg < 2; sg++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const double y = eq ? 0.0 : f.s[sg][c];
        const double u = f.n[sg][c] + y;
        const double v = eq ? 0.0 : f.n[sg][c] - y;
#pragma unroll
        for (int r = 0; r < 2; r++) {
          acc[sg][0][r][c] = mfma64(u, p[0][r], acc[sg][0][r][c]);
          acc[sg][1][r][c] = mfma64(v, p[1][r], acc[sg][1][r][c]);
        }
      }
  };
  const int last = (d.nth_h + 3) / 4 - 1;
  const bool eq = (d.nth & 1) && 4 * last + (lane >> 4) >= d.nth_h - 1;
  Step f0, f1;
  load(0, f0);
  int s = 0;
  for (; s + 2 <= last; s += 2) {
    load(s + 1, f1);
    mul(f0, false);
    load(s + 2, f0);
    mul(f1, false);
  }
  if (s < last) {
    load(s + 1, f1);
    mul(f0, false);
    f0 = f1;
  }
  mul(f0, eq);
  fwd_scl_store(d, acc, M, i0, ct, lane, sp, sa, jst);
}

// One launch for all fields: a work-group's waves take consecutive tiles of
// one column tile (they share its rows), and the column tiles of a tile group
// run on one XCD (they share the P rows).
__global__ void __launch_bounds__(256, 2) k_leg_fwd(
    LegDims d, const double *__restrict__ in, GridAddr ga, double *__restrict__ sp, SpecAddr sa,
    const int *__restrict__ jst, const long long *__restrict__ offf,
    const int *__restrict__ ipad, const double *__restrict__ Pf,
    const double *__restrict__ dPf, const double *__restrict__ radius,
    const double2 *__restrict__ wt) {
  const int nw = blockDim.x >> 6;
  if (blockIdx.x < d.nbv) {
    const long long b = xcd_group_order(blockIdx.x, d.nbv, d.ncv);
    const long long id = b / d.ncv * nw + wave_of_group();
    if (id < d.ntv)
      leg_fwd_vec(d, id, (int)(b % d.ncv), in, ga, sp, sa, jst, offf, ipad, Pf, dPf, radius, wt);
  } else {
    const int nct = (d.ncs + 1) / 2;
    const long long b = xcd_group_order(blockIdx.x - d.nbv, gridDim.x - d.nbv, nct);
    const long long id = b / nct * nw + wave_of_group();
    if (id < d.nts)
      leg_fwd_scl(d, id, (int)(b % nct) * 2, in, ga, sp, sa, jst, offf, ipad, Pf, wt);
  }
}

// ---------------------------------------------------------------------------
// Forward, staged: a work-group's rows in LDS, as symmetric and antisymmetric
// combinations, once for its four waves instead of once a wave.  A wave then
// reads 4 fragments of P a K step from global memory where the direct form
// reads 16 (rows that start anywhere in a line cost two L1 accesses each), and
// the combinations' FP64 operations, which take the matrix unit's time, are
// shared.  Weights and 1/sin go to the P fragments and every accumulator takes
// its K steps in order, as in the direct form: the two give the same bits, so
// that the choice between them, made for a launch (one tile of orders with P
// per call), does not show in the results.
//
// NT waves along the pair indices by NC = 4 / NT along the columns, as the
// tiles of an order divide: groups of four tiles (NT = 4), then a remainder of
// two and of one, so that no wave idles.  A chunk is 4 NT rows of 16 NC
// columns, one (row, column) per thread, in two LDS buffers; the rows of the
// next chunk travel while this one is multiplied.
constexpr int kFwdWaves = 4, kPlane = 64 * kFwdWaves;  // doubles of a staged component: 4 NT x 16 NC

// sum over y = 0 .. n of floor(y / D)
__host__ __device__ inline int floor_sum(int n, int D) {
  const int q = (n + 1) / D, r = (n + 1) % D;
  return D * (q * (q - 1) / 2) + q * r;
}
// Tiles of U degrees of the orders with n, n - 8, n - 16, ... degrees: those
// of one XCD (8 divides U, so that floor((n + U - 1 - 8 j) / U) counts eighths).
template <int U>
__host__ __device__ inline int xcd_tiles(int n) {
  return n <= 0 ? 0 : floor_sum((n + U - 1) / 8, U / 8);
}
// Work-group b of a launch, eight classes of orders M0 + x, M0 + x + 8, ...
// dealt to the XCDs: all tiles of four columns tiles in turn, so that the
// groups that read the same rows run side by side on one L2.  An order of c
// tiles has c work-groups per four column tiles.
struct FwdGroup {
  int M, c, sc, r;  // order (-1: none), its tiles, column block, group within it
};
template <int U>
__device__ __forceinline__ FwdGroup fwd_group(const LegDims &d, unsigned b, int nsc) {
  const int x = b & 7, i = (int)(b >> 3), n = d.L + 1 - d.M0 - x;
  if (x >= d.nM) return FwdGroup{-1, 0, 0, 0};
  const int all = xcd_tiles<U>(n);
  int lo = 0, hi = (d.nM - 1 - x) / 8;
  while (lo < hi) {  // the last order that starts at or before i
    const int mid = (lo + hi + 1) / 2;
    if ((all - xcd_tiles<U>(n - 8 * mid)) * nsc <= i)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int c = (n - 8 * lo + U - 1) / U, in = i - (all - xcd_tiles<U>(n - 8 * lo)) * nsc;
  if (in >= c * nsc) return FwdGroup{-1, 0, 0, 0};
  return FwdGroup{d.M0 + x + 8 * lo, c, in / c, in % c};
}

// LDS position of a chunk's (column tile, row, column).  Rows of radius-slowest
// input are written along the colatitude: the columns of a row are permuted so
// that neither that nor the fragments' reads meet in a bank.
template <bool KFAST, int NT>
__device__ __forceinline__ int stage_pos(int ctl, int row, int col) {
  return (ctl * 4 * NT + row) * 16 + (KFAST ? col : col ^ (row & 15));
}

// fwd_vec_store by way of LDS, 16 x 96 doubles of the wave's own: the (r, t, p)
// of a radius's 32 degrees lie side by side there, so that a store covers runs
// of three doubles of 21 degrees, some 24 pieces of 64 bytes, instead of 64
// single doubles apart.  L = 255, Nr = 129, 9 components 1586 -> 1529 us,
// L = 511, Nr = 257 18.0 -> 17.6 ms.
__device__ __forceinline__ void fwd_vec_store_lds(const LegDims &d, const d4 (&acc)[2][2][5],
                                                  int M, int i0, int ct, int lane,
                                                  double *__restrict__ sp, const SpecAddr &sa,
                                                  const int *__restrict__ jst,
                                                  const double *__restrict__ radius,
                                                  double *__restrict__ lds) {
  const int L = d.L, nsig = (M == 0) ? 1 : 2;
  const int ii = i0 + (lane & 15);
  // element 64 s + lane of two radii: radius, degree and component
  int kk[3];
  long long off[3];
  bool in[3];
#pragma unroll
  for (int s = 0; s < 3; s++) {
    const int e = 64 * s + lane, x = e % 96 / 3;
    kk[s] = e / 96;
    off[s] = x * sa.s_j + e % 3 * sa.s_nd;
    in[s] = M + 2 * i0 + x <= L;
  }
  const FwdCol fc = fwd_col(d, ct, lane & 15, d.nv);
  const int cq = fc.ok ? fc.q : -1;
  double r1[4], g7[2];
#pragma unroll
  for (int r = 0; r < 4; r++) r1[r] = radius[fwd_col(d, ct, 4 * r + (lane >> 4), d.nv).k];
#pragma unroll
  for (int par = 0; par < 2; par++) g7[par] = g7_of(M + 2 * ii + par, M);
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
    if (sg >= nsig) continue;
    const double ms = (sg == 0) ? (double)M : -(double)M;
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int par = 0; par < 2; par++) {
        double *o = lds + (4 * r + (lane >> 4)) * 96 + (2 * (lane & 15) + par) * 3;
        o[0] = r1[r] * r1[r] * g7[par] * acc[sg][par][0][r];
        o[1] = r1[r] * g7[par] * (acc[sg][par][1][r] - ms * acc[sg][par][2][r]);
        o[2] = r1[r] * g7[par] * (-acc[sg][par][3][r] - ms * acc[sg][par][4][r]);
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double *base = sp + (long long)(jst[sg == 0 ? L + M : L - M] + 2 * i0) * sa.s_j;
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
      for (int s = 0; s < 3; s++) {
        const int c = 2 * j + kk[s], q = __shfl(cq, c), k = __shfl(fc.k, c);
        const double z = lds[192 * j + 64 * s + lane];
        if (in[s] && q >= 0) base[off[s] + 3 * q * sa.s_nd + k * sa.s_k] = z;
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// VEC: components (r, t, p) of a tile of columns; else two tiles of scalars
template <bool VEC, bool KFAST, int NT>
__device__ __forceinline__ void leg_fwd_staged(
    const LegDims &d, const FwdGroup &fg, double *__restrict__ lds,
    const double *__restrict__ in, const GridAddr &ga, double *__restrict__ sp,
    const SpecAddr &sa, const int *__restrict__ jst, const long long *__restrict__ offf,
    const int *__restrict__ ipad, const double *__restrict__ Pf,
    const double *__restrict__ dPf, const double *__restrict__ radius,
    const double2 *__restrict__ wt) {
  constexpr int NC = kFwdWaves / NT, R = 4 * NT, NX = VEC ? 3 : 2;
  constexpr int kBuf = 4 * NX * kPlane;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_of_group();
  const int L = d.L, M = fg.M, c4 = fg.c / 4;
  const int ctl = wave / NT;
  // groups of four tiles first, then those of two and of one
  const int cg = NT == 4 ? fg.sc * 4 + fg.r / c4 : NT == 2 ? fg.sc * 2 + (fg.r & 1) : fg.sc;
  const int i0 = ((NT == 4 ? fg.r % c4 * 4 : NT == 2 ? 4 * c4 : fg.c - 1) + wave % NT) * (VEC ? 16 : 32);
  if (cg * NC >= (VEC ? d.ncv : (d.ncs + 1) / 2)) return;
  const int ip0 = ipad[2 * M], ip1 = ipad[2 * M + 1];
  const long long so[2] = {ga.slot_off[L + M] * ga.slot_mul, ga.slot_off[L - M] * ga.slot_mul};

  // this thread's row and column(s)
  const int srow = KFAST ? (tid >> 4) % R : tid % R, scol = KFAST ? tid & 15 : (tid / R) & 15;
  const int sct = tid / (16 * R);
  const double *xs[VEC ? 1 : 2];
#pragma unroll
  for (int j = 0; j < (VEC ? 1 : 2); j++) {
    const int nf = VEC ? d.nv : d.ns;
    int c = VEC ? (cg * NC + sct) * 16 + scol : ((cg * NC + sct) * 2 + j) * 16 + scol;
    c = c < nf * d.nr ? c : nf * d.nr - 1;
    const int q = c / d.nr, k = c - q * d.nr;
    xs[j] = in + (VEC ? 3 * q : 3 * d.nv + q) * ga.s_nd + k * ga.s_k;
  }
  const int spos = stage_pos<KFAST, NT>(sct, srow, scol);
  const unsigned pitch = (unsigned)ga.s_t * 8;
  // pair y of the chunk's rows: slot y / NX, component y % NX
  double xn[2 * NX], xm[2 * NX];
  double2 xw;
  bool xeq;
  unsigned on = 0, os = 0;  // its rows of the chunk, bytes
  auto stage_rows = [&](int c) {
    const int i = c * R + srow, t = i < d.nth_h ? i : d.nth_h - 1;
    on = (unsigned)t * pitch;
    os = (unsigned)(d.nth - 1 - t) * pitch;
    xw = wt[i];  // 0 past the equator
    xeq = 2 * t + 1 == d.nth;
  };
  auto stage_load = [&](int y) {
    const int sg = y / NX, f = y % NX;
    const double *x = xs[VEC ? 0 : f] + so[sg] + (VEC ? f * ga.s_nd : 0);
    xn[y] = ldu(x, on);
    xm[y] = ldu(x, os);
  };
  auto stage_store = [&](double *buf, int y) {
    const double z = xeq ? 0.0 : xm[y];
    double *o = buf + 2 * y * kPlane + spos;
    o[0] = xn[y] + z;
    o[kPlane] = xeq ? 0.0 : xn[y] - z;
    if (y == 0 && scol == 0 && sct == 0) *reinterpret_cast<double2 *>(buf + kBuf + 2 * srow) = xw;
  };
  // columns of P: an odd block may end before the even one (read what is
  // there: its products are not stored), and a scalar tile's second half with
  // it.  Planes: P and dP of both parities, or P of both halves.
  const bool has_o = VEC ? i0 < ip1 : ip1 > 0;
  const int ipo = has_o ? ip1 : ip0;
  const long long oe = offf[2 * M], oo = has_o ? offf[2 * M + 1] : oe;
  const double *p1 = VEC ? dPf : Pf;
  unsigned ve[2], vo[2];
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const int i = VEC ? i0 : i0 + 16 * r;
    ve[r] = (unsigned)(((lane >> 4) * ip0 + (i < ip0 ? i : 0) + (lane & 15)) * 8);
    vo[r] = (unsigned)(((lane >> 4) * ipo + (i < ipo ? i : 0) + (lane & 15)) * 8);
  }
  struct Step {
    double a[2][2];
  };
  auto pload = [&](int s, Step &f) {
    f.a[0][0] = ldu(Pf + oe + 4LL * s * ip0, ve[0]);
    f.a[0][1] = ldu(p1 + oe + 4LL * s * ip0, ve[1]);
    f.a[1][0] = ldu(Pf + oo + 4LL * s * ipo, vo[0]);
    f.a[1][1] = ldu(p1 + oo + 4LL * s * ipo, vo[1]);
  };

  constexpr int NA = VEC ? 5 : 4;
  d4 acc[2][2][NA];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int c = 0; c < NA; c++) acc[s][u][c] = d4{0.0, 0.0, 0.0, 0.0};
  auto mul = [&](Step &f, const double *buf, int s) {
    const double *x = buf + stage_pos<KFAST, NT>(ctl, 4 * s + (lane >> 4), lane & 15);
    const double2 z = *reinterpret_cast<const double2 *>(buf + kBuf + 2 * (4 * s + (lane >> 4)));
#pragma unroll
    for (int r = 0; r < 4; r++) f.a[r >> 1][r & 1] *= z.x;
    const double ps[2] = {f.a[0][0] * z.y, f.a[1][0] * z.y};
#pragma unroll
    for (int sg = 0; sg < 2; sg++)
#pragma unroll
      for (int c = 0; c < NX; c++) {
        const double u = x[(sg * NX + c) * 2 * kPlane];            // symmetric
        const double v = x[((sg * NX + c) * 2 + 1) * kPlane];      // antisymmetric
        if (!VEC) {
#pragma unroll
          for (int r = 0; r < 2; r++) {
            acc[sg][0][2 * r + c] = mfma64(u, f.a[0][r], acc[sg][0][2 * r + c]);
            acc[sg][1][2 * r + c] = mfma64(v, f.a[1][r], acc[sg][1][2 * r + c]);
          }
        } else if (c == 0) {
          acc[sg][0][0] = mfma64(u, f.a[0][0], acc[sg][0][0]);
          acc[sg][1][0] = mfma64(v, f.a[1][0], acc[sg][1][0]);
        } else {
          // v_t: dP own slot (1), P / sin conjugate slot (4); v_p: 3 and 2
          const int o = c == 1 ? 1 : 3, k = c == 1 ? 4 : 2;
          acc[sg][0][o] = mfma64(v, f.a[0][1], acc[sg][0][o]);
          acc[sg][1][o] = mfma64(u, f.a[1][1], acc[sg][1][o]);
          acc[1 - sg][0][k] = mfma64(u, ps[0], acc[1 - sg][0][k]);
          acc[1 - sg][1][k] = mfma64(v, ps[1], acc[1 - sg][1][k]);
        }
      }
  };
  const int nstep = (d.nth_h + 3) / 4, last = nstep - 1;
  constexpr int kPitch = kBuf + 32;  // a buffer and (weight, 1/sin) of its rows
  Step f[2];
  pload(0, f[0]);
  stage_rows(0);
#pragma unroll
  for (int y = 0; y < 2 * NX; y++) stage_load(y);
#pragma unroll
  for (int y = 0; y < 2 * NX; y++) stage_store(lds, y);
  __syncthreads();
  // P one step ahead; the pairs of the next chunk a few per step, each
  // written a step after its load where the chunk has four
  constexpr int kPer = NT == 4 ? (2 * NX + 2) / 3 : 2 * NX;
  int cur = 0;
  for (int q = 0; q < nstep; q += 4) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int st = q + s, sc = s % NT;
      if (st >= nstep) break;
      const double *buf = lds + cur;
      double *nxt = lds + (kPitch - cur);
      pload(st + 1 < nstep ? st + 1 : last, f[(s + 1) & 1]);
      if (sc == 0) stage_rows(st + NT < nstep ? st / NT + 1 : 0);
#pragma unroll
      for (int y = sc * kPer; y < (sc + 1) * kPer && y < 2 * NX; y++) stage_load(y);
      __builtin_amdgcn_sched_barrier(0);
      mul(f[s & 1], buf, sc);
      __builtin_amdgcn_sched_barrier(0);
      // pairs loaded a step ago (all of them at the end of a shorter chunk)
#pragma unroll
      for (int y = NT == 4 ? (sc - 1) * kPer : sc == NT - 1 ? 0 : 2 * NX;
           y < (NT == 4 ? sc * kPer : 2 * NX) && y < 2 * NX; y++)
        if (y >= 0) stage_store(nxt, y);
      if (sc == NT - 1) {
        __syncthreads();
        cur = kPitch - cur;
      }
    }
  }
  if constexpr (VEC) {
    // a last chunk of fewer steps leaves the loop without its barrier: other
    // waves may still read the rows that the store overwrites
    __syncthreads();
    fwd_vec_store_lds(d, acc, M, i0, cg * NC + ctl, lane, sp, sa, jst, radius, lds + wave * 1536);
  } else {
    d4 q[2][2][2][2];
#pragma unroll
    for (int i = 0; i < 16; i++)
      q[i >> 3][(i >> 2) & 1][(i >> 1) & 1][i & 1] = acc[i >> 3][(i >> 2) & 1][i & 3];
    fwd_scl_store(d, q, M, i0, (cg * NC + ctl) * 2, lane, sp, sa, jst);
  }
}

// One launch for all fields: the scalars' work-groups follow the vectors'.
template <bool KFAST>
__global__ void __launch_bounds__(64 * kFwdWaves, 2) k_leg_fwd_lds(
    LegDims d, const double *__restrict__ in, GridAddr ga, double *__restrict__ sp, SpecAddr sa,
    const int *__restrict__ jst, const long long *__restrict__ offf,
    const int *__restrict__ ipad, const double *__restrict__ Pf,
    const double *__restrict__ dPf, const double *__restrict__ radius,
    const double2 *__restrict__ wt) {
  __shared__ __align__(16) double lds[2 * (12 * kPlane + 32)];
  const bool vec = blockIdx.x < d.nbv;
  const FwdGroup g = vec ? fwd_group<32>(d, blockIdx.x, (d.ncv + kFwdWaves - 1) / kFwdWaves)
                         : fwd_group<64>(d, blockIdx.x - d.nbv, ((d.ncs + 1) / 2 + kFwdWaves - 1) / kFwdWaves);
  if (g.M < 0) return;
  const int rest = g.r - (g.c & ~3);  // below 0: of a group of four
#define KSHT_KIND(VEC, NT)                                                                       \
  leg_fwd_staged<VEC, KFAST, NT>(d, g, lds, in, ga, sp, sa, jst, offf, ipad, Pf, dPf, radius, wt)
  if (vec) {
    if (rest < 0)
      KSHT_KIND(true, 4);
    else if ((g.c & 2) && rest < 2)
      KSHT_KIND(true, 2);
    else
      KSHT_KIND(true, 1);
  } else {
    if (rest < 0)
      KSHT_KIND(false, 4);
    else if ((g.c & 2) && rest < 2)
      KSHT_KIND(false, 2);
    else
      KSHT_KIND(false, 1);
  }
#undef KSHT_KIND
}

// Packed spectra: all orders of a call up to 1 GiB, else that much of them at
// a time (at least the largest order).
static int col_tiles(const sht_plan *p, int nf) { return (nf * p->nr + 15) / 16; }
static long long pack_elems(const sht_plan *p, int W) {
  const long long cap = (1LL << 30) / 8;
  const long long all = pack_rows_sum(p->L + 1) * W, one = pack_rows(p->L + 1) * W;
  return all < cap ? all : one > cap ? one : cap;
}

// Packing pays once its launch (6 to 10 us) costs less than the waves lose
// to scattered loads: L = 31, 8 components, Nr = 33 (416 waves) 14 us direct
// against 8 + 11 packed, L = 63, 4, Nr = 17 (512) 18 / 10 + 13; L = 127, 7,
// Nr = 65 (8000) 270 / 34 + 164, L = 361, 4, Nr = 63 (31000) 1400 / 130 + 720.
// Spectra past the 32-bit offsets of the direct loads are packed always.
static bool packs(const sht_plan *p, int nv, int ns) {
  const long long waves =
      (p->L + 1) * ((nv ? (long long)col_tiles(p, nv) * ((p->nth_h + 15) / 16) : 0) +
                    (ns ? (long long)((col_tiles(p, ns) + 1) / 2) * ((p->nth_h + 31) / 32) : 0));
  return waves >= 2048 || (3LL * nv + ns) * p->jmax * p->nr >= (1LL << 28);
}

int leg_init(sht_plan *p) {
  bool any = false;  // a call of the plan's that packs
  for (int nv = 0; 3 * nv <= p->max_ncomp; nv++) any |= packs(p, nv, p->max_ncomp - 3 * nv);
  // the widest rows of any call: max_ncomp scalars, or as many vectors; where
  // memory is short, fewer orders at a time
  const int W = 2 * 16 * (col_tiles(p, p->max_ncomp) + 3);
  const long long one = pack_rows(p->L + 1) * W;
  p->bp_elems = any ? pack_elems(p, W) : 0;
  std::vector<double2> wt(p->nth_hp, make_double2(0.0, 0.0));
  for (int t = 0; t < p->nth_h; t++) wt[t] = make_double2(p->weight[t], p->asin_t[t]);
  const size_t wb = sizeof(double2) * wt.size();
  while (p->bp_elems && hipMalloc(&p->Bp, sizeof(double) * (size_t)p->bp_elems) != hipSuccess) {
    p->Bp = nullptr;
    (void)hipGetLastError();
    if (p->bp_elems == one) {
      set_error("sht_plan_create: packed spectra of %lld bytes: out of device memory", 8 * one);
      return SHT_ERR_OOM;
    }
    p->bp_elems = p->bp_elems / 4 > one ? p->bp_elems / 4 : one;
  }
  KSHT_HIP(hipMalloc(&p->t.wt, wb));
  KSHT_HIP(hipMemcpy(p->t.wt, wt.data(), wb, hipMemcpyHostToDevice));
  p->device_bytes += 8 * p->bp_elems + (long long)wb;
  return SHT_OK;
}

static LegDims make_dims(const sht_plan *p, int nv, int ns) {
  LegDims d;
  d.L = p->L;
  d.nr = p->nr;
  d.nth = p->nth;
  d.nth_h = p->nth_h;
  d.nth_hp = p->nth_hp;
  d.nv = nv;
  d.ns = ns;
  d.ncomp = 3 * nv + ns;
  d.M0 = 0;
  d.nM = p->L + 1;
  d.ncv = nv ? col_tiles(p, nv) : 0;
  d.ncs = ns ? col_tiles(p, ns) : 0;
  d.ntv = (p->nth_h + 15) / 16;
  d.nts = (p->nth_h + 31) / 32;
  d.nbv = 0;
  d.W = 2 * 16 * (3 * d.ncv + d.ncs);
  return d;
}

// Waves of a work-group: four share their operands through L1; launches of
// fewer waves than the chip has SIMDs spread them one by one.
static int group_waves(long long waves) { return waves < 1024 ? 1 : 4; }
static unsigned groups(long long waves, int nw) { return (unsigned)((waves + nw - 1) / nw); }

int launch_leg_bwd(sht_plan *p, const Workspace &ws, int nv, int ns, const double *sp,
                   SpecAddr sa, double *out, GridAddr ga) {
  LegDims d = make_dims(p, nv, ns);
  const long long W = d.W, cap = ws.bp_elems > 0 ? ws.bp_elems : 1;
  const long long per_v = (long long)d.ncv * d.ntv, per_s = (long long)((d.ncs + 1) / 2) * d.nts;
  // the fixed workspace may not hold one order's rows beside the call's
  // Fourier workspace: unpacked then, the same products in the same order (its
  // calls are far below the 32-bit offsets that packs() asks about)
  const bool pack = packs(p, nv, ns) && cap >= pack_rows(p->L + 1) * W;
  int dt = 1;  // degrees of a packed run
  while (2 * dt * d.ncomp <= kPackRun) dt *= 2;
  for (int ti = 0; ti < ptile_count(p); ti++) {
    PTile pt;
    int rc = ptile_prepare(p, ti, false, &pt);
    if (rc) return rc;
    // about equal shares of the tile's orders that fit the packed buffer
    const long long all = (pack_rows_sum(p->L - pt.M0 + 1) - pack_rows_sum(p->L - pt.M1 + 1)) * W;
    const long long parts = (all + cap - 1) / cap, share = (all + parts - 1) / parts;
    for (int M0 = pt.M0, M1 = pt.M0; M0 < pt.M1; M0 = M1) {
      long long used = 0;
      if (!pack)
        M1 = pt.M1;
      else
        do used += pack_rows(p->L - M1 + 1) * W, M1++;
        while (M1 < pt.M1 && used < share && used + pack_rows(p->L - M1 + 1) * W <= cap);
      d.M0 = M0;
      d.nM = M1 - M0;
      if (pack) {
        const int nz = (int)((pack_rows(p->L - M0 + 1) + dt - 1) / dt);
        const long long nb = (p->nr + 15) / 16 * 2LL * d.nM * nz;
        hipLaunchKernelGGL(k_leg_pack, dim3((unsigned)nb), dim3(256), 0, p->stream, d, dt, nz, sp,
                           sa.s_k, p->t.jst, ws.Bp);
        KSHT_HIP(hipGetLastError());
      }
      StageTimer tk(p, 5);
      const int nw = group_waves(d.nM * (per_v + per_s));
      d.nbv = groups(d.nM * per_v, nw);
      const dim3 g(d.nbv + groups(d.nM * per_s, nw)), bl(64 * nw);
      if (pack)
        hipLaunchKernelGGL(k_leg_bwd<true>, g, bl, 0, p->stream, d, ws.Bp, sa.s_k, out, ga,
                           p->t.jst, pt.offb, p->t.ipad, pt.Pb, pt.dPb, p->t.a_r, p->t.asin_t);
      else
        hipLaunchKernelGGL(k_leg_bwd<false>, g, bl, 0, p->stream, d, sp, sa.s_k, out, ga,
                           p->t.jst, pt.offb, p->t.ipad, pt.Pb, pt.dPb, p->t.a_r, p->t.asin_t);
      KSHT_HIP(hipGetLastError());
    }
  }
  return SHT_OK;
}

// Staged from this many waves of a launch (with P per call, a tile of orders)
// on: it reads the rows once for four waves but starts and ends them together.
// Direct / staged: L = 127, 7 components, Nr = 65 (2900 waves) 143 / 163 us,
// L = 361, 4, Nr = 63 (11000) 834 / 820, L = 255, 9, Nr = 129 (29000) 1593 /
// 1446, 18, Nr = 65 (29000) 1756 / 1515, L = 511, 9, Nr = 257 (210000) 17.2 ms
// both.
constexpr long long kFwdStaged = 16384;

// work-groups of the staged forward: eight times the most of an XCD's orders
template <int U>
static unsigned fwd_groups(const LegDims &d, int nct) {
  int most = 0;
  for (int x = 0; x < 8 && x < d.nM; x++) {
    const int n = d.L + 1 - d.M0 - x, j = (d.nM - 1 - x) / 8 + 1;
    const int t = xcd_tiles<U>(n) - xcd_tiles<U>(n - 8 * j);
    most = t > most ? t : most;
  }
  return 8u * (unsigned)most * (unsigned)((nct + kFwdWaves - 1) / kFwdWaves);
}

int launch_leg_fwd(sht_plan *p, int nv, int ns, const double *in, GridAddr ga, double *sp,
                   SpecAddr sa) {
  LegDims d = make_dims(p, nv, ns);
  for (int ti = 0; ti < ptile_count(p); ti++) {
    PTile pt;
    int rc = ptile_prepare(p, ti, true, &pt);
    if (rc) return rc;
    StageTimer tk(p, 6);
    d.M0 = pt.M0;
    d.nM = pt.M1 - pt.M0;
    // direct: the lanes of a flattened tile reach every field by a 32-bit offset
    const long long lim = (1LL << 32) - 8LL * p->nr * p->nth, nd8 = 8 * ga.s_nd;
    d.ntv = (int)(ceil_sum(p->L + 1 - pt.M0, 32) - ceil_sum(p->L + 1 - pt.M1, 32));
    d.nts = (int)(ceil_sum(p->L + 1 - pt.M0, 64) - ceil_sum(p->L + 1 - pt.M1, 64));
    const long long nct = (d.ncs + 1) / 2, waves = (long long)d.ntv * d.ncv + d.nts * nct;
    if (ga.s_k == 1 && lim > 3LL * (nv - 1) * nd8 && lim > (ns - 1) * nd8 && waves < kFwdStaged) {
      const int nw = group_waves(waves);
      d.nbv = groups(d.ntv, nw) * (unsigned)d.ncv;
      const dim3 g(d.nbv + groups(d.nts, nw) * (unsigned)nct), bl(64 * nw);
      hipLaunchKernelGGL(k_leg_fwd, g, bl, 0, p->stream, d, in, ga, sp, sa, p->t.jst, pt.offf,
                         p->t.ipad, pt.Pf, pt.dPf, p->t.radius, p->t.wt);
    } else {
      d.nbv = nv ? fwd_groups<32>(d, d.ncv) : 0;
      const unsigned nb = d.nbv + (ns ? fwd_groups<64>(d, (int)nct) : 0);
      const auto kern = ga.s_k == 1 ? k_leg_fwd_lds<true> : k_leg_fwd_lds<false>;
      hipLaunchKernelGGL(kern, dim3(nb), dim3(64 * kFwdWaves), 0, p->stream, d, in, ga, sp, sa, p->t.jst,
                         pt.offf, p->t.ipad, pt.Pf, pt.dPf, p->t.radius, p->t.wt);
    }
    KSHT_HIP(hipGetLastError());
  }
  return SHT_OK;
}

}  // namespace ksht
