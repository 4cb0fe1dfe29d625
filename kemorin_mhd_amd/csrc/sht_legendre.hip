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
// The matrix units are busy 78 % of the time where a wave has many steps (low
// orders, L = 511) and about half of it for few steps or where the forward's
// rows, not multiples of a line, double its L1 accesses.  L = 511, Nr = 257:
// backward (8 components) 26.4 ms staged through LDS in its own layout, now
// 2.3 to pack and 13.2; forward (9) 36.0, now 19.4.  L = 255, Nr = 129:
// forward (9) 3.14, now 1.6.
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
  int tpv, tps;    // forward: column tiles of a group of fields, and whether
  bool flat_v, flat_s;  // it holds all of them
  int W;           // doubles per packed row
};
// the LDS-staged forward of the reference's rtm buffers
struct LegDimsLds {
  int L, nr, nth, nth_h, nth_hp, nv, ns, n_rt, ncg, nblk;
  int M0, nM;
};
constexpr int kSclPer = 4;

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

// Field and radius of element e of column tile ct; nf fields of step planes.
// Flattened over all fields (tpg = all tiles) where the fields' planes lie
// within 32-bit offsets of each other, else field by field.
struct FwdCol {
  int q, k;
  bool ok;
};
__device__ __forceinline__ FwdCol fwd_col(const LegDims &d, int ct, int e, int nf, int tpg, bool flat) {
  const int g = flat ? 0 : ct / tpg, i = (flat ? ct : ct - g * tpg) * 16 + e;
  const int q = flat ? i / d.nr : 0;
  const FwdCol c = {g + q, i - q * d.nr, i < (flat ? nf * d.nr : d.nr)};
  return c.ok ? c : FwdCol{flat ? nf - 1 : g, d.nr - 1, false};
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
  const FwdCol fc = fwd_col(d, ct, lane & 15, d.nv, d.tpv, d.flat_v);
  const int q0 = d.flat_v ? 0 : ct / d.tpv;  // uniform part of the field
  const double *x = in + (long long)(3 * q0) * ga.s_nd;
  const unsigned vx = (unsigned)(((fc.q - q0) * 3 * ga.s_nd + fc.k) * 8);
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
  const int ii = i0 + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const FwdCol fr = fwd_col(d, ct, 4 * r + (lane >> 4), d.nv, d.tpv, d.flat_v);
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
    const FwdCol fc = fwd_col(d, cc, lane & 15, d.ns, d.tps, d.flat_s);
    const int q0 = d.flat_s ? 0 : cc / d.tps;
    x[c] = in + (long long)(3 * d.nv + q0) * ga.s_nd;
    vx[c] = (unsigned)(((fc.q - q0) * ga.s_nd + fc.k) * 8);
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
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      if (ct + c >= d.ncs) continue;
      const FwdCol fr = fwd_col(d, ct + c, 4 * r + (lane >> 4), d.ns, d.tps, d.flat_s);
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
// Forward of the reference's rtm buffers, radius slowest, whose rows have to
// be transposed through LDS.  Work-group = (M, radius tile,
// component group, degree block); 4 waves, wave w owns pair indices
// i in [64*ib + 16*w, +16) of both parities (l = M + 2i + parity).  The
// reduction runs over hemisphere rows in chunks of 16 staged in LDS as
// weighted symmetric / antisymmetric combinations of the mirrored rows; the
// rows of chunk tc+1 and the P/dP fragments are prefetched into registers
// while chunk tc is reduced.
template <bool VEC>
__global__ void __launch_bounds__(256) k_leg_fwd_lds(
    LegDimsLds d, int cg0, const double *__restrict__ in, GridAddr ga, double *__restrict__ sp,
    SpecAddr sa, const int *__restrict__ jst, const long long *__restrict__ offf,
    const int *__restrict__ ipad, const double *__restrict__ Pf,
    const double *__restrict__ dPf, const double *__restrict__ radius,
    const double *__restrict__ weight, const double *__restrict__ asin_t) {
  constexpr int NC = VEC ? 3 : kSclPer;
  constexpr int NQ = VEC ? 5 : kSclPer;
  constexpr int NU = NC * 2;  // staging items per thread: 2 sig x NC x 256 / 256
  constexpr int SBUF = 2 * NC * 2 * 256;
  __shared__ double sA[2][SBUF];  // [buf][sig][f][sym/asym][tt][kk]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // logical id = ((ib (L+1) + M) n_rt + rt) ncg + cgl in runs of one (M, row
  // block) per XCD (xcd_group_order), sharing the P rows on one L2; the run
  // index ib (L+1) + M puts consecutive orders on consecutive XCDs (row
  // blocks past the degrees of M are empty, and the work of row block ib
  // would otherwise all land on two XCDs)
  long long b = xcd_group_order(blockIdx.x, gridDim.x, (long long)d.n_rt * d.ncg);
  const int cgl = (int)(b % d.ncg);
  b /= d.ncg;
  const int rt = (int)(b % d.n_rt);
  b /= d.n_rt;
  const int M = d.M0 + (int)(b % d.nM);
  const int ib = (int)(b / d.nM);
  const int L = d.L;
  const int ip0 = ipad[2 * M], ip1 = ipad[2 * M + 1];
  if (ib * 64 >= ip0) return;  // whole work-group beyond the degrees of M
  const int nsig = (M == 0) ? 1 : 2;
  const int k0 = rt * 16;
  const int i0 = ib * 64 + wave * 16;
  const bool active = i0 < ip0;
  const int cg = cg0 + cgl;
  const int nc = VEC ? 3 : min(kSclPer, d.ns - kSclPer * (cg - d.nv));
  const int nd0 = VEC ? 3 * cg : 3 * d.nv + kSclPer * (cg - d.nv);
  const long long of0 = offf[2 * M], of1 = offf[2 * M + 1];
  const int slot0 = L + M, slot1 = L - M;
  const bool odd_nth = (d.nth & 1) != 0;
  const int t_eq = odd_nth ? d.nth / 2 : -1;

  d4 acc[2][2][NQ];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < NQ; q++) acc[s][p][q] = d4{0.0, 0.0, 0.0, 0.0};

  double vn[NU], vs[NU];
  auto stage_load = [&](int tc) {
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int idx = tid + 256 * u;
      const int kk = idx & 15, tt = (idx >> 4) & 15, f = (idx >> 8) % NC, sg = idx / (256 * NC);
      const int t = tc * 16 + tt, k = k0 + kk;
      const bool valid = sg < nsig && f < nc && t < d.nth_h && k < d.nr;
      const long long base = ga.slot_off[sg == 0 ? slot0 : slot1] * ga.slot_mul +
                             (long long)(nd0 + f) * ga.s_nd + (long long)k * ga.s_k;
      vn[u] = valid ? in[base + (long long)t * ga.s_t] : 0.0;
      vs[u] = (valid && t != t_eq) ? in[base + (long long)(d.nth - 1 - t) * ga.s_t] : 0.0;
    }
  };
  auto stage_store = [&](int tc, double *buf) {
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int idx = tid + 256 * u;
      const int kk = idx & 15, tt = (idx >> 4) & 15, f = (idx >> 8) % NC, sg = idx / (256 * NC);
      const int t = tc * 16 + tt;
      const double w = t < d.nth_h ? weight[t] : 0.0;
      double *dst = buf + (((sg * NC + f) * 2) * 16 + tt) * 16 + kk;
      dst[0] = (vn[u] + vs[u]) * w;
      dst[256] = (t == t_eq) ? 0.0 : (vn[u] - vs[u]) * w;
    }
  };
  double pc[4][2], dpc[4][2], pn[4][2], dpn[4][2], asc[4], asn_[4];
  auto pload = [&](int tc, double (&a)[4][2], double (&da)[4][2], double (&as)[4]) {
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      const int t = tc * 16 + ks * 4 + (lane >> 4);
      const long long c = i0 + (lane & 15);
      const bool v1 = i0 < ip1;
      a[ks][0] = Pf[of0 + (long long)t * ip0 + c];
      a[ks][1] = v1 ? Pf[of1 + (long long)t * ip1 + c] : 0.0;
      da[ks][0] = VEC ? dPf[of0 + (long long)t * ip0 + c] : 0.0;
      da[ks][1] = (VEC && v1) ? dPf[of1 + (long long)t * ip1 + c] : 0.0;
      as[ks] = (VEC && t < d.nth_h) ? asin_t[t] : 0.0;
    }
  };

  const int nchunk = (d.nth_h + 15) / 16;
  stage_load(0);
  if (active) pload(0, pc, dpc, asc);
  for (int tc = 0; tc < nchunk; tc++) {
    double *buf = sA[tc & 1];
    stage_store(tc, buf);
    __syncthreads();
    const bool more = tc + 1 < nchunk;
    if (more) {
      stage_load(tc + 1);
      if (active) pload(tc + 1, pn, dpn, asn_);
    }
    if (active) {
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        const int tt = ks * 4 + (lane >> 4);
        const double asn = asc[ks];
#pragma unroll
        for (int par = 0; par < 2; par++) {
          if (i0 >= (par ? ip1 : ip0)) continue;
          const double bP = pc[ks][par], bdP = dpc[ks][par];
          const int sP = par, sdP = 1 - par;  // P: sym for even, dP: asym for even
#pragma unroll
          for (int sg = 0; sg < 2; sg++) {
            if (sg >= nsig) continue;
            const int sc = (nsig == 1) ? 0 : 1 - sg;
            const double *aa = buf + ((sg * NC * 2) * 16 + tt) * 16 + (lane & 15);
            const double *ac = buf + ((sc * NC * 2) * 16 + tt) * 16 + (lane & 15);
            if (VEC) {
              const double avr = aa[(0 * 2 + sP) * 256];
              const double avt = aa[(1 * 2 + sdP) * 256];
              const double avp = aa[(2 * 2 + sdP) * 256];
              const double avpc = ac[(2 * 2 + sP) * 256] * asn;
              const double avtc = ac[(1 * 2 + sP) * 256] * asn;
              acc[sg][par][0] = mfma64(avr, bP, acc[sg][par][0]);
              acc[sg][par][1] = mfma64(avt, bdP, acc[sg][par][1]);
              acc[sg][par][2] = mfma64(avpc, bP, acc[sg][par][2]);
              acc[sg][par][3] = mfma64(avp, bdP, acc[sg][par][3]);
              acc[sg][par][4] = mfma64(avtc, bP, acc[sg][par][4]);
            } else {
#pragma unroll
              for (int c = 0; c < NQ; c++)
                if (c < nc) acc[sg][par][c] = mfma64(aa[(c * 2 + sP) * 256], bP, acc[sg][par][c]);
            }
          }
        }
      }
    }
    if (more && active) {
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        asc[ks] = asn_[ks];
#pragma unroll
        for (int par = 0; par < 2; par++) {
          pc[ks][par] = pn[ks][par];
          dpc[ks][par] = dpn[ks][par];
        }
      }
    }
  }
  if (!active) return;
  const int ii = i0 + (lane & 15);
#pragma unroll
  for (int par = 0; par < 2; par++) {
    const int l = M + 2 * ii + par;
    if (l > L) continue;
    const double g7 = g7_of(l, M), g6 = g6_of(l, M);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int k = k0 + 4 * r + (lane >> 4);
      if (k >= d.nr) continue;
      const double r1 = radius[k], r2 = r1 * r1;
#pragma unroll
      for (int sg = 0; sg < 2; sg++) {
        if (sg >= nsig) continue;
        const double ms = (sg == 0) ? (double)M : -(double)M;
        const long long o = (long long)(jst[sg == 0 ? slot0 : slot1] + l - M) * sa.s_j +
                            (long long)k * sa.s_k + (long long)nd0 * sa.s_nd;
        if (VEC) {
          sp[o] = r2 * g7 * acc[sg][par][0][r];
          sp[o + sa.s_nd] = r1 * g7 * (acc[sg][par][1][r] - ms * acc[sg][par][2][r]);
          sp[o + 2 * sa.s_nd] = r1 * g7 * (-acc[sg][par][3][r] - ms * acc[sg][par][4][r]);
        } else {
#pragma unroll
          for (int c = 0; c < NQ; c++)
            if (c < nc) sp[o + (long long)c * sa.s_nd] = g6 * acc[sg][par][c][r];
        }
      }
    }
  }
}

// Packed spectra: all orders of a call up to 1 GiB, else that much of them at
// a time (at least the largest order).
static int col_tiles(const sht_plan *p, int nf) { return (nf * p->nr + 15) / 16; }
static long long pack_elems(const sht_plan *p, int W) {
  const long long cap = (1LL << 30) / 8;
  const long long all = pack_rows_sum(p->L + 1) * W, one = pack_rows(p->L + 1) * W;
  return all < cap ? all : one > cap ? one : cap;
}

int leg_init(sht_plan *p) {
  // the widest rows of any call: max_ncomp scalars, or as many vectors
  const int W = 2 * 16 * (col_tiles(p, p->max_ncomp) + 3);
  p->bp_elems = pack_elems(p, W);
  std::vector<double2> wt(p->nth_hp, make_double2(0.0, 0.0));
  for (int t = 0; t < p->nth_h; t++) wt[t] = make_double2(p->weight[t], p->asin_t[t]);
  const size_t bytes = sizeof(double) * (size_t)p->bp_elems, wb = sizeof(double2) * wt.size();
  if (hipMalloc(&p->Bp, bytes) != hipSuccess) {
    p->Bp = nullptr;
    set_error("sht_plan_create: packed spectra of %zu bytes: out of device memory", bytes);
    return SHT_ERR_OOM;
  }
  KSHT_HIP(hipMalloc(&p->t.wt, wb));
  KSHT_HIP(hipMemcpy(p->t.wt, wt.data(), wb, hipMemcpyHostToDevice));
  p->device_bytes += (long long)(bytes + wb);
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
  d.tpv = d.tps = 1;
  d.flat_v = d.flat_s = true;
  d.W = 2 * 16 * (3 * d.ncv + d.ncs);
  return d;
}

// Waves of a work-group: four share their operands through L1; launches of
// fewer waves than the chip has SIMDs spread them one by one.
static int group_waves(long long waves) { return waves < 1024 ? 1 : 4; }
static unsigned groups(long long waves, int nw) { return (unsigned)((waves + nw - 1) / nw); }

int launch_leg_bwd(sht_plan *p, int nv, int ns, const double *sp, SpecAddr sa, double *out,
                   GridAddr ga) {
  LegDims d = make_dims(p, nv, ns);
  const long long W = d.W, cap = p->bp_elems;
  const long long per_v = (long long)d.ncv * d.ntv, per_s = (long long)((d.ncs + 1) / 2) * d.nts;
  // Packing pays once its launch (6 to 10 us) costs less than the waves lose
  // to scattered loads: L = 31, 8 components, Nr = 33 (416 waves) 14 us direct
  // against 8 + 11 packed, L = 63, 4, Nr = 17 (512) 18 / 10 + 13; L = 127, 7,
  // Nr = 65 (8000) 270 / 34 + 164, L = 361, 4, Nr = 63 (31000) 1400 / 130 + 720.
  const bool pack = (p->L + 1) * (per_v + per_s) >= 2048 ||
                    (long long)p->nr * sa.s_k >= (1LL << 28);
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
                           sa.s_k, p->t.jst, p->Bp);
        KSHT_HIP(hipGetLastError());
      }
      StageTimer tk(p, 5);
      const int nw = group_waves(d.nM * (per_v + per_s));
      d.nbv = groups(d.nM * per_v, nw);
      const dim3 g(d.nbv + groups(d.nM * per_s, nw)), bl(64 * nw);
      if (pack)
        hipLaunchKernelGGL(k_leg_bwd<true>, g, bl, 0, p->stream, d, p->Bp, sa.s_k, out, ga,
                           p->t.jst, pt.offb, p->t.ipad, pt.Pb, pt.dPb, p->t.a_r, p->t.asin_t);
      else
        hipLaunchKernelGGL(k_leg_bwd<false>, g, bl, 0, p->stream, d, sp, sa.s_k, out, ga,
                           p->t.jst, pt.offb, p->t.ipad, pt.Pb, pt.dPb, p->t.a_r, p->t.asin_t);
      KSHT_HIP(hipGetLastError());
    }
  }
  return SHT_OK;
}

static int launch_leg_fwd_lds(sht_plan *p, const PTile &pt, int nv, int ns, const double *in,
                              GridAddr ga, double *sp, SpecAddr sa) {
  LegDimsLds d;
  d.L = p->L;
  d.nr = p->nr;
  d.nth = p->nth;
  d.nth_h = p->nth_h;
  d.nth_hp = p->nth_hp;
  d.nv = nv;
  d.ns = ns;
  d.n_rt = p->nr_p / 16;
  d.nblk = ((p->L + 2) / 2 + 63) / 64;
  d.M0 = pt.M0;
  d.nM = pt.M1 - pt.M0;
  const int nsg = (ns + kSclPer - 1) / kSclPer;
  ForkJoin fj(p, nv > 0 && nsg > 0);  // scalar groups beside the vector groups
  for (int vec = 1; vec >= 0; vec--) {
    d.ncg = vec ? nv : nsg;
    if (d.ncg == 0) continue;
    const hipStream_t st = fj.stream(!vec);
    const dim3 g((unsigned)((long long)d.nM * d.n_rt * d.ncg * d.nblk)), bl(256);
    if (vec) {
      StageTimer tk(p, 6);
      hipLaunchKernelGGL(k_leg_fwd_lds<true>, g, bl, 0, st, d, 0, in, ga, sp, sa, p->t.jst,
                         pt.offf, p->t.ipad, pt.Pf, pt.dPf, p->t.radius, p->t.weight, p->t.asin_t);
    } else
      hipLaunchKernelGGL(k_leg_fwd_lds<false>, g, bl, 0, st, d, nv, in, ga, sp, sa, p->t.jst,
                         pt.offf, p->t.ipad, pt.Pf, pt.dPf, p->t.radius, p->t.weight, p->t.asin_t);
    KSHT_HIP(hipGetLastError());
  }
  return SHT_OK;
}

int launch_leg_fwd(sht_plan *p, int nv, int ns, const double *in, GridAddr ga, double *sp,
                   SpecAddr sa) {
  LegDims d = make_dims(p, nv, ns);
  // the lanes of a flattened tile reach every field by a 32-bit offset
  const long long lim = (1LL << 32) - 8LL * p->nr * p->nth, nd8 = 8 * ga.s_nd;
  d.flat_v = 3LL * (nv - 1) * nd8 < lim;
  d.flat_s = (ns - 1) * nd8 < lim;
  const int tp1 = col_tiles(p, 1);
  d.tpv = d.flat_v ? d.ncv : tp1;
  d.tps = d.flat_s ? d.ncs : tp1;
  if (!d.flat_v) d.ncv = nv * tp1;
  if (!d.flat_s) d.ncs = ns * tp1;
  const long long nct = (d.ncs + 1) / 2;
  for (int ti = 0; ti < ptile_count(p); ti++) {
    PTile pt;
    int rc = ptile_prepare(p, ti, true, &pt);
    if (rc) return rc;
    if (ga.s_k != 1 || lim <= 0) {
      if ((rc = launch_leg_fwd_lds(p, pt, nv, ns, in, ga, sp, sa))) return rc;
      continue;
    }
    StageTimer tk(p, 6);
    d.M0 = pt.M0;
    d.nM = pt.M1 - pt.M0;
    d.ntv = (int)(ceil_sum(p->L + 1 - pt.M0, 32) - ceil_sum(p->L + 1 - pt.M1, 32));
    d.nts = (int)(ceil_sum(p->L + 1 - pt.M0, 64) - ceil_sum(p->L + 1 - pt.M1, 64));
    const int nw = group_waves((long long)d.ntv * d.ncv + d.nts * nct);
    d.nbv = groups(d.ntv, nw) * (unsigned)d.ncv;
    const dim3 g(d.nbv + groups(d.nts, nw) * (unsigned)nct), bl(64 * nw);
    hipLaunchKernelGGL(k_leg_fwd, g, bl, 0, p->stream, d, in, ga, sp, sa, p->t.jst, pt.offf,
                       p->t.ipad, pt.Pf, pt.dPf, p->t.radius, p->t.wt);
    KSHT_HIP(hipGetLastError());
  }
  return SHT_OK;
}

}  // namespace ksht
