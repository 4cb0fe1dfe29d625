// sht_zfold.hip -- the zonal transform as a folded real DFT on FP64 MFMA.
//
// FFTPACK's convention, as the FFT kernels (sht_fft.hip):
//   backward x_j = a_0 + sum_m (a_m cos(2 pi m j / N) + b_m sin(2 pi m j / N)),
//   forward  a_0 = (1/N) sum_j x_j, a_m = (2/N) sum_j x_j cos(.),
//            b_m = (2/N) sum_j x_j sin(.),   m <= L < N/2, N even.
// With H = N/2, the points j, N-j, H-j, H+j (0 <= j <= N/4) share one product
// per term: cos is even and sin odd under j -> N-j, and j -> H-j multiplies
// cos by (-1)^m and sin by -(-1)^m.  So with the sums over even and odd m
// kept apart (Ce, Co, Se, So),
//   x_j     = Ce + Co + Se + So,   x_(N-j) = Ce + Co - Se - So,
//   x_(H-j) = Ce - Co - Se + So,   x_(H+j) = Ce - Co + Se - So,
// and the forward folds the four points before its products.  Four GEMMs of
// (N/4) x (L/2) remain: N L flops a line, a quarter of the plain DFT, for any
// even N.
//
// A wave owns 32 rows by 32 lines of all four products (128 accumulator
// registers, two waves per SIMD) and reads both operands straight into MFMA
// fragments, one K step of 4 ahead: at 64 cycles per FP64 MFMA the 8 KB of a
// step are 8 bytes per cycle and SIMD, which L1 and L2 deliver, so nothing
// goes through LDS and no wave waits for another.  Lanes take neighbouring
// lines in pairs: 16-byte accesses, 256 contiguous bytes per row.
// Bound by HBM up to N of about 400 (N = 192: 3.4 TB/s of 1.21 before) and by
// the FP64 matrix rate above (N = 1086: 48 of about 72 TF; 8.4 ns per line
// against 82 for the mixed-radix form with its Bluestein pass).
#include <cmath>
#include <vector>

#include "sht_internal.h"

namespace ksht {

typedef double d2 __attribute__((ext_vector_type(2)));
// two neighbouring lines: rows start anywhere (odd line counts), so the
// 16-byte accesses are only 8-byte aligned
typedef d2 d2u __attribute__((aligned(8)));

struct ZfoldDims {
  int N, L, nrow, nrb, k4;    // output rows, blocks of 32 of them, K steps of 4
  int wr, ncomp, nd_inner;    // waves of a work-group along the rows; component order
  unsigned nrg, nlg, nlb;     // row groups, line groups, 32-line blocks
  long long nline;
};

struct ZfoldWave {
  int rb, nd;
  unsigned lb;
  bool ok;
};

// Logical work-group: row groups fastest (they share their lines' input),
// then lines, then components; where the components interleave, components
// before lines.  Contiguous ranges per XCD keep a line's rows in one L2.
__device__ __forceinline__ ZfoldWave zfold_wave(const ZfoldDims &d) {
  const unsigned nb = gridDim.x, per = nb / 8, b = blockIdx.x;
  const unsigned lid = b >= per * 8 ? b : (b % 8) * per + b / 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const unsigned rg = lid % d.nrg, rest = lid / d.nrg;
  const unsigned lg = d.nd_inner ? rest / d.ncomp : rest % d.nlg;
  ZfoldWave w;
  w.nd = (int)(d.nd_inner ? rest % d.ncomp : rest / d.nlg);
  w.rb = (int)rg * d.wr + wave % d.wr;
  w.lb = lg * (unsigned)(nw / d.wr) + (unsigned)(wave / d.wr);
  w.ok = w.rb < d.nrb && w.lb < d.nlb;
  return w;
}

__device__ __forceinline__ d4 zmfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// table element of (row block, K step): [type][lane][row tile]
__device__ __forceinline__ void zfold_tab(const double *__restrict__ t, int lane, d2 (&a)[4]) {
#pragma unroll
  for (int ty = 0; ty < 4; ty++) a[ty] = *reinterpret_cast<const d2 *>(t + ty * 128 + lane * 2);
}

template <bool ADJ>
__device__ __forceinline__ d2 zfold_ld(const double *__restrict__ p, long long s) {
  if constexpr (ADJ)
    return *reinterpret_cast<const d2u *>(p);
  else
    return d2{p[0], p[s]};
}

__device__ __forceinline__ void zfold_mul(const d2 (&a)[4], const d2 (&b)[4], d4 (&acc)[4][2][2]) {
#pragma unroll
  for (int ty = 0; ty < 4; ty++)
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
      for (int ct = 0; ct < 2; ct++) acc[ty][rt][ct] = zmfma(a[ty][rt], b[ty][ct], acc[ty][rt][ct]);
}

// Fourier coefficients -> grid.  ADJ: neighbouring lines are adjacent on the
// Fourier side.
template <bool ADJ>
__global__ void __launch_bounds__(256, 2) k_zfold_bwd(ZfoldDims d, const double *__restrict__ X,
                                                      FourierAddr xa, double *__restrict__ v,
                                                      const double *__restrict__ tab) {
  const ZfoldWave w = zfold_wave(d);
  if (!w.ok) return;
  const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
  const long long line = (long long)w.lb * 32 + 2 * col;
  const long long l0 = line < d.nline - 1 ? line : d.nline - 2;
  const double *x = X + (long long)w.nd * xa.s_nd + l0 * xa.s_line;
  const double *t = tab + (long long)w.rb * d.k4 * 512;
  const int Le = d.L & ~1, Lo = (d.L - 1) | 1;  // largest even and odd orders
  d4 acc[4][2][2];
#pragma unroll
  for (int ty = 0; ty < 4; ty++)
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
      for (int ct = 0; ct < 2; ct++) acc[ty][rt][ct] = d4{0.0, 0.0, 0.0, 0.0};
  // The highest orders first: coefficients fall with m, so the partial sums
  // stay small until the last steps.  Falling as (m + 1)^-1.5, N = 192, 540,
  // 1086, relative L2 against 80-bit sums: 1.2e-16 each; lowest first 2.6, 4.5,
  // 6.3e-16, the mixed-radix FFT 1.3, 1.8, 2.4e-16.  Equal coefficients, either
  // order: 2.1, 3.3, 4.6e-16, the FFT 1.8, 2.6, 2.9e-16.
  // Rows past the last order repeat it (their table entries are zero), and
  // the sine row of m = 0 is the cosine's (sin 0 = 0).
  auto load = [&](int step, d2 (&a)[4], d2 (&b)[4]) {
    const int ks = d.k4 - 1 - step, i = ks * 4 + kq;
    const int me = 2 * i < Le ? 2 * i : Le, mo = 2 * i + 1 < Lo ? 2 * i + 1 : Lo;
    const int f = xa.fftpack;
    const int qe = me ? 2 * me - 1 + f : 0, qs = me ? qe + 1 : 0, qo = 2 * mo - 1 + f;
    zfold_tab(t + (long long)ks * 512, lane, a);
    b[0] = zfold_ld<ADJ>(x + (unsigned long long)(unsigned)qe * (unsigned)xa.q_stride, xa.s_line);
    b[1] = zfold_ld<ADJ>(x + (unsigned long long)(unsigned)qo * (unsigned)xa.q_stride, xa.s_line);
    b[2] = zfold_ld<ADJ>(x + (unsigned long long)(unsigned)qs * (unsigned)xa.q_stride, xa.s_line);
    b[3] = zfold_ld<ADJ>(x + (unsigned long long)(unsigned)(qo + 1) * (unsigned)xa.q_stride, xa.s_line);
  };
  d2 a0[4], b0[4], a1[4], b1[4];
  load(0, a0, b0);
  int ks = 0;
  for (; ks + 2 <= d.k4; ks += 2) {
    load(ks + 1, a1, b1);
    zfold_mul(a0, b0, acc);
    load(ks + 2 < d.k4 ? ks + 2 : ks + 1, a0, b0);
    zfold_mul(a1, b1, acc);
  }
  if (ks < d.k4) zfold_mul(a0, b0, acc);
  if (line >= d.nline) return;
  const int N = d.N, H = N / 2;
  double *o = v + (long long)w.nd * N * d.nline + l0;
#pragma unroll
  for (int rt = 0; rt < 2; rt++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int j = w.rb * 32 + rt * 16 + 4 * r + kq;
      if (j >= d.nrow) continue;
      d2 e, f, g, h;
#pragma unroll
      for (int ct = 0; ct < 2; ct++) {
        e[ct] = acc[0][rt][ct][r] + acc[1][rt][ct][r];
        f[ct] = acc[0][rt][ct][r] - acc[1][rt][ct][r];
        g[ct] = acc[2][rt][ct][r] + acc[3][rt][ct][r];
        h[ct] = acc[3][rt][ct][r] - acc[2][rt][ct][r];
      }
      *reinterpret_cast<d2u *>(o + (long long)j * d.nline) = e + g;
      if (j) *reinterpret_cast<d2u *>(o + (long long)(N - j) * d.nline) = e - g;
      if (2 * j != H) {
        *reinterpret_cast<d2u *>(o + (long long)(H - j) * d.nline) = f + h;
        if (j) *reinterpret_cast<d2u *>(o + (long long)(H + j) * d.nline) = f - h;
      }
    }
}

// grid -> Fourier coefficients (orders m <= L).
template <bool ADJ>
__global__ void __launch_bounds__(256, 2) k_zfold_fwd(ZfoldDims d, const double *__restrict__ v,
                                                      double *__restrict__ X, FourierAddr xa,
                                                      const double *__restrict__ tab) {
  const ZfoldWave w = zfold_wave(d);
  if (!w.ok) return;
  const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
  const long long line = (long long)w.lb * 32 + 2 * col;
  const long long l0 = line < d.nline - 1 ? line : d.nline - 2;
  const int N = d.N, H = N / 2, jm = N / 4;
  const double *x = v + (long long)w.nd * N * d.nline + l0;
  const double *t = tab + (long long)w.rb * d.k4 * 512;
  d4 acc[4][2][2];
#pragma unroll
  for (int ty = 0; ty < 4; ty++)
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
      for (int ct = 0; ct < 2; ct++) acc[ty][rt][ct] = d4{0.0, 0.0, 0.0, 0.0};
  const unsigned ls = (unsigned)d.nline;
  // No such order here: the points weigh alike, and a sum of N/4 rounds more
  // than an FFT's log N levels: N = 192, 540, 1086, 2160 2.7, 4.4, 6.6, 8.7e-16
  // against 1.6, 2.0, 3.0, 2.2e-16.  The Legendre sums of a whole transform add
  // ten times that and more, and its error is the same with either.
  // j = 0 reads x_0 and x_H twice and j = N/4 its two points twice: their
  // table entries are halved; rows past N/4 repeat it against zeros
  auto load = [&](int ks, d2 (&a)[4], d2 (&b)[4]) {
    const int i = ks * 4 + kq, j = i < jm ? i : jm;
    zfold_tab(t + (long long)ks * 512, lane, a);
    b[0] = zfold_ld<true>(x + (unsigned long long)(unsigned)j * ls, 1);
    b[1] = zfold_ld<true>(x + (unsigned long long)(unsigned)(j ? N - j : 0) * ls, 1);
    b[2] = zfold_ld<true>(x + (unsigned long long)(unsigned)(H - j) * ls, 1);
    b[3] = zfold_ld<true>(x + (unsigned long long)(unsigned)(H + j) * ls, 1);
  };
  auto mul = [&](const d2 (&a)[4], const d2 (&b)[4]) {
    const d2 p = b[0] + b[1], q = b[2] + b[3], u = b[0] - b[1], e = b[2] - b[3];
    const d2 g[4] = {p + q, p - q, u - e, u + e};
    zfold_mul(a, g, acc);
  };
  d2 a0[4], b0[4], a1[4], b1[4];
  load(0, a0, b0);
  int ks = 0;
  for (; ks + 2 <= d.k4; ks += 2) {
    load(ks + 1, a1, b1);
    mul(a0, b0);
    load(ks + 2 < d.k4 ? ks + 2 : ks + 1, a0, b0);
    mul(a1, b1);
  }
  if (ks < d.k4) mul(a0, b0);
  if (line >= d.nline) return;
  double *o = X + (long long)w.nd * xa.s_nd + l0 * xa.s_line;
  auto put = [&](int q, int ty, int rt, int r) {
    double *p = o + q_offset(xa, q);
    const d2 z = {acc[ty][rt][0][r], acc[ty][rt][1][r]};
    if constexpr (ADJ)
      *reinterpret_cast<d2u *>(p) = z;
    else {
      p[0] = z.x;
      p[xa.s_line] = z.y;
    }
  };
#pragma unroll
  for (int rt = 0; rt < 2; rt++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = 2 * (w.rb * 32 + rt * 16 + 4 * r + kq);
      if (m <= d.L) {
        put(m ? 2 * m - 1 : 0, 0, rt, r);
        if (m) put(2 * m, 2, rt, r);
      }
      if (m + 1 <= d.L) {
        put(2 * m + 1, 1, rt, r);
        put(2 * m + 2, 3, rt, r);
      }
    }
}

// Tables of both directions, in the order the waves read them.
int zfold_init(sht_plan *p) {
  if (p->t.zfb) return SHT_OK;
  const int N = p->nphi, H = N / 2, L = p->L, J = N / 4 + 1, I = L / 2 + 1;
  // cos and sin of 2 pi k / N from the first quarter (N is even)
  const long double w0 = 2.0L * 3.14159265358979323846264338327950288L / (long double)N;
  std::vector<long double> root[2] = {std::vector<long double>(N), std::vector<long double>(N)};
  std::vector<long double> &c = root[0], &s = root[1];
  for (int k = 0; k <= N / 4; k++) {
    c[k] = 4 * k == N ? 0.0L : cosl(w0 * k);
    s[k] = sinl(w0 * k);
    c[H - k] = 4 * k == N ? 0.0L : -c[k];
    s[H - k] = s[k];
  }
  for (int k = 1; k < H; k++) {
    c[N - k] = c[k];
    s[N - k] = -s[k];
  }
  for (int dir = 0; dir < 2; dir++) {
    const bool bwd = dir == 0;
    const int rows = bwd ? J : I, kd = bwd ? I : J;
    const int nrb = (rows + 31) / 32, k4 = (kd + 3) / 4;
    std::vector<double> z[2] = {std::vector<double>(N), std::vector<double>(N)};
    for (int f = 0; f < 2; f++)
      for (int k = 0; k < N; k++)
        z[f][k] = (double)(bwd ? root[f][k] : 2.0L * root[f][k] / (long double)N);
    std::vector<double> tab((size_t)nrb * k4 * 512, 0.0);
    for (int r = 0; r < rows; r++) {
      double *row = tab.data() + (size_t)(r / 32) * k4 * 512 + (r & 15) * 2 + ((r >> 4) & 1);
      for (int par = 0; par < 2; par++) {
        // m j mod N along the row: m = 2i + par
        const long long m0 = bwd ? par : 2 * r + par;
        if (m0 > L) continue;
        int a = bwd ? par * r : 0;
        const int step = (int)((bwd ? 2LL * r : m0) % N);
        for (int k = 0; k < kd; k++) {
          if (bwd && 2 * k + par > L) break;
          // the points 0, H and N/4, 3N/4 are read twice by the forward
          const double h = !bwd && (k == 0 || 4 * k == N) ? 0.5 : 1.0;
          double *e = row + (size_t)(k / 4) * 512 + (k & 3) * 32 + par * 128;
          e[0] = h * z[0][a];
          e[256] = h * z[1][a];
          a += step;
          if (a >= N) a -= N;
        }
      }
    }
    if (!bwd)  // m = 0 has weight 1/N
      for (int k = 0; k < kd; k++) tab[(size_t)(k / 4) * 512 + (k & 3) * 32] *= 0.5;
    double **dst = bwd ? &p->t.zfb : &p->t.zff;
    const size_t bytes = sizeof(double) * tab.size();
    if (hipMalloc(dst, bytes) != hipSuccess) {
      *dst = nullptr;
      set_error("zonal DFT tables of %zu bytes: out of device memory", bytes);
      return SHT_ERR_OOM;
    }
    KSHT_HIP(hipMemcpy(*dst, tab.data(), bytes, hipMemcpyHostToDevice));
    p->device_bytes += (long long)bytes;
  }
  return SHT_OK;
}

int launch_zfold(sht_plan *p, int ncomp, bool bwd, const double *in, double *out, FourierAddr xa) {
  ZfoldDims d;
  const int J = p->nphi / 4 + 1, I = p->L / 2 + 1;
  d.N = p->nphi;
  d.L = p->L;
  d.nrow = bwd ? J : I;
  d.nrb = (d.nrow + 31) / 32;
  d.k4 = ((bwd ? I : J) + 3) / 4;
  d.ncomp = ncomp;
  d.nd_inner = xa.s_line != 1;
  d.nline = (long long)p->nr * p->nth;
  d.nlb = (unsigned)((d.nline + 31) / 32);
  // few waves: one per work-group spreads them over the CUs; otherwise four,
  // two by two over rows and lines where the row blocks pair up
  const int nw = (long long)d.nrb * d.nlb * ncomp < 4096 ? 1 : 4;
  d.wr = nw == 4 && d.nrb % 2 == 0 ? 2 : 1;
  d.nrg = (unsigned)((d.nrb + d.wr - 1) / d.wr);
  d.nlg = (d.nlb + (unsigned)(nw / d.wr) - 1) / (unsigned)(nw / d.wr);
  const long long nb = (long long)d.nrg * d.nlg * ncomp;
  if (nb > 0x7fffffffLL || xa.q_stride > 0x7fffffffLL) {
    set_error("zonal DFT: %lld work-groups, row stride %lld: out of range", nb, xa.q_stride);
    return SHT_ERR_UNSUPPORTED;
  }
  const dim3 g((unsigned)nb), bl(64 * nw);
  if (bwd) {
    if (xa.s_line == 1)
      hipLaunchKernelGGL(k_zfold_bwd<true>, g, bl, 0, p->stream, d, in, xa, out, p->t.zfb);
    else
      hipLaunchKernelGGL(k_zfold_bwd<false>, g, bl, 0, p->stream, d, in, xa, out, p->t.zfb);
  } else {
    if (xa.s_line == 1)
      hipLaunchKernelGGL(k_zfold_fwd<true>, g, bl, 0, p->stream, d, in, out, xa, p->t.zff);
    else
      hipLaunchKernelGGL(k_zfold_fwd<false>, g, bl, 0, p->stream, d, in, out, xa, p->t.zff);
  }
  KSHT_HIP(hipGetLastError());
  return SHT_OK;
}

}  // namespace ksht
