// tcsem_upmat.hip -- the air boundary as matrix products (gfx950, FP64 matrix cores).
//
// The upward continuation Bz(0) -> BxAir, ByAir (UpContinuation_gpu.cu:166-274) is linear and
// its three parts -- resampling to the regular plane, the wavenumber filter, sampling back -- are
// separable but for the filter, which couples x and y through exp(-|k|)/|k| only.  So with the x
// axis in wavenumbers, a(kx, j) = sum_i Ax(kx, i) Bz(j, i) with Ax the transform of the resampling
// weights, what is left per kx is a real matrix over the irregular rows,
//   Kx(kx) = Sy F^-1 diag(gx(., kx)) F Wy,
// (Wy resamples to the regular rows, Sy samples them back), and the result is a sum over kx again:
//   BxAir(j, i) = sum_kx Re( i Kx(kx) a(kx, .) V(kx, i) ),  V the sampled inverse transform.
// The regular plane never exists.  Three launches: k_dn_x (Ax), k_dn_y (the row operators), k_dn_out.
// The rows mirror about the middle of the plane (the y padding is symmetric), so each operator is
// two blocks of half the rows, one on the even and one on the odd part of a column: half the bytes.
// Built once per model on the device; FP64 data and sums throughout (the row operators are kept in
// FP32 where the FFT chain that they replace computes in FP32: their sums are FP64 here).
//
// Bound: k_dn_y reads every operator entry once per four slots (M (M + 1/2) H words), which the FFT chain
// replaces by transforms: the matrix form wins where those are long against the irregular rows or not powers of
// two (the rule is dense_pays).  The two products run at a fraction of the FP64 matrix rate
// (6 M L L1 flops).
#include "tcsem_internal.h"

namespace tcsem {

typedef double d4 __attribute__((ext_vector_type(4)));

// v_mfma_f64_16x16x4: lane l holds A[l & 15][l >> 4], B[l >> 4][l & 15] and D[4 t + (l >> 4)][l & 15].
__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

template <bool GEO, typename U>
__device__ inline U dense_record(const U &u0, const U *geo) {
  if constexpr (GEO) return geo[blockIdx.y];
  else return u0;
}

// ---- a(kx, j): P[q][j] = sum_i ax[i][q] Bz[j][i], q = 2 kx + (0 re, 1 im) -----------------------
// One workgroup per 32 x 32 tile of P: its four wavefronts take every fourth block of 16 columns i and
// meet in LDS (the sum is short, so the tile alone leaves the chip idle).  A lane's four
// columns of a block are consecutive in memory, so that a row of Bz is read as runs.
constexpr int kXWaves = 4;
template <typename T, bool GEO>
__global__ void __launch_bounds__(64 * kXWaves) k_dn_x(const UpcontArgs<T> u0, const UpcontArgs<T> *geo) {
  const UpcontArgs<T> u = dense_record<GEO>(u0, geo);
  const int W2 = 2 * u.H, M = u.M, L = u.L, slot = GEO ? 0 : (int)blockIdx.y;
  if (u.H == 0) return;  // a model batch's finished member
  const int ntj = (M + 31) / 32, tile = blockIdx.x, q0 = tile / ntj * 32, j0 = tile % ntj * 32;
  if (q0 >= W2) return;
  __shared__ double red[kXWaves][32][33];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, r = lane & 15;
  const T *bz = u.bz0 + (long long)slot * u.pstride;
  const T *b0 = bz + (long long)min(j0 + r, M - 1) * u.pz, *b1 = bz + (long long)min(j0 + 16 + r, M - 1) * u.pz;
  const double *ax = u.d.ax + q0 + r;  // columns padded to the tile
  d4 c[2][2] = {};
  for (int i0 = 16 * w; i0 < L; i0 += 16 * kXWaves) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int i = i0 + 4 * g + t, ic = min(i, L - 1);  // ax has zero rows past L
      const double y0 = (double)b0[ic], y1 = (double)b1[ic];
      const double x0 = ax[(long long)i * u.d.ldax], x1 = ax[(long long)i * u.d.ldax + 16];
      c[0][0] = mfma(x0, y0, c[0][0]);
      c[0][1] = mfma(x0, y1, c[0][1]);
      c[1][0] = mfma(x1, y0, c[1][0]);
      c[1][1] = mfma(x1, y1, c[1][1]);
    }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int t = 0; t < 4; ++t) red[w][16 * m + 4 * t + g][16 * n + r] = c[m][n][t];
  __syncthreads();
  double *P = u.d.P + (long long)slot * u.d.sP;
  for (int e = threadIdx.x; e < 1024; e += 64 * kXWaves) {
    const int q = e >> 5, j = e & 31;
    double v = red[0][q][j];
#pragma unroll
    for (int s = 1; s < kXWaves; ++s) v += red[s][q][j];
    if (q0 + q < W2 && j0 + j < M) P[(long long)(q0 + q) * u.d.MP + j0 + j] = v;
  }
}

// ---- the row operators of one kx -----------------------------------------------------------------
// One workgroup per kx and NS slots: the columns' even and odd parts in LDS, one thread per operator
// row (kop is column-major within a block, so lanes read runs), the halves' sums and differences
// through LDS.  Bound by the operator's bytes; NS slots share one read of it.
template <typename T, typename TK, int NS, bool GEO>
__global__ void __launch_bounds__(1024) k_dn_y(const UpcontArgs<T> u0, const UpcontArgs<T> *geo, int nslot) {
  const UpcontArgs<T> u = dense_record<GEO>(u0, geo);
  const int kx = blockIdx.x, M = u.M, MP = u.d.MP;
  if (kx >= u.H) return;
  const int s0 = GEO ? 0 : (int)blockIdx.y * NS;
  const int ne = (M + 1) / 2, no = M / 2, nye = M / 2 + 1, nyo = (M + 1) / 2;
  const int We = ne + nyo, Wo = no + nye;
  extern __shared__ double2 lds2[];
  double2 *in = lds2, *res = in + NS * (ne + no);  // in: [slot][even ne, odd no]; res: [slot][We + Wo]
  double2 *tau = res + NS * (We + Wo);             // [slot]
  for (int s = 0; s < NS; ++s) {
    const double *p = u.d.P + (long long)min(s0 + s, nslot - 1) * u.d.sP + (long long)(2 * kx) * MP;
    for (int j = threadIdx.x; j < ne; j += blockDim.x) {
      const double2 a = make_double2(p[j], p[MP + j]), b = make_double2(p[M - 1 - j], p[MP + M - 1 - j]);
      const bool mid = j >= no;
      in[s * M + j] = mid ? a : make_double2(a.x + b.x, a.y + b.y);
      if (!mid) in[s * M + ne + j] = make_double2(a.x - b.x, a.y - b.y);
    }
  }
  __syncthreads();
  const TK *k = (const TK *)u.d.kop + (long long)kx * u.d.kstride;
  for (int row = threadIdx.x; row < We + Wo; row += blockDim.x) {
    const bool ev = row < We;
    const int n = ev ? ne : no, ld = ev ? We : Wo;
    const TK *kr = ev ? k + row : k + (long long)ne * We + (row - We);
    const double2 *v = in + (ev ? 0 : ne);
    double2 c[NS] = {};
#pragma unroll 8
    for (int j = 0; j < n; ++j) {
      const double kv = (double)kr[(long long)j * ld];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const double2 x = v[s * M + j];
        c[s].x += kv * x.x;
        c[s].y += kv * x.y;
      }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) res[s * (We + Wo) + row] = c[s];
  }
  // the y-Nyquist bin of an even plane: By gets i gN ns(j) sum_j' nt(j') odd(j')
  const bool nyq = u.d.nt != nullptr;
  if (nyq && (int)threadIdx.x < 64) {
    for (int s = 0; s < NS; ++s) {
      double2 t = make_double2(0.0, 0.0);
      for (int j = threadIdx.x; j < no; j += 64) {
        const double2 x = in[s * M + ne + j];
        t.x += u.d.nt[j] * x.x;
        t.y += u.d.nt[j] * x.y;
      }
      for (int d = 32; d; d >>= 1) {
        t.x += __shfl_down(t.x, d);
        t.y += __shfl_down(t.y, d);
      }
      if (threadIdx.x == 0) tau[s] = make_double2(-u.d.ng[kx] * t.y, u.d.ng[kx] * t.x);
    }
  }
  __syncthreads();
  for (int s = 0; s < NS && s0 + s < nslot; ++s) {
    double *rx = u.d.Rx + (long long)(s0 + s) * u.d.sP + (long long)(2 * kx) * MP;
    double *ry = u.d.Ry + (long long)(s0 + s) * u.d.sP + (long long)(2 * kx) * MP;
    const double2 *q = res + s * (We + Wo);
    for (int j = threadIdx.x; j < ne; j += blockDim.x) {
      const double2 a = q[j];
      const bool mid = j >= no;
      const double2 b = mid ? make_double2(0.0, 0.0) : q[We + j];
      rx[j] = a.x + b.x;
      rx[MP + j] = a.y + b.y;
      if (!mid) {
        rx[M - 1 - j] = a.x - b.x;
        rx[MP + M - 1 - j] = a.y - b.y;
      }
    }
    for (int j = threadIdx.x; j < nye; j += blockDim.x) {
      const double2 a = q[We + no + j];
      const bool mid = j >= nyo;
      double2 b = mid ? make_double2(0.0, 0.0) : q[ne + j];
      if (nyq && !mid) {
        b.x += u.d.ns[j] * tau[s].x;
        b.y += u.d.ns[j] * tau[s].y;
      }
      ry[j] = a.x + b.x;
      ry[MP + j] = a.y + b.y;
      if (!mid) {
        ry[M - j] = a.x - b.x;
        ry[MP + M - j] = a.y - b.y;
      }
    }
  }
}

// ---- back to the irregular points: out[j][i] = sum_q R[q][j] b[q][i] -------------------------------
// One workgroup per 32 x 16 tile of an air plane; its wavefronts share the sum over q.  A plane gives few tiles
// (182 on 220 x 200) and the sum may be long (q < 3916 under 3914 regular columns), so latency bounds it: there 16
// wavefronts with eight loads of a stream in flight take 42 us, 8 with four took 66; short sums are the same either way.
constexpr int kOutWaves = 16;
template <typename T, bool GEO>
__global__ void __launch_bounds__(64 * kOutWaves) k_dn_out(const UpcontArgs<T> u0, const UpcontArgs<T> *geo) {
  const UpcontArgs<T> u = dense_record<GEO>(u0, geo);
  const int W2 = 2 * u.H, comp = blockIdx.z, slot = GEO ? 0 : (int)blockIdx.y;
  const int rows = comp ? u.M + 1 : u.M, cols = comp ? u.L : u.L + 1;
  const int nti = (u.L + 1 + 15) / 16, j0 = (int)blockIdx.x / nti * 32, i0 = (int)blockIdx.x % nti * 16;
  if (j0 >= rows || u.H == 0) return;
  __shared__ double red[kOutWaves][32][17];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, r = lane & 15, MP = u.d.MP, ldb = u.d.ldb;
  const double *R = (comp ? u.d.Ry : u.d.Rx) + (long long)slot * u.d.sP + j0 + r;
  const double *B = (comp ? u.d.by : u.d.bx) + i0 + r;
  d4 c0 = {}, c1 = {};
#pragma unroll 8
  for (int q = 4 * w + g; q < ((W2 + 3) & ~3); q += 4 * kOutWaves) {
    const long long o = (long long)min(q, W2 - 1) * MP;  // b has zero rows past W2
    const double b = B[(long long)q * ldb];
    c0 = mfma(R[o], b, c0);
    c1 = mfma(R[o + 16], b, c1);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    red[w][4 * t + g][r] = c0[t];
    red[w][16 + 4 * t + g][r] = c1[t];
  }
  __syncthreads();
  if (threadIdx.x >= 512) return;
  const int j = threadIdx.x >> 4, i = threadIdx.x & 15;
  double v = red[0][j][i];
#pragma unroll
  for (int s = 1; s < kOutWaves; ++s) v += red[s][j][i];
  if (j0 + j < rows && i0 + i < cols) {
    if (comp) u.byair[(long long)slot * u.pstride + (long long)(j0 + j) * u.pya + i0 + i] = (T)v;
    else u.bxair[(long long)slot * u.pstride + (long long)(j0 + j) * u.pxa + i0 + i] = (T)v;
  }
}

template <typename T, typename TK, int NS, bool GEO>
hipError_t launch_dn_y(const UpcontArgs<T> &u, int nslot, hipStream_t s, const UpcontArgs<T> *geo) {
  const size_t lds = (size_t)NS * (u.M + 2 * u.M + 1 + 1) * sizeof(double2);
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void *)k_dn_y<T, TK, NS, GEO>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const int thr = min(1024, (2 * u.M + 1 + 63) / 64 * 64);
  hipLaunchKernelGGL((k_dn_y<T, TK, NS, GEO>), dim3(u.H, GEO ? nslot : (nslot + NS - 1) / NS), dim3(thr), lds, s, u, geo,
                     GEO ? 1 : nslot);
  return hipGetLastError();
}
template <typename T, typename TK, bool GEO>
hipError_t launch_dn_y_ns(const UpcontArgs<T> &u, int nslot, hipStream_t s, const UpcontArgs<T> *geo) {
  if constexpr (!GEO) {
    const int ns = dense_share(nslot);
    if (ns == 4) return launch_dn_y<T, TK, 4, GEO>(u, nslot, s, geo);
    if (ns == 2) return launch_dn_y<T, TK, 2, GEO>(u, nslot, s, geo);
  }
  return launch_dn_y<T, TK, 1, GEO>(u, nslot, s, geo);
}
template <typename T, bool GEO>
hipError_t launch_dense_g(const UpcontArgs<T> &u, int nslot, hipStream_t s, hipEvent_t e0, hipEvent_t e1,
                          const UpcontArgs<T> *geo) {
  hipError_t e;
  const int tx = (2 * u.H + 31) / 32 * ((u.M + 31) / 32);
  launch_k(k_dn_x<T, GEO>, dim3(tx, nslot), dim3(64 * kXWaves), 0u, s, e0, nullptr, u, geo);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  e = u.d.kf32 ? launch_dn_y_ns<T, float, GEO>(u, nslot, s, geo) : launch_dn_y_ns<T, double, GEO>(u, nslot, s, geo);
  if (e != hipSuccess) return e;
  const int to = (u.M + 1 + 31) / 32 * ((u.L + 1 + 15) / 16);
  launch_k(k_dn_out<T, GEO>, dim3(to, nslot, 2), dim3(64 * kOutWaves), 0u, s, nullptr, e1, u, geo);
  return hipGetLastError();
}
// geo (model batch): u carries the largest L, M, H over the records.
template <typename T>
hipError_t launch_dense(const UpcontArgs<T> &u, int nslot, hipStream_t s, hipEvent_t e0, hipEvent_t e1,
                        const UpcontArgs<T> *geo) {
  return geo ? launch_dense_g<T, true>(u, nslot, s, e0, e1, geo) : launch_dense_g<T, false>(u, nslot, s, e0, e1, geo);
}
template hipError_t launch_dense<float>(const UpcontArgs<float> &, int, hipStream_t, hipEvent_t, hipEvent_t,
                                        const UpcontArgs<float> *);
template hipError_t launch_dense<double>(const UpcontArgs<double> &, int, hipStream_t, hipEvent_t, hipEvent_t,
                                         const UpcontArgs<double> *);

// ---- building the operators (once per model) -------------------------------------------------------
// Sum over the regular points c that irregular point i feeds, weights of the resampling windows
// (left: c < na from the first nl nodes, right: from node o on; core: one to one), of w(c) f(c).
template <typename F>
__device__ inline void each_target(int i, int na, int pad, int core, int n, int nl, int o, F &&f) {
  if (i < nl)
    for (int c = 0; c < na; ++c) f(c, 0, c, i);
  if (i >= pad && i < pad + core) f(na + i - pad, 1, 0, 0);
  if (i >= o)
    for (int c = na + core; c < n; ++c) f(c, 2, c - na - core, i - o);
}

__global__ void k_dnb_ax(const DenseBuild b, const UpcontArgs<double> u) {
  const int kx = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
  if (kx >= u.H) return;
  double re = 0.0, im = 0.0;
  each_target(i, u.AnLx, u.AL, u.Nx, u.L1, u.n1, u.Nx + u.AL - kNPad, [&](int c, int part, int p, int q) {
    const double w = part == 0 ? u.wl[(long long)q * u.AnLx + p] : part == 1 ? 1.0 : u.wr[(long long)q * u.AnRx + p];
    const double2 e = b.tx[(int)((long long)kx * c % u.L1)];
    re += w * e.x;
    im -= w * e.y;
  });
  b.ax[(long long)i * b.ldax + 2 * kx] = re;
  b.ax[(long long)i * b.ldax + 2 * kx + 1] = im;
}

__global__ void k_dnb_b(const DenseBuild b, const UpcontArgs<double> u) {
  const int ix = blockIdx.x * blockDim.x + threadIdx.x, kx = blockIdx.y;
  if (ix > u.L) return;
  const double nrm = ((kx == 0 || 2 * kx == u.L1) ? 1.0 : 2.0) / ((double)u.L1 * (double)u.M1);
  auto v = [&](int map, double x) {
    const int i1 = min(max(map, 1), u.L1 - 1);
    const double l = (x - u.Xn[i1 - 1]) / (u.Xn[i1] - u.Xn[i1 - 1]);
    const double2 e0 = b.tx[(int)((long long)kx * (i1 - 1) % u.L1)], e1 = b.tx[(int)((long long)kx * i1 % u.L1)];
    return make_double2(nrm * ((1.0 - l) * e0.x + l * e1.x), nrm * ((1.0 - l) * e0.y + l * e1.y));
  };
  const double2 e = v(u.xBx2N[ix], ix == u.L ? u.X[u.L - 1] + 0.5 * u.dx[u.L - 1] : u.X[ix] - 0.5 * u.dx[ix]);
  b.bx[(long long)(2 * kx) * b.ldb + ix] = -e.y;
  b.bx[(long long)(2 * kx + 1) * b.ldb + ix] = -e.x;
  if (ix < u.L) {
    const double2 c = v(u.xo2N[ix], u.X[ix]);
    b.by[(long long)(2 * kx) * b.ldb + ix] = c.x;
    b.by[(long long)(2 * kx + 1) * b.ldb + ix] = -c.y;
  }
}

// Cosines and sines about the plane's middle, per ky: of the resampling (cw, sw: columns j < ne), of the
// centre rows sampled back (cs, ss: j < ne) and of the edge rows (ce, se: j < M/2 + 1).
__global__ void k_dnb_y(const DenseBuild b, const UpcontArgs<double> u) {
  const int ky = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (ky >= b.Hy) return;
  const int M = u.M, M1 = u.M1, ne = (M + 1) / 2;
  auto ph = [&](int r) {  // exp(i 2 pi ky (r - (M1-1)/2) / M1)
    long long q = (long long)ky * (2 * r - M1 + 1) % (2 * M1);
    return b.ty[(int)(q < 0 ? q + 2 * M1 : q)];
  };
  const long long o = (long long)ky * b.ldy + j;
  if (j < ne) {
    double c = 0.0, s = 0.0;
    each_target(j, u.Any, u.AY, u.Ny, M1, u.n3, u.Ny + u.AY - kNPad, [&](int r, int part, int p, int q) {
      const double w = part == 0 ? u.wf[(long long)p * u.n3 + q] : part == 1 ? 1.0 : u.wb[(long long)p * u.n3 + q];
      const double2 e = ph(r);
      c += w * e.x;
      s += w * e.y;
    });
    b.cw[o] = c;
    b.sw[o] = s;
  }
  auto row = [&](int map, double y, double *c, double *s) {
    const int i1 = min(max(map, 1), M1 - 1);
    const double l = (y - u.Yn[i1 - 1]) / (u.Yn[i1] - u.Yn[i1 - 1]);
    const double2 e0 = ph(i1 - 1), e1 = ph(i1);
    c[o] = (1.0 - l) * e0.x + l * e1.x;
    s[o] = (1.0 - l) * e0.y + l * e1.y;
  };
  if (j < ne) row(u.yo2N[j], u.Y[j], b.cs, b.ss);
  row(u.yBy2N[j], u.Y[j] - 0.5 * u.dy[j], b.ce, b.se);
  if (M1 % 2 == 0 && 2 * ky == M1) {
    if (j < M / 2) b.nt[j] = b.sw[o];
    if (j < (M + 1) / 2) b.ns[j] = b.se[o];
  }
}

// Filter gains (UpContinuation_gpu.cu:113-164) of ky = 0 .. M1/2 with both signs of ky folded in, the bins
// that a real-output inverse drops set to zero; the y-Nyquist bin of By is apart (ng).
__global__ void k_dnb_gain(const DenseBuild b, const UpcontArgs<double> u) {
  const int ky = blockIdx.x * blockDim.x + threadIdx.x, kx = blockIdx.y;
  if (ky >= b.Hy) return;
  const double v = (1.0 * kPi * ky) / u.M1 * b.dzdy, w = (1.0 * kPi * kx) / u.L1 * b.dzdx;
  const bool xn = 2 * kx == u.L1, yn = 2 * ky == u.M1;
  double gx = 0.0, gy = 0.0;
  if (kx || ky) {
    const double k = sqrt(w * w + v * v), f = exp(-k) / k;
    gx = xn ? 0.0 : b.rxy * w * f * (ky == 0 || yn ? 1.0 : 2.0);
    gy = b.ryx * v * f;
  }
  b.gx[(long long)kx * b.Hy + ky] = gx;
  b.gy[(long long)kx * b.Hy + ky] = yn ? 0.0 : 2.0 * gy;
  if (yn) b.ng[kx] = kx == 0 || xn ? 0.0 : gy;
}

// The row operators: per kx four products over ky (even and odd parts of Kx and Ky), a wavefront per 32 x 32
// tile; the tables stay in L2.
template <typename TK>
__global__ void __launch_bounds__(256) k_dnb_k(const DenseBuild b, const UpcontArgs<double> u) {
  const int M = u.M, ne = (M + 1) / 2, no = M / 2, nye = M / 2 + 1, nyo = (M + 1) / 2, We = ne + nyo, Wo = no + nye;
  const int kx = blockIdx.z, part = blockIdx.y, lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const bool ev = part < 2, xc = part == 0 || part == 2;
  const int m = ev ? ne : no, n = part == 0 ? ne : part == 1 ? nyo : part == 2 ? no : nye, ld = ev ? We : Wo;
  const int tn = (n + 31) / 32, tile = blockIdx.x * 4 + (threadIdx.x >> 6), m0 = tile / tn * 32, n0 = tile % tn * 32;
  if (m0 >= m) return;
  const double *A = (ev ? b.cw : b.sw) + m0 + r;
  const double *B = (part == 0 ? b.cs : part == 1 ? b.se : part == 2 ? b.ss : b.ce) + n0 + r;
  const double *G = (xc ? b.gx : b.gy) + (long long)kx * b.Hy;
  const double sgn = part == 1 ? -1.0 : 1.0;
  d4 c[2][2] = {};
#pragma unroll 2
  for (int k0 = 0; k0 < b.Hy; k0 += 4) {
    const int ky = min(k0 + g, b.Hy - 1);
    const long long o = (long long)ky * b.ldy;
    const double w = k0 + g < b.Hy ? sgn * G[ky] : 0.0;
    const double a0 = w * A[o], a1 = w * A[o + 16], b0 = B[o], b1 = B[o + 16];
    c[0][0] = mfma(a0, b0, c[0][0]);
    c[0][1] = mfma(a0, b1, c[0][1]);
    c[1][0] = mfma(a1, b0, c[1][0]);
    c[1][1] = mfma(a1, b1, c[1][1]);
  }
  TK *K = (TK *)b.kop + (long long)kx * b.kstride + (ev ? 0 : (long long)ne * We) + (part == 1 ? ne : part == 3 ? no : 0);
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int i = m0 + 16 * p + 4 * t + g, j = n0 + 16 * q + r;
        if (i < m && j < n) K[(long long)i * ld + j] = (TK)c[p][q][t];
      }
}

hipError_t launch_dense_build(const DenseBuild &b, const UpcontArgs<double> &u, bool kf32, hipStream_t s) {
  hipError_t e;
  hipLaunchKernelGGL(k_dnb_ax, dim3((u.H + 63) / 64, u.L), dim3(64), 0, s, b, u);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_dnb_b, dim3((u.L + 1 + 63) / 64, u.H), dim3(64), 0, s, b, u);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_dnb_y, dim3((b.Hy + 63) / 64, u.M / 2 + 1), dim3(64), 0, s, b, u);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_dnb_gain, dim3((b.Hy + 63) / 64, u.H), dim3(64), 0, s, b, u);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const int t = (u.M / 2 + 1 + 31) / 32;
  const dim3 grid((t * t + 3) / 4, 4, u.H);
  if (kf32) hipLaunchKernelGGL((k_dnb_k<float>), grid, dim3(256), 0, s, b, u);
  else hipLaunchKernelGGL((k_dnb_k<double>), grid, dim3(256), 0, s, b, u);
  return hipGetLastError();
}

}  // namespace tcsem
