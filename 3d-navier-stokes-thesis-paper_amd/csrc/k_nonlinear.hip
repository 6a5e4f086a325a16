// Physical-space pass of the nonlinear term (PFC/pass1.f90:26-252) and of
// its linearized variant (PFC/pass1_linearized.f90:135-509), fused per z-row.
//
// A workgroup owns `rz` physical z-rows and a chunk of y-planes.  Thread
// (r, n) owns the two physical points x = 2n, 2n+1 of row r, which are the
// real and imaginary parts of point n of the half-length complex FFT used
// for every x transform.  Walking up the chunk, it keeps in registers the
// velocity at planes k and k+1 and the wall-normal fluxes at y(k-1), yh(k),
// exactly the sliding window of the reference (u = up at :81), so each plane
// is inverse transformed once per chunk plus one halo plane.
//
// Per plane k the workgroup
//   1. x-c2r's the z-inverse rows of u, v, w at plane k+1 (three half-length
//      backward FFTs per row),
//   2. forms the flux products and y-differences (:138-195),
//   3. forward x-transforms the 8 distinct real fields (u^2, d/dy flux_u,
//      w u, d/dy flux_w, w^2, the two interpolated v fluxes, d/dy flux_v),
//   4. combines A = F(fy) + i kx F(fx) and B = F(fz) for each component
//      (PFC/transform.f90:613) and writes them for the z-forward pass.
// At rk_step == 1 it also accumulates the per-plane CFL maxima (:202-217).
#include <type_traits>
#include "chan_internal.h"

__device__ __forceinline__ double2 c2r_pack_nl(const double2* __restrict__ row, int nxh, int M,
                                               int n, double2 wconj) {
  double2 a = make_double2(0.0, 0.0), b = make_double2(0.0, 0.0);
  if (n < nxh) { a = row[n]; if (n == 0 || n == M) a.y = 0.0; }
  int m = M - n;
  if (m < nxh) { b = row[m]; if (m == 0 || m == M) b.y = 0.0; b.y = -b.y; }
  return c2r_combine(a, b, wconj);
}

// Twice the real transform's coefficient k from the half-length transform
// (Z_k + conj Z_{M-k}) - i w^k (Z_k - conj Z_{M-k}); the z-forward pass halves
// it with its own scale.
template <int MC>
__device__ __forceinline__ double2 r2c_post_nl(const double2* __restrict__ Zs, int M, int k, double2 wk) {
  const double2 a = Zs[fft_out_pos<MC>(k % M)], b = cconj(Zs[fft_out_pos<MC>((M - k) % M)]);
  return r2c_combine(a, b, wk);
}

// elementwise helpers on the pair of points (x = 2n, 2n+1)
__device__ __forceinline__ double2 pmul(double2 a, double2 b) { return make_double2(a.x * b.x, a.y * b.y); }
__device__ __forceinline__ double2 padd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 psub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 psc(double s, double2 a) { return make_double2(s * a.x, s * a.y); }
__device__ __forceinline__ double pabsmax(double2 a) { return fmax(fabs(a.x), fabs(a.y)); }

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

template <bool LIN, int MC>
__global__ __launch_bounds__(640) void k_xpass(XZGeom g, const double2* __restrict__ tw, DevOps ops,
                                                XPassArgs a) {
  extern __shared__ double2 lds[];
  const int M = MC > 0 ? MC : g.nx2 / 2, SS = fft_seq_cells(M), RZ = a.rz;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int r = tid / M, n = tid - r * M;
  const bool act = r < RZ;
  const int zz = blockIdx.x * RZ + (act ? r : 0);
  const int ny = a.ny, nyp = ny + 1;
  const int ka = a.ka + blockIdx.y * a.chunk;
  const int kb = min(a.kb, ka + a.chunk - 1);
  const int nz2 = g.nz2, kxp = g.kxpad, nxh = g.nxh;
  const double2* rootx = tw + g.twx;
  const double2 wconj = cconj(rootx[n < M ? n : 0]);
  double2* rl = lds + 8 * RZ * SS;
  load_tw2<MC>(rl, tw + g.px.tw, tid, nthr);
  const int pin = fft_in_pos<MC>(n < M ? n : 0), pout = fft_out_pos<MC>(n < M ? n : 0);
  const long rowoff = (long)zz * kxp;

  double2 buf = make_double2(0.0, 0.0);
  const bool hasbuf = ops.buffer != nullptr;
  if (hasbuf && act) buf = *reinterpret_cast<const double2*>(ops.buffer + (long)zz * g.nx2 + 2 * n);

  // c2r of plane p (1-based reference plane) for the components in cmask
  auto load_plane = [&](int p, double2& U, double2& V, double2& W, bool needv) {
    const int nc = 3;
    for (int c = 0; c < nc; ++c) {
      double2 v = make_double2(0.0, 0.0);
      if (act && (c != 1 || needv)) {
        const double2* row = a.Z + ((long)(c * nyp + (p - 1)) * nz2) * kxp + rowoff;
        v = c2r_pack_nl(row, nxh, M, n, wconj);
      }
      if (act) lds[(c * RZ + r) * SS + pin] = v;
    }
    __syncthreads();
    fft_run<MC, 1, 12>(lds, SS, 3 * RZ, g.px, tw, rl, tid, nthr);
    if (act) {
      U = lds[(0 * RZ + r) * SS + pout];
      V = lds[(1 * RZ + r) * SS + pout];
      W = lds[(2 * RZ + r) * SS + pout];
    }
    __syncthreads();
  };
  auto load_base = [&](int p, double2& U, double2& V, double2& W) {
    if (!LIN || !act) return;
    const double* b = a.base;
    long o = ((long)(p - 1) * nz2 + zz) * g.nx2 + 2 * n;
    long cs = (long)nyp * nz2 * g.nx2;
    U = *reinterpret_cast<const double2*>(b + o);
    V = *reinterpret_cast<const double2*>(b + cs + o);
    W = *reinterpret_cast<const double2*>(b + 2 * cs + o);
  };

  double2 U0 = {0, 0}, V0 = {0, 0}, W0 = {0, 0}, U1 = {0, 0}, V1 = {0, 0}, W1 = {0, 0};
  double2 BU0 = {0, 0}, BV0 = {0, 0}, BW0 = {0, 0}, BU1 = {0, 0}, BV1 = {0, 0}, BW1 = {0, 0};
  double2 FU, FW, GV;
  const double half = 0.5, two = 2.0;

  // prologue: planes ka-1 and ka, fluxes at y(ka-1) and yh(ka)
  load_plane(ka - 1, U0, V0, W0, true);
  load_base(ka - 1, BU0, BV0, BW0);
  load_plane(ka, U1, V1, W1, true);
  load_base(ka, BU1, BV1, BW1);
  if (!LIN) {
    if (ka - 1 == 1) { FU = pmul(V0, U0); FW = pmul(V0, W0); }                 // :53,56
    else { FU = pmul(V0, psc(half, padd(U0, U1))); FW = pmul(V0, psc(half, padd(W0, W1))); }
    double2 t = psc(half, padd(V0, V1)); GV = pmul(t, t);                        // :54-55
  } else {
    if (ka - 1 == 1) {                                                          // lin :160-170
      FU = padd(pmul(BV0, U0), pmul(V0, BU0));
      FW = padd(pmul(BV0, W0), pmul(V0, BW0));
    } else {                                                                    // lin :265-273
      FU = padd(pmul(psc(half, BV0), padd(U0, U1)), pmul(psc(half, V0), padd(BU0, BU1)));
      FW = padd(pmul(psc(half, BV0), padd(W0, W1)), pmul(psc(half, V0), padd(BW0, BW1)));
    }
    double2 t = psc(half, padd(V0, V1)), tb = psc(half, padd(BV0, BV1));
    GV = pmul(psc(two, t), tb);
  }
  U0 = U1; V0 = V1; W0 = W1; BU0 = BU1; BV0 = BV1; BW0 = BW1;

  for (int k = ka; k <= kb; ++k) {
    const bool top = (k == ny);
    load_plane(k + 1, U1, V1, W1, !top);
    load_base(k + 1, BU1, BV1, BW1);
    const int kk = k - 1;  // 0-based plane index
    const double dh = ops.dh[kk];
    // wall-parallel fluxes at y(k) (:138-146)
    double2 Fu, Fw;
    if (!LIN) {
      if (!top) { Fu = pmul(V0, psc(half, padd(U0, U1))); Fw = pmul(V0, psc(half, padd(W0, W1))); }
      else { Fu = pmul(V0, U1); Fw = pmul(V0, W1); }
    } else {
      if (!top) {
        Fu = padd(pmul(psc(half, BV0), padd(U0, U1)), pmul(psc(half, V0), padd(BU0, BU1)));
        Fw = padd(pmul(psc(half, BV0), padd(W0, W1)), pmul(psc(half, V0), padd(BW0, BW1)));
      } else {
        Fu = padd(pmul(BV0, U1), pmul(V0, BU1));
        Fw = padd(pmul(BV0, W1), pmul(V0, BW1));
      }
    }
    double2 yfu = psc(dh, psub(Fu, FU));
    double2 yfw = psc(dh, psub(Fw, FW));
    if (hasbuf) {
      double tu = ops.target[0 * nyp + kk], tw_ = ops.target[2 * nyp + kk];
      yfu = padd(yfu, pmul(buf, make_double2(U0.x - tu, U0.y - tu)));
      yfw = padd(yfw, pmul(buf, make_double2(W0.x - tw_, W0.y - tw_)));
    }
    const int nf = top ? 5 : 8;
    double2 fld[8];
    if (!LIN) {
      fld[0] = pmul(U0, U0);          // x-flux of u
      fld[2] = pmul(W0, U0);          // z-flux of u == x-flux of w
      fld[4] = pmul(W0, W0);          // z-flux of w
    } else {
      fld[0] = pmul(psc(two, BU0), U0);
      fld[2] = padd(pmul(BW0, U0), pmul(W0, BU0));
      fld[4] = pmul(psc(two, BW0), W0);
    }
    fld[1] = yfu;
    fld[3] = yfw;
    double2 G1 = {0, 0};
    if (!top) {
      const double i1 = ops.iu[2 * kk], i2 = ops.iu[2 * kk + 1];
      if (!LIN) {
        double2 t = psc(half, padd(V0, V1)); G1 = pmul(t, t);
        fld[5] = pmul(V0, padd(psc(i1, U0), psc(i2, U1)));
        fld[7] = pmul(V0, padd(psc(i1, W0), psc(i2, W1)));
      } else {
        double2 t = psc(half, padd(V0, V1)), tb = psc(half, padd(BV0, BV1));
        G1 = pmul(psc(two, t), tb);
        fld[5] = padd(pmul(BV0, padd(psc(i1, U0), psc(i2, U1))), pmul(V0, padd(psc(i1, BU0), psc(i2, BU1))));
        fld[7] = padd(pmul(BV0, padd(psc(i1, W0), psc(i2, W1))), pmul(V0, padd(psc(i1, BW0), psc(i2, BW1))));
      }
      double2 yfv = psc(ops.dn[kk], psub(G1, GV));                                 // :188-189
      if (hasbuf) {
        double tv = ops.target[1 * nyp + kk];
        yfv = padd(yfv, pmul(buf, make_double2(V0.x - tv, V0.y - tv)));
      }
      fld[6] = yfv;
    }
    // CFL maxima for this plane (check_cfl :211-213)
    if (a.cflbits) {
      double au = act ? pabsmax(padd(U0, U1)) : 0.0;
      double av = act ? pabsmax(V0) : 0.0;
      double aw = act ? pabsmax(padd(W0, W1)) : 0.0;
      if (LIN && act) {
        au = fmax(au, pabsmax(padd(BU0, BU1)));
        av = fmax(av, pabsmax(BV0));
        aw = fmax(aw, pabsmax(padd(BW0, BW1)));
      }
      au = wave_max(au); av = wave_max(av); aw = wave_max(aw);
      if ((tid & 63) == 0) {
        unsigned long long* cb = a.cflbits + 3 * kk;
        atomicMax(cb + 0, (unsigned long long)__double_as_longlong(au));
        atomicMax(cb + 1, (unsigned long long)__double_as_longlong(av));
        atomicMax(cb + 2, (unsigned long long)__double_as_longlong(aw));
      }
    }
    // forward x transforms of the nf fields
    if (act) {
#pragma unroll
      for (int f = 0; f < 8; ++f)
        if (f < nf) lds[(f * RZ + r) * SS + pin] = fld[f];
    }
    __syncthreads();
    fft_run<MC, -1, 12>(lds, SS, nf * RZ, g.px, tw, rl, tid, nthr);
    if (act) {
      // outputs kx = n (and kx = M for an undealiased x grid)
      for (int kq = n; kq < nxh; kq += M) {
        const double2 wk = rootx[kq];
        const double kxv = ops.kx[kq];
        auto X = [&](int f) { return r2c_post_nl<MC>(lds + (f * RZ + r) * SS, M, kq, wk); };
        auto ikxm = [&](double2 v) { return make_double2(-kxv * v.y, kxv * v.x); };
        double2 X0 = X(0), X1 = X(1), X2 = X(2), X3 = X(3), X4 = X(4);
        double2 Au = cadd(X1, ikxm(X0));
        double2 Aw = cadd(X3, ikxm(X2));
        const long ab0 = ((long)((0 * nyp + kk) * 2) * nz2 + zz) * kxp + kq;
        const long ab2 = ((long)((2 * nyp + kk) * 2) * nz2 + zz) * kxp + kq;
        const long bst = (long)nz2 * kxp;
        a.AB[ab0] = Au;
        a.AB[ab0 + bst] = X2;
        a.AB[ab2] = Aw;
        a.AB[ab2 + bst] = X4;
        if (!top) {
          double2 X5 = X(5), X6 = X(6), X7 = X(7);
          const long ab1 = ((long)((1 * nyp + kk) * 2) * nz2 + zz) * kxp + kq;
          a.AB[ab1] = cadd(X6, ikxm(X5));
          a.AB[ab1 + bst] = X7;
        }
      }
    }
    __syncthreads();
    // slide the window (:81, :170-171, :198)
    FU = Fu; FW = Fw; GV = G1;
    U0 = U1; V0 = V1; W0 = W1; BU0 = BU1; BV0 = BV1; BW0 = BW1;
  }
}

// Two rows of 96 pairs keep the roots w_{2M}^n (n <= M) and the wavenumbers in
// LDS tables instead of registers: of the 31 registers that went to scratch,
// whose loads waited behind the prefetch, 5 are left.  A step at 128x129x128
// 858 -> 827 us, 128x200x64 681 -> 665.  Level at one row of 192 pairs (17
// registers in scratch) and two of 72 (13).
__host__ __device__ constexpr bool xpass_tables(int M, int rw) { return rw == 2 && M == 96; }
__host__ __device__ constexpr int xpass_table_cells(int M, int rw, int nxh) {
  return xpass_tables(M, rw) ? M + 1 + (nxh + 1) / 2 : 0;
}

// ---------------------------------------------------------------------------
// Wave-centric x-pass for the compile-time lengths M <= 192.  A wavefront
// owns RW consecutive z-rows and walks a chunk of planes on its own: the
// RW*M physical point pairs of its rows are spread over the lanes (lane l
// holds the pairs v = l + 64q, q < PPL; pair v is point n = v mod M of row
// v / M), and the x transforms of the rows run in the wavefront's private
// LDS slice, ordered with wavefront-scope fences only.  The eight forward
// fields go through the slice in two batches of four per row: {u^2, d/dy
// flux_u, w u, d/dy flux_w} give Au, Bu, Aw, and {w^2, v-interp u, d/dy
// flux_v, v-interp w} give Bw, Av, Bv.  Sequence (f, r) of a batch, field f
// of row r, sits at f*RW + r.  Short rows take RW > 1: one row of 36 pairs
// leaves 28 of 64 lanes idle in every pointwise step, and its 4-sequence
// transform batches give the lanes 24 tasks.  The four wavefronts of a
// workgroup share only the root table.
// ---------------------------------------------------------------------------
//
// With PF the raw rows of the next plane are streamed into a per-wavefront
// LDS buffer by direct global-to-LDS loads (global_load_lds_dwordx4: lane i
// writes cells base + i) as soon as the current rows have been consumed, so
// their latency overlaps a whole plane of work instead of stalling the
// wavefront at the start of every plane.  A raw row takes M + 1 cells rounded
// up to 64 with one row per wavefront or below 64 pairs, otherwise nxh cells:
// the next row follows, so the lanes past a row's end are masked.
//
// What bounds it: LDS round trips and vector issue in turn (M = 144: two
// wavefronts per SIMD, a forward transform phase of 2900 cycles of which
// 1280 issue vector instructions; LDS 48 % busy), so the steps are laid out
// for few waits: lanes without work run along and only their stores are
// masked, which lets every load of a step issue before the first wait, and
// the wait for the next raw rows leaves the stores behind them in flight.
// x-pass at 256x193x192 (M = 192, rows read in place): 796 us with a branch
// per cell and one wavefront per SIMD, 388 now; 32x65x32 16.6 and 15.5.
//
// (bx, by): the workgroup's group of 4*RW z-rows and its plane range
// (blockIdx, or a work-list entry of the batched form)
template <bool LIN, int M, bool PF, bool LES = false, int RW = 1>
__device__ __forceinline__ void xpass_w_body(const XZGeom& g, const double2* __restrict__ tw, const DevOps& ops,
                                             const XPassArgs& a, int bx, int by) {
  extern __shared__ double2 lds[];
  constexpr int SEQ = fft_seq_cells(M), NP = RW * M, PPL = (NP + 63) / 64;
  constexpr int FS = RW * SEQ;                      // cells between the fields of a batch
  // the wavefront index is uniform: as a scalar it keeps the row and plane
  // offsets on the scalar unit
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nz2 = g.nz2, kxp = g.kxpad, nxh = g.nxh;
  // a constant raw-row stride (M + 1 cells rounded up) where it costs no LDS, so that the
  // LDS offsets of the raw rows fold into the reads
  const int rawn = (RW == 1 || M < 64) ? xpass_raw_cells(M + 1) : nxh;
  double2* rl = lds;
  load_tw2<M>(rl, tw + g.px.tw, tid, 256);
  constexpr bool TAB = xpass_tables(M, RW);
  double2* const RT = lds + M;                                    // TAB: roots, then wavenumbers
  double* const KX = reinterpret_cast<double*>(lds + M + M + 1);
  if constexpr (TAB) {
    for (int i = tid; i <= M; i += 256) RT[i] = tw[g.twx + i];
    for (int i = tid; i < nxh; i += 256) KX[i] = ops.kx[i];
  }
  __syncthreads();
  const int zb = (bx * 4 + wv) * RW;  // first z-row of the wavefront
  if (zb >= nz2) return;  // after the only workgroup barrier
  const long rowoff = (long)zb * kxp, prow = (long)zb * g.nx2;
  double2* W = lds + M + xpass_table_cells(M, RW, nxh) + wv * (4 * FS + (PF ? 3 * RW * rawn : 0));
  double2* RAW = W + 4 * FS;
  const double2* rg = tw + g.px.tw;
  const double2* rootx = tw + g.twx;
  const int ny = a.ny, nyp = ny + 1;
  const int ka = a.ka + by * a.chunk;
  const int kb = min(a.kb, ka + a.chunk - 1);
  const bool hasbuf = ops.buffer != nullptr;

  // pair q of the lane: point nq[q] of row rq(q); pin/pout carry the row's
  // sequence offset.  A lane past the last pair works on point 0 of row 0 and
  // its values are not stored: everything but the stores runs without a
  // branch, so that the loads of a step are all issued before the first wait.
  int nq[PPL], pin[PPL], pout[PPL];
  bool vq[PPL];
  double2 wc[TAB ? 1 : PPL];
  auto rq = [&](int q) { return RW == 1 ? 0 : (vq[q] ? (lane + 64 * q) / M : 0); };
#pragma unroll
  for (int q = 0; q < PPL; ++q) {
    const int v = lane + 64 * q;
    vq[q] = 64 * (q + 1) <= NP || v < NP;
    const int vv = vq[q] ? v : 0;
    const int r = RW == 1 ? 0 : vv / M, n = vv - r * M;
    nq[q] = n;
    if (!TAB) wc[TAB ? 0 : q] = cconj(rootx[RW == 1 ? min(v, M) : n]);   // one row: also the root of output column v <= M
    pin[q] = r * SEQ + fft2_in_pos<M>(n);
    pout[q] = r * SEQ + fft2_out_pos<M>(n);
  }

  // raw rows of plane p (1-based) into RAW[c*RW + r][0..nxh) (PF only); every
  // global address is clamped to an element of the row
  auto fetch = [&](int p) {
    if constexpr (PF) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): earlier reads of RAW are done
#pragma unroll
      for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int r = 0; r < RW; ++r) {
          const double2* row = a.Z + ((long)(c * nyp + (p - 1)) * nz2 + r) * kxp + rowoff;
#pragma unroll
          for (int i = 0; i < (M + 64) / 64; ++i) {   // nxh <= M + 1
            if (64 * i >= nxh) break;
            const int idx = min(64 * i + lane, nxh - 1);
            if (RW > 1 && M >= 64 && 64 * i + lane >= nxh) continue;   // the next row's cells follow
            __builtin_amdgcn_global_load_lds((const void*)(row + idx),
                                             (__attribute__((address_space(3))) void*)(RAW + (c * RW + r) * rawn + 64 * i),
                                             16, 0, 0);
          }
        }
      }
    }
  };
  // The raw rows have landed.  Vector memory operations complete in the order
  // they were issued, so the `later` stores issued since the fetch need not
  // have: waiting for them too would add their latency to every plane.  This
  // holds for global and scratch accesses, not for FLAT ones (as_global): no
  // pointer of this body may be generic.
  auto ready = [&](int later) {
    if constexpr (PF) {
      switch (later) {
        case 6: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
        case 12: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
        case 18: asm volatile("s_waitcnt vmcnt(18)" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
      }
      wave_sync();
    }
  };
  // c2r of plane p (1-based) into U, V, Wv at the owned points; the raw rows
  // of plane pnext (0: none) are fetched as soon as those of p are in registers.
  // The half-length packing (c2r_pack_nl) with the cells of both modes clamped
  // into the row and their parts zeroed by selects.
  auto c2r_plane = [&](int p, double2* U, double2* V, double2* Wv, int pnext) {
    constexpr int CB = RW == 1 ? 3 : 1;   // components whose cells are in flight together
#pragma unroll
    for (int c0 = 0; c0 < 3; c0 += CB) {
      double2 ya[CB][PPL], yb[CB][PPL];
#pragma unroll
      for (int c = 0; c < CB; ++c) {
#pragma unroll
        for (int q = 0; q < PPL; ++q) {
          const double2* row = PF ? RAW + ((c0 + c) * RW + rq(q)) * rawn
                                  : a.Z + ((long)((c0 + c) * nyp + (p - 1)) * nz2 + rq(q)) * kxp + rowoff;
          ya[c][q] = row[min(nq[q], nxh - 1)];
          yb[c][q] = row[min(M - nq[q], nxh - 1)];
        }
      }
      if (c0 + CB == 3 && pnext) fetch(pnext);
#pragma unroll
      for (int q = 0; q < PPL; ++q) {
        const int n = nq[q];
        const bool ha = n < nxh, hb = M - n < nxh, im = n != 0;
        const double2 wq = TAB ? cconj(RT[n]) : wc[TAB ? 0 : q];
        double2 z[CB];
#pragma unroll
        for (int c = 0; c < CB; ++c) {
          const double2 A = make_double2(ha ? ya[c][q].x : 0.0, ha && im ? ya[c][q].y : 0.0);
          const double2 B = make_double2(hb ? yb[c][q].x : 0.0, hb && im ? -yb[c][q].y : 0.0);
          z[c] = c2r_combine(A, B, wq);
        }
        if (vq[q]) {
#pragma unroll
          for (int c = 0; c < CB; ++c) W[(c0 + c) * FS + pin[q]] = z[c];
        }
      }
    }
    wave_sync();
    fft2p_wave<M, 1>(W, SEQ, 3 * RW, rl, rg, lane);
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      U[q] = W[0 * FS + pout[q]];
      V[q] = W[1 * FS + pout[q]];
      Wv[q] = W[2 * FS + pout[q]];
    }
    wave_sync();
  };
  // offset of pair q in a physical [nz2][nx2] plane
  auto poff = [&](int q) { return prow + (long)rq(q) * g.nx2 + 2 * nq[q]; };
  auto load_base = [&](int p, double2* U, double2* V, double2* Wv) {
    if (!LIN) return;
    const double* b = a.base;
    const long cs = (long)nyp * nz2 * g.nx2;
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      const long o = (long)(p - 1) * nz2 * g.nx2 + poff(q);
      U[q] = *reinterpret_cast<const double2*>(b + o);
      V[q] = *reinterpret_cast<const double2*>(b + cs + o);
      Wv[q] = *reinterpret_cast<const double2*>(b + 2 * cs + o);
    }
  };
  // Everything the plane loop reads from global memory besides the raw rows
  // is loaded ahead of the wait for those rows: with PF a later vector load
  // would make its consumer wait for the in-flight prefetch as well.
  // The output columns of the rows: output u = lane + 64i is column
  // u mod nxh of row u / nxh.  The columns of the first KP iterations (all of
  // them with 3/2 dealiasing, nxh = 2M/3 + 1) have their root (with one row,
  // that of the pair with the same index) and wavenumber in registers; wider
  // rows load the rest in place.
  constexpr int KQ = (RW * (M + 1) + 63) / 64;              // nxh <= M + 1
  constexpr int KPD = (RW * ((2 * M) / 3 + 1) + 63) / 64;
  constexpr int KP = KPD < KQ ? KPD : KQ;
  constexpr int G0 = RW == 1 && KP > 1 ? 2 : 1;             // columns of the first output group
  const int nout = RW * nxh;
  auto orow = [&](int i) {
    const int u = min(lane + 64 * i, nout - 1);
    int r = 0;
#pragma unroll
    for (int j = 1; j < RW; ++j) r += (u >= j * nxh) ? 1 : 0;
    return r;
  };
  auto ocol = [&](int i) { return min(lane + 64 * i, nout - 1) - orow(i) * nxh; };
  static_assert(RW > 1 || KP <= PPL, "the columns' roots are those of the pairs");
  double2 rxl[RW == 1 || TAB ? 1 : KP];
  double kxl[TAB ? 1 : KP];
  if (!TAB) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int kq = ocol(i);
      if (RW > 1) rxl[RW == 1 || TAB ? 0 : i] = rootx[kq];
      kxl[TAB ? 0 : i] = ops.kx[kq];
    }
  }
  auto root_of = [&](int i, int kq) {
    if (TAB) return RT[kq];
    if (i >= KP) return rootx[kq];
    return RW == 1 ? cconj(wc[!TAB && i < PPL ? i : 0]) : rxl[!TAB && RW > 1 && i < KP ? i : 0];
  };
  auto kx_of = [&](int i, int kq) { return TAB ? KX[kq] : i < KP ? kxl[!TAB && i < KP ? i : 0] : ops.kx[kq]; };
  auto bufv = [&](int q) { return *reinterpret_cast<const double2*>(ops.buffer + poff(q)); };
  // Subgrid stress (LES): tau_ij is added to the flux u_i u_j wherever the
  // flux is formed, so the divergence of the fluxes carries -div(tau) with the
  // same discrete operators.  tau lives at the cell centres yh; at the v-points
  // y(k) tau_12 and tau_23 are interpolated with the iu weights, as u and w are.
  constexpr bool les = LES;
  auto tauv = [&](int c, int kk, int q) {
    return *reinterpret_cast<const double2*>(a.tau + ((long)c * nyp + kk) * nz2 * g.nx2 + poff(q));
  };

  const double2 z2 = make_double2(0.0, 0.0);
  double2 U0[PPL], V0[PPL], W0[PPL], U1[PPL], V1[PPL], W1[PPL];
  double2 BU0[PPL], BV0[PPL], BW0[PPL], BU1[PPL], BV1[PPL], BW1[PPL];
  double2 FU[PPL], FW[PPL], GV[PPL];
#pragma unroll
  for (int q = 0; q < PPL; ++q) {
    U0[q] = V0[q] = W0[q] = U1[q] = V1[q] = W1[q] = z2;
    BU0[q] = BV0[q] = BW0[q] = BU1[q] = BV1[q] = BW1[q] = z2;
  }
  const double half = 0.5, two = 2.0;

  // prologue: planes ka-1 and ka, fluxes at y(ka-1) and yh(ka)
  fetch(ka - 1);
  ready(0);
  c2r_plane(ka - 1, U0, V0, W0, ka);
  load_base(ka - 1, BU0, BV0, BW0);
  load_base(ka, BU1, BV1, BW1);
  ready(0);
  c2r_plane(ka, U1, V1, W1, ka + 1);
#pragma unroll
  for (int q = 0; q < PPL; ++q) {
    if (!LIN) {
      if (ka - 1 == 1) { FU[q] = pmul(V0[q], U0[q]); FW[q] = pmul(V0[q], W0[q]); }   // :53,56
      else {
        FU[q] = pmul(V0[q], psc(half, padd(U0[q], U1[q])));
        FW[q] = pmul(V0[q], psc(half, padd(W0[q], W1[q])));
      }
      double2 t = psc(half, padd(V0[q], V1[q]));
      GV[q] = pmul(t, t);                                                                 // :54-55
    } else {
      if (ka - 1 == 1) {                                                                  // lin :160-170
        FU[q] = padd(pmul(BV0[q], U0[q]), pmul(V0[q], BU0[q]));
        FW[q] = padd(pmul(BV0[q], W0[q]), pmul(V0[q], BW0[q]));
      } else {                                                                            // lin :265-273
        FU[q] = padd(pmul(psc(half, BV0[q]), padd(U0[q], U1[q])), pmul(psc(half, V0[q]), padd(BU0[q], BU1[q])));
        FW[q] = padd(pmul(psc(half, BV0[q]), padd(W0[q], W1[q])), pmul(psc(half, V0[q]), padd(BW0[q], BW1[q])));
      }
      double2 t = psc(half, padd(V0[q], V1[q])), tb = psc(half, padd(BV0[q], BV1[q]));
      GV[q] = pmul(psc(two, t), tb);
    }
    if (les) {
      const int k0 = ka - 2;  // 0-based plane ka-1
      if (ka - 1 != 1) {      // the bottom wall carries no subgrid stress
        const double j1 = ldro(ops.iu, 2 * k0), j2 = ldro(ops.iu, 2 * k0 + 1);
        FU[q] = padd(FU[q], padd(psc(j1, tauv(1, k0, q)), psc(j2, tauv(1, k0 + 1, q))));
        FW[q] = padd(FW[q], padd(psc(j1, tauv(4, k0, q)), psc(j2, tauv(4, k0 + 1, q))));
      }
      GV[q] = padd(GV[q], tauv(3, k0 + 1, q));
    }
    U0[q] = U1[q]; V0[q] = V1[q]; W0[q] = W1[q];
    BU0[q] = BU1[q]; BV0[q] = BV1[q]; BW0[q] = BW1[q];
  }

  // stores of a plane below the top one: two batches of three per 64 columns
  const int nst = 6 * ((nout + 63) / 64);
  int later = 0;   // stores issued since the last fetch, at least
  for (int k = ka; k <= kb; ++k) {
    const bool top = (k == ny);
    const int kk = k - 1;  // 0-based plane index
    const double dh = ldro(ops.dh, kk);
    const double dnk = top ? 0.0 : ldro(ops.dn, kk);
    const double i1 = top ? 0.0 : ldro(ops.iu, 2 * kk), i2 = top ? 0.0 : ldro(ops.iu, 2 * kk + 1);
    double tgu = 0.0, tgv = 0.0, tgw = 0.0;
    if (hasbuf) { tgu = ldro(ops.target, 0 * nyp + kk); tgv = ldro(ops.target, 1 * nyp + kk); tgw = ldro(ops.target, 2 * nyp + kk); }
    load_base(k + 1, BU1, BV1, BW1);
    ready(later);
    later = nst;
    c2r_plane(k + 1, U1, V1, W1, k < kb ? k + 2 : 0);
    double2 Fu[PPL], Fw[PPL], G1[PPL];
    // batch 1: u^2, d/dy flux_u, w u, d/dy flux_w (:138-155)
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      if (!LIN) {
        if (!top) {
          Fu[q] = pmul(V0[q], psc(half, padd(U0[q], U1[q])));
          Fw[q] = pmul(V0[q], psc(half, padd(W0[q], W1[q])));
        } else {
          Fu[q] = pmul(V0[q], U1[q]);
          Fw[q] = pmul(V0[q], W1[q]);
        }
      } else {
        if (!top) {
          Fu[q] = padd(pmul(psc(half, BV0[q]), padd(U0[q], U1[q])), pmul(psc(half, V0[q]), padd(BU0[q], BU1[q])));
          Fw[q] = padd(pmul(psc(half, BV0[q]), padd(W0[q], W1[q])), pmul(psc(half, V0[q]), padd(BW0[q], BW1[q])));
        } else {
          Fu[q] = padd(pmul(BV0[q], U1[q]), pmul(V0[q], BU1[q]));
          Fw[q] = padd(pmul(BV0[q], W1[q]), pmul(V0[q], BW1[q]));
        }
      }
      if (les && !top) {
        Fu[q] = padd(Fu[q], padd(psc(i1, tauv(1, kk, q)), psc(i2, tauv(1, kk + 1, q))));
        Fw[q] = padd(Fw[q], padd(psc(i1, tauv(4, kk, q)), psc(i2, tauv(4, kk + 1, q))));
      }
      double2 yfu = psc(dh, psub(Fu[q], FU[q]));
      double2 yfw = psc(dh, psub(Fw[q], FW[q]));
      if (hasbuf) {
        const double2 bf = bufv(q);
        const double tu = tgu, tw_ = tgw;
        yfu = padd(yfu, pmul(bf, make_double2(U0[q].x - tu, U0[q].y - tu)));
        yfw = padd(yfw, pmul(bf, make_double2(W0[q].x - tw_, W0[q].y - tw_)));
      }
      double2 f0, f2;
      if (!LIN) { f0 = pmul(U0[q], U0[q]); f2 = pmul(W0[q], U0[q]); }
      else { f0 = pmul(psc(two, BU0[q]), U0[q]); f2 = padd(pmul(BW0[q], U0[q]), pmul(W0[q], BU0[q])); }
      if (les) { f0 = padd(f0, tauv(0, kk, q)); f2 = padd(f2, tauv(2, kk, q)); }
      if (vq[q]) {
        W[0 * FS + pin[q]] = f0;
        W[1 * FS + pin[q]] = yfu;
        W[2 * FS + pin[q]] = f2;
        W[3 * FS + pin[q]] = yfw;
      }
    }
    // CFL maxima for this plane (check_cfl :211-213)
    if (a.cflbits) {
      double au = 0.0, av = 0.0, aw = 0.0;
#pragma unroll
      for (int q = 0; q < PPL; ++q) {
        au = fmax(au, pabsmax(padd(U0[q], U1[q])));
        av = fmax(av, pabsmax(V0[q]));
        aw = fmax(aw, pabsmax(padd(W0[q], W1[q])));
        if (LIN) {
          au = fmax(au, pabsmax(padd(BU0[q], BU1[q])));
          av = fmax(av, pabsmax(BV0[q]));
          aw = fmax(aw, pabsmax(padd(BW0[q], BW1[q])));
        }
      }
      au = wave_max(au); av = wave_max(av); aw = wave_max(aw);
      if (lane == 0) {
        unsigned long long* cb = a.cflbits + 3 * kk;
        atomicMax(cb + 0, (unsigned long long)__double_as_longlong(au));
        atomicMax(cb + 1, (unsigned long long)__double_as_longlong(av));
        atomicMax(cb + 2, (unsigned long long)__double_as_longlong(aw));
      }
    }
    wave_sync();
    fft2p_wave<M, -1>(W, SEQ, 4 * RW, rl, rg, lane);
    const long bst = (long)nz2 * kxp;
    const long ab0 = ((long)((0 * nyp + kk) * 2) * nz2) * kxp + rowoff;
    const long ab1 = ((long)((1 * nyp + kk) * 2) * nz2) * kxp + rowoff;
    const long ab2 = ((long)((2 * nyp + kk) * 2) * nz2) * kxp + rowoff;
    // The columns i0 .. i1-1 (x 64) of the first batch: the loads of all of
    // them (in groups, for the registers), then the stores
    auto out1 = [&](auto i0_, auto i1_) {
      constexpr int i0 = decltype(i0_)::value, i1 = decltype(i1_)::value;
      double2 Au[i1 - i0], Bu[i1 - i0], Aw[i1 - i0];
#pragma unroll
      for (int i = i0; i < i1; ++i) {
        const int kq = ocol(i);
        const double2* S = W + orow(i) * SEQ;
        const double2 wk = root_of(i, kq);
        const double kxv = kx_of(i, kq);
        const double2 X0 = r2c_post_nl<M>(S + 0 * FS, M, kq, wk), X1 = r2c_post_nl<M>(S + 1 * FS, M, kq, wk);
        const double2 X2 = r2c_post_nl<M>(S + 2 * FS, M, kq, wk), X3 = r2c_post_nl<M>(S + 3 * FS, M, kq, wk);
        Au[i - i0] = add_ik(X1, kxv, X0);
        Bu[i - i0] = X2;
        Aw[i - i0] = add_ik(X3, kxv, X2);
      }
#pragma unroll
      for (int i = i0; i < i1; ++i) {
        if (lane + 64 * i >= nout) break;
        const long oo = (long)orow(i) * kxp + ocol(i);
        a.AB[ab0 + oo] = Au[i - i0];
        a.AB[ab0 + bst + oo] = Bu[i - i0];
        a.AB[ab2 + oo] = Aw[i - i0];
      }
    };
    out1(std::integral_constant<int, 0>{}, std::integral_constant<int, G0>{});
    if constexpr (KP > G0) out1(std::integral_constant<int, G0>{}, std::integral_constant<int, KP>{});
    if constexpr (KQ > KP) {
      if (64 * KP < nout) out1(std::integral_constant<int, KP>{}, std::integral_constant<int, KQ>{});
    }
    wave_sync();
    // batch 2: w^2 and, below the top plane, the v fluxes (:183-195)
    const int nb2 = top ? 1 : 4;
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      if (!LIN) {
        if (!top) { double2 t = psc(half, padd(V0[q], V1[q])); G1[q] = pmul(t, t); }
        else G1[q] = z2;
      } else {
        if (!top) {
          double2 t = psc(half, padd(V0[q], V1[q])), tb = psc(half, padd(BV0[q], BV1[q]));
          G1[q] = pmul(psc(two, t), tb);
        } else {
          G1[q] = z2;
        }
      }
      if (les && !top) G1[q] = padd(G1[q], tauv(3, kk + 1, q));
      double2 f4 = LIN ? pmul(psc(two, BW0[q]), W0[q]) : pmul(W0[q], W0[q]);
      if (les) f4 = padd(f4, tauv(5, kk, q));
      if (vq[q]) W[0 * FS + pin[q]] = f4;
      if (!top) {
        double2 f5, f7;
        if (!LIN) {
          f5 = pmul(V0[q], padd(psc(i1, U0[q]), psc(i2, U1[q])));
          f7 = pmul(V0[q], padd(psc(i1, W0[q]), psc(i2, W1[q])));
        } else {
          f5 = padd(pmul(BV0[q], padd(psc(i1, U0[q]), psc(i2, U1[q]))),
                    pmul(V0[q], padd(psc(i1, BU0[q]), psc(i2, BU1[q]))));
          f7 = padd(pmul(BV0[q], padd(psc(i1, W0[q]), psc(i2, W1[q]))),
                    pmul(V0[q], padd(psc(i1, BW0[q]), psc(i2, BW1[q]))));
        }
        if (les) {
          f5 = padd(f5, padd(psc(i1, tauv(1, kk, q)), psc(i2, tauv(1, kk + 1, q))));
          f7 = padd(f7, padd(psc(i1, tauv(4, kk, q)), psc(i2, tauv(4, kk + 1, q))));
        }
        double2 yfv = psc(dnk, psub(G1[q], GV[q]));                                    // :188-189
        if (hasbuf) {
          const double tv = tgv;
          yfv = padd(yfv, pmul(bufv(q), make_double2(V0[q].x - tv, V0[q].y - tv)));
        }
        if (vq[q]) {
          W[1 * FS + pin[q]] = f5;
          W[2 * FS + pin[q]] = yfv;
          W[3 * FS + pin[q]] = f7;
        }
      }
    }
    wave_sync();
    fft2p_wave<M, -1>(W, SEQ, nb2 * RW, rl, rg, lane);
    auto out2 = [&](auto i0_, auto i1_) {
      constexpr int i0 = decltype(i0_)::value, i1 = decltype(i1_)::value;
      double2 Bw[i1 - i0], Av[i1 - i0], Bv[i1 - i0];
#pragma unroll
      for (int i = i0; i < i1; ++i) {
        const int kq = ocol(i);
        const double2* S = W + orow(i) * SEQ;
        const double2 wk = root_of(i, kq);
        const double kxv = kx_of(i, kq);
        Bw[i - i0] = r2c_post_nl<M>(S + 0 * FS, M, kq, wk);
        const double2 X5 = r2c_post_nl<M>(S + 1 * FS, M, kq, wk), X6 = r2c_post_nl<M>(S + 2 * FS, M, kq, wk);
        Av[i - i0] = add_ik(X6, kxv, X5);
        Bv[i - i0] = r2c_post_nl<M>(S + 3 * FS, M, kq, wk);   // at the top plane Av and Bv are not stored
      }
#pragma unroll
      for (int i = i0; i < i1; ++i) {
        if (lane + 64 * i >= nout) break;
        const long oo = (long)orow(i) * kxp + ocol(i);
        a.AB[ab2 + bst + oo] = Bw[i - i0];
        if (!top) {
          a.AB[ab1 + oo] = Av[i - i0];
          a.AB[ab1 + bst + oo] = Bv[i - i0];
        }
      }
    };
    out2(std::integral_constant<int, 0>{}, std::integral_constant<int, G0>{});
    if constexpr (KP > G0) out2(std::integral_constant<int, G0>{}, std::integral_constant<int, KP>{});
    if constexpr (KQ > KP) {
      if (64 * KP < nout) out2(std::integral_constant<int, KP>{}, std::integral_constant<int, KQ>{});
    }
    wave_sync();
    // slide the window (:81, :170-171, :198)
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      FU[q] = Fu[q]; FW[q] = Fw[q]; GV[q] = G1[q];
      U0[q] = U1[q]; V0[q] = V1[q]; W0[q] = W1[q];
      BU0[q] = BU1[q]; BV0[q] = BV1[q]; BW0[q] = BW1[q];
    }
  }
}

// Wavefronts per SIMD the registers are held to: two (a few of them go to
// scratch at M = 192 and two rows of 72), but one for the linearized pass of
// 128 and more pairs, whose base flow would go there.  Three at two rows of
// 36 or 48 cost 20 registers of scratch: 337 against 334 ms for 60 steps of
// the 48-member ensemble (with the generic pointers its kernels had then).
template <bool LIN, int M, int RW>
constexpr int xpass_w_waves() { return LIN && RW * M >= 128 ? 1 : 2; }

template <bool LIN, int M, bool PF, bool LES = false, int RW = 1>
__global__ __launch_bounds__(256, (xpass_w_waves<LIN, M, RW>())) void k_xpass_w(XZGeom g, const double2* __restrict__ tw, DevOps ops,
                                                  XPassArgs a) {
  xpass_w_body<LIN, M, PF, LES, RW>(g, tw, ops, a, blockIdx.x, blockIdx.y);
}

// Batched form: workgroup i runs work-list entry it[i] of channel it[i].m.
// The pointers of the entry go to the body as global ones: its counted waits
// (ready) hold for global accesses only, and a FLAT load of a root or a
// twiddle waited for the whole prefetch (60 steps of the 48-member ensemble
// 333 ms with generic pointers, 311 so).
template <bool LIN, int M, bool PF, int RW>
__global__ __launch_bounds__(256, (xpass_w_waves<LIN, M, RW>())) void k_xpass_w_b(const XBatchArgs* __restrict__ args,
                                                    const BatchItem* __restrict__ it) {
  const BatchItem w = it[blockIdx.x];
  XBatchArgs x = args[w.m];
  x.tw = as_global(x.tw);
  DevOps& o = x.ops;
  for (const double** p : {&o.d2h, &o.d2n, &o.dm, &o.dh, &o.dn, &o.hn, &o.iu, &o.dyh, &o.dy, &o.kx, &o.kz, &o.buffer,
                           &o.target, &x.a.base, &x.a.tau})
    *p = as_global(*p);
  x.a.Z = as_global(x.a.Z);
  x.a.AB = as_global(x.a.AB);
  x.a.cflbits = as_global(x.a.cflbits);
  xpass_w_body<LIN, M, PF, false, RW>(x.g, x.tw, x.ops, x.a, w.bx, w.by);
}

using XPassFn = void (*)(XZGeom, const double2*, DevOps, XPassArgs);
using XPassBFn = void (*)(const XBatchArgs*, const BatchItem*);

// Rows per wavefront with a kernel: 1 at every length, 2 for M <= 72 and 96,
// 4 for M <= 24, the last two with the row prefetch only.
static bool xpass_rw_built(int M, int rw, bool pf) {
  return rw == 1 || (pf && ((rw == 2 && (M <= 72 || M == 96)) || (rw == 4 && M <= 24)));
}

// The default.  The pass issues vector instructions most of the time at the
// short lengths (three wavefronts per SIMD at 64x97x64 finish at 43, 54 and 66
// thousand cycles in the order of their age), and the transform tasks of one
// row leave half of the lanes or more idle in every one of them.  A whole step
// with one row and two: 32x129x64 238 and 198 us, 64x97x64 244 and 238,
// 72x81x108 356 and 335, 96x193x96 811 and 739.  Two rows of 96 pairs leave one
// workgroup's registers and LDS twice per compute unit and pay where they
// leave its plane ranges four planes or more: 128x65x64 294 and 301,
// 128x200x64 694 and 665, 128x129x128 912 and 827.  With base-flow loads (lin)
// the registers set the line, 64x65x64 188 and 183, 96x97x96 421 and 426; with
// the stress loads (les), which wait behind the prefetch, one row and its four
// wavefronts per SIMD hide more: 48x65x48 234 and 240, 64x97x64 388 and 406.
int xpass_rows(int M, int nz2, int req, bool pf, bool lin, bool les, int nplanes) {
  auto ok = [&](int r) { return xpass_rw_built(M, r, pf) && nz2 % r == 0; };
  if (req > 0 && ok(req)) return req;
  const bool two = les ? M <= 27 : lin ? M <= 48 : M <= 72 || (M == 96 && (long)nz2 / 8 * nplanes >= 4 * 512);
  return two && ok(2) ? 2 : 1;
}

// LDS of a wavefront x-pass workgroup: the root table and, per wavefront, 4*rw
// sequences and (with the prefetch) 3*rw raw rows (of M + 1 cells rounded up
// to 64 for one row per wavefront and below 64 pairs, of nxh cells otherwise)
size_t xpass_w_lds(int M, int rw, int nxh, bool pf) {
  const int rawn = rw == 1 || M < 64 ? xpass_raw_cells(M + 1) : nxh;
  return sizeof(double2) *
         (M + xpass_table_cells(M, rw, nxh) + 4 * (4 * rw * fft_seq_cells(M) + (pf ? 3 * rw * rawn : 0)));
}

template <int N, bool PF, int RW>
static XPassFn xpass_w_variant(bool les, bool lin) {
  if constexpr (fft2_batched(N)) {
    if (les) return k_xpass_w<false, N, PF, true, RW>;
  }
  return lin ? (XPassFn)k_xpass_w<true, N, PF, false, RW> : (XPassFn)k_xpass_w<false, N, PF, false, RW>;
}

template <int N>
static XPassFn xpass_w_fn(bool les, bool lin, bool pf, int rw) {
  if constexpr (N <= 144) {
    if (pf) {
      if constexpr (N <= 24) {
        if (rw == 4) return xpass_w_variant<N, true, 4>(les, lin);
      }
      if constexpr (N <= 72 || N == 96) {
        if (rw == 2) return xpass_w_variant<N, true, 2>(les, lin);
      }
      return rw == 1 ? xpass_w_variant<N, true, 1>(les, lin) : nullptr;
    }
  }
  return rw == 1 ? xpass_w_variant<N, false, 1>(les, lin) : nullptr;
}

template <int N, int RW>
static XPassBFn xpass_wb_variant(bool lin) {
  constexpr bool pf = N <= 144;
  return lin ? (XPassBFn)k_xpass_w_b<true, N, pf, RW> : (XPassBFn)k_xpass_w_b<false, N, pf, RW>;
}

// Rows per wavefront the batched form is built for: the single one's but two
// rows of 96 pairs, which leave a compute unit one workgroup.
static constexpr bool xpass_wb_built(int M, int rw) {
  return rw == 1 || (rw == 2 && M <= 72) || (rw == 4 && M <= 24);
}
int xpass_batched_rows(int M, int nz2, int req) {
  return xpass_rows(M, nz2, xpass_wb_built(M, req) ? req : 0, M <= 144, false, false, 0);
}

template <int N>
static XPassBFn xpass_wb_fn(bool lin, int rw) {
  if constexpr (xpass_wb_built(N, 4)) {
    if (rw == 4) return xpass_wb_variant<N, 4>(lin);
  }
  if constexpr (xpass_wb_built(N, 2)) {
    if (rw == 2) return xpass_wb_variant<N, 2>(lin);
  }
  return rw == 1 ? xpass_wb_variant<N, 1>(lin) : nullptr;
}

static XPassBFn xpass_wb_pick(int M, bool lin, int rw) {
  XPassBFn fn = nullptr;
#define XPASSB_CASE(N)                                   \
  if constexpr (fft2_batched(N) && N <= 192) fn = xpass_wb_fn<N>(lin, rw);
  FFT_DISPATCH(M, XPASSB_CASE)
#undef XPASSB_CASE
  if (!fn) throw chan_error("batched x-pass: no wavefront kernel for nx2/2 = " + std::to_string(M) + " with " +
                            std::to_string(rw) + " rows per wavefront");
  return fn;
}

// The wavefront x-pass of several channels with the same nx2/2 = M in one
// launch (the batched ensemble); the row prefetch is on wherever the single
// launch uses it (M <= 144).  rw: rows per wavefront (every member's nz2 a
// multiple of it); nxh: the largest nx/2+1 of the members.
bool xpass_batchable(int M) { return fft2_batched(M) && M <= 192; }

void launch_xpass_batched(int M, bool lin, int rw, int nxh, const XBatchArgs* args, const BatchItem* items,
                          int nitems, hipStream_t s) {
  if (nitems <= 0) return;
  if (!xpass_batchable(M)) throw chan_error("batched x-pass: nx2/2 = " + std::to_string(M) + " has no wavefront kernel");
  const XPassBFn fn = xpass_wb_pick(M, lin, rw);
  hipLaunchKernelGGL(fn, dim3(nitems), dim3(256), xpass_w_lds(M, rw, nxh, M <= 144), s, args, items);
  LAUNCH_CHECK("k_xpass_w_b");
}

// Resident workgroups of the batched wavefront x-pass at length M on the
// current device (the plane-range rule of the single launch, over the whole batch).
long xpass_batched_resident(int M, bool lin, int rw, int nxh) {
  const void* fn = (const void*)xpass_wb_pick(M, lin, rw);
  int dev = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
    cus = 256;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, xpass_w_lds(M, rw, nxh, M <= 144)) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  return (long)per_cu * cus;
}

// Planes per workgroup of the wavefront x-pass when no chunk is set: the
// plane-rows of the pass spread evenly over the `res` workgroups resident at
// a time, so that one wave of workgroups with full ranges covers nearly all
// of them and the short last ranges fill the remaining slots; at least two
// planes per range.
static int xpass_chunk_auto(long zw, int np, long res) {
  const long c = (zw * np + res - 1) / res;
  return (int)std::max(2L, std::min<long>(c, std::max(2, np)));
}

void launch_xpass(const XZGeom& g, const double2* tw, const DevOps& ops, const XPassArgs& a0,
                  hipStream_t s) {
  XPassArgs a = a0;
  const int M = g.nx2 / 2;
  if (a.kb < a.ka) return;
  // rows per workgroup: largest divisor of nz2 with rz*M <= maxthr
  const int maxthr = (a.maxthr >= 64 && a.maxthr <= 640) ? a.maxthr : 640;
  int rz = 1;
  for (int d = 1; d <= g.nz2; ++d)
    if (g.nz2 % d == 0 && d * M <= std::max(maxthr, M)) rz = d;
  a.rz = rz;
  int nthr = ((rz * M + 63) / 64) * 64;
  if (nthr > 640) throw chan_error("x-pass: nx2/2 above 640 is not supported");
  const bool ct = fft2_split(M).n1 > 0;
  // staging bound of the runtime-planned in-place FFT: 8*rz sequences of length M
  if (!ct)
    for (int i = 0; i < g.px.nst; ++i) {
      int R = g.px.rad[i];
      long nbf = (long)8 * rz * (M / R);
      if (((nbf + nthr - 1) / nthr) * R > 12) throw chan_error("x-pass FFT staging bound");
    }
  const int nplanes = a.kb - a.ka + 1;
  if (a.tau && !(a.wave && fft2_batched(M) && M <= 192))
    throw chan_error("the subgrid closure needs the wavefront x-pass and nx2/2 one of " + batched_lengths(192));
  if (a.wave && ct && M <= 192) {
    const bool pf = a.prefetch && M <= 144;
    if (a.tau && a.base) throw chan_error("the subgrid closure is not defined for the linearized pass");
    const int rw = xpass_rows(M, g.nz2, a.rows, pf, a.base != nullptr, a.tau != nullptr, nplanes);
    const size_t ldw = xpass_w_lds(M, rw, g.nxh, pf);
    XPassFn fn = nullptr;
#define XPASSW_CASE(N)                                                                  \
  if constexpr (N > 0 && N <= 192) fn = xpass_w_fn<N>(a.tau != nullptr, a.base != nullptr, pf, rw);
    FFT_DISPATCH(M, XPASSW_CASE)
#undef XPASSW_CASE
    if (!fn) throw chan_error("x-pass: no wavefront kernel for this length");
    const long zw = (g.nz2 / rw + 3) / 4;
    if (a.chunk <= 0) {
      // resident workgroups of this kernel on the current device
      int dev = 0, cus = 0;
      if (hipGetDevice(&dev) != hipSuccess ||
          hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
      int per_cu = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, ldw) != hipSuccess || per_cu < 1) per_cu = 1;
      a.chunk = xpass_chunk_auto(zw, nplanes, (long)per_cu * cus);
    }
    const int nch = (nplanes + a.chunk - 1) / a.chunk;
    hipLaunchKernelGGL(fn, dim3((unsigned)zw, nch), dim3(256), ldw, s, g, tw, ops, a);
    LAUNCH_CHECK("k_xpass_w");
    return;
  }
  if (a.chunk <= 0) a.chunk = 6;
  const int nch = (nplanes + a.chunk - 1) / a.chunk;
  dim3 grid(g.nz2 / rz, nch);
  size_t lds = sizeof(double2) * (8 * rz * fft_seq_cells(M) + (ct ? M : 0));
#define XPASS_CASE(N)                                                                 \
  if (a.base) hipLaunchKernelGGL((k_xpass<true, N>), grid, dim3(nthr), lds, s, g, tw, ops, a); \
  else hipLaunchKernelGGL((k_xpass<false, N>), grid, dim3(nthr), lds, s, g, tw, ops, a)
  FFT_DISPATCH(M, XPASS_CASE)
#undef XPASS_CASE
  LAUNCH_CHECK("k_xpass");
}
