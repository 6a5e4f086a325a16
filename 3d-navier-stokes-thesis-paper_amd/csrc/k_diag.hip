// Diagnostics on the device: the l2 deviation from the laminar profile
// (l2_norm, PFC/read_write.f90:1432-1462), the per-mode kinetic energy
// (PFC/pass2.f90:113-118) and the per-plane velocity moments of
// compute_velocity_moments (PFC/stats.f90:423-440) for one field.
#include "chan_internal.h"

// Sum over the workgroup (256 threads); every thread gets the total.
__device__ __forceinline__ double block_sum(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) t += red[i];
  return t;
}

// One workgroup per plane j of one component: part[j] = dy(j) * sum (u - lam(j))^2
// over the nx2 x nz2 points of the plane.
__global__ __launch_bounds__(256) void k_l2_planes(const double* __restrict__ phys, long ps, const double* __restrict__ lam,
                                                   const double* __restrict__ dy, double* __restrict__ part) {
  __shared__ double red[4];
  const int j = blockIdx.x;
  const double* p = phys + (long)j * ps;
  const double l = lam ? lam[j] : 0.0;
  double s = 0.0;
  for (long i = threadIdx.x; i < ps; i += blockDim.x) {
    const double d = p[i] - l;
    s += d * d;
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) part[j] = s * dy[j];
}

// The same parts on a grid dealiased in x and z, without a transform: by
// Parseval the sum over the points of the padded inverse transform is nx2 nz2
// times the sum of the squared coefficients, each kx > 0 mode twice.  The
// halved Nyquist modes (the last kx column, and kz = nz/2 split over both
// signs) count 1/4 of that per halving and the split twice; of the kx = 0
// column the real inverse transform keeps the Hermitian part.  Workgroup
// (b, p) sums the b-th share of the modes of plane p = c (ny+1) + j.
//
// Bounded by reading the velocity once: 480 us for the three components at
// 192x129x192 through z-inverse, x c2r (288x288 points a plane) and k_l2_planes.
#define L2_SHARES 4
__global__ __launch_bounds__(256) void k_l2_modes(const double2* __restrict__ vel, int nxh, int nz, int nyp,
                                                  double npts, const double* __restrict__ lam,
                                                  const double* __restrict__ dy, double* __restrict__ part) {
  __shared__ double red[4];
  const int p = blockIdx.y, c = p / nyp, j = p - c * nyp, nm = nxh * nz, h = nz / 2;
  const double2* u = vel + (long)p * nm;
  const int per = (nm + L2_SHARES - 1) / L2_SHARES, m0 = blockIdx.x * per, m1 = min(nm, m0 + per);
  double s = 0.0;
  constexpr int IN = 4;   // loads in flight
  for (int mb = m0 + (int)threadIdx.x; mb < m1; mb += IN * 256) {
    double2 v[IN];
#pragma unroll
    for (int i = 0; i < IN; ++i) v[i] = u[min(mb + 256 * i, nm - 1)];
#pragma unroll
    for (int i = 0; i < IN; ++i) {
      const int m = mb + 256 * i;
      if (m >= m1) break;
      const int ix = m / nz, iz = m - ix * nz;
      const double wz = iz == h ? 0.5 : 1.0;
      double2 a = v[i];
      double wx = ix == nxh - 1 ? 0.5 : 2.0;
      if (ix == 0) {
        wx = 1.0;
        if (iz != h) {
          const double2 b = u[iz == 0 ? 0 : nz - iz];   // mode -kz
          a = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
          if (iz == 0 && c == 0) a.x -= lam[j];
        }
      }
      s += wx * wz * (a.x * a.x + a.y * a.y);
    }
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) part[p * L2_SHARES + blockIdx.x] = s * npts * dy[j];
}

// l2 = sqrt(sum of the n plane parts / (nx2 nz2) / 2); drag = d_um_dy(1) - d_um_dy(ny).
__global__ __launch_bounds__(256) void k_l2_final(const double* __restrict__ part, int n, double npts,
                                                  const double* __restrict__ dudy, int ny, double* __restrict__ out) {
  __shared__ double red[4];
  double t = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) t += part[i];
  t = block_sum(t, red);
  if (threadIdx.x != 0) return;
  out[0] = sqrt(t / npts / 2.0);
  out[1] = dudy[0] - dudy[ny - 1];
}

// sum over j of Re u(0,0)(j) dyh(j), one wavefront
__global__ __launch_bounds__(64) void k_mass_flux(const double2* __restrict__ vel, long nm, int nyp,
                                                  const double* __restrict__ dyh, double* __restrict__ out) {
  double t = 0.0;
  for (int j = threadIdx.x; j < nyp; j += 64) t += vel[j * nm].x * dyh[j];
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  if (threadIdx.x == 0) out[0] = t;
}

// KE of every mode: int_y(|u|^2 + |w|^2 + |v at yh|^2, dyh); written as
// ke(x, z) with x fastest.  A workgroup takes 32 modes (512-byte row pieces)
// in 16 shares of the planes, which are summed in LDS in their order: one
// thread per mode walked all planes in 73 workgroups at 192x129x192, 83 us
// for 116 MB.
#define KE_MODES 32
#define KE_SHARES 16
__global__ __launch_bounds__(KE_MODES * KE_SHARES) void k_mode_energy(DevOps ops, int ny, int nxh, int nz,
                                                                      const double2* __restrict__ vel,
                                                                      double* __restrict__ ke) {
  __shared__ double sum[KE_SHARES][KE_MODES];
  const long nm = (long)nxh * nz;
  const int l = threadIdx.x % KE_MODES, sh = threadIdx.x / KE_MODES;
  const long mg = (long)blockIdx.x * KE_MODES + l, m = mg < nm ? mg : nm - 1;
  const int nyp = ny + 1, per = (nyp + KE_SHARES - 1) / KE_SHARES;
  const int j0 = sh * per, j1 = min(nyp, j0 + per);
  auto at = [&](int c, int j) { return vel[((long)c * nyp + j) * nm + m]; };
  auto a2 = [](double2 v) { return v.x * v.x + v.y * v.y; };
  double s = 0.0;
  if (j0 < j1) {
    double2 vp = at(1, j0 > 0 ? j0 - 1 : 0);
#pragma unroll 4
    for (int j = j0; j < j1; ++j) {
      const double2 u = at(0, j), w = at(2, j), v = at(1, j < ny ? j : ny - 1);
      // v at yh: the mean of the two faces, at the walls the face itself
      const double2 vc = (j == 0 || j == ny) ? v : make_double2(0.5 * (v.x + vp.x), 0.5 * (v.y + vp.y));
      s += (a2(u) + a2(w) + a2(vc)) * ops.dyh[j];
      vp = v;
    }
  }
  sum[sh][l] = s;
  __syncthreads();
  if (sh != 0 || mg >= nm) return;
  for (int i = 1; i < KE_SHARES; ++i) s += sum[i][l];
  const int ix = (int)(m / nz), iz = (int)(m - (long)ix * nz);
  ke[(long)iz * nxh + ix] = s;
}

// x-inverse of `rows` z-rows at a time of the three components of one plane,
// and the sums over its points of the deviations d from the plane's mean coefficient,
// their powers d^2, d^3, d^4 and products with v's: part[plane][block][15]
// (k_moments_final).  Fused, the points stay in LDS: written out and read by
// one workgroup per plane they took 58 + 168 us at 192x129x192.  A workgroup
// takes several row groups, for its 15 sums over the lanes (180 LDS
// permutes a wavefront) are a quarter of its time with one: 78 us, 65 with four.
template <int NC>
__global__ __launch_bounds__(512) void k_xmoments(XZGeom g, const double2* __restrict__ tw,
                                                  const double2* __restrict__ Z, long z_ps, int nyp, int rows,
                                                  const double2* __restrict__ vel, long nm, double* __restrict__ part) {
  extern __shared__ double2 lds[];
  __shared__ double red[8][15];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int M = NC > 0 ? NC : g.nx2 / 2, ss = fft_seq_cells(M);
  const int j = blockIdx.y;
  const double2* rootx = tw + g.twx;
  double2* rl = lds + 3 * rows * ss;
  load_tw2<NC>(rl, tw + g.px.tw, tid, nthr);
  double mean[3], acc[15];
#pragma unroll
  for (int c = 0; c < 3; ++c) mean[c] = vel[((long)c * nyp + j) * nm].x;
#pragma unroll
  for (int k = 0; k < 15; ++k) acc[k] = 0.0;
  for (int z0 = blockIdx.x * rows; z0 < g.nz2; z0 += gridDim.x * rows) {
    // the cells of up to five points per thread (moments_rows) are in flight
    // together, clamped into their row and zeroed by selects (c2r_pack)
    constexpr int IT = 5;
    for (int e0 = tid; e0 < 3 * rows * M; e0 += IT * nthr) {
      double2 ya[IT], yb[IT], wc[IT];
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const int e = min(e0 + i * nthr, 3 * rows * M - 1);
        const int q = e / M, n = e - q * M, c = q / rows, r = q - c * rows;
        const double2* row = Z + ((long)c * nyp + j) * z_ps + (long)(z0 + r) * g.kxpad;
        ya[i] = row[min(n, g.nxh - 1)];
        yb[i] = row[min(M - n, g.nxh - 1)];
        wc[i] = cconj(rootx[n]);
      }
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const int e = e0 + i * nthr;
        if (e >= 3 * rows * M) break;
        const int q = e / M, n = e - q * M;
        const bool ha = n < g.nxh, hb = M - n < g.nxh;
        const double2 a = make_double2(ha ? ya[i].x : 0.0, ha && n ? ya[i].y : 0.0);
        const double2 b = make_double2(hb ? yb[i].x : 0.0, hb && n ? -yb[i].y : 0.0);
        lds[q * ss + fft_in_pos<NC>(n)] = c2r_combine(a, b, wc[i]);
      }
    }
    __syncthreads();
    fft_run<NC, 1, FFT_MAXV>(lds, ss, 3 * rows, g.px, tw, rl, tid, nthr);
    for (int e = tid; e < rows * M; e += nthr) {
      const int r = e / M, n = e - r * M;
      double2 u[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) u[c] = lds[(c * rows + r) * ss + fft_out_pos<NC>(n)];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const double dv = (i ? u[1].y : u[1].x) - mean[1];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const double d = (i ? u[c].y : u[c].x) - mean[c], d2 = d * d;
          acc[c] += d;
          acc[3 + c] += d2;
          acc[6 + c] += d2 * d;
          acc[9 + c] += d2 * d2;
          acc[12 + c] += d * dv;
        }
      }
    }
    __syncthreads();
  }
  const int w = tid >> 6, nw = nthr >> 6;
#pragma unroll
  for (int k = 0; k < 15; ++k) {
    double v = acc[k];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((tid & 63) == 0) red[w][k] = v;
  }
  __syncthreads();
  if (tid < 15) {
    double t = red[0][tid];
    for (int i = 1; i < nw; ++i) t += red[i][tid];
    part[((long)j * gridDim.x + blockIdx.x) * 15 + tid] = t;
  }
}

// Mean, 2nd/3rd/4th central moments of u, v, w and <u_i' v'> of plane
// blockIdx.x from its partial sums: out(ny+1, 15) with the plane fastest.
// The mean coefficient differs from the mean of the points by round-off,
// which the sum of the deviations carries (and any NaN with it).
__global__ __launch_bounds__(64) void k_moments_final(const double* __restrict__ part, int nb, double sc,
                                                      const double2* __restrict__ vel, long nm, int nyp,
                                                      double* __restrict__ out) {
  const int j = blockIdx.x, k = threadIdx.x;
  if (k >= 15) return;
  double t = 0.0;
#pragma unroll 8
  for (int b = 0; b < nb; ++b) t += part[((long)j * nb + b) * 15 + k];
  t *= sc;
  if (k < 3) t += vel[((long)k * nyp + j) * nm].x;
  out[(long)k * nyp + j] = t;
}

// The same from the points in memory, one workgroup per plane: for rows too
// long for three of them in LDS (nx/2 above 2048) and for many short ones
// (plane_moments_fused).
__global__ __launch_bounds__(256) void k_plane_moments(const double* __restrict__ phys, long ps, long cs, int nyp,
                                                       double* __restrict__ out) {
  __shared__ double red[4];
  const int j = blockIdx.x;
  const double sc = 1.0 / (double)ps;
  const double* u[3] = {phys + (long)j * ps, phys + cs + (long)j * ps, phys + 2 * cs + (long)j * ps};
  double m[3];
  for (int c = 0; c < 3; ++c) {
    double s = 0.0;
    for (long i = threadIdx.x; i < ps; i += blockDim.x) s += u[c][i];
    m[c] = sc * block_sum(s, red);
  }
  double acc[12];
  for (int k = 0; k < 12; ++k) acc[k] = 0.0;
  for (long i = threadIdx.x; i < ps; i += blockDim.x) {
    const double dv = u[1][i] - m[1];
    for (int c = 0; c < 3; ++c) {
      const double d = u[c][i] - m[c], d2 = d * d;
      acc[c] += d2;
      acc[3 + c] += d2 * d;
      acc[6 + c] += d2 * d2;
      acc[9 + c] += d * dv;
    }
  }
  for (int k = 0; k < 12; ++k) {
    const double t = sc * block_sum(acc[k], red);
    if (threadIdx.x == 0) out[(long)(3 + k) * nyp + j] = t;
  }
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) out[(long)c * nyp + j] = m[c];
}

void launch_l2_planes(const double* phys, long ps, int nplanes, const double* lam, const double* dy, double* part,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_l2_planes, dim3(nplanes), dim3(256), 0, s, phys, ps, lam, dy, part);
  LAUNCH_CHECK("k_l2_planes");
}

// The parts of k_l2_modes: L2_SHARES per plane
int l2_modes_parts(int nyp) { return 3 * nyp * L2_SHARES; }
void launch_l2_modes(const XZGeom& g, const double2* vel, int nyp, const double* lam, const double* dy, double* part,
                     hipStream_t s) {
  if (!(g.nx2 > g.nx && g.nz2 > g.nz)) throw chan_error("k_l2_modes: the grid is not dealiased");
  hipLaunchKernelGGL(k_l2_modes, dim3(L2_SHARES, 3 * nyp), dim3(256), 0, s, vel, g.nxh, g.nz, nyp,
                     (double)g.nx2 * g.nz2, lam, dy, part);
  LAUNCH_CHECK("k_l2_modes");
}

void launch_l2_final(const double* part, int n, double npts, const double* dudy, int ny, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_l2_final, dim3(1), dim3(256), 0, s, part, n, npts, dudy, ny, out);
  LAUNCH_CHECK("k_l2_final");
}

void launch_mass_flux(const double2* vel, long nm, int nyp, const double* dyh, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_mass_flux, dim3(1), dim3(64), 0, s, vel, nm, nyp, dyh, out);
  LAUNCH_CHECK("k_mass_flux");
}

void launch_mode_energy(const DevOps& ops, int ny, int nxh, int nz, const double2* vel, double* ke, hipStream_t s) {
  const long nm = (long)nxh * nz;
  hipLaunchKernelGGL(k_mode_energy, dim3((unsigned)((nm + KE_MODES - 1) / KE_MODES)), dim3(KE_MODES * KE_SHARES), 0, s,
                     ops, ny, nxh, nz, vel, ke);
  LAUNCH_CHECK("k_mode_energy");
}

// z-rows per workgroup of the moments: the largest divisor of nz whose rows
// fit 768 points per component (three points per thread and component with
// the compile-time lengths, at most 170 points with the runtime-planned
// transform, whose staging is bounded).
static int moments_rows(const XZGeom& g) {
  const int M = g.nx2 / 2, cap = fft2_split(M).n1 > 0 ? 768 : 170;
  int best = 1;
  for (int d = 1; d <= g.nz2; ++d)
    if (g.nz2 % d == 0 && d * M <= cap) best = d;
  return best;
}
// Rows below 16 pairs take the runtime-planned transform, whose workgroups run
// one to a compute unit: up to one round of them the fused form is 7 to 30 %
// ahead, from the second on the points in memory are.  A call at nx = 16: 31.2 us
// fused and 34.8 through memory at 66 planes of 32 rows (132 workgroups), 38.6 and
// 34.9 at 130 (260), 68.2 and 57.4 at 501 (1002).
bool plane_moments_fused(const XZGeom& g, int nyp) {
  const int M = g.nx2 / 2;
  return M <= 2048 && (M >= 16 || (long)nyp * (g.nz2 / moments_rows(g)) <= 256);
}
// Workgroups per plane: about a thousand in all, each with the same number of row groups but the last
static int moments_blocks(const XZGeom& g, int nyp) {
  const int ng = g.nz2 / moments_rows(g), want = std::min(ng, std::max(1, 1024 / nyp)), per = (ng + want - 1) / want;
  return (ng + per - 1) / per;
}
long plane_moments_part(const XZGeom& g, int nyp) { return (long)nyp * moments_blocks(g, nyp) * 15; }
void launch_plane_moments_points(const double* phys, long ps, long cs, int nyp, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_plane_moments, dim3(nyp), dim3(256), 0, s, phys, ps, cs, nyp, out);
  LAUNCH_CHECK("k_plane_moments");
}

// Z: the z-inverse rows of the 3 nyp planes; part: plane_moments_part doubles
void launch_plane_moments(const XZGeom& g, const double2* tw, const double2* Z, long z_ps, int nyp, const double2* vel,
                          double* part, double* out, hipStream_t s) {
  const int M = g.nx2 / 2, rows = moments_rows(g), nb = moments_blocks(g, nyp);
  const bool ct = fft2_split(M).n1 > 0;
  const int nthr = std::min(512, std::max(64, ((3 * rows * M + 63) / 64) * 64));
  if (!ct) check_stage_fit(g.px, 3 * rows, nthr);
  const size_t lds = sizeof(double2) * (3 * rows * fft_seq_cells(M) + (ct ? M : 0));
  const long nm = (long)g.nxh * g.nz;
#define XMOM_CASE(N)                                                                                             \
  hipLaunchKernelGGL(k_xmoments<N>, dim3(nb, nyp), dim3(nthr), lds, s, g, tw, Z, z_ps, nyp, rows, vel, nm, part)
  FFT_DISPATCH(M, XMOM_CASE)
#undef XMOM_CASE
  LAUNCH_CHECK("k_xmoments");
  hipLaunchKernelGGL(k_moments_final, dim3(nyp), dim3(64), 0, s, part, nb, 1.0 / ((double)g.nx2 * g.nz2), vel, nm, nyp,
                     out);
  LAUNCH_CHECK("k_moments_final");
}

// Spectral field of the VTK output: u and w at plane j, v at yh(j) as
// half*(v(j-1) + v(j)), v(1) at the bottom and v(ny) at the top plane
// (PFC/read_write.f90:418-432, yskip = 1).
__global__ __launch_bounds__(256) void k_vtk_field(int ny, long nm, const double2* __restrict__ vel,
                                                   double2* __restrict__ out) {
  const int nyp = ny + 1;
  const long tot = 3L * nyp * nm;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    const long m = e % nm, t = e / nm;
    const int j = (int)(t % nyp), c = (int)(t / nyp);
    double2 v;
    if (c != 1) v = vel[e];
    else if (j == 0) v = vel[(1L * nyp + 0) * nm + m];
    else if (j == ny) v = vel[(1L * nyp + ny - 1) * nm + m];
    else {
      const double2 a = vel[(1L * nyp + j - 1) * nm + m], b = vel[(1L * nyp + j) * nm + m];
      v = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y + b.y));
    }
    out[e] = v;
  }
}

void launch_vtk_field(int ny, long nm, const double2* vel, double2* out, hipStream_t s) {
  const long tot = 3L * (ny + 1) * nm;
  const unsigned blocks = (unsigned)std::min<long>((tot + 255) / 256, 8192);
  hipLaunchKernelGGL(k_vtk_field, dim3(blocks), dim3(256), 0, s, ny, nm, vel, out);
  LAUNCH_CHECK("k_vtk_field");
}
