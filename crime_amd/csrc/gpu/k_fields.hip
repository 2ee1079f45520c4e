// Field stage of the GetHI density-to-sky path on gfx950: create_d_and_vr_fields
// (src/fourier.c:234-305, 375-438) as three HBM passes over one complex N^3 grid.
//
// delta and the velocity potential phi are both real, so the two inverse real FFTs of the
// reference (fourier.c:391-392) are done as ONE complex inverse FFT of
//     F(k) = delta_k + i phi_k,   phi_k = delta_k f0 H0 / k^2            (fourier.c:297-298)
// over the Hermitian completion of the half spectrum: the output is delta in the real part and phi
// in the imaginary part of each cell.  Bytes moved equal those of two r2c-layout transforms, the
// map stage then reads (delta, phi) of a cell in one 8-byte load.  The kx = 0 and kx = N/2 planes,
// which the reference fills without Hermitian symmetry (fourier.c:275-299), enter through their
// Hermitian part (X(k) + X*(-k))/2, which is what a c2r transform uses of them.
//
//   pass 1  k_fill_z : generate F on the fly (P(k) amplitude x unit mode) and transform along kz
//   pass 2  k_fft_y  : transform along ky
//   pass 3  k_fft_x  : transform along kx (contiguous), scale by (sqrt(2 pi)/L)^3 (fourier.c:403),
//                      FP64 partial sums of delta and delta^2 (compute_sigma_dens, fourier.c:24-76)
//   k_sigma_finalize : fixed-order FP64 reduction of the partials -> sigma^2, <delta>, and the largest
//                      |phi| of the grid (bounds the map stage's velocities)
#include "gh_kernels.hpp"

namespace crime {

// ---------------------------------------------------------------------------------------------
// mode fill
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ double pk_linear0(const FillParams &f, double lgk)
{
#pragma clang fp contract(off)
  // src/cosmo.c:153-170; the last half-open bin uses the k^-3 tail instead of reading past the table
  int ik = (int)((lgk - f.logkmin) * f.idlogk);
  if (ik < 0) return f.pk[0] * pow(10.0, f.n_s * (lgk - f.logkmin));
  if (ik < f.numk - 1) return f.pk[ik] + (lgk - f.logk[ik]) * (f.pk[ik + 1] - f.pk[ik]) * f.idlogk;
  return f.pk[f.numk - 1] * pow(10.0, -3 * (lgk - f.logkmax));
}

// Philox words of half-spectrum mode idx -> the two uniforms (53-bit) of rng_delta_gauss
__device__ __forceinline__ void mode_uniforms(const FillParams &f, size_t idx, double &u1, double &u2)
{
  u32x4 c;
  c.v[0] = (uint32_t)idx;
  c.v[1] = (uint32_t)(idx >> 32);
  c.v[2] = 0;
  c.v[3] = 0;
  u32x4 r = philox4x32_10(c, f.seed, PHILOX_KEY1);
  u1 = u53(r.v[0], r.v[1]);
  u2 = u53(r.v[2], r.v[3]);
}

// Unit-variance complex mode at half-spectrum position (kx in [0,N/2], ky, kz):
// rng_delta_gauss (src/common.c:154-164), phase 2 pi u1 and modulus sqrt(-ln(1-u2)).  FP64 grids
// evaluate it in FP64; FP32 grids evaluate the logarithm, root and sin/cos in FP32 from the exact
// FP64 value of 1-u2 (relative error ~1e-7 per mode, the precision the mode is stored in).
template <typename T, int N>
__device__ __forceinline__ cx<T> unit_mode(const FillParams &f, int kx, int ky, int kz)
{
  size_t idx = (size_t)kx + (size_t)(N / 2 + 1) * ((size_t)ky + (size_t)N * (size_t)kz);
  if (f.mode_source == 1) return {(T)f.unit_modes[2 * idx], (T)f.unit_modes[2 * idx + 1]};
  double u1, u2;
  mode_uniforms(f, idx, u1, u2);
  if constexpr (sizeof(T) == 8) {
    double mod = sqrt(-log(1.0 - u2));
    double s, co;
    sincos(2.0 * M_PI * u1, &s, &co);
    return {mod * co, mod * s};
  }
  else {
    float mod = sqrtf(-logf((float)(1.0 - u2)));
    float s, co;
    sincospif(2.0f * (float)u1, &s, &co);
    return {mod * co, mod * s};
  }
}

// Amplitude per k^2 = m dk^2: A = sqrt(P(k)/dk^3 [e^{-r_s^2 k^2}]) (fourier.c:292-295) and, for
// FP64 grids, also A psi with the velocity-potential factor psi = phi_scale f0 H0 / k^2
// (fourier.c:298).  FP32 grids keep A alone (4 bytes per entry, 3 MB at N=1024, L2-sized) and form
// psi = psi_c / m in registers.  Built once per handle.
template <typename T>
__global__ __launch_bounds__(256) void k_amp_table(FillParams f, AmpEntry<T> *__restrict__ tab, int mmax)
{
  int m = blockIdx.x * 256 + threadIdx.x;
  if (m > mmax) return;
  double amp = 0, psi = 0;
  if (m > 0) {
    double k2 = (double)m * (f.dk * f.dk);
    double sigma2 = pk_linear0(f, 0.5 * log10(k2)) * f.idk3;
    if (f.do_smoothing) sigma2 *= exp(-f.r2_smooth * k2);
    amp = sqrt(sigma2);
    psi = f.phi_scale * (f.f0h0 / k2);
  }
  if constexpr (sizeof(T) == 8) tab[m] = {amp, amp * psi};
  else tab[m] = (float)amp;
}

// (A, A psi) of mode (kx, ky, kz): a function of |k|^2 only, so kz and N - kz share it
template <typename T, int N>
__device__ __forceinline__ cx<T> mode_amp(const FillParams &f, const AmpEntry<T> *__restrict__ amp, int kx, int ky,
                                          int kz)
{
  constexpr int n = N, h = N / 2;
  // |k| components with the reference's +Nyquist convention (fourier.c:264-283); only squares matter
  int ax = kx <= h ? kx : n - kx;
  int ay = ky <= h ? ky : n - ky;
  int az = kz <= h ? kz : n - kz;
  int m2 = ax * ax + ay * ay + az * az;
  cx<T> ab;
  if constexpr (sizeof(T) == 8) ab = amp[m2];
  else {
    // psi = psi_c / m2 through the hardware reciprocal (1 ulp): FP32 fields carry ~1e-7 relative error
    // anyway, and a correctly rounded division costs ten instructions per element
    float a = amp[m2];
    ab = {a, a * ((float)f.psi_c * __builtin_amdgcn_rcpf((float)m2))};
  }
  return ab;
}

// F = delta + i phi_scale phi at full-grid position (kx, ky, kz), kx in [0, N), from the amplitude pair
// ab = mode_amp(kx, ky, kz) and the unit-variance mode g.  The products are written as fused operations of one order:
// a mode and its mirror (g conjugate) round alike.
template <typename T>
__device__ __forceinline__ cx<T> fill_element(const FillParams &f, cx<T> ab, cx<T> g, int kx, int ky, int kz)
{
  if ((kx | ky | kz) == 0) return {(T)0, (T)0};
  if (f.vmode == 0) {
    // delta = A g, phi_scale phi = A psi g; F = delta + i phi_scale phi = A g (1 + i psi)
    return {fma(ab.x, g.x, -(ab.y * g.y)), fma(ab.y, g.x, ab.x * g.y)};
  }
  // spectral velocities: with A psi = A phi_scale f0 H0 / k^2 and S_j = sin(k_j dx)/dx,
  //   grid 0: delta + i phi_scale vx = A g + i (i S_x A psi g) = (A - S_x A psi) g
  //   grid 1: phi_scale (vy + i vz)  = i S_y A psi g - S_z A psi g = A psi (-S_z + i S_y) g
  // S_j is odd in k_j, so each v_j(k) is Hermitian wherever delta_k is (the kx = 0, N/2 planes included).
  if (f.comp == 0) {
    const T c = fma(-(T)f.sin_dx[kx], ab.y, ab.x);
    return {c * g.x, c * g.y};
  }
  const cx<T> c = {-(T)f.sin_dx[kz] * ab.y, (T)f.sin_dx[ky] * ab.y};
  return {fma(c.x, g.x, -(c.y * g.y)), fma(c.x, g.y, c.y * g.x)};
}

// ---------------------------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------------------------
// A workgroup holds TX columns (kx, ky), 0 <= kx < N/2, and their mirrors (N - kx, N - ky): F there is made of the
// conjugates of the same modes, so each mode is drawn once.  The draw (ten Philox rounds, a logarithm, a root, a
// sine and cosine: some 300 instructions) bounds the pass up to 512^3 (474 us, 697 with a draw for each element); above,
// the amplitude gathers and writes a plane apart weigh as much (1024^3 5.6 ms, 6.85).  Column kx = 0 has kx = N/2 of the same ky in its
// mirror's place; the two are drawn after the others by all threads, two modes to an element.
template <typename T, int N, int V>
__global__ __launch_bounds__((FillCfg<T, N, V>::NTG)) void k_fill_z(cx<T> *__restrict__ F, FillParams f,
                                                                 const cx<T> *__restrict__ tw)
{
  using C = FillCfg<T, N, V>;
  constexpr int TX = C::TX / 2, NX = N / 2 / TX, h = N / 2;
  __shared__ cx<T> lds[N * C::TX];
  stamp(f.stamp, STAMP_FILL);
  // neighbouring tiles on one XCD: they share lines of 128 bytes, which leave its L2 whole
  const int tile = xcd_swizzle((int)blockIdx.x, NX * N);
  const int x0 = tile % NX * TX, ky = tile / NX, my = (N - ky) % N;
  const size_t n2 = (size_t)N * N;
  // the generator is too large to unroll into the register tile: stage the modes in LDS first
  const AmpEntry<T> *amp = (const AmpEntry<T> *)f.amp;
  {
    const int q = threadIdx.x % TX, kx = x0 + q;
    // kz = e and N - e, of the column and its mirror, in one step: one read of their shared amplitude (a scattered
    // gather, a cache line per lane) for four elements
    for (int e = threadIdx.x / TX; e <= h; e += C::NTG / TX) {
      if (kx == 0) continue;
      const cx<T> ab = mode_amp<T, N>(f, amp, kx, ky, e);
      const int m = (N - e) % N;
      const cx<T> g = unit_mode<T, N>(f, kx, ky, e);
      lds[e * C::TX + q] = fill_element<T>(f, ab, g, kx, ky, e);
      lds[m * C::TX + TX + q] = fill_element<T>(f, ab, {g.x, -g.y}, N - kx, my, m);
      if (e == 0 || e == h) continue;
      const cx<T> g2 = unit_mode<T, N>(f, kx, ky, m);
      lds[m * C::TX + q] = fill_element<T>(f, ab, g2, kx, ky, m);
      lds[e * C::TX + TX + q] = fill_element<T>(f, ab, {g2.x, -g2.y}, N - kx, my, e);
    }
  }
  if (x0 == 0) {
    // kx == 0 or kx == N/2: Hermitian part of the plane
    for (int i = threadIdx.x; i < 2 * N; i += C::NTG) {
      const int kx = i < N ? 0 : h, kz = i % N;
      const cx<T> ab = mode_amp<T, N>(f, amp, kx, ky, kz);
      const cx<T> a = unit_mode<T, N>(f, kx, ky, kz), b = unit_mode<T, N>(f, kx, my, (N - kz) % N);
      const cx<T> g = {(T)0.5 * (a.x + b.x), (T)0.5 * (a.y - b.y)};
      lds[kz * C::TX + (i < N ? 0 : TX)] = fill_element<T>(f, ab, g, kx, ky, kz);
    }
  }
  __syncthreads();
  if (C::NTG > C::NT && threadIdx.x >= C::NT) {   // whole waves
    Stockham<T, N, C::TC, C::MAXR>::template idle<true>();
    return;
  }
  const int c = threadIdx.x % C::TX, t = threadIdx.x / C::TX, kx = x0 + c % TX;
  cx<T> *col = F + (c < TX ? (size_t)kx + (size_t)N * ky
                           : (kx == 0 ? (size_t)h + (size_t)N * ky : (size_t)(N - kx) + (size_t)N * my));
  auto load = [&](int e) { return lds[e * C::TX + c]; };
  auto store = [&](int e, cx<T> v) { col[(size_t)e * n2] = v; };
  auto slot = [&](int e) -> cx<T> & { return lds[e * C::TX + c]; };
  Stockham<T, N, C::TC, C::MAXR>::template run<true>(t, load, store, slot, tw);
}

template <typename T, int N, int V>
__global__ __launch_bounds__((ColCfg<T, N, V>::NT)) void k_fft_y(cx<T> *__restrict__ F,
                                                               const cx<T> *__restrict__ tw, unsigned long long *st)
{
  using C = ColCfg<T, N, V>;
  __shared__ cx<T> lds[N * C::TX];
  stamp(st, STAMP_Y);
  const int c = threadIdx.x % C::TX, t = threadIdx.x / C::TX;
  // XCD-aware tile order: neighbouring column tiles of one plane run on one XCD, so tiles narrower
  // than a 128-byte line share each line through that XCD's L2 instead of fetching it twice
  const int b = xcd_swizzle((int)(blockIdx.y * gridDim.x + blockIdx.x), (int)(gridDim.x * gridDim.y));
  const int kx = (b % (int)gridDim.x) * C::TX + c, kz = b / (int)gridDim.x;
  cx<T> *col = F + (size_t)kx + (size_t)N * N * kz;
  auto load = [&](int e) { return col[(size_t)e * N]; };
  auto store = [&](int e, cx<T> v) { col[(size_t)e * N] = v; };
  auto slot = [&](int e) -> cx<T> & { return lds[e * C::TX + c]; };
  Stockham<T, N, C::TC, C::MAXR>::run(t, load, store, slot, tw);
}

template <typename T, int N, int V>
__global__ __launch_bounds__((RowCfg<T, N, V>::NT)) void k_fft_x(cx<T> *__restrict__ F,
                                                               const cx<T> *__restrict__ tw,
                                                               double norm, double norm_phi,
                                                               double *__restrict__ partials, unsigned long long *st)
{
  using C = RowCfg<T, N, V>;
  stamp(st, STAMP_X);
  __shared__ cx<T> lds[N * C::TY];
  __shared__ double red[2 * C::NT];
  __shared__ unsigned long long imax;
  const int t = threadIdx.x % C::TC, b = threadIdx.x / C::TC;
  const size_t row = (size_t)blockIdx.x * C::TY + b;
  cx<T> *line = F + row * N;
  double s1 = 0, s2 = 0, am = 0;
  if (threadIdx.x == 0) imax = 0;
  __syncthreads();
  auto load = [&](int e) { return line[e]; };
  auto store = [&](int e, cx<T> v) {
    cx<T> o = {(T)((double)v.x * norm), (T)((double)v.y * norm_phi)};
    double d = (double)o.x;
    s1 += d;
    s2 += d * d;
    am = fmax(am, fabs((double)o.y));
    line[e] = o;
  };
  auto slot = [&](int e) -> cx<T> & { return lds[b * N + e]; };
  Stockham<T, N, C::TC, C::MAXR>::run(t, load, store, slot, tw);
  red[threadIdx.x] = s1;
  red[C::NT + threadIdx.x] = s2;
  // largest |imaginary part| of the block: non-negative doubles order as their bit patterns
  atomicMax(&imax, (unsigned long long)__double_as_longlong(am));
  __syncthreads();
  for (int w = C::NT / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      red[threadIdx.x] += red[threadIdx.x + w];
      red[C::NT + threadIdx.x] += red[C::NT + threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = red[0];
    partials[2 * blockIdx.x + 1] = red[C::NT];
    partials[2 * gridDim.x + blockIdx.x] = __longlong_as_double((long long)imax);
  }
}

// ---------------------------------------------------------------------------------------------
// P(k) estimator: forward DFT of the resident grid as conj(IDFT(conj F)) -- kx pass on conj(F),
// the ky pass, and a kz pass that bins |delta_k|^2 into shells.
// ---------------------------------------------------------------------------------------------
template <typename T, int N>
__global__ __launch_bounds__((RowCfg<T, N>::NT)) void k_fft_x_conj(cx<T> *__restrict__ F,
                                                                 const cx<T> *__restrict__ tw)
{
  using C = RowCfg<T, N>;
  __shared__ cx<T> lds[N * C::TY];
  const int t = threadIdx.x % C::TC, b = threadIdx.x / C::TC;
  cx<T> *line = F + ((size_t)blockIdx.x * C::TY + b) * N;
  auto load = [&](int e) { return cconj(line[e]); };
  auto store = [&](int e, cx<T> v) { line[e] = v; };
  auto slot = [&](int e) -> cx<T> & { return lds[b * N + e]; };
  Stockham<T, N, C::TC>::run(t, load, store, slot, tw);
}

// G = IDFT(conj F) = conj(DFT F).  delta real => DFT(delta)_k = (DFT F_k + conj(DFT F_{-k}))/2
// = (conj G_k + G_{-k})/2; P_est = |DFT(delta)_k|^2 L^3 / N^6 summed into |k|/dk shells of width binw.
// acc[3*i] += P, acc[3*i+1] += |k|/dk, acc[3*i+2] += 1 (every k of the full grid).
//
// The kz pass bins where the columns stand: a workgroup transforms TX columns (kx, ky) with their mirrors
// (-kx, -ky), so every k it holds meets its -k, and nothing is written.  512^3 FP32 takes 505 us for its 1.07 GB, bound
// by the reads (segments of 64 bytes a plane apart) and the LDS sums; a pass that wrote the columns and one that read
// each mode and its mirror back took 641 + 691, three sums for every entry instead of a quarter of them 522.
template <typename T, int N>
struct PkCfg {
  static constexpr int TC = ColCfg<T, N>::TC;
  // at most 8 columns beside their mirrors and 64 KB: two workgroups or more share a CU, neighbours share lines
  // through their XCD's L2
  static constexpr int tx_for()
  {
    int tx = cmin(8, cpow2_div(N / 2));
    while (tx > 1 && (2 * tx * N * (int)sizeof(cx<T>) > 65536 || 2 * tx * TC > 1024)) tx /= 2;
    return tx;
  }
  static constexpr int TX = tx_for(), NT = 2 * TX * TC;
  // a column's place in LDS when it is binned, padded so that the store of the columns and a wave's read along one
  // column both spread over the banks
  static constexpr int LZ = N + 8;
  // kx in [0, N/2), TX of them to a tile, for every ky; then kx = N/2, TX of its ky to a tile
  static constexpr int TILES = N / 2 / TX * N + N / TX;
};

// A workgroup takes several tiles (neighbouring workgroups of an XCD neighbouring tiles) and hands its shell sums
// over once: a workgroup for each tile would end in 10^7 atomics on the same few hundred words.  The shells of a
// wave's 64 places decide how many of its LDS atomics meet in one word, so a wave goes along kz.
template <typename T, int N, int HB>
__global__ __launch_bounds__((PkCfg<T, N>::NT)) void k_pk_z(const cx<T> *__restrict__ F, const cx<T> *__restrict__ tw,
                                                            double pscale, double binw, int nbins,
                                                            double *__restrict__ acc)
{
  using C = PkCfg<T, N>;
  __shared__ cx<T> lds[C::LZ * 2 * C::TX];
  __shared__ double h[3 * HB];
  constexpr int NX = N / 2 / C::TX, HF = N / 2, CHUNK = (C::TILES + 7) / 8;
  const int c = threadIdx.x % (2 * C::TX), t = threadIdx.x / (2 * C::TX);
  const size_t n2 = (size_t)N * N;
  for (int i = threadIdx.x; i < 3 * nbins; i += C::NT) h[i] = 0;
  const int xcd = blockIdx.x % 8, end = cmin((xcd + 1) * CHUNK, C::TILES);
  for (int tile = xcd * CHUNK + (int)blockIdx.x / 8; tile < end; tile += (int)gridDim.x / 8) {
    const bool nyq = tile >= NX * N;
    const int x0 = nyq ? HF : tile % NX * C::TX, y0 = nyq ? (tile - NX * N) * C::TX : tile / NX;
    int kx = x0 + (nyq ? 0 : c % C::TX), ky = y0 + (nyq ? c % C::TX : 0);
    if (c >= C::TX) {
      kx = (N - kx) % N;
      ky = (N - ky) % N;
    }
    const cx<T> *col = F + (size_t)kx + (size_t)N * ky;
    auto load = [&](int e) { return col[(size_t)e * n2]; };
    auto slot = [&](int e) -> cx<T> & { return lds[e * 2 * C::TX + c]; };
    auto store = [&](int e, cx<T> v) { lds[c * C::LZ + e] = v; };   // every read through slot() has ended
    Stockham<T, N, C::TC>::run(t, load, store, slot, tw);
    __syncthreads();
    for (int i = threadIdx.x; i < C::TX * (HF + 1); i += C::NT) {
      const int q = i / (HF + 1), e = i % (HF + 1), m = (N - e) % N;
      const int bx = x0 + (nyq ? 0 : q), by = y0 + (nyq ? q : 0), ay = by <= HF ? by : N - by;
      const double kk = sqrt((double)(bx * bx + ay * ay + e * e));
      const int bin = (int)(kk / binw);
      if (bin >= nbins) continue;
      const cx<T> *g = lds + q * C::LZ, *gm = g + C::TX * C::LZ;
      const double re = 0.5 * ((double)g[e].x + (double)gm[m].x), im = 0.5 * ((double)gm[m].y - (double)g[e].y);
      double p = re * re + im * im;
      const bool two = e > 0 && e < HF;   // kz = N - e beside e
      if (two) {
        const double re2 = 0.5 * ((double)g[m].x + (double)gm[e].x), im2 = 0.5 * ((double)gm[e].y - (double)g[m].y);
        p += re2 * re2 + im2 * im2;
      }
      const bool mir = bx > 0 && !nyq;    // the mirrors' own modes: kx = 0 and N/2 have theirs at another ky of theirs
      atomicAdd(&h[3 * bin], (mir ? 2 * p : p) * pscale);
      // the shell's count and |k| are the same for +-ky, and for ky and kz exchanged: one entry stands for all
      if (by <= HF && e <= by) {
        const double w = (mir ? 2.0 : 1.0) * (two ? 2.0 : 1.0) * (by > 0 && by < HF ? 2.0 : 1.0) * (e < by ? 2.0 : 1.0);
        atomicAdd(&h[3 * bin + 1], w * kk);
        atomicAdd(&h[3 * bin + 2], w);
      }
    }
    __syncthreads();
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 3 * nbins; i += C::NT)
    if (h[i] != 0) atomicAdd(&acc[i], h[i]);
}

template <typename T, int N>
static hipError_t launch_pk_n(cx<T> *F, const cx<T> *tw, double pscale, double binw, int nbins, double *acc,
                              hipStream_t s)
{
  using CC = ColCfg<T, N>;
  using RC = RowCfg<T, N>;
  using PC = PkCfg<T, N>;
  hipLaunchKernelGGL((k_fft_x_conj<T, N>), dim3((N * N) / RC::TY), dim3(RC::NT), 0, s, F, tw);
  hipLaunchKernelGGL((k_fft_y<T, N, 0>), dim3(N / CC::TX, N), dim3(CC::NT), 0, s, F, tw, (unsigned long long *)nullptr);
  // four workgroups for each CU at most, a multiple of 8 (the XCDs)
  const unsigned nb = (unsigned)cmin((PC::TILES + 7) / 8 * 8, 1024);
  if (nbins <= 512)
    hipLaunchKernelGGL((k_pk_z<T, N, 512>), dim3(nb), dim3(PC::NT), 0, s, F, tw, pscale, binw, nbins, acc);
  else
    hipLaunchKernelGGL((k_pk_z<T, N, PK_MAX_BINS>), dim3(nb), dim3(PC::NT), 0, s, F, tw, pscale, binw, nbins, acc);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_power_spectrum(int n, cx<T> *F, const cx<T> *tw, double pscale, double binw, int nbins,
                                 double *acc, hipStream_t s)
{
  switch (n) {
#define CRIME_CASE(NN) \
  case NN: return launch_pk_n<T, NN>(F, tw, pscale, binw, nbins, acc, s);
    CRIME_FOR_EACH_N(CRIME_CASE)
#undef CRIME_CASE
  default: return hipErrorInvalidValue;
  }
}
template hipError_t launch_power_spectrum<float>(int, cx<float> *, const cx<float> *, double, double, int,
                                                 double *, hipStream_t);
template hipError_t launch_power_spectrum<double>(int, cx<double> *, const cx<double> *, double, double, int,
                                                  double *, hipStream_t);

// Partials of n blocks: sums p[2 i], sums of squares p[2 i + 1], largest |imaginary part| p[2 n + i].  The block's
// thread t takes the entries of index t mod NT (from first, every stride), then a tree: a fixed order.
template <int NT>
__device__ __forceinline__ void sigma_reduce(const double *__restrict__ p, int n, int first, int stride, double &a,
                                             double &b, double &c)
{
  __shared__ double r1[NT], r2[NT], r3[NT];
  a = b = c = 0;
  for (int i = first; i < n; i += stride) {
    a += p[2 * i];
    b += p[2 * i + 1];
    c = fmax(c, p[2 * n + i]);
  }
  const int t = threadIdx.x;
  r1[t] = a;
  r2[t] = b;
  r3[t] = c;
  __syncthreads();
  for (int w = NT / 2; w > 0; w >>= 1) {
    if (t < w) {
      r1[t] += r1[t + w];
      r2[t] += r2[t + w];
      r3[t] = fmax(r3[t], r3[t + w]);
    }
    __syncthreads();
  }
  a = r1[0];
  b = r2[0];
  c = r3[0];
}

// first step of a long reduction: one workgroup over 1024^3's half million partials took 265 us
__global__ __launch_bounds__(256) void k_sigma_blocks(const double *__restrict__ p, int n, double *__restrict__ out,
                                                      unsigned long long *st)
{
  stamp(st, STAMP_SIGMA);
  double a, b, c;
  sigma_reduce<256>(p, n, blockIdx.x * 256 + threadIdx.x, 256 * SIGMA_BLOCKS, a, b, c);
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = a;
    out[2 * blockIdx.x + 1] = b;
    out[2 * SIGMA_BLOCKS + blockIdx.x] = c;
  }
}

__global__ __launch_bounds__(1024) void k_sigma_finalize(const double *__restrict__ partials, int nparts, double ncells,
                                                         double *__restrict__ out, unsigned long long *st,
                                                         unsigned long long *st_end)
{
  stamp(st, STAMP_SIGMA);
  double a, b, c;
  sigma_reduce<1024>(partials, nparts, threadIdx.x, 1024, a, b, c);
  if (threadIdx.x == 0) {
    double mean = a / ncells;
    out[0] = b / ncells - mean * mean;  // sigma2_gauss (fourier.c:74)
    out[1] = mean;
    out[2] = c;  // max |imaginary part| of the grid (the map stage's bound on the velocity)
    stamp(st_end, STAMP_FIELDS_END);
  }
}

__global__ __launch_bounds__(64) void k_run_end(const double *__restrict__ sig, unsigned long long *stamps,
                                                RunEnd *__restrict__ out)
{
  const int t = threadIdx.x;
  if (t < 2) out->sig[t] = sig[t];
  if (t < N_STAMPS) out->stamp[t] = t == STAMP_END ? (unsigned long long)wall_clock64() : stamps[t];
  __threadfence_system();
}

hipError_t launch_run_end(const double *sig, unsigned long long *stamps, RunEnd *out, hipStream_t s)
{
  hipLaunchKernelGGL(k_run_end, dim3(1), dim3(64), 0, s, sig, stamps, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
template <typename T, int N, int V>
static void launch_fill_v(cx<T> *F, const FillParams &f, const cx<T> *tw, hipStream_t s)
{
  using FC = FillCfg<T, N, V>;
  hipLaunchKernelGGL((k_fill_z<T, N, V>), dim3(N / FC::TX * N), dim3(FC::NTG), 0, s, F, f, tw);
}

template <typename T, int N, int V>
static void launch_y_v(cx<T> *F, const cx<T> *tw, hipStream_t s, unsigned long long *st)
{
  using CC = ColCfg<T, N, V>;
  hipLaunchKernelGGL((k_fft_y<T, N, V>), dim3(N / CC::TX, N), dim3(CC::NT), 0, s, F, tw, st);
}

template <typename T, int N, int V>
static int launch_x_v(cx<T> *F, const cx<T> *tw, double norm, double norm_phi, double *partials, hipStream_t s,
                      unsigned long long *st)
{
  using RC = RowCfg<T, N, V>;
  const int nrowblk = (N * N) / RC::TY;
  hipLaunchKernelGGL((k_fft_x<T, N, V>), dim3(nrowblk), dim3(RC::NT), 0, s, F, tw, norm, norm_phi, partials, st);
  return nrowblk;
}

template <typename T, int N>
static void fill_sched(cx<T> *F, const FillParams &f, const cx<T> *tw, hipStream_t s, const Schedule &sc)
{
  constexpr bool tuned = N >= TUNE_MIN_N;
  if (tuned && sc.fill == 1) launch_fill_v<T, N, tuned ? 1 : 0>(F, f, tw, s);
  else if (tuned && sc.fill == 2) launch_fill_v<T, N, tuned ? 2 : 0>(F, f, tw, s);
  else if (tuned && sc.fill == 3) launch_fill_v<T, N, tuned ? 3 : 0>(F, f, tw, s);
  else launch_fill_v<T, N, 0>(F, f, tw, s);
}

template <typename T, int N>
static void y_sched(cx<T> *F, const cx<T> *tw, hipStream_t s, const Schedule &sc, unsigned long long *st)
{
  constexpr bool tuned = N >= TUNE_MIN_N;
  if (tuned && sc.y == 1) launch_y_v<T, N, tuned ? 1 : 0>(F, tw, s, st);
  else if (tuned && sc.y == 2) launch_y_v<T, N, tuned ? 2 : 0>(F, tw, s, st);
  else if (tuned && sc.y == 3) launch_y_v<T, N, tuned ? 3 : 0>(F, tw, s, st);
  else launch_y_v<T, N, 0>(F, tw, s, st);
}

template <typename T, int N>
static int x_sched(cx<T> *F, const cx<T> *tw, double nre, double nim, double *partials, hipStream_t s,
                   const Schedule &sc, unsigned long long *st)
{
  constexpr bool tuned = N >= TUNE_MIN_N;
  if (tuned && sc.x == 1) return launch_x_v<T, N, tuned ? 1 : 0>(F, tw, nre, nim, partials, s, st);
  if (tuned && sc.x == 2) return launch_x_v<T, N, tuned ? 2 : 0>(F, tw, nre, nim, partials, s, st);
  if (tuned && sc.x == 3) return launch_x_v<T, N, tuned ? 3 : 0>(F, tw, nre, nim, partials, s, st);
  return launch_x_v<T, N, 0>(F, tw, nre, nim, partials, s, st);
}

// Stage times cover both grids of a spectral handle: the second grid's pass runs right before the same pass of F
// (and is the one stamped), and its sigma^2 partials are overwritten by F's kx pass.
template <typename T, int N>
static hipError_t launch_fields_n(cx<T> *F, cx<T> *G, const FillParams &f, const cx<T> *tw, double norm,
                                  double *partials, double *sig, hipStream_t s, const Schedule &sc)
{
  const bool two = f.vmode != 0;
  unsigned long long *const st = f.stamp, *const st2 = two ? nullptr : st;
  FillParams f0 = f, f1 = f;
  f0.stamp = st2;
  f1.comp = 1;
  if (two) fill_sched<T, N>(G, f1, tw, s, sc);
  fill_sched<T, N>(F, f0, tw, s, sc);
  if (two) y_sched<T, N>(G, tw, s, sc, st);
  y_sched<T, N>(F, tw, s, sc, st2);
  const double nphi = norm / f.phi_scale;
  if (two) x_sched<T, N>(G, tw, nphi, nphi, partials, s, sc, st);
  int n = x_sched<T, N>(F, tw, norm, nphi, partials, s, sc, st2);
  unsigned long long *sts = st;
  if (n > 16 * SIGMA_BLOCKS) {
    double *out = partials + 3 * (size_t)n;
    hipLaunchKernelGGL(k_sigma_blocks, dim3(SIGMA_BLOCKS), dim3(256), 0, s, partials, n, out, st);
    partials = out;
    n = SIGMA_BLOCKS;
    sts = nullptr;
  }
  hipLaunchKernelGGL(k_sigma_finalize, dim3(1), dim3(1024), 0, s, partials, n, (double)N * N * N, sig, sts, st);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_fields(int n, cx<T> *F, cx<T> *G, const FillParams &f, const cx<T> *tw, double norm,
                         double *partials, double *sig, hipStream_t s, const Schedule &sc)
{
  if (f.vmode != 0 && (!G || !f.sin_dx)) return hipErrorInvalidValue;
  switch (n) {
#define CRIME_CASE(NN) \
  case NN: return launch_fields_n<T, NN>(F, G, f, tw, norm, partials, sig, s, sc);
    CRIME_FOR_EACH_N(CRIME_CASE)
#undef CRIME_CASE
  default: return hipErrorInvalidValue;
  }
}

template hipError_t launch_fields<float>(int, cx<float> *, cx<float> *, const FillParams &, const cx<float> *,
                                         double, double *, double *, hipStream_t, const Schedule &);
template hipError_t launch_fields<double>(int, cx<double> *, cx<double> *, const FillParams &, const cx<double> *,
                                          double, double *, double *, hipStream_t, const Schedule &);

template <typename T>
hipError_t launch_amp_table(const FillParams &f, void *tab, hipStream_t s)
{
  int mmax = amp_count(f.n) - 1;
  hipLaunchKernelGGL(k_amp_table<T>, dim3((mmax + 256) / 256), dim3(256), 0, s, f, (AmpEntry<T> *)tab, mmax);
  return hipGetLastError();
}
template hipError_t launch_amp_table<float>(const FillParams &, void *, hipStream_t);
template hipError_t launch_amp_table<double>(const FillParams &, void *, hipStream_t);

// the most row blocks any schedule variant launches (variant 1 has the fewest rows per block)
int fields_partials_count(int n, int prec)
{
  switch (n) {
#define CRIME_CASE(NN) \
  case NN: return prec ? (NN * NN) / RowCfg<double, NN, 1>::TY : (NN * NN) / RowCfg<float, NN, 1>::TY;
    CRIME_FOR_EACH_N(CRIME_CASE)
#undef CRIME_CASE
  default: return 0;
  }
}

}  // namespace crime
