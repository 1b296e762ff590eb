// grad.hip -- adjoint of the solve (no counterpart in the reference).
//
// For the potentials phi = A(x) q of m charge vectors and a loss with
// g = dLoss/dphi, the FMM operator A is symmetric (the same interpolants
// in P2M and L2P, M2M the transpose of L2L, E_{-v} = E_v^T over the
// interaction lists), so
//     dLoss/dq_v   = A g_v                       (a solve with charges g),
//     dLoss/dx_k   = sum_v g_vk grad Phi_{q_v}(x_k) + q_vk grad Phi_{g_v}(x_k),
// where Phi_c is the FMM potential of charges c.  One solve of the 2m
// stacked vectors [q; g] recomputes all expansions; the far part of the
// position gradient is the gradient of the L2P interpolant (Chebyshev
// derivative) of the leaf's local values F, the near part the gradient of
// 1/r over the same leaf neighbourhoods as P2P.
#include "common.h"
#include "kernels.h"

namespace bb {

__device__ __forceinline__ real rsqrt_g(real x)
{
#ifdef SINGLE
  return __builtin_amdgcn_rsqf(x);
#else
  return 1.0 / sqrt(x);
#endif
}

// S_n(x_m, xi) and dS_n/dxi for m = 0..NN-1, xi in [-1, 1]:
// S = 1/2 + sum_{k>=1} T_k(x_m) T_k(xi),  dS/dxi = sum_{k>=1} T_k(x_m) k U_{k-1}(xi).
template <int NN>
__device__ __forceinline__ void cheb_val_der(const real *__restrict__ Tkz, real xi, real *s, real *ds)
{
  real T[NN], Ud[NN];
  T[0] = 1;
  Ud[0] = 1;  // U_0
  if (NN > 1) {
    T[1] = xi;
    Ud[1] = 2 * xi;  // U_1
  }
#pragma unroll
  for (int k = 2; k < NN; k++) {
    T[k] = 2 * xi * T[k - 1] - T[k - 2];
    Ud[k] = 2 * xi * Ud[k - 1] - Ud[k - 2];
  }
#pragma unroll
  for (int m = 0; m < NN; m++) {
    real v = (real)0.5 * Tkz[m * NN], d = 0;
#pragma unroll
    for (int k = 1; k < NN; k++) {
      const real c = Tkz[m * NN + k];
      v += c * T[k];
      d += c * (real)k * Ud[k - 1];
    }
    s[m] = v;
    ds[m] = d;
  }
}

// Far part: dx[c][i] = prefac3 / (L_leaf / 2) * d/dxi_c sum_l S_l(xi) Fc_l,
// Fc = sum_v g_vi F_{q_v} + q_vi F_{g_v} on the particle's leaf.  One block
// per leaf, a thread per particle; a slab of nodes (fixed l1) of the leaf's
// F is staged in LDS for all of them (every value as a uniform load of its
// own, one at a time: 128 us at N = 262144, depth 4, n = 4, 8 vectors; so
// staged 32).
template <int NN, int MMAX, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_l2p_grad(GradArgs a)
{
  constexpr int N2 = NN * NN, N3 = NN * N2;
  __shared__ real sF[N2][2 * MMAX] __attribute__((aligned(16)));
  const int leaf = blockIdx.x;
  const int A = a.leafcell[leaf];
  const real ih = a.leafihalf[leaf];
  const int sta = a.leafsta[leaf], cnt = a.leafcnt[leaf];
  const real4 c = a.center[A];
  for (int j0 = 0; j0 < cnt; j0 += BLOCK) {
    const bool act = j0 + (int)threadIdx.x < cnt;
    const int i = sta + min(j0 + (int)threadIdx.x, cnt - 1);
    const real4 x = a.pos[i];
    real sx[NN], dsx[NN], sy[NN], dsy[NN], sz[NN], dsz[NN];
    cheb_val_der<NN>(a.Tkz, ih * (x.x - c.x), sx, dsx);
    cheb_val_der<NN>(a.Tkz, ih * (x.y - c.y), sy, dsy);
    cheb_val_der<NN>(a.Tkz, ih * (x.z - c.z), sz, dsz);
    if (NN % 4 == 3 && a.l2p_ref) {  // the reference's L2P z weights (anotherDownwardPassX.c:304)
      sz[NN - 1] = sz[NN - 2];
      dsz[NN - 1] = dsz[NN - 2];
    }
    real w[2 * MMAX];  // g for the values of q, q for those of g
#pragma unroll
    for (int v = 0; v < MMAX; v++) {
      w[v] = v < a.mb ? a.qg[(size_t)(a.m + a.v0 + v) * a.N + i] : (real)0;
      w[MMAX + v] = v < a.mb ? a.qg[(size_t)(a.v0 + v) * a.N + i] : (real)0;
    }
    real gx = 0, gy = 0, gz = 0;
#pragma unroll 1
    for (int l1 = 0; l1 < NN; l1++) {
      __syncthreads();  // the previous slab has been read
      for (int o = threadIdx.x; o < N2 * 2 * MMAX; o += BLOCK) {
        const int v = o / N2, l = o - v * N2, u = v < MMAX ? v : v - MMAX;
        sF[l][v] = u < a.mb ? a.F[((size_t)((v < MMAX ? 0 : a.m) + a.v0 + u) * a.ncell + A) * N3 + l1 * N2 + l] : (real)0;
      }
      __syncthreads();
      real s1 = 0, d1 = 0;
#pragma unroll
      for (int k = 0; k < NN; k++) {
        s1 = k == l1 ? sx[k] : s1;
        d1 = k == l1 ? dsx[k] : d1;
      }
#pragma unroll
      for (int l2 = 0; l2 < NN; l2++) {
        real in_s = 0, in_d = 0;
#pragma unroll
        for (int l3 = 0; l3 < NN; l3++) {
          real f = 0;
#pragma unroll
          for (int v = 0; v < 2 * MMAX; v++) f += w[v] * sF[l2 * NN + l3][v];
          in_s += sz[l3] * f;
          in_d += dsz[l3] * f;
        }
        gx += d1 * sy[l2] * in_s;
        gy += s1 * dsy[l2] * in_s;
        gz += s1 * sy[l2] * in_d;
      }
    }
    if (!act) continue;
    const real sc = a.prefac3 * ih;
    if (a.v0 > 0) {  // a later block of vectors: add to the earlier blocks' sum
      a.dx[i] += sc * gx;
      a.dx[(size_t)a.N + i] += sc * gy;
      a.dx[(size_t)2 * a.N + i] += sc * gz;
    } else {
      a.dx[i] = sc * gx;
      a.dx[(size_t)a.N + i] = sc * gy;
      a.dx[(size_t)2 * a.N + i] = sc * gz;
    }
  }
}

// ---------------------------------------------------------------- near part
// For target k of the leaf, with q and g the charges of the block's vectors:
//   dx_k += sum_j (sum_v g_vk q_vj + q_vk g_vj) (x_j - x_k) / r_kj^3
//   phi_{g_v}(k) += sum_j g_vj / r_kj
// over the particles j of the neighbour leaves with r_kj != 0: the gradient
// and the near field of the potentials it returns share 1/r (as two kernels,
// a lane a target and the 16-vector P2P of q and g, they took 818 + 233 us at
// N = 262144, depth 4, 8 vectors; this one 525).  r != 0 is tested in the leaf
// itself only: coordinates that fall into different leaves differ by an ulp of
// x + L/2 or more, 3e-8 of a leaf in fp32, so that r^2 between two leaves
// vanishes only in root cells so small (1e-15 fp32, 3e-146 fp64, twice as
// large with each level) that 1 / r^3 overflows for every pair.
//
// Lanes are 16 targets (l % 16) by 4 source groups (l / 16), NT tiles of
// targets share the sources that a wave stages in LDS, kStage at a time across
// leaves (a lane finds its source's leaf by bisection), the next chunk's loads
// in flight during a chunk's sums, padded to a multiple of 16 with copies of its
// last source that carry no charge.  The W waves of a block take the chunks in turn, their sums
// added through LDS; the passes over target tiles go to gridDim.y blocks.
// Bound by the matrix unit and the vector ALUs, which do not overlap in fp32
// (8 vectors: 8 products of 32 cycles and about 190 cycles of 1/r per 256
// pairs, 0.6 of which is reached), half of the potentials' product idle at 8.
// MFMA (fp32, NR = 8 or 16): the weights of 16 sources x 16 targets are one
// product over the 2 NR charges (v_mfma_f32_16x16x4_f32; a lane gets those of
// its target and the sources 4 (l / 16) .. + 3), and the potentials another
// over the sources, as in the 16-vector P2P.  Else: FMAs, a lane taking the
// sources l / 16, l / 16 + 4, ...
constexpr int kStage = 64;  // one source a lane
typedef real rx4 __attribute__((ext_vector_type(4)));

template <int NR>
struct GradStage {
  rx4 s[kStage];
  real c[kStage][2 * NR + 4] __attribute__((aligned(16)));  // q, then g (+ 4: LDS banks)
};

template <int NR, int NT>
struct GradSums {
  rx4 x[NT];              // targets' positions
  real ax[NT], ay[NT], az[NT];
  real tc[NT][2 * NR];    // targets' charges: g, then q (FMA form)
  rx4 tm[NT][NR / 8 ? NR / 8 : 1];  // those of the lane's k slots (MFMA form)
  real phi[NT][NR];       // FMA form
  rx4 pm[NT][1];          // MFMA form: vectors 4 (l / 16) .. + 3 of the lane's target
};

template <int NR, bool MFMA, int NT, bool SELF>
__device__ __forceinline__ void grad_sweep(const GradStage<NR> &st, int n16, int ti, int h, GradSums<NR, NT> &u)
{
#ifdef SINGLE
  if constexpr (MFMA) {
    constexpr int NB = NR / 8;
    for (int k = 0; k < n16; k += 16) {
      rx4 ca[NB], z[4];
      real pa[4];
#pragma unroll
      for (int c = 0; c < NB; c++) ca[c] = *reinterpret_cast<const rx4 *>(&st.c[k + ti][16 * c + 4 * h]);
#pragma unroll
      for (int v = 0; v < 4; v++) {
        z[v] = st.s[k + 4 * h + v];
        pa[v] = st.c[k + 4 * h + v][NR + (NR == 8 ? ti & 7 : ti)];  // NR = 8: rows 8 .. 15 repeat, not stored
      }
#pragma unroll
      for (int t = 0; t < NT; t++) {
        rx4 w = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < NB; c++)
#pragma unroll
          for (int e = 0; e < 4; e++) w = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[c][e], u.tm[t][c][e], w, 0, 0, 0);
        real ri[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const real dx = z[v].x - u.x[t].x, dy = z[v].y - u.x[t].y, dz = z[v].z - u.x[t].z;
          const real rr = dx * dx + dy * dy + dz * dz;
          ri[v] = SELF && rr == (real)0 ? (real)0 : rsqrt_g(rr);
          const real f = w[v] * (ri[v] * ri[v] * ri[v]);
          u.ax[t] += f * dx;
          u.ay[t] += f * dy;
          u.az[t] += f * dz;
        }
#pragma unroll
        for (int v = 0; v < 4; v++) u.pm[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[v], ri[v], u.pm[t][0], 0, 0, 0);
      }
    }
    return;
  }
#endif
  for (int k4 = 0; k4 < n16; k4 += 4) {
    const int k = k4 + h;
    const rx4 z = st.s[k];
    real c[2 * NR];
#pragma unroll
    for (int v = 0; v < 2 * NR; v++) c[v] = st.c[k][v];
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const real dx = z.x - u.x[t].x, dy = z.y - u.x[t].y, dz = z.z - u.x[t].z;
      const real rr = dx * dx + dy * dy + dz * dz;
      const real ri = SELF && rr == (real)0 ? (real)0 : rsqrt_g(rr);
      real w = 0;
#pragma unroll
      for (int v = 0; v < 2 * NR; v++) w += u.tc[t][v] * c[v];
#pragma unroll
      for (int v = 0; v < NR; v++) u.phi[t][v] += ri * c[NR + v];
      const real f = w * (ri * ri * ri);
      u.ax[t] += f * dx;
      u.ay[t] += f * dy;
      u.az[t] += f * dz;
    }
  }
}

template <int NR, bool MFMA, int NT, int W>
__device__ __forceinline__ void grad_tiles(const GradArgs &a, int tb, int sta, int cnt, const int *end,
                                           const int *delta, int total, GradStage<NR> &st, real *red)
{
  const int lane = threadIdx.x & 63;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  const int ti = lane & 15, h = lane >> 4;
  const size_t N = a.N;
  const rx4 *pos = reinterpret_cast<const rx4 *>(a.pos);
  // charge k of particle i: q of the block's vectors, then g, zero past mb
  auto charge = [&](int k, int i) -> real {
    const int v = k < NR ? k : k - NR;
    return v < a.mb ? a.qg[(size_t)((k < NR ? 0 : a.m) + a.v0 + v) * N + i] : (real)0;
  };
  GradSums<NR, NT> u;
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int i = sta + min(tb + 16 * t + ti, cnt - 1);  // targets past the leaf's end are not stored
    u.x[t] = pos[i];
    u.ax[t] = u.ay[t] = u.az[t] = 0;
    if constexpr (MFMA) {
#pragma unroll
      for (int c = 0; c < NR / 8; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) u.tm[t][c][e] = charge((16 * c + 4 * h + e + NR) % (2 * NR), i);
      u.pm[t][0] = rx4{0, 0, 0, 0};
    } else {
#pragma unroll
      for (int v = 0; v < 2 * NR; v++) u.tc[t][v] = charge((v + NR) % (2 * NR), i);
#pragma unroll
      for (int v = 0; v < NR; v++) u.phi[t][v] = 0;
    }
  }
  // a chunk of kStage sources: a lane's is loaded into registers (past the
  // end, on = false: the last one, without charge), later moved into LDS
  rx4 rp;
  real rc[2 * NR];
  auto load = [&](bool on, int j) {
    rp = pos[j];
#pragma unroll
    for (int k = 0; k < 2 * NR; k++) rc[k] = 0;
    if (on) {
#pragma unroll
      for (int k = 0; k < 2 * NR; k++) rc[k] = charge(k, j);
    }
  };
  auto put = [&]() {
    st.s[lane] = rp;
#pragma unroll
    for (int k = 0; k < 2 * NR; k++) st.c[lane][k] = rc[k];
  };
  // source n of the other leaves, one after the other
  auto load_other = [&](int n) {
    const int m = min(n, total - 1);
    int b = 0;
#pragma unroll
    for (int d = 16; d > 0; d >>= 1)
      if (end[b + d - 1] <= m) b += d;
    load(n < total, m + delta[b]);
  };
  if (wave == 0)  // the leaf itself
    for (int j = 0; j < cnt; j += kStage) {
      load(j + lane < cnt, sta + min(j + lane, cnt - 1));
      put();
      wave_sync();
      grad_sweep<NR, MFMA, NT, true>(st, min(kStage, (cnt - j + 15) & ~15), ti, h, u);
      wave_sync();
    }
  int n = kStage * wave;
  if (n < total) load_other(n + lane);
  for (; n < total; n += kStage * W) {
    put();
    if (n + kStage * W < total) load_other(n + kStage * W + lane);  // in flight during the sums
    wave_sync();
    grad_sweep<NR, MFMA, NT, false>(st, min(kStage, (total - n + 15) & ~15), ti, h, u);
    wave_sync();
  }
  // sums over the lane groups (the MFMA potentials are whole already)
  auto groups = [&](real v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
  };
#pragma unroll
  for (int t = 0; t < NT; t++) {
    u.ax[t] = groups(u.ax[t]);
    u.ay[t] = groups(u.ay[t]);
    u.az[t] = groups(u.az[t]);
    if constexpr (!MFMA)
#pragma unroll
      for (int v = 0; v < NR; v++) u.phi[t][v] = groups(u.phi[t][v]);
  }
  // values of a lane: the gradient, and 4 potentials (MFMA) or all of them
  constexpr int NV = 3 + (MFMA ? 4 : NR);
  auto value = [&](int t, int v) -> real & {
    if (v == 0) return u.ax[t];
    if (v == 1) return u.ay[t];
    if (v == 2) return u.az[t];
    return u.phi[t][v - 3];
  };
  if (W > 1) {
    __syncthreads();  // the previous pass's sums have been read
    if (wave > 0)
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int v = 0; v < NV; v++)
          red[(((wave - 1) * NT + t) * NV + v) * 64 + lane] = MFMA && v >= 3 ? u.pm[t][0][(v - 3) & 3] : value(t, v < 3 || !MFMA ? v : 0);
    __syncthreads();
    if (wave > 0) return;
    for (int w = 0; w < W - 1; w++)
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int v = 0; v < NV; v++) {
          const real r = red[((w * NT + t) * NV + v) * 64 + lane];
          if (MFMA && v >= 3) u.pm[t][0][(v - 3) & 3] += r;
          else value(t, v < 3 || !MFMA ? v : 0) += r;
        }
  }
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int k = tb + 16 * t + ti, i = sta + k;
    if (k >= cnt) continue;
    if (h == 0) {
      a.dx[i] += u.ax[t];
      a.dx[N + i] += u.ay[t];
      a.dx[2 * N + i] += u.az[t];
    }
    if constexpr (MFMA) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (4 * h + e < a.mb) a.phi[(size_t)(a.m + a.v0 + 4 * h + e) * N + i] += u.pm[t][0][e];
    } else {
#pragma unroll
      for (int v = 0; v < NR; v++)
        if ((v & 3) == h && v < a.mb) a.phi[(size_t)(a.m + a.v0 + v) * N + i] += u.phi[t][v];
    }
  }
}

// tiles of targets that share the staged sources
constexpr int grad_tiles_max(int nr, bool mfma) { return mfma ? (nr == 8 ? 3 : 2) : nr <= 2 ? 3 : nr <= 4 ? 2 : 1; }

template <int NR, bool MFMA, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(sizeof(real) == 8 ? 1 : NR > 8 ? 3 : 4))) k_near_grad(GradArgs a)
{
  constexpr int NTM = grad_tiles_max(NR, MFMA), NV = 3 + (MFMA ? 4 : NR);
  __shared__ GradStage<NR> stage[W];
  __shared__ real red[W > 1 ? (W - 1) * NTM * NV * 64 : 1];
  // the other leaves' sources, one after the other: where leaf b's end in
  // that order, and from there to its particles
  __shared__ int end[32], delta[32];
  const int leaf = xcd_leaf(blockIdx.x, a.nleaf);
  const int sta = a.leafsta[leaf], cnt = a.leafcnt[leaf], nn = a.nnbr[leaf];
  // as few passes of equal tiles as NTM allows
  const int tiles = (cnt + 15) >> 4, np = (tiles + NTM - 1) / NTM;
  if ((int)blockIdx.y >= np) return;
  int total;
  {
    const int lane = threadIdx.x & 63;
    int s0 = 0, c = 0;
    if (lane < nn) {
      const int B = a.nbr[(size_t)leaf * 27 + lane];
      s0 = a.leafsta[B];
      c = B == leaf ? 0 : a.leafcnt[B];
    }
    int e = c;
    for (int d = 1; d < 32; d <<= 1) {
      const int o = __shfl_up(e, d);
      if (lane >= d) e += o;
    }
    total = __builtin_amdgcn_readlane(e, 31);
    if (threadIdx.x < 32) {
      end[lane] = lane < nn ? e : 0x7fffffff;
      delta[lane] = s0 - (e - c);
    }
  }
  __syncthreads();
  GradStage<NR> &st = stage[threadIdx.x >> 6];
  for (int p = blockIdx.y; p < np; p += gridDim.y) {
    const int t0 = tiles * p / np, nt = tiles * (p + 1) / np - t0, tb = 16 * t0;
    if (NTM >= 3 && nt == 3) grad_tiles<NR, MFMA, NTM >= 3 ? 3 : 1, W>(a, tb, sta, cnt, end, delta, total, st, red);
    else if (NTM >= 2 && nt == 2) grad_tiles<NR, MFMA, NTM >= 2 ? 2 : 1, W>(a, tb, sta, cnt, end, delta, total, st, red);
    else grad_tiles<NR, MFMA, 1, W>(a, tb, sta, cnt, end, delta, total, st, red);
  }
}

// dx (leaf order, [3][N]) -> out (original order, [N][3])
__global__ void k_scatter_vec3(int N, const int *__restrict__ iperm, const real *__restrict__ src,
                               real *__restrict__ out)
{
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  const int i = iperm[j];
  out[(size_t)3 * j] = src[i];
  out[(size_t)3 * j + 1] = src[(size_t)N + i];
  out[(size_t)3 * j + 2] = src[(size_t)2 * N + i];
}

template <int NN, int MMAX>
static void l2p_grad_t(const GradArgs &a, hipStream_t s)
{
  if (a.N > 48LL * a.nleaf)  // leaves of more than a wavefront
    hipLaunchKernelGGL((k_l2p_grad<NN, MMAX, 128>), dim3(a.nleaf), dim3(128), 0, s, a);
  else
    hipLaunchKernelGGL((k_l2p_grad<NN, MMAX, 64>), dim3(a.nleaf), dim3(64), 0, s, a);
}

template <int NN>
static void l2p_grad(const GradArgs &a, hipStream_t s)
{
  if (a.mb <= 1) l2p_grad_t<NN, 1>(a, s);
  else if (a.mb <= 4) l2p_grad_t<NN, 4>(a, s);
  else if (a.mb <= 8) l2p_grad_t<NN, 8>(a, s);
  else l2p_grad_t<NN, 16>(a, s);
}

// Waves of a block: leaves by the thousand leave the last round uneven and
// fewer do not fill the chip, so they split their sources over 4 waves (2
// where a wave's registers and LDS allow few of them).  dq and dx of the
// whole gradient in us with 1, 2, 4 waves: N = 262144, 4096 leaves, 8 vectors
// 800, 776, 766, 1 vector 376, 352, 343, 16 vectors 1223, 1212, 1263; 50000,
// 512 leaves, 12 vectors 514, 434, 409; 900000, 32768 leaves, 8 vectors 2153,
// 2179, 2255; fp64 60000, 4096 leaves, 8 vectors 733, 725, 775.
template <int NR, bool MFMA>
static void near_grad_t(const GradArgs &a, hipStream_t s)
{
  const dim3 grid(a.nleaf, 4);
  const bool large = NR * sizeof(real) >= 64;  // (16 vectors, or 8 in fp64)
  if (a.nleaf > 8192) hipLaunchKernelGGL((k_near_grad<NR, MFMA, 1>), grid, dim3(64), 0, s, a);
  else if (large && a.nleaf > 1024) hipLaunchKernelGGL((k_near_grad<NR, MFMA, 2>), grid, dim3(128), 0, s, a);
  else hipLaunchKernelGGL((k_near_grad<NR, MFMA, 4>), grid, dim3(256), 0, s, a);
}

static void near_grad(const GradArgs &a, hipStream_t s)
{
#ifdef SINGLE
  if (a.mb > 8) return near_grad_t<16, true>(a, s);
  if (a.mb > 4) return near_grad_t<8, true>(a, s);
#endif
  if (a.mb > 4) near_grad_t<8, false>(a, s);
  else if (a.mb > 2) near_grad_t<4, false>(a, s);
  else if (a.mb == 2) near_grad_t<2, false>(a, s);
  else near_grad_t<1, false>(a, s);
}

int launch_gradient(const GradArgs &a0, const int *iperm, real *dx_out, hipStream_t s)
{
  if (a0.nleaf <= 0 || a0.N <= 0) return BBFMM_OK;
  // blocks of vectors, summed into dx in order: the far part first
  for (int v0 = 0; v0 < a0.m; v0 += 16) {
    GradArgs a = a0;
    a.v0 = v0;
    a.mb = a0.m - v0 < 16 ? a0.m - v0 : 16;
    BB_WITH_ORDER(a.n, l2p_grad<NN>(a, s));
  }
  BB_HIP(hipGetLastError());
  constexpr int MB = sizeof(real) == 4 ? 16 : 8;
  for (int v0 = 0; v0 < a0.m; v0 += MB) {
    GradArgs a = a0;
    a.v0 = v0;
    a.mb = a0.m - v0 < MB ? a0.m - v0 : MB;
    near_grad(a, s);
  }
  BB_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_scatter_vec3, dim3((a0.N + 255) / 256), dim3(256), 0, s, a0.N, iperm, a0.dx, dx_out);
  BB_HIP(hipGetLastError());
  return BBFMM_OK;
}

} // namespace bb
