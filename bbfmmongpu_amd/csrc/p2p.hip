// p2p.hip -- near-field P2P on the leaf level: for every particle i of leaf A,
//   phi_i += q_i * sum_{B in neighbours(A)} sum_{j in B, r_ij != 0} q_j / r_ij
// (the semantics of the reference GPU kernel direct.cu:69-209 and the CPU
// anotherNearField.c:137-206; the r != 0 test is applied in the self leaf).
//
// Up to 8 right-hand sides are processed together so that the geometry (dx,
// dy, dz, 1/r) is computed once per pair and shared by their charges; 16 take
// the kernels on the padded layout.
// 1/r: fp32 uses the hardware v_rsq_f32 (AMD's own reciprocal square root,
// about 1 ulp); fp64 one iteration from v_rsq_f64 (rsqrt_r).
#include "common.h"
#include "kernels.h"

#include <type_traits>

namespace bb {

__device__ __forceinline__ real rsqrt_r(real x)
{
#ifdef SINGLE
  return __builtin_amdgcn_rsqf(x);
#else
  // the hardware's estimate (5e-8) and one third-order step: as exact as the
  // library's rsqrt (1.4e-16 at most over 1e-12 .. 100) without its special
  // cases, 47 against 60 cycles a wavefront: x is positive and finite here, or
  // the result is not used (r^2 overflows in root cells of 1e154: NaN, not 0)
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-x * y, y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
#endif
}

// Sparse forests, where leaves hold a few particles: a lane per target
// particle, sweeping its own leaf's neighbour list (the neighbour leaves'
// particles straight from memory; lanes of one leaf read the same source at
// the same time).  Same sums as above; the r != 0 test is applied to every
// neighbour leaf, which changes nothing since coincident particles share a
// leaf.
template <int NR>
__global__ void __launch_bounds__(256) k_p2p_lane(P2PArgs a, int rhs0)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.N) return;
  const int lf = a.leafof[i];
  const real4 x = a.pos[i];
  const int nn = a.nnbr[lf];
  const int *nb = a.nbr + (size_t)lf * 27;
  const size_t N = a.N;
  real acc[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) acc[r] = 0;
  // the next neighbour's range is fetched while this one's sources are summed
  int Bn = nb[0];  // nn >= 1: the leaf itself
  int j0n = a.leafsta[Bn], cn = a.leafcnt[Bn];
  for (int b = 0; b < nn; b++) {
    const int j0 = j0n, j1 = j0 + cn;
    if (b + 1 < nn) {
      Bn = nb[b + 1];
      j0n = a.leafsta[Bn];
      cn = a.leafcnt[Bn];
    }
    for (int j = j0; j < j1; j++) {
      const real4 y = a.pos[j];
      const real dx = y.x - x.x, dy = y.y - x.y, dz = y.z - x.z;
      const real rr = dx * dx + dy * dy + dz * dz;
      const real w = rr != (real)0 ? rsqrt_r(rr) : (real)0;
#pragma unroll
      for (int r = 0; r < NR; r++) acc[r] += w * a.q[(size_t)(rhs0 + r) * N + j];
    }
  }
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const size_t o = (size_t)(rhs0 + r) * N + i;
    a.phi[o] += (a.potential ? (real)1 : a.q[o]) * acc[r];
  }
}

// The same for one vector, the sources read as (x, y, z, q) in one load.
__global__ void __launch_bounds__(256) k_p2p_lane_pq(P2PArgs a, int rhs)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.N) return;
  const int lf = a.leafof[i];
  const real4 x = a.pq[i];
  const int nn = a.nnbr[lf];
  const int *nb = a.nbr + (size_t)lf * 27;
  real acc = 0;
  // the next neighbour's range is fetched while this one's sources are summed
  int Bn = nb[0];  // nn >= 1: the leaf itself
  int j0n = a.leafsta[Bn], cn = a.leafcnt[Bn];
  for (int b = 0; b < nn; b++) {
    const int j0 = j0n, j1 = j0 + cn;
    if (b + 1 < nn) {
      Bn = nb[b + 1];
      j0n = a.leafsta[Bn];
      cn = a.leafcnt[Bn];
    }
    for (int j = j0; j < j1; j++) {
      const real4 y = a.pq[j];
      const real dx = y.x - x.x, dy = y.y - x.y, dz = y.z - x.z;
      const real rr = dx * dx + dy * dy + dz * dz;
      const real w = rr != (real)0 ? rsqrt_r(rr) : (real)0;
      acc += w * y.w;
    }
  }
  const size_t o = (size_t)rhs * a.N + i;
  a.phi[o] += (a.potential ? (real)1 : x.w) * acc;
}

// pq[i] = (pos[i].xyz, q[rhs][i])
__global__ void k_pack_pq(int N, const real4 *__restrict__ pos, const real *__restrict__ q, real4 *__restrict__ pq)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  real4 v = pos[i];
  v.w = q[i];
  pq[i] = v;
}

// ---------------------------------------------------------------- 1 to 8 vectors
// A wavefront's lanes are 16 targets x 4 source groups (fp64: 8 x 8): group h
// takes the staged sources h, h + 4, ... for up to NTMAX tiles of targets of the
// leaf, so that leaves of a few dozen particles keep the lanes busy (a lane a
// target left half of them idle at 33 to 48 particles) and every source read
// from LDS serves NT targets.  The groups' sums are added across lanes at the
// end.  The W waves of a block take the neighbour leaves in turn, their sums
// added through LDS; the target tiles of a leaf go to gridDim.y blocks, so
// that few large leaves fill the chip too.  Each wave stages up to kP2PLeaves
// leaves (64 sources of each) at a time in its own part of LDS, their loads
// in flight together, padded to a multiple of 8 (16) with sources of zero charge
// outside the root cell (no tail masks; copies of a leaf's last particle, as the
// 16-vector layout has, cost 64K particles 1.5 us here).  The r != 0 test is
// applied in the self leaf, which wave 0 stages by itself.
// Bound by the vector ALUs (7 + NR fp32 operations and a reciprocal square
// root a pair; fp64: rsqrt_r).  N = 1M, depth 5, one vector: 467 -> 244
// us (45 cycles of a SIMD per 64 pairs of whole tiles; the operations alone
// measure 37); 4096, depth 2 (64 leaves of 64): 192 -> 11.7 us; 65536, depth
// 4: 33 -> 21.5 us; fp64 100003, depth 4: 117 -> 57.6 us; 4 vectors of 150001
// on a sphere, depth 5: 249 -> 85 us.
constexpr int kP2PLeaves = 4;  // leaves staged together
constexpr int kP2PStage = 64 * kP2PLeaves;
// Targets of a tile.  fp64: 8 leave fewer lanes without a target, 100003
// particles, depth 4, 66.9 -> 57.6 us, 500000, depth 5, 206 -> 191; fp32 gains
// nothing (1M 246 and 246, 65536 20.6 and 22.4), its pairs being cheap against
// the staged sources' padding to 16 and the longer sums across lanes.
constexpr int kTile = sizeof(real) == 4 ? 16 : 8;
constexpr int kGroups = 64 / kTile;    // source groups

typedef real realx4 __attribute__((ext_vector_type(4)));

// position and, for one vector, charge of the staged sources; more charges beside them
template <int NR>
struct P2PStage {
  realx4 s[kP2PStage];
  real q[NR > 1 ? kP2PStage : 1][NR] __attribute__((aligned(16)));
};

// acc += the sums over the n2 (a multiple of 2 kGroups) staged sources, two of a lane's at a time
template <int NR, int NT, bool SELF>
__device__ __forceinline__ void p2p_sweep(const P2PStage<NR> &st, int n2, int h, const realx4 *x, real (&acc)[NT][NR])
{
  for (int k = 0; k < n2; k += 2 * kGroups) {
    realx4 z[2];
    real q[2][NR];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      z[u] = st.s[k + kGroups * u + h];
#pragma unroll
      for (int r = 0; r < NR; r++) q[u][r] = NR > 1 ? st.q[k + kGroups * u + h][r] : z[u].w;
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const real dx = z[u].x - x[t].x, dy = z[u].y - x[t].y, dz = z[u].z - x[t].z;
        const real rr = dx * dx + dy * dy + dz * dz;
        const real g = SELF && rr == (real)0 ? (real)0 : rsqrt_r(rr);
#pragma unroll
        for (int r = 0; r < NR; r++) acc[t][r] += g * q[u][r];
      }
  }
}

template <int NR, int NT>
__device__ __forceinline__ void p2p_tiles(const P2PArgs &a, int rhs0, int nv, int leaf, int tb, int sta, int cnt,
                                          int nsta, int ncnt, int nn, P2PStage<NR> &st, real *red)
{
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), W = blockDim.x >> 6;
  const int ti = lane % kTile, h = lane / kTile;
  const size_t N = a.N;
  const realx4 *pos = reinterpret_cast<const realx4 *>(a.pos);
  realx4 x[NT];
  real acc[NT][NR];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    x[t] = pos[sta + min(tb + kTile * t + ti, cnt - 1)];  // targets past the leaf's end are not stored
#pragma unroll
    for (int r = 0; r < NR; r++) acc[t][r] = 0;
  }
  // source `at` of the staged ones (lanes below n) from particle j + lane
  auto load = [&](int j, int n, realx4 &p, real (&q)[NR]) {
    const int i = j + min(lane, n - 1);
    p = pos[i];
#pragma unroll
    for (int r = 0; r < NR; r++) q[r] = r < nv ? a.q[(size_t)(rhs0 + r) * N + i] : (real)0;
  };
  auto put = [&](int at, int n, const realx4 &p, const real (&q)[NR]) {
    if (lane < n) {
      realx4 v = p;
      v.w = q[0];
      st.s[at + lane] = v;
      if (NR > 1)
#pragma unroll
        for (int r = 0; r < NR; r++) st.q[at + lane][r] = q[r];
    }
  };
  auto pad = [&](int n) {  // to a multiple of 2 kGroups
    const int n2 = (n + 2 * kGroups - 1) & ~(2 * kGroups - 1);
    if (lane < n2 - n) {
      st.s[n + lane] = realx4{a.beyond, a.beyond, a.beyond, 0};
      if (NR > 1)
#pragma unroll
        for (int r = 0; r < NR; r++) st.q[n + lane][r] = 0;
    }
    return n2;
  };
  if (wave == 0) {  // the leaf itself
    for (int j = 0; j < cnt; j += 64) {
      const int n = min(64, cnt - j);
      realx4 p;
      real q[NR];
      load(sta + j, n, p, q);
      put(0, n, p, q);
      const int n2 = pad(n);
      wave_sync();
      p2p_sweep<NR, NT, true>(st, n2, h, x, acc);
      wave_sync();
    }
  }
  // the other leaves: items (leaf b, 64 sources from j) of this wave
  int b = wave, j = 0;
  while (b < nn) {
    realx4 p[kP2PLeaves];
    real q[kP2PLeaves][NR];
    int n[kP2PLeaves];
#pragma unroll
    for (int g = 0; g < kP2PLeaves; g++) {
      // (an empty leaf, the leaf itself: a step without sources)
      n[g] = 0;
      if (b < nn) {
        const int c = __builtin_amdgcn_readlane(ncnt, b);
        n[g] = min(64, c - j);
        if (n[g] > 0) load(__builtin_amdgcn_readlane(nsta, b) + j, n[g], p[g], q[g]);
        j += 64;
        if (j >= c) {
          j = 0;
          b += W;
        }
      }
    }
    int at = 0;
#pragma unroll
    for (int g = 0; g < kP2PLeaves; g++)
      if (n[g] > 0) {
        put(at, n[g], p[g], q[g]);
        at += n[g];
      }
    if (at > 0) {
      const int n2 = pad(at);
      wave_sync();
      p2p_sweep<NR, NT, false>(st, n2, h, x, acc);
      wave_sync();
    }
  }
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int r = 0; r < NR; r++) {
      for (int k = kTile; k < 64; k <<= 1) acc[t][r] += __shfl_xor(acc[t][r], k);
    }
  if (W > 1) {
    __syncthreads();  // the previous pass's sums have been read
    if (h == 0)
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < NR; r++) red[((wave * NT + t) * NR + r) * kTile + ti] = acc[t][r];
    __syncthreads();
    if (wave > 0) return;
    for (int w = 1; w < W; w++)
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < NR; r++) acc[t][r] += red[((w * NT + t) * NR + r) * kTile + ti];
  }
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int i = tb + kTile * t + ti;
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const size_t o = (size_t)(rhs0 + r) * N + sta + i;
      if (i < cnt && r < nv && (r & (kGroups - 1)) == h) {
        const real v = a.phi[o] + (a.potential ? (real)1 : a.q[o]) * acc[t][r];
        if (a.out) a.out[(size_t)(rhs0 + r) * N + a.perm[sta + i]] = v;
        else a.phi[o] = v;
      }
    }
  }
}

// vectors rhs0 .. rhs0 + nv - 1 (nv <= NR)
template <int NR, int NTMAX, int MAXW>
__global__ void __launch_bounds__(64 * MAXW) k_p2p(P2PArgs a, int rhs0, int nv)
{
  __shared__ P2PStage<NR> stage[MAXW];
  __shared__ real red[MAXW > 1 ? MAXW * NTMAX * NR * kTile : 1];
  const int leaf = xcd_leaf(blockIdx.x, a.nleaf);
  const int lane = threadIdx.x & 63;
  const int sta = a.leafsta[leaf], cnt = a.leafcnt[leaf], nn = a.nnbr[leaf];
  int nsta = 0, ncnt = 0;  // lane b: neighbour leaf b (the leaf itself without sources)
  if (lane < nn) {
    const int B = a.nbr[(size_t)leaf * 27 + lane];
    nsta = a.leafsta[B];
    ncnt = B == leaf ? 0 : a.leafcnt[B];
  }
  P2PStage<NR> &st = stage[threadIdx.x >> 6];
  // passes of NTMAX tiles, dealt to the gridDim.y blocks
  for (int tb = blockIdx.y * kTile * NTMAX; tb < cnt; tb += gridDim.y * kTile * NTMAX) {
    const int nt = min(NTMAX, (cnt - tb + kTile - 1) / kTile);
    auto run = [&](auto k) {
      constexpr int NT = decltype(k)::value;
      if constexpr (NT <= NTMAX)
        p2p_tiles<NR, NT>(a, rhs0, nv, leaf, tb, sta, cnt, nsta, ncnt, nn, st, red);
    };
    switch (nt) {
    case 1: run(std::integral_constant<int, 1>()); break;
    case 2: run(std::integral_constant<int, 2>()); break;
    case 3: run(std::integral_constant<int, 3>()); break;
    case 4: run(std::integral_constant<int, 4>()); break;
    case 5: run(std::integral_constant<int, 5>()); break;
    default: run(std::integral_constant<int, 6>()); break;
    }
  }
}

#ifdef SINGLE
typedef float f32x4 __attribute__((ext_vector_type(4)));

#endif

// ---------------------------------------------------------------- padded layout
// The kernel below reads a private copy of the particles in which every
// leaf's range starts at a multiple of 4 and is padded to a multiple of 4
// with copies of its last particle of zero charge, so that its source loops
// need no tail masks.  seg[leaf][0..nseg) lists the
// (padded start, padded count) of the leaf's non-empty neighbours, the leaf
// itself first.  Targets are read from the same copy; dummy targets are
// never written.

#ifdef SINGLE
template <int NT>
__device__ __forceinline__ void p2p16_step(const float4 &z, float bq, const float4 *x, f32x4 *acc)
{
  float g[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const float dx = z.x - x[t].x, dy = z.y - x[t].y, dz = z.z - x[t].z;
    g[t] = __builtin_amdgcn_rsqf(dx * dx + dy * dy + dz * dz);
  }
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(bq, g[t], acc[t], 0, 0, 0);
}

// results of NT target tiles of the transposed product (lane l holds the
// vectors 4 (l / 16) .. 4 (l / 16) + 3 of target tb + 16 t + l % 16) added
// into phi (q * potential, or the potential), the particle rows (one
// 16-byte piece of a row per lane), or the near rows
template <int NT>
__device__ __forceinline__ void p2p16_store_t(const P2PArgs &a, int rhs0, int sta, int cnt, int psta, int tb,
                                              const f32x4 *acc)
{
  const int l = threadIdx.x & 63;
  const int ti = l & 15, kq = l >> 4;
  if (a.phin) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int i = tb + 16 * t + ti;
      if (i < cnt) *reinterpret_cast<f32x4 *>(a.phin + (size_t)(psta + i) * 16 + 4 * kq) = acc[t];
    }
    return;
  }
  if (a.phit) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int i = tb + 16 * t + ti;
      if (i < cnt) {
        const size_t o = (size_t)(psta + i) * 16 + 4 * kq;
        const f32x4 far = *reinterpret_cast<const f32x4 *>(a.phit + o);
        const f32x4 q = a.potential ? f32x4{1.f, 1.f, 1.f, 1.f} : *reinterpret_cast<const f32x4 *>(a.qt + o);
        *reinterpret_cast<f32x4 *>(a.phit + o) = q * (far + acc[t]);
      }
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int i = tb + 16 * t + ti;
    if (i < cnt)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const size_t o = (size_t)(rhs0 + 4 * kq + e) * a.N + sta + i;
        a.phi[o] += (a.potential ? 1.0f : a.q[o]) * acc[t][e];
      }
  }
}

// results of NT target tiles (accumulator layout of the 16x16 MFMA: lane l
// holds targets tb + 16 t + 4 (l / 16) + v, vector l % 16) added into phi
// (q * potential, or the potential), the particle rows, or the near rows
template <int NT>
__device__ __forceinline__ void p2p16_store(const P2PArgs &a, int rhs0, int sta, int cnt, int psta, int tb,
                                            const f32x4 *acc)
{
  const int l = threadIdx.x;
  const int ti = l & 15, kq = l >> 4;
  const float *Qt = a.qt;
  if (a.phin) {
    // particle rows of their own: the near-field potential
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int i = tb + 16 * t + 4 * kq + v;
        if (i < cnt) a.phin[(size_t)(psta + i) * 16 + ti] = acc[t][v];
      }
    return;
  }
  if (a.phit) {
    // particle rows: far field + near field, then the output's q factor
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int i = tb + 16 * t + 4 * kq + v;
        const size_t o = (size_t)(psta + i) * 16 + ti;
        if (i < cnt) a.phit[o] = (a.potential ? 1.0f : Qt[o]) * (a.phit[o] + acc[t][v]);
      }
    return;
  }
  const size_t row = (size_t)(rhs0 + ti) * a.N + sta;
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int i = tb + 16 * t + 4 * kq + v;
      if (i < cnt) a.phi[row + i] += (a.potential ? 1.0f : a.q[row + i]) * acc[t][v];
    }
}

// One pass over all sources for NT tiles of 16 targets starting at target
// tb of the leaf; results added into phi (q * potential, or the potential).
// BUF: the source positions and charge rows are read with buffer loads whose
// group offset is a scalar register (the padded arrays then stay below 2 GB),
// so no vector instructions go into the per-group addresses.
template <int NT, bool BUF, int W>
__device__ __forceinline__ void p2p16_pass(const P2PArgs &a, int rhs0, int2 sg, int nseg, int T, int sta,
                                           int cnt, int psta, int pself, int tb, f32x4 *red)
{
  const int l = threadIdx.x & 63;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  const int ti = l & 15, kq = l >> 4;
  const float4 *P = reinterpret_cast<const float4 *>(a.ppos);
  const float *Qt = a.qt;
  const int qoff = kq * 16 + ti;
  const __amdgpu_buffer_rsrc_t rP = __builtin_amdgcn_make_buffer_rsrc((void *)a.ppos, 0, a.npad * 16, 0x00020000);
  const __amdgpu_buffer_rsrc_t rQ = __builtin_amdgcn_make_buffer_rsrc((void *)a.qt, 0, a.npad * 64, 0x00020000);
  // source group at padded index p: lane l reads the position of source p + l / 16 and its charge of vector l % 16
  auto src_pos = [&](int p) -> float4 {
    if (BUF) return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rP, kq * 16, p * 16, 0));
    return P[p + kq];
  };
  auto src_q = [&](int p) -> float {
    if (BUF) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rQ, qoff * 4, p * 64, 0));
    return Qt[(size_t)p * 16 + qoff];
  };
  float4 x[NT];
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    x[t] = P[psta + min(tb + 16 * t + ti, cnt - 1)];
    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the self leaf (r != 0 exclusion), loaded one group ahead
  auto self_step = [&](const float4 &z, float bq) {
    float g[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const float dx = z.x - x[t].x, dy = z.y - x[t].y, dz = z.z - x[t].z;
      const float rr = dx * dx + dy * dy + dz * dz;
      g[t] = rr != 0.f ? __builtin_amdgcn_rsqf(rr) : 0.f;
    }
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(bq, g[t], acc[t], 0, 0, 0);
  };
  if (pself > 0 && wave == 0) {
    float4 zA = src_pos(psta);
    float qA = src_q(psta);
    for (int k = 0; k < pself; k += 8) {
      const int k1 = min(k + 4, pself - 4);
      const float4 zB = src_pos(psta + k1);
      const float qB = src_q(psta + k1);
      self_step(zA, qA);
      if (k + 4 >= pself) break;
      const int k2 = min(k + 8, pself - 4);
      zA = src_pos(psta + k2);
      qA = src_q(psta + k2);
      self_step(zB, qB);
    }
  }
  // this wave's groups of the other leaves (W > 1: the first wave, which has
  // the self leaf too, takes the fewer)
  const int T0 = W > 1 ? max(0, (int)((T + (pself >> 2)) * wave / W) - (pself >> 2)) : 0;
  const int Tn = (W > 1 ? max(0, (int)((T + (pself >> 2)) * (wave + 1) / W) - (pself >> 2)) : T) - T0;
  if (Tn > 0) {
    int b = 1;
    int pos = __builtin_amdgcn_readlane(sg.x, 1);
    int end = pos + __builtin_amdgcn_readlane(sg.y, 1);
    if (W > 1) {
      int skip = 4 * T0;
      while (skip >= end - pos) {
        skip -= end - pos;
        b++;
        pos = __builtin_amdgcn_readlane(sg.x, b);
        end = pos + __builtin_amdgcn_readlane(sg.y, b);
      }
      pos += skip;
    }
    // next group; stays on the last group at the end (loaded, never summed)
    auto advance = [&]() {
      if (pos + 4 < end) {
        pos += 4;
      } else if (b + 1 < nseg) {
        b++;
        pos = __builtin_amdgcn_readlane(sg.x, b);
        end = pos + __builtin_amdgcn_readlane(sg.y, b);
      }
    };
    // four groups in flight: a ring of four register sets, loaded three
    // groups ahead (the loop is unrolled so that no set is copied)
    float4 y0, y1, y2, y3;
    float q0, q1, q2, q3;
    auto load = [&](float4 &y, float &q) {
      y = src_pos(pos);
      q = src_q(pos);
      advance();
    };
    load(y0, q0);
    load(y1, q1);
    load(y2, q2);
    for (int t = 0; t < Tn; t += 4) {
      load(y3, q3);
      p2p16_step<NT>(y0, q0, x, acc);
      if (t + 1 >= Tn) break;
      load(y0, q0);
      p2p16_step<NT>(y1, q1, x, acc);
      if (t + 2 >= Tn) break;
      load(y1, q1);
      p2p16_step<NT>(y2, q2, x, acc);
      if (t + 3 >= Tn) break;
      load(y2, q2);
      p2p16_step<NT>(y3, q3, x, acc);
    }
  }
  if (W > 1) {
    __syncthreads();  // the previous pass's sums have been read
    if (wave > 0)
#pragma unroll
      for (int t = 0; t < NT; t++) red[((wave - 1) * NT + t) * 64 + l] = acc[t];
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int t = 0; t < NT; t++)
      for (int w = 0; w < W - 1; w++) acc[t] += red[(w * NT + t) * 64 + l];
  }
  p2p16_store_t<NT>(a, rhs0, sta, cnt, psta, tb, acc);
}

// Sixteen vectors on MFMA; qt is [padded N][16].  Lane l computes
// G[target l%16 of each 16-target tile][source 4j + l/16] and feeds it as the
// B operand, the charges of that source for vector l%16 as the A operand
// (the transposed product: a lane ends with four consecutive vectors of one
// target, stored as one 16-byte piece of its row).  The self leaf is
// summed first with the r != 0 exclusion; the other neighbours form one
// flattened sequence of 4-source groups, loaded three groups ahead into a
// ring of four register sets.  Up to ntp target tiles share a pass; the
// passes are dealt to gridDim.y blocks, and the W waves of a block take equal
// parts of the groups, their sums added through LDS.
template <bool BUF, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(W > 4 ? 5 : W > 1 ? 6 : 7)))
    k_p2p_seg16(P2PArgs a, int rhs0, int ntp)
{
  __shared__ f32x4 red[W > 1 ? (W - 1) * 4 * 64 : 1];
  const int leaf = xcd_leaf(blockIdx.x, a.nleaf);
  const int l = threadIdx.x & 63;
  const int sta = a.leafsta[leaf], cnt = a.leafcnt[leaf];
  // as few passes of equal tiles as ntp allows
  const int tiles = (cnt + 15) >> 4, np = W > 1 ? (tiles + ntp - 1) / ntp : 1;
  if (cnt == 0 || (int)blockIdx.y >= np) return;
  const int nseg = a.nseg[leaf];
  const int2 sg = l < nseg ? a.seg[(size_t)leaf * 27 + l] : make_int2(0, 0);
  const int psta = __builtin_amdgcn_readfirstlane(sg.x);
  const int pself = __builtin_amdgcn_readfirstlane(sg.y);
  int T = 0;
  for (int b = 1; b < nseg; b++) T += __builtin_amdgcn_readlane(sg.y, b) >> 2;
  if (W == 1) {  // all passes here, up to 4 tiles each
    for (int tb = 0; tb < cnt;) {
      const int nt = (cnt - tb + 15) >> 4;
      if (nt >= 4) {
        p2p16_pass<4, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
        tb += 64;
      } else if (nt == 3) {
        p2p16_pass<3, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
        tb += 48;
      } else if (nt == 2) {
        p2p16_pass<2, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
        tb += 32;
      } else {
        p2p16_pass<1, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
        tb += 16;
      }
    }
    return;
  }
  for (int p = blockIdx.y; p < np; p += gridDim.y) {
    const int t0 = tiles * p / np, nt = tiles * (p + 1) / np - t0, tb = 16 * t0;
    if (nt >= 4) p2p16_pass<4, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
    else if (nt == 3) p2p16_pass<3, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
    else if (nt == 2) p2p16_pass<2, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
    else p2p16_pass<1, BUF, W>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb, red);
  }
}

// ------------------------------------------------ split-BF16 accumulation
// On gfx950 the FP32 MFMA and the FP32 vector ALU of a SIMD do not run at the
// same time, so in k_p2p_seg16 the 1/r work and the MFMA accumulation (32
// cycles per 64 pairs) add up.  Here G = 1/r (fp32) and the charges are each
// split into bf16 hi + lo parts and the sum over sources takes three
// products (hi*hi + hi*lo + lo*hi) of v_mfma_f32_16x16x16_bf16: 16 targets x
// 16 sources x 16 vectors per product, fp32 accumulation.  The relative
// error of one term is below 3 * 2^-16 (the dropped lo*lo and the rounding of
// the lo parts).
#ifdef SINGLE
typedef __bf16 bf16x4p __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2p __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x3 __attribute__((ext_vector_type(3)));

// two fp32 values -> their bf16 hi parts (round to nearest even) and the
// bf16 of the remainders, each pair in one conversion
__device__ __forceinline__ void split2(float g0, float g1, unsigned &h, unsigned &lo)
{
  h = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{g0, g1}, bf16x2p));
  const float h0 = __builtin_bit_cast(float, h << 16), h1 = __builtin_bit_cast(float, h & 0xffff0000u);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{g0 - h0, g1 - h1}, bf16x2p));
}

// qt [Npad][16] -> hi and lo parts at [padded source / 4][vector][4 sources]
__global__ void k_split_q16(int ngroups, const float *__restrict__ qt, bf16x4p *__restrict__ qh,
                            bf16x4p *__restrict__ ql)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;  // (group of 4 sources, vector)
  if (i >= ngroups * 16) return;
  const int g = i >> 4, v = i & 15;
  bf16x4p h, lo;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float x = qt[(size_t)(4 * g + e) * 16 + v];
    h[e] = (__bf16)x;
    lo[e] = (__bf16)(x - (float)h[e]);
  }
  qh[i] = h;
  ql[i] = lo;
}

typedef short i16x4 __attribute__((ext_vector_type(4)));

// One pass over all sources for NT tiles of 16 targets starting at target tb.
// A step takes 4 groups of 4 sources: lane l (target l % 16 of each tile)
// computes G for group l / 16 of the step, whose 4 sources are also its
// k-slots in the A and B operands, so no data moves between lanes.  The self
// leaf's groups are contiguous; the neighbours' groups follow the segment
// table in the order of k_p2p_seg16, walked with scalar registers, two steps
// in flight.  Groups past the end take the last group's position with zero
// charges.
template <int NT>
__device__ __forceinline__ void p2p16x_pass(const P2PArgs &a, int rhs0, int2 sg, int nseg, int T, int sta, int cnt,
                                            int psta, int pself, int tb)
{
  const int l = threadIdx.x;
  const int ti = l & 15, kq = l >> 4;
  const float4 *P = reinterpret_cast<const float4 *>(a.ppos);
  const __amdgpu_buffer_rsrc_t rP = __builtin_amdgcn_make_buffer_rsrc((void *)a.ppos, 0, a.npad * 16, 0x00020000);
  const __amdgpu_buffer_rsrc_t rH = __builtin_amdgcn_make_buffer_rsrc(a.qsh, 0, a.npad * 32, 0x00020000);
  const __amdgpu_buffer_rsrc_t rL = __builtin_amdgcn_make_buffer_rsrc(a.qsl, 0, a.npad * 32, 0x00020000);
  float4 x[NT];
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    x[t] = P[psta + min(tb + 16 * t + ti, cnt - 1)];
    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the lane's group at padded position pa (x, y, z of its 4 sources and
  // their hi / lo charges of vector ti); va: it counts
  struct Src {
    f32x3 y[4];
    i16x4 h, lo;
  };
  auto load = [&](Src &u, int pa, bool va) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      u.y[e] = __builtin_bit_cast(f32x3, __builtin_amdgcn_raw_buffer_load_b96(rP, (pa + e) * 16, 0, 0));
    const int oa = ((pa >> 2) * 16 + ti) * 8;
    u.h = __builtin_bit_cast(i16x4, __builtin_amdgcn_raw_buffer_load_b64(rH, oa, 0, 0));
    u.lo = __builtin_bit_cast(i16x4, __builtin_amdgcn_raw_buffer_load_b64(rL, oa, 0, 0));
    const i16x4 z = {};
    if (!va) u.h = u.lo = z;
  };
  auto step = [&](const Src &u, bool self) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      float g[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float dx = u.y[e].x - x[t].x, dy = u.y[e].y - x[t].y, dz = u.y[e].z - x[t].z;
        const float rr = dx * dx + dy * dy + dz * dz;
        g[e] = __builtin_amdgcn_rsqf(rr);
        if (self) g[e] = rr != 0.f ? g[e] : 0.f;
      }
      unsigned hw[2], lw[2];
      split2(g[0], g[1], hw[0], lw[0]);
      split2(g[2], g[3], hw[1], lw[1]);
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      const i16x4 gh = __builtin_bit_cast(i16x4, u32x2{hw[0], hw[1]});
      const i16x4 gl = __builtin_bit_cast(i16x4, u32x2{lw[0], lw[1]});
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gh, u.h, acc[t], 0, 0, 0);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gh, u.lo, acc[t], 0, 0, 0);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(gl, u.h, acc[t], 0, 0, 0);
    }
  };
  // self leaf: groups 0 .. pself/4 - 1 from psta
  const int gs = pself >> 2;
  for (int g0 = 0; g0 < gs; g0 += 4) {
    const int ga = g0 + kq;
    Src u;
    load(u, psta + 4 * min(ga, gs - 1), ga < gs);
    step(u, true);
  }
  if (T > 0) {
    int b = 1;
    int pos = __builtin_amdgcn_readlane(sg.x, 1);
    int end = pos + __builtin_amdgcn_readlane(sg.y, 1);
    // next group; stays on the last group at the end
    auto advance = [&]() {
      if (pos + 4 < end) {
        pos += 4;
      } else if (b + 1 < nseg) {
        b++;
        pos = __builtin_amdgcn_readlane(sg.x, b);
        end = pos + __builtin_amdgcn_readlane(sg.y, b);
      }
    };
    // the 4 group positions of the next step, the lane's picked out
    auto next = [&](Src &u, int g0) {
      int p[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        p[j] = pos;
        advance();
      }
      const int pa = kq == 0 ? p[0] : kq == 1 ? p[1] : kq == 2 ? p[2] : p[3];
      load(u, pa, g0 + kq < T);
    };
    Src u0, u1;
    next(u0, 0);
    for (int g0 = 0; g0 < T; g0 += 8) {
      if (g0 + 4 < T) next(u1, g0 + 4);
      step(u0, false);
      if (g0 + 4 >= T) break;
      if (g0 + 8 < T) next(u0, g0 + 8);
      step(u1, false);
    }
  }
  p2p16_store<NT>(a, rhs0, sta, cnt, psta, tb, acc);
}

// k_p2p_seg16 with the split-BF16 accumulation; qsh / qsl filled from qt.
// At most NTMAX target tiles per pass: the registers of a kernel are those of
// its largest pass (NTMAX = 3: 80 VGPRs, 6 waves per SIMD; NTMAX = 4: 100).
template <int NTMAX>
__global__ void __launch_bounds__(64) k_p2p_seg16x(P2PArgs a, int rhs0)
{
  const int leaf = xcd_leaf(blockIdx.x, a.nleaf);
  const int l = threadIdx.x;
  const int sta = a.leafsta[leaf], cnt = a.leafcnt[leaf];
  if (cnt == 0) return;
  const int nseg = a.nseg[leaf];
  const int2 sg = l < nseg ? a.seg[(size_t)leaf * 27 + l] : make_int2(0, 0);
  const int psta = __builtin_amdgcn_readfirstlane(sg.x);
  const int pself = __builtin_amdgcn_readfirstlane(sg.y);
  int T = 0;
  for (int b = 1; b < nseg; b++) T += __builtin_amdgcn_readlane(sg.y, b) >> 2;
  for (int tb = 0; tb < cnt;) {
    const int tiles = min((cnt - tb + 15) >> 4, NTMAX);
    if (NTMAX >= 4 && tiles >= 4) {
      p2p16x_pass<NTMAX >= 4 ? 4 : 1>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb);
      tb += 64;
    } else if (NTMAX >= 3 && tiles == 3) {
      p2p16x_pass<NTMAX >= 3 ? 3 : 1>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb);
      tb += 48;
    } else if (tiles == 2) {
      p2p16x_pass<2>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb);
      tb += 32;
    } else {
      p2p16x_pass<1>(a, rhs0, sg, nseg, T, sta, cnt, psta, pself, tb);
      tb += 16;
    }
  }
}
#endif

// charges of vectors rhs0..rhs0+15, leaf order [16][N] -> padded [Npad][16]
__global__ void k_pad_charges16(int N, const int *__restrict__ pad_of, const float *__restrict__ q,
                                float *__restrict__ qt)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  float4 *o = reinterpret_cast<float4 *>(qt + (size_t)pad_of[i] * 16);
#pragma unroll
  for (int r = 0; r < 16; r += 4)
    o[r / 4] = make_float4(q[(size_t)r * N + i], q[(size_t)(r + 1) * N + i], q[(size_t)(r + 2) * N + i],
                           q[(size_t)(r + 3) * N + i]);
}
#endif

template <int NR, int NTMAX, int W>
static void p2p_few_t(const P2PArgs &a, int rhs, int nv, hipStream_t s)
{
  hipLaunchKernelGGL((k_p2p<NR, NTMAX, W>), dim3(a.nleaf, 4), dim3(64 * W), 0, s, a, rhs, nv);
}

// Tiles of a pass and waves of a block.  Many leaves fill the chip with a
// wave each, and more tiles a pass read fewer staged sources per pair; few
// leaves need their sources split over waves, as far as the waves' LDS leaves
// room for enough of them.  The target tiles of a leaf are dealt to 4 blocks
// (those without tiles end at once): N = 50000, 512 leaves 42.9 against 52.5
// us on one block, surface 150001 85 against 130.  P2P in us, tiles x waves:
//   fp32, 1 vector:  1M, 32768 leaves 4x1 244, 4x4 262; 262144, 4096 leaves
//                    4x4 118, 4x1 123; 65536, 4096 leaves 2x4 21.5, 4x1 24.8;
//                    50000, 512 leaves 2x8 42.9, 2x4 47.1; 4096, 64 leaves
//                    2x8 11.7, 2x4 14.5, 4x8 15.1
//   fp32, 4 vectors: 262144 4x4 170.5, 4x1 171.9; 65536 2x1 33.6, 2x4 39.7;
//                    50000 2x4 63.4, 2x8 65.8; 4096 2x8 15.2, 2x4 19.1
//   fp32, 7 vectors: 1M 4x1 524, 2x1 633; 16384, 512 leaves 2x4 24.1
//   fp32, 16 vectors of the plain form, as two times 8 (all 16 at once, a lane
//                    a target: in brackets): 4096 51 (547), 65536 114 (109),
//                    262144 490 (1082), 1M 1112 (1585)
//   fp64:            100003, 4096 leaves, 1 vector 4x4 57.4, 4x1 57.6, 4
//                    vectors 4x1 95.1, 4x4 134; 500000, 32768 leaves, 1
//                    vector 4x1 191, 4x4 275; 8000, 64 leaves, 1 vector 6x4
//                    38.6, 4x4 45.7, 4x1 111; 40000, 512 leaves, 4 vectors 6x4
//                    97.5, 4x4 101, 4x1 117
template <int NR>
static void p2p_few_n(const P2PArgs &a, int rhs, int nv, hipStream_t s)
{
#ifdef SINGLE
  if (a.nleaf <= 1024) {
    if (NR == 1 || (NR < 8 && a.nleaf <= 128)) p2p_few_t<NR, 2, NR < 8 ? 8 : 4>(a, rhs, nv, s);
    else p2p_few_t<NR, 2, 4>(a, rhs, nv, s);
  } else if (a.N > 24LL * a.nleaf) {
    if (NR == 1 && a.nleaf <= 6144) p2p_few_t<NR, 4, NR == 1 ? 4 : 1>(a, rhs, nv, s);
    else p2p_few_t<NR, 4, 1>(a, rhs, nv, s);
  } else {
    if (NR == 1 && a.nleaf <= 6144) p2p_few_t<NR, 2, 4>(a, rhs, nv, s);
    else p2p_few_t<NR, 2, 1>(a, rhs, nv, s);
  }
#else
  if (a.nleaf <= (NR < 8 ? 1024 : 128)) p2p_few_t<NR, NR < 8 ? 6 : 4, 4>(a, rhs, nv, s);
  else if (NR == 1 && a.nleaf <= 6144) p2p_few_t<NR, 4, 4>(a, rhs, nv, s);
  else p2p_few_t<NR, 4, 1>(a, rhs, nv, s);
#endif
}

// nv (1 to 8) vectors from rhs
static void p2p_few(const P2PArgs &a, int rhs, int nv, hipStream_t s)
{
  if (nv > 4) p2p_few_n<8>(a, rhs, nv, s);
  else if (nv > 2) p2p_few_n<4>(a, rhs, nv, s);
  else if (nv == 2) p2p_few_n<2>(a, rhs, nv, s);
  else p2p_few_n<1>(a, rhs, nv, s);
}

#ifdef SINGLE
template <bool BUF, int W>
static void p2p_seg16_t(const P2PArgs &a, int rhs, int ntp, hipStream_t s)
{
  hipLaunchKernelGGL((k_p2p_seg16<BUF, W>), dim3(a.nleaf, W > 1 ? 4 : 1), dim3(64 * W), 0, s, a, rhs, ntp);
}

// Tiles of a pass and waves of a block of the 16-vector near field, as for
// few vectors.  Many leaves fill the chip with a wave each and are spared the
// blocks without tiles.  Less than 8
// particles a leaf on average means that most are empty (a surface) and the
// others are large.  P2P in us, tiles x waves (4 blocks a leaf), and one wave
// a leaf of up to 4 tiles before:
//   4096, 64 leaves 2x8 16.3, 2x4 21.1 (118); 50021, 512 leaves 2x4 78.7, 4x4
//   86.0 (265); 262144, 4096 leaves 4x4 233, 4x2 235 (350); 131072 4x4 78.2
//   (106); 65536 4x4 36.1, 4x2 35.8 (44.6); 1M, 32768 leaves 4x1 490 (4 blocks
//   502), 4x2 504; 150001 on a sphere, 32768 leaves 4x4 85.1, 4x2 97.8 (201)
template <bool BUF>
static void p2p_seg16(const P2PArgs &a, int rhs, hipStream_t s)
{
  if (a.nleaf <= 128) p2p_seg16_t<BUF, 8>(a, rhs, 2, s);
  else if (a.nleaf <= 1024) p2p_seg16_t<BUF, 4>(a, rhs, 2, s);
  else if (a.nleaf <= 8192 || a.N < 8LL * a.nleaf) p2p_seg16_t<BUF, 4>(a, rhs, 4, s);
  else p2p_seg16_t<BUF, 1>(a, rhs, 4, s);
}
#endif

int launch_p2p(const P2PArgs &a, hipStream_t s)
{
  if (a.nleaf <= 0 || a.N <= 0) return BBFMM_OK;
  int rhs = 0;
  const bool lane = a.leafof && !a.phit && !a.phin;  // a lane per target particle
#ifdef SINGLE
  const bool mfma = a.use_mfma && a.qt && a.ppos && a.seg;  // 16 vectors at a time
#else
  const bool mfma = false;
#endif
  if (a.out && (lane || (mfma && a.nrhs >= 16)))  // these leave the sums in phi
    return set_error(BBFMM_E_ARG, "internal: near field asked to scatter by a kernel that does not");
  if (lane) {
    const int nb = (a.N + 255) / 256;
    while (rhs < a.nrhs) {
      const int left = a.nrhs - rhs;
      if (left >= 4) {
        hipLaunchKernelGGL(k_p2p_lane<4>, dim3(nb), dim3(256), 0, s, a, rhs);
        rhs += 4;
      } else if (a.pq) {
        hipLaunchKernelGGL(k_pack_pq, dim3(nb), dim3(256), 0, s, a.N, a.pos, a.q + (size_t)rhs * a.N, a.pq);
        BB_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_p2p_lane_pq, dim3(nb), dim3(256), 0, s, a, rhs);
        rhs += 1;
      } else {
        hipLaunchKernelGGL(k_p2p_lane<1>, dim3(nb), dim3(256), 0, s, a, rhs);
        rhs += 1;
      }
      BB_HIP(hipGetLastError());
    }
    return BBFMM_OK;
  }
  while (rhs < a.nrhs) {
    const int left = a.nrhs - rhs;
    if (left >= 16) {
#ifdef SINGLE
      if (mfma) {
        if (!a.phit && !a.phin) {  // particle rows arrive filled
          hipLaunchKernelGGL(k_pad_charges16, dim3((a.N + 255) / 256), dim3(256), 0, s, a.N, a.pad_of,
                             a.q + (size_t)rhs * a.N, a.qt);
          BB_HIP(hipGetLastError());
        }
        if (a.qsh && a.qsl && a.npad > 0 && a.npad < (1 << 25)) {  // split-BF16 accumulation
          const int ng = a.npad >> 2;
          hipLaunchKernelGGL(k_split_q16, dim3((ng * 16 + 255) / 256), dim3(256), 0, s, ng, a.qt,
                             (bf16x4p *)a.qsh, (bf16x4p *)a.qsl);
          BB_HIP(hipGetLastError());
          if (a.N <= 40LL * a.nleaf)  // up to about 40 particles per leaf: passes of 1 to 3 tiles
            hipLaunchKernelGGL(k_p2p_seg16x<3>, dim3(a.nleaf), dim3(64), 0, s, a, rhs);
          else
            hipLaunchKernelGGL(k_p2p_seg16x<4>, dim3(a.nleaf), dim3(64), 0, s, a, rhs);
        } else if (!a.flat && a.npad > 0 && a.npad < (1 << 25))  // charge rows below 2 GB: scalar-offset buffer loads
          p2p_seg16<true>(a, rhs, s);
        else
          p2p_seg16<false>(a, rhs, s);
      } else
#endif
        for (int v = 0; v < 16; v += 8) p2p_few(a, rhs + v, 8, s);
      rhs += 16;
    } else {
      const int nv = left < 8 ? left : 8;
      p2p_few(a, rhs, nv, s);
      rhs += nv;
    }
    BB_HIP(hipGetLastError());
  }
  return BBFMM_OK;
}

} // namespace bb
