// m2l_grid.hip -- dense-grid M2L (schemes CL and IJ).
//
// At level l (2^l cells per axis) a field cell f = 2p + s has parent p and
// sibling class s in {0,1}^3.  Its interaction list is every cell c = f + v
// whose parent is a neighbour of p (|p(c) - p|_inf <= 1) and which is not a
// neighbour of f (|v|_inf >= 2) -- 189 offsets per class, with
//   source class  s' = (s + v) mod 2,   parent shift  d = floor((s + v) / 2),
// so the sources of all class-s cells for one offset v form the class-s'
// parent grid shifted by d.  M is scattered into eight per-class parent grids
// with one ghost layer of zeros on every side; then for every class s and
// offset v
//     L_s[:, p] += K_v M_{s'}[:, p + d]      (an r x r by r x ncols product)
// which is a GEMM per (s, v) accumulated in registers -- the natural MFMA
// form.  Cells at the domain boundary read ghost zeros, so the result equals
// the list-driven M2L (anotherInteractionList.c:11-111).
//
// Columns are (parent position, right-hand side) pairs, so many charge
// vectors widen every product.  One launch covers all levels.
//
// Forms:
//   PLAIN   the build's precision on the matrix unit (fp32 or fp64 operands
//           and sums), any rank 1..512;
//   BF16X2  K and M split into bf16 hi + lo, three MFMA products
//           (hi*hi + hi*lo + lo*hi) accumulated in fp32 (fp32 build);
//   FP32    the same kernel on the vectors of the particle-row form (fp32 build);
//   FP16X3  K and M each split into three fp16 terms t1 + t2 + t3 (about 33
//           bits), six MFMA products (t1t1, t1t2, t2t1, t1t3, t2t2, t3t1)
//           accumulated in fp32 (fp32 build).  fp16 has a narrow exponent
//           range, so K is scaled by a power of two chosen from its largest
//           entry and the M of every level by one chosen from that level's
//           largest entry (measured on the device each solve); all sources
//           of a field cell lie on its level, so the product is unscaled
//           exactly in the epilogue.
// The split forms use r = 32 (one 32 x 32 output tile per 32 columns), FP32
// r = 32 and 256.
#include "common.h"
#include "kernels.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>
#include <vector>

namespace bb {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kOffsets = 189;
constexpr int kMaxLev = 10;

struct GridArgs {
  int r, nrhs, ncell, minlev, maxlev;
  int blk0[kMaxLev + 2];      // first block of each level (flattened launch)
  int lvl_slot0[kMaxLev + 1];  // first slot of each level's 8 class grids
  int levsta[kMaxLev + 2];
  const int4 *tab;  // [8][189]: (k, source class, packed shift, 0)
  const void *Ka;   // operators in the form's layout
  const void *Mg0;  // grids (hi / real)
  const void *Mg1;  // grids (lo) for BF16X2, (t2) for FP16X3
  const void *Mg2;  // grids (t3) for FP16X3
  unsigned *lvl_max;  // FP16X3: [kMaxLev + 1] bits of each level's largest |M|
  float kscale_inv;   // FP16X3: 1 / the power of two K is scaled by
  real *L;
  int wave_cols;    // columns per wave
  const int *steps;  // [class group][208][kStepWords] step records (step_table)
  int nsteps[8];     // steps of each class group
  int ss;            // source-stationary kernel: field classes per wave (8, 4 or 2); 0: not used
  int ss_tpw;        // source-stationary kernel: 32-column tiles per wave (1 or 2)
  int ss_pair;       // 1: both class groups of a column group in one block sharing source tiles
                     // (k_m2l_mfma_ss_pair: 4 classes, 2 tiles per wave, the 8-class step table)
  int gbytes;        // bytes of one grid array when below 2 GB (scalar-offset buffer loads), else 0
  int kbytes;        // bytes of the operator array
  // source-stationary kernel: each class group's step list in nsplit parts
  // (one block each); part 0 stores into L, part k >= 1 into Lx
  // [k - 1][rhs][up_ncell][32] (cells up_cell0 ...), added to L afterwards
  int nsplit;
  int up_cell0, up_ncell;
  float *Lx;
  // full-precision kernel (k_m2l_real): rank in tiles of 16; a block's row
  // tiles, column tiles and waves (offset slices); row groups of a column
  // group; 1: buffer loads
  int kt, rt, ct, ws, nrg, buf;
  size_t plane;  // values of one coefficient plane of the grids
  // full-precision kernel on trees with many empty leaves: a bit per grid
  // slot, set when the cell holds particles; null: every source is multiplied
  const unsigned long long *occ;
  int few;       // 1: split-BF16 on few columns (k_m2l_bf16_few; ct, ws, plane as above)
};

constexpr int kSteps = 208;  // 8 source classes x 26 non-zero parent shifts
constexpr int kStepWords = 8;  // words per step record (see step_table)
constexpr int kZeroOp = kNumOps;  // all-zero operator slot of the split-BF16 layout
// s_waitcnt immediate (gfx9 encoding) for vmcnt(0), expcnt and lgkmcnt not waited on
constexpr int kWaitVm0 = 0x0F70;

struct GridM2L {
  int r = 0, maxlev = 0, nrhs = 1, form = 0, ncell_cap = 0, minlev = kMinLev, variant = 0;
  int flat = 0;  // 1: pointer-form loads even on grids below 2 GB
  // split-BF16 source-stationary kernel with a class-group size of its own
  // for the levels above the deepest: part[0] those levels, part[1] the
  // deepest (one launch each); nparts = 1: one launch, args
  int nparts = 1;
  GridArgs part[2];
  int part_blocks[2] = {0, 0};
  float *d_Lx = nullptr;  // partial sums of the upper part's steps beyond the first part
  GridArgs args{};
  int nblocks = 0;
  size_t nslots = 0;
  int4 *d_tab = nullptr;
  int *d_steps = nullptr;
  void *d_K = nullptr;
  void *d_Mg0 = nullptr;
  void *d_Mg1 = nullptr;
  void *d_Mg2 = nullptr;
  unsigned *d_lvl_max = nullptr;
  unsigned long long *d_occ = nullptr;
};

__device__ __forceinline__ int morton3(int x, int y, int z, int bits)
{
  int m = 0;
  for (int b = 0; b < bits; b++)
    m |= ((((x >> b) & 1) << 2) | (((y >> b) & 1) << 1) | ((z >> b) & 1)) << (3 * b);
  return m;
}

__device__ __forceinline__ void demorton3(int m, int bits, int &x, int &y, int &z)
{
  x = y = z = 0;
  for (int b = 0; b < bits; b++) {
    const int s = (m >> (3 * b)) & 7;
    x |= ((s >> 2) & 1) << b;
    y |= ((s >> 1) & 1) << b;
    z |= (s & 1) << b;
  }
}

// slot of (level, class, parent p) in the ghost-padded grids
__device__ __forceinline__ int grid_slot(const GridArgs &g, int l, int c, int px, int py, int pz)
{
  const int PP = (1 << (l - 1)) + 2;
  return g.lvl_slot0[l] + ((c * PP + px + 1) * PP + py + 1) * PP + pz + 1;
}

// ---------------------------------------------------------------- FP16X3 scaling
// The power of two that maps a largest magnitude m (bits of a non-negative
// float) into [2^14, 2^15): 2^(15 - e) with m = f 2^e, f in [0.5, 1).
__device__ __forceinline__ int fp16_scale_exp(unsigned mbits)
{
  int e = 0;
  (void)frexpf(__uint_as_float(mbits), &e);
  return 15 - e;
}

__device__ __forceinline__ void split3_f16(float v, _Float16 &t1, _Float16 &t2, _Float16 &t3)
{
  t1 = (_Float16)v;
  const float r1 = v - (float)t1;
  t2 = (_Float16)r1;
  t3 = (_Float16)(r1 - (float)t2);
}

__global__ void k_zero_u32(unsigned *p, int n)
{
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0u;
}

// Largest |M| of every level minlev..maxlev: blockIdx.y = level - minlev; a
// block reduces a grid-strided slice of the level's [rhs][cells][r] values
// and posts one atomicMax on the bits (order-preserving for non-negative
// floats).
__global__ void __launch_bounds__(256) k_level_absmax(GridArgs g, const real *__restrict__ M)
{
  __shared__ unsigned red[4];
  const int l = g.minlev + blockIdx.y;
  const int c0 = g.levsta[l], nc = g.levsta[l + 1] - c0;
  const long long per = (long long)nc * g.r / 4;  // float4 per vector
  const long long total = per * g.nrhs;
  float m = 0.0f;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long long)gridDim.x * blockDim.x) {
    const int rhs = (int)(t / per);
    const long long k = t - (long long)rhs * per;
    const float4 v = *reinterpret_cast<const float4 *>(M + ((size_t)rhs * g.ncell + c0) * g.r + 4 * k);
    m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
  }
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = __float_as_uint(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned b = red[0];
    for (int w = 1; w < 4; w++) b = max(b, red[w]);
    atomicMax(g.lvl_max + l, b);
  }
}

// ---------------------------------------------------------------- scatter
// M [rhs][ncell][r] -> per-class grids [slot][rhs][r]; one thread per
// (cell, rhs, 8 consecutive coefficients).
template <int FORM>
__global__ void k_grid_scatter(GridArgs g, const real *__restrict__ M)
{
  constexpr int CW = 8;
  const int chunks = g.r / CW;
  const long long total = (long long)(g.levsta[g.maxlev + 1] - g.levsta[g.minlev]) * g.nrhs * chunks;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int ch = (int)(t % chunks);
  const long long cr = t / chunks;
  const int rhs = (int)(cr % g.nrhs);
  const int A = g.levsta[g.minlev] + (int)(cr / g.nrhs);
  int l = g.minlev;
  while (A >= g.levsta[l + 1]) l++;
  int x, y, z;
  demorton3(A - g.levsta[l], l, x, y, z);
  const int c = ((x & 1) << 2) | ((y & 1) << 1) | (z & 1);
  const size_t slot = grid_slot(g, l, c, x >> 1, y >> 1, z >> 1);
  const real *src = M + ((size_t)rhs * g.ncell + A) * g.r + ch * CW;
  const size_t dst = (slot * g.nrhs + rhs) * g.r + ch * CW;
  if (FORM == BBFMM_M2L_BF16X2) {
    bf16x8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float v = (float)src[e];
      const __bf16 h = (__bf16)v;
      hi[e] = h;
      lo[e] = (__bf16)(v - (float)h);
    }
    *reinterpret_cast<bf16x8 *>((__bf16 *)g.Mg0 + dst) = hi;
    *reinterpret_cast<bf16x8 *>((__bf16 *)g.Mg1 + dst) = lo;
  } else {  // FP16X3
    const float sc = ldexpf(1.0f, fp16_scale_exp(g.lvl_max[l]));
    f16x8 t1, t2, t3;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      _Float16 a1, a2, a3;
      split3_f16((float)src[e] * sc, a1, a2, a3);
      t1[e] = a1;
      t2[e] = a2;
      t3[e] = a3;
    }
    *reinterpret_cast<f16x8 *>((_Float16 *)g.Mg0 + dst) = t1;
    *reinterpret_cast<f16x8 *>((_Float16 *)g.Mg1 + dst) = t2;
    *reinterpret_cast<f16x8 *>((_Float16 *)g.Mg2 + dst) = t3;
  }
}

// Blocks are dealt to the 8 XCDs round-robin (block b on XCD b % 8): the
// logical block of launch block b gives each XCD a contiguous run of logical
// blocks -- the 8 classes of a column group and neighbouring column groups,
// which read the same shifted source tiles -- so they share its L2.  The
// launch is rounded up to a multiple of 8; blocks past the end get -1.
__device__ __forceinline__ int xcd_block(const GridArgs &g, int b)
{
  const int nb = g.blk0[g.maxlev + 1];
  const int lb = (b & 7) * ((nb + 7) >> 3) + (b >> 3);
  return lb < nb ? lb : -1;
}

// level / class / column-group of a block of the flattened launch
__device__ __forceinline__ void decode_block(const GridArgs &g, int b, int &l, int &s, int &grp)
{
  l = g.minlev;
  while (l < g.maxlev && b >= g.blk0[l + 1]) l++;
  const int rel = b - g.blk0[l];
  s = rel & 7;
  grp = rel >> 3;
}

// ---------------------------------------------------------------- MFMA kernel
// 256 threads = 4 waves, all of one class s at one level; each wave owns
// TPW tiles of 32 columns.  Per offset v: A = K_v (bf16 hi/lo or fp32, read
// in lane order), B = the shifted sources of the wave's columns.
template <int FORM, int TPW>
__global__ void __launch_bounds__(256) k_m2l_mfma(GridArgs g)
{
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int lb = xcd_block(g, blockIdx.x);
  if (lb < 0) return;
  int l, s, grp;
  decode_block(g, lb, l, s, grp);
  const int P = 1 << (l - 1);
  const int PP = P + 2;
  const int ncols = P * P * P * g.nrhs;
  const int half = lane >> 5;  // which k-half of the operand this lane holds
  int base[TPW], rhs[TPW], pcol[TPW];
  bool valid[TPW];
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    const int col = ((grp * 4 + wave) * TPW + t) * 32 + (lane & 31);
    valid[t] = col < ncols;
    const int c = valid[t] ? col : 0;
    const int pl = c / g.nrhs;
    rhs[t] = c - pl * g.nrhs;
    pcol[t] = pl;
    const int pz = pl % P, py = (pl / P) % P, px = pl / (P * P);
    base[t] = ((px + 1) * PP + py + 1) * PP + pz + 1;
  }
  f32x16 acc[TPW];
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[t][e] = 0.0f;

  const int4 *tab = g.tab + s * kOffsets;
  const int slot0 = g.lvl_slot0[l];
  for (int v = 0; v < kOffsets; v++) {
    const int4 e = tab[v];
    const int k = e.x;
    const int sc = e.y;
    const int dx = ((e.z >> 4) & 3) - 1, dy = ((e.z >> 2) & 3) - 1, dz = (e.z & 3) - 1;
    const int off = slot0 + sc * PP * PP * PP + (dx * PP + dy) * PP + dz;
    if (FORM == BBFMM_M2L_BF16X2) {
      // A: [k][kstep][hi/lo][lane] bf16x8
      const bf16x8 *Ka = (const bf16x8 *)g.Ka + (size_t)k * 4 * 64 + lane;
      const bf16x8 a0h = Ka[0 * 64], a0l = Ka[1 * 64], a1h = Ka[2 * 64], a1l = Ka[3 * 64];
      const __bf16 *Mh = (const __bf16 *)g.Mg0;
      const __bf16 *Ml = (const __bf16 *)g.Mg1;
#pragma unroll
      for (int t = 0; t < TPW; t++) {
        const size_t o = ((size_t)(off + base[t]) * g.nrhs + rhs[t]) * 32 + half * 8;
        bf16x8 b0h = *(const bf16x8 *)(Mh + o), b0l = *(const bf16x8 *)(Ml + o);
        bf16x8 b1h = *(const bf16x8 *)(Mh + o + 16), b1l = *(const bf16x8 *)(Ml + o + 16);
        if (!valid[t]) {
#pragma unroll
          for (int q = 0; q < 8; q++) b0h[q] = b0l[q] = b1h[q] = b1l[q] = (__bf16)0.0f;
        }
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0h, b0h, acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0h, b0l, acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0l, b0h, acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1h, b1h, acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1h, b1l, acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1l, b1h, acc[t], 0, 0, 0);
      }
    } else if (FORM == BBFMM_M2L_FP16X3) {
      // A: [k][kstep][term][lane] f16x8, as the BF16X2 layout with three terms
      const f16x8 *Ka = (const f16x8 *)g.Ka + (size_t)k * 6 * 64 + lane;
      f16x8 a[2][3];
#pragma unroll
      for (int ks = 0; ks < 2; ks++)
#pragma unroll
        for (int q = 0; q < 3; q++) a[ks][q] = Ka[(ks * 3 + q) * 64];
      const _Float16 *Mt[3] = {(const _Float16 *)g.Mg0, (const _Float16 *)g.Mg1, (const _Float16 *)g.Mg2};
#pragma unroll
      for (int t = 0; t < TPW; t++) {
        const size_t o = ((size_t)(off + base[t]) * g.nrhs + rhs[t]) * 32 + half * 8;
        f16x8 b[2][3];
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
          for (int q = 0; q < 3; q++) {
            b[ks][q] = *(const f16x8 *)(Mt[q] + o + 16 * ks);
            if (!valid[t]) b[ks][q] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
          }
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks][0], b[ks][0], acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks][0], b[ks][1], acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks][1], b[ks][0], acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks][0], b[ks][2], acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks][1], b[ks][1], acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks][2], b[ks][0], acc[t], 0, 0, 0);
        }
      }
    }
  }
  // epilogue: lane holds rows 8*(e/4) + 4*half + e%4 of its column
  float unscale = 1.0f;
  if (FORM == BBFMM_M2L_FP16X3) unscale = ldexpf(g.kscale_inv, -fp16_scale_exp(g.lvl_max[l]));
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    if (!valid[t]) continue;
    if (FORM == BBFMM_M2L_FP16X3)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[t][e] *= unscale;
    const int pl = pcol[t];
    const int pz = pl % P, py = (pl / P) % P, px = pl / (P * P);
    const int fx = 2 * px + ((s >> 2) & 1), fy = 2 * py + ((s >> 1) & 1), fz = 2 * pz + (s & 1);
    const int A = g.levsta[l] + morton3(fx, fy, fz, l);
    float *Lp = (float *)g.L + ((size_t)rhs[t] * g.ncell + A) * 32 + 4 * half;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      f32x4 o = {acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
      *reinterpret_cast<f32x4 *>(Lp + 8 * q) = o;
    }
  }
}

// ---------------------------------------------------------------- ghost steps of a wave
// The parents of a wave's span columns (columns are (parent, vector) pairs,
// vector fastest, then pz, py, px) lie in the box [lo, hi] per axis (the
// whole axis where the columns span more than one row).  A step of shift d
// whose shifted box lies outside [0, P) in some axis reads only the ghost
// layer (zeros) for every column of the wave: its products add nothing, and
// the wave skips them.  A wave without valid columns skips every step.
struct WaveBox {
  int lo[3], hi[3];
};

__device__ __forceinline__ WaveBox wave_box(int col0, int ncols, int nrhs, int P, int span)
{
  WaveBox b;
  if (col0 >= ncols) {
    for (int a = 0; a < 3; a++) {
      b.lo[a] = 2 * P;
      b.hi[a] = -2 * P;
    }
    return b;
  }
  const int f = col0 / nrhs, t = min(col0 + span - 1, ncols - 1) / nrhs;
  const int fx = f / (P * P), fy = (f / P) % P, fz = f % P;
  const int tx = t / (P * P), ty = (t / P) % P, tz = t % P;
  b.lo[0] = fx;
  b.hi[0] = tx;
  const bool row = fx == tx, line = row && fy == ty;
  b.lo[1] = row ? fy : 0;
  b.hi[1] = row ? ty : P - 1;
  b.lo[2] = line ? fz : 0;
  b.hi[2] = line ? tz : P - 1;
  return b;
}

// the step record's first word: source class | packed shift << 3
__device__ __forceinline__ bool ghost_step(const WaveBox &b, int e0, int P)
{
  const int pk = e0 >> 3;
  const int d[3] = {((pk >> 4) & 3) - 1, ((pk >> 2) & 3) - 1, (pk & 3) - 1};
  bool g = false;
#pragma unroll
  for (int a = 0; a < 3; a++) g |= (b.hi[a] + d[a] < 0) | (b.lo[a] + d[a] >= P);
  return g;
}

// ---------------------------------------------------------------- source-stationary MFMA kernel
// Same products, loop order inverted: a field cell of class s at parent p and
// a source of class s' at parent p + d interact through the offset
// v = 2d + s' - s, so for one (s', d) the shifted source tile M_{s'}[p + d]
// serves every field class.  A wave owns TPW tiles of 32 columns (parent,
// vector) of CLS field classes (TPW x CLS accumulators); per step (s', d) it
// loads its source tiles once and multiplies them by the CLS operators K_v,
// which the block stages in LDS (double-buffered) for all its waves.  CLS = 8
// takes all classes of a column group in one block; CLS = 4 or 2 splits a
// column group over 2 or 4 blocks (class groups), which evens out the work
// per CU when the column groups do not fill whole rounds of the chip, and
// drops the steps in which every class of the group has a near-field offset.
// With TPW = 2 every operator fragment read from LDS serves two tiles.
// Split-BF16 (fp32 build).
template <int CLS, int TPW, bool BUF>
__global__ void __launch_bounds__(256) k_m2l_mfma_ss(GridArgs g)
{
  constexpr int WAVES = 4;  // one k-part (k-step x hi/lo) of the operators per wave
  constexpr int NCG = 8 / CLS;
  __shared__ bf16x8 sK[2][CLS][4][64];  // [buffer][class of the group][kstep*2 + hi/lo][lane]
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  // Blocks are dealt to the 8 XCDs round-robin (block b on XCD b % 8); the
  // logical order gives each XCD a contiguous run of column groups, i.e.
  // neighbouring parents, whose shifted source tiles then share its L2; the
  // class groups of one column group are adjacent.
  const int nb = g.blk0[g.maxlev + 1];
  const int lb = (blockIdx.x & 7) * ((nb + 7) >> 3) + (blockIdx.x >> 3);
  if (lb >= nb) return;
  int l = g.minlev;
  while (l < g.maxlev && lb >= g.blk0[l + 1]) l++;
  const int nsp = g.nsplit > 1 ? g.nsplit : 1;
  const int rel = lb - g.blk0[l];
  const int part = rel % nsp, rq = rel / nsp;
  const int grp = rq / NCG, cg = rq - grp * NCG;
  const int P = 1 << (l - 1);
  const int PP = P + 2;
  const int ncols = P * P * P * g.nrhs;
  const int half = lane >> 5;
  const int sh0 = PP * PP + PP + 1;
  const int col0 = (grp * WAVES + wave) * 32 * TPW;
  // per tile: columns past the end compute a copy of column 0 and are not stored
  bool valid[TPW];
  int rh[TPW], px[TPW], py[TPW], pz[TPW], base[TPW], voff[TPW];
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    const int col = col0 + 32 * t + (lane & 31);
    valid[t] = col < ncols;
    const int cc = valid[t] ? col : 0;
    const int pl = cc / g.nrhs;
    rh[t] = cc - pl * g.nrhs;
    pz[t] = pl % P;
    py[t] = (pl / P) % P;
    px[t] = pl / (P * P);
    base[t] = ((px[t] + 1) * PP + py[t] + 1) * PP + pz[t] + 1;
    // the scalar offset of a buffer load is unsigned: the shift's most
    // negative value, -(PP^2 + PP + 1), moves to the lane part (base >= PP^2 + PP + 1)
    voff[t] = (((base[t] - sh0) * g.nrhs + rh[t]) * 32 + half * 8) * 2;
  }
  const int slot0 = g.lvl_slot0[l];
  const int cls = PP * PP * PP;
  const bf16x8 *Kl = (const bf16x8 *)g.Ka + wave * 64 + lane;
  const __bf16 *Mh = (const __bf16 *)g.Mg0;
  const __bf16 *Ml = (const __bf16 *)g.Mg1;
  const WaveBox box =
      wave_box((grp * WAVES + __builtin_amdgcn_readfirstlane(wave)) * 32 * TPW, ncols, g.nrhs, P, 32 * TPW);

  f32x16 acc[TPW][CLS];
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int c = 0; c < CLS; c++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[t][c][e] = 0.0f;

  // Step record of the class group: e[0] = source class | packed shift << 3,
  // e[1 + i/2] holds the operator of the group's classes i (low 16 bits) and
  // i + 1 (high); near-field pairs point at the zero operator, so every step
  // runs all CLS classes.  Each wave moves its k-part of the step's operators
  // (1 KB each) from global memory straight into the other LDS buffer
  // (global_load_lds, 16 bytes per lane at lane-contiguous addresses) while
  // the MFMAs of the current step run; the source tiles of the next step are
  // loaded into registers at the same time.  Records are read two steps ahead.
  typedef __attribute__((address_space(3))) void lds_void;
  // BUF: buffer loads whose per-step part is a scalar offset (the operator's
  // index, the step's shift) and whose per-lane part is fixed, so that no
  // vector instructions go into the step's addresses (grids below 2 GB)
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void *)g.Ka, 0, g.kbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rMh = __builtin_amdgcn_make_buffer_rsrc((void *)g.Mg0, 0, g.gbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rMl = __builtin_amdgcn_make_buffer_rsrc((void *)g.Mg1, 0, g.gbytes, 0x00020000);
  auto load_k = [&](const int *e, int buf) {
#pragma unroll
    for (int i = 0; i < CLS; i++) {
      const int k = (e[1 + (i >> 1)] >> (16 * (i & 1))) & 0xffff;
      if (BUF)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rK, (lds_void *)&sK[buf][i][wave][0], 16, (wave * 64 + lane) * 16,
                                                 k * 256 * 16, 0, 0);
      else
        __builtin_amdgcn_global_load_lds((const void *)(Kl + (size_t)k * 256), (lds_void *)&sK[buf][i][wave][0], 16,
                                         0, 0);
    }
  };
  // source tiles of step e: hi and lo of k-steps 0 and 1
  struct Src {
    bf16x8 h0, l0, h1, l1;
  };
  auto load_src = [&](const int *e, Src *d) {
    const int sc = e[0] & 7, pk = e[0] >> 3;
    const int dx = ((pk >> 4) & 3) - 1, dy = ((pk >> 2) & 3) - 1, dz = (pk & 3) - 1;
    const int sft = slot0 + sc * cls + (dx * PP + dy) * PP + dz;
#pragma unroll
    for (int t = 0; t < TPW; t++) {
      if (BUF) {
        const int so = (sft + sh0) * g.nrhs * 64;
        d[t].h0 = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rMh, voff[t], so, 0));
        d[t].l0 = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rMl, voff[t], so, 0));
        d[t].h1 = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rMh, voff[t] + 32, so, 0));
        d[t].l1 = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rMl, voff[t] + 32, so, 0));
      } else {
        const size_t o = ((size_t)(sft + base[t]) * g.nrhs + rh[t]) * 32 + half * 8;
        d[t].h0 = *(const bf16x8 *)(Mh + o);
        d[t].l0 = *(const bf16x8 *)(Ml + o);
        d[t].h1 = *(const bf16x8 *)(Mh + o + 16);
        d[t].l1 = *(const bf16x8 *)(Ml + o + 16);
      }
    }
  };
  // this block's part of the class group's steps (all of them when nsplit = 1)
  const int s_lo = part * g.nsteps[cg] / nsp;
  const int nst = (part + 1) * g.nsteps[cg] / nsp - s_lo;
  const int *S = g.steps + ((size_t)cg * kSteps + s_lo) * kStepWords;
  int e1[5];
  int ec = S[0];  // first word of the current step's record
  Src cur[TPW];
  {
    int e0[5];
#pragma unroll
    for (int i = 0; i < 5; i++) e0[i] = S[i];
    const int s1 = nst > 1 ? 1 : 0;
#pragma unroll
    for (int i = 0; i < 5; i++) e1[i] = S[s1 * kStepWords + i];
    load_k(e0, 0);
    load_src(e0, cur);
  }
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  __syncthreads();
  for (int st = 0; st < nst; st++) {
    const int b = st & 1;
    // the last steps reload their own data (harmless, never used)
    const int n2 = st + 2 < nst ? st + 2 : nst - 1;
    // vector loads (operators arriving by DMA keep the compiler from scalar
    // loads here); moved to scalar registers after the end-of-step wait
    const int4 r2a = *reinterpret_cast<const int4 *>(S + n2 * kStepWords);
    const int r2b = CLS > 6 ? S[n2 * kStepWords + 4] : 0;
    const bool skip = ghost_step(box, ec, P);
    // k-step 0 of all classes, then the k-step-1 fragments; only then the
    // loads into the other buffer (the compiler orders LDS reads after any
    // earlier global_load_lds), then k-step 1
    bf16x8 ah[CLS], al[CLS];
    if (!skip) {
#pragma unroll
      for (int c = 0; c < CLS; c++) {
        ah[c] = sK[b][c][0][lane];
        al[c] = sK[b][c][1][lane];
      }
      // all reads issued before the first product (otherwise the scheduler
      // puts each read just before its MFMA, which then waits on it)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CLS; c++)
#pragma unroll
        for (int t = 0; t < TPW; t++) {
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], cur[t].h0, acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], cur[t].l0, acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[c], cur[t].h0, acc[t][c], 0, 0, 0);
        }
#pragma unroll
      for (int c = 0; c < CLS; c++) {
        ah[c] = sK[b][c][2][lane];
        al[c] = sK[b][c][3][lane];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_k(e1, b ^ 1);
    Src nxt[TPW];
    load_src(e1, nxt);
    __builtin_amdgcn_sched_barrier(0);
    if (!skip) {
#pragma unroll
      for (int c = 0; c < CLS; c++)
#pragma unroll
        for (int t = 0; t < TPW; t++) {
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], cur[t].h1, acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], cur[t].l1, acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[c], cur[t].h1, acc[t][c], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < TPW; t++) cur[t] = nxt[t];
    // the next step's operators are in LDS for every wave after this (the
    // scheduling barrier keeps the MFMAs above the wait)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    ec = e1[0];
    e1[0] = __builtin_amdgcn_readfirstlane(r2a.x);
    e1[1] = __builtin_amdgcn_readfirstlane(r2a.y);
    e1[2] = __builtin_amdgcn_readfirstlane(r2a.z);
    e1[3] = __builtin_amdgcn_readfirstlane(r2a.w);
    e1[4] = __builtin_amdgcn_readfirstlane(r2b);
  }
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    if (!valid[t]) continue;
#pragma unroll
    for (int i = 0; i < CLS; i++) {
      const int c = cg * CLS + i;
      const int fx = 2 * px[t] + ((c >> 2) & 1), fy = 2 * py[t] + ((c >> 1) & 1), fz = 2 * pz[t] + (c & 1);
      const int A = g.levsta[l] + morton3(fx, fy, fz, l);
      float *Lp = part == 0 ? (float *)g.L + ((size_t)rh[t] * g.ncell + A) * 32 + 4 * half
                            : g.Lx + (((size_t)(part - 1) * g.nrhs + rh[t]) * g.up_ncell + (A - g.up_cell0)) * 32 +
                                  4 * half;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f32x4 v = {acc[t][i][4 * q], acc[t][i][4 * q + 1], acc[t][i][4 * q + 2], acc[t][i][4 * q + 3]};
        *reinterpret_cast<f32x4 *>(Lp + 8 * q) = v;
      }
    }
  }
}

// ---------------------------------------------------------------- class-group pairs sharing source tiles
// k_m2l_mfma_ss with 4 classes and two 32-column tiles per wave, and both
// class groups of a column group in one block of 8 waves (waves 0-3 classes
// 0-3, waves 4-7 classes 4-7, wave w on the columns of tile pair w % 4).
// The block walks the union of the two groups' step lists (the 8-class
// table: 208 steps; a group's classes that are near in a step take the zero
// operator), so the shifted source tiles of a step are the same for both
// groups: the block moves them into LDS once (wave w moves tile w / 4 of its
// own columns, global_load_lds, double-buffered like the operators) and
// every wave reads its B fragments from there.  Per 48 MFMAs a wave moves
// 4 KB of operators and 4 KB of sources from memory (8 + 4 KB when each
// group loads its own tiles).  LDS: 64 KB of operators + 64 KB of source
// tiles, one block per CU.
template <bool BUF>
__global__ void __launch_bounds__(512) k_m2l_mfma_ss_pair(GridArgs g)
{
  constexpr int CLS = 4, TPW = 2;
  __shared__ bf16x8 sK[2][8][4][64];         // [buffer][class][kstep*2 + hi/lo][lane]
  __shared__ bf16x8 sS[2][4][TPW][4][64];    // [buffer][tile pair][tile][h0, l0, h1, l1][lane]
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int tp = wave & 3, cg = wave >> 2;
  const int nb = g.blk0[g.maxlev + 1];
  const int lb = (blockIdx.x & 7) * ((nb + 7) >> 3) + (blockIdx.x >> 3);
  if (lb >= nb) return;
  int l = g.minlev;
  while (l < g.maxlev && lb >= g.blk0[l + 1]) l++;
  const int grp = lb - g.blk0[l];
  const int P = 1 << (l - 1);
  const int PP = P + 2;
  const int ncols = P * P * P * g.nrhs;
  const int half = lane >> 5;
  const int sh0 = PP * PP + PP + 1;
  const int col0 = (grp * 4 + tp) * 32 * TPW;
  bool valid[TPW];
  int rh[TPW], px[TPW], py[TPW], pz[TPW], base[TPW], voff[TPW];
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    const int col = col0 + 32 * t + (lane & 31);
    valid[t] = col < ncols;
    const int cc = valid[t] ? col : 0;
    const int pl = cc / g.nrhs;
    rh[t] = cc - pl * g.nrhs;
    pz[t] = pl % P;
    py[t] = (pl / P) % P;
    px[t] = pl / (P * P);
    base[t] = ((px[t] + 1) * PP + py[t] + 1) * PP + pz[t] + 1;
    voff[t] = (((base[t] - sh0) * g.nrhs + rh[t]) * 32 + half * 8) * 2;
  }
  const int slot0 = g.lvl_slot0[l];
  const int cls = PP * PP * PP;
  const WaveBox box = wave_box((grp * 4 + __builtin_amdgcn_readfirstlane(tp)) * 32 * TPW, ncols, g.nrhs, P, 32 * TPW);
  f32x16 acc[TPW][CLS];
#pragma unroll
  for (int t = 0; t < TPW; t++)
#pragma unroll
    for (int c = 0; c < CLS; c++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[t][c][e] = 0.0f;

  typedef __attribute__((address_space(3))) void lds_void;
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void *)g.Ka, 0, g.kbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rMh = __builtin_amdgcn_make_buffer_rsrc((void *)g.Mg0, 0, g.gbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rMl = __builtin_amdgcn_make_buffer_rsrc((void *)g.Mg1, 0, g.gbytes, 0x00020000);
  const bf16x8 *Kl = (const bf16x8 *)g.Ka + tp * 64 + lane;
  const __bf16 *Mh = (const __bf16 *)g.Mg0;
  const __bf16 *Ml = (const __bf16 *)g.Mg1;
  const int my_t = cg;  // the tile of its own columns this wave moves into LDS
  // operators: wave w moves k-part w % 4 of its group's 4 classes
  auto load_k = [&](const int *e, int buf) {
#pragma unroll
    for (int i = 0; i < CLS; i++) {
      const int k = (e[1 + 2 * cg + (i >> 1)] >> (16 * (i & 1))) & 0xffff;
      if (BUF)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rK, (lds_void *)&sK[buf][4 * cg + i][tp][0], 16,
                                                 (tp * 64 + lane) * 16, k * 256 * 16, 0, 0);
      else
        __builtin_amdgcn_global_load_lds((const void *)(Kl + (size_t)k * 256), (lds_void *)&sK[buf][4 * cg + i][tp][0],
                                         16, 0, 0);
    }
  };
  // source tile my_t of this wave's columns for step e: h0, l0, h1, l1
  auto load_s = [&](const int *e, int buf) {
    const int sc = e[0] & 7, pk = e[0] >> 3;
    const int dx = ((pk >> 4) & 3) - 1, dy = ((pk >> 2) & 3) - 1, dz = (pk & 3) - 1;
    const int sft = slot0 + sc * cls + (dx * PP + dy) * PP + dz;
    lds_void *d = (lds_void *)&sS[buf][tp][my_t][0][0];
    if (BUF) {
      const int so = (sft + sh0) * g.nrhs * 64;
      const int vo = my_t ? voff[1] : voff[0];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rMh, d, 16, vo, so, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rMl, (lds_void *)&sS[buf][tp][my_t][1][0], 16, vo, so, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rMh, (lds_void *)&sS[buf][tp][my_t][2][0], 16, vo + 32, so, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rMl, (lds_void *)&sS[buf][tp][my_t][3][0], 16, vo + 32, so, 0, 0);
    } else {
      const int bs = my_t ? base[1] : base[0];
      const int rr = my_t ? rh[1] : rh[0];
      const size_t o = ((size_t)(sft + bs) * g.nrhs + rr) * 32 + half * 8;
      __builtin_amdgcn_global_load_lds((const void *)(Mh + o), d, 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void *)(Ml + o), (lds_void *)&sS[buf][tp][my_t][1][0], 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void *)(Mh + o + 16), (lds_void *)&sS[buf][tp][my_t][2][0], 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void *)(Ml + o + 16), (lds_void *)&sS[buf][tp][my_t][3][0], 16, 0, 0);
    }
  };
  const int nst = g.nsteps[0];
  const int *S = g.steps;
  int e1[5];
  int ec = S[0];
  {
    int e0[5];
#pragma unroll
    for (int i = 0; i < 5; i++) e0[i] = S[i];
    const int s1 = nst > 1 ? 1 : 0;
#pragma unroll
    for (int i = 0; i < 5; i++) e1[i] = S[s1 * kStepWords + i];
    load_k(e0, 0);
    load_s(e0, 0);
  }
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  __syncthreads();
  for (int st = 0; st < nst; st++) {
    const int b = st & 1;
    const int n2 = st + 2 < nst ? st + 2 : nst - 1;
    const int4 r2a = *reinterpret_cast<const int4 *>(S + n2 * kStepWords);
    const int r2b = S[n2 * kStepWords + 4];
    const bool skip = ghost_step(box, ec, P);
    // every LDS read of the step comes before the DMA into the other buffer
    bf16x8 ah[CLS], al[CLS], bh[TPW], bl[TPW];
    if (!skip) {
#pragma unroll
      for (int c = 0; c < CLS; c++) {
        ah[c] = sK[b][4 * cg + c][0][lane];
        al[c] = sK[b][4 * cg + c][1][lane];
      }
#pragma unroll
      for (int t = 0; t < TPW; t++) {
        bh[t] = sS[b][tp][t][0][lane];
        bl[t] = sS[b][tp][t][1][lane];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CLS; c++)
#pragma unroll
        for (int t = 0; t < TPW; t++) {
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], bh[t], acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], bl[t], acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[c], bh[t], acc[t][c], 0, 0, 0);
        }
#pragma unroll
      for (int c = 0; c < CLS; c++) {
        ah[c] = sK[b][4 * cg + c][2][lane];
        al[c] = sK[b][4 * cg + c][3][lane];
      }
#pragma unroll
      for (int t = 0; t < TPW; t++) {
        bh[t] = sS[b][tp][t][2][lane];
        bl[t] = sS[b][tp][t][3][lane];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_k(e1, b ^ 1);
    load_s(e1, b ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    if (!skip) {
#pragma unroll
      for (int c = 0; c < CLS; c++)
#pragma unroll
        for (int t = 0; t < TPW; t++) {
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], bh[t], acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[c], bl[t], acc[t][c], 0, 0, 0);
          acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[c], bh[t], acc[t][c], 0, 0, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    ec = e1[0];
    e1[0] = __builtin_amdgcn_readfirstlane(r2a.x);
    e1[1] = __builtin_amdgcn_readfirstlane(r2a.y);
    e1[2] = __builtin_amdgcn_readfirstlane(r2a.z);
    e1[3] = __builtin_amdgcn_readfirstlane(r2a.w);
    e1[4] = __builtin_amdgcn_readfirstlane(r2b);
  }
#pragma unroll
  for (int t = 0; t < TPW; t++) {
    if (!valid[t]) continue;
#pragma unroll
    for (int i = 0; i < CLS; i++) {
      const int c = 4 * cg + i;
      const int fx = 2 * px[t] + ((c >> 2) & 1), fy = 2 * py[t] + ((c >> 1) & 1), fz = 2 * pz[t] + (c & 1);
      const int A = g.levsta[l] + morton3(fx, fy, fz, l);
      float *Lp = (float *)g.L + ((size_t)rh[t] * g.ncell + A) * 32 + 4 * half;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f32x4 v = {acc[t][i][4 * q], acc[t][i][4 * q + 1], acc[t][i][4 * q + 2], acc[t][i][4 * q + 3]};
        *reinterpret_cast<f32x4 *>(Lp + 8 * q) = v;
      }
    }
  }
}

// L of the cells up_cell0 .. up_cell0 + up_ncell - 1 += the partial sums of
// parts 1 .. nsplit - 1 (in part order), one float4 per thread
__global__ void __launch_bounds__(256) k_m2l_add_parts(GridArgs g)
{
  const size_t n4 = (size_t)g.nrhs * g.up_ncell * 8;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const size_t rc = i >> 3;  // rhs * up_ncell + cell
  const int q = (int)(i & 7);
  const size_t rh = rc / g.up_ncell, c = rc - rh * g.up_ncell;
  f32x4 *Lp = reinterpret_cast<f32x4 *>(g.L + (rh * g.ncell + g.up_cell0 + c) * 32) + q;
  f32x4 v = *Lp;
  const f32x4 *X = reinterpret_cast<const f32x4 *>(g.Lx);
  for (int k = 0; k + 1 < g.nsplit; k++) v += X[((size_t)k * g.nrhs * g.up_ncell + rc) * 8 + q];
  *Lp = v;
}

// ---------------------------------------------------------------- full-precision kernel
// L_s[:, p] += K_v M_{s'}[:, p + d] in the build's own precision on
// v_mfma_f32_16x16x4_f32 / v_mfma_f64_16x16x4_f64 (fp32 / fp64 operands and
// sums), any rank 1..512, padded with zeros to kt tiles of 16.
//
// Operators: [k][row tile][k chunk of 16][lane] (k_real_layout): lane l
// holds row 16 tile + real_row(l % 16) and columns 16 chunk + 4 (l / 16) ..
// + 3, the operands of four products, in 16-byte pieces; the B fragment is
// the same four coefficients of the lane's source column.
//
// A block is one class, RT tiles of rows and CT tiles of 16 columns (parents
// x vectors) of one level; its waves take the offsets in ws slices, whose
// sums are added through LDS in slice order.  Offsets
// whose shifted tile lies outside the level in some axis for all CT tiles
// read only ghost zeros: wave 0 lists the others once (with 16 vectors a
// tile is one parent and no ghost is multiplied).  The fragments of the next
// k chunk are loaded while the current one is multiplied.
// Class s takes the blocks b % 8 = s, which run on one XCD: its L2 then holds
// that class's operators only.
//
// Bound by the matrix unit at many columns (the fragments' loads come from L2
// at 8 to 24 bytes a clock and CU), by the operators' bytes beyond L2 at high
// rank and few columns, by latency at the smallest sizes.  M2L alone, scatter
// included, against the kernels before it (fp32 or fp64 FMAs, a thread a row
// or a lane a column; 32-column MFMA tiles without offset slices):
//   n = 4, one vector: N = 65536 315 -> 32 us, 1M 553 -> 131 us (93 TFLOP/s
//   of list products), fp64 100003 380 -> 54 us, 1M 1023 -> 242 us;
//   n = 4, 16 vectors, 1M, fp32: 2640 -> 1600 us; n = 6, 80000, one vector:
//   10120 -> 204 us (fp64 14250 -> 400); n = 8, 131072: one vector
//   24.5 -> 0.96 ms, 16 vectors 19.25 -> 9.95 ms (135 TFLOP/s).
#ifdef SINGLE
typedef float realx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ realx4 mfma_real(real a, real b, realx4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// row of the tile that A's lane i holds (accumulator v of lane group h is row 4 h + v)
__host__ __device__ __forceinline__ int real_row(int i) { return i; }
#else
typedef double realx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ realx4 mfma_real(real a, real b, realx4 c)
{
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// the fp64 product leaves its row 4 v + h in accumulator v of lane group h:
// A's rows are permuted so that it too is row 4 h + v of the tile
__host__ __device__ __forceinline__ int real_row(int i) { return 4 * (i & 3) + (i >> 2); }
#endif
typedef real realx __attribute__((ext_vector_type(16 / sizeof(real))));  // a 16-byte piece
// L of any caller is stored four values at a time whatever its alignment
typedef real realx4u __attribute__((ext_vector_type(4), aligned(sizeof(real))));

constexpr int kVW = 16 / (int)sizeof(real);  // coefficients of a 16-byte piece
constexpr int kPW = 4 / kVW;                  // pieces of the four coefficients of a fragment

// out [k][tile][chunk][piece][lane][kVW] from the column-major operators (K_k(i, j) at k r^2 + j r + i)
__global__ void __launch_bounds__(256) k_real_layout(int r, int kt, const real *__restrict__ K, real *__restrict__ out)
{
  const long long n = (long long)kNumOps * kt * kt * 256;
  const long long o = (long long)blockIdx.x * 256 + threadIdx.x;
  if (o >= n) return;
  const int e = (int)(o % kVW), lane = (int)(o / kVW % 64), h = (int)(o / (64 * kVW) % kPW);
  const long long tc = o >> 8;
  const int c = (int)(tc % kt), t = (int)((tc / kt) % kt), k = (int)(tc / kt / kt);
  const int row = 16 * t + real_row(lane & 15), col = 16 * c + 4 * (lane >> 4) + kVW * h + e;
  out[o] = row < r && col < r ? K[((size_t)k * r + col) * r + row] : (real)0;
}

// M [rhs][ncell][r] -> grids [plane][slot][rhs][kVW], plane p holding the
// coefficients kVW p .. kVW p + kVW - 1 (zeros from r on): the 16 columns of
// a fragment are then one 256-byte piece of a plane wherever the shift puts
// them (as [slot][rhs][r] every lane's 16 bytes were a separate access of
// the cache: the M2L of 131072 particles, n = 8, 16 vectors took 18.5 ms)
__global__ void __launch_bounds__(256) k_real_scatter(GridArgs g, const real *__restrict__ M)
{
  const int np = 16 * g.kt / kVW;
  const long long total = (long long)(g.levsta[g.maxlev + 1] - g.levsta[g.minlev]) * g.nrhs * np;
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= total) return;
  const int rhs = (int)(t % g.nrhs);
  const long long cp = t / g.nrhs;
  const int p = (int)(cp % np);
  const int A = g.levsta[g.minlev] + (int)(cp / np);
  int l = g.minlev;
  while (A >= g.levsta[l + 1]) l++;
  int x, y, z;
  demorton3(A - g.levsta[l], l, x, y, z);
  const size_t slot = grid_slot(g, l, ((x & 1) << 2) | ((y & 1) << 1) | (z & 1), x >> 1, y >> 1, z >> 1);
  const real *src = M + ((size_t)rhs * g.ncell + A) * g.r + kVW * p;
  realx v;
#pragma unroll
  for (int e = 0; e < kVW; e++) v[e] = kVW * p + e < g.r ? src[e] : (real)0;
  *reinterpret_cast<realx *>((real *)g.Mg0 + p * g.plane + (slot * g.nrhs + rhs) * kVW) = v;
}

// One thread per leaf: its cell and those above it marked in occ
__global__ void __launch_bounds__(256) k_mark_occupied(GridArgs g, const int *__restrict__ leafcnt, int nleaf,
                                                       unsigned *occ)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nleaf || leafcnt[i] == 0) return;
  int A = g.levsta[g.maxlev] + i;
  for (int l = g.maxlev; l >= g.minlev; l--, A = (A - 1) >> 3) {
    int x, y, z;
    demorton3(A - g.levsta[l], l, x, y, z);
    const int slot = grid_slot(g, l, ((x & 1) << 2) | ((y & 1) << 1) | (z & 1), x >> 1, y >> 1, z >> 1);
    atomicOr(&occ[slot >> 5], 1u << (slot & 31));
  }
}

// whether one of the slots [at, at + len) holds particles (len above 64: taken so)
__device__ __forceinline__ bool occupied(const unsigned long long *occ, int at, int len)
{
  if (len > 64) return true;
  const unsigned long long *w = occ + (at >> 6);
  const int o = at & 63;
  const unsigned long long b = w[0] >> o | w[1] << 1 << (63 - o);
  return (b << (64 - len)) != 0;
}

// Trees with many empty leaves (occ): the offsets at which no cell of a tile
// has a source with particles are left out; they add K_v times zeros.
// 150000 particles on a sphere, depth 5 (a seventh of the leaves), 4 vectors:
// 418 -> 177 us, one vector (tiles of 16 cells instead of 4) 124 -> 97.
//
// BUF: fragments by buffer loads (the uniform part of an address in the
// resource, a 32-bit lane offset; planes of a k chunk within 4 GB), else by
// 64-bit lane addresses, which cost the address path about twice as much
// (131072 particles, n = 8, 16 vectors, CT = RT = 4: 13.2 against 15.7 ms).
template <int RT, int CT, int KC, int MAXW, bool BUF>
__global__ void __launch_bounds__(64 * MAXW) k_m2l_real(GridArgs g)
{
  extern __shared__ __align__(32) unsigned char smem_raw[];
  realx4 *red = reinterpret_cast<realx4 *>(smem_raw);  // [slice][tile][64]
  __shared__ int2 lst[192];  // offsets to multiply: operator | tiles << 16, slot shift
  __shared__ int nlst;
  const int lane = threadIdx.x & 63;
  const int ws = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // offset slice
  const int s = blockIdx.x & 7, gr = blockIdx.x >> 3;
  const int gb = gr / g.nrg;               // column group
  const int rt0 = (gr - gb * g.nrg) * RT;  // first row tile
  int l = g.minlev;
  while (l < g.maxlev && gb >= g.blk0[l + 1]) l++;
  const int P = 1 << (l - 1);
  const int PP = P + 2;
  const int ncols = P * P * P * g.nrhs;
  const int col0 = (gb - g.blk0[l]) * (16 * CT);
  if (ws == 0) {
    WaveBox box[CT];
    int first[CT], len[CT];  // the slots of a tile's cells, before a shift
#pragma unroll
    for (int t = 0; t < CT; t++) {
      box[t] = wave_box(col0 + 16 * t, ncols, g.nrhs, P, 16);
      auto slot = [&](int col) {
        const int pl = min(col, ncols - 1) / g.nrhs;
        return (pl / (P * P) * PP + pl / P % P) * PP + pl % P;
      };
      first[t] = slot(col0 + 16 * t);
      len[t] = slot(col0 + 16 * t + 15) - first[t] + 1;
    }
    int n = 0;
    for (int q = 0; q < 3; q++) {
      const int v = 64 * q + lane;
      const int4 e = g.tab[s * kOffsets + min(v, kOffsets - 1)];
      const int dx = (e.z >> 4) & 3, dy = (e.z >> 2) & 3, dz = e.z & 3;  // shift + 1
      const int shift = e.y * PP * PP * PP + (dx * PP + dy) * PP + dz;
      int m = 0;
#pragma unroll
      for (int t = 0; t < CT; t++) {
        const bool on = !ghost_step(box[t], e.z << 3, P) &&
                        (!g.occ || occupied(g.occ, g.lvl_slot0[l] + first[t] + shift, len[t]));
        m |= on ? 1 << t : 0;
      }
      if (v >= kOffsets) m = 0;
      const unsigned long long act = __ballot(m != 0);
      if (m) lst[n + __popcll(act & ((1ull << lane) - 1))] = make_int2(e.x | (m << 16), shift);
      n += __popcll(act);
    }
    if (lane == 0) nlst = n;
  }
  const int kt = g.kt;
  const int nrt = min(RT, kt - rt0);  // row tiles
  // sources and operators: a uniform address plus a lane offset
  size_t bo[CT];
#pragma unroll
  for (int t = 0; t < CT; t++) {
    const int col = min(col0 + 16 * t + (lane & 15), ncols - 1);  // columns past the end are not stored
    const int pl = col / g.nrhs, rh = col - pl * g.nrhs;
    const int pz = pl % P, py = (pl / P) % P, px = pl / (P * P);
    const int slot = (px * PP + py) * PP + pz;  // shifts add PP (PP + 1) + 1 at most, 0 at least
    bo[t] = ((size_t)(lane >> 4) * kPW * g.plane + ((size_t)slot * g.nrhs + rh) * kVW) * sizeof(real);
  }
  const char *bbase = (const char *)((const real *)g.Mg0 + (size_t)g.lvl_slot0[l] * g.nrhs * kVW);
  const size_t plane = g.plane * sizeof(real);
  const int ktile = kt * 256 * (int)sizeof(real);
  const char *abase = (const char *)g.Ka + (size_t)rt0 * ktile;
  struct Frag {
    realx a[RT][KC][kPW], b[CT][KC][kPW];
  };
  auto load = [&](Frag &f, int2 w, int c) {
    const char *a = abase + (size_t)(w.x & 0xffff) * kt * ktile + (size_t)c * (256 * sizeof(real));
    const char *b = bbase + (size_t)w.y * (g.nrhs * 16) + (size_t)c * (16 / kVW) * plane;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)a, 0, -1, 0x00020000);
#pragma unroll
    for (int q = 0; q < KC; q++) {
      const char *bq = b + (size_t)q * (16 / kVW) * plane;
      const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)bq, 0, -1, 0x00020000);
#pragma unroll
      for (int h = 0; h < kPW; h++) {
#pragma unroll
        for (int i = 0; i < RT; i++) {
          const int at = min(i, nrt - 1) * ktile, al = q * (256 * (int)sizeof(real)) + h * 1024 + lane * 16;
          if (BUF)
            f.a[i][q][h] = __builtin_bit_cast(realx, __builtin_amdgcn_raw_buffer_load_b128(ra, al, at, 0));
          else
            f.a[i][q][h] = *reinterpret_cast<const realx *>(a + at + al);
        }
#pragma unroll
        for (int t = 0; t < CT; t++)
          if (BUF)
            f.b[t][q][h] =
                __builtin_bit_cast(realx, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)bo[t], (int)(h * plane), 0));
          else
            f.b[t][q][h] = *reinterpret_cast<const realx *>(bq + h * plane + bo[t]);
      }
    }
  };
  realx4 acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int t = 0; t < CT; t++) acc[i][t] = realx4{0, 0, 0, 0};
  // the fragments of the current iteration have arrived once only the next
  // one's loads are outstanding (waited for here, whatever products follow)
  constexpr int kLoads = (RT + CT) * KC * kPW;
  static_assert(kLoads < 64, "vmcnt immediate");
  auto mac = [&](const Frag &f, int2 w) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitVm0 | (kLoads & 15) | ((kLoads >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < CT; t++) {
      if (CT > 1 && !((w.x >> (16 + t)) & 1)) continue;
#pragma unroll
      for (int i = 0; i < RT; i++) {
        if (RT > 1 && i >= nrt) break;
#pragma unroll
        for (int q = 0; q < KC; q++)
#pragma unroll
          for (int e = 0; e < 4; e++)
            acc[i][t] = mfma_real(f.a[i][q][e / kVW][e % kVW], f.b[t][q][e / kVW][e % kVW], acc[i][t]);
      }
    }
  };
  __syncthreads();
  const int n = __builtin_amdgcn_readfirstlane(nlst);
  if (ws < n) {
    // iterations (offset, k chunk); the next one's fragments are in flight
    // while the current one's are multiplied (past the last offset of the
    // slice, that offset's again)
    const int jlast = ws + (n - 1 - ws) / g.ws * g.ws;
    int j = ws, c = 0;
    auto entry = [&](int i) {
      const int2 e = lst[i];
      return make_int2(__builtin_amdgcn_readfirstlane(e.x), __builtin_amdgcn_readfirstlane(e.y));
    };
    int2 w = entry(j);
    int2 wn = w;
    Frag f0, f1;
    load(f0, w, c);
    auto advance = [&]() {
      c += KC;
      if (c >= kt) {
        c = 0;
        j = min(j + g.ws, jlast);
      }
      wn = entry(j);
    };
    const int nit = (jlast - ws) / g.ws * (kt / KC) + kt / KC;
    for (int it = nit >> 1; it > 0; it--) {
      advance();
      load(f1, wn, c);
      mac(f0, w);
      w = wn;
      advance();
      load(f0, wn, c);
      mac(f1, w);
      w = wn;
    }
    if (nit & 1) {
      load(f1, wn, c);  // (the count of outstanding loads that mac waits for)
      mac(f0, w);
    }
  }
  auto store = [&](int rt, int t, realx4 v) {
    const int col = col0 + 16 * t + (lane & 15);
    const int row = 16 * rt + 4 * (lane >> 4);
    if (col >= ncols || row >= g.r) return;
    const int pl = col / g.nrhs, rh = col - pl * g.nrhs;
    const int pz = pl % P, py = (pl / P) % P, px = pl / (P * P);
    const int fx = 2 * px + ((s >> 2) & 1), fy = 2 * py + ((s >> 1) & 1), fz = 2 * pz + (s & 1);
    const int A = g.levsta[l] + morton3(fx, fy, fz, l);
    real *Lp = g.L + ((size_t)rh * g.ncell + A) * g.r + row;
    if (row + 4 <= g.r) {
      *reinterpret_cast<realx4u *>(Lp) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 3; e++)
        if (row + e < g.r) Lp[e] = v[e];
    }
  };
  if (g.ws == 1) {
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int t = 0; t < CT; t++) store(rt0 + i, t, acc[i][t]);  // rows past r are not stored
    return;
  }
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int t = 0; t < CT; t++) red[(ws * RT * CT + i * CT + t) * 64 + lane] = acc[i][t];
  __syncthreads();
  for (int f = ws; f < RT * CT; f += g.ws) {
    realx4 v = red[f * 64 + lane];
    for (int q = 1; q < g.ws; q++) v += red[(q * RT * CT + f) * 64 + lane];
    store(rt0 + f / CT, f % CT, v);
  }
}

#ifdef SINGLE
// ---------------------------------------------------------------- split-BF16, few columns
// The split-BF16 products on few columns, blocked as the full-precision
// kernel: a block is one class, all 32 rows and CT tiles of 16 columns of one
// level, its waves take the offsets in slices; v_mfma_f32_16x16x32_bf16 takes
// the whole rank at once.  Two offsets' fragments are loaded while the two
// before are multiplied (past a slice's end: the zero operator).  Operators
// [k][row tile][hi, lo][lane][8] (k_few_layout): lane l holds row 16 tile +
// l % 16, columns 8 (l / 16) .. + 7.  Grids, hi and lo: [plane][slot][rhs][8],
// plane p the coefficients 8 p .. 8 p + 7 (k_few_scatter).
// Bound by latency and by the loads (6 KB per 6 products of 16 cycles at CT =
// 1).  M2L of 50021 particles, depth 3, 16 vectors: 86 us with 32-column
// tiles a wave and all offsets in turn, so 23; 4096, depth 2: 74 and 10.5.
__global__ void __launch_bounds__(256) k_few_layout(const float *__restrict__ K, __bf16 *__restrict__ out)
{
  const int o = blockIdx.x * 256 + threadIdx.x;  // [k][tile][lane][8]
  if (o >= (kNumOps + 1) * 1024) return;
  const int e = o & 7, lane = (o >> 3) & 63, t = (o >> 9) & 1, k = o >> 10;
  const int row = 16 * t + (lane & 15), col = 8 * (lane >> 4) + e;
  const float v = k < kNumOps ? K[(size_t)k * 1024 + col * 32 + row] : 0.0f;
  const __bf16 h = (__bf16)v;
  const size_t at = ((size_t)(2 * k + t) * 2 * 64 + lane) * 8 + e;
  out[at] = h;
  out[at + 64 * 8] = (__bf16)(v - (float)h);
}

// M [rhs][ncell][32] -> the hi and lo planes, a thread 8 coefficients of a cell and vector
__global__ void __launch_bounds__(256) k_few_scatter(GridArgs g, const float *__restrict__ M)
{
  const int total = (g.levsta[g.maxlev + 1] - g.levsta[g.minlev]) * g.nrhs * 4;
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= total) return;
  const int rhs = t % g.nrhs, p = t / g.nrhs & 3, A = g.levsta[g.minlev] + t / g.nrhs / 4;
  int l = g.minlev;
  while (A >= g.levsta[l + 1]) l++;
  int x, y, z;
  demorton3(A - g.levsta[l], l, x, y, z);
  const size_t slot = grid_slot(g, l, ((x & 1) << 2) | ((y & 1) << 1) | (z & 1), x >> 1, y >> 1, z >> 1);
  const float *src = M + ((size_t)rhs * g.ncell + A) * 32 + 8 * p;
  bf16x8 hi, lo;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const __bf16 h = (__bf16)src[e];
    hi[e] = h;
    lo[e] = (__bf16)(src[e] - (float)h);
  }
  const size_t dst = p * g.plane + (slot * g.nrhs + rhs) * 8;
  *reinterpret_cast<bf16x8 *>((__bf16 *)g.Mg0 + dst) = hi;
  *reinterpret_cast<bf16x8 *>((__bf16 *)g.Mg1 + dst) = lo;
}

template <int CT>
__global__ void __launch_bounds__(512) k_m2l_bf16_few(GridArgs g)
{
  constexpr int G = CT == 1 ? 2 : 1;  // offsets per iteration
  extern __shared__ __align__(16) unsigned char smem_raw[];
  f32x4 *red = reinterpret_cast<f32x4 *>(smem_raw);  // [slice][tile][64]
  __shared__ int2 lst[192];  // offsets to multiply: operator, slot shift
  __shared__ int nlst;
  const int lane = threadIdx.x & 63;
  const int ws = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int s = blockIdx.x & 7, gb = blockIdx.x >> 3;
  int l = g.minlev;
  while (l < g.maxlev && gb >= g.blk0[l + 1]) l++;
  const int P = 1 << (l - 1);
  const int PP = P + 2;
  const int ncols = P * P * P * g.nrhs;
  const int col0 = (gb - g.blk0[l]) * (16 * CT);
  if (ws == 0) {
    const WaveBox box = wave_box(col0, ncols, g.nrhs, P, 16 * CT);
    int n = 0;
    for (int q = 0; q < 3; q++) {
      const int v = 64 * q + lane;
      const int4 e = g.tab[s * kOffsets + min(v, kOffsets - 1)];
      const bool on = v < kOffsets && !ghost_step(box, e.z << 3, P);
      const unsigned long long act = __ballot(on);
      const int dx = (e.z >> 4) & 3, dy = (e.z >> 2) & 3, dz = e.z & 3;  // shift + 1
      if (on)
        lst[n + __popcll(act & ((1ull << lane) - 1))] =
            make_int2(e.x, (e.y * PP * PP * PP + (dx * PP + dy) * PP + dz) * g.nrhs);
      n += __popcll(act);
    }
    if (lane == 0) nlst = n;
  }
  unsigned bo[CT];
#pragma unroll
  for (int t = 0; t < CT; t++) {
    const int col = min(col0 + 16 * t + (lane & 15), ncols - 1);  // columns past the end are not stored
    const int pl = col / g.nrhs, rh = col - pl * g.nrhs;
    const int pz = pl % P, py = (pl / P) % P, px = pl / (P * P);
    const int slot = g.lvl_slot0[l] + (px * PP + py) * PP + pz;  // shifts count from (-1, -1, -1)
    bo[t] = (unsigned)(((lane >> 4) * g.plane + ((size_t)slot * g.nrhs + rh) * 8) * 2);
  }
  // few columns: operators and grids are far below 2 GB
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void *)g.Ka, 0, g.kbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rH = __builtin_amdgcn_make_buffer_rsrc((void *)g.Mg0, 0, g.gbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rL = __builtin_amdgcn_make_buffer_rsrc((void *)g.Mg1, 0, g.gbytes, 0x00020000);
  struct Frag {
    bf16x8 a[G][2][2], h[G][CT], l[G][CT];
  };
  constexpr int kLoads = G * (4 + 2 * CT);
  auto load = [&](Frag &f, int j, int n) {
#pragma unroll
    for (int u = 0; u < G; u++) {
      const int jj = j + u * g.ws;
      const int2 e = lst[min(jj, n - 1)];
      const int k = __builtin_amdgcn_readfirstlane(jj < n ? e.x : kZeroOp);
      const int so = __builtin_amdgcn_readfirstlane(e.y) * 16;
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int q = 0; q < 2; q++)
          f.a[u][t][q] = __builtin_bit_cast(
              bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rK, lane * 16 + (2 * t + q) * 1024, k * 4096, 0));
#pragma unroll
      for (int t = 0; t < CT; t++) {
        f.h[u][t] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rH, (int)bo[t], so, 0));
        f.l[u][t] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rL, (int)bo[t], so, 0));
      }
    }
  };
  f32x4 acc[2][CT];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int t = 0; t < CT; t++) acc[i][t] = f32x4{0, 0, 0, 0};
  auto mac = [&](const Frag &f) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitVm0 | (kLoads & 15) | ((kLoads >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < G; u++)
#pragma unroll
      for (int q = 0; q < 3; q++)  // hi hi, hi lo, lo hi
#pragma unroll
        for (int t = 0; t < CT; t++)
#pragma unroll
          for (int i = 0; i < 2; i++)
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.a[u][i][q == 2], q == 1 ? f.l[u][t] : f.h[u][t],
                                                                acc[i][t], 0, 0, 0);
  };
  __syncthreads();
  const int n = __builtin_amdgcn_readfirstlane(nlst);
  if (ws < n) {
    Frag f0, f1;
    int j = ws;
    const int step = G * g.ws, nit = (n - ws + step - 1) / step;
    load(f0, j, n);
    for (int it = nit >> 1; it > 0; it--) {
      load(f1, j += step, n);
      mac(f0);
      load(f0, j += step, n);
      mac(f1);
    }
    if (nit & 1) {
      load(f1, j, n);  // (the count of outstanding loads that mac waits for)
      mac(f0);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int t = 0; t < CT; t++) red[(ws * 2 * CT + i * CT + t) * 64 + lane] = acc[i][t];
  __syncthreads();
  for (int f = ws; f < 2 * CT; f += g.ws) {
    f32x4 v = red[f * 64 + lane];
    for (int q = 1; q < g.ws; q++) v += red[(q * 2 * CT + f) * 64 + lane];
    const int col = col0 + 16 * (f % CT) + (lane & 15);
    if (col >= ncols) continue;
    const int pl = col / g.nrhs, rh = col - pl * g.nrhs;
    const int pz = pl % P, py = (pl / P) % P, px = pl / (P * P);
    const int fx = 2 * px + ((s >> 2) & 1), fy = 2 * py + ((s >> 1) & 1), fz = 2 * pz + (s & 1);
    const int A = g.levsta[l] + morton3(fx, fy, fz, l);
    *reinterpret_cast<realx4u *>(g.L + ((size_t)rh * g.ncell + A) * 32 + 16 * (f / CT) + 4 * (lane >> 4)) = v;
  }
}
#endif

// ---------------------------------------------------------------- host side
static void offset_table(std::vector<int4> &tab)
{
  int Kt[343];
  ktable(Kt);
  tab.assign(8 * kOffsets, int4{0, 0, 0, 0});
  for (int s = 0; s < 8; s++) {
    const int sb[3] = {(s >> 2) & 1, (s >> 1) & 1, s & 1};
    int nv = 0;
    for (int vx = -2 - sb[0]; vx <= 3 - sb[0]; vx++)
      for (int vy = -2 - sb[1]; vy <= 3 - sb[1]; vy++)
        for (int vz = -2 - sb[2]; vz <= 3 - sb[2]; vz++) {
          if (vx >= -1 && vx <= 1 && vy >= -1 && vy <= 1 && vz >= -1 && vz <= 1) continue;
          const int v[3] = {vx, vy, vz};
          int sc = 0, packed = 0;
          for (int a = 0; a < 3; a++) {
            const int t = sb[a] + v[a];           // in [-2, 3]
            const int d = t >= 0 ? t / 2 : -1;    // floor(t / 2) in {-1, 0, 1}
            sc |= (t - 2 * d) << (2 - a);
            packed |= (d + 1) << (2 * (2 - a));
          }
          tab[s * kOffsets + nv] = int4{Kt[49 * (vx + 3) + 7 * (vy + 3) + (vz + 3)], sc, packed, 0};
          nv++;
        }
  }
}

// (s', d) steps of the source-stationary kernel for field classes split into
// groups of cls: for every source class s' and non-zero parent shift d, the
// operator index of each field class s of the group (offset v = 2d + s' - s),
// or the zero operator when v is a near-field offset; steps in which every
// class of the group is near are left out.  Record: [0] = s' | packed shift
// << 3, [1 + i/2] = operators of the group's classes i (low 16 bits) and
// i + 1 (high 16 bits), rest unused.  Layout [group][kSteps][kStepWords].
static void step_table(std::vector<int> &steps, int cls, int *nsteps)
{
  int Kt[343];
  ktable(Kt);
  const int ncg = 8 / cls;
  steps.assign((size_t)ncg * kSteps * kStepWords, 0);
  for (int cg = 0; cg < ncg; cg++) {
    int st = 0;
    for (int sc = 0; sc < 8; sc++)
      for (int dxi = 0; dxi < 3; dxi++)
        for (int dyi = 0; dyi < 3; dyi++)
          for (int dzi = 0; dzi < 3; dzi++) {
            if (dxi == 1 && dyi == 1 && dzi == 1) continue;
            int *e = &steps[((size_t)cg * kSteps + st) * kStepWords];
            e[0] = sc | (((dxi << 4) | (dyi << 2) | dzi) << 3);
            bool far_any = false;
            for (int i = 0; i < cls; i++) {
              const int c = cg * cls + i;
              const int vx = 2 * (dxi - 1) + ((sc >> 2) & 1) - ((c >> 2) & 1);
              const int vy = 2 * (dyi - 1) + ((sc >> 1) & 1) - ((c >> 1) & 1);
              const int vz = 2 * (dzi - 1) + (sc & 1) - (c & 1);
              const bool near = vx >= -1 && vx <= 1 && vy >= -1 && vy <= 1 && vz >= -1 && vz <= 1;
              far_any |= !near;
              const int k = near ? kZeroOp : Kt[49 * (vx + 3) + 7 * (vy + 3) + (vz + 3)];
              e[1 + (i >> 1)] |= k << (16 * (i & 1));
            }
            if (far_any) {
              st++;
            } else {
              for (int w = 0; w < kStepWords; w++) e[w] = 0;
            }
          }
    nsteps[cg] = st;
  }
}

// field classes per wave of the source-stationary variants (1 / 4, 7 / 5, 6),
// 0 otherwise, and their 32-column tiles per wave
static int ss_classes(int variant)
{
  return variant == 1 ? 8 : (variant == 4 || variant == 7 || variant == 8) ? 4 : (variant == 5 || variant == 6) ? 2 : 0;
}

static int ss_tiles(int variant) { return variant == 6 || variant == 7 || variant == 8 ? 2 : 1; }

// waves of a block of the full-precision kernel at most (their registers)
constexpr int real_max_waves(int rt, int ct) { return rt * ct <= 4 ? 16 : 8; }
// Tiles and slices of a block of the full-precision kernel, from the number
// of 16 x 16 tiles of L.  Larger blocks load fewer fragments per product,
// smaller ones fill the chip and even out its last round; beyond r = 32 the
// operators no longer fit L2, so the columns widen first.  Where the lines
// lie (us, fp32 unless said; columns x rank tiles):
//   r = 32:  37 x 2 tiles a class (1 vector, depth 4): 1 x 2 32, 1 x 1 33,
//            2 x 2 36; 73 x 2 (16 vectors, depth 3): 2 x 2 34, 1 x 2 35;
//            585 x 2: 2 x 2 203, 2 x 4 209; 4681 x 2: 2 x 4 1599, 2 x 2 1639;
//            fp64 37 x 2: 1 x 2 54, 2 x 1 60; 293 x 2: 2 x 1 242, 2 x 2 > 280
//   r = 108: 37 x 7: 1 x 4 204, 2 x 2 235, 2 x 4 260; 147 x 7: 2 x 4 664,
//            4 x 4 695; r = 256, 584 x 16: 4 x 4 9948, 2 x 4 11973;
//            fp64 147 x 7: 4 x 2 1291, 2 x 2 1657
// Slices: 8 (64K one vector 32 us, 2 slices 61), 4 once the blocks alone give
// several rounds (1M, 4 vectors: 4 slices 426, 8 442), 16 at the smallest.
// The pointer form takes the same column tiles and slices, so that its sums are
// the same to the bit, and one row tile a block (n = 8, 16 vectors, 131072
// particles 15.8 ms, with blocks of 1 x 1 35.8; 1M, one vector 180 us and 191).
static void real_shape(GridM2L *g)
{
  GridArgs &a = g->args;
  long long t16 = 0;  // tiles of 16 columns of one class
  for (int l = a.minlev; l <= a.maxlev; l++) t16 += ((1LL << (3 * (l - 1))) * a.nrhs + 15) / 16;
  const long long u = 8 * t16 * a.kt;
  auto take = [&](int rt, int ct) {
    a.rt = rt;
    a.ct = ct;
  };
  constexpr bool f64 = sizeof(real) == 8;
  if (g->variant == 2) take(2, 2);  // 32 columns of r = 32
  else if (g->variant == 3) take(2, 4);  // 64
  else if (a.kt <= 2) {
    if (f64 && a.kt == 2 && u >= 2 * 1024) take(2, 1);
    else if (!f64 && a.kt == 2 && u >= 8 * 4096) take(2, 4);
    else if (!f64 && a.kt == 2 && u >= 4 * 256) take(2, 2);
    else take(1, u >= 2 * 256 ? 2 : 1);
  } else {
    if (!f64 && u >= 16 * 2048) take(4, 4);
    else if (u >= 8 * 512) take(f64 ? 4 : 2, f64 ? 2 : 4);
    else take(1, u >= 4 * 384 ? 4 : u >= 2 * 256 ? 2 : 1);
  }
  a.nrg = (a.kt + a.rt - 1) / a.rt;
  int groups = 0;
  for (int l = a.minlev; l <= a.maxlev; l++) {
    a.blk0[l] = groups;
    groups += (int)(((1LL << (3 * (l - 1))) * a.nrhs + 16 * a.ct - 1) / (16 * a.ct));
  }
  a.blk0[a.maxlev + 1] = groups;
  g->nblocks = 8 * groups * a.nrg;
  a.ws = std::min(g->nblocks >= 2048 ? 4 : g->nblocks >= 128 ? 8 : 16, real_max_waves(a.rt, a.ct));
  // buffer loads: the planes of a k chunk within their 32-bit offsets
  a.buf = !g->flat && a.plane * sizeof(real) * (16 / kVW) < ((size_t)1 << 32);
  if (!a.buf) {
    a.rt = 1;
    a.nrg = a.kt;
    g->nblocks = 8 * groups * a.nrg;
  }
}

// Split-BF16 on fewer columns of the deepest level than this runs
// k_m2l_bf16_few, on more the source-stationary kernel, whose step parts then
// fill the chip (us, 4096 columns 80 against 141; 8192 of depth 5 119 against
// 104, of depth 4 106 against 103).
constexpr long long kFewColumns = 8192;

// Two tiles of 16 columns a block once they leave 128 blocks and more (us:
// 37 tiles a class 22.9 against 27.5, 72 22.7 against 26.6, 23 20.1 against
// 17.1, 8 13.1 against 10.5), with 8 offset slices, else 4.
static void few_shape(GridM2L *g)
{
  GridArgs &a = g->args;
  a.plane = ((g->nslots * a.nrhs * 16 + 4095) / 4096 * 4096 + 256) / 2;
  a.gbytes = (int)(a.plane * 4 * 2);
  long long t16 = 0;
  for (int l = a.minlev; l <= a.maxlev; l++) t16 += ((1LL << (3 * (l - 1))) * a.nrhs + 15) / 16;
  a.ct = t16 >= 32 ? 2 : 1;
  a.ws = a.ct == 2 ? 8 : 4;
  int groups = 0;
  for (int l = a.minlev; l <= a.maxlev; l++) {
    a.blk0[l] = groups;
    groups += (int)(((1LL << (3 * (l - 1))) * a.nrhs + 16 * a.ct - 1) / (16 * a.ct));
  }
  a.blk0[a.maxlev + 1] = groups;
  g->nblocks = 8 * groups;
}

int grid_m2l_create(GridM2L **out, int r, int maxlev, int nrhs, int form, const real *K, hipStream_t s,
                    int minlev, int variant, int variant_upper, int upper_split, const real *K_dev)
{
  *out = nullptr;
  // variant 0 on a deepest level of 64 K columns (parents x vectors) or more,
  // one block of 256 columns and both class groups per CU on 256 CUs: that
  // level with two tiles per wave and the class groups sharing the source
  // tiles (variant 8; fewer bytes moved per product), the levels above in a
  // launch of one tile per wave, their steps in 4 parts while they have
  // fewer blocks than 3 per CU (N = 1M uniform, depth 5, 16 vectors: 0.579
  // against 0.595 ms with variant 7 on the deepest level and 0.601 ms for
  // one launch of one tile per wave)
  if (variant == 0 && variant_upper == 0 && upper_split == 1 && form == BBFMM_M2L_BF16X2 && r == 32 &&
      maxlev > minlev && (long long)(1 << (3 * (maxlev - 1))) * nrhs >= 64 * 1024) {
    long long up_blocks = 0;
    for (int l = minlev; l < maxlev; l++) up_blocks += 2 * (((long long)(1 << (3 * (l - 1))) * nrhs + 127) / 128);
    variant = 8;
    variant_upper = 4;
    upper_split = up_blocks * 4 <= 3 * 256 ? 4 : 1;
  }
  if (upper_split < 1 || upper_split > 16)
    return set_error(BBFMM_E_ARG, "dense-grid M2L: step parts %d outside 1..16", upper_split);
  // step parts without an upper-level variant: the whole (single) launch
  int whole_split = 1;
  if (variant_upper == 0 && upper_split > 1) {
    whole_split = upper_split;
    upper_split = 1;
  }
  if (variant_upper != 0 && (!(ss_classes(variant_upper) && ss_classes(variant)) || variant_upper == 8))
    return set_error(BBFMM_E_ARG, "dense-grid M2L: a variant for the upper levels (%d) needs source-stationary "
                     "variants for both (1, 4 to 7 above the deepest level)", variant_upper);
  if (maxlev > kMaxLev) return set_error(BBFMM_E_ARG, "dense-grid M2L: maxlev %d > %d", maxlev, kMaxLev);
  if (minlev < kMinLev || minlev > maxlev)
    return set_error(BBFMM_E_ARG, "dense-grid M2L: first level %d outside [%d, %d]", minlev, kMinLev, maxlev);
  if (variant < 0 || variant > 8) return set_error(BBFMM_E_ARG, "dense-grid M2L: variant %d", variant);
  if ((variant == 1 || variant >= 4) && form != BBFMM_M2L_BF16X2)
    return set_error(BBFMM_E_ARG, "dense-grid M2L: the source-stationary variant is split-BF16 only");
  if (variant >= 2 && (form == BBFMM_M2L_PLAIN || r != 32))
    return set_error(BBFMM_E_ARG, "dense-grid M2L: tile variants are for the r = 32 MFMA forms");
  if (r < 1 || r > kMaxRank) return set_error(BBFMM_E_ARG, "dense-grid M2L: r=%d outside 1..%d", r, kMaxRank);
  if (form != BBFMM_M2L_PLAIN && r != 32 && r != 256)
    return set_error(BBFMM_E_ARG, "dense-grid M2L: the MFMA forms need r = 32 or 256 (got r=%d)", r);
#ifdef SINGLE
  if (form == BBFMM_M2L_BF16X2 && r != 32)
    return set_error(BBFMM_E_ARG, "the split-BF16 M2L form is built for r = 32 (got r=%d)", r);
  if (form == BBFMM_M2L_FP16X3 && r != 32)
    return set_error(BBFMM_E_ARG, "the split-FP16 M2L form is built for r = 32 (got r=%d)", r);
#else
  if (form != BBFMM_M2L_PLAIN) return set_error(BBFMM_E_ARG, "MFMA M2L forms need the fp32 build");
#endif
  GridM2L *g = new GridM2L();
  g->r = r;
  g->maxlev = maxlev;
  g->nrhs = nrhs;
  g->form = form;
  GridArgs &a = g->args;
  a.r = r;
  a.nrhs = nrhs;
  a.minlev = minlev;
  a.maxlev = maxlev;
  a.nsplit = 1;
  g->minlev = minlev;
  g->variant = variant;
  for (int l = 0; l <= maxlev + 1; l++) a.levsta[l] = ((1 << (3 * l)) - 1) / 7;
  a.ncell = a.levsta[maxlev + 1];
  size_t slots = 0;
  for (int l = minlev; l <= maxlev; l++) {
    a.lvl_slot0[l] = (int)slots;
    const size_t PP = ((size_t)1 << (l - 1)) + 2;
    slots += 8 * PP * PP * PP;
  }
  g->nslots = slots;
  {
    const size_t gb = slots * (size_t)nrhs * r * 2;  // split-BF16 grids: 2 bytes per value
    a.gbytes = gb < ((size_t)1 << 31) ? (int)gb : 0;
  }
  const bool real_form = form == BBFMM_M2L_PLAIN || form == BBFMM_M2L_FP32MFMA;
  a.kt = (r + 15) / 16;
  // plane stride an odd multiple of 256 bytes: the planes of a fragment start
  // on different L2 channels (at a multiple of 4 KB they all share one)
  a.plane = ((slots * nrhs * kVW * sizeof(real) + 4095) / 4096 * 4096 + 256) / sizeof(real);
  int tpw = 1, cpb;
  // variant 0 (automatic): split-BF16 takes the source-stationary blocking (4
  // classes per wave) once the deepest level has kFewColumns columns (parents
  // x vectors) or more, k_m2l_bf16_few below;
  // 1 / 4 / 5: source-stationary with 8 / 4 / 2 field classes per wave and
  // one 32-column tile, 6 / 7: 2 / 4 classes and two tiles per wave;
  // 2 / 3: class-stationary, one / two 32-column tiles per wave
  const long long deep = (long long)(1 << (3 * (maxlev - 1))) * nrhs;
  a.ss = 0;
  if (form == BBFMM_M2L_BF16X2) {
    a.few = variant == 0 && deep < kFewColumns;
    a.ss = variant == 0 && deep >= 8 * 1024 ? 4 : ss_classes(variant);
    if (a.few) a.ss = 0;
    a.ss_tpw = ss_tiles(variant);
    a.ss_pair = variant == 8;
  }
  if (real_form || a.few) {
    cpb = 1 << 30;  // blocks: real_shape, few_shape
  } else if (a.ss) {
    cpb = 4 * 32 * a.ss_tpw;  // 4 waves x 32 or 64 columns, one class group per block
  } else {
    // two tiles per wave once there are enough columns to fill the chip
    tpw = variant == 3 ? 2 : variant == 2 ? 1 : (deep >= 8 * 1024 ? 2 : 1);
    cpb = 4 * tpw * 32;
  }
  a.wave_cols = tpw * 32;
  if (whole_split > 1 && !a.ss) {
    delete g;
    return set_error(BBFMM_E_ARG, "dense-grid M2L: step parts need the split-BF16 source-stationary kernel");
  }
  // variant 0 on a deepest level of 8 K to 64 K columns (one launch, 4
  // classes and one tile per wave): each class group's step list in as many
  // parts as keep the blocks to one round at 3 per CU on 256 CUs (N = 262144
  // uniform, depth 4, 16 vectors: 146 column-group blocks, 5 parts)
  if (variant == 0 && variant_upper == 0 && whole_split == 1 && a.ss == 4 && a.ss_tpw == 1 && !a.ss_pair) {
    long long nb1 = 0;
    for (int l = minlev; l <= maxlev; l++) nb1 += 2 * (((long long)(1 << (3 * (l - 1))) * nrhs + cpb - 1) / cpb);
    whole_split = (int)std::max(1LL, std::min(16LL, 3 * 256 / nb1));
  }
  a.nsplit = whole_split;
  a.up_cell0 = a.levsta[minlev];
  a.up_ncell = a.levsta[maxlev + 1] - a.levsta[minlev];
  int nb = 0;
  for (int l = minlev; l <= maxlev; l++) {
    a.blk0[l] = nb;
    const long long cols = (long long)(1 << (3 * (l - 1))) * nrhs;
    nb += whole_split * (a.ss_pair ? 1 : a.ss ? 8 / a.ss : 8) * (int)((cols + cpb - 1) / cpb);
  }
  a.blk0[maxlev + 1] = nb;
  g->nblocks = nb;
  if (real_form) real_shape(g);
  if (a.few) few_shape(g);

  std::vector<int4> tab;
  offset_table(tab);
  std::vector<int> steps;
  step_table(steps, a.ss && !a.ss_pair ? a.ss : 8, a.nsteps);
  // levels above the deepest with their own class-group size: two launches
  const int ss_up = ss_classes(variant_upper), tpw_up = ss_tiles(variant_upper);
  size_t steps_up_off = 0;
  if (a.ss && ss_up && (ss_up != a.ss || tpw_up != a.ss_tpw || upper_split > 1) && maxlev > minlev) {
    g->nparts = 2;
    GridArgs &u = g->part[0], &d = g->part[1];
    u = a;
    d = a;
    u.maxlev = maxlev - 1;
    u.ss = ss_up;
    u.ss_tpw = tpw_up;
    u.ss_pair = 0;
    u.wave_cols = 32 * tpw_up;
    u.nsplit = upper_split;
    u.up_cell0 = a.levsta[minlev];
    u.up_ncell = a.levsta[maxlev] - a.levsta[minlev];
    const int cpb_up = 4 * 32 * tpw_up;
    int nbu = 0;
    for (int l = minlev; l <= maxlev - 1; l++) {
      u.blk0[l] = nbu;
      const long long cols = (long long)(1 << (3 * (l - 1))) * nrhs;
      nbu += upper_split * (8 / ss_up) * (int)((cols + cpb_up - 1) / cpb_up);
    }
    u.blk0[maxlev] = nbu;
    d.minlev = maxlev;
    d.blk0[maxlev] = 0;
    d.blk0[maxlev + 1] = a.blk0[maxlev + 1] - a.blk0[maxlev];
    g->part_blocks[0] = nbu;
    g->part_blocks[1] = d.blk0[maxlev + 1];
    std::vector<int> su;
    step_table(su, ss_up, u.nsteps);
    steps_up_off = steps.size();
    steps.insert(steps.end(), su.begin(), su.end());
  }
  int rc = BBFMM_OK;
  auto fail = [&](hipError_t e, const char *what) {
    rc = set_error(BBFMM_E_HIP, "dense-grid M2L: %s: %s", what, hipGetErrorString(e));
  };
  hipError_t e;
  if ((e = hipMalloc(&g->d_tab, sizeof(int4) * tab.size())) != hipSuccess) fail(e, "hipMalloc");
  if (rc == BBFMM_OK && (e = hipMemcpyAsync(g->d_tab, tab.data(), sizeof(int4) * tab.size(), hipMemcpyHostToDevice, s)) != hipSuccess)
    fail(e, "copy");
  if (rc == BBFMM_OK && (e = hipMalloc(&g->d_steps, sizeof(int) * steps.size())) != hipSuccess) fail(e, "hipMalloc");
  if (rc == BBFMM_OK && (e = hipMemcpyAsync(g->d_steps, steps.data(), sizeof(int) * steps.size(), hipMemcpyHostToDevice, s)) != hipSuccess)
    fail(e, "copy");
  // operators in the form's layout
  if (rc == BBFMM_OK) {
    if (real_form) {
      // the column-major operators go up as they are (unless the caller has
      // them on the device) and are laid out there
      const size_t nk = (size_t)kNumOps * a.kt * a.kt * 256, nc = (size_t)kNumOps * r * r;
      const size_t ng = sizeof(real) * a.plane * (16 * a.kt / kVW);
      real *up = nullptr;
      if ((e = hipMalloc(&g->d_K, sizeof(real) * nk)) != hipSuccess) fail(e, "hipMalloc");
      if (rc == BBFMM_OK && !K_dev) {
        if ((e = hipMalloc((void **)&up, sizeof(real) * nc)) != hipSuccess) fail(e, "hipMalloc");
        else if ((e = hipMemcpyAsync(up, K, sizeof(real) * nc, hipMemcpyHostToDevice, s)) != hipSuccess) fail(e, "copy");
      }
      if (rc == BBFMM_OK) {
        hipLaunchKernelGGL(k_real_layout, dim3((unsigned)((nk + 255) / 256)), dim3(256), 0, s, r, a.kt,
                           K_dev ? K_dev : up, (real *)g->d_K);
        if ((e = hipGetLastError()) != hipSuccess) fail(e, "operator layout");
      }
      if (rc == BBFMM_OK && (e = hipMalloc(&g->d_Mg0, ng)) != hipSuccess) fail(e, "hipMalloc");
      if (rc == BBFMM_OK && (e = hipMemsetAsync(g->d_Mg0, 0, ng, s)) != hipSuccess) fail(e, "memset");
      if (up) {
        (void)hipStreamSynchronize(s);
        (void)hipFree(up);
      }
    }
#ifdef SINGLE
    else if (a.few) {
      a.kbytes = (kNumOps + 1) * 4096;
      float *up = nullptr;
      if ((e = hipMalloc(&g->d_K, a.kbytes)) != hipSuccess) fail(e, "hipMalloc");
      if (rc == BBFMM_OK && !K_dev) {
        if ((e = hipMalloc((void **)&up, sizeof(float) * kNumOps * 1024)) != hipSuccess) fail(e, "hipMalloc");
        else if ((e = hipMemcpyAsync(up, K, sizeof(float) * kNumOps * 1024, hipMemcpyHostToDevice, s)) != hipSuccess)
          fail(e, "copy");
      }
      if (rc == BBFMM_OK) {
        hipLaunchKernelGGL(k_few_layout, dim3((kNumOps + 1) * 4), dim3(256), 0, s, K_dev ? K_dev : up, (__bf16 *)g->d_K);
        if ((e = hipGetLastError()) != hipSuccess) fail(e, "operator layout");
      }
      void **grids[2] = {&g->d_Mg0, &g->d_Mg1};
      for (void **gp : grids) {
        if (rc == BBFMM_OK && (e = hipMalloc(gp, a.gbytes)) != hipSuccess) fail(e, "hipMalloc");
        if (rc == BBFMM_OK && (e = hipMemsetAsync(*gp, 0, a.gbytes, s)) != hipSuccess) fail(e, "memset");
      }
      if (up) {
        (void)hipStreamSynchronize(s);
        (void)hipFree(up);
      }
    } else if (form == BBFMM_M2L_BF16X2) {
      // [k][kstep][hi/lo][lane][8]: lane l holds row l%32, k = 16*kstep + 8*(l/32) + e
      // one extra all-zero operator (kZeroOp) after the 316
      std::vector<__bf16> Kb((size_t)(kNumOps + 1) * 2 * 2 * 64 * 8, (__bf16)0.0f);
      for (int k = 0; k < kNumOps; k++)
        for (int ks = 0; ks < 2; ks++)
          for (int lane = 0; lane < 64; lane++)
            for (int q = 0; q < 8; q++) {
              const int row = lane & 31, col = 16 * ks + 8 * (lane >> 5) + q;
              const float v = K[(size_t)k * 32 * 32 + (size_t)col * 32 + row];
              const __bf16 h = (__bf16)v;
              const __bf16 lo = (__bf16)(v - (float)h);
              Kb[((((size_t)k * 2 + ks) * 2 + 0) * 64 + lane) * 8 + q] = h;
              Kb[((((size_t)k * 2 + ks) * 2 + 1) * 64 + lane) * 8 + q] = lo;
            }
      if ((e = hipMalloc(&g->d_K, sizeof(__bf16) * Kb.size())) != hipSuccess) fail(e, "hipMalloc");
      else if ((e = hipMemcpyAsync(g->d_K, Kb.data(), sizeof(__bf16) * Kb.size(), hipMemcpyHostToDevice, s)) != hipSuccess)
        fail(e, "copy");
      a.kbytes = (int)(sizeof(__bf16) * Kb.size());
      const size_t nb2 = sizeof(__bf16) * slots * nrhs * r;
      if (rc == BBFMM_OK && (e = hipMalloc(&g->d_Mg0, nb2)) != hipSuccess) fail(e, "hipMalloc");
      if (rc == BBFMM_OK && (e = hipMalloc(&g->d_Mg1, nb2)) != hipSuccess) fail(e, "hipMalloc");
      if (rc == BBFMM_OK && (e = hipMemsetAsync(g->d_Mg0, 0, nb2, s)) != hipSuccess) fail(e, "memset");
      if (rc == BBFMM_OK && (e = hipMemsetAsync(g->d_Mg1, 0, nb2, s)) != hipSuccess) fail(e, "memset");
    } else if (form == BBFMM_M2L_FP16X3) {
      // [k][kstep][term][lane][8]: lane l holds row l%32, k = 16*kstep + 8*(l/32) + e,
      // scaled by 2^(15 - e) for the largest |K| = f 2^e
      float kmax = 0.0f;
      for (size_t i = 0; i < (size_t)kNumOps * 32 * 32; i++) kmax = std::max(kmax, std::fabs((float)K[i]));
      int ke = 0;
      (void)std::frexp(kmax, &ke);
      const float ksc = std::ldexp(1.0f, 15 - ke);
      a.kscale_inv = std::ldexp(1.0f, ke - 15);
      std::vector<_Float16> Kh((size_t)kNumOps * 2 * 3 * 64 * 8);
      for (int k = 0; k < kNumOps; k++)
        for (int ks = 0; ks < 2; ks++)
          for (int lane = 0; lane < 64; lane++)
            for (int q = 0; q < 8; q++) {
              const int row = lane & 31, col = 16 * ks + 8 * (lane >> 5) + q;
              const float v = (float)K[(size_t)k * 32 * 32 + (size_t)col * 32 + row] * ksc;
              const _Float16 t1 = (_Float16)v;
              const float r1 = v - (float)t1;
              const _Float16 t2 = (_Float16)r1;
              const _Float16 t3 = (_Float16)(r1 - (float)t2);
              const size_t b = (((size_t)k * 2 + ks) * 3) * 64 * 8 + (size_t)lane * 8 + q;
              Kh[b] = t1;
              Kh[b + 64 * 8] = t2;
              Kh[b + 2 * 64 * 8] = t3;
            }
      if ((e = hipMalloc(&g->d_K, sizeof(_Float16) * Kh.size())) != hipSuccess) fail(e, "hipMalloc");
      else if ((e = hipMemcpyAsync(g->d_K, Kh.data(), sizeof(_Float16) * Kh.size(), hipMemcpyHostToDevice, s)) != hipSuccess)
        fail(e, "copy");
      // the host copy must outlive the asynchronous copy
      if (rc == BBFMM_OK && (e = hipStreamSynchronize(s)) != hipSuccess) fail(e, "sync");
      const size_t nb2 = sizeof(_Float16) * slots * nrhs * r;
      void **grids[3] = {&g->d_Mg0, &g->d_Mg1, &g->d_Mg2};
      for (void **gp : grids) {
        if (rc == BBFMM_OK && (e = hipMalloc(gp, nb2)) != hipSuccess) fail(e, "hipMalloc");
        if (rc == BBFMM_OK && (e = hipMemsetAsync(*gp, 0, nb2, s)) != hipSuccess) fail(e, "memset");
      }
      if (rc == BBFMM_OK && (e = hipMalloc(&g->d_lvl_max, sizeof(unsigned) * (kMaxLev + 1))) != hipSuccess)
        fail(e, "hipMalloc");
    }
#endif
  }
  if (rc == BBFMM_OK && g->nparts == 2 && g->part[0].nsplit > 1) {
    const size_t nx = (size_t)(g->part[0].nsplit - 1) * nrhs * g->part[0].up_ncell * 32;
    if ((e = hipMalloc(&g->d_Lx, sizeof(float) * nx)) != hipSuccess) fail(e, "hipMalloc");
  }
  if (rc == BBFMM_OK && g->nparts == 1 && a.nsplit > 1) {  // the whole launch in step parts
    const size_t nx = (size_t)(a.nsplit - 1) * nrhs * a.up_ncell * 32;
    if ((e = hipMalloc(&g->d_Lx, sizeof(float) * nx)) != hipSuccess) fail(e, "hipMalloc");
  }
  if (rc == BBFMM_OK && (e = hipStreamSynchronize(s)) != hipSuccess) fail(e, "sync");
  if (rc != BBFMM_OK) {
    grid_m2l_destroy(g);
    return rc;
  }
  a.tab = g->d_tab;
  a.steps = g->d_steps;
  a.Ka = g->d_K;
  a.Mg0 = g->d_Mg0;
  a.Mg1 = g->d_Mg1;
  a.Mg2 = g->d_Mg2;
  a.lvl_max = g->d_lvl_max;
  a.Lx = g->nparts == 1 ? g->d_Lx : nullptr;
  if (g->nparts == 2) {
    // everything from the final args (operator and grid pointers and sizes),
    // then each part's own levels, blocks, class-group size, tiles and steps
    for (int pi = 0; pi < 2; pi++) {
      const GridArgs own = g->part[pi];
      GridArgs &q = g->part[pi];
      q = a;
      q.minlev = own.minlev;
      q.maxlev = own.maxlev;
      for (int l = 0; l < kMaxLev + 2; l++) q.blk0[l] = own.blk0[l];
      q.ss = own.ss;
      q.ss_tpw = own.ss_tpw;
      q.ss_pair = own.ss_pair;
      q.wave_cols = own.wave_cols;
      for (int c = 0; c < 8; c++) q.nsteps[c] = own.nsteps[c];
      q.steps = g->d_steps + (pi == 0 ? steps_up_off : 0);
      q.nsplit = own.nsplit;
      q.up_cell0 = own.up_cell0;
      q.up_ncell = own.up_ncell;
      q.Lx = pi == 0 ? g->d_Lx : nullptr;
    }
  }
  *out = g;
  return BBFMM_OK;
}

void grid_m2l_set_flat(GridM2L *g, int flat)
{
  if (!g || g->flat == (flat != 0)) return;
  g->flat = flat != 0;
  if (g->form == BBFMM_M2L_PLAIN || g->form == BBFMM_M2L_FP32MFMA) real_shape(g);
}

void grid_m2l_destroy(GridM2L *g)
{
  if (!g) return;
  if (g->d_tab) (void)hipFree(g->d_tab);
  if (g->d_steps) (void)hipFree(g->d_steps);
  if (g->d_K) (void)hipFree(g->d_K);
  if (g->d_Mg0) (void)hipFree(g->d_Mg0);
  if (g->d_Mg1) (void)hipFree(g->d_Mg1);
  if (g->d_Mg2) (void)hipFree(g->d_Mg2);
  if (g->d_lvl_max) (void)hipFree(g->d_lvl_max);
  if (g->d_occ) (void)hipFree(g->d_occ);
  if (g->d_Lx) (void)hipFree(g->d_Lx);
  delete g;
}

template <int RT, int CT, int KC, bool BUF = true>
static int launch_real_t(const GridArgs &a, int nblocks, hipStream_t s)
{
  // (4 column tiles never come with more than 8 slices)
  constexpr int MAXW = !BUF && CT == 4 ? 8 : real_max_waves(RT, CT);
  const int lds = a.ws > 1 ? (int)(a.ws * RT * CT * 64 * sizeof(realx4)) : 0;
  const auto kernel = k_m2l_real<RT, CT, KC, MAXW, BUF>;
  hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(64 * a.ws), lds, s, a);
  BB_HIP(hipGetLastError());
  return BBFMM_OK;
}

// One k chunk per iteration; two where they come in pairs, in blocks of up to 8
// tiles.  In fp64 blocks of 1 x 4 that overruns the registers (143 of them in
// scratch): M2L of 80000 particles, n = 5, 3 vectors 1252 us, against 380 of
// the pointer form with its one chunk.
static int launch_real(const GridArgs &a, int nb, hipStream_t s)
{
  const bool two = a.kt % 2 == 0;
  if (!a.buf) {
    if (a.ct == 1) return launch_real_t<1, 1, 1, false>(a, nb, s);
    if (a.ct == 2) return launch_real_t<1, 2, 1, false>(a, nb, s);
    return launch_real_t<1, 4, 1, false>(a, nb, s);
  }
  switch (a.rt * 10 + a.ct) {
  case 11: return two ? launch_real_t<1, 1, 2>(a, nb, s) : launch_real_t<1, 1, 1>(a, nb, s);
  case 12: return two ? launch_real_t<1, 2, 2>(a, nb, s) : launch_real_t<1, 2, 1>(a, nb, s);
  case 14: return two ? launch_real_t<1, 4, 2>(a, nb, s) : launch_real_t<1, 4, 1>(a, nb, s);
#ifdef SINGLE
  case 22: return launch_real_t<2, 2, 2>(a, nb, s);  // r = 32 only
  case 24: return two ? launch_real_t<2, 4, 2>(a, nb, s) : launch_real_t<2, 4, 1>(a, nb, s);
  case 44: return launch_real_t<4, 4, 1>(a, nb, s);
#else
  case 21: return launch_real_t<2, 1, 2>(a, nb, s);  // r = 17 .. 32 only
  case 42: return launch_real_t<4, 2, 1>(a, nb, s);
#endif
  default: return set_error(BBFMM_E_ARG, "internal: block of %d x %d tiles", a.rt, a.ct);
  }
}

#ifdef SINGLE
// grids below 2 GB take the scalar-offset buffer-load form of the kernel
template <int CLS>
static void launch_ss(const GridM2L *g, const GridArgs &a, int nblocks, hipStream_t s)
{
  const dim3 grid((nblocks + 7) & ~7);
  const bool buf = a.gbytes > 0 && !g->flat;
  if (a.ss_pair) {
    if (buf)
      hipLaunchKernelGGL(k_m2l_mfma_ss_pair<true>, grid, dim3(512), 0, s, a);
    else
      hipLaunchKernelGGL(k_m2l_mfma_ss_pair<false>, grid, dim3(512), 0, s, a);
  } else if (CLS <= 4 && a.ss_tpw == 2) {  // two tiles per wave: 2 or 4 classes
    constexpr int C = CLS <= 4 ? CLS : 4;
    if (buf)
      hipLaunchKernelGGL((k_m2l_mfma_ss<C, 2, true>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((k_m2l_mfma_ss<C, 2, false>), grid, dim3(256), 0, s, a);
  } else if (buf)
    hipLaunchKernelGGL((k_m2l_mfma_ss<CLS, 1, true>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_m2l_mfma_ss<CLS, 1, false>), grid, dim3(256), 0, s, a);
}
#endif

int grid_m2l_leaf_grids(const GridM2L *g, void **hi, void **lo, int *slot0)
{
#ifdef SINGLE
  if (g && g->form == BBFMM_M2L_BF16X2 && !g->args.few && g->nrhs == 16 && g->args.minlev <= g->args.maxlev) {
    *hi = g->d_Mg0;
    *lo = g->d_Mg1;
    *slot0 = g->args.lvl_slot0[g->args.maxlev];
    return 1;
  }
#endif
  (void)g;
  (void)hi;
  (void)lo;
  (void)slot0;
  return 0;
}

int grid_m2l_occupied(GridM2L *g, const int *d_leafcnt, int nleaf, hipStream_t s)
{
  if (g->form != BBFMM_M2L_PLAIN && g->form != BBFMM_M2L_FP32MFMA) return BBFMM_OK;
  const size_t bytes = sizeof(unsigned long long) * (g->nslots / 64 + 2);
  BB_HIP(hipMalloc(&g->d_occ, bytes));
  BB_HIP(hipMemsetAsync(g->d_occ, 0, bytes, s));
  hipLaunchKernelGGL(k_mark_occupied, dim3((nleaf + 255) / 256), dim3(256), 0, s, g->args, d_leafcnt, nleaf,
                     (unsigned *)g->d_occ);
  BB_HIP(hipGetLastError());
  return BBFMM_OK;
}

int grid_m2l_run(GridM2L *g, const real *M, real *L, int ncell, hipStream_t s, hipEvent_t mid, int deep_in_grid,
                 bool zero_empty)
{
  GridArgs a = g->args;
  a.occ = zero_empty ? g->d_occ : nullptr;
  if (ncell != a.ncell) return set_error(BBFMM_E_ARG, "dense-grid M2L: ncell %d != %d", ncell, a.ncell);
  a.L = L;
  const long long cells = (long long)(a.levsta[a.maxlev + 1] - a.levsta[a.minlev]) * a.nrhs;
  const int sb = (int)((cells * (a.r / 8) + 255) / 256);
  switch (g->form) {
  case BBFMM_M2L_PLAIN:
  case BBFMM_M2L_FP32MFMA:
    hipLaunchKernelGGL(k_real_scatter, dim3((unsigned)((cells * (16 * a.kt / kVW) + 255) / 256)), dim3(256), 0, s, a, M);
    BB_HIP(hipGetLastError());
    if (mid) BB_HIP(hipEventRecord(mid, s));
    return launch_real(a, g->nblocks, s);
#ifdef SINGLE
  case BBFMM_M2L_BF16X2:
    if (a.few) {
      hipLaunchKernelGGL(k_few_scatter, dim3((unsigned)((cells * 4 + 255) / 256)), dim3(256), 0, s, a, M);
      BB_HIP(hipGetLastError());
      if (mid) BB_HIP(hipEventRecord(mid, s));
      const size_t lds = (size_t)a.ws * 2 * a.ct * 64 * sizeof(f32x4);
      if (a.ct == 1) hipLaunchKernelGGL(k_m2l_bf16_few<1>, dim3(g->nblocks), dim3(64 * a.ws), lds, s, a);
      else hipLaunchKernelGGL(k_m2l_bf16_few<2>, dim3(g->nblocks), dim3(64 * a.ws), lds, s, a);
      BB_HIP(hipGetLastError());
      return BBFMM_OK;
    }
    if (deep_in_grid) {  // the levels above the deepest only
      if (a.maxlev > a.minlev) {
        GridArgs u = a;
        u.maxlev = a.maxlev - 1;
        const long long ucells = (long long)(a.levsta[a.maxlev] - a.levsta[a.minlev]) * a.nrhs;
        hipLaunchKernelGGL(k_grid_scatter<BBFMM_M2L_BF16X2>, dim3((int)((ucells * (a.r / 8) + 255) / 256)), dim3(256),
                           0, s, u, M);
      }
    } else {
      hipLaunchKernelGGL(k_grid_scatter<BBFMM_M2L_BF16X2>, dim3(sb), dim3(256), 0, s, a, M);
    }
    BB_HIP(hipGetLastError());
    if (mid) BB_HIP(hipEventRecord(mid, s));
    if (a.ss) {  // one launch, or the upper levels then the deepest
      const int np = g->nparts;
      for (int pi = 0; pi < np; pi++) {
        GridArgs pa = np == 2 ? g->part[pi] : a;
        pa.L = L;
        const int nbk = np == 2 ? g->part_blocks[pi] : g->nblocks;
        if (nbk == 0) continue;
        if (pa.ss == 8)  // rounded up to whole rounds of the 8 XCDs; the extra blocks exit
          launch_ss<8>(g, pa, nbk, s);
        else if (pa.ss == 4)
          launch_ss<4>(g, pa, nbk, s);
        else
          launch_ss<2>(g, pa, nbk, s);
        if (pa.nsplit > 1) {  // the upper part's steps in parts: add parts 1.. to L
          const size_t n4 = (size_t)pa.nrhs * pa.up_ncell * 8;
          hipLaunchKernelGGL(k_m2l_add_parts, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, pa);
        }
      }
    } else if (a.wave_cols == 64)
      hipLaunchKernelGGL((k_m2l_mfma<BBFMM_M2L_BF16X2, 2>), dim3((g->nblocks + 7) & ~7), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((k_m2l_mfma<BBFMM_M2L_BF16X2, 1>), dim3((g->nblocks + 7) & ~7), dim3(256), 0, s, a);
    BB_HIP(hipGetLastError());
    return BBFMM_OK;
  case BBFMM_M2L_FP16X3:
    // per-level scales first (a fill kernel, not a memset: the solve may be captured)
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, a.lvl_max, kMaxLev + 1);
    hipLaunchKernelGGL(k_level_absmax, dim3(256, a.maxlev - a.minlev + 1), dim3(256), 0, s, a, M);
    hipLaunchKernelGGL(k_grid_scatter<BBFMM_M2L_FP16X3>, dim3(sb), dim3(256), 0, s, a, M);
    BB_HIP(hipGetLastError());
    if (mid) BB_HIP(hipEventRecord(mid, s));
    if (a.wave_cols == 64)
      hipLaunchKernelGGL((k_m2l_mfma<BBFMM_M2L_FP16X3, 2>), dim3((g->nblocks + 7) & ~7), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((k_m2l_mfma<BBFMM_M2L_FP16X3, 1>), dim3((g->nblocks + 7) & ~7), dim3(256), 0, s, a);
    BB_HIP(hipGetLastError());
    return BBFMM_OK;
#endif
  default: return set_error(BBFMM_E_ARG, "dense-grid M2L: unknown form %d", g->form);
  }
}

// ---------------------------------------------------------------- list MFMA (sparse trees)
// For trees that store only occupied cells (batches of instances) the dense
// grids do not exist; the same (class, offset) products are formed on
// gathered columns.  The field cells of levels >= 2 are grouped by sibling
// class s; for class s and its 189 offsets v (the dense-grid table order)
// vsrc[F * 189 + j] names the source cell F + v, or the zero cell ncell when
// that cell holds no points.  M is copied per solve to one 128-byte line a
// cell and vector, [rhs][ncell + 1] (bf16 hi and lo, or the 32 floats) with a
// zero last cell; k_m2l_list_packed multiplies them.

// A wave's units of k_m2l_list_packed, of 64 columns and of 32, and the first
// entry of each.
struct ListPart {
  int unit[2], count[2];
  long long entry[2];
};

struct ListArgs {
  int ncell, nrhs;
  int cls_off[9];  // class c cells: cls_cells[cls_off[c] .. cls_off[c + 1])
  const int *cls_cells;
  const int *vsrc;  // [ncell * 189]
  const int4 *tab;  // [8][189] (operator, ...)
  // blocks of at most cw cells x vb vectors, ws waves with their accumulators
  // in ts LDS slots each; in launch order, the classes interleaved in proportion to their
  // sizes, so that the blocks running at one time (and the contiguous range
  // each XCD takes) cover one region of the forest for all 8 classes and
  // share its source cells in L2
  int nblk, vb, cw, ts, ws;
  const int2 *blk;             // [nblk] first of cls_cells, cells
  const ListPart *part;        // [nblk * ws]
  const unsigned *unit;        // operator | entries << 16
  const int *esrc;             // entries: source cell
  const unsigned char *eslot;  // and target (cell within the block)
  const void *Ka;
  const void *M0;
  real *L;
  int kbytes;  // bytes of Ka
  int mbytes;  // bytes of M0 when below 2 GB (32-bit buffer offsets), else 0
};

struct ListM2L {
  int form = 0;
  int flat = 0;  // 1: pointer-form loads even on arrays below 2 GB
  ListArgs args{};
  int4 *d_tab = nullptr;
  int2 *d_blk = nullptr;
  ListPart *d_part = nullptr;
  unsigned *d_unit = nullptr;
  int *d_esrc = nullptr;
  unsigned char *d_eslot = nullptr;
  void *d_K = nullptr, *d_M0 = nullptr;
};

template <int FORM>
__global__ void __launch_bounds__(256) k_m2l_list_prep(ListArgs g, const real *__restrict__ M)
{
  const long long total = (long long)g.nrhs * g.ncell * 4;  // 8 coefficients per thread
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int ch = (int)(t & 3);
  const long long cr = t >> 2;
  const int A = (int)(cr % g.ncell), rh = (int)(cr / g.ncell);
  const real *src = M + ((size_t)rh * g.ncell + A) * 32 + ch * 8;
  const size_t row = (size_t)rh * (g.ncell + 1) + A;  // one 128-byte line a cell and vector
  if (FORM == BBFMM_M2L_BF16X2) {
    bf16x8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float v = (float)src[e];
      const __bf16 h = (__bf16)v;
      hi[e] = h;
      lo[e] = (__bf16)(v - (float)h);
    }
    __bf16 *d = (__bf16 *)g.M0 + row * 64 + ch * 8;  // hi, lo
    *reinterpret_cast<bf16x8 *>(d) = hi;
    *reinterpret_cast<bf16x8 *>(d + 32) = lo;
  } else {
    float *d = (float *)g.M0 + row * 32 + ch * 8;
#pragma unroll
    for (int e = 0; e < 8; e++) d[e] = (float)src[e];
  }
}

// slot j of offset v in class s's order (offset_table), or -1
static void slot_table(std::vector<int> &slot)
{
  slot.assign(8 * 343, -1);
  for (int s = 0; s < 8; s++) {
    const int sb[3] = {(s >> 2) & 1, (s >> 1) & 1, s & 1};
    int nv = 0;
    for (int vx = -2 - sb[0]; vx <= 3 - sb[0]; vx++)
      for (int vy = -2 - sb[1]; vy <= 3 - sb[1]; vy++)
        for (int vz = -2 - sb[2]; vz <= 3 - sb[2]; vz++) {
          if (vx >= -1 && vx <= 1 && vy >= -1 && vy <= 1 && vz >= -1 && vz <= 1) continue;
          slot[s * 343 + 49 * (vx + 3) + 7 * (vy + 3) + (vz + 3)] = nv++;
        }
  }
}

void slot_operators(std::vector<int> &op)
{
  std::vector<int4> tab;
  offset_table(tab);
  op.resize(tab.size());
  for (size_t i = 0; i < tab.size(); i++) op[i] = tab[i].x;
}

int class_slot(int s, int vx, int vy, int vz)
{
  static const std::vector<int> slot = [] {  // built once, thread-safe
    std::vector<int> t;
    slot_table(t);
    return t;
  }();
  if (vx < -3 || vx > 3 || vy < -3 || vy > 3 || vz < -3 || vz > 3) return -1;
  return slot[s * 343 + 49 * (vx + 3) + 7 * (vy + 3) + (vz + 3)];
}

typedef __attribute__((ext_vector_type(4))) int i32x4;

// Entries of a unit of R columns of k_m2l_list_packed: whole cells of vb vectors.
template <int R>
__host__ __device__ constexpr int unit_cells(int vb)
{
  return R / vb;
}

// What a block of k_m2l_list_packed multiplies: units of 64 columns and of 32
// (kind 0, 1), and their entries.
struct ListCount {
  int unit[2], entry[2];
};

// The units and entries of each block of k_m2l_list_packed (FILL: written;
// else counted).  An entry is a (target, source) pair of non-empty cells; a
// unit holds entries of one offset, the last of an offset those that are left.
// base: first unit and entry of the block (kind 0, then kind 1).  The cells'
// rows of vsrc are read into LDS whole (1.65M cells: 0.5 ms to count, 1.7 ms
// to write; with a wave a block and a lane a cell, 10.9 ms together).
template <bool FILL>
__global__ void __launch_bounds__(1024) k_m2l_list_pack(ListArgs g, const int *__restrict__ cls, ListCount *cnt,
                                                       const longlong2 *__restrict__ base, unsigned *unit, int *esrc,
                                                       unsigned char *eslot, ListPart *part)
{
  extern __shared__ int rows[];  // [cells][189]
  __shared__ int cells[128];
  __shared__ ListCount sum[256];  // inclusive over the offsets
  const int w = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int2 d = g.blk[w];
  const int4 *tab = g.tab + cls[w] * kOffsets;
  const int e64 = unit_cells<64>(g.vb), e32 = unit_cells<32>(g.vb);
  if (tid < d.y) cells[tid] = g.cls_cells[d.x + tid];
  __syncthreads();
  for (int i0 = tid; i0 < d.y * kOffsets; i0 += 8 * 1024) {
    int S[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int i = min(i0 + k * 1024, d.y * kOffsets - 1), j = i / kOffsets;
      S[k] = g.vsrc[(size_t)cells[j] * kOffsets + (i - j * kOffsets)];
    }
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (i0 + k * 1024 < d.y * kOffsets) rows[i0 + k * 1024] = S[k];
  }
  __syncthreads();
  // an offset of n entries: u0 units of 64 columns with the first m, then u1
  // (at most one) of 32 with the rest
  int n = 0;
  if (tid < kOffsets)
    for (int j = 0; j < d.y; j++) n += rows[j * kOffsets + tid] != g.ncell;
  const int rem = n % e64;
  const int u0 = n / e64 + (rem > e32 ? 1 : 0), u1 = rem > 0 && rem <= e32 ? 1 : 0;
  const int m = u1 ? n - rem : n;
  ListCount at{{u0, u1}, {m, n - m}};
  for (int k = 1; k < 256; k <<= 1) {
    if (tid < 256) sum[tid] = at;
    __syncthreads();
    if (tid >= k && tid < 256) {
      const ListCount o = sum[tid - k];
      for (int i = 0; i < 2; i++) {
        at.unit[i] += o.unit[i];
        at.entry[i] += o.entry[i];
      }
    }
    __syncthreads();
  }
  if (!FILL) {
    if (tid == kOffsets - 1) cnt[w] = at;
    return;
  }
  if (tid < 256) sum[tid] = at;
  __syncthreads();
  const ListCount tot = cnt[w];
  const longlong2 bs = base[w];
  const long long eb = bs.y + tot.entry[0];  // entries of kind 1
  if (tid < kOffsets) {
    const unsigned op = (unsigned)tab[tid].x;
    for (int i = 0; i < u0; i++)
      unit[bs.x + at.unit[0] - u0 + i] = op | (unsigned)min(e64, m - i * e64) << 16;
    if (u1) unit[bs.x + tot.unit[0] + at.unit[1] - 1] = op | (unsigned)rem << 16;
  }
  if (tid < g.ws) {
    ListPart p;
    for (int k = 0; k < 2; k++) {
      const int first = (int)((long long)tot.unit[k] * tid / g.ws);
      p.unit[k] = (int)bs.x + (k ? tot.unit[0] : 0) + first;
      p.count[k] = (int)((long long)tot.unit[k] * (tid + 1) / g.ws) - first;
      int v = 0;  // the offset that holds unit `first`
      while (v < kOffsets - 1 && sum[v].unit[k] <= first) v++;
      const int u = v ? sum[v - 1].unit[k] : 0, e = v ? sum[v - 1].entry[k] : 0;
      p.entry[k] = (k ? eb : bs.y) + e + (first - u) * (k ? 1 : e64);
    }
    part[w * g.ws + tid] = p;
  }
  const unsigned long long below = (1ull << lane) - 1;
  for (int v = tid >> 6; v < kOffsets; v += 16) {
    ListCount o{};
    if (v) o = sum[v - 1];
    const int mv = sum[v].entry[0] - o.entry[0];
    int first = 0;
    for (int j0 = 0; j0 < d.y; j0 += 64) {
      const int j = j0 + lane;
      const int S = j < d.y ? rows[j * kOffsets + v] : g.ncell;
      const unsigned long long mask = __ballot(S != g.ncell);
      const int at_v = first + __popcll(mask & below);
      if (S != g.ncell) {
        const long long k = at_v < mv ? bs.y + o.entry[0] + at_v : eb + o.entry[1] + at_v - mv;
        esrc[k] = S;
        eslot[k] = (unsigned char)j;
      }
      first += __popcll(mask);
    }
  }
}

__device__ __forceinline__ int quad_xor(int x, int p)
{
  return p == 1   ? __builtin_amdgcn_mov_dpp(x, 0xb1, 0xf, 0xf, false)
         : p == 2 ? __builtin_amdgcn_mov_dpp(x, 0x4e, 0xf, 0xf, false)
                  : __builtin_amdgcn_mov_dpp(x, 0x1b, 0xf, 0xf, false);
}
// exchange the odd rows of 16 lanes of x with the even rows of y; the upper
// half of x with the lower half of y
__device__ __forceinline__ void row_swap(unsigned &x, unsigned &y)
{
  const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}
__device__ __forceinline__ void half_swap(unsigned &x, unsigned &y)
{
  const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}

// 64 lines of 64 bytes, v[j] of lane 4 Q + i holding piece i ^ j of line
// 4 Q + j: to v[t] of lane 16 q + c holding piece q of line 16 t + c.
__device__ __forceinline__ void lines_to_columns(i32x4 (&v)[4], bool b0, bool b1)
{
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int x0 = v[0][e], x1 = v[1][e], x2 = v[2][e], x3 = v[3][e];
    const int y0 = b0 ? x1 : x0, y1 = b0 ? x0 : x1, y2 = b0 ? x3 : x2, y3 = b0 ? x2 : x3;
    // piece p of the lane's own line: lane i ^ p holds it in its register i
    unsigned u[4];
    u[0] = b1 ? y2 : y0;
    u[1] = quad_xor(b1 ? y3 : y1, 1);
    u[2] = quad_xor(b1 ? y0 : y2, 2);
    u[3] = quad_xor(b1 ? y1 : y3, 3);
    half_swap(u[0], u[2]);
    half_swap(u[1], u[3]);
    row_swap(u[0], u[1]);
    row_swap(u[2], u[3]);
#pragma unroll
    for (int t = 0; t < 4; t++) v[t][e] = u[t];
  }
}

// List M2L over the non-empty (target, source) pairs only.  In a sparse tree
// a cell has a source at 67 of the 189 offsets (a batch of Plummer spheres and
// surfaces, 1.65M cells), while 32 neighbouring cells have some source at 165
// of them: columns that stay with their cells, accumulated in registers,
// multiply 2.5 times as many as there are.  Here the accumulators of a
// block's 127 columns lie in LDS, one set a wave, and per offset only the
// cells with a source are packed into units of 64 or 32 columns, built once a
// plan: the unit's accumulators are read, multiplied into and written back.
// The block's units are split over its 4 waves (summed at the end in wave
// order), so that the cells in flight on an XCD are few enough for their
// sources to stay in its L2 (misses 32M lines -> 8.6M).
//
// Bound: the cache's return path (TD busy 84%, TA 73%; LDS about 70%).  A
// load whose adjacent lanes take 16 bytes each of different lines costs an
// access a lane, 64; so the 4 lanes of a quad take the 64 bytes of one line
// (16 accesses), and the columns are put where the products want them in
// registers (lines_to_columns; through ds_bpermute for 32 columns).
// Measured, split BF16, against 32 columns a wave with block-shared
// operators: 64 instances of 4096 to 131072 points 2970 -> 1840 us, 16 up to
// 32768 371 -> 204, 16 up to 65536 with 2 vectors 1553 -> 718, 8 up to 16384
// 120 -> 80.
template <int FORM, bool BUF>
__global__ void __launch_bounds__(256) k_m2l_list_packed(ListArgs g)
{
  extern __shared__ f32x4 accs[];  // [wave][row quad 8][slot ts]
  typedef __attribute__((ext_vector_type(8))) __bf16 b8;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x;
  const int lb = (b & 7) * ((g.nblk + 7) >> 3) + (b >> 3);
  if (lb >= g.nblk) return;  // whole block
  const int ts = g.ts, vb = g.vb;
  const int2 d = g.blk[lb];
  const ListPart part = g.part[lb * g.ws + wave];
  f32x4 *acc = accs + wave * 8 * ts;
  for (int i = lane; i < 8 * ts; i += 64) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  __syncthreads();
  const int rh0 = blockIdx.y * vb, nv = min(vb, g.nrhs - rh0);
  const int dummy = ts - 1;  // columns past a unit's last
  const int c = lane & 15, q = lane >> 4;
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void *)g.Ka, 0, g.kbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rM = __builtin_amdgcn_make_buffer_rsrc((void *)g.M0, 0, g.mbytes, 0x00020000);
  // two tiles of 16 columns: accumulator columns sl, sources b0, b1
  auto products = [&](const f32x4 *k, const i32x4 *b0, const i32x4 *b1, const int *sl) {
    f32x4 C[2][2];
    int a[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      a[i] = q * ts + sl[i];
      C[i][0] = acc[a[i]];
      C[i][1] = acc[a[i] + 4 * ts];
    }
    if (FORM == BBFMM_M2L_BF16X2) {
#pragma unroll
      for (int p = 0; p < 3; p++)  // hi x hi, hi x lo, lo x hi
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int m = 0; m < 2; m++)
            C[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, k[2 * m + (p == 2)]),
                                                              __builtin_bit_cast(b8, (p == 1 ? b1 : b0)[i]), C[i][m],
                                                              0, 0, 0);
    } else {
#pragma unroll
      for (int p = 0; p < 8; p++)  // step p: k = 4 q + p % 4 (+ 16)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int m = 0; m < 2; m++)
            C[i][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[2 * m + (p >> 2)][p & 3],
                                                           __builtin_bit_cast(f32x4, (p < 4 ? b0 : b1)[i])[p & 3],
                                                           C[i][m], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      acc[a[i]] = C[i][0];
      acc[a[i] + 4 * ts] = C[i][1];
    }
    wave_sync();
  };
  // the units of R columns
  auto phase = [&](auto rc) {
    constexpr int R = decltype(rc)::value, kind = R == 64 ? 0 : 1;
    constexpr int NB = R / 16, NE = R == 64 ? 1 : 2;
    struct Entry {
      int src[NE], slot[NE];
    };
    struct Buf {
      f32x4 k[4];
      i32x4 b0[NB], b1[NB];  // the two 64-byte halves of the lines
      int slot[NE];
    };
    const int nu = part.count[kind];
    if (nu <= 0) return;
    const unsigned *unit = g.unit + part.unit[kind];
    const int *esrc = g.esrc + part.entry[kind];
    const unsigned char *eslot = g.eslot + part.entry[kind];
    // R = 64: a lane reads the line and slot of column `lane`.  R = 32: the
    // lines of columns lane / 4 (+ 16), which its quad loads, and the slots
    // of columns lane % 16 (+ 16), which it multiplies.
    int es[NE], rs[NE], ed[NE], rd[NE];  // entry and vector of the line, of the slot
    bool ls[NE], ld[NE];
#pragma unroll
    for (int i = 0; i < NE; i++) {
      const int cs = R == 64 ? lane : 16 * i + (lane >> 2), cd = R == 64 ? lane : 16 * i + c;
      es[i] = cs / vb;
      rs[i] = cs - es[i] * vb;
      ed[i] = cd / vb;
      rd[i] = cd - ed[i] * vb;
      ls[i] = es[i] < unit_cells<R>(vb) && rs[i] < nv;
      ld[i] = ed[i] < unit_cells<R>(vb) && rd[i] < nv;
      rs[i] = (rh0 + rs[i]) * (g.ncell + 1);
    }
    auto word = [&](int i) { return i < nu ? unit[i] : 0u; };
    auto entries = [&](int start) {
      Entry e;
#pragma unroll
      for (int i = 0; i < NE; i++) {
        e.src[i] = esrc[start + es[i]];
        e.slot[i] = eslot[start + ed[i]];
      }
      return e;
    };
    auto load = [&](unsigned u, const Entry &e, Buf &t) {
      const int n = (int)(u >> 16), k = (int)(u & 0xffff);
      int row[NE];
#pragma unroll
      for (int i = 0; i < NE; i++) {
        row[i] = ls[i] && es[i] < n ? rs[i] + e.src[i] : g.ncell;
        t.slot[i] = ld[i] && ed[i] < n ? e.slot[i] * vb + rd[i] : dummy;
      }
      // load j: the 4 lanes of a quad share a line
      int rj[4];
      if (R == 64) {
        rj[0] = __builtin_amdgcn_mov_dpp(row[0], 0x00, 0xf, 0xf, false);
        rj[1] = __builtin_amdgcn_mov_dpp(row[0], 0x55, 0xf, 0xf, false);
        rj[2] = __builtin_amdgcn_mov_dpp(row[0], 0xaa, 0xf, 0xf, false);
        rj[3] = __builtin_amdgcn_mov_dpp(row[0], 0xff, 0xf, 0xf, false);
      } else {
        rj[0] = row[0];
        rj[1] = row[NE - 1];
      }
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const int piece = R == 64 ? (lane & 3) ^ j : lane & 3;
        if (BUF) {
          const int o = rj[j] * 128 + piece * 16;
          t.b0[j] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rM, o, 0, 0));
          t.b1[j] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rM, o + 64, 0, 0));
        } else {
          const char *o = (const char *)g.M0 + (size_t)rj[j] * 128 + piece * 16;
          t.b0[j] = *(const i32x4 *)o;
          t.b1[j] = *(const i32x4 *)(o + 64);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
        t.k[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rK, lane * 16 + i * 1024, k * 4096, 0));
    };
    auto run = [&](Buf &t) {
      if constexpr (R == 64) {
        lines_to_columns(t.b0, lane & 1, lane & 2);
        lines_to_columns(t.b1, lane & 1, lane & 2);
        unsigned sl[4];
        sl[0] = sl[2] = t.slot[0];
        half_swap(sl[0], sl[2]);
        sl[1] = sl[0];
        sl[3] = sl[2];
        row_swap(sl[0], sl[1]);
        row_swap(sl[2], sl[3]);
        products(t.k, t.b0, t.b1, (const int *)sl);
        products(t.k, t.b0 + 2, t.b1 + 2, (const int *)sl + 2);
      } else {
        // line 16 j + Q, piece i in lane 4 Q + i: to lane 16 i + Q
        const int from = 4 * (4 * c + q);
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int x = t.b0[j][e], y = t.b1[j][e];
            t.b0[j][e] = __builtin_amdgcn_ds_bpermute(from, x);
            t.b1[j][e] = __builtin_amdgcn_ds_bpermute(from, y);
          }
        products(t.k, t.b0, t.b1, t.slot);
      }
    };
    Buf X, Y;
    unsigned u0 = word(0), u1 = word(1), u2 = word(2);
    int start = 0;
    Entry e0 = entries(0);
    start += u0 >> 16;
    Entry e1 = entries(start);
    start += u1 >> 16;
    load(u0, e0, X);
    for (int i = 0;;) {
      // entries of unit i + 2, operator and sources of i + 1, products of i
      const Entry e2 = entries(start);
      start += u2 >> 16;
      load(u1, e1, Y);
      const unsigned u3 = word(i + 3);
      __builtin_amdgcn_sched_barrier(0);
      run(X);
      __builtin_amdgcn_sched_barrier(0);
      if (++i >= nu) break;
      e1 = entries(start);
      start += u3 >> 16;
      load(u2, e2, X);
      const unsigned u4 = word(i + 3);
      __builtin_amdgcn_sched_barrier(0);
      run(Y);
      __builtin_amdgcn_sched_barrier(0);
      if (++i >= nu) break;
      u0 = u2;
      u1 = u3;
      u2 = u4;
    }
  };
  phase(std::integral_constant<int, 64>());
  phase(std::integral_constant<int, 32>());
  __syncthreads();
  // columns of the block: 8 lanes a column
  for (int i = threadIdx.x; i < d.y * vb * 8; i += blockDim.x) {
    const int col = i >> 3, p = i & 7;
    const int cell = col / vb, rh = rh0 + col - cell * vb;
    f32x4 v = accs[p * ts + col];
    for (int w = 1; w < g.ws; w++) v += accs[(8 * w + p) * ts + col];
    if (rh < g.nrhs)
      *(f32x4 *)((float *)g.L + ((size_t)rh * g.ncell + g.cls_cells[d.x + cell]) * 32 + 4 * p) = v;
  }
}

#ifdef SINGLE
// The blocks of k_m2l_list_packed, their units and entries.
static int pack_lists(ListM2L *g, hipStream_t s)
{
  ListArgs &a = g->args;
  const int nv = (a.nrhs + 15) / 16;
  a.vb = (a.nrhs + nv - 1) / nv;
  // 128 slots and 4 waves: 64 KB of LDS, 2 blocks a CU.  64 slots leave the
  // units 40% emptier (batch of 1.65M cells 2391 us against 2050), 96 the same
  // time; 1 wave a block 2215, and 222 against 92 where 8 small instances
  // give too few blocks; 8 waves leave each too few units (2896)
  a.ts = 128;
  a.ws = 4;
  a.cw = (a.ts - 1) / a.vb;
  // the classes' blocks interleaved in proportion to their sizes
  std::vector<std::pair<double, int2>> order;
  for (int c = 0; c < 8; c++) {
    const int n = a.cls_off[c + 1] - a.cls_off[c], nb = (n + a.cw - 1) / a.cw;
    for (int k = 0; k < nb; k++) order.push_back({(k + 0.5) / nb, make_int2(c, a.cls_off[c] + k * a.cw)});
  }
  std::stable_sort(order.begin(), order.end(), [](const auto &x, const auto &y) { return x.first < y.first; });
  const int nb = a.nblk = (int)order.size();
  if (nb == 0) return BBFMM_OK;
  std::vector<int2> blk(nb);
  std::vector<int> cls(nb);
  for (int w = 0; w < nb; w++) {
    const int2 o = order[w].second;
    cls[w] = o.x;
    blk[w] = make_int2(o.y, std::min(a.cw, a.cls_off[o.x + 1] - o.y));
  }
  int *d_cls = nullptr;
  ListCount *d_cnt = nullptr;
  longlong2 *d_base = nullptr;
  std::vector<ListCount> cnt(nb);
  std::vector<longlong2> base(nb);
  const size_t rows = sizeof(int) * kOffsets * std::min(a.cw, a.cls_off[8]);
  const char *what = "hipMalloc";
  auto set_up = [&]() -> hipError_t {
    hipError_t e;
    if ((e = hipMalloc(&d_cls, sizeof(int) * nb)) != hipSuccess) return e;
    if ((e = hipMalloc(&d_cnt, sizeof(ListCount) * nb)) != hipSuccess) return e;
    if ((e = hipMalloc(&d_base, sizeof(longlong2) * nb)) != hipSuccess) return e;
    if ((e = hipMalloc(&g->d_blk, sizeof(int2) * nb)) != hipSuccess) return e;
    if ((e = hipMalloc(&g->d_part, sizeof(ListPart) * nb * a.ws)) != hipSuccess) return e;
    a.blk = g->d_blk;
    a.part = g->d_part;
    what = "list set-up";
    if ((e = hipMemcpyAsync(d_cls, cls.data(), sizeof(int) * nb, hipMemcpyHostToDevice, s)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(g->d_blk, blk.data(), sizeof(int2) * nb, hipMemcpyHostToDevice, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_m2l_list_pack<false>, dim3(nb), dim3(1024), rows, s, a, d_cls, d_cnt, d_base, nullptr, nullptr,
                       nullptr, nullptr);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(cnt.data(), d_cnt, sizeof(ListCount) * nb, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
    long long nu = 0, ne = 0;
    for (int w = 0; w < nb; w++) {
      base[w] = make_longlong2(nu, ne);
      nu += cnt[w].unit[0] + cnt[w].unit[1];
      ne += (long long)cnt[w].entry[0] + cnt[w].entry[1];
    }
    what = "list of more than 2^31 units";
    if (nu > INT_MAX) return hipErrorInvalidValue;
    what = "hipMalloc";
    if ((e = hipMalloc(&g->d_unit, sizeof(unsigned) * (nu + 1))) != hipSuccess) return e;
    // a unit's entries are read as if it were full, two units ahead
    const size_t ahead = 256;
    if ((e = hipMalloc(&g->d_esrc, sizeof(int) * (ne + ahead))) != hipSuccess) return e;
    if ((e = hipMalloc(&g->d_eslot, (size_t)ne + ahead)) != hipSuccess) return e;
    what = "list set-up";
    if ((e = hipMemcpyAsync(d_base, base.data(), sizeof(longlong2) * nb, hipMemcpyHostToDevice, s)) != hipSuccess)
      return e;
    hipLaunchKernelGGL(k_m2l_list_pack<true>, dim3(nb), dim3(1024), rows, s, a, d_cls, d_cnt, d_base, g->d_unit, g->d_esrc,
                       g->d_eslot, g->d_part);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return hipStreamSynchronize(s);
  };
  const hipError_t rc = set_up();
  if (d_cls) (void)hipFree(d_cls);
  if (d_cnt) (void)hipFree(d_cnt);
  if (d_base) (void)hipFree(d_base);
  if (rc != hipSuccess) return set_error(BBFMM_E_HIP, "list M2L: %s: %s", what, hipGetErrorString(rc));
  a.unit = g->d_unit;
  a.esrc = g->d_esrc;
  a.eslot = g->d_eslot;
  return BBFMM_OK;
}
#endif

int list_m2l_create(ListM2L **out, int r, int nrhs, int form, const real *K, int ncell, const int *cls_off,
                    const int *d_cls_cells, const int *d_vsrc, hipStream_t s)
{
  *out = nullptr;
#ifndef SINGLE
  (void)r; (void)nrhs; (void)form; (void)K; (void)ncell; (void)cls_off; (void)d_cls_cells; (void)d_vsrc; (void)s;
  return set_error(BBFMM_E_ARG, "the list MFMA M2L needs the fp32 build");
#else
  if (r != 32) return set_error(BBFMM_E_ARG, "the list MFMA M2L is built for r = 32 (got r=%d)", r);
  if (form != BBFMM_M2L_BF16X2 && form != BBFMM_M2L_FP32MFMA)
    return set_error(BBFMM_E_ARG, "the list MFMA M2L runs the split-BF16 or FP32 MFMA form");
  ListM2L *g = new ListM2L();
  g->form = form;
  ListArgs &a = g->args;
  a.ncell = ncell;
  a.nrhs = nrhs;
  for (int c = 0; c <= 8; c++) a.cls_off[c] = cls_off[c];
  std::vector<int4> tab;
  offset_table(tab);
  int rc = BBFMM_OK;
  auto fail = [&](hipError_t e, const char *what) {
    rc = set_error(BBFMM_E_HIP, "list M2L: %s: %s", what, hipGetErrorString(e));
  };
  hipError_t e;
  if ((e = hipMalloc(&g->d_tab, sizeof(int4) * tab.size())) != hipSuccess) fail(e, "hipMalloc");
  if (rc == BBFMM_OK && (e = hipMemcpy(g->d_tab, tab.data(), sizeof(int4) * tab.size(), hipMemcpyHostToDevice)) != hipSuccess)
    fail(e, "copy");
  if (rc == BBFMM_OK) {
    if (form == BBFMM_M2L_BF16X2) {
      // 16x16x32 products: [operator][row half][hi, lo][lane][8]
      std::vector<__bf16> Kb((size_t)kNumOps * 2 * 2 * 64 * 8);
      for (int k = 0; k < kNumOps; k++)
        for (int m = 0; m < 2; m++)
          for (int lane = 0; lane < 64; lane++)
            for (int q = 0; q < 8; q++) {
              const int row = 16 * m + (lane & 15), col = 8 * (lane >> 4) + q;
              const float v = K[(size_t)k * 32 * 32 + (size_t)col * 32 + row];
              const __bf16 h = (__bf16)v;
              Kb[((((size_t)k * 2 + m) * 2 + 0) * 64 + lane) * 8 + q] = h;
              Kb[((((size_t)k * 2 + m) * 2 + 1) * 64 + lane) * 8 + q] = (__bf16)(v - (float)h);
            }
      if ((e = hipMalloc(&g->d_K, sizeof(__bf16) * Kb.size())) != hipSuccess) fail(e, "hipMalloc");
      else if ((e = hipMemcpy(g->d_K, Kb.data(), sizeof(__bf16) * Kb.size(), hipMemcpyHostToDevice)) != hipSuccess)
        fail(e, "copy");
    } else {
      // 16x16x4 products, k = 4 (lane / 16) + step % 4 (+ 16): [operator][row half][step / 4][lane][step % 4]
      std::vector<float> Kf((size_t)kNumOps * 64 * 16);
      for (int k = 0; k < kNumOps; k++)
        for (int m = 0; m < 2; m++)
          for (int lane = 0; lane < 64; lane++)
            for (int p = 0; p < 8; p++) {
              const int row = 16 * m + (lane & 15), col = 4 * (lane >> 4) + (p & 3) + 16 * (p >> 2);
              Kf[((((size_t)k * 2 + m) * 2 + (p >> 2)) * 64 + lane) * 4 + (p & 3)] =
                  K[(size_t)k * 32 * 32 + (size_t)col * 32 + row];
            }
      if ((e = hipMalloc(&g->d_K, sizeof(float) * Kf.size())) != hipSuccess) fail(e, "hipMalloc");
      else if ((e = hipMemcpy(g->d_K, Kf.data(), sizeof(float) * Kf.size(), hipMemcpyHostToDevice)) != hipSuccess)
        fail(e, "copy");
    }
  }
  // the sources: one 128-byte line a cell and vector, the last a zero cell
  const size_t mb = (size_t)128 * nrhs * (ncell + 1);
  a.kbytes = kNumOps * 4096;
  a.mbytes = mb < ((size_t)1 << 31) ? (int)mb : 0;
  if (rc == BBFMM_OK && (e = hipMalloc(&g->d_M0, mb)) != hipSuccess) fail(e, "hipMalloc");
  if (rc == BBFMM_OK && (e = hipMemsetAsync(g->d_M0, 0, mb, s)) != hipSuccess) fail(e, "memset");
  if (rc == BBFMM_OK && (e = hipStreamSynchronize(s)) != hipSuccess) fail(e, "sync");
  if (rc != BBFMM_OK) {
    list_m2l_destroy(g);
    return rc;
  }
  a.cls_cells = d_cls_cells;
  a.vsrc = d_vsrc;
  a.tab = g->d_tab;
  a.Ka = g->d_K;
  a.M0 = g->d_M0;
  if ((rc = pack_lists(g, s)) != BBFMM_OK) {
    list_m2l_destroy(g);
    return rc;
  }
  *out = g;
  return BBFMM_OK;
#endif
}

void list_m2l_set_flat(ListM2L *g, int flat)
{
  if (g) g->flat = flat != 0;
}

void list_m2l_destroy(ListM2L *g)
{
  if (!g) return;
  for (void *p : {(void *)g->d_tab, (void *)g->d_blk, (void *)g->d_part, (void *)g->d_unit, (void *)g->d_esrc,
                  (void *)g->d_eslot, g->d_K, g->d_M0})
    if (p) (void)hipFree(p);
  delete g;
}

int list_m2l_run(ListM2L *g, const real *M, real *L, hipStream_t s, hipEvent_t mid)
{
  ListArgs a = g->args;
  a.L = L;
  const long long prep = (long long)a.nrhs * a.ncell * 4;
  const int pb = (int)((prep + 255) / 256);
#ifdef SINGLE
  const bool bf16 = g->form == BBFMM_M2L_BF16X2;
  const bool buf = a.mbytes > 0 && !g->flat;  // grids below 2 GB: 32-bit buffer offsets
  if (bf16) hipLaunchKernelGGL(k_m2l_list_prep<BBFMM_M2L_BF16X2>, dim3(pb), dim3(256), 0, s, a, M);
  else hipLaunchKernelGGL(k_m2l_list_prep<BBFMM_M2L_FP32MFMA>, dim3(pb), dim3(256), 0, s, a, M);
  BB_HIP(hipGetLastError());
  if (mid) BB_HIP(hipEventRecord(mid, s));
  if (a.nblk > 0) {
    const dim3 grid((a.nblk + 7) & ~7, (a.nrhs + a.vb - 1) / a.vb);
    const size_t lds = sizeof(f32x4) * 8 * a.ts * a.ws;
    auto launch = [&](auto *k) { hipLaunchKernelGGL(k, grid, dim3(64 * a.ws), lds, s, a); };
    if (bf16 && buf) launch(k_m2l_list_packed<BBFMM_M2L_BF16X2, true>);
    else if (bf16) launch(k_m2l_list_packed<BBFMM_M2L_BF16X2, false>);
    else if (buf) launch(k_m2l_list_packed<BBFMM_M2L_FP32MFMA, true>);
    else launch(k_m2l_list_packed<BBFMM_M2L_FP32MFMA, false>);
  }
  BB_HIP(hipGetLastError());
  return BBFMM_OK;
#else
  (void)pb; (void)M; (void)s; (void)mid;
  return set_error(BBFMM_E_ARG, "the list MFMA M2L needs the fp32 build");
#endif
}

} // namespace bb
