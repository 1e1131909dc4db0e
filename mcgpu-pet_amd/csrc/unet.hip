// unet.hip — learned scatter surrogate: a small 3D U-Net on the rebinned scatter sinogram,
// trained on simulator output (no reference counterpart; the reference only runs Monte Carlo),
// and the device rebinning of sinograms onto its grid.
//
// Every convolution product (forward, input gradient, weight gradient) is an implicit GEMM
//   C[m][n] (+)= sum_k A(m, k) * B(k, n)
// on BF16 MFMA tiles (v_mfma_f32_16x16x32_bf16: 16x16 outputs, K = 32 per instruction, FP32
// accumulation); operands are rounded to BF16 (im2col is never materialised). Parameters, optimiser
// state, the input, the output and all gradients are kept in FP32; the activations between the
// layers exist only as the BF16 operands of the products that read them. k_conv_tiled, k_conv_planes,
// k_conv_cols and k_conv_short hold the forward and input-gradient products, k_bwgt_tiled and
// k_bwgt_point the weight gradients; k_gemm is a plain GEMM on the same tiles, used by the self test
// of the MFMA operand layout.
// MFMA lane layout (16x16x32 BF16): lane l holds A row (l % 16), k = 8 (l / 16) .. +7; B column
// (l % 16), the same k; the accumulator's 4 values are rows 4 (l / 16) .. +3 of column (l % 16).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "host_internal.h"
#include "mcpet.h"
#include "runtime_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ __bf16 to_bf16(float x) { return (__bf16)x; }   // round to nearest even

// ------------------------------------------------------------------ the plain GEMM (self test)

struct Dense {      // row-major matrix, element (r, c) at p[r * ld + c]
  const float* p;
  int rows, cols, ld;
  __device__ __forceinline__ float operator()(int r, int c) const { return (r < rows && c < cols) ? p[(size_t)r * ld + c] : 0.0f; }
};

// Block: 4 waves; block tile 32 (m) x 64 (n); wave w owns columns [16 w, 16 w + 16) and both
// 16-row halves. Grid: (ceil(N/64), ceil(M/32), split). Split > 1 accumulates partial sums
// over K ranges with atomics.
template <class AOp, class BOp>
__global__ __launch_bounds__(256) void k_gemm(AOp A, BOp B, float* __restrict__ C, int M, int N, int K, int ldc,
                                              const float* __restrict__ bias, int k_per_split, int accumulate)
{
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 64 + wave * 16;
  const int kb = blockIdx.z * k_per_split;
  const int ke = min(K, kb + k_per_split);
  floatx4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = kb; k0 < ke; k0 += 32) {
    bf16x8 a0, a1, b;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int k = k0 + kg * 8 + j;
      const bool in = k < ke;
      a0[j] = to_bf16(in ? A(m0 + r, k) : 0.0f);
      a1[j] = to_bf16(in ? A(m0 + 16 + r, k) : 0.0f);
      b[j] = to_bf16(in ? B(k, n0 + r) : 0.0f);
    }
    acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b, acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b, acc1, 0, 0, 0);
  }
  const int col = n0 + r;
  if (col >= N) return;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row0 = m0 + kg * 4 + i, row1 = row0 + 16;
    if (row0 < M) {
      float v = acc0[i];
      if (accumulate) atomicAdd(&C[(size_t)row0 * ldc + col], v);
      else C[(size_t)row0 * ldc + col] = v + (bias ? bias[row0] : 0.0f);
    }
    if (row1 < M) {
      float v = acc1[i];
      if (accumulate) atomicAdd(&C[(size_t)row1 * ldc + col], v);
      else C[(size_t)row1 * ldc + col] = v + (bias ? bias[row1] : 0.0f);
    }
  }
}

// accumulate: add into C with atomics (C holds earlier partial sums); else store (+ bias).
template <class AOp, class BOp>
hipError_t gemm(AOp A, BOp B, float* C, int M, int N, int K, int ldc, const float* bias, int split, bool accumulate,
                hipStream_t st)
{
  if (M <= 0 || N <= 0) return hipSuccess;
  if (split < 1) split = 1;
  if (split > 1) accumulate = true;
  int kps = (K + split - 1) / split;
  kps = (kps + 31) / 32 * 32;
  split = (K + kps - 1) / kps;
  if (split < 1) split = 1;
  dim3 grid((N + 63) / 64, (M + 31) / 32, split);
  hipLaunchKernelGGL((k_gemm<AOp, BOp>), grid, dim3(256), 0, st, A, B, C, M, N, K, ldc, bias, kps, accumulate ? 1 : 0);
  return hipGetLastError();
}

// ------------------------------------------------------------------ convolution kernels
//
// Each convolution product is one implicit GEMM with a tap-major reduction index
// k = t * Cp + c (t: kernel tap, 27 for 3x3x3 or 1 for 1x1x1; c: channel, padded to
// Cp = roundup(C, 8)), so a lane's 8 consecutive k share one tap: one address and bounds
// computation, then one 16-byte load.
//   FWD   : Y[co][p]        = act(sum_k Wf[co][k] X[c][s p + d_t] + b[co])    m = co, n = output voxel
//   BDATA : dX[ci][p]      (+)= mask(sum_k Wb[ci][k] dY[c][q], s q + d_t = p)  m = ci, n = input voxel
// and the weight gradient (k_bwgt_tiled, k_bwgt_point) is
//           G[co][ci][t]    += sum_q dY[co][q] X[ci][s q + d_t]              m = co, n = ci, k = q
// Wf, Wb: BF16 copies of the FP32 weights in those layouts (zero padded, in MFMA fragment order). FWD
// and BDATA read their B tensor from a channels-last BF16 copy ([voxel][Cp], padding zero), so a
// lane's 8 channels are one 16-byte load; their epilogues write such a copy of what they produce: FWD
// nothing else (but the output layer, which writes FP32), as the next product, the weight gradient and, by its
// sign, the ReLU mask read it; BDATA beside the FP32 gradient, which the bias gradient reads.

// FWDUP: FWD of a concatenation whose first Cu channels are the nearest x2 upsampling of a tensor of
// half the size, read where it is.
enum { FWD = 0, BDATA = 1, FWDUP = 2 };

// Where an epilogue writes a channels-last BF16 copy of its output: element (m, n) at
// p[n * ld + off + m] (p null: no copy).
struct ClOut {
  __bf16* p;
  int ld, off;
};

struct ConvK {
  const __bf16* A;     // FWD, BDATA: BF16 weights [Kp / 32][nrb][64 lanes][8] (k_derive)
  const __bf16* Xl;    // FWD: input activations [D][H][W][ldx]; BDATA: dY [oD][oH][oW][ldx] (channels-last BF16)
  const __bf16* Xu;    // FWDUP: channels 0 .. Cu - 1 at half size, [D/2][H/2][W/2][ldu]; Xl holds the others
  int ldx, ldu, Cu;
  ClOut o1;            // FWD, BDATA: channels-last copy of the output
  float* C;            // FWD: Y [M][N], may be null; BDATA: dX [M][N]
  const float* bias;   // FWD
  const __bf16* mask;  // BDATA: the layer input's channels from mask0 on, [N][ldm] (gradient zero where it is
  int ldm, mask0;      // not positive: the ReLU before it); may be null
  const float* res;    // FWD with M = 1: added to the output; may be null
  int relu, beta;      // FWD: ReLU on the output; BDATA: add to C
  int M, N, K, Kp;     // GEMM sizes; Kp: K padded to whole k-steps
  int nrb;             // 16-row blocks of A
  int Cb, Cbp;         // channels of the B tensor (FWD: Cin; BDATA: Cout) and Cb rounded up to 8
  int D, H, W, oD, oH, oW, ks, stride, T;
  size_t sX, sXu, sC, sR;   // from one sample to the next (blockIdx.z): B tensor(s); C; res
  int samples;
};

// the tensors of sample z
__device__ __forceinline__ void to_sample(ConvK& a, size_t z)
{
  a.Xl += z * a.sX;
  if (a.Xu) a.Xu += z * a.sXu;
  if (a.C) a.C += z * a.sC;
  if (a.res) a.res += z * a.sR;
  if (a.mask) a.mask += z * a.N * a.ldm;
  if (a.o1.p) a.o1.p += z * a.N * a.o1.ld;
}

// What the epilogue of rows row0 .. row0 + 3 of column n reads: FWD the bias, BDATA the ReLU mask (the
// sign of the forward's BF16 copy) and what it adds to. Read apart from the stores, so that a wave's
// reads are in flight together.
struct ConvIn {
  float c[4];   // FWD: bias; BDATA: the earlier C, 0 without beta
  bool on[4];   // BDATA: not masked
};
template <int MODE>
__device__ __forceinline__ ConvIn conv_in(const ConvK& a, int row0, int n)
{
  ConvIn q;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    q.c[v] = 0.0f;
    q.on[v] = true;
  }
  if (row0 >= a.M || (MODE == BDATA && n >= a.N)) return q;
  if (MODE != BDATA) {
#pragma unroll
    for (int v = 0; v < 4; v++) q.c[v] = row0 + v < a.M ? a.bias[row0 + v] : 0.0f;
    return q;
  }
  if (a.beta)
#pragma unroll
    for (int v = 0; v < 4; v++) q.c[v] = row0 + v < a.M ? a.C[(size_t)(row0 + v) * a.N + n] : 0.0f;
  if (a.mask && row0 + 3 >= a.mask0) {
    const __bf16* m = a.mask + (size_t)n * a.ldm - a.mask0;
    if ((a.mask0 & 3) == 0) {   // ldm is a multiple of 8: the four exist
      const bf16x4 m4 = *(const bf16x4*)(m + row0);
#pragma unroll
      for (int v = 0; v < 4; v++) q.on[v] = (float)m4[v] > 0.0f;
    } else {
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (row0 + v >= a.mask0 && row0 + v < a.M) q.on[v] = (float)m[row0 + v] > 0.0f;
    }
  }
  return q;
}

// Those four rows (FWD: bias, ReLU; BDATA: add, mask) and their channels-last copy.
template <int MODE>
__device__ __forceinline__ void conv_out(const ConvK& a, const ConvIn& q, const floatx4& s, int row0, int n)
{
  if (row0 >= a.M) return;
  float ov[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int row = row0 + v;
    ov[v] = 0.0f;
    if (row >= a.M) continue;
    const size_t idx = (size_t)row * a.N + n;
    float o = s[v] + q.c[v];
    if (MODE != BDATA) {
      if (a.relu) o = fmaxf(o, 0.0f);
      if (a.C) a.C[idx] = a.res ? a.res[n] + o : o;   // null: no FP32 copy
    } else {
      if (!q.on[v]) o = 0.0f;
      a.C[idx] = o;
    }
    ov[v] = o;
  }
  // the four channels in one 8-byte store when they all exist
  if (!a.o1.p) return;
  __bf16* dst = a.o1.p + (size_t)n * a.o1.ld + a.o1.off + row0;
  if (row0 + 3 < a.M && ((a.o1.ld | a.o1.off) & 3) == 0) {
    bf16x4 w;
#pragma unroll
    for (int v = 0; v < 4; v++) w[v] = to_bf16(ov[v]);
    *(bf16x4*)dst = w;
  } else {
#pragma unroll
    for (int v = 0; v < 4; v++)
      if (row0 + v < a.M) dst[v] = to_bf16(ov[v]);
  }
}

// what a lane reads as its 8 channels outside the volume
__device__ __attribute__((aligned(16))) const unsigned k_zeros[4] = {0u, 0u, 0u, 0u};

// 8 channels of a voxel, or zeros; a global load (a pointer chosen between the two is a generic one,
// whose loads also count as LDS accesses)
__device__ __forceinline__ bf16x8 load_cl(const __bf16* p, bool in)
{
  return *(const __attribute__((address_space(1))) bf16x8*)(in ? (unsigned long long)p : (unsigned long long)k_zeros);
}

// the 8 channels from c on of input voxel (z, y, x)
template <int MODE>
__device__ __forceinline__ const __bf16* voxel_cl(const ConvK& a, int z, int y, int x, int c)
{
  if (MODE == FWDUP) {
    const bool up = c < a.Cu;
    const size_t v = up ? ((size_t)(z >> 1) * (a.H >> 1) + (y >> 1)) * (a.W >> 1) + (x >> 1) : ((size_t)z * a.H + y) * a.W + x;
    return (up ? a.Xu : a.Xl) + v * (up ? a.ldu : a.ldx) + (up ? c : c - a.Cu);
  }
  return a.Xl + (((size_t)z * a.H + y) * a.W + x) * a.ldx + c;
}

// A thread's place in a halo tile that begins one voxel before (z0, y0, x0): halo coordinates packed
// once, so that a load is a few integer operations (divisions by the halo's sides and 64-bit index
// products took longer than the products that they feed).
__device__ __forceinline__ unsigned halo_pack(int hx, int hy, int hz) { return (unsigned)(hx | hy << 8 | hz << 16); }

// Where a thread's 8 channels come from: Xl, or (up) the tensor of half the size. The tile's first voxel
// is even, so the half-size offset of a halo voxel does not depend on the tile. Offsets in units of 8
// channels fit 32 bits: two planes of a tensor that the device can hold have fewer than 2^34 elements.
struct HaloFrom {
  const __bf16* base;   // the tile's first voxel (not the halo's), the thread's channels
  int row, plane, ld8, up;
};
__device__ __forceinline__ HaloFrom halo_from(const __bf16* Xl, int ldx, const __bf16* Xu, int ldu, int Cu, int H, int W, int z, int y,
                                              int x, int c)
{
  HaloFrom f;
  f.up = c < Cu;
  f.row = f.up ? W >> 1 : W;
  f.plane = f.up ? (H >> 1) * (W >> 1) : H * W;
  f.ld8 = (f.up ? ldu : ldx) >> 3;
  const size_t v = f.up ? ((size_t)(z >> 1) * (H >> 1) + (y >> 1)) * (W >> 1) + (x >> 1) : ((size_t)z * H + y) * W + x;
  f.base = (f.up ? Xu : Xl) + v * (f.up ? ldu : ldx) + (f.up ? c : c - Cu);
  return f;
}
__device__ __forceinline__ bf16x8 halo_load(const HaloFrom& f, unsigned h, bool in)
{
  const int dx = ((int)(h & 255u) - 1) >> f.up, dy = ((int)(h >> 8 & 255u) - 1) >> f.up, dz = ((int)(h >> 16) - 1) >> f.up;
  return load_cl(f.base + (ptrdiff_t)((dz * f.plane + dy * f.row + dx) * f.ld8) * 8, in);
}

// bits t of the taps t = 9 (dz + 1) + 3 (dy + 1) + (dx + 1) whose three bits are all set
__device__ __forceinline__ unsigned tap_mask(unsigned vz, unsigned vy, unsigned vx)
{
  const unsigned row = (vy & 1 ? vx : 0u) | (vy & 2 ? vx << 3 : 0u) | (vy & 4 ? vx << 6 : 0u);
  return (vz & 1 ? row : 0u) | (vz & 2 ? row << 9 : 0u) | (vz & 4 ? row << 18 : 0u);
}

// Forward and input-gradient products on NC tiles of 16 voxels and MT blocks of 16 channels per
// workgroup; the four waves split the k-steps (wave w: steps w, w + 4, ...) and their sums are
// added in wave order through LDS. A lane's taps inside the volume are one bit mask and its input
// voxel is linear in the tap, so a k-step is the tap's offset, MT + NC 16-byte loads (weights 1 KB
// contiguous) and MT NC MFMAs; the loads of CONV_PF steps are in flight (one workgroup or two per CU
// at the coarse levels, where a k-step without prefetch took 1.2 to 1.5 us). Width 16 on 16 x 28 x 28
// voxels, all products of a forward: 95 -> 61 us; 192 -> 64 channels on 16 x 28 x 28: 61 -> 40 us.
// Stride-2 input gradients: output voxels are taken parity class by parity class (D, H, W even),
// so a tile's voxels share their 1 to 8 taps and the other k-steps are skipped (64 -> 32 channels on
// 32 x 56 x 56: 60 -> 29 us).
#define CONV_PF 4
template <int MODE, int MT, int NC, bool kSkip>
__global__ __launch_bounds__(256) void k_conv_cols(ConvK a)
{
  __shared__ floatx4 red[4][NC * MT][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int rb0 = blockIdx.y * MT;
  to_sample(a, blockIdx.z);
  int nn[NC], base[NC], cx[NC], cy[NC], cz[NC];   // c?: FWDUP's input voxel
  unsigned mask[NC];
  // the tap's step in the B tensor: rows and planes of that tensor
  const int bW = MODE != BDATA ? a.W : a.oW, bH = MODE != BDATA ? a.H : a.oH;
#pragma unroll
  for (int j = 0; j < NC; j++) {
    int n = (blockIdx.x * NC + j) * 16 + r;   // this lane's column in tile j
    const int w = MODE != BDATA ? a.oW : a.W, h = MODE != BDATA ? a.oH : a.H, d = MODE != BDATA ? a.oD : a.D;
    int x, y, z;
    if (kSkip) {
      const int per = a.N >> 3, cls = n / per, i = n - cls * per, w2 = w >> 1, h2 = h >> 1;
      x = 2 * (i % w2) + (cls & 1);
      y = 2 * ((i / w2) % h2) + ((cls >> 1) & 1);
      z = 2 * (i / (w2 * h2)) + (cls >> 2);
      const bool ok = n < a.N;
      n = ok ? (z * h + y) * w + x : a.N;
    } else {
      x = n % w;
      y = (n / w) % h;
      z = n / (w * h);
    }
    nn[j] = n;
    unsigned vx = 7, vy = 7, vz = 7;
    if (MODE != BDATA) {
      x *= a.stride;
      y *= a.stride;
      z *= a.stride;
      if (x == 0) vx &= ~1u;
      if (y == 0) vy &= ~1u;
      if (z == 0) vz &= ~1u;
      if (x + 1 >= a.W) vx &= ~4u;
      if (y + 1 >= a.H) vy &= ~4u;
      if (z + 1 >= a.D) vz &= ~4u;
      base[j] = (z * a.H + y) * a.W + x;
    } else if (kSkip) {   // 2 q + d = p: p even d = 0, p odd d = -1 (q = (p + 1) / 2) and +1 (q one less)
      vx = x & 1 ? 5u : 2u;
      vy = y & 1 ? 5u : 2u;
      vz = z & 1 ? 5u : 2u;
      x = (x + 1) >> 1;
      y = (y + 1) >> 1;
      z = (z + 1) >> 1;
      if (x >= a.oW) vx &= ~3u;
      if (y >= a.oH) vy &= ~3u;
      if (z >= a.oD) vz &= ~3u;
      base[j] = (z * a.oH + y) * a.oW + x;
    } else {                      // q = p - d
      if (x == 0) vx &= ~4u;
      if (y == 0) vy &= ~4u;
      if (z == 0) vz &= ~4u;
      if (x + 1 >= w) vx &= ~1u;
      if (y + 1 >= h) vy &= ~1u;
      if (z + 1 >= d) vz &= ~1u;
      base[j] = (z * h + y) * w + x;
    }
    cx[j] = x;
    cy[j] = y;
    cz[j] = z;
    mask[j] = n < a.N ? (a.ks == 3 ? tap_mask(vz, vy, vx) : 1u) : 0u;
  }
  floatx4 acc[NC][MT];
#pragma unroll
  for (int j = 0; j < NC; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  // the lane's tap t and channel c0 of k = t Cbp + c0 are carried from step to step
  const int Cbp = a.Cbp, dt = 128 / Cbp, dc = 128 - dt * Cbp;
  const int n_steps = (a.K + 31) >> 5, n_mine = (n_steps - wave + 3) >> 2;
  int t, c0, step = wave;
  {
    const int k = wave * 32 + kg * 8;
    t = k / Cbp;
    c0 = k - t * Cbp;
  }
  const __bf16* ap = a.A + ((size_t)wave * a.nrb + rb0) * 512 + lane * 8;
  const size_t astep = (size_t)a.nrb * 2048;
  bf16x8 av[CONV_PF][MT], bv[CONV_PF][NC];
  auto advance = [&]() {
    step += 4;
    ap += astep;
    c0 += dc;
    t += dt;
    if (c0 >= Cbp) {
      c0 -= Cbp;
      t++;
    }
  };
  auto fetch = [&](bf16x8* fa, bf16x8* fb) {   // step `step`, then on to the wave's next one
    int off = 0, oz = 0, oy = 0, ox = 0;
    if (a.ks == 3) {   // t / 9 = (7282 t) >> 16 and t / 3 = (21846 t) >> 16, exact for t < 32
      const int q9 = (t * 7282) >> 16, q3 = (t * 21846) >> 16;
      const int uz = q9, uy = q3 - 3 * q9, ux = t - 3 * q3;   // d + 1
      if (kSkip) off = -(((uz >> 1) * bH + (uy >> 1)) * bW + (ux >> 1));
      else {
        oz = uz - 1;
        oy = uy - 1;
        ox = ux - 1;
        off = (oz * bH + oy) * bW + ox;
        if (MODE == BDATA) off = -off;
      }
    }
#pragma unroll
    for (int i = 0; i < MT; i++) fa[i] = *(const bf16x8*)(ap + i * 512);
#pragma unroll
    for (int j = 0; j < NC; j++) {
      const bool in = t < 32 && ((mask[j] >> t) & 1u);
      const __bf16* p = MODE == FWDUP ? voxel_cl<MODE>(a, cz[j] + oz, cy[j] + oy, cx[j] + ox, c0)
                                      : a.Xl + ((size_t)(unsigned)(base[j] + off) * (unsigned)a.ldx + (unsigned)c0);
      fb[j] = load_cl(p, in);
    }
    advance();
  };
  auto mult = [&](const bf16x8* fa, const bf16x8* fb) {
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
      for (int i = 0; i < MT; i++) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[j][i], 0, 0, 0);
  };
  if constexpr (kSkip) {
    unsigned any = 0;
#pragma unroll
    for (int j = 0; j < NC; j++) any |= mask[j];
    auto live = [&]() {   // on to the next step with a tap of one of the tiles
      while (step < n_steps && !__any(t < 32 && ((any >> t) & 1u))) advance();
      return step < n_steps;
    };
    while (live()) {
      fetch(av[0], bv[0]);
      const bool two = live();
      if (two) fetch(av[1], bv[1]);
      mult(av[0], bv[0]);
      if (two) mult(av[1], bv[1]);
    }
  } else if (n_mine > 0) {
    int left = n_mine;
#pragma unroll
    for (int p = 0; p < CONV_PF; p++) {
      if (left > 0) fetch(av[p], bv[p]);
      left--;
    }
    int i = 0;
    for (; i + 2 * CONV_PF <= n_mine; i += CONV_PF) {
#pragma unroll
      for (int p = 0; p < CONV_PF; p++) {
        mult(av[p], bv[p]);
        fetch(av[p], bv[p]);
        __builtin_amdgcn_sched_barrier(0);   // the loads are issued here, CONV_PF steps ahead of their use
      }
    }
#pragma unroll
    for (int p = 0; p < CONV_PF; p++) {
      if (i + p < n_mine) mult(av[p], bv[p]);
      if (i + p + CONV_PF < n_mine) fetch(av[p], bv[p]);
    }
    i += CONV_PF;
#pragma unroll
    for (int p = 0; p < CONV_PF; p++)
      if (i + p < n_mine) mult(av[p], bv[p]);
  }
#pragma unroll
  for (int j = 0; j < NC; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) red[wave][j * MT + i][lane] = acc[j][i];
  // wave w finishes the (tile, row block) pairs w, w + 4, ...
  ConvIn pre[(NC * MT + 3) / 4];
#pragma unroll
  for (int q = 0; q < NC * MT; q++)
    if ((q & 3) == wave) pre[q / 4] = conv_in<MODE>(a, (rb0 + q % MT) * 16 + kg * 4, nn[q / MT]);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NC * MT; q++) {
    if ((q & 3) != wave) continue;
    const floatx4 s = red[0][q][lane] + red[1][q][lane] + red[2][q][lane] + red[3][q][lane];
    const int j = q / MT;
    if (nn[j] < a.N) conv_out<MODE>(a, pre[q / 4], s, (rb0 + q % MT) * 16 + kg * 4, nn[j]);
  }
}

// Forward and input-gradient products of a stride-1 3x3x3 convolution whose B tensor (the input, or
// the output gradient) has a multiple of 32 (padded) channels, in tiles of 16 x 8 x 2 voxels per
// workgroup: wave w has the 16 x 4 voxels from row 4 (w % 2) of plane w / 2, one row per MFMA column
// tile. The B tile with its one-voxel halo (18 x 10 x 4 voxels) is staged in LDS 32 channels at a time,
// zero outside the volume, as [channel group of 8][voxel] (a fragment read is 16 consecutive voxels:
// no bank conflict); the six rows x three shifts that a tap plane's nine taps read are read once, and
// each weight fragment serves the wave's four rows. FWD reads voxel p + d_t for tap t, BDATA
// (q = p - d_t) voxel p - d_t. Waiting for loads bounds it: the compiler sinks them to their use, so
// they are pinned FT_PF taps ahead, and a thread's halo loads are all issued before the first store.
// 96 -> 32 channels on four volumes of 32 x 56 x 56 (66.6 GFLOP): 169 us with 128-voxel tiles and
// loads at their use, 136 with the larger tile and batched halo loads, 93 with pinned loads.
#define FT_X 16
#define FT_Y 8
#define FT_Z 2
#define FT_HX (FT_X + 2)
#define FT_HY (FT_Y + 2)
#define FT_HALO ((FT_Z + 2) * FT_HY * FT_HX)
#define FT_HP (FT_HALO + 2)   // voxels per channel group, padded: the four groups of a voxel on different banks

// Workgroups are dealt to the eight XCDs in turn: number b of n, such that each XCD (and its L2) gets
// consecutive tiles, which share their halos.
__device__ __forceinline__ int xcd_order(int b, int n)
{
  const int per = n >> 3;
  return b < per * 8 ? (b & 7) * per + (b >> 3) : b;
}

#define FT_PF 3
template <int MODE, int MT>
__global__ __launch_bounds__(256) void k_conv_tiled(ConvK a)
{
  __shared__ bf16x8 s_halo[4 * FT_HP];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int tiles_x = (a.W + FT_X - 1) / FT_X, tiles_y = (a.H + FT_Y - 1) / FT_Y;
  int b = xcd_order(blockIdx.x, gridDim.x);
  const int x0 = (b % tiles_x) * FT_X;
  b /= tiles_x;
  const int y0 = (b % tiles_y) * FT_Y;
  const int z0 = (b / tiles_y) * FT_Z;
  const int rb0 = blockIdx.y * MT;
  to_sample(a, blockIdx.z);
  floatx4 acc[4][MT];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  const __bf16* ap = a.A + (size_t)rb0 * 512 + lane * 8;
  const size_t atap = (size_t)(a.Cbp >> 5) * a.nrb * 512;   // weights of the next tap
  constexpr int kLoads = (FT_HALO * 4 + 255) / 256;
  unsigned at[kLoads], ok = 0;
#pragma unroll
  for (int l = 0; l < kLoads; l++) {
    const int v = (threadIdx.x + 256 * l) >> 2, hx = v % FT_HX, hy = (v / FT_HX) % FT_HY, hz = v / (FT_HX * FT_HY);
    const int gz = z0 + hz - 1, gy = y0 + hy - 1, gx = x0 + hx - 1;
    at[l] = halo_pack(hx, hy, hz);
    if (v < FT_HALO && (unsigned)gz < (unsigned)a.D && (unsigned)gy < (unsigned)a.H && (unsigned)gx < (unsigned)a.W) ok |= 1u << l;
  }
  const bf16x8* const hp = s_halo + kg * FT_HP + ((wave >> 1) * FT_HY + 4 * (wave & 1)) * FT_HX + r;
  for (int c0 = 0; c0 < a.Cbp; c0 += 32, ap += (size_t)a.nrb * 512) {
    bf16x8 av[FT_PF + 1][MT];   // the weights of FT_PF taps in flight
#pragma unroll
    for (int t = 0; t < FT_PF; t++)
#pragma unroll
      for (int i = 0; i < MT; i++) av[t][i] = *(const bf16x8*)(ap + t * atap + i * 512);
    // all of the thread's loads in flight at once, then the stores
    const HaloFrom from = halo_from(a.Xl, a.ldx, a.Xu, a.ldu, MODE == FWDUP ? a.Cu : 0, a.H, a.W, z0, y0, x0, c0 + (threadIdx.x & 3) * 8);
    bf16x8 hv[kLoads];
#pragma unroll
    for (int l = 0; l < kLoads; l++) hv[l] = halo_load(from, at[l], ok >> l & 1u);
#pragma unroll
    for (int l = 0; l < kLoads; l++) {
      const int i = threadIdx.x + 256 * l;
      if (i < FT_HALO * 4) s_halo[(i & 3) * FT_HP + (i >> 2)] = hv[l];
    }
    __syncthreads();
    bf16x8 bv[6][3];
#pragma unroll
    for (int t = 0; t < 27; t++) {
      const int dz = MODE != BDATA ? t / 9 : 2 - t / 9;            // halo coordinates of p + d_t or p - d_t
      const int dy = MODE != BDATA ? (t / 3) % 3 : 2 - (t / 3) % 3;
      const int dx = MODE != BDATA ? t % 3 : 2 - t % 3;
      if (t % 9 == 0) {
#pragma unroll
        for (int y = 0; y < 6; y++)
#pragma unroll
          for (int x = 0; x < 3; x++) bv[y][x] = hp[(dz * FT_HY + y) * FT_HX + x];
      }
      if (t + FT_PF < 27) {
#pragma unroll
        for (int i = 0; i < MT; i++)
          av[(t + FT_PF) % (FT_PF + 1)][i] = *(const bf16x8*)(ap + (t + FT_PF) * atap + i * 512);
      }
      __builtin_amdgcn_sched_barrier(0);   // the loads stay ahead of the taps that they do not belong to
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < MT; i++)
          acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[t % (FT_PF + 1)][i], bv[j + dy][dx], acc[j][i], 0, 0, 0);
    }
    __syncthreads();
  }
  // this lane's columns are voxels (z, y0 + 4 (w % 2) + j, x0 + r)
  const int x = x0 + r, z = z0 + (wave >> 1);
  if (x >= a.W || z >= a.D) return;
  constexpr int kIn = MODE == BDATA ? 4 : 1;   // FWD: the rows' bias serves every column
  ConvIn pre[kIn][MT];
  const int yw = y0 + 4 * (wave & 1);
#pragma unroll
  for (int j = 0; j < kIn; j++)
#pragma unroll
    for (int i = 0; i < MT; i++)
      pre[j][i] = conv_in<MODE>(a, (rb0 + i) * 16 + kg * 4, yw + j < a.H ? (z * a.H + yw + j) * a.W + x : a.N);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (yw + j >= a.H) continue;
    const int n = (z * a.H + yw + j) * a.W + x;
#pragma unroll
    for (int i = 0; i < MT; i++) conv_out<MODE>(a, pre[j % kIn][i], acc[j][i], (rb0 + i) * 16 + kg * 4, n);
  }
}

// The products of k_conv_cols (the same k-steps per wave, the same order of every sum) for stride-1
// 3x3x3 convolutions with a multiple of 32 (padded) channels, in tiles of 16 x 4 voxels: k runs tap
// plane by tap plane, so LDS holds one halo plane (18 x 6 voxels) of all channels at a time, as
// [channel group of 8][voxel], and a weight fragment serves 64 voxels (k_conv_cols: 32, and its
// workgroups read each weight once per 16 or 32 voxels from L2, which bounds it). 192 -> 64 channels on
// four volumes of 16 x 28 x 28: 102 -> 60 us; 64 -> 64: 45 -> 33 us.
#define FP_HALO (6 * 18)
#define FP_HP (FP_HALO + 2)

template <int MODE, int MT>
__global__ __launch_bounds__(256) void k_conv_planes(ConvK a)
{
  extern __shared__ __attribute__((aligned(16))) char s_planes[];
  bf16x8* const halo = (bf16x8*)s_planes;                 // [Cbp / 8][FP_HP]
  floatx4* const red = (floatx4*)s_planes;                // [4 waves][2 rows x MT][64]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int tiles_x = (a.W + 15) >> 4, tiles_y = (a.H + 3) >> 2;
  int b = xcd_order(blockIdx.x, gridDim.x);
  const int x0 = (b % tiles_x) * 16;
  b /= tiles_x;
  const int y0 = (b % tiles_y) * 4;
  const int z = b / tiles_y;
  const int rb0 = blockIdx.y * MT;
  to_sample(a, blockIdx.z);
  floatx4 acc[4][MT];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int nsl = a.Cbp >> 5, groups = a.Cbp >> 3, per_plane = 9 * nsl;
  const int dt = 4 / nsl, dc = 4 - dt * nsl;
  const size_t astep = (size_t)a.nrb * 2048;
  const bf16x8* const hp = halo + kg * FP_HP + r;
  constexpr int kLoads = 6;   // halo loads of a thread in flight
  const int v_first = threadIdx.x / groups, q_first = threadIdx.x - v_first * groups, dv = 256 / groups, dq = 256 - dv * groups;
  for (int p = 0; p < 3; p++) {
    // the wave's steps w, w + 4, ... inside this tap plane
    const int first = wave + 4 * ((p * per_plane - wave + 3) >> 2);
    const int n_mine = ((p + 1) * per_plane - first + 3) >> 2;
    int t = (first - p * per_plane) / nsl, sl = first - p * per_plane - t * nsl;
    const __bf16* ap = a.A + ((size_t)first * a.nrb + rb0) * 512 + lane * 8;
    bf16x8 av[CONV_PF][MT];
    auto fetch = [&](bf16x8* fa) {
#pragma unroll
      for (int i = 0; i < MT; i++) fa[i] = *(const bf16x8*)(ap + i * 512);
      ap += astep;
    };
    auto mult = [&](const bf16x8* fa) {
      const int q3 = (t * 21846) >> 16, dy = MODE != BDATA ? q3 : 2 - q3, dx = MODE != BDATA ? t - 3 * q3 : 2 - (t - 3 * q3);
      const bf16x8* h = hp + sl * (4 * FP_HP) + dy * 18 + dx;
      bf16x8 bv[4];
#pragma unroll
      for (int j = 0; j < 4; j++) bv[j] = h[j * 18];
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], bv[j], acc[j][i], 0, 0, 0);
      sl += dc;
      t += dt;
      if (sl >= nsl) {
        sl -= nsl;
        t++;
      }
    };
#pragma unroll
    for (int f = 0; f < CONV_PF; f++)
      if (f < n_mine) fetch(av[f]);
    if (p) __syncthreads();   // every wave is done with the last plane
    const int gz = MODE != BDATA ? z + p - 1 : z + 1 - p;
    for (int v = v_first, q = q_first; v < FP_HALO;) {
      bf16x8 hv[kLoads];
      int at[kLoads];
#pragma unroll
      for (int l = 0; l < kLoads; l++) {
        const int hy = (v * 3641) >> 16, hx = v - 18 * hy;   // v / 18, exact for v < 2^11
        const int gy = y0 + hy - 1, gx = x0 + hx - 1;
        const bool in = v < FP_HALO && (unsigned)gz < (unsigned)a.D && (unsigned)gy < (unsigned)a.H && (unsigned)gx < (unsigned)a.W;
        hv[l] = load_cl(voxel_cl<MODE>(a, gz, gy, gx, q * 8), in);
        at[l] = v < FP_HALO ? q * FP_HP + v : -1;
        v += dv;
        q += dq;
        if (q >= groups) {
          q -= groups;
          v++;
        }
      }
#pragma unroll
      for (int l = 0; l < kLoads; l++)
        if (at[l] >= 0) halo[at[l]] = hv[l];
    }
    __syncthreads();
    int i = 0;
    for (; i + 2 * CONV_PF <= n_mine; i += CONV_PF) {
#pragma unroll
      for (int f = 0; f < CONV_PF; f++) {
        mult(av[f]);
        fetch(av[f]);
        __builtin_amdgcn_sched_barrier(0);   // the loads are issued here, CONV_PF steps ahead of their use
      }
    }
#pragma unroll
    for (int f = 0; f < CONV_PF; f++) {
      if (i + f < n_mine) mult(av[f]);
      if (i + f + CONV_PF < n_mine) fetch(av[f]);
    }
    i += CONV_PF;
#pragma unroll
    for (int f = 0; f < CONV_PF; f++)
      if (i + f < n_mine) mult(av[f]);
  }
  // the waves' sums, two rows at a time
  const int x = x0 + r;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int i = 0; i < MT; i++) red[(wave * 2 * MT + j * MT + i) * 64 + lane] = acc[2 * h + j][i];
    ConvIn pre[(2 * MT + 3) / 4];
#pragma unroll
    for (int q = 0; q < 2 * MT; q++) {
      const int y = y0 + 2 * h + q / MT;
      if ((q & 3) == wave)
        pre[q / 4] = conv_in<MODE>(a, (rb0 + q % MT) * 16 + kg * 4, x < a.W && y < a.H ? (z * a.H + y) * a.W + x : a.N);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2 * MT; q++) {
      if ((q & 3) != wave) continue;
      const floatx4* s = red + q * 64 + lane;
      const floatx4 sum = s[0] + s[2 * MT * 64] + s[4 * MT * 64] + s[6 * MT * 64];
      const int y = y0 + 2 * h + q / MT;
      if (x < a.W && y < a.H) conv_out<MODE>(a, pre[q / 4], sum, (rb0 + q % MT) * 16 + kg * 4, (z * a.H + y) * a.W + x);
    }
  }
}

// The products of k_conv_cols with at most SHORT_STEPS k-steps (8 or fewer padded channels, or a
// 1x1x1 kernel): reading and writing bounds them, so the weights stay in registers and each wave takes
// 16-voxel tiles by itself, all steps of one (the four sums that k_conv_cols' waves would hold, added
// in their order), the next tile's voxels in flight. Four volumes of 32 x 56 x 56: 4 -> 32 channels
// 49 -> 32 us, 32 -> 1 22 -> 8 us, the latter's input gradient 50 -> 22 us.
#define SHORT_STEPS 8
template <int MODE, int MT, int NS>
__global__ __launch_bounds__(256) void k_conv_short(ConvK a)
{
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int rb0 = blockIdx.y * MT;
  to_sample(a, blockIdx.z);
  bf16x8 av[NS][MT], bv[NS];
  int t[NS], c0[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
#pragma unroll
    for (int i = 0; i < MT; i++)   // steps that K does not have multiply zeros
      av[s][i] = load_cl(a.A + ((size_t)s * a.nrb + rb0 + i) * 512 + lane * 8, 32 * s < a.K);
    const int k = 32 * s + 8 * kg;
    t[s] = k / a.Cbp;
    c0[s] = k - t[s] * a.Cbp;
  }
  const int tiles = (a.N + 15) >> 4, step = gridDim.x * 4;
  auto fetch = [&](int tile) {
    const int n = tile * 16 + r;
    const int x = n % a.W, y = (n / a.W) % a.H, z = n / (a.W * a.H);
    unsigned vx = 7, vy = 7, vz = 7;
    constexpr unsigned lo = MODE == BDATA ? 4u : 1u, hi = 5u - lo;   // the taps that leave at 0 and at the end
    if (x == 0) vx &= ~lo;
    if (y == 0) vy &= ~lo;
    if (z == 0) vz &= ~lo;
    if (x + 1 >= a.W) vx &= ~hi;
    if (y + 1 >= a.H) vy &= ~hi;
    if (z + 1 >= a.D) vz &= ~hi;
    const unsigned mask = n < a.N ? (a.ks == 3 ? tap_mask(vz, vy, vx) : 1u) : 0u;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      int off = 0;
      if (a.ks == 3) {
        const int q9 = (t[s] * 7282) >> 16, q3 = (t[s] * 21846) >> 16;
        off = ((q9 - 1) * a.H + (q3 - 3 * q9 - 1)) * a.W + (t[s] - 3 * q3 - 1);
        if (MODE == BDATA) off = -off;
      }
      const bool in = t[s] < 32 && ((mask >> t[s]) & 1u);
      const size_t v = (unsigned)(n + off);
      bv[s] = load_cl(a.Xl + v * a.ldx + c0[s], in);
    }
  };
  int tile = blockIdx.x * 4 + wave;
  ConvIn pre[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) pre[i] = conv_in<MODE>(a, (rb0 + i) * 16 + kg * 4, tile * 16 + r);
  if (tile < tiles) fetch(tile);
  while (tile < tiles) {
    floatx4 acc[MT][4];   // steps 0, 4, ...; 1, 5, ...; 2, 6, ...; 3, 7, ...
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
      for (int i = 0; i < MT; i++) acc[i][s & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[s][i], bv[s], acc[i][s & 3], 0, 0, 0);
    const int n = tile * 16 + r;
    tile += step;
    if (tile < tiles) fetch(tile);
    ConvIn now[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
      now[i] = pre[i];
      if (MODE == BDATA && tile < tiles) pre[i] = conv_in<MODE>(a, (rb0 + i) * 16 + kg * 4, tile * 16 + r);
    }
    if (n < a.N) {
#pragma unroll
      for (int i = 0; i < MT; i++)
        conv_out<MODE>(a, now[i], acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3], (rb0 + i) * 16 + kg * 4, n);
    }
  }
}

inline int mt_for(int M)
{
  const int mt = (M + 15) / 16;
  if (mt <= 4) return mt;
  for (int c = 4; c >= 2; c--)
    if (mt % c == 0) return c;
  return 4;
}
inline int rows_for(int M)
{
  const int t = 16 * mt_for(M);
  return (M + t - 1) / t * t;
}
inline int rup(int x, int m) { return (x + m - 1) / m * m; }

template <int MODE, int NC, bool kSkip>
void launch_cols(const ConvK& a, int mt, hipStream_t st)
{
  const dim3 g((a.N + 16 * NC - 1) / (16 * NC), a.nrb / mt, a.samples);
  switch (mt) {
    case 1: hipLaunchKernelGGL((k_conv_cols<MODE, 1, NC, kSkip>), g, dim3(256), 0, st, a); break;
    case 2: hipLaunchKernelGGL((k_conv_cols<MODE, 2, NC, kSkip>), g, dim3(256), 0, st, a); break;
    case 3: hipLaunchKernelGGL((k_conv_cols<MODE, 3, NC, kSkip>), g, dim3(256), 0, st, a); break;
    default: hipLaunchKernelGGL((k_conv_cols<MODE, 4, NC, kSkip>), g, dim3(256), 0, st, a); break;
  }
}

// Forward and input-gradient products outside the tiled form. The tile of a workgroup does not
// change the order of any sum: it is the largest of the list that still gives COLS_WGS workgroups
// (two per CU), the smallest where none does.
#define COLS_WGS 512
// k_conv_planes takes a shape when its halo plane fits LDS beside a second workgroup's and its tiles
// give PLANES_WGS workgroups: with fewer, k_conv_cols' smaller tiles end as soon. Forward at width 32, device
// us a sample, with a threshold of 1 / 100 / 200 / 256 / 512 / never: one sample of 32 x 56 x 56 (its half
// resolution has 224) 145 / 144 / 144 / 158 / 157 / 157, four 83 / 82 / 83 / 82 / 84 / 95; 24 x 40 x 40
// one 117 / 109 / 102 / 102 / 101 / 114, four 51 / 51 / 51 / 51 / 56 / 65; 16 x 28 x 28 one 103 / 77 / 77 /
// 77 / 77 / 77, eight 20 / 20 / 20 / 20 / 21 / 25; 12 x 20 x 36 four 29 / 27 / 25 / 25 / 25 / 28; 16 x 56 x 56
// two 81 / 81 / 81 / 87 / 85 / 103; 64^3 one 210 / 212 / 209 / 209 / 209 / 244; width 16, one of
// 32 x 56 x 56: 117 / 110 / 109 / 107 / 107 / 107.
#define PLANES_WGS 200
inline long long planes_tiles(const ConvK& a) { return (long long)((a.W + 15) / 16) * ((a.H + 3) / 4) * a.D; }
inline size_t planes_lds(const ConvK& a, int mt) { return std::max<size_t>(16 * (size_t)(a.Cbp / 8) * FP_HP, 16 * 512 * (size_t)mt); }
inline bool use_planes(const ConvK& a)
{
  const int mt = mt_for(a.M);
  return a.ks == 3 && a.stride == 1 && a.Cbp % 32 == 0 && planes_lds(a, mt) <= 65536 && planes_tiles(a) <= 0x7fffffffLL &&
         planes_tiles(a) * (a.nrb / mt) * a.samples >= PLANES_WGS;
}
template <int MODE>
hipError_t launch_planes(const ConvK& a, hipStream_t st)
{
  const int mt = mt_for(a.M);
  const dim3 g((unsigned)planes_tiles(a), a.nrb / mt, a.samples);
  const unsigned lds = (unsigned)planes_lds(a, mt);
  switch (mt) {
    case 1: hipLaunchKernelGGL((k_conv_planes<MODE, 1>), g, dim3(256), lds, st, a); break;
    case 2: hipLaunchKernelGGL((k_conv_planes<MODE, 2>), g, dim3(256), lds, st, a); break;
    case 3: hipLaunchKernelGGL((k_conv_planes<MODE, 3>), g, dim3(256), lds, st, a); break;
    default: hipLaunchKernelGGL((k_conv_planes<MODE, 4>), g, dim3(256), lds, st, a); break;
  }
  return hipGetLastError();
}

inline bool use_short(const ConvK& a) { return a.stride == 1 && a.K <= 32 * SHORT_STEPS; }
template <int MODE, int MT>
void launch_short_ns(const ConvK& a, dim3 g, hipStream_t st)
{
  const int ns = (a.K + 31) / 32;
  if (ns == 1) hipLaunchKernelGGL((k_conv_short<MODE, MT, 1>), g, dim3(256), 0, st, a);
  else if (ns == 2) hipLaunchKernelGGL((k_conv_short<MODE, MT, 2>), g, dim3(256), 0, st, a);
  else if (ns <= 4) hipLaunchKernelGGL((k_conv_short<MODE, MT, 4>), g, dim3(256), 0, st, a);
  else if constexpr (MT <= 2) hipLaunchKernelGGL((k_conv_short<MODE, MT, 8>), g, dim3(256), 0, st, a);
}
template <int MODE>
hipError_t launch_short(const ConvK& a, hipStream_t st)
{
  int mt = mt_for(a.M);
  if (a.K > 128) mt = mt == 4 ? 2 : mt == 3 ? 1 : mt;   // eight steps' weights of more blocks take over 256 registers
  const int tiles = (a.N + 15) / 16;
  // the workgroups that are resident together, so that a wave's weights serve several tiles
  const int most = std::max(1, (a.K > 128 ? 512 : 2048) / (a.samples * (a.nrb / mt)));
  const dim3 g(std::min((tiles + 3) / 4, most), a.nrb / mt, a.samples);
  switch (mt) {
    case 1: launch_short_ns<MODE, 1>(a, g, st); break;
    case 2: launch_short_ns<MODE, 2>(a, g, st); break;
    case 3: launch_short_ns<MODE, 3>(a, g, st); break;
    default: launch_short_ns<MODE, 4>(a, g, st); break;
  }
  return hipGetLastError();
}

template <int MODE>
hipError_t launch_conv(const ConvK& a, hipStream_t st)
{
  if (MODE != FWDUP && use_short(a)) return launch_short<MODE == FWDUP ? FWD : MODE>(a, st);
  if (use_planes(a)) return launch_planes<MODE>(a, st);
  int mt = mt_for(a.M), nc = 2;
  auto wgs = [&](int m, int c) { return (long long)a.samples * (a.nrb / m) * ((a.N + 16 * c - 1) / (16 * c)); };
  if (wgs(mt, nc) < COLS_WGS) {
    nc = 1;
    while (mt > 1 && wgs(mt, nc) < COLS_WGS) mt = mt % 2 == 0 ? mt / 2 : 1;
  }
  if (MODE == BDATA && a.stride == 2) {
    if (a.ks != 3 || a.D % 2 || a.H % 2 || a.W % 2) return hipErrorInvalidValue;
    if (nc == 2) launch_cols<BDATA, 2, true>(a, mt, st);
    else launch_cols<BDATA, 1, true>(a, mt, st);
  } else {
    if (nc == 2) launch_cols<MODE, 2, false>(a, mt, st);
    else launch_cols<MODE, 1, false>(a, mt, st);
  }
  return hipGetLastError();
}

// Stride-1 3x3x3 FWD / BDATA products with Cbp % 32 == 0 (k_conv_tiled); the row blocks as
// k_conv_cols', so the A rows read stay inside the padded weight copy. Counted in 4-row tiles.
inline long long tiled_blocks(const ConvK& a)
{
  return (long long)((a.W + FT_X - 1) / FT_X) * ((a.H + 3) / 4) * a.D * ((a.M + 16 * mt_for(a.M) - 1) / (16 * mt_for(a.M)));
}
// The tiled products on volumes with at least 1024 four-row tiles (the full-resolution level);
// smaller volumes (the coarser U-Net levels) take the 16-voxel tiles and in-workgroup k split of
// k_conv_planes and k_conv_cols.
#define TILED_MIN 1024
inline bool use_tiled(const ConvK& a)
{
  return a.ks == 3 && a.stride == 1 && a.Cbp % 32 == 0 && tiled_blocks(a) >= TILED_MIN;
}

template <int MODE>
hipError_t launch_conv_tiled(const ConvK& a, hipStream_t st)
{
  const int mt = mt_for(a.M);
  const long long tiles = (long long)((a.W + FT_X - 1) / FT_X) * ((a.H + FT_Y - 1) / FT_Y) * ((a.D + FT_Z - 1) / FT_Z);
  if (a.ks != 3 || a.stride != 1 || a.D != a.oD || a.H != a.oH || a.W != a.oW || a.Cbp % 32 != 0 || a.Kp < 27 * a.Cbp ||
      tiles > 0x7fffffffLL)
    return hipErrorInvalidValue;
  dim3 grid((unsigned)tiles, (a.M + 16 * mt - 1) / (16 * mt), a.samples);
  switch (mt) {
    case 1: hipLaunchKernelGGL((k_conv_tiled<MODE, 1>), grid, dim3(256), 0, st, a); break;
    case 2: hipLaunchKernelGGL((k_conv_tiled<MODE, 2>), grid, dim3(256), 0, st, a); break;
    case 3: hipLaunchKernelGGL((k_conv_tiled<MODE, 3>), grid, dim3(256), 0, st, a); break;
    default: hipLaunchKernelGGL((k_conv_tiled<MODE, 4>), grid, dim3(256), 0, st, a); break;
  }
  return hipGetLastError();
}

// Weight gradient of a 3x3x3 convolution of stride S (1 or 2) from channels-last BF16 copies of
// its input X and of its output gradient dY:
//   G[co][ci][t] = sum_q dY[co][q] X[ci][S q + d_t]      (MFMA m = co, n = ci, k = q)
// A workgroup owns one block of 32 output and 32 input channels and a slab of output-voxel tiles
// (16 x 8 x 2 voxels for S = 1, 16 x 4 x 1 for S = 2); each half of a tile's voxels has six waves, which
// split the accumulators by tap plane dz (3) and input-channel half (2), each holding the 3 x 3 (dy, dx)
// taps x 2 output-channel halves = 18 MFMA tiles. dY of the tile and X of the region its taps read (18 x 10 x 4 voxels, 33 x 9 x 3 for
// S = 2) are staged in LDS as they are, [voxel][32 channels], and the fragments, which want 8 voxels of
// a channel per lane, are transposing reads (16 lanes give the addresses of 4 voxels x 4 channel quads
// and get 4 voxels of one channel each), so a tap is an address offset. The next tile is on its way to
// registers while one is multiplied. Each half writes its slab's sums to part[2 slab + half][t][co][ci];
// k_bwgt_reduce adds the slabs in a fixed order into the gradient (deterministic, no atomics).
// 96 -> 32 channels on four volumes of 32 x 56 x 56: 234 us with element-wise transposed
// stores, 140 with these reads and six waves per CU, 101 with twelve, 89 with the loads' places packed once
#define BW_X 16
#define BW_THREADS 768
template <int S>
struct BwTile {
  static constexpr int Y = S == 1 ? 8 : 4, Z = S == 1 ? 2 : 1;
  static constexpr int HX = S * (BW_X - 1) + 3, HY = S * (Y - 1) + 3, HZ = S * (Z - 1) + 3;
  static constexpr int NX = (HX * HY * HZ * 4 + BW_THREADS - 1) / BW_THREADS, NG = (BW_X * Y * Z * 4 + BW_THREADS - 1) / BW_THREADS;
};

struct BwK {
  const __bf16* Xl;   // input, channels-last [vox][ldx] (channels >= ldx: zero)
  const __bf16* Xu;   // its first Cu channels at half size, [vox / 8][ldu] (Cu = 0: none; Xl then holds the others)
  int ldu, Cu;
  const __bf16* Gl;   // output gradient, channels-last [ovox][ldg]
  float* part;        // [n_slabs][27][32 cob][32 cib]
  int ldx, ldg, gch, Cin, Cout, D, H, W, oD, oH, oW;   // gch: channels from Gl on
  int tiles_x, tiles_y, tiles_z, n_tiles, per_slab, cob, cib;   // n_tiles: of all samples
  size_t sX, sXu, sG;                                  // from one sample to the next
};

typedef short short4v __attribute__((ext_vector_type(4)));

// the lane's 8 voxels of its channel: two transposing reads, the second `next` bytes on
__device__ __forceinline__ bf16x8 read_tr(const char* lds, int next)
{
  typedef __attribute__((address_space(3))) short4v lds4;
  const short4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)lds);
  const short4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)(lds + next));
  typedef short short8v __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(bf16x8, (short8v)__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int S>
__global__ __launch_bounds__(BW_THREADS, 3) void k_bwgt_tiled(BwK a)
{
  typedef BwTile<S> T;
  __shared__ __attribute__((aligned(16))) char s_x[T::HX * T::HY * T::HZ * 64];   // [voxel][32 channels]
  __shared__ __attribute__((aligned(16))) char s_g[BW_X * T::Y * T::Z * 64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, g = lane >> 4;
  const int dz = wave % 3, nj = wave / 3 & 1, half = wave / 6;   // tap plane, input-channel half, half of the k-steps
  const int slab = blockIdx.x, co0 = blockIdx.y * 32, ci0 = blockIdx.z * 32;
  floatx4 acc[3][3][2];
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int m = 0; m < 2; m++) acc[i][j][m] = floatx4{0.f, 0.f, 0.f, 0.f};
  // the thread's channels and places are the same in every tile (BW_THREADS is a multiple of 4)
  const int cx = ci0 + (threadIdx.x & 3) * 8, cg = co0 + (threadIdx.x & 3) * 8;
  const bool x_in = cx < a.Cu + a.ldx;
  unsigned at[T::NX];
#pragma unroll
  for (int l = 0; l < T::NX; l++) {
    const int v = (threadIdx.x + l * BW_THREADS) >> 2, hz = v / (T::HX * T::HY);
    // 0xffff: past the region (the last one only)
    at[l] = halo_pack(v % T::HX, (v / T::HX) % T::HY, hz < T::HZ ? hz : 0xffff);
  }
  bf16x8 xv[T::NX], gv[T::NG];
  auto load = [&](int tile) {
    int b = tile;
    const int x0 = (b % a.tiles_x) * BW_X;
    b /= a.tiles_x;
    const int y0 = (b % a.tiles_y) * T::Y;
    b /= a.tiles_y;
    const int z0 = (b % a.tiles_z) * T::Z, smp = b / a.tiles_z;
    const __bf16* const Xl = a.Xl + smp * a.sX;
    const __bf16* const Xu = a.Xu + smp * a.sXu;
    const __bf16* const Gl = a.Gl + smp * a.sG;
    // input region: voxel (S z0 - 1 + hz, S y0 - 1 + hy, S x0 - 1 + hx), 4 groups of 8 channels
    const int xz = S * z0, xy = S * y0, xx = S * x0;
    const HaloFrom from = halo_from(Xl, a.ldx, Xu, a.ldu, a.Cu, a.H, a.W, xz, xy, xx, cx);
#pragma unroll
    for (int l = 0; l < T::NX; l++) {
      const int gz = xz + (int)(at[l] >> 16) - 1, gy = xy + (int)(at[l] >> 8 & 255u) - 1, gx = xx + (int)(at[l] & 255u) - 1;
      const bool in = x_in && (l + 1 < T::NX || at[l] >> 16 != 0xffff) && (unsigned)gz < (unsigned)a.D &&
                      (unsigned)gy < (unsigned)a.H && (unsigned)gx < (unsigned)a.W;
      xv[l] = halo_load(from, at[l], in);
    }
    const __bf16* const gb = Gl + (((size_t)z0 * a.oH + y0) * a.oW + x0) * a.ldg + cg;
#pragma unroll
    for (int l = 0; l < T::NG; l++) {
      const int v = (threadIdx.x + l * BW_THREADS) >> 2, dx = v % BW_X, dy = (v / BW_X) % T::Y, dz = v / (BW_X * T::Y);
      const bool in = dz < T::Z && z0 + dz < a.oD && y0 + dy < a.oH && x0 + dx < a.oW && cg < a.gch;
      gv[l] = load_cl(gb + (ptrdiff_t)((dz * a.oH + dy) * a.oW + dx) * a.ldg, in);
    }
  };
  // what this lane reads of each fragment: voxel (lr / 4) of four, channels 4 (lr % 4) .. + 3 of 16
  const int vj = lr >> 2, qb = (lr & 3) * 8;
  const int hz = S == 1 ? half : 0, hy = S == 1 ? 0 : 2 * half;   // where the half begins: a plane, or two rows
  const char* const ga = s_g + ((hz * T::Y + hy + (g >> 1)) * BW_X + (g & 1) * 8 + vj) * 64 + qb;
  const char* const xa = s_x + (((S * hz + dz) * T::HY + S * (hy + (g >> 1))) * T::HX + S * ((g & 1) * 8 + vj)) * 64 + 32 * nj + qb;
  const int t_end = min(a.n_tiles, (slab + 1) * a.per_slab);
  int tile = slab * a.per_slab;
  if (tile < t_end) load(tile);
  for (; tile < t_end; tile++) {
#pragma unroll
    for (int l = 0; l < T::NX; l++) {
      const int i = threadIdx.x + l * BW_THREADS;
      if (i < T::HX * T::HY * T::HZ * 4) *(bf16x8*)(s_x + i * 16) = xv[l];
    }
#pragma unroll
    for (int l = 0; l < T::NG; l++) {
      const int i = threadIdx.x + l * BW_THREADS;
      if (i < BW_X * T::Y * T::Z * 4) *(bf16x8*)(s_g + i * 16) = gv[l];
    }
    __syncthreads();
    if (tile + 1 < t_end) load(tile + 1);
    __builtin_amdgcn_sched_barrier(0);   // the loads are issued before the products
#pragma unroll
    for (int ks = 0; ks < T::Y * T::Z / 4; ks++) {   // 32 voxels: two rows of the wave's half of the tile
      constexpr int rows = T::Y / (S == 1 ? 2 : 4);   // pairs of rows in a plane of the half
      const int oz = ks / rows, oy = 2 * (ks % rows);
      bf16x8 av[2];
#pragma unroll
      for (int m = 0; m < 2; m++) av[m] = read_tr(ga + (oz * T::Y + oy) * (BW_X * 64) + 32 * m, 256);
#pragma unroll
      for (int dy = 0; dy < 3; dy++)
#pragma unroll
        for (int dx = 0; dx < 3; dx++) {
          const bf16x8 bx = read_tr(xa + ((S * oz * T::HY + S * oy + dy) * T::HX + dx) * 64, S * 256);
#pragma unroll
          for (int m = 0; m < 2; m++)
            acc[dy][dx][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bx, acc[dy][dx][m], 0, 0, 0);
        }
    }
    __syncthreads();
  }
  // this lane: columns ci = ci0 + 16 nj + lr, rows co = co0 + 16 m + 4 g + v of each tap's tile
  const int CoutR = 32 * a.cob, CinR = 32 * a.cib;
#pragma unroll
  for (int dy = 0; dy < 3; dy++)
#pragma unroll
    for (int dx = 0; dx < 3; dx++) {
      const int t = dz * 9 + dy * 3 + dx;
      float* p = a.part + ((size_t)(2 * slab + half) * 27 + t) * CoutR * CinR + (ci0 + 16 * nj + lr);
#pragma unroll
      for (int m = 0; m < 2; m++)
#pragma unroll
        for (int v = 0; v < 4; v++) p[(size_t)(co0 + 16 * m + 4 * g + v) * CinR] = acc[dy][dx][m][v];
    }
}

// G[co][ci][t] += sum over slabs of part[slab][t][co][ci]. A workgroup takes 64 consecutive
// outputs in the partial sums' (t, co, ci) order (each slab's reads contiguous across them) and
// four slab phases: thread (j, ph) adds slabs ph, ph + 4, ... of output j, and the four phase
// sums are added in a fixed order (deterministic).
__global__ __launch_bounds__(256) void k_bwgt_reduce(const float* __restrict__ part, float* __restrict__ G, int Cout, int Cin,
                                                     int CoutR, int CinR, int n_slabs)
{
  __shared__ float ps[4][64];
  const long long n = (long long)Cout * Cin * 27;
  const int j = threadIdx.x & 63, ph = threadIdx.x >> 6;
  const long long i = (long long)blockIdx.x * 64 + j;
  float s = 0.0f;
  int ci = 0, co = 0, t = 0;
  if (i < n) {
    ci = (int)(i % Cin);
    co = (int)((i / Cin) % Cout);
    t = (int)(i / ((long long)Cin * Cout));
    const size_t stride = (size_t)27 * CoutR * CinR;
    const float* p = part + ((size_t)t * CoutR + co) * CinR + ci;
#pragma unroll 8
    for (int k = ph; k < n_slabs; k += 4) s += p[(size_t)k * stride];
  }
  ps[ph][j] = s;
  __syncthreads();
  if (ph == 0 && i < n) G[((size_t)co * Cin + ci) * 27 + t] += ((ps[0][j] + ps[1][j]) + ps[2][j]) + ps[3][j];
}

// Workgroups of the tiled weight gradient: about BW_WGS in total (one per CU), the output-voxel tiles
// dealt to slabs of equal length; each workgroup's two halves write their own partial sums.
#define BW_WGS 256
inline void bwgt_shape(int samples, int stride, BwK& b, int& n_slabs)
{
  const int ty = stride == 1 ? BwTile<1>::Y : BwTile<2>::Y, tz = stride == 1 ? BwTile<1>::Z : BwTile<2>::Z;
  b.tiles_x = (b.oW + BW_X - 1) / BW_X;
  b.tiles_y = (b.oH + ty - 1) / ty;
  b.tiles_z = (b.oD + tz - 1) / tz;
  b.n_tiles = b.tiles_x * b.tiles_y * b.tiles_z * samples;
  b.cob = (b.Cout + 31) / 32;
  b.cib = (b.Cin + 31) / 32;
  n_slabs = std::max(1, std::min(b.n_tiles, BW_WGS / (b.cob * b.cib)));
  b.per_slab = (b.n_tiles + n_slabs - 1) / n_slabs;
  n_slabs = (b.n_tiles + b.per_slab - 1) / b.per_slab;
}
constexpr size_t kBwPartFloats = (size_t)BW_WGS * 2 * 27 * 1024;   // half a workgroup writes 27 x 32 x 32

// The input x and its gradient's copy gyl as in conv_bwd_weights; stride 1 (input and output volumes
// equal) or 2 (output (D/2, H/2, W/2)). Output channels go in passes of as many 32-channel blocks as
// the partial sums have room for (all of them up to 256 blocks of 32 x 32: each workgroup writes two halves).
hipError_t launch_bwgt_tiled(int samples, int stride, BwK b, const __bf16* gyl, float* G, hipStream_t st)
{
  if (b.ldx % 8 != 0 || b.ldg % 8 != 0 || (stride != 1 && stride != 2)) return hipErrorInvalidValue;
  const int cout = b.Cout, cib = (b.Cin + 31) / 32, most = BW_WGS / cib * 32;
  if (most == 0) return hipErrorInvalidValue;
  for (int co = 0; co < cout; co += most) {
    b.Cout = std::min(most, cout - co);
    b.Gl = gyl + co;
    b.gch = b.ldg - co;
    int n_slabs = 0;
    bwgt_shape(samples, stride, b, n_slabs);
    const dim3 g(n_slabs, b.cob, b.cib);
    if (stride == 1) hipLaunchKernelGGL(k_bwgt_tiled<1>, g, dim3(BW_THREADS), 0, st, b);
    else hipLaunchKernelGGL(k_bwgt_tiled<2>, g, dim3(BW_THREADS), 0, st, b);
    const long long n = (long long)b.Cout * b.Cin * 27;
    hipLaunchKernelGGL(k_bwgt_reduce, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, st, (const float*)b.part,
                       G + (size_t)co * b.Cin * 27, b.Cout, b.Cin, 32 * b.cob, 32 * b.cib, 2 * n_slabs);
  }
  return hipGetLastError();
}

// BF16 weight copies in the order in which the MFMA fragments read them: k-step s = k / 32, then
// the 16-row block, then the lane (row m % 16, k-group (k % 32) / 8) and its 8 k, so that a fragment
// is one contiguous 1 KB load (row by row it was 16 segments of 64 bytes). Element (m, k = t Cp + c)
// is W[co][ci][t] with (co, ci) = (m, c) (forward) or (c, m) (transposed, for the input gradient);
// zero outside the real channels.
__global__ void k_derive(const float* __restrict__ w, __bf16* __restrict__ out, int rows, int Kp, int Cout, int Cin, int T, int Cp,
                         int transpose)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)rows * Kp) return;
  const int step = (int)(i / ((size_t)rows * 32)), q = (int)(i % ((size_t)rows * 32)), l = (q & 511) >> 3;
  const int m = (q >> 9) * 16 + (l & 15), k = step * 32 + (l >> 4) * 8 + (q & 7);
  const int t = k / Cp, c = k - t * Cp;
  const int co = transpose ? c : m, ci = transpose ? m : c;
  const bool ok = t < T && co < Cout && ci < Cin;
  out[i] = to_bf16(ok ? w[((size_t)co * Cin + ci) * T + t] : 0.0f);
}

// ------------------------------------------------------------------ elementwise kernels

// Elementwise kernels take sample blockIdx.y; a tensor that is part of a larger one comes with its
// step from sample to sample.
// Channels-last concatenation of the nearest x2 upsampling of u [D/2][H/2][W/2][ldu] (Cu channels) and of
// l [D][H][W][ldl] (Cl channels) into o: where Cu is not a multiple of 8 (else the products read u and l
// themselves).
__global__ void k_concat(const __bf16* __restrict__ u, int Cu, int ldu, const __bf16* __restrict__ l, int Cl, int ldl, int D, int H,
                         int W, ClOut o)
{
  const size_t vox = (size_t)D * H * W, i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vox * (Cu + Cl)) return;
  const size_t v = i / (Cu + Cl), vl = blockIdx.y * vox + v;
  const int c = (int)(i % (Cu + Cl));
  const int x = (int)(v % W), y = (int)((v / W) % H), z = (int)(v / ((size_t)W * H));
  const size_t vu = blockIdx.y * (vox / 8) + ((size_t)(z / 2) * (H / 2) + y / 2) * (W / 2) + x / 2;
  o.p[vl * o.ld + c] = c < Cu ? u[vu * ldu + c] : l[vl * ldl + c - Cu];
}
// Input voxels v0 .. v0 + range - 1 (x: FP32 [sample][C][range], device or pinned host memory) into their
// channels-last BF16 copy o (zero padded) and, where x0 is given, the FP32 input [sample][C][vox]; 8
// channels of a voxel per thread.
__global__ void k_input(const float* __restrict__ x, int C, size_t vox, size_t v0, size_t range, float* __restrict__ x0, ClOut o)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= range * (o.ld / 8)) return;
  const size_t v = i % range;
  const int c0 = (int)(i / range) * 8;
  float f[8];
  bf16x8 q;
#pragma unroll
  for (int k = 0; k < 8; k++) f[k] = c0 + k < C ? x[(blockIdx.y * (size_t)C + c0 + k) * range + v] : 0.0f;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    q[k] = to_bf16(f[k]);
    if (x0 && c0 + k < C) x0[(blockIdx.y * (size_t)C + c0 + k) * vox + v0 + v] = f[k];
  }
  *(bf16x8*)(o.p + (blockIdx.y * vox + v0 + v) * o.ld + c0) = q;
}
// Gradient of the x2 upsampling: the eight voxels' sum, zero where the upsampled tensor's own copy
// (mask, [d h w][o.ld]) is not positive, and its channels-last copy. A thread takes 8 channels of a voxel.
__global__ void k_upsample_bwd(const float* __restrict__ gy, size_t sy, const __bf16* __restrict__ mask, float* __restrict__ gx,
                               int C, int d, int h, int w, ClOut o)
{
  const size_t vin = (size_t)d * h * w;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vin * (size_t)((C + 7) / 8)) return;
  gy += blockIdx.y * sy;
  gx += blockIdx.y * (C * vin);
  const size_t v = i % vin, vl = blockIdx.y * vin + v;
  const int c0 = (int)(i / vin) * 8;
  const int xx = (int)(v % w), yy = (int)((v / w) % h), zz = (int)(v / ((size_t)w * h));
  const int W2 = 2 * w, H2 = 2 * h, D2 = 2 * d;
  const bf16x8 m = *(const bf16x8*)(mask + vl * o.ld + c0);
  bf16x8 q;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    q[k] = to_bf16(0.0f);
    if (c0 + k >= C) continue;
    float s = 0.0f;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const float2 p = *(const float2*)(gy + (((size_t)(c0 + k) * D2 + 2 * zz + a) * H2 + 2 * yy + b) * W2 + 2 * xx);
        s += p.x;
        s += p.y;
      }
    if (!((float)m[k] > 0.0f)) s = 0.0f;
    gx[(c0 + k) * vin + v] = s;
    q[k] = to_bf16(s);
  }
  *(bf16x8*)(o.p + vl * o.ld + c0) = q;
}
// per-channel sum (bias gradient): workgroups (channel, chunk of `per` voxels, sample), added
// atomically; four voxels a read where the channels' beginnings allow it
__global__ __launch_bounds__(256) void k_channel_sum(const float* __restrict__ g, size_t sg, float* __restrict__ out, int vox, int per)
{
  __shared__ float sh[4];
  const float* p = g + blockIdx.z * sg + (size_t)blockIdx.x * vox;
  const int b = blockIdx.y * per, e = min(vox, b + per);
  float s = 0.0f;
  if ((vox & 3) == 0 && ((uintptr_t)p & 15) == 0) {   // per is a multiple of 4
    const float4* p4 = (const float4*)p;
    float4 t = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int i = b / 4 + threadIdx.x; i < e / 4; i += 256) {
      const float4 v = p4[i];
      t.x += v.x;
      t.y += v.y;
      t.z += v.z;
      t.w += v.w;
    }
    s = (t.x + t.y) + (t.z + t.w);
  } else {
    for (int i = b + threadIdx.x; i < e; i += 256) s += p[i];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(&out[blockIdx.x], (sh[0] + sh[1]) + (sh[2] + sh[3]));
}
// loss gradient (and its channels-last copy) and squared error of the output
__global__ void k_loss(const float* __restrict__ out, const float* __restrict__ target, float* __restrict__ g, float scale,
                       float* __restrict__ sse, int n, ClOut gl)
{
  __shared__ float sh[256];
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t i = blockIdx.y * (size_t)n + v;
  float e2 = 0.0f;
  if (v < n) {
    const float d = out[i] - target[i];
    g[i] = 2.0f * d * scale;
    gl.p[i * gl.ld] = to_bf16(g[i]);
    e2 = d * d;
  }
  sh[threadIdx.x] = e2;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(sse, sh[0]);
}
// Weight gradient of the 1x1x1 output layer (one output channel): the sum over voxels of the output
// gradient (channel 0 of gl, [vox][8]) times the input copy xl [vox][ld]. A thread adds 8 channels of
// every (256 / groups)th voxel of its workgroup's chunk; bounded by reading xl once.
__global__ __launch_bounds__(256) void k_bwgt_point(const __bf16* __restrict__ xl, int ld, const __bf16* __restrict__ gl,
                                                    float* __restrict__ G, int C, size_t n, int chunk)
{
  __shared__ float sh[256][9];
  const int groups = ld >> 3, per = 256 / groups, q = threadIdx.x % groups, first = threadIdx.x / groups;
  const size_t b = (size_t)blockIdx.x * chunk, e = min(n, b + chunk);
  float s[8];
#pragma unroll
  for (int k = 0; k < 8; k++) s[k] = 0.0f;
  if (first < per)
#pragma unroll 4
    for (size_t v = b + first; v < e; v += per) {
      const bf16x8 x = *(const bf16x8*)(xl + v * ld + q * 8);
      const float g = (float)gl[v * 8];
#pragma unroll
      for (int k = 0; k < 8; k++) s[k] = __builtin_fmaf(g, (float)x[k], s[k]);   // the product is exact
    }
#pragma unroll
  for (int k = 0; k < 8; k++) sh[threadIdx.x][k] = s[k];
  __syncthreads();
  for (int c = threadIdx.x; c < C; c += 256) {
    float t = 0.0f;
    for (int i = 0; i < per; i++) t += sh[i * groups + (c >> 3)][c & 7];
    atomicAdd(&G[c], t);
  }
}
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v, size_t n,
                       float lr, float b1, float b2, float eps, float c1, float c2)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
__global__ void k_zero(float* __restrict__ p, size_t n)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0f;
}

// Total of a float array in double, in a fixed order: 256 workgroups sum contiguous chunks,
// then one workgroup sums their results. Integer-valued inputs (counts) give the exact total.
__global__ void k_sum_partial(const float* __restrict__ x, size_t n, double* __restrict__ partial)
{
  __shared__ double sh[256];
  const size_t chunk = (n + gridDim.x - 1) / gridDim.x, b = blockIdx.x * chunk, e = min(n, b + chunk);
  double s = 0.0;
  for (size_t i = b + threadIdx.x; i < e; i += blockDim.x) s += (double)x[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}
__global__ void k_sum_final(const double* __restrict__ partial, int m, double* __restrict__ out)
{
  __shared__ double sh[256];
  sh[threadIdx.x] = (int)threadIdx.x < m ? partial[threadIdx.x] : 0.0;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0];
}
// network input: scatter and trues counts times float(voxels / total trues)
__global__ void k_normalize(const float* __restrict__ s, const float* __restrict__ t, float* __restrict__ x0, size_t n,
                            const double* __restrict__ total)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double tot = total[0];
  const float scale = tot > 0.0 ? (float)((double)n / tot) : 0.0f;
  x0[i] = s[i] * scale;
  x0[n + i] = t[i] * scale;
}
// scatter per decay: max(output, 0) times float(total trues / (voxels * decays))
__global__ void k_estimate(const float* __restrict__ out, float* __restrict__ est, size_t n, const double* __restrict__ total,
                           const unsigned long long* __restrict__ decay_counter)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double tot = total[0], decays = (double)(long long)*decay_counter;
  const float f = (tot > 0.0 && decays > 0.0) ? (float)(tot / ((double)n * decays)) : 0.0f;
  est[i] = fmaxf(out[i], 0.0f) * f;
}

inline unsigned blocks_for(size_t n) { return (unsigned)((n + 255) / 256); }

// ------------------------------------------------------------------ the network

// One convolution layer: W [Cout][Cin][T] and b [Cout] at offsets of the flat parameter
// vector; BF16 copies at offsets of the BF16 buffer.
struct Conv {
  int cin, cout, ks, stride;
  size_t w, b;                 // offsets into the parameter vector
  size_t wf, wb;               // offsets of the forward / transposed BF16 copies
  int rows_f, kp_f, rows_b, kp_b;
};

struct Vol {
  int C, D, H, W;
  size_t vox() const { return (size_t)D * H * W; }
  size_t size() const { return (size_t)C * vox(); }
};

}  // namespace

// 3D U-Net: enc1 (2 convs, width c) -> stride-2 conv (2c) -> conv -> stride-2 conv (4c) -> conv
// -> upsample, concat with the enc2 skip -> conv (2c) -> upsample, concat with enc1 -> conv (c)
// -> 1x1x1 conv -> residual added to input channel 0. ReLU after every 3x3x3 convolution.
struct mcpet_surrogate {
  int D, H, W, cin, c;
  Conv L[9];
  size_t n_params = 0, n_bf16 = 0;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  __bf16* wbf = nullptr;
  // the input, the output and the gradients; the concatenations' gradients hold the skip tensors' ones
  Vol vx, va1, vcat1, vd1, vcat2, vd2, vb3, ve2, ve1, vr;
  float *x0 = nullptr, *out = nullptr;
  float *ga1 = nullptr, *gcat1 = nullptr, *gd1 = nullptr, *gcat2 = nullptr, *gd2 = nullptr, *gb3 = nullptr, *ge2 = nullptr,
        *ge1 = nullptr, *gr = nullptr, *sse = nullptr;
  // channels-last BF16 copies: the activations (post-ReLU), then the gradients read as B operands
  __bf16 *x0l = nullptr, *a1l = nullptr, *b1l = nullptr, *cat1l = nullptr, *d1l = nullptr, *b2l = nullptr, *cat2l = nullptr,
         *d2l = nullptr, *b3l = nullptr, *e2l = nullptr, *e1l = nullptr;
  __bf16 *grl = nullptr, *ge1l = nullptr, *ge2l = nullptr, *gb3l = nullptr, *gd2l = nullptr, *gb2l = nullptr, *gd1l = nullptr,
         *gb1l = nullptr, *ga1l = nullptr;
  float *raw_s = nullptr, *raw_t = nullptr, *est = nullptr;   // the fused estimate's buffers
  int slots = 0, grad_slots = 0;   // samples that the tensors above have room for: the forward's, the gradients'
  bool grad_full = false;          // more gradients did not fit
  void *held = nullptr, *grad_held = nullptr;
  double* sums = nullptr;                                       // 256 partial totals + the total
  float* bw_part = nullptr;                                     // slab sums of the tiled weight gradient
  long long t_adam = 0;
  int device = 0;
  hipStream_t st = nullptr;
  hipEvent_t ev_f0 = nullptr, ev_f1 = nullptr;   // around the last forward of mcpet_surrogate_forward
  float* h_stage = nullptr;   // pinned: a group's outputs or targets; the fused estimate's two outputs
  float* h_in = nullptr;      // pinned: the two halves of stage_input's buffer, stage_in floats
  size_t stage_in = 0;
  int in_turn = 0;                      // the half that stage_input fills next
  bool in_used[2] = {false, false};     // halves that kernels of the current call may still read (until ev_in)
  hipEvent_t ev_in[2] = {nullptr, nullptr}, ev_out = nullptr;
  unsigned long long* h_decays = nullptr;   // pinned: the estimated run's decays
  int fwd_timed = 0;   // samples between the two events
  std::vector<void*> allocs;
  std::string err;
  double flops_fwd = 0.0;
};

namespace {

mcpet_status serr(mcpet_surrogate* s, mcpet_status st, const std::string& m)
{
  if (s) s->err = m;
  mcpet_host_set_error(m.c_str());
  return st;
}

#define SHIP(s, call)                                                                                  \
  do {                                                                                                 \
    hipError_t e_ = (call);                                                                            \
    if (e_ != hipSuccess) return serr(s, MCPET_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

template <class T>
hipError_t dalloc_t(mcpet_surrogate* s, T** p, size_t n)
{
  hipError_t e = hipMalloc((void**)p, sizeof(T) * std::max<size_t>(1, n));
  if (e == hipSuccess) {
    s->allocs.push_back(*p);
    e = hipMemset(*p, 0, sizeof(T) * std::max<size_t>(1, n));
  }
  return e;
}

// refresh the BF16 weight copies from the FP32 parameters
hipError_t derive(mcpet_surrogate* s)
{
  for (int i = 0; i < 9; i++) {
    const Conv& l = s->L[i];
    const int T = l.ks * l.ks * l.ks;
    size_t n = (size_t)l.rows_f * l.kp_f;
    hipLaunchKernelGGL(k_derive, dim3(blocks_for(n)), dim3(256), 0, s->st, s->p + l.w, s->wbf + l.wf, l.rows_f, l.kp_f, l.cout,
                       l.cin, T, rup(l.cin, 8), 0);
    n = (size_t)l.rows_b * l.kp_b;
    hipLaunchKernelGGL(k_derive, dim3(blocks_for(n)), dim3(256), 0, s->st, s->p + l.w, s->wbf + l.wb, l.rows_b, l.kp_b, l.cout,
                       l.cin, T, rup(l.cout, 8), 1);
  }
  return hipGetLastError();
}

ConvK conv_args(const Conv& l, const Vol& vin, const Vol& vout)
{
  ConvK a{};
  a.D = vin.D;
  a.H = vin.H;
  a.W = vin.W;
  a.oD = vout.D;
  a.oH = vout.H;
  a.oW = vout.W;
  a.ks = l.ks;
  a.stride = l.stride;
  a.T = l.ks * l.ks * l.ks;
  return a;
}

const ClOut kNoCl{nullptr, 0, 0};

// A layer's input as channels-last copies: xl alone, or the concatenation of xu's x2 upsampling (its
// first Cu channels) and xl.
struct ClIn {
  const __bf16* xl;
  int ld;
  const __bf16* xu;
  int Cu;
};

// act(conv(x) + b) into the channels-last copy o1 and, where y is given, FP32 (with res: res + it)
hipError_t conv_fwd(mcpet_surrogate* s, int ns, const Conv& l, const Vol& vin, ClIn x, const Vol& vout, bool relu, ClOut o1,
                    float* y = nullptr, const float* res = nullptr)
{
  ConvK a = conv_args(l, vin, vout);
  a.A = s->wbf + l.wf;
  a.Xl = x.xl;
  a.ldx = x.ld;
  a.sX = vin.vox() * x.ld;
  a.Xu = x.xu;
  a.Cu = a.ldu = x.Cu;
  a.sXu = vin.vox() / 8 * x.Cu;
  a.C = y;
  a.sC = vout.size();
  a.res = res;
  a.sR = s->vx.size();
  a.o1 = o1;
  a.bias = s->p + l.b;
  a.relu = relu ? 1 : 0;
  a.M = l.cout;
  a.N = (int)vout.vox();
  a.Cb = l.cin;
  a.Cbp = rup(l.cin, 8);
  a.samples = ns;
  a.K = a.T * a.Cbp;
  a.Kp = l.kp_f;
  a.nrb = l.rows_f / 16;
  s->flops_fwd += 2.0 * l.cout * (double)l.cin * a.T * a.N;
  if (x.Cu) return use_tiled(a) ? launch_conv_tiled<FWDUP>(a, s->st) : launch_conv<FWDUP>(a, s->st);
  return use_tiled(a) ? launch_conv_tiled<FWD>(a, s->st) : launch_conv<FWD>(a, s->st);
}
// gx (+)= dL/dx of the layer input; from channel mask0 on zeroed where the input's copy mask is not
// positive; gy read from its channels-last copy
hipError_t conv_bwd_data(mcpet_surrogate* s, int ns, const Conv& l, const Vol& vin, const Vol& vout, const __bf16* gyl, float* gx,
                         size_t sx, ClOut mask, int mask0, bool add, ClOut o1)
{
  ConvK a = conv_args(l, vin, vout);
  a.A = s->wbf + l.wb;
  a.Xl = gyl;
  a.C = gx;
  a.o1 = o1;
  a.mask = mask.p;
  a.ldm = mask.ld;
  a.mask0 = mask0;
  a.beta = add ? 1 : 0;
  a.M = l.cin;
  a.N = (int)vin.vox();
  a.Cb = l.cout;
  a.Cbp = rup(l.cout, 8);
  a.ldx = a.Cbp;
  a.samples = ns;
  a.sX = vout.vox() * a.Cbp;
  a.sC = sx;
  a.K = a.T * a.Cbp;
  a.Kp = l.kp_b;
  a.nrb = l.rows_b / 16;
  return use_tiled(a) ? launch_conv_tiled<BDATA>(a, s->st) : launch_conv<BDATA>(a, s->st);
}
// weight and bias gradients accumulated from gy (dL/d pre-activation, with its channels-last copy
// gyl) and the layer input x
hipError_t conv_bwd_weights(mcpet_surrogate* s, int ns, const Conv& l, const Vol& vin, ClIn x, const Vol& vout, const float* gy,
                            size_t sg, const __bf16* gyl)
{
  const int vox = (int)vout.vox(), per = 4096;
  hipError_t e = hipSuccess;
  if (l.ks == 1) {   // the output layer: one channel from at most 256
    const size_t n = (size_t)ns * vox;
    const int chunk = (int)std::max<size_t>(256, (n + 1023) / 1024);
    hipLaunchKernelGGL(k_bwgt_point, dim3((unsigned)((n + chunk - 1) / chunk)), dim3(256), 0, s->st, x.xl, x.ld, gyl, s->g + l.w,
                       l.cin, n, chunk);
    e = hipGetLastError();
  } else {
    BwK b{};
    b.Xl = x.xl;
    b.Xu = x.xu;
    b.ldu = b.Cu = x.Cu;
    b.part = s->bw_part;
    b.ldx = x.ld;
    b.ldg = rup(l.cout, 8);
    b.Cin = l.cin;
    b.Cout = l.cout;
    b.D = vin.D, b.H = vin.H, b.W = vin.W;
    b.oD = vout.D, b.oH = vout.H, b.oW = vout.W;
    b.sX = vin.vox() * x.ld;
    b.sXu = vin.vox() / 8 * x.Cu;
    b.sG = vout.vox() * b.ldg;
    e = launch_bwgt_tiled(ns, l.stride, b, gyl, s->g + l.w, s->st);
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_channel_sum, dim3(l.cout, (vox + per - 1) / per, ns), dim3(256), 0, s->st, gy, sg, s->g + l.b, vox, per);
  return hipGetLastError();
}
hipError_t upsample_bwd(mcpet_surrogate* s, int ns, const Vol& v, const float* gy, size_t sy, const __bf16* mask, float* gx, ClOut o)
{
  hipLaunchKernelGGL(k_upsample_bwd, dim3(blocks_for(v.vox() * ((v.C + 7) / 8)), ns), dim3(256), 0, s->st, gy, sy, mask, gx, v.C,
                     v.D, v.H, v.W, o);
  return hipGetLastError();
}
ClOut cl(__bf16* p, int channels, int off = 0) { return ClOut{p, rup(channels, 8), off}; }

ClIn in(const __bf16* p, int channels) { return ClIn{p, rup(channels, 8), nullptr, 0}; }

// The input of a layer after an upsampling: its two tensors where they are, or their concatenation cat
// (written by concat) where the products cannot read them so.
ClIn in_up(const __bf16* u, int Cu, const __bf16* l, int Cl, const __bf16* cat)
{
  return Cu % 8 == 0 ? ClIn{l, rup(Cl, 8), u, Cu} : in(cat, Cu + Cl);
}
hipError_t concat(mcpet_surrogate* s, int ns, const Vol& v, const __bf16* u, int Cu, const __bf16* l, int Cl, __bf16* cat)
{
  if (Cu % 8 == 0) return hipSuccess;
  hipLaunchKernelGGL(k_concat, dim3(blocks_for(v.vox() * (Cu + Cl)), ns), dim3(256), 0, s->st, u, Cu, rup(Cu, 8), l, Cl, rup(Cl, 8),
                     v.D, v.H, v.W, cl(cat, Cu + Cl));
  return hipGetLastError();
}

// n samples of the batch into s->x0 and their copy. A pageable copy of 100 KB takes 48 us, of 6.4 MB
// 200; so the host fills the two halves of a pinned buffer in turn (whole samples where they fit, else
// voxel ranges) and k_input reads them where they are. A half that was filled before in this call, for
// this group of samples or an earlier one, is filled again only after its k_input has ended.
hipError_t stage_input(mcpet_surrogate* s, const float* x, int n)
{
  const size_t C = s->cin, vox = s->vx.vox(), half = s->stage_in / 2;
  const size_t range = std::min(vox, half / C);
  const int per = range == vox ? (int)std::min<size_t>(n, half / (C * vox)) : 1;
  for (int b = 0; b < n; b += per)
    for (size_t v0 = 0; v0 < vox; v0 += range, s->in_turn ^= 1) {
      const int m = std::min(per, n - b), turn = s->in_turn;
      const size_t r = std::min(range, vox - v0);
      float* h = s->h_in + turn * half;
      hipError_t e = s->in_used[turn] ? hipEventSynchronize(s->ev_in[turn]) : hipSuccess;
      if (e != hipSuccess) return e;
      if (r == vox) std::memcpy(h, x + b * C * vox, sizeof(float) * m * C * vox);
      else
        for (size_t c = 0; c < C; c++) std::memcpy(h + c * r, x + (b * C + c) * vox + v0, sizeof(float) * r);
      const ClOut o{s->x0l + (size_t)b * vox * rup(s->cin, 8), rup(s->cin, 8), 0};
      hipLaunchKernelGGL(k_input, dim3(blocks_for(r * (o.ld / 8)), m), dim3(256), 0, s->st, (const float*)h, (int)C, vox, v0, r,
                         s->x0 + (size_t)b * C * vox, o);
      e = hipGetLastError();
      if (e == hipSuccess) e = hipEventRecord(s->ev_in[turn], s->st);
      if (e != hipSuccess) return e;
      s->in_used[turn] = true;
    }
  return hipSuccess;
}

// Forward of the ns samples already in s->x0 and their copy, into out (device, or pinned host memory).
// The layers pass their outputs on as channels-last BF16 copies, which are also the weight gradients'
// operands and, by their signs, the ReLU masks.
hipError_t forward(mcpet_surrogate* s, int ns, float* out)
{
  hipError_t e = hipSuccess;
  const int c = s->c;
  const Vol vb1{c, s->D, s->H, s->W}, vb2{2 * c, s->D / 2, s->H / 2, s->W / 2};
  s->flops_fwd = 0.0;
#define STEP(x) \
  if (e == hipSuccess) e = (x)
  STEP(conv_fwd(s, ns, s->L[0], s->vx, in(s->x0l, s->cin), s->va1, true, cl(s->a1l, c)));
  STEP(conv_fwd(s, ns, s->L[1], s->va1, in(s->a1l, c), vb1, true, cl(s->b1l, c)));
  STEP(conv_fwd(s, ns, s->L[2], vb1, in(s->b1l, c), s->vd1, true, cl(s->d1l, 2 * c)));
  STEP(conv_fwd(s, ns, s->L[3], s->vd1, in(s->d1l, 2 * c), vb2, true, cl(s->b2l, 2 * c)));
  STEP(conv_fwd(s, ns, s->L[4], vb2, in(s->b2l, 2 * c), s->vd2, true, cl(s->d2l, 4 * c)));
  STEP(conv_fwd(s, ns, s->L[5], s->vd2, in(s->d2l, 4 * c), s->vb3, true, cl(s->b3l, 4 * c)));
  STEP(concat(s, ns, s->vcat2, s->b3l, 4 * c, s->b2l, 2 * c, s->cat2l));
  STEP(conv_fwd(s, ns, s->L[6], s->vcat2, in_up(s->b3l, 4 * c, s->b2l, 2 * c, s->cat2l), s->ve2, true, cl(s->e2l, 2 * c)));
  STEP(concat(s, ns, s->vcat1, s->e2l, 2 * c, s->b1l, c, s->cat1l));
  STEP(conv_fwd(s, ns, s->L[7], s->vcat1, in_up(s->e2l, 2 * c, s->b1l, c, s->cat1l), s->ve1, true, cl(s->e1l, c)));
  STEP(conv_fwd(s, ns, s->L[8], s->ve1, in(s->e1l, c), s->vr, false, kNoCl, out, s->x0));
#undef STEP
  return e;
}

// Backward of ns samples from gr (= dL/dr, with its channels-last copy); accumulates the
// parameter gradients. The ReLU derivative is applied where each gradient is produced (mask = the
// sign of the post-ReLU activation), for an upsampled tensor after the sum over its copies. A
// gradient's channels-last copy is written by the product that completes it.
hipError_t backward(mcpet_surrogate* s, int ns)
{
  hipError_t e = hipSuccess;
  const int c = s->c;
  const Vol vb1{c, s->D, s->H, s->W}, vb2{2 * c, s->D / 2, s->H / 2, s->W / 2};
  const size_t s1 = s->vcat1.size(), s2 = s->vcat2.size();
  float* gb1 = s->gcat1 + (size_t)2 * c * vb1.vox();
  float* gb2 = s->gcat2 + (size_t)4 * c * vb2.vox();
#define STEP(x) \
  if (e == hipSuccess) e = (x)
#define WGT(l, vin, x, vout, gy, sg, gyl) STEP(conv_bwd_weights(s, ns, s->L[l], vin, x, vout, gy, sg, gyl))
#define DATA(l, vin, vout, gyl, gx, sx, mask, mask0, add, o1) \
  STEP(conv_bwd_data(s, ns, s->L[l], vin, vout, gyl, gx, sx, mask, mask0, add, o1))
  WGT(8, s->ve1, in(s->e1l, c), s->vr, s->gr, s->vr.size(), s->grl);
  DATA(8, s->ve1, s->vr, s->grl, s->ge1, s->ve1.size(), cl(s->e1l, c), 0, false, cl(s->ge1l, c));
  WGT(7, s->vcat1, in_up(s->e2l, 2 * c, s->b1l, c, s->cat1l), s->ve1, s->ge1, s->ve1.size(), s->ge1l);
  DATA(7, s->vcat1, s->ve1, s->ge1l, s->gcat1, s1, cl(s->b1l, c), 2 * c, false, kNoCl);   // g(up1), g(b1 skip)
  STEP(upsample_bwd(s, ns, s->ve2, s->gcat1, s1, s->e2l, s->ge2, cl(s->ge2l, 2 * c)));
  WGT(6, s->vcat2, in_up(s->b3l, 4 * c, s->b2l, 2 * c, s->cat2l), s->ve2, s->ge2, s->ve2.size(), s->ge2l);
  DATA(6, s->vcat2, s->ve2, s->ge2l, s->gcat2, s2, cl(s->b2l, 2 * c), 4 * c, false, kNoCl);   // g(up2), g(b2 skip)
  STEP(upsample_bwd(s, ns, s->vb3, s->gcat2, s2, s->b3l, s->gb3, cl(s->gb3l, 4 * c)));
  WGT(5, s->vd2, in(s->d2l, 4 * c), s->vb3, s->gb3, s->vb3.size(), s->gb3l);
  DATA(5, s->vd2, s->vb3, s->gb3l, s->gd2, s->vd2.size(), cl(s->d2l, 4 * c), 0, false, cl(s->gd2l, 4 * c));
  WGT(4, vb2, in(s->b2l, 2 * c), s->vd2, s->gd2, s->vd2.size(), s->gd2l);
  DATA(4, vb2, s->vd2, s->gd2l, gb2, s2, cl(s->b2l, 2 * c), 0, true, cl(s->gb2l, 2 * c));      // + the skip's gradient
  WGT(3, s->vd1, in(s->d1l, 2 * c), vb2, gb2, s2, s->gb2l);
  DATA(3, s->vd1, vb2, s->gb2l, s->gd1, s->vd1.size(), cl(s->d1l, 2 * c), 0, false, cl(s->gd1l, 2 * c));
  WGT(2, vb1, in(s->b1l, c), s->vd1, s->gd1, s->vd1.size(), s->gd1l);
  DATA(2, vb1, s->vd1, s->gd1l, gb1, s1, cl(s->b1l, c), 0, true, cl(s->gb1l, c));              // + the skip's gradient
  WGT(1, s->va1, in(s->a1l, c), vb1, gb1, s1, s->gb1l);
  DATA(1, s->va1, vb1, s->gb1l, s->ga1, s->va1.size(), cl(s->a1l, c), 0, false, cl(s->ga1l, c));
  WGT(0, s->vx, in(s->x0l, s->cin), s->va1, s->ga1, s->va1.size(), s->ga1l);
#undef WGT
#undef DATA
#undef STEP
  return e;
}

// The tensors held per sample: the forward's (the weight gradients' operands and the ReLU masks too), and
// what only the gradients need.
struct Slot {
  void** p;
  size_t bytes;   // of one sample
  bool zero;
};

std::vector<Slot> sample_tensors(mcpet_surrogate* s, bool gradients)
{
  const int c = s->c, ci = s->cin;
  const size_t v0 = s->vx.vox(), v1 = s->vd1.vox(), v2 = s->vd2.vox();
  std::vector<Slot> t;
  auto f = [&](float** p, const Vol& v) { t.push_back({(void**)p, sizeof(float) * v.size(), false}); };
  auto h = [&](__bf16** p, size_t vox, int ch) { t.push_back({(void**)p, sizeof(__bf16) * vox * rup(ch, 8), true}); };
  if (!gradients) {
    const bool cat = 2 * c % 8 != 0;   // the concatenations are written (concat)
    f(&s->x0, s->vx), f(&s->out, s->vr);
    h(&s->x0l, v0, ci), h(&s->a1l, v0, c), h(&s->b1l, v0, c), h(&s->cat1l, cat ? v0 : 0, 3 * c);
    h(&s->d1l, v1, 2 * c), h(&s->b2l, v1, 2 * c), h(&s->cat2l, cat ? v1 : 0, 6 * c), h(&s->d2l, v2, 4 * c);
    h(&s->e1l, v0, c), h(&s->e2l, v1, 2 * c), h(&s->b3l, v2, 4 * c);
  } else {
    f(&s->ga1, s->va1), f(&s->gcat1, s->vcat1), f(&s->gd1, s->vd1), f(&s->gcat2, s->vcat2);
    f(&s->gd2, s->vd2), f(&s->gb3, s->vb3), f(&s->ge2, s->ve2), f(&s->ge1, s->ve1), f(&s->gr, s->vr);
    h(&s->grl, v0, 8), h(&s->ge1l, v0, c), h(&s->ge2l, v1, 2 * c), h(&s->gb3l, v2, 4 * c);
    h(&s->gd2l, v2, 4 * c), h(&s->gb2l, v1, 2 * c), h(&s->gd1l, v1, 2 * c), h(&s->gb1l, v0, c), h(&s->ga1l, v0, c);
  }
  return t;
}

// Room for n samples of the tensors t in one allocation, the BF16 copies first: zeroed, their padding
// channels stay zero. The tensors' pointers change only where it succeeds.
hipError_t hold(mcpet_surrogate* s, const std::vector<Slot>& t, int n, void** block)
{
  auto room = [n](const Slot& b) { return (b.bytes * n + 255) / 256 * 256; };
  size_t zeroed = 0, plain = 0;
  for (const Slot& b : t) (b.zero ? zeroed : plain) += room(b);
  char* q = nullptr;
  const hipError_t e = hipMalloc((void**)&q, zeroed + plain);
  if (e != hipSuccess) return e;
  *block = q;
  char *z = q, *p = q + zeroed;
  for (const Slot& b : t) {
    char*& at = b.zero ? z : p;
    *b.p = at;
    at += room(b);
  }
  return hipMemsetAsync(q, 0, zeroed, s->st);
}

// Samples that go through the network together: one launch per layer serves them all, so the
// coarse levels and the short launches fill the device. About 2^19 voxels are enough, and at most
// 1 GiB is held for them, the gradients' part of it (four fifths; one sample's until then) from the first
// gradients of more than one sample. Four samples of 32 x 56 x 56 on width 32: 1.09 ms of device time one by
// one, 0.56 together; eight of 16 x 28 x 28 on width 16: 0.77 and 0.11.
hipError_t hold_samples(mcpet_surrogate* s)
{
  const std::vector<Slot> t = sample_tensors(s, false), g = sample_tensors(s, true);
  size_t per = 0;
  for (const auto* v : {&t, &g})
    for (const Slot& b : *v) per += b.bytes;
  const size_t by_vox = (((size_t)1 << 19) + s->vr.vox() - 1) / s->vr.vox(), by_mem = ((size_t)1 << 30) / per;
  s->slots = (int)std::max<size_t>(1, std::min(std::min<size_t>(by_vox, 64), by_mem));
  hipError_t e = hold(s, t, s->slots, &s->held);
  if (e != hipSuccess && s->slots > 1) {
    (void)hipGetLastError();
    s->slots = 1;
    e = hold(s, t, 1, &s->held);
  }
  s->grad_slots = 1;
  return e == hipSuccess ? hold(s, g, 1, &s->grad_held) : e;
}

// The gradients' tensors for as many samples as the forward's, at the first batch that has more than one;
// one sample at a time stays possible where the device has no room. No kernel of the network is running.
hipError_t hold_gradients(mcpet_surrogate* s, int batch)
{
  if (batch <= s->grad_slots || s->grad_slots == s->slots || s->grad_full) return hipSuccess;
  void* const one = s->grad_held;
  const hipError_t e = hold(s, sample_tensors(s, true), s->slots, &s->grad_held);
  if (s->grad_held == one) {   // no room
    (void)hipGetLastError();
    s->grad_full = true;
    return hipSuccess;
  }
  s->grad_slots = s->slots;
  const hipError_t f = hipFree(one);
  return e == hipSuccess ? f : e;
}

// samples per pass of a batch: equal groups of at most `slots`
int sample_group(int slots, int batch)
{
  const int groups = (batch + slots - 1) / slots;
  return (batch + groups - 1) / groups;
}

}  // namespace

extern "C" mcpet_status mcpet_surrogate_create(int32_t D, int32_t H, int32_t W, int32_t in_channels, int32_t width, uint64_t seed,
                                               mcpet_surrogate** out)
{
  if (!out) return serr(nullptr, MCPET_E_ARG, "mcpet_surrogate_create: null output pointer");
  *out = nullptr;
  if (D < 4 || H < 4 || W < 4 || D % 4 || H % 4 || W % 4 || in_channels < 1 || width < 1 || in_channels > 64 || width > 256 ||
      (long long)D * H * W > (1LL << 28))
    return serr(nullptr, MCPET_E_ARG, "mcpet_surrogate_create: sizes must be multiples of 4 (at most 2^28 voxels), "
                                      "1 <= channels <= 64, 1 <= width <= 256");
  mcpet_surrogate* s = new mcpet_surrogate();
  s->D = D;
  s->H = H;
  s->W = W;
  s->cin = in_channels;
  s->c = width;
  const int c = width;
  const int spec[9][4] = {{in_channels, c, 3, 1}, {c, c, 3, 1},         {c, 2 * c, 3, 2},     {2 * c, 2 * c, 3, 1}, {2 * c, 4 * c, 3, 2},
                          {4 * c, 4 * c, 3, 1},    {6 * c, 2 * c, 3, 1}, {3 * c, c, 3, 1},     {c, 1, 1, 1}};
  size_t off = 0, offb = 0;
  for (int i = 0; i < 9; i++) {
    Conv& l = s->L[i];
    l.cin = spec[i][0];
    l.cout = spec[i][1];
    l.ks = spec[i][2];
    l.stride = spec[i][3];
    const int T = l.ks * l.ks * l.ks;
    l.w = off;
    off += (size_t)l.cout * l.cin * T;
    l.b = off;
    off += (size_t)l.cout;
    l.rows_f = rows_for(l.cout);
    l.kp_f = rup(T * rup(l.cin, 8), 32);
    l.rows_b = rows_for(l.cin);
    l.kp_b = rup(T * rup(l.cout, 8), 32);
    l.wf = offb;
    offb += (size_t)l.rows_f * l.kp_f;
    l.wb = offb;
    offb += (size_t)l.rows_b * l.kp_b;
  }
  s->n_params = off;
  s->n_bf16 = offb;
  s->vx = {in_channels, D, H, W};
  s->va1 = {c, D, H, W};
  s->vcat1 = {3 * c, D, H, W};
  s->vd1 = {2 * c, D / 2, H / 2, W / 2};
  s->vcat2 = {6 * c, D / 2, H / 2, W / 2};
  s->vd2 = {4 * c, D / 4, H / 4, W / 4};
  s->vb3 = {4 * c, D / 4, H / 4, W / 4};
  s->ve2 = {2 * c, D / 2, H / 2, W / 2};
  s->ve1 = {c, D, H, W};
  s->vr = {1, D, H, W};
  hipError_t e = hipGetDevice(&s->device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&s->st, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreate(&s->ev_f0);
  if (e == hipSuccess) e = hipEventCreate(&s->ev_f1);
  for (hipEvent_t* ev : {&s->ev_in[0], &s->ev_in[1], &s->ev_out})
    if (e == hipSuccess) e = hipEventCreateWithFlags(ev, hipEventDisableTiming);
  if (e == hipSuccess) e = hipHostMalloc((void**)&s->h_decays, sizeof(unsigned long long), hipHostMallocDefault);
  struct A {
    float** p;
    size_t n;
  } al[] = {{&s->p, off},          {&s->g, off},          {&s->m, off},           {&s->v, off},
            {&s->sse, 1}, {&s->raw_s, s->vr.size()}, {&s->raw_t, s->vr.size()}, {&s->est, s->vr.size()}};
  for (auto& a : al)
    if (e == hipSuccess) e = dalloc_t(s, a.p, a.n);
  if (e == hipSuccess) e = dalloc_t(s, &s->wbf, s->n_bf16);
  if (e == hipSuccess) e = dalloc_t(s, &s->sums, 257);
  if (e == hipSuccess) e = dalloc_t(s, &s->bw_part, kBwPartFloats);
  if (e == hipSuccess) e = hold_samples(s);
  const size_t vox = (size_t)D * H * W;
  if (e == hipSuccess)
    e = hipHostMalloc((void**)&s->h_stage, sizeof(float) * vox * std::max(2, s->slots), hipHostMallocDefault);
  // at most 2 MB a half
  s->stage_in = 2 * std::min<size_t>((size_t)1 << 19, vox * in_channels * s->slots);
  if (e == hipSuccess) e = hipHostMalloc((void**)&s->h_in, sizeof(float) * s->stage_in, hipHostMallocDefault);
  if (e != hipSuccess) {
    std::string m = std::string("mcpet_surrogate_create: ") + hipGetErrorString(e);
    mcpet_surrogate_destroy(s);
    return serr(nullptr, MCPET_E_NOMEM, m);
  }
  // He-normal weights from a seeded generator (splitmix64 + Box-Muller), zero biases; the 1x1x1
  // output layer is zero, so the untrained network returns its input channel 0
  std::vector<float> hp(off, 0.0f);
  uint64_t z = seed ? seed : 0x9E3779B97F4A7C15ull;
  auto next = [&]() {
    z += 0x9E3779B97F4A7C15ull;
    uint64_t x = z;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    x ^= x >> 31;
    return (double)((x >> 11) + 1) * 0x1.0p-53;
  };
  for (int i = 0; i < 9; i++) {
    const Conv& l = s->L[i];
    const int T = l.ks * l.ks * l.ks;
    const double sd = i == 8 ? 0.0 : std::sqrt(2.0 / (l.cin * T));   // the output layer starts at zero: identity
    for (size_t k = 0; k < (size_t)l.cout * l.cin * T; k++)
      hp[l.w + k] = (float)(sd * std::sqrt(-2.0 * std::log(next())) * std::cos(6.283185307179586 * next()));
  }
  e = hipMemcpy(s->p, hp.data(), sizeof(float) * off, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = derive(s);
  if (e == hipSuccess) e = hipStreamSynchronize(s->st);
  if (e != hipSuccess) {
    mcpet_surrogate_destroy(s);
    return serr(nullptr, MCPET_E_HIP, "mcpet_surrogate_create: upload");
  }
  *out = s;
  return MCPET_OK;
}

extern "C" int64_t mcpet_surrogate_param_count(const mcpet_surrogate* s) { return s ? (int64_t)s->n_params : 0; }

extern "C" mcpet_status mcpet_surrogate_get_params(mcpet_surrogate* s, float* out)
{
  if (!s || !out) return serr(s, MCPET_E_ARG, "mcpet_surrogate_get_params: null argument");
  SHIP(s, hipStreamSynchronize(s->st));
  SHIP(s, hipMemcpy(out, s->p, sizeof(float) * s->n_params, hipMemcpyDeviceToHost));
  return MCPET_OK;
}
extern "C" mcpet_status mcpet_surrogate_set_params(mcpet_surrogate* s, const float* in)
{
  if (!s || !in) return serr(s, MCPET_E_ARG, "mcpet_surrogate_set_params: null argument");
  SHIP(s, hipStreamSynchronize(s->st));
  SHIP(s, hipMemcpy(s->p, in, sizeof(float) * s->n_params, hipMemcpyHostToDevice));
  SHIP(s, derive(s));
  SHIP(s, hipStreamSynchronize(s->st));
  return MCPET_OK;
}

// The pinned buffers (h_in, h_stage) are free whenever a call begins: every call that uses them waits for
// its stream before it returns, also where it returns an error (staged_end).
static mcpet_status staged_end(mcpet_surrogate* s, mcpet_status st)
{
  if (st != MCPET_OK) (void)hipStreamSynchronize(s->st);
  s->in_turn = 0;
  s->in_used[0] = s->in_used[1] = false;
  return st;
}

static mcpet_status batch_forward(mcpet_surrogate* s, const float* x, int32_t batch, float* y, double* gflop)
{
  const size_t nx = s->vx.size(), nv = s->vr.size();
  const int group = sample_group(s->slots, batch);
  SHIP(s, stage_input(s, x, std::min(group, batch)));
  for (int b = 0; b < batch; b += group) {
    const int n = std::min(group, batch - b), next = std::min(group, batch - b - n);
    const bool last = next == 0;
    if (last) SHIP(s, hipEventRecord(s->ev_f0, s->st));
    SHIP(s, forward(s, n, s->h_stage));   // the last layer writes to the host
    if (last) SHIP(s, hipEventRecord(s->ev_f1, s->st));
    if (last) {
      SHIP(s, hipStreamSynchronize(s->st));
    } else {
      SHIP(s, hipEventRecord(s->ev_out, s->st));
      SHIP(s, stage_input(s, x + (b + n) * nx, next));   // the next group's input, behind this one's layers
      SHIP(s, hipEventSynchronize(s->ev_out));
    }
    std::memcpy(y + b * nv, s->h_stage, sizeof(float) * nv * n);
  }
  s->fwd_timed = batch - (batch - 1) / group * group;
  if (gflop) *gflop = s->flops_fwd * 1e-9;
  return MCPET_OK;
}

// x: batch x cin x D x H x W, y (out): batch x D x H x W; returns the forward GFLOP per sample.
extern "C" mcpet_status mcpet_surrogate_forward(mcpet_surrogate* s, const float* x, int32_t batch, float* y, double* gflop)
{
  if (!s || !x || !y || batch < 1) return serr(s, MCPET_E_ARG, "mcpet_surrogate_forward: bad arguments");
  return staged_end(s, batch_forward(s, x, batch, y, gflop));
}

// Device time per sample of the network in the last mcpet_surrogate_forward (its last samples that
// went through together: the layers from the converted input to the output, HIP events on the network's
// stream; k_input, which converts the input while it reads it from pinned host memory, comes before).
extern "C" mcpet_status mcpet_surrogate_forward_ms(mcpet_surrogate* s, double* ms)
{
  if (!s || !ms) return serr(s, MCPET_E_ARG, "mcpet_surrogate_forward_ms: null argument");
  if (!s->fwd_timed) return serr(s, MCPET_E_STATE, "mcpet_surrogate_forward_ms: no forward yet");
  float t = 0.0f;
  SHIP(s, hipEventElapsedTime(&t, s->ev_f0, s->ev_f1));
  *ms = t / s->fwd_timed;
  return MCPET_OK;
}

// One estimate from the last run of ctx, all on the device: rebinning of its scatter and
// trues onto the network's grid, normalisation (counts times float(voxels / total trues), the
// total exact in double), the network, and scatter per decay = max(output, 0) times
// float(total trues / (voxels * decays)).
void mcpet_surrogate_dims(const mcpet_surrogate* s, int* D, int* H, int* W, int* cin)
{
  *D = s->D;
  *H = s->H;
  *W = s->W;
  *cin = s->cin;
}

static mcpet_status run_estimate(mcpet_surrogate* s, mcpet_ctx* ctx, float* estimate, float* scatter_counts, int64_t* decays)
{
  if (s->cin != 2 && s->cin != 4)
    return serr(s, MCPET_E_ARG, "mcpet_surrogate_estimate: the network must take 2 or 4 input channels");
  if (mcpet_ctx_device(ctx) != s->device) return serr(s, MCPET_E_ARG, "mcpet_surrogate_estimate: context on another device");
  SHIP(s, hipSetDevice(s->device));
  const size_t nv = s->vr.size();
  // everything below is enqueued behind the context's run on the device: the host waits once,
  // for the outputs
  mcpet_status st = mcpet_ctx_rebin2_device(ctx, 1, 0, s->D, s->H, s->W, s->raw_s, s->raw_t, s->st);
  const unsigned long long* d_decays = mcpet_ctx_decay_counter(ctx);
  const float* maps = nullptr;
  if (st == MCPET_OK && s->cin == 4) st = mcpet_ctx_project_device(ctx, s->D, s->H, s->W, &maps);
  if (st != MCPET_OK) return serr(s, st, std::string("mcpet_surrogate_estimate: ") + mcpet_last_error(ctx));
  if (maps)   // the scaled activity integrals and the attenuation factors
    SHIP(s, hipMemcpyAsync(s->x0 + 2 * nv, maps + nv, 2 * sizeof(float) * nv, hipMemcpyDeviceToDevice, s->st));
  hipLaunchKernelGGL(k_sum_partial, dim3(256), dim3(256), 0, s->st, s->raw_t, nv, s->sums);
  hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(256), 0, s->st, s->sums, 256, s->sums + 256);
  hipLaunchKernelGGL(k_normalize, dim3(blocks_for(nv)), dim3(256), 0, s->st, s->raw_s, s->raw_t, s->x0, nv, s->sums + 256);
  SHIP(s, hipGetLastError());
  hipLaunchKernelGGL(k_input, dim3(blocks_for(nv * (rup(s->cin, 8) / 8))), dim3(256), 0, s->st, (const float*)s->x0, s->cin, nv,
                     (size_t)0, nv, (float*)nullptr, cl(s->x0l, s->cin));
  SHIP(s, hipGetLastError());
  SHIP(s, forward(s, 1, s->out));
  hipLaunchKernelGGL(k_estimate, dim3(blocks_for(nv)), dim3(256), 0, s->st, s->out, s->est, nv, s->sums + 256, d_decays);
  SHIP(s, hipGetLastError());
  // through pinned staging (one DMA per output), then host copies into the caller's buffers
  SHIP(s, hipMemcpyAsync(s->h_stage, s->est, sizeof(float) * nv, hipMemcpyDeviceToHost, s->st));
  if (scatter_counts) SHIP(s, hipMemcpyAsync(s->h_stage + nv, s->raw_s, sizeof(float) * nv, hipMemcpyDeviceToHost, s->st));
  SHIP(s, hipMemcpyAsync(s->h_decays, d_decays, sizeof(unsigned long long), hipMemcpyDeviceToHost, s->st));
  SHIP(s, hipStreamSynchronize(s->st));
  std::memcpy(estimate, s->h_stage, sizeof(float) * nv);
  if (scatter_counts) std::memcpy(scatter_counts, s->h_stage + nv, sizeof(float) * nv);
  if (decays) *decays = (int64_t)*s->h_decays;
  return MCPET_OK;
}

extern "C" mcpet_status mcpet_surrogate_estimate(mcpet_surrogate* s, mcpet_ctx* ctx, float* estimate, float* scatter_counts,
                                                 int64_t* decays)
{
  if (!s || !ctx || !estimate) return serr(s, MCPET_E_ARG, "mcpet_surrogate_estimate: null argument");
  return staged_end(s, run_estimate(s, ctx, estimate, scatter_counts, decays));
}

// Mean-squared-error gradients of the batch (loss = mean over batch and voxels); leaves them
// in the device buffer for an optimiser step.
static mcpet_status batch_gradients(mcpet_surrogate* s, const float* x, const float* target, int32_t batch, float* loss)
{
  const size_t nx = s->vx.size(), nv = s->vr.size();
  SHIP(s, hold_gradients(s, batch));
  hipLaunchKernelGGL(k_zero, dim3(blocks_for(s->n_params)), dim3(256), 0, s->st, s->g, s->n_params);
  hipLaunchKernelGGL(k_zero, dim3(1), dim3(256), 0, s->st, s->sse, (size_t)1);
  SHIP(s, hipGetLastError());
  const float scale = 1.0f / ((float)nv * (float)batch);
  const int group = sample_group(s->grad_slots, batch);
  for (int b = 0; b < batch; b += group) {
    const int n = std::min(group, batch - b);
    if (b) SHIP(s, hipEventSynchronize(s->ev_out));   // the last group's targets have been read
    std::memcpy(s->h_stage, target + b * nv, sizeof(float) * nv * n);
    SHIP(s, stage_input(s, x + b * nx, n));
    SHIP(s, forward(s, n, s->out));
    hipLaunchKernelGGL(k_loss, dim3(blocks_for(nv), n), dim3(256), 0, s->st, s->out, (const float*)s->h_stage, s->gr, scale, s->sse,
                       (int)nv, ClOut{s->grl, 8, 0});
    SHIP(s, hipEventRecord(s->ev_out, s->st));
    SHIP(s, hipGetLastError());
    SHIP(s, backward(s, n));
  }
  float sse = 0.0f;
  SHIP(s, hipMemcpyAsync(&sse, s->sse, sizeof(float), hipMemcpyDeviceToHost, s->st));
  SHIP(s, hipStreamSynchronize(s->st));
  if (loss) *loss = sse * scale;
  return MCPET_OK;
}

extern "C" mcpet_status mcpet_surrogate_gradients(mcpet_surrogate* s, const float* x, const float* target, int32_t batch,
                                                  float* loss, float* grad)
{
  if (!s || !x || !target || batch < 1) return serr(s, MCPET_E_ARG, "mcpet_surrogate_gradients: bad arguments");
  mcpet_status st = staged_end(s, batch_gradients(s, x, target, batch, loss));
  if (st != MCPET_OK || !grad) return st;
  SHIP(s, hipMemcpy(grad, s->g, sizeof(float) * s->n_params, hipMemcpyDeviceToHost));
  return MCPET_OK;
}

// One Adam step (beta 0.9, 0.999, eps 1e-8) on the batch's MSE.
extern "C" mcpet_status mcpet_surrogate_train_step(mcpet_surrogate* s, const float* x, const float* target, int32_t batch,
                                                   float lr, float* loss)
{
  if (!s || !x || !target || batch < 1 || !(lr > 0.0f)) return serr(s, MCPET_E_ARG, "mcpet_surrogate_train_step: bad arguments");
  mcpet_status st = staged_end(s, batch_gradients(s, x, target, batch, loss));
  if (st != MCPET_OK) return st;
  s->t_adam++;
  const float c1 = 1.0f - std::pow(0.9f, (float)s->t_adam), c2 = 1.0f - std::pow(0.999f, (float)s->t_adam);
  hipLaunchKernelGGL(k_adam, dim3(blocks_for(s->n_params)), dim3(256), 0, s->st, s->p, s->g, s->m, s->v, s->n_params, lr, 0.9f,
                     0.999f, 1e-8f, c1, c2);
  SHIP(s, hipGetLastError());
  SHIP(s, derive(s));
  SHIP(s, hipStreamSynchronize(s->st));
  return MCPET_OK;
}

extern "C" void mcpet_surrogate_destroy(mcpet_surrogate* s)
{
  if (!s) return;
  if (s->st) (void)hipStreamSynchronize(s->st);
  for (void* p : s->allocs) (void)hipFree(p);
  for (void* p : {s->held, s->grad_held})
    if (p) (void)hipFree(p);
  if (s->h_stage) (void)hipHostFree(s->h_stage);
  if (s->h_in) (void)hipHostFree(s->h_in);
  for (hipEvent_t ev : {s->ev_in[0], s->ev_in[1], s->ev_out})
    if (ev) (void)hipEventDestroy(ev);
  if (s->h_decays) (void)hipHostFree(s->h_decays);
  if (s->ev_f0) (void)hipEventDestroy(s->ev_f0);
  if (s->ev_f1) (void)hipEventDestroy(s->ev_f1);
  if (s->st) (void)hipStreamDestroy(s->st);
  delete s;
}

extern "C" const char* mcpet_surrogate_last_error(const mcpet_surrogate* s)
{
  if (s && !s->err.empty()) return s->err.c_str();
  return mcpet_last_error(nullptr);
}

namespace {

// ------------------------------------------------------------------ sinogram rebinning

// One workgroup per (angle group h, plane group d): the sinograms of the plane group (CSR list)
// times the group's angle rows are read as whole radial rows (coalesced), each count added to
// the LDS sum of its radial group. out[(d H + h) W + w] = float(sum).
__global__ __launch_bounds__(256) void k_rebin(const int* __restrict__ sino, const int* __restrict__ grp_off,
                                               const int* __restrict__ grp_sino, int nangles, int nrad, int H, int W, int gh,
                                               int gw, float* __restrict__ out)
{
  __shared__ unsigned long long acc[256];
  const int h = blockIdx.x, d = blockIdx.y;
  for (int i = threadIdx.x; i < W; i += blockDim.x) acc[i] = 0ull;
  __syncthreads();
  const int a0 = h * gh, rows = max(0, min(gh, nangles - a0));
  const int j0 = grp_off[d], nj = grp_off[d + 1] - j0;
  const long long items = (long long)nj * rows * nrad;
  for (long long it = threadIdx.x; it < items; it += blockDim.x) {
    const int r = (int)(it % nrad);
    const long long q = it / nrad;
    const int a = (int)(q % rows), j = (int)(q / rows);
    const int v = sino[((size_t)grp_sino[j0 + j] * nangles + a0 + a) * nrad + r];
    if (v) atomicAdd(&acc[r / gw], (unsigned long long)(unsigned)v);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < W; i += blockDim.x) out[((size_t)d * H + h) * W + i] = (float)acc[i];
}

// The same sums for NRAD <= 256 without atomics: thread r owns radial bin r and adds it up
// over the group's sinogram rows (each row read whole, coalesced), then the radial groups are
// summed from LDS in order.
__global__ __launch_bounds__(256) void k_rebin_rows(const int* __restrict__ sino, const int* __restrict__ grp_off,
                                                    const int* __restrict__ grp_sino, int nangles, int nrad, int H, int W,
                                                    int gh, int gw, float* __restrict__ out)
{
  __shared__ unsigned long long bin[256];
  const int h = blockIdx.x, d = blockIdx.y, r = threadIdx.x;
  const int a0 = h * gh, rows = max(0, min(gh, nangles - a0));
  const int j0 = grp_off[d], nj = grp_off[d + 1] - j0;
  unsigned long long acc = 0ull;
  if (r < nrad)
    for (int j = 0; j < nj; j++) {
      const int* row = sino + ((size_t)grp_sino[j0 + j] * nangles + a0) * nrad + r;
      for (int a = 0; a < rows; a++) acc += (unsigned)row[(size_t)a * nrad];
    }
  bin[r] = acc;
  __syncthreads();
  if (r < W) {
    unsigned long long t = 0ull;
    for (int i = r * gw; i < min(nrad, r * gw + gw); i++) t += bin[i];
    out[((size_t)d * H + h) * W + r] = (float)t;
  }
}

// k_rebin_rows for two tallies of the same geometry in one pass, with the group's sinogram rows
// dealt to RB_SLICES slices of RB_LANES threads (thread r of slice s adds rows j = s, s + RB_SLICES,
// ... of radial bin r), so five times as many rows are read at once; the slices' integer sums
// are added in LDS in slice order. The same integer sums as two k_rebin_rows launches.
#define RB_LANES 192
#define RB_SLICES 5
__global__ __launch_bounds__(RB_LANES * RB_SLICES) void k_rebin_rows2(const int* __restrict__ sa, const int* __restrict__ sb,
                                                                      const int* __restrict__ grp_off,
                                                                      const int* __restrict__ grp_sino, int nangles, int nrad,
                                                                      int H, int W, int gh, int gw, float* __restrict__ oa,
                                                                      float* __restrict__ ob)
{
  __shared__ unsigned long long bin[RB_SLICES][2][RB_LANES];
  const int h = blockIdx.x, d = blockIdx.y;
  const int r = threadIdx.x % RB_LANES, sl = threadIdx.x / RB_LANES;
  const int a0 = h * gh, rows = max(0, min(gh, nangles - a0));
  const int j0 = grp_off[d], nj = grp_off[d + 1] - j0;
  unsigned long long acc_a = 0ull, acc_b = 0ull;
  if (r < nrad && rows > 0) {
    // rows (j, a) of the group, a fastest, dealt round-robin to the slices; the loop is unrolled
    // so that several rows' loads are in flight per thread
    const int items = nj * rows;
#pragma unroll 4
    for (int it = sl; it < items; it += RB_SLICES) {
      const int j = it / rows, a = it - j * rows;
      const size_t off = ((size_t)grp_sino[j0 + j] * nangles + a0 + a) * nrad + r;
      acc_a += (unsigned)sa[off];
      acc_b += (unsigned)sb[off];
    }
  }
  bin[sl][0][r] = acc_a;
  bin[sl][1][r] = acc_b;
  __syncthreads();
  if (sl == 0 && r < W) {
    unsigned long long ta = 0ull, tb = 0ull;
    for (int i = r * gw; i < min(nrad, r * gw + gw); i++)
      for (int k = 0; k < RB_SLICES; k++) {
        ta += bin[k][0][i];
        tb += bin[k][1][i];
      }
    oa[((size_t)d * H + h) * W + r] = (float)ta;
    ob[((size_t)d * H + h) * W + r] = (float)tb;
  }
}

__global__ void k_i2f2(const int* __restrict__ a, const int* __restrict__ b, float* __restrict__ oa, float* __restrict__ ob,
                       size_t n)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  oa[i] = (float)a[i];
  ob[i] = (float)b[i];
}

}  // namespace

hipError_t mcpet_launch_i2f2(const int* a, const int* b, float* oa, float* ob, size_t n, hipStream_t st)
{
  hipLaunchKernelGGL(k_i2f2, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, b, oa, ob, n);
  return hipGetLastError();
}

hipError_t mcpet_launch_rebin2(const int* sa, const int* sb, const int* grp_off, const int* grp_sino, int nangles, int nrad, int D,
                               int H, int W, int gh, int gw, float* oa, float* ob, hipStream_t st)
{
  if (W > RB_LANES || nrad > RB_LANES) {
    hipError_t e = mcpet_launch_rebin(sa, grp_off, grp_sino, nangles, nrad, D, H, W, gh, gw, oa, st);
    return e == hipSuccess ? mcpet_launch_rebin(sb, grp_off, grp_sino, nangles, nrad, D, H, W, gh, gw, ob, st) : e;
  }
  hipLaunchKernelGGL(k_rebin_rows2, dim3(H, D), dim3(RB_LANES * RB_SLICES), 0, st, sa, sb, grp_off, grp_sino, nangles, nrad, H,
                     W, gh, gw, oa, ob);
  return hipGetLastError();
}

hipError_t mcpet_launch_rebin(const int* sino, const int* grp_off, const int* grp_sino, int nangles, int nrad, int D, int H, int W,
                              int gh, int gw, float* out, hipStream_t st)
{
  if (W > 256) return hipErrorInvalidValue;
  if (nrad <= 256)
    hipLaunchKernelGGL(k_rebin_rows, dim3(H, D), dim3(256), 0, st, sino, grp_off, grp_sino, nangles, nrad, H, W, gh, gw, out);
  else
    hipLaunchKernelGGL(k_rebin, dim3(H, D), dim3(256), 0, st, sino, grp_off, grp_sino, nangles, nrad, H, W, gh, gw, out);
  return hipGetLastError();
}

// ------------------------------------------------------------------ self test of the GEMM

extern "C" mcpet_status mcpet_selftest_gemm_bf16(const float* a, const float* b, int32_t M, int32_t N, int32_t K, int32_t split,
                                                 float* c)
{
  if (!a || !b || !c || M < 1 || N < 1 || K < 1 || split < 1) {
    mcpet_host_set_error("selftest_gemm_bf16: bad args");
    return MCPET_E_ARG;
  }
  float *da = nullptr, *db = nullptr, *dc = nullptr;
  hipError_t e = hipMalloc((void**)&da, 4 * (size_t)M * K);
  if (e == hipSuccess) e = hipMalloc((void**)&db, 4 * (size_t)K * N);
  if (e == hipSuccess) e = hipMalloc((void**)&dc, 4 * (size_t)M * N);
  if (e == hipSuccess) e = hipMemcpy(da, a, 4 * (size_t)M * K, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(db, b, 4 * (size_t)K * N, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(dc, 0, 4 * (size_t)M * N);
  if (e == hipSuccess) e = gemm(Dense{da, M, K, K}, Dense{db, K, N, N}, dc, M, N, K, N, nullptr, split, false, 0);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(c, dc, 4 * (size_t)M * N, hipMemcpyDeviceToHost);
  if (da) (void)hipFree(da);
  if (db) (void)hipFree(db);
  if (dc) (void)hipFree(dc);
  if (e != hipSuccess) {
    mcpet_host_set_error((std::string("selftest_gemm_bf16: ") + hipGetErrorString(e)).c_str());
    return MCPET_E_HIP;
  }
  return MCPET_OK;
}
