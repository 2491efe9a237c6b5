// 3-D convolutional surrogate of the multi-scale Frangi stack (gfx950).
//
// The network (5 layers of 3x3x3 "valid" convolutions, 24 channels, GELU
// between layers) has no counterpart in the reference; it stands in for
// filters/ridges.py:322-476 (python/cucim/src/cucim/skimage/) and its output
// is compared with the plain kernels'.
//
// Activations are channels-last bfloat16 volumes (D, H, W, C); weights are
// bfloat16, accumulation float32 on the matrix cores:
//
//   k_conv3d_24x24  24 -> 24 channels, GELU: implicit GEMM with M = output
//       channels (16 per tile), N = 16 voxels along x, K = taps x channels
//   k_conv3d_1x24   1 -> 24, GELU
//   k_conv3d_24x1   24 -> 1
//       all on v_mfma_f32_16x16x32_bf16: lane l holds A[l % 16][8 (l / 16) + j],
//       B[8 (l / 16) + j][l % 16] and D[4 (l / 16) + r][l % 16].  The weights
//       are the A operand, so a lane ends with four consecutive channels of
//       one voxel and stores them as one word.  The bias is added to the
//       finished sum (as the accumulators' start it would cost the products'
//       partial sums its bits).  Weights arrive pre-packed in each kernel's A
//       order (k_pack_weights).
//   k_pad_bf16        reflect / nearest / ... padding of a float32 volume into
//                     the bfloat16 single-channel input of the first layer
//   training kernels  (float32): MSE gradient, Adam step, bf16 packing.  The
//                     training step takes its gradients from k_cnn3d_bwd.hip;
//                     the GELU backward, input gradient and weight / bias
//                     gradients here (one work-item per sum) serve the C
//                     entries for one patch of any channel counts.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "hc_cnn.h"

namespace hc {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
// the caller's output arrays need no more than their elements' alignment
typedef __bf16 bf16x4_out __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4_out __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kC = 24;
constexpr int kBY = 8, kBX = 16;             // output block rows / columns
constexpr int kTY = kBY + 2, kTX = kBX + 2;  // input tile rows / columns

enum { ACT_NONE = 0, ACT_GELU = 1, ACT_CLAMP01 = 2 };

struct ConvArgs {
  const __bf16* in;   // (B, D, H, W, CI)
  void* out;          // (B, D-2, H-2, W-2, CO): bf16, or float32 (24 -> 1)
  float* pre;         // optional float32 pre-activation (training), or null
  const bf16x8* wpk;  // packed weights
  const float* bias;  // CO
  int D, H, W;        // input extents
  int nbx, nby, nbz;  // blocks along x, y, z of one patch
  int64_t nblocks;    // of the whole batch
  int act;            // 24 -> 1
};

// Block b of the output grid (x fastest, patches slowest; fewer than 2^31
// blocks) -> origin; returns the patch.
template <int BZ>
__device__ __forceinline__ int64_t block_origin(const ConvArgs& a, int64_t b, int& x0, int& y0,
                                                int& z0) {
  unsigned q = (unsigned)b;
  unsigned r = q / (unsigned)a.nbx;
  x0 = (int)(q - r * a.nbx) * kBX;
  q = r / (unsigned)a.nby;
  y0 = (int)(r - q * a.nby) * kBY;
  r = q / (unsigned)a.nbz;
  z0 = (int)(q - r * a.nbz) * BZ;
  return r;
}

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// GELU of four channels of a voxel, stored as bf16 (and the pre-activations
// as float32 in training).
__device__ __forceinline__ void store_gelu4(const ConvArgs& a, int64_t o, f32x4 p) {
  if (a.pre) *reinterpret_cast<f32x4_out*>(a.pre + o) = p;
  bf16x4 y;
#pragma unroll
  for (int r = 0; r < 4; ++r) y[r] = f2bf(gelu(p[r]));
  *reinterpret_cast<bf16x4_out*>(reinterpret_cast<__bf16*>(a.out) + o) = y;
}

// The second channel tile holds 8 channels (16 .. 23) in lanes 0 .. 31 only;
// the results of two rows are joined, so that every lane has four channels to
// activate: lanes 0 .. 31 those of `lo`, lanes 32 .. 63 those of `hi`'s lanes
// 0 .. 31.
__device__ __forceinline__ f32x4 join_halves(f32x4 lo, f32x4 hi) {
  f32x4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo[r]), __float_as_uint(hi[r]),
                                                    false, false);
    v[r] = __uint_as_float(s[0]);
  }
  return v;
}

// 24 -> 24.  A work-group of eight waves computes BZ x 8 x 16 voxels, a wave
// MR = BZ rows of one plane.  K is ordered (dy)(dz, dx, octet of channels): the
// 27 (dz, dx, octet) groups of 8 make 7 steps of 4, and one 16-byte LDS read
// per lane (an input row) serves the three dy of a step, i.e. three output
// rows: 10 reads and 6 weight reads for 48 matrix instructions (MR = 8),
// against 16 + 8 for 32 with a row read per tap, which left LDS the bound.
// The activation takes about as long on the vector ALU as the products on the
// matrix cores, so of the two waves of a SIMD the first activates a block
// after its products and the second before those of its next block: one's
// activation runs during the other's products.  The input tile of the next
// block is loaded into registers meanwhile, a wave per row, clamped to the
// volume (what lies outside reaches no stored output).  A layer of 260^3
// voxels: 1.30 ms with a row read per tap, 0.83 with rows shared by three dy,
// 0.75 with hand-pipelined LDS reads and the two waves' phases apart; the same
// without the products takes 0.44 (2.1 GB at memory speed) and without the
// activation 0.73.
constexpr int k24Steps = 7;
constexpr int k24Row = kTX * kC / 8;  // 16-byte words of a tile row (54)

template <int BZ>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void
k_conv3d_24x24(const ConvArgs a) {
  constexpr int MR = BZ, NR = MR + 2, ROWS = (BZ + 2) * kTY;
  constexpr int NW = k24Steps * 3 * 2 * 64;  // 16-byte words of weights
  constexpr int NPF = (ROWS + 7) / 8;        // rows that a wave stages
  extern __shared__ __align__(16) unsigned char smem[];
  bf16x8* Wl = reinterpret_cast<bf16x8*>(smem);
  bf16x8* T = Wl + NW;  // [ROWS][54]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kg = lane >> 4;
  for (int i = tid; i < NW; i += 512) Wl[i] = a.wpk[i];
  const int64_t G = gridDim.x;
  const int64_t slot = xcd_swizzle(blockIdx.x, G);
  const int OD = a.D - 2, OH = a.H - 2, OW = a.W - 2;
  const int lw = min(lane, k24Row - 1);  // this lane's word of a row
  bf16x8 pf[NPF];
  auto fetch = [&](int64_t b) {
    int x0, y0, z0;
    const int64_t n = block_origin<BZ>(a, b, x0, y0, z0);
    const int xo = min(x0 + lw / 3, a.W - 1) * 3 + lw % 3;
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int r = wv + 8 * u;
      const int gy = min(y0 + r % kTY, a.H - 1), gz = min(z0 + r / kTY, a.D - 1);
      pf[u] = reinterpret_cast<const bf16x8*>(a.in + ((n * a.D + gz) * a.H + gy) * a.W * kC)[xo];
    }
  };
  // this lane's input word of K group 4 s + kg, relative to its voxel
  int koff[k24Steps];
#pragma unroll
  for (int s = 0; s < k24Steps; ++s) {
    const int q = 4 * s + kg;  // (dz, dx, octet); group 27 has zero weights
    koff[s] = q < 27 ? (q / 9 * kTY * kTX + q / 3 % 3) * 3 + q % 3 : 0;
  }
  f32x4 bias0, bias1;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    bias0[r] = a.bias[4 * kg + r];
    bias1[r] = a.bias[16 + 4 * (kg & 1) + r];
  }
  const int pz = wv * MR / kBY, py = wv * MR % kBY;  // this wave's plane and first row
  f32x4 acc[MR][2];
  auto activate = [&](int64_t b) {
    int x0, y0, z0;
    const int64_t n = block_origin<BZ>(a, b, x0, y0, z0);
    const int gz = z0 + pz, gx = x0 + li, gy = y0 + py;
    const int64_t o0 = (((n * OD + gz) * OH + gy) * OW + x0) * kC;
    const int ol = li * kC + 4 * kg, oh = li * kC + 16 + 4 * (kg & 1), k = kg >> 1;
    const bool in = gz < OD && gx < OW;
#pragma unroll
    for (int m = 0; m < MR; m += 2) {
      const int64_t o = o0 + (int64_t)m * OW * kC;
      if (in && gy + m < OH) store_gelu4(a, o + ol, acc[m][0] + bias0);
      if (in && gy + m + 1 < OH) store_gelu4(a, o + OW * kC + ol, acc[m + 1][0] + bias0);
      const f32x4 v = join_halves(acc[m][1], acc[m + 1][1]) + bias1;
      if (in && gy + m + k < OH) store_gelu4(a, o + k * OW * kC + oh, v);
    }
  };
  // the loads above are waited for here, not in the loop, where the wait would
  // include the next block's tile
  __builtin_amdgcn_s_waitcnt(0);
  const bool late = wv >= 4;  // the second wave of a SIMD
  int64_t prev = -1;
  if (slot < a.nblocks) fetch(slot);
  for (int64_t blk = slot; blk < a.nblocks; blk += G) {  // uniform per work-group
    __syncthreads();  // the previous block's reads are done
#pragma unroll
    for (int u = 0; u < NPF; ++u) {
      const int r = wv + 8 * u;
      if (lane < k24Row && r < ROWS) T[r * k24Row + lane] = pf[u];
    }
    if (blk + G < a.nblocks) fetch(blk + G);  // in flight during the products
    __syncthreads();
    if (late && prev >= 0) activate(prev);
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8* row = T + (pz * kTY + py) * k24Row + li * 3;
    // Pipelined by hand (left alone, the compiler reads a row right before its
    // products and waits for it): row i + 3 and one of the next step's weights
    // are read while the products of row i run.
    bf16x8 x[4], w[2][6];
    auto load_x = [&](int i) { return row[koff[i / NR] + i % NR * k24Row]; };
    auto load_w = [&](int s, int k) { return Wl[(s * 6 + k) * 64 + lane]; };
#pragma unroll
    for (int k = 0; k < 6; ++k) w[0][k] = load_w(0, k);
#pragma unroll
    for (int i = 0; i < 3; ++i) x[i] = load_x(i);
#pragma unroll
    for (int i = 0; i < k24Steps * NR; ++i) {
      const int s = i / NR, r = i % NR;
      if (i + 3 < k24Steps * NR) x[(i + 3) % 4] = load_x(i + 3);
      if (r < 6 && s + 1 < k24Steps) w[(s + 1) % 2][r] = load_w(s + 1, r);
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 xi = x[i % 4];
      if (s == k24Steps - 1 && kg == 3) xi = bf16x8{};  // no weight: not even inf * 0
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int m = r - d;
        if (m < 0 || m >= MR) continue;
        acc[m][0] = mfma_bf16(w[s % 2][2 * d], xi, acc[m][0]);
        acc[m][1] = mfma_bf16(w[s % 2][2 * d + 1], xi, acc[m][1]);
      }
    }
    if (!late) activate(blk);
    prev = blk;
  }
  if (late && prev >= 0) activate(prev);
}

// 1 -> 24.  The tile holds, per voxel, its value and the next two along x (and
// a zero) as one 8-byte word: a lane's 8 values of K are two (dz, dy) rows of
// three dx, and the ninth row's values take the free fourth places of the
// first three lane groups, so one step holds all 27 taps (with a second step
// for the ninth row the float32 sums were rounded once more).  Bound by the
// activation and the stores: 8 waves of 8 rows, several work-groups per CU
// (0.69 ms of 264^3 voxels with a 2-byte LDS read per K value and a byte-wise
// store, 0.31 now).
constexpr int k1BZ = 8;

__global__ __launch_bounds__(64 * k1BZ) __attribute__((amdgpu_waves_per_eu(4))) void
k_conv3d_1x24(const ConvArgs a) {
  constexpr int TVOX = (k1BZ + 2) * kTY * kTX;
  __shared__ __align__(16) bf16x4 T[TVOX];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kg = lane >> 4;
  const int OD = a.D - 2, OH = a.H - 2, OW = a.W - 2;
  const bf16x8 w0 = a.wpk[lane], w1 = a.wpk[64 + lane];
  f32x4 bias0, bias1;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    bias0[r] = a.bias[4 * kg + r];
    bias1[r] = a.bias[16 + 4 * (kg & 1) + r];
  }
  // rows 2 kg and 2 kg + 1 of (dz, dy), and dx = kg of row 8 (kg < 3)
  const int g0 = 2 * kg, g1 = 2 * kg + 1;
  const int off0 = (g0 / 3 * kTY + g0 % 3) * kTX, off1 = (g1 / 3 * kTY + g1 % 3) * kTX;
  const int off8 = (2 * kTY + 2) * kTX + (kg < 3 ? kg : 0);
  const int64_t G = gridDim.x;
  for (int64_t blk = xcd_swizzle(blockIdx.x, G); blk < a.nblocks; blk += G) {
    int x0, y0, z0;
    const int64_t n = block_origin<k1BZ>(a, blk, x0, y0, z0);
    __syncthreads();  // the previous block's reads are done
    for (int e = tid; e < TVOX; e += 64 * k1BZ) {
      const int gx = x0 + e % kTX, gy = y0 + e / kTX % kTY, gz = z0 + e / (kTX * kTY);
      bf16x4 v = {};
      if (gy < a.H && gz < a.D) {
        const __bf16* p = a.in + ((n * a.D + gz) * a.H + gy) * a.W + gx;
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (gx + d < a.W) v[d] = p[d];
      }
      T[e] = v;
    }
    __syncthreads();
    const int gz = z0 + wv, gx = x0 + li;
    const int64_t o0 = (((n * OD + gz) * OH + y0) * OW + gx) * kC;
    const bool in = gz < OD && gx < OW;
    const bf16x4* row = T + wv * kTY * kTX + li;
#pragma unroll
    for (int m = 0; m < kBY; m += 2) {
      f32x4 acc[2][2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const bf16x4* p = row + (m + k) * kTX;
        bf16x4 u = p[off0];
        const bf16x4 v = p[off1];
        const __bf16 q = p[off8][0];
        u[3] = kg < 3 ? q : (__bf16)0.0f;  // no weight: not even inf * 0
        const bf16x8 x = __builtin_shufflevector(u, v, 0, 1, 2, 3, 4, 5, 6, 7);
        acc[k][0] = mfma_bf16(w0, x, f32x4{0.f, 0.f, 0.f, 0.f});
        acc[k][1] = mfma_bf16(w1, x, f32x4{0.f, 0.f, 0.f, 0.f});
      }
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (in && y0 + m + k < OH)
          store_gelu4(a, o0 + (int64_t)(m + k) * OW * kC + 4 * kg, acc[k][0] + bias0);
      const f32x4 v = join_halves(acc[0][1], acc[1][1]) + bias1;
      const int k = kg >> 1;
      if (in && y0 + m + k < OH)
        store_gelu4(a, o0 + (int64_t)(m + k) * OW * kC + 16 + 4 * (kg & 1), v);
    }
  }
}

// 24 -> 1.  One output channel would fill one of 16 matrix rows; here M = the
// nine (dz, dy), K = (dx, octet of channels) in three steps, and the products
// P[(dz, dy)][input voxel] are summed over (dz, dy) from LDS: 3 matrix
// instructions per 16 input voxels instead of 21 per 16 outputs.  Inputs are
// read straight from memory, seven rows of a wave at a time.  Bound by reading
// them: 0.88 ms of 258^3 voxels with 21 instructions per 16 outputs, 0.45 with
// three and four rows in flight, 0.35 with seven.
constexpr int k9BZ = 8;

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void
k_conv3d_24x1(const ConvArgs a) {
  constexpr int ROWS = (k9BZ + 2) * kTY;
  __shared__ float P[9 * ROWS * kBX];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kg = lane >> 4;
  const int OD = a.D - 2, OH = a.H - 2, OW = a.W - 2;
  bf16x8 w[3];
  int dx[3], oct[3];
  bool use[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    w[c] = a.wpk[c * 64 + lane];
    const int q = 4 * c + kg;
    use[c] = q < 9;
    dx[c] = use[c] ? q / 3 : 0;
    oct[c] = use[c] ? q % 3 : 0;
  }
  const float bias = a.bias[0];
  const int64_t G = gridDim.x;
  for (int64_t blk = xcd_swizzle(blockIdx.x, G); blk < a.nblocks; blk += G) {
    int x0, y0, z0;
    const int64_t n = block_origin<k9BZ>(a, blk, x0, y0, z0);
    __syncthreads();  // the previous block's reads are done
    // rows past the volume are computed from its last row and never used
    int xo[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) xo[c] = min(x0 + li + dx[c], a.W - 1) * kC + 8 * oct[c];
    constexpr int NB = 7;  // rows of a wave whose loads are issued together
#pragma unroll 1
    for (int r0 = wv; r0 < ROWS; r0 += 8 * NB) {
      bf16x8 x[NB][3];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int r = r0 + 8 * u;
        const int gy = min(y0 + r % kTY, a.H - 1), gz = min(z0 + r / kTY, a.D - 1);
        const __bf16* p = a.in + ((n * a.D + gz) * a.H + gy) * (int64_t)a.W * kC;
#pragma unroll
        for (int c = 0; c < 3; ++c) x[u][c] = *reinterpret_cast<const bf16x8*>(p + xo[c]);
      }
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int r = r0 + 8 * u;
        if (r >= ROWS) break;
        if (!use[2]) x[u][2] = bf16x8{};  // no weight: not even inf * 0
        f32x4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 3; ++c) acc = mfma_bf16(w[c], x[u][c], acc);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (4 * kg + k < 9) P[((4 * kg + k) * ROWS + r) * kBX + li] = acc[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < k9BZ * kBY * kBX / 512; ++u) {
      const int e = tid + 512 * u;
      const int lx = e % kBX, ly = e / kBX % kBY, lz = e / (kBX * kBY);
      float s = 0.f;
#pragma unroll
      for (int g = 0; g < 9; ++g)
        s += P[(g * ROWS + (lz + g / 3) * kTY + ly + g % 3) * kBX + lx];
      s += bias;
      const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
      if (gx < OW && gy < OH && gz < OD) {
        const int64_t o = ((n * OD + gz) * OH + gy) * OW + gx;
        if (a.pre) a.pre[o] = s;
        reinterpret_cast<float*>(a.out)[o] =
            a.act == ACT_CLAMP01 ? fminf(fmaxf(s, 0.f), 1.f) : s;
      }
    }
  }
}

// --------------------------------------------------------------- padding --
// out (D + 2p, H + 2p, W + 2p) bf16 = in (D, H, W) float32 boundary-extended
// One wave per row: the row's source is found once, and only the x index is
// mapped per element.
__global__ __launch_bounds__(256) void k_pad_bf16(const float* __restrict__ in,
                                                  __bf16* __restrict__ out, int D, int H, int W,
                                                  int p, int mode, float cval) {
  const int PD = D + 2 * p, PH = H + 2 * p, PW = W + 2 * p;
  const int64_t nrows = (int64_t)PD * PH;
  const int lane = threadIdx.x & 63;
  for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < nrows;
       row += (int64_t)gridDim.x * 4) {
    const int y = (int)(row % PH), z = (int)(row / PH);
    const int64_t sy = remap(y - p, H, mode), sz = remap(z - p, D, mode);
    const bool row_in = sy >= 0 && sz >= 0;
    const float* src = in + (row_in ? (sz * H + sy) * W : 0);
    __bf16* dst = out + row * PW;
    for (int x = lane; x < PW; x += 64) {
      const int64_t sx = remap(x - p, W, mode);
      dst[x] = f2bf(row_in && sx >= 0 ? src[sx] : cval);
    }
  }
}

// ------------------------------------------------------------- training --
// g (out-shaped, float32) *= gelu'(pre)
__global__ __launch_bounds__(256) void k_gelu_bwd(float* __restrict__ g,
                                                  const float* __restrict__ pre, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256)
    g[i] *= gelu_grad(pre[i]);
}

// Input gradient of a valid 3x3x3 convolution: dx[p][ci] =
// sum_{tap, co} dy[p - off(tap)][co] * w[tap][ci][co] over valid p - off.
// w: float32 [27][CI][CO].
__global__ __launch_bounds__(256) void k_conv3d_dgrad(const float* __restrict__ dy,
                                                      const float* __restrict__ w,
                                                      float* __restrict__ dx, int D, int H,
                                                      int W, int CI, int CO) {
  const int OD = D - 2, OH = H - 2, OW = W - 2;
  const int64_t n = (int64_t)D * H * W * CI;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256) {
    const int ci = (int)(i % CI);
    const int64_t v = i / CI;
    const int x = (int)(v % W), y = (int)((v / W) % H), z = (int)(v / ((int64_t)W * H));
    float s = 0.f;
    for (int dz = 0; dz < 3; ++dz) {
      const int oz = z - dz;
      if (oz < 0 || oz >= OD) continue;
      for (int dyy = 0; dyy < 3; ++dyy) {
        const int oy = y - dyy;
        if (oy < 0 || oy >= OH) continue;
        for (int dxx = 0; dxx < 3; ++dxx) {
          const int ox = x - dxx;
          if (ox < 0 || ox >= OW) continue;
          const int tap = (dz * 3 + dyy) * 3 + dxx;
          const float* g = dy + (((int64_t)oz * OH + oy) * OW + ox) * CO;
          const float* wr = w + ((int64_t)tap * CI + ci) * CO;
          for (int co = 0; co < CO; ++co) s = fmaf(g[co], wr[co], s);
        }
      }
    }
    dx[i] = s;
  }
}

// Weight gradient: dw[tap][ci][co] += sum_p x[p + off(tap)][ci] * dy[p][co],
// one work-group per slab of output voxels; db[co] += sum_p dy[p][co].
// x: bf16 activations (the forward input), dy: float32.
__global__ __launch_bounds__(256) void k_conv3d_wgrad(const __bf16* __restrict__ x,
                                                      const float* __restrict__ dy,
                                                      float* __restrict__ dw,
                                                      float* __restrict__ db, int D, int H,
                                                      int W, int CI, int CO, int64_t per_block) {
  const int OD = D - 2, OH = H - 2, OW = W - 2;
  const int64_t nvox = (int64_t)OD * OH * OW;
  const int64_t v0 = (int64_t)blockIdx.x * per_block;
  const int64_t v1 = v0 + per_block < nvox ? v0 + per_block : nvox;
  const int nw = 27 * CI * CO;
  for (int j = threadIdx.x; j < nw + CO; j += 256) {
    float s = 0.f;
    if (j < nw) {
      const int co = j % CO, ci = (j / CO) % CI, tap = j / (CO * CI);
      const int dz = tap / 9, dyy = (tap / 3) % 3, dxx = tap % 3;
      for (int64_t v = v0; v < v1; ++v) {
        const int ox = (int)(v % OW), oy = (int)((v / OW) % OH),
                  oz = (int)(v / ((int64_t)OW * OH));
        const float xv =
            bf2f(x[(((int64_t)(oz + dz) * H + (oy + dyy)) * W + (ox + dxx)) * CI + ci]);
        s = fmaf(xv, dy[v * CO + co], s);
      }
      atomicAdd(dw + j, s);
    } else {
      const int co = j - nw;
      for (int64_t v = v0; v < v1; ++v) s += dy[v * CO + co];
      atomicAdd(db + co, s);
    }
  }
}

// MSE gradient over the interior: g = 2 (y - t) / count where mask, else 0;
// loss partial sums atomically added to *loss.
__global__ __launch_bounds__(256) void k_mse_grad(const float* __restrict__ y,
                                                  const float* __restrict__ t,
                                                  float* __restrict__ g, int64_t n, float inv_n,
                                                  float* __restrict__ loss) {
  __shared__ float red[256];
  float s = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256) {
    const float d = y[i] - t[i];
    g[i] = 2.f * d * inv_n;
    s += d * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0] * inv_n);
}

// Adam on float32 master weights.
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v,
                                              int64_t n, float lr, float b1, float b2, float eps,
                                              float c1, float c2) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// Pack float32 weights [27][CI][CO] into the bf16 A operands (16 channels or
// rows x 8 K values per lane) of the kernel of their shape; other shapes, for
// which no kernel is compiled, in (tap, channel) order.
__global__ __launch_bounds__(256) void k_pack_weights(const float* __restrict__ w,
                                                      bf16x8* __restrict__ pk, int CI, int CO,
                                                      int n) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int lane = i % 64, row = lane & 15, kg = lane >> 4;
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      int tap = -1, ci = 0, co = 0;
      if (CI == 24 && CO == 24) {  // [step][dy][tile][lane]
        const int t = i / 64 % 2, dy = i / 128 % 3, q = 4 * (i / 384) + kg;
        if (q < 27) tap = q / 9 * 9 + dy * 3 + q / 3 % 3;
        ci = q % 3 * 8 + j;
        co = 16 * t + row;
      } else if (CI == 1 && CO == 24) {  // [tile][lane]
        if (j % 4 < 3)
          tap = (2 * kg + j / 4) * 3 + j % 4;
        else if (j == 3 && kg < 3)
          tap = 24 + kg;
        co = 16 * (i / 64) + row;
      } else if (CI == 24 && CO == 1) {  // [step][lane], row = (dz, dy)
        const int q = 4 * (i / 64) + kg;
        if (q < 9 && row < 9) tap = row * 3 + q / 3;
        ci = q % 3 * 8 + j;
      } else {
        const int NT = (CO + 15) / 16, k = 32 * (i / (64 * NT)) + 8 * kg + j;
        if (k < 27 * CI) tap = k / CI;
        ci = k % CI;
        co = 16 * (i / 64 % NT) + row;
      }
      float f = 0.f;
      if (tap >= 0 && co < CO) f = w[((int64_t)tap * CI + ci) * CO + co];
      v[j] = f2bf(f);
    }
    pk[i] = v;
  }
}

namespace {

int64_t grid_of(int64_t n) { return n <= 0 ? 1 : std::min<int64_t>((n + 255) / 256, 256 * 64); }

int conv_blocks(ConvArgs* a, int64_t batch, int bz) {
  a->nbx = (a->W - 2 + kBX - 1) / kBX;
  a->nby = (a->H - 2 + kBY - 1) / kBY;
  a->nbz = (a->D - 2 + bz - 1) / bz;
  a->nblocks = batch * a->nbx * a->nby * a->nbz;
  if (a->nblocks > 0x7fffffff) return fail(HC_ERR_VALUE, "volume too large");
  return HC_OK;
}

template <int BZ>
int launch_24x24(ConvArgs a, int64_t batch, hipStream_t st) {
  const int rc = conv_blocks(&a, batch, BZ);
  if (rc != HC_OK) return rc;
  // weights, then the input tile
  const int smem = k24Steps * 6 * 64 * 16 + (BZ + 2) * kTY * kTX * kC * 2;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)k_conv3d_24x24<BZ>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (e != hipSuccess) return hip_check(e, "hipFuncSetAttribute(k_conv3d_24x24)");
  // persistent: one work-group per CU (95 or 129 KB of LDS)
  const int grid = (int)std::min<int64_t>(a.nblocks, 256);
  HC_LAUNCH("k_conv3d_24x24", st, k_conv3d_24x24<BZ>, dim3(grid), dim3(512), smem, a);
  return HC_OK;
}

int conv_24x24(const ConvArgs& a, int64_t batch, hipStream_t st) {
  // Blocks of 8 planes read less halo and fewer LDS words per product; blocks
  // of 4 are half the work and divide better over 256 CUs where there are few.
  // By rounds of work-groups, one layer with 8 against 4 planes (us): 64 / 128
  // (258^3) 652 / 681, 16 / 32 (162^3) 160 / 166, 1 / 2 (58^3) 14.9 / 16.4; 12 /
  // 23 (146^3) 124.9 / 123.1, 6 / 11 (114^3) 64.7 / 62.1, 4 / 7 (98^3) 47.0 /
  // 42.7, 1 / 1 (22^3) 12.9 / 8.7.
  ConvArgs b = a;
  int rc = conv_blocks(&b, batch, 8);
  if (rc != HC_OK) return rc;
  const int64_t n8 = (b.nblocks + 255) / 256;
  rc = conv_blocks(&b, batch, 4);
  if (rc != HC_OK) return rc;
  const int64_t n4 = (b.nblocks + 255) / 256;
  return 25 * n8 <= 13 * n4 ? launch_24x24<8>(a, batch, st) : launch_24x24<4>(a, batch, st);
}

}  // namespace
}  // namespace hc

using namespace hc;

extern "C" {

int hc_cnn3d_packed_size(int ci, int co) {
  if (ci < 1 || co < 1) return -1;
  if (ci == 24 && co == 24) return k24Steps * 6 * 64 * 16;
  if (ci == 1 && co == 24) return 2 * 64 * 16;
  if (ci == 24 && co == 1) return 3 * 64 * 16;
  return ((27 * ci + 31) / 32) * ((co + 15) / 16) * 64 * 16;
}

int hc_cnn3d_pack(const float* w_dev, void* packed_dev, int ci, int co, void* stream) {
  if (!w_dev || !packed_dev) return fail(HC_ERR_VALUE, "null argument");
  if (ci < 1 || co < 1) return fail(HC_ERR_VALUE, "channel counts must be positive");
  const int n = hc_cnn3d_packed_size(ci, co) / 16;
  hipStream_t st = (hipStream_t)stream;
  HC_LAUNCH("k_pack_weights", st, k_pack_weights, dim3((unsigned)grid_of(n)), dim3(256), 0, w_dev,
            (bf16x8*)packed_dev, ci, co, n);
  return HC_OK;
}

int hc_cnn3d_conv(const hc_array* in, const hc_array* out, const void* packed,
                  const float* bias_dev, int act, float* pre_dev, void* stream) {
  if (!in || !out || !packed || !bias_dev) return fail(HC_ERR_VALUE, "null argument");
  if (in->dtype != HC_BFLOAT16 || (in->ndim != 4 && in->ndim != 5) || !is_c_contiguous(in))
    return fail(HC_ERR_VALUE, "input must be a C-contiguous ([B,] D, H, W, C) bfloat16 array");
  if (out->ndim != in->ndim || !is_c_contiguous(out))
    return fail(HC_ERR_VALUE, "output must be a C-contiguous ([B,] D-2, H-2, W-2, C) array");
  const int d0 = in->ndim - 4;  // a leading batch dimension
  const int64_t batch = d0 ? in->shape[0] : 1;
  if (d0 && out->shape[0] != batch) return fail(HC_ERR_VALUE, "batch sizes differ");
  if (batch == 0) return HC_OK;
  const int ci = (int)in->shape[d0 + 3], co = (int)out->shape[d0 + 3];
  for (int d = d0; d < d0 + 3; ++d)
    if (out->shape[d] != in->shape[d] - 2 || in->shape[d] < 3)
      return fail(HC_ERR_VALUE, "valid convolution: output extents are input extents - 2");
  if (((uintptr_t)in->data | (uintptr_t)packed) % 16)
    return fail(HC_ERR_VALUE, "input and packed weights must be 16-byte aligned");
  ConvArgs a;
  std::memset(&a, 0, sizeof(a));
  a.in = (const __bf16*)in->data;
  a.out = out->data;
  a.pre = pre_dev;
  a.wpk = (const bf16x8*)packed;
  a.bias = bias_dev;
  a.D = (int)in->shape[d0];
  a.H = (int)in->shape[d0 + 1];
  a.W = (int)in->shape[d0 + 2];
  hipStream_t st = (hipStream_t)stream;
  const bool f32 = out->dtype == HC_FLOAT32;
  if (!f32 && out->dtype != HC_BFLOAT16) return fail(HC_ERR_VALUE, "output must be bf16 or f32");
  if (ci == 24 && co == 24 && act == ACT_GELU && !f32) return conv_24x24(a, batch, st);
  if (ci == 1 && co == 24 && act == ACT_GELU && !f32) {
    const int rc = conv_blocks(&a, batch, k1BZ);
    if (rc != HC_OK) return rc;
    const int grid = (int)std::min<int64_t>(a.nblocks, 256 * 8);
    HC_LAUNCH("k_conv3d_1x24", st, k_conv3d_1x24, dim3(grid), dim3(64 * k1BZ), 0, a);
    return HC_OK;
  }
  if (ci == 24 && co == 1 && (act == ACT_CLAMP01 || act == ACT_NONE) && f32) {
    const int rc = conv_blocks(&a, batch, k9BZ);
    if (rc != HC_OK) return rc;
    a.act = act;
    const int grid = (int)std::min<int64_t>(a.nblocks, 256 * 8);
    HC_LAUNCH("k_conv3d_24x1", st, k_conv3d_24x1, dim3(grid), dim3(512), 0, a);
    return HC_OK;
  }
  return fail(HC_ERR_UNSUPPORTED, "layer shape / activation not compiled");
}

int hc_cnn3d_pad(const hc_array* in, const hc_array* out, int pad, int mode, double cval,
                 void* stream) {
  if (!in || !out) return fail(HC_ERR_VALUE, "null argument");
  if (in->dtype != HC_FLOAT32 || in->ndim != 3 || !is_c_contiguous(in))
    return fail(HC_ERR_VALUE, "input must be a C-contiguous 3-D float32 array");
  if (out->dtype != HC_BFLOAT16 || !is_c_contiguous(out) || out->ndim < 3)
    return fail(HC_ERR_VALUE, "output must be a C-contiguous bfloat16 array");
  for (int d = 0; d < 3; ++d)
    if (out->shape[d] != in->shape[d] + 2 * pad)
      return fail(HC_ERR_VALUE, "output extents must be input + 2 pad");
  if (out->ndim == 4 && out->shape[3] != 1) return fail(HC_ERR_VALUE, "one channel expected");
  const int64_t n = numel(out);
  if (n == 0) return HC_OK;
  hipStream_t st = (hipStream_t)stream;
  const int64_t rows = n / (in->shape[2] + 2 * pad);
  HC_LAUNCH("k_pad_bf16", st, k_pad_bf16,
            dim3((unsigned)std::min<int64_t>((rows + 3) / 4, 256 * 32)), dim3(256), 0,
            (const float*)in->data, (__bf16*)out->data, (int)in->shape[0], (int)in->shape[1],
            (int)in->shape[2], pad, mode, (float)cval);
  return HC_OK;
}

int hc_cnn3d_gelu_bwd(float* g, const float* pre, int64_t n, void* stream) {
  if (!g || !pre || n < 0) return fail(HC_ERR_VALUE, "bad argument");
  if (n == 0) return HC_OK;
  hipStream_t st = (hipStream_t)stream;
  HC_LAUNCH("k_gelu_bwd", st, k_gelu_bwd, dim3((unsigned)grid_of(n)), dim3(256), 0, g, pre, n);
  return HC_OK;
}

int hc_cnn3d_dgrad(const float* dy, const float* w, float* dx, int D, int H, int W, int ci,
                   int co, void* stream) {
  if (!dy || !w || !dx || D < 3 || H < 3 || W < 3 || ci < 1 || co < 1)
    return fail(HC_ERR_VALUE, "bad argument");
  const int64_t n = (int64_t)D * H * W * ci;
  hipStream_t st = (hipStream_t)stream;
  HC_LAUNCH("k_conv3d_dgrad", st, k_conv3d_dgrad, dim3((unsigned)grid_of(n)), dim3(256), 0, dy,
            w, dx, D, H, W, ci, co);
  return HC_OK;
}

int hc_cnn3d_wgrad(const void* x_bf16, const float* dy, float* dw, float* db, int D, int H,
                   int W, int ci, int co, void* stream) {
  if (!x_bf16 || !dy || !dw || !db || D < 3 || H < 3 || W < 3 || ci < 1 || co < 1)
    return fail(HC_ERR_VALUE, "bad argument");
  const int64_t nvox = (int64_t)(D - 2) * (H - 2) * (W - 2);
  const int64_t blocks = std::min<int64_t>(nvox, 2048);
  const int64_t per = (nvox + blocks - 1) / blocks;
  hipStream_t st = (hipStream_t)stream;
  HC_LAUNCH("k_conv3d_wgrad", st, k_conv3d_wgrad, dim3((unsigned)blocks), dim3(256), 0,
            (const __bf16*)x_bf16, dy, dw, db, D, H, W, ci, co, per);
  return HC_OK;
}

int hc_cnn3d_mse_grad_batch(const float* y, const float* t, float* g, int64_t n, int64_t batch,
                            float* loss, void* stream) {
  if (!y || !t || !g || !loss || n <= 0 || batch <= 0) return fail(HC_ERR_VALUE, "bad argument");
  hipStream_t st = (hipStream_t)stream;
  const int64_t total = n * batch;
  HC_LAUNCH("k_mse_grad", st, k_mse_grad,
            dim3((unsigned)std::min<int64_t>(grid_of(total), 1024)), dim3(256), 0, y, t, g, total,
            1.0f / (float)n, loss);
  return HC_OK;
}

int hc_cnn3d_mse_grad(const float* y, const float* t, float* g, int64_t n, float* loss,
                      void* stream) {
  return hc_cnn3d_mse_grad_batch(y, t, g, n, 1, loss, stream);
}

int hc_cnn3d_adam(float* p, const float* g, float* m, float* v, int64_t n, double lr,
                  double b1, double b2, double eps, int step, void* stream) {
  if (!p || !g || !m || !v || n < 0 || step < 1) return fail(HC_ERR_VALUE, "bad argument");
  if (n == 0) return HC_OK;
  const float c1 = (float)(1.0 - std::pow(b1, step)), c2 = (float)(1.0 - std::pow(b2, step));
  hipStream_t st = (hipStream_t)stream;
  HC_LAUNCH("k_adam", st, k_adam, dim3((unsigned)grid_of(n)), dim3(256), 0, p, g, m, v, n,
            (float)lr, (float)b1, (float)b2, (float)eps, c1, c2);
  return HC_OK;
}

}  // extern "C"
