// Backward kernels of the surrogate network's layers on the float32 matrix
// cores (gfx950), over a batch of equally sized patches: activations
// (B, D, H, W, C) bfloat16, gradients (B, D-2, H-2, W-2, C) float32.
//
// v_mfma_f32_16x16x4f32: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and
// D[4 (l / 16) + r][l % 16].  Every sum over voxels or channels is a float32
// sum of exact products of float32 values (a bfloat16 activation widens
// exactly), as in the per-output kernels these replace; only the order of the
// terms differs.  No operand that pads a block is multiplied by one that may be
// infinite or NaN: sums hold their own terms only, with such values too.
//
// One training step of eight 64^3 patches took 269 ms with one work-item per
// output and one launch per patch (weight gradients 40 launches of 3.4 ms,
// each with an atomic add per weight and work-group; input gradients 32 of
// 4.1 ms); it takes 5.8 ms with these (24 -> 24 layers: three launches of
// 0.76 ms and three of 0.87 ms for all patches, the matrix cores busy for 71
// and 63 % of them, on 24 of 32 rows or columns).
#include <algorithm>
#include <cstring>

#include "hc_cnn.h"

namespace hc {

namespace {

constexpr int kC = 24;                     // channels of a hidden layer
constexpr int kBZ = 2, kBY = 8, kBX = 16;  // voxels of one block
constexpr int kTZ = kBZ + 2, kTY = kBY + 2, kTX = kBX + 2;  // with halo
constexpr int kTV = kTZ * kTY * kTX;                        // 720
constexpr int kBV = kBZ * kBY * kBX;                        // 256

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct BwdArgs {
  const __bf16* x;   // layer input (B, D, H, W, ci)
  const float* dy;   // gradient of the layer's output (B, D-2, H-2, W-2, co)
  const float* w;    // float32 weights [27][ci][co]
  const float* pre;  // pre-activation of the layer before (dx's shape), or null
  float* out;        // dx, or the weight gradient's partial sums
  int D, H, W;       // extents of x
  int nbx, nby, nbz;  // blocks per patch
  int64_t nblocks;    // of the batch
};

struct Origin {
  int x, y, z;
  int64_t n;  // patch
};

// Block b (fewer than 2^31) -> its first voxel and patch.
__device__ __forceinline__ Origin origin_of(const BwdArgs& a, int64_t b) {
  Origin o;
  unsigned q = (unsigned)b;
  unsigned r = q / (unsigned)a.nbx;
  o.x = (int)(q - r * a.nbx) * kBX;
  q = r / (unsigned)a.nby;
  o.y = (int)(r - q * a.nby) * kBY;
  r = q / (unsigned)a.nbz;
  o.z = (int)(q - r * a.nbz) * kBZ;
  o.n = r;
  return o;
}

}  // namespace

// ------------------------------------------------------ weight gradient --
// dw[tap][ci][co] = sum_p x[p + off(tap)][ci] dy[p][co], db[co] = sum_p dy[p][co]:
// a product with M = co (24 of 32 rows), N = the flattened (tap, ci) and one
// column of ones for db (649 of 656 columns), K = the voxels, four along x
// per instruction.  Both operands are read from LDS in their own channels-last
// order.  The 41 column tiles are dealt to the four waves; a persistent
// work-group keeps its whole 24 x 649 sum in accumulators over all its blocks
// (88 registers per lane) and writes it once; k_sum_parts adds the
// work-groups' sums in a fixed order.  Bound by the matrix cores: 22
// instructions of 32 cycles per wave for 2 + 11 LDS words per lane.
constexpr int kWgT = 11;                  // column tiles per wave
constexpr int kWgN = 27 * kC + 1;         // columns: weights per output channel, ones
constexpr int kWgPart = kWgN * kC;        // floats of one partial sum

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
k_conv3d_wgrad_mfma(const BwdArgs a) {
  __shared__ __align__(16) __bf16 X[kTV * kC];
  __shared__ __align__(16) float G[kBV * kC + 8];  // + 8: row tile 1 reads to channel 31
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kg = lane >> 4;
  const int OD = a.D - 2, OH = a.H - 2, OW = a.W - 2;
  constexpr int NX = (kTV * 3 + 255) / 256, NG = kBV * 6 / 256;
  bf16x8 px[NX];
  f32x4 pg[NG];
  auto fetch = [&](int64_t b) {
    const Origin o = origin_of(a, b);
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + 256 * u;
      const int v = e % 3, vox = e / 3;
      const int gx = o.x + vox % kTX, gy = o.y + vox / kTX % kTY, gz = o.z + vox / (kTX * kTY);
      bf16x8 val = {};
      if (e < kTV * 3 && gx < a.W && gy < a.H && gz < a.D)
        val = reinterpret_cast<const bf16x8*>(
            a.x + (((o.n * a.D + gz) * a.H + gy) * a.W + gx) * kC)[v];
      px[u] = val;
    }
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int e = tid + 256 * u;
      const int v = e % 6, vox = e / 6;
      const int gx = o.x + vox % kBX, gy = o.y + vox / kBX % kBY, gz = o.z + vox / (kBX * kBY);
      f32x4 val = {};
      if (gx < OW && gy < OH && gz < OD)
        val = reinterpret_cast<const f32x4*>(
            a.dy + (((o.n * OD + gz) * OH + gy) * OW + gx) * kC)[v];
      pg[u] = val;
    }
  };
  int toff[kWgT];  // element offset of the column's (tap, ci) in the tile
  bool one = false;
#pragma unroll
  for (int j = 0; j < kWgT; ++j) {
    const int n = 16 * (wv + 4 * j) + li;
    const int tap = n / kC, ci = n - tap * kC;
    toff[j] = n < 27 * kC ? ((tap / 9 * kTY + tap / 3 % 3) * kTX + tap % 3) * kC + ci : 0;
    if (n == 27 * kC) one = true;  // only in the last tile
  }
  f32x4 acc[2][kWgT];
#pragma unroll
  for (int j = 0; j < kWgT; ++j) acc[0][j] = acc[1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (tid < 8) G[kBV * kC + tid] = 0.f;
  const int64_t NB = gridDim.x;
  int64_t blk = xcd_swizzle(blockIdx.x, NB);
  if (blk < a.nblocks) fetch(blk);
  for (; blk < a.nblocks; blk += NB) {  // uniform per work-group
    __syncthreads();  // the previous block's reads are done
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int e = tid + 256 * u;
      if (e < kTV * 3) reinterpret_cast<bf16x8*>(X)[e] = px[u];
    }
#pragma unroll
    for (int u = 0; u < NG; ++u) reinterpret_cast<f32x4*>(G)[tid + 256 * u] = pg[u];
    if (blk + NB < a.nblocks) fetch(blk + NB);  // in flight during the products
    __syncthreads();
    // outputs past the patch take no part: their rows and steps are left out,
    // and in a row's last step the activations next to them are zeroed (only
    // the gradient's tile is padded; 0 * inf would spoil a sum)
    const Origin o = origin_of(a, blk);
    const int nz = min(kBZ, OD - o.z), ny = min(kBY, OH - o.y), nx = min(kBX, OW - o.x);
#pragma unroll 1
    for (int r = 0; r < nz * kBY; ++r) {
      const int z = r / kBY, y = r - z * kBY;
      if (y >= ny) continue;
      const __bf16* xr = X + ((z * kTY + y) * kTX + kg) * kC;
      const float* gr = G + (r * kBX + kg) * kC + li;
      auto step = [&](int s, bool in) {
        const float a0 = gr[4 * s * kC], a1 = gr[4 * s * kC + 16];
        float b[kWgT];
#pragma unroll
        for (int j = 0; j < kWgT; ++j) b[j] = in ? bf2f(xr[toff[j] + 4 * s * kC]) : 0.f;
        if (one) b[kWgT - 1] = 1.f;
#pragma unroll
        for (int j = 0; j < kWgT; ++j) {
          acc[0][j] = mfma_f32(a0, b[j], acc[0][j]);
          acc[1][j] = mfma_f32(a1, b[j], acc[1][j]);
        }
      };
#pragma unroll 2
      for (int s = 0; s < nx / 4; ++s) step(s, true);
      if (nx % 4) step(nx / 4, kg < nx % 4);
    }
  }
  // rows 4 kg + r (+ 16), column 16 tile + li -> part[column][channel]
  float* P = a.out + (int64_t)blockIdx.x * kWgPart;
#pragma unroll
  for (int j = 0; j < kWgT; ++j) {
    const int n = 16 * (wv + 4 * j) + li;
    if (n >= kWgN) continue;
    *reinterpret_cast<f32x4*>(P + n * kC + 4 * kg) = acc[0][j];
    if (kg < 2) *reinterpret_cast<f32x4*>(P + n * kC + 16 + 4 * kg) = acc[1][j];
  }
}

// The same for the layers with one channel on one side: F the 24-channel
// field, S the other, K = the positions of F.
//   FIRST (1 -> 24): dw[tap][co] = sum_p S[p + off(tap)] F[p][co], F = dy, S = x
//   else (24 -> 1):  dw[tap][ci] = sum_p F[p][ci] S[p - off(tap)], F = x, S = dy
// M = the 24 channels (and, for 24 -> 1, a row of ones: its product with tap 0
// is the sum of dy), N = the 27 taps (and, for 1 -> 24, a column of ones).
// F is read straight from memory (each wave 4 rows of 16 voxels), S from LDS;
// bound by reading F.  Where F is padded (1 -> 24), S is zeroed beside it; where
// S is (24 -> 1, outputs off the patch), which positions are depends on the
// tap, so a wave with an infinite or NaN activation takes its products tap by
// tap with both operands zeroed.
template <bool FIRST>
__global__ __launch_bounds__(256) void k_conv3d_wgrad_1c(const BwdArgs a) {
  __shared__ float S[kTV];
  __shared__ float R[4][32 * 33];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kg = lane >> 4;
  const int OD = a.D - 2, OH = a.H - 2, OW = a.W - 2;
  const int FD = FIRST ? OD : a.D, FH = FIRST ? OH : a.H, FW = FIRST ? OW : a.W;
  int toff[2];
  bool colone = false;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tap = 16 * j + li;
    int dz = tap / 9, dy = tap / 3 % 3, dx = tap % 3;
    if (!FIRST) dz = 2 - dz, dy = 2 - dy, dx = 2 - dx;
    toff[j] = tap < 27 ? (dz * kTY + dy) * kTX + dx : 0;
    if (FIRST && tap == 27) colone = true;
  }
  const bool rowone = !FIRST && li == 8;  // row 24
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int64_t blk = xcd_swizzle(blockIdx.x, gridDim.x); blk < a.nblocks; blk += gridDim.x) {
    const Origin o = origin_of(a, blk);
    // this wave's F values: 4 rows x 4 steps x 2 channel tiles
    float f0[16], f1[16];
    unsigned fin = 0;   // bit u: step u's position is in F
    float chk = 0.f;    // stays 0 while every value is finite
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int r = 4 * wv + u / 4, z = o.z + r / kBY, y = o.y + r % kBY;
      const int x = o.x + 4 * (u % 4) + kg;
      const bool in = z < FD && y < FH && x < FW;
      const int64_t v = ((o.n * FD + z) * FH + y) * FW + x;
      f0[u] = f1[u] = 0.f;
      fin |= (unsigned)in << u;
      if (in) {
        if (FIRST) {
          f0[u] = a.dy[v * kC + li];
          if (li < 8) f1[u] = a.dy[v * kC + 16 + li];
        } else {
          f0[u] = bf2f(a.x[v * kC + li]);
          if (li < 8) f1[u] = bf2f(a.x[v * kC + 16 + li]);
        }
      }
      if (!FIRST) chk = fmaf(f1[u], 0.f, fmaf(f0[u], 0.f, chk));
      if (rowone) f1[u] = 1.f;
    }
    __syncthreads();
    for (int e = tid; e < kTV; e += 256) {
      int x = o.x + e % kTX, y = o.y + e / kTX % kTY, z = o.z + e / (kTX * kTY);
      float v = 0.f;
      if (FIRST) {
        if (x < a.W && y < a.H && z < a.D) v = bf2f(a.x[((o.n * a.D + z) * a.H + y) * a.W + x]);
      } else {
        x -= 2, y -= 2, z -= 2;
        if (x >= 0 && y >= 0 && z >= 0 && x < OW && y < OH && z < OD)
          v = a.dy[((o.n * OD + z) * OH + y) * OW + x];
      }
      S[e] = v;
    }
    __syncthreads();
    if (!FIRST && __any(!(chk == 0.f))) {
#pragma unroll 1
      for (int tap = 0; tap < 27; ++tap) {
        const int dz = tap / 9, dy = tap / 3 % 3, dx = tap % 3;
        const int off = ((2 - dz) * kTY + 2 - dy) * kTX + 2 - dx;
        f32x4 t0{0.f, 0.f, 0.f, 0.f}, t1 = t0;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int r = 4 * wv + u / 4;
          const int z = o.z + r / kBY - dz, y = o.y + r % kBY - dy;
          const int x = o.x + 4 * (u % 4) + kg - dx;
          const bool in = z >= 0 && y >= 0 && x >= 0 && z < OD && y < OH && x < OW;
          const float b =
              in ? S[(r / kBY * kTY + r % kBY) * kTX + 4 * (u % 4) + kg + off] : 0.f;
          t0 = mfma_f32(in ? f0[u] : 0.f, b, t0);
          t1 = mfma_f32(in ? f1[u] : 0.f, b, t1);
        }
        if (li == tap % 16) {
          if (tap < 16)
            acc[0][0] += t0, acc[1][0] += t1;
          else
            acc[0][1] += t0, acc[1][1] += t1;
        }
      }
      continue;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int r = 4 * wv + u / 4;
      const float* s = S + (r / kBY * kTY + r % kBY) * kTX + 4 * (u % 4) + kg;
      const bool in = !FIRST || (fin >> u & 1);
      const float b0 = in ? s[toff[0]] : 0.f, b1 = colone ? 1.f : in ? s[toff[1]] : 0.f;
      acc[0][0] = mfma_f32(f0[u], b0, acc[0][0]);
      acc[0][1] = mfma_f32(f0[u], b1, acc[0][1]);
      acc[1][0] = mfma_f32(f1[u], b0, acc[1][0]);
      acc[1][1] = mfma_f32(f1[u], b1, acc[1][1]);
    }
  }
  // R[column][row] of every wave, summed in wave order
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        R[wv][(16 * j + li) * 33 + 16 * i + 4 * kg + r] = acc[i][j][r];
  __syncthreads();
  constexpr int NP = 27 * kC + (FIRST ? kC : 1);
  float* P = a.out + (int64_t)blockIdx.x * NP;
  for (int e = tid; e < NP; e += 256) {
    const int q = FIRST || e < 27 * kC ? e / kC * 33 + e % kC : 24;
    P[e] = (R[0][q] + R[1][q]) + (R[2][q] + R[3][q]);
  }
}

// dw[j] += sum_p part[p][j] (j < nw), db[j - nw] likewise: 64 columns per
// work-group, 16 rows at a time, then a tree over the 16 sums.
__global__ __launch_bounds__(1024) void k_sum_parts(const float* __restrict__ part, int nparts,
                                                    int n, int nw, float* __restrict__ dw,
                                                    float* __restrict__ db) {
  __shared__ float red[16][64];
  const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int j = blockIdx.x * 64 + c;
  float s = 0.f;
  if (j < n) {
#pragma unroll 8
    for (int p = g; p < nparts; p += 16) s += part[(int64_t)p * n + j];
  }
  red[g][c] = s;
  __syncthreads();
  for (int k = 8; k > 0; k >>= 1) {
    if (g < k) red[g][c] += red[g + k][c];
    __syncthreads();
  }
  if (g == 0 && j < n) {
    if (j < nw)
      dw[j] += red[0][c];
    else
      db[j - nw] += red[0][c];
  }
}

// ------------------------------------------------------- input gradient --
// dx[p][ci] = sum_{tap, co} dy[p - off(tap)][co] w[tap][ci][co], times
// gelu'(pre[p][ci]) when pre is given (the layer before's activation): M = 16
// voxels along x, N = ci (24 of 32 columns), K = 27 taps x 24 channels.  Eight
// waves, two rows of 16 voxels each; the gradient's tile with halo (zero
// outside the patch) and all the weights are in LDS.  A lane's K group kg
// holds channels 6 kg .. 6 kg + 5, so a tap's six instructions read three
// 8-byte words per operand row; rows are 26 words apart, which spreads them
// over the banks (24 would put every eighth row on the same ones).  Bound by
// the matrix cores: 24 instructions of 32 cycles per wave and tap for 12
// 8-byte words.  An infinite or NaN weight (times the zeros around the
// gradient) sends a work-group to sums over its own terms, one per work-item.
constexpr int kDgS = 26;
constexpr int kDgLds = (kTV + 27 * kC) * kDgS * 4;

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void
k_conv3d_dgrad_mfma(const BwdArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* G = reinterpret_cast<float*>(smem);  // [kTV][26]
  float* Wl = G + kTV * kDgS;                 // [27 * 24][26]
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kg = lane >> 4;
  const int OD = a.D - 2, OH = a.H - 2, OW = a.W - 2;
  auto put = [&](float* row, int v, f32x4 x) {
    *reinterpret_cast<f32x2*>(row + 4 * v) = f32x2{x[0], x[1]};
    *reinterpret_cast<f32x2*>(row + 4 * v + 2) = f32x2{x[2], x[3]};
  };
  float chk = 0.f;  // stays 0 while every weight is finite
  for (int e = tid; e < 27 * kC * 6; e += 512) {
    const f32x4 w = reinterpret_cast<const f32x4*>(a.w)[e];
    chk = fmaf(w[3], 0.f, fmaf(w[2], 0.f, fmaf(w[1], 0.f, fmaf(w[0], 0.f, chk))));
    put(Wl + e / 6 * kDgS, e % 6, w);
  }
  const bool wbad = __syncthreads_or(!(chk == 0.f));
  constexpr int NG = (kTV * 6 + 511) / 512;
  f32x4 pg[NG];
  auto fetch = [&](int64_t b) {
    const Origin o = origin_of(a, b);
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int e = tid + 512 * u;
      const int v = e % 6, vox = e / 6;
      const int gx = o.x + vox % kTX - 2, gy = o.y + vox / kTX % kTY - 2,
                gz = o.z + vox / (kTX * kTY) - 2;
      f32x4 val = {};
      if (e < kTV * 6 && gx >= 0 && gy >= 0 && gz >= 0 && gx < OW && gy < OH && gz < OD)
        val = reinterpret_cast<const f32x4*>(
            a.dy + (((o.n * OD + gz) * OH + gy) * OW + gx) * kC)[v];
      pg[u] = val;
    }
  };
  const int64_t NB = gridDim.x;
  int64_t blk = xcd_swizzle(blockIdx.x, NB);
  if (blk < a.nblocks) fetch(blk);
  const int z = wv >> 2, y0 = (wv & 3) * 2;  // this wave's rows
  // column tile 1 holds ci = 16 .. 23 only; its other lanes' results are unused
  const float* w0 = Wl + li * kDgS + 6 * kg;
  const float* w1 = Wl + (16 + (li & 7)) * kDgS + 6 * kg;
  for (; blk < a.nblocks; blk += NB) {  // uniform per work-group
    const Origin o = origin_of(a, blk);
    __syncthreads();  // the previous block's reads are done
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int e = tid + 512 * u;
      if (e < kTV * 6) put(G + e / 6 * kDgS, e % 6, pg[u]);
    }
    if (blk + NB < a.nblocks) fetch(blk + NB);  // in flight during the products
    __syncthreads();
    if (wbad) {  // uniform
#pragma unroll 1
      for (int e = tid; e < kBV * kC; e += 512) {
        const int ci = e % kC, v = e / kC;
        const int lx = v % kBX, ly = v / kBX % kBY, lz = v / (kBX * kBY);
        const int gx = o.x + lx, gy = o.y + ly, gz = o.z + lz;
        if (gx >= a.W || gy >= a.H || gz >= a.D) continue;
        float s = 0.f;
#pragma unroll 1
        for (int tap = 0; tap < 27; ++tap) {
          const int dz = tap / 9, dy = tap / 3 % 3, dx = tap % 3;
          if (gz < dz || gy < dy || gx < dx || gz - dz >= OD || gy - dy >= OH || gx - dx >= OW)
            continue;
          const float* g = G + (((lz + 2 - dz) * kTY + ly + 2 - dy) * kTX + lx + 2 - dx) * kDgS;
          for (int c = 0; c < kC; ++c) s = fmaf(g[c], Wl[(tap * kC + ci) * kDgS + c], s);
        }
        const int64_t q = (((o.n * a.D + gz) * a.H + gy) * a.W + gx) * kC + ci;
        a.out[q] = a.pre ? s * gelu_grad(a.pre[q]) : s;
      }
      continue;
    }
    f32x4 acc[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m) acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 3
    for (int tap = 0; tap < 27; ++tap) {
      const int dz = tap / 9, dy = tap / 3 % 3, dx = tap % 3;
      const float* g = G + (((z + 2 - dz) * kTY + y0 + 2 - dy) * kTX + li + 2 - dx) * kDgS +
                       6 * kg;
      f32x2 g0[3], g1[3], b0[3], b1[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        g0[k] = *reinterpret_cast<const f32x2*>(g + 2 * k);
        g1[k] = *reinterpret_cast<const f32x2*>(g + kTX * kDgS + 2 * k);
        b0[k] = *reinterpret_cast<const f32x2*>(w0 + tap * kC * kDgS + 2 * k);
        b1[k] = *reinterpret_cast<const f32x2*>(w1 + tap * kC * kDgS + 2 * k);
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        acc[0][0] = mfma_f32(g0[k / 2][k % 2], b0[k / 2][k % 2], acc[0][0]);
        acc[1][0] = mfma_f32(g1[k / 2][k % 2], b0[k / 2][k % 2], acc[1][0]);
        acc[0][1] = mfma_f32(g0[k / 2][k % 2], b1[k / 2][k % 2], acc[0][1]);
        acc[1][1] = mfma_f32(g1[k / 2][k % 2], b1[k / 2][k % 2], acc[1][1]);
      }
    }
    const int gz = o.z + z;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int gy = o.y + y0 + m;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int ci = 16 * t + li;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int gx = o.x + 4 * kg + r;
          if (ci < kC && gx < a.W && gy < a.H && gz < a.D) {
            const int64_t q = (((o.n * a.D + gz) * a.H + gy) * a.W + gx) * kC + ci;
            a.out[q] = a.pre ? acc[m][t][r] * gelu_grad(a.pre[q]) : acc[m][t][r];
          }
        }
      }
    }
  }
}

// The same for 24 -> 1: one voxel per work-item, its 27 gradients from LDS,
// 24 sums over the taps with wave-uniform weights (taps off the patch are left
// out where a weight is not finite).  Bound by writing dx.
__global__ __launch_bounds__(256) void k_conv3d_dgrad_1c(const BwdArgs a) {
  __shared__ float S[kTV];
  const int tid = threadIdx.x;
  const int OD = a.D - 2, OH = a.H - 2, OW = a.W - 2;
  float chk = 0.f;  // stays 0 while every weight is finite
  for (int e = tid; e < 27 * kC; e += 256) chk = fmaf(a.w[e], 0.f, chk);
  const bool wbad = __syncthreads_or(!(chk == 0.f));
  for (int64_t blk = xcd_swizzle(blockIdx.x, gridDim.x); blk < a.nblocks; blk += gridDim.x) {
    const Origin o = origin_of(a, blk);
    __syncthreads();
    for (int e = tid; e < kTV; e += 256) {
      const int x = o.x + e % kTX - 2, y = o.y + e / kTX % kTY - 2, z = o.z + e / (kTX * kTY) - 2;
      S[e] = x >= 0 && y >= 0 && z >= 0 && x < OW && y < OH && z < OD
                 ? a.dy[((o.n * OD + z) * OH + y) * OW + x]
                 : 0.f;
    }
    __syncthreads();
    const int lx = tid % kBX, ly = tid / kBX % kBY, lz = tid / (kBX * kBY);
    float acc[kC];
#pragma unroll
    for (int c = 0; c < kC; ++c) acc[c] = 0.f;
    const int px = o.x + lx, py = o.y + ly, pz = o.z + lz;
#pragma unroll 3
    for (int tap = 0; tap < 27; ++tap) {
      if (wbad) {
        const int z = pz - tap / 9, y = py - tap / 3 % 3, x = px - tap % 3;
        if (x < 0 || y < 0 || z < 0 || x >= OW || y >= OH || z >= OD) continue;
      }
      const float g =
          S[((lz + 2 - tap / 9) * kTY + ly + 2 - tap / 3 % 3) * kTX + lx + 2 - tap % 3];
#pragma unroll
      for (int c = 0; c < kC; ++c) acc[c] = fmaf(g, a.w[tap * kC + c], acc[c]);
    }
    if (px < a.W && py < a.H && pz < a.D) {
      const int64_t q = (((o.n * a.D + pz) * a.H + py) * a.W + px) * kC;
#pragma unroll
      for (int v = 0; v < kC / 4; ++v) {
        f32x4 r{acc[4 * v], acc[4 * v + 1], acc[4 * v + 2], acc[4 * v + 3]};
        if (a.pre) {
          const f32x4 p = reinterpret_cast<const f32x4*>(a.pre + q)[v];
#pragma unroll
          for (int k = 0; k < 4; ++k) r[k] *= gelu_grad(p[k]);
        }
        reinterpret_cast<f32x4*>(a.out + q)[v] = r;
      }
    }
  }
}

namespace {

// Work-groups of the weight gradient: two per CU (59 KB of LDS and four waves
// each), so one's loads and barriers are covered by the other's products.
constexpr int kWgGrid = 512;

int bwd_args(BwdArgs* a, int64_t batch, int D, int H, int W, int ez, int ey, int ex) {
  std::memset(a, 0, sizeof(*a));
  a->D = D;
  a->H = H;
  a->W = W;
  a->nbx = (ex + kBX - 1) / kBX;
  a->nby = (ey + kBY - 1) / kBY;
  a->nbz = (ez + kBZ - 1) / kBZ;
  a->nblocks = batch * a->nbx * a->nby * a->nbz;
  if (a->nblocks > 0x7fffffff) return fail(HC_ERR_VALUE, "volume too large");
  return HC_OK;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace
}  // namespace hc

using namespace hc;

extern "C" {

int64_t hc_cnn3d_wgrad_work(int ci, int co) {
  if (ci == 24 && co == 24) return (int64_t)kWgGrid * kWgPart;
  if (ci == 1 && co == 24) return (int64_t)kWgGrid * 28 * kC;
  if (ci == 24 && co == 1) return (int64_t)kWgGrid * (27 * kC + 1);
  return -1;
}

int hc_cnn3d_wgrad_batch(const void* x_bf16, const float* dy, float* dw, float* db, int64_t batch,
                         int D, int H, int W, int ci, int co, float* work, int64_t work_elems,
                         void* stream) {
  if (!x_bf16 || !dy || !dw || !db || !work || batch < 1 || D < 3 || H < 3 || W < 3)
    return fail(HC_ERR_VALUE, "bad argument");
  const int64_t need = hc_cnn3d_wgrad_work(ci, co);
  if (need < 0) return fail(HC_ERR_UNSUPPORTED, "layer shape not compiled");
  if (work_elems < need) return fail(HC_ERR_VALUE, "work buffer too small");
  if (!aligned16(x_bf16) || !aligned16(dy) || !aligned16(work))
    return fail(HC_ERR_VALUE, "arrays must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  BwdArgs a;
  const bool last = co == 1;  // the blocks cover the 24-channel side
  const int rc =
      bwd_args(&a, batch, D, H, W, last ? D : D - 2, last ? H : H - 2, last ? W : W - 2);
  if (rc != HC_OK) return rc;
  a.x = (const __bf16*)x_bf16;
  a.dy = dy;
  a.out = work;
  const int grid = (int)std::min<int64_t>(a.nblocks, kWgGrid);
  const int nw = 27 * ci * co, n = nw + co;
  if (ci == 24 && co == 24)
    HC_LAUNCH("k_conv3d_wgrad_mfma", st, k_conv3d_wgrad_mfma, dim3(grid), dim3(256), 0, a);
  else if (ci == 1)
    HC_LAUNCH("k_conv3d_wgrad_1c", st, k_conv3d_wgrad_1c<true>, dim3(grid), dim3(256), 0, a);
  else
    HC_LAUNCH("k_conv3d_wgrad_1c", st, k_conv3d_wgrad_1c<false>, dim3(grid), dim3(256), 0, a);
  HC_LAUNCH("k_sum_parts", st, k_sum_parts, dim3((n + 63) / 64), dim3(1024), 0, work, grid, n, nw,
            dw, db);
  return HC_OK;
}

int hc_cnn3d_dgrad_batch(const float* dy, const float* w, const float* pre, float* dx,
                         int64_t batch, int D, int H, int W, int ci, int co, void* stream) {
  if (!dy || !w || !dx || batch < 1 || D < 3 || H < 3 || W < 3)
    return fail(HC_ERR_VALUE, "bad argument");
  if (ci != 24 || (co != 24 && co != 1))
    return fail(HC_ERR_UNSUPPORTED, "layer shape not compiled");
  if (!aligned16(dy) || !aligned16(w) || !aligned16(dx) || !aligned16(pre))
    return fail(HC_ERR_VALUE, "arrays must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  BwdArgs a;
  const int rc = bwd_args(&a, batch, D, H, W, D, H, W);
  if (rc != HC_OK) return rc;
  a.dy = dy;
  a.w = w;
  a.pre = pre;
  a.out = dx;
  if (co == 1) {
    const int grid = (int)std::min<int64_t>(a.nblocks, 256 * 8);
    HC_LAUNCH("k_conv3d_dgrad_1c", st, k_conv3d_dgrad_1c, dim3(grid), dim3(256), 0, a);
    return HC_OK;
  }
  const hipError_t e = hipFuncSetAttribute((const void*)k_conv3d_dgrad_mfma,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kDgLds);
  if (e != hipSuccess) return hip_check(e, "hipFuncSetAttribute(k_conv3d_dgrad_mfma)");
  const int grid = (int)std::min<int64_t>(a.nblocks, 256);  // one per CU: 142 KB of LDS
  HC_LAUNCH("k_conv3d_dgrad_mfma", st, k_conv3d_dgrad_mfma, dim3(grid), dim3(512), kDgLds, a);
  return HC_OK;
}

}  // extern "C"
