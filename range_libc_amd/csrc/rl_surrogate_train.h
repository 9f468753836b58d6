// Training kernels of the learned range surrogate: one minibatch is three
// launches (forward + loss + data gradients; weight and bias gradient partials;
// their sums and the Adam update).
//
// Included by rl_surrogate_impl.h (network, loss and parameter layout there).
//
// A minibatch of 16384 rays is 14.6 GFLOP and, kept in HBM between launches,
// 52 MB of activations and gradients: 6 us of matrix instructions at the
// 16x16x16 rate and 10 us of HBM.  One launch per layer and direction, with
// 2-byte strided loads staged through LDS, took 0.81 ms per minibatch; these
// three launches take 73 us (43 + 23 + 7).  Here a workgroup carries 64 rays through the whole forward and data-gradient chain
// with the activation tile in LDS, and writes what the weight gradients need
// transposed (one feature's values of consecutive rays contiguous), so that
// these are a product of two K-contiguous operands.
//
// The arithmetic keeps a fixed order: the 16x16x32 instruction over ascending k
// in the forward hidden layers, 16x16x16 over ascending k in the heads, the
// data gradients and the weight gradients; weight gradients in slices of
// sg_split(n).kchunk rows, added in slice order; bias gradients row by row in
// chunks of sg_split(n).cchunk rows, added in chunk order.

#define RL_SGT_ROWS 64    // rays per workgroup of k_sg_fwd_bwd
#define RL_SGT_THREADS 512
#define RL_SGT_BIAS (3 * RL_SG_H + RL_SG_OUT)

// Rows of the transposed training matrices (each ld bf16 values): features,
// activations a1..a3, gradients of the pre-activations dz1..dz3 and the output.
struct SgT {
  static constexpr int X = 0;
  static constexpr int A1 = X + RL_SG_F;
  static constexpr int A2 = A1 + RL_SG_H;
  static constexpr int A3 = A2 + RL_SG_H;
  static constexpr int D1 = A3 + RL_SG_H;
  static constexpr int D2 = D1 + RL_SG_H;
  static constexpr int D3 = D2 + RL_SG_H;
  static constexpr int DO = D3 + RL_SG_H;
  static constexpr int N = DO + RL_SG_OUT;
};

// Position of element k inside its 32-element group such that lane group g =
// lane >> 4 finds its operands of two 16x16x16 instructions (k = 4 g .. + 3 of
// each half) in 16 consecutive bytes.
__host__ __device__ __forceinline__ int sg_perm(int k) {
  return (k & ~31) | (((k & 15) >> 2) << 3) | (((k >> 4) & 1) << 2) | (k & 3);
}

// Parameter i with value v into the bf16 copies: the flat vector, and W2 / W3
// transposed with permuted rows, pt[l][in][sg_perm(out)] (data gradients).
__device__ __forceinline__ void sg_store_bf16(int i, float v, bf16_t* __restrict__ pb, bf16_t* __restrict__ pt) {
  const bf16_t h = f2bf(v);
  pb[i] = h;
  int e = -1, l = 0;
  if (i >= SgLayout::W2 && i < SgLayout::B2) e = i - SgLayout::W2;
  if (i >= SgLayout::W3 && i < SgLayout::B3) e = i - SgLayout::W3, l = 1;
  if (e >= 0) pt[l * RL_SG_H * RL_SG_H + (e & (RL_SG_H - 1)) * RL_SG_H + sg_perm(e / RL_SG_H)] = h;
}

__global__ void k_sg_to_bf16(const float* __restrict__ p, bf16_t* __restrict__ pb, bf16_t* __restrict__ pt, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) sg_store_bf16(i, p[i], pb, pt);
}

struct SgPass {
  const float4* rays;   // n x (x0, y0, sin h, cos h)
  const float* target;  // n ranges
  const float* freq;
  float inv_w, inv_h, max_range, inv_n;
  const bf16_t* P;      // bf16 parameters, flat
  const bf16_t* Pt;     // W2, W3 transposed (sg_store_bf16)
  const float* Pf;      // fp32 parameters
  bf16_t* T;            // SgT::N x ld
  bf16_t* x_rows;       // n x 64 features, row-major (optional)
  float* partial;       // loss partial of each workgroup
  int n, ld;            // ld: n rounded up to RL_SGT_ROWS
};

// A wave's output tile: 64 rows x 32 columns (columns 32 wave .. + 31) as 4 x 2
// MFMA tiles; lane l holds column l & 15 of a tile, rows 4 (l >> 4) .. + 3.
typedef sg_float4 SgAcc[4][2];

// Weight fragments of a forward layer: rows (output columns) of W [256][K].
template <int K>
__device__ __forceinline__ void sgt_load_fwd(sg_bf16x8 (&b)[8][2], const bf16_t* __restrict__ W, int wave, int lane) {
#pragma unroll
  for (int s = 0; s < K / 32; ++s)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      b[s][j] = *(const sg_bf16x8*)(W + (size_t)(wave * 32 + j * 16 + (lane & 15)) * K + s * 32 + (lane >> 4) * 8);
}

template <int K>
__device__ __forceinline__ void sgt_mul_fwd(SgAcc& acc, const bf16_t* act, const sg_bf16x8 (&b)[8][2], int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sg_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < K / 32; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const sg_bf16x8 a = *(const sg_bf16x8*)(act + (i * 16 + (lane & 15)) * RL_SG_ACT_PAD + s * 32 + (lane >> 4) * 8);
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[s][j], acc[i][j], 0, 0, 0);
    }
}

// The data gradient's product: act holds dz with its columns at sg_perm, b the
// fragments of pt (loaded as a forward layer of K = 256).
__device__ __forceinline__ void sgt_mul_bwd(SgAcc& acc, const bf16_t* act, const sg_bf16x8 (&b)[8][2], int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sg_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 8; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 a = *(const uint4*)(act + (i * 16 + (lane & 15)) * RL_SG_ACT_PAD + s * 32 + (lane >> 4) * 8);
      const sg_short4 a0 = __builtin_bit_cast(sg_short4, make_uint2(a.x, a.y));
      const sg_short4 a1 = __builtin_bit_cast(sg_short4, make_uint2(a.z, a.w));
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 w = __builtin_bit_cast(uint4, b[s][j]);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
            a0, __builtin_bit_cast(sg_short4, make_uint2(w.x, w.y)), acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
            a1, __builtin_bit_cast(sg_short4, make_uint2(w.z, w.w)), acc[i][j], 0, 0, 0);
      }
    }
}

// Four consecutive rows of one column to their transposed place; rows past n
// are stored as zeros, so that the weight gradients may read whole tiles.
__device__ __forceinline__ void sgt_store_t(bf16_t* __restrict__ Tc, int row, int rows_left, const bf16_t (&h)[4]) {
  bf16_t v[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = row + q < rows_left ? h[q] : (bf16_t)0;
  *(uint2*)(Tc + row) = make_uint2((unsigned)v[0] | ((unsigned)v[1] << 16), (unsigned)v[2] | ((unsigned)v[3] << 16));
}

// Forward epilogue: bias, relu, bf16; the tile rewritten in LDS, the transposed
// copy stored, bit 8 i + 4 j + q of the result set where the value is positive.
__device__ __forceinline__ unsigned sgt_out_fwd(const SgAcc& acc, bf16_t* act, const float* sb, bf16_t* __restrict__ T,
                                                int ld, int r0, int left, int wave, int lane) {
  unsigned pos = 0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = wave * 32 + j * 16 + (lane & 15);
    const float bb = sb[c];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = i * 16 + 4 * (lane >> 4);
      bf16_t h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v = acc[i][j][q] + bb;
        v = v < 0.0f ? 0.0f : v;
        h[q] = f2bf_hw(v);
        pos |= (bf2f(h[q]) > 0.0f ? 1u : 0u) << (8 * i + 4 * j + q);
        act[(row + q) * RL_SG_ACT_PAD + c] = h[q];
      }
      sgt_store_t(T + (size_t)c * ld + r0, row, left, h);
    }
  }
  return pos;
}

// Data-gradient epilogue: zero where the activation was not positive.
__device__ __forceinline__ void sgt_out_bwd(const SgAcc& acc, unsigned pos, bf16_t* act, bf16_t* __restrict__ T, int ld,
                                            int r0, int left, int wave, int lane, bool to_lds) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = wave * 32 + j * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = i * 16 + 4 * (lane >> 4);
      bf16_t h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        h[q] = f2bf_hw((pos >> (8 * i + 4 * j + q)) & 1u ? acc[i][j][q] : 0.0f);
        if (to_lds) act[(row + q) * RL_SG_ACT_PAD + sg_perm(c)] = h[q];
      }
      sgt_store_t(T + (size_t)c * ld + r0, row, left, h);
    }
  }
}

// Forward, loss and data gradients of 64 rays: 8 waves, each 32 of the 256
// columns.  At 16384 rays there is one workgroup per CU, so a layer's weight
// fragments (64 registers per lane) are all requested a layer ahead: the L2
// round trips, not the matrix instructions, are what the chain would wait for.
__global__ __launch_bounds__(RL_SGT_THREADS, 2) void k_sg_fwd_bwd(SgPass g) {
  __shared__ __align__(16) bf16_t act[RL_SGT_ROWS * RL_SG_ACT_PAD];
  __shared__ float sbias[RL_SGT_BIAS];
  __shared__ __align__(16) bf16_t sw4[RL_SG_OUT * RL_SG_H];
  __shared__ float sout[RL_SGT_ROWS][RL_SG_OUT];
  __shared__ bf16_t sdo[RL_SGT_ROWS][RL_SG_OUT];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r0 = blockIdx.x * RL_SGT_ROWS;
  const int left = g.n - r0;  // rays from this workgroup's first on
  const int ld = g.ld;
  sg_bf16x8 w1[8][2], w2[8][2];
  sgt_load_fwd<RL_SG_F>(w1, g.P + SgLayout::W1, wave, lane);
  sgt_load_fwd<RL_SG_H>(w2, g.P + SgLayout::W2, wave, lane);
  if (tid < RL_SG_H) {
    sbias[tid] = g.Pf[SgLayout::B1 + tid];
    sbias[RL_SG_H + tid] = g.Pf[SgLayout::B2 + tid];
    sbias[2 * RL_SG_H + tid] = g.Pf[SgLayout::B3 + tid];
    if (tid < RL_SG_OUT) sbias[3 * RL_SG_H + tid] = g.Pf[SgLayout::B4 + tid];
    sw4[tid] = g.P[SgLayout::W4 + tid];
    sw4[RL_SG_H + tid] = g.P[SgLayout::W4 + RL_SG_H + tid];
  }
  // features (k_sg_features' expression); rays past n: zeros
#pragma unroll
  for (int e = tid; e < RL_SGT_ROWS * RL_SG_NF; e += RL_SGT_THREADS) {
    const int r = e / RL_SG_NF, j = e - r * RL_SG_NF;
    bf16_t s = 0, c = 0;
    if (r < left) {
      const float4 rr = g.rays[r0 + r];
      const float v0 = rr.x * g.inv_w, v1 = rr.y * g.inv_h, v2 = rr.z, v3 = rr.w;
      const float p = 6.283185307179586f * (g.freq[4 * j] * v0 + g.freq[4 * j + 1] * v1 + g.freq[4 * j + 2] * v2 +
                                            g.freq[4 * j + 3] * v3);
      s = f2bf(sinf(p));
      c = f2bf(cosf(p));
    }
    act[r * RL_SG_ACT_PAD + j] = s;
    act[r * RL_SG_ACT_PAD + RL_SG_NF + j] = c;
  }
  __syncthreads();
  {  // 64 features x 8 groups of 8 rows: the features transposed
    const int f = tid >> 3, r = (tid & 7) * 8;
    unsigned v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = (unsigned)act[(r + 2 * q) * RL_SG_ACT_PAD + f] | ((unsigned)act[(r + 2 * q + 1) * RL_SG_ACT_PAD + f] << 16);
    *(uint4*)(g.T + (size_t)(SgT::X + f) * ld + r0 + r) = make_uint4(v[0], v[1], v[2], v[3]);
    if (g.x_rows) {  // and as they are: row tid >> 3, 8 features
      const int row = tid >> 3, c = (tid & 7) * 8;
      if (row < left)
        *(uint4*)(g.x_rows + (size_t)(r0 + row) * RL_SG_F + c) = *(const uint4*)(act + row * RL_SG_ACT_PAD + c);
    }
  }
  SgAcc acc;
  sgt_mul_fwd<RL_SG_F>(acc, act, w1, lane);
  sgt_load_fwd<RL_SG_H>(w1, g.P + SgLayout::W3, wave, lane);
  __syncthreads();
  const unsigned pos1 = sgt_out_fwd(acc, act, sbias, g.T + (size_t)SgT::A1 * ld, ld, r0, left, wave, lane);
  __syncthreads();
  sgt_mul_fwd<RL_SG_H>(acc, act, w2, lane);
  sgt_load_fwd<RL_SG_H>(w2, g.Pt + RL_SG_H * RL_SG_H, wave, lane);  // W3 transposed
  __syncthreads();
  const unsigned pos2 = sgt_out_fwd(acc, act, sbias + RL_SG_H, g.T + (size_t)SgT::A2 * ld, ld, r0, left, wave, lane);
  __syncthreads();
  sgt_mul_fwd<RL_SG_H>(acc, act, w1, lane);
  sgt_load_fwd<RL_SG_H>(w1, g.Pt, wave, lane);  // W2 transposed
  __syncthreads();
  const unsigned pos3 = sgt_out_fwd(acc, act, sbias + 2 * RL_SG_H, g.T + (size_t)SgT::A3 * ld, ld, r0, left, wave, lane);
  __syncthreads();
  if (wave < 4) {  // heads: wave w takes rows 16 w .. 16 w + 15, columns 0 and 1 of one tile
    const int col = lane & 15, kb = 4 * (lane >> 4);
    sg_float4 o = sg_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < RL_SG_H; k += 16) {
      const sg_short4 a = *(const sg_short4*)(act + (wave * 16 + col) * RL_SG_ACT_PAD + k + kb);
      const sg_short4 b = col < RL_SG_OUT ? *(const sg_short4*)(sw4 + col * RL_SG_H + k + kb) : sg_short4{0, 0, 0, 0};
      o = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, o, 0, 0, 0);
    }
    if (col < RL_SG_OUT)
#pragma unroll
      for (int q = 0; q < 4; ++q) sout[wave * 16 + kb + q][col] = o[q] + sbias[3 * RL_SG_H + col];
  }
  __syncthreads();
  if (wave == 0) {  // loss and output gradient, one ray per lane
    float l = 0.0f;
    bf16_t d0 = 0, d1 = 0;
    if (lane < left) {
      const float tau = 0.95f;
      const float e = g.max_range * sout[lane][0] - g.target[r0 + lane];
      const float ae = fabsf(e);
      const float lr = ae <= 1.0f ? 0.5f * e * e : ae - 0.5f;
      const float ge = ae <= 1.0f ? e : (e > 0.0f ? 1.0f : -1.0f);
      const float lb0 = sout[lane][1];
      const float lb = lb0 > 20.0f ? 20.0f : (lb0 < -20.0f ? -20.0f : lb0);
      const float b = expf(lb);
      const float lq = ae > b ? tau * (ae - b) : (1.0f - tau) * (b - ae);
      const float gb = lb == lb0 ? (ae > b ? -tau : (1.0f - tau)) * b : 0.0f;
      l = lr + 0.1f * lq;
      d0 = f2bf(ge * g.max_range * g.inv_n);
      d1 = f2bf(0.1f * gb * g.inv_n);
    }
    sdo[lane][0] = d0;
    sdo[lane][1] = d1;
    g.T[(size_t)SgT::DO * ld + r0 + lane] = d0;
    g.T[(size_t)(SgT::DO + 1) * ld + r0 + lane] = d1;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) l += __shfl_down(l, s);
    if (lane == 0) g.partial[blockIdx.x] = l * g.inv_n;
  }
  __syncthreads();
  {  // dz3 = dout W4: k = 0, 1 of one 16x16x16 instruction
    const bool k0 = (lane >> 4) == 0;
    const int r16 = lane & 15;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const sg_short4 a = k0 ? sg_short4{(short)sdo[i * 16 + r16][0], (short)sdo[i * 16 + r16][1], 0, 0}
                             : sg_short4{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int c = wave * 32 + j * 16 + r16;
        const sg_short4 b = k0 ? sg_short4{(short)sw4[c], (short)sw4[RL_SG_H + c], 0, 0} : sg_short4{0, 0, 0, 0};
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, sg_float4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
    }
  }
  sgt_out_bwd(acc, pos3, act, g.T + (size_t)SgT::D3 * ld, ld, r0, left, wave, lane, true);  // a3 was read before
  __syncthreads();
  sgt_mul_bwd(acc, act, w2, lane);
  __syncthreads();
  sgt_out_bwd(acc, pos2, act, g.T + (size_t)SgT::D2 * ld, ld, r0, left, wave, lane, true);
  __syncthreads();
  sgt_mul_bwd(acc, act, w1, lane);
  sgt_out_bwd(acc, pos1, act, g.T + (size_t)SgT::D1 * ld, ld, r0, left, wave, lane, false);
}

// How the gradient sums over n rays are cut: weight gradients into nz slices
// of kchunk rows (about 1024, at most RL_SG_MAX_SPLIT slices), bias gradients
// into ncz chunks of cchunk rows (at least 256, at most 256 chunks).
struct SgSplit {
  int kchunk, nz, cchunk, ncz;
};
static SgSplit sg_split(int n) {
  SgSplit s;
  const int splits = std::max(1, std::min(RL_SG_MAX_SPLIT, (n + 1023) / 1024));
  s.kchunk = ((n + splits - 1) / splits + 31) / 32 * 32;
  s.nz = (n + s.kchunk - 1) / s.kchunk;
  s.cchunk = std::max(256, (n + 255) / 256);
  s.ncz = (n + s.cchunk - 1) / s.cchunk;
  return s;
}

// Gradient partials of one launch.  Workgroups [0, 8 ceil(nz / 8) RL_SGT_TILES):
// a 64 x 64 tile of one layer's weight gradient over one slice of rows,
// dW[o][i] = sum_b dz[b][o] act[b][i], both operands with b contiguous (T).
// All tiles of a slice are on one XCD (workgroup b runs on XCD b mod 8): the
// slice's rows, 3.2 MB at 1024, are read from HBM once and then from that
// XCD's 4 MB L2.  The remaining workgroups: the bias gradients' column sums.
#define RL_SGT_TILES 40  // 64 x 64 tiles of dW3 (16), dW2 (16), dW1 (4), dW4 (4)
#define RL_SGT_PAD 72    // LDS row stride in elements: the 8-byte reads of 16 rows fall on distinct banks
__global__ __launch_bounds__(256) void k_sg_wgrad(const bf16_t* __restrict__ T, int n, int ld, SgSplit sp, int gemm_blocks,
                                                  float* __restrict__ part, float* __restrict__ bpart) {
  __shared__ __align__(16) bf16_t As[64 * RL_SGT_PAD];
  __shared__ __align__(16) bf16_t Bs[64 * RL_SGT_PAD];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if ((int)blockIdx.x >= gemm_blocks) {
    // one thread per (column, chunk): its rows in order, 8 per load (rows
    // outside the chunk add +0)
    const int e = ((int)blockIdx.x - gemm_blocks) * 256 + tid;
    const int z = e / RL_SGT_BIAS, c = e - z * RL_SGT_BIAS;
    if (z >= sp.ncz) return;
    const bf16_t* src = T + (size_t)(SgT::D1 + c) * ld;  // dz1, dz2, dz3, dout follow each other
    const int b0 = z * sp.cchunk, b1 = min(n, b0 + sp.cchunk);
    float s = 0.0f;
#pragma unroll 4
    for (int b = b0 & ~7; b < b1; b += 8) {
      const uint4 v = *(const uint4*)(src + b);
      const unsigned u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float x = bf2f((bf16_t)(u[q >> 1] >> (16 * (q & 1))));
        s += (b + q >= b0 && b + q < b1) ? x : 0.0f;
      }
    }
    bpart[(size_t)z * RL_SGT_BIAS + c] = s;
    return;
  }
  const int x = (int)blockIdx.x & 7, q8 = (int)blockIdx.x >> 3;
  const int slice = x + 8 * (q8 / RL_SGT_TILES), tile = q8 % RL_SGT_TILES;
  if (slice >= sp.nz) return;  // the same in every thread
  int a_row, b_row, o0, i0, fin, out, rows;
  if (tile < 32) {
    const bool l3 = tile < 16;
    const int t = tile & 15;
    o0 = (t >> 2) * 64, i0 = (t & 3) * 64, fin = RL_SG_H, rows = 64;
    a_row = l3 ? SgT::D3 : SgT::D2, b_row = l3 ? SgT::A2 : SgT::A1;
    out = l3 ? SgLayout::W3 : SgLayout::W2;
  } else if (tile < 36) {
    o0 = (tile - 32) * 64, i0 = 0, fin = RL_SG_F, rows = 64;
    a_row = SgT::D1, b_row = SgT::X, out = SgLayout::W1;
  } else {
    o0 = 0, i0 = (tile - 36) * 64, fin = RL_SG_H, rows = RL_SG_OUT;
    a_row = SgT::DO, b_row = SgT::A3, out = SgLayout::W4;
  }
  const bf16_t* A = T + (size_t)(a_row + o0) * ld;
  const bf16_t* B = T + (size_t)(b_row + i0) * ld;
  const int kbeg = slice * sp.kchunk, kend = min(ld, kbeg + sp.kchunk);  // multiples of 32
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  sg_float4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sg_float4{0.f, 0.f, 0.f, 0.f};
  // 64 rows of k per stage: rows r and r + 32 of each operand, 8 values per load
  const int r = tid >> 3, c8 = (tid & 7) * 8;
  uint4 va[2], vb[2];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = r + 32 * h;
      const bool in = k0 + c8 < kend;
      va[h] = in && row < rows ? *(const uint4*)(A + (size_t)row * ld + k0 + c8) : make_uint4(0u, 0u, 0u, 0u);
      vb[h] = in ? *(const uint4*)(B + (size_t)row * ld + k0 + c8) : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  fetch(kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += 64) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      *(uint4*)(As + (r + 32 * h) * RL_SGT_PAD + c8) = va[h];
      *(uint4*)(Bs + (r + 32 * h) * RL_SGT_PAD + c8) = vb[h];
    }
    __syncthreads();
    fetch(k0 + 64);  // past the slice: zeros, not used
#pragma unroll
    for (int ks = 0; ks < 64; ks += 16) {
      const int kb = ks + 4 * (lane >> 4);
      sg_short4 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = *(const sg_short4*)(As + (wm + i * 16 + (lane & 15)) * RL_SGT_PAD + kb);
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = *(const sg_short4*)(Bs + (wn + j * 16 + (lane & 15)) * RL_SGT_PAD + kb);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  float* dst = part + (size_t)slice * RL_SG_NPARAM + out;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int o = wm + i * 16 + 4 * (lane >> 4) + q;
        if (o < rows) dst[(size_t)(o0 + o) * fin + i0 + wn + j * 16 + (lane & 15)] = acc[i][j][q];
      }
}

// Sums of the gradient partials in slice / chunk order (SUM) into grad, and the
// Adam step with it (ADAM; without SUM, with the gradient grad holds), which
// writes the bf16 copies as well.  One thread per parameter.
template <bool SUM, bool ADAM>
__global__ __launch_bounds__(256) void k_sg_update(const float* __restrict__ part, const float* __restrict__ bpart, int nz,
                                                   int ncz, float* __restrict__ grad, float* __restrict__ p,
                                                   float* __restrict__ m1, float* __restrict__ m2,
                                                   bf16_t* __restrict__ pb, bf16_t* __restrict__ pt, float lr, float b1,
                                                   float b2, float c1, float c2, float eps) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= RL_SG_NPARAM) return;
  float g;
  if (SUM) {
    int bias = -1;  // column of bpart, -1: a weight
    if (i >= SgLayout::B1 && i < SgLayout::W2) bias = i - SgLayout::B1;
    if (i >= SgLayout::B2 && i < SgLayout::W3) bias = RL_SG_H + i - SgLayout::B2;
    if (i >= SgLayout::B3 && i < SgLayout::W4) bias = 2 * RL_SG_H + i - SgLayout::B3;
    if (i >= SgLayout::B4) bias = 3 * RL_SG_H + i - SgLayout::B4;
    const float* src = bias < 0 ? part + i : bpart + bias;
    const size_t stride = bias < 0 ? RL_SG_NPARAM : RL_SGT_BIAS;
    const int cnt = bias < 0 ? nz : ncz;
    g = 0.0f;
#pragma unroll 8
    for (int z = 0; z < cnt; ++z) g += src[z * stride];  // loads issued ahead, sums in order
    grad[i] = g;
  } else {
    g = grad[i];
  }
  if (ADAM) {
    const float a = b1 * m1[i] + (1.0f - b1) * g;
    const float b = b2 * m2[i] + (1.0f - b2) * g * g;
    m1[i] = a;
    m2[i] = b;
    const float v = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    p[i] = v;
    sg_store_bf16(i, v, pb, pt);
  }
}
