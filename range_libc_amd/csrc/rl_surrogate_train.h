// Training kernels of the learned range surrogate: one minibatch is three
// launches (forward + loss + data gradients; weight and bias gradient partials;
// their sums and the Adam update).
//
// Included by rl_surrogate_impl.h (network, loss and parameter layout there).
//
// A minibatch of 16384 rays is 14.6 GFLOP and, kept in HBM between launches,
// 52 MB of activations and gradients: 6 us of matrix instructions and 10 us of
// HBM each way.  One launch per layer and direction, with 2-byte strided loads
// staged through LDS, took 0.81 ms per minibatch; now 24 + 21 + 7 us.  Here a workgroup carries 64 rays
// through the whole forward and data-gradient chain with the activation tile
// in LDS, and the weight gradients of all layers are one launch.
//
// The arithmetic keeps a fixed order: every product sums ascending k with
// v_mfma_f32_16x16x32_bf16 (its bits are those of two 16x16x16 instructions in
// turn, and do not depend on which operand comes first: no difference in
// 512,000 random tiles over 14 binades); weight gradients in slices of
// sg_split(n).kchunk rows, added in slice order; bias gradients row by row in
// chunks of sg_split(n).cchunk rows, added in chunk order; the loss in a tree over each
// workgroup's 64 rays, whose sums the host adds in order.

#define RL_SGT_ROWS 64    // rays per workgroup of k_sg_fwd_bwd
#define RL_SGT_RT (RL_SGT_ROWS / 16)
#define RL_SGT_THREADS 512
#define RL_SGT_BIAS (3 * RL_SG_H + RL_SG_OUT)
#define RL_SGT_PART ((RL_SG_NPARAM + 3) / 4 * 4)  // floats of a slice of gradient partials

// The training matrices, each `ld` rows (rays) of its width, one after the
// other: matrix M starts at T + M * ld.  Features, activations a1..a3, gradients
// of the pre-activations dz1..dz3 and of the output (two values in rows of 8).
#define RL_SGT_DO 8
struct SgT {
  static constexpr int X = 0;
  static constexpr int A1 = X + RL_SG_F;
  static constexpr int A2 = A1 + RL_SG_H;
  static constexpr int A3 = A2 + RL_SG_H;
  static constexpr int D1 = A3 + RL_SG_H;
  static constexpr int D2 = D1 + RL_SG_H;
  static constexpr int D3 = D2 + RL_SG_H;
  static constexpr int DO = D3 + RL_SG_H;
  static constexpr int N = DO + RL_SGT_DO;
};

// Parameter i with value v into the bf16 copies: the flat vector, and the hidden
// layers' weights as matrix operands (SgFrag).
__device__ __forceinline__ void sg_store_bf16(int i, float v, bf16_t* __restrict__ pb, bf16_t* __restrict__ pf) {
  const bf16_t h = f2bf(v);
  pb[i] = h;
  if (i < SgLayout::B1) pf[SgFrag::W1 + SgFrag::at(i / RL_SG_F, i % RL_SG_F, RL_SG_F)] = h;
  int e = -1, w = SgFrag::W2, wt = SgFrag::W2T;
  if (i >= SgLayout::W2 && i < SgLayout::B2) e = i - SgLayout::W2;
  if (i >= SgLayout::W3 && i < SgLayout::B3) e = i - SgLayout::W3, w = SgFrag::W3, wt = SgFrag::W3T;
  if (e >= 0) {
    pf[w + SgFrag::at(e / RL_SG_H, e % RL_SG_H, RL_SG_H)] = h;
    pf[wt + SgFrag::at(e % RL_SG_H, e / RL_SG_H, RL_SG_H)] = h;
  }
}

__global__ void k_sg_to_bf16(const float* __restrict__ p, bf16_t* __restrict__ pb, bf16_t* __restrict__ pf, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) sg_store_bf16(i, p[i], pb, pf);
}

struct SgPass {
  const float4* rays;   // n x (x0, y0, sin h, cos h)
  const float* target;  // n ranges
  const float* freq;
  float inv_w, inv_h, max_range, inv_n;
  const bf16_t* P;      // bf16 parameters, flat
  const bf16_t* F;      // the weights as matrix operands (SgFrag)
  const float* Pf;      // fp32 parameters
  bf16_t* T;            // training matrices (SgT)
  float* partial;       // loss partial of each workgroup
  int n, ld;            // ld: n rounded up to 64
};

// A wave's output tile: all rows x 32 columns (columns 32 wave .. + 31) as RT x 2
// MFMA tiles, the weights as the first operand: lane l holds row l & 15 of a
// tile and its columns 4 (l >> 4) .. + 3, four neighbours in the row-major tile.
typedef sg_float4 SgAcc[RL_SGT_RT][2];

// Weight fragments of a layer for columns 32 wave .. + 31 (W: its place in SgFrag).
template <int K>
__device__ __forceinline__ void sgt_load(sg_bf16x8 (&b)[8][2], const bf16_t* __restrict__ W, int wave, int lane) {
#pragma unroll
  for (int s = 0; s < K / 32; ++s)
#pragma unroll
    for (int j = 0; j < 2; ++j) b[s][j] = *(const sg_bf16x8*)(W + (((wave * 2 + j) * (K / 32) + s) * 64 + lane) * 8);
}

template <int K>
__device__ __forceinline__ void sgt_mul(SgAcc& acc, const bf16_t* act, const sg_bf16x8 (&b)[8][2], int lane) {
#pragma unroll
  for (int i = 0; i < RL_SGT_RT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sg_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < K / 32; ++s)
#pragma unroll
    for (int i = 0; i < RL_SGT_RT; ++i) {
      const sg_bf16x8 a = *(const sg_bf16x8*)(act + (i * 16 + (lane & 15)) * RL_SG_ACT_PAD + s * 32 + (lane >> 4) * 8);
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][j], a, acc[i][j], 0, 0, 0);
    }
}

// Forward epilogue: bias, relu, bf16 into the LDS tile; bit 8 i + 4 j + q of
// the result is set where the rounded value is positive.
__device__ __forceinline__ unsigned sgt_out_fwd(const SgAcc& acc, bf16_t* act, const float* sb, int wave, int lane) {
  unsigned pos = 0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = wave * 32 + j * 16 + 4 * (lane >> 4);
    const sg_float4 bb = *(const sg_float4*)(sb + c);
#pragma unroll
    for (int i = 0; i < RL_SGT_RT; ++i) {
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = acc[i][j][q] + bb[q];
        v[q] = v[q] < 0.0f ? 0.0f : v[q];
        // values up to 2^-134 round to zero
        pos |= v[q] > 0x1p-134f ? 1u << (8 * i + 4 * j + q) : 0u;
      }
      *(uint2*)(act + (i * 16 + (lane & 15)) * RL_SG_ACT_PAD + c) = make_uint2(sg_pack2(v[0], v[1]), sg_pack2(v[2], v[3]));
    }
  }
  return pos;
}

// Data-gradient epilogue: zero where the activation was not positive.
__device__ __forceinline__ void sgt_out_bwd(const SgAcc& acc, unsigned pos, bf16_t* act, int wave, int lane) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = wave * 32 + j * 16 + 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < RL_SGT_RT; ++i) {
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int keep = (int)(pos << (31 - (8 * i + 4 * j + q))) >> 31;  // the bit over the whole word
        v[q] = __int_as_float(__float_as_int(acc[i][j][q]) & keep);
      }
      *(uint2*)(act + (i * 16 + (lane & 15)) * RL_SG_ACT_PAD + c) = make_uint2(sg_pack2(v[0], v[1]), sg_pack2(v[2], v[3]));
    }
  }
}

// The LDS tile (64 rows x 256) to its rows of a training matrix; rows past n
// are stored as zeros, so that the weight gradients may read whole tiles.
__device__ __forceinline__ void sgt_store(const bf16_t* act, bf16_t* __restrict__ M, int left, int tid) {
#pragma unroll
  for (int t = 0; t < RL_SGT_ROWS * RL_SG_H / 8 / RL_SGT_THREADS; ++t) {
    const int e = tid + t * RL_SGT_THREADS, row = e >> 5, c = (e & 31) * 8;
    uint4 v = *(const uint4*)(act + row * RL_SG_ACT_PAD + c);
    if (row >= left) v = make_uint4(0u, 0u, 0u, 0u);
    *(uint4*)(M + (size_t)row * RL_SG_H + c) = v;
  }
}

// Forward, loss and data gradients of 64 rays: 8 waves, each 32 of the 256
// columns.  At 16384 rays there is one workgroup per CU, so its serial chain is
// the launch's time: a layer's weight fragments are requested before the
// previous layer's epilogue and stores (loads and stores are waited for in
// order), and the layers are loops, so that their code is fetched once.  24 us
// at 16384 rays (35 with fragments from the row-major weights and unrolled
// layers); with 32 rays per workgroup, two of them per CU, 27.
__global__ __launch_bounds__(RL_SGT_THREADS, 2) void k_sg_fwd_bwd(SgPass g) {
  __shared__ __align__(16) bf16_t act[RL_SGT_ROWS * RL_SG_ACT_PAD];
  __shared__ __align__(16) float sbias[RL_SGT_BIAS];
  __shared__ __align__(16) bf16_t sw4[RL_SG_OUT * RL_SG_H];
  __shared__ float sout[RL_SGT_ROWS][RL_SG_OUT];
  __shared__ unsigned sdo[RL_SGT_ROWS];  // output gradient, two bf16
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r0 = blockIdx.x * RL_SGT_ROWS;
  const int left = g.n - r0;  // rays from this workgroup's first on
  const size_t ld = (size_t)g.ld;
  auto mat = [&](int m) { return g.T + m * ld + (size_t)r0 * RL_SG_H; };  // this workgroup's rows of a 256-wide matrix
  // loads return in order: what the features need first, then the weights
  constexpr int FR = RL_SGT_ROWS * RL_SG_NF / RL_SGT_THREADS;  // rows of a thread, all of frequency tid % 32
  const int fj = tid & (RL_SG_NF - 1), fr = tid / RL_SG_NF;
  const float4 fq = ((const float4*)g.freq)[fj];
  float4 ray[FR];
#pragma unroll
  for (int k = 0; k < FR; ++k) {
    const int r = fr + k * (RL_SGT_THREADS / RL_SG_NF);
    ray[k] = g.rays[r0 + (r < left ? r : 0)];
  }
  const float target = g.target[r0 + (lane < left ? lane : 0)];
  float b[4];
#pragma unroll
  for (int k = 0; k < 3; ++k) b[k] = g.Pf[(k == 0 ? SgLayout::B1 : k == 1 ? SgLayout::B2 : SgLayout::B3) + (tid & (RL_SG_H - 1))];
  b[3] = g.Pf[SgLayout::B4 + (tid & 1)];
  const bf16_t w4 = g.P[SgLayout::W4 + tid];
  sg_bf16x8 w[8][2];
  sgt_load<RL_SG_F>(w, g.F + SgFrag::W1, wave, lane);
  __builtin_amdgcn_sched_barrier(0);
  if (tid < RL_SG_H) {
#pragma unroll
    for (int k = 0; k < 3; ++k) sbias[k * RL_SG_H + tid] = b[k];
    if (tid < RL_SG_OUT) sbias[3 * RL_SG_H + tid] = b[3];
  }
  sw4[tid] = w4;  // RL_SGT_THREADS = RL_SG_OUT * RL_SG_H
  // features (k_sg_features' expression); rays past n: zeros
#pragma unroll 1
  for (int k = 0; k < FR; ++k) {
    const int r = fr + k * (RL_SGT_THREADS / RL_SG_NF);
    const float v0 = ray[0].x * g.inv_w, v1 = ray[0].y * g.inv_h, v2 = ray[0].z, v3 = ray[0].w;
#pragma unroll
    for (int q = 0; q + 1 < FR; ++q) ray[q] = ray[q + 1];  // the next row's, at a fixed index
    const float p = 6.283185307179586f * (fq.x * v0 + fq.y * v1 + fq.z * v2 + fq.w * v3);
    act[r * RL_SG_ACT_PAD + fj] = r < left ? f2bf(sinf(p)) : (bf16_t)0;
    act[r * RL_SG_ACT_PAD + RL_SG_NF + fj] = r < left ? f2bf(cosf(p)) : (bf16_t)0;
  }
  __syncthreads();
  {  // the features: row tid >> 3, 8 of them (zeros past n)
    const int row = tid >> 3, c = (tid & 7) * 8;
    *(uint4*)(g.T + SgT::X * ld + (size_t)(r0 + row) * RL_SG_F + c) = *(const uint4*)(act + row * RL_SG_ACT_PAD + c);
  }
  SgAcc acc;
  sgt_mul<RL_SG_F>(acc, act, w, lane);
  sgt_load<RL_SG_H>(w, g.F + SgFrag::W2, wave, lane);
  __syncthreads();
  unsigned p1 = 0, p2 = 0, p3 = sgt_out_fwd(acc, act, sbias, wave, lane);
  __syncthreads();
#pragma unroll 1
  for (int l = 0; l < 2; ++l) {
    sgt_store(act, mat(SgT::A1 + l * RL_SG_H), left, tid);
    sgt_mul<RL_SG_H>(acc, act, w, lane);
    sgt_load<RL_SG_H>(w, g.F + (l == 0 ? SgFrag::W3 : SgFrag::W3T), wave, lane);
    __syncthreads();
    p1 = p2, p2 = p3;
    p3 = sgt_out_fwd(acc, act, sbias + (l + 1) * RL_SG_H, wave, lane);
    __syncthreads();
  }
  sgt_store(act, mat(SgT::A3), left, tid);
  if (wave < RL_SGT_RT) {  // heads: wave w takes rows 16 w .. 16 w + 15, columns 0 and 1 of one tile
    const int col = lane & 15, kb = 4 * (lane >> 4);
    sg_float4 o = sg_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < RL_SG_H; k += 32) {
      const sg_bf16x8 a = *(const sg_bf16x8*)(act + (wave * 16 + col) * RL_SG_ACT_PAD + k + 2 * kb);
      sg_bf16x8 b{};
      if (col < RL_SG_OUT) b = *(const sg_bf16x8*)(sw4 + col * RL_SG_H + k + 2 * kb);
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, o, 0, 0, 0);
    }
    if (col < RL_SG_OUT)
#pragma unroll
      for (int q = 0; q < 4; ++q) sout[wave * 16 + kb + q][col] = o[q] + sbias[3 * RL_SG_H + col];
  }
  __syncthreads();
  if (tid < RL_SGT_ROWS) {  // loss and output gradient, one ray per lane
    float l = 0.0f;
    bf16_t d0 = 0, d1 = 0;
    if (lane < left) {
      const float tau = 0.95f;
      const float e = g.max_range * sout[lane][0] - target;
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
    const unsigned d01 = (unsigned)d0 | ((unsigned)d1 << 16);
    sdo[lane] = d01;
    *(uint4*)(g.T + SgT::DO * ld + (size_t)(r0 + lane) * RL_SGT_DO) = make_uint4(d01, 0u, 0u, 0u);
#pragma unroll
    for (int s = RL_SGT_ROWS / 2; s > 0; s >>= 1) l += __shfl_down(l, s);
    if (lane == 0) g.partial[blockIdx.x] = l * g.inv_n;
  }
  __syncthreads();
  {  // dz3 = dout W4: k = 0, 1 of one instruction
    const bool k0 = (lane >> 4) == 0;
    const int r16 = lane & 15;
    uint4 v[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = wave * 32 + j * 16 + r16;
      v[j] = make_uint4(k0 ? (unsigned)sw4[c] | ((unsigned)sw4[RL_SG_H + c] << 16) : 0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int i = 0; i < RL_SGT_RT; ++i) {
      const uint4 d = make_uint4(k0 ? sdo[i * 16 + r16] : 0u, 0u, 0u, 0u);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sg_bf16x8, v[j]),
                                                            __builtin_bit_cast(sg_bf16x8, d),
                                                            sg_float4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
  }
  sgt_out_bwd(acc, p3, act, wave, lane);  // a3 was read before
  __syncthreads();
#pragma unroll 1
  for (int l = 0; l < 2; ++l) {
    sgt_store(act, mat(SgT::D3 - l * RL_SG_H), left, tid);
    sgt_mul<RL_SG_H>(acc, act, w, lane);
    if (l == 0) sgt_load<RL_SG_H>(w, g.F + SgFrag::W2T, wave, lane);
    __syncthreads();
    sgt_out_bwd(acc, p2, act, wave, lane);
    p2 = p1;
    __syncthreads();
  }
  sgt_store(act, mat(SgT::D1), left, tid);
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

// Gradient partials of one launch.  The first bias_blocks workgroups (a multiple
// of 8): the bias gradients' column sums, one thread per (column, chunk), its
// rows in order.  Then 8 ceil(nz / 8) RL_SGT_TILES workgroups: a 64 x 64 tile of
// one layer's weight gradient over one slice of rows, dW[o][i] = sum_b dz[b][o]
// act[b][i].  All tiles of a slice are on one XCD (workgroup b runs on XCD b mod
// 8): the slice's rows, 3.2 MB at 1024, are read from HBM once and then from
// that XCD's 4 MB L2.  Both operands have the summed index b as their row, so
// their tiles sit in LDS as they come and are read through the transposing LDS
// load.  A slice is a chain of 16 stages of 64 rows, RL_SGT_AHEAD of which are
// requested before they are needed.  21 us at 16384 rays, 17 without the column
// sums, and as long when every stage reads the same rows: the tiles' way from
// L2 through LDS bounds it, not HBM.
#define RL_SGT_TILES 40  // 64 x 64 tiles of dW3 (16), dW2 (16), dW1 (4), dW4 (4)
#define RL_SGT_PAD 80    // LDS row stride in elements: the 32-byte runs of 8 rows fall on distinct banks
#define RL_SGT_AHEAD 4

// Operand of a 16x16x32 instruction from an LDS tile [k][m]: lane l gets m =
// m0 + (l & 15), k = k0 + 8 (l >> 4) .. + 7.  The transposing load gives 16 lanes
// the transpose of the 4 x 16 block whose 8-byte pieces their addresses name.
__device__ __forceinline__ sg_bf16x8 sgt_frag(const bf16_t* tile, int k0, int m0, int lane) {
  const bf16_t* p = tile + (k0 + 8 * (lane >> 4) + ((lane & 15) >> 2)) * RL_SGT_PAD + m0 + 4 * (lane & 3);
  const sg_short4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((RL_LDS sg_short4*)p);
  const sg_short4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((RL_LDS sg_short4*)(p + 4 * RL_SGT_PAD));
  return __builtin_bit_cast(sg_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

__global__ __launch_bounds__(256) void k_sg_wgrad(const bf16_t* __restrict__ T, int n, int ld, SgSplit sp, int bias_blocks,
                                                  float* __restrict__ part, float* __restrict__ bpart) {
  __shared__ __align__(16) bf16_t As[2][64 * RL_SGT_PAD];
  __shared__ __align__(16) bf16_t Bs[2][64 * RL_SGT_PAD];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if ((int)blockIdx.x < bias_blocks) {
    const int e = (int)blockIdx.x * 256 + tid;
    const int z = e / RL_SGT_BIAS, c = e - z * RL_SGT_BIAS;
    if (z >= sp.ncz) return;
    const int w = c < 3 * RL_SG_H ? RL_SG_H : RL_SGT_DO, l = c / RL_SG_H;  // dz1, dz2, dz3, dout follow each other
    const bf16_t* src = T + (size_t)(SgT::D1 + l * RL_SG_H) * ld + (c - l * RL_SG_H);
    const int b0 = z * sp.cchunk, b1 = min(n, b0 + sp.cchunk);
    float s = 0.0f;
#pragma unroll 32
    for (int b = b0; b < b1; ++b) s += bf2f(src[(size_t)b * w]);  // loads issued ahead, sums in order
    bpart[(size_t)z * RL_SGT_BIAS + c] = s;
    return;
  }
  const int blk = (int)blockIdx.x - bias_blocks;
  const int x = blk & 7, q8 = blk >> 3;
  const int slice = x + 8 * (q8 / RL_SGT_TILES), tile = q8 % RL_SGT_TILES;
  if (slice >= sp.nz) return;  // the same in every thread
  int a_mat, b_mat, o0, i0, fin, out;
  if (tile < 32) {
    const bool l3 = tile < 16;
    const int t = tile & 15;
    o0 = (t >> 2) * 64, i0 = (t & 3) * 64, fin = RL_SG_H;
    a_mat = l3 ? SgT::D3 : SgT::D2, b_mat = l3 ? SgT::A2 : SgT::A1;
    out = l3 ? SgLayout::W3 : SgLayout::W2;
  } else if (tile < 36) {
    o0 = (tile - 32) * 64, i0 = 0, fin = RL_SG_F;
    a_mat = SgT::D1, b_mat = SgT::X, out = SgLayout::W1;
  } else {
    o0 = 0, i0 = (tile - 36) * 64, fin = RL_SG_H;
    a_mat = SgT::DO, b_mat = SgT::A3, out = SgLayout::W4;
  }
  const bool head = a_mat == SgT::DO;  // two columns of dz, the tile's others are zeros
  const int aw = head ? RL_SGT_DO : RL_SG_H;
  const int kbeg = slice * sp.kchunk, kend = min(ld, kbeg + sp.kchunk);
  // the slice's rows through buffer resources: rows past its end read as zeros
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(T + (size_t)a_mat * ld + (size_t)kbeg * aw + o0), (short)0, ((kend - kbeg) * aw - o0) * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(T + (size_t)b_mat * ld + (size_t)kbeg * fin + i0), (short)0, ((kend - kbeg) * fin - i0) * 2, 0x00020000);
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  sg_float4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sg_float4{0.f, 0.f, 0.f, 0.f};
  // a stage: rows r and r + 32 of both operands, 8 values per load
  const int r = tid >> 3, c8 = (tid & 7) * 8;
  const unsigned oa = head && c8 ? 0x80000000u : (unsigned)(r * aw + c8) * 2u, ob = (unsigned)(r * fin + c8) * 2u;
  uint4 va[RL_SGT_AHEAD][2], vb[RL_SGT_AHEAD][2];
  auto fetch = [&](int k0, uint4 (&fa)[2], uint4 (&fb)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      fa[h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ra, oa + (unsigned)((k0 + 32 * h) * aw) * 2u, 0, 0));
      fb[h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rb, ob + (unsigned)((k0 + 32 * h) * fin) * 2u, 0, 0));
    }
  };
#pragma unroll
  for (int s = 0; s < RL_SGT_AHEAD; ++s) {
    fetch(64 * s, va[s], vb[s]);
    __builtin_amdgcn_sched_barrier(0);  // in order: the first stage's wait must not cover the later ones' loads
  }
  // whole groups of stages (past the slice they add zeros), so that each stage
  // waits for its own loads only.  One barrier per stage: a buffer is written again only after the barrier
  // that follows the other buffer's writes, which every wave reaches after it
  // has read this one
  for (int k0 = 0; k0 < kend - kbeg; k0 += 64 * RL_SGT_AHEAD) {
#pragma unroll
    for (int s = 0; s < RL_SGT_AHEAD; ++s) {
      bf16_t *as = As[s & 1], *bs = Bs[s & 1];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        *(uint4*)(as + (r + 32 * h) * RL_SGT_PAD + c8) = va[s][h];
        *(uint4*)(bs + (r + 32 * h) * RL_SGT_PAD + c8) = vb[s][h];
      }
      fetch(k0 + 64 * (s + RL_SGT_AHEAD), va[s], vb[s]);
      __syncthreads();
#pragma unroll
      for (int ks = 0; ks < 64; ks += 32) {
        sg_bf16x8 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) a[i] = sgt_frag(as, ks, wm + i * 16, lane);
#pragma unroll
        for (int j = 0; j < 2; ++j) b[j] = sgt_frag(bs, ks, wn + j * 16, lane);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
      }
    }
  }
  // act first: lane l holds row o = l & 15 of a tile, columns 4 (l >> 4) .. + 3
  float* dst = part + (size_t)slice * RL_SGT_PART + out;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int o = o0 + wm + i * 16 + (lane & 15);
    if (!head || o < RL_SG_OUT)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        *(sg_float4*)(dst + (size_t)o * fin + i0 + wn + j * 16 + 4 * (lane >> 4)) = acc[i][j];
  }
}

// Sums of the gradient partials in slice / chunk order (SUM) into grad, and the
// Adam step with it (ADAM; without SUM, with the gradient grad holds), which
// writes the bf16 copies as well.  One thread per parameter.
template <bool SUM, bool ADAM>
__global__ __launch_bounds__(256) void k_sg_update(const float* __restrict__ part, const float* __restrict__ bpart, int nz,
                                                   int ncz, float* __restrict__ grad, float* __restrict__ p,
                                                   float* __restrict__ m1, float* __restrict__ m2,
                                                   bf16_t* __restrict__ pb, bf16_t* __restrict__ pf, float lr, float b1,
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
    const size_t stride = bias < 0 ? RL_SGT_PART : RL_SGT_BIAS;
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
    sg_store_bf16(i, v, pb, pf);
  }
}
