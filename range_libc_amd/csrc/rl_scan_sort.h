// Device-wide exclusive sum of 64-bit counts and per-segment ascending sort of
// float keys, used by the CDDT table build (bin offsets from bin counts, then
// each bin's entries in order).
//
// Included by rl_cddt_impl.h (uses rl_lib.hip's fail/TRY/HIP_TRY and DevBuf).
//
// Scan: tiles of 2048 counts (256 threads x 8 consecutive items); pass 1 sums
// each tile, pass 2 (one workgroup) turns the tile sums into tile offsets,
// pass 3 rescans each tile from its offset.  Wave scans use 64-lane shuffles.
//
// Sort: floats are sorted by their order-preserving unsigned keys (sign bit
// set: all bits inverted; clear: sign bit set), the order of a radix sort of
// float bit patterns (-0 before +0).  Segments of up to 512 keys are sorted by
// one wave each in registers, up to 2048 by a 256-thread workgroup in LDS, up to 16384 by a
// 1024-thread workgroup (64 KiB of LDS), all with bitonic networks over the
// segment padded to a power of two with the largest key; longer segments
// (maps far above 4096 cells a side) are sorted in global memory, one
// bitonic stage per launch.

#define RL_SCAN_ITEMS 8
#define RL_SCAN_BLOCK 256
#define RL_SCAN_TILE (RL_SCAN_ITEMS * RL_SCAN_BLOCK)

__device__ __forceinline__ unsigned long long wave_incl_scan_u64(unsigned long long v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned long long o = __shfl_up(v, (unsigned)d, 64);
    if (lane >= d) v += o;
  }
  return v;
}

// Exclusive scan of one value per thread over a RL_SCAN_BLOCK-thread block;
// *total receives the block's sum.  Every thread of the block must call it.
__device__ __forceinline__ unsigned long long block_excl_scan_u64(unsigned long long v, unsigned long long* wsum,
                                                                  unsigned long long* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned long long inc = wave_incl_scan_u64(v);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  unsigned long long off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < RL_SCAN_BLOCK / 64; ++i) {
    const unsigned long long s = wsum[i];
    off += (i < w) ? s : 0ull;
    tot += s;
  }
  __syncthreads();  // wsum is rewritten by the next call
  *total = tot;
  return off + inc - v;
}

__global__ void __launch_bounds__(RL_SCAN_BLOCK) k_scan_tiles(const unsigned long long* __restrict__ in, long long n,
                                                              unsigned long long* __restrict__ tile_sum) {
  __shared__ unsigned long long wsum[RL_SCAN_BLOCK / 64];
  const long long base = (long long)blockIdx.x * RL_SCAN_TILE + (long long)threadIdx.x * RL_SCAN_ITEMS;
  unsigned long long s = 0;
#pragma unroll
  for (int k = 0; k < RL_SCAN_ITEMS; ++k) s += (base + k < n) ? in[base + k] : 0ull;
  unsigned long long tot;
  (void)block_excl_scan_u64(s, wsum, &tot);
  if (threadIdx.x == 0) tile_sum[blockIdx.x] = tot;
}

// One workgroup: tile_sum[0..nt) becomes its own exclusive prefix sum.
__global__ void __launch_bounds__(RL_SCAN_BLOCK) k_scan_spine(unsigned long long* __restrict__ tile_sum, long long nt) {
  __shared__ unsigned long long wsum[RL_SCAN_BLOCK / 64];
  unsigned long long carry = 0;
  for (long long b0 = 0; b0 < nt; b0 += RL_SCAN_TILE) {
    const long long base = b0 + (long long)threadIdx.x * RL_SCAN_ITEMS;
    unsigned long long v[RL_SCAN_ITEMS], s = 0;
#pragma unroll
    for (int k = 0; k < RL_SCAN_ITEMS; ++k) {
      v[k] = (base + k < nt) ? tile_sum[base + k] : 0ull;
      s += v[k];
    }
    unsigned long long tot;
    unsigned long long ex = block_excl_scan_u64(s, wsum, &tot) + carry;
#pragma unroll
    for (int k = 0; k < RL_SCAN_ITEMS; ++k) {
      if (base + k < nt) tile_sum[base + k] = ex;
      ex += v[k];
    }
    carry += tot;
  }
}

__global__ void __launch_bounds__(RL_SCAN_BLOCK) k_scan_out(const unsigned long long* __restrict__ in, long long n,
                                                            const unsigned long long* __restrict__ tile_off,
                                                            unsigned long long* __restrict__ out) {
  __shared__ unsigned long long wsum[RL_SCAN_BLOCK / 64];
  const long long base = (long long)blockIdx.x * RL_SCAN_TILE + (long long)threadIdx.x * RL_SCAN_ITEMS;
  unsigned long long v[RL_SCAN_ITEMS], s = 0;
#pragma unroll
  for (int k = 0; k < RL_SCAN_ITEMS; ++k) {
    v[k] = (base + k < n) ? in[base + k] : 0ull;
    s += v[k];
  }
  unsigned long long tot;
  unsigned long long ex = block_excl_scan_u64(s, wsum, &tot) + tile_off[blockIdx.x];
#pragma unroll
  for (int k = 0; k < RL_SCAN_ITEMS; ++k) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
}

// out[i] = in[0] + ... + in[i - 1] for i < n, on the stream; `tiles` is scratch
// for one call.
int exclusive_sum_u64(hipStream_t st, const unsigned long long* in, unsigned long long* out, long long n,
                      DevBuf* tiles) {
  if (n <= 0) return RL_OK;
  const long long nt = (n + RL_SCAN_TILE - 1) / RL_SCAN_TILE;
  if (nt > 0x7fffffffLL) return fail(RL_ERR_ARG, "scan: %lld items is too many", n);
  TRY(tiles->alloc((size_t)nt * sizeof(unsigned long long)));
  hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)nt), dim3(RL_SCAN_BLOCK), 0, st, in, n,
                     tiles->as<unsigned long long>());
  hipLaunchKernelGGL(k_scan_spine, dim3(1), dim3(RL_SCAN_BLOCK), 0, st, tiles->as<unsigned long long>(), nt);
  hipLaunchKernelGGL(k_scan_out, dim3((unsigned)nt), dim3(RL_SCAN_BLOCK), 0, st, in, n,
                     (const unsigned long long*)tiles->p, out);
  HIP_TRY(hipGetLastError());
  return RL_OK;
}

__device__ __forceinline__ unsigned sort_key(float f) {
  const unsigned u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float sort_key_value(unsigned k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Ascending bitonic sort of s[0..P) in LDS, P a power of two >= 2, by the
// workgroup's threads tid = 0..nt-1.
__device__ __forceinline__ void bitonic_lds(unsigned* s, int P, int tid, int nt) {
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = tid; i < (P >> 1); i += nt) {
        const int a = ((i & ~(j - 1)) << 1) | (i & (j - 1)), b = a + j;
        const unsigned x = s[a], y = s[b];
        if ((x > y) == ((a & k) == 0)) {
          s[a] = y;
          s[b] = x;
        }
      }
      __syncthreads();
    }
}

__device__ __forceinline__ int pow2_at_least(long long n) {
  int p = 2;
  while (p < n) p <<= 1;
  return p;
}

#define RL_SORT_WAVE_MAX 512
#define RL_SORT_MID_MAX 2048
#define RL_SORT_BIG_MAX 16384

// Ascending bitonic sort of 64 E keys by one wave, key e of lane l being element
// l E + e: stages between elements of one lane are min / max of its registers,
// stages between lanes one exchange per register.
template <int E>
__device__ __forceinline__ void bitonic_regs(unsigned (&r)[E], int lane) {
#pragma unroll
  for (int k = 2; k <= 64 * E; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (j >= E) {
        // elements l E + e and (l ^ d) E + e; ascending where bit k of the element
        // is clear (k > j >= E: a bit of the lane, or none when k is all of them)
        const int d = j / E;
        const bool keep_min = ((lane & d) == 0) == ((lane & (k / E)) == 0);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const unsigned o = (unsigned)__shfl_xor((int)r[e], d);
          r[e] = keep_min ? min(r[e], o) : max(r[e], o);
        }
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          if (e & j) continue;
          const bool up = k < E ? (e & k) == 0 : (lane & (k / E)) == 0;
          const unsigned lo = min(r[e], r[e | j]), hi = max(r[e], r[e | j]);
          r[e] = up ? lo : hi;
          r[e | j] = up ? hi : lo;
        }
      }
    }
  }
}

template <int E>
__device__ __forceinline__ void sort_wave(const float* __restrict__ in, float* __restrict__ out, int n, int lane) {
  unsigned r[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {  // (any order will do: the loads take consecutive elements)
    const int i = e * 64 + lane;
    r[e] = i < n ? sort_key(in[i]) : 0xffffffffu;
  }
  bitonic_regs<E>(r, lane);
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (lane * E + e < n) out[lane * E + e] = sort_key_value(r[e]);
}

// Segments of at most RL_SORT_WAVE_MAX keys, one wave each (4 per workgroup);
// longer segments are left to the other kernels.  32.9 M keys in 140,000
// segments of up to 512: 204 us (a wave sorting at most 256 in LDS, workgroups
// the others: 120 + 490 us).
__global__ void __launch_bounds__(256) k_seg_sort_wave(const float* __restrict__ in, float* __restrict__ out,
                                                       const long long* __restrict__ start, long long nseg) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long seg = (long long)blockIdx.x * 4 + w;
  if (seg >= nseg) return;
  const long long b = start[seg], n = start[seg + 1] - b;
  if (n > RL_SORT_WAVE_MAX || n <= 0) return;
  if (n <= 64)
    sort_wave<1>(in + b, out + b, (int)n, lane);
  else if (n <= 128)
    sort_wave<2>(in + b, out + b, (int)n, lane);
  else if (n <= 256)
    sort_wave<4>(in + b, out + b, (int)n, lane);
  else
    sort_wave<8>(in + b, out + b, (int)n, lane);
}

// Workgroups of NT threads over the listed segments (at most MAXN keys each).
template <int NT, int MAXN>
__global__ void __launch_bounds__(NT) k_seg_sort_block(const float* __restrict__ in, float* __restrict__ out,
                                                       const long long* __restrict__ start,
                                                       const unsigned* __restrict__ list,
                                                       const unsigned* __restrict__ count) {
  __shared__ unsigned s[MAXN];
  for (unsigned l = blockIdx.x; l < *count; l += gridDim.x) {  // the same in every thread
    const long long seg = list[l];
    const long long b = start[seg], n = start[seg + 1] - b;
    const int P = pow2_at_least(n);
    for (int i = threadIdx.x; i < P; i += NT) s[i] = (i < n) ? sort_key(in[b + i]) : 0xffffffffu;
    __syncthreads();
    bitonic_lds(s, P, threadIdx.x, NT);
    for (int i = threadIdx.x; i < n; i += NT) out[b + i] = sort_key_value(s[i]);
    __syncthreads();  // stored before the next segment is loaded
  }
}

// Lists the segments longer than RL_SORT_WAVE_MAX by size class: class 0
// (<= RL_SORT_MID_MAX), 1 (<= RL_SORT_BIG_MAX), 2 (longer).  One atomic per
// wave and class.
__global__ void __launch_bounds__(256) k_seg_classify(const long long* __restrict__ start, long long nseg,
                                                      unsigned* __restrict__ lists, unsigned* __restrict__ counts) {
  const long long seg = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long n = 0;
  if (seg < nseg) n = start[seg + 1] - start[seg];
  const int cls = n <= RL_SORT_WAVE_MAX ? -1 : (n <= RL_SORT_MID_MAX ? 0 : (n <= RL_SORT_BIG_MAX ? 1 : 2));
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const unsigned long long m = __ballot(cls == c);
    if (!m) continue;
    const int leader = __builtin_ctzll(m);
    unsigned base = 0;
    if (lane == leader) base = atomicAdd(&counts[c], (unsigned)__popcll(m));
    base = __shfl(base, leader, 64);
    if (cls == c) lists[(size_t)c * (size_t)nseg + base + (unsigned)__popcll(m & ((1ull << lane) - 1ull))] = (unsigned)seg;
  }
}

__global__ void k_sort_global_load(const float* __restrict__ in, unsigned* __restrict__ keys, long long n, long long P) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < P) keys[i] = (i < n) ? sort_key(in[i]) : 0xffffffffu;
}
__global__ void k_sort_global_step(unsigned* __restrict__ keys, long long P, long long j, long long k) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (P >> 1)) return;
  const long long a = ((i & ~(j - 1)) << 1) | (i & (j - 1)), b = a + j;
  const unsigned x = keys[a], y = keys[b];
  if ((x > y) == ((a & k) == 0)) {
    keys[a] = y;
    keys[b] = x;
  }
}
__global__ void k_sort_global_store(const unsigned* __restrict__ keys, float* __restrict__ out, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = sort_key_value(keys[i]);
}

// out[start[s] .. start[s + 1]) = in[start[s] .. start[s + 1]) sorted ascending,
// for every segment s < nseg (start on the device, nseg + 1 entries, nseg < 2^32);
// `lists` is scratch for one call.  Waits for the stream only to learn whether
// a segment is left to the global-memory sort.
int segmented_sort_f32(hipStream_t st, const float* in, float* out, const long long* start, long long nseg,
                       DevBuf* lists) {
  if (nseg <= 0) return RL_OK;
  if (nseg >= 0xffffffffLL) return fail(RL_ERR_ARG, "sort: %lld segments is too many", nseg);
  hipLaunchKernelGGL(k_seg_sort_wave, dim3((unsigned)((nseg + 3) / 4)), dim3(256), 0, st, in, out, start, nseg);
  TRY(lists->alloc((4 + (size_t)nseg * 3) * sizeof(unsigned)));
  unsigned* counts = lists->as<unsigned>();  // 4, then the three lists
  const unsigned* L = counts + 4;
  HIP_TRY(hipMemsetAsync(counts, 0, 4 * sizeof(unsigned), st));
  hipLaunchKernelGGL(k_seg_classify, dim3((unsigned)((nseg + 255) / 256)), dim3(256), 0, st, start, nseg, counts + 4,
                     counts);
  hipLaunchKernelGGL((k_seg_sort_block<256, RL_SORT_MID_MAX>), dim3((unsigned)std::min<long long>(nseg, 1024)), dim3(256),
                     0, st, in, out, start, L, (const unsigned*)counts);
  hipLaunchKernelGGL((k_seg_sort_block<1024, RL_SORT_BIG_MAX>), dim3((unsigned)std::min<long long>(nseg, 512)), dim3(1024),
                     0, st, in, out, start, L + nseg, (const unsigned*)counts + 1);
  HIP_TRY(hipGetLastError());
  unsigned* cnt;
  TRY(lists->c->pinned((void**)&cnt));
  HIP_TRY(hipMemcpyAsync(cnt, counts, 4 * sizeof(unsigned), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  if (cnt[2]) {
    std::vector<unsigned> big(cnt[2]);
    std::vector<long long> se(2);
    HIP_TRY(hipMemcpyAsync(big.data(), L + 2 * nseg, big.size() * sizeof(unsigned), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    for (unsigned s : big) {
      HIP_TRY(hipMemcpy(se.data(), start + s, 2 * sizeof(long long), hipMemcpyDeviceToHost));
      const long long b = se[0], n = se[1] - se[0];
      long long P = 2;
      while (P < n) P <<= 1;
      DevBuf keys(lists->c);
      TRY(keys.alloc((size_t)P * sizeof(unsigned)));
      const unsigned gp = (unsigned)((P + 255) / 256), gh = (unsigned)((P / 2 + 255) / 256);
      hipLaunchKernelGGL(k_sort_global_load, dim3(gp), dim3(256), 0, st, in + b, keys.as<unsigned>(), n, P);
      for (long long k = 2; k <= P; k <<= 1)
        for (long long j = k >> 1; j > 0; j >>= 1)
          hipLaunchKernelGGL(k_sort_global_step, dim3(gh), dim3(256), 0, st, keys.as<unsigned>(), P, j, k);
      hipLaunchKernelGGL(k_sort_global_store, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                         (const unsigned*)keys.p, out + b, n);
      HIP_TRY(hipGetLastError());
    }
  }
  return RL_OK;
}
