// CDDTCast / PCDDT (RangeLib.h:971-1770) built on the GPU.
//
// Included at the end of rl_lib.hip (uses its types and helpers).  The query
// is rl::cddt_calc_range in rl_device.h; this file builds and prunes the
// tables:
//   1. per-angle constants (one thread per angle, the library's sinf/cosf);
//   2. edge cells (occupied with a free 8-neighbour, OMap::make_edge_map);
//   3. every (edge cell, angle < td/2) pair projects the cell centre into the
//      bins its footprint covers: a counting pass (in LDS, in memory for the widest
//      maps), an exclusive scan into bin offsets, and a filling pass;
//   4. each bin sorted (segmented bitonic sort, rl_scan_sort.h) and its
//      duplicates dropped;
//   5. prune: the entries that a query from some free cell can return are found by
//      intervals between entries, the others are dropped.
// The result equals the reference's compressed_lut bin for bin: the order in
// which entries arrive does not matter after sorting and deduplication.

#define RL_CDDT_EPS 0.00001

// 1. Constants of angle a (RangeLib.h:991-1058).
__global__ void k_cddt_consts(TrigDev trig, int td, int W, int H, float m2pi_div_td, int* __restrict__ width,
                              float* __restrict__ trans, float* __restrict__ cosv, float* __restrict__ sinv) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= td) return;
  const float angle = (float)a * m2pi_div_td;
  float sn, cs;
  rl::sincos_libc(angle, trig, &sn, &cs);
  cosv[a] = cs;
  sinv[a] = sn;
  const float rotated_height = fabsf((float)W * sn) + fabsf((float)H * cs);
  width[a] = (int)(unsigned)ceil((double)rotated_height - RL_CDDT_EPS);
  const float lt = (float)H * cs, rt = (float)W * sn + (float)H * cs, rb = (float)W * sn;
  const float m2 = (rb < rt) ? rb : rt;  // std::min(rt, rb)
  const float mn = (m2 < lt) ? m2 : lt;  // std::min(lt, ...)
  const double t = -1.0 * (double)mn - RL_CDDT_EPS;
  trans[a] = (float)(t > 0.0 ? t : 0.0);  // std::max(0.0, t)
}

// Bin offsets of the angles (one workgroup of 1024): exclusive sums of the
// widths, and the build's sizes into pinned memory.
struct CddtSizes {
  long long nb, nba;  // bins of all angles, of the first nang
  unsigned ne, occupied;  // edge cells, occupied cells
  int max_width;
};
__global__ __launch_bounds__(1024) void k_cddt_offsets(const int* __restrict__ width, int td, int nang,
                                                       const unsigned long long* __restrict__ n_edges,
                                                       long long* __restrict__ off,
                                                       CddtSizes* __restrict__ out) {
  __shared__ long long sum[1024];
  __shared__ int top[1024];
  const int t = threadIdx.x, per = (td + 1023) / 1024;
  const int a0 = min(td, t * per), a1 = min(td, a0 + per);
  long long s = 0;
  int mw = 0;
  for (int a = a0; a < a1; ++a) s += width[a], mw = max(mw, width[a]);
  sum[t] = s;
  top[t] = mw;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {  // inclusive sums and maxima
    const long long o = t >= d ? sum[t - d] : 0;
    const int q = t >= d ? top[t - d] : 0;
    __syncthreads();
    sum[t] += o;
    top[t] = max(top[t], q);
    __syncthreads();
  }
  long long run = sum[t] - s;
  for (int a = a0; a < a1; ++a) {
    off[a] = run;
    if (a == nang) out->nba = run;
    run += width[a];
  }
  if (t == 1023) {
    off[td] = sum[t];
    out->nb = sum[t];
    out->ne = (unsigned)*n_edges;
    out->occupied = (unsigned)(*n_edges >> 32);
    out->max_width = top[t];
    if (nang == td) out->nba = sum[t];
  }
}

// 2. Edge cells as (x << 16) | y (sides are below 65536), in any order, their number
// in the low half of *n_out and that of the occupied cells in the high half.  A
// workgroup gathers the edge cells of 4096 in LDS and takes their place in the
// list with one atomic: with one per wave, 65,536 atomics on one address took
// 0.65 ms for a 2048^2 map; 0.04 so.
#define RL_CDDT_EDGE_ITEMS 16
__global__ __launch_bounds__(256) void k_cddt_edges(const uint8_t* __restrict__ occ, int W, int H,
                                                    unsigned* __restrict__ list, unsigned long long* __restrict__ n_out) {
  __shared__ unsigned found[256 * RL_CDDT_EDGE_ITEMS];
  __shared__ unsigned cnt, base, occupied;
  if (threadIdx.x == 0) cnt = occupied = 0;
  __syncthreads();
  const unsigned n = (unsigned)W * (unsigned)H;  // < 2^31 (checked by the caller)
  const unsigned first = blockIdx.x * (256 * RL_CDDT_EDGE_ITEMS) + threadIdx.x;
  const int lane = threadIdx.x & 63;
  unsigned full = 0;  // occupied cells of the wave
  for (int k = 0; k < RL_CDDT_EDGE_ITEMS; ++k) {
    const unsigned i = first + (unsigned)k * 256u;
    const bool o = i < n && occ[i];
    full += (unsigned)__popcll(__ballot(o));
    bool e = false;
    int x = 0, y = 0;
    if (o) {
      x = (int)(i / (unsigned)H), y = (int)(i - (unsigned)x * (unsigned)H);
      const uint8_t* c = occ + i;
      const bool l = x > 0, r = x + 1 < W, d = y > 0, u = y + 1 < H;
      e = (r && !c[H]) || (l && !*(c - H)) || (u && !c[1]) || (d && !*(c - 1)) || (r && u && !c[H + 1]) ||
          (l && u && !*(c - H + 1)) || (r && d && !c[H - 1]) || (l && d && !*(c - H - 1));
    }
    const unsigned long long m = __ballot(e);
    unsigned at = 0;
    if (lane == 0 && m) at = atomicAdd(&cnt, (unsigned)__popcll(m));
    at = __shfl(at, 0);
    if (e) found[at + __popcll(m & ((1ull << lane) - 1ull))] = ((unsigned)x << 16) | (unsigned)y;
  }
  if (lane == 0) atomicAdd(&occupied, full);
  __syncthreads();
  if (threadIdx.x == 0) base = (unsigned)atomicAdd(n_out, (unsigned long long)occupied << 32 | cnt);
  __syncthreads();
  for (unsigned i = threadIdx.x; i < cnt; i += 256) list[base + i] = found[i];
}

// Footprint of an edge cell at angle a (RangeLib.h:1096-1115): the projected
// centre and the bins [lower, upper] it is stored in.
struct CddtProj {
  float cx;
  int lower, upper;
};
__device__ __forceinline__ CddtProj cddt_project(unsigned cell, float cs, float sn, float tr) {
  const float px = (float)(cell >> 16) + 0.5f, py = (float)(cell & 0xffffu) + 0.5f;  // exact
  const float half = (float)((double)(fabsf(sn) + fabsf(cs)) / 2.0);
  CddtProj p;
  p.cx = px * cs - py * sn;
  const float cy = (px * sn + py * cs) + tr;
  p.upper = (int)((double)(cy + half) - RL_CDDT_EPS);
  p.lower = (int)((double)(cy - half) + RL_CDDT_EPS);
  return p;
}

// 3. Counting (FILL == false) and filling (FILL == true) passes over the (edge
// cell, angle) pairs.  A workgroup takes one angle and one of G chunks of the
// edge list and counts into the angle's bins in LDS (up to RL_CDDT_LDS_BINS of
// them): the first pass stores the chunk's counts, k_cddt_chunks turns them into
// each chunk's offsets in the bins, and the second pass starts its LDS cursors
// there.  All chunks of an angle run on one XCD (workgroup b is on XCD b mod 8),
// so an angle's entries, about 1 MB at 2048^2, are put together in its L2.
// 2048^2 corridor map, 54 headings, 32.9 M entries: 1.00 + 1.19 ms with an atomic
// on a 64-bit counter in memory per entry and pass; 0.05 + 0.27 so.
// Bins outside [0, width) are skipped (the reference would write outside its
// table; it does not happen for maps whose edge cells project inside the
// rotated bounding box, which the translation and width are built to cover).
#define RL_CDDT_LDS_BINS 16384  // 64 KB: maps of up to about 11,500 cells a side
template <bool FILL>
__global__ __launch_bounds__(256) void k_cddt_hist(const unsigned* __restrict__ edges, int n_edges, int nang, int G,
                                                   const int* __restrict__ width, const float* __restrict__ trans,
                                                   const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                   const long long* __restrict__ bin_off,
                                                   const long long* __restrict__ start, unsigned* __restrict__ chunks,
                                                   long long nb, float* __restrict__ vals) {
  extern __shared__ unsigned bins[];
  const int k = (int)(blockIdx.x >> 3);
  const int a = (int)(blockIdx.x & 7) + 8 * (k / G), g = k % G;
  if (a >= nang) return;  // the same in every thread
  const int w = width[a];
  const long long off = bin_off[a];
  unsigned* mine = chunks + (size_t)g * (size_t)nb + off;
  for (int b = threadIdx.x; b < w; b += 256) bins[b] = FILL ? (unsigned)start[off + b] + mine[b] : 0u;
  __syncthreads();
  const float cs = cosv[a], sn = sinv[a], tr = trans[a];
  const int per = (n_edges + G - 1) / G, e0 = g * per, e1 = min(n_edges, e0 + per);
  for (int e = e0 + (int)threadIdx.x; e < e1; e += 256) {
    const CddtProj p = cddt_project(edges[e], cs, sn, tr);
    for (int b = p.lower; b <= p.upper; ++b) {
      if (b < 0 || b >= w) continue;
      const unsigned pos = atomicAdd(&bins[b], 1u);
      if (FILL) vals[pos] = p.cx;
    }
  }
  if (FILL) return;
  __syncthreads();
  for (int b = threadIdx.x; b < w; b += 256) mine[b] = bins[b];
}

// Per bin (the first nba of nb): the chunks' counts become their offsets in the
// bin, their sum the bin's count.
__global__ __launch_bounds__(256) void k_cddt_chunks(unsigned* __restrict__ chunks, int G, long long nb,
                                                     unsigned long long* __restrict__ counts, long long nba) {
  const long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nba) return;
  unsigned s = 0;
  for (int g = 0; g < G; ++g) {
    const unsigned c = chunks[(size_t)g * (size_t)nb + b];
    chunks[(size_t)g * (size_t)nb + b] = s;
    s += c;
  }
  counts[b] = s;
}

// The same passes for maps whose angles have more bins than LDS holds: one
// thread per (edge cell, angle a0 + blockIdx.y), counting in memory.
template <bool FILL>
__global__ __launch_bounds__(256) void k_cddt_scatter(const unsigned* __restrict__ edges, int n_edges, int a0,
                                                      const int* __restrict__ width, const float* __restrict__ trans,
                                                      const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                      const long long* __restrict__ bin_off,
                                                      unsigned long long* __restrict__ counter,
                                                      float* __restrict__ vals) {
  const int e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (e >= n_edges) return;
  const int a = a0 + (int)blockIdx.y;
  const CddtProj p = cddt_project(edges[e], cosv[a], sinv[a], trans[a]);
  for (int b = p.lower; b <= p.upper; ++b) {
    if (b < 0 || b >= width[a]) continue;
    const unsigned long long pos = atomicAdd(&counter[bin_off[a] + b], 1ull);
    if (FILL) vals[pos] = p.cx;
  }
}

// 4./5. One wave per bin: count the entries kept (COPY == false) or copy them to
// their new place (COPY == true).  mode 0 keeps the first of each run of equal
// values (after sorting), mode 1 keeps the entries marked used.  Lanes take
// consecutive entries, so a bin's loads are whole lines (one thread per bin read
// 4 bytes of a line at a time: 0.47 and 0.95 ms on the 2048^2 corridor map with 108
// headings; 0.07 and 0.08 ms so).
template <bool COPY>
__global__ __launch_bounds__(256) void k_cddt_compact(long long nb, const long long* __restrict__ start,
                                                      const float* __restrict__ vals, const uint8_t* __restrict__ used,
                                                      int mode, const long long* __restrict__ new_start,
                                                      long long* __restrict__ kept, float* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  for (long long b = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); b < nb; b += (long long)gridDim.x * 4) {
    const long long s = start[b], e = start[b + 1];
    long long o = COPY ? new_start[b] : 0;
    for (long long j0 = s; j0 < e; j0 += 64) {
      const long long j = j0 + lane;
      bool keep = false;
      float v = 0.0f;
      if (j < e) {
        v = vals[j];
        keep = mode == 0 ? (j == s || v != vals[j - 1]) : used[j] != 0;
      }
      const unsigned long long m = __ballot(keep);
      if (COPY && keep) out[o + __popcll(m & ((1ull << lane) - 1ull))] = v;
      o += __popcll(m);
    }
    if (!COPY && lane == 0) kept[b] = o;
  }
}

// 5. Prune marks (RangeLib.h:1172-1275).  In the reference every free cell looks
// up its bin under every angle and marks the entries around it: the first entry
// at or beyond its projection and the one before (where the reference's linear
// search leaves its index unset, the lower_bound value is taken, as its binary
// search; past the last entry that entry is marked whatever max_range is).  So
// entry i is used exactly when a free cell of the bin's strip projects into
// (v[i - 1], v[i]] or (v[i], v[i + 1]] (unbounded at the ends), and one such cell
// per interval is enough: a lane takes an interval and walks the cells of the
// strip that can project into it until it finds a free one.  The walk's bounds
// are real geometry with a margin far above float rounding; a cell counts only
// if its own float projection (the reference's expressions) falls in the bin and
// the interval.  2048^2 corridor map, 108 headings: one lookup
// (binary search) per cell and angle, 226 M of them, took 4.65 ms; 0.46 so
// (0.96 with every lane walking its interval to the end).
// SOLID, for maps whose occupied cells are mostly inside blocks (cddt_solid): a walk
// through a block skips its solid 8 x 8 tiles by the occupancy bitmap.  2048^2, 108
// headings, call times: rooms in solid ground 2.11 -> 0.54 ms (one lookup per free cell
// and angle: 0.52), half the map solid 1.38 -> 0.35 (1.08), a block in an open map 1.04 ->
// 0.35 (1.94); the corridor map, which takes the other, 0.57 -> 0.61 (7.2).
// One wave per bin, angle blockIdx.y; used[i] of every entry is written, and the
// bin's number of used entries.
template <bool SOLID>
__global__ __launch_bounds__(256) void k_cddt_prune_mark(const uint8_t* __restrict__ occ, int W, int H,
                                                         const unsigned long long* __restrict__ bits, int ntx, int nty,
                                                         const int* __restrict__ width, const float* __restrict__ trans,
                                                         const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                         const long long* __restrict__ bin_off,
                                                         const long long* __restrict__ start,
                                                         const float* __restrict__ vals, uint8_t* __restrict__ used,
                                                         long long* __restrict__ kept, int a0) {
  const int a = a0 + (int)blockIdx.y;
  const unsigned li = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (li >= (unsigned)width[a]) return;
  const long long b = bin_off[a] + li, s = start[b];
  const int n = (int)(start[b + 1] - s);  // fewer than 2^31 entries in all (checked at build)
  if (n == 0) {
    if (lane == 0) kept[b] = 0;
    return;
  }
  const float* v = vals + s;
  const float cs = cosv[a], sn = sinv[a], tr = trans[a];
  // a cell centre (fx, fy) is at lx = fx cs - fy sn along the strip and l = fx sn +
  // fy cs across it, l in [l0, l1) up to rounding; fx = lx cs + l sn, fy = l cs - lx sn
  const float mg = 0.05f + 4.0e-6f * (float)(W + H);
  // (bin 0 also takes the projections that truncate to it from (-1, 0))
  const float l0 = (li ? (float)li : -1.0f) - tr - mg, l1 = (float)li - tr + 1.0f + mg;
  // p: the axis along which the strip advances fastest, q the other; np, nq their
  // sizes.  l = fp * kp + fq * kq with |kq| >= 0.7
  const bool along_x = fabsf(cs) >= fabsf(sn);
  const float kp = along_x ? sn : cs, kq = along_x ? cs : sn;
  const int np = along_x ? W : H, nq = along_x ? H : W;
  const float inv_kq = 1.0f / kq;
  // positions p for which the strip crosses the map: fp in [0, np], fp * kp = l - fq * kq
  float pmin = 0.0f, pmax = (float)np;
  if (fabsf(kp) > 1.0e-3f) {
    const float e = (float)nq * kq;
    const float u = l0 - fmaxf(e, 0.0f), w = l1 - fminf(e, 0.0f);
    const float r0 = u / kp, r1 = w / kp;
    pmin = fmaxf(pmin, fminf(r0, r1) - 1.0f);
    pmax = fminf(pmax, fmaxf(r0, r1) + 1.0f);
  }
  // lx's part of fp: along x fp = lx cs + l sn, along y fp = -lx sn + l cs
  const float kx = along_x ? cs : -sn, kl = along_x ? sn : cs;
  const float lmin = fminf(l0 * kl, l1 * kl) - mg, lmax = fmaxf(l0 * kl, l1 * kl) + mg;
  // whether a free cell at position p of the strip projects into (lo, hi]
  auto column = [&](int p, float lo, float hi) {
    const float fp = (float)p + 0.5f;
    const float c0 = (l0 - fp * kp) * inv_kq, c1 = (l1 - fp * kp) * inv_kq;
    const int q0 = max(0, (int)ceilf(fminf(c0, c1) - 0.5f)), q1 = min(nq - 1, (int)floorf(fmaxf(c0, c1) - 0.5f));
    for (int q = q0; q <= q1; ++q) {
      const int x = along_x ? p : q, y = along_x ? q : p;
      const float fx = (float)x + 0.5f, fy = (float)y + 0.5f;  // (exact, as the reference's 0.5 + x in double)
      const float lx = fx * cs - fy * sn;
      const float ly = (fx * sn + fy * cs) + tr;
      if (lx > lo && lx <= hi && (unsigned)rl::trunc_x86(ly) == li && !occ[(size_t)x * (unsigned)H + (unsigned)y])
        return true;
    }
    return false;
  };
  // whether the bitmap's tiles under the strip at positions p0 .. p0 + 7 (p0 a
  // multiple of 8) have no free cell.  (Each bound of a column's cells is monotone in
  // the position, rounding included, so the ends' bounds hold all eight columns'.)
  const unsigned long long* row0 = bits + (along_x ? 0 : (size_t)ntx * nty);
  const int nt = along_x ? nty : ntx;
  auto solid = [&](int p0) {
    if (p0 >= np) return true;
    const float fa = (float)p0 + 0.5f, fb = (float)(p0 + 7) + 0.5f;
    const float a0 = (l0 - fa * kp) * inv_kq, a1 = (l1 - fa * kp) * inv_kq;
    const float b0 = (l0 - fb * kp) * inv_kq, b1 = (l1 - fb * kp) * inv_kq;
    const int q0 = max(0, (int)ceilf(fminf(fminf(a0, a1), fminf(b0, b1)) - 0.5f));
    const int q1 = min(nq - 1, (int)floorf(fmaxf(fmaxf(a0, a1), fmaxf(b0, b1)) - 0.5f));
    unsigned long long t = ~0ull;
    for (int q = q0 >> 3; q <= q1 >> 3; ++q) t &= row0[(size_t)(p0 >> 3) * (unsigned)nt + q];
    return t == ~0ull;
  };
  __shared__ int sel[4][8];
  int* slot = sel[threadIdx.x >> 6];
  long long cnt = 0;
  // 64 intervals a round, the last of them again the first of the next round:
  // entry i is used by intervals i and i + 1
  for (int i0 = 0; i0 < n; i0 += 63) {
    const int i = i0 + lane;
    bool found = false;
    int p = 0, p1 = -1;
    float lo = 0.0f, hi = 0.0f;
    if (i <= n) {
      lo = i > 0 ? v[i - 1] : -FLT_MAX, hi = i < n ? v[i] : FLT_MAX;
      const float g0 = lo * kx, g1 = hi * kx;
      const float f0 = fmaxf(pmin, fminf(g0, g1) + lmin), f1 = fminf(pmax, fmaxf(g0, g1) + lmax);
      p = max(0, (int)ceilf(f0 - 0.5f)), p1 = min(np - 1, (int)floorf(f1 - 0.5f));
      for (int k = 0; k < 2 && p <= p1 && !found; ++k, ++p) found = column(p, lo, hi);
    }
    // the few lanes that are left cross a wall or a solid block: eight of them at a
    // time are helped by eight lanes each, which take the next eight positions (SOLID:
    // from the second time on, after those of the next 64 whose tiles are solid)
    for (bool again = false;; again = true) {  // the same in every lane
      const bool left = !found && p <= p1;
      const unsigned long long lm = __ballot(left);
      if (!lm) break;
      const int rank = __popcll(lm & ((1ull << lane) - 1ull)), grp = lane >> 3;
      if (left && rank < 8) slot[rank] = lane;
      wave_lds_sync();
      const bool helps = grp < __popcll(lm);
      const int owner = helps ? slot[grp] : lane;
      wave_lds_sync();  // read before the next round's writes
      const float olo = __shfl(lo, owner), ohi = __shfl(hi, owner);
      int op = __shfl(p, owner);
      const int op1 = __shfl(p1, owner);
      if (SOLID && again) {
        const unsigned long long open = __ballot(helps && !solid((op & ~7) + 8 * (lane & 7)));
        const auto ahead = [open](int g, int at) {
          const unsigned o = (unsigned)(open >> (8 * g)) & 0xffu;
          return o & 1u ? at : (at & ~7) + 8 * (o ? __builtin_ctz(o) : 8);
        };
        op = ahead(grp, op);
        if (left && rank < 8) p = ahead(rank, p);
      }
      op += lane & 7;
      const bool hit = helps && op <= op1 && column(op, olo, ohi);
      const unsigned long long hm = __ballot(hit);
      if (left && rank < 8) {
        found = (hm >> (8 * rank)) & 0xffull;
        p += 8;
      }
    }
    const unsigned long long f = __ballot(found);
    const unsigned long long u = (f | (f >> 1)) & 0x7fffffffffffffffull;  // entries i0 .. i0 + 62
    const bool mine = lane < 63 && i < n;
    if (mine) used[s + i] = (uint8_t)((u >> lane) & 1ull);
    cnt += __popcll(u & __ballot(mine));
  }
  if (lane == 0) kept[b] = cnt;
}

// RangeMethod::calc_range_many_radial_optimized (RangeLib.h:616-676), one
// thread per output slot s of particle p.  The reference loops a = 0..mpi
// writing pair(a).r to slot a and pair(a).r_inv to slot a + off, then a =
// mpi+1..off-1 writing calc_range to slot a, the beam angle growing by `step`
// each iteration; a slot keeps its last write.  So slot s is: the single ray
// if mpi < s < off; else pair(s - off).r_inv if that iteration exists and
// either off <= 0 or s > mpi; else pair(s).r if s <= mpi; else untouched.
// Pairs exist for CDDTCast only (-1, -1 for the other methods, RangeLib.h:419).
template <int METHOD>
__global__ __launch_bounds__(256) void k_radial(MapDev m, TrigDev trig, float max_range, const float* __restrict__ ins,
                                                float* __restrict__ outs, int N, int nr, float min_angle, float step,
                                                int mpi, int off) {
  __shared__ float lut[RL_LUT_SIZE];
  stage_lut<METHOD>(m, lut);
  const unsigned r = blockIdx.x * blockDim.x + threadIdx.x;  // N * nr < 2^31 (checked by the caller)
  if (r >= (unsigned)N * (unsigned)nr) return;
  const int p = (int)(r / (unsigned)nr), s = (int)(r - (unsigned)p * (unsigned)nr);
  int kind = 0, a = 0;  // 1: pair r, 2: pair r_inv, 3: single ray
  if (s > mpi && s < off) {
    kind = 3;
    a = s;
  } else {
    const bool first = s <= mpi;
    const int a2 = s - off;
    const bool second = a2 >= 0 && a2 <= mpi;
    if (second && (off <= 0 || !first)) {
      kind = 2;
      a = a2;
    } else if (first) {
      kind = 1;
      a = s;
    }
  }
  if (kind == 0) return;
  float angle = min_angle;
  for (int k = 0; k < a; ++k) angle += step;
  float gx, gy;
  rl::to_grid(m.world, ins[3 * (size_t)p], ins[3 * (size_t)p + 1], &gx, &gy);
  const float h = (-ins[3 * (size_t)p + 2] + m.world.rotation_const) - angle;
  float v;
  if (kind == 3) {
    int unused;
    v = cast_one<METHOD, false>(m, lut, rl::Box{nullptr, 0, 0}, trig, max_range, gy, gx, h, &unused);
  } else {
    float r0 = -1.0f, r1 = -1.0f;
    if (METHOD == RL_METHOD_CDDT) rl::cddt_calc_range_pair(m, max_range, gy, gx, h, &r0, &r1);
    v = kind == 1 ? r0 : r1;
  }
  outs[r] = v * m.world.scale;
}

namespace {

// A build's scratch from the context's pool, given back when the build's scope
// ends (after waiting for what it launched).
struct DevBuf {
  rl_ctx* c;
  void* p = nullptr;
  explicit DevBuf(rl_ctx* ctx) : c(ctx) {}
  DevBuf(const DevBuf&) = delete;
  ~DevBuf() {
    if (!p) return;
    (void)hipStreamSynchronize(c->stream);
    c->pool.release(p, true);
  }
  int alloc(size_t bytes) {
    if (c->pool.alloc(&p, bytes) != hipSuccess) {
      (void)hipGetLastError();
      return fail(RL_ERR_NOMEM, "CDDT: device allocation of %zu bytes failed", bytes);
    }
    return RL_OK;
  }
  template <class T>
  T* as() const {
    return (T*)p;
  }
};

#include "rl_scan_sort.h"

void cddt_free(rl_map* m) {
  void* ps[] = {m->cddt_width, m->cddt_trans, m->cddt_cos, m->cddt_sin, m->cddt_bin_off, m->cddt_start, m->cddt_vals};
  for (void* p : ps) m->ctx->pool.release(p, false);
  m->cddt_width = nullptr;
  m->cddt_trans = m->cddt_cos = m->cddt_sin = m->cddt_vals = nullptr;
  m->cddt_bin_off = m->cddt_start = nullptr;
  m->cddt_td = 0;
  m->cddt_nb = m->cddt_nv = 0;
}

// Table buffer from the pool.
template <class T>
int cddt_table(rl_map* m, T** p, size_t count) {
  if (m->ctx->pool.alloc(p, count * sizeof(T)) != hipSuccess) {
    (void)hipGetLastError();
    return fail(RL_ERR_NOMEM, "CDDT: device allocation of %zu bytes failed", count * sizeof(T));
  }
  return RL_OK;
}

// A 64-bit value of the device, after the stream's work so far (through the
// context's pinned block: its mutex is held).
int cddt_read(rl_map* m, const long long* d, long long* out) {
  long long* h;
  TRY(m->ctx->pinned((void**)&h));
  HIP_TRY(hipMemcpyAsync(h, d, sizeof(long long), hipMemcpyDeviceToHost, m->ctx->stream));
  HIP_TRY(hipStreamSynchronize(m->ctx->stream));
  *out = *h;
  return RL_OK;
}

// One wave per bin, striding from 2^20 workgroups on (a grid's threads stay below
// 2^32; 65536 headings of a 1200^2 map have 10^8 bins).
dim3 cddt_compact_grid(long long nb) { return dim3((unsigned)std::min<long long>((nb + 3) / 4, 1 << 20)); }

// Keeps the entries selected by `mode` (see k_cddt_compact): new start and
// values.  kept: the bins' numbers of entries to keep (nb + 1, the last 0).
int cddt_compact(rl_map* m, int mode, const uint8_t* used, const DevBuf& kept) {
  rl_ctx* c = m->ctx;
  hipStream_t st = c->stream;
  const long long nb = m->cddt_nb;
  DevBuf tiles(c), nstart(c), nvals(c);  // (the new tables leave through .p)
  TRY(nstart.alloc((size_t)(nb + 1) * sizeof(long long)));
  // the scan writes n + 1 values: its input has a trailing zero
  TRY(exclusive_sum_u64(st, kept.as<unsigned long long>(), nstart.as<unsigned long long>(), nb + 1, &tiles));
  long long total = 0;
  TRY(cddt_read(m, nstart.as<long long>() + nb, &total));
  TRY(nvals.alloc((size_t)total * sizeof(float)));
  hipLaunchKernelGGL(k_cddt_compact<true>, cddt_compact_grid(nb), dim3(256), 0, st, nb,
                     (const long long*)m->cddt_start, (const float*)m->cddt_vals, used, mode, (const long long*)nstart.p,
                     (long long*)nullptr, nvals.as<float>());
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(st));
  c->pool.release(m->cddt_start, false);
  c->pool.release(m->cddt_vals, false);
  m->cddt_start = nstart.as<long long>();
  m->cddt_vals = nvals.as<float>();
  nstart.p = nvals.p = nullptr;
  m->cddt_nv = total;
  return RL_OK;
}

// nb + 1 zeroed counts.
int cddt_counts(rl_map* m, DevBuf* kept) {
  const size_t bytes = (size_t)(m->cddt_nb + 1) * sizeof(unsigned long long);
  TRY(kept->alloc(bytes));
  HIP_TRY(hipMemsetAsync(kept->p, 0, bytes, m->ctx->stream));
  return RL_OK;
}

// Rule for k_cddt_prune_mark<true>: more than four occupied cells inside for one at an
// edge, walls of some ten cells in the mean, from where tiles are solid often enough
// (per edge cell: corridor maps 1.8 to 2.1, prune 3% slower with the tiles' tests; disks and
// rectangles of a 1024^2 map 11, 0.50 -> 0.46 ms; stripes of 32 15, 0.87 -> 0.47 ms).
bool cddt_solid(unsigned edges, unsigned occupied) { return (occupied - edges) / 4 > edges; }

int cddt_build_locked(rl_map* m, int td) {
  rl_ctx* c = m->ctx;
  hipStream_t st = c->stream;
  const int W = m->width, H = m->height;
  if ((long long)W * H > 0x7fffffffLL) return fail(RL_ERR_ARG, "CDDT: maps above 2^31 cells are not supported");
  cddt_free(m);
  m->cddt_td = td;
  int nang = 0;
  while (nang < td && nang < td / 2.0) ++nang;  // a < theta_discretization / 2.0
  m->cddt_nang = nang;
  m->cddt_td_div_2pi = (float)((double)td / 6.28318530718);          // RangeLib.h:976
  const float m2pi_div_td = (float)(6.28318530718 / (double)(float)td);  // :977
  TRY(cddt_table(m, &m->cddt_width, (size_t)td));
  TRY(cddt_table(m, &m->cddt_trans, (size_t)td));
  TRY(cddt_table(m, &m->cddt_cos, (size_t)td));
  TRY(cddt_table(m, &m->cddt_sin, (size_t)td));
  TRY(cddt_table(m, &m->cddt_bin_off, (size_t)td + 1));
  hipLaunchKernelGGL(k_cddt_consts, dim3(grid_for(td, 64)), dim3(64), 0, st, c->trig, td, W, H, m2pi_div_td,
                     m->cddt_width, m->cddt_trans, m->cddt_cos, m->cddt_sin);
  HIP_TRY(hipGetLastError());
  // edge cells
  const long long N = (long long)W * H;
  DevBuf edges(c), n_edges(c);
  TRY(edges.alloc((size_t)N * sizeof(unsigned)));
  TRY(n_edges.alloc(sizeof(unsigned long long)));
  HIP_TRY(hipMemsetAsync(n_edges.p, 0, sizeof(unsigned long long), st));
  hipLaunchKernelGGL(k_cddt_edges, dim3(grid_for(N, 256 * RL_CDDT_EDGE_ITEMS)), dim3(256), 0, st,
                     (const uint8_t*)m->d_occ, W, H, edges.as<unsigned>(), n_edges.as<unsigned long long>());
  HIP_TRY(hipGetLastError());
  CddtSizes* sz;
  TRY(c->pinned((void**)&sz));
  hipLaunchKernelGGL(k_cddt_offsets, dim3(1), dim3(1024), 0, st, (const int*)m->cddt_width, td, nang,
                     (const unsigned long long*)n_edges.p, m->cddt_bin_off, sz);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(st));
  const long long nb = sz->nb, nba = sz->nba;
  const unsigned ne = sz->ne;
  m->cddt_solid = cddt_solid(ne, sz->occupied);
  const int max_width = sz->max_width;
  m->cddt_nb = nb;
  // count, scan, fill.  In LDS where an angle's bins fit; about 1024 workgroups,
  // each of at least 2048 edge cells and at most 32 chunks of an angle
  DevBuf counter(c), chunks(c), tiles(c), raw(c), kept(c), lists(c);
  TRY(cddt_counts(m, &counter));
  const bool in_lds = max_width <= RL_CDDT_LDS_BINS;
  const int G = std::max(1, std::min(std::min(32, 1024 / nang + 1), (int)(ne / 2048u)));
  const unsigned hist_grid = 8u * (unsigned)((nang + 7) / 8) * (unsigned)G;
  const unsigned hist_lds = (unsigned)max_width * sizeof(unsigned);
  if (ne && in_lds) {
    TRY(chunks.alloc((size_t)G * (size_t)nb * sizeof(unsigned)));
    hipLaunchKernelGGL(k_cddt_hist<false>, dim3(hist_grid), dim3(256), hist_lds, st, (const unsigned*)edges.p, (int)ne,
                       nang, G, (const int*)m->cddt_width, (const float*)m->cddt_trans, (const float*)m->cddt_cos,
                       (const float*)m->cddt_sin, (const long long*)m->cddt_bin_off, (const long long*)nullptr,
                       chunks.as<unsigned>(), nb, (float*)nullptr);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_cddt_chunks, dim3((unsigned)grid_for(nba, 256)), dim3(256), 0, st, chunks.as<unsigned>(), G, nb,
                       counter.as<unsigned long long>(), nba);
    HIP_TRY(hipGetLastError());
  }
  for (int a0 = 0; ne && !in_lds && a0 < nang; a0 += 65535) {  // grid rows: at most 65535 angles per launch
    hipLaunchKernelGGL(k_cddt_scatter<false>, dim3(grid_for(ne, 256), (unsigned)std::min(65535, nang - a0)), dim3(256),
                       0, st, (const unsigned*)edges.p, (int)ne, a0, (const int*)m->cddt_width,
                       (const float*)m->cddt_trans, (const float*)m->cddt_cos, (const float*)m->cddt_sin,
                       (const long long*)m->cddt_bin_off, counter.as<unsigned long long>(), (float*)nullptr);
    HIP_TRY(hipGetLastError());
  }
  TRY(cddt_table(m, &m->cddt_start, (size_t)nb + 1));
  TRY(exclusive_sum_u64(st, counter.as<unsigned long long>(), (unsigned long long*)m->cddt_start, nb + 1, &tiles));
  long long total = 0;
  TRY(cddt_read(m, m->cddt_start + nb, &total));
  if (total > 0x7fffffffLL) return fail(RL_ERR_ARG, "CDDT: %lld table entries exceed 2^31", total);
  TRY(raw.alloc((size_t)total * sizeof(float)));
  if (ne && in_lds) {
    hipLaunchKernelGGL(k_cddt_hist<true>, dim3(hist_grid), dim3(256), hist_lds, st, (const unsigned*)edges.p, (int)ne,
                       nang, G, (const int*)m->cddt_width, (const float*)m->cddt_trans, (const float*)m->cddt_cos,
                       (const float*)m->cddt_sin, (const long long*)m->cddt_bin_off, (const long long*)m->cddt_start,
                       chunks.as<unsigned>(), nb, raw.as<float>());
    HIP_TRY(hipGetLastError());
  } else if (ne) {
    HIP_TRY(hipMemcpyAsync(counter.p, m->cddt_start, (size_t)(nb + 1) * sizeof(long long), hipMemcpyDeviceToDevice, st));
    for (int a0 = 0; a0 < nang; a0 += 65535) {
      hipLaunchKernelGGL(k_cddt_scatter<true>, dim3(grid_for(ne, 256), (unsigned)std::min(65535, nang - a0)), dim3(256),
                         0, st, (const unsigned*)edges.p, (int)ne, a0, (const int*)m->cddt_width,
                         (const float*)m->cddt_trans, (const float*)m->cddt_cos, (const float*)m->cddt_sin,
                         (const long long*)m->cddt_bin_off, counter.as<unsigned long long>(), raw.as<float>());
      HIP_TRY(hipGetLastError());
    }
  }
  // sort each bin
  TRY(cddt_table(m, &m->cddt_vals, (size_t)total));
  if (total > 0) TRY(segmented_sort_f32(st, raw.as<float>(), m->cddt_vals, m->cddt_start, nb, &lists));
  m->cddt_nv = total;
  // drop duplicates
  TRY(cddt_counts(m, &kept));
  hipLaunchKernelGGL(k_cddt_compact<false>, cddt_compact_grid(nb), dim3(256), 0, st, nb,
                     (const long long*)m->cddt_start, (const float*)m->cddt_vals, (const uint8_t*)nullptr, 0,
                     (const long long*)nullptr, kept.as<long long>(), (float*)nullptr);
  HIP_TRY(hipGetLastError());
  return cddt_compact(m, 0, nullptr, kept);
}

// CDDTCast::prune: max_range does not change which entries stay (k_cddt_prune_mark).
int cddt_prune_locked(rl_map* m) {
  hipStream_t st = m->ctx->stream;
  const int W = m->width, H = m->height;
  DevBuf used(m->ctx), kept(m->ctx);
  TRY(used.alloc((size_t)m->cddt_nv + 1));
  TRY(cddt_counts(m, &kept));
  // widths are at most |W sin| + |H cos| rounded up
  const int max_width = (int)ceil(sqrt((double)W * W + (double)H * H)) + 1;
  for (int a0 = 0; a0 < m->cddt_nang; a0 += 65535) {  // grid rows: at most 65535 angles per launch
    const int na = std::min(65535, m->cddt_nang - a0);
    hipLaunchKernelGGL(m->cddt_solid ? k_cddt_prune_mark<true> : k_cddt_prune_mark<false>,
                       dim3((unsigned)grid_for(max_width, 4), (unsigned)na), dim3(256), 0, st,
                       (const uint8_t*)m->d_occ, W, H, (const unsigned long long*)m->d_bits, (W + 7) / 8, (H + 7) / 8,
                       (const int*)m->cddt_width, (const float*)m->cddt_trans, (const float*)m->cddt_cos,
                       (const float*)m->cddt_sin, (const long long*)m->cddt_bin_off, (const long long*)m->cddt_start,
                       (const float*)m->cddt_vals, used.as<uint8_t>(), kept.as<long long>(), a0);
    HIP_TRY(hipGetLastError());
  }
  return cddt_compact(m, 1, used.as<uint8_t>(), kept);
}

template <int METHOD>
int launch_radial_t(rl_map* m, float max_range, const float* ins, float* outs, int N, int nr, float min_angle,
                    float step, int mpi, int off) {
  const long long n = (long long)N * nr;
  if (n == 0) return RL_OK;
  hipLaunchKernelGGL(k_radial<METHOD>, dim3(grid_for(n, 256)), dim3(256), 0, m->ctx->stream, m->dev(),
                     m->ctx->trig, max_range, ins, outs, N, nr, min_angle, step, mpi, off);
  HIP_TRY(hipGetLastError());
  return RL_OK;
}

int launch_radial(rl_map* m, int method, float max_range, const float* ins, float* outs, int N, int nr,
                  float min_angle, float max_angle) {
  TRY(check_map(m, method, max_range));
  if ((long long)N * nr > 0x7fffffffLL) return fail(RL_ERR_ARG, "batch too large");
  // RangeLib.h:631-641
  const float step = (max_angle - min_angle) / (float)(nr - 1);
  const int mpi = (int)((double)(float)nr / 3.0);
  const float iof = (float)(((double)nr - 1.0) * 3.14159265358979323846 / (double)(max_angle - min_angle));
  const int off = (int)roundf(iof);
  switch (method) {
    case RL_METHOD_BL: return launch_radial_t<RL_METHOD_BL>(m, max_range, ins, outs, N, nr, min_angle, step, mpi, off);
    case RL_METHOD_GLT: return launch_radial_t<RL_METHOD_GLT>(m, max_range, ins, outs, N, nr, min_angle, step, mpi, off);
    case RL_METHOD_CDDT: return launch_radial_t<RL_METHOD_CDDT>(m, max_range, ins, outs, N, nr, min_angle, step, mpi, off);
    default: return launch_radial_t<RL_METHOD_RM>(m, max_range, ins, outs, N, nr, min_angle, step, mpi, off);
  }
}

}  // namespace

extern "C" {

int rl_calc_range_many_radial_optimized_dev(rl_map* m, int method, float max_range, const float* d_ins,
                                            float* d_outs, int num_particles, int num_rays, float min_angle,
                                            float max_angle) {
  CHECK_ARG(m && d_ins && d_outs && num_particles >= 0 && num_rays >= 2, "bad argument");
  std::lock_guard<std::mutex> lk(m->ctx->mu);
  TRY(use_device(m->ctx));
  return launch_radial(m, method, max_range, d_ins, d_outs, num_particles, num_rays, min_angle, max_angle);
}

int rl_calc_range_many_radial_optimized(rl_map* m, int method, float max_range, const float* ins, float* outs,
                                        int num_particles, int num_rays, float min_angle, float max_angle) {
  CHECK_ARG(m && ins && outs && num_particles >= 0 && num_rays >= 2, "bad argument");
  rl_ctx* c = m->ctx;
  std::lock_guard<std::mutex> lk(c->mu);
  TRY(use_device(c));
  const long long n = (long long)num_particles * num_rays;
  if (n > 0x7fffffffLL) return fail(RL_ERR_ARG, "batch too large");
  if (n == 0) return RL_OK;
  void *d_ins, *d_out;
  TRY(c->staging(0, (size_t)num_particles * 3 * sizeof(float), &d_ins));
  TRY(c->staging(1, (size_t)n * sizeof(float), &d_out));
  HIP_TRY(hipMemcpyAsync(d_ins, ins, (size_t)num_particles * 3 * sizeof(float), hipMemcpyHostToDevice, c->stream));
  // slots the reference leaves untouched keep the caller's values
  HIP_TRY(hipMemcpyAsync(d_out, outs, (size_t)n * sizeof(float), hipMemcpyHostToDevice, c->stream));
  TRY(launch_radial(m, method, max_range, (const float*)d_ins, (float*)d_out, num_particles, num_rays, min_angle,
                    max_angle));
  HIP_TRY(hipMemcpyAsync(outs, d_out, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  return RL_OK;
}

int rl_map_build_cddt(rl_map* m, int theta_disc) {
  CHECK_ARG(m, "map is NULL");
  CHECK_ARG(theta_disc >= 1 && theta_disc <= 65536, "theta_discretization outside 1..65536");
  rl_ctx* c = m->ctx;
  std::lock_guard<std::mutex> lk(c->mu);
  TRY(use_device(c));
  HIP_TRY(hipStreamSynchronize(c->stream));
  m->gen.fetch_add(1);
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  (void)hipEventRecord(e0, c->stream);
  int rc = cddt_build_locked(m, theta_disc);
  (void)hipEventRecord(e1, c->stream);
  (void)hipEventSynchronize(e1);
  (void)hipEventElapsedTime(&m->cddt_ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc != RL_OK) {
    std::string msg = g_err;
    cddt_free(m);
    return fail(rc, "%s", msg.c_str());
  }
  return RL_OK;
}

int rl_map_prune_cddt(rl_map* m, float /*max_range*/) {
  CHECK_ARG(m, "map is NULL");
  rl_ctx* c = m->ctx;
  std::lock_guard<std::mutex> lk(c->mu);
  TRY(use_device(c));
  if (!m->cddt_vals) return fail(RL_ERR_STATE, "no CDDT tables (call rl_map_build_cddt first)");
  HIP_TRY(hipStreamSynchronize(c->stream));
  m->gen.fetch_add(1);
  return cddt_prune_locked(m);
}

int rl_map_get_cddt(rl_map* m, int* theta_disc, long long* nbins, long long* nvals, int* widths, float* trans,
                    long long* start, float* vals, float* build_ms) {
  CHECK_ARG(m, "map is NULL");
  rl_ctx* c = m->ctx;
  std::lock_guard<std::mutex> lk(c->mu);
  TRY(use_device(c));
  if (!m->cddt_vals) return fail(RL_ERR_STATE, "no CDDT tables (call rl_map_build_cddt first)");
  HIP_TRY(hipStreamSynchronize(c->stream));
  if (theta_disc) *theta_disc = m->cddt_td;
  if (nbins) *nbins = m->cddt_nb;
  if (nvals) *nvals = m->cddt_nv;
  if (build_ms) *build_ms = m->cddt_ms;
  if (widths) HIP_TRY(hipMemcpy(widths, m->cddt_width, m->cddt_td * sizeof(int), hipMemcpyDeviceToHost));
  if (trans) HIP_TRY(hipMemcpy(trans, m->cddt_trans, m->cddt_td * sizeof(float), hipMemcpyDeviceToHost));
  if (start)
    HIP_TRY(hipMemcpy(start, m->cddt_start, (size_t)(m->cddt_nb + 1) * sizeof(long long), hipMemcpyDeviceToHost));
  if (vals && m->cddt_nv)
    HIP_TRY(hipMemcpy(vals, m->cddt_vals, (size_t)m->cddt_nv * sizeof(float), hipMemcpyDeviceToHost));
  return RL_OK;
}

int rl_debug_exclusive_sum_dev(rl_ctx* c, const unsigned long long* in, unsigned long long* out, long long n) {
  CHECK_ARG(c && (n <= 0 || (in && out)), "bad argument");
  std::lock_guard<std::mutex> lk(c->mu);
  TRY(use_device(c));
  DevBuf tiles(c);
  TRY(exclusive_sum_u64(c->stream, in, out, n, &tiles));
  HIP_TRY(hipStreamSynchronize(c->stream));
  return RL_OK;
}

int rl_debug_segmented_sort_dev(rl_ctx* c, const float* in, float* out, const long long* start, long long nseg) {
  CHECK_ARG(c && (nseg <= 0 || (in && out && start)), "bad argument");
  std::lock_guard<std::mutex> lk(c->mu);
  TRY(use_device(c));
  DevBuf lists(c);
  TRY(segmented_sort_f32(c->stream, in, out, start, nseg, &lists));
  HIP_TRY(hipStreamSynchronize(c->stream));
  return RL_OK;
}

}  // extern "C"
