// CIC paint of particles in any order, by mesh tiles (part of paint.hip).
//
// Three launches, almost without device-scope atomics:
// k_bin_sort: one workgroup per kBinChunk consecutive particles sorts the
//   chunk's particle numbers by the mesh tiles their corners touch (mostly
//   one; at the faces of a tile up to eight), with a histogram in LDS, and
//   leaves them with where each tile's run starts.
// k_bin_paint: one workgroup per tile collects its runs of all chunks, reads
//   those particles, adds the corners that lie in the tile to a box in LDS in
//   float64, and adds the box to the mesh (or writes it) with plain accesses.
// k_bin_tail: what a tile holds beyond kBinShare entries (k_bin_paint counts
//   such tiles with an atomic) is shared out to further workgroups, which add
//   their boxes with float atomics (a catalogue within one tile of 120^3: 300001
//   particles 412 us by the scatter, 1730 in one workgroup, 63 in shares).
// The sums are float64 (the LDS atomics' order shows in the 53rd bit), so a cell
// of a tile of up to kBinShare entries is rounded once, and repeats but for that;
// in a fuller tile it is rounded once per share, in an order that may vary.
// float64 LDS atomics run at 2.8 per clock and CU here, 32-bit integers at 8.8,
// 64-bit ones at 5.3, float32 at 0.3.
// The scatter's device-scope atomics run at 27 per ns on the whole chip: the
// paint of 300007 particles on 120^3 126 us -> 30, that of 2 x 96^3 in the
// readout's adjoint 485 -> 62.
#pragma once

namespace pmx {

constexpr int kBinChunk = 2048, kBinT = 512, kBinPPT = kBinChunk / kBinT;
constexpr int kBinX = 8, kBinY = 16, kBinZ = 16;  // tile: a float64 box of 16 KB
constexpr int kBinCells = kBinX * kBinY * kBinZ;
constexpr int kBinTiles = 8192;  // most tiles: a 32 KB histogram
constexpr int kBinPT = 512, kBinU = 2;  // threads, entries in flight of each
constexpr int kBinShare = 8192;  // entries of a tile per workgroup
constexpr int kBinTail = 512;    // workgroups for the rest
// Fewest particles: the two launches cost 10 us and a pass over the tiles, the
// scatter 0.39 ns per particle.  Uniform ones, scatter / tiles in us: 32^3
// 42599 19.1 / 20.2; 64^3 16385 8.9 / 13.0, 45511 20.0 / 14.0; 120^3 34561
// 16.1 / 18.5, 108001 45 / 19, 1.3 per cell 863 / 114; 192^3 70779 31.7 / 38.2,
// 141557 58 / 39; 250^3 156251 64 / 74, 312501 122 / 78.  The line lies where
// some 10 us are gained, as two launches more take the host as long (63975
// particles on 5 x 48 x 48 x 24: 126 us a call by tiles, 122 by the scatter).
constexpr long long kBinMin = 32 * 2048, kBinSparse = 80;

struct BinArgs {
  float* mesh;
  const float* base;  // added to, or null; may be the mesh itself
  const float* pos;
  const float* w;  // or null (ones)
  float ps;
  MeshDims d;
  int nty, ntz, ntiles;
  int nchunk;    // chunks per batch member
  int row, cap;  // 16-bit words per chunk: run starts, particle numbers
  unsigned short* start;  // [chunk][row]: starts of the tiles' runs, the end
  unsigned short* list;   // [chunk][cap]: numbers within the chunk
  int* heavy;             // count, then (tile, member, entries) of the tiles
                          // with more than kBinShare
};

struct BinAxis {
  int i0, i1;  // wrapped corner cells
};
__device__ __forceinline__ BinAxis bin_axis(float x, int n) {
  BinAxis c;
  c.i0 = (int)floorf(x);
  if ((unsigned)c.i0 >= (unsigned)n) c.i0 = imod(c.i0, n);
  c.i1 = c.i0 + 1 == n ? 0 : c.i0 + 1;
  return c;
}

// (17 us for 2 x 96^3 particles on 864 tiles each, 8 for 300007 on 960)
__global__ __launch_bounds__(kBinT) void k_bin_sort(BinArgs a) {
  extern __shared__ unsigned hist[];  // [ntiles]: counts, then cursors
  __shared__ unsigned wsum[kBinT / 64];
  const int tid = threadIdx.x, ln = tid & 63, wv = tid >> 6;
  const int b = blockIdx.y;
  const long long q = (long long)b * a.nchunk + blockIdx.x;
  const long long first = (long long)blockIdx.x * kBinChunk;
  const int n = (int)min((long long)kBinChunk, a.d.N - first);
  const float* const X = a.pos + 3 * ((long long)b * a.d.N + first);
  if (q == 0 && tid == 0) a.heavy[0] = 0;
  for (int i = tid; i < a.ntiles; i += kBinT) hist[i] = 0;
  // the particles' first tiles, and the steps to the next tile of each axis
  // (0: both corners in one)
  int t0[kBinPPT], sx[kBinPPT], sy[kBinPPT], sz[kBinPPT];
  float px[kBinPPT], py[kBinPPT], pz[kBinPPT];
#pragma unroll
  for (int u = 0; u < kBinPPT; ++u) {
    const int t = min(tid + u * kBinT, n - 1);
    px[u] = X[3 * t] * a.ps;
    py[u] = X[3 * t + 1] * a.ps;
    pz[u] = X[3 * t + 2] * a.ps;
  }
#pragma unroll
  for (int u = 0; u < kBinPPT; ++u) {
    t0[u] = -1;
    sx[u] = sy[u] = sz[u] = 0;
    if (tid + u * kBinT < n && ok_pos(px[u], py[u], pz[u])) {
      const BinAxis x = bin_axis(px[u], a.d.nx), y = bin_axis(py[u], a.d.ny),
                    z = bin_axis(pz[u], a.d.nz);
      const int tx = x.i0 / kBinX, ty = y.i0 / kBinY, tz = z.i0 / kBinZ;
      t0[u] = (tx * a.nty + ty) * a.ntz + tz;
      sx[u] = (x.i1 / kBinX - tx) * a.nty * a.ntz;
      sy[u] = (y.i1 / kBinY - ty) * a.ntz;
      sz[u] = z.i1 / kBinZ - tz;
    }
  }
  __syncthreads();
  // f(tile, u) for every tile that particle u touches
  auto tiles = [&](auto&& f) {
#pragma unroll
    for (int u = 0; u < kBinPPT; ++u) {
      if (t0[u] < 0) continue;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (((k & 1) && sx[u] == 0) || ((k & 2) && sy[u] == 0) ||
            ((k & 4) && sz[u] == 0))
          continue;
        f(t0[u] + (k & 1 ? sx[u] : 0) + (k & 2 ? sy[u] : 0) +
              (k & 4 ? sz[u] : 0), u);
      }
    }
  };
  tiles([&](int t, int) { atomicAdd(&hist[t], 1u); });
  __syncthreads();
  // exclusive scan: a run of consecutive tiles per thread
  const int per = (a.ntiles + kBinT - 1) / kBinT, i0 = tid * per;
  unsigned s = 0;
  for (int i = 0; i < per; ++i)
    if (i0 + i < a.ntiles) s += hist[i0 + i];
  unsigned sc = s;
#pragma unroll
  for (int k = 1; k < 64; k <<= 1) {
    const unsigned v = __shfl_up(sc, k);
    if (ln >= k) sc += v;
  }
  if (ln == 63) wsum[wv] = sc;
  __syncthreads();
  unsigned at = sc - s;
  for (int w = 0; w < wv; ++w) at += wsum[w];
  for (int i = 0; i < per; ++i)
    if (i0 + i < a.ntiles) {
      const unsigned h = hist[i0 + i];
      hist[i0 + i] = at;
      at += h;
    }
  __syncthreads();
  unsigned short* const row = a.start + q * a.row;
  for (int i = tid; i < a.ntiles; i += kBinT)
    row[i] = (unsigned short)hist[i];
  if (tid == 0) {
    unsigned end = 0;
    for (int w = 0; w < kBinT / 64; ++w) end += wsum[w];
    row[a.ntiles] = (unsigned short)end;  // <= 8 kBinChunk
  }
  __syncthreads();
  unsigned short* const out = a.list + q * a.cap;
  tiles([&](int t, int u) {
    out[atomicAdd(&hist[t], 1u)] = (unsigned short)(tid + u * kBinT);
  });
}

struct BinLds {
  double box[kBinCells];
  int pre[kBinPT];  // entries before a chunk's run
  int beg[kBinPT];  // where the run starts, less those
  int wsum[kBinPT / 64];
};

// Adds the tile's entries number [lo, hi) (of those of all chunks, in chunk
// order) to the cleared box; returns how many entries the tile has (at least
// hi, if it stops there).
__device__ __forceinline__ long long bin_deposit(const BinArgs& a, BinLds& l,
                                                 int tile, int b, long long lo,
                                                 long long hi, bool stop) {
  const MeshDims& d = a.d;
  const int tid = threadIdx.x, ln = tid & 63, wv = tid >> 6;
  const int tz = tile % a.ntz, r = tile / a.ntz, ty = r % a.nty, tx = r / a.nty;
  const int x0 = tx * kBinX, y0 = ty * kBinY, z0 = tz * kBinZ;
  const long long q0 = (long long)b * a.nchunk;
  const float* const X = a.pos + 3 * (long long)b * d.N;
  const float* const W = a.w ? a.w + (long long)b * d.N : nullptr;
  long long seen = 0;
  for (int c0 = 0; c0 < a.nchunk && !(stop && seen >= hi); c0 += kBinPT) {
    int s = 0, cnt = 0;
    if (c0 + tid < a.nchunk) {
      const unsigned short* const row = a.start + (q0 + c0 + tid) * a.row + tile;
      s = row[0];
      cnt = row[1] - s;
    }
    int sc = cnt;
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) {
      const int v = __shfl_up(sc, k);
      if (ln >= k) sc += v;
    }
    __syncthreads();  // (the last round's reads of pre and beg; the box)
    if (ln == 63) l.wsum[wv] = sc;
    __syncthreads();
    int off = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kBinPT / 64; ++w) {
      if (w < wv) off += l.wsum[w];
      total += l.wsum[w];
    }
    l.pre[tid] = off + sc - cnt;
    l.beg[tid] = s - (off + sc - cnt);
    __syncthreads();
    const int e0 = (int)max(lo - seen, 0LL),
              e1 = (int)min(hi - seen, (long long)total);
    seen += total;
    for (int e = e0 + tid; e < e1; e += kBinU * kBinPT) {
      float x[kBinU], y[kBinU], z[kBinU], wt[kBinU];
      int j[kBinU];
#pragma unroll
      for (int u = 0; u < kBinU; ++u) j[u] = 0;
      // the last run that starts at or before the entry
#pragma unroll
      for (int k = kBinPT / 2; k > 0; k >>= 1)
#pragma unroll
        for (int u = 0; u < kBinU; ++u)
          if (l.pre[j[u] + k] <= min(e + u * kBinPT, e1 - 1)) j[u] += k;
      int num[kBinU];
#pragma unroll
      for (int u = 0; u < kBinU; ++u)
        num[u] = a.list[(q0 + c0 + j[u]) * a.cap + l.beg[j[u]] +
                        min(e + u * kBinPT, e1 - 1)];
#pragma unroll
      for (int u = 0; u < kBinU; ++u) {
        const long long p = (long long)(c0 + j[u]) * kBinChunk + num[u];
        x[u] = X[3 * p];
        y[u] = X[3 * p + 1];
        z[u] = X[3 * p + 2];
        wt[u] = W ? W[p] : 1.0f;
      }
#pragma unroll
      for (int u = 0; u < kBinU; ++u) {
        if (u > 0 && e + u * kBinPT >= e1) break;
        const float px = x[u] * a.ps, py = y[u] * a.ps, pz = z[u] * a.ps;
        const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
        const float wx[2] = {1.0f - fabsf(px - fx), 1.0f - fabsf(px - (fx + 1.0f))};
        const float wy[2] = {1.0f - fabsf(py - fy), 1.0f - fabsf(py - (fy + 1.0f))};
        const float wz[2] = {1.0f - fabsf(pz - fz), 1.0f - fabsf(pz - (fz + 1.0f))};
        const BinAxis cx = bin_axis(px, d.nx), cy = bin_axis(py, d.ny),
                      cz = bin_axis(pz, d.nz);
        const int lx[2] = {cx.i0 - x0, cx.i1 - x0};
        const int ly[2] = {cy.i0 - y0, cy.i1 - y0};
        const int lz[2] = {cz.i0 - z0, cz.i1 - z0};
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int ox = k & 1, oy = (k >> 1) & 1, oz = k >> 2;
          if ((unsigned)lx[ox] < kBinX && (unsigned)ly[oy] < kBinY &&
              (unsigned)lz[oz] < kBinZ)
            atomicAdd(&l.box[(lx[ox] * kBinY + ly[oy]) * kBinZ + lz[oz]],
                      (double)(wt[u] * ((wx[ox] * wy[oy]) * wz[oz])));
        }
      }
    }
  }
  return seen;
}

// mesh cell of box cell i of a tile, or -1 beyond the mesh's end
__device__ __forceinline__ long long bin_cell(const BinArgs& a, int tile,
                                              int b, int i) {
  const int tz = tile % a.ntz, r = tile / a.ntz, ty = r % a.nty, tx = r / a.nty;
  const int z = tz * kBinZ + i % kBinZ, y = ty * kBinY + i / kBinZ % kBinY,
            x = tx * kBinX + i / (kBinZ * kBinY);
  if (x >= a.d.nx || y >= a.d.ny || z >= a.d.nz) return -1;
  return (((long long)b * a.d.nx + x) * a.d.ny + y) * a.d.nz + z;
}

// Bound by the latency of each entry's chain (search, number, position,
// atomics) and the tiles' unequal loads: 512 threads with two entries each in
// flight take 40 us for 2 x 96^3 particles, 256 threads with one 55, with two
// 45, 1024 with two 43.
__global__ __launch_bounds__(kBinPT) void k_bin_paint(BinArgs a) {
  __shared__ BinLds l;
  const int b = blockIdx.y;
  const int tile = (int)xcd_block(blockIdx.x, gridDim.x);
  for (int i = threadIdx.x; i < kBinCells; i += kBinPT) l.box[i] = 0.0;
  const long long n = bin_deposit(a, l, tile, b, 0, kBinShare, false);
  if (threadIdx.x == 0 && n > kBinShare) {
    int* const h = a.heavy + 4 + 4LL * atomicAdd(a.heavy, 1);
    h[0] = tile;
    h[1] = b;
    h[2] = (int)((n - 1) / kBinShare);  // further workgroups' shares
  }
  if (a.base == a.mesh && n == 0) return;
  __syncthreads();
  for (int i = threadIdx.x; i < kBinCells; i += kBinPT) {
    const long long c = bin_cell(a, tile, b, i);
    if (c >= 0)
      a.mesh[c] = (float)(a.base ? (double)a.base[c] + l.box[i] : l.box[i]);
  }
}

// The shares of the tiles that hold more than one, added with float atomics.
__global__ __launch_bounds__(kBinPT) void k_bin_tail(BinArgs a) {
  __shared__ BinLds l;
  const int nh = a.heavy[0];
  int base = 0;  // shares of the tiles before, modulo the grid
  for (int h = 0; h < nh; ++h) {
    const int tile = a.heavy[4 + 4 * h], b = a.heavy[5 + 4 * h],
              shares = a.heavy[6 + 4 * h];
    int k = (int)blockIdx.x - base;
    if (k < 0) k += gridDim.x;
    base = (base + shares) % gridDim.x;
    for (; k < shares; k += gridDim.x) {
      for (int i = threadIdx.x; i < kBinCells; i += kBinPT) l.box[i] = 0.0;
      const long long lo = (k + 1LL) * kBinShare;
      bin_deposit(a, l, tile, b, lo, lo + kBinShare, true);
      __syncthreads();
      for (int i = threadIdx.x; i < kBinCells; i += kBinPT) {
        const long long c = bin_cell(a, tile, b, i);
        if (c >= 0 && l.box[i] != 0.0) atomicAdd(a.mesh + c, (float)l.box[i]);
      }
      __syncthreads();
    }
  }
}

static int bin_tiles(int n, int t) { return (n + t - 1) / t; }

bool bin_paint_ok(const MeshDims& d) {
  if (d.B > 65535 || d.N < 1 || d.N > (1LL << 40)) return false;
  const long long nt = (long long)bin_tiles(d.nx, kBinX) *
                       bin_tiles(d.ny, kBinY) * bin_tiles(d.nz, kBinZ);
  return nt <= kBinTiles &&
         d.B * (d.N - (long long)d.nx * d.ny * d.nz / kBinSparse) >= kBinMin;
}

static BinArgs bin_args(const MeshDims& d) {
  BinArgs a{};
  a.d = d;
  const int ntx = bin_tiles(d.nx, kBinX);
  a.nty = bin_tiles(d.ny, kBinY);
  a.ntz = bin_tiles(d.nz, kBinZ);
  a.ntiles = ntx * a.nty * a.ntz;
  a.nchunk = (int)((d.N + kBinChunk - 1) / kBinChunk);
  a.row = (a.ntiles + 2) & ~1;
  // a particle touches two tiles of an axis that has more than one
  a.cap = kBinChunk * (ntx > 1 ? 2 : 1) * (a.nty > 1 ? 2 : 1) *
          (a.ntz > 1 ? 2 : 1);
  return a;
}

long long bin_work_floats(const MeshDims& d) {
  const BinArgs a = bin_args(d);
  return (long long)d.B * a.nchunk * (a.row + a.cap) / 2 +
         4 + 4LL * d.B * a.ntiles;
}

// (the caller has asked bin_paint_ok)
int launch_bin_paint(float* mesh, const float* base, const float* pos,
                     const float* w, float ps, const MeshDims& d, float* work,
                     ProfKind kind, hipStream_t s) {
  BinArgs a = bin_args(d);
  a.mesh = mesh;
  a.base = base;
  a.pos = pos;
  a.w = w;
  a.ps = ps;
  a.heavy = reinterpret_cast<int*>(work);
  a.start = reinterpret_cast<unsigned short*>(work + 4 + 4LL * d.B * a.ntiles);
  a.list = a.start + (long long)d.B * a.nchunk * a.row;
  ProfScope prof_(kind, s);
  hipLaunchKernelGGL(k_bin_sort, dim3(a.nchunk, d.B), dim3(kBinT),
                     a.ntiles * sizeof(unsigned), s, a);
  PMX_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_bin_paint, dim3(a.ntiles, d.B), dim3(kBinPT), 0, s, a);
  PMX_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_bin_tail, dim3(kBinTail), dim3(kBinPT), 0, s, a);
  PMX_LAUNCH_CHECK();
  return kOk;
}

}  // namespace pmx
