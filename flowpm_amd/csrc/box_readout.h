// Force readout of the particle grid straight from the potential, for gfx950
// (part of cic.hip).
//
// F = fac * readout(D phi), D the fourth-order central difference of
// stencil.hip, phi the potential: the same values as the force mesh of
// k_grad_mesh read by k_readout_kick_drift (cic.hip), without that mesh.
// One workgroup takes one brick of the particle grid (particles that start
// close stay close), loads the box of potential cells its particles' stencils
// reach into LDS, and every particle forms the gradient at its 8 corners
// there; closing kick, opening kick and drift follow in registers.
//
// What bounds it: memory, 48 bytes of state per particle and step and about 11
// of potential (the boxes overlap, about 2.7 times the mesh at a = 0.5), 210
// of the 255 us it takes at 256^3 at the rate of a large copy; then the LDS
// reads (56 potential values per particle as 28 two-float reads; late
// positions spread them unevenly over the banks, 10 clocks a read instead of
// 4) and the VALU work, each about 130 us.  The gradient mesh it replaces
// costs 12 bytes per cell written and 8 scattered 12-byte gathers per
// particle.  Gradient + readout before -> here, one force evaluation: 256^3
// (a = 0.1 to 1) 327 -> 255 us, 512^3 (a = 0.5, with the copies of a first
// step) 2760 -> 2290, 16 x 64^3 73 -> 55, 64^3 10.5 -> 9.6, 32^3 8 -> 6.7.
#pragma once
#include "pmx_internal.h"

namespace pmx {

constexpr float kD1 = 2.0f / 3.0f, kD2 = 1.0f / 12.0f;
static __device__ __forceinline__ float dstencil(float m2, float m1, float p1,
                                                 float p2) {
  return kD1 * (p1 - m1) - kD2 * (p2 - m2);
}

// n / d by one high multiplication with m = ceil(2^32 / d), d >= 2: exact while
// n d < 2^32 (here n < 2^14 quads, d < 2^12)
static __device__ __forceinline__ unsigned magic(unsigned d) {
  return 0xffffffffu / d + 1u;
}

static __device__ __forceinline__ bool finite_pos(float x, float y, float z) {
  return fabsf(x) < 1.0e9f && fabsf(y) < 1.0e9f && fabsf(z) < 1.0e9f;
}

// (a caller's tape, and the potentials in it, may lie at any float)
typedef float V4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float V2 __attribute__((ext_vector_type(2)));
typedef float V2u __attribute__((ext_vector_type(2), aligned(4)));

// Gradient readout at one particle: the differences at the 8 corners of its
// cell and their weighted sum, in the corner order of cic.hip.
// pair(a, b, c) is the potential at the lower corner + (a, b, c) and
// + (a, b, c + 1), a, b, c in -2 .. 3 with one of a, b outside 0 .. 1 only
// where c = 0: 28 loads of two values for the 56 cells of the differences,
// which are those of k_grad_mesh, as the sum is k_readout_kick_drift's.
template <class Pair>
static __device__ __forceinline__ void grad_readout(const Pair& pair, float x,
                                                    float y, float z,
                                                    float (&out)[3]) {
  constexpr int OX[8] = {0, 1, 0, 0, 1, 1, 0, 1};
  constexpr int OY[8] = {0, 0, 1, 0, 1, 0, 1, 1};
  constexpr int OZ[8] = {0, 0, 0, 1, 0, 1, 1, 1};
  V2 vx[6][2], vy[2][6], vz[2][2][3];
#pragma unroll
  for (int e = 0; e < 6; ++e)
#pragma unroll
    for (int b = 0; b < 2; ++b) vx[e][b] = pair(e - 2, b, 0);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int e = 0; e < 6; ++e)
      vy[a][e] = e == 2 || e == 3 ? vx[a + 2][e - 2] : pair(a, e - 2, 0);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      vz[a][b][0] = pair(a, b, -2);
      vz[a][b][1] = vx[a + 2][b];
      vz[a][b][2] = pair(a, b, 2);
    }
  const float fx = floorf(x), fy = floorf(y), fz = floorf(z);
  const float wx[2] = {1.0f - fabsf(x - fx), 1.0f - fabsf(x - (fx + 1.0f))};
  const float wy[2] = {1.0f - fabsf(y - fy), 1.0f - fabsf(y - (fy + 1.0f))};
  const float wz[2] = {1.0f - fabsf(z - fz), 1.0f - fabsf(z - (fz + 1.0f))};
  float ax = 0.f, ay = 0.f, az = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int a = OX[q], b = OY[q], c = OZ[q];
    const float k = (wx[a] * wy[b]) * wz[c];
    ax += dstencil(vx[a][b][c], vx[a + 1][b][c], vx[a + 3][b][c],
                   vx[a + 4][b][c]) * k;
    ay += dstencil(vy[a][b][c], vy[a][b + 1][c], vy[a][b + 3][c],
                   vy[a][b + 4][c]) * k;
    const V2* const l = vz[a][b];
    az += dstencil(l[c / 2][c % 2], l[(c + 1) / 2][(c + 1) % 2],
                   l[(c + 3) / 2][(c + 3) % 2], l[(c + 4) / 2][(c + 4) % 2]) *
          k;
  }
  out[0] = ax;
  out[1] = ay;
  out[2] = az;
}

// element e of the 12-byte record at byte offset off of a uniform base: one
// 32-bit address register
static __device__ __forceinline__ float ldo(const float* base, unsigned off,
                                            int e) {
  return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) +
                                        off)[e];
}
static __device__ __forceinline__ void sto(float v, float* base, unsigned off,
                                           int e) {
  reinterpret_cast<float*>(reinterpret_cast<char*>(base) + off)[e] = v;
}

constexpr int kBoxT = 512;  // 4 particles per thread, one after the other
static_assert(kWalkRounds * kBoxT == 2048, "bricks hold up to 2048 particles");
// LDS window, floats: two workgroups per CU.  A box longer than it is taken in
// x windows that overlap by 5 planes: with 13568 floats and three workgroups
// (80 VGPRs) the late boxes take two, 287 us against 262 at 256^3.
constexpr int kBoxWin = 20224;

// A box of mesh cells in the LDS window: planes of py rows of nzq quads, row
// pitch pz floats, plane pitch plane floats.
struct Box {
  int z0, nzq, y0, py, x0, px;  // first cells (unwrapped) and lengths
  int pz, plane;
};
// the cells lo - h .. lo + ext - 1 + h per axis (ext: lower corners and their
// upper neighbours), in z widened to whole quads from a multiple of 4 on.
// The row pitch is odd (the fill's rows start on other banks), the plane
// pitch 16 mod 64: the 4 planes a wave's 4 x 16 lanes read start 16 banks
// apart.
static __device__ __forceinline__ Box make_box(const int (&lo)[3],
                                               const int (&ext)[3], int h) {
  Box q;
  q.x0 = lo[0] - h;
  q.px = ext[0] + 2 * h;
  q.y0 = lo[1] - h;
  q.py = ext[1] + 2 * h;
  q.z0 = (lo[2] - h) & ~3;
  q.nzq = (lo[2] + ext[2] + h - q.z0 + 3) >> 2;
  q.pz = 4 * q.nzq + 1;
  q.plane = ((q.py * q.pz + 47) & ~63) + 16;
  return q;
}

// i modulo n, of an i that is mostly in range or one side off (a scalar
// division is some 40 instructions of the scalar unit the whole CU shares)
static __device__ __forceinline__ int near_mod(int i, int n) {
  if (i < 0) i += n;
  if (i >= n) i -= n;
  if ((unsigned)i >= (unsigned)n) i = imod(i, n);
  return i;
}

// Planes s0 .. s0 + np - 1 of the box of mesh pm into win: the quads of all
// rows in one sequence, T at a time, U loads in flight per thread.
// ONCE: rows and planes wrap at most once (the box is not longer than the
// sides).
template <int T, bool ONCE>
static __device__ __forceinline__ void fill_box(float* win, const float* pm,
                                                const MeshDims& d,
                                                const Box& q, int s0, int np) {
  constexpr int U = 4;
  const unsigned x0 = near_mod(q.x0 + s0, d.nx), y0 = near_mod(q.y0, d.ny),
                 z0 = near_mod(q.z0, d.nz);
  const unsigned nx = d.nx, ny = d.ny, nz = d.nz;
  const int quads = np * q.py * q.nzq;
  const unsigned my = magic(q.py), mz = magic(q.nzq);
  for (int i0 = threadIdx.x; i0 < quads; i0 += T * U) {
    V4 v[U];
    int at[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned i = min(i0 + u * T, quads - 1);
      const unsigned r = __umulhi(i, mz), zq = i - r * q.nzq;
      const unsigned xx = __umulhi(r, my), yy = r - xx * q.py;
      at[u] = (int)(xx * q.plane + yy * q.pz + 4 * zq);
      unsigned x = x0 + xx, y = y0 + yy, z = z0 + 4 * zq;
      if (ONCE) {
        x = min(x, x - nx);
        y = min(y, y - ny);
        z = min(z, z - nz);
      } else {
        x %= nx;
        y %= ny;
        z %= nz;
      }
      // 32-bit byte offset: a member has at most 2^30 cells
      v[u] = *reinterpret_cast<const V4*>(reinterpret_cast<const char*>(pm) +
                                          4u * ((x * ny + y) * nz + z));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i0 + u * T < quads) {
        float* const w = win + at[u];
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = v[u][e];
      }
    }
  }
}

// potential pairs of the cell whose lower corner is (ix, iy, iz), from the
// mesh itself: the wrapped offsets of the 6 planes and rows and of the 3 pairs
// of cells, taken once.  A pair is one 8-byte load; the few that wrap between
// their cells take the second one by itself (two 4-byte loads each: 256^3 with 4
// cells rms of noise 7970 us a force, so 7709; two members of 12 x 256 x 256
// with 1 cell, a run of two steps, 1333 / 1212).
struct MeshPair {
  const float* pm;
  unsigned ox[6], oy[6], oz[6];
  unsigned last;  // the last cell of a row
  __device__ __forceinline__ MeshPair(const float* pm_, int ix, int iy, int iz,
                                      const MeshDims& d)
      : pm(pm_), last(d.nz - 1) {
    axis(ox, ix, d.nx, (unsigned)d.ny * d.nz);
    axis(oy, iy, d.ny, (unsigned)d.nz);
    axis(oz, iz, d.nz, 1u);
  }
  static __device__ __forceinline__ void axis(unsigned (&o)[6], int i, int n,
                                              unsigned stride) {
    // sides are 8 or more: - 2 .. 3 wraps at most once
    const int w = near_mod(i, n);
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      int v = w + e - 2;
      v = v < 0 ? v + n : (v >= n ? v - n : v);
      o[e] = (unsigned)v * stride;
    }
  }
  __device__ __forceinline__ V2 operator()(int a, int b, int c) const {
    const float* const r = pm + (ox[a + 2] + oy[b + 2]);
    const unsigned z = oz[c + 2];
    V2 v = *reinterpret_cast<const V2u*>(r + min(z, last - 1));
    if (z == last) v = V2{v.y, *r};
    return v;
  }
};
// The same readout from the packed force mesh of the member: three values at each
// corner, in the same order.
static __device__ __forceinline__ void mesh_readout(const float* m, int ix,
                                                    int iy, int iz, float x,
                                                    float y, float z,
                                                    const MeshDims& d,
                                                    float (&out)[3]) {
  constexpr int OX[8] = {0, 1, 0, 0, 1, 1, 0, 1};
  constexpr int OY[8] = {0, 0, 1, 0, 1, 0, 1, 1};
  constexpr int OZ[8] = {0, 0, 0, 1, 0, 1, 1, 1};
  const int n[3] = {d.nx, d.ny, d.nz};
  const int i[3] = {ix, iy, iz};
  unsigned o[3][2];
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const unsigned w = (unsigned)near_mod(i[e], n[e]);
    o[e][0] = w;
    o[e][1] = w + 1 == (unsigned)n[e] ? 0u : w + 1;
  }
  float v[8][3];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float* const g =
        m + 3LL * ((o[0][OX[q]] * (unsigned)d.ny + o[1][OY[q]]) *
                       (unsigned)d.nz + o[2][OZ[q]]);
#pragma unroll
    for (int e = 0; e < 3; ++e) v[q][e] = g[e];
  }
  const float fx = floorf(x), fy = floorf(y), fz = floorf(z);
  const float wx[2] = {1.0f - fabsf(x - fx), 1.0f - fabsf(x - (fx + 1.0f))};
  const float wy[2] = {1.0f - fabsf(y - fy), 1.0f - fabsf(y - (fy + 1.0f))};
  const float wz[2] = {1.0f - fabsf(z - fz), 1.0f - fabsf(z - (fz + 1.0f))};
  out[0] = out[1] = out[2] = 0.0f;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float k = (wx[OX[q]] * wy[OY[q]]) * wz[OZ[q]];
#pragma unroll
    for (int e = 0; e < 3; ++e) out[e] += v[q][e] * k;
  }
}
// and from a window whose cell (ix - 2, iy - 2, iz - 2) is w
struct WinPair {
  const float* w;
  int plane, pz;
  __device__ __forceinline__ V2 operator()(int a, int b, int c) const {
    return *reinterpret_cast<const V2u*>(w + (a + 2) * plane + (b + 2) * pz +
                                         c + 2);
  }
};

// META: the bricks' boxes are those the paint of the same positions stored
// (paint.hip), so the potential and the particles are loaded together;
// otherwise the workgroup finds the box first.
// PLAIN: none of the copies of a tape, of a first step or of kept positions.
template <bool META, bool PLAIN>
__global__ __launch_bounds__(kBoxT, 4) void k_readout_box(
    float* X, float* P, float* F, const float* __restrict__ phi,
    const int* __restrict__ meta, BoxlessMesh b3, MeshDims d, BrickGrid g,
    KickDrift c, int rounds_each) {
  __shared__ float win[kBoxWin];
  __shared__ int red[META ? 1 : kBoxT / 64][6];
  const int tid = threadIdx.x;
  const int bid = xcd_block32(blockIdx.x, gridDim.x);
  const int b = blockIdx.y;
  // this workgroup's rounds of kBoxT particles
  const int ua = blockIdx.z * rounds_each, ub = ua + rounds_each;
  int q0[3], cnt[3];
  brick_block(g, bid, q0, cnt);
  // z fastest, then x: the 4 rows of a wave are a plane apart in LDS
  const BrickWalk wk = brick_walk(g, cnt, kBoxT);
  const int nloc = wk.nloc;
  // the brick's first particle (uniform); particle t of the brick is poff(t)
  // bytes from there
  const long long o0 =
      3 * ((long long)b * d.N +
           ((long long)q0[0] * g.gy + q0[1]) * g.gz + q0[2]);
  auto poff = [&](int t) { return 12u * walk_at(wk, t); };
  const bool kick = c.do_k2 || c.do_k1d;
  const bool useP = kick || (!PLAIN && c.copy_xp);
  const float* const Xl = (c.xin ? c.xin : X) + o0;
  const float* const Pl = (c.pin ? c.pin : P) + o0;
  const unsigned t_first = walk_at(wk, tid + ua * kBoxT);
  unsigned tn = t_first, on = 12u * tn;
  float xn[3], pn[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 3; ++e) xn[e] = ldo(Xl, on, e);
  if (useP) {
#pragma unroll
    for (int e = 0; e < 3; ++e) pn[e] = ldo(Pl, on, e);
  }
  int lo[3], ext[3];  // first cell and extent of the brick's deposits
  bool boxed;
  if (META) {
    const int* m = meta + 8LL * ((long long)b * g.nbricks + bid);
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      lo[e] = m[e];
      ext[e] = m[3 + e];
    }
    boxed = ext[0] > 0;
  } else {
    int hi[3] = {INT_MIN, INT_MIN, INT_MIN};
    lo[0] = lo[1] = lo[2] = INT_MAX;
    for (int t = tid; t < nloc; t += kBoxT) {
      const unsigned o = poff(t);
      const float x[3] = {ldo(Xl, o, 0), ldo(Xl, o, 1), ldo(Xl, o, 2)};
      if (!finite_pos(x[0], x[1], x[2])) continue;
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const int f = (int)floorf(x[e]);
        lo[e] = min(lo[e], f);
        hi[e] = max(hi[e], f);
      }
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) {
#pragma unroll
      for (int k = 32; k > 0; k >>= 1) {
        lo[e] = min(lo[e], __shfl_xor(lo[e], k));
        hi[e] = max(hi[e], __shfl_xor(hi[e], k));
      }
      if ((tid & 63) == 0) {
        red[META ? 0 : tid >> 6][e] = lo[e];
        red[META ? 0 : tid >> 6][3 + e] = hi[e];
      }
    }
    __syncthreads();
    boxed = true;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      int l = red[0][e], h = red[0][3 + e];
#pragma unroll
      for (int w = 1; w < (META ? 1 : kBoxT / 64); ++w) {
        l = min(l, red[w][e]);
        h = max(h, red[w][3 + e]);
      }
      l = __builtin_amdgcn_readfirstlane(l);
      h = __builtin_amdgcn_readfirstlane(h);
      // wider than the window in any case: not boxed
      boxed = boxed && l <= h && (long long)h - l < 4096;
      lo[e] = boxed ? l : 0;
      ext[e] = boxed ? h - l + 2 : 0;
    }
  }
  const Box q = make_box(lo, ext, 2);
  // planes per window; a particle needs 6
  const int hx =
      boxed && 6 * q.plane <= kBoxWin ? min(q.px, kBoxWin / q.plane) : 0;
  const float* const pm =
      phi + (long long)b * ((long long)d.nx * d.ny * d.nz);
  const long long tot = (long long)d.B * d.N;
  const float* const m3 =
      hx < 6 && b3.mesh && *b3.count >= b3.need
          ? b3.mesh + 3LL * b * ((long long)d.nx * d.ny * d.nz)
          : nullptr;
  // without a box every particle reads the mesh, in one round
  const int rounds = hx >= 6 ? q.px - 5 : 1, step = hx >= 6 ? hx - 5 : 1;
  unsigned done = 0;
  for (int s0 = 0; s0 < rounds; s0 += step) {
    int nxw = 0;
    if (hx >= 6) {
      nxw = min(hx, q.px - s0);
      if (s0 > 0) __syncthreads();  // the window is reused
      if (q.px <= d.nx && q.py <= d.ny && 4 * q.nzq <= d.nz)
        fill_box<kBoxT, true>(win, pm, d, q, s0, nxw);
      else
        fill_box<kBoxT, false>(win, pm, d, q, s0, nxw);
      __syncthreads();
    }
#pragma unroll 1
    for (int u = ua; u < ub; ++u) {
      const int t = tid + u * kBoxT;
      const unsigned o = on;
      float x[3], p[3];
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        x[e] = xn[e];
        p[e] = pn[e];
      }
      // the next particle's loads (the first one's again for a next window)
      tn = u == ub - 1 ? t_first : walk_next(wk, tn, t);
      on = 12u * tn;
#pragma unroll
      for (int e = 0; e < 3; ++e) xn[e] = ldo(Xl, on, e);
      if (useP) {
#pragma unroll
        for (int e = 0; e < 3; ++e) pn[e] = ldo(Pl, on, e);
      }
      if (t >= nloc || (done >> u & 1)) continue;
      float r[3] = {0.f, 0.f, 0.f};
      if (finite_pos(x[0], x[1], x[2])) {
        const int ix = (int)floorf(x[0]), iy = (int)floorf(x[1]),
                  iz = (int)floorf(x[2]);
        if (hx >= 6) {
          const int i = ix - lo[0] - s0;
          if (i < 0 || i + 5 >= nxw) continue;  // another window's
          grad_readout(WinPair{win + i * q.plane + (iy - lo[1]) * q.pz +
                                   (iz - 2 - q.z0),
                               q.plane, q.pz},
                       x[0], x[1], x[2], r);
        } else if (m3) {
          mesh_readout(m3, ix, iy, iz, x[0], x[1], x[2], d, r);
        } else {
          grad_readout(MeshPair(pm, ix, iy, iz, d), x[0], x[1], x[2], r);
        }
      }
      done |= 1u << u;
#pragma unroll
      for (int e = 0; e < 3; ++e) r[e] *= c.fac;
      auto store = [&](const float (&v)[3], float* q) {
#pragma unroll
        for (int e = 0; e < 3; ++e) sto(v[e], q + o0, o, e);
      };
      if (!c.skip_f) store(r, F);
      if (!PLAIN) {
        if (c.xkeep) store(x, c.xkeep);
        if (c.copy_xp) {
          store(x, X);
          store(p, P);
        }
        if (c.ckpt) {
          store(x, c.ckpt);
          store(r, c.ckpt + 6 * tot);
        }
      }
      if (kick) {
        if (c.do_k2) {
#pragma unroll
          for (int e = 0; e < 3; ++e) p[e] = p[e] + c.k2 * r[e];
        }
        if (!PLAIN && c.ckpt) store(p, c.ckpt + 3 * tot);
        if (c.do_k1d) {
#pragma unroll
          for (int e = 0; e < 3; ++e) {
            p[e] = p[e] + c.k1 * r[e];
            x[e] = x[e] + c.d * p[e];
          }
          store(x, c.xout ? c.xout : X);
          if (!PLAIN && c.xcopy) store(x, c.xcopy);
        }
        store(p, P);
      }
    }
  }
}

bool readout_box_ok(const MeshDims& d, const KickDrift& c) {
  return c.f == 1.0f && c.gx == d.nx && c.gy == d.ny && c.gz == d.nz &&
         d.nz % 4 == 0 && (long long)d.nx * d.ny * d.nz == d.N;
}

int launch_readout_box(float* X, float* P, float* F, const float* phi,
                       const int* meta, const BoxlessMesh& b3,
                       const MeshDims& d, const KickDrift& c, hipStream_t s) {
  if ((long long)d.B * d.N == 0) return kOk;
  PMX_REQUIRE(readout_box_ok(d, c), "readout_box: one particle per cell");
  ProfScope prof_(kProfReadoutKD, s);
  const BrickGrid g = make_brick_grid(d.nx, d.ny, d.nz, 1);
  const bool plain = !c.xkeep && !c.copy_xp && !c.ckpt && !c.xcopy;
  auto kern = meta ? (plain ? k_readout_box<true, true>
                            : k_readout_box<true, false>)
                   : (plain ? k_readout_box<false, true>
                            : k_readout_box<false, false>);
  // few bricks, which leave most of the chip idle: their particles by several
  // workgroups, each with the whole box: 32 bricks (32^3) 10.8 us by one, 7.9
  // by two, 6.7 by four; 128 (64^3) 12.8 / 9.6 / 11.2; 2048 55 / 68 / 96
  const long long nb = (long long)g.nbricks * d.B;
  const int parts = nb <= 64 ? 4 : (nb <= 128 ? 2 : 1);
  hipLaunchKernelGGL(kern, dim3(g.nbricks, d.B, parts), dim3(kBoxT), 0, s, X,
                     P, F, phi, meta, b3, d, g, c, kWalkRounds / parts);
  PMX_LAUNCH_CHECK();
  return kOk;
}

}  // namespace pmx
