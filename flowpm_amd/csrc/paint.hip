// Atomic-free CIC paint of a Lagrangian particle grid ("brick paint").
//
// Same deposit as flowpm/utils.py:32-91 (8 corners, weight (wx*wy)*wz times
// the particle weight, periodic wrap), organised for gfx950:
//
// phase 1 (k_brick_deposit): one workgroup per Lagrangian brick of
//   particles (e.g. 8x16x16).  Particles that start close stay close, so
//   the brick's deposits fit a small box.  The workgroup finds the box,
//   accumulates the 8 deposits per particle in LDS (in x slabs when the box
//   exceeds the 39.5 KB window) as 32-bit fixed point
//   (integer LDS atomics run several times faster than float ones on
//   gfx950, and integer sums do not depend on their order), and stores the
//   dense box, converted back to float, to a piece of the arena of its own.
//   The fixed-point scale is a power of two chosen per brick and channel from
//   the sum S of the channel's |weights| so no cell can overflow: the scale
//   is 2^(30 - ex) with S = m 2^ex, m in [0.5, 1), so one deposit is rounded
//   by at most half a unit, 2^(ex - 31) <= 2^-30 S.  That unit is coarse where
//   a cell holds little of S: of boxes beyond 64 KB (which at first were added
//   to the mesh as floats) the mesh would be off by 3.4e-6 rms of itself.
//   Those are accumulated in doubles, as whole numbers of the unit 2^(ex - 52)
//   (exact, so in any order): 3.4e-8.  Twice the passes, in a few bricks:
//   force and gradient at 256^3, a = 1, 2157 -> 2166 us; where the few bricks
//   are the last ones to end, 3-channel deposit at 128 x 160 x 96 22.7 -> 31.1
//   (64-bit integers 36.6: a conversion takes some 12 instructions).
//   Every brick has a 64 KB piece of the arena per channel; a larger box, up
//   to 128 KB (of many particles: box_max), goes to a pool of 8 KB per brick
//   (where a box lies does not change what is in it).  Without the pool the
//   late boxes beyond their pieces spilled: at 256^3, a = 1, 100 us of float
//   atomics per density paint and 231 per three-channel one.
//   A brick whose box is larger still, or finds the pool full, falls back to
//   device-scope float atomics into the finished mesh (k_brick_spill, after
//   phase 2).
// phase 2 (k_brick_gather): one workgroup per mesh tile (4, 8 or 16 x planes
//   of 16 x 16 cells) evaluates the candidate bricks in parallel, compacts
//   those whose boxes meet the tile (in candidate order), and every wave adds
//   them, in that order, to the x planes it owns; the tile is written with
//   plain stores, no barrier per brick, so the mesh is never cleared first.
//
// Device-scope float atomics cannot complete inside one XCD's L2 (the eight
// L2s are not coherent with each other), so the plain scatter pays a far
// memory transaction per deposit; here the mesh sees none in the common
// case.  C = 1 is the density paint, C = 3 the weighted paint of the force
// VJP (three mesh cotangents at once).
#include <type_traits>

#include "pmx_internal.h"

namespace pmx {

struct BrickArgs {
  float* mesh[3];        // C output meshes [B][nx][ny][nz] (overwritten)
  float* arena;          // box arena
  const float* base;     // C = 1: the mesh the paint is added to, or null
  int own_r;             // the gather finds its largest R itself
  int vec4;              // the gather may store the mesh 16 bytes at a time
  int* meta;             // 8 ints per brick: lo[3], ext[3], R (how far the
                         // box reaches past the brick), where its box lies in
                         // the arena (16-float units; kNoBox: it spills)
  int* ctr;              // [kCtrPool] the pool's fill count, [kCtrR] the
                         // largest R; zero before and after every paint.
                         // [kCtrBoxless] bricks without a box, left for the
                         // readout until the next paint's gather clears it
  const float* X;        // positions [B][N][3]
  const float* w;        // weights [B][N][wstride] or null
  int wstride;
  float wscale;
  float ps;              // position scale (pm_nc_factor)
  MeshDims d;            // mesh dims and N
  BrickGrid g;
};

constexpr int kNoBox = -1;
// The arena: a piece of kBoxFloats (and a little, so that the pieces do not all
// start on the same memory channels: 256^3 with 1 cell rms of noise 220 -> 216
// us) per brick and channel, and kPoolFloats of each as a pool for the boxes
// beyond that, handed out by a fill count.  (Every brick taking what it needs
// from the count would pack the arena, but 8192 returning device-scope atomics
// on one line take 400 us.  With pieces of 56 KB and the pool cut out of them,
// states whose boxes are mostly around 60 KB filled the pool and spilled: 256^3
// with 1.8 cells rms of noise 1003 us, 327 here.)
constexpr int kPieceFloats = kBoxFloats + 272, kPoolFloats = 2048;
constexpr int kCtrPool = 0, kCtrR = 2, kCtrInts = 8;  // (the fill: 64 bits)
constexpr int kCtrBoxless = 4;

// Reductions along a wave by DPP moves (no LDS traffic): the result of the
// first 8 << k lanes of a row ends up in the last of them; wave_* in lane 63.
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp_from(int old, int v) {
  return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xf, false);
}
// (lanes without a source take the identity, so that each step is one
// instruction with a DPP operand)
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp_min(int v) {
  return min(v, dpp_from<CTRL, ROWS>(INT_MAX, v));
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp_max(int v) {
  return max(v, dpp_from<CTRL, ROWS>(INT_MIN, v));
}
__device__ __forceinline__ int min8(int v) {
  return dpp_min<0x114>(dpp_min<0x112>(dpp_min<0x111>(v)));  // row_shr
}
__device__ __forceinline__ int max8(int v) {
  return dpp_max<0x114>(dpp_max<0x112>(dpp_max<0x111>(v)));
}
__device__ __forceinline__ int wave_min(int v) {
  // then row_shr 8, row_bcast 15, row_bcast 31
  return dpp_min<0x143, 0xc>(dpp_min<0x142, 0xa>(dpp_min<0x118>(min8(v))));
}
__device__ __forceinline__ int wave_max(int v) {
  return dpp_max<0x143, 0xc>(dpp_max<0x142, 0xa>(dpp_max<0x118>(max8(v))));
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(dpp_from<CTRL, ROWS>(0, __float_as_int(v)));
}
__device__ __forceinline__ float sum8(float v) {
  return dpp_add<0x114>(dpp_add<0x112>(dpp_add<0x111>(v)));
}
__device__ __forceinline__ float wave_sum(float v) {
  return dpp_add<0x143, 0xc>(dpp_add<0x142, 0xa>(dpp_add<0x118>(sum8(v))));
}

__device__ __forceinline__ bool ok_pos(float x, float y, float z) {
  return fabsf(x) < 1.0e9f && fabsf(y) < 1.0e9f && fabsf(z) < 1.0e9f;
}

// deposit workgroup: 512 threads (8 waves; four workgroups per CU give 32
// waves to hide the loads and the LDS atomics), 4 particles per thread;
// bricks hold <= 2048 particles.  A box is accumulated through an LDS window
// of kWinFloats ints: four windows and the workgroups' other LDS fit a CU's
// 160 KB; a larger box is deposited in slabs of whole x planes, one pass over
// the particles per slab and channel.
constexpr int kDT = 512;
constexpr int kWinFloats = 10112;
constexpr int kDW = kDT / 64;
constexpr int kPPT = 2048 / kDT;
// The largest box of a brick of nloc particles.  Those of a finer force mesh
// have 256 (f = 2) or 32 (f = 4): added one by one they cost less than the many
// passes over a large box take the workgroup, which ends last.  Force and
// gradient, boxes up to 128 / 80 / 64 KB in us: 64 x 80 x 48, f = 2, a = 1 261.5
// / 263.7 / 270; grids with 2 spacings rms of noise, f = 2 32^3 191 / 172 / 168,
// 64^3 604 / 562 / 565, 64 x 80 x 48 604 / 594 / 565; f = 4, 1 spacing 32^3 278 /
// 274 / 251, 64^3 1620 / 1602 / 1561.
PMX_HD long long box_max(int nloc) {
  return nloc <= 64    ? kBoxFloats
         : nloc <= 512 ? 5 * kBoxFloats / 4
                       : 2 * kBoxFloats;
}
static_assert(kDW == 8, "the workgroup reductions take 8 waves");

// four consecutive floats of a box row, at any dword
typedef float Vec4u __attribute__((ext_vector_type(4), aligned(4)));

// A deposit is bound by its VALU work, then the LDS atomics (8 per particle
// and channel).  Particles a constant stride apart instead of two divisions
// each, DPP instead of permute reductions, the box set up by every wave from
// one LDS read instead of by one thread between two barriers, clearing and
// storing 16 bytes at a time, and the three channels unrolled: density at
// 256^3 105 -> 92 us, 16 x 64^3 28.4 -> 24.7, three channels at a = 1 in 256^3
// 296 (a twelfth of the boxes not among them) -> 271, 128 x 160 x 96 31 -> 22.
// (The three channels in one pass, so that the corner weights are formed once,
// leave each a third of the window and take 381 us; the loop over them not
// unrolled takes 360.)
template <int C>
// (launch bounds: at least 8 waves per SIMD, i.e. at most 64 VGPRs, so that
// four 512-thread workgroups share a CU; their LDS windows fit its 160 KB)
__global__ __launch_bounds__(kDT, 8) void k_brick_deposit(BrickArgs a) {
  __shared__ __align__(16) int box[kWinFloats];  // fixed-point accumulators
  __shared__ int red[6 * kDW];
  __shared__ float redw[C * kDW];
  __shared__ int sh_off;
  const BrickGrid& g = a.g;
  // XCD-aware: each XCD deposits one contiguous run of bricks, so the
  // cache lines that z-neighbouring bricks share are fetched into one L2
  const int bid = xcd_block32(blockIdx.x, gridDim.x);
  const int b = blockIdx.y;
  const int tid = threadIdx.x, ln = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float ps = a.ps;
  int q0[3], cnt[3];
  brick_block(g, bid, q0, cnt);
  const int cy = cnt[1], cz = cnt[2], nloc = cnt[0] * cy * cz;
  // the brick's first particle (uniform) and each particle's offset from it;
  // in bricks of whole rounds of kDT particles a constant apart
  const long long p0 = (long long)b * a.d.N +
                       ((long long)q0[0] * g.gy + q0[1]) * g.gz + q0[2];
  const bool even = nloc == kDT * kPPT && kDT % (cy * cz) == 0;
  const unsigned pstep =
      even ? (unsigned)(kDT / (cy * cz)) * g.gy * g.gz : 0u;
  const float rz = 1.0f / (float)cz, ry = 1.0f / (float)cy;
  auto part = [&](int t) {
    // exact divisions: t < 2048, and (t + 1/2) / c is 1 / 2c off a whole
    // number
    const int q = (int)(((float)t + 0.5f) * rz), lz = t - q * cz,
              lx = (int)(((float)q + 0.5f) * ry), ly = q - lx * cy;
    return (unsigned)((lx * g.gy + ly) * g.gz + lz);
  };
  const float* const X0 = a.X + 3 * p0;
  const float* const w0 = a.w ? a.w + p0 * a.wstride : nullptr;
  // every load issued up front, branch-free: lanes past the brick's end load
  // its first particle and drop it; the weight test is one uniform branch
  float px[kPPT], py[kPPT], pz[kPPT], wc[kPPT][C];
  unsigned q[kPPT];
  bool ok[kPPT];
  q[0] = part(tid < nloc ? tid : 0);
#pragma unroll
  for (int u = 0; u < kPPT; ++u) {
    const int t = tid + u * kDT;
    ok[u] = t < nloc;
    if (u > 0) q[u] = even ? q[u - 1] + pstep : part(ok[u] ? t : 0);
    px[u] = X0[3 * q[u]];
    py[u] = X0[3 * q[u] + 1];
    pz[u] = X0[3 * q[u] + 2];
  }
  if (a.w) {
#pragma unroll
    for (int u = 0; u < kPPT; ++u)
#pragma unroll
      for (int c = 0; c < C; ++c) wc[u][c] = w0[q[u] * a.wstride + c];
  }
  // bounds and sums of |weight|
  int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {INT_MIN, INT_MIN, INT_MIN};
  float sw[C];
#pragma unroll
  for (int c = 0; c < C; ++c) sw[c] = 0.0f;
#pragma unroll
  for (int u = 0; u < kPPT; ++u) {
    px[u] *= ps;
    py[u] *= ps;
    pz[u] *= ps;
    ok[u] = ok[u] && ok_pos(px[u], py[u], pz[u]);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      wc[u][c] = ok[u] ? (a.w ? wc[u][c] * a.wscale : a.wscale) : 0.0f;
      sw[c] += fabsf(wc[u][c]);
    }
    if (ok[u]) {
      const float p[3] = {px[u], py[u], pz[u]};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int f = (int)floorf(p[d]);
        mn[d] = min(mn[d], f);
        mx[d] = max(mx[d], f);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int l = wave_min(mn[d]), h = wave_max(mx[d]);
    if (ln == 63) {
      red[d * kDW + wv] = l;
      red[(3 + d) * kDW + wv] = h;
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const float m = wave_sum(sw[c]);
    if (ln == 63) redw[c * kDW + wv] = m;
  }
  __syncthreads();
  // every wave finishes the reductions: 8 lanes per bound, 8 per channel
  const int rv = red[ln < 6 * kDW ? ln : 0];
  const int rmin = min8(rv), rmax = max8(rv);
  const float rw = sum8(redw[ln < C * kDW ? ln : 0]);
  int lo[3], hi[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    lo[d] = __builtin_amdgcn_readlane(rmin, 8 * d + 7);
    hi[d] = __builtin_amdgcn_readlane(rmax, 8 * d + 31);
  }
  // fixed-point scale 2^e with (sum of |weights|) * 2^e < 2^30: no cell
  // total (nor a partial sum) can leave the int32 range
  float fxs[C], fxinv[C];
  bool wfin = true;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const float swt = __int_as_float(
        __builtin_amdgcn_readlane(__float_as_int(rw), 8 * c + 7));
    int e = 0;
    wfin = wfin && swt <= 3.0e38f;  // false for inf / nan weights
    if (swt <= 3.0e38f && swt > 0.0f) {
      int ex;
      frexpf(swt, &ex);  // swt = m 2^ex, m in [0.5, 1)
      e = min(max(30 - ex, -120), 120);
    }
    // 2^e and 2^-e (|e| <= 120), uniform
    const int es = __builtin_amdgcn_readfirstlane(e);
    fxs[c] = __int_as_float((127 + es) << 23);
    fxinv[c] = __int_as_float((127 - es) << 23);
  }
  const int n[3] = {a.d.nx, a.d.ny, a.d.nz};
  BrickBox bx = brick_box(lo, hi, n, q0, cnt, g.f, wfin, box_max(nloc));
  // (the window has to hold a plane of the deposits' two)
  if (bx.mode == 1 && 2LL * bx.ext[1] * bx.ext[2] > kWinFloats) bx.mode = 2;
  int* const m = a.meta + 8LL * ((long long)b * g.nbricks + bid);
  const bool box_ok = bx.mode == 1;
  const int e0 = bx.ext[0], e1 = bx.ext[1], e2 = bx.ext[2];
  const int vol4 = (int)((bx.vol + 3) & ~3LL);  // channel stride in the arena
  // where the box goes, in 16-float units; a piece of the pool is asked for
  // by thread 0, and its answer used after the first pass
  const long long nb = (long long)gridDim.x * gridDim.y;
  constexpr int kPiece = C * kPieceFloats / 16, kPool = C * kPoolFloats / 16;
  const bool pooled = vol4 > kBoxFloats;
  const int units = (C * vol4 + 15) / 16;
  unsigned long long got = 0;
  if (tid == 0 && box_ok && pooled)
    got = atomicAdd(reinterpret_cast<unsigned long long*>(a.ctr + kCtrPool),
                    (unsigned long long)units);
  if (!box_ok) {
    if (tid == 0) {
      m[3] = m[4] = m[5] = m[6] = 0;
      m[7] = bx.mode == 2 ? kNoBox : 0;
    }
    return;
  }
  // planes per pass; a box of the pool is accumulated in doubles
  const bool wide = pooled;
  const int plane = e1 * e2, hx = (wide ? kWinFloats / 2 : kWinFloats) / plane;
  const bool clip = hx < e0;  // (always, if wide)
  float* dst = nullptr;
  double* const box64 = reinterpret_cast<double*>(box);
  // deposits channel c of the particles; with CLIP those whose corners fall
  // in x planes [x0, x0 + nxw) of the box, else all
  auto deposit = [&](auto clip_, int c, int x0, int nxw) {
    constexpr bool CLIP = decltype(clip_)::value;
    // the positions are opaque here, so the corner weights are computed
    // per pass instead of being kept live across the passes and channels
#pragma unroll
    for (int u = 0; u < kPPT; ++u)
      asm volatile("" : "+v"(px[u]), "+v"(py[u]), "+v"(pz[u]));
#pragma unroll
    for (int u = 0; u < kPPT; ++u) {
      const float x = px[u], y = py[u], z = pz[u];
      const float flx = floorf(x), fly = floorf(y), flz = floorf(z);
      const int ix = (int)flx - lo[0] - x0;
      if (!ok[u] || (CLIP && !(ix >= -1 && ix < nxw))) continue;
      const float w0x = 1.0f - fabsf(x - flx), w1x = 1.0f - fabsf(x - (flx + 1.0f));
      const float w0y = 1.0f - fabsf(y - fly), w1y = 1.0f - fabsf(y - (fly + 1.0f));
      const float w0z = 1.0f - fabsf(z - flz), w1z = 1.0f - fabsf(z - (flz + 1.0f));
      const int at = (ix * e1 + ((int)fly - lo[1])) * e2 + ((int)flz - lo[2]);
      const float wq = wc[u][c] * fxs[c];
#pragma unroll
      for (int ox = 0; ox < 2; ++ox) {
        if (CLIP && (unsigned)(ix + ox) >= (unsigned)nxw) continue;
        const int to = at + ox * plane;
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          v[k] = wq * (((ox ? w1x : w0x) * (k & 2 ? w1y : w0y)) *
                       (k & 1 ? w1z : w0z));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int o = to + (k >> 1) * e2 + (k & 1);
          if (CLIP && wide)
            atomicAdd(box64 + o, (double)rintf(v[k] * 0x1p22f));
          else
            atomicAdd(box + o, __float2int_rn(v[k]));
        }
      }
    }
  };
#pragma unroll
  for (int c = 0; c < C; ++c) {
    for (int x0 = 0; x0 < e0; x0 += hx) {
      const int nxw = min(hx, e0 - x0), nw = nxw * plane;
      const bool first_pass = c == 0 && x0 == 0;
      if (!first_pass) __syncthreads();  // the window is reused
      for (int i = tid; 4 * i < (wide ? 2 * nw : nw); i += kDT)
        reinterpret_cast<int4*>(box)[i] = make_int4(0, 0, 0, 0);
      __syncthreads();
      if (clip)
        deposit(std::true_type{}, c, x0, nxw);
      else
        deposit(std::false_type{}, c, 0, nxw);
      if (first_pass && tid == 0) {
        const bool fits = !pooled || (long long)got + units <= nb * kPool;
        const long long at =
            pooled ? nb * kPiece + (long long)got
                   : ((long long)b * g.nbricks + bid) * kPiece;
        const int off = fits ? (int)(unsigned)at : kNoBox;
        sh_off = off;
        m[0] = lo[0];
        m[1] = lo[1];
        m[2] = lo[2];
        m[3] = fits ? e0 : 0;
        m[4] = fits ? e1 : 0;
        m[5] = fits ? e2 : 0;
        m[6] = fits ? bx.R : 0;
        m[7] = off;
      }
      __syncthreads();
      if (first_pass) {
        const int off = sh_off;
        if (off == kNoBox) return;
        dst = a.arena + 16LL * (unsigned)off;
      }
      const float fi = fxinv[c];
      float* const o = dst + c * vol4 + x0 * plane;
      for (int i = tid; 4 * i < nw; i += kDT) {
        Vec4u r;
        if (wide) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            r[e] = (float)box64[4 * i + e] * 0x1p-22f * fi;
        } else {
          const int4 v = reinterpret_cast<const int4*>(box)[i];
          r = Vec4u{(float)v.x * fi, (float)v.y * fi, (float)v.z * fi,
                    (float)v.w * fi};
        }
        if (4 * i + 4 <= nw) {
          *reinterpret_cast<Vec4u*>(o + 4 * i) = r;
        } else {
          o[4 * i] = r.x;
          if (4 * i + 1 < nw) o[4 * i + 1] = r.y;
          if (4 * i + 2 < nw) o[4 * i + 2] = r.z;
        }
      }
    }
  }
}

// The largest R of the paint, read by the gather (one workgroup).
__global__ __launch_bounds__(1024) void k_brick_reduce(
    const int* __restrict__ meta, long long nb, int* __restrict__ ctr) {
  __shared__ int smax[16];
  int r = 0;
  // 8 bricks per thread and round, all loads issued before the first is used
  // (indices past the end reload the last brick)
  constexpr int U = 8;
  for (long long i0 = threadIdx.x; i0 < nb; i0 += 1024LL * U) {
    int v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = meta[8 * min(i0 + 1024LL * u, nb - 1) + 6];
#pragma unroll
    for (int u = 0; u < U; ++u) r = max(r, v[u]);
  }
#pragma unroll
  for (int k = 32; k > 0; k >>= 1) r = max(r, __shfl_xor(r, k));
  if ((threadIdx.x & 63) == 0) smax[threadIdx.x >> 6] = r;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) r = max(r, smax[w]);
    ctr[kCtrR] = max(r, smax[0]);
  }
}

// the counters of a workspace that no paint has used
__global__ void k_brick_init(int* __restrict__ ctr) {
  if (threadIdx.x < kCtrInts) ctr[threadIdx.x] = 0;
}

// One workgroup of 4 waves per mesh tile of 4 PX x 16 x 16 cells: wave w owns
// the x planes w PX .. w PX + PX - 1, a lane 4 consecutive z cells of one y
// row in each of them, so one 16-byte load per lane covers a whole 16 x 16
// plane of a box.  Bound by the load instructions and, on few tiles, by the
// chain of boxes each wave walks: a wave visits only the boxes that meet its
// own planes (one ballot), and has the loads of kGatherU boxes in flight
// together.  Against a thread per (y, z) column reading 16 x cells one float
// at a time, with the cells outside the box loaded and dropped: density at
// 256^3 122 -> 92 us, 16 x 64^3 38 -> 26, 128^3 37 -> 22, 64^3 28 -> 12.5,
// 32^3 21 -> 7.8; the three channels, which had one float of 4 cells per
// load, gain little: at 128 x 160 x 96 31 -> 29, at 64^3 12.4 -> 12.9.
// The sums, and their order, are the same: so are the results, bit for bit.
constexpr int kGatherU = 2;
template <int C, int PX>
__global__ __launch_bounds__(256) void k_brick_gather(BrickArgs a) {
  constexpr int U = kGatherU;
  constexpr int TX = 4 * PX;
  __shared__ short cand[3][1024];
  __shared__ int ncand[3];
  __shared__ int lst[256][8];  // overlapping bricks of one chunk
  __shared__ int wcnt[4];
  const BrickGrid& g = a.g;
  const MeshDims& d = a.d;
  const int tid = threadIdx.x;
  const int b = blockIdx.y;
  const int ntx = (d.nx + TX - 1) / TX, nty = (d.ny + kTile - 1) / kTile,
            ntz = (d.nz + kTile - 1) / kTile;
  if (blockIdx.x == 0 && b == 0 && tid == 0) a.ctr[kCtrBoxless] = 0;
  const int tt = (int)xcd_block(blockIdx.x, gridDim.x);
  const int tz = tt % ntz, ty = (tt / ntz) % nty, tx = tt / (ntz * nty);
  const int t0x = tx * TX, t0y = ty * kTile, t0z = tz * kTile;
  const int Tx = min(TX, d.nx - t0x), Ty = min(kTile, d.ny - t0y),
            Tz = min(kTile, d.nz - t0z);
  int R = 0;
  if (a.own_r) {
    __shared__ int rmax[4];
    for (int k = tid; k < g.nbricks; k += 256)
      R = max(R, a.meta[8LL * ((long long)b * g.nbricks + k) + 6]);
    R = wave_max(R);
    if ((tid & 63) == 63) rmax[tid >> 6] = R;
    __syncthreads();
    R = max(max(rmax[0], rmax[1]), max(rmax[2], rmax[3]));
  } else {
    R = a.ctr[kCtrR];
  }
  // candidate bricks per dimension (wave w builds list w)
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), ln = tid & 63;
  if (wv < 3) {
    const int e = wv == 0 ? g.ex : (wv == 1 ? g.ey : g.ez);
    const int gd = wv == 0 ? g.gx : (wv == 1 ? g.gy : g.gz);
    const int nb = wv == 0 ? g.nbx : (wv == 1 ? g.nby : g.nbz);
    const int t0 = wv == 0 ? t0x : (wv == 1 ? t0y : t0z);
    const int T = wv == 0 ? Tx : (wv == 1 ? Ty : Tz);
    const int n = wv == 0 ? d.nx : (wv == 1 ? d.ny : d.nz);
    int base = 0;
    for (int k0 = 0; k0 < nb; k0 += 64) {
      const int k = k0 + ln;
      const bool hit = k < nb && brick_hits(k, e, gd, g.f, R, t0, T, n);
      const unsigned long long mask = __ballot(hit);
      if (hit) {
        const int pos = base + __popcll(mask & ((1ULL << ln) - 1ULL));
        if (pos < 1024) cand[wv][pos] = (short)k;
      }
      base += __popcll(mask);
    }
    if (ln == 0) ncand[wv] = min(base, 1024);
  }
  __syncthreads();
  const int nc0 = ncand[0], nc1 = ncand[1], nc2 = ncand[2];
  const int total = nc0 * nc1 * nc2;
  // owned cells: x = x0w + k (k < PX), y = cy, z = cz + i (i < 4)
  const int x0w = t0x + wv * PX;
  const int cy = t0y + (ln >> 2), cz = t0z + 4 * (ln & 3);
  const bool yz_ok = cy < d.ny && cz < d.nz;
  float acc[C][PX][4];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int k = 0; k < PX; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[c][k][i] = 0.0f;
  for (int base = 0; base < total; base += 256) {
    // 1. evaluate one candidate per thread, compact the overlapping ones in
    //    candidate order (ballot within a wave, wave counts across)
    const int ci = base + tid;
    bool ok = false;
    int rec[7];
    if (ci < total) {
      const int i2 = ci % nc2, r = ci / nc2, i1 = r % nc1, i0 = r / nc1;
      const int bid = (cand[0][i0] * g.nby + cand[1][i1]) * g.nbz + cand[2][i2];
      const int4* m = reinterpret_cast<const int4*>(
          a.meta + 8LL * ((long long)b * g.nbricks + bid));
      const int4 ma = m[0], mb = m[1];
      const int e0 = ma.w, e1 = mb.x, e2 = mb.y;
      if (e0 > 0) {
        const int a0 = imod(ma.x, d.nx), a1 = imod(ma.y, d.ny),
                  a2 = imod(ma.z, d.nz);
        ok = box_meets(a0, e0, t0x, Tx, d.nx) &&
             box_meets(a1, e1, t0y, Ty, d.ny) &&
             box_meets(a2, e2, t0z, Tz, d.nz);
        rec[0] = mb.w;
        rec[1] = a0;
        rec[2] = a1;
        rec[3] = a2;
        rec[4] = e0;
        rec[5] = e1;
        rec[6] = e2;
      }
    }
    const unsigned long long mask = __ballot(ok);
    if (ln == 0) wcnt[wv] = __popcll(mask);
    __syncthreads();
    int off = 0, nl = 0;
    for (int w = 0; w < 4; ++w) {
      if (w < wv) off += wcnt[w];
      nl += wcnt[w];
    }
    if (ok) {
      const int pos = off + __popcll(mask & ((1ULL << ln) - 1ULL));
#pragma unroll
      for (int q = 0; q < 7; ++q) lst[pos][q] = rec[q];
    }
    __syncthreads();
    // 2. every wave adds the bricks that meet its planes, in list order, to
    //    its own cells, the loads of U bricks in flight together
    for (int l0 = 0; l0 < nl; l0 += 64) {
      bool meets = false;
      if (l0 + ln < nl) {
        const int a0 = lst[l0 + ln][1], e0 = lst[l0 + ln][4];
#pragma unroll
        for (int k = 0; k < PX; ++k)
          meets = meets || (x0w + k < d.nx && wrap_off(x0w + k, a0, d.nx) < e0);
      }
      unsigned long long todo = __ballot(meets);
      while (todo) {
        float v[U][C][PX][4];
        bool in[U][PX], inz[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const bool any = todo != 0;  // wave-uniform
          const int j = l0 + (any ? __ffsll(todo) - 1 : 0);
          todo &= todo - 1;
          auto rd = [&](int q) {
            return __builtin_amdgcn_readfirstlane(lst[j][q]);
          };
          const int a0 = rd(1), a1 = rd(2), a2 = rd(3), e0 = rd(4), e1 = rd(5),
                    e2 = rd(6);
          const int vol = (e0 * e1 * e2 + 3) & ~3, pl = e1 * e2;
          const float* src = a.arena + 16LL * (unsigned)rd(0);
          const int oy = wrap_off(cy, a1, d.ny);
          const bool yin = any && yz_ok && oy < e1;
          const int o = cz - a2;
          if (e2 <= d.nz - 4) {
            // the four cells lie in one run of box offsets: o .. o + 3 from
            // o = -3 on, o + nz .. below that (nothing of o + i < 0 with
            // o > -4 is in a box this short)
            const int oz = o > -4 ? o : o + d.nz;
            const bool lane = yin && oz < e2;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              inz[u][i] = lane && oz + i >= 0 && oz + i < e2;
            const int bi = lane ? oy * e2 + oz : 0;
#pragma unroll
            for (int k = 0; k < PX; ++k) {
              const int ox = wrap_off(x0w + k, a0, d.nx);
              in[u][k] = x0w + k < d.nx && ox < e0;
              const float* p = src + (in[u][k] ? ox * pl : 0);
#pragma unroll
              for (int c = 0; c < C; ++c) {
                const Vec4u q =
                    *reinterpret_cast<const Vec4u*>(p + c * vol + bi);
                v[u][c][k][0] = q.x;
                v[u][c][k][1] = q.y;
                v[u][c][k][2] = q.z;
                v[u][c][k][3] = q.w;
              }
            }
          } else {
            // a box that nearly spans the mesh: each cell by itself
            int zi[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const bool zok = cz + i < d.nz;
              const int oz = wrap_off(cz + (zok ? i : 0), a2, d.nz);
              inz[u][i] = yin && zok && oz < e2;
              zi[i] = inz[u][i] ? oy * e2 + oz : 0;
            }
#pragma unroll
            for (int k = 0; k < PX; ++k) {
              const int ox = wrap_off(x0w + k, a0, d.nx);
              in[u][k] = x0w + k < d.nx && ox < e0;
              const float* p = src + (in[u][k] ? ox * pl : 0);
#pragma unroll
              for (int c = 0; c < C; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[u][c][k][i] = p[c * vol + zi[i]];
            }
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int k = 0; k < PX; ++k)
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[c][k][i] +=
                    in[u][k] && inz[u][i] ? v[u][c][k][i] : 0.0f;
      }
    }
    __syncthreads();  // lst is rewritten by the next chunk
  }
  if (!yz_ok) return;
  // every cell of the mesh is written here (the mesh needs no clearing);
  // the painted values are added to the base's, if there is one
  const bool whole = a.vec4 && cz + 4 <= d.nz;
#pragma unroll
  for (int k = 0; k < PX; ++k) {
    if (x0w + k < d.nx) {
      const long long cell =
          (((long long)b * d.nx + x0w + k) * d.ny + cy) * d.nz + cz;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        float* out = a.mesh[c] + cell;
        if (whole) {
          float4 r = make_float4(acc[c][k][0], acc[c][k][1], acc[c][k][2],
                                 acc[c][k][3]);
          if (C == 1 && a.base) {
            const float4 o = *reinterpret_cast<const float4*>(a.base + cell);
            r = make_float4(o.x + r.x, o.y + r.y, o.z + r.z, o.w + r.w);
          }
          *reinterpret_cast<float4*>(out) = r;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (cz + i < d.nz)
              out[i] = C == 1 && a.base ? a.base[cell + i] + acc[c][k][i]
                                        : acc[c][k][i];
        }
      }
    }
  }
}

template <int C>
__device__ __forceinline__ void spill_brick(const BrickArgs& a, long long q) {
  const BrickGrid& g = a.g;
  const MeshDims& d = a.d;
  const int b = (int)(q / g.nbricks), bid = (int)(q % g.nbricks);
  int q0[3], cnt[3];
  brick_block(g, bid, q0, cnt);
  const int cy = cnt[1], cz = cnt[2];
  const int nloc = cnt[0] * cy * cz;
  for (int t = threadIdx.x; t < nloc; t += blockDim.x) {
    const int lz = t % cz, r = t / cz, ly = r % cy, lx = r / cy;
    const long long pi =
        (long long)b * d.N +
        ((long long)(q0[0] + lx) * g.gy + (q0[1] + ly)) * g.gz + q0[2] + lz;
    const float x = a.X[3 * pi] * a.ps, y = a.X[3 * pi + 1] * a.ps,
                z = a.X[3 * pi + 2] * a.ps;
    if (!ok_pos(x, y, z)) continue;
    float wc[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
      wc[c] = a.w ? a.w[pi * a.wstride + c] * a.wscale : a.wscale;
    const float flx = floorf(x), fly = floorf(y), flz = floorf(z);
    const float wx[2] = {1.0f - fabsf(x - flx), 1.0f - fabsf(x - (flx + 1.0f))};
    const float wy[2] = {1.0f - fabsf(y - fly), 1.0f - fabsf(y - (fly + 1.0f))};
    const float wz[2] = {1.0f - fabsf(z - flz), 1.0f - fabsf(z - (flz + 1.0f))};
    const int ix = (int)flx, iy = (int)fly, iz = (int)flz;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int ox = k & 1, oy = (k >> 1) & 1, oz = k >> 2;
      const float kw = (wx[ox] * wy[oy]) * wz[oz];
      const long long cell =
          (((long long)b * d.nx + imod(ix + ox, d.nx)) * d.ny +
           imod(iy + oy, d.ny)) * d.nz + imod(iz + oz, d.nz);
#pragma unroll
      for (int c = 0; c < C; ++c) atomicAdd(a.mesh[c] + cell, wc[c] * kw);
    }
  }
}

// Bricks whose box did not fit (too large, or the arena was full; positions
// spread over more than the mesh; non-finite weights) are added to the
// gathered mesh with device-scope float atomics, one thread per particle.
// Every workgroup looks through the flags of its own bricks at once; without
// a marked one it returns after that load.  The pool's and R's counters are
// left zero.
template <int C>
__global__ __launch_bounds__(256) void k_brick_spill(BrickArgs a) {
  if (blockIdx.x == 0 && threadIdx.x < kCtrBoxless) a.ctr[threadIdx.x] = 0;
  const long long nq = (long long)a.d.B * a.g.nbricks;
  for (long long k0 = blockIdx.x; k0 < nq; k0 += 256LL * gridDim.x) {
    const long long mine = k0 + (long long)threadIdx.x * gridDim.x;
    const bool hit = mine < nq && a.meta[8 * mine + 7] == kNoBox;
    const int n = __syncthreads_count(hit);
    if (n == 0) continue;
    if (threadIdx.x == 0) atomicAdd(a.ctr + kCtrBoxless, n);
    for (int w = 0; w < 256; ++w) {
      const long long q = k0 + (long long)w * gridDim.x;
      if (q >= nq) break;
      if (a.meta[8 * q + 7] == kNoBox) spill_brick<C>(a, q);
    }
  }
}

bool brick_paint_ok(const MeshDims& d, const BrickGrid& g) {
  // (the limits on the bricks: brick_block's divisions, the candidate lists)
  return g.ex * g.ey * g.ez <= kDT * kPPT && g.gx * g.f == d.nx &&
         (long long)g.nbx * g.nby * g.nbz < (1LL << 22) &&
         g.gy * g.f == d.ny && g.gz * g.f == d.nz &&
         (long long)g.gx * g.gy * g.gz == d.N && g.nbx <= 1024 &&
         g.nby <= 1024 && g.nbz <= 1024;
}

static long long arena_floats(const MeshDims& d, const BrickGrid& g, int C) {
  return (long long)d.B * g.nbricks * C * (kPieceFloats + kPoolFloats);
}

long long brick_work_floats(const MeshDims& d, const BrickGrid& g, int C) {
  // counters and alignment take the rest
  const long long arena = arena_floats(d, g, C);
  const long long meta = 8LL * d.B * g.nbricks;
  return arena + meta + 16;
}

// The counters come first, at a place that does not depend on C, and the
// arena is 16-byte aligned with at least 3 floats in front: the gather's
// 16-byte loads may start 3 floats before a box (those values are dropped).
static int* brick_ctr(float* work) {
  return reinterpret_cast<int*>(
      (reinterpret_cast<uintptr_t>(work) + 15) & ~uintptr_t(15));
}
static float* brick_arena(float* work) {
  return reinterpret_cast<float*>(brick_ctr(work) + kCtrInts);
}
const int* brick_meta(const MeshDims& d, const BrickGrid& g, int C,
                      float* work) {
  return reinterpret_cast<const int*>(brick_arena(work) +
                                      arena_floats(d, g, C));
}

const int* brick_boxless(float* work) { return brick_ctr(work) + kCtrBoxless; }

int launch_brick_paint(float* const* mesh, int C, const float* X,
                       const float* w, int wstride, float wscale, float ps,
                       const MeshDims& d, const BrickGrid& g, float* work,
                       hipStream_t s, const float* base, bool* ready) {
  if ((long long)d.B * d.N == 0) return kOk;
  BrickArgs a{};
  a.base = base;
  for (int c = 0; c < C; ++c) a.mesh[c] = mesh[c];
  a.arena = brick_arena(work);
  a.meta = const_cast<int*>(brick_meta(d, g, C, work));
  a.ctr = brick_ctr(work);
  if (!ready || !*ready) {
    hipLaunchKernelGGL(k_brick_init, dim3(1), dim3(64), 0, s, a.ctr);
    PMX_LAUNCH_CHECK();
    if (ready) *ready = true;
  }
  a.vec4 = d.nz % 4 == 0 && reinterpret_cast<uintptr_t>(base) % 16 == 0;
  for (int c = 0; c < C; ++c)
    if (reinterpret_cast<uintptr_t>(mesh[c]) % 16 != 0) a.vec4 = 0;
  a.X = X;
  a.w = w;
  a.wstride = wstride;
  a.wscale = wscale;
  a.ps = ps;
  a.d = d;
  a.g = g;
  {
    ProfScope prof_(C == 1 ? kProfPaint : kProfPaintW, s);
    dim3 grid(g.nbricks, d.B);
    if (C == 1)
      hipLaunchKernelGGL(k_brick_deposit<1>, grid, dim3(kDT), 0, s, a);
    else
      hipLaunchKernelGGL(k_brick_deposit<3>, grid, dim3(kDT), 0, s, a);
    PMX_LAUNCH_CHECK();
  }
  // Up to 1024 bricks per member every tile finds the largest R of its member
  // itself, which saves a launch (and 5 us of the host): at 960 bricks the
  // gather takes 1.7 us more (20.1 of 18.4) and the reduction took 4.4, at 128
  // bricks 11.3 of 11.8 and 3.3.  At 8192 it would take 146 us of 95.
  a.own_r = g.nbricks <= 1024;
  if (!a.own_r) {
    hipLaunchKernelGGL(k_brick_reduce, dim3(1), dim3(1024), 0, s, a.meta,
                       (long long)d.B * g.nbricks, a.ctr);
    PMX_LAUNCH_CHECK();
  }
  {
    ProfScope prof_(C == 1 ? kProfPaintGather : kProfPaintWGather, s);
    // tiles of 16 planes where they fill the chip four times over (1024
    // workgroups), else of 8 (two workgroups per CU or more), else of 4: at
    // 1024 tiles of 16 (16 x 64^3) 25.8 us against 29.0 with 8 and 37.8 with
    // 4, at 512 (128^3) 24.4 / 21.5 / 27.2, at 64 (64^3) 17.1 / 13.9 / 12.5.
    // The three channels always take 4, 72 VGPRs against 106 with 8: 312 us
    // against 324 at 256^3, 29.4 against 31.3 at 128 x 160 x 96.
    const long long yz = (long long)((d.ny + kTile - 1) / kTile) *
                         ((d.nz + kTile - 1) / kTile);
    const long long t16 = (d.nx + 15) / 16 * yz * d.B;
    const int px = t16 < 256 || C == 3 ? 1 : (t16 < 1024 ? 2 : 4);
    dim3 grid((unsigned)((d.nx + 4 * px - 1) / (4 * px) * yz), d.B);
    auto kern = C == 1 ? (px == 1   ? k_brick_gather<1, 1>
                          : px == 2 ? k_brick_gather<1, 2>
                                    : k_brick_gather<1, 4>)
                       : k_brick_gather<3, 1>;
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a);
    PMX_LAUNCH_CHECK();
    const long long nq = (long long)d.B * g.nbricks;
    const dim3 sgrid((unsigned)std::min<long long>(nq, 256));
    if (C == 1)
      hipLaunchKernelGGL(k_brick_spill<1>, sgrid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL(k_brick_spill<3>, sgrid, dim3(256), 0, s, a);
    PMX_LAUNCH_CHECK();
  }
  return kOk;
}

}  // namespace pmx

#include "bin_paint.h"
