// Power-series propagator exp(-i H dt) ~ sum_{n<=p} (-i H dt)^n / n! (gfx950).
//
// The reference evaluates the series by the recurrence
//   s_n = (i dt / n) [ (1/2m) L s_{n-1} - V s_{n-1} ],  psi += s_n
// with one kernel launch per term (sources/sim_state.py:721-752,
// sources/cuda_kernels/power_series_operator.cu:3-65).  The same polynomial is
// evaluated here by Horner's rule,
//   u <- psi;  for n = p..1:  u <- psi + (-i dt / n) H u,
// which reads u (stencil), psi and V and writes u once per stage: 32 B per
// point per stage in complex64 instead of 40.
//
// H u = -(1/2m) L u + V u with L the 7-point Laplacian whose neighbour index
// falls back to the voxel itself at a face (edge replication) and whose sum is
// divided by dx_x^2 on every axis (power_series_operator.cu:23-58).
//
// Each thread owns one (y, z) column of a block tile and marches along x over
// a 16-plane slab, keeping u(x-1), u(x), u(x+1) in registers; the y/z
// neighbours come from the same plane, which the block's other lanes load at
// the same time (L1/L2 hits).
#include "wfs_internal.h"

namespace wfs {

// One Horner update at a point: psi + (-i c) (-(1/2m) L u + V u), with L u * dx^2 summed in the
// reference's order.  Shared by the single-stage and the two-stage kernels so that both round
// identically.
template <typename R>
__device__ __forceinline__ cx<R> horner_point(cx<R> cur, cx<R> xm, cx<R> xp, cx<R> ym, cx<R> yp, cx<R> zm,
                                              cx<R> zp, cx<R> ps, float2 v, R c, R inv_2m, R inv_dx2) {
  cx<R> lap;
  lap.x = xm.x + xp.x + ym.x - R(6) * cur.x + yp.x + zm.x + zp.x;
  lap.y = xm.y + xp.y + ym.y - R(6) * cur.y + yp.y + zm.y + zp.y;
  cx<R> hu;
  hu.x = -inv_2m * inv_dx2 * lap.x + (R(v.x) * cur.x - R(v.y) * cur.y);
  hu.y = -inv_2m * inv_dx2 * lap.y + (R(v.x) * cur.y + R(v.y) * cur.x);
  // psi + (-i c) H u = psi + c (Hu.y, -Hu.x)
  cx<R> o;
  o.x = ps.x + c * hu.y;
  o.y = ps.y - c * hu.x;
  return o;
}

template <typename R, int TZ, int TY>
__global__ __launch_bounds__(TZ* TY) void horner_stage_kernel(const cx<R>* __restrict__ u_in, cx<R>* u_out,
                                                             const cx<R>* psi, const float2* __restrict__ V,
                                                             int nx, int ny, int nz, R dt_over_n, R inv_2m,
                                                             R inv_dx2, int tile_x, int ntiles) {
  using C = cx<R>;
  const int z = blockIdx.x * TZ + threadIdx.x;
  const int y = blockIdx.y * TY + threadIdx.y;
  const int packet = blockIdx.z / ntiles;          // independent grids stacked along x
  const int x0 = (blockIdx.z % ntiles) * tile_x;
  if (z >= nz || y >= ny) return;
  const long poff = long(packet) * nx * ny * nz;
  u_in += poff;
  u_out += poff;
  psi += poff;
  V += poff;
  int x1 = x0 + tile_x;
  if (x1 > nx) x1 = nx;
  const long sx = long(ny) * nz;
  const long sy = nz;
  const int zm = z > 0 ? z - 1 : z;
  const int zp = z < nz - 1 ? z + 1 : z;
  const int ym = y > 0 ? y - 1 : y;
  const int yp = y < ny - 1 ? y + 1 : y;

  auto at = [&](int x, int yy, int zz) -> long { return long(x) * sx + long(yy) * sy + zz; };

  C prev = u_in[at(x0 > 0 ? x0 - 1 : x0, y, z)];
  C cur = u_in[at(x0, y, z)];
  for (int x = x0; x < x1; ++x) {
    const C next = u_in[at(x < nx - 1 ? x + 1 : x, y, z)];
    const C uym = u_in[at(x, ym, z)];
    const C uyp = u_in[at(x, yp, z)];
    const C uzm = u_in[at(x, y, zm)];
    const C uzp = u_in[at(x, y, zp)];
    const long i = at(x, y, z);
    u_out[i] = horner_point<R>(cur, prev, next, uym, uyp, uzm, uzp, psi[i], V[i], dt_over_n, inv_2m, inv_dx2);
    prev = cur;
    cur = next;
  }
}

// S Horner stages in one pass (temporal blocking): w_1 = psi + (-i c_1) H u, w_2 = psi +
// (-i c_2) H w_1, ..., u_out = w_S.  A block owns a window of uy x w (y, z) cells -- its output
// tile and a halo of S cells on every side that is not a grid face -- and marches along x.  A
// thread owns a strip of RC rows at one column.  While plane t of u arrives, stage s works on
// plane t - s, so the stages of an iteration read only what earlier iterations left behind:
//   - level s - 1 (u is level 0) holds its plane t - s in one LDS buffer and plane t - s - 1 in the
//     other, which this iteration overwrites: one barrier a plane;
//   - a cell's z neighbours, its centre and its previous plane come from LDS, the y neighbours
//     inside the strip from the thread's own centres, only the rows above and below it from LDS;
//   - the next plane of level s - 1 is the thread's own, computed by stage s - 1 just before (or
//     loaded an iteration ahead for u);
//   - psi and V of a cell are read once, one iteration ahead, and stay in registers for S planes
//     (three slots, the loop unrolled by three so that nothing is moved).
// Faces: a neighbour outside the grid is the voxel itself (the reference's clamped index): an LDS
// position chosen once for z and for the strip's ends, a copy of the edge row for a face inside a
// strip, the centre for x.  Cells outside the window's valid part compute values that nothing
// reads.  Each stage rounds as the single-stage kernel does, so the result equals S single stages
// bit for bit.  u_out must alias neither psi nor u_in (other blocks read their halos).
//
// Every fused launch moves 32 B per point (complex64), 16 at S = 2 and 10.7 at S = 3 per stage:
// at 256^3 two stages take 112 us (4.9 TB/s, the rate of a large copy) and three 136 us, where the
// arithmetic and the LDS reads of the halo cells bound the launch (530 MB, 3.6 to 3.9 TB/s).  Keeping the centre and the
// previous plane of every level in registers spilled 30 of them (290 us at S = 3).  The pair
// kernel before this one held three planes of every level in LDS, took 111 us at 256^3 and, with
// too few blocks on smaller grids, 49 us at 128^3 (now 20), 46 at 64^3 (7.8), and in complex128
// 63 us at 64 x 96 x 128 (16 to 19) and 322 at 256^3 (185 to 225).
struct ChainArgs {
  int nx, ny, nz;
  int w;                    // window columns
  int ty, tz, tx;           // output tile (rows, columns) and x planes per block
  int nty, ntz, ntx;        // tiles per grid
  int batch;
};
template <typename R, int S> struct ChainCoef { R c[S], inv_2m, inv_dx2; };

// W: the window's columns where they are known at compile time (LDS row offsets become immediates)
template <typename R, int S, int NT, int RC, int W>
__global__ __launch_bounds__(NT) void horner_chain_kernel(const cx<R>* __restrict__ u_in, cx<R>* __restrict__ u_out,
                                                          const cx<R>* __restrict__ psi,
                                                          const float2* __restrict__ V, const ChainArgs g,
                                                          const ChainCoef<R, S> k) {
  using C = cx<R>;
  static_assert(S == 2 || S == 3, "psi and V are kept in three slots");
  constexpr int CELLS = NT * RC;
  constexpr unsigned EB = unsigned(sizeof(C));
  __shared__ C lev[2][S][CELLS];            // [buffer][level][row][column]
  const int tid = threadIdx.x;
  // Blocks are dispatched round-robin over the 8 XCDs.  Each XCD gets a contiguous run of tiles
  // (z fastest, then y, then x slab), so the tiles of one XCD march the same x planes together and
  // the halo cells one tile fetches are L2 hits for its neighbours.
  const long total = long(g.ntz) * g.nty * g.ntx * g.batch;
  const long q8 = total / 8, r8 = total % 8, xcd = blockIdx.x % 8;
  long tile = xcd * q8 + (xcd < r8 ? xcd : r8) + blockIdx.x / 8;
  const int bz = int(tile % g.ntz);
  tile /= g.ntz;
  const int by = int(tile % g.nty);
  tile /= g.nty;
  const int bx = int(tile % g.ntx);
  const long poff = (tile / g.ntx) * long(g.nx) * g.ny * g.nz;
  u_in += poff;
  u_out += poff;
  psi += poff;
  V += poff;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int w = W ? W : g.w;
  const int strips = NT / w;
  const int x0 = bx * g.tx, x1 = min(x0 + g.tx, nx);
  const int yb = by * g.ty - S;                       // first window row
  const int zb = g.ntz > 1 ? bz * g.tz - S : 0;       // first window column (whole rows: no halo)
  const long sx = long(ny) * nz;

  // the strip: rows j0 .. j0 + RC - 1 of column c
  const int strip = tid / w, c = tid % w;
  const int j0 = strip * RC;
  const int gy0 = yb + j0, gz = zb + c;
  const bool live = strip < strips && gz >= 0 && gz < nz && gy0 < ny && gy0 + RC > 0;
  // depth: the stages the strip takes part in, its largest distance from a window edge that is not
  // a grid face; outmask: its output cells; off: their voxels in an x plane (clamped)
  int depth = 0;
  unsigned outmask = 0;
  unsigned off[RC];
#pragma unroll
  for (int i = 0; i < RC; ++i) {
    const int j = j0 + i, gy = gy0 + i;
    off[i] = unsigned(min(max(gy, 0), ny - 1)) * unsigned(nz) + unsigned(min(max(gz, 0), nz - 1));
    int d = S;
    if (yb > 0) d = min(d, j);
    if (yb + strips * RC < ny) d = min(d, strips * RC - 1 - j);
    if (live && gy >= 0 && gy < ny) {
      depth = max(depth, d);
      if (gy >= by * g.ty && gy < (by + 1) * g.ty && gz >= bz * g.tz && gz < (bz + 1) * g.tz) outmask |= 1u << i;
    }
  }
  // LDS elements of a level plane: the strip's first cell, its z neighbours, the rows above and
  // below the strip; a neighbour outside the grid (or the window) is the cell itself
  const int own = strip < strips ? j0 * w + c : 0;
  const int ezm = (c > 0 && gz > 0) ? own - 1 : own;
  const int ezp = (c < w - 1 && gz < nz - 1) ? own + 1 : own;
  const int etop = (j0 > 0 && gy0 > 0) ? own - w : own;
  const int ebot = (strip < strips - 1 && gy0 + RC < ny) ? own + RC * w : own + (RC - 1) * w;
  // a y face inside the strip: row lo - 1 repeats the grid's first row, row hi + 1 its last
  const int lo = live && gy0 < 0 ? -gy0 : 0;
  const int hi = live && gy0 + RC > ny ? ny - 1 - gy0 : RC - 1;
  const bool face = lo > 0 || hi < RC - 1;

  C un[RC];                                           // u(t)
  C ps[3][RC];                                        // psi, V of plane q in slot (q - t0) mod 3
  float2 vs[3][RC];
  const int t0 = max(x0 - S, 0), t1 = x1 - 1 + S;
#pragma unroll
  for (int i = 0; i < RC; ++i) {
    un[i] = mk<R>(R(0), R(0));
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      ps[f][i] = mk<R>(R(0), R(0));
      vs[f][i] = make_float2(0.0f, 0.0f);
    }
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < RC; ++i) un[i] = byte_at(u_in + long(t0) * sx, off[i] * EB);
  }

  // iteration t, f = (t - t0) mod 3
  auto iteration = [&](int t, auto fc) {
    constexpr int f = decltype(fc)::value;
    const int b = t & 1;
    // loads of the next iteration: u(t + 1); psi and V of plane t, whose first stage is next
    C ua[RC], pa[RC];
    float2 va[RC];
    if (live) {
      const C* __restrict__ ub = u_in + long(min(t + 1, nx - 1)) * sx;
      const C* __restrict__ pb = psi + long(min(t, nx - 1)) * sx;
      const float2* __restrict__ vb = V + long(min(t, nx - 1)) * sx;
#pragma unroll
      for (int i = 0; i < RC; ++i) ua[i] = byte_at(ub, off[i] * EB);
#pragma unroll
      for (int i = 0; i < RC; ++i) {
        pa[i] = byte_at(pb, off[i] * EB);
        va[i] = byte_at(vb, off[i] * unsigned(sizeof(float2)));
      }
    }
    C* wr = &lev[b ^ 1][0][0];
    const C* rd = &lev[b][0][0];
    C nxt[RC], prv[RC];                               // level s - 1: planes t - s + 1 and t - s - 1
    if (strip < strips) {
#pragma unroll
      for (int i = 0; i < RC; ++i) {
        nxt[i] = un[i];
        prv[i] = wr[own + i * w];
        wr[own + i * w] = un[i];
      }
    }
    static_for<S>([&](auto lc) {
      constexpr int l = decltype(lc)::value, s = l + 1;
      const int q = t - s;                            // this stage's plane; the first one needed: x0 - (S - s)
      if (q >= x0 - (S - s) && q >= 0 && q < nx && depth >= s) {
        const C* cl = rd + l * CELLS;
        C cur[RC];
#pragma unroll
        for (int i = 0; i < RC; ++i) cur[i] = cl[own + i * w];
        if (q == 0) {
#pragma unroll
          for (int i = 0; i < RC; ++i) prv[i] = cur[i];
        }
        if (q == nx - 1) {
#pragma unroll
          for (int i = 0; i < RC; ++i) nxt[i] = cur[i];
        }
        C o[RC];
#pragma unroll
        for (int i = 0; i < RC; ++i) {
          const C ym = i > 0 ? cur[i > 0 ? i - 1 : 0] : cl[etop];
          const C yp = i < RC - 1 ? cur[i < RC - 1 ? i + 1 : 0] : cl[ebot];
          o[i] = horner_point<R>(cur[i], prv[i], nxt[i], ym, yp, cl[ezm + i * w], cl[ezp + i * w],
                                 ps[(f + 3 - s) % 3][i], vs[(f + 3 - s) % 3][i], k.c[l], k.inv_2m, k.inv_dx2);
        }
        if constexpr (s < S) {
          if (face) {
#pragma unroll
            for (int i = RC - 1; i > 0; --i)
              if (i == lo) o[i - 1] = o[i];
#pragma unroll
            for (int i = 0; i < RC - 1; ++i)
              if (i == hi) o[i + 1] = o[i];
          }
          C* wl = wr + s * CELLS;
#pragma unroll
          for (int i = 0; i < RC; ++i) {
            nxt[i] = o[i];
            prv[i] = wl[own + i * w];
            wl[own + i * w] = o[i];
          }
        } else {
          C* __restrict__ ob = u_out + long(q) * sx;
#pragma unroll
          for (int i = 0; i < RC; ++i)
            if (outmask & (1u << i)) byte_at(ob, off[i] * EB) = o[i];
        }
      } else if constexpr (s < S) {
        // no plane for this stage (before its first, past the grid): the next one still needs the
        // plane before its own
#pragma unroll
        for (int i = 0; i < RC; ++i) prv[i] = wr[s * CELLS + own + i * w];
      }
    });
#pragma unroll
    for (int i = 0; i < RC; ++i) {
      un[i] = ua[i];
      ps[f][i] = pa[i];
      vs[f][i] = va[i];
    }
    __syncthreads();
  };
  for (int t = t0; t <= t1; t += 3) {
    iteration(t, std::integral_constant<int, 0>{});
    if (t + 1 > t1) break;
    iteration(t + 1, std::integral_constant<int, 1>{});
    if (t + 2 > t1) break;
    iteration(t + 2, std::integral_constant<int, 2>{});
  }
}

// g: grid and batch, tz = output columns of a tile (at least nz: whole rows)
template <typename R, int S, int NT, int RC, int W>
static int launch_chain_form(ChainArgs g, const void* u_in, void* u_out, const void* psi, const float2* V,
                             const double* c, double inv_2m, double inv_dx2, hipStream_t s) {
  constexpr long lds = long(2) * S * NT * RC * long(sizeof(cx<R>));
  static_assert(lds <= 160 * 1024, "levels do not fit in LDS");
  if (g.tz > g.nz) g.tz = g.nz;
  g.ntz = (g.nz + g.tz - 1) / g.tz;
  g.w = g.ntz > 1 ? g.tz + 2 * S : g.nz;
  const int uy = (NT / g.w) * RC;
  if ((W && g.w != W) || uy <= 2 * S) {
    set_last_error("power series: %d stages on %d columns do not fit the window", S, g.w);
    return WFS_ERR_INVALID;
  }
  g.ty = uy - 2 * S < g.ny ? uy - 2 * S : g.ny;
  g.nty = (g.ny + g.ty - 1) / g.ty;
  g.ty = (g.ny + g.nty - 1) / g.nty;                  // even tiles
  // x planes per block: a block takes tx + 2 S iterations; of the slab counts up to four rounds of
  // blocks, the one with the fewest iterations over all rounds
  constexpr long fit = 160 * 1024 / lds;
  constexpr long slots = 256 * (fit < 1024 / NT ? fit : 1024 / NT);
  const long tiles = long(g.ntz) * g.nty * g.batch;
  const int most = int(g.nx < 4 * slots / tiles + 1 ? g.nx : 4 * slots / tiles + 1);
  long best = -1;
  for (int m = 1; m <= most; ++m) {
    const int tx = (g.nx + m - 1) / m;
    const int ntx = (g.nx + tx - 1) / tx;
    const long cost = (tiles * ntx + slots - 1) / slots * (tx + 2 * S);
    if (best < 0 || cost < best) {
      best = cost;
      g.tx = tx;
      g.ntx = ntx;
    }
  }
  const long blocks = tiles * g.ntx;
  if (blocks > 0x7fffffffL) { set_last_error("power series: grid too large"); return WFS_ERR_INVALID; }
  ChainCoef<R, S> k;
  for (int i = 0; i < S; ++i) k.c[i] = R(c[i]);
  k.inv_2m = R(inv_2m);
  k.inv_dx2 = R(inv_dx2);
  WFS_LAUNCH((horner_chain_kernel<R, S, NT, RC, W>), dim3(unsigned(blocks)), dim3(NT), 0, s,
             static_cast<const cx<R>*>(u_in), static_cast<cx<R>*>(u_out), static_cast<const cx<R>*>(psi), V, g, k);
  return int(hipGetLastError());
}

int horner_chain_stages(int precision) { return precision == WFS_C128 ? 2 : 3; }

// The window by grid, measured per launch in us, the forms of a pair of figures side by side on one box (on another
// box, by the launches' own times: S = 3 256^3 140, 192^3 55, 128^3 26, 64^3 13, 32^3 9.7; S = 2 256^3 108, 192^3 41,
// 128^3 19, 64^3 9.4, 64 x 64 x 512 19; complex128 256^3 225, 64 x 96 x 128 16, 32^3 6.4):
// complex64, S = 3: columns past 64 in tiles of 64 (a wide tile has few rows, most of them halo):
//   256^3 136 (whole rows 157, tiles of 128 143), 192^3 54 (59), 128^3 28 (26); nz <= 64 whole
//   rows, 512 threads (64^3 11.5 against 15 with 1024) or 256 on small grids (32^3 9.0 against 10.2)
// complex64, S = 2: whole rows at nz = 256 (256^3 112; tiles of 64 123), else tiles of 64, 512
//   threads (192^3 43, whole rows 45; 128^3 20, 21; 64 x 64 x 512 20, 27); 96 columns whole (13);
//   nz <= 64 whole rows, 256 threads (64^3 7.8, with 1024 10.7; 512 x 512 x 64 116, 120)
// complex128 (S = 2): whole rows, 1024 threads (256^3 185, 256 threads 231; 64 x 96 x 128 14.6,
//   17.5), 256 threads on small grids (32^3 5.5, 8.2); 512 columns in tiles of 128
int launch_horner_chain(int precision, int stages, int batch, int nx, int ny, int nz, const void* u_in, void* u_out,
                        const void* psi, const float2* V, const double* c, double inv_2m, double inv_dx2,
                        hipStream_t s) {
  ChainArgs g{};
  g.nx = nx;
  g.ny = ny;
  g.nz = nz;
  g.batch = batch;
  g.tz = nz;
  const bool small = long(batch) * nx * ny * nz <= 1L << 16;
#define WFS_CHAIN(R, S, NT, RC, W) \
  return launch_chain_form<R, S, NT, RC, W>(g, u_in, u_out, psi, V, c, inv_2m, inv_dx2, s)
  if (precision == WFS_C128) {
    if (stages == 2) {
      if (small && nz <= 64) WFS_CHAIN(double, 2, 256, 2, 0);
      if (nz > 256) g.tz = 128;
      WFS_CHAIN(double, 2, 1024, 2, 0);
    }
  } else if (stages == 3) {
    if (nz <= 64) {
      if (small) WFS_CHAIN(float, 3, 256, 3, 0);
      WFS_CHAIN(float, 3, 512, 3, 0);
    }
    if (nz % 64 == 0) {
      g.tz = 64;
      WFS_CHAIN(float, 3, 1024, 3, 70);
    }
    WFS_CHAIN(float, 3, 1024, 3, 0);
  } else if (stages == 2) {
    if (nz <= 64) WFS_CHAIN(float, 2, 256, 3, 0);
    if (nz == 256) WFS_CHAIN(float, 2, 1024, 3, 256);
    if (nz % 64 == 0) {
      g.tz = 64;
      WFS_CHAIN(float, 2, 512, 3, 68);
    }
    WFS_CHAIN(float, 2, 512, 3, 0);
  }
#undef WFS_CHAIN
  set_last_error("power series: no fused launch of %d stages", stages);
  return WFS_ERR_INVALID;
}

int launch_horner_stage(int precision, int batch, int nx, int ny, int nz, const void* u_in, void* u_out,
                        const void* psi, const float2* V, double dt_over_n, double inv_2m, double inv_dx2,
                        int tile_x, hipStream_t s) {
  // 64 z x 4 y threads per block, each marching 16 x planes: 16x more blocks
  // than whole-column marching (which left one block per CU, latency bound).
  constexpr int TZ = 64, TY = 4;
  if (tile_x <= 0) tile_x = nx < 16 ? nx : 16;
  const int ntiles = (nx + tile_x - 1) / tile_x;
  dim3 grid((nz + TZ - 1) / TZ, (ny + TY - 1) / TY, unsigned(ntiles * batch));
  dim3 block(TZ, TY, 1);
  if (precision == WFS_C128) {
    WFS_LAUNCH((horner_stage_kernel<double, TZ, TY>), grid, block, 0, s,
                       static_cast<const double2*>(u_in), static_cast<double2*>(u_out),
                       static_cast<const double2*>(psi), V, nx, ny, nz, dt_over_n, inv_2m, inv_dx2, tile_x, ntiles);
  } else {
    WFS_LAUNCH((horner_stage_kernel<float, TZ, TY>), grid, block, 0, s,
                       static_cast<const float2*>(u_in), static_cast<float2*>(u_out),
                       static_cast<const float2*>(psi), V, nx, ny, nz, float(dt_over_n), float(inv_2m),
                       float(inv_dx2), tile_x, ntiles);
  }
  return int(hipGetLastError());
}

}  // namespace wfs
