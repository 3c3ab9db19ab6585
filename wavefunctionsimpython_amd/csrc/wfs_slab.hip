// Two-launch split step for complex64 grids with ny = nz in {96, 128, 192, 256, 512} and complex128 grids
// with ny = nz in {64, 96, 128, 192} (gfx950), nx <= 512 in complex64 and <= 256 in complex128; planes of unequal
// sides (wfs_rect.hip) share the x launch.  Compiled twice: WFS_SLAB_PREC=0 (complex64) and 1 (complex128).
//
// A 256^2 y-z plane (512 KiB) or a 192^2 one (288 KiB) does not fit in one CU, so the y
// transform is split in two stages, ny = LY * B (B = 4, LY = 64 or 48; at 128 and 96, B = 2 and
// LY = 64 and 48; at 512, B = 8 and LY = 64), y = B a + b, ky = ka + LY kb:
//   X[ka + LY kb] = sum_b W_B^{b kb} W_NY^{b ka} sum_a x[B a + b] W_LY^{a ka}
// and each stage rides on a pass that is needed anyway:
//
//   yz_lines_kernel<NZ, LY, B>  (one block per x plane and residue b: the LY rows
//     y = B a + b with all z, 128 KiB at 256, 72 KiB at 192, 66 KiB at 128; half of it where the
//     exchanges go in parts, 64 KiB at 256 and 136 KiB at 512):  length-LY
//     inverse y stage over a, z inverse, potential phase, z forward, length-LY forward y stage
//   x_rows_kernel or x_slab_kernel  (one block per packet, ka and 8 to 32 consecutive z: the B rows
//     y = B ka + b with all x):  twiddles W_NY^{b ka} and length-B forward y stage over b,
//     x forward, kinetic phase K(kx, ky, kz), x inverse, length-B inverse y stage and twiddles
//
// Between the passes the y axis holds the half-transformed Y[b][ka] at row B ka + b.  The
// y-z launch reads the potential phase table in lines order (LinesOrder), one contiguous run
// per wavefront load.  A step moves 16 B per point in each pass (+8 for a potential table)
// against 64 (+8) for the four axis passes.  The arithmetic differs from the axis passes only
// in how the y transform is factored, so the results agree with theirs to float rounding, not
// bit for bit.
#include "wfs_yz_lines.h"

namespace wfs {

namespace {

// z points per x block of the complex128 launch: half lines where whole ones leave too few blocks
// (128^3: 16.5 us with 8, 18.3 with 4)
template <int N> constexpr int kZB128 = N <= 64 ? 4 : 8;

// rows y = B a + b of a row group: the length-B stage rides on the x launch (complex64: B = 4 at
// 256 and 192, LY = 64 and 48 rows per group; B = 2 at 128 and 96, LY = 64 and 48; B = 8 at 512, LY = 64; complex128: B = 2 up to 128,
// where the x launch then holds one row a lane: 33, 74 and 129 KiB of LDS per group at 64, 96 and
// 128, B = 4 at 192, 148 KiB).  Measured at 64^3 and 128^3 complex128, y-z and x launch: B = 2 8.0 +
// 5.7 and 25.9 + 16.5 us, B = 4 7.3 + 7.5 and 24.2 + 21.9.
template <typename R, int N> struct SlabShape {
  static constexpr int B = N <= 128 ? 2 : N <= 256 ? 4 : 8;
  static constexpr int LY = N / B;
};

// Lane pairs: the partner lanes tid and tid ^ ZB share the (x, z) points of a block; lane
// q = (tid / ZB) % 2 holds rows b = q and q + 2 (and, after the forward y stage, ky
// columns kb = q and q + 2).  The length-4 y stage is a 2-point stage in each lane, one
// complex value swapped with the partner, and a second 2-point stage:
//   forward, Z[b] = W_NY^{b ka} Y[b]:  E_q[k'] = Z[q] + (-1)^k' Z[q + 2],
//            X[k' + 2 k''] = E_0[k'] + (-1)^k'' W_4^{k'} E_1[k']
//   inverse: F_q[beta] = X[q] + (-1)^beta X[q + 2],
//            out[b] = F_0[b mod 2] + W_4^{-b} F_1[b mod 2],  Y'[b] = W_NY^{-b ka} out[b]
// Lane q keeps the k' = q (beta = q) values and receives the partner's.  For B = 2 (128^2
// planes) each lane holds the one row b = q and the length-2 stage is one swap:
//   X[kb] = Z[0] + (-1)^kb Z[1],  out[b] = X[0] + (-1)^b X[1].
// Lane-dependent choices are signs, not selects: with s = (-1)^q, lane q of a B = 4 pair
// holds s times its second column through the x transforms (all linear) and uses s W_NY^{b ka}
// as that row's twiddle.  Negation commutes exactly with every rounded operation, so the
// results are bit for bit those of the selecting form, with one select per value left.
// the partner's value, partner = tid ^ ZB, by DPP moves and row swaps (xor_lane)
template <int ZB, typename R>
__device__ __forceinline__ cx<R> partner_c(cx<R> v) {
  if constexpr (sizeof(R) == 4) {
    return mk<R>(__int_as_float(xor_lane_b32<ZB>(__float_as_int(v.x))), __int_as_float(xor_lane_b32<ZB>(__float_as_int(v.y))));
  } else {
    return mk<R>(xor_lane<ZB>(v.x), xor_lane<ZB>(v.y));
  }
}

// complex64 grids of few blocks and complex128.  ZB = 8 runs four waves per SIMD where a lane holds at most 16 points of an x line (at most 128
// VGPRs: the x transforms' table twiddles are read from LDS one at a time where they are applied,
// so no twiddle array is held; at nx = 256 one spilled register, 52.4 against 55.8 us per launch
// with three waves, bit-identical); the 24 points of nx = 96 or 192 do not fit in 128.
// 64-byte segments (ZB = 8, complex128 ZB = 4): a block reads and writes halves of 128-byte lines; the two blocks of a line
// get the block indices 16 g + x and 16 g + 8 + x, which the dispatcher sends to the same XCD
// (blocks go round-robin over the 8 XCDs) one after the other, so the second half comes from
// that XCD's L2.
template <typename R, int NX, int NY, int NZ, int B, int ZB>
__global__ __launch_bounds__(2 * ZB * split_of<NX>::n2)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 && ZB == 8 && NX / split_of<NX>::n2 <= 16 ? 4 : 1))) void x_slab_kernel(
    cx<R>* __restrict__ data, const XSlabParams p) {
  constexpr int N2 = split_of<NX>::n2;
  constexpr int N1 = NX / N2;
  constexpr int A = NY / B;
  constexpr int TZ = NZ / ZB;
  static_assert(B == 4 || B == 2, "the lane-pair y stage is written for B = 4 and B = 2");
  constexpr int RPL = B / 2;               // rows (columns after the y stage) per lane
  static_assert(N1 * N2 == NX && N1 % N2 == 0 && NZ % ZB == 0 && NY % B == 0 && 2 * ZB <= 64, "bad slab split");
  using C = cx<R>;
  using CC = const __attribute__((address_space(4))) C;
  constexpr int LINES = 2 * ZB;            // x lines per round: (q, z)
  __shared__ C lds[LINES * NX];

  const int tid = threadIdx.x;
  const int zl = tid % ZB;                 // z within the block's segment
  const int q = (tid / ZB) % 2;            // lane-pair half
  const int t = tid / (2 * ZB);            // thread of the x line: x = t + N2 i
  const int line = q * ZB + zl;
  long bid = blockIdx.x;
  if constexpr (ZB * sizeof(C) == 64) bid = 2 * (8 * (bid / 16) + bid % 8) + (bid / 8) % 2;
  const int zt = int(bid % TZ);
  const int ka = int((bid / TZ) % A);
  const long pk = bid / (long(TZ) * A);
  C* __restrict__ blk = data + pk * (long(NX) * NY * NZ) + long(B * ka) * NZ + long(zt) * ZB;
  constexpr unsigned XS = unsigned(NY) * NZ;   // x stride
  constexpr unsigned EB = unsigned(sizeof(C));  // byte offsets within a packet: NX NY NZ 8 <= 2^27
  static_assert(long(NX) * NY * NZ * sizeof(C) <= (1L << 32), "32-bit byte offsets");
  // element i of row q + 2 j
  auto off = [&](int i, int j) { return unsigned(zl) + unsigned(q + 2 * j) * NZ + unsigned(t + N2 * i) * XS; };

  // y-stage twiddles W_NY^{b ka} of this lane's rows b = q (+ 2)
  C wq[RPL];
  {
    CC* twy = (CC*)(p.tw_y);
    C wb[B];
#pragma unroll
    for (int b = 0; b < B; ++b) wb[b] = mk<R>(twy[(b * ka) % NY].x, twy[(b * ka) % NY].y);
    wq[0] = q ? wb[1] : wb[0];
    if constexpr (RPL == 2) wq[RPL - 1] = q ? mk<R>(-wb[B - 1].x, -wb[B - 1].y) : wb[B - 2];   // s W_NY^{b ka}
  }

  C a[RPL][N1];
#pragma unroll
  for (int j = 0; j < RPL; ++j)
#pragma unroll
    for (int i = 0; i < N1; ++i) a[j][i] = byte_at(blk, off(i, j) * EB);

  // the x transforms' table twiddles W_NX^{t k1} (t < N2, k1 < N1) and the kinetic factors
  // kx(x), staged in LDS once per block (their loads in flight with the points'); every
  // transform of both columns reads them from there
  __shared__ C tws[N2 * N1];
  __shared__ C kxs[NX];
  {
    const C* __restrict__ tw = reinterpret_cast<const C*>(p.tw_x);
    const C* __restrict__ kx = reinterpret_cast<const C*>(p.kx);
    for (int e = tid; e < N2 * N1; e += 2 * ZB * N2) tws[e] = tw[((e / N1) * (e % N1)) % NX];
    for (int e = tid; e < NX; e += 2 * ZB * N2) kxs[e] = kx[e];
  }

  const R sgn = q ? R(-1) : R(1);          // s = (-1)^q
  if constexpr (B == 2) {
    // forward y stage, B = 2: X[kb] = Z[0] + (-1)^kb Z[1], lane q keeps X[q] = recv + s z
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      const C z = cmul(a[0][i], wq[0]);
      const C recv = partner_c<ZB, R>(z);
      a[0][i] = mk<R>(fma_r(sgn, z.x, recv.x), fma_r(sgn, z.y, recv.y));
    }
  } else {
    // forward y stage, B = 4: a[0] <- X[q], a[1] <- s X[q + 2].  With z1 = s Z[q + 2] the
    // kept value z0 + z1 is E_q[q] and the sent one E_q[1 - q]; lane 0 then holds E_0[0]
    // and receives E_1[0], lane 1 holds E_1[1] and receives E_0[1]:
    //   X[q] = kk + recv,  X[q + 2] = s (kk - recv),  kk = keep or W_4 keep (lane 1)
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      const C z0 = cmul(a[0][i], wq[0]);
      const C z1 = cmul(a[RPL - 1][i], wq[RPL - 1]);
      const C keep = cadd(z0, z1);
      const C recv = partner_c<ZB, R>(csub(z0, z1));
      const C kk = q ? mk<R>(keep.y, -keep.x) : keep;     // W_4^q keep, W_4 = -i
      a[0][i] = cadd(kk, recv);
      a[RPL - 1][i] = csub(kk, recv);
    }
  }

  // x forward, kinetic phase, x inverse on the columns ky = ka + A kb, kb = q + 2 j, one
  // column at a time: the table twiddles and kinetic factors are read where they are used
  // (opaque indices), so that only the other column's points stay live besides the transform
  auto lidx = [&](int k1, int n2) { return (k1 * N2 + n2) * LINES + line; };
  const C* __restrict__ ky = reinterpret_cast<const C*>(p.ky);
  const C* __restrict__ kz = reinterpret_cast<const C*>(p.kz);
  __syncthreads();                         // tws, kxs staged
  // one column transform: the in-register DFT, then each table twiddle read from LDS where it
  // is applied (no twiddle array held across the DFT), then the LDS exchange
  auto column = [&](C (&col)[N1], auto sign_c) {
    constexpr int SG = decltype(sign_c)::value;
    DFT<N1, SG>::run(col);
    const C* tr = tws + opaque_v(t) * N1;
#pragma unroll
    for (int k1 = 1; k1 < N1; ++k1) {
      const C w = tr[k1];
      col[k1] = SG < 0 ? cmul(col[k1], w) : cmulc(col[k1], w);
    }
    column_dft_second<NX, N2, SG>(col, lds, t, lidx);
  };
#pragma unroll
  for (int j = 0; j < RPL; ++j) {
    if (j) __syncthreads();
    column(a[j], std::integral_constant<int, -1>{});
    {
      const C* kr = kxs + opaque_v(t);
      const C kyz = cmul(ky[ka + A * (q + 2 * j)], kz[zt * ZB + zl]);
#pragma unroll
      for (int i = 0; i < N1; ++i) a[j][i] = cmul(a[j][i], cmul(kr[N2 * i], kyz));
    }
    __syncthreads();
    column(a[j], std::integral_constant<int, +1>{});
  }

  if constexpr (B == 2) {
    // inverse y stage, B = 2: out[b] = X[0] + (-1)^b X[1], Y'[q] = W_NY^{-q ka} out[q]
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      const C v = a[0][i];
      const C recv = partner_c<ZB, R>(v);
      a[0][i] = cmulc(mk<R>(fma_r(sgn, v.x, recv.x), fma_r(sgn, v.y, recv.y)), wq[0]);
    }
  } else {
    // inverse y stage, B = 4, from a[0] = X[q] and a[1] = s X[q + 2]: the kept a[0] + a[1] is
    // F_q[q] and the sent a[0] - a[1] is F_q[1 - q]; with kk = keep or W_4^{-1} keep (lane 1)
    //   out[q] = kk + recv,  out[q + 2] = s (kk - recv),  a[0] <- Y'[q], a[1] <- Y'[q + 2]
    // (s W_NY^{(q+2) ka} is the second row's twiddle, so the sign cancels)
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      const C keep = cadd(a[0][i], a[RPL - 1][i]);
      const C recv = partner_c<ZB, R>(csub(a[0][i], a[RPL - 1][i]));
      const C kk = q ? mk<R>(-keep.y, keep.x) : keep;     // W_4^{-q} keep, W_4^{-1} = +i
      a[0][i] = cmulc(cadd(kk, recv), wq[0]);
      a[RPL - 1][i] = cmulc(csub(kk, recv), wq[RPL - 1]);
    }
  }

  // store addresses recomputed from an opaque copy of the thread index, so the load
  // addresses do not stay live through the transforms
  {
    const int tt = opaque_v(tid);
    const unsigned base = unsigned(tt % ZB) + unsigned((tt / ZB) % 2) * NZ + unsigned(tt / (2 * ZB)) * XS;
#pragma unroll
    for (int j = 0; j < RPL; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) byte_at(blk, (base + unsigned(2 * j) * NZ + unsigned(N2 * i) * XS) * EB) = a[j][i];
  }
}

// The complex64 x launch (and complex128 at 192^2).  A block owns the B rows of one ka over 64 / B z points (64, 128 or 256 bytes of a
// row) and all x; lane q 64 / B + z of every wavefront holds row b = q at x = t + N2 i, t the wavefront's
// index, so that the x transforms' twiddles and the kinetic factors are the same in all lanes and come
// through the scalar cache.  For the y stage the B rows are brought into one lane (transpose_rows, B x
// points at a time), transformed there and sent back; the x transforms exchange one part at a time through
// 256 NX bytes of LDS.  At nx = 256 that leaves 44 registers and 64 KiB, two blocks of 1024 threads a CU, at
// nx = 512 (128 registers, 128 KiB) one.  Whole lines (B < 8) go down the rows, ka fastest (256^3 49.8 us against
// 51.6 with z fastest); the half lines of B = 8 go with all z tiles of a ka to one XCD (blocks go round-robin
// over the 8 of them), whose L2 then joins them.
//   us per launch, lane pairs (x_slab_kernel, the better of 8 and 16 z points) against this form: 2 x 256^3
//   134 -> 105 (536 MB: 5.1 TB/s), 192 x 256^2 53 -> 38, 192^3 37 -> 28, 3 of them 85 -> 69, 12 x 96^3 37 -> 28,
//   8 x 128^3 45 -> 42, 256^3 alike at 50 (5.4 TB/s); the bits are the same.
//   512^2 planes (B = 8): 512^3 597 us, 646 with the tiles of a ka in pairs over the XCDs (the axis pass alone
//   688), 256 x 512^2 317 -> 233, 64 x 512^2 46 -> 50; 400 us of arithmetic beside one block's waits.  Lanes along
//   x instead of the rows at the loads save a transposition and lose more to eight pages a load: 692 us.
// N: the sides of square planes at compile time, or 0 (256^3 49.3 us, with sides at run time 52).
template <typename R, int NX, int B, int N>
__global__ __launch_bounds__(64 * split_of<NX>::n2)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 && NX == 256 && B >= 4 ? 8 : 1))) void x_rows_kernel(cx<R>* __restrict__ data,
                                                                        const XSlabParams p) {
  constexpr int ZB = 64 / B;
  // B = 1: 64 consecutive points of the plane, taken as one row
  const unsigned NY = N ? unsigned(N) : B == 1 ? 1u : unsigned(p.ny);
  const unsigned NZ = N ? unsigned(N) : B == 1 ? unsigned(p.ny) * unsigned(p.nz) : unsigned(p.nz);
  const unsigned A = NY / B, TZ = NZ / ZB;
  constexpr int N2 = split_of<NX>::n2, N1 = NX / N2;
  static_assert(N1 % B == 0, "bad split of the x line");
  using C = cx<R>;
  using CC = const __attribute__((address_space(4))) C;
  __shared__ R lds[64 * NX];

  const int lane = threadIdx.x & 63;
  const int t = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned pk = blockIdx.x / (TZ * A), bid = blockIdx.x % (TZ * A);
  const bool by_xcd = B == 8 && A % 8 == 0;
  const int zt = int(by_xcd ? (bid / 8) % TZ : bid / A);
  const int ka = int(by_xcd ? (bid / (8 * TZ)) * 8 + bid % 8 : bid % A);
  const unsigned XS = NY * NZ;
  constexpr unsigned EB = unsigned(sizeof(C));           // byte offsets within a packet: nx ny nz 8 <= 2^32
  C* __restrict__ blk = data + long(pk) * NX * XS + long(B * ka) * NZ + long(zt) * ZB;

  auto off = [&](int l, int i) {
    return (unsigned(l % ZB) + unsigned(l / ZB) * NZ + (unsigned(t) + unsigned(N2) * unsigned(i)) * XS) * EB;
  };
  C a[N1];
#pragma unroll
  for (int i = 0; i < N1; ++i) a[i] = byte_at(blk, off(lane, i));

  CC* twy = (CC*)(p.tw_y);
  // forward y stage X[kb] = sum_b W_B^{b kb} W_N^{b ka} Y[b] on B x points at a time
#pragma unroll
  for (int g = 0; g < (B > 1 ? N1 : 0); g += B) {
    transpose_rows<B, R>(a + g);
    C r[B];
    r[0] = a[g];
#pragma unroll
    for (int b = 1; b < B; ++b) r[b] = cmul(a[g + b], mk<R>(twy[b * ka].x, twy[b * ka].y));
    DFT<B, -1>::run(r);
#pragma unroll
    for (int b = 0; b < B; ++b) a[g + b] = r[b];
    transpose_rows<B, R>(a + g);
  }
  CC* twx = (CC*)(p.tw_x);
  auto lidx = [&](int k1, int n2) { return (k1 * N2 + n2) * 64 + lane; };
  auto transform_x = [&](auto sign_c) {
    constexpr int SG = decltype(sign_c)::value;
    DFT<N1, SG>::run(a);
#pragma unroll
    for (int k1 = 1; k1 < N1; ++k1) {
      const C w = mk<R>(twx[(t * k1) % NX].x, twx[(t * k1) % NX].y);
      a[k1] = SG < 0 ? cmul(a[k1], w) : cmulc(a[k1], w);
    }
    column_dft_second_parts<NX, N2, SG>(a, lds, t, lidx);
  };

  transform_x(std::integral_constant<int, -1>{});
  {
    const int y = B == 1 ? (zt * ZB + lane) / p.nz : ka + int(A) * (lane / ZB);
    const int z = B == 1 ? (zt * ZB + lane) % p.nz : zt * ZB + lane % ZB;
    const C kyz = cmul(reinterpret_cast<const C*>(p.ky)[y], reinterpret_cast<const C*>(p.kz)[z]);
    CC* kx = (CC*)(p.kx) + t;
#pragma unroll
    for (int i = 0; i < N1; ++i) a[i] = cmul(a[i], cmul(mk<R>(kx[N2 * i].x, kx[N2 * i].y), kyz));
  }
  __syncthreads();
  transform_x(std::integral_constant<int, +1>{});

  // inverse y stage Y'[b] = W_N^{-b ka} sum_kb W_B^{-b kb} X[kb], stored B x points at a time
  const int l = opaque_v(lane);
#pragma unroll
  for (int g = 0; g < N1; g += B) {
    if constexpr (B > 1) {
      transpose_rows<B, R>(a + g);
      C r[B];
#pragma unroll
      for (int b = 0; b < B; ++b) r[b] = a[g + b];
      DFT<B, +1>::run(r);
      a[g] = r[0];
#pragma unroll
      for (int b = 1; b < B; ++b) a[g + b] = cmulc(r[b], mk<R>(twy[b * ka].x, twy[b * ka].y));
      transpose_rows<B, R>(a + g);
    }
#pragma unroll
    for (int i = g; i < g + B; ++i) byte_at(blk, off(l, i)) = a[i];
  }
}

#if WFS_SLAB_PREC == 0
// flags[p] = 1 when x plane p equals plane p - 1 of the same packet bit for bit, else 0
__global__ __launch_bounds__(256) void plane_equal_kernel(const unsigned long long* __restrict__ table,
                                                          long plane_elems, int nx, long first,
                                                          int* __restrict__ flags) {
  const long p = first + blockIdx.x;
  int differ = 0;
  if (p % nx == 0) {
    differ = 1;
  } else {
    const unsigned long long* a = table + p * plane_elems;
    const unsigned long long* b = a - plane_elems;
    // 16 independent pairs of loads per round, issued together (no bound test between them;
    // the early exit is tested once a round): a 256^2 plane takes 16 rounds, not 256 dependent
    // steps.  The last partial round goes one element at a time.
    constexpr int U = 16;
    const long full = plane_elems - 256L * (U - 1);   // rounds starting below this hold U elements
    long i0 = threadIdx.x;
    for (; i0 < full && !differ; i0 += 256L * U) {
      unsigned long long v[U], w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        v[u] = a[i0 + 256L * u];
        w[u] = b[i0 + 256L * u];
      }
      unsigned long long d = 0;
#pragma unroll
      for (int u = 0; u < U; ++u) d |= v[u] ^ w[u];
      differ = d != 0;
    }
    for (; i0 < plane_elems && !differ; i0 += 256) differ = a[i0] != b[i0];
  }
  differ = __syncthreads_or(differ);
  if (threadIdx.x == 0) flags[p] = differ ? 0 : 1;
}

// src[p] = the first plane of p's run of identical planes, one block per packet: plane x of the
// packet maps to the last x' <= x whose flag is 0 (plane 0 of a packet always starts a run).
// Each thread takes a chunk of planes, the chunks' last run starts are max-scanned across the
// block, and each thread fills its chunk from the start carried in -- instead of one thread
// walking the packet's planes one dependent load at a time.
__global__ __launch_bounds__(256) void plane_runs_kernel(const int* __restrict__ flags, int nx,
                                                         int* __restrict__ src) {
  __shared__ int last[256];
  const long base = long(blockIdx.x) * nx;
  const int t = threadIdx.x;
  const int chunk = (nx + 255) / 256;
  const int x0 = t * chunk < nx ? t * chunk : nx;
  const int x1 = x0 + chunk < nx ? x0 + chunk : nx;
  int l = -1;
  for (int x = x0; x < x1; ++x)
    if (!flags[base + x]) l = x;
  last[t] = l;
  __syncthreads();
  for (int d = 1; d < 256; d <<= 1) {   // inclusive max-scan over the chunks
    const int v = t >= d ? last[t - d] : -1;
    __syncthreads();
    if (v > last[t]) last[t] = v;
    __syncthreads();
  }
  int cur = t > 0 ? last[t - 1] : -1;
  for (int x = x0; x < x1; ++x) {
    if (!flags[base + x]) cur = x;
    src[base + x] = int(base) + cur;
  }
}

#endif

// compute units of the current device (cached per device)
int cu_count() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] > 0) return cache[dev];
  int n = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
  cache[dev] = n;
  return n;
}

template <typename R, int N, int MODE, int PARTS = 0, int PV = PV_ANY>
int launch_lines_m(void* data, const YzPlaneParams& p, hipStream_t s) {
  constexpr int LY = SlabShape<R, N>::LY, B = SlabShape<R, N>::B;
  static_assert(yz_lines_lds_bytes<R, N, LY, B, 1, PARTS>() <= 160 * 1024, "rows do not fit in LDS");
  const long groups = p.planes * B;
  WFS_LAUNCH((yz_lines_kernel<R, N, LY, B, 1, MODE, true, PARTS, PV>), dim3(unsigned(groups)),
                     dim3(yz_lines_threads<N, LY, 1>()), 0, s, reinterpret_cast<cx<R>*>(data), p);
  return int(hipGetLastError());
}

// Waves per SIMD asked of the compiler for the form that exchanges one part at a time (PARTS in
// wfs_yz_lines.h; the bits are those of the whole form), 0 where the whole form is the better one at any
// size.  256^2: a 1024-thread block in 64 VGPRs and 66 KB of LDS leaves room for a second one, so that one
// block's loads and stores run beside the other's transforms.  192^2: one 768-thread block either way, but
// the transforms no longer wait for the factor loads hoisted over them.  Not for complex128 (128^3 27.3 ->
// 28.6, 192^3 80.3 -> 85.6, 96^3 17.2 -> 18.3 us: its 3 and more exchanges cost what the second block
// gains) nor for complex64 128^2 planes (19.0 -> 19.3).  512^2: the only form that fits, 136 KiB of LDS and 128
// registers a block of 1024 threads; 512^3 701 us a full launch (3.3 GB: 4.7 TB/s), 465 an entry or exit.
template <typename R, int N> constexpr int lines_parts() { return sizeof(R) == 8 ? 0 : N == 512 ? 4 : N == 256 ? 8 : N == 192 ? 3 : 0; }

// The parts form is taken where the groups are more than the CUs.  us of the full / entry or exit launch,
// whole against parts: 256^2 256 planes 85 / 57 -> 76 / 49, 192 planes 64 / 44 -> 57 / 39, 128 planes
// 46 / 30 -> 36 / 26, 96 planes 40 / 27 -> 33 / 24; 192^2 256 planes 64 / 43 -> 59 / 39, 192 planes
// 50 / 34 -> 40 / 27, 128 planes 34 / 22 -> 26 / 18.  With one group per CU there is nothing to overlap
// and the extra barriers show: 256^2 64 planes 24.1 / 15.3 -> 26.2 / 16.4, 192^2 17.9 -> 19.0.
template <typename R, int N>
bool lines_in_parts(long planes) {
  return N == 512 || (lines_parts<R, N>() != 0 && planes * SlabShape<R, N>::B > cu_count());
}

// complex128 has the one-block-per-group forms only, and takes its box moments in their own launches
// (the sums of the plane pass and the axis passes, bit for bit)
template <typename R, int N>
int launch_lines_n(int mode, void* data, const YzPlaneParams& p, hipStream_t s) {
  if constexpr (lines_parts<R, N>() != 0) {
    constexpr int W = lines_parts<R, N>();
    if (lines_in_parts<R, N>(p.planes)) {
      if (mode == LINES_FULL)
        return p.spx ? launch_lines_m<R, N, LINES_FULL, W, PV_AXES>(data, p, s)
                     : launch_lines_m<R, N, LINES_FULL, W, PV_TABLE>(data, p, s);
      if (mode == LINES_ENTRY) return launch_lines_m<R, N, LINES_ENTRY, W>(data, p, s);
      if (mode == LINES_EXIT) return launch_lines_m<R, N, LINES_EXIT, W>(data, p, s);
    }
  }
  if constexpr (N < 512) {
    if (mode == LINES_FULL) return launch_lines_m<R, N, LINES_FULL>(data, p, s);
    if (mode == LINES_ENTRY) return launch_lines_m<R, N, LINES_ENTRY>(data, p, s);
    if (mode == LINES_EXIT) return launch_lines_m<R, N, LINES_EXIT>(data, p, s);
  }
  if constexpr (sizeof(R) == 4 && N >= 128 && N < 512) {
    if (mode == LINES_OBSERVE) return launch_lines_m<R, N, LINES_OBSERVE>(data, p, s);
    if (mode == LINES_ENTRY_OBSERVE) return launch_lines_m<R, N, LINES_ENTRY_OBSERVE>(data, p, s);
  }
  set_last_error("slab y-z pass: bad mode %d", mode);
  return WFS_ERR_INVALID;
}

template <typename R, int NX, int N, int ZB>
int launch_x_slab_z(void* data, const XSlabParams& p, hipStream_t s) {
  constexpr int B = SlabShape<R, N>::B;
  constexpr long per_packet = long(N / B) * (N / ZB);
  static_assert(per_packet % 16 == 0, "the XCD pairing needs a multiple of 16 blocks");
  WFS_LAUNCH((x_slab_kernel<R, NX, N, N, B, ZB>), dim3(unsigned(p.packets * per_packet)),
                     dim3(2 * ZB * split_of<NX>::n2), 0, s, reinterpret_cast<cx<R>*>(data), p);
  return int(hipGetLastError());
}

// z points per block: complex64 8 (256 threads at nx = 256), complex128 kZB128
template <typename R, int N>
int launch_x_slab_ny(int nx, void* data, const XSlabParams& p, hipStream_t s) {
#define WFS_X_SLAB_CASE(NX)                                                                                    \
  case NX:                                                                                                     \
    return launch_x_slab_z<R, NX, N, sizeof(R) == 8 ? kZB128<N> : 8>(data, p, s);
  switch (nx) {
    WFS_X_SLAB_CASE(8)
    WFS_X_SLAB_CASE(16)
    WFS_X_SLAB_CASE(32)
    WFS_X_SLAB_CASE(64)
    WFS_X_SLAB_CASE(96)
    WFS_X_SLAB_CASE(128)
    WFS_X_SLAB_CASE(192)
    WFS_X_SLAB_CASE(256)
    default:
      set_last_error("slab x pass: unsupported length %d", nx);
      return WFS_ERR_UNSUPPORTED;
  }
#undef WFS_X_SLAB_CASE
}

// x_rows_kernel's N^2 / 64 blocks a packet fill the card from 1.5 of them a CU on; below that the smaller blocks
// of x_slab_kernel are the faster ones or level.  us per launch, lane pairs against rows: 256 x 128^2 (256
// blocks a packet) 17.0 / 16.7, 2 packets 27.9 / 26.2; 128^3 11.4 / 11.8, 2 packets 14.6 / 14.1, 4 packets 25.5 /
// 21.1; 256 x 96^2 (144 blocks a packet) 14.6 / 16.3, 2 packets 18.1 / 20.9, 3 packets 24.2 / 22.2; 128 x 96^2
// 9.7 / 10.4, 14.0 / 15.3.  192^2 and 256^2 planes have 576 and 1024 blocks a packet.
bool x_rows_fill(int n, long packets) { return packets * (long(n) * n / 64) * 2 >= 3L * cu_count(); }

template <typename R, int B, int N = 0>
int launch_x_rows(int nx, void* data, const XSlabParams& p, hipStream_t s) {
  const unsigned blocks = unsigned(p.packets * (long(p.ny) * p.nz / 64));
#define WFS_X_ROWS_CASE(NX)                                                                                  \
  case NX:                                                                                                   \
    if constexpr ((NX / split_of<NX>::n2) % B == 0 && (NX <= 256 || (N == 0 && sizeof(R) == 4))) {                                                    \
      WFS_LAUNCH((x_rows_kernel<R, NX, B, N>), dim3(blocks), dim3(64 * split_of<NX>::n2), 0, s,                     \
                 reinterpret_cast<cx<R>*>(data), p);                                                         \
      return int(hipGetLastError());                                                                         \
    }                                                                                                        \
    break;
  switch (nx) {
    WFS_X_ROWS_CASE(8)
    WFS_X_ROWS_CASE(16)
    WFS_X_ROWS_CASE(32)
    WFS_X_ROWS_CASE(64)
    WFS_X_ROWS_CASE(96)
    WFS_X_ROWS_CASE(128)
    WFS_X_ROWS_CASE(192)
    WFS_X_ROWS_CASE(256)
    WFS_X_ROWS_CASE(512)
    default: break;
  }
#undef WFS_X_ROWS_CASE
  set_last_error("slab x pass: unsupported length %d", nx);
  return WFS_ERR_UNSUPPORTED;
}

template <typename R, int N>
SlabRows slab_rows_n() {
  SlabRows g;
  g.b = SlabShape<R, N>::B;
  g.n1y = g.n1z = N / split_of<N>::n2;
  g.uy = SlabShape<R, N>::LY / g.n1y;
  g.uz = split_of<N>::n2;
  return g;
}

}  // namespace

#if WFS_SLAB_PREC == 0
int launch_plane_dedup(const void* table, long plane_elems, int nx, int packets, long first, long count, int* flags,
                       int* src, hipStream_t s) {
  const long planes = long(nx) * packets;
  if (planes < 1 || planes > 0x7fffffffL || plane_elems < 1 || first < 0 || count < 1 || first + count > planes) {
    set_last_error("potential plane sharing: bad sizes");
    return WFS_ERR_INVALID;
  }
  WFS_LAUNCH(plane_equal_kernel, dim3(unsigned(count)), dim3(256), 0, s,
                     static_cast<const unsigned long long*>(table), plane_elems, nx, first, flags);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return int(e);
  WFS_LAUNCH(plane_runs_kernel, dim3(unsigned(packets)), dim3(256), 0, s, flags, nx, src);
  return int(hipGetLastError());
}

// complex64, ny = nz in {128, 192, 256}, nx a supported FFT length up to 256 (at 512 the x
// lines of a lane pair do not fit in registers)
bool slab_supported(int precision, const int n[3]) {
  return precision == WFS_C64 && n[1] == n[2] && (n[1] == 128 || n[1] == 192 || n[1] == 256) && n[0] <= 256 &&
         fft_length_supported(n[0]);
}

// complex128, ny = nz in {64, 96, 128, 192}: a row group of 256^2 planes (LY = 64 rows, 257 KiB)
// does not fit in a CU.  us per step with a potential table, passes or plane pass against the two
// launches: 64^3 18.1 -> 14.8, 96^3 54.8 -> 37.7, 128^3 57.5 -> 44.4, 192^3 198.7 -> 166.1, 64 x
// 192^2 76.4 -> 46.0, 48 x 64^3 192 -> 144; only long x lines beside 64^2 planes were slower
// (192 x 64^2 27.6 -> 29.9, 256 x 64^2 28.7 -> 34.6: x blocks of 128 and more points a lane pair),
// so the plan leaves those to the plane pass.
//
// complex64, ny = nz = 96 or 128: the plane pass holds a whole plane per block, a 96^2 plane in 74 KB with 12
// points of two lines a thread and one block a CU, against row groups of half a plane.  us per step with a
// potential table / with per-axis factors: 96^2 8 planes 24.4 / 21.6 -> 15.1 / 15.3, 64 planes 29.5 / 26.8 ->
// 20.0 / 20.2, 96^3 35.2 / 32.6 -> 26.8 / 27.0, 3 packets of it 57.9 / 56.8 -> 34.8 / 39.0, 12 packets 147 / 132
// -> 93 / 90; 128^2 256 planes 49.6 / 43.3 -> 40.6 / 39.4, 512 planes 78 / 71 -> 70 / 68, 1536 planes 240 / 182
// -> 191 / 172.  Not at 64^2: 14.0 / 12.7 -> 11.3 / 11.5 for one packet, but 12 packets of 96 x 64^2 47 / 42 ->
// 45 / 44, and the tuned 64^2 forms are bit for bit the axis passes.
//
// complex64 512^2 planes (B = 8, x_rows_kernel), us per step with a potential table against the four axis
// passes: 512^3 2407 -> 1367 (20 steps a call, entry and exit counted in; the two launches alone 1311), 256 x 512^2
// 1158 -> 798, 64 x 512^2 230 -> 182.  Its x launch takes 8 x points of a lane at a time, so nx = 8 and 16 (4 points
// a lane) stay with the passes.
//
// complex64 with 512 x planes (x_rows_kernel alone takes them): 512 x 96^2 75 / 69 -> 56 / 55, x 128^2 87 / 81 -> 81 /
// 78, x 192^2 256 / 243 -> 218 / 200, x 256^2 450 / 374 -> 339 / 310.
bool split_supported(int precision, const int n[3]) {
  if (n[1] != n[2]) return rect_supported(precision, n);
  if (!fft_length_supported(n[0])) return false;
  if (precision == WFS_C128) return (n[1] == 64 || n[1] == 96 || n[1] == 128 || n[1] == 192) && n[0] <= 256;
  if (n[1] == 512) return n[0] >= 32;
  return n[1] == 96 || n[1] == 128 || (n[0] == 512 && (n[1] == 192 || n[1] == 256));
}

SlabRows slab_rows_c128(int n);
int launch_yz_slab_c128(int n, int mode, void* data, const YzPlaneParams& p, hipStream_t s);
int launch_x_slab_c128(int nx, int n, void* data, const XSlabParams& p, hipStream_t s);

SlabRows slab_rows(int precision, const int nn[3]) {
  if (nn[1] != nn[2]) return rect_rows(nn[1], nn[2]);
  const int n = nn[1];
  if (precision == WFS_C128) return slab_rows_c128(n);
  if (n == 96) return slab_rows_n<float, 96>();
  if (n == 512) return slab_rows_n<float, 512>();
  return n == 128 ? slab_rows_n<float, 128>() : n == 192 ? slab_rows_n<float, 192>() : slab_rows_n<float, 256>();
}

LinesOrder slab_lines_order(int precision, const int n[3]) {
  const SlabRows g = slab_rows(precision, n);
  LinesOrder m;
  m.ny = n[1];
  m.nz = n[2];
  m.b = g.b;
  m.ly = m.rh = n[1] / g.b;
  m.n2z = g.uz;
  m.n1 = g.n1z;
  m.threads = g.uz * m.rh;
  return m;
}

int launch_yz_slab(int precision, const int nn[3], int mode, void* data, const YzPlaneParams& p, hipStream_t s) {
  if (nn[1] != nn[2]) return launch_yz_rect(nn[1], nn[2], mode, data, p, s);
  const int n = nn[1];
  if (p.planes <= 0 || p.planes * 8 > 0x7fffffffL) {
    set_last_error("slab y-z pass: bad plane count %ld", p.planes);
    return WFS_ERR_INVALID;
  }
  if (precision == WFS_C128) return launch_yz_slab_c128(n, mode, data, p, s);
  if (n == 256) return launch_lines_n<float, 256>(mode, data, p, s);
  if (n == 192) return launch_lines_n<float, 192>(mode, data, p, s);
  if (n == 128) return launch_lines_n<float, 128>(mode, data, p, s);
  if (n == 96) return launch_lines_n<float, 96>(mode, data, p, s);
  if (n == 512) return launch_lines_n<float, 512>(mode, data, p, s);
  set_last_error("slab y-z pass: unsupported plane %d", n);
  return WFS_ERR_UNSUPPORTED;
}

int launch_x_slab(int precision, const int nn[3], void* data, const XSlabParams& p, hipStream_t s) {
  const int nx = nn[0], n = nn[1];
  const long blocks = p.packets * (nn[1] == nn[2] ? long(n / 2) * (n / 4) : long(nn[1]) * nn[2] / 64);
  if (p.packets <= 0 || blocks > 0x7fffffffL || p.ny != nn[1] || p.nz != nn[2]) {
    set_last_error("slab x pass: bad packet count %ld", p.packets);
    return WFS_ERR_INVALID;
  }
  if (nn[1] != nn[2]) {
    const int b = rect_rows(nn[1], nn[2]).b;
    return b == 1   ? launch_x_rows<float, 1>(nx, data, p, s)
           : b == 2 ? launch_x_rows<float, 2>(nx, data, p, s)
           : b == 4 ? launch_x_rows<float, 4>(nx, data, p, s) : launch_x_rows<float, 8>(nx, data, p, s);
  }
  if (precision == WFS_C128) return launch_x_slab_c128(nx, n, data, p, s);
  if (n == 512) return launch_x_rows<float, 8>(nx, data, p, s);
  if (n == 256) return nx <= 256 ? launch_x_rows<float, 4, 256>(nx, data, p, s) : launch_x_rows<float, 4>(nx, data, p, s);
  if (n == 192) return nx <= 256 ? launch_x_rows<float, 4, 192>(nx, data, p, s) : launch_x_rows<float, 4>(nx, data, p, s);
  const bool rows = nx == 512 || x_rows_fill(n, p.packets);
  if (n == 128) return rows ? launch_x_rows<float, 2>(nx, data, p, s) : launch_x_slab_ny<float, 128>(nx, data, p, s);
  if (n == 96) return rows ? launch_x_rows<float, 2>(nx, data, p, s) : launch_x_slab_ny<float, 96>(nx, data, p, s);
  set_last_error("slab x pass: unsupported plane %d", n);
  return WFS_ERR_UNSUPPORTED;
}
#else
SlabRows slab_rows_c128(int n) {
  return n == 64 ? slab_rows_n<double, 64>() : n == 96 ? slab_rows_n<double, 96>()
         : n == 128 ? slab_rows_n<double, 128>() : slab_rows_n<double, 192>();
}

int launch_yz_slab_c128(int n, int mode, void* data, const YzPlaneParams& p, hipStream_t s) {
  if (n == 64) return launch_lines_n<double, 64>(mode, data, p, s);
  if (n == 96) return launch_lines_n<double, 96>(mode, data, p, s);
  if (n == 128) return launch_lines_n<double, 128>(mode, data, p, s);
  if (n == 192) return launch_lines_n<double, 192>(mode, data, p, s);
  set_last_error("slab y-z pass: unsupported complex128 plane %d", n);
  return WFS_ERR_UNSUPPORTED;
}

int launch_x_slab_c128(int nx, int n, void* data, const XSlabParams& p, hipStream_t s) {
  if (n == 64) return launch_x_slab_ny<double, 64>(nx, data, p, s);
  if (n == 96) return launch_x_slab_ny<double, 96>(nx, data, p, s);
  if (n == 128) return launch_x_slab_ny<double, 128>(nx, data, p, s);
  // 192^2 (B = 4: a lane pair holds two rows a lane): rows in one lane, but for 128 and 256 x planes (16 points
  // a lane), us per launch lane pairs / rows: nx = 192 79 / 67, 96 47 / 26, 64 16.8 / 15.9, 32 15.0 / 12.5, 8 6.5 / 4.9, 3
  // packets of 96 107 / 65; 128 32.4 / 34.2, 256 63 / 76.  B = 2 planes stay with lane pairs: 64^3 5.5 / 6.8, 128^3
  // 15.4 / 16.2, 96^3 15.1 / 17.1 (6 packets 44 / 37).
  if (n == 192)
    return nx % 128 ? launch_x_rows<double, 4, 192>(nx, data, p, s) : launch_x_slab_ny<double, 192>(nx, data, p, s);
  set_last_error("slab x pass: unsupported complex128 plane %d", n);
  return WFS_ERR_UNSUPPORTED;
}
#endif

}  // namespace wfs
