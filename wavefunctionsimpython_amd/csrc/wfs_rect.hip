// y-z launch of the two-launch split step on planes of unequal sides (complex64, ny != nz in {32, 64, 96, 128,
// 192, 256, 512}, gfx950): the scheme of wfs_slab.hip, rows y = B a + b of an x plane in one block with all
// z, LY = ny / B of them, in lengths that the square kernel cannot mix: its threads hold the same number of
// points of a y line and of a z line, which 128 = 16 x 8 and 48 = 24 x 2 do not share.  Here the two
// directions have their own split and their own number of active threads.
//
// Four axis passes of a 96 x 192 x 128 grid (19 MB) take 10 to 16 us each, bound by their latency and by the
// 64 to 96 bytes a point that they move.  us per step with a potential table, passes against two launches:
// 96 x 192 x 128 55 -> 34, 32 x 32 x 64 15.3 -> 9.9, 96 x 96 x 64 30 -> 20, 256 x 128 x 96 55 -> 38, 256 x 192 x 256
// 153 -> 111, 96 x 512 x 96 83 -> 46, 96 x 256 x 512 164 -> 125, 8 packets of 64 x 64 x 128 54 -> 36.  The y-z
// launch then runs at 2 to 4 TB/s: small groups' latency and their six exchanges.
#include "wfs_yz_lines.h"

namespace wfs {

namespace {

// Points per thread of a y line of LY points beside z lines of NZ: the split N1 x N2 (N1 a multiple of N2, at
// most 32 points) whose thread count is nearest to that of the z lines.
template <int NZ, int LY>
constexpr int rect_n1y() {
  const int tz = LY * split_of<NZ>::n2;
  int best = 0, far = 1 << 30;
  for (int n1 = 4; n1 <= 32; ++n1) {
    if (LY % n1 || n1 % (LY / n1)) continue;
    const int ty = NZ * (LY / n1), d = ty > tz ? ty - tz : tz - ty;
    if (ty <= 1024 && d < far) { best = n1; far = d; }
  }
  return best;
}

template <int NZ, int LY>
struct RectShape {
  static constexpr int N2Z = split_of<NZ>::n2, N1Z = NZ / N2Z;
  static constexpr int N1Y = rect_n1y<NZ, LY>(), N2Y = LY / N1Y;
  static constexpr int TY = NZ * N2Y, TZ = LY * N2Z, T = TY > TZ ? TY : TZ;
  static constexpr int TS = NZ + 1;      // odd row stride of the transposition
  static_assert(N1Y > 0 && T <= 1024 && long(LY) * TS * 8 <= 160 * 1024, "bad row group");
};

// MODE as in wfs_yz_lines.h (LINES_FULL, LINES_ENTRY, LINES_EXIT); B rows stride, runtime
template <int NZ, int LY, int MODE>
__global__ __launch_bounds__((RectShape<NZ, LY>::T)) void yz_rect_kernel(cx<float>* __restrict__ data,
                                                                        const YzPlaneParams p, int B) {
  using S = RectShape<NZ, LY>;
  using C = cx<float>;
  using CC = const __attribute__((address_space(4))) C;
  constexpr int NA = S::N1Y > S::N1Z ? S::N1Y : S::N1Z;
  __shared__ C lds[LY * S::TS];

  const int tid = threadIdx.x;
  const long group = blockIdx.x;
  const long plane = group / B;
  const int bres = int(group % B);
  C* __restrict__ blk = data + plane * (long(LY) * B * NZ) + long(bres) * NZ;
  const unsigned RS = unsigned(B) * NZ;      // element stride between the block's rows
  const bool in_y = S::TY == S::T || tid < S::TY, in_z = S::TZ == S::T || tid < S::TZ;
  C a[NA];

  // one transform of the lines a thread group holds: thread (c, u) has points u + N2 i of line c; STRIDE
  // lines.  Ends with LDS reads where N2 > 1.
  auto transform = [&](auto n1_c, auto n2_c, auto stride_c, bool active, const void* twp, auto sign_c) {
    constexpr int N1 = decltype(n1_c)::value, N2 = decltype(n2_c)::value, STRIDE = decltype(stride_c)::value;
    constexpr int SG = decltype(sign_c)::value, M = N1 / N2;
    const int t = opaque_v(tid), c = t % STRIDE;
    const int u = STRIDE % 64 == 0 ? __builtin_amdgcn_readfirstlane(t / STRIDE) : t / STRIDE;
    C(&v)[N1] = reinterpret_cast<C(&)[N1]>(a);
    if (active) {
      DFT<N1, SG>::run(v);
      if constexpr (N2 > 1) {
#pragma unroll
        for (int k1 = 1; k1 < N1; ++k1) {
          C w;
          if constexpr (STRIDE % 64 == 0) {
            CC* tw = (CC*)(twp) + u * N1;
            w = mk<float>(tw[k1].x, tw[k1].y);
          } else {
            w = reinterpret_cast<const C*>(twp)[u * N1 + k1];
          }
          v[k1] = SG < 0 ? cmul(v[k1], w) : cmulc(v[k1], w);
        }
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) lds[(k1 * N2 + u) * STRIDE + c] = v[k1];
      }
    }
    if constexpr (N2 > 1) {
      __syncthreads();
      if (active) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
          C b[N2];
#pragma unroll
          for (int n2 = 0; n2 < N2; ++n2) b[n2] = lds[((u + N2 * m) * N2 + n2) * STRIDE + c];
          DFT<N2, SG>::run(b);
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) v[m + M * k2] = b[k2];
        }
      }
    }
  };
  using std::integral_constant;
  auto transform_y = [&](auto sign_c) {
    transform(integral_constant<int, S::N1Y>{}, integral_constant<int, S::N2Y>{}, integral_constant<int, NZ>{}, in_y,
              decltype(sign_c)::value > 0 ? p.tw_yi : p.tw_yf, sign_c);
  };
  auto transform_z = [&](auto sign_c) {
    transform(integral_constant<int, S::N1Z>{}, integral_constant<int, S::N2Z>{}, integral_constant<int, LY>{}, in_z,
              p.tw_z, sign_c);
  };
  // y lines to z lines and back; LDS is free at entry, read at exit
  auto cols_to_rows = [&]() {
    const int t = opaque_v(tid);
    if (in_y) {
#pragma unroll
      for (int i = 0; i < S::N1Y; ++i) lds[(t / NZ + S::N2Y * i) * S::TS + t % NZ] = a[i];
    }
    __syncthreads();
    if (in_z) {
#pragma unroll
      for (int i = 0; i < S::N1Z; ++i) a[i] = lds[(t % LY) * S::TS + t / LY + S::N2Z * i];
    }
  };
  auto rows_to_cols = [&]() {
    const int t = opaque_v(tid);
    if (in_z) {
#pragma unroll
      for (int i = 0; i < S::N1Z; ++i) lds[(t % LY) * S::TS + t / LY + S::N2Z * i] = a[i];
    }
    __syncthreads();
    if (in_y) {
#pragma unroll
      for (int i = 0; i < S::N1Y; ++i) a[i] = lds[(t / NZ + S::N2Y * i) * S::TS + t % NZ];
    }
  };

  if (in_y) {
#pragma unroll
    for (int i = 0; i < S::N1Y; ++i) a[i] = blk[unsigned(tid % NZ) + unsigned(tid / NZ + S::N2Y * i) * RS];
  }
  const integral_constant<int, +1> inverse{};
  const integral_constant<int, -1> forward{};
  if constexpr (MODE != LINES_ENTRY) {
    transform_y(inverse);
    __syncthreads();
  }
  cols_to_rows();
  __syncthreads();
  if constexpr (MODE != LINES_ENTRY) transform_z(inverse);
  if constexpr (MODE == LINES_FULL) {
    if (in_z) {
      const int t = opaque_v(tid), c = t % LY, v = t / LY;
      if (p.spx) {
        const long pk = plane / p.nx;
        const C* __restrict__ pz = reinterpret_cast<const C*>(p.spz) + pk * NZ;
        const C pxy = cmul(reinterpret_cast<const C*>(p.spx)[plane],
                           reinterpret_cast<const C*>(p.spy)[pk * (long(LY) * B) + bres + B * c]);
#pragma unroll
        for (int i = 0; i < S::N1Z; ++i) a[i] = cmul(a[i], cmul(pz[v + S::N2Z * i], pxy));
      } else {
        const long tg = p.pv_planes ? long(p.pv_planes[plane]) * B + bres : group;
        const C* __restrict__ pv = reinterpret_cast<const C*>(p.pv) + tg * (long(LY) * NZ);
#pragma unroll
        for (int i = 0; i < S::N1Z; ++i) a[i] = cmul(a[i], pv[unsigned(i * S::TZ) + unsigned(t)]);
      }
    }
    __syncthreads();
  }
  if constexpr (MODE != LINES_EXIT) transform_z(forward);
  __syncthreads();
  rows_to_cols();
  if constexpr (MODE != LINES_EXIT) {
    __syncthreads();
    transform_y(forward);
  }
  if (in_y) {
    const int t = opaque_v(tid);
#pragma unroll
    for (int i = 0; i < S::N1Y; ++i) blk[unsigned(t % NZ) + unsigned(t / NZ + S::N2Y * i) * RS] = a[i];
  }
}

template <int NZ, int LY>
int launch_rect(int mode, int b, void* data, const YzPlaneParams& p, hipStream_t s) {
  const dim3 grid(unsigned(p.planes * b)), block(RectShape<NZ, LY>::T);
  cx<float>* d = static_cast<cx<float>*>(data);
  if (mode == LINES_FULL) WFS_LAUNCH((yz_rect_kernel<NZ, LY, LINES_FULL>), grid, block, 0, s, d, p, b);
  else if (mode == LINES_ENTRY) WFS_LAUNCH((yz_rect_kernel<NZ, LY, LINES_ENTRY>), grid, block, 0, s, d, p, b);
  else if (mode == LINES_EXIT) WFS_LAUNCH((yz_rect_kernel<NZ, LY, LINES_EXIT>), grid, block, 0, s, d, p, b);
  else { set_last_error("two-launch y-z pass: bad mode %d", mode); return WFS_ERR_INVALID; }
  return int(hipGetLastError());
}

constexpr int kSides[] = {32, 64, 96, 128, 192, 256, 512};

constexpr bool rect_length(int n) {
  for (int m : kSides)
    if (n == m) return true;
  return false;
}

// Residue classes of the y axis: the whole plane while it has at most 4608 points (36 KiB), else the fewest
// that leave row groups of at most 8192 points (two or more blocks a CU), at most 8, and of at most 128 rows.
constexpr int rect_b(int ny, int nz) {
  if (ny <= 128 && ny * nz <= 4608) return 1;
  int b = 2;
  while (b < 8 && (ny * nz / b > 8192 || ny / b > 128)) b *= 2;
  return b;
}

// calls f with the row group's (NZ, LY) as types; false where there is no such row group
template <typename F>
constexpr bool rect_dispatch(int nz, int ly, F f) {
#define WFS_RECT(NZ, LY) \
  if (nz == NZ && ly == LY) { f(std::integral_constant<int, NZ>{}, std::integral_constant<int, LY>{}); return true; }
  WFS_RECT(32, 64) WFS_RECT(32, 96) WFS_RECT(32, 128)
  WFS_RECT(64, 32) WFS_RECT(64, 48) WFS_RECT(64, 64) WFS_RECT(64, 96) WFS_RECT(64, 128)
  WFS_RECT(96, 32) WFS_RECT(96, 48) WFS_RECT(96, 64)
  WFS_RECT(128, 32) WFS_RECT(128, 48) WFS_RECT(128, 64)
  WFS_RECT(192, 16) WFS_RECT(192, 24) WFS_RECT(192, 32) WFS_RECT(192, 64)
  WFS_RECT(256, 16) WFS_RECT(256, 24) WFS_RECT(256, 32) WFS_RECT(256, 64)
  WFS_RECT(512, 12) WFS_RECT(512, 16) WFS_RECT(512, 24) WFS_RECT(512, 32)
#undef WFS_RECT
  return false;
}

// every pair of sides that rect_supported takes has its row group above
constexpr bool rect_complete() {
  for (int ny : kSides)
    for (int nz : kSides)
      if (ny != nz && !rect_dispatch(nz, ny / rect_b(ny, nz), [](auto, auto) {})) return false;
  return true;
}
static_assert(rect_complete(), "a pair of sides without its row group");

}  // namespace

// Not beside 512 x planes under 3072 points: 32 x blocks of 1024 threads (512 x 32 x 64 30.6 -> 34.2 us a step).
bool rect_supported(int precision, const int n[3]) {
  return precision == WFS_C64 && n[1] != n[2] && rect_length(n[1]) && rect_length(n[2]) && fft_length_supported(n[0]) &&
         (rect_b(n[1], n[2]) < 8 || n[0] >= 32) && (n[0] < 512 || n[1] * n[2] >= 3072);
}

SlabRows rect_rows(int ny, int nz) {
  const int b = rect_b(ny, nz);
  SlabRows g;
  rect_dispatch(nz, ny / b, [&](auto z, auto y) {
    using S = RectShape<decltype(z)::value, decltype(y)::value>;
    g.b = b;
    g.uy = S::N2Y;
    g.n1y = S::N1Y;
    g.uz = S::N2Z;
    g.n1z = S::N1Z;
  });
  return g;
}

int launch_yz_rect(int ny, int nz, int mode, void* data, const YzPlaneParams& p, hipStream_t s) {
  const int b = rect_b(ny, nz);
  int rc = 0;
  if (p.planes <= 0 || p.planes * b > 0x7fffffffL || !rect_length(ny) || !rect_length(nz) || ny == nz ||
      !rect_dispatch(nz, ny / b, [&](auto z, auto y) {
        rc = launch_rect<decltype(z)::value, decltype(y)::value>(mode, b, data, p, s);
      })) {
    set_last_error("two-launch y-z pass: unsupported %d x %d planes", ny, nz);
    return WFS_ERR_UNSUPPORTED;
  }
  return rc;
}

}  // namespace wfs
