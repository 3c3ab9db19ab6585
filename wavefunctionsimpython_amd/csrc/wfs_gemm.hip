// Strided batched GEMM on the bf16 matrix cores of gfx950, FP32 accumulation.
//
//   C[b](m, n) = alpha * sum_k A[b](m, k) B[b](k, n) + beta * C[b](m, n)
//
// with every operand addressed by explicit element strides, so one kernel
// serves all contractions of the Fourier neural operator (truncated DFTs along
// each axis, channel mixing, spectral weights) and their backward passes
// (which are the same contractions with swapped strides).  A and B are FP32 in
// memory and rounded to bf16 (nearest even) as they are staged into LDS; the
// bf16 inputs are what the matrix cores multiply.
//
// Split operands (flags bit 0: A, bit 1: B): the operand is staged as two bf16
// parts, hi = bf16(x) and lo = bf16(x - hi), and the tile product adds
// Ahi Bhi + Alo Bhi + Ahi Blo (lo lo is dropped), so that operand carries about
// 16 significant bits.  The Fourier neural operator splits its activations and
// keeps weights and transform tables in plain bf16: rounding a fixed operand
// perturbs the map by a fixed amount, while rounding activations adds noise
// that does not shrink with the change of the input.
//
// Block tile (32*WM) x (32*WN) x 32, one wavefront per 32 x 32 sub-tile, using
// gfx950's v_mfma_f32_32x32x16_bf16 (16 k per instruction, twice the rate of the 8-k
// form): lane l gives 8 k values of row l%32 of A and the same 8 k values of column l%32
// of B; accumulator item v of lane l is C[8(v/4)+4(l/32)+v%4][l%32].  Which k a lane's
// element stands for needs no care: the instruction sums A[i][k] B[k][j] over the 16
// (lane half, element) slots, so any assignment of a step's 16 k values to those slots
// that A and B share gives the same sum.  Lane l's elements e are k = k0 + 8(e/4) +
// 4(l/32) + e%4 here (the two 4-element runs of the 8-k form's layout side by side).
//
// Split-K: gridDim.z = batch * splits; with splits > 1 each block writes its
// partial tile to a workspace and a second kernel adds the splits in a fixed
// order (deterministic), then applies alpha/beta.
#include "wfs_internal.h"

namespace wfs {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// the k values of two 4-element runs as one 8-element operand
__device__ __forceinline__ s16x8 cat8(const bf16x4& a, const bf16x4& b) {
  return s16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// C += A B over 16 k on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16)
__device__ __forceinline__ f32x16 mfma16(const s16x8& a, const s16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                  0, 0);
}

// round to nearest even (gfx950 converts in hardware: v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned short f32_to_bf16(float f) {
  return __builtin_bit_cast(unsigned short, (__bf16)f);
}

struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  float* work;         // split-K partials [batch][splits][M][N]
  long M, N, K;
  long sAb, sAm, sAk;
  long sBb, sBm_unused, sBk, sBn;
  long sCb, sCm, sCn;
  float alpha, beta;
  int batch, splits;
  int flags;           // bit 0: split A into hi + lo; bit 1: split B; bit 2: do not store C
  const float* bias;   // per-row bias added after alpha/beta (may be null)
  float* act;          // GELU of the result, same strides as C (may be null)
  long kchunk;         // K range per split (multiple of 32)
};

constexpr int kBK = 32;

// C = alpha acc + beta C (+ bias[m]); act = GELU(C); C not stored with flag bit 2
__device__ __forceinline__ void epilogue(const GemmArgs& g, long b, long m, long n, float accv) {
  const long off = b * g.sCb + m * g.sCm + n * g.sCn;
  float val = (g.beta != 0.0f) ? g.alpha * accv + g.beta * g.C[off] : g.alpha * accv;
  if (g.bias) val = val + g.bias[m];
  if (!(g.flags & 4)) g.C[off] = val;
  if (g.act) g.act[off] = gelu_f(val);
}

template <int WM, int WN, bool SA, bool SB>
__global__ __launch_bounds__(64 * WM * WN) void gemm_bf16_kernel(GemmArgs g) {
  constexpr int BM = 32 * WM, BN = 32 * WN;
  constexpr int NT = 64 * WM * WN;
  // k-contiguous bf16 tiles, padded by 4 elements against bank conflicts
  __shared__ unsigned short As[BM][kBK + 4];
  __shared__ unsigned short Bs[BN][kBK + 4];
  __shared__ unsigned short Al[SA ? BM : 1][kBK + 4];
  __shared__ unsigned short Bl[SB ? BN : 1][kBK + 4];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const int b = blockIdx.z / g.splits;
  const int split = blockIdx.z % g.splits;
  const long n0 = long(blockIdx.x) * BN;   // x: column tiles (the long dimension of the network's GEMMs)
  const long m0 = long(blockIdx.y) * BM;
  const long kbeg = long(split) * g.kchunk;
  long kend = kbeg + g.kchunk;
  if (kend > g.K) kend = g.K;

  const float* __restrict__ A = g.A + long(b) * g.sAb;
  const float* __restrict__ B = g.B + long(b) * g.sBb;
  const bool a_k_fast = (g.sAk == 1);
  const bool b_n_fast = (g.sBn == 1);
  // 16-byte loads of four consecutive elements along the contiguous axis when every
  // quad start is 16-byte aligned (k0 is a multiple of 32)
  const bool a_vec = a_k_fast && (g.sAm % 4 == 0) && (g.sAb % 4 == 0) &&
                     (reinterpret_cast<unsigned long>(g.A) % 16 == 0);
  const bool b_vec = b_n_fast && (g.sBk % 4 == 0) && (g.sBb % 4 == 0) &&
                     (reinterpret_cast<unsigned long>(g.B) % 16 == 0);

  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;

  for (long k0 = kbeg; k0 < kend; k0 += kBK) {
    // stage A (BM x 32) and B (32 x BN) as bf16
    if (a_vec) {
      for (int e = tid; e < BM * (kBK / 4); e += NT) {
        const int mm = e / (kBK / 4), kk = (e % (kBK / 4)) * 4;
        const long m = m0 + mm, k = k0 + kk;
        float v[4];
        if (m < g.M && k + 3 < kend) {
          const float4 q = *reinterpret_cast<const float4*>(A + m * g.sAm + k);
          v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = (m < g.M && k + j < kend) ? A[m * g.sAm + k + j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const unsigned short h = f32_to_bf16(v[j]);
          As[mm][kk + j] = h;
          if constexpr (SA) Al[mm][kk + j] = f32_to_bf16(v[j] - __uint_as_float(unsigned(h) << 16));
        }
      }
    } else {
      for (int e = tid; e < BM * kBK; e += NT) {
        int mm, kk;
        if (a_k_fast) { mm = e / kBK; kk = e % kBK; } else { kk = e / BM; mm = e % BM; }
        const long m = m0 + mm, k = k0 + kk;
        const float v = (m < g.M && k < kend) ? A[m * g.sAm + k * g.sAk] : 0.0f;
        const unsigned short h = f32_to_bf16(v);
        As[mm][kk] = h;
        if constexpr (SA) Al[mm][kk] = f32_to_bf16(v - __uint_as_float(unsigned(h) << 16));
      }
    }
    if (b_vec) {
      for (int e = tid; e < kBK * (BN / 4); e += NT) {
        const int kk = e / (BN / 4), nn = (e % (BN / 4)) * 4;
        const long n = n0 + nn, k = k0 + kk;
        float v[4];
        if (k < kend && n + 3 < g.N) {
          const float4 q = *reinterpret_cast<const float4*>(B + k * g.sBk + n);
          v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = (k < kend && n + j < g.N) ? B[k * g.sBk + n + j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const unsigned short h = f32_to_bf16(v[j]);
          Bs[nn + j][kk] = h;
          if constexpr (SB) Bl[nn + j][kk] = f32_to_bf16(v[j] - __uint_as_float(unsigned(h) << 16));
        }
      }
    } else {
      for (int e = tid; e < BN * kBK; e += NT) {
        int nn, kk;
        if (b_n_fast) { kk = e / BN; nn = e % BN; } else { nn = e / kBK; kk = e % kBK; }
        const long n = n0 + nn, k = k0 + kk;
        const float v = (n < g.N && k < kend) ? B[k * g.sBk + n * g.sBn] : 0.0f;
        const unsigned short h = f32_to_bf16(v);
        Bs[nn][kk] = h;
        if constexpr (SB) Bl[nn][kk] = f32_to_bf16(v - __uint_as_float(unsigned(h) << 16));
      }
    }
    __syncthreads();
    const int row = wm * 32 + (lane & 31);
    const int col = wn * 32 + (lane & 31);
    const int kq = 4 * (lane >> 5);
#pragma unroll
    for (int kk = 0; kk < kBK; kk += 16) {
      s16x8 a, bb;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[j] = (short)As[row][kk + kq + j];
        a[4 + j] = (short)As[row][kk + 8 + kq + j];
        bb[j] = (short)Bs[col][kk + kq + j];
        bb[4 + j] = (short)Bs[col][kk + 8 + kq + j];
      }
      if constexpr (SA) {
        s16x8 al;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          al[j] = (short)Al[row][kk + kq + j];
          al[4 + j] = (short)Al[row][kk + 8 + kq + j];
        }
        acc = mfma16(al, bb, acc);
      }
      if constexpr (SB) {
        s16x8 bl;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          bl[j] = (short)Bl[col][kk + kq + j];
          bl[4 + j] = (short)Bl[col][kk + 8 + kq + j];
        }
        acc = mfma16(a, bl, acc);
      }
      acc = mfma16(a, bb, acc);
    }
    __syncthreads();
  }

  const long n = n0 + wn * 32 + (lane & 31);
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const long m = m0 + wm * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
    if (m < g.M && n < g.N) {
      if (g.splits == 1) {
        epilogue(g, b, m, n, acc[v]);
      } else {
        g.work[((long(b) * g.splits + split) * g.M + m) * g.N + n] = acc[v];
      }
    }
  }
}

// one wavefront per output element: lane l adds splits l, l + 64, ... in order, then a
// fixed xor tree across the lanes (deterministic)
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(GemmArgs g) {
  const long mn = g.M * g.N;
  const long total = long(g.batch) * mn;
  const int lane = threadIdx.x & 63;
  const long e = long(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (e >= total) return;   // uniform per wavefront
  const long b = e / mn, r = e % mn;
  const float* __restrict__ w = g.work + long(b) * g.splits * mn + r;
  float s = 0.0f;
  for (int sp = lane; sp < g.splits; sp += 64) s += w[long(sp) * mn];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) epilogue(g, b, r / g.N, r % g.N, s);
}

// ---------------------------------------------------------------------------
// One layer of the Fourier neural operator, fused over a grid line.  For the line
// r = (x, y) (all n = 32 NZC points along z) and all channels:
//   u  = W v + Z Gz + b        (W: C x cin, v: cin channels, Z: the layer's inverse
//                               spectral path before its last (z) stage, C x tm per line)
//   v' = GELU(u) or u
//   T' = v' Fz                 (the next layer's first (z) spectral stage, C x tm per line)
// which the unfused network computes as four GEMMs and writes S = Z Gz and u to HBM in
// between.  Operand rounding is that of those GEMMs: W, Gz, Fz plain bf16, v, Z and v'
// split into bf16 hi + lo; products accumulate in FP32 (in another order).
//
// One wavefront per line, no LDS and no barriers.  The transposed product is formed,
// u^T = v^T W^T + Gz^T Z^T, so that (in 8-k runs: lane l holds A[l%32][8s+4(l/32)..+3],
// B[8s+4(l/32)..+3][l%32], two runs s = 2S, 2S + 1 per 16-k instruction, and
// accumulator item i is C[8(i/4)+4(l/32)+i%4][l%32]) every operand comes straight from
// memory or from the previous product: the A fragment of v^T is four channel rows at one
// z (each load instruction reads 2 x 128 contiguous bytes), W^T, Gz^T and Fz are per-lane
// constants held in registers, Z^T is one 16-byte load per run, and the accumulator of a
// 32-point z chunk of u^T, items 4q..4q+3, is already the A run of v' for the z run q of
// T = v' Fz.  A chunk takes 12 matrix instructions (W v, Z Gz and v' Fz, two each per
// 16 k for the hi and lo parts).  C, cin, tm <= 32.
//
// BWD: the layer's transposed product in the same form, for the backward pass
//   vn = (W^T g + T' Fz^T) GELU'(u),  T = vn Gz^T
// with g in v, T' (the gradient of the layer's z stage) in Z, W stored [cin][C], the two tables
// exchanged, u in up (null: no factor) and no bias: what the composition writes and reads in
// between (W^T g, its sum with the spectral term, the product with GELU') stays in registers.
// At 64^3, C = 32: 41 us, against 150 us for the four launches it replaces (27 + 27 us for the two
// GEMMs that write W^T g and add the spectral term, 23 for GELU', 73 for the z stage).
//
// Wavefronts in flight: the kernel waits for memory.  n <= 64 has at most 4096 lines, one a wavefront (ONE_LINE):
// its next chunk's loads go into the registers of the chunk that the matrix cores have just taken, and the
// unrolled chunk loop (rolled, its addresses spill 12 to 21 registers) holds 128 registers at most, four
// wavefronts per SIMD; at three, 64^3 was 1.33 rounds of the card: 64^3 forward 253 -> 226 us, a training sample
// 805 -> 727 (C = 32, 4 layers).  Larger n keeps three (four spill: a training sample at 128^3 3415 -> 3512 us) and
// two chunk buffers, and its blocks, as many as fit the card at once (kLayerBlocks), walk the lines: the
// tables are staged once a block and no load waits for a block's start.  us, 2048 blocks against 768: 128^3 forward
// 981 -> 890 (942 with four wavefronts), C = 16 with 16 modes 628 -> 530, C = 18 506 -> 441, 96^3 with C = 24 285 ->
// 241, training samples at 128^3 3525 -> 3415, at 96^3 with C = 20 826 -> 770.
//
// LAYER_LAST: the last layer with the projection, out = base + rscale (Q u + qb) for one or two
// rows (Q bf16 as in the GEMM, u FP32): the lanes sum their half of the channels of one z from the
// chunk's LDS tile.  Without it the layer wrote u and a GEMM with 2 useful rows of 32 and an
// elementwise pass read it back: 161 + 79 + 14 us at 128^3, C = 32; here 111 (165 where u is stored).
// ---------------------------------------------------------------------------
struct LayerArgs {
  const float* W;
  const float* v;
  const float* Z;      // may be null (no spectral term)
  const float* bias;
  const float* Gz;     // [tm][n]
  const float* Fz;     // [n][tm]
  float* u;            // may be null
  float* vn;           // may be null
  float* T;            // may be null
  int cin, C, tm, act;
  long rows;           // lines (n * n)
  const float* up = nullptr;   // backward form: pre-activations [C][n^3] whose GELU' multiplies vn (may be null)
  // last form: out = base + rscale (Q u + qb), cout <= 2 rows
  const float* Q = nullptr;    // [cout][C]
  const float* qb = nullptr;
  const float* base = nullptr; // [cout][n^3] (may be null: zero)
  float* out = nullptr;        // [cout][n^3]
  float rscale = 1.0f;
  int cout = 0;
};
enum { LAYER_FORWARD = 0, LAYER_BACKWARD = 1, LAYER_LAST = 2 };

__device__ __forceinline__ void split4(const float (&x)[4], bf16x4& hi, bf16x4& lo) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned short h = f32_to_bf16(x[j]);
    hi[j] = (short)h;
    lo[j] = (short)f32_to_bf16(x[j] - __uint_as_float(unsigned(h) << 16));
  }
}

template <int NZC, int MODE, bool QUADS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NZC <= 2 ? 4 : 3))) void fno_layer_kernel(LayerArgs g) {
  constexpr bool BWD = MODE == LAYER_BACKWARD;
  constexpr bool ONE_LINE = NZC <= 2;                // a wavefront per line
  constexpr int n = 32 * NZC;
  constexpr int GP = kBK + 4;                        // padded rows of the transform tables
  __shared__ unsigned short GzT[n][GP];              // A = Gz^T: [z][j]
  __shared__ unsigned short FzT[32][n + 4];          // B = Fz:   [j][z]
  __shared__ float tiles[4][32][36];                 // per wavefront: a 32 x 32 (channel, z) chunk
  const int lane = threadIdx.x & 63;
  const int lc = lane & 31;
  const int kq = 4 * (lane >> 5);
  const int C = g.C, cin = g.cin, tm = g.tm;
  const long rows = g.rows;
  const unsigned P = unsigned(rows * n);             // C * P * 4 bytes < 2^32 (n <= 128, C <= 32)
  const int kin = (cin + 7) / 8;                     // k steps of W v
  const int ktm = g.Z ? (tm + 7) / 8 : 0;            // k steps of Z Gz

  for (int e = threadIdx.x; e < n * 32; e += blockDim.x) {
    const int z = e / 32, j = e % 32;
    const float gz = j < tm && (BWD ? g.T : g.Z) ? g.Gz[j * n + z] : 0.0f;
    const float fz = j < tm && (BWD ? g.Z : g.T) ? g.Fz[z * tm + j] : 0.0f;
    GzT[z][j] = f32_to_bf16(BWD ? fz : gz);
    FzT[j][z] = f32_to_bf16(BWD ? gz : fz);
  }
  __shared__ float proj[2][MODE == LAYER_LAST ? 32 : 1];   // the projection's rows (bf16 values)
  if constexpr (MODE == LAYER_LAST) {
    if (threadIdx.x < 64) {
      const int o = threadIdx.x >> 5, c = threadIdx.x & 31;
      proj[o][c] = o < g.cout && c < C ? __uint_as_float(unsigned(f32_to_bf16(g.Q[o * C + c])) << 16) : 0.0f;
    }
  }
  bf16x4 Wf[4];                                      // B = W^T: (k = c_in, n = c_out = lc)
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 8 * s + kq + j;
      Wf[s][j] = (short)((lc < C && k < cin) ? f32_to_bf16(g.W[BWD ? k * C + lc : lc * cin + k]) : 0);
    }
  const float bias_c = !BWD && lc < C ? g.bias[lc] : 0.0f;
  __syncthreads();

  // 32-bit byte offsets from the buffers' base addresses (C * n^3 * 4 < 2^32); loads past
  // the operand's extent read a valid element instead, whose weight (W, table) is zero, so no
  // load is conditional; rows past C come out of no store
  const char* __restrict__ vb = reinterpret_cast<const char*>(g.v);
  const char* __restrict__ zb = reinterpret_cast<const char*>(g.Z);
  char* __restrict__ ub = reinterpret_cast<char*>(g.u);
  char* __restrict__ nb = reinterpret_cast<char*>(g.vn);
  char* __restrict__ tb = reinterpret_cast<char*>(g.T);
  const char* __restrict__ pb = reinterpret_cast<const char*>(g.up);
  const unsigned lcC = unsigned(lc < C ? lc : C - 1);
  const long stride = long(gridDim.x) * (blockDim.x / 64);
  // the A fragments of v^T for one 32-point chunk; the next chunk's (or the next line's
  // first chunk's) are loaded while the current one is computed
  // QUADS (cin a multiple of 4): the channels 8 s + kq .. + 3 exist together or not at all, so four
  // lane offsets and four scalar bases address all rows
  unsigned vrow[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) vrow[s] = unsigned(8 * s + kq < cin ? 8 * s + kq : 0) * P + unsigned(lc);
  auto load_v = [&](unsigned ru, int ch, float (&x)[16]) {
    const unsigned at = ru * n + 32 * ch;
    if constexpr (QUADS) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const char* __restrict__ base = vb + (long(j) * P + at) * 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) x[4 * s + j] = *reinterpret_cast<const float*>(base + vrow[s] * 4u);
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = 8 * s + kq + j;
          x[4 * s + j] =
              *reinterpret_cast<const float*>(vb + ((c < cin ? unsigned(c) : unsigned(cin - 1)) * P + at + lc) * 4u);
        }
    }
  };
  // A chunk goes to and comes from memory as whole 128-byte lines: lane l holds z = 4 (l % 8) ..
  // + 3 of channel 8 i + l / 8 in part i.  The wavefront's own LDS tile turns that into the
  // matrix layout (four consecutive z of channel l % 32) and back.  Stored from the matrix layout,
  // an instruction wrote 32-byte pieces of 32 channels, whose lines lie n^3 floats apart (a power
  // of two at 64 and 128: one memory channel): a bare copy in that pattern takes 202 us at 128^3,
  // in whole lines 114.  A 128^3 layer went from 250 to 188 us (422 to 246 where u is stored too,
  // backward 401 to 285), a 64^3 one from 43 to 35 (46 to 38, 56 to 47).  What is left is those
  // power-of-two strides: with 4 KiB more between channels a layer takes 170 us.  Loading up or Z
  // a chunk or a line ahead was slower (backward 320 us, spilled registers).
  float (*tile)[36] = tiles[threadIdx.x >> 6];
  const float qbias = MODE == LAYER_LAST && (kq >> 2) < g.cout ? g.qb[kq >> 2] : 0.0f;
  const int mc = lane >> 3, mz = 4 * (lane & 7);
  auto to_memory = [&](char* base, unsigned at) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 8 * i + mc;
      const float4 y = *reinterpret_cast<const float4*>(&tile[c][mz]);
      if (c < C) *reinterpret_cast<float4*>(base + (unsigned(c) * P + at + unsigned(mz)) * 4u) = y;
    }
    __builtin_amdgcn_wave_barrier();
  };
  auto load_up = [&](unsigned ru, int ch, float4 (&y)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned c = unsigned(8 * i + mc < C ? 8 * i + mc : C - 1);
      y[i] = *reinterpret_cast<const float4*>(pb + (c * P + ru * n + 32 * ch + unsigned(mz)) * 4u);
    }
  };
  float xv[16];
  long r = long(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
  if (r < rows) load_v(unsigned(r), 0, xv);
  for (; r < rows; r += stride) {
    const unsigned ru = unsigned(r);
    bf16x4 Zh[4], Zl[4];                             // B = Z^T: (k = j, n = c = lc)
#pragma unroll
    for (int s = 0; s < 4; ++s) { Zh[s] = bf16x4{0, 0, 0, 0}; Zl[s] = bf16x4{0, 0, 0, 0}; }
    if (zb) {
      // four consecutive j per lane: one 16-byte load (tm is a multiple of 4, so a quad lies
      // wholly inside or wholly past the row; past it, the row's last quad meets zero table rows)
      const unsigned row = (lcC * unsigned(rows) + ru) * unsigned(tm);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k0 = 8 * s + kq;
        const float4 y = *reinterpret_cast<const float4*>(zb + (row + unsigned(k0 < tm ? k0 : tm - 4)) * 4u);
        const float x[4] = {y.x, y.y, y.z, y.w};
        split4(x, Zh[s], Zl[s]);
      }
    }
    f32x16 accT;
#pragma unroll
    for (int i = 0; i < 16; ++i) accT[i] = 0.0f;
    const unsigned line = ru * n;
    const long rnext = r + stride;
    // the chunk after ch: this line's ch + 1, or the next line's first
    auto prefetch = [&](int ch, float (&x)[16]) {
      if (ch + 1 < NZC) load_v(ru, ch + 1, x);
      else if (!ONE_LINE && rnext < rows) load_v(unsigned(rnext), 0, x);
    };
    // chunk ch of this line from x (its loads were issued one chunk earlier)
    auto process = [&](int ch, float (&x)[16]) {
      float4 up[4];
      if constexpr (BWD) {
        if (pb) load_up(ru, ch, up);
      }
      f32x16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
      // k steps of 16: the 8-k steps 2S and 2S + 1 side by side (past cin and tm the
      // operands are zero)
#pragma unroll
      for (int S = 0; S < 2; ++S) {
        if (2 * S < kin) {
          bf16x4 ah0, al0, ah1, al1;
          float x0[4] = {x[8 * S], x[8 * S + 1], x[8 * S + 2], x[8 * S + 3]};
          float x1[4] = {x[8 * S + 4], x[8 * S + 5], x[8 * S + 6], x[8 * S + 7]};
          split4(x0, ah0, al0);
          split4(x1, ah1, al1);
          const s16x8 w = cat8(Wf[2 * S], Wf[2 * S + 1]);
          acc = mfma16(cat8(al0, al1), w, acc);
          acc = mfma16(cat8(ah0, ah1), w, acc);
        }
      }
      if constexpr (ONE_LINE) prefetch(ch, x);
#pragma unroll
      for (int S = 0; S < 2; ++S) {
        if (2 * S < ktm) {
          s16x8 a;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            a[j] = (short)GzT[32 * ch + lc][16 * S + kq + j];
            a[4 + j] = (short)GzT[32 * ch + lc][16 * S + 8 + kq + j];
          }
          acc = mfma16(a, cat8(Zl[2 * S], Zl[2 * S + 1]), acc);
          acc = mfma16(a, cat8(Zh[2 * S], Zh[2 * S + 1]), acc);
        }
      }
      // lane: column c = lc; items 4q..4q+3: z = 32 ch + 8 q + kq + 0..3; the items of q = 2Q
      // and 2Q + 1 are the A operand of one 16-k step of T = v' Fz
      const unsigned at = line + 32 * ch;
      float gv[16];
      if constexpr (BWD) {
        if (pb) {
#pragma unroll
          for (int i = 0; i < 4; ++i) *reinterpret_cast<float4*>(&tile[8 * i + mc][mz]) = up[i];
          __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float4 y = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          if (pb) y = *reinterpret_cast<const float4*>(&tile[lc][8 * q + kq]);
          const float uv[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float val = acc[4 * q + j];
            gv[4 * q + j] = pb ? val * gelu_grad(uv[j]) : val;
          }
        }
        __builtin_amdgcn_wave_barrier();
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = acc[i] + bias_c;
        if (ub || MODE == LAYER_LAST) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(&tile[lc][8 * q + kq]) =
                make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
          if (ub) to_memory(ub, at);
        }
        if constexpr (MODE == LAYER_LAST) {
          // lane: z = lc, channels 16 (l / 32) ..; then the other half's sums, and half o stores row o
          __builtin_amdgcn_wave_barrier();
          float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float y = tile[4 * kq + i][lc];
            s0 = __builtin_fmaf(proj[0][4 * kq + i], y, s0);
            s1 = __builtin_fmaf(proj[1][4 * kq + i], y, s1);
          }
          __builtin_amdgcn_wave_barrier();
          const float mine = kq ? s1 : s0, other = __shfl_xor(kq ? s0 : s1, 32, 64);
          const int o = kq >> 2;
          if (o < g.cout) {
            const unsigned e = unsigned(o) * P + at + unsigned(lc);
            const float y = g.rscale * (mine + other + qbias);
            g.out[e] = g.base ? g.base[e] + y : y;
          }
          return;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) gv[i] = g.act ? gelu_f(acc[i]) : acc[i];
      }
      if (nb) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4*>(&tile[lc][8 * q + kq]) =
              make_float4(gv[4 * q], gv[4 * q + 1], gv[4 * q + 2], gv[4 * q + 3]);
        to_memory(nb, at);
      }
      if (tb) {
#pragma unroll
        for (int Q = 0; Q < 2; ++Q) {
          bf16x4 ahq[2], alq[2], bq[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int q = 2 * Q + h;
            const float gq[4] = {gv[4 * q], gv[4 * q + 1], gv[4 * q + 2], gv[4 * q + 3]};
            split4(gq, ahq[h], alq[h]);
#pragma unroll
            for (int j = 0; j < 4; ++j) bq[h][j] = (short)FzT[lc][32 * ch + 8 * q + kq + j];
          }
          const s16x8 b = cat8(bq[0], bq[1]);
          accT = mfma16(cat8(alq[0], alq[1]), b, accT);
          accT = mfma16(cat8(ahq[0], ahq[1]), b, accT);
        }
      }
    };
    if constexpr (ONE_LINE) {
#pragma unroll
      for (int ch = 0; ch < NZC; ++ch) process(ch, xv);
    } else {
      // chunks in pairs through two buffers, so that no register copy waits for a load in flight
      float xw[16];
#pragma unroll 1
      for (int ch = 0; ch < NZC; ch += 2) {
        prefetch(ch, xw);
        process(ch, xv);
        if (ch + 1 < NZC) {
          prefetch(ch + 1, xv);
          process(ch + 1, xw);
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) xv[i] = xw[i];   // odd chunk count: next line's first chunk
        }
      }
    }
    if (tb && lc < tm) {
      // accumulator: column j = lc, rows c = 8(i/4) + 4(l/32) + i%4
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int c = 8 * (i / 4) + kq + (i % 4);
        if (c < C)
          *reinterpret_cast<float*>(tb + ((unsigned(c) * unsigned(rows) + ru) * unsigned(tm) + lc) * 4u) = accT[i];
      }
    }
    if constexpr (ONE_LINE) break;
  }
}

// ---------------------------------------------------------------------------
// One stage of the truncated DFT along an axis between the z stages: for every slab s
//   out[s][i][c] = sum_k A[i][k] in[s][k][c],   c < ncol,
// A a transform table in bf16 ([ceil32(M)][ceil16(K)], zero padded), in as bf16 hi + lo, FP32
// accumulation (the operand rounding of wfs_gemm_bf16).  The columns of all slabs are numbered
// through, so a tile of 32 columns is full for any ncol; a tile's A fragments (8 consecutive k of a
// row) are one 16-byte load each, its B fragments eight loads of 32 columns each, both straight
// from memory: no LDS on the way to the matrix cores and no barriers.
//
// Reducing stages (M = 2 m <= 32 rows, K = 2 n): the block's four wavefronts take a quarter of k
// each and add their tiles in LDS, so that the x stage (m^2 columns per channel, 144 tiles at 12
// modes and 32 channels) still has four wavefronts a tile.  Expanding stages (K = 2 m <= 32,
// M = 2 n): a wavefront holds its tile's B fragments and the four wavefronts share the rows.
// The strided GEMM staged both operands element by element through LDS with 64-bit index
// arithmetic, a 32 x 32 tile per 12 useful columns: per launch at 128^3, C = 32, m = 12 (y, x,
// inverse x, inverse y) 44, 23, 7, 33 us; here 16, 5, 5, 15 (the y stages move 63 MB: 4 TB/s).
// ---------------------------------------------------------------------------
__device__ __forceinline__ s16x8 load_a8(const unsigned short* __restrict__ A, long at) {
  return *reinterpret_cast<const s16x8*>(A + at);
}

// eight rows k0 .. k0 + 7 of a column, rows from K on zero (their addresses clamped)
__device__ __forceinline__ void load_b8(const float* __restrict__ col, int ncol, int k0, int K, float (&x)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = col[long(k0 + j < K ? k0 + j : K - 1) * ncol];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (k0 + j >= K) x[j] = 0.0f;
}

__device__ __forceinline__ void split8v(const float (&x)[8], s16x8& hi, s16x8& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const unsigned short h = f32_to_bf16(x[j]);
    hi[j] = (short)h;
    lo[j] = (short)f32_to_bf16(x[j] - __uint_as_float(unsigned(h) << 16));
  }
}

// M <= 32
__global__ __launch_bounds__(256) void fno_reduce_stage_kernel(const unsigned short* __restrict__ A,
                                                               const float* __restrict__ in, float* __restrict__ out,
                                                               int M, int K, int ncol, long cols) {
  __shared__ float red[3][64][17];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5;
  const long j = long(blockIdx.x) * 32 + (lane & 31);
  const long jj = j < cols ? j : cols - 1;
  const long slab = jj / ncol;
  const int c = int(jj - slab * ncol);
  const float* __restrict__ col = in + slab * K * ncol + c;
  const int kp = (K + 15) / 16 * 16;
  const long arow = long(lane & 31) * kp;
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  // k steps of 16: wavefront w takes steps w, w + 4, ...; a lane half takes 8 consecutive k
  const int steps = kp / 16;
  for (int s = wave; s < steps; s += 8) {
    // two steps' loads in flight together (past the last step: zero fragments)
    float x[2][8];
    s16x8 a[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k0 = 16 * (s + 4 * u) + 8 * half;
      load_b8(col, ncol, k0, K, x[u]);
      a[u] = load_a8(A, arow + (k0 < kp ? k0 : 8 * half));
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s16x8 bh, bl;
      split8v(x[u], bh, bl);
      acc = mfma16(a[u], bl, acc);
      acc = mfma16(a[u], bh, acc);
    }
  }
  if (wave) {
#pragma unroll
    for (int i = 0; i < 16; ++i) red[wave - 1][lane][i] = acc[i];
  }
  __syncthreads();
  if (wave == 0 && j < cols) {
    float* __restrict__ o = out + slab * M * ncol + c;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 8 * (i / 4) + 4 * half + i % 4;
      const float v = (acc[i] + red[0][lane][i]) + (red[1][lane][i] + red[2][lane][i]);
      if (row < M) o[long(row) * ncol] = v;
    }
  }
}

// K <= 32; blockIdx.y: this block's share of the 32-row tiles
__global__ __launch_bounds__(256) void fno_expand_stage_kernel(const unsigned short* __restrict__ A,
                                                               const float* __restrict__ in, float* __restrict__ out,
                                                               int M, int K, int ncol, long cols) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5;
  const long j = long(blockIdx.x) * 32 + (lane & 31);
  const long jj = j < cols ? j : cols - 1;
  const long slab = jj / ncol;
  const int c = int(jj - slab * ncol);
  const float* __restrict__ col = in + slab * K * ncol + c;
  const int kp = (K + 15) / 16 * 16;
  s16x8 bh[2], bl[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    float x[8];
    load_b8(col, ncol, 16 * s + 8 * half, K, x);
    split8v(x, bh[s], bl[s]);
  }
  float* __restrict__ o = out + slab * M * ncol + c;
  const int tiles = (M + 31) / 32;
  for (int t = int(blockIdx.y) * 4 + wave; t < tiles; t += 4 * int(gridDim.y)) {
    const long arow = long(32 * t + (lane & 31)) * kp + 8 * half;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    const s16x8 a0 = load_a8(A, arow);
    acc = mfma16(a0, bl[0], acc);
    acc = mfma16(a0, bh[0], acc);
    if (kp > 16) {
      const s16x8 a1 = load_a8(A, arow + 16);
      acc = mfma16(a1, bl[1], acc);
      acc = mfma16(a1, bh[1], acc);
    }
    if (j < cols) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = 32 * t + 8 * (i / 4) + 4 * half + i % 4;
        if (row < M) o[long(row) * ncol] = acc[i];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Complex per-mode channel mixing of the Fourier neural operator:
//   O[o][q] = sum_i R[q][i][o] X[i][q]     (complex: Or = Rr Xr - Ri Xi, Oi = Ri Xr + Rr Xi)
// for m3 modes q and C channels, with the GEMM path's operand rounding (R plain bf16,
// X as bf16 hi + lo, FP32 accumulation).  The GEMM path issues it as four strided
// batched GEMMs with N = 1 (one 32 x 32 tile per mode for one useful column); here four
// lanes own one (mode, output channel) pair.  Layouts: R [m3][C][C] ([q][i][o]),
// X and O [C][2][m3] (real parts, then imaginary parts).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fno_modes_kernel(const float* __restrict__ Rr, const float* __restrict__ Ri,
                                                        const float* __restrict__ X, float* __restrict__ O,
                                                        int m3, int C) {
  // four lanes per (mode, output channel): lane h sums input channels i = h, h + 4, ...,
  // then the four partial sums are added across the lanes (xor 1, xor 2)
  const long t = long(blockIdx.x) * 256 + threadIdx.x;
  const long pair = t >> 2;
  const int h = int(t & 3);
  const bool live = pair < long(m3) * C;
  const long pp = live ? pair : 0;
  const int q = int(pp / C), o = int(pp % C);
  const float* __restrict__ rr = Rr + long(q) * C * C + o;
  const float* __restrict__ ri = Ri + long(q) * C * C + o;
  float srr = 0.0f, sii = 0.0f, sir = 0.0f, sri = 0.0f;   // Rr Xr, Ri Xi, Ri Xr, Rr Xi
  for (int i = h; i < C; i += 4) {
    const float a = __uint_as_float(unsigned(f32_to_bf16(rr[long(i) * C])) << 16);
    const float b = __uint_as_float(unsigned(f32_to_bf16(ri[long(i) * C])) << 16);
    const float xr = X[long(i) * 2 * m3 + q], xi = X[long(i) * 2 * m3 + m3 + q];
    const float xrh = __uint_as_float(unsigned(f32_to_bf16(xr)) << 16);
    const float xih = __uint_as_float(unsigned(f32_to_bf16(xi)) << 16);
    const float xrl = __uint_as_float(unsigned(f32_to_bf16(xr - xrh)) << 16);
    const float xil = __uint_as_float(unsigned(f32_to_bf16(xi - xih)) << 16);
    srr = __builtin_fmaf(a, xrh, __builtin_fmaf(a, xrl, srr));
    sii = __builtin_fmaf(b, xih, __builtin_fmaf(b, xil, sii));
    sir = __builtin_fmaf(b, xrh, __builtin_fmaf(b, xrl, sir));
    sri = __builtin_fmaf(a, xih, __builtin_fmaf(a, xil, sri));
  }
#pragma unroll
  for (int off = 1; off < 4; off <<= 1) {
    srr += __shfl_xor(srr, off, 64);
    sii += __shfl_xor(sii, off, 64);
    sir += __shfl_xor(sir, off, 64);
    sri += __shfl_xor(sri, off, 64);
  }
  if (live && h == 0) {
    O[long(o) * 2 * m3 + q] = srr - sii;
    O[long(o) * 2 * m3 + m3 + q] = sir + sri;
  }
}

// ---------------------------------------------------------------------------
// Weight and bias gradients of a pointwise layer, gW[o][i] += sum_p g[o][p] v[i][p] and
// gb[o] += sum_p g[o][p], for up to 32 channels on both sides: one 32 x 32 tile whose k is the
// grid.  Both operands are contiguous along k, so a lane's fragments -- 16 points of row lane % 32
// of g and of v, the two lane halves side by side -- come straight from memory, with no LDS and no
// barriers.  Both operands are split into bf16 hi + lo (hi hi + lo hi + hi lo, FP32 accumulation,
// as the GEMM's split operands); the bias sum adds the FP32 values themselves.  Each wavefront
// takes every (4 gridDim.x)-th run of 32 points, the block's four tiles are added in LDS, and a
// second kernel adds the blocks' records in a fixed order.
// Reads 4 (C + cin) P bytes.  The strided GEMM it replaces computed this tile in blocks of 128 x 32
// with one wavefront in four at work, and the bias in a second pass over g: 114 + 13 us at 64^3,
// C = cin = 32 (67 MB); this pair of launches takes 15 + 5 us (4.5 TB/s in the first).
// ---------------------------------------------------------------------------
constexpr int kGradRecord = 33 * 32;   // floats per block: the tile [o][i], then the bias sums

__device__ __forceinline__ void split8(const float4& a, const float4& b, s16x8& hi, s16x8& lo) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const unsigned short h = f32_to_bf16(x[j]);
    hi[j] = (short)h;
    lo[j] = (short)f32_to_bf16(x[j] - __uint_as_float(unsigned(h) << 16));
  }
}

__global__ __launch_bounds__(256) void fno_weight_grad_kernel(const float* __restrict__ g, const float* __restrict__ v,
                                                              float* __restrict__ work, int C, int cin, long P) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane & 31;
  // rows past the channels read a valid row and count as zero
  const bool ga = row < C, va = row < cin;
  const float* __restrict__ gr = g + long(ga ? row : 0) * P + 16 * (lane >> 5);
  const float* __restrict__ vr = v + long(va ? row : 0) * P + 16 * (lane >> 5);
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  float bsum = 0.0f;
  const long stride = long(gridDim.x) * 4 * 32;
  long p = (long(blockIdx.x) * 4 + wave) * 32;
  float4 a[4], b[4];
  const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  auto load = [&](long at) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[j] = *reinterpret_cast<const float4*>(gr + at + 4 * j);
      b[j] = *reinterpret_cast<const float4*>(vr + at + 4 * j);
    }
  };
  if (p < P) load(p);
  for (; p < P; p += stride) {
    float4 ca[4], cb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ca[j] = ga ? a[j] : zero;
      cb[j] = va ? b[j] : zero;
    }
    if (p + stride < P) load(p + stride);
#pragma unroll
    for (int j = 0; j < 4; ++j) bsum += (ca[j].x + ca[j].y) + (ca[j].z + ca[j].w);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s16x8 ah, al, bh, bl;
      split8(ca[2 * h], ca[2 * h + 1], ah, al);
      split8(cb[2 * h], cb[2 * h + 1], bh, bl);
      acc = mfma16(al, bh, acc);
      acc = mfma16(ah, bl, acc);
      acc = mfma16(ah, bh, acc);
    }
  }
  bsum += __shfl_xor(bsum, 32, 64);
  // lane: column i = row; items: o = 8(v/4) + 4(lane/32) + v%4
  __shared__ float red[4][kGradRecord];
#pragma unroll
  for (int i = 0; i < 16; ++i) red[wave][(8 * (i / 4) + 4 * (lane >> 5) + i % 4) * 32 + row] = acc[i];
  if (lane < 32) red[wave][32 * 32 + row] = bsum;
  __syncthreads();
  for (int e = threadIdx.x; e < kGradRecord; e += 256)
    work[long(blockIdx.x) * kGradRecord + e] = (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
}

// block b: row b of the records (32: the bias), 32 columns by 16 strided parts of the blocks
__global__ __launch_bounds__(512) void fno_weight_grad_sum_kernel(const float* __restrict__ work, int nblk,
                                                                  float* __restrict__ gW, float* __restrict__ gb,
                                                                  int C, int cin) {
  const int col = threadIdx.x & 31, part = threadIdx.x >> 5;
  const int row = blockIdx.x;
  float s = 0.0f;
#pragma unroll 8
  for (int b = part; b < nblk; b += 16) s += work[long(b) * kGradRecord + row * 32 + col];
  __shared__ float red[16][32];
  red[part][col] = s;
  __syncthreads();
  if (part == 0) {
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += red[k][col];
    if (row < 32) {
      if (row < C && col < cin) gW[row * cin + col] += t;
    } else if (col < C) {
      gb[col] += t;
    }
  }
}

// ---------------------------------------------------------------------------
// Backward of the per-mode channel mixing O = R (.) X (fno_modes_kernel), one block per mode q:
//   gRr[q][i][o] += Xr[i] dOr[o] + Xi[i] dOi[o],  gRi[q][i][o] += Xr[i] dOi[o] - Xi[i] dOr[o]
//   dXr[i] = sum_o Rr dOr + Ri dOi,               dXi[i] = sum_o Rr dOi - Ri dOr
// R plain bf16 and dO as bf16 hi + lo in the sums, as the mixing itself takes them; the outer
// products are FP32.  32 lanes own a row i (o along the lanes, contiguous in memory), the row sums
// go over the lanes.  R is read and gR read and written once: 24 C^2 bytes per mode, 42 MB at 12
// modes and C = 32.  The eight strided GEMMs it replaces (K or N of 1 in a 32 x 32 tile) read and
// wrote gR twice and took 16 and 12 us each; this launch takes 12 us.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fno_modes_backward_kernel(const float* __restrict__ Rr,
                                                                 const float* __restrict__ Ri,
                                                                 const float* __restrict__ X,
                                                                 const float* __restrict__ dO, float* __restrict__ dX,
                                                                 float* __restrict__ gRr, float* __restrict__ gRi,
                                                                 int m3, int C) {
  __shared__ float x[2][256], d[2][256];
  const int q = blockIdx.x;
  for (int e = threadIdx.x; e < 2 * C; e += 256) {
    const int c = e % C, part = e / C;
    x[part][c] = X[(long(c) * 2 + part) * m3 + q];
    d[part][c] = dO[(long(c) * 2 + part) * m3 + q];
  }
  __syncthreads();
  const int lane = threadIdx.x & 31;
  for (int i = threadIdx.x >> 5; i < C; i += 8) {
    const float xr = x[0][i], xi = x[1][i];
    float sr = 0.0f, si = 0.0f;
    for (int o = lane; o < C; o += 32) {
      const long e = (long(q) * C + i) * C + o;
      const float dr = d[0][o], di = d[1][o];
      gRr[e] += __builtin_fmaf(xr, dr, xi * di);
      gRi[e] += __builtin_fmaf(xr, di, -(xi * dr));
      const float a = __uint_as_float(unsigned(f32_to_bf16(Rr[e])) << 16);
      const float b = __uint_as_float(unsigned(f32_to_bf16(Ri[e])) << 16);
      const float drh = __uint_as_float(unsigned(f32_to_bf16(dr)) << 16);
      const float dih = __uint_as_float(unsigned(f32_to_bf16(di)) << 16);
      const float drl = __uint_as_float(unsigned(f32_to_bf16(dr - drh)) << 16);
      const float dil = __uint_as_float(unsigned(f32_to_bf16(di - dih)) << 16);
      sr = __builtin_fmaf(a, drh, __builtin_fmaf(a, drl, sr));
      sr = __builtin_fmaf(b, dih, __builtin_fmaf(b, dil, sr));
      si = __builtin_fmaf(a, dih, __builtin_fmaf(a, dil, si));
      si = __builtin_fmaf(-b, drh, __builtin_fmaf(-b, drl, si));
    }
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {
      sr += __shfl_xor(sr, off, 64);
      si += __shfl_xor(si, off, 64);
    }
    if (lane == 0) {
      dX[long(i) * 2 * m3 + q] = sr;
      dX[(long(i) * 2 + 1) * m3 + q] = si;
    }
  }
}

}  // namespace wfs

using namespace wfs;

extern "C" int wfs_fno_modes(const float* Rr, const float* Ri, const float* X, float* O, int m3, int C,
                             void* stream) {
  if (!Rr || !Ri || !X || !O || m3 < 1 || C < 1) { set_last_error("wfs_fno_modes: bad argument"); return WFS_ERR_INVALID; }
  const long total = long(m3) * C * 4;
  hipLaunchKernelGGL(fno_modes_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), Rr, Ri, X, O, m3, C);
  WFS_HIP_CHECK(hipGetLastError());
  return 0;
}

constexpr long kLayerBlocks = 3 * 256;   // three blocks of four wavefronts on each of the 256 CUs

// a block takes four lines at a time
template <int NZC, int MODE, bool QUADS>
static void launch_layer_form(const LayerArgs& g, hipStream_t s) {
  const long want = (g.rows + 3) / 4;
  const unsigned blocks = unsigned(NZC <= 2 || want < kLayerBlocks ? want : kLayerBlocks);   // ONE_LINE: all lines
  hipLaunchKernelGGL((fno_layer_kernel<NZC, MODE, QUADS>), dim3(blocks), dim3(256), 0, s, g);
}

template <int MODE>
static void launch_layer(const LayerArgs& g, int n, hipStream_t s) {
#define WFS_LAYER(NZC)                                                   \
  if (g.cin % 4 == 0) launch_layer_form<NZC, MODE, true>(g, s);          \
  else launch_layer_form<NZC, MODE, false>(g, s);
  switch (n / 32) {
    case 1: WFS_LAYER(1) break;
    case 2: WFS_LAYER(2) break;
    case 3: WFS_LAYER(3) break;
    default: WFS_LAYER(4) break;
  }
#undef WFS_LAYER
}

// layer of the Fourier neural operator fused over grid lines (see fno_layer_kernel)
extern "C" int wfs_fno_layer(const float* W, const float* v, const float* Z, const float* bias, const float* Gz,
                             const float* Fz, float* u, float* vn, float* T, int cin, int C, int n, int tm, int act,
                             void* stream) {
  if (!W || !v || !bias) { set_last_error("wfs_fno_layer: null argument"); return WFS_ERR_INVALID; }
  if (n % 32 != 0 || n < 32 || n > 128 || C < 1 || C > 32 || cin < 1 || cin > 32 || tm < 4 || tm > 32 || tm % 4) {
    set_last_error("wfs_fno_layer: needs n in {32, 64, 96, 128}, C, cin <= 32 and tm a multiple of 4 up to 32 "
                   "(n=%d C=%d cin=%d tm=%d)", n, C, cin, tm);
    return WFS_ERR_UNSUPPORTED;
  }
  if ((Z && !Gz) || (T && (!Fz || !vn)) || (!u && !vn)) {
    set_last_error("wfs_fno_layer: Z needs Gz; T needs Fz and vn; one of u, vn is required");
    return WFS_ERR_INVALID;
  }
  if ((reinterpret_cast<unsigned long>(u) % 16) != 0 || (reinterpret_cast<unsigned long>(vn) % 16) != 0 ||
      (reinterpret_cast<unsigned long>(Z) % 16) != 0) {
    set_last_error("wfs_fno_layer: u, vn and Z must be 16-byte aligned");
    return WFS_ERR_INVALID;
  }
  const LayerArgs g{W, v, Z, bias, Gz, Fz, u, vn, T, cin, C, tm, act, long(n) * n};
  launch_layer<LAYER_FORWARD>(g, n, static_cast<hipStream_t>(stream));
  WFS_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int wfs_fno_last_layer(const float* W, const float* v, const float* Z, const float* bias, const float* Gz,
                                  const float* Q, const float* qb, const float* base, float rscale, float* u,
                                  float* out, int cin, int C, int cout, int n, int tm, void* stream) {
  if (!W || !v || !bias || !Q || !qb || !out || (Z && !Gz)) { set_last_error("wfs_fno_last_layer: null argument"); return WFS_ERR_INVALID; }
  if (n % 32 != 0 || n < 32 || n > 128 || C < 1 || C > 32 || cin < 1 || cin > 32 || cout < 1 || cout > 2 || tm < 4 ||
      tm > 32 || tm % 4) {
    set_last_error("wfs_fno_last_layer: needs n in {32, 64, 96, 128}, C, cin <= 32, cout <= 2 and tm a multiple of 4 "
                   "up to 32 (n=%d C=%d cin=%d cout=%d tm=%d)", n, C, cin, cout, tm);
    return WFS_ERR_UNSUPPORTED;
  }
  if ((reinterpret_cast<unsigned long>(u) % 16) != 0 || (reinterpret_cast<unsigned long>(Z) % 16) != 0) {
    set_last_error("wfs_fno_last_layer: u and Z must be 16-byte aligned");
    return WFS_ERR_INVALID;
  }
  LayerArgs g{W, v, Z, bias, Gz, nullptr, u, nullptr, nullptr, cin, C, tm, 0, long(n) * n};
  g.Q = Q;
  g.qb = qb;
  g.base = base;
  g.out = out;
  g.rscale = rscale;
  g.cout = cout;
  launch_layer<LAYER_LAST>(g, n, static_cast<hipStream_t>(stream));
  WFS_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int wfs_fno_layer_backward(const float* W, const float* g, const float* Tg, const float* u, const float* Gz,
                                      const float* Fz, float* gn, float* Tn, int cin, int C, int n, int tm,
                                      void* stream) {
  if (!W || !g || !gn || (Tg && !Fz) || (Tn && !Gz)) { set_last_error("wfs_fno_layer_backward: null argument"); return WFS_ERR_INVALID; }
  if (n % 32 != 0 || n < 32 || n > 128 || C < 1 || C > 32 || cin < 1 || cin > 32 || tm < 4 || tm > 32 || tm % 4) {
    set_last_error("wfs_fno_layer_backward: needs n in {32, 64, 96, 128}, C, cin <= 32 and tm a multiple of 4 up to 32 "
                   "(n=%d C=%d cin=%d tm=%d)", n, C, cin, tm);
    return WFS_ERR_UNSUPPORTED;
  }
  if ((reinterpret_cast<unsigned long>(u) % 16) != 0 || (reinterpret_cast<unsigned long>(gn) % 16) != 0 ||
      (reinterpret_cast<unsigned long>(Tg) % 16) != 0) {
    set_last_error("wfs_fno_layer_backward: u, gn and Tg must be 16-byte aligned");
    return WFS_ERR_INVALID;
  }
  const LayerArgs a{W, g, Tg, nullptr, Gz, Fz, nullptr, gn, Tn, cin, C, tm, 0, long(n) * n, u};
  launch_layer<LAYER_BACKWARD>(a, n, static_cast<hipStream_t>(stream));
  WFS_HIP_CHECK(hipGetLastError());
  return 0;
}

// gW += g v^T and gb += sum_p g (see fno_weight_grad_kernel)
extern "C" int wfs_fno_weight_grad(const float* g, const float* v, float* gW, float* gb, int C, int cin, long P,
                                   float* work, long work_elems, void* stream) {
  if (!g || !v || !gW || !gb || !work) { set_last_error("wfs_fno_weight_grad: null argument"); return WFS_ERR_INVALID; }
  if (C < 1 || C > 32 || cin < 1 || cin > 32 || P < 32 || P % 32) {
    set_last_error("wfs_fno_weight_grad: needs C, cin <= 32 and P a multiple of 32 (C=%d cin=%d P=%ld)", C, cin, P);
    return WFS_ERR_UNSUPPORTED;
  }
  if ((reinterpret_cast<unsigned long>(g) % 16) != 0 || (reinterpret_cast<unsigned long>(v) % 16) != 0) {
    set_last_error("wfs_fno_weight_grad: g and v must be 16-byte aligned");
    return WFS_ERR_INVALID;
  }
  // about 256 points per wavefront, at most two blocks per CU
  const long steps = P / 32;
  long blocks = (steps + 31) / 32;
  if (blocks > 512) blocks = 512;
  if (work_elems < blocks * kGradRecord) {
    set_last_error("wfs_fno_weight_grad: workspace needs %ld floats", blocks * kGradRecord);
    return WFS_ERR_INVALID;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(fno_weight_grad_kernel, dim3(unsigned(blocks)), dim3(256), 0, s, g, v, work, C, cin, P);
  WFS_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(fno_weight_grad_sum_kernel, dim3(33), dim3(512), 0, s, work, int(blocks), gW, gb, C, cin);
  WFS_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int wfs_fno_stage(const void* A, const float* in, float* out, int M, int K, int ncol, long slabs,
                             void* stream) {
  if (!A || !in || !out) { set_last_error("wfs_fno_stage: null argument"); return WFS_ERR_INVALID; }
  if (M < 1 || K < 1 || ncol < 1 || slabs < 1 || (M > 32 && K > 32) || M > 1 << 20 || K > 1 << 20) {
    set_last_error("wfs_fno_stage: needs M <= 32 or K <= 32 (M=%d K=%d ncol=%d slabs=%ld)", M, K, ncol, slabs);
    return WFS_ERR_UNSUPPORTED;
  }
  if (reinterpret_cast<unsigned long>(A) % 16) { set_last_error("wfs_fno_stage: A must be 16-byte aligned"); return WFS_ERR_INVALID; }
  const long cols = slabs * ncol;
  const long blocks = (cols + 31) / 32;
  if (blocks > 0x7fffffffL) { set_last_error("wfs_fno_stage: too many columns"); return WFS_ERR_INVALID; }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned short* a = static_cast<const unsigned short*>(A);
  if (M <= 32) {
    hipLaunchKernelGGL(fno_reduce_stage_kernel, dim3(unsigned(blocks)), dim3(256), 0, s, a, in, out, M, K, ncol, cols);
  } else {
    // few columns (the inverse x stage): the row tiles over several blocks as well
    const long tiles = (M + 31) / 32;
    const long share = (tiles + 3) / 4;
    const unsigned gy = unsigned(blocks < 512 ? share : 1);
    hipLaunchKernelGGL(fno_expand_stage_kernel, dim3(unsigned(blocks), gy), dim3(256), 0, s, a, in, out, M, K, ncol,
                       cols);
  }
  WFS_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int wfs_fno_modes_backward(const float* Rr, const float* Ri, const float* X, const float* dO, float* dX,
                                      float* gRr, float* gRi, int m3, int C, void* stream) {
  if (!Rr || !Ri || !X || !dO || !dX || !gRr || !gRi || m3 < 1 || C < 1 || C > 256) {
    set_last_error("wfs_fno_modes_backward: bad argument");
    return WFS_ERR_INVALID;
  }
  hipLaunchKernelGGL(fno_modes_backward_kernel, dim3(unsigned(m3)), dim3(256), 0, static_cast<hipStream_t>(stream), Rr,
                     Ri, X, dO, dX, gRr, gRi, m3, C);
  WFS_HIP_CHECK(hipGetLastError());
  return 0;
}

// The spectral path between the z stages, T -> Z, in one call: its five launches are 4 to 10 us each, and
// called one by one from Python they cost more host time than that (32^3, width 32, 12 modes, 4 layers:
// 246 -> 153 us a forward, 750 -> 470 a training sample with the gradients cleared in one launch).
extern "C" int wfs_fno_spectral(const void* F2, const void* G2, const float* Rr, const float* Ri, const float* T,
                                float* U, float* X, float* O, float* Y, float* Z, int n, int m, int C, void* stream) {
  const int m2 = m * m;
  if (int rc = wfs_fno_stage(F2, T, U, 2 * m, 2 * n, m, long(C) * n, stream)) return rc;
  if (int rc = wfs_fno_stage(F2, U, X, 2 * m, 2 * n, m2, C, stream)) return rc;
  if (int rc = wfs_fno_modes(Rr, Ri, X, O, m2 * m, C, stream)) return rc;
  if (int rc = wfs_fno_stage(G2, O, Y, 2 * n, 2 * m, m2, C, stream)) return rc;
  return wfs_fno_stage(G2, Y, Z, 2 * n, 2 * m, m, long(C) * n, stream);
}

// its transposition, Tg -> Zg (Zg may be Tg): G2t and F2t are the transposed tables
extern "C" int wfs_fno_spectral_backward(const void* G2t, const void* F2t, const float* Rr, const float* Ri,
                                         const float* X, const float* Tg, float* Y, float* O, float* dX, float* U,
                                         float* Zg, float* gRr, float* gRi, int n, int m, int C, void* stream) {
  const int m2 = m * m;
  if (int rc = wfs_fno_stage(G2t, Tg, Y, 2 * m, 2 * n, m, long(C) * n, stream)) return rc;
  if (int rc = wfs_fno_stage(G2t, Y, O, 2 * m, 2 * n, m2, C, stream)) return rc;
  if (int rc = wfs_fno_modes_backward(Rr, Ri, X, O, dX, gRr, gRi, m2 * m, C, stream)) return rc;
  if (int rc = wfs_fno_stage(F2t, dX, U, 2 * n, 2 * m, m2, C, stream)) return rc;
  return wfs_fno_stage(F2t, U, Zg, 2 * n, 2 * m, m, long(C) * n, stream);
}

template <int WM, int WN>
static void launch_tile(dim3 grid, hipStream_t s, const GemmArgs& g) {
  switch (g.flags & 3) {
    case 0: hipLaunchKernelGGL((gemm_bf16_kernel<WM, WN, false, false>), grid, dim3(64 * WM * WN), 0, s, g); break;
    case 1: hipLaunchKernelGGL((gemm_bf16_kernel<WM, WN, true, false>), grid, dim3(64 * WM * WN), 0, s, g); break;
    case 2: hipLaunchKernelGGL((gemm_bf16_kernel<WM, WN, false, true>), grid, dim3(64 * WM * WN), 0, s, g); break;
    default: hipLaunchKernelGGL((gemm_bf16_kernel<WM, WN, true, true>), grid, dim3(64 * WM * WN), 0, s, g); break;
  }
}

// dims = {batch, M, N, K}; strides = {sAb, sAm, sAk, sBb, sBk, sBn, sCb, sCm, sCn} (elements)
extern "C" int wfs_gemm_bf16(const float* A, const float* B, float* C, const long dims[4], const long strides[9],
                             float alpha, float beta, int flags, int splits, float* work, long work_elems,
                             const float* bias, float* act, void* stream) {
  if (!A || !B || !C || !dims || !strides) { set_last_error("wfs_gemm_bf16: null argument"); return WFS_ERR_INVALID; }
  GemmArgs g{};
  g.A = A; g.B = B; g.C = C; g.work = work;
  g.batch = int(dims[0]); g.M = dims[1]; g.N = dims[2]; g.K = dims[3];
  g.sAb = strides[0]; g.sAm = strides[1]; g.sAk = strides[2];
  g.sBb = strides[3]; g.sBk = strides[4]; g.sBn = strides[5];
  g.sCb = strides[6]; g.sCm = strides[7]; g.sCn = strides[8];
  g.alpha = alpha; g.beta = beta; g.flags = flags; g.bias = bias; g.act = act;
  if (flags & ~7) { set_last_error("wfs_gemm_bf16: unknown flags"); return WFS_ERR_INVALID; }
  if ((flags & 4) && !act) { set_last_error("wfs_gemm_bf16: WFS_GEMM_NO_C needs an activation output"); return WFS_ERR_INVALID; }
  if (g.batch < 1 || g.M < 1 || g.N < 1 || g.K < 1 || g.batch > 65535) { set_last_error("wfs_gemm_bf16: bad sizes"); return WFS_ERR_INVALID; }
  if (splits < 1) splits = 1;
  const long kblocks = (g.K + kBK - 1) / kBK;
  if (splits > kblocks) splits = int(kblocks);
  g.kchunk = ((kblocks + splits - 1) / splits) * kBK;
  splits = int((g.K + g.kchunk - 1) / g.kchunk);
  g.splits = splits;
  if (splits > 1 && (!work || work_elems < long(g.batch) * splits * g.M * g.N)) {
    set_last_error("wfs_gemm_bf16: split-K needs a workspace of batch*splits*M*N floats");
    return WFS_ERR_INVALID;
  }
  if (long(g.batch) * splits > 65535) { set_last_error("wfs_gemm_bf16: batch*splits too large"); return WFS_ERR_INVALID; }
  hipStream_t s = static_cast<hipStream_t>(stream);
  // tile shape by output shape: 32-row outputs use one wave row (32 x 128 tiles when wide, one
  // 32 x 32 wave when small and the k range per block is short), tall-skinny outputs and long-k
  // small outputs 128 x 32 (four waves share the staging), the rest 64 x 64
  int wm, wn;
  if (g.M <= 32 && g.N > 32) { wm = 1; wn = 4; }
  else if (g.M <= 32 && g.kchunk <= 256) { wm = 1; wn = 1; }
  else if (g.N <= 32) { wm = 4; wn = 1; }
  else { wm = 2; wn = 2; }
  const long gy = (g.M + 32 * wm - 1) / (32 * wm);
  const long gx = (g.N + 32 * wn - 1) / (32 * wn);
  if (gy > 65535 || gx > 0x7fffffffL) { set_last_error("wfs_gemm_bf16: output too large for the launch grid"); return WFS_ERR_INVALID; }
  dim3 grid(unsigned(gx), unsigned(gy), unsigned(g.batch * splits));
  if (wm == 1 && wn == 1) launch_tile<1, 1>(grid, s, g);
  else if (wm == 1) launch_tile<1, 4>(grid, s, g);
  else if (wm == 4) launch_tile<4, 1>(grid, s, g);
  else launch_tile<2, 2>(grid, s, g);
  WFS_HIP_CHECK(hipGetLastError());
  if (splits > 1) {
    const long total = long(g.batch) * g.M * g.N;
    const long blocks = (total + 3) / 4;
    if (blocks > 0x7fffffffL) { set_last_error("wfs_gemm_bf16: split-K output too large"); return WFS_ERR_INVALID; }
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3(unsigned(blocks)), dim3(256), 0, s, g);
    WFS_HIP_CHECK(hipGetLastError());
  }
  return 0;
}
