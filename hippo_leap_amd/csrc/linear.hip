// fp32 linear layer over the reference's column-major activations: the
// drop-in for gpuLinearCol (backends/naive.nim:3519-3547), which the forward
// pass calls for the Q/K/V projections in front of attention and the O
// projection behind it (naive.nim:4064-4066, 4079).
//
//   Y[M, T] = W[M, K] . X[K, T]
//
// W is row-major with K fastest (the GGUF weight as loaded, naive.nim:4091);
// X and Y keep the token index fastest (ggml column-major [dim, T]).
//
// * T == 1 (decode): linear_gemv_kernel reads W once from HBM with
//   non-temporal 16-byte loads, eight in flight per lane; the bound is HBM
//   bandwidth over M*K*4 bytes.  One wave per row (four per row when M is
//   small, so the grid still covers the chip), one cross-lane reduction per
//   row.  x is re-read from L2 by every wave (staging it in LDS measured
//   slower).
// * T > 1 (prefill): linear_split_kernel, six bf16 MFMAs
//   (v_mfma_f32_32x32x16_bf16) on the three bf16 parts of the fp32 operands
//   per fp32 product; fp32 MFMAs for the output tiles where that is not
//   possible.
//
// Accumulation is fp32 as in the reference; only the summation order
// differs (the reference's decode kernel reduces 256 strided partial sums,
// its prefill kernel sums k = 0..K-1 in order).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "launch.h"

namespace hl {
namespace {

__device__ inline float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// ---------------------------------------------------------------------------
// GEMV (T == 1)
// ---------------------------------------------------------------------------
// WPR waves share one row (each takes every WPR-th 16-byte chunk); the
// workgroup's 4 waves cover 4 / WPR rows.  VEC: K % 4 == 0 and 16-byte
// aligned w and x; otherwise one float per lane per step.
template <int WPR, bool VEC>
__global__ __launch_bounds__(256) void linear_gemv_kernel(const float* __restrict__ w,
                                                          const float* __restrict__ x,
                                                          float* __restrict__ y, int M, int K) {
  constexpr int RPW = 4 / WPR;
  constexpr int U = 8;  // 16-byte loads in flight per lane
  __shared__ float part[4];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int row = blockIdx.x * RPW + wave / WPR;
  const int share = wave % WPR;
  float acc = 0.f;
  if (row < M) {
    const float* wr = w + (size_t)row * K;
    if (VEC) {
      const f32x4* w4 = (const f32x4*)wr;
      const f32x4* x4 = (const f32x4*)x;
      const int K4 = K >> 2;
      constexpr int STEP = 64 * WPR;
      float s[4] = {0.f, 0.f, 0.f, 0.f};
      int k = lane + 64 * share;
      for (; k + (U - 1) * STEP < K4; k += U * STEP) {
        f32x4 wv[U], xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          wv[u] = __builtin_nontemporal_load(&w4[k + u * STEP]);  // W is read once
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = x4[k + u * STEP];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          s[u & 3] += wv[u].x * xv[u].x;
          s[u & 3] += wv[u].y * xv[u].y;
          s[u & 3] += wv[u].z * xv[u].z;
          s[u & 3] += wv[u].w * xv[u].w;
        }
      }
      for (; k < K4; k += STEP) {
        const f32x4 wv = __builtin_nontemporal_load(&w4[k]), xv = x4[k];
        s[0] += wv.x * xv.x;
        s[1] += wv.y * xv.y;
        s[2] += wv.z * xv.z;
        s[3] += wv.w * xv.w;
      }
      acc = (s[0] + s[1]) + (s[2] + s[3]);
    } else {
      for (int k = lane + 64 * share; k < K; k += 64 * WPR) acc += wr[k] * x[k];
    }
  }
  acc = wave_sum(acc);
  if (WPR == 1) {
    if (lane == 0 && row < M) y[row] = acc;
  } else {
    if (lane == 0) part[wave] = acc;
    __syncthreads();
    if (share == 0 && lane == 0 && row < M) {
      float t = 0.f;
#pragma unroll
      for (int i = 0; i < WPR; ++i) t += part[wave + i];
      y[row] = t;
    }
  }
}

// ---------------------------------------------------------------------------
// GEMM (T > 1) on bf16 MFMA over split fp32 operands
// ---------------------------------------------------------------------------
// Every operand x is the sum of three bf16 numbers, each the rounded rest of
// the one before: p0 = bf16(x), p1 = bf16(x - p0), p2 = x - p0 - p1.  bf16 has
// the exponents of fp32, so this needs no scale and holds all 24 bits of any
// element, however large its neighbours are.  A product is the six products of
// parts p0 p2', p2 p0', p1 p1', p0 p1', p1 p0', p0 p0'; the three left out are
// at most 2^-24 of it, the rounding of one fp32 product.  The matrix cores
// take bf16 subnormals, and give fp32 ones, as they are (test_small_parts).
//
// Bits below the smallest bf16 subnormal (of elements below 2^-109) are the
// only ones that the parts miss: the rests are collected, and a workgroup that
// has met one, or whose partial sums hold an inf or a NaN, computes its tile
// once more with fp32 MFMAs (body<false>), so that those come out as fp32
// arithmetic gives them.  Nothing else goes there: two f16 parts and a scale
// from a row's first elements (three products, 1.3 to 1.5 times as fast) lost
// elements 2^14 and more below those, and did every tile twice that met one
// 2^9 above them.
//
// Cost: 6 x 32 matrix-core cycles per 32x32x16 block where
// v_mfma_f32_32x32x2_f32 takes 8 x 64, and 6 VALU instructions per element
// and lane, spread part by part over the MFMAs of the blocks before (in bursts
// of a whole split: 14336 x 4096, 1000 columns 681 us, so 618).
// v_dot2_f32_bf16, which would halve the subtractions, took twice the time in
// all and did not subtract exactly.
//
// The small products have sums of their own: an MFMA cuts what lies below the
// last place of its largest addend towards minus infinity, so that small
// products (and a full fp32 sum added to larger products) shift every output
// the same way, by 1e-7 of their spread, which the layers of a model add up
// (Llama-3.2-1B, 16 layers, logits against 64 bits: 2.0e-6, now 7.7e-7; fp32
// MFMAs 2.1e-6).  Large
// products lose nothing in acc.  CROSS keeps accumulators of the small ones over
// all of K; the 64x64 tiles have no registers for those and sum a block's five
// small products of 16 k, which the VALU adds to acc behind the next block's
// MFMAs.  Error against a 64-bit product: 1.3e-7 at K = 2048, 1.4e-7 to 1.9e-7 at
// 4096, 3.7e-7 at 14336, where all six into one accumulator gave 2.5e-7, 3.5e-7
// to 5.0e-7 and 9.9e-7, and fp32 MFMAs in one chain of K 4.1e-7 at 2048 and
// 1.1e-6 at 4096.  The sums by VALU cost 7 to 10% (2048 x 8192, 301 columns: 82
// -> 91 us; added at the end of their own block: 97), CROSS 2%.
//
// The KW waves of a workgroup share one (32 WM) x (32 WN) output tile and
// split K between them in chunks of CK (wave w takes chunks w, w + KW, ...),
// each with its own staging area: no barrier until the partial sums meet in
// LDS.  W comes in rows of 4 CK bytes through LDS (16-byte pieces swizzled by
// the row, fp32; every wave splits what it reads itself); X goes straight to
// registers, XD 16-k steps ahead: lane ln of a half holds columns
// WN ln .. WN ln + WN - 1 of 8 k, so one load of 4 WN bytes serves the WN
// column blocks, and neither K nor T nor an address has to be a multiple of
// anything.
//
// A launch takes up to three matrices on the same X, a residual to add, or
// gate and up with SiLU * up on the sums: a prompt's layers then need four
// GEMM launches for ten kernels, tiles of small matrices share a round, and
// the sums of gate and up never go to memory.  Llama-3.2-1B shapes, 301
// tokens, a whole prefill, when this was done: 6.17 -> 5.46 ms (Q/K/V 51 -> 28
// us a layer, gate, up and SiLU 131 -> 105, the two additions 10 -> 0).
//
// What bounds it: bytes into the CUs on the small tiles (128 B per k of a
// 64x64 tile from L2; the prefetch depth did not matter), the matrix cores
// at six products on 64x128 tiles (1.1 PFLOP/s of bf16).  Before: fp32 MFMAs on
// 128x128 tiles staged through LDS, scalar loads whenever K or T was no
// multiple of 4.
//   M x K, T              before      now
//   4096 x 4096,    37    130 us     28     (32x32 tiles)
//   2048 x 2048,   301     76        28     (64x64)
//   2048 x 8192,   301    267        91     (64x64)
//   14336 x 4096, 1000   1080       650     (64x128: 181 TFLOP/s)
//   4096 x 4096,  4096   1044       728     (64x128: 189 TFLOP/s)
// (14336 x 4096, 1000, with a NaN in every tile, so that all are computed twice:
// 1530 us.  An element below 2^-109 does the same, however little the outputs
// feel it: telling takes the largest element too, one more VALU instruction a
// pair, 2 to 4% of every launch.)
// Measured and not kept: x loads four steps ahead (no change), 64-k chunks on
// 64x64 tiles (17% slower), sixteen waves (slower), 128x64 and 128x128 tiles;
// sums by VALU on 64x128 tiles (784 us instead of 650).

// N floats at a 4-byte aligned address.
template <int N>
struct FVec {
  typedef float T __attribute__((ext_vector_type(N), aligned(4)));
};
template <int N>
__device__ __forceinline__ void load_n(const float* p, float* v) {
  if constexpr (N == 1) {
    v[0] = *p;
  } else {
    const typename FVec<N>::T t = *(const typename FVec<N>::T*)p;
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  }
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// Two values rounded to bf16; through an empty asm, or the compiler would
// convert once more for each use of a half.
__device__ __forceinline__ uint32_t pack_bf16(float v0, float v1) {
  uint32_t r = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)v0, (__bf16)v1});
  asm("" : "+v"(r));
  return r;
}
// Parts 0 (largest) to 2 of eight values.
struct Split8 {
  u32x4 part[3];
};
__device__ __forceinline__ bf16x8 as_bf16(const u32x4& v) { return __builtin_bit_cast(bf16x8, v); }
// Part i of a pair of values, j of the eight; leaves what is below it in v.
// lost collects the bits that are in no part.
struct Pair {
  float v0, v1;
};
__device__ __forceinline__ void split_part(Pair& v, Split8& r, int j, int i, uint32_t& lost) {
  const uint32_t h = pack_bf16(v.v0, v.v1);
  r.part[i][j] = h;
  if (i < 2) {
    v.v0 -= __uint_as_float(h << 16);
    v.v1 -= __uint_as_float(h & 0xFFFF0000u);
  } else {
    // In asm, so that the collection is not put off (the rests of a whole
    // step would be live, which spills).
    asm("v_or3_b32 %0, %1, %2, %0" : "+v"(lost) : "v"(v.v0), "v"(v.v1));
  }
}
__device__ __forceinline__ Split8 split8(const float* v, uint32_t& lost) {
  Split8 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    Pair p = {v[2 * j], v[2 * j + 1]};
#pragma unroll
    for (int i = 0; i < 3; ++i) split_part(p, r, j, i, lost);
  }
  return r;
}
// The six products of parts that are kept, smallest first.
constexpr int kProducts = 6;
constexpr int kPartA[kProducts] = {0, 2, 1, 0, 1, 0}, kPartB[kProducts] = {2, 0, 1, 1, 0, 0};

// Orders a wave's LDS writes and reads (each wave has its own staging area).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct SplitArgs {
  const float* w[3];
  float* y[3];
  int rows[3];
  int tend[2];  // row tiles up to and including the first and second matrix
  const float* x;
  const float* res;  // added to y[0] (may be y[0]); null: none
  int K, T, tiles_m, tiles_n;
  int group_m;  // tiles are walked group_m row tiles at a time, row tiles fastest
};

// PAIR: w[0] and w[1] are gate and up, y[0] = silu(gate x) * (up x): each 32
// rows of a tile are 16 of gate and the same 16 of up, which meet in one lane
// of the final sums.  Otherwise the row tiles run over the matrices in order.
template <int WM, int WN, int KW, int CK, int XD, bool PAIR>
__global__ __launch_bounds__(64 * KW, WM * WN == 8 ? 1 : 2) void linear_split_kernel(SplitArgs p) {
  constexpr int ST = CK / 16;            // 16-k steps per chunk
  constexpr int BM = 32 * WM, BN = 32 * WN;
  constexpr int C16 = CK / 4;            // 16-byte pieces per staged row
  constexpr int NL = BM * CK / 4 / 64;   // 16-byte loads per lane and chunk
  constexpr int RPL = 64 / C16;          // rows per load
  constexpr int STAGE = BM * CK;         // floats of a wave's staging area
  constexpr int PART = BM * BN;          // floats of a wave's partial sums
  // The 64x64 tiles have 256 registers a wave: no accumulators for the small
  // products, and the next step's rows are split behind this one's MFMAs (a
  // second wave on the SIMD has MFMAs meanwhile; 2 to 3%).
  constexpr bool CROSS = WM * WN != 4, PIPE_A = CROSS;
  static_assert(XD <= ST && ST % XD == 0, "x buffers");
  __shared__ __attribute__((aligned(16))) float lds[KW * (STAGE > PART ? STAGE : PART)];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, hh = lane >> 5;

  // Each XCD (workgroup id mod 8) walks its own contiguous run of tiles, so
  // that its L2 serves the rows and columns its workgroups share.
  const int K = p.K, T = p.T;
  const int total = p.tiles_m * p.tiles_n, xcd = blockIdx.x % 8, rem = total % 8;
  const int id = xcd * (total / 8) + min(xcd, rem) + (int)blockIdx.x / 8;
  const int gi = id / (p.group_m * p.tiles_n), in = id - gi * (p.group_m * p.tiles_n);
  const int gm = min(p.group_m, p.tiles_m - gi * p.group_m);
  const int tm = gi * p.group_m + in % gm, n0 = (in / gm) * BN;
  const int mat = PAIR || tm < p.tend[0] ? 0 : tm < p.tend[1] ? 1 : 2;
  const int M = mat == 0 ? p.rows[0] : mat == 1 ? p.rows[1] : p.rows[2];
  const float* const w = mat == 0 ? p.w[0] : mat == 1 ? p.w[1] : p.w[2];
  float* const y = mat == 0 ? p.y[0] : mat == 1 ? p.y[1] : p.y[2];
  const float* const x = p.x;
  const int m0 = PAIR ? tm * (BM / 2) : (tm - (mat == 0 ? 0 : mat == 1 ? p.tend[0] : p.tend[1])) * BM;

  float* stage = lds + wave * STAGE;
  const int lrow = lane / C16, lp = lane % C16;
  // This lane's first column; the last lanes move back so that their WN
  // columns stay inside the row (and store only their own).
  const int nom = n0 + WN * ln, col0 = min(nom, T - WN);
  const float* const wt = w + (size_t)m0 * K;
  [[maybe_unused]] const float* const wt2 = PAIR ? p.w[1] + (size_t)m0 * K : nullptr;
  const int mlast = M - 1 - m0;  // rows past it read row mlast and store nothing
  // Tile row r: its matrix and its row there behind m0.
  auto wbase = [&](int r) { return PAIR && (r & 16) ? wt2 : wt; };
  auto wrow = [&](int r) { return min(PAIR ? 16 * (r >> 5) + (r & 15) : r, mlast); };
  // Offsets inside a tile: 32 bits hold those of all but the longest rows,
  // which get the smallest tile (linear_plan).
  typedef std::conditional_t<WM * WN == 1, size_t, uint32_t> Off;
  Off woff[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int r = RPL * i + lrow;
    woff[i] = (Off)wrow(r) * (Off)K + (Off)(4 * (lp ^ (r & (C16 - 1))));
  }
  const Off xoff = (Off)(8 * hh) * (Off)T + (Off)col0;
  const int nfull = K / CK;
  const int nmine = wave < nfull ? (nfull - wave + KW - 1) / KW : 0;  // full chunks of this wave
  const bool tail = K % CK != 0 && wave == nfull % KW;                 // the last, partial chunk

  f32x16 acc[WM][WN];

  // This wave's share of K into acc, on split operands or (false) on fp32
  // MFMAs.  Returns true when the parts do not hold every bit of a value.
  auto body = [&](auto split_tag) -> bool {
    constexpr bool SPLIT = decltype(split_tag)::value;
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
      for (int b = 0; b < WN; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;
    f32x4 wr[NL];
    float xr[XD][8][WN];
    [[maybe_unused]] uint32_t lost = 0;
    [[maybe_unused]] f32x16 cross[WM][WN], sums = {}, done;
    if constexpr (SPLIT && CROSS)
#pragma unroll
      for (int a = 0; a < WM; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b) cross[a][b] = f32x16{};
    auto load_w = [&](int c) {
      const float* src = wt + (size_t)c * CK;
      [[maybe_unused]] const float* src2 = PAIR ? wt2 + (size_t)c * CK : nullptr;
#pragma unroll
      for (int i = 0; i < NL; ++i) {  // RPL divides 16: one matrix per load
        const FVec<4>::T t = *(const FVec<4>::T*)((PAIR && (RPL * i & 16) ? src2 : src) + woff[i]);
        wr[i] = f32x4{t[0], t[1], t[2], t[3]};
      }
    };
    auto load_x = [&](int k0, float (*xv)[WN]) {
      const float* src = x + (size_t)k0 * T;
#pragma unroll
      for (int j = 0; j < 8; ++j) load_n<WN>(src + (size_t)j * T + xoff, xv[j]);
    };
    auto put_w = [&]() {
#pragma unroll
      for (int i = 0; i < NL; ++i) *(f32x4*)(stage + (RPL * i + lrow) * CK + 4 * lp) = wr[i];
      wave_lds_sync();
    };
    // k 16 s + 8 hh .. + 7 of staged row 32 a + ln
    auto read_a = [&](int a, int s, float* v) {
      const int r = 32 * a + ln, sw = r & (C16 - 1);
      const f32x4 v0 = *(const f32x4*)(stage + r * CK + 4 * ((4 * s + 2 * hh) ^ sw));
      const f32x4 v1 = *(const f32x4*)(stage + r * CK + 4 * ((4 * s + 2 * hh + 1) ^ sw));
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = v0[j], v[4 + j] = v1[j];
    };
    auto split_a = [&](int a, int s, Split8* A) {
      float v[8];
      read_a(a, s, v);
      A[a] = split8(v, lost);
    };
    auto split_b = [&](const float (*xv)[WN], int b) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = xv[j][b];
      return split8(v, lost);
    };
    // The products of 16 k of column block b, work(i) behind MFMA i.
    auto products = [&](const Split8* A, const Split8& B, int b, auto work) {
#pragma unroll
      for (int i = 0; i < kProducts * WM; ++i) {
        const int a = CROSS ? i % WM : i / kProducts, q = CROSS ? i / WM : i % kProducts;
        const bf16x8 pa = as_bf16(A[a].part[kPartA[q]]), pb = as_bf16(B.part[kPartB[q]]);
        const bool small = q < kProducts - 1;
        if (!CROSS && q == 0) done = sums;
        f32x16& c = !small ? acc[a][b] : CROSS ? cross[a][b] : sums;
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa, pb, !CROSS && q == 0 ? f32x16{} : c, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        work(i);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!CROSS) {
          const int at = (b * WM + a + WM * WN - 1) % (WM * WN);  // block that done belongs to
#pragma unroll
          for (int e = 16 * q / kProducts; e < 16 * (q + 1) / kProducts; ++e) acc[at % WM][at / WM][e] += done[e];
          asm volatile("" : "+v"(acc[at % WM][at / WM]));  // here, or the sums of all blocks would be live
        }
      }
    };
    // Step s on operands split before (A, B of column block 0); splits those
    // of the next step (its x in xn, its A if next_a) and of the other column
    // blocks between the MFMAs.  load_next overwrites xv once it is split.
    auto piped = [&](int s, const float (*xv)[WN], const float (*xn)[WN], Split8* A, Split8& B, bool next_a,
                     auto load_next) {
      constexpr int N = kProducts * WM;
      float va[8];
      Split8 A2[WM];
      Pair pa, pb;
      if (PIPE_A && next_a) read_a(0, s + 1, va);
#pragma unroll
      for (int b = 0; b < WN; ++b) {
        Split8 B2;
        const int nb = (b + 1) % WN;
        if (b == WN - 1) {
          __builtin_amdgcn_sched_barrier(0);
          load_next();
        }
        __builtin_amdgcn_sched_barrier(0);
        products(A, B, b, [&](int i) {
#pragma unroll
          for (int u = 12 * i / N; u < 12 * (i + 1) / N; ++u) {  // of the next column block
            const int j = u / 3, q = u % 3;
            const float(*src)[WN] = nb ? xv : xn;
            if (q == 0) pb = Pair{src[2 * j][nb], src[2 * j + 1][nb]};
            split_part(pb, B2, j, q, lost);
          }
          const int at = b * N + i;
          if (PIPE_A && next_a)
#pragma unroll
            for (int u = 12 * WM * at / (N * WN); u < 12 * WM * (at + 1) / (N * WN); ++u) {  // of the next step's A
              const int a = u / 12, j = u / 3 % 4, q = u % 3;
              if (q == 0) pa = Pair{va[2 * j], va[2 * j + 1]};
              split_part(pa, A2[a], j, q, lost);
              if (j == 3 && q == 2 && a + 1 < WM) read_a(a + 1, s + 1, va);
            }
        });
        B = B2;
      }
      if (next_a)
#pragma unroll
        for (int a = 0; a < WM; ++a) {
          if constexpr (PIPE_A) A[a] = A2[a];
          else split_a(a, s + 1, A);
        }
    };
    auto step = [&](int s, const float (*xv)[WN]) {
      if constexpr (SPLIT) {
        Split8 A[WM];
#pragma unroll
        for (int a = 0; a < WM; ++a) split_a(a, s, A);
#pragma unroll
        for (int b = 0; b < WN; ++b) products(A, split_b(xv, b), b, [](int) {});
      } else {
        // MFMA j pairs k 8 hh + j of the two lane halves
#pragma unroll
        for (int a = 0; a < WM; ++a) {
          float v[8];
          read_a(a, s, v);
#pragma unroll
          for (int b = 0; b < WN; ++b)
#pragma unroll
            for (int j = 0; j < 8; ++j)
              acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[j], xv[j][b], acc[a][b], 0, 0, 0);
        }
      }
    };
    if (nmine > 0) {
      // The loads are unconditional (the last ones repeat the last chunk and
      // are not used) and kept in program order, so that every wait counts
      // the loads behind it exactly.
      load_w(wave);
#pragma unroll
      for (int s = 0; s < XD; ++s) load_x(wave * CK + 16 * s, xr[s]);
      [[maybe_unused]] Split8 A[WM], B;
      for (int n = 0, c = wave; n < nmine; ++n, c += KW) {
        put_w();
        const int cn = min(c + KW, nfull - 1);
        __builtin_amdgcn_sched_barrier(0);
        load_w(cn);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SPLIT) {
          if (n == 0) B = split_b(xr[0], 0);
#pragma unroll
          for (int a = 0; a < WM; ++a) split_a(a, 0, A);
        }
#pragma unroll
        for (int s = 0; s < ST; ++s) {
          auto load_next = [&]() {
            load_x(s + XD < ST ? c * CK + 16 * (s + XD) : cn * CK + 16 * (s + XD - ST), xr[s % XD]);
          };
          if constexpr (SPLIT) {
            piped(s, xr[s % XD], xr[(s + 1) % XD], A, B, s + 1 < ST, load_next);
          } else {
            step(s, xr[s % XD]);
            __builtin_amdgcn_sched_barrier(0);
            load_next();
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (tail) {
      const int k0 = nfull * CK;
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int r = RPL * i + lrow, kk = k0 + 4 * (lp ^ (r & (C16 - 1)));
        const float* src = wbase(RPL * i) + (size_t)wrow(r) * K;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = src[min(kk + e, K - 1)];
          wr[i][e] = kk + e < K ? v : 0.f;
        }
      }
      wave_lds_sync();
      put_w();
      for (int s = 0; s < ST && k0 + 16 * s < K; ++s) {
        const int kb = k0 + 16 * s + 8 * hh;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          load_n<WN>(x + (size_t)min(kb + j, K - 1) * T + col0, xr[0][j]);
#pragma unroll
          for (int b = 0; b < WN; ++b) xr[0][j][b] = kb + j < K ? xr[0][j][b] : 0.f;
        }
        step(s, xr[0]);
      }
    }
    if constexpr (SPLIT && !CROSS) acc[WM - 1][WN - 1] += sums;
    if constexpr (SPLIT && CROSS)
#pragma unroll
      for (int a = 0; a < WM; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b) acc[a][b] += cross[a][b];
    return (lost & 0xFFFFu) != 0;
  };

  // The waves' partial sums meet in LDS ([wave][a][b][q][lane], four rows
  // each) and are added in wave order.  CHECK: if one is inf or NaN (or a
  // wave met bits outside its parts) nothing is stored and the result is false.
  auto finish = [&](auto check_tag, bool bad) -> bool {
    constexpr bool CHECK = decltype(check_tag)::value;
    // Units of four rows per lane: (a, q) of the tile, for PAIR q = 0, 1 (gate)
    // with q + 2 (up).
    constexpr int QN = PAIR ? 2 : 4, UPT = (WM * QN + KW - 1) / KW;  // units per wave
    __syncthreads();                                                 // the staging areas are free
    f32x4* part = (f32x4*)lds + wave * (PART / 4);
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
      for (int b = 0; b < WN; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          part[((a * WN + b) * 4 + q) * 64 + lane] =
              f32x4{acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
    __syncthreads();
    f32x4 sum[UPT][WN];
    float z = 0.f;
    auto added = [&](int a, int b, int q) {
      const f32x4* src = (const f32x4*)lds + ((a * WN + b) * 4 + q) * 64 + lane;
      f32x4 t = src[0];
#pragma unroll
      for (int k = 1; k < KW; ++k) t += src[k * (PART / 4)];
      if (CHECK) z += t.x * 0.f + t.y * 0.f + (t.z * 0.f + t.w * 0.f);
      return t;
    };
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const int aq = wave + KW * u;
      if (aq >= WM * QN) break;
#pragma unroll
      for (int b = 0; b < WN; ++b) {
        f32x4 t = added(aq / QN, b, aq % QN);
        if constexpr (PAIR) {
          const f32x4 up = added(aq / QN, b, aq % QN + 2);
#pragma unroll
          for (int e = 0; e < 4; ++e) t[e] = t[e] * (1.0f / (1.0f + expf(-t[e]))) * up[e];  // gpuSiluMul
        }
        sum[u][b] = t;
      }
    }
    if (CHECK && __syncthreads_or(bad || z != 0.f)) return false;
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const int aq = wave + KW * u;
      if (aq >= WM * QN) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + (PAIR ? 16 : 32) * (aq / QN) + 8 * (aq % QN) + 4 * hh + e;
        if (m >= M || nom >= T) continue;
        const size_t at = (size_t)m * T + col0;
        float* dst = y + at;
        if (WN > 1 && col0 == nom) {
          typedef typename FVec<WN == 1 ? 2 : WN>::T V;
          V v = {};
          if (p.res) v = *(const V*)(p.res + at);
#pragma unroll
          for (int b = 0; b < WN; ++b) v[b] = p.res ? v[b] + sum[u][b][e] : sum[u][b][e];
          *(V*)dst = v;
        } else {
#pragma unroll
          for (int b = 0; b < WN; ++b)
            if (col0 + b >= nom) dst[b] = p.res ? p.res[at + b] + sum[u][b][e] : sum[u][b][e];
        }
      }
    }
    return true;
  };
  const bool bad = body(std::true_type{});
  if (finish(std::true_type{}, bad)) return;
  body(std::false_type{});
  finish(std::false_type{}, false);
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

// The split GEMM's variants: tile, workgroups resident on a CU, and the model
// of their time by which one is chosen, in us:
//   2 + rounds of workgroups * (fixed + K / 1000 * (only round ? one : more)).
// Fitted to 200 timed shapes (4 .. 14336 rows, 2 .. 14336 k, 2 .. 4096 columns):
// the choice is 0.2% off the best of the four on average, 7% at worst; always
// taking one would cost 1.35 to 1.9 times as much on average.
struct SplitVariant {
  int bm, bn, per_cu;
  float fixed, one, more;
};
constexpr SplitVariant kSplit[] = {
    {32, 32, 1, 2.57f, 4.58f, 4.90f},    // 8 waves
    {64, 64, 1, 3.80f, 10.39f, 13.15f},  // 8 waves
    {64, 64, 2, 3.61f, 15.37f, 15.70f},  // 4 waves
    {64, 128, 1, 8.80f, 14.06f, 12.22f}, // 4 waves
};

LinearPlan linear_plan(const LinearCall& c) {
  LinearPlan p{};
  float best = 0.f;
  const int cus = cu_count();
  for (int v = 0; v < (int)(sizeof(kSplit) / sizeof(kSplit[0])); ++v) {
    const SplitVariant& s = kSplit[v];
    if (c.T < s.bn / 32) continue;  // a lane holds bn / 32 columns
    // Offsets of 32 bits inside a tile: 64 rows of K and 9 of T.
    if (v > 0 && (c.K > (1 << 26) || c.T > (1 << 28))) continue;
    const int bm = c.pair ? s.bm / 2 : s.bm;
    long long tm[3] = {0, 0, 0};
    for (int i = 0; i < (c.pair ? 1 : c.nmat); ++i) tm[i] = ((long long)c.rows[i] + bm - 1) / bm;
    const long long all = tm[0] + tm[1] + tm[2], tn = ((long long)c.T + s.bn - 1) / s.bn;
    if (all * tn > 0x7FFFFFFFLL) continue;
    const long long rounds = (all * tn + (long long)cus * s.per_cu - 1) / ((long long)cus * s.per_cu);
    float t = 2.f + (float)rounds * (s.fixed + (rounds > 1 ? s.more : s.one) * (float)c.K * 1e-3f);
    if (c.pair && s.bn == 128) t *= 1.1f;  // gate and up of 8192 x 2048, 301 columns: 159 us, on 64x64 tiles 155
    if (p.tiles_m == 0 || t < best) {
      best = t;
      p.variant = v;
      p.tiles_m = (int)all;
      p.tiles_n = (int)tn;
      p.tend[0] = (int)tm[0];
      p.tend[1] = (int)(tm[0] + tm[1]);
    }
  }
  return p;
}

template <int WM, int WN, int KW, int CK, int XD>
static void launch_split(const SplitArgs& a, bool pair, hipStream_t stream) {
  const dim3 grid((unsigned)a.tiles_m * (unsigned)a.tiles_n), block(64 * KW);
  if (pair) hipLaunchKernelGGL((linear_split_kernel<WM, WN, KW, CK, XD, true>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((linear_split_kernel<WM, WN, KW, CK, XD, false>), grid, block, 0, stream, a);
}

static thread_local long long g_linear_launches[HL_LK_KINDS];

void count_linear(int kernel) { ++g_linear_launches[kernel]; }

hipError_t linear_cols_launch(const LinearCall& c, hipStream_t stream) {
  const LinearPlan p = linear_plan(c);
  if (p.tiles_m == 0) return hipErrorInvalidValue;
  SplitArgs a{};
  for (int i = 0; i < c.nmat; ++i) {
    a.w[i] = c.w[i];
    a.y[i] = c.y[i];
    a.rows[i] = c.rows[i];
  }
  a.tend[0] = p.tend[0];
  a.tend[1] = p.tend[1];
  a.x = c.x;
  a.res = c.res;
  a.K = c.K;
  a.T = c.T;
  a.tiles_m = p.tiles_m;
  a.tiles_n = p.tiles_n;
  a.group_m = kSplit[p.variant].bn == 128 ? 4 : 8;
  if (p.variant == 0) launch_split<1, 1, 8, 64, 4>(a, c.pair, stream);
  else if (p.variant == 1) launch_split<2, 2, 8, 32, 2>(a, c.pair, stream);
  else if (p.variant == 2) launch_split<2, 2, 4, 32, 2>(a, c.pair, stream);
  else launch_split<2, 4, 4, 32, 2>(a, c.pair, stream);
  count_linear(HL_LK_SPLIT_32X32 + p.variant);
  return hipGetLastError();
}

hipError_t linear_col_launch(float* y, const float* x, const float* w, int K, int M, int T,
                             hipStream_t stream) {
  if (T > 1) return linear_cols_launch(LinearCall{1, {w}, {y}, {M}, x, nullptr, false, K, T}, stream);
  count_linear(HL_LK_GEMV);
  const bool vec = K % 4 == 0 && aligned16(w) && aligned16(x);
  const int wpr = M >= 2048 ? 1 : 4;
  const dim3 grid((M + 4 / wpr - 1) / (4 / wpr)), block(256);
  if (wpr == 1) {
    if (vec) hipLaunchKernelGGL((linear_gemv_kernel<1, true>), grid, block, 0, stream, w, x, y, M, K);
    else hipLaunchKernelGGL((linear_gemv_kernel<1, false>), grid, block, 0, stream, w, x, y, M, K);
  } else {
    if (vec) hipLaunchKernelGGL((linear_gemv_kernel<4, true>), grid, block, 0, stream, w, x, y, M, K);
    else hipLaunchKernelGGL((linear_gemv_kernel<4, false>), grid, block, 0, stream, w, x, y, M, K);
  }
  return hipGetLastError();
}

}  // namespace hl

extern "C" long long hl_linear_launches(int kernel) {
  return kernel >= 0 && kernel < HL_LK_KINDS ? hl::g_linear_launches[kernel] : 0;
}
