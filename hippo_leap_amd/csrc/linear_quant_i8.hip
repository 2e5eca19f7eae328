// Quantized decode GEMV on the int8 matrix cores: gpuLinearColQuant and its
// fused forms (backends/naive.nim:1580-1592, 1693-1708, 1799-1814, 1905-1920)
// for Q4_K, Q5_K, Q6_K and Q8_0 rows of whole 256-weight superblocks.
//
//   y[M] = dequant(W)[M, K] . x[K]
//
// x is held exactly to fixed point: the 256 values of a superblock become
// 32-bit integers X = rint(x 2^(30 - e)), e the exponent of the largest, and
// each X four signed 8-bit digits.  The weights' own integer quants are the
// other operand of v_mfma_i32_16x16x64_i8, so every product and every sum
// inside a scale group is exact (fp32 products of q and x round each); what
// is left in fp32 are the group's scale, its min and the sum over groups.
// Elements within 2^-6 of their superblock's largest keep all 24 bits; the
// absolute error of smaller ones is 2^-31 of the largest.
//
// MFMA operands: column n of B is row n of 16 weight rows, lane 16 g + n
// holds 16 consecutive quants ("run") of it; A's 16 rows are 4 digits for
// each of the 4 lane groups g, zero outside the group's own 16 k, so that
// C[4 g + t][n], the four results of lane 16 g + n, are the digit sums of
// that lane's own run: no value crosses lanes, runs of one scale group are
// chained through C, and each lane scales its own sums.
//
// A workgroup (NSB <= 16 waves) takes 16 rows at a time (8 gate and 8 up rows for
// the fused gate / up), a step being NSB superblocks of them: all threads
// load the rows' bytes (16 bytes each, contiguous along a row) three steps
// ahead into registers and put them into LDS (rows an odd number of 16-byte
// units apart, which spreads the 16 rows over the banks); wave w computes
// superblock w of every row.  One barrier per step.  Workgroups are
// persistent; a wave converts the x of its own superblocks once.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace hl {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Bytes per 256 weights, and the run of x (16 consecutive elements) that the
// lanes of group g take in MFMA m, as m and g of run r.
template <int QT>
struct QM;
template <>
struct QM<HL_GGML_Q4_K> {
  static constexpr int SB = 144;
  static constexpr bool MINS = true;
  static __device__ int pos(int r) { return 4 * (r & 3) + (r >> 2); }  // sub-blocks 2g, 2g + 1
};
template <>
struct QM<HL_GGML_Q5_K> {
  static constexpr int SB = 176;
  static constexpr bool MINS = true;
  static __device__ int pos(int r) { return 4 * (r & 3) + (r >> 2); }
};
template <>
struct QM<HL_GGML_Q6_K> {
  static constexpr int SB = 210;
  static constexpr bool MINS = false;
  static __device__ int pos(int r) { return 4 * ((r >> 1) & 3) + 2 * (r >> 3) + (r & 1); }  // r = 8n + 2m + h, g = 2n + h
};
template <>
struct QM<HL_GGML_Q8_0> {
  static constexpr int SB = 272;
  static constexpr bool MINS = false;
  static __device__ int pos(int r) { return 4 * (2 * (r >> 3) + (r & 1)) + ((r >> 1) & 3); }  // r = 8u + 2g + h, m = 2u + h
};

struct QmArgs {
  const uint8_t* w[3];
  float* y[3];
  int m[3];     // rows of each matrix
  int gend[3];  // row groups up to and including each matrix
  int ngroups, K;
  uint32_t magic;  // 2^24 / (16-byte units of a row in a step), rounded up
  const float* x;
  const float* res;  // NORM: x becomes rmsnorm(x + res) * nrm, x + res goes to xsum
  const float* nrm;
  float* xsum;
  float eps;
};

// 4 N bytes at a 2-byte aligned LDS address: the dwords that hold them,
// shifted (16-byte LDS reads off 16 bytes are far slower).
template <int N>
__device__ __forceinline__ void lds_dwords(const uint8_t* p, uint32_t* v) {
  const uint32_t ps = (uint32_t)(uintptr_t)p & 2u;
  const uint32_t* q = (const uint32_t*)(p - ps);
  uint32_t t[N + 1];
#pragma unroll
  for (int i = 0; i <= N; ++i) t[i] = q[i];
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = __builtin_amdgcn_alignbyte(t[i + 1], t[i], ps);
}
__device__ __forceinline__ u32x4 lds16(const uint8_t* p) {
  uint32_t v[4];
  lds_dwords<4>(p, v);
  return u32x4{v[0], v[1], v[2], v[3]};
}
__device__ __forceinline__ float lds_half(const uint8_t* p) { return f16_bits_to_f32(*(const uint16_t*)p); }

__device__ __forceinline__ i32x4 mfma_i8(u32x4 a, u32x4 b, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}
// The value of a run's digit sums.
__device__ __forceinline__ float digits_value(i32x4 c) {
  return fmaf((float)(c[2] + (c[3] << 8)), 65536.f, (float)(c[0] + (c[1] << 8)));
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kHalfMirror = 0x141, kMirror = 0x140;

// 6-bit scales and mins of sub-blocks 2g and 2g + 1 (getScaleMinK4,
// quant.nim:235-242), as in k4_pair of the direct kernel.
__device__ __forceinline__ void scale_min_pair(const u32x4& hdr, int g, float& sc0, float& sc1, float& mn0, float& mn1) {
  const uint32_t sh = 16 * (g & 1);
  const uint32_t Y = hdr.y >> sh, Z = hdr.z >> sh, W = hdr.w >> sh;
  const bool lo = g < 2;
  const uint32_t m1 = lo ? 0x3F3Fu : 0x0F0Fu, m2 = lo ? 0u : 0x3030u;
  const uint32_t SC = ((lo ? Y : W) & m1) | ((Y >> 2) & m2);
  const uint32_t MN = ((lo ? Z : (W >> 4)) & m1) | ((Z >> 2) & m2);
  sc0 = (float)(SC & 255u);
  sc1 = (float)((SC >> 8) & 255u);
  mn0 = (float)(MN & 255u);
  mn1 = (float)((MN >> 8) & 255u);
}

// Lane (g, n)'s share of one superblock of one row (bytes at p): the sum of
// its runs' scaled digit sums (times 2^(30 - e)), and the mins term.
template <int QT>
__device__ __forceinline__ void superblock(const uint8_t* p, int g, const u32x4* A, const float2& X, float& dot,
                                           float& mins) {
  const i32x4 zero = {0, 0, 0, 0};
  mins = 0.f;
  if constexpr (QT == HL_GGML_Q4_K || QT == HL_GGML_Q5_K) {
    const u32x4 hdr = *(const u32x4*)p;
    const uint8_t* qp = p + (QT == HL_GGML_Q4_K ? 16 : 48) + 32 * g;
    const u32x4 q0 = *(const u32x4*)qp, q1 = *(const u32x4*)(qp + 16);
    u32x4 b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      b[0][i] = q0[i] & 0x0F0F0F0Fu;
      b[1][i] = q1[i] & 0x0F0F0F0Fu;
      b[2][i] = (q0[i] >> 4) & 0x0F0F0F0Fu;
      b[3][i] = (q1[i] >> 4) & 0x0F0F0F0Fu;
    }
    if constexpr (QT == HL_GGML_Q5_K) {  // bits 2g and 2g + 1 of qh as bit 4
      const u32x4 h0 = *(const u32x4*)(p + 16), h1 = *(const u32x4*)(p + 32);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t s0 = h0[i] >> (2 * g), s1 = h1[i] >> (2 * g);
        b[0][i] |= (s0 & 0x01010101u) << 4;
        b[1][i] |= (s1 & 0x01010101u) << 4;
        b[2][i] |= (s0 & 0x02020202u) << 3;
        b[3][i] |= (s1 & 0x02020202u) << 3;
      }
    }
    const i32x4 c0 = mfma_i8(A[1], b[1], mfma_i8(A[0], b[0], zero));
    const i32x4 c1 = mfma_i8(A[3], b[3], mfma_i8(A[2], b[2], zero));
    float sc0, sc1, mn0, mn1;
    scale_min_pair(hdr, g, sc0, sc1, mn0, mn1);
    const float d = f16_bits_to_f32((uint16_t)(hdr.x & 0xFFFFu));
    const float dmin = f16_bits_to_f32((uint16_t)(hdr.x >> 16));
    dot = d * fmaf(sc0, digits_value(c0), sc1 * digits_value(c1));
    mins = dmin * fmaf(mn0, X.x, mn1 * X.y);
  } else if constexpr (QT == HL_GGML_Q6_K) {
    // Group g = 2n + h: elements 128n + 32m + 16h + 0..15 for m = 0..3.  The
    // 6-bit quants go to the top of their byte and flip its sign bit, which
    // makes them 4 (q - 32) as int8.
    const int n = g >> 1, h = g & 1;
    const u32x4 qa = lds16(p + 64 * n + 16 * h), qb = lds16(p + 64 * n + 32 + 16 * h);
    const u32x4 qh = lds16(p + 128 + 32 * n + 16 * h);
    const uint8_t* sp = p + 192 + 8 * n + h;  // scales of m = 0..3: two bytes apart
    u32x4 b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t hx = qh[i] ^ 0xAAAAAAAAu;
      b[0][i] = ((qa[i] << 2) & 0x3C3C3C3Cu) | ((hx << 6) & 0xC0C0C0C0u);
      b[1][i] = ((qb[i] << 2) & 0x3C3C3C3Cu) | ((hx << 4) & 0xC0C0C0C0u);
      b[2][i] = ((qa[i] >> 2) & 0x3C3C3C3Cu) | ((hx << 2) & 0xC0C0C0C0u);
      b[3][i] = ((qb[i] >> 2) & 0x3C3C3C3Cu) | (hx & 0xC0C0C0C0u);
    }
    const float d = 0.25f * lds_half(p + 208);
    float s = 0.f;
#pragma unroll
    for (int m = 0; m < 4; ++m)
      s = fmaf((float)(int8_t)sp[2 * m], digits_value(mfma_i8(A[m], b[m], zero)), s);
    dot = d * s;
  } else {  // Q8_0: blocks g and 4 + g of the eight
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint8_t* bp = p + 34 * (4 * u + g);
      uint32_t q[8];
      lds_dwords<8>(bp + 2, q);
      const i32x4 c = mfma_i8(A[2 * u + 1], u32x4{q[4], q[5], q[6], q[7]}, mfma_i8(A[2 * u], u32x4{q[0], q[1], q[2], q[3]}, zero));
      s = fmaf(lds_half(bp), digits_value(c), s);
    }
    dot = s;
  }
}

// NSB = blockDim / 64 superblocks per step, one per wave, MAX at most.  PAIR:
// w[0] and w[1] are gate and up, y[0] = silu(gate x) * (up x).  Otherwise the
// groups run over the matrices of the list in order.  XQ: superblocks of x
// per wave at most (1: K fits one step, and a wave keeps its x operands in
// registers).
template <int QT, int MAX, bool PAIR, bool NORM, int XQ>
__global__ __launch_bounds__(64 * MAX) void quant_i8_kernel(QmArgs a) {
  constexpr int SB = QM<QT>::SB;
  constexpr int NLD = (SB + 63) / 64;            // 16-byte units per thread and step: 16 NSB SB / 16 / (64 NSB)
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int NSB = (int)blockDim.x >> 6, NT = (int)blockDim.x;
  const int RU = NSB * SB / 16;                  // 16-byte units of a full step of one row
  const int STR = (RU | 1) * 16;                 // row pitch in LDS
  const int nb = a.K / 256, nseg = XQ == 1 ? 1 : (nb + NSB - 1) / NSB;
  uint8_t* stage = lds;                                        // [2][16 STR]
  uint8_t* dig = stage + 2 * 16 * STR;                         // [nseg NSB][16 runs][4 digits][16]
  float* xs = (float*)(dig + (size_t)nseg * NSB * 1024);       // [nseg NSB][8] sums of x per sub-block
  float2* xf = (float2*)(xs + nseg * NSB * 8);                 // [nseg NSB] 2^(e - 30) as two factors
  float* red = (float*)(xf + nseg * NSB);                      // [2][NSB][16]
  float* ssum = red + 2 * NSB * 16;                            // [NSB]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const uint32_t rowbytes = (uint32_t)nb * SB;

  // This thread's units of a step: row r of the 16, byte c of its segment.
  uint32_t ur[NLD], uc[NLD], ul[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const uint32_t u = (uint32_t)min(tid + NT * i, 16 * RU - 1);  // < 16 * 272
    ur[i] = (u * a.magic) >> 24;
    uc[i] = (u - ur[i] * (uint32_t)RU) * 16u;
    ul[i] = ur[i] * (uint32_t)STR + uc[i];
  }
  const int mine = ((int)a.ngroups - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;  // groups of this workgroup
  const int nsteps = mine * nseg;
  struct At {  // a step's group and segment
    int group, seg;
  };
  auto advance = [&](At& t) {
    if (++t.seg == nseg) {
      t.seg = 0;
      t.group += gridDim.x;
    }
  };
  // Matrix and first row of a group; the last group of a matrix moves back to
  // its last rows (computed twice, to the same bits).
  auto locate = [&](int group, int& mat, int& row0) {
    if constexpr (PAIR) {
      mat = 0;
      row0 = min(8 * group, a.m[0] - 8);
    } else {
      mat = group < a.gend[0] ? 0 : group < a.gend[1] ? 1 : 2;
      const int first = mat == 0 ? 0 : a.gend[mat - 1];
      row0 = min(16 * (group - first), a.m[mat] - 16);
    }
  };
  auto load = [&](const At& t, u32x4* r) {
    int mat, row0;
    locate(min(t.group, a.ngroups - 1), mat, row0);
    const uint32_t segbytes = (uint32_t)min(NSB, nb - t.seg * NSB) * SB;
    const size_t at = (size_t)row0 * rowbytes + (size_t)t.seg * (NSB * SB);
    const uint8_t* base = a.w[mat] + at;
    [[maybe_unused]] const uint8_t* base2 = PAIR ? a.w[1] + at : nullptr;
    typedef uint32_t V __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      // past a short last segment: its last bytes again, which nobody reads
      const uint32_t c = min(uc[i], segbytes - 16u);
      const uint8_t* src;
      if constexpr (PAIR) src = (ur[i] < 8u ? base : base2) + ((ur[i] & 7u) * rowbytes + c);
      else src = base + (ur[i] * rowbytes + c);
      const V v = __builtin_nontemporal_load((const V*)src);
      r[i] = u32x4{v[0], v[1], v[2], v[3]};
    }
  };

  // x (and the norm's inputs) first, then the first three steps' weights,
  // which stay in flight while x is converted.
  f32x4 xv[XQ];
  [[maybe_unused]] f32x4 rv[XQ], nv[XQ];
#pragma unroll
  for (int q = 0; q < XQ; ++q) {
    const int sb = wave + NSB * q;
    if (sb < nb) {
      const size_t o = (size_t)sb * 64 + lane;
      xv[q] = ((const f32x4*)a.x)[o];
      if constexpr (NORM) {
        rv[q] = ((const f32x4*)a.res)[o];
        nv[q] = ((const f32x4*)a.nrm)[o];
      }
    }
  }
  u32x4 ra[NLD], rb[NLD], rc[NLD];
  At ahead = {(int)blockIdx.x, 0};
  __builtin_amdgcn_sched_barrier(0);
  load(ahead, ra);
  advance(ahead);
  load(ahead, rb);
  advance(ahead);
  load(ahead, rc);
  advance(ahead);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
      const int sb = wave + NSB * q;
      if (sb < nb) {
        xv[q] += rv[q];
        if (blockIdx.x == 0) ((f32x4*)a.xsum)[(size_t)sb * 64 + lane] = xv[q];
        ss += (xv[q].x * xv[q].x + xv[q].y * xv[q].y) + (xv[q].z * xv[q].z + xv[q].w * xv[q].w);
      }
    }
    ss = wave_sum(ss);
    if (lane == 0) ssum[wave] = ss;
    __syncthreads();
    float t = 0.f;
    for (int i = 0; i < NSB; ++i) t += ssum[i];
    const float inv = 1.0f / sqrtf(t / (float)a.K + a.eps);
#pragma unroll
    for (int q = 0; q < XQ; ++q)
      if (wave + NSB * q < nb)
        xv[q] = f32x4{xv[q].x * inv * nv[q].x, xv[q].y * inv * nv[q].y, xv[q].z * inv * nv[q].z, xv[q].w * inv * nv[q].w};
  }
#pragma unroll
  for (int q = 0; q < XQ; ++q) {
    const int sb = wave + NSB * q;
    if (sb >= nb) break;
    const f32x4 v = xv[q];
    float am = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    float sum = (v.x + v.y) + (v.z + v.w);
    am = fmaxf(am, dpp<kXor1>(am));
    am = fmaxf(am, dpp<kXor2>(am));
    am = fmaxf(am, dpp<kHalfMirror>(am));
    am = fmaxf(am, dpp<kMirror>(am));
    am = fmaxf(am, __shfl_xor(am, 16, 64));
    am = fmaxf(am, __shfl_xor(am, 32, 64));
    if constexpr (QM<QT>::MINS) {
      sum += dpp<kXor1>(sum);
      sum += dpp<kXor2>(sum);
      sum += dpp<kHalfMirror>(sum);  // the sub-block's 8 lanes
      if ((lane & 7) == 0) xs[sb * 8 + (lane >> 3)] = sum;
    }
    // |x| < 2^e
    const int e = __builtin_amdgcn_frexp_expf(am);
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      d[i] = ((uint32_t)(int)rintf(ldexpf(v[i], 30 - e)) + 0x00808080u) ^ 0x00808080u;  // signed digits
    const uint32_t a0 = __builtin_amdgcn_perm(d[1], d[0], 0x05010400u), b0 = __builtin_amdgcn_perm(d[3], d[2], 0x05010400u);
    const uint32_t a1 = __builtin_amdgcn_perm(d[1], d[0], 0x07030602u), b1 = __builtin_amdgcn_perm(d[3], d[2], 0x07030602u);
    uint32_t* dst = (uint32_t*)(dig + (size_t)sb * 1024 + QM<QT>::pos(lane >> 2) * 64) + (lane & 3);
    dst[0] = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
    dst[4] = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
    dst[8] = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
    dst[12] = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
    // An inf or NaN in the superblock makes every row's result NaN.
    const float inf = __uint_as_float(kInfBits);
    const bool fin = !__any(!(fabsf(v.x) < inf && fabsf(v.y) < inf && fabsf(v.z) < inf && fabsf(v.w) < inf));
    if (lane == 0) {
      const int h = (e - 30) >> 1;
      xf[sb] = float2{fin ? ldexpf(1.0f, h) : __uint_as_float(0x7FC00000u), ldexpf(1.0f, e - 30 - h)};
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // This lane's A operands and factors of superblock sb (its wave's own).
  const bool own = (n >> 2) == g;
  u32x4 A[4];
  float2 X = {0.f, 0.f}, f = {0.f, 0.f};
  auto operands = [&](int sb) {
    const uint8_t* dp = dig + (size_t)sb * 1024 + g * 64 + (n & 3) * 16;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const u32x4 v = *(const u32x4*)(dp + 256 * m);
#pragma unroll
      for (int i = 0; i < 4; ++i) A[m][i] = own ? v[i] : 0u;
    }
    if constexpr (QM<QT>::MINS) X = *(const float2*)(xs + sb * 8 + 2 * g);
    f = xf[sb];
  };
  if (XQ == 1 && wave < nb) operands(wave);

  At now = {(int)blockIdx.x, 0};
  float acc = 0.f;
  int pending = -1;  // group whose sums wait in red
  auto finalize = [&](int buf) {
    if (tid < (PAIR ? 8 : 16)) {
      const float* rp = red + buf * NSB * 16 + tid;
      float s = 0.f, s2 = 0.f;
#pragma unroll 4
      for (int i = 0; i < NSB; ++i) {
        s += rp[16 * i];
        if (PAIR) s2 += rp[16 * i + 8];
      }
      int mat, row0;
      locate(pending, mat, row0);
      a.y[mat][row0 + tid] = PAIR ? s * (1.0f / (1.0f + expf(-s))) * s2 : s;  // gpuSiluMul
    }
  };
  auto step = [&](int k, u32x4* r) {
    uint8_t* buf = stage + (k & 1) * (16 * STR);
#pragma unroll
    for (int i = 0; i < NLD; ++i)
      if (64 * (i + 1) <= SB || tid + NT * i < 16 * RU) *(u32x4*)(buf + ul[i]) = r[i];
    __builtin_amdgcn_sched_barrier(0);
    load(ahead, r);  // past the last step: the last group again, not used
    __builtin_amdgcn_sched_barrier(0);
    advance(ahead);
    __syncthreads();
    if (pending >= 0) {
      finalize((k - 1) & 1);
      pending = -1;
    }
    const int sb = now.seg * NSB + wave;
    if (sb < nb) {
      if (XQ > 1) operands(sb);
      float dot, mins;
      superblock<QT>(buf + n * STR + wave * SB, g, A, X, dot, mins);
      acc += dot * f.x * f.y - mins;
    }
    if (now.seg == nseg - 1) {
      float s = acc + __shfl_xor(acc, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (lane < 16) red[(k & 1) * NSB * 16 + wave * 16 + n] = s;
      pending = now.group;
      acc = 0.f;
    }
    advance(now);
  };
  int k = 0;
  for (; k + 2 < nsteps; k += 3) {
    step(k, ra);
    step(k + 1, rb);
    step(k + 2, rc);
  }
  if (k < nsteps) step(k, ra);
  if (k + 1 < nsteps) step(k + 1, rb);
  __syncthreads();
  finalize((nsteps - 1) & 1);
}

constexpr int kMaxLds = 160 * 1024;

template <int QT>
size_t lds_bytes(int nb, int nsb) {
  const int RU = nsb * QM<QT>::SB / 16, nseg = (nb + nsb - 1) / nsb;
  return (size_t)2 * 16 * (RU | 1) * 16 + (size_t)nseg * nsb * (1024 + 32 + 8) + 2 * nsb * 16 * 4 + nsb * 4;
}

template <int QT, int MAX, bool PAIR, bool NORM, int XQ>
bool launch(QmArgs a, int nsb, hipStream_t stream) {
  const size_t shm = lds_bytes<QT>(a.K / 256, nsb);
  // Set once per instantiation: without it 64 KiB is the limit.
  static const hipError_t attr = hipFuncSetAttribute((const void*)quant_i8_kernel<QT, MAX, PAIR, NORM, XQ>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
  if (shm > (size_t)kMaxLds || (attr != hipSuccess && shm > 64 * 1024)) {
    (void)hipGetLastError();  // the failed attribute call's error is not this launch's
    return false;
  }
  const uint32_t ru = (uint32_t)(nsb * QM<QT>::SB / 16);
  a.magic = ((1u << 24) + ru - 1) / ru;
  const int slots = std::max(1, std::min<int>(16 / nsb, (int)(kMaxLds / shm))) * cu_count();
  // Every workgroup takes whole groups: a last round that is mostly empty
  // costs as much as a full one, and the direct kernels are then faster
  // (2x 2304 x 14336 Q4_K, 288 groups on 256 CUs: 12.7 us against 15.2; 5632 x
  // 6912, 352 groups: 9.5 against 10.5; 6400 x 2816 twice, 800 groups: 9.6
  // against 8.3).  Not asked where the norm is folded in: that saves a launch.
  const int rounds = (a.ngroups + slots - 1) / slots;
  constexpr float full = QT == HL_GGML_Q5_K || QT == HL_GGML_Q8_0 ? 0.6f : XQ == 1 ? 0.75f : 0.9f;
  if (!NORM && (float)a.ngroups < full * (float)rounds * (float)slots) return false;
  const int grid = std::min(a.ngroups, slots);
  hipLaunchKernelGGL((quant_i8_kernel<QT, MAX, PAIR, NORM, XQ>), dim3(grid), dim3(64 * nsb), shm, stream, a);
  count_linear(NORM ? HL_LK_I8_NORM : HL_LK_I8);
  return true;
}

template <int QT, int MAX, int XQ>
bool launch_forms(const QmArgs& a, bool pair, int nsb, hipStream_t stream) {
  if (a.res) return pair ? launch<QT, MAX, true, true, XQ>(a, nsb, stream) : launch<QT, MAX, false, true, XQ>(a, nsb, stream);
  return pair ? launch<QT, MAX, true, false, XQ>(a, nsb, stream) : launch<QT, MAX, false, false, XQ>(a, nsb, stream);
}

// K goes to steps of 16 superblocks and a rest, or to as many equal steps
// where that rest would be less than half (K = 8704: 12, 12 and 10
// superblocks, not 16, 16 and 2: 4096 x 8704 Q4_K 10.6 -> 9.1 us; but 4096 x
// 14336 in 16, 16, 16 and 8 10.8, in four times 14 11.5).  Eight waves for
// K <= 2048, which has no work for more, where LDS does not hold two stages of
// 16 superblocks and the digits of x, and for Q8_0, whose superblocks are too
// large.  Q6_K: multiples of eight superblocks (210 bytes each) are whole
// 16-byte units.
template <int QT>
bool launch_type(const QmArgs& a, bool pair, hipStream_t stream) {
  const int nb = a.K / 256;
  auto even = [&](int most) {
    const int nseg = (nb + most - 1) / most, nsb = nb % most >= most / 2 || nb % most == 0 ? most : (nb + nseg - 1) / nseg;
    return QT == HL_GGML_Q6_K ? (nsb + 7) / 8 * 8 : nsb;
  };
  if (nb <= 8) return launch_forms<QT, 8, 1>(a, pair, nb, stream);
  if constexpr (QT != HL_GGML_Q8_0) {
    if (nb <= 16) return launch_forms<QT, 16, 1>(a, pair, nb, stream);
    if (lds_bytes<QT>(nb, even(16)) <= (size_t)kMaxLds) return launch_forms<QT, 16, 4>(a, pair, even(16), stream);
  }
  if (a.res) return nb <= 32 ? launch_forms<QT, 8, 4>(a, pair, even(8), stream) : false;  // the norm's inputs fill the registers
  return launch_forms<QT, 8, 8>(a, pair, even(8), stream);
}

}  // namespace

bool linear_quant_i8_launch(const QuantI8Call& c, hipStream_t stream) {
  const int nb = c.K / 256;
  if (c.nmat < 1 || c.nmat > 3 || c.K % 256 || nb < 8 || nb > 64 || ((uintptr_t)c.x & 15)) return false;
  if (c.qtype == HL_GGML_Q6_K && nb % 8) return false;  // 210-byte superblocks: 16-byte units of whole rows
  if (c.res && (((uintptr_t)c.res | (uintptr_t)c.nrm | (uintptr_t)c.xsum) & 15)) return false;
  QmArgs a{};
  int groups = 0;
  for (int i = 0; i < c.nmat; ++i) {
    if (((uintptr_t)c.w[i] & 15) || c.rows[i] < (c.pair ? 8 : 16)) return false;
    a.w[i] = (const uint8_t*)c.w[i];
    a.y[i] = c.y[i];
    a.m[i] = c.rows[i];
    groups += (c.rows[i] + 15) / 16;
    a.gend[i] = groups;
  }
  for (int i = c.nmat; i < 3; ++i) a.gend[i] = groups;
  a.ngroups = c.pair ? (c.rows[0] + 7) / 8 : groups;
  a.K = c.K;
  a.x = c.x;
  a.res = c.res;
  a.nrm = c.nrm;
  a.xsum = c.xsum;
  a.eps = c.eps;
  switch (c.qtype) {
    case HL_GGML_Q4_K: return launch_type<HL_GGML_Q4_K>(a, c.pair, stream);
    case HL_GGML_Q5_K: return launch_type<HL_GGML_Q5_K>(a, c.pair, stream);
    case HL_GGML_Q6_K: return launch_type<HL_GGML_Q6_K>(a, c.pair, stream);
    case HL_GGML_Q8_0: return launch_type<HL_GGML_Q8_0>(a, c.pair, stream);
    default: return false;
  }
}

}  // namespace hl
