// Device building blocks shared by the MTE and adjoint kernels: the MFMA
// traits (operand and accumulator lane layouts of the two matrix
// instructions used), the k-permuted LDS layout, the packed B-operand order,
// the growth law and the per-year product loop.
#ifndef ROADMC_MTE_COMMON_H
#define ROADMC_MTE_COMMON_H

#include <hip/hip_runtime.h>

#include <type_traits>

#include "mte_kernels.h"
#include "rng.h"

namespace roadmc {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef double doublex2 __attribute__((ext_vector_type(2)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

enum { kLawLognormal = 0, kLawRefCpu = 1, kLawRefGpu = 2 };
enum { kEndPost = 0, kEndPre = 1 };

// v_mfma_f32_32x32x2_f32: A lane l = A[l%32][l/32]; B lane l = B[l/32][l%32];
// D item r of lane l = D[8(r/4) + 4(l/32) + r%4][l%32].
struct TraitsF32 {
  using T = float;
  using VecT = floatx4;
  using AccT = floatx16;
  static constexpr int TM = 32, TN = 32, KV = 4, NACC = 16, NT = 4, PAD = 4;
  static constexpr bool kQuadItems = true;  // items 4q..4q+3 are 4 paths
  static constexpr bool kSplit = false;
  __device__ static AccT mfma(float a, float b, AccT c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
  __device__ static int acc_row(int lane, int r) {
    return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
  }
  __device__ static int acc_col(int lane) { return lane & 31; }
  __device__ static int a_row(int lane) { return lane & 31; }
  __device__ static int k_lane(int lane) { return lane >> 5; }
  // k = 8g + 2s + h  ->  8g + 4h + s
  __host__ __device__ static int perm(int k) {
    return (k & ~7) | ((k & 1) << 2) | ((k >> 1) & 3);
  }
  __device__ static float expo(float x) { return __expf(x); }
  __device__ static void normal4(uint32_t q, uint32_t y, uint32_t p,
                                 uint32_t tag, uint32_t k0, uint32_t k1,
                                 float z[4]) {
    rmc_normal4_f(q, y, p, tag, k0, k1, z);
  }
};

// v_mfma_f64_16x16x4_f64: A lane l = A[l%16][l/16]; B lane l = B[l/16][l%16];
// D item r of lane l = D[l/16 + 4r][l%16].
struct TraitsF64 {
  using T = double;
  using VecT = doublex2;
  using AccT = doublex4;
  static constexpr int TM = 16, TN = 16, KV = 2, NACC = 4, NT = 8, PAD = 2;
  static constexpr bool kQuadItems = false;
  static constexpr bool kSplit = false;
  __device__ static AccT mfma(double a, double b, AccT c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int acc_row(int lane, int r) { return (lane >> 4) + 4 * r; }
  __device__ static int acc_col(int lane) { return lane & 15; }
  __device__ static int a_row(int lane) { return lane & 15; }
  __device__ static int k_lane(int lane) { return lane >> 4; }
  // k = 8g + 4s + h  ->  8g + 2h + s
  __host__ __device__ static int perm(int k) {
    return (k & ~7) | ((k & 3) << 1) | ((k >> 2) & 1);
  }
  __device__ static double expo(double x) { return exp(x); }
  __device__ static void normal4(uint32_t q, uint32_t y, uint32_t p,
                                 uint32_t tag, uint32_t k0, uint32_t k1,
                                 double z[4]) {
    rmc_normal4_d(q, y, p, tag, k0, k1, z);
  }
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Split-bf16 products on v_mfma_f32_32x32x16_bf16 (FP32 accumulate).  A value
// x is held as the pair hi = bf16(x), lo = bf16(x - hi), which carries about
// 17 significant bits; a product x.m is hi.m_hi + hi.m_lo + lo.m_hi (the
// dropped lo.m_lo is below 2^-16 of it).  The population tile lives in LDS as
// two bf16 arrays (hi, then lo), k in natural order; a lane's operand is the
// 8 consecutive k of its row and lane half: A lane l = A[l%32][8(l/32) + i],
// B lane l = B[8(l/32) + i][l%32], i = 0..7 (one 16-byte vector).  The
// accumulator layout is the one of v_mfma_f32_32x32x2_f32.
struct TraitsB3 {
  using T = float;
  using VecT = floatx4;  // 16 bytes: 8 bf16 operands
  using AccT = floatx16;
  // Each bf16 row has Pp + PAD slots (16 bytes of padding), so the hi and lo
  // arrays together take BM (Pp + PAD) 4-byte units, as lds_bytes_t counts.
  static constexpr int TM = 32, TN = 32, KV = 1, NACC = 16, NT = 4, PAD = 8;
  static constexpr bool kQuadItems = true;
  static constexpr bool kSplit = true;
  __device__ static AccT mfma(floatx4 a, floatx4 b, AccT c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                    __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  __device__ static int acc_row(int lane, int r) {
    return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
  }
  __device__ static int acc_col(int lane) { return lane & 31; }
  __device__ static int a_row(int lane) { return lane & 31; }
  __device__ static int k_lane(int lane) { return lane >> 5; }
  __host__ __device__ static int perm(int k) { return k; }
  __device__ static float expo(float x) { return __expf(x); }
  __device__ static void normal4(uint32_t q, uint32_t y, uint32_t p,
                                 uint32_t tag, uint32_t k0, uint32_t k1,
                                 float z[4]) {
    rmc_normal4_f(q, y, p, tag, k0, k1, z);
  }
  // The split pair of x, hi in the low half.
  __device__ static uint32_t split(float x) {
    const __bf16 h = (__bf16)x;
    const __bf16 l = (__bf16)(x - (float)h);
    return (uint32_t)__builtin_bit_cast(uint16_t, h) |
           ((uint32_t)__builtin_bit_cast(uint16_t, l) << 16);
  }
};

// FP32 products on v_mfma_f32_32x32x16_bf16.  An FP32 value is exactly the sum
// of three bf16 terms x = h + m + l (each the rounding of what is left; down to
// 2^-110, below which l underflows), and a
// product x.y is taken as the six of the nine term products that reach 2^-24
// of it: h.h' in one FP32 accumulator, l.h' + h.l' + m.m' + m.h' + h.m' in a
// second one, added to the first at the end.  The dropped m.l', l.m' and l.l'
// are below 2^-25 of the product each, of either sign.
// Why two accumulators: the matrix cores add 8 products at a time (their sum
// aligned to the largest one's exponent - 24) to the accumulator and round to
// nearest, but cut the sum to 2^-8 of the accumulator's last place, downwards.
// In one accumulator, twelve such cuts per 16 products lower every sum by
// 2e-8 of it at 256 terms, each year alike; in two the bias is below 1e-9 and
// the rms error of a dot product over landscape rows is less than half that
// of v_mfma_f32_32x32x2_f32 (5.1e-8 against 1.2e-7 at 64 terms, 9.1e-8
// against 2.3e-7 at 256, 1.8e-7 against 4.8e-7 at 1024).
// The matrix cores run the six at 1.8 PFLOP/s (random operands), 305 TFLOP/s
// of FP32 products against 155 for the FP32 MFMA, and leave the VALU to the
// other waves of the SIMD, which the FP32 MFMA does not.
// The population tile stays FP32 in LDS, k in natural order, and is split as
// it is read (28 VALU operations per 8 values); the movement matrix is split
// once when it is packed.  Operand and accumulator lane layouts are those of
// TraitsB3.
// The tile of a job with little noise (MteJob::scaled) holds a path's
// populations times its row's scale, one of 32 in (0.5, 1].  The sums of h.h'
// depend on the populations' first 8 bits only, so that paths closer to each
// other than that would round alike in every sum, and their mean would keep one
// path's error: 7e-8 of a patch's mean at 512 patches under REF_CPU, where the
// FP32 MFMA's larger errors average to 2e-8.  Scaled, paths have different first
// bits whatever the noise (1.3e-8).  The product and the growth factor commute
// with the scale; only the level in the growth law takes its inverse, one
// multiplication per value and year.
struct TraitsX6 {
  using T = float;
  using VecT = floatx4;
  using AccT = floatx16;
  static constexpr int TM = 32, TN = 32, KV = 8, NACC = 16, NT = 4, PAD = 4;
  static constexpr bool kQuadItems = true;
  static constexpr bool kSplit = false;
  __device__ static AccT mfma(floatx4 a, floatx4 b, AccT c) { return TraitsB3::mfma(a, b, c); }
  // Inverse scale of a row, the product of the factors of its accumulator item
  // r and of its lane half, row = acc_row(lane, r).  Exact short numbers: one
  // that rounds would move the level of every patch of a row alike (5e-10 of
  // the mean total a year).
  __host__ __device__ static constexpr float unscale(int row) {
    return (float)((32 + 2 * ((row >> 1 & 12) | (row & 3))) * (32 + (row >> 2 & 1))) / 1024.f;
  }
  __device__ static constexpr float unscale_item(int r) { return (float)(32 + 2 * r) / 32.f; }
  __device__ static float unscale_half(int lane) { return lane < 32 ? 1.f : 33.f / 32.f; }
  __device__ static int acc_row(int lane, int r) {
    return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
  }
  __device__ static int acc_col(int lane) { return lane & 31; }
  __device__ static int a_row(int lane) { return lane & 31; }
  __device__ static int k_lane(int lane) { return lane >> 5; }
  __host__ __device__ static int perm(int k) { return k; }
  __device__ static float expo(float x) { return __expf(x); }
  __device__ static void normal4(uint32_t q, uint32_t y, uint32_t p,
                                 uint32_t tag, uint32_t k0, uint32_t k1,
                                 float z[4]) {
    rmc_normal4_f(q, y, p, tag, k0, k1, z);
  }
};

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// The three bf16 terms of a pair of FP32 values, packed (first value in the
// low half), each the rounding to nearest of what the ones before leave, so
// that m and l have either sign and h + m + l is the value.  x - h is one v_dot2_f32_bf16 of the
// packed pair with (-1, 0) or (0, -1), exact because the difference is
// representable; the constants stay in scalar registers (as inline constants
// they would read as a 32-bit -1.0).
__device__ __forceinline__ void split3_pair(float x0, float x1, uint32_t& h, uint32_t& m,
                                            uint32_t& l) {
  uint32_t c0 = 0x0000bf80u, c1 = 0xbf800000u;
  asm("" : "+s"(c0), "+s"(c1));
  const bf16x2 n0 = __builtin_bit_cast(bf16x2, c0), n1 = __builtin_bit_cast(bf16x2, c1);
  auto pack = [](float a, float b) -> uint32_t {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){a, b}, bf16x2));
  };
  auto minus = [](uint32_t pk, bf16x2 which, float x) -> float {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pk), which, x, false);
  };
  h = pack(x0, x1);
  const float r0 = minus(h, n0, x0), r1 = minus(h, n1, x1);
  m = pack(r0, r1);
  l = pack(minus(m, n0, r0), minus(m, n1, r1));
}

// The split operands of 8 consecutive FP32 values.
struct Split8 {
  floatx4 h, m, l;
};
__device__ __forceinline__ Split8 split3_8(const floatx4 x0, const floatx4 x1) {
  uint32_t h[4], m[4], l[4];
  split3_pair(x0[0], x0[1], h[0], m[0], l[0]);
  split3_pair(x0[2], x0[3], h[1], m[1], l[1]);
  split3_pair(x1[0], x1[1], h[2], m[2], l[2]);
  split3_pair(x1[2], x1[3], h[3], m[3], l[3]);
  typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));
  Split8 s;
  s.h = __builtin_bit_cast(floatx4, (uint32x4){h[0], h[1], h[2], h[3]});
  s.m = __builtin_bit_cast(floatx4, (uint32x4){m[0], m[1], m[2], m[3]});
  s.l = __builtin_bit_cast(floatx4, (uint32x4){l[0], l[1], l[2], l[3]});
  return s;
}

__host__ __device__ static inline size_t align16(size_t x) {
  return (x + 15) & ~(size_t)15;
}

// LDS of one MTE workgroup: the BM x (Pp + PAD) population tile, the per-row
// growth-rate means, 8 x 4 doubles for the tally reduction and, when
// remainder tiles are split into k-quarters, 4 partial accumulators per
// remainder tile.
template <class TR>
__host__ __device__ static inline size_t lds_bytes_t(int BM, int Pp, int n_rem_split) {
  using T = typename TR::T;
  return align16((size_t)BM * (Pp + TR::PAD) * sizeof(T)) +
         align16((size_t)BM * sizeof(T)) + 8 * 4 * sizeof(double) +
         (size_t)n_rem_split * 4 * TR::NACC * 64 * sizeof(T);
}

// n' = level grown by a year, times x / level.
template <typename T, int LAW>
__device__ __forceinline__ T grow(T x, T level, T z, T K, T Kinv, T r, T sig,
                                  T half_var, T dt, T mu, T sd, T grm, T lv) {
  if constexpr (LAW == kLawRefCpu) {
    const T g = dt * (mu + sd * z) * (T)0.01;
    return x * ((T)1 + g * (K - level) * Kinv);
  }
  if constexpr (LAW == kLawRefGpu) {
    const T g = lv * z * grm + grm;
    return x * ((T)1 + g * (K - level) * Kinv);
  }
  T e;
  if constexpr (sizeof(T) == 4)
    // sig and half_var arrive pre-scaled by log2(e): one FMA and v_exp_f32.
    e = __builtin_amdgcn_exp2f(fmaf(sig, z, -half_var));
  else
    e = exp(sig * z - half_var);
  return x * ((T)1 + r * ((T)1 - level * Kinv)) * e;
}

template <typename T>
__device__ __forceinline__ void path_scalars(uint32_t path, uint32_t year,
                                             uint32_t tag, uint32_t k0,
                                             uint32_t k1, T* zb, T* zj,
                                             T* uj) {
  const rmc_u4 x = rmc_philox(path, year, 0u, tag, k0, k1);
  if constexpr (sizeof(T) == 4) {
    rmc_box_muller_f(rmc_u01f(x.x), rmc_u01f(x.y), zb, zj);
    *uj = rmc_u01f(x.z);
  } else {
    rmc_box_muller_d(rmc_u01d(x.x), rmc_u01d(x.y), zb, zj);
    *uj = rmc_u01d(x.z);
  }
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Global-address-space view of a device pointer, so that loads compile to
// global_load (not flat_load).
template <typename V>
__device__ __forceinline__ const __attribute__((address_space(1))) V* as_global(const V* p) {
  return (const __attribute__((address_space(1))) V*)(p);
}

// Movement matrix of one job in MFMA B-operand order, read through a buffer
// resource: the k-group step goes into the scalar offset and the tile's
// column block into a 32-bit vector offset, so operand loads need no vector
// address arithmetic.  Reads past `bytes` return zero instead of faulting.
struct PackedB {
  __amdgpu_buffer_rsrc_t rsrc;
  int nkg;  // k-groups per column block
};

__device__ __forceinline__ PackedB packed_b(const void* p, int nkg, size_t bytes) {
  PackedB b;
  // Word 3 of the descriptor: raw 32-bit data format of the gfx9 family.
  b.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
  b.nkg = nkg;
  return b;
}

// Byte offset of lane `lane`'s 16-byte operand in column block `tcol`.
__device__ __forceinline__ uint32_t b_voff(const PackedB& B, int tcol, int lane) {
  return ((uint32_t)tcol * (uint32_t)B.nkg * 64u + (uint32_t)lane) * 16u;
}

template <class VecT>
__device__ __forceinline__ VecT load_b(const PackedB& B, uint32_t voff, int kg) {
  static_assert(sizeof(VecT) == 16, "B operands are 16-byte vectors");
  return __builtin_bit_cast(
      VecT, __builtin_amdgcn_raw_buffer_load_b128(B.rsrc, (int)voff, kg * 64 * 16, 0));
}

// One year's product for the NTILE output tiles of a wave:
// acc[t] = A[rows of tile t, :] . M[:, cols of tile t].
// Two register stages ping-pong over the k-groups (the k-group count B.nkg is
// even): the B operands and LDS A operands of k-group kg+1 are in flight while
// the MFMAs of k-group kg run.
// On entry b0 holds the B operands of k-group 0; on exit it holds them again
// (the last stage-0 load re-fetches k-group 0, which the next year starts
// with, so that load's latency is hidden behind the epilogue).
template <class TR, int NTILE, bool SHARED_A = false>
__device__ __forceinline__ void year_product(typename TR::AccT* acc,
                                             typename TR::VecT* b0,
                                             const PackedB& B,
                                             const typename TR::T* A,
                                             const int* trow, const int* tcol,
                                             int LDA, int arow, int akoff, int lane) {
  using T = typename TR::T;
  using VecT = typename TR::VecT;
  using AccT = typename TR::AccT;
  constexpr int TM = TR::TM, KV = TR::KV;
  // With SHARED_A all NTILE tiles lie in one row block: one A fragment per
  // k-group serves every tile.
  constexpr int NA = SHARED_A ? 1 : NTILE;
  const int nkg = B.nkg;
  uint32_t boff[NTILE];
  const T* ap[NA];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) boff[t] = b_voff(B, tcol[t], lane);
#pragma unroll
  for (int t = 0; t < NA; ++t) ap[t] = A + (trow[t] * TM + arow) * LDA + akoff;
  auto ldb = [&](int t, int kg) -> VecT { return load_b<VecT>(B, boff[t], kg); };
  auto ia = [](int t) { return SHARED_A ? 0 : t; };
  VecT b1[NTILE], a0[NA], a1[NA];
#pragma unroll
  for (int t = 0; t < NA; ++t) a0[t] = *reinterpret_cast<const VecT*>(ap[t]);
  // Two k-groups per step.  FIRST: the step's first MFMA per tile starts
  // from a zero accumulator (an inline constant, no register clearing).
  auto step = [&](const int kg, auto first) {
    // stage 1 loads (k-group kg+1 < nkg always: nkg is even)
#pragma unroll
    for (int t = 0; t < NTILE; ++t) b1[t] = ldb(t, kg + 1);
#pragma unroll
    for (int t = 0; t < NA; ++t) a1[t] = *reinterpret_cast<const VecT*>(ap[t] + 8);
    // Keep the loads ahead of the MFMAs that do not need them: the scheduler
    // would otherwise sink them next to their use and expose their latency.
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      if constexpr (decltype(first)::value)
        acc[t] = TR::mfma(a0[ia(t)][0], b0[t][0], AccT{});
      else
        acc[t] = TR::mfma(a0[ia(t)][0], b0[t][0], acc[t]);
#pragma unroll
      for (int s = 1; s < KV; ++s) acc[t] = TR::mfma(a0[ia(t)][s], b0[t][s], acc[t]);
    }
    // stage 0 loads for k-group kg+2.  After the last step b0 re-fetches
    // k-group 0, which the next year starts with; a0 then reads the 8 values
    // past column Pk - 1 of its row (inside the LDS allocation, never used:
    // the next call reloads a0), which keeps its address an immediate offset.
    const int k2 = (kg + 2 < nkg) ? kg + 2 : 0;
#pragma unroll
    for (int t = 0; t < NTILE; ++t) b0[t] = ldb(t, k2);
#pragma unroll
    for (int t = 0; t < NA; ++t) {
      a0[t] = *reinterpret_cast<const VecT*>(ap[t] + 16);
      ap[t] += 16;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
#pragma unroll
      for (int s = 0; s < KV; ++s) acc[t] = TR::mfma(a1[ia(t)][s], b1[t][s], acc[t]);
    }
  };
  step(0, std::true_type{});
  for (int kg = 2; kg < nkg; kg += 2) step(kg, std::false_type{});
}

// Split-bf16 form of year_product (TraitsB3).  A k-chunk is 16 k: the A
// operands are 8 bf16 of the hi and of the lo array (Ah and Ah + lo_off), the
// B operands packed k-groups 2c (hi) and 2c + 1 (lo).  Each chunk issues the
// three products of every tile, one product kind at a time across the tiles,
// so that consecutive MFMAs are independent.  Stages ping-pong over the chunks
// (the chunk count is even).  Unlike year_product, no operands stay in
// registers between years: the epilogue needs them.
template <int NTILE, bool SHARED_A = false>
__device__ __forceinline__ void year_product_b3(floatx16* acc, const PackedB& B,
                                                const uint16_t* Ah,
                                                int lo_off, const int* trow, const int* tcol,
                                                int LDA, int arow, int akoff, int lane) {
  constexpr int NA = SHARED_A ? 1 : NTILE;
  const int nch = B.nkg >> 1;
  uint32_t boff[NTILE];
  const uint16_t* ap[NA];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) boff[t] = b_voff(B, tcol[t], lane);
#pragma unroll
  for (int t = 0; t < NA; ++t) ap[t] = Ah + (trow[t] * 32 + arow) * LDA + akoff;
  auto ldb = [&](int t, int kg) -> floatx4 { return load_b<floatx4>(B, boff[t], kg); };
  auto lda = [&](int t, int off) -> floatx4 {
    return *reinterpret_cast<const floatx4*>(ap[t] + off);
  };
  auto ia = [](int t) { return SHARED_A ? 0 : t; };
  floatx4 bh0[NTILE], bl0[NTILE], bh1[NTILE], bl1[NTILE], ah0[NA], al0[NA], ah1[NA], al1[NA];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) {
    bh0[t] = ldb(t, 0);
    bl0[t] = ldb(t, 1);
  }
#pragma unroll
  for (int t = 0; t < NA; ++t) {
    ah0[t] = lda(t, 0);
    al0[t] = lda(t, lo_off);
  }
  auto products = [&](const floatx4* ah, const floatx4* al, const floatx4* bh,
                      const floatx4* bl, auto first) {
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      if constexpr (decltype(first)::value)
        acc[t] = TraitsB3::mfma(ah[ia(t)], bh[t], floatx16{});
      else
        acc[t] = TraitsB3::mfma(ah[ia(t)], bh[t], acc[t]);
    }
#pragma unroll
    for (int t = 0; t < NTILE; ++t) acc[t] = TraitsB3::mfma(ah[ia(t)], bl[t], acc[t]);
#pragma unroll
    for (int t = 0; t < NTILE; ++t) acc[t] = TraitsB3::mfma(al[ia(t)], bh[t], acc[t]);
  };
  auto step = [&](const int c, auto first) {
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      bh1[t] = ldb(t, 2 * c + 2);
      bl1[t] = ldb(t, 2 * c + 3);
    }
#pragma unroll
    for (int t = 0; t < NA; ++t) {
      ah1[t] = lda(t, 16);
      al1[t] = lda(t, lo_off + 16);
    }
    __builtin_amdgcn_sched_barrier(0);
    products(ah0, al0, bh0, bl0, first);
    // The last step's stage-0 loads read chunk 0 again (B) and past the
    // row's last chunk (A: inside the LDS allocation); both are never used.
    const int c2 = (c + 2 < nch) ? c + 2 : 0;
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      bh0[t] = ldb(t, 2 * c2);
      bl0[t] = ldb(t, 2 * c2 + 1);
    }
#pragma unroll
    for (int t = 0; t < NA; ++t) {
      ah0[t] = lda(t, 32);
      al0[t] = lda(t, lo_off + 32);
      ap[t] += 32;
    }
    __builtin_amdgcn_sched_barrier(0);
    products(ah1, al1, bh1, bl1, std::false_type{});
  };
  step(0, std::true_type{});
  for (int c = 2; c < nch; c += 2) step(c, std::false_type{});
}

// acc += the split-bf16 product over k-chunks c0 .. c1 (c1 > c0) of one tile,
// with year_product_b3's ping-pong and an odd tail step.
__device__ __forceinline__ void range_product_b3(floatx16& acc, const PackedB& B,
                                                 const uint16_t* Ah, int lo_off, int trow,
                                                 int tcol, int c0, int c1, int LDA, int arow,
                                                 int akoff, int lane) {
  const uint32_t boff = b_voff(B, tcol, lane);
  const uint16_t* ap = Ah + (trow * 32 + arow) * LDA + akoff;
  auto lda = [&](int off) -> floatx4 { return *reinterpret_cast<const floatx4*>(ap + off); };
  floatx4 bh0 = load_b<floatx4>(B, boff, 2 * c0), bl0 = load_b<floatx4>(B, boff, 2 * c0 + 1);
  floatx4 ah0 = lda(16 * c0), al0 = lda(lo_off + 16 * c0);
  auto products = [&](floatx4 ah, floatx4 al, floatx4 bh, floatx4 bl) {
    acc = TraitsB3::mfma(ah, bh, acc);
    acc = TraitsB3::mfma(ah, bl, acc);
    acc = TraitsB3::mfma(al, bh, acc);
  };
  int c = c0;
  for (; c + 1 < c1; c += 2) {
    const floatx4 bh1 = load_b<floatx4>(B, boff, 2 * c + 2);
    const floatx4 bl1 = load_b<floatx4>(B, boff, 2 * c + 3);
    const floatx4 ah1 = lda(16 * (c + 1)), al1 = lda(lo_off + 16 * (c + 1));
    __builtin_amdgcn_sched_barrier(0);
    products(ah0, al0, bh0, bl0);
    const int k2 = min(c + 2, c1 - 1);
    bh0 = load_b<floatx4>(B, boff, 2 * k2);
    bl0 = load_b<floatx4>(B, boff, 2 * k2 + 1);
    ah0 = lda(16 * k2);
    al0 = lda(lo_off + 16 * k2);
    __builtin_amdgcn_sched_barrier(0);
    products(ah1, al1, bh1, bl1);
  }
  if (c < c1) products(ah0, al0, bh0, bl0);
}

// Byte offset of lane `lane`'s operands of column block `tcol` in a matrix
// packed for TraitsX6 (nch 16-k chunks, each 3 x 1 KB: the h, m and l
// operands of the 64 lanes).
__device__ __forceinline__ uint32_t b6_voff(int nch, int tcol, int lane) {
  return ((uint32_t)tcol * (uint32_t)nch * 192u + (uint32_t)lane) * 16u;
}

// acc[c * NR + r] = A[row tile r, chunks c0 .. c1) . M[those chunks, column
// tile c] for NR row tiles x NC column tiles (TraitsX6), c1 > c0; ap is the
// lane's first operand of row tile 0 (chunk 0), rstep the row tiles' distance
// and boff[c] the column tiles' offsets.  Blocks of 2 x 2 tiles use each split
// and each B operand for two tiles: 14 VALU operations and 1.5 KB of L2
// traffic per six MFMAs, against 28 and 3 KB for single tiles.  The B operands
// of the next chunk are in flight while this chunk's products run; the A
// operands are split first, then reloaded for the next chunk.
// AP: ap(r) is row tile r's operand pointer.
template <int NR, int NC, class AP>
__device__ __forceinline__ void product_x6_rows(floatx16* acc, const PackedB& B, const AP& ap,
                                                const uint32_t* boff, int c0, int c1) {
  floatx16 sm[NR * NC];
#pragma unroll
  for (int t = 0; t < NR * NC; ++t) acc[t] = sm[t] = floatx16{};
  floatx4 b0[NC][3], b1[NC][3], a[NR][2];
  auto ldb = [&](floatx4 (&b)[NC][3], int c) {
#pragma unroll
    for (int t = 0; t < NC; ++t)
#pragma unroll
      for (int i = 0; i < 3; ++i) b[t][i] = load_b<floatx4>(B, boff[t], 3 * c + i);
  };
  auto lda = [&](int c) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const floatx4* q = reinterpret_cast<const floatx4*>(ap(r) + 16 * c);
      a[r][0] = q[0];
      a[r][1] = q[1];
    }
  };
  auto step = [&](const floatx4 (&b)[NC][3], floatx4 (&bn)[NC][3], const int c) {
    const int cn = min(c + 1, c1 - 1);
    ldb(bn, cn);
    Split8 x[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) x[r] = split3_8(a[r][0], a[r][1]);
    lda(cn);
    // Keep the loads ahead of the products, which do not need them.
    __builtin_amdgcn_sched_barrier(0);
    // One term product at a time over the tiles, so that consecutive MFMAs
    // are independent.
#define RMC_X6(d, ta, ib)                                                      \
  _Pragma("unroll") for (int t = 0; t < NC; ++t)                               \
      _Pragma("unroll") for (int r = 0; r < NR; ++r) d[t * NR + r] =           \
          TraitsX6::mfma(x[r].ta, b[t][ib], d[t * NR + r])
    RMC_X6(sm, l, 0);
    RMC_X6(sm, h, 2);
    RMC_X6(sm, m, 1);
    RMC_X6(sm, m, 0);
    RMC_X6(sm, h, 1);
    RMC_X6(acc, h, 0);
#undef RMC_X6
  };
  ldb(b0, c0);
  lda(c0);
  int c = c0;
  for (; c + 1 < c1; c += 2) {
    step(b0, b1, c);
    step(b1, b0, c + 1);
  }
  if (c < c1) step(b0, b1, c);
#pragma unroll
  for (int t = 0; t < NR * NC; ++t) acc[t] += sm[t];
}

// The same with the row tiles at a fixed distance rstep.
template <int NR, int NC>
__device__ __forceinline__ void product_x6(floatx16* acc, const PackedB& B, const float* ap,
                                           int rstep, const uint32_t* boff, int c0, int c1) {
  product_x6_rows<NR, NC>(acc, B, [&](int r) { return ap + r * rstep; }, boff, c0, c1);
}

}  // namespace roadmc

#endif
