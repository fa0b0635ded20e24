// kdecay_internal.h — what the kernel files of libkdecay.so share: element
// conversion, the normaliser, the look-back words and workspace header, the
// scans' argument blocks and the host helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <math.h>
#include <mutex>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "kdecay.h"

// The reference rounds lam*s and (lam*s)+v separately (two torch ops).  The
// decode step and the sequential scan keep those two roundings (their state is
// bit-identical to the reference's); nothing is contracted implicitly.  The
// chunked scan, which reassociates the recurrence anyway and is checked to a
// tolerance, fuses each lam*s+v into one explicit fmaf: one rounding instead
// of two, and half the vector instructions of its hot loops.
#pragma clang fp contract(off)

namespace kd {

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }

// --------------------------------------------------------------------------
// Element conversion
// --------------------------------------------------------------------------
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(__bf16 x) { return (float)x; }
__device__ __forceinline__ float to_f32(_Float16 x) { return (float)x; }
__device__ __forceinline__ float to_f32(double x) { return (float)x; }

template <typename T>
__device__ __forceinline__ T from_f32(float x);
template <>
__device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <>
__device__ __forceinline__ __bf16 from_f32<__bf16>(float x) { return (__bf16)x; }
template <>
__device__ __forceinline__ _Float16 from_f32<_Float16>(float x) { return (_Float16)x; }
template <>
__device__ __forceinline__ double from_f32<double>(float x) { return (double)x; }

// 16 bytes of T -> 16/sizeof(T) floats.
template <typename T>
__device__ __forceinline__ void unpack16(const uint4& u, float* f);

template <>
__device__ __forceinline__ void unpack16<float>(const uint4& u, float* f) {
  f[0] = __uint_as_float(u.x);
  f[1] = __uint_as_float(u.y);
  f[2] = __uint_as_float(u.z);
  f[3] = __uint_as_float(u.w);
}

template <>
__device__ __forceinline__ void unpack16<__bf16>(const uint4& u, float* f) {
  const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f[2 * k] = __uint_as_float(w[k] << 16);
    f[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
  }
}

template <>
__device__ __forceinline__ void unpack16<_Float16>(const uint4& u, float* f) {
  const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const f16x2 h = __builtin_bit_cast(f16x2, w[k]);
    f[2 * k] = (float)h.x;
    f[2 * k + 1] = (float)h.y;
  }
}

// Two doubles, each rounded to float (round to nearest even), as the
// fp32-arithmetic kernels take every input type.
template <>
__device__ __forceinline__ void unpack16<double>(const uint4& u, float* f) {
  f[0] = (float)__hiloint2double((int)u.y, (int)u.x);
  f[1] = (float)__hiloint2double((int)u.w, (int)u.z);
}

__device__ __forceinline__ unsigned pack2(__bf16*, float a, float b) {
  bf16x2 p;
  p.x = (__bf16)a;
  p.y = (__bf16)b;
  return __builtin_bit_cast(unsigned, p);
}
__device__ __forceinline__ unsigned pack2(_Float16*, float a, float b) {
  f16x2 p;
  p.x = (_Float16)a;
  p.y = (_Float16)b;
  return __builtin_bit_cast(unsigned, p);
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// 16-byte store of data written once and not read back by this kernel
// (non-temporal: it does not displace cached data).
__device__ __forceinline__ void store16_stream(void* p, unsigned a, unsigned b, unsigned c, unsigned d) {
  const u32x4 v = {a, b, c, d};
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}

// Store N floats (N = 4 or 8; 2 for double) as N elements of T at p (16-byte aligned).
// Eight floats take two 16-byte stores, each of which covers every other 16
// bytes of the row's range across the lanes: through the cache, whose lines
// the second store completes before they are written back (non-temporal,
// bf16 in / fp32 out at B=8 N=4096 H=12 D=64 took 52.2 us; cached, 29.7 us).
// With 8 lanes per row the scan pairs lanes instead (ChunkScan::store_chunk).
template <typename T, int N>
__device__ __forceinline__ void store_vec(T* p, const float* f) {
  if constexpr (sizeof(T) == 4 && N == 8) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const u32x4 v = {__float_as_uint(f[4 * k]), __float_as_uint(f[4 * k + 1]), __float_as_uint(f[4 * k + 2]),
                       __float_as_uint(f[4 * k + 3])};
      *reinterpret_cast<u32x4*>(p + 4 * k) = v;
    }
  } else if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int k = 0; k < N / 4; ++k)
      store16_stream(p + 4 * k, __float_as_uint(f[4 * k]), __float_as_uint(f[4 * k + 1]),
                     __float_as_uint(f[4 * k + 2]), __float_as_uint(f[4 * k + 3]));
  } else if constexpr (sizeof(T) == 8) {
    static_assert(N == 2, "8-byte outputs are stored 2 at a time");
    const double d0 = (double)f[0], d1 = (double)f[1];
    store16_stream(p, (unsigned)__double2loint(d0), (unsigned)__double2hiint(d0), (unsigned)__double2loint(d1),
                   (unsigned)__double2hiint(d1));
  } else {
    static_assert(N == 8, "2-byte outputs are stored 8 at a time");
    store16_stream(p, pack2((T*)nullptr, f[0], f[1]), pack2((T*)nullptr, f[2], f[3]),
                   pack2((T*)nullptr, f[4], f[5]), pack2((T*)nullptr, f[6], f[7]));
  }
}

// --------------------------------------------------------------------------
// Normaliser, as the reference's torch expression evaluates it:
//   z = (1.0 - lam ** (t+1)) / (1.0 - lam + 1e-6)
// torch's pow(tensor, int scalar) returns lam for e == 1, lam*lam for e == 2,
// (lam*lam)*lam for e == 3, and a float power otherwise.  For e >= 4 this
// takes the float rounding of lam^e evaluated in double by binary
// exponentiation (at most 2*64 double products, relative error < 2^-45, so
// the float result is the correctly rounded power except within 2^-45 of a
// rounding tie).  Every other operation is one rounded fp32 op.
// --------------------------------------------------------------------------
__device__ __forceinline__ double ipow_f64(double x, int64_t e) {
  double r = 1.0;
  while (e > 0) {
    if (e & 1) r *= x;
    x *= x;
    e >>= 1;
  }
  return r;
}

__device__ __forceinline__ float pow_like_torch(float x, int64_t e) {
  if (e == 1) return x;
  if (e == 2) return x * x;
  if (e == 3) return (x * x) * x;
  if (e == 0) return 1.0f;
  return (float)ipow_f64((double)x, e);
}

// Wait until at most N vector memory operations of this wavefront are
// outstanding (vmcnt only; the other counters are left alone).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

__device__ __forceinline__ float z_of(float lam, int64_t t) {
  const float num = 1.0f - pow_like_torch(lam, t + 1);
  const float den = (1.0f - lam) + 1e-6f;
  return num / den;
}

// The same values with lower latency, for the decode step, where z is on the
// critical path of a launch-latency-bound kernel: for e < 2^16 the binary
// exponentiation is unrolled and branch-free (the same products in the same
// order as ipow_f64; squarings past the top bit do not reach r), 12 steps
// instead of 16 for e < 2^12 (C3 decode step 2.22 -> 2.18 us), and the small
// cases are selects instead of branches.  The scan kernels keep the
// loop: they build their z tables while their rows are in flight, and there
// the shorter form measured 3.7% slower (bf16, B=8 N=4096 H=12 D=64).
// x^e by binary exponentiation for 0 <= e < 2^BITS, unrolled and branch-free
// (the products of ipow_f64, in the same order).
template <int BITS>
__device__ __forceinline__ double ipow_f64_bits(double x, unsigned e) {
  double r = 1.0;
#pragma unroll
  for (int k = 0; k < BITS; ++k) {
    const double rx = r * x;
    r = (e >> k) & 1u ? rx : r;
    x *= x;
  }
  return r;
}

// ipow_f64 with the unrolled form for exponents below 2^16.
__device__ __forceinline__ double ipow_f64_fast(double x, int64_t e) {
  if (e >= 0 && e < (1 << 12)) return ipow_f64_bits<12>(x, (unsigned)e);
  if (e >= 0 && e < (1 << 16)) return ipow_f64_bits<16>(x, (unsigned)e);
  return ipow_f64(x, e);
}

__device__ __forceinline__ float pow_like_torch_fast(float x, int64_t e) {
  const double r = ipow_f64_fast((double)x, e);
  const float p2 = x * x;
  const float p3 = p2 * x;
  return e == 1 ? x : e == 2 ? p2 : e == 3 ? p3 : e == 0 ? 1.0f : (float)r;
}

__device__ __forceinline__ float z_of_fast(float lam, int64_t t) {
  const float num = 1.0f - pow_like_torch_fast(lam, t + 1);
  const float den = (1.0f - lam) + 1e-6f;
  return num / den;
}

// --------------------------------------------------------------------------
// Division by a divisor fixed for the launch: a multiply and a shift
// (Granlund & Montgomery, "Division by invariant integers using
// multiplication", PLDI 1994, theorem 4.2 with N = 31: for 2^(l-1) < d <= 2^l
// and m = ceil(2^(31+l) / d) < 2^32, floor(n * m / 2^(31+l)) = floor(n / d)
// for 0 <= n < 2^31).  A compiled division by a runtime value is a chain of
// about 25 dependent instructions (a 64-bit one about 100); the kernels do
// theirs before their first load.
// --------------------------------------------------------------------------
struct FastDiv {
  uint32_t d, m, s;
  __host__ __device__ uint32_t div(uint32_t n) const { return (uint32_t)(((uint64_t)n * m) >> s); }
  __host__ __device__ uint32_t mod(uint32_t n) const { return n - div(n) * d; }
};

// d >= 1.
inline FastDiv make_fastdiv(uint32_t d) {
  uint32_t l = 0;
  while (l < 32 && ((uint64_t)1 << l) < d) ++l;
  const uint32_t s = 31 + l;
  const uint64_t p = (uint64_t)1 << s;  // s <= 63
  return FastDiv{d, (uint32_t)((p + d - 1) / d), s};
}

// --------------------------------------------------------------------------
// Look-back words and the workspace header
// --------------------------------------------------------------------------
typedef unsigned long long u64;

// Header words (first 256 bytes of the workspace).
//   EPOCH  launch generation: look-back words of older launches never match
//   ERROR  sticky fault word (1: a bounded wait gave up).  Every launch reads
//          it with the epoch (one 64-bit load) and, when it is set, writes
//          NaN to all its outputs instead of trusting the workspace: after a
//          give-up, words of the launch that gave up may carry a later
//          launch's tag, so only a cleared workspace computes again.
//   DONE   workgroups of the running launch that have counted toward the
//          epoch's advance (the forward: each stream's last chunk, directly
//          or through a sub-count; the backward: see ChunkBwd::run)
// From byte 256: kCountSlots sub-counts, 32 bytes apart (count_done_2).
enum { HDR_EPOCH = 0, HDR_ERROR = 1, HDR_DONE = 2 };
constexpr unsigned kCountSlots = 64;
constexpr unsigned kCountBase = 64;    // word index of the first sub-count (byte 256)
constexpr unsigned kCountStride = 8;   // words between sub-counts (32 bytes)
constexpr size_t kHeaderBytes = 4 * (kCountBase + kCountSlots * kCountStride);  // 2304

// The epoch and the error word of a workspace header, as one load.
struct EpochErr {
  unsigned epoch, err;
};

__device__ __forceinline__ EpochErr split_header(u64 w) { return EpochErr{(unsigned)w, (unsigned)(w >> 32)}; }

// Tag of a word published in launch `epoch`: kind 0 = aggregate, 1 = inclusive.
// Zeroed memory (tag 0) never matches a live tag.
__device__ __forceinline__ unsigned tag_of(unsigned epoch, unsigned kind) {
  return (((epoch & 0x3fffffffu) + 1u) << 1) | kind;
}

__device__ __forceinline__ void publish(u64* p, unsigned tag, float v) {
  const u64 w = ((u64)tag << 32) | (u64)__float_as_uint(v);
  __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ u64 peek(const u64* p) {
  return __hip_atomic_load(const_cast<u64*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Polls before a look-back gives up (well over a second): the kernel then
// exits normally and flags the header instead of hanging.
constexpr int kSpinLimit = 1 << 20;

// Look-back window.  When every workgroup of a launch is resident at once, a
// wider window resolves the chunk chains in fewer polls; when the launch runs
// in several rounds, the chunks a workgroup waits on have mostly finished in
// an earlier round, and reading fewer words per poll wins.  Measured (bf16,
// same-box A/B): B=8 N=4096 H=12 D=64 (768 chunks, one round) window 4
// 18.3 us, 2 18.5 us; B=1 N=65536 H=16 D=128 (4096 chunks, four rounds)
// window 4 96.0 us, 3 94.5 us, 2 93.4 us.
constexpr int kW = 4;        // the whole grid resident at once
constexpr int kWRounds = 2;  // several rounds

// Look-back words of the W chunks before chunk c (c >= 1) for channel d:
// w[k] = word of chunk c-1-k.  The reads are unconditional (a load under a
// branch is waited for at the branch join): where c-1-k < 0 the word of chunk
// 0 is read again, and a fold never gets past chunk 0's word, which is always
// inclusive; a lane past the last channel reads the last channel's words.
template <int W, int DG>
__device__ __forceinline__ void read_window(const u64* base, int c, int d, u64 (&w)[W]) {
  const u64* col = base + (d < DG ? d : DG - 1);
#pragma unroll
  for (int k = 0; k < W; ++k) {
    const int ck = c - 1 - k > 0 ? c - 1 - k : 0;
    w[k] = peek(col + (int64_t)ck * DG);
  }
}

// F(c-1) for one channel from the words of the W chunks before chunk c, if
// they determine it: the nearest inclusive word, then the aggregates after
// it folded oldest first (F = mL * F + agg).  Every inclusive word is the same
// left fold from the start of the stream, so the result does not depend on
// which inclusive word is the nearest one.  Returns false when a word the fold
// needs is not (yet) published.
template <int W>
__device__ __forceinline__ bool fold_window(const u64 (&w)[W], unsigned tag_agg, unsigned tag_inc, float mL,
                                            float& carry) {
  int m = -1;
  bool open = true;
#pragma unroll
  for (int k = 0; k < W; ++k) {
    const unsigned tag = (unsigned)(w[k] >> 32);
    if (open && tag == tag_inc) m = k;
    if (tag != tag_agg) open = false;
  }
  if (m < 0) return false;
  float f = __uint_as_float((unsigned)w[m]);
#pragma unroll
  for (int k = W - 1; k >= 0; --k)
    if (k < m) f = __builtin_fmaf(mL, f, __uint_as_float((unsigned)w[k]));
  carry = f;
  return true;
}

// Look-back of wavefront 0 for chunk c (c >= 1): carry[q] = F(c-1) of channel
// lane + 64q.  Re-reads the window until every channel's fold succeeds.  A
// look-back that gives up sets the sticky error word and returns a NaN carry
// for the channels it could not resolve: every output that carry reaches
// (the chunk's rows, its inclusive word, and through it later chunks and the
// final state) is NaN, so a caller that checks its outputs for finite values
// sees the fault, not a plausible wrong number.
template <int W, int DG, int DQ>
__device__ void look_back(const u64* base, int c, unsigned tag_agg, unsigned tag_inc, float mL, unsigned* hdr,
                          int spin_limit, float (&carry)[DQ]) {
  const int lane = threadIdx.x & 63;
  bool done[DQ];
#pragma unroll
  for (int q = 0; q < DQ; ++q) done[q] = lane + 64 * q >= DG;
  for (int spin = 0;; ++spin) {
#pragma unroll
    for (int q = 0; q < DQ; ++q) {
      if (!done[q]) {
        u64 w[W];
        read_window<W, DG>(base, c, lane + 64 * q, w);
        done[q] = fold_window<W>(w, tag_agg, tag_inc, mL, carry[q]);
      }
    }
    bool all = true;
#pragma unroll
    for (int q = 0; q < DQ; ++q) all &= done[q];
    if (__ballot(!all) == 0ull) return;
    if (spin >= spin_limit) {
      __hip_atomic_store(hdr + HDR_ERROR, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int q = 0; q < DQ; ++q)
        if (!done[q]) carry[q] = __builtin_nanf("");
      return;
    }
    __builtin_amdgcn_s_sleep(1);
  }
}

// Sum of x over the 64 lanes of the wavefront, in a fixed order (the same
// result on every run): DPP butterflies inside each row of 16 lanes, then the
// four row sums.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

__device__ __forceinline__ float wave_sum(float x) {
  x += dpp_f32<0xB1>(x);   // quad_perm [1,0,3,2]
  x += dpp_f32<0x4E>(x);   // quad_perm [2,3,0,1]
  x += dpp_f32<0x141>(x);  // row_half_mirror
  x += dpp_f32<0x140>(x);  // row_mirror
  const int xi = __builtin_bit_cast(int, x);
  return (__builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 0)) +
          __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 16))) +
         (__builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 32)) +
          __builtin_bit_cast(float, __builtin_amdgcn_readlane(xi, 48)));
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// wave_sum in double, same fixed order.
__device__ __forceinline__ double wave_sum_f64(double x) {
  x += dpp_f64<0xB1>(x);
  x += dpp_f64<0x4E>(x);
  x += dpp_f64<0x141>(x);
  x += dpp_f64<0x140>(x);
  return (readlane_f64(x, 0) + readlane_f64(x, 16)) + (readlane_f64(x, 32) + readlane_f64(x, 48));
}

// Index of the calling wavefront in its workgroup, as a wavefront-uniform
// (scalar) value: loops and branches on it are then scalar, not exec-masked.
__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// Value of `x` held K row groups below (row groups are S lanes apart, GW per
// wavefront; lanes whose group index is below K get an unspecified value).
// Adjacent groups of up to 16 lanes use a DPP row shift (no LDS traffic);
// anything else a lane permute.
template <int K, int GW, int S>
__device__ __forceinline__ float lane_shr(float x) {
  if constexpr (S == 1 && GW <= 16) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x110 | K, 0xf, 0xf, false));
  } else {
    return __shfl_up(x, K * S, 64);
  }
}

// Inclusive scan of the per-lane states over the GW row groups of a
// wavefront: acc(g) = lam^(R*K) * acc(g - K) + acc(g) for K = 1, 2, 4, ...
// pw[K] holds lam^(R*K).
template <int K, int GW, int VW, int S>
__device__ __forceinline__ void group_scan(float (&acc)[VW], int gw, const float* pw) {
  if constexpr (K < GW) {
    const float m = pw[K];
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      const float o = lane_shr<K, GW, S>(acc[j]);
      if (gw >= K) acc[j] = __builtin_fmaf(m, o, acc[j]);
    }
    group_scan<2 * K, GW, VW, S>(acc, gw, pw);
  }
}

// --------------------------------------------------------------------------
// Chunked single-pass scan
// --------------------------------------------------------------------------
struct ScanArgs {
  const void* V;
  void* out;
  const float* lam;
  const float* init;  // [B*H*D] or null
  float* fin;         // [B*H*D] or null
  int64_t vb, vh, vn; // element strides of V (d stride 1)
  int64_t ob, oh, on; // element strides of out (d stride 1)
  int64_t H, N, t_offset;
  int64_t D;    // head dim (channels of a (b,h) pair)
  int ng;       // channel groups per head: a stream is (b, h, group)
  int nchunk;   // chunks per stream
  int nstream;  // B*H*ng
  u64* flags;   // [nstream][nchunk][DG] look-back words (null if nchunk == 1)
  unsigned* hdr;
  // Optional: the state after every `state_rows` rows, for the backward pass.
  // states[(bh * nsaved + k) * D + d] = s of channel d of head bh at row
  // k * state_rows - 1 (1 <= k < nsaved = ceil(N / state_rows); entry 0 is
  // not written): by head and channel, so the backward may group a head's
  // channels into streams other than the forward's.
  float* states;
  int64_t state_rows;
  int64_t nsaved;
  // With the states: the backward's terms of every row of every head,
  // rowtab[h * N + t] = (1/z, d(1/z)/dlam) at row t (bwd_row_terms), written
  // by the streams of batch 0, first channel group.
  float2* rowtab;
  int spin_limit;  // polls before a look-back gives up (kSpinLimit unless a test lowers it)
  FastDiv f_nstream, f_ng, f_H;  // division by nstream, ng and H
};

// 16-byte load of data read exactly once (non-temporal: no cache residency).
__device__ __forceinline__ uint4 load16_stream(const void* p) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Buffer resource over `rows` rows of a stream of DG channels, `stride`
// elements apart (stride >= DG), starting at p: the range ends with the last
// row's channels, so a buffer load of any later row returns zeros without
// touching memory.  Offsets are 32-bit: the host keeps a chunk's rows within
// 2^31 bytes.
template <int DG, typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_buffer(const T* p, int64_t rows, int64_t stride) {
  const int64_t bytes = rows > 0 ? ((rows - 1) * stride + DG) * (int64_t)sizeof(T) : 0;
  const int n = bytes > 0x7fffffffLL ? 0x7fffffff : (int)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), (short)0, n, 0x00020000);
}

// 16-byte non-temporal buffer load at byte offset `off`.
__device__ __forceinline__ uint4 load16_buffer(__amdgpu_buffer_rsrc_t r, unsigned off) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 2);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// The launch epoch from the workspace header, kept in a vector register:
// read through a uniform address, the value was moved to a scalar register
// at once, which waited for the load (and every load issued before it).
// One of n workgroups that each finish a launch's use of the epoch: the
// last of them resets the count and advances the epoch for the next launch.
__device__ __forceinline__ void count_done(unsigned* hdr, unsigned n, unsigned epoch) {
  const unsigned d = __hip_atomic_fetch_add(hdr + HDR_DONE, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (d == n - 1u) {
    __hip_atomic_store(hdr + HDR_DONE, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(hdr + HDR_EPOCH, epoch + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// count_done for n workgroups numbered s = 0..n-1 in two levels: workgroup s
// counts on sub-count s % kCountSlots, and the one that completes a sub-count
// counts on DONE (min(n, kCountSlots) of them).  With every count on one word
// the n atomics of a launch queue on that word at the launch's end.  Measured
// (the forward, bf16 D=64, same-box A/B, us, one word / 64 sub-counts 32
// bytes apart): B=128 N=512 H=12 (1536 streams) 106.6 / 42.7, B=64 N=4096
// H=12 (768) 171.3 / 143.5, B=64 N=1024 H=12 44.1 / 39.4, B=40 N=4096 H=16
// (640) 132.5 / 120.6, B=48 N=4096 H=12 (576) 117.2 / 110.8; 16 sub-counts in
// one 64-byte segment did not help (109.6 at 1536 streams), 16 of them 256
// bytes apart nearly did (46.3).  With fewer streams the second atomic is the
// cost: B=16 N=4096 H=12 (192 streams) 38.4 / 38.7, B=8 (96) 17.36 / 17.59;
// between them no gain (B=20, 24, 32 H=12: 48.6 / 48.7, 57.8 / 57.7, 72.2 /
// 72.0; B=16 H=16, 256 streams: 46.6 / 47.1).
__device__ __forceinline__ void count_done_2(unsigned* hdr, unsigned n, unsigned s, unsigned epoch) {
  const unsigned k = s % kCountSlots;
  const unsigned nk = n / kCountSlots + (k < n % kCountSlots ? 1u : 0u);
  unsigned* c = hdr + kCountBase + k * kCountStride;
  const unsigned d = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (d == nk - 1u) {
    __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    count_done(hdr, n < kCountSlots ? n : kCountSlots, epoch);
  }
}

// Streams up to which the forward counts each stream's last chunk on DONE
// directly (count_done_2 above it).
constexpr int kFwdPerStreamCount = 384;

__device__ __forceinline__ EpochErr read_epoch_v(const unsigned* hdr) {
  unsigned zero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
  return split_header(__hip_atomic_load(reinterpret_cast<u64*>(const_cast<unsigned*>(hdr)) + zero, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT));
}

// Keeps `x` opaque to the optimiser at this point, so values derived from it
// are recomputed after the barrier rather than held in registers across it.
__device__ __forceinline__ void opaque(uint4& x) {
  asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));
}

// Pins the values of x at this point of the program: computations feeding
// them are done before it and uses come after it (a row-by-row sweep then
// stays row by row instead of running one chain ahead and holding its values).
template <int N>
__device__ __forceinline__ void pin(float (&x)[N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) asm volatile("" : "+v"(x[j]));
}

// Stream of item j (0 <= j < nstream) of a chunk row rotated by `rot`.
// Items are numbered row by row (every item of chunk row r precedes every
// item of row r+1), so the chunk an item waits on always has a smaller item
// number, whatever the order inside a row.  Inside a row the streams are
// rotated by a different amount per row: workgroups go to the XCDs round-robin
// by index, so without the rotation, whenever nstream is a multiple of 8,
// every chunk of a stream would run on one XCD and each XCD's traffic would
// stay inside its own streams' address ranges.  Spread over the XCDs, the
// same launches ran 10% faster for B=1 N=65536 H=16 D=128 and about 2% faster
// (and steadier from one allocation to the next) for B=8 N=4096 H=12 D=64.
__device__ __forceinline__ int rotated_stream(int j, int rot, int nstream) {
  const int k = j + rot;  // rot < nstream
  return k >= nstream ? k - nstream : k;
}

// Where item `item` of a launch is: chunk (row of chunks), stream, and the
// stream's (b, h, channel group).  Computed once per workgroup.
struct Pos {
  int chunk, stream, bh, grp, b, h;
};

__device__ __forceinline__ Pos pos_of(const ScanArgs& a, int item) {
  Pos p;
  p.chunk = (int)a.f_nstream.div((uint32_t)item);
  const int j = item - p.chunk * a.nstream;
  p.stream = rotated_stream(j, (int)a.f_nstream.mod((uint32_t)p.chunk), a.nstream);
  p.bh = (int)a.f_ng.div((uint32_t)p.stream);
  p.grp = p.stream - p.bh * a.ng;
  p.b = (int)a.f_H.div((uint32_t)p.bh);
  p.h = p.bh - p.b * (int)a.H;
  return p;
}

// The backward's terms of one row with exponent e = t + 1, from p = lam^(e-1):
//   x = 1/z = ((1 - lam) + 1e-6) / (1 - lam^e)   (lam^e as z_of takes it)
//   y = d(1/z)/dlam = (e lam^(e-1) ((1 - lam) + 1e-6) - (1 - lam^e)) / (1 - lam^e)^2
// lam^e is p times lam (in double); y's numerator, a small difference of
// nearly equal terms when lam is close to 1, stays in double, and both
// quotients are fp32 divisions.  (Two double-precision power loops and a
// double division per row were most of the table's cost; it is built by
// every workgroup for its chunk's rows, on the critical path after the rows
// arrive.)
__device__ __forceinline__ void bwd_row_terms(float lam, int64_t e, double p, float& x, float& y) {
  const double l = lam;
  const double pe = p * l;
  const float pf = e == 1 ? lam : e == 2 ? lam * lam : e == 3 ? (lam * lam) * lam : (float)pe;
  x = ((1.0f - lam) + 1e-6f) / (1.0f - pf);
  const double A = 1.0 - pe;
  y = (float)((double)e * p * ((1.0 - l) + 1e-6) - A) / (float)(A * A);
}

// The launch epoch and the error word, read by every thread before it loads
// any rows (so that waiting for them does not wait for the rows).  A launch
// of one chunk per stream has no workspace.
__device__ __forceinline__ EpochErr read_epoch(const ScanArgs& a) {
  if (a.nchunk <= 1) return EpochErr{0u, 0u};
  return split_header(__hip_atomic_load(reinterpret_cast<u64*>(a.hdr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

struct BwdArgs {
  const void* V;
  const void* gy;
  void* dv;
  const float* lam;
  const float* init;    // [B*H*D] or null
  const float* states;  // forward states at chunk starts (ScanArgs::states layout, by head and channel), null if nchunk == 1
  const float2* rowtab; // the training forward's per-row terms (ScanArgs::rowtab), null if nchunk == 1
  const float* gfin;    // [B*H*D] or null: gradient of the final state
  float* dinit;         // [B*H*D] or null
  float* dlam;          // [H]
  u64* partial;         // [nchunk * nstream] dlam partial per chunk (rc * nstream + stream), epoch-tagged words
  int64_t vb, vh, vn, gb, gh, gn, db, dh, dn;
  int64_t B, H, N, t_offset, D;
  int ng, nchunk, nstream;
  int64_t nsaved;
  u64* flags;
  unsigned* hdr;
  int spin_limit;  // as ScanArgs::spin_limit, for the look-back and the dlam reduction
  int ndone;       // workgroups that count toward the epoch's advance (ChunkBwd::run)
  int per_stream;  // 1: the first chunk of every stream counts instead
  FastDiv f_nstream, f_ng, f_H, f_nchunk;  // division by nstream, ng, H and nchunk
  // Batch slices (kdecay_scan_bwd): this launch is slice `slice` of `nslice`;
  // the earlier slices' per-head dlam sums, in double ([nslice - 1][H]).
  int slice, nslice;
  double* dlam_slices;
};

// XCDs of the device: workgroups are handed to them round-robin by index, and
// each XCD dispatches its share in index order.
constexpr int kXcds = 8;

// dlam[h] = the sum of head h's chunk partials in double, in a fixed order
// whatever the order in which they arrive (deterministic): wavefront 0
// alone, each lane summing a strided subset (all its reads issued at
// once), then a fixed butterfly across the lanes.
// SL: a launch over a batch slice (BwdArgs::nslice).
template <bool SL>
__device__ __forceinline__ void reduce_head(const BwdArgs& a, int h, unsigned epoch, bool poisoned) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  const unsigned tag = tag_of(epoch, 0u);
  const int n = (int)a.B * a.ng * a.nchunk;
  constexpr int K = 8;
  double acc = 0.0;
  for (int i0 = 0; i0 < n; i0 += 64 * K) {
    const u64* p[K];
    u64 w[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int idx = i0 + lane + 64 * k < n ? i0 + lane + 64 * k : n - 1;
      const int bg = (int)a.f_nchunk.div((uint32_t)idx), rc = idx - bg * a.nchunk;
      const int b = (int)a.f_ng.div((uint32_t)bg), grp = bg - b * a.ng;
      p[k] = a.partial + (int64_t)rc * a.nstream + ((int64_t)b * a.H + h) * a.ng + grp;
      w[k] = peek(p[k]);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (i0 + lane + 64 * k >= n) continue;
      for (int spin = 0; (unsigned)(w[k] >> 32) != tag; ++spin) {
        if (spin >= a.spin_limit) {  // give up: flag it, and the head's dlam becomes NaN
          __hip_atomic_store(a.hdr + HDR_ERROR, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          w[k] = ((u64)tag << 32) | 0x7fc00000u;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        w[k] = peek(p[k]);
      }
      acc += (double)__uint_as_float((unsigned)w[k]);
    }
  }
  acc = wave_sum_f64(acc);
  if (lane == 0) {
    // Only the batch-slice kernels carry this (compiled into every kernel,
    // it cost one more VGPR, and five waves per SIMD, in the 4-row
    // narrow-group kernels and 1.2% at the B=8 N=4096 H=12 backward).
    if constexpr (SL) {
      if (a.slice + 1 < a.nslice) {
        a.dlam_slices[(int64_t)a.slice * a.H + h] = acc;  // the last slice adds it
      } else {
        double t = acc;
        if (a.slice > 0) {  // the earlier slices' sums in slice order, then this one's
          t = a.dlam_slices[h];
          for (int sl = 1; sl < a.slice; ++sl) t += a.dlam_slices[(int64_t)sl * a.H + h];
          t += acc;
        }
        a.dlam[h] = (float)t;
      }
    } else {
      a.dlam[h] = (float)acc;
    }
    if (!a.per_stream && !poisoned) count_done(a.hdr, (unsigned)a.ndone, epoch);
  }
}

// --------------------------------------------------------------------------
// Host helpers (kdecay.hip)
// --------------------------------------------------------------------------
int fail(int code, const char* fmt, ...);
int hip_check(const char* what);
int elem_size(int dt);
bool dtype_ok(int dt);
bool fwd_dtype_ok(int dt);
int spin_limit();
int cu_count();
int check_scan_args(const void* V, int v_dtype, const int64_t* v_strides, const void* out, int out_dtype,
                    const int64_t* out_strides, const float* lam, int64_t B, int64_t H, int64_t N, int64_t D);
int empty_final_state(const float* init, float* fin, int64_t n, hipStream_t s);
int empty_backward(const float* g_final, float* d_init, float* dlam, int64_t B, int64_t H, int64_t D, hipStream_t s);
int bwd_done_count(int64_t B, int64_t H, int64_t ng, int64_t nchunk);

// Streams up to which every stream's first chunk counts toward the epoch's
// advance (ChunkBwd::run).  Measured (bf16, same-box A/B, per stream / per
// head and XCD, us): D=64 B=8 N=1024 H=6 (48 streams) 11.13 / 11.48; B=8
// N=4096 H=12 (96) 28.77 / 29.17; B=12 N=2048 H=16 (192) 29.31 / 29.61;
// B=16 N=2048 H=16 (256) 40.68 / 40.86; B=16 N=1024 H=16 (256) 23.96 /
// 23.21; B=24 N=1024 H=16 (384) 37.23 / 29.21.
constexpr int64_t kBwdPerStreamCount = 192;

}  // namespace kd
