// kdecay_rows.hip — the global-decay scan for head dims and alignments that the
// channel-group kernels of kdecay.hip do not take (head dims such as 48, 80, 96
// or 100, rows or bases off the 16-byte grid), straight from and to the
// caller's arrays.
//
// The algorithm is that of kdecay.hip (one workgroup per chunk of rows of one
// stream, rows in registers, look-back across chunks); what differs is how a
// row is split among lanes.  A stream is one (b,h) pair and whole rows of up to
// 256 bytes: lpr lanes of 16 bytes each, any number from 1 to 16, so a wavefront
// holds 64 / lpr row groups and its last 64 % lpr lanes are idle.  Wider rows
// are split into the fewest equal streams.  Where a row is not a whole number
// of 16-byte vectors, its last vector starts early enough to end with the row:
// the channels it shares with the vector before it are computed twice, with
// the same operations and so the same bits, and stored twice.  Loads and
// stores assume the element type's alignment only (gfx950 takes 16-byte
// accesses at any address).
//
// Against zero-padding the rows to the next head dim of kdecay.hip (fill, copy
// in, scan, copy out: four more passes over memory) this is bounded, as those
// kernels are, by one read of V and one write of y.
#include "kdecay_internal.h"

#pragma clang fp contract(off)  // as kdecay_internal.h: nothing is contracted implicitly

namespace kd {

// How a head's rows are split: the same for the forward and the backward.
struct RowSplit {
  int lpr;   // lanes (16-byte vectors) per row of a stream
  int ng;    // streams per head
  bool ok;
};

constexpr int kMaxLanes = 16;  // 256-byte rows

// Head dims of less than one vector have no last vector that fits the row.
// (A last stream of one vector that overlaps the stream before it is left out
// too: with out written over V, one workgroup could read what the other has
// already written.)
RowSplit row_split(int v_dtype, int64_t D) {
  const int64_t vw = 16 / elem_size(v_dtype);
  RowSplit s{0, 0, false};
  if (D < vw) return s;
  const int64_t nv = (D + vw - 1) / vw;
  const int64_t ng = (nv + kMaxLanes - 1) / kMaxLanes;
  if (ng > 1 << 20) return s;
  s.ng = (int)ng;
  s.lpr = (int)((nv + ng - 1) / ng);
  const int64_t left = nv - (ng - 1) * s.lpr;  // vectors of the last stream
  s.ok = left >= 1 && (ng == 1 || left >= 2 || D % vw == 0);
  return s;
}

struct RowScanArgs {
  ScanArgs s;  // ng: streams per head; flags: [nstream][nchunk][slots] words
  int lpr, gw;  // lanes per row, row groups per wavefront
  int slots;    // lpr * channels per vector: a stream's channels, shared ones twice
  FastDiv f_lpr;
};

// 16 bytes at any element boundary (the smallest element is 2 bytes).
typedef u32x4 u32x4_any __attribute__((aligned(2)));

template <typename T>
__device__ __forceinline__ uint4 load16_any(const T* p) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

// One 16-byte store, non-temporal (NT) or through the cache.
//
// Rows of whole 64-byte pieces are stored non-temporally, as in kdecay.hip;
// others leave pieces that another instruction, lane group or workgroup
// completes, which non-temporal stores send to memory one by one.  Measured
// (us, non-temporal / cached stores, buffers past the Infinity Cache): fp16
// D=80 (160-byte rows) B=8 H=16 N=2047 25.3 / 19.9 from the projection layout,
// 23.3 / 20.0 contiguous; bf16 D=100 B=8 H=12 N=2048 21.5 / 16.9; bf16 D=48 B=8
// H=16 N=4096 contiguous 33.7 / 22.0; but bf16 D=96 (192-byte rows) B=8 H=8
// N=3001 17.6 / 19.3, B=16 H=16 N=4096 92.2 / 105.5.  Cached loads lose with
// either (D=80 23.4, D=96 22.6, D=100 20.8).
template <bool NT>
__device__ __forceinline__ void store16_any(void* p, u32x4 v) {
  if constexpr (NT)
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4_any*>(p));
  else
    *reinterpret_cast<u32x4_any*>(p) = v;
}

// N floats as elements of T at p: one 16-byte store, or two for the fp32 output
// of a 2-byte V (those always through the cache, see store_vec).
template <typename T, int N, bool NT>
__device__ __forceinline__ void store_any(T* p, const float* f) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int k = 0; k < N / 4; ++k) {
      const u32x4 v = {__float_as_uint(f[4 * k]), __float_as_uint(f[4 * k + 1]), __float_as_uint(f[4 * k + 2]),
                       __float_as_uint(f[4 * k + 3])};
      store16_any<NT && N == 4>(p + 4 * k, v);
    }
  } else if constexpr (sizeof(T) == 8) {
    const double d0 = (double)f[0], d1 = (double)f[1];
    const u32x4 v = {(unsigned)__double2loint(d0), (unsigned)__double2hiint(d0), (unsigned)__double2loint(d1),
                     (unsigned)__double2hiint(d1)};
    store16_any<NT>(p, v);
  } else {
    const u32x4 v = {pack2((T*)nullptr, f[0], f[1]), pack2((T*)nullptr, f[2], f[3]), pack2((T*)nullptr, f[4], f[5]),
                     pack2((T*)nullptr, f[6], f[7])};
    store16_any<NT>(p, v);
  }
}

// First channel of vector `vec` of a head's row (the last one ends with the
// row; vectors past it, of the last stream's surplus lanes, repeat it).
template <int VW>
__device__ __forceinline__ int vec_channel(int vec, int D) {
  return vec * VW < D - VW ? vec * VW : D - VW;
}

// Where item `item` of a launch is (pos_of), with the streams of a chunk row
// numbered so that consecutive ones land on one XCD (workgroups go to the XCDs
// round-robin by index): adjacent heads of the projection layout share the
// memory lines where one row piece ends and the next begins, and then share
// them in one L2.  Measured (us, pos_of's order / this one, projection layout,
// buffers past the Infinity Cache): fp16 D=80 B=8 H=16 N=2047 28.7 / 19.9, bf16
// D=96 B=8 H=8 N=3001 19.1 / 17.6, B=16 H=16 N=4096 99.4 / 92.2, bf16 D=24 B=8
// H=12 N=4096 26.4 / 15.1, D=72 B=128 H=12 N=200 34.9 / 22.4; contiguous
// layouts equal.
__device__ __forceinline__ Pos rows_pos(const ScanArgs& a, int item) {
  Pos p;
  p.chunk = (int)a.f_nstream.div((uint32_t)item);
  const int j = rotated_stream(item - p.chunk * a.nstream, (int)a.f_nstream.mod((uint32_t)p.chunk), a.nstream);
  const int x = j % kXcds, most = a.nstream % kXcds;
  p.stream = x * (a.nstream / kXcds) + (x < most ? x : most) + j / kXcds;
  p.bh = (int)a.f_ng.div((uint32_t)p.stream);
  p.grp = p.stream - p.bh * a.ng;
  p.b = (int)a.f_H.div((uint32_t)p.bh);
  p.h = p.bh - p.b * (int)a.H;
  return p;
}

// look_back of kdecay_internal.h for a number of channels known at run time
// (slots, at most 64 * DQ).
template <int W, int DQ>
__device__ void look_back_rows(const u64* base, int c, int slots, unsigned tag_agg, unsigned tag_inc, float mL,
                               unsigned* hdr, int spin_limit, float (&carry)[DQ]) {
  const int lane = threadIdx.x & 63;
  bool done[DQ];
#pragma unroll
  for (int q = 0; q < DQ; ++q) done[q] = lane + 64 * q >= slots;
  for (int spin = 0;; ++spin) {
#pragma unroll
    for (int q = 0; q < DQ; ++q) {
      if (!done[q]) {
        const u64* col = base + lane + 64 * q;
        u64 w[W];
#pragma unroll
        for (int k = 0; k < W; ++k) {
          const int ck = c - 1 - k > 0 ? c - 1 - k : 0;
          w[k] = peek(col + (int64_t)ck * slots);
        }
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

// The forward.  As scan_chunked (kdecay.hip): tables and a sequential pass per
// lane, a scan across the wavefront's row groups, a fold across wavefronts, the
// look-back, and a second pass that stores y.
// NT: non-temporal stores.  THR: at most two rows' stores in flight.
template <typename TI, typename TO, int R, int NW, int W, int WPE, bool THR, bool NT>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
void scan_rows(RowScanArgs ra) {
  constexpr int VW = 16 / (int)sizeof(TI);
  constexpr int NTH = NW * 64;  // threads
  constexpr int DQ = (kMaxLanes * VW + 63) / 64;  // channels per lane of wavefront 0
  const ScanArgs& a = ra.s;
  const EpochErr eh = read_epoch(a);
  const Pos p = rows_pos(a, (int)blockIdx.x);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lpr = ra.lpr, GW = ra.gw, S = ra.slots;
  const int G = NW * GW, L = G * R;
  const int D = (int)a.D;
  const int chunk = p.chunk, stream = p.stream;
  const bool multi = a.nchunk > 1, last = chunk == a.nchunk - 1;
  const int64_t row0 = (int64_t)chunk * L;
  const int vec0 = p.grp * lpr;

  extern __shared__ float4 smem4[];  // 16-byte aligned
  float* const rz = reinterpret_cast<float*>(smem4);  // [L] 1 / z of each row of the chunk
  float* const wt = rz + L;           // [NW][S] per-wavefront totals (zero carry in)
  float* const sm_carry = wt + NW * S;  // [S] F(chunk - 1)
  float* const pw = sm_carry + S;     // [G + 1] lam^(R*k)

  // Idle lanes (past the last whole row group) repeat the last group's rows.
  const int gq = (int)ra.f_lpr.div((uint32_t)lane);
  const int ds = lane - gq * lpr;
  const bool idle = gq >= GW;
  const int gw = idle ? GW - 1 : gq;
  const int g = wave * GW + gw;
  const int ch = vec_channel<VW>(vec0 + ds, D);
  const int64_t rbase = row0 + (int64_t)g * R;

  // Decay factor and carry-in first, unconditionally (see ChunkScan::load).
  const float lam = a.lam[p.h];
  float init[DQ];
#pragma unroll
  for (int q = 0; q < DQ; ++q) {
    const int d = lane + 64 * q < S ? lane + 64 * q : S - 1;
    const bool has = chunk == 0 && a.init != nullptr;
    const float* ip = has ? a.init + (int64_t)p.bh * a.D + vec_channel<VW>(vec0 + d / VW, D) + d % VW : a.lam;
    const float v = *ip;
    init[q] = has ? v : 0.0f;
  }
  uint4 raw[R];
  {
    const TI* vp = static_cast<const TI*>(a.V) + p.b * a.vb + p.h * a.vh + ch;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t r = rbase + i < a.N ? rbase + i : a.N - 1;
      raw[i] = load16_any(vp + r * a.vn);
    }
  }

  // Tables, while the rows are in flight.
  for (int k = tid; k <= G; k += NTH) pw[k] = pow_like_torch(lam, (int64_t)k * R);
  for (int r = tid; r < L; r += NTH) {
    if (row0 + r < a.N) rz[r] = 1.0f / (R == 8 ? z_of_fast(lam, a.t_offset + row0 + r) : z_of(lam, a.t_offset + row0 + r));
  }
  float acc[VW];
#pragma unroll
  for (int j = 0; j < VW; ++j) acc[j] = 0.0f;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    float v[VW];
    unpack16<TI>(raw[i], v);
#pragma unroll
    for (int j = 0; j < VW; ++j) acc[j] = __builtin_fmaf(lam, acc[j], v[j]);
  }
  __syncthreads();  // tables

  // Inclusive scan over the wavefront's row groups.
  for (int K = 1; K < GW; K *= 2) {
    const float m = pw[K];
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      const float o = __shfl_up(acc[j], K * lpr, 64);
      if (gw >= K) acc[j] = __builtin_fmaf(m, o, acc[j]);
    }
  }
  if (!idle && gw == GW - 1) {
#pragma unroll
    for (int j = 0; j < VW; ++j) wt[wave * S + ds * VW + j] = acc[j];
  }
#pragma unroll
  for (int j = 0; j < VW; ++j) {
    const float o = __shfl_up(acc[j], lpr, 64);
    acc[j] = gw > 0 ? o : 0.0f;
  }
  __syncthreads();

  // Carry into the chunk (see ChunkScan::scan_chunk).
  const float mW = pw[GW];
  bool poisoned = false;
  if (wave == 0) {
    const float mL = pw[G];
    const unsigned tag_agg = tag_of(eh.epoch, 0u), tag_inc = tag_of(eh.epoch, 1u);
    poisoned = __builtin_amdgcn_readfirstlane(eh.err) != 0;
    u64* const base = multi ? a.flags + (int64_t)stream * a.nchunk * S : nullptr;
    float agg[DQ], carry[DQ];
#pragma unroll
    for (int q = 0; q < DQ; ++q) {
      const int d = lane + 64 * q;
      agg[q] = 0.0f;
      carry[q] = init[q];
      if (d < S) {
#pragma unroll
        for (int w = 0; w < NW; ++w) agg[q] = __builtin_fmaf(mW, agg[q], wt[w * S + d]);
        if (chunk > 0 && !last) publish(base + (int64_t)chunk * S + d, tag_agg, agg[q]);
      }
    }
    if (poisoned) {
#pragma unroll
      for (int q = 0; q < DQ; ++q) carry[q] = __builtin_nanf("");
    } else if (chunk > 0) {
      look_back_rows<W, DQ>(base, chunk, S, tag_agg, tag_inc, mL, a.hdr, a.spin_limit, carry);
    }
#pragma unroll
    for (int q = 0; q < DQ; ++q) {
      const int d = lane + 64 * q;
      if (d < S) {
        if (multi && !last) publish(base + (int64_t)chunk * S + d, tag_inc, __builtin_fmaf(mL, carry[q], agg[q]));
        sm_carry[d] = carry[q];
      }
    }
  }
  // Training forward: the backward's row terms (see ChunkScan::scan_chunk).
  if (a.rowtab && p.b == 0 && p.grp == 0 && wave > 0) {
    for (int r = tid - 64; r < L; r += NTH - 64) {
      const int64_t row = row0 + r;
      if (row < a.N) {
        const int64_t t = a.t_offset + row;
        float x, y;
        bwd_row_terms(lam, t + 1, ipow_f64((double)lam, t), x, y);
        a.rowtab[p.h * a.N + row] = make_float2(x, y);
      }
    }
  }
  __syncthreads();

  // The epoch's advance (see ChunkScan::scan_chunk).
  if (multi && last && tid == 0 && !poisoned) {
    if (a.nstream <= kFwdPerStreamCount)
      count_done(a.hdr, (unsigned)a.nstream, eh.epoch);
    else
      count_done_2(a.hdr, (unsigned)a.nstream, (unsigned)stream, eh.epoch);
  }

  // The lane's true start state, then its rows again.
  float st[VW];
  {
    float ew[VW];
#pragma unroll
    for (int j = 0; j < VW; ++j) ew[j] = 0.0f;
    for (int w = 0; w < wave; ++w) {
#pragma unroll
      for (int j = 0; j < VW; ++j) ew[j] = __builtin_fmaf(mW, ew[j], wt[w * S + ds * VW + j]);
    }
    const float mg = pw[g], mgw = pw[gw];
#pragma unroll
    for (int j = 0; j < VW; ++j)
      st[j] = __builtin_fmaf(mg, sm_carry[ds * VW + j], __builtin_fmaf(mgw, ew[j], acc[j]));
  }
  if (idle) return;
  TO* const op = static_cast<TO*>(a.out) + p.b * a.ob + p.h * a.oh + ch + rbase * a.on;
  const int64_t c0 = (int64_t)p.bh * a.D + ch;
  const int nvalid = a.N - rbase >= R ? R : (a.N - rbase > 0 ? (int)(a.N - rbase) : 0);
  const int64_t fr = a.N - 1 - rbase;
  const int ifin = a.fin != nullptr && fr >= 0 && fr < R ? (int)fr : -1;
  float rzl[R];
#pragma unroll
  for (int k = 0; k < R / 4; ++k) {
    const float4 q = *reinterpret_cast<const float4*>(&rz[g * R + 4 * k]);
    rzl[4 * k] = q.x;
    rzl[4 * k + 1] = q.y;
    rzl[4 * k + 2] = q.z;
    rzl[4 * k + 3] = q.w;
  }
  auto row = [&](int i) {
    float v[VW], y[VW];
    opaque(raw[i]);
    unpack16<TI>(raw[i], v);
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      st[j] = __builtin_fmaf(lam, st[j], v[j]);
      y[j] = st[j] * rzl[i];
    }
    store_any<TO, VW, NT>(op + (int64_t)i * a.on, y);
    if constexpr (THR) {
      if (i >= 2) wait_vmcnt<2 * (VW * (int)sizeof(TO) / 16)>();
    }
  };
  if (nvalid == R && (ifin < 0 || ifin == R - 1)) {
#pragma unroll
    for (int i = 0; i < R; ++i) row(i);
    if (ifin == R - 1) {
#pragma unroll
      for (int j = 0; j < VW; ++j) a.fin[c0 + j] = st[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i < nvalid) {
        row(i);
        if (i == ifin) {
#pragma unroll
          for (int j = 0; j < VW; ++j) a.fin[c0 + j] = st[j];
        }
      }
    }
  }
  if (a.states) {
    const int64_t e = rbase + R;  // st is the state at row e - 1
    if (e < a.N && e % a.state_rows == 0) {
      float* sp = a.states + ((int64_t)p.bh * a.nsaved + e / a.state_rows) * a.D + ch;
#pragma unroll
      for (int j = 0; j < VW; ++j) sp[j] = st[j];
    }
  }
}

// Chunk shape: 4 wavefronts of 16 rows per lane; 8 rows for grids that would
// leave much of the device idle (the limit of kdecay.hip's chunk_shape) and for
// sequences that an 8-row chunk holds; 8 wavefronts of 8 rows for small grids of
// long chains (half the hops a carry takes).
constexpr int64_t kRowsSmallGrid = 416;
constexpr int64_t kRowsLongChain = 64;

struct RowShape {
  int R, NW;
};

int64_t rows_chunk(const RowSplit& s, RowShape c) { return (int64_t)c.NW * (64 / s.lpr) * c.R; }

RowShape rows_shape(const RowSplit& s, int64_t B, int64_t H, int64_t N) {
  const int64_t L = rows_chunk(s, RowShape{16, 4}), L8 = L / 2;
  if (N > L8 && (N + L - 1) / L * B * H * s.ng > kRowsSmallGrid) return RowShape{16, 4};
  return RowShape{8, (N + L8 - 1) / L8 >= kRowsLongChain ? 8 : 4};
}

template <typename TI, typename TO, bool NT>
int launch_rows_nt(const RowScanArgs& ra, int64_t grid, RowShape c, hipStream_t s) {
  const ScanArgs& a = ra.s;
  const int G = c.NW * ra.gw;
  const size_t lds = sizeof(float) * ((size_t)G * c.R + (size_t)(c.NW + 1) * ra.slots + G + 1);
  // The look-back windows as launch_chunked chooses them: wide where few
  // streams make long chains in one round, narrow in several rounds (four
  // workgroups per CU, by registers).
  if (c.NW == 8) {
    hipLaunchKernelGGL((scan_rows<TI, TO, 8, 8, 16, 4, false, NT>), dim3((unsigned)grid), dim3(512), lds, s, ra);
  } else if (c.R == 8) {
    auto* const k = a.nchunk > 16 ? scan_rows<TI, TO, 8, 4, 16, 4, false, NT> : scan_rows<TI, TO, 8, 4, 4, 4, false, NT>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(256), lds, s, ra);
  } else {
    const int64_t resident = 4 * (int64_t)cu_count();
    auto* const k = resident > 0 && grid > resident ? scan_rows<TI, TO, 16, 4, kWRounds, 4, false, NT>
                                                    : scan_rows<TI, TO, 16, 4, kW, 4, true, NT>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(256), lds, s, ra);
  }
  return hip_check("scan_rows launch");
}

// Whether every row piece that a workgroup stores is whole 64-byte pieces
// (store16_any): strides in elements of es bytes.
bool whole_pieces(const void* p, int64_t sb, int64_t sh, int64_t sn, int64_t D, int64_t es, int lpr) {
  return ((uintptr_t)p | (uintptr_t)(sb * es) | (uintptr_t)(sh * es) | (uintptr_t)(sn * es) | (uintptr_t)(D * es) |
          (uintptr_t)(lpr * 16)) % 64 == 0;
}

template <typename TI, typename TO>
int launch_rows(const RowScanArgs& ra, int64_t grid, RowShape c, hipStream_t s) {
  // fp32 outputs of a 2-byte V are stored through the cache either way.
  if constexpr (sizeof(TI) == sizeof(TO)) {
    const ScanArgs& a = ra.s;
    if (whole_pieces(a.out, a.ob, a.oh, a.on, a.D, sizeof(TO), ra.lpr))
      return launch_rows_nt<TI, TO, true>(ra, grid, c, s);
  }
  return launch_rows_nt<TI, TO, false>(ra, grid, c, s);
}

}  // namespace kd

using namespace kd;

extern "C" {

size_t kdecay_scan_rows_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t D, int v_dtype) {
  if (B <= 0 || H <= 0 || N <= 0 || !fwd_dtype_ok(v_dtype)) return 0;
  const RowSplit s = row_split(v_dtype, D);
  if (!s.ok) return 0;
  const int64_t L = rows_chunk(s, rows_shape(s, B, H, N));
  const int64_t nchunk = (N + L - 1) / L;
  if (nchunk <= 1) return 0;
  return kHeaderBytes + (size_t)(B * H * s.ng * nchunk * s.lpr * (16 / elem_size(v_dtype))) * sizeof(u64);
}

int kdecay_scan_fwd_rows(const void* V, int v_dtype, const int64_t* v_strides, void* out, int out_dtype,
                         const int64_t* out_strides, const float* lam, const float* init_state,
                         float* final_state, int64_t B, int64_t H, int64_t N, int64_t D, int64_t t_offset,
                         void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_scan_args(V, v_dtype, v_strides, out, out_dtype, out_strides, lam, B, H, N, D);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (B * H * D == 0) return 0;
  if (N == 0) return empty_final_state(init_state, final_state, B * H * D, s);
  const RowSplit sp = row_split(v_dtype, D);
  if (!sp.ok) return fail(KDECAY_ESHAPE, "head dim D=%lld: no split into 16-byte vectors", (long long)D);
  if (v_strides[3] != 1 || out_strides[3] != 1) return fail(KDECAY_ELAYOUT, "channel (d) stride must be 1");
  if ((uintptr_t)V % elem_size(v_dtype) || (uintptr_t)out % elem_size(out_dtype))
    return fail(KDECAY_ELAYOUT, "V and out must be aligned to their elements");
  const RowShape shape = rows_shape(sp, B, H, N);
  const int64_t L = rows_chunk(sp, shape);
  const int64_t nchunk = (N + L - 1) / L, nstream = B * H * sp.ng, grid = nchunk * nstream;
  if (grid > 0x7fffffffLL) return fail(KDECAY_EINVAL, "problem too large (%lld chunks)", (long long)grid);
  const size_t need = kdecay_scan_rows_workspace_bytes(B, H, N, D, v_dtype);
  if (need && (!workspace || workspace_bytes < need))
    return fail(KDECAY_EWORKSPACE, "workspace of %zu bytes required, %zu given", need, workspace_bytes);
  if (need && ((uintptr_t)workspace & 255u)) return fail(KDECAY_EWORKSPACE, "workspace must be 256-byte aligned");

  RowScanArgs ra;
  ScanArgs& a = ra.s;
  a.V = V;
  a.out = out;
  a.lam = lam;
  a.init = init_state;
  a.fin = final_state;
  a.vb = v_strides[0];
  a.vh = v_strides[1];
  a.vn = v_strides[2];
  a.ob = out_strides[0];
  a.oh = out_strides[1];
  a.on = out_strides[2];
  a.H = H;
  a.N = N;
  a.t_offset = t_offset;
  a.D = D;
  a.ng = sp.ng;
  a.nchunk = (int)nchunk;
  a.nstream = (int)nstream;
  a.f_nstream = make_fastdiv((uint32_t)nstream);
  a.f_ng = make_fastdiv((uint32_t)sp.ng);
  a.f_H = make_fastdiv((uint32_t)H);
  a.hdr = nchunk > 1 ? static_cast<unsigned*>(workspace) : nullptr;
  a.flags = nchunk > 1 ? reinterpret_cast<u64*>(static_cast<char*>(workspace) + kHeaderBytes) : nullptr;
  a.spin_limit = spin_limit();
  a.state_rows = 0;
  a.nsaved = 0;
  a.states = nullptr;
  a.rowtab = nullptr;
  ra.lpr = sp.lpr;
  ra.gw = 64 / sp.lpr;
  ra.slots = sp.lpr * (16 / elem_size(v_dtype));
  ra.f_lpr = make_fastdiv((uint32_t)sp.lpr);
  switch (v_dtype) {
    case KDECAY_F32: return launch_rows<float, float>(ra, grid, shape, s);
    case KDECAY_F64: return launch_rows<double, double>(ra, grid, shape, s);
    case KDECAY_BF16:
      return out_dtype == KDECAY_BF16 ? launch_rows<__bf16, __bf16>(ra, grid, shape, s)
                                      : launch_rows<__bf16, float>(ra, grid, shape, s);
    default:
      return out_dtype == KDECAY_F16 ? launch_rows<_Float16, _Float16>(ra, grid, shape, s)
                                     : launch_rows<_Float16, float>(ra, grid, shape, s);
  }
}

}  // extern "C"
