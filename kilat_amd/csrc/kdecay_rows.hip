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

int row_slots(const RowSplit& s, int v_dtype) { return s.lpr * (16 / elem_size(v_dtype)); }

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
    if (row0 + r < a.N) rz[r] = 1.0f / (R <= 8 ? z_of_fast(lam, a.t_offset + row0 + r) : z_of(lam, a.t_offset + row0 + r));
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

// --------------------------------------------------------------------------
// Backward
// --------------------------------------------------------------------------
// As scan_bwd (kdecay.hip; the sums and their names are explained there):
// chunks from the end of the sequence, one forward sweep over V and gy from
// the saved state, the reverse look-back, and a dV pass over gy.  Channels a
// row's last vector shares with the one before it are computed in both, but
// count once in dlam: the later vector's copy of V and of the incoming state is
// zeroed, which zeroes every term of dlam that the lane adds for them, while
// its dV depends on gy alone.  A gy there that is not finite makes dlam NaN
// (infinity times zero) where the sum alone might be an infinity.  Summing such
// lanes once more without the copies cost every lane registers the kernels do not
// have to spare, whole-vector head dims included: 500 training passes at 1.027 of
// the time (1.135 at most), and at 1.023 (1.112) channel by channel.
struct RowBwdArgs {
  BwdArgs s;  // ng: streams per head; flags: [nstream][nchunk][slots] words
  int lpr, gw, slots;
  FastDiv f_lpr;
};

// Channels [ch, ch + VW) of a vector with the first `skip` zeroed.
template <typename T>
__device__ __forceinline__ uint4 skip_mask(int skip) {
  unsigned m[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (sizeof(T) == 2)
      m[k] = (2 * k < skip ? 0u : 0xffffu) | (2 * k + 1 < skip ? 0u : 0xffff0000u);
    else
      m[k] = k < skip ? 0u : ~0u;
  }
  return make_uint4(m[0], m[1], m[2], m[3]);
}

template <typename T, int R, int NW, int W, int WPE, bool NT>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
void scan_rows_bwd(RowBwdArgs ra) {
  constexpr int VW = 16 / (int)sizeof(T);
  constexpr int NTH = NW * 64;  // threads
  constexpr int DQ = (kMaxLanes * VW + 63) / 64;
  constexpr int TS = R + 1;  // table entries per row group: padded, see ChunkBwd::Smem
  constexpr int NR = 2;      // rows of the table per thread whose saved terms are loaded early
  const BwdArgs& a = ra.s;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int lpr = ra.lpr, GW = ra.gw, S = ra.slots;
  const int G = NW * GW, L = G * R, KS = S + 1;
  const int D = (int)a.D;
  const bool multi = a.nchunk > 1;
  const int item = blockIdx.x;
  // rc: position from the end.  Consecutive streams on one XCD (rows_pos), but
  // in the last row of items (chunk 0), whose order reduce_head relies on.
  const int rc = (int)a.f_nstream.div((uint32_t)item);
  const int chunk = a.nchunk - 1 - rc;
  int stream = item - rc * a.nstream;
  if (chunk > 0) {
    const int j = rotated_stream(stream, (int)a.f_nstream.mod((uint32_t)chunk), a.nstream);
    const int x = j % kXcds, most = a.nstream % kXcds;
    stream = x * (a.nstream / kXcds) + (x < most ? x : most) + j / kXcds;
  }
  const int bh = (int)a.f_ng.div((uint32_t)stream), grp = stream - bh * a.ng;
  const int b = (int)a.f_H.div((uint32_t)bh), h = bh - b * (int)a.H;
  const int64_t row0 = (int64_t)chunk * L;
  const int vec0 = grp * lpr;

  extern __shared__ float4 smem4[];
  float4* const rt4 = smem4;                                 // [G * TS] row terms (ChunkBwd::Smem)
  double* const red = reinterpret_cast<double*>(rt4 + G * TS);  // [NW]
  float* const kq = reinterpret_cast<float*>(red + NW);      // [G][KS]
  float* const wt = kq + G * KS;                             // [NW][S] forward wavefront totals
  float* const rt = wt + NW * S;                             // [NW][S] reverse wavefront totals
  float* const carry_s = rt + NW * S;                        // [S]
  float* const carry_g = carry_s + S;                        // [S]
  float* const gfin = carry_g + S;                           // [S]
  float* const pw = gfin + S;                                // [G + 1] lam^(R*k)
  float* const pl = pw + G + 1;                              // [R + 1] lam^i

  const int gq = (int)ra.f_lpr.div((uint32_t)lane);
  const int ds = lane - gq * lpr;
  const bool idle = gq >= GW;
  const int gw = idle ? GW - 1 : gq;
  const int g = wave * GW + gw;
  const int gr = g * R;  // the lane's first row within the chunk
  const int ch = vec_channel<VW>(vec0 + ds, D);
  const float lam = a.lam[h];

  // Slots tid (< S <= NTH: at most 128, or 64 with one wavefront): the state before the chunk's first row (zero
  // for the second copy of a channel) and the final-state gradient.  Loaded
  // before the rows and unconditionally (see ChunkBwd::run).
  float cs, cf;
  {
    const int d = tid < S ? tid : S - 1;
    const int c = vec_channel<VW>(vec0 + d / VW, D) + d % VW;
    const int64_t at = (int64_t)bh * a.D + c;
    const float* cp = chunk > 0 ? a.states + ((int64_t)bh * a.nsaved + chunk) * a.D + c : (a.init ? a.init + at : a.lam);
    const bool fin = rc == 0 && a.gfin != nullptr;
    const float* fp = fin ? a.gfin + at : a.lam;
    cs = *cp;
    cf = *fp;
    if ((chunk == 0 && !a.init) || c < (vec0 + d / VW) * VW) cs = 0.0f;
    if (!fin) cf = 0.0f;
  }
  float tx[NR], ty[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    const int rr = tid + k * NTH < L ? tid + k * NTH : L - 1;
    const int64_t r = row0 + rr < a.N ? row0 + rr : a.N - 1;
    const float* tp = a.rowtab ? reinterpret_cast<const float*>(a.rowtab + h * a.N + r) : a.lam;
    tx[k] = tp[0];
    ty[k] = (a.rowtab ? tp + 1 : a.lam)[0];
  }

  // Rows past the end read row N-1 and are zeroed below.
  const int64_t left = a.N - 1 - row0;  // the chunk's last row inside the sequence
  const int li = left - gr < R - 1 ? (int)(left - gr) : R - 1;
  uint4 rv[R], rg[R];
  {
    const T* vp = static_cast<const T*>(a.V) + b * a.vb + h * a.vh + ch;
    const T* gp = static_cast<const T*>(a.gy) + b * a.gb + h * a.gh + ch;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t r = row0 + gr + i < a.N ? row0 + gr + i : a.N - 1;
      rv[i] = load16_any(vp + r * a.vn);
      rg[i] = load16_any(gp + r * a.gn);
    }
  }

  __syncthreads();
  for (int k = tid; k <= G; k += NTH) pw[k] = pow_like_torch(lam, (int64_t)k * R);
  if (tid >= NTH - (R + 1)) pl[tid - (NTH - (R + 1))] = pow_like_torch(lam, (int64_t)(tid - (NTH - (R + 1))));
  {
    static_assert(NTH % R == 0, "rows of a thread share their index in the lane");
    const int i = tid % R;
    const float p = pow_like_torch(lam, i);
    const float p1 = p * lam;
    auto entry = [&](int r, float x, float y) {
      const float w = x * p;
      rt4[r + r / R] = make_float4(x, y, __builtin_fmaf(w, (float)(i + 1), y * p1), w);
    };
    if (a.rowtab) {
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        const int r = tid + k * NTH;
        const bool in = row0 + r < a.N;
        if (r < L) entry(r, in ? tx[k] : 0.0f, in ? ty[k] : 0.0f);
      }
      for (int r = tid + NR * NTH; r < L; r += NTH) {  // fewer than 4 lanes per row
        const bool in = row0 + r < a.N;
        const float2 t = in ? a.rowtab[h * a.N + row0 + r] : make_float2(0.0f, 0.0f);
        entry(r, t.x, t.y);
      }
    } else {
      for (int r = tid; r < L; r += NTH) {
        const int64_t t = a.t_offset + row0 + r;
        float x = 0.0f, y = 0.0f;
        if (row0 + r < a.N) bwd_row_terms(lam, t + 1, ipow_f64((double)lam, t), x, y);
        entry(r, x, y);
      }
    }
  }
  if (tid < S) {
    carry_s[tid] = cs;
    gfin[tid] = cf;
  }
  __syncthreads();  // tables

  // Rows past the end, and second copies of channels of V.
  const int skip = (vec0 + ds) * VW - ch < VW ? (vec0 + ds) * VW - ch : VW;
  if (rc == 0 || D % VW != 0 || a.ng * lpr * VW != D) {
    const uint4 m = skip_mask<T>(skip);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const bool in = i <= li;
      rv[i].x = in ? rv[i].x & m.x : 0u;
      rv[i].y = in ? rv[i].y & m.y : 0u;
      rv[i].z = in ? rv[i].z & m.z : 0u;
      rv[i].w = in ? rv[i].w & m.w : 0u;
      rg[i].x = in ? rg[i].x : 0u;
      rg[i].y = in ? rg[i].y : 0u;
      rg[i].z = in ? rg[i].z : 0u;
      rg[i].w = in ? rg[i].w : 0u;
    }
  }
  const int fin_i = rc == 0 && a.gfin != nullptr && li >= 0 && gr + li == left ? li : -1;

  // Forward sweep (ChunkBwd::sweep_fwd): with 16 rows it takes the gy-only sums
  // (qz, ra_) of rows F0 and later, and rows below F0 get a pass of their own
  // once V's registers are free.
  constexpr int F0 = R <= 8 ? 0 : R / 2;
  float sl[VW], wl[VW], qz[VW], ra_[VW], dq = 0.0f;
#pragma unroll
  for (int j = 0; j < VW; ++j) sl[j] = wl[j] = qz[j] = ra_[j] = 0.0f;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const float4 t = rt4[g * TS + i];
    float v[VW], gv[VW];
    unpack16<T>(rv[i], v);
    unpack16<T>(rg[i], gv);
    float pws = 0.0f, ps = 0.0f;
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      wl[j] = __builtin_fmaf(lam, wl[j], sl[j]);
      sl[j] = __builtin_fmaf(lam, sl[j], v[j]);
      pws = __builtin_fmaf(gv[j], wl[j], pws);
      ps = __builtin_fmaf(gv[j], sl[j], ps);
      if (i >= F0) {
        qz[j] = __builtin_fmaf(gv[j], t.z, qz[j]);
        ra_[j] = __builtin_fmaf(gv[j], t.w, ra_[j]);
      }
    }
    dq = __builtin_fmaf(t.x, pws, __builtin_fmaf(t.y, ps, dq));
    if (i == fin_i) {
#pragma unroll
      for (int j = 0; j < VW; ++j) dq = __builtin_fmaf(gfin[ds * VW + j], wl[j], dq);
    }
    pin(sl);
    pin(wl);
    asm volatile("" : "+v"(dq));
    if (i >= F0) {
      pin(qz);
      pin(ra_);
    }
  }
#pragma unroll
  for (int i = 0; i < F0; ++i) {
    const float2 t = *reinterpret_cast<const float2*>(&rt4[g * TS + i].z);
    float gv[VW];
    opaque(rg[i]);
    unpack16<T>(rg[i], gv);
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      qz[j] = __builtin_fmaf(gv[j], t.x, qz[j]);
      ra_[j] = __builtin_fmaf(gv[j], t.y, ra_[j]);
    }
    pin(qz);
    pin(ra_);
  }
  if (fin_i >= 0) {
    const float p = pl[fin_i];
    const float c = p * (float)(fin_i + 1);
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      const float gf = gfin[ds * VW + j];
      qz[j] = __builtin_fmaf(gf, c, qz[j]);
      ra_[j] = __builtin_fmaf(gf, p, ra_[j]);
    }
  }
  const EpochErr eh = read_epoch_v(a.hdr);
  const unsigned epoch = eh.epoch;

  // Scans over the wavefront's row groups, both directions.
  for (int K = 1; K < GW; K *= 2) {
    const float m = pw[K];
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      const float o = __shfl_up(sl[j], K * lpr, 64);
      const float p = __shfl_down(ra_[j], K * lpr, 64);
      if (gw >= K) sl[j] = __builtin_fmaf(m, o, sl[j]);
      if (gw + K < GW) ra_[j] = __builtin_fmaf(m, p, ra_[j]);
    }
  }
  if (!idle && gw == GW - 1) {
#pragma unroll
    for (int j = 0; j < VW; ++j) wt[wave * S + ds * VW + j] = sl[j];
  }
  if (gq == 0) {
#pragma unroll
    for (int j = 0; j < VW; ++j) rt[wave * S + ds * VW + j] = ra_[j];
  }
  float xin[VW], rin[VW];
#pragma unroll
  for (int j = 0; j < VW; ++j) {
    const float o = __shfl_up(sl[j], lpr, 64);
    xin[j] = gw > 0 ? o : 0.0f;
    const float p = __shfl_down(ra_[j], lpr, 64);
    rin[j] = gw < GW - 1 ? p : 0.0f;
  }
  __syncthreads();

  // Reverse carry of the chunk (wavefront 0).
  const float mW = pw[GW];
  float cg[DQ];
  bool poisoned = false;
  if (wave == 0) {
    const float mL = pw[G];
    const unsigned tag_agg = tag_of(epoch, 0u), tag_inc = tag_of(epoch, 1u);
    u64* const base = multi ? a.flags + (int64_t)stream * a.nchunk * S : nullptr;
    float agg[DQ];
#pragma unroll
    for (int q = 0; q < DQ; ++q) {
      const int d = lane + 64 * q;
      agg[q] = 0.0f;
      cg[q] = 0.0f;
      if (d < S) {
#pragma unroll
        for (int w = NW - 1; w >= 0; --w) agg[q] = __builtin_fmaf(mW, agg[q], rt[w * S + d]);
        if (rc > 0 && chunk > 0) publish(base + (int64_t)rc * S + d, tag_agg, agg[q]);
      }
    }
    poisoned = __builtin_amdgcn_readfirstlane(eh.err) != 0;
    if (poisoned) {
#pragma unroll
      for (int q = 0; q < DQ; ++q) cg[q] = __builtin_nanf("");
    } else if (rc > 0) {
      look_back_rows<W, DQ>(base, rc, S, tag_agg, tag_inc, mL, a.hdr, a.spin_limit, cg);
    }
#pragma unroll
    for (int q = 0; q < DQ; ++q) {
      const int d = lane + 64 * q;
      if (d < S) {
        if (multi && chunk > 0) publish(base + (int64_t)rc * S + d, tag_inc, __builtin_fmaf(mL, cg[q], agg[q]));
        carry_g[d] = cg[q];
      }
    }
  }

  // s_in, g_out without the chunk's carry, and the lane's share of dlam, in
  // double from here (see ChunkBwd::run).
  const float mg = pw[g], mgw = pw[gw];
  const float mr = pw[G - 1 - g], mrw = pw[GW - 1 - gw];
  const float rlr = (float)R * pw[1];
  float gh0[VW];
  double dsum = idle ? 0.0 : (double)dq;
  {
    float ew[VW], er[VW];
#pragma unroll
    for (int j = 0; j < VW; ++j) ew[j] = er[j] = 0.0f;
    for (int w = 0; w < wave; ++w) {
#pragma unroll
      for (int j = 0; j < VW; ++j) ew[j] = __builtin_fmaf(mW, ew[j], wt[w * S + ds * VW + j]);
    }
    for (int w = NW - 1; w > wave; --w) {
#pragma unroll
      for (int j = 0; j < VW; ++j) er[j] = __builtin_fmaf(mW, er[j], rt[w * S + ds * VW + j]);
    }
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      const float sin = __builtin_fmaf(mg, carry_s[ds * VW + j], __builtin_fmaf(mgw, ew[j], xin[j]));
      gh0[j] = __builtin_fmaf(mrw, er[j], rin[j]);
      const float x = __builtin_fmaf(sin, rlr, lam * wl[j]);  // Q2 + s_in R lam^R
      if (!idle) {
        dsum = __builtin_fma((double)gh0[j], (double)x, __builtin_fma((double)sin, (double)qz[j], dsum));
        kq[g * KS + ds * VW + j] = mr * x;
      }
    }
  }
  dsum = wave_sum_f64(dsum);
  if (lane == 0) red[wave] = dsum;
  __syncthreads();  // carry_g, kq, red

  if (wave == 0) {
    double e = 0.0;
#pragma unroll
    for (int q = 0; q < DQ; ++q) {
      const int d = lane + 64 * q;
      if (d < S) {
        double kc = 0.0;
        for (int r = 0; r < G; ++r) kc += (double)kq[r * KS + d];
        e = __builtin_fma((double)cg[q], kc, e);
      }
    }
    e = wave_sum_f64(e);
    if (lane == 0) {
      double sum = e;
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += red[w];
      publish(a.partial + (int64_t)rc * a.nstream + stream, tag_of(epoch, 0u), (float)sum);
    }
  }
  if (a.per_stream && chunk == 0 && tid == 0 && !poisoned) count_done(a.hdr, (unsigned)a.nstream, epoch);

  // dV with the true carry.
  float gn[VW];
#pragma unroll
  for (int j = 0; j < VW; ++j) gn[j] = __builtin_fmaf(mr, carry_g[ds * VW + j], gh0[j]);
  T* const dp = static_cast<T*>(a.dv) + b * a.db + h * a.dh + ch + (row0 + gr) * a.dn;
#pragma unroll
  for (int i = R - 1; i >= 0; --i) {
    float gv[VW];
    opaque(rg[i]);
    unpack16<T>(rg[i], gv);
    const float rz = rt4[g * TS + i].x;
#pragma unroll
    for (int j = 0; j < VW; ++j) gn[j] = __builtin_fmaf(lam, gn[j], gv[j] * rz);
    if (i == fin_i) {
#pragma unroll
      for (int j = 0; j < VW; ++j) gn[j] += gfin[ds * VW + j];
    }
    if (i <= li && !idle) store_any<T, VW, NT>(dp + (int64_t)i * a.dn, gn);
    pin(gn);
  }
  if (a.dinit && row0 + gr == 0 && !idle) {
#pragma unroll
    for (int j = 0; j < VW; ++j) a.dinit[(int64_t)bh * a.D + ch + j] = lam * gn[j];
  }

  // The head's sum and the epoch's advance (see ChunkBwd::run).
  if (rc == a.nchunk - 1 && b == a.B - 1 && grp == a.ng - 1)
    reduce_head<false>(a, h, epoch, poisoned);
  else if (!a.per_stream && item + kXcds >= (int)gridDim.x && tid == 0 && !poisoned)
    count_done(a.hdr, (unsigned)a.ndone, epoch);
}

// Chunk shape: 4 wavefronts of 16 rows per lane; 8 rows for grids that would
// leave much of the device idle (the limit of kdecay.hip's chunk_shape); 8
// wavefronts of 8 rows for small grids of long chains (half the hops a carry
// takes); short sequences take the smallest of 4 rows x 1 wavefront, 8 x 1, 4 x
// 4 and 8 x 4 that holds them (chunk_shape).
constexpr int64_t kRowsSmallGrid = 416;
constexpr int64_t kRowsLongChain = 64;

struct RowShape {
  int R, NW;
};

int64_t rows_chunk(const RowSplit& s, RowShape c) { return (int64_t)c.NW * (64 / s.lpr) * c.R; }

RowShape rows_shape(const RowSplit& s, int64_t B, int64_t H, int64_t N) {
  const int64_t gw = 64 / s.lpr;
  if (N <= 4 * gw) return RowShape{4, 1};
  if (N <= 8 * gw) return RowShape{8, 1};
  if (N <= 16 * gw) return RowShape{4, 4};
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
  if (c.NW == 1 || c.R == 4) {  // one chunk per stream
    auto* const k = c.R == 8    ? scan_rows<TI, TO, 8, 1, 1, 4, false, NT>
                    : c.NW == 1 ? scan_rows<TI, TO, 4, 1, 1, 4, false, NT>
                                : scan_rows<TI, TO, 4, 4, 1, 4, false, NT>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(c.NW * 64), lds, s, ra);
  } else if (c.NW == 8) {
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

// Backward chunk shape, 4 wavefronts: 8 rows per lane (four workgroups per CU);
// 4 rows for grids that would leave much of the device idle; 16 rows (three per
// CU) for grids that fill most of one round of them.  Measured (us, 16 / 8 / 4
// rows; chunks at 16 rows): bf16 D=96 B=8 H=8 N=3001 (640) 29.7 / 32.4 / 37.7,
// fp16 D=80 B=8 H=16 N=2047 (768) 35.2 / 37.1 / 41.4, bf16 D=100 B=8 H=12 N=2048
// (768) 31.8 / 34.2 / 40.3, bf16 D=160 B=8 H=8 N=2048 (768) 35.5 / 37.2 / 41.3;
// but D=48 B=8 H=16 N=4096 (896) 46.6 / 41.5 / 47.4, D=24 B=8 H=12 N=4096 (384)
// 36.3 / 27.5 / 28.9, D=96 B=16 H=16 N=2048 (1792) 81.2 / 72.3 / 78.1, fp32 D=40
// B=4 H=16 N=2048 (384) 21.4 / 17.9 / 20.2, bf16 D=96 B=2 H=16 N=512 (64; 128 at
// 8 rows) - / 13.2 / 12.4, fp32 D=48 B=2 H=6 N=1024 - / 11.1 / 10.3.
constexpr int64_t kRowsBwdSmallGrid = 384;  // chunks of 8 rows per lane
constexpr int64_t kRowsBwdFullLo = 512;     // chunks of 16
constexpr int64_t kRowsBwdFullHi = 768;
// 16 rows only where three workgroups' LDS fits a CU: rows of one lane (8 bf16 or
// 4 fp32 channels) take 80 KB each, two to a CU, and run 8 rows instead.  300
// training passes of such rows with 513 to 768 chunks of 16: 0.90 of the time with
// 16 (0.75 to 1.00, one 1.06); bf16 D=8 B=284 H=1 N=4917 112.3 / 89.8 us, D=8 B=46
// H=6 N=4836 141.2 / 107.1, fp32 D=4 B=37 H=9 N=4754 149.7 / 115.9.
constexpr size_t kCuLds = 160 << 10;

// Dynamic LDS of scan_rows_bwd (its layout is at the kernel's head).
size_t rows_bwd_lds(const RowSplit& s, RowShape c, int slots) {
  const int64_t G = (int64_t)c.NW * (64 / s.lpr), S = slots;
  return 16 * G * (c.R + 1) + 8 * c.NW + 4 * (G * (S + 1) + 2 * c.NW * S + 3 * S + (G + 1) + (c.R + 1));
}

// Short sequences as the forward's, with one wavefront only where its 64 lanes
// hold a stream's channels (slots), and of 8 rows only for many streams
// (bwd_shape).
RowShape rows_bwd_shape(const RowSplit& s, int64_t B, int64_t H, int64_t N, int slots) {
  const int64_t gw = 64 / s.lpr;
  if (slots <= 64 && N <= 4 * gw) return RowShape{4, 1};
  if (slots <= 64 && N <= 8 * gw && B * H * s.ng > kRowsBwdSmallGrid) return RowShape{8, 1};
  if (N <= 16 * gw) return RowShape{4, 4};
  const int64_t L = rows_chunk(s, RowShape{8, 4}), n = B * H * s.ng;
  if (N <= L) return RowShape{8, 4};
  const int64_t grid16 = (N + 2 * L - 1) / (2 * L) * n;
  if (grid16 > kRowsBwdFullLo && grid16 <= kRowsBwdFullHi && 3 * rows_bwd_lds(s, RowShape{16, 4}, slots) <= kCuLds)
    return RowShape{16, 4};
  return RowShape{(N + L - 1) / L * n > kRowsBwdSmallGrid ? 8 : 4, 4};
}

template <typename T, bool NT>
int launch_rows_bwd_nt(const RowBwdArgs& ra, int64_t grid, RowShape c, hipStream_t s) {
  const BwdArgs& a = ra.s;
  const size_t lds = rows_bwd_lds(RowSplit{ra.lpr, a.ng, true}, c, ra.slots);
  // Windows as launch_bwd's: narrow in several rounds, else by chain length.
  const int64_t resident = 4 * (int64_t)cu_count();
  const bool rounds = resident > 0 && grid > resident;
  const int n = a.nchunk;
  if (c.NW == 1) {  // one chunk of one wavefront per stream
    auto* const k1 = c.R == 8 ? scan_rows_bwd<T, 8, 1, 1, 4, NT> : scan_rows_bwd<T, 4, 1, 1, 4, NT>;
    hipLaunchKernelGGL(k1, dim3((unsigned)grid), dim3(64), lds, s, ra);
    return hip_check("scan_rows_bwd launch");
  }
  auto* const k = c.R == 16 ? (n > 8 ? scan_rows_bwd<T, 16, 4, 8, 3, NT> : scan_rows_bwd<T, 16, 4, kW, 3, NT>)
                  : c.R == 8 ? (rounds  ? scan_rows_bwd<T, 8, 4, kWRounds, 4, NT>
                                : n > 8 ? scan_rows_bwd<T, 8, 4, 8, 4, NT>
                                        : scan_rows_bwd<T, 8, 4, kW, 4, NT>)
                             : (n > 32  ? scan_rows_bwd<T, 4, 4, 16, 3, NT>
                                : n > 8 ? scan_rows_bwd<T, 4, 4, 8, 4, NT>
                                        : scan_rows_bwd<T, 4, 4, kW, 4, NT>);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(c.NW * 64), lds, s, ra);
  return hip_check("scan_rows_bwd launch");
}

template <typename T>
int launch_rows_bwd(const RowBwdArgs& ra, int64_t grid, RowShape c, hipStream_t s) {
  const BwdArgs& a = ra.s;
  return whole_pieces(a.dv, a.db, a.dh, a.dn, a.D, sizeof(T), ra.lpr) ? launch_rows_bwd_nt<T, true>(ra, grid, c, s)
                                                                      : launch_rows_bwd_nt<T, false>(ra, grid, c, s);
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
  return kHeaderBytes + (size_t)(B * H * s.ng * nchunk * row_slots(s, v_dtype)) * sizeof(u64);
}

static int rows_fwd_impl(const void* V, int v_dtype, const int64_t* v_strides, void* out, int out_dtype,
                         const int64_t* out_strides, const float* lam, const float* init_state,
                         float* final_state, int64_t B, int64_t H, int64_t N, int64_t D, int64_t t_offset,
                         void* workspace, size_t workspace_bytes, float* states, void* stream) {
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
  a.state_rows = rows_chunk(sp, rows_bwd_shape(sp, B, H, N, row_slots(sp, v_dtype)));
  a.nsaved = (N + a.state_rows - 1) / a.state_rows;
  a.states = a.nsaved > 1 ? states : nullptr;
  a.rowtab = a.states ? reinterpret_cast<float2*>(states + B * H * D * a.nsaved) : nullptr;
  // One wavefront's chunks hold sequences that are one backward chunk too: no
  // states (scan_rows writes the row terms from its other wavefronts).
  if (shape.NW == 1 && a.states) return fail(KDECAY_EINVAL, "no saving kernel of one wavefront");
  ra.lpr = sp.lpr;
  ra.gw = 64 / sp.lpr;
  ra.slots = row_slots(sp, v_dtype);
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

int kdecay_scan_fwd_rows(const void* V, int v_dtype, const int64_t* v_strides, void* out, int out_dtype,
                         const int64_t* out_strides, const float* lam, const float* init_state,
                         float* final_state, int64_t B, int64_t H, int64_t N, int64_t D, int64_t t_offset,
                         void* workspace, size_t workspace_bytes, void* stream) {
  return rows_fwd_impl(V, v_dtype, v_strides, out, out_dtype, out_strides, lam, init_state, final_state, B, H, N, D,
                       t_offset, workspace, workspace_bytes, nullptr, stream);
}

size_t kdecay_scan_rows_saved_states_floats(int64_t B, int64_t H, int64_t N, int64_t D, int v_dtype) {
  if (B <= 0 || H <= 0 || N <= 0 || !dtype_ok(v_dtype)) return 0;
  const RowSplit sp = row_split(v_dtype, D);
  if (!sp.ok) return 0;
  const int64_t Lb = rows_chunk(sp, rows_bwd_shape(sp, B, H, N, row_slots(sp, v_dtype)));
  const int64_t nsaved = (N + Lb - 1) / Lb;
  return nsaved <= 1 ? 0 : (size_t)(B * H * D * nsaved + 2 * H * N);
}

int kdecay_scan_fwd_rows_train(const void* V, int v_dtype, const int64_t* v_strides, void* out, int out_dtype,
                               const int64_t* out_strides, const float* lam, const float* init_state,
                               float* final_state, float* states, size_t states_floats, int64_t B, int64_t H,
                               int64_t N, int64_t D, int64_t t_offset, void* workspace, size_t workspace_bytes,
                               void* stream) {
  if (!dtype_ok(v_dtype) || !dtype_ok(out_dtype))
    return fail(KDECAY_EDTYPE, "training forward: dtype code (v=%d out=%d) not F32/BF16/F16", v_dtype, out_dtype);
  const size_t need = kdecay_scan_rows_saved_states_floats(B, H, N, D, v_dtype);
  if (need && (!states || states_floats < need))
    return fail(KDECAY_EINVAL, "states buffer of %zu floats required, %zu given", need, states_floats);
  return rows_fwd_impl(V, v_dtype, v_strides, out, out_dtype, out_strides, lam, init_state, final_state, B, H, N, D,
                       t_offset, workspace, workspace_bytes, states, stream);
}

size_t kdecay_scan_rows_bwd_workspace_bytes(int64_t B, int64_t H, int64_t N, int64_t D, int v_dtype) {
  if (B <= 0 || H <= 0 || N <= 0 || !dtype_ok(v_dtype)) return 0;
  const RowSplit sp = row_split(v_dtype, D);
  if (!sp.ok) return 0;
  const int64_t Lb = rows_chunk(sp, rows_bwd_shape(sp, B, H, N, row_slots(sp, v_dtype)));
  const int64_t nchunk = (N + Lb - 1) / Lb, nstream = B * H * sp.ng;
  const size_t flags = nchunk > 1 ? (size_t)(nstream * nchunk * row_slots(sp, v_dtype)) * sizeof(u64) : 0;
  return kHeaderBytes + flags + (size_t)(nstream * nchunk) * sizeof(u64);
}

int kdecay_scan_rows_bwd(const void* V, int v_dtype, const int64_t* v_strides, const void* gy,
                         const int64_t* gy_strides, void* dV, const int64_t* dv_strides, const float* lam,
                         const float* init_state, const float* states, const float* g_final, float* dlam,
                         float* d_init, int64_t B, int64_t H, int64_t N, int64_t D, int64_t t_offset,
                         void* workspace, size_t workspace_bytes, void* stream) {
  if (B < 0 || H < 0 || N < 0 || D < 0) return fail(KDECAY_EINVAL, "negative size");
  if (!dtype_ok(v_dtype)) return fail(KDECAY_EDTYPE, "unknown dtype code %d", v_dtype);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (B * H * D == 0) return 0;
  if (!lam || !dlam) return fail(KDECAY_EINVAL, "null pointer argument");
  if (N == 0) return empty_backward(g_final, d_init, dlam, B, H, D, s);
  if (!V || !gy || !dV || !v_strides || !gy_strides || !dv_strides) return fail(KDECAY_EINVAL, "null pointer argument");
  const RowSplit sp = row_split(v_dtype, D);
  if (!sp.ok) return fail(KDECAY_ESHAPE, "head dim D=%lld: no split into 16-byte vectors", (long long)D);
  if (v_strides[3] != 1 || gy_strides[3] != 1 || dv_strides[3] != 1)
    return fail(KDECAY_ELAYOUT, "channel (d) stride must be 1");
  const uintptr_t es = (uintptr_t)elem_size(v_dtype);
  if ((uintptr_t)V % es || (uintptr_t)gy % es || (uintptr_t)dV % es)
    return fail(KDECAY_ELAYOUT, "V, gy and dV must be aligned to their elements");
  const RowShape shape = rows_bwd_shape(sp, B, H, N, row_slots(sp, v_dtype));
  const int64_t Lb = rows_chunk(sp, shape);
  const int64_t nchunk = (N + Lb - 1) / Lb, nstream = B * H * sp.ng, grid = nchunk * nstream;
  if (grid > 0x7fffffffLL) return fail(KDECAY_EINVAL, "problem too large (%lld chunks)", (long long)grid);
  if (nchunk > 1 && !states) return fail(KDECAY_EINVAL, "saved states (kdecay_scan_fwd_rows_train) required");
  const size_t need = kdecay_scan_rows_bwd_workspace_bytes(B, H, N, D, v_dtype);
  if (!workspace || workspace_bytes < need)
    return fail(KDECAY_EWORKSPACE, "workspace of %zu bytes required, %zu given", need, workspace_bytes);
  if ((uintptr_t)workspace & 255u) return fail(KDECAY_EWORKSPACE, "workspace must be 256-byte aligned");

  RowBwdArgs ra;
  BwdArgs& a = ra.s;
  a.V = V;
  a.gy = gy;
  a.dv = dV;
  a.lam = lam;
  a.init = init_state;
  a.states = states;
  a.rowtab = nchunk > 1 ? reinterpret_cast<const float2*>(states + B * H * D * nchunk) : nullptr;
  a.gfin = g_final;
  a.dinit = d_init;
  a.dlam = dlam;
  a.vb = v_strides[0];
  a.vh = v_strides[1];
  a.vn = v_strides[2];
  a.gb = gy_strides[0];
  a.gh = gy_strides[1];
  a.gn = gy_strides[2];
  a.db = dv_strides[0];
  a.dh = dv_strides[1];
  a.dn = dv_strides[2];
  a.B = B;
  a.H = H;
  a.N = N;
  a.t_offset = t_offset;
  a.D = D;
  a.ng = sp.ng;
  a.nchunk = (int)nchunk;
  a.nstream = (int)nstream;
  a.nsaved = nchunk;
  a.f_nstream = make_fastdiv((uint32_t)nstream);
  a.f_ng = make_fastdiv((uint32_t)sp.ng);
  a.f_H = make_fastdiv((uint32_t)H);
  a.f_nchunk = make_fastdiv((uint32_t)nchunk);
  a.hdr = static_cast<unsigned*>(workspace);
  a.spin_limit = spin_limit();
  a.per_stream = nstream <= kBwdPerStreamCount;
  a.ndone = bwd_done_count(B, H, sp.ng, nchunk);
  const int slots = row_slots(sp, v_dtype);
  const size_t flag_bytes = nchunk > 1 ? (size_t)(nstream * nchunk * slots) * sizeof(u64) : 0;
  a.flags = nchunk > 1 ? reinterpret_cast<u64*>(static_cast<char*>(workspace) + kHeaderBytes) : nullptr;
  a.partial = reinterpret_cast<u64*>(static_cast<char*>(workspace) + kHeaderBytes + flag_bytes);
  a.slice = 0;
  a.nslice = 1;
  a.dlam_slices = nullptr;
  ra.lpr = sp.lpr;
  ra.gw = 64 / sp.lpr;
  ra.slots = slots;
  ra.f_lpr = make_fastdiv((uint32_t)sp.lpr);
  switch (v_dtype) {
    case KDECAY_F32: return launch_rows_bwd<float>(ra, grid, shape, s);
    case KDECAY_BF16: return launch_rows_bwd<__bf16>(ra, grid, shape, s);
    default: return launch_rows_bwd<_Float16>(ra, grid, shape, s);
  }
}

}  // extern "C"
