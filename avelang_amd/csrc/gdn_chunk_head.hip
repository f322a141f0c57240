// Forward chain of the chunked prefill, whole-head form (gfx950).
//
// One workgroup per (sequence or segment of one, v-head).  Compute wave w
// carries the 32 value columns 32 w .. 32 w + 31 of the head's fp32 state in
// VGPRs (every key row, 64 registers at K = 128) through the chunks of 64
// tokens and forms those columns' output too:
//     X = K S,  Y = V - e^G X,  vnew = Tb Y,  o = scale e^G (Q S) + P vnew,
//     S = e^G_last S + K^T (e^(G_last - G) vnew)
// with the row orders of the state-wave chain (gdn_chunk_chain.hip), in which
// every product's result tile is the next product's B operand where it
// stands; so the compute waves exchange nothing and one barrier per chunk
// hands the operand buffers over.  Every product takes fp16 operands rounded
// from fp32 (K and V rows as fp16, exact in fp16's normal range; the caller's
// Q rows times a power of two, taken back from the output's factor: Q S is then
// as exact for a q outside fp16's range as the state-wave form's bf16 product).
//
// What bounds it: with a workgroup on every compute unit HBM (64 packed
// sequences x 32 heads: 3.9 GB in 876 us, 4.5 TB/s; the state-wave form, whose
// eight workgroups per head each pull the chunk's 44 KiB of K, Q, Tb and P into
// their compute units, ~1700 us); on its own 2.1 to 2.4 us per chunk (transfer
// pass 1.3 to 1.5), instruction issue: per SIMD 120 MFMAs (1,920 cycles of its
// matrix pipe), ~665 VALU and ~112 LDS instructions of its compute and its
// helper wave, at the ~5 cycles a SIMD takes per VALU or MFMA instruction.  32
// columns per wave halve the LDS reads per product of 16 (one 1 KiB fragment,
// two MFMAs): eight compute waves of 16 columns, staging themselves, took 2.5
// us per chunk, and a split into state and output waves 2.8.
//
// Staging: as many helper waves hold the next three chunks' K, Q and V units
// and Tb / P fragments in registers (a load has two steps to land) and write
// them to the other of two LDS buffers, K (KLayout) and Q as fp16 -- COPY
// (use_qk_l2norm): the prep kernel's normalised fp16 copies as they are
// (normalising here instead made the helper the longer wave: 2.9 us per
// chunk) -- V as fp16, and the chunk's gate factors.
//
// Registers: K = V = 128 takes 256 VGPRs, unspilled but for saves and o in one
// launch, which spills 15 to 17 and is 2 to 15 % faster than a launch for each,
// in segments too (W = 4, T = 20000 148 -> 129 us, W = 32, T = 16384 526 -> 476,
// W = 64 897 -> 811; at 32 spilled registers it was slower there).
// K = 128 with V = 64 (four waves, 106 KB of LDS: alone on its compute
// unit) takes up to 422 with the AGPRs.  K = V = 64 (74 KB) takes 244 with COPY
// and 275 without, where a compute unit then holds one workgroup instead of
// two (held to 256 it would spill 32).
//
// Segments (few long chains): a chunk maps the state by S -> M_c S + B_c, so a
// sequence is cut into segments whose own contributions B (from a zero state)
// and transfer matrices M (from I, with V = 0) are formed in parallel (XFER),
// chunk_combine_kernel runs S_j = M_j S_(j-1) + B_j over them, and the
// segments' outputs then start from those states, again in parallel.
#include <algorithm>
#include <type_traits>

#include "gdn_chunk.h"

namespace gdn {

struct HeadArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const float* h0;
  float* ht;
  uint16_t* o;
  const int32_t* cu;
  int N, T, total, Hqk, Hv;
  float scale;
  int seg;      // chunks per segment (0: whole sequences)
  int member;   // if ws.longs lists any, sequences of more chunks are (the state-wave form's)
  bool ht_in_segs;   // (segments, ht == h0) a cut sequence's final state goes to ws.segs
  TokenStride ts;
};

// Segments.  Sequence n's chunks are cut into segments of `seg` chunks (one
// at least, also for an empty sequence); ws.soff[n] is its first segment's
// global index with cu_seqlens (chunk_table_kernel, which leaves those of
// WsPlan::cut chunks and less in one), n times a constant without.  Every
// segment but a sequence's last is full; ws.segs and ws.segm hold the full ones
// alone, so without the last ones of the n sequences before: segment j of
// sequence n is full segment first + j - n.
__device__ __forceinline__ void seg_range(int n, int seg, const int32_t* cu, int T,
                                          const ChunkWs& ws, int& first, int& count) {
  if (cu) {
    first = ws.soff[n];
    count = ws.soff[n + 1] - first;
  } else {
    count = max(1, ((T + kChunk - 1) / kChunk + seg - 1) / seg);
    first = n * count;
  }
}
struct SegPos {
  int n;            // sequence, -1 past the last segment
  int full;         // index among the full segments (a last segment: one past the
                    // full segment that it follows)
  int first;        // its sequence's chunk it starts at
  int c_begin, nc;  // global first chunk, chunks
  bool last;        // the sequence's last segment
};
// i-th segment -- or (full) the i-th that is not its sequence's last, or
// (seg == 0) the i-th sequence as a whole
__device__ __forceinline__ SegPos seg_pos(int i, bool full, int seg, const int32_t* cu, int N,
                                          int T, const ChunkWs& ws) {
  SegPos r{i, i, 0, 0, 0, true};
  const int nct = (T + kChunk - 1) / kChunk;
  int j = 0, cnt = 1;
  if (seg) {
    if (cu) {
      if (i >= ws.soff[N] - (full ? N : 0)) return SegPos{-1, 0, 0, 0, 0, true};
      int lo = 0, hi = N;   // the largest n whose first segment is i or before
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ws.soff[mid] - (full ? mid : 0) <= i) lo = mid; else hi = mid;
      }
      r.n = lo;
    } else {
      const int per = max(1, (nct + seg - 1) / seg) - (full ? 1 : 0);
      r.n = i / per;
    }
    int first;
    seg_range(r.n, seg, cu, T, ws, first, cnt);
    r.full = full ? i : i - r.n;
    j = r.full - (first - r.n);
  }
  const int c0 = cu ? ws.off[r.n] : r.n * nct;
  const int c1 = cu ? ws.off[r.n + 1] : c0 + nct;
  r.first = j * seg;
  r.c_begin = c0 + r.first;
  r.last = j + 1 == cnt;
  r.nc = r.last ? c1 - r.c_begin : seg;
  return r;
}

// Q rows in LDS: row-major, 2 K bytes per row, 16-byte units permuted so that
// the 16 rows of a fragment read fall on distinct banks.
template <int K>
__device__ __forceinline__ constexpr int qrow_off(int r, int u) {
  return r * 2 * K + 16 * (u ^ (K == 128 ? (r & 15) : ((r >> 1) & 7)));
}
// V rows in LDS: row-major, 2 V bytes per row, 32-byte tiles permuted so that
// the 4 rows of a transposing read (and the next 8-row group's) fall on
// distinct banks.
template <int V>
__device__ __forceinline__ constexpr int vrow_swz(int r) {
  return V == 128 ? ((r & 3) | (((r >> 3) & 1) << 2)) : (((r >> 1) & 1) | (((r >> 3) & 1) << 1));
}

// round(a b + c) to fp16 per element, c fp16 (v_fma_mixlo / mixhi_f16: the
// product and sum in fp32, one rounding)
__device__ __forceinline__ u16x4 fma_h4(f32x4 a, f32x4 b, u16x4 c) {
  const f16x4 ch = __builtin_bit_cast(f16x4, c);
  f16x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r[i] = static_cast<_Float16>(__builtin_fmaf(a[i], b[i], static_cast<float>(ch[i])));
  return __builtin_bit_cast(u16x4, r);
}

// Eight bf16 values times s (a power of two), as fp16 in one rounding.
__device__ __forceinline__ u16x8 scale_h8(u16x8 x, float s) {
  constexpr u16x4 kNegZero4 = {0x8000, 0x8000, 0x8000, 0x8000};
  const f32x8 f = __builtin_convertvector(__builtin_bit_cast(bf16x8, x), f32x8);
  const f32x4 s4 = {s, s, s, s};
  return cat8(fma_h4(f32x4{f[0], f[1], f[2], f[3]}, s4, kNegZero4),
              fma_h4(f32x4{f[4], f[5], f[6], f[7]}, s4, kNegZero4));
}
// The larger of m and every |x| of eight bf16 values (NaN left out).
__device__ __forceinline__ float max_abs8(u32x4 x, float m) {
#pragma unroll
  for (int y = 0; y < 4; ++y)
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(x[y] << 16), "v"(x[y] & 0xffff0000u));
  return m;
}

// Workgroup bid of nb with a qk-head group's workgroups on one XCD (they read the
// same K, Q rows; workgroups are dealt to the 8 XCDs in turn).
__device__ __forceinline__ int group_block(int bid, int nb, int G) {
  if (nb % (8 * G)) return bid;
  const int i = bid >> 3;
  return ((i / G) * 8 + (bid & 7)) * G + i % G;
}

// LDS accesses done, then a bare barrier (global loads and stores stay in
// flight).
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0) alone
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

template <int K, int V, bool COPY, bool SAVE, bool OUT, bool XFER>
__global__ __launch_bounds__(4 * V) void chunk_head_kernel(HeadArgs a, ChunkWs ws) {
  static_assert(!XFER || (!SAVE && !OUT && K == V), "XFER leaves only segment states");
  constexpr int NW = V / 32, HT = 64 * NW;   // compute waves (and helper waves), helper threads
  constexpr int KB = K / 32, ST = K / 16;    // k-blocks over the keys, state tiles
  using KL = KLayout<K>;
  constexpr int UPR = K / 8;                 // 16-byte units per K / Q row
  constexpr int KPT = 64 * UPR / HT;         // K (Q) units per helper thread
  constexpr int VPT = 64 * (V / 8) / HT;     // V units per helper thread
  constexpr int NSL = OUT ? 12 : 6;          // fragment slots: Tb, then P
  constexpr int SPW = (NSL + NW - 1) / NW;   // fragment slots per helper wave
  constexpr bool kRowsQ = OUT && !COPY;      // Q from the caller's rows
  // Operand buffer b of the two sits at byte kBufStep b of one block: every
  // fragment address is then a per-lane offset of the step's buffer plus an
  // immediate (under 64 KiB), with no address registers per buffer.
  constexpr int kQ = KL::BYTES, kV = kQ + (OUT ? 128 * K : 0), kF = kV + 128 * V;
  constexpr int kG = kF + NSL * 1024, kO = kG + 512, kE = kO + (OUT ? 256 : 0);
  constexpr int kBufStep = (kE + 16 + 255) / 256 * 256;
  static_assert(kBufStep <= 65536, "a buffer's offsets fit the LDS immediates");
  __shared__ __attribute__((aligned(256))) unsigned char buf[2 * kBufStep];
  __shared__ __attribute__((aligned(16))) u16x8 Vx[SAVE ? 2 * NW : 1][2][64];

  const int G = a.Hv / a.Hqk;
  // XFER: a second half of the grid forms the transfer matrices
  const int nb = XFER ? gridDim.x / 2 : gridDim.x;
  const bool mpart = XFER && (int)blockIdx.x >= nb;
  const int bid = group_block(mpart ? blockIdx.x - nb : blockIdx.x, nb, G);
  const int h = bid % a.Hv;
  const int hq = h / G;
  const int lane = threadIdx.x % 64;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r16 = lane % 16, grp = lane / 16;

  // this workgroup's chunks: a sequence's, or one segment of them (XFER: one
  // that another follows)
  const SegPos sp = seg_pos(bid / a.Hv, XFER, a.seg, a.cu, a.N, a.T, ws);
  if (sp.n < 0) return;
  if (ws.longs && sp.nc > a.member && ws.longs[0] > 0) return;
  const int n = sp.n, full = sp.full;
  int s, e;
  seq_bounds(a.cu, n, a.T, a.total, s, e);
  const int c_begin = sp.c_begin, nc = sp.nc;
  s += sp.first * kChunk;
  if (mpart && sp.first == 0) return;   // the first segment starts from h0: no M needed

  if (w >= NW) {
    // ---------------------------------------------------- helper waves ----
    const int hw = w - NW, tid = 64 * hw + lane;
    struct Regs {
      u32x4 k[KPT], q[OUT ? KPT : 1], v[VPT], f[SPW];
      float g;
    };
    Regs r0, r1, r2;
    auto load = [&](Regs& r, int j) {
      const int ci = c_begin + j, t0 = s + j * kChunk, L = min(kChunk, e - t0);
      // K, Q: the prep kernel's fp16 copies (contiguous), or the caller's rows
      // (rows past the sequence end read as 0)
      const size_t co = (size_t)ci * a.Hqk + hq;
      const uint16_t* kp = a.k + (size_t)t0 * a.ts.k + hq * K;
      const uint16_t* qp = a.q + (size_t)t0 * a.ts.q + hq * K;
      const __amdgpu_buffer_rsrc_t rk =
          COPY ? __builtin_amdgcn_make_buffer_rsrc(ws.k16 + co * KL::BYTES, 0, KL::BYTES,
                                                   kBufferFlags)
               : __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kp), 0, L * a.ts.k * 2,
                                                   kBufferFlags);
      const __amdgpu_buffer_rsrc_t rq =
          COPY ? __builtin_amdgcn_make_buffer_rsrc(ws.q16 + co * 4 * KB * 64, 0, 128 * K,
                                                   kBufferFlags)
               : __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(qp), 0, L * a.ts.q * 2,
                                                   kBufferFlags);
#pragma unroll
      for (int i = 0; i < KPT; ++i) {
        const int x = tid + HT * i;
        const int row = x / UPR, unit = 16 * (x % UPR);
        r.k[i] = __builtin_amdgcn_raw_buffer_load_b128(
            rk, COPY ? 16 * x : row * a.ts.k * 2 + unit, 0, 0);
        if constexpr (OUT)
          r.q[i] = __builtin_amdgcn_raw_buffer_load_b128(
              rq, COPY ? 16 * x : row * a.ts.q * 2 + unit, 0, 0);
      }
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint16_t*>(a.v + (size_t)t0 * a.ts.v + h * V), 0,
          mpart ? 0 : L * a.ts.v * 2, kBufferFlags);   // (a transfer matrix has V = 0)
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        const int x = tid + HT * i;
        r.v[i] = __builtin_amdgcn_raw_buffer_load_b128(
            rv, (x / (V / 8)) * a.ts.v * 2 + 16 * (x % (V / 8)), 0, 0);
      }
      const size_t fo = ((size_t)ci * a.Hv + h) * 6 * 64;
#pragma unroll
      for (int i = 0; i < SPW; ++i) {
        const int sl = min(hw + NW * i, NSL - 1);
        const u16x8* p = (sl < 6 ? ws.tfrag : ws.pfrag) + fo + (sl < 6 ? sl : sl - 6) * 64;
        const __amdgpu_buffer_rsrc_t rf =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<u16x8*>(p), 0, 1024, kBufferFlags);
        r.f[i] = __builtin_amdgcn_raw_buffer_load_b128(rf, 16 * lane, 0, 0);
      }
      const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(
          ws.gate + ((size_t)ci * a.Hv + h) * 64, 0, 256, kBufferFlags);
      r.g = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rg, lane * 4, 0, 0));
    };
    auto stage = [&](const Regs& r, int j, int b) {
      unsigned char* bp = buf + b * kBufStep;
#pragma unroll
      for (int i = 0; i < KPT; ++i) {
        const int x = tid + HT * i;
        if constexpr (COPY) {   // already laid out
          *reinterpret_cast<u32x4*>(bp + 16 * x) = r.k[i];
          if constexpr (OUT) *reinterpret_cast<u32x4*>(bp + kQ + 16 * x) = r.q[i];
        } else {
          *reinterpret_cast<u16x8*>(bp + KL::off(x / UPR, x % UPR)) =
              bf2h8(__builtin_bit_cast(u16x8, r.k[i]));
        }
      }
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        const int x = tid + HT * i, row = x / (V / 8), u = x % (V / 8);
        *reinterpret_cast<u16x8*>(bp + kV + row * 2 * V + 16 * (u ^ (2 * vrow_swz<V>(row)))) =
            bf2h8(__builtin_bit_cast(u16x8, r.v[i]));
      }
#pragma unroll
      for (int i = 0; i < SPW; ++i)
        if (hw + NW * i < NSL)
          *reinterpret_cast<u32x4*>(bp + kF + 1024 * (hw + NW * i) + 16 * lane) = r.f[i];
      // Q rows as fp16 times a power of two, and the output's factor scale e^G with
      // it taken back: 2^8 where this wave's rows are in range of it, else one for
      // each row by its largest element
      if constexpr (kRowsQ) {
        float top = 0.f;
#pragma unroll
        for (int i = 0; i < KPT; ++i) top = max_abs8(r.q[i], top);
        if (!__any(top >= 256.f) && __any(top >= 0x1p-13f)) {
#pragma unroll
          for (int i = 0; i < KPT; ++i) {
            const int x = tid + HT * i;
            *reinterpret_cast<u16x8*>(bp + kQ + qrow_off<K>(x / UPR, x % UPR)) =
                scale_h8(__builtin_bit_cast(u16x8, r.q[i]), 256.f);
          }
          if (lane / (64 / UPR) % NW == hw)
            *reinterpret_cast<float*>(bp + kO + 4 * lane) = a.scale * __expf(r.g) * 0x1p-8f;
        } else {
#pragma unroll
          for (int i = 0; i < KPT; ++i) {
            const int x = tid + HT * i, row = x / UPR;
            unsigned m = __float_as_uint(max_abs8(r.q[i], 0.f));
#pragma unroll
            for (int d = 1; d < UPR; d *= 2) m = max(m, (unsigned)__shfl_xor((int)m, d));
            // the largest element to 2^14 .. 2^15, both factors normal floats
            const int e = max((int)(m >> 23), 15);
            *reinterpret_cast<u16x8*>(bp + kQ + qrow_off<K>(row, x % UPR)) =
                scale_h8(__builtin_bit_cast(u16x8, r.q[i]), __int_as_float((268 - e) << 23));
            const float g = __shfl(r.g, row);
            if (x % UPR == 0)
              *reinterpret_cast<float*>(bp + kO + 4 * row) =
                  a.scale * __expf(g) * __int_as_float((e - 14) << 23);
          }
        }
      } else if constexpr (OUT) {
        if (lane / (64 / UPR) % NW == hw)
          *reinterpret_cast<float*>(bp + kO + 4 * lane) = a.scale * __expf(r.g);
      }
      if (hw == NW - 1) {
        const int L = min(kChunk, e - (s + j * kChunk));
        const float GL = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.g), L - 1));
        const float eg = __expf(r.g);
        float* gp = reinterpret_cast<float*>(bp + kG);
        gp[lane] = eg;
        gp[64 + lane] = __expf(GL - r.g);
        if (lane == L - 1) *reinterpret_cast<float*>(bp + kE) = eg;
      }
    };
    if (nc > 0) {
      // during step j chunk j+1 is written from its set and chunk j+4
      // requested into that set, so a load has two to three steps to land
      // (past the last chunk repeated, into a buffer no step reads)
      load(r0, 0);
      load(r1, min(1, nc - 1));
      load(r2, min(2, nc - 1));
      stage(r0, 0, 0);
      load(r0, min(3, nc - 1));
      lds_barrier();
      auto turn = [&](Regs& r, int j) {
        stage(r, min(j + 1, nc - 1), (j + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
        load(r, min(j + 4, nc - 1));
        lds_barrier();
      };
      int j = 0;
      for (; j + 2 < nc; j += 3) {
        turn(r1, j);
        turn(r2, j + 1);
        turn(r0, j + 2);
      }
      if (j < nc) turn(r1, j);
      if (j + 1 < nc) turn(r2, j + 1);
    }
    return;
  }

  // ------------------------------------------------------ compute waves ----
  // state tile t of column tile x: lane (r16, grp), element r =
  // S[rho(16t + 4grp + r)][32 w + 16 x + r16]
  const size_t lane_tile = 32 * w + r16, kv = (size_t)K * V;
  // the state to start from: the caller's, or the state after the segment
  // before (chunk_combine_kernel)
  const float* init = a.h0 ? a.h0 + ((size_t)n * a.Hv + h) * kv : nullptr;
  if (sp.first > 0) init = XFER ? nullptr : ws.segs + ((size_t)(full - 1) * a.Hv + h) * kv;
  f32x4 S[2][ST];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
#pragma unroll
    for (int t = 0; t < ST; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rho_row(t, 4 * grp + r);
        if (mpart) S[x][t][r] = row == (int)lane_tile + 16 * x ? 1.f : 0.f;
        else S[x][t][r] = init ? init[lane_tile + 16 * x + (size_t)row * V] : 0.f;
      }
    }
  }
  // per-lane byte offsets of the fragment reads in the step's buffer (see
  // KLayout; the rest of every address is an immediate, but for the k-block,
  // which a row's unit permutation takes as an XOR of byte address bits 6 and
  // up: one instruction per read block where an offset per k-block held nine
  // registers more, and 16 were spilled)
  const int m4 = r16 >> 2, q4 = r16 & 3;
  int ka_off = KL::off(rho_row(0, r16), grp), tr_off = KL::off(8 * grp + m4, q4),
      q_off = kQ + (COPY ? 16 * lane : qrow_off<K>(r16, grp)), v_off[2], f_off = kF + 16 * lane,
      g_off = kG + 32 * grp, e_off = kO + 4 * r16;
#pragma unroll
  for (int x = 0; x < 2; ++x)
    v_off[x] = kV + (8 * grp + m4) * 2 * V + 32 * ((2 * w + x) ^ vrow_swz<V>(8 * grp + m4)) + 8 * q4;
  auto lds8 = [&](int off) { return *reinterpret_cast<const u16x8*>(buf + off); };
  auto lds4 = [&](int off) { return *reinterpret_cast<const f32x4*>(buf + off); };
  auto ldst = [&](int off) { return lds_tr16(reinterpret_cast<const uint16_t*>(buf + off)); };

  float decay = 1.f;   // (XFER) of the state over the segment's chunks so far
  // What chunk j - 1 leaves for step j to finish: its output's Q S term
  // (scaled), vnew and P fragments.
  f32x4 O[2][4];
  u16x8 vx[2][2], pf[6];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) O[x][ti] = zero4();
    vx[x][0] = vx[x][1] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
#pragma unroll
  for (int f = 0; f < 6; ++f) pf[f] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  auto fence = [] { __builtin_amdgcn_sched_barrier(0); };

  // o += P vnew, row tiles tb .. te - 1
  auto out_mfma = [&](int tb, int te) {
#pragma unroll
    for (int ti = tb; ti < te; ++ti) {
#pragma unroll
      for (int x = 0; x < 2; ++x) O[x][ti] = mfma16h(vx[x][0], pf[tb_slot(ti, 0)], O[x][ti]);
    }
#pragma unroll
    for (int ti = tb; ti < te; ++ti) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
        if (ti >= 2) O[x][ti] = mfma16h(vx[x][1], pf[tb_slot(ti, 1)], O[x][ti]);
    }
  };
  // row tile ti of chunk j's o: one 16-byte store (v_permlane16_swap: lane
  // grp then holds columns 8 (grp / 2) .. + 7 of column tile grp % 2), the
  // four lanes of a row covering 64 contiguous bytes; j < 0 stores nothing
  auto out_store = [&](int ti, int j) {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const int t0 = s + max(j, 0) * kChunk, L = j < 0 ? 0 : min(kChunk, e - t0);
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        a.o + ((size_t)t0 * a.Hv + h) * V, 0, L * a.Hv * V * 2, kBufferFlags);
    const u32x2 o0 = __builtin_bit_cast(u32x2, f2bf4(O[0][ti]));
    const u32x2 o1 = __builtin_bit_cast(u32x2, f2bf4(O[1][ti]));
    u32x4 row;
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const auto sw = __builtin_amdgcn_permlane16_swap(o0[y], o1[y], false, false);
      row[y] = sw[0];
      row[2 + y] = sw[1];
    }
    __builtin_amdgcn_raw_buffer_store_b128(
        row, ro, ((16 * ti + r16) * a.Hv * V + 32 * w + 16 * (grp & 1) + 8 * (grp >> 1)) * 2, 0, 0);
  };

  // A step's products run in blocks of four fragments (eight MFMAs); a
  // block's LDS reads are issued one block ahead of it, and the fences keep
  // the compiler from sinking them to their use, which would expose the LDS
  // latency at every product.  Blocks: K 0..KB-1 (X = K S), Q 0..KB-1
  // ((Q S)^T), K^T in fours of state tiles.  The conversions and gate factors
  // are dealt among MFMAs that do not depend on them (kMix), the previous
  // chunk's P vnew covering the state's conversion.
  constexpr u16x4 kNegZero4 = {0x8000, 0x8000, 0x8000, 0x8000};
#define kReads(N) __builtin_amdgcn_sched_group_barrier(0x100, (N), 0);
#define kMix(NM, NV)                                       \
  _Pragma("unroll") for (int z = 0; z < (NM); ++z) {       \
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     \
    __builtin_amdgcn_sched_group_barrier(0x002, (NV), 0);  \
  }
  auto step = [&](int j) {
    constexpr int NB = OUT ? 2 * KB : KB;   // K and Q blocks
    constexpr int NK = 2 * (ST / 4);        // K^T blocks
    u16x8 win[2][4];   // block i in win[i % 2]
    auto read_blk = [&](int i) {
      u16x8 (&f)[4] = win[i % 2];
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        if (i < KB) {
          f[y] = lds8((ka_off ^ 64 * i) + KL::RS * (32 * (y >> 1) + 4 * (y & 1)));
        } else if (i < NB) {
          f[y] = lds8(COPY ? q_off + 1024 * (i - KB) + y * KB * 1024 : (q_off ^ 64 * (i - KB)) + y * 32 * K);
        } else if (i < NB + NK) {
          // element i of lane (m, grp): K[32 b + 8 grp + i][rho(16 t + m)]
          const int b = (i - NB) / (ST / 4), t = 4 * ((i - NB) % (ST / 4)) + y;
          const int p = (tr_off ^ 64 * (t >> 1)) + KL::RS * 32 * b + 8 * (t & 1);
          f[y] = cat8(ldst(p), ldst(p + KL::RS * 4));
        }
      }
    };
    const float egl = *reinterpret_cast<const float*>(buf + (g_off - 32 * grp) + (kE - kG));
    if constexpr (XFER) decay *= egl;
    read_blk(0);
    if constexpr (SAVE) {
      // the chunk's start state: hs[chunk][v-head] = S^T (bf16), row 32 w +
      // 16 x + r16, keys 32 b + 8 grp .. + 7
      const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(
          ws.hs + ((size_t)(c_begin + j) * a.Hv + h) * V * K, 0, V * K * 2, kBufferFlags);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
#pragma unroll
        for (int b = 0; b < KB; ++b)
          __builtin_amdgcn_raw_buffer_store_b128(
              __builtin_bit_cast(u32x4, cat8(f2bf4(S[x][2 * b]), f2bf4(S[x][2 * b + 1]))), hr,
              ((32 * w + 16 * x + r16) * K + 32 * b + 8 * grp) * 2, 0, kStoreStream);
      }
    }
    // the state as fp16 B fragments, beside the previous chunk's P vnew
    u16x8 sh[2][KB];
    if constexpr (OUT) out_mfma(0, 4);
#pragma unroll
    for (int b = 0; b < KB; ++b) {
#pragma unroll
      for (int x = 0; x < 2; ++x) sh[x][b] = cat8(f2h4(S[x][2 * b]), f2h4(S[x][2 * b + 1]));
    }
    kReads(5)
    if constexpr (OUT) kMix(12, KB == 4 ? 3 : 2)
    fence();
    // X = K S on the four rho-ordered token tiles
    f32x4 X[2][4], eg[4];
    u16x4 v4[2][4];
    u16x8 ta[6];
    auto read_v = [&](int b) {
#pragma unroll
      for (int ti = 2 * b; ti < 2 * b + 2; ++ti) {
        const int r0 = 32 * b + 4 * (ti & 1);
#pragma unroll
        for (int x = 0; x < 2; ++x) v4[x][ti] = ldst(v_off[x] + r0 * 2 * V);
        eg[ti] = lds4(g_off + 4 * r0);
      }
    };
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      read_blk(b + 1);
      if (b == KB - 1) read_v(0);
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
          X[x][ti] = mfma16h(win[b % 2][ti], sh[x][b], b ? X[x][ti] : zero4());
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        S[x][2 * b] = S[x][2 * b] * egl;
        S[x][2 * b + 1] = S[x][2 * b + 1] * egl;
      }
      if constexpr (OUT) {
#pragma unroll
        for (int ti = b * 4 / KB; ti < (b + 1) * 4 / KB; ++ti) out_store(ti, j - 1);
      }
      kReads(8)
      kMix(8, OUT ? 4 : 2)
      fence();
    }
    // Y = V - e^G X as B fragments, vnew = Tb Y, U = e^(G_last - G) vnew
    u16x8 yf[2][2], uh[2][2];
    f32x4 vn[2][4], dc[4];
    auto form_y = [&](int b) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        u16x4 yy[2];
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          yy[y] = fma_h4(-eg[2 * b + y], X[x][2 * b + y], v4[x][2 * b + y]);
        }
        yf[x][b] = cat8(yy[0], yy[1]);
      }
    };
    auto read_ta = [&] {
#pragma unroll
      for (int f = 0; f < 6; ++f) ta[f] = lds8(f_off + 1024 * f);
    };
    auto read_dc = [&] {
#pragma unroll
      for (int ti = 0; ti < 4; ++ti)
        dc[ti] = lds4(g_off + 256 + 4 * (32 * (ti >> 1) + 4 * (ti & 1)));
    };
    auto form_vn = [&](int b) {
#pragma unroll
      for (int ti = 2 * b; ti < 4; ++ti) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
          vn[x][ti] = mfma16h(ta[tb_slot(ti, b)], yf[x][b], b ? vn[x][ti] : zero4());
      }
    };
    auto form_u = [&](int b) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        uh[x][b] = cat8(fma_h4(dc[2 * b], vn[x][2 * b], kNegZero4),
                        fma_h4(dc[2 * b + 1], vn[x][2 * b + 1], kNegZero4));
        if constexpr (OUT || SAVE) vx[x][b] = cat8(f2h4(vn[x][2 * b]), f2h4(vn[x][2 * b + 1]));
      }
    };
    // (Q S)^T: lane (r16, grp) of tile ti holds token 16 ti + r16, columns
    // 32 w + 16 x + 4 grp .. + 3
    auto q_blk = [&](int b) {
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
          O[x][ti] = mfma16h(sh[x][b], win[(KB + b) % 2][ti], b ? O[x][ti] : zero4());
      }
    };
    if constexpr (OUT) {
      read_blk(KB + 1);
      read_v(1);
      q_blk(0);
      form_y(0);
      kReads(12)
      kMix(8, 5)
      fence();
      if constexpr (KB == 4) read_blk(KB + 2);
      read_ta();
      q_blk(1);
      form_y(1);
      kReads(12)
      kMix(8, 5)
      fence();
      form_vn(0);
      form_vn(1);
      read_dc();
      fence();
      if constexpr (KB == 4) {
        read_blk(KB + 3);
        q_blk(2);
        form_u(0);
        kReads(8)
        kMix(8, 4)
        fence();
        read_blk(NB);
        q_blk(3);
        form_u(1);
        kReads(8)
        kMix(8, 4)
      } else {
        read_blk(NB);
        form_u(0);
        form_u(1);
      }
      fence();
    } else {
      read_v(1);
      read_ta();
      read_dc();
      form_y(0);
      form_y(1);
      form_vn(0);
      form_vn(1);
      form_u(0);
      form_u(1);
      fence();
    }
    // S = e^G_last S + K^T U, K^T block by block
    float ego[4];
#pragma unroll
    for (int y = 0; y < NK; ++y) {
      const int i = NB + y, b = y / (ST / 4);
      if (y + 1 < NK) read_blk(i + 1);
      if (OUT && y == 0) {
#pragma unroll
        for (int ti = 0; ti < 4; ++ti)
          ego[ti] = *reinterpret_cast<const float*>(buf + e_off + 64 * ti);
      }
      if (OUT && y == NK - 1) {
#pragma unroll
        for (int f = 0; f < 6; ++f) pf[f] = lds8(f_off + 6144 + 1024 * f);
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const int t = 4 * (y % (ST / 4)) + f;
#pragma unroll
        for (int x = 0; x < 2; ++x) S[x][t] = mfma16h(win[i % 2][f], uh[x][b], S[x][t]);
      }
      if (OUT && y >= NK - 2) {
#pragma unroll
        for (int ti = 2 * (y - (NK - 2)); ti < 2 * (y - (NK - 2)) + 2; ++ti) {
#pragma unroll
          for (int x = 0; x < 2; ++x) O[x][ti] = ego[ti] * O[x][ti];
        }
        kReads(14)
        kMix(8, 2)
      }
      fence();
    }
    if constexpr (SAVE) {
      // the chunk's deltas: lane t stores token row t (16 columns per tile),
      // through this wave's own LDS rows and four transposing reads per tile
      const int L = min(kChunk, e - (s + j * kChunk));
      const __amdgpu_buffer_rsrc_t dr = __builtin_amdgcn_make_buffer_rsrc(
          ws.dl + ((size_t)(c_begin + j) * a.Hv + h) * 64 * V, 0, 64 * V * 2, kBufferFlags);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int ct = 2 * w + x;
#pragma unroll
        for (int b = 0; b < 2; ++b) Vx[ct][b][lane] = vx[x][b];
        __builtin_amdgcn_wave_barrier();
        const uint16_t* src =
            reinterpret_cast<const uint16_t*>(
                &Vx[ct][grp >> 1][16 * (2 * (grp & 1) + (q4 >> 1)) + m4]) + 4 * (q4 & 1);
        u16x8 d0 = cat8(lds_tr16(src), lds_tr16(src + 32));
        u16x8 d1 = cat8(lds_tr16(src + 64), lds_tr16(src + 96));
        const u16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
        d0 = lane < L ? h2bf8(d0) : zero;
        d1 = lane < L ? h2bf8(d1) : zero;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, d0), dr,
                                               ((2 * ct) * 64 + lane) * 16, 0, kStoreStream);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, d1), dr,
                                               ((2 * ct + 1) * 64 + lane) * 16, 0, kStoreStream);
      }
    }
  };
  auto next = [&](int j) {
    lds_barrier();
    // the next step's buffer
    const int d = (j & 1) ? -kBufStep : kBufStep;
    ka_off += d;
    q_off += d;
    tr_off += d;
    v_off[0] += d;
    v_off[1] += d;
    f_off += d;
    g_off += d;
    e_off += d;
  };
#undef kMix
#undef kReads

  if (nc > 0) {
    lds_barrier();
    for (int j = 0; j < nc; ++j) {
      step(j);
      next(j);
    }
    if constexpr (OUT) {
      out_mfma(0, 4);
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) out_store(ti, nc - 1);
    }
  }
  if (mpart) {
    // E = M - decay I as hi + lo (bf16), the combine's A fragments (row tile t,
    // k-block w), transposed through this wave's share of the operand buffers
    constexpr int LD = 20;
    static_assert(2 * 32 * LD * 2 <= 4096 && 4096 * NW <= 2 * kBufStep, "a wave's share");
    uint16_t* X = reinterpret_cast<uint16_t*>(buf + 4096 * w);
    u16x8* dst = ws.segm + ((size_t)full * a.Hv + h) * (2 * ST * KB * 64) + w * 64 + lane;
    if (threadIdx.x == 0) ws.sdecay[(size_t)full * a.Hv + h] = decay;
#pragma unroll
    for (int t = 0; t < ST; ++t) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        f32x4 e = S[x][t];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (rho_row(t, 4 * grp + r) == (int)lane_tile + 16 * x) e[r] -= decay;
        u16x4 hi, lo;
        split_bf4(e, hi, lo);
        *reinterpret_cast<u16x4*>(X + (16 * x + r16) * LD + 4 * grp) = hi;
        *reinterpret_cast<u16x4*>(X + (32 + 16 * x + r16) * LD + 4 * grp) = lo;
      }
      __builtin_amdgcn_wave_barrier();
      dst[t * KB * 64] = lds_colfrag(X, LD, 0, 0, lane);
      dst[(ST + t) * KB * 64] = lds_colfrag(X, LD, 32, 0, lane);
      __builtin_amdgcn_wave_barrier();
    }
    return;
  }
  float* out = sp.last && a.ht ? a.ht + ((size_t)n * a.Hv + h) * kv : nullptr;
  // in place the first segment's workgroup may yet read the state here: it
  // goes over the one that this workgroup, and no other, started from
  if (out && a.ht_in_segs && sp.first > 0) out = ws.segs + ((size_t)(full - 1) * a.Hv + h) * kv;
  if constexpr (XFER) out = ws.segs + ((size_t)full * a.Hv + h) * kv;
  if (out) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
#pragma unroll
      for (int t = 0; t < ST; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[lane_tile + 16 * x + (size_t)rho_row(t, 4 * grp + r) * V] = S[x][t][r];
      }
    }
  }
}

// States at the segment starts: S_j = M_j S_(j-1) + B_j from the segments' own
// contributions B (ws.segs; the first segment's is already the state after
// it) and transfer matrices M (ws.segm, ws.sdecay), in place of B.  One workgroup
// per (sequence, v-head, 16 value columns), wave w the state rows rho(16 w + m).
// M = decay I + E: the decay goes over the fp32 state in fp32, as within a
// chunk (g = beta = 0 leaves every bit), and E S, what the segment's tokens
// take out, is a product of bf16 hi + lo halves (three MFMA passes, ~2^-17
// relative, where the chunks' own take fp16 operands, 2^-11).  Errors against
// 64 bits are those of a chain in one piece to three digits.  ~1.2 us per
// segment (25 of 4 heads 30.0 us, the call 98); M itself in three parts and six
// products, exact too, took 37.0 and 105, on fp32 MFMA 42.
// The state passes between the waves through LDS, and a segment's E fragments
// are requested two segments ahead.
template <int K>
__global__ __launch_bounds__(4 * K) void chunk_combine_kernel(HeadArgs a, ChunkWs ws) {
  constexpr int ST = K / 16, KB = K / 32;   // row tiles (waves), k-blocks
  __shared__ __attribute__((aligned(16))) u16x8 St[2][2][KB][64];   // [parity][hi, lo]
  const int h = blockIdx.x % a.Hv, vt = blockIdx.x / a.Hv;
  const int lane = threadIdx.x % 64;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r16 = lane % 16, grp = lane / 16;
  // The sequences with three segments or more (with fewer nothing but the first
  // segment is started from), every gridDim.y-th of them here: found NT at a
  // time, a bit per thread.
  constexpr int NT = 4 * K;
  __shared__ unsigned long long many[NT / 64];
  if (a.cu && ws.soff[a.N] == a.N) return;   // none is cut
  int seen = 0;
  for (int base = 0; base < a.N; base += NT) {
    int first = 0, count = 0;   // a sequence's segments
    if (base + (int)threadIdx.x < a.N)
      seg_range(base + threadIdx.x, a.seg, a.cu, a.T, ws, first, count);
    const unsigned long long mine = __ballot(count >= 3);
    if (lane == 0) many[w] = mine;
    lds_barrier();
    for (int word = 0; word < NT / 64; ++word) {
      for (unsigned long long left = many[word]; left; left &= left - 1) {
        if (seen++ % (int)gridDim.y != (int)blockIdx.y) continue;
        const int n = __builtin_amdgcn_readfirstlane(base + 64 * word + __builtin_ctzll(left));
        seg_range(n, a.seg, a.cu, a.T, ws, first, count);
        auto head = [&](int j) { return (size_t)(first - n + j) * a.Hv + h; };
        auto load_e = [&](u16x8 (&m)[2][KB], int j) {
          const u16x8* p = ws.segm + head(j) * (2 * ST * KB * 64) + w * KB * 64 + lane;
#pragma unroll
          for (int y = 0; y < 2; ++y) {
#pragma unroll
            for (int b = 0; b < KB; ++b) m[y][b] = p[(y * ST * KB + b) * 64];
          }
        };
        // this wave's state tile: lane (r16, grp), element r = row rho(16 w + 4 grp
        // + r), column 16 vt + r16
        auto tile_at = [&](int j) {
          return ws.segs + head(j) * K * K + (size_t)rho_row(w, 4 * grp) * K + 16 * vt + r16;
        };
        auto load_b = [&](int j) {
          const float* p = tile_at(j);
          return f32x4{p[0], p[K], p[2 * K], p[3 * K]};
        };
        auto publish = [&](f32x4 x, int par) {
          u16x4 part[2];
          split_bf4(x, part[0], part[1]);
#pragma unroll
          for (int y = 0; y < 2; ++y)   // (a B fragment: tile w's half of k-block w / 2)
            reinterpret_cast<u16x4*>(&St[par][y][w >> 1][lane])[w & 1] = part[y];
          lds_barrier();
        };
        // segment j's E fragments, decay and B tile in set j % 3
        u16x8 m[3][2][KB];
        f32x4 bt[3];
        float dec[3];
        auto load = [&](auto set, int j) {
          constexpr int c = decltype(set)::value;
          load_e(m[c], j);
          bt[c] = load_b(j);
          dec[c] = ws.sdecay[head(j)];
        };
        load(std::integral_constant<int, 1>{}, 1);
        load(std::integral_constant<int, 2>{}, min(2, count - 2));
        f32x4 state = load_b(0);   // this wave's tile of the state after the segment before
        publish(state, 0);
        auto step = [&](int j, auto jc) {
          constexpr int c = decltype(jc)::value;   // j % 3
          load(std::integral_constant<int, (c + 2) % 3>{}, min(j + 2, count - 2));
          f32x4 acc = zero4(), acc1 = zero4(), acc2 = zero4();
#pragma unroll
          for (int b = 0; b < KB; ++b) {
            const u16x8 hi = St[(j + 1) & 1][0][b][lane], lo = St[(j + 1) & 1][1][b][lane];
            acc = mfma16(m[c][0][b], hi, acc);
            acc1 = mfma16(m[c][0][b], lo, acc1);
            acc2 = mfma16(m[c][1][b], hi, acc2);
          }
          state = dec[c] * state + (bt[c] + (acc + (acc1 + acc2)));
          float* o = tile_at(j);
#pragma unroll
          for (int r = 0; r < 4; ++r) o[(size_t)r * K] = state[r];
          publish(state, j & 1);
        };
        for (int j = 1; j < count - 1;) {
          step(j++, std::integral_constant<int, 1>{});
          if (j < count - 1) step(j++, std::integral_constant<int, 2>{});
          if (j < count - 1) step(j++, std::integral_constant<int, 0>{});
        }
        lds_barrier();   // St is free for the next sequence
      }
    }
    lds_barrier();   // as is `many`
  }
}

// ht_in_segs: the cut sequences' final states from where chunk_head_kernel left
// them.  One workgroup per v-head and, as far as the grid goes, sequence.
__global__ __launch_bounds__(256) void chunk_final_state_kernel(HeadArgs a, ChunkWs ws, int kv) {
  const int h = blockIdx.x;
  for (int n = blockIdx.y; n < a.N; n += gridDim.y) {
    int first, count;
    seg_range(n, a.seg, a.cu, a.T, ws, first, count);
    if (count < 2) continue;
    const float* src = ws.segs + ((size_t)(first - n + count - 2) * a.Hv + h) * kv;
    float* dst = a.ht + ((size_t)n * a.Hv + h) * kv;
    for (int i = threadIdx.x; i < kv; i += 256) dst[i] = src[i];
  }
}

template <int K, bool SAVE, bool OUT>
void launch_chain_head(const uint16_t* q, const uint16_t* k, const uint16_t* v, const float* h0,
                       float* ht, uint16_t* o, const int32_t* cu, int N, int T, int total, int Hqk,
                       int Hv, int V, float scale, bool l2, TokenStride ts, const WsPlan& p,
                       const ChunkWs& ws, hipStream_t st) {
  const bool ht_in_segs = p.seg && p.nfull > 0 && ht && ht == h0;
  const HeadArgs a{q, k, v, h0, ht, o, cu, N, T, total, Hqk, Hv, scale, p.seg,
                   p.member, ht_in_segs, ts};
  const unsigned grid = (unsigned)((p.seg ? p.nseg : N) * Hv);
  auto go = [&](auto kern, unsigned g) {
    hipLaunchKernelGGL(kern, dim3(g), dim3(4 * V), 0, st, a, ws);
  };
  if (p.seg && p.nfull > 0 && V == K) {   // (segments are planned for K == V only)
    const unsigned full = (unsigned)(p.nfull * Hv);
    if (l2) go(chunk_head_kernel<K, K, true, false, false, true>, 2 * full);
    else go(chunk_head_kernel<K, K, false, false, false, true>, 2 * full);
    // a workgroup per (v-head, column tile) and, as far as the GPU holds them,
    // sequence; with many sequences the rest in turn (most have no segments)
    const unsigned tiles = (unsigned)(Hv * (V / 16));
    const unsigned seqs = std::min<unsigned>(N, std::max(1u, 4u * device_cus() / tiles));
    hipLaunchKernelGGL((chunk_combine_kernel<K>), dim3(tiles, seqs), dim3(4 * K), 0, st, a, ws);
  }
  if (V == 128) {
    if (l2) go(chunk_head_kernel<K, 128, true, SAVE, OUT, false>, grid);
    else go(chunk_head_kernel<K, 128, false, SAVE, OUT, false>, grid);
  } else {
    if (l2) go(chunk_head_kernel<K, 64, true, SAVE, OUT, false>, grid);
    else go(chunk_head_kernel<K, 64, false, SAVE, OUT, false>, grid);
  }
  if (ht_in_segs)
    hipLaunchKernelGGL(chunk_final_state_kernel, dim3(Hv, std::min(N, 1024)), dim3(256), 0, st, a,
                       ws, K * V);
}

#define GDN_HEAD_INST(K_, SAVE_, OUT_)                                                       \
  template void launch_chain_head<K_, SAVE_, OUT_>(                                          \
      const uint16_t*, const uint16_t*, const uint16_t*, const float*, float*, uint16_t*,    \
      const int32_t*, int, int, int, int, int, int, float, bool, TokenStride, const WsPlan&, \
      const ChunkWs&, hipStream_t);
GDN_HEAD_INST(64, false, true)
GDN_HEAD_INST(64, true, false)
GDN_HEAD_INST(64, true, true)
GDN_HEAD_INST(128, false, true)
GDN_HEAD_INST(128, true, false)
GDN_HEAD_INST(128, true, true)
#undef GDN_HEAD_INST

}  // namespace gdn
