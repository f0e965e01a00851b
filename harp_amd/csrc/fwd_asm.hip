// Forward kernel for head dim 128 with a hand-scheduled main loop.
//
// Reference math: gemm/ring_attention/ring_attn.cpp:2412-2575
// (ring_attention_forward: Q-stationary online softmax over the KV chunks of
// the ring), as fwd_kernel in ra_kernels.hip computes it.
//
// Work split: a block is 4 waves x 64 queries (one wave per SIMD).  A wave's
// 64 queries are two 32-query groups, so every K or V^T fragment read from
// LDS feeds two MFMAs (0.5 KB of LDS per MFMA against 1 KB in fwd_kernel);
// O^T (128 x 64 fp32 per wave) lives in AGPRs a0..a127 and Q in a128..a191.
// Keys go in 32-key blocks through eight LDS block buffers, copied
// global -> LDS five blocks ahead, with a barrier every second block.  The loop over the blocks is one inline-asm
// statement generated by fwd_asm_gen.py (fwd_asm.inc): it issues every
// instruction in a fixed order, with the wait states gfx950 requires between
// dependent MFMA / VALU instructions inserted by the generator.  Its state
// stays in the pinned register tuples below across the whole loop.
//
// Numerics match fwd_kernel: fp32 S, lazy rescale of O and l when a row's
// maximum grows by more than 2^8 (tested here on the exps themselves: a lane
// whose block sum exceeds 2^8 makes the wave move its reference points up to
// that block's maxima and compute the block's exps again), P rounded to bf16
// only as the MFMA operand, row sums of the unrounded exps in fp32, exp2 with
// log2(e) folded into the scale.  One difference: m is the reference point of
// the exps (at most 8 log2 units below the exact row maximum that fwd_kernel
// writes) and l is relative to it, so m + log l is the same LSE.
#include <cstddef>
#include <type_traits>

#include "fwd_asm.inc"
#include "q_epilogue.h"
#include "ra_common.h"
#include "ra_kernels.h"

namespace harp_ra {

namespace {

typedef int v32i __attribute__((ext_vector_type(32)));

constexpr int kAsmWaves = 4;
constexpr int kAsmRows = 64 * kAsmWaves;  // queries per block
static_assert(kAsmRows == kQueryBlockRows, "the host sizes KV splits with kQueryBlockRows");
constexpr int kLoopLds = 2 * 65536;  // K block buffers, then V block buffers (8 x 8 KiB each)
// the epilogue's staging rows reuse the same memory after the loop
constexpr int kLdsBytes = kLoopLds > q_epi::kStageBytes ? kLoopLds : q_epi::kStageBytes;
static_assert(q_epi::kWaves == kAsmWaves && q_epi::kRowsPerWave * kAsmWaves == kAsmRows, "epilogue geometry");

// The ChunkTable fields the loop reads from the kernel arguments (s_load
// from the kernarg segment: FwdParams is the kernel's only argument).
constexpr int kCtOff = (int)offsetof(FwdParams, ct);
constexpr int kOrderOff = kCtOff + (int)offsetof(ChunkTable, order);
constexpr int kLenOff = kCtOff + (int)offsetof(ChunkTable, len);
constexpr int kKOff = kCtOff + (int)offsetof(ChunkTable, k);
constexpr int kVOff = kCtOff + (int)offsetof(ChunkTable, v);

}  // namespace

__global__ __launch_bounds__(64 * kAsmWaves, 1) void fwd_asm_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(16))) char lds[kLdsBytes];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  int qt, h, b;
  decode_block((p.T + kAsmRows - 1) / kAsmRows, p.H, qt, h, b);
  const KvSplit sp = kv_split(p.ct.n);
  const float c2 = p.scale * kLog2e;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)lds;

  // V block buffer 7 holds the "block -1" that the first slot's O MFMAs read
  // with P = 0: zeros, so no stale bit pattern can make a NaN
  {
    const uint4 z = make_uint4(0u, 0u, 0u, 0u);
    uint4* vb7 = (uint4*)(lds + 65536 + 7 * 8192);
    vb7[tid] = z;
    vb7[tid + 256] = z;
  }

  // Q of query qi = qt * 256 + 64 wave + 32 qg + l32, elements 16 ks + 8 g
  // .. + 7: the B operand of S^T = K Q^T, at a[128 + (8 qg + ks) * 4].  The
  // block's 256 rows go global -> LDS first, by direct-to-LDS loads that
  // move whole rows per 16 lanes (rows past T load as zero: the buffer range
  // ends at row T), into the loop's K-buffer layout, and from there into the
  // registers (the V buffer 7 zeros above lie outside the rows' 64 KiB)
  v32i q0, q1;
  {
    const int r0 = qt * kAsmRows;
    const rsrc_t rq = rows_rsrc(p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh, p.sqt, r0, p.T - r0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {  // 64 copies of 1 KiB (4 rows), 16 per wave
      const int inst = wave * 16 + i, row = inst * 4 + (lane >> 4);
      const uint32_t chunk = (uint32_t)(((lane & 15) ^ swz(row)) << 4);
      lds_dma_b128(rq, lds0 + inst * 1024, (uint32_t)(row * p.sqt * 2) + chunk);
    }
    wait_lds_loads();
    __syncthreads();
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
      const int row = wave * 64 + qg * 32 + l32;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const uint4 x = *(const uint4*)(lds + row * 256 + (((2 * ks + g) ^ swz(row)) << 4));
        v32i& q = qg ? q1 : q0;
        q[ks * 4 + 0] = (int)x.x;
        q[ks * 4 + 1] = (int)x.y;
        q[ks * 4 + 2] = (int)x.z;
        q[ks * 4 + 3] = (int)x.w;
      }
    }
    __syncthreads();  // every wave has its rows before the loop's copies overwrite them
  }
  asm volatile("" : "+{a[128:159]}"(q0), "+{a[160:191]}"(q1));

  // per-lane constants and the softmax state (v32..v63) and v192..v223
  const int64_t sbytes = p.skt * 2;
  v32i misc, misc2;
  {
    int mv[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) mv[i] = 0;
    // K row fragments: row l32 of a block buffer, chunk 2 ks + g (XOR layout)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) mv[ks] = (int)(lds0 + l32 * 256 + (((2 * ks + g) ^ swz(l32)) << 4));
    // V^T fragments by ds_read_b64_tr_b16: rows 8 hh + 4 g + s of a 16-row
    // group, columns 32 db + l32
    const int j = lane >> 4, s = (lane >> 2) & 3, m = lane & 3;
    const int cl = 2 * (j & 1) + (m >> 1);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const int row = 8 * hh + 4 * g + s;
        mv[8 + hh * 4 + db] =
            (int)(lds0 + 65536 + 2 * (row * 128 + (((4 * db + cl) ^ swz(row)) << 3) + 4 * (m & 1)));
      }
    // copy offsets: instruction i of this wave fills rows 4 (2 wave + i) ..
    // + 3 of a block, 16 bytes per lane, chunk (lane % 16) ^ swz(row)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = (2 * wave + i) * 4 + (lane >> 4);
      mv[16 + i] = (int)(r * sbytes + (((lane & 15) ^ swz(r)) << 4));
    }
    mv[18] = mv[19] = __float_as_int(-INFINITY);  // m_ref (the loop starts it at -FLT_MAX)
    mv[26] = mv[27] = __float_as_int(-INFINITY);  // m_new
#pragma unroll
    for (int i = 0; i < 32; ++i) misc[i] = mv[i];
#pragma unroll
    for (int i = 0; i < 32; ++i) misc2[i] = 0;
    misc2[1] = 4 * g;                             // c_row(r, g) - c_row(r, 0)
    misc2[2] = __float_as_int(-INFINITY);         // the tail mask's value
  }
  asm volatile("" : "+{v[32:63]}"(misc), "+{v[192:223]}"(misc2));
  // fragments, P, S and O: outputs of the loop statement, which zeroes what
  // it reads before writing it (O ends zero when the split has no keys)
  v32i frag, pp, s0, s1, o0, o1, o2, o3;

  // the key cursor (first non-empty chunk of this split) and the number of
  // 32-key blocks of the split
  const int64_t kvo = (int64_t)b * p.skb + (int64_t)h * p.skh;
  KvCursor cur;
  kv_enter(p.ct, kvo, sp.begin, sp.end, cur);
  int nb = 0;
  for (int st = sp.begin; st < sp.end; ++st) nb += (p.ct.len[p.ct.order[st]] + 31) >> 5;
  const bool any = cur.step < sp.end;
  const uint64_t kp0 = any ? (uint64_t)(uintptr_t)cur.k : 0, vp0 = any ? (uint64_t)(uintptr_t)cur.v : 0;
  const int left0 = any ? cur.len : 0;
  const uint64_t ctp = (uint64_t)(uintptr_t)(const void*)__builtin_amdgcn_kernarg_segment_ptr();
  const uint64_t kvb = (uint64_t)(kvo * 2);
  const uint32_t dbase = lds0 + (uint32_t)wave * 2048u;
  const uint32_t blkb = (uint32_t)(32 * sbytes);

  {
    asm volatile(HARP_FWD_ASM_LOOP
                 : "+{v[32:63]}"(misc), "={v[64:95]}"(frag), "={v[96:127]}"(pp), "={v[128:159]}"(s0),
                   "={v[160:191]}"(s1), "+{v[192:223]}"(misc2), "={a[0:31]}"(o0), "={a[32:63]}"(o1),
                   "={a[64:95]}"(o2), "={a[96:127]}"(o3), "+{a[128:159]}"(q0), "+{a[160:191]}"(q1)
                 : [c2] "s"(sgpr_of(c2)), [dbase] "s"(dbase), [sbytes] "s"((uint32_t)sbytes), [blkb] "s"(blkb),
                   [kvl] "s"((uint32_t)kvb), [kvh] "s"((uint32_t)(kvb >> 32)), [ctp] "s"(ctp), [end] "s"(sp.end),
                   [nb] "s"(nb), [kp0] "s"(kp0), [vp0] "s"(vp0), [left0] "s"(left0), [step0] "s"(cur.step),
                   [ooff] "n"(kOrderOff), [loff] "n"(kLenOff), [koff] "n"(kKOff), [voff] "n"(kVOff)
                 : "memory", "vcc", HARP_FWD_ASM_SGPR_CLOBBERS);
  }

  // epilogue: O / l, and the row statistics m = m_ref (the loop's reference
  // point, the same in both lane halves of a row) and l relative to it (a
  // row without keys: m = -inf, l = 0).  O is staged through LDS so that
  // every query row is stored by 32 lanes as one contiguous row; every
  // address comes from q_epilogue.h, which the host bounds check compiles too
  namespace E = q_epi;
  const int lane_e = lane_id_fresh(), g_e = lane_e >> 5;
  float* const st = (float*)lds + E::stage_base(wave);
  __syncthreads();  // every wave is done with the loop's block buffers
#pragma unroll
  for (int qg = 0; qg < 2; ++qg) {
    const float l_tot = wave_half_sum(__int_as_float(misc[22 + qg]));
    const float m_ref = (l_tot > 0.f) ? __int_as_float(misc[18 + qg]) : -INFINITY;
    const float inv = (l_tot > 0.f) ? 1.f / l_tot : 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const v32i& acc = db < 2 ? (qg ? o2 : o0) : (qg ? o3 : o1);
        const int idx = (db & 1) * 16 + 4 * i;
        const f32x4 x = {__int_as_float(acc[idx]) * inv, __int_as_float(acc[idx + 1]) * inv,
                         __int_as_float(acc[idx + 2]) * inv, __int_as_float(acc[idx + 3]) * inv};
        *(f32x4*)(st + E::stage_write(qg, db, i, lane_e)) = x;
      }
    const int qi = qt * kAsmRows + wave * 64 + qg * 32 + (lane_e & 31);
    if (qi < p.T && g_e == 0) {
      const int64_t si = sp.index * p.split_ml + ((int64_t)b * p.H + h) * p.T + qi;
      const float m_nat = m_ref * kLn2;
      if (p.m_bf16) {
        const bf16 mh = (bf16)m_nat;
        const float mhf = (float)mh;
        ((bf16*)p.m)[si] = mh;
        p.l[si] = (l_tot > 0.f) ? l_tot * __expf(m_nat - mhf) : 0.f;
      } else {
        ((float*)p.m)[si] = m_nat;
        p.l[si] = l_tot;
      }
    }
  }
  __syncthreads();
  const int qtile0 = qt * kAsmRows;
  const int64_t bh = sp.index * p.split_o + (int64_t)b * p.sob + (int64_t)h * p.soh;
  const int64_t bhb = (int64_t)b * p.sbb + (int64_t)h * p.sbh;
#pragma unroll 1
  for (int it0 = 0; it0 < E::kRowsPerWave / 2; it0 += 8) {
    f32x4 x[8];  // eight rows read back before any is stored: one LDS latency
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = *(const f32x4*)(st + E::stage_read(it0 + j, lane_e));
    // which outputs are wanted is decided once per eight rows, in a loop that
    // is not unrolled (three unrolled epilogues cost their instruction fetch):
    // one block of 64 keys 10.1 -> 9.7 us with O alone, 10.6 -> 10.5 with both
    auto store_rows = [&](auto f32_out, auto rounded_out) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int qi = E::out_query(qtile0, wave, it0 + j, lane_e);
        if (qi >= p.T) continue;
        if constexpr (f32_out) {
          float* o = p.out + E::out_elem(bh, qi, p.sot, lane_e);
          o[0] = x[j].x;
          o[1] = x[j].y;
          o[2] = x[j].z;
          o[3] = x[j].w;
        }
        // the rounded output straight from the staged row: a cast pass over O
        // took 4 us at 30 heads x 256 rows and 24 us at 24 x 8192 (4.2 TB/s)
        if constexpr (rounded_out)
          *(bf16x4*)(p.outb + E::out_elem(bhb, qi, p.sbt, lane_e)) = __builtin_convertvector(x[j], bf16x4);
      }
    };
    if (!p.outb) store_rows(std::true_type{}, std::false_type{});
    else if (p.out) store_rows(std::true_type{}, std::true_type{});
    else store_rows(std::false_type{}, std::true_type{});
  }
}

// D = 128 exactly (the copies fill whole 256-byte rows).
bool fwd_asm_applies(const FwdParams& p) { return p.D == 128; }

hipError_t launch_fwd_asm(const FwdParams& p, hipStream_t st) {
  const int n = ((p.T + kAsmRows - 1) / kAsmRows) * p.H * p.B;
  hipLaunchKernelGGL(fwd_asm_kernel, dim3(n, p.n_split), dim3(64 * kAsmWaves), 0, st, p);
  return hipGetLastError();
}

}  // namespace harp_ra
