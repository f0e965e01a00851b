// Backward dQ kernel for head dim 128 with a hand-scheduled main loop.
//
// Reference math: gemm/ring_attention/ring_attn.cpp:2577-2829
// (ring_attention_backward: P = exp(S - LSE), dS = P (dP - D), dQ = dS K
// scaled), Q-stationary with S and dP recomputed, as dq_kernel in
// ra_kernels.hip computes it.
//
// Work split and memory path as fwd_asm_kernel (fwd_asm.hip): a block is 4
// waves x 64 queries (one wave per SIMD), two 32-query groups per wave, so
// every K, V or K^T fragment read from LDS feeds two MFMAs.  dQ^T (128 x 64
// fp32 per wave) accumulates in AGPRs a0..a127; Q and dO, the B operands of
// S^T = K Q^T and dP^T = V dO^T, sit in a128..a255.  Keys go in 32-key blocks
// through eight LDS block buffers, copied five blocks ahead, with a barrier
// every second block.  The loop over the blocks is one inline-asm statement
// generated by dq_asm_gen.py (dq_asm.inc).
//
// Numerics match dq_kernel: fp32 S and dP (its accumulators start at -D, so
// dP - D comes out of the MFMAs), P = exp2(S c2 - LSE2) clamped to
// [0, 1] (exact for valid keys; pad keys' zero K rows then contribute
// nothing), dS rounded to bf16 only as the MFMA operand, fp32 dQ scaled once.
#include <cstddef>

#include "dq_asm.inc"
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

constexpr int kCtOff = (int)offsetof(BwdParams, ct);
constexpr int kOrderOff = kCtOff + (int)offsetof(ChunkTable, order);
constexpr int kLenOff = kCtOff + (int)offsetof(ChunkTable, len);
constexpr int kKOff = kCtOff + (int)offsetof(ChunkTable, k);
constexpr int kVOff = kCtOff + (int)offsetof(ChunkTable, v);

// 16 bytes of row `row` starting at element 16 ks + 8 g into a v32i at 4 ks
__device__ __forceinline__ void put4(v32i& t, int ks, const uint4& x) {
  t[ks * 4 + 0] = (int)x.x;
  t[ks * 4 + 1] = (int)x.y;
  t[ks * 4 + 2] = (int)x.z;
  t[ks * 4 + 3] = (int)x.w;
}

}  // namespace

__global__ __launch_bounds__(64 * kAsmWaves, 1) void dq_asm_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(16))) char lds[kLdsBytes];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  int qt, h, b;
  decode_block((p.T + kAsmRows - 1) / kAsmRows, p.H, qt, h, b);
  const KvSplit sp = kv_split(p.ct.n);
  const float c2 = p.scale * kLog2e;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)lds;

  // Q and dO of query qi = qt * 256 + 64 wave + 32 qg + l32, elements
  // 16 ks + 8 g .. + 7, at a[128 + (8 qg + ks) * 4] and a[192 + ...].  The
  // block's 256 rows of each go global -> LDS first, by direct-to-LDS loads
  // that move whole rows per 16 lanes (rows past T load as zero: the buffer
  // range ends at row T), into the loop's K-buffer layout (row r, 16-byte
  // chunk c at r * 256 + ((c ^ swz(r)) << 4)), and from there into the
  // registers: one row per lane straight from global memory took twice as
  // long per block.
  v32i q0, q1, g0, g1;
  float dsum[16];  // without p.delta: dsum[0] = D of the wave's row 4 (lane % 16) + lane / 16
  {
    const int r0 = qt * kAsmRows;
    const rsrc_t rq = rows_rsrc(p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh, p.sqt, r0, p.T - r0);
    const rsrc_t rg = rows_rsrc(p.dout + (int64_t)b * p.sdb + (int64_t)h * p.sdh, p.sdt, r0, p.T - r0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {  // 64 copies of 1 KiB (4 rows) per tensor, 16 per wave
      const int inst = wave * 16 + i, row = inst * 4 + (lane >> 4);
      const uint32_t chunk = (uint32_t)(((lane & 15) ^ swz(row)) << 4);
      lds_dma_b128(rq, lds0 + inst * 1024, (uint32_t)(row * p.sqt * 2) + chunk);
      lds_dma_b128(rg, lds0 + 65536 + inst * 1024, (uint32_t)(row * p.sdt * 2) + chunk);
    }
    // D = rowsum(dO O) of the wave's 64 rows, 16 lanes x 8 elements per row,
    // four rows a step: O's rows are requested here, beside the copies, and
    // dO's are read back from LDS, so the block pays no launch and no second
    // read of dO for it (delta_kernel took 4 us at 30 heads x 256 rows, 24 us
    // at 24 x 8192).  One forward + backward at 30 x 256 rows, 8 chunks: 128
    // us before, 102 with D, the cast and the fill of m in these kernels.
    // The sums run in delta_kernel's order (8 elements of a lane in turn, then
    // lanes 8, 4, 2, 1 apart), so both entry points give the same D and dS
    const int sub = lane & 15, rr = lane >> 4;
    f32x4u ox[16], oy[16];
    if (!p.delta) {
      const float* ob = p.out + (int64_t)b * p.sob + (int64_t)h * p.soh + sub * 8;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int qi = r0 + wave * 64 + 4 * i + rr;
        const float* orow = ob + (int64_t)(qi < p.T ? qi : r0) * p.sot;  // past T: any row, its dO is zero
        ox[i] = *(const f32x4u*)orow;
        oy[i] = *(const f32x4u*)(orow + 4);
      }
    }
    wait_lds_loads();
    __syncthreads();
    if (!p.delta) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = wave * 64 + 4 * i + rr;
        const bf16x8 x = *(const bf16x8*)(lds + 65536 + row * 256 + ((sub ^ swz(row)) << 4));
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc = __builtin_fmaf((float)x[j], j < 4 ? ox[i][j] : oy[i][j - 4], acc);
        dsum[i] = acc;
      }
      // 16 sums over the 16 lanes of a row at once: each exchange halves the
      // values a lane still holds (15 exchanges, not 64), lane `sub` ends
      // with the sum of step i = sub
#pragma unroll
      for (int w = 8; w >= 1; w >>= 1) {
        const bool up = (sub & w) != 0;
#pragma unroll
        for (int i = 0; i < w; ++i) {
          const float keep = up ? dsum[i + w] : dsum[i], give = up ? dsum[i] : dsum[i + w];
          dsum[i] = keep + __shfl_xor(give, w, 16);
        }
      }
    }
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
      const int row = wave * 64 + qg * 32 + l32;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const int off = row * 256 + (((2 * ks + g) ^ swz(row)) << 4);
        put4(qg ? q1 : q0, ks, *(const uint4*)(lds + off));
        put4(qg ? g1 : g0, ks, *(const uint4*)(lds + 65536 + off));
      }
    }
    __syncthreads();  // every wave has its rows before the loop's buffers are written
  }

  // K block buffer 7 holds the "block -1" that the first slot's dQ MFMAs
  // read with dS = 0: zeros, so no stale bit pattern can make a NaN
  {
    uint4* kb7 = (uint4*)(lds + 7 * 8192);
    kb7[tid] = make_uint4(0u, 0u, 0u, 0u);
    kb7[tid + 256] = make_uint4(0u, 0u, 0u, 0u);
  }
  asm volatile("" : "+{a[128:159]}"(q0), "+{a[160:191]}"(q1), "+{a[192:223]}"(g0), "+{a[224:255]}"(g1));

  const int64_t sbytes = p.skt * 2;
  // the statistics of the lane's two queries (bwd_stat_lse and -D; 0 past T),
  // written once (split 0, lanes 0-31) for the dK/dV kernel
  float st0[2], st1[2];
  {
    const int64_t nrows = (int64_t)p.B * p.H * p.T;
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
      const int qi = qt * kAsmRows + wave * 64 + qg * 32 + l32;
      const bool ok = qi < p.T;
      const int64_t si = ((int64_t)b * p.H + h) * p.T + (ok ? qi : 0);
      st0[qg] = ok ? bwd_stat_lse(p, si) : 0.f;
      const int row = qg * 32 + l32;  // of the wave: step row / 4, lane group row % 4
      const float d = p.delta ? p.delta[si] : __shfl(dsum[0], (row & 3) * 16 + (row >> 2));
      st1[qg] = ok ? -d : 0.f;
      if (ok && g == 0 && sp.index == 0) {
        p.stats[si] = st0[qg];
        p.stats[nrows + si] = st1[qg];
      }
    }
  }
  v32i misc;
  {
    int mv[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) mv[i] = 0;
    // K and V row fragments: row l32 of a block buffer, chunk 2 ks + g
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      mv[ks] = (int)(lds0 + l32 * 256 + (((2 * ks + g) ^ swz(l32)) << 4));
      mv[8 + ks] = mv[ks] + 65536;
    }
    // K^T fragments by ds_read_b64_tr_b16: rows 8 hh + 4 g + s of a 16-row
    // group, columns 32 db + l32
    const int j = lane >> 4, s = (lane >> 2) & 3, m = lane & 3;
    const int cl = 2 * (j & 1) + (m >> 1);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const int row = 8 * hh + 4 * g + s;
        mv[16 + hh * 4 + db] = (int)(lds0 + 2 * (row * 128 + (((4 * db + cl) ^ swz(row)) << 3) + 4 * (m & 1)));
      }
    // copy offsets, as in the forward
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = (2 * wave + i) * 4 + (lane >> 4);
      mv[24 + i] = (int)(r * sbytes + (((lane & 15) ^ swz(r)) << 4));
    }
    // LSE2 = -c * plane 0 (+inf for a query past T: P = 0)
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
      const int qi = qt * kAsmRows + wave * 64 + qg * 32 + l32;
      mv[26 + qg] = __float_as_int(qi < p.T ? -st0[qg] * c2 : INFINITY);
      mv[28 + qg] = 0;
    }
#pragma unroll
    for (int i = 0; i < 32; ++i) misc[i] = mv[i];
  }
  asm volatile("" : "+{v[32:63]}"(misc));

  // -D of the lane's query (plane 1; 0 past T), 16 copies per query group:
  // the initial value of the dP^T accumulators, so dP - D costs no VALU
  v32i negd;
#pragma unroll
  for (int qg = 0; qg < 2; ++qg) {
    const int d = __float_as_int(st1[qg]);
#pragma unroll
    for (int i = 0; i < 16; ++i) negd[qg * 16 + i] = d;
  }

  // fragments, dS, S, dP and dQ: outputs of the loop statement, which zeroes
  // what it reads before writing it (dQ ends zero when the split has no keys)
  v32i fr0, fr1, s0, s1, d0, d1, o0, o1, o2, o3;

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

  asm volatile(HARP_DQ_ASM_LOOP
               : "+{v[0:31]}"(negd), "+{v[32:63]}"(misc), "={v[64:95]}"(fr0), "={v[96:127]}"(fr1),
                 "={v[128:159]}"(s0),
                 "={v[160:191]}"(s1), "={v[192:223]}"(d0), "={v[224:255]}"(d1), "={a[0:31]}"(o0),
                 "={a[32:63]}"(o1), "={a[64:95]}"(o2), "={a[96:127]}"(o3), "+{a[128:159]}"(q0),
                 "+{a[160:191]}"(q1), "+{a[192:223]}"(g0), "+{a[224:255]}"(g1)
               : [c2] "s"(sgpr_of(c2)), [dbase] "s"(dbase), [sbytes] "s"((uint32_t)sbytes), [blkb] "s"(blkb),
                 [kvl] "s"((uint32_t)kvb), [kvh] "s"((uint32_t)(kvb >> 32)), [ctp] "s"(ctp), [end] "s"(sp.end),
                 [nb] "s"(nb), [kp0] "s"(kp0), [vp0] "s"(vp0), [left0] "s"(left0), [step0] "s"(cur.step),
                 [ooff] "n"(kOrderOff), [loff] "n"(kLenOff), [koff] "n"(kKOff), [voff] "n"(kVOff)
               : "memory", "vcc", HARP_DQ_ASM_SGPR_CLOBBERS);

  // epilogue: dQ = scale * (dQ^T)^T, staged through LDS so that every query
  // row is stored by 32 lanes as one contiguous row; every address comes
  // from q_epilogue.h, which the host bounds check compiles too
  namespace E = q_epi;
  const int lane_e = lane_id_fresh();
  float* const st = (float*)lds + E::stage_base(wave);
  __syncthreads();  // every wave is done with the loop's block buffers
#pragma unroll
  for (int qg = 0; qg < 2; ++qg)
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const v32i& acc = db < 2 ? (qg ? o2 : o0) : (qg ? o3 : o1);
        const int idx = (db & 1) * 16 + 4 * i;
        const f32x4 x = {__int_as_float(acc[idx]) * p.scale, __int_as_float(acc[idx + 1]) * p.scale,
                         __int_as_float(acc[idx + 2]) * p.scale, __int_as_float(acc[idx + 3]) * p.scale};
        *(f32x4*)(st + E::stage_write(qg, db, i, lane_e)) = x;
      }
  __syncthreads();
  const int qtile0 = qt * kAsmRows;
  const int64_t bh = sp.index * p.split_dq + (int64_t)b * p.sdqb + (int64_t)h * p.sdqh;
#pragma unroll
  for (int it0 = 0; it0 < E::kRowsPerWave / 2; it0 += 8) {
    f32x4 x[8];  // eight rows read back before any is stored: one LDS latency
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = *(const f32x4*)(st + E::stage_read(it0 + j, lane_e));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int qi = E::out_query(qtile0, wave, it0 + j, lane_e);
      if (qi >= p.T) continue;
      const int64_t e = E::out_elem(bh, qi, p.sdqt, lane_e);
      if (p.dq_f32) {
        float* o = (float*)p.dq + e;
        o[0] = x[j].x;
        o[1] = x[j].y;
        o[2] = x[j].z;
        o[3] = x[j].w;
      } else {
        // 8-byte aligned: the C ABI requires it of bf16 dQ at head dim 128
        *(bf16x4*)((bf16*)p.dq + e) = __builtin_convertvector(x[j], bf16x4);
      }
    }
  }
}

// D = 128 exactly (the copies fill whole 256-byte rows).
bool dq_asm_applies(const BwdParams& p) { return p.D == 128; }

hipError_t launch_dq_asm(const BwdParams& p, hipStream_t st) {
  const int n = ((p.T + kAsmRows - 1) / kAsmRows) * p.H * p.B;
  hipLaunchKernelGGL(dq_asm_kernel, dim3(n, p.n_split), dim3(64 * kAsmWaves), 0, st, p);
  return hipGetLastError();
}

}  // namespace harp_ra
