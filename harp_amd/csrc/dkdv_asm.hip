// Backward dK/dV kernel for head dim 128 with a hand-scheduled main loop.
//
// Reference math: gemm/ring_attention/ring_attn.cpp:2577-2829
// (ring_attention_backward: P = exp(S - LSE), dS = P (dP - D), dV = P^T dO,
// dK = dS^T Q scaled), KV-stationary as the reference and as dkdv_kernel in
// ra_kernels.hip.
//
// A block owns 256 keys of one (b, h): 4 waves x 64 keys, one wave per SIMD,
// two 32-key groups per wave, so every Q, dO, Q^T or dO^T fragment read from
// LDS feeds two MFMAs.  dK and dV (2 x 128 x 64 fp32 per wave) accumulate in
// the 256 AGPRs; the wave's K rows, the B operands of S = Q K^T, sit in
// v32..v95 for the whole block; V rows are read from the block's padded V
// tile in LDS.  Queries stream in 32-query blocks through five LDS buffers,
// copied three blocks ahead, with their statistics rows (-LSE / scale and
// -D, written by the dQ kernel, which runs first) as the S and dP
// accumulators' initial values.  The loop over the query blocks is one
// inline-asm statement generated by dkdv_asm_gen.py (dkdv_asm.inc); it binds
// every VGPR, so nothing lane-dependent is kept across it.
//
// Numerics match dkdv_kernel: fp32 S and dP, P = exp2(S' c) clamped to [0, 1],
// dS = P dP', P and dS rounded to bf16 only as MFMA operands, fp32 dK / dV;
// dK scaled once in the epilogue; pad keys written as zero.
#include <cstddef>

#include "dkdv_asm.inc"
#include "dkdv_epilogue.h"
#include "ra_common.h"
#include "ra_kernels.h"

namespace harp_ra {

namespace {

typedef int v32i __attribute__((ext_vector_type(32)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kAsmWaves = 4;
constexpr int kKeysPerWave = 64;
static_assert(kAsmWaves * kKeysPerWave == kDkdvBlockKeys, "the host sizes the key tiles with kDkdvBlockKeys");
constexpr int kBufBytes = 16384;                           // Q rows 8 KiB, dO rows 8 KiB
constexpr int kNumBuf = 5;
constexpr int kVOff = kNumBuf * kBufBytes;                 // 81920
constexpr int kVRow = 272;                                 // padded V row: 256 + 16 bytes
constexpr int kStatsOff = kVOff + kDkdvBlockKeys * kVRow;  // 151552
constexpr int kStatsPerWave = kNumBuf * 512;               // two 256-byte planes per buffer
constexpr int kLdsBytes = kStatsOff + kAsmWaves * kStatsPerWave;
static_assert(kLdsBytes <= 163840, "LDS of one CU");
static_assert(dkdv_epi::kWaves == kAsmWaves && dkdv_epi::kKeysPerWave == kKeysPerWave, "epilogue geometry");
static_assert(dkdv_epi::stage_base(kAsmWaves) * 4 <= kLdsBytes, "epilogue staging fits the LDS");

__device__ __forceinline__ void put4(v32i& t, int i, const uint4& x) {
  t[i * 4 + 0] = (int)x.x;
  t[i * 4 + 1] = (int)x.y;
  t[i * 4 + 2] = (int)x.z;
  t[i * 4 + 3] = (int)x.w;
}

}  // namespace

__global__ __launch_bounds__(64 * kAsmWaves, 1) void dkdv_asm_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(16))) char lds[kLdsBytes];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  int kt, h, b;
  decode_block(p.n_key_tiles, p.H, kt, h, b);
  int c = 0;
#pragma unroll 1
  for (int i = 1; i < p.ct.n; ++i)
    if (kt >= p.ct.tile0[i]) c = i;
  c = __builtin_amdgcn_readfirstlane(c);
  const int kblk0 = (kt - p.ct.tile0[c]) * kDkdvBlockKeys;
  const int len = p.ct.len[c];
  // in an SGPR for the loop statement, which owns every VGPR
  const uint32_t c2 = sgpr_of(p.scale * kLog2e);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)lds;
  const bool any = kblk0 < len;  // block-uniform: the block has a valid key
  const int64_t kvo = (int64_t)b * p.skb + (int64_t)h * p.skh;

  // The block's V rows into the padded tile (rows past the valid length: 0)
  // and the wave's K rows, the B operands of S = Q K^T (key kblk0 + 64 wave +
  // 32 kg + l32, elements 16 ks + 8 g .. + 7, at v[32 + 32 kg + 4 ks]); buffer
  // 4's Q / dO rows zeroed: the first slot's dV / dK MFMAs read them as
  // "block -1" with P = dS = 0, and a stale bit pattern could be NaN.  All 32
  // row loads are issued before any is used (one memory round trip): from a
  // clamped row (row kblk0 is valid when the block has a valid key), then
  // selected, since a load under the lane condition makes each one wait for
  // the previous.
  v32i kb0, kb1;
  {
    uint4 vx[16], kx[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) vx[i] = kx[i] = make_uint4(0u, 0u, 0u, 0u);
    if (any) {
      const bf16* vb = p.ct.v[c] + kvo;
      const bf16* kb = p.ct.k[c] + kvo;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = kblk0 + ((i * 256 + tid) >> 4), ch = tid & 15;
        vx[i] = *(const uint4*)(vb + (int64_t)(key < len ? key : kblk0) * p.skt + ch * 8);
      }
#pragma unroll
      for (int kg = 0; kg < 2; ++kg) {
        const int key = kblk0 + wave * kKeysPerWave + kg * 32 + l32;
        const bf16* krow = kb + (int64_t)(key < len ? key : kblk0) * p.skt;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) kx[kg * 8 + ks] = *(const uint4*)(krow + ks * 16 + g * 8);
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int idx = i * 256 + tid, row = idx >> 4, ch = idx & 15;
      const bool ok = kblk0 + row < len;
      *(uint4*)(lds + kVOff + row * kVRow + ch * 16) = ok ? vx[i] : make_uint4(0u, 0u, 0u, 0u);
    }
    uint4* b4 = (uint4*)(lds + 4 * kBufBytes);
#pragma unroll
    for (int i = 0; i < 4; ++i) b4[i * 256 + tid] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int kg = 0; kg < 2; ++kg) {
      const bool ok = kblk0 + wave * kKeysPerWave + kg * 32 + l32 < len;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) put4(kg ? kb1 : kb0, ks, ok ? kx[kg * 8 + ks] : make_uint4(0u, 0u, 0u, 0u));
    }
  }
  __syncthreads();

  const int64_t qrow = p.sqt * 2, grow = p.sdt * 2;  // bytes between query rows
  v32i misc;
  {
    int mv[32];
    // Q / dO row fragments: row l32 of a 32-row tile, chunk 2 ks + g, buffer 0
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) mv[ks] = (int)(lds0 + l32 * 256 + (((2 * ks + g) ^ swz(l32)) << 4));
    // dO^T / Q^T fragments by ds_read_b64_tr_b16: rows 8 hh + 4 g + s of a
    // 16-row group, columns 32 db + l32, buffer 1 (the loop's base for the
    // first slot, whose reads select buffer 4 by offset)
    const int j = lane >> 4, sr = (lane >> 2) & 3, m = lane & 3;
    const int cl = 2 * (j & 1) + (m >> 1);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const int row = 8 * hh + 4 * g + sr;
        mv[8 + hh * 4 + db] =
            (int)(lds0 + kBufBytes + 2 * (row * 128 + (((4 * db + cl) ^ swz(row)) << 3) + 4 * (m & 1)));
      }
    mv[16] = (int)(lds0 + kVOff + (wave * kKeysPerWave + l32) * kVRow + g * 16);
    mv[17] = (int)(lds0 + kStatsOff + wave * kStatsPerWave + g * 16);
    // copy offsets: instruction i of wave w copies rows (2 w + i) * 4 + lane / 16
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = (2 * wave + i) * 4 + (lane >> 4);
      const int chunk = ((lane & 15) ^ swz(r)) << 4;
      mv[18 + i] = (int)(r * qrow + chunk);
      mv[20 + i] = (int)(r * grow + chunk);
    }
    mv[22] = lane * 4;
    // unused slots (v23; v24..v31 hold fragments in the loop): a copy of the
    // V address, which nothing after the loop needs (a constant there, e.g.
    // 0, would be taken from the tuple after the loop and cost it a copy in
    // scratch)
#pragma unroll
    for (int i = 23; i < 32; ++i) mv[i] = mv[16];
#pragma unroll
    for (int i = 0; i < 32; ++i) misc[i] = mv[i];
  }

  const QSplit qs = q_split(p);
  const int nb = any ? (qs.rows + 31) >> 5 : 0;
  const bf16* qb = p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh + qs.begin * p.sqt;
  const bf16* gb = p.dout + (int64_t)b * p.sdb + (int64_t)h * p.sdh + qs.begin * p.sdt;
  const int64_t sbase = ((int64_t)b * p.H + h) * p.T + qs.begin;
  const int64_t nrows = (int64_t)p.B * p.H * p.T;
  const uint64_t qp = (uint64_t)(uintptr_t)qb, gp = (uint64_t)(uintptr_t)gb;
  const uint64_t sp0 = (uint64_t)(uintptr_t)(p.stats + sbase), sp1 = (uint64_t)(uintptr_t)(p.stats + nrows + sbase);
  const uint32_t qnr = (uint32_t)(qs.rows * qrow), gnr = (uint32_t)(qs.rows * grow), snr = (uint32_t)(qs.rows * 4);
  const uint32_t qstep = (uint32_t)(32 * qrow), gstep = (uint32_t)(32 * grow);
  const uint32_t dbase = lds0 + (uint32_t)wave * 2048u;
  const uint32_t stb = lds0 + kStatsOff + (uint32_t)wave * kStatsPerWave;

  v32i sacc, dacc, pbds, init, frag, o0, o1, o2, o3, o4, o5, o6, o7;
  asm volatile(HARP_DKDV_ASM_LOOP
               : "+{v[0:31]}"(misc), "+{v[32:63]}"(kb0), "+{v[64:95]}"(kb1), "={v[96:127]}"(sacc),
                 "={v[128:159]}"(dacc), "={v[160:191]}"(pbds), "={v[192:223]}"(init), "={v[224:255]}"(frag),
                 "={a[0:31]}"(o0), "={a[32:63]}"(o1), "={a[64:95]}"(o2), "={a[96:127]}"(o3), "={a[128:159]}"(o4),
                 "={a[160:191]}"(o5), "={a[192:223]}"(o6), "={a[224:255]}"(o7)
               : [c2] "s"(c2), [dbase] "s"(dbase), [sbase] "s"(stb), [qp] "s"(qp), [gp] "s"(gp), [sp0] "s"(sp0),
                 [sp1] "s"(sp1), [qnr] "s"(qnr), [gnr] "s"(gnr), [snr] "s"(snr), [qstep] "s"(qstep),
                 [gstep] "s"(gstep), [nb] "s"(nb)
               : "memory", "vcc", HARP_DKDV_ASM_SGPR_CLOBBERS);

  // epilogue: C layout row = key kblk0 + 64 wave + 32 kg + c_row(r, g), col
  // = d = 32 db + lane; dK at a[64 kg + 16 db], dV at a[128 + 64 kg + 16 db]
  const int lane_e = lane_id_fresh(), g_e = lane_e >> 5;
  const int64_t base = (int64_t)b * p.sdkb + (int64_t)h * p.sdkh;
  if (!p.dkv_f32) {
    // bf16 outputs through LDS: each wave's 64 x 128 fp32 tile of dK, then
    // of dV, as rows of 136 floats (rows 4 apart, written by one
    // instruction, fall on disjoint banks), read back as 4 consecutive d per
    // lane and stored 8 bytes at a time (32 stores per tensor and wave
    // instead of 256 two-byte ones; the C ABI refuses bf16 dK / dV rows that
    // are not 8-byte aligned).  Every address comes from dkdv_epilogue.h,
    // which the host bounds check compiles too.
    namespace E = dkdv_epi;
    float* st = (float*)lds + E::stage_base(wave);
    __syncthreads();  // every wave is done with the loop's buffers
#pragma unroll
    for (int tn = 0; tn < 2; ++tn) {
      const float sc = tn == 0 ? p.scale : 1.f;
#pragma unroll
      for (int kg = 0; kg < 2; ++kg)
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int t = kg * 2 + (db >> 1), idx = (db & 1) * 16 + r;
            const v32i& acc = tn == 0 ? (t == 0 ? o0 : (t == 1 ? o1 : (t == 2 ? o2 : o3)))
                                      : (t == 0 ? o4 : (t == 1 ? o5 : (t == 2 ? o6 : o7)));
            st[E::stage_write(kg, db, r, lane_e)] = __int_as_float(acc[idx]) * sc;
          }
      __syncthreads();
      bf16* const out = tn == 0 ? p.ct.dk[c] : p.ct.dv[c];
      const int rows_c = p.ct_rows[c];
      const int64_t sdkt = p.sdkt;
#pragma unroll
      for (int it0 = 0; it0 < kKeysPerWave / 2; it0 += 8) {
        f32x4 x[8];  // eight rows read back before any is used: one LDS latency
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = *(const f32x4*)(st + E::stage_read(it0 + j, lane_e));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int kk = E::out_row(kblk0, wave, it0 + j, lane_e);
          if (kk >= rows_c) continue;
          bf16x4 y = __builtin_convertvector(x[j], bf16x4);
          if (kk >= len) y = bf16x4{};
          *(bf16x4*)(out + E::out_elem(base, kk, sdkt, lane_e)) = y;  // 8-byte aligned: the C ABI requires it
        }
      }
      __syncthreads();  // the staging rows are rewritten with dV
    }
    return;
  }
#pragma unroll
  for (int kg = 0; kg < 2; ++kg)
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const int d = db * 32 + (lane_e & 31);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kk = kblk0 + wave * kKeysPerWave + kg * 32 + c_row(r, g_e);
        if (kk >= p.ct_rows[c]) continue;
        const int t = kg * 2 + (db >> 1), idx = (db & 1) * 16 + r;
        const v32i& dkt = t == 0 ? o0 : (t == 1 ? o1 : (t == 2 ? o2 : o3));
        const v32i& dvt = t == 0 ? o4 : (t == 1 ? o5 : (t == 2 ? o6 : o7));
        // only fp32 outputs, the query splits' partials among them, come here
        const int64_t e = base + (int64_t)blockIdx.y * p.split_dkv + (int64_t)kk * p.sdkt + d;
        const bool valid = kk < len;
        const float vk = valid ? __int_as_float(dkt[idx]) * p.scale : 0.f;
        const float vv = valid ? __int_as_float(dvt[idx]) : 0.f;
        ((float*)p.ct.dk[c])[e] = vk;
        ((float*)p.ct.dv[c])[e] = vv;
      }
    }
}

// D = 128 exactly (the copies fill whole 256-byte rows), and byte offsets of
// 32 query rows within 32 bits
bool dkdv_asm_applies(const BwdParams& p) {
  return p.D == 128 && (int64_t)p.T * p.sqt * 2 < (1LL << 31) && (int64_t)p.T * p.sdt * 2 < (1LL << 31);
}

hipError_t launch_dkdv_asm(const BwdParams& p, hipStream_t st) {
  const int n = p.n_key_tiles * p.H * p.B;
  hipLaunchKernelGGL(dkdv_asm_kernel, dim3(n, p.n_split), dim3(64 * kAsmWaves), 0, st, p);
  return hipGetLastError();
}

}  // namespace harp_ra
