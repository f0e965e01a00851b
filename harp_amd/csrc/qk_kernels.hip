// gfx950 kernels for the step before the ring-attention block: per-head
// RMSNorm of Q and K and the rotary embedding (RoPE), forward and backward,
// separately and fused.
//
// Reference math (HARP's async runtime, ARM SVE, run on the CPU):
//   rmsnormForwardKernelBF16   async_rt/csrc/rms_norm.cc:20-105
//     rms = sqrt(sum(x^2) / D + eps), out = bf16((x * (1 / rms)) * w), rms saved
//   rmsnormBackwardKernelBF16  async_rt/csrc/rms_norm.cc:107-240
//     xn = x / rms, g = dy * w, dx = bf16((g - xn * sum(g * xn) / D) / rms),
//     grad_w = sum over rows of dy * xn
//   ropeForwardKernelBF16      async_rt/csrc/rope.cc:9-86
//     pairs (x[2i], x[2i+1]) times (f[2i], f[2i+1]) as complex numbers
//   ropeBackwardKernelBF16     async_rt/csrc/rope.cc:88-183
//     times the conjugate of f
// Every bf16 result is truncated (the reference stores the high 16 bits of
// the fp32 value, async_rt/csrc/async_op_math.h:24-35), so these kernels do
// the same and match the reference's results to the last bit wherever the
// fp32 arithmetic agrees (sums of squares are reduced in a different order,
// which can move a result by one bf16 unit).
//
// Layout: x and every per-row tensor are [B, H, S, D] views with unit D
// stride (the ring-attention kernels read Q and K token-major, strides
// (S*H*D, D, H*D, 1)).  freqs is fp32 [B or 1, S, D] with (cos, sin)
// interleaved, i.e. torch.view_as_real of the complex [.., S, D/2] table.
//
// Mapping: LPR lanes per row (16, or 8 at D <= 64), each lane owning NCH chunks
// of 8 consecutive elements (chunk j of lane i covers elements 8*(LPR*j + i)
// ..); a row's sums are DPP adds over its lanes.  All loads are 16-byte (bf16)
// or 32-byte (fp32 freqs) per lane.
//
// The kernels are HBM-bound: per row they read and write D bf16 once.  A
// RMSNorm row's loads, sum, square root and division are one serial chain, so
// the kernels with RMSNorm walk their rows with the next loads in flight, and
// the forward takes two heads of a token at once (one RoPE row, one root and
// division for both).  Calls back to back over buffers cycled through 800 MB,
// one row group per block without a prefetch -> this, at [B,H,S,D]:
// [1,24,8192,128] forward 26.7 -> 22.8 us, backward with its reduction 42.1 ->
// 31.4 (5.0 TB/s, the rate of a large copy); [1,30,16384,128] 59.1 -> 53.2 and
// 104.8 -> 80.5; [2,16,8192,64] 31.0 -> 17.5 and 48.4 -> 24.2 (16 lanes per row
// left half of them idle); [1,30,256,128] backward 12.6 -> 9.7 (one reduction
// launch fewer).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qk_kernels.h"

namespace harp_qk {

typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// fp32 -> bf16 by truncation, as the reference stores bf16
__device__ __forceinline__ uint16_t f32_to_bf16_trunc(float f) { return (uint16_t)(__float_as_uint(f) >> 16); }
// the truncated value, kept as fp32
__device__ __forceinline__ float trunc_f32(float f) { return __uint_as_float(__float_as_uint(f) & 0xffff0000u); }

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// sum over the LPR lanes of a group, the same in every lane (each step adds
// the same two values in both partners): lanes 8 (16 per row), 4, 2 and 1
// apart, so a row's sum is the same fp32 value with 8 and with 16 lanes
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
  static_assert(LPR == 16 || LPR == 8);
  if constexpr (LPR == 16) {
    v += dpp<0x128>(v);  // row_ror:8
    v += dpp<0x124>(v);  // row_ror:4
  } else {
    v += dpp<0x1b>(dpp<0x141>(v));  // row_half_mirror, then quad_perm:[3,2,1,0]: lane ^ 4
  }
  v += dpp<0x4e>(v);  // quad_perm:[2,3,0,1]
  v += dpp<0xb1>(v);  // quad_perm:[1,0,3,2]
  return v;
}
// the value of lane r (0 <= r < 8) of the lane's group
template <int LPR, int r>
__device__ __forceinline__ float group_bcast(float v) {
  const float lo = dpp<0x150 + r>(v);  // row_newbcast:r
  if constexpr (LPR == 16) return lo;
  const float hi = dpp<0x158 + r>(v);
  return (threadIdx.x & 8) ? hi : lo;
}

// The units of a launch: (batch, token, heads u + r * hg, r < R) with u (< hg =
// ceil(H / R)) fastest, so that in the token-major layout the r-th load of
// consecutive groups reads one contiguous run, and they share one row of the
// RoPE table.  A block-uniform position is advanced in 32
// bits; only its start takes a 64-bit division.
struct UnitPos {
  uint32_t b, s, u;
};
__device__ __forceinline__ uint32_t head_groups(const QkShape& sh, int R) { return (uint32_t)(sh.H + R - 1) / R; }
__device__ __forceinline__ UnitPos unit_at(const QkShape& sh, uint32_t hg, int64_t unit) {
  const int64_t bs = unit / hg;
  UnitPos p;
  p.u = (uint32_t)(unit - bs * hg);
  p.b = (uint32_t)(bs / sh.S);
  p.s = (uint32_t)(bs - (int64_t)p.b * sh.S);
  return p;
}
__device__ __forceinline__ UnitPos unit_after(const QkShape& sh, uint32_t hg, UnitPos p, uint32_t n) {
  const uint32_t v = p.u + n, dt = v / hg, s = p.s + dt, db = s / (uint32_t)sh.S;
  return UnitPos{p.b + db, s - db * (uint32_t)sh.S, v - dt * hg};
}
__device__ __forceinline__ int64_t unit_count(const QkShape& sh, uint32_t hg) { return (int64_t)sh.B * sh.S * hg; }
__device__ __forceinline__ int64_t elem_off(const Strides4& st, const UnitPos& p, int h) {
  return (int64_t)p.b * st.b + (int64_t)h * st.h + (int64_t)p.s * st.s;
}
__device__ __forceinline__ int64_t rms_off(const QkShape& sh, const UnitPos& p, int h) {
  return ((int64_t)p.b * sh.H + h) * sh.S + p.s;
}
// One lane's chunks of a row as loaded, and as fp32
template <int NCH>
struct Raw {
  u16x8 c[NCH];
};
template <int LPR, int NCH>
__device__ __forceinline__ Raw<NCH> load_raw(const uint16_t* base, int D, int sub) {
  Raw<NCH> r;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int e0 = 8 * (LPR * j + sub);
    r.c[j] = e0 < D ? *(const u16x8*)(base + e0) : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  return r;
}
template <int NCH>
__device__ __forceinline__ void to_f32(const Raw<NCH>& r, float (&v)[NCH][8]) {
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) v[j][k] = bf16_to_f32(r.c[j][k]);
}
template <int LPR, int NCH>
__device__ __forceinline__ void store_row(uint16_t* base, int D, int sub, const float (&v)[NCH][8]) {
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int e0 = 8 * (LPR * j + sub);
    if (e0 < D) {
      u32x4 u;
#pragma unroll
      for (int k = 0; k < 4; ++k)  // the high halves of two values: truncation and packing in one v_perm
        u[k] = __builtin_amdgcn_perm(__float_as_uint(v[j][2 * k + 1]), __float_as_uint(v[j][2 * k]), 0x07060302u);
      *(u32x4*)(base + e0) = u;
    }
  }
}
// weight (bf16 or fp32) chunk as fp32; absent weight = 1.  The weight is a
// separate allocation of D elements: 16-byte loads stay inside it because D
// is a multiple of 8 and allocations are at least 16-byte aligned.
template <int LPR, int NCH>
__device__ __forceinline__ void load_weight(const void* w, int w_f32, int D, int sub, float (&v)[NCH][8]) {
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int e0 = 8 * (LPR * j + sub);
    if (!w || e0 >= D) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[j][k] = 1.f;
    } else if (w_f32) {
      const f32x4 a = *(const f32x4*)((const float*)w + e0), c = *(const f32x4*)((const float*)w + e0 + 4);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[j][k] = a[k];
        v[j][k + 4] = c[k];
      }
    } else {
      const u16x8 u = *(const u16x8*)((const uint16_t*)w + e0);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[j][k] = bf16_to_f32(u[k]);
    }
  }
}
template <int LPR, int NCH>
__device__ __forceinline__ void load_freqs(const float* f, int D, int sub, float (&v)[NCH][8]) {
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int e0 = 8 * (LPR * j + sub);
    if (e0 < D) {
      const f32x4 a = *(const f32x4*)(f + e0), c = *(const f32x4*)(f + e0 + 4);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[j][k] = a[k];
        v[j][k + 4] = c[k];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[j][k] = 0.f;
    }
  }
}

// RMSNorm forward (rms_norm.cc:39-103): a lane's share of a row's sum of squares
template <int NCH>
__device__ __forceinline__ float square_sum(const float (&v)[NCH][8]) {
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) ss = __builtin_fmaf(v[j][k], v[j][k], ss);
  return ss;
}
__device__ __forceinline__ float rms_of(float ss, int D, float eps) { return __fsqrt_rn(__fdiv_rn(ss, (float)D) + eps); }
// bf16-truncated (x * (1 / rms)) * w, kept as fp32 values
template <int NCH>
__device__ __forceinline__ void normalise(float (&v)[NCH][8], const float (&w)[NCH][8], float inv) {
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) v[j][k] = trunc_f32(__fmul_rn(__fmul_rn(v[j][k], inv), w[j][k]));
}
// RoPE of one row (rope.cc:34-38): complex multiply by f, or by conj(f)
// (rope.cc:115-134), then bf16-truncated.  The reference forms each part with
// one rounded product and one fused multiply-add.
template <int NCH, bool CONJ>
__device__ __forceinline__ void rope_row(float (&v)[NCH][8], const float (&f)[NCH][8]) {
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
      const float xr = v[j][k], xi = v[j][k + 1], fr = f[j][k], fi = f[j][k + 1];
      float re, im;
      if (CONJ) {
        re = __builtin_fmaf(xi, fi, __fmul_rn(xr, fr));
        im = __builtin_fmaf(-xr, fi, __fmul_rn(xi, fr));
      } else {
        re = __builtin_fmaf(-xi, fi, __fmul_rn(xr, fr));
        im = __builtin_fmaf(xi, fr, __fmul_rn(xr, fi));
      }
      v[j][k] = trunc_f32(re);
      v[j][k + 1] = trunc_f32(im);
    }
}

// RMSNorm backward of one row (rms_norm.cc:139-230): the lane's share of
// sum(g * xn), then dy becomes dx (fp32, not yet truncated) and wgrad
// accumulates dy * xn.
template <int NCH>
__device__ __forceinline__ float bwd_dot(const float (&x)[NCH][8], const float (&dy)[NCH][8], const float (&w)[NCH][8],
                                         float inv) {
  float dot = 0.f;
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) dot = __builtin_fmaf(__fmul_rn(dy[j][k], w[j][k]), __fmul_rn(x[j][k], inv), dot);
  return dot;
}
template <int NCH>
__device__ __forceinline__ void bwd_apply(const float (&x)[NCH][8], float (&dy)[NCH][8], const float (&w)[NCH][8],
                                          float inv, float coeff, float (&wgrad)[NCH][8]) {
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float xn = __fmul_rn(x[j][k], inv);
      const float g = __fmul_rn(dy[j][k], w[j][k]);
      wgrad[j][k] = __builtin_fmaf(dy[j][k], xn, wgrad[j][k]);
      dy[j][k] = __fmul_rn(__fsub_rn(g, __fmul_rn(xn, coeff)), inv);
    }
}

// A lane's R values, one per row of the unit -> the value of row `sub` on lane
// sub (any value on the other lanes), and back: row r's value from lane r
template <int R>
__device__ __forceinline__ float pick(const float (&v)[R], int sub) {
  float x = v[0];
#pragma unroll
  for (int r = 1; r < R; ++r) x = sub == r ? v[r] : x;
  return x;
}
template <int LPR, int R, int r = 0>
__device__ __forceinline__ void spread(float v, float (&out)[R]) {
  if constexpr (r < R) {
    out[r] = group_bcast<LPR, r>(v);
    spread<LPR, R, r + 1>(v, out);
  }
}

// The steps (kGroups units each) of a block: begin, begin + stride, .. below
// end.  Workgroups are dealt to the 8 XCDs round-robin; each XCD takes one
// contiguous range of the steps, so that a token's rows, its RoPE table row
// and the neighbouring rms entries of a head are fetched into, and merged in,
// one L2, and its blocks take the range's steps in turn, so that what runs at
// one time is one contiguous window of memory.
struct Steps {
  int64_t begin, end;
  uint32_t stride;
};
__device__ __forceinline__ Steps block_steps(int64_t steps) {
  const uint32_t nx = min(gridDim.x, 8u), x = blockIdx.x % nx, local = blockIdx.x / nx;
  return Steps{steps * x / nx + local, steps * (x + 1) / nx, (gridDim.x - x + nx - 1) / nx};
}

// ---------------------------------------------------------------------------
// Forward: RMSNorm, then (ROPE) RoPE; the intermediate is truncated to bf16
// exactly as between the two reference ops.  A block walks its steps with the
// next step's loads in flight while it works on the current one.
// ---------------------------------------------------------------------------
template <int LPR, int NCH, bool ROPE, int R>
__global__ __launch_bounds__(256) void qk_forward_kernel(QkFwdParams p) {
  constexpr int kGroups = 256 / LPR;
  const int grp = threadIdx.x / LPR, sub = threadIdx.x % LPR;
  const uint32_t hg = head_groups(p.sh, R);
  const int64_t units = unit_count(p.sh, hg);
  const Steps st = block_steps((units + kGroups - 1) / kGroups);
  if (st.begin >= st.end || st.begin * kGroups + grp >= units) return;  // whole groups exit together
  float w[NCH][8];
  load_weight<LPR, NCH>(p.weight, p.weight_f32, p.sh.D, sub, w);
  // a row past H repeats the unit's first one and is not stored
  auto ok = [&](const UnitPos& u, int r) { return (int)(u.u + r * hg) < p.sh.H; };
  auto head = [&](const UnitPos& u, int r) { return (int)(ok(u, r) ? u.u + r * hg : u.u); };
  Raw<NCH> raw[R];
  float f[NCH][8];
  auto load = [&](const UnitPos& u) {
#pragma unroll
    for (int r = 0; r < R; ++r) raw[r] = load_raw<LPR, NCH>(p.x + elem_off(p.sx, u, head(u, r)), p.sh.D, sub);
    if (ROPE)
      load_freqs<LPR, NCH>(p.freqs + (int64_t)u.b * p.f_stride_b + (int64_t)u.s * p.f_stride_s, p.sh.D, sub, f);
  };
  UnitPos pos = unit_after(p.sh, hg, unit_at(p.sh, hg, st.begin * kGroups), grp);
  load(pos);
  for (int64_t si = st.begin;; si += st.stride) {
    const UnitPos cur = pos;
    float v[R][NCH][8], fc[NCH][8];
#pragma unroll
    for (int r = 0; r < R; ++r) to_f32(raw[r], v[r]);
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
      for (int k = 0; k < 8; ++k) fc[j][k] = f[j][k];
    // only the last step of all is short, so the groups of a wave leave the
    // loop together or have no later step of their own
    const bool more = si + st.stride < st.end && (si + st.stride) * kGroups + grp < units;
    if (more) {
      pos = unit_after(p.sh, hg, pos, kGroups * st.stride);
      load(pos);
    }
    float ss[R], inv[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ss[r] = group_sum<LPR>(square_sum(v[r]));
    const float rms = rms_of(pick<R>(ss, sub), p.sh.D, p.eps);
    if (sub < R && ok(cur, sub) && p.rms) p.rms[rms_off(p.sh, cur, head(cur, sub))] = rms;
    spread<LPR, R>(__fdiv_rn(1.f, rms), inv);
#pragma unroll
    for (int r = 0; r < R; ++r) normalise(v[r], w, inv[r]);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (ROPE) rope_row<NCH, false>(v[r], fc);
      if (ok(cur, r)) store_row<LPR, NCH>(p.out + elem_off(p.so, cur, head(cur, r)), p.sh.D, sub, v[r]);
    }
    if (!more) break;
  }
}

// ---------------------------------------------------------------------------
// Backward: (ROPE) RoPE backward, then RMSNorm backward, one row per group and
// step, walked as the forward (two rows a step took 129 registers and was
// 5-10% slower).  Each block writes its fp32 weight-gradient partial sums to
// wpart[block][D]; the partials are summed in a second kernel (deterministic,
// no atomics).
// ---------------------------------------------------------------------------
template <int LPR, int NCH, bool ROPE>
__global__ __launch_bounds__(256) void qk_backward_kernel(QkBwdParams p) {
  constexpr int kGroups = 256 / LPR;
  __shared__ float wsum[kGroups][LPR * NCH * 8 + 4];
  const int grp = threadIdx.x / LPR, sub = threadIdx.x % LPR;
  const uint32_t hg = (uint32_t)p.sh.H;
  const int64_t units = unit_count(p.sh, hg);
  const Steps st = block_steps((units + kGroups - 1) / kGroups);
  float wg[NCH][8], w[NCH][8];
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) wg[j][k] = 0.f;
  if (st.begin < st.end && st.begin * kGroups + grp < units) {
    load_weight<LPR, NCH>(p.weight, p.weight_f32, p.sh.D, sub, w);
    Raw<NCH> rg, rx;
    float f[NCH][8], rms = 1.f;
    auto load = [&](const UnitPos& u) {
      rg = load_raw<LPR, NCH>(p.dy + elem_off(p.sdy, u, (int)u.u), p.sh.D, sub);
      rx = load_raw<LPR, NCH>(p.x + elem_off(p.sx, u, (int)u.u), p.sh.D, sub);
      rms = p.rms[rms_off(p.sh, u, (int)u.u)];
      if (ROPE)
        load_freqs<LPR, NCH>(p.freqs + (int64_t)u.b * p.f_stride_b + (int64_t)u.s * p.f_stride_s, p.sh.D, sub, f);
    };
    UnitPos pos = unit_after(p.sh, hg, unit_at(p.sh, hg, st.begin * kGroups), grp);
    load(pos);
    for (int64_t si = st.begin;; si += st.stride) {
      const UnitPos cur = pos;
      float g[NCH][8], x[NCH][8];
      to_f32(rg, g);
      to_f32(rx, x);
      if (ROPE) rope_row<NCH, true>(g, f);
      const float inv = __fdiv_rn(1.f, rms);
      const bool more = si + st.stride < st.end && (si + st.stride) * kGroups + grp < units;
      if (more) {
        pos = unit_after(p.sh, hg, pos, kGroups * st.stride);
        load(pos);
      }
      const float coeff = __fdiv_rn(group_sum<LPR>(bwd_dot(x, g, w, inv)), (float)p.sh.D);
      bwd_apply(x, g, w, inv, coeff, wg);
      store_row<LPR, NCH>(p.dx + elem_off(p.sdx, cur, (int)cur.u), p.sh.D, sub, g);
      if (!more) break;
    }
  }
  // block partial of the weight gradient: sum the groups through LDS
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) wsum[grp][8 * (LPR * j + sub) + k] = wg[j][k];
  __syncthreads();
  for (int e = threadIdx.x; e < p.sh.D; e += 256) {
    float acc = 0.f;
#pragma unroll
    for (int gi = 0; gi < kGroups; ++gi) acc += wsum[gi][e];
    p.wpart[(int64_t)blockIdx.x * p.sh.D + e] = acc;
  }
}

// ---------------------------------------------------------------------------
// RoPE alone, forward and (CONJ) backward: one row per group, no walk.  There
// is no chain to hide, and one short block per 16 or 32 rows streams better
// than the walk does ([1,30,16384,128]: 45 us, 5.5 TB/s, against 51).
// ---------------------------------------------------------------------------
template <int LPR, int NCH, bool CONJ>
__global__ __launch_bounds__(256) void rope_kernel(RopeParams p) {
  const int64_t q = gridDim.x / 8, r = gridDim.x % 8, x = blockIdx.x % 8, local = blockIdx.x / 8;
  const int64_t blk = x < r ? x * (q + 1) + local : r * (q + 1) + (x - r) * q + local;  // XCD ranges, as block_steps
  const int sub = threadIdx.x % LPR;
  const int64_t row = blk * (256 / LPR) + threadIdx.x / LPR;
  if (row >= (int64_t)p.sh.B * p.sh.H * p.sh.S) return;
  const int64_t bs = row / p.sh.H;
  const int h = (int)(row - bs * p.sh.H);
  UnitPos u;
  u.b = (uint32_t)(bs / p.sh.S);
  u.s = (uint32_t)(bs - (int64_t)u.b * p.sh.S);
  float v[NCH][8], f[NCH][8];
  to_f32(load_raw<LPR, NCH>(p.x + elem_off(p.sx, u, h), p.sh.D, sub), v);
  load_freqs<LPR, NCH>(p.freqs + (int64_t)u.b * p.f_stride_b + (int64_t)u.s * p.f_stride_s, p.sh.D, sub, f);
  rope_row<NCH, CONJ>(v, f);
  store_row<LPR, NCH>(p.out + elem_off(p.so, u, h), p.sh.D, sub, v);
}

// grad_weight[e] = sum over blocks of wpart[block][e], in one launch with a
// fixed order (so the result is deterministic), stored as fp32 or bf16
// (truncated, like the reference's other bf16 stores).  A launch behind
// another costs about 4.5 us here whatever it does: with at most
// kQkBwdMaxLaunch rows one launch ends sooner than two levels of 64-row groups
// did (12.6 -> 9.7 us for the whole backward at 30 heads x 256 rows).  Block x
// sums columns 8x .. 8x + 7 with 128 row lanes, each taking every 128th row (at
// most kQkBwdMaxLaunch / 128 independent loads in flight per thread), and LDS
// adds the lane sums in order.  (The order, and so the last bit, of a weight
// gradient depends on the number of partial rows; y, rms and dx depend on
// neither the grid nor the lanes per row.)
constexpr int kWgCols = 8, kWgLanes = 128;
__global__ __launch_bounds__(kWgCols* kWgLanes) void wgrad_sum_kernel(const float* src, int nrows, int D, void* dst,
                                                                      int dst_f32) {
  __shared__ float part[kWgLanes][kWgCols + 1];
  const int tx = threadIdx.x % kWgCols, ty = threadIdx.x / kWgCols;
  const int e = blockIdx.x * kWgCols + tx;  // D is a multiple of 8
  float acc = 0.f;
#pragma unroll 4
  for (int i = ty; i < nrows; i += kWgLanes) acc += src[(int64_t)i * D + e];
  part[ty][tx] = acc;
  __syncthreads();
  // 128 lane sums -> 8 per column -> 1, both in lane order
  if (ty < 8) {
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < kWgLanes / 8; ++k) v += part[ty * (kWgLanes / 8) + k][tx];
    acc = v;
  }
  __syncthreads();
  if (ty < 8) part[ty][tx] = acc;
  __syncthreads();
  if (ty != 0) return;
  float v = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) v += part[k][tx];
  if (dst_f32) ((float*)dst)[e] = v;
  else ((uint16_t*)dst)[e] = f32_to_bf16_trunc(v);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
// Lanes per row, heads per unit (forward) and blocks.  Two heads once the
// units still fill kFillBlocks blocks (smaller calls spread over the chip, one
// head per group) and unless an odd H leaves more than 1 lane in 8 idle; at
// most max_blocks blocks, as few as leave the busiest one no more steps.
constexpr int64_t kFillBlocks = 1024;
struct Plan {
  int lpr, R, blocks;
};
static Plan plan(const QkShape& sh, bool pairs, int64_t max_blocks) {
  Plan q;
  q.lpr = sh.D > 64 ? 16 : 8;
  const int64_t hg2 = (sh.H + 1) / 2, units2 = (int64_t)sh.B * sh.S * hg2;
  q.R = pairs && sh.D <= 128 && hg2 * 2 * 7 <= (int64_t)sh.H * 8 && units2 * q.lpr / 256 >= kFillBlocks ? 2 : 1;
  const int64_t units = q.R == 2 ? units2 : (int64_t)sh.B * sh.S * sh.H;
  const int64_t steps = (units * q.lpr + 255) / 256, per = (steps + max_blocks - 1) / max_blocks;
  q.blocks = (int)((steps + per - 1) / per);
  return q;
}

template <int LPR, int NCH, bool CONJ>
static hipError_t rope_t(const RopeParams& p, hipStream_t st) {
  const int64_t rows = (int64_t)p.sh.B * p.sh.H * p.sh.S;
  const dim3 grid((unsigned)((rows * LPR + 255) / 256));
  hipLaunchKernelGGL((rope_kernel<LPR, NCH, CONJ>), grid, dim3(256), 0, st, p);
  return hipGetLastError();
}
template <bool CONJ>
static hipError_t launch_rope(const RopeParams& p, hipStream_t st) {
  if (p.sh.D > 128) return rope_t<16, 2, CONJ>(p, st);
  return p.sh.D > 64 ? rope_t<16, 1, CONJ>(p, st) : rope_t<8, 1, CONJ>(p, st);
}

template <int LPR, int NCH, int R>
static hipError_t fwd_t(const QkFwdParams& p, int mode, int blocks, hipStream_t st) {
  const dim3 grid((unsigned)blocks), block(256);
  if (mode == 1) hipLaunchKernelGGL((qk_forward_kernel<LPR, NCH, false, R>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((qk_forward_kernel<LPR, NCH, true, R>), grid, block, 0, st, p);
  return hipGetLastError();
}
hipError_t launch_qk_forward(const QkFwdParams& p, int mode, hipStream_t st) {
  if (mode == 2) return launch_rope<false>(RopeParams{p.sh, p.x, p.sx, p.out, p.so, p.freqs, p.f_stride_b, p.f_stride_s}, st);
  const Plan q = plan(p.sh, true, kQkFwdMaxLaunch);
  if (p.sh.D > 128) return fwd_t<16, 2, 1>(p, mode, q.blocks, st);
  if (p.sh.D > 64) return q.R == 2 ? fwd_t<16, 1, 2>(p, mode, q.blocks, st) : fwd_t<16, 1, 1>(p, mode, q.blocks, st);
  return q.R == 2 ? fwd_t<8, 1, 2>(p, mode, q.blocks, st) : fwd_t<8, 1, 1>(p, mode, q.blocks, st);
}

int bwd_blocks(const QkShape& sh) {
  const int64_t rows = (int64_t)sh.B * sh.H * sh.S;
  const int64_t need = (rows + 15) / 16;
  return (int)(need < kQkBwdMaxBlocks ? need : kQkBwdMaxBlocks);
}
int bwd_launch_blocks(const QkShape& sh) { return plan(sh, false, kQkBwdMaxLaunch).blocks; }

template <int LPR, int NCH>
static hipError_t bwd_t(const QkBwdParams& p, int mode, hipStream_t st) {
  const dim3 grid((unsigned)bwd_launch_blocks(p.sh)), block(256);
  if (mode == 1) hipLaunchKernelGGL((qk_backward_kernel<LPR, NCH, false>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((qk_backward_kernel<LPR, NCH, true>), grid, block, 0, st, p);
  return hipGetLastError();
}
hipError_t launch_qk_backward(const QkBwdParams& p, int mode, hipStream_t st) {
  if (mode == 2) return launch_rope<true>(RopeParams{p.sh, p.dy, p.sdy, p.dx, p.sdx, p.freqs, p.f_stride_b, p.f_stride_s}, st);
  if (p.sh.D > 128) return bwd_t<16, 2>(p, mode, st);
  return p.sh.D > 64 ? bwd_t<16, 1>(p, mode, st) : bwd_t<8, 1>(p, mode, st);
}

hipError_t launch_wgrad_reduce(const float* wpart, int nblk, int D, void* gw, int gw_f32, hipStream_t st) {
  hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)(D / kWgCols)), dim3(kWgCols * kWgLanes), 0, st, wpart, nblk, D,
                     gw, gw_f32);
  return hipGetLastError();
}

}  // namespace harp_qk
