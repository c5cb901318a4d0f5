// r4.hip -- Q4R4 / Q8R4 matmuls: 4-row blocks, groups of 32, f16 group
// scales, group-32 int8 activations.
//
// Reference: hw/hw_q4r4.h (format, kernels), nn/quant.c:110-179 (packers),
// nn/matmul.c:365-466 (moty_matmul_q4r4_s / moty_matmul_q8r4_s).
//
// Layout (unchanged from the reference): weight rows in blocks of 4; per
// (block, group) Q4R4 stores 64 bytes = 4 rows x 16 bytes, row byte j =
// c[j] | c[j+16] << 4 with codes c = v + 8 in 0..15; Q8R4 stores 128 bytes =
// 4 rows x 32 signed codes.  Scales: f16 [block][group][4].
//
// Activations: per group of 32, s = amax/127 (clamped at 1e-30), q =
// rint(x/s) and the code sum xsum (hw/hw_q4r4.h:36-46).
//
// Arithmetic, as the reference's x86 build evaluates it (its portable
// kernels are the scalar references): per output, groups in order,
//   tokens t < 4*floor(S/4) (the 4-token tile kernel):
//       s = sum c*x;  acc = fma(s, dd*xs, acc);  acc = fma(-dd, (8*xsum)*xs, acc)
//   the remaining tokens (the per-token kernel):
//       s = sum c*x - 8*xsum;  acc = fma(s, dd*xs, acc)
//   Q8R4 (no offset): acc = fma(sum c*x, dd*xs, acc).
// The integer group sums are exact, so only the float chain's order is
// fixed; the kernels below keep it.
#include "common.h"
#include "kernels.h"

#include <type_traits>

namespace moty {

// ---------------------------------------------------------------------------
// Group-32 activation quantization: a lane pair per group, 16 elements
// (4 float4) per lane.  Each lane reduces its half in registers; one
// exchange with the partner lane joins amax and the code sum, so the scale's
// two divisions run once per half group.  The arithmetic per element is the
// reference's: s = amax/127 (at least 1e-30), q = rint(x * (1/s)).
// Returns the group's code sum; q gets the lane's 16 codes, s the scale.
__device__ __forceinline__ int quant_half_g32(const float4 (&v)[4], uint4& q, float& s) {
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < 4; j++)
    amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[j].x), fabsf(v[j].y)), fmaxf(fabsf(v[j].z), fabsf(v[j].w))));
  amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
  s = amax / 127.f;
  if (s < 1e-30f) s = 1e-30f;
  const float inv = 1.f / s;
  int sum = 0;
  uint32_t w[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int a = rne_int(v[j].x * inv), b = rne_int(v[j].y * inv), c = rne_int(v[j].z * inv),
              d = rne_int(v[j].w * inv);
    sum += a + b + c + d;
    w[j] = (uint32_t)(a & 0xff) | ((uint32_t)(b & 0xff) << 8) | ((uint32_t)(c & 0xff) << 16) |
           ((uint32_t)(d & 0xff) << 24);
  }
  q = make_uint4(w[0], w[1], w[2], w[3]);
  return sum + __shfl_xor(sum, 1, 64);
}

// One lane per 16 elements of a row: lanes 2i, 2i+1 share group i.
__global__ __launch_bounds__(256) void k_quant_g32(const float* __restrict__ x, int8_t* __restrict__ xq,
                                                   float* __restrict__ xs, int32_t* __restrict__ xm, int I) {
  const int64_t row = blockIdx.y;
  const int e = (blockIdx.x * 256 + threadIdx.x) * 16;
  const bool ok = e < I;
  const float4* src = (const float4*)(x + row * I + (ok ? e : 0));
  float4 v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = sel4(ok, src[j]);
  uint4 q;
  float s;
  const int sum = quant_half_g32(v, q, s);
  if (!ok) return;
  *(uint4*)(xq + row * I + e) = q;
  if ((threadIdx.x & 1) == 0) {
    const int nb = I / 32;
    xs[row * nb + e / 32] = s;
    xm[row * nb + e / 32] = sum;
  }
}

int launch_quant_g32(const float* x, int8_t* xq, float* xs, int32_t* xm, int S, int I, hipStream_t st) {
  if (S <= 0) return MOTY_OK;
  if (I % 32) return MOTY_EUNSUP;
  hipLaunchKernelGGL(k_quant_g32, dim3((I + 4095) / 4096, S), dim3(256), 0, st, x, xq, xs, xm, I);
  LAUNCH_TRY("k_quant_g32");
  return MOTY_OK;
}

// low / high nibbles of 16 packed Q4R4 bytes as 16 + 16 unsigned int8 codes
__device__ __forceinline__ int4 r4_lo(int4 w) {
  return int4{w.x & 0x0f0f0f0f, w.y & 0x0f0f0f0f, w.z & 0x0f0f0f0f, w.w & 0x0f0f0f0f};
}
__device__ __forceinline__ int4 r4_hi(int4 w) {
  return int4{(w.x >> 4) & 0x0f0f0f0f, (w.y >> 4) & 0x0f0f0f0f, (w.z >> 4) & 0x0f0f0f0f, (w.w >> 4) & 0x0f0f0f0f};
}

// ---------------------------------------------------------------------------
// Decode GEMV, S_ <= 3 tokens (all in the per-token kernel's form), I <=
// 1024*IC.  KS waves share one 4-row block, split along K: chunk index kk
// (64 lanes x 16 bytes, GPC groups) belongs to part kk % KS, so a block
// count near the SIMD count still puts several waves on every SIMD.  The
// activation rows are loaded and land first; the weight chunks of the part
// (each load instruction reads 1 KiB of the contiguous block) and the f16
// scale of each chunk's (row, group) are then kept PD chunks ahead of the
// one being consumed.  The workgroup quantizes the activation rows into LDS
// from registers (every workgroup derives the same codes).  Each lane forms
// the exact integer group sums of its chunks (Q8R4: half a row per chunk,
// the halves joined across the lane pair) and parks the two operands of the
// chain step, (s - 8*xsum, dd*xs), in the block's LDS slice
// ([row][token][group]); after its k-th chunk a part raises its progress
// flag to k+1.  One lane per (row, token) of part 0 runs acc = fma(a, b,
// acc) over the groups in order, chunk index by chunk index, each one as
// soon as its part's flag says it is parked.  Only part 0 ever waits, on
// flags that every other part raises unconditionally, so every wait ends.
template <bool Q8, int S_, int IC, int NT, bool PAIR = false, int KS = 1>
__global__ __launch_bounds__(NT) void k_r4_gemv(const float* __restrict__ x, const uint8_t* __restrict__ W,
                                                const uint16_t* __restrict__ d16, float* __restrict__ y, int S,
                                                int I, int O) {
  static_assert(!PAIR || S_ == 1, "the fused gate/up form serves one token");
  constexpr int NM = PAIR ? 2 : 1;  // matrices: gate (and up)
  constexpr int GB = Q8 ? 128 : 64;        // bytes per (block, group)
  constexpr int NCH = IC * (Q8 ? 4 : 2);   // chunk indices per block
  static_assert(NCH % KS == 0, "K parts of whole chunks");
  constexpr int NCW = NCH / KS;            // chunks per lane per wave
  // chunks in flight ahead of the one consumed: one for a single token (the
  // C3 shapes on MI355X: 4096 x 12288 9.5 us against 10.9 with four ahead,
  // the fused 2 x 12288 x 4096 gate_up 11.6 against 13.7 -- each row's chain
  // then keeps pace with its data), four for more tokens
  constexpr int PD = S_ == 1 ? 1 : (NCW < 4 ? NCW : 4);
  constexpr int P0 = PD < 2 ? PD : 2;      // of them issued before the quantization
  constexpr int GPC = Q8 ? 8 : 16;         // groups per chunk index
  constexpr int WAVES = NT / MOTY_WAVE;
  static_assert(WAVES % KS == 0, "whole blocks per workgroup");
  constexpr int BPW = WAVES / KS;          // blocks per workgroup
  constexpr int XU = (IC * 64 + NT - 1) / NT;  // activation half groups (16 floats) per thread per row
  extern __shared__ __align__(16) int8_t lds[];
  __shared__ int flag_s[BPW * KS];
  const int nb = I / 32, O4 = (O + 3) / 4;
  const int lane = threadIdx.x % MOTY_WAVE, wv = threadIdx.x / MOTY_WAVE;
  const int part = wv % KS, bw = wv / KS;
  // LDS: xq [S_][I] | xs [S_][nb] | xm [S_][nb] | per block: operands [NM*4][S_][nb] float2
  int8_t* xq_s = lds;
  float* xs_s = (float*)(lds + S_ * I);
  int* xm_s = (int*)(xs_s + S_ * nb);
  // operand rows padded to an even length past nb: the four rows of a
  // block that lanes 4g..4g+3 write land in distinct banks (rows nb apart
  // shared banks: 8-16 % of LDS cycles in bank conflicts)
  const int ldo = nb + 2 - (nb & 1);
  float2* op_s = (float2*)(xm_s + S_ * nb) + (size_t)bw * (4 * NM * S_ * ldo);
  int blk = blockIdx.x * BPW + bw;
  const bool live = blk < O4;
  blk = live ? blk : O4 - 1;

  // 1. activation rows
  float4 xr[S_][XU][4];
#pragma unroll
  for (int t = 0; t < S_; t++)
#pragma unroll
    for (int c = 0; c < XU; c++) {
      const int e = (c * NT + threadIdx.x) * 16;
      const float4* src = (const float4*)(x + (size_t)(t < S ? t : 0) * I + (e < I ? e : 0));
#pragma unroll
      for (int j = 0; j < 4; j++) xr[t][c][j] = src[j];
    }
  if (KS > 1 && threadIdx.x < BPW * KS) flag_s[threadIdx.x] = 0;

  // 2. weight chunks of the part and their scales, PD chunks ahead: chunk
  // k + PD is issued just before chunk k is consumed, so the integer dots
  // and the chain run while the stream is still arriving (a wave that
  // issued all of its loads first would sit in the issue stall until the
  // memory path had taken them all).  The activation rows land first (the
  // wait and the bare barrier: queued behind the weight stream in the CU's
  // load path and in L2 they would arrive with it), then the first P0
  // chunks go out before the quantization, the rest of the PD after it.
  // PAIR: W is the row-fused [gate; up] matrix (moty_mat_fuse_rows), the up
  // rows' blocks start O/4 blocks after the gate rows'
  const int nchunk = nb * GB / 16;
  int4 wc[NM][NCW];
  uint16_t dc[NM][NCW];
  auto issue = [&](int k) {
#pragma unroll
    for (int m = 0; m < NM; m++) {
      const int ci = lane + 64 * (k * KS + part);
      const int cc = ci < nchunk ? ci : 0;
      {
        const v4i t = __builtin_nontemporal_load((const v4i*)(W + ((size_t)(blk + m * O4) * nb * GB + (size_t)cc * 16)));
        wc[m][k] = int4{t.x, t.y, t.z, t.w};
      }
      // chunk ci: group ci/4, row ci%4 (Q8R4: group ci/8, row (ci/2)%4)
      dc[m][k] = __builtin_nontemporal_load(d16 + (size_t)(blk + m * O4) * nb * 4 + (Q8 ? (cc >> 3) * 4 + ((cc >> 1) & 3) : cc));
    }
  };
  MOTY_WAIT_VMCNT(0);
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int k = 0; k < P0; k++) issue(k);
  __builtin_amdgcn_sched_barrier(0);

  // 3. group-32 quantization of the activation rows into LDS (k_quant_g32's
  // arithmetic)
#pragma unroll
  for (int t = 0; t < S_; t++)
#pragma unroll
    for (int c = 0; c < XU; c++) {
      const int e = (c * NT + threadIdx.x) * 16;
      const bool ok = e < I;
      float4 v[4];
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = sel4(ok, xr[t][c][j]);
      uint4 q;
      float sc;
      const int sum = quant_half_g32(v, q, sc);
      if (ok) {
        *(uint4*)(xq_s + t * I + e) = q;
        if ((threadIdx.x & 1) == 0) {
          xs_s[t * nb + e / 32] = sc;
          xm_s[t * nb + e / 32] = sum;
        }
      }
    }
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int k = P0; k < PD; k++) issue(k);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();

  // 4. per chunk: the exact integer group sum and the chain step's
  // operands; then part 0's lane (m*4 + r)*S_ + t continues row r's chain
  // for token t (PAIR: m = 1 is the up row) over chunk indices k*KS ..
  // k*KS + KS-1 in order, while later chunks may still be in flight.
  // part 0 carries the serial chain: its wave gets the SIMD's issue
  // priority over the parts that only form group sums
  if (KS > 1 && part == 0) __builtin_amdgcn_s_setprio(3);
  const bool chain = part == 0 && lane < 4 * NM * S_;
  const float2* opc = op_s + (lane < 4 * NM * S_ ? lane : 0) * ldo;  // lane = (m*4 + r)*S_ + t
  const bool even = (nb & 1) == 0;  // 16-byte reads of two groups' operands stay aligned
  float acc = 0.f;
#pragma unroll
  for (int k = 0; k < NCW; k++) {
    if (k + PD < NCW) issue(k + PD);
    __builtin_amdgcn_sched_barrier(0);
    const int ci = lane + 64 * (k * KS + part);
    const int g = Q8 ? (ci >> 3) : (ci >> 2), r = Q8 ? ((ci >> 1) & 3) : (ci & 3), h = Q8 ? (ci & 1) : 0;
    const bool ok = ci < nchunk;
    const int gc = ok ? g : 0;
#pragma unroll
    for (int m = 0; m < NM; m++) {
      const float dd = f16_to_f32(dc[m][k]);
#pragma unroll
      for (int t = 0; t < S_; t++) {
        const int8_t* xg = xq_s + t * I + gc * 32;
        int sacc;
        if (Q8) {
          sacc = dot16(wc[m][k], *(const int4*)(xg + 16 * h), 0);
          sacc += __shfl_xor(sacc, 1, 64);  // the row's other half: lanes 2i, 2i+1 hold (g, r, h = 0/1)
        } else {
          sacc = dot16(r4_lo(wc[m][k]), *(const int4*)xg, dot16(r4_hi(wc[m][k]), *(const int4*)(xg + 16), 0));
          sacc -= 8 * xm_s[t * nb + gc];
        }
        if (ok && h == 0) op_s[((m * 4 + r) * S_ + t) * ldo + g] = float2{(float)sacc, dd * xs_s[t * nb + gc]};
      }
    }
    if (KS > 1 && part != 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if (lane == 0) __hip_atomic_store(&flag_s[bw * KS + part], k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      continue;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (chain) {
#pragma unroll
      for (int p = 0; p < KS; p++) {
        if (p > 0) {
          while (__hip_atomic_load(&flag_s[bw * KS + p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= k)
            __builtin_amdgcn_s_sleep(1);
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
        const int g0 = (k * KS + p) * GPC, g1 = nb < g0 + GPC ? nb : g0 + GPC;
        if (g1 - g0 == GPC && even) {
          const float4* p4 = (const float4*)(opc + g0);
          float4 v[GPC / 2];
#pragma unroll
          for (int u = 0; u < GPC / 2; u++) v[u] = p4[u];
#pragma unroll
          for (int u = 0; u < GPC / 2; u++) {
            acc = __fmaf_rn(v[u].x, v[u].y, acc);
            acc = __fmaf_rn(v[u].z, v[u].w, acc);
          }
        } else {
          for (int gg = g0; gg < g1; gg++) acc = __fmaf_rn(opc[gg].x, opc[gg].y, acc);
        }
      }
    }
  }
  if (part != 0) return;
  if (PAIR) {
    const float u = __shfl(acc, (lane + 4) & 63, 64);
    const int o = blk * 4 + lane;
    if (live && lane < 4 && o < O) y[o] = ref_silu_mul(acc, u);
  } else if (lane < 4 * S_) {
    // lane = r*S_ + t
    const int r = lane / S_, t = lane % S_;
    const int o = blk * 4 + r;
    if (live && t < S && o < O) y[(size_t)t * O + o] = acc;
  }
}

template <int S_, int NT, bool PAIR, int KS>
static size_t r4_gemv_lds(int I) {
  const int nb = I / 32;
  const int ldo = nb + 2 - (nb & 1);
  return (size_t)S_ * I + (size_t)S_ * nb * 8 + (size_t)(NT / MOTY_WAVE / KS) * 4 * (PAIR ? 2 : 1) * S_ * ldo * 8;
}

template <bool Q8, int S_, int IC, int NT, bool PAIR, int KS>
static int go_r4_gemv(const float* x, const uint8_t* W, const uint16_t* d16, float* y, int S, int I, int O,
                      hipStream_t st) {
  const int O4 = (O + 3) / 4, bpw = NT / MOTY_WAVE / KS;
  const size_t lds = r4_gemv_lds<S_, NT, PAIR, KS>(I);
  if (lds + 256 > 64 * 1024) return MOTY_EUNSUP;  // 256: the static progress flags
  hipLaunchKernelGGL((k_r4_gemv<Q8, S_, IC, NT, PAIR, KS>), dim3((unsigned)((O4 + bpw - 1) / bpw)), dim3(NT), lds,
                     st, x, W, d16, y, S, I, O);
  LAUNCH_TRY("k_r4_gemv");
  return MOTY_OK;
}

// Waves per block: K is split until the blocks give every SIMD (1024 on the
// chip) about four waves, within the chunks a lane holds.  Workgroups of
// 4 * KS... waves as the LDS allows.
template <bool Q8, int S_, int IC, bool PAIR>
static int go_r4_gemv_nt(const float* x, const uint8_t* W, const uint16_t* d16, float* y, int S, int I, int O,
                         hipStream_t st) {
  constexpr int NCH = IC * (Q8 ? 4 : 2);
  const int O4 = (O + 3) / 4;
  if constexpr (NCH % 4 == 0 && NCH >= 8) {
    if (O4 <= 1024) {
      int rc = go_r4_gemv<Q8, S_, IC, 1024, PAIR, 4>(x, W, d16, y, S, I, O, st);
      if (rc != MOTY_EUNSUP) return rc;
      rc = go_r4_gemv<Q8, S_, IC, 512, PAIR, 4>(x, W, d16, y, S, I, O, st);
      if (rc != MOTY_EUNSUP) return rc;
    }
  }
  if constexpr (NCH % 2 == 0 && NCH >= 4) {
    if (O4 <= 2048) {
      int rc = go_r4_gemv<Q8, S_, IC, 512, PAIR, 2>(x, W, d16, y, S, I, O, st);
      if (rc != MOTY_EUNSUP) return rc;
      rc = go_r4_gemv<Q8, S_, IC, 256, PAIR, 2>(x, W, d16, y, S, I, O, st);
      if (rc != MOTY_EUNSUP) return rc;
    }
  }
  int rc = go_r4_gemv<Q8, S_, IC, 256, PAIR, 1>(x, W, d16, y, S, I, O, st);
  if (rc != MOTY_EUNSUP) return rc;
  return go_r4_gemv<Q8, S_, IC, 128, PAIR, 1>(x, W, d16, y, S, I, O, st);
}

// instances: activation float4 per thread and weight chunks per lane stay
// within a register budget (S_ * IC <= 16, Q8R4 IC <= 8; PAIR IC <= 8)
template <bool Q8, int S_, bool PAIR = false>
static int go_r4_gemv_ic(const float* x, const uint8_t* W, const uint16_t* d16, float* y, int S, int I, int O,
                         hipStream_t st) {
  const int ic = (I + 1023) / 1024;
  if (ic <= 1) return go_r4_gemv_nt<Q8, S_, 1, PAIR>(x, W, d16, y, S, I, O, st);
  if (ic <= 2) return go_r4_gemv_nt<Q8, S_, 2, PAIR>(x, W, d16, y, S, I, O, st);
  if (ic <= 4) return go_r4_gemv_nt<Q8, S_, 4, PAIR>(x, W, d16, y, S, I, O, st);
  if constexpr (S_ <= 2 && !(Q8 && PAIR)) {
    if (ic <= 8) return go_r4_gemv_nt<Q8, S_, 8, PAIR>(x, W, d16, y, S, I, O, st);
  }
  if constexpr (!Q8 && !PAIR && S_ == 1) {
    if (ic <= 12) return go_r4_gemv_nt<Q8, S_, 12, PAIR>(x, W, d16, y, S, I, O, st);
    if (ic <= 16) return go_r4_gemv_nt<Q8, S_, 16, PAIR>(x, W, d16, y, S, I, O, st);
  }
  return MOTY_EUNSUP;
}

template <bool Q8>
static int launch_r4_gemv(const float* x, const uint8_t* W, const uint16_t* d16, float* y, int S, int I, int O,
                          hipStream_t st) {
  switch (S) {
    case 1: return go_r4_gemv_ic<Q8, 1>(x, W, d16, y, S, I, O, st);
    case 2: return go_r4_gemv_ic<Q8, 2>(x, W, d16, y, S, I, O, st);
    case 3: return go_r4_gemv_ic<Q8, 3>(x, W, d16, y, S, I, O, st);
  }
  return MOTY_EUNSUP;  // S = 4 is the reference's 4-token tile: the GEMM path
}

// ---------------------------------------------------------------------------
// Prefill GEMM on int8 MFMA, one per group (K = 32 = the group), so each
// group's integer sum comes out separately and is folded into the float chain
// per output in group order:
//   acc = fma(float(s + m8), dd*xs, acc);  acc = fma(-dd, xct, acc)
// with m8 = -8*xsum for per-token-kernel tokens (t >= 4*floor(S/4); else 0)
// and xct the tile kernel's offset term (8*xsum)*xs (0 for per-token tokens)
// reproduces both reference forms (the second FMA adds -dd*0 to a nonzero-
// signed or +0 accumulator: exactly nothing).  Q8R4 runs the first FMA only.
//
// The weight rows are the MFMA's rows and the tokens its columns: a lane then
// holds one token (of each token tile), whose xs and xct it reads once per
// group, and reads the scales dd of its 16 rows as four float4s, shared by
// all its token tiles.  With the operands the other way round
// (k_r4_gemm_tok) the per-token xs, xct and m8 are 8-12 ds_read_b128 per group
// and 32 x 32 outputs, three times the LDS instructions per output.  What bounds
// this one on full grids is the vector work of the chains, 64 operations
// (convert, dd*xs, two FMAs) per 16 registers and MFMA: 24576 x 4096, 256
// tokens, counters: vector pipes busy 73 % of the kernel's time, MFMA 7 %, LDS
// bank conflicts 5 %.
//
// Tiles of MT x MT outputs (32: v_mfma_i32_32x32x32_i8; 16: 16x16x32, for
// grids that leave SIMDs idle), RT row tiles x TT token tiles per wave, WR x
// WT waves.  PAIR: W is a row-fused [gate; up] matrix of 2*O rows, RT = 2,
// tile 0 gate rows and tile 1 the same up rows, y [S][O] = silu(gate) * up
// (the gate_up + silu_rows of nn/ffn.c:28-37).  Steps of 4 groups are
// double-buffered in LDS, one barrier each, with the next two on their way to
// registers (with one, the load latency of a step was its time on small grids).
constexpr int R4M_KG = 4;                 // groups per K step
constexpr int R4M_AS = R4M_KG * 32 + 16;  // LDS row stride of the token codes (bytes)

typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

template <bool Q8, bool PAIR, int MT, int RT, int TT, int WR, int WT>
__global__ __launch_bounds__(64 * WR * WT, 2) void k_r4_gemm(const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                          const int32_t* __restrict__ xm,
                                                          const uint8_t* __restrict__ W,
                                                          const uint16_t* __restrict__ d16, float* __restrict__ y,
                                                          int S, int I, int O) {
  static_assert(!PAIR || RT == 2, "PAIR: a gate and an up tile");
  constexpr int NT = 64 * WR * WT;
  constexpr int GB = Q8 ? 128 : 64, RB = Q8 ? 32 : 16;  // bytes of a block and group, of a row and group
  constexpr int BT = MT * TT * WT, BR = MT * RT * WR;   // tokens, weight rows of the tile
  constexpr int OC = PAIR ? BR / 2 : BR;                // output columns
  constexpr int BS = R4M_KG * RB + 16;                  // LDS row stride of the weight codes (bytes)
  constexpr int ND = MT == 32 ? 16 : 4;                 // registers of a tile
  constexpr int AC = BT * R4M_KG * 2, BC = BR * R4M_KG * (RB / 16), DC = BR / 4 * R4M_KG, TC = BT * R4M_KG;
  constexpr int NA = (AC + NT - 1) / NT, NB = (BC + NT - 1) / NT, NDC = (DC + NT - 1) / NT, NTC = (TC + NT - 1) / NT;
  __shared__ __align__(16) int8_t sA[2][BT * R4M_AS];
  __shared__ __align__(16) uint8_t sB[2][BR * BS];
  __shared__ __align__(16) float sD[2][R4M_KG * BR];  // [group][row]
  __shared__ __align__(16) float sX[2][R4M_KG * BT], sC[2][Q8 ? 4 : R4M_KG * BT];  // [group][token]
  __shared__ int sM[2][Q8 ? 4 : R4M_KG * BT];
  __shared__ uint64_t s_exp[PAIR ? 32 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wr = wv % WR, wt = wv / WR;
  const int rl = lane % MT, hk = lane / MT;  // this lane's row / token of a tile, its K part
  const int mb = blockIdx.y * BT, ob = blockIdx.x * OC;
  const int nb = I / 32, S4 = S / 4 * 4, nstep = (nb + R4M_KG - 1) / R4M_KG;
  const int O4 = ((PAIR ? 2 * O : O) + 3) / 4;
  const bool tile = Q8 || mb + BT <= S4 || S == S4;  // no per-token tokens here: m8 is 0 throughout
  if (PAIR) exp_tab_lds(s_exp);

  // staging.  Rows past the end re-read the last block or token; groups past
  // the end hold the row's first group and are never chained (compute takes a
  // short step's groups one by one).
  auto blk = [&](int r4) {  // global 4-row block of tile row 4 * r4
    const int row = 4 * r4, o = PAIR && row >= OC ? O + ob + row - OC : ob + row;
    return o / 4 < O4 ? o / 4 : O4 - 1;
  };
  // Every load is unconditional, from clamped piece numbers and addresses
  // (the last piece is then stored more than once, the same bytes): with no
  // branch around a load the compiler waits for the set it needs alone.
  struct Set {
    v4i a[NA], b[NB];
    u32x2_a2 d[NDC];
    float x[NTC];
    int m[NTC];
  };
  Set s0, s1;
  auto piece = [&](int i, int n) { return n % NT == 0 || tid + i * NT < n ? tid + i * NT : n - 1; };
  // The pieces' addresses are set up once and move by the same bytes every
  // step; only a last step that is not full looks at each piece's group.
  const int8_t* pa[NA];
  const uint8_t* pb[NB];
  const uint16_t* pd[NDC];
  uint32_t px[NTC];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int c = piece(i, AC), t = c / (2 * R4M_KG), m = mb + t < S ? mb + t : S - 1;
    pa[i] = xq + (int64_t)m * I + c % (2 * R4M_KG) * 16;
  }
  constexpr int PB = R4M_KG * GB / 16;  // a block's 16-byte pieces of a step: consecutive threads take consecutive ones
#pragma unroll
  for (int i = 0; i < NB; i++) {
    const int c = piece(i, BC);
    pb[i] = W + (size_t)blk(c / PB) * nb * GB + c % PB * 16;
  }
#pragma unroll
  for (int i = 0; i < NDC; i++) {
    const int c = piece(i, DC);
    pd[i] = d16 + ((size_t)blk(c / R4M_KG) * nb + c % R4M_KG) * 4;
  }
#pragma unroll
  for (int i = 0; i < NTC; i++) {
    const int c = piece(i, TC), t = c / R4M_KG, m = mb + t < S ? mb + t : S - 1;
    px[i] = (uint32_t)m * nb + c % R4M_KG;
  }
  auto gload = [&](int st, Set& v) {
    const int s = st < nstep ? st : nstep - 1, left = nb - s * R4M_KG;  // uniform
    // a piece of a group past the row's end takes the row's first piece
#pragma unroll
    for (int i = 0; i < NA; i++) {
      const int k = piece(i, AC) % (2 * R4M_KG);
      v.a[i] = *(const v4i*)(pa[i] + (k / 2 < left ? s * (R4M_KG * 32) : -k * 16));
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int q = piece(i, BC) % PB;
      v.b[i] = *(const v4i*)(pb[i] + (q / (GB / 16) < left ? s * (R4M_KG * GB) : -q * 16));
    }
#pragma unroll
    for (int i = 0; i < NDC; i++) {
      const int k = piece(i, DC) % R4M_KG;
      v.d[i] = *(const u32x2_a2*)(pd[i] + (k < left ? s * (R4M_KG * 4) : -k * 4));
    }
#pragma unroll
    for (int i = 0; i < NTC; i++) {
      const int k = piece(i, TC) % R4M_KG;
      const uint32_t at = px[i] + (k < left ? s * R4M_KG : -k);
      v.x[i] = xs[at];
      if (!Q8) v.m[i] = xm[at];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto put = [&](int p, const Set& v) {
#pragma unroll
    for (int i = 0; i < NA; i++) {
      const int c = piece(i, AC), t = c / (2 * R4M_KG), k = c % (2 * R4M_KG);
      *(v4i*)(sA[p] + t * R4M_AS + k * 16) = v.a[i];
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
      constexpr int PR = RB / 16;
      const int c = piece(i, BC), r4 = c / PB, q = c % PB, k = q / (GB / 16), h = q % (GB / 16);
      *(v4i*)(sB[p] + (r4 * 4 + h / PR) * BS + k * RB + h % PR * 16) = v.b[i];
    }
#pragma unroll
    for (int i = 0; i < NDC; i++) {
      const int c = piece(i, DC), r4 = c / R4M_KG, k = c % R4M_KG;
      const auto h = [](uint32_t u) { return (float)__builtin_bit_cast(_Float16, (uint16_t)u); };  // exact
      *(float4*)(sD[p] + k * BR + r4 * 4) = float4{h(v.d[i].x & 0xffffu), h(v.d[i].x >> 16),
                                                   h(v.d[i].y & 0xffffu), h(v.d[i].y >> 16)};
    }
#pragma unroll
    for (int i = 0; i < NTC; i++) {
      const int c = piece(i, TC), t = c / R4M_KG, k = c % R4M_KG;
      sX[p][k * BT + t] = v.x[i];
      if (!Q8) {
        const bool per_token = mb + t >= S4;
        sC[p][k * BT + t] = per_token ? 0.f : (8.f * (float)v.m[i]) * v.x[i];
        sM[p][k * BT + t] = per_token ? -8 * v.m[i] : 0;
      }
    }
  };

  float acc[RT][TT][ND];
#pragma unroll
  for (int j = 0; j < RT; j++)
#pragma unroll
    for (int i = 0; i < TT; i++)
#pragma unroll
      for (int r = 0; r < ND; r++) acc[j][i][r] = 0.f;
  auto row0 = [&](int j) { return PAIR ? j * OC + wr * MT : (wr * RT + j) * MT; };  // first tile row of row tile j

  // NG groups from gg on: every fragment and MFMA first, then the chains in
  // group order, so the reads and MFMAs of one group hide behind another's
  typedef typename std::conditional<MT == 32, v16i, v4i>::type vd;
  auto groups = [&](int p, int gg, auto ngs, auto tl) {
    constexpr int NG = decltype(ngs)::value;
    constexpr bool TILE = decltype(tl)::value;
    vd d[NG][RT][TT];
    float xv[NG][TT], cv[NG][TT];
    int mv[NG][TT];
#pragma unroll
    for (int g = 0; g < NG; g++) {
      if constexpr (MT == 32) {
        v4i fb[TT];
#pragma unroll
        for (int i = 0; i < TT; i++)
          fb[i] = *(const v4i*)(sA[p] + ((wt * TT + i) * 32 + rl) * R4M_AS + (gg + g) * 32 + hk * 16);
#pragma unroll
        for (int j = 0; j < RT; j++) {
          v4i fa;
          if (Q8) {
            fa = *(const v4i*)(sB[p] + (row0(j) + rl) * BS + (gg + g) * RB + hk * 16);
          } else {  // low nibbles for hk = 0 (codes 0..15), high for hk = 1
            const v4i w = *(const v4i*)(sB[p] + (row0(j) + rl) * BS + (gg + g) * RB);
#pragma unroll
            for (int q = 0; q < 4; q++) fa[q] = (w[q] >> (4 * hk)) & 0x0f0f0f0f;
          }
#pragma unroll
          for (int i = 0; i < TT; i++) d[g][j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb[i], vd{}, 0, 0, 0);
        }
      } else {
        long fb[TT];
#pragma unroll
        for (int i = 0; i < TT; i++)
          fb[i] = *(const long*)(sA[p] + ((wt * TT + i) * 16 + rl) * R4M_AS + (gg + g) * 32 + hk * 8);
#pragma unroll
        for (int j = 0; j < RT; j++) {
          long fa;
          if (Q8) {
            fa = *(const long*)(sB[p] + (row0(j) + rl) * BS + (gg + g) * RB + hk * 8);
          } else {  // K part hk: codes 8 hk .. + 8, nibbles hk / 2 of bytes 8 (hk % 2) ..
            const uint2 w = *(const uint2*)(sB[p] + (row0(j) + rl) * BS + (gg + g) * RB + (hk & 1) * 8);
            const int sh = (hk >> 1) * 4;
            fa = (long)(((w.x >> sh) & 0x0f0f0f0fu) | ((uint64_t)((w.y >> sh) & 0x0f0f0f0fu) << 32));
          }
#pragma unroll
          for (int i = 0; i < TT; i++) d[g][j][i] = __builtin_amdgcn_mfma_i32_16x16x32_i8(fa, fb[i], vd{}, 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < TT; i++) {
        const int t = (gg + g) * BT + (wt * TT + i) * MT + rl;
        xv[g][i] = sX[p][t];
        cv[g][i] = Q8 ? 0.f : sC[p][t];
        mv[g][i] = TILE ? 0 : sM[p][t];
      }
    }
    // register r of a tile: row 8 (r / 4) + 4 hk + r % 4 (MT 32), 4 hk + r (MT 16)
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
      for (int j = 0; j < RT; j++)
#pragma unroll
        for (int q = 0; q < ND / 4; q++) {
          const float4 dv = *(const float4*)(sD[p] + (gg + g) * BR + row0(j) + 8 * q + 4 * hk);
          const float dd[4] = {dv.x, dv.y, dv.z, dv.w};
#pragma unroll
          for (int i = 0; i < TT; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
              float& a = acc[j][i][4 * q + r];
              a = __fmaf_rn((float)(d[g][j][i][4 * q + r] + mv[g][i]), dd[r] * xv[g][i], a);
              if (!Q8) a = __fmaf_rn(-dd[r], cv[g][i], a);
            }
        }
  };
  // as many groups at once as 64 registers of sums allow
  constexpr int NGB = RT * TT * ND * 4 <= 64 ? 4 : (RT * TT * ND * 2 <= 64 ? 2 : 1);
  auto compute = [&](int p, int n, auto tl) {
    if (n == R4M_KG) {  // uniform; straight-line: a branch per group would wait for each on its own
#pragma unroll
      for (int gg = 0; gg < R4M_KG; gg += NGB) groups(p, gg, std::integral_constant<int, NGB>{}, tl);
    } else {
#pragma unroll 1
      for (int gg = 0; gg < n; gg++) groups(p, gg, std::integral_constant<int, 1>{}, tl);
    }
  };

  auto step = [&](int st, Set& v) {  // v: step st + 1's pieces; step st + 3's next
    __syncthreads();  // step st is staged; every wave is done with step st - 1
    const int p = st & 1;
    put(p ^ 1, v);
    gload(st + 3, v);
    const int n = nb - st * R4M_KG < R4M_KG ? nb - st * R4M_KG : R4M_KG;
    if (tile) compute(p, n, std::true_type{});  // workgroup-uniform
    else compute(p, n, std::false_type{});
  };
  gload(0, s0);
  gload(1, s1);
  put(0, s0);
  gload(2, s0);
  for (int st = 0; st < nstep; st += 2) {
    step(st, s1);
    if (st + 1 < nstep) step(st + 1, s0);
  }
  // retire the clamped prefetches once before the conditional stores
  __builtin_amdgcn_s_waitcnt(0);
  // a lane's registers 4q..4q+3 are four consecutive columns of its token
  const bool vec = (O & 3) == 0 && (((uintptr_t)y) & 15) == 0;
#pragma unroll
  for (int i = 0; i < TT; i++) {
    const int t = mb + (wt * TT + i) * MT + rl;
#pragma unroll
    for (int j = 0; j < (PAIR ? 1 : RT); j++)
#pragma unroll
      for (int q = 0; q < ND / 4; q++) {
        const int o = ob + row0(j) + 8 * q + 4 * hk;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          v[r] = acc[j][i][4 * q + r];
          if constexpr (PAIR) v[r] = ref_silu_mul(v[r], acc[1][i][4 * q + r], s_exp);
        }
        if (t >= S || o >= O) continue;
        float* yp = y + (int64_t)t * O + o;
        if (vec) {
          *(float4*)yp = float4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (o + r < O) yp[r] = v[r];
        }
      }
  }
}

// ---------------------------------------------------------------------------
// The same for a few tokens: tiles of 16 TT tokens x 16 RT weight rows (PAIR:
// RT = 2, gate and up rows of the same 16 columns) whose K steps of KG groups
// are split over 8 waves by group.  Each wave forms its groups' integer dots
// by one v_mfma_i32_16x16x32_i8 per tile and hands (float)(s + m8) over
// through LDS, where a wave per register and tile continues the two-FMA
// chains one step behind.  A step's barrier, LDS and load latencies (0.5-0.7
// us, whatever it holds) bound k_r4_gemm's 4-group steps on grids this small.
template <bool Q8, bool PAIR, int TT, int KG>
__global__ __launch_bounds__(512, 2) void k_r4_few(const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                   const int32_t* __restrict__ xm, const uint8_t* __restrict__ W,
                                                   const uint16_t* __restrict__ d16, float* __restrict__ y, int S,
                                                   int I, int O) {
  constexpr int NT = 512, KS = 8, RT = PAIR ? 2 : 1;
  constexpr int GB = Q8 ? 128 : 64, RB = Q8 ? 32 : 16;  // bytes of a block and group, of a row and group
  constexpr int BT = 16 * TT, BR = 16 * RT;             // tokens, weight rows of the tile
  constexpr int AS = KG * 32 + 16, BS = KG * RB + 16;   // LDS row strides of the codes (bytes)
  constexpr int FS = KG + 4;                            // and of the per-group floats: 16 rows' float4s on 64 banks
  constexpr int PB = KG * GB / 16;                      // a block's 16-byte pieces of a step
  constexpr int AC = BT * KG * 2, BC = BR / 4 * PB, DC = BR / 4 * KG, TC = BT * KG;
  constexpr int NA = (AC + NT - 1) / NT, NB = (BC + NT - 1) / NT, NTC = (TC + NT - 1) / NT;
  constexpr int NTL = RT * TT;                // tiles
  constexpr int NC = (NTL * 4 + KS - 1) / KS;  // (tile, register) chains per wave
  static_assert(KG % KS == 0 && DC <= NT, "groups of a step over the K waves, one scale piece a thread");
  __shared__ __align__(16) int8_t sA[2][BT * AS];
  __shared__ __align__(16) uint8_t sB[2][BR * BS];
  __shared__ __align__(16) float sD[2][BR * FS], sX[2][BT * FS], sC[2][Q8 ? 4 : BT * FS];  // [row or token][group]
  __shared__ int sM[2][Q8 ? 4 : BT * FS];
  __shared__ float rs[2][KG * NTL * 256];
  __shared__ uint64_t s_exp[PAIR ? 32 : 1];
  const int tid = threadIdx.x, lane = tid & 63, ks = tid >> 6;
  const int rl = lane & 15, hk = lane >> 4;  // this lane's row / token of a tile, its K part
  const int mb = blockIdx.y * BT, ob = blockIdx.x * 16;
  const int nb = I / 32, S4 = S / 4 * 4, nstep = (nb + KG - 1) / KG;
  const int O4 = ((PAIR ? 2 * O : O) + 3) / 4;
  if (PAIR) exp_tab_lds(s_exp);

  // staging, two steps ahead, every load unconditional as in k_r4_gemm: rows
  // past the end re-read the last block or token, groups past the end group 0
  auto blk = [&](int r4) {
    const int row = 4 * r4, o = row >= 16 ? O + ob + row - 16 : ob + row;
    return o / 4 < O4 ? o / 4 : O4 - 1;
  };
  struct Set {
    v4i a[NA], b[NB];
    u32x2_a2 d;
    float x[NTC];
    int m[NTC];
  };
  Set s0, s1;
  auto piece = [&](int i, int n) { return n % NT == 0 || tid + i * NT < n ? tid + i * NT : n - 1; };
  const int8_t* pa[NA];
  const uint8_t* pb[NB];
  uint32_t px[NTC];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int c = piece(i, AC), t = c / (2 * KG), m = mb + t < S ? mb + t : S - 1;
    pa[i] = xq + (int64_t)m * I + c % (2 * KG) * 16;
  }
#pragma unroll
  for (int i = 0; i < NB; i++) {
    const int c = piece(i, BC);
    pb[i] = W + (size_t)blk(c / PB) * nb * GB + c % PB * 16;
  }
  const uint16_t* pd = d16 + ((size_t)blk(piece(0, DC) / KG) * nb + piece(0, DC) % KG) * 4;
#pragma unroll
  for (int i = 0; i < NTC; i++) {
    const int c = piece(i, TC), t = c / KG, m = mb + t < S ? mb + t : S - 1;
    px[i] = (uint32_t)m * nb + c % KG;
  }
  auto gload = [&](int st, Set& v) {
    const int s = st < nstep ? st : nstep - 1, left = nb - s * KG;  // uniform
#pragma unroll
    for (int i = 0; i < NA; i++) {
      const int k = piece(i, AC) % (2 * KG);
      v.a[i] = *(const v4i*)(pa[i] + (k / 2 < left ? s * (KG * 32) : -k * 16));
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int q = piece(i, BC) % PB;
      v.b[i] = *(const v4i*)(pb[i] + (q / (GB / 16) < left ? s * (KG * GB) : -q * 16));
    }
    {
      const int k = piece(0, DC) % KG;
      v.d = *(const u32x2_a2*)(pd + (k < left ? s * (KG * 4) : -k * 4));
    }
#pragma unroll
    for (int i = 0; i < NTC; i++) {
      const int k = piece(i, TC) % KG;
      const uint32_t at = px[i] + (k < left ? s * KG : -k);
      v.x[i] = xs[at];
      if (!Q8) v.m[i] = xm[at];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto put = [&](int p, const Set& v) {
#pragma unroll
    for (int i = 0; i < NA; i++) {
      const int c = piece(i, AC);
      *(v4i*)(sA[p] + c / (2 * KG) * AS + c % (2 * KG) * 16) = v.a[i];
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
      constexpr int PR = RB / 16;
      const int c = piece(i, BC), r4 = c / PB, q = c % PB, k = q / (GB / 16), h = q % (GB / 16);
      *(v4i*)(sB[p] + (r4 * 4 + h / PR) * BS + k * RB + h % PR * 16) = v.b[i];
    }
    {
      const int c = piece(0, DC), r4 = c / KG, k = c % KG;
      const auto h = [](uint32_t u) { return (float)__builtin_bit_cast(_Float16, (uint16_t)u); };  // exact
      float* o = sD[p] + r4 * 4 * FS + k;
      o[0] = h(v.d.x & 0xffffu), o[FS] = h(v.d.x >> 16), o[2 * FS] = h(v.d.y & 0xffffu), o[3 * FS] = h(v.d.y >> 16);
    }
#pragma unroll
    for (int i = 0; i < NTC; i++) {
      const int c = piece(i, TC), t = c / KG, at = t * FS + c % KG;
      sX[p][at] = v.x[i];
      if (!Q8) {
        const bool per_token = mb + t >= S4;
        sC[p][at] = per_token ? 0.f : (8.f * (float)v.m[i]) * v.x[i];
        sM[p][at] = per_token ? -8 * v.m[i] : 0;
      }
    }
  };

  // chain c of this wave: id = ks + 8 c, register id % 4 (row 4 hk + id % 4)
  // of tile id / 4 (row tile id / 4 / TT, token tile id / 4 % TT)
  float acc[NC], sc[NC][KG], nd[NC][KG], cv[NC][KG];
#pragma unroll
  for (int c = 0; c < NC; c++) acc[c] = 0.f;
  auto chain = [&](int st) {
    const int n = nb - st * KG < KG ? nb - st * KG : KG;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int id = ks + KS * c;
      if (id >= NTL * 4) break;  // wave-uniform
      const float* rp = rs[st & 1] + id * 64 + lane;
      auto link = [&](int k) {
        acc[c] = __fmaf_rn(rp[k * NTL * 256], sc[c][k], acc[c]);
        if (!Q8) acc[c] = __fmaf_rn(nd[c][k], cv[c][k], acc[c]);
      };
      if (n == KG) {
#pragma unroll
        for (int k = 0; k < KG; k++) link(k);
      } else {
#pragma unroll
        for (int k = 0; k < KG; k++)
          if (k < n) link(k);
      }
    }
  };
  auto step = [&](int st, Set& v) {  // v: step st + 1's pieces; step st + 3's next
    // step st is staged, the dots of step st - 1 are handed over, and every
    // wave is done with the buffers of step st - 1
    __syncthreads();
    const int p = st & 1;
    if (st > 0) chain(st - 1);
    put(p ^ 1, v);
    gload(st + 3, v);
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int id = ks + KS * c, tl = id / 4 % NTL;
      const float* dp = sD[p] + (tl / TT * 16 + 4 * hk + id % 4) * FS;
      const int t = (tl % TT * 16 + rl) * FS;
#pragma unroll
      for (int k = 0; k < KG; k += 4) {
        const float4 dv = *(const float4*)(dp + k), xv = *(const float4*)(sX[p] + t + k);
        sc[c][k] = dv.x * xv.x, sc[c][k + 1] = dv.y * xv.y, sc[c][k + 2] = dv.z * xv.z, sc[c][k + 3] = dv.w * xv.w;
        if (!Q8) {
          const float4 cc = *(const float4*)(sC[p] + t + k);
          nd[c][k] = -dv.x, nd[c][k + 1] = -dv.y, nd[c][k + 2] = -dv.z, nd[c][k + 3] = -dv.w;
          cv[c][k] = cc.x, cv[c][k + 1] = cc.y, cv[c][k + 2] = cc.z, cv[c][k + 3] = cc.w;
        }
      }
    }
    // groups past the end are computed on the rows' first and never chained
    v4i d[KG / KS][RT][TT];
    int mv[KG / KS][TT];
#pragma unroll
    for (int g = 0; g < KG / KS; g++) {
      const int k = g * KS + ks;
      long fb[TT];
#pragma unroll
      for (int i = 0; i < TT; i++) {
        fb[i] = *(const long*)(sA[p] + (i * 16 + rl) * AS + k * 32 + hk * 8);
        mv[g][i] = Q8 ? 0 : sM[p][(i * 16 + rl) * FS + k];
      }
#pragma unroll
      for (int j = 0; j < RT; j++) {
        long fa;
        const uint8_t* wp = sB[p] + (j * 16 + rl) * BS + k * RB;
        if (Q8) {
          fa = *(const long*)(wp + hk * 8);
        } else {  // K part hk: codes 8 hk .. + 8, nibbles hk / 2 of bytes 8 (hk % 2) ..
          const uint2 w = *(const uint2*)(wp + (hk & 1) * 8);
          const int sh = (hk >> 1) * 4;
          fa = (long)(((w.x >> sh) & 0x0f0f0f0fu) | ((uint64_t)((w.y >> sh) & 0x0f0f0f0fu) << 32));
        }
#pragma unroll
        for (int i = 0; i < TT; i++)
          d[g][j][i] = __builtin_amdgcn_mfma_i32_16x16x32_i8(fa, fb[i], v4i{0, 0, 0, 0}, 0, 0, 0);
      }
    }
#pragma unroll
    for (int g = 0; g < KG / KS; g++)
#pragma unroll
      for (int j = 0; j < RT; j++)
#pragma unroll
        for (int i = 0; i < TT; i++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            rs[p][((g * KS + ks) * NTL + j * TT + i) * 256 + r * 64 + lane] = (float)(d[g][j][i][r] + mv[g][i]);
  };
  gload(0, s0);
  gload(1, s1);
  put(0, s0);
  gload(2, s0);
  for (int st = 0; st < nstep; st += 2) {
    step(st, s1);
    if (st + 1 < nstep) step(st + 1, s0);
  }
  __syncthreads();
  chain(nstep - 1);
  __builtin_amdgcn_s_waitcnt(0);  // the clamped prefetches
  // the chains of a token's columns sit in different waves: through LDS, then
  // a wave per token tile and register writes its outputs
  float* ex = rs[nstep & 1];  // the half the last chain did not read
#pragma unroll
  for (int c = 0; c < NC; c++) {
    const int id = ks + KS * c;
    if (id < NTL * 4) ex[id * 64 + lane] = acc[c];
  }
  __syncthreads();
  // 64 outputs at a time, 16 consecutive columns of 4 tokens
  for (int q = ks; q < TT * 4; q += KS) {
    const int t = q * 4 + hk, i = t / 16, o = rl;  // token and column of the tile
    const int at = (i * 4 + o % 4) * 64 + o / 4 * 16 + t % 16;
    float v = ex[at];
    if constexpr (PAIR) v = ref_silu_mul(v, ex[TT * 256 + at], s_exp);
    if (mb + t < S && ob + o < O) y[(int64_t)(mb + t) * O + ob + o] = v;
  }
}

// Q4R4 with the operands the other way round: the tokens are the MFMA's rows
// and the weights its columns, a lane holding one weight row's dd and reading
// the xs, xct and m8 of its 16 (4) tokens per group.  Block tile 64 tokens x 64
// weight rows, K steps of 4 groups single-buffered in LDS with two more in
// registers.  Slower per output than k_r4_gemm on full grids, but its small LDS
// and register shares hold more waves on a CU, so it is the faster one where
// k_r4_gemm's tiles leave CUs idle or a last round nearly empty (4096 x 12288,
// 256 tokens: 94.8 us against 99.9 in any of k_r4_gemm's tiles; 10240 x 1024,
// 400 tokens: 34.2 and 39.0).
// WV = 4: waves of 32 x 32.  WV = 16, for at most one workgroup per CU: waves
// of 16 x 16, the first four stage (4096 x 12288, 256 tokens: 92.7 us against
// 132 with four).  PAIR (WV = 4): 32 gate rows and the same up rows, y [S][O] =
// silu(gate) * up, the up waves handing their sums over through LDS.
constexpr int R4T_NT = 256;  // staging threads

template <int WV, bool PAIR>
__global__ __launch_bounds__(64 * WV, WV <= 8 ? 8 / WV : 1) void k_r4_gemm_tok(const int8_t* __restrict__ xq,
                                                                               const float* __restrict__ xs,
                                                                               const int32_t* __restrict__ xm,
                                                                               const uint8_t* __restrict__ W,
                                                                               const uint16_t* __restrict__ d16,
                                                                               float* __restrict__ y, int S, int I,
                                                                               int O) {
  static_assert(WV == 16 ? !PAIR : WV == 4, "waves");
  constexpr int GB = 64, RB = 16;       // bytes of a block and group, of a row and group
  constexpr int BS = R4M_KG * RB + 16;  // LDS row stride of the weight codes
  __shared__ __align__(16) int8_t sA[64 * R4M_AS];
  __shared__ __align__(16) uint8_t sB[64 * BS];
  __shared__ float sD[64 * R4M_KG];                                 // [row][group]
  __shared__ __align__(16) float sX[R4M_KG * 64], sC[R4M_KG * 64];  // [group][token]
  __shared__ __align__(16) int sM[R4M_KG * 64];
  const int tid = threadIdx.x, lane = tid % MOTY_WAVE, wv = tid / MOTY_WAVE;
  const int mb = blockIdx.y * 64, nb0 = blockIdx.x * (PAIR ? 32 : 64);
  const int nb = I / 32, S4 = S / 4 * 4;
  const bool tile = mb + 64 <= S4 || S == S4;  // no per-token tokens here: m8 is 0 throughout
  const int O4 = ((PAIR ? 2 * O : O) + 3) / 4;

  // staging: thread -> two 16-byte chunks of the tokens' codes, 16 bytes and
  // one scale of weight row tid / 4, group tid % 4, the scales of token
  // tid % 64, group tid / 64.  Rows past the end re-read the last; groups past
  // the end re-read others and are never chained.
  const int8_t* srcA[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int q = tid + i * R4T_NT, m = mb + (q >> 3) < S ? mb + (q >> 3) : S - 1;
    srcA[i] = xq + (int64_t)m * I + (q & 7) * 16;
  }
  const int trow = tid >> 2;
  const int orow = !PAIR ? nb0 + trow : trow < 32 ? nb0 + trow : O + nb0 + trow - 32;
  const int ob = orow / 4 < O4 ? orow / 4 : O4 - 1;
  const uint8_t* srcB = W + (size_t)ob * nb * GB + (size_t)(orow & 3) * RB;
  const uint16_t* srcD = d16 + (size_t)ob * nb * 4 + (orow & 3);
  const int st_g = (tid >> 6) & 3, st_t = mb + (tid & 63) < S ? mb + (tid & 63) : S - 1;
  struct Set {
    v4i a[2], b;
    uint32_t d;
    float x;
    int m;
  };
  Set s0, s1;
  const bool stager = WV == 4 || tid < R4T_NT;  // wave-uniform
  const int glast = (nb - 1) / R4M_KG * R4M_KG;
  auto gload = [&](int g0, Set& v) {
    if (!stager) return;
    const int gc = g0 < nb ? g0 : glast;
    const int kb = gc * 32;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int k = ((tid + i * R4T_NT) & 7) * 16;
      v.a[i] = *(const v4i*)(srcA[i] + (kb + k < I ? kb : -k));
    }
    const int g = gc + (tid & 3) < nb ? gc + (tid & 3) : 0;
    v.b = *(const v4i*)(srcB + (size_t)g * GB);
    v.d = srcD[(size_t)g * 4];
    const int gt = gc + st_g < nb ? gc + st_g : 0;
    v.x = xs[(size_t)st_t * nb + gt];
    v.m = xm[(size_t)st_t * nb + gt];
    __builtin_amdgcn_sched_barrier(0);
  };
  float acc[WV == 16 ? 4 : 16];
#pragma unroll
  for (float& v : acc) v = 0.f;
  auto compute = [&](int ngk, auto tl) {
    constexpr bool TILE = decltype(tl)::value;
#pragma unroll
    for (int gg = 0; gg < R4M_KG; gg++) {
      if (gg >= ngk) break;  // wave-uniform
      if constexpr (WV == 16) {
        // tokens wm * 16 + [0, 16) x rows wn * 16 + [0, 16)
        const int wm = wv / 4, row = wv % 4 * 16 + (lane & 15), q4 = lane >> 4;
        const long a = *(const long*)(sA + (wm * 16 + (lane & 15)) * R4M_AS + gg * 32 + q4 * 8);
        const int t = gg * 64 + wm * 16 + 4 * q4;  // this lane's 4 tokens
        const float4 xv = *(const float4*)(sX + t), cv = *(const float4*)(sC + t);
        const int4 mv = TILE ? int4{0, 0, 0, 0} : *(const int4*)(sM + t);
        // codes 8 q4 .. + 8: nibbles q4 / 2 of bytes 8 (q4 % 2) ..
        const uint2 w = *(const uint2*)(sB + row * BS + gg * RB + (q4 & 1) * 8);
        const int sh = (q4 >> 1) * 4;
        const long b = (long)(((w.x >> sh) & 0x0f0f0f0fu) | ((uint64_t)((w.y >> sh) & 0x0f0f0f0fu) << 32));
        const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, v4i{0, 0, 0, 0}, 0, 0, 0);
        const float dd = sD[row * R4M_KG + gg];
        acc[0] = __fmaf_rn(-dd, cv.x, __fmaf_rn((float)(d[0] + mv.x), dd * xv.x, acc[0]));
        acc[1] = __fmaf_rn(-dd, cv.y, __fmaf_rn((float)(d[1] + mv.y), dd * xv.y, acc[1]));
        acc[2] = __fmaf_rn(-dd, cv.z, __fmaf_rn((float)(d[2] + mv.z), dd * xv.z, acc[2]));
        acc[3] = __fmaf_rn(-dd, cv.w, __fmaf_rn((float)(d[3] + mv.w), dd * xv.w, acc[3]));
      } else {
        const int wm = wv >> 1, row = (wv & 1) * 32 + (lane & 31), hk = lane >> 5;
        const v4i a = *(const v4i*)(sA + (wm * 32 + (lane & 31)) * R4M_AS + gg * 32 + hk * 16);
        v4i w = *(const v4i*)(sB + row * BS + gg * RB);
#pragma unroll
        for (int q = 0; q < 4; q++) w[q] = (w[q] >> (4 * hk)) & 0x0f0f0f0f;  // low nibbles for hk = 0, high for 1
        const v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, w, v16i{}, 0, 0, 0);
        const float dd = sD[row * R4M_KG + gg];
        // register r: token 8 (r / 4) + 4 hk + r % 4
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int t = gg * 64 + wm * 32 + 8 * q + 4 * hk;
          const float4 xv = *(const float4*)(sX + t), cv = *(const float4*)(sC + t);
          const int4 mv = TILE ? int4{0, 0, 0, 0} : *(const int4*)(sM + t);
          acc[4 * q] = __fmaf_rn(-dd, cv.x, __fmaf_rn((float)(d[4 * q] + mv.x), dd * xv.x, acc[4 * q]));
          acc[4 * q + 1] = __fmaf_rn(-dd, cv.y, __fmaf_rn((float)(d[4 * q + 1] + mv.y), dd * xv.y, acc[4 * q + 1]));
          acc[4 * q + 2] = __fmaf_rn(-dd, cv.z, __fmaf_rn((float)(d[4 * q + 2] + mv.z), dd * xv.z, acc[4 * q + 2]));
          acc[4 * q + 3] = __fmaf_rn(-dd, cv.w, __fmaf_rn((float)(d[4 * q + 3] + mv.w), dd * xv.w, acc[4 * q + 3]));
        }
      }
    }
  };
  auto stage = [&](int g0, Set& v) {
    if (stager) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int q = tid + i * R4T_NT;
        *(v4i*)(sA + (q >> 3) * R4M_AS + (q & 7) * 16) = v.a[i];
      }
      *(v4i*)(sB + trow * BS + (tid & 3) * RB) = v.b;
      sD[trow * R4M_KG + (tid & 3)] = f16_to_f32(v.d);
      sX[st_g * 64 + (tid & 63)] = v.x;
      const bool per_token = mb + (tid & 63) >= S4;
      sC[st_g * 64 + (tid & 63)] = per_token ? 0.f : (8.f * (float)v.m) * v.x;
      sM[st_g * 64 + (tid & 63)] = per_token ? -8 * v.m : 0;
    }
    __syncthreads();
    gload(g0 + 2 * R4M_KG, v);
    const int ngk = nb - g0 < R4M_KG ? nb - g0 : R4M_KG;
    if (tile) compute(ngk, std::true_type{});  // workgroup-uniform
    else compute(ngk, std::false_type{});
    __syncthreads();
  };
  gload(0, s0);
  gload(R4M_KG, s1);
  for (int g0 = 0; g0 < nb; g0 += 2 * R4M_KG) {
    stage(g0, s0);
    stage(g0 + R4M_KG, s1);
  }
  // retire the clamped prefetches once before the conditional stores
  __builtin_amdgcn_s_waitcnt(0);
  if constexpr (WV == 16) {
    const int col = nb0 + wv % 4 * 16 + (lane & 15);
    if (col >= O) return;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int t = mb + wv / 4 * 16 + 4 * (lane >> 4) + r;
      if (t < S) y[(int64_t)t * O + col] = acc[r];
    }
  } else {
    const int wm = wv >> 1, wn = wv & 1, hk = lane >> 5;
    float* xch = (float*)sA;  // up sums, [r][wm][lane]
    if constexpr (PAIR) {
      if (wn == 1) {
#pragma unroll
        for (int r = 0; r < 16; r++) xch[r * 128 + wm * 64 + lane] = acc[r];
      }
      __syncthreads();
    }
    const int col = nb0 + (PAIR ? 0 : wn * 32) + (lane & 31);
    if ((PAIR && wn == 1) || col >= O) return;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int t = mb + wm * 32 + 8 * (r >> 2) + 4 * hk + (r & 3);
      float v = acc[r];
      if constexpr (PAIR) v = ref_silu_mul(v, xch[r * 128 + wm * 64 + lane]);
      if (t < S) y[(int64_t)t * O + col] = v;
    }
  }
}

// The kernels' tile shapes and times: a launch of j tiles on the busiest CU
// (ceil(tiles / 256)) and n steps of 4 groups takes a + b * j + n * g[j] us,
// past eight tiles n * g[8] * j / 8.  The tiles on a CU share its SIMDs, so g
// is no multiple of j: two small tiles cost hardly more than one, and odd
// numbers of 64 x 64 tiles waste a slot.  Fitted on MI355X to 240 to 304
// points each: S = 4..4096 over the FFNs' gate + up (1024 x 3072 to 4096 x
// 14336) and down, 1024 x 10240 and 4096 x 4096, weights rotating past the
// Infinity Cache; off by 2 to 4 % (root mean square).  Where each wins: the
// few-token kernel to about 64 tokens, 16 x 32 tiles (MFMA 16 x 16) to a few
// hundred on narrow matrices, large tiles where several rounds of them fill
// the chip, and for Q4R4 k_r4_gemm_tok between.
enum R4Kern { R4_FEW16, R4_FEW32, R4_16x32, R4_32x64, R4_64x64, R4_64x128, R4_TOK, R4_NONE };
struct R4Tile {
  R4Kern kern;
  int bt, oc;  // tokens, output columns
  double a, b, g[8];
};
static constexpr R4Tile R4_ONE_Q4[] = {
    {R4_FEW16, 16, 16, 3.18, 1.17, {0.196, 0.404, 0.609, 0.815, 0.994, 1.137, 1.327, 1.516}},
    {R4_FEW32, 32, 16, 2.93, 1.52, {0.269, 0.549, 0.791, 1.035, 1.288, 1.542, 1.799, 2.056}},
    {R4_16x32, 16, 32, 4.65, 0.04, {0.570, 0.643, 0.685, 0.767, 0.920, 0.984, 1.148, 1.312}},
    {R4_32x64, 32, 64, 3.42, 0.95, {0.802, 0.990, 1.360, 1.903, 2.191, 2.457, 2.866, 3.276}},
    {R4_TOK, 64, 64, 2.50, 1.15, {0.938, 1.502, 2.022, 2.475, 3.176, 3.287, 3.835, 4.383}},
    {R4_64x128, 64, 128, 2.22, 3.64, {1.355, 2.758, 4.078, 5.439, 6.767, 8.121, 9.475, 10.828}},
};
static constexpr R4Tile R4_PAIR_Q4[] = {
    {R4_FEW16, 16, 16, 2.70, 2.01, {0.250, 0.489, 0.737, 0.990, 1.169, 1.472, 1.653, 1.813}},
    {R4_16x32, 16, 32, 5.03, 0.43, {0.766, 0.960, 1.015, 1.117, 1.405, 1.534, 1.793, 2.053}},
    {R4_32x64, 32, 64, 4.70, 1.69, {1.196, 1.488, 2.577, 2.984, 3.828, 4.423, 5.301, 5.815}},
    {R4_TOK, 64, 32, 6.36, 0.88, {1.169, 1.499, 1.966, 2.536, 3.352, 3.909, 4.705, 5.084}},
    {R4_64x64, 64, 64, 3.71, 2.16, {1.868, 2.270, 3.933, 4.603, 5.963, 6.761, 7.864, 8.966}},
};
static constexpr R4Tile R4_ONE_Q8[] = {
    {R4_FEW16, 16, 16, 3.69, 0.50, {0.167, 0.302, 0.450, 0.591, 0.720, 0.805, 0.939, 1.073}},
    {R4_FEW32, 32, 16, 2.81, 1.52, {0.235, 0.480, 0.697, 0.903, 1.111, 1.323, 1.543, 1.764}},
    {R4_16x32, 16, 32, 4.46, 0.00, {0.469, 0.529, 0.604, 0.697, 0.812, 0.930, 1.085, 1.240}},
    {R4_32x64, 32, 64, 4.02, 0.82, {0.672, 0.920, 1.231, 1.685, 2.011, 2.269, 2.647, 3.025}},
    {R4_64x64, 64, 64, 3.15, 1.97, {0.862, 1.112, 1.856, 2.160, 2.826, 3.081, 3.595, 4.108}},
    {R4_64x128, 64, 128, 1.15, 4.50, {1.083, 2.115, 3.048, 3.978, 4.968, 5.961, 6.955, 7.948}},
};
static constexpr R4Tile R4_PAIR_Q8[] = {
    {R4_FEW16, 16, 16, 4.00, 0.79, {0.250, 0.454, 0.732, 0.968, 1.139, 1.239, 1.446, 1.652}},
    {R4_16x32, 16, 32, 5.57, 0.03, {0.607, 0.809, 0.970, 1.146, 1.442, 1.595, 1.861, 2.127}},
    {R4_32x64, 32, 64, 3.80, 1.08, {1.110, 1.624, 2.480, 3.036, 3.823, 4.515, 5.267, 6.020}},
    {R4_64x64, 64, 64, 3.76, 2.13, {1.638, 2.033, 3.450, 4.130, 5.306, 5.920, 6.907, 7.893}},
};

// the fastest shape; its grid's extents in `grid`
template <int N>
static R4Kern r4_pick(const R4Tile (&t)[N], int S, int I, int O, dim3& grid) {
  R4Kern best = R4_NONE;
  double bt = 0;
  for (int k = 0; k < N; k++) {
    if (t[k].bt < 64 && S > t[k].bt * 65535) continue;  // a grid's rows
    const int64_t gx = (O + t[k].oc - 1) / t[k].oc, gy = (S + t[k].bt - 1) / t[k].bt, j = (gx * gy + 255) / 256;
    const double n = (I + 32 * R4M_KG - 1) / (32 * R4M_KG), g = j <= 8 ? t[k].g[j - 1] : t[k].g[7] * j / 8;
    double us = t[k].a + t[k].b * j + n * g;
    // its workgroups with per-token tokens read and add m8, and are waited for
    if (t[k].kern == R4_TOK && S % 4) us *= 1.08;
    if (best != R4_NONE && us >= bt) continue;
    best = t[k].kern;
    bt = us;
    grid = dim3((unsigned)gx, (unsigned)gy);
  }
  return best;
}

#define R4_LAUNCH(KERN, THREADS) \
  hipLaunchKernelGGL((KERN), grid, dim3(THREADS), 0, st, xq, xs, xm, W, d16, y, S, I, O)

// y [S][O] from quantized activations
template <bool Q8>
static int r4_one(const int8_t* xq, const float* xs, const int32_t* xm, const uint8_t* W, const uint16_t* d16, float* y,
                  int S, int I, int O, hipStream_t st) {
  dim3 grid;
  R4Kern k;
  if constexpr (Q8) k = r4_pick(R4_ONE_Q8, S, I, O, grid);
  else k = r4_pick(R4_ONE_Q4, S, I, O, grid);
  if (k == R4_FEW16) R4_LAUNCH((k_r4_few<Q8, false, 1, 16>), 512);
  else if (k == R4_FEW32) R4_LAUNCH((k_r4_few<Q8, false, 2, 16>), 512);
  else if (k == R4_16x32) R4_LAUNCH((k_r4_gemm<Q8, false, 16, 1, 1, 2, 1>), 128);
  else if (k == R4_32x64) R4_LAUNCH((k_r4_gemm<Q8, false, 16, 1, 2, 4, 1>), 256);
  else if (k == R4_64x128) R4_LAUNCH((k_r4_gemm<Q8, false, 32, 1, 1, 4, 2>), 512);
  else if constexpr (Q8) R4_LAUNCH((k_r4_gemm<true, false, 32, 1, 1, 2, 2>), 256);
  else if ((int64_t)grid.x * grid.y <= 256) R4_LAUNCH((k_r4_gemm_tok<16, false>), 1024);
  else R4_LAUNCH((k_r4_gemm_tok<4, false>), 256);
  LAUNCH_TRY("R4 matmul");
  return MOTY_OK;
}

// y [S][O] = silu(gate) * up, W the row-fused [gate; up] of 2 O rows
template <bool Q8>
static int r4_pair(const int8_t* xq, const float* xs, const int32_t* xm, const uint8_t* W, const uint16_t* d16,
                   float* y, int S, int I, int O, hipStream_t st) {
  dim3 grid;
  R4Kern k;
  if constexpr (Q8) k = r4_pick(R4_PAIR_Q8, S, I, O, grid);
  else k = r4_pick(R4_PAIR_Q4, S, I, O, grid);
  if (k == R4_FEW16) R4_LAUNCH((k_r4_few<Q8, true, 1, Q8 ? 8 : 16>), 512);
  else if (k == R4_16x32) R4_LAUNCH((k_r4_gemm<Q8, true, 16, 2, 1, 2, 1>), 128);
  else if (k == R4_32x64) R4_LAUNCH((k_r4_gemm<Q8, true, 16, 2, 2, 4, 1>), 256);
  else if (Q8 || k == R4_64x64) R4_LAUNCH((k_r4_gemm<Q8, true, 32, 2, 1, 2, 2>), 256);
  else R4_LAUNCH((k_r4_gemm_tok<4, true>), 256);
  LAUNCH_TRY("R4 gate + up");
  return MOTY_OK;
}
#undef R4_LAUNCH

// y [S][O] = R4 matmul of x [S][I]; xq/xs/xm: scratch for the activation
// codes (S*I bytes, S*(I/32) floats and ints)
int launch_r4_matmul(bool q8, const float* x, const uint8_t* W, const uint16_t* d16, float* y, int S, int I, int O,
                     int8_t* xq, float* xs, int32_t* xm, hipStream_t st) {
  if (I % 32 || I <= 0) return MOTY_EUNSUP;
  if (S <= 0 || O <= 0) return MOTY_OK;
  if (S <= 3) {
    const int rc = q8 ? launch_r4_gemv<true>(x, W, d16, y, S, I, O, st) : launch_r4_gemv<false>(x, W, d16, y, S, I, O, st);
    if (rc != MOTY_EUNSUP) return rc;
  }
  if (!xq || !xs || !xm) return MOTY_EINVAL;  // the GEMM path needs the activation scratch
  int rc = launch_quant_g32(x, xq, xs, xm, S, I, st);
  if (rc) return rc;
  return q8 ? r4_one<true>(xq, xs, xm, W, d16, y, S, I, O, st) : r4_one<false>(xq, xs, xm, W, d16, y, S, I, O, st);
}

// gate/up + SiLU over a row-fused [gate; up] R4 matrix (2*I rows) for S > 3
// tokens: h [S][I] = silu(x.gate^T) * (x.up^T) in one GEMM pass (PAIR tiles)
int launch_r4_gate_up_gemm(bool q8, const float* x, const uint8_t* W, const uint16_t* d16, float* h, int S, int D,
                           int I, int8_t* xq, float* xs, int32_t* xm, hipStream_t st) {
  if (D % 32 || D <= 0 || I % 4 || I <= 0) return MOTY_EUNSUP;
  if (S <= 0) return MOTY_OK;
  int rc = launch_quant_g32(x, xq, xs, xm, S, D, st);
  if (rc) return rc;
  return q8 ? r4_pair<true>(xq, xs, xm, W, d16, h, S, D, I, st) : r4_pair<false>(xq, xs, xm, W, d16, h, S, D, I, st);
}

// Decode gate/up + SiLU over a row-fused [gate; up] R4 matrix (2*I rows,
// the gate_up of nn/ffn.c:28-37): h [I] = silu(x.gate^T) * (x.up^T), one token.
int launch_r4_gate_up_silu(bool q8, const float* x, const uint8_t* W, const uint16_t* d16, float* h, int D, int I,
                           hipStream_t st) {
  if (D % 32 || D <= 0 || I % 4 || I <= 0) return MOTY_EUNSUP;
  return q8 ? go_r4_gemv_ic<true, 1, true>(x, W, d16, h, 1, D, I, st)
            : go_r4_gemv_ic<false, 1, true>(x, W, d16, h, 1, D, I, st);
}

// ---------------------------------------------------------------------------
// Packers (nn/quant.c:130-177): thread per (block, group, row).  The group
// scale is the "no-clip Q4_0" rule: mx = the largest-magnitude weight (the
// first one on ties), opp = the largest |w| of the other sign, d =
// -sign(mx) * max(|mx|/lo, opp/hi) rounded to f16 (nearest even), codes
// rint(w / d) via the reciprocal of the rounded scale, clipped.

// float -> IEEE half, round to nearest even (nn/quant.c:111-128)
__device__ __forceinline__ uint32_t f32_to_f16(float f) {
  const uint32_t x = __float_as_uint(f);
  const uint32_t sign = (x >> 16) & 0x8000u, e = (x >> 23) & 0xffu;
  uint32_t m = x & 0x7fffffu;
  if (e == 0xffu) return sign | 0x7c00u | (m ? 0x200u : 0u);
  const int ne = (int)e - 127 + 15;
  if (ne >= 31) return sign | 0x7c00u;
  if (ne <= 0) {
    if (ne < -10) return sign;
    m |= 0x800000u;
    const int sh = 14 - ne;
    uint32_t h = m >> sh;
    const uint32_t rem = m & ((1u << sh) - 1), half = 1u << (sh - 1);
    if (rem > half || (rem == half && (h & 1))) h++;
    return sign | h;
  }
  uint32_t h = ((uint32_t)ne << 10) | (m >> 13);
  const uint32_t rem = m & 0x1fffu;
  if (rem > 0x1000u || (rem == 0x1000u && (h & 1))) h++;
  return sign | h;
}

template <bool Q8>
__global__ __launch_bounds__(256) void k_pack_r4(const float* __restrict__ w, uint8_t* __restrict__ q,
                                                 uint16_t* __restrict__ d16, int O, int I) {
  const int nb = I / 32, O4 = (O + 3) / 4;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (block, group, row)
  if (id >= (int64_t)O4 * nb * 4) return;
  const int r = (int)(id & 3);
  const int64_t bg = id >> 2;
  const int g = (int)(bg % nb), b = (int)(bg / nb);
  const int row = b * 4 + r;
  constexpr int GB = Q8 ? 128 : 64;
  uint8_t* dst = q + (size_t)bg * GB + r * (Q8 ? 32 : 16);
  if (row >= O) {
#pragma unroll
    for (int j = 0; j < (Q8 ? 32 : 16); j += 4) *(uint32_t*)(dst + j) = Q8 ? 0u : 0x88888888u;
    d16[(size_t)bg * 4 + r] = 0;
    return;
  }
  const float* wg = w + (size_t)row * I + g * 32;
  float v[32];
#pragma unroll
  for (int j = 0; j < 32; j += 4) *(float4*)(v + j) = *(const float4*)(wg + j);
  float mx = 0.f;
#pragma unroll
  for (int j = 0; j < 32; j++) mx = fabsf(v[j]) > fabsf(mx) ? v[j] : mx;
  float opp = 0.f;
#pragma unroll
  for (int j = 0; j < 32; j++) opp = ((v[j] > 0) != (mx > 0) && fabsf(v[j]) > opp) ? fabsf(v[j]) : opp;
  const float lo = Q8 ? 128.f : 8.f, hi = Q8 ? 127.f : 7.f;
  const float dm = fmaxf(fabsf(mx) / lo, opp / hi);
  const uint32_t h = f32_to_f16(mx > 0 ? -dm : dm);
  const float dd = f16_to_f32(h), inv = dd != 0.f ? 1.f / dd : 0.f;
  d16[(size_t)bg * 4 + r] = (uint16_t)h;
  int c[32];
#pragma unroll
  for (int j = 0; j < 32; j++) {
    int t = rne_int(v[j] * inv);
    t = t < (Q8 ? -128 : -8) ? (Q8 ? -128 : -8) : t;
    t = t > (Q8 ? 127 : 7) ? (Q8 ? 127 : 7) : t;
    c[j] = t;
  }
  if (Q8) {
#pragma unroll
    for (int j = 0; j < 32; j += 4)
      *(uint32_t*)(dst + j) = (uint32_t)(c[j] & 0xff) | ((uint32_t)(c[j + 1] & 0xff) << 8) |
                              ((uint32_t)(c[j + 2] & 0xff) << 16) | ((uint32_t)(c[j + 3] & 0xff) << 24);
  } else {
#pragma unroll
    for (int j = 0; j < 16; j += 4) {
      uint32_t p = 0;
#pragma unroll
      for (int u = 0; u < 4; u++)
        p |= ((uint32_t)(c[j + u] + 8) | ((uint32_t)(c[j + u + 16] + 8) << 4)) << (8 * u);
      *(uint32_t*)(dst + j) = p;
    }
  }
}

int launch_pack_r4(bool q8, const float* w, uint8_t* q, uint16_t* d16, int O, int I, hipStream_t st) {
  if (I % 32 || I <= 0) return MOTY_EUNSUP;
  if (O <= 0) return MOTY_OK;
  const int64_t n = (int64_t)((O + 3) / 4) * (I / 32) * 4;
  const unsigned nbk = (unsigned)((n + 255) / 256);
  if (q8)
    hipLaunchKernelGGL(k_pack_r4<true>, dim3(nbk), dim3(256), 0, st, w, q, d16, O, I);
  else
    hipLaunchKernelGGL(k_pack_r4<false>, dim3(nbk), dim3(256), 0, st, w, q, d16, O, I);
  LAUNCH_TRY("k_pack_r4");
  return MOTY_OK;
}

}  // namespace moty
