// q4g.hip -- grouped int4 (group 32, f32 group scales) GEMV/GEMM.
//
// Reference: moty_matmul_i4_grouped_s (nn/matmul.c:164-197).
//  IDOT4=1 (gs == 32, I % 64 == 0):  xq = qrow_i8(x), then per output
//    acc = 0; for g ascending: acc = fma(scl[o][g], (float)(d_g - 8*xg_g), acc)
//    y = sx * acc                      (hw/hw_avx512.h:155-176, matmul.c:148-160)
//  default (exact f32 activations):  per group
//    t[j] = fma(x[j], w[j], x[j+16]*w[j+16]), j < 16; r = hsum16(t);
//    a = fma(r, scl[o][g], a)           (nn/matmul.c:199-253)
//
// The integer group dot d_g - 8*xg_g equals sum (n-8)*x exactly, so the
// kernels expand nibbles straight to signed int8 (n-8) and never need the
// group sums xg.  Group scales multiply a float chain whose order is fixed,
// so each output's chain runs in ascending group order in one lane.
#include "common.h"
#include "kernels.h"

#include <type_traits>

namespace moty {

// v_cvt_off_f32_i4 of byte K of w: the signed nibble in bits [8K, 8K+4)
// divided by 16 (exact), one SDWA-selected conversion
template <int K>
__device__ __forceinline__ float cvt_off_b(uint32_t w) {
  float r;
  if (K == 0)
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(r) : "v"(w));
  else if (K == 1)
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(r) : "v"(w));
  else if (K == 2)
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(r) : "v"(w));
  else
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(r) : "v"(w));
  return r;
}

// ---------------------------------------------------------------------------
// IDOT4 GEMV for decode (S = 1), optionally PAIR (gate + up + SiLU).
// Workgroup = 4 waves; a wave owns RW consecutive output rows (of W, and of
// W2 in PAIR mode):
//   1. it issues the nibble loads of its rows' first PD 64-group chunks --
//      lane l takes group l of each chunk (16 B, coalesced along the row) --
//      and each further chunk as the one PD before it is consumed;
//   2. the workgroup quantizes x into LDS (qrow_i8) while those loads fly;
//   3. per chunk, each lane forms its group's exact integer dot sum (n-8)*x
//      and parks it, with the group scale, in the wave's LDS slice;
//   4. one lane per row extends the reference's FMA chain over the chunk's
//      groups in order; y = sx * acc (PAIR: h = silu(g) * u).
// MT: several tokens, blockIdx.y, where a call must not keep its activation
// codes in memory (the weights of all but the first come from the caches).
template <int RW, int NGC, bool PAIR, int NT, int PD = NGC, bool XF = false, bool MT = false>
__global__ __launch_bounds__(NT) void k_gemv1_i4g(const float* __restrict__ x, const uint8_t* __restrict__ q4,
                                                      const float* __restrict__ scl,
                                                      const uint8_t* __restrict__ q4b,
                                                      const float* __restrict__ sclb, float* __restrict__ y, int I,
                                                      int O) {
  constexpr int NM = PAIR ? 2 : 1;
  constexpr int WAVES = NT / MOTY_WAVE;
  constexpr int XV = (NGC * 64 * 32) / (NT * 4);  // float4 of x per thread (I <= 2048 * NGC)
  extern __shared__ __align__(16) int8_t lds[];
  __shared__ float red[WAVES];
  __shared__ float sx_s;
  const int lane = threadIdx.x % MOTY_WAVE, wv = threadIdx.x / MOTY_WAVE;
  const int ng = I / 32, rb = I / 2;
  if constexpr (MT) {
    x += (int64_t)blockIdx.y * I;
    y += (int64_t)blockIdx.y * O;
  }
  constexpr int ldv = 66;  // one chunk's 64 groups, padded (even: float4 reads stay aligned)
  int8_t* xq_s = lds;                                                          // [I]
  int* xg8 = (int*)(lds + I);                                                  // [ng] -8 * group sums
  float* xf_s = (float*)lds;  // XF: [ng][36] f32 -- each group's 32 values, rows padded to 144 B so
                              // the lanes' 16-byte reads of their groups spread over the banks
  float2* dv = (float2*)(lds + (XF ? 4 * ng * 36 : I + ng * 4)) + (size_t)wv * (NM * RW * ldv);  // [NM*RW][ldv] (scale, dot) of one chunk
  const int o0 = (blockIdx.x * WAVES + wv) * RW;

  // 1. x (one pass, kept in registers), then every nibble load of this wave
  float4 xr[XV];
#pragma unroll
  for (int j = 0; j < XV; j++) {
    const int i = (threadIdx.x + j * NT) * 4;
    xr[j] = *(const float4*)(x + (i < I ? i : 0));  // clamped: zeroed below
  }
  int4 wb[NM][RW][NGC];
  float wsc[NM][RW][NGC];  // group scales, loaded with the nibbles
  // chunk-major issue order, PD chunks ahead: chunk c of every row is
  // issued before chunk c+1, and chunk c+PD only when chunk c is consumed,
  // so each row's data arrives spread over the stream and its FMA chain
  // (one dependent FMA per group) runs behind it; with every chunk issued
  // at once a row's whole chain would start after its last byte lands
  // (the compiler waits only for the chunk it consumes)
  auto issue = [&](int c) {
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
      for (int r = 0; r < RW; r++) {
        const int64_t o = o0 + r < O ? o0 + r : O - 1;
        // clamped (unused past ng): unconditional loads keep the wave's
        // loads in one straight run, with no wait at branch joins
        const int g = c * 64 + lane < ng ? c * 64 + lane : 0;
        {
          const v4i t = __builtin_nontemporal_load((const v4i*)((m ? q4b : q4) + o * rb + g * 16));
          wb[m][r][c] = int4{t.x, t.y, t.z, t.w};
        }
        wsc[m][r][c] = __builtin_nontemporal_load((m ? sclb : scl) + o * ng + g);
      }
  };
#pragma unroll
  for (int c = 0; c < PD; c++) issue(c);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < XV; j++) xr[j] = sel4((threadIdx.x + j * NT) * 4 < I, xr[j]);
  // XF: x into LDS as 16 x (exact) when every |x| < 2^123 -- then the
  // nibbles convert as (n - 8) / 16 and each product, hence each rounding,
  // is the reference's -- else as it is, for the full-width conversion
  bool x16 = false;
  if (XF) {
    bool big = false;
#pragma unroll
    for (int j = 0; j < XV; j++)
      big |= fmaxf(fmaxf(fabsf(xr[j].x), fabsf(xr[j].y)), fmaxf(fabsf(xr[j].z), fabsf(xr[j].w))) >= 0x1p123f;
    x16 = !__syncthreads_or(big);
#pragma unroll
    for (int j = 0; j < XV; j++) {
      const int i = (threadIdx.x + j * NT) * 4;
      float4 v = xr[j];
      if (x16) v = float4{16.f * v.x, 16.f * v.y, 16.f * v.z, 16.f * v.w};
      if (i < I) *(float4*)(xf_s + (i >> 5) * 36 + (i & 31)) = v;
    }
    __syncthreads();
  } else {
  // 2. qrow_i8 of x into LDS
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < XV; j++)
    amax = fmaxf(amax, fmaxf(fmaxf(fabsf(xr[j].x), fabsf(xr[j].y)), fmaxf(fabsf(xr[j].z), fabsf(xr[j].w))));
  amax = wave_max_f32(amax);
  if (lane == 0) red[wv] = amax;
  __syncthreads();
  {
    float mx = red[0];
#pragma unroll
    for (int i = 1; i < WAVES; i++) mx = fmaxf(mx, red[i]);
    float sc = mx / 127.f;
    if (sc < 1e-12f) sc = 1e-12f;
    const float inv = 1.f / sc;
    if (threadIdx.x == 0) sx_s = sc;
#pragma unroll
    for (int j = 0; j < XV; j++) {
      const int i = (threadIdx.x + j * NT) * 4;
      const float4 v = xr[j];
      if (i < I)
        *(uint32_t*)(xq_s + i) = (uint32_t)(rne_int(v.x * inv) & 0xff) | ((uint32_t)(rne_int(v.y * inv) & 0xff) << 8) |
                                 ((uint32_t)(rne_int(v.z * inv) & 0xff) << 16) |
                                 ((uint32_t)(rne_int(v.w * inv) & 0xff) << 24);
    }
  }
  __syncthreads();
  // -8 * each group's activation sum: the dots run on the unsigned codes n
  // and start from it, giving sum (n-8)*x exactly
  for (int g = threadIdx.x; g < ng; g += NT) {
    const int4 a = *(const int4*)(xq_s + g * 32), b = *(const int4*)(xq_s + g * 32 + 16);
    xg8[g] = -8 * dot16(b, int4{0x01010101, 0x01010101, 0x01010101, 0x01010101},
                        dot16(a, int4{0x01010101, 0x01010101, 0x01010101, 0x01010101}, 0));
  }
  __syncthreads();
  }
  // 3./4. per 64-group chunk: every lane forms its group's exact integer dot
  // for each row and parks (scale, dot) in the wave's LDS slice; then lane
  // j < NM*RW continues the FMA chain of its row (j % RW of matrix j / RW)
  // over the chunk's groups in order, while later chunks may still arrive.
  // 16-byte LDS reads carry two groups' pairs.
  float acc = 0.f;
#pragma unroll
  for (int c = 0; c < NGC; c++) {
    if (c + PD < NGC) {
      issue(c + PD);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int g = c * 64 + lane;
    if (XF && g < ng) {
      // the reference's exact f32 group sum (nn/matmul.c:222-233, the
      // AVX-512 form with FMA contraction): t[j] = fma(x[j], w[j],
      // x[16+j]*w[16+j]), then the 16 -> 8 -> 4 -> 1 reduction tree
      float xv[32];
#pragma unroll
      for (int q = 0; q < 8; q++) *(float4*)(xv + 4 * q) = *(const float4*)(xf_s + g * 36 + 4 * q);
#pragma unroll
      for (int m = 0; m < NM; m++)
#pragma unroll
        for (int r = 0; r < RW; r++) {
          const int4 w = wb[m][r][c];
          const uint32_t wd[4] = {(uint32_t)w.x, (uint32_t)w.y, (uint32_t)w.z, (uint32_t)w.w};
          float wf[32];  // element e = byte e/2, low nibble when e is even, minus 8 (exact)
          if (x16) {
            // (n - 8) / 16: n ^ 8 is n - 8 as a signed nibble, and
            // v_cvt_off_f32_i4 gives a signed nibble / 16 from the low
            // 4 bits of its byte-selected operand
#pragma unroll
            for (int q = 0; q < 4; q++) {
              const uint32_t a = wd[q] ^ 0x88888888u, b = a >> 4;
              wf[8 * q + 0] = cvt_off_b<0>(a);
              wf[8 * q + 1] = cvt_off_b<0>(b);
              wf[8 * q + 2] = cvt_off_b<1>(a);
              wf[8 * q + 3] = cvt_off_b<1>(b);
              wf[8 * q + 4] = cvt_off_b<2>(a);
              wf[8 * q + 5] = cvt_off_b<2>(b);
              wf[8 * q + 6] = cvt_off_b<3>(a);
              wf[8 * q + 7] = cvt_off_b<3>(b);
            }
          } else {
#pragma unroll
            for (int q = 0; q < 4; q++) {
              // n - 8 as signed bytes ((n + 0x78) ^ 0x80, carry-free),
              // each then converted from its byte position
              const uint32_t lo = ((wd[q] & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
              const uint32_t hi = (((wd[q] >> 4) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
#pragma unroll
              for (int k = 0; k < 4; k++) {
                wf[8 * q + 2 * k] = (float)(int8_t)(lo >> (8 * k));
                wf[8 * q + 2 * k + 1] = (float)(int8_t)(hi >> (8 * k));
              }
            }
          }
          float t[16];
#pragma unroll
          for (int j = 0; j < 16; j++) t[j] = __fmaf_rn(xv[j], wf[j], xv[16 + j] * wf[16 + j]);
          float u[8], v[4];
#pragma unroll
          for (int j = 0; j < 8; j++) u[j] = t[j + 8] + t[j];
#pragma unroll
          for (int j = 0; j < 4; j++) v[j] = u[j + 4] + u[j];
          dv[(m * RW + r) * ldv + lane] = float2{wsc[m][r][c], (v[0] + v[2]) + (v[1] + v[3])};
        }
    }
    if (!XF && g < ng) {
      const int4 x0 = *(const int4*)(xq_s + g * 32);
      const int4 x1 = *(const int4*)(xq_s + g * 32 + 16);
      const int c8 = xg8[g];
#pragma unroll
      for (int m = 0; m < NM; m++)
#pragma unroll
        for (int r = 0; r < RW; r++) {
          const int4 w = wb[m][r][c];
          const int4 w0 = unpack_nib16_u(uint2{(uint32_t)w.x, (uint32_t)w.y});
          const int4 w1 = unpack_nib16_u(uint2{(uint32_t)w.z, (uint32_t)w.w});
          const int d = dot16(w1, x1, dot16(w0, x0, c8));
          dv[(m * RW + r) * ldv + lane] = float2{wsc[m][r][c], (float)d};
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < NM * RW) {
      const int gend = ng < (c + 1) * 64 ? ng : (c + 1) * 64;
      const float4* dr = (const float4*)(dv + lane * ldv - c * 64);
      int gg = c * 64;
      for (; gg + 16 <= gend; gg += 16) {
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = dr[gg / 2 + u];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          acc = __fmaf_rn(v[u].x, v[u].y, acc);
          acc = __fmaf_rn(v[u].z, v[u].w, acc);
        }
      }
      const float2* d2 = dv + lane * ldv - c * 64;
      for (; gg < gend; gg++) acc = __fmaf_rn(d2[gg].x, d2[gg].y, acc);
    }
    // the next chunk's dots overwrite the slice: after these reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // XF: y = a (no activation scale)
  const float sxv = XF ? 0.f : sx_s;
  if (PAIR) {
    const float u = __shfl(acc, (lane + RW) & 63, 64);  // lane r < RW: the up row's chain
    const int o = o0 + lane;
    if (lane < RW && o < O) y[o] = XF ? ref_silu_mul(acc, u) : ref_silu_mul(sxv * acc, sxv * u);
  } else {
    const int o = o0 + lane;
    if (lane < RW && o < O) y[o] = XF ? acc : sxv * acc;
  }
}

// ---------------------------------------------------------------------------
// IDOT4 GEMM on v_mfma_i32_32x32x32_i8: one MFMA per group (K = 32 exactly),
// so each group's integer dot comes out separately and is folded into a
// float accumulator per output, in group order:
//     accf = fma(scl[o][g], (float)d, accf)
// Workgroup: 4 waves as 2 (tokens) x 2 (rows), block tile 64 x 64.  Per
// K block of 4 groups the workgroup stages, by whole-line loads, the int8
// activations (64 x 128 B), the nibbles (64 x 64 B) and the group scales
// (64 x 4) in LDS, the next block's loads in flight in registers.
// Lane l's A fragment is 16 bytes of token row (l % 32) at offset 16*(l/32)
// of the group; its B fragment the matching 8 nibble bytes of weight row
// (l % 32), expanded to signed n-8 -- one scale per lane per group.
constexpr int Q4M_NT = 256;
constexpr int Q4M_KG = 4;             // groups per K block
constexpr int Q4M_AS = 128 + 16;      // LDS row stride: activations
constexpr int Q4M_BS = 64 + 16;       // nibbles
constexpr int Q4M_SS = Q4M_KG + 1;    // scales

template <int NS = 2>
__global__ __launch_bounds__(Q4M_NT, 2) void k_gemm_i4g(const int8_t* __restrict__ xq, const float* __restrict__ sx,
                                                        const uint8_t* __restrict__ q4,
                                                        const float* __restrict__ scl, float* __restrict__ y,
                                                        int M, int I, int O) {
  __shared__ __align__(16) int8_t sA[64 * Q4M_AS];
  __shared__ __align__(16) uint8_t sB[64 * Q4M_BS];
  __shared__ float sS[64 * Q4M_SS];
  const int tid = threadIdx.x, lane = tid % MOTY_WAVE, wv = tid / MOTY_WAVE;
  const int wm = wv >> 1, wn = wv & 1;
  const int r32 = lane & 31, hk = lane >> 5;
  const int mb = blockIdx.y * 64, nb = blockIdx.x * 64;
  const int ng = I / 32, rb = I / 2;
  // copy assignments: A 2 x 16 B chunks (row = q/8, col16 = q%8), B 1 chunk
  // (row = tid/4, col16 = tid%4), S 1 float (row = tid/4, group = tid%4)
  const int8_t* srcA[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int q = tid + i * Q4M_NT;
    int m = mb + (q >> 3);
    m = m < M ? m : M - 1;
    srcA[i] = xq + (int64_t)m * I + (q & 7) * 16;
  }
  int nrow = nb + (tid >> 2);
  nrow = nrow < O ? nrow : O - 1;
  const uint8_t* srcB = q4 + (int64_t)nrow * rb + (tid & 3) * 16;
  const float* srcS = scl + (int64_t)nrow * ng + (tid & 3);
  // epilogue: the activation scale of tile row tid % 64, loaded now so its
  // latency hides behind the K loop (to LDS after it)
  __shared__ float s_sx[64];
  const float sxr = sx[mb + (tid & 63) < M ? mb + (tid & 63) : M - 1];
  // Two register sets: while one K block is consumed from LDS, the next two
  // are in flight.  Loads are unconditional, from clamped addresses (a block
  // past the end re-reads the last one; a chunk past the row end re-reads
  // the row start), and are masked when written to LDS: with no branch
  // around a load the compiler waits only for the set about to be consumed.
  // I % 64 == 0, so a K block of 4 groups (128 elements) is whole or the
  // last 2 groups of the row are missing (I % 128 == 64).
  struct Set {
    int4 a[2];
    int4 b;
    float s;
  };
  Set sets[NS];
  const int glast = (ng - 1) / Q4M_KG * Q4M_KG;
  auto gload = [&](int g0, Set& st) {
    const int gc = g0 < ng ? g0 : glast;
    const int kb = gc * 32;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int q = tid + i * Q4M_NT;
      st.a[i] = *(const int4*)(srcA[i] + (kb + (q & 7) * 16 < I ? kb : -(q & 7) * 16));
    }
    st.b = *(const int4*)(srcB + (gc * 16 + (tid & 3) * 16 < rb ? gc * 16 : -(tid & 3) * 16));
    st.s = srcS[gc + (tid & 3) < ng ? gc : -(tid & 3)];
    __builtin_amdgcn_sched_barrier(0);
  };
  float accf[16];
#pragma unroll
  for (int r = 0; r < 16; r++) accf[r] = 0.f;
  auto stage = [&](int g0, Set& st) {
    const int kb = g0 * 32;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int q = tid + i * Q4M_NT;
      *(int4*)(sA + (q >> 3) * Q4M_AS + (q & 7) * 16) = sel4(kb + (q & 7) * 16 < I, st.a[i]);
    }
    *(int4*)(sB + (tid >> 2) * Q4M_BS + (tid & 3) * 16) = sel4(g0 * 16 + (tid & 3) * 16 < rb, st.b);
    sS[(tid >> 2) * Q4M_SS + (tid & 3)] = g0 + (tid & 3) < ng ? st.s : 0.f;
    __syncthreads();
    gload(g0 + NS * Q4M_KG, st);
    // Straight-line over the block's 4 groups -- fragments, then the 4
    // MFMAs, then the 4 epilogues in group order -- so the MFMAs overlap
    // each other and the fragment reads.  Groups past the row end hold zero
    // codes, activations and scales: their step fma(0, 0, acc) adds
    // exactly nothing (acc is never -0: it starts at +0, and an exact zero
    // result rounds to +0).
    if (g0 < ng) {
      v4i a[Q4M_KG];
      int4 w[Q4M_KG];
      float sc[Q4M_KG];
#pragma unroll
      for (int gg = 0; gg < Q4M_KG; gg++) {
        a[gg] = *(const v4i*)(sA + (wm * 32 + r32) * Q4M_AS + gg * 32 + hk * 16);
        w[gg] = unpack_nib16(*(const uint2*)(sB + (wn * 32 + r32) * Q4M_BS + gg * 16 + hk * 8));
        sc[gg] = sS[(wn * 32 + r32) * Q4M_SS + gg];
      }
      v16i d[Q4M_KG];
#pragma unroll
      for (int gg = 0; gg < Q4M_KG; gg++)
        d[gg] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[gg], *(const v4i*)&w[gg], v16i{}, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);  // all four MFMAs issue before the epilogues
#pragma unroll
      for (int gg = 0; gg < Q4M_KG; gg++)
#pragma unroll
        for (int r = 0; r < 16; r++) accf[r] = __fmaf_rn(sc[gg], (float)d[gg][r], accf[r]);
    }
    __syncthreads();
  };
#pragma unroll
  for (int i = 0; i < NS; i++) gload(i * Q4M_KG, sets[i]);
  for (int g0 = 0; g0 < ng; g0 += NS * Q4M_KG) {
#pragma unroll
    for (int i = 0; i < NS; i++) stage(g0 + i * Q4M_KG, sets[i]);
  }
  // retire the clamped prefetch still in flight once, here: otherwise the
  // compiler waits for every memory operation before each conditional store
  __builtin_amdgcn_s_waitcnt(0);
  if (tid < 64) s_sx[tid] = sxr;
  __syncthreads();
  const int col = nb + wn * 32 + r32;
  if (col >= O) return;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int rl = wm * 32 + 8 * (r >> 2) + 4 * hk + (r & 3);
    if (mb + rl < M) y[(int64_t)(mb + rl) * O + col] = s_sx[rl] * accf[r];
  }
}

// ---------------------------------------------------------------------------
// IDOT4 GEMM on f16 MFMA (v_mfma_f32_32x32x16_f16, two per group).  The
// reference's per-group step is acc = fma(scl[o][g], (float)d_g, acc) in group
// order, d_g = sum over the group of (n - 8) * xq: an exact integer.  With f16
// operands -- activation codes in [-127, 127] and weight codes n - 8 in
// [-8, 7] are exact halves, every partial sum is an integer below 2^24 -- the
// MFMA returns d_g already as an exact float, so the epilogue is one FMA per
// output per group instead of a conversion and an FMA.
//
// Weight nibbles become halves with one v_and_or_b32 per pair and no
// float op: in a dword of 4 weight bytes, (w & 0x000f000f) | 0x64006400 is
// the half pair (1024 + n) of the low nibbles of bytes 0 and 2, the mask
// 0x00f000f0 gives (1024 + 16 n) for their high nibbles, and w >> 8 serves
// bytes 1 and 3 alike.  So a lane's 8 bytes of a group (16 codes e0..e15)
// become two 8-half fragments, low nibbles [e0,e4,e2,e6,e8,e12,e10,e14] and
// high nibbles [e1,e5,...] at 16x, matched by k_qrow_f16p's activation
// fragments x and x/16.  With the activations x, the two MFMAs give
//   sum_lo x (1024 + n) + sum_hi x (64 + n) = d_g + 1032 sum_lo x + 72 sum_hi x,
// and two more MFMAs of the same activation fragments against constant
// fragments (-1032 and -1152 = -72 * 16) give the offset, once per token
// tile and group for every weight tile: it enters the first product MFMA as
// its accumulator.  Every value is an integer below 2^23 in magnitude (|x|
// <= 127, 16 terms of each kind), so every sum is exact and d_g comes out
// exactly as the reference's integer group dot.
//
// Block tile BM tokens x BN weight rows, 4 waves as 2 x 2, each wave FM x FN
// 32 x 32 tiles.  K blocks of 4 groups (128 elements) move global -> LDS by
// DMA, S - 1 blocks ahead: per stage BM activation rows of 256 B (16-byte
// chunk c of row r in slot c ^ (r & 15): a ds_read_b128 cycle's 16 rows hit
// 16 distinct bank groups), BN nibble rows of 64 B (chunk c in slot
// c ^ ((r >> 2) & 3)) and BN scale rows of 16 B (the block's 4 group scales).
// Lane l takes, for group j, half h = l / 32 of its rows' group: elements
// [16h, 16h + 16) -- the low-nibble fragment for MFMA 0, the high for MFMA 1.
constexpr int Q4H_NT = 256;

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

// A lane's 8 nibble bytes of a group -> the low- and high-nibble fragments.
// m = 0x000f000f, m4 = 0x00f000f0 and o = 0x64006400 arrive in VGPRs so that
// each pair is one v_and_or_b32 (VOP3 takes no literal here).
__device__ __forceinline__ void nib16_to_h(uint2 w, uint32_t m, uint32_t m4, uint32_t o, v8h& lo, v8h& hi) {
  const uint32_t t0 = w.x >> 8, t1 = w.y >> 8;
  typedef uint32_t u4v __attribute__((ext_vector_type(4)));
  lo = __builtin_bit_cast(v8h, u4v{(w.x & m) | o, (t0 & m) | o, (w.y & m) | o, (t1 & m) | o});
  hi = __builtin_bit_cast(v8h, u4v{(w.x & m4) | o, (t0 & m4) | o, (w.y & m4) | o, (t1 & m4) | o});
}
// T16 (16 x 16 x 32 MFMA, a whole group per instruction): one dword of 4
// weight bytes (codes e0..e7 of a lane's 8-element slice) -> the fragment
// [e0,e4,e2,e6 | e1,e5,e3,e7 at 16x] with the offsets taken off: n - 8 and
// 16 (n - 8), matched by activations [x0,x4,x2,x6 | x1,x5,x3,x7 / 16].
__device__ __forceinline__ v8h nib8_to_h_c(uint32_t w, uint32_t m, uint32_t m4, uint32_t o) {
  typedef uint32_t u4v __attribute__((ext_vector_type(4)));
  const uint32_t t = w >> 8;
  return __builtin_bit_cast(v8h, u4v{(w & m) | o, (t & m) | o, (w & m4) | o, (t & m4) | o}) +
         v8h{-1032, -1032, -1032, -1032, -1152, -1152, -1152, -1152};
}
// The same fragments with the offsets taken off in the halves (packed f16
// adds, exact): n - 8 and 16 (n - 8).
__device__ __forceinline__ void nib16_to_h_c(uint2 w, uint32_t m, uint32_t m4, uint32_t o, v8h& lo, v8h& hi) {
  nib16_to_h(w, m, m4, o, lo, hi);
  lo += v8h{-1032, -1032, -1032, -1032, -1032, -1032, -1032, -1032};
  hi += v8h{-1152, -1152, -1152, -1152, -1152, -1152, -1152, -1152};
}

// PAIR: gate and up rows of the same block tile in one pass (the activation
// fragments serve both), epilogue y = silu(sx*gate) * (sx*up) -- the
// gate_up + silu_rows of nn/ffn.c:28-37.
template <int BM, int BN, int S, int WGM, int NW, bool PAIR, bool T16 = false>
__global__ __launch_bounds__(NW * 64, NW <= 8 ? 8 / NW : 1) void k_gemm_i4g_h(const uint16_t* __restrict__ xh,
                                                                const float* __restrict__ sx,
                                                                const uint8_t* __restrict__ q4,
                                                                const float* __restrict__ scl,
                                                                const uint8_t* __restrict__ q4b,
                                                                const float* __restrict__ sclb,
                                                                float* __restrict__ y, int M, int I, int O) {
  constexpr int NP = PAIR ? 2 : 1;  // weight matrices
  // stage: BM activation rows x 256 B | NP x BN nibble rows x 64 B | NP x BN scale rows x 16 B
  constexpr int SA = BM * 256, SB = BN * 64, SS = BN * 16, STAGE = SA + NP * (SB + SS);
  // 1 KiB DMA instructions per stage: A 4 rows each, B 16 rows, scales 64
  // rows; wave wv takes instruction j * NW + wv of each region (the last
  // repeats when a region's count is not a multiple of NW)
  constexpr int JA = BM / 4, JB = NP * BN / 16, JS = NP * BN / 64;
  constexpr int NA = (JA + NW - 1) / NW, NB = (JB + NW - 1) / NW, NS = (JS + NW - 1) / NW;
  constexpr int NI = NA + NB + NS;
  constexpr int WGN = NW / WGM;  // waves along the tokens x along the rows
  constexpr int MT = T16 ? 16 : 32;  // MFMA tile edge
  constexpr int TM = BM / WGM, TN = BN / WGN, FM = TM / MT, FN = TN / MT;
  constexpr int NR = T16 ? 4 : 16;   // accumulators per lane and tile
  static_assert(BN % 64 == 0 && BM % 64 == 0 && FM >= 1 && FN >= 1, "whole 1 KiB DMA rows");
  __shared__ __align__(1024) uint8_t lds[S * STAGE];
  __shared__ float s_sx[BM];
  const int tid = threadIdx.x, lane = tid % MOTY_WAVE;
  const int wv = __builtin_amdgcn_readfirstlane(tid / MOTY_WAVE);
  const int wm = wv / WGN, wn = wv % WGN;
  const int r32 = lane & 31, h = lane >> 5;
  const int mb = blockIdx.y * BM, nb = blockIdx.x * BN;
  const int ng = I / 32;
  const v4i rA = buf_rsrc(xh, (uint32_t)M * I * 2);
  const v4i rB0 = buf_rsrc(q4, (uint32_t)O * (I / 2)), rS0 = buf_rsrc(scl, (uint32_t)O * ng * 4);
  const v4i rB1 = PAIR ? buf_rsrc(q4b, (uint32_t)O * (I / 2)) : rB0;
  const v4i rS1 = PAIR ? buf_rsrc(sclb, (uint32_t)O * ng * 4) : rS0;
  // per-lane source offsets of this wave's DMAs: A chunk c of row r goes to
  // slot c ^ (r & 15), B chunk c of row r to slot c ^ ((r >> 2) & 3); B and
  // scale instructions past the first matrix's count serve the second
  uint32_t voA[NA], voB[NB], voS[NS];
  int jA[NA], jB[NB], jS[NS];
#pragma unroll
  for (int j = 0; j < NA; j++) {
    jA[j] = j * NW + wv < JA ? j * NW + wv : JA - 1;
    const int row = jA[j] * 4 + (lane >> 4);
    const int c = (lane & 15) ^ (row & 15);
    const int m = mb + row < M ? mb + row : M - 1;
    voA[j] = (uint32_t)m * (uint32_t)I * 2u + (uint32_t)c * 16u;
  }
#pragma unroll
  for (int j = 0; j < NB; j++) {
    jB[j] = j * NW + wv < JB ? j * NW + wv : JB - 1;
    const int row = (jB[j] % (BN / 16)) * 16 + (lane >> 2);
    const int c = (lane & 3) ^ ((row >> 2) & 3);
    const int n = nb + row < O ? nb + row : O - 1;
    voB[j] = (uint32_t)n * (uint32_t)(I / 2) + (uint32_t)c * 16u;
  }
#pragma unroll
  for (int j = 0; j < NS; j++) {
    jS[j] = j * NW + wv < JS ? j * NW + wv : JS - 1;
    const int row = (jS[j] % (BN / 64)) * 64 + lane;
    const int n = nb + row < O ? nb + row : O - 1;
    voS[j] = (uint32_t)n * (uint32_t)ng * 4u;
  }
  const int nk = I / 128;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  auto issue = [&](int kb) {
    const uint32_t st0 = lds0 + (uint32_t)(kb % S) * STAGE;
#pragma unroll
    for (int j = 0; j < NA; j++) bdma16_to_lds(rA, voA[j], (uint32_t)kb * 256u, st0 + jA[j] * 1024);
#pragma unroll
    for (int j = 0; j < NB; j++)
      bdma16_to_lds(jB[j] < BN / 16 ? rB0 : rB1, voB[j], (uint32_t)kb * 64u, st0 + SA + jB[j] * 1024);
#pragma unroll
    for (int j = 0; j < NS; j++)
      bdma16_to_lds(jS[j] < BN / 64 ? rS0 : rS1, voS[j], (uint32_t)kb * 16u, st0 + SA + NP * SB + jS[j] * 1024);
  };
  // the tile's activation scales: the oldest load, covered by the waits below
  float sxr;
  {
    const int m = mb + tid % BM;
    sxr = sx[m < M ? m : M - 1];
  }
  uint32_t km, km4, ko;
  asm volatile("v_mov_b32 %0, 0x000f000f" : "=v"(km));
  asm volatile("v_mov_b32 %0, 0x00f000f0" : "=v"(km4));
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(ko));
  const v8h c_lo = v8h{-1032, -1032, -1032, -1032, -1032, -1032, -1032, -1032};
  const v8h c_hi = v8h{-1152, -1152, -1152, -1152, -1152, -1152, -1152, -1152};
  float acc[NP][FM][FN][NR];
#pragma unroll
  for (int p = 0; p < NP; p++)
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++)
#pragma unroll
        for (int r = 0; r < NR; r++) acc[p][i][j][r] = 0.f;
  // A K block's operands in registers: the activation fragments, the raw
  // nibble pairs and the scales of its 4 groups.  The next block's are read
  // from LDS while this one is unpacked and multiplied.
  struct Frags32 {
    v8h a[4][FM][2];
    uint2 b[4][NP][FN];
    float4 s[NP][FN];
  };
  // T16: one 8-half activation fragment and one nibble dword per group
  struct Frags16 {
    v8h a[4][FM];
    uint32_t b[4][NP][FN];
    float4 s[NP][FN];
  };
  using Frags = typename std::conditional<T16, Frags16, Frags32>::type;
  auto read = [&](int kb, Frags& f) {
    const uint8_t* st = lds + (kb % S) * STAGE;
    if constexpr (T16) {
      const int r16 = lane & 15, q = lane >> 4;
#pragma unroll
      for (int p = 0; p < NP; p++)
#pragma unroll
        for (int j = 0; j < FN; j++)
          f.s[p][j] = *(const float4*)(st + SA + NP * SB + p * SS + (wn * TN + j * 16 + r16) * 16);
#pragma unroll
      for (int gl = 0; gl < 4; gl++) {
#pragma unroll
        for (int i = 0; i < FM; i++) {
          const int row = wm * TM + i * 16 + r16;
          f.a[gl][i] = *(const v8h*)(st + row * 256 + (((4 * gl + q) ^ (row & 15)) * 16));
        }
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
          for (int j = 0; j < FN; j++) {
            const int row = wn * TN + j * 16 + r16;
            f.b[gl][p][j] = *(const uint32_t*)(st + SA + p * SB + row * 64 + ((gl ^ ((row >> 2) & 3)) * 16) + 4 * q);
          }
      }
      return;
    } else {
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (int j = 0; j < FN; j++)
        f.s[p][j] = *(const float4*)(st + SA + NP * SB + p * SS + (wn * TN + j * 32 + r32) * 16);
#pragma unroll
    for (int gl = 0; gl < 4; gl++) {
#pragma unroll
      for (int i = 0; i < FM; i++) {
        const int row = wm * TM + i * 32 + r32;
#pragma unroll
        for (int m = 0; m < 2; m++) {
          const int c = 4 * gl + 2 * h + m;
          f.a[gl][i][m] = *(const v8h*)(st + row * 256 + ((c ^ (row & 15)) * 16));
        }
      }
#pragma unroll
      for (int p = 0; p < NP; p++)
#pragma unroll
        for (int j = 0; j < FN; j++) {
          const int row = wn * TN + j * 32 + r32;
          f.b[gl][p][j] = *(const uint2*)(st + SA + p * SB + row * 64 + ((gl ^ ((row >> 2) & 3)) * 16) + 8 * h);
        }
    }
    }
  };
  // PAIR takes the offsets off in the weight halves (two packed adds per
  // 4 halves, shared by the FM token tiles); the single-matrix form, with
  // one weight tile per wave, computes them on the matrix core instead
  constexpr bool OFS_MFMA = !PAIR;
  auto compute = [&](const Frags& f) {
    if constexpr (T16) {
#pragma unroll
      for (int gl = 0; gl < 4; gl++) {
        v8h fb[NP][FN];
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
          for (int j = 0; j < FN; j++) fb[p][j] = nib8_to_h_c(f.b[gl][p][j], km, km4, ko);
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
          for (int p = 0; p < NP; p++)
#pragma unroll
            for (int j = 0; j < FN; j++) {
              const v4f d = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.a[gl][i], fb[p][j], v4f{}, 0, 0, 0);
              const float4 sv = f.s[p][j];
              const float s = gl == 0 ? sv.x : gl == 1 ? sv.y : gl == 2 ? sv.z : sv.w;
#pragma unroll
              for (int r = 0; r < 4; r++) acc[p][i][j][r] = __fmaf_rn(s, d[r], acc[p][i][j][r]);
            }
      }
      return;
    } else {
#pragma unroll
    for (int gl = 0; gl < 4; gl++) {
      v8h fb[NP][FN][2];
#pragma unroll
      for (int p = 0; p < NP; p++)
#pragma unroll
        for (int j = 0; j < FN; j++) {
          if (OFS_MFMA) nib16_to_h(f.b[gl][p][j], km, km4, ko, fb[p][j][0], fb[p][j][1]);
          else nib16_to_h_c(f.b[gl][p][j], km, km4, ko, fb[p][j][0], fb[p][j][1]);
        }
#pragma unroll
      for (int i = 0; i < FM; i++) {
        // the offset -1032 sum_lo x - 72 sum_hi x of each token row
        v16f d3 = v16f{};
        if (OFS_MFMA) {
          d3 = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[gl][i][0], c_lo, d3, 0, 0, 0);
          d3 = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[gl][i][1], c_hi, d3, 0, 0, 0);
        }
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
          for (int j = 0; j < FN; j++) {
            v16f d = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[gl][i][0], fb[p][j][0], d3, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[gl][i][1], fb[p][j][1], d, 0, 0, 0);
            const float4 sv = f.s[p][j];
            const float s = gl == 0 ? sv.x : gl == 1 ? sv.y : gl == 2 ? sv.z : sv.w;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[p][i][j][r] = __fmaf_rn(s, d[r], acc[p][i][j][r]);
          }
      }
    }
    }
  };
  // every stage of the ring in flight, then block 0's operands to registers
#pragma unroll
  for (int s = 0; s < S; s++) issue(s);
  MOTY_WAIT_VMCNT((S - 1) * NI);
  __syncthreads();
  Frags f0, f1;
  read(0, f0);
  for (int kb = 0; kb < nk; kb += 2) {
    // block kb + 1 has landed (the S - 2 later ones may still fly); the
    // barrier also retires every wave's reads of block kb's stage, which the
    // next DMA overwrites.  Blocks past the end read zeros, never consumed.
    MOTY_WAIT_VMCNT((S - 2) * NI);
    __syncthreads();
    issue(kb + S);
    read(kb + 1, f1);
    compute(f0);
    if (kb + 1 >= nk) break;
    MOTY_WAIT_VMCNT((S - 2) * NI);
    __syncthreads();
    issue(kb + 1 + S);
    read(kb + 2, f0);
    compute(f1);
  }
  __builtin_amdgcn_s_waitcnt(0);
  if (tid < BM) s_sx[tid] = sxr;
  __syncthreads();
  if constexpr (T16) {
    const int r16 = lane & 15, q = lane >> 4;
#pragma unroll
    for (int j = 0; j < FN; j++) {
      const int n = nb + wn * TN + j * 16 + r16;
      if (n >= O) continue;
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int ml = wm * TM + i * 16 + 4 * q + r;
          if (mb + ml >= M) continue;
          const float sv = s_sx[ml];
          y[(int64_t)(mb + ml) * O + n] =
              PAIR ? ref_silu_mul(sv * acc[0][i][j][r], sv * acc[NP - 1][i][j][r]) : sv * acc[0][i][j][r];
        }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < FN; j++) {
    const int n = nb + wn * TN + j * 32 + r32;
    if (n >= O) continue;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int ml = wm * TM + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (mb + ml >= M) continue;
        const float sv = s_sx[ml];
        y[(int64_t)(mb + ml) * O + n] =
            PAIR ? ref_silu_mul(sv * acc[0][i][j][r], sv * acc[NP - 1][i][j][r]) : sv * acc[0][i][j][r];
      }
  }
}

// The f16-MFMA GEMM (q4b/sclb non-null: PAIR, y = silu(x.q4^T) * (x.q4b^T)).
// Tiles from sweeps on MI355X at M = 256: 128 x 128 block tiles of 8 waves
// when they give at least 160 workgroups (PAIR gate + up, K = 4096, N =
// 12288: three stages 86 us, two 92, 64 x 128 93, 64 x 64 94; the 16 x 16
// form 93) -- except PAIR, where 64 x 192 tiles take over while 128 x 128
// ones would leave CUs idle and they number at least 192 (the same GEMM:
// 256 workgroups on 256 CUs against 192, 81 us against 86-91 alone; three
// stages 84, the 16 x 16 form 87-95).  Their 6 waves each take all 64 tokens
// of 32 gate and 32 up rows, so each unpacked weight fragment serves two
// token tiles: 78-80 us against 80-84 for 12 waves of 32 tokens (the FFN
// 157.0 against 159.6 us), though 6 waves leave two SIMDs a wave short;
// otherwise 64 x 64 tiles, PAIR of 4 waves in three stages, the
// single matrix in the 16 x 16 form: 8 waves of 32 x 16, four stages (down,
// K = 12288, N = 4096: 57 us; five or six stages 57.5 / 58, three 62; the
// 32 x 32 form of 4 waves 66, four stages 69, 128 x 128 113).
static bool gemm_i4g_h_big(int M, int O) { return (int64_t)((M + 127) / 128) * ((O + 127) / 128) >= 160; }
// 128 x 128 tiles give every CU a workgroup
static bool gemm_i4g_h_full(int M, int O) { return (int64_t)((M + 127) / 128) * ((O + 127) / 128) >= 256; }
static bool gemm_i4g_h_pair192(int M, int O) {
  return !gemm_i4g_h_full(M, O) && (int64_t)((M + 63) / 64) * ((O + 191) / 192) >= 192;
}
int gemm_i4g_h_f8(int M, int O, bool pair) { return !pair && !gemm_i4g_h_big(M, O); }

// the f16 GEMM's 32-bit buffer offsets: activations and nibbles under 4 GiB
bool gemm_i4g_h_fits(int M, int I, int O) {
  return (I % 128) == 0 && (int64_t)M * I * 2 < ((int64_t)1 << 32) && (int64_t)O * I / 2 < ((int64_t)1 << 32);
}

int launch_gemm_i4g_h(const uint16_t* xh, const float* sx, const uint8_t* q4, const float* scl, const uint8_t* q4b,
                      const float* sclb, float* y, int M, int I, int O, hipStream_t st) {
  if ((I % 128) || ((((uintptr_t)xh) | ((uintptr_t)q4) | ((uintptr_t)scl) | ((uintptr_t)q4b) | ((uintptr_t)sclb)) & 15))
    return MOTY_EUNSUP;
  if (!gemm_i4g_h_fits(M, I, O)) return MOTY_EUNSUP;
  if (M <= 0 || O <= 0) return MOTY_OK;
  const bool big = gemm_i4g_h_big(M, O);
#define Q4H(BM, BN, S, WGM, NW, P, T16)                                                                         \
  hipLaunchKernelGGL((k_gemm_i4g_h<BM, BN, S, WGM, NW, P, T16>), dim3((O + BN - 1) / BN, (M + BM - 1) / BM),   \
                     dim3(NW * 64), 0, st, xh, sx, q4, scl, q4b, sclb, y, M, I, O)
  if (q4b) {
    if (gemm_i4g_h_pair192(M, O)) Q4H(64, 192, 2, 1, 6, true, false);
    else if (big) Q4H(128, 128, 3, 2, 8, true, false);
    else Q4H(64, 64, 3, 2, 4, true, false);
  } else {
    if (big) Q4H(128, 128, 2, 2, 8, false, false);
    else Q4H(64, 64, 4, 2, 8, false, true);
  }
#undef Q4H
  LAUNCH_TRY("k_gemm_i4g_h");
  return MOTY_OK;
}

// ---------------------------------------------------------------------------
// Exact f32 path, any S: one lane per (row, token); x rows staged in LDS.
constexpr int Q4F_NT = 256;

__global__ __launch_bounds__(Q4F_NT) void k_i4g_f32(const float* __restrict__ x, const uint8_t* __restrict__ q4,
                                                    const float* __restrict__ scl, float* __restrict__ y, int S,
                                                    int I, int O) {
  const int s = blockIdx.y;
  const int o = blockIdx.x * Q4F_NT + threadIdx.x;
  if (o >= O) return;
  const int ng = I / 32, rb = I / 2;
  const float* xs = x + (int64_t)s * I;
  const uint8_t* w = q4 + (int64_t)o * rb;
  const float* sp = scl + (int64_t)o * ng;
  float a = 0.f;
  for (int g = 0; g < ng; g++) {
    const int4 wb = *(const int4*)(w + g * 16);
    const uint32_t wd[4] = {(uint32_t)wb.x, (uint32_t)wb.y, (uint32_t)wb.z, (uint32_t)wb.w};
    float t[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      // element j (bytes 0..7) and element 16+j (bytes 8..15)
      const uint32_t b0 = (wd[j >> 3] >> (8 * ((j >> 1) & 3))) & 0xffu;
      const uint32_t b1 = (wd[2 + (j >> 3)] >> (8 * ((j >> 1) & 3))) & 0xffu;
      const int n0 = (j & 1) ? (int)(b0 >> 4) : (int)(b0 & 0xf);
      const int n1 = (j & 1) ? (int)(b1 >> 4) : (int)(b1 & 0xf);
      const float p1 = xs[g * 32 + 16 + j] * (float)(n1 - 8);
      t[j] = __fmaf_rn(xs[g * 32 + j], (float)(n0 - 8), p1);
    }
    float u[8], v[4];
#pragma unroll
    for (int j = 0; j < 8; j++) u[j] = t[j + 8] + t[j];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = u[j + 4] + u[j];
    const float r = (v[0] + v[2]) + (v[1] + v[3]);
    a = __fmaf_rn(r, sp[g], a);
  }
  y[(int64_t)s * O + o] = a;
}

// ---------------------------------------------------------------------------
// Per-row int4 (WF_I4), exact f32 path of moty_matmul_i4_s
// (nn/matmul.c:102-145) in the x86-64 AVX2 order: eight accumulator lanes,
// lane j takes elements i+j then i+8+j of each 16-element step (an FMA each),
// then simd_hsum256_f32's tree (hw/hw_avx2.h:16-20), y = a * scale.  Lane
// per (row, token), I % 16 == 0.
__global__ __launch_bounds__(256) void k_i4row_f32(const float* __restrict__ x, const uint8_t* __restrict__ q4,
                                                   const float* __restrict__ scale, float* __restrict__ y, int S,
                                                   int I, int O) {
  const int s = blockIdx.y;
  const int o = blockIdx.x * 256 + threadIdx.x;
  if (o >= O) return;
  const float* xs = x + (int64_t)s * I;
  const uint8_t* w = q4 + (int64_t)o * (I / 2);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < I; i += 16) {
    const uint2 wb = *(const uint2*)(w + i / 2);
    const uint32_t wd[2] = {wb.x, wb.y};
    float xv[16];
#pragma unroll
    for (int q = 0; q < 4; q++) *(float4*)(xv + 4 * q) = *(const float4*)(xs + i + 4 * q);
#pragma unroll
    for (int half = 0; half < 2; half++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int e = 8 * half + j;  // element i + e: byte e / 2, low nibble when even
        const uint32_t byte = (wd[e >> 3] >> (8 * ((e >> 1) & 3))) & 0xffu;
        const int n = (e & 1) ? (int)(byte >> 4) : (int)(byte & 15u);
        acc[j] = __fmaf_rn(xv[e], (float)(n - 8), acc[j]);
      }
  }
  const float a0 = acc[0] + acc[4], a1 = acc[1] + acc[5], a2 = acc[2] + acc[6], a3 = acc[3] + acc[7];
  const float b0 = a0 + a2, b1 = a1 + a3;
  y[(int64_t)s * O + o] = (b0 + b1) * scale[o];
}

int launch_i4row_f32(const float* x, const uint8_t* q4, const float* scale, float* y, int S, int I, int O,
                     hipStream_t st) {
  if (I % 16 || (((uintptr_t)q4) & 7) || (((uintptr_t)x) & 15)) return MOTY_EUNSUP;
  if (S <= 0 || O <= 0) return MOTY_OK;
  hipLaunchKernelGGL(k_i4row_f32, dim3((O + 255) / 256, S), dim3(256), 0, st, x, q4, scale, y, S, I, O);
  LAUNCH_TRY("k_i4row_f32");
  return MOTY_OK;
}

// NT = 256 or 512 threads: wider workgroups amortize the activation row
// (read once per workgroup) over more weight rows when I is large
template <int RW, int NGC, bool PAIR, int NT, int PD = NGC, bool XF = false, bool MT = false>
static int go_gemv1_i4g(const float* x, const uint8_t* q4, const float* scl, const uint8_t* q4b, const float* sclb,
                        float* y, int I, int O, hipStream_t st, int S = 1) {
  constexpr int NM = PAIR ? 2 : 1;
  const int ng = I / 32;
  const size_t lds = (XF ? (size_t)ng * 36 * 4 : (size_t)I + (size_t)ng * 4) + (size_t)(NT / MOTY_WAVE) * NM * RW * 66 * 8;
  if (lds > 150 * 1024) return MOTY_EUNSUP;  // within the CU's 160 KiB, static arrays included
  if (lds > 64 * 1024) {
    // past 64 KiB of dynamic LDS: raise the instance's allowance on this
    // device to what this launch needs (kept when larger)
    static size_t allowed[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
      (void)hipGetLastError();
      return MOTY_EUNSUP;
    }
    if (lds > allowed[dev]) {
      if (hipFuncSetAttribute((const void*)&k_gemv1_i4g<RW, NGC, PAIR, NT, PD, XF, MT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
        (void)hipGetLastError();  // leave no error for a later call to find
        return MOTY_EUNSUP;
      }
      allowed[dev] = lds;
    }
  }
  const unsigned nb = (unsigned)((O + RW * (NT / MOTY_WAVE) - 1) / (RW * (NT / MOTY_WAVE)));
  hipLaunchKernelGGL((k_gemv1_i4g<RW, NGC, PAIR, NT, PD, XF, MT>), dim3(nb, S), dim3(NT), lds, st, x, q4, scl, q4b, sclb, y, I, O);
  LAUNCH_TRY("k_gemv1_i4g");
  return MOTY_OK;
}

// The exact-f32 path (IDOT4 unset) for one token: the same workgroup
// structure with x kept as f32 in LDS and each lane's group sum formed in
// the reference's float order.  I % 32 == 0, I <= 16384 (x in LDS: past
// 12288 more than 64 KiB of it), 16-byte aligned x and nibbles.  PAIR (q4b):
// gate + up + SiLU.
int launch_gemv_i4g_xf(const float* x, const uint8_t* q4, const float* scl, const uint8_t* q4b, const float* sclb,
                       float* y, int I, int O, hipStream_t st) {
  if ((I % 32) || I > 16384 || ((((uintptr_t)x) | ((uintptr_t)q4) | ((uintptr_t)q4b)) & 15)) return MOTY_EUNSUP;
  if (O <= 0) return MOTY_OK;
  const int ngc = (I / 32 + 63) / 64;
  if (q4b) {
    // 2 gate + 2 up rows per wave (C3 M = 1 exact-f32 FFN 25.7 -> 25.2 us against 4 + 4)
    if (ngc <= 2) return go_gemv1_i4g<2, 2, true, 256, 1, true>(x, q4, scl, q4b, sclb, y, I, O, st);
    if (ngc <= 4) return go_gemv1_i4g<2, 4, true, 256, 1, true>(x, q4, scl, q4b, sclb, y, I, O, st);
    if (ngc <= 6) return go_gemv1_i4g<2, 6, true, 256, 1, true>(x, q4, scl, q4b, sclb, y, I, O, st);
    return go_gemv1_i4g<2, 8, true, 256, 1, true>(x, q4, scl, q4b, sclb, y, I, O, st);
  }
  if (ngc <= 2) return go_gemv1_i4g<8, 2, false, 256, 1, true>(x, q4, scl, nullptr, nullptr, y, I, O, st);
  if (ngc <= 4) return go_gemv1_i4g<4, 4, false, 256, 1, true>(x, q4, scl, nullptr, nullptr, y, I, O, st);
  // 2 rows per wave (4096 x 12288: 10.6 -> 10.2 us against 4)
  if (ngc <= 6) return go_gemv1_i4g<2, 6, false, 256, 1, true>(x, q4, scl, nullptr, nullptr, y, I, O, st);
  return go_gemv1_i4g<2, 8, false, 256, 1, true>(x, q4, scl, nullptr, nullptr, y, I, O, st);
}

// one matrix: the widest instance whose LDS fits, else the next narrower one
template <bool MT>
static int go_gemv_i4g(const float* x, const uint8_t* q4, const float* scl, float* y, int I, int O, hipStream_t st, int S) {
  const int ngc = (I / 32 + 63) / 64;
  int rc = MOTY_EUNSUP;
  if (ngc <= 2) rc = go_gemv1_i4g<8, 2, false, 256, 2, false, MT>(x, q4, scl, nullptr, nullptr, y, I, O, st, S);
  else if (ngc <= 4) {
    rc = go_gemv1_i4g<4, 4, false, 512, 4, false, MT>(x, q4, scl, nullptr, nullptr, y, I, O, st, S);
    if (rc == MOTY_EUNSUP) rc = go_gemv1_i4g<4, 4, false, 256, 4, false, MT>(x, q4, scl, nullptr, nullptr, y, I, O, st, S);
  } else if (ngc <= 6) {
    // 4096 x 12288 (8B down) in a sweep of rows/wave x workgroup size x
    // chunks in flight on MI355X, graph replays over rotating weights:
    // 4 rows x 256 threads, one chunk ahead 8.0 us; two ahead 9.3, all six
    // 10.9 (the whole row's chains then run after its last byte lands);
    // 2 rows 9.6 / 10.9; 8 rows x 128 threads 10.1
    rc = go_gemv1_i4g<4, 6, false, 256, 1, false, MT>(x, q4, scl, nullptr, nullptr, y, I, O, st, S);
  } else if (ngc <= 8) {
    rc = go_gemv1_i4g<2, 8, false, 256, 8, false, MT>(x, q4, scl, nullptr, nullptr, y, I, O, st, S);
  }
  return rc;
}

int launch_gemv_i4g(const float* x, const uint8_t* q4, const float* scl, const uint8_t* q4b, const float* sclb,
                    float* y, int I, int O, hipStream_t st, int S) {
  if ((I % 64) || I > 16384 || (q4b && S > 1)) return MOTY_EUNSUP;
  if (O <= 0 || S <= 0) return MOTY_OK;
  if (q4b) {
    const int ngc = (I / 32 + 63) / 64;
    int rc = MOTY_EUNSUP;
    // up to 2 chunks (I <= 4096): 2 gate + 2 up rows per wave (12288 x
    // 4096 pair: 12.2 us against 12.5 with 4 + 4, 14.2 with 1 + 1, 13.6
    // for 2 + 2 in 2-wave workgroups or with both chunks issued at once)
    if (ngc <= 2) rc = go_gemv1_i4g<2, 2, true, 256, 1>(x, q4, scl, q4b, sclb, y, I, O, st);
    else if (ngc <= 4) {
      rc = go_gemv1_i4g<2, 4, true, 512>(x, q4, scl, q4b, sclb, y, I, O, st);
      if (rc == MOTY_EUNSUP) rc = go_gemv1_i4g<2, 4, true, 256>(x, q4, scl, q4b, sclb, y, I, O, st);
    } else if (ngc <= 8) {
      rc = go_gemv1_i4g<1, 8, true, 512>(x, q4, scl, q4b, sclb, y, I, O, st);
      if (rc == MOTY_EUNSUP) rc = go_gemv1_i4g<1, 8, true, 256>(x, q4, scl, q4b, sclb, y, I, O, st);
    }
    return rc;
  }
  return S == 1 ? go_gemv_i4g<false>(x, q4, scl, y, I, O, st, 1) : go_gemv_i4g<true>(x, q4, scl, y, I, O, st, S);
}

int launch_gemm_i4g(const int8_t* xq, const float* sx, const uint8_t* q4, const float* scl, float* y, int M,
                    int I, int O, hipStream_t st) {
  if (I % 64) return MOTY_EUNSUP;
  if (M <= 0 || O <= 0) return MOTY_OK;
  dim3 grid((O + 63) / 64, (M + 63) / 64);
  // three K blocks in flight for long rows (I = 4096, O = 12288, M = 256:
  // 76 us vs 82 with two, in a sweep on MI355X)
  if (I >= 4096)
    hipLaunchKernelGGL(k_gemm_i4g<3>, grid, dim3(Q4M_NT), 0, st, xq, sx, q4, scl, y, M, I, O);
  else
    hipLaunchKernelGGL(k_gemm_i4g<2>, grid, dim3(Q4M_NT), 0, st, xq, sx, q4, scl, y, M, I, O);
  LAUNCH_TRY("k_gemm_i4g");
  return MOTY_OK;
}

// ---------------------------------------------------------------------------
// The exact-f32 path (IDOT4 unset) for several tokens, on f32 matrix
// instructions.  v_mfma_f32_16x16x1_4b_f32 is four independent 16 x 16 outer
// products with one fused multiply-add per output (k = 1), bit for bit
// v_fma_f32 of the same operands (checked on random triples, wide exponents,
// denormals and signed zeros), so block b of one instruction carries one j of
// the reference's group step (nn/matmul.c:222-233 with FMA contraction):
//   p    = fma(x[16+j], w[16+j], -0)          the rounded product, its sign of zero kept
//   t[j] = fma(x[j], w[j], p)                 (j < 16)
//   u[j] = t[j+8] + t[j];  v[j] = u[j+4] + u[j];  r = (v0 + v2) + (v1 + v3)
//   a    = fma(r, scale[g], a)                (groups in ascending order)
// Instruction q takes j = q, q+4, q+8, q+12 in its four blocks, whose results
// for one output land in one lane, so the tree is 15 adds per output and group
// in registers, and a lane's operands are two float4s of its x row (elements
// 4b.. and 16 + 4b.., b = lane / 16) and the four nibble bytes of the same
// elements of its weight row.
//
// Wave (wm, wn, ks) owns TM x TN tiles of 16 tokens x 16 weight rows (PAIR:
// TN = 2, the same 16 gate and up rows) and, of every K step's KG groups,
// those with index ks mod KS.  With KS = 4 the waves of a tile hand the group
// sums r over through LDS and wave ks continues the chains of the tile's
// register ks: the r of different groups are independent, only the chain, one
// FMA per group, is serial.  Steps are double-buffered in LDS, one barrier
// per step.
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));

// signed byte K of w as a float
template <int K>
__device__ __forceinline__ float cvt_sb(uint32_t w) { return (float)(int)(int8_t)(w >> (8 * K)); }

template <int TM, int TN, int WM, int WN, int KS, int KG, bool PAIR>
__global__ __launch_bounds__(64 * WM * WN * KS) void k_gemm_i4g_xf(const float* __restrict__ x,
                                                                   const uint8_t* __restrict__ q4,
                                                                   const float* __restrict__ scl,
                                                                   const uint8_t* __restrict__ q4b,
                                                                   const float* __restrict__ sclb,
                                                                   float* __restrict__ y, int M, int I, int O) {
  static_assert(!PAIR || TN == 2, "PAIR: one gate and one up tile per wave");
  static_assert(KG % KS == 0 && (KS == 1 || KS == 4 || KS == 8), "groups of a step over the K waves");
  constexpr int NT = 64 * WM * WN * KS;
  constexpr int BM = 16 * TM * WM, BW = 16 * TN * WN;  // tokens, weight rows of the tile
  constexpr int OC = PAIR ? BW / 2 : BW;               // output columns
  constexpr int XS = KG * 128;      // LDS row stride of x: 16-byte chunks, XOR-swizzled by row
  constexpr int WS = KG * 16 + 16;  // of the nibbles: padded, the 2-byte reads of 16 rows hit 16 banks
  constexpr int XC = BM * KG * 8, WC = BW * KG;  // a step's 16-byte pieces of x and of the nibbles
  constexpr int NX = (XC + NT - 1) / NT, NW = (WC + NT - 1) / NT;
  constexpr int NR = KS == 1 ? 4 : 1;  // chains per tile and lane
  __shared__ __align__(16) uint8_t xs[2][BM * XS];
  __shared__ __align__(16) uint8_t ws[2][BW * WS];
  __shared__ __align__(16) float ss[2][BW * KG];
  __shared__ float rs[2][KS > 1 ? WM * WN * KG * TM * TN * 256 : 1];  // group sums of a step
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int ks = wv % KS, wt = wv / KS, wm = wt / WN, wn = wt % WN;
  const int r16 = lane & 15, b = lane >> 4;
  const int tb = blockIdx.y * BM, ob = blockIdx.x * OC;
  const int ng = I / 32, rb = I / 2;

  // staging: piece c of x is chunk c % (8 KG) of row c / (8 KG), of the
  // nibbles group c % KG of row c / KG.  Rows past the end re-read the last
  // one; pieces past a row's end re-read its first (never used).
  float4 px[NX];
  u32x4_a8 pw[NW];
  float ps[NW];
  auto gload = [&](int g0) {
#pragma unroll
    for (int i = 0; i < NX; i++) {
      const int c = tid + i * NT, row = c / (8 * KG), k = c % (8 * KG);
      if (XC % NT == 0 || c < XC) {
        const int t = tb + row < M ? tb + row : M - 1;
        const int e = g0 * 32 + k * 4;
        px[i] = *(const float4*)(x + (int64_t)t * I + (e < I ? e : 0));
      }
    }
#pragma unroll
    for (int i = 0; i < NW; i++) {
      const int c = tid + i * NT, row = c / KG, k = c % KG;
      if (WC % NT == 0 || c < WC) {
        const bool up = PAIR && row >= OC;
        const int on = ob + (up ? row - OC : row);
        const int64_t o = on < O ? on : O - 1;
        const int g = g0 + k < ng ? g0 + k : 0;
        pw[i] = *(const u32x4_a8*)((up ? q4b : q4) + o * rb + g * 16);
        ps[i] = (up ? sclb : scl)[o * ng + g];
      }
    }
  };
  auto put = [&](int p) {
#pragma unroll
    for (int i = 0; i < NX; i++) {
      const int c = tid + i * NT, row = c / (8 * KG), k = c % (8 * KG);
      if (XC % NT == 0 || c < XC) *(float4*)(xs[p] + row * XS + ((k ^ (row & 15)) << 4)) = px[i];
    }
#pragma unroll
    for (int i = 0; i < NW; i++) {
      const int c = tid + i * NT, row = c / KG, k = c % KG;
      if (WC % NT == 0 || c < WC) {
        *(u32x4_a8*)(ws[p] + row * WS + k * 16) = pw[i];
        ss[p][row * KG + k] = ps[i];
      }
    }
  };

  v16f neg0;
#pragma unroll
  for (int i = 0; i < 16; i++) neg0[i] = -0.f;
  asm("" : "+v"(neg0));  // keeps it in registers: else rebuilt every step
  float a[TM][TN][NR];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < NR; r++) a[i][j][r] = 0.f;
  float sc[TN][KG];  // this lane's weight rows' scales of the step
  const int nstep = (ng + KG - 1) / KG;

  // KS > 1: this wave's share of the chains over step st's group sums
  auto chain = [&](int st) {
    if (ks >= 4) return;
    const int n = ng - st * KG < KG ? ng - st * KG : KG;
    const float* rp = rs[st & 1] + wt * (KG * TM * TN * 256) + ks * 64 + lane;
#pragma unroll
    for (int k = 0; k < KG; k++)
      if (k < n)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++)
            a[i][j][0] = __fmaf_rn(rp[((k * TM + i) * TN + j) * 256], sc[j][k], a[i][j][0]);
  };

  gload(0);
  put(0);
  if (nstep > 1) gload(KG);
  for (int st = 0; st < nstep; st++) {
    // step st is staged, the group sums of step st - 1 are handed over, and
    // every wave is done with the buffers of step st - 1
    __syncthreads();
    if (KS > 1 && st > 0) chain(st - 1);
    const int p = st & 1;
    if (st + 1 < nstep) {
      put(p ^ 1);
      if (st + 2 < nstep) gload((st + 2) * KG);
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int row = PAIR ? j * OC + wn * 16 + r16 : (wn * TN + j) * 16 + r16;
#pragma unroll
      for (int k = 0; k < KG; k++) sc[j][k] = ss[p][row * KG + k];
    }
#pragma unroll
    for (int gi = 0; gi < KG / KS; gi++) {
      const int g = gi * KS + ks;
      if (st * KG + g >= ng) break;  // wave-uniform
      float4 xl[TM], xh[TM];
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const uint8_t* base = xs[p] + ((wm * TM + i) * 16 + r16) * XS;
        xl[i] = *(const float4*)(base + (((g * 8 + b) ^ r16) << 4));
        xh[i] = *(const float4*)(base + (((g * 8 + 4 + b) ^ r16) << 4));
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int row = PAIR ? j * OC + wn * 16 + r16 : (wn * TN + j) * 16 + r16;
        const uint8_t* base = ws[p] + row * WS + g * 16 + 2 * b;
        const uint32_t n = (uint32_t)*(const uint16_t*)base | ((uint32_t)*(const uint16_t*)(base + 8) << 16);
        // bytes: elements 4b, 4b+2, 16+4b, 16+4b+2 (even) and their odd neighbours, as n - 8
        const uint32_t ev = nib_minus8(n & 0x0f0f0f0fu), od = nib_minus8((n >> 4) & 0x0f0f0f0fu);
        const float wl[4] = {cvt_sb<0>(ev), cvt_sb<0>(od), cvt_sb<1>(ev), cvt_sb<1>(od)};
        const float wh[4] = {cvt_sb<2>(ev), cvt_sb<2>(od), cvt_sb<3>(ev), cvt_sb<3>(od)};
#pragma unroll
        for (int i = 0; i < TM; i++) {
          const float xlo[4] = {xl[i].x, xl[i].y, xl[i].z, xl[i].w}, xhi[4] = {xh[i].x, xh[i].y, xh[i].z, xh[i].w};
          // the eight matrix instructions together, then the adds: left to
          // itself the compiler chains each pair and waits for it (M = 250,
          // I = 4096, O = 12288 gate/up 937 -> 860 us); memory and scalar
          // instructions may cross
          v16f t[4];
          __builtin_amdgcn_sched_barrier(0x4 | 0x10 | 0x80);
#pragma unroll
          for (int q = 0; q < 4; q++) t[q] = __builtin_amdgcn_mfma_f32_16x16x1f32(xhi[q], wh[q], neg0, 0, 0, 0);
#pragma unroll
          for (int q = 0; q < 4; q++) t[q] = __builtin_amdgcn_mfma_f32_16x16x1f32(xlo[q], wl[q], t[q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0x4 | 0x10 | 0x80);
          float v[4][4];
#pragma unroll
          for (int q = 0; q < 4; q++)
#pragma unroll
            for (int r = 0; r < 4; r++) v[q][r] = (t[q][12 + r] + t[q][4 + r]) + (t[q][8 + r] + t[q][r]);
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float s = (v[0][r] + v[2][r]) + (v[1][r] + v[3][r]);
            if constexpr (KS == 1)
              a[i][j][r] = __fmaf_rn(s, sc[j][g], a[i][j][r]);
            else
              rs[p][((wt * KG + g) * TM * TN + i * TN + j) * 256 + r * 64 + lane] = s;
          }
        }
      }
    }
  }
  if constexpr (KS > 1) {
    __syncthreads();
    chain(nstep - 1);
  }
  if (KS > 4 && ks >= 4) return;
  // lane l, register r of a tile: token 4 (l / 16) + r, weight row l % 16
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int t = tb + (wm * TM + i) * 16 + 4 * b + (KS == 1 ? r : ks);
      if (t >= M) continue;
      if constexpr (PAIR) {
        const int o = ob + wn * 16 + r16;
        if (o < O) y[(int64_t)t * O + o] = ref_silu_mul(a[i][0][r], a[i][1][r]);
      } else {
#pragma unroll
        for (int j = 0; j < TN; j++) {
          const int o = ob + (wn * TN + j) * 16 + r16;
          if (o < O) y[(int64_t)t * O + o] = a[i][j][r];
        }
      }
    }
}

// ---------------------------------------------------------------------------
// IDOT4 for a few tokens: tiles of 16 TM tokens x 16 TN WN weight rows whose
// K steps are split over KS waves by group, as the exact-f32 form above.  One
// v_mfma_i32_16x16x32_i8 is a group's integer dots of 16 tokens and 16 rows;
// the waves hand them over as floats through LDS and a wave per register (and
// tile) continues the chains acc = fma(scale, d, acc), y = sx * acc.  A step
// is KG = 8 or 16 groups long: its barrier, LDS and load latencies (0.5-0.7
// us, whatever it holds) and not the weight stream were the time of the
// kernels that take 4 groups a step (M = 6..40, 8B FFN: 97 us for 19 us of
// bytes).  Lane l takes bytes [4 (l / 16), +4) of a row's 16 nibble bytes of
// the group, low nibbles then high, and the same 8 elements of its token, the
// even ones first (a k-permutation shared by both operands).
template <int TM, int TN, int WN, int KS, int KG, bool PAIR>
__global__ __launch_bounds__(64 * WN * KS, 2) void k_gemm_i4g_few(const int8_t* __restrict__ xq,
                                                                  const float* __restrict__ sx,
                                                                  const uint8_t* __restrict__ q4,
                                                                  const float* __restrict__ scl,
                                                                  const uint8_t* __restrict__ q4b,
                                                                  const float* __restrict__ sclb,
                                                                  float* __restrict__ y, int M, int I, int O) {
  static_assert(!PAIR || TN == 2, "PAIR: one gate and one up tile per wave");
  static_assert(KG % KS == 0 && KS == 8, "groups of a step over the K waves");
  constexpr int NT = 64 * WN * KS;
  constexpr int BM = 16 * TM, BW = 16 * TN * WN;  // tokens, weight rows of the tile
  constexpr int OC = PAIR ? BW / 2 : BW;          // output columns
  constexpr int XS = KG * 32 + 16, WS = KG * 16 + 16;  // LDS row strides of codes and nibbles (bytes)
  constexpr int XC = BM * KG * 2, WC = BW * KG;        // a step's 16-byte pieces of x and of the nibbles
  constexpr int NX = (XC + NT - 1) / NT, NW = (WC + NT - 1) / NT;
  constexpr int NTL = TM * TN;                         // tiles of a wave
  constexpr int NC = (NTL * 4 + KS - 1) / KS;          // (tile, register) chains per wave of the tile
  __shared__ __align__(16) int8_t xs[2][BM * XS];
  __shared__ __align__(16) uint8_t ws[2][BW * WS];
  __shared__ float ss[2][KG * BW];  // [group][row]
  __shared__ float rs[2][WN * KG * NTL * 256];
  __shared__ uint64_t s_exp[PAIR ? 32 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int ks = wv % KS, wn = wv / KS;
  const int r16 = lane & 15, b = lane >> 4;
  const int tb = blockIdx.y * BM, ob = blockIdx.x * OC;
  const int ng = I / 32, rb = I / 2, nstep = (ng + KG - 1) / KG;
  if (PAIR) exp_tab_lds(s_exp);

  // staging, two steps ahead: every load unconditional, from clamped piece
  // numbers (the last piece stored more than once, the same bytes), rows past
  // the end re-reading the last and groups past the end a row's first
  struct Set {
    v4i x[NX], w[NW];
    float s[NW];
  };
  Set s0, s1;
  auto piece = [&](int i, int n) { return n % NT == 0 || tid + i * NT < n ? tid + i * NT : n - 1; };
  const int8_t* px[NX];
  const uint8_t* pw[NW];
  const float* ps[NW];
#pragma unroll
  for (int i = 0; i < NX; i++) {
    const int c = piece(i, XC), row = c / (2 * KG), t = tb + row < M ? tb + row : M - 1;
    px[i] = xq + (int64_t)t * I + c % (2 * KG) * 16;
  }
#pragma unroll
  for (int i = 0; i < NW; i++) {
    const int c = piece(i, WC), row = c / KG, k = c % KG;
    const bool up = PAIR && row >= OC;
    const int on = ob + (up ? row - OC : row);
    const int64_t o = on < O ? on : O - 1;
    pw[i] = (up ? q4b : q4) + o * rb + k * 16;
    ps[i] = (up ? sclb : scl) + o * ng + k;
  }
  auto gload = [&](int st, Set& v) {
    const int s = st < nstep ? st : nstep - 1, left = ng - s * KG;  // uniform
#pragma unroll
    for (int i = 0; i < NX; i++) {
      const int k = piece(i, XC) % (2 * KG);
      v.x[i] = *(const v4i*)(px[i] + (k / 2 < left ? s * (KG * 32) : -k * 16));
    }
#pragma unroll
    for (int i = 0; i < NW; i++) {
      const int k = piece(i, WC) % KG;
      v.w[i] = *(const v4i*)(pw[i] + (k < left ? s * (KG * 16) : -k * 16));
      v.s[i] = ps[i][k < left ? s * KG : -k];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto put = [&](int p, const Set& v) {
#pragma unroll
    for (int i = 0; i < NX; i++) {
      const int c = piece(i, XC);
      *(v4i*)(xs[p] + c / (2 * KG) * XS + c % (2 * KG) * 16) = v.x[i];
    }
#pragma unroll
    for (int i = 0; i < NW; i++) {
      const int c = piece(i, WC);
      *(v4i*)(ws[p] + c / KG * WS + c % KG * 16) = v.w[i];
      ss[p][c % KG * BW + c / KG] = v.s[i];
    }
  };

  auto row_of = [&](int j) { return PAIR ? j * OC + wn * 16 + r16 : (wn * TN + j) * 16 + r16; };
  float acc[NC], sc[NC][KG];
#pragma unroll
  for (int c = 0; c < NC; c++) acc[c] = 0.f;
  // chain c of this wave: register and tile of index ks + KS c
  auto chain = [&](int st) {
    const int n = ng - st * KG < KG ? ng - st * KG : KG;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int id = ks + KS * c;
      if (id >= NTL * 4) break;  // wave-uniform
      const float* rp = rs[st & 1] + wn * (KG * NTL * 256) + id * 64 + lane;
      if (n == KG) {
#pragma unroll
        for (int k = 0; k < KG; k++) acc[c] = __fmaf_rn(sc[c][k], rp[k * NTL * 256], acc[c]);
      } else {
#pragma unroll
        for (int k = 0; k < KG; k++)
          if (k < n) acc[c] = __fmaf_rn(sc[c][k], rp[k * NTL * 256], acc[c]);
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
      const int id = ks + KS * c, row = row_of(id / 4 % NTL % TN);
#pragma unroll
      for (int k = 0; k < KG; k++) sc[c][k] = ss[p][k * BW + row];
    }
    // groups past the end are computed on the row's first and never chained
    long fa[KG / KS][TM];
    v4i d[KG / KS][TM][TN];
#pragma unroll
    for (int g = 0; g < KG / KS; g++) {
      const int k = g * KS + ks;
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const uint2 c = *(const uint2*)(xs[p] + (i * 16 + r16) * XS + k * 32 + b * 8);
        fa[g][i] = (long)((uint64_t)__builtin_amdgcn_perm(c.y, c.x, 0x06040200u) |
                          ((uint64_t)__builtin_amdgcn_perm(c.y, c.x, 0x07050301u) << 32));
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const uint32_t w = *(const uint32_t*)(ws[p] + row_of(j) * WS + k * 16 + b * 4);
        const long fb = (long)((uint64_t)nib_minus8(w & 0x0f0f0f0fu) | ((uint64_t)nib_minus8((w >> 4) & 0x0f0f0f0fu) << 32));
#pragma unroll
        for (int i = 0; i < TM; i++)
          d[g][i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(fa[g][i], fb, v4i{0, 0, 0, 0}, 0, 0, 0);
      }
    }
#pragma unroll
    for (int g = 0; g < KG / KS; g++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            rs[p][((wn * KG + g * KS + ks) * NTL + i * TN + j) * 256 + r * 64 + lane] = (float)d[g][i][j][r];
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
  if constexpr (PAIR) {
    // gate and up chains of one output sit in different waves: through LDS
    float* ex = rs[nstep & 1];  // the half the last chain did not read
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int id = ks + KS * c;
      if (id < NTL * 4) ex[(wn * NTL * 4 + id) * 64 + lane] = acc[c];
    }
    __syncthreads();
    for (int q = ks; q < TM * 4; q += KS) {  // (token tile, register)
      const int i = q / 4, r = q % 4, t = tb + i * 16 + 4 * b + r, o = ob + wn * 16 + r16;
      const float s = sx[t < M ? t : M - 1];
      const float g = s * ex[(wn * NTL * 4 + (i * 2) * 4 + r) * 64 + lane];
      const float u = s * ex[(wn * NTL * 4 + (i * 2 + 1) * 4 + r) * 64 + lane];
      const float v = ref_silu_mul(g, u, s_exp);
      if (t < M && o < O) y[(int64_t)t * O + o] = v;
    }
  } else {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int id = ks + KS * c, tl = id / 4, r = id % 4;
      if (id >= NTL * 4) break;
      const int t = tb + tl / TN * 16 + 4 * b + r, o = ob + row_of(tl % TN);
      if (t < M && o < O) y[(int64_t)t * O + o] = sx[t] * acc[c];
    }
  }
}

// The IDOT4 kernels' tiles (tokens, columns) and times: a launch with j tiles on
// the busiest CU (ceil(tiles / 256)) takes a + b * j + g[j] * groups us, past
// eight tiles g[8] * j / 8.  Fitted on MI355X to M = 5..512 over 25 (I, O) pairs
// from 576 x 1536 to 12352 x 4096, weights rotating past the Infinity Cache, to
// 2 to 6 % (root mean square).  Gate + up of 4096 x 12288: few-token kernel 25.7
// us up to 16 tokens (16 groups a step 27.8, two column tiles 33) and 42 up to
// 32, f16-MFMA tiles 42 to 64; 12288 x 4096 16.5 (8 groups 29), 22 (29) and 57.
struct I4Tile {
  int bm, oc;
  double a, b, g[8];
};
static constexpr I4Tile I4_FEW_ONE[] = {{16, 16, 3.80, 0.59, {0.0336, 0.0577, 0.0868, 0.1127, 0.1396, 0.1649, 0.1904, 0.2053}},
                                        {32, 16, 3.04, 1.62, {0.0481, 0.0963, 0.1414, 0.1863, 0.2325, 0.2758, 0.3237, 0.3641}}};
static constexpr I4Tile I4_FEW_PAIR[] = {{16, 16, 3.76, 0.59, {0.0642, 0.1029, 0.1445, 0.1905, 0.2309, 0.2731, 0.3146, 0.3380}},
                                         {32, 16, 2.60, 1.83, {0.0895, 0.1737, 0.2592, 0.3435, 0.4265, 0.5089, 0.5972, 0.6635}}};
static constexpr I4Tile I4_INT8 = {64, 64, 2.79, 2.00, {0.1816, 0.2434, 0.3393, 0.4399, 0.4933, 0.5706, 0.6657, 0.7608}};
static constexpr I4Tile I4_H_ONE = {64, 64, 2.90, 2.71, {0.1335, 0.2746, 0.4106, 0.5474, 0.6843, 0.8212, 0.9580, 1.0949}};
static constexpr I4Tile I4_H_ONE_BIG = {128, 128, 4.03, 4.08, {0.3722, 0.7232, 1.0848, 1.4465, 1.8081, 2.1697, 2.5313, 2.8929}};
static constexpr I4Tile I4_H_PAIR = {64, 64, 6.80, 1.85, {0.2382, 0.3787, 0.6003, 0.8004, 1.0005, 1.2006, 1.4007, 1.6008}};
static constexpr I4Tile I4_H_PAIR_BIG = {128, 128, 6.87, 9.34, {0.5647, 1.0630, 1.5946, 2.1261, 2.6576, 3.1891, 3.7206, 4.2521}};
static constexpr I4Tile I4_H_PAIR_192 = {64, 192, 3.69, 10.11, {0.5399, 1.0007, 1.5011, 2.0014, 2.5018, 3.0022, 3.5025, 4.0029}};

static double i4_us(const I4Tile& t, int M, int I, int O) {
  const int64_t j = ((int64_t)((M + t.bm - 1) / t.bm) * ((O + t.oc - 1) / t.oc) + 255) / 256;
  return t.a + t.b * j + (I / 32) * (j <= 8 ? t.g[j - 1] : t.g[7] * j / 8);
}

static double few_us(int M, int I, int O, bool pair, bool* two) {
  const I4Tile* t = pair ? I4_FEW_PAIR : I4_FEW_ONE;
  const double t1 = i4_us(t[0], M, I, O), t2 = i4_us(t[1], M, I, O);
  *two = t2 < t1;
  return *two ? t2 : t1;
}

// against the f16-MFMA tiles or, for other row lengths, the int8-MFMA GEMM (one
// each for gate and up, and silu_mul)
bool i4g_few_wins(int M, int I, int O, bool pair, bool f16) {
  if (M > 512) return false;
  bool two;
  const double few = few_us(M, I, O, pair, &two);
  if (!f16) return few < (pair ? 2 * i4_us(I4_INT8, M, I, O) + 4 : i4_us(I4_INT8, M, I, O));
  const bool big = gemm_i4g_h_big(M, O);
  const I4Tile& h = !pair ? (big ? I4_H_ONE_BIG : I4_H_ONE)
                          : gemm_i4g_h_pair192(M, O) ? I4_H_PAIR_192 : big ? I4_H_PAIR_BIG : I4_H_PAIR;
  return few < i4_us(h, M, I, O);
}

int launch_gemm_i4g_few(const int8_t* xq, const float* sx, const uint8_t* q4, const float* scl, const uint8_t* q4b,
                        const float* sclb, float* y, int M, int I, int O, hipStream_t st) {
  if (I % 32) return MOTY_EUNSUP;
  if (M <= 0 || O <= 0) return MOTY_OK;
  bool two;
  few_us(M, I, O, q4b != nullptr, &two);
  const dim3 grid((O + 15) / 16, (M + (two ? 31 : 15)) / (two ? 32 : 16)), blk(512);
#define FEW(TM, TN, KG, P) \
  hipLaunchKernelGGL((k_gemm_i4g_few<TM, TN, 1, 8, KG, P>), grid, blk, 0, st, xq, sx, q4, scl, q4b, sclb, y, M, I, O)
  if (q4b) {
    if (two) FEW(2, 2, 8, true);
    else FEW(1, 2, 8, true);
  } else {
    if (two) FEW(2, 1, 16, false);
    else FEW(1, 1, 16, false);
  }
#undef FEW
  LAUNCH_TRY("k_gemm_i4g_few");
  return MOTY_OK;
}

// The tile shapes, by the time one workgroup takes alone on a CU per 4096
// elements of I (measured on MI355X over M = 1..500 and six (I, O) pairs;
// workgroups on one CU share its SIMDs, so a launch takes about
// ceil(workgroups / 256) of these).  Small tiles with the K steps split over
// waves fill the chip when there are few, large ones cost less per output:
//   gate + up, tokens x columns: 16 x 32 47 us, 16 x 64 78, 64 x 64 250
//   one matrix:  16 x 32 25 us, 16 x 64 43, 32 x 64 71, 64 x 64 128
// (a SIMD spends 584 clocks per 16 x 16 tile and group in the 64 x 64 ones,
// 256 of them MFMA: at 24576 x 4096, 256 tokens the counters show the matrix
// cores busy 44 % of the kernel's time and the vector pipes 65 %).
struct XfTile {
  int bm, oc;
  double us;
};
static constexpr XfTile XF_PAIR[] = {{16, 32, 47}, {16, 64, 78}, {64, 64, 250}};
static constexpr XfTile XF_ONE[] = {{16, 32, 25}, {16, 64, 43}, {32, 64, 71}, {64, 64, 128}};

static int xf_pick(int M, int I, int O, bool pair, double* us) {
  const XfTile* t = pair ? XF_PAIR : XF_ONE;
  const int n = pair ? 3 : 4;
  int best = 0;
  double bt = 0;
  for (int k = 0; k < n; k++) {
    const int64_t wgs = (int64_t)((M + t[k].bm - 1) / t[k].bm) * ((O + t[k].oc - 1) / t[k].oc);
    const double us_k = (double)((wgs + 255) / 256) * t[k].us * I / 4096;
    if (k == 0 || us_k < bt) best = k, bt = us_k;
  }
  *us = bt;
  return best;
}

// S tokens: the one-token GEMV once per token, its row's latency or, from the
// second token out of the Infinity Cache, the matrix bytes at 5.6 TB/s each
// (1024 x 3072 gate + up 4.4 us a token, 4096 x 12288 13.4, 14336 x 4096 11.5),
// or the GEMM above?  Measured at 2 to 10 tokens over 23 shapes: the GEMM wins
// from 2 to 4 tokens at the smaller shapes, at the larger ones from 6 (gate + up
// of 4096 x 12288, 5 / 6 tokens: 71 / 85 us against 84) or 8.
bool xf_gemv_per_token(int S, int I, int O, bool pair) {
  if (S <= 1) return true;
  if (S > 64) return false;
  double gemm_us;
  xf_pick(S, I, O, pair, &gemm_us);
  const double row_us = 3.8 + 0.54e-3 * I, bytes_us = 3.9 + 0.178e-6 * ((double)O * I * (pair ? 1.25 : 0.625));
  return S * (row_us > bytes_us ? row_us : bytes_us) < gemm_us + 1.6;
}

// I % 32 == 0, 16-byte aligned x and 8-byte aligned nibbles; PAIR (q4b):
// y = silu(gate) * up
int launch_gemm_i4g_xf(const float* x, const uint8_t* q4, const float* scl, const uint8_t* q4b, const float* sclb,
                       float* y, int M, int I, int O, hipStream_t st) {
  if ((I % 32) || (((uintptr_t)x) & 15) || ((((uintptr_t)q4) | ((uintptr_t)q4b)) & 7)) return MOTY_EUNSUP;
  if (M <= 0 || O <= 0) return MOTY_OK;
  double us;
  const int k = xf_pick(M, I, O, q4b != nullptr, &us);
  const XfTile t = q4b ? XF_PAIR[k] : XF_ONE[k];
  const dim3 grid((O + t.oc - 1) / t.oc, (M + t.bm - 1) / t.bm);
#define XF(TM, TN, WM, WN, KS, KG, P)                                                                          \
  hipLaunchKernelGGL((k_gemm_i4g_xf<TM, TN, WM, WN, KS, KG, P>), grid, dim3(64 * WM * WN * KS), 0, st, x, q4, \
                     scl, q4b, sclb, y, M, I, O)
  if (q4b) {
    if (k == 0) XF(1, 2, 1, 2, 4, 4, true);
    else if (k == 1) XF(1, 2, 1, 4, 4, 4, true);
    else XF(1, 2, 4, 4, 1, 2, true);
  } else {
    if (k == 0) XF(1, 1, 1, 2, 8, 8, false);
    else if (k == 1) XF(1, 1, 1, 4, 4, 4, false);
    else if (k == 2) XF(2, 1, 1, 4, 4, 4, false);
    else XF(1, 1, 4, 4, 1, 2, false);
  }
#undef XF
  LAUNCH_TRY("k_gemm_i4g_xf");
  return MOTY_OK;
}

int launch_i4g_f32(const float* x, const uint8_t* q4, const float* scl, float* y, int S, int I, int O,
                   hipStream_t st) {
  if (I % 32) return MOTY_EUNSUP;
  if (S <= 0 || O <= 0) return MOTY_OK;
  dim3 grid((O + Q4F_NT - 1) / Q4F_NT, S);
  hipLaunchKernelGGL(k_i4g_f32, grid, dim3(Q4F_NT), 0, st, x, q4, scl, y, S, I, O);
  LAUNCH_TRY("k_i4g_f32");
  return MOTY_OK;
}

}  // namespace moty
