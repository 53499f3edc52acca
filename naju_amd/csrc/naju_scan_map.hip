// naju_scan_map.hip -- time-segment maps of the chunked scan (9 <= N <= 128,
// above 64 in two launches over halves of the entries).
//
// When T is split into segments, the state (adjoint carry) entering a segment
// comes from composing the maps of the segments before (after) it, s -> F s + Z
// per channel, with (reference naju/chunk_affine_triton.py:3-5)
//   forward:  F = prod_t f_t,  Z[n] = sum_t (prod_{k>t} f_k) w_t B_t[n]
//   backward: F = prod_t f_t,  Z[n] = sum_t (prod_{k<=t} f_k) dy_t C_t[n]
// over the segment's rows. Nothing but the segment's end is needed here, so the
// sum is formed as one matrix product over all of its rows, Z = B^T (c w) with
// c_t the decay from row t to the segment's end: walking the rows from that end
// keeps c as a running product per channel, and the accumulator is never
// rescaled. (The scan kernels step the state over 16-row sub-blocks instead,
// X <- Pall X + B^T (Pe w), with the gates passed through LDS, because they need
// the state in between.)
//
// Layout. A wave owns 16 V channels and a run of rows, in blocks of 32. Lane
// (j, g) = (l % 16, l / 16) loads rows 8g .. 8g+7 of channels V j .. V j + V - 1:
// whole 128-byte lines per row, and at the same time the B operand of one
// K = 32 product per channel tile c (column j = channel V j + c), so the gates
// never leave the lane's registers. The decays of a lane's 8 rows are a
// product chain, those of the four lane groups two lane swaps. B (or C) of the
// block goes through the wave's own LDS as [n][row], whose 8 rows per lane are
// the A operand in two 8-byte reads (bf16; 16-byte ones for float32). There is no barrier in the walk;
// the W waves of a workgroup take consecutive runs of a segment's rows and add
// their maps in wave order at the end.
//
// What bounds it: reading the streams in 64- and 128-byte pieces of rows (a
// timing copy with no products and no sigmoids takes 51 of the 54 us below).
// Measured against stepping the state over 16-row sub-blocks as the scan does
// (N = 64, kernel time, forward / backward maps): bf16 8 x 4096 x 1024 82 / 69
// -> 54 / 47 us; bf16 8 x 8192 x 512 forward 81 -> 57 us; the LM layer
// (8 x 2048 x 1536, float32 gates) 65 / 54 -> 47 / 43 us; float32
// 8 x 2048 x 512 39 / 30 -> 39 / 26 us. Two blocks of loads in flight per wave,
// or twice the waves, change it by less than 3%.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mc_ops.h"
#include "naju_scan.h"
#include "scan_internal.h"

namespace naju_detail {
namespace {

constexpr int kMapMaxW = 4;
constexpr int KB = 32;  // rows per block

// V consecutive elements as loaded (2 to 16 bytes, 32 as two loads).
template <typename TT, int V>
struct RawV {
  static constexpr int NW = V * (int)sizeof(TT) < 4 ? 1 : V * (int)sizeof(TT) / 4;
  uint32_t w[NW];
  __device__ __forceinline__ float get(int e) const {
    if constexpr (sizeof(TT) == 4) {
      return __builtin_bit_cast(float, w[e]);
    } else {
      const uint16_t h = (uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu));
      return to_f32(__builtin_bit_cast(TT, h));
    }
  }
  __device__ __forceinline__ void fill(float x) {
    const TT v = (TT)x;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      if constexpr (sizeof(TT) == 4)
        w[k] = __builtin_bit_cast(uint32_t, v);
      else
        w[k] = (uint32_t)__builtin_bit_cast(uint16_t, v) * 0x10001u;
    }
  }
  __device__ __forceinline__ void load(const void* base, uint32_t byte_off) {
    typedef typename UserVec<uint32_t, NW, sizeof(TT)>::type vw;
    if constexpr (V * sizeof(TT) == 2) {
      w[0] = *(const uint16_t*)((const char*)base + byte_off);
    } else {
      const vw v = *(const vw*)((const char*)base + byte_off);
#pragma unroll
      for (int k = 0; k < NW; ++k) w[k] = v[k];
    }
  }
};

// Whether the A operand goes through LDS as bf16 (exact) or as float32.
template <typename TB>
constexpr bool kMap16 = __is_same(TB, bf16_t);
// LDS row pitch of the [n][row] tile in elements: 88 bytes for bf16 (so rows
// are 8-byte aligned), 144 for float32.
template <typename TB>
constexpr int kMapPitch = kMap16<TB> ? 44 : 36;
// Bytes of a wave's LDS: the tile, or its part of the final sum.
template <int NP, int V, typename TB>
constexpr int kMapLds = NP * kMapPitch<TB> * (kMap16<TB> ? 2 : 4) > NP / 16 * V * 1024
                            ? NP * kMapPitch<TB> * (kMap16<TB> ? 2 : 4)
                            : NP / 16 * V * 1024;

template <int NP, int V, bool BWD, typename TU, typename TG, typename TB>
__global__ __launch_bounds__(64 * kMapMaxW) __attribute__((amdgpu_waves_per_eu(3))) void mc_map_kernel(const ScanArgs a, int wave_rows, int n_ctiles) {
  constexpr int MT = NP / 16;
  constexpr int PT = kMapPitch<TB>;
  extern __shared__ __align__(16) char lds[];
  const int W = (int)(blockDim.x >> 6);
  const int lane = (int)(threadIdx.x & 63);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  char* my = lds + wv * kMapLds<NP, V, TB>;
  float* s_F = (float*)(lds + W * kMapLds<NP, V, TB>);  // [W][16 V]

  const int N = a.N;
  const int64_t T = a.T, D = a.D;
  const int per = n_ctiles * a.batch;
  const uint32_t id = xcd_item();
  const int seg = (int)(id / (uint32_t)per) + (BWD ? 1 : 0);
  const int rem = (int)(id % (uint32_t)per);
  const int b = rem / n_ctiles;
  const int64_t dw = (int64_t)(rem - b * n_ctiles) * (16 * V);
  const int64_t r0 = (int64_t)seg * a.seg_sc * kMcQ;
  const int64_t r1 = r0 + (int64_t)a.seg_sc * kMcQ < T ? r0 + (int64_t)a.seg_sc * kMcQ : T;
  const int64_t w0 = r0 + (int64_t)wv * wave_rows;
  const int64_t w1 = w0 + wave_rows < r1 ? w0 + wave_rows : r1;
  const int nblk = w1 > w0 ? (int)((w1 - w0 + KB - 1) / KB) : 0;
  // the lane's channels V j .. V j + V - 1 of the tile: all inside [0, D) or
  // all past it (D % V == 0), where the loads are clamped in bounds
  const bool cok = dw + V * j < D;
  const uint32_t cb = (uint32_t)(cok ? dw + V * j : D - V);

  // B (or C): lane < NP takes rows ra .. ra + 3, entries nb .. nb + 7 of the
  // block, when they can be loaded whole
  constexpr int NG = NP / 8;
  const int ra = 4 * (lane / NG), nb = 8 * (lane % NG);
  const bool bvec = N == NP && a.ldbc % 8 == 0;
  const TB* const bp = (const TB*)(BWD ? a.Cm : a.Bm) + (int64_t)b * T * a.ldbc;

  // a block's inputs as loaded
  struct Blk {
    RawV<TG, V> f[8], i[BWD ? 1 : 8];
    RawV<TU, V> u[8];  // u, or dy
    RawV<TB, 8> b[4];
  } blk;
  auto load = [&](Blk& x, int k) {
    const int64_t t = w0 + (int64_t)(BWD ? k : nblk - 1 - k) * KB;
    const uint32_t last = (uint32_t)(T - 1 - t < KB ? T - 1 - t : KB);  // rows stay inside T
    const int64_t base = ((int64_t)b * T + t) * D;
    const uint32_t lo = (uint32_t)(8 * g * D) + cb, hi = last * (uint32_t)D + cb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t o = min(lo + (uint32_t)(e * D), hi);
      x.f[e].load((const TG*)a.fl + base, o * (uint32_t)sizeof(TG));
      if constexpr (!BWD) x.i[e].load((const TG*)a.il + base, o * (uint32_t)sizeof(TG));
      x.u[e].load((const TU*)(BWD ? a.dy : a.u) + base, o * (uint32_t)sizeof(TU));
    }
    if (bvec && lane < NP) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        x.b[q].load(bp + t * a.ldbc,
                    (min((uint32_t)(ra + q), last) * (uint32_t)a.ldbc + nb) * (uint32_t)sizeof(TB));
    }
  };

  f4_t acc[MT][V];
  float R[V];
#pragma unroll
  for (int c = 0; c < V; ++c) {
    R[c] = 1.f;
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][c] = f4_t{0.f, 0.f, 0.f, 0.f};
  }
  auto work = [&](Blk& x, int k) {
    const int64_t t = w0 + (int64_t)(BWD ? k : nblk - 1 - k) * KB;
    const int left = (int)(w1 - t < KB ? w1 - t : KB);  // rows of this block
    if (left < KB) {
      // rows past the run: the neutral step f = 1, u (dy) = 0
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (8 * g + e >= left) {
          x.f[e].fill(__builtin_inff());
          if constexpr (!BWD) x.i[e].fill(0.f);
          x.u[e].fill(0.f);
        }
    }
    // ---- B (C) into the wave's tile as [n][row]; rows past the run (a
    // duplicated row could hold a value that is not finite) and entries past
    // N are zero
    if (bvec && lane < NP) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (kMap16<TB>) {
          const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
          uint32_t p0 = __builtin_amdgcn_perm(x.b[1].w[e >> 1], x.b[0].w[e >> 1], sel);
          uint32_t p1 = __builtin_amdgcn_perm(x.b[3].w[e >> 1], x.b[2].w[e >> 1], sel);
          if (left < KB) {
            if (ra + 1 >= left) p0 &= ra < left ? 0xffffu : 0u;
            if (ra + 3 >= left) p1 &= ra + 2 < left ? 0xffffu : 0u;
          }
          *(uint2*)(my + ((nb + e) * PT + ra) * 2) = make_uint2(p0, p1);
        } else {
          float v[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = ra + q < left ? x.b[q].get(e) : 0.f;
          *(float4*)(my + ((nb + e) * PT + ra) * 4) = make_float4(v[0], v[1], v[2], v[3]);
        }
      }
    } else if (!bvec) {
      using TL = std::conditional_t<kMap16<TB>, TB, float>;
#pragma unroll 2
      for (int i = lane; i < NP * KB; i += 64) {
        const int row = i / NP, n = i % NP;
        const bool ok = row < left && n < N;
        const TB v = bp[t * a.ldbc + (ok ? row * a.ldbc + n : 0)];
        ((TL*)my)[n * PT + row] = ok ? (TL)v : (TL)0.f;
      }
    }
    // ---- the lane's coefficients c_t w_t (c_t dy_t) of 8 rows and V channels
    float wp[V][8];
#pragma unroll
    for (int c = 0; c < V; ++c) {
      float f[8], s[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        f[e] = sigm(x.f[e].get(c));
        wp[c][e] = x.u[e].get(c);
        if constexpr (!BWD) wp[c][e] *= sigm(x.i[e].get(c));
      }
      float tot;
      if constexpr (BWD) {
        s[0] = f[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) s[e] = s[e - 1] * f[e];
        tot = s[7];
      } else {
        s[7] = 1.f;
#pragma unroll
        for (int e = 6; e >= 0; --e) s[e] = s[e + 1] * f[e + 1];
        tot = s[0] * f[0];
      }
      // products of the lane groups: pairs (0, 1), (2, 3), then all four
      const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(tot), __float_as_uint(tot), false, false);
      const float pe = __uint_as_float(p[0]), po = __uint_as_float(p[1]);
      const float pr = pe * po;
      const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(pr), __float_as_uint(pr), false, false);
      const float ql = __uint_as_float(q[0]), qh = __uint_as_float(q[1]);
      const float s1 = BWD ? ((g & 1) ? pe : 1.f) : ((g & 1) ? 1.f : po);
      const float s2 = BWD ? ((g & 2) ? ql : 1.f) : ((g & 2) ? 1.f : qh);
      const float cf = R[c] * (s1 * s2);
#pragma unroll
      for (int e = 0; e < 8; ++e) wp[c][e] *= cf * s[e];
      R[c] *= ql * qh;
      // as rounded here: the split below must not be fused with the product
#pragma unroll
      for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(wp[c][e]));
    }
    asm volatile("" ::: "memory");
    // the next block's loads take the registers that this block's are done with
    if (k + 1 < nblk) load(x, k + 1);
    // ---- Z += B^T (c w)
    if constexpr (kMap16<TB>) {
      typedef __bf16 v8 __attribute__((ext_vector_type(8)));
      typedef uint32_t u4 __attribute__((ext_vector_type(4)));
      v8 bt[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const uint2 q0 = *(const uint2*)(my + ((16 * m + j) * PT + 8 * g) * 2);
        const uint2 q1 = *(const uint2*)(my + ((16 * m + j) * PT + 8 * g + 4) * 2);
        bt[m] = __builtin_bit_cast(v8, (u4{q0.x, q0.y, q1.x, q1.y}));
      }
#pragma unroll
      for (int c = 0; c < V; ++c) {
        uint32_t h0[2], m0[2], l0[2], h1[2], m1[2], l1[2];
        split4_bf16({wp[c][0], wp[c][1], wp[c][2], wp[c][3]}, h0, m0, l0);
        split4_bf16({wp[c][4], wp[c][5], wp[c][6], wp[c][7]}, h1, m1, l1);
        const v8 hi = __builtin_bit_cast(v8, (u4{h0[0], h0[1], h1[0], h1[1]}));
        const v8 md = __builtin_bit_cast(v8, (u4{m0[0], m0[1], m1[0], m1[1]}));
        const v8 lo = __builtin_bit_cast(v8, (u4{l0[0], l0[1], l1[0], l1[1]}));
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt[m], hi, acc[m][c], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt[m], md, acc[m][c], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt[m], lo, acc[m][c], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        float bt[8];
        const float4 b0 = *(const float4*)(my + ((16 * m + j) * PT + 8 * g) * 4);
        const float4 b1 = *(const float4*)(my + ((16 * m + j) * PT + 8 * g + 4) * 4);
        bt[0] = b0.x, bt[1] = b0.y, bt[2] = b0.z, bt[3] = b0.w;
        bt[4] = b1.x, bt[5] = b1.y, bt[6] = b1.z, bt[7] = b1.w;
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int c = 0; c < V; ++c) acc[m][c] = mma(bt[e], wp[c][e], acc[m][c]);
      }
    }
    asm volatile("" ::: "memory");
  };
  if (nblk > 0) load(blk, 0);
  for (int k = 0; k < nblk; ++k) work(blk, k);

  // ---- the segment's map from its waves': F = prod F_w, Z = sum_w S_w Z_w
  // with S_w the decay from wave w's rows to the segment's end (start)
  if (g == 0)
#pragma unroll
    for (int c = 0; c < V; ++c) s_F[wv * 16 * V + V * j + c] = R[c];
  __syncthreads();
  float S[V], F[V];
#pragma unroll
  for (int c = 0; c < V; ++c) {
    S[c] = 1.f, F[c] = 1.f;
    for (int w = 0; w < W; ++w) {
      const float f = s_F[w * 16 * V + V * j + c];
      F[c] *= f;
      if (BWD ? w < wv : w > wv) S[c] *= f;
    }
  }
  const int64_t o = ((int64_t)b * a.nseg + seg) * D + dw + V * j;
  if (wv == 0 && g == 0 && cok)
#pragma unroll
    for (int c = 0; c < V; ++c) a.segF[o + c] = F[c];
  if (W > 1) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int c = 0; c < V; ++c) *(f4_t*)(my + ((m * V + c) * 64 + lane) * 16) = acc[m][c] * S[c];
    __syncthreads();
  }
  // wave w adds and stores the tiles m = w, w + W, ..
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m % W != wv) continue;
    f4_t z[V];
#pragma unroll
    for (int c = 0; c < V; ++c) {
      z[c] = acc[m][c];
      if (W > 1) {
        const char* p = lds + ((m * V + c) * 64 + lane) * 16;
        z[c] = *(const f4_t*)p;
        for (int w = 1; w < W; ++w) z[c] += *(const f4_t*)(p + w * kMapLds<NP, V, TB>);
      }
    }
    if (!cok) continue;
    const int n = 16 * m + 4 * g;
#pragma unroll
    for (int c = 0; c < V; ++c) {
      float* p = a.segZ + (o + c) * a.ldn + n;
      if (((N | a.ldn) & 3) == 0) {
        if (n < N) *(f4_t*)p = z[c];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) p[r] = z[c][r];
      }
    }
  }
}

typedef void (*mc_map_t)(ScanArgs, int, int);

struct MapPick {
  mc_map_t k;
  int V, lds;  // channels per lane, LDS bytes per wave
};

// V channels per lane, 1 where D does not divide
template <bool BWD, typename TU, typename TG, typename TB, int NP>
MapPick map_np(int64_t D) {
  constexpr int V = 2;
  if (D % V) return {mc_map_kernel<NP, 1, BWD, TU, TG, TB>, 1, kMapLds<NP, 1, TB>};
  return {mc_map_kernel<NP, V, BWD, TU, TG, TB>, V, kMapLds<NP, V, TB>};
}
template <bool BWD, typename TU, typename TG, typename TB>
MapPick map_n(int64_t N, int64_t D) {
  return N <= 16   ? map_np<BWD, TU, TG, TB, 16>(D)
         : N <= 32 ? map_np<BWD, TU, TG, TB, 32>(D)
                   : map_np<BWD, TU, TG, TB, 64>(D);
}
template <bool BWD, typename TU>
MapPick map_u(int g_dt, int bc_dt, int64_t N, int64_t D) {
  const bool gf = g_dt == NAJU_DTYPE_F32, bf = bc_dt == NAJU_DTYPE_F32;
  if (gf) return bf ? map_n<BWD, TU, float, float>(N, D) : map_n<BWD, TU, float, TU>(N, D);
  return bf ? map_n<BWD, TU, TU, float>(N, D) : map_n<BWD, TU, TU, TU>(N, D);
}
template <bool BWD>
MapPick map_pick(int x_dt, int g_dt, int bc_dt, int64_t N, int64_t D) {
  return x_dt == NAJU_DTYPE_F32    ? map_n<BWD, float, float, float>(N, D)
         : x_dt == NAJU_DTYPE_BF16 ? map_u<BWD, bf16_t>(g_dt, bc_dt, N, D)
                                   : map_u<BWD, f16_t>(g_dt, bc_dt, N, D);
}

}  // namespace

// As many as leave each four blocks of rows. More waves hide more latency
// (bf16, 8 x 4096 x 1024, N = 64, 512-row segments: 1 / 2 / 4 waves took 62 / 57
// / 55 us), but their maps are added at the end (float32, 8 x 2048 x 512, 128
// rows, backward: 1 / 2 waves 26 / 31 us).
int mc_map_waves(int rows) {
  int W = 1;
  while (W < kMapMaxW && rows >= 2 * W * 4 * KB) W *= 2;
  return W;
}

hipError_t mc_map_launch(const ScanArgs& a, bool bwd, int x_dt, int g_dt, hipStream_t st) {
  if (a.nseg <= 1) return hipSuccess;
  const MapPick p = bwd ? map_pick<true>(x_dt, g_dt, a.bc_dt, a.N, a.D)
                        : map_pick<false>(x_dt, g_dt, a.bc_dt, a.N, a.D);
  const int64_t n_ctiles = (a.D + 16 * p.V - 1) / (16 * p.V);
  const int64_t wgs = n_ctiles * a.batch * (a.nseg - 1);
  if (wgs > 0x7fffffff) return hipErrorInvalidValue;
  const int rows = a.seg_sc * kMcQ;
  const int W = mc_map_waves(rows);
  const int wave_rows = (rows + W * KB - 1) / (W * KB) * KB;
  hipLaunchKernelGGL(p.k, dim3((unsigned)wgs), dim3(64 * W), (size_t)W * (p.lds + 16 * p.V * 4), st, a, wave_rows,
                     (int)n_ctiles);
  return hipGetLastError();
}

}  // namespace naju_detail
