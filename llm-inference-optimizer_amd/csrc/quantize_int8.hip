// The int8 weight quantiser of QuantizedLinearInt8.from_linear
// (src/quantization/int8.py:45-50) for gfx950, plus its launcher.  Per weight
// row:
//   amax = max_k |w|,  scale = max(amax / 127, 1e-8),
//   q = clamp(rint(w / scale), -127, 127)   (IEEE fp32 division, ties to even)
// bit-identical to the reference's torch expression.
//
// Bound by HBM: each weight is read once and each code written once (3 bytes
// per 16-bit weight), so the row stays in registers between the two passes
// and both passes keep to a few VALU operations per element:
//   amax      on the packed bits: the magnitudes of 16-bit (32-bit) floats
//             order like their bit patterns, so one AND and one packed u16 max
//             cover two elements.  A NaN's pattern lies above infinity's, so
//             the same max finds rows that hold either; they take the plain
//             formula (amax with fmaxf, which skips NaN; division; clamp).
//   codes     t = fma(w, 1 / scale, 1.5 * 2^23) rounds w / scale to an integer
//             in t's low bits.  1 / scale is correctly rounded, so the
//             product is within 127 * 2^-24 of the quotient, as is the
//             reference's own rounded quotient: the integers agree unless the
//             product lies within 2^-15 of a half-integer.  A packet with a
//             lane nearer than 2^-14 (a few percent of them) is redone with
//             the division.  No clamp: |w| <= amax keeps |w / scale| <= 127
//             (1 + 2^-23), below 127.5.
// One wave per row up to 8 packets a lane (k 4096 in 16 bits); wider rows are
// spread over up to 16 waves that exchange their maxima through LDS.
// Measured on MI355X, [18944, 3584] bf16 (204 MB): 37.5 us, 5.4 TB/s; the
// kernel before (one wave per row, 2-byte loads, the row read twice, a
// division per weight) 124.8 us.
#include "common.h"
#include "quantize_plan.h"

namespace mi355 {
namespace {

constexpr float kRound = 12582912.0f;              // 1.5 * 2^23
constexpr float kSafe = 0.5f - 1.0f / 16384.0f;    // nearest-integer distance that settles the rounding

template <int CTRL> __device__ __forceinline__ uint32_t dpp_max(uint32_t v) {
  const uint32_t o = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, false));
  return v > o ? v : o;
}

// Largest v of the wave, in every lane (the pairing of wave_allreduce_sum).
__device__ __forceinline__ uint32_t wave_allreduce_max(uint32_t v) {
  v = dpp_max<0xb1>(v);
  v = dpp_max<0x4e>(v);
  v = dpp_max<0x141>(v);
  v = dpp_max<0x140>(v);
  {
    auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    const uint32_t lo = r[0], hi = r[1];
    v = lo > hi ? lo : hi;
  }
  {
    auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const uint32_t lo = r[0], hi = r[1];
    v = lo > hi ? lo : hi;
  }
  return v;
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Magnitude bits: two per dword for 16-bit types, one for fp32.
template <typename TW> __device__ __forceinline__ uint32_t mag_max(uint32_t acc, uint32_t d) {
  if constexpr (is_half_width<TW>::value) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, acc),
                                                                  __builtin_bit_cast(u16x2, d & 0x7fff7fffu)));
  } else {
    const uint32_t m = d & 0x7fffffffu;
    return acc > m ? acc : m;
  }
}
// The lane's largest magnitude as fp32 bits (NaN and infinity stay at or
// above infinity's pattern, and in order).
template <typename TW> __device__ __forceinline__ uint32_t mag_f32(uint32_t acc) {
  if constexpr (is_half_width<TW>::value) {
    const uint32_t lo = acc & 0xffffu, hi = acc >> 16;
    const uint32_t m = lo > hi ? lo : hi;
    return as_u32(load_elem<TW>(&m, 0)) & 0x7fffffffu;
  } else {
    return acc;
  }
}

// The reference's expression, operation by operation.
__device__ __forceinline__ int code_exact(float w, float sc) {
  float v = __builtin_rintf(w / sc);
  v = __builtin_fminf(__builtin_fmaxf(v, -127.0f), 127.0f);
  return static_cast<int>(v);
}

__device__ __forceinline__ float row_scale(float amax) {
  float sc = amax / 127.0f;  // IEEE division (HIP's default for fp32 '/')
  return sc < 1e-8f ? 1e-8f : sc;
}

// VPL packets per lane; BLOCK: the workgroup's waves share one row, else one
// row per wave.
template <typename TW, int VPL, bool BLOCK>
__global__ __launch_bounds__(BLOCK ? 1024 : 256) void quantize_int8_rows(const void* __restrict__ w,
                                                                         int8_t* __restrict__ q,
                                                                         float* __restrict__ scale, int64_t n, int k,
                                                                         int64_t ws, int64_t qs) {
  constexpr int W = pack_width<TW>::value;
  using TB = typename TW::bits;
  __shared__ uint32_t wave_max[16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r = BLOCK ? static_cast<int64_t>(blockIdx.x) : static_cast<int64_t>(blockIdx.x) * 4 + wave;
  if (r >= n) return;
  const int slot = BLOCK ? threadIdx.x : (threadIdx.x & 63), stride = BLOCK ? blockDim.x : 64;
  const rsrc_t rw = make_rsrc(static_cast<const TB*>(w) + r * ws, static_cast<uint32_t>(k) * sizeof(TB));
  const rsrc_t rq = make_rsrc(q + r * qs, static_cast<uint32_t>(k));

  Packet<TW> x[VPL];  // packets past k read 0
#pragma unroll
  for (int j = 0; j < VPL; ++j) x[j].raw = buf_load16(rw, static_cast<uint32_t>(slot + j * stride) * 16u);
  uint32_t acc = 0;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = mag_max<TW>(acc, x[j].raw[i]);
  }
  uint32_t top = wave_allreduce_max(mag_f32<TW>(acc));
  if constexpr (BLOCK) {
    if ((threadIdx.x & 63) == 0) wave_max[wave] = top;
    __syncthreads();
    for (int i = 0; i < static_cast<int>(blockDim.x >> 6); ++i) top = top > wave_max[i] ? top : wave_max[i];
  }
  const bool special = top >= 0x7f800000u;  // the row holds a NaN or an infinity
  float amax = as_f32(top);
  if (special) {  // amax over the values that are no NaN
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      float f[W];
      x[j].unpack(f);
#pragma unroll
      for (int e = 0; e < W; ++e) m = __builtin_fmaxf(m, __builtin_fabsf(f[e]));
    }
    top = wave_allreduce_max(as_u32(m));
    if constexpr (BLOCK) {
      __syncthreads();  // every wave of the row is here: `special` is the same in all
      if ((threadIdx.x & 63) == 0) wave_max[wave] = top;
      __syncthreads();
      for (int i = 0; i < static_cast<int>(blockDim.x >> 6); ++i) top = top > wave_max[i] ? top : wave_max[i];
    }
    amax = as_f32(top);
  }
  const float sc = row_scale(amax);
  if (slot == 0) scale[r] = sc;
  const float rc = 1.0f / sc;

#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    float f[W], t[W], worst = 0.f;
    x[j].unpack(f);
#pragma unroll
    for (int e = 0; e < W; ++e) {
      t[e] = __builtin_fmaf(f[e], rc, kRound);
      const float d = __builtin_fmaf(f[e], rc, kRound - t[e]);
      worst = __builtin_fmaxf(worst, __builtin_fabsf(d));
    }
    uint32_t code[W / 4];
#pragma unroll
    for (int i = 0; i < W / 4; ++i) {
      const uint32_t lo = __builtin_amdgcn_perm(as_u32(t[4 * i + 1]), as_u32(t[4 * i]), 0x0c0c0400u);
      const uint32_t hi = __builtin_amdgcn_perm(as_u32(t[4 * i + 3]), as_u32(t[4 * i + 2]), 0x04000c0cu);
      code[i] = lo | hi;
    }
    if (special || __builtin_amdgcn_ballot_w64(worst > kSafe) != 0) {
#pragma unroll
      for (int i = 0; i < W / 4; ++i) {
        code[i] = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) code[i] |= (static_cast<uint32_t>(code_exact(f[4 * i + b], sc)) & 0xffu) << (8 * b);
      }
    }
    const uint32_t off = static_cast<uint32_t>(slot + j * stride) * W;
    if constexpr (W == 8) buf_store8(rq, off, u32x2{code[0], code[1]});
    else __builtin_amdgcn_raw_buffer_store_b32(code[0], rq, off, 0, kStreamAux);
  }
}

// Any k, stride or alignment: a wave per row, scalar accesses, two passes.
template <typename TW>
__global__ __launch_bounds__(256) void quantize_int8_generic(const void* __restrict__ w, int8_t* __restrict__ q,
                                                             float* __restrict__ scale, int64_t n, int k, int64_t ws,
                                                             int64_t qs) {
  const int lane = threadIdx.x & 63;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= n) return;
  float m = 0.f;
  for (int c = lane; c < k; c += 64) m = __builtin_fmaxf(m, __builtin_fabsf(load_elem<TW>(w, r * ws + c)));
  const float sc = row_scale(as_f32(wave_allreduce_max(as_u32(m))));  // magnitudes order like their bits
  if (lane == 0) scale[r] = sc;
  for (int c = lane; c < k; c += 64) q[r * qs + c] = static_cast<int8_t>(code_exact(load_elem<TW>(w, r * ws + c), sc));
}

struct QuantArgs {
  const void* w;
  void* q;
  void* scale;
  int64_t n;
  int k;
  int64_t ws, qs;
};

template <typename K>
int launch_quant(K kernel, int64_t grid, int block, const QuantArgs& a, hipStream_t s) {
  void* args[] = {const_cast<void**>(&a.w), const_cast<void**>(&a.q), const_cast<void**>(&a.scale),
                  const_cast<int64_t*>(&a.n), const_cast<int*>(&a.k), const_cast<int64_t*>(&a.ws),
                  const_cast<int64_t*>(&a.qs)};
  return hip_status(hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(static_cast<unsigned>(grid)),
                                    dim3(block), args, 0, s),
                    "quantize_int8 launch");
}

// Packets need whole ones per row, 16-byte aligned weight rows and code rows
// aligned to a packet's codes.
template <typename TW>
int quant_typed(const QuantArgs& a, hipStream_t s) {
  constexpr int W = pack_width<TW>::value;
  const int64_t eb = sizeof(typename TW::bits);
  const bool vec = a.k % W == 0 && aligned16(a.w) && a.ws * eb % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(a.q) % W == 0 && a.qs % W == 0;
  const QuantPlan p = quant_plan(a.n, vec ? a.k / W : 0);
  if (p.block) {
    if (p.vpl == 4) return launch_quant(quantize_int8_rows<TW, 4, true>, p.grid, p.threads, a, s);
    return launch_quant(quantize_int8_rows<TW, 8, true>, p.grid, p.threads, a, s);
  }
  switch (p.vpl) {
    case 1: return launch_quant(quantize_int8_rows<TW, 1, false>, p.grid, p.threads, a, s);
    case 2: return launch_quant(quantize_int8_rows<TW, 2, false>, p.grid, p.threads, a, s);
    case 3: return launch_quant(quantize_int8_rows<TW, 3, false>, p.grid, p.threads, a, s);
    case 4: return launch_quant(quantize_int8_rows<TW, 4, false>, p.grid, p.threads, a, s);
    case 5: return launch_quant(quantize_int8_rows<TW, 5, false>, p.grid, p.threads, a, s);
    case 6: return launch_quant(quantize_int8_rows<TW, 6, false>, p.grid, p.threads, a, s);
    case 7: return launch_quant(quantize_int8_rows<TW, 7, false>, p.grid, p.threads, a, s);
    case 8: return launch_quant(quantize_int8_rows<TW, 8, false>, p.grid, p.threads, a, s);
    default: return launch_quant(quantize_int8_generic<TW>, p.grid, p.threads, a, s);
  }
}

}  // namespace

int quantize_int8_launch(const void* w, void* q, void* scale, int64_t n, int k, int64_t ws, int64_t qs, int w_dtype,
                         hipStream_t stream) {
  const QuantArgs a{w, q, scale, n, k, ws, qs};
  if (w_dtype == MI355_F32) return quant_typed<F32>(a, stream);
  if (w_dtype == MI355_F16) return quant_typed<F16>(a, stream);
  if (w_dtype == MI355_BF16) return quant_typed<BF16>(a, stream);
  set_error("mi355_quantize_int8_fwd: unsupported weight dtype %d", w_dtype);
  return MI355_ERR_UNSUPPORTED;
}

}  // namespace mi355
