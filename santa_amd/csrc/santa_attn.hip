// santa_attn.hip -- exact attention of the model-level runtime
// (santa_amd/runtime.py) at head_dim 128: the causal attention of a prefill.
// The reference leaves it to the HF model's own attention
// (tutorial_code/runtime_common.py:501-571).
#include "santa_device.h"
#include "santa_amd.h"
#include "santa_internal.h"

#include <type_traits>

namespace santa {
namespace attn {

constexpr int kD = 128;
constexpr int kBufWord3 = 0x00020000;  // raw buffer descriptor, gfx9 family

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

template <bool BF16>
struct Half8 {
  typedef __bf16 T __attribute__((ext_vector_type(8)));
};
template <>
struct Half8<false> {
  typedef _Float16 T __attribute__((ext_vector_type(8)));
};

// Eight 16-bit values travel as u32x4: the kernels' own code names no 16-bit
// vector type, which the host pass does not have.
template <bool BF16>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  typedef typename Half8<BF16>::T H8;
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(H8, a), __builtin_bit_cast(H8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(H8, a), __builtin_bit_cast(H8, b), c, 0, 0, 0);
  }
}

// Eight floats rounded to nearest even into the 16-bit type.
template <bool BF16>
__device__ __forceinline__ u32x4 pack8(const float (&e)[8]) {
  typedef typename Half8<BF16>::T H8;
  H8 v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = static_cast<std::remove_reference_t<decltype(v[0])>>(e[i]);
  return __builtin_bit_cast(u32x4, v);
}

// v of lane i ^ 32.
__device__ __forceinline__ float other_half(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float((threadIdx.x & 32) ? s[0] : s[1]);
}

// This lane's column of two 4-row groups of a row-major 16-bit LDS tile, 8
// rows (2048 bytes) apart, through the transposing read: in each 16-lane
// group, lane i passes the address of 4 elements of row i / 4 and receives
// the 4 rows' elements of column i.
__device__ __forceinline__ u32x4 read_tr8(const char* p) {
  typedef __attribute__((address_space(3))) s16x4* lds4;
  struct Two {
    s16x4 a, b;
  };
  const Two f = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p)),
                 __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 2048))};
  return __builtin_bit_cast(u32x4, f);
}

// 16 bytes per lane from rs + off (this lane's byte offset) to LDS, 1 KiB from
// dst on in lane order; nothing waits for it here.
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t rs, u32x4* dst, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(dst), 16, off, 0, 0, 0);
}

constexpr int kTileKeys = 64;
constexpr int kTileVecs = kTileKeys * kD * 2 / 16;  // 16-byte LDS slots of one K or V tile

// Element strides of [B, P, heads, 128] tensors whose last dimension is
// contiguous.
struct Strides {
  long long b, p, h;
};

// Causal GQA attention of P positions: flash attention over 64-key tiles.
// A wave owns one unit, 32 consecutive positions of one query head; the NW
// waves of a workgroup take NW consecutive units of one (sequence, KV head),
// heads fastest, so they walk the same keys.
//
// Per tile the wave forms S^T = K Q^T (v_mfma 32x32x16: the 32 x 32 result
// holds one query per lane, 16 keys of it in registers), so the softmax
// statistics of a query are per-lane scalars (the two lane halves hold
// different keys and meet once for the maximum), and P^T, rounded to 16 bits
// in place, is the B operand of O^T += V^T P^T without leaving its lane: V^T's
// fragments are read with the keys in the order S^T's registers have them.
// They come from the row-major V tile through the transposing LDS read
// (ds_read_b64_tr_b16).  Scores, statistics and both sums are float32; the
// probabilities are rounded to the 16-bit type as the torch path rounds them
// before its second product, the scores are not.
//
// K and V tiles are loaded straight into LDS (no registers held), two buffers
// deep, one barrier per tile.  A K row's 16-byte pieces sit at slot
// piece ^ (row & 15), a V row's at piece ^ 4 (row & 3), which leaves both
// reads without bank conflicts.
//
// Bound by the matrix cores and the softmax's vector work beside them.  At
// B = 2, P = 4096, 32q/8kv the call takes 289 us, 954 TFLOP/s over the causal
// pairs (a large library matrix product reaches 1,349 on this card); the torch
// expressions it replaces (all P x P scores of a query chunk, written and read
// back five times over) took 8,513 us.
//
// The workgroups of one (sequence, KV head) are NG apart, so with NG a
// multiple of 8 they share an XCD and its L2 holds their K and V; the longest
// (last positions) start first.
template <bool BF16, int NW>
__global__ __launch_bounds__(64 * NW, 2) void causal_attention_kernel(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V,
    uint16_t* __restrict__ O, Strides sq, Strides sk, Strides sv, Strides so, int P, int GH, int KVH, int NG, int W,
    float scale_log2) {
  __shared__ u32x4 s_kv[2][2 * kTileVecs];  // per buffer: the K tile, the V tile
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ng = blockIdx.x % NG;
  const int idx = W - 1 - blockIdx.x / NG;
  const int b = ng / KVH, kv = ng % KVH;
  const int half = lane >> 5, ql = lane & 31;
  const int units = ((P + 31) / 32) * GH;
  const int u = idx * NW + wave;
  const bool active = u < units;
  const int pb = min(u, units - 1) / GH;  // position block of this wave
  const int g = min(u, units - 1) % GH;
  const int qpos = 32 * pb + ql;
  const int pb_last = min(idx * NW + NW - 1, units - 1) / GH;
  const int nt = pb_last / 2 + 1;            // tiles of the workgroup
  const int my_nt = active ? pb / 2 + 1 : 0; // tiles of this wave

  const char* Kg = reinterpret_cast<const char*>(K + b * sk.b + kv * sk.h);
  const char* Vg = reinterpret_cast<const char*>(V + b * sv.b + kv * sv.h);
  const uint32_t k_row = static_cast<uint32_t>(sk.p * 2), v_row = static_cast<uint32_t>(sv.p * 2);
  // load group c: rows 4c .. 4c+3 of the tile, 16 lanes each
  const uint32_t lrow = lane >> 4, lslot = lane & 15;
  uint32_t k_off[16 / NW];
#pragma unroll
  for (int i = 0; i < 16 / NW; ++i) {
    const uint32_t r = 4 * (wave + NW * i) + lrow;
    k_off[i] = r * k_row + 16 * (lslot ^ (r & 15));
  }
  const uint32_t v_off = (4 * wave + lrow) * v_row + 16 * (lslot ^ (4 * lrow));
  auto load_tile = [&](int t, int buf) {
    const int n0 = t * kTileKeys;
    const int nvalid = min(P - n0, kTileKeys);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(Kg) + static_cast<size_t>(n0) * k_row, static_cast<short>(0),
        static_cast<int>((nvalid - 1) * k_row + 2 * kD), kBufWord3);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(Vg) + static_cast<size_t>(n0) * v_row, static_cast<short>(0),
        static_cast<int>((nvalid - 1) * v_row + 2 * kD), kBufWord3);
    u32x4* const dst = s_kv[buf];
#pragma unroll
    for (int i = 0; i < 16 / NW; ++i) {
      const int c = wave + NW * i;
      load_lds16(rk, dst + 64 * c, k_off[i]);
      load_lds16(rv, dst + kTileVecs + 64 * c, v_off + static_cast<uint32_t>(4 * NW * i) * v_row);
    }
  };
  load_tile(0, 0);

  // Q fragments: dims 16c + 8 half .. + 7 of this lane's query
  u32x4 qf[8];
  {
    const uint16_t* qr = Q + b * sq.b + static_cast<long long>(min(qpos, P - 1)) * sq.p + (kv * GH + g) * sq.h + 8 * half;
#pragma unroll
    for (int c = 0; c < 8; ++c) qf[c] = *reinterpret_cast<const u32x4*>(qr + 16 * c);
  }
  // LDS byte offsets of this lane's fragments inside a buffer
  uint32_t ko[8], vo[4];
#pragma unroll
  for (int c = 0; c < 8; ++c) ko[c] = ql * 256 + 16 * ((2 * c + half) ^ (lane & 15));
  const int r3 = (lane & 15) >> 2;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
    vo[mb] = 16 * kTileVecs + (4 * half + r3) * 256 + 16 * (4 * (mb ^ r3) + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) +
             8 * (lane & 1);

  f32x16 o[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[mb][i] = 0.0f;
  float m = -__builtin_inff(), l = 0.0f;  // running max (of the raw scores) and this half's sum

  for (int t = 0; t < nt; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // tile t is in LDS, and no wave reads the other buffer any more
    if (t + 1 < nt) load_tile(t + 1, (t + 1) & 1);
    if (t >= my_nt) continue;
    const char* buf = reinterpret_cast<const char*>(s_kv[t & 1]);
    f32x16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kb][i] = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c)
        s[kb] = mfma32<BF16>(*reinterpret_cast<const u32x4*>(buf + ko[c] + 32 * 256 * kb), qf[c], s[kb]);
    }
    if (t == my_nt - 1) {  // the tile on the diagonal: keys after the query take no part
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = t * kTileKeys + 32 * kb + 8 * (i >> 2) + 4 * half + (i & 3);
          if (key > qpos) s[kb][i] = -__builtin_inff();
        }
    }
    float mx = s[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb][i]);
    mx = fmaxf(mx, other_half(mx));
    const float m_new = fmaxf(m, mx);
    if (__any(m_new > m)) {
      const float a = __builtin_amdgcn_exp2f((m - m_new) * scale_log2);
      l *= a;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[mb][i] *= a;
      m = m_new;
    }
    const float mc = m * scale_log2;
    u32x4 p[4];
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        e[i] = __builtin_amdgcn_exp2f(fmaf(s[kc >> 1][8 * (kc & 1) + i], scale_log2, -mc));
        l += e[i];
      }
      p[kc] = pack8<BF16>(e);
    }
#pragma unroll
    for (int kc = 0; kc < 4; ++kc)
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        o[mb] = mfma32<BF16>(read_tr8(buf + vo[mb] + 4096 * kc), p[kc], o[mb]);
      }
  }
  if (!active || qpos >= P) return;
  l += other_half(l);
  const float inv = 1.0f / l;
  uint16_t* orow = O + b * so.b + static_cast<long long>(qpos) * so.p + (kv * GH + g) * so.h;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      uint2 w;
      w.x = f32_to_h16<BF16>(o[mb][i] * inv) | (static_cast<uint32_t>(f32_to_h16<BF16>(o[mb][i + 1] * inv)) << 16);
      w.y = f32_to_h16<BF16>(o[mb][i + 2] * inv) | (static_cast<uint32_t>(f32_to_h16<BF16>(o[mb][i + 3] * inv)) << 16);
      *reinterpret_cast<uint2*>(orow + 32 * mb + 2 * i + 4 * half) = w;
    }
}

}  // namespace attn
}  // namespace santa

using namespace santa;

namespace {
// Strides of one [B, P, heads, 128] tensor the kernels can address: 16-byte
// aligned rows, a tile's rows within 32-bit offsets.
bool strides_fit(const attn::Strides& s, const void* p) {
  return reinterpret_cast<uintptr_t>(p) % 16 == 0 && s.b >= 0 && s.p >= 0 && s.h >= 0 && s.b % 8 == 0 &&
         s.p % 8 == 0 && s.h % 8 == 0 && s.p < (1LL << 24);
}
}  // namespace

extern "C" int santa_rt_causal_attention(const void* q, const void* k, const void* v, void* out, int dtype, int B,
                                         int P, int H, int KVH, int D, const long long* strides, hipStream_t stream) {
  if (!q || !k || !v || !out || !strides || (dtype != SANTA_BF16 && dtype != SANTA_F16) || B <= 0 || P <= 0 ||
      KVH <= 0 || H <= 0 || H % KVH != 0)
    return set_error(SANTA_ERR_INVALID, "bad causal_attention arguments");
  if (D != attn::kD) return set_error(SANTA_ERR_UNSUPPORTED, "causal_attention: D must be 128. Got D=%d", D);
  const attn::Strides sq{strides[0], strides[1], strides[2]}, sk{strides[3], strides[4], strides[5]};
  const attn::Strides sv{strides[6], strides[7], strides[8]}, so{strides[9], strides[10], strides[11]};
  if (!strides_fit(sq, q) || !strides_fit(sk, k) || !strides_fit(sv, v) || !strides_fit(so, out))
    return set_error(SANTA_ERR_INVALID, "causal_attention: strides must be multiples of 8 elements (the position "
                                        "stride below 2^24) and the tensors 16-byte aligned");
  constexpr int NW = 4;
  const int GH = H / KVH;
  const long long units = static_cast<long long>((P + 31) / 32) * GH;
  const long long W = (units + NW - 1) / NW, NG = static_cast<long long>(B) * KVH;
  if (units > 0x7fffff00LL || W * NG > 0x7fffffffLL)
    return set_error(SANTA_ERR_INVALID, "causal_attention: too many positions");
  const float scale_log2 = 1.44269504088896340736f / sqrtf(static_cast<float>(D));
  const dim3 grid(static_cast<unsigned>(W * NG)), block(64 * NW);
  const uint16_t *qp = static_cast<const uint16_t*>(q), *kp = static_cast<const uint16_t*>(k),
                 *vp = static_cast<const uint16_t*>(v);
  if (dtype == SANTA_BF16)
    hipLaunchKernelGGL((attn::causal_attention_kernel<true, NW>), grid, block, 0, stream, qp, kp, vp,
                       static_cast<uint16_t*>(out), sq, sk, sv, so, P, GH, KVH, static_cast<int>(NG),
                       static_cast<int>(W), scale_log2);
  else
    hipLaunchKernelGGL((attn::causal_attention_kernel<false, NW>), grid, block, 0, stream, qp, kp, vp,
                       static_cast<uint16_t*>(out), sq, sk, sv, so, P, GH, KVH, static_cast<int>(NG),
                       static_cast<int>(W), scale_log2);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(SANTA_ERR_HIP, "causal_attention launch failed: %s", hipGetErrorString(e));
  return clear_error();
}
