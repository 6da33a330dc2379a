// santa_attn.hip -- exact attention of the model-level runtime
// (santa_amd/runtime.py) at head_dim 128: the causal attention of a prefill and
// the decode attention of the exact comparator.  The reference leaves both to
// torch's and the HF model's own attention (tutorial_code/runtime_common.py:
// 501-571, tutorial_code/attention_backends.py:70-89).
#include "santa_device.h"
#include "santa_amd.h"
#include "santa_internal.h"

#include <algorithm>
#include <type_traits>

namespace santa {
namespace attn {

constexpr int kD = 128;
constexpr int kBufWord3 = 0x00020000;  // raw buffer descriptor, gfx9 family
constexpr int kBufNontemporal = 2;     // the "nt" cache-policy bit

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

// Where running maxima start: below every finite score, so that scores of -inf
// (masked through K) weigh nothing as long as one key of the query is finite;
// relative to a maximum of -inf they would be NaN.
constexpr float kLowest = -3.402823466e38f;

// Above this a maximum in log2 units is subtracted from the scores before they
// are scaled: fma(score, scale, -round(max * scale)) is off by half an ulp of
// the product, up to a factor 2^(1/4) common to a query's probabilities here but
// an overflow from 2^31 on (scores from about 2e10).
constexpr float kHugeMax = 4194304.0f;

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
// B = 2, P = 4096, 32q/8kv the call takes 280 to 310 us on one card or another,
// 890 to 980 TFLOP/s over the causal pairs (a large library matrix product
// reaches 1,349); the torch expressions it replaces (all P x P scores of a query
// chunk, written and read back five times over) took 8,536 us.
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
  float m = kLowest, l = 0.0f;  // running max (of the raw scores) and this half's sum
  // mc: m in log2 units, or 0 where the scores have m subtracted (kHugeMax);
  // grows: m, or -inf there, so that every tile's scores pass that way
  float mc = 0.0f, grows = -__builtin_inff();

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
    // Rescaling whenever a maximum grows, not only once it has grown by some
    // factor (273 us at the size above), keeps the largest probability exactly
    // 1: rounded relative to an older maximum it would be off by up to an ulp,
    // and with it the whole output of a query that attends to one key.
    if (__any(m_new > grows)) {
      const float a = __builtin_amdgcn_exp2f((m - m_new) * scale_log2);
      l *= a;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[mb][i] *= a;
      grows = m = m_new;
      mc = m * scale_log2;
      if (__any(fabsf(mc) > kHugeMax)) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[kb][i] -= m;
        mc = 0.0f;
        grows = -__builtin_inff();
      }
    }
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

// ------------------------------------------------------------ exact decode
// Exact decode attention: one query row per sequence over its first L cached
// positions, everything in float32 (the 16-bit operands are exact; products,
// scores, probabilities and sums are float32).
//
// A wave takes one item, a chunk of positions of one (sequence, KV head, up to
// GHP of its query heads).  16 lanes hold a K or V row (16 bytes each), so a
// load instruction covers 4 rows and a step 32 positions: the scores are
// v_dot2 chains over the lane's 8 dims summed over the row's 16 lanes by
// halving exchanges (each head's score ends in 16 / GHP of them), the step's
// maximum meets across the 4 rows, and each probability goes back to its row's
// lanes by a DPP broadcast for the V sums.  Matrix cores would not help: at GH
// query rows the call reads 2 bytes per 2 GH multiply-adds.  The next step's
// K rows are loaded once this step's scores are formed and its V rows once
// this step's are summed, so 8 to 16 KiB per wave are in flight throughout.
// The KV heads of a chunk are neighbours in launch order (8 waves of a
// workgroup), so whole NHD rows are read at about the same time.  Bound by
// reading K and V once (us per call with the merge, K and V tensors of their
// own): B = 8, 32k, 32q/8kv 168 (6.4 TB/s), 32q/32kv at 8k 168 (6.4 TB/s); eight
// heads per KV head double the vector work per row (64q/8kv 202 to 216, 5.0 to 5.3
// TB/s).  The torch products on float32 copies of both caches it replaces took
// 1,679, 1,797 and 2,000; B = 4, 4k: 21 against 135.
constexpr int kDecWaves = 8;
constexpr int kDecStep = 32;              // positions per step
constexpr int kPartStride = kD + 2;       // chunk partial: max (log2 units), mass, numerator[128]
constexpr int kMaxChunks = 256;           // chunks per sequence (the merge holds one per thread)

template <bool BF16>
__device__ __forceinline__ float dot8(u32x4 a, u32x4 b) {
  typedef typename Half8<BF16>::T H8;
  const H8 x = __builtin_bit_cast(H8, a), y = __builtin_bit_cast(H8, b);
  float acc = 0.0f;
  if constexpr (BF16) {
    acc = __builtin_amdgcn_fdot2_f32_bf16(x.s01, y.s01, acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(x.s23, y.s23, acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(x.s45, y.s45, acc, false);
    return __builtin_amdgcn_fdot2_f32_bf16(x.s67, y.s67, acc, false);
  } else {
    acc = __builtin_amdgcn_fdot2(x.s01, y.s01, acc, false);
    acc = __builtin_amdgcn_fdot2(x.s23, y.s23, acc, false);
    acc = __builtin_amdgcn_fdot2(x.s45, y.s45, acc, false);
    return __builtin_amdgcn_fdot2(x.s67, y.s67, acc, false);
  }
}

// v of lane N of this lane's 16-lane row.
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xF, 0xF, true));
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>).
template <int N, class F, int I = 0>
__device__ __forceinline__ void static_for(F f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, F, I + 1>(f);
  }
}

template <bool BF16, int GHP>
__global__ __launch_bounds__(64 * kDecWaves) void exact_decode_kernel(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V, Strides sk,
    Strides sv, int L, int H, int KVH, int GH, int groups, int chunk, int cpg, long long items, float scale_log2,
    float* __restrict__ part) {
  constexpr int SH = GHP == 1 ? 0 : GHP == 2 ? 1 : GHP == 4 ? 2 : 3;
  const int lane = threadIdx.x & 63;
  const long long item =
      static_cast<long long>(blockIdx.x) * kDecWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= items) return;
  // items: (sequence, chunk, KV head, head group), the last fastest
  const int grp = static_cast<int>(item % groups);
  const int kv = static_cast<int>(item / groups % KVH);
  const int c = static_cast<int>(item / groups / KVH % cpg);
  const int b = static_cast<int>(item / groups / KVH / cpg);
  const int h0 = kv * GH + grp * GHP;
  const int nh = min(GHP, GH - grp * GHP);
  const int n_begin = c * chunk, n_end = min(L, n_begin + chunk);
  const int r = lane >> 4, p = lane & 15;

  u32x4 q[GHP];
#pragma unroll
  for (int g = 0; g < GHP; ++g)
    q[g] = *reinterpret_cast<const u32x4*>(Q + (static_cast<size_t>(b) * H + h0 + min(g, nh - 1)) * kD + 8 * p);

  const char* Kg = reinterpret_cast<const char*>(K + b * sk.b + kv * sk.h);
  const char* Vg = reinterpret_cast<const char*>(V + b * sv.b + kv * sv.h);
  const uint32_t k_row = static_cast<uint32_t>(sk.p * 2), v_row = static_cast<uint32_t>(sv.p * 2);
  // rows n .. n + 31, 4 per load; rows at or past the chunk's end read as zero
  auto load = [&](u32x4 (&w)[8], const char* base, uint32_t row, int n) {
    const int nvalid = min(n_end - n, kDecStep);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(base) + static_cast<size_t>(nvalid > 0 ? n : n_begin) * row, static_cast<short>(0),
        nvalid > 0 ? static_cast<int>((nvalid - 1) * row + 2 * kD) : 0, kBufWord3);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      w[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (4 * i + r) * row + 16 * p, 0,
                                                                             kBufNontemporal));
  };
  u32x4 kw[8], vw[8];
  load(kw, Kg, k_row, n_begin);
  load(vw, Vg, v_row, n_begin);

  float o[GHP][8];
#pragma unroll
  for (int g = 0; g < GHP; ++g)
#pragma unroll
    for (int d = 0; d < 8; ++d) o[g][d] = 0.0f;
  // of the head whose scores end in this lane: running max (raw scores) and
  // the mass of this row's positions
  float m = kLowest, l = 0.0f;
  float mc = 0.0f, grows = -__builtin_inff();  // as in causal_attention_kernel

  for (int n = n_begin; n < n_end; n += kDecStep) {
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      typedef float acc_t __attribute__((ext_vector_type(GHP == 1 ? 2 : GHP)));
      acc_t a = {};
#pragma unroll
      for (int g = 0; g < GHP; ++g) a[g] = dot8<BF16>(kw[i], q[g]);
      lane_reduce<GHP, 8>(a, lane);
      s[i] = (n + 4 * i + r < n_end) ? a[0] : -__builtin_inff();
    }
    load(kw, Kg, k_row, n + kDecStep);
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, s[i]);
    mx = fmaxf(mx, fxor<16>(mx, lane));
    mx = fmaxf(mx, fxor<32>(mx, lane));
    const float m_new = fmaxf(m, mx);
    if (__any(m_new > grows)) {
      const float a = __builtin_amdgcn_exp2f((m - m_new) * scale_log2);
      l *= a;
      static_for<GHP>([&](auto gc) {
        constexpr int g = decltype(gc)::value;
        const float ag = row_bcast<g << (4 - SH)>(a);
#pragma unroll
        for (int d = 0; d < 8; ++d) o[g][d] *= ag;
      });
      grows = m = m_new;
      mc = m * scale_log2;
      if (__any(fabsf(mc) > kHugeMax)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] -= m;
        mc = 0.0f;
        grows = -__builtin_inff();
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], scale_log2, -mc));
      l += s[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float v[8];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        v[2 * d] = lo16_to_f32<BF16>(vw[i][d]);
        v[2 * d + 1] = hi16_to_f32<BF16>(vw[i][d]);
      }
      static_for<GHP>([&](auto gc) {
        constexpr int g = decltype(gc)::value;
        const float pg = row_bcast<g << (4 - SH)>(s[i]);
#pragma unroll
        for (int d = 0; d < 8; ++d) o[g][d] = fmaf(pg, v[d], o[g][d]);
      });
    }
    load(vw, Vg, v_row, n + kDecStep);
  }
  // the 4 rows' sums
  l += fxor<16>(l, lane);
  l += fxor<32>(l, lane);
  static_for<GHP>([&](auto gc) {
    constexpr int g = decltype(gc)::value;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      o[g][d] += fxor<16>(o[g][d], lane);
      o[g][d] += fxor<32>(o[g][d], lane);
    }
    const float mg = row_bcast<g << (4 - SH)>(m), lg = row_bcast<g << (4 - SH)>(l);
    if (g < nh && r == (g & 3)) {
      // partials [sequence, head, chunk]
      float* pp = part + ((static_cast<size_t>(b) * H + h0 + g) * cpg + c) * kPartStride;
      if (p == 0) *reinterpret_cast<float2*>(pp) = make_float2(mg * scale_log2, lg);
#pragma unroll
      for (int d = 0; d < 8; d += 2) *reinterpret_cast<float2*>(pp + 2 + 8 * p + d) = make_float2(o[g][d], o[g][d + 1]);
    }
  });
}

// out[d] = sum_c w_c num_c[d] / sum_c w_c mass_c, w_c = 2^(max_c - max), per
// (sequence, head): 256 threads, thread c weighing chunk c, then two threads
// per dim over the even and the odd chunks.
template <bool BF16>
__global__ __launch_bounds__(256) void exact_merge_kernel(const float* __restrict__ part, int cpg,
                                                          uint16_t* __restrict__ out) {
  __shared__ float s_w[kMaxChunks];
  __shared__ float s_red[8];
  __shared__ float s_o[kD];
  const size_t bh = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* pb = part + bh * cpg * kPartStride;
  float2 ml = make_float2(-__builtin_inff(), 0.0f);
  if (tid < cpg) ml = *reinterpret_cast<const float2*>(pb + static_cast<size_t>(tid) * kPartStride);
  float mx = ml.x;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
  if (lane == 0) s_red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  const float w = tid < cpg ? __builtin_amdgcn_exp2f(ml.x - mx) : 0.0f;
  s_w[tid] = w;
  float z = tid < cpg ? w * ml.y : 0.0f;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) z += __shfl_xor(z, d, 64);
  if (lane == 0) s_red[4 + wave] = z;
  __syncthreads();
  z = (s_red[4] + s_red[5]) + (s_red[6] + s_red[7]);
  const int d = tid & (kD - 1);
  float acc = 0.0f;
#pragma unroll 16
  for (int c = tid >> 7; c < cpg; c += 2) acc = fmaf(s_w[c], pb[static_cast<size_t>(c) * kPartStride + 2 + d], acc);
  if (tid >= kD) s_o[d] = acc;
  __syncthreads();
  if (tid < kD) out[bh * kD + d] = f32_to_h16<BF16>((acc + s_o[d]) / z);
}

// Chunks of the exact decode: about one resident round of waves (two per SIMD,
// what the widest form's registers hold), at least 64 positions each, at most
// kMaxChunks per sequence.
void plan_decode(int B, int L, int KVH, int groups, int* chunk, int* cpg) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  const long long per_seq = static_cast<long long>(KVH) * groups * B;
  const long long want = (8LL * cus + per_seq - 1) / per_seq;  // chunks per sequence
  const long long n = want < 1 ? 1 : want > kMaxChunks ? kMaxChunks : want;
  long long len = (L + n - 1) / n;
  len = (len + kDecStep - 1) / kDecStep * kDecStep;
  if (len < 64) len = 64;
  *chunk = static_cast<int>(len);
  *cpg = static_cast<int>((L + len - 1) / len);
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
  const long long W = (units + NW - 1) / NW;
  // a launch holds fewer than 2^32 threads and drops the rest without an error:
  // at most this many sequences each
  const long long per_seq = W * KVH;
  const long long fit = (1LL << 32) / (64 * NW) - 1;
  if (units > 0x7fffff00LL || per_seq > fit)
    return set_error(SANTA_ERR_INVALID, "causal_attention: too many positions");
  const float scale_log2 = 1.44269504088896340736f / sqrtf(static_cast<float>(D));
  const dim3 block(64 * NW);
  for (long long b0 = 0, step = fit / per_seq; b0 < B; b0 += step) {
    const long long n = std::min<long long>(step, B - b0) * KVH;
    const dim3 grid(static_cast<unsigned>(W * n));
    const uint16_t *qp = static_cast<const uint16_t*>(q) + b0 * sq.b, *kp = static_cast<const uint16_t*>(k) + b0 * sk.b,
                   *vp = static_cast<const uint16_t*>(v) + b0 * sv.b;
    uint16_t* op = static_cast<uint16_t*>(out) + b0 * so.b;
    if (dtype == SANTA_BF16)
      hipLaunchKernelGGL((attn::causal_attention_kernel<true, NW>), grid, block, 0, stream, qp, kp, vp, op, sq, sk, sv,
                         so, P, GH, KVH, static_cast<int>(n), static_cast<int>(W), scale_log2);
    else
      hipLaunchKernelGGL((attn::causal_attention_kernel<false, NW>), grid, block, 0, stream, qp, kp, vp, op, sq, sk,
                         sv, so, P, GH, KVH, static_cast<int>(n), static_cast<int>(W), scale_log2);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(SANTA_ERR_HIP, "causal_attention launch failed: %s", hipGetErrorString(e));
  return clear_error();
}

extern "C" size_t santa_rt_exact_decode_workspace_size(int B, int L, int H, int KVH) {
  if (B <= 0 || L <= 0 || KVH <= 0 || H <= 0 || H % KVH != 0) return 0;
  int chunk, cpg;
  attn::plan_decode(B, L, KVH, (H / KVH + 7) / 8, &chunk, &cpg);
  return static_cast<size_t>(B) * H * cpg * attn::kPartStride * sizeof(float);
}

extern "C" int santa_rt_exact_decode(const void* q, const void* k, const void* v, void* out, int dtype, int B, int L,
                                     int H, int KVH, int D, const long long* strides, void* workspace,
                                     size_t workspace_bytes, hipStream_t stream) {
  if (!q || !k || !v || !out || !strides || !workspace || (dtype != SANTA_BF16 && dtype != SANTA_F16) || B <= 0 ||
      L <= 0 || KVH <= 0 || H <= 0 || H % KVH != 0)
    return set_error(SANTA_ERR_INVALID, "bad exact_decode arguments");
  if (D != attn::kD) return set_error(SANTA_ERR_UNSUPPORTED, "exact_decode: D must be 128. Got D=%d", D);
  const attn::Strides sk{strides[0], strides[1], strides[2]}, sv{strides[3], strides[4], strides[5]};
  if (reinterpret_cast<uintptr_t>(q) % 16 != 0 || !strides_fit(sk, k) || !strides_fit(sv, v))
    return set_error(SANTA_ERR_INVALID, "exact_decode: strides must be multiples of 8 elements (the position stride "
                                        "below 2^24) and the tensors 16-byte aligned");
  if (workspace_bytes < santa_rt_exact_decode_workspace_size(B, L, H, KVH))
    return set_error(SANTA_ERR_WORKSPACE, "exact_decode: workspace too small");
  const int GH = H / KVH, groups = (GH + 7) / 8;
  int chunk, cpg;
  attn::plan_decode(B, L, KVH, groups, &chunk, &cpg);
  // a launch holds fewer than 2^32 threads: at most this many sequences each
  // (a wave per item, 256 threads a head in the merge)
  const long long per_seq = static_cast<long long>(KVH) * groups * cpg;
  const long long step = std::min((1LL << 25) / per_seq, (1LL << 23) / H);
  if (step == 0) return set_error(SANTA_ERR_INVALID, "exact_decode: too many heads");
  const float scale_log2 = 1.44269504088896340736f / sqrtf(static_cast<float>(D));
  for (long long b0 = 0; b0 < B; b0 += step) {
    const long long n = std::min<long long>(step, B - b0);
    const long long items = n * per_seq;
    const dim3 grid(static_cast<unsigned>((items + attn::kDecWaves - 1) / attn::kDecWaves));
    const dim3 heads(static_cast<unsigned>(n * H));
    const uint16_t *qp = static_cast<const uint16_t*>(q) + b0 * H * D, *kp = static_cast<const uint16_t*>(k) + b0 * sk.b,
                   *vp = static_cast<const uint16_t*>(v) + b0 * sv.b;
    uint16_t* op = static_cast<uint16_t*>(out) + b0 * H * D;
    float* part = static_cast<float*>(workspace) + b0 * H * cpg * attn::kPartStride;
    auto launch = [&](auto bf, auto ghp) {
      constexpr bool BF16 = decltype(bf)::value;
      constexpr int GHP = decltype(ghp)::value;
      hipLaunchKernelGGL((attn::exact_decode_kernel<BF16, GHP>), grid, dim3(64 * attn::kDecWaves), 0, stream, qp, kp,
                         vp, sk, sv, L, H, KVH, GH, groups, chunk, cpg, items, scale_log2, part);
    };
    auto pick = [&](auto bf) {
      if (GH == 1) launch(bf, std::integral_constant<int, 1>{});
      else if (GH == 2) launch(bf, std::integral_constant<int, 2>{});
      else if (GH <= 4) launch(bf, std::integral_constant<int, 4>{});
      else launch(bf, std::integral_constant<int, 8>{});
    };
    if (dtype == SANTA_BF16) {
      pick(std::true_type{});
      hipLaunchKernelGGL(attn::exact_merge_kernel<true>, heads, dim3(256), 0, stream, part, cpg, op);
    } else {
      pick(std::false_type{});
      hipLaunchKernelGGL(attn::exact_merge_kernel<false>, heads, dim3(256), 0, stream, part, cpg, op);
    }
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(SANTA_ERR_HIP, "exact_decode launch failed: %s", hipGetErrorString(e));
  return clear_error();
}
