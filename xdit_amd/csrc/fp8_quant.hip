// fp8 (OCP e4m3fn) quantiser with abs-max scaling for gfx950: the step in front of the fp8
// attention kernel.  Restates per_tensor_quant (xfuser/core/distributed/attention_backend.py:606-615):
//     scale = absmax(x) / 448 ;  y = fp8(x / scale) ;  descale = scale broadcast to (B, H)
// with the abs-max taken over the whole tensor (`per_tensor`) or per (batch, head) slice, or a
// caller-supplied static scale.  With a scratch buffer of the caller: two launches on the
// caller's stream, (1) abs-max reduction, every workgroup storing its maximum in a scratch slot
// of its own, (2) scale and cast, every workgroup folding its slice's partial maxima first and
// the first one of a slice storing the descale; a static scale needs launch (2) only.  Without
// scratch: four launches, (1) clear the (B,H) abs-max buffer (a fill kernel, so the sequence can
// be captured in a HIP graph), (2) abs-max reduction with one atomic max per workgroup, (3) scale
// and cast, (4) turn the abs-max buffer into the descale values.  An optional second tensor (the
// joint keys or values) shares the scales of the first.  Both tensor passes are HBM-bound and read
// 16 bytes per lane; the quotient rounds to the byte of a true fp32 division, so results match the
// reference's `x / scale` bit for bit.  Optionally both passes first rotate each row along head_dim by a
// block Hadamard matrix (_fp8_hadamard_rotate, attention_backend.py:703-714), in registers.
// Several tensors (the q, k and v of one attention call) go through the same launches, blockIdx.z
// selecting the tensor.  Flux-1024's q, k and v (85 MB) with the rotation of q and k: 17.2 us for the
// abs-max (4.9 TB/s) and 23.7 us for the cast (5.4 TB/s), two launches; with a launch pair per tensor, the
// rotation by shuffles and a compiler-made division it was six launches and 116 us.
#include "attn_split.h"
#include "common.h"
#include "launchers.h"

namespace xdit {

namespace quant {

constexpr float kFp8Max = 448.0f;
constexpr int kFiniteNonZero = 0x198;  // class mask: normal and subnormal numbers of either sign
constexpr int kFinite = 0x1f8;         // ... and zeros

// Eight consecutive elements as they are in memory, in 16-byte loads.
template <typename T> struct Chunk {
  static constexpr int N = sizeof(T) / 2;
  typedef __attribute__((ext_vector_type(8 / N))) T vec;
  vec x[N];
};

// The value of the lane whose index differs in exactly bit log2(M) (M = 1, 2, 4 or 8), within the 16
// lanes of a DPP row: quad permutes, the rotation by 8, and for 4 the half-row mirror (lane ^ 7)
// followed by the quad mirror (^ 3).  A DPP operand rides on the addition that uses it, where a
// shuffle is an LDS-pipe instruction per value and level (32 of them per 8 elements at block 128).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int M>
__device__ __forceinline__ float lane_xor(float x) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8, "within a DPP row");
  if constexpr (M == 1) return dpp_move<0xB1>(x);        // quad_perm [1,0,3,2]
  else if constexpr (M == 2) return dpp_move<0x4E>(x);   // quad_perm [2,3,0,1]
  else if constexpr (M == 4) return dpp_move<0x1B>(dpp_move<0x141>(x));  // row_half_mirror, quad_perm [3,2,1,0]
  else return dpp_move<0x128>(x);                        // row_ror:8
}
// One butterfly level across chunks: the upper chunk of a pair takes (other - own), the lower (own + other).
template <int M>
__device__ __forceinline__ void hadamard_level(float (&v)[8], int c) {
  const unsigned flip = (c & M) != 0 ? 0x80000000u : 0u;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float own = __uint_as_float(__float_as_uint(v[j]) ^ flip);
    v[j] = lane_xor<M>(v[j]) + own;
  }
}

// The same level up to a sign that the lane keeps in `r`: own + other or own - other, one multiply-add whose DPP
// operand is the other's value, where the form above changes the sign first (and for 4 moves twice).  Both partners of
// a later level carry the same sign, so it passes through sums unchanged and every rounding is that of the level above
// (one instruction per element for two: the two passes over q, k and v of Flux-1024 49.5 -> 46 us).
// The waits at both ends are the two states between a VALU write and a DPP read of a register.
#define XDIT_FMAC8(CTRL) \
  asm("s_nop 1\n" \
      "v_fmac_f32_dpp %0, %0, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "v_fmac_f32_dpp %1, %1, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "v_fmac_f32_dpp %2, %2, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "v_fmac_f32_dpp %3, %3, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "v_fmac_f32_dpp %4, %4, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "v_fmac_f32_dpp %5, %5, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "v_fmac_f32_dpp %6, %6, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "v_fmac_f32_dpp %7, %7, %8 " CTRL " row_mask:0xf bank_mask:0xf\n" \
      "s_nop 1" \
      : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]) : "v"(sign))
template <int M>
__device__ __forceinline__ void hadamard_signed_level(float (&v)[8], int c, float& r) {
  const float sign = (c & M) != 0 ? -1.f : 1.f;
  r *= sign;
  if constexpr (M == 1) XDIT_FMAC8("quad_perm:[1,0,3,2]");
  else if constexpr (M == 2) XDIT_FMAC8("quad_perm:[2,3,0,1]");
  else if constexpr (M == 8) XDIT_FMAC8("row_ror:8");
  else {
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = __builtin_fmaf(lane_xor<M>(v[j]), sign, v[j]);
  }
}
#undef XDIT_FMAC8

// x r rounded to T.  fp16: one rounding of the exact product, zeros positive (the mixed multiply-add, named
// here because the compiler takes it or a rounded fp32 product and a conversion by the code around).
template <typename T, bool SIGNED_ZERO = false>
__device__ __forceinline__ float rounded_product(float x, float r) {
  if constexpr (sizeof(T) == 2 && !__is_same(T, __bf16)) {
    unsigned y;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(y) : "v"(x), "v"(r));
    return (float)__builtin_bit_cast(_Float16, (unsigned short)y);
  }
  return (float)(T)(SIGNED_ZERO ? x * r : __builtin_fmaf(x, r, 0.f));  // a sum of zero is a positive zero
}

// Rotates the N rows by the Sylvester-Hadamard matrix of size `block` along head_dim, in place in
// the 8-element chunks the threads hold: the three butterfly levels inside a chunk in
// registers, the levels across chunks by exchanging with the lane that holds chunk c ^ m of the
// same row (the chunks of a block, at most 16, sit in consecutive, block-aligned lanes of one wavefront).
// Entries are +-r with r = `scale` rounded to T and the result is rounded to T, like the output
// of a matmul with the matrix held in T.  `c` is the chunk's index within its row.
template <typename T, int N>
__device__ __forceinline__ void hadamard_rows(float (&x)[N][8], int block, float scale, int c) {
  float r = (float)(T)scale;
  int plain = 1, least = 0;
#pragma unroll
  for (int n = 0; n < N; n++) {
    float (&v)[8] = x[n];
    if (block >= 2) {
#pragma unroll
      for (int j = 0; j < 8; j += 2) { const float a = v[j], b = v[j + 1]; v[j] = a + b; v[j + 1] = a - b; }
    }
    if (block >= 4) {
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
#pragma unroll
        for (int i = 0; i < 2; i++) { const float a = v[j + i], b = v[j + i + 2]; v[j + i] = a + b; v[j + i + 2] = a - b; }
      }
    }
    if (block >= 8) {
#pragma unroll
      for (int i = 0; i < 4; i++) { const float a = v[i], b = v[i + 4]; v[i] = a + b; v[i + 4] = a - b; }
    }
    plain &= __builtin_amdgcn_classf(v[0], kFinite);
#pragma unroll
    for (int j = 0; j < 8; j++) least = min(least, __float_as_int(v[j]));
  }
  // The signed form where a chunk holds no infinity or NaN (its first element is the sum of all) and, from here on, no negative
  // zero, whose bits are the least integer: the signed form ends in positive zeros only, and so does the other one
  // then, as its sums are negative zeros only where both terms are.
  if (block >= 64 && __builtin_amdgcn_ballot_w64(!plain || least == (int)0x80000000) == 0) {
#pragma unroll
    for (int n = 0; n < N; n++) {
      float rn = r;
      hadamard_signed_level<1>(x[n], c, rn);
      hadamard_signed_level<2>(x[n], c, rn);
      hadamard_signed_level<4>(x[n], c, rn);
      if (block >= 128) hadamard_signed_level<8>(x[n], c, rn);
#pragma unroll
      for (int j = 0; j < 8; j++) x[n][j] = rounded_product<T>(x[n][j], rn);
    }
    return;
  }
#pragma unroll
  for (int n = 0; n < N; n++) {
    if (block >= 16) hadamard_level<1>(x[n], c);
    if (block >= 32) hadamard_level<2>(x[n], c);
    if (block >= 64) hadamard_level<4>(x[n], c);
    if (block >= 128) hadamard_level<8>(x[n], c);
#pragma unroll
    for (int j = 0; j < 8; j++) x[n][j] = rounded_product<T, true>(x[n][j], r);
  }
}

__global__ void fill_zero_kernel(float* p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

// Both tensor passes: grid = (most blocks per slice, most B*H, tensors of the batch); a job's slices
// have `blocks` workgroups, what is beyond them leaves at once.  A row of D elements is held by D/8
// consecutive threads (8 elements each), a workgroup covers 256 / (D/8) rows per step and every
// thread works on kRowsInFlight rows while the next ones are on their way; rows advance by whole grid steps, so there is
// no division in the loop and the trip count is the same for every thread of a workgroup (the
// lanes of a row exchange data in the Hadamard rotation).  Two rows: the rotation is close behind the loads (about 150
// VALU instructions per 16 bytes), so what hides it is wavefronts, five to seven to a SIMD by registers.
// q, k and v of Flux-1024 and of a 75600 x 5 shard: 45.9 and 161 us with four rows (eight in the abs-max) at once and no request
// ahead, at four to five wavefronts, 40.5 and 144 now; three or four rows a step of the abs-max are no faster at the rule below.
constexpr int kRowsInFlight = 2;
// Rows per thread: eight, and for bf16 9 to 18 where that is a single round of the workgroups that fit at once, 94 % of it work
// (rows of a workgroup come in pairs, so an odd number costs the next even one).  Of 2936 problems in that band (one tensor or q, k and
// v, with and without rotation, 500 to 60000 rows, inputs in the cache or not) the 1230 of such rounds take 3.2 % less than with eight
// rows, 4 % of them over 1 % longer; in the emptier ones it depends on the rest (one rotated tensor 2 % longer, one without rotation 7 %
// less), 26 % over 1 % longer, up to 9 %.  Beyond 18 rows the memory is left to a few workgroups at the end (45 % of 557 longer,
// 40 heads of 9450 by 10 %), and fp16 and fp32, with other numbers of wavefronts, take 2.5 and 3.2 % longer in a round of nine rows or more.
// q, k and v with the rotation, eight rows and one round: 24 heads of 4608 43.6 and 41.6 us, 24 of 6000 56.6 and 53.9.
constexpr int kRowsPerThread = 8;

// `before` runs once per step, between a step's loads and their use.
template <typename T, typename G, typename F>
__device__ __forceinline__ void for_each_chunk(const QuantParams& p, const T* x, int64_t S, int64_t xs_s, int blocks, G&& before, F&& f) {
  const int cpr = p.D >> 3;
  const int rpb = 256 / cpr;              // rows per workgroup step
  const int c = threadIdx.x % cpr;
  const int r = threadIdx.x / cpr;
  const bool lane_live = r < rpb;
  const int64_t step = (int64_t)blocks * rpb;
  // the rows of the next step are requested before those of this one are used
  Chunk<T> next[kRowsInFlight];
  auto request = [&](int64_t base) {
#pragma unroll
    for (int j = 0; j < kRowsInFlight; j++) {
      const int64_t s = base + j * step + r;
      next[j] = *(const Chunk<T>*)(x + (s < S ? s : S - 1) * xs_s + c * 8);  // rows past the end re-read the last row
    }
  };
  int64_t base = (int64_t)blockIdx.x * rpb;
  if (base < S) request(base);
  for (; base < S; base += step * kRowsInFlight) {
    float v[kRowsInFlight][8];
    before();
#pragma unroll
    for (int j = 0; j < kRowsInFlight; j++)
#pragma unroll
      for (int i = 0; i < 8; i++) v[j][i] = (float)next[j].x[i / (8 / Chunk<T>::N)][i % (8 / Chunk<T>::N)];
    if (base + step * kRowsInFlight < S) request(base + step * kRowsInFlight);
    if (p.had_block > 1) hadamard_rows<T>(v, p.had_block, p.had_scale, c);
#pragma unroll
    for (int j = 0; j < kRowsInFlight; j++) {
      const int64_t s = base + j * step + r;
      f(v[j], s, c, lane_live && s < S);
    }
  }
}

// Maximum of a value over the workgroup (256 threads), returned to every thread.
__device__ __forceinline__ float block_max(float m) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  __shared__ float wm[4];
  __syncthreads();  // a previous use of wm is over
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  return fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
}

// Abs-max of a (batch, head) slice over both tensors.  With `partials` every workgroup stores
// its maximum in a slot of its own (no clearing, no atomics); otherwise one atomic max per
// workgroup goes to the slice's entry of the (cleared) amax buffer.
template <typename T>
__global__ __launch_bounds__(256) void absmax_kernel(const QuantBatch batch) {
  const QuantParams& p = batch.job[blockIdx.z];
  const int bh = blockIdx.y;
  if ((int)blockIdx.x >= p.reduce_blocks || bh >= p.B * p.H) return;
  const int b = bh / p.H, h = bh - b * p.H;
  float m = 0.f;
  auto take = [&](float (&v)[8], int64_t, int, bool live) {
    if (live) {
#pragma unroll
      for (int j = 0; j < 8; j++) m = fmaxf(m, fabsf(v[j]));  // fmaxf drops NaN operands
    }
  };
  for_each_chunk<T>(p, (const T*)p.x + b * p.xs_b + h * p.xs_h, p.S, p.xs_s, p.reduce_blocks, [] {}, take);
  if (p.S2 > 0) for_each_chunk<T>(p, (const T*)p.x2 + b * p.x2s_b + h * p.x2s_h, p.S2, p.x2s_s, p.reduce_blocks, [] {}, take);
  m = block_max(m);
  if (threadIdx.x == 0) {
    if (p.partials != nullptr) p.partials[(int64_t)bh * p.reduce_blocks + blockIdx.x] = m;
    // non-negative floats order like their bit patterns
    else atomicMax((unsigned int*)(p.amax + (p.per_tensor ? 0 : bh)), __float_as_uint(m));
  }
}

// x / scale to the fp8 byte of a true fp32 division, in three instructions instead of the dozen of the
// compiler's sequence: with r the correctly rounded 1 / scale, y = q + r (x - q scale) with q = x r
// (Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", 1990).  q is
// within 1.5 units of the quotient (one from r, for quotients near two, and half from its own rounding), the
// remainder in one fused multiply-add has at most 25 bits and so is off by at most 2^-23 units of the quotient, and
// the sum before its last rounding is within 1.75 * 2^-23 units of it.  What can round to another byte than the
// division are thus only quotients that close to the middle between an fp8 rounding point and a neighbouring fp32
// number, a few hundred pairs of mantissas that a host test enumerates: none does.  (The fp32 quotient was the
// division's in 4 * 10^9 random cases as well.)  The bounds need the remainder's and the reciprocal's exponents in range:
// scales outside [2^-80, 2^80] take the division itself, and where q is a zero, an infinity or a NaN it
// is the quotient already (the remainder would cost a negative zero its sign and make an infinity a NaN).
struct Divider {
  float scale, r;
  bool plain;
  __device__ __forceinline__ explicit Divider(float s) : scale(s), r(1.0f / s), plain(!(s >= 0x1p-80f && s <= 0x1p80f)) {}
  __device__ __forceinline__ float operator()(float x) const {
    const float q = x * r;
    const float y = __builtin_fmaf(__builtin_fmaf(-q, scale, x), r, q);
    return __builtin_amdgcn_classf(q, kFiniteNonZero) ? y : q;
  }
};

// Scale and cast of a (batch, head) slice of both tensors.  The scale is the static one, or comes
// from the partial maxima of the abs-max pass (folded here by every workgroup while its first rows
// are on their way; the first workgroup of a slice also stores the slice's descale), or from the amax
// buffer.
template <typename T>
__global__ __launch_bounds__(256) void cast_kernel(const QuantBatch batch) {
  const QuantParams& p = batch.job[blockIdx.z];
  const int bh = blockIdx.y;
  if ((int)blockIdx.x >= p.cast_blocks || bh >= p.B * p.H) return;
  const int b = bh / p.H, h = bh - b * p.H;
  Divider div(1.0f);
  bool have_scale = false;
  auto need_scale = [&] {
    if (have_scale) return;
    have_scale = true;
    float scale;
    if (p.scale_in != nullptr) {
      scale = *p.scale_in;
    } else if (p.partials != nullptr) {
      const int n = p.per_tensor ? p.reduce_blocks * p.B * p.H : p.reduce_blocks;
      const float* src = p.partials + (p.per_tensor ? 0 : (int64_t)bh * p.reduce_blocks);
      float am = 0.f;
      for (int i = threadIdx.x; i < n; i += 256) am = fmaxf(am, src[i]);
      am = block_max(am);
      scale = am > 0.f ? am / kFp8Max : 1.0f;
    } else {
      const float am = p.amax[p.per_tensor ? 0 : bh];
      scale = am > 0.f ? am / kFp8Max : 1.0f;
    }
    if ((p.scale_in != nullptr || p.partials != nullptr) && blockIdx.x == 0 && threadIdx.x == 0) p.descale[bh] = scale;
    div = Divider(scale);
  };
  auto cast_to = [&](unsigned char* y, int64_t ys_s) {
    return [&, y, ys_s](float (&v)[8], int64_t s, int c, bool live) {
      if (div.plain) {
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = v[j] / div.scale;
      } else {
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = div(v[j]);
      }
      int w0 = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
      w0 = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], w0, true);
      int w1 = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], 0, false);
      w1 = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], w1, true);
      i32x2 w = {w0, w1};
      if (live) *(i32x2*)(y + s * ys_s + c * 8) = w;
    };
  };
  for_each_chunk<T>(p, (const T*)p.x + b * p.xs_b + h * p.xs_h, p.S, p.xs_s, p.cast_blocks, need_scale,
                    cast_to((unsigned char*)p.y + b * p.ys_b + h * p.ys_h, p.ys_s));
  if (p.S2 > 0)
    for_each_chunk<T>(p, (const T*)p.x2 + b * p.x2s_b + h * p.x2s_h, p.S2, p.x2s_s, p.cast_blocks, need_scale,
                      cast_to((unsigned char*)p.y2 + b * p.y2s_b + h * p.y2s_h, p.y2s_s));
}

// amax buffer -> descale values, for all B*H entries (the path without a scratch buffer).
__global__ void finalize_kernel(const QuantParams p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  // every thread reads its source before any thread overwrites entry 0 (single workgroup launch
  // when per_tensor; otherwise each thread only touches its own entry)
  float am = p.amax[p.per_tensor ? 0 : (i < n ? i : 0)];
  __syncthreads();
  if (i >= n) return;
  p.descale[i] = am > 0.f ? am / kFp8Max : 1.0f;
}

// The rule above.  Workgroups are rounded up per (batch, head), so they are counted for each number of rows.
template <typename T>
static int rows_per_thread(const QuantBatch& batch) {
  if (!__is_same(T, __bf16)) return kRowsPerThread;
  const int64_t slots = (int64_t)resident_cus() * 6;  // six to a compute unit by the registers of the cast (the abs-max: seven)
  for (int rows = kRowsPerThread; rows <= 18; rows++) {
    int64_t workgroups = 0, steps = 0;  // steps: of one row per thread
    for (int i = 0; i < batch.n; i++) {
      const QuantParams& p = batch.job[i];
      const int64_t rpb = 256 / (p.D >> 3), slice = ((int64_t)p.S + p.S2 + rpb - 1) / rpb;
      steps += (int64_t)p.B * p.H * slice;
      workgroups += (int64_t)p.B * p.H * ((slice + rows - 1) / rows);
    }
    if (workgroups > slots) continue;
    const int64_t room = slots * ((rows + kRowsInFlight - 1) / kRowsInFlight * kRowsInFlight);
    return steps * 100 >= room * 94 ? rows : kRowsPerThread;
  }
  return kRowsPerThread;
}

template <typename T>
static hipError_t run(QuantBatch& batch, hipStream_t stream) {
  const int per_thread = rows_per_thread<T>(batch);
  int cast_x = 1, reduce_x = 0, bh_max = 1;
  for (int i = 0; i < batch.n; i++) {
    QuantParams& p = batch.job[i];
    const int BH = p.B * p.H;
    const int rpb = 256 / (p.D >> 3);
    const int64_t rows = (int64_t)p.S + p.S2;
    int per_slice = (int)((rows + rpb * per_thread - 1) / (rpb * per_thread));
    if (per_slice < 1) per_slice = 1;
    if (per_slice > 2048) per_slice = 2048;
    p.cast_blocks = per_slice;
    p.reduce_blocks = 0;
    if (p.scale_in == nullptr) {
      if (p.partials != nullptr) {
        // one slot per workgroup: as many workgroups as the scratch holds slots for
        p.reduce_blocks = (int)(p.partial_slots / BH);
        if (p.reduce_blocks > per_slice) p.reduce_blocks = per_slice;
        if (p.reduce_blocks < 1) return hipErrorInvalidValue;
      } else {
        // every workgroup ends in one atomic max on its slice's entry: keep their number near 1024,
        // same-address atomics are served one at a time
        p.reduce_blocks = 1024 / BH;
        if (p.reduce_blocks < 1) p.reduce_blocks = 1;
        if (p.reduce_blocks > per_slice) p.reduce_blocks = per_slice;
        hipLaunchKernelGGL(fill_zero_kernel, dim3((BH + 255) / 256), dim3(256), 0, stream, p.amax, BH);
      }
    }
    if (p.cast_blocks > cast_x) cast_x = p.cast_blocks;
    if (p.reduce_blocks > reduce_x) reduce_x = p.reduce_blocks;
    if (BH > bh_max) bh_max = BH;
  }
  const dim3 block(256);
  if (reduce_x > 0) hipLaunchKernelGGL((absmax_kernel<T>), dim3(reduce_x, bh_max, batch.n), block, 0, stream, batch);
  hipLaunchKernelGGL((cast_kernel<T>), dim3(cast_x, bh_max, batch.n), block, 0, stream, batch);
  for (int i = 0; i < batch.n; i++) {
    const QuantParams& p = batch.job[i];
    if (p.scale_in == nullptr && p.partials == nullptr) {
      // per_tensor broadcasts entry 0: keep it to one workgroup so the barrier orders read/write
      const int BH = p.B * p.H;
      if (p.per_tensor && BH > 1024) return hipErrorInvalidValue;
      const int fb = p.per_tensor ? BH : 256;
      hipLaunchKernelGGL(finalize_kernel, dim3((BH + fb - 1) / fb), dim3(fb < 64 ? 64 : fb), 0, stream, p, BH);
    }
  }
  return hipGetLastError();
}

}  // namespace quant

hipError_t launch_fp8_quant(QuantBatch& b, int in_dtype, hipStream_t stream) {
  if (in_dtype == 0) return quant::run<__bf16>(b, stream);
  if (in_dtype == 1) return quant::run<_Float16>(b, stream);
  if (in_dtype == 2) return quant::run<float>(b, stream);
  return hipErrorInvalidValue;
}

}  // namespace xdit
