// Non-causal attention forward for fp32 tensors on gfx950, any head_dim that is a multiple of 8 up to 128
// (e.g. 72), with fp32 accumulation.  (16-bit tensors of every such head_dim run on the 16-bit kernel.)  Same
// orientation as the 16-bit kernel:
//   S^T = K Q^T  (A = K rows, B = Q^T in registers),  O^T = V^T P^T  (B = P^T = the S^T registers).
// Two loops: split_loop runs the products on the bf16 matrix cores with operands split into three bf16
// values, and the loop in the kernel itself on the fp32 ones (v_mfma_f32_32x32x2_f32) for the values that the
// split has no room for.  The fp32 instruction runs at a sixteenth of the bf16 rate; six split products cost
// 3/8 of it.  2 x 16 heads of 4096 rows at head_dim 72: 1465 -> 964 us, 24 heads of 4608 at 128: 2625 -> 1646,
// 16 heads of 1024 at 72: 67 -> 53, one head of 39500 at 64: 5753 -> 3029 (same box); relative error against
// float64 1.26e-6 -> 2.8e-7, 1.37e-6 -> 3.1e-7, 5.2e-7 -> 1.8e-7, 3.9e-6 -> 7.9e-7, because a tile's products are
// summed by themselves before they are added to O^T (added one by one: 1.06e-6, 1.10e-6, 3.9e-7, 3.3e-6, at 930,
// 1651, 53, 3010 us).  Bound by the VALU work of splitting and softmax beside the MFMAs (busy 33 % with one
// wavefront per SIMD, 49 % with two, before the tile sums).
// In the fp32 loop, with a contraction depth of 2 per instruction every operand is ONE float per lane, so V^T
// is a plain LDS read (lanes along head_dim) and needs no transposing load.
//
// workgroup = 256 threads = 4 wavefronts, each with 32 query rows and 32 of the keys of a tile.
// KS = 1: four row groups (128 query rows) share tiles of 32 keys.  KS = 2: two row groups (64
// query rows), and the two wavefronts of a row group each take one half of every 64-key tile and
// fold their partial results through LDS at the end: twice the workgroups and wavefronts, for
// problems whose 128-row tiles would leave compute units idle (PixArt-512: 16 heads x 1024 rows
// are 128 such tiles for 256 compute units).  Every wavefront is bound by its own chain of MFMAs
// (64 cycles each), so what counts is how many SIMDs have one.
//
// In the fp32 loop K/V tiles are double buffered in LDS and filled by direct global->LDS loads (16 bytes
// per lane, one barrier per tile).  A tile is an array of 16-byte chunks in the order the loads write them:
// K rows of DP/4 + 1 chunks, V rows of DP/4 + 2 chunks (DP = head_dim rounded up to 32); the
// lanes of the chunks a row does not have stay idle.  The K pitch of DP + 4 floats makes the
// 16-byte fragment reads of 16 consecutive rows hit 64 different banks; the V pitch of DP + 8
// floats puts the rows that the two halves of a wavefront read (4 keys apart) 32 banks apart.
//
// The contraction index of the first product is permuted so that a lane's K operands of four
// consecutive steps are 16 contiguous bytes: step s of lane half hh is column 8(s/4) + 4hh + s%4.
#include "attn_split.h"
#include "launchers.h"

namespace xdit {

namespace f32path {

template <int D8, int KS> struct Geom {
  static constexpr int D = 8 * D8;
  static constexpr int DB = (D + 31) / 32;
  static constexpr int DP = 32 * DB;   // padded head_dim of the second product
  static constexpr int KCH = DP / 4 + 1;   // 16-byte chunks per K row in LDS
  static constexpr int VCH = DP / 4 + 2;   // ... per V row
  static constexpr int TK = 32 * KS;       // keys per tile
  static constexpr int RQ = 4 / KS;        // row groups (of 32 query rows) per workgroup
  static constexpr int ROWS = 32 * RQ;
  static constexpr int K_CHUNKS = TK * KCH;
  static constexpr int V_CHUNKS = TK * VCH;
  static constexpr int K_INSTR = (K_CHUNKS + 63) / 64;   // wavefront load instructions per K tile
  static constexpr int V_INSTR = (V_CHUNKS + 63) / 64;
  static constexpr int K_BYTES = K_INSTR * 1024;
  static constexpr int V_BYTES = V_INSTR * 1024;
  static constexpr int BUF_BYTES = K_BYTES + V_BYTES;
  // partial result of a wavefront for the fold between key halves: 16 DB + 2 floats per lane
  static constexpr int PART_BYTES = (16 * DB + 2) * 64 * 4;
  // split loop: three bf16 planes per tensor, rows of DS (K) and DP (V) columns
  static constexpr int KST = (D + 15) / 16;    // contraction steps of the first product
  static constexpr int SK_PITCH = 32 * KST + 16;                          // an odd number of 16-byte units
  static constexpr int SV_PITCH = DB == 1 ? 64 : (DB == 4 ? 320 : 192);   // +-64 modulo 256
  static constexpr int SK_PLANE = TK * SK_PITCH;
  static constexpr int SV_PLANE = TK * SV_PITCH;
  static constexpr int SBUF_BYTES = 3 * (SK_PLANE + SV_PLANE);
  static constexpr int SBUFS = 2 * SBUF_BYTES <= 159 * 1024 ? 2 : 1;
  static constexpr int TPR = 256 / TK;                      // threads that load a row
  static constexpr int CPT = (D / 4 + TPR - 1) / TPR;       // 16-byte chunks of a row per thread
  static constexpr int MAX2(int a, int b) { return a > b ? a : b; }
  static constexpr int LDS_BYTES = MAX2(MAX2(2 * BUF_BYTES, SBUFS * SBUF_BYTES), RQ * PART_BYTES);
};

// Two fp32 values as the sum of three bf16 values each, packed (first value in the low half): round to
// nearest, three times eight bits, so nothing of a value is left (short of underflow).
__device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& mid, unsigned& lo) {
  f32x2 v = {a, b};
  hi = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
  v[0] -= __uint_as_float(hi << 16);
  v[1] -= __uint_as_float(hi & 0xffff0000u);
  mid = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
  v[0] -= __uint_as_float(mid << 16);
  v[1] -= __uint_as_float(mid & 0xffff0000u);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
// A pointer that is the same in every lane, as the scalar the compiler does not prove it to be.
__device__ __forceinline__ const unsigned char* uniform(const unsigned char* x) {
  const uint64_t v = (uint64_t)x;
  return (const unsigned char*)(((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)v));
}
constexpr float kValueScale = 0x1p24f;  // of the V planes of the split loop
constexpr float kValueMost = 0x1p80f;   // of those, so that the sums of 2^31 of them times probabilities of up to 2^8 stay finite
constexpr float kDotMost = 0x1p120f;
__device__ __forceinline__ float max_abs(float m, float a, float b) { return fmaxf(fmaxf(m, fabsf(a)), fabsf(b)); }

// The KV loop on the bf16 matrix cores.  Every fp32 operand x is split into x0 + x1 + x2 (split2; |x1| is at
// most 2^-8 of x, |x2| 2^-17) and a product is x0 y0 + (x0 y1 + x1 y0) + (x0 y2 + x1 y1 + x2 y0): what is left
// out, x1 y2 + x2 y1 and less, is at most 2^-24 of the product (2^-24.04 seen over random operands), which is the
// rounding of an fp32 product, and the accumulation is in fp32: one rounding per 32 keys at the size of O^T
// instead of one per 2.  Six bf16 instructions of 32 cycles do the work of eight fp32 ones of 64.
// K and V tiles are split once per workgroup on their way into LDS (row-major planes; V^T is read
// transposed, as in the 16-bit kernel), Q once, P per tile in registers.
// The split has no room at the ends of fp32's range, and 0 x inf turns up where the plain product has
// none: false (results meaningless) if the largest magnitudes seen do not leave it that room; the caller
// then runs the fp32 loop.  NaN goes through as in the plain products.
// The pieces of an element below 2^-110 reach below bf16's smallest subnormal, where up to 2^-134 of it is lost.
//   V is multiplied by 2^24 on its way into the planes (and O^T by 2^-24 at the end), which leaves nothing of
//   what fp32 holds below that, whatever the other columns hold.
//   Q and K: the loop is used only where that puts no logit off by 2^-30, with a margin of 2^9 (which
//   covers an instruction that takes subnormals as zeros).
//   P: a probability below 2^-110 is off by up to 2^-134, and one below 2^-126 is zero, beside a row's sum
//   of at least 2^-8.
template <int D8, int KS>
__device__ __forceinline__ bool split_loop(const AttnParams& p, unsigned char* smem, int b, int h, int qrow_c, int rg, int ksl,
                                           float c, f32x16 (&oacc)[Geom<D8, KS>::DB], float& m_used, float& l_part) {
  typedef Geom<D8, KS> G;
  constexpr int D = G::D, DB = G::DB, TK = G::TK, KST = G::KST, TPR = G::TPR, CPT = G::CPT;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  XDIT_LDS unsigned char* const lds = (XDIT_LDS unsigned char*)smem;
  typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
  typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
  typedef __attribute__((ext_vector_type(8))) short s16x8;

  float mq = 0.f, mk = 0.f, mv = 0.f;  // largest magnitudes seen by this thread
  const float qk_limit = fminf(0x1p95f / (fabsf(c) * (float)D) - 4.f, kDotMost);   // of |q| + |k|
  bf16x8 qf[3][KST];
  const float* qptr = (const float*)p.q + b * p.qs_b + h * p.qs_h + (int64_t)qrow_c * p.qs_s + 8 * hh;
#pragma unroll
  for (int ks = 0; ks < KST; ks++) {
    u32x4 pl[3] = {};
    if (16 * ks + 8 * hh < D) {
      const f32x4 x0 = *(const f32x4*)(qptr + 16 * ks), x1 = *(const f32x4*)(qptr + 16 * ks + 4);
      const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        unsigned a, m, l;
        split2(x[2 * e], x[2 * e + 1], a, m, l);
        pl[0][e] = a; pl[1][e] = m; pl[2][e] = l;
        mq = max_abs(mq, x[2 * e], x[2 * e + 1]);
      }
    }
#pragma unroll
    for (int n = 0; n < 3; n++) qf[n][ks] = __builtin_bit_cast(bf16x8, pl[n]);
  }

  const int nt1 = (p.Sk + TK - 1) / TK;
  const int nt = nt1 + (p.Sk2 + TK - 1) / TK;
  const int row = tid / TPR, c0 = tid % TPR;   // this thread's row of every tile and its first chunk
  f32x4 kr[CPT], vr[CPT];
  // (in registers: selected from the kernel arguments per tile, they came through scratch memory and flat loads)
  const float* const kbase1 = (const float*)p.k + b * p.ks_b + h * p.ks_h;
  const float* const vbase1 = (const float*)p.v + b * p.vs_b + h * p.vs_h;
  const float* kbase2 = kbase1;
  const float* vbase2 = vbase1;
  const int kss1 = (int)p.ks_s, vss1 = (int)p.vs_s;  // below 2^24 bytes
  int kss2 = kss1, vss2 = vss1;
  if (p.Sk2 > 0) {
    kbase2 = (const float*)p.k2 + b * p.k2s_b + h * p.k2s_h;
    vbase2 = (const float*)p.v2 + b * p.v2s_b + h * p.v2s_h;
    kss2 = (int)p.k2s_s;
    vss2 = (int)p.v2s_s;
  }
  // Chunk n of this thread; past the end of the row the last one again (its loads and stores repeat).
  auto chunk = [&](int n) { const int cc = c0 + TPR * n; return (D / 4) % TPR == 0 || cc < D / 4 ? cc : D / 4 - 1; };
  auto load_tile = [&](int t) {
    const bool second = t >= nt1;
    const int row0 = (second ? t - nt1 : t) * TK;
    int r = row0 + row;
    const int last = (second ? p.Sk2 : p.Sk) - 1;
    r = r < last ? r : last;  // rows past the end of a KV segment re-read its last row (their logits are masked)
    const float* kp = (second ? kbase2 : kbase1) + (int64_t)r * (second ? kss2 : kss1);
    const float* vp = (second ? vbase2 : vbase1) + (int64_t)r * (second ? vss2 : vss1);
#pragma unroll
    for (int n = 0; n < CPT; n++) {
      const int cc = n + 1 < CPT ? c0 + TPR * n : chunk(n);
      kr[n] = *(const f32x4*)(kp + 4 * cc);
      vr[n] = *(const f32x4*)(vp + 4 * cc);
    }
  };
  // Piece i of splitting the loaded tile into buffer `buf`: one half of one 16-byte chunk, the stores with the
  // second half.  4 CPT pieces: K and V in turn.
  constexpr int PIECES = 4 * CPT;
  unsigned ph = 0, pm = 0, pl = 0;  // the first half of the chunk being split
  auto store_piece = [&](auto I, int buf) {
    constexpr int i = I, n = i / 4;
    constexpr bool is_v = (i / 2) % 2 != 0;
    constexpr int e = 2 * (i % 2);
    const f32x4 x = is_v ? vr[n] : kr[n];
    const float xa = is_v ? x[e] * kValueScale : x[e], xb = is_v ? x[e + 1] * kValueScale : x[e + 1];
    if (is_v) mv = max_abs(mv, xa, xb); else mk = max_abs(mk, xa, xb);
    if constexpr (i % 2 == 0) {
      split2(xa, xb, ph, pm, pl);
    } else {
      unsigned h1, m1, l1;
      split2(xa, xb, h1, m1, l1);
      const int cc = n + 1 < CPT ? c0 + TPR * n : chunk(n);
      const unsigned at = buf * G::SBUF_BYTES + (is_v ? 3 * G::SK_PLANE + row * G::SV_PITCH : row * G::SK_PITCH) + 8 * cc;
      constexpr int plane = is_v ? G::SV_PLANE : G::SK_PLANE;
      *(XDIT_LDS u32x2*)(lds + at) = u32x2{ph, h1};
      *(XDIT_LDS u32x2*)(lds + at + plane) = u32x2{pm, m1};
      *(XDIT_LDS u32x2*)(lds + at + 2 * plane) = u32x2{pl, l1};
    }
  };
  if constexpr (D % 16 != 0) {  // K columns past D meet zeros of Q: they have to be finite
    for (int i = tid; i < G::SBUFS * 3 * TK; i += 256) {
      const int buf = i / (3 * TK), r = i % (3 * TK);
      *(XDIT_LDS u32x4*)(lds + buf * G::SBUF_BYTES + r * G::SK_PITCH + 2 * D) = u32x4{0, 0, 0, 0};
    }
  }

  const unsigned kfrag = (32 * ksl + l32) * G::SK_PITCH + 16 * hh;
  // V^T fragments as in the 16-bit kernel: lane (group g = lane / 16, s = lane % 16) points at key 4hh + s/4
  // (+ 8rd + 16j), columns 32db + 16 (g % 2) + 4 (s % 4)
  const unsigned vfrag = 3 * G::SK_PLANE + (32 * ksl + 4 * hh + ((lane & 15) >> 2)) * G::SV_PITCH + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;

  load_tile(0);
  if constexpr (G::SBUFS == 2) {
    static_for<PIECES>([&](auto I) { store_piece(I, 0); });
    load_tile(nt > 1 ? 1 : 0);
  }
  for (int t = 0; t < nt; t++) {
    const int buf = G::SBUFS == 2 ? t & 1 : 0;
    __syncthreads();  // two buffers: tile t is there and nobody reads the other buffer; one: nobody reads it any more
    if constexpr (G::SBUFS == 1) {
      static_for<PIECES>([&](auto I) { store_piece(I, 0); });
      load_tile(t + 1 < nt ? t + 1 : t);
      __syncthreads();
    }
    const XDIT_LDS unsigned char* const base = lds + buf * G::SBUF_BYTES;

    // S^T = K Q^T : 32 keys x 32 queries; the small products in an accumulator of their own.  With two buffers the
    // next tile is split between the MFMAs: a wavefront issues in order, so VALU work runs beside the matrix
    // pipe only if it stands between two MFMAs.
    f32x16 sacc, low;
#pragma unroll
    for (int i = 0; i < 16; i++) sacc[i] = low[i] = 0.f;
    {
      bf16x8 kf[2][3];
#pragma unroll
      for (int n = 0; n < 3; n++) kf[0][n] = *(const XDIT_LDS bf16x8*)(base + kfrag + n * G::SK_PLANE);
      static_for<6 * KST>([&](auto I) {
        constexpr int i = I, ks = i / 6, op = i % 6;
        if constexpr (op == 0 && ks + 1 < KST) {
#pragma unroll
          for (int n = 0; n < 3; n++) kf[(ks + 1) % 2][n] = *(const XDIT_LDS bf16x8*)(base + kfrag + n * G::SK_PLANE + 32 * (ks + 1));
        }
        constexpr int kn = op == 0 ? 2 : (op == 3 || op == 4 ? 1 : 0);   // lo hi, hi hi, hi lo, mid mid, mid hi, hi mid
        constexpr int qn = op == 2 ? 2 : (op == 3 || op == 5 ? 1 : 0);
        if constexpr (op == 1) sacc = Mfma16<__bf16>::mma(kf[ks % 2][kn], qf[qn][ks], sacc);
        else low = Mfma16<__bf16>::mma(kf[ks % 2][kn], qf[qn][ks], low);
        if constexpr (G::SBUFS == 2) {
          constexpr int first = i * PIECES / (6 * KST), past = (i + 1) * PIECES / (6 * KST);
          static_for<past - first>([&](auto J) { store_piece(std::integral_constant<int, first + J>{}, buf ^ 1); });
          __builtin_amdgcn_sched_barrier(0);
        }
      });
    }
    if constexpr (G::SBUFS == 2) load_tile(t + 2 < nt ? t + 2 : nt - 1);
    const int valid = ((t < nt1) ? p.Sk - t * TK : p.Sk2 - (t - nt1) * TK) - 32 * ksl;  // keys of this wavefront's slice
    if (valid <= 0) continue;
#pragma unroll
    for (int i = 0; i < 16; i++) sacc[i] += low[i];
    if (valid < 32) {
      asm volatile("");  // a branch, not a select per element on every tile
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int key = 8 * (i >> 2) + 4 * hh + (i & 3);
        if (key >= valid) sacc[i] = -INFINITY;
      }
    }
    float mx = sacc[0];
#pragma unroll
    for (int i = 1; i < 16; i++) mx = fmaxf(mx, sacc[i]);
    mx = max_halves(mx);
    const float m_new = fmaxf(m_used, mx);
    const bool grow = (m_new - m_used) * c > kLazyRescaleLog2;  // true on the first tile (-inf)
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float alpha = fast_exp2((m_used - m_new) * c);  // 0 on the first tile
      m_used = m_new;
      l_part *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
    }
    const float mc = m_used * c;
    // P^T as B operands: plane n, key step j (16 keys): registers 8j .. 8j+7 of S^T.  Results below 2^-126 are zero:
    // the row's sum is at least 2^-8.
    u32x4 pf[3][2];
    float l_tile = 0.f;  // summed by itself: one rounding at the size of the row's sum per tile
    auto probabilities = [&](int j, int e) {
      const float p0 = fast_exp2(__builtin_fmaf(sacc[8 * j + 2 * e], c, -mc)), p1 = fast_exp2(__builtin_fmaf(sacc[8 * j + 2 * e + 1], c, -mc));
      l_tile += p0 + p1;
      unsigned a, m, l;
      split2(p0, p1, a, m, l);
      pf[0][j][e] = a; pf[1][j][e] = m; pf[2][j][e] = l;
    };
#pragma unroll
    for (int e = 0; e < 4; e++) probabilities(0, e);
    // O^T += V^T P^T.  A tile's products are summed by themselves, small ones first, and added once: O^T grows
    // with the number of keys and every addition to it rounds at its size.  The second key step's probabilities
    // stand between the first MFMAs, the additions of one block of columns between the next one's.
    {
      bf16x8 vf[2][3];
      auto read_v = [&](int g, int n) {
        const XDIT_LDS unsigned char* at = base + vfrag + n * G::SV_PLANE + 16 * (g % 2) * G::SV_PITCH + 64 * (g / 2);
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((XDIT_LDS s16x4*)at);
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((XDIT_LDS s16x4*)(at + 8 * G::SV_PITCH));
        vf[g % 2][n] = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      };
#pragma unroll
      for (int n = 0; n < 3; n++) read_v(0, n);
      // One sum or two, by measurement: with two wavefronts per SIMD head_dims 72 to 96 leave a few registers over 256
      // to scratch memory either way (14 to 22).  16 heads of 4000 at head_dim 88, 96: 535, 536 us with two, 524, 528 with
      // one; at 72, 80: 487, 489 with two, 491 to 499, 489 with one; 2 heads of 37000 at 72, 80: 6325, 6375 with two,
      // 6460, 6425 with one.
      constexpr int NS = KS == 1 && (D8 == 11 || D8 == 12) ? 1 : 2;
      f32x16 sum[NS];
      static_for<12 * DB>([&](auto I) {
        constexpr int i = I, g = i / 6, op = i % 6, db = g / 2, j = g % 2;
        if constexpr (op == 0 && g + 1 < 2 * DB) {
#pragma unroll
          for (int n = 0; n < 3; n++) read_v(g + 1, n);
        }
        if constexpr (op == 0 && j == 0) {
#pragma unroll
          for (int e = 0; e < 16; e++) sum[db % NS][e] = 0.f;
        }
        constexpr int vn = op == 0 ? 2 : (op == 2 || op == 3 ? 1 : 0);   // lo hi, hi lo, mid mid, mid hi, hi mid, hi hi
        constexpr int pn = op == 1 ? 2 : (op == 2 || op == 4 ? 1 : 0);
        sum[db % NS] = Mfma16<__bf16>::mma(vf[g % 2][vn], __builtin_bit_cast(bf16x8, pf[pn][j]), sum[db % NS]);
        if constexpr (g == 0) {
          constexpr int first = i * 4 / 6, past = (i + 1) * 4 / 6;
          static_for<past - first>([&](auto J) { probabilities(1, first + J); });
          __builtin_amdgcn_sched_barrier(0);
        } else if constexpr (NS == 2 && db > 0 && j == 0 && op >= 2) {
#pragma unroll
          for (int e = 4 * (op - 2); e < 4 * (op - 1); e++) oacc[db - 1][e] += sum[(db - 1) % NS][e];
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (j == 1 && op == 5 && (NS == 1 || db == DB - 1)) {
#pragma unroll
          for (int e = 0; e < 16; e++) oacc[db][e] += sum[db % NS][e];
        }
      });
    }
    l_part += l_tile;
  }

  // did the split have room?  The largest magnitudes of Q and K in [2^-90, 2^120) (or zero throughout) and within
  // the limit on what their small elements lose, that of V as split below 2^80 and the dot products below 2^120
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mq = fmaxf(mq, __shfl_xor(mq, off));
    mk = fmaxf(mk, __shfl_xor(mk, off));
    mv = fmaxf(mv, __shfl_xor(mv, off));
  }
  __shared__ float seen[4][3];
  if (lane == 0) { seen[tid >> 6][0] = mq; seen[tid >> 6][1] = mk; seen[tid >> 6][2] = mv; }
  __syncthreads();  // also: the tile buffers are no longer read
#pragma unroll
  for (int w = 0; w < 4; w++) { mq = fmaxf(mq, seen[w][0]); mk = fmaxf(mk, seen[w][1]); mv = fmaxf(mv, seen[w][2]); }
#pragma unroll
  for (int db = 0; db < DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) oacc[db][i] *= 1.f / kValueScale;
  auto room = [](float m) { return m == 0.f || m >= 0x1p-90f; };
  const bool ok = room(mq) && room(mk) && mq + mk < qk_limit && mv < kValueMost && mq * mk * (float)D < kDotMost;
  return __builtin_amdgcn_readfirstlane((int)ok) != 0;  // the same for the whole workgroup
}

// FUSED: the ring step; the block is folded into the fp32 accumulator (p.acc_out, p.acc_lse) with
// the arithmetic of the merge kernel instead of being written out.
template <int D8, int KS, bool FUSED>
__global__ __launch_bounds__(256, KS == 1 && D8 <= 12 ? 2 : 1) void attn_fwd_f32_kernel(const AttnParams p) {
  typedef Geom<D8, KS> G;
  constexpr int D = G::D, DB = G::DB, TK = G::TK, RQ = G::RQ;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hh = lane >> 5;
  const int rg = wave % RQ;    // row group of this wavefront
  const int ksl = wave / RQ;   // which 32 keys of a tile it takes

  const int tile = xcd_tile_index(blockIdx.x, p.tiles_per_xcd);
  if (tile >= p.total_tiles) return;
  const int bh = tile / p.nq_tiles;
  const int qt = tile - bh * p.nq_tiles;
  const int b = bh / p.H;
  const int h = bh - b * p.H;

  const int qrow = qt * G::ROWS + rg * 32 + l32;
  const int qrow_c = qrow < p.Sq ? qrow : p.Sq - 1;
  const float c = p.scale * kLog2e;
  float m_used;   // running (lazily updated) row maximum of the raw dot products
  float l_part;
  f32x16 oacc[DB];
  auto clear = [&] {
    m_used = -INFINITY;
    l_part = 0.f;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = 0.f;
  };
  clear();

  if (!split_loop<D8, KS>(p, smem, b, h, qrow_c, rg, ksl, c, oacc, m_used, l_part)) {
  clear();
  // Q^T fragments: lane (query l32, half hh) holds Q[query][8j + 4hh + i] as step 4j + i.
  const float* qptr = (const float*)p.q + b * p.qs_b + h * p.qs_h + (int64_t)qrow_c * p.qs_s + 4 * hh;
  f32x4 qf[D8];
#pragma unroll
  for (int j = 0; j < D8; j++) qf[j] = *(const f32x4*)(qptr + 8 * j);

  const unsigned char* kbase1 = (const unsigned char*)((const float*)p.k + b * p.ks_b + h * p.ks_h);
  const unsigned char* vbase1 = (const unsigned char*)((const float*)p.v + b * p.vs_b + h * p.vs_h);
  const unsigned char* kbase2 = p.Sk2 > 0 ? (const unsigned char*)((const float*)p.k2 + b * p.k2s_b + h * p.k2s_h) : kbase1;
  const unsigned char* vbase2 = p.Sk2 > 0 ? (const unsigned char*)((const float*)p.v2 + b * p.v2s_b + h * p.v2s_h) : vbase1;
  const unsigned kss1 = (unsigned)p.ks_s * 4, vss1 = (unsigned)p.vs_s * 4;
  const unsigned kss2 = p.Sk2 > 0 ? (unsigned)p.k2s_s * 4 : kss1, vss2 = p.Sk2 > 0 ? (unsigned)p.v2s_s * 4 : vss1;
  const int nt1 = (p.Sk + TK - 1) / TK;
  const int nt = nt1 + (p.Sk2 + TK - 1) / TK;
  const unsigned lds_base = (unsigned)(uintptr_t)(XDIT_LDS unsigned char*)smem;

  // Loads KV tile t into buffer `buf`: load instruction n of a tile (n = wave, wave + 4, ...)
  // writes chunks 64n .. 64n+63; chunk x is row x / CH, 16-byte column x % CH.  Rows past the end
  // of a KV segment re-read its last row (their logits are masked, their P is exactly zero).
  auto issue_tile = [&](int t, int buf) {
    const bool second = t >= nt1;
    const unsigned row0 = (unsigned)(second ? t - nt1 : t) * TK;
    const unsigned kss = second ? kss2 : kss1, vss = second ? vss2 : vss1;
    const unsigned char* kp = (second ? kbase2 : kbase1) + (uint64_t)row0 * kss;
    const unsigned char* vp = (second ? vbase2 : vbase1) + (uint64_t)row0 * vss;
    const int left = (second ? p.Sk2 : p.Sk) - (int)row0;
    const int last = (left < TK ? left : TK) - 1;
    const unsigned bo = lds_base + buf * G::BUF_BYTES;
#pragma unroll
    for (int n = 0; n < (G::K_INSTR + 3) / 4; n++) {
      const int instr = 4 * n + wave;
      const int x = instr * 64 + lane;
      int r = x / G::KCH;
      const int cchunk = x - r * G::KCH;
      r = r < last ? r : last;
      if (instr < G::K_INSTR && x < G::K_CHUNKS && cchunk < D / 4)
        load_lds_16(uniform(kp), (unsigned)r * kss + cchunk * 16, bo + instr * 1024);
    }
#pragma unroll
    for (int n = 0; n < (G::V_INSTR + 3) / 4; n++) {
      const int instr = 4 * n + wave;
      const int x = instr * 64 + lane;
      int r = x / G::VCH;
      const int cchunk = x - r * G::VCH;
      r = r < last ? r : last;
      if (instr < G::V_INSTR && x < G::V_CHUNKS && cchunk < D / 4)
        load_lds_16(uniform(vp), (unsigned)r * vss + cchunk * 16, bo + G::K_BYTES + instr * 1024);
    }
  };

  issue_tile(0, 0);
  for (int t = 0; t < nt; t++) {
    const int buf = t & 1;
    // tile t has landed (this thread's loads, after the barrier everyone's), and every wavefront
    // is done reading the other buffer, which the next tile now overwrites
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + 1 < nt) issue_tile(t + 1, buf ^ 1);

    const int valid = ((t < nt1) ? p.Sk - t * TK : p.Sk2 - (t - nt1) * TK) - 32 * ksl;  // keys of this wavefront's slice
    if (valid <= 0) continue;
    const XDIT_LDS unsigned char* kt = (const XDIT_LDS unsigned char*)smem + buf * G::BUF_BYTES;
    const XDIT_LDS unsigned char* vt = kt + G::K_BYTES;

    // S^T = K Q^T : 32 keys x 32 queries
    f32x16 sacc;
#pragma unroll
    for (int i = 0; i < 16; i++) sacc[i] = 0.f;
    const XDIT_LDS unsigned char* krow = kt + ((32 * ksl + l32) * G::KCH + hh) * 16;
#pragma unroll
    for (int j = 0; j < D8; j++) {
      const f32x4 kf = *(const XDIT_LDS f32x4*)(krow + 32 * j);
#pragma unroll
      for (int i = 0; i < 4; i++) sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[i], qf[j][i], sacc, 0, 0, 0);
    }
    if (valid < 32) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int key = 8 * (i >> 2) + 4 * hh + (i & 3);
        if (key >= valid) sacc[i] = -INFINITY;
      }
    }
    float mx = sacc[0];
#pragma unroll
    for (int i = 1; i < 16; i++) mx = fmaxf(mx, sacc[i]);
    mx = max_halves(mx);
    const float m_new = fmaxf(m_used, mx);
    const bool grow = (m_new - m_used) * c > kLazyRescaleLog2;  // true on the first tile (-inf)
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float alpha = fast_exp2((m_used - m_new) * c);  // 0 on the first tile
      m_used = m_new;
      l_part *= alpha;
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[db][i] *= alpha;
    }
    const float mc = m_used * c;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      sacc[i] = exp2f(__builtin_fmaf(sacc[i], c, -mc));
      l_part += sacc[i];
    }
    // O^T += V^T P^T : register i of P^T is keys {8(i/4) + i%4, +4} for the two lane halves
    const XDIT_LDS float* vcol = (const XDIT_LDS float*)(vt + (32 * ksl + 4 * hh) * G::VCH * 16) + l32;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int key = 8 * (i >> 2) + (i & 3);
#pragma unroll
      for (int db = 0; db < DB; db++) {
        const float vf = vcol[key * G::VCH * 4 + 32 * db];
        oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf, sacc[i], oacc[db], 0, 0, 0);
      }
    }
  }
  }

  if constexpr (KS > 1) {
    // fold the partial results of the key halves of a row group: the wavefronts of the second half
    // leave theirs in LDS ([value][lane], so that lanes write and read consecutive floats)
    __syncthreads();  // the tile buffers are no longer read
    XDIT_LDS float* part = (XDIT_LDS float*)smem + rg * (G::PART_BYTES / 4) + lane;
    if (ksl != 0) {
#pragma unroll
      for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) part[(16 * db + i) * 64] = oacc[db][i];
      part[16 * DB * 64] = m_used;
      part[(16 * DB + 1) * 64] = l_part;
    }
    __syncthreads();
    if (ksl != 0) return;
    const float m1 = part[16 * DB * 64], l1 = part[(16 * DB + 1) * 64];
    const float m = fmaxf(m_used, m1);   // m_used is finite: the first half of tile 0 holds key 0
    const float a0 = fast_exp2((m_used - m) * c), a1 = fast_exp2((m1 - m) * c);  // a1 = 0 for a half that saw no key
    m_used = m;
    l_part = l_part * a0 + l1 * a1;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = oacc[db][i] * a0 + part[(16 * db + i) * 64] * a1;
  }

  const float l_tot = sum_halves(l_part);
  const float inv = 1.0f / l_tot;
  const float lse = (m_used * c + log2f(l_tot)) * kLn2;
  if (qrow >= p.Sq) return;
  if constexpr (!FUSED) {
    float* optr = (float*)p.out + b * p.os_b + h * p.os_h + (int64_t)qrow * p.os_s;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const int d = 32 * db + 8 * a + 4 * hh;   // registers 4a..4a+3 are d .. d+3 of this lane's query
        if (d < D) {
          const f32x4 o = {oacc[db][4 * a] * inv, oacc[db][4 * a + 1] * inv, oacc[db][4 * a + 2] * inv, oacc[db][4 * a + 3] * inv};
          *(f32x4*)(optr + d) = o;
        }
      }
    if (p.lse != nullptr && hh == 0) p.lse[b * p.ls_b + h * p.ls_h + qrow] = lse;
  } else {
    // ring step: the arithmetic of the merge kernel on this block (fp32, so nothing is rounded in
    // between); both halves of the wavefront read the row's log-sum-exp before one of them
    // overwrites it (program order within the wavefront)
    const bool first = p.acc_first != 0;
    float* alp = p.acc_lse + b * p.al_b + h * p.al_h + (int64_t)qrow * p.al_s;
    float w = 0.f, new_lse = lse;
    if (!first) {
      const float la = *alp;
      w = sigmoid(lse - la);
      new_lse = la - log_sigmoid(la - lse);
    }
    float* aptr = p.acc_out + b * p.ao_b + h * p.ao_h + (int64_t)qrow * p.ao_s;
    float* optr = p.out != nullptr ? (float*)p.out + b * p.os_b + h * p.os_h + (int64_t)qrow * p.os_s : nullptr;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const int d = 32 * db + 8 * a + 4 * hh;
        if (d < D) {
          f32x4 m = {oacc[db][4 * a] * inv, oacc[db][4 * a + 1] * inv, oacc[db][4 * a + 2] * inv, oacc[db][4 * a + 3] * inv};
          if (!first) {
            const f32x4 acc = *(const f32x4*)(aptr + d);
#pragma unroll
            for (int e = 0; e < 4; e++) m[e] = fold_value(acc[e], m[e], w);
          }
          if (p.acc_store) *(f32x4*)(aptr + d) = m;
          if (optr != nullptr) *(f32x4*)(optr + d) = m;
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (hh == 0) {
      *alp = new_lse;
      if (p.lse != nullptr) p.lse[b * p.ls_b + h * p.ls_h + qrow] = new_lse;
    }
  }
}

template <int D8, int KS, bool FUSED>
static hipError_t launch_kernel(const AttnParams& q, dim3 grid, hipStream_t stream) {
  typedef Geom<D8, KS> G;
  static std::atomic<bool> lds_ready[kMaxDevices];
  const int slot = current_device_slot();
  if (G::LDS_BYTES > 65536 && !lds_ready[slot].load(std::memory_order_relaxed)) {  // > 64 KiB of dynamic LDS must be enabled once per kernel and device
    hipError_t e = hipFuncSetAttribute((const void*)attn_fwd_f32_kernel<D8, KS, FUSED>, hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS_BYTES);
    if (e != hipSuccess) return e;
    lds_ready[slot].store(true, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL((attn_fwd_f32_kernel<D8, KS, FUSED>), grid, dim3(256), G::LDS_BYTES, stream, q);
  return hipGetLastError();
}

template <int D8, int KS, bool FUSED>
static hipError_t launch_d(const AttnParams& q, int d8, dim3 grid, hipStream_t stream) {
  if constexpr (D8 <= 16) {
    if (d8 == D8) return launch_kernel<D8, KS, FUSED>(q, grid, stream);
    return launch_d<D8 + 1, KS, FUSED>(q, d8, grid, stream);
  } else {
    return hipErrorInvalidValue;
  }
}

}  // namespace f32path

// Query rows per workgroup: 128, or 64 with the keys of a tile split between two wavefronts when
// 128-row tiles would leave more than a quarter of the compute units without a workgroup.
// (Smaller workgroups without the key split were measured and do not help: PixArt-512 fp32,
// 16 x 1024 rows: 136 / 140 / 156 us at 128 / 64 / 32 rows, since the number of wavefronts, each
// bound by its own chain of MFMAs, stays the same.)
int attn_fwd_f32_rows(const AttnParams& p) {
  const int64_t tiles128 = (int64_t)p.B * p.H * ((p.Sq + 127) / 128);
  return tiles128 * 4 < (int64_t)resident_cus(p.cu_count) * 3 ? 64 : 128;
}

hipError_t launch_attn_fwd_f32(const AttnParams& p, int D, hipStream_t stream) {
  if (D <= 0 || D % 8 != 0 || D > 128) return hipErrorInvalidValue;
  AttnParams q = p;
  const int rows = attn_fwd_f32_rows(p);
  q.nq_tiles = (p.Sq + rows - 1) / rows;
  q.total_tiles = p.B * p.H * q.nq_tiles;
  q.tiles_per_xcd = (q.total_tiles + 7) / 8;
  dim3 grid(q.tiles_per_xcd * 8);
  const bool fused = p.acc_out != nullptr;
  if (rows == 64) return fused ? f32path::launch_d<1, 2, true>(q, D / 8, grid, stream) : f32path::launch_d<1, 2, false>(q, D / 8, grid, stream);
  return fused ? f32path::launch_d<1, 1, true>(q, D / 8, grid, stream) : f32path::launch_d<1, 1, false>(q, D / 8, grid, stream);
}

}  // namespace xdit
