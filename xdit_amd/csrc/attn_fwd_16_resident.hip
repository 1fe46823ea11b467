// 16-bit attention forward over few keys (cross-attention on text tokens): every key and value of a (batch, head)
// stays in LDS, and the wavefronts of a workgroup run over query rows without meeting again.
//
// The kernel of attn_fwd_16_impl.h pays for every query tile what a long key range hides: the load of the
// first keys, a barrier per KV tile and the store of the rows, for two to eight KV tiles of products.  Here a workgroup
// loads the KV tiles of its head once (resident_walk.h deals it consecutive groups of 32 rows of that head), and after the
// one barrier behind that load each wavefront takes group after group by itself: the queries of the next group are on their
// way while it computes, and one wavefront's loads and stores run beside another's products.
// The arithmetic of a row is that of the tiled kernel, in the same order (TileMath), so the bits are the same.
//
// It is taken where it is expected to take less time (resident_path in api.hip).  us of a call with the tiled kernel and
// here (bf16): head_dim 128, 24 heads of 40000 rows on 77 / 120 keys 114 -> 99.7 / 118 -> 102, 40 of 32760 on 226 249 -> 218, 48 of 32760 on
// 77 202 -> 181; head_dim 72, 24 of 40000 on 120 97.8 -> 78.7 (BSHD memory 104 -> 84.7), 2 x 16 of 4096 on 120 16.7 -> 13.6; 88, 48 of
// 60000 on 120 336 -> 267; 96, 24 of 40000 on 256 144 -> 134; 64, 24 of 14933 on 512 61.4 -> 59.3.
// What is left (2 x 16 heads at 72 on 120 keys, eight workgroups a head): 11.9 us with one row group per wavefront (3072 rows),
// then 6.1 to 7.1 us for each further one (two to six: 19.0, 25.1, 32.1, 38.9, 46.0 us), in which 28 MB of rows come in and go out:
// 4.2 TB/s, near the rate of a copy.  So about five are the launch and the way of the keys and first queries.
#include "attn_fwd_16_impl.h"
#include "resident_walk.h"

namespace xdit {

// Output staging block of a wavefront: 16 rows of 64 columns (half the rows of the tiled kernel's, so that four
// KV tiles at head_dim 128 and eight at 64 fit beside it).
constexpr int kResidentStageRows = 16;
constexpr int kResidentStageBytes = kResidentStageRows * kStagePitchBytes;

template <int D, int NW>
constexpr int resident_lds_bytes(int nt) { return nt * TileGeom<D>::BUF_BYTES + NW * kResidentStageBytes; }

template <typename T, int D, int DC, int NW, bool PAD>
__global__ __launch_bounds__(64 * NW, NW == 12 ? 3 : 2) void attn_fwd_16_resident_kernel(const AttnParams p) {
  typedef TileGeom<D> G;
  typedef TileMath<T, D, DC> M;
  typedef typename Mfma16<T>::vec8 vec8;
  typedef __attribute__((ext_vector_type(4))) T vec4;
  constexpr int KSTEPS = M::KSTEPS, DBLOCKS = M::DBLOCKS;
  constexpr bool AHEAD = D == 64 || NW == 8;  // the next group's queries are requested a group ahead (there are registers for it)
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];  // nt KV tiles, then a staging block per wavefront

  ResidentPart part;
  if (!resident_part((int)blockIdx.x, p.tiles_per_xcd, p.total_tiles, p.nq_tiles, p.Sq, part)) return;
  const int b = part.bh / p.H, h = part.bh - b * p.H;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
  const int dact = PAD ? p.d_actual : D;
  const int nt1 = (p.Sk + kKeysPerTile - 1) / kKeysPerTile;
  const int nt = nt1 + (p.Sk2 + kKeysPerTile - 1) / kKeysPerTile;

  // Q fragments of row group g: lane (query l32, contraction half hh), as in the tiled kernel.
  const T* const q1 = (const T*)p.q + b * p.qs_b + h * p.qs_h;
  const T* const q2 = (const T*)p.q2 + b * p.q2s_b + h * p.q2s_h;
  auto load_queries = [&](int g, vec8 (&qf)[KSTEPS]) {
    const int qrow = 32 * g + l32;
    const int row = qrow < p.Sq ? qrow : p.Sq - 1;
    const T* at = row < p.Sq1 ? q1 + (int64_t)row * p.qs_s : q2 + (int64_t)(row - p.Sq1) * p.q2s_s;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      const int col = ks * 16 + hh * 8;
      qf[ks] = *(const vec8*)(at + (!PAD || col < dact ? col : 0));  // past the head_dim any 8 elements of the row: zeros take their place
    }
  };
  auto clear_pad_queries = [&](vec8 (&qf)[KSTEPS]) {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++)
      if (PAD && ks * 16 + hh * 8 >= dact) {
#pragma unroll
        for (int e = 0; e < 8; e++) qf[ks][e] = (T)0.f;
      }
  };
  vec8 qnext[KSTEPS];
  const int g_last = part.g1 - 1;
  load_queries(part.g0 + wave < g_last ? part.g0 + wave : g_last, qnext);

  // ---- all KV tiles: piece i (1 KiB of K and 1 KiB of V, see attn_tiles.h) by wavefront i % NW ----------
  {
    constexpr int LANES_PER_ROW = G::ROW_BYTES / 16;
    const unsigned colb = (lane % LANES_PER_ROW) * 16;
    const unsigned lds_base = (unsigned)(uintptr_t)(XDIT_LDS unsigned char*)smem;
    const unsigned kss1 = (unsigned)p.ks_s * 2, vss1 = (unsigned)p.vs_s * 2, kss2 = (unsigned)p.k2s_s * 2, vss2 = (unsigned)p.v2s_s * 2;  // below 2^24
    const unsigned char* const k1 = (const unsigned char*)((const T*)p.k + b * p.ks_b + h * p.ks_h);
    const unsigned char* const v1 = (const unsigned char*)((const T*)p.v + b * p.vs_b + h * p.vs_h);
    const unsigned char* const k2 = (const unsigned char*)((const T*)p.k2 + b * p.k2s_b + h * p.k2s_h);
    const unsigned char* const v2 = (const unsigned char*)((const T*)p.v2 + b * p.v2s_b + h * p.v2s_h);
    for (int i = wave; i < nt * G::NG; i += NW) {
      const int t = i / G::NG, g = i - t * G::NG;
      const bool second = t >= nt1;
      const int row0 = (second ? t - nt1 : t) * kKeysPerTile;
      const int left = (second ? p.Sk2 : p.Sk) - row0;
      const int last = (left < kKeysPerTile ? left : kKeysPerTile) - 1;
      int r = G::NG * (lane / LANES_PER_ROW) + g;
      r = r < last ? r : last;  // rows past the end of the segment re-read its last row
      const unsigned kss = second ? kss2 : kss1, vss = second ? vss2 : vss1;
      if (!PAD || colb < (unsigned)dact * 2) {  // lanes of columns the tensors do not have stay idle
        load_lds_16((second ? k2 : k1) + (uint64_t)(unsigned)row0 * kss, __umul24((unsigned)r, kss) + colb, lds_base + t * G::BUF_BYTES + g * G::K_PITCH);
        load_lds_16((second ? v2 : v1) + (uint64_t)(unsigned)row0 * vss, __umul24((unsigned)r, vss) + colb, lds_base + t * G::BUF_BYTES + G::K_BYTES + g * G::V_PITCH);
      }
    }
  }
  if (PAD) {  // K columns between the tensors' head_dim and the computed one meet zeros of Q and have to be finite
    typedef __attribute__((ext_vector_type(4))) int i32x4_;
    const i32x4_ zero = {0, 0, 0, 0};
    const int chunks = DC / 8 - dact / 8;
    for (int i = threadIdx.x; i < nt * kKeysPerTile * chunks; i += 64 * NW) {
      const int row = i % kKeysPerTile, rest = i / kKeysPerTile, t = rest / chunks, chunk = dact / 8 + rest - t * chunks;
      *(XDIT_LDS i32x4_*)((XDIT_LDS unsigned char*)smem + t * G::BUF_BYTES + (row % G::NG) * G::K_PITCH + (row / G::NG) * G::ROW_BYTES + chunk * 16) = zero;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const unsigned lds0 = (unsigned)(uintptr_t)(XDIT_LDS unsigned char*)smem;
  unsigned kaddr0 = M::k_read_address(lds0, l32, hh), vaddr0 = M::v_read_address(lds0, lane, hh);
  asm volatile("" : "+v"(kaddr0), "+v"(vaddr0));  // one register each through the loop
  XDIT_LDS unsigned char* const stage = (XDIT_LDS unsigned char*)smem + nt * G::BUF_BYTES + wave * kResidentStageBytes;
  const float c = p.scale * kLog2e;  // logits are kept in log2 units
  T* const obase = (T*)p.out + b * p.os_b + h * p.os_h;

  for (int g = part.g0 + wave; g < part.g1; g += NW) {
    vec8 qf[KSTEPS];
    if (!AHEAD && g != part.g0 + wave) load_queries(g, qnext);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      qf[ks] = qnext[ks];
      asm volatile("" : "+v"(qf[ks]));  // the loads are awaited here
    }
    if (AHEAD) load_queries(g + NW < part.g1 ? g + NW : g, qnext);
    clear_pad_queries(qf);

    float m_used = -INFINITY, l_part = 0.f;
    f32x16 oacc[DBLOCKS];
#pragma unroll
    for (int db = 0; db < DBLOCKS; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) oacc[db][i] = 0.f;
    int left = p.Sk;
    for (int t = 0; t < nt; t++) {
      if (t == nt1) left = p.Sk2;
      f32x16 sacc[2];
      M::logits(sacc, qf, kaddr0 + t * G::BUF_BYTES);
      if (left < kKeysPerTile) M::mask(sacc, left);
      const float mx = M::row_max(sacc);
      if (t == 0) {
        m_used = fmaxf(m_used, mx);  // -inf where all logits are NaN, as in the tiled kernel: a later tile may rescale the rows beside such a row
      } else {
        const float m_new = fmaxf(m_used, mx);
        const bool grow = (m_new - m_used) * c > kLazyRescaleLog2;
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
          const float alpha = fast_exp2((m_used - m_new) * c);
          m_used = m_new;
          l_part *= alpha;
#pragma unroll
          for (int db = 0; db < DBLOCKS; db++)
#pragma unroll
            for (int e = 0; e < 16; e++) oacc[db][e] *= alpha;
        }
      }
      vec8 pf[4];
      M::probabilities(sacc, c, m_used * c, l_part, pf);
      M::values(oacc, pf, vaddr0 + t * G::BUF_BYTES);
      left -= kKeysPerTile;
    }

    // ---- rows out, 16 of them and 64 columns at a time through the wavefront's staging block ----
    const float l_tot = sum_halves(l_part);
    const float inv = 1.0f / l_tot;
    const int row0 = 32 * g, rows_live = p.Sq - row0;  // at least 1
    const int rd_row = lane >> 3, rd_col = (lane & 7) * 8;
#pragma unroll
    for (int half = 0; half < (DBLOCKS + 1) / 2; half++) {
#pragma unroll
      for (int rows = 0; rows < 32; rows += kResidentStageRows) {
        if ((l32 & 16) == rows) {
#pragma unroll
          for (int dbl = 0; dbl < 2; dbl++) {
            const int db = 2 * half + dbl;
            if (db < DBLOCKS) {
#pragma unroll
              for (int a = 0; a < 4; a++) {
                // registers 4a..4a+3 are d = 32db + 8a + 4hh + 0..3 of this lane's query
                f32x4 o = {oacc[db][4 * a] * inv, oacc[db][4 * a + 1] * inv, oacc[db][4 * a + 2] * inv, oacc[db][4 * a + 3] * inv};
                *(XDIT_LDS vec4*)(stage + (l32 & 15) * kStagePitchBytes + (32 * dbl + 8 * a + 4 * hh) * 2) = __builtin_convertvector(o, vec4);
              }
            }
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < 2; r++) {
          // lanes past the last row store it again (the same bytes) instead of being masked: the number of stores
          // behind the next queries' loads is then known to the wait for these
          int row = rd_row + 8 * r;
          const int col = 64 * half + rd_col;
          const int here = rows_live - rows;   // rows of this block that exist
          if (here > 0) {
            row = row < here ? row : here - 1;
            const vec8 x = *(const XDIT_LDS vec8*)(stage + row * kStagePitchBytes + rd_col * 2);
            vec8* const at = (vec8*)(obase + (int64_t)(row0 + rows + row) * p.os_s + col);
            // Whole lines leave the cache as they are written; rows of head_dims that are no whole lines go out by
            // ordinary stores, which the cache puts together (48 heads of 60000 rows at 88: 429 -> 271 us)
            if (!PAD) __builtin_nontemporal_store(x, at);
            else if (col < dact) *at = x;
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
    if (p.lse != nullptr && hh == 0 && row0 + l32 < p.Sq) {
      float mc = m_used * c;
      asm volatile("" : "+v"(mc));  // rounded before the sum, as in the tiled kernel (where the loop has this product)
      p.lse[b * p.ls_b + h * p.ls_h + row0 + l32] = (mc + fast_log2(l_tot)) * kLn2;
    }
  }
}

template <typename T, int D, int DC, int NW, bool PAD>
static hipError_t launch_resident(const AttnParams& p, int nt, hipStream_t stream) {
  static std::atomic<bool> lds_ready[kMaxDevices];
  const int slot = current_device_slot();
  if (!lds_ready[slot].load(std::memory_order_relaxed)) {
    hipError_t e = hipFuncSetAttribute((const void*)attn_fwd_16_resident_kernel<T, D, DC, NW, PAD>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       resident_lds_bytes<D, NW>(kResidentTiles<D>));
    if (e != hipSuccess) return e;
    lds_ready[slot].store(true, std::memory_order_relaxed);
  }
  AttnParams q = p;
  q.nq_tiles = resident_parts(p.B * p.H, p.Sq, nt, NW, resident_cus(p.cu_count));
  q.total_tiles = p.B * p.H * q.nq_tiles;
  q.tiles_per_xcd = (q.total_tiles + 7) / 8;
  hipLaunchKernelGGL((attn_fwd_16_resident_kernel<T, D, DC, NW, PAD>), dim3((unsigned)q.tiles_per_xcd * 8), dim3(64 * NW), (resident_lds_bytes<D, NW>(nt)), stream, q);
  return hipGetLastError();
}

template <typename T>
static hipError_t launch_typed_resident(const AttnParams& p, int D, int nt, hipStream_t stream) {
  const int d = p.d_actual == D ? 0 : p.d_actual;
  AttnParams q = p;
  q.d_actual = d;
  // Computed over 80 columns twelve wavefronts are ahead of eight with the queries requested ahead (2 x 16 heads of 4096
  // on 120 keys 15.5 against 16.5 us, 24 of 40000 80.7 against 84), over 96 behind (24 of 40000 on 256 keys 141 against 138).
  if (D == 128) {
    if (d == 0) return launch_resident<T, 128, 128, resident_wavefronts(128), false>(q, nt, stream);
    if (d <= 80) return launch_resident<T, 128, 80, resident_wavefronts(80), true>(q, nt, stream);
    if (d <= 96) return launch_resident<T, 128, 96, resident_wavefronts(96), true>(q, nt, stream);
    if (d <= 112) return launch_resident<T, 128, 112, resident_wavefronts(112), true>(q, nt, stream);
    return launch_resident<T, 128, 128, resident_wavefronts(128), true>(q, nt, stream);
  }
  if (d == 0) return launch_resident<T, 64, 64, resident_wavefronts(64), false>(q, nt, stream);
  if (d <= 32) return launch_resident<T, 64, 32, resident_wavefronts(32), true>(q, nt, stream);
  return launch_resident<T, 64, 64, resident_wavefronts(64), true>(q, nt, stream);
}

hipError_t launch_attn_fwd_16_resident(const AttnParams& p, int dtype_is_fp16, int D, hipStream_t stream) {
  const int nt = (p.Sk + kKeysPerTile - 1) / kKeysPerTile + (p.Sk2 + kKeysPerTile - 1) / kKeysPerTile;
  return dtype_is_fp16 ? launch_typed_resident<_Float16>(p, D, nt, stream) : launch_typed_resident<__bf16>(p, D, nt, stream);
}

}  // namespace xdit
