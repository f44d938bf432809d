// Attention kernels for gfx950.
//
// flash_kernel: flash-style multi-head attention on v_mfma_f32_16x16x32_bf16 with an
//   online softmax. A workgroup of NW waves serves one (frame, head) and NW blocks of
//   16 queries; K and V^T for 64-key chunks are staged in LDS and shared by the waves.
//   The scores are computed transposed (S^T = K Q^T) so that every lane's scores all
//   belong to one query (lane & 15): the running max/sum and the rescale of the output
//   accumulators need only lane-group reductions, and the probabilities feed the
//   P V product (as O^T = V^T P^T) straight from registers without an LDS round trip.
//   Used for sequences of up to 64 and for the reference's sdpa / sdpa_causal surface with an additive
//   bias, a causal mask or fp32 operands.
//
// flash_ring_kernel: the same products without bias and mask on bf16, K and V staged as they lie:
//   spatial attention (144 tokens per frame), the VAE (576 tokens) and the sdpa surface.
//
// temporal_kernel: causal attention over the T frames of one (stream, position, head)
//   group. At T=2 each group is 2 queries x 2 keys, far below an MFMA tile, so it is a
//   VALU kernel: 16 lanes per group, 4 head dims per lane, dot products by 16-lane
//   butterfly reductions and an online softmax over the causal keys.
#include <type_traits>

#include "oasis_common.h"

namespace {

constexpr int KPITCH = 64 + 8;
constexpr float LOG2E = 1.4426950408889634f;

template <typename T>
__device__ __forceinline__ bf16x8 load8_bf16(const T* p);
template <>
__device__ __forceinline__ bf16x8 load8_bf16<bf16>(const bf16* p) {
  return *reinterpret_cast<const bf16x8*>(p);
}
template <>
__device__ __forceinline__ bf16x8 load8_bf16<float>(const float* p) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p);
  const f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
  float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return pack8(v);
}

// 8 consecutive K / V elements at element offset e of a (frame, head) block: bf16 blocks through a
// buffer resource (scalar base, 32-bit lane offset), which stages faster than 64-bit addresses
template <typename T>
__device__ __forceinline__ bf16x8 load8_kv(__amdgpu_buffer_rsrc_t r, const T* base, int e);
template <>
__device__ __forceinline__ bf16x8 load8_kv<bf16>(__amdgpu_buffer_rsrc_t r, const bf16*, int e) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, (uint32_t)e * 2, 0, 0));
}
template <>
__device__ __forceinline__ bf16x8 load8_kv<float>(__amdgpu_buffer_rsrc_t, const float* base, int e) {
  return load8_bf16<float>(base + e);
}

template <typename T>
__device__ __forceinline__ void store4(T* p, float a, float b, float c, float d);
template <>
__device__ __forceinline__ void store4<bf16>(bf16* p, float a, float b, float c, float d) {
  *reinterpret_cast<bf16x4*>(p) = bf16x4{f2bf(a), f2bf(b), f2bf(c), f2bf(d)};
}
template <>
__device__ __forceinline__ void store4<float>(float* p, float a, float b, float c, float d) {
  *reinterpret_cast<f32x4*>(p) = f32x4{a, b, c, d};
}

struct AttnArgs {
  int Lq, Lk;
  int64_t q_bh, kv_bh;      // element stride between (frame, head) blocks of Q and K/V
  float scale_log2;         // softmax scale * log2(e)
  const float* bias;        // [Lq, Lk] or nullptr
  int causal;
  int H;                    // heads per frame (output addressing)
  // out offset of query i, dim d of block bh: with f = bh / H, h = bh % H,
  // (f / f_inner) * o_sfo + (f % f_inner) * o_sf + h * o_sh + i * o_si + d
  int f_inner;
  int64_t o_sfo, o_sf, o_sh, o_si;
  // > 0: the output is a token-major [rows, frag_ks * 32] matrix stored in MFMA fragment order
  // (bf16): the row-major offset above names the element
  int frag_ks = 0;
  // byte ranges read by the grid slice blockIdx.z == 1 (launched when any is set)
  oasis::Prefetch pf = {{nullptr, nullptr, nullptr, nullptr}, {0, 0, 0, 0}, 7};
  // set: the output goes out as fp8 activation blocks instead (e4m3 bytes at o8 + the row-major
  // offset, the e8m0 scale of each 32-column block at o8s + offset / 32), the bf16-rounded values
  // quantized as oasis_quantize_act_fp8 would; the row-major offsets are multiples of 64 there
  uint8_t* o8 = nullptr;
  uint8_t* o8s = nullptr;
};

// Four consecutive bf16-rounded outputs r of a 32-column block whose max |v| over the block is
// amax -> e4m3 bytes (a u32) at q, and the block's e8m0 scale byte at *sc when sc is set.
__device__ __forceinline__ void store_fp8x4(uint8_t* q, uint8_t* sc, const float* r, float amax) {
  const int sb = fp8_block_scale(amax);
  const float inv = fp8_block_inv(sb);
  *reinterpret_cast<uint32_t*>(q) = pack4_fp8(r[0] * inv, r[1] * inv, r[2] * inv, r[3] * inv);
  if (sc) *sc = (uint8_t)sb;
}

// One query's output in the O^T accumulators of its 4 lanes (o[dt][i]: dim 16 dt + 4 g + i of the head, times
// inv), at row-major element offset off: as T, in fragment order, or as fp8 activation blocks. Called by all 4
// lanes (the ones that share lane % 16) of a query together.
template <typename T>
__device__ __forceinline__ void store_head(T* O, int64_t off, const f32x4* o, float inv, int g, int frag_ks,
                                           uint8_t* o8, uint8_t* o8s) {
  if (o8) {
    // dims 0..31 of the head are o[0..1] of the 4 lanes (lane groups g), 32..63 o[2..3]
    float r[4][4], m[2] = {0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[dt][i] = bf2f(f2bf(o[dt][i] * inv));
        m[dt >> 1] = fmaxf(m[dt >> 1], fabsf(r[dt][i]));
      }
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) m[h2] = max_xor32(max_xor16(m[h2]));
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const int64_t e = off + dt * 16 + 4 * g;
      store_fp8x4(o8 + e, (g == 0 && (dt & 1) == 0) ? o8s + e / 32 : nullptr, r[dt], m[dt >> 1]);
    }
    return;
  }
  const int64_t ocols = (int64_t)frag_ks * 32, orow = frag_ks ? off / ocols : 0;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) {
    const int d = dt * 16 + 4 * g;
    T* dst = frag_ks ? O + frag_index(orow, off - orow * ocols + d, frag_ks) : O + off + d;
    store4<T>(dst, o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
  }
}

// KS keys are staged in LDS at a time (K rows and V^T columns; KS >= Lk stages the whole
// sequence once, with no barrier in the key loop) and consumed in KC-key chunks.
// V^T is built from 8x8 blocks: a thread loads 8 key rows x 8 dims and transposes them in
// registers. Each V^T row (one head dim) holds its keys in k-slot order: within a 32-key
// block, position 8g + j holds the key that k-slot j of lane group g multiplies in the P V
// product (key 4g + j for j < 4, 16 + 4g + j - 4 for j >= 4), so a V fragment is one
// 16-byte LDS read. The 16-byte units of a row are XOR-swizzled by (row >> 3) & 7 within
// each 64-key group: the 8-byte staging writes of 8 dims x the same keys (rows 8 apart) and
// the fragment reads of 8 consecutive rows then fall in distinct LDS banks.
// KSPLIT = 2: two waves per 16-query block, each taking every other key chunk (two waves
// per SIMD, half the serial softmax chain each); their running (max, sum, output) states
// are merged through LDS at the end.
// PLAIN: no bias and no causal mask (only keys past Lk are masked).
template <int NW, int KC, int KS, typename T, int KSPLIT = 1, bool PLAIN = false>
__global__ __launch_bounds__(NW * KSPLIT * 64) void flash_kernel(const T* __restrict__ Q, const T* __restrict__ K,
                                                                 const T* __restrict__ V, T* __restrict__ O,
                                                                 AttnArgs a) {
  static_assert(KS % KC == 0 && KC % 32 == 0 && KS % 8 == 0, "chunking");
  static_assert(KSPLIT == 1 || KSPLIT == 2, "key split");
  static_assert(KSPLIT == 1 || KS * KPITCH * 2 >= NW * 64 * 18 * 4, "merge slots fit in the K staging");
  constexpr int VPITCH = (KS + 63) / 64 * 64 + 8;  // whole 64-key swizzle groups, +8 against bank repeats
  constexpr int KT = KC / 16;   // 16-key tiles per chunk
  constexpr int NT = NW * KSPLIT * 64;
  constexpr int KCH = KS * 8;             // 16-byte K chunks per stage
  constexpr int VBL = KS;                 // 8x8 V blocks per stage (KS/8 key blocks x 8 dim blocks)
  constexpr int KPER = (KCH + NT - 1) / NT;
  constexpr int VPER = (VBL + NT - 1) / NT;
  __shared__ __attribute__((aligned(16))) bf16 Ks[KS * KPITCH];
  __shared__ __attribute__((aligned(16))) bf16 Vt[64 * VPITCH];
  if (blockIdx.z) {  // the prefetching slice
    prefetch_lines(a.pf);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wq = wave % NW, wk = wave / NW;  // query block, key-chunk parity
  // work id -> (head, query block) with a head's query blocks on consecutive ids: xcd_remap puts
  // them on one XCD, whose L2 then fetches the head's K and V once for all of them
  const int nqb = gridDim.x;
  const int wid = xcd_remap(blockIdx.y * nqb + blockIdx.x, nqb * gridDim.y);
  const int bh = wid / nqb;
  const int q0 = ((wid - bh * nqb) * NW + wq) * 16;
  const int lr = lane & 15, g = lane >> 4;
  const T* Qb = Q + (int64_t)bh * a.q_bh;
  const T* Kb = K + (int64_t)bh * a.kv_bh;
  const T* Vb = V + (int64_t)bh * a.kv_bh;

  // this lane's query row (B operand of S^T = K Q^T): 8 dims at 8g and 32 + 8g
  const int qrow = min(q0 + lr, a.Lq - 1);
  const bf16x8 qf0 = load8_bf16<T>(Qb + (int64_t)qrow * 64 + g * 8);
  const bf16x8 qf1 = load8_bf16<T>(Qb + (int64_t)qrow * 64 + 32 + g * 8);
  const int my_q = q0 + lr;

  float m = -INFINITY, lsum = 0.f;
  f32x4 o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const __amdgpu_buffer_rsrc_t Krs = buffer_rsrc(Kb), Vrs = buffer_rsrc(Vb);  // bf16 blocks: Lk * 128 bytes
  for (int ks0 = 0; ks0 < a.Lk; ks0 += KS) {
    __syncthreads();
    {
      bf16x8 kv[KPER], vv[VPER][8];
      // all loads of the stage first (keys past Lk read the last key; masked below)
#pragma unroll
      for (int u = 0; u < KPER; ++u) {
        const int c = min(tid + u * NT, KCH - 1);
        kv[u] = load8_kv<T>(Krs, Kb, min(ks0 + (c >> 3), a.Lk - 1) * 64 + (c & 7) * 8);
      }
#pragma unroll
      for (int u = 0; u < VPER; ++u) {
        const int b = min(tid + u * NT, VBL - 1);
        const int kb = b >> 3, db = b & 7;
#pragma unroll
        for (int r = 0; r < 8; ++r) vv[u][r] = load8_kv<T>(Vrs, Vb, min(ks0 + kb * 8 + r, a.Lk - 1) * 64 + db * 8);
      }
#pragma unroll
      for (int u = 0; u < KPER; ++u) {
        const int c = tid + u * NT;
        if (c < KCH) *reinterpret_cast<bf16x8*>(Ks + (c >> 3) * KPITCH + (c & 7) * 8) = kv[u];
      }
#pragma unroll
      for (int u = 0; u < VPER; ++u) {
        const int b = tid + u * NT;
        if (b < VBL) {
          const int kb = b >> 3, db = b & 7;
          // keys 8kb..8kb+3 go to k-slot positions p0..p0+3, keys 8kb+4..8kb+7 to p0+8..p0+11;
          // rows db*8..db*8+7 share the swizzle db
          const int p0 = (kb >> 2) * 32 + 16 * (kb & 1) + 4 * ((kb >> 1) & 1);
          const int e0 = (((p0 >> 3) ^ db) << 3) + (p0 & 7);
          const int e1 = ((((p0 >> 3) + 1) ^ db) << 3) + (p0 & 7);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            bf16* row = Vt + (db * 8 + j) * VPITCH;
            *reinterpret_cast<bf16x4*>(row + e0) = bf16x4{vv[u][0][j], vv[u][1][j], vv[u][2][j], vv[u][3][j]};
            *reinterpret_cast<bf16x4*>(row + e1) = bf16x4{vv[u][4][j], vv[u][5][j], vv[u][6][j], vv[u][7][j]};
          }
        }
      }
    }
    __syncthreads();
    if (q0 >= a.Lq) continue;

  for (int kc0 = ks0 + wk * KC; kc0 < min(ks0 + KS, a.Lk); kc0 += KC * KSPLIT) {
    const int kl = kc0 - ks0;  // chunk offset inside the staged keys
    // S^T for KT key tiles of 16: s[kt][i] = score(key kc0 + kt*16 + 4g + i, query my_q)
    float s[KT][4];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const bf16* kp = Ks + (kl + kt * 16 + lr) * KPITCH + g * 8;
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
      acc = mfma16(*reinterpret_cast<const bf16x8*>(kp), qf0, acc);
      acc = mfma16(*reinterpret_cast<const bf16x8*>(kp + 32), qf1, acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kc0 + kt * 16 + 4 * g + i;
        float x = acc[i] * a.scale_log2;
        if (!PLAIN && a.bias && key < a.Lk && my_q < a.Lq) x += a.bias[(int64_t)my_q * a.Lk + key] * LOG2E;
        if (key >= a.Lk || (!PLAIN && a.causal && key > my_q)) x = -INFINITY;
        s[kt][i] = x;
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kt][i]);
    mx = max_xor32(max_xor16(mx));
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m - m_use);
    float ps = 0.f;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kt][i] = __builtin_amdgcn_exp2f(s[kt][i] - m_use);
        ps += s[kt][i];
      }
    ps = sum_xor32(sum_xor16(ps));
    lsum = lsum * alpha + ps;
    m = m_new;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[dt][i] *= alpha;

    // O^T += V^T P^T over KT/2 sub-chunks of 32 keys; k-slot j of lane group g maps to
    // key 32kc + 4g + j (j < 4) and 32kc + 16 + 4g + (j - 4) (j >= 4).
#pragma unroll
    for (int kc = 0; kc < KT / 2; ++kc) {
      bf16x8 pb;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pb[i] = f2bf(s[2 * kc][i]);
        pb[4 + i] = f2bf(s[2 * kc + 1][i]);
      }
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const int row = dt * 16 + lr, unit = ((kl + kc * 32) >> 3) + g;
        const bf16x8 va = *reinterpret_cast<const bf16x8*>(Vt + row * VPITCH + ((unit ^ ((row >> 3) & 7)) << 3));
        o[dt] = mfma16(va, pb, o[dt]);
      }
    }
  }
  }
  if (KSPLIT > 1) {
    // lane-wise merge: both waves of a query block hold query lr's state in the same lanes
    __syncthreads();  // every wave is done with the staged K / V^T
    float* slot = reinterpret_cast<float*>(Ks) + (wq * 64 + lane) * 18;
    if (wk == 1) {
      slot[0] = m;
      slot[1] = lsum;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) slot[2 + dt * 4 + i] = o[dt][i];
    }
    __syncthreads();
    if (wk == 1) return;
    const float m2 = slot[0], m_new = fmaxf(m, m2);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float a1 = __builtin_amdgcn_exp2f(m - m_use), a2 = __builtin_amdgcn_exp2f(m2 - m_use);
    lsum = lsum * a1 + slot[1] * a2;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[dt][i] = o[dt][i] * a1 + slot[2 + dt * 4 + i] * a2;
  }
  if (q0 >= a.Lq || my_q >= a.Lq) return;
  const float inv = 1.0f / lsum;
  const int f = bh / a.H, h = bh - f * a.H;
  const int fo = f / a.f_inner, fi = f - fo * a.f_inner;
  const int64_t off = fo * a.o_sfo + fi * a.o_sf + h * a.o_sh + (int64_t)my_q * a.o_si;
  store_head<T>(O, off, o, inv, g, a.frag_ks, a.o8, a.o8s);
}

// PLAIN variants (no bias, not causal) exist for bf16 sequences of up to 64; longer ones run flash_ring_kernel
template <int NW, int KC, int KS, typename T, int KSPLIT = 1>
void flash_go(dim3 g, const T* q, const T* k, const T* v, T* o, const AttnArgs& a, hipStream_t s) {
  const dim3 b(NW * KSPLIT * 64);
  if (oasis::prefetch_any(&a.pf)) g.z = 2;
  if constexpr (std::is_same<T, bf16>::value && KS <= 64) {
    if (!a.bias && !a.causal) {
      hipLaunchKernelGGL((flash_kernel<NW, KC, KS, T, KSPLIT, true>), g, b, 0, s, q, k, v, o, a);
      return;
    }
  }
  hipLaunchKernelGGL((flash_kernel<NW, KC, KS, T, KSPLIT, false>), g, b, 0, s, q, k, v, o, a);
}

// Attention without bias or causal mask on bf16 (every spatial and VAE call). K and V rows go to LDS as they lie,
// by direct-to-LDS loads into a ring of ST stages of KS keys (ST = 1: the whole sequence), and V is transposed on
// the way out by ds_read_b64_tr_b16, so nothing passes through registers and stages are small enough for two or
// three workgroups per CU: flash_kernel stages K and V^T at once (158 KB at 576 keys, one workgroup per CU) and
// its time stepped with rounds of 256 workgroups. Rows are XOR-swizzled against bank repeats: a K row's 16-byte
// units by row % 8, a V row's 32-byte groups by (row / 2) % 4. A stage is consumed in chunks of CT 16-key tiles;
// KSPLIT = 2: two waves per query block, each half of every stage. The sum of the probabilities is of the fp32 ones.
// FINE: what rounding the probabilities to bf16 leaves goes through the products as a second bf16 (one stage, one
// chunk), and their sum is a product with ones of both parts: chunks of 4 to 10 tiles round more probabilities than the
// 32-key chunks of flash_kernel did, where every chunk's largest is 1. Relative rms error against fp64, standard normal
// operands: at 144 keys 2.07e-3 there, 2.17e-3 without FINE, 1.66e-3 (the output's own rounding) with it, for 0.3-0.9
// us; at 576 keys 2.16e-3 there and 2.15e-3 here.
// Measured, before -> now: 576 tokens x 1, 2, 3, 4, 8 latents 9.9, 19.3, 20.1, 28.2, 44.8 -> 9.0, 13.2, 14.0, 18.4,
// 29.1 us; 144 tokens x 1, 8, 12, 32, 64 frames 5.1, 8.1, 11.7, 15.8, 33.1 -> 4.8, 7.0, 8.5, 11.5, 23.7 (64 frames: 75 MB,
// 3.2 TB/s).
// TAIL: keys past the sequence in the last stage; their value rows are cleared.
template <int NW, int KSPLIT, int KS, int ST, int CT, bool FINE, bool TAIL>
__global__ __launch_bounds__(NW * KSPLIT * 64) void flash_ring_kernel(const bf16* __restrict__ Q,
                                                                      const bf16* __restrict__ K,
                                                                      const bf16* __restrict__ V, bf16* __restrict__ O,
                                                                      AttnArgs a) {
  constexpr int W = NW * KSPLIT, KT = KS / KSPLIT / 16;   // 16-key tiles of a wave in a stage
  constexpr int BLKS = KS / 4, LPW = (BLKS + W - 1) / W;  // 1 KB blocks of 8 rows, K's then V's
  constexpr int STAGE = KS * 256, MERGE = KSPLIT > 1 ? NW * 64 * 18 * 4 : 0;
  constexpr int SMEM = ST * STAGE > MERGE ? ST * STAGE : MERGE;
  constexpr int VM = ST > 1 ? (ST - 2) * LPW : 0;
  constexpr int WAIT = (VM & 15) | ((VM >> 4) << 14) | (0x7 << 4) | (0xF << 8);
  static_assert(KT * 16 * KSPLIT == KS && KS % 8 == 0 && SMEM <= 160 * 1024 && VM <= 63, "stages");
  static_assert(!FINE || (ST == 1 && KSPLIT == 1 && CT == KT), "the remainders are not rescaled");
  static_assert((KSPLIT == 1 || KSPLIT == 2) && (CT % 2 == 0 || CT == KT) && CT <= KT, "key split, chunks");
  __shared__ __attribute__((aligned(1024))) char smem[SMEM];
  if (blockIdx.z) {  // the prefetching slice
    prefetch_lines(a.pf);
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = wave % NW, wk = wave / NW;  // query block, key half of each stage
  const int nqb = gridDim.x, wid = xcd_remap(blockIdx.y * nqb + blockIdx.x, nqb * gridDim.y);
  const int bh = wid / nqb, q0 = ((wid - bh * nqb) * NW + wq) * 16;
  const int lr = lane & 15, g = lane >> 4, my_q = q0 + lr;
  const bf16* qp = Q + (int64_t)bh * a.q_bh + (int64_t)min(my_q, a.Lq - 1) * 64 + g * 8;
  const bf16x8 qf0 = load8_bf16<bf16>(qp), qf1 = load8_bf16<bf16>(qp + 32);
  const __amdgpu_buffer_rsrc_t Krs = buffer_rsrc(K + (int64_t)bh * a.kv_bh), Vrs = buffer_rsrc(V + (int64_t)bh * a.kv_bh);

  const int n = (a.Lk + KS - 1) / KS;
  auto issue = [&](int st, int buf) {  // rows past Lk are the last key's; masked and zeroed below
    char* base = smem + buf * STAGE;
#pragma unroll
    for (int u = 0; u < LPW; ++u) {
      const int blk = min(wave * LPW + u, BLKS - 1);
      const bool isv = blk >= KS / 8;
      const int r = (isv ? blk - KS / 8 : blk) * 8 + (lane >> 3), s = lane & 7;
      const int unit = isv ? ((((s >> 1) ^ ((r >> 1) & 3)) << 1) | (s & 1)) : s ^ (r & 7);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(isv ? Vrs : Krs, (__attribute__((address_space(3))) void*)(base + blk * 1024),
                                               16, (uint32_t)min(st * KS + r, a.Lk - 1) * 128u + unit * 16, 0, 0, 0);
    }
  };
#pragma unroll
  for (int st = 0; st < (ST > 1 ? ST - 1 : 1); ++st) issue(min(st, n - 1), st);

  float m = -INFINITY;
  float lsum = 0.f;  // of this lane's keys only (4 of 16); the 4 lanes of a query add up at the end
  f32x4 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 osum = f32x4{0.f, 0.f, 0.f, 0.f};  // FINE: the sum, as a product with ones of both bf16 parts
  const bf16 one = f2bf(1.f);
  const bf16x8 ones = {one, one, one, one, one, one, one, one};
  f32x4 ol[4];  // FINE: the products of the remainders, apart: against an infinite value they are not finite
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) ol[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int st = 0; st < n; ++st) {
    __builtin_amdgcn_s_waitcnt(WAIT);
    __builtin_amdgcn_s_barrier();
    if constexpr (ST > 1) issue(min(st + ST - 1, n - 1), (st + ST - 1) % ST);  // into the buffer read at st - 1
    if (TAIL && (st + 1) * KS > a.Lk) {  // the last key's value once only: against the 0 of a masked key an infinite one is NaN
      char* v0 = smem + (ST > 1 ? st % ST : 0) * STAGE + KS * 128;
      for (int i = (a.Lk - st * KS) * 8 + threadIdx.x; i < KS * 8; i += W * 64)
        *reinterpret_cast<f32x4*>(v0 + i * 16) = f32x4{0.f, 0.f, 0.f, 0.f};
      __syncthreads();
    }
    if (q0 >= a.Lq) continue;
    const char* kb = smem + (ST > 1 ? st % ST : 0) * STAGE + wk * KT * 16 * 128;
    const char* vb = kb + KS * 128;
    const int key0 = st * KS + wk * KT * 16;
#pragma unroll
    for (int c = 0; c < KT; c += CT) {
      const int nt = KT - c < CT ? KT - c : CT;  // tiles of this chunk, known at compile time
      // S^T: s[kt][i] = score(key key0 + (c + kt) * 16 + 4g + i, query my_q)
      float s[CT][4], mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < nt; ++kt) {
        const char* kr = kb + ((c + kt) * 16 + lr) * 128;
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        acc = mfma16(*reinterpret_cast<const bf16x8*>(kr + ((g ^ (lr & 7)) << 4)), qf0, acc);
        acc = mfma16(*reinterpret_cast<const bf16x8*>(kr + (((4 + g) ^ (lr & 7)) << 4)), qf1, acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[kt][i] = acc[i] * a.scale_log2;
      }
      if (key0 + (c + nt) * 16 > a.Lk) {
#pragma unroll
        for (int kt = 0; kt < nt; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (key0 + (c + kt) * 16 + 4 * g + i >= a.Lk) s[kt][i] = -INFINITY;
      }
#pragma unroll
      for (int kt = 0; kt < nt; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kt][i]);
      mx = max_xor32(max_xor16(mx));
      const float m_new = fmaxf(m, mx), m_use = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m - m_use);
      m = m_new;
      float ps[4] = {0.f, 0.f, 0.f, 0.f};  // four chains: one of up to 48 adds takes longer than the products
#pragma unroll
      for (int kt = 0; kt < nt; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[kt][i] = __builtin_amdgcn_exp2f(s[kt][i] - m_use);
          if constexpr (!FINE) ps[i] += s[kt][i];
        }
      lsum = lsum * alpha + ((ps[0] + ps[1]) + (ps[2] + ps[3]));
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[dt][i] *= alpha;
      // O^T += V^T P^T over pairs of key tiles (of an odd count's last pair one): k-slot j of lane group g is key
      // 4g + j (j < 4) of the first tile and 4g + j - 4 of the second
#pragma unroll
      for (int kp = 0; kp < (nt + 1) / 2; ++kp) {
        typedef short i16x4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) i16x4* lds4;
        const bool two = 2 * kp + 1 < nt;
        bf16x8 pb;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pb[i] = f2bf(s[2 * kp][i]);
          pb[4 + i] = two ? f2bf(s[two ? 2 * kp + 1 : 0][i]) : f2bf(0.f);
        }
        bf16x8 pl;  // FINE: what the rounding to pb left
        if constexpr (FINE) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            pl[i] = f2bf(s[2 * kp][i] - bf2f(pb[i]));
            pl[4 + i] = two ? f2bf(s[two ? 2 * kp + 1 : 0][i] - bf2f(pb[4 + i])) : f2bf(0.f);
          }
          osum = mfma16(ones, pb, osum);
          osum = mfma16(ones, pl, osum);
        }
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          const int r = (c + 2 * kp) * 16 + 4 * g + (lr >> 2);  // 16 rows on: the same swizzle
          const char* vr = vb + r * 128 + ((dt ^ ((r >> 1) & 3)) << 5) + (lr & 3) * 8;
          const i16x4 t0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)vr);
          i16x4 t1 = i16x4{0, 0, 0, 0};
          if (two) t1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(vr + 16 * 128));
          const bf16x8 va = __builtin_bit_cast(bf16x8, __builtin_shufflevector(t0, t1, 0, 1, 2, 3, 4, 5, 6, 7));
          o[dt] = mfma16(va, pb, o[dt]);
          if constexpr (FINE) ol[dt] = mfma16(va, pl, ol[dt]);
        }
      }
    }
  }
  if constexpr (KSPLIT > 1) {
    // lane-wise merge: both waves of a query block hold query lr's state in the same lanes
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // no load into the stages is in flight, every wave is done with them
    float* slot = reinterpret_cast<float*>(smem) + (wq * 64 + lane) * 18;
    if (wk == 1) {
      slot[0] = m;
      slot[1] = lsum;
#pragma unroll
      for (int j = 0; j < 16; ++j) slot[2 + j] = o[j / 4][j % 4];
    }
    __syncthreads();
    if (wk == 1) return;
    const float m2 = slot[0], m_new = fmaxf(m, m2), m_use = m_new == -INFINITY ? 0.f : m_new;
    const float a1 = __builtin_amdgcn_exp2f(m - m_use), a2 = __builtin_amdgcn_exp2f(m2 - m_use);
    lsum = lsum * a1 + slot[1] * a2;
#pragma unroll
    for (int j = 0; j < 16; ++j) o[j / 4][j % 4] = o[j / 4][j % 4] * a1 + slot[2 + j] * a2;
  }
  const float inv = 1.0f / (FINE ? osum[0] : sum_xor32(sum_xor16(lsum)));
  if (my_q >= a.Lq) return;  // the 4 lanes of a query leave together
  if constexpr (FINE)
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (fabsf(ol[j / 4][j % 4]) < INFINITY) o[j / 4][j % 4] += ol[j / 4][j % 4];
  const int f = bh / a.H, h = bh - f * a.H;
  const int fo = f / a.f_inner, fi = f - fo * a.f_inner;
  const int64_t off = fo * a.o_sfo + fi * a.o_sf + h * a.o_sh + (int64_t)my_q * a.o_si;
  store_head<bf16>(O, off, o, inv, g, a.frag_ks, a.o8, a.o8s);
}

template <int NW, int KSPLIT, int KS, int ST, int CT, bool FINE = false>
int ring_go(const bf16* q, const bf16* k, const bf16* v, bf16* o, int64_t n_bh, const AttnArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.Lq + NW * 16 - 1) / (NW * 16)), (unsigned)n_bh, oasis::prefetch_any(&a.pf) ? 2 : 1);
  // whole frames without the tail: the two-frame step 1553 us, 1560 with it compiled in; elsewhere it costs nothing
  constexpr bool WHOLE = KS == 144;
  const auto fn = !WHOLE || a.Lk % KS ? &flash_ring_kernel<NW, KSPLIT, KS, ST, CT, FINE, true>
                                      : &flash_ring_kernel<NW, KSPLIT, KS, ST, CT, FINE, !WHOLE>;
  hipLaunchKernelGGL(fn, grid, dim3(NW * KSPLIT * 64), 0, s, q, k, v, o, a);
  return oasis::check_launch("attention");
}

template <typename T>
int flash_launch(const T* q, const T* k, const T* v, T* o, int64_t n_bh, const AttnArgs& a, hipStream_t s) {
  OASIS_REQUIRE(n_bh > 0 && n_bh <= 65535, OASIS_ERR_SHAPE, "attention: bad head count %lld", (long long)n_bh);
  OASIS_REQUIRE((a.Lq / 16 + 1) * n_bh < (1ll << 31), OASIS_ERR_SHAPE, "attention: too many query blocks");
  OASIS_REQUIRE(a.Lq > 0 && a.Lk > 0, OASIS_ERR_SHAPE, "attention: empty sequence");
  // K and V rows are addressed by 32-bit offsets within a (frame, head) block
  OASIS_REQUIRE(a.Lk < (1 << 24), OASIS_ERR_SHAPE, "attention: Lk=%d must be below 2^24", a.Lk);
  // With a bias, a causal mask or fp32 operands, and up to 64 queries and keys: one chunk for up to 32, 64, 160 and
  // 192 keys, beyond that 576-key stages (158 KB of LDS) consumed in 64-key chunks by two waves per query block.
  // 48-row query counts take 48 queries per workgroup (each 16-query block on two waves taking alternate 32-key
  // chunks), or with 256+ heads of 144 queries all 144 (9 waves share one K/V staging).
  const unsigned nb = (unsigned)n_bh;
  if (a.Lq <= 32 && a.Lk <= 32) {
    flash_go<2, 32, 32>(dim3(1, nb), q, k, v, o, a, s);
    return oasis::check_launch("attention");
  }
  if (a.Lq <= 64 && a.Lk <= 64) {
    flash_go<4, 64, 64>(dim3(1, nb), q, k, v, o, a, s);
    return oasis::check_launch("attention");
  }
  if constexpr (std::is_same<T, bf16>::value) {
    if (!a.bias && !a.causal) {
      // The smallest single stage that takes the sequence, beyond 192 keys a ring. Up to 160 keys the probabilities
      // keep their remainders, but with 256 heads of whole-frame or 64-row queries, which flash_kernel took in one
      // chunk: there 64 frames take 23.7 us without, 25.4 with them. 64-, 96- and 128-key stages keep short sequences
      // from computing 144 (200 heads of 144 x 64: 9.1 us on flash_kernel, 6.7 on 96 keys, 5.6 on 64; 255 heads of
      // 128 x 128: 8.0 us on flash_kernel, 8.8 on 144 keys, 6.9 on 128). At 160 keys 64-query workgroups where 48-query ones would be more than two per CU, or one if 64 divides the
      // queries (200 heads of 160 x 160: 48 9.2 us, 64 8.5; 64 x 160: 6.9, 5.7), else 48 (32 heads of 160 x 160:
      // 5.3, with 64 5.4). A ring with one workgroup per CU at most stages 128 keys (96 KB; 16 x 1000 x
      // 1000 13.2 us, with 64 15.3), with more of them 64 (48 KB, three per CU; 3 latents 14.6, with 128 18.3).
      if (a.Lk <= 64) return ring_go<3, 1, 64, 1, 4, true>(q, k, v, o, n_bh, a, s);
      if (a.Lk <= 96) return ring_go<3, 1, 96, 1, 6, true>(q, k, v, o, n_bh, a, s);
      if (a.Lk <= 128) return ring_go<4, 1, 128, 1, 8, true>(q, k, v, o, n_bh, a, s);
      if (a.Lk <= 144)
        return n_bh >= 256 && a.Lq % 144 == 0 ? ring_go<3, 1, 144, 1, 9>(q, k, v, o, n_bh, a, s)
                                              : ring_go<3, 1, 144, 1, 9, true>(q, k, v, o, n_bh, a, s);
      if (a.Lk <= 160) {
        const bool q64 = a.Lq % 64 == 0 || a.Lq % 48 != 0;
        if (q64 && n_bh >= 256) return ring_go<4, 1, 160, 1, 10>(q, k, v, o, n_bh, a, s);
        if (q64 && (a.Lq + 47) / 48 * n_bh > (a.Lq % 64 == 0 ? 256 : 512))
          return ring_go<4, 1, 160, 1, 10, true>(q, k, v, o, n_bh, a, s);
        return ring_go<3, 1, 160, 1, 10, true>(q, k, v, o, n_bh, a, s);
      }
      if (a.Lk <= 192) return ring_go<4, 1, 192, 1, 12>(q, k, v, o, n_bh, a, s);
      if ((a.Lq + 63) / 64 * n_bh <= 256) return ring_go<4, 2, 128, 3, 4>(q, k, v, o, n_bh, a, s);
      return ring_go<4, 2, 64, 3, 2>(q, k, v, o, n_bh, a, s);
    }
  }
  const int kind = a.Lk <= 160 ? 0 : (a.Lk <= 192 ? 1 : 2);
  if (a.Lq % 64 != 0 && a.Lq % 48 == 0) {
    if (kind == 0 && a.Lq % 144 == 0 && n_bh >= 256) {
      flash_go<9, 160, 160>(dim3((unsigned)(a.Lq / 144), nb), q, k, v, o, a, s);
    } else {
      const dim3 g((unsigned)(a.Lq / 48), nb);
      if (kind == 0 && n_bh <= 16)  // one frame: a workgroup per 16-query block (3x the workgroups)
        flash_go<1, 32, 160, T, 2>(dim3((unsigned)(a.Lq / 16), nb), q, k, v, o, a, s);
      else if (kind == 0)  // two waves per query block over alternate 32-key chunks
        flash_go<3, 32, 160, T, 2>(g, q, k, v, o, a, s);
      else if (kind == 1)
        flash_go<3, 192, 192>(g, q, k, v, o, a, s);
      else
        flash_go<3, 64, 576, T, 2>(g, q, k, v, o, a, s);
    }
  } else {
    const dim3 g((unsigned)((a.Lq + 63) / 64), nb);
    if (kind == 0)
      flash_go<4, 160, 160>(g, q, k, v, o, a, s);
    else if (kind == 1)
      flash_go<4, 192, 192>(g, q, k, v, o, a, s);
    else
      flash_go<4, 64, 576, T, 2>(g, q, k, v, o, a, s);
  }
  return oasis::check_launch("attention");
}

// q,k,v: [B][P][H][T][64] bf16; out: token-major [(b*T + t)*P + p][h*64 + d], row-major or
// (fks = 2H) in MFMA fragment order. TW >= 3: windows of TW frames, every row loaded up front (the general loop
// loads a key and a value row per (query, key) pair, a dependent chain of round trips: T = 3 at 432 tokens 4.0 us,
// T = 5 at 1440 10.1, T = 7 at 3024 15.7; with the loads ahead 3.0, 6.2 and 9.1)
template <int TW>
__global__ __launch_bounds__(256) void temporal_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k,
                                                       const bf16* __restrict__ v, bf16* __restrict__ out,
                                                       int64_t G, int T, int P, int H, float scale_log2, int qf,
                                                       int fks, oasis::Prefetch pf, uint8_t* __restrict__ out8,
                                                       uint8_t* __restrict__ out8s) {
  if (blockIdx.z) {  // the prefetching slice
    prefetch_lines(pf);
    return;
  }
  const int64_t grp = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int j = threadIdx.x & 15;
  if (grp >= G) return;  // whole 16-lane groups exit together; no cross-group shuffles
  const int h = (int)(grp % H);
  const int64_t bp = grp / H;
  const int p = (int)(bp % P);
  const int64_t b = bp / P;
  const int64_t base = grp * T * 64 + j * 4;
  // output row `row`, this lane's 4 dims: bf16 (row-major or fragment order) or, with out8, fp8
  // blocks (the 8 lanes of an aligned 32-dim half of the head share a block)
  auto put = [&](int64_t row, float a0, float a1, float a2, float a3) {
    const int col = h * 64 + j * 4;
    if (out8) {
      const float r[4] = {bf2f(f2bf(a0)), bf2f(f2bf(a1)), bf2f(f2bf(a2)), bf2f(f2bf(a3))};
      const float amax = oct_max(fmaxf(fmaxf(fabsf(r[0]), fabsf(r[1])), fmaxf(fabsf(r[2]), fabsf(r[3]))));
      const int64_t e = row * (int64_t)(H * 64) + col;
      store_fp8x4(out8 + e, (j & 7) == 0 ? out8s + e / 32 : nullptr, r, amax);
      return;
    }
    bf16* dst = fks ? out + frag_index(row, col, fks) : out + row * (int64_t)(H * 64) + col;
    *reinterpret_cast<bf16x4*>(dst) = bf16x4{f2bf(a0), f2bf(a1), f2bf(a2), f2bf(a3)};
  };
  if constexpr (TW >= 3) {
    bf16x4 qr[TW], kr[TW], vr[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      qr[t] = *reinterpret_cast<const bf16x4*>(q + base + t * 64);
      kr[t] = *reinterpret_cast<const bf16x4*>(k + base + t * 64);
      vr[t] = *reinterpret_cast<const bf16x4*>(v + base + t * 64);
    }
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      float m = -INFINITY, l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s <= t; ++s) {
        float dot = bf2f(qr[t][0]) * bf2f(kr[s][0]) + bf2f(qr[t][1]) * bf2f(kr[s][1]) +
                    bf2f(qr[t][2]) * bf2f(kr[s][2]) + bf2f(qr[t][3]) * bf2f(kr[s][3]);
        dot = row16_sum(dot);
        const float x = dot * scale_log2;
        const float m_new = fmaxf(m, x);
        const float alpha = exp2f(m - m_new);
        const float pexp = exp2f(x - m_new);
        l = l * alpha + pexp;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = acc[i] * alpha + pexp * bf2f(vr[s][i]);
        m = m_new;
      }
      const float inv = 1.0f / l;
      put((b * TW + t) * P + p, acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
    }
    return;
  }
  // qf >= 0: only query frame qf is computed, written as the single frame of a T=1 output
  // (out row b*P + p); the K/V cache path runs the current frame against cached context K/V.
  if (T == 2) {  // the DiT's 2-frame window: one round trip for all six rows
    const bf16x4 q0 = *reinterpret_cast<const bf16x4*>(q + base), q1 = *reinterpret_cast<const bf16x4*>(q + base + 64);
    const bf16x4 k0 = *reinterpret_cast<const bf16x4*>(k + base), k1 = *reinterpret_cast<const bf16x4*>(k + base + 64);
    const bf16x4 v0 = *reinterpret_cast<const bf16x4*>(v + base), v1 = *reinterpret_cast<const bf16x4*>(v + base + 64);
    // query 0 sees one causal key (softmax weight exactly 1): out_0 = v_0
    float d10 = 0.f, d11 = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      d10 += bf2f(q1[i]) * bf2f(k0[i]);
      d11 += bf2f(q1[i]) * bf2f(k1[i]);
    }
    d10 = row16_sum(d10);
    d11 = row16_sum(d11);
    (void)q0;
    const float x0 = d10 * scale_log2, x1 = d11 * scale_log2;
    const float mx = fmaxf(x0, x1);
    const float p0 = exp2f(x0 - mx), p1 = exp2f(x1 - mx);
    const float inv = 1.0f / (p0 + p1);
    const int T_out = qf < 0 ? T : 1;
    const int64_t row0 = b * T_out * P + p, row1 = qf < 0 ? row0 + P : row0;
    if (qf <= 0) put(row0, bf2f(v0[0]), bf2f(v0[1]), bf2f(v0[2]), bf2f(v0[3]));
    if (qf == 0) return;
    put(row1, (p0 * bf2f(v0[0]) + p1 * bf2f(v1[0])) * inv, (p0 * bf2f(v0[1]) + p1 * bf2f(v1[1])) * inv,
        (p0 * bf2f(v0[2]) + p1 * bf2f(v1[2])) * inv, (p0 * bf2f(v0[3]) + p1 * bf2f(v1[3])) * inv);
    return;
  }
  for (int t = qf < 0 ? 0 : qf; t < (qf < 0 ? T : qf + 1); ++t) {
    const bf16x4 qv4 = *reinterpret_cast<const bf16x4*>(q + base + t * 64);
    float qv[4] = {bf2f(qv4[0]), bf2f(qv4[1]), bf2f(qv4[2]), bf2f(qv4[3])};
    float m = -INFINITY, l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s <= t; ++s) {
      const bf16x4 kv4 = *reinterpret_cast<const bf16x4*>(k + base + s * 64);
      float dot = qv[0] * bf2f(kv4[0]) + qv[1] * bf2f(kv4[1]) + qv[2] * bf2f(kv4[2]) + qv[3] * bf2f(kv4[3]);
      dot = row16_sum(dot);
      const float x = dot * scale_log2;
      const float m_new = fmaxf(m, x);
      const float alpha = exp2f(m - m_new);
      const float pexp = exp2f(x - m_new);
      const bf16x4 vv4 = *reinterpret_cast<const bf16x4*>(v + base + s * 64);
      l = l * alpha + pexp;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = acc[i] * alpha + pexp * bf2f(vv4[i]);
      m = m_new;
    }
    const float inv = 1.0f / l;
    const int64_t frame = qf < 0 ? b * T + t : b;
    put(frame * P + p, acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
  }
}

// Causal windows of 8 to 32 frames: one wave per tile of NT x 16 consecutive rows of the [group][T][64] layout
// (NT = 1: floor(16 / T) whole groups; NT = 2: one group of up to 32 frames), no barrier and no shared staging.
// Q and K rows go straight into the MFMA operands of S^T = K Q^T; V rows go to the wave's own LDS as they lie
// (32-byte groups XOR-swizzled by (row / 2) % 4, so that half a wave's 8 rows fall in distinct banks) and
// ds_read_b64_tr_b16 transposes them into the operand of O^T = V^T P^T: k-slot j of lane group g is key 4g + j
// (j < 4) and 16 + 4g + j - 4. Memory-bound: 4 x 18.9 MB at 9216 tokens. flash_kernel ran a two-wave workgroup per
// group there, one wave without queries up to 16 frames: 34.6 us at 8 streams x 8 frames, 22.6 at 4 x 16, 17.1 at
// 2 x 24, 10.6 at 1 x 32; here 19.3, 19.3, 16.4 and 10.1.
// A masked key's probability is 0, but 0 x inf is not: where a tile's V holds a non-finite value the wave adds
// the unmasked products one key at a time, so that frames and groups stay independent.
template <int NT>
__global__ __launch_bounds__(256) void temporal_tile_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k,
                                                            const bf16* __restrict__ v, bf16* __restrict__ out,
                                                            int rows, int T, int groups, int P, int H,
                                                            float scale_log2, int fks, uint8_t* __restrict__ out8,
                                                            uint8_t* __restrict__ out8s, oasis::Prefetch pf) {
  __shared__ __attribute__((aligned(1024))) char vs_all[4 * NT * 2048];
  if (blockIdx.z) {  // the prefetching slice
    prefetch_lines(pf);
    return;
  }
  const int lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = blockIdx.x * (blockDim.x >> 6) + wave, r0 = tile * groups * T;
  if (r0 >= rows) return;
  const int n = min(rows - r0, groups * T);
  char* vs = vs_all + wave * NT * 2048;
  const int64_t e0 = (int64_t)r0 * 64;
  const __amdgpu_buffer_rsrc_t Qrs = buffer_rsrc(q + e0), Krs = buffer_rsrc(k + e0), Vrs = buffer_rsrc(v + e0);
  // rows past the tile read its last row; what they give is masked or not stored
#pragma unroll
  for (int b = 0; b < NT * 2; ++b) {
    const int r = b * 8 + (lane >> 3), s = lane & 7;
    const int col = ((((s >> 1) ^ ((r >> 1) & 3)) << 1) | (s & 1)) * 8;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(Vrs, (__attribute__((address_space(3))) void*)(vs + b * 1024), 16,
                                             (min(r, n - 1) * 64 + col) * 2, 0, 0, 0);
  }
  bf16x8 qf[NT][2], kf[NT][2];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int r = min(t * 16 + lr, n - 1) * 64 + g * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      kf[t][h] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(Krs, (r + h * 32) * 2, 0, 0));
      qf[t][h] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(Qrs, (r + h * 32) * 2, 0, 0));
    }
  }
  float p[NT][NT][4], inv[NT];  // [query tile][key tile]
#pragma unroll
  for (int qt = 0; qt < NT; ++qt) {
    // score - max as written, so that the largest score gives exactly 0: fused into one multiply-add with the scale
    // (only where a tile of keys needs no mask, the queries past the first 16) the maximum's rounding remains, which
    // above 2^31 overflows exp2
#pragma clang fp contract(off)
    const int my_q = qt * 16 + lr, first = NT == 1 ? my_q - my_q % T : 0;  // the query's group starts at row `first`
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt <= qt; ++kt) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
      acc = mfma16(kf[kt][0], qf[qt][0], acc);
      acc = mfma16(kf[kt][1], qf[qt][1], acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kt * 16 + 4 * g + i;
        p[qt][kt][i] = key <= my_q && key >= first ? acc[i] * scale_log2 : -INFINITY;
        mx = fmaxf(mx, p[qt][kt][i]);
      }
    }
    mx = max_xor32(max_xor16(mx));
    const float m_use = mx == -INFINITY ? 0.f : mx;
    float ps = 0.f;
#pragma unroll
    for (int kt = 0; kt <= qt; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[qt][kt][i] = __builtin_amdgcn_exp2f(p[qt][kt][i] - m_use);
        ps += p[qt][kt][i];
      }
    inv[qt] = 1.0f / sum_xor32(sum_xor16(ps));
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8));  // vmcnt(0): the wave's V rows are in its LDS
  __builtin_amdgcn_sched_barrier(0);
  typedef short i16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) i16x4* lds4;
  bf16x8 va[4];
  bool finite = true;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) {
    i16x4 t[2] = {i16x4{0, 0, 0, 0}, i16x4{0, 0, 0, 0}};
#pragma unroll
    for (int kt = 0; kt < NT; ++kt) {
      const int r = kt * 16 + 4 * g + (lr >> 2);
      t[kt] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(vs + r * 128 + ((dt ^ ((r >> 1) & 3)) << 5) + (lr & 3) * 8));
#pragma unroll
      for (int i = 0; i < 4; ++i) finite &= (t[kt][i] & 0x7F80) != 0x7F80;
    }
    va[dt] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(t[0], t[1], 0, 1, 2, 3, 4, 5, 6, 7));
  }
  const bool all_finite = __builtin_amdgcn_ballot_w64(!finite) == 0;
#pragma unroll
  for (int qt = 0; qt < NT; ++qt) {
    f32x4 o[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int my_q = qt * 16 + lr;
    if (all_finite) {
      bf16x8 pb;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pb[i] = f2bf(p[qt][0][i]);
        pb[4 + i] = qt > 0 ? f2bf(p[qt][NT - 1][i]) : f2bf(0.f);
      }
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] = mfma16(va[dt], pb, o[dt]);
    } else {
      const int first = NT == 1 ? my_q - my_q % T : 0;
#pragma unroll
      for (int kt = 0; kt <= qt; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int kg = 0; kg < 4; ++kg) {
            const int key = kt * 16 + 4 * kg + i;
            const float pk = bf2f(f2bf(__shfl(p[qt][kt][i], kg * 16 + lr, 64)));
            if (key > my_q || key < first) continue;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const bf16* row = reinterpret_cast<const bf16*>(vs + key * 128 + ((dt ^ ((key >> 1) & 3)) << 5));
                o[dt][e] += pk * bf2f(row[4 * g + e]);
              }
          }
    }
    if (my_q >= n) continue;  // the 4 lanes of a query leave together
    const unsigned gi = NT == 1 ? (unsigned)my_q / (unsigned)T : 0, grp = tile * groups + gi, t = my_q - gi * T;
    const unsigned bp = grp / (unsigned)H, h = grp - bp * H, b = bp / (unsigned)P, pos = bp - b * P;
    store_head<bf16>(out, (int64_t)((b * T + t) * P + pos) * (H * 64) + h * 64, o, inv[qt], g, fks, out8, out8s);
  }
}

}  // namespace

namespace {

int attention_impl(const void* q, const void* k, const void* v, void* out, int64_t n_frames, int64_t L,
                   int64_t n_heads, float scale, hipStream_t stream, bool out_frag,
                   const oasis::Prefetch* pf = nullptr, uint8_t* out8 = nullptr, uint8_t* out8_scale = nullptr) {
  OASIS_REQUIRE(q && k && v && out, OASIS_ERR_NULL, "attention: null pointer");
  OASIS_REQUIRE(!out8 || (out8_scale && !out_frag), OASIS_ERR_ARG,
                "attention: an fp8 output needs its scales and a row-major layout");
  OASIS_REQUIRE(!out_frag || (n_frames * L) % 16 == 0, OASIS_ERR_SHAPE,
                "attention: a fragment-order output needs a multiple of 16 rows");
  OASIS_REQUIRE(oasis_aligned(16, q, k, v, out), OASIS_ERR_ARG, "attention: pointers must be 16-byte aligned");
  OASIS_REQUIRE(n_frames > 0 && L > 0 && n_heads > 0 && L < (1 << 30), OASIS_ERR_SHAPE, "attention: bad shape");
  AttnArgs a;
  a.Lq = a.Lk = (int)L;
  a.q_bh = a.kv_bh = L * 64;
  a.scale_log2 = scale * LOG2E;
  a.bias = nullptr;
  a.causal = 0;
  a.H = (int)n_heads;
  a.f_inner = 1 << 30;
  a.o_sfo = 0;
  a.o_sf = L * n_heads * 64;
  a.o_sh = 64;
  a.o_si = n_heads * 64;
  a.frag_ks = out_frag ? (int)(n_heads * 2) : 0;
  a.pf = oasis::prefetch_or_none(pf);
  a.o8 = out8;
  a.o8s = out8_scale;
  return flash_launch<bf16>(static_cast<const bf16*>(q), static_cast<const bf16*>(k), static_cast<const bf16*>(v),
                            static_cast<bf16*>(out), n_frames * n_heads, a, stream);
}

}  // namespace

extern "C" int oasis_attention(const void* q, const void* k, const void* v, void* out, int64_t n_frames, int64_t L,
                               int64_t n_heads, float scale, oasis_stream_t stream) {
  return attention_impl(q, k, v, out, n_frames, L, n_heads, scale, static_cast<hipStream_t>(stream), false);
}

extern "C" int oasis_sdpa(const void* Q, const void* K, const void* V, void* out, int64_t n_heads_total, int64_t sq,
                          int64_t skv, int64_t head_dim, float scale, const float* bias, int causal, int dtype,
                          oasis_stream_t stream) {
  OASIS_REQUIRE(Q && K && V && out, OASIS_ERR_NULL, "sdpa: null pointer");
  OASIS_REQUIRE(oasis_aligned(16, Q, K, V, out), OASIS_ERR_ARG, "sdpa: pointers must be 16-byte aligned");
  OASIS_REQUIRE(head_dim == 64, OASIS_ERR_SHAPE, "sdpa: head_dim must be 64");
  OASIS_REQUIRE(sq > 0 && skv > 0 && sq < (1 << 30) && skv < (1 << 30), OASIS_ERR_SHAPE, "sdpa: bad shape");
  AttnArgs a;
  a.Lq = (int)sq;
  a.Lk = (int)skv;
  a.q_bh = sq * 64;
  a.kv_bh = skv * 64;
  a.scale_log2 = scale * LOG2E;
  a.bias = bias;
  a.causal = causal;
  a.H = 1;
  a.f_inner = 1 << 30;
  a.o_sfo = 0;
  a.o_sf = sq * 64;
  a.o_sh = 0;
  a.o_si = 64;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == OASIS_BF16)
    return flash_launch<bf16>(static_cast<const bf16*>(Q), static_cast<const bf16*>(K), static_cast<const bf16*>(V),
                              static_cast<bf16*>(out), n_heads_total, a, s);
  if (dtype == OASIS_F32)
    return flash_launch<float>(static_cast<const float*>(Q), static_cast<const float*>(K),
                               static_cast<const float*>(V), static_cast<float*>(out), n_heads_total, a, s);
  oasis::set_error("sdpa: unsupported dtype %d", dtype);
  return OASIS_ERR_DTYPE;
}

namespace oasis {

int attention(const void* q, const void* k, const void* v, void* out, int64_t n_frames, int64_t L, int64_t n_heads,
              float scale, hipStream_t stream, bool out_frag, const Prefetch* pf, uint8_t* out8, uint8_t* out8_scale) {
  return attention_impl(q, k, v, out, n_frames, L, n_heads, scale, stream, out_frag, pf, out8, out8_scale);
}

int attention_frag(const void* q, const void* k, const void* v, void* out, int64_t n_frames, int64_t L,
                   int64_t n_heads, float scale, hipStream_t stream) {
  return attention_impl(q, k, v, out, n_frames, L, n_heads, scale, stream, true);
}

int temporal_attention(const void* q, const void* k, const void* v, void* out, int64_t B, int64_t T, int64_t P,
                       int64_t n_heads, float scale, int q_frame, hipStream_t stream, bool out_frag,
                       const Prefetch* pf, uint8_t* out8, uint8_t* out8_scale) {
  OASIS_REQUIRE(q && k && v && out, OASIS_ERR_NULL, "temporal_attention: null pointer");
  OASIS_REQUIRE(!out8 || (out8_scale && !out_frag), OASIS_ERR_ARG,
                "temporal_attention: an fp8 output needs its scales and a row-major layout");
  OASIS_REQUIRE(!out_frag || (B * (q_frame < 0 ? T : 1) * P) % 16 == 0, OASIS_ERR_SHAPE,
                "temporal_attention: a fragment-order output needs a multiple of 16 rows");
  OASIS_REQUIRE(oasis_aligned(16, q, k, v, out), OASIS_ERR_ARG, "temporal_attention: pointers must be 16-byte aligned");
  OASIS_REQUIRE(B > 0 && T > 0 && P > 0 && n_heads > 0 && T <= 4096, OASIS_ERR_SHAPE,
                "temporal_attention: bad shape");
  OASIS_REQUIRE(q_frame < T, OASIS_ERR_ARG, "temporal_attention: q_frame must be < T");
  const int64_t G = B * P * n_heads;
  const bf16 *qp = static_cast<const bf16*>(q), *kp = static_cast<const bf16*>(k), *vp = static_cast<const bf16*>(v);
  bf16* op = static_cast<bf16*>(out);
  const float sl = scale * LOG2E;
  const int fks = out_frag ? (int)(n_heads * 2) : 0;
  const unsigned gz = prefetch_any(pf) ? 2 : 1;
  const Prefetch pfv = prefetch_or_none(pf);
  if (T >= 8 && q_frame < 0) {
    // long causal windows: each (stream, position, head) group is a contiguous [T][64] block; outputs land
    // token-major at row (b*T + t)*P + p. Up to 32 frames a wave per tile of rows, beyond on flash_kernel.
    OASIS_REQUIRE(G <= 65535, OASIS_ERR_SHAPE, "temporal_attention: too many (stream, position, head) groups");
    if (T <= 32) {
      const int groups = T <= 16 ? (int)(16 / T) : 1;
      const int64_t tiles = (G + groups - 1) / groups;
      // up to 12 tiles per CU a workgroup each: four waves in one leave CUs idle (256 groups of 24 frames 4.2 us on
      // flash_kernel, 4.9 with four waves, 4.3 with one; 2304 groups of 16: 7.1, 5.6, 5.2); beyond, four start faster
      // (9216 groups of 32: 25.8 us, 27.2 with one). As fp8 blocks 256 groups of 24 take 5.0 us, 4.3 on flash_kernel,
      // which lets a masked frame's infinite value into the earlier ones.
      const int waves = tiles <= 12 * 256 ? 1 : 4;
      const dim3 grid((unsigned)((tiles + waves - 1) / waves), 1, gz), block(waves * 64);
      if (T <= 16)
        hipLaunchKernelGGL((temporal_tile_kernel<1>), grid, block, 0, stream, qp, kp, vp, op, (int)(G * T), (int)T, groups,
                           (int)P, (int)n_heads, sl, fks, out8, out8_scale, pfv);
      else
        hipLaunchKernelGGL((temporal_tile_kernel<2>), grid, block, 0, stream, qp, kp, vp, op, (int)(G * T), (int)T, groups,
                           (int)P, (int)n_heads, sl, fks, out8, out8_scale, pfv);
      return check_launch("temporal_attention");
    }
    AttnArgs a;
    a.Lq = a.Lk = (int)T;
    a.q_bh = a.kv_bh = T * 64;
    a.scale_log2 = scale * LOG2E;
    a.bias = nullptr;
    a.causal = 1;
    a.H = (int)n_heads;
    a.f_inner = (int)P;  // f = b*P + p
    a.o_sfo = T * P * n_heads * 64;
    a.o_sf = n_heads * 64;
    a.o_sh = 64;
    a.o_si = P * n_heads * 64;
    a.frag_ks = out_frag ? (int)(n_heads * 2) : 0;
    a.pf = prefetch_or_none(pf);
    a.o8 = out8;
    a.o8s = out8_scale;
    return flash_launch<bf16>(static_cast<const bf16*>(q), static_cast<const bf16*>(k), static_cast<const bf16*>(v),
                              static_cast<bf16*>(out), G, a, stream);
  }
  const dim3 grid((unsigned)((G + 15) / 16), 1, gz);
  const int qfr = q_frame < 0 ? -1 : q_frame;
#define OASIS_TEMPORAL(TWV)                                                                                           \
  hipLaunchKernelGGL((temporal_kernel<TWV>), grid, dim3(256), 0, stream, qp, kp, vp, op, G, (int)T, (int)P, (int)n_heads, \
                     sl, qfr, fks, pfv, out8, out8_scale)
  switch (q_frame < 0 ? T : 0) {
    case 3: OASIS_TEMPORAL(3); break;
    case 4: OASIS_TEMPORAL(4); break;
    case 5: OASIS_TEMPORAL(5); break;
    case 6: OASIS_TEMPORAL(6); break;
    case 7: OASIS_TEMPORAL(7); break;
    default: OASIS_TEMPORAL(0);
  }
#undef OASIS_TEMPORAL
  return check_launch("temporal_attention");
}

}  // namespace oasis

extern "C" int oasis_temporal_attention(const void* q, const void* k, const void* v, void* out, int64_t B, int64_t T,
                                        int64_t P, int64_t n_heads, float scale, oasis_stream_t stream) {
  return oasis::temporal_attention(q, k, v, out, B, T, P, n_heads, scale, -1, static_cast<hipStream_t>(stream));
}

extern "C" int oasis_attention_fp8(const void* q, const void* k, const void* v, void* out8, void* out8_scale,
                                   int64_t n_frames, int64_t L, int64_t n_heads, float scale, oasis_stream_t stream) {
  OASIS_REQUIRE(out8 && out8_scale, OASIS_ERR_NULL, "attention_fp8: null output");
  return attention_impl(q, k, v, out8, n_frames, L, n_heads, scale, static_cast<hipStream_t>(stream), false, nullptr,
                        static_cast<uint8_t*>(out8), static_cast<uint8_t*>(out8_scale));
}

extern "C" int oasis_temporal_attention_fp8(const void* q, const void* k, const void* v, void* out8, void* out8_scale,
                                            int64_t B, int64_t T, int64_t P, int64_t n_heads, float scale,
                                            oasis_stream_t stream) {
  OASIS_REQUIRE(out8 && out8_scale, OASIS_ERR_NULL, "temporal_attention_fp8: null output");
  return oasis::temporal_attention(q, k, v, out8, B, T, P, n_heads, scale, -1, static_cast<hipStream_t>(stream), false,
                                   nullptr, static_cast<uint8_t*>(out8), static_cast<uint8_t*>(out8_scale));
}
