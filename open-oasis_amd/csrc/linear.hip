// The reference surface's linear layer, out = x @ w with w in its [K, N] layout (src/linear.py:10-53).
//
// linear_kernel: the direct-to-LDS ring of gemm_big_kernel with B staged as it lies in memory, 64 k rows of BN
// columns, and transposed on the way out of LDS by ds_read_b64_tr_b16: lane i of each 16 lanes points at
// 4 columns (i % 4) of k row i / 4 of a 4 x 16 block and receives the 4 rows of column i, so two reads give a
// lane the 8 consecutive k of its column that v_mfma_f32_16x16x32_bf16 takes. The 32-byte column groups of row
// r are stored XOR-swizzled by f(r), which sends the 8 rows that half a wave reads to distinct banks.
#include <algorithm>

#include "gemm_epilogue.h"

namespace {

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));

// swizzle of row r's 32-byte groups (BN / 16 of them): half a wave reads rows 8g + i, g in {0, 1} or {2, 3} and
// i in 0..3 (then 4..7), of one group; a 64-column row is half of the 256 bytes the banks cover
template <int BN>
__device__ __forceinline__ int group_swizzle(int r) {
  return BN == 64 ? ((r >> 1) & 1) | (((r >> 3) & 1) << 1) : (r & 3) | (((r >> 3) & 1) << 2);
}

template <int BM, int BN, int WM, int WN, int STAGES, bool F32, bool WIDE = false>
__global__ __launch_bounds__(WM * WN * 64) void linear_kernel(const bf16* __restrict__ A, int64_t lda,
                                                             const bf16* __restrict__ B, int64_t ldb, int M, int N,
                                                             int K, void* __restrict__ out) {
  constexpr int NW = WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
  static_assert(FM * 16 == TM && FN * 16 == TN && (BN == 64 || BN == 128), "tile");
  constexpr int ABLK = BM / 8, BBLK = BN / 8, NBLK = ABLK + BBLK;  // 1 KB blocks: 8 A rows; 512 / BN rows of B
  constexpr int BROWS = 512 / BN;
  constexpr int LPW = (NBLK + NW - 1) / NW;
  constexpr int STAGE_BYTES = NBLK * 1024;
  constexpr int EP = TN + 4;
  constexpr int EPI_BYTES = NW * 16 * EP * 4;
  constexpr int SMEM = STAGES * STAGE_BYTES > EPI_BYTES ? STAGES * STAGE_BYTES : EPI_BYTES;
  static_assert(SMEM <= 160 * 1024 && STAGES >= 2 && (STAGES - 2) * LPW <= 63, "LDS, vmcnt");
  __shared__ __attribute__((aligned(1024))) char smem[SMEM];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int Mt = (M + BM - 1) / BM, Nt = (N + BN - 1) / BN;
  int split, mt, nt;
  grouped_tile(xcd_remap(blockIdx.x, Mt * Nt), Mt, Nt, 8, split, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN, nk = K / 64;

  // this lane's source in each of its LPW blocks. A: row r, K chunk (lane % 8) ^ ((r >> 1) & 7), a scalar
  // offset per K tile. B: row r of the K tile, the 16 columns whose swizzled group the lane's slot is, clamped
  // to the last 8 columns (N is a multiple of 8; what they feed is dropped), and a scalar base per K tile.
  const __amdgpu_buffer_rsrc_t Ars = buffer_rsrc(A + (int64_t)m0 * lda);
  uint32_t off[LPW];
  int64_t woff[WIDE ? LPW : 1];  // WIDE: rows too long for 32-bit byte offsets (elements)
  int dst[LPW];
  bool from_a[LPW];
#pragma unroll
  for (int u = 0; u < LPW; ++u) {
    const int blk = min(wave * LPW + u, NBLK - 1);
    from_a[u] = blk < ABLK;
    if (from_a[u]) {
      const int r = blk * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
      const int64_t o = (int64_t)(min(m0 + r, M - 1) - m0) * lda + c * 8;
      off[u] = (uint32_t)(o * 2);
      if constexpr (WIDE) woff[u] = o;
    } else {
      const int r = (blk - ABLK) * BROWS + lane / (BN / 8), s = lane % (BN / 8);
      const int col = ((((s >> 1) ^ group_swizzle<BN>(r)) << 1) | (s & 1)) * 8;
      const int64_t o = (int64_t)r * ldb + min(n0 + col, N - 8) - n0;
      off[u] = (uint32_t)(o * 2);
      if constexpr (WIDE) woff[u] = o;
    }
    dst[u] = blk * 1024;
  }
  auto issue = [&](int kt, int buf) {
    char* base = smem + buf * STAGE_BYTES;
    const bf16* Bk = B + (int64_t)kt * 64 * ldb + n0;
    const __amdgpu_buffer_rsrc_t Brs = buffer_rsrc(Bk);
#pragma unroll
    for (int u = 0; u < LPW; ++u) {
      if constexpr (WIDE)
        load_lds16(from_a[u] ? A + (int64_t)m0 * lda + kt * 64 + woff[u] : Bk + woff[u], base + dst[u]);
      else
        buffer_load_lds16(from_a[u] ? Ars : Brs, off[u], from_a[u] ? kt * 128 : 0, base + dst[u]);
    }
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int lr = lane & 15, g = lane >> 4;
  // B: this lane's row within a 32-wide K step (+ 4 for the second read) and its 8 bytes of the group
  const int br = 8 * g + (lr >> 2), bsw = group_swizzle<BN>(br), bo = br * BN * 2 + (lr & 3) * 8;
  auto compute = [&](int buf) {
    const char* base = smem + buf * STAGE_BYTES;
    const char* bb = base + ABLK * 1024 + bo;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int c = ks * 4 + g;
      bf16x8 af[FM], bfr[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int r = wm * TM + i * 16 + lr;
        af[i] = *reinterpret_cast<const bf16x8*>(base + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const char* p = bb + ks * 32 * BN * 2 + (((wn * FN + j) ^ bsw) << 5);
        typedef __attribute__((address_space(3))) i16x4* lds4;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)p);
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 4 * BN * 2));
        bfr[j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma16(af[i], bfr[j], acc[i][j]);
    }
  };

  constexpr int VM = (STAGES - 2) * LPW;
  constexpr int WAIT = (VM & 15) | ((VM >> 4) << 14) | (0x7 << 4) | (0xF << 8);
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) issue(min(s, nk - 1), s);
  for (int k = 0; k < nk; ++k) {
    __builtin_amdgcn_s_waitcnt(WAIT);
    __builtin_amdgcn_s_barrier();
    issue(min(k + STAGES - 1, nk - 1), (k + STAGES - 1) % STAGES);  // into the buffer read at k - 1
    compute(k % STAGES);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // 16 rows of the wave's tile at a time through its own LDS: 8 consecutive columns of a row per lane
  float* st = reinterpret_cast<float*>(smem) + wave * 16 * EP;
  constexpr int UPR = TN / 8;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[(g * 4 + r) * EP + j * 16 + lr] = acc[i][j][r];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int u = lane; u < 16 * UPR; u += 64) {
      const int r = u / UPR, c8 = (u - r * UPR) * 8;
      const int gm = m0 + wm * TM + i * 16 + r, gn = n0 + wn * TN + c8;
      if (gm >= M || gn >= N) continue;
      const f32x4 c0 = *reinterpret_cast<const f32x4*>(st + r * EP + c8);
      const f32x4 c1 = *reinterpret_cast<const f32x4*>(st + r * EP + c8 + 4);
      if constexpr (F32) {
        float* d = static_cast<float*>(out) + (int64_t)gm * N + gn;
        *reinterpret_cast<f32x4*>(d) = c0;
        *reinterpret_cast<f32x4*>(d + 4) = c1;
      } else {
        const float v[8] = {c0[0], c0[1], c0[2], c0[3], c1[0], c1[1], c1[2], c1[3]};
        store8_bf16(static_cast<bf16*>(out) + (int64_t)gm * N + gn, v);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// Up to a few hundred rows, where the tiles do not fill the CUs and each ring tile waits out a memory latency
// per few K tiles: the 4 waves of a workgroup split K four ways, each over its own STG-deep LDS ring with no
// workgroup barrier in the K loop (as gemm_wave_kernel), and the partial tiles are summed through LDS. BN = 64;
// K a multiple of 256; rows within 32-bit byte offsets.
template <int BM, int STG, bool F32>
__global__ __launch_bounds__(256) void linear_wave_kernel(const bf16* __restrict__ A, int64_t lda,
                                                          const bf16* __restrict__ B, int64_t ldb, int M, int N, int K,
                                                          void* __restrict__ out) {
  constexpr int BN = 64, NW = 4, FM = BM / 16, FN = BN / 16;
  constexpr int ABLK = BM / 8, NBLK = ABLK + 8;  // 1 KB blocks of a K tile, one load instruction each
  constexpr int STAGE_BYTES = NBLK * 1024, WAVE_BYTES = STG * STAGE_BYTES;
  constexpr int PITCH = BN + 4;
  static_assert(NW * WAVE_BYTES <= 160 * 1024 && BM * PITCH * 4 <= WAVE_BYTES && (STG - 1) * NBLK <= 63, "LDS, vmcnt");
  __shared__ __attribute__((aligned(1024))) char smem[NW * WAVE_BYTES];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int Mt = (M + BM - 1) / BM, Nt = (N + BN - 1) / BN;
  const int pid = xcd_remap(blockIdx.x, Mt * Nt);
  const int nt = pid / Mt, mt = pid - nt * Mt;  // m fastest: an XCD's workgroups share weight columns
  const int m0 = mt * BM, n0 = nt * BN;
  const int nk = K / (64 * NW), k0 = wave * nk;  // this wave's K tiles
  char* ring = smem + wave * WAVE_BYTES;

  const __amdgpu_buffer_rsrc_t Ars = buffer_rsrc(A + (int64_t)m0 * lda);
  uint32_t off[NBLK];
#pragma unroll
  for (int b = 0; b < NBLK; ++b) {
    if (b < ABLK) {
      const int r = b * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
      off[b] = (uint32_t)(((int64_t)(min(m0 + r, M - 1) - m0) * lda + c * 8) * 2);
    } else {
      const int r = (b - ABLK) * 8 + (lane >> 3), s = lane & 7;
      const int col = ((((s >> 1) ^ group_swizzle<BN>(r)) << 1) | (s & 1)) * 8;
      off[b] = (uint32_t)(((int64_t)r * ldb + min(n0 + col, N - 8) - n0) * 2);
    }
  }
  auto issue = [&](int kt, int buf) {
    char* base = ring + buf * STAGE_BYTES;
    const __amdgpu_buffer_rsrc_t Brs = buffer_rsrc(B + (int64_t)(k0 + kt) * 64 * ldb + n0);
#pragma unroll
    for (int b = 0; b < NBLK; ++b)
      buffer_load_lds16(b < ABLK ? Ars : Brs, off[b], b < ABLK ? (k0 + kt) * 128 : 0, base + b * 1024);
  };
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int lr = lane & 15, g = lane >> 4;
  const int br = 8 * g + (lr >> 2), bsw = group_swizzle<BN>(br), bo = br * BN * 2 + (lr & 3) * 8;
  auto compute = [&](int buf) {
    const char* base = ring + buf * STAGE_BYTES;
    const char* bb = base + ABLK * 1024 + bo;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int c = ks * 4 + g;
      bf16x8 af[FM], bfr[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int r = i * 16 + lr;
        af[i] = *reinterpret_cast<const bf16x8*>(base + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const char* p = bb + ks * 32 * BN * 2 + ((j ^ bsw) << 5);
        typedef __attribute__((address_space(3))) i16x4* lds4;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)p);
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 4 * BN * 2));
        bfr[j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma16(af[i], bfr[j], acc[i][j]);
    }
  };
  // tile k's loads are followed by those of tiles k + 1 .. k + STG - 1 (the last tile's again at the end, so
  // that one bound holds); the buffer of tile k is reloaded only after its reads, which the MFMAs that use
  // them have waited for
  constexpr int VM = (STG - 1) * NBLK;
  constexpr int WAIT = (VM & 15) | ((VM >> 4) << 14) | (0x7 << 4) | (0xF << 8);
#pragma unroll
  for (int s = 0; s < STG; ++s) issue(min(s, nk - 1), s);
  int buf = 0;
  for (int k = 0; k < nk; ++k) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(WAIT);
    __builtin_amdgcn_sched_barrier(0);
    compute(buf);
    __builtin_amdgcn_sched_barrier(0);
    issue(min(k + STG, nk - 1), buf);
    buf = buf + 1 == STG ? 0 : buf + 1;
  }
  __builtin_amdgcn_s_waitcnt(0);

  float* mine = reinterpret_cast<float*>(ring);  // each wave's partial tile over its own ring
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) mine[(i * 16 + g * 4 + r) * PITCH + j * 16 + lr] = acc[i][j][r];
  __syncthreads();
#pragma unroll
  for (int u = tid; u < BM * 8; u += 256) {
    const int r = u >> 3, c8 = (u & 7) * 8;
    const int gm = m0 + r, gn = n0 + c8;
    if (gm >= M || gn >= N) continue;
    f32x4 c0 = f32x4{0.f, 0.f, 0.f, 0.f}, c1 = c0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* p = reinterpret_cast<const float*>(smem + w * WAVE_BYTES) + r * PITCH + c8;
      c0 += *reinterpret_cast<const f32x4*>(p);
      c1 += *reinterpret_cast<const f32x4*>(p + 4);
    }
    if constexpr (F32) {
      float* d = static_cast<float*>(out) + (int64_t)gm * N + gn;
      *reinterpret_cast<f32x4*>(d) = c0;
      *reinterpret_cast<f32x4*>(d + 4) = c1;
    } else {
      const float v[8] = {c0[0], c0[1], c0[2], c0[3], c1[0], c1[1], c1[2], c1[3]};
      store8_bf16(static_cast<bf16*>(out) + (int64_t)gm * N + gn, v);
    }
  }
}

typedef void (*linear_fn)(const bf16*, int64_t, const bf16*, int64_t, int, int, int, void*, bool, hipStream_t);
template <int BM, int BN, int WM, int WN, int STAGES, bool WIDE = false>
void launch_linear(const bf16* A, int64_t lda, const bf16* B, int64_t ldb, int M, int N, int K, void* out, bool f32,
                   hipStream_t s) {
  const dim3 grid((unsigned)((M + BM - 1) / BM * ((N + BN - 1) / BN))), block(WM * WN * 64);
  if (f32)
    hipLaunchKernelGGL((linear_kernel<BM, BN, WM, WN, STAGES, true, WIDE>), grid, block, 0, s, A, lda, B, ldb, M, N, K, out);
  else
    hipLaunchKernelGGL((linear_kernel<BM, BN, WM, WN, STAGES, false, WIDE>), grid, block, 0, s, A, lda, B, ldb, M, N, K, out);
}
template <int BM, int STG>
void launch_linear_wave(const bf16* A, int64_t lda, const bf16* B, int64_t ldb, int M, int N, int K, void* out, bool f32,
                        hipStream_t s) {
  const dim3 grid((unsigned)((M + BM - 1) / BM * ((N + 63) / 64)));
  if (f32)
    hipLaunchKernelGGL((linear_wave_kernel<BM, STG, true>), grid, dim3(256), 0, s, A, lda, B, ldb, M, N, K, out);
  else
    hipLaunchKernelGGL((linear_wave_kernel<BM, STG, false>), grid, dim3(256), 0, s, A, lda, B, ldb, M, N, K, out);
}

// Tile by measured cost (hipGraphs of 24 launches over cold weights, 32 to 5120 rows, K = 1024 and 4096,
// N = 64 to 4096): with W = ceil(tiles / 256) workgroups on the busiest CU and nk = K / 64,
//     c + max(lat * nk, W * (a * nk + b))  microseconds,
// lat the time of a K tile of a workgroup that has its CU to itself (a ring tile waits out the memory latency
// every few K tiles; a wave-split one is four rings at once). The pick is within 3% of the fastest of them at
// every measured shape. 320 x 3072 x 1024 takes 9.6 us, 5120 x 4096 x 1024 51 us (840 TFLOP/s); the 4-wave
// register ring with 2-byte transposing LDS stores before took 23.9 and 369 us.
struct LinearTile {
  int bm, bn, kgran;  // K a multiple of kgran
  float c, lat, a, b;
  linear_fn fn;
};
const LinearTile kLinear[] = {
    {16, 64, 256, 1.7f, 0.0f, 0.14f, 2.56f, launch_linear_wave<16, 3>},
    {32, 64, 256, 1.7f, 0.0f, 0.167f, 2.6f, launch_linear_wave<32, 2>},
    {48, 64, 256, 2.1f, 0.0f, 0.185f, 2.7f, launch_linear_wave<48, 2>},
    {64, 64, 256, 2.4f, 0.0f, 0.233f, 3.1f, launch_linear_wave<64, 2>},
    {64, 64, 64, 2.4f, 0.58f, 0.36f, -0.5f, launch_linear<64, 64, 2, 2, 4>},
    {96, 64, 64, 3.0f, 0.69f, 0.35f, 0.6f, launch_linear<96, 64, 2, 2, 4>},
    {128, 128, 64, 2.6f, 0.88f, 0.88f, 1.6f, launch_linear<128, 128, 2, 4, 3>},
    {192, 128, 64, 4.8f, 0.97f, 0.6f, 1.3f, launch_linear<192, 128, 4, 2, 2>},  // two workgroups per CU
};

const LinearTile& linear_tile(int64_t M, int64_t N, int64_t K) {
  const LinearTile* best = nullptr;
  float best_us = 0.f;
  const float nk = (float)(K / 64);
  for (const LinearTile& t : kLinear) {
    if (K % t.kgran != 0) continue;
    const int64_t tiles = (M + t.bm - 1) / t.bm * ((N + t.bn - 1) / t.bn);
    const float us = t.c + std::max(t.lat * nk, (float)((tiles + 255) / 256) * (t.a * nk + t.b));
    if (!best || us < best_us) {
      best = &t;
      best_us = us;
    }
  }
  return *best;
}

// a K tile's 64 rows, or a tile's rows of x, beyond 32-bit byte offsets (2^32 / 2 / 192 rows)
bool linear_wide(int64_t K, int64_t N) { return N >= (1ll << 24) || K >= (1ll << 23); }

}  // namespace

extern "C" int oasis_linear_tile(int64_t M, int64_t K, int64_t N) {
  OASIS_REQUIRE(M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 8 == 0 && M < (1ll << 31) && N < (1ll << 31),
                OASIS_ERR_SHAPE, "linear_tile: need K %% 64 == 0 and N %% 8 == 0");
  if (linear_wide(K, N)) return (int)(sizeof(kLinear) / sizeof(kLinear[0]));
  return (int)(&linear_tile(M, N, K) - kLinear);
}

extern "C" int oasis_linear(const void* x, const void* w, void* out, int64_t M, int64_t K, int64_t N,
                            int w_layout, int out_dtype, oasis_stream_t stream) {
  OASIS_REQUIRE(x && w && out, OASIS_ERR_NULL, "linear: null pointer");
  OASIS_REQUIRE(oasis_aligned(16, x, w, out), OASIS_ERR_ARG, "linear: pointers must be 16-byte aligned");
  OASIS_REQUIRE(M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 8 == 0 && M < (1ll << 31) && N < (1ll << 31),
                OASIS_ERR_SHAPE, "linear: need K %% 64 == 0 and N %% 8 == 0");
  OASIS_REQUIRE(w_layout == 0 || w_layout == 1, OASIS_ERR_ARG, "linear: w_layout must be 0 ([K,N]) or 1 ([N,K])");
  OASIS_REQUIRE(out_dtype == OASIS_F32 || out_dtype == OASIS_BF16, OASIS_ERR_DTYPE, "linear: bad out dtype %d",
                out_dtype);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (w_layout == 1) {
    oasis_epilogue_t ex;
    memset(&ex, 0, sizeof(ex));
    ex.kind = out_dtype == OASIS_F32 ? OASIS_EPI_STORE_F32 : OASIS_EPI_STORE_BF16;
    ex.out_f32 = static_cast<float*>(out);
    ex.out_bf16 = out;
    ex.ld_out = N;
    return oasis::gemm_launch(static_cast<const bf16*>(x), K, static_cast<const bf16*>(w), K, M, N, K, ex, s);
  }
  if (linear_wide(K, N)) {
    launch_linear<64, 64, 2, 2, 4, true>(static_cast<const bf16*>(x), K, static_cast<const bf16*>(w), N, (int)M, (int)N,
                                         (int)K, out, out_dtype == OASIS_F32, s);
    return oasis::check_launch("linear");
  }
  const LinearTile& t = linear_tile(M, N, K);
  t.fn(static_cast<const bf16*>(x), K, static_cast<const bf16*>(w), N, (int)M, (int)N, (int)K, out, out_dtype == OASIS_F32,
       s);
  return oasis::check_launch("linear");
}
