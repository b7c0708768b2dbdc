// bf16 MFMA GEMM for the DiT projections, with fused epilogues.
//
//   C[m, n] = epilogue( sum_k A[m, k] * W[n, k] + bias[n] )
//
// A is the token-major activation [M, K]; W is an nn.Linear weight [N, K]; both
// are K-contiguous, which is what the MFMA operands want (each lane feeds 8
// consecutive k values).  The kernel computes C^T tiles: the MFMA "A" operand
// is a 16-row slice of W and the "B" operand a 16-token slice of the
// activation, so every lane ends up owning one token and 4 consecutive output
// features per accumulator tile -> 8-byte row-major staging writes.
//
// Tiling (gfx950, v_mfma_f32_16x16x32_bf16, which draws less power per FLOP
// than the 32x32x16 form): a 512-thread workgroup computes a 256 (tokens) x 256
// (features) tile as 2 x 4 waves of 128 tokens x 64 features (4 x 8
// accumulator tiles of 16 x 16 per wave), two waves per SIMD so one wave's
// MFMAs issue while the other waits on its DMA or LDS reads.  K advances
// through 128 KiB of LDS stages filled by direct global->LDS DMA (no register
// staging): two stages of 64 k when K % 64 == 0, else four of 32 k.
//
// The k-loop order is fixed and there is no split-K, so every output element is
// computed the same way whatever M is and wherever its row sits: packed and
// per-request projections agree bitwise.
#include <atomic>

#include "ditk_common.h"
#include "gemm_l4_clobbers.h"

namespace {

enum Epilogue : int {
  EPI_BIAS = 0,      // bf16(acc + b)
  EPI_GELU = 1,      // bf16(gelu_tanh(bf16(acc + b)))
  EPI_GATE_RES = 2,  // bf16(R + bf16(acc + b) * gate[seg, n])   (fp32 math)
  EPI_RES = 3,       // bf16(R + bf16(acc + b))
  EPI_F32 = 4,       // fp32(acc + b)
  EPI_SILU = 5,      // bf16(silu(bf16(acc + b)))
};

// Workgroup tile configurations.  A wave computes WTM tokens x 64 features (the
// epilogue staging swizzle below assumes 64 features); the GW = WM x WN waves of
// a workgroup are laid out WM along tokens and WN along features.
//   TILE_LARGE  256 x 256, 8 waves of 128 x 64, 128 KiB of LDS stages, one
//               workgroup per CU (two waves per SIMD).
//   TILE_SMALL   64 x 128, 4 waves of 32 x 64, 72 KiB, two workgroups per CU:
//               for GEMMs whose large tiles would leave CUs idle (the few hundred
//               text rows of a step, two-row conditioning projections).
// Both run the same MFMA (W rows as the A operand) over the same k-chunk order
// with the same epilogue arithmetic, so an output element is bitwise the same
// whichever tile computed it.
enum TileCfg : int { TILE_LARGE = 0, TILE_SMALL = 1 };
template <int T> struct Tile;
template <> struct Tile<TILE_LARGE> {
  static constexpr int GBM = 256, GBN = 256, WM = 2, WN = 4, LDS_BYTES = 128 * 1024, WAVES_PER_EU = 1;
};
template <> struct Tile<TILE_SMALL> {
  static constexpr int GBM = 64, GBN = 128, WM = 2, WN = 2, LDS_BYTES = 72 * 1024, WAVES_PER_EU = 2;
};

// k-stage geometry for BK k values per stage (BK = 64 when K allows, else 32)
template <int BK, int T>
struct Stages {
  static constexpr int GBM = Tile<T>::GBM;            // tokens per workgroup tile
  static constexpr int GBN = Tile<T>::GBN;            // features per workgroup tile
  static constexpr int GW = Tile<T>::WM * Tile<T>::WN;  // waves per workgroup
  static constexpr int WTM = GBM / Tile<T>::WM;       // tokens per wave tile
  static constexpr int WTN = GBN / Tile<T>::WN;       // features per wave tile
  static constexpr int GBK = BK;
  static constexpr int NCH = BK / 32;                 // 32-k MFMA chunks per stage
  static constexpr int CPRW = BK / 8;                 // 16-byte chunks per LDS row
  static constexpr int RPG = 64 / CPRW;               // rows filled by one DMA instruction (1 KiB)
  static constexpr int DPW_A = GBM / RPG / GW;        // A DMA instructions per wave and stage
  static constexpr int DPW_W = GBN / RPG / GW;        // W DMA instructions per wave and stage
  static constexpr int ND = DPW_A + DPW_W;            // DMA instructions per wave and stage
  static constexpr int NSTAGE = Tile<T>::LDS_BYTES / ((GBM + GBN) * BK * 2);
  static_assert(WTN == 64 && DPW_A >= 1 && DPW_W >= DPW_A && DPW_A * GW * RPG == GBM &&
                    DPW_W * GW * RPG == GBN && (BK == 32 || BK == 64) && NSTAGE >= 2 &&
                    GW * WTM * WTN * 2 <= Tile<T>::LDS_BYTES,
                "tile configuration");
  // LDS stage layout (A and W alike): row r of BK k-values = CPRW chunks of
  // 16 B, slot(r, u) = r*CPRW + (u ^ swz(r)).  A DMA instruction fills 64
  // contiguous slots (RPG whole rows); 16 consecutive lanes reading chunk u of
  // 16 consecutive rows hit 16 distinct 16-byte bank groups.
  static __device__ __forceinline__ int swz(int r) { return CPRW == 4 ? (r >> 2) & 3 : (r >> 1) & 7; }
  // wait until at most `stages` DMA stages (ND instructions each) of this wave are in flight
  static __device__ __forceinline__ void dma_wait(int stages) {
    constexpr int P = ND;
    if (stages >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * P) : "memory");
    else if (stages == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
};

// Tile order: groups of `group_m` m-tiles walked m-fastest within the group, so
// the tiles running together share A rows and W rows in L2.  Chosen per shape
// (measured on the block GEMMs, same box): long K favours narrow groups
// (ffn-down: 1.39 ms at 1 vs 1.46 at 8), many n-tiles favour 4 (ffn-up: 1.58 vs
// 1.73), the rest 8.  The order does not change any result.
int gemm_group_m(int K, int tiles_n) { return K >= 4096 ? 1 : (tiles_n >= 24 ? 4 : 8); }

// 16 bytes per lane, global -> LDS; the wave's 64 lanes fill 1 KiB starting at
// the wave-uniform lds_slot0 (lane l writes bytes 16l .. 16l+15).
__device__ __forceinline__ void lds_dma16(const bf16_t* gsrc, u32x4_t* lds_slot0) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)gsrc,
                                   (__attribute__((address_space(3))) void*)lds_slot0, 16, 0, 0);
}
// Per 32 k a wave reads 4 feature fragments (double-buffered) and 8 token
// fragments (single-buffered: token fragment j of the next chunk is read right
// after the 4 MFMAs that use fragment j of this one).  Accumulator lane layout:
// features f = i*16 + 4*(lane/16) + e, token t = j*16 + lane % 16 of the wave
// tile.  The bias is loaded after the k loop (holding it through the loop would
// spill).
// STREAM: output stored past the caches (see stream_output; a run-time choice in the
// epilogue's stores costs 3% at 65520 x 1536 x 1536).
template <int EPI, int BK, int T, bool STREAM>
__global__ __launch_bounds__(Tile<T>::WM * Tile<T>::WN * 64, Tile<T>::WAVES_PER_EU) void gemm_kernel(
    const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W, int64_t ldw,
    const float* __restrict__ bias, void* __restrict__ Cv, int64_t ldc, int M, int N, int K,
    const bf16_t* R, int64_t ldr, const float* __restrict__ gate, int64_t gate_stride,
    const int32_t* __restrict__ cu, int nseg, int tiles_m, int tiles_n, int group_m, int row_base) {
  using S = Stages<BK, T>;
  constexpr int GBM = S::GBM, GBN = S::GBN, GW = S::GW, WTM = S::WTM, WTN = S::WTN;
  constexpr int CPRW = S::CPRW, RPG = S::RPG, NSTAGE = S::NSTAGE, DPW_A = S::DPW_A, DPW_W = S::DPW_W;
  constexpr int ND = S::ND, NCH = S::NCH;
  constexpr int FI = WTN / 16, FJ = WTM / 16;  // feature / token fragments per wave (4; 8 or 2)
  __shared__ u32x4_t lds[NSTAGE * (GBM + GBN) * CPRW];
  auto As = [&](int s) { return lds + s * (GBM * CPRW); };
  auto Ws = [&](int s) { return lds + NSTAGE * GBM * CPRW + s * (GBN * CPRW); };

  const int nb = gridDim.x, b = blockIdx.x;
  const int L = (b & 7) * (nb >> 3) + (b >> 3);
  if (L >= tiles_m * tiles_n) return;
  const int group = L / (group_m * tiles_n);
  const int first_m = group * group_m;
  const int gm = min(group_m, tiles_m - first_m);
  const int pid = L % (group_m * tiles_n);
  const int mt = first_m + pid % gm, nt = pid / gm;
  const int m0 = mt * GBM, n0 = nt * GBN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ql = lane & 15, g = lane >> 4;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int wm = wave_u % Tile<T>::WM, wn = wave_u / Tile<T>::WM;
  const int a_row0 = wm * WTM, w_row0 = wn * WTN;

  const bf16_t* Ablk = A + (int64_t)m0 * lda;
  const bf16_t* Wblk = W + (int64_t)n0 * ldw;
  uint32_t a_off[DPW_A], w_off[DPW_W];
#pragma unroll
  for (int i = 0; i < DPW_W; ++i) {
    const int gi = i * GW + wave_u;
    const int row = gi * RPG + lane / CPRW;
    const int ksw = ((lane % CPRW) ^ S::swz(row)) * 8;
    if (i < DPW_A) a_off[i] = (uint32_t)(min(row, M - 1 - m0) * lda + ksw);
    w_off[i] = (uint32_t)(min(row, N - 1 - n0) * ldw + ksw);
  }
  // DMA instruction d of a stage: A and W alternate while both have
  // instructions left, then the remaining W ones
  auto dma_one = [&](int kt, int d) {
    const int s = kt % NSTAGE;
    if (d < 2 * DPW_A) {
      const int i = d >> 1, gi = i * GW + wave_u;
      if ((d & 1) == 0) lds_dma16(Ablk + kt * BK + a_off[i], &As(s)[gi * 64]);
      else lds_dma16(Wblk + kt * BK + w_off[i], &Ws(s)[gi * 64]);
    } else {
      const int i = d - DPW_A, gi = i * GW + wave_u;
      lds_dma16(Wblk + kt * BK + w_off[i], &Ws(s)[gi * 64]);
    }
  };
  auto issue = [&](int kt) {
#pragma unroll
    for (int d = 0; d < ND; ++d) dma_one(kt, d);
  };

  // operand read base of chunk c: row x*16 + ql, 16-byte chunk c*4 + g (the
  // stage swizzle of row x*16 + ql depends on ql only)
  int rbase[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) rbase[c] = ql * CPRW + ((c * 4 + g) ^ S::swz(ql));

  f32x4_t bvec[FI];
  auto load_bias = [&]() {
#pragma unroll
    for (int i = 0; i < FI; ++i)
      bvec[i] = bias != nullptr ? *reinterpret_cast<const f32x4_t*>(bias + min(n0 + w_row0 + i * 16 + 4 * g, N - 4))
                                : f32x4_t{0.f, 0.f, 0.f, 0.f};
  };

  f32x4_t acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int nk = K / BK;
  bf16x8_t fw[2][FI], fx[FJ];
  auto read_w = [&](int s, int c, int i, bf16x8_t (&dst)[FI]) {
    dst[i] = __builtin_bit_cast(bf16x8_t, Ws(s)[rbase[c] + (w_row0 + i * 16) * CPRW]);
  };
  auto read_x = [&](int s, int c, int j) {
    fx[j] = __builtin_bit_cast(bf16x8_t, As(s)[rbase[c] + (a_row0 + j * 16) * CPRW]);
  };
#pragma unroll
  for (int kt = 0; kt < NSTAGE; ++kt)
    if (kt < nk) issue(kt);
  S::dma_wait(min(NSTAGE - 1, nk - 1));
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FI; ++i) read_w(0, 0, i, fw[0]);
#pragma unroll
  for (int j = 0; j < FJ; ++j) read_x(0, 0, j);

  auto publish = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  };
  // group j of a chunk (operand set p for the feature fragments): the FI MFMAs of
  // token fragment j, then the reads of the next chunk (cn of stage sn): token
  // fragment j into fx[j] and this group's share of the feature fragments into
  // set p^1 (one every other group when FJ = 8, two per group when FJ = 2);
  // and DMA instructions j, j + FJ, ... of stage kd
  auto step = [&](int j, int p, int sn, int cn, int kd, bool reads, bool dmas) {
#pragma unroll
    for (int i = 0; i < FI; ++i)
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[p][i], fx[j], acc[i][j], 0, 0, 0);
    if (reads) {
      read_x(sn, cn, j);
      if (FJ >= FI) {
        if (j % (FJ / FI) == FJ / FI - 1) read_w(sn, cn, j / (FJ / FI), fw[p ^ 1]);
      } else {
#pragma unroll
        for (int i = j * (FI / FJ); i < (j + 1) * (FI / FJ); ++i) read_w(sn, cn, i, fw[p ^ 1]);
      }
    }
    if (dmas) {
#pragma unroll
      for (int d = j; d < ND; d += FJ) dma_one(kd, d);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  static_assert((FJ % FI == 0 || FI % FJ == 0) && (NCH % 2 == 0 || NCH == 1), "group layout");
  // with one chunk per stage the next stage's feature fragments land in set 1:
  // swap the two sets after each stage (4 fragments, only the 32-k stage path)
  auto rotate = [&]() {
    if (NCH % 2 == 1) {
#pragma unroll
      for (int i = 0; i < FI; ++i) {
        const bf16x8_t t = fw[0][i];
        fw[0][i] = fw[1][i];
        fw[1][i] = t;
      }
    }
  };
  int kt = 0;
  for (; kt + NSTAGE < nk; ++kt) {
    const int s = kt % NSTAGE;
#pragma unroll
    for (int c = 0; c + 1 < NCH; ++c)
#pragma unroll
      for (int j = 0; j < FJ; ++j) step(j, c & 1, s, c + 1, 0, true, false);
    S::dma_wait(NSTAGE - 2);
    publish();
#pragma unroll
    for (int j = 0; j < FJ; ++j) step(j, (NCH - 1) & 1, (kt + 1) % NSTAGE, 0, kt + NSTAGE, true, true);
    rotate();
  }
  for (; kt < nk; ++kt) {
    const int s = kt % NSTAGE;
#pragma unroll
    for (int c = 0; c + 1 < NCH; ++c)
#pragma unroll
      for (int j = 0; j < FJ; ++j) step(j, c & 1, s, c + 1, 0, true, false);
    const bool next = kt + 1 < nk;
    if (next) {
      S::dma_wait(nk - 2 - kt);
      publish();
    }
#pragma unroll
    for (int j = 0; j < FJ; ++j) step(j, (NCH - 1) & 1, (kt + 1) % NSTAGE, 0, 0, next, false);
    rotate();
  }
  __syncthreads();
  load_bias();

  if (EPI == EPI_F32) {
#pragma unroll
    for (int j = 0; j < FJ; ++j) {
      const int m = m0 + a_row0 + j * 16 + ql;
      if (m >= M) continue;
#pragma unroll
      for (int i = 0; i < FI; ++i) {
        const int n = n0 + w_row0 + i * 16 + 4 * g;
        if (n >= N) continue;
        *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(Cv) + (int64_t)m * ldc + n) = acc[i][j] + bvec[i];
      }
    }
    return;
  }
  // bf16 epilogues through a per-wave LDS tile [WTM tokens][WTN features]: 8-byte
  // unit u (features 4u..4u+3) of row t stored at u ^ (2 * ((t >> 1) & 7)), so the
  // 16 rows of one write hit distinct banks and 16-byte unit pairs stay together.
  constexpr int CPR = WTN / 8;
  constexpr int RPP = 64 / CPR;
  constexpr int NPASS = WTM / RPP;
  constexpr bool HAS_RES = EPI == EPI_GATE_RES || EPI == EPI_RES;
  const int c8 = lane % CPR;
  const int n = n0 + w_row0 + c8 * 8;
  const int mrow = m0 + a_row0 + lane / CPR;
  u32x4_t res[HAS_RES ? NPASS : 1];
  if (HAS_RES) {
#pragma unroll
    for (int r = 0; r < NPASS; ++r) {
      const int m = mrow + r * RPP;
      res[r] = (m < M && n < N) ? *reinterpret_cast<const u32x4_t*>(R + (int64_t)m * ldr + n) : u32x4_t{0, 0, 0, 0};
    }
  }
  int seg_lo = 0;
  bool one_seg = true;
  f32x4_t g0 = {0.f, 0.f, 0.f, 0.f}, g1 = {0.f, 0.f, 0.f, 0.f};
  if (EPI == EPI_GATE_RES) {
    seg_lo = find_segment(cu, nseg, row_base + m0 + a_row0);
    one_seg = seg_lo == find_segment(cu, nseg, row_base + min(m0 + a_row0 + WTM, M) - 1);
    if (one_seg && n < N) {
      const float* gp = gate + (int64_t)seg_lo * gate_stride + n;
      g0 = *reinterpret_cast<const f32x4_t*>(gp);
      g1 = *reinterpret_cast<const f32x4_t*>(gp + 4);
    }
  }
  u32x2_t* stage8 = reinterpret_cast<u32x2_t*>(lds + wave_u * (WTM * CPR));
  const u32x4_t* stage16 = lds + wave_u * (WTM * CPR);
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) {
      const int t = j * 16 + ql;
      const int u = (i * 4 + g) ^ (2 * ((t >> 1) & 7));
      const f32x4_t y = acc[i][j] + bvec[i];
      stage8[t * (2 * CPR) + u] = u32x2_t{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3])};
    }
  __syncthreads();
  if (n >= N) return;
#pragma unroll
  for (int r = 0; r < NPASS; ++r) {
    const int t = r * RPP + lane / CPR;
    const int m = mrow + r * RPP;
    if (m >= M) continue;
    u32x4_t v = stage16[t * CPR + (c8 ^ ((t >> 1) & 7))];
    if (EPI != EPI_BIAS) {
      float x[8];
      unpack8(v, x);
      if (EPI == EPI_GELU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = gelu_tanh_f(x[e]);
      } else if (EPI == EPI_SILU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = silu_f(x[e]);
      } else {
        float rv[8];
        unpack8(res[HAS_RES ? r : 0], rv);
        if (EPI == EPI_GATE_RES) {
          f32x4_t h0 = g0, h1 = g1;
          if (!one_seg) {
            const float* gp = gate + (int64_t)find_segment(cu, nseg, row_base + m) * gate_stride + n;
            h0 = *reinterpret_cast<const f32x4_t*>(gp);
            h1 = *reinterpret_cast<const f32x4_t*>(gp + 4);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[e] = fmaf(x[e], h0[e], rv[e]);
            x[e + 4] = fmaf(x[e + 4], h1[e], rv[e + 4]);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = rv[e] + x[e];
        }
      }
      v = pack8(x);
    }
    u32x4_t* dst = reinterpret_cast<u32x4_t*>(reinterpret_cast<bf16_t*>(Cv) + (int64_t)m * ldc + n);
    if (STREAM) __builtin_nontemporal_store(v, dst);
    else *dst = v;
  }
}

// Up to 16 rows by many features (SD3.5's stacked modulations of a step: 2 rows by
// 499 k features of K = 1536, 1.5 GB of weights): bound by streaming the weights
// once.  One wave computes 16 features for all rows with the weights straight from
// global memory into MFMA operands (no LDS, no barriers, no tile of 254 idle rows):
// lane l loads 16 bytes of weight row n0 + l % 16 at k 8 (l / 16), a batch of SK_U
// 32-k chunks ahead of the MFMAs: 341 -> 292 us, 4.5 -> 5.25 TB/s.  Fewer features
// are bound by one wave's walk along K and gain nothing (9216: 10.8 against 11.0 us,
// 1536: 5.5 against 6.2).  Same MFMA, k order, bias add and rounding as gemm_kernel:
// bitwise its results.
constexpr int kSkinnyM = 16, kSkinnyN = 16384;
constexpr int SK_U = 8;
template <int EPI>
__global__ __launch_bounds__(256) void gemm_skinny(
    const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W, int64_t ldw,
    const float* __restrict__ bias, void* __restrict__ Cv, int64_t ldc, int M, int N, int K, const bf16_t* R,
    int64_t ldr, const float* __restrict__ gate, int64_t gate_stride, const int32_t* __restrict__ cu, int nseg) {
  const int lane = threadIdx.x & 63, ql = lane & 15, g = lane >> 4;
  const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
  if (n0 >= N) return;
  const bf16_t* wp = W + (int64_t)min(n0 + ql, N - 1) * ldw + g * 8;
  const bf16_t* xp = A + (int64_t)min(ql, M - 1) * lda + g * 8;
  const int chunks = K / 32;
  bf16x8_t w[2][SK_U], x[2][SK_U];
  auto load = [&](int set, int c0) {
#pragma unroll
    for (int u = 0; u < SK_U; ++u) {
      const int c = min(c0 + u, chunks - 1);  // past the end: the last chunk again, not used
      w[set][u] = *reinterpret_cast<const bf16x8_t*>(wp + (int64_t)c * 32);
      x[set][u] = *reinterpret_cast<const bf16x8_t*>(xp + (int64_t)c * 32);
    }
  };
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  auto use = [&](int set, int c0) {
#pragma unroll
    for (int u = 0; u < SK_U; ++u)
      if (c0 + u < chunks) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[set][u], x[set][u], acc, 0, 0, 0);
  };
  load(0, 0);
  for (int c = 0; c < chunks; c += 2 * SK_U) {
    load(1, c + SK_U);
    use(0, c);
    load(0, c + 2 * SK_U);
    use(1, c + SK_U);
  }
  // this lane: row ql, features n .. n + 3
  const int n = n0 + 4 * g;
  if (ql >= M || n >= N) return;
  const f32x4_t y = acc + (bias != nullptr ? *reinterpret_cast<const f32x4_t*>(bias + n) : f32x4_t{0.f, 0.f, 0.f, 0.f});
  if (EPI == EPI_F32) {
    *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(Cv) + (int64_t)ql * ldc + n) = y;
    return;
  }
  auto lo = [](uint32_t w2) { return __uint_as_float(w2 << 16); };
  auto hi = [](uint32_t w2) { return __uint_as_float(w2 & 0xffff0000u); };
  u32x2_t v{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3])};
  if (EPI != EPI_BIAS) {
    float f[4] = {lo(v[0]), hi(v[0]), lo(v[1]), hi(v[1])};
    if (EPI == EPI_GELU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = gelu_tanh_f(f[e]);
    } else if (EPI == EPI_SILU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = silu_f(f[e]);
    } else {
      const u32x2_t r = *reinterpret_cast<const u32x2_t*>(R + (int64_t)ql * ldr + n);
      const float rv[4] = {lo(r[0]), hi(r[0]), lo(r[1]), hi(r[1])};
      if (EPI == EPI_GATE_RES) {
        const f32x4_t h = *reinterpret_cast<const f32x4_t*>(gate + (int64_t)find_segment(cu, nseg, ql) * gate_stride + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = fmaf(f[e], h[e], rv[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = rv[e] + f[e];
      }
    }
    v = u32x2_t{pack_bf2(f[0], f[1]), pack_bf2(f[2], f[3])};
  }
  *reinterpret_cast<u32x2_t*>(reinterpret_cast<bf16_t*>(Cv) + (int64_t)ql * ldc + n) = v;
}

template <int EPI>
int launch_skinny(const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C, int64_t ldc,
                  int M, int N, int K, const void* R, int64_t ldr, const float* gate, int64_t gate_stride,
                  const int32_t* cu, int nseg, hipStream_t stream) {
  gemm_skinny<EPI><<<(unsigned)((N + 63) / 64), 256, 0, stream>>>((const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, C,
                                                                 ldc, M, N, K, (const bf16_t*)R, ldr, gate,
                                                                 gate_stride, cu, nseg);
  return ditk_check_launch("ditk_gemm");
}

// One wave per SIMD (every epilogue but fp32, K % 64 == 0): a workgroup tile as
// four wave tiles, their accumulators in the AGPRs (all 256 of them for the
// 256 x 256 tile's 128 x 128 wave tiles).  The k loop and the bf16 staging are
// generated assembly (gen_gemm.py -> gemm_l4_*_body.inc: 64-k stages through
// NBUF LDS buffers filled by direct DMA, the next chunk's fragments read under
// the current MFMAs); this C++ part computes the per-lane addresses and runs the
// same epilogue arithmetic as gemm_kernel on the staged rows.  Same MFMA
// (16x16x32, W rows as the A operand), same k order, same bias add and rounding:
// bitwise equal to gemm_kernel.
// A wave tile is FI feature and FJ token fragments of 16; the six tiles generated
// are listed with their times at kL4 below.  What bounds them, by counters at K =
// 8192-8960: a 256 x 256 tile's stage takes 2464 cycles, 2048 of them MFMA (83%); a
// 128 x 128 one 845 for 512 (60%), a 128 x 96 one 707 for 384 (54%).  Waves wait for 9,
// 12 and 15% of their time, and the LDS reads of a 128 x 128 stage take 262 cycles
// without bank conflicts, so what a smaller tile adds is mostly issue: the one wave of a
// SIMD issues as many reads, DMAs and address instructions for fewer MFMAs.
// (1560 x 1536 x 8960 on 64 x 128 tiles of gemm_kernel 81 us, 128 x 96 here 54 us;
// 2048 x 6144 x 1536 on 256 x 192 as before.)
template <int FI, int FJ>
struct L4 {
  static constexpr int WTM = 16 * FJ, WTN = 16 * FI, GBM = 2 * WTM, GBN = 2 * WTN;
  static constexpr int NBUF = FJ == 8 ? 2 : FI >= 6 ? 3 : FI == 3 ? 5 : 4;  // stage buffers, as generated
  static constexpr int BUF = (GBM + GBN) * 128;            // one 64-k stage: A rows, then W rows
  static constexpr int STG_ROW = 2 * WTN + 16;             // staging row bytes
  // the stage buffers and the prefetch's spare line, or the staging rows
  static constexpr int LDS_BYTES = NBUF * BUF + 1024 > 4 * WTM * STG_ROW ? NBUF * BUF + 1024 : 4 * WTM * STG_ROW;
};
#define DITK_L4_OPERANDS                                                                                        \
  [a_lo] "s"(su((uint32_t)abase)), [a_hi] "s"(su((uint32_t)(abase >> 32))), [w_lo] "s"(su((uint32_t)wbase)),   \
      [w_hi] "s"(su((uint32_t)(wbase >> 32))), [nk] "s"(su(K / 64)), [lds] "s"(su(lds0)),                       \
      [wave1k] "s"(su(wave_u * 1024u)), [pf_lo] "s"(su((uint32_t)(uint64_t)(uintptr_t)W)),                       \
      [pf_hi] "s"(su((uint32_t)((uint64_t)(uintptr_t)W >> 32))), [pfn] "s"(su(pf.n)), [pfn0] "s"(su(pf.n0)),     \
      [pflpr] "s"(su(pf.lines)), [pfstep] "s"(su(pf.lines * 128u)), [pfmax] "v"(pf_max), [pfoff] "v"(pf_off), [rdx00] "v"(rdx[0][0]), [rdx01] "v"(rdx[0][1]), [rdx10] "v"(rdx[1][0]), \
      [rdx11] "v"(rdx[1][1]), [rdx20] "v"(rdx[2][0]), [rdx21] "v"(rdx[2][1]), [rdx30] "v"(rdx[3][0]),           \
      [rdx31] "v"(rdx[3][1]), [rdx40] "v"(rdx[4][0]), [rdx41] "v"(rdx[4][1]), [rdw00] "v"(rdw[0][0]),           \
      [rdw01] "v"(rdw[0][1]), [rdw10] "v"(rdw[1][0]), [rdw11] "v"(rdw[1][1]), [rdw20] "v"(rdw[2][0]),           \
      [rdw21] "v"(rdw[2][1]), [rdw30] "v"(rdw[3][0]), [rdw31] "v"(rdw[3][1]), [rdw40] "v"(rdw[4][0]),           \
      [rdw41] "v"(rdw[4][1]), [aoff0] "v"(aoff[0]), [aoff1] "v"(aoff[1]), [aoff2] "v"(aoff[2]),                 \
      [aoff3] "v"(aoff[3]), [aoff4] "v"(aoff[4]), [aoff5] "v"(aoff[5]), [aoff6] "v"(aoff[6]),                   \
      [aoff7] "v"(aoff[7]), [woff0] "v"(woff[0]), [woff1] "v"(woff[1]), [woff2] "v"(woff[2]),                   \
      [woff3] "v"(woff[3]), [woff4] "v"(woff[4]), [woff5] "v"(woff[5]), [woff6] "v"(woff[6]),                   \
      [woff7] "v"(woff[7]), [stg] "v"(stg), [b0] "v"(bv[0]), [b1] "v"(bv[1]), [b2] "v"(bv[2]), [b3] "v"(bv[3]),  \
      [b4] "v"(bv[4]), [b5] "v"(bv[5]), [b6] "v"(bv[6]), [b7] "v"(bv[7]), [b8] "v"(bv[8]), [b9] "v"(bv[9]),      \
      [b10] "v"(bv[10]), [b11] "v"(bv[11]), [b12] "v"(bv[12]), [b13] "v"(bv[13]), [b14] "v"(bv[14]),            \
      [b15] "v"(bv[15]), [b16] "v"(bv[16]), [b17] "v"(bv[17]), [b18] "v"(bv[18]), [b19] "v"(bv[19]),            \
      [b20] "v"(bv[20]), [b21] "v"(bv[21]), [b22] "v"(bv[22]), [b23] "v"(bv[23]), [b24] "v"(bv[24]),            \
      [b25] "v"(bv[25]), [b26] "v"(bv[26]), [b27] "v"(bv[27]), [b28] "v"(bv[28]), [b29] "v"(bv[29]),            \
      [b30] "v"(bv[30]), [b31] "v"(bv[31])
// Weight prefetch (see prefetch_start in gen_gemm.py): the launch's `count`
// workgroups together touch every 128-byte line of W [N, K] once, in k order, a
// batch of `lines` 64-k stages of all rows at a time and a few stages ahead of
// their use, so that only the first reader of a line waits for HBM.
struct L4Prefetch {
  uint32_t n = 0, n0 = 0, lines = 1;  // batches, batches before the k loop, lines per row and batch
  int rank = 0;
};
__device__ __forceinline__ L4Prefetch l4_prefetch(int rank, int count, int N, int K, bool on) {
  L4Prefetch p;
  p.lines = (uint32_t)(count * 256) / (uint32_t)N;
  if (!on || p.lines == 0) return L4Prefetch{};
  p.n = ((uint32_t)(K / 64) + p.lines - 1) / p.lines;
  p.n0 = min(p.n, 1 + (8 + p.lines - 1) / p.lines);
  p.rank = rank;
  return p;
}
template <int EPI, int FI, int FJ>
__device__ __forceinline__ void l4_tile(u32x4_t* lds, int L, const bf16_t* __restrict__ A, int64_t lda,
                                        const bf16_t* __restrict__ W, int64_t ldw, const float* __restrict__ bias,
                                        void* __restrict__ Cv, int64_t ldc, int M, int N, int K, const bf16_t* R,
                                        int64_t ldr, const float* __restrict__ gate, int64_t gate_stride,
                                        const int32_t* __restrict__ cu, int nseg, int tiles_m, int tiles_n,
                                        int group_m, L4Prefetch pf, bool stream_out,
                                        int row_base);
template <int EPI, int FI, int FJ>
__global__ __launch_bounds__(256, 1) void gemm_kernel_l4(
    const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W, int64_t ldw,
    const float* __restrict__ bias, void* __restrict__ Cv, int64_t ldc, int M, int N, int K,
    const bf16_t* R, int64_t ldr, const float* __restrict__ gate, int64_t gate_stride,
    const int32_t* __restrict__ cu, int nseg, int tiles_m, int tiles_n, int group_m, bool prefetch, bool stream_out,
    int row_base) {
  __shared__ u32x4_t lds[L4<FI, FJ>::LDS_BYTES / 16];
  // Persistent: XCD x (= blockIdx % 8) owns the tiles [x * per_xcd, (x + 1) *
  // per_xcd), which its workgroups take in turn (the order a one-tile-per-
  // workgroup launch would run them in), so each workgroup loads its kernel
  // arguments once and a tile's k loop starts while the previous tile's
  // stores drain.
  const int nb = gridDim.x, b = blockIdx.x;
  const int ntiles = tiles_m * tiles_n, per_xcd = (ntiles + 7) / 8;
  const int tlo = (b & 7) * per_xcd, thi = min(tlo + per_xcd, ntiles);
  // the epilogue's arguments are loaded here, under the first stages' DMA: first
  // touched after the k loop, they cost a trip to memory (2 us of 18 at
  // 2560 x 1536 x 1536)
  if (EPI == EPI_GATE_RES) asm volatile("" ::"s"(R), "s"(ldr), "s"(gate), "s"(gate_stride), "s"(cu), "s"(nseg), "s"(row_base));
  if (EPI == EPI_RES) asm volatile("" ::"s"(R), "s"(ldr));
  asm volatile("" ::"s"(Cv), "s"(ldc));
  L4Prefetch pf = l4_prefetch(b, nb, N, K, prefetch);
  for (int L = tlo + (b >> 3); L < thi; L += nb >> 3) {
    l4_tile<EPI, FI, FJ>(lds, L, A, lda, W, ldw, bias, Cv, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, tiles_m,
                     tiles_n, group_m, pf, stream_out, row_base);
    pf.n = 0;  // once per workgroup
  }
}

// One product of a paired launch (see gemm_kernel_l4_pair).
struct L4Prob {
  const bf16_t* A;
  int64_t lda;
  const bf16_t* W;
  int64_t ldw;
  const float* bias;
  void* C;
  int64_t ldc;
  const bf16_t* R;
  int64_t ldr;
  const float* gate;
  int64_t gate_stride;
  const int32_t* cu;
  int nseg, M, N, tiles_m, tiles_n, group_m;
};

// Two products of the same K and epilogue (their own inputs, features, weights,
// bias, residual, gate and segments) in one persistent launch: the tile list is the
// first product's tiles, then the second's, taken per XCD as gemm_kernel_l4
// takes one product's.  Each tile is computed exactly as a launch of its own
// product would compute it.
template <int EPI, int FI, int FJ>
__global__ __launch_bounds__(256, 1) void gemm_kernel_l4_pair(L4Prob p0, L4Prob p1, int K, bool prefetch, bool stream_out) {
  __shared__ u32x4_t lds[L4<FI, FJ>::LDS_BYTES / 16];
  const int nb = gridDim.x, b = blockIdx.x;
  const int t0 = p0.tiles_m * p0.tiles_n, ntiles = t0 + p1.tiles_m * p1.tiles_n, per_xcd = (ntiles + 7) / 8;
  const int tlo = (b & 7) * per_xcd, thi = min(tlo + per_xcd, ntiles);
  // Workgroups in the order of their first tiles: the first c0 start in product 0
  // and prefetch its weights, the others product 1's.
  const int wpx = nb >> 3, x0 = t0 / per_xcd, rank = (b & 7) * wpx + (b >> 3);
  const int c0 = min(nb, x0 * wpx + min(t0 - x0 * per_xcd, wpx));
  L4Prefetch pf = rank < c0 ? l4_prefetch(rank, c0, p0.N, K, prefetch)
                            : l4_prefetch(rank - c0, nb - c0, p1.N, K, prefetch);
  for (int L = tlo + (b >> 3); L < thi; L += nb >> 3) {
    const bool s = L >= t0;  // wave-uniform: the fields below are scalar selects
    l4_tile<EPI, FI, FJ>(lds, s ? L - t0 : L, s ? p1.A : p0.A, s ? p1.lda : p0.lda, s ? p1.W : p0.W,
                     s ? p1.ldw : p0.ldw, s ? p1.bias : p0.bias, s ? p1.C : p0.C, s ? p1.ldc : p0.ldc,
                     s ? p1.M : p0.M, s ? p1.N : p0.N, K, s ? p1.R : p0.R, s ? p1.ldr : p0.ldr, s ? p1.gate : p0.gate,
                     s ? p1.gate_stride : p0.gate_stride, s ? p1.cu : p0.cu, s ? p1.nseg : p0.nseg,
                     s ? p1.tiles_m : p0.tiles_m, s ? p1.tiles_n : p0.tiles_n, s ? p1.group_m : p0.group_m, pf,
                         stream_out, 0);
    pf.n = 0;
  }
}

template <int EPI, int FI, int FJ>
__device__ __forceinline__ void l4_tile(u32x4_t* lds, int L, const bf16_t* __restrict__ A, int64_t lda,
                                        const bf16_t* __restrict__ W, int64_t ldw, const float* __restrict__ bias,
                                        void* __restrict__ Cv, int64_t ldc, int M, int N, int K, const bf16_t* R,
                                        int64_t ldr, const float* __restrict__ gate, int64_t gate_stride,
                                        const int32_t* __restrict__ cu, int nseg, int tiles_m, int tiles_n,
                                        int group_m, L4Prefetch pf, bool stream_out,
                                        int row_base) {
  using G = L4<FI, FJ>;
  constexpr int GBM = G::GBM, GBN = G::GBN, WTM = G::WTM, WTN = G::WTN, STG_ROW = G::STG_ROW;
  const int group = L / (group_m * tiles_n);
  const int first_m = group * group_m;
  const int gm = min(group_m, tiles_m - first_m);
  const int pid = L % (group_m * tiles_n);
  const int mt = first_m + pid % gm, nt = pid / gm;
  const int m0 = mt * GBM, n0 = nt * GBN;

  // the lane's values are recomputed per tile (an opaque copy of the thread id
  // keeps them out of the registers that stay live across the k loop)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int ql = lane & 15, g = lane >> 4;
  const int wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int a_row0 = (wave_u & 1) * WTM, w_row0 = (wave_u >> 1) * WTN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4_t*)&lds[0];
  // fragment reads of 32-k chunk c: row ql of a 16-row fragment, 16-byte unit
  // 4 c + g of its 64 k, stored at unit (4 c + g) ^ ((row >> 1) & 7) of the
  // 128-byte LDS row (as gemm_kernel's 64-k stages)
  uint32_t rdx[5][2] = {}, rdw[5][2] = {};
#pragma unroll
  for (int s = 0; s < G::NBUF; ++s)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const uint32_t lane_part = (uint32_t)(ql * 128 + (((c * 4 + g) ^ ((ql >> 1) & 7)) * 16));
      rdx[s][c] = lds0 + s * G::BUF + a_row0 * 128 + lane_part;
      rdw[s][c] = lds0 + s * G::BUF + GBM * 128 + w_row0 * 128 + lane_part;
    }
  // DMA instruction d of this wave fills rows 8 (4 d + wave) .. +7 (1 KiB):
  // lane l -> row l / 8, LDS unit l % 8 <- k unit (l % 8) ^ ((row >> 1) & 7)
  uint32_t aoff[8], woff[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const int row = (d * 4 + wave_u) * 8 + lane / 8;
    const int usw = ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    aoff[d] = d < FJ ? (uint32_t)((int64_t)min(row, M - 1 - m0) * lda * 2 + usw) : 0u;
    woff[d] = d < FI ? (uint32_t)((int64_t)min(row, N - 1 - n0) * ldw * 2 + usw) : 0u;
  }
  // this lane's prefetch row (of lane 256 rank + tid over `lines` lanes a row) and
  // the first and last of its lines, as byte offsets into W
  const uint32_t pf_lane = (uint32_t)(pf.rank * 256 + tid), pf_row = min(pf_lane / pf.lines, (uint32_t)(N - 1));
  const uint32_t pf_base = pf_row * (uint32_t)(ldw * 2), pf_off = pf_base + (pf_lane % pf.lines) * 128u;
  const uint32_t pf_max = pf_base + (uint32_t)(K / 64 - 1) * 128u;
  const uint32_t stg = lds0 + wave_u * (WTM * STG_ROW) + ql * STG_ROW + g * 8;
  float bv[32];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const f32x4_t x = bias != nullptr && i < FI
                          ? *reinterpret_cast<const f32x4_t*>(bias + min(n0 + w_row0 + i * 16 + 4 * g, N - 4))
                          : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) bv[i * 4 + e] = x[e];
  }
  auto su = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
  const uint64_t abase = (uint64_t)(uintptr_t)(A + (int64_t)m0 * lda);
  const uint64_t wbase = (uint64_t)(uintptr_t)(W + (int64_t)n0 * ldw);
  static_assert(FI == 8 || FI == 6 || (FJ == 4 && (FI == 4 || FI == 3)), "a generated wave tile");
  if constexpr (FI == 8 && FJ == 8)
    asm volatile(
#include "gemm_l4_256x256_body.inc"
        : : DITK_L4_OPERANDS : DITK_GEMM_L4_CLOBBERS "scc", "memory");
  else if constexpr (FI == 6 && FJ == 8)
    asm volatile(
#include "gemm_l4_256x192_body.inc"
        : : DITK_L4_OPERANDS : DITK_GEMM_L4_CLOBBERS "scc", "memory");
  else if constexpr (FI == 8 && FJ == 4)
    asm volatile(
#include "gemm_l4_128x256_body.inc"
        : : DITK_L4_OPERANDS : DITK_GEMM_L4_CLOBBERS "scc", "memory");
  else if constexpr (FI == 6 && FJ == 4)
    asm volatile(
#include "gemm_l4_128x192_body.inc"
        : : DITK_L4_OPERANDS : DITK_GEMM_L4_CLOBBERS "scc", "memory");
  else if constexpr (FI == 4 && FJ == 4)
    asm volatile(
#include "gemm_l4_128x128_body.inc"
        : : DITK_L4_OPERANDS : DITK_GEMM_L4_CLOBBERS "scc", "memory");
  else if constexpr (FI == 3 && FJ == 4)
    asm volatile(
#include "gemm_l4_128x96_body.inc"
        : : DITK_L4_OPERANDS : DITK_GEMM_L4_CLOBBERS "scc", "memory");

  // epilogue on this wave's staged rows (the wave wrote them and waited for them).
  // The output (and residual) rows go through buffer descriptors whose range
  // ends at the last row of the matrix: a store past it is dropped and a load
  // returns 0, so the passes have no branches and the staged-row reads and
  // residual loads of many passes are in flight together.
  constexpr int CPR = WTN / 8;                    // 16-byte units per row (16, 12, 8 or 6)
  constexpr int RPP = 64 / CPR;                   // rows per pass (4, 5, 8 or 10; lanes past RPP * CPR idle)
  constexpr int NPASS = (WTM + RPP - 1) / RPP;
  constexpr bool HAS_RES = EPI == EPI_GATE_RES || EPI == EPI_RES;
  constexpr uint32_t kOut = 0x80000000u;          // an offset past every descriptor's range
  const int row0 = m0 + a_row0;                   // this wave tile's first row
  const int rows = max(0, min(WTM, M - row0));    // its rows inside the matrix
  const uint32_t ldc2 = (uint32_t)(ldc * 2), ldr2 = (uint32_t)(ldr * 2);
  // descriptors from wave-uniform (scalar) base addresses
  auto sptr = [&](const void* p) {
    const uint64_t x = (uint64_t)(uintptr_t)p;
    const uint64_t lo = su((uint32_t)x), hi = su((uint32_t)(x >> 32));
    return reinterpret_cast<void*>((uintptr_t)(lo | (hi << 32)));
  };
  const int rec_c = (int)su((uint32_t)rows * ldc2), rec_r = (int)su((uint32_t)rows * ldr2);
  const __amdgpu_buffer_rsrc_t cdesc = __builtin_amdgcn_make_buffer_rsrc(
      sptr(reinterpret_cast<bf16_t*>(Cv) + (int64_t)row0 * ldc + n0 + w_row0), 0, rec_c, 0x00020000);
  const __amdgpu_buffer_rsrc_t rdesc = __builtin_amdgcn_make_buffer_rsrc(
      sptr(HAS_RES ? R + (int64_t)row0 * ldr + n0 + w_row0 : nullptr), 0, HAS_RES ? rec_r : 0, 0x00020000);
  const int c8 = lane % CPR;
  const int n = n0 + w_row0 + c8 * 8;
  const bool lane_on = n < N && lane < RPP * CPR;   // lanes past N or past a pass's units store nothing
  const char* stage = reinterpret_cast<const char*>(lds) + wave_u * (WTM * STG_ROW);
  int seg_lo = 0;
  bool one_seg = true;
  f32x4_t g0 = {0.f, 0.f, 0.f, 0.f}, g1 = {0.f, 0.f, 0.f, 0.f};
  if (EPI == EPI_GATE_RES) {
    seg_lo = find_segment(cu, nseg, row_base + min(row0, M - 1));
    one_seg = seg_lo == find_segment(cu, nseg, row_base + min(row0 + WTM, M) - 1);
    if (one_seg) {
      const float* gp = gate + (int64_t)seg_lo * gate_stride + min(n, N - 8);
      g0 = *reinterpret_cast<const f32x4_t*>(gp);
      g1 = *reinterpret_cast<const f32x4_t*>(gp + 4);
    }
  }
  // every residual row is loaded first (one latency for the tile), then the
  // staged rows are read and stored in batches of RB passes
  u32x4_t res[HAS_RES ? NPASS : 1];
  if (HAS_RES) {
#pragma unroll
    for (int r = 0; r < NPASS; ++r) {
      const int t = r * RPP + lane / CPR;
      res[r] = __builtin_amdgcn_raw_buffer_load_b128(rdesc, t < rows && lane_on ? (uint32_t)t * ldr2 + c8 * 16 : kOut, 0, 0);
    }
  }
  constexpr int RB = 8;
#pragma unroll
  for (int r0 = 0; r0 < NPASS; r0 += RB) {
    u32x4_t v[RB];
    uint32_t off[RB];
#pragma unroll
    for (int q = 0; q < RB && r0 + q < NPASS; ++q) {
      const int t = (r0 + q) * RPP + lane / CPR;  // row in the wave tile
      off[q] = t < rows && lane_on ? (uint32_t)t * ldc2 + c8 * 16 : kOut;
      v[q] = *reinterpret_cast<const u32x4_t*>(stage + min(t, WTM - 1) * STG_ROW + c8 * 16);
    }
#pragma unroll
    for (int q = 0; q < RB && r0 + q < NPASS; ++q) {
      if (EPI != EPI_BIAS) {
        float x[8];
        unpack8(v[q], x);
        if (EPI == EPI_GELU) {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = gelu_tanh_f(x[e]);
        } else if (EPI == EPI_SILU) {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = silu_f(x[e]);
        } else {
          float rv[8];
          unpack8(res[HAS_RES ? r0 + q : 0], rv);
          if (EPI == EPI_GATE_RES) {
            f32x4_t h0 = g0, h1 = g1;
            if (!one_seg) {
              const int m = min(row0 + (r0 + q) * RPP + lane / CPR, M - 1);
              const float* gp = gate + (int64_t)find_segment(cu, nseg, row_base + m) * gate_stride + min(n, N - 8);
              h0 = *reinterpret_cast<const f32x4_t*>(gp);
              h1 = *reinterpret_cast<const f32x4_t*>(gp + 4);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x[e] = fmaf(x[e], h0[e], rv[e]);
              x[e + 4] = fmaf(x[e + 4], h1[e], rv[e + 4]);
            }
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = rv[e] + x[e];
          }
        }
        v[q] = pack8(x);
      }
      if (stream_out) __builtin_amdgcn_raw_buffer_store_b128(v[q], cdesc, off[q], 0, 2);  // non-temporal
      else __builtin_amdgcn_raw_buffer_store_b128(v[q], cdesc, off[q], 0, 0);
    }
  }
}

// The tile configurations of gemm_kernel_l4: workgroup tile (tokens x features)
// and its measured time in us, start + rounds x (tile + stage x K / 64) with a round
// one tile per CU (least squares over 14 weight shapes of the Wan and SD3.5 blocks,
// 8 to 28000 rows, weights from HBM; 8-9% rms.  Longer products lose clock and take
// more, 56400 x 1536 x 8960 1199 us for 949 predicted; there it only ranks the
// tiles).  A 256 x 256 tile's stage does 1.78 PFLOP/s over the chip, a 128 x 96 one's
// 1.06, but the small tiles let 1000-row products use most of the CUs.
struct L4Cfg {
  int gbm, gbn;
  float start, tile, stage;
};
constexpr int kL4Cfgs = 6;
constexpr L4Cfg kL4[kL4Cfgs] = {{256, 256, -4.4f, 10.2f, 1.207f}, {256, 192, -2.3f, 6.6f, 1.054f},
                                {128, 256, -0.1f, 5.1f, 0.744f},  {128, 192, 0.6f, 3.7f, 0.592f},
                                {128, 128, 1.2f, 2.6f, 0.439f},   {128, 96, 1.7f, 2.5f, 0.381f}};

// Tile order of gemm_kernel_l4.  Up to two rounds of tiles, all of an XCD's tiles
// run about together, so its block of them is made about square in operand rows:
// it then pulls the fewest operand bytes into its L2 (2048 x 1536 x 8960: 63.5 us
// in the long-K order below, 61 us in groups of 4-6 m-tiles).  More rounds:
// gemm_group_m's orders.
int l4_group_m(int64_t tiles_m, int64_t tiles_n, int gbm, int gbn, int K) {
  const int64_t tiles = tiles_m * tiles_n, per_xcd = (tiles + 7) / 8;
  if (tiles > 2 * ditk_cu_count()) return gemm_group_m(K, (int)tiles_n);
  int64_t g = 1;
  while (g < tiles_m && (g + 1) * (g + 1) * gbm <= per_xcd * gbn) ++g;
  const int64_t groups = (tiles_m + g - 1) / g;
  return (int)((tiles_m + groups - 1) / groups);
}

// Whether a launch prefetches its weights (see L4Prefetch).  Where every tile row
// is full, the workgroups run in step and all wait for HBM at the first touch of
// each weight line: 2048 x 1536 x 8960 at 128 x 128 tiles 78 -> 61 us, x 6144
// 55 -> 42 us, 6400 x 1536 x 8960 at 256 x 192 160 -> 142 us, 4608 x 1536 33.0 ->
// 29.7 us.  A short last tile row (its missing rows re-read one row) runs ahead and
// does the same for nothing: with up to a third of a tile left the prefetch costs
// 0-3%, beyond that it wins by as much as with full tiles, but with 256-row tiles
// only at long K.  Few tile rows share too little: at 512 rows 11.7 -> 12.1 us
// (1536 x 1536) but 69 -> 55 us (1536 x 8960), at 100 rows (one) 55 -> 80 us.
bool l4_prefetch_on(int M, int N, int K, int64_t ldw, int gbm) {
  const int rem = M % gbm, tiles_m = (M + gbm - 1) / gbm;
  if (tiles_m < (K >= 4096 ? 4 : 8)) return false;
  return (int64_t)N * ldw * 2 < (1ll << 31) && (rem == 0 || (3 * rem > gbm && (gbm == 128 || K >= 4096)));
}
// Whether the output (all of it, where two launches write it) is stored past the caches.  Outputs of 64 MB and more
// are (2.6-3.6% faster on the K = 1536 products of 65520 rows: they would not stay
// cached until the next kernel reads them); smaller ones stay, and the next kernel
// finds them (one-frame Wan block 300 -> 281 us, preview step of 2 x 1280 rows
// 11.20 -> 10.90 ms, SD3.5 512 step 8.65 -> 8.37 ms; gated residual of K = N = 1536 on
// gemm_kernel and the AdaLN after it: 9300 rows 59.1 -> 57.8 us, 20000 113.2 -> 110.7;
// 21800 rows 129 past the caches, 132 in them).
bool stream_output(int64_t M, int N) { return M * N * 2 >= (64ll << 20); }
template <int EPI, int FI, int FJ>
int launch_l4(const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C, int64_t ldc,
              int M, int N, int K, const void* R, int64_t ldr, const float* gate, int64_t gate_stride,
              const int32_t* cu, int nseg, hipStream_t stream, int row_base, bool stream_out) {
  constexpr int GBM = L4<FI, FJ>::GBM, GBN = L4<FI, FJ>::GBN;
  const int tiles_m = (M + GBM - 1) / GBM, tiles_n = (N + GBN - 1) / GBN;
  // one persistent workgroup per CU (a multiple of 8: the same number per XCD)
  const int64_t nblocks = std::min<int64_t>(((int64_t)tiles_m * tiles_n + 7) / 8 * 8, std::max(8, ditk_cu_count() / 8 * 8));
  gemm_kernel_l4<EPI, FI, FJ><<<(unsigned)nblocks, 256, 0, stream>>>(
      (const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, C, ldc, M, N, K, (const bf16_t*)R, ldr, gate,
      gate_stride, cu, nseg, tiles_m, tiles_n, l4_group_m(tiles_m, tiles_n, GBM, GBN, K), l4_prefetch_on(M, N, K, ldw, GBM),
      stream_out, row_base);
  return ditk_check_launch("ditk_gemm");
}

template <int EPI, int FI, int FJ>
int launch_l4_pair(L4Prob p0, L4Prob p1, int K, hipStream_t stream) {
  constexpr int GBM = L4<FI, FJ>::GBM, GBN = L4<FI, FJ>::GBN;
  for (L4Prob* p : {&p0, &p1}) {
    p->tiles_m = (p->M + GBM - 1) / GBM;
    p->tiles_n = (p->N + GBN - 1) / GBN;
    p->group_m = l4_group_m(p->tiles_m, p->tiles_n, GBM, GBN, K);
  }
  const int64_t tiles = (int64_t)p0.tiles_m * p0.tiles_n + (int64_t)p1.tiles_m * p1.tiles_n;
  const int64_t nblocks = std::min<int64_t>((tiles + 7) / 8 * 8, std::max(8, ditk_cu_count() / 8 * 8));
  gemm_kernel_l4_pair<EPI, FI, FJ><<<(unsigned)nblocks, 256, 0, stream>>>(
      p0, p1, K, l4_prefetch_on(p0.M, p0.N, K, p0.ldw, GBM) && (int64_t)p1.N * p1.ldw * 2 < (1ll << 31),
      stream_output((int64_t)p0.M * p0.N + (int64_t)p1.M * p1.N, 1));
  return ditk_check_launch("ditk_gemm_pair");
}

template <int EPI, int BK, int T>
int launch_tile(const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C,
                int64_t ldc, int M, int N, int K, const void* R, int64_t ldr, const float* gate,
                int64_t gate_stride, const int32_t* cu, int nseg, hipStream_t stream, int row_base, bool stream_out) {
  using S = Stages<BK, T>;
  const int tiles_m = (M + S::GBM - 1) / S::GBM, tiles_n = (N + S::GBN - 1) / S::GBN;
  const int64_t tiles = (int64_t)tiles_m * tiles_n;
  const int64_t nblocks = (tiles + 7) / 8 * 8;
  DITK_REQUIRE(nblocks < (1ll << 31), "ditk_gemm: grid too large");
  constexpr bool kMayStream = T == TILE_LARGE && EPI != EPI_F32;
  auto kern = kMayStream && stream_out ? gemm_kernel<EPI, BK, T, kMayStream> : gemm_kernel<EPI, BK, T, false>;
  kern<<<(unsigned)nblocks, S::GW * 64, 0, stream>>>(
      (const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, C, ldc, M, N, K, (const bf16_t*)R, ldr, gate,
      gate_stride, cu, nseg, tiles_m, tiles_n, gemm_group_m(K, tiles_n), row_base);
  return ditk_check_launch("ditk_gemm");
}

// One product on the one-wave-per-SIMD kernel's tile configuration `cfg`.
template <int EPI>
int launch_l4_cfg(int cfg, const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C,
                  int64_t ldc, int M, int N, int K, const void* R, int64_t ldr, const float* gate,
                  int64_t gate_stride, const int32_t* cu, int nseg, hipStream_t stream, int row_base,
                  bool stream_out) {
  switch (cfg) {
    case 0: return launch_l4<EPI, 8, 8>(A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream, row_base, stream_out);
    case 1: return launch_l4<EPI, 6, 8>(A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream, row_base, stream_out);
    case 2: return launch_l4<EPI, 8, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream, row_base, stream_out);
    case 3: return launch_l4<EPI, 6, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream, row_base, stream_out);
    case 4: return launch_l4<EPI, 4, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream, row_base, stream_out);
    default: return launch_l4<EPI, 3, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream, row_base, stream_out);
  }
}

template <int EPI>
int launch_l4_pair_cfg(int cfg, const L4Prob& p0, const L4Prob& p1, int K, hipStream_t stream) {
  switch (cfg) {
    case 0: return launch_l4_pair<EPI, 8, 8>(p0, p1, K, stream);
    case 1: return launch_l4_pair<EPI, 6, 8>(p0, p1, K, stream);
    case 2: return launch_l4_pair<EPI, 8, 4>(p0, p1, K, stream);
    case 3: return launch_l4_pair<EPI, 6, 4>(p0, p1, K, stream);
    case 4: return launch_l4_pair<EPI, 4, 4>(p0, p1, K, stream);
    default: return launch_l4_pair<EPI, 3, 4>(p0, p1, K, stream);
  }
}

// Estimated time (us) of `tiles` tiles of configuration c on `cus` CUs, and of M x N on
// the 64 x 128 tiles of gemm_kernel while each has a CU to itself (two sharing one run at
// half the rate each, where the configurations above are the faster ones).
float l4_cost(int c, int64_t tiles, int K, int cus) {
  const int64_t ncu = std::max(8, cus / 8 * 8), rounds = (tiles + ncu - 1) / ncu;
  return kL4[c].start + (float)rounds * (kL4[c].tile + kL4[c].stage * (float)(K / 64));
}
float small_cost(int M, int N, int K, int cus) {
  const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 127) / 128);
  return tiles <= cus ? 2.8f + 0.411f * (float)(K / 64) : 1e30f;
}
int64_t l4_tiles(int c, int M, int N) {
  return (int64_t)((M + kL4[c].gbm - 1) / kL4[c].gbm) * ((N + kL4[c].gbn - 1) / kL4[c].gbn);
}

// The kernels and tiles a product can run on (as numbered by ditk_gemm_plan).
enum GemmTile : int {
  GT_SMALL = 0,                    // gemm_kernel, 64 x 128
  GT_LARGE = 1,                    // gemm_kernel, 256 x 256
  GT_L4 = 2,                       // + a configuration of kL4: gemm_kernel_l4
  GT_SKINNY = GT_L4 + kL4Cfgs,     // gemm_skinny
};

// How one product runs: the first `rows` rows on `tile`, the others in a second launch
// on `rest`.  A second launch pays where the tiles of one configuration leave the last
// round of CUs mostly idle: full rounds of it, then smaller tiles for the remaining rows
// (14336 x 1536 x 8960: 336 tiles of 256 x 256 are 1.3 rounds, 367 -> 314 us;
// 54560 x 3072 x 14336, whose last tile row has 32 rows, 3.89 -> 3.56 ms).  A short
// last tile row is split off for any predicted gain, more rows at long K from
// kSplitGain on: over several rounds the workgroups drift apart and the last round
// costs less than a whole one (7000 x 4608 x 1536, 0.3% predicted: 78 -> 82 us; 28080
// x 1536 x 1536, 8% predicted: 126 -> 133 us).
// Every row is computed the same way whichever tile holds it, so the choice changes
// no result.  Without splits the choice loses 0.4% on average against the fastest of
// all configurations at each measured size.
struct GemmPlan {
  int tile, rows, rest;
  float us;
};
GemmPlan gemm_plan_one(int M, int N, int K, int cus) {
  GemmPlan best{GT_SMALL, M, GT_SMALL, small_cost(M, N, K, cus)};
  for (int c = 0; c < kL4Cfgs; ++c) {
    const float us = l4_cost(c, l4_tiles(c, M, N), K, cus);
    if (us < best.us) best = GemmPlan{GT_L4 + c, M, GT_SMALL, us};
  }
  return best;
}
constexpr float kSplitGain = 0.92f;
GemmPlan gemm_plan_l4(int M, int N, int K, int cus) {
  GemmPlan best = gemm_plan_one(M, N, K, cus);
  const float one = best.us;
  const int64_t ncu = std::max(8, cus / 8 * 8);
  for (int c = 0; c < kL4Cfgs; ++c) {
    const int64_t tn = (N + kL4[c].gbn - 1) / kL4[c].gbn, tm = (M + kL4[c].gbm - 1) / kL4[c].gbm;
    const int64_t main_m = tm * tn / ncu * ncu / tn;  // tile rows of the full rounds
    if (main_m == 0 || main_m >= tm || tm * tn % ncu == 0) continue;
    const int rows = (int)main_m * kL4[c].gbm;
    const GemmPlan rest = gemm_plan_one(M - rows, N, K, cus);
    const float us = l4_cost(c, main_m * tn, K, cus) + rest.us;
    if (us < best.us && (main_m == tm - 1 || (K >= 4096 && us < kSplitGain * one)))
      best = GemmPlan{GT_L4 + c, rows, rest.tile, us};
  }
  return best;
}

// narrow: every output and residual row stride below 2^22 (the one-wave-per-SIMD kernel's
// epilogue addresses a wave tile's rows by 32-bit offsets).  fp32 outputs and K % 64 != 0:
// gemm_kernel, on small tiles when the large ones would number fewer than
// kSmallBelow (666 rows 1.3-3x faster at 54-72 large tiles, 8192 x 1536 1.25-1.5x
// slower at 192).
constexpr int64_t kSmallBelow = 128;
GemmPlan gemm_plan(int M, int N, int K, int epilogue, bool narrow, int cus) {
  if (M <= kSkinnyM && N >= kSkinnyN)  // its weights at 5.25 TB/s
    return GemmPlan{GT_SKINNY, M, GT_SMALL, 2.f + (float)N * (float)K * (2.f / 5.25e6f)};
  if (epilogue == EPI_F32 || K % 64 != 0 || !narrow) {
    const int64_t large_tiles = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
    return GemmPlan{large_tiles < kSmallBelow ? GT_SMALL : GT_LARGE, M, GT_SMALL, 0.f};
  }
  GemmPlan p = gemm_plan_l4(M, N, K, cus);
  // the gated residual at short K: the 8-wave kernel's two waves per SIMD hide
  // more of the residual and gate reads (1536 x 1536, with the AdaLN that reads the
  // output next: 28080 rows 175 -> 166 us, 20000 115 -> 110, 9300 62 -> 58; at N = K = 3072
  // it is 0-3% slower)
  if (epilogue == EPI_GATE_RES && K < 3072)
    for (int* t : {&p.tile, &p.rest})
      if (*t == GT_L4) *t = GT_LARGE;
  return p;
}

template <int EPI, int BK>
int launch(const GemmPlan& plan, const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C,
           int64_t ldc, int M, int N, int K, const void* R, int64_t ldr, const float* gate,
           int64_t gate_stride, const int32_t* cu, int nseg, hipStream_t stream) {
  const bool stream_out = stream_output(M, N);
  // rows [m0, m0 + m) on tile
  auto part = [&](int tile, int m0, int m) {
    constexpr int esize = EPI == EPI_F32 ? 4 : 2;
    const void* Am = static_cast<const bf16_t*>(A) + (int64_t)m0 * lda;
    void* Cm = static_cast<char*>(C) + (int64_t)m0 * ldc * esize;
    const void* Rm = R ? static_cast<const bf16_t*>(R) + (int64_t)m0 * ldr : nullptr;
    if (tile == GT_SKINNY)
      return launch_skinny<EPI>(Am, lda, W, ldw, bias, Cm, ldc, m, N, K, Rm, ldr, gate, gate_stride, cu, nseg, stream);
    if (tile == GT_SMALL)
      return launch_tile<EPI, BK, TILE_SMALL>(Am, lda, W, ldw, bias, Cm, ldc, m, N, K, Rm, ldr, gate, gate_stride,
                                              cu, nseg, stream, m0, stream_out);
    if constexpr (EPI != EPI_F32 && BK == 64)
      if (tile >= GT_L4)
        return launch_l4_cfg<EPI>(tile - GT_L4, Am, lda, W, ldw, bias, Cm, ldc, m, N, K, Rm, ldr, gate, gate_stride, cu,
                                  nseg, stream, m0, stream_out);
    return launch_tile<EPI, BK, TILE_LARGE>(Am, lda, W, ldw, bias, Cm, ldc, m, N, K, Rm, ldr, gate, gate_stride,
                                            cu, nseg, stream, m0, stream_out);
  };
  const int rc = part(plan.tile, 0, plan.rows);
  return rc != 0 || plan.rows == M ? rc : part(plan.rest, plan.rows, M - plan.rows);
}

template <int EPI>
int launch_k(const GemmPlan& plan, const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C,
             int64_t ldc, int M, int N, int K, const void* R, int64_t ldr, const float* gate,
             int64_t gate_stride, const int32_t* cu, int nseg, hipStream_t stream) {
  // 64-k stages when K allows (half the barriers); the MFMA k order is the
  // same for both, so results do not depend on the choice
  return K % 64 == 0 ? launch<EPI, 64>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream)
                     : launch<EPI, 32>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu, nseg, stream);
}

}  // namespace

namespace {
int gemm_validate(const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C, int64_t ldc,
                  int M, int N, int K, int epilogue, const void* R, int64_t ldr, const float* gate,
                  int64_t gate_stride, const int32_t* cu_seqlens, int nseg) {
  // A, C and R may be NULL when there are no rows (an empty tensor's pointer)
  DITK_REQUIRE(W && (M == 0 || (A && C)), "ditk_gemm: null operand");
  DITK_REQUIRE(M >= 0 && N > 0 && K > 0, "ditk_gemm: bad shape M=%d N=%d K=%d", M, N, K);
  DITK_REQUIRE(K % 32 == 0, "ditk_gemm: K=%d must be a multiple of 32", K);
  DITK_REQUIRE(N % 8 == 0, "ditk_gemm: N=%d must be a multiple of 8", N);
  DITK_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K,
               "ditk_gemm: lda/ldw must be multiples of 8 and >= K");
  DITK_REQUIRE((int64_t)256 * lda < (1ll << 31) && (int64_t)256 * ldw < (1ll << 31),
               "ditk_gemm: leading dimensions too large");
  DITK_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)C % 16) == 0 &&
                   ((uintptr_t)bias % 16) == 0,
               "ditk_gemm: A, W, C and bias must be 16-byte aligned");
  DITK_REQUIRE(ldc % 8 == 0 && ldc >= N, "ditk_gemm: ldc must be a multiple of 8 and >= N");
  DITK_REQUIRE(epilogue >= 0 && epilogue <= 5, "ditk_gemm: unknown epilogue %d", epilogue);
  DITK_REQUIRE(!(epilogue == EPI_GATE_RES || epilogue == EPI_RES) ||
               ((R || M == 0) && ldr % 8 == 0 && ldr >= N && ((uintptr_t)R % 16) == 0),
               "ditk_gemm: residual epilogue needs a 16-byte aligned R with ldr %% 8 == 0");
  DITK_REQUIRE(epilogue != EPI_GATE_RES || (gate_stride % 4 == 0 && ((uintptr_t)gate % 16) == 0),
               "ditk_gemm: gate rows must be 16-byte aligned");
  DITK_REQUIRE(epilogue != EPI_GATE_RES || (gate && cu_seqlens && nseg > 0),
               "ditk_gemm: gated epilogue needs gate and cu_seqlens");
  return 0;
}

bool narrow(int64_t ldc, int64_t ldr) { return ldc < (1 << 22) && ldr < (1 << 22); }

// The configuration of kL4 that takes two products in one launch, where its rounds over
// both tile lists cost less than the two launches p0 and p1; -1 where none does.
int pair_plan(const GemmPlan& p0, const GemmPlan& p1, int M0, int N0, int M1, int N1, int K, int epilogue, bool narrow,
              int cus) {
  if (M0 <= 0 || M1 <= 0 || epilogue == EPI_F32 || K % 64 != 0 || !narrow) return -1;
  int cfg = -1;
  float us = p0.us + p1.us;
  for (int c = 0; c < kL4Cfgs; ++c) {
    const float t = l4_cost(c, l4_tiles(c, M0, N0) + l4_tiles(c, M1, N1), K, cus);
    if (t < us) {
      us = t;
      cfg = c;
    }
  }
  return cfg;
}

int gemm_run(const GemmPlan& plan, const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias, void* C,
             int64_t ldc, int M, int N, int K, int epilogue, const void* R, int64_t ldr, const float* gate,
             int64_t gate_stride, const int32_t* cu_seqlens, int nseg, hipStream_t stream) {
  if (M == 0) return 0;
  switch (epilogue) {
    case EPI_BIAS: return launch_k<EPI_BIAS>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu_seqlens, nseg, stream);
    case EPI_GELU: return launch_k<EPI_GELU>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu_seqlens, nseg, stream);
    case EPI_GATE_RES: return launch_k<EPI_GATE_RES>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu_seqlens, nseg, stream);
    case EPI_RES: return launch_k<EPI_RES>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu_seqlens, nseg, stream);
    case EPI_F32: return launch_k<EPI_F32>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu_seqlens, nseg, stream);
    default: return launch_k<EPI_SILU>(plan, A, lda, W, ldw, bias, C, ldc, M, N, K, R, ldr, gate, gate_stride, cu_seqlens, nseg, stream);
  }
}
}  // namespace

DITK_EXPORT int ditk_gemm(const void* A, int64_t lda, const void* W, int64_t ldw, const float* bias,
                          void* C, int64_t ldc, int M, int N, int K, int epilogue, const void* R,
                          int64_t ldr, const float* gate, int64_t gate_stride,
                          const int32_t* cu_seqlens, int nseg, hipStream_t stream) {
  if (int rc = gemm_validate(A, lda, W, ldw, bias, C, ldc, M, N, K, epilogue, R, ldr, gate, gate_stride,
                             cu_seqlens, nseg))
    return rc;
  return gemm_run(gemm_plan(M, N, K, epilogue, narrow(ldc, ldr), ditk_cu_count()), A, lda, W, ldw, bias, C, ldc, M, N,
                  K, epilogue, R, ldr, gate, gate_stride, cu_seqlens, nseg, stream);
}

DITK_EXPORT int ditk_gemm_pair_n(const void* A0, int64_t lda0, const void* W0, int64_t ldw0, const float* bias0,
                               void* C0, int64_t ldc0, int M0, const void* R0, int64_t ldr0, const float* gate0,
                               int64_t gate_stride0, const int32_t* cu_seqlens0, int nseg0, const void* A1,
                               int64_t lda1, const void* W1, int64_t ldw1, const float* bias1, void* C1,
                               int64_t ldc1, int M1, const void* R1, int64_t ldr1, const float* gate1,
                               int64_t gate_stride1, const int32_t* cu_seqlens1, int nseg1, int N0, int N1,
                                 int K, int epilogue, hipStream_t stream) {
  if (int rc = gemm_validate(A0, lda0, W0, ldw0, bias0, C0, ldc0, M0, N0, K, epilogue, R0, ldr0, gate0,
                             gate_stride0, cu_seqlens0, nseg0))
    return rc;
  if (int rc = gemm_validate(A1, lda1, W1, ldw1, bias1, C1, ldc1, M1, N1, K, epilogue, R1, ldr1, gate1,
                             gate_stride1, cu_seqlens1, nseg1))
    return rc;
  const int cus = ditk_cu_count();
  const bool narrow0 = narrow(ldc0, ldr0), narrow1 = narrow(ldc1, ldr1);
  const GemmPlan g0 = gemm_plan(M0, N0, K, epilogue, narrow0, cus), g1 = gemm_plan(M1, N1, K, epilogue, narrow1, cus);
  const int cfg = pair_plan(g0, g1, M0, N0, M1, N1, K, epilogue, narrow0 && narrow1, cus);
  if (cfg >= 0) {
    const L4Prob p0{(const bf16_t*)A0, lda0, (const bf16_t*)W0, ldw0, bias0, C0, ldc0, (const bf16_t*)R0, ldr0,
                    gate0, gate_stride0, cu_seqlens0, nseg0, M0, N0, 0, 0, 0};
    const L4Prob p1{(const bf16_t*)A1, lda1, (const bf16_t*)W1, ldw1, bias1, C1, ldc1, (const bf16_t*)R1, ldr1,
                    gate1, gate_stride1, cu_seqlens1, nseg1, M1, N1, 0, 0, 0};
    switch (epilogue) {
      case EPI_BIAS: return launch_l4_pair_cfg<EPI_BIAS>(cfg, p0, p1, K, stream);
      case EPI_GELU: return launch_l4_pair_cfg<EPI_GELU>(cfg, p0, p1, K, stream);
      case EPI_GATE_RES: return launch_l4_pair_cfg<EPI_GATE_RES>(cfg, p0, p1, K, stream);
      case EPI_RES: return launch_l4_pair_cfg<EPI_RES>(cfg, p0, p1, K, stream);
      default: return launch_l4_pair_cfg<EPI_SILU>(cfg, p0, p1, K, stream);
    }
  }
  if (int rc = gemm_run(g0, A0, lda0, W0, ldw0, bias0, C0, ldc0, M0, N0, K, epilogue, R0, ldr0, gate0, gate_stride0,
                        cu_seqlens0, nseg0, stream))
    return rc;
  return gemm_run(g1, A1, lda1, W1, ldw1, bias1, C1, ldc1, M1, N1, K, epilogue, R1, ldr1, gate1, gate_stride1,
                  cu_seqlens1, nseg1, stream);
}

DITK_EXPORT int ditk_gemm_plan(int M, int N, int K, int epilogue, int* plan) {
  DITK_REQUIRE(plan && M > 0 && N > 0 && K > 0 && K % 32 == 0 && epilogue >= 0 && epilogue <= 5,
               "ditk_gemm_plan: bad arguments");
  const GemmPlan p = gemm_plan(M, N, K, epilogue, true, ditk_cu_count());
  plan[0] = p.tile;
  plan[1] = p.rows;
  plan[2] = p.rest;
  return 0;
}

DITK_EXPORT int ditk_gemm_pair_plan(int M0, int N0, int M1, int N1, int K, int epilogue) {
  if (M0 <= 0 || M1 <= 0 || N0 <= 0 || N1 <= 0 || K <= 0 || K % 32 != 0) return -1;
  const int cus = ditk_cu_count();
  const int cfg = pair_plan(gemm_plan(M0, N0, K, epilogue, true, cus), gemm_plan(M1, N1, K, epilogue, true, cus), M0, N0,
                            M1, N1, K, epilogue, true, cus);
  return cfg < 0 ? -1 : GT_L4 + cfg;
}

DITK_EXPORT int ditk_gemm_pair(const void* A0, int64_t lda0, const void* W0, int64_t ldw0, const float* bias0,
                               void* C0, int64_t ldc0, int M0, const void* R0, int64_t ldr0, const float* gate0,
                               int64_t gate_stride0, const int32_t* cu_seqlens0, int nseg0, const void* A1,
                               int64_t lda1, const void* W1, int64_t ldw1, const float* bias1, void* C1,
                               int64_t ldc1, int M1, const void* R1, int64_t ldr1, const float* gate1,
                               int64_t gate_stride1, const int32_t* cu_seqlens1, int nseg1, int N, int K,
                               int epilogue, hipStream_t stream) {
  return ditk_gemm_pair_n(A0, lda0, W0, ldw0, bias0, C0, ldc0, M0, R0, ldr0, gate0, gate_stride0, cu_seqlens0, nseg0,
                          A1, lda1, W1, ldw1, bias1, C1, ldc1, M1, R1, ldr1, gate1, gate_stride1, cu_seqlens1, nseg1,
                          N, N, K, epilogue, stream);
}
