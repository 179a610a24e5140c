// gemm.hip — K2: INT4 x activation-plane GEMM on gfx950 MFMA.
//
// y[M][N] = planes(x)[M][K] . W^T past the decode GEMV's rows (decode batches
// of 3 or more lanes, prompt chunks), with the same tile layout and fused
// epilogues as the decode GEMV (K1). Two plane layouts (kernels.h):
//   * Q8: the per-group arithmetic is the reference's Q8 dot
//     (int4_matmul.zig:365-418), an exact integer dot per 32-element group
//     scaled by the weight and activation group scales and summed in f32. One
//     i8 MFMA with K = 32 covers one group of an output tile. The codes are
//     made signed (u - 7), so its result is the group dot T itself; the
//     accumulator starts at the bits of 1.5 * 2^23 and fma(that as f32, ws,
//     -12582912 * ws) = RN(T * ws) (int4_ops.h), then one fma applies the
//     activation scale into the running sum.
//   * split-16: f32 activations as an fp16 pair per element (x / 2^e = hi + lo
//     to the larger of 2^-23 of x and 2^-39 of the group's largest), codes as
//     exact halves, two fp16 MFMAs (one onto the
//     other) per group with f32 accumulation, then the same two scales. Against
//     three 7-bit digits on i8 MFMAs (three of them and five f32 / integer
//     operations per output and group): 1999 x 3584 x 18944 1302 -> 840 us,
//     error against 64-bit sums 5.9e-7 -> 4.7e-7.
//
// The tall tiles' largest known cost is the vector work of the per-group
// scaling (two f32 operations per output and group), not the matrix cores (see
// there). Two kernels:
//   * up to 32 rows, gemm_kernel: 4 waves over 16 or 32 rows, each wave its
//     own weight row blocks. Each lane loads its own 16-byte tile slot per row
//     block and quad (1 KB per wave, fully coalesced), two quads in flight;
//     the words are transposed across lanes into MFMA operands
//     (quad_transpose) and the lane-ordered fp16 scales gathered per column
//     (column_gather). The workgroup stages each quad's activation planes in
//     LDS, double buffered, one barrier per quad;
//   * prompt chunks, gemm_tile_kernel: 64 or 128 rows x 128 columns by 8
//     waves, both operands in LDS.
// Small grids split K over workgroups: each split writes its partial sums and
// a finishing kernel (or the last split to arrive) adds them in a fixed order
// and runs the epilogue (deterministic).
#include "epilogue.h"
#include "int4_ops.h"
#include "kernels.h"

#include <algorithm>

namespace gk {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef long v2l __attribute__((ext_vector_type(2)));

constexpr int kWaves = 4;            // waves per workgroup, side by side in N
constexpr int kU = 2;                // weight quads in flight per wave
constexpr int kFoldSplits = 4;       // K splits a folded tile adds at most

// Activation staging of the 16- and 32-row tiles: a quad's planes as 16-byte
// units, then the group scales [4][BM].
//   Q8:       [group][half][row][16 B], a half's stride padded by 64 bytes;
//   split-16: [group][hi, lo][unit][row][16 B], a unit's stride padded by 32.
// A wave's operand read takes 16 bytes of consecutive rows (no bank
// conflicts), and the pads keep the staging writes, whose lanes take the
// units of a row in turn, on distinct banks.
template <int D, int BM>
struct ActStage {
  static constexpr int SG = 4;
  static constexpr int kRowUnits = D == kPlanesQ8 ? 2 : 4;      // per plane row
  static constexpr int kPlanes = D == kPlanesQ8 ? 1 : 2;        // planes per group
  static constexpr int kUnitStride = BM * 16 + (D == kPlanesQ8 ? 64 : 32);
  static constexpr int kPlaneStride = kRowUnits * kUnitStride;
  static constexpr int kActBytes = SG * kPlanes * kPlaneStride;
  static constexpr int kBufBytes = kActBytes + SG * BM * 4;
  static constexpr int kUnitCount = SG * kPlanes * BM * kRowUnits;
  static constexpr int kUnits = (kUnitCount + 255) / 256;       // per thread
  static_assert(kUnits <= 4 && SG * BM <= 256, "ActRegs holds four units and a scale per thread");
};

// One thread's share of a stage as named members, read and written through
// at() with indices that are constants once the loops are unrolled (an array
// member of them was kept in scratch memory, whose stores waited for the
// loads as soon as they were issued).
struct ActRegs {
  uint4 v0, v1, v2, v3;
  float sc;
  __device__ __forceinline__ uint4 &at(int i) {
    switch (i) {
      case 0: return v0;
      case 1: return v1;
      case 2: return v2;
      default: return v3;
    }
  }
};

// Where a thread's units and scale of a stage lie: byte offsets from the
// stage's first group in the planes (rows m0 .. m0 + BM - 1, clamped to
// M - 1) and into the LDS buffer. Loads are base + 32-bit offset.
template <int D, int BM>
struct ActMap {
  using S = ActStage<D, BM>;
  uint32_t src[S::kUnits], dst[S::kUnits], msrc, mdst;
  __device__ __forceinline__ ActMap(int M, int m0) {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < S::kUnits; ++i) {
      // (16-row tiles have fewer units than threads: the extra threads
      // repeat the last unit, branch-free)
      const int u = min(t + 256 * i, S::kUnitCount - 1);
      const int sub = u % S::kRowUnits, row = u / S::kRowUnits % BM, pl = u / S::kRowUnits / BM;
      src[i] = ((uint32_t)pl * M + min(m0 + row, M - 1)) * (16 * S::kRowUnits) + 16 * sub;
      dst[i] = pl * S::kPlaneStride + sub * S::kUnitStride + row * 16;
    }
    const int ts = t % (S::SG * BM);  // threads past SG * BM repeat another's scale
    msrc = ((uint32_t)(ts / BM) * M + min(m0 + ts % BM, M - 1)) * sizeof(ActMeta);
    mdst = S::kActBytes + ts * 4;
  }
  // the stage that starts at group g
  __device__ __forceinline__ ActRegs load(const GemvArgs &p, int g) const {
    ActRegs r;
    const char *q = (const char *)p.act_q + (size_t)g * p.M * plane_group_bytes(D);
    const char *mp = (const char *)(p.act_meta + (size_t)g * p.M);
#pragma unroll
    for (int i = 0; i < S::kUnits; ++i) r.at(i) = *(const uint4 *)(q + src[i]);
    r.sc = *(const float *)(mp + msrc);
    return r;
  }
  __device__ __forceinline__ void store(unsigned char *buf, ActRegs &r) const {
#pragma unroll
    for (int i = 0; i < S::kUnits; ++i) *(uint4 *)(buf + dst[i]) = r.at(i);
    *(float *)(buf + mdst) = r.sc;
  }
};

// A value the compiler may not see through: keeps a converted fp16 scale in
// its own f32 register instead of folded into v_fma_mix_f32, which issues at
// half the rate of v_fma_f32 (4.7 against 2.8 cycles).
static __device__ __forceinline__ float opaque(float v) {
  asm("" : "+v"(v));
  return v;
}

// First quad of K split s of ks (a power of two, at most 16). By a shift: as
// 64-bit divisions the two bounds were 300 instructions in front of every
// load: 16 x 9728 x 896 10.1 -> 9.7 us, 5 x 4608 x 3584 10.7 -> 10.2.
static __device__ __forceinline__ int split_quad(uint32_t s, int KQ, int ks) {
  return (int)(s * (uint32_t)KQ >> __builtin_ctz(ks));
}

// A lane offset the compiler may not widen outside the loop: loads then take a
// scalar base and this one register (a 64-bit address pair per load otherwise).
static __device__ __forceinline__ uint32_t here(uint32_t v) {
  asm("" : "+v"(v));
  return v;
}

// kRB: 16-row weight blocks per wave (kRowBlocks<D>; the workgroup covers
// 4 kRB); BM: activation rows per workgroup (16 or 32). The K quads are split over
// blockIdx.y (ks_count splits); with part set each split writes its partial
// sums to part [ks_count][M][N] (no epilogue; a finishing kernel runs it),
// unless fold: then the splits of a tile meet at p.splitk_counters and the
// last to arrive runs the epilogue (the SwiGLU plane emission included).
// Lane (c, n) of a 16 x 16 output tile (row block i, row tile mt) holds rows
// 16 mt + 4 c + r of column n.
template <int D>
constexpr int kRowBlocks = D == kPlanesQ8 ? 1 : 2;
template <int D, int BM>
__global__ __launch_bounds__(256, kRowBlocks<D> == 2 ? 4 : 5) void gemm_kernel(
    GemvArgs p, int m_tiles, int ks_count, float *part, int fold) {
  constexpr int kRB = kRowBlocks<D>;
  using S = ActStage<D, BM>;
  constexpr int MT = BM / 16;         // 16-row activation tiles per wave
  constexpr int kNBW = kWaves * kRB;  // weight row blocks per workgroup
  constexpr int NO = 32 * kRB;        // SwiGLU outputs per workgroup and row
  constexpr int kStageBytes = BM * NO * 4, kParkBytes = MT * 4 * 256 * 4;
  constexpr int kLds = 2 * S::kBufBytes > kStageBytes ? 2 * S::kBufBytes : kStageBytes;
  __shared__ __align__(16) unsigned char lds[kLds > kParkBytes ? kLds : kParkBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform
  const int n_local = lane & 15, c = lane >> 4;
  const int NB = p.N >> 4, KQ = p.K >> 7;
  // XCD-aware block order: XCD x runs logical blocks [first_x, first_x + cnt_x)
  const int nblk = gridDim.x, b = blockIdx.x;
  const int xcd = b & 7, idx = b >> 3;
  const int logical = xcd * (nblk >> 3) + min(xcd, nblk & 7) + idx;
  const int n_tile = logical / m_tiles, m_tile = logical % m_tiles;
  const int m0 = m_tile * BM;
  const int nb0 = n_tile * kNBW + wave * kRB;  // this wave's first row block
  // this split's quads kq0 .. kq0 + nq - 1
  const int kq0 = split_quad(blockIdx.y, KQ, ks_count);
  const int nq = split_quad(blockIdx.y + 1, KQ, ks_count) - kq0;
  const auto row_of = [&](int mt, int r) {
    return m0 + 16 * mt + 4 * c + r;
  };
  const auto block_of = [&](int i) { return nb0 + i; };

  // weight slots of this wave's row blocks: one per-lane base pointer plus
  // uniform tile offsets (row blocks past NB are clamped into range, compute
  // on a copy and are never stored)
  const uint4 *cp = p.codes + lane;
  const uint16_t *spp = (const uint16_t *)p.scales + lane;
  size_t toff[kRB];
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb) toff[rb] = ((size_t)min(nb0 + rb, NB - 1) * KQ + kq0) * 64;
  uint4 wb[kU][kRB];
  uint32_t sb[kU][kRB];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int q = min(u, nq - 1);
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      wb[u][rb] = load_stream(cp + toff[rb] + (size_t)q * 64);
      sb[u][rb] = spp[toff[rb] + (size_t)q * 64];
    }
  }
  const ActMap<D, BM> map(p.M, m0);
  {
    ActRegs r = map.load(p, 4 * kq0);
    map.store(lds, r);
  }
  __syncthreads();

  float acc[kRB][MT][4];
#pragma unroll
  for (int i = 0; i < kRB; ++i)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][mt][r] = 0.0f;

  for (int q0 = 0; q0 < nq; q0 += kU) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int q = q0 + u;  // local quad index (absolute kq0 + q)
      if (q >= nq) break;
      // this quad's weights; the slot is refilled with quad q + kU
      uint4 wc[kRB];
      uint32_t sc[kRB];
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        wc[rb] = wb[u][rb];
        sc[rb] = sb[u][rb];
      }
      // (branch-free: past the end the last quad is loaded again and never
      // used, so the quad's work stays one block for the scheduler)
      const int qn = min(q + kU, nq - 1);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        wb[u][rb] = load_stream(cp + toff[rb] + (size_t)qn * 64);
        sb[u][rb] = spp[toff[rb] + (size_t)qn * 64];
      }
      // MFMA operand words of the quad's groups and the scales of this
      // lane's columns
      uint32_t wt[kRB][4];
      float ws[kRB][4];
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        const uint4 t4 = quad_transpose(wc[rb]);
        wt[rb][0] = t4.x;
        wt[rb][1] = t4.y;
        wt[rb][2] = t4.z;
        wt[rb][3] = t4.w;
      }
      {
        // two row blocks' u16 scales per register, all four groups' rows
        uint32_t g4[4];
        column_gather((sc[0] & 0xFFFFu) | (kRB > 1 ? sc[kRB - 1] << 16 : 0u), g4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ws[0][j] = opaque(h2f(g4[j] & 0xFFFFu));
          if (kRB > 1) ws[kRB - 1][j] = opaque(h2f(g4[j] >> 16));
        }
      }
      // this quad's buffer (q0 is even, so u: constant LDS offsets) and, into
      // the other one, the next quad's activations, loaded while this one
      // computes (the last quad stages a copy of itself)
      ActRegs nxt = map.load(p, 4 * (kq0 + min(q + 1, nq - 1)));
      const unsigned char *buf = lds + u * S::kBufBytes;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned char *gb = buf + j * S::kPlanes * S::kPlaneStride;
        const unsigned char *sb4 = buf + S::kActBytes + j * BM * 4;
        long bw[kRB];
        v8h bh[kRB];
#pragma unroll
        for (int i = 0; i < kRB; ++i) {
          if constexpr (D == kPlanesQ8) bw[i] = signed_codes(wt[i][j]);
          else bh[i] = half_codes(wt[i][j]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const float4 as4 = *(const float4 *)(sb4 + (16 * mt + 4 * c) * 4);
          const float as[4] = {as4.x, as4.y, as4.z, as4.w};
          if constexpr (D == kPlanesQ8) {
            const long av = *(const long *)(gb + (c >> 1) * S::kUnitStride +
                                            (16 * mt + n_local) * 16 + 8 * (c & 1));
            const v4i magic = {kMagic, kMagic, kMagic, kMagic};
#pragma unroll
            for (int i = 0; i < kRB; ++i) {
              const v4i dd = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bw[i], magic, 0, 0, 0);
              const float wcorr = -kMagicF * ws[i][j];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float t = fmaf(__int_as_float(dd[r]), ws[i][j], wcorr);
                acc[i][mt][r] = fmaf(t, as[r], acc[i][mt][r]);
              }
            }
          } else {
            const unsigned char *ab = gb + c * S::kUnitStride + (16 * mt + n_local) * 16;
            const v8h ahi = *(const v8h *)ab, alo = *(const v8h *)(ab + S::kPlaneStride);
            v4f dd[kRB];
#pragma unroll
            for (int i = 0; i < kRB; ++i)
              dd[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bh[i], v4f{0.f, 0.f, 0.f, 0.f}, 0,
                                                             0, 0);
#pragma unroll
            for (int i = 0; i < kRB; ++i)
              dd[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bh[i], dd[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < kRB; ++i)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                acc[i][mt][r] = fmaf(dd[i][r] * ws[i][j], as[r], acc[i][mt][r]);
          }
          // one activation tile's MFMAs at a time: their results are
          // consumed before the next tile's are issued (register budget)
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // publish the next quad's activations (the other buffer was last read
      // before the previous barrier)
      map.store(lds + (u ^ 1) * S::kBufBytes, nxt);
      __syncthreads();
    }
  }

  if (fold) {
    if (ks_count > 1) {
      // Publish this split's partial sums; the tile's last split to arrive
      // adds every split's in split order (the finishing kernel's order, so
      // the sums are the same) and runs the epilogue. The publication is the
      // cross-workgroup contract attn_o_kernel's merge documents:
      // agent-scope stores written through to the level every XCD reads,
      // waited for (s_waitcnt covers stores), then an agent-scope counter
      // increment; the last arriver reads with agent-scope loads.
      const size_t MN = (size_t)p.M * p.N;
      float *dst = part + (size_t)blockIdx.y * MN;
#pragma unroll
      for (int i = 0; i < kRB; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = row_of(mt, r), nb = block_of(i);
            if (m < p.M && nb < NB)
              __hip_atomic_store(dst + (size_t)m * p.N + nb * 16 + n_local, acc[i][mt][r],
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
      __builtin_amdgcn_s_waitcnt(0);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      __shared__ int tile_last;
      if (threadIdx.x == 0)
        tile_last = __hip_atomic_fetch_add(p.splitk_counters + blockIdx.x, 1u, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(ks_count - 1);
      __syncthreads();
      if (!tile_last) return;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      // one (row block, row tile) at a time: its up to kFoldSplits splits'
      // loads issued together, then added in split order
#pragma unroll
      for (int i = 0; i < kRB; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          float v[kFoldSplits][4];
#pragma unroll
          for (int sp = 0; sp < kFoldSplits; ++sp)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int m = row_of(mt, r), nb = block_of(i);
              const size_t idx = m < p.M && nb < NB ? (size_t)m * p.N + nb * 16 + n_local : 0;
              v[sp][r] = sp < ks_count ? __hip_atomic_load(part + sp * MN + idx, __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT)
                                       : 0.0f;
            }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float tot = v[0][r];
#pragma unroll
            for (int sp = 1; sp < kFoldSplits; ++sp)
              if (sp < ks_count) tot += v[sp][r];
            acc[i][mt][r] = tot;
          }
        }
      if (threadIdx.x == 0)
        __hip_atomic_store(p.splitk_counters + blockIdx.x, 0u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    if (p.epi == EPI_SWIGLU && p.out_q) {
      // The SwiGLU plane emission of splitk_swiglu_emit_kernel for this
      // tile: its 4 kRB row blocks hold 32 kRB SwiGLU outputs (kRB whole
      // quantisation groups) of each activation row; silu(g) * u into LDS
      // [BM][32 kRB], then a half-wave quantises each (row, group).
      float *stage = (float *)lds;
      __syncthreads();  // the staging buffers were last read before the loop's end
#pragma unroll
      for (int i = 0; i < kRB; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float tot = acc[i][mt][r];
            const float partner = row_xor8(tot);
            if (n_local < 8)
              stage[(row_of(mt, r) - m0) * NO + (block_of(i) - n_tile * kNBW) * 8 + n_local] =
                  silu_mul(tot, partner);
          }
      __syncthreads();
      const int No = p.N >> 1;
      const int half = threadIdx.x >> 5, hl = threadIdx.x & 31;
      for (int it = half; it < BM * kRB; it += 8) {
        const int row = it / kRB, gl = it % kRB, m = m0 + row;
        const int o = (n_tile * kNBW) * 8 + gl * 32 + hl;  // SwiGLU output index
        if (m >= p.M || o >= No) continue;  // whole half-waves: No is a multiple of 32
        const float v = stage[row * NO + gl * 32 + hl];
        if (p.y) p.y[(size_t)m * No + o] = v;
        quantize_group_d(p.out_D, v, hl, o >> 5, m, p.M, p.out_q, p.out_meta);
      }
      return;
    }
  } else if (part) {
    // split K (or a finishing pass that emits planes): this split's partial
    // sums, part[split][m][n]
    float *dst = part + (size_t)blockIdx.y * p.M * p.N;
#pragma unroll
    for (int i = 0; i < kRB; ++i)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = row_of(mt, r), nb = block_of(i);
          if (m < p.M && nb < NB) dst[(size_t)m * p.N + nb * 16 + n_local] = acc[i][mt][r];
        }
    return;
  }
  // The SwiGLU / RoPE partner row n ^ 8 lives in lane ^ 8. The epilogue runs
  // as a loop over each row block's values parked in this thread's own LDS
  // column (the staging buffers are free after the last barrier): unrolled
  // over the large inlined epilogue it would index the accumulators
  // dynamically and push them to scratch.
  const bool paired = p.epi == EPI_SWIGLU || p.epi == EPI_QKV;
  float *park = (float *)lds + threadIdx.x;
#pragma unroll
  for (int i = 0; i < kRB; ++i) {
    const int nb = block_of(i);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) park[(mt * 4 + r) * 256] = acc[i][mt][r];
#pragma unroll 1
    for (int k = 0; k < MT * 4; ++k) {
      const float tot = park[k * 256];
      const float partner = paired ? row_xor8(tot) : 0.0f;
      const int m = row_of(k >> 2, k & 3);
      if (m < p.M && nb < NB)
        store_output(p, p.epi, nb, n_local, m, tot, partner, epi_load(p, p.epi, nb, n_local, m));
    }
  }
}

// ---------------------------------------------------------------------------
// Prompt chunks (more than 32 rows): BM x 128 output tiles by 8 waves, both
// operands in LDS.
//
// Cost: per output and group two f32 operations (scale by ws, then by as into
// the running sum) against one MFMA worth 1/128 of its time;
// MFMAs and vector work add up on this chip (a 32x32x32 i8 MFMA alone 35
// cycles, 32 fmas alone 86, together 106), f32 operations issue at 2.4-2.9
// cycles when at least two waves of a SIMD are ready and all operands are
// plain vector registers (v_fma_mix_f32, conversions and scalar operands
// 4.4-4.9), a single wave at 5-8. At those rates the instructions of the 2048
// x 37888 x 3584 Q8 launch are 518 of its 745 us (counted: 4.1e8 VALU, 8.5e6
// MFMAs over 1024 SIMDs at 2.4 GHz); what the other 30% is (the clock under
// load, LDS reads, barriers) has not been measured. Hence:
//   * the workgroup unpacks each quad's codes once (one 32-code slot, or one
//     word, per thread) into LDS operands every wave reads, so unpacking
//     costs 1/BM of an output instead of 1/(rows of a wave);
//   * at most 128 registers: four waves a SIMD, two workgroups a CU;
//   * Q8 on 32 x 32 x 32 MFMAs (half the time of 16 x 16 ones, whose K of 32
//     leaves half the multipliers idle), split-16 on 16 x 16 x 32;
//   * results are scaled by ws in one run and added in another (a dependent
//     instruction right behind costs the double rate).
// Stage: Q8 a quad in two buffers, split-16 a group in three, one barrier a
// stage.
// ---------------------------------------------------------------------------
constexpr int kTileThreads = 512;
constexpr int kTileN = 128;  // columns: 8 row blocks

template <int D, int BM>
struct TileStage {
  static constexpr bool Q8 = D == kPlanesQ8;
  static constexpr int SG = Q8 ? 4 : 1;                   // groups per stage
  static constexpr int kRowUnits = Q8 ? 2 : 4;            // 16-byte units per plane row
  static constexpr int kPlanes = Q8 ? 1 : 2;              // planes per group
  static constexpr int kPad = Q8 ? 64 : 32;               // staging writes of 8 lanes: distinct banks
  static constexpr int kBufs = Q8 ? 2 : 3;
  static constexpr int kAUnit = BM * 16 + kPad, kAPlane = kRowUnits * kAUnit;
  static constexpr int kBUnit = kTileN * 16 + kPad, kBPlane = kRowUnits * kBUnit;
  static constexpr int kB = SG * kPlanes * kAPlane;       // weight operands
  static constexpr int kAs = kB + SG * kBPlane;           // activation scales [SG][BM]
  static constexpr int kWs = kAs + SG * BM * 4;           // weight scales [SG][128]
  static constexpr int kBufBytes = kWs + SG * kTileN * 4;
  static constexpr int kUnits = SG * kPlanes * BM * kRowUnits / kTileThreads;  // per thread
  static constexpr int kScales = SG * BM;                 // threads past it repeat others'
};

template <int D, int BM>
__global__ __launch_bounds__(kTileThreads, 4) void gemm_tile_kernel(GemvArgs p, int m_tiles,
                                                                    int n_tiles, int ks_count,
                                                                    float *part, int fold) {
  using S = TileStage<D, BM>;
  constexpr bool Q8 = D == kPlanesQ8;
  constexpr int WM = BM / 32, WN = 8 / WM;      // waves in M (32 rows each) and N
  constexpr int NC = kTileN / WN;               // columns per wave
  constexpr int TS = Q8 ? 32 : 16;              // output tile size
  constexpr int NI = NC / TS, MT = 32 / TS, NR = TS * TS / 64;
  constexpr int kStageBytes = BM * (kTileN / 2) * 4, kParkBytes = 16 * kTileThreads * 4;
  constexpr int kLds0 = S::kBufs * S::kBufBytes > kStageBytes ? S::kBufs * S::kBufBytes : kStageBytes;
  __shared__ __align__(16) unsigned char lds[kLds0 > kParkBytes ? kLds0 : kParkBytes];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n_local = lane & 15, c = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;
  const int KQ = p.K >> 7, NB = p.N >> 4;
  // Block order: XCD x (block b runs on XCD b % 8) takes a contiguous run of
  // logical blocks, row tiles fastest in bands of kBand, so the workgroups that
  // run together on an XCD (about 64) read each operand's bytes about equally
  // often past its L2 (a Q8 row is 1.125 bytes a column, a split-16 one 4.25,
  // a weight 0.56).
  const int nblk = gridDim.x, b = blockIdx.x;
  const int xcd = b & 7;
  const int logical = xcd * (nblk >> 3) + min(xcd, nblk & 7) + (b >> 3);
  constexpr int kBand = Q8 ? 8 : 4;
  const int band = logical / (kBand * n_tiles), in_band = logical - band * kBand * n_tiles;
  const int band_rows = min(kBand, m_tiles - kBand * band);
  const int n_tile = in_band / band_rows, m_tile = kBand * band + in_band % band_rows;
  const int m0 = m_tile * BM, nb_wg = n_tile * 8;
  // (not split_quad: with the shifts in front of it the loop's code lies
  // differently, and 1999 x 3584 x 18944 takes 848 us instead of 845)
  const int kq0 = (int)(((long)blockIdx.y * KQ) / ks_count);
  const int nq = (int)(((long)(blockIdx.y + 1) * KQ) / ks_count) - kq0;
  const auto row_of = [&](int mt, int r) {
    return m0 + 32 * wm + (Q8 ? 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3) : 16 * mt + 4 * c + r);
  };
  const auto block_of = [&](int i) {
    return nb_wg + wn * (NC / 16) + (Q8 ? 2 * i + (c & 1) : i);
  };

  // staging: this thread's activation units (unit i lies kPlaneStep planes
  // after unit 0, or at the same place of a taller tile's next rows) and scale
  constexpr int kSpan = kTileThreads / S::kRowUnits;  // rows a pass covers
  static_assert(kSpan % BM == 0, "whole planes per pass");
  constexpr int kPlaneStep = kSpan / BM;
  const int sub = t % S::kRowUnits, arow = t / S::kRowUnits % BM, apl = t / S::kRowUnits / BM;
  const uint32_t asrc =
      ((uint32_t)apl * p.M + min(m0 + arow, p.M - 1)) * (16 * S::kRowUnits) + 16 * sub;
  const uint32_t adst = apl * S::kAPlane + sub * S::kAUnit + arow * 16;
  const uint32_t astep = (uint32_t)kPlaneStep * p.M * (16 * S::kRowUnits);  // uniform
  const int ts = t % S::kScales;
  const uint32_t ssrc = ((uint32_t)(ts / BM) * p.M + min(m0 + ts % BM, p.M - 1)) * sizeof(ActMeta);
  // ... and weight slot: wave w stages row block nb_wg + w (clamped into
  // range: computed on a copy, never stored). Q8: lane 16 j + n unpacks
  // group j of row n; split-16: lane 16 w + n word w of row n, for each group
  // of the quad in turn.
  const size_t tile0 = ((size_t)min(nb_wg + wave, NB - 1) * KQ + kq0) * 64;
  const char *wbase = (const char *)(p.codes + tile0);
  const char *sbase = (const char *)((const uint16_t *)p.scales + tile0);
  const uint32_t woff = Q8 ? lane * 16 : n_local * 16 + c * 4, scoff = 2 * (Q8 ? lane : n_local);
  // (named native vectors: HIP's uint4 class or an array of them was kept in
  // scratch memory, whose stores waited for the loads)
  static_assert(S::kUnits <= 2, "two units per thread");
  v4u a0, a1, b0, b1;  // two stages' units
  float asc, bsc;
  v4u wreg;                 // Q8: this thread's slot
  uint32_t aw, bw, aws, bws;  // split-16: a stage's code word; either: weight scale
  const auto load_acts = [&](v4u &v0, v4u &v1, float &sc, int g) {
    const char *q = (const char *)p.act_q + (size_t)g * p.M * plane_group_bytes(D);
    const uint32_t ao = here(asrc);
    v0 = *(const v4u *)(q + ao);
    if constexpr (S::kUnits > 1) v1 = *(const v4u *)(q + astep + ao);
    sc = *(const float *)((const char *)(p.act_meta + (size_t)g * p.M) + here(ssrc));
  };
  const auto load_slot = [&](int q) {
    wreg = *(const v4u *)(wbase + (size_t)q * 1024 + here(woff));
    aws = *(const uint16_t *)(sbase + (size_t)q * 128 + here(scoff));
  };
  const auto load_word = [&](uint32_t &w, uint32_t &sc, int g) {
    w = *(const uint32_t *)(wbase + (size_t)g * 256 + here(woff));
    sc = *(const uint16_t *)(sbase + (size_t)g * 32 + here(scoff));
  };
  const auto store_stage = [&](unsigned char *buf, v4u v0, v4u v1, float as, v4u w, uint32_t word,
                               uint32_t sc) {
    *(v4u *)(buf + adst) = v0;
    if constexpr (S::kUnits > 1) *(v4u *)(buf + kPlaneStep * S::kAPlane + adst) = v1;
    *(float *)(buf + S::kAs + ts * 4) = as;
    const int col = 16 * wave + n_local;
    if constexpr (Q8) {
      const v2l lo = {signed_codes(w.x), signed_codes(w.y)};
      const v2l hi = {signed_codes(w.z), signed_codes(w.w)};
      unsigned char *d = buf + S::kB + c * S::kBPlane + col * 16;
      *(v2l *)d = lo;
      *(v2l *)(d + S::kBUnit) = hi;
      *(float *)(buf + S::kWs + (c * kTileN + col) * 4) = h2f(sc);
    } else {
      *(v8h *)(buf + S::kB + c * S::kBUnit + col * 16) = half_codes(word);
      *(float *)(buf + S::kWs + col * 4) = h2f(sc);
    }
  };

  float acc[NI][MT][NR];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < NR; ++r) acc[i][mt][r] = 0.0f;

  // Q8: one group into the running sums. Its operands (av, bv, ws) were read
  // by the group before it; the next group's (of `nbuf`, if any) are requested
  // when this group's last MFMA has been issued, two runs of f32 work before
  // they are needed.
  const int h32 = lane >> 5, l32 = lane & 31;
  v4i av, bv[NI];
  float wsv[NI];
  const auto operand_b = [&](const unsigned char *buf, int gl, int i) {
    bv[i] = *(const v4i *)(buf + S::kB + gl * S::kBPlane + h32 * S::kBUnit +
                           (wn * NC + 32 * i + l32) * 16);
    wsv[i] = *(const float *)(buf + S::kWs + (gl * kTileN + wn * NC + 32 * i + l32) * 4);
  };
  const auto operands = [&](const unsigned char *buf, int gl) {
    av = *(const v4i *)(buf + gl * S::kAPlane + h32 * S::kAUnit + (32 * wm + l32) * 16);
    operand_b(buf, gl, 0);
  };
  const auto group8 = [&](const unsigned char *buf, int gl, bool more) {
    float4 as[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      as[k] = *(const float4 *)(buf + S::kAs + (gl * BM + 32 * wm + 8 * k + 4 * h32) * 4);
#pragma unroll
    for (int i = 1; i < NI; ++i) operand_b(buf, gl, i);
    v16i magic;
#pragma unroll
    for (int r = 0; r < 16; ++r) magic[r] = kMagic;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const v16i dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv[i], magic, 0, 0, 0);
      const float ws = wsv[i], wcorr = -kMagicF * ws;
      __builtin_amdgcn_sched_barrier(0);
      if (i == NI - 1 && more) operands(buf, gl + 1);
      float tt[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) tt[r] = fmaf(__int_as_float(dd[r]), ws, wcorr);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float a4[4] = {as[k].x, as[k].y, as[k].z, as[k].w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[i][0][4 * k + r] = fmaf(tt[4 * k + r], a4[r], acc[i][0][4 * k + r]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // split-16: one staged group into the running sums. Its weight operands and
  // its first row tile's were read by the group before it, whose last MFMAs
  // had been issued (three buffers: the next group's is complete a barrier
  // earlier), so LDS trips pass under the f32 runs, the staging writes and
  // the barrier.
  v8h hb[NI], ahi, alo;
  const auto rows16 = [&](const unsigned char *buf, int mt) {
    const unsigned char *ar = buf + c * S::kAUnit + (32 * wm + 16 * mt + n_local) * 16;
    ahi = *(const v8h *)ar;
    alo = *(const v8h *)(ar + S::kAPlane);
  };
  const auto operands16 = [&](const unsigned char *buf) {
    rows16(buf, 0);
#pragma unroll
    for (int i = 0; i < NI; ++i)
      hb[i] = *(const v8h *)(buf + S::kB + c * S::kBUnit + (wn * NC + 16 * i + n_local) * 16);
  };
  const auto group16 = [&](const unsigned char *buf, const unsigned char *next) {
    float ws[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
      ws[i] = *(const float *)(buf + S::kWs + (wn * NC + 16 * i + n_local) * 4);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const float4 as = *(const float4 *)(buf + S::kAs + (32 * wm + 16 * mt + 4 * c) * 4);
      const float a4[4] = {as.x, as.y, as.z, as.w};
      v4f dd[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i)
        dd[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, hb[i], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < NI; ++i)
        dd[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, hb[i], dd[i], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (mt + 1 < MT) rows16(buf, mt + 1);
      else operands16(next);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) dd[i][r] *= ws[i];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][mt][r] = fmaf(dd[i][r], a4[r], acc[i][mt][r]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  load_acts(a0, a1, asc, 4 * kq0);
  if constexpr (Q8) {
    load_slot(0);
    store_stage(lds, a0, a1, asc, wreg, 0, aws);
  } else {
    load_word(aw, aws, 0);
    load_acts(b0, b1, bsc, 4 * kq0 + 1);
    load_word(bw, bws, 1);
    store_stage(lds, a0, a1, asc, v4u{}, aw, aws);
    store_stage(lds + S::kBufBytes, b0, b1, bsc, v4u{}, bw, bws);
    load_acts(a0, a1, asc, 4 * kq0 + 2);
    load_word(aw, aws, 2);
  }
  __syncthreads();
  if constexpr (Q8) {
    for (int q = 0; q < nq; ++q) {
      // (past the end the last quad is staged again, into the idle buffer)
      const int qn = min(q + 1, nq - 1);
      load_acts(a0, a1, asc, 4 * (kq0 + qn));
      load_slot(qn);
      const unsigned char *buf = lds + (q & 1) * S::kBufBytes;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (g == 0) operands(buf, 0);
        group8(buf, g, g < 3);
      }
      store_stage(lds + ((q & 1) ^ 1) * S::kBufBytes, a0, a1, asc, wreg, 0, aws);
      __syncthreads();
    }
  } else {
    // a group's stage is shorter than a trip past the L2: requested three
    // stages ahead, stored two ahead
    int cur = 0, nxt = S::kBufBytes, far = 2 * S::kBufBytes;
    operands16(lds);
    const int ng = 4 * nq;
    for (int g0 = 0; g0 < ng; g0 += 2) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int ag = min(g0 + e + 3, ng - 1);  // (past the end the last group again, never used)
        if (e) {
          load_acts(a0, a1, asc, 4 * kq0 + ag);
          load_word(aw, aws, ag);
        } else {
          load_acts(b0, b1, bsc, 4 * kq0 + ag);
          load_word(bw, bws, ag);
        }
        group16(lds + cur, lds + nxt);
        if (e) store_stage(lds + far, b0, b1, bsc, v4u{}, bw, bws);
        else store_stage(lds + far, a0, a1, asc, v4u{}, aw, aws);
        const int was = cur;
        cur = nxt;
        nxt = far;
        far = was;
        __syncthreads();
      }
    }
  }

  if (part) {
    // split K (or a finishing pass that emits planes): this split's partial
    // sums, part[split][m][n]
    float *dst = part + (size_t)blockIdx.y * p.M * p.N;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const int m = row_of(mt, r), nb = block_of(i);
          if (m < p.M && nb < NB) dst[(size_t)m * p.N + nb * 16 + n_local] = acc[i][mt][r];
        }
    return;
  }
  if (fold) {
    // SwiGLU plane emission (splitk_swiglu_emit_kernel's) for this tile's
    // 64 outputs (two quantisation groups) of each row: silu(g) * u into
    // LDS [BM][64], then a half-wave quantises each (row, group).
    float *stage = (float *)lds;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const float tot = acc[i][mt][r];
          const float partner = row_xor8(tot);
          if (n_local < 8)
            stage[(row_of(mt, r) - m0) * 64 + (block_of(i) - nb_wg) * 8 + n_local] =
                silu_mul(tot, partner);
        }
    __syncthreads();
    const int No = p.N >> 1, half = t >> 5, hl = t & 31;
    for (int it = half; it < BM * 2; it += kTileThreads / 32) {
      const int row = it >> 1, gl = it & 1, m = m0 + row;
      const int o = nb_wg * 8 + gl * 32 + hl;  // SwiGLU output index
      if (m >= p.M || o >= No) continue;  // whole half-waves: No is a multiple of 32
      const float v = stage[row * 64 + gl * 32 + hl];
      if (p.y) p.y[(size_t)m * No + o] = v;
      quantize_group_d(p.out_D, v, hl, o >> 5, m, p.M, p.out_q, p.out_meta);
    }
    return;
  }
  if (p.epi == EPI_PLAIN) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int nb = block_of(i);
      if (nb >= NB) continue;
      const int n = nb * 16 + n_local;
      const float bias = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const int m = row_of(mt, r);
          if (m < p.M) p.y[(size_t)m * p.N + n] = p.bias ? bias + acc[i][mt][r] : acc[i][mt][r];
        }
    }
    return;
  }
  // The other epilogues run as a loop over 16 values at a time parked in this
  // thread's own LDS column: unrolled over the large inlined epilogue they
  // would index the accumulators dynamically and push them to scratch. The
  // SwiGLU / RoPE partner row n ^ 8 lives in lane ^ 8.
  const bool paired = p.epi == EPI_SWIGLU || p.epi == EPI_QKV;
  float *park = (float *)lds + t;
  constexpr int PT = Q8 ? 1 : 2;  // output tiles in N parked at a time
#pragma unroll
  for (int i0 = 0; i0 < NI; i0 += PT) {
#pragma unroll
    for (int i = 0; i < PT; ++i)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < NR; ++r)
          park[((i * MT + mt) * NR + r) * kTileThreads] = acc[i0 + i][mt][r];
#pragma unroll 1
    for (int k = 0; k < PT * MT * NR; ++k) {
      const float tot = park[k * kTileThreads];
      const float partner = paired ? row_xor8(tot) : 0.0f;
      const int nb = block_of(i0 + k / (MT * NR));
      const int m = row_of(k / NR % MT, k % NR);
      if (m < p.M && nb < NB)
        store_output(p, p.epi, nb, n_local, m, tot, partner, epi_load(p, p.epi, nb, n_local, m));
    }
  }
}

// Split-K finish: y = the fixed-order sum over splits of part[s][m][n],
// through the same epilogue as the one-split kernel. One thread per output
// (m, n); the SwiGLU / RoPE partner n ^ 8 is summed by the same thread.
// Every load is issued before the first add.
template <int KS>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(GemvArgs p, const float *part) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t MN = (size_t)p.M * p.N;
  if (idx >= MN) return;
  const int m = (int)(idx / p.N), n = (int)(idx % p.N);
  const int nb = n >> 4, n_local = n & 15;
  const bool paired = p.epi == EPI_SWIGLU || p.epi == EPI_QKV;
  // the partner of an unpaired output is itself (loaded, never used)
  const size_t pi = paired ? (size_t)m * p.N + (n ^ 8) : idx;
  float tv[KS], pv[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    tv[s] = part[s * MN + idx];
    pv[s] = part[s * MN + pi];
  }
  float tot = tv[0], partner = pv[0];
#pragma unroll
  for (int s = 1; s < KS; ++s) {
    tot += tv[s];
    partner += pv[s];
  }
  if (!paired) partner = 0.0f;
  store_output(p, p.epi, nb, n_local, m, tot, partner, epi_load(p, p.epi, nb, n_local, m));
}

// Split-K finish of the gate/up GEMM that also emits the down projection's
// planes: one thread per SwiGLU output (m, o), o < N / 2, whose gate
// and up rows are device rows 16 (o / 8) + o % 8 and that + 8 (the
// interleaved layout); every split sum in a fixed order, then the epilogue's
// silu(g) * u. A half-wave holds 32 consecutive outputs of one row, which
// is one quantisation group of the planes.
template <int KS, int D>
__global__ __launch_bounds__(256) void splitk_swiglu_emit_kernel(GemvArgs p, const float *part) {
  const int No = p.N >> 1;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t MN = (size_t)p.M * p.N;
  if (idx >= (size_t)p.M * No) return;  // whole half-waves: No is a multiple of 32
  const int m = (int)(idx / No), o = (int)(idx % No);
  const size_t gi = (size_t)m * p.N + ((o >> 3) << 4) + (o & 7), ui = gi + 8;
  float gv[KS], uv[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    gv[s] = part[s * MN + gi];
    uv[s] = part[s * MN + ui];
  }
  float g = gv[0], u = uv[0];
#pragma unroll
  for (int s = 1; s < KS; ++s) {
    g += gv[s];
    u += uv[s];
  }
  const float v = silu_mul(g, u);
  if (p.y) p.y[(size_t)m * No + o] = v;
  quantize_group<D>(v, o & 31, o >> 5, m, p.M, p.out_q, p.out_meta);
}

// Split-K finish of a residual GEMM (O, down) that also produces the next
// projection's input: y = resid + (fixed-order sum of the splits) is
// written, then the row's RMSNorm with emit_norm_w (kernels.zig:141-220:
// y / sqrt(mean(y^2) + eps) * w) and the group quantiser give the
// planes prep_act_kernel would make from y. One workgroup per row; each
// thread owns 8 consecutive outputs (two 16-byte loads per split, all of a
// thread's loads issued before the first add), so 4 threads (one quad) hold
// a 32-wide group and reduce it with quad DPP exchanges.
constexpr int kEmitThreads = 512;  // rows of up to 4096
template <int KS, int D>
__global__ __launch_bounds__(kEmitThreads) void splitk_resid_emit_kernel(GemvArgs p,
                                                                         const float *part) {
  const int m = blockIdx.x, t = threadIdx.x, N = p.N;
  const size_t MN = (size_t)p.M * N, row = (size_t)m * N;
  const bool act = 8 * t < N;  // N is a multiple of 32: whole quads
  const int n0 = act ? 8 * t : 0;
  __shared__ float red[kEmitThreads / 64 + 1];
  float4 pv[KS][2], rv[2], wv[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    rv[h] = *(const float4 *)(p.resid + row + n0 + 4 * h);
    wv[h] = *(const float4 *)(p.emit_norm_w + n0 + 4 * h);
#pragma unroll
    for (int s = 0; s < KS; ++s) pv[s][h] = *(const float4 *)(part + s * MN + row + n0 + 4 * h);
  }
  float y[8], w8[8];
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int h = i >> 2, e = i & 3;
    float tot = pv[0][h][e];
#pragma unroll
    for (int s = 1; s < KS; ++s) tot += pv[s][h][e];
    y[i] = rv[h][e] + tot;
    w8[i] = wv[h][e];
    ss = fmaf(y[i], y[i], ss);
  }
  if (act) {
    *(float4 *)(p.y + row + n0) = make_float4(y[0], y[1], y[2], y[3]);
    *(float4 *)(p.y + row + n0 + 4) = make_float4(y[4], y[5], y[6], y[7]);
  } else {
    ss = 0.0f;
  }
  ss = wave_sum(ss);
  if ((t & 63) == 0) red[t >> 6] = ss;
  __syncthreads();
  if (t == 0) {
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < kEmitThreads / 64; ++w) sum += red[w];
    red[kEmitThreads / 64] = 1.0f / sqrtf(sum / (float)N + p.in_eps);
  }
  __syncthreads();
  const float inv = red[kEmitThreads / 64];
  // quantize_group's arithmetic over the quad's 32 values
  float v[8];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[i] = (y[i] * inv) * w8[i];
    amax = fmaxf(amax, fabsf(v[i]));
  }
  amax = fmaxf(amax, quad_xor1(amax));
  amax = fmaxf(amax, quad_xor2(amax));
  const int g = n0 >> 5, qp = (n0 >> 3) & 3;
  ActMeta mm;
  if constexpr (D == kPlanesSplit16) {
    const float inv_s = split16_scale(amax, &mm.scale);
    v8h hi, lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      _Float16 hv, lv;
      split16(v[i] * inv_s, hv, lv);
      hi[split16_pos(i)] = hv;
      lo[split16_pos(i)] = lv;
    }
    mm.corr = 0;
    if (act) {
      v8h *q = (v8h *)p.out_q;
      q[(((size_t)g * 2 + 0) * p.M + m) * 4 + qp] = hi;
      q[(((size_t)g * 2 + 1) * p.M + m) * 4 + qp] = lo;
      if (qp == 0) p.out_meta[(size_t)g * p.M + m] = mm;
    }
  } else {
    const float scale = amax / 127.0f;
    const float inv_s = scale == 0.0f ? 0.0f : 1.0f / scale;
    uint64_t packed = 0;
    int csum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int q0 = (int)fminf(fmaxf(roundf(v[i] * inv_s), -127.0f), 127.0f);
      packed |= (uint64_t)(uint8_t)(int8_t)q0 << (8 * i);
      csum += q0;
    }
    csum += quad_xor1(csum);
    csum += quad_xor2(csum);
    if (act) {
      *(uint64_t *)(p.out_q + ((size_t)g * p.M + m) * 32 + qp * 8) = packed;
      mm.scale = scale;
      mm.corr = 7 * csum;
      if (qp == 0) p.out_meta[(size_t)g * p.M + m] = mm;
    }
  }
}

}  // namespace

// Tiles of bm rows x nt row blocks, K split over workgroups (at least 2 quads
// each) toward `target` of them, as far as the partial sums fit the workspace.
static GemmShape tiles(int N, int M, int K, int bm, int nt, int target, size_t ws_floats) {
  GemmShape s;
  const int NB = N / 16, KQ = K / 128;
  s.nt = nt;
  s.mt = bm / 16;
  s.m_tiles = (M + bm - 1) / bm;
  s.n_tiles = (NB + s.nt - 1) / s.nt;
  s.grid = s.m_tiles * s.n_tiles;
  s.ks = 1;
  while (s.grid * s.ks < target && 2 * s.ks <= KQ / 2 && s.ks < 16 &&
         (size_t)(2 * s.ks) * M * N <= ws_floats)
    s.ks *= 2;
  return s;
}

// What a tile kernel's launch and its finishing pass take, in us to within the
// choice this serves (fitted to both heights at 7 shapes of 40 to 2048 rows):
// the most workgroups of a CU, two at a time (one alone takes 1.2 of its share
// of two), times a workgroup's rows and quads (0.0103 us a row and quad with
// Q8, 0.0184 with split-16, 1.3 times that in a 64-row tile); for a K split a
// launch, its loads of ks partial sums and their bytes.
static float tile_cost(const GemmShape &s, int N, int M, int K, int D) {
  const int bm = 16 * s.mt, per_cu = (s.grid * s.ks + 255) / 256;
  const float row = (D == kPlanesQ8 ? 0.0103f : 0.0184f) * (bm == 128 ? 1.0f : 1.3f);
  const float run = (per_cu + 0.2f * (per_cu & 1)) * bm * row * (K / 128) / s.ks;
  return s.ks == 1 ? run : run + 2.0f + 0.6f * s.ks + 0.5e-6f * s.ks * M * N;
}

GemmShape plan_gemm(int N, int M, int K, int D, size_t ws_floats) {
  // decode lanes (16 rows up to 16, so small batches do not pay for 32 rows
  // of MFMA and scaling work): 1 row block per wave for Q8, 2 for split-16,
  // toward about 1024 workgroups (sweeps of the 7B shapes)
  if (M <= 32)
    return tiles(N, M, K, M <= 16 ? 16 : 32,
                 kWaves * (D == kPlanesQ8 ? kRowBlocks<kPlanesQ8> : kRowBlocks<kPlanesSplit16>),
                 1024, ws_floats);
  // prompt chunks: 128- or 64-row tiles toward one workgroup a CU (M = 100,
  // 3584 x 18944: 65 us with 256, 66 with 1024), whichever tile_cost finds
  // cheaper: a row of a 64-row tile costs more, but they round M up to fewer
  // rows, leave a fuller last round and split K less (us, 64 / 128 rows: 2048
  // x 18944 x 3584 454 / 390, 554 x 3584 x 3584 43 / 53, 200 x 9728 x 896 19 /
  // 28, 160 x 3584 x 18944 133 / 113)
  const GemmShape s64 = tiles(N, M, K, 64, kTileN / 16, 256, ws_floats);
  const GemmShape s128 = tiles(N, M, K, 128, kTileN / 16, 256, ws_floats);
  return tile_cost(s64, N, M, K, D) < tile_cost(s128, N, M, K, D) ? s64 : s128;
}

size_t gemm_splitk_floats(int N, int M, int K, int D) {
  const GemmShape s = plan_gemm(N, M, K, D, (size_t)-1);
  return s.ks > 1 ? (size_t)s.ks * M * N : 0;
}

// The launch shape of these arguments; false when they are invalid.
static bool gemm_plan(const GemvArgs &a, GemmShape &s) {
  if (a.N % 16 || a.K % 128 || a.M < 1 || !a.act_q || !a.act_meta ||
      (a.D != kPlanesQ8 && a.D != kPlanesSplit16))
    return false;
  if (a.ss_out || a.arg_parts || a.x_in) return false;  // GEMV-only
  s = plan_gemm(a.N, a.M, a.K, a.D, a.splitk_ws ? a.splitk_ws_floats : 0);
  return true;
}

// A SwiGLU GEMM without a K split emits down's planes from its own tiles
// (their sums are complete), with no partial sums.
static bool gemm_direct_emit(const GemvArgs &a, const GemmShape &s) {
  return a.out_q && a.epi == EPI_SWIGLU && s.ks == 1;
}

// Whether the SwiGLU planes a launch emits overlap the planes it reads: a
// finished tile would overwrite what the others still read.
static bool emit_overlaps_input(const GemvArgs &a) {
  const size_t in_bytes = (size_t)(a.K / 32) * plane_group_bytes(a.D) * a.M;
  const size_t out_bytes = (size_t)(a.N / 64) * plane_group_bytes(a.out_D) * a.M;
  return a.out_q < a.act_q + in_bytes && a.act_q < a.out_q + out_bytes;
}

bool gemm_emit_ok(const GemvArgs &a) {
  GemmShape s;
  if (!a.out_q || !a.out_meta || (a.out_D != kPlanesQ8 && a.out_D != kPlanesSplit16) ||
      !gemm_plan(a, s)) return false;
  if (a.epi == EPI_SWIGLU && ((a.N / 2) % 32 || emit_overlaps_input(a))) return false;
  if (gemm_direct_emit(a, s)) return true;
  if (!a.splitk_ws || (size_t)s.ks * a.M * a.N > a.splitk_ws_floats) return false;
  if (a.epi == EPI_SWIGLU) return true;
  if (a.epi == EPI_RESID)
    return a.emit_norm_w && a.resid && a.y && a.N % 32 == 0 && a.N <= 8 * kEmitThreads;
  return false;
}

hipError_t launch_gemm(const GemvArgs &a, hipStream_t st) {
  GemmShape s;
  if (!gemm_plan(a, s)) return hipErrorInvalidValue;
  const bool emit = a.out_q != nullptr;
  if (emit && !gemm_emit_ok(a)) return hipErrorInvalidValue;
  const dim3 grid(s.grid, s.ks), block(256);
  // the last-arriving split finishes its tile (no finishing kernel) when the
  // counters cover the grid, the tile has at most 32 rows and kFoldSplits
  // splits (their partial sums are read at once), and the epilogue is the
  // tile's own: any but the residual plane emission (whole-row RMSNorm);
  // without a K split any tile emits SwiGLU's planes itself
  const bool fold = (a.splitk_counters && s.grid <= a.splitk_counter_count && s.mt <= 2 &&
                     (!emit || a.epi == EPI_SWIGLU) && (s.ks > 1 || emit) &&
                     s.ks <= kFoldSplits) ||
                    gemm_direct_emit(a, s);
  float *part = s.ks > 1 || (emit && !fold) ? a.splitk_ws : nullptr;
  // (an emission that cannot fold needs the partial sums in the workspace)
  if ((s.ks > 1 || (emit && !fold)) &&
      (!a.splitk_ws || (size_t)s.ks * a.M * a.N > a.splitk_ws_floats))
    return hipErrorInvalidValue;
#define GK_GEMM(DD, BM)                                                                      \
  hipLaunchKernelGGL((gemm_kernel<DD, BM>), grid, block, 0, st, a, s.m_tiles, s.ks, part, \
                     fold ? 1 : 0)
#define GK_TILE(DD, BM)                                                                          \
  hipLaunchKernelGGL((gemm_tile_kernel<DD, BM>), grid, dim3(kTileThreads), 0, st, a, s.m_tiles,  \
                     s.n_tiles, s.ks, part, fold ? 1 : 0)
  if (s.mt > 2) {
    if (a.D == kPlanesQ8) {
      if (s.mt == 4) GK_TILE(kPlanesQ8, 64); else GK_TILE(kPlanesQ8, 128);
    } else {
      if (s.mt == 4) GK_TILE(kPlanesSplit16, 64); else GK_TILE(kPlanesSplit16, 128);
    }
  } else if (a.D == kPlanesQ8) {
    if (s.mt == 1) GK_GEMM(kPlanesQ8, 16); else GK_GEMM(kPlanesQ8, 32);
  } else {
    if (s.mt == 1) GK_GEMM(kPlanesSplit16, 16); else GK_GEMM(kPlanesSplit16, 32);
  }
#undef GK_TILE
#undef GK_GEMM
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || fold) return e;
  if (emit) {
    const float *pc = part;
    const unsigned sw_grid = (unsigned)(((size_t)a.M * (a.N / 2) + 255) / 256);
#define GK_EMIT(KS, DD)                                                                      \
  do {                                                                                      \
    if (a.epi == EPI_SWIGLU)                                                                \
      hipLaunchKernelGGL((splitk_swiglu_emit_kernel<KS, DD>), dim3(sw_grid), dim3(256), 0, \
                         st, a, pc);                                                        \
    else                                                                                    \
      hipLaunchKernelGGL((splitk_resid_emit_kernel<KS, DD>), dim3(a.M), dim3(kEmitThreads), \
                         0, st, a, pc);                                                     \
  } while (0)
#define GK_EMIT_D(KS)                                  \
  do {                                                \
    if (a.out_D == kPlanesQ8) GK_EMIT(KS, kPlanesQ8); else GK_EMIT(KS, kPlanesSplit16); \
  } while (0)
    switch (s.ks) {
      case 1: GK_EMIT_D(1); break;
      case 2: GK_EMIT_D(2); break;
      case 4: GK_EMIT_D(4); break;
      case 8: GK_EMIT_D(8); break;
      default: GK_EMIT_D(16); break;
    }
#undef GK_EMIT_D
#undef GK_EMIT
    return hipGetLastError();
  }
  if (s.ks == 1) return e;
  const size_t MN = (size_t)a.M * a.N;
  const dim3 rg((unsigned)((MN + 255) / 256));
  const float *pc = part;
  switch (s.ks) {
    case 2: hipLaunchKernelGGL((splitk_reduce_kernel<2>), rg, dim3(256), 0, st, a, pc); break;
    case 4: hipLaunchKernelGGL((splitk_reduce_kernel<4>), rg, dim3(256), 0, st, a, pc); break;
    case 8: hipLaunchKernelGGL((splitk_reduce_kernel<8>), rg, dim3(256), 0, st, a, pc); break;
    default: hipLaunchKernelGGL((splitk_reduce_kernel<16>), rg, dim3(256), 0, st, a, pc); break;
  }
  return hipGetLastError();
}

}  // namespace gk
