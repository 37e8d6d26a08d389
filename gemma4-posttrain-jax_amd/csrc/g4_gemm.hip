// Decode-step projection GEMM (g4_linear_bf16): Y[M, N] = X[M, K] . W[N, K]^T, bf16 in, f32
// accumulation, bf16 out, for the rollout's decode batch (M <= 256 rows). Replaces the dense
// projections of forward_attention / forward_mlp (model.py:463-482, 393-396, 500) at S = 1.
//
// At M = 256 the projection is a stream of the weight matrix: every weight byte is used by all
// 256 rows once. A workgroup owns 128 rows x 128 columns of the output (the two row halves of a
// column tile on one XCD, so W is read from HBM once; 256 rows x 64 columns below 129 rows), and
// X (shared by every workgroup) comes from L2. K is walked in stages of 64: the X and W stages are
// DMA'd into a 4-deep LDS ring (buffer_load ... lds), three stages in flight while the fourth is
// multiplied.
//
// LDS layout of a stage: groups of 8 rows x 128 bytes (one DMA instruction: 64 lanes x 16 bytes,
// 8 full 128-byte lines of the row-major operand); within a group, row r's
// 16-byte piece kc sits at slot kc ^ r, so the 16 rows an MFMA operand read touches fall on
// different banks. Each lane DMAs the piece that belongs at its slot.
//
// MFMA v_mfma_f32_16x16x32_bf16 with A = 16 rows of W (output columns) and B = 16 rows of X
// (output rows): lane (grp, col) accumulates Y[m = 16 rb + col][n = 16 cb + 4 grp .. + 3], four
// consecutive outputs of one row. Each of the 8 waves owns a 64 x 32 block of the 128 x 128 or
// 256 x 64 tile (4 x 2 accumulator blocks).
//
// Split-K (ksplit > 1): a workgroup of split s covers K range s; partial sums go to an f32
// workspace [ksplit][M][N] and a second kernel adds them in split order and rounds to bf16, or,
// with no y given, they are left there for a consumer that adds them itself
// (g4_residual_norm_splitk, the residual norm after the MLP's down projection).
#include "g4_common.h"
#include "g4_internal.h"

namespace g4 {
namespace {

constexpr int kGemmRows = 256;  // M rows at most
constexpr int kGemmKT = 64;     // K per stage
constexpr int kGroupBytes = 1024;  // 8 rows x 128 B

// A workgroup's tile: TR rows x TC columns (TR / 64 waves along the rows, TC / WCOLS along the
// columns). TR = 256: all rows, 64 columns (X re-read once per 64 columns). TR = 128: half
// the rows, 128 columns (per CU 1/4 less X + W traffic; the two row halves of a column tile go to
// one XCD, so the second read of its W is an L2 hit).
// Every wave owns 64 x 32 outputs: 8 waves per workgroup, two per SIMD, so one's MFMAs run while the
// other waits on its stage; each output keeps the same K order as with 4 waves of 64 x 64, so the
// results are identical. TR = 128 (M 256): gate/up 31.4-33.2 -> 29.5-31.1 us, down 18.2-18.6 ->
// 17.7-18.0 us, E2B decode step 4.542 -> 4.505 ms; TR = 256 (M 128 / 64): gate/up 29.3-31.3 ->
// 25.9-27.5 / 28.8-29.7 -> 25.4-26.4 us, down 16.2-16.5 -> 14.2-14.9 / 15.0 -> 12.9-13.2 us.
template <int TR>
struct GemmTile {
  static constexpr int TC = 16384 / TR;
  static constexpr int WR = TR / 64;                  // waves along the rows
  static constexpr int WCOLS = 32;                    // columns per wave
  static constexpr int CB = WCOLS / 16;               // 16-column MFMA blocks per wave
  static constexpr int WAVES = WR * (TC / WCOLS);
  static constexpr int THREADS = WAVES * 64;
  static constexpr int XG = TR / 8;   // 8-row groups of X per stage
  static constexpr int WG = TC / 8;   // of W
  static constexpr int DMA = (XG + WG) / WAVES;  // DMA instructions per wave and stage
  static constexpr int STAGE = (XG + WG) * kGroupBytes;        // 40 KiB (TR 256) / 32 KiB (TR 128)
  static_assert(TR == 256 || TR == 128, "tile rows");
  static_assert((XG + WG) % WAVES == 0 && WAVES * 64 <= 1024, "every wave issues the same DMA count");
};

// First weight row of W group j (8 rows) of column tile `tile`. Plain: rows tile * TC + 8 j. Gated
// GELU: each WCOLS-column wave slice holds the WCOLS / 2 gate rows and the WCOLS / 2 up rows of the
// same outputs (gate rows of output o at o, up rows at half + o), tile * TC / 2 outputs before this
// tile.
template <int TC, int WCOLS>
__device__ __forceinline__ int gemm_wrow(bool gelu, int half, int tile, int j) {
  if (!gelu) return tile * TC + 8 * j;
  constexpr int GS = WCOLS / 8;  // 8-row groups per wave slice: the first GS / 2 are gate rows
  const int o = tile * (TC / 2) + (WCOLS / 2) * (j / GS) + 8 * (j % (GS / 2));
  return j % GS < GS / 2 ? o : half + o;
}

// DMA of the stage at K offset k0 into `buf`: wave w moves groups w, w + WAVES, ... of X then of W.
// Lane l of a group instruction takes row 8 g + l / 8 and the 16-byte piece (l % 8) ^ (row % 8) of
// its 128-byte K slice. Past the last stage every load reads beyond its resource (zeros, no memory
// request), so every wave always issues the same number of loads per stage.
template <int TR>
__device__ __forceinline__ void gemm_dma(unsigned char* __restrict__ buf, __amdgpu_buffer_rsrc_t rx,
                                         __amdgpu_buffer_rsrc_t rw, int K, int k0, bool live, uint32_t oob_x,
                                         uint32_t oob_w, int w, int lane, int m0, bool gelu, int half, int tile) {
  using T = GemmTile<TR>;
  const int rl = lane >> 3;        // row within the group
  const int kc = (lane & 7) ^ rl;  // 16-byte piece this lane fetches (row % 8 == rl)
#pragma unroll
  for (int i = 0; i < T::DMA; ++i) {
    const int g = w + T::WAVES * i;  // groups 0..XG-1: X, then W
    const bool is_x = g < T::XG;
    const int row = is_x ? m0 + 8 * g + rl : gemm_wrow<T::TC, T::WCOLS>(gelu, half, tile, g - T::XG) + rl;
    const uint32_t off = (uint32_t)(row * K + k0 + 8 * kc) * 2u;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(is_x ? rx : rw,
                                             (__attribute__((address_space(3))) void*)(buf + g * kGroupBytes), 16,
                                             live ? off : (is_x ? oob_x : oob_w), 0, 0, 0);
  }
}

// LDS byte offset of the 16-byte MFMA operand piece kc of row `row` (within the X or W part of a
// stage).
__device__ __forceinline__ uint32_t gemm_operand_at(uint32_t part, int row, int kc) {
  const int r = row & 7;
  return part + (uint32_t)((row >> 3) * kGroupBytes + (8 * r + (kc ^ r)) * 16);
}

// The operand reads are issued as ds_read_b128 in inline assembly (lds_read16) and waited for
// explicitly (lgkmcnt, tied to the eight operand registers). Read through C++, the compiler cannot
// tell the stage being multiplied from the stages the DMA is still filling, and at some steps of
// the ring waited for every DMA in flight (vmcnt(0)); the stage's own DMAs are already covered by
// the s_waitcnt vmcnt + s_barrier that starts each step.
// Wave (wr, wc) multiplies rows [64 wr, 64 wr + 64) of the X part by rows [WCOLS wc, WCOLS wc +
// WCOLS) of the W part.
template <int TR>
__device__ __forceinline__ void gemm_compute(const unsigned char* __restrict__ buf,
                                             floatx4 (&acc)[4][GemmTile<TR>::CB], int wr, int wc, int col, int grp) {
  constexpr int CB = GemmTile<TR>::CB, WCOLS = GemmTile<TR>::WCOLS;
  const uint32_t xs = lds_addr(buf);
  const uint32_t ws = xs + GemmTile<TR>::XG * kGroupBytes;
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) {
    static_assert(CB == 2, "operand wait list");
    u32x4 a[CB], b[4];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) a[cb] = lds_read16(gemm_operand_at(ws, WCOLS * wc + 16 * cb + col, 4 * kh + grp));
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) b[rb] = lds_read16(gemm_operand_at(xs, 64 * wr + 16 * rb + col, 4 * kh + grp));
    __asm__ volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0]), "+v"(a[1]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mfma16x16x32(as_bf16x8(a[cb]), as_bf16x8(b[rb]), acc[rb][cb]);
  }
}

// Waits until at most min(lines, MAX) lines' loads (G each) are outstanding.
template <int G, int MAX>
__device__ __forceinline__ void wait_lines(int lines) {
  if constexpr (MAX > 0) {
    if (lines >= MAX)
      __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX * G) : "memory");
    else
      wait_lines<G, MAX - 1>(lines);
  } else {
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}

struct GemmLoop {
  __amdgpu_buffer_rsrc_t rx, rw;
  int K, kbeg, nst;
  uint32_t oob_x, oob_w;
  int w, lane, col, grp, wr, wc, m0, half, tile;
  bool gelu;
};

// One pipeline step: stage s is in `cur` (stages s + 1, s + 2 in flight); stage s + 3 is
// requested into `fre` (the buffer of stage s - 1, which every wave has finished with) after the
// stage's MFMAs are issued, so a DMA issue that waits for room in the memory queue does not hold
// them back (down projection 19.3 -> 18.6 us).
template <int TR>
__device__ __forceinline__ void gemm_step(const unsigned char* __restrict__ cur, unsigned char* __restrict__ fre,
                                          floatx4 (&acc)[4][GemmTile<TR>::CB], const GemmLoop& L, int s) {
  // this wave's DMAs of stage s have landed (stages s + 1, s + 2 may not have), then every wave's
  __asm__ volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * GemmTile<TR>::DMA) : "memory");
  gemm_compute<TR>(cur, acc, L.wr, L.wc, L.col, L.grp);
  gemm_dma<TR>(fre, L.rx, L.rw, L.K, L.kbeg + (s + 3) * kGemmKT, s + 3 < L.nst, L.oob_x, L.oob_w, L.w, L.lane, L.m0,
               L.gelu, L.half, L.tile);
}

// Work units (column tile, K split), each covered by n_halves = ceil(M / TR) workgroups (row
// halves). Workgroups are dealt to the 8 XCDs round robin (i mod 8); when the unit count is a
// multiple of 8, workgroup i takes unit 8 (j / n_halves) + i mod 8 and half j mod n_halves
// (j = i / 8), so all halves of a unit share an XCD (one HBM read of its W) and, with ksplit
// dividing 8, every XCD works on one K split, whose slice of X its L2 then holds for all its
// column tiles. The unit is (tile u / ksplit, split u mod ksplit). K / ksplit must be a multiple
// of 64.
template <int TR>
__global__ __launch_bounds__(GemmTile<TR>::THREADS) void linear_bf16_kernel(G4LinearArgs a, float* partials) {
  using T = GemmTile<TR>;
  __shared__ __attribute__((aligned(1024))) unsigned char b0[T::STAGE], b1[T::STAGE], b2[T::STAGE], b3[T::STAGE];
  GemmLoop L;
  L.lane = threadIdx.x & 63;
  L.w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  L.col = L.lane & 15;
  L.grp = L.lane >> 4;
  L.wr = L.w % T::WR;
  L.wc = L.w / T::WR;
  const int n_halves = (a.m + TR - 1) / TR;
  const int n_units = a.n / T::TC * a.ksplit;
  const int i = (int)blockIdx.x;
  int unit, hf;
  if (n_units % 8 == 0) {
    const int j = i >> 3;
    unit = 8 * (j / n_halves) + (i & 7);
    hf = j % n_halves;
  } else {
    unit = i / n_halves;
    hf = i % n_halves;
  }
  L.tile = unit / a.ksplit;
  const int split = unit - L.tile * a.ksplit;
  L.m0 = hf * TR;
  const int n0 = L.tile * T::TC;
  L.K = a.k;
  const int kper = L.K / a.ksplit;
  L.kbeg = split * kper;
  L.nst = kper / kGemmKT;
  const uint32_t xbytes = (uint32_t)a.m * (uint32_t)L.K * 2u;  // rows >= M read as zeros
  const uint32_t wbytes = (uint32_t)a.n * (uint32_t)L.K * 2u;
  L.oob_x = xbytes;
  L.oob_w = wbytes;
  L.rx = make_rsrc(a.x, xbytes);
  L.rw = make_rsrc(a.w, wbytes);
  L.gelu = a.epilogue == G4_LINEAR_GELU_MUL;
  L.half = a.n / 2;

  constexpr int CB = T::CB;
  floatx4 acc[4][CB];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[r][c] = floatx4{0.f, 0.f, 0.f, 0.f};

  gemm_dma<TR>(b0, L.rx, L.rw, L.K, L.kbeg, true, xbytes, wbytes, L.w, L.lane, L.m0, L.gelu, L.half, L.tile);
  gemm_dma<TR>(b1, L.rx, L.rw, L.K, L.kbeg + kGemmKT, L.nst > 1, xbytes, wbytes, L.w, L.lane, L.m0, L.gelu, L.half,
               L.tile);
  gemm_dma<TR>(b2, L.rx, L.rw, L.K, L.kbeg + 2 * kGemmKT, L.nst > 2, xbytes, wbytes, L.w, L.lane, L.m0, L.gelu,
               L.half, L.tile);
  for (int s = 0; s < L.nst; s += 4) {
    gemm_step<TR>(b0, b3, acc, L, s);
    if (s + 1 < L.nst) gemm_step<TR>(b1, b0, acc, L, s + 1);
    if (s + 2 < L.nst) gemm_step<TR>(b2, b1, acc, L, s + 2);
    if (s + 3 < L.nst) gemm_step<TR>(b3, b2, acc, L, s + 3);
  }
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the trailing (zero) DMAs

  // lane (grp, col) holds Y[m = m0 + 64 wr + 16 rb + col][n = n0 + WCOLS wc + 16 cb + 4 grp + j]
  if (L.gelu) {  // cb < CB / 2: gate columns; cb + CB / 2: the up columns of the same outputs
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      const int m = L.m0 + 64 * L.wr + 16 * rb + L.col;
      if (m < a.m) {
#pragma unroll
        for (int cb = 0; cb < CB / 2; ++cb) {
          float y[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            y[j] = gelu_tanh_mul(round_bf16(acc[rb][cb][j]), round_bf16(acc[rb][cb + CB / 2][j]));
          uint16_t* dst = reinterpret_cast<uint16_t*>(a.y) + (int64_t)m * a.ldy + L.tile * (T::TC / 2) +
                          (T::WCOLS / 2) * L.wc + 16 * cb + 4 * L.grp;
          *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
        }
      }
    }
    return;
  }
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const int m = L.m0 + 64 * L.wr + 16 * rb + L.col;
    if (m < a.m) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const int n = n0 + T::WCOLS * L.wc + 16 * cb + 4 * L.grp;
        if (a.ksplit == 1) {
          uint16_t* y = reinterpret_cast<uint16_t*>(a.y) + (int64_t)m * a.ldy + n;
          *reinterpret_cast<uint2*>(y) = make_uint2(pack_bf16x2(acc[rb][cb][0], acc[rb][cb][1]),
                                                    pack_bf16x2(acc[rb][cb][2], acc[rb][cb][3]));
        } else {
          float* p = partials + ((int64_t)split * a.m + m) * a.n + n;
          *reinterpret_cast<floatx4*>(p) = acc[rb][cb];
        }
      }
    }
  }
}

// --- few rows --------------------------------------------------------------------------------------
//
// A batch of a few rows only streams the weights: what counts is how many of their bytes are in flight
// and how short the chain of one launch is, not the tile's reuse. A workgroup of NW waves owns 16 CB
// columns x 8 XG rows of one K split; its waves divide the K range into 128-byte lines and each streams
// its own lines of W and X into its own LDS slots (NBUF lines in flight), so there is no barrier until
// the waves' partial sums meet in LDS at the end (added in wave order). The ring kernel above keeps one
// stage sequence per workgroup, three stages ahead, and half its tile on padding rows here.
// In HIP graphs over rotating weights (us; the ring kernel, for q/k/v and o hipBLASLt, before; now):
//   rows   down, 8 K splits   q/k/v (N 3072)   o (N 2048)    K = 2048 (down 8192)
//      1      12.0    7.3       11.3    4.2     11.0   4.0
//     32      12.3    9.0       11.5    6.0     11.2   4.7
//     64      12.8   11.0       11.9    7.1     11.7   5.7
//    128      14.1 (ring)       14.4    9.1     11.1   6.7
// (gate/up: launch_skinny_wide). Loaded straight into operand registers, the 16 rows of
// an operand make every lane of an instruction a request of its own, 64 cycles per KiB instead of 16: q/k/v
// at 32 rows 8.2 us. A load past a wave's last line costs the same time although it reads nothing, so
// none is issued.
constexpr int kSkinnyWaves = 4;
// It takes every shape up to 64 rows, and beyond what one round of its largest tile covers (gate/up at
// 128 rows takes two: 27.3 us against the ring kernel's 24.6).
constexpr int kSkinnyRows = 64;
constexpr int kSkinnyMaxCost = 16;
constexpr int kSkinnyWideCols = 4096;  // columns from which one wave per column block fills the chip

template <int NW, int CB, int XG, int NBUF, bool GELU>
__global__ __launch_bounds__(NW * 64) void linear_skinny_kernel(G4LinearArgs a, float* partials) {
  constexpr int MB = XG / 2, BLKS = CB * MB;
  constexpr int GROUPS = 2 * CB + XG;  // DMA instructions (8 rows x 128 bytes) per line: W, then X
  static_assert(!GELU || CB == 1 || CB % 2 == 0, "gate and up blocks in pairs, or halves of one block");
  static_assert(BLKS <= NBUF * GROUPS, "the partial sums reuse the wave's slots");
  static_assert((NBUF - 1) * GROUPS < 64, "vmcnt counts up to 63");
  __shared__ __attribute__((aligned(1024))) unsigned char slots[NW][NBUF][GROUPS][kGroupBytes];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  // row groups of a (column tile, K split) unit go to one XCD, as in linear_bf16_kernel
  const int n_rg = (a.m + 8 * XG - 1) / (8 * XG), n_units = a.n / (16 * CB) * a.ksplit;
  const int j = (int)blockIdx.x >> 3;
  const bool dealt = n_units % 8 == 0;
  const int unit = dealt ? 8 * (j / n_rg) + ((int)blockIdx.x & 7) : (int)blockIdx.x / n_rg;
  const int m0 = 8 * XG * (dealt ? j % n_rg : (int)blockIdx.x % n_rg);
  const int tile = unit / a.ksplit, split = unit - tile * a.ksplit;
  const int K = a.k, kper = K / a.ksplit;
  const int lines = kper / 64;
  const int s0 = lines * w / NW, cnt = lines * (w + 1) / NW - s0;  // this wave's lines
  const int half = a.n / 2;
  const uint32_t wbytes = (uint32_t)a.n * (uint32_t)K * 2u, xbytes = (uint32_t)a.m * (uint32_t)K * 2u;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.w, wbytes), rx = make_rsrc(a.x, xbytes);
  const uint32_t rl = (uint32_t)lane >> 3;
  const uint32_t lane_ofs = rl * (uint32_t)K * 2u + (((uint32_t)lane & 7u) ^ rl) * 16u + (uint32_t)(split * kper) * 2u;

  floatx4 acc[CB][MB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[cb][mb] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto load = [&](int buf, int i) {
    const uint32_t k2 = (uint32_t)(s0 + i) * 128u;
#pragma unroll
    for (int g = 0; g < 2 * CB; ++g) {
      const int row = !GELU    ? tile * 16 * CB + 8 * g  // the first CB groups of a gated tile: gate rows
                      : g < CB ? tile * 8 * CB + 8 * g
                               : half + tile * 8 * CB + 8 * (g - CB);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void*)&slots[w][buf][g][0], 16,
                                               lane_ofs + (uint32_t)row * (uint32_t)K * 2u + k2, 0, 0, kNonTemporal);
    }
#pragma unroll
    for (int g = 0; g < XG; ++g)  // rows >= M: beyond the resource, zeros
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rx, (__attribute__((address_space(3))) void*)&slots[w][buf][2 * CB + g][0], 16,
          lane_ofs + (uint32_t)(m0 + 8 * g) * (uint32_t)K * 2u + k2, 0, 0, 0);
  };
  const uint32_t slot0 = lds_addr(&slots[w][0][0][0]);
  const int orow = col & 7;
  const uint32_t opnd[2] = {slot0 + (uint32_t)((col >> 3) * kGroupBytes + (8 * orow + (grp ^ orow)) * 16),
                            slot0 + (uint32_t)((col >> 3) * kGroupBytes + (8 * orow + ((4 + grp) ^ orow)) * 16)};
  auto mac = [&](int buf) {
    u32x4 wv[2][CB], xv[2][MB];
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      const uint32_t at = opnd[kh] + (uint32_t)(buf * GROUPS * kGroupBytes);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) xv[kh][mb] = lds_read16_at(at, (2 * CB + 2 * mb) * kGroupBytes);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) wv[kh][cb] = lds_read16_at(at, 2 * cb * kGroupBytes);
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) lgkm_wait(0, xv[kh][mb]);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) lgkm_wait(0, wv[kh][cb]);
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          acc[cb][mb] = mfma16x16x32(as_bf16x8(wv[kh][cb]), as_bf16x8(xv[kh][mb]), acc[cb][mb]);
  };
  // line i sits in slot i % NBUF; while it is multiplied lines i + 1 .. i + NBUF - 1 are in flight. Its
  // slot's operand reads have returned before the next line is requested into it.
#pragma unroll
  for (int i = 0; i < NBUF; ++i)
    if (i < cnt) load(i, i);
#pragma unroll 1
  for (int i = 0; i < cnt; i += NBUF) {
#pragma unroll
    for (int u = 0; u < NBUF; ++u) {
      if (i + u < cnt) {
        // this line has landed; the lines requested after it, min(cnt - 1 - i - u, NBUF - 1), may not have
        wait_lines<GROUPS, NBUF - 1>(cnt - 1 - (i + u));
        mac(u);
        if (i + u + NBUF < cnt) load(u, i + u + NBUF);
      }
    }
  }
  floatx4* red = reinterpret_cast<floatx4*>(&slots[w][0][0][0]);  // [BLKS][64] in this wave's own slots
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) red[(cb * MB + mb) * 64 + lane] = acc[cb][mb];
  __syncthreads();

  // quad q: block q / 64, lane q % 64 of the MFMA result: Y[m = m0 + 16 mb + col][4 consecutive columns]
  auto sum = [&](int blk, int l) {
    floatx4 t = reinterpret_cast<const floatx4*>(&slots[0][0][0][0])[blk * 64 + l];
#pragma unroll
    for (int i = 1; i < NW; ++i) t += reinterpret_cast<const floatx4*>(&slots[i][0][0][0])[blk * 64 + l];
    return t;
  };
  // (gated GELU: the up quad of a gate quad is CB / 2 column blocks on; with CB = 1, rows 0 .. 7 of the
  // block are gate rows and 8 .. 15 their up rows, 32 lanes on)
  constexpr int QL = GELU && CB == 1 ? 32 : 64;
  constexpr int QUADS = GELU && CB > 1 ? BLKS / 2 * 64 : BLKS * QL;
  for (int q = threadIdx.x; q < QUADS; q += NW * 64) {
    const int blk = q / QL, l = q % QL, cb = blk / MB, mb = blk - cb * MB;
    const int m = m0 + 16 * mb + (l & 15);
    if (m >= a.m) continue;
    const floatx4 t = sum(blk, l);
    if (GELU) {
      const floatx4 up = CB == 1 ? sum(blk, l + 32) : sum(blk + BLKS / 2, l);
      float y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = gelu_tanh_mul(round_bf16(t[j]), round_bf16(up[j]));
      uint16_t* dst = reinterpret_cast<uint16_t*>(a.y) + (int64_t)m * a.ldy + tile * 8 * CB + 16 * cb + 4 * (l >> 4);
      *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
    } else {
      const int n = tile * 16 * CB + 16 * cb + 4 * (l >> 4);
      if (a.ksplit == 1) {
        uint16_t* dst = reinterpret_cast<uint16_t*>(a.y) + (int64_t)m * a.ldy + n;
        *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(t[0], t[1]), pack_bf16x2(t[2], t[3]));
      } else {
        *reinterpret_cast<floatx4*>(partials + ((int64_t)split * a.m + m) * a.n + n) = t;
      }
    }
  }
}

// LDS slots per wave (lines in flight): what lets two workgroups share a CU where a line is small
// (64 - 80 KiB; (CB 2, XG 4): 2 slots 14.5 us, 4 slots 16.2 for gate/up at 32 rows), else all of it. A
// one-wave workgroup takes 40 KiB, four to a CU (80 KiB: 24576 columns at 16 rows 28.8 -> 36.5 us).
template <int NW, int CB, int XG>
constexpr int skinny_slots() {
  if (NW == 1) return 40 / (2 * CB + XG);
  return CB == 1 ? (XG == 2 ? 4 : XG == 4 ? 3 : 2) : CB == 2 ? (XG == 4 ? 2 : 3) : (XG == 8 ? 2 : 3);
}

template <int NW, int CB, int XG>
void launch_skinny(const G4LinearArgs& a, float* partials, hipStream_t st) {
  constexpr int NBUF = skinny_slots<NW, CB, XG>();
  const int n_rg = (a.m + 8 * XG - 1) / (8 * XG);
  const dim3 grid((unsigned)(a.n / (16 * CB) * a.ksplit * n_rg)), block(NW * 64);
  if constexpr (CB % 2 == 0 || NW == 1)
    if (a.epilogue == G4_LINEAR_GELU_MUL) {
      hipLaunchKernelGGL((linear_skinny_kernel<NW, CB, XG, NBUF, true>), grid, block, 0, st, a, partials);
      return;
    }
  hipLaunchKernelGGL((linear_skinny_kernel<NW, CB, XG, NBUF, false>), grid, block, 0, st, a, partials);
}

// Many columns, one K range (gate/up): one wave per workgroup walks all of K for its 16 CB columns, so the
// sums keep the ring kernel's order (split over four waves the 16384 columns take 12.9 us instead of 15.9
// at 16 rows, but the gated GELU's roundings then move 3e-4 of the MLP's output). One column block per
// wave while that leaves at most two per CU, else two (gate/up + GELU, K = 2048, us at 1 / 16 / 64 rows,
// ring kernel, now: 4096 columns 18.3 / 18.2 / 19.9, 7.5 / 7.7 / 11.1; 8192 19.0 / 19.0 / 20.8, 9.6 / 9.2 /
// 13.0; 16384 21.8 / 21.7 / 23.5, 16.3 / 15.9 / 19.3; 24576 x 3072 54 / 52 / 56, 28 / 29 / 40).
template <int CB>
void launch_skinny_wide(const G4LinearArgs& a, float* partials, hipStream_t st) {
  if (a.m <= 16)
    launch_skinny<1, CB, 2>(a, partials, st);
  else if (a.m <= 32)
    launch_skinny<1, CB, 4>(a, partials, st);
  else
    launch_skinny<1, CB, 8>(a, partials, st);
}

// Rows up to which it takes a shape of many columns. Its workgroups (32 columns, 40 KiB of LDS) sit four to a
// CU; where their last round is less than half full and long, the ring kernel is as fast from 57 rows (us at 48
// / 64 rows, ring kernel / this: 43008 x 5376 134.5 / 128.7, 138.5 / 142.4; x 4096 108 / 100, 109 / 107;
// at 49152 x 4096 116 / 113, 32768 x 5376 96 / 80 at 64 rows).
int skinny_wide_rows(const G4LinearArgs& a) {
  const int groups = a.n / 32;
  return a.k > 4096 && groups >= 1152 && groups < 1536 ? 56 : kSkinnyRows;
}

// The tile (16 CB columns x 8 XG rows) whose workgroups bring the least through each of the 256 CUs:
// cost = ceil(workgroups / 256) x (2 CB + XG) KiB per line.
struct SkinnyTile {
  int cb, xg;
  int64_t cost;
};

SkinnyTile skinny_tile(const G4LinearArgs& a, bool gelu) {
  SkinnyTile best = {0, 0, 0};
  for (int cb = gelu ? 2 : 1; cb <= 4; cb *= 2)
    for (int xg = 2; xg <= 8; xg *= 2) {
      if (xg > 2 && 4 * xg >= a.m) break;  // half the rows would do
      const int64_t groups = (int64_t)(a.n / (16 * cb)) * a.ksplit * ((a.m + 8 * xg - 1) / (8 * xg));
      // (4, 2) leaves one workgroup per CU, whose last lines nothing overlaps: gate/up at 16 rows 13.4 us
      // against 12.9 with two (2, 2) workgroups per CU
      const int64_t cost = (groups + 255) / 256 * (2 * cb + xg) + (cb == 4 && xg == 2 ? 3 : 0);
      if (!best.cb || cost < best.cost) best = {cb, xg, cost};
    }
  return best;
}

void launch_skinny_tile(const SkinnyTile& t, const G4LinearArgs& a, float* partials, hipStream_t st) {
  switch (t.cb * 16 + t.xg) {
    case 16 + 2: return launch_skinny<kSkinnyWaves, 1, 2>(a, partials, st);
    case 16 + 4: return launch_skinny<kSkinnyWaves, 1, 4>(a, partials, st);
    case 16 + 8: return launch_skinny<kSkinnyWaves, 1, 8>(a, partials, st);
    case 32 + 2: return launch_skinny<kSkinnyWaves, 2, 2>(a, partials, st);
    case 32 + 4: return launch_skinny<kSkinnyWaves, 2, 4>(a, partials, st);
    case 32 + 8: return launch_skinny<kSkinnyWaves, 2, 8>(a, partials, st);
    case 64 + 2: return launch_skinny<kSkinnyWaves, 4, 2>(a, partials, st);
    case 64 + 4: return launch_skinny<kSkinnyWaves, 4, 4>(a, partials, st);
    default: return launch_skinny<kSkinnyWaves, 4, 8>(a, partials, st);
  }
}

// Y = sum of the split partials (split order), rounded to bf16; 4 outputs per thread.
__global__ __launch_bounds__(256) void linear_reduce_kernel(G4LinearArgs a, const float* partials) {
  const int64_t i4 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t total = (int64_t)a.m * a.n;
  if (i4 >= total) return;
  floatx4 s = *reinterpret_cast<const floatx4*>(partials + i4);
  for (int k = 1; k < a.ksplit; ++k) s += *reinterpret_cast<const floatx4*>(partials + (int64_t)k * total + i4);
  const int64_t m = i4 / a.n, n = i4 - m * a.n;
  uint16_t* y = reinterpret_cast<uint16_t*>(a.y) + m * a.ldy + n;
  *reinterpret_cast<uint2*>(y) = make_uint2(pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]));
}

}  // namespace
}  // namespace g4

extern "C" size_t g4_linear_workspace_size(const G4LinearArgs* args) {
  if (!args || args->ksplit <= 1 || args->m <= 0 || args->n <= 0) return 0;
  return (size_t)args->ksplit * (size_t)args->m * (size_t)args->n * 4u;
}

extern "C" int g4_linear_bf16(const G4LinearArgs* args, void* stream) {
  using namespace g4;
  if (!args) return fail(G4_ERR_INVALID, "g4_linear_bf16: args is NULL");
  const G4LinearArgs& a = *args;
  if (!a.x || !a.w || (!a.y && a.ksplit <= 1)) return fail(G4_ERR_INVALID, "g4_linear_bf16: NULL x/w/y");
  if (a.m <= 0 || a.m > kGemmRows) return fail(G4_ERR_UNSUPPORTED, "g4_linear_bf16: m %d (1..%d)", a.m, kGemmRows);
  if (a.n <= 0 || a.n % 64) return fail(G4_ERR_UNSUPPORTED, "g4_linear_bf16: n %d (a multiple of 64)", a.n);
  if (a.ksplit < 1 || a.ksplit > 64) return fail(G4_ERR_INVALID, "g4_linear_bf16: ksplit %d (1..64)", a.ksplit);
  if (a.k <= 0 || a.k % (kGemmKT * a.ksplit))
    return fail(G4_ERR_UNSUPPORTED, "g4_linear_bf16: k %d (a multiple of %d x ksplit %d)", a.k, kGemmKT, a.ksplit);
  if ((int64_t)a.m * a.k * 2 >= (int64_t)1 << 31 || (int64_t)a.n * a.k * 2 >= (int64_t)1 << 31)
    return fail(G4_ERR_UNSUPPORTED, "g4_linear_bf16: operands beyond 2 GiB");
  if (a.epilogue != G4_LINEAR_PLAIN && a.epilogue != G4_LINEAR_GELU_MUL)
    return fail(G4_ERR_INVALID, "g4_linear_bf16: epilogue %d", a.epilogue);
  if (a.epilogue == G4_LINEAR_GELU_MUL && (a.ksplit != 1 || !a.y))
    return fail(G4_ERR_UNSUPPORTED, "g4_linear_bf16: the gated-GELU epilogue needs ksplit 1 and y");
  const int ycols = a.epilogue == G4_LINEAR_GELU_MUL ? a.n / 2 : a.n;
  if (a.y && (a.ldy < ycols || a.ldy % 4))
    return fail(G4_ERR_INVALID, "g4_linear_bf16: ldy %d (>= n, a multiple of 4)", a.ldy);
  if ((reinterpret_cast<uintptr_t>(a.y) & 7) || (reinterpret_cast<uintptr_t>(a.x) & 15) ||
      (reinterpret_cast<uintptr_t>(a.w) & 15))
    return fail(G4_ERR_INVALID, "g4_linear_bf16: x/w need 16-byte and y 8-byte alignment");
  const size_t need = g4_linear_workspace_size(args);
  if (need && (!a.workspace || a.workspace_bytes < need))
    return fail(G4_ERR_WORKSPACE, "g4_linear_bf16: ksplit %d needs %zu B of workspace (have %zu)", a.ksplit, need,
                a.workspace ? a.workspace_bytes : (size_t)0);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  float* partials = reinterpret_cast<float*>(a.workspace);
  // few rows: the streaming kernel (neither the choice nor the order of the sums depends on the epilogue:
  // the gated GELU's products are the plain call's bit for bit); else 128 x 128 tiles when the rows fill
  // two halves and the columns divide by 128; else 256 x 64
  const bool wide = a.n >= kSkinnyWideCols && a.ksplit == 1;
  if (wide && a.m <= skinny_wide_rows(a)) {
    if (a.n / 16 <= 512)
      launch_skinny_wide<1>(a, partials, st);
    else
      launch_skinny_wide<2>(a, partials, st);
  } else if (!wide && (a.m <= kSkinnyRows || skinny_tile(a, false).cost <= kSkinnyMaxCost))
    launch_skinny_tile(skinny_tile(a, a.epilogue == G4_LINEAR_GELU_MUL), a, partials, st);
  else if (a.m > 128 && a.n % 128 == 0)
    hipLaunchKernelGGL(linear_bf16_kernel<128>, dim3((unsigned)(a.n / 128 * a.ksplit * 2)), dim3(GemmTile<128>::THREADS), 0,
                       st, a, partials);
  else
    hipLaunchKernelGGL(linear_bf16_kernel<256>, dim3((unsigned)(a.n / 64 * a.ksplit)), dim3(GemmTile<256>::THREADS), 0, st,
                       a, partials);
  if (int rc = check_launch("g4_linear_bf16")) return rc;
  if (a.ksplit > 1 && a.y) {  // without y the partials stay in the workspace for the consumer
    const int64_t quads = ((int64_t)a.m * a.n) / 4;
    hipLaunchKernelGGL(linear_reduce_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, a,
                       (const float*)partials);
    return check_launch("g4_linear_bf16 (split-K sum)");
  }
  return G4_OK;
}
