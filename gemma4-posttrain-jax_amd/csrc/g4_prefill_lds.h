// bf16 prefill attention with the key / value chunks staged through LDS (head dims 128, 256, 512);
// included by g4_prefill.hip after prefill_bf16_kernel.
//
// A workgroup of NW waves owns NW * NB * 16/R consecutive query positions of one (b, kv head);
// each wave owns NB column blocks of 16 query rows (16/R positions x R heads each), so every K and
// V^T operand tile it reads from LDS feeds NB MFMAs. The key range is walked in 32-key chunks:
// every chunk's K and V^T are DMA'd into LDS once per workgroup (buffer_load ... lds, each wave
// issuing an equal share, into rings of 4 slots, 2 at head dim 512, where a chunk's operand is 32 KiB)
// as lane-ordered MFMA operand tiles, and all waves read them from there (head dim 512, 4 x 1024 tokens
// without pads, 2 kv heads of 4: 630 us with one wave per SIMD loading its own operands, 102-106 us here). The
// key-mask bytes of the row are staged in LDS once, so a chunk's validity is one LDS byte per lane and a ballot.
//
// Same two passes as prefill_bf16_kernel (the reference rounds probabilities after the full-row
// softmax): pass 1 streams K for each row's max and sum, pass 2 streams K and V and forms the bf16
// probabilities of the full-row softmax for the value product, at head dims 128 and 256 evaluated as
// __expf(s - m) * (1/l): the hardware exp and the row's reciprocal instead of expf and a division per score,
// a few f32 ulps from exp(s - m) / l, so a probability at a bf16 rounding boundary may round one bf16 step
// the other way (head dim 512: pf_exp, pf_prob). Workgroups are launched heaviest (latest positions, longest causal key range)
// first.
//
// What bounds it is the issue rate of each SIMD's two waves, VALU work included, more than the
// MFMAs, so the schedule is built around three things:
//  - a wave-uniform fast path: a chunk whose 32 keys every row of the wave may see (key mask,
//    causal limit, window) skips the per-key selects, and its scores are rounded two per
//    conversion instruction;
//  - operand tiles read from LDS through a rolling window: tile t + W is requested right after the
//    MFMAs of tile t, so the LDS latency hides behind the MFMAs in flight;
//  - in pass 2 the two waves sharing a SIMD (w, w + NW/2) are half a step apart. One runs the
//    MFMA phase (the values of chunk c-1, then the QK of chunk c) while the other runs the VALU
//    phase (the probabilities of a chunk), at raised priority while in the MFMA phase.

constexpr int kPfMaxSeq = 32768;  // key-mask bytes staged in LDS

template <int D, int NW>
struct PfShape {
  static constexpr int KT = 2 * (D / 32);  // K operand tiles per chunk: (bb, s)
  static constexpr int VT = D / 16;        // V^T operand tiles per chunk: d-blocks
  static constexpr int SLOTS = D >= 512 ? 2 : 4;  // ring slots of each operand in pass 2
  static constexpr int CHUNK = KT * 1024;         // LDS bytes of a chunk's K (and V^T) tiles
  static_assert(KT == VT, "K and V^T chunks share the ring");
  static constexpr int KT_W = KT / NW;     // DMA'd by each wave
  static constexpr int VT_W = VT / NW;
  static_assert(KT % NW == 0 && VT % NW == 0, "tiles split evenly over the waves");
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The 8 scores of one column block (both 16-key halves), each rounded to bf16, two values per
// conversion instruction; element e is key 8 * grp + e of the chunk.
__device__ __forceinline__ void pf_round8(const floatx4 (&acc)[2], float (&sc)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t w = pack_bf16x2(acc[j >> 1][2 * (j & 1)], acc[j >> 1][2 * (j & 1) + 1]);
    sc[2 * j] = __uint_as_float(w << 16);
    sc[2 * j + 1] = __uint_as_float(w & 0xffff0000u);
  }
}

// S^T of one chunk for the wave's NB column blocks: K operand tiles (KT = 2 halves x KS d-slices,
// 1 KiB each, this lane's pieces from LDS address kbase) against the q operands in registers, a rolling window of WIN
// tiles in flight (each read waited for right before its MFMAs; the chunk's DMA is covered by the
// caller's vmcnt wait + barrier).
template <int KT, int KS, int NB, int WIN>
__device__ __forceinline__ void pf_qk(uint32_t kbase, const bf16x8 (&qop)[NB][KS], floatx4 (&acc)[NB][2]) {
  static_assert(WIN >= 1 && WIN <= 8 && WIN <= KT, "window of LDS reads (lgkm_wait counts up to 7)");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) acc[cb][0] = acc[cb][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  u32x4 kv[WIN];
#pragma unroll
  for (int j = 0; j < WIN; ++j) kv[j] = lds_read16_at(kbase, 1024 * j);
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const int bb = t / KS, s = t - bb * KS;
    const int later = KT - 1 - t < WIN - 1 ? KT - 1 - t : WIN - 1;  // reads issued after tile t's
    lgkm_wait(later, kv[t % WIN]);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) acc[cb][bb] = mfma16x16x32(as_bf16x8(kv[t % WIN]), qop[cb][s], acc[cb][bb]);
    if (t + WIN < KT) kv[t % WIN] = lds_read16_at(kbase, 1024 * (t + WIN));
  }
  __builtin_amdgcn_sched_barrier(0);
}

// O^T += V^T P^T over one chunk: VT value operand tiles (one per 16-dim block, 1 KiB each, this
// lane's pieces from LDS address vbase) against the wave's probabilities, a rolling window of WIN tiles in flight.
template <int VT, int NB, int WIN>
__device__ __forceinline__ void pf_pv(uint32_t vbase, const bf16x8 (&pop)[NB], floatx4 (&oacc)[NB][VT]) {
  static_assert(WIN >= 1 && WIN <= 8 && WIN <= VT, "window of LDS reads (lgkm_wait counts up to 7)");
  __builtin_amdgcn_sched_barrier(0);
  u32x4 vv[WIN];
#pragma unroll
  for (int i = 0; i < WIN; ++i) vv[i] = lds_read16_at(vbase, 1024 * i);
#pragma unroll
  for (int i = 0; i < VT; ++i) {
    const int later = VT - 1 - i < WIN - 1 ? VT - 1 - i : WIN - 1;
    lgkm_wait(later, vv[i % WIN]);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) oacc[cb][i] = mfma16x16x32(as_bf16x8(vv[i % WIN]), pop[cb], oacc[cb][i]);
    if (i + WIN < VT) vv[i % WIN] = lds_read16_at(vbase, 1024 * (i + WIN));
  }
  __builtin_amdgcn_sched_barrier(0);
}

// exp(x) for x <= 0 (NaN stays NaN) as 2^hi exp(r): hi = x log2(e) rounded, 2^hi from v_exp_f32, and
// r = x - hi ln 2 by fmas with ln 2 in two parts, so that the rounding of hi does not enter (Cody and Waite's
// reduction), exp(r) = 1 + r for |r| < 2^-17. About 1 ulp at any x, where __expf's error grows with |x|;
// results below the smallest normal float are 0.
__device__ __forceinline__ float exp_nonpos(float x) {
  constexpr float kLog2e = 0x1.715476p+0f, kLn2Hi = 0x1.62e42ep-1f, kLn2Lo = 0x1.efa39ep-25f;
  const float hi = x * kLog2e;
  const float r = fmaf(-hi, kLn2Lo, fmaf(-hi, kLn2Hi, x));
  const float e = __builtin_amdgcn_exp2f(hi);
  return fmaf(e, fminf(r, 1.f), e);  // (x at the lowest bf16, a masked key: hi = -inf, r = inf, e = 0)
}

// The softmax's exp and a probability exp(x) / sum. Head dims 128 and 256: the hardware exp and the row's
// reciprocal (see the head of this file). Head dim 512 keeps the precision of prefill_bf16_kernel's expf and
// division, which its rows took before (4 x 1024 tokens: 100.1 us with the other head dims' two, 102.3 with
// these, about 118 with expf and a division).
template <int D>
__device__ __forceinline__ float pf_exp(float x) {
  if constexpr (D == 512) return exp_nonpos(x);
  return __expf(x);
}
template <int D>
__device__ __forceinline__ float pf_prob(float x, float sum, float rsum) {
  if constexpr (D == 512) {  // the quotient from the reciprocal with one residual correction (Markstein)
    const float e = exp_nonpos(x), q = e * rsum;
    return fmaf(fmaf(-q, sum, e), rsum, q);
  }
  return __expf(x) * rsum;
}

template <int D, int NB, int NW>
__global__ __launch_bounds__(NW * 64) void prefill_bf16_lds_kernel(G4PrefillArgs a) {
  using S_ = PfShape<D, NW>;
  constexpr int KS = D / 32;
  constexpr int SLOTS = S_::SLOTS;
  // one array for the DMA's slots, read with inline-assembly LDS reads only: the compiler adds no
  // waits of its own for the DMAs in flight (the key-mask bytes and the statistics are other arrays)
  __shared__ __attribute__((aligned(1024))) unsigned char ring[2 * SLOTS][S_::CHUNK];
  __shared__ int first_valid[NW];
  extern __shared__ float smem[];
  uint8_t* km_lds = reinterpret_cast<uint8_t*>(smem);  // key_mask[b, 0:S]

  const int R = a.group;
  const int ppc = 16 / R;              // positions per 16-row column block
  const int ppw = NB * ppc;            // positions per wave
  const int ppb = NW * ppw;            // positions per workgroup
  const int S = a.seq, H = a.kv_heads;
  const int nblk = (S + ppb - 1) / ppb;
  // One-dimensional grid. Causal rows (no window, or one that spans the sequence): a block's cost
  // grows with its position, so workgroup i takes block nblk - 1 - i / (B H) of pair i % (B H): the
  // latest blocks of every pair are dispatched before anyone's shorter ones (config 4's global layer:
  // 1.10 -> 0.99 ms against pair-major order). Windowed rows cost the same from block to block;
  // pair-major order (workgroup i: block nblk - 1 - i % nblk of pair i / nblk) keeps the workgroups in
  // flight on different key offsets, which measured faster there (sliding layer 0.36 against
  // 0.49 ms block-major). There, with a multiple of 8 pairs, consecutive blocks of a pair go to one
  // XCD (workgroups are dealt to the 8 XCDs round robin, i mod 8), so the overlapping key windows
  // of neighbouring blocks meet in one L2 (0.290-0.294 -> 0.278-0.283 ms); block-major order already
  // keeps a pair on one XCD.
  const int npairs = a.batch * H;
  const bool blk_major = a.window <= 0 || a.window >= S;
  int blk, pair;
  if (blk_major) {
    blk = nblk - 1 - (int)(blockIdx.x / (unsigned)npairs);
    pair = (int)(blockIdx.x % (unsigned)npairs);
  } else if (npairs % 8 == 0) {
    const int i = (int)blockIdx.x, j = i >> 3;
    blk = nblk - 1 - j % nblk;
    pair = (j / nblk) * 8 + (i & 7);
  } else {
    blk = nblk - 1 - (int)(blockIdx.x % (unsigned)nblk);
    pair = (int)(blockIdx.x / (unsigned)nblk);
  }
  const int b = pair / H, h = pair - b * H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int p0 = blk * ppb;                       // first position of the workgroup
  const int r = col - (col / R) * R;
  int my_pos[NB];                                 // this lane's query row (column col) of each block
  bool row_ok[NB];
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) {
    my_pos[cb] = p0 + w * ppw + cb * ppc + col / R;
    row_ok[cb] = my_pos[cb] < S;
  }
  const int64_t bh = (int64_t)b * H + h;
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(reinterpret_cast<const uint16_t*>(a.k) + bh * a.k_stride * D,
                                              (uint32_t)a.k_stride * D * 2u);
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(reinterpret_cast<const uint16_t*>(a.vt) + bh * D * a.k_stride,
                                              (uint32_t)a.k_stride * D * 2u);

  // q operands (registers) and the row's key-mask bytes (LDS)
  bf16x8 qop[NB][KS];
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) {
    const uint16_t* qrow =
        reinterpret_cast<const uint16_t*>(a.q) + ((((int64_t)b * S + my_pos[cb]) * H + h) * R + r) * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (row_ok[cb]) v = load16(qrow + 32 * s + 8 * grp);
      qop[cb][s] = as_bf16x8(v);
    }
  }
  // ... and the row's first valid key: the keys before it (a left-padded prompt's pads) score
  // nothing, so the passes start at its chunk
  const uint8_t* km = a.key_mask + (int64_t)b * a.key_mask_stride;
  int first = S;
  for (int i = tid; i < S; i += blockDim.x) {
    const uint8_t v = km[i];
    km_lds[i] = v;
    if (v && i < first) first = i;
  }
  // the q operands have landed here: waited for inside the loops, the compiler's count (it does not see
  // the loops' own waits) would drain the DMAs in flight at every chunk
#pragma unroll
  for (int cb = 0; cb < NB; ++cb)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4 v = __builtin_bit_cast(u32x4, qop[cb][s]);
      __asm__ volatile("" : "+v"(v));
      qop[cb][s] = as_bf16x8(v);
    }
#pragma unroll
  for (int msk = 32; msk >= 1; msk >>= 1) first = min(first, __shfl_xor(first, msk, 64));
  if (lane == 0) first_valid[w] = first;
  __syncthreads();  // key-mask bytes and first valid keys in LDS (no DMA in flight yet)
#pragma unroll
  for (int i = 0; i < NW; ++i) first = min(first, first_valid[i]);
  first = __builtin_amdgcn_readfirstlane(first);

  const int pos_last = min(p0 + ppb - 1, S - 1);
  const int kmin = max(first, a.window > 0 ? p0 - a.window + 1 : 0);
  // chunks c_begin .. c_end hold every key a row of this workgroup may see (none: c_begin > c_end)
  const int c_begin = kmin >> 5, c_end = kmin <= pos_last ? pos_last >> 5 : c_begin - 1;

  // This wave's share of a chunk's K / V^T operand tiles into LDS. Both layouts put chunk c at byte
  // 64 * D * c; a tile's place in it is uniform too and rides in soffset with it, so each operand
  // takes one lane offset (every chunk issued lies inside the cache rows: c <= (S - 1) / 32 and
  // S <= k_stride).
  const uint32_t k_lane = (uint32_t)(col * 64 + grp * 16);    // kt_index: lane col's 64-byte run, dims 8 grp ..
  const uint32_t v_lane = vt_operand_bytes(grp, col, D);
  auto issue_k = [&](int c, int slot) {
#pragma unroll
    for (int i = 0; i < S_::KT_W; ++i) {
      const int t = w * S_::KT_W + i, bb = t / KS, s = t - bb * KS;
      const uint32_t ofs = (uint32_t)c * (uint32_t)(64 * D) + (uint32_t)(2 * s + bb) * 1024u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)&ring[slot][1024 * t], 16,
                                               k_lane, ofs, 0, 0);
    }
  };
  auto issue_v = [&](int c, int slot) {
#pragma unroll
    for (int i = 0; i < S_::VT_W; ++i) {
      const int t = w * S_::VT_W + i;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)&ring[slot][1024 * t], 16,
                                               v_lane, (uint32_t)c * (uint32_t)(64 * D) + 256u * t, 0, 0);
    }
  };
  // Hides the chunk index from the compiler, which would otherwise keep one register per lane for every
  // bound of valid_bits and advance them from chunk to chunk (9 registers in pass 2: spills).
  auto hide_chunk = [](int& c) { __asm__ volatile("" : "+s"(c)); };
  // key-mask ballot of the chunk's 32 keys (lanes l and l + 32 both hold key 32 c + l % 32)
  auto chunk_ballot = [&](int c) -> uint64_t {
    const int key = (c << 5) + (lane & 31);
    return __ballot(key < S && km_lds[key < S ? key : 0] != 0);
  };
  // Wave-uniform: every row of this wave sees all 32 keys of chunk c (key mask, causal limit,
  // window, rows inside the sequence).
  const int wpos_min = p0 + w * ppw;
  const int wpos_max = wpos_min + (NB - 1) * ppc + 15 / R;
  auto chunk_full = [&](int c, uint64_t mb) -> bool {
    const int k0 = c << 5;
    return (uint32_t)mb == 0xffffffffu && k0 + 31 <= wpos_min && wpos_max < S &&
           (a.window <= 0 || k0 >= wpos_max - a.window + 1);
  };
  // this lane's key bits of the chunk (bit e <-> key 32 c + 8 grp + e) for block cb's row: the key
  // mask, causal, and the window
  auto valid_bits = [&](int c, uint64_t mb, int cb) -> uint32_t {
    uint32_t bits = (uint32_t)(mb >> (8 * grp)) & 0xffu;
    const int lo = (c << 5) + 8 * grp;
    const int hi_ok = my_pos[cb] - lo;  // keys lo + e valid for e <= hi_ok
    bits &= hi_ok >= 7 ? 0xffu : (hi_ok < 0 ? 0u : (0xffu >> (7 - hi_ok)));
    if (a.window > 0) {
      const int lo_ok = my_pos[cb] - a.window + 1 - lo;  // need e >= lo_ok
      bits &= lo_ok <= 0 ? 0xffu : (lo_ok > 7 ? 0u : (0xffu << lo_ok) & 0xffu);
    }
    return row_ok[cb] ? bits : 0u;
  };

  // ---- pass 1: row max and sum --------------------------------------------------------------------
  float m[NB], l[NB];
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) {
    m[cb] = kBf16Min;
    l[cb] = 0.f;
  }
  // one rescale per chunk: l <- l * exp(m - m') + sum exp(s - m') with m' = max(m, chunk max)
  // (masked keys score the fill value, whose exp vanishes against any real maximum)
  const uint32_t ring0 = lds_addr(&ring[0][0]) + 16u * (uint32_t)lane;  // this lane's piece of a tile
  auto stats = [&](int c, int slot) {
    floatx4 acc[NB][2];
    pf_qk<S_::KT, KS, NB, 8>(ring0 + (uint32_t)(slot * S_::CHUNK), qop, acc);  // pass 1 holds no value accumulators
    hide_chunk(c);
    const uint64_t mb = chunk_ballot(c);
    if (chunk_full(c, mb)) {
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        float sc[8], mx = kBf16Min;
        pf_round8(acc[cb], sc);
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, sc[e]);
        const float mn = fmaxf(m[cb], mx);
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += pf_exp<D>(sc[e] - mn);
        l[cb] = l[cb] * pf_exp<D>(m[cb] - mn) + sum;
        m[cb] = mn;
      }
      return;
    }
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const uint32_t bits = valid_bits(c, mb, cb);
      float sc[8], mx = kBf16Min;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        sc[e] = ((bits >> e) & 1u) ? round_bf16(acc[cb][e >> 2][e & 3]) : kBf16Min;
        mx = fmaxf(mx, sc[e]);
      }
      const float mn = fmaxf(m[cb], mx);
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += pf_exp<D>(sc[e] - mn);
      l[cb] = l[cb] * pf_exp<D>(m[cb] - mn) + sum;
      m[cb] = mn;
    }
  };
  // One pipeline step: wait for this wave's DMA of chunk c (chunks c+1, c+2 may stay in flight),
  // barrier (every wave's share of chunk c has landed, and every wave is done with chunk c-1, whose
  // slot the DMA of chunk c+3 reuses), queue chunk c+3, compute chunk c.
  auto wait_chunk = [&](int c, int c_last) {
    constexpr int n = S_::KT_W;
    const int ahead = min(c_last - c, 2);  // chunks queued after c
    if (ahead >= 2) wait_vmcnt<2 * n>();
    else if (ahead == 1) wait_vmcnt<n>();
    else wait_vmcnt<0>();
    wg_barrier();
  };
  // pass 1 rings through four slots whatever SLOTS is (the V^T slots are idle)
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if (c_begin + j <= c_end) issue_k(c_begin + j, j);
#pragma unroll 1
  for (int c = c_begin, i = 0; c <= c_end; ++c, ++i) {
    wait_chunk(c, c_end);
    if (c + 3 <= c_end) issue_k(c + 3, (i + 3) & 3);
    stats(c, i & 3);
  }
  bool row_masked[NB], mine_masked = false;
  float rl[NB];
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) {
#pragma unroll
    for (int msk = 16; msk <= 32; msk <<= 1) {
      const float m2 = __shfl_xor(m[cb], msk, 64);
      const float l2 = __shfl_xor(l[cb], msk, 64);
      const float mm = fmaxf(m[cb], m2);
      l[cb] = l[cb] * pf_exp<D>(m[cb] - mm) + l2 * pf_exp<D>(m2 - mm);
      m[cb] = mm;
    }
    // A row with no valid key is the reference's softmax over S equal fills: 1/S on every key.
    row_masked[cb] = row_ok[cb] && m[cb] == kBf16Min;
    mine_masked = mine_masked || row_masked[cb];
    rl[cb] = 1.0f / l[cb];
  }
  const bool any_masked = __syncthreads_or(mine_masked);  // (also: every wave is done with pass 1's LDS)

  // ---- pass 2: exact probabilities and O^T = V^T P^T -------------------------------------------------
  floatx4 oacc[NB][S_::VT];
#pragma unroll
  for (int cb = 0; cb < NB; ++cb)
#pragma unroll
    for (int i = 0; i < S_::VT; ++i) oacc[cb][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  // exact bf16 probabilities of chunk c from its score accumulators (the B operand of O^T += V^T P^T)
  auto probs = [&](int c, const floatx4 (&acc)[NB][2], bf16x8 (&pop)[NB]) {
    hide_chunk(c);
    const uint64_t mb = chunk_ballot(c);
    const bool full = chunk_full(c, mb);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      uint32_t pw[4];
      if (full) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t sw = pack_bf16x2(acc[cb][j >> 1][2 * (j & 1)], acc[cb][j >> 1][2 * (j & 1) + 1]);
          pw[j] = pack_bf16x2(pf_prob<D>(__uint_as_float(sw << 16) - m[cb], l[cb], rl[cb]),
                              pf_prob<D>(__uint_as_float(sw & 0xffff0000u) - m[cb], l[cb], rl[cb]));
        }
        // (keeps the packing here: sunk below the branches, eight floats per block stay live over them)
        __asm__ volatile("" : "+v"(pw[0]), "+v"(pw[1]), "+v"(pw[2]), "+v"(pw[3]));
      } else {
        const uint32_t bits = valid_bits(c, mb, cb);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t sw = pack_bf16x2(acc[cb][j >> 1][2 * (j & 1)], acc[cb][j >> 1][2 * (j & 1) + 1]);
          const float p0 = pf_prob<D>(__uint_as_float(sw << 16) - m[cb], l[cb], rl[cb]);
          const float p1 = pf_prob<D>(__uint_as_float(sw & 0xffff0000u) - m[cb], l[cb], rl[cb]);
          pw[j] = pack_bf16x2((bits >> (2 * j)) & 1u ? p0 : 0.f, (bits >> (2 * j + 1)) & 1u ? p1 : 0.f);
        }
      }
      pop[cb] = as_bf16x8(u32x4{pw[0], pw[1], pw[2], pw[3]});
    }
  };
  // One barrier per chunk step. After the barrier of chunk c every wave runs two phases:
  // M(c) = the values of chunk c-1 (its V^T tiles x the probabilities formed earlier) and the QK of
  // chunk c (MFMA work), and P(c) = the probabilities of chunk c (VALU work). Waves 0..NW/2-1 run
  // M(c) then P(c); waves NW/2.. run P(c-1) then M(c). Chunk j sits in slot (j - c_begin) % SLOTS of
  // both rings (K in slots 0 .. SLOTS-1, V^T behind them); K(c) and V(c-1) are read only in step c, and
  // the barrier of chunk c queues K(c+SLOTS-1) and V(c+SLOTS-2) into the slots of K(c-1) and V(c-2),
  // which step c-1 finished reading.
  const bool lead = w < NW / 2;
  // this wave's DMAs of K(c) and V(c-1) have landed: queued after them are, with four slots, V(c) and,
  // where they exist, K(c+1), K(c+2) and V(c+1); with two slots nothing
  auto wait_step = [&](int c, int c_last) {
    constexpr int nk = S_::KT_W, nv = S_::VT_W;
    if (SLOTS == 2) wait_vmcnt<0>();
    else if (c + 2 <= c_last) wait_vmcnt<2 * nk + 2 * nv>();
    else if (c + 1 <= c_last) wait_vmcnt<nk + 2 * nv>();
    else wait_vmcnt<nv>();
    wg_barrier();
  };
  if (c_begin <= c_end) {  // (uniform over the workgroup)
    floatx4 acc[NB][2];
    bf16x8 pop[NB];
    // prologue, in the steady state's order: K(b), then K(b+1), V(b), K(b+2), V(b+1) with four slots
    issue_k(c_begin, 0);
    if constexpr (SLOTS == 4) {
      if (c_begin + 1 <= c_end) issue_k(c_begin + 1, 1);
      issue_v(c_begin, SLOTS);
      if (c_begin + 2 <= c_end) issue_k(c_begin + 2, 2);
      if (c_begin + 1 <= c_end) issue_v(c_begin + 1, SLOTS + 1);
    }
#pragma unroll 1
    for (int c = c_begin, i = 0; c <= c_end; ++c, ++i) {
      wait_step(c, c_end);
      if (c + SLOTS - 1 <= c_end) issue_k(c + SLOTS - 1, (i + SLOTS - 1) & (SLOTS - 1));
      if (c + SLOTS - 2 <= c_end) issue_v(c + SLOTS - 2, SLOTS + ((i + SLOTS - 2) & (SLOTS - 1)));
      if (!lead && c > c_begin) probs(c - 1, acc, pop);
      __builtin_amdgcn_s_setprio(1);
      if (c > c_begin)
        pf_pv<S_::VT, NB, 4>(ring0 + (uint32_t)((SLOTS + ((i - 1) & (SLOTS - 1))) * S_::CHUNK), pop, oacc);
      pf_qk<S_::KT, KS, NB, 4>(ring0 + (uint32_t)((i & (SLOTS - 1)) * S_::CHUNK), qop, acc);
      __builtin_amdgcn_s_setprio(0);
      if (lead) probs(c, acc, pop);
    }
    // the last chunk's values: every wave's share of its V^T tiles has landed after this barrier
    wait_vmcnt<0>();
    wg_barrier();
    if (!lead) probs(c_end, acc, pop);
    pf_pv<S_::VT, NB, 4>(ring0 + (uint32_t)((SLOTS + ((c_end - c_begin) & (SLOTS - 1))) * S_::CHUNK), pop, oacc);
  }

  // the output row's address is computed here afresh (the lane is hidden from the compiler), not kept in
  // registers over both passes since the q loads
  int lane_o = lane;
  __asm__ volatile("" : "+v"(lane_o));
  auto out_row = [&](int cb) {
    const int c = lane_o & 15, pos = p0 + w * ppw + cb * ppc + c / R;
    return reinterpret_cast<uint16_t*>(a.out) + ((((int64_t)b * S + pos) * H + h) * R + c % R) * D;
  };
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) {
    if (row_ok[cb] && !row_masked[cb]) {
      uint16_t* orow = out_row(cb);
#pragma unroll
      for (int i = 0; i < S_::VT; ++i) {
        *reinterpret_cast<uint2*>(orow + 16 * i + 4 * grp) =
            make_uint2(pack_bf16x2(oacc[cb][i][0], oacc[cb][i][1]), pack_bf16x2(oacc[cb][i][2], oacc[cb][i][3]));
      }
    }
  }

  // ---- rows with no valid key: the average of all S values ------------------------------------------
  // The reference's softmax over S equal fills is 1/S on every key, the same output for every such row
  // of the pair. Wave w forms dims 16 VT_W w .. of it straight from memory, chunk after chunk into one
  // accumulator (the same MFMA, the uniform probability in every column: the bits that pass 2 over all S
  // keys gives), kUniform loads at a time; the average meets in LDS and each wave writes its masked rows.
  // S D values read once per workgroup with a masked row, instead of both passes over all S keys (11
  // prompts of 1999 left-padded tokens, window 512, with the pads' chunks skipped: 404 -> 186 us; a share
  // of the keys per wave, added at the end, takes the same time but rounds differently).
  if (!any_masked) return;
  float* usum = reinterpret_cast<float*>(&ring[0][0]);  // [D]
  const float p_uniform = round_bf16(1.0f / (float)S);
  constexpr int kUniform = 16, UC = kUniform / S_::VT_W;  // loads in flight, the chunks they cover
  const int u_last = (S - 1) >> 5;
  floatx4 uacc[S_::VT_W];
#pragma unroll
  for (int i = 0; i < S_::VT_W; ++i) uacc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int c = 0; c <= u_last; c += UC) {
    u32x4 v[UC][S_::VT_W];
#pragma unroll
    for (int u = 0; u < UC; ++u)
      if (c + u <= u_last) {
#pragma unroll
        for (int i = 0; i < S_::VT_W; ++i)
          v[u][i] = buffer_load16(rv, v_lane, (uint32_t)(c + u) * (uint32_t)(64 * D) + 256u * (w * S_::VT_W + i));
      }
    __builtin_amdgcn_sched_barrier(0);  // every load of the group requested before the first wait
#pragma unroll
    for (int u = 0; u < UC; ++u)
      if (c + u <= u_last) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = ((c + u) << 5) + 8 * grp + e < S ? p_uniform : 0.f;
        const bf16x8 pu = as_bf16x8(u32x4{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]),
                                          pack_bf16x2(p[6], p[7])});
#pragma unroll
        for (int i = 0; i < S_::VT_W; ++i) uacc[i] = mfma16x16x32(as_bf16x8(v[u][i]), pu, uacc[i]);
      }
  }
  __syncthreads();  // every wave is done with the ring
  if (col == 0) {
#pragma unroll
    for (int i = 0; i < S_::VT_W; ++i)
      *reinterpret_cast<floatx4*>(usum + 16 * (w * S_::VT_W + i) + 4 * grp) = uacc[i];
  }
  __syncthreads();
#pragma unroll
  for (int cb = 0; cb < NB; ++cb) {
    if (row_masked[cb]) {
      uint16_t* orow = out_row(cb);
#pragma unroll
      for (int i = 0; i < S_::VT; ++i) {
        const floatx4 o = *reinterpret_cast<const floatx4*>(usum + 16 * i + 4 * grp);
        *reinterpret_cast<uint2*>(orow + 16 * i + 4 * grp) =
            make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      }
    }
  }
}
