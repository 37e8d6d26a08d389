// Fused q/k/v preparation + KV-cache append (g4_kv_append).
//
// Replaces forward_rms_norm / forward_rotary_embedding on q and k, the unscaled v norm, and
// _update_layer_cache of gemma4_posttrain_jax/model.py:463-491, 368-390 with one launch per
// layer. append_kernel: one workgroup per token (b, s); append_tile_kernel (below): one per 8
// tokens of a row, for prefill-sized bf16 chunks. Each wave takes whole head vectors, with lane l
// owning elements [l*D/64, (l+1)*D/64) so a RoPE partner (d +- D/2) is lane l^32 in the same
// register. K rows go to the head-major key cache, V to the transposed value cache
// (cache_vt[b, h, d, slot]) that the MFMA attention kernels read as contiguous key runs.
#include <initializer_list>

#include "g4_common.h"
#include "g4_internal.h"
#include "g4_prep.h"

namespace g4 {
namespace {

enum VecKind { kQ = 0, kK = 1, kV = 2 };

// VEC: bf16 with D >= 128 and every row aligned to its lane's PER elements (checked on the host):
// each lane's elements move in one access per array instead of one per element.
template <bool BF16, int D, bool VEC = false>
__global__ __launch_bounds__(1024) void append_kernel(G4AppendArgs a) {
  using E = Elem<BF16>;
  using T = typename E::T;
  // D >= 64: lane l owns d in [l*D/64, (l+1)*D/64) and its RoPE partner is lane l^32;
  // D < 64: lane l < D owns d = l and its partner is lane l^(D/2).
  constexpr int PER = D >= 64 ? D / 64 : 1;
  constexpr int PARTNER = D >= 64 ? 32 : D / 2;
  const int lane = threadIdx.x & 63;
  const bool lane_on = D >= 64 || lane < D;
  const int wave = threadIdx.x >> 6;
  const int nwaves = blockDim.x >> 6;
  const int S = a.seq;
  const int token = blockIdx.x;
  const int b = token / S;
  const int s = token - b * S;
  const int H = a.kv_heads;
  const int R = a.group;
  const int nq = a.q ? H * R : 0;
  const int nvec = nq + (a.k ? 2 * H : 0);

  // Destination slot (model.py:373-390): linear writes at start + s with XLA's
  // dynamic_update_slice start clamp; a ring keeps only the chunk's last Wc tokens.
  const int64_t start = a.write_pos ? (int64_t)a.write_pos[b] : (int64_t)a.write_pos_scalar;
  const int64_t cap = a.capacity;
  int64_t slot;
  bool to_cache;
  if (a.kind == G4_CACHE_RING) {
    const int64_t keep = S < cap ? S : cap;
    to_cache = s >= S - keep;
    slot = floor_mod(start + s, cap);
  } else {
    int64_t st = start < 0 ? 0 : start;
    if (st > cap - S) st = cap - S;
    slot = st + s;
    to_cache = true;
  }

  const int64_t in_base = (int64_t)token * a.in_row_stride;
  const int64_t rope_base = (int64_t)token * D;

  for (int vec = wave; vec < nvec; vec += nwaves) {
    int kind, head, r = 0;
    const T* src;
    if (vec < nq) {
      kind = kQ;
      head = vec / R;
      r = vec - head * R;
      src = reinterpret_cast<const T*>(a.q) + in_base + (int64_t)vec * D;
    } else if (vec < nq + H) {
      kind = kK;
      head = vec - nq;
      src = reinterpret_cast<const T*>(a.k) + in_base + (int64_t)head * D;
    } else {
      kind = kV;
      head = vec - nq - H;
      src = reinterpret_cast<const T*>(a.v) + in_base + (int64_t)head * D;
    }

    const bool norm = (kind == kQ && (a.flags & G4_APPEND_NORM_Q)) || (kind == kK && (a.flags & G4_APPEND_NORM_K)) ||
                      (kind == kV && (a.flags & G4_APPEND_NORM_V));
    const bool rope = (kind == kQ && (a.flags & G4_APPEND_ROPE_Q)) || (kind == kK && (a.flags & G4_APPEND_ROPE_K));
    const T* w = norm ? (kind == kQ ? reinterpret_cast<const T*>(a.q_norm_weight)
                                    : (kind == kK ? reinterpret_cast<const T*>(a.k_norm_weight) : nullptr))
                      : nullptr;
    float x[PER];
    prep_head<BF16, D, VEC>(src, w, norm, rope, a.rope_cos + rope_base, a.rope_sin + rope_base, a.eps, lane, x);

    const int64_t bh = (int64_t)b * H + head;
    if (!lane_on) continue;
    // this lane's PER consecutive elements at p (they never cross a 32-element run of the key layout)
    auto store_run = [&](T* p) {
      if constexpr (VEC) {
        st_bf16<PER>(reinterpret_cast<uint16_t*>(p), x);
      } else {
#pragma unroll
        for (int e = 0; e < PER; ++e) E::store(p, e, x[e]);
      }
    };
    auto store_row = [&](T* dst) { store_run(dst + lane * PER); };
    if (kind == kQ) {
      store_row(reinterpret_cast<T*>(a.q_out) + ((((int64_t)token) * H + head) * R + r) * D);
    } else if (kind == kK) {
      if (to_cache) store_run(reinterpret_cast<T*>(a.cache_k) + bh * a.slot_stride * D + kt_index(slot, lane * PER, D));
      if (a.k_out) store_run(reinterpret_cast<T*>(a.k_out) + bh * a.chunk_stride * D + kt_index(s, lane * PER, D));
    } else {
      if (to_cache) {
        T* dst = reinterpret_cast<T*>(a.cache_vt) + bh * D * a.slot_stride;
#pragma unroll
        for (int e = 0; e < PER; ++e) E::store(dst, vt_index(slot, lane * PER + e, D), x[e]);
      }
      if (a.vt_out) {
        T* dst = reinterpret_cast<T*>(a.vt_out) + bh * D * a.chunk_stride;
#pragma unroll
        for (int e = 0; e < PER; ++e) E::store(dst, vt_index(s, lane * PER + e, D), x[e]);
      }
    }
  }
}

// Prefill-sized appends (bf16, the vectorized rows, S >= 8): one 8-wave workgroup per 8 consecutive
// tokens of a row, one token per wave. A token's cos / sin row and the norm weights are read and
// rounded once for its H (R + 2) head vectors, whose loads are issued kTileVecs at a time (8 waves
// per SIMD; D = 512 runs at 4). The value cache groups 8 slots per 16-byte piece
// (cache_vt[b, h, slot / 8, d, slot % 8]), so one token's V row is D two-byte pieces spread over
// D / 8 cache lines; when the 8 tokens land in one aligned 8-slot group (a cache start and ring size
// that are multiples of 8) their V rows are staged in LDS and stored as whole 16-byte pieces, 16 D
// contiguous bytes per head, and the chunk copy (vt_out) likewise. Other workgroups store V element
// by element as append_kernel does. Same arithmetic and destinations as append_kernel.
// Bound by HBM: 256 x 256 tokens of 2 x (4 + 2) heads of 256 with the chunk copy move 1.07 GB in 202 - 209
// us, 5.2 TB/s (a copy of 4 GiB reaches 4.8); with a wave per head vector, which read the cos / sin row and
// formed the slot anew for each of the 12 vectors of a token and rotated through LDS, 354 us.
constexpr int kTileTok = 8;
constexpr int kTileThreads = 64 * kTileTok;
constexpr int kTileVtBytes = 32 * 1024;  // LDS for the staged V rows: kv_heads * D * 16 bytes at most
constexpr int kTileVecs = 4;             // head vectors of a token in flight per wave

__device__ __forceinline__ void swap_halves(float& x, float& y) {  // x's lanes 32 .. 63 <-> y's lanes 0 .. 31
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}

// The lane's PER elements as packed bf16 pairs, one access (PER = 2, 4 or 8).
template <int W>
__device__ __forceinline__ void ld_words(const uint16_t* p, uint32_t (&w)[W]) {
  if constexpr (W == 1) {
    w[0] = *reinterpret_cast<const uint32_t*>(p);
  } else if constexpr (W == 2) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    w[0] = v.x, w[1] = v.y;
  } else {
    const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = v[i];
  }
}
template <int W>
__device__ __forceinline__ void st_words(uint16_t* p, const uint32_t (&w)[W]) {
  if constexpr (W == 1) {
    *reinterpret_cast<uint32_t*>(p) = w[0];
  } else if constexpr (W == 2) {
    *reinterpret_cast<uint2*>(p) = make_uint2(w[0], w[1]);
  } else {
    *reinterpret_cast<u32x4*>(p) = u32x4{w[0], w[1], w[2], w[3]};
  }
}

// One token's RoPE row, rounded to bf16. Element pair (e, e + PER / 2) of a lane after swap_halves:
// lanes 0 .. 31 hold dims d and d + D / 2 of element e, lanes 32 .. 63 those of element e + PER / 2,
// so both members of a rotated pair sit in one lane and no partner is fetched.
template <int PER>
struct TileRope {
  float c[PER], s[PER];
  __device__ __forceinline__ void load(const float* rcos, const float* rsin, int lane) {
    ld_f32<PER>(rcos + lane * PER, c);
    ld_f32<PER>(rsin + lane * PER, s);
  }
  __device__ __forceinline__ void arrange() {
#pragma unroll
    for (int e = 0; e < PER / 2; ++e) {
      swap_halves(c[e], c[e + PER / 2]);
      swap_halves(s[e], s[e + PER / 2]);
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) c[e] = round_bf16(c[e]), s[e] = round_bf16(s[e]);
  }
};

// prep_math on packed pairs: the same operations in the same order, so the same bits.
template <int D, bool HAS_W>
__device__ __forceinline__ void tile_prep(uint32_t (&w)[D / 128], bool norm, const float (&wv)[D / 64], bool rope,
                                          const TileRope<D / 64>& tr, float eps) {
#pragma clang fp contract(off)
  constexpr int PER = D / 64, W = D / 128;
  float x[PER];
#pragma unroll
  for (int i = 0; i < W; ++i) {
    x[2 * i] = __uint_as_float(w[i] << 16);
    x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
  if (norm) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < PER; ++e) ss += x[e] * x[e];
    ss = wave_sum(ss);
    const float inv = 1.0f / __fsqrt_rn(ss / (float)D + eps);
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      x[e] = x[e] * inv;
      if (HAS_W) x[e] = x[e] * wv[e];
    }
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
  }
  if (rope) {
#pragma unroll
    for (int i = 0; i < W; ++i) {
      x[2 * i] = __uint_as_float(w[i] << 16);
      x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
#pragma unroll
    for (int e = 0; e < PER / 2; ++e) {
      float lo = x[e], hi = x[e + PER / 2];
      swap_halves(lo, hi);
      const float lc = lo * tr.c[e], hs = -hi * tr.s[e];
      const float hc = hi * tr.c[e + PER / 2], ls = lo * tr.s[e + PER / 2];
      lo = lc + hs;
      hi = hc + ls;
      swap_halves(lo, hi);
      x[e] = lo;
      x[e + PER / 2] = hi;
    }
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
  }
}

template <int D>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(D >= 512 ? 4 : 8))) void
append_tile_kernel(G4AppendArgs a) {
  using T = uint16_t;
  constexpr int PER = D / 64, W = D / 128;
  extern __shared__ __attribute__((aligned(16))) uint16_t v_lds[];  // [H][8 tokens][D]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int S = a.seq, H = a.kv_heads;
  const int ntile = (S + kTileTok - 1) / kTileTok;
  const int b = (int)blockIdx.x / ntile;
  const int s0 = ((int)blockIdx.x - b * ntile) * kTileTok;
  const int n_tok = S - s0 < kTileTok ? S - s0 : kTileTok;

  // destination slot of token s0 + t (model.py:373-390), as in append_kernel
  const int64_t start = a.write_pos ? (int64_t)a.write_pos[b] : (int64_t)a.write_pos_scalar;
  const int cap = a.capacity;
  const bool ring = a.kind == G4_CACHE_RING;
  const int drop = ring && S > cap ? S - cap : 0;  // a ring keeps the chunk's last `cap` tokens
  int64_t first = start < 0 ? 0 : start;
  if (ring) {
    first = floor_mod(start + s0, (int64_t)cap);
  } else {
    if (first > cap - S) first = cap - S;
    first += s0;
  }
  auto slot_of = [&](int t) -> int64_t {
    return ring ? (int64_t)(((uint32_t)first + (uint32_t)t) % (uint32_t)cap) : first + t;
  };
  // whole 8-slot groups: 8 tokens, consecutive slots from a multiple of 8, all or none of them kept
  const bool grouped = a.k && n_tok == kTileTok && first % 8 == 0 && slot_of(kTileTok - 1) == first + kTileTok - 1 &&
                       (s0 >= drop) == (s0 + kTileTok - 1 >= drop);

  if (wave < n_tok) {
    const int t = wave, s = s0 + t;
    const int64_t token = (int64_t)b * S + s;
    const int64_t in_off = token * a.in_row_stride + lane * PER;
    const bool rope_q = a.q && (a.flags & G4_APPEND_ROPE_Q), rope_k = a.k && (a.flags & G4_APPEND_ROPE_K);
    TileRope<PER> tr;
    if (rope_q || rope_k) tr.load(a.rope_cos + token * D, a.rope_sin + token * D, lane);
    uint32_t w[kTileVecs][W];
    float wv[PER];
    bool arranged = false;
    if (a.q) {
      const bool norm = a.flags & G4_APPEND_NORM_Q;
      const int nq = H * a.group;
      const T* src = reinterpret_cast<const T*>(a.q) + in_off;
      T* dst = reinterpret_cast<T*>(a.q_out) + token * nq * D + lane * PER;
      if (norm) ld_bf16<PER>(reinterpret_cast<const T*>(a.q_norm_weight) + lane * PER, wv);
      for (int v0 = 0; v0 < nq; v0 += kTileVecs) {
#pragma unroll
        for (int i = 0; i < kTileVecs; ++i)
          if (v0 + i < nq) ld_words<W>(src + (v0 + i) * D, w[i]);
        if (!arranged && (rope_q || rope_k)) tr.arrange();
        arranged = true;
#pragma unroll
        for (int i = 0; i < kTileVecs; ++i) {
          if (v0 + i < nq) {
            tile_prep<D, true>(w[i], norm, wv, rope_q, tr, a.eps);
            st_words<W>(dst + (v0 + i) * D, w[i]);
          }
        }
      }
    }
    if (a.k) {
      const bool norm_k = a.flags & G4_APPEND_NORM_K, norm_v = a.flags & G4_APPEND_NORM_V;
      const T* ksrc = reinterpret_cast<const T*>(a.k) + in_off;
      const T* vsrc = reinterpret_cast<const T*>(a.v) + in_off;
      const bool to_cache = s >= drop;
      const int64_t slot = slot_of(t);
      const int64_t k_lane = kt_index(0, lane * PER, D);
      if (norm_k) ld_bf16<PER>(reinterpret_cast<const T*>(a.k_norm_weight) + lane * PER, wv);
      for (int h0 = 0; h0 < H; h0 += kTileVecs / 2) {
#pragma unroll
        for (int i = 0; i < kTileVecs / 2; ++i) {
          if (h0 + i < H) {
            ld_words<W>(ksrc + (h0 + i) * D, w[2 * i]);
            ld_words<W>(vsrc + (h0 + i) * D, w[2 * i + 1]);
          }
        }
        if (!arranged && rope_k) tr.arrange();
        arranged = true;
#pragma unroll
        for (int i = 0; i < kTileVecs / 2; ++i) {
          const int head = h0 + i;
          if (head >= H) break;
          const int64_t bh = (int64_t)b * H + head;
          tile_prep<D, true>(w[2 * i], norm_k, wv, rope_k, tr, a.eps);
          if (to_cache)
            st_words<W>(reinterpret_cast<T*>(a.cache_k) + bh * a.slot_stride * D + kt_index(slot, 0, D) + k_lane, w[2 * i]);
          if (a.k_out)
            st_words<W>(reinterpret_cast<T*>(a.k_out) + bh * a.chunk_stride * D + kt_index(s, 0, D) + k_lane, w[2 * i]);
          uint32_t(&vw)[W] = w[2 * i + 1];
          tile_prep<D, false>(vw, norm_v, wv, false, tr, a.eps);
          if (grouped) {
            st_words<W>(v_lds + (head * kTileTok + t) * D + lane * PER, vw);
          } else {
            auto scatter = [&](T* dst, int64_t to) {
#pragma unroll
              for (int e = 0; e < PER; ++e) dst[vt_index(to, lane * PER + e, D)] = (uint16_t)(vw[e / 2] >> (16 * (e & 1)));
            };
            if (to_cache) scatter(reinterpret_cast<T*>(a.cache_vt) + bh * D * a.slot_stride, slot);
            if (a.vt_out) scatter(reinterpret_cast<T*>(a.vt_out) + bh * D * a.chunk_stride, s);
          }
        }
      }
    }
  }
  if (!grouped) return;  // uniform over the workgroup
  __syncthreads();
  // piece (head, d): the 8 tokens' values of dim d, 16 bytes at slot group first / 8
  for (int i = threadIdx.x; i < H * D; i += kTileThreads) {
    const int hh = i / D, d = i - hh * D;
    const uint16_t* col = v_lds + hh * kTileTok * D + d;
    u32x4 piece;
#pragma unroll
    for (int j = 0; j < 4; ++j) piece[j] = (uint32_t)col[2 * j * D] | ((uint32_t)col[(2 * j + 1) * D] << 16);
    const int64_t bh = (int64_t)b * H + hh;
    if (s0 >= drop)
      *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(a.cache_vt) + bh * D * a.slot_stride + vt_index(first, d, D)) = piece;
    if (a.vt_out)
      *reinterpret_cast<u32x4*>(reinterpret_cast<T*>(a.vt_out) + bh * D * a.chunk_stride + vt_index(s0, d, D)) = piece;
  }
}

// The vectorized path needs every row start aligned to one lane's D/64 bf16 elements (and the
// f32 RoPE rows to 16 bytes).
bool vec_rows_ok(const G4AppendArgs& a) {
  const uintptr_t al = (uintptr_t)(a.head_dim / 64) * 2;
  for (const void* p : std::initializer_list<const void*>{a.q, a.k, a.v, a.q_out, a.cache_k, a.k_out,
                                                        a.q_norm_weight, a.k_norm_weight})
    if (reinterpret_cast<uintptr_t>(p) % al) return false;
  for (const void* p : std::initializer_list<const void*>{a.rope_cos, a.rope_sin})
    if (reinterpret_cast<uintptr_t>(p) % 16) return false;
  return (a.in_row_stride * 2) % (int64_t)al == 0;
}

template <bool BF16>
int launch_append(const G4AppendArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)((int64_t)a.batch * a.seq));
  // one wave per head vector (q heads, k heads, v heads) up to 16 waves; more vectors loop
  const int nvec = (a.q ? a.kv_heads * a.group : 0) + (a.k ? 2 * a.kv_heads : 0);
  const dim3 block((unsigned)(64 * (nvec < 1 ? 1 : (nvec > 16 ? 16 : nvec))));
  if (BF16 && a.head_dim >= 128 && vec_rows_ok(a)) {
    const size_t vt_bytes = a.k ? (size_t)a.kv_heads * a.head_dim * 16 : 0;
    // prefill-sized: 8 tokens per workgroup (its 16-byte V stores need 16-byte aligned value arrays)
    const bool vt_aligned = reinterpret_cast<uintptr_t>(a.cache_vt) % 16 == 0 && reinterpret_cast<uintptr_t>(a.vt_out) % 16 == 0;
    if (a.seq >= kTileTok && vt_bytes <= (size_t)kTileVtBytes && vt_aligned) {
      const dim3 tgrid((unsigned)((int64_t)a.batch * ((a.seq + kTileTok - 1) / kTileTok)));
      switch (a.head_dim) {
        case 128: hipLaunchKernelGGL((append_tile_kernel<128>), tgrid, dim3(kTileThreads), vt_bytes, st, a); break;
        case 256: hipLaunchKernelGGL((append_tile_kernel<256>), tgrid, dim3(kTileThreads), vt_bytes, st, a); break;
        case 512: hipLaunchKernelGGL((append_tile_kernel<512>), tgrid, dim3(kTileThreads), vt_bytes, st, a); break;
        default: return fail(G4_ERR_UNSUPPORTED, "g4_kv_append: head_dim %d", a.head_dim);
      }
      return check_launch("g4_kv_append");
    }
    switch (a.head_dim) {
      case 128: hipLaunchKernelGGL((append_kernel<true, 128, true>), grid, block, 0, st, a); break;
      case 256: hipLaunchKernelGGL((append_kernel<true, 256, true>), grid, block, 0, st, a); break;
      case 512: hipLaunchKernelGGL((append_kernel<true, 512, true>), grid, block, 0, st, a); break;
      default: return fail(G4_ERR_UNSUPPORTED, "g4_kv_append: head_dim %d", a.head_dim);
    }
    return check_launch("g4_kv_append");
  }
  switch (a.head_dim) {
    case 8: hipLaunchKernelGGL((append_kernel<BF16, 8>), grid, block, 0, st, a); break;
    case 16: hipLaunchKernelGGL((append_kernel<BF16, 16>), grid, block, 0, st, a); break;
    case 32: hipLaunchKernelGGL((append_kernel<BF16, 32>), grid, block, 0, st, a); break;
    case 64: hipLaunchKernelGGL((append_kernel<BF16, 64>), grid, block, 0, st, a); break;
    case 128: hipLaunchKernelGGL((append_kernel<BF16, 128>), grid, block, 0, st, a); break;
    case 256: hipLaunchKernelGGL((append_kernel<BF16, 256>), grid, block, 0, st, a); break;
    case 512: hipLaunchKernelGGL((append_kernel<BF16, 512>), grid, block, 0, st, a); break;
    default: return fail(G4_ERR_UNSUPPORTED, "g4_kv_append: head_dim %d", a.head_dim);
  }
  return check_launch("g4_kv_append");
}

}  // namespace
}  // namespace g4

extern "C" int g4_kv_append(const G4AppendArgs* args, void* stream) {
  using g4::fail;
  if (!args) return fail(G4_ERR_INVALID, "g4_kv_append: args is NULL");
  const G4AppendArgs& a = *args;
  if (a.dtype != G4_DTYPE_F32 && a.dtype != G4_DTYPE_BF16) return fail(G4_ERR_INVALID, "g4_kv_append: dtype %d", a.dtype);
  if (a.kind != G4_CACHE_LINEAR && a.kind != G4_CACHE_RING) return fail(G4_ERR_INVALID, "g4_kv_append: kind %d", a.kind);
  if (a.batch <= 0 || a.seq <= 0 || a.kv_heads <= 0)
    return fail(G4_ERR_INVALID, "g4_kv_append: batch/seq/kv_heads must be positive (%d, %d, %d)", a.batch, a.seq,
                a.kv_heads);
  if (!g4::supported_head_dim(a.head_dim)) return fail(G4_ERR_UNSUPPORTED, "g4_kv_append: head_dim %d", a.head_dim);
  if (a.capacity <= 0 || a.slot_stride < a.capacity || a.slot_stride % 64)
    return fail(G4_ERR_INVALID, "g4_kv_append: capacity %d / slot_stride %d (need stride >= capacity, multiple of 64)",
                a.capacity, a.slot_stride);
  if (a.kind == G4_CACHE_LINEAR && a.seq > a.capacity)
    return fail(G4_ERR_INVALID, "g4_kv_append: %d tokens do not fit a linear cache of %d slots", a.seq, a.capacity);
  if (a.k || a.v) {
    if (!a.k || !a.v || !a.cache_k || !a.cache_vt)
      return fail(G4_ERR_INVALID, "g4_kv_append: k/v/cache pointer is NULL");
  } else if (!a.q) {
    return fail(G4_ERR_INVALID, "g4_kv_append: nothing to do (q, k and v are NULL)");
  }
  if (a.in_row_stride < (int64_t)a.kv_heads * a.head_dim)
    return fail(G4_ERR_INVALID, "g4_kv_append: in_row_stride %lld too small", (long long)a.in_row_stride);
  if (a.q) {
    if (a.group <= 0 || !a.q_out) return fail(G4_ERR_INVALID, "g4_kv_append: q needs group > 0 and q_out");
  }
  if ((a.flags & (G4_APPEND_ROPE_K | G4_APPEND_ROPE_Q)) && (!a.rope_cos || !a.rope_sin))
    return fail(G4_ERR_INVALID, "g4_kv_append: RoPE flags need rope_cos/rope_sin");
  if ((a.flags & G4_APPEND_NORM_K) && !a.k_norm_weight) return fail(G4_ERR_INVALID, "g4_kv_append: NORM_K needs k_norm_weight");
  if ((a.flags & G4_APPEND_NORM_Q) && a.q && !a.q_norm_weight)
    return fail(G4_ERR_INVALID, "g4_kv_append: NORM_Q needs q_norm_weight");
  if ((a.k_out || a.vt_out) && (a.chunk_stride < a.seq || a.chunk_stride % 64))
    return fail(G4_ERR_INVALID, "g4_kv_append: chunk_stride %d (need >= seq, multiple of 64)", a.chunk_stride);
  if ((int64_t)a.batch * a.seq > 0x7fffffffLL) return fail(G4_ERR_UNSUPPORTED, "g4_kv_append: too many tokens");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return a.dtype == G4_DTYPE_BF16 ? g4::launch_append<true>(a, st) : g4::launch_append<false>(a, st);
}
