// Slot-mapped KV append for gfx950.
//
// Semantics follow the reference kernels reshape_and_cache
// (paged_attention/metal/cache/reshape_and_cache.metal:35-69) and
// reshape_and_cache_flash (:115-136): token i is written to slot
// slot_mapping[i] (block = slot / block_size, offset = slot % block_size);
// negative slots are skipped.  Element conversion is static_cast semantics
// (:9-12): identical types copy bits, float -> f16/bf16 rounds to nearest even.
//
// Two layouts:
//  * paged 5-D: K [nb, H, D/x, bs, x], V [nb, H, D, bs].  One workgroup per
//    window of bs batch tokens and head: tokens that together fill a whole
//    block in order (a prefill) leave as whole lines; other tokens leave one
//    (token, head) per wavefront, K as D/x 16-byte chunks at a stride of bs*16
//    bytes, V as D single elements at a stride of bs elements (the layout
//    makes V token-minor, so one token's stores cannot be wider than one
//    element).
//  * FP8 caches (E4M3 codes of x / scale, either layout): see below.
//  * token-major (MHATokenPool / flash): K and V [num_slots, H, D].  A token's
//    K row and V row are each one contiguous H*D run in both source and
//    destination, so every lane moves 16-byte vectors and every wavefront
//    covers 1 KiB of one row.  Rows of at least 64 vectors go one token per
//    wavefront with nontemporal stores; shorter rows one token per
//    workgroup.
#include <algorithm>

#include "pkv_fp8.h"
#include "pkv_launch.h"

namespace pkv {

// ---- vector helpers ----------------------------------------------------------
// Load VE elements of type S starting at src (aligned when ALIGNED) and
// convert them to VE elements of type D written to dst.
template <class S, class D, int VE, bool ALIGNED>
__device__ __forceinline__ void convert_run(const typename Elem<S>::storage* __restrict__ src,
                                            typename Elem<D>::storage* __restrict__ dst) {
  if constexpr (ALIGNED && Elem<S>::kBytes == Elem<D>::kBytes && Elem<S>::kBytes * VE == 16 &&
                std::is_same<S, D>::value) {
    *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
  } else if constexpr (ALIGNED && Elem<D>::kBytes == 2 && Elem<S>::kBytes == 4 && VE == 8) {
    const float4 a = reinterpret_cast<const float4*>(src)[0];
    const float4 b = reinterpret_cast<const float4*>(src)[1];
    uint4 o;
    o.x = pack2(from_f32<D>(a.x), from_f32<D>(a.y));
    o.y = pack2(from_f32<D>(a.z), from_f32<D>(a.w));
    o.z = pack2(from_f32<D>(b.x), from_f32<D>(b.y));
    o.w = pack2(from_f32<D>(b.z), from_f32<D>(b.w));
    *reinterpret_cast<uint4*>(dst) = o;
  } else {
#pragma unroll
    for (int i = 0; i < VE; ++i) dst[i] = convert_elem<S, D>(src[i]);
  }
}

// One 16-byte cache vector (16 / sizeof(CT) elements) read from an aligned
// source run and converted.
template <class S, class D>
__device__ __forceinline__ uint4 load_vec16(const typename Elem<S>::storage* __restrict__ src) {
  constexpr int VE = 16 / Elem<D>::kBytes;
  if constexpr (std::is_same<S, D>::value) {
    return *reinterpret_cast<const uint4*>(src);
  } else {
    typename Elem<D>::storage t[VE];
    convert_run<S, D, VE, true>(src, t);
    return *reinterpret_cast<const uint4*>(t);
  }
}

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

// ---- FP8 caches: E4M3 codes of x / scale (pkv_fp8.h) -------------------------------
// Eight source elements -> eight codes.
template <class KT>
__device__ __forceinline__ uint2 encode8(const typename Elem<KT>::storage* __restrict__ src, const Fp8Scale& s) {
  float v[8];
  if constexpr (std::is_same<KT, F32>::value) {
    const float4 a = reinterpret_cast<const float4*>(src)[0], b = reinterpret_cast<const float4*>(src)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
    const uint4 w = *reinterpret_cast<const uint4*>(src);
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = to_f32<KT>((uint16_t)(u[i] & 0xffffu));
      v[2 * i + 1] = to_f32<KT>((uint16_t)(u[i] >> 16));
    }
  }
  return make_uint2(fp8_encode4_scaled(v, s), fp8_encode4_scaled(v + 4, s));
}

// ---- paged 5-D layout, windows of one block's tokens ------------------------------
// One workgroup (SPLIT: several that share its tasks) per (window of BS
// consecutive batch tokens, group of `hg` heads), for block sizes 8, 16 and
// 32.  When BS consecutive batch tokens write slots blk*BS .. blk*BS + BS-1 in
// order (a prefill writing whole blocks, a "run"), the (block, head) regions
// of K ([D/x][BS][x]) and V ([D][BS]) are each one contiguous run of D*BS
// elements that these tokens fill completely.  The workgroup of the window in which a run starts (at
// most one run starts in BS consecutive tokens, as runs do not overlap)
// writes both regions whole; the other tokens of the window, which lie
// between the end of the previous window's run and the start of its own, are
// written token by token.
//
// Run tasks, one per thread, eight elements of each region, index u:
//   K: 16-bit caches: the 16-byte unit u = c*BS + t (dimensions 8c .. 8c+7 of
//      token t), one 16-byte load of 8 source elements; FP8 caches: the
//      8-byte half u of the units of 16 codes.
//   V: u = (dim pair) * BS/4 + (token quad): two dimensions of four tokens in
//      four loads; v_perm regroups them by dimension and one exchange with
//      the neighbouring lane (the pair's other quad) leaves each lane eight
//      tokens of one dimension, so 64 lanes store 1 KiB (FP8: 512 bytes) of
//      the region in one piece.
// Bound: HBM traffic.  Measured (ragged prompts of 97 .. 927 tokens, 8 heads
// x 128, blocks of 16; passes back to back): 16,384 bf16 tokens 51.2 -> 22.4
// us (134 MB, 6.0 TB/s), 8192 tokens into FP8 36.4 -> 13.9 us (50 MB; kernel
// 38.2 -> 15.1 us under the profiler), against a wavefront per (token, head)
// that gathered a 1/BS slice of each region with 2-byte loads: 131,072
// wavefronts, and eight load instructions where one does.  The run stores are nontemporal: whole lines that
// nothing in the launch reads back (a decode right after the append then
// finds its own lines in the caches: radix-shared workload 84.0 -> 77.3 us
// per launch).
//
// Per-token stores: a token's V elements lie BS elements apart, each store a
// partial write of its line.  They keep the default policy, as the L2 combines
// the tokens of a block into lines (nontemporal, they made the radix
// workload's append 4.5x slower).  K chunks of a large call are stored
// nontemporally (p.stream_k): a token's 16-byte chunks sit BS*16 bytes apart,
// one per line, and a call writing more K than one XCD's L2 holds (4 MiB) has
// its lines evicted before a later token fills their neighbours (4096 random
// slots, 8 MiB of K: 76.4 -> 65.0 us).

// Batch positions of a window that each wavefront needs: the run that started
// in the previous window (prev) and the one that starts in this window (run),
// -1 if there is none; every lane gets the same values.  slot: the slot of
// token (window - 1) * BS + lane, -1 outside the batch.
template <int BS>
__device__ __forceinline__ void rac_window_runs(const RacParams& p, int64_t window, int lane, int64_t& prev,
                                                int64_t& run, int& slot) {
  const int64_t base = (window - 1) * BS;  // the lanes look at [base, base + 3 BS)
  // Bit i: token base + i's slot is followed by its successor's.
  auto links = [&](int64_t pos, int& slot) -> uint64_t {
    slot = pos >= 0 && pos < p.num_tokens ? p.slot_mapping[pos] : -1;
    const int next = pos >= 0 && pos + 1 < p.num_tokens ? p.slot_mapping[pos + 1] : -1;
    return __ballot(slot >= 0 && slot < INT32_MAX && next == slot + 1);
  };
  int unused;
  const uint64_t lo = links(base + lane, slot);
  uint64_t follow = lo >> lane;
  if constexpr (3 * BS > 64) {
    const uint64_t hi = links(base + 64 + lane, unused);
    if (lane > 0) follow |= hi << (64 - lane);
  }
  constexpr uint64_t kAll = ((uint64_t)1 << (BS - 1)) - 1;
  const bool starts = lane < 2 * BS && slot >= 0 && slot % BS == 0 && (int64_t)slot + BS <= p.num_slots &&
                      (follow & kAll) == kAll;
  const uint64_t m = __ballot(starts);
  constexpr uint64_t kWin = ((uint64_t)1 << BS) - 1;
  const uint64_t mp = m & kWin, mr = (m >> BS) & kWin;
  prev = mp ? base + __builtin_ctzll(mp) : -1;
  run = mr ? base + BS + __builtin_ctzll(mr) : -1;
}

// Eight cache elements of a source run: one 16-byte vector (16-bit caches)
// or 8 code bytes (FP8).
template <class CT> struct Vec8 { using type = uint4; };
template <> struct Vec8<FP8> { using type = uint2; };

template <class KT, class CT>
__device__ __forceinline__ typename Vec8<CT>::type load8(const typename Elem<KT>::storage* src, const Fp8Scale& s) {
  if constexpr (std::is_same<CT, FP8>::value)
    return encode8<KT>(src, s);
  else
    return load_vec16<KT, CT>(src);
}

template <bool NT> __device__ __forceinline__ void store8(void* dst, uint4 v) {
  if constexpr (NT)
    __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, v), reinterpret_cast<u32x4_t*>(dst));
  else
    *reinterpret_cast<uint4*>(dst) = v;
}
template <bool NT> __device__ __forceinline__ void store8(void* dst, uint2 v) {
  if constexpr (NT)
    __builtin_nontemporal_store(__builtin_bit_cast(u32x2_t, v), reinterpret_cast<u32x2_t*>(dst));
  else
    *reinterpret_cast<uint2*>(dst) = v;
}

// Two neighbouring source elements as floats (or raw 16-bit words when the
// cache has the source's type).
template <class KT> struct Pair { float a, b; };
template <class KT>
__device__ __forceinline__ Pair<KT> load_pair(const typename Elem<KT>::storage* src) {
  if constexpr (std::is_same<KT, F32>::value) {
    const float2 x = *reinterpret_cast<const float2*>(src);
    return {x.x, x.y};
  } else {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(src);
    return {to_f32<KT>((uint16_t)(w & 0xffffu)), to_f32<KT>((uint16_t)(w >> 16))};
  }
}

// A V task's four tokens of two dimensions -> eight tokens of one: this
// lane's four of dimension d0 + (lane & 1) and its neighbour's.  (Both
// dimensions are exchanged and the lane keeps one: the exchange then reads
// registers as loaded, never a select's result.)
__device__ __forceinline__ uint32_t swap_pair(uint32_t x) {
  constexpr int kSwap1 = 1 | (0 << 2) | (3 << 4) | (2 << 6);  // quad_perm: lane ^ 1
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kSwap1, 0xf, 0xf, false);
}

template <class KT, class CT>
__device__ __forceinline__ typename Vec8<CT>::type load_v_task(const typename Elem<KT>::storage* src, int64_t stride,
                                                               bool odd, const Fp8Scale& s) {
  if constexpr (std::is_same<CT, FP8>::value) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const Pair<KT> w = load_pair<KT>(src + e * stride);
      x[e] = w.a;
      x[4 + e] = w.b;
    }
    const uint32_t d0 = fp8_encode4_scaled(x, s), d1 = fp8_encode4_scaled(x + 4, s);
    const uint32_t s0 = swap_pair(d0), s1 = swap_pair(d1);
    return odd ? make_uint2(s1, d1) : make_uint2(d0, s0);
  } else {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (std::is_same<KT, CT>::value) {
        w[e] = *reinterpret_cast<const uint32_t*>(src + e * stride);
      } else {
        const Pair<KT> x = load_pair<KT>(src + e * stride);
        w[e] = pack2(from_f32<CT>(x.a), from_f32<CT>(x.b));
      }
    }
    // Low halves: dimension d0 of tokens 0 1 | 2 3; high halves: d0 + 1.
    const uint2 d0 = make_uint2(__builtin_amdgcn_perm(w[1], w[0], 0x05040100u),
                                __builtin_amdgcn_perm(w[3], w[2], 0x05040100u));
    const uint2 d1 = make_uint2(__builtin_amdgcn_perm(w[1], w[0], 0x07060302u),
                                __builtin_amdgcn_perm(w[3], w[2], 0x07060302u));
    const uint2 s0 = make_uint2(swap_pair(d0.x), swap_pair(d0.y)), s1 = make_uint2(swap_pair(d1.x), swap_pair(d1.y));
    return odd ? make_uint4(s1.x, s1.y, d1.x, d1.y) : make_uint4(d0.x, d0.y, s0.x, s0.y);
  }
}

// FEW: every token on its own, in runs too, without the search for them, and
// SPLIT's division of the work: calls of fewer than BS tokens, in which no run
// exists, and small ones (the line is at window_few).  Such a call is a chain
// of round trips (kernel arguments, slots, stores), and a search between them
// shows: single tokens, kernel times, 2 heads x 64 1.84 us in a kernel without
// any search, 2.20 with it and all of SPLIT's wavefronts, 1.70 in this form;
// 8 x 128, blocks of 8, 2.44, 2.70 and 2.42.
template <class KT, class CT, int BS, bool SPLIT, bool FEW>
__global__ __launch_bounds__(256) void rac_paged_window_kernel(RacParams p, int hg, int head_groups) {
  static_assert(SPLIT || !FEW, "few tokens are split over workgroups");
  using KS = typename Elem<KT>::storage;
  using CS = typename Elem<CT>::storage;
  constexpr bool F8 = std::is_same<CT, FP8>::value;
  constexpr int X = 16 / Elem<CT>::kBytes;  // elements per 16-byte K chunk
  const int tid = threadIdx.x, lane = tid & 63;
  const int part = SPLIT ? (int)blockIdx.y : 0, parts = SPLIT ? (int)gridDim.y : 1;
  const int64_t window = head_groups == 1 ? blockIdx.x : blockIdx.x / (uint32_t)head_groups;
  const int h0 = (int)(blockIdx.x - (uint32_t)window * (uint32_t)head_groups) * hg;
  const int first = part * 256 + tid, step = parts * 256;  // this thread's tasks
  const int nh = min(hg, p.num_heads - h0);
  const int D = p.head_size;
  const Fp8Scale ks{p.k_scale, p.k_inv, p.fast_div != 0}, vs{p.v_scale, p.v_inv, p.fast_div != 0};
  const KS* key = static_cast<const KS*>(p.key) + (int64_t)h0 * D;
  const KS* val = static_cast<const KS*>(p.value) + (int64_t)h0 * D;
  CS* kc = static_cast<CS*>(p.key_cache);
  CS* vc = static_cast<CS*>(p.value_cache);

  // SPLIT, 16-bit caches: the wavefront's own (token, head) of the window, whose
  // loads go out before the slots are known.
  constexpr bool kOwn = SPLIT && !F8;
  const int64_t w0 = window * BS;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint4 own_k = make_uint4(0, 0, 0, 0);
  KS own_v0 = 0, own_v1 = 0;
  const int own_tok = part * 4 + wave;  // (one head per workgroup)
  if constexpr (kOwn) {
    const int64_t tok = min(w0 + own_tok, p.num_tokens - 1);
    const KS* ksrc = key + tok * p.key_stride;
    const KS* vsrc = val + tok * p.value_stride;
    own_k = load8<KT, CT>(ksrc + 8 * min(lane, D / 8 - 1), ks);
    own_v0 = vsrc[min(lane, D - 1)];
    own_v1 = vsrc[min(lane + 64, D - 1)];
  }

  int64_t prev = -1, run = -1;
  int lane_slot;  // lanes BS .. 2 BS - 1: the window's slots
  if constexpr (FEW)
    lane_slot = lane >= BS && lane < 2 * BS && w0 + lane - BS < p.num_tokens ? p.slot_mapping[w0 + lane - BS] : -1;
  else
    rac_window_runs<BS>(p, window, lane, prev, run, lane_slot);

  if (!FEW && run >= 0) {
    const int units = D * (BS / 8);  // tasks per head
    const int64_t blk = __builtin_amdgcn_readlane(lane_slot, BS + (int)(run - w0)) / BS;
    const KS* k0 = key + run * p.key_stride;
    const KS* v0 = val + run * p.value_stride;
    const int64_t region0 = (blk * p.num_heads + h0) * (int64_t)D * BS;
    for (int i = first; i < nh * units; i += step) {
      const int h = nh == 1 ? 0 : i / units;
      const int u = i - h * units;
      const int64_t region = region0 + (int64_t)h * D * BS;
      // K: eight dimensions of one token.
      int t, d;
      if constexpr (F8) {
        t = (u >> 1) % BS;
        d = (u >> 1) / BS * 16 + (u & 1) * 8;
      } else {
        t = u % BS;
        d = u / BS * 8;
      }
      const auto kv = load8<KT, CT>(k0 + t * p.key_stride + h * D + d, ks);
      // V: dimensions 2 pair, 2 pair + 1 of tokens 4 quad .. +3.
      const int quad = u % (BS / 4), pair = u / (BS / 4);
      const auto vv = load_v_task<KT, CT>(v0 + (int64_t)(4 * quad) * p.value_stride + h * D + 2 * pair,
                                          p.value_stride, (quad & 1) != 0, vs);
      store8<true>(kc + region + 8 * u, kv);
      store8<true>(vc + region + (2 * pair + (quad & 1)) * BS + 8 * (quad >> 1), vv);
    }
  }

  // The window's other tokens.
  const int64_t s0 = prev >= 0 ? prev + BS : w0;  // prev + BS >= w0
  const int64_t s1 = run >= 0 ? run : min(w0 + BS, p.num_tokens);
  if (s0 >= s1) return;
  const int lane0 = (int)(s0 - w0) + BS;  // the lane that holds token s0's slot
  if constexpr (F8) {
    // Eight elements of a token's K and V per thread: the encoder works on
    // groups of four, and one V element per lane (as below) took an
    // 8192-token prefill of ragged prompts from 15.3 to 18.5 us.  (A
    // wavefront's trips are the same in every lane: the slots come from other
    // lanes.)
    const int per = nh * D / 8, total = (int)(s1 - s0) * per;
    for (int i = first; i - lane < total; i += step) {
      const int j = i / per, c = i - j * per;
      const int64_t tok = s0 + j;
      const int32_t slot = __shfl(lane_slot, (lane0 + j) & 63);
      if (i >= total || slot < 0 || (int64_t)slot >= p.num_slots) continue;
      const int h = nh == 1 ? 0 : 8 * c / D;
      const int d = 8 * c - h * D;
      const uint2 kv = load8<KT, CT>(key + tok * p.key_stride + 8 * c, ks);
      const uint2 vv = load8<KT, CT>(val + tok * p.value_stride + 8 * c, vs);
      const int64_t region = ((int64_t)(slot / BS) * p.num_heads + h0 + h) * (int64_t)D * BS;
      store8<false>(kc + region + ((int64_t)(d / X) * BS + slot % BS) * X + d % X, kv);
      CS* vd = vc + region + d * BS + slot % BS;
#pragma unroll
      for (int r = 0; r < 8; ++r) vd[r * BS] = (uint8_t)((r < 4 ? vv.x : vv.y) >> (8 * (r & 3)));
    }
    return;
  } else {
    // One (token, head) per wavefront and turn, lanes over the K chunks and over
    // the dimensions of V, so that a store instruction's accesses to one line
    // (64 / BS dimensions of the token) leave as one request.  (Eight dimensions
    // per lane: 2,200 random slots of 32-token blocks 40 us against 30.)  The
    // loads of U turns are issued together and unconditionally, padding lanes
    // and turns reading the last valid place.  SPLIT: one turn per wavefront.
    auto put = [&](int tok, int head, uint4 kx, KS v0, KS v1) {  // tok: counted from w0
      const int32_t slot = __builtin_amdgcn_readlane(lane_slot, BS + tok);
      if (slot < 0 || (int64_t)slot >= p.num_slots) return;
      const int64_t region = ((int64_t)(slot / BS) * p.num_heads + h0 + head) * (int64_t)D * BS;
      CS* kd = kc + region + (slot % BS) * X;
      CS* vd = vc + region + slot % BS;
      auto put_k = [&](int c, uint4 x) {
        CS* to = kd + (int64_t)c * BS * X;
        if (p.stream_k)
          store8<true>(to, x);
        else
          store8<false>(to, x);
      };
      auto put_v = [&](int d, KS x) { vd[(int64_t)d * BS] = convert_elem<KT, CT>(x); };
      if (lane < D / 8) put_k(lane, kx);
      if (lane < D) put_v(lane, v0);
      if (lane + 64 < D) put_v(lane + 64, v1);
      const KS* ksrc = key + (w0 + tok) * p.key_stride + head * D;
      const KS* vsrc = val + (w0 + tok) * p.value_stride + head * D;
      for (int c = lane + 64; c < D / 8; c += 64) put_k(c, load8<KT, CT>(ksrc + 8 * c, ks));
      for (int d = lane + 128; d < D; d += 64) put_v(d, vsrc[d]);
    };
    if constexpr (kOwn) {
      if (own_tok >= s0 - w0 && own_tok < s1 - w0) put(own_tok, 0, own_k, own_v0, own_v1);
    } else {
      constexpr int U = 4;
      const int pairs = (int)(s1 - s0) * nh;
      for (int q0 = wave; q0 < pairs; q0 += 4 * U) {
        uint4 kv[U];
        KS v0[U], v1[U];
        int tok[U], head[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int q = min(q0 + 4 * u, pairs - 1);
          tok[u] = (int)(s0 - w0) + (nh == 1 ? q : q / nh);
          head[u] = q - (tok[u] - (int)(s0 - w0)) * nh;
          const KS* ksrc = key + (w0 + tok[u]) * p.key_stride + head[u] * D;
          const KS* vsrc = val + (w0 + tok[u]) * p.value_stride + head[u] * D;
          kv[u] = load8<KT, CT>(ksrc + 8 * min(lane, D / 8 - 1), ks);
          v0[u] = vsrc[min(lane, D - 1)];
          v1[u] = vsrc[min(lane + 64, D - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (q0 + 4 * u < pairs) put(tok[u], head[u], kv[u], v0[u], v1[u]);
      }
    }
  }
}

// ---- paged 5-D layout, float32 caches, unaligned sources and other block sizes:
// one wavefront per (token, head) ------------------------------------------------
template <class KT, class CT, bool ALIGNED>
__global__ __launch_bounds__(256) void rac_paged5d_kernel(RacParams p) {
  using KS = typename Elem<KT>::storage;
  using CS = typename Elem<CT>::storage;
  constexpr int X = 16 / Elem<CT>::kBytes;  // elements per 16-byte K chunk
  const int lane = threadIdx.x & 63;
  const int64_t wid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wid >= p.num_tokens * p.num_heads) return;
  const int64_t tok = wid / p.num_heads;
  const int head = (int)(wid - tok * p.num_heads);
  const int32_t slot = p.slot_mapping[tok];
  if (slot < 0 || (int64_t)slot >= p.num_slots) return;
  const int64_t blk = slot / p.block_size;
  const int off = slot - (int)blk * p.block_size;
  const int D = p.head_size;
  const KS* ksrc = static_cast<const KS*>(p.key) + tok * p.key_stride + (int64_t)head * D;
  const KS* vsrc = static_cast<const KS*>(p.value) + tok * p.value_stride + (int64_t)head * D;
  const int64_t region = ((int64_t)blk * p.num_heads + head) * (int64_t)D * p.block_size;
  CS* kdst = static_cast<CS*>(p.key_cache) + region;    // [D/X][bs][X]
  CS* vdst = static_cast<CS*>(p.value_cache) + region;  // [D][bs]
  const int nchunk = D / X;
  // K chunks of a large call are stored nontemporally, as in the window kernel
  // (a small call keeps default stores: 8 tokens, rewritten back to back, 2.45
  // us default, 3.1 us nontemporal).
  if (ALIGNED && p.stream_k) {
    for (int c = lane; c < nchunk; c += 64)
      __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, load_vec16<KT, CT>(ksrc + c * X)),
                                  reinterpret_cast<u32x4_t*>(kdst + ((int64_t)c * p.block_size + off) * X));
  } else {
    for (int c = lane; c < nchunk; c += 64)
      convert_run<KT, CT, X, ALIGNED>(ksrc + c * X, kdst + ((int64_t)c * p.block_size + off) * X);
  }
  for (int d = lane; d < D; d += 64)
    vdst[(int64_t)d * p.block_size + off] = convert_elem<KT, CT>(vsrc[d]);
}

// ---- token-major layout: one workgroup per token, 16-byte vectors ----------------
template <class KT, class CT, int VE, bool ALIGNED>
__global__ __launch_bounds__(256) void rac_token_major_kernel(RacParams p) {
  using KS = typename Elem<KT>::storage;
  using CS = typename Elem<CT>::storage;
  const int64_t tok = blockIdx.x;
  const int32_t slot = p.slot_mapping[tok];
  if (slot < 0 || (int64_t)slot >= p.num_slots) return;
  const int row = p.num_heads * p.head_size;
  const int nvec = row / VE;  // vectors per K (or V) row
  const KS* ksrc = static_cast<const KS*>(p.key) + tok * p.key_stride;
  const KS* vsrc = static_cast<const KS*>(p.value) + tok * p.value_stride;
  CS* kdst = static_cast<CS*>(p.key_cache) + (int64_t)slot * row;
  CS* vdst = static_cast<CS*>(p.value_cache) + (int64_t)slot * row;
  for (int v = threadIdx.x; v < 2 * nvec; v += blockDim.x) {
    const bool is_v = v >= nvec;
    const int e = (is_v ? v - nvec : v) * VE;
    convert_run<KT, CT, VE, ALIGNED>((is_v ? vsrc : ksrc) + e, (is_v ? vdst : kdst) + e);
  }
}

// ---- token-major layout, wide rows: one wavefront per token -----------------------
// Each lane moves 16-byte cache vectors lane, lane+64, ... of the token's K
// row and V row (NV of each, 64 * NV / 2 < vectors per row <= 64 * NV).  All
// loads are issued, the workgroup's wavefronts meet at a barrier, then all
// store: keeping a CU's reads and writes in separate phases (rather than each
// wavefront storing the moment its loads land) measured ~10% faster on
// MI355X.  The row loads do not wait for the slot id: a padding token's row
// is read and dropped.  The stores are nontemporal: each cache line is
// written once and nothing in this launch reads it back.  (Inactive lanes
// take zeros through a conditional expression; guarding the loads with an
// if-statement instead measured ~15% slower at the same instruction count.)
// The source rows are loaded with the nontemporal policy when no conversion
// is needed: each is read once.

// Measured at 4096 tokens x 8 heads x D 128, bf16, 65,536 slots (median of
// interleaved runs, one process per variant): one token per wavefront, four
// wavefronts per workgroup, default-policy source loads 6.64 us; with
// nontemporal source loads (each source row is read once) 6.29 us; two or
// eight wavefronts per workgroup 6.62 / 6.60 us; two tokens per wavefront
// 6.85 us; one wavefront per (token, head) 9.68 us.
constexpr int kRacWaves = 4;  // wavefronts (tokens) per workgroup

template <class KT, class CT>
__device__ __forceinline__ uint4 load_src16(const typename Elem<KT>::storage* src) {
  if constexpr (std::is_same<KT, CT>::value) {
    return __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(src)));
  } else {
    return load_vec16<KT, CT>(src);
  }
}

template <class KT, class CT, int NV>
__global__ __launch_bounds__(64 * kRacWaves) void rac_token_major_wave_kernel(RacParams p) {
  using KS = typename Elem<KT>::storage;
  using CS = typename Elem<CT>::storage;
  constexpr int VE = 16 / Elem<CT>::kBytes;  // elements per 16-byte cache vector
  constexpr int TPW = 1;  // tokens per wavefront
  const int lane = threadIdx.x & 63;
  const int tok0 = ((int)blockIdx.x * kRacWaves + (int)(threadIdx.x >> 6)) * TPW;
  const int row = p.num_heads * p.head_size;
  const int nvec = row / VE;  // 64 * (NV/2) < nvec <= 64 * NV
  uint4 kx[TPW][NV], vx[TPW][NV];
  int32_t slot[TPW];
#pragma unroll
  for (int u = 0; u < TPW; ++u) {
    const int tok = tok0 + u;
    // Wavefronts past the last token stay for the barrier and move nothing.
    const bool live = tok < p.num_tokens;
    slot[u] = live ? p.slot_mapping[tok] : -1;
    const KS* ksrc = static_cast<const KS*>(p.key) + (int64_t)tok * p.key_stride;
    const KS* vsrc = static_cast<const KS*>(p.value) + (int64_t)tok * p.value_stride;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      const int i = 64 * c + lane;
      const bool ok = live && i < nvec;
      kx[u][c] = ok ? load_src16<KT, CT>(ksrc + i * VE) : make_uint4(0, 0, 0, 0);
      vx[u][c] = ok ? load_src16<KT, CT>(vsrc + i * VE) : make_uint4(0, 0, 0, 0);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TPW; ++u) {
    if (slot[u] >= 0 && (int64_t)slot[u] < p.num_slots) {
      CS* kdst = static_cast<CS*>(p.key_cache) + (int64_t)slot[u] * row;
      CS* vdst = static_cast<CS*>(p.value_cache) + (int64_t)slot[u] * row;
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        const int i = 64 * c + lane;
        if (i < nvec) {
          __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, kx[u][c]), reinterpret_cast<u32x4_t*>(kdst + i * VE));
          __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, vx[u][c]), reinterpret_cast<u32x4_t*>(vdst + i * VE));
        }
      }
    }
  }
}

// ---- FP8 caches, token-major: one wavefront per token, each lane turning 8
// source elements into 8 code bytes per step of the K row and of the V row. ------
template <class KT>
__global__ __launch_bounds__(256) void rac_fp8_token_major_kernel(RacParams p) {
  using KS = typename Elem<KT>::storage;
  const int lane = threadIdx.x & 63;
  const int64_t tok = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tok >= p.num_tokens) return;
  const int32_t slot = p.slot_mapping[tok];
  if (slot < 0 || (int64_t)slot >= p.num_slots) return;
  const int row = p.num_heads * p.head_size;  // a multiple of 8
  const int n8 = row / 8;
  const Fp8Scale ks{p.k_scale, p.k_inv, p.fast_div != 0}, vs{p.v_scale, p.v_inv, p.fast_div != 0};
  const KS* ksrc = static_cast<const KS*>(p.key) + tok * p.key_stride;
  const KS* vsrc = static_cast<const KS*>(p.value) + tok * p.value_stride;
  uint8_t* kdst = static_cast<uint8_t*>(p.key_cache) + (int64_t)slot * row;
  uint8_t* vdst = static_cast<uint8_t*>(p.value_cache) + (int64_t)slot * row;
  for (int i = lane; i < n8; i += 64) {
    const uint2 k = encode8<KT>(ksrc + 8 * i, ks);
    const uint2 v = encode8<KT>(vsrc + 8 * i, vs);
    __builtin_nontemporal_store(k.x, reinterpret_cast<uint32_t*>(kdst + 8 * i));
    __builtin_nontemporal_store(k.y, reinterpret_cast<uint32_t*>(kdst + 8 * i) + 1);
    __builtin_nontemporal_store(v.x, reinterpret_cast<uint32_t*>(vdst + 8 * i));
    __builtin_nontemporal_store(v.y, reinterpret_cast<uint32_t*>(vdst + 8 * i) + 1);
  }
}

// ---- FP8 caches, paged 5-D layout, other block sizes: one wavefront per (token,
// head), K as 8-byte halves of the 16-byte chunks, V as single bytes. -------------
template <class KT>
__global__ __launch_bounds__(256) void rac_fp8_paged5d_kernel(RacParams p) {
  using KS = typename Elem<KT>::storage;
  const int lane = threadIdx.x & 63;
  const int64_t wid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wid >= p.num_tokens * p.num_heads) return;
  const int64_t tok = wid / p.num_heads;
  const int head = (int)(wid - tok * p.num_heads);
  const int32_t slot = p.slot_mapping[tok];
  if (slot < 0 || (int64_t)slot >= p.num_slots) return;
  const int64_t blk = slot / p.block_size;
  const int off = slot - (int)blk * p.block_size;
  const int D = p.head_size;  // a multiple of 16
  const Fp8Scale ks{p.k_scale, p.k_inv, p.fast_div != 0}, vs{p.v_scale, p.v_inv, p.fast_div != 0};
  const KS* ksrc = static_cast<const KS*>(p.key) + tok * p.key_stride + (int64_t)head * D;
  const KS* vsrc = static_cast<const KS*>(p.value) + tok * p.value_stride + (int64_t)head * D;
  const int64_t region = ((int64_t)blk * p.num_heads + head) * (int64_t)D * p.block_size;
  uint8_t* kdst = static_cast<uint8_t*>(p.key_cache) + region;    // [D/16][bs][16]
  uint8_t* vdst = static_cast<uint8_t*>(p.value_cache) + region;  // [D][bs]
  for (int c = lane; c < D / 8; c += 64) {  // 8-element halves of the 16-byte chunks
    const uint2 k = encode8<KT>(ksrc + 8 * c, ks);
    *reinterpret_cast<uint2*>(kdst + ((int64_t)(c >> 1) * p.block_size + off) * 16 + (c & 1) * 8) = k;
  }
  for (int d = lane; d < D; d += 64)
    vdst[(int64_t)d * p.block_size + off] =
        (uint8_t)fp8_e4m3_encode(__fdiv_rn(to_f32<KT>(vsrc[d]), vs.scale));
}

// Paged 5-D caches of 16-bit and FP8 elements with blocks of 8, 16 or 32
// tokens: the window kernel at every number of tokens (*ok: it took the call).
// Heads per window and 256 threads: as many as give every thread a run task.
// A small call takes one head per workgroup and splits each window over as
// many workgroups as give every token (FP8: eight elements) a wavefront
// (thread) of its own; the split index is the grid's slower one, so that the
// parts of a window mostly share an XCD and its L2 combines a block's tokens
// into lines (902 ragged tokens of 32-token blocks: 5.7 us, as with a wavefront
// per token and head; whole windows per workgroup 11.0).  The line:
// the (token, head) wavefronts that the chip holds at once (32 per CU).
// (Four heads of one token per workgroup instead of four tokens of one head:
// 500 scattered windows of 16 5.2 -> 7.4 us.)
constexpr int64_t kWindowSplitBelow = 8192;
// Whether a call takes the FEW form: in fewer than BS tokens no run exists, and
// below the line writing a run's tokens one by one costs less than finding it.
// FP8 codes always search: a run's tasks encode half as often (64 tokens in
// order, 8 x 128, blocks of 16: 3.06 us, FEW 3.73).  Measured with every token
// in a run (device time of captured calls, search -> FEW), bf16:
//   32 x 8 x 64, blocks of 32 (16K elements)    2.66  2.10
//   96 x 8 x 128, blocks of 16 (98K)            2.54  2.26
//   128 x 8 x 128, blocks of 32 (131K)          2.85  2.54
//   64 x 8 x 256, blocks of 32 (131K)           2.76  2.92
//   384 x 8 x 64, blocks of 32 (197K)           2.87  3.02
//   256 x 8 x 128, blocks of 16 (262K)          2.66  2.80
// and from float32, whose run tasks load twice the bytes:
//   128 x 8 x 128, blocks of 16 (131K)          2.97  2.38
//   256 x 8 x 128, blocks of 16 (262K)          3.11  2.81
//   512 x 8 x 128, blocks of 16 (524K)          3.26  3.81
// Scattered tokens take 0.2 to 0.4 us less in the FEW form at every size.
template <class KT, class CT, int BS>
static bool window_few(const RacParams& p) {
  if (p.num_tokens * p.num_heads >= kWindowSplitBelow) return false;
  if (p.num_tokens < BS) return true;
  if (std::is_same<CT, FP8>::value) return false;
  const int64_t line = (std::is_same<KT, F32>::value ? 1 << 18 : 1 << 17) / (p.head_size > 128 ? 2 : 1);
  return p.num_tokens * p.num_heads * p.head_size <= line;
}
template <class KT, class CT, int BS>
static hipError_t launch_window_bs(const RacParams& p, hipStream_t stream) {
  const int64_t windows = (p.num_tokens + BS - 1) / BS;
  if (window_few<KT, CT, BS>(p)) {
    // A call of one window: only wavefronts (FP8: threads) that have a token.
    const int tokens = (int)std::min<int64_t>(p.num_tokens, BS);
    const int parts = std::is_same<CT, FP8>::value ? (tokens * p.head_size + 2047) / 2048 : (tokens + 3) / 4;
    hipLaunchKernelGGL((rac_paged_window_kernel<KT, CT, BS, true, true>),
                       dim3((unsigned)(windows * p.num_heads), (unsigned)parts), dim3(256), 0, stream, p, 1,
                       p.num_heads);
  } else if (p.num_tokens * p.num_heads < kWindowSplitBelow) {
    const int parts = std::is_same<CT, FP8>::value ? std::max(1, BS * p.head_size / 2048) : BS / 4;
    hipLaunchKernelGGL((rac_paged_window_kernel<KT, CT, BS, true, false>),
                       dim3((unsigned)(windows * p.num_heads), (unsigned)parts), dim3(256), 0, stream, p, 1,
                       p.num_heads);
  } else {
    const int units = p.head_size * (BS / 8);
    const int hg = std::min(p.num_heads, (256 + units - 1) / units);
    const int groups = (p.num_heads + hg - 1) / hg;
    hipLaunchKernelGGL((rac_paged_window_kernel<KT, CT, BS, false, false>), dim3((unsigned)(windows * groups)),
                       dim3(256), 0, stream, p, hg, groups);
  }
  return hipGetLastError();
}

template <class KT, class CT>
static hipError_t launch_paged_window(const RacParams& p, hipStream_t stream, bool* ok) {
  *ok = p.head_size % 8 == 0;
  if (*ok && p.block_size == 8) return launch_window_bs<KT, CT, 8>(p, stream);
  if (*ok && p.block_size == 16) return launch_window_bs<KT, CT, 16>(p, stream);
  if (*ok && p.block_size == 32) return launch_window_bs<KT, CT, 32>(p, stream);
  *ok = false;
  return hipSuccess;
}

template <class KT>
static hipError_t launch_rac_fp8(const RacParams& p, hipStream_t stream) {
  if (p.layout == 0) {
    bool ok;
    const hipError_t e = launch_paged_window<KT, FP8>(p, stream, &ok);
    if (ok) return e;
    const int64_t waves = p.num_tokens * p.num_heads;
    hipLaunchKernelGGL((rac_fp8_paged5d_kernel<KT>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, stream, p);
  } else {
    hipLaunchKernelGGL((rac_fp8_token_major_kernel<KT>), dim3((unsigned)((p.num_tokens + 3) / 4)), dim3(256), 0,
                       stream, p);
  }
  return hipGetLastError();
}

// ---- host launchers -----------------------------------------------------------------
template <class KT, class CT>
static hipError_t launch_rac_typed(const RacParams& p, bool aligned, hipStream_t stream) {
  if (p.layout == 0) {
    if constexpr (Elem<CT>::kBytes == 2) {
      if (aligned) {
        bool ok;
        const hipError_t e = launch_paged_window<KT, CT>(p, stream, &ok);
        if (ok) return e;
      }
    }
    const int64_t waves = p.num_tokens * p.num_heads;
    const dim3 grid((unsigned)((waves + 3) / 4));
    if (aligned)
      hipLaunchKernelGGL((rac_paged5d_kernel<KT, CT, true>), grid, dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((rac_paged5d_kernel<KT, CT, false>), grid, dim3(256), 0, stream, p);
  } else {
    constexpr int VE = 16 / Elem<CT>::kBytes;
    const int row = p.num_heads * p.head_size;
    const bool vec = aligned && (row % VE == 0);
    int threads = vec ? 2 * (row / VE) : 2 * row;
    threads = threads >= 256 ? 256 : ((threads + 63) / 64) * 64;
    const dim3 grid((unsigned)p.num_tokens);
    // The one-wavefront-per-token kernels index tokens with 32-bit ints
    // (a workgroup covers at most 64 tokens).
    const int nvec = (vec && p.num_tokens <= INT32_MAX - 64) ? row / VE : 0;
    const dim3 wgrid((unsigned)((p.num_tokens + kRacWaves - 1) / kRacWaves));
    if (vec && nvec > 64 && nvec <= 128)
      hipLaunchKernelGGL((rac_token_major_wave_kernel<KT, CT, 2>), wgrid, dim3(64 * kRacWaves), 0, stream, p);
    else if (vec && nvec > 128 && nvec <= 256)
      hipLaunchKernelGGL((rac_token_major_wave_kernel<KT, CT, 4>), wgrid, dim3(64 * kRacWaves), 0, stream, p);
    else if (vec && nvec > 256 && nvec <= 512)
      hipLaunchKernelGGL((rac_token_major_wave_kernel<KT, CT, 8>), wgrid, dim3(64 * kRacWaves), 0, stream, p);
    else if (vec && nvec > 512 && nvec <= 1024)
      hipLaunchKernelGGL((rac_token_major_wave_kernel<KT, CT, 16>), wgrid, dim3(64 * kRacWaves), 0, stream, p);
    else if (vec)
      hipLaunchKernelGGL((rac_token_major_kernel<KT, CT, VE, true>), grid, dim3(threads), 0, stream, p);
    else
      hipLaunchKernelGGL((rac_token_major_kernel<KT, CT, 1, false>), grid, dim3(threads), 0, stream, p);
  }
  return hipGetLastError();
}

hipError_t launch_reshape_and_cache(const RacParams& params, bool aligned, hipStream_t stream) {
  if (params.num_tokens == 0) return hipSuccess;
  RacParams p = params;
  const int64_t cache_elem = p.cache_dtype == kF32 ? 4 : p.cache_dtype == kFP8 ? 1 : 2;
  p.stream_k = p.num_tokens * p.num_heads * p.head_size * cache_elem >= kRacStreamKBytes;
  const int kt = p.kv_dtype, ct = p.cache_dtype;
  if (kt == kF32 && ct == kF32) return launch_rac_typed<F32, F32>(p, aligned, stream);
  if (kt == kF16 && ct == kF16) return launch_rac_typed<F16, F16>(p, aligned, stream);
  if (kt == kBF16 && ct == kBF16) return launch_rac_typed<BF16, BF16>(p, aligned, stream);
  if (kt == kF32 && ct == kF16) return launch_rac_typed<F32, F16>(p, aligned, stream);
  if (kt == kF32 && ct == kBF16) return launch_rac_typed<F32, BF16>(p, aligned, stream);
  if (ct == kFP8) {
    if (!aligned) return hipErrorInvalidValue;  // the ABI checks alignment first
    if (kt == kF32) return launch_rac_fp8<F32>(p, stream);
    if (kt == kF16) return launch_rac_fp8<F16>(p, stream);
    if (kt == kBF16) return launch_rac_fp8<BF16>(p, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace pkv
