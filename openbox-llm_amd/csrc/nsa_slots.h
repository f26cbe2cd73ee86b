// The sum over a query row's selection slots: the forward's partials merged
// into the selection output, and the dQ partials added up.  Used by the
// merges of their own (nsa_selbo.hip) and by the range kernels that finish
// the rows (nsa_range.hip).
//
// A row of D elements is handled by D / 8 consecutive lanes, 16 bytes of every
// slot each.  These kernels stream 8 to 34 GB per launch at the full shapes
// and are bound by how many loads they issue: the 16 slots' row pieces are one
// load a lane each, but the slots' indices and (m, l) pairs, the same for all
// lanes of a row, are loaded once per row (16 / (D / 8) slots a lane) and
// passed between the row's lanes in registers.  With one index and one pair
// loaded per lane and slot (48 load instructions for 16 KB instead of 18, and
// 16 exponentials a lane instead of one) the merge ran at 5.2 TB/s.
#pragma once

#include "nsa_items.h"
#include "nsa_tile32.h"

namespace nsa {

template <int D> struct SlotLanes {
  static constexpr int CPR = D / 8;         // lanes per row
  static constexpr int SPL = 16 / CPR;      // slots of a batch of 16 whose index a lane loads
  template <int CTRL> static __device__ __forceinline__ float dpp(float x) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(x), CTRL, 0xF, 0xF, false));
  }
  // butterfly over the row's lanes (quad swaps, half-row and row mirrors)
  template <typename Op> static __device__ __forceinline__ float reduce(float x, Op op) {
    x = op(x, dpp<0xB1>(x));                           // quad_perm [1,0,3,2]
    if constexpr (CPR >= 4) x = op(x, dpp<0x4E>(x));   // quad_perm [2,3,0,1]
    if constexpr (CPR >= 8) x = op(x, dpp<0x141>(x));  // row_half_mirror
    if constexpr (CPR >= 16) x = op(x, dpp<0x140>(x)); // row_mirror
    return x;
  }
  // the value that lane K % CPR of the row holds for slot K of the batch
  template <int K> static __device__ __forceinline__ float of(const float (&v)[SPL]) {
    constexpr int c = K % CPR;
    const float x = v[K / CPR];
    if constexpr (CPR == 16) {
      return dpp<0x150 + c>(x);   // row_newbcast
    } else if constexpr (CPR == 8) {
      int y = __builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x150 + c, 0xF, 0x3, false);
      y = __builtin_amdgcn_update_dpp(y, (int)__float_as_uint(x), 0x158 + c, 0xF, 0xC, false);
      return __uint_as_float((uint32_t)y);
    } else if constexpr (CPR == 4) {
      return dpp<0x55 * c>(x);    // quad_perm [c,c,c,c]
    } else {
      return dpp<(c | (c << 2) | ((2 + c) << 4) | ((2 + c) << 6))>(x);   // quad_perm [c,c,2+c,2+c]
    }
  }
};

// A lane's address as a wave-uniform base (the first lane's; a wave's rows
// ascend) and an unsigned 32-bit offset: the slots' loads then share one
// offset register, their distance is scalar arithmetic.
struct LaneAddr {
  uint64_t base;
  uint32_t off;
};
__device__ __forceinline__ LaneAddr lane_addr(const void* p) {
  const uint64_t a = (uint64_t)(uintptr_t)p;
  LaneAddr r;
  r.base = u64_from_halves(__builtin_amdgcn_readfirstlane((uint32_t)a),
                           __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32)));
  r.off = (uint32_t)(a - r.base);
  return r;
}

// Slots whose row pieces are in flight together: a float piece is two loads and
// eight registers.  TIGHT: in a range kernel, beside the row's accumulators and
// operands; with eight pieces the float32 forward spilled 15 to 64 registers
// and finishing a D = 64 window (T8192 Hq4 B2) took 161 us, with four it takes
// 147.
template <typename P> constexpr int slot_loads(bool tight) { return sizeof(P) == 4 ? (tight ? 4 : 8) : 16; }

// Merge of the selection partials of one row (query t of pair row qs = (b Hkv
// + hkv) T + t, head gl of the group): this lane's 8 elements (chunk c8) of
// acc / Ls are o, M + log2(Ls) the row's log-sum-exp in log2 units.  Slots
// that do not count were maybe never written: nothing of them is used.  A
// running maximum over batches of 16 slots.  Whole rows of lanes call this.
template <typename P, int D, bool TIGHT>
__device__ __forceinline__ void merge_slots(const P* __restrict__ opart, const float2* __restrict__ ml,
                                            const int32_t* __restrict__ idx, int64_t qs, int t, int gl, int G, int S,
                                            int nsub, int n_csr, int L, int c8, float (&acc)[8], float& M,
                                            float& Ls) {
  using SL = SlotLanes<D>;
  const int NS = S * nsub;
  const int32_t* irow = idx + qs * S;
  const LaneAddr pa = lane_addr(opart + (qs * NS * G + gl) * D + 8 * c8);
  const uint32_t pitch = (uint32_t)(G * D * (int)sizeof(P));   // bytes between a row's slots
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
  M = -__builtin_inff();
  Ls = 0.0f;
  for (int s0 = 0; s0 < NS; s0 += 16) {
    float2 p[SL::SPL];
    int j[SL::SPL];
#pragma unroll
    for (int u = 0; u < SL::SPL; ++u) {
      const int sl = s0 + c8 + SL::CPR * u < NS ? s0 + c8 + SL::CPR * u : NS - 1;
      j[u] = irow[sl / nsub];
      p[u] = ml[(qs * NS + sl) * G + gl];
    }
    constexpr int XB = slot_loads<P>(TIGHT);
    Raw8<P> x[XB];
    auto load = [&](int k0) {
#pragma unroll
      for (int k = 0; k < XB; ++k) {
        const int sl = s0 + k0 + k < NS ? s0 + k0 + k : NS - 1;
        x[k].load_nt(reinterpret_cast<const P*>((const char*)(uintptr_t)(pa.base + (uint64_t)sl * pitch) + pa.off));
      }
    };
    load(0);
    float w[SL::SPL], bm = M;
#pragma unroll
    for (int u = 0; u < SL::SPL; ++u) {
      const bool ok = s0 + c8 + SL::CPR * u < NS && sel_slot_valid(j[u], n_csr, L, t) && p[u].y > 0.0f;
      w[u] = ok ? p[u].x : -__builtin_inff();
      p[u].y = ok ? p[u].y : 0.0f;
      bm = fmaxf(bm, w[u]);
    }
    bm = SL::reduce(bm, [](float a, float b) { return fmaxf(a, b); });
    if (bm == -__builtin_inff()) continue;   // nothing valid yet (the same for the row's lanes)
    float ls = 0.0f;
    bool all = true;
#pragma unroll
    for (int u = 0; u < SL::SPL; ++u) {
      // a weight that underflows to 0 still counts (0 times an infinite or NaN
      // partial is NaN); negative: the slot does not, its l is 0
      w[u] = p[u].y > 0.0f ? fast_exp2(w[u] - bm) : -1.0f;
      ls += w[u] * p[u].y;
      all &= p[u].y > 0.0f;
    }
    const float rs = M == -__builtin_inff() ? 0.0f : fast_exp2(M - bm);
    Ls = Ls * rs + SL::reduce(ls, [](float a, float b) { return a + b; });
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] *= rs;
    static_for<0, 16 / XB>([&](auto half) {
      constexpr int k0 = half.value * XB;
      if constexpr (k0 > 0) {
        __builtin_amdgcn_sched_barrier(0);   // not before the first half is added: its registers are needed
        load(k0);
      }
      if (!__all(all)) {
        static_for<0, XB>([&](auto k) { x[k.value].keep_if(!(SL::template of<k0 + k.value>(w) < 0.0f)); });
      }
      static_for<0, XB>([&](auto k) {
        const float wk = SL::template of<k0 + k.value>(w);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += wk * x[k.value].get(i);
      });
    });
    M = bm;
  }
}

// v += the dQ partials of the row's valid slots, in slot order (arguments as
// merge_slots).  The partials are read once, past the caches, but for float
// pieces in a launch of their own: their two loads share each line (T8192 Hq16
// D64, us, cached / past the caches: B1 128 MiB 23.5 / 28.5, B4 2 GiB 403 / 451;
// bf16 B4 1 GiB 219 / 191).
template <typename T, int D, bool TIGHT>
__device__ __forceinline__ void add_slots(const T* __restrict__ part, const int32_t* __restrict__ idx, int64_t qs,
                                          int t, int gl, int G, int S, int nsub, int n_csr, int L, int c8, int lane,
                                          float (&v)[8]) {
  using SL = SlotLanes<D>;
  const int NS = S * nsub;
  const int32_t* irow = idx + qs * S;
  const LaneAddr pa = lane_addr(part + (qs * NS * G + gl) * D + 8 * c8);
  const uint32_t pitch = (uint32_t)(G * D * (int)sizeof(T));   // bytes between a row's slots
  for (int s0 = 0; s0 < NS; s0 += 16) {
    int j[SL::SPL];
#pragma unroll
    for (int u = 0; u < SL::SPL; ++u) {
      const int sl = s0 + c8 + SL::CPR * u < NS ? s0 + c8 + SL::CPR * u : NS - 1;
      j[u] = irow[sl / nsub];
    }
    constexpr int XB = slot_loads<T>(TIGHT);
    Raw8<T> x[XB];
    auto load = [&](int k0) {
#pragma unroll
      for (int k = 0; k < XB; ++k) {
        const int sl = s0 + k0 + k < NS ? s0 + k0 + k : NS - 1;
        const T* src = reinterpret_cast<const T*>((const char*)(uintptr_t)(pa.base + (uint64_t)sl * pitch) + pa.off);
        if constexpr (sizeof(T) == 2 || TIGHT)
          x[k].load_nt(src);
        else
          x[k].load(src);
      }
    };
    load(0);
    uint32_t bits = 0;   // bit k: slot s0 + k counts
#pragma unroll
    for (int u = 0; u < SL::SPL; ++u) {
      const uint64_t m = __ballot(s0 + c8 + SL::CPR * u < NS && sel_slot_valid(j[u], n_csr, L, t));
      bits |= ((uint32_t)(m >> (lane & ~(SL::CPR - 1))) & ((1u << SL::CPR) - 1u)) << (SL::CPR * u);
    }
    const bool all = __all(bits == 0xFFFFu);
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += XB) {
      if (k0 > 0) {
        __builtin_amdgcn_sched_barrier(0);   // not before the first half is added: its registers are needed
        load(k0);
      }
      if (!all) {
#pragma unroll
        for (int k = 0; k < XB; ++k) x[k].keep_if((bits >> (k0 + k)) & 1u);
      }
#pragma unroll
      for (int k = 0; k < XB; ++k)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += x[k].get(i);
    }
  }
}

}  // namespace nsa
