// fa2_decode_walk.h - the balanced walk of the decode kernels: every
// workgroup streams an equal share of the K/V tiles of the call.
//
// A call's units are (sequence, kv head, q-block).  The kv heads and
// q-blocks form a.walk_streams streams; stream s holds the units (b, s) of
// all sequences in order, unit b weighing max(1, ceil(Lk_b / kBN)) tiles
// of kBN = 64 keys.  The grid starts with walk_streams * walk_segs workgroups:
// workgroup g takes stream g % walk_streams and segment k = g / walk_streams of
// it, tiles [k C, (k + 1) C) with C = ceil(total / walk_segs), at least
// a.walk_min.  The kv heads of a sequence are therefore read at about the same
// time (paged rows hold all of them side by side), whatever the spread of the
// lengths every workgroup streams at most C tiles, and no plan kernel is
// launched.  A unit that a segment boundary cuts runs as pieces whose partials
// the last one to finish merges, in piece order (merge_count, merge_pieces): the
// cut points follow from the lengths alone, so results do not depend on timing.
//
// Whole units: cutting one costs its partials' round trip, about walk_whole tiles
// of a workgroup's time.  So when no unit has more than walk_short tiles, or the
// longest workgroup would take no more than walk_whole tiles beyond C with whole
// units, workgroup g takes the whole units g, g + gridDim.x, ... of the call, in
// the order (sequence, stream).
//
// Without a walk (walk_segs == 0, a forced split count) workgroup (x, y) runs
// split y of unit x.
#pragma once

#include "fa2_device.h"

namespace fa2 {

// Sequences one lane of the locating wave adds up at most.
constexpr int kWalkMaxPer = 1024;

// One piece of a unit for this workgroup.
struct DecPiece {
  Work w;
  int t0, T;     // first KV tile and tile count
  int np, mine;  // pieces of the unit, this one's index
  int us, W;     // walk: the unit's start in its stream and its weight
  int unit;      // merge word
};

template <int MODE>
__device__ __forceinline__ int walk_len(const KArgs& a, int b) {
  int n;
  if constexpr (MODE == FA2_LAYOUT_DENSE) n = a.kv_len;
  else if constexpr (MODE == FA2_LAYOUT_RAGGED) n = a.kv_indptr[b + 1] - a.kv_indptr[b];
  else n = a.kv_indptr[b];
  return n > 0 ? n : 0;
}

__device__ __forceinline__ int walk_weight(int Lk) {
  const int t = (Lk + kBN - 1) / kBN;
  return t > 1 ? t : 1;
}

// The Work of packed-head unit (sequence b, kv head kvh, q-block qblk).
template <int MODE>
__device__ __forceinline__ Work packed_work(const KArgs& a, int b, int kvh, int qblk) {
  Work w;
  w.valid = true;
  w.b = b;
  w.kvh = kvh;
  w.qblk = qblk;
  w.hg = 0;
  w.pair = 0;
  w.h = kvh * (a.hq / a.hkv);
  w.Lq = a.q_len;
  w.q_base = b * a.q_sb + w.h * a.q_sh;
  w.o_base = b * a.o_sb + w.h * a.o_sh;
  if constexpr (MODE == FA2_LAYOUT_DENSE) {
    w.Lk = a.kv_len;
    w.k_base = b * a.k_sb + kvh * a.k_sh;
    w.v_base = b * a.v_sb + kvh * a.v_sh;
  } else if constexpr (MODE == FA2_LAYOUT_RAGGED) {
    const int ks = a.kv_indptr[b];
    w.Lk = a.kv_indptr[b + 1] - ks;
    w.k_base = ks * a.k_ss + kvh * a.k_sh;
    w.v_base = ks * a.v_ss + kvh * a.v_sh;
  } else {
    w.Lk = a.kv_indptr[b];
    w.k_base = kvh * a.k_sh;
    w.v_base = kvh * a.v_sh;
  }
  if (w.Lk < 0) w.Lk = 0;
  w.off = a.mask == FA2_MASK_CAUSAL_BOTTOM_RIGHT ? w.Lk - a.pack_m : 0;
  return w;
}

// The first piece's place, from walk_locate: sequence, the unit's start in
// the stream, the segment [s0, s1) and C; C == 0: whole units.
struct DecSegment {
  int j, us, s0, s1, C;
};

// Whether units of up to `longest` tiles stay whole, walk_rounds of them per
// workgroup, rather than C tiles of cut ones; `cost`: tiles' time of cutting them.
__device__ __forceinline__ bool walk_keep_whole(const KArgs& a, int longest, int C, int cost) {
  return longest <= a.walk_short || a.walk_rounds <= (C + cost) / longest;
}

// By one wave: segment k of a stream into *sh (LDS); k >= walk_segs: empty.
template <int MODE>
__device__ __forceinline__ void walk_locate(const KArgs& a, int k, DecSegment* sh) {
  const int lane = threadIdx.x & 63;
  const int segs = a.walk_segs;
  if constexpr (MODE == FA2_LAYOUT_DENSE) {
    if (lane == 0) {
      const int W = walk_weight(a.kv_len);
      const int total = W * a.batch;
      const int C = max((total + segs - 1) / segs, a.walk_min);
      // (shares that no two units lie in have one piece to merge, not two)
      if (walk_keep_whole(a, W, C, W % C == 0 ? a.walk_whole / 2 : a.walk_whole)) {
        *sh = DecSegment{k, 0, 0, 0, 0};
        return;
      }
      const int s0 = min(k * C, total);
      *sh = DecSegment{s0 / W, (s0 / W) * W, s0, min(s0 + C, total), C};
    }
    return;
  }
  const int per = (a.batch + 63) / 64;
  const int j0 = min(a.batch, lane * per), j1 = min(a.batch, j0 + per);
  int sum = 0, longest = 0;
  for (int j = j0; j < j1; ++j) {
    const int W = walk_weight(walk_len<MODE>(a, j));
    sum += W;
    longest = max(longest, W);
  }
  if (!__any(longest > a.walk_short)) {
    if (lane == 0) *sh = DecSegment{k, 0, 0, 0, 0};
    return;
  }
  int incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(incl, d);
    if (lane >= d) incl += y;
    longest = max(longest, __shfl_xor(longest, d));
  }
  const int total = __shfl(incl, 63);
  const int C = max((total + segs - 1) / segs, a.walk_min);
  if (walk_keep_whole(a, longest, C, a.walk_whole)) {
    if (lane == 0) *sh = DecSegment{k, 0, 0, 0, 0};
    return;
  }
  const int s0 = min(k * C, total);
  const int excl = incl - sum;
  if (excl <= s0 && s0 < incl) {  // one lane, or none past the end
    int us = excl, j = j0;
    for (;; ++j) {
      const int W = walk_weight(walk_len<MODE>(a, j));
      if (s0 < us + W) break;
      us += W;
    }
    *sh = DecSegment{j, us, s0, min(s0 + C, total), C};
  } else if (lane == 0 && s0 >= total) {
    *sh = DecSegment{a.batch, total, total, total, C};
  }
}

// The piece of sequence j's unit (starting at us in its stream) that falls
// in segment g (whole units: all of it); false past the segment's end.
template <int MODE>
__device__ __forceinline__ bool walk_piece(const KArgs& a, const DecSegment& g, int stream, int k,
                                           int j, int us, DecPiece& p) {
  const bool whole = g.C == 0;
  if (j >= a.batch || (!whole && us >= g.s1)) return false;
  p.w = packed_work<MODE>(a, j, stream % a.hkv, stream / a.hkv);
  const int tiles = (p.w.Lk + kBN - 1) / kBN;
  p.us = us;
  p.W = tiles > 1 ? tiles : 1;
  p.unit = j * a.walk_streams + stream;
  if (whole) {
    p.t0 = 0;
    p.T = tiles;
    p.np = 1;
    p.mine = 0;
    return true;
  }
  const int b = max(us, g.s0), e = min(us + p.W, g.s1);
  p.t0 = b - us;
  p.T = tiles > 0 ? e - b : 0;
  const int kf = us / g.C;
  p.np = (us + p.W - 1) / g.C - kf + 1;
  p.mine = k - kf;
  return true;
}

// The sequence whose unit follows that of sequence b in segment g.
__device__ __forceinline__ int walk_next(const KArgs& a, const DecSegment& g, int b) {
  return b + (g.C == 0 ? a.walk_segs : 1);
}

// The sequence and stream of the next piece where whole units go round all
// workgroups: the unit gridDim.x = walk_dj * walk_streams + walk_ds further.
__device__ __forceinline__ void walk_next_unit(const KArgs& a, const DecSegment& g, int& j,
                                               int& stream) {
  if (g.C != 0) {
    ++j;
    return;
  }
  j += a.walk_dj;
  stream += a.walk_ds;
  if (stream >= a.walk_streams) {
    stream -= a.walk_streams;
    ++j;
  }
}

// Split blockIdx.y of unit blockIdx.x (no walk); false: no such unit.
template <int MODE>
__device__ __forceinline__ bool split_piece(const KArgs& a, DecPiece& p) {
  p.w = decode_work<MODE>(a, blockIdx.x);
  if (!p.w.valid) return false;
  const int tiles = (p.w.Lk + kBN - 1) / kBN;
  // (splits past the unit's tiles would have none: they are not counted)
  const int S = a.merge_ctr ? min(a.num_splits, max(tiles, 1)) : a.num_splits;
  const int split = blockIdx.y;
  if (split >= S) return false;
  p.t0 = (tiles * split) / S;
  p.T = (tiles * (split + 1)) / S - p.t0;
  p.np = S;
  p.mine = split;
  p.us = p.W = 0;
  p.unit = blockIdx.x;
  return true;
}

// Part slot of piece s of unit p: its workgroup's first piece (kind 0, from
// the segment's start) or last one (kind 1, from inside to the end).
__device__ __forceinline__ int64_t walk_slot(const KArgs& a, int C, int us, int stream, int s) {
  const int kf = us / C;
  const int kind = (s == 0 && us != kf * C) ? 1 : 0;
  return (static_cast<int64_t>(kf + s) * a.walk_streams + stream) * 2 + kind;
}

// LDS of merge_pieces
template <int NT>
constexpr int kMergePieceBytes = NT * 6 * 4;

// The last piece of a unit merges all of them: rows [0, rows) (rows <= MAXR)
// of the partials in part slots slot_of(s), s < np, read at device scope, the
// output of row r at o_base + (row0 + r) * o_ss.  NT threads, 4 columns each.
// With fewer rows than the threads cover, the threads split the pieces into
// groups as well, whose sums meet in LDS; pieces go four at a time, one memory
// round trip for their (m, l) and O together.  The order is fixed, whichever
// piece is last.
template <int DT, int D, int NT, int MAXR, typename SlotOf>
__device__ __forceinline__ void merge_pieces(const KArgs& a, SlotOf slot_of, int np, int rows,
                                             int64_t o_base, int row0, char* lds) {
  constexpr int kTPR = D / 4;
  constexpr int kRP = NT / kTPR;  // rows per pass of the workgroup
  constexpr int kRows = (MAXR + kRP - 1) / kRP;
  constexpr int kIt = kRows < 4 ? kRows : 4;  // rows per thread at once
  constexpr int kB = 4;                       // pieces at once
  const int tid = threadIdx.x;
  const int col = (tid % kTPR) * 4;
  const int t = tid / kTPR;
  int span = 1;  // threads' rows per group: a power of two >= rows, or all
  while (span < rows && span < kRP) span <<= 1;
  const int groups = kRP / span;
  const int gp = t / span;
  const uint32_t R = static_cast<uint32_t>(a.part_rows);
  // one descriptor each over all part slots (make_plan_packed bounds them)
  const uint32_t slots = 2u * a.walk_streams * a.walk_segs;
  const __amdgpu_buffer_rsrc_t rm = make_rsrc_uniform(a.part_ml, slots * R * 8);
  const __amdgpu_buffer_rsrc_t ro = make_rsrc_uniform(a.part_o, slots * R * D * 4);
  constexpr uint32_t kOut = 0xFFFFFF00u;  // past every range: reads zeros
  // (bit_cast through scalars: this compiler reads element 0 when bit_cast
  // is applied to a subscripted vector element)
  auto fl = [](uint32_t w) { return __builtin_bit_cast(float, w); };
  for (int c0 = 0; c0 < rows; c0 += kIt * span) {
    float m[kIt], l[kIt];
    f32x4 acc[kIt];
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
      m[it] = -INFINITY;
      l[it] = 0.f;
      acc[it] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    for (int s0 = gp; s0 < np; s0 += kB * groups) {
      u32x2 ml[kB][kIt];
      u32x4 x[kB][kIt];
#pragma unroll
      for (int j = 0; j < kB; ++j) {
        const int s = s0 + j * groups;
        const uint32_t slot = static_cast<uint32_t>(slot_of(s < np ? s : s0));
#pragma unroll
        for (int it = 0; it < kIt; ++it) {
          const uint32_t r = c0 + it * span + t % span;
          const bool ok = s < np && r < static_cast<uint32_t>(rows);
          ml[j][it] = __builtin_amdgcn_raw_buffer_load_b64(rm, ok ? (slot * R + r) * 8 : kOut, 0,
                                                           kCpolSc1);
          x[j][it] = __builtin_amdgcn_raw_buffer_load_b128(
              ro, ok ? ((slot * R + r) * D + col) * 4 : kOut, 0, kCpolSc1);
        }
      }
#pragma unroll
      for (int j = 0; j < kB; ++j)
#pragma unroll
        for (int it = 0; it < kIt; ++it)
          if (s0 + j * groups >= np) ml[j][it] = (u32x2){0xFF800000u, 0u};  // (-inf, 0)
#pragma unroll
      for (int it = 0; it < kIt; ++it) {
        float mn = m[it];
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const uint32_t mw = ml[j][it][0];
          mn = fmaxf(mn, fl(mw));
        }
        const float mu = mn == -INFINITY ? 0.f : mn;
        const float al = fast_exp2(m[it] - mu);
        l[it] *= al;
        acc[it] *= al;
        m[it] = mn;
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const uint32_t mw = ml[j][it][0], lw = ml[j][it][1];
          const float wgt = fast_exp2(fl(mw) - mu);
          l[it] += wgt * fl(lw);
          acc[it] += wgt * __builtin_bit_cast(f32x4, x[j][it]);
        }
      }
    }
    if (groups > 1) {  // (then kIt * span >= rows: one pass, one row per thread)
      float* sh = reinterpret_cast<float*>(lds);
      __syncthreads();
      *reinterpret_cast<f32x4*>(sh + tid * 4) = acc[0];
      sh[NT * 4 + tid * 2] = m[0];
      sh[NT * 4 + tid * 2 + 1] = l[0];
      __syncthreads();
      if (gp != 0) return;
      float mn = -INFINITY;
      for (int q = 0; q < groups; ++q) mn = fmaxf(mn, sh[NT * 4 + (tid + q * span * kTPR) * 2]);
      const float mu = mn == -INFINITY ? 0.f : mn;
      l[0] = 0.f;
      acc[0] = (f32x4){0.f, 0.f, 0.f, 0.f};
      for (int q = 0; q < groups; ++q) {
        const int o = tid + q * span * kTPR;
        const float wgt = fast_exp2(sh[NT * 4 + o * 2] - mu);
        l[0] += wgt * sh[NT * 4 + o * 2 + 1];
        acc[0] += wgt * *reinterpret_cast<const f32x4*>(sh + o * 4);
      }
    }
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
      const int r = c0 + it * span + t % span;
      if (r >= rows) continue;
      const float inv = 1.f / l[it];  // 0/0 -> NaN for a row with no key, as the reference
      const int64_t off = o_base + static_cast<int64_t>(row0 + r) * a.o_ss + col;
      if constexpr (DT == FA2_DTYPE_F32) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(a.o) + off) = acc[it] * inv;
      } else {
        constexpr bool BF = Elt<DT>::kBF;
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.o) + off) =
            (u32x2){pack2<BF>(acc[it][0] * inv, acc[it][1] * inv),
                    pack2<BF>(acc[it][2] * inv, acc[it][3] * inv)};
      }
    }
  }
}

}  // namespace fa2
