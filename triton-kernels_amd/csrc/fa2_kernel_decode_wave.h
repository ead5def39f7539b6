// fa2_kernel_decode_wave.h - fp16/bf16 decode_attention and
// speculative_decode_attention (packed-head mode, KArgs::pack_m > 0) with
// automatic splits: every wave streams its own K/V tiles.
//
// These calls read every K/V row once per kv head and do 4 * rows FLOP per
// element, so what counts is that each CU always has enough bytes in flight.
//   * Workgroup = 8 waves, one per CU.  A wave walks its own tiles (32 keys at
//     D = 128, 64 at D = 64: 8 KB of K and 8 KB of V; tile i of the
//     workgroup's range to wave i % 8) through its own LDS slots, filled by
//     direct-to-LDS loads of whole rows, and keeps its own (m, l, O).  No
//     barrier or hand-over stands between a load and its use: K(t + 1) goes
//     out once S(t) has read K(t), V(t + 1) once PV(t) has read V(t), and as a
//     tile's arithmetic takes a fraction of its share of the HBM time, nearly
//     all of the 128 KB per CU are in flight all the time.
//   * v_mfma_f32_16x16x32, the unit's rows (up to 16) as columns: S^T = K Q^T (A: lane l
//     holds key l % 16, dims 32 j + 8 (l / 16) ..+7), O^T = V^T P^T with the
//     32 keys of a step in the order the S^T accumulators hold them (lane
//     group g: keys 4 g ..+3 and 16 + 4 g ..+3), V^T by two transpose reads.
//   * Block-table entries of a window of keys lie in LDS, loaded a window
//     ahead, so that no vector load of the compiler's (whose wait would drain
//     the tiles in flight) is part of the tile loop, for any page size.
//   * The running max is raised, and O rescaled, only when a score passes it by
//     2^8; the cross-lane maximum is skipped otherwise.
//   * Workgroups share the KV tiles evenly (fa2_decode_walk.h).  At the end of a
//     piece each wave issues its first tile of the next one, then the waves'
//     states meet in LDS, a few rows at a time, added up in wave order.
//
// Measured on MI355X, us per call, against the producer / consumer ring of
// fa2_kernel_decode.h with a plan kernel or splits: 64 sequences of 512-8192
// keys Hq32/Hkv8 D128 208 -> 189 (6.15 TB/s; a plain read reaches 6.9), 16 x
// 8200 keys, 8 heads of D64, 8 drafts 69 -> 59, one sequence of 8000 keys
// 41 -> 21, 4 x 1023 dense 17.5 -> 12.7, 4 x 500-1500 keys Hkv8 D64 15.8 -> 10.3.
// Keys are read once (1.00 of their bytes from HBM); what is left is uneven
// service: equal shares end 121 to 186 us into the first of these calls, by kv
// head (the channels its rows fall on) and by XCD.
#pragma once

#include "fa2_decode_walk.h"
#include "fa2_kernel_lds.h"

namespace fa2 {

constexpr int kDwWaves = 8;
constexpr int kDwThreads = 64 * kDwWaves;
constexpr int kDwTable = 512;     // block-table entries of a window (K and V each)
constexpr int kDwRows = 16;       // rows of a unit at most
// rows that pass through LDS at once beside the tiles in flight
template <int D>
constexpr int kDwMergeRows = 512 / D;

typedef __attribute__((address_space(3))) f32x4 lds_f32x4_t;

template <bool BF>
__device__ __forceinline__ f32x4 mma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Non-temporal direct-to-LDS load of 16 bytes per lane from a scalar base and a
// 32-bit offset per lane (wait states as dma_buffer_x4).
__device__ __forceinline__ void dma_global_base_x4(uint64_t base, uint32_t off,
                                                   uint32_t lds_addr) {
  asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1 nt"
               :
               : "v"(off), "s"(base),
                 "{m0}"(__builtin_amdgcn_readfirstlane(static_cast<int>(lds_addr))));
}

// Wait for this wave's loads and stores in a form the compiler's own wait
// counting sees.  It does not see the asm loads: a value of its own still in
// flight when the tile loop starts would get a wait at its first use there,
// draining the tiles on every iteration.
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
}

template <int DT, int D, int MODE>
__global__ __launch_bounds__(kDwThreads, 1) void fa2_decode_wave_kernel(KArgs a) {
  static_assert(DT != FA2_DTYPE_F32, "fp32 decode runs fa2_decode_f32_kernel");
  constexpr bool BF = Elt<DT>::kBF;
  constexpr int R = kDwRows;
  constexpr int kRow = D * 2;                // bytes of a K or V row
  constexpr int NC = kRow / 16;              // 16-byte chunks of a row
  constexpr int TKW = 8192 / kRow;           // keys of a wave's tile
  constexpr int KB = TKW / 16;               // 16-key blocks of a tile
  constexpr int KK = TKW / 32;               // 32-key PV steps
  constexpr int DJ = D / 32;                 // S k-steps
  constexpr int DB = D / 16;                 // 16-dim blocks of O^T
  constexpr int kI = 8;                      // 1 KB loads of a tile's K (or V)
  constexpr int RPI = 64 / NC;               // rows of one load
  constexpr int kPitch = (D + 4) * 4;        // merge rows
  constexpr int MR = kDwMergeRows<D>;
  constexpr int kMrg = kDwWaves * MR * kPitch;
  static_assert(kDwWaves * 16 * kPitch <= kDwWaves * 16384, "merge in the tile slots");
  constexpr bool kPaged = MODE == FA2_LAYOUT_PAGED;

  __shared__ __attribute__((aligned(1024))) char tiles[kDwWaves * 16384];
  __shared__ __attribute__((aligned(16)))
  char mrg[kMrg > kMergePieceBytes<kDwThreads> ? kMrg : kMergePieceBytes<kDwThreads>];
  __shared__ float mrg_ml[kDwWaves][R][2];
  __shared__ int tab[kPaged ? 2 : 1][2][kPaged ? kDwTable : 1];
  __shared__ DecSegment seg_sh;
  __shared__ int merge_flag;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const bool causal = a.mask != FA2_MASK_NONE;
  const int stream = static_cast<int>(blockIdx.x) % a.walk_streams;
  const int seg_k = static_cast<int>(blockIdx.x) / a.walk_streams;

  if (wave == 0) walk_locate<MODE>(a, seg_k, &seg_sh);
  __syncthreads();
  DecSegment sg;
  sg.j = __builtin_amdgcn_readfirstlane(seg_sh.j);
  sg.us = __builtin_amdgcn_readfirstlane(seg_sh.us);
  sg.s0 = __builtin_amdgcn_readfirstlane(seg_sh.s0);
  sg.s1 = __builtin_amdgcn_readfirstlane(seg_sh.s1);
  sg.C = __builtin_amdgcn_readfirstlane(seg_sh.C);

  // A window: keys [ka, kb) of a piece, all of it unless its block-table
  // entries exceed the LDS table.
  struct Window {
    DecPiece p;
    int ka, kb, kend;  // kend: the piece's end
    int page0;         // first logical page
  };
  auto window_at = [&](Window& v, int ka) {
    v.ka = ka;
    v.kb = v.kend;
    v.page0 = 0;
    if constexpr (kPaged) {
      v.page0 = a.page_shift >= 0 ? ka >> a.page_shift : ka / a.page_size;
      const int64_t lim = (static_cast<int64_t>(v.page0) + kDwTable) * a.page_size;
      if (lim < v.kend) {  // whole tiles, so that every window starts at one
        const int n = (static_cast<int>(lim) - ka) / TKW * TKW;
        v.kb = ka + max(n, TKW);
      }
    }
  };
  auto first_window = [&](Window& v, int j, int us) -> bool {
    if (!walk_piece<MODE>(a, sg, stream, seg_k, j, us, v.p)) return false;
    v.kend = min((v.p.t0 + v.p.T) * kBN, v.p.w.Lk);
    window_at(v, v.p.t0 * kBN);
    return true;
  };
  auto next_window = [&](const Window& c, Window& v) -> bool {
    if (c.kb < c.kend) {
      v = c;
      window_at(v, c.kb);
      return true;
    }
    return first_window(v, walk_next(a, sg, c.p.w.b), c.p.us + c.p.W);
  };
  auto load_table = [&](const Window& v, int buf) {
    if constexpr (kPaged) {
      if (v.ka >= v.kb) return;
      const int last = a.page_shift >= 0 ? (v.kb - 1) >> a.page_shift : (v.kb - 1) / a.page_size;
      for (int i = tid; i <= last - v.page0; i += kDwThreads) {
        tab[buf][0][i] = a.k_table[v.p.w.b * a.k_table_stride + v.page0 + i];
        tab[buf][1][i] = a.v_table[v.p.w.b * a.v_table_stride + v.page0 + i];
      }
    }
  };

  Window cur, nxt;
  if (!first_window(cur, sg.j, sg.us)) return;
  bool has_next = next_window(cur, nxt);
  load_table(cur, 0);
  if (has_next) load_table(nxt, 1);
  int buf = 0;
  const int rows = min(cur.p.w.Lq, R);
  const bool ahead = rows <= 2 * MR;
  const int mr = ahead ? MR : 16;
  const uint32_t area = ahead ? lds_addr_of(mrg) : lds_addr_of(tiles);

  // LDS addresses.  K row r: chunk c at c ^ ksw(r), so that 16 lanes reading
  // one chunk of 16 rows hit distinct banks; V row r: chunk pair (32 bytes) p
  // at p ^ vsw(r), distinct for the 8 rows that 32 lanes of a transpose read.
  auto ksw = [](int r) { return D == 128 ? r & 15 : (r >> 1) & 7; };
  auto vsw = [](int r) { return D == 128 ? r & 7 : (r >> 1) & 3; };
  const uint32_t kbuf = lds_addr_of(tiles) + wave * 16384;
  const uint32_t vbuf = kbuf + 8192;
  const uint32_t qbuf = lds_addr_of(mrg);
  const uint32_t koff = l16 * kRow + ((g ^ ksw(l16)) * 16);
  const int vr = 4 * g + (l16 >> 2);
  const uint32_t voff = vr * kRow + vsw(vr) * 32 + (l16 & 3) * 8;
  const int64_t ksb = a.k_ss * 2, vsb = a.v_ss * 2;

  // loads of the tile of window v at key n0 (keys past the window are its last
  // one: finite data under a zero weight); a row outside a pool of known size
  // is clamped into it (no read outside the allocation)
  auto issue_rows = [&](auto is_v, auto pow2, const Window& v, int n0, int tb) {
    constexpr bool V = decltype(is_v)::value;
    const char* base = static_cast<const char*>(V ? a.v : a.k) + (V ? v.p.w.v_base : v.p.w.k_base) * 2;
    const int64_t sb = V ? vsb : ksb;
    const uint32_t dst = V ? vbuf : kbuf;
    int row[kI];
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      const int n = min(n0 + i * RPI + lane / NC, v.kb - 1);
      row[i] = n;
      if constexpr (kPaged) {
        const int pg = decltype(pow2)::value ? n >> a.page_shift : n / a.page_size;
        row[i] = tab[tb][V ? 1 : 0][pg - v.page0] * a.page_size + (n - pg * a.page_size);
        if (a.kv_len > 0) row[i] = min(max(row[i], 0), a.kv_len - 1);
      }
    }
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      const int r = i * RPI + lane / NC;
      const int c = (lane % NC) ^ (V ? 2 * vsw(r) : ksw(r));
      dma_global_x4<true>(base + row[i] * sb + c * 16, dst + i * 1024);
    }
  };
  // The rows of one load of a whole tile are evenly spaced in memory when they
  // lie in one page (or the layout has none): a scalar base per load and a
  // fixed offset per lane.  Lane i % 8 derives load i's base.
  const bool even = !kPaged || (a.page_shift >= 0 && a.page_size >= RPI &&
                                (a.kv_len <= 0 || a.kv_len >= RPI));
  auto issue_even = [&](auto is_v, const Window& v, int n0, int tb) {
    constexpr bool V = decltype(is_v)::value;
    const char* base = static_cast<const char*>(V ? a.v : a.k) + (V ? v.p.w.v_base : v.p.w.k_base) * 2;
    const int64_t sb = V ? vsb : ksb;
    const uint32_t dst = V ? vbuf : kbuf;
    const int n = n0 + (lane & 7) * RPI;
    int row = n;
    if constexpr (kPaged) {
      const int pg = n >> a.page_shift;
      row = tab[tb][V ? 1 : 0][pg - v.page0] * a.page_size + (n & (a.page_size - 1));
      if (a.kv_len > 0) row = min(max(row, 0), a.kv_len - RPI);
    }
    const uint64_t at = reinterpret_cast<uint64_t>(base + row * sb);
    const int lo = static_cast<int>(at), hi = static_cast<int>(at >> 32);
    const uint32_t off0 = static_cast<uint32_t>((lane / NC) * sb);
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      const int r = i * RPI + lane / NC;
      const uint32_t off = off0 + ((lane % NC) ^ (V ? 2 * vsw(r) : ksw(r))) * 16;
      const uint64_t sbase =
          (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(hi, i))) << 32) |
          static_cast<uint32_t>(__builtin_amdgcn_readlane(lo, i));
      dma_global_base_x4(sbase, off, dst + i * 1024);
    }
  };
  auto issue = [&](auto is_v, const Window& v, int n0, int tb) {
    if (even && n0 + TKW <= v.kb)
      issue_even(is_v, v, n0, tb);
    else if (!kPaged || a.page_shift >= 0)
      issue_rows(is_v, std::integral_constant<bool, true>{}, v, n0, tb);
    else
      issue_rows(is_v, std::integral_constant<bool, false>{}, v, n0, tb);
  };
  using IsK = std::integral_constant<bool, false>;
  using IsV = std::integral_constant<bool, true>;

  // Q^T (B operand, lane: row l16, dims 32 j + 8 g ..+7) lies in LDS in fragment
  // order, in the merge area between merges; one 16-byte chunk per thread.
  constexpr int kQChunks = DJ * 64;
  static_assert(kQChunks <= kDwThreads && kQChunks * 16 <= sizeof(mrg), "Q area");
  auto load_q = [&](const Work& w) -> u32x4 {
    if (tid >= kQChunks || l16 >= rows) return (u32x4){0u, 0u, 0u, 0u};
    return *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.q) + w.q_base +
                                           static_cast<int64_t>(l16) * a.q_ss + 8 * g + 32 * wave);
  };
  auto put_q = [&](const u32x4& x) {
    if (tid < kQChunks) *reinterpret_cast<u32x4*>(mrg + tid * 16) = x;
  };
  float m, l;
  f32x4 o[DB];
  auto reset = [&]() {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int d = 0; d < DB; ++d) o[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
  };

  put_q(load_q(cur.p.w));
  reset();
  __syncthreads();  // the tables and Q are in LDS
  // This wave's first tile of a window: the tiles of consecutive windows go
  // round the waves without a gap, so that none gets more than its share.
  int turn = wave;
  if (cur.ka + turn * TKW < cur.kb) {
    issue(IsK{}, cur, cur.ka + turn * TKW, buf);
    issue(IsV{}, cur, cur.ka + turn * TKW, buf);
  }

  for (;;) {
    const Work& w = cur.p.w;
    constexpr int kStep = TKW * kDwWaves;
    // last visible key of this lane's row
    const int last = causal ? min(cur.kb - 1, w.off + diag_row(a, l16)) : cur.kb - 1;
    // no key below this one is hidden from any row
    const int full = causal ? min(cur.kb, w.off + 1) : cur.kb;

    for (int n0 = cur.ka + turn * TKW; n0 < cur.kb; n0 += kStep) {
      const bool more = n0 + kStep < cur.kb;
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kI) : "memory");  // K(t)
      f32x4 s[KB];
      u32x4 kf[KB][DJ], q[DJ];
#pragma unroll
      for (int j = 0; j < DJ; ++j)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
          kf[kb][j] = *(const lds_u32x4_t*)(lds_ptr(kbuf + kb * 16 * kRow + (koff ^ (64u * j))));
#pragma unroll
      for (int j = 0; j < DJ; ++j)
        q[j] = *(const lds_u32x4_t*)(lds_ptr(qbuf + (j * 64 + lane) * 16));
      __builtin_amdgcn_sched_barrier(0);  // all reads first: one latency, not eight
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) s[kb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < DJ; ++j)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) s[kb] = mma16<BF>(kf[kb][j], q[j], s[kb]);
      // the reads of K(t) are complete: its slot takes K(t + 1)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (more) issue(IsK{}, cur, n0 + kStep, buf);

      if (n0 + TKW > full) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            s[kb][r] = n0 + 16 * kb + 4 * g + r <= last ? s[kb][r] : -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[kb][r]);
      mx *= a.scale_log2;
      if (__any(mx > m + kRescaleThreshold)) {
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float alpha = fast_exp2(m - (mn == -INFINITY ? 0.f : mn));
        m = mn;
        l *= alpha;
#pragma unroll
        for (int d = 0; d < DB; ++d) o[d] *= alpha;
      }
      const float mu = m == -INFINITY ? 0.f : m;
      u32x4 pf[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        float e[8];
#pragma unroll
        for (int r = 0; r < 8; ++r)
          e[r] = fast_exp2(__builtin_fmaf(s[2 * kk + (r >> 2)][r & 3], a.scale_log2, -mu));
        pf[kk] = (u32x4){pack2<BF>(e[0], e[1]), pack2<BF>(e[2], e[3]), pack2<BF>(e[4], e[5]),
                         pack2<BF>(e[6], e[7])};
        // row sum of the rounded weights, those that PV applies
#pragma unroll
        for (int x = 0; x < 4; ++x) l = dot2_ones<BF>(pf[kk][x], l);
      }
      if (more)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kI) : "memory");  // V(t)
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      // half of a step's V^T fragments are read before their MFMAs
      constexpr int kH = DB / 2;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          u32x4 vf[kH];
#pragma unroll
          for (int d = 0; d < kH; ++d) {
            const uint32_t va = vbuf + kk * 32 * kRow + (voff ^ (32u * (h * kH + d)));
            const u32x2 lo = __builtin_bit_cast(
                u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)lds_ptr(va)));
            const u32x2 hi = __builtin_bit_cast(
                u32x2,
                __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)lds_ptr(va + 16 * kRow)));
            vf[d] = (u32x4){lo[0], lo[1], hi[0], hi[1]};
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int d = 0; d < kH; ++d)
            o[h * kH + d] = mma16<BF>(vf[d], pf[kk], o[h * kH + d]);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (more) issue(IsV{}, cur, n0 + kStep, buf);
    }
    // This wave's first tile of the next window goes out under the merge; with
    // many rows the merge takes the tile slots instead and the tile follows it.
    turn = (turn - (cur.kb - cur.ka + TKW - 1) / TKW) & (kDwWaves - 1);
    auto issue_next = [&]() {
      if (has_next && nxt.ka + turn * TKW < nxt.kb) {
        issue(IsK{}, nxt, nxt.ka + turn * TKW, buf ^ 1);
        issue(IsV{}, nxt, nxt.ka + turn * TKW, buf ^ 1);
      }
    };
    const bool piece_end = cur.kb >= cur.kend;
    u32x4 qn = (u32x4){0u, 0u, 0u, 0u};
    if (piece_end && has_next) qn = load_q(nxt.p.w);
    if (ahead || !piece_end) issue_next();

    if (piece_end) {
      // ---- the piece's end: merge the waves' states ------------------------
      const DecPiece& p = cur.p;
      l += __shfl_xor(l, 16);
      l += __shfl_xor(l, 32);
      if (g == 0) {
        mrg_ml[wave][l16][0] = m;
        mrg_ml[wave][l16][1] = l;
      }
      __syncthreads();
      float mg = -INFINITY;
#pragma unroll
      for (int x = 0; x < kDwWaves; ++x) mg = fmaxf(mg, mrg_ml[x][l16][0]);
      const float f = fast_exp2(m - (mg == -INFINITY ? 0.f : mg));
      const int64_t slot = p.np == 1 ? 0 : walk_slot(a, sg.C, p.us, stream, p.mine);
      const uint32_t pr = static_cast<uint32_t>(a.part_rows);
      const __amdgpu_buffer_rsrc_t rm = make_rsrc_uniform(a.part_ml + slot * pr * 2, pr * 8);
      const __amdgpu_buffer_rsrc_t ro = make_rsrc_uniform(a.part_o + slot * pr * D, pr * D * 4);
      for (int r0 = 0; r0 < rows; r0 += mr) {
        if (l16 >= r0 && l16 < r0 + mr) {
          const uint32_t po = area + (wave * mr + l16 - r0) * kPitch + 16 * g;
#pragma unroll
          for (int d = 0; d < DB; ++d) *(lds_f32x4_t*)lds_ptr(po + 64 * d) = o[d] * f;
        }
        __syncthreads();
        constexpr int kTPR = D / 4;
        const int lr = tid / kTPR;
        const int r = r0 + lr;
        const int col = (tid % kTPR) * 4;
        if (lr < mr && r < rows) {
          float mt = -INFINITY;
#pragma unroll
          for (int x = 0; x < kDwWaves; ++x) mt = fmaxf(mt, mrg_ml[x][r][0]);
          const float mu = mt == -INFINITY ? 0.f : mt;
          float lt = 0.f;
          f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < kDwWaves; ++x) {
            lt += mrg_ml[x][r][1] * fast_exp2(mrg_ml[x][r][0] - mu);
            acc += *(const lds_f32x4_t*)lds_ptr(area + (x * mr + lr) * kPitch + col * 4);
          }
          if (p.np == 1) {  // 0/0 -> NaN for a row with no key, as the reference
            const float inv = 1.f / lt;
            *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.o) + w.o_base +
                                      static_cast<int64_t>(r) * a.o_ss + col) =
                (u32x2){pack2<BF>(acc[0] * inv, acc[1] * inv), pack2<BF>(acc[2] * inv, acc[3] * inv)};
          } else {
            if (col == 0)
              __builtin_amdgcn_raw_buffer_store_b64(
                  (u32x2){__builtin_bit_cast(uint32_t, mt), __builtin_bit_cast(uint32_t, lt)}, rm,
                  r * 8, 0, kCpolSc1);
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), ro,
                                                   (r * D + col) * 4, 0, kCpolSc1);
          }
        }
        __syncthreads();
      }
      if (p.np > 1) {
        merge_publish();
        __syncthreads();
        if (merge_count(a, p.unit, p.np, &merge_flag))
          merge_pieces<DT, D, kDwThreads, R>(
              a, [&](int s) { return walk_slot(a, sg.C, p.us, stream, s); }, p.np, rows, w.o_base, 0,
              mrg);
      }
      reset();
    }
    if (!has_next) return;
    __syncthreads();  // the finished window's table and the merge area are free
    if (piece_end) {
      put_q(qn);
      if (!ahead) issue_next();
    }
    cur = nxt;
    buf ^= 1;
    has_next = next_window(cur, nxt);
    if (has_next) load_table(nxt, buf ^ 1);
    __syncthreads();  // Q (and, read at this window's end, the table) is in LDS
    wait_loads();  // stores count as well
  }
}

}  // namespace fa2
