// fa2_kernel_decode_f32.h - fp32 decode_attention / speculative_decode_attention
// on v_mfma_f32_16x16x4_f32, K and V streamed from HBM into registers.
//
// The references compute fp32 decode in fp32 (decode.py:84, 92-160;
// speculative_decode.py:91-175).  A unit's rows are the query heads of one kv
// head times the drafts (packed-head mode, KArgs::pack_m), in blocks of 16 NB
// rows; a key costs 4 * D * 16 NB FLOP of matrix work against 8 * D bytes.
// With one block the MFMAs could take 17 TB/s of K/V, so the kernel is bound by
// HBM; with two (17 to 32 rows) they take about 8.6, close to what HBM gives.
//   * Workgroup = 8 waves, one per CU (4, two per CU, in calls of many units of
//     one block: make_plan_packed).  Each wave walks its own 16-key tiles
//     (tile i of the workgroup's range to wave i % NW) with its own (m, l, O), so
//     all four matrix cores work whatever the row count and no barrier stands
//     between a load and its use.
//   * S^T = K Q^T: the A operand of k-step (i, e) is K[key][16 i + 4 g + e] for
//     lane group g = lane / 16, key = lane % 16, so one 16-byte load of a K row
//     feeds four MFMAs per row block straight from its registers.  Q^T lies in
//     LDS in the same fragment order.
//   * O^T = V^T P^T: k-step r takes key 4 g + r from lane group g, which is
//     register r of the S^T accumulator, so P stays where the softmax left it.
//     Lane i of a group loads V[key][64 h + 4 i ..+3]; element e feeds the dim
//     block (h, e) of dims 64 h + 4 i + e, and register r of O^T block (h, e)
//     holds dim 64 h + 16 g + 4 r + e.
//   * K(t + 1) is issued once S(t) has read K(t), V(t + 1) once PV(t) has read
//     V(t): two waves per SIMD keep 64 to 128 KB per CU in flight.  (A second
//     K buffer, issued a phase earlier, gained 3 % on large two-block calls and
//     spilled with one block at D = 128.)
//   * The running max is raised, and O rescaled, only when a score passes it by
//     2^8; the cross-lane maximum is skipped otherwise.  The largest weight is
//     finite and not zero for scores of any finite size (Max32).
//   * Rounding: with one block S is summed in eight chains and O in two levels
//     (kFlush), so that the error against 64 bits stays at or below that of a
//     tree over many lanes (2.1e-7 relative at 8192 keys).
//   * The waves' states meet in LDS, added up by all threads in wave order; cut
//     units merge through their partials (fa2_decode_walk.h).  The next piece's
//     first tile and Q are loaded under the merge of a whole unit: 256 x 50-150 keys
//     Hq32/Hkv32 D128 302 -> 276 us, with four-wave workgroups 220.
//   * With several blocks per unit K and V stay in L2 for the others (no nt loads):
//     64 x 2000-6000 keys, 8 kv heads x 128 rows D64 960 -> 830 us, with blocks of 64
//     rows 700.
//
// Measured on MI355X, us per call, against a dot-product kernel on the VALU
// (up to 8 rows) and 32x32x2 MFMAs with one 32-row block per wave (above):
// 16 sequences of 512-4096 keys, Hq16/Hkv4 D128, 8 drafts (32 rows): 806 -> 49;
// 64 sequences of 512-8192 keys, Hq32/Hkv8 D128, decode: 459 -> 368 (6.1 TB/s),
// 8 drafts: 1238 -> 462 (77 TFLOP/s); 16 x 8192 keys, 8 heads of D64, decode:
// 124 -> 113, 8 drafts: 171 -> 120; one sequence of 4000 keys: 178 -> 24.
#pragma once

#include "fa2_decode_walk.h"

namespace fa2 {

constexpr int kDecF32Waves = 8;  // waves of a CU: one workgroup, or two of four each

__device__ __forceinline__ f32x4 mma16_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// NB: 16-row blocks of a unit (block_rows = 16 NB); NW: waves of a workgroup
template <int D, int MODE, int NB, int NW>
__global__ __launch_bounds__(64 * NW, kDecF32Waves / 4) void fa2_decode_f32_kernel(KArgs a) {
  constexpr int kThr = 64 * NW;
  constexpr int DJ = D / 16;  // 16-dim groups of K and Q: 4 MFMA k-steps each
  constexpr int DH = D / 64;  // 64-dim groups of V and O
  constexpr int R = 16 * NB;
  constexpr int kSChains = NB == 1 ? 8 : 2;
  // O and l are summed over kFlush tiles at a time (NB = 1), which keeps the
  // chains of rounded sums as short as a tree over more lanes would
  constexpr bool kTwoLevel = NB == 1;
  constexpr int kFlush = 2;
  constexpr int kQBytes = NB * DJ * 64 * 16;       // Q fragments
  // one wave's O, rows padded so that 16 lanes write 16 rows conflict-free
  constexpr int kOPitch = (D + 4) * 4;
  constexpr int kOBytes = R * kOPitch;
  constexpr int kLds = NW * kOBytes;  // (Q first, then every wave's O)
  static_assert(kLds >= kQBytes && kLds >= kMergePieceBytes<kThr>, "LDS areas");
  __shared__ __attribute__((aligned(16))) char lds[kLds];
  __shared__ float mrg_ml[NW][R][2];
  __shared__ DecSegment seg_sh;
  __shared__ int merge_flag;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const bool causal = a.mask != FA2_MASK_NONE;
  const bool walk = a.walk_segs > 0;
  int stream = walk ? static_cast<int>(blockIdx.x) % a.walk_streams : 0;
  const int seg_k = walk ? static_cast<int>(blockIdx.x) / a.walk_streams : 0;

  const float scale = a.scale_log2;

  DecPiece p;
  DecSegment sg{};
  if (walk) {
    if (wave == 0) walk_locate<MODE>(a, seg_k, &seg_sh);
    __syncthreads();
    sg.j = __builtin_amdgcn_readfirstlane(seg_sh.j);
    sg.us = __builtin_amdgcn_readfirstlane(seg_sh.us);
    sg.s0 = __builtin_amdgcn_readfirstlane(seg_sh.s0);
    sg.s1 = __builtin_amdgcn_readfirstlane(seg_sh.s1);
    sg.C = __builtin_amdgcn_readfirstlane(seg_sh.C);
    if (!walk_piece<MODE>(a, sg, stream, seg_k, sg.j, sg.us, p)) return;
  } else if (!split_piece<MODE>(a, p)) {
    return;
  }

  // The piece whose tiles are being loaded: its sequence, keys, and this wave's
  // next tile.
  int b, k_end, n0;
  const float *kbase, *vbase;
  constexpr int kStep = 16 * NW;
  // physical rows (in K and V) of key n, clamped to the range, and to the
  // pool where its size is known (no read outside the allocation)
  auto row_of = [&](const int32_t* table, int64_t stride, int n) -> int {
    n = max(min(n, k_end - 1), 0);
    if constexpr (MODE == FA2_LAYOUT_PAGED) {
      const int pidx = a.page_shift >= 0 ? n >> a.page_shift : n / a.page_size;
      const int row = table[b * stride + pidx] * a.page_size + (n - pidx * a.page_size);
      return a.kv_len > 0 ? min(max(row, 0), a.kv_len - 1) : row;
    } else {
      return n;
    }
  };
  auto krow_of = [&](int n) { return row_of(a.k_table, a.k_table_stride, n); };
  auto vrow_of = [&](int n) { return row_of(a.v_table, a.v_table_stride, n); };

  f32x4 kx[DJ], vx[4][DH];
  auto load_k = [&](int row) {
    const f32x4* kp = reinterpret_cast<const f32x4*>(kbase + static_cast<int64_t>(row) * a.k_ss);
#pragma unroll
    for (int i = 0; i < DJ; ++i) kx[i] = NB > 1 ? kp[4 * i] : __builtin_nontemporal_load(kp + 4 * i);
  };
  auto load_v = [&](int row16) {  // row16: the physical row of key lane % 16
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = __shfl(row16, 4 * g + r);
      const f32x4* vp = reinterpret_cast<const f32x4*>(vbase + static_cast<int64_t>(row) * a.v_ss);
#pragma unroll
      for (int h = 0; h < DH; ++h) vx[r][h] = NB > 1 ? vp[16 * h] : __builtin_nontemporal_load(vp + 16 * h);
    }
  };
  int krow = 0, vrow = 0;  // of the tile after the one loaded
  constexpr int kQF = (NB * DJ * 64 + kThr - 1) / kThr;
  f32x4 qx[kQF];  // Q in fragment order, on its way to LDS
  // the first tile's and Q's loads of piece x
  auto begin = [&](const DecPiece& x) {
    b = x.w.b;
    k_end = min((x.t0 + x.T) * kBN, x.w.Lk);
    n0 = x.t0 * kBN + wave * 16;
    kbase = static_cast<const float*>(a.k) + x.w.k_base + 4 * g;
    vbase = static_cast<const float*>(a.v) + x.w.v_base + 4 * l16;
    const int row0 = x.w.qblk * R;
    const int rows = min(x.w.Lq - row0, R);
    const float* qp = static_cast<const float*>(a.q) + x.w.q_base;
#pragma unroll
    for (int y = 0; y < kQF; ++y) {
      const int f = tid + y * kThr;
      const int fl = f & 63, fj = (f >> 6) % DJ, fn = (f >> 6) / DJ;
      const int row = fn * 16 + (fl & 15);
      qx[y] = f < NB * DJ * 64 && row < rows
                  ? *reinterpret_cast<const f32x4*>(
                        qp + static_cast<int64_t>(row0 + row) * a.q_ss + 16 * fj + 4 * (fl >> 4))
                  : (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    if (n0 < k_end) {
      krow = krow_of(n0 + l16);
      vrow = vrow_of(n0 + l16);
      load_k(krow);
      load_v(vrow);
      krow = krow_of(n0 + kStep + l16);
      vrow = vrow_of(n0 + kStep + l16);
    }
  };

  begin(p);
  for (;;) {
    const Work& w = p.w;
    const int row0 = w.qblk * R;
    const int rows = min(w.Lq - row0, R);
#pragma unroll
    for (int y = 0; y < kQF; ++y) {
      const int f = tid + y * kThr;
      if (f < NB * DJ * 64) *reinterpret_cast<f32x4*>(lds + f * 16) = qx[y];
    }
    DecPiece next;
    bool has_next = walk;
    if (walk) {
      int j = w.b;
      walk_next_unit(a, sg, j, stream);
      has_next = walk_piece<MODE>(a, sg, stream, seg_k, j, p.us + p.W, next);
    }
    int last[NB];  // last visible key of this lane's row
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      last[nb] = causal ? min(k_end - 1, w.off + diag_row(a, row0 + nb * 16 + l16)) : k_end - 1;
    // no key of a tile below this one is hidden from any row
    const int full = causal ? min(k_end, w.off + 1) : k_end;

    Max32 m[NB];
    float l[NB];
    f32x4 o[NB][DH][4];
    f32x4 o2[DH][4];  // kTwoLevel: the flushed sums
    float l2 = 0.f;
    int left = kFlush;
#pragma unroll
    for (int h = 0; h < DH; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) o2[h][e] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      m[nb] = Max32{-INFINITY, 0.f};
      l[nb] = 0.f;
#pragma unroll
      for (int h = 0; h < DH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[nb][h][e] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();

    for (; n0 < k_end; n0 += kStep) {
      const bool more = n0 + kStep < k_end;
      // (several chains per block: shorter sums, less rounding)
      f32x4 s[NB], sc[NB][kSChains];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int c = 0; c < kSChains; ++c) sc[nb][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < DJ; ++i) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const f32x4 q = *reinterpret_cast<const f32x4*>(lds + ((nb * DJ + i) * 64 + lane) * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sc[nb][(4 * i + e) % kSChains] =
                mma16_f32(kx[i][e], q[e], sc[nb][(4 * i + e) % kSChains]);
        }
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int c = kSChains / 2; c > 0; c /= 2)
#pragma unroll
          for (int x = 0; x < c; ++x) sc[nb][x] += sc[nb][x + c];
        s[nb] = sc[nb][0];
      }
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        load_k(krow);
        krow = krow_of(n0 + 2 * kStep + l16);
      }
      __builtin_amdgcn_sched_barrier(0);
      float mx[NB];
      bool need = false;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if (n0 + 16 > full) {
#pragma unroll
          for (int r = 0; r < 4; ++r) s[nb][r] = n0 + 4 * g + r <= last[nb] ? s[nb][r] : -INFINITY;
        }
        mx[nb] = fmaxf(fmaxf(s[nb][0], s[nb][1]), fmaxf(s[nb][2], s[nb][3]));
        need |= over32(mx[nb], scale, m[nb]) > kRescaleThreshold;
      }
      if (__any(need)) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          float x = mx[nb];
          x = fmaxf(x, __shfl_xor(x, 16));
          x = fmaxf(x, __shfl_xor(x, 32));
          const float alpha = raise32(m[nb], x, scale);
          l[nb] *= alpha;
#pragma unroll
          for (int h = 0; h < DH; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              o[nb][h][e] *= alpha;
              if (kTwoLevel) o2[h][e] *= alpha;
            }
          if (kTwoLevel) l2 *= alpha;
        }
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const Max32 ref = m[nb].mu == -INFINITY ? Max32{0.f, 0.f} : m[nb];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[nb][r] = fast_exp2(over32(s[nb][r], scale, ref));
          l[nb] += s[nb][r];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int h = 0; h < DH; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              o[nb][h][e] = mma16_f32(vx[r][h][e], s[nb][r], o[nb][h][e]);
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        load_v(vrow);
        vrow = vrow_of(n0 + 2 * kStep + l16);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (kTwoLevel && --left == 0) {
        left = kFlush;
        l2 += l[0];
        l[0] = 0.f;
#pragma unroll
        for (int h = 0; h < DH; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            o2[h][e] += o[0][h][e];
            o[0][h][e] = (f32x4){0.f, 0.f, 0.f, 0.f};
          }
      }
    }
    if constexpr (kTwoLevel) {
      l[0] += l2;
#pragma unroll
      for (int h = 0; h < DH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[0][h][e] += o2[h][e];
    }

    // the next piece's first loads run under this one's merge (a cut unit's piece
    // publishes its partials and counts first: both wait for all earlier loads)
    if (has_next && p.np == 1) begin(next);

    // merge the waves: their (m, l), then every wave's O scaled to the common
    // max goes through LDS and all threads add up rows, in wave order
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      l[nb] += __shfl_xor(l[nb], 16);
      l[nb] += __shfl_xor(l[nb], 32);
      if (g == 0) {
        mrg_ml[wave][nb * 16 + l16][0] = m[nb].mu;
        mrg_ml[wave][nb * 16 + l16][1] = l[nb];
      }
    }
    __syncthreads();  // (also: every wave is done with Q)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      float mg = -INFINITY;
#pragma unroll
      for (int x = 0; x < NW; ++x) mg = fmaxf(mg, mrg_ml[x][nb * 16 + l16][0]);
      const float f = fast_exp2(m[nb].mu - (mg == -INFINITY ? 0.f : mg));
      char* po = lds + wave * kOBytes + (nb * 16 + l16) * kOPitch + 16 * g * 4;
      if (nb * 16 + l16 < rows) {
#pragma unroll
        for (int h = 0; h < DH; ++h)
#pragma unroll
          for (int x = 0; x < 4; ++x)
            *reinterpret_cast<f32x4*>(po + (64 * h + 4 * x) * 4) =
                (f32x4){o[nb][h][0][x] * f, o[nb][h][1][x] * f, o[nb][h][2][x] * f,
                        o[nb][h][3][x] * f};
      }
    }
    __syncthreads();
    {
      const int64_t slot = p.np == 1 ? 0
                           : walk    ? walk_slot(a, sg.C, p.us, stream, p.mine)
                                     : static_cast<int64_t>(p.mine) * a.part_slots + p.unit;
      const uint32_t pr = static_cast<uint32_t>(a.part_rows);
      const __amdgpu_buffer_rsrc_t rm = make_rsrc_uniform(a.part_ml + slot * pr * 2, pr * 8);
      const __amdgpu_buffer_rsrc_t ro = make_rsrc_uniform(a.part_o + slot * pr * D, pr * D * 4);
      constexpr int kTPR = D / 4;
      const int col = (tid % kTPR) * 4;
      for (int r = tid / kTPR; r < rows; r += kThr / kTPR) {
        float mg = -INFINITY;
#pragma unroll
        for (int x = 0; x < NW; ++x) mg = fmaxf(mg, mrg_ml[x][r][0]);
        const float mu = mg == -INFINITY ? 0.f : mg;
        float lt = 0.f;
        f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < NW; ++x) {
          lt += mrg_ml[x][r][1] * fast_exp2(mrg_ml[x][r][0] - mu);
          acc += *reinterpret_cast<const f32x4*>(lds + x * kOBytes + r * kOPitch + col * 4);
        }
        if (p.np == 1) {  // 0/0 -> NaN for a row with no key, as the reference
          *reinterpret_cast<f32x4*>(static_cast<float*>(a.o) + w.o_base +
                                    static_cast<int64_t>(row0 + r) * a.o_ss + col) =
              acc * (1.f / lt);
        } else {
          if (col == 0)
            __builtin_amdgcn_raw_buffer_store_b64(
                (u32x2){__builtin_bit_cast(uint32_t, mg), __builtin_bit_cast(uint32_t, lt)}, rm,
                r * 8, 0, kCpolSc1);
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), ro,
                                                 (r * D + col) * 4, 0, kCpolSc1);
        }
      }
    }
    if (p.np > 1) {
      merge_publish();
      __syncthreads();
      if (merge_count(a, p.unit, p.np, &merge_flag)) {
        if (walk)
          merge_pieces<FA2_DTYPE_F32, D, kThr, R>(
              a, [&](int s) { return walk_slot(a, sg.C, p.us, stream, s); }, p.np, rows, w.o_base,
              row0, lds);
        else
          merge_rows<FA2_DTYPE_F32, D, kThr, R>(a, p.unit, p.np, rows, w.o_base, row0);
      }
    }
    if (!has_next) return;
    if (p.np > 1) begin(next);
    p = next;
    __syncthreads();  // the merge area becomes Q again
  }
}

}  // namespace fa2
