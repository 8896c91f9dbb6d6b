// kquant_mid.hip -- Q4_K / Q6_K x Q8_K projections of 5 to 63 columns (a
// draft, a short prompt; some of 2 to 4; host calls of more) on the gfx950
// matrix cores, bit-exact with the reference's WASM path (packages/engine/
// wasm-kernels/src/lib.rs:224-426 with the vec-dots 2116-2172 and 1923-1968).
//
// Numerics are those of kquant_prefill.hip's bit-exact kernel: per (row,
// column, block) one v_mfma_f32_16x16x32_f16 per lane class l gives aux32[l]
// exactly (Q6_K weights enter as two exact f16 operands, q6_split, so any
// int8 scale is exact), and nine f32 chains per output run in block order:
//   sums[l] += (dW_b * dX_b) * f32(aux32[l]);  Q4_K: sumf -= (dminW_b * dX_b) * f32(sumi)
//   result = [sumf +] ((((-0 + s0) + s1) + ...) + s7)
//
// Two kernels.  Few segments (Q/K/V, O, down: 160 to 192): what bounds them is
// neither the bytes (a layer's 59 MB stream in 10 us) nor the matrix cores, but
// the chains' serial walk over a row's blocks and the loads' latency along it.
// There a wave keeps two classes of a segment ("class pairs", below).  Many
// segments (gate/up, the head): instructions per weight; there a wave keeps a
// whole segment ("row waves").  Either way every column set rides on the
// weights' one trip to registers.
//
// Measured on MI355X against what these launches ran before (the vector-ALU
// kernels 8 columns at a time, or kquant_mfma's 8): with full-range Q6_K
// weights, three layers of 21 tokens 1086 -> 271 us, of 5 tokens 345 -> 245;
// gate/up + GeGLU + down 64 -> 38 us at 5 columns, 225 -> 46 at 21, 482 -> 73
// at 60; the 262144-row head at 5 columns 411 -> 137 us.  hp_mid_policy.h has
// the launches these kernels take, and both sides' times at each line.
#include "hp_common.h"
#include "hp_f2tile.h"
#include "hp_gelu.h"
#include "hp_mfma.h"
#include "hp_mid_policy.h"
#include "hp_wfrag.h"

namespace hp {

namespace {

struct MidWeight {
  const uint8_t *seg;      // segments of this weight (null: kept in one layout)
  const uint8_t *wt;       // tiles of this weight
  const uint16_t *dplane;  // Q6_K d plane
  float *out;
  int type, rows, tiles, tile_begin;  // tiles: 16-row segments
};

struct MidArgs {
  MidWeight w[kMaxWeights];
  int count, total_tiles, nb, cols;
  int S, R;  // tile geometry of the weights
  const uint8_t *xt;
  int items, col_groups;  // row waves: work items (rows x column groups)
  // gate/up + GeGLU (w[0] gate, w[1] up of equal rows): pair_out[m][row]
  float *pair_out;
  const uint16_t *gelu_lut;
};

// A column group: C sets of 16 columns, group cg at columns 16 C cg ..; a set's
// activation tiles (hp_f2tile.h) are nb * kMidXTile bytes after the set before's.
template <int C>
__device__ __forceinline__ const uint8_t *group_tiles(const uint8_t *xt, int cg, int nb) {
  return xt + (size_t)(C * cg) * nb * kMidXTile;
}

// ---- class pairs: launches with few segments --------------------------------
//
// A workgroup of four waves takes one segment and one column group; wave w
// keeps classes 2w and 2w + 1 (KL = 2; 640 waves for the 2560 rows of O or
// down, where a wave per segment would leave most SIMDs empty) and a quarter of
// the min chain's columns.  With no more workgroups than CUs, one wave a SIMD
// waits on each of its own instructions, and eight waves of one class (KL = 1)
// are faster over long rows although they unpack every header twice as often.
// The waves' classes are disjoint, so neither weights nor activations have a
// second reader in the workgroup: both go straight from global memory to
// registers, mid_depth blocks ahead, with no stage in LDS and no barrier until
// the chains meet (measured against activations copied through a ring of LDS
// stages by waves of their own: the copies, 46 bytes per clock and CU, bounded
// it).  Those loads share the CU's L1 (64 bytes and one address group a clock),
// so what lanes share is loaded once and spread by lane swaps: a row's header
// as one dword per lane, a column's d as one dword per lane of a four-lane
// group.
constexpr int mid_depth(int C) { return C == 1 ? 5 : 4; }

// The chains' exchange at the end: [9][16 C columns][16 rows, padded to 20]
// floats per segment (the padding spreads a wave's store over all banks).
constexpr int kMidRowPad = 20;

// One block of a lane's weights: row n = lane % 16 of the segment, quarter
// q = lane / 16 (elements j = 2q, 2q + 1) of classes l = KL w + g, g < KL.
template <int KL, bool Q4>
struct MidW;
template <int KL>
struct MidW<KL, true> {
  uint32_t hdr;     // dword q of the row's header (d | dmin, 12 scale/min bytes)
  uint32_t ql[KL];  // quant dwords D[q][l]
};
template <int KL>
struct MidW<KL, false> {
  uint32_t gs, d16;  // scales of groups 4q .. 4q + 3, f16 d
  uint32_t ql[KL];   // low bits D[q][l]
  uint32_t qh[KL];   // high bits Dqh[q / 2][l] (tiles: ^ 0xAA per byte)
};
// The block as loaded.  A segment stores a row's four dwords of a class side
// by side; loaded where its fragment needs it, lane (n, q) dword 4 n + q, a
// dword load touches four times the bytes it takes (16-byte strides: the L1's
// address unit was busy 84 % of the down launch).  So lane i loads dword i
// (wq: quant dwords of class l, wh: high-bit dwords, ws: header or
// scales) and mid_place spreads them.  From tiles: already in place, w.
template <int C, int KL, bool Q4, bool TILE>
struct MidRaw {
  MidW<KL, Q4> w;
  uint32_t wq[KL], wh, ws, d16;
  uint4 B[KL][C], bm[C];  // activations of column nrot(n) of each set
  float dx[C];
};

// Lane 16 q + n's weights (classes l0 ..) from the lanes that loaded them.
template <int C, int KL, bool Q4, bool TILE>
__device__ __forceinline__ MidW<KL, Q4> mid_place(const MidRaw<C, KL, Q4, TILE> &r, uint32_t n, uint32_t q,
                                                  uint32_t l0) {
  if constexpr (TILE) {
    return r.w;
  } else {
    auto from = [](uint32_t lane, uint32_t v) {
      return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(4u * lane), (int)v);
    };
    MidW<KL, Q4> w;
#pragma unroll
    for (int g = 0; g < KL; g++) w.ql[g] = from(4u * n + q, r.wq[g]);
    if constexpr (Q4) {
      w.hdr = from(4u * n + q, r.ws);
    } else {
#pragma unroll
      for (int g = 0; g < KL; g++) w.qh[g] = from(4u * n + 2u * (q >> 1) + ((l0 + g) & 1u), r.wh);
      w.gs = from(4u * n + q, r.ws);
      w.d16 = r.d16;
    }
    return w;
  }
}

template <class T>
__device__ __forceinline__ T ldg(const uint8_t *base, uint32_t off) {
  return *reinterpret_cast<const T *>(base + off);
}

// Lane dwords v (one per 16-lane row) of all four rows, in every lane.
__device__ __forceinline__ uint4 row_gather(uint32_t v) {
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  const auto e = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);
  const auto o = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
  return make_uint4(e[0], o[0], e[1], o[1]);
}

// A lane's quarter as masks: selects of loaded values that stay selects (the
// compiler turns nested ones into branches around the header's registers).
struct QuarterMasks {
  uint32_t lo, q0, q1;  // q < 2, q == 0, q == 1
};
__device__ __forceinline__ QuarterMasks quarter_masks(uint32_t q) {
  QuarterMasks m{q < 2 ? ~0u : 0u, q == 0 ? ~0u : 0u, q == 1 ? ~0u : 0u};
  asm("" : "+v"(m.lo), "+v"(m.q0), "+v"(m.q1));
  return m;
}

// The value of lane J of each four-lane group.
template <int J>
__device__ __forceinline__ float quad_lane(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), J * 0x55, 0xf, 0xf, false));
}

// Every block of one segment (tile tt of W) for the wave's two classes, and
// the Q4_K min chain of a quarter of the columns.  Sum j of lane (n, q) is row
// n, column 16 cs + 4q + (j + w) % 4: the columns are turned by w within each
// four, so that sum 0, the min chain's, is another column in each wave.
template <int C, int KL, bool Q4, bool TILE>
__device__ __forceinline__ void mid_tile(float (&s)[KL][C][4], float (&f)[C], const MidWeight &W, int tt, int nb,
                                         int S, int R, const uint8_t *xt, int w, int lane) {
  constexpr int PD = mid_depth(C), segb = Q4 ? 2304 : 3360;
  const uint32_t l0 = KL * w;
  const uint32_t n = lane & 15, q = lane >> 4;
  const uint32_t exp = magic_nib_exp();
  const QuarterMasks mq = quarter_masks(q);
  TileRow tr{};
  if constexpr (TILE) tr = tile_row(min(16 * tt + (int)n, W.rows - 1), W.rows, nb, S, R, Q4 ? 9 : 13);
  // lane offsets: within a segment, and within an activation tile
  const uint32_t os = 4u * (uint32_t)lane, oh = 2336u + 256u * (l0 >> 1) + os;
  const uint32_t oq = (Q4 ? 256u : 288u) + 1024u * (l0 & 1u) + 256u * (l0 >> 1) + os;  // (class l0 + 1 is 1024 on)
  const uint32_t od = 256u + 2u * n;
  const uint32_t nrot = (n & ~3u) | ((n + w) & 3u);
  const uint32_t ox = ((4u * l0 + q) * 16u + nrot) * 16u;       // class l0; class l0 + 1 is 1024 on
  const uint32_t ob = 8192u + ((q & 1u) * 16u + nrot) * 16u;    // (quarters 2, 3 meet zero mins)
  const uint32_t ods = 8704u + 4u * (4u * q + ((n + w) & 3u));
  auto load = [&](int b) {  // unconditional: a block past the last re-reads it
    b = min(b, nb - 1);
    MidRaw<C, KL, Q4, TILE> r;
    if constexpr (TILE) {
      // D[q][l] is dword l % 4 of quant chunk 2q + l / 4
      int i, sl;
      block_split(b, S, i, sl);
      const uint32_t off = tr.base + (uint32_t)i * tr.iter + 16u * (uint32_t)sl, at = 4u * (l0 & 3u), c = l0 >> 2;
      const uint32_t lq = off + ((Q4 ? 1u : 0u) + 2u * q + c) * tr.chunk + at;
      const uint32_t lh = off + (8u + 2u * (q >> 1) + c) * tr.chunk + at;
#pragma unroll
      for (int g = 0; g < KL; g++) r.w.ql[g] = ldg<uint32_t>(W.wt, lq + 4u * g);
      if constexpr (Q4) {
        r.w.hdr = ldg<uint32_t>(W.wt, off + 4u * q);
      } else {
        r.w.gs = ldg<uint32_t>(W.wt, off + 12u * tr.chunk + 4u * q);
        r.w.d16 = W.dplane[tr.dbase + (uint32_t)i * tr.diter + (uint32_t)sl];
#pragma unroll
        for (int g = 0; g < KL; g++) r.w.qh[g] = ldg<uint32_t>(W.wt, lh + 4u * g);
      }
    } else {
      const uint8_t *seg = W.seg + ((size_t)b * W.tiles + tt) * segb;
#pragma unroll
      for (int g = 0; g < KL; g++) r.wq[g] = ldg<uint32_t>(seg + 1024 * g, oq);
      r.ws = ldg<uint32_t>(seg, os);
      if constexpr (!Q4) {
        r.wh = ldg<uint32_t>(seg, oh);
        r.d16 = ldg<uint16_t>(seg, od);
      }
    }
#pragma unroll
    for (int cs = 0; cs < C; cs++) {
      const uint8_t *x = xt + ((size_t)cs * nb + b) * kMidXTile;
#pragma unroll
      for (int g = 0; g < KL; g++) r.B[g][cs] = ldg<uint4>(x + 1024 * g, ox);
      if constexpr (Q4) r.bm[cs] = ldg<uint4>(x, ob);
      r.dx[cs] = ldg<float>(x, ods);
    }
    return r;
  };
  // block b's products from its weights v and activations r; block b + 1's
  // weights (rn) are put in place meanwhile
  MidW<KL, Q4> v;
  auto compute = [&](const MidRaw<C, KL, Q4, TILE> &r, const MidRaw<C, KL, Q4, TILE> &rn) {
    const MidW<KL, Q4> vn = mid_place(rn, n, q, l0);
    half8 a[KL], odd[KL], mins;
    float dw, dmw = 0.0f;
    if constexpr (Q4) {
      const uint4 hdr = row_gather(v.hdr);
      const uint32_t sclo = hdr.y & 0x3F3F3F3Fu;
      const uint32_t schi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
      const uint32_t sc = ((sclo & mq.lo) | (schi & ~mq.lo)) >> (16 * (q & 1));
      const half2v S0 = dup_byte(sc, 0, 1024.0f), S1 = dup_byte_16th(sc, 1);
      const half2v m1024 = (half2v){(_Float16)-1024.0f, (_Float16)-1024.0f};
      const half2v N0 = S0 * m1024, N1 = S1 * m1024;
#pragma unroll
      for (int g = 0; g < KL; g++) {
        const uint32_t d0 = v.ql[g], d8 = d0 >> 8;
        a[g] = cat(fma2(magic_nib<kNibLo>(d0, exp), S0, N0), fma2(magic_nib<kNibLo>(d8, exp), S0, N0),
                   fma2(magic_nib<kNibHi>(d0, exp), S1, N1), fma2(magic_nib<kNibHi>(d8, exp), S1, N1));
      }
      // sumi by one MFMA: quarter q < 2 carries k = 8q + e -> (j = 4q + e/2, half e%2)
      const uint32_t mn0 = hdr.z & 0x3F3F3F3Fu, mn1 = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
      const uint32_t mn = (mn0 & mq.q0) | (mn1 & mq.q1);
      mins = cat(dup_byte(mn, 0, 1024.0f), dup_byte(mn, 1, 1024.0f), dup_byte(mn, 2, 1024.0f),
                 dup_byte(mn, 3, 1024.0f));
      dw = h2f_bits(hdr.x & 0xFFFFu);
      dmw = h2f_bits(hdr.x >> 16);
    } else {
      half2v S[2];
      uint32_t M[2];
      q6_split_scales(S, M, v.gs);
      const int jj = 2 * (q & 1);
#pragma unroll
      for (int g = 0; g < KL; g++) {
        const uint32_t ql = v.ql[g], qh = v.qh[g] ^ (TILE ? 0xAAAAAAAAu : 0u);
        const uint32_t lo = (ql & 0x0F0F0F0Fu) | (((qh >> (2 * jj)) & 0x03030303u) << 4);
        const uint32_t hi = ((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (2 * jj + 2)) & 0x03030303u) << 4);
        q6_split(a[g], odd[g], lo, hi, S, M);
      }
      dw = h2f_bits(v.d16);
    }
    f32x4 D[KL][C], sm[C];
    const f32x4 zero = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int cs = 0; cs < C; cs++) {
#pragma unroll
      for (int g = 0; g < KL; g++) D[g][cs] = mfma(__builtin_bit_cast(half8, r.B[g][cs]), a[g], zero);
      if constexpr (Q4) sm[cs] = mfma(__builtin_bit_cast(half8, r.bm[cs]), mins, zero);
    }
    if constexpr (!Q4) {
#pragma unroll
      for (int cs = 0; cs < C; cs++)
#pragma unroll
        for (int g = 0; g < KL; g++) D[g][cs] = mfma(__builtin_bit_cast(half8, r.B[g][cs]), odd[g], D[g][cs]);
    }
#pragma unroll
    for (int cs = 0; cs < C; cs++) {
      const float dx[4] = {quad_lane<0>(r.dx[cs]), quad_lane<1>(r.dx[cs]), quad_lane<2>(r.dx[cs]),
                           quad_lane<3>(r.dx[cs])};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float dd = __fmul_rn(dw, dx[j]);
#pragma unroll
        for (int g = 0; g < KL; g++) s[g][cs][j] = __fadd_rn(s[g][cs][j], __fmul_rn(dd, D[g][cs][j]));
      }
      if constexpr (Q4) f[cs] = __fsub_rn(f[cs], __fmul_rn(__fmul_rn(dmw, dx[0]), sm[cs][0]));
    }
    v = vn;
  };
  MidRaw<C, KL, Q4, TILE> r[PD];
  // the scheduling barriers keep the loads in block order: the first wait in
  // the loop would otherwise be for all of them
#pragma unroll
  for (int i = 0; i < PD; i++) {
    r[i] = load(i);
    __builtin_amdgcn_sched_barrier(0);
  }
  v = mid_place(r[0], n, q, l0);
  // (blocks past the last are skipped by a branch around them: an exit inside
  // the loop would join its back edge, and the waits at its head would then be
  // for every load)
  for (int b0 = 0; b0 < nb; b0 += PD) {
#pragma unroll
    for (int i = 0; i < PD; i++) {
      if (b0 + i < nb) compute(r[i], r[(i + 1) % PD]);
      r[i] = load(b0 + i + PD);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// PAIR: eight waves, segment tt of gate (waves 0-3) and of up (4-7); their
// totals meet in the final sum, which stores fround(gelu(gate) * up).
// TILE: every weight is read from its tiles (a launch with a weight kept in
// one layout); else from its segments.
template <int C, int KL, bool PAIR, bool TILE>
__global__ __launch_bounds__(512 / KL * (PAIR ? 2 : 1)) __attribute__((amdgpu_waves_per_eu(C == 1 ? 3 : 2))) void
kquant_mid_kernel(const MidArgs a) {
  kernarg_warm<MidArgs>();
  constexpr int cols = 16 * C, kChain = cols * kMidRowPad;
  __shared__ float fin[(PAIR ? 2 : 1) * 9 * kChain];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int kThreads = 512 / KL;  // of a segment
  const int grp = PAIR ? wave / (8 / KL) : 0, w = wave & (8 / KL - 1);
  // the column groups of a segment are 8 workgroups apart: one XCD, whose L2
  // holds the segment's weights for all of them
  const int G = a.col_groups, tg = blockIdx.x / (8 * G), rem = blockIdx.x - tg * 8 * G;
  const int t = 8 * tg + (rem & 7), cg = rem >> 3;
  if (t >= a.total_tiles) return;
  MidWeight W = a.w[0];
  if (PAIR) {
    if (grp) W = a.w[1];
  } else {
    if (a.count > 1 && t >= a.w[1].tile_begin) W = a.w[1];
    if (a.count > 2 && t >= a.w[2].tile_begin) W = a.w[2];
    if (a.count > 3 && t >= a.w[3].tile_begin) W = a.w[3];
  }
  const int tt = PAIR ? t : t - W.tile_begin;
  float s[KL][C][4], f[C];
#pragma unroll
  for (int cs = 0; cs < C; cs++) {
    f[cs] = 0.0f;
#pragma unroll
    for (int g = 0; g < KL; g++)
#pragma unroll
      for (int j = 0; j < 4; j++) s[g][cs][j] = 0.0f;
  }
  const uint8_t *xt = group_tiles<C>(a.xt, cg, a.nb);
  if (W.type == kTypeQ4K)
    mid_tile<C, KL, true, TILE>(s, f, W, tt, a.nb, a.S, a.R, xt, w, lane);
  else
    mid_tile<C, KL, false, TILE>(s, f, W, tt, a.nb, a.S, a.R, xt, w, lane);
  {
    const int n = lane & 15, q = lane >> 4;
    float *fg = fin + grp * 9 * kChain + n;
#pragma unroll
    for (int cs = 0; cs < C; cs++) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int col = 16 * cs + 4 * q + ((j + w) & 3);
#pragma unroll
        for (int g = 0; g < KL; g++) fg[(KL * w + g) * kChain + col * kMidRowPad] = s[g][cs][j];
        if (j == 0 && w < 4) fg[8 * kChain + col * kMidRowPad] = f[cs];
      }
    }
  }
  __syncthreads();
  // the chains of one output in class order, then [sumf +]
  auto total = [&](int g, bool q4, int row, int col) {
    const float *p = fin + g * 9 * kChain + col * kMidRowPad + row;
    float v = -0.0f;
#pragma unroll
    for (int l = 0; l < 8; l++) v = __fadd_rn(v, p[l * kChain]);
    return q4 ? __fadd_rn(p[8 * kChain], v) : v;
  };
  const int row16 = tid & 15, row = 16 * tt + row16;
  if constexpr (PAIR) {
    const bool q4g = a.w[0].type == kTypeQ4K, q4u = a.w[1].type == kTypeQ4K;
    const int rows = a.w[0].rows;
    for (int col = tid >> 4; col < cols; col += kThreads / 8) {
      const int m = cols * cg + col;
      if (row < rows && m < a.cols)
        a.pair_out[(size_t)m * rows + row] = geglu_lut(total(0, q4g, row16, col), total(1, q4u, row16, col), a.gelu_lut);
    }
  } else {
    for (int col = tid >> 4; col < cols; col += kThreads / 16) {
      const int m = cols * cg + col;
      const float v = total(0, W.type == kTypeQ4K, row16, col);
      if (row < W.rows && m < a.cols) W.out[(size_t)m * W.rows + row] = v;
    }
  }
}

template <int C, int KL, bool PAIR>
void launch_mid_kernel(MidArgs a, bool tiles, hipStream_t s) {
  a.col_groups = (a.cols + 16 * C - 1) / (16 * C);
  if (PAIR) a.total_tiles = a.w[0].tiles;
  auto *k = tiles ? kquant_mid_kernel<C, KL, PAIR, true> : kquant_mid_kernel<C, KL, PAIR, false>;
  hipLaunchKernelGGL(k, dim3((a.total_tiles + 7) / 8 * 8 * a.col_groups), dim3(512 / KL * (PAIR ? 2 : 1)), 0, s, a);
}

// ---- row waves: launches with many segments ---------------------------------
//
// With several segments to every SIMD (gate/up 1280, the head 16384) the walk
// along a row no longer bounds the launch; instructions per weight and the
// restart of the loads at each segment do.  So here a wave owns a whole
// segment (all eight classes and the min chain: one header, no exchange of
// chains), a workgroup of up to kRowWaves computing waves shares one ring, and
// a workgroup walks its items without a break: the weight loads and activation
// copies of the next item are issued during the current one's last blocks.
// All weights of such a launch have one type.  PAIR: the first half of the
// computing waves take segments of gate, the second half the same of up.
// One block's activation tiles of a column group in LDS, set after set.
constexpr int mid_stage(int C) { return C * kMidXTile; }
// Stages in the ring.  A tile was written by the previous launch, so its first
// read on each XCD comes from beyond the L2 (about 2000 clocks).
constexpr int mid_ring(int C) { return C == 1 ? 10 : 7; }

// A use of v's registers at this point of the program (no instruction).
__device__ __forceinline__ void pin(uint4 &v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }

// s_waitcnt immediates (vmcnt in bits 3:0 and 15:14, lgkmcnt in 11:8).
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }
constexpr int kWaitLgkm0 = 0xC07F;

// Workgroup barrier without the waits of __syncthreads (weight loads stay in
// flight across it); memory operations are not moved past it.
__device__ __forceinline__ void mid_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

constexpr int kMidCopiers = 2;

// Waits until at most n (0 <= n <= N) steps' copies, PER of them each, are in flight.
template <int N, int PER>
__device__ __forceinline__ void mid_wait(int n) {
  if (n >= N) {
    __builtin_amdgcn_s_waitcnt(wait_vm(N * PER));
    return;
  }
  if constexpr (N > 0) mid_wait<N - 1, PER>(n);
}

// A copying wave (P of kMidCopiers) of a workgroup that walks items it =
// blockIdx.x, + gridDim.x, ... below `items`: step k (block k % nb of item k /
// nb, whose column group is item % col_groups) into stage k % NB, NB - 1 steps
// ahead, with direct global->LDS loads of 1 KB.  item_barrier: one more barrier
// ends each item.
template <int C, int P>
__device__ __forceinline__ void mid_copy(const uint8_t *xt, int nb, int items, int col_groups, bool item_barrier,
                                         uint8_t *ring, int lane) {
  constexpr int NB = mid_ring(C), kAll = (mid_stage(C) + 1023) / 1024;  // 1 KB copies per block, the last a part
  constexpr int kPer = (kAll - P + kMidCopiers - 1) / kMidCopiers;       // of this wave
  static_assert((NB - 2) * kPer < 64, "vmcnt range");
  int left = (items - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x * nb;  // steps not yet copied
  int ahead = 0;                                                                     // steps copied and not yet waited for
  int cit = blockIdx.x, cb = 0;  // the next copy's item and block
  uint8_t *dst = ring;
  auto copy = [&]() {
    const uint8_t *src = group_tiles<C>(xt, cit % col_groups, nb) + (size_t)cb * kMidXTile;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      // stage byte o: byte o % kMidXTile of set o / kMidXTile's tile
      const int o = 1024 * (kMidCopiers * j + P) + 16 * lane, cs = o / kMidXTile;
      const uint8_t *from = src + (size_t)cs * nb * kMidXTile + (o - cs * kMidXTile);
      if (o < mid_stage(C))
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const void *>(from),
                                         (__attribute__((address_space(3))) void *)(dst + 1024 * (kMidCopiers * j + P)),
                                         16, 0, 0);
    }
    dst = dst == ring + (NB - 1) * mid_stage(C) ? ring : dst + mid_stage(C);
    left--;
    ahead++;
    if (++cb == nb) {
      cit += gridDim.x;
      cb = 0;
    }
  };
  for (int i = 0; i < NB - 1 && left > 0; i++) copy();
  for (int it = blockIdx.x; it < items; it += gridDim.x) {
    for (int b = 0; b < nb; b++) {
      mid_wait<NB - 2, kPer>(--ahead);  // the step's copies have landed
      mid_barrier();                    // and the step before is read
      if (left > 0) copy();
    }
    if (item_barrier) mid_barrier();
  }
}

constexpr int row_waves(int C) { return C == 1 ? 8 : 6; }
// Blocks of weights in registers (a third of Q6_K's 18 registers, or of the
// tiles' with their addresses, would spill).
constexpr int row_depth(int C, bool q4, bool tile) { return C == 1 && q4 && !tile ? 3 : 2; }

template <int C, bool Q4, bool PAIR, bool TILE>
__global__ __launch_bounds__(64 * (row_waves(C) + kMidCopiers)) void kquant_rows_kernel(const MidArgs a) {
  kernarg_warm<MidArgs>();
  extern __shared__ __align__(16) uint8_t smem[];
  constexpr int NB = mid_ring(C), PD = row_depth(C, Q4, TILE), segb = Q4 ? 2304 : 3360, cols = 16 * C;
  const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = (int)(blockDim.x >> 6) - kMidCopiers, nb = a.nb;
  if (wave >= nw) {
    if (wave == nw)
      mid_copy<C, 0>(a.xt, nb, a.items, a.col_groups, PAIR, smem, lane);
    else
      mid_copy<C, 1>(a.xt, nb, a.items, a.col_groups, PAIR, smem, lane);
    return;
  }
  const int per = PAIR ? nw >> 1 : nw;  // segments of an item (of each of gate and up)
  const bool up = PAIR && wave >= per;
  const int my = up ? wave - per : wave;
  const uint32_t exp = magic_nib_exp();
  const QuarterMasks mq = quarter_masks(q);
  // this wave's segment of an item (one past the last re-reads the last, and is never stored)
  auto weight_of = [&](int it, int &tt) {
    const int t = min(it / a.col_groups * per + my, a.total_tiles - 1);
    MidWeight W = a.w[0];
    if (PAIR) {
      if (up) W = a.w[1];
    } else {
      if (a.count > 1 && t >= a.w[1].tile_begin) W = a.w[1];
      if (a.count > 2 && t >= a.w[2].tile_begin) W = a.w[2];
      if (a.count > 3 && t >= a.w[3].tile_begin) W = a.w[3];
    }
    tt = t - (PAIR ? 0 : W.tile_begin);
    return W;
  };
  // the next load's item and block (past the last step it repeats the last block)
  int lit = blockIdx.x, lb = 0, ltt;
  MidWeight LW = weight_of(lit, ltt);
  F3Row fr{};
  if constexpr (TILE) fr = f3_row<Q4>(min(16 * ltt + n, LW.rows - 1), LW.rows, nb, a.S, a.R, q);
  auto load = [&](typename WSel<Q4>::T &r) {
    if constexpr (TILE) {
      int bi, bs;
      block_split(lb, a.S, bi, bs);
      f3_wload_tile<Q4>(r, LW.wt, LW.dplane, fr, bi, bs, q);
    } else {
      f3_wload_seg<Q4>(r, LW.seg + ((size_t)lb * LW.tiles + ltt) * segb, lane);
    }
    if (++lb == nb) {
      if (lit + (int)gridDim.x < a.items) {
        lit += gridDim.x;
        lb = 0;
        LW = weight_of(lit, ltt);
        if constexpr (TILE) fr = f3_row<Q4>(min(16 * ltt + n, LW.rows - 1), LW.rows, nb, a.S, a.R, q);
      } else {
        lb = nb - 1;
      }
    }
  };
  typename WSel<Q4>::T r[PD];
#pragma unroll
  for (int i = 0; i < PD; i++) {
    load(r[i]);
    __builtin_amdgcn_sched_barrier(0);  // in block order, so that the first wait is for the first block
  }
  float s[8][C][4], f[C][4];
  auto clear = [&]() {
#pragma unroll
    for (int cs = 0; cs < C; cs++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        f[cs][j] = 0.0f;
#pragma unroll
        for (int l = 0; l < 8; l++) s[l][cs][j] = 0.0f;
      }
  };
  clear();
  const uint8_t *st = smem;
  int it = blockIdx.x, b = 0;
  // one block; the item's totals after its last
  auto step = [&](typename WSel<Q4>::T &rw) {
    // nothing made from the block's registers moves up into the loop's latch,
    // where its wait would be for every load
    if constexpr (Q4) {
      pin(rw.hdr);
      pin(rw.qa[0]);
      pin(rw.qa[1]);
    }
    // scales and quants of the block, before its stage is waited for
    half2v S[2], N[2];
    uint32_t odd[2], qd[2][4];
    float dw, dmw = 0.0f;
    half8 mins;
    if constexpr (Q4) {
      const uint4 hdr = rw.hdr;
      const uint32_t sclo = hdr.y & 0x3F3F3F3Fu;
      const uint32_t schi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
      const uint32_t sc = ((sclo & mq.lo) | (schi & ~mq.lo)) >> (16 * (q & 1));
      S[0] = dup_byte(sc, 0, 1024.0f);
      S[1] = dup_byte_16th(sc, 1);
      const half2v m1024 = (half2v){(_Float16)-1024.0f, (_Float16)-1024.0f};
      N[0] = S[0] * m1024;
      N[1] = S[1] * m1024;
      const uint32_t mn0 = hdr.z & 0x3F3F3F3Fu, mn1 = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
      const uint32_t mn = (mn0 & mq.q0) | (mn1 & mq.q1);
      mins = cat(dup_byte(mn, 0, 1024.0f), dup_byte(mn, 1, 1024.0f), dup_byte(mn, 2, 1024.0f),
                 dup_byte(mn, 3, 1024.0f));
      dw = h2f_bits(hdr.x & 0xFFFFu);
      dmw = h2f_bits(hdr.x >> 16);
    } else {
      q6_split_scales(S, odd, rw.gs);
      dw = h2f_bits(rw.d16);
    }
#pragma unroll
    for (int g = 0; g < 2; g++) {
      if constexpr (TILE) {
#pragma unroll
        for (int t = 0; t < 4; t++) qd[g][t] = u4at(rw.qa[t >> 1], 2 * (t & 1) + g);
      } else {
        const uint4 v = rw.qa[g];
        qd[g][0] = v.x;
        qd[g][1] = v.y;
        qd[g][2] = v.z;
        qd[g][3] = v.w;
        f3_transpose(qd[g]);
      }
    }
    mid_barrier();  // the step's stage is complete
    f32x4 dx[C];
    float dd[C][4];
#pragma unroll
    for (int cs = 0; cs < C; cs++) {
      dx[cs] = *reinterpret_cast<const f32x4 *>(st + cs * kMidXTile + 8704 + 16 * q);
#pragma unroll
      for (int j = 0; j < 4; j++) dd[cs][j] = __fmul_rn(dw, dx[cs][j]);
    }
    // class l's MFMAs run while class l + 1 is unpacked and class l - 1
    // enters its chains; its activations are read two classes ahead
    half8 B[3][C], A, Al;
    f32x4 D[2][C];
    auto bread = [&](int l) {
#pragma unroll
      for (int cs = 0; cs < C; cs++)
        B[l % 3][cs] = __builtin_bit_cast(
            half8, *reinterpret_cast<const uint4 *>(st + cs * kMidXTile + ((l * 4 + q) * 16 + n) * 16));
    };
    auto unpack = [&](int l) {
      if constexpr (Q4)
        A = f3_a<true, TILE>(rw, qd, l, q, S, N, exp);
      else
        f3_a6_split<TILE>(A, Al, rw, qd, l, q, S, odd);
    };
    auto chain = [&](int l) {
#pragma unroll
      for (int cs = 0; cs < C; cs++)
#pragma unroll
        for (int j = 0; j < 4; j++) s[l][cs][j] = __fadd_rn(s[l][cs][j], __fmul_rn(dd[cs][j], D[l & 1][cs][j]));
    };
    bread(0);
    bread(1);
    unpack(0);
#pragma unroll
    for (int l = 0; l < 8; l++) {
      if (l + 2 < 8) bread(l + 2);
#pragma unroll
      for (int cs = 0; cs < C; cs++) {
        D[l & 1][cs] = mfma(B[l % 3][cs], A, (f32x4){0.0f, 0.0f, 0.0f, 0.0f});
        if constexpr (!Q4) D[l & 1][cs] = mfma(B[l % 3][cs], Al, D[l & 1][cs]);
      }
      if (l < 7) unpack(l + 1);
      if (l > 0) chain(l - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    chain(7);
    if constexpr (Q4) {
      // sumi by one MFMA: quarter q < 2 carries k = 8q + e -> (j = 4q +
      // e/2, half e%2); quarters 2, 3 meet zero mins
#pragma unroll
      for (int cs = 0; cs < C; cs++) {
        const half8 bm = __builtin_bit_cast(
            half8, *reinterpret_cast<const uint4 *>(st + cs * kMidXTile + 8192 + ((q & 1) * 16 + n) * 16));
        const f32x4 sm = mfma(bm, mins, (f32x4){0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
        for (int j = 0; j < 4; j++)
          f[cs][j] = __fsub_rn(f[cs][j], __fmul_rn(__fmul_rn(dmw, dx[cs][j]), sm[j]));
      }
    }
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);  // this stage is read: the next barrier lets it be refilled
    st = st == smem + (NB - 1) * mid_stage(C) ? smem : st + mid_stage(C);
    if (++b < nb) return;
    // the item's totals: the chains in class order, then [sumf +]
    int tt;
    const MidWeight W = weight_of(it, tt);
    const int row = 16 * tt + n, cg = it % a.col_groups;
    const bool live = it / a.col_groups * per + my < a.total_tiles && row < W.rows;
    float *xch = reinterpret_cast<float *>(smem + NB * mid_stage(C)) + my * C * 256 + lane;
#pragma unroll
    for (int cs = 0; cs < C; cs++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float t = -0.0f;
#pragma unroll
        for (int l = 0; l < 8; l++) t = __fadd_rn(t, s[l][cs][j]);
        if constexpr (Q4) t = __fadd_rn(f[cs][j], t);
        if constexpr (PAIR) {
          if (up) xch[(cs * 4 + j) * 64] = t;
          s[0][cs][j] = t;
        } else {
          const int m = cols * cg + 16 * cs + 4 * q + j;
          if (live && m < a.cols) W.out[(size_t)m * W.rows + row] = t;
        }
      }
    if constexpr (PAIR) {
      __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      mid_barrier();
      if (!up) {
        // every table read before the first store
        float h[C][4];
#pragma unroll
        for (int cs = 0; cs < C; cs++)
#pragma unroll
          for (int j = 0; j < 4; j++) h[cs][j] = geglu_lut(s[0][cs][j], xch[(cs * 4 + j) * 64], a.gelu_lut);
#pragma unroll
        for (int cs = 0; cs < C; cs++)
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const int m = cols * cg + 16 * cs + 4 * q + j;
            if (live && m < a.cols) a.pair_out[(size_t)m * W.rows + row] = h[cs][j];
          }
        __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      }
    }
    clear();
    b = 0;
    it += gridDim.x;
  };
  int left = (a.items - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x * nb;
  for (; left > 0; left -= PD) {  // (no exit inside: see mid_tile)
#pragma unroll
    for (int i = 0; i < PD; i++) {
      if (i < left) step(r[i]);
      load(r[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

constexpr int row_lds(int C, bool pair, int nw) {
  return mid_ring(C) * mid_stage(C) + (pair ? nw / 2 * C * 1024 : 0);
}

template <int C, bool PAIR>
void launch_rows_kernel(MidArgs a, bool tiles, int num_cus, hipStream_t s) {
  const int gy = (a.cols + 16 * C - 1) / (16 * C);
  // computing waves per workgroup: as few as still give one item per CU
  int nw = row_waves(C);
  const int segs = PAIR ? 2 * a.w[0].tiles : a.total_tiles;
  while (nw > 4 && (segs + nw - 3) / (nw - 2) * gy <= num_cus) nw -= 2;
  const int per = PAIR ? nw / 2 : nw;
  if (PAIR) a.total_tiles = a.w[0].tiles;
  a.col_groups = gy;
  a.items = (a.total_tiles + per - 1) / per * gy;
  const bool q4 = a.w[0].type == kTypeQ4K;
  auto *k = q4 ? (tiles ? kquant_rows_kernel<C, true, PAIR, true> : kquant_rows_kernel<C, true, PAIR, false>)
               : (tiles ? kquant_rows_kernel<C, false, PAIR, true> : kquant_rows_kernel<C, false, PAIR, false>);
  hipLaunchKernelGGL(k, dim3(a.items < num_cus ? a.items : num_cus), dim3(64 * (nw + kMidCopiers)),
                     row_lds(C, PAIR, nw), s, a);
}

}  // namespace

size_t mid_bytes(int k, int cols) { return (size_t)(mid_pad_cols(cols) / kMidCols) * (k / kQK) * kMidXTile; }

size_t mid_lds_bytes() {
  const int r1 = row_lds(1, true, row_waves(1)), r2 = row_lds(2, true, row_waves(2));
  return r1 > r2 ? r1 : r2;
}

int mid_pad_cols(int cols) { return cols <= 16 ? 16 : (cols + 31) / 32 * 32; }

hipError_t launch_mid(const MfmaLaunch &l, const uint8_t *xt, const uint16_t *gelu_lut, float *pair_out, int num_cus,
                      hipStream_t s) {
  if (l.count < 1 || l.count > kMaxWeights || l.cols < 1 || l.k % kQK != 0 || !mfma_geometry_ok(l) ||
      (pair_out && (l.count != 2 || l.rows[0] != l.rows[1] || !gelu_lut)))
    return hipErrorInvalidValue;
  MidArgs a{};
  a.count = l.count;
  for (int i = 0; i < l.count; i++) {
    a.w[i].seg = l.seg[i];
    a.w[i].wt = l.wt[i];
    a.w[i].dplane = l.dplane[i];
    a.w[i].out = l.out[i];
    a.w[i].type = l.type[i];
    a.w[i].rows = l.rows[i];
    a.w[i].tiles = (l.rows[i] + 15) / 16;
    a.w[i].tile_begin = a.total_tiles;
    a.total_tiles += a.w[i].tiles;
  }
  a.nb = l.k / kQK;
  a.cols = l.cols;
  a.S = l.S;
  a.R = l.R;
  a.xt = xt;
  a.pair_out = pair_out;
  a.gelu_lut = gelu_lut;
  const bool tiles = launch_reads_tiles(l);
  // row waves from two segments of one type a CU on
  MidShape shape{};
  shape.segs = a.total_tiles;
  shape.cus = num_cus;
  for (int i = 0; i < l.count; i++) (l.type[i] == kTypeQ4K ? shape.q4 : shape.q6) = true;
  if (!mid_grid_fits(shape, l.cols)) return hipErrorInvalidValue;
  if (mid_row_waves(shape)) {
    if (pair_out && l.cols <= 16)
      launch_rows_kernel<1, true>(a, tiles, num_cus, s);
    else if (pair_out)
      launch_rows_kernel<2, true>(a, tiles, num_cus, s);
    else if (l.cols <= 16)
      launch_rows_kernel<1, false>(a, tiles, num_cus, s);
    else
      launch_rows_kernel<2, false>(a, tiles, num_cus, s);
    return hipGetLastError();
  }
  // class pairs; for long rows single classes, while a workgroup per segment
  // fits the CUs (down, 40 blocks, with its tile launch: 18.8 -> 17.1 us at 5
  // columns, 24.2 -> 21.0 at 21; Q/K/V and O, 10 and 8 blocks: 9.6 -> 9.7, 8.8 -> 9.1)
  const bool single = a.total_tiles <= num_cus && a.nb >= 20;
  if (!pair_out && single && l.cols <= 32) {
    if (l.cols <= 16)
      launch_mid_kernel<1, 1, false>(a, tiles, s);
    else
      launch_mid_kernel<2, 1, false>(a, tiles, s);
    return hipGetLastError();
  }
  // a workgroup per 16 columns while those fit the CUs three to each (three
  // groups of down 30.5 -> 25.1 us against two of 32), else per 32
  const bool narrow = l.cols <= 16 || (long long)a.total_tiles * ((l.cols + 15) / 16) <= 3 * num_cus;
  if (pair_out && narrow)
    launch_mid_kernel<1, 2, true>(a, tiles, s);
  else if (pair_out)
    launch_mid_kernel<2, 2, true>(a, tiles, s);
  else if (narrow)
    launch_mid_kernel<1, 2, false>(a, tiles, s);
  else
    launch_mid_kernel<2, 2, false>(a, tiles, s);
  return hipGetLastError();
}

}  // namespace hp
