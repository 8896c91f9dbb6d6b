// hp_wfrag.h -- a 16-row weight segment's block in a wave's registers and its
// f16 MFMA fragments of all eight lane classes, shared by the kernels in which
// one wave owns whole rows (the fast prefill kernel, kquant_prefill.hip, and
// the row waves of kquant_mid.hip).
#pragma once

#include "hp_common.h"
#include "hp_mfma.h"

namespace hp {

// One segment's weights in a lane's registers, loaded with 16- and 8-byte
// loads (few memory instructions), from one of two places:
//   segments (matrix-core layout): lane (n, r) holds unit n + 16r of chunk g,
//     dwords u = 0..3, and f3_transpose turns them into what the A fragments
//     take: lane (n, q) holds dword q of units n + 16t, t = 0..3 (class
//     l = 2t + g);
//   tiles (a weight kept in one layout, hp_common.h): lane (row n, quarter
//     q) takes the two quant chunks holding dwords D[q][l], l = 0..3 and
//     4..7, which are what its A fragments need (class l = 2t + g: dword
//     l % 4 of chunk l / 4), no transpose.
// Q4_K: row n's header (d | dmin, then the 12 bytes of 6-bit scales and
// mins) and the quants (qa[g] / qa[l / 4]).
struct W4 {
  uint4 hdr;
  uint4 qa[2];
};
// Q6_K: low-bit units or chunks as Q4_K's; high bits: for class l = 2t + g
// dword 2 (t % 2) + g of qh[t / 2] (segments: the two dwords of unit n + 16t
// for quarter pair q / 2; tiles: chunks 8 + 2h, 9 + 2h, h = q / 2, fields
// stored ^ 2); row n's scales 4q .. 4q + 3 and its d (f16 bits).
struct W6 {
  uint4 qa[2];
  uint4 qh[2];
  uint32_t gs, d16;
};
template <bool Q4>
struct WSel {
  using T = W6;
};
template <>
struct WSel<true> {
  using T = W4;
};

// A lane's offsets into one of its rows' row-blocks (tile_row) and the
// chunks it loads: oq = its first quant chunk, oh = its first high-bit chunk.
struct F3Row {
  TileRow tr;
  uint32_t oq, oh;
};

template <bool Q4>
__device__ __forceinline__ F3Row f3_row(int row, int rows, int nb, int S, int R, int q) {
  F3Row f;
  f.tr = tile_row(row, rows, nb, S, R, Q4 ? 9 : 13);
  f.oq = (uint32_t)(Q4 ? 1 + 2 * q : 2 * q) * f.tr.chunk;
  f.oh = (uint32_t)(8 + 2 * (q >> 1)) * f.tr.chunk;
  return f;
}

// Segment layouts of the matrix-core repack (kquant_mfma.hip): Q4_K [16 rows
// x 16-byte header][2 chunks x 64 units x 16 bytes of quants]; Q6_K [16 rows x
// 16 scales][16 x f16 d][2 chunks x 1024 low bits][1024 high bits].
template <bool Q4>
__device__ __forceinline__ void f3_wload_seg(typename WSel<Q4>::T &w, const uint8_t *seg, int lane) {
  const int n = lane & 15, q = lane >> 4;
  if constexpr (Q4) {
    w.hdr = *reinterpret_cast<const uint4 *>(seg + 16 * n);
#pragma unroll
    for (int g = 0; g < 2; g++) w.qa[g] = *reinterpret_cast<const uint4 *>(seg + 256 + 1024 * g + 16 * lane);
  } else {
    w.gs = *reinterpret_cast<const uint32_t *>(seg + 16 * n + 4 * q);
    w.d16 = *reinterpret_cast<const uint16_t *>(seg + 256 + 2 * n);
#pragma unroll
    for (int g = 0; g < 2; g++) w.qa[g] = *reinterpret_cast<const uint4 *>(seg + 288 + 1024 * g + 16 * lane);
    uint2 h[4];
#pragma unroll
    for (int t = 0; t < 4; t++) h[t] = *reinterpret_cast<const uint2 *>(seg + 2336 + 256 * t + 16 * n + 8 * (q >> 1));
    w.qh[0] = make_uint4(h[0].x, h[0].y, h[1].x, h[1].y);
    w.qh[1] = make_uint4(h[2].x, h[2].y, h[3].x, h[3].y);
  }
}

// 4 x 4 transpose across the wave's four 16-lane rows: in, lane (n, r) holds
// v[u] = element (r, u); out, lane (n, q) holds v[t] = element (t, q).
__device__ __forceinline__ void f3_transpose(uint32_t (&v)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  v[0] = c[0];
  v[1] = c[1];
  v[2] = d[0];
  v[3] = d[1];
}

// Block (bi, bs) = bi * S + bs of row f into w, from the tiles.
template <bool Q4>
__device__ __forceinline__ void f3_wload_tile(typename WSel<Q4>::T &w, const uint8_t *wt, const uint16_t *dplane,
                                              const F3Row &f, int bi, int bs, int q) {
  const uint32_t off = f.tr.base + (uint32_t)bi * f.tr.iter + 16u * (uint32_t)bs;
  auto ld16 = [&](uint32_t o) { return *reinterpret_cast<const uint4 *>(wt + o); };
  w.qa[0] = ld16(off + f.oq);
  w.qa[1] = ld16(off + f.oq + f.tr.chunk);
  if constexpr (Q4) {
    w.hdr = ld16(off);
  } else {
    w.qh[0] = ld16(off + f.oh);
    w.qh[1] = ld16(off + f.oh + f.tr.chunk);
    w.gs = *reinterpret_cast<const uint32_t *>(wt + off + 12u * f.tr.chunk + 4u * (uint32_t)q);
    w.d16 = dplane[f.tr.dbase + (uint32_t)bi * f.tr.diter + (uint32_t)bs];
  }
}

// Weight fragment of class l = 2t + g (sc * q as exact f16); qd[g][t] are the
// quant dwords D[q][l].  Element order: bytes 0, 2, 1, 3 of the dword's
// low nibbles (or low 6-bit values), then the same of its high ones -- the
// activation tiles store their runs the same way.  Q4_K: (S[0], N[0]) scale
// the low nibbles, (S[1], N[1]) the high ones as 16 q (their scale / 16).
// Q6_K: S[0] = (s0, s1) for the low values, S[1] = (s2, s3) for the high.
template <bool Q4, bool TILE>
__device__ __forceinline__ half8 f3_a(const typename WSel<Q4>::T &w, const uint32_t (&qd)[2][4], int l, int q,
                                      const half2v (&S)[2], const half2v (&N)[2], uint32_t exp) {
  const int g = l & 1, t = l >> 1;
  if constexpr (Q4) {
    const uint32_t dw = qd[g][t], d8 = dw >> 8;
    return cat(fma2(magic_nib<kNibLo>(dw, exp), S[0], N[0]), fma2(magic_nib<kNibLo>(d8, exp), S[0], N[0]),
               fma2(magic_nib<kNibHi>(dw, exp), S[1], N[1]), fma2(magic_nib<kNibHi>(d8, exp), S[1], N[1]));
  } else {
    const int jj = 2 * (q & 1);
    // the tiles store the fields as hi ^ 2
    const uint32_t ql = qd[g][t], qh = u4at(w.qh[t >> 1], 2 * (t & 1) + g) ^ (TILE ? 0xAAAAAAAAu : 0u);
    const uint32_t lo = (ql & 0x0F0F0F0Fu) | (((qh >> (2 * jj)) & 0x03030303u) << 4);
    const uint32_t hi = ((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (2 * jj + 2)) & 0x03030303u) << 4);
    return cat(fma2(magic_pair<kSel02>(lo), S[0], N[0]), fma2(magic_pair<kSel13>(lo), S[0], N[0]),
               fma2(magic_pair<kSel02>(hi), S[1], N[1]), fma2(magic_pair<kSel13>(hi), S[1], N[1]));
  }
}

// Q6_K weights whose scales reach beyond what one f16 holds exactly (an odd
// scale of 67 and more against an odd q - 32; hp_mfma.h): the fragment as two
// exact ones, (sc & ~1) * (q - 32), at most 4096 and even, and (sc & 1) *
// (q - 32).  S are the even parts (pairs as f3_a's), M the odd bits as masks.
// Costs twice the MFMAs and 8 more vector-ALU instructions per fragment; the
// vector-ALU kernels these weights took before re-read them every 8 columns:
// three layers over 512 tokens 14.65 -> 0.88 ms, over 150 tokens 4.42 -> 0.44.
template <bool TILE>
__device__ __forceinline__ void f3_a6_split(half8 &hi8, half8 &lo8, const W6 &w, const uint32_t (&qd)[2][4], int l,
                                            int q, const half2v (&S)[2], const uint32_t (&M)[2]) {
  const int g = l & 1, t = l >> 1, jj = 2 * (q & 1);
  const uint32_t ql = qd[g][t], qh = u4at(w.qh[t >> 1], 2 * (t & 1) + g) ^ (TILE ? 0xAAAAAAAAu : 0u);
  const uint32_t lo = (ql & 0x0F0F0F0Fu) | (((qh >> (2 * jj)) & 0x03030303u) << 4);
  const uint32_t hi = ((ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (2 * jj + 2)) & 0x03030303u) << 4);
  q6_split(hi8, lo8, lo, hi, S, M);
}

}  // namespace hp
