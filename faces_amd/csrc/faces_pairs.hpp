// faces_pairs.hpp -- one work item of the DSS step moved in 16-byte pairs: S
// or fewer consecutive elements of one element row, loaded into LDS, summed
// and stored back by one block (load width 3 of the one-item kernel, and the
// batched step's item).
//
// The item owns the lower-corner nodes (ix, iy, iz < n-1) of its elements;
// the copies of those nodes form its footprint: its own planes iz < n-1 (but
// for the x-rows iy = n-1), the x-rows iy = n-1 of those planes in the row
// jy-1 (y), plane iz = n-1 of the row (jy, jz-1) (z; yz its x-row iy = n-1 in
// the row (jy-1, jz-1)), and the seam, the column ix = n-1 of the element
// before it in the four rows.  Its last element's column ix = n-1 is the next
// item's.  Every field location belongs to exactly one item.
//
// Layout in LDS.  The four regions fill each other's gaps: an element's
// copies lie at their own offsets inside the element, so that the element
// takes n^3 doubles, a double's LDS position is its offset from the item's
// start, and a node's copies lie at fixed distances from the node -- (n-1)*n
// for y, (n-1)*n^2 for z, n-1 minus an element for x -- which the LDS
// instructions carry as immediate offsets.  The seam follows as n^2 doubles.
//
// What bounds it.  Blocks are short (one item, dispatched in memory order:
// walking several items per block is slower, the more the longer), 8 waves
// per SIMD, and a wave waits for its turn to issue for half its life, so
// instructions count as much as bytes for small n: slots of a wave lie in one
// region (regions start on multiples of 64), their indices come from 24-bit
// multiplications, and nodes are taken class by class (faces, edges, corners)
// so that a wave mostly runs one class's loads and stores.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "faces_stream.hpp"

namespace faces {

// u / D for u < 4096, by a 24-bit multiplication (full rate; the 32-bit
// high product of a general division by a constant takes four times as long).
// D < 16: M = ceil(2^18 / D), u * (M*D - 2^18) < 4096 * 16 < 2^18; else M =
// ceil(2^24 / D) <= 2^20, u * (M*D - 2^24) < 4096 * D, which is below 2^24
// for D < 4096.
template <int D>
__device__ __forceinline__ unsigned div24(unsigned u)
{
  static_assert(D >= 1 && D < 4096, "divisor");
  if constexpr (D == 1) {
    return u;
  } else {
    constexpr int sh = D < 16 ? 18 : 24;
    constexpr unsigned M = ((1u << sh) + D - 1) / D;
    return __umul24(u, M) >> sh;
  }
}

// Pair slots of an item of S elements of n^3 points, the regions' starts on
// multiples of 64 (the counts explained in pairs_item).
constexpr int pair_slots(int n, int S)
{
  const int K = n - 1, LP = K > 1 ? n / 2 : 0, XP = (n + 1) / 2, RP = K * n / 2;
  auto up64 = [](int v) { return (v + 63) / 64 * 64; };
  return up64((S - 1) * K * RP + K * K * LP) + up64((S - 1) * K * XP + K * LP) + up64((S - 1) * RP + K * LP) +
         (S - 1) * XP + LP;
}

template <int N, int S>
struct PairShape {
  static constexpr int n3 = N * N * N;
  static constexpr int rS = S * n3;             // LDS position of the seam
  static constexpr int P = (rS + N * N + 1) / 2 * 2;  // LDS doubles
  static constexpr int kMarkWords = (P + 31) / 32;
};

// The four element rows of an item (their starts, jx = 0), whose copies its
// nodes have: own (jy, jz), y (jy-1, jz), z (jy, jz-1), yz (jy-1, jz-1).
struct ItemRows {
  double *own, *y, *z, *yz;
  unsigned bytes;  // of a row
};

// One item: elements [jx0, jx0 + count) of the rows R, count <= S; jxs the element
// before them (the last one for jx0 = 0).  MODE, TREE: as in faces_flow.hpp
// (modes 0 to 2); surf: axes (bit 0 x) on which the item holds the rank
// surface.  T threads; lds: PairShape::P doubles, and for MODE 1 kMarkWords
// words after them.
template <int N, int S, int T, int MODE, int TREE>
__device__ __forceinline__ void pairs_item(const ItemRows R, int jx0, int count, int jxs, unsigned surf, int nbr_mask,
                                           double *lds)
{
  using SH = PairShape<N, S>;
  constexpr int n = N, K = N - 1, K1 = K > 1 ? K - 1 : 0, n2 = N * N;
  constexpr unsigned n3 = (unsigned)(N * N * N);
  constexpr unsigned kOOB = kOobBase;
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  const unsigned tid = threadIdx.x;
  const unsigned wave0 = __builtin_amdgcn_readfirstlane(tid & ~63u);

  // ---- pair slots.  Owned runs, each cut into pairs from its start (a pair
  // may start on any double): per element but the last one of (n-1)*n doubles
  // per own plane and in the z plane, one of n per plane of the y row and in
  // the yz row; per last element one of n-1 per x-row.  The last pair of an
  // odd run starts one double early, on the last double of the pair before
  // it: both move the same value.  (n = 2: the last element's runs are
  // singles.)
  constexpr unsigned RP = (K * n) / 2, PNL = K * RP;          // own: pairs of a plane, of an element
  constexpr unsigned XP = (n + 1) / 2, LP = K > 1 ? n / 2 : 0;  // pairs of a whole x-row, of the last element's
  constexpr unsigned LP1 = LP > 0 ? LP : 1;
  auto xpos = [](unsigned i) { return n & 1 ? min(2 * i, (unsigned)n - 2) : 2 * i; };                // in a whole x-row
  auto lpos = [](unsigned i) { return K > 1 && (K & 1) ? min(2 * i, (unsigned)K - 2) : 2 * i; };  // in the last element's
  auto po = [](unsigned e) { return (e - 1) * PNL + K * K * LP; };
  auto py = [](unsigned e) { return (e - 1) * K * XP + K * LP; };
  auto pz = [](unsigned e) { return (e - 1) * RP + K * LP; };
  auto pw = [](unsigned e) { return (e - 1) * XP + LP; };
  auto up64 = [](unsigned v) { return (v + 63) / 64 * 64; };
  constexpr unsigned PY = up64(po(S)), PZ = PY + up64(py(S)), PW = PZ + up64(pz(S)), PE = PW + pw(S);
  constexpr int JR = (PE + T - 1) / T > 0 ? (PE + T - 1) / T : 1;
  static_assert(JR * T <= 4096 && PE == (unsigned)pair_slots(n, S), "div24, slots");
  const unsigned E = S == 1 ? 1u : (unsigned)count, e1 = E - 1, last = e1 * n3;
  const unsigned bytes = E * n3 * 8;  // of the item in each row
  unsigned xo[JR];  // byte offset from the item's start, in its row and in LDS; kOOB: no pair
  u32x4 wr[JR];
  // the row of a wave's slots from t0 on (addresses as numbers: a choice
  // among the members of R would keep R in scratch memory)
  const unsigned long own = (unsigned long)R.own, yrow = (unsigned long)R.y, zrow = (unsigned long)R.z,
                      yzrow = (unsigned long)R.yz;
  const unsigned rowbytes = R.bytes;
  auto pair_row = [=](unsigned t0) {
    const unsigned long p = t0 < PY ? own : t0 < PZ ? yrow : t0 < PW ? zrow : yzrow;
    return __builtin_amdgcn_make_buffer_rsrc((double *)p + (long)jx0 * n3, 0, (int)bytes, 0x00020000);
  };
#pragma unroll
  for (int j = 0; j < JR; j++) {
    const unsigned t0 = j * T + wave0, t = j * T + tid;
    if ((j + 1) * T > PE && t0 >= PE) {
      xo[j] = kOOB;
      continue;
    }
    unsigned x = 0, u, cnt, f;  // offset in the item; index in the region; pairs there; of whole elements
    if (t0 < PY) {
      u = t;
      cnt = po(E);
      f = e1 * PNL;
      const unsigned e = div24<PNL>(u), r = u - e * PNL, iz = div24<RP>(r);
      x = e * n3 + 2 * r + iz * n;
      if (t0 + 63 >= f) {
        const unsigned v = u - f, row = div24<LP1>(v & 4095u), z = div24<K>(row);
        if (u >= f) x = last + (row + z) * n + lpos(v - row * LP);
      }
    } else if (t0 < PZ) {
      u = t - PY;
      cnt = py(E);
      f = e1 * (K * XP);
      const unsigned run = div24<XP>(u), e = div24<K>(run);
      x = e * n3 + (run - e * K) * n2 + K * n + xpos(u - run * XP);
      if (t0 + 63 >= PY + f) {
        const unsigned v = u - f, row = div24<LP1>(v & 4095u);
        if (u >= f) x = last + row * n2 + K * n + lpos(v - row * LP);
      }
    } else if (t0 < PW) {
      u = t - PZ;
      cnt = pz(E);
      f = e1 * RP;
      const unsigned e = div24<RP>(u);
      x = e * n3 + K * n2 + 2 * (u - e * RP);
      if (t0 + 63 >= PZ + f) {
        const unsigned v = u - f, row = div24<LP1>(v & 4095u);
        if (u >= f) x = last + K * n2 + row * n + lpos(v - row * LP);
      }
    } else {
      u = t - PW;
      cnt = pw(E);
      f = e1 * XP;
      const unsigned e = div24<XP>(u);
      x = (u >= f ? last + lpos(u - f) : e * n3 + xpos(u - e * XP)) + K * n2 + K * n;
    }
    xo[j] = u < cnt ? x * 8 : kOOB;
    wr[j] = __builtin_amdgcn_raw_buffer_load_b128(pair_row(t0), xo[j], 0, 0);
  }

  // ---- singles: the seam; for n = 2 the last element's runs before it
  constexpr unsigned one = K == 1;
  constexpr unsigned QY = up64(one + K * K), QZ = QY + up64(one + K), QW = QZ + up64(one + K), QE = QW + one + 1;
  constexpr int JG = (QE + T - 1) / T;
  unsigned go[JG], gq[JG];  // byte offset in the row (kOOB: none), in LDS
  double wg[JG];
  auto single_row = [=](unsigned t0) {
    const unsigned long p = t0 < QY ? own : t0 < QZ ? yrow : t0 < QW ? zrow : yzrow;
    return __builtin_amdgcn_make_buffer_rsrc((double *)p, 0, (int)rowbytes, 0x00020000);
  };
#pragma unroll
  for (int j = 0; j < JG; j++) {
    const unsigned t0 = j * T + wave0, t = j * T + tid;
    if ((j + 1) * T > QE && t0 >= QE) {
      go[j] = kOOB;
      gq[j] = 0;
      continue;
    }
    unsigned u, x, q, cnt;  // index in the row's group; offset in its element, LDS position in the seam; all
    if (t0 < QY) {
      u = t;
      cnt = K * K;
      const unsigned iz = div24<K>((u - one) & 4095u), iy = u - one - iz * K;
      x = iz * n2 + iy * n + K;
      q = iz * n + iy;
    } else if (t0 < QZ) {
      u = t - QY;
      cnt = K;
      x = (u - one) * n2 + K * n + K;
      q = (u - one) * n + K;
    } else if (t0 < QW) {
      u = t - QZ;
      cnt = K;
      x = K * n2 + (u - one) * n + K;
      q = K * n + u - one;
    } else {
      u = t - QW;
      cnt = 1;
      x = K * n2 + K * n + K;
      q = K * n + K;
    }
    const bool run = one && u == 0;  // the last element's one double of this row
    if (run) x = last + (t0 < QY ? 0 : t0 < QZ ? K * n : t0 < QW ? K * n2 : K * n2 + K * n);
    go[j] = u < one + cnt ? (x + (unsigned)(run ? jx0 : jxs) * n3) * 8 : kOOB;
    gq[j] = (run ? x : SH::rS + q) * 8;
    wg[j] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(single_row(t0), go[j], 0, 0));
  }

  // ---- the shared nodes this thread sums (computed while the loads are in
  // flight), class by class: z faces (iz = 0 only), y faces, x faces; from
  // FB on, a multiple of 64, the edges yz, xz, xy and the corners.  np: byte
  // position of the node in LDS, its low bits cx, cy, cz (copies on both
  // sides of that axis); nq: of its x partner, low bit 0 set in the item's
  // first element, whose x partners are the seam's.
  constexpr unsigned FB = up64(3 * K1 * K1 * S);
  constexpr int NN = (FB + (3 * K1 + 1) * S + T - 1) / T;
  static_assert(NN * T <= 4096, "div24");
  constexpr unsigned kNone = 0xffffffffu;
  unsigned np[NN], nq[NN];
#pragma unroll
  for (int i = 0; i < NN; i++) {
    constexpr int KF = K1 * K1 > 0 ? K1 * K1 : 1, KE = K1 > 0 ? K1 : 1;
    unsigned k = i * T + tid;
    unsigned p, q = 0, f, e;  // position, the seam's, flags, element
    if (i * T + wave0 < FB) {
      const unsigned nf = E * (K1 * K1), c = (k >= nf ? 1u : 0u) + (k >= 2 * nf ? 1u : 0u);
      const unsigned r0 = k - c * nf;
      e = k < 3 * nf ? div24<KF>(r0) : E;
      const unsigned r = r0 - e * KF, a = div24<KE>(r & 4095u), b = r - a * KE;  // a + 1, b + 1: the face's indices
      p = c == 0 ? (a + 1) * n + b + 1 : c == 1 ? (a + 1) * n2 + b + 1 : (a + 1) * n2 + (b + 1) * n;
      q = (a + 1) * n + b + 1;
      f = 4u >> c;
    } else {
      k -= FB;
      const unsigned nd = E * K1, c = (k >= nd ? 1u : 0u) + (k >= 2 * nd ? 1u : 0u) + (k >= 3 * nd ? 1u : 0u);
      const unsigned r = k - c * nd, d = div24<KE>(r), b = r - d * KE + 1;
      e = c == 3 ? r : d;
      p = c == 0 ? b : c == 1 ? b * n : c == 2 ? b * n2 : 0;
      q = c == 1 ? b : c == 2 ? b * n : 0;
      f = c == 3 ? 7u : 7u ^ (1u << c);
    }
    p += e * n3;
    const bool first = e == 0;
    np[i] = e < E ? p * 8 | f : kNone;
    nq[i] = first ? (SH::rS + q) * 8 | 1u : (p - n3 + K) * 8;
  }

  char *const lb = reinterpret_cast<char *>(lds);
  auto L = [&](unsigned b) -> double & { return *reinterpret_cast<double *>(lb + b); };
#pragma unroll
  for (int j = 0; j < JR; j++) {
    if (xo[j] == kOOB) continue;
    const u32x2 lo = {wr[j][0], wr[j][1]}, hi = {wr[j][2], wr[j][3]};
    L(xo[j]) = __builtin_bit_cast(double, lo);
    L(xo[j] + 8) = __builtin_bit_cast(double, hi);
  }
#pragma unroll
  for (int j = 0; j < JG; j++)
    if (go[j] != kOOB) L(gq[j]) = wg[j];
  unsigned *const smark = reinterpret_cast<unsigned *>(lds + SH::P);
  if (MODE == 1 && surf) {
    for (unsigned w = tid; w < SH::kMarkWords; w += T) smark[w] = 0u;
  }
  __syncthreads();

  // ---- sums: x pairs, then y, then z (TREE 1: z, y, x); the sum goes to
  // every copy
  constexpr unsigned DY = K * n * 8, DZ = K * n2 * 8;    // y, z partners
  constexpr unsigned SY = K * 8, SZ8 = K * n * 8;        // of a seam double
#pragma unroll
  for (int i = 0; i < NN; i++) {
    if (np[i] == kNone) continue;
    const unsigned f = np[i] & 7u, p = np[i] & ~7u, q = nq[i] & ~7u;
    const bool first = nq[i] & 1u;
    const bool cx = f & 1u, cy = f & 2u, cz = f & 4u;
    const unsigned qy = q + (first ? SY : DY), qz = q + (first ? SZ8 : DZ), qyz = qy + (first ? SZ8 : DZ);
    if (MODE) {
      // a node whose x pair (the first element's only), y or z pair crosses
      // the rank surface
      const unsigned wrap = surf & ((f & 6u) | (first ? f & 1u : 0u));
      if (wrap) {
        if constexpr (MODE == 1) {
          // the surface sums': its copies are marked, and not stored here
          const unsigned at[8] = {p, q, p + DY, qy, p + DZ, qz, p + DY + DZ, qyz};
#pragma unroll
          for (int c = 0; c < 8; c++)
            if ((c & ~(int)f) == 0) atomicOr(&smark[at[c] >> 8], 1u << ((at[c] >> 3) & 31));
        }
        if constexpr (MODE == 2) {
          // Each side of the surface sums its copies, and those across it
          // where the rank has a neighbour on that side.  Copy sx | sy << 1 |
          // sz << 2, side 1 = the partner across that axis; copies the node
          // does not have read as the node.  Tree 1: the axes x and z
          // exchanged in the copy numbering, the flags, the split axes and
          // the neighbour mask, so that the levels below run z, y, x.
          const unsigned dy = cy ? DY : 0u, dz = cz ? DZ : 0u;
          const unsigned qb = cx ? q : p;
          const unsigned qdy = cy ? (cx && first ? SY : DY) : 0u, qdz = cz ? (cx && first ? SZ8 : DZ) : 0u;
          const unsigned c1 = qb, c2 = p + dy, c3 = qb + qdy, c4 = p + dz, c5 = qb + qdz, c6 = p + dy + dz,
                         c7 = qb + qdy + qdz;
          const unsigned pp[8] = {p, TREE ? c4 : c1, c2, TREE ? c6 : c3, TREE ? c1 : c4, c5, TREE ? c3 : c6, c7};
          auto swap = [](unsigned a) { return (a & 2u) | ((a & 1u) << 2) | ((a >> 2) & 1u); };
          const unsigned ft = TREE ? swap(f) : f, wt = TREE ? swap(wrap) : wrap;
          const int nbr = TREE ? (nbr_mask & 12) | ((nbr_mask & 3) << 4) | ((nbr_mask >> 4) & 3) : nbr_mask;
          double c[8];
#pragma unroll
          for (int m = 0; m < 8; m++) c[m] = L(pp[m]);
          // pair[a][side]: that side of axis a sums both copies -- a pair
          // inside the rank, or across the surface with a neighbour on that side
          bool pair[3][2];
#pragma unroll
          for (int a = 0; a < 3; a++)
#pragma unroll
            for (int sd = 0; sd < 2; sd++)
              pair[a][sd] = (ft & (1u << a)) && (!(wt & (1u << a)) || (nbr & (1 << (2 * a + sd))));
          // the tree level by level for both sides of every axis
          double A[2][2][2], Q[2][2][2], Rs[2][2][2];
#pragma unroll
          for (int gx = 0; gx < 2; gx++)
#pragma unroll
            for (int m = 0; m < 4; m++) {
              const double x0 = c[2 * m], x1 = c[2 * m + 1];
              A[gx][m & 1][m >> 1] = pair[0][gx] ? x0 + x1 : (gx ? x1 : x0);
            }
#pragma unroll
          for (int gx = 0; gx < 2; gx++)
#pragma unroll
            for (int gy = 0; gy < 2; gy++)
#pragma unroll
              for (int az = 0; az < 2; az++)
                Q[gx][gy][az] = pair[1][gy] ? A[gx][0][az] + A[gx][1][az] : A[gx][gy][az];
#pragma unroll
          for (int gx = 0; gx < 2; gx++)
#pragma unroll
            for (int gy = 0; gy < 2; gy++)
#pragma unroll
              for (int gz = 0; gz < 2; gz++)
                Rs[gx][gy][gz] = pair[2][gz] ? Q[gx][gy][0] + Q[gx][gy][1] : Q[gx][gy][gz];
#pragma unroll
          for (int m = 0; m < 8; m++) {
            if (m & ~(int)ft) continue;  // a copy the node does not have
            // copy m's side on each split axis
            const bool gx = (wt & 1u) && (m & 1), gy = (wt & 2u) && (m & 2), gz = (wt & 4u) && (m & 4);
            double rz[2][2];
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
              for (int b = 0; b < 2; b++) rz[a][b] = gz ? Rs[a][b][1] : Rs[a][b][0];
            const double ry0 = gy ? rz[0][1] : rz[0][0], ry1 = gy ? rz[1][1] : rz[1][0];
            L(pp[m]) = gx ? ry1 : ry0;
          }
        }
        continue;
      }
    }
    if (i * T + wave0 < FB) {  // a face: two copies
      const unsigned o = cz ? p + DZ : cy ? p + DY : q;
      const double r = L(p) + L(o);
      L(p) = r;
      L(o) = r;
    } else if (f != 7u) {  // an edge: pairs along the tree's first axis of its two, then the other
      const unsigned ox = q, oy = p + DY, oz = p + DZ;
      const unsigned a = TREE ? (cz ? oz : oy) : (cx ? ox : oy), b = TREE ? (cx ? ox : oy) : (cz ? oz : oy);
      const unsigned ab = cx ? (cy ? qy : qz) : p + DY + DZ;
      const double r = (L(p) + L(a)) + (L(b) + L(ab));
      L(p) = r;
      L(a) = r;
      L(b) = r;
      L(ab) = r;
    } else {
      const unsigned o[8] = {p, q, p + DY, qy, p + DZ, qz, p + DY + DZ, qyz};
      double v[8];
#pragma unroll
      for (int c = 0; c < 8; c++) v[c] = L(o[TREE ? (c & 2) | (c & 1) << 2 | c >> 2 : c]);
      const double r = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
      for (int c = 0; c < 8; c++) L(o[c]) = r;
    }
  }
  __syncthreads();

  // ---- stores of the locations the item owns (MODE 1: but the copies of
  // rank-surface nodes, which the surface blocks may be summing)
  if (MODE == 1 && surf) {
    // (block-uniform) a pair with a rank-surface half stores its other half alone
    auto marked = [&](unsigned b) { return ((smark[b >> 8] >> ((b >> 3) & 31)) & 1u) != 0u; };
#pragma unroll
    for (int j = 0; j < JR; j++) {
      const auto d = pair_row(j * T + wave0);
      if (xo[j] == kOOB) continue;
      const u32x2 lo = __builtin_bit_cast(u32x2, L(xo[j])), hi = __builtin_bit_cast(u32x2, L(xo[j] + 8));
      const bool m0 = marked(xo[j]), m1 = marked(xo[j] + 8);
      if (m0 || m1) {
        if (!m0) __builtin_amdgcn_raw_buffer_store_b64(lo, d, xo[j], 0, 0);
        if (!m1) __builtin_amdgcn_raw_buffer_store_b64(hi, d, xo[j] + 8, 0, 0);
      } else {
        const u32x4 x = {lo[0], lo[1], hi[0], hi[1]};
        __builtin_amdgcn_raw_buffer_store_b128(x, d, xo[j], 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < JG; j++) {
      const auto d = single_row(j * T + wave0);
      if (go[j] == kOOB || marked(gq[j])) continue;
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, L(gq[j])), d, go[j], 0, 0);
    }
    return;
  }
  // (read at once, slots without a location from position 0; their stores
  // are out of range)
#pragma unroll
  for (int j = 0; j < JR; j++) {
    const unsigned a = xo[j] == kOOB ? 0u : xo[j];
    const u32x2 lo = __builtin_bit_cast(u32x2, L(a)), hi = __builtin_bit_cast(u32x2, L(a + 8));
    wr[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
#pragma unroll
  for (int j = 0; j < JG; j++) wg[j] = L(go[j] == kOOB ? 0u : gq[j]);
#pragma unroll
  for (int j = 0; j < JG; j++)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, wg[j]), single_row(j * T + wave0), go[j], 0, 0);
#pragma unroll
  for (int j = 0; j < JR; j++) __builtin_amdgcn_raw_buffer_store_b128(wr[j], pair_row(j * T + wave0), xo[j], 0, 0);
}

}  // namespace faces
