// mlp_prune.h -- the sweep of a DVND round (ADS row map): only the moves that
// can improve the tour.  Included by mlp_kernels.hip after the tiled sweep.
//
// A DVND merge reads nothing but the rows whose best move improves the tour
// (delta < 0), so a block of moves none of which can improve needs no
// evaluation.  Every delta is a sum of terms known per row, terms known per
// column, and positive multiples of distances between a position near the
// row's and one near the column's:
//   swap    Cs(i) + Bs(j) + (N-i) d(i-1,j) + (N-i-1) d(j,i+1)
//                         + (N-j) d(j-1,i) + (N-j-1) d(i,j+1)
//   or-opt  R(i) + C(c) - (column) S(i) + two such products
//   2-opt   (N-i) (d(i-1,j) - w[i]) + (N-j-1) (d(i,j+1) - w[j+1]) + inner(i,j)
// The gap between the bounding boxes of the rows' and the columns' positions
// bounds every such distance from below (the rounded distance is monotone in
// dx^2 + dy^2), and the extremes of the other terms over eight rows and a
// block of 16 columns are cheap: a lower bound of the block's deltas.  Blocks
// with a bound below zero, and those around the diagonal, are evaluated;
// the others hold no improving move.  The rows that improve are therefore
// exactly those of the full sweep, with the same best move and the same
// lowest index among equal ones.  Rows that do not improve may stay empty;
// info[PARTIAL] says so.
//
// One wave owns eight rows x W columns: its lanes test one block each (16 of
// W columns), the survivors are listed in LDS, and 64 lanes evaluate four
// listed blocks at a time, a lane a column, for the eight rows.  A lane
// computes its column's distances to the rows' positions once; the
// neighbouring column's come from the neighbouring lane (DPP), and those of
// the column beyond the block's edge are computed one row a lane and shifted
// to the edge lane.  Nothing but the block list goes through LDS, and no wave
// waits for another (2-opt, whose rows are diagonals, collects the workgroup's
// improving moves per diagonal).
//
// Blocks left of all (rows x 16 columns, recorded solves): n = 1000 a quarter
// in the late rounds, n = 2000 an eighth, n = 9001 one in 25.  What bounds it
// then is the latency of a wave's chain (row set-up, test, column loads, a
// few hundred VALU instructions a group) and, in long launches, the waves
// whose rows survive against most columns.  Clustered n = 9001, mean over a
// solve, against the 16 x 1024 tiles: 83 us a neighborhood before, swap 14,
// 2-opt 17, or-opt-1/2/3 25 / 31 / 32 us now (the solve 365-420 -> 205-234 ms);
// 64 instances n in [50, 2000] in one call 34.1 -> 27.1 ms.
#ifndef MLP_PRUNE_H_
#define MLP_PRUNE_H_

namespace {

constexpr int kPR = 8;                    // rows of a wave
constexpr int kPWg = kPR * kBlock / kWave;  // rows of a workgroup
constexpr int kPMaxW = 1024;              // columns of a wave at most
constexpr int kPMaxBlk = kPMaxW / MLP_BLK;

// What a wave reads first: xy, w and T of position b0 + lane % 16, and the
// summary of the lane's first block with T before it.  All of it is loaded
// beside the slot's info words, before any of them is looked at (one wait
// instead of three: n = 1000 5.7 -> 5.4 us a neighborhood).
struct PruneFirst {
  int rxy, rw, rt, tp;
  int4v sm;
  __device__ __forceinline__ PruneFirst(const SlotDev& s, int b0, int wb0) {
    const int lane = threadIdx.x % kWave, rp = min(b0 + (lane & 15), s.N - 1);
    const int B = min(wb0 + lane, (s.N + MLP_BLK - 1) / MLP_BLK - 1);
    rxy = ldg(s.xy + rp);
    rw = ldg(s.w + rp);
    rt = ldg(s.t32 + rp);
    sm = *(gptr<const int4v>)(blk_of(s) + B);
    tp = ldg(s.t32 + max(B * MLP_BLK - 1, 0));
  }
  __device__ __forceinline__ void arrive() {
    asm volatile("" : "+v"(rxy), "+v"(rw), "+v"(rt), "+v"(tp), "+v"(sm));
  }
};

struct PruneLds {
  uint16_t list[kBlock / kWave][kPMaxBlk];  // surviving blocks of each wave
};
// 2-opt: the best improving key per diagonal D = j - i of the workgroup's
// rows and columns, and of the middle diagonals that belong to a second row.
struct PruneDiag {
  int64_t dgx[4];
  int64_t dg[1];  // W + kPWg
};

__device__ __forceinline__ short2v as_s2(int v) { return __builtin_bit_cast(short2v, v); }
__device__ __forceinline__ int as_i(short2v v) { return __builtin_bit_cast(int, v); }

// Lane l of each 16-lane row gets lane l + S (0 beyond the row's end).
template <int S>
__device__ __forceinline__ int row_shl(int v) {
  if constexpr (S == 0) return v;
  else return __builtin_amdgcn_update_dpp(0, v, 0x100 | S, 0xf, 0xf, true);
}
template <int S>
__device__ __forceinline__ int row_shr(int v) {
  if constexpr (S == 0) return v;
  else return __builtin_amdgcn_update_dpp(0, v, 0x110 | S, 0xf, 0xf, true);
}

// The bounding box of lanes 0..15's packed coordinates (uniform).
__device__ __forceinline__ void row_box(int xy, int& lo, int& hi) {
  short2v a = as_s2(xy), b = a;
#define MLP_BOX_STEP(S)                                                                            \
  a = __builtin_elementwise_min(a, as_s2(__builtin_amdgcn_update_dpp(as_i(a), as_i(a), 0x120 | S, 0xf, 0xf, false))); \
  b = __builtin_elementwise_max(b, as_s2(__builtin_amdgcn_update_dpp(as_i(b), as_i(b), 0x120 | S, 0xf, 0xf, false)));
  MLP_BOX_STEP(1)  // rotations within the row of 16
  MLP_BOX_STEP(2)
  MLP_BOX_STEP(4)
  MLP_BOX_STEP(8)
#undef MLP_BOX_STEP
  lo = __builtin_amdgcn_readlane(as_i(a), 0);
  hi = __builtin_amdgcn_readlane(as_i(b), 0);
}

// Smallest distance between a point of box [alo, ahi] and one of [blo, bhi].
__device__ __forceinline__ int box_gap(int alo, int ahi, int blo, int bhi, float dr) {
  const short2v z = {0, 0};
  const short2v g = __builtin_elementwise_max(
      z, __builtin_elementwise_max(as_s2(blo) - as_s2(ahi), as_s2(alo) - as_s2(bhi)));
  return dist_s(__builtin_amdgcn_sdot2(g, g, 0, false), dr);
}

// A wave's eight rows x W columns of neighborhood NB (0 swap, 1 2-opt,
// 2..4 or-opt-1..3).  WIDE: 2-opt deltas or their bounds beyond 32 bits.
// first: the loads that every wave begins with, issued by the caller.
template <int NB, bool WIDE>
__device__ __forceinline__ void prune_wave(const SlotDev& s, int b0, int ct, int W, uint16_t* list,
                                           PruneDiag* G, int dlo, int par, const PruneFirst& first) {
  constexpr int K = NB >= 2 ? NB - 1 : 0;
  // positions b0 + A0 .. b0 + A1 appear in the rows' distances
  constexpr int A0 = NB >= 2 ? 1 : 0;
  constexpr int A1 = NB == 0 ? kPR + 1 : NB == 1 ? kPR : kPR + K;
  constexpr int NA = A1 + 1;
  using U = std::conditional_t<WIDE, int64_t, uint32_t>;
  using S = std::conditional_t<WIDE, int64_t, int32_t>;
  const int N = s.N, lane = threadIdx.x % kWave;
  const float dr = round_dr(s.round);
  // rows by = b0 + r: swap i = by + 1 <= N - 4; 2-opt i = by + 1 <= N - 3;
  // or-opt by <= N - K - 3
  const int rv = min(kPR, (NB == 0 ? N - 4 : NB == 1 ? N - 3 : N - K - 2) - b0);
  if (rv <= 0) return;
  // column positions c of this wave: swap j = c; 2-opt j = c - 1; or-opt
  // forward j = c - K, backward j = c
  const int nblk = (N + MLP_BLK - 1) / MLP_BLK;
  const int wb0 = ct * (W / MLP_BLK), wb1 = min(nblk, wb0 + W / MLP_BLK);
  if (wb0 >= wb1) return;
  // swap and 2-opt columns lie right of the rows
  if (NB < 2 && wb1 * MLP_BLK <= b0 + 3) return;

  // row side: position b0 + (lane & 15) in each row of 16 lanes
  const int rl = lane & 15;
  const int rp = min(b0 + rl, N - 1);
  const int rxy = first.rxy, rw = first.rw, rt = first.rt;
  int64_t rq = 0;
  int rg = 0;
  if (NB == 1) {
    if (WIDE) rq = ldg(s.q64 + rp);
    else rg = ldg(s.g32 + rp);
  }
  int boxlo, boxhi;
  {
    const int inb = min(max(rl, A0), min(A1, A0 + rv + A1 - A0 - kPR));
    const int bxy = __builtin_amdgcn_ds_bpermute(inb * 4, rxy);
    row_box(bxy, boxlo, boxhi);
  }
  int xa[NA];
#pragma unroll
  for (int a = A0; a < NA; ++a) xa[a] = __builtin_amdgcn_readlane(rxy, a);

  // row constants (lane r < 8: row r)
  uint32_t Cs[kPR], RF[kPR], RB[kPR];  // swap Cs; or-opt forward / backward
  int SF[kPR], SB[kPR];
  U Ai[kPR];                            // 2-opt: -(N - i) w[i] - Z[i]
  int Ti[kPR], wi[kPR];
  int rowmin = 0, rowminB = 0, segmax = 0;
  const int rowi = b0 + rl + 1;  // i of swap, 2-opt and forward or-opt
  const bool rok = rl < rv;
  if (NB == 0) {
    const uint32_t w1 = (uint32_t)row_shl<1>(rw), w2 = (uint32_t)row_shl<2>(rw);
    const uint32_t c = 0u - umul(N - rowi, w1) - umul(N - rowi - 1, w2);
    rowmin = wave_min_i32(rok ? (int)c : INT32_MAX);
#pragma unroll
    for (int r = 0; r < kPR; ++r) Cs[r] = lane_bcast(c, r);
  } else if (NB == 1) {
    const int w1 = row_shl<1>(rw), t1 = row_shl<1>(rt);
    U a;
    if constexpr (WIDE) {
      const int qlo = row_shl<1>((int)(uint32_t)(uint64_t)rq);
      const int qhi = row_shl<1>((int)(uint32_t)((uint64_t)rq >> 32));
      const int64_t q = (int64_t)(((uint64_t)(uint32_t)qhi << 32) | (uint32_t)qlo);
      a = -(int64_t)(N - rowi) * w1 - (2 * q - (int64_t)(2 * rowi + 1) * t1);
    } else {
      a = (uint32_t)row_shl<1>(rg);
    }
#pragma unroll
    for (int r = 0; r < kPR; ++r) {
      if constexpr (WIDE) {
        const uint32_t lo = lane_bcast((uint32_t)(uint64_t)a, r);
        const uint32_t hi = lane_bcast((uint32_t)((uint64_t)a >> 32), r);
        Ai[r] = (int64_t)(((uint64_t)hi << 32) | lo);
      } else {
        Ai[r] = lane_bcast((uint32_t)a, r);
      }
      Ti[r] = __builtin_amdgcn_readlane(t1, r);
      wi[r] = __builtin_amdgcn_readlane(w1, r);
    }
  } else {
    // forward i = by + 1, backward i = by + 2 (lane shifts of 1 and 2)
    const int wF = row_shl<1>(rw), wB = row_shl<2>(rw);
    const int wFk = row_shl<1 + K>(rw), wBk = row_shl<2 + K>(rw);
    const int tF = row_shl<1>(rt), tB = row_shl<2>(rt);
    const int sF = row_shl<K>(rt) - tF, sB = row_shl<1 + K>(rt) - tB;  // T[i+K-1] - T[i]
    const int tFk = row_shl<1 + K>(rt);
    const int iF = rowi, iB = rowi + 1;
    const uint32_t dF = (uint32_t)dist_xy(rxy, row_shl<1 + K>(rxy), dr);
    const uint32_t dB = (uint32_t)dist_xy(row_shl<1>(rxy), row_shl<2 + K>(rxy), dr);
    // delta = f + (its column's terms) + (i - j) S, without the S term
    const uint32_t f = (uint32_t)(N - iF) * (dF - (uint32_t)wF) -
                       (uint32_t)(N - iF - K) * (uint32_t)wFk - (uint32_t)K * (uint32_t)tFk;
    const uint32_t g = (uint32_t)(N - iB - K) * (dB - (uint32_t)wBk) -
                       (uint32_t)(N - iB) * (uint32_t)wB - (uint32_t)K * (uint32_t)tF;
    rowmin = wave_min_i32(rok ? (int)(f + (uint32_t)(iF - b0) * (uint32_t)sF) : INT32_MAX);
    rowminB = wave_min_i32(rok ? (int)g : INT32_MAX);
    segmax = K > 1 ? wave_max_i32(rok ? sF : 0) : 0;
    const uint32_t rf = f + (uint32_t)iF * (uint32_t)sF, rb = g + (uint32_t)iB * (uint32_t)sB;
#pragma unroll
    for (int r = 0; r < kPR; ++r) {
      RF[r] = lane_bcast(rf, r);
      RB[r] = lane_bcast(rb, r);
      SF[r] = __builtin_amdgcn_readlane(sF, r);
      SB[r] = __builtin_amdgcn_readlane(sB, r);
    }
  }

  // --- test: one block a lane, survivors appended to the wave's list
  const int ilo = b0 + 1, ihi = b0 + rv;  // rows' i (backward or-opt: one more)
  int cnt = 0;
  for (int q0 = wb0; q0 < wb1; q0 += kWave) {
    const int B = q0 + lane;
    const int Bc = min(B, wb1 - 1);
    const int c0 = Bc * MLP_BLK, c1 = min(c0 + MLP_BLK - 1, N - 1);
    // block Bc's summary and T[c0 - 1]
    int4v sm = first.sm;
    int tp = first.tp;
    if (q0 > wb0) {
      sm = *(gptr<const int4v>)(blk_of(s) + Bc);
      tp = ldg(s.t32 + max(c0 - 1, 0));
    }
    bool keep;
    const uint32_t D = (uint32_t)box_gap(boxlo, boxhi, sm.x, sm.y, dr);
    if (NB == 0) {
      const int jhi = min(c1, N - 2);
      const bool none = jhi < ilo + 2, pure = c0 >= ihi + 2;
      const int lb = rowmin - (int)umul(N - c0, sm.w) + (int)umul(2 * (N - ihi) - 1, D) +
                     (int)umul(2 * (N - jhi) - 1, D);
      keep = !none && !(pure && lb >= 0);
    } else if (NB == 1) {
      const int j0 = c0 - 1, jhi = min(c1 - 1, N - 2);
      const bool none = jhi < ilo + 1, pure = j0 > ihi;
      // inner(i, j) = Z[j] - Z[i] + (j - i)(T[i] + T[j]), Z = 2 Q - (2p + 1) T:
      // exactly for each row at j0 = c0 - 1, then for j = j0 + u
      //   inner(i, j) - inner(i, j0) = (j0 - i - 1) t + (2 q - u t) - u (T[j0] - T[i])
      // with t and q the sums of w and of (p - j0) w over (j0, j]: least over
      // the rows at the last i in the first term and the first i in the last
      // one; over u exactly
      keep = !none;
      if (keep && pure) {
        U zj;
        if constexpr (WIDE) zj = 2 * ldg(s.q64 + j0) - (int64_t)(2 * j0 + 1) * tp;
        else zj = (uint32_t)ldg(s.h32 + j0) + umul(N - j0 - 1, ldg(s.w + c0));
        S fm = std::numeric_limits<S>::max();
#pragma unroll
        for (int r = 0; r < kPR; ++r) {
          const int i = b0 + r + 1;
          const U f = zj + Ai[r] + (U)(N - i) * (U)D + (U)(j0 - i) * (U)(Ti[r] + tp);
          if (r < rv) fm = min(fm, (S)f);
        }
        const S alpha = j0 - ihi - 1, beta = tp - Ti[0];
        S gm = std::numeric_limits<S>::max();
        int t = 0, q = 0;
#pragma unroll
        for (int u = 0; u < MLP_BLK; u += 4) {
          int w4[4];
          if (c0 + MLP_BLK <= N) {
            const int4 v = *(const int4*)(s.w + c0 + u);
            w4[0] = v.x; w4[1] = v.y; w4[2] = v.z; w4[3] = v.w;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) w4[e] = ldg(s.w + min(c0 + u + e, N - 1));
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int uu = u + e;
            const U g = (U)alpha * (U)t + (U)(2 * q - uu * t) - (U)uu * (U)beta -
                        (U)(N - j0 - uu - 1) * (U)w4[e];
            if (j0 + uu <= jhi) gm = min(gm, (S)g);
            t += w4[e];
            q += (uu + 1) * w4[e];
          }
        }
        const U lb = (U)fm + (U)gm + (U)(N - jhi - 1) * (U)D;
        keep = (S)lb < 0;
      }
    } else {
      // forward moves need c >= by + 2 + K, backward ones c <= by + 1
      const bool fwd = c0 >= b0 + rv + 1 + K, bwd = c1 <= b0 + 1;
      const int colT = K * tp;
      const int colW = (int)umul(N - c0, sm.z);
      // forward j = c - K: (N - j - K) + (N - j) = 2 (N - c) + K
      const int lbF = rowmin - (c1 - K - b0) * segmax - colW + colT + (int)umul(2 * (N - c1) + K, D);
      // backward j = c: (N - j) + (N - j - K); (i - j) S >= 0
      const int lbB = rowminB - colW + colT + (int)umul(2 * (N - c1) - K, D);
      keep = !((fwd && lbF >= 0) || (bwd && lbB >= 0));
    }
    keep = keep && B < wb1;
    const uint64_t m = __builtin_amdgcn_ballot_w64(keep);
    if (keep) list[cnt + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)B;
    cnt += __popcll(m);
  }
  if (cnt == 0) return;
  __builtin_amdgcn_wave_barrier();

  // --- evaluation of the listed blocks, four at a time
  int32_t bd[kPR], bc[kPR];
#pragma unroll
  for (int r = 0; r < kPR; ++r) {
    bd[r] = 0;  // improving moves only
    bc[r] = -1;
  }
  const int rows2 = (N + 1) >> 1, mid0 = N - 1 - rows2;
  const int x = lane & 15;
  struct Col {
    int c, xy, xl, xr, w, w1, t, h;
    int64_t q;
    bool ok;
  };
  auto load = [&](int g) {
    Col o;
    const int e = g * 4 + (lane >> 4);
    const int B = list[min(e, cnt - 1)];
    const int c = B * MLP_BLK + x;
    const int cc = min(c, N - 1);
    o.c = cc;
    o.ok = e < cnt && c < N;
    o.xy = ldg(s.xy + cc);
    o.xl = ldg(s.xy + max(B * MLP_BLK - 1, 0));
    if (NB == 0) o.xr = ldg(s.xy + min(B * MLP_BLK + MLP_BLK, N - 1));
    o.w = ldg(s.w + cc);
    if (NB == 0) o.w1 = ldg(s.w + min(cc + 1, N - 1));
    if (NB >= 2) o.t = ldg(s.t32 + cc);
    if (NB == 1) {
      const int j = max(cc - 1, 0);
      o.t = ldg(s.t32 + j);
      if (WIDE) o.q = ldg(s.q64 + j);
      else o.h = ldg(s.h32 + j);
    }
    return o;
  };
  Col nx = load(0);
  const int groups = (cnt + 3) >> 2;
  for (int g = 0; g < groups; ++g) {
    const Col o = nx;
    if (g + 1 < groups) nx = load(g + 1);
    const int c = o.c;
    const uint32_t nc = (uint32_t)(N - c);
    // own[a]: distance of row position a to the lane's column; hl, hr: of row
    // position lane % 16 to the columns beyond the block's edges
    int own[NA], hl, hr = 0;
    auto dists = [&](const auto& dist) {
#pragma unroll
      for (int a = A0; a < NA; ++a) own[a] = dist_by(xa[a], o.xy, dist);
      hl = dist_by(rxy, o.xl, dist);
      if constexpr (NB == 0) hr = dist_by(rxy, o.xr, dist);
    };
    if (s.small) dists(fast_dist(s.round));
    else dists(FullDist{dr});
    // left[a]: distance of row position a to the column on the left; the
    // block's first lane takes it from lane a, which computed row a's
    int left[NA];
#define MLP_LEFT(A)                                                                          \
  if constexpr ((A) >= A0 && (A) < NA)                                                       \
    left[A] = __builtin_amdgcn_update_dpp(row_shl<A>(hl), own[A], 0x111, 0xf, 0xf, false);
    MLP_LEFT(0) MLP_LEFT(1) MLP_LEFT(2) MLP_LEFT(3) MLP_LEFT(4) MLP_LEFT(5) MLP_LEFT(6)
    MLP_LEFT(7) MLP_LEFT(8) MLP_LEFT(9) MLP_LEFT(10) MLP_LEFT(11)
#undef MLP_LEFT
    int right[kPR + 1];
    if constexpr (NB == 0) {
#define MLP_RIGHT(A)                                                                         \
  right[A] = __builtin_amdgcn_update_dpp(row_shr<15 - (A)>(hr), own[A], 0x101, 0xf, 0xf, false);
      MLP_RIGHT(1) MLP_RIGHT(2) MLP_RIGHT(3) MLP_RIGHT(4) MLP_RIGHT(5) MLP_RIGHT(6) MLP_RIGHT(7)
      MLP_RIGHT(8)
#undef MLP_RIGHT
    }
    if constexpr (NB == 0) {
      // j = c in [i + 2, N - 2]
      const uint32_t cs = opaque(0u - umul(nc, o.w) - umul(nc - 1u, o.w1));
      const bool okc = o.ok && c <= N - 2;
      int32_t d[kPR], any = 0;
#pragma unroll
      for (int r = 0; r < kPR; ++r) {
        const uint32_t a1 = (uint32_t)(N - b0 - r - 1);
        const uint32_t v = Cs[r] + cs + umul(a1, own[r]) + umul(a1 - 1u, own[r + 2]) +
                           umul(nc, left[r + 1]) + umul(nc - 1u, right[r + 1]);
        const bool ok = okc && r < rv && c >= b0 + r + 3;
        d[r] = ok ? (int32_t)v : 0;
        any |= d[r];
      }
      if (__builtin_amdgcn_ballot_w64(any < 0)) {
#pragma unroll
        for (int r = 0; r < kPR; ++r) take_min(bd[r], bc[r], (uint32_t)d[r], c);
      }
    } else if constexpr (NB == 1) {
      // j = c - 1 in [i + 1, N - 2]
      const int j = c - 1;
      U hj;
      if constexpr (WIDE)
        hj = 2 * o.q - (int64_t)(2 * j + 1) * o.t - (int64_t)(N - j - 1) * o.w;
      else
        hj = (uint32_t)o.h;
#pragma unroll
      for (int r = 0; r < kPR; ++r) {
        const int i = b0 + r + 1;
        U v;
        if constexpr (WIDE)
          v = Ai[r] + hj + (int64_t)(int32_t)(umul((uint32_t)(N - i), left[r])) +
              (int64_t)(int32_t)umul((uint32_t)(N - j - 1), own[r + 1]) +
              (int64_t)(j - i) * (int64_t)(Ti[r] + o.t);
        else
          v = Ai[r] + hj + umul((uint32_t)(N - i), left[r]) +
              umul((uint32_t)(N - j - 1), own[r + 1]) +
              (uint32_t)(j - i) * (uint32_t)(Ti[r] + o.t);
        if (o.ok && r < rv && j >= i + 1 && (S)v < 0) {
          const int Dg = j - i;
          const int64_t base = (int64_t)(S)v * (int64_t)(1 << MLP_KEY_SHIFT);
          atomicMin((long long*)&G->dg[Dg - dlo], (long long)(base + (Dg <= rows2 ? j - 2 : N - 2 - j)));
          if (Dg >= mid0 && Dg <= rows2)
            atomicMin((long long*)&G->dgx[Dg - mid0], (long long)(base + (N - 2 - j)));
        }
      }
    } else {
      // lanes left of the rows hold backward moves (j = c), lanes right of
      // them forward ones (j = c - K), lanes among them either by row
      const uint32_t wt = umul(nc, o.w);
      const uint32_t kt = (uint32_t)K * (uint32_t)o.t;
      const uint32_t CB = opaque(kt - wt), CF = opaque(kt - (uint32_t)K * (uint32_t)o.w - wt);
      int32_t d[kPR], any = 0;
      // own and left are indexed by the direction's row offset
#pragma unroll
      for (int r = 0; r < kPR; ++r) {
        const bool bw = c <= b0 + r + 1;
        const uint32_t v1 = (uint32_t)(bw ? own[r + 1 + K] : own[r + K]);
        const uint32_t v2 = (uint32_t)(bw ? left[r + 2] : left[r + 1]);
        const uint32_t n1 = nc - (bw ? (uint32_t)K : 0u), n2 = nc + (bw ? 0u : (uint32_t)K);
        uint32_t v = (bw ? RB[r] + CB : RF[r] + CF) + umul(n1, v1) + umul(n2, v2);
        if (K > 1) v -= bw ? umul(c, SB[r]) : (uint32_t)__mul24(c - K, SF[r]);
        const bool ok = o.ok && r < rv && c >= 1 && (bw ? c <= N - K - 1 : c >= b0 + r + 2 + K);
        d[r] = ok ? (int32_t)v : 0;
        any |= d[r];
      }
      if (__builtin_amdgcn_ballot_w64(any < 0)) {
#pragma unroll
        for (int r = 0; r < kPR; ++r)
          take_min(bd[r], bc[r], (uint32_t)d[r], c <= b0 + r + 1 ? c - 1 : c - K - 1);
      }
    }
  }
  if constexpr (NB != 1) {
    int64_t* out = row_buf(s, NB, par) + b0;
#pragma unroll
    for (int r = 0; r < kPR; ++r)
      if (__builtin_amdgcn_ballot_w64(bd[r] < 0)) {
        const int64_t key = wave_argmin(bd[r], bc[r]);
        if (lane == 0) fold_key(out + r, key);
      }
  }
}

}  // namespace

// One workgroup: 32 rows x W columns of one slot (SweepSeg: slot, first item,
// column chunks).
template <int NB>
__global__ __launch_bounds__(kBlock) void k_psweep(const SlotDev* __restrict__ table,
                                                   SweepSegsInline inl, const SweepSeg* segs_dev,
                                                   int nsegs, int W) {
  __shared__ PruneLds L;
  extern __shared__ int64_t pdyn[];  // 2-opt: PruneDiag with W + kPWg diagonals
  const int item = blockIdx.x;
  const SweepSeg sg = segs_dev ? find_sweep(segs_dev, nsegs, item) : find_sweep_inline(inl, nsegs, item);
  const SlotDev& s = table[sg.slot];
  const int N = s.N, tid = threadIdx.x, wave = wave_id();
  const int b = item - sg.blk0;
  const int rb = b / sg.ncols, ct = b % sg.ncols;
  const int w0 = rb * kPWg, rows = rows_of(NB, 0, N);
  PruneFirst first(s, w0 + wave * kPR, ct * (W / MLP_BLK));
  const int64_t active = ldg(s.info + MLP_INFO_ACTIVE), pf = ldg(s.info + MLP_INFO_PATH32);
  const int par = 1 - (int)(ldg(s.info + MLP_INFO_PARITY0 + NB) & 1);
  first.arrive();
  if (active == 0) return;
  if (b == 0 && tid == 0) s.info[MLP_INFO_PARTIAL] = s.info[MLP_INFO_ROUNDS] + 1;
  if (ct == 0) reset_other(s, NB, par, w0, min(w0 + kPWg, rows), rb == 0);
  if constexpr (NB != 1) {
    if (!(pf & MLP_P32_SWAP_OROPT)) {  // deltas beyond 32 bits: whole rows, one wave each
      if (ct != 0) return;
      for (int by = w0 + wave; by < min(w0 + kPWg, rows); by += kBlock / kWave)
        eval_row<NB == 0 ? 0 : 2, false>(s, NB, 0, by, tid % kWave, row_buf(s, NB, par) + by);
      return;
    }
    prune_wave<NB, false>(s, w0 + wave * kPR, ct, W, L.list[wave], nullptr, 0, par, first);
  } else {
    PruneDiag* G = reinterpret_cast<PruneDiag*>(pdyn);
    // diagonals D = c - 1 - i of the workgroup's rows i = w0 + 1 .. w0 + 32
    const int c0 = ct * W, nd = W + kPWg;
    if (c0 + W <= w0 + 3) return;  // no column right of the rows
    const int dlo = c0 - 1 - w0 - kPWg;
    int64_t* dg = G->dg;
    for (int q = tid; q < nd; q += kBlock) dg[q] = MLP_KEY_NONE;
    if (tid < 4) G->dgx[tid] = MLP_KEY_NONE;
    __syncthreads();
    if (pf & MLP_LB32_2OPT) prune_wave<1, false>(s, w0 + wave * kPR, ct, W, L.list[wave], G, dlo, par, first);
    else prune_wave<1, true>(s, w0 + wave * kPR, ct, W, L.list[wave], G, dlo, par, first);
    __syncthreads();
    const int rows2 = (N + 1) >> 1, mid0 = N - 1 - rows2;
    int64_t* out = row_buf(s, 1, par);
    for (int q = tid; q < nd; q += kBlock) {
      const int64_t key = dg[q];
      if (key == MLP_KEY_NONE) continue;
      const int D = dlo + q;
      fold_key_filtered(out + (D <= rows2 ? D - 1 : N - 2 - D), key);
    }
    if (tid < 4) fold_key(out + (N - 2 - (mid0 + tid)), G->dgx[tid]);
  }
}

#endif  // MLP_PRUNE_H_

