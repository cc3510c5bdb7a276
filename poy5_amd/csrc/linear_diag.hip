// Non-affine DO alignment (POY algn_nw, src/algn.c:2972) swept by
// anti-diagonals: a lane owns 2R neighbouring diagonals of the band for a
// whole round, and step s computes every band cell with i + j = s.
//
// Why this shape.  A band of half-width newk holds W = D + 2 newk + 1
// diagonals (D = L2 - L1), and no cell of a pair can be finished before
// anti-diagonal i + j, so a round takes L1 + L2 steps at least.  Sweeping
// rows in 64-row stripes reaches that count only with a boundary row and a
// wait between stripes, and leaves half of a wavefront idle when W < 128.
// Here the band's edges are fixed lanes (no per-cell band tests), the row
// above and the column to the left are the lane's own values or one DPP move
// away, and nothing but directions leaves the registers.
//
// Cells.  Diagonals k = j - i are taken in slots of an even and the next odd
// one; a band lane holds R consecutive slots.  Even diagonals are computed on
// even steps (E steps), odd ones on odd steps (O steps), so with E[r], O[r]
// the newest values of a slot's two diagonals
//   E step: up O[r], left O[r-1] (r = 0: lane - 1's O[R-1]), diagonal E[r]
//   O step: up E[r+1] (r = R-1: lane + 1's E[0]), left E[r], diagonal O[r].
// Slots outside the band are kept above every band value by an OR with the
// slot's constant; the host checks that a launch's sums stay below it, so
// such a value never wins, ties or wraps.
//
// Symbols.  From an E step to the following O step every cell moves one
// column on, from an O step to the next E step one row on; the arrays of row
// and column records shift by one slot, and in 16 steps a lane takes in 8 new
// row symbols and 8 new column symbols: two unaligned 8-byte loads, issued
// two blocks ahead.  A record holds the symbol's table offset and its
// deletion or insertion cost.
//
// Several wavefronts.  With NW > 1 wavefront w owns U = 64 - 2H lanes of the
// band and keeps H halo lanes on either side (2RH >= 16 diagonals).  A halo
// lane's values go stale by one diagonal per step from the outside, so the
// owned lanes stay right for 16 steps; after each block the halos are
// refreshed from the neighbours through LDS with one barrier.
//
// Sweeps.  A pair's doubling rounds differ in their bands only, and each band
// is about half as wide as the next; a sweep runs as many consecutive rounds
// side by side as its lanes hold, a lane outside every band between them.
// Rounds past the one that stops use lanes that were idle.
//
// Directions: 2 bits per cell and step, a word of 16 steps per slot, at
// word (block * stride + slot), stride the band's slots rounded up to 8 (see
// diag_stride): the layout depends on the band only, not on R or NW.  Bit 1 of a cell is set unless
// its move is diagonal, bit 0 says up (else left).
//
// What bounds it: the issue of a lone wavefront (one instruction in 8 cycles)
// while pairs are few, VALU issue when they are many: about 15 instructions
// per cell and step in key form, 20 in wide form.  Measured against the
// stripe fills: 1,024 pairs of 300-700 symbols 2.43 -> 0.39 ms, one pair of
// 1,500 symbols 2.94 -> 0.33 ms, 4,000 rejoin costs through the server
// 20.9 -> 4.8 ms.
#pragma once
#include "poyhip_device.h"
#include "poyhip_layout.h"

namespace poyhip {

// The substitution table's rows are placed as in the workgroup fill
// (mw_ag_row: the 16 lookups of two plain symbols fall in 16 different LDS
// banks); word 32 of row a holds its tail cost, row 32 the prepend costs.
constexpr int kDgPrepend = 32 * 64;
constexpr int kDgInf = 1 << 30;

constexpr int kDgRounds = 4;  // rounds of a sweep, at most

template <int R, int NW>
struct DiagGeom {
  static constexpr int H = NW == 1 ? 1 : (16 + 2 * R - 1) / (2 * R);  // halo lanes a side
  static constexpr int U = 64 - 2 * H;                                // owned lanes
  static constexpr int kLanes = NW * U;
  static constexpr int kMaxBand = kLanes * 2 * R - 1;                 // diagonals
};

// Table offset and deletion / insertion cost of a symbol as a row / column.
struct DiagRec {
  unsigned off;
  int cost;
};
// The wide form holds both in one register (offset below, cost above): its
// eight slots a lane spill less of their 128 registers than with two (128
// pairs of 16,000-100,000 symbols: 1.36 s in the stripe fills, 1.16 s with two
// registers a record, 1.02 s with one).
struct DiagPacked {
  unsigned v;
};
template <bool kKey>
struct DiagRecOf {
  typedef DiagRec type;
};
template <>
struct DiagRecOf<false> {
  typedef DiagPacked type;
};

__device__ __forceinline__ DiagRec dg_rec(DiagRec*, unsigned off, int cost) {
  return DiagRec{off, cost};
}
__device__ __forceinline__ DiagPacked dg_rec(DiagPacked*, unsigned off, int cost) {
  return DiagPacked{off | ((unsigned)cost << 16)};
}
__device__ __forceinline__ int dg_cost(DiagRec r) { return r.cost; }
__device__ __forceinline__ int dg_cost(DiagPacked r) { return (int)(r.v >> 16); }
__device__ __forceinline__ unsigned dg_off(DiagRec r) { return r.off; }
__device__ __forceinline__ unsigned dg_off(DiagPacked r) { return r.v & 0xFFFFu; }
// table offset of a row and a column symbol
__device__ __forceinline__ unsigned dg_addr(DiagRec a, DiagRec b) { return a.off + b.off; }
__device__ __forceinline__ unsigned dg_addr(DiagPacked a, DiagPacked b) {
  unsigned r;  // 16-bit adds clear the upper half
  asm("v_add_u16_e32 %0, %1, %2" : "=v"(r) : "v"(a.v), "v"(b.v));
  return r;
}
// x + the record's cost
__device__ __forceinline__ int dg_plus(int x, DiagRec r) { return x + r.cost; }
__device__ __forceinline__ int dg_plus(int x, DiagPacked p) {
  int r;
  asm("v_add_u32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
      : "=v"(r)
      : "v"(x), "v"(p.v));
  return r;
}

template <int NW, bool kKey>
struct DiagShared {
  typedef typename DiagRecOf<kKey>::type Rec;
  Rec row[32];
  Rec col[32];
  int tab[33 * 64];
  int tail[32];
  int tail_below;  // some tail cost is below its symbol's deletion cost
  int pair[2];
  int fin[kDgRounds][2];
  int scan[NW];
  // edge slots of each wavefront: values and delete counts of 16 diagonals a
  // side, double-buffered
  int halo[NW > 1 ? 2 : 1][NW > 1 ? NW : 1][2][NW > 1 ? 32 : 1];
};

template <int R, bool kKey>
struct DiagState {
  typedef typename DiagRecOf<kKey>::type Rec;
  int vE[R], vO[R], dE[R], dO[R];
  int oob[2 * R];    // kDgInf for slots outside the band (even, odd)
  Rec A[R];          // row records i0 - 1 - r before an E step
  Rec B[R];          // column records j0 + r
};

__device__ __forceinline__ int dg_from_left(int v) {   // lane - 1's value
  return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xF, 0xF, true);
}
__device__ __forceinline__ int dg_from_right(int v) {  // lane + 1's value
  return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xF, 0xF, true);
}
__device__ __forceinline__ int dg_lds(const char* base, unsigned off) {
  return *reinterpret_cast<const int*>(base + off);
}

// Steps of a block: kDgInner every cell lies inside rows and columns 1 and
// up and before the last cell; kDgEdge cells of row 0 and column 0 keep the
// border value they start with until their diagonal's first step (step |k|,
// k = j - i) is past, and nothing changes after the last cell; kDgTail also
// prices deletions in the last column by the tail costs.
constexpr int kDgInner = 0, kDgEdge = 1, kDgTail = 2;

// A cell is carried in one of two forms.
//   wide: its value and its delete count in a register each.
//   key:  value << (nd + 2) | delete count, below 2^31 (the host checks that
//         the launch's sums and counts fit).  Table costs are shifted alike
//         and carry, between value and count, the candidate's rank in the
//         order align (0), insert (2), delete (3; its cost also adds 1 to the
//         count): one minimum picks value, rank and count together, and the
//         rank is the move (bit 1: not diagonal, bit 0: up).  Slots outside
//         the band have bit 31 set.
struct DiagKey {
  int nd;           // bits of the delete count
  unsigned keep;    // ~(3 << nd)
  unsigned one;     // 1 << (nd + 2): a value of 1
};

template <bool kKey>
struct DiagOob {
  static constexpr int value = kKey ? (int)0x80000000u : kDgInf;
};

__device__ __forceinline__ unsigned dg_umin3(unsigned a, unsigned b, unsigned c) {
  const unsigned x = a < b ? a : b;
  return x < c ? x : c;
}

// One cell: the recurrence and tie order of algn_fill_row (src/algn.c:458)
// and backtrace_2d_gaps (978): align, insert, delete for the delete count;
// align, then delete / insert by the swap flag for the move.  `pack` takes
// the move: bit 0 up, bit 1 not diagonal, earlier steps lower once the block
// is done (dg_finish).
template <bool kKey, bool kDm, bool kDc, bool kSw, bool kEdge, class Rec>
__device__ __forceinline__ void dg_cell(const DiagKey& key, bool sw, int up, int left, int diag,
                                        Rec del_c, Rec ins_c, int sub, int udc, int ldc, int oob,
                                        bool upd, int& v, int& d, unsigned& pack) {
  const int del = dg_plus(up, del_c);
  const int ins = dg_plus(left, ins_c);
  const int aln = diag + sub;
  if (kKey) {
    const unsigned m = dg_umin3((unsigned)del, (unsigned)ins, (unsigned)aln);
    if (kDm) {
      if (kSw) {
        pack = __builtin_amdgcn_alignbit(m >> key.nd, pack, 2);
      } else {
        // up wherever the deletion ties with the minimum: the keys then
        // differ by ranks and counts only
        pack = __builtin_amdgcn_alignbit(pack, (unsigned)del - m - key.one, 31);
        pack = __builtin_amdgcn_alignbit(pack, m << (30 - key.nd), 31);
      }
    }
    const int vn = (int)((m & key.keep) | (unsigned)oob);
    v = !kEdge || upd ? vn : v;
  } else {
    const int val = imin(imin(del, ins), aln);
    if (kDm) {
      const lmask nI = ballot(ins != val), D = ballot(del == val);
      pack = shift_in(pack, sw ? nI : D);
      pack = shift_in(pack, ballot(aln != val));
    }
    if (kDc) {
      const int dn = aln == val ? d : (ins == val ? ldc : udc + 1);
      d = !kEdge || upd ? dn : d;
    }
    const int vn = val | oob;
    v = !kEdge || upd ? vn : v;
  }
}

// What the border cells of a block need: the lane's first diagonal, and the
// steps of the block and of the last cell and column.
struct DiagEdge {
  int k0;      // j - i of the lane's first slot's even diagonal
  int s0;      // first step of the block
  int s_fin;   // step of the last cell
  int L2;
};

// Sixteen steps.  rx / cx: the block's new symbols.  The steps run in groups
// of P pairs (E, O); records are read a group ahead and table entries kLook
// steps ahead of their cells, so that a lone wavefront does not wait for
// LDS; the group loop bounds the live registers.
template <int R, bool kKey, bool kDm, bool kDc, bool kSw, int NW, int kMode>
__device__ __forceinline__ void dg_block(DiagState<R, kKey>& S, const DiagShared<NW, kKey>& sh,
                                         const DiagKey& key, bool sw, unsigned long long rx,
                                         unsigned long long cx, const DiagEdge& e,
                                         unsigned pack[R]) {
  typedef typename DiagRecOf<kKey>::type Rec;
  constexpr int P = R <= 2 ? 4 : 2;
  constexpr int kLook = R >= 4 ? 1 : 4 / R;
  constexpr bool kEdge = kMode != kDgInner;
  const char* const tab = reinterpret_cast<const char*>(sh.tab);
  Rec rr[P], cr[P];
  unsigned rlo = (unsigned)rx, clo = (unsigned)cx;
  unsigned rhi = (unsigned)(rx >> 32), chi = (unsigned)(cx >> 32);
  // the next P records; the symbols move down by P bytes
  auto records = [&](Rec r_[P], Rec c_[P]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < P; t++) {
      r_[t] = sh.row[(rlo >> (8 * t)) & 255u];
      c_[t] = sh.col[(clo >> (8 * t)) & 255u];
    }
    rlo = P == 4 ? rhi : (unsigned)((((unsigned long long)rhi << 32) | rlo) >> 16);
    clo = P == 4 ? chi : (unsigned)((((unsigned long long)chi << 32) | clo) >> 16);
    rhi >>= 16;
    chi >>= 16;
  };
  records(rr, cr);
  int sub[2 * P + kLook][R];  // of the group's steps and the next group's first
#pragma unroll
  for (int u = 0; u < kLook; u++)
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int ia = (u >> 1) - r, jb = ((u + 1) >> 1) + r;
      sub[u][r] = dg_lds(tab, dg_addr(ia >= 0 ? rr[ia >= 0 ? ia : 0] : S.A[ia < 0 ? -ia - 1 : 0],
                                      jb < R ? S.B[jb < R ? jb : 0] : cr[jb >= R ? jb - R : 0]));
    }
#pragma unroll 1
  for (int grp = 0; grp < 8 / P; grp++) {
    Rec RA[R - 1 + P], CB[R + P], rn[P], cn[P];
#pragma unroll
    for (int r = 0; r < R - 1; r++) RA[R - 2 - r] = S.A[r];
#pragma unroll
    for (int r = 0; r < R; r++) CB[r] = S.B[r];
#pragma unroll
    for (int t = 0; t < P; t++) {
      RA[R - 1 + t] = rr[t];
      CB[R + t] = cr[t];
    }
    records(rn, cn);  // past the block's end: symbol 0, not used
#pragma unroll
    for (int u = 0; u < 2 * P; u++) {
      const int x = u + kLook;  // this group's step, or the next group's
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int ra = R - 1 + (x >> 1) - r, cb = ((x + 1) >> 1) + r;
        const Rec va = ra < R - 1 + P ? RA[ra < R - 1 + P ? ra : 0]
                                      : rn[ra >= R - 1 + P ? ra - (R - 1 + P) : 0];
        const Rec vb = cb < R + P ? CB[cb < R + P ? cb : 0]
                                  : cn[cb >= R + P ? cb - (R + P) : 0];
        sub[x][r] = dg_lds(tab, dg_addr(va, vb));
      }
      const int s = e.s0 + 2 * P * grp + u;
      const int s_upd = s <= e.s_fin ? s : -1;
      const bool odd = u & 1;
      // the value a cell takes from the next lane
      const int xv = odd ? dg_from_right(S.vE[0]) : dg_from_left(S.vO[R - 1]);
      const int xd = !kDc ? 0 : (odd ? dg_from_right(S.dE[0]) : dg_from_left(S.dO[R - 1]));
#pragma unroll
      for (int r = 0; r < R; r++) {
        const Rec ra = RA[R - 1 + (u >> 1) - r], cb = CB[((u + 1) >> 1) + r];
        Rec del_c = ra;
        bool upd = true;
        if (kEdge) {
          const int k = e.k0 + 2 * r + (odd ? 1 : 0);
          upd = imax(k, -k) < s_upd;
          if (kMode == kDgTail && s + k == 2 * (e.L2 - 1))
            del_c = dg_rec((Rec*)nullptr, dg_off(ra),
                           imin(dg_cost(ra), dg_lds(tab, dg_off(ra) + 32 * 4)));
        }
        if (!odd)
          dg_cell<kKey, kDm, kDc, kSw, kEdge>(key, sw, S.vO[r], r ? S.vO[r ? r - 1 : 0] : xv, S.vE[r], del_c,
                                   cb, sub[u][r], S.dO[r], r ? S.dO[r ? r - 1 : 0] : xd,
                                   S.oob[2 * r], upd, S.vE[r], S.dE[r], pack[r]);
        else
          dg_cell<kKey, kDm, kDc, kSw, kEdge>(key, sw, r < R - 1 ? S.vE[r < R - 1 ? r + 1 : 0] : xv, S.vE[r],
                                   S.vO[r], del_c, cb, sub[u][r],
                                   r < R - 1 ? S.dE[r < R - 1 ? r + 1 : 0] : xd, S.dE[r],
                                   S.oob[2 * r + 1], upd, S.vO[r], S.dO[r], pack[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < R - 1; r++) S.A[r] = RA[R - 2 + P - r];
#pragma unroll
    for (int r = 0; r < R; r++) S.B[r] = CB[P + r];
#pragma unroll
    for (int t = 0; t < P; t++) {
      rr[t] = rn[t];
      cr[t] = cn[t];
    }
#pragma unroll
    for (int u = 0; u < kLook; u++)
#pragma unroll
      for (int r = 0; r < R; r++) sub[u][r] = sub[2 * P + u][r];
  }
  if (kDm && !(kKey && kSw)) {
    // the shifts put step 0 in the top bits
#pragma unroll
    for (int r = 0; r < R; r++) pack[r] = __builtin_bitreverse32(pack[r]);
  }
}

// Eight symbols s[at .. at + 7]; positions outside the sequence read as 0.
// `inside`: every lane that owns band cells has all eight inside.
__device__ __forceinline__ unsigned long long dg_load8(const uint8_t* __restrict__ s, int n, int at,
                                                       bool inside) {
  typedef unsigned long long __attribute__((aligned(1), may_alias)) u64u;
  if (n < 8) {
    unsigned long long x = 0;
    for (int t = 0; t < 8; t++) {
      const int p = at + t;
      if ((unsigned)p < (unsigned)n) x |= (unsigned long long)s[p] << (8 * t);
    }
    return x;
  }
  const int a = imin(imax(at, 0), n - 8);
  unsigned long long x = *reinterpret_cast<const u64u*>(s + a);
  if (!inside) {
    const int off = at - a;  // < 0 before the start, > 0 past the end
    if (off < 0) x = off > -8 ? x << (-8 * off) : 0;
    if (off > 0) x = off < 8 ? x >> (8 * off) : 0;
  }
  return x;
}

// Refreshes the halo lanes of every wavefront from its neighbours' edge lanes
// (buffer buf; one barrier).  A slot outside the band keeps its own value
// (its owner may hold no band lane and write nothing).
template <int R, int NW, bool kKey>
__device__ __forceinline__ void dg_exchange(DiagShared<NW, kKey>& S, DiagState<R, kKey>& st, int buf, int w,
                                            int lane, bool active) {
  constexpr int H = DiagGeom<R, NW>::H;
  const bool lo = lane >= H && lane < 2 * H, hi = lane >= 64 - 2 * H && lane < 64 - H;
  if (active && (lo || hi)) {
    int* const q = S.halo[buf][w][lo ? 0 : 1] + (lo ? lane - H : lane - (64 - 2 * H)) * 4 * R;
#pragma unroll
    for (int r = 0; r < R; r++) {
      q[4 * r] = st.vE[r];
      q[4 * r + 1] = st.vO[r];
      if (!kKey) {
        q[4 * r + 2] = st.dE[r];
        q[4 * r + 3] = st.dO[r];
      }
    }
  }
  __syncthreads();
  const bool fl = lane < H && w > 0, fr = lane >= 64 - H && w + 1 < NW;
  if (active && (fl || fr)) {
    const int* const q = fl ? S.halo[buf][w > 0 ? w - 1 : 0][1] + lane * 4 * R
                            : S.halo[buf][w + 1 < NW ? w + 1 : 0][0] + (lane - (64 - H)) * 4 * R;
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (st.oob[2 * r] == 0) {
        st.vE[r] = q[4 * r];
        if (!kKey) st.dE[r] = q[4 * r + 2];
      }
      if (st.oob[2 * r + 1] == 0) {
        st.vO[r] = q[4 * r + 1];
        if (!kKey) st.dO[r] = q[4 * r + 3];
      }
    }
  }
}

// The rounds of a sweep: round m has half-width newk[m] and owns band lanes
// [start[m], start[m] + lanes[m]), its direction words start at word dm[m].
struct DiagSweep {
  int n = 0;
  int newk[kDgRounds], start[kDgRounds], lanes[kDgRounds];
  long long dm[kDgRounds];
  int cost[kDgRounds], dcnt[kDgRounds];
};

// One sweep of a pair on the workgroup: fills the rounds' last values and
// delete counts; counts the lane-steps into `slots`.
template <int R, int NW, bool kKey, bool kDm, bool kDc, bool kSw>
__device__ __forceinline__ void dg_sweep(DiagShared<NW, kKey>& S, const DiagKey& key, const uint8_t* __restrict__ sa,
                                         const uint8_t* __restrict__ sb, int L1, int L2,
                                         DiagSweep& sp, bool full, bool sw, unsigned* dm,
                                         long long& slots) {
  typedef DiagGeom<R, NW> Geo;
  constexpr int H = Geo::H, U = Geo::U;
  const int w = NW == 1 ? 0 : (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int Dd = L2 - L1;
  const int g = w * U + lane - H;
  // this lane's round, the widest round and the lanes in use
  int newk = -1, g0 = 0, wide = 0, used = 0;
  long long dm0 = 0;
#pragma unroll
  for (int m = 0; m < kDgRounds; m++) {
    if (m < sp.n) {
      if (g >= sp.start[m] && g < sp.start[m] + sp.lanes[m]) {
        newk = sp.newk[m];
        g0 = sp.start[m];
        dm0 = sp.dm[m];
      }
      wide = imax(wide, sp.newk[m]);
      used = sp.start[m] + sp.lanes[m];
    }
  }
  const bool in_round = newk >= 0;
  const int newke = (newk + 1) & ~1;
  const int k0 = in_round ? 2 * R * (g - g0) - newke : 0;  // the lane's first diagonal
  const bool own = lane >= H && lane < 64 - H && in_round;
  const bool active = NW == 1 || w * U - H < used;  // the wavefront holds band lanes
  const int stride = diag_stride(Dd, imax(newk, 0));
  unsigned* dmp = dm + dm0 + (in_round ? (g - g0) * R : 0);
  const int s_fin = L1 + L2 - 2;
  const int nblk = (s_fin >> 4) + 1;
  // of block 0: row of the lane's r = 0 cell on its first step, and the
  // column of its r = 0 cell
  const int i00 = -(k0 >> 1);
  const int j00 = k0 >> 1;
  // symbols of block b: rows i00 + 8b .., columns j00 + R + 8b ..; the band
  // lanes' lowest and highest
  const int widee = (wide + 1) & ~1;
  const int k_last = imax(Dd + wide, -widee) + 2 * R;
  auto rows_in = [&](int b) {
    return -(k_last >> 1) - 1 + 8 * b >= 0 && (widee >> 1) + 8 * b + 7 < L1;
  };
  auto cols_in = [&](int b) {
    return -(widee >> 1) + R + 8 * b >= 0 && (k_last >> 1) + R + 1 + 8 * b + 7 < L2;
  };
  unsigned long long rx[2], cx[2];  // two blocks ahead
#pragma unroll
  for (int b = 0; b < 2; b++) {
    rx[b] = dg_load8(sa, L1, i00 + 8 * b, rows_in(b));
    cx[b] = dg_load8(sb, L2, j00 + R + 8 * b, cols_in(b));
  }
  DiagState<R, kKey> st;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int ia = i00 - 1 - r, jb = j00 + r;
    st.A[r] = S.row[(unsigned)ia < (unsigned)L1 ? sa[ia] & 31 : 0];
    st.B[r] = S.col[(unsigned)jb < (unsigned)L2 ? sb[jb] & 31 : 0];
  }
  // Border values: cell (0, k) of row 0 on diagonal k >= 0 (prefix sums of
  // the prepend costs, algn_fill_first_row) and cell (-k, 0) of column 0 on
  // k < 0 (prefix sums of the deletion or tail costs, one deletion a row).
  // One running sum F over the band's diagonals serves both sides: it
  // subtracts column 0's costs below k = 0 and adds row 0's above.
  DiagEdge edge;
  edge.k0 = k0;
  edge.s_fin = s_fin;
  edge.L2 = L2;
  {
    int f[2 * R];
    int tot = 0;
#pragma unroll
    for (int x = 0; x < 2 * R; x++) {
      const int k = k0 + x;
      const bool in = in_round && (NW == 1 || own) && k < L2 && -k < L1 && k <= Dd + newk;
      int c = 0;
      if (in && k > 0) c = S.tab[kDgPrepend + (sb[k] & 31)];
      if (in && k < 0) {
        const int a = sa[-k] & 31;
        c = full ? -(kKey ? dg_cost(S.row[a]) >> (key.nd + 2) : dg_cost(S.row[a])) : -S.tail[a];
      }
      f[x] = c;
      tot += c;
    }
    int sum;
    int ex = wave_excl_sum_lane(tot, lane, sum);
    if (NW > 1) {
      if (lane == 0) S.scan[w] = sum;
      __syncthreads();
      for (int k = 0; k < w; k++) ex += S.scan[k];
    }
    // each round's F at its k = 0 (whose own entry is 0)
    int fz = ex;
#pragma unroll
    for (int x = 0; x < 2 * R; x++)
      if (k0 + x < 0) fz += f[x];
    int zero = 0;
#pragma unroll
    for (int m = 0; m < kDgRounds; m++) {
      if (m < sp.n) {
        const int gz = sp.start[m] + ((sp.newk[m] + 1) >> 1) / R;
        const int wz = gz / U, lz = gz - wz * U + H;
        int z = __builtin_amdgcn_readlane(fz, lz);
        if (NW > 1) {
          if (w == wz && lane == 0) S.fin[m][0] = z;
        } else if (g0 == sp.start[m]) {
          zero = z;
        }
      }
    }
    if (NW > 1) {
      __syncthreads();
#pragma unroll
      for (int m = 0; m < kDgRounds; m++)
        if (m < sp.n && g0 == sp.start[m]) zero = S.fin[m][0];
      // (S.fin and S.scan are next written after further barriers)
    }
    int F = ex - zero;
    if (NW > 1) {
      // the scan covers the owned lanes; a halo lane's border values come
      // with the first exchange
      if (!own) F = 0;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int odd = 0; odd < 2; odd++) {
        const int k = k0 + 2 * r + odd;
        const bool in = in_round && k >= -newk && k <= Dd + newk;
        const int before = F;
        F += f[2 * r + odd];
        const int d = in && k < 0 ? -k : 0;
        int v = k < 0 ? before : F;
        if (kKey) v = (v << (key.nd + 2)) | d;
        if (!in) v = DiagOob<kKey>::value;
        st.oob[2 * r + odd] = in ? 0 : DiagOob<kKey>::value;
        if (odd) {
          st.vO[r] = v;
          st.dO[r] = d;
        } else {
          st.vE[r] = v;
          st.dE[r] = d;
        }
      }
    }
  }
  const int s_inner = Dd + wide;           // the last step with a border cell
  const int s_outer = L1 + L2 - 1 - wide;  // the first step with a last-column cell
  const bool tails = S.tail_below != 0;
  for (int b = 0; b < nblk; b++) {
    const int s0 = 16 * b;
    if (NW > 1) dg_exchange<R, NW, kKey>(S, st, b & 1, w, lane, active);
    const unsigned long long rcur = rx[0], ccur = cx[0];
    rx[0] = rx[1];
    cx[0] = cx[1];
    if (active) {
      rx[1] = dg_load8(sa, L1, i00 + 8 * (b + 2), rows_in(b + 2));
      cx[1] = dg_load8(sb, L2, j00 + R + 8 * (b + 2), cols_in(b + 2));
      unsigned pack[R];
#pragma unroll
      for (int r = 0; r < R; r++) pack[r] = 0;
      edge.s0 = s0;
      // (a key launch has no tail cost below its symbol's deletion cost)
      if (!kKey && tails && s0 + 15 >= s_outer)
        dg_block<R, kKey, kDm, kDc, kSw, NW, kDgTail>(st, S, key, sw, rcur, ccur, edge, pack);
      else if (s0 > s_inner && s0 + 15 <= s_fin)
        dg_block<R, kKey, kDm, kDc, kSw, NW, kDgInner>(st, S, key, sw, rcur, ccur, edge, pack);
      else
        dg_block<R, kKey, kDm, kDc, kSw, NW, kDgEdge>(st, S, key, sw, rcur, ccur, edge, pack);
      if (kDm && own) {
        unsigned* const p = dmp;
        if (R == 1) {
          p[0] = pack[0];
        } else if (R == 2) {
          *reinterpret_cast<uint2*>(p) = make_uint2(pack[0], pack[R > 1 ? 1 : 0]);
        } else {
#pragma unroll
          for (int r = 0; r < R; r += 4)
            *reinterpret_cast<uint4*>(p + r) =
                make_uint4(pack[r], pack[r + 1 < R ? r + 1 : 0], pack[r + 2 < R ? r + 2 : 0],
                           pack[r + 3 < R ? r + 3 : 0]);
        }
      }
      if (kDm) dmp += stride;
    }
  }
  // each round's last cell, on diagonal D
#pragma unroll
  for (int m = 0; m < kDgRounds; m++) {
    if (m < sp.n) {
      const int kf = Dd + ((sp.newk[m] + 1) & ~1), cf = kf >> 1;
      const int gf = sp.start[m] + cf / R, rf = cf % R;
      const int wf = gf / U, lf = gf - wf * U + H;
      int v = 0, d = 0;
#pragma unroll
      for (int r = 0; r < R; r++)
        if (r == rf) {
          v = (kf & 1) ? st.vO[r] : st.vE[r];
          d = (kf & 1) ? st.dO[r] : st.dE[r];
        }
      v = __builtin_amdgcn_readlane(v, lf);
      d = __builtin_amdgcn_readlane(d, lf);
      if (NW > 1) {
        if (w == wf && lane == 0) {
          S.fin[m][0] = v;
          S.fin[m][1] = d;
        }
      } else {
        sp.cost[m] = kKey ? v >> (key.nd + 2) : v;
        sp.dcnt[m] = kKey ? v & ((1 << key.nd) - 1) : d;
      }
    }
  }
  if (NW > 1) {
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kDgRounds; m++) {
      if (m < sp.n) {
        const int v = __builtin_amdgcn_readfirstlane(S.fin[m][0]);
        const int d = __builtin_amdgcn_readfirstlane(S.fin[m][1]);
        sp.cost[m] = kKey ? v >> (key.nd + 2) : v;
        sp.dcnt[m] = kKey ? v & ((1 << key.nd) - 1) : d;
      }
    }
    __syncthreads();
  }
  const int nact = NW == 1 ? 1 : imin(NW, (used + H + U - 1) / U);
  slots += (long long)nblk * 16 * 64 * R * nact;
}

// Whether a round's direction words fit the pair's region: the stripe
// layout's full width in phase 0; in phase 2 the host sizes the region for
// either layout of the round's band (lin_region_bytes), this one while it
// fits the budget.
__device__ __forceinline__ bool dg_fits(const LinFillArgs& A, int L1, int L2, int64_t bytes) {
  return bytes <= (A.phase == 2 ? A.budget : lin_dm_bytes(L1, L2));
}

// Band cells of a round, as the reference's loops count them: row i covers
// columns max(i - newk, 0) .. min(i + D + newk, L2 - 1).
__device__ __forceinline__ long long dg_cells(int L1, int L2, int newk, bool full, int p) {
  const long long m = imax(0, L1 - 1 - newk);
  return m * (L2 - L1 + newk) + (L1 - 1 - m) * (long long)(L2 - 1) + (L1 - 1) +
         (full ? L2 : imin(L2 - L1 + 1 + p, L2));
}

template <int NW, bool kKey, bool kDm, bool kDc>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_linear_diag(LinFillArgs A) {
  __shared__ DiagShared<NW, kKey> S;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // a second fill takes only what the first left
  if (A.left_in && __builtin_amdgcn_readfirstlane(*A.left_in) == 0) return;
  DiagKey key;
  key.nd = kKey ? A.nd : 0;
  key.keep = ~(3u << key.nd);
  key.one = 4u << key.nd;
  const int sh = kKey ? key.nd + 2 : 0;
  for (int k = tid; k < 1024; k += 64 * NW)
    S.tab[mw_ag_row(k >> 5) + (k & 31)] = A.cm->cost[k] << sh;
  if (tid < 64) {
    const int a = tid & 31;
    const int tl = A.cm->tail[a], del = A.cm->cost[(a << 5) + kGap];
    const bool below = ballot(a > 0 && tl < del) != 0;
    if (tid < 32) {
      S.tab[mw_ag_row(a) + 32] = tl;
      S.tab[kDgPrepend + a] = A.cm->prepend[a];
      S.tail[a] = tl;
      typedef typename DiagRecOf<kKey>::type Rec;
      const int ins = A.cm->cost[(kGap << 5) + a];
      S.row[a] = dg_rec((Rec*)nullptr, (unsigned)(mw_ag_row(a) * 4),
                        kKey ? (del << sh) | (3 << key.nd) | 1 : del);
      S.col[a] = dg_rec((Rec*)nullptr, (unsigned)(a * 4),
                        kKey ? (ins << sh) | (2 << key.nd) : ins);
    }
    if (tid == 0) S.tail_below = below ? 1 : 0;
  }
  __syncthreads();
  const int delta = A.cm->delta;
  for (;;) {
    int q;
    if (NW == 1) {
      q = wave_grab(A.counter);
    } else {
      if (tid == 0) S.pair[0] = atomicAdd(A.counter, 1);
      __syncthreads();
      q = __builtin_amdgcn_readfirstlane(S.pair[0]);
      __syncthreads();  // the next grab rewrites S.pair
    }
    if (q >= A.pt.n) break;
    const int pid = __builtin_amdgcn_readfirstlane(A.pt.order[q]);
    PairResult r1;
    if (A.left_in || A.phase == 2) r1 = A.res[pid];
    if (A.left_in && r1.full != kLinLeft) continue;
    const uint8_t* sa = A.pt.blob + rows_off(A.pt, pid);
    const uint8_t* sb = A.pt.blob + cols_off(A.pt, pid);
    const int L1 = __builtin_amdgcn_readfirstlane(A.pt.len_a[pid]);
    const int L2 = __builtin_amdgcn_readfirstlane(A.pt.len_b[pid]);
    const bool sw = __builtin_amdgcn_readfirstlane(A.pt.prio[pid]) != 0;
    const bool full = lin_full_plane(L1, L2, __builtin_amdgcn_readfirstlane(A.pt.deltawh[pid]));
    const int Dd = L2 - L1;
    unsigned* dm = reinterpret_cast<unsigned*>(A.dm + (kDm ? A.pt.dm_off[pid] : 0));
    int T = (Dd + 1) * delta, rounds = 0;
    long long cells = 0, slots = 0, cells1 = 0;
    if (A.phase == 2) {
      T = __builtin_amdgcn_readfirstlane(r1.pad);
      rounds = __builtin_amdgcn_readfirstlane(r1.rounds) - 1;
      cells1 = r1.cells;
      slots = r1.slots;
    } else if (A.left_in) {
      T = __builtin_amdgcn_readfirstlane(r1.pad);
      rounds = __builtin_amdgcn_readfirstlane(r1.rounds);
      cells = r1.cells;
      slots = r1.slots;
    }
    int newk = 0, cost = 0, gap_num = 0, Tfin = T, dm_word = 0;
    bool left = false;
    for (bool done = false; !done;) {
      Tfin = T;
      const int p = (T - Dd) / 2;
      // band rounds whose stop test cannot pass are skipped (see
      // k_linear_fill)
      if (!full && A.phase != 2 && p <= Dd + 1 && (2 * T - Dd) / 2 - L2 + 1 < 0) {
        rounds++;
        T *= 2;
        continue;
      }
      if (L1 == 1) {
        newk = 0;
        int sum = 0;
        for (int j = 1 + lane; j < L2; j += 64) sum += S.tab[kDgPrepend + (sb[j] & 31)];
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        cost = __builtin_amdgcn_readfirstlane(sum);
        gap_num = L2 - 1;
        cells += full ? L2 : imin(L2 - L1 + 1 + p, L2);
        rounds++;
        const int newp = (2 * T - Dd) / 2;
        done = full || A.phase == 2 || (gap_num + 1) < p || newp - L2 + 1 >= 0;
        if (!done) T *= 2;
        continue;
      }
      // the sweep: the pending round on the fewest cells per lane that hold
      // its band, and the rounds after it while lanes and directions fit
      DiagSweep sp;
      int R = 0, cap = 0, lanes = 0;
      int64_t words = 0;
      int Tm = T;
#pragma unroll
      for (int m = 0; m < kDgRounds; m++) {
        if (m == sp.n) {
          const int pm = (Tm - Dd) / 2;
          const int nk = full ? L1 - 1 : (pm >= L1 ? L1 - 1 : pm);
          const int c = diag_slots(Dd, nk);
          if (m == 0) {
            R = c <= DiagGeom<1, NW>::kLanes       ? 1
                : c <= 2 * DiagGeom<2, NW>::kLanes ? 2
                : c <= 4 * DiagGeom<4, NW>::kLanes ? 4
                                                   : 8;
            cap = R == 1   ? DiagGeom<1, NW>::kLanes
                  : R == 2 ? DiagGeom<2, NW>::kLanes
                  : R == 4 ? DiagGeom<4, NW>::kLanes
                           : DiagGeom<8, NW>::kLanes;
          }
          const int need = (c + R - 1) / R;
          const int at = m ? lanes + 1 : 0;
          const int64_t bytes = diag_dm_bytes(L1, L2, nk);
          // a SIMD runs two wavefronts at little more than one's pace: the
          // rounds after the first share a sweep up to that
          if (at + need <= (m && NW == 16 ? imin(cap, 9 * DiagGeom<1, NW>::U) : cap) && (!kDm || dg_fits(A, L1, L2, 4 * words + bytes))) {
            sp.newk[m] = nk;
            sp.start[m] = at;
            sp.lanes[m] = need;
            sp.dm[m] = words;
            sp.n = m + 1;
            lanes = at + need;
            words += bytes / 4;
            // nothing follows a full plane, phase 2's round or the last one
            if (full || A.phase == 2 || (2 * Tm - Dd) / 2 - L2 + 1 >= 0) sp.n = -(m + 1);
            Tm *= 2;
          }
        }
      }
      if (sp.n < 0) sp.n = -sp.n;
      left = sp.n == 0;
      if (left) break;
#define POYHIP_DG_SWEEP(R_)                                                                     \
  if (!kKey || !kDm || sw)                                                                      \
    dg_sweep<R_, NW, kKey, kDm, kDc, true>(S, key, sa, sb, L1, L2, sp, full, sw, dm, slots);    \
  else                                                                                          \
    dg_sweep<R_, NW, kKey, kDm, kDc, false>(S, key, sa, sb, L1, L2, sp, full, sw, dm, slots);
      if (R == 1) {
        POYHIP_DG_SWEEP(1)
      } else if (R == 2) {
        POYHIP_DG_SWEEP(2)
      } else if (R == 4) {
        POYHIP_DG_SWEEP(4)
      } else {
        POYHIP_DG_SWEEP(8)
      }
#undef POYHIP_DG_SWEEP
#pragma unroll
      for (int m = 0; m < kDgRounds; m++) {
        if (m < sp.n && !done) {
          const int pm = (T - Dd) / 2;
          Tfin = T;
          newk = sp.newk[m];
          cost = sp.cost[m];
          gap_num = sp.dcnt[m] + Dd;
          dm_word = (int)(sp.dm[m] >> 6);
          cells += dg_cells(L1, L2, newk, full, pm);
          rounds++;
          const int newp = (2 * T - Dd) / 2;
          done = full || A.phase == 2 || (gap_num + 1) < pm || newp - L2 + 1 >= 0;
          if (!done) T *= 2;
        }
      }
    }
    if (tid == 0) {
      PairResult r;
      r.cost = cost;
      r.gap_num = gap_num;
      r.newk = newk;
      r.rounds = rounds;
      r.full = left ? kLinLeft : ((full ? 1 : 0) | kLinDiag);
      r.pad = Tfin;
      r.cells = cells;
      if (A.phase == 2) {
        // phase 2 repeats phase 1's last round and reports phase 1's cells;
        // a pair left for the next fill keeps its phase-1 figures
        r.cells = cells1;
        if (left) r.rounds = rounds + 1;
      }
      r.slots = slots;
      A.res[pid] = r;
      if (kDm && !left) A.stab[A.pt.stab_off[pid]] = dm_word;
      if (left) atomicAdd(A.left_out, 1);
    }
    if (NW > 1) __syncthreads();
  }
}

}  // namespace poyhip
