// Banded affine-gap alignment of gap-free pairs (POY algn_CAML_align_affine_3,
// src/algn.c:2359) swept by anti-diagonals: the lanes, sweeps, halos and
// symbol records of linear_diag.hip with Gotoh's cell.
//
// Cell.  Without gap bits POY's four states reduce to H, V and C (close), the
// horizontal and vertical extensions to plain costs, and the gap-gap block
// never wins (affine.hip, aff_cell_fast_core).  Costs and gap counts fit one
// 32-bit key, value << nd | (2^nd - 1 - horizontal gap count): the reference
// keeps the largest count over the moves that tie for the minimum, which is
// the smallest key.  A diagonal keeps
//   F   the cell's key: min over C, H, V, each with the count of the cell it
//       comes from (one more for H)
//   MH  min(H, C + opening): what the next column's H extends or opens from
//   MV  min(V, C + opening): the same for the next row's V
// (MH and MV with the count bits zero).  Every path into a cell has the same
// difference of horizontal and vertical moves, so the largest horizontal
// count is POY's gap number where the doubling tests it.
//
// The host checks that every finite sum, shifted, stays below 2^29; kAdInf
// (2^30) stands for POY's HIGH_NUM, which is above every finite sum too, so
// that no comparison that matters depends on its value.  Slots outside the
// band take kAdInf for the opening, and lanes outside every round read symbol
// 0, whose costs are kAdInf: their MH and MV never drop below it.
//
// Directions: 4 bits per cell and step, 8 steps a word, at word
// (step / 8 * stride + slot): V is a minimum, H is a minimum, V >= C + opening,
// H >= C + opening.  The last two belong to the cell a run of gaps starts
// from, so a walk reads them one cell on; the swap flag is the walk's.
//
// What bounds it: VALU issue, 22 to 24 instructions per cell and step against
// about 53 for the rotating stripes (whose lanes are busy 87% of the time, these
// 65 to 70%: bands fill whole lane counts), and for a few long pairs the
// issue of their own wavefronts.  Measured against the stripes: 16,384 pairs of
// 50-5,000 symbols 47 -> 20 ms, 65,536 of them 69 -> 61 ms, one pair of 110
// symbols 131 -> 46 us.
#pragma once
#include "linear_diag.hip"

namespace poyhip {

constexpr int kAdInf = 1 << 30;
template <int NW>
struct AdShared {
  DiagRec row[32];  // cost: vertical extension
  DiagRec col[32];  // cost: horizontal extension
  int tab[32 * 64];
  int pair[2];
  int fin[kDgRounds];
  int scan[NW];
  int halo[NW > 1 ? 2 : 1][NW > 1 ? NW : 1][2][NW > 1 ? 54 : 1];
};

template <int R>
struct AdState {
  unsigned fE[R], fO[R], hE[R], hO[R], vE[R], vO[R];
  unsigned open[2 * R];  // C + opening: the opening, kAdInf outside the band
  DiagRec A[R];
  DiagRec B[R];
};

__device__ __forceinline__ unsigned ad_umin(unsigned a, unsigned b) { return a < b ? a : b; }

template <bool kEdge>
__device__ __forceinline__ void ad_cell(unsigned low, unsigned upF, unsigned upV, unsigned leftF,
                                        unsigned leftH, unsigned ge, unsigned gr, unsigned sub,
                                        unsigned open, bool upd, unsigned& F, unsigned& MH,
                                        unsigned& MV, unsigned& pack) {
  const unsigned c = F + sub;
  const unsigned cg = (c & ~low) + open;
  const unsigned h = leftH + gr;
  const unsigned v = upV + ge;
  const unsigned ch = h + (leftF & low) - 1;
  const unsigned cv = v + (upF & low);
  const unsigned f = dg_umin3(c, ch, cv);
  const unsigned fv = f & ~low;
  pack = shift_in(pack, ballot(v == fv));
  pack = shift_in(pack, ballot(h == fv));
  pack = shift_in(pack, ballot(v >= cg));
  pack = shift_in(pack, ballot(h >= cg));
  const unsigned mh = ad_umin(h, cg), mv = ad_umin(v, cg);
  F = !kEdge || upd ? f : F;
  MH = !kEdge || upd ? mh : MH;
  MV = !kEdge || upd ? mv : MV;
}

// Sixteen steps (see dg_block); the two direction words of each slot go to
// dmp and dmp + stride.
template <int R, int NW, bool kEdge>
__device__ __forceinline__ void ad_block(AdState<R>& S, const AdShared<NW>& sh, unsigned low,
                                         unsigned long long rx, unsigned long long cx,
                                         const DiagEdge& e, unsigned* dmp, int stride, bool own) {
  constexpr int P = 4;  // a group of 8 steps fills a direction word
  constexpr int kLook = R >= 3 ? 1 : 4 / R;
  const char* const tab = reinterpret_cast<const char*>(sh.tab);
  DiagRec rr[P], cr[P];
  unsigned rlo = (unsigned)rx, clo = (unsigned)cx;
  const unsigned rhi = (unsigned)(rx >> 32), chi = (unsigned)(cx >> 32);
  auto records = [&](DiagRec r_[P], DiagRec c_[P]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < P; t++) {
      r_[t] = sh.row[(rlo >> (8 * t)) & 31u];
      c_[t] = sh.col[(clo >> (8 * t)) & 31u];
    }
    rlo = rhi;
    clo = chi;
  };
  records(rr, cr);
  int sub[2 * P + kLook][R];
#pragma unroll
  for (int u = 0; u < kLook; u++)
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int ia = (u >> 1) - r, jb = ((u + 1) >> 1) + r;
      sub[u][r] = dg_lds(tab, (ia >= 0 ? rr[ia >= 0 ? ia : 0] : S.A[ia < 0 ? -ia - 1 : 0]).off +
                                  (jb < R ? S.B[jb < R ? jb : 0] : cr[jb >= R ? jb - R : 0]).off);
    }
#pragma unroll 1
  for (int grp = 0; grp < 2; grp++) {
    DiagRec RA[R - 1 + P], CB[R + P], rn[P], cn[P];
#pragma unroll
    for (int r = 0; r < R - 1; r++) RA[R - 2 - r] = S.A[r];
#pragma unroll
    for (int r = 0; r < R; r++) CB[r] = S.B[r];
#pragma unroll
    for (int t = 0; t < P; t++) {
      RA[R - 1 + t] = rr[t];
      CB[R + t] = cr[t];
    }
    records(rn, cn);
    unsigned pack[R];
#pragma unroll
    for (int r = 0; r < R; r++) pack[r] = 0;
#pragma unroll
    for (int u = 0; u < 2 * P; u++) {
      const int x = u + kLook;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int ra = R - 1 + (x >> 1) - r, cb = ((x + 1) >> 1) + r;
        const unsigned va = ra < R - 1 + P ? RA[ra < R - 1 + P ? ra : 0].off
                                           : rn[ra >= R - 1 + P ? ra - (R - 1 + P) : 0].off;
        const unsigned vb = cb < R + P ? CB[cb < R + P ? cb : 0].off
                                       : cn[cb >= R + P ? cb - (R + P) : 0].off;
        sub[x][r] = dg_lds(tab, va + vb);
      }
      const int s = e.s0 + 2 * P * grp + u;
      const int s_upd = s <= e.s_fin ? s : -1;
      const bool odd = u & 1;
      // what a cell takes from the next lane: up (odd steps) or left
      const unsigned xF = odd ? dg_from_right(S.fE[0]) : dg_from_left(S.fO[R - 1]);
      const unsigned xM = odd ? dg_from_right(S.vE[0]) : dg_from_left(S.hO[R - 1]);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const unsigned ge = RA[R - 1 + (u >> 1) - r].cost, gr = CB[((u + 1) >> 1) + r].cost;
        bool upd = true;
        if (kEdge) {
          const int k = e.k0 + 2 * r + (odd ? 1 : 0);
          upd = imax(k, -k) < s_upd;
        }
        if (!odd)
          ad_cell<kEdge>(low, S.fO[r], S.vO[r], r ? S.fO[r ? r - 1 : 0] : xF,
                         r ? S.hO[r ? r - 1 : 0] : xM, ge, gr, sub[u][r], S.open[2 * r], upd,
                         S.fE[r], S.hE[r], S.vE[r], pack[r]);
        else
          ad_cell<kEdge>(low, r < R - 1 ? S.fE[r < R - 1 ? r + 1 : 0] : xF,
                         r < R - 1 ? S.vE[r < R - 1 ? r + 1 : 0] : xM, S.fE[r], S.hE[r], ge, gr,
                         sub[u][r], S.open[2 * r + 1], upd, S.fO[r], S.hO[r], S.vO[r], pack[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++) pack[r] = __builtin_bitreverse32(pack[r]);
    if (own) {
      unsigned* const p = dmp + (long long)grp * stride;
      if (R == 1)
        p[0] = pack[0];
      else if (R == 2)
        *reinterpret_cast<uint2*>(p) = make_uint2(pack[0], pack[R > 1 ? 1 : 0]);
      else if (R == 3) {
        // three slots a lane may pass the row's end (a multiple of 8 slots)
        const int c = (e.k0 - e.k_first) >> 1;
#pragma unroll
        for (int r = 0; r < 3; r++)
          if (c + r < stride) p[r] = pack[r < R ? r : 0];
      } else
        *reinterpret_cast<uint4*>(p) = make_uint4(pack[0], pack[R > 1 ? 1 : 0],
                                                  pack[R > 2 ? 2 : 0], pack[R > 3 ? 3 : 0]);
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
}

template <int R, int NW>
__device__ __forceinline__ void ad_exchange(AdShared<NW>& S, AdState<R>& st, int buf, int w,
                                            int lane, bool active, bool in_round) {
  constexpr int H = DiagGeom<R, NW>::H;
  const bool lo = lane >= H && lane < 2 * H, hi = lane >= 64 - 2 * H && lane < 64 - H;
  if (active && (lo || hi)) {
    int* const q = S.halo[buf][w][lo ? 0 : 1] + (lo ? lane - H : lane - (64 - 2 * H)) * 6 * R;
#pragma unroll
    for (int r = 0; r < R; r++) {
      q[6 * r] = st.fE[r];
      q[6 * r + 1] = st.fO[r];
      q[6 * r + 2] = st.hE[r];
      q[6 * r + 3] = st.hO[r];
      q[6 * r + 4] = st.vE[r];
      q[6 * r + 5] = st.vO[r];
    }
  }
  __syncthreads();
  const bool fl = lane < H && w > 0, fr = lane >= 64 - H && w + 1 < NW;
  // every slot of a band lane, those outside the band too: nothing else would
  // clear what reached them from the wavefront's end (the other halo lanes
  // stay above kAdInf by their symbols)
  if (in_round && (fl || fr)) {
    const int* const q = fl ? S.halo[buf][w > 0 ? w - 1 : 0][1] + lane * 6 * R
                            : S.halo[buf][w + 1 < NW ? w + 1 : 0][0] + (lane - (64 - H)) * 6 * R;
#pragma unroll
    for (int r = 0; r < R; r++) {
      st.fE[r] = q[6 * r];
      st.fO[r] = q[6 * r + 1];
      st.hE[r] = q[6 * r + 2];
      st.hO[r] = q[6 * r + 3];
      st.vE[r] = q[6 * r + 4];
      st.vO[r] = q[6 * r + 5];
    }
  }
}

// One sweep (see dg_sweep): cost[m] and dcnt[m] are the round's cost and
// horizontal gap count.
template <int R, int NW>
__device__ __forceinline__ void ad_sweep(AdShared<NW>& S, int nd, int go,
                                         const uint8_t* __restrict__ sa,
                                         const uint8_t* __restrict__ sb, int L1, int L2,
                                         DiagSweep& sp, unsigned* dm, long long& slots) {
  typedef DiagGeom<R, NW> Geo;
  constexpr int H = Geo::H, U = Geo::U;
  const int w = NW == 1 ? 0 : (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int Dd = L2 - L1;
  const unsigned low = (1u << nd) - 1;
  const unsigned gos = (unsigned)go << nd;
  const int g = w * U + lane - H;
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
  const int k0 = in_round ? 2 * R * (g - g0) - newke : 0;
  const bool own = lane >= H && lane < 64 - H && in_round;
  const bool active = NW == 1 || w * U - H < used;
  const int stride = diag_stride(Dd, imax(newk, 0));
  unsigned* dmp = dm + dm0 + (in_round ? (g - g0) * R : 0);
  const int s_fin = L1 + L2 - 2;
  const int nblk = (s_fin >> 4) + 1;
  const int i00 = -(k0 >> 1);
  const int j00 = k0 >> 1;
  const int widee = (wide + 1) & ~1;
  const int k_last = imax(Dd + wide, -widee) + 2 * R;
  auto rows_in = [&](int b) {
    return -(k_last >> 1) - 1 + 8 * b >= 0 && (widee >> 1) + 8 * b + 7 < L1;
  };
  auto cols_in = [&](int b) {
    return -(widee >> 1) + R + 8 * b >= 0 && (k_last >> 1) + R + 1 + 8 * b + 7 < L2;
  };
  // a lane outside every round reads symbol 0
  const unsigned long long keep = in_round ? ~0ull : 0ull;
  unsigned long long rx[2], cx[2];
#pragma unroll
  for (int b = 0; b < 2; b++) {
    rx[b] = dg_load8(sa, L1, i00 + 8 * b, rows_in(b));
    cx[b] = dg_load8(sb, L2, j00 + R + 8 * b, cols_in(b));
  }
  AdState<R> st;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int ia = i00 - 1 - r, jb = j00 + r;
    st.A[r] = S.row[in_round && (unsigned)ia < (unsigned)L1 ? sa[ia] & 31 : 0];
    st.B[r] = S.col[in_round && (unsigned)jb < (unsigned)L2 ? sb[jb] & 31 : 0];
  }
  // Border values: row 0 holds go + the prefix sums of the prepend costs and
  // j horizontal gaps, column 0 go + the prefix sums of the extensions and
  // none; V can open from row 0, H never from column 0.  F runs as in
  // dg_sweep.
  DiagEdge edge;
  edge.k0 = k0;
  edge.k_first = -newke;
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
      if (in && k > 0) c = (int)(S.col[sb[k] & 31].cost >> nd);
      if (in && k < 0) c = -(int)(S.row[sa[-k] & 31].cost >> nd);
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
        const int z = __builtin_amdgcn_readlane(fz, lz);
        if (NW > 1) {
          if (w == wz && lane == 0) S.fin[m] = z;
        } else if (g0 == sp.start[m]) {
          zero = z;
        }
      }
    }
    if (NW > 1) {
      __syncthreads();
#pragma unroll
      for (int m = 0; m < kDgRounds; m++)
        if (m < sp.n && g0 == sp.start[m]) zero = S.fin[m];
      // (S.fin and S.scan are next written after further barriers)
    }
    // (the scan covers the owned lanes; a halo lane's border values come with
    // the first exchange)
    int F = NW == 1 || own ? ex - zero : 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int odd = 0; odd < 2; odd++) {
        const int k = k0 + 2 * r + odd;
        const bool in = in_round && k >= -newk && k <= Dd + newk;
        const int before = F;
        F += f[2 * r + odd];
        const unsigned val = k == 0 ? 0u : ((unsigned)(k < 0 ? before : F) << nd) + gos;
        const unsigned fv = !in ? (unsigned)kAdInf : val | (low - (unsigned)imax(k, 0));
        const unsigned mv = !in ? (unsigned)kAdInf : (k < 0 ? val : val + gos);
        st.open[2 * r + odd] = in ? gos : (unsigned)kAdInf;
        if (odd) {
          st.fO[r] = fv;
          st.hO[r] = kAdInf;
          st.vO[r] = mv;
        } else {
          st.fE[r] = fv;
          st.hE[r] = kAdInf;
          st.vE[r] = mv;
        }
      }
    }
  }
  const int s_inner = Dd + wide;
  for (int b = 0; b < nblk; b++) {
    if (NW > 1) ad_exchange<R, NW>(S, st, b & 1, w, lane, active, in_round);
    const unsigned long long rcur = rx[0] & keep, ccur = cx[0] & keep;
    rx[0] = rx[1];
    cx[0] = cx[1];
    if (active) {
      rx[1] = dg_load8(sa, L1, i00 + 8 * (b + 2), rows_in(b + 2));
      cx[1] = dg_load8(sb, L2, j00 + R + 8 * (b + 2), cols_in(b + 2));
      edge.s0 = 16 * b;
      if (edge.s0 > s_inner && edge.s0 + 15 <= s_fin)
        ad_block<R, NW, false>(st, S, low, rcur, ccur, edge, dmp, stride, own);
      else
        ad_block<R, NW, true>(st, S, low, rcur, ccur, edge, dmp, stride, own);
      dmp += 2 * stride;
    }
  }
#pragma unroll
  for (int m = 0; m < kDgRounds; m++) {
    if (m < sp.n) {
      const int kf = Dd + ((sp.newk[m] + 1) & ~1), cf = kf >> 1;
      const int gf = sp.start[m] + cf / R, rf = cf % R;
      const int wf = gf / U, lf = gf - wf * U + H;
      int v = 0;
#pragma unroll
      for (int r = 0; r < R; r++)
        if (r == rf) v = (kf & 1) ? (int)st.fO[r] : (int)st.fE[r];
      v = __builtin_amdgcn_readlane(v, lf);
      if (NW > 1) {
        if (w == wf && lane == 0) S.fin[m] = v;
      } else {
        sp.cost[m] = v >> nd;
        sp.dcnt[m] = (int)(low - ((unsigned)v & low));
      }
    }
  }
  if (NW > 1) {
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kDgRounds; m++) {
      if (m < sp.n) {
        const int v = __builtin_amdgcn_readfirstlane(S.fin[m]);
        sp.cost[m] = v >> nd;
        sp.dcnt[m] = (int)(low - ((unsigned)v & low));
      }
    }
    __syncthreads();
  }
  const int nact = NW == 1 ? 1 : imin(NW, (used + H + U - 1) / U);
  slots += (long long)nblk * 16 * 64 * R * nact;
}

// Fills the gap-free pairs (cls 1, or every pair without classes).  A pair
// that does not fit (no DP rows, a band wider than the lanes, directions
// larger than its region) is marked kAffLeft and counted in left_out for the
// stripe fill.
template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_affine_diag(AffFillArgs A) {
  __shared__ AdShared<NW> S;
  const int tid = threadIdx.x;
  if (A.left_in && __builtin_amdgcn_readfirstlane(*A.left_in) == 0) return;
  const int nd = A.nd;
  for (int k = tid; k < 1024; k += 64 * NW)
    S.tab[mw_ag_row(k >> 5) + (k & 31)] = A.cm->cost[k] << nd;
  if (tid < 32) {
    S.row[tid].off = (unsigned)(mw_ag_row(tid) * 4);
    S.row[tid].cost = tid == 0 ? kAdInf : A.cm->cost[(tid << 5) + kGap] << nd;
    S.col[tid].off = (unsigned)(tid * 4);
    S.col[tid].cost = tid == 0 ? kAdInf : A.cm->prepend[tid] << nd;
  }
  __syncthreads();
  const int delta = A.cm->delta, go = A.cm->gap_open;
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
    if (A.cls != nullptr && A.cls[pid] != 1) continue;
    PairResult r1;
    if (A.left_in) {
      r1 = A.res[pid];
      if (r1.full != kAffLeft) continue;
    }
    const uint8_t* sa = A.pt.blob + rows_off(A.pt, pid);
    const uint8_t* sb = A.pt.blob + cols_off(A.pt, pid);
    const int L1 = __builtin_amdgcn_readfirstlane(A.pt.len_a[pid]);
    const int L2 = __builtin_amdgcn_readfirstlane(A.pt.len_b[pid]);
    const int leni = L1 - 1, lenj = L2 - 1, Dd = lenj - leni;
    unsigned* dm = reinterpret_cast<unsigned*>(A.dm + A.pt.dm_off[pid]);
    const int64_t region = aff_dm_bytes(L1, L2);
    int T = (Dd + 1) * delta, rounds = 0;
    long long cells = 0, slots = 0;
    if (A.left_in) {
      T = __builtin_amdgcn_readfirstlane(r1.pad);
      rounds = __builtin_amdgcn_readfirstlane(r1.rounds);
      cells = r1.cells;
      slots = r1.slots;
    }
    int newk = 0, cost = 0, gap_num = 0, dm_word = 0;
    bool left = leni == 0;
    for (bool done = left; !done;) {
      const int p = (T - Dd) / 2;
      // rounds whose stop test cannot pass are skipped (see k_affine_fill)
      if (Dd >= p && (2 * T - Dd) / 2 - lenj + 1 < 0) {
        rounds++;
        T *= 2;
        continue;
      }
      DiagSweep sp;
      int R = 0, cap = 0, lanes = 0;
      int64_t words = 0;
      int Tm = T;
#pragma unroll
      for (int m = 0; m < kDgRounds; m++) {
        if (m == sp.n) {
          const int pm = (Tm - Dd) / 2;
          const int nk = pm >= leni ? leni - 1 : pm;
          const int c = diag_slots(Dd, nk);
          if (m == 0) {
            R = c <= DiagGeom<1, NW>::kLanes       ? 1
                : c <= 2 * DiagGeom<2, NW>::kLanes ? 2
                : c <= 3 * DiagGeom<3, NW>::kLanes ? 3
                                                   : 4;
            cap = R == 1   ? DiagGeom<1, NW>::kLanes
                  : R == 2 ? DiagGeom<2, NW>::kLanes
                  : R == 3 ? DiagGeom<3, NW>::kLanes
                           : DiagGeom<4, NW>::kLanes;
          }
          const int need = (c + R - 1) / R;
          const int at = m ? lanes + 1 : 0;
          const int64_t bytes = aff_diag_bytes(L1, L2, nk);
          if (at + need <= (m && NW == 16 ? imin(cap, 9 * DiagGeom<1, NW>::U) : cap) &&
              4 * words + bytes <= region) {
            sp.newk[m] = nk;
            sp.start[m] = at;
            sp.lanes[m] = need;
            sp.dm[m] = words;
            sp.n = m + 1;
            lanes = at + need;
            words += bytes / 4;
            if ((2 * Tm - Dd) / 2 - lenj + 1 >= 0) sp.n = -(m + 1);  // the last round
            Tm *= 2;
          }
        }
      }
      if (sp.n < 0) sp.n = -sp.n;
      left = sp.n == 0;
      if (left) break;
      if (R == 1)
        ad_sweep<1, NW>(S, nd, go, sa, sb, L1, L2, sp, dm, slots);
      else if (R == 2)
        ad_sweep<2, NW>(S, nd, go, sa, sb, L1, L2, sp, dm, slots);
      else if (R == 3)
        ad_sweep<3, NW>(S, nd, go, sa, sb, L1, L2, sp, dm, slots);
      else
        ad_sweep<4, NW>(S, nd, go, sa, sb, L1, L2, sp, dm, slots);
#pragma unroll
      for (int m = 0; m < kDgRounds; m++) {
        if (m < sp.n && !done) {
          const int pm = (T - Dd) / 2;
          newk = sp.newk[m];
          cost = sp.cost[m];
          gap_num = sp.dcnt[m];
          dm_word = (int)(sp.dm[m] >> 6);
          const long long rows = imax(0, leni - newk);
          cells += rows * (Dd + newk) + (leni - rows) * (long long)lenj + leni;
          rounds++;
          done = gap_num < pm || (2 * T - Dd) / 2 - lenj + 1 >= 0;
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
      r.full = left ? kAffLeft : kAffDiag;
      r.pad = T;
      r.cells = cells;
      r.slots = slots;
      A.res[pid] = r;
      if (left) atomicAdd(A.left_out, 1);
      else A.stab[A.pt.stab_off[pid]] = dm_word;
    }
    if (NW > 1) __syncthreads();
  }
}

}  // namespace poyhip
