// Union merge of POY's implied-alignment unions (src/union.c: union_merge
// 170, behind union_CAML_make 318) on gfx950.
//
// A merge walks the two children's aligned sequences and their unions from
// the right, prepending the new union's symbols and writing its offset and
// child-offset arrays; the steps depend on each other through five cursors.
// One wavefront runs one merge, up to 64 columns at a time (un_chunk): where
// the unions' counts form whole runs, a column's cursors follow from bit
// counts over the columns right of it, and only what does not (a cursor
// that runs out, a run longer than the wavefront, counts of another shape,
// the closing column) is walked column by column (un_column).  A union is a sequence right-aligned in
// `cap` bytes of the byte blob plus three int32 arrays of `cap` entries in
// the int blob (offset, union_c1, union_c2), their live part at the right
// end; the child unions need only their sequence and offsets.
#include "poyhip.h"
#include "poyhip_device.h"

namespace poyhip {

struct UnCursor {
  const uint8_t* s;  // sequence buffer (cap bytes)
  int cap, len;
  int end, position;  // offset-array and sequence cursors
};

struct UnOut {
  uint8_t* s;
  int32_t *off, *ca, *cb;
  int cap, len;
  int end, pca, pcb;
  int last;  // the symbol prepended last
};

__device__ __forceinline__ int un_get(const UnCursor& u, int pos) {
  return u.s[u.cap - u.len + pos];
}

// seq_prepend (src/seq.c:155); false when the capacity is exhausted
__device__ __forceinline__ bool un_prepend(UnOut& c, int v) {
  if (c.len >= c.cap) return false;
  c.len++;
  c.s[c.cap - c.len] = (uint8_t)v;
  c.last = v;
  return true;
}

// union_prepend_item (src/union.c:79)
__device__ __forceinline__ bool un_item(UnCursor& src, UnOut& c, int v) {
  if (src.position >= 0) {
    v |= un_get(src, src.position);
    src.position--;
    src.end--;
  }
  return un_prepend(c, v);
}

// union_prepend_and_fill_items (src/union.c:136): the counts prep..1 of the
// items prepended since the last fill, their child offsets 0, then the
// column's symbol with the children's positions (the new union is cleared
// before the walk, so writes of 0 only move a cursor)
__device__ __forceinline__ bool un_fill(UnOut& c, int interm, int prep, int apos, int bpos) {
  if (c.end - prep < 0 || c.pca - prep < 0 || c.pcb - prep < 0) return false;
  for (int i = prep; i > 0; i--) c.off[c.end--] = i;
  c.pca -= prep;
  c.pcb -= prep;
  if (apos != 0) c.ca[c.pca] = apos;
  if (bpos != 0) c.cb[c.pcb] = bpos;
  c.pca--;
  c.pcb--;
  const bool ok = un_prepend(c, interm);
  c.end--;  // offset 0
  return ok;
}

struct UnJob {
  const uint8_t *a, *b, *median;
  const int32_t *aoff, *boff;
  int abeg, bbeg;  // first live entries; a union holds items while begin <= end
};

enum { kUnGoes, kUnEnds, kUnFails };

// One column of union_merge (src/union.c:170-274); i moves left.  Fails
// where the reference fails (the aligned sequences end while a union still
// has items) or the new union's capacity is exhausted.
__device__ __forceinline__ int un_column(const UnJob& J, UnCursor& au, UnCursor& bu, UnOut& c,
                                         int& items, int& i) {
  const int gap = kGap;
  if (c.end < 0 || c.pca < 0 || c.pcb < 0) return kUnFails;
  // union_copy_non_homologous (src/union.c:118): the count at each child's
  // cursor is the number of its items copied across as they are
  const int ka = au.position > -1 ? J.aoff[au.end] : 0;
  const int kb = bu.position > -1 ? J.boff[bu.end] : 0;
  items += ka;
  for (int k = ka; k > 0; k--)
    if (!un_item(au, c, gap)) return kUnFails;
  items += kb;
  for (int k = kb; k > 0; k--)
    if (!un_item(bu, c, gap)) return kUnFails;
  if (i < 0) return kUnFails;  // "infinit loop" in the reference
  int interm = J.median[i];
  const int ai = J.a[i], bi = J.b[i];
  if (interm == gap) {
    if (i == 0) {
      if (!un_fill(c, gap, items, 0, 0)) return kUnFails;
      au.end--;
      bu.end--;
      return kUnEnds;
    }
    bool ok;
    if (ai == gap) ok = un_item(bu, c, gap);
    else if (bi == gap) ok = un_item(au, c, gap);
    else {
      // union_prepend_pair (src/union.c:38)
      int v = gap;
      if (au.position >= 0) {
        v |= un_get(au, au.position);
        au.position--;
        au.end--;
      }
      ok = un_item(bu, c, v);
    }
    if (!ok) return kUnFails;
    items += 1;
  } else {
    int apos = 0, bpos = 0;
    // union_move_left (src/union.c:161) as the three cases call it; in the
    // last case each guard tests the other union's cursor, as written: a
    // guard that passes with the union's own cursor below 0 reads the byte
    // before its live part, as the reference does
    const bool ma = ai != gap, mb = ai == gap || bi != gap;
    if (mb) bpos = bu.position;
    if (ma) apos = au.position;
    if (ma && (mb ? bpos : apos) >= 0) {
      interm |= un_get(au, au.position);
      au.position--;
      au.end--;
    }
    if (mb && (ma ? apos : bpos) >= 0) {
      interm |= un_get(bu, bu.position);
      bu.position--;
      bu.end--;
    }
    if (!un_fill(c, interm, items, apos, bpos)) return kUnFails;
    items = 0;
  }
  i--;
  return kUnGoes;
}

struct UnShared {
  int zero[2][64];   // window lane of a child's m-th entry without a count
  int col[2][64];    // the column lane that copies the items before it
  int at[64];        // a column's first prepend
  int pre[2][64];    // the items a column copies from each child
  int fill[64];      // prepend index of the first filled column from here on
};

// Up to 64 columns at once: lane l looks at column i - l and, for each child,
// at the entry l left of its cursor.  Counts that run k, k-1, .., 1, 0
// leftwards are items of one copy; the entries of count 0 are taken in order
// by the columns that move the child's cursor, so a column's entry is the
// m-th one, m the number of such columns right of it, and it copies the
// items in front of that entry if it is the first column to reach them.
// Returns the number of columns done, a prefix of those looked at: up to one
// whose entry is not in the window, whose child has run out though it moves,
// that finds both run out, that would close the merge or pass the capacity.
__device__ __forceinline__ int un_chunk(UnShared& S, const UnJob& J, UnCursor& au, UnCursor& bu,
                                        UnOut& c, int& items, int& i) {
  const int lane = threadIdx.x & 63;
  const lmask below = ((lmask)1 << lane) - 1;
  const int gap = kGap;
  const int ci = i - lane;
  const bool here = ci >= 0;
  const int med = here ? J.median[ci] : gap;
  const int ai = here ? J.a[ci] : gap;
  const int bi = here ? J.b[ci] : gap;
  const bool live[2] = {lane <= au.position, lane <= bu.position};
  const int cnt[2] = {live[0] ? J.aoff[au.end - lane] : -1, live[1] ? J.boff[bu.end - lane] : -1};
  const int sym[2] = {live[0] ? un_get(au, au.position - lane) : 0,
                      live[1] ? un_get(bu, bu.position - lane) : 0};
  const int pos[2] = {au.position, bu.position};
  const bool move[2] = {ai != gap, ai == gap || bi != gap};
  __syncthreads();  // the tables' last readers are done
  int nz[2], rank[2], lim[2];
  bool head[2];
#pragma unroll
  for (int x = 0; x < 2; x++) {
    const int next = __shfl_down(cnt[x], 1);
    const bool good = cnt[x] == 0 || (cnt[x] > 0 && lane < 63 && next == cnt[x] - 1);
    const lmask bad = ~ballot(good);
    lim[x] = bad ? __builtin_ctzll(bad) : 64;
    const lmask zeros = ballot(cnt[x] == 0 && lane < lim[x]);
    nz[x] = __builtin_popcountll(zeros);
    if ((zeros >> lane) & 1) S.zero[x][__builtin_popcountll(zeros & below)] = lane;
    const lmask moves = ballot(move[x]);
    rank[x] = __builtin_popcountll(moves & below);
    head[x] = lane == 0 || ((moves >> (lane - 1)) & 1);
    if (head[x]) S.col[x][rank[x]] = lane;
  }
  __syncthreads();
  int cur[2], pre[2], z[2];
  bool out[2];
  bool ok = here && !(ci == 0 && med == gap);
#pragma unroll
  for (int x = 0; x < 2; x++) {
    // the child's cursor as this column finds it
    cur[x] = rank[x] == 0 ? 0 : rank[x] <= nz[x] ? S.zero[x][rank[x] - 1] + 1 : 64;
    out[x] = cur[x] > pos[x];
    const bool in = rank[x] < nz[x];
    z[x] = in ? S.zero[x][rank[x]] : cur[x];
    pre[x] = in && head[x] ? z[x] - cur[x] : 0;
    ok = ok && rank[x] <= nz[x] && (in || (out[x] && !move[x]));
  }
  ok = ok && !(out[0] && out[1]);
  const int step = ok ? 1 + pre[0] + pre[1] : 0;
  int total;
  const int at = c.len + wave_excl_sum_lane(step, lane, total);
  ok = ok && at + step <= c.cap;
  const lmask stop = ~ballot(ok);
  const int n = stop ? __builtin_ctzll(stop) : 64;
  if (n == 0) return 0;
  const bool mine = lane < n;
  const int f = at + pre[0] + pre[1];  // this column's own prepend
  const bool fills = mine && med != gap;
  const lmask fm = ballot(fills);
  S.at[lane] = at;
  S.pre[0][lane] = pre[0];
  S.pre[1][lane] = pre[1];
  const lmask ahead = fm & ~below;
  const int fnext = __shfl(f, ahead ? __builtin_ctzll(ahead) : 0);
  S.fill[lane] = ahead ? fnext : -1;
  const int sa = __shfl(sym[0], z[0] & 63), sb = __shfl(sym[1], z[1] & 63);
  __syncthreads();
  int v = med;
  if (mine) {
    if (move[0]) v |= sa;
    if (move[1]) v |= sb;
    const int k = c.cap - 1 - f;
    c.s[k] = (uint8_t)v;
    if (fills) {
      const int apos = move[0] ? pos[0] - z[0] : 0, bpos = move[1] ? pos[1] - z[1] : 0;
      if (apos != 0) c.ca[k] = apos;
      if (bpos != 0) c.cb[k] = bpos;
    } else if (S.fill[lane] >= 0) {
      c.off[k] = S.fill[lane] - f;
    }
  }
  // the copied items, by the lanes that hold their entries
#pragma unroll
  for (int x = 0; x < 2; x++) {
    const lmask zeros = ballot(cnt[x] == 0 && lane < lim[x]);
    const lmask moves = ballot(move[x]);
    const int m = __builtin_popcountll(zeros & below);
    if (cnt[x] > 0 && lane < lim[x] && m <= (int)__builtin_popcountll(moves << 1)) {
      const int j = S.col[x][m];
      if (j < n) {
        const int p = S.at[j] + (x ? S.pre[0][j] : 0) + S.pre[x][j] - cnt[x];
        const int k = c.cap - 1 - p;
        c.s[k] = (uint8_t)(gap | sym[x]);
        if (S.fill[j] >= 0) c.off[k] = S.fill[j] - p;
      }
    }
  }
  // items of earlier columns wait for the first filled column
  if (fm) {
    const int f0 = __shfl(f, __builtin_ctzll(fm));
    for (int p = c.len - items + lane; p < c.len; p += 64) c.off[c.cap - 1 - p] = f0 - p;
  }
  const int e = n - 1;
  const int len = __builtin_amdgcn_readlane(f, e) + 1;
  const int flast = fm ? __builtin_amdgcn_readlane(f, 63 - __builtin_clzll(fm)) : 0;
  items = fm ? len - 1 - flast : items + len - c.len;
  c.last = __builtin_amdgcn_readlane(v, e) & 255;
  c.len = len;
  c.end = c.pca = c.pcb = c.cap - 1 - len + items;
  const int da = __builtin_amdgcn_readlane(z[0] + (move[0] ? 1 : 0), e);
  const int db = __builtin_amdgcn_readlane(z[1] + (move[1] ? 1 : 0), e);
  au.position -= da;
  au.end -= da;
  bu.position -= db;
  bu.end -= db;
  i -= n;
  return n;
}

// union_merge (src/union.c:170-274) by a wavefront; `chunks` allows whole
// runs of columns at once.
__device__ __forceinline__ bool union_merge_one(UnShared& S, const UnJob& J, int lena,
                                                UnCursor& au, UnCursor& bu, UnOut& c,
                                                bool chunks) {
  int items = 0;
  int i = lena - 1;
  int walk = 1;  // columns to walk after a chunk that did none
  while (J.abeg <= au.end || J.bbeg <= bu.end) {
    // a chunk takes the pending items for the last prepends
    if (chunks && i >= 0 && items >= 0 && c.end == c.cap - 1 - c.len + items && c.pca == c.end &&
        c.pcb == c.end) {
      if (un_chunk(S, J, au, bu, c, items, i) > 0) {
        walk = 1;
        continue;
      }
    }
    for (int k = 0; k < walk && (J.abeg <= au.end || J.bbeg <= bu.end); k++) {
      const int r = un_column(J, au, bu, c, items, i);
      if (r != kUnGoes) return r == kUnEnds;
    }
    walk = imin(2 * walk, 64);
  }
  if (c.len == 0 || c.last != kGap) {
    if (c.end < 0 || c.pca < 0 || c.pcb < 0 || !un_prepend(c, kGap)) return false;
  }
  return true;
}

// every range the job names lies inside its blob
__device__ __forceinline__ bool un_in(int64_t off, int64_t n, int64_t size) {
  return off >= 0 && n >= 0 && off <= size && n <= size - off;
}

__device__ __forceinline__ bool un_job_fits(const poyhip_union_job& J, int64_t seq_bytes,
                                            int64_t n_ints) {
  return J.lena >= 0 && J.ua_len >= 0 && J.ub_len >= 0 && J.ua_cap >= 1 && J.ub_cap >= 1 &&
         J.c_cap >= 1 && J.ua_len <= J.ua_cap && J.ub_len <= J.ub_cap &&
         un_in(J.a, J.lena, seq_bytes) && un_in(J.b, J.lena, seq_bytes) &&
         un_in(J.median, J.lena, seq_bytes) && un_in(J.ua_s, J.ua_cap, seq_bytes) &&
         un_in(J.ub_s, J.ub_cap, seq_bytes) && un_in(J.c_s, J.c_cap, seq_bytes) &&
         un_in(J.ua_off, J.ua_cap, n_ints) && un_in(J.ub_off, J.ub_cap, n_ints) &&
         un_in(J.c_off, J.c_cap, n_ints) && un_in(J.c_c1, J.c_cap, n_ints) &&
         un_in(J.c_c2, J.c_cap, n_ints);
}

__device__ __forceinline__ bool un_meet(int64_t x, int64_t nx, int64_t y, int64_t ny) {
  return x < y + ny && y < x + nx;
}

// the new union lies apart from what the merge reads, and its arrays apart
// from each other (a chunk reads ahead of what it writes)
__device__ __forceinline__ bool un_apart(const poyhip_union_job& J) {
  const int64_t n = J.c_cap;
  return !(un_meet(J.c_s, n, J.a, J.lena) || un_meet(J.c_s, n, J.b, J.lena) ||
           un_meet(J.c_s, n, J.median, J.lena) || un_meet(J.c_s, n, J.ua_s, J.ua_cap) ||
           un_meet(J.c_s, n, J.ub_s, J.ub_cap) || un_meet(J.c_off, n, J.c_c1, n) ||
           un_meet(J.c_off, n, J.c_c2, n) || un_meet(J.c_c1, n, J.c_c2, n) ||
           un_meet(J.c_off, n, J.ua_off, J.ua_cap) || un_meet(J.c_off, n, J.ub_off, J.ub_cap) ||
           un_meet(J.c_c1, n, J.ua_off, J.ua_cap) || un_meet(J.c_c1, n, J.ub_off, J.ub_cap) ||
           un_meet(J.c_c2, n, J.ua_off, J.ua_cap) || un_meet(J.c_c2, n, J.ub_off, J.ub_cap));
}

// One wavefront (one 64-thread block) takes one merge.  It first clears the
// new union with coalesced stores (entries the merge does not write are 0;
// the reference leaves them uninitialised).
//
// What bounds it: the longest merge's chain of chunks, each a round trip to
// memory and some 150 instructions.  Columns walked one by one by a lane,
// four merges to a wavefront, took 5.6 ms for 4,096 merges of 50-5,000
// columns; in chunks they take 0.20 ms.
__global__ __launch_bounds__(64) void k_union_merge(const poyhip_union_job* jobs, int n,
                                                    uint8_t* seq, int64_t seq_bytes,
                                                    int32_t* ints, int64_t n_ints, int* c_len,
                                                    int* status) {
  __shared__ UnShared S;
  const int lane = threadIdx.x;
  const int k = blockIdx.x;
  if (k >= n) return;
  const poyhip_union_job& Q = jobs[k];
  if (!un_job_fits(Q, seq_bytes, n_ints)) {
    if (lane == 0) {
      c_len[k] = 0;
      status[k] = POYHIP_EINVAL;
    }
    return;
  }
  UnOut c;
  c.s = seq + Q.c_s;
  c.off = ints + Q.c_off;
  c.ca = ints + Q.c_c1;
  c.cb = ints + Q.c_c2;
  c.cap = Q.c_cap;
  c.len = 0;
  c.last = 0;
  c.end = c.pca = c.pcb = c.cap - 1;
  for (int q = lane; q < c.cap; q += 64) {
    c.s[q] = 0;
    c.off[q] = 0;
    c.ca[q] = 0;
    c.cb[q] = 0;
  }
  // the clearing stores complete before any lane writes the union
  __syncthreads();
  UnCursor au, bu;
  au.s = seq + Q.ua_s;
  au.cap = Q.ua_cap;
  au.len = Q.ua_len;
  au.end = au.cap - 1;
  au.position = au.len - 1;
  bu.s = seq + Q.ub_s;
  bu.cap = Q.ub_cap;
  bu.len = Q.ub_len;
  bu.end = bu.cap - 1;
  bu.position = bu.len - 1;
  UnJob J;
  J.a = seq + Q.a;
  J.b = seq + Q.b;
  J.median = seq + Q.median;
  J.aoff = ints + Q.ua_off;
  J.boff = ints + Q.ub_off;
  // begin cursors stay put
  J.abeg = au.len == 0 ? au.cap - 1 : au.cap - au.len;
  J.bbeg = bu.len == 0 ? bu.cap - 1 : bu.cap - bu.len;
  const bool chunks = au.len > 0 && bu.len > 0 && un_apart(Q);
  const bool ok = union_merge_one(S, J, Q.lena, au, bu, c, chunks);
  if (lane == 0) {
    c_len[k] = c.len;
    status[k] = ok ? POYHIP_OK : POYHIP_EINVAL;
  }
}

}  // namespace poyhip
