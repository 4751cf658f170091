// colouring.hpp -- the constraint colouring of the coloured solver.
//
// Jones-Plassmann rounds over the constraint graph: a round's winners are the
// constraints whose (unique, hashed) priority is the largest among the still
// uncoloured ones at both their bodies; they share no body.  First fit,
// capped: the winners, in constraint order, each take the lowest colour that
// neither body has taken and that has fewer than the workgroup's width (at
// most 256) members (a colour is then one pass of the block); past 64 colours,
// one colour of their own per round.
//
// Rounds work on lists that shrink (the constraints left, and the round's
// winners, both in constraint order), not on all constraints again: a world
// of 11 236 contacts has 44 full colours, each settled in a pass of its own.
// What the passes touch at random -- per body the largest priority left and
// the colours taken -- is kept in LDS even where the lists are too long for
// it.
//
// Included by step_kernels.hip inside namespace odemi, after its workgroup
// helpers.
#pragma once

// Placement: everything in the LDS pool; the bodies' part of it; nothing.
enum { COL_IN_LDS = 0, COL_BODIES_LDS = 1, COL_IN_GLOBAL = 2 };

__device__ inline long long col_bodies_bytes(int nb) { return 12LL * nb; }
__device__ inline long long col_lists_bytes(int ncons) { return 20LL * ncons; }

// a constraint's priority: unique, hashed
__device__ inline int col_priority(int i) { return (int)(((unsigned)i * 2654435761u) & 0x7fffffffu); }

// Colours the constraints with rows and buckets them by colour, stably (index
// order inside a colour): the sweep result does not depend on the order inside
// a colour, but the block sums of the stopping test and the CG step do, so the
// layout is kept reproducible from run to run.  corder: the constraints by
// colour, cstart: the first of each colour and the end; returns the number of
// colours.  bmax, lists: the world's scratch (nb, and 5 ncons ints).
template <int PLACE>
__device__ __attribute__((noinline)) int colour_constraints(const Cons *cons, float *bt, int *bmax_g, int *lists_g,
                                                            LdsChar *pool, int nb, int ncons, int *corder, int *cstart,
                                                            Shared &sh) {
  cons = uniform_global(cons);
  bt = uniform_global(bt);
  corder = uniform_global(corder);
  cstart = uniform_global(cstart);
  nb = uniform(nb);
  ncons = uniform(ncons);
  char *const lds = (char *)uniform(pool);
  unsigned long long *const mask = (unsigned long long *)lds;   // colours taken at each body
  int *const bmax = PLACE == COL_IN_GLOBAL ? uniform_global(bmax_g) : (int *)(mask + nb);
  int *const col = PLACE == COL_IN_LDS ? bmax + nb : uniform_global(lists_g);
  int *const cb1 = col + ncons, *const cb2 = cb1 + ncons, *const left = cb2 + ncons, *const win = left + ncons;
  const int nt = blockDim.x, t = threadIdx.x, width = min(nt, COLOUR_WIDTH);
  auto taken = [&](int b) -> unsigned long long & {
    if constexpr (PLACE == COL_IN_GLOBAL) return *(unsigned long long *)(bt + 32 * b + 24);   // unused temp words
    else return mask[b];
  };
  // the lowest colour below 64 neither body has taken and that is not full
  auto first_free = [&](int i, unsigned long long full) {
    unsigned long long used = taken(cb1[i]) | full;
    if (cb2[i] >= 0) used |= taken(cb2[i]);
    return used == ~0ull ? 64 : __ffsll((long long)~used) - 1;
  };
  auto take = [&](int i, int c) {
    col[i] = c;
    taken(cb1[i]) |= 1ull << c;
    if (cb2[i] >= 0) taken(cb2[i]) |= 1ull << c;
  };
  for (int b = t; b < nb; b += nt) {
    bmax[b] = -1;
    taken(b) = 0ull;
  }
  // members of each of the first 64 colours, and the mask of full ones
  for (int k = t; k < 64; k += nt) sh.ccount[k] = 0;
  if (t == 0) sh.ival[9] = sh.ival[10] = 0;
  int nleft = 0;
  for (int start = 0; start < ncons; start += nt) {
    const int i = start + t;
    bool rows = false;
    if (i < ncons) {
      const Cons q = cons[i];
      rows = q.m > 0;
      col[i] = rows ? -1 : -2;
      cb1[i] = q.b1;
      cb2[i] = q.b2;
    }
    int tot;
    const int off = block_excl_scan(rows ? 1 : 0, tot, sh);
    if (rows) left[nleft + off] = i;
    nleft += tot;
  }
  __syncthreads();
  for (int round = 0; nleft > 0; round++) {
    // bmax: the largest priority left at each body.  A body whose largest one
    // did not win keeps it; the winners' bodies start over below.
    for (int x = t; x < nleft; x += nt) {
      const int i = left[x], pr = col_priority(i);
      atomicMax(&bmax[cb1[i]], pr);
      if (cb2[i] >= 0) atomicMax(&bmax[cb2[i]], pr);
    }
    __syncthreads();
    int nwin = 0, nkeep = 0;
    for (int start = 0; start < nleft; start += nt) {
      const int x = start + t, i = x < nleft ? left[x] : 0;
      bool w = false;
      if (x < nleft) {
        const int pr = col_priority(i);
        w = bmax[cb1[i]] == pr && (cb2[i] < 0 || bmax[cb2[i]] == pr);
      }
      // places of the winners (low half) and of the others; the reads of this
      // stretch of `left` are done before the scan's barriers, and it only
      // moves forward
      int tot;
      const int off = block_excl_scan(x < nleft ? (w ? 1 : 1 << 16) : 0, tot, sh);
      if (x < nleft) {
        if (w) win[nwin + (off & 0xffff)] = i;
        else left[nkeep + (off >> 16)] = i;
      }
      nwin += tot & 0xffff;
      nkeep += tot >> 16;
    }
    nleft = nkeep;
    __syncthreads();
    for (int x = t; x < nwin; x += nt) {
      const int i = win[x];
      bmax[cb1[i]] = -1;
      if (cb2[i] >= 0) bmax[cb2[i]] = -1;
    }
    // Colours are settled in increasing order: below the lowest colour the
    // winners would overfill every proposal stands; that colour goes to its
    // first proposers in constraint order and is full, and the rest propose
    // again.  A winner's proposal only rises, and a round's winners share no
    // body (each mask has one writer per round), so this equals the sequential
    // assignment.
    while (true) {
      const unsigned long long full = ((unsigned long long)(unsigned)sh.ival[10] << 32) | (unsigned)sh.ival[9];
      for (int k = t; k < 64; k += nt) sh.ccur[k] = 0;
      __syncthreads();
      for (int x = t; x < nwin; x += nt) {
        const int i = win[x];
        if (col[i] != -1) continue;
        const int p = first_free(i, full);
        if (p < 64) atomicAdd(&sh.ccur[p], 1);
      }
      __syncthreads();
      if (t < 64) {
        const unsigned long long over = __ballot(sh.ccount[t] + sh.ccur[t] > width);
        if (t == 0) sh.ival[8] = over ? __ffsll((long long)over) - 1 : 64;
      }
      __syncthreads();
      const int cs = sh.ival[8];
      for (int x = t; x < nwin; x += nt) {
        const int i = win[x];
        if (col[i] != -1) continue;
        const int p = first_free(i, full);
        if (p < cs) take(i, p);
        else if (p >= 64) col[i] = 64 + round;
      }
      for (int k = t; k < cs; k += nt) sh.ccount[k] += sh.ccur[k];
      if (cs == 64) break;
      const int room = width - sh.ccount[cs];
      int base = 0;
      for (int start = 0; start < nwin && base < room; start += nt) {
        const int x = start + t, i = x < nwin ? win[x] : 0;
        const bool want = x < nwin && col[i] == -1 && first_free(i, full) == cs;
        int tot;
        const int r = base + block_excl_scan(want ? 1 : 0, tot, sh);
        if (want && r < room) take(i, cs);
        base += tot;
      }
      __syncthreads();
      if (t == 0) {
        sh.ccount[cs] = width;
        if (cs < 32) sh.ival[9] |= (int)(1u << cs);
        else sh.ival[10] |= (int)(1u << (cs - 32));
      }
      __syncthreads();
    }
    __syncthreads();
  }
  int mc = -1;
  for (int i = t; i < ncons; i += nt) mc = max(mc, col[i]);
  const int ngroups = (int)block_max((float)mc, sh) + 1;
  if (ngroups <= MAX_COLORS_LDS) {
    for (int k = t; k <= ngroups; k += nt) sh.ccount[k] = 0;
    __syncthreads();
    for (int i = t; i < ncons; i += nt)
      if (col[i] >= 0) atomicAdd(&sh.ccount[col[i]], 1);
    __syncthreads();
    int base = 0;
    for (int k0 = 0; k0 <= ngroups; k0 += nt) {
      const int k = k0 + t;
      int tot;
      const int off = base + block_excl_scan(k < ngroups ? sh.ccount[k] : 0, tot, sh);
      if (k <= ngroups) cstart[k] = off;
      if (k < ngroups) sh.ccur[k] = off;
      base += tot;
    }
    __syncthreads();
    // stably: the rank among a wavefront's equal colours from ballots, the
    // wavefronts of a stretch one after another
    const int lane = t & 63, wid = t >> 6, nw = (nt + 63) >> 6;
    for (int start = 0; start < ncons; start += nt) {
      const int i = start + t;
      const int ci = i < ncons ? col[i] : -1;
      unsigned long long peers = __ballot(ci >= 0);
      for (int b = 0; (1 << b) < ngroups; b++) {
        const unsigned long long m = __ballot((ci >> b) & 1);
        peers &= ((ci >> b) & 1) ? m : ~m;
      }
      const int rank = __popcll(peers & ((1ull << lane) - 1)), cnt = __popcll(peers);
      for (int w = 0; w < nw; w++) {
        if (w == wid && ci >= 0) {
          const int at = sh.ccur[ci];
          corder[at + rank] = i;
          if (rank == cnt - 1) sh.ccur[ci] = at + cnt;
        }
        lds_barrier();
      }
    }
  } else if (t == 0) {
    for (int k = 0; k <= ngroups; k++) cstart[k] = 0;
    for (int i = 0; i < ncons; i++)
      if (col[i] >= 0) cstart[col[i] + 1]++;
    for (int k = 0; k < ngroups; k++) cstart[k + 1] += cstart[k];
    int *cur = cstart + ngroups + 1;
    for (int k = 0; k < ngroups; k++) cur[k] = cstart[k];
    for (int i = 0; i < ncons; i++)
      if (col[i] >= 0) corder[cur[col[i]]++] = i;
  }
  __syncthreads();
  return ngroups;
}
