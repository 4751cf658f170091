// ref_order.hpp -- the reference's constraint and row order of one world
// (ode/src/util.cpp:420-487, quickstep.cpp:473-482, 670-830): islands by a
// depth-first walk from the newest body, each body's constraints newest
// attach first, rows in island order, every island's generator state.
//
// Only the walk itself is one lane's; its steps are dependent LDS accesses
// (about 250 cycles an adjacency entry), so it reads one word per entry (the
// constraint and its other body) ahead of the step that needs it, and
// everything around it is done by all lanes: the bodies' lists (each entry
// counts the newer ones in its list), row offsets (a scan over the walk's
// order), generator states (skipped ahead by the draws of the islands before)
// and Info2's running erp.
//
// Included by step_kernels.hip inside namespace odemi, after its workgroup
// helpers.
#pragma once

// flags of a constraint: its rows, whether the walk takes it, whether it has
// met it
enum { RO_ROWS = 7, RO_ENABLED = 8, RO_IN = 16, RO_OUT = 32 };

// LDS bytes: per constraint two adjacency words, two unsorted entries (then
// its place in the order), sequence number (then row offset) and flags; per
// body list start, cursor (then the stack), tag and island
__device__ inline long long ref_order_lds_bytes(int nb, int ncons) {
  return 17LL * ncons + 13LL * nb + 64;
}

// Orders cons[0, ncons), nk contacts first.  Writes corder (constraints in
// island order), after it the bodies in visit order, the island table isl
// ([cons0, ncons, row0, nrows, seed] each), each constraint's row0 (m = 0 where
// no island has it) and erp, misc[0..3] (rows, islands, ordered constraints,
// visited bodies) and the world's next generator state.  ncons, nb < 65535.
__device__ __attribute__((noinline)) void ref_order_lds(Cons *cons, const JointDev *joints, const float *invMass,
                                                        WorldParams *P, int nb, int nk, int ncons, bool host, int *corder,
                                                        int *isl, float *erp_out, int *misc, LdsChar *pool,
                                                        Shared &sh) {
  cons = uniform_global(cons);
  joints = uniform_global(joints);
  invMass = uniform_global(invMass);
  P = uniform_global(P);
  corder = uniform_global(corder);
  isl = uniform_global(isl);
  erp_out = uniform_global(erp_out);
  misc = uniform_global(misc);
  nb = uniform(nb);
  nk = uniform(nk);
  ncons = uniform(ncons);
  host = uniform(host);
  const int nt = blockDim.x, t = threadIdx.x;
  unsigned *adj = (unsigned *)(char *)uniform(pool);      // constraint | other body << 16 (0xffff: none)
  int *cseq = (int *)(adj + 2 * ncons), *pre = cseq;      // sequence number, then row offset by place
  int *adjs = cseq + ncons;                               // nb + 1
  int *fill = adjs + nb + 1;                              // cursors, then the stack
  unsigned short *adju = (unsigned short *)(fill + nb), *cord = adju;   // unsorted lists, then the order
  unsigned short *icons = adju + 2 * ncons, *icnt = icons + nb;         // island: first constraint, count
  unsigned char *flag = (unsigned char *)(icnt + nb), *tag = flag + ncons;
  int *border = corder + ncons;
  for (int b = t; b <= nb; b += nt) adjs[b] = 0;
  __syncthreads();
  // Constraints with rows, and contacts, are in their bodies' lists.  Newest
  // is the largest sequence number; contacts of the host count in the order
  // they were created, a joint after the last of them that is not newer (so a
  // contact's number is the least from it on), which the device's contacts
  // are in anyway.
  for (int i = t; i < ncons; i += nt) {
    const Cons q = cons[i];
    cseq[i] = q.seq;
    int f = q.m > 0 ? q.m : 0;
    if (q.b1 >= 0 && (q.m > 0 || q.kind == JT_CONTACT)) {
      if (invMass[q.b1] > 0.f || (q.b2 >= 0 && invMass[q.b2] > 0.f)) f |= RO_ENABLED;
      atomicAdd(&adjs[q.b1 + 1], 1);
      if (q.b2 >= 0) atomicAdd(&adjs[q.b2 + 1], 1);
    }
    flag[i] = (unsigned char)f;
  }
  __syncthreads();
  {
    const int per = (nb + 1 + nt - 1) / nt, d0 = min(t * per, nb + 1), d1 = min(d0 + per, nb + 1);
    int loc = 0;
    for (int d = d0; d < d1; d++) loc += adjs[d];
    int tot;
    int run = block_excl_scan(loc, tot, sh);
    for (int d = d0; d < d1; d++) { run += adjs[d]; adjs[d] = run; }
  }
  __syncthreads();
  for (int b = t; b < nb; b += nt) {
    fill[b] = adjs[b];
    tag[b] = 0;
  }
  __syncthreads();
  if (host) {
    int *least = (int *)adju;   // of each lane's stretch
    const int per = (nk + nt - 1) / nt, x0 = min(t * per, nk), x1 = min(x0 + per, nk);
    int run = 0x7fffffff;
    for (int x = x0; x < x1; x++) run = min(run, cseq[x]);
    if (x0 < x1) least[t] = run;
    __syncthreads();
    run = 0x7fffffff;
    for (int u = t + 1; u * per < nk; u++) run = min(run, least[u]);
    for (int x = x1 - 1; x >= x0; x--) cseq[x] = run = min(run, cseq[x]);
    __syncthreads();
  }
  auto in_lists = [](const Cons &q) { return q.b1 >= 0 && (q.m > 0 || q.kind == JT_CONTACT); };
  for (int i = t; i < ncons; i += nt) {
    const Cons q = cons[i];
    if (!in_lists(q)) continue;
    adju[atomicAdd(&fill[q.b1], 1)] = (unsigned short)i;
    if (q.b2 >= 0) adju[atomicAdd(&fill[q.b2], 1)] = (unsigned short)i;
  }
  __syncthreads();
  // newest first (body joint lists prepend, ode.cpp:1382-1389)
  for (int i = t; i < ncons; i += nt) {
    const Cons q = cons[i];
    if (!in_lists(q)) continue;
    const int si = cseq[i];
    for (int side = 0; side < 2; side++) {
      const int b = side ? q.b2 : q.b1, o = side ? q.b1 : q.b2;
      if (b < 0) continue;
      int at = adjs[b];
      const int e = adjs[b + 1];
      for (int k = adjs[b]; k < e; k++) {
        const int c = adju[k], sc = cseq[c];
        at += sc > si || (sc == si && c > i);
      }
      adj[at] = (unsigned)i | (unsigned)(o >= 0 ? o : 0xffff) << 16;
    }
  }
  __syncthreads();
  int *stack = fill;
  if (t == 0) {
    int nic = 0, nib = 0, nisl = 0;
    for (int bb = nb - 1; bb >= 0; bb--) {
      if (tag[bb]) continue;
      tag[bb] = 1;
      const int c0 = nic;
      border[nib++] = bb;
      int sp = 0, b = bb;
      while (true) {
        const int k1 = adjs[b + 1];
        int k = adjs[b];
        unsigned next = k < k1 ? adj[k] : 0;
        for (; k < k1; k++) {
          const unsigned a = next;
          if (k + 1 < k1) next = adj[k + 1];
          const int qi = (int)(a & 0xffff), other = (int)(a >> 16);
          const int f = flag[qi], seen = other != 0xffff ? tag[other] : 1;
          if (f & (RO_IN | RO_OUT)) continue;
          if (!(f & RO_ENABLED)) { flag[qi] = (unsigned char)(f | RO_OUT); continue; }
          flag[qi] = (unsigned char)(f | RO_IN);
          cord[nic++] = (unsigned short)qi;
          if (!seen) {
            tag[other] = 1;
            stack[sp++] = other;
          }
        }
        if (sp == 0) break;
        b = stack[--sp];
        border[nib++] = b;
      }
      icons[nisl] = (unsigned short)c0;
      icnt[nisl] = (unsigned short)(nic - c0);
      nisl++;
    }
    sh.ival[5] = nic;
    sh.ival[6] = nisl;
    sh.ival[7] = nib;
  }
  __syncthreads();
  const int nic = uniform(sh.ival[5]), nisl = uniform(sh.ival[6]), nib = uniform(sh.ival[7]);
  int nrows = 0;
  for (int x0 = 0; x0 < nic; x0 += nt) {
    const int x = x0 + t, i = x < nic ? cord[x] : 0;
    int tot;
    const int off = nrows + block_excl_scan(x < nic ? (int)(flag[i] & RO_ROWS) : 0, tot, sh);
    if (x < nic) {
      pre[x] = off;
      corder[x] = i;
      cons[i].row0 = off;
    }
    nrows += tot;
  }
  for (int i = t; i < ncons; i += nt)
    if (!(flag[i] & RO_IN)) cons[i].m = 0;
  __syncthreads();
  // generator states: an island with m rows makes ceil(iterations / 8) (m - 1)
  // draws
  const unsigned seed = P->seed;
  const unsigned long long shuffles = (unsigned long long)((P->iterations + 7) / 8);
  unsigned long long draws = 0;
  for (int k0 = 0; k0 < nisl; k0 += nt) {
    const int k = k0 + t;
    int c0 = 0, cn = 0, r0 = 0, m = 0;
    if (k < nisl) {
      c0 = icons[k];
      cn = icnt[k];
      r0 = c0 < nic ? pre[c0] : nrows;
      m = (c0 + cn < nic ? pre[c0 + cn] : nrows) - r0;
    }
    int tot;
    const int off = block_excl_scan(m > 1 ? m - 1 : 0, tot, sh);
    if (k < nisl) {
      isl[5 * k + 0] = c0;
      isl[5 * k + 1] = cn;
      isl[5 * k + 2] = r0;
      isl[5 * k + 3] = m;
      isl[5 * k + 4] = (int)lcg_skip(seed, shuffles * (draws + (unsigned long long)off));
    }
    draws += (unsigned long long)tot;
  }
  // Info2's erp is reset per island; a ball joint sets it for the constraints
  // after it (quickstep.cpp:777-779)
  const float erp0 = P->erp;
  if (ncons == nk) {
    for (int x = t; x < nic; x += nt) erp_out[cord[x]] = erp0;
  } else {
    for (int k = t; k < nisl; k += nt) {
      float erp = erp0;
      for (int x = icons[k], e = x + icnt[k]; x < e; x++) {
        const int i = cord[x];
        if (i >= nk && joints[i - nk].type == JT_BALL) erp = joints[i - nk].erp;
        erp_out[i] = erp;
      }
    }
  }
  __syncthreads();
  if (t == 0) {
    P->seed = lcg_skip(seed, shuffles * draws);
    misc[0] = nrows;
    misc[1] = nisl;
    misc[2] = nic;
    misc[3] = nib;
  }
  __syncthreads();
}
