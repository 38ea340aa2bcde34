// gh_complex.inl -- Greiner-Hormann clipping of complex polygons (several
// rings per side: outer rings, holes, islands) and their union, on gfx950.
// Included at the end of gh.hip (same translation unit: it shares the node
// lists, the output buffers and the predicates).
//
// The reference clips complex polygons with its multi-polygon program
// (GH-CUDA/ghcuda-multiPolygon.cpp:259-330 with
// gppolyclip_mDIV512-multiPolygon.cu for phase 1) and the CPU labelling of
// GH-CUDA/lib/polyclip.h, whose loops run over every component of P and Q
// (vector<polygon>) and whose global UNION switch (polyclip.h:42) turns the
// intersection into the union.
//
// Here one wave takes one pair of complex polygons:
//   1. the lanes classify every source edge of every ring of P against every
//      source edge of every ring of Q (intersect(), polyclip.h:60-179), 64
//      Q edges at a time held one per lane and read by readlane, and write
//      the non-zero records, each P edge's in Q order, at scanned offsets;
//   2. a pair in general position whose arrays fit the launch's LDS
//      (complex_fast) is spliced, labelled, traced and cleaned up by the
//      whole wave in LDS;
//   3. every other pair is replayed by lane 0 in global memory: the records
//      in the reference's loop order (P ring, P edge, Q ring, Q edge;
//      polyclip.h:200-277), inserting vertices by alpha with the reference's
//      tie rule (polygon.h:101-113), then label_trace_multi over all
//      components and the clean-up (polyclip.h:791-807).
//
// What bounds it: dependent accesses, one pair at a time.  On one MI355X 300
// pairs of 120 vertices took 881 us in the clip launch when lane 0 replayed
// every pair from global memory and each lane read every Q edge by itself
// (another 144 us in the counting launch); see complex_fast for what it
// takes now.

constexpr int kComplexW = 64;

// ---------------------------------------------------- multi-ring labelling
__device__ bool node_pip_comps(const Nodes &N, const int *roots, int n, pt R) {
  bool in = false;  // even-odd over the components (polyclip.h:505-507)
  for (int c = 0; c < n; c++)
    if (node_pip(N, roots[c], R)) in = !in;
  return in;
}

__device__ bool node_on_ring(const Nodes &N, int root, int V) {
  int W = root;
  do {
    if (W == V) return true;
    W = N.next[W];
  } while (W != root);
  return false;
}

// polygon::noCrossingVertex(union_case), polygon.h:465-475
__device__ bool node_no_crossing(const Nodes &N, int root, bool U) {
  int V = root;
  do {
    if (isint(N, V)) {
      const int l = N.lab[V];
      if (l == L_CROSSING || l == L_DELAYED_CROSSING) return false;
      if (U && (l == L_BOUNCING || l == L_DELAYED_BOUNCING)) return false;
    }
    V = N.next[V];
  } while (V != root);
  return true;
}

__device__ bool node_all_on_on(const Nodes &N, int root) {
  int V = root;
  do {
    if (N.lab[V] != L_ON_ON) return false;
    V = N.next[V];
  } while (V != root);
  return true;
}

// polygon::getNonIntersectionPoint, polygon.h:480-491
__device__ bool node_nonint_point(const Nodes &N, int root, pt &p) {
  int V = root;
  do {
    if (!isint(N, V)) {
      p = P_(N, V);
      return true;
    }
    V = N.next[V];
  } while (V != root);
  V = root;
  do {
    const int n = N.next[V], nb = N.nb[V], nnb = N.nb[n];
    if (nb >= 0 && nnb != N.prev[nb] && nnb != N.next[nb]) {
      const pt a = P_(N, V), b = P_(N, n);
      p = pt{0.5 * (a.x + b.x), 0.5 * (a.y + b.y)};
      return true;
    }
    V = n;
  } while (V != root);
  return false;
}

// polygon::getNonIntersectionVertex, polygon.h:496-512 (a midpoint vertex
// is inserted when every vertex is an intersection); -1 none, -2 overflow
__device__ int node_nonint_vertex(Nodes &N, int root) {
  int V = root;
  do {
    if (!isint(N, V)) return V;
    V = N.next[V];
  } while (V != root);
  V = root;
  do {
    const int n = N.next[V], nb = N.nb[V], nnb = N.nb[n];
    if (nb >= 0 && nnb != N.prev[nb] && nnb != N.next[nb]) {
      const pt a = P_(N, V), b = P_(N, n), ao = ld(N.po, V), bo = ld(N.po, n);
      const int T = node_new(N, pt{0.5 * (a.x + b.x), 0.5 * (a.y + b.y)},
                             pt{0.5 * (ao.x + bo.x), 0.5 * (ao.y + bo.y)});
      if (T < 0) return -2;
      node_insert_after(N, T, V);
      return T;
    }
    V = n;
  } while (V != root);
  return -1;
}

// labelIntersections (polyclip.h:335-735, steps 1 and 3 restored),
// createResult (:743-783) over every component of P and Q, for the
// intersection or (U) the union.  roots[0] / roots[1] hold the rings' start
// nodes; the result components go to O in the reference's order.
__device__ int label_trace_multi(Nodes &N, const int *const *roots, const int *nr, OutBuf &O,
                                 bool U) {
  // step 1 (restored, :343-397) and step 3 (:461-465) over P's components
  for (int c = 0; c < nr[0]; c++) {
    const int r = roots[0][c];
    int I = r;
    do {
      if (isint(N, I) && N.nb[I] >= 0) {
        const int Pm = N.prev[I], Pp = N.next[I], Qm = N.prev[N.nb[I]], Qp = N.next[N.nb[I]];
        const int tm = node_rel(N, Qm, Pm, I, Pp), tp = node_rel(N, Qp, Pm, I, Pp);
        int l = N.lab[I];
        if ((tm == 0 && tp == 1) || (tm == 1 && tp == 0)) l = L_CROSSING;
        if ((tm == 0 && tp == 0) || (tm == 1 && tp == 1)) l = L_BOUNCING;
        if ((tp == 3 && tm == 1) || (tm == 3 && tp == 1)) l = L_LEFT_ON;
        if ((tp == 3 && tm == 0) || (tm == 3 && tp == 0)) l = L_RIGHT_ON;
        if ((tp == 3 && tm == 2) || (tm == 3 && tp == 2)) l = L_ON_ON;
        if ((tm == 2 && tp == 1) || (tp == 2 && tm == 1)) l = L_ON_LEFT;
        if ((tm == 2 && tp == 0) || (tp == 2 && tm == 0)) l = L_ON_RIGHT;
        N.lab[I] = (signed char)l;
      }
      I = N.next[I];
    } while (I != r);
  }
  for (int c = 0; c < nr[0]; c++) {
    const int r = roots[0][c];
    int I = r;
    do {
      if (isint(N, I) && N.nb[I] >= 0) N.lab[N.nb[I]] = N.lab[I];
      I = N.next[I];
    } while (I != r);
  }
  // step 2: intersection chains (:398-451)
  for (int c = 0; c < nr[0]; c++) {
    const int r = roots[0][c];
    int it = r;
    do {
      if (isint(N, it) && (N.lab[it] == L_LEFT_ON || N.lab[it] == L_RIGHT_ON)) {
        int I = it;
        const int x = N.lab[I] == L_LEFT_ON ? 0 : 1;
        const int X = I;
        do {
          N.lab[I] = L_NONE;
          if (N.nb[I] >= 0) N.lab[N.nb[I]] = L_NONE;
          I = N.next[I];
        } while (N.lab[I] == L_ON_ON);
        const int y = N.lab[I] == L_ON_LEFT ? 0 : 1;
        const signed char ct = (x != y) ? L_DELAYED_CROSSING : L_DELAYED_BOUNCING;
        N.lab[X] = ct;
        N.lab[I] = ct;
        if (N.nb[X] >= 0) N.lab[N.nb[X]] = ct;
        if (N.nb[I] >= 0) N.lab[N.nb[I]] = ct;
      }
      it = N.next[it];
    } while (it != r);
  }
  // step 3.5: components without crossings (:474-543); the per-component
  // flags are kept in the split bit of the root node (free until step 4)
  // as: bit F_SPLIT set = no intersection, bit F_CROSS set = identical
  for (int i = 0; i < 2; i++) {
    for (int c = 0; c < nr[i]; c++) {
      const int Pr = roots[i][c];
      if (!node_no_crossing(N, Pr, U)) continue;
      N.fl[Pr] |= F_SPLIT;
      if (node_all_on_on(N, Pr)) {
        N.fl[Pr] |= F_CROSS;
        continue;
      }
      pt p;
      if (!node_nonint_point(N, Pr, p)) return GH_TRACE_FAIL;
      if (node_pip_comps(N, roots[1 - i], nr[1 - i], p) != U)
        if (!out_copy_ring(O, N, Pr)) return GH_OVERFLOW;
    }
  }
  // components of P identical to one of Q: added when both or neither are
  // holes (:517-541)
  for (int c = 0; c < nr[0]; c++) {
    const int Pr = roots[0][c];
    if (!(N.fl[Pr] & F_SPLIT) || !(N.fl[Pr] & F_CROSS)) continue;
    bool pHole = false;
    for (int c2 = 0; c2 < nr[0]; c2++)
      if (roots[0][c2] != Pr && node_pip(N, roots[0][c2], P_(N, Pr))) pHole = !pHole;
    for (int q = 0; q < nr[1]; q++) {
      const int Qr = roots[1][q];
      if (!(N.fl[Qr] & F_SPLIT) || !(N.fl[Qr] & F_CROSS) || !node_on_ring(N, Qr, N.nb[Pr]))
        continue;
      bool qHole = false;
      for (int q2 = 0; q2 < nr[1]; q2++)
        if (roots[1][q2] != Qr && node_pip(N, roots[1][q2], P_(N, Qr))) qHole = !qHole;
      if (pHole == qHole && !out_copy_ring(O, N, Pr)) return GH_OVERFLOW;
      break;
    }
  }
  // the component flags back to per-node split / crossing candidates
  bool skip[2][64];  // components without intersections (at most 64 per side here)
  for (int i = 0; i < 2; i++)
    for (int c = 0; c < nr[i]; c++) {
      const int Pr = roots[i][c];
      skip[i][c] = (N.fl[Pr] & F_SPLIT) != 0;
      N.fl[Pr] &= (unsigned char)~(F_SPLIT | F_CROSS);
    }
  // step 4: entry/exit flags (:549-655)
  for (int i = 0; i < 2; i++) {
    for (int c = 0; c < nr[i]; c++) {
      if (skip[i][c]) continue;
      const int Pr = roots[i][c];
      const int V = node_nonint_vertex(N, Pr);
      if (V == -2) return GH_OVERFLOW;
      if (V < 0) return GH_TRACE_FAIL;
      int status = ENTRY;
      if (node_pip_comps(N, roots[1 - i], nr[1 - i], P_(N, V))) toggle(status);
      bool first = true;
      int I = V;
      do {
        I = N.next[I];
      } while (!isint(N, I) && I != V);
      while (I != V) {
        if (N.lab[I] == L_CROSSING) {
          N.enex[I] = (signed char)status;
          toggle(status);
        }
        if (N.lab[I] == L_BOUNCING && ((status == EXIT) != U)) N.fl[I] |= F_SPLIT;
        if (N.lab[I] == L_DELAYED_CROSSING) {
          N.enex[I] = (signed char)status;
          if (first) {
            if ((status == EXIT) != U) N.lab[I] = L_CROSSING;
            first = false;
          } else {
            if ((status == ENTRY) != U) N.lab[I] = L_CROSSING;
            first = true;
            toggle(status);
          }
        }
        if (N.lab[I] == L_DELAYED_BOUNCING) {
          N.enex[I] = (signed char)status;
          if (first) {
            if ((status == EXIT) != U) N.fl[I] |= F_CROSS;
            first = false;
          } else {
            if ((status == ENTRY) != U) N.fl[I] |= F_CROSS;
            first = true;
          }
          toggle(status);
        }
        do {
          I = N.next[I];
        } while (!isint(N, I) && I != V);
      }
    }
  }
  // step 5: split bouncing vertex pairs (:661-714), P's candidates in the
  // order in which step 4 met them (a vertex of Q that several vertices of P
  // link to is split more than once, and the order decides the links); step 6
  // (:722-734)
  for (int c = 0; c < nr[0]; c++) {
    if (skip[0][c]) continue;
    const int r = node_nonint_vertex(N, roots[0][c]);  // step 4's start
    int I = r;
    do {
      const int nextI = N.next[I];
      if ((N.fl[I] & F_SPLIT) && N.nb[I] >= 0 && (N.fl[N.nb[I]] & F_SPLIT)) {
        const int IQ = N.nb[I];
        const int VP = node_new(N, P_(N, I), ld(N.po, I));
        const int VQ = node_new(N, P_(N, IQ), ld(N.po, IQ));
        if (VP < 0 || VQ < 0) return GH_OVERFLOW;
        const double sP = triA(P_(N, N.prev[I]), P_(N, I), P_(N, N.next[I]));
        const double sQ = triA(P_(N, N.prev[IQ]), P_(N, IQ), P_(N, N.next[IQ]));
        if (sP * sQ > 0) {
          node_link(N, I, VQ);
          node_link(N, IQ, VP);
        } else {
          node_link(N, VP, VQ);
        }
        node_insert_after(N, VP, I);
        node_insert_after(N, VQ, IQ);
        const signed char ex = U ? ENTRY : EXIT, en = U ? EXIT : ENTRY;
        N.enex[I] = ex;
        N.enex[VP] = en;
        N.enex[IQ] = ex;
        N.enex[VQ] = en;
        N.lab[I] = N.lab[VP] = N.lab[IQ] = N.lab[VQ] = L_CROSSING;
        N.fl[I] &= (unsigned char)~F_SPLIT;
      }
      I = nextI;
    } while (I != r);
  }
  for (int c = 0; c < nr[0]; c++) {
    const int r = roots[0][c];
    int I = r;
    do {
      if ((N.fl[I] & F_CROSS) && N.nb[I] >= 0 && (N.fl[N.nb[I]] & F_CROSS)) {
        N.lab[I] = L_CROSSING;
        N.lab[N.nb[I]] = L_CROSSING;
      }
      I = N.next[I];
    } while (I != r);
  }
  // createResult (:743-783) over P's components
  const long long guard = 4LL * N.n + 64;
  for (int c = 0; c < nr[0]; c++) {
    const int r = roots[0][c];
#define IS_CI(v) (isint(N, (v)) && N.lab[(v)] == L_CROSSING)
    int I = r;
    bool have = IS_CI(I);
    if (!have) {
      do {
        I = N.next[I];
      } while (!IS_CI(I) && I != r);
      have = I != r;
    }
    while (have) {
      if (O.ncomp >= O.capComp) return GH_OVERFLOW;
      int R = -1, V = I;
      N.fl[V] &= (unsigned char)~F_INT;
      long long steps = 0;
      do {
        int status = N.enex[V];
        toggle(status);
        do {
          V = ((status == EXIT) != U) ? N.next[V] : N.prev[V];
          N.fl[V] &= (unsigned char)~F_INT;
          const int w = out_new(O, P_(N, V), ld(N.po, V));
          if (w < 0) return GH_OVERFLOW;
          if (R < 0) R = w;
          else out_append(O, R, w);
          if (++steps > guard) return GH_TRACE_FAIL;
        } while (!(N.enex[V] == status) && V != I);
        if (V != I) {
          V = N.nb[V];
          if (V < 0) return GH_TRACE_FAIL;
          N.fl[V] &= (unsigned char)~F_INT;
        }
      } while (V != I);
      O.compRoot[O.ncomp++] = R;
      do {
        I = N.next[I];
      } while (!IS_CI(I) && I != r);
      have = I != r;
    }
#undef IS_CI
  }
  return GH_OK;
}

// ------------------------------------------------------------- kernels ----
// The pair's parts: base rings [b0, b0 + bn), overlay rings [o0, o0 + on).
struct ComplexPair {
  int b0, bn, o0, on;
};

__device__ __forceinline__ ComplexPair complex_pair(const int *parts, long k) {
  return ComplexPair{parts[4 * k], parts[4 * k + 1], parts[4 * k + 2], parts[4 * k + 3]};
}

// ring r of a side: its first vertex in the layer and its length without the
// closing vertex
__device__ __forceinline__ void ring_of(const int *vnum, const long *vpsnum, int r, long &s,
                                        int &n) {
  n = vnum[r] - 1;
  s = vpsnum[r] - vnum[r];
}

// The pair's predicate frame (ComplexArgs::norm): the MBRs over every ring,
// the CMBR, then as the single-ring clip (k_pair_setup) with the vertex
// totals; a union of polygons with disjoint MBRs uses their joint MBR.
// Status GH_DISJOINT for an intersection of disjoint MBRs (or an empty side).
struct ComplexArgs {
  const int *parts;
  long B, O;  // rings in the base and overlay layers
  const double *bCoords, *oCoords;
  const int *bVNum, *oVNum;
  const long *bVPSNum, *oVPSNum;
  int normalize, unionOp;
  int *status;
  double *norm;          // [3M]
  long long *nodeOff;    // [M+1] node / output capacity prefix
  long long *compOff;    // [M+1] component capacity prefix
  long long *recOff;     // [M+1] record capacity prefix
  long long *ringOff;    // [M+1] ring-root prefix
  long long *edgeOff;    // [M+1] P edge prefix (record offsets per P edge)
  unsigned long long *bad;  // pairs whose parts lie outside the layers
};

// The rings of both sides of a pair (at most 64 each), by a block's first
// wave: off[s][r]
// the first vertex of ring r counted over side s's rings, src[s][r] its first
// vertex in the layer.
struct ComplexRings {
  int off[2][65];
  long src[2][64];
};

__device__ __forceinline__ void complex_rings(const ComplexArgs &a, const ComplexPair &cp,
                                              ComplexRings &R) {
  const int lane = threadIdx.x;
  for (int side = 0; side < 2 && lane < kComplexW; side++) {
    const int r0 = side ? cp.o0 : cp.b0, rn = side ? cp.on : cp.bn;
    long s = 0;
    int n = 0;
    if (lane < rn)
      ring_of(side ? a.oVNum : a.bVNum, side ? a.oVPSNum : a.bVPSNum, r0 + lane, s, n);
    int tot;
    const int pre = grp_scan<kComplexW>(n, tot);
    if (lane < rn) {
      R.off[side][lane] = pre;
      R.src[side][lane] = s;
    }
    if (lane == 0) R.off[side][rn] = tot;
  }
  __syncthreads();
}

// ring of vertex v of a side with rn rings
__device__ __forceinline__ int ring_at(const int *off, int rn, int v) {
  int r = 0;
  while (r + 1 < rn && v >= off[r + 1]) r++;
  return r;
}

struct ComplexSide {
  const double *C;
  const int *off;
  const long *src;
  int rn;
  // original coordinates of vertex v, which lies in ring r
  __device__ __forceinline__ pt orig(int v, int r) const {
    return ld(C, src[r] + (v - off[r]));
  }
  // the vertex after v on its ring r
  __device__ __forceinline__ int next(int v, int r) const {
    return v + 1 == off[r + 1] ? off[r] : v + 1;
  }
};

__device__ __forceinline__ ComplexSide complex_side(const ComplexArgs &a, const ComplexPair &cp,
                                                    const ComplexRings &R, int side) {
  return ComplexSide{side ? a.oCoords : a.bCoords, R.off[side], R.src[side],
                     side ? cp.on : cp.bn};
}

// edge v of a side in the frame nrm
__device__ __forceinline__ void complex_edge(const ComplexSide &S, int v, const double nrm[3],
                                             pt &A, pt &B) {
  const int r = ring_at(S.off, S.rn, v);
  const pt a = S.orig(v, r), b = S.orig(S.next(v, r), r);
  A = pt{(a.x - nrm[0]) * nrm[2], (a.y - nrm[1]) * nrm[2]};
  B = pt{(b.x - nrm[0]) * nrm[2], (b.y - nrm[1]) * nrm[2]};
}

// Every P edge against every Q edge, by a block of nw waves: f(p, q, type,
// alpha, beta) for the non-zero types.  Wave w takes the w-th of every nw
// chunks of kCxChunk Q edges, held one per lane and read by readlane, four at
// a time for independent chains; a lane holds one P edge.  With nw = 1 each
// P edge's calls come in Q order, from lane p % 64.
constexpr int kCxChunk = 16;
template <class F>
__device__ __forceinline__ void complex_records(const ComplexSide &P, const ComplexSide &Q,
                                                const double nrm[3], int nw, F &&f) {
  const int lane = __lane_id(), nP = P.off[P.rn], nQ = Q.off[Q.rn];
  const int w = threadIdx.x >> 6;
  for (int p0 = 0; p0 < nP; p0 += 64) {
    const int p = p0 + lane;
    pt P1{0.0, 0.0}, P2{0.0, 0.0};
    if (p < nP) complex_edge(P, p, nrm, P1, P2);
    for (int q0 = w * kCxChunk; q0 < nQ; q0 += nw * kCxChunk) {
      pt A{0.0, 0.0}, B{0.0, 0.0};
      if (lane < kCxChunk && q0 + lane < nQ) complex_edge(Q, q0 + lane, nrm, A, B);
      const int m = min(kCxChunk, nQ - q0);
      for (int l = 0; l < m; l += 4) {
        bool apart[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const pt Q1{lane_d(A.x, l + u), lane_d(A.y, l + u)};
          const pt Q2{lane_d(B.x, l + u), lane_d(B.y, l + u)};
          apart[u] = p >= nP || l + u >= m || edges_apart(P1, P2, Q1, Q2);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (!__ballot(!apart[u])) continue;
          const pt Q1{lane_d(A.x, l + u), lane_d(A.y, l + u)};
          const pt Q2{lane_d(B.x, l + u), lane_d(B.y, l + u)};
          if (apart[u]) continue;
          double al, be;
          const int t = itype(P1, P2, Q1, Q2, al, be);
          if (t != 0) f(p, q0 + l + u, t, al, be);
        }
      }
    }
  }
}

// the most LDS a pair's arrays may take (a block's default limit): pairs of
// up to about 1500 vertices
constexpr long kComplexLds = 65536 - 4096;

// bytes of LDS complex_fast needs for a pair of n vertices in nr rings with
// R intersection records (LDS arrays each rounded up to 16 bytes)
__host__ __device__ constexpr long complex_fast_bytes(long n, long nr, long R) {
  return 36 * n + 160 * R + 48 * nr + 32 * 16;
}

// One block per pair: the frame, then the number of intersection records and
// with it the pair's capacities; the edges (p, q) of the first kCxHits
// records, in any order, at hits, so that the clip classifies only those
// again.  need[0]: the largest complex_fast_bytes of the launch's pairs that
// are at most ldsMax.  Four waves share a pair's edge pairs, since a call's
// few hundred pairs leave most SIMDs empty otherwise.
constexpr int kCxSetup = 256;
constexpr int kCxHits = 64;
__global__ void __launch_bounds__(kCxSetup)
    k_complex_setup(long M, ComplexArgs a, int *nodeCap, int *compCap, int *rings,
                    int *edgesP, int *recCnt, int *swapped, unsigned long long *need,
                    long ldsMax, int2 *hits) {
  const long k = blockIdx.x;
  if (k >= M) return;
  const int lane = threadIdx.x;
  const ComplexPair cp = complex_pair(a.parts, k);
  // parts outside the layers: counted and nothing read (the call fails)
  if (cp.b0 < 0 || cp.bn < 0 || cp.o0 < 0 || cp.on < 0 || (long)cp.b0 + cp.bn > a.B ||
      (long)cp.o0 + cp.on > a.O) {
    if (lane == 0) {
      a.status[k] = GH_DISJOINT;
      atomicAdd(a.bad, 1ULL);
      rings[k] = edgesP[k] = nodeCap[k] = compCap[k] = recCnt[k] = swapped[k] = 0;
    }
    return;
  }
  __shared__ ComplexRings R;
  __shared__ int nHits;
  if (lane == 0) nHits = 0;
  const bool few = cp.bn <= 64 && cp.on <= 64;
  if (few) complex_rings(a, cp, R);
  double m[2][4];
  long long nv[2] = {0, 0};
  bool emptyRing = false;
  for (int side = 0; side < 2 && few; side++) {
    const ComplexSide S = complex_side(a, cp, R, side);
    nv[side] = S.off[S.rn];
    for (int r = 0; r < S.rn; r++) emptyRing |= S.off[r + 1] - S.off[r] < 1;
    double x0 = INFINITY, y0 = INFINITY, x1 = -INFINITY, y1 = -INFINITY;
    for (int v = lane; v < S.off[S.rn]; v += kCxSetup) {
      const pt c = S.orig(v, ring_at(S.off, S.rn, v));
      x0 = fmin(x0, c.x);
      y0 = fmin(y0, c.y);
      x1 = fmax(x1, c.x);
      y1 = fmax(y1, c.y);
    }
    pgrp_minmax<kCxSetup>(x0, x1);
    pgrp_minmax<kCxSetup>(y0, y1);
    m[side][0] = x0;
    m[side][1] = y0;
    m[side][2] = x1;
    m[side][3] = y1;
  }
  int st = GH_OK;
  const bool apart = few && (m[0][0] > m[1][2] || m[0][2] < m[1][0] || m[0][1] > m[1][3] ||
                     m[0][3] < m[1][1]);
  if (!few || nv[0] < 1 || nv[1] < 1 || emptyRing) st = GH_DISJOINT;
  if (apart && !a.unionOp) st = GH_DISJOINT;
  double nrm[3] = {0.0, 0.0, 1.0};
  if (st == GH_OK && (a.normalize & 1)) {
    double b[4];
    if (apart) {  // the joint MBR (a union only)
      b[0] = fmin(m[0][0], m[1][0]);
      b[1] = fmin(m[0][1], m[1][1]);
      b[2] = fmax(m[0][2], m[1][2]);
      b[3] = fmax(m[0][3], m[1][3]);
    } else {  // the CMBR, as getCMBR (ghcuda.cpp:94-125)
      b[0] = m[0][0] < m[1][0] ? m[1][0] : m[0][0];
      b[1] = m[0][1] < m[1][1] ? m[1][1] : m[0][1];
      b[2] = m[1][2] < m[0][2] ? m[1][2] : m[0][2];
      b[3] = m[1][3] < m[0][3] ? m[1][3] : m[0][3];
    }
    const double w = b[2] - b[0], h = b[3] - b[1], e = w > h ? w : h;
    nrm[0] = b[0];
    nrm[1] = b[1];
    nrm[2] = e > 0.0 ? 1.0 / e : 1.0;
    if (a.normalize & 4) {
      const double rr = sqrt((double)nv[0] * (double)nv[1]) / 1024.0;
      double f = 1.0;
      while (f < rr) f *= 2.0;
      nrm[2] *= f;
    }
  }
  if (lane == 0) {
    a.status[k] = st;
    a.norm[3 * k] = nrm[0];
    a.norm[3 * k + 1] = nrm[1];
    a.norm[3 * k + 2] = nrm[2];
    swapped[k] = 0;
  }
  int cnt = 0;
  if (st == GH_OK) {
    complex_records(complex_side(a, cp, R, 0), complex_side(a, cp, R, 1), nrm, kCxSetup / 64,
                    [&](int p, int q, int, double, double) {
                      const int i = atomicAdd(&nHits, 1);
                      if (i < kCxHits) hits[k * kCxHits + i] = make_int2(p, q);
                    });
    __syncthreads();
    cnt = nHits;
  }
  if (lane != 0) return;
  const int nr = cp.bn + cp.on;
  recCnt[k] = cnt;
  rings[k] = st == GH_OK ? nr : 0;
  edgesP[k] = st == GH_OK ? (int)nv[0] : 0;
  // two nodes per record, two more per split pair, and the result
  nodeCap[k] = st == GH_OK ? (int)(nv[0] + nv[1]) + 4 * nr + 16 + 4 * cnt : 0;
  compCap[k] = st == GH_OK ? nr + 8 + cnt : 0;
  const long b = complex_fast_bytes(nv[0] + nv[1], nr, cnt);
  if (st == GH_OK && b <= ldsMax) atomicMax(need, (unsigned long long)b);
}

struct ComplexWork {
  double *npn, *npo, *nalpha;
  int *nnext, *nprev, *nnb;
  unsigned char *nfl;
  signed char *nlab, *nenex;
  double *opn, *opo;
  int *onext, *oprev, *ocompRoot;
  int *roots;             // [ring total] ring start nodes
  int *recP, *recQ, *recT;  // [records] P edge, Q edge and type
  double *recA, *recB;    // [records] alpha, beta
  int *edgeRec;           // [P edges + M] per-P-edge record offsets within the pair
  int *outNComp, *outNVerts, *compLen;
  double *xyTmp;
  int cleanup;
};

// The winding of the segment P0 -> P1 about R (polygon::pointInPoly,
// polygon.h:427-448)
__device__ __forceinline__ int seg_wind(pt P0, pt P1, pt R) {
  if ((P0.y < R.y) == (P1.y < R.y)) return 0;
  const int w = 2 * (P1.y > P0.y) - 1;
  if (P0.x >= R.x)
    return P1.x > R.x || (triA(P0, P1, R) > 0) == (P1.y > P0.y) ? w : 0;
  return P1.x > R.x && (triA(P0, P1, R) > 0) == (P1.y > P0.y) ? w : 0;
}

// Splicing, labelling, tracing and clean-up of one pair in general position,
// by one wave in LDS.  General position: every record is of type 1 (both
// edges crossed inside) and every crossing is labelled CROSSING, so that no
// source vertex carries a link, links are mutual, and steps 2, 5 and 6 of
// the labelling have nothing to do.  Then
//   - the list of a ring is its source vertices, each followed by its edge's
//     crossings by alpha (a later record before an earlier one on ties,
//     polygon.h:101-113), so a crossing's place in its side's list is (its
//     edge) + (its rank among the side's crossings) + 1, and rings own
//     contiguous ranges of the crossings;
//   - step 4 starts at the ring's first vertex and alternates, so a
//     crossing's enex is the start status and its rank's parity;
//   - createResult goes from crossing to crossing: lane 0 walks those (a few
//     per pair) and notes the segments, and all lanes write the vertices.
// Returns false, having written nothing but xy, when the pair is not in
// general position (lane 0's replay then takes it).
// All accesses but the layer's coordinates and the result are to LDS.
//
// Measured on one MI355X (set-up and count, then clip): 300 pairs of 120
// vertices 6 + 144 + 881 -> 34 + 57 us, the unions of 7 pairs 6 + 96 + 769 ->
// 31 + 53 us.  With one wave and no edges_apart the set-up took 78 us, and
// the clip, counting and classifying by itself, 197.
struct FastRecs {  // the pair's records, in LDS
  int *er, *rp, *rq;  // [nP + 1] offsets per P edge; P and Q edge per record
  double *al, *be;
};

__device__ bool complex_fast(const ComplexSide &P, const ComplexSide &Q, int nRec,
                             const FastRecs &rec, const double *pn,
                             Arena &ar, bool U, int cleanup, long long cap, long long capComp,
                             double *xy, int *clenOut, int *outComps, int *outVerts) {
  const int lane = threadIdx.x;
  const int nP = P.off[P.rn], nQ = Q.off[Q.rn], nS = nP + nQ;
  const int rn[2] = {P.rn, Q.rn}, nR = P.rn + Q.rn;
  // every take below fits: the caller checked complex_fast_bytes
  int *qo = ar.take<int>(nQ + 1, nullptr);
  int *ord[2] = {ar.take<int>(nRec, nullptr), ar.take<int>(nRec, nullptr)};
  int *inv[2] = {ar.take<int>(nRec, nullptr), ar.take<int>(nRec, nullptr)};
  // -- each edge's records by alpha (P) and beta (Q)
  for (int i = lane; i <= nQ; i += kComplexW) qo[i] = 0;
  __syncthreads();
  for (int r = lane; r < nRec; r += kComplexW) atomicAdd(&qo[rec.rq[r]], 1);
  __syncthreads();
  grp_scan_range<kComplexW, int>(nQ, [&](int q) { return qo[q]; },
                                 [&](int q, int pre, int) { qo[q] = pre; });
  __syncthreads();
  for (int r = lane; r < nRec; r += kComplexW) ord[1][atomicAdd(&qo[rec.rq[r]], 1)] = r;
  __syncthreads();
  // qo[q] is now the end of edge q's run
  for (int q = lane; q < nQ; q += kComplexW) {
    const int b = q ? qo[q - 1] : 0, z = qo[q];
    for (int i = b + 1; i < z; i++) {
      const int r = ord[1][i];
      const double v = rec.be[r];
      int j = i - 1;
      while (j >= b && (rec.be[ord[1][j]] > v || (rec.be[ord[1][j]] == v && ord[1][j] < r))) {
        ord[1][j + 1] = ord[1][j];
        j--;
      }
      ord[1][j + 1] = r;
    }
  }
  for (int p = lane; p < nP; p += kComplexW) {
    const int b = rec.er[p], z = rec.er[p + 1];
    for (int i = b; i < z; i++) {
      const double v = rec.al[i];
      int j = i - 1;
      while (j >= b && rec.al[ord[0][j]] >= v) {
        ord[0][j + 1] = ord[0][j];
        j--;
      }
      ord[0][j + 1] = i;
    }
  }
  __syncthreads();
  for (int j = lane; j < nRec; j += kComplexW) {
    inv[0][ord[0][j]] = j;
    inv[1][ord[1][j]] = j;
  }
  // first crossing of edge e of a side
  auto first = [&](int s, int e) { return s ? (e ? qo[e - 1] : 0) : rec.er[e]; };
  auto edge_of = [&](int s, int r) { return s ? rec.rq[r] : rec.rp[r]; };
  // a node: a source vertex of P or (from nP) of Q, or (from nS) a record's
  // crossing
  auto src = [&](int s, int v) { return (s ? nP : 0) + v; };
  // -- the lists, each ring's crossings and each crossing's ring
  int *lst[2] = {ar.take<int>(nP + nRec, nullptr), ar.take<int>(nQ + nRec, nullptr)};
  int *crng[2] = {ar.take<int>(nRec, nullptr), ar.take<int>(nRec, nullptr)};
  int *rc[2] = {ar.take<int>(P.rn + 1, nullptr), ar.take<int>(Q.rn + 1, nullptr)};
  int *in = ar.take<int>(nR, nullptr);
  int *vis = ar.take<int>(nRec, nullptr);
  __syncthreads();
  for (int s = 0; s < 2; s++) {
    const ComplexSide &S = s ? Q : P;
    const int n = s ? nQ : nP;
    for (int v = lane; v < n; v += kComplexW) {
      const int f = first(s, v);
      lst[s][v + f] = src(s, v);
    }
    for (int j = lane; j < nRec; j += kComplexW) {
      const int r = ord[s][j], e = edge_of(s, r);
      lst[s][e + 1 + j] = nS + r;
      crng[s][j] = ring_at(S.off, S.rn, e);
    }
    for (int r = lane; r <= rn[s]; r += kComplexW)
      rc[s][r] = S.off[r] < n ? first(s, S.off[r]) : nRec;
  }
  for (int j = lane; j < nRec; j += kComplexW) vis[j] = 0;
  __syncthreads();
  // -- labels (polyclip.h:343-397), every one CROSSING, and an even number
  // of crossings on every ring (else the statuses do not alternate round it)
  bool slow = false;
  for (int r = lane; r < nRec; r += kComplexW) {
    int nb[2][2];  // the nodes before and after the crossing on both lists
    for (int s = 0; s < 2; s++) {
      const ComplexSide &S = s ? Q : P;
      const int e = edge_of(s, r), j = inv[s][r], b = first(s, e);
      const int z = s ? qo[e] : rec.er[e + 1];
      nb[s][0] = j > b ? nS + ord[s][j - 1] : src(s, e);
      nb[s][1] = j + 1 < z ? nS + ord[s][j + 1] : src(s, S.next(e, crng[s][j]));
    }
    const pt Pm = ld(pn, nb[0][0]), I = ld(pn, nS + r), Pp = ld(pn, nb[0][1]);
    int t[2];
    for (int d = 0; d < 2; d++) {
      const int q = nb[1][d];  // linked to a P neighbour: the same crossing
      t[d] = rel_pos(q >= nS && q == nb[0][0], q >= nS && q == nb[0][1], ld(pn, q), Pm, I, Pp);
    }
    if (!((t[0] == 0 && t[1] == 1) || (t[0] == 1 && t[1] == 0))) slow = true;
  }
  for (int s = 0; s < 2; s++)
    for (int r = lane; r < rn[s]; r += kComplexW)
      if ((rc[s][r + 1] - rc[s][r]) & 1) slow = true;
  if (grp_any<kComplexW>(slow)) return false;
  // -- every ring's first vertex inside the other polygon (steps 3.5 and 4)
  for (int g = 0; g < nR; g++) {
    const int s = g >= P.rn ? 1 : 0, o = 1 - s;
    const ComplexSide &S = s ? Q : P, &O = o ? Q : P;
    const pt X = ld(pn, src(s, S.off[g - (s ? P.rn : 0)]));
    const int n = o ? nQ : nP;
    int w = 0;
    for (int v = lane; v < n; v += kComplexW) {
      const int ring = ring_at(O.off, O.rn, v);
      const int b = first(o, v), z = o ? qo[v] : rec.er[v + 1];
      pt A = ld(pn, src(o, v));
      for (int j = b; j < z; j++) {
        const pt B = ld(pn, nS + ord[o][j]);
        w += seg_wind(A, B, X);
        A = B;
      }
      w += seg_wind(A, ld(pn, src(o, O.next(v, ring))), X);
    }
    w = grp_sum<kComplexW>(w);
    if (lane == 0) in[g] = w & 1;
  }
  // -- createResult (polyclip.h:743-783): the segments, in order.  The
  // departures from the crossings form cycles, so there are at most two
  // segments per record, and one per ring without crossings.
  const int maxSeg = 2 * nRec + nR;
  int *so = ar.take<int>(maxSeg + 1, nullptr);  // first output position
  int *sp = ar.take<int>(maxSeg, nullptr);      // first list position
  int *sx = ar.take<int>(maxSeg, nullptr);      // component and direction
  int *sr = ar.take<int>(maxSeg, nullptr);      // side and ring
  const int maxComp = nRec + nR;
  int *compRoot = ar.take<int>(maxComp, nullptr), *clen = ar.take<int>(maxComp, nullptr);
  __shared__ int sh[3];
  __syncthreads();
  if (lane == 0) {
    int ns = 0, nc = 0, tot = 0;
    bool fits = true;
    auto ring_list = [&](int s, int r, int &b, int &len) {
      const ComplexSide &S = s ? Q : P;
      b = S.off[r] + rc[s][r];
      len = S.off[r + 1] + rc[s][r + 1] - b;
    };
    auto put = [&](int s, int r, bool fwd, int p, int len) {
      if (ns >= maxSeg) {
        fits = false;
        return;
      }
      so[ns] = tot;
      sp[ns] = p;
      sx[ns] = 2 * nc + (fwd ? 1 : 0);
      sr[ns] = 64 * s + r;
      ns++;
      tot += len;
    };
    for (int g = 0; g < nR; g++) {  // step 3.5: rings without crossings
      const int s = g >= P.rn ? 1 : 0, r = g - (s ? P.rn : 0);
      if (rc[s][r + 1] != rc[s][r] || (in[g] != 0) == U) continue;
      int b, len;
      ring_list(s, r, b, len);
      compRoot[nc] = tot;
      clen[nc] = len;
      put(s, r, true, b, len);
      nc++;
    }
    for (int c0 = 0; c0 < nRec && fits; c0++) {
      if (vis[ord[0][c0]]) continue;
      vis[ord[0][c0]] = 1;
      const int start = tot;
      int s = 0, j = c0;
      while (fits) {
        const int r = crng[s][j], lo = rc[s][r], hi = rc[s][r + 1];
        int b, len;
        ring_list(s, r, b, len);
        const int st0 = in[(s ? P.rn : 0) + r] ? EXIT : ENTRY;
        const int enex = ((j - lo) & 1) ? (st0 == ENTRY ? EXIT : ENTRY) : st0;
        const bool fwd = (enex == ENTRY) != U;
        const int j2 = fwd ? (j + 1 == hi ? lo : j + 1) : (j == lo ? hi - 1 : j - 1);
        const int p = edge_of(s, ord[s][j]) + 1 + j, r2 = ord[s][j2];
        const int p2 = edge_of(s, r2) + 1 + j2;
        int d = fwd ? p2 - p : p - p2;
        if (d <= 0) d += len;
        int q = fwd ? p + 1 : p - 1;
        if (q >= b + len) q -= len;
        if (q < b) q += len;
        put(s, r, fwd, q, d);
        vis[r2] = 1;
        if (s == 0 && j2 == c0) break;
        s = 1 - s;
        j = inv[s][r2];
        if (s == 0 && j == c0) break;
      }
      if (nc < maxComp) {
        compRoot[nc] = start;
        clen[nc] = tot - start;
      }
      nc++;
    }
    so[ns] = tot;
    if (tot > nS + 2 * nRec || tot > cap || nc > maxComp || nc > capComp) fits = false;
    sh[0] = ns;
    sh[1] = nc;
    sh[2] = fits ? tot : -1;
  }
  __syncthreads();
  const int ns = sh[0], nc = sh[1], tot = sh[2];
  if (tot < 0) return false;
  // -- the result vertices
  int *omap = ar.take<int>(nS + 2 * nRec, nullptr), *cw = ar.take<int>(nS + 2 * nRec, nullptr);
  for (int w = lane; w < tot; w += kComplexW) {
    int a = 0, z = ns;  // the segment with so[a] <= w < so[a + 1]
    while (z - a > 1) {
      const int m = (a + z) >> 1;
      if (so[m] <= w) a = m;
      else z = m;
    }
    const int s = sr[a] >> 6, r = sr[a] & 63;
    const ComplexSide &S = s ? Q : P;
    const int b = S.off[r] + rc[s][r], len = S.off[r + 1] + rc[s][r + 1] - b;
    int q = (sx[a] & 1) ? sp[a] + (w - so[a]) : sp[a] - (w - so[a]);
    if (q >= b + len) q -= len;
    if (q < b) q += len;
    const int v = lst[s][q];
    omap[w] = v;
    cw[w] = sx[a] >> 1;
    pt o;
    if (v < nS) {
      o = S.orig(v - (s ? nP : 0), r);
    } else {  // (1 - alpha) P1 + alpha P2 in the original coordinates
      const int e = rec.rp[v - nS], pr = ring_at(P.off, P.rn, e);
      const double al = rec.al[v - nS];
      const pt A = P.orig(e, pr), B = P.orig(P.next(e, pr), pr);
      o = pt{(1.0 - al) * A.x + al * B.x, (1.0 - al) * A.y + al * B.y};
    }
    st(xy, w, o);
  }
  __syncthreads();
  OutBuf O;
  O.n = tot;
  O.ncomp = nc;
  O.compRoot = compRoot;
  if (cleanup) {
    int *sc = ar.take<int>(3 * nc + tot, nullptr);
    grp_cleanup_compact<kComplexW>(O, xy, clen, cw, sc, pn, omap, 0);
    __syncthreads();
  }
  for (int c = lane; c < O.ncomp; c += kComplexW) clenOut[c] = clen[c];
  if (lane == 0) {
    *outComps = O.ncomp;
    *outVerts = O.n;
  }
  return true;
}

__global__ void __launch_bounds__(kComplexW)
    k_complex_clip(long M, ComplexArgs a, ComplexWork w, const int2 *hits, int ldsBytes) {
  const long k = blockIdx.x;
  if (k >= M) return;
  const int lane = threadIdx.x;
  if (a.status[k] != GH_OK) {
    if (lane == 0) {
      w.outNComp[k] = 0;
      w.outNVerts[k] = 0;
    }
    return;
  }
  const ComplexPair cp = complex_pair(a.parts, k);
  __shared__ ComplexRings R;
  complex_rings(a, cp, R);
  const ComplexSide P = complex_side(a, cp, R, 0), Q = complex_side(a, cp, R, 1);
  const int nP = P.off[P.rn], nQ = Q.off[Q.rn], base = nP + nQ, nSrcP = nP;
  const double nrm[3] = {a.norm[3 * k], a.norm[3 * k + 1], a.norm[3 * k + 2]};
  const long long rb = a.recOff[k], nRec = a.recOff[k + 1] - rb;
  // -- the records: in LDS when the pair fits there, else in the pair's
  // global region
  extern __shared__ __align__(16) char complex_lds[];
  const bool fits = complex_fast_bytes(base, cp.bn + cp.on, nRec) <= ldsBytes;
  Arena ar{fits ? complex_lds : nullptr, ldsBytes};
  int *er = ar.take<int>(nSrcP + 1, w.edgeRec + a.edgeOff[k] + k);
  int *recP = ar.take<int>(nRec, w.recP + rb), *recQ = ar.take<int>(nRec, w.recQ + rb);
  int *recT = ar.take<int>(nRec, w.recT + rb);
  double *recA = ar.take<double>(nRec, w.recA + rb), *recB = ar.take<double>(nRec, w.recB + rb);
  for (int e = lane; e <= nSrcP; e += kComplexW) er[e] = 0;
  __syncthreads();
  bool plain = true;  // every record of type 1
  auto scan_er = [&] {
    __syncthreads();
    const int tot = grp_scan_range<kComplexW, int>(
        nSrcP, [&](int e) { return er[e]; }, [&](int e, int pre, int) { er[e] = pre; });
    if (lane == 0) er[nSrcP] = tot;
    __syncthreads();
  };
  if (nRec <= kCxHits) {
    // the set-up's hits, one per lane, ranked by (P edge, Q edge)
    const int2 h = lane < nRec ? hits[k * kCxHits + lane] : make_int2(0x7fffffff, 0);
    int o = 0;
    for (int l = 0; l < (int)nRec; l++) {
      const int p = __builtin_amdgcn_readlane(h.x, l), q = __builtin_amdgcn_readlane(h.y, l);
      o += p < h.x || (p == h.x && q < h.y) ? 1 : 0;
    }
    if (lane < nRec) {
      pt P1, P2, Q1, Q2;
      complex_edge(P, h.x, nrm, P1, P2);
      complex_edge(Q, h.y, nrm, Q1, Q2);
      double al, be;
      const int t = itype(P1, P2, Q1, Q2, al, be);
      recP[o] = h.x;
      recQ[o] = h.y;
      recT[o] = t;
      recA[o] = al;
      recB[o] = be;
      plain = t == 1;
      atomicAdd(&er[h.x], 1);
    }
    scan_er();
  } else {
    complex_records(P, Q, nrm, 1, [&](int p, int, int, double, double) { er[p]++; });
    scan_er();
    int p0 = -1, o = 0;  // the lane's P edge and its next record
    complex_records(P, Q, nrm, 1, [&](int p, int q, int t, double al, double be) {
      if (p != p0) {
        p0 = p;
        o = er[p];
      }
      recP[o] = p;
      recQ[o] = q;
      recT[o] = t;
      recA[o] = al;
      recB[o] = be;
      o++;
      plain = plain && t == 1;
    });
    __syncthreads();
  }
  double *xy = w.xyTmp + 2 * a.nodeOff[k];
  int *clen = w.compLen + a.compOff[k];
  if (fits && !grp_any<kComplexW>(!plain)) {
    double *pn = ar.take<double>(2 * (base + nRec), nullptr);
    for (int v = lane; v < base; v += kComplexW) {
      const bool onQ = v >= nP;
      const ComplexSide &S = onQ ? Q : P;
      const int i = onQ ? v - nP : v;
      const pt o = S.orig(i, ring_at(S.off, S.rn, i));
      st(pn, v, pt{(o.x - nrm[0]) * nrm[2], (o.y - nrm[1]) * nrm[2]});
    }
    __syncthreads();
    for (int r = lane; r < nRec; r += kComplexW) {
      const int e = recP[r];
      const pt P1 = ld(pn, e), P2 = ld(pn, P.next(e, ring_at(P.off, P.rn, e)));
      const double al = recA[r];
      st(pn, base + r, pt{(1.0 - al) * P1.x + al * P2.x, (1.0 - al) * P1.y + al * P2.y});
    }
    __syncthreads();
    if (complex_fast(P, Q, (int)nRec, FastRecs{er, recP, recQ, recA, recB}, pn, ar,
                     a.unionOp != 0, w.cleanup, a.nodeOff[k + 1] - a.nodeOff[k],
                     a.compOff[k + 1] - a.compOff[k], xy, clen, w.outNComp + k,
                     w.outNVerts + k))
      return;
    __syncthreads();
  }
  // -- lane 0's replay: the source nodes, ring by ring (P's rings, then Q's)
  const long long nb0 = a.nodeOff[k], cap = a.nodeOff[k + 1] - nb0;
  Nodes N;
  N.pn = w.npn + 2 * nb0;
  N.po = w.npo + 2 * nb0;
  N.next = w.nnext + nb0;
  N.prev = w.nprev + nb0;
  N.nb = w.nnb + nb0;
  N.fl = w.nfl + nb0;
  N.lab = w.nlab + nb0;
  N.enex = w.nenex + nb0;
  N.cap = (int)cap;
  double *alpha = w.nalpha + nb0;
  int *roots = w.roots + a.ringOff[k];
  for (int v = lane; v < base; v += kComplexW) {
    const bool onQ = v >= nP;
    const ComplexSide &S = onQ ? Q : P;
    const int sb = onQ ? nP : 0, i = v - sb, r = ring_at(S.off, S.rn, i);
    const pt o = S.orig(i, r);
    st(N.pn, v, pt{(o.x - nrm[0]) * nrm[2], (o.y - nrm[1]) * nrm[2]});
    st(N.po, v, o);
    N.next[v] = sb + S.next(i, r);
    N.prev[v] = sb + (i == S.off[r] ? S.off[r + 1] - 1 : i - 1);
    N.nb[v] = -1;
    N.fl[v] = F_SRC;
    N.lab[v] = L_NONE;
    N.enex[v] = NEITHER;
    alpha[v] = -2.0;
  }
  for (int r = lane; r < P.rn + Q.rn; r += kComplexW)
    roots[r] = r < P.rn ? P.off[r] : nP + Q.off[r - P.rn];
  N.n = base;
  __syncthreads();
  if (lane != 0) return;
  // -- the insertions in the reference's loop order (polyclip.h:200-277)
  auto insert = [&](int V, int curr, double al) {  // insertVertex, polygon.h:101-113
    do {
      curr = N.next[curr];
    } while (!(N.fl[curr] & F_SRC) && alpha[curr] < al);
    N.next[N.prev[curr]] = V;
    N.prev[V] = N.prev[curr];
    N.next[V] = curr;
    N.prev[curr] = V;
  };
  auto fresh = [&](pt p, pt o, double al) {
    const int v = node_new(N, p, o);
    if (v >= 0) alpha[v] = al;
    return v;
  };
  int rc = GH_OK;
  for (int e = 0; e < nSrcP && rc == GH_OK; e++) {
    const int one = e;  // P's source nodes are 0 .. nSrcP - 1 in edge order
    int two = N.next[one];
    while (!(N.fl[two] & F_SRC)) two = N.next[two];
    const pt P1 = P_(N, one), P2 = P_(N, two), P1o = ld(N.po, one), P2o = ld(N.po, two);
    for (int j = er[e]; j < er[e + 1]; j++) {
      const int q1 = nSrcP + recQ[j], t = recT[j];
      const double al = recA[j], be = recB[j];
      const pt Q1 = P_(N, q1), Q1o = ld(N.po, q1);
      int IP, IQ;
      switch (t) {
        case 1: {
          const pt I = {(1.0 - al) * P1.x + al * P2.x, (1.0 - al) * P1.y + al * P2.y};
          const pt Io = {(1.0 - al) * P1o.x + al * P2o.x, (1.0 - al) * P1o.y + al * P2o.y};
          IP = fresh(I, Io, al);
          IQ = fresh(I, Io, be);
          if (IP < 0 || IQ < 0) {
            rc = GH_OVERFLOW;
            break;
          }
          insert(IP, one, al);
          insert(IQ, q1, be);
          node_link(N, IP, IQ);
          break;
        }
        case 5:
          IQ = fresh(P1, P1o, be);
          if (IQ < 0) {
            rc = GH_OVERFLOW;
            break;
          }
          insert(IQ, q1, be);
          node_link(N, one, IQ);
          IP = fresh(Q1, Q1o, al);
          if (IP < 0) {
            rc = GH_OVERFLOW;
            break;
          }
          insert(IP, one, al);
          node_link(N, IP, q1);
          break;
        case 2:
        case 6:
          IQ = fresh(P1, P1o, be);
          if (IQ < 0) {
            rc = GH_OVERFLOW;
            break;
          }
          insert(IQ, q1, be);
          node_link(N, one, IQ);
          break;
        case 3:
        case 7:
          IP = fresh(Q1, Q1o, al);
          if (IP < 0) {
            rc = GH_OVERFLOW;
            break;
          }
          insert(IP, one, al);
          node_link(N, IP, q1);
          break;
        default:  // 4, 8
          node_link(N, one, q1);
          break;
      }
      if (rc != GH_OK) break;
    }
  }
  // -- labelling, tracing, clean-up
  OutBuf O;
  O.pn = w.opn + 2 * nb0;
  O.po = w.opo + 2 * nb0;
  O.next = w.onext + nb0;
  O.prev = w.oprev + nb0;
  O.n = 0;
  O.cap = (int)cap;
  O.compRoot = w.ocompRoot + a.compOff[k];
  O.ncomp = 0;
  O.capComp = (int)(a.compOff[k + 1] - a.compOff[k]);
  if (rc == GH_OK) {
    const int *rts[2] = {roots, roots + cp.bn};
    const int nrs[2] = {cp.bn, cp.on};
    rc = label_trace_multi(N, rts, nrs, O, a.unionOp != 0);
  }
  if (rc != GH_OK) {
    a.status[k] = rc;
    w.outNComp[k] = 0;
    w.outNVerts[k] = 0;
    return;
  }
  int nc = 0, nv = 0;
  for (int c = 0; c < O.ncomp; c++) {
    int r = O.compRoot[c];
    if (w.cleanup) r = out_cleanup(O, r);
    if (r < 0) continue;
    int len = 0, v = r;
    do {
      st(xy, nv + len, ld(O.po, v));
      len++;
      v = O.next[v];
    } while (v != r);
    clen[nc++] = len;
    nv += len;
  }
  w.outNComp[k] = nc;
  w.outNVerts[k] = nv;
}

// ----------------------------------------------------------------- host ----
void clip_complex(Context &c, const JoinInputs &in, const int *parts, long M,
                  const ClipOptions &opt, bool unionOp, ClipResult &res) {
  res = ClipResult();
  res.M = M;
  if (M <= 0) return;
  ComplexArgs a;
  a.parts = parts;
  a.bCoords = in.bCoords;
  a.oCoords = in.oCoords;
  a.bVNum = in.bVNum;
  a.oVNum = in.oVNum;
  a.bVPSNum = in.bVPSNum;
  a.oVPSNum = in.oVPSNum;
  a.normalize = opt.normalize;
  a.unionOp = unionOp ? 1 : 0;
  a.B = in.B;
  a.O = in.O;
  // [0] bad parts, [1] LDS the fast path needs, [2, 6) status counts
  unsigned long long *ctr = wsT<unsigned long long>(c, "cx_counters", 6);
  a.bad = ctr;
  fill_i32(c, (int *)ctr, 0, 12);
  a.status = wsT<int>(c, "cx_status", M);
  a.norm = wsT<double>(c, "cx_norm", 3 * M);
  int *nodeCap = wsT<int>(c, "cx_nodeCap", M), *compCap = wsT<int>(c, "cx_compCap", M);
  int *rings = wsT<int>(c, "cx_rings", M), *edgesP = wsT<int>(c, "cx_edgesP", M);
  int *recCnt = wsT<int>(c, "cx_recCnt", M);
  a.nodeOff = wsT<long long>(c, "cx_nodeOff", M + 1);
  a.compOff = wsT<long long>(c, "cx_compOff", M + 1);
  a.recOff = wsT<long long>(c, "cx_recOff", M + 1);
  a.ringOff = wsT<long long>(c, "cx_ringOff", M + 1);
  a.edgeOff = wsT<long long>(c, "cx_edgeOff", M + 1);
  res.swapped = wsT<int>(c, "cx_swapped", M);
  int2 *hits = wsT<int2>(c, "cx_hits", (long long)kCxHits * M);
  {
    LaunchTimer t(c, "gh_complex_count");
    hipLaunchKernelGGL(k_complex_setup, dim3((unsigned)M), dim3(kCxSetup), 0, c.stream, M, a,
                       nodeCap, compCap, rings, edgesP, recCnt, res.swapped, ctr + 1,
                       kComplexLds, hits);
    HIP_CHECK(hipGetLastError());
  }
  scan_i32_to_i64_multi(c, {{nodeCap, a.nodeOff, M},
                            {compCap, a.compOff, M},
                            {recCnt, a.recOff, M},
                            {rings, a.ringOff, M},
                            {edgesP, a.edgeOff, M}});
  long long tot[7];
  read_scalars(c, {a.nodeOff + M, a.compOff + M, a.recOff + M, a.ringOff + M, a.edgeOff + M,
                   (const long long *)a.bad, (const long long *)ctr + 1},
               tot);
  if (tot[5] != 0)
    throw Error{GCMF_ERR_ARG, "complex clip: a pair's rings lie outside its layer"};
  const long long nodes = tot[0], comps = tot[1], recs = tot[2], nrings = tot[3],
                  nedges = tot[4];
  if (nodes >= 0x7fffffffLL || recs >= 0x7fffffffLL)
    throw Error{GCMF_ERR_OVERFLOW, "complex clip batch exceeds 2^31 nodes or records"};
  ComplexWork w;
  w.npn = wsT<double>(c, "cx_npn", 2 * nodes);
  w.npo = wsT<double>(c, "cx_npo", 2 * nodes);
  w.nalpha = wsT<double>(c, "cx_nalpha", nodes);
  w.nnext = wsT<int>(c, "cx_nnext", nodes);
  w.nprev = wsT<int>(c, "cx_nprev", nodes);
  w.nnb = wsT<int>(c, "cx_nnb", nodes);
  w.nfl = wsT<unsigned char>(c, "cx_nfl", nodes);
  w.nlab = wsT<signed char>(c, "cx_nlab", nodes);
  w.nenex = wsT<signed char>(c, "cx_nenex", nodes);
  w.opn = wsT<double>(c, "cx_opn", 2 * nodes);
  w.opo = wsT<double>(c, "cx_opo", 2 * nodes);
  w.onext = wsT<int>(c, "cx_onext", nodes);
  w.oprev = wsT<int>(c, "cx_oprev", nodes);
  w.ocompRoot = wsT<int>(c, "cx_ocompRoot", comps);
  w.roots = wsT<int>(c, "cx_roots", nrings);
  w.recP = wsT<int>(c, "cx_recP", recs);
  w.recQ = wsT<int>(c, "cx_recQ", recs);
  w.recT = wsT<int>(c, "cx_recT", recs);
  w.recA = wsT<double>(c, "cx_recA", recs);
  w.recB = wsT<double>(c, "cx_recB", recs);
  w.edgeRec = wsT<int>(c, "cx_edgeRec", nedges + M);
  w.outNComp = wsT<int>(c, "cx_outNComp", M);
  w.outNVerts = wsT<int>(c, "cx_outNVerts", M);
  w.compLen = wsT<int>(c, "cx_compLen", comps);
  w.xyTmp = wsT<double>(c, "cx_xyTmp", 2 * nodes);
  w.cleanup = opt.cleanup;
  {
    LaunchTimer t(c, "gh_complex_clip");
    const int lds = (int)((tot[6] + 15) & ~15LL);
    hipLaunchKernelGGL(k_complex_clip, dim3((unsigned)M), dim3(kComplexW), (size_t)lds, c.stream,
                       M, a, w, (const int2 *)hits, lds);
    HIP_CHECK(hipGetLastError());
  }
  res.vertOff = wsT<long long>(c, "cx_vOff", M + 1);
  res.compOff = wsT<long long>(c, "cx_cOff", M + 1);
  scan_i32_to_i64_multi(c, {{w.outNVerts, res.vertOff, M}, {w.outNComp, res.compOff, M}});
  res.xy = wsT<double>(c, "cx_out_xy", 2 * nodes);
  res.compSizes = wsT<int>(c, "cx_out_comp", comps);
  hipLaunchKernelGGL(k_gather_out<64>, dim3(pgrp_grid(M, 64)), dim3(pgrp_block(64)), 0, c.stream,
                     M, 1, (const long long *)a.nodeOff, (const long long *)a.compOff,
                     (const long long *)res.vertOff, (const long long *)res.compOff, w.xyTmp,
                     w.compLen, res.xy, res.compSizes);
  HIP_CHECK(hipGetLastError());
  res.status = a.status;
  res.ncomp = w.outNComp;
  res.nverts = w.outNVerts;
  unsigned long long *sc = ctr + 2;
  hipLaunchKernelGGL(k_status_counts, dim3(std::min<unsigned>(kStatBlocks, grid_for(M, 256))),
                     dim3(256), 0, c.stream, M, (const int *)a.status, sc);
  HIP_CHECK(hipGetLastError());
  long long rb[6];
  const long long *sl = (const long long *)sc;
  read_scalars(c, {res.vertOff + M, res.compOff + M, sl, sl + 1, sl + 2, sl + 3}, rb);
  res.totalVerts = (long)rb[0];
  res.totalComps = (long)rb[1];
  res.nOk = rb[2];
  res.nInvalid = rb[3];
  res.nDisjoint = rb[4];
  res.nFailed = rb[5];
  res.totalIntersections = recs;
}
