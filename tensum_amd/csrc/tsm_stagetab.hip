// tsm_stagetab.hip -- the tables of the stage kernel (tsm_stage.hip), built on
// the device from a tiling and the mesh incidences.
//
// The stage kernel forms the gradients of a tile's owned vertices and of the
// first halo ring itself, so a tile's slots are its owned vertices, the first
// ring (the tiling's halo) and, for schemes with gradients, the second ring:
// the corners of the first ring's cells.  Around each of these "gradient
// slots" the kernel walks the neighbours in ring order, so every neighbour is
// read once and each pair of successive neighbours is a cell (a fan).  Every
// per-tile table has one stride for all tiles: a block finds its entries from
// its tile number alone, without first loading an offset.
//
// Fans depend on the cell order and orientation only, never on the tiles, so
// the sums taken along them are the same bit for bit whatever the tile size
// and whichever tile forms them.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <functional>
#include <string>
#include <type_traits>
#include <vector>

#include "tsm_device.h"

namespace tsm {
namespace {

constexpr unsigned FAN_START = 0x80000000u, FAN_CLOSED = 0x40000000u, FAN_V = 0x3fffffffu;

inline unsigned nblk(long long n) { return (unsigned)((std::max(n, 1LL) + 255) / 256); }

// The fan of a vertex with n cells: chains of neighbours such that each successive
// pair (b, d) is a cell (v, b, d) in counter-clockwise order; in a closed chain the
// last and the first are one too.  A closed ring starts at the vertex's first cell,
// an open one at the cell without a predecessor.  b(k), d(k): cell k's pair; used(k)
// and use(k): the cells taken so far, none at the start.  Returns the entry count, at
// most two a cell.
template <class B, class D, class Used, class Use>
__device__ __forceinline__ int fan_walk(int n, B&& b, D&& d, Used&& used, Use&& use, unsigned* out) {
  int m = 0, left = n;
  while (left > 0) {
    int cur = -1;
    for (int e = 0; e < n; ++e) {
      if (used(e)) continue;
      if (cur < 0) cur = e;
      const int be = b(e);
      bool pred = false;
      for (int f = 0; f < n && !pred; ++f) pred = !used(f) && f != e && d(f) == be;
      if (!pred) { cur = e; break; }
    }
    const int first = b(cur), m0 = m;
    unsigned head = (unsigned)first | FAN_START;
    ++m;
    while (cur >= 0) {
      use(cur);
      --left;
      const int from = d(cur);
      if (from == first) { head |= FAN_CLOSED; break; }  // back where the chain began
      out[m++] = (unsigned)from;
      cur = -1;
      for (int f = 0; f < n && cur < 0; ++f)
        if (!used(f) && b(f) == from) cur = f;
    }
    out[m0] = head;
  }
  return m;
}
// ... of every vertex, at twice the start of its cells.  Bound by the latency of its
// searches, so the pairs are held in LDS and the taken cells in a register; vertices of
// more cells than fit read the mesh again instead.
constexpr int FAN_LDS = 16;
__global__ __launch_bounds__(64) void k_fan(DevGeo G, unsigned char* used, int* cnt, unsigned* fan) {
  __shared__ int2 pair[FAN_LDS][64];
  const int v = blockIdx.x * 64 + threadIdx.x, lane = threadIdx.x;
  if (v >= G.nv) return;
  const int e0 = G.vc_ptr[v], n = G.vc_ptr[v + 1] - e0;
  auto ends = [&](int k) -> int2 {
    const int c = G.vc[e0 + k] & 0x7fffffff;
    const int a0 = G.cv[3 * (size_t)c], a1 = G.cv[3 * (size_t)c + 1], a2 = G.cv[3 * (size_t)c + 2];
    return a0 == v ? make_int2(a1, a2) : (a1 == v ? make_int2(a2, a0) : make_int2(a0, a1));
  };
  unsigned* out = fan + 2 * (size_t)e0;
  if (n <= FAN_LDS) {
#pragma unroll 4
    for (int k = 0; k < n; ++k) pair[k][lane] = ends(k);
    unsigned taken = 0;
    cnt[v] = fan_walk(n, [&](int k) { return pair[k][lane].x; }, [&](int k) { return pair[k][lane].y; },
                      [&](int k) { return (taken >> k & 1u) != 0; }, [&](int k) { taken |= 1u << k; }, out);
  } else {
    for (int k = 0; k < n; ++k) used[e0 + k] = 0;
    cnt[v] = fan_walk(n, [&](int k) { return ends(k).x; }, [&](int k) { return ends(k).y; },
                      [&](int k) { return used[e0 + k] != 0; }, [&](int k) { used[e0 + k] = 1; }, out);
  }
}

struct TabIn {
  DevGeo G;
  int nt, grad;
  const int *vbeg, *hbeg, *halo;   // the tiling: owned ranges, first ring
  const int *h2beg, *halo2;        // second ring (null while it is being found)
  const int *fan_n;                // entries of each vertex's fan
  const unsigned* fan;
  const int *btbeg, *bt;           // boundary terms (null while they are being found)
};

// gradient slots of all tiles as one range: those of tile t start at
// vbeg[t] + hbeg[t] (owned and first ring), or at vbeg[t] without gradients
__device__ __forceinline__ int gs_beg(const TabIn& T, int t) {
  return T.vbeg[t] + (T.grad ? T.hbeg[t] : 0);
}
__device__ __forceinline__ void gs_find(const TabIn& T, int q, int& t, int& k, int& v) {
  int lo = 0, hi = T.nt;
  while (hi - lo > 1) {
    const int m = (lo + hi) >> 1;
    if (gs_beg(T, m) <= q) lo = m; else hi = m;
  }
  t = lo;
  k = q - gs_beg(T, t);
  const int nown = T.vbeg[t + 1] - T.vbeg[t];
  v = k < nown ? T.vbeg[t] + k : T.halo[T.hbeg[t] + k - nown];
}
__device__ __forceinline__ int tile_of(const TabIn& T, int v) {
  int lo = 0, hi = T.nt;
  while (hi - lo > 1) {
    const int m = (lo + hi) >> 1;
    if (T.vbeg[m] <= v) lo = m; else hi = m;
  }
  return lo;
}
__device__ __forceinline__ int find32(const int* a, int lo, int hi, int k) {
  while (lo < hi) {
    const int m = (lo + hi) >> 1;
    if (a[m] < k) lo = m + 1; else hi = m;
  }
  return lo;
}
// slot of vertex u in tile t, -1 if it has none (yet)
__device__ __forceinline__ int slot_in(const TabIn& T, int t, int u) {
  const int b0 = T.vbeg[t], b1 = T.vbeg[t + 1];
  if (u >= b0 && u < b1) return u - b0;
  const int h0 = T.hbeg[t], h1 = T.hbeg[t + 1];
  int k = find32(T.halo, h0, h1, u);
  if (k < h1 && T.halo[k] == u) return (b1 - b0) + (k - h0);
  if (!T.h2beg) return -1;
  const int r0 = T.h2beg[t], r1 = T.h2beg[t + 1];
  k = find32(T.halo2, r0, r1, u);
  return (k < r1 && T.halo2[k] == u) ? (b1 - b0) + (h1 - h0) + (k - r0) : -1;
}

// The items of a gradient slot: for each member of the vertex's periodic set
// (the vertex alone without one), a centre entry where the centre is not the
// slot itself from the start, then the member's fan, then the boundary terms of
// all members' cells.  f(kind, id, closed): kind 0 neighbour (closed: first of a
// closed chain), 1 centre, 2 boundary term of bface id.
template <class F>
__device__ void walk_items(const TabIn& T, int v, F&& f) {
  const DevGeo& G = T.G;
  const int p = G.pset[v];
  const int m0 = p < 0 ? 0 : G.pptr[p], m1 = p < 0 ? 1 : G.pptr[p + 1];
  for (int i = m0; i < m1; ++i) {
    const int m = p < 0 ? v : G.pv[i];
    if (!(i == m0 && m == v)) f(1, m, false);
    const unsigned* fan = T.fan + 2 * (size_t)G.vc_ptr[m];
    const int n = T.fan_n[m];
    for (int e = 0; e < n; ++e) {
      const unsigned x = fan[e];
      if ((x & FAN_START) && e > 0) f(1, m, false);
      f(0, (int)(x & FAN_V), (x & FAN_CLOSED) != 0);
    }
  }
  for (int i = m0; i < m1; ++i) {
    const int m = p < 0 ? v : G.pv[i];
    for (int e = G.vc_ptr[m]; e < G.vc_ptr[m + 1]; ++e) {
      if (G.vc[e] >= 0) continue;  // no bface
      const int c = G.vc[e] & 0x7fffffff;
      for (int z = 0; z < 2; ++z) {
        const int b = G.cbf[2 * (size_t)c + z];
        if (b < 0) break;
        if (bc_sets_state(G.btype[b])) f(2, b, false);
      }
    }
  }
}

// Counts of a build, read back together: largest counts of a tile (k_desc, k_be_max),
// totals, cursors of k_gs_emit, and whether an entry did not fit its bits.
enum { N_MS, N_MS1, N_MF, N_MBT, N_MWT, N_MC, N_MB, N_BE, N_RING2, N_TERMS, N_OV, N_AT2, N_ATB, N_BAD, N_COUNTS };

// Sum over the threads of the block before this one; total: over all of them
__device__ __forceinline__ int block_before(int x, int& total) {
  __shared__ int part[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = x;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  __syncthreads();  // the sums before these have been read
  if (lane == 63) part[wave] = incl;
  __syncthreads();
  int before = incl - x;
  total = 0;
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += part[w];
    total += part[w];
  }
  return before;
}
// Over the gradient slots: second-ring candidates (corners of first-ring cells: an
// owned vertex's are all owned or in the first ring), boundary terms, and for each at
// least as many groups of items as follow its first
__global__ __launch_bounds__(256) void k_gs_count(TabIn T, int nq, int2* cnt, int* ng, int* n) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  int c2 = 0, cb = 0, nbr = 0, centres = 0;
  if (q < nq) {
    int t, k, v;
    gs_find(T, q, t, k, v);
    const bool ring = k >= T.vbeg[t + 1] - T.vbeg[t];
    walk_items(T, v, [&](int kind, int id, bool) {
      cb += kind == 2;
      nbr += kind == 0;
      centres += kind == 1;
      if (ring && kind != 2 && slot_in(T, t, id) < 0) ++c2;
    });
    cnt[q] = make_int2(c2, cb);
  }
  if (q <= nq) ng[q] = cb == 0 && centres == 0 && nbr <= 8 ? 0 : nbr / 7 + centres + (cb + 6) / 7;
  int s2, sb;
  block_before(c2, s2);
  block_before(cb, sb);
  if (threadIdx.x == 0) {
    if (s2) atomicAdd(n + N_RING2, s2);
    if (sb) atomicAdd(n + N_TERMS, sb);
  }
}
// their keys, the blocks' in any order (sorted next)
__global__ __launch_bounds__(256) void k_gs_emit(TabIn T, int nq, const int2* cnt, unsigned long long* k2,
                                                 unsigned long long* kb, int* n) {
  __shared__ int base[2];
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int2 c = q < nq ? cnt[q] : make_int2(0, 0);
  int s2, sb;
  int a2 = block_before(c.x, s2), ab = block_before(c.y, sb);
  if (threadIdx.x == 0) {
    base[0] = s2 ? atomicAdd(n + N_AT2, s2) : 0;
    base[1] = sb ? atomicAdd(n + N_ATB, sb) : 0;
  }
  __syncthreads();
  if (c.x + c.y == 0) return;
  a2 += base[0];
  ab += base[1];
  int t, k, v;
  gs_find(T, q, t, k, v);
  walk_items(T, v, [&](int kind, int id, bool) {
    const unsigned long long key = ((unsigned long long)(unsigned)t << 32) | (unsigned)id;
    if (kind == 2) kb[ab++] = key;
    else if (c.x && slot_in(T, t, id) < 0) k2[a2++] = key;
  });
}
__global__ void k_totals(const int* be, const int* ov, int* n) {
  n[N_BE] = *be;
  if (ov) n[N_OV] = *ov;
}
// first of the keys at or past each tile; entries to be left out are all ones and
// sort past them all
__global__ void k_seg(int n, const unsigned long long* keys, const int* nkeys, int* ptr) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  const unsigned long long k = (unsigned long long)(unsigned)i << 32;
  int lo = 0, hi = *nkeys;
  while (lo < hi) {
    const int m = (lo + hi) >> 1;
    if (keys[m] < k) lo = m + 1; else hi = m;
  }
  ptr[i] = lo;
}
__global__ void k_low(const int* n, const unsigned long long* keys, int* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < *n) out[i] = (int)(unsigned)(keys[i] & 0xffffffffull);
}
__global__ void k_zero_int(int n, int* p) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// descriptors and the largest counts
__global__ void k_desc(TabIn T, const int* fbeg, const int* wtbeg, const int* tcbeg,
                       const unsigned char* special, int4* desc, int* mx) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T.nt) return;
  const int nown = T.vbeg[t + 1] - T.vbeg[t], n1 = nown + T.hbeg[t + 1] - T.hbeg[t];
  const int ns = n1 + (T.h2beg ? T.h2beg[t + 1] - T.h2beg[t] : 0);
  const int nf = fbeg[t + 1] - fbeg[t];
  if (desc) desc[t] = make_int4(T.vbeg[t], nown, n1, nf | (special[t] ? 0x40000000 : 0));
  if (mx) {
    atomicMax(mx + N_MS, ns);
    atomicMax(mx + N_MS1, n1);
    atomicMax(mx + N_MF, nf);
    if (T.btbeg) atomicMax(mx + N_MBT, T.btbeg[t + 1] - T.btbeg[t]);
    if (wtbeg) atomicMax(mx + N_MWT, wtbeg[t + 1] - wtbeg[t]);
    if (tcbeg) atomicMax(mx + N_MC, tcbeg[t + 1] - tcbeg[t]);
  }
}
__global__ void k_fill_sid(TabIn T, int ms, int* sid) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)T.nt * ms) return;
  const int t = (int)(i / ms);
  int k = (int)(i % ms);
  const int nown = T.vbeg[t + 1] - T.vbeg[t], nh = T.hbeg[t + 1] - T.hbeg[t];
  const int n2 = T.h2beg ? T.h2beg[t + 1] - T.h2beg[t] : 0;
  int v = -1;
  if (k < nown) v = T.vbeg[t] + k;
  else if ((k -= nown) < nh) v = T.halo[T.hbeg[t] + k];
  else if ((k -= nh) < n2) v = T.halo2[T.h2beg[t] + k];
  sid[i] = v;
}
__global__ void k_fill_faces(int nt, int mf, const int* fbeg, const unsigned* f_lr,
                             const double* f_n, unsigned* lr, double2* n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)nt * mf) return;
  const int t = (int)(i / mf), j = (int)(i % mf);
  const bool in = j < fbeg[t + 1] - fbeg[t];
  const size_t o = (size_t)fbeg[t] + j;
  lr[i] = in ? f_lr[o] : 0u;
  n[i] = in ? make_double2(f_n[2 * o], f_n[2 * o + 1]) : make_double2(1.0, 0.0);
}
__global__ void k_xy(int nv, const double* x, const double* y, double2* xy) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nv) xy[i] = make_double2(x[i], y[i]);
}
__device__ __forceinline__ uint4 pack8(const unsigned* w) {
  return make_uint4(w[0] | (w[1] << 16), w[2] | (w[3] << 16), w[4] | (w[5] << 16), w[6] | (w[7] << 16));
}
// the items of each gradient slot (codes in tsm_device.h): the first chain in
// items if it has up to eight neighbours, everything else in groups (read by tiles
// marked special only); special[t] is set where a tile has anything but such chains
// around the slots themselves.
__global__ void k_fill_items(TabIn T, int nq, int ms1, const int* ovp, uint4* items, uint4* items2,
                             int2* item_x, uint4* ov, unsigned char* special, int* bad) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  int t, k, v;
  gs_find(T, q, t, k, v);
  int first = 0, pos = 0;  // neighbours of the first chain
  bool open = true;
  walk_items(T, v, [&](int kind, int, bool) {
    if (kind == 0 && open) ++first;
    else if (!(pos == 0 && kind == 1)) open = false;
    ++pos;
  });
  const bool inl = first <= 8;
  unsigned w[8], g[8];
  for (int u = 0; u < 8; ++u) w[u] = g[u] = SI_END;
  int n = 0, groups = 0, seen = 0, at = 0, start = k, centre = k;
  uint4 g0 = pack8(g);
  auto put = [&]() {  // the group is full or the next item needs another
    if (groups == 0) g0 = pack8(g);
    else ov[ovp[q] + groups - 1] = pack8(g);
    ++groups;
    n = 0;
    for (int u = 0; u < 8; ++u) g[u] = SI_END;
  };
  walk_items(T, v, [&](int kind, int id, bool closed) {
    if (kind == 2) {
      const int b0 = T.btbeg[t], b1 = T.btbeg[t + 1];
      const int j = find32(T.bt, b0, b1, id) - b0;
      if (j > SI_MASK) atomicOr(bad, 1);
      if (n > 0 && ((g[0] & 0xc000u) != SI_TERM || n == 8)) put();
      if (n == 0) g[n++] = SI_TERM;
      g[n++] = SI_TERM | (unsigned)(j & SI_MASK);
    } else {
      const int s = slot_in(T, t, id);
      if (s < 0 || s > SI_MASK) atomicOr(bad, 1);
      if (kind == 1) {
        centre = s;
        if (at == 0) start = s;
        if (n > 0) put();
      } else {
        const unsigned e = (closed ? SI_CLOSED : 0u) | (unsigned)(s & SI_MASK);
        if (inl && seen < first) {
          w[seen] = e;
        } else {
          if (n == 8) {  // the chain goes on
            g[0] |= SI_CLOSED;
            put();
            g[n++] = SI_CENTRE | SI_FLAG | (unsigned)(centre & SI_MASK);
          } else if (n == 0) {
            g[n++] = SI_CENTRE | (unsigned)(centre & SI_MASK);
          }
          g[n++] = e;
        }
        ++seen;
      }
    }
    ++at;
  });
  if (n > 0) put();
  if (groups - 1 > ovp[q + 1] - ovp[q]) atomicOr(bad, 1);
  const size_t o = (size_t)t * ms1 + k;
  items[o] = pack8(w);
  items2[o] = g0;
  item_x[o] = make_int2((start & SI_MASK) | (max(groups - 1, 0) << 12), ovp[q]);
  if (groups > 0 || start != k) special[t] = 1;
}
// boundary entries: per vertex their count, then the entries
__device__ __forceinline__ int vertex_faces(const int* gptr, const unsigned short* gent, int v) {
  const int k0 = gptr[v], n = gptr[v + 1] - k0;
  int nf = 0;
  while (nf < n && !(gent[k0 + nf] & 0x4000u)) ++nf;
  return nf;
}
__global__ void k_be_count(int nv, const int* gptr, const unsigned short* gent, int* cnt) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v <= nv) cnt[v] = v < nv ? gptr[v + 1] - gptr[v] - vertex_faces(gptr, gent, v) : 0;
}
__global__ void k_be_fill(TabIn T, const int* gptr, const unsigned short* gent, const int* bbeg,
                          const int* tbf, const int* vbp, int2* be) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= T.G.nv) return;
  const int n = vbp[v + 1] - vbp[v];
  if (n == 0) return;
  const int t = tile_of(T, v), k0 = gptr[v + 1] - n;
  for (int i = 0; i < n; ++i) {
    const int b = tbf[bbeg[t] + (gent[k0 + i] & 0x3fffu)];
    be[vbp[v] + i] = make_int2(b, (v - T.vbeg[t]) | (bc_end(T.G, b, v) << 16));
  }
}
__global__ void k_be_max(TabIn T, const int* vbp, int* mx) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < T.nt) atomicMax(mx + N_MB, vbp[T.vbeg[t + 1]] - vbp[T.vbeg[t]]);
}
// the first eight gather entries of each vertex
__global__ void k_ge8(TabIn T, int bf0, const int* gptr, const unsigned short* gent, const int* vbp,
                      uint4* ge8, int* bad) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= T.G.nv) return;
  const int k0 = gptr[v], n = gptr[v + 1] - k0, nf = n - (vbp[v + 1] - vbp[v]);
  int k = 0;  // the tile's boundary entries before this vertex's
  if (nf < n) k = vbp[v] - vbp[T.vbeg[tile_of(T, v)]];
  unsigned w[8];
  for (int u = 0; u < 8; ++u) w[u] = GE_END;
  const int m = n <= 8 ? n : 7;
  for (int u = 0; u < m; ++u) w[u] = u < nf ? gent[k0 + u] : (unsigned)(bf0 + k + u - nf);
  if (bf0 + k + n - nf > 0x3fff) atomicOr(bad, 1);
  if (m < n) w[m] = GE_MORE;
  ge8[v] = pack8(w);
}
// boundary terms with their vertices
__global__ void k_bt4(DevGeo G, const int* n, const int* bt, int4* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= *n) return;
  const int b = bt[i];
  out[i] = make_int4(b, G.bv[2 * b], G.bv[2 * b + 1], 0);
}
// viscous cells: (tile, cell) of every cell of an owned vertex that is no wall cell
__global__ void k_vcell_keys(TabIn T, unsigned long long* keys) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= T.G.nv) return;
  const int t = tile_of(T, v);
  for (int e = T.G.vc_ptr[v]; e < T.G.vc_ptr[v + 1]; ++e) {
    const int c = T.G.vc[e] & 0x7fffffff;
    keys[e] = T.G.cnb[c] ? ~0ull : ((unsigned long long)(unsigned)t << 32) | (unsigned)c;
  }
}
// their corners as slots, one stride per tile
__global__ void k_vcells(TabIn T, int mc, const int* beg, const int* cells, unsigned* out, int* bad) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)T.nt * mc) return;
  const int t = (int)(i / mc), j = (int)(i % mc);
  unsigned x = ~0u;
  if (j < beg[t + 1] - beg[t]) {
    const int c = cells[beg[t] + j];
    x = 0;
    for (int z = 0; z < 3; ++z) {
      const int s = slot_in(T, t, T.G.cv[3 * (size_t)c + z]);
      if (s < 0 || s > 1023) atomicOr(bad, 1);
      x |= (unsigned)(s & 1023) << (10 * z);
    }
  }
  out[i] = x;
}
// per vertex, in cell order: the tile's viscous cell | the vertex's corner << 13
// (along G.vc; wall cells leave no entry), and the first eight of them packed
__global__ void k_vcell_entries(TabIn T, const int* beg, const int* cells, unsigned short* ent,
                                int* cnt, uint4* vc8, int* bad) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= T.G.nv) return;
  const int t = tile_of(T, v);
  int n = 0;
  unsigned w[8];
  for (int u = 0; u < 8; ++u) w[u] = GE_END;
  for (int e = T.G.vc_ptr[v]; e < T.G.vc_ptr[v + 1]; ++e) {
    const int c = T.G.vc[e] & 0x7fffffff;
    if (T.G.cnb[c]) continue;
    const int j = find32(cells, beg[t], beg[t + 1], c) - beg[t];
    const int z = T.G.cv[3 * (size_t)c] == v ? 0 : (T.G.cv[3 * (size_t)c + 1] == v ? 1 : 2);
    if (j > 0x1fff) atomicOr(bad, 1);
    const unsigned x = ((unsigned)z << 13) | (unsigned)(j & 0x1fff);
    ent[T.G.vc_ptr[v] + n] = (unsigned short)x;
    if (n < 8) w[n] = x;
    ++n;
  }
  cnt[v] = n;
  vc8[v] = pack8(w);
}
// wall terms: (tile, bface) of every bface whose cell holds an owned vertex
__global__ void k_wall_keys(TabIn T, unsigned long long* keys) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= T.G.nv) return;
  const int t = tile_of(T, v);
  for (int e = T.G.vbe_ptr[v]; e < T.G.vbe_ptr[v + 1]; ++e)
    keys[e] = ((unsigned long long)(unsigned)t << 32) | ((unsigned)T.G.vbe[e] & 0x7fffffffu);
}
__global__ void k_wall_cells(TabIn T, const int* wtbeg, const int* wt, uint4* wcell, int* bad) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= wtbeg[T.nt]) return;
  const DevGeo& G = T.G;
  int t = 0, end = T.nt;
  while (end - t > 1) {
    const int m = (t + end) >> 1;
    if (wtbeg[m] <= j) t = m; else end = m;
  }
  const int c = G.blc[wt[j]];
  int s[3];
  for (int z = 0; z < 3; ++z) {
    s[z] = slot_in(T, t, G.cv[3 * (size_t)c + z]);
    if (s[z] < 0 || s[z] > SI_MASK) { atomicOr(bad, 1); s[z] = 0; }
  }
  unsigned jt[2] = {0xffffu, 0xffffu};
  for (int z = 0; z < 2; ++z) {
    const int b = G.cbf[2 * (size_t)c + z];
    if (b < 0) break;
    if (!bc_sets_state(G.btype[b])) continue;
    jt[z] = (unsigned)z;
    if (T.grad) {
      const int k = find32(T.bt, T.btbeg[t], T.btbeg[t + 1], b);
      if (k >= T.btbeg[t + 1] || T.bt[k] != b) atomicOr(bad, 1);
      jt[z] = (unsigned)(k - T.btbeg[t]) & 0xffffu;
    }
  }
  uint4* o = wcell + 3 * (size_t)j;
  o[0] = make_uint4((unsigned)wt[j], (unsigned)s[0] | ((unsigned)s[1] << 16), (unsigned)s[2],
                    jt[0] | (jt[1] << 16));
  for (int z = 0; z < 2; ++z) {
    const int f = G.cwf[2 * c + z];
    uint4 q = make_uint4(0, 0, 0, 0xffffffffu);
    if (f >= 0) {
      const int b = G.cwb[2 * c + z], v0 = G.fv[2 * f], v1 = G.fv[2 * f + 1];
      if (b > 0x3fffffff) atomicOr(bad, 1);
      q = make_uint4((unsigned)v0, (unsigned)v1,
                     (unsigned)b | ((unsigned)bc_end(G, b, v0) << 30) | ((unsigned)bc_end(G, b, v1) << 31),
                     (unsigned)f);
    }
    o[1 + z] = q;
  }
}
// per (vertex, bface) in bface order: the tile's wall term, the vertex's corner
// of the cell and whether the vertex ends the bface
__global__ void k_wall_entries(TabIn T, const int* wtbeg, const int* wt, unsigned short* wvent, int* bad) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= T.G.nv) return;
  const int t = tile_of(T, v);
  for (int e = T.G.vbe_ptr[v]; e < T.G.vbe_ptr[v + 1]; ++e) {
    const unsigned x = (unsigned)T.G.vbe[e];
    const int b = (int)(x & 0x7fffffffu), c = T.G.blc[b];
    const int j = find32(wt, wtbeg[t], wtbeg[t + 1], b) - wtbeg[t];
    const int z = T.G.cv[3 * (size_t)c] == v ? 0 : (T.G.cv[3 * (size_t)c + 1] == v ? 1 : 2);
    if (j > SI_MASK) atomicOr(bad, 1);
    wvent[e] = (unsigned short)((x >> 31 ? 0x8000u : 0u) | ((unsigned)z << 13) | (unsigned)(j & SI_MASK));
  }
}
__global__ void k_zero(long long n, unsigned char* p) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace

int build_stage_tables(const DevGeo& G, const TileGeo& TG, bool grad, bool ns, int n_wall,
                       StageTab& S, const std::function<int(void**, size_t)>& dalloc, hipStream_t st,
                       std::string& msg) {
#define TT(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { msg = std::string("stage tables: ") + hipGetErrorString(e_); return TSM_E_HIP; } } while (0)
#define TA(ptr, n) do { void* q_ = nullptr; int r_ = dalloc(&q_, std::max<size_t>((size_t)(n), 1) * sizeof(*(ptr))); if (r_) { msg = "stage tables: allocation"; return r_; } (ptr) = static_cast<std::remove_reference_t<decltype(ptr)>>(q_); } while (0)
#define GO(k, n, ...) hipLaunchKernelGGL(k, dim3(nblk(n)), dim3(256), 0, st, __VA_ARGS__)
  const int nv = G.nv, nt = TG.ntiles, n_inc = 3 * G.nc;
  S = StageTab{};
  S.ntiles = nt; S.tb = TG.tb; S.fu_block = TG.fu_block; S.n_periodic_tiles = TG.n_periodic_tiles;
  S.tper = TG.tper; S.pinfo = TG.pinfo; S.gptr = TG.gptr; S.gent = TG.gent;
  const int nq = nv + (grad ? TG.nhalo : 0);
  TabIn T{};
  T.G = G; T.nt = nt; T.grad = grad ? 1 : 0;
  T.vbeg = TG.vbeg; T.hbeg = TG.hbeg; T.halo = TG.halo;
  TmpPool tmp;
  auto scan = [&](const int* in, int* out, int n) -> hipError_t {
    size_t b = 0;
    char* p = nullptr;
    hipError_t e = hipcub::DeviceScan::ExclusiveSum(nullptr, b, in, out, n, st);
    if (e == hipSuccess) e = tmp.get(&p, b);
    return e == hipSuccess ? hipcub::DeviceScan::ExclusiveSum(p, b, in, out, n, st) : e;
  };
  // sorted distinct keys: where each tile's start (beg), their low words (list)
  auto group = [&](unsigned long long* k, int n, int* beg, int** list) -> int {
    unsigned long long *ks = nullptr, *ku = nullptr;
    int* nu = nullptr;
    TT(tmp.get(&ks, n)); TT(tmp.get(&ku, n)); TT(tmp.get(&nu, 1)); TT(tmp.get(list, n));
    if (n > 0) {
      size_t b1 = 0, b2 = 0;
      char* p = nullptr;
      TT(hipcub::DeviceRadixSort::SortKeys(nullptr, b1, k, ks, n, 0, 64, st));
      TT(hipcub::DeviceSelect::Unique(nullptr, b2, ks, ku, nu, n, st));
      TT(tmp.get(&p, std::max(b1, b2)));
      TT(hipcub::DeviceRadixSort::SortKeys(p, b1, k, ks, n, 0, 64, st));
      TT(hipcub::DeviceSelect::Unique(p, b2, ks, ku, nu, n, st));
      GO(k_low, n, nu, ku, *list);
    } else {
      GO(k_zero_int, 1, 1, nu);
    }
    GO(k_seg, nt + 1, nt, ku, nu, beg);
    return 0;
  };
  int *mx = nullptr, h[N_COUNTS];
  TT(tmp.get(&mx, N_COUNTS));
  GO(k_zero_int, N_COUNTS, (int)N_COUNTS, mx);
  int* bad = mx + N_BAD;
  auto counts = [&]() -> hipError_t {
    hipError_t e = hipMemcpyAsync(h, mx, sizeof(h), hipMemcpyDeviceToHost, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  };
  unsigned char* special = nullptr;
  TT(tmp.get(&special, nt));
  GO(k_zero, nt, (long long)nt, special);
  // ---- boundary entries ---------------------------------------------------------
  int *becnt = nullptr, *vbp = nullptr;
  TT(tmp.get(&becnt, nv + 1));
  TA(vbp, nv + 1);
  GO(k_be_count, nv + 1, nv, TG.gptr, TG.gent, becnt);
  TT(scan(becnt, vbp, nv + 1));
  GO(k_be_max, nt, T, vbp, mx);
  // ---- fans, second ring and boundary terms ---------------------------------------
  int *ovp = nullptr, *halo2 = nullptr, *btbeg = nullptr, *bt = nullptr;
  if (grad) {
    unsigned char* used = nullptr;
    int *fan_n = nullptr, *ng = nullptr, *h2beg = nullptr;
    unsigned* fan = nullptr;
    TT(tmp.get(&used, n_inc)); TT(tmp.get(&fan_n, nv)); TT(tmp.get(&fan, 2 * (size_t)n_inc));
    int2* gs = nullptr;
    TT(tmp.get(&ng, nq + 1)); TT(tmp.get(&ovp, nq + 1)); TT(tmp.get(&h2beg, nt + 1)); TT(tmp.get(&gs, nq));
    TA(btbeg, nt + 1);
    hipLaunchKernelGGL(k_fan, dim3((nv + 63) / 64), dim3(64), 0, st, G, used, fan_n, fan);
    T.fan_n = fan_n;
    T.fan = fan;
    GO(k_gs_count, nq + 1, T, nq, gs, ng, mx);
    TT(scan(ng, ovp, nq + 1));
    GO(k_totals, 1, vbp + nv, ovp + nq, mx);
    TT(counts());
    const int c2 = h[N_RING2], cb = h[N_TERMS];
    if (c2 < 0 || cb < 0) { msg = "stage tables: too many entries"; return 1; }
    unsigned long long *k2 = nullptr, *kb = nullptr;
    TT(tmp.get(&k2, c2)); TT(tmp.get(&kb, cb));
    GO(k_gs_emit, nq, T, nq, gs, k2, kb, mx);
    if (int r = group(k2, c2, h2beg, &halo2)) return r;
    if (int r = group(kb, cb, btbeg, &bt)) return r;
    T.h2beg = h2beg; T.halo2 = halo2; T.btbeg = btbeg; T.bt = bt;
  } else {
    GO(k_totals, 1, vbp + nv, (const int*)nullptr, mx);
  }
  // ---- wall terms -------------------------------------------------------------
  int *wtbeg = nullptr, *wt = nullptr;
  if (n_wall > 0) {
    unsigned long long* k = nullptr;
    TT(tmp.get(&k, n_wall));
    TA(wtbeg, nt + 1);
    GO(k_wall_keys, nv, T, k);
    if (int r = group(k, n_wall, wtbeg, &wt)) return r;
    uint4* wcell = nullptr;
    unsigned short* wvent = nullptr;
    TA(wcell, 3 * (size_t)n_wall);
    TA(wvent, n_wall);
    GO(k_wall_cells, n_wall, T, wtbeg, wt, wcell, bad);
    GO(k_wall_entries, nv, T, wtbeg, wt, wvent, bad);
    S.wtbeg = wtbeg; S.wcell = wcell; S.wvent = wvent;
  }
  // ---- viscous cells ----------------------------------------------------------
  int *tcbeg = nullptr, *tc = nullptr;
  if (ns) {
    unsigned long long* k = nullptr;
    TT(tmp.get(&k, n_inc));
    TT(tmp.get(&tcbeg, nt + 1));
    GO(k_vcell_keys, nv, T, k);
    if (int r = group(k, n_inc, tcbeg, &tc)) return r;
    unsigned short* ent = nullptr;
    int* cnt = nullptr;
    uint4* vc8 = nullptr;
    TA(ent, n_inc); TA(cnt, nv); TA(vc8, nv);
    GO(k_vcell_entries, nv, T, tcbeg, tc, ent, cnt, vc8, bad);
    S.vcent = ent; S.vccnt = cnt; S.vc8 = vc8;
  }
  GO(k_desc, nt, T, TG.fbeg, wtbeg, tcbeg, special, (int4*)nullptr, mx);
  TT(counts());
  S.ms = h[N_MS]; S.ms1 = h[N_MS1]; S.mf = h[N_MF]; S.mbt = h[N_MBT]; S.mwt = h[N_MWT]; S.mc = h[N_MC];
  S.mb = h[N_MB];
  S.bf0 = stage_main_records(S, grad, ns);
  if (S.ms > SI_MASK || h[N_BAD]) { msg = "stage tables: too many slots or entries"; return 1; }
  // ---- padded tables ------------------------------------------------------------
  int* sid = nullptr;
  unsigned* lr = nullptr;
  double2 *fn = nullptr, *xy = nullptr;
  uint4 *it = nullptr, *it2 = nullptr, *ge = nullptr;
  int4* desc = nullptr;
  TA(sid, (size_t)nt * S.ms); TA(lr, (size_t)nt * S.mf); TA(fn, (size_t)nt * S.mf);
  TA(xy, nv); TA(ge, nv); TA(desc, nt);
  GO(k_fill_sid, (long long)nt * S.ms, T, S.ms, sid);
  GO(k_fill_faces, (long long)nt * S.mf, nt, S.mf, TG.fbeg, TG.f_lr, TG.f_n, lr, fn);
  GO(k_xy, nv, nv, G.x, G.y, xy);
  int2* be = nullptr;
  TA(be, h[N_BE]);
  GO(k_be_fill, nv, T, TG.gptr, TG.gent, TG.bbeg, TG.tbf, vbp, be);
  GO(k_ge8, nv, T, S.bf0, TG.gptr, TG.gent, vbp, ge, bad);
  S.vbp = vbp; S.be = be;
  if (grad) {
    int2* itx = nullptr;
    uint4* ov = nullptr;
    int4* bt4 = nullptr;
    TA(it, (size_t)nt * S.ms1); TA(it2, (size_t)nt * S.ms1); TA(itx, (size_t)nt * S.ms1);
    TA(ov, h[N_OV]); TA(bt4, h[N_TERMS]);
    if (h[N_TERMS] > 0) GO(k_bt4, h[N_TERMS], G, btbeg + nt, bt, bt4);
    GO(k_fill_items, nq, T, nq, S.ms1, ovp, it, it2, itx, ov, special, bad);
    S.items = it; S.items2 = it2; S.item_x = itx; S.ov = ov; S.btbeg = btbeg; S.bt = bt4;
  }
  if (ns) {
    unsigned* vcells = nullptr;
    TA(vcells, (size_t)nt * S.mc);
    GO(k_vcells, (long long)nt * S.mc, T, S.mc, tcbeg, tc, vcells, bad);
    S.vcells = vcells;
  }
  GO(k_desc, nt, T, TG.fbeg, wtbeg, tcbeg, special, desc, (int*)nullptr);
  TT(hipGetLastError());
  TT(counts());
  if (h[N_BAD]) { msg = "stage tables: entry out of range"; return 1; }
  S.desc = desc; S.sid = sid; S.f_lr = lr; S.f_n = fn; S.xy = xy; S.ge8 = ge;
#undef TT
#undef TA
#undef GO
  return 0;
}

}  // namespace tsm
