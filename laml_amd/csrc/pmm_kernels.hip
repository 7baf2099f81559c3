// PMM inside / outside / posterior / M-step kernels for gfx950.
//
// Layout (one forest = many trees, grouped into problems):
//  - nodes are numbered in height-level order; a level is a contiguous range.
//  - every (node, site) value lives in a row of K_t contiguous sites; leaf rows
//    (int16 codes) and internal rows (beta, alpha, labels) are packed
//    separately, row_off[v] giving the row start in the matching array.
//  - internal rows hold beta = (b0, bA) mantissas with a shared exponent bE
//    (inside, below the node), the az-partition label, and the outside state
//    alpha = (a0, aX), conditional on all data (see cond_post).
//
// A segment of W lanes handles one node and strides over its K sites, so
// per-node reductions over sites are segment shuffles.
#include "pmm_kernels.hpp"

#include <algorithm>
#include <map>
#include <mutex>

namespace laml {

__device__ __forceinline__ Coef branch_coef(double dv, double nv) {
  Coef c;
  c.p1n = exp(-(1.0 + nv) * dv);
  c.pn = exp(-nv * dv);
  c.mut = -expm1(-dv) * c.pn;
  int es;
  c.msil = frexp(-expm1(-nv * dv), &es);
  c.esil = c.msil != 0.0 ? es : 0;
  c.pad = 0;
  return c;
}

// branch v's coefficients to its place in the steps of the clade plan
__device__ __forceinline__ void clade_coef(const DevForest& F, int v, const Coef& c) {
  const int q = F.clade_pos[v];
  if (q < 0) return;
  CladeCoef& r = F.clade_coef[q >> 1];
  const int i = q & 1;
  r.p1n[i] = c.p1n;
  r.mut[i] = c.mut;
  r.pn[i] = c.pn;
  r.msil[i] = c.msil;
  r.esil[i] = c.esil;
}

__global__ void k_coef(DevForest F, const double* __restrict__ d, const double* __restrict__ nu,
                       const int32_t* __restrict__ done) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= F.num_nodes) return;
  const int p = F.tree_prob[F.tree_of[v]];
  if (done && done[p]) return;
  const Coef c = branch_coef(d[v], nu[p]);
  F.coef[v] = c;
  if (F.clade_pos) clade_coef(F, v, c);
}

// the resident coefficients into a clade plan's steps
__global__ void k_clade_coef(DevForest F) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < F.num_nodes) clade_coef(F, v, F.coef[v]);
}

// Segment mapping shared by the level kernels: a block of 256 threads holds
// 256/W segments of W lanes; segment s of a level handles node beg+s, and
// blockIdx.y selects the chunk of W consecutive sites of that node.
template <int W>
struct Seg {
  int v, lane, k;
  __device__ __forceinline__ bool init(int beg, int cnt) {
    const int seg = blockIdx.x * (256 / W) + (int)(threadIdx.x / W);
    lane = threadIdx.x & (W - 1);
    if (seg >= cnt) return false;
    v = beg + seg;
    k = (int)blockIdx.y * W + lane;
    return true;
  }
};

template <int W>
__global__ void __launch_bounds__(256) k_labels(DevForest F, int beg, int cnt) {
  Seg<W> g;
  if (!g.init(beg, cnt)) return;
  const int v = g.v, k = g.k;
  const int t = F.tree_of[v];
  if (k >= F.tree_nsites[t]) return;
  const int c1 = F.child0[v], c2 = F.child1[v];
  const int la = c1 < F.num_leaves ? code_label(F.codes[F.row_off[c1] + k]) : (int)F.labels[F.row_off[c1] + k];
  const int lb = c2 < F.num_leaves ? code_label(F.codes[F.row_off[c2] + k]) : (int)F.labels[F.row_off[c2] + k];
  F.labels[F.row_off[v] + k] = (int16_t)combine_label(la, lb);
}

// Prior-weight rows of every node (a wavefront per row; sites past the
// tree's up to the row stride get 0).
__global__ void __launch_bounds__(256) k_qrows(DevForest F, double* __restrict__ qleaf, double* __restrict__ qint) {
  const int lane = (int)(threadIdx.x & 63);
  const int W = F.chunk_w;
  for (int v = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6); v < F.num_nodes; v += (int)gridDim.x * 4) {
    const int t = F.tree_of[v];
    const int K = F.tree_nsites[t];
    const int stride = (K + W - 1) / W * W;
    const int sb = F.tree_site_base[t];
    const int64_t ro = F.row_off[v];
    const bool leaf = v < F.num_leaves;
    double* dst = (leaf ? qleaf : qint) + ro;
    for (int k = lane; k < stride; k += 64) {
      double q = 0.0;
      if (k < K) {
        const int lab = leaf ? code_label(F.codes[ro + k]) : (int)F.labels[ro + k];
        q = lab > 0 ? F.prior[F.site_qoff[sb + k] - 1 + lab] : F.site_qsum[sb + k];
      }
      dst[k] = q;
    }
  }
}

// Leaf code rows from the caller's packed layout (leaf v's K codes at
// packed_off[v], rows back to back) into the device rows, padded to a
// multiple of the segment width with code 0; a wavefront per row.
__global__ void __launch_bounds__(256) k_pad_codes(DevForest F, const int16_t* __restrict__ packed,
                                                   const int64_t* __restrict__ packed_off) {
  const int lane = (int)(threadIdx.x & 63);
  const int W = F.chunk_w;
  int16_t* codes = const_cast<int16_t*>(F.codes);
  for (int v = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6); v < F.num_leaves; v += (int)gridDim.x * 4) {
    const int K = F.tree_nsites[F.tree_of[v]];
    const int stride = (K + W - 1) / W * W;
    const int16_t* src = packed + packed_off[v];
    int16_t* dst = codes + F.row_off[v];
    for (int k = lane; k < stride; k += 64) dst[k] = k < K ? src[k] : (int16_t)0;
  }
}

// load the inside state of node c at site k (labels/codes by row_off, the
// inside vector by brow, which differs from row_off under level checkpointing)
__device__ __forceinline__ void load_child(const DevForest& F, int c, bool leaf, int k, double phi, int& lab,
                                           double& b0, double& bA, int& E, int& code) {
  const int64_t r = F.row_off[c];
  if (leaf) {
    code = F.codes[r + k];
    leaf_beta(code, phi, lab, b0, bA);
    E = 0;
  } else {
    code = 0;
    lab = F.labels[r + k];
    const int64_t br = F.brow[c];
    const double2 bb = F.beta[br + k];
    b0 = bb.x;
    bA = bb.y;
    E = F.bE[br + k];
  }
}

// Element k of a row: the byte offset is formed in 32 bits, so that with a
// wave-uniform row pointer the access is a scalar base plus a 32-bit lane
// offset (rows hold fewer than 2^24 sites; the forest checks it).
template <typename T>
__device__ __forceinline__ T& row_at(T* p, unsigned k) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(p) + k * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ const T& row_at(const T* p, unsigned k) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + k * (unsigned)sizeof(T));
}

// A load of data that no kernel writes while it runs (launch plans, node
// records, branch coefficients), through the constant address space: at a
// wave-uniform address the compiler may then issue it as a scalar load into
// SGPRs even after the kernel's own stores, where it must otherwise assume
// the store may have changed it and load it into VGPRs of every lane (other
// addresses stay vector loads).
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "loaded as 32-bit words");
  typedef const __attribute__((address_space(4))) uint32_t* WordPtr;
  const WordPtr q = (WordPtr)(uintptr_t)p;
  uint32_t w[sizeof(T) / 4];
#pragma unroll
  for (unsigned i = 0; i < sizeof(T) / 4; ++i) w[i] = q[i];
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// the wavefront's LDS stores so far are done and visible to its own loads
__device__ __forceinline__ void lds_wave_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Kinds of child a pass kernel meets.  A *cherry* is an internal node whose
// children are both leaves; when the pass fuses cherries (F.cherry_end >
// F.num_leaves: nodes [num_leaves, cherry_end) are exactly the cherries, the
// whole height-1 level) no cherry row is stored: its parent forms the
// cherry's inside vector from the two leaf codes, and in the outside pass
// runs the cherry's posterior step itself, so the height-1 level costs no
// launch and no row traffic.
// Template kind arguments: a fixed kind, or kNoCherry (leaf or internal,
// read at run time: kernels that never meet a fused cherry carry no cherry
// code).
constexpr int kInternal = 0, kLeaf = 1, kCherry = 2, kNoCherry = -2;

__device__ __forceinline__ int child_kind(const DevForest& F, int c) {
  return c < F.num_leaves ? kLeaf : (c < F.cherry_end ? kCherry : kInternal);
}

template <int KT>
__device__ __forceinline__ int resolve_kind(int k) {
  return KT >= 0 ? KT : (KT == kNoCherry ? (k == kLeaf ? kLeaf : kInternal) : k);
}

// Rows of one child node at its parent's sites: leaf codes, label + inside
// vector, or (cherry) the codes and branch coefficients of its two leaves.
// Held as pointers to the row start so that, where the node is wave-uniform,
// every per-site access is a scalar base plus a 32-bit lane offset.
struct ChildRows {
  const int16_t* code;   // leaf codes (leaf), az-partition labels (internal), first leaf's codes (cherry)
  const double2* beta;   // inside mantissas (internal)
  const int32_t* bE;     // inside exponent (internal)
  const int16_t* code2;  // second leaf's codes (cherry)
  Coef g[2];             // the cherry's leaf branches
  int gc[2];             // the cherry's leaves
};

__device__ __forceinline__ ChildRows child_rows(const DevForest& F, int c, int kind) {
  ChildRows r;
  r.beta = nullptr;
  r.bE = nullptr;
  r.code2 = nullptr;
  r.gc[0] = r.gc[1] = -1;
  if (kind == kLeaf) {
    r.code = F.codes + F.row_off[c];
  } else if (kind == kCherry) {
    const int a = F.child0[c], b = F.child1[c];
    r.code = F.codes + F.row_off[a];
    r.code2 = F.codes + F.row_off[b];
    r.g[0] = F.coef[a];
    r.g[1] = F.coef[b];
    r.gc[0] = a;
    r.gc[1] = b;
  } else {
    const int64_t br = F.brow[c];
    r.code = F.labels + F.row_off[c];
    r.beta = F.beta + br;
    r.bE = F.bE + br;
  }
  return r;
}
__device__ __forceinline__ ChildRows child_rows(const DevForest& F, int c, bool leaf) {
  return child_rows(F, c, leaf ? kLeaf : kInternal);
}

// inside vector of a leaf at site k, seen from its parent over its branch
__device__ __forceinline__ Eps leaf_edge(int code, double phi, const double* __restrict__ prior, int qo, double qs,
                                         const Coef& cf, int& lab) {
  double b0, bA;
  leaf_beta(code, phi, lab, b0, bA);
  const double q = lab > 0 ? row_at(prior, (unsigned)(qo + lab)) : qs;
  return edge(lab, b0, bA, 0, q, cf);
}

// The inside vector a cherry's node would store at site k: the same
// operations as the inside pass for a node with two leaf children.
__device__ __forceinline__ void cherry_beta(const ChildRows& r, int k, double phi, const double* __restrict__ prior,
                                            int qo, double qs, int& lab, double& b0, double& bA, int& E) {
  int la, lb;
  const Eps ea = leaf_edge(row_at(r.code, k), phi, prior, qo, qs, r.g[0], la);
  const Eps eb = leaf_edge(row_at(r.code2, k), phi, prior, qo, qs, r.g[1], lb);
  lab = combine_label(la, lb);
  const double B0 = ea.e0 * eb.e0;
  const double BA = lab != 0 ? ea.eA * eb.eA : 0.0;
  const int sh = min(-exp_of(fmax(B0, BA)), 1000);
  const double sc = ldexp(1.0, sh);
  b0 = B0 * sc;
  bA = BA * sc;
  E = ea.e + eb.e - sh;
}

// inside state of a child at site k (qo, qs: the site's prior offset and
// mass, used for a cherry's leaves).  stream: read the inside row with the
// non-temporal hint (the inside pass reads each row once).
__device__ __forceinline__ void load_child_rows(const ChildRows& r, int kind, int k, double phi,
                                                const double* __restrict__ prior, int qo, double qs, int& lab,
                                                double& b0, double& bA, int& E, int& code, bool stream = false) {
  if (kind == kLeaf) {
    code = row_at(r.code, k);
    leaf_beta(code, phi, lab, b0, bA);
    E = 0;
  } else if (kind == kCherry) {
    code = 0;
    cherry_beta(r, k, phi, prior, qo, qs, lab, b0, bA, E);
  } else {
    code = 0;
    lab = row_at(r.code, k);
    const double2 bb = stream ? load_stream(&row_at(r.beta, k)) : row_at(r.beta, k);
    b0 = bb.x;
    bA = bb.y;
    E = row_at(r.bE, k);
  }
}
__device__ __forceinline__ void load_child_rows(const ChildRows& r, bool leaf, int k, double phi, int& lab,
                                                double& b0, double& bA, int& E, int& code) {
  load_child_rows(r, leaf ? kLeaf : kInternal, k, phi, nullptr, 0, 0.0, lab, b0, bA, E, code);
}

// per-node values of the inside pass (uniform over the sites of the node)
struct InNode {
  int K;
  int kind[2];
  Coef cf[2];
  ChildRows c[2];
  const int16_t* lab;    // the node's labels
  double2* beta;         // the node's inside row
  int32_t* bE;
  const int32_t* qoff;   // prior offsets of the tree's sites
  const double* qsum;    // prior mass of the tree's sites
  double phi;
  bool stream;           // rows with the non-temporal hint
};

// CH: the node may have a fused cherry child (otherwise children are leaves
// or stored internal nodes, and no cherry code is generated)
template <bool CH>
__device__ __forceinline__ void in_node_load(const DevForest& F, int v, int t, int p, int K, InNode& n) {
  n.K = K;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = i == 0 ? F.child0[v] : F.child1[v];
    n.kind[i] = CH ? child_kind(F, c) : (c < F.num_leaves ? kLeaf : kInternal);
    n.cf[i] = F.coef[c];
    n.c[i] = child_rows(F, c, n.kind[i]);
  }
  n.lab = F.labels + F.row_off[v];
  const int64_t bv = F.brow[v];
  n.beta = F.beta + bv;
  n.bE = F.bE + bv;
  n.qoff = F.site_qoff + F.tree_site_base[t];
  n.qsum = F.site_qsum + F.tree_site_base[t];
  n.phi = F.phi[p];
  n.stream = F.stream_rows != 0;
}

// The inside step of one site in three phases: row loads, prior gathers
// (they need the loaded labels), then arithmetic and stores.
struct InSite {
  int lv, qo, la, lb, Ea, Eb, ca, cb;
  double qs, a0, aA, b0, bA, qa, qb;
};

template <int K0, int K1>
__device__ __forceinline__ void inside_load(const DevForest& F, const InNode& n, int k, InSite& x) {
  const int kind[2] = {resolve_kind<K0>(n.kind[0]), resolve_kind<K1>(n.kind[1])};
  x.lv = row_at(n.lab, k);
  x.qo = row_at(n.qoff, k) - 1;
  // a missing ('?') child may be in any edit state: its prior weight is the
  // site's total prior mass
  x.qs = row_at(n.qsum, k);
  load_child_rows(n.c[0], kind[0], k, n.phi, F.prior, x.qo, x.qs, x.la, x.a0, x.aA, x.Ea, x.ca, n.stream);
  load_child_rows(n.c[1], kind[1], k, n.phi, F.prior, x.qo, x.qs, x.lb, x.b0, x.bA, x.Eb, x.cb, n.stream);
}

__device__ __forceinline__ void inside_gather(const DevForest& F, InSite& x) {
  x.qa = x.la > 0 ? row_at(F.prior, (unsigned)(x.qo + x.la)) : x.qs;
  x.qb = x.lb > 0 ? row_at(F.prior, (unsigned)(x.qo + x.lb)) : x.qs;
}

__device__ __forceinline__ void inside_finish(const InNode& n, int k, const InSite& x) {
  const Eps ea = edge(x.la, x.a0, x.aA, x.Ea, x.qa, n.cf[0]);
  const Eps eb = edge(x.lb, x.b0, x.bA, x.Eb, x.qb, n.cf[1]);
  const double B0 = ea.e0 * eb.e0;
  const double BA = x.lv != 0 ? ea.eA * eb.eA : 0.0;
  // renormalise the pair by a power of two (bounded so that a denormal pair
  // cannot produce an infinite scale)
  const int sh = min(-exp_of(fmax(B0, BA)), 1000);
  const double sc = ldexp(1.0, sh);
  const double2 b = make_double2(B0 * sc, BA * sc);
  if (n.stream)
    store_stream(&row_at(n.beta, k), b);
  else
    row_at(n.beta, k) = b;
  row_at(n.bE, k) = ea.e + eb.e - sh;
}

// inside vector (below the node) of internal node n at site k.  K0 / K1: the
// kind of each child (kLeaf, kInternal, kCherry), or kNoCherry to read
// n.kind at run time.
template <int K0, int K1>
__device__ __forceinline__ void inside_site(const DevForest& F, const InNode& n, int k) {
  InSite x;
  inside_load<K0, K1>(F, n, k, x);
  inside_gather(F, x);
  inside_finish(n, k, x);
}
// the same with the children's prior weights read from their prior-weight
// rows q0, q1 (no load waits for the labels)
__device__ __forceinline__ void inside_site_q(const DevForest& F, const InNode& n, int k, const double* q0,
                                              const double* q1) {
  InSite x;
  inside_load<kNoCherry, kNoCherry>(F, n, k, x);
  x.qa = row_at(q0, k);
  x.qb = row_at(q1, k);
  inside_finish(n, k, x);
}

// The inside-pass values of internal node v from its record (children that
// are leaves or stored internal nodes).
__device__ __forceinline__ void in_node_rec(const DevForest& F, const NodeRec& r, InNode& n) {
  n.K = r.K;
  const int ch[2] = {r.ch0, r.ch1};
  const int64_t ro[2] = {r.ro0, r.ro1}, bro[2] = {r.bro0, r.bro1};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    n.kind[i] = ch[i] < F.num_leaves ? kLeaf : kInternal;
    n.cf[i] = uniform_load(F.coef + ch[i]);
    n.c[i].code = (n.kind[i] == kLeaf ? F.codes : F.labels) + ro[i];
    n.c[i].beta = F.beta + bro[i];
    n.c[i].bE = F.bE + bro[i];
    n.c[i].code2 = nullptr;
    n.c[i].gc[0] = n.c[i].gc[1] = -1;
  }
  n.lab = F.labels + r.ro;
  n.beta = F.beta + r.bro;
  n.bE = F.bE + r.bro;
  n.qoff = F.site_qoff + r.sb;
  n.qsum = F.site_qsum + r.sb;
  n.phi = uniform_load(F.phi + r.p);
  n.stream = F.stream_rows != 0;
}

// segment form: one site k of node v
__device__ __forceinline__ void inside_node(const DevForest& F, int v, int k, const int32_t* __restrict__ done) {
  const NodeRec r = F.nrec[v - F.num_leaves];
  if (k >= r.K) return;
  if (done && done[r.p]) return;
  InNode n;
  in_node_rec(F, r, n);
  inside_site<kNoCherry, kNoCherry>(F, n, k);
}

template <int W>
__global__ void __launch_bounds__(256) k_inside(DevForest F, int beg, int cnt, const int32_t* __restrict__ done) {
  Seg<W> g;
  if (!g.init(beg, cnt)) return;
  inside_node(F, g.v, g.k, done);
}

// Row form (K > 32): one wavefront per node walks chunks [c0, c0 + cpw) of 64
// sites.  The node number is wave-uniform, so the node's metadata are scalar
// loads and the child-kind tests scalar branches.
template <int K0, int K1>
__device__ __forceinline__ void inside_row_run(const DevForest& F, const InNode& n, int c0, int c1, int lane) {
  // software-pipelined over the wave's chunks: the rows and prior gathers of
  // chunk c + 1 are issued before chunk c's arithmetic and stores (they touch
  // other sites, so the order of memory accesses is free)
  InSite x;
  int k = c0 * 64 + lane;
  bool on = k < n.K;
  if (on) {
    inside_load<K0, K1>(F, n, k, x);
    inside_gather(F, x);
  }
  for (int c = c0; c < c1; ++c) {
    InSite y;
    const int kn = k + 64;
    const bool onn = c + 1 < c1 && kn < n.K;
    if (onn) inside_load<K0, K1>(F, n, kn, y);
    if (on) inside_finish(n, k, x);
    if (onn) inside_gather(F, y);
    x = y;
    k = kn;
    on = onn;
  }
}

// Both children leaves (the cherry level, whose rows are mostly written):
// the codes, labels and site values of the wavefront's chunks (at most
// kLeafGroup, their number a template argument so that the code is
// straight-line) are loaded first, then their prior gathers, then the
// arithmetic and stores, so that a wavefront waits twice instead of twice
// per chunk (a load issued after a store waits for the store too).  The
// per-chunk state is kept compact (raw codes until the arithmetic); same
// operations as inside_site, so the same bits.
constexpr int kLeafGroup = 8;
template <int NG>
__device__ __forceinline__ void inside_row_run_leaves_n(const DevForest& F, const InNode& n, int c0, int lane) {
  // lanes past the tree's sites load its last site, so that no load depends
  // on the lane mask
  int lv[NG], ca[NG], cb[NG], qo[NG];
  double qs[NG], ga[NG], gb[NG];
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    const unsigned kk = min((c0 + j) * 64 + lane, n.K - 1);
    lv[j] = row_at(n.lab, kk);
    qo[j] = row_at(n.qoff, kk);
    qs[j] = row_at(n.qsum, kk);
    ca[j] = row_at(n.c[0].code, kk);
    cb[j] = row_at(n.c[1].code, kk);
  }
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    const int la = code_label(ca[j]), lb = code_label(cb[j]);
    ga[j] = row_at(F.prior, (unsigned)(la > 0 ? qo[j] - 1 + la : 0));
    gb[j] = row_at(F.prior, (unsigned)(lb > 0 ? qo[j] - 1 + lb : 0));
  }
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    const int k = (c0 + j) * 64 + lane;
    if (k < n.K) {
      InSite x;
      x.lv = lv[j];
      x.qo = qo[j] - 1;
      x.qs = qs[j];
      x.ca = ca[j];
      x.cb = cb[j];
      leaf_beta(ca[j], n.phi, x.la, x.a0, x.aA);
      leaf_beta(cb[j], n.phi, x.lb, x.b0, x.bA);
      x.Ea = 0;
      x.Eb = 0;
      x.qa = x.la > 0 ? ga[j] : x.qs;
      x.qb = x.lb > 0 ? gb[j] : x.qs;
      inside_finish(n, k, x);
    }
  }
}
__device__ __forceinline__ void inside_row_run_leaves(const DevForest& F, const InNode& n, int c0, int c1, int lane) {
  switch (c1 - c0) {
    case 1: inside_row_run_leaves_n<1>(F, n, c0, lane); break;
    case 2: inside_row_run_leaves_n<2>(F, n, c0, lane); break;
    case 3: inside_row_run_leaves_n<3>(F, n, c0, lane); break;
    case 4: inside_row_run_leaves_n<4>(F, n, c0, lane); break;
    case 5: inside_row_run_leaves_n<5>(F, n, c0, lane); break;
    case 6: inside_row_run_leaves_n<6>(F, n, c0, lane); break;
    case 7: inside_row_run_leaves_n<7>(F, n, c0, lane); break;
    default: inside_row_run_leaves_n<8>(F, n, c0, lane); break;
  }
}

// The wave's node: entry beg + wv of a node list, or of the level range.
// Returns -1 past the end.
__device__ __forceinline__ int row_node(int beg, int cnt, const int32_t* __restrict__ nodes) {
  const int wv = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  if (wv >= cnt) return -1;
  return nodes ? __builtin_amdgcn_readfirstlane(nodes[beg + wv]) : beg + wv;
}

// Nodes whose children are leaves or stored internal nodes.
__global__ void __launch_bounds__(256) k_inside_rows(DevForest F, int beg, int cnt, int cpw,
                                                      const int32_t* __restrict__ done,
                                                      const int32_t* __restrict__ nodes) {
  const int v = row_node(beg, cnt, nodes);
  if (v < 0) return;
  const int lane = threadIdx.x & 63;
  const NodeRec r = F.nrec[v - F.num_leaves];
  const int nch = (r.K + 63) >> 6;
  const int c0 = (int)blockIdx.y * cpw;
  if (c0 >= nch) return;
  if (done && done[r.p]) return;
  const int c1 = min(c0 + cpw, nch);
  InNode n;
  in_node_rec(F, r, n);
  if (n.kind[0] == kLeaf) {
    if (n.kind[1] == kLeaf) inside_row_run<kLeaf, kLeaf>(F, n, c0, c1, lane);
    else inside_row_run<kLeaf, kInternal>(F, n, c0, c1, lane);
  } else {
    if (n.kind[1] == kLeaf) inside_row_run<kInternal, kLeaf>(F, n, c0, c1, lane);
    else inside_row_run<kInternal, kInternal>(F, n, c0, c1, lane);
  }
}

// The same for level 1, whose nodes have two leaf children (a separate
// kernel: its loads-first path needs more registers than the other levels'
// kernel should carry).
__global__ void __launch_bounds__(256) k_inside_rows_leaves(DevForest F, int beg, int cnt, int cpw,
                                                             const int32_t* __restrict__ done) {
  const int v = row_node(beg, cnt, nullptr);
  if (v < 0) return;
  const int lane = threadIdx.x & 63;
  const NodeRec r = F.nrec[v - F.num_leaves];
  const int nch = (r.K + 63) >> 6;
  const int c0 = (int)blockIdx.y * cpw;
  if (c0 >= nch) return;
  if (done && done[r.p]) return;
  const int c1 = min(c0 + cpw, nch);
  InNode n;
  in_node_rec(F, r, n);
  if (n.kind[0] == kLeaf && n.kind[1] == kLeaf) {
    if (c1 - c0 <= kLeafGroup) inside_row_run_leaves(F, n, c0, c1, lane);
    else inside_row_run<kLeaf, kLeaf>(F, n, c0, c1, lane);
  } else if (n.kind[0] == kLeaf) inside_row_run<kLeaf, kInternal>(F, n, c0, c1, lane);
  else if (n.kind[1] == kLeaf) inside_row_run<kInternal, kLeaf>(F, n, c0, c1, lane);
  else inside_row_run<kInternal, kInternal>(F, n, c0, c1, lane);
}

// Nodes with at least one fused cherry child (a separate kernel, so that the
// cherry code does not raise the register count of the common case).
__global__ void __launch_bounds__(256) k_inside_rows_ch(DevForest F, int beg, int cnt, int cpw,
                                                         const int32_t* __restrict__ done,
                                                         const int32_t* __restrict__ nodes) {
  const int v = row_node(beg, cnt, nodes);
  if (v < 0) return;
  const int lane = threadIdx.x & 63;
  const int t = F.tree_of[v];
  const int p = F.tree_prob[t];
  const int K = F.tree_nsites[t];
  const int nch = (K + 63) >> 6;
  const int c0 = (int)blockIdx.y * cpw;
  if (c0 >= nch) return;
  if (done && done[p]) return;
  const int c1 = min(c0 + cpw, nch);
  InNode n;
  in_node_load<true>(F, v, t, p, K, n);
  if (n.kind[0] == kCherry) {
    if (n.kind[1] == kCherry) inside_row_run<kCherry, kCherry>(F, n, c0, c1, lane);
    else if (n.kind[1] == kLeaf) inside_row_run<kCherry, kLeaf>(F, n, c0, c1, lane);
    else inside_row_run<kCherry, kInternal>(F, n, c0, c1, lane);
  } else if (n.kind[0] == kLeaf) {
    inside_row_run<kLeaf, kCherry>(F, n, c0, c1, lane);
  } else {
    inside_row_run<kInternal, kCherry>(F, n, c0, c1, lane);
  }
}

// Inside pass along heavy-path chains (row form, one 64-site chunk per
// wavefront): the wavefront walks its chain from the deepest node (whose
// children are both leaves) up to the head, keeping each node's inside
// state in registers for its parent, so only light children's inside rows
// are read.  Every node's inside row is still written (the outside pass
// reads it).  The same operations as the level kernels, the same bits.
struct InCarry {
  int lab, E;
  double b0, bA;
};

// one site of node n whose child HV (0 or 1) is the carried heavy child and
// whose other child has kind KL; HV < 0: both children are leaves
template <int HV, int KL>
__device__ __forceinline__ void chain_in_site(const DevForest& F, const InNode& n, int k, int qo, double qs,
                                              InCarry& c) {
  InSite x;
  x.lv = row_at(n.lab, k);
  x.qo = qo;
  x.qs = qs;
  if (HV == 0) {
    x.la = c.lab;
    x.a0 = c.b0;
    x.aA = c.bA;
    x.Ea = c.E;
    load_child_rows(n.c[1], KL, k, n.phi, F.prior, qo, qs, x.lb, x.b0, x.bA, x.Eb, x.cb, n.stream);
  } else if (HV == 1) {
    load_child_rows(n.c[0], KL, k, n.phi, F.prior, qo, qs, x.la, x.a0, x.aA, x.Ea, x.ca, n.stream);
    x.lb = c.lab;
    x.b0 = c.b0;
    x.bA = c.bA;
    x.Eb = c.E;
  } else {
    load_child_rows(n.c[0], kLeaf, k, n.phi, F.prior, qo, qs, x.la, x.a0, x.aA, x.Ea, x.ca, n.stream);
    load_child_rows(n.c[1], kLeaf, k, n.phi, F.prior, qo, qs, x.lb, x.b0, x.bA, x.Eb, x.cb, n.stream);
  }
  inside_gather(F, x);
  const Eps ea = edge(x.la, x.a0, x.aA, x.Ea, x.qa, n.cf[0]);
  const Eps eb = edge(x.lb, x.b0, x.bA, x.Eb, x.qb, n.cf[1]);
  const double B0 = ea.e0 * eb.e0;
  const double BA = x.lv != 0 ? ea.eA * eb.eA : 0.0;
  const int sh = min(-exp_of(fmax(B0, BA)), 1000);
  const double sc = ldexp(1.0, sh);
  const double2 b = make_double2(B0 * sc, BA * sc);
  if (n.stream)
    store_stream(&row_at(n.beta, k), b);
  else
    row_at(n.beta, k) = b;
  const int E = ea.e + eb.e - sh;
  row_at(n.bE, k) = E;
  c.lab = x.lv;
  c.b0 = b.x;
  c.bA = b.y;
  c.E = E;
}

// Chains [cbeg, cbeg + cnt) of an inside chain order (chain c is
// cnodes[chains[c].x .. chains[c].x + chains[c].y), head first; the walk
// starts at the last node).  Wavefront w runs chain w / max_chunks at chunk
// w % max_chunks; light children's inside rows must be complete.
__global__ void __launch_bounds__(256) k_inside_chain(DevForest F, const int2* __restrict__ chains, int cbeg,
                                                       int cnt, const int32_t* __restrict__ cnodes,
                                                       const int32_t* __restrict__ done) {
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int wv = w / F.max_chunks;
  if (wv >= cnt) return;
  const int2 cd = chains[cbeg + wv];
  const int nb = __builtin_amdgcn_readfirstlane(cd.x);
  const int len = __builtin_amdgcn_readfirstlane(cd.y);
  int prev = -1;
  int v = __builtin_amdgcn_readfirstlane(cnodes[nb + len - 1]);
  const int t = F.tree_of[v];
  const int p = F.tree_prob[t];
  const int K = F.tree_nsites[t];
  const int chunk = w - wv * F.max_chunks;
  if (chunk * 64 >= K) return;
  if (done && done[p]) return;
  const int k = chunk * 64 + (int)(threadIdx.x & 63);
  const bool on = k < K;
  const int sb = F.tree_site_base[t];
  int qo = 0;
  double qs = 0.0;
  if (on) {
    qo = F.site_qoff[sb + k] - 1;
    qs = F.site_qsum[sb + k];
  }
  InCarry c{0, 0, 0.0, 0.0};
  // each step's node record is loaded one step ahead
  NodeRec r = uniform_load(F.nrec + (v - F.num_leaves));
  for (int j = len - 1;; --j) {
    NodeRec rn = r;
    int vn = v;
    if (j > 0) {
      vn = uniform_load(cnodes + nb + j - 1);
      rn = uniform_load(F.nrec + (vn - F.num_leaves));
    }
    InNode n;
    in_node_rec(F, r, n);
    const int hv = prev < 0 ? -1 : (r.ch0 == prev ? 0 : 1);
    if (on) {
      if (hv < 0) {
        chain_in_site<-1, kLeaf>(F, n, k, qo, qs, c);
      } else if (hv == 0) {
        if (n.kind[1] == kLeaf) chain_in_site<0, kLeaf>(F, n, k, qo, qs, c);
        else chain_in_site<0, kInternal>(F, n, k, qo, qs, c);
      } else {
        if (n.kind[0] == kLeaf) chain_in_site<1, kLeaf>(F, n, k, qo, qs, c);
        else chain_in_site<1, kInternal>(F, n, k, qo, qs, c);
      }
    }
    if (j == 0) break;
    prev = v;
    v = vn;
    r = rn;
  }
}

// Inside pass over clades: a wavefront walks a clade's nodes in postorder at
// one 64-site chunk.  The state of the node just done stays in registers, that
// of a finished subtree whose sibling is still to come waits in the
// wavefront's LDS slice (children with the larger need for slots first, so
// two slots suffice for most subtrees of a few dozen leaves).  Rows are only
// written, never read, and nothing is gathered for internal nodes: a node's
// label comes from its children's, and its prior weight is that of the child
// with the same label.  A load waits for all stores before it, so the steps
// make none: the codes of kCladeBatch leaves at a time come with one load into
// the LDS slice, a batch ahead.  The wavefronts of a block share a tree and a
// chunk, whose prior weights (one contiguous piece of the table) they keep in
// LDS: gathered from global memory, every lane of a gather touches another
// cache line, and the L1 caches hold too few of them.  Sixteen trees of 10,000
// leaves x 300 sites: 223 us (4.7 TB/s of rows written and codes read) and 112
// us in the rounds above, where level launches took 653 us; 50,000 x 500: 100
// and 70 us, 351.  Bound by the row stores and the latency of a step's chain
// (LDS reads, then the arithmetic of one node) at six wavefronts a SIMD.  The
// same operations as the level kernels, the same bits.
struct CladeIn {
  int lab, E;
  double b0, bA, q;
};
struct CladeCtx {
  double2* beta;
  int32_t* bE;
  double phi, qs;
  unsigned k;
  bool on, stream;
  const int16_t* code;  // the lane's place in the wavefront's batch of leaf codes
  const double* q;      // q[j]: the site's weight of edit state j (LDS)
};
// prior weight of a label (a leaf's code does as well)
__device__ __forceinline__ double clade_q(const CladeCtx& x, int lab) {
  const double g = x.q[max(lab, 1)];
  return lab > 0 ? g : x.qs;
}
__device__ __forceinline__ CladeIn clade_leaf(const CladeCtx& x, int slot) {
  const int code = x.code[slot * 64];
  CladeIn a;
  leaf_beta(code, x.phi, a.lab, a.b0, a.bA);
  a.E = 0;
  a.q = clade_q(x, code);
  return a;
}
// the node of children a and b
__device__ __forceinline__ CladeIn clade_node(const CladeCtx& x, int64_t ro, const CladeCoef& r, const CladeIn& a,
                                              const CladeIn& b) {
  const Eps ea = edge(a.lab, a.b0, a.bA, a.E, a.q, Coef{r.p1n[0], r.mut[0], r.pn[0], r.msil[0], r.esil[0], 0});
  const Eps eb = edge(b.lab, b.b0, b.bA, b.E, b.q, Coef{r.p1n[1], r.mut[1], r.pn[1], r.msil[1], r.esil[1], 0});
  const int lv = combine_label(a.lab, b.lab);
  const double B0 = ea.e0 * eb.e0;
  const double BA = lv != 0 ? ea.eA * eb.eA : 0.0;
  const int sh = min(-exp_of(fmax(B0, BA)), 1000);
  const double sc = ldexp(1.0, sh);
  CladeIn c;
  c.q = lv > 0 ? (a.lab > 0 ? a.q : b.q) : x.qs;
  c.lab = lv;
  c.b0 = B0 * sc;
  c.bA = BA * sc;
  c.E = ea.e + eb.e - sh;
  if (x.on) {
    const double2 o = make_double2(c.b0, c.bA);
    if (x.stream)
      store_stream(&row_at(x.beta + ro, x.k), o);
    else
      row_at(x.beta + ro, x.k) = o;
    row_at(x.bE + ro, x.k) = c.E;
  }
  return c;
}

// a block: up to kCladeWaves clades of one tree, at one chunk
__global__ void __launch_bounds__(64 * kCladeWaves) k_inside_clade(DevForest F, const int4* __restrict__ blocks,
                                                                   const int4* __restrict__ clades,
                                                                   const CladeStep* __restrict__ steps,
                                                                   const int32_t* __restrict__ leaf_row,
                                                                   int num, const int32_t* __restrict__ done) {
  extern __shared__ __attribute__((aligned(16))) char clade_lds[];
  // the chunks of a block's clades, eight workgroups apart, on one XCD: its
  // L2 cache then serves their step records
  const int g = (int)blockIdx.x >> 3, b = g / F.max_chunks * 8 + ((int)blockIdx.x & 7), chunk = g % F.max_chunks;
  if (b >= num) return;
  const int4 bd = uniform_load(blocks + b);
  const int t = bd.z, k0 = chunk * 64;
  const int K = F.tree_nsites[t], p = F.tree_prob[t];
  if (k0 >= K) return;
  if (done && done[p]) return;
  const int lane = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int sb = F.tree_site_base[t];
  CladeCtx x;
  x.k = (unsigned)(k0 + lane);
  x.on = k0 + lane < K;
  // lanes past the tree's sites run on their rows' pad codes (0) and store
  // nothing
  const unsigned ks = (unsigned)min(k0 + lane, K - 1);
  x.qs = row_at(F.site_qsum + sb, ks);
  {
    double* q = (double*)(clade_lds + kCladeWaves * kCladeLds);
    const int q0 = uniform_load(F.site_qoff + sb + k0), q1 = uniform_load(F.site_qoff + sb + min(k0 + 64, K));
    for (int i = (int)threadIdx.x; i < q1 - q0; i += 64 * kCladeWaves) q[i] = F.prior[q0 + i];
    // (a site without edit states reads q[1] all the same: the piece has a
    // spare entry)
    x.q = q + (row_at(F.site_qoff + sb, ks) - 1 - q0);
    __syncthreads();
  }
  if (wave >= bd.y) return;
  const int4 cd = uniform_load(clades + bd.x + wave);
  x.phi = uniform_load(F.phi + p);
  x.beta = F.beta;
  x.bE = F.bE;
  x.stream = F.stream_rows != 0;
  char* slice = clade_lds + wave * kCladeLds;
  char* batch = slice + kCladeSlots * kCladeSlotBytes;
  x.code = (const int16_t*)batch + lane;
  // a batch: eight lanes a leaf, eight sites a lane
  const int32_t* lr = leaf_row + cd.z * kCladeBatch + (lane >> 3);
  const int16_t* codes = F.codes + k0 + (lane & 7) * 8;
  int nb = 1;
  uint4 w = *(const uint4*)(codes + (int64_t)lr[0] * 64);
  int row = lr[min(1, cd.w - 1) * kCladeBatch];
  const CladeStep* st = steps + cd.x;
  const CladeCoef* sc = F.clade_coef + cd.x;
  CladeStep r = uniform_load(st);
  CladeCoef cf = uniform_load(sc);
  CladeIn c{0, 0, 0.0, 0.0, 0.0};
  for (int j = 1;; ++j) {
    if (r.flags & 128) {
      *(uint4*)(batch + lane * 16) = w;
      lds_wave_sync();
      w = *(const uint4*)(codes + (int64_t)row * 64);
      nb = min(nb + 1, cd.w - 1);
      row = lr[nb * kCladeBatch];
    }
    const int kind = r.flags & 3;
    CladeIn b;
    if (kind == 2) {
      const char* l = slice + ((r.flags >> 2) & 3) * kCladeSlotBytes;
      const double2 u = *(const double2*)(l + lane * 16);
      const int2 v = *(const int2*)(l + 1024 + lane * 8);
      b = CladeIn{v.y, v.x, u.x, u.y, clade_q(x, v.y)};
    } else {
      b = clade_leaf(x, (r.flags >> 11) & 7);
      if (kind == 0) c = clade_leaf(x, (r.flags >> 8) & 7);
    }
    // the next step's record, once the operands are there: LDS and scalar
    // loads share a counter
    int jn = min(j, cd.y - 1);
    asm volatile("" : "+s"(jn) : "v"(b.q), "v"(c.q));
    const CladeStep rn = uniform_load(st + jn);
    const CladeCoef cn = uniform_load(sc + jn);
    c = clade_node(x, (int64_t)r.row * 64, cf, c, b);
    if (j == cd.y) break;
    const int push = (r.flags >> 4) & 7;
    if (push) {
      char* l = slice + (push - 1) * kCladeSlotBytes;
      *(double2*)(l + lane * 16) = make_double2(c.b0, c.bA);
      *(int2*)(l + 1024 + lane * 8) = make_int2(c.E, c.lab);
    }
    r = rn;
    cf = cn;
  }
}

// Inside pass over the top levels [h0, h1): one block per site chunk walks
// the levels in order (its segments share each level's nodes), so the small
// upper levels cost one launch instead of one each.
template <int W>
__global__ void __launch_bounds__(1024) k_inside_top(DevForest F, int h0, int h1, const int32_t* __restrict__ done) {
  const int segs = 1024 / W;
  const int seg = threadIdx.x / W;
  const int k = (int)blockIdx.x * W + (int)(threadIdx.x & (W - 1));
  for (int h = h0; h < h1; ++h) {
    const int e = F.level_off[h + 1];
    for (int v = F.level_off[h] + seg; v < e; v += segs) inside_node(F, v, k, done);
    __syncthreads();
  }
}

// Root of tree t at the sites of one chunk: site likelihood L = P(D | stem
// starts unedited), the outside state at the root, and the root branch's
// posterior counts (partial number `chunk`).  All W lanes of the segment call
// this together.
template <int W>
__device__ __forceinline__ void root_chunk(const DevForest& F, int t, int chunk, int lane,
                                           double* __restrict__ site_llh_out) {
  const int p = F.tree_prob[t];
  const int K = F.tree_nsites[t];
  const int k = chunk * W + lane;
  const int r = F.tree_root[t];
  const bool act = k < K;
  double acc0 = 0, acc1 = 0, acc2 = 0;
  if (act) {
    const int sb = F.tree_site_base[t];
    const Coef cf = F.coef[r];
    const double phi = F.phi[p];
    const bool leaf = r < F.num_leaves;
    const int64_t rr = F.row_off[r];
    int lab, E, code;
    double b0, bA;
    load_child(F, r, leaf, k, phi, lab, b0, bA, E, code);
    const int qo = F.site_qoff[sb + k] - 1;
    const double q = lab > 0 ? F.prior[qo + lab] : F.site_qsum[sb + k];
    const Eps er = edge(lab, b0, bA, E, q, cf);
    const int ex = exp_of(er.e0);
    const double Lm = ldexp(er.e0, -ex);
    const int LE = er.e + ex;
    const double sl = log(Lm) + (double)LE * 0.69314718055994530942;
    F.site_llh[sb + k] = sl;
    if (site_llh_out) site_llh_out[sb + k] = sl;
    // the stem starts unedited: given the data, its top is unedited with
    // probability 1, as below a node with label 'z'
    const double A = 1.0 / er.e0;
    const double a0 = cf.p1n * A * er.s0;
    const double m = cf.mut * q * A * er.s0;
    const double sil = lab < 0 ? er.s1 * A : 0.0;
    if (!leaf) {
      F.alpha[rr + k] = make_double2(a0, m);
      if (lab < 0) F.pS[rr + k] = sil;
    }
    acc0 = lab == 0 ? 1.0 : a0 * b0;
    if (lab != 0) acc1 = m * bA;
    acc2 = sil;
  }
  acc0 = seg_sum_last<W>(acc0);
  acc1 = seg_sum_last<W>(acc1);
  acc2 = seg_sum_last<W>(acc2);
  if (lane == W - 1) {
    double* c = F.cpart + ((int64_t)r * F.max_chunks + chunk) * 5;
    c[0] = acc0;
    c[1] = acc1;
    c[2] = acc2;
    c[3] = 0.0;
    c[4] = 0.0;
  }
}

// Root step of every tree (segments index trees, blockIdx.y the site chunk).
template <int W>
__global__ void __launch_bounds__(256) k_root(DevForest F, double* __restrict__ site_llh_out,
                                              const int32_t* __restrict__ done) {
  Seg<W> g;
  if (!g.init(0, F.num_trees)) return;
  const int t = g.v;
  if ((int)blockIdx.y * W >= F.tree_nsites[t]) return;
  if (done && done[F.tree_prob[t]]) return;
  root_chunk<W>(F, t, (int)blockIdx.y, g.lane, site_llh_out);
}

// Outside pass for the children of the internal nodes of one level, with the
// posterior expected transition counts of both child branches and the
// dropout responsibilities of missing leaf children.

// per-node values of the outside pass (uniform over the sites of the node)
struct OutNode {
  int K;
  int ch[2];
  int kind[2];
  Coef cf[2];
  ChildRows c[2];
  double2* ca[2];        // children's outside rows (internal children)
  double* cS[2];         // children's silenced posteriors (internal children)
  const int16_t* lab;    // the node's labels
  const double2* a;      // the node's outside row
  const double* aS;      // the node's silenced posteriors ('?' sites)
  const int32_t* qoff;
  const double* qsum;
  double phi;
  bool stream;           // rows with the non-temporal hint
};

template <bool CH>
__device__ __forceinline__ void out_node_load(const DevForest& F, int u, int t, int p, int K, OutNode& n) {
  n.K = K;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = i == 0 ? F.child0[u] : F.child1[u];
    n.ch[i] = c;
    n.kind[i] = CH ? child_kind(F, c) : (c < F.num_leaves ? kLeaf : kInternal);
    n.cf[i] = F.coef[c];
    n.c[i] = child_rows(F, c, n.kind[i]);
    const int64_t rc = F.row_off[c];
    n.ca[i] = F.alpha + rc;
    n.cS[i] = F.pS + rc;
  }
  const int64_t ru = F.row_off[u];
  n.lab = F.labels + ru;
  n.a = F.alpha + ru;
  n.aS = F.pS + ru;
  const int sb = F.tree_site_base[t];
  n.qoff = F.site_qoff + sb;
  n.qsum = F.site_qsum + sb;
  n.phi = F.phi[p];
  n.stream = F.stream_rows != 0;
}

// The outside-pass values of internal node u from its record (children that
// are leaves or stored internal nodes).
__device__ __forceinline__ void out_node_rec(const DevForest& F, const NodeRec& r, OutNode& n) {
  n.K = r.K;
  const int ch[2] = {r.ch0, r.ch1};
  const int64_t ro[2] = {r.ro0, r.ro1}, bro[2] = {r.bro0, r.bro1};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    n.ch[i] = ch[i];
    n.kind[i] = ch[i] < F.num_leaves ? kLeaf : kInternal;
    n.cf[i] = uniform_load(F.coef + ch[i]);
    n.c[i].code = (n.kind[i] == kLeaf ? F.codes : F.labels) + ro[i];
    n.c[i].beta = F.beta + bro[i];
    n.c[i].bE = F.bE + bro[i];
    n.c[i].code2 = nullptr;
    n.c[i].gc[0] = n.c[i].gc[1] = -1;
    n.ca[i] = F.alpha + ro[i];
    n.cS[i] = F.pS + ro[i];
  }
  n.lab = F.labels + r.ro;
  n.a = F.alpha + r.ro;
  n.aS = F.pS + r.ro;
  n.qoff = F.site_qoff + r.sb;
  n.qsum = F.site_qsum + r.sb;
  n.phi = uniform_load(F.phi + r.p);
  n.stream = F.stream_rows != 0;
}

// The posterior step of one node u at one site.
//
// Outside states are kept conditional on all the data and on the scale of the
// node's own inside vector: with beta_u = (b0, bA) 2^E and the site
// likelihood L, u's state is
//   a0 = alpha_u(0) 2^E / L,  aX = sum over the edit states a that the data
//   below u allow (the label's state, or any state of a '?' node) of
//   alpha_u(a) 2^E / L,
// so a0 b0 = P(u unedited | D) and aX bA = P(u edited | D) and no exponent or
// site likelihood is carried.  Two facts make the pair enough.  The posterior
// counts and the states below need no other part of alpha_u (its silenced
// part enters only P(u silenced | D), kept beside where '?' nodes need it).
// And a node with label 'z' is unedited given the data below it: a0 = 1 / b0
// and aX = 0 whatever lies outside, so its row is not read (and may hold
// anything).
// Range: the scale sc of u's vector goes to the siblings' edge values and not
// to the state, since 1 / B0 alone leaves a double's range where two unedited
// children hang on branches of 300 or more.  a0 is at most 1 / b0, so it stays
// finite while a node's unedited value is within 1e-308 of its edited one; the
// ratio is at least (edit probability x prior weight) ^ 2 of one branch, 0
// below that (then a0 counts for nothing).
// A row is 16 bytes where the unconditional state (three more values, an
// exponent and a specific state) took 38, and a step needs about half the
// arithmetic: on 16 trees of 10,000 leaves x 300 sites the chain rounds below
// level 10 went from 0.66 to 0.52 ms a pass (114 -> 87 VGPRs, 5 wavefronts a
// SIMD), an EM step from 1.79 to 1.61 ms.
//
// In: u's label lu and state (a0, aX), silenced posterior pSu (read where
// lu < 0), and for both children their label, inside mantissas, prior weight
// q (the site's prior mass for '?'), edge values ep, branch coefficients and
// leaf code.  Out: the children's states ca, silenced posteriors cS (kS), the
// counts S of both child branches, and the dropout responsibility rt of
// missing leaf children.
struct PostOut {
  double a0[2], aX[2], pS[2];
  double S[2][5];
  double rt;
};
template <bool kS>
__device__ __forceinline__ void cond_post(int lu, double a0, double aX, double pSu, double phi, const int (&lab)[2],
                                          const double (&b0)[2], const double (&bA)[2], const double (&q)[2],
                                          const Eps (&ep)[2], const Coef (&cfs)[2], const bool (&lf)[2],
                                          const int (&code)[2], PostOut& o) {
  // every pass kernel gives the same bits: fused operations are written out
#pragma clang fp contract(off)
  const bool z = lu == 0;
  const double B0 = ep[0].e0 * ep[1].e0;
  const double BA = z ? 0.0 : ep[0].eA * ep[1].eA;
  // the power of two that the inside pass scaled u's vector by
  const double sc = ldexp(1.0, min(-exp_of(fmax(B0, BA)), 1000));
  const double f0 = z ? rcp_normal(B0 * sc) : a0;
  const double fX = z ? 0.0 : aX;
  o.rt = 0.0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int w = 1 - i;
    const Coef& cf = cfs[i];
    // A, G: the data outside the child's branch joint with u unedited / in
    // an allowed edit state, over L and on the child's edge exponent
    const double A = f0 * (ep[w].e0 * sc);
    const double G = fX * (ep[w].eA * sc);
    const double As = A * ep[i].s0, Gs = G * ep[i].s0;
    const double m = cf.mut * q[i] * As;
    const double pg = cf.pn * Gs;
    o.a0[i] = cf.p1n * As;
    o.aX[i] = fma(cf.pn, Gs, m);
    const bool cz = lab[i] == 0;
    o.S[i][0] = cz ? 1.0 : o.a0[i] * b0[i];
    o.S[i][1] = m * bA[i];  // bA = 0 at 'z' nodes, s1 = 0 but at '?' nodes
    o.S[i][2] = ep[i].s1 * A;
    o.S[i][3] = pg * bA[i];
    o.S[i][4] = ep[i].s1 * G;
    if (kS) o.pS[i] = o.S[i][2] + o.S[i][4] + (lu < 0 ? pSu : 0.0);
    if (lf[i]) o.rt = fma(code[i] == -1 ? phi : 0.0, o.a0[i] + o.aX[i], o.rt);
  }
}

// The posterior step a fused cherry's own node would run at site k, from the
// state (a0, aX) its parent just formed and its label: counts of its two leaf
// branches into cacc, dropout responsibility of its missing leaves into crt.
__device__ __forceinline__ void cherry_post(const DevForest& F, const ChildRows& r, int k, int lu, double a0,
                                            double aX, int qo, double qs, double phi, double (&cacc)[2][5],
                                            double& crt) {
  int lab[2], code[2];
  double b0[2], bA[2], q[2];
  Eps ep[2];
  code[0] = row_at(r.code, k);
  code[1] = row_at(r.code2, k);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    leaf_beta(code[j], phi, lab[j], b0[j], bA[j]);
    q[j] = lab[j] > 0 ? row_at(F.prior, (unsigned)(qo + lab[j])) : qs;
    ep[j] = edge(lab[j], b0[j], bA[j], 0, q[j], r.g[j]);
  }
  const bool lf[2] = {true, true};
  PostOut o;
  cond_post<false>(lu, a0, aX, 0.0, phi, lab, b0, bA, q, ep, r.g, lf, code, o);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int m = 0; m < 5; ++m) cacc[j][m] += o.S[j][m];
  crt += o.rt;
}

// The outside step of one site in three phases: row loads, prior gathers,
// then arithmetic and stores.
struct OutSite {
  double2 au;
  double pS;
  int lu, qo;
  double qs;
  int lab[2], E[2], code[2];
  double b0[2], bA[2], q[2];
};

// the children's rows at site k (x.qo, x.qs already loaded)
template <int K0, int K1>
__device__ __forceinline__ void outside_load_children(const DevForest& F, const OutNode& n, int k, OutSite& x) {
  const int kind[2] = {resolve_kind<K0>(n.kind[0]), resolve_kind<K1>(n.kind[1])};
#pragma unroll
  for (int i = 0; i < 2; ++i)
    load_child_rows(n.c[i], kind[i], k, n.phi, F.prior, x.qo, x.qs, x.lab[i], x.b0[i], x.bA[i], x.E[i], x.code[i]);
}

template <int K0, int K1>
__device__ __forceinline__ void outside_load(const DevForest& F, const OutNode& n, int k, OutSite& x) {
  x.au = row_at(n.a, k);
  x.lu = row_at(n.lab, k);
  x.pS = 0.0;
  if (x.lu < 0) x.pS = row_at(n.aS, k);
  x.qo = row_at(n.qoff, k) - 1;
  x.qs = row_at(n.qsum, k);
  outside_load_children<K0, K1>(F, n, k, x);
}

__device__ __forceinline__ void outside_gather(const DevForest& F, OutSite& x) {
#pragma unroll
  for (int i = 0; i < 2; ++i) x.q[i] = x.lab[i] > 0 ? row_at(F.prior, (unsigned)(x.qo + x.lab[i])) : x.qs;
}

// One site k of node n: the children's outside states and the posterior
// counts of both child branches, added to acc; the dropout responsibility of
// missing leaf children added to rt.  A fused cherry child's outside state is
// not stored: the cherry's own posterior step runs here, into cacc[i] and
// crt[i].  K0 / K1: the kind of each child, or kNoCherry to read n.kind.
template <int K0, int K1>
__device__ __forceinline__ void outside_finish(const DevForest& F, const OutNode& n, int k, const OutSite& x,
                                               double (&acc)[2][5], double& rt, double (&cacc)[2][2][5],
                                               double (&crt)[2]) {
  const int kind[2] = {resolve_kind<K0>(n.kind[0]), resolve_kind<K1>(n.kind[1])};
  const bool lf[2] = {kind[0] == kLeaf, kind[1] == kLeaf};
  Eps ep[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) ep[i] = edge(x.lab[i], x.b0[i], x.bA[i], x.E[i], x.q[i], n.cf[i]);
  PostOut o;
  cond_post<true>(x.lu, x.au.x, x.au.y, x.pS, n.phi, x.lab, x.b0, x.bA, x.q, ep, n.cf, lf, x.code, o);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int m = 0; m < 5; ++m) acc[i][m] += o.S[i][m];
    if (kind[i] == kCherry) {
      cherry_post(F, n.c[i], k, x.lab[i], o.a0[i], o.aX[i], x.qo, x.qs, n.phi, cacc[i], crt[i]);
    } else if (kind[i] != kLeaf) {
      const double2 a = make_double2(o.a0[i], o.aX[i]);
      if (n.stream)
        store_stream(&row_at(n.ca[i], k), a);
      else
        row_at(n.ca[i], k) = a;
      if (x.lab[i] < 0) row_at(n.cS[i], k) = o.pS[i];
    }
  }
  rt += o.rt;
}

template <int K0, int K1>
__device__ __forceinline__ void outside_site(const DevForest& F, const OutNode& n, int k, double (&acc)[2][5],
                                             double& rt, double (&cacc)[2][2][5], double (&crt)[2]) {
  OutSite x;
  outside_load<K0, K1>(F, n, k, x);
  outside_gather(F, x);
  outside_finish<K0, K1>(F, n, k, x, acc, rt, cacc, crt);
}
// the same with the children's prior weights read from their prior-weight
// rows q0, q1, for nodes without fused cherry children
__device__ __forceinline__ void outside_site_q(const DevForest& F, const OutNode& n, int k, double (&acc)[2][5],
                                               double& rt, const double* q0, const double* q1) {
  double cacc[2][2][5];
  double crt[2];
  OutSite x;
  outside_load<kNoCherry, kNoCherry>(F, n, k, x);
  x.q[0] = row_at(q0, k);
  x.q[1] = row_at(q1, k);
  outside_finish<kNoCherry, kNoCherry>(F, n, k, x, acc, rt, cacc, crt);
}

// outside_site for kernels that never meet a fused cherry
template <int K0, int K1>
__device__ __forceinline__ void outside_site(const DevForest& F, const OutNode& n, int k, double (&acc)[2][5],
                                             double& rt) {
  double cacc[2][2][5];
  double crt[2];
  outside_site<K0, K1>(F, n, k, acc, rt, cacc, crt);
}

// segment sums of a fused cherry's leaf-branch counts and dropout sum for one
// chunk; the last lane of the segment writes them as partial number `slot`
// of the leaf branches and of the cherry.  All lanes of the segment call this.
template <int W>
__device__ __forceinline__ void cherry_write_partials(const DevForest& F, int c, const ChildRows& r, int lane,
                                                      int slot, double (&cacc)[2][5], double crt) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int m = 0; m < 5; ++m) cacc[j][m] = seg_sum_last<W>(cacc[j][m]);
  crt = seg_sum_last<W>(crt);
  if (lane == W - 1) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      double* o = F.cpart + ((int64_t)r.gc[j] * F.max_chunks + slot) * 5;
#pragma unroll
      for (int m = 0; m < 5; ++m) o[m] = cacc[j][m];
    }
    F.rt_part[(int64_t)c * F.max_chunks + slot] = crt;
  }
}

// segment sums of the partial counts; they are written as partial number
// `slot` of each child branch (and of the node's dropout sum), and partials
// slot+1 .. slot_end-1 are cleared.  64-lane segments: one butterfly sum of
// all eleven values, each total stored by one lane, the clearing by
// coalesced vector stores; narrower segments: DPP segment sums, stored by
// the segment's last lane.
template <int W>
__device__ __forceinline__ void out_write_partials(const DevForest& F, int u, const int (&ch)[2], int lane, int slot,
                                                   int slot_end, double (&acc)[2][5], double rt) {
  if constexpr (W == 64) {
    double v[12];
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      v[j] = acc[0][j];
      v[5 + j] = acc[1][j];
    }
    v[10] = rt;
    v[11] = 0.0;
    const double x = wave_sum12(v);
    // totals 0..4: counts of child 0, 5..9: of child 1, 10: the dropout sum
    const int vi = sum12_value(lane);
    if (vi >= 0 && vi < 10) {
      const int i = vi >= 5 ? 1 : 0;
      F.cpart[((int64_t)ch[i] * F.max_chunks + slot) * 5 + (vi - 5 * i)] = x;
    } else if (vi == 10) {
      F.rt_part[(int64_t)u * F.max_chunks + slot] = x;
    }
    const int nz = slot_end - slot - 1;
    if (nz > 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        double* c = F.cpart + ((int64_t)ch[i] * F.max_chunks + slot + 1) * 5;
        for (int b = lane; b < 5 * nz; b += 64) c[b] = 0.0;
      }
      for (int b = lane; b < nz; b += 64) F.rt_part[(int64_t)u * F.max_chunks + slot + 1 + b] = 0.0;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 5; ++j) acc[i][j] = seg_sum_last<W>(acc[i][j]);
  rt = seg_sum_last<W>(rt);
  if (lane == W - 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      double* c = F.cpart + ((int64_t)ch[i] * F.max_chunks + slot) * 5;
#pragma unroll
      for (int j = 0; j < 5; ++j) c[j] = acc[i][j];
      for (int s2 = slot + 1; s2 < slot_end; ++s2)
#pragma unroll
        for (int j = 0; j < 5; ++j) F.cpart[((int64_t)ch[i] * F.max_chunks + s2) * 5 + j] = 0.0;
    }
    F.rt_part[(int64_t)u * F.max_chunks + slot] = rt;
    for (int s2 = slot + 1; s2 < slot_end; ++s2) F.rt_part[(int64_t)u * F.max_chunks + s2] = 0.0;
  }
}

__device__ __forceinline__ void zero_acc(double (&acc)[2][5]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 5; ++j) acc[i][j] = 0.0;
}

// Segment form: the W lanes of a segment handle sites chunk*W + lane of node
// u (all lanes of the segment call this together).
template <int W>
__device__ __forceinline__ void outside_node(const DevForest& F, int u, int chunk, int lane,
                                             const int32_t* __restrict__ done) {
  const int k = chunk * W + lane;
  const NodeRec r = F.nrec[u - F.num_leaves];
  const int K = r.K;
  if (chunk * W >= K) return;
  if (done && done[r.p]) return;
  OutNode n;
  out_node_rec(F, r, n);
  double acc[2][5];
  zero_acc(acc);
  double rt = 0.0;
  if (k < K) outside_site<kNoCherry, kNoCherry>(F, n, k, acc, rt);
  out_write_partials<W>(F, u, n.ch, lane, chunk, chunk + 1, acc, rt);
}

// Row form (K > 32): one wavefront per node, so the node number is
// wave-uniform (its metadata are scalar loads and the child-kind tests
// scalar branches); the wave walks chunks [c0, c0 + cpw) of 64 sites,
// accumulating per lane, and reduces once.  The leaf-branch counts of a
// fused cherry child are reduced and written per chunk.
template <int K0, int K1>
__device__ __forceinline__ void outside_row_run(const DevForest& F, int u, const OutNode& n, int c0, int c1,
                                                int lane) {
  double acc[2][5];
  zero_acc(acc);
  double rt = 0.0;
  for (int c = c0; c < c1; ++c) {
    const int k = c * 64 + lane;
    double cacc[2][2][5];
    double crt[2] = {0.0, 0.0};
    if (K0 == kCherry) zero_acc(cacc[0]);
    if (K1 == kCherry) zero_acc(cacc[1]);
    if (k < n.K) outside_site<K0, K1>(F, n, k, acc, rt, cacc, crt);
    if (K0 == kCherry) cherry_write_partials<64>(F, n.ch[0], n.c[0], lane, c, cacc[0], crt[0]);
    if (K1 == kCherry) cherry_write_partials<64>(F, n.ch[1], n.c[1], lane, c, cacc[1], crt[1]);
  }
  out_write_partials<64>(F, u, n.ch, lane, c0, c1, acc, rt);
}

// Nodes whose children are leaves or stored internal nodes.
__global__ void __launch_bounds__(256) k_outside_rows(DevForest F, int beg, int cnt, int cpw,
                                                       const int32_t* __restrict__ done,
                                                       const int32_t* __restrict__ nodes) {
  const int u = row_node(beg, cnt, nodes);
  if (u < 0) return;
  const int lane = threadIdx.x & 63;
  const NodeRec r = F.nrec[u - F.num_leaves];
  const int nch = (r.K + 63) >> 6;
  const int c0 = (int)blockIdx.y * cpw;
  if (c0 >= nch) return;
  if (done && done[r.p]) return;
  const int c1 = min(c0 + cpw, nch);
  OutNode n;
  out_node_rec(F, r, n);
  if (n.kind[0] == kLeaf) {
    if (n.kind[1] == kLeaf) outside_row_run<kLeaf, kLeaf>(F, u, n, c0, c1, lane);
    else outside_row_run<kLeaf, kInternal>(F, u, n, c0, c1, lane);
  } else {
    if (n.kind[1] == kLeaf) outside_row_run<kInternal, kLeaf>(F, u, n, c0, c1, lane);
    else outside_row_run<kInternal, kInternal>(F, u, n, c0, c1, lane);
  }
}

// Nodes with at least one fused cherry child.
__global__ void __launch_bounds__(256) k_outside_rows_ch(DevForest F, int beg, int cnt, int cpw,
                                                          const int32_t* __restrict__ done,
                                                          const int32_t* __restrict__ nodes) {
  const int u = row_node(beg, cnt, nodes);
  if (u < 0) return;
  const int lane = threadIdx.x & 63;
  const int t = F.tree_of[u];
  const int p = F.tree_prob[t];
  const int K = F.tree_nsites[t];
  const int nch = (K + 63) >> 6;
  const int c0 = (int)blockIdx.y * cpw;
  if (c0 >= nch) return;
  if (done && done[p]) return;
  const int c1 = min(c0 + cpw, nch);
  OutNode n;
  out_node_load<true>(F, u, t, p, K, n);
  if (n.kind[0] == kCherry) {
    if (n.kind[1] == kCherry) outside_row_run<kCherry, kCherry>(F, u, n, c0, c1, lane);
    else if (n.kind[1] == kLeaf) outside_row_run<kCherry, kLeaf>(F, u, n, c0, c1, lane);
    else outside_row_run<kCherry, kInternal>(F, u, n, c0, c1, lane);
  } else if (n.kind[0] == kLeaf) {
    outside_row_run<kLeaf, kCherry>(F, u, n, c0, c1, lane);
  } else {
    outside_row_run<kInternal, kCherry>(F, u, n, c0, c1, lane);
  }
}

// Outside pass along heavy-path chains (row form, one 64-site chunk per
// wavefront).  A chain is a node followed by its successive heavy children
// (each the child with the larger subtree among the internal ones).  The
// wavefront runs the posterior step of every node of its chain from the top,
// keeping the heavy child's outside state in registers as the next node's
// own: only light children's outside rows are written and only the head's
// is read, which removes most of the outside-row traffic of the level
// passes.  The site's likelihood and prior values are read once per chain.
// Partial counts go to the chunk's slot as in the level kernels with one
// chunk per wavefront, so the results are the same bits.
//
// The steps are software-pipelined so that each waits for memory once, on
// operations issued a whole step earlier.  The inside rows, branch
// coefficients, prior-weight rows and codes of step j + 1 are copied to the
// wavefront's slice of LDS during step j by direct global-to-LDS loads,
// which occupy no registers in flight.  At the top of step j every
// outstanding access completes, step j's operands are read from LDS and the
// step records from the scalar cache, and the next copies are issued; step
// j itself runs on registers.
// No register written by a memory load is carried from one step to the
// next, so the compiler never waits for one mid-step.  The vector memory
// counter counts loads and stores together, so the partial counts of step j
// are stored at the top of step j + 1, after its wait.

// the codes (leaf) or az-partition labels (internal) of child c at row ro
__device__ __forceinline__ const int16_t* chain_code_row(const DevForest& F, int c, int64_t ro) {
  return (c < F.num_leaves ? F.codes : F.labels) + ro;
}
__device__ __forceinline__ const double* chain_q_row(const DevForest& F, int c, int64_t ro) {
  return (c < F.num_leaves ? F.qleaf : F.qint) + ro;
}

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void glb_void;

// One wavefront's LDS slice: the next step's inside rows of both children,
// both children's prior weights, both children's branch coefficients (10
// words each), both children's codes (the aligned 32-bit word holding each
// lane's 16-bit code), and in a pack the next head's outside state and labels.
constexpr int kChainLdsBeta = 0;       // [2][64] double2
constexpr int kChainLdsBE = 2048;      // [2][64] int32
constexpr int kChainLdsQ = 2560;       // [2][64] double
constexpr int kChainLdsCoef = 3584;    // [64] uint32 (20 used)
constexpr int kChainLdsCode = 3840;    // [2][64] uint32
constexpr int kChainLdsHeadA = 4352;   // [64] double2: a head's outside state
constexpr int kChainLdsHeadL = 5376;   // [64] uint32: the word holding its label
constexpr int kChainLdsBytes = 5632;

// copy `size` (4 or 16) bytes at src (per lane) to dst + size * lane; rows
// read once per pass carry the non-temporal hint, so that the per-site
// tables and priors every chain of a tree reads stay in the L2 cache
__device__ __forceinline__ void to_lds(const void* src, char* dst, unsigned size, bool stream = false) {
  if (size == 16) {
    if (stream)
      __builtin_amdgcn_global_load_lds((glb_void*)src, (lds_void*)dst, 16, 0, 2);
    else
      __builtin_amdgcn_global_load_lds((glb_void*)src, (lds_void*)dst, 16, 0, 0);
  } else {
    if (stream)
      __builtin_amdgcn_global_load_lds((glb_void*)src, (lds_void*)dst, 4, 0, 2);
    else
      __builtin_amdgcn_global_load_lds((glb_void*)src, (lds_void*)dst, 4, 0, 0);
  }
}
template <typename T>
__device__ __forceinline__ T lds_at(const char* base, unsigned byte_off) {
  return *(const __attribute__((address_space(3))) T*)(base + byte_off);
}
template <>
__device__ __forceinline__ double2 lds_at<double2>(const char* base, unsigned byte_off) {
  const nt_double2 v = *(const __attribute__((address_space(3))) nt_double2*)(base + byte_off);
  return make_double2(v.x, v.y);
}

// a wave-uniform double in scalar registers
__device__ __forceinline__ double uniform_double(double x) {
  const int lo = __builtin_amdgcn_readfirstlane(__double2loint(x));
  const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(x));
  return __hiloint2double(hi, lo);
}

// every memory access issued so far has completed; nothing is moved across
__device__ __forceinline__ void chain_wait_all() {
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_sched_barrier(0);
}
// every LDS read and scalar load issued so far has completed
__device__ __forceinline__ void chain_wait_lgkm() {
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_sched_barrier(0);
}

// the 16-bit code at site kk of a row, from the aligned word that holds it
__device__ __forceinline__ int code_of_word(uint32_t wd, unsigned kk) {
  return (int)(int16_t)(kk & 1u ? wd >> 16 : wd & 0xffffu);
}

// Copy step r's codes.
__device__ __forceinline__ void chain_stage_codes(const DevForest& F, const ChainStep& r, unsigned kk, char* lds) {
  const int16_t* row0 = chain_code_row(F, r.ch0, r.ro0) + (kk & ~1u);
  const int16_t* row1 = chain_code_row(F, r.ch1, r.ro1) + (kk & ~1u);
  to_lds(row0, lds + kChainLdsCode, 4, true);
  to_lds(row1, lds + kChainLdsCode + 256, 4, true);
}

// Copy step r's operands: branch coefficients of both children, inside rows
// of internal children, and both children's prior-weight rows over the
// chunk's 64 sites (k0 .. k0 + 63, inside the padded rows; 16 bytes by each
// of the first 32 lanes).
__device__ __forceinline__ void chain_stage(const DevForest& F, const ChainStep& r, unsigned k0, unsigned kk,
                                            int lane, char* lds) {
  {
    const int c = lane < 10 ? r.ch0 : r.ch1;
    const int wd = lane < 10 ? lane : min(lane - 10, 9);
    to_lds(reinterpret_cast<const uint32_t*>(F.coef + c) + wd, lds + kChainLdsCoef, 4);
  }
  const int ch[2] = {r.ch0, r.ch1};
  const int64_t ro[2] = {r.ro0, r.ro1};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool leaf = ch[i] < F.num_leaves;
    if (!leaf) {
      to_lds(&row_at(F.beta + ro[i], kk), lds + kChainLdsBeta + 1024 * i, 16, true);
      to_lds(&row_at(F.bE + ro[i], kk), lds + kChainLdsBE + 256 * i, 4, true);
    }
    if (lane < 32) to_lds(chain_q_row(F, ch[i], ro[i]) + k0 + 2 * lane, lds + kChainLdsQ + 512 * i, 16, true);
  }
}

// Copy the stored outside state and the labels of the node whose rows start
// at ru: the head of the next chain of a pack.
__device__ __forceinline__ void chain_stage_head(const DevForest& F, int64_t ru, unsigned kk, char* lds) {
  to_lds(&row_at(F.alpha + ru, kk), lds + kChainLdsHeadA, 16, true);
  to_lds(F.labels + ru + (kk & ~1u), lds + kChainLdsHeadL, 4, true);
}

// One chain step at one site, on registers: the children's raw row values
// (leaf codes or labels), prior weights, inside rows (ignored for leaves)
// and branch coefficients.  The heavy child's outside state and label replace
// (a0, aX, lu); the light internal child's state is stored at row ro[light].
template <int K0, int K1, typename Stage>
__device__ __forceinline__ void chain_compute(const DevForest& F, const char* lds, int lane, const Coef (&cf)[2],
                                              double phi, int hv, const int (&raw)[2], const int64_t (&ro)[2],
                                              unsigned kk, bool on, bool stream, Stage&& stage, double& a0,
                                              double& aX, int& lu, PostOut& o) {
  const bool lf[2] = {K0 == kLeaf, K1 == kLeaf};
  int lab[2], E[2], code[2];
  double b0[2], bA[2], q[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    q[i] = lds_at<double>(lds, kChainLdsQ + 512 * i + 8 * lane);
    if (lf[i]) {
      code[i] = raw[i];
      leaf_beta(raw[i], phi, lab[i], b0[i], bA[i]);
      E[i] = 0;
    } else {
      code[i] = 0;
      lab[i] = raw[i];
      const double2 bb = lds_at<double2>(lds, kChainLdsBeta + 1024 * i + 16 * lane);
      b0[i] = bb.x;
      bA[i] = bb.y;
      E[i] = lds_at<int>(lds, kChainLdsBE + 256 * i + 4 * lane);
    }
  }
  // the slice is read: the next step's copies may overwrite it
  chain_wait_lgkm();
  stage();
  Eps ep[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) ep[i] = edge(lab[i], b0[i], bA[i], E[i], q[i], cf[i]);
  cond_post<false>(lu, a0, aX, 0.0, phi, lab, b0, bA, q, ep, cf, lf, code, o);
  if (!on) {
    // lanes past the tree's sites add nothing to the counts
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int m = 0; m < 5; ++m) o.S[i][m] = 0.0;
    o.rt = 0.0;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (lf[i]) continue;
    if (i == hv) {
      a0 = o.a0[i];
      aX = o.aX[i];
      lu = lab[i];
    } else if (on) {
      const double2 a = make_double2(o.a0[i], o.aX[i]);
      if (stream)
        store_stream(&row_at(F.alpha + ro[i], kk), a);
      else
        row_at(F.alpha + ro[i], kk) = a;
    }
  }
}

// Packs [cbeg, cbeg + cnt) of a chain plan: pack c's steps are
// steps[packs[c].x .. packs[c].x + packs[c].y), one or more chains of one
// tree back to back, each head first; a head's node id is stored
// complemented (~u) and head_ro holds its row offset.  Wavefront w runs pack
// w / max_chunks at chunk w % max_chunks, so that every chunk of the
// (longest, first) packs starts first.  The first head's outside state is
// loaded in the prologue; a later head's is staged into the slice during the
// step before it, like every other operand.  Lanes past the tree's sites
// read its last site (every address stays inside the rows) and neither
// store nor add to the counts.  Grid: ceil(cnt * max_chunks / 4) blocks of
// 256; the heads' outside rows must be complete.
template <bool kPacked>
__global__ void __launch_bounds__(256) k_outside_chain(DevForest F, const int2* __restrict__ packs, int cbeg,
                                                        int cnt, const ChainStep* __restrict__ steps,
                                                        const int64_t* __restrict__ head_ro,
                                                        const int32_t* __restrict__ done) {
  __shared__ __align__(16) char lds_all[4 * kChainLdsBytes];
  const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int wv = w / F.max_chunks;
  if (wv >= cnt) return;
  const int2 cd = uniform_load(packs + cbeg + wv);
  const int nb = cd.x, len = cd.y;
  const ChainStep* cs = steps + nb;
  const int64_t* hro = head_ro + nb;
  ChainStep r0 = uniform_load(cs);
  const int u0 = r0.u < 0 ? ~r0.u : r0.u;
  const int t = F.tree_of[u0];
  const int p = F.tree_prob[t];
  const int K = F.tree_nsites[t];
  const int chunk = w - wv * F.max_chunks;
  if (chunk * 64 >= K) return;
  if (done && done[p]) return;
  char* lds = lds_all + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * kChainLdsBytes;
  const int lane = threadIdx.x & 63;
  const int k = chunk * 64 + lane;
  const bool on = k < K;
  const unsigned kk = on ? k : K - 1;
  const double phi = F.phi[p];
  const bool stream = F.stream_rows != 0;
  const unsigned k0 = (unsigned)chunk * 64u;
  const int64_t ru = F.row_off[u0];
  const double2 au = row_at(F.alpha + ru, kk);
  double a0 = au.x, aX = au.y;
  int lu = row_at(F.labels + ru, kk);

  // prologue: step 0's operands and codes and step 1's codes staged
  {
    chain_stage_codes(F, r0, kk, lds);
    chain_stage(F, r0, k0, kk, lane, lds);
  }
  int touch = 0;  // first word of the record four steps ahead (brings its line into the scalar cache)
  if (len > 2) touch = uniform_load(&cs[min(len - 1, 4)].u);

  const int vi = sum12_value(lane);
  double* pp = nullptr;  // partial count held back from the previous step
  double pv = 0.0;
  for (int j = 0;;) {
    chain_wait_all();
    asm volatile("" ::"s"(touch));
    if (pp) *pp = pv;
    const bool more = j + 1 < len;
    r0 = uniform_load(cs + j);
    const ChainStep r1 = uniform_load(cs + (more ? j + 1 : j));
    const bool head1 = kPacked && more && r1.u < 0;
    const int64_t ru1 = head1 ? uniform_load(hro + j + 1) : 0;
    if (j + 4 < len) touch = uniform_load(&cs[j + 4].u);
    // a later chain's head: its outside state, staged during the last step
    const bool head0 = r0.u < 0;
    const int u = head0 ? ~r0.u : r0.u;
    if (kPacked && j > 0 && head0) {
      const double2 h = lds_at<double2>(lds, kChainLdsHeadA + 16 * lane);
      a0 = h.x;
      aX = h.y;
      lu = code_of_word(lds_at<uint32_t>(lds, kChainLdsHeadL + 4 * lane), kk);
    }
    // this step's operands, from the slice (wave-uniform: moved to scalar
    // registers)
    Coef cf[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      cf[i].p1n = uniform_double(lds_at<double>(lds, kChainLdsCoef + 40 * i));
      cf[i].mut = uniform_double(lds_at<double>(lds, kChainLdsCoef + 40 * i + 8));
      cf[i].pn = uniform_double(lds_at<double>(lds, kChainLdsCoef + 40 * i + 16));
      cf[i].msil = uniform_double(lds_at<double>(lds, kChainLdsCoef + 40 * i + 24));
      cf[i].esil = __builtin_amdgcn_readfirstlane(lds_at<int>(lds, kChainLdsCoef + 40 * i + 32));
      cf[i].pad = 0;
    }
    const int raw[2] = {code_of_word(lds_at<uint32_t>(lds, kChainLdsCode + 4 * lane), kk),
                        code_of_word(lds_at<uint32_t>(lds, kChainLdsCode + 256 + 4 * lane), kk)};
    // operands and codes of step j + 1, issued once this step's are read
    // from the slice
    auto stage = [&]() {
      if (more) {
        chain_stage(F, r1, k0, kk, lane, lds);
        chain_stage_codes(F, r1, kk, lds);
        if (head1) chain_stage_head(F, ru1, kk, lds);
      }
    };
    // step j
    PostOut o;
    const int hv = r0.hv;
    const int64_t ro[2] = {r0.ro0, r0.ro1};
    if (r0.ch0 < F.num_leaves) {
      if (r0.ch1 < F.num_leaves)
        chain_compute<kLeaf, kLeaf>(F, lds, lane, cf, phi, hv, raw, ro, kk, on, stream, stage, a0, aX, lu, o);
      else
        chain_compute<kLeaf, kInternal>(F, lds, lane, cf, phi, hv, raw, ro, kk, on, stream, stage, a0, aX, lu, o);
    } else {
      if (r0.ch1 < F.num_leaves)
        chain_compute<kInternal, kLeaf>(F, lds, lane, cf, phi, hv, raw, ro, kk, on, stream, stage, a0, aX, lu, o);
      else
        chain_compute<kInternal, kInternal>(F, lds, lane, cf, phi, hv, raw, ro, kk, on, stream, stage, a0, aX, lu,
                                            o);
    }
    // partial counts (0..4 of child 0, of child 1, the dropout sum), stored at
    // the top of the next step
    double v[12];
#pragma unroll
    for (int m = 0; m < 5; ++m) {
      v[m] = o.S[0][m];
      v[5 + m] = o.S[1][m];
    }
    v[10] = o.rt;
    v[11] = 0.0;
    pv = wave_sum12(v);
    pp = nullptr;
    if (vi >= 0 && vi < 10) {
      const int c = vi >= 5 ? 1 : 0;
      pp = F.cpart + ((int64_t)(c ? r0.ch1 : r0.ch0) * F.max_chunks + chunk) * 5 + (vi - 5 * c);
    } else if (vi == 10) {
      pp = F.rt_part + (int64_t)u * F.max_chunks + chunk;
    }
    if (!more) break;
    ++j;
  }
  if (pp) *pp = pv;
}

// Outside pass over clades: the steps of k_inside_clade's walk in reverse, from
// the clade's root, whose outside state comes from above.  The carried child's
// state stays in registers, the other internal child's waits in the
// wavefront's LDS slice, so that no outside row is written or read below a
// clade's root.  The children's inside rows, labels and codes of the next step
// are copied to the slice during the step, as in k_outside_chain; prior
// weights come from the chunk's piece in LDS and the coefficients in walking
// order, as in k_inside_clade.  EM step of sixteen trees of 10,000 leaves x 300
// sites: 335 us and 126 in the rounds above, where the chain rounds and the
// levels above took 675 us; 50,000 x 500: 178 and 86, 325.  Bound by instruction
// issue (82 % of the VALU cycles at six wavefronts a SIMD).
constexpr int kOutLdsBeta = 0;     // [2][64] double2
constexpr int kOutLdsE = 2048;     // [2][64] int32
constexpr int kOutLdsCode = 2560;  // [2][64] int16
constexpr int kOutLdsSlots = 2816;  // [kCladeSlots][64] double2
constexpr int kOutLdsBytes = kOutLdsSlots + kCladeSlots * 1024;

__device__ __forceinline__ void clade_stage(const DevForest& F, const CladeOut& r, unsigned k0, int lane, char* lds,
                                            bool stream) {
  const int kind = r.flags & 3;
  // codes or labels of both children, a row by each half of the wavefront
  const int16_t* c0 = (kind == 0 ? F.codes : F.labels) + (int64_t)r.row[0] * 64 + k0;
  const int16_t* c1 = (kind == 2 ? F.labels : F.codes) + (int64_t)r.row[1] * 64 + k0;
  to_lds((lane < 32 ? c0 : c1) + 2 * (lane & 31), lds + kOutLdsCode, 4, stream);
  if (kind == 0) return;
  to_lds(&row_at(F.beta + (int64_t)r.row[0] * 64 + k0, (unsigned)lane), lds + kOutLdsBeta, 16, stream);
  to_lds(&row_at(F.bE + (int64_t)r.row[0] * 64 + k0, (unsigned)lane), lds + kOutLdsE, 4, stream);
  if (kind == 1) return;
  to_lds(&row_at(F.beta + (int64_t)r.row[1] * 64 + k0, (unsigned)lane), lds + kOutLdsBeta + 1024, 16, stream);
  to_lds(&row_at(F.bE + (int64_t)r.row[1] * 64 + k0, (unsigned)lane), lds + kOutLdsE + 256, 4, stream);
}

template <int kKind, typename Stage>
__device__ __forceinline__ void clade_out_step(const char* lds, int lane, const CladeCoef& r, double phi, double qs,
                                               const double* q, bool on, Stage&& stage, double a0, double aX,
                                               PostOut& o) {
  const bool lf[2] = {kKind == 0, kKind != 2};
  int lab[2], E[2], code[2];
  double b0[2], bA[2], qv[2];
  Coef cf[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    cf[i] = Coef{r.p1n[i], r.mut[i], r.pn[i], r.msil[i], r.esil[i], 0};
    // (lanes past the tree's sites: label 0)
    const int raw = on ? lds_at<int16_t>(lds, kOutLdsCode + 128 * i + 2 * lane) : 0;
    const double g = q[max(raw, 1)];
    code[i] = raw;
    if (lf[i]) {
      leaf_beta(raw, phi, lab[i], b0[i], bA[i]);
      E[i] = 0;
    } else {
      lab[i] = raw;
      const double2 bb = lds_at<double2>(lds, kOutLdsBeta + 1024 * i + 16 * lane);
      b0[i] = bb.x;
      bA[i] = bb.y;
      E[i] = lds_at<int>(lds, kOutLdsE + 256 * i + 4 * lane);
    }
    qv[i] = lab[i] > 0 ? g : qs;
  }
  // the slice is read: the next step's copies may overwrite it
  chain_wait_lgkm();
  stage();
  Eps ep[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) ep[i] = edge(lab[i], b0[i], bA[i], E[i], qv[i], cf[i]);
  cond_post<false>(combine_label(lab[0], lab[1]), a0, aX, 0.0, phi, lab, b0, bA, qv, ep, cf, lf, code, o);
  if (!on) {
    // lanes past the tree's sites add nothing to the counts
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int m = 0; m < 5; ++m) o.S[i][m] = 0.0;
    o.rt = 0.0;
  }
}

__global__ void __launch_bounds__(64 * kCladeOutWaves)
    k_outside_clade(DevForest F, const int4* __restrict__ blocks, const int4* __restrict__ clades,
                    const CladeOut* __restrict__ steps, int num, const int32_t* __restrict__ done) {
  extern __shared__ __attribute__((aligned(16))) char clade_lds[];
  const int g = (int)blockIdx.x >> 3, b = g / F.max_chunks * 8 + ((int)blockIdx.x & 7), chunk = g % F.max_chunks;
  if (b >= num) return;
  const int4 bd = uniform_load(blocks + b);
  const int t = bd.z, k0 = chunk * 64;
  const int K = F.tree_nsites[t], p = F.tree_prob[t];
  if (k0 >= K) return;
  if (done && done[p]) return;
  const int lane = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int sb = F.tree_site_base[t];
  const bool on = k0 + lane < K;
  const unsigned ks = (unsigned)min(k0 + lane, K - 1);
  const double qs = row_at(F.site_qsum + sb, ks);
  double* qt = (double*)(clade_lds + kCladeOutWaves * kOutLdsBytes);
  const int q0 = uniform_load(F.site_qoff + sb + k0), q1 = uniform_load(F.site_qoff + sb + min(k0 + 64, K));
  for (int i = (int)threadIdx.x; i < q1 - q0; i += 64 * kCladeOutWaves) qt[i] = F.prior[q0 + i];
  const double* q = qt + (row_at(F.site_qoff + sb, ks) - 1 - q0);
  __syncthreads();
  if (wave >= bd.y) return;
  const int4 cd = uniform_load(clades + bd.x + wave);
  const double phi = uniform_load(F.phi + p);
  const bool stream = F.stream_rows != 0;
  char* lds = clade_lds + wave * kOutLdsBytes;
  int j = cd.x + cd.y - 1;
  CladeOut r = uniform_load(steps + j);
  CladeOut r1 = uniform_load(steps + max(j - 1, cd.x));
  CladeCoef cf = uniform_load(F.clade_coef + j);
  double a0, aX;
  {
    const double2 a = row_at(F.alpha + uniform_load(F.row_off + r.u), ks);
    a0 = a.x;
    aX = a.y;
  }
  clade_stage(F, r, (unsigned)k0, lane, lds, stream);
  const int vi = sum12_value(lane);
  double* pp = nullptr;  // partial count held back from the previous step
  double pv = 0.0;
  for (;; --j) {
    chain_wait_all();
    if (pp) *pp = pv;
    const int pop = (r.flags >> 4) & 7;
    if (pop) {
      const double2 a = lds_at<double2>(lds, kOutLdsSlots + (pop - 1) * 1024 + 16 * lane);
      a0 = a.x;
      aX = a.y;
    }
    const int kind = r.flags & 3;
    const bool more = j > cd.x;
    CladeOut r2;
    CladeCoef c1;
    auto stage = [&]() {
      if (more) clade_stage(F, r1, (unsigned)k0, lane, lds, stream);
      r2 = uniform_load(steps + max(j - 2, cd.x));
      c1 = uniform_load(F.clade_coef + max(j - 1, cd.x));
    };
    PostOut o;
    if (kind == 0) clade_out_step<0>(lds, lane, cf, phi, qs, q, on, stage, a0, aX, o);
    else if (kind == 1) clade_out_step<1>(lds, lane, cf, phi, qs, q, on, stage, a0, aX, o);
    else {
      clade_out_step<2>(lds, lane, cf, phi, qs, q, on, stage, a0, aX, o);
      *(double2*)(lds + kOutLdsSlots + ((r.flags >> 2) & 3) * 1024 + 16 * lane) = make_double2(o.a0[1], o.aX[1]);
    }
    a0 = o.a0[0];
    aX = o.aX[0];
    // partial counts (as in k_outside_chain)
    double v[12];
#pragma unroll
    for (int m = 0; m < 5; ++m) {
      v[m] = o.S[0][m];
      v[5 + m] = o.S[1][m];
    }
    v[10] = o.rt;
    v[11] = 0.0;
    pv = wave_sum12(v);
    pp = nullptr;
    if (vi >= 0 && vi < 10) {
      const int c = vi >= 5 ? 1 : 0;
      pp = F.cpart + ((int64_t)(c ? r.ch[1] : r.ch[0]) * F.max_chunks + chunk) * 5 + (vi - 5 * c);
    } else if (vi == 10) {
      pp = F.rt_part + (int64_t)r.u * F.max_chunks + chunk;
    }
    if (!more) break;
    r = r1;
    r1 = r2;
    cf = c1;
  }
  if (pp) *pp = pv;
}

template <int W>
__global__ void __launch_bounds__(256) k_outside(DevForest F, int beg, int cnt, const int32_t* __restrict__ done) {
  Seg<W> g;
  if (!g.init(beg, cnt)) return;
  outside_node<W>(F, g.v, (int)blockIdx.y, g.lane, done);
}

// Outside pass over the top levels, from level h1-1 down to h0, one block per
// site chunk (see k_inside_top).
template <int W>
__global__ void __launch_bounds__(1024) k_outside_top(DevForest F, int h0, int h1, const int32_t* __restrict__ done) {
  const int segs = 1024 / W;
  const int seg = threadIdx.x / W;
  const int lane = threadIdx.x & (W - 1);
  for (int h = h1 - 1; h >= h0; --h) {
    const int e = F.level_off[h + 1];
    for (int u = F.level_off[h] + seg; u < e; u += segs) outside_node<W>(F, u, (int)blockIdx.x, lane, done);
    __syncthreads();
  }
}



// threads per tree-walk block (16 wavefronts share each level of the tree)
constexpr int kWalkThreads = 1024;

// Tree walk: one block per (tree, chunk of W sites) runs the whole pass of
// that tree at those sites -- inside levels bottom-up, the root step, outside
// levels top-down -- with block barriers between levels.  Sites of one chunk
// never depend on other chunks, so blocks are independent: a forest of many
// trees of uneven sizes is one launch per pass, and each block stops at its
// own tree's height.  phases: 1 inside, 2 root, 4 outside (any combination,
// in that order).  Levels below h_lo are left to level launches (the hybrid
// pass: the walk covers the small top levels of every tree at once).
template <int W>
__global__ void __launch_bounds__(kWalkThreads) k_tree_walk(DevForest F, TreeWalk TW, int phases, int h_lo,
                                                            double* __restrict__ site_llh_out,
                                                            const int32_t* __restrict__ done) {
  const int t = TW.blk_tree[blockIdx.x];
  const int chunk = TW.blk_chunk[blockIdx.x];
  const int p = F.tree_prob[t];
  if (done && done[p]) return;
  const int K = F.tree_nsites[t];
  constexpr int kSegs = kWalkThreads / W;
  const int seg = (int)(threadIdx.x / W);
  const int lane = threadIdx.x & (W - 1);
  const int k = chunk * W + lane;
  const int lb = TW.lvl_base[t];
  const int H = TW.lvl_base[t + 1] - lb;
  const int hb = max(1, h_lo);
  if (phases & 1) {
    for (int h = hb; h < H; ++h) {
      const int beg = uniform_load(TW.lvl_beg + lb + h), cnt = uniform_load(TW.lvl_cnt + lb + h);
      for (int i = seg; i < cnt; i += kSegs) {
        const int v = W == 64 ? __builtin_amdgcn_readfirstlane(beg + i) : beg + i;
        if (k < K) {
          InNode n;
          const NodeRec r = uniform_load(F.nrec + (v - F.num_leaves));
          in_node_rec(F, r, n);
          if constexpr (W == 64)
            inside_site_q(F, n, k, chain_q_row(F, r.ch0, r.ro0), chain_q_row(F, r.ch1, r.ro1));
          else
            inside_site<kNoCherry, kNoCherry>(F, n, k);
        }
      }
      __syncthreads();
    }
  }
  if (phases & 2) {
    if (seg == 0) root_chunk<W>(F, t, chunk, lane, site_llh_out);
    __syncthreads();
  }
  if (phases & 4) {
    for (int h = H - 1; h >= hb; --h) {
      const int beg = uniform_load(TW.lvl_beg + lb + h), cnt = uniform_load(TW.lvl_cnt + lb + h);
      for (int i = seg; i < cnt; i += kSegs) {
        const int u = W == 64 ? __builtin_amdgcn_readfirstlane(beg + i) : beg + i;
        OutNode n;
        const NodeRec r = uniform_load(F.nrec + (u - F.num_leaves));
        out_node_rec(F, r, n);
        double acc[2][5];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int j = 0; j < 5; ++j) acc[a][j] = 0.0;
        double rt = 0.0;
        if constexpr (W == 64) {
          if (k < K) outside_site_q(F, n, k, acc, rt, chain_q_row(F, r.ch0, r.ro0), chain_q_row(F, r.ch1, r.ro1));
        } else {
          if (k < K) outside_site<kNoCherry, kNoCherry>(F, n, k, acc, rt);
        }
        out_write_partials<W>(F, u, n.ch, lane, chunk, chunk + 1, acc, rt);
      }
      __syncthreads();
    }
  }
}

// Per-node counts: fixed-order sum of the per-chunk partials, one thread per
// (node, count), so that a wavefront's loads of one chunk slot cover a few
// whole partial records instead of one value per 200-byte record.
__global__ void __launch_bounds__(256) k_counts(DevForest F, double* __restrict__ counts) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)F.num_nodes * 5) return;
  const int v = (int)(idx / 5);
  const int j = (int)(idx - (int64_t)v * 5);
  const int C = (F.tree_nsites[F.tree_of[v]] + F.chunk_w - 1) / F.chunk_w;
  const double* src = F.cpart + v * F.cp_v + j;
  double s = 0.0;
  for (int c = 0; c < C; ++c) s += src[c * 5];
  counts[idx] = s;
}

// ---------------------------------------------------------------------------
// per-problem reductions (one block per problem, fixed order => deterministic)
// ---------------------------------------------------------------------------
template <int NT>
__device__ __forceinline__ double block_sum(double x, double* sh) {
  x = seg_sum<64>(x);
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) sh[wid] = x;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) s += sh[i];
  __syncthreads();
  return s;
}

// Sum of per-site log-likelihoods of every tree of a problem, plus the EM
// bookkeeping of the device loop when em.done != nullptr.
// Per-problem log-likelihood; inside the EM loop also the convergence test
// of EM_solver.EM_optimization (EM_solver.py:483-512).  The EM step number of
// each problem lives on the device (em.step), so that a captured EM step can
// be replayed unchanged.
__global__ void __launch_bounds__(256) k_llh(DevForest F, double* __restrict__ nll, EmState em, int max_iter,
                                             double tol) {
  __shared__ double sh[4];
  const int p = blockIdx.x;
  if (em.done && em.done[p]) return;
  double s = 0.0;
  for (int t = F.prob_tree_off[p]; t < F.prob_tree_off[p + 1]; ++t) {
    const int K = F.tree_nsites[t];
    const int sb = F.tree_site_base[t];
    for (int k = threadIdx.x; k < K; k += 256) s += F.site_llh[sb + k];
  }
  const double llh = block_sum<256>(s, sh);
  if (threadIdx.x != 0) return;
  if (nll) nll[p] = -llh;
  if (!em.done) return;
  const int step = em.step[p];
  em.step[p] = step + 1;
  if (em.trace) em.trace[(int64_t)step * F.num_problems + p] = -llh;
  if (step > 0) {
    const double pre = em.pre[p];
    if (tol > 0.0 && fabs((llh - pre) / pre) < tol) {
      em.done[p] = 1;
      em.iters[p] = step;
      return;
    }
  }
  em.pre[p] = llh;
  if (step >= max_iter) {
    em.done[p] = 1;
    em.iters[p] = max_iter + 1;
  }
}

constexpr int kRedThreads = 1024;

// adds node v's per-chunk dropout sums, chunks 0 .. C-1 in order, to s; up
// to 8 chunks are loaded together before the additions
__device__ __forceinline__ void add_node_rt(const DevForest& F, int64_t v, int C, double& s) {
  constexpr int kC = 8;
  const double* src = F.rt_part + v * F.rt_v;
  if (C <= kC) {
    double x[kC];
#pragma unroll
    for (int c = 0; c < kC; ++c) x[c] = c < C ? src[c] : 0.0;
#pragma unroll
    for (int c = 0; c < kC; ++c)
      if (c < C) s += x[c];
  } else {
    for (int c = 0; c < C; ++c) s += src[c];
  }
}

// sum over the problem's internal nodes of the per-node dropout sums
__device__ __forceinline__ double problem_rtilde(const DevForest& F, int p, double* sh) {
  double s = 0.0;
  const int b = F.prob_int_off[p], e = F.prob_node_off[p + 1];
  const int C = (F.tree_nsites[F.prob_tree_off[p]] + F.chunk_w - 1) / F.chunk_w;
  for (int i = b + threadIdx.x; i < e; i += kRedThreads) add_node_rt(F, F.prob_nodes[i], C, s);
  return block_sum<kRedThreads>(s, sh);
}

// Sum of the dropout responsibilities of missing leaf entries of a problem.
__global__ void __launch_bounds__(kRedThreads) k_rtilde(DevForest F, double* __restrict__ rtilde,
                                                        const int32_t* __restrict__ done) {
  __shared__ double sh[kRedThreads / 64];
  const int p = blockIdx.x;
  if (done && done[p]) return;
  const double rt = problem_rtilde(F, p, sh);
  if (threadIdx.x == 0) rtilde[p] = rt;
}

// ---------------------------------------------------------------------------
// M-step
// ---------------------------------------------------------------------------
// the objective of a branch with expected counts s (clamped and renormalised
// in place) over K sites
__device__ __forceinline__ BranchObj branch_obj(double (&s)[5], double K, double nu0) {
  double tot = 0.0;
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    s[j] = fmax(kEpsS, s[j]);
    tot += s[j];
  }
#pragma unroll
  for (int j = 0; j < 5; ++j) s[j] = s[j] / tot * K;
  BranchObj o;
  o.nu = nu0;
  o.A = (nu0 + 1.0) * s[0] + nu0 * s[1] + nu0 * s[3];
  o.S1 = s[1];
  o.B = nu0 > kEpsNu ? (s[2] + s[4]) : 0.0;
  return o;
}
// the new length of a free branch, and its coefficients of the nu problem
__device__ __forceinline__ double branch_length(const DevForest& F, double (&s)[5], double K, double nu0, double d,
                                                double& na, double& nb) {
  const BranchObj o = branch_obj(s, K, nu0);
  na = s[0] + s[1] + s[3];
  nb = s[2] + s[4];
  return solve_branch(o, F.dmin, F.dmax, d);
}

// nu maximises a concave function of one variable over [0, 1] given the new
// branch lengths (EM_solver.py:392-407); its derivative
// h'(x) = sum_v d_v (b_v / expm1(x d_v) - a_v) sums over every branch of the
// problem.  Warm-started solves take one evaluation of h' and its derivatives,
// two when nu moves by more than kNuDone x (Newton steps to 1e-12 took three
// to five).  Each problem's branches are split into spans of kNuThreads, a
// block each, in two launches of an evaluation each, which write their spans'
// sums; the next kernel's blocks all add the sums of their problem (in an
// order set by the problem alone) and take the step.  So the kernels need no
// fence between blocks: one with a last block that adds the sums took 80 us
// for 16 problems of 20k branches, 30 us of it in the write-back that the
// fence asks of the L2 caches.  The first evaluation follows the branch solves
// in the same kernel and also sums the dropout responsibilities, for phi in
// closed form (EM_solver.py:318-326).  k_nu_finish, a block per problem, takes
// the last step and goes on alone where the solve is still open.
constexpr int kNuThreads = kNuSpan;
// evaluations a nu solve may take in all before its M-step reports failure:
// the bracket halves at least every other evaluation, so this is far more
// than [0, 1] needs to close to 1e-12 relative at any optimum the clamped
// counts allow (nu* >= ~1e-12)
constexpr int kNuMaxEvals = 200;
constexpr int kNuFinishThreads = 512;

// Sums over the block in every thread, in one pass through LDS (sh: 6 NT / 64
// doubles).
template <int NT>
__device__ __forceinline__ void nu_block_sum(NuSum& n, double& rt, double& bad, double* sh) {
  double v[6] = {n.g, n.g1, n.g2, n.g3, rt, bad};
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    v[j] = seg_sum_last<64>(v[j]);
    if ((threadIdx.x & 63) == 63) sh[(threadIdx.x >> 6) * 6 + j] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    v[j] = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) v[j] += sh[w * 6 + j];
  }
  __syncthreads();
  n = NuSum{v[0], v[1], v[2], v[3]};
  rt = v[4];
  bad = v[5];
}

// the sums of the span of block blk, evaluation e
__device__ __forceinline__ double* nu_span(const DevForest& F, int e, int blk) {
  return F.nu_part + ((int64_t)e * F.num_nu_blocks + blk) * 6;
}
__device__ __forceinline__ void nu_store(const DevForest& F, int e, NuSum n, double rt, double bad, double* sh) {
  nu_block_sum<kNuThreads>(n, rt, bad, sh);
  if (threadIdx.x != 0) return;
  double* o = nu_span(F, e, (int)blockIdx.x);
  o[0] = n.g;
  o[1] = n.g1;
  o[2] = n.g2;
  o[3] = n.g3;
  if (e != 0) return;
  o[4] = rt;
  o[5] = bad;
}

// the sums of evaluation e of problem p in every thread (the same bits for
// every NT)
template <int NT>
__device__ __forceinline__ void nu_load(const DevForest& F, int p, int e, NuSum& n, double& rt, double& bad,
                                        double* sh) {
  const int b0 = F.prob_blk_off[p], nparts = F.prob_blk_off[p + 1] - b0;
  n = NuSum{0.0, 0.0, 0.0, 0.0};
  rt = bad = 0.0;
  if ((int)threadIdx.x < kNuThreads)
    for (int q = (int)threadIdx.x; q < nparts; q += kNuThreads) {
      const double* o = nu_span(F, e, b0 + q);
      n.g += o[0];
      n.g1 += o[1];
      n.g2 += o[2];
      n.g3 += o[3];
      rt += o[4];
      bad += o[5];
    }
  nu_block_sum<NT>(n, rt, bad, sh);
}

// the problem whose spans hold block blk, by binary search over prob_blk_off
__device__ __forceinline__ int nu_problem(const DevForest& F, int blk) {
  int lo_p = 0, hi_p = F.num_problems;
  while (hi_p - lo_p > 1) {
    const int mid = (lo_p + hi_p) >> 1;
    if (F.prob_blk_off[mid] <= blk) lo_p = mid; else hi_p = mid;
  }
  return lo_p;
}

// Branch lengths of every free branch (EM_solver.py:328-366): counts are
// clamped at eps_s and renormalised to sum K, then the per-branch concave
// problem is solved exactly with the current nu; then the first nu
// evaluation, at the current nu (or 1/2 when outside (0, 1)).  The branch's
// nu coefficients are staged at its position in the problem for the later
// evaluations.  Ultrametric forests solve their lengths together: for them
// the objective of every branch is written instead, and k_nu_eval<true>
// follows k_ultra.  Bound by latency (counts, then the dependent steps of the
// solves, then the sums): 20k branches of one problem 9 us with the first nu
// evaluation, 16 such problems 31 us; the M-step of the first with the two
// kernels below 20 us, 58 us when nu took six Newton launches after the branch
// solves, of the second 47 us, 111 us.
template <bool kUltra>
__global__ void __launch_bounds__(kNuThreads) k_branch(DevForest F, const double* __restrict__ counts,
                                                       const double* __restrict__ rtilde_in, double* __restrict__ d,
                                                       const double* __restrict__ nu,
                                                       const int32_t* __restrict__ done, UltraDev U) {
  __shared__ double sh[6 * (kNuThreads / 64)];
  const int p = nu_problem(F, (int)blockIdx.x);
  const int part = (int)blockIdx.x - F.prob_blk_off[p];
  if (done && done[p]) return;
  const int pos = F.prob_node_off[p] + part * kNuThreads + (int)threadIdx.x;
  const double nu0 = nu[p];
  const uint32_t flags = F.prob_flags[p];
  double na = 0.0, nb = 0.0, dn = 0.0, rt = 0.0, bad = 0.0;
  if (pos < F.prob_node_off[p + 1]) {
    const int v = F.prob_nodes[pos];
    dn = d[v];
    const int Kt = F.tree_nsites[F.tree_of[v]];
    const int C = (Kt + F.chunk_w - 1) / F.chunk_w;
    if (!kUltra && (flags & 1u) && !rtilde_in && pos >= F.prob_int_off[p]) add_node_rt(F, v, C, rt);
    if (F.free_branch[v]) {
      double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
      if (counts) {
#pragma unroll
        for (int j = 0; j < 5; ++j) s[j] = counts[(int64_t)v * 5 + j];
      } else {
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int j = 0; j < 5; ++j) s[j] += F.cpart[v * F.cp_v + c * 5 + j];
      }
      if (kUltra) {
        const BranchObj o = branch_obj(s, (double)Kt, nu0);
        U.bA[v] = o.A;
        U.bS1[v] = o.S1;
        U.bB[v] = o.B;
        na = s[0] + s[1] + s[3];
        nb = s[2] + s[4];
      } else {
        dn = branch_length(F, s, (double)Kt, nu0, dn, na, nb);
        if (!isfinite(dn)) bad = 1.0;
        d[v] = dn;
      }
    }
    F.nu_a[pos] = na;
    F.nu_b[pos] = nb;
    F.nu_d[pos] = dn;  // (ultrametric: of fixed branches; k_ultra sets the others)
  }
  if (kUltra) return;
  const bool opt_nu = (flags & 2u) && F.prob_nfree[p] > 0;
  NuSum n{0.0, 0.0, 0.0, 0.0};
  if (opt_nu) nu_term(na, nb, dn, nu_start(nu0), n);
  nu_store(F, 0, n, rt, bad, sh);
}

// An evaluation of the nu solves: the first one (after k_ultra), or the second
// one of those that the first has not brought to their end.
template <bool kFirst>
__global__ void __launch_bounds__(kNuThreads) k_nu_eval(DevForest F, const double* __restrict__ rtilde_in,
                                                        const double* __restrict__ nu,
                                                        const int32_t* __restrict__ done) {
  __shared__ double sh[6 * (kNuThreads / 64)];
  const int p = nu_problem(F, (int)blockIdx.x);
  if (done && done[p]) return;
  const uint32_t flags = F.prob_flags[p];
  const bool opt_nu = (flags & 2u) && F.prob_nfree[p] > 0;
  const int pos = F.prob_node_off[p] + ((int)blockIdx.x - F.prob_blk_off[p]) * kNuThreads + (int)threadIdx.x;
  const bool on = pos < F.prob_node_off[p + 1];
  double x = nu_start(nu[p]), rt = 0.0;
  NuSum n{0.0, 0.0, 0.0, 0.0};
  if (!kFirst) {
    if (!opt_nu) return;
    double r, b, lo = 0.0, hi = 2.0, xn;
    nu_load<kNuThreads>(F, p, 0, n, r, b, sh);
    const bool fin = nu_step(x, n, lo, hi, xn);
    if (threadIdx.x == 0) {
      // the step as k_nu_finish is to take it
      double* o = nu_span(F, 1, (int)blockIdx.x);
      o[4] = xn;
      o[5] = fin ? 1.0 : 0.0;
    }
    if (fin) return;
    x = xn;
    n = NuSum{0.0, 0.0, 0.0, 0.0};
  } else if (on && (flags & 1u) && !rtilde_in && pos >= F.prob_int_off[p]) {
    const int C = (F.tree_nsites[F.prob_tree_off[p]] + F.chunk_w - 1) / F.chunk_w;
    add_node_rt(F, F.prob_nodes[pos], C, rt);
  }
  if (on && opt_nu) nu_term(F.nu_a[pos], F.nu_b[pos], F.nu_d[pos], x, n);
  nu_store(F, kFirst ? 0 : 1, n, rt, 0.0, sh);
}

// phi, the end of the nu solve and the status of the M-step, a block per
// problem: the steps of the two evaluations, and more of them where the solve
// is still open.
__global__ void __launch_bounds__(kNuFinishThreads) k_nu_finish(DevForest F, const double* __restrict__ rtilde_in,
                                                               double* __restrict__ nu, double* __restrict__ phi,
                                                               const int32_t* __restrict__ done) {
  __shared__ double sh[6 * (kNuFinishThreads / 64)];
  const int p = blockIdx.x;
  if (done && done[p]) return;
  const uint32_t flags = F.prob_flags[p];
  const bool opt_nu = (flags & 2u) && F.prob_nfree[p] > 0;
  double x = nu_start(nu[p]), rt, bad, lo = 0.0, hi = 2.0, xn;  // (hi > 1: x = 1 not evaluated)
  NuSum n;
  nu_load<kNuFinishThreads>(F, p, 0, n, rt, bad, sh);
  bool fin = true;
  if (opt_nu) {
    nu_step(x, n, lo, hi, xn);
    const double* o = nu_span(F, 1, F.prob_blk_off[p]);
    x = o[4];
    fin = o[5] != 0.0;
    const int e = F.prob_node_off[p + 1];
    for (int evals = 1; evals < kNuMaxEvals && !fin; ++evals) {
      double z0 = 0.0, z1 = 0.0;
      if (evals == 1) {
        nu_load<kNuFinishThreads>(F, p, 1, n, z0, z1, sh);
      } else {
        n = NuSum{0.0, 0.0, 0.0, 0.0};
        for (int i = F.prob_node_off[p] + (int)threadIdx.x; i < e; i += kNuFinishThreads)
          nu_term(F.nu_a[i], F.nu_b[i], F.nu_d[i], x, n);
        nu_block_sum<kNuFinishThreads>(n, z0, z1, sh);
      }
      fin = nu_step(x, n, lo, hi, xn);
      x = xn;
    }
  }
  if (threadIdx.x != 0) return;
  if (opt_nu) nu[p] = x;
  if (flags & 1u) {
    const double r = rtilde_in ? rtilde_in[p] : rt;
    double phi_star = r / (F.prob_nobs[p] + r);
    if (fabs(phi_star) < F.prob_phimin[p]) phi_star = 0.0;
    phi[p] = phi_star;
  }
  // a branch length came out non-finite: reported as the reference's failed
  // branch solve (EM_solver.py:415-418,450-459)
  F.mstep_status[p] = (bad != 0.0 ? 1 : 0) | (fin ? 0 : 2);
}

// ---------------------------------------------------------------------------
// Gradient of the negative log-likelihood (Fisher identity: the gradient of
// log L is the posterior expectation of the complete-data score).  With raw
// per-branch expected counts S0..S4 from the outside pass:
//   dlogL/dd_v  = -(1+nu) S0 + S1 (1/expm1(d) - nu) + (S2+S4) nu/expm1(nu d) - nu S3
//   dlogL/dnu   = sum_v d_v (-S0 - S1 - S3 + (S2+S4)/expm1(nu d_v))
//   dlogL/dphi  = -n_obs/(1-phi) + Rt/phi
// n_obs counts leaf entries observed as 0 or an edit (an explicit -1 entry
// does not depend on phi); Rt sums P(leaf not silenced | D) over '?' entries.
// ---------------------------------------------------------------------------
// a branch of length dv with counts s: dlogL/dd, and its part of dlogL/dnu but
// -dv (S0 + S1 + S3)
__device__ __forceinline__ double grad_length(const double (&s)[5], double dv, double x) {
  double g = -(1.0 + x) * s[0] + s[1] * (1.0 / expm1(dv) - x) - x * s[3];
  if (s[2] + s[4] != 0.0) g += (s[2] + s[4]) * x / expm1(x * dv);
  return g;
}
__device__ __forceinline__ double grad_nu_part(double b, double dv, double x) {
  return b != 0.0 ? b * dv / expm1(x * dv) : 0.0;
}
__device__ __forceinline__ double grad_phi_of(double nobs, double rt, double ph) {
  return nobs / (1.0 - ph) - (rt != 0.0 ? rt / ph : 0.0);
}

__global__ void k_grad_branch(DevForest F, const double* __restrict__ d, const double* __restrict__ nu,
                              double* __restrict__ grad_d) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= F.num_nodes) return;
  const int t = F.tree_of[v];
  const int p = F.tree_prob[t];
  const int C = (F.tree_nsites[t] + F.chunk_w - 1) / F.chunk_w;
  double s[5] = {0, 0, 0, 0, 0};
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int j = 0; j < 5; ++j) s[j] += F.cpart[v * F.cp_v + c * 5 + j];
  const double dv = d[v];
  grad_d[v] = -grad_length(s, dv, nu[p]);
  F.nu_a[F.node_pos[v]] = s[0] + s[1] + s[3];
  F.nu_b[F.node_pos[v]] = s[2] + s[4];
  F.nu_d[F.node_pos[v]] = dv;
}

__global__ void __launch_bounds__(kRedThreads) k_grad_problem(DevForest F, const double* __restrict__ nu,
                                                              const double* __restrict__ phi,
                                                              double* __restrict__ grad_nu,
                                                              double* __restrict__ grad_phi) {
  __shared__ double sh[kRedThreads / 64];
  const int p = blockIdx.x;
  const double x = nu[p];
  double g = 0.0;
  for (int i = F.prob_node_off[p] + threadIdx.x; i < F.prob_node_off[p + 1]; i += kRedThreads) {
    const double dv = F.nu_d[i];
    g -= dv * F.nu_a[i];
    g += grad_nu_part(F.nu_b[i], dv, x);
  }
  g = block_sum<kRedThreads>(g, sh);
  const double rt = problem_rtilde(F, p, sh);
  if (threadIdx.x == 0) {
    grad_nu[p] = -g;
    grad_phi[p] = grad_phi_of(F.prob_nobs_phi[p], rt, phi[p]);
  }
}

// ---------------------------------------------------------------------------
// Ultrametric branch-length M-step (EM_solver.py:349-366 with the equality
// system of EM_solver.py:53-89).  Heights of the variable height classes are
// the unknowns, d_v = t(parent side) - t(child side).  A log-barrier keeps
// every free branch in (dmin, dmax); each Newton system is a weighted tree
// Laplacian over the classes and is solved exactly by eliminating classes
// bottom-up and substituting top-down (two level sweeps).  One block per
// problem; every decision depends on block-reduced values, so control flow is
// uniform across the block.
// ---------------------------------------------------------------------------
constexpr int kUltraThreads = 1024;

template <int NT>
__device__ __forceinline__ double block_min(double x, double* sh) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = fmin(x, __shfl_xor(x, off, 64));
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) sh[wid] = x;
  __syncthreads();
  double s = sh[0];
#pragma unroll
  for (int i = 1; i < NT / 64; ++i) s = fmin(s, sh[i]);
  __syncthreads();
  return s;
}

__device__ __forceinline__ double ult_height(const UltraDev& U, int c, double off) {
  return c >= 0 ? U.t[c] + off : off;
}

// height at t + a dt (only called with a finite direction)
__device__ __forceinline__ double ult_height_at(const UltraDev& U, int c, double off, double a) {
  return c >= 0 ? fma(a, U.dt[c], U.t[c]) + off : off;
}

// branch objective (barrier excluded): value, first and second derivative
__device__ __forceinline__ void ult_obj(double A, double S1, double B, double nu, double d, double& f, double& g,
                                        double& h) {
  const double em = expm1(d);
  f = -A * d + S1 * log(-expm1(-d));
  g = -A + S1 / em;
  h = -S1 * (em + 1.0) / (em * em);
  if (B > 0.0) {
    const double en = expm1(nu * d);
    f += B * log(-expm1(-nu * d));
    g += B * nu / en;
    h -= B * nu * nu * (en + 1.0) / (en * en);
  }
}

// barrier objective of problem p's free branches at heights t + a dt
__device__ double ult_phi(const DevForest& F, const UltraDev& U, int nb, int ne, double nu0, double mu, double a,
                          double* sh) {
  double s = 0.0;
  for (int i = nb + threadIdx.x; i < ne; i += kUltraThreads) {
    const int v = F.prob_nodes[i];
    if (!F.free_branch[v]) continue;
    const double dv =
        ult_height_at(U, U.up_cls[v], U.up_off[v], a) - ult_height_at(U, U.dn_cls[v], U.dn_off[v], a);
    const double lo = dv - F.dmin, hi = F.dmax - dv;
    if (!(lo > 0.0 && hi > 0.0)) {
      s = -INFINITY;
      continue;
    }
    double f, g, h;
    ult_obj(U.bA[v], U.bS1[v], U.bB[v], nu0, dv, f, g, h);
    s += f + mu * (log(lo) + log(hi));
  }
  return block_sum<kUltraThreads>(s, sh);
}

// The barrier method: mu falls tenfold a round, each round a damped Newton
// solve (60 to 135 Newton systems a solve, more where the warm start lies at
// the bounds).  Solves that the primal-dual method below does not finish.
__device__ void ultra_barrier(const DevForest& F, const UltraDev& U, double* __restrict__ d,
                              const double* __restrict__ nu, int p, double* sh) {
  const int P = F.num_problems;
  const int nb = F.prob_node_off[p], ne = F.prob_node_off[p + 1];
  const double nu0 = nu[p];
  const double dmin = F.dmin, dmax = F.dmax;
  const double K = (double)F.tree_nsites[F.prob_tree_off[p]];
  const int H = U.num_levels;
  int status = 0;
  double mu = 1e-2 * K;
  const double mu_end = 1e-13 * K;
  for (int outer = 0; outer < 40; ++outer) {
    for (int it = 0; it < 60; ++it) {
      // branch derivatives of the barrier objective
      for (int i = nb + threadIdx.x; i < ne; i += kUltraThreads) {
        const int v = F.prob_nodes[i];
        if (!F.free_branch[v]) continue;
        const double dv = ult_height(U, U.up_cls[v], U.up_off[v]) - ult_height(U, U.dn_cls[v], U.dn_off[v]);
        const double lo = dv - dmin, hi = dmax - dv;
        double f, g, h;
        ult_obj(U.bA[v], U.bS1[v], U.bB[v], nu0, dv, f, g, h);
        U.gp[v] = g + mu * (1.0 / lo - 1.0 / hi);
        U.w[v] = -h + mu * (1.0 / (lo * lo) + 1.0 / (hi * hi));
      }
      __syncthreads();
      // eliminate classes bottom-up.  The eliminated diagonal of class c is
      // D_c = G_c + w(edge to the parent class), where G_c, the conductance of
      // c's subtree to the pinned heights, sums positive terms only: pinned
      // neighbours add w, a child class k adds the series conductance
      // w G_k / (w + G_k).  (Forming D_c as sum(w) - sum(w^2 / D_k) cancels to
      // zero when one branch's barrier weight dominates.)
      for (int lv = 0; lv < H; ++lv) {
        const int cb = U.plo[lv * P + p], ce = U.plo[lv * P + p + 1];
        for (int c = cb + threadIdx.x; c < ce; c += kUltraThreads) {
          double gg = 0.0, G = 0.0, wup = 0.0, rr = 0.0;
          for (int j = U.inc_off[c]; j < U.inc_off[c + 1]; ++j) {
            const int v = U.inc_branch[j];
            const double wv = U.w[v];
            if (U.inc_sign[j] > 0) {
              gg += U.gp[v];
              const int kc = U.dn_cls[v];
              if (kc >= 0) {
                const double Dk = U.Dd[kc];
                G += wv * (U.Gg[kc] / Dk);
                rr += wv * (U.r[kc] / Dk);
              } else {
                G += wv;
              }
            } else {
              gg -= U.gp[v];
              if (U.up_cls[v] >= 0) wup += wv; else G += wv;
            }
          }
          U.g[c] = gg;
          U.Gg[c] = G;
          U.Dd[c] = G + wup;
          U.r[c] = gg + rr;
        }
        __syncthreads();
      }
      // substitute top-down
      for (int lv = H - 1; lv >= 0; --lv) {
        const int cb = U.plo[lv * P + p], ce = U.plo[lv * P + p + 1];
        for (int c = cb + threadIdx.x; c < ce; c += kUltraThreads) {
          const int pc = U.cls_parent[c];
          U.dt[c] = pc < 0 ? U.r[c] / U.Dd[c] : (U.r[c] + U.w[U.cls_pedge[c]] * U.dt[pc]) / U.Dd[c];
        }
        __syncthreads();
      }
      // Newton decrement, largest step keeping every branch inside the box
      double lam = 0.0, step = 0.0;
      const int c0 = U.plo[p], c1 = U.plo[(H - 1) * P + p + 1];
      for (int lv = 0; lv < H; ++lv) {
        const int cb = U.plo[lv * P + p], ce = U.plo[lv * P + p + 1];
        for (int c = cb + threadIdx.x; c < ce; c += kUltraThreads) {
          lam += U.g[c] * U.dt[c];
          step = fmax(step, fabs(U.dt[c]) / (1.0 + fabs(U.t[c])));
        }
      }
      (void)c0;
      (void)c1;
      double amax = 1.0;
      for (int i = nb + threadIdx.x; i < ne; i += kUltraThreads) {
        const int v = F.prob_nodes[i];
        if (!F.free_branch[v]) continue;
        const double dv = ult_height(U, U.up_cls[v], U.up_off[v]) - ult_height(U, U.dn_cls[v], U.dn_off[v]);
        const double dd = (U.up_cls[v] >= 0 ? U.dt[U.up_cls[v]] : 0.0) - (U.dn_cls[v] >= 0 ? U.dt[U.dn_cls[v]] : 0.0);
        if (dd < 0.0) amax = fmin(amax, 0.99 * (dv - dmin) / (-dd));
        else if (dd > 0.0) amax = fmin(amax, 0.99 * (dmax - dv) / dd);
      }
      lam = block_sum<kUltraThreads>(lam, sh);
      step = -block_min<kUltraThreads>(-step, sh);
      amax = block_min<kUltraThreads>(amax, sh);
      if (!isfinite(lam) || !isfinite(step)) {
        status = 2;  // singular Newton system: keep the current heights
        break;
      }
      if (!(lam > 0.0) || step * amax <= 1e-15) break;
      double a = amax;
      const double phi0 = ult_phi(F, U, nb, ne, nu0, mu, 0.0, sh);
      if (lam > 1e-12 * (1.0 + fabs(phi0))) {
        // backtracking (Armijo) while the predicted gain is measurable
        int k = 0;
        for (; k < 40; ++k) {
          const double phi1 = ult_phi(F, U, nb, ne, nu0, mu, a, sh);
          if (phi1 >= phi0 + 0.25 * a * lam) break;
          a *= 0.5;
        }
        if (k == 40) {
          status = 1;
          break;
        }
      }
      for (int lv = 0; lv < H; ++lv) {
        const int cb = U.plo[lv * P + p], ce = U.plo[lv * P + p + 1];
        for (int c = cb + threadIdx.x; c < ce; c += kUltraThreads) U.t[c] += a * U.dt[c];
      }
      __syncthreads();
      if (step * a <= 1e-15) break;
    }
    if (mu <= mu_end) break;
    mu = fmax(mu * 0.1, mu_end);
  }
  for (int i = nb + threadIdx.x; i < ne; i += kUltraThreads) {
    const int v = F.prob_nodes[i];
    if (!F.free_branch[v]) continue;
    const double dv = ult_height(U, U.up_cls[v], U.up_off[v]) - ult_height(U, U.dn_cls[v], U.dn_off[v]);
    d[v] = dv;
    F.nu_d[F.node_pos[v]] = dv;
  }
  if (threadIdx.x == 0) U.status[p] = status;
}

// ---------------------------------------------------------------------------
// Quartet-local EM of NNI candidates (Topology_search.py:242-322 with
// local_brlen_opt): nu, phi and every branch except the five around the move
// are fixed, so the subtrees hanging off the quartet (A and W below u, C below
// v) keep their inside vectors and the data above v keeps its outside state.
// A candidate's EM then needs, per site, only those inputs and the five free
// branches: each EM step is O(K) instead of a pass over the tree.
//
// Candidate c (after the move): v has children u and C, u has children A and
// W; p is v's parent and s v's sibling (p = -1: v is the root and its branch
// is the stem from the unedited ancestor).  Free branches in the order
// (A, W, u, C, v); opt bit j set = branch j is optimised.
// ---------------------------------------------------------------------------
namespace {

// Data outside a branch joint with its top unedited (A) / in an edit state
// that the data below allow (G), over the site likelihood and on a power of
// two of the caller's choice (cond_post's A and G).
struct QTop {
  double A, G;
};

// posterior counts of the branch above a node with inside mantissas (b0, bA),
// prior weight q and edge values ep (t on the scale of ep, over the candidate's
// site likelihood)
__device__ __forceinline__ void q_post(const QTop& t, const Coef& cf, int lv, double b0, double bA, double q,
                                       const Eps& ep, double* S) {
  // ('z': bA = 0 and s1 = 0)
  const double A = t.A * ep.s0, G = t.G * ep.s0;
  S[0] = lv == 0 ? 1.0 : cf.p1n * A * b0;
  S[1] = cf.mut * q * A * bA;
  S[2] = ep.s1 * t.A;
  S[3] = cf.pn * G * bA;
  S[4] = ep.s1 * t.G;
}

// outside state (a0, aX) at the node below a branch, on the scale of its
// inside mantissas; aX = 0 at 'z' nodes
__device__ __forceinline__ QTop q_node(const QTop& t, const Coef& cf, int lv, double q, const Eps& ep) {
  QTop a;
  const double A = t.A * ep.s0, G = t.G * ep.s0;
  a.A = cf.p1n * A;
  a.G = lv == 0 ? 0.0 : fma(cf.pn, G, cf.mut * q * A);
  return a;
}

// top of a child's branch from its parent's state (scaled by sc, the power
// of two the parent's vector was scaled by) and the sibling's edge values
__device__ __forceinline__ QTop q_top(const QTop& a, double sc, const Eps& ew) {
  QTop t;
  t.A = a.A * (sc * ew.e0);
  t.G = a.G * (sc * ew.eA);
  return t;
}

// inside of a node from its two children's edge values, and the power of two
// sc that it was scaled by; returns the label
__device__ __forceinline__ int q_combine(int la, int lb, const Eps& ea, const Eps& eb, double& B0, double& BA,
                                         int& E, double& scale) {
  const int lv = combine_label(la, lb);
  const double b0 = ea.e0 * eb.e0;
  const double bA = lv != 0 ? ea.eA * eb.eA : 0.0;
  const int sh = min(-exp_of(fmax(b0, bA)), 1000);
  const double sc = ldexp(1.0, sh);
  B0 = b0 * sc;
  BA = bA * sc;
  E = ea.e + eb.e - sh;
  scale = sc;
  return lv;
}

}  // namespace

// What a candidate's EM needs of one site and does not change: the moved
// subtrees' inside state and prior weights, labels and prior weights of u and
// v, the data outside v's branch over the likelihood before the move (top,
// with exponent x0), the part c of the likelihood free of v's branch, and the
// log-likelihood before the move.
struct QSite {
  double b0[3], bA[3], q[3];  // A, W, C
  double qU, qV, topA, topG, c, base;
  int lab[3], E[3], labU, labV, x0;
};

struct QCand {
  ChildRows r[3], rS;
  bool lf[3], lfS, top_root;
  Coef cs;
  const double2 *aP, *bP;
  const int32_t* bEP;
  const int16_t* labP;
  const double *pSP, *qsum, *site_llh;
  const int32_t* qoff;
  double phi;
};

__device__ __forceinline__ void q_load(const DevForest& F, const QCand& n, int k, QSite& x) {
  const int qo = row_at(n.qoff, (unsigned)k) - 1;
  const double qs = row_at(n.qsum, (unsigned)k);
  auto weight = [&](int lab) { return lab > 0 ? row_at(F.prior, (unsigned)(qo + lab)) : qs; };
  int code;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    load_child_rows(n.r[i], n.lf[i], k, n.phi, x.lab[i], x.b0[i], x.bA[i], x.E[i], code);
    x.q[i] = weight(x.lab[i]);
  }
  x.labU = combine_label(x.lab[0], x.lab[1]);
  x.labV = combine_label(x.labU, x.lab[2]);
  x.qU = weight(x.labU);
  x.qV = weight(x.labV);
  x.c = x.base = 0.0;
  if (n.top_root) {
    // the unedited ancestor
    x.topA = 1.0;
    x.topG = 0.0;
    x.x0 = 0;
    return;
  }
  int labS, ES;
  double b0S, bAS;
  load_child_rows(n.rS, n.lfS, k, n.phi, labS, b0S, bAS, ES, code);
  const Eps eS = edge(labS, b0S, bAS, ES, weight(labS), n.cs);
  const int lp = row_at(n.labP, (unsigned)k);
  const double2 ap = row_at(n.aP, (unsigned)k);
  const double b0p = row_at(n.bP, (unsigned)k).x;
  x.topA = (lp == 0 ? 1.0 / b0p : ap.x) * eS.e0;
  x.topG = lp == 0 ? 0.0 : ap.y * eS.eA;
  if (lp < 0) x.c = row_at(n.pSP, (unsigned)k);  // p silenced: free of v's branch
  x.x0 = eS.e - row_at(n.bEP, (unsigned)k);
  x.base = row_at(n.site_llh, (unsigned)k);
}

// One site's log-likelihood and posterior counts of the five branches.  Each
// branch's five counts go to emit(branch, S) as soon as they are formed (v,
// u, C, A, W), so that few are held at a time.
template <typename Emit>
__device__ __forceinline__ double q_eval(const QSite& x, const Coef (&cf)[5], Emit&& emit) {
  const Eps eA = edge(x.lab[0], x.b0[0], x.bA[0], x.E[0], x.q[0], cf[0]);
  const Eps eW = edge(x.lab[1], x.b0[1], x.bA[1], x.E[1], x.q[1], cf[1]);
  double b0u, bAu, b0v, bAv, scU, scV;
  int Eu, Ev;
  q_combine(x.lab[0], x.lab[1], eA, eW, b0u, bAu, Eu, scU);
  const Eps eU = edge(x.labU, b0u, bAu, Eu, x.qU, cf[2]);
  const Eps eC = edge(x.lab[2], x.b0[2], x.bA[2], x.E[2], x.q[2], cf[3]);
  q_combine(x.labU, x.lab[2], eU, eC, b0v, bAv, Ev, scV);
  const Eps eV = edge(x.labV, b0v, bAv, Ev, x.qV, cf[4]);
  // site likelihood L' of the candidate: L' / L = t1 2^xe + c
  const int xe = x.x0 + eV.e;
  const double t1 = fma(x.topA, eV.e0, x.topG * eV.eA);
  const int e1 = t1 != 0.0 ? xe + exp_of(t1) : kZeroTop;
  const int e = max(e1, x.c != 0.0 ? exp_of(x.c) : kZeroTop);
  const double Lm = ldexp(t1, min(xe - e, 1000)) + ldexp(x.c, min(-e, 1000));
  // from here on over L'
  const double iL = ldexp(rcp_normal(Lm), min(xe - e, 1000));
  const QTop tv{x.topA * iL, x.topG * iL};
  double S[5];
  // v's branch, then u and C below v, then A and W below u
  q_post(tv, cf[4], x.labV, b0v, bAv, x.qV, eV, S);
  emit(4, S);
  const QTop av = q_node(tv, cf[4], x.labV, x.qV, eV);
  const QTop tu = q_top(av, scV, eC);
  q_post(tu, cf[2], x.labU, b0u, bAu, x.qU, eU, S);
  emit(2, S);
  const QTop tc = q_top(av, scV, eU);
  q_post(tc, cf[3], x.lab[2], x.b0[2], x.bA[2], x.q[2], eC, S);
  emit(3, S);
  const QTop au = q_node(tu, cf[2], x.labU, x.qU, eU);
  q_post(q_top(au, scU, eW), cf[0], x.lab[0], x.b0[0], x.bA[0], x.q[0], eA, S);
  emit(0, S);
  q_post(q_top(au, scU, eA), cf[1], x.lab[1], x.b0[1], x.bA[1], x.q[1], eW, S);
  emit(1, S);
  return log(Lm) + (double)e * 0.69314718055994530942 + x.base;
}

// A block of NW wavefronts per candidate, a site a lane (more than 64 NW
// sites: in turns, loaded anew each EM step).  The sums over sites go through
// LDS once a step; then five lanes of the first wavefront solve the five
// branches side by side and form their coefficients, which a wavefront per
// candidate did one after the other in every lane (3,996 candidates on 2,000
// leaves x 200 sites: 790 us then, 270 now).  The coefficients of a step are
// wave-uniform and held in scalar registers.  Bound by latency: half of the
// wave cycles wait for the step's barriers, sums and solves, 37 % of the issue
// slots are used; three wavefronts a SIMD (168 registers) in place of two
// measured the same.
template <int NW>
__global__ void __launch_bounds__(64 * NW) k_quartet_em(DevForest F, const int32_t* __restrict__ qnodes,
                                                        const double* __restrict__ len_in,
                                                        const uint8_t* __restrict__ opt_mask,
                                                        const double* __restrict__ llh_const,
                                                        const double* __restrict__ nu_p,
                                                        const double* __restrict__ phi_p, int max_iter, double tol,
                                                        double* __restrict__ len_out, double* __restrict__ nll_out,
                                                        int32_t* __restrict__ iters_out) {
  // values 0 .. 24: counts of the branches in the order they are formed (v,
  // u, C, A, W); 25: the log-likelihood
  __shared__ double sh[NW][27];
  __shared__ double tot[25];
  __shared__ Coef scf[5];
  const int c = (int)blockIdx.x;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int p = uniform_load(qnodes + c * 5), sib = uniform_load(qnodes + c * 5 + 1);
  const int nd[3] = {uniform_load(qnodes + c * 5 + 2), uniform_load(qnodes + c * 5 + 3),
                     uniform_load(qnodes + c * 5 + 4)};
  const int t = F.tree_of[nd[0]];
  const int prob = F.tree_prob[t];
  const int K = F.tree_nsites[t];
  const int sb = F.tree_site_base[t];
  const double nu = nu_p[prob];
  const uint32_t opt = opt_mask[c];
  QCand n;
  n.phi = phi_p[prob];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    n.lf[i] = nd[i] < F.num_leaves;
    n.r[i] = child_rows(F, nd[i], n.lf[i]);
  }
  n.top_root = p < 0;
  n.qoff = F.site_qoff + sb;
  n.qsum = F.site_qsum + sb;
  n.site_llh = F.site_llh + sb;
  if (!n.top_root) {
    n.cs = F.coef[sib];
    n.lfS = sib < F.num_leaves;
    n.rS = child_rows(F, sib, n.lfS);
    const int64_t rp = F.row_off[p];
    n.aP = F.alpha + rp;
    n.labP = F.labels + rp;
    n.pSP = F.pS + rp;
    n.bP = F.beta + F.brow[p];
    n.bEP = F.bE + F.brow[p];
  }
  // lane j < 5 of the first wavefront owns branch j
  double d = tid < 5 ? len_in[c * 5 + tid] : 0.0;
  if (tid < 5) scf[tid] = branch_coef(d, nu);
  __syncthreads();
  QSite x{};  // (a lane without a site evaluates zeros, which count for nothing)
  double llh_prev = 0.0, llh = 0.0;
  int iters = max_iter + 1;
  for (int it = 0; it <= max_iter; ++it) {
    // wave-uniform: in scalar registers
    Coef cf[5];
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      cf[j].p1n = uniform_double(scf[j].p1n);
      cf[j].mut = uniform_double(scf[j].mut);
      cf[j].pn = uniform_double(scf[j].pn);
      cf[j].msil = uniform_double(scf[j].msil);
      cf[j].esil = __builtin_amdgcn_readfirstlane(scf[j].esil);
    }
    const int vi = sum12_value(lane);
    for (int k0 = 0; k0 < K; k0 += 64 * NW) {
      const int k = k0 + tid;
      const bool on = k < K;
      if (on && (it == 0 || K > 64 * NW)) q_load(F, n, k, x);
      // totals over the wavefront, a dozen values at a time, added to the
      // earlier turns'
      double v[12];
      int nv = 0, base = 0;
      auto put = [&](double s) {
        v[nv++] = on ? s : 0.0;
        if (nv < 12) return;
        const double y = wave_sum12(v);
        if (vi >= 0) {
          double* o = &sh[wave][base + vi];
          *o = k0 == 0 ? y : *o + y;
        }
        nv = 0;
        base += 12;
      };
      double ll = q_eval(x, cf, [&](int, const double(&S)[5]) {
#pragma unroll
        for (int m = 0; m < 5; ++m) put(S[m]);
      });
      const double s24 = seg_sum_last<64>(v[0]);
      ll = seg_sum_last<64>(on ? ll : 0.0);
      if (lane == 63) {
        sh[wave][24] = k0 == 0 ? s24 : sh[wave][24] + s24;
        sh[wave][25] = k0 == 0 ? ll : sh[wave][25] + ll;
      }
    }
    __syncthreads();
    double lsum = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) lsum += sh[w][25];
    llh = lsum + llh_const[c];
    // EM_solver.py:483-512: stop when the relative change is below tol, or
    // after max_iter M-steps (iteration count max_iter + 1)
    if (it > 0 && tol > 0.0 && fabs((llh - llh_prev) / llh_prev) < tol) {
      iters = it;
      break;
    }
    if (it == max_iter) break;
    llh_prev = llh;
    // M-step of the free branches (EM_solver.py:339-366 for one branch)
    if (wave == 0) {
      if (lane < 25) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) s += sh[w][lane];
        tot[lane] = s;
      }
      lds_wave_sync();
      if (lane < 5 && ((opt >> lane) & 1u)) {
        double sj[5];
#pragma unroll
        for (int m = 0; m < 5; ++m) sj[m] = tot[5 * (lane == 4 ? 0 : (lane == 2 ? 1 : (lane == 3 ? 2 : lane + 3))) + m];
        d = solve_branch(branch_obj(sj, (double)K, nu), F.dmin, F.dmax, d);
        scf[lane] = branch_coef(d, nu);
      }
    }
    __syncthreads();
  }
  if (tid < 5) len_out[c * 5 + tid] = d;
  if (tid == 0) {
    nll_out[c] = -llh;
    iters_out[c] = iters;
  }
}

// the wavefronts a candidate takes: one per 64 sites of the longest row, up
// to 8
void run_quartet_em(const DevForest& F, int ncand, const int32_t* qnodes, const double* len_in,
                    const uint8_t* opt_mask, const double* llh_const, const double* nu, const double* phi,
                    int max_iter, double tol, double* len_out, double* nll_out, int32_t* iters_out, hipStream_t s) {
  if (ncand <= 0) return;
  const int waves = F.chunk_w < 64 ? 1 : F.max_chunks;
#define LAML_QUARTET(NW)                                                                                       \
  hipLaunchKernelGGL(k_quartet_em<NW>, dim3(ncand), dim3(64 * NW), 0, s, F, qnodes, len_in, opt_mask, llh_const, \
                     nu, phi, max_iter, tol, len_out, nll_out, iters_out)
  if (waves <= 1) LAML_QUARTET(1);
  else if (waves == 2) LAML_QUARTET(2);
  else if (waves <= 4) LAML_QUARTET(4);
  else LAML_QUARTET(8);
#undef LAML_QUARTET
}

// ---------------------------------------------------------------------------
// LDS passes: a block keeps the state of every internal node of one tree at
// its sites in LDS and runs the pass (inside levels, root, outside levels)
// with barriers between levels.  A level then costs an LDS round trip and the
// arithmetic (0.4 us inside, 0.8 us outside for narrow levels) where rows in
// global memory cost a store, a barrier and a load through the L2, or a
// launch.
//
// A thread takes two neighbouring sites of a node, kLdsCells (node, site)
// cells a step.  What they need besides the LDS state (where the children's
// vectors are, label flags, prior weights, branch coefficients) does not
// depend on the level below, is laid out in the order the threads read it, and
// is loaded one step ahead, across the barrier, into one of two register sets
// used in turn: copying a set would wait for it.  A leaf child's vector is one
// of four constant cells, so that leaves and internal children take the same
// path.  The outside pass writes a child's state over its inside vector (its
// last use is the parent's step) and a node's partial counts over its own
// state, so that no store to global memory is pending when a step waits for
// its loads.  Wide levels are bound by the CU's L1 and instruction issue
// (hence two sites a thread, which share coefficients and sums, and silencing
// terms only in wavefronts that hold a '?' cell), narrow ones by latency.
//
// Eight sites of a node share a partial-count slot.  Their four lanes lie in
// the four 16-lane rows (lane 16 r + c: sites 2 r and 2 r + 1 of group c), so
// that the eleven sums over them take two halving row swaps.
// ---------------------------------------------------------------------------
constexpr int kLdsThreads = 512;
constexpr int kLdsCells = 2 * kLdsThreads;  // cells a step
constexpr int kLdsWave = 128;               // of them a wavefront's
// the 8 x 16 bytes of state of the sites that share a slot hold its eleven sums
constexpr int kLdsR = kLdsSlotSites;

// flags of a cell: label kinds of the node and its children, kinds of child
enum : uint32_t {
  kLdsUz = 1,                       // the node is 'z' (label 0)
  kLdsZ0 = 2, kLdsZ1 = 4,           // child 0 / 1 is 'z'
  kLdsQ0 = 8, kLdsQ1 = 16,          // child 0 / 1 is '?'
  kLdsLeaf0 = 32, kLdsLeaf1 = 64,
  kLdsDrop0 = 128, kLdsDrop1 = 256  // child 0 / 1 is a leaf with a missing entry
};                                  // (the upper 16 bits: the cell's own place)
// cells of the constant leaf vectors: unedited, edited, missing, none
// (explicitly silenced entries, and the sites past the tree's); a cell that
// is written and never read
constexpr int kLdsLeafCells = 8, kLdsNoCell = 4;

// Where cell c (node-major) lies: the sites of a group of eight in an order
// that depends on the group, so that the lanes of a row (the same site of 16
// groups) fall into different banks.
__device__ __forceinline__ int lds_place(int c) {
  return (c + kLdsLeafCells) ^ (((c >> 4) & 3) << 1) ^ ((c >> 6) & 1);
}
// the first cell of thread t's pair, of a step's cells
__device__ __forceinline__ int lds_pair(unsigned t) {
  return (int)((t >> 6) * kLdsWave + 8u * (t & 15u) + 2u * ((t >> 4) & 3u));
}

// every LDS access of the block so far is done; global loads and stores stay
// in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct LdsItem {
  uint4 w;        // per cell: places of the children's vectors; flags and its own place
  double2 q[2];   // per cell: prior weights of the children
  LdsCoef cf;
  bool on;        // whether the lane has cells
};

// one block's tree
struct LdsCtx {
  int sb, nint, H, K;
  unsigned magic;          // floor(i / sb) = umulhi(i, magic) for i < 2^20
  const uint4* w;
  const double4* q;
  const LdsRec* rec;
  const LdsCoef* lcoef;
  double phi;
  double2* st;             // LDS: the cells' vectors
  int* sE;                 // LDS: their exponents
  int2* lvl;               // LDS: first local number and first table entry of level h (level H: the end)
  int2 lreg;               // lane i of a wavefront: lvl[i]
  double* rpart;           // LDS: the stem's sums, 3 per kLdsR sites
};

// element i (wave-uniform) of an array that no kernel writes while it runs
template <typename T>
__device__ __forceinline__ T uniform_at(const T* p, int i) {
  return uniform_load(p + __builtin_amdgcn_readfirstlane(i));
}

// the constant leaf vectors (as leaf_beta)
__device__ __forceinline__ void lds_leaves(LdsCtx& x, double phi) {
  const int t = (int)threadIdx.x;
  x.phi = phi;
  if (t < kLdsLeafCells) {
    x.st[t] = make_double2(t == 0 ? 1.0 - phi : (t == 2 ? phi : 0.0), t == 1 ? 1.0 - phi : (t == 2 ? phi : 0.0));
    x.sE[t] = 0;
  }
}

__device__ __forceinline__ LdsCtx lds_ctx(const DevForest& F, const LdsPlan& L, const TreeWalk& TW, const LdsBlk& B,
                                          double phi, char* lds) {
  LdsCtx x;
  x.sb = B.sb;
  x.nint = B.nint;
  x.K = uniform_at(F.tree_nsites, B.tree);
  const int lb = uniform_at(TW.lvl_base, B.tree);
  x.H = uniform_at(TW.lvl_base, B.tree + 1) - lb;
  const int ib = uniform_at(L.int_base, B.tree);
  x.magic = 0xffffffffu / (unsigned)B.sb + 1u;
  x.w = L.w + B.tab;
  x.q = L.q + B.tab;
  x.rec = L.rec + ib;
  x.lcoef = L.lcoef + ib;
  const int cells = B.nint * B.sb + kLdsLeafCells;
  x.st = reinterpret_cast<double2*>(lds);
  x.rpart = reinterpret_cast<double*>(x.st + cells);
  x.lvl = reinterpret_cast<int2*>(x.rpart + 3 * (B.sb / kLdsR));
  x.sE = reinterpret_cast<int*>(x.lvl + x.H + 1);
  lds_leaves(x, phi);
  for (int h = (int)threadIdx.x; h < x.H; h += kLdsThreads) x.lvl[h + 1] = L.lvl_off[lb + h];
  lds_barrier();
  x.lreg = x.lvl[min((int)(threadIdx.x & 63), x.H)];
  return x;
}

// The uniform walk over a tree's steps: level h, its cells from i0 on, n in
// all; up or down the levels.
struct LdsStep {
  int h, i0, n, l0, e0;  // the level's first local number and table entry
};
__device__ __forceinline__ void lds_level(const LdsCtx& x, int h, LdsStep& p) {
  p.h = h;
  p.i0 = 0;
  int l1;
  if (h < 63) {
    p.l0 = __builtin_amdgcn_readlane(x.lreg.x, h);
    p.e0 = __builtin_amdgcn_readlane(x.lreg.y, h);
    l1 = __builtin_amdgcn_readlane(x.lreg.x, h + 1);
  } else {
    p.l0 = __builtin_amdgcn_readfirstlane(x.lvl[h].x);
    p.e0 = __builtin_amdgcn_readfirstlane(x.lvl[h].y);
    l1 = __builtin_amdgcn_readfirstlane(x.lvl[h + 1].x);
  }
  p.n = (l1 - p.l0) * x.sb;
}
// the step after p among levels 1 .. H - 1 (n = 0: none), of `width` cells;
// whether it starts a level
__device__ __forceinline__ bool lds_next(const LdsCtx& x, int dir, int width, const LdsStep& p, LdsStep& o) {
  o = p;
  o.i0 += width;
  if (o.i0 < p.n) return false;
  o.h = p.h + dir;
  o.n = 0;
  if (o.h >= 1 && o.h < x.H) lds_level(x, o.h, o);
  return true;
}

// The wavefront's cells of step p, t the thread's number in the step: every
// lane loads (lanes past the level's cells its last one), so that the number
// of loads in flight is known.
__device__ __forceinline__ void lds_fetch(const LdsCtx& x, const LdsStep& p, unsigned t, LdsItem& it) {
  const int i = p.i0 + lds_pair(t);
  const unsigned l = (unsigned)p.l0 + __umulhi((unsigned)min(i, p.n - 1), x.magic);
  it.on = i < p.n;
  const unsigned e = (unsigned)(p.e0 + p.i0 / 2) + t;
  it.w = row_at(x.w, e);
  const double4 q = row_at(x.q, e);
  it.q[0] = make_double2(q.x, q.y);
  it.q[1] = make_double2(q.z, q.w);
  it.cf = row_at(x.lcoef, l);
}
__device__ __forceinline__ bool lds_any_q(const LdsItem& it) {
  return __any(it.on && ((it.w.y | it.w.w) & (kLdsQ0 | kLdsQ1)));
}

// What a thread's two cells read from LDS: their children's vectors, loaded
// before anything is stored (a load may not pass a store).
struct LdsIn {
  double2 b[2][2];
  int E[2][2], pl[2][2];
};
template <bool kE>
__device__ __forceinline__ void lds_load(const LdsCtx& x, const LdsItem& it, LdsIn& o) {
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint32_t w = c == 0 ? it.w.x : it.w.z;
    o.pl[c][0] = w & 0xffffu;
    o.pl[c][1] = w >> 16;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      o.b[c][i] = x.st[o.pl[c][i]];
      o.E[c][i] = kE ? x.sE[o.pl[c][i]] : 0;
    }
  }
}
// Edge values of child i of a cell (edge() with the label kinds from the
// flags: the inside vector is 0 where edge() selects 0; kQ false: no '?' cell
// in the wavefront, s0 = 1 and s1 = 0).
template <bool kQ>
__device__ __forceinline__ Eps lds_edge(const LdsCoef& c, int i, uint32_t fl, const double2& b, int E, double mq) {
#pragma clang fp contract(off)
  Eps r;
  r.e0 = fma(mq, b.y, c.p1n[i] * b.x);
  r.eA = c.pn[i] * b.y;
  r.e = E;
  r.s0 = 1.0;
  r.s1 = 0.0;
  if (kQ) {
    const int es = fl & (i == 0 ? kLdsQ0 : kLdsQ1) ? c.esil[i] : kZeroTop;
    r.e = max(E, es);
    r.s0 = ldexp(1.0, E - r.e);
    r.s1 = ldexp(c.msil[i], es - r.e);
    r.e0 = fma(r.e0, r.s0, r.s1);
    r.eA = fma(r.eA, r.s0, r.s1);
  }
  return r;
}

template <bool kQ>
__device__ __forceinline__ void lds_inside_cells(const LdsCtx& x, const LdsItem& it) {
#pragma clang fp contract(off)
  LdsIn in;
  lds_load<true>(x, it, in);
  double2 o[2];
  int E[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint32_t fl = c == 0 ? it.w.y : it.w.w;
    const Eps e0 = lds_edge<kQ>(it.cf, 0, fl, in.b[c][0], in.E[c][0], it.cf.mut[0] * it.q[c].x);
    const Eps e1 = lds_edge<kQ>(it.cf, 1, fl, in.b[c][1], in.E[c][1], it.cf.mut[1] * it.q[c].y);
    const double B0 = e0.e0 * e1.e0;
    const double BA = fl & kLdsUz ? 0.0 : e0.eA * e1.eA;
    const int sh = min(-exp_of(fmax(B0, BA)), 1000);
    o[c] = make_double2(ldexp(B0, sh), ldexp(BA, sh));
    E[c] = e0.e + e1.e - sh;
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int pl = (c == 0 ? it.w.y : it.w.w) >> 16;
    x.st[pl] = o[c];
    x.sE[pl] = E[c];
  }
}

// (as cond_post; products that do not need the node's own state are formed
// before it is known, which shortens the chain from a node to its children)
template <bool kQ>
__device__ __forceinline__ void lds_outside_cells(const LdsCtx& x, const LdsItem& it, double (&v)[12]) {
#pragma clang fp contract(off)
  LdsIn in;
  const double2 a[2] = {x.st[it.w.y >> 16], x.st[it.w.w >> 16]};
  lds_load<kQ>(x, it, in);
  double2 o[2][2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint32_t fl = c == 0 ? it.w.y : it.w.w;
    const double mq[2] = {it.cf.mut[0] * it.q[c].x, it.cf.mut[1] * it.q[c].y};
    const Eps ep[2] = {lds_edge<kQ>(it.cf, 0, fl, in.b[c][0], in.E[c][0], mq[0]),
                       lds_edge<kQ>(it.cf, 1, fl, in.b[c][1], in.E[c][1], mq[1])};
    const bool z = fl & kLdsUz;
    const double B0 = ep[0].e0 * ep[1].e0;
    const double BA = z ? 0.0 : ep[0].eA * ep[1].eA;
    const int sh = min(-exp_of(fmax(B0, BA)), 1000);
    const double f0 = z ? rcp_normal(ldexp(B0, sh)) : a[c].x;
    const double fX = z ? 0.0 : a[c].y;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const Eps& ew = ep[1 - i];
      double k0 = ldexp(ew.e0, sh), kX = ldexp(ew.eA, sh);
      if (kQ) {
        v[5 * i + 2] = fma(f0, ep[i].s1 * k0, v[5 * i + 2]);
        v[5 * i + 4] = fma(fX, ep[i].s1 * kX, v[5 * i + 4]);
        k0 *= ep[i].s0;
        kX *= ep[i].s0;
      }
      const double a0 = f0 * (it.cf.p1n[i] * k0);
      const double m = f0 * (mq[i] * k0);
      const double pg = fX * (it.cf.pn[i] * kX);
      const double aX = pg + m;
      const bool cz = fl & (i == 0 ? kLdsZ0 : kLdsZ1);
      v[5 * i] = fma(cz ? 1.0 : a0, cz ? 1.0 : in.b[c][i].x, v[5 * i]);
      v[5 * i + 1] = fma(m, in.b[c][i].y, v[5 * i + 1]);
      v[5 * i + 3] = fma(pg, in.b[c][i].y, v[5 * i + 3]);
      if (kQ) v[10] = fma(fl & (i == 0 ? kLdsDrop0 : kLdsDrop1) ? x.phi : 0.0, a0 + aX, v[10]);
      o[c][i] = make_double2(a0, aX);
    }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint32_t fl = c == 0 ? it.w.y : it.w.w;
#pragma unroll
    for (int i = 0; i < 2; ++i)  // (a leaf's state goes to a cell that nothing reads)
      x.st[fl & (i == 0 ? kLdsLeaf0 : kLdsLeaf1) ? kLdsNoCell : in.pl[c][i]] = o[c][i];
  }
}

template <int dir>
__device__ __forceinline__ void lds_cells(const LdsCtx& x, const LdsItem& it) {
  const bool any_q = lds_any_q(it);
  if (dir > 0) {
    if (!it.on) return;
    if (any_q) lds_inside_cells<true>(x, it);
    else lds_inside_cells<false>(x, it);
    return;
  }
  double v[12];
#pragma unroll
  for (int m = 0; m < 12; ++m) v[m] = 0.0;
  if (it.on) {
    if (any_q) lds_outside_cells<true>(x, it, v);
    else lds_outside_cells<false>(x, it, v);
  }
  // sums over the lanes of the group: row r ends with values 3 r .. 3 r + 2
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    swap32(v[j], v[j + 6]);
    v[j] += v[j + 6];
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    swap16(v[j], v[j + 3]);
    v[j] += v[j + 3];
  }
  if (it.on) {
    // the group's cells lie in one aligned run of 8 places
    double* c = reinterpret_cast<double*>(x.st + ((it.w.y >> 16) & ~7u)) + 3 * ((threadIdx.x >> 4) & 3);
    c[0] = v[0];
    c[1] = v[1];
    c[2] = v[2];
  }
}

// One step on the cells in A while the next step's load into B.  Whether the
// wavefront has cells at either step is uniform over it, and each case has
// code of its own: where paths with and without the loads of B join, the
// compiler would wait for B with A.
template <int dir>
__device__ __forceinline__ bool lds_turn(const LdsCtx& x, const LdsStep& p, LdsStep& o, int wave0, LdsItem& A,
                                         LdsItem& B) {
  const bool lvl = lds_next(x, dir, kLdsCells, p, o);
  if (dir > 0 && o.n <= kLdsWave) o.n = 0;  // the narrow levels follow
  const bool cur = p.i0 + wave0 < p.n;
  if (o.i0 + wave0 < o.n) {
    lds_fetch(x, o, threadIdx.x, B);
    if (cur) lds_cells<dir>(x, A);
  } else if (cur) {
    lds_cells<dir>(x, A);
  }
  if (lvl) lds_barrier();
  return o.n != 0;
}
// the same for the levels that one wavefront holds (it runs them without
// barriers: its LDS accesses are in order)
template <int dir>
__device__ __forceinline__ bool lds_turn1(const LdsCtx& x, const LdsStep& p, LdsStep& o, LdsItem& A, LdsItem& B) {
  lds_next(x, dir, kLdsWave, p, o);
  if (dir < 0 && o.n > kLdsWave) o.n = 0;  // the wide levels follow
  if (o.n != 0) {
    lds_fetch(x, o, threadIdx.x & 63u, B);
    lds_cells<dir>(x, A);
  } else {
    lds_cells<dir>(x, A);
  }
  return o.n != 0;
}

// The levels from h on, bottom up (dir 1) or top down (dir -1), two steps a
// turn of the loop (one register set each): the wide ones by the block, those
// of at most kLdsWave cells by the first wavefront (levels only get narrower
// upwards).
template <int dir>
__device__ __forceinline__ void lds_wide(const LdsCtx& x, int h) {
  LdsStep p, o;
  LdsItem A, B;
  const int wave0 = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * kLdsWave;
  lds_level(x, h, p);
  if (p.n <= kLdsWave) return;
  if (wave0 < p.n) lds_fetch(x, p, threadIdx.x, A);
  for (;;) {
    if (!lds_turn<dir>(x, p, o, wave0, A, B)) break;
    if (!lds_turn<dir>(x, o, p, wave0, B, A)) break;
  }
}
template <int dir>
__device__ __forceinline__ void lds_narrow(const LdsCtx& x, int h) {
  LdsStep p, o;
  LdsItem A, B;
  lds_level(x, h, p);
  lds_fetch(x, p, threadIdx.x & 63u, A);
  for (;;) {
    if (!lds_turn1<dir>(x, p, o, A, B)) break;
    if (!lds_turn1<dir>(x, o, p, B, A)) break;
  }
}
// the first narrow level (H: none)
__device__ __forceinline__ int lds_first_narrow(const LdsCtx& x) {
  int h = 1;
  for (; h < x.H; ++h) {
    LdsStep p;
    lds_level(x, h, p);
    if (p.n <= kLdsWave) break;
  }
  return h;
}

// Root step of the block's tree (as root_chunk): site log-likelihoods, the
// root's state, the stem's counts.  Returns the log-likelihood of the
// thread's site (0: none).
__device__ __forceinline__ double lds_root(const DevForest& F, const LdsCtx& x, int t, double* site_llh_out) {
  double sl = 0.0;
  const int s = (int)threadIdx.x;
  if (s < x.sb) {
    const int r = uniform_at(F.tree_root, t);
    const int pl = lds_place((x.nint - 1) * x.sb + s);
    const bool real = s < x.K;
    const int kc = min(s, x.K - 1);
    const int sk = uniform_at(F.tree_site_base, t) + kc;
    const int lab = F.labels[F.row_off[r] + kc];
    const double q = lab > 0 ? F.prior[F.site_qoff[sk] - 1 + lab] : F.site_qsum[sk];
    const double2 b = x.st[pl];
    const Coef cf = F.coef[r];
    const Eps er = edge(lab, b.x, b.y, x.sE[pl], q, cf);
    const int ex = exp_of(er.e0);
    const double Lm = ldexp(er.e0, -ex);
    // the sites past the tree's carry zeros
    const double A = real ? 1.0 / er.e0 : 0.0;
    const double a0 = cf.p1n * A * er.s0;
    const double m = cf.mut * q * A * er.s0;
    const double sil = lab < 0 ? er.s1 * A : 0.0;
    x.st[pl] = make_double2(a0, m);
    double acc[3] = {lab == 0 ? 1.0 : a0 * b.x, lab != 0 ? m * b.y : 0.0, sil};
    if (real) {
      sl = log(Lm) + (double)(er.e + ex) * 0.69314718055994530942;
      F.site_llh[sk] = sl;
      if (site_llh_out) site_llh_out[sk] = sl;
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      acc[j] = seg_sum_last<kLdsR>(real ? acc[j] : 0.0);
      if ((s & (kLdsR - 1)) == kLdsR - 1) x.rpart[3 * (s / kLdsR) + j] = acc[j];
    }
  }
  lds_barrier();
  return sl;
}

// The block's passes: inside, root() (lds_root), outside when `out`; hn: the
// first narrow level.
template <typename Root>
__device__ __forceinline__ double lds_pass(const LdsCtx& x, int hn, bool out, Root&& root) {
  const bool first = __builtin_amdgcn_readfirstlane((int)threadIdx.x) < 64;
  lds_wide<1>(x, 1);
  if (hn < x.H && first) lds_narrow<1>(x, hn);
  lds_barrier();
  const double sl = root();
  if (!out) return sl;
  if (hn < x.H && first) lds_narrow<-1>(x, x.H - 1);
  lds_barrier();
  if (hn > 1) lds_wide<-1>(x, hn - 1);
  return sl;
}

// Sums the block's partial counts over its sites, in site order, and leaves
// them in the nodes' first slots: 16 threads a node, thread m its value m
// (counts 0..4 of both child branches, the dropout sum).
__device__ __forceinline__ double* lds_slot(const LdsCtx& x, int l, int g) {
  return reinterpret_cast<double*>(x.st + (kLdsLeafCells + l * x.sb + kLdsR * g));
}
__device__ __forceinline__ void lds_fold(const LdsCtx& x) {
  const int G = x.sb / kLdsR;
  const int m = (int)threadIdx.x & 15;
  for (int l = (int)threadIdx.x >> 4; l < x.nint; l += kLdsThreads / 16) {
    if (m > 10) continue;
    double s = lds_slot(x, l, 0)[m];
    for (int g = 1; g < G; ++g) s += lds_slot(x, l, g)[m];
    lds_slot(x, l, 0)[m] = s;
  }
  if (threadIdx.x < 3)
    for (int g = 1; g < G; ++g) x.rpart[threadIdx.x] += x.rpart[3 * g + threadIdx.x];
  lds_barrier();
}
// branch r of the block's tree: child r & 1 of internal node r / 2, the stem last
__device__ __forceinline__ int lds_branch_node(const DevForest& F, const LdsCtx& x, int t, int r) {
  if (r == 2 * x.nint) return F.tree_root[t];
  return r & 1 ? x.rec[r >> 1].g1 : x.rec[r >> 1].g0;
}
__device__ __forceinline__ void lds_branch_counts(const LdsCtx& x, int r, double (&s)[5]) {
  const bool stem = r == 2 * x.nint;
  const double* c = stem ? x.rpart : lds_slot(x, r >> 1, 0) + 5 * (r & 1);
#pragma unroll
  for (int m = 0; m < 5; ++m) s[m] = stem && m > 2 ? 0.0 : c[m];
}
// the folded counts into F's partials
__device__ __forceinline__ void lds_flush(const DevForest& F, const LdsCtx& x, int t) {
  for (int r = (int)threadIdx.x; r <= 2 * x.nint; r += kLdsThreads) {
    double s[5];
    lds_branch_counts(x, r, s);
    double* c = F.cpart + lds_branch_node(F, x, t, r) * F.cp_v;
#pragma unroll
    for (int m = 0; m < 5; ++m) c[m] = s[m];
    if (r < 2 * x.nint && !(r & 1)) F.rt_part[x.rec[r >> 1].v * F.rt_v] = lds_slot(x, r >> 1, 0)[10];
  }
}

// coefficients of branch r of the tree with records from ib on
__device__ __forceinline__ void lds_set_coef(const LdsPlan& L, int ib, int r, const Coef& c) {
  LdsCoef* o = L.lcoef + ib + (r >> 1);
  const int i = r & 1;
  o->p1n[i] = c.p1n;
  o->mut[i] = c.mut;
  o->pn[i] = c.pn;
  o->msil[i] = c.msil;
  o->esil[i] = c.msil != 0.0 ? c.esil : kZeroTop;
}

// sums of kN values over the block's threads (sh: kN kLdsThreads / 64 doubles, free again after the next barrier)
template <int kN>
__device__ __forceinline__ void lds_sum(double (&v)[kN], double* sh) {
  constexpr int kW = kLdsThreads / 64;
#pragma unroll
  for (int j = 0; j < kN; ++j) {
    v[j] = seg_sum_last<64>(v[j]);
    if ((threadIdx.x & 63) == 63) sh[kN * (threadIdx.x >> 6) + j] = v[j];
  }
  lds_barrier();
#pragma unroll
  for (int j = 0; j < kN; ++j) {
    v[j] = 0.0;
#pragma unroll
    for (int i = 0; i < kW; ++i) v[j] += sh[kN * i + j];
  }
}

// Whole problems of one tree, a block each: likelihood, outside pass (the
// inside pass again first), or the EM loop, for problems of at most
// kPbMaxSites sites whose state fits LDS.  The
// loop needs no launch, no host and no other block between EM steps.  A
// thread keeps to the same branches throughout; the M-step reads their counts
// from LDS.  One 250 x 30 problem: 43 us an EM step (inside 16, outside 19,
// M-step 8), 101 us in the general passes' 13 launches; 200 trees of 20-200
// leaves x 20 sites: 51 us, 187 us; one likelihood of 250 x 30: 23 us, 35 us.
struct PbArgs {
  DevForest F;
  LdsPlan L;
  TreeWalk TW;
  double *d, *nu, *phi, *nll, *site_llh_out;
  int32_t* iters_out;
  EmState em;
  int max_steps, max_iter;
  double tol;
  int what;
  GradOut grad;
};
// The kernel's arguments, read where they are used: from an address that the
// compiler cannot tell from the last one, so that it loads again instead of
// keeping some 200 scalar registers' worth of pointers alive (spilled to
// vector lanes) across the passes.
__device__ __forceinline__ const PbArgs& pb_args() {
  uintptr_t p = (uintptr_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const PbArgs*)(const __attribute__((address_space(4))) PbArgs*)p;
}
__global__ void __launch_bounds__(kLdsThreads) k_problem(PbArgs) {
  extern __shared__ __align__(16) char lds[];
  __shared__ double sh[2][6 * (kLdsThreads / 64)];
  const int p = (int)blockIdx.x;
  const int t = p;  // one tree a problem
  const int what = pb_args().what;
  int step = 0;
  double pre = 0.0, nv, pv;
  LdsCtx x;
  {
    const PbArgs& A = pb_args();
    if (A.em.done && A.em.done[p]) return;
    if (what & kPbEm) {
      step = A.em.step[p];
      pre = A.em.pre[p];
    }
    nv = A.nu ? A.nu[p] : 0.0;
    pv = A.phi[p];
    x = lds_ctx(A.F, A.L, A.TW, uniform_at(A.L.blk, p), pv, lds);
  }
  const int hn = lds_first_narrow(x);
  const int nbr = 2 * x.nint + 1;
  for (int it = 0; it < pb_args().max_steps; ++it) {
    {
      const PbArgs& A = pb_args();
      const DevForest& F = A.F;
      const int ib = uniform_at(A.L.int_base, t);
      for (int r = (int)threadIdx.x; r < nbr; r += kLdsThreads) {
        const int v = lds_branch_node(F, x, t, r);
        Coef c;
        if (what & kPbCoef) {
          c = branch_coef(A.d[v], nv);
          F.coef[v] = c;
        } else {
          c = F.coef[v];  // (those of the last call, whichever kernels ran it)
        }
        if (r < nbr - 1) lds_set_coef(A.L, ib, r, c);
      }
      __syncthreads();
    }
    const bool out = (what & kPbOut) && !((what & kPbEm) && step == pb_args().max_iter);
    double lsum[1] = {lds_pass(x, hn, out, [&] { return lds_root(pb_args().F, x, t, pb_args().site_llh_out); })};
    lds_sum<1>(lsum, sh[0]);
    const double llh = lsum[0];
    if (out) lds_fold(x);
    const PbArgs& A = pb_args();
    const DevForest& F = A.F;
    if (!(what & kPbEm)) {
      if (threadIdx.x == 0 && A.nll) A.nll[p] = -llh;
      if (what & kPbGrad) {
        double g[2] = {0.0, 0.0};  // dlogL/dnu, the dropout sum
        for (int r = (int)threadIdx.x; r < nbr; r += kLdsThreads) {
          const int v = lds_branch_node(F, x, t, r);
          const double dv = A.d[v];
          double s[5];
          lds_branch_counts(x, r, s);
          A.grad.d[v] = -grad_length(s, dv, nv);
          g[0] -= dv * (s[0] + s[1] + s[3]);
          g[0] += grad_nu_part(s[2] + s[4], dv, nv);
          if (r < nbr - 1 && !(r & 1)) g[1] += lds_slot(x, r >> 1, 0)[10];
        }
        lds_sum<2>(g, sh[1]);
        if (threadIdx.x == 0) {
          A.grad.nu[p] = -g[0];
          A.grad.phi[p] = grad_phi_of(F.prob_nobs_phi[p], g[1], pv);
        }
      } else if (out) {
        lds_flush(F, x, t);
      }
      return;
    }
    const EmState& em = A.em;
    // bookkeeping of the EM loop (as k_llh; every thread decides alike)
    const bool conv = step > 0 && A.tol > 0.0 && fabs((llh - pre) / pre) < A.tol;
    const bool stop = conv || step >= A.max_iter;
    if (threadIdx.x == 0) {
      A.nll[p] = -llh;
      if (em.trace) em.trace[(int64_t)step * F.num_problems + p] = -llh;
      if (!conv) em.pre[p] = llh;
      em.step[p] = step + 1;
      if (stop) {
        const int n = conv ? step : A.max_iter + 1;
        em.done[p] = 1;
        em.iters[p] = n;
        A.iters_out[p] = n;
      }
    }
    if (stop) return;
    pre = llh;
    ++step;
    const uint32_t flags = uniform_at(F.prob_flags, p);
    const bool opt_nu = (flags & 2u) && uniform_at(F.prob_nfree, p) > 0;
    const double K = (double)x.K;
    // M-step: branch lengths (as k_branch), the dropout sum on the way
    double a0 = 0.0, b0 = 0.0, d0 = 0.0;  // the thread's first branch, as nu_a, nu_b, nu_d
    double rt = 0.0, bad = 0.0;
    for (int r = (int)threadIdx.x; r < nbr; r += kLdsThreads) {
      const int v = lds_branch_node(F, x, t, r);
      double s[5];
      lds_branch_counts(x, r, s);
      if (r < nbr - 1 && !(r & 1)) rt += lds_slot(x, r >> 1, 0)[10];
      double dn = A.d[v], na = 0.0, nb = 0.0;
      if (F.free_branch[v]) {
        dn = branch_length(F, s, K, nv, dn, na, nb);
        if (!isfinite(dn)) bad = 1.0;
        A.d[v] = dn;
      }
      if (r == (int)threadIdx.x) {
        a0 = na;
        b0 = nb;
        d0 = dn;
      } else {
        F.nu_a[F.node_pos[v]] = na;
        F.nu_b[F.node_pos[v]] = nb;
        F.nu_d[F.node_pos[v]] = dn;
      }
    }
    // phi, then nu (as k_nu_finish)
    double xx = nu_start(nv), lo = 0.0, hi = 2.0;
    bool fin = !opt_nu;
    int evals = 0;
    for (; evals == 0 || (!fin && evals < kNuMaxEvals); ++evals) {
      NuSum n{0.0, 0.0, 0.0, 0.0};
      if (opt_nu) {
        nu_term(a0, b0, d0, xx, n);
        for (int r = (int)threadIdx.x + kLdsThreads; r < nbr; r += kLdsThreads) {
          const int pos = F.node_pos[lds_branch_node(F, x, t, r)];
          nu_term(F.nu_a[pos], F.nu_b[pos], F.nu_d[pos], xx, n);
        }
      }
      double* const s = sh[1 - (evals & 1)];
      if (evals == 0) {
        double v[6] = {n.g, n.g1, n.g2, n.g3, rt, bad};
        lds_sum<6>(v, s);
        n = NuSum{v[0], v[1], v[2], v[3]};
        rt = v[4];
        bad = v[5];
        if (flags & 1u) {
          pv = rt / (F.prob_nobs[p] + rt);
          if (fabs(pv) < F.prob_phimin[p]) pv = 0.0;
        }
        if (!opt_nu) break;
      } else {
        double v[4] = {n.g, n.g1, n.g2, n.g3};
        lds_sum<4>(v, s);
        n = NuSum{v[0], v[1], v[2], v[3]};
      }
      double xn;
      fin = nu_step(xx, n, lo, hi, xn);
      xx = xn;
    }
    if (opt_nu) nv = xx;
    if (threadIdx.x == 0) {
      A.phi[p] = pv;
      A.nu[p] = nv;
      F.mstep_status[p] = (bad != 0.0 ? 1 : 0) | (fin ? 0 : 2);
    }
    lds_leaves(x, pv);
  }
}

// The cell tables of the blocks (blockIdx.y), a thread per pair of cells.
__global__ void __launch_bounds__(256) k_lds_tables(DevForest F, LdsPlan L, TreeWalk TW) {
  const LdsBlk B = L.blk[blockIdx.y];
  const LdsRec* recs = L.rec + L.int_base[B.tree];
  const int K = F.tree_nsites[B.tree], sb0 = F.tree_site_base[B.tree];
  const int lb = TW.lvl_base[B.tree], H = TW.lvl_base[B.tree + 1] - lb;
  for (int h = 1; h < H; ++h) {
    const int l0 = L.lvl_off[lb + h - 1].x, e0 = L.lvl_off[lb + h - 1].y;
    const int n = (L.lvl_off[lb + h].x - l0) * B.sb, ne = L.lvl_off[lb + h].y - e0;
    for (int e = (int)(blockIdx.x * 256 + threadIdx.x); e < ne; e += (int)gridDim.x * 256) {
      uint32_t w[4];
      double q[4];
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const int i = lds_pair((unsigned)e) + c2;
        uint32_t pl[2] = {3, 3}, fl = kLdsLeaf0 | kLdsLeaf1;
        q[2 * c2] = q[2 * c2 + 1] = 0.0;
        const int j = l0 + i / B.sb, s = i % B.sb, k = s;
        if (i < n) {
          const LdsRec r = recs[j];
          int lab[2] = {0, 0};
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const int g = c == 0 ? r.g0 : r.g1, l = c == 0 ? r.l0 : r.l1;
            if (l >= 0) {
              pl[c] = (uint32_t)lds_place(l * B.sb + s);
              fl &= ~(c == 0 ? kLdsLeaf0 : kLdsLeaf1);
            }
            if (k >= K) continue;
            const int code = l < 0 ? F.codes[F.row_off[g] + k] : F.labels[F.row_off[g] + k];
            lab[c] = l < 0 ? code_label(code) : code;
            if (l < 0) {
              pl[c] = code == 0 ? 0 : (code > 0 ? 1 : (code == -1 ? 2 : 3));
              if (code == -1) fl |= c == 0 ? kLdsDrop0 : kLdsDrop1;
            }
            if (lab[c] == 0) fl |= c == 0 ? kLdsZ0 : kLdsZ1;
            if (lab[c] < 0) fl |= c == 0 ? kLdsQ0 : kLdsQ1;
            q[2 * c2 + c] = lab[c] > 0 ? F.prior[F.site_qoff[sb0 + k] - 1 + lab[c]] : F.site_qsum[sb0 + k];
          }
          if (k < K && combine_label(lab[0], lab[1]) == 0) fl |= kLdsUz;
          fl |= (uint32_t)lds_place(j * B.sb + s) << 16;
        }
        w[2 * c2] = pl[0] | (pl[1] << 16);
        w[2 * c2 + 1] = fl;
      }
      L.w[B.tab + e0 + e] = make_uint4(w[0], w[1], w[2], w[3]);
      L.q[B.tab + e0 + e] = make_double4(q[0], q[1], q[2], q[3]);
    }
  }
}

void run_lds_tables(const DevForest& F, const LdsPlan& L, const TreeWalk& TW, hipStream_t s) {
  hipLaunchKernelGGL(k_lds_tables, dim3(8, L.num_blocks), dim3(256), 0, s, F, L, TW);
}

void run_problem(const DevForest& F, const LdsPlan& L, const TreeWalk& TW, double* d, double* nu, double* phi,
                 double* nll, double* site_llh_out, int32_t* iters_out, const EmState& em, int max_steps,
                 int max_iter, double tol, int what, hipStream_t s, GradOut grad) {
  const PbArgs a{F, L, TW, d, nu, phi, nll, site_llh_out, iters_out, em, max_steps, max_iter, tol, what, grad};
  hipLaunchKernelGGL(k_problem, dim3(F.num_problems), dim3(kLdsThreads), L.lds_bytes, s, a);
}

// Primal-dual interior-point solve of the same problem.  With duals zl, zh of
// the bounds (zl (d - dmin) -> mu, zh (dmax - d) -> mu) a Newton step is the
// same Laplacian system with branch weights -f'' + zl / (d - dmin) + zh /
// (dmax - d); mu follows the complementarity down superlinearly, and no line
// search is needed: 8 to 15 systems a solve against the barrier's 60 to 135,
// ending at the same point (mu_end is the same).  It starts from the last
// solution drawn a tenth towards the strictly interior heights that the
// caller set, since a start at the bounds costs the barrier method one
// doubling of the distance a step.
//
// A system's two level sweeps are latency: everything they do not need is
// formed before (branch derivatives, each class's own sums), a class passes
// up the two values its parent adds (cG, cR) and down one fma, state is in
// LDS where it fits, and levels of at most 64 classes are the first
// wavefront's, without barriers.  250 leaves x 30 sites: 210 us a solve,
// the barrier method 7,750.
constexpr int kUltraIters = 60;

// LDS or global arrays of one problem's solve
struct UltraWork {
  double *t, *dt, *gg, *G0, *wup, *cG, *cR, *f, *u;  // classes
  double *w, *gp, *zl, *zh;                          // free branches
  const int4* link;  // classes: two child classes and the parent class (-1: none), whether there are more children
};
constexpr int kUltraClsDoubles = 9, kUltraBrDoubles = 4;

template <bool kLds>
__device__ __forceinline__ void ultra_sync() {
  if (kLds) lds_barrier(); else __syncthreads();
}

// the block's minimum of a and b, maximum of c
__device__ __forceinline__ void ultra_reduce(double& a, double& b, double& c, double* sh) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a = fmin(a, __shfl_xor(a, off, 64));
    b = fmin(b, __shfl_xor(b, off, 64));
    c = fmax(c, __shfl_xor(c, off, 64));
  }
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sh[3 * wid] = a;
    sh[3 * wid + 1] = b;
    sh[3 * wid + 2] = c;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kUltraThreads / 64; ++i) {
    a = fmin(a, sh[3 * i]);
    b = fmin(b, sh[3 * i + 1]);
    c = fmax(c, sh[3 * i + 2]);
  }
  __syncthreads();
}

__device__ __forceinline__ void ultra_up(const UltraDev& U, const UltraWork& W, int c0, int c, int nc) {
  if (c >= nc) return;
  const int4 link = W.link[c];
  double G = W.G0[c], r = W.gg[c];
  if (link.x >= 0) {
    G += W.cG[link.x];
    r += W.cR[link.x];
  }
  if (link.y >= 0) {
    G += W.cG[link.y];
    r += W.cR[link.y];
  }
  if (link.w)
    for (int j = U.pk_more_off[c0 + c]; j < U.pk_more_off[c0 + c + 1]; ++j) {
      G += W.cG[U.pk_more[j]];
      r += W.cR[U.pk_more[j]];
    }
  const double iD = 1.0 / (G + W.wup[c]);
  const double f = W.wup[c] * iD;
  W.f[c] = f;
  W.u[c] = r * iD;
  W.cG[c] = f * G;
  W.cR[c] = f * r;
}
__device__ __forceinline__ void ultra_down(const UltraWork& W, int c, int nc) {
  if (c >= nc) return;
  const int pc = W.link[c].z;
  W.dt[c] = pc < 0 ? W.u[c] : fma(W.f[c], W.dt[pc], W.u[c]);
}

// Returns whether the solve converged (d, nu_d, heights and status written);
// nothing is written otherwise.
template <bool kLds>
__device__ bool ultra_pd(const DevForest& F, const UltraDev& U, double* __restrict__ d, double nu0, int p,
                         const UltraWork& W, double* sh) {
  const int tid = (int)threadIdx.x;
  const int c0 = uniform_at(U.pk_cls_off, p), V = uniform_at(U.pk_cls_off, p + 1) - c0;
  const int b0 = uniform_at(U.pk_br_off, p), B = uniform_at(U.pk_br_off, p + 1) - b0;
  const int H = U.num_levels;
  const int* lo_ = U.pk_lvl + p * (H + 1);
  const double dmin = F.dmin, dmax = F.dmax;
  const double K = (double)uniform_at(F.tree_nsites, uniform_at(F.prob_tree_off, p));
  const double mu_end = 1e-13 * K;
  double mu = 1e-2 * K;
  // the narrow levels (at most 64 classes; levels only get narrower)
  int hn = H;
  if (kLds) {
    hn = 0;
    for (int h = 0; h < H; ++h)
      if (uniform_at(lo_, h + 1) - uniform_at(lo_, h) > 64) hn = h + 1;
  }
  for (int c = tid; c < V; c += kUltraThreads) {
    const int g = U.pk_cls[c0 + c];
    W.t[c] = fma(0.9, U.t[g], 0.1 * U.t0[g]);
  }
  ultra_sync<kLds>();
  auto height = [&](const double* t, int cls, double off) { return cls >= 0 ? t[cls] + off : off; };
  auto diff = [&](const double* t, int cls) { return cls >= 0 ? t[cls] : 0.0; };
  double bad = 0.0;
  for (int i = tid; i < B; i += kUltraThreads) {
    const UltraBranch br = U.pk_br[b0 + i];
    const double x = height(W.t, br.up, br.up_off) - height(W.t, br.dn, br.dn_off);
    const double lo = x - dmin, hi = dmax - x;
    if (!(lo > 0.0 && hi > 0.0)) bad = 1.0;
    W.zl[i] = mu / lo;
    W.zh[i] = mu / hi;
  }
  {
    double a = 0.0, b = 0.0;
    ultra_reduce(a, b, bad, sh);
  }
  if (bad != 0.0) return false;
  double last = INFINITY;
  bool ok = false;
  for (int it = 0; it < kUltraIters; ++it) {
    for (int i = tid; i < B; i += kUltraThreads) {
      const UltraBranch br = U.pk_br[b0 + i];
      const double x = height(W.t, br.up, br.up_off) - height(W.t, br.dn, br.dn_off);
      const double il = 1.0 / (x - dmin), ih = 1.0 / (dmax - x);
      const double S1 = U.bS1[br.v], Bq = U.bB[br.v];
      const double r1 = 1.0 / expm1(x);
      double g = fma(S1, r1, -U.bA[br.v]), w = S1 * r1 * (1.0 + r1);
      if (Bq > 0.0) {
        const double rn = nu0 / expm1(nu0 * x);
        g = fma(Bq, rn, g);
        w = fma(Bq * rn, nu0 + rn, w);
      }
      W.gp[i] = g + mu * (il - ih);
      W.w[i] = w + W.zl[i] * il + W.zh[i] * ih;
    }
    ultra_sync<kLds>();
    for (int c = tid; c < V; c += kUltraThreads) {
      double gg = 0.0, G = 0.0, wup = 0.0;
      for (int j = U.pk_inc_off[c0 + c]; j < U.pk_inc_off[c0 + c + 1]; ++j) {
        // branch, and its kind here: 0 below the class, to a pinned height; 1
        // below, to a child class; 2 above, from a pinned height; 3 above,
        // from the parent class
        const int e = U.pk_inc[j], i = e >> 2, k = e & 3;
        gg += k < 2 ? W.gp[i] : -W.gp[i];
        if (k == 0 || k == 2) G += W.w[i];
        if (k == 3) wup += W.w[i];
      }
      W.gg[c] = gg;
      W.G0[c] = G;
      W.wup[c] = wup;
    }
    ultra_sync<kLds>();
    for (int h = 0; h < hn; ++h) {
      const int e = uniform_at(lo_, h + 1);
      for (int c = uniform_at(lo_, h) + tid; c < e; c += kUltraThreads) ultra_up(U, W, c0, c, e);
      ultra_sync<kLds>();
    }
    if (kLds && tid < 64) {
      for (int h = hn; h < H; ++h) ultra_up(U, W, c0, uniform_at(lo_, h) + tid, uniform_at(lo_, h + 1));
      for (int h = H - 1; h >= hn; --h) ultra_down(W, uniform_at(lo_, h) + tid, uniform_at(lo_, h + 1));
    }
    ultra_sync<kLds>();
    for (int h = hn - 1; h >= 0; --h) {
      const int e = uniform_at(lo_, h + 1);
      for (int c = uniform_at(lo_, h) + tid; c < e; c += kUltraThreads) ultra_down(W, c, e);
      ultra_sync<kLds>();
    }
    // step lengths that keep the lengths and the duals inside
    const double tau = fmin(0.9999, fmax(0.99, 1.0 - mu / K));
    double ap = 1.0, ad = 1.0, step = 0.0;
    for (int c = tid; c < V; c += kUltraThreads) {
      const double s = fabs(W.dt[c]) / (1.0 + fabs(W.t[c]));
      step = s >= 0.0 ? fmax(step, s) : INFINITY;  // (NaN: not a step)
    }
    for (int i = tid; i < B; i += kUltraThreads) {
      const UltraBranch br = U.pk_br[b0 + i];
      const double x = height(W.t, br.up, br.up_off) - height(W.t, br.dn, br.dn_off);
      const double dx = diff(W.dt, br.up) - diff(W.dt, br.dn);
      const double lo = x - dmin, hi = dmax - x, zl = W.zl[i], zh = W.zh[i];
      const double dzl = (mu - zl * dx) / lo - zl, dzh = (mu + zh * dx) / hi - zh;
      if (dx < 0.0) ap = fmin(ap, tau * lo / -dx);
      if (dx > 0.0) ap = fmin(ap, tau * hi / dx);
      if (dzl < 0.0) ad = fmin(ad, tau * zl / -dzl);
      if (dzh < 0.0) ad = fmin(ad, tau * zh / -dzh);
    }
    ultra_reduce(ap, ad, step, sh);
    if (!isfinite(step)) return false;
    double comp = 0.0;
    for (int i = tid; i < B; i += kUltraThreads) {
      const UltraBranch br = U.pk_br[b0 + i];
      const double x = height(W.t, br.up, br.up_off) - height(W.t, br.dn, br.dn_off);
      const double dx = diff(W.dt, br.up) - diff(W.dt, br.dn);
      const double lo = x - dmin, hi = dmax - x;
      const double zl = fma(ad, (mu - W.zl[i] * dx) / lo - W.zl[i], W.zl[i]);
      const double zh = fma(ad, (mu + W.zh[i] * dx) / hi - W.zh[i], W.zh[i]);
      W.zl[i] = zl;
      W.zh[i] = zh;
      comp += zl * fma(ap, dx, lo) + zh * fma(-ap, dx, hi);
    }
    comp = block_sum<kUltraThreads>(comp, sh) / (2.0 * B);  // (all have read t)
    for (int c = tid; c < V; c += kUltraThreads) W.t[c] = fma(ap, W.dt[c], W.t[c]);
    ultra_sync<kLds>();
    step *= ap;
    if (mu <= mu_end) {
      // at the rounding floor of the steps where they stop falling
      if (step <= 1e-15 || (step <= 1e-12 && step > 0.25 * last)) {
        ok = true;
        break;
      }
      last = step;
    }
    mu = fmax(mu_end, fmin(mu, comp * fmax(0.1 * (1.0 - fmin(ap, ad)), fmin(0.1, comp / K))));
  }
  if (!ok) return false;
  for (int c = tid; c < V; c += kUltraThreads) U.t[U.pk_cls[c0 + c]] = W.t[c];
  for (int i = tid; i < B; i += kUltraThreads) {
    const UltraBranch br = U.pk_br[b0 + i];
    const double x = height(W.t, br.up, br.up_off) - height(W.t, br.dn, br.dn_off);
    d[br.v] = x;
    F.nu_d[F.node_pos[br.v]] = x;
  }
  if (tid == 0) U.status[p] = 0;
  return true;
}

template <bool kLds>
__global__ void __launch_bounds__(kUltraThreads) k_ultra(DevForest F, UltraDev U, double* __restrict__ d,
                                                         const double* __restrict__ nu,
                                                         const int32_t* __restrict__ done) {
  extern __shared__ __align__(16) char lds[];
  __shared__ double sh[3 * (kUltraThreads / 64)];
  const int p = blockIdx.x;
  if ((done && done[p]) || !U.has_free[p]) return;
  const int c0 = U.pk_cls_off[p], V = U.pk_cls_off[p + 1] - c0;
  const int b0 = U.pk_br_off[p], B = U.pk_br_off[p + 1] - b0;
  // (16-byte records first, the doubles after them)
  double* base = kLds ? reinterpret_cast<double*>(lds) + 2 * V
                      : U.pk_work + (int64_t)kUltraClsDoubles * c0 + (int64_t)kUltraBrDoubles * b0;
  double* bb = base + (int64_t)kUltraClsDoubles * V;
  const UltraWork W{base,         base + V,     base + 2 * V, base + 3 * V, base + 4 * V, base + 5 * V, base + 6 * V,
                    base + 7 * V, base + 8 * V, bb,           bb + B,       bb + 2 * B,   bb + 3 * B,
                    kLds ? reinterpret_cast<const int4*>(lds) : U.pk_link + c0};
  if (kLds)
    for (int c = (int)threadIdx.x; c < V; c += kUltraThreads) reinterpret_cast<int4*>(lds)[c] = U.pk_link[c0 + c];
  if (V > 0 && ultra_pd<kLds>(F, U, d, nu[p], p, W, sh)) return;
  __syncthreads();
  ultra_barrier(F, U, d, nu, p, sh);
}

void run_ultra(const DevForest& F, const UltraDev& U, double* d, const double* nu, const int32_t* done,
               hipStream_t s) {
  if (U.lds_bytes <= kLdsMaxBytes)
    hipLaunchKernelGGL(k_ultra<true>, dim3(F.num_problems), dim3(kUltraThreads), U.lds_bytes, s, F, U, d, nu, done);
  else
    hipLaunchKernelGGL(k_ultra<false>, dim3(F.num_problems), dim3(kUltraThreads), 0, s, F, U, d, nu, done);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
int seg_width(int max_k) {
  if (max_k <= 8) return 8;
  if (max_k <= 16) return 16;
  if (max_k <= 32) return 32;
  return 64;
}

#define LAML_DISPATCH_W(W, BODY)                     \
  switch (W) {                                       \
    case 8: { constexpr int WW = 8; BODY; } break;   \
    case 16: { constexpr int WW = 16; BODY; } break; \
    case 32: { constexpr int WW = 32; BODY; } break; \
    default: { constexpr int WW = 64; BODY; } break; \
  }

static dim3 seg_grid(int cnt, int W, int chunks) {
  const int segs = 256 / W;
  return dim3((cnt + segs - 1) / segs, chunks);
}

void run_labels(const DevForest& F, const std::vector<int32_t>& lvl, int W, hipStream_t s) {
  for (size_t h = 1; h + 1 < lvl.size(); ++h) {
    const int beg = lvl[h], cnt = lvl[h + 1] - lvl[h];
    if (cnt <= 0) continue;
    LAML_DISPATCH_W(W, {
      hipLaunchKernelGGL(k_labels<WW>, seg_grid(cnt, WW, F.max_chunks), dim3(256), 0, s, F, beg, cnt);
    });
  }
}

void run_qrows(const DevForest& F, double* qleaf, double* qint, hipStream_t s) {
  const int grid = std::max(1, std::min((F.num_nodes + 3) / 4, 8192));
  hipLaunchKernelGGL(k_qrows, dim3(grid), dim3(256), 0, s, F, qleaf, qint);
}

void run_pad_codes(const DevForest& F, const int16_t* packed, const int64_t* packed_off, hipStream_t s) {
  const int grid = std::max(1, std::min((F.num_leaves + 3) / 4, 8192));
  hipLaunchKernelGGL(k_pad_codes, dim3(grid), dim3(256), 0, s, F, packed, packed_off);
}

void run_coef(const DevForest& F, const double* d, const double* nu, const int32_t* done, hipStream_t s) {
  const int grid = (F.num_nodes + 255) / 256;
  hipLaunchKernelGGL(k_coef, dim3(grid), dim3(256), 0, s, F, d, nu, done);
}

void run_clade_coef(const DevForest& F, hipStream_t s) {
  hipLaunchKernelGGL(k_clade_coef, dim3((F.num_nodes + 255) / 256), dim3(256), 0, s, F);
}

static void launch_inside_rows(dim3 grid, hipStream_t s, const DevForest& F, int beg, int cnt, int cpw,
                               const int32_t* done, const int32_t* nodes) {
  hipLaunchKernelGGL(k_inside_rows, grid, dim3(256), 0, s, F, beg, cnt, cpw, done, nodes);
}

static void launch_outside_rows(dim3 grid, hipStream_t s, const DevForest& F, int beg, int cnt, int cpw,
                                const int32_t* done, const int32_t* nodes) {
  hipLaunchKernelGGL(k_outside_rows, grid, dim3(256), 0, s, F, beg, cnt, cpw, done, nodes);
}

// one level of the inside pass: row kernels when a per-level shape is given
// (W == 64), segment kernels otherwise
static void inside_level(const DevForest& F, const std::vector<int32_t>& lvl, int W, const std::vector<int32_t>& cpw,
                         int h, const int32_t* done, hipStream_t s) {
  const int beg = lvl[h], cnt = lvl[h + 1] - lvl[h];
  if (cnt <= 0) return;
  if (W == 64 && !cpw.empty() && cpw[h] > 0) {
    const int c = cpw[h];
    const dim3 grid((cnt + 3) / 4, (F.max_chunks + c - 1) / c);
    if (h == 1)
      hipLaunchKernelGGL(k_inside_rows_leaves, grid, dim3(256), 0, s, F, beg, cnt, c, done);
    else
      launch_inside_rows(grid, s, F, beg, cnt, c, done, nullptr);
    return;
  }
  LAML_DISPATCH_W(W, {
    hipLaunchKernelGGL(k_inside<WW>, seg_grid(cnt, WW, F.max_chunks), dim3(256), 0, s, F, beg, cnt, done);
  });
}

static void outside_level(const DevForest& F, const std::vector<int32_t>& lvl, int W, const std::vector<int32_t>& cpw,
                          int h, const int32_t* done, hipStream_t s) {
  const int beg = lvl[h], cnt = lvl[h + 1] - lvl[h];
  if (cnt <= 0) return;
  if (W == 64 && !cpw.empty() && cpw[h] > 0) {
    const int c = cpw[h];
    launch_outside_rows(dim3((cnt + 3) / 4, (F.max_chunks + c - 1) / c), s, F, beg, cnt, c, done, nullptr);
    return;
  }
  LAML_DISPATCH_W(W, {
    hipLaunchKernelGGL(k_outside<WW>, seg_grid(cnt, WW, F.max_chunks), dim3(256), 0, s, F, beg, cnt, done);
  });
}

std::vector<int32_t> default_cpw(const std::vector<int32_t>& lvl, int W, int max_chunks) {
  std::vector<int32_t> c;
  if (W != 64) return c;
  const int H = (int)lvl.size() - 1;
  c.assign(H, 1);
  for (int h = 1; h < H; ++h) {
    const int64_t cnt = lvl[h + 1] - lvl[h];
    // enough wavefronts to keep every SIMD busy (kRowTargetWaves), then as
    // many chunks per wavefront as that allows
    const int64_t want = cnt * max_chunks / kRowTargetWaves;
    c[h] = (int32_t)std::max<int64_t>(1, std::min<int64_t>(max_chunks, want));
  }
  return c;
}

// One level of a pass with fused cherries (row kernels): the level's nodes
// without a cherry child, then those with one, each from its node list.
static void split_level(bool outside, const DevForest& F, const CherrySplit& cs, const std::vector<int32_t>& cpw,
                        int h, const int32_t* done, hipStream_t s) {
  const int c = std::max(1, cpw[h]);
  const int pb = cs.off[2 * h], pe = cs.off[2 * h + 1], ce = cs.off[2 * h + 2];
  const unsigned gy = (unsigned)((F.max_chunks + c - 1) / c);
  if (pe > pb) {
    const int cnt = pe - pb;
    if (outside)
      launch_outside_rows(dim3((cnt + 3) / 4, gy), s, F, pb, cnt, c, done, cs.nodes);
    else
      launch_inside_rows(dim3((cnt + 3) / 4, gy), s, F, pb, cnt, c, done, cs.nodes);
  }
  if (ce > pe) {
    const int cnt = ce - pe;
    if (outside)
      hipLaunchKernelGGL(k_outside_rows_ch, dim3((cnt + 3) / 4, gy), dim3(256), 0, s, F, pe, cnt, c, done,
                         cs.nodes);
    else
      hipLaunchKernelGGL(k_inside_rows_ch, dim3((cnt + 3) / 4, gy), dim3(256), 0, s, F, pe, cnt, c, done, cs.nodes);
  }
}

void run_inside(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h_top, const std::vector<int32_t>& cpw,
                const int32_t* done, hipStream_t s, const CherrySplit* cs, const ChainPlan* cp, const CladePlan* cl) {
  const int H = (int)lvl.size() - 1;
  if (cs) {
    // fused cherries: row kernels on every level from 2 up, no top kernel
    for (int h = 2; h < H; ++h) split_level(false, F, *cs, cpw, h, done, s);
    return;
  }
  const int ht = std::max(1, std::min(h_top, H));
  // chains below the chain plan's top level or clades and their rounds below
  // theirs, level launches from there
  const int h0 = cl ? std::min(cl->h_split, ht) : (cp ? std::min(cp->h_split, ht) : 1);
  if (cl) run_inside_clades(F, *cl, done, s);
  else if (cp) run_inside_chains(F, *cp, done, s);
  for (int h = h0; h < ht; ++h) inside_level(F, lvl, W, cpw, h, done, s);
  if (ht < H) {
    LAML_DISPATCH_W(W, {
      hipLaunchKernelGGL(k_inside_top<WW>, dim3(F.max_chunks), dim3(1024), 0, s, F, ht, H, done);
    });
  }
}

void run_root(const DevForest& F, int W, double* site_llh_out, const int32_t* done, hipStream_t s) {
  LAML_DISPATCH_W(W, {
    hipLaunchKernelGGL(k_root<WW>, seg_grid(F.num_trees, WW, F.max_chunks), dim3(256), 0, s, F, site_llh_out,
                       done);
  });
}

void run_outside_ckpt(const DevForest& F, const std::vector<int32_t>& lvl, int W, int L,
                      const std::vector<int32_t>& in_cpw, const std::vector<int32_t>& out_cpw, const int32_t* done,
                      hipStream_t s) {
  const int H = (int)lvl.size() - 1;
  const int nseg = (H - 1 + L - 1) / L;  // internal levels 1..H-1
  for (int sg = nseg - 1; sg >= 0; --sg) {
    const int a = 1 + sg * L, b = std::min(H, 1 + (sg + 1) * L);
    // recompute the segment's inside vectors (working area), then its
    // outside levels from the top of the segment down
    if (sg != nseg - 1)
      for (int h = a; h < b; ++h) inside_level(F, lvl, W, in_cpw, h, done, s);
    for (int h = b - 1; h >= a; --h) outside_level(F, lvl, W, out_cpw, h, done, s);
  }
}

void run_outside(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h_top,
                 const std::vector<int32_t>& cpw, const int32_t* done, hipStream_t s, const CherrySplit* cs,
                 const ChainPlan* cp, const CladePlan* cl) {
  const int H = (int)lvl.size() - 1;
  if (cs) {
    for (int h = H - 1; h >= 2; --h) split_level(true, F, *cs, cpw, h, done, s);
    return;
  }
  const int ht = std::max(1, std::min(h_top, H));
  if (ht < H) {
    LAML_DISPATCH_W(W, {
      hipLaunchKernelGGL(k_outside_top<WW>, dim3(F.max_chunks), dim3(1024), 0, s, F, ht, H, done);
    });
  }
  const int h0 = cl ? std::min(cl->h_split, ht) : (cp ? std::min(cp->h_split, ht) : 1);
  for (int h = ht - 1; h >= h0; --h) outside_level(F, lvl, W, cpw, h, done, s);
  if (cl) run_outside_clades(F, *cl, done, s);
  else if (cp) run_outside_chains(F, *cp, done, s);
}

void run_inside_clades(const DevForest& F, const CladePlan& cl, const int32_t* done, hipStream_t s) {
  if (cl.num > 0) {
    const dim3 g((unsigned)((cl.num + 7) / 8 * 8 * F.max_chunks)), b(64 * kCladeWaves);
    hipLaunchKernelGGL(k_inside_clade, g, b, (size_t)kCladeWaves * kCladeLds + cl.q_bytes, s, F, cl.blocks, cl.clades,
                       cl.steps, cl.leaf_row, cl.num, done);
  }
  for (size_t r = 0; r + 1 < cl.round_off.size(); ++r) {
    const int beg = cl.round_off[r], cnt = cl.round_off[r + 1] - beg;
    launch_inside_rows(dim3((cnt + 3) / 4, F.max_chunks), s, F, beg, cnt, 1, done, cl.rest);
  }
}

void run_outside_clades(const DevForest& F, const CladePlan& cl, const int32_t* done, hipStream_t s) {
  for (size_t r = cl.round_off.size() - 1; r-- > 0;) {
    const int beg = cl.round_off[r], cnt = cl.round_off[r + 1] - beg;
    launch_outside_rows(dim3((cnt + 3) / 4, F.max_chunks), s, F, beg, cnt, 1, done, cl.rest);
  }
  if (cl.out_num == 0) return;
  const size_t lds = (size_t)kCladeOutWaves * kOutLdsBytes + cl.q_bytes;
  hipLaunchKernelGGL(k_outside_clade, dim3((unsigned)((cl.out_num + 7) / 8 * 8 * F.max_chunks)),
                     dim3(64 * kCladeOutWaves), lds, s, F, cl.out_blocks, cl.clades, cl.out_steps, cl.out_num, done);
}

void run_inside_chains(const DevForest& F, const ChainPlan& cp, const int32_t* done, hipStream_t s) {
  for (size_t r = 0; r + 1 < cp.in_round_off.size(); ++r) {
    const int beg = cp.in_round_off[r], cnt = cp.in_round_off[r + 1] - beg;
    if (cnt <= 0) continue;
    const int64_t waves = (int64_t)cnt * F.max_chunks;
    hipLaunchKernelGGL(k_inside_chain, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, F, cp.in_chains, beg, cnt,
                       cp.nodes, done);
  }
}

void run_outside_chains(const DevForest& F, const ChainPlan& cp, const int32_t* done, hipStream_t s) {
  for (size_t r = 0; r + 1 < cp.pack_round_off.size(); ++r) {
    const int beg = cp.pack_round_off[r], cnt = cp.pack_round_off[r + 1] - beg;
    if (cnt <= 0) continue;
    const int64_t waves = (int64_t)cnt * F.max_chunks;
    if (cp.round_packed[r])
      hipLaunchKernelGGL(k_outside_chain<true>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, F, cp.packs, beg,
                         cnt, cp.pack_steps, cp.pack_head_ro, done);
    else
      hipLaunchKernelGGL(k_outside_chain<false>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, F, cp.packs, beg,
                         cnt, cp.pack_steps, cp.pack_head_ro, done);
  }
}

void run_tree_walk(const DevForest& F, const TreeWalk& TW, int W, int phases, double* site_llh_out,
                   const int32_t* done, hipStream_t s, int h_lo) {
  LAML_DISPATCH_W(W, {
    hipLaunchKernelGGL(k_tree_walk<WW>, dim3(TW.num_blocks), dim3(kWalkThreads), 0, s, F, TW, phases, h_lo,
                       site_llh_out, done);
  });
}

void run_inside_levels(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h0, int h1,
                       const std::vector<int32_t>& cpw, const int32_t* done, hipStream_t s) {
  for (int h = h0; h < h1; ++h) inside_level(F, lvl, W, cpw, h, done, s);
}

void run_outside_levels(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h0, int h1,
                        const std::vector<int32_t>& cpw, const int32_t* done, hipStream_t s) {
  for (int h = h1 - 1; h >= h0; --h) outside_level(F, lvl, W, cpw, h, done, s);
}

// Posterior state probabilities of every (node, site): P(v = 0 | D) and
// P(v = -1 | D), the post0 / post1 of EM_solver.Estep_posterior
// (EM_solver.py:247-300, in linear space), from the resident inside and
// outside state.  Segments index internal nodes; a leaf child's posteriors
// are formed from its parent's state as in the outside pass.  Outputs are
// packed as laml_forest_labels' are, so that they go to the caller in one copy
// each: leaf entries, then internal entries at leaf_sites; desc_off[v] is the
// node's first entry in its part.  (Padded rows, copied and then packed row by
// row on the host, took 0.4 ms of a call on 1,000 leaves x 100 sites.)
template <int W>
__global__ void __launch_bounds__(256) k_node_post(DevForest F, const int64_t* __restrict__ desc_off,
                                                   int64_t leaf_sites, double* __restrict__ p0,
                                                   double* __restrict__ pS) {
  Seg<W> g;
  if (!g.init(F.num_leaves, F.num_nodes - F.num_leaves)) return;
  const int u = g.v, k = g.k;
  const int t = F.tree_of[u];
  const int prob = F.tree_prob[t];
  const int K = F.tree_nsites[t];
  if (k >= K) return;
  const int sb = F.tree_site_base[t];
  const double phi = F.phi[prob];
  const int64_t ru = F.row_off[u];
  const int lu = F.labels[ru + k];
  const double2 au = F.alpha[ru + k];
  const double b0u = F.beta[F.brow[u] + k].x;
  const double pSu = lu < 0 ? F.pS[ru + k] : 0.0;
  const int64_t o = leaf_sites + desc_off[u] + k;
  p0[o] = lu == 0 ? 1.0 : au.x * b0u;
  pS[o] = pSu;
  const int ch[2] = {F.child0[u], F.child1[u]};
  const bool lf[2] = {ch[0] < F.num_leaves, ch[1] < F.num_leaves};
  if (!lf[0] && !lf[1]) return;
  const int qo = F.site_qoff[sb + k] - 1;
  const double qs = F.site_qsum[sb + k];
  int lab[2], E[2], code[2];
  double b0[2], bA[2], q[2];
  Eps ep[2];
  const Coef cf[2] = {F.coef[ch[0]], F.coef[ch[1]]};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    load_child(F, ch[i], lf[i], k, phi, lab[i], b0[i], bA[i], E[i], code[i]);
    q[i] = lab[i] > 0 ? F.prior[qo + lab[i]] : qs;
    ep[i] = edge(lab[i], b0[i], bA[i], E[i], q[i], cf[i]);
  }
  PostOut po;
  cond_post<true>(lu, au.x, au.y, pSu, phi, lab, b0, bA, q, ep, cf, lf, code, po);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (!lf[i]) continue;
    const int64_t ov = desc_off[ch[i]] + k;
    p0[ov] = po.S[i][0];
    pS[ov] = lab[i] < 0 ? po.pS[i] : 0.0;
  }
}

void run_node_post(const DevForest& F, int W, const int64_t* desc_off, int64_t leaf_sites, double* p0, double* pS,
                   hipStream_t s) {
  const int cnt = F.num_nodes - F.num_leaves;
  if (cnt <= 0) return;
  LAML_DISPATCH_W(W, {
    hipLaunchKernelGGL(k_node_post<WW>, seg_grid(cnt, WW, F.max_chunks), dim3(256), 0, s, F, desc_off, leaf_sites,
                       p0, pS);
  });
}

// ---------------------------------------------------------------------------
// Staging area of laml_posteriors_noalloc: a file-scope device array, so that
// the entry point needs no allocation.  In host code the name `scratch` is a
// host-side stand-in, never a device address: the address every kernel
// argument and copy uses is the one hipGetSymbolAddress returns for the
// device that is current, looked up once per device by post_scratch().
// ---------------------------------------------------------------------------
static __device__ __align__(256) double scratch[kPostScratchDoubles];

int post_scratch(int device, double** out) {
  static std::mutex mu;
  static std::map<int, double*> by_device;
  std::lock_guard<std::mutex> lock(mu);
  auto it = by_device.find(device);
  if (it == by_device.end()) {
    // the caller has made `device` current: each device holds its own copy
    // of the array at its own address
    double* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    it = by_device.emplace(device, ptr).first;
  }
  *out = it->second;
  return 0;
}

int max_lds(int device) {
  static std::mutex mu;
  static std::map<int, int> by_device;
  std::lock_guard<std::mutex> lock(mu);
  auto it = by_device.find(device);
  if (it == by_device.end()) {
    // kernel attributes are the current device's, as `device` is
    bool ok = true;
    for (const void* k : {reinterpret_cast<const void*>(k_problem), reinterpret_cast<const void*>(k_ultra<true>),
                          reinterpret_cast<const void*>(k_outside_clade)})
      ok = ok && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMaxBytes) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    it = by_device.emplace(device, ok ? kLdsMaxBytes : 0).first;
  }
  return it->second;
}

void run_counts(const DevForest& F, double* counts, hipStream_t s) {
  hipLaunchKernelGGL(k_counts, dim3((unsigned)(((int64_t)F.num_nodes * 5 + 255) / 256)), dim3(256), 0, s, F,
                     counts);
}

// clears the EM bookkeeping of every problem (a kernel rather than a memset,
// so that the call stays valid inside a caller's stream capture)
__global__ void k_em_reset(EmState em, int P) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  em.done[p] = 0;
  em.iters[p] = 0;
  em.step[p] = 0;
}

void run_em_reset(const EmState& em, int P, hipStream_t s) {
  hipLaunchKernelGGL(k_em_reset, dim3((P + 255) / 256), dim3(256), 0, s, em, P);
}

void run_llh(const DevForest& F, double* nll, EmState em, int max_iter, double tol, hipStream_t s) {
  hipLaunchKernelGGL(k_llh, dim3(F.num_problems), dim3(256), 0, s, F, nll, em, max_iter, tol);
}

void run_grad(const DevForest& F, const double* d, const double* nu, const double* phi, double* grad_d,
              double* grad_nu, double* grad_phi, hipStream_t s) {
  hipLaunchKernelGGL(k_grad_branch, dim3((F.num_nodes + 255) / 256), dim3(256), 0, s, F, d, nu, grad_d);
  hipLaunchKernelGGL(k_grad_problem, dim3(F.num_problems), dim3(kRedThreads), 0, s, F, nu, phi, grad_nu, grad_phi);
}

void run_rtilde(const DevForest& F, double* rtilde, const int32_t* done, hipStream_t s) {
  hipLaunchKernelGGL(k_rtilde, dim3(F.num_problems), dim3(kRedThreads), 0, s, F, rtilde, done);
}

void run_mstep(const DevForest& F, const double* counts, const double* rtilde, double* d, double* nu, double* phi,
               const int32_t* done, hipStream_t s, const UltraDev* U) {
  const dim3 g(F.num_nu_blocks), b(kNuThreads);
  if (U) {
    hipLaunchKernelGGL(k_branch<true>, g, b, 0, s, F, counts, rtilde, d, nu, done, *U);
    run_ultra(F, *U, d, nu, done, s);
    hipLaunchKernelGGL(k_nu_eval<true>, g, b, 0, s, F, rtilde, nu, done);
  } else {
    hipLaunchKernelGGL(k_branch<false>, g, b, 0, s, F, counts, rtilde, d, nu, done, UltraDev{});
  }
  hipLaunchKernelGGL(k_nu_eval<false>, g, b, 0, s, F, rtilde, nu, done);
  hipLaunchKernelGGL(k_nu_finish, dim3(F.num_problems), dim3(kNuFinishThreads), 0, s, F, rtilde, nu, phi, done);
}

}  // namespace laml
