// Internal interface between the kernels and the C ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "pmm_device.hpp"

namespace laml {

// branches of a problem that a block of the nu evaluations takes
constexpr int kNuSpan = 256;

// Per internal node, what the inside row kernel reads before its row loads
// (one scalar load instead of chains of dependent ones): children, problem,
// sites and first site of the tree, and the row offsets of the node's labels
// and inside row and of its children's.
struct NodeRec {
  int32_t ch0, ch1, p, K;
  int32_t sb, pad;
  int64_t ro, bro;
  int64_t ro0, bro0, ro1, bro1;
};

// Device view of a forest; passed by value to every kernel.
struct DevForest {
  int32_t num_nodes, num_leaves, num_trees, num_problems;
  int32_t chunk_w;     // sites per segment (W)
  int32_t max_chunks;  // ceil(max K / W)
  // nodes [num_leaves, cherry_end) are fused cherries in the current pass
  // (their parents form and consume their inside and outside states; no
  // cherry row is read or written); cherry_end == num_leaves: no fusion
  int32_t cherry_end;
  // 1: the inside/outside rows of a pass exceed the last-level cache, and
  // the row kernels read and write them with the non-temporal hint
  int32_t stream_rows;
  double dmin, dmax;
  // topology (level order)
  const int32_t* level_off;  // [levels+1]
  const int32_t* child0;
  const int32_t* child1;
  const int32_t* tree_of;
  const int64_t* row_off;
  const int64_t* brow;  // [N] row of the node's inside vector (beta, bE)
  const NodeRec* nrec;  // [N - num_leaves] by internal node
  const uint8_t* free_branch;
  // trees / problems
  const int32_t* tree_root;
  const int32_t* tree_prob;
  const int32_t* tree_nsites;
  const int32_t* tree_site_base;
  const int32_t* prob_tree_off;  // [P+1]
  const int32_t* prob_node_off;  // [P+1]
  const int32_t* prob_nodes;     // nodes grouped by problem (leaves first)
  const int32_t* prob_int_off;   // [P] first internal node of each problem in prob_nodes
  const int32_t* prob_nfree;     // [P] number of optimised branches
  const int32_t* node_pos;       // [N] position of each node in prob_nodes
  const int32_t* prob_blk_off;   // [P+1] blocks of the nu solve per problem
  int32_t num_nu_blocks;
  const uint32_t* prob_flags;
  const double* prob_nobs;
  const double* prob_phimin;
  const double* prob_nobs_phi;  // [P] leaf entries observed as 0 or an edit
  // sites
  const int32_t* site_qoff;  // 1-based local state j -> prior[site_qoff[s] + j - 1]
  const double* site_qsum;   // prior mass of each site's alphabet (1 for normalised priors)
  const double* prior;
  const int16_t* codes;  // leaf rows
  // prior weight of each node's label at each site (leaf rows by the leaf
  // row offsets, internal rows by the internal ones): prior[site_qoff[s] - 1 +
  // label] for an edit label, the site's prior mass site_qsum[s] otherwise;
  // fixed for the forest's life (labels and priors are)
  const double* qleaf;
  const double* qint;
  // per-call parameters
  const double* phi;  // [P]
  // state
  int16_t* labels;  // internal rows
  Coef* coef;       // [N]
  // the coefficients of the clade plan of the next inside pass (null: none),
  // written by k_coef, and their places by branch
  struct CladeCoef* clade_coef;
  const int32_t* clade_pos;
  double2* beta;    // internal rows
  int32_t* bE;
  // outside state (a0, aX) of internal nodes given all data, on the scale of
  // beta (undefined where the label is 'z'), and P(silenced | D) where the
  // label is '?'
  double2* alpha;
  double* pS;
  double* site_llh;
  double* rt_part;  // [N * max_chunks] dropout sums of leaf children per chunk
  double* cpart;    // [N * max_chunks * 5] per-chunk branch count partials
  // where the readers of the partials find node v's chunk c: cpart + v cp_v +
  // 5 c, rt_part + v rt_v + c (a node's chunks side by side; one chunk holds
  // all sites of the problems that k_problem runs)
  int64_t cp_v, rt_v;
  double* nu_a;     // [N] by position in prob_nodes: S0+S1+S3 of the branch
  double* nu_b;     // [N] S2+S4 (0 for fixed branches)
  double* nu_d;     // [N] new branch length
  double* nu_part;  // [2][num_nu_blocks][6] partial sums of the nu solve
  int32_t* mstep_status;  // [P] last M-step: bit 0 a branch length came out non-finite, bit 1 the nu solve did
                          // not converge (kept at its last iterate)
};

// a free branch of the ultrametric solve: its node, and the class (numbered
// within the problem, -1: pinned) and offset of its upper and lower end
struct UltraBranch {
  int32_t v, up, dn, pad;
  double up_off, dn_off;
};

// Height-class model of the ultrametric constraint (one per forest)
struct UltraDev {
  int32_t num_classes, num_levels;
  const int32_t* plo;        // [num_levels * P + 1] class ranges by (level, problem)
  const int32_t* up_cls;     // [N] parent-side class of each free branch (-1 pinned)
  const int32_t* dn_cls;     // [N] child-side class (-1 pinned)
  const double* up_off;      // [N] offset (absolute height when pinned)
  const double* dn_off;      // [N]
  const int32_t* cls_parent; // [V]
  const int32_t* cls_pedge;  // [V] branch joining the class to its parent class
  const int32_t* inc_off;    // [V+1]
  const int32_t* inc_branch; // incident free branches
  const int8_t* inc_sign;    // +1: class is the parent side
  const uint8_t* has_free;   // [P]
  double* t;                 // [V] heights (warm start / solution)
  double* dt;                // [V] Newton direction
  double* Dd;                // [V] eliminated diagonal (= Gg + weight of the edge to the parent class)
  double* Gg;                // [V] conductance of the class subtree to the pinned heights
  double* r;                 // [V] eliminated right-hand side
  double* g;                 // [V] gradient
  double* gp;                // [N] branch first derivative
  double* w;                 // [N] branch curvature (positive)
  double* bA;                // [N] branch objective: -A d + S1 log(1-e^-d) + B log(1-e^-nu d)
  double* bS1;
  double* bB;
  int32_t* status;           // [P] 0 ok, 1 line search stalled, 2 singular Newton system
  double* t0;                // [V] the strictly interior heights that the caller set
  // the same model by problem (classes and branches numbered within it,
  // classes in level order), for the primal-dual solve
  int32_t lds_bytes;         // state of the largest problem's solve
  const int32_t* pk_cls_off; // [P + 1] into the class arrays below
  const int32_t* pk_cls;     // the class's number in t
  const int32_t* pk_lvl;     // [P][num_levels + 1] first class of each level
  const int4* pk_link;       // the first two child classes, the parent class (-1: none), whether there are more
  const int32_t* pk_more_off;  // further child classes
  const int32_t* pk_more;
  const int32_t* pk_inc_off; // incident branches: 4 * branch + kind (see ultra_pd)
  const int32_t* pk_inc;
  const int32_t* pk_br_off;  // [P + 1] into pk_br
  const UltraBranch* pk_br;
  double* pk_work;           // state of the solves that do not fit LDS
};

// Tree-walk launch plan: block b runs tree blk_tree[b] at site chunk
// blk_chunk[b]; tree t's internal levels are lvl_base[t] + 1 ..
// lvl_base[t+1] - 1, level h holding the contiguous node range
// [lvl_beg[lvl_base[t] + h], + lvl_cnt[...]).
struct TreeWalk {
  int32_t num_blocks;
  const int32_t* blk_tree;
  const int32_t* blk_chunk;
  const int32_t* lvl_base;  // [T+1]
  const int32_t* lvl_beg;
  const int32_t* lvl_cnt;
};

// Plan of k_problem: block b runs tree blk[b].tree at all its sites (sb: their
// number rounded up to a multiple of the reduction width), the state of every
// internal node in LDS.  Internal nodes are numbered within their tree in level
// order ("local"), so the root is last.
struct LdsBlk {
  int32_t tree, sb, nint, pad;  // nint: internal nodes of the tree
  int64_t tab;                  // first entry of the block's cell tables
};
// an internal node: its children's local numbers (-1: leaf) and node ids, its
// own id
struct LdsRec {
  int32_t l0, l1, g0, g1, v, pad;
};
// coefficients of the branches to a record's two children (as Coef; esil
// kZeroTop where msil is 0)
struct LdsCoef {
  double p1n[2], mut[2], pn[2], msil[2];
  int32_t esil[2];
  int32_t pad[2];
};
struct LdsPlan {
  int32_t num_blocks;
  int32_t lds_bytes;           // dynamic LDS of a block
  const LdsBlk* blk;
  const int32_t* int_base;     // [T] first record of each tree
  const LdsRec* rec;           // [internal nodes] by tree, then local
  const int2* lvl_off;         // [as the tree walk's levels] local number and table entry after level h
  LdsCoef* lcoef;              // [internal nodes] branch coefficients of both children of each record
  // per block and pair of (node, site) cells, in the order the block's threads
  // read them: where the children's vectors lie in LDS and label flags, and
  // the children's prior weights; fixed for the forest's life
  uint4* w;
  double4* q;
  double* cpart;               // partials
  double* rt_part;
};

struct EmState {
  int32_t* done;   // [P] or nullptr outside the EM loop
  int32_t* iters;  // [P]
  int32_t* step;   // [P] EM steps taken (read and advanced on the device)
  double* pre;     // [P]
  double* trace;   // [(max_iter+1)*P] or nullptr
};

int seg_width(int max_k);
// dynamic LDS a block of the LDS passes may take (160 KiB less their static
// arrays)
constexpr int kLdsMaxBytes = 160 * 1024 - 1024;
// what they may take on `device` (which must be current), set up once per
// device: kLdsMaxBytes, or 0 where the runtime refuses it (the passes then run
// without these kernels)
int max_lds(int device);
// sites of a block that share a partial-count slot in its LDS (a block's
// sites are a multiple)
constexpr int kLdsSlotSites = 8;
// Forests that k_problem takes.  Sites: a block holds all sites of a problem,
// and 64 x 120 leaves fill the LDS.  Problems: a CU's blocks run in turns, so
// the general passes overtake it when blocks are many and tiny (EM step, block
// / general: 256 problems of 250 x 30 89 / 308 us, 1,024 of them 308 / 658,
// 2,048 of 100 x 20 373 / 576, 4,096 of 60 x 16 720 / 588).
// A likelihood (with its gradient) goes through blocks up to kPbMaxSingle: 1,024
// problems of 10 x 8 41 (115) us, 46 (104) in the general passes, of 60 x 40
// 67 (204) and 73 (188), of 120 x 60 89 (286) and 97 (281); 768 of them 30 (84)
// and 35 (89), 51 (154) and 69 (172), 70 (221) and 90 (243); 1,280 of them 55
// (151) and 45 (106), 85 (259) and 85 (216), 136 (411) and 118 (334).
constexpr int kPbMaxSites = 64;
constexpr int kPbMaxProblems = 2048;
constexpr int kPbMaxSingle = 1024;
// the cell tables of an LDS plan (after run_labels)
void run_lds_tables(const DevForest& F, const LdsPlan& L, const TreeWalk& TW, hipStream_t s);
// What k_problem does, a block per problem: branch coefficients from d and nu
// (else those of the last call), the outside pass with counts (else inside
// and likelihood alone), EM steps (at most max_steps, of the max_iter that
// the run has in all), the gradient from the counts
constexpr int kPbCoef = 1, kPbOut = 2, kPbEm = 4, kPbGrad = 8;
struct GradOut {
  double *d, *nu, *phi;
};
void run_problem(const DevForest& F, const LdsPlan& L, const TreeWalk& TW, double* d, double* nu, double* phi,
                 double* nll, double* site_llh_out, int32_t* iters_out, const EmState& em, int max_steps,
                 int max_iter, double tol, int what, hipStream_t s, GradOut grad = {});
void run_labels(const DevForest& F, const std::vector<int32_t>& lvl, int W, hipStream_t s);
// the prior-weight rows qleaf / qint from the codes and labels (after run_labels)
void run_qrows(const DevForest& F, double* qleaf, double* qint, hipStream_t s);
// leaf code rows from the packed host layout (uploaded as it is) into the
// padded device rows of F.codes
void run_pad_codes(const DevForest& F, const int16_t* packed, const int64_t* packed_off, hipStream_t s);
void run_coef(const DevForest& F, const double* d, const double* nu, const int32_t* done, hipStream_t s);
// wavefronts a row-kernel launch aims for before it gives each wavefront
// more than one chunk of 64 sites (8 per SIMD of the 256 CUs)
constexpr int64_t kRowTargetWaves = 8192;
// default chunks per wavefront of the row kernels for each level (empty
// unless W == 64)
std::vector<int32_t> default_cpw(const std::vector<int32_t>& lvl, int W, int max_chunks);
// Per-level node lists of a pass with fused cherries: for level h >= 2,
// nodes[off[2h] .. off[2h+1]) have no cherry child, nodes[off[2h+1] ..
// off[2h+2]) have at least one (device list, host offsets).
struct CherrySplit {
  const int32_t* nodes = nullptr;
  std::vector<int32_t> off;
};

// Heavy-path chains over the levels below h_split (k_outside_chain,
// k_inside_chain): a chain is a node and its successive heavy children,
// head first.  Outside rounds: the heads of round 0 get their outside state
// from the levels above h_split or the root step, those of round r > 0 from
// round r - 1; round r's packs are [pack_round_off[r], pack_round_off[r +
// 1]), longest first, each the steps of one or more of the round's chains of
// one tree.  in_chains lists the chains (offset into nodes, length) in
// inside rounds: a chain runs one round after the last chain hanging off it
// (its light internal children's), round 0 holding chains with none (device
// arrays, host offsets).
// One node of a chain, as the outside chain kernel reads it: the node, its
// children, which child continues the chain (-1: none), and the children's
// row offsets.
struct ChainStep {
  int32_t u, ch0, ch1, hv;
  int64_t ro0, ro1;
};

struct ChainPlan {
  int32_t h_split = -1;
  int32_t pack_cap = 0;              // most steps per outside pack the plan was built for
  bool inside = false;               // with the inside rounds (only where inside chains are asked for)
  const int2* in_chains = nullptr;
  const int32_t* nodes = nullptr;
  // outside packs: (offset into pack_steps, steps), each one or more chains
  // of one tree back to back; a chain's first record holds ~u and
  // pack_head_ro its row offset
  const int2* packs = nullptr;
  const ChainStep* pack_steps = nullptr;
  const int64_t* pack_head_ro = nullptr;
  std::vector<int32_t> pack_round_off, in_round_off;
  std::vector<uint8_t> round_packed;  // per round: some pack holds more than one chain
};
// wavefronts an outside chain round keeps: its packs hold at most
// max(1, min(cap, (steps x chunks) / kPackWaves)) steps, so that packing
// only thins rounds with wavefronts to spare (16 per SIMD)
constexpr int64_t kPackWaves = 16384;

// Clades of the inside pass (k_inside_clade): maximal subtrees below level
// h_split of at most `cap` internal nodes whose walk keeps at most kCladeSlots
// pending states.  A wavefront walks a clade's nodes in postorder at a 64-site
// chunk, so that their rows are written and never read; the other nodes below
// h_split follow in rounds of row launches (`rest`: node list, round_off: host
// offsets), each after the rounds of its children.
constexpr int kCladeSlots = 2;
constexpr int kCladeBatch = 8;  // leaves whose codes a wavefront loads at a time
constexpr int kCladeSlotBytes = 64 * 24;
constexpr int kCladeLds = kCladeSlots * kCladeSlotBytes + kCladeBatch * 128;  // a wavefront's slice
// One node of a clade: its row, in units of 64 sites, and bits of flags: 0-1
// kind (0 two leaves, 1 carried and leaf, 2 carried and pending), 2-3 slot of
// the pending state, 4-6 one more than the slot that the result goes to (0:
// carried only), 7 the next batch of leaves comes before this step, 8-10 and
// 11-13 place of the children's codes in the batch.
struct CladeStep {
  int32_t row, flags;
};
// The same node for the outside walk, which runs the steps in reverse: the
// node, its children and their rows (codes of a leaf, inside row and labels of
// an internal node).
struct CladeOut {
  int32_t u, flags, ch[2], row[2];
};
// The coefficients of its branches in one piece, written by k_coef (scalar
// loads of coefficients by branch took most of the walk's time); children
// ordered so that the first is the one whose state the wavefront carries (or
// both are leaves).
struct CladeCoef {
  double p1n[2], mut[2], pn[2], msil[2];
  int32_t esil[2];
};
struct CladePlan {
  int32_t h_split = -1, cap = 0;
  int32_t count = 0, largest = 0;  // clades, internal nodes of the largest
  int32_t num = 0;               // blocks
  int32_t q_bytes = 0;           // LDS for the prior weights of a chunk
  const int4* blocks = nullptr;  // first clade, clades, tree
  const int4* clades = nullptr;  // offset into steps, steps, first batch, batches
  const CladeStep* steps = nullptr;
  CladeCoef* coef = nullptr;     // by step
  int32_t out_num = 0;           // blocks of the outside pass (0: it takes none, see kCladeOutFill)
  const int4* out_blocks = nullptr;
  const CladeOut* out_steps = nullptr;
  const int32_t* pos = nullptr;  // [N] place of a branch's coefficients: 2 step + child, -1 none
  const int32_t* leaf_row = nullptr;  // [batch][kCladeBatch] code rows of the leaves, in units of 64 sites
  const int32_t* rest = nullptr;
  std::vector<int32_t> round_off;
};
constexpr int kCladeWaves = 8;      // wavefronts of a block, inside
constexpr int kCladeOutWaves = 12;  // and outside
// Most nodes of a clade: one per kCladePairs (internal node, 64-site chunk)
// pairs of the forest, between kCladeMin and kCladeCap.  Longer walks read
// fewer rows back, but the wavefronts have to fill the chip.  E-step of 10,000
// leaves x 300 (50k pairs): 216 us at 16, 219 at 24, 234 at 32; of sixteen such
// trees (800k) 1052 at 16, 929 at 32, 899 at 64.
constexpr int64_t kCladePairs = 4096;
constexpr int kCladeMin = 16, kCladeCap = 64;
// Forests of at least this many pairs take clades in the inside pass: 2,000 x
// 500 (16k pairs) 63 us, 76 by levels; 1,000 x 500 (8k) 48 and 53, but a forest
// that is solved once and dropped does not earn its plan back.
constexpr int64_t kCladeForest = 12288;
// Forests below kCladeEager pairs lay clades out once their calls would have
// saved the time: the plan takes 0.11 ms (4,000 leaves x 300, 20k pairs), a
// likelihood saves 12 us of 82 there, an E-step 30, an EM step 55.  From
// kCladeEager pairs on (where outside chains had their plan to lay out) at
// once.
constexpr int64_t kCladeEager = 32768;
constexpr int64_t kCladeEarn = 10;
// And of at least this many in the outside pass as well: E-step of 300 trees of
// 300 leaves x 300 (60k pairs) 172 us, 203 by chains; of 10,000 x 300 (50k) 216
// and 221, but its gradient, whose launches are not in a graph, 291 and 267.
constexpr int64_t kCladeOutForest = 57344;
// Nor where a block holds at most this many clades on average: its wavefronts
// walk clades of one tree, and with few of them the CU idles.  E-step by clades
// a block, clades / chains: 1 (2,048 trees of 20 leaves x 300) 794 / 472 us,
// 1.5 (2,048 of 40 x 70) 538 / 328, 4 (1,024 of 60 x 70) 290 / 241, 5.5 (500 of
// 100 x 130) 294 / 266, 7.4 (300 of 300 x 300) 576 / 612, 8 (300 of 100 x 70)
// 169 / 176, 9.7 (100 of 400 x 200) 270 / 286.
constexpr int kCladeOutFill = 6;
// most LDS for a chunk's prior weights: 64 sites of 62 edit states (up to 21 KB
// three blocks fit a CU)
constexpr int kCladeMaxQ = 31 * 1024;

// cp: the levels below the top kernel's run as heavy-path chains; cl: as
// clades
void run_inside(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h_top, const std::vector<int32_t>& cpw,
                const int32_t* done, hipStream_t s, const CherrySplit* cs = nullptr, const ChainPlan* cp = nullptr,
                const CladePlan* cl = nullptr);
void run_clade_coef(const DevForest& F, hipStream_t s);
void run_inside_clades(const DevForest& F, const CladePlan& cl, const int32_t* done, hipStream_t s);
void run_outside_clades(const DevForest& F, const CladePlan& cl, const int32_t* done, hipStream_t s);
void run_inside_chains(const DevForest& F, const ChainPlan& cp, const int32_t* done, hipStream_t s);
// cp: the levels below the top kernel's run as heavy-path chains
void run_outside(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h_top,
                 const std::vector<int32_t>& cpw, const int32_t* done, hipStream_t s, const CherrySplit* cs = nullptr,
                 const ChainPlan* cp = nullptr, const CladePlan* cl = nullptr);
void run_outside_chains(const DevForest& F, const ChainPlan& cp, const int32_t* done, hipStream_t s);
void run_outside_ckpt(const DevForest& F, const std::vector<int32_t>& lvl, int W, int L,
                      const std::vector<int32_t>& in_cpw, const std::vector<int32_t>& out_cpw, const int32_t* done,
                      hipStream_t s);
void run_root(const DevForest& F, int W, double* site_llh_out, const int32_t* done, hipStream_t s);
void run_counts(const DevForest& F, double* counts, hipStream_t s);
void run_tree_walk(const DevForest& F, const TreeWalk& TW, int W, int phases, double* site_llh_out,
                   const int32_t* done, hipStream_t s, int h_lo = 1);
// levels [h0, h1) of the inside pass (bottom up) / outside pass (top down)
void run_inside_levels(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h0, int h1,
                       const std::vector<int32_t>& cpw, const int32_t* done, hipStream_t s);
void run_outside_levels(const DevForest& F, const std::vector<int32_t>& lvl, int W, int h0, int h1,
                        const std::vector<int32_t>& cpw, const int32_t* done, hipStream_t s);
void run_llh(const DevForest& F, double* nll, EmState em, int max_iter, double tol, hipStream_t s);
void run_em_reset(const EmState& em, int P, hipStream_t s);
void run_node_post(const DevForest& F, int W, const int64_t* desc_off, int64_t leaf_sites, double* p0, double* pS,
                   hipStream_t s);
// doubles in the file-scope staging array of laml_posteriors_noalloc (64 MiB
// per device, held until the process ends)
constexpr int64_t kPostScratchDoubles = (int64_t)8 << 20;
// device address of that array on `device` (which must be current), looked
// up once per device; 0 or a hipError_t
int post_scratch(int device, double** out);
void run_quartet_em(const DevForest& F, int ncand, const int32_t* qnodes, const double* len_in,
                    const uint8_t* opt_mask, const double* llh_const, const double* nu, const double* phi,
                    int max_iter, double tol, double* len_out, double* nll_out, int32_t* iters_out, hipStream_t s);
void run_rtilde(const DevForest& F, double* rtilde, const int32_t* done, hipStream_t s);
void run_grad(const DevForest& F, const double* d, const double* nu, const double* phi, double* grad_d,
              double* grad_nu, double* grad_phi, hipStream_t s);
void run_ultra(const DevForest& F, const UltraDev& U, double* d, const double* nu, const int32_t* done,
               hipStream_t s);
void run_mstep(const DevForest& F, const double* counts, const double* rtilde, double* d, double* nu, double* phi,
               const int32_t* done, hipStream_t s, const UltraDev* U = nullptr);

}  // namespace laml
