// Kernel argument blocks shared by the host plan code and the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gscf {

// ---------------------------------------------------------------------------
// Plan data (device, structure-of-arrays where lanes gather)
// ---------------------------------------------------------------------------
struct PrimPair {
  double p;        // alpha_a + alpha_b
  double px, py, pz;
  double e;        // c_a c_b K_AB sqrt(2 pi^{5/2}) / p
  double aa;       // alpha_a (first-centre exponent)
  double ab;       // alpha_b
  double ip;       // 1 / p
};

// Per primitive pair, for the basis-parameter derivatives only: primitive
// indices inside the two segmented shells, their coefficients (s/p factor
// included) and the coefficient-free factor K_AB sqrt(2 pi^{5/2}) / p.
struct PrimAux {
  int ia, ib;
  double ca, cb;
  double ek;
};

// Column coefficients (s/p factor included) of a primitive pair of a
// contracted pair: primitive i of shell A in columns 0/1, primitive j of shell
// B in columns 0/1 (zero where a shell has one column).  The primitive pair's
// e then carries no coefficients.
struct PrimCoef {
  double ca[2];
  double cb[2];
};

// Column pattern of a pair: columns of (A, B) = (1 + (p & 1), 1 + (p >> 1)).
__host__ __device__ constexpr bool pattern_valid(int la, int lb, int p) {
  return p == 0 || (la == 0 && lb == 0 && (p == 1 || p == 3)) || (la > 0 && lb == 0 && p == 2);
}

struct Pair {
  int sa, sb;      // segmented shells, l(sa) >= l(sb)
  int poff, np;    // primitive-pair range
};

struct ShellXYZ {
  double x, y, z;
  int ao;          // Cartesian AO offset inside its molecule
  int l;
  int mol;         // molecule of a batched plan
  int lseg;        // segmented-shell index inside its molecule
};

// Per-molecule layout of a (batched) plan: Cartesian matrices of molecule m
// live at base .. base + n*n of every density/J/K batch; dbase/nseg address
// its shell-block density maxima.
struct MolInfo {
  int64_t base;
  int64_t dbase;
  int32_t n;
  int32_t nseg;
  int32_t nuc0;   // nuclei of the molecule: [nuc0, nuc0 + nnuc) of the plan's list
  int32_t nnuc;
  int64_t sbase;  // the molecule's matrix in the requested AO basis, ns x ns
  int32_t ns;
  int32_t pad;
};


// Work of one quartet class is a list of canonical quartets (bra pair, ket
// pair), grouped into sub-tasks of similar primitive counts.  Sub-task t owns
// quartets [q0, q0+nq) and work items [item0, item0 + S*nq): item
// item0 + s*nq + g processes quartet q0+g for slice s of its primitive
// quartets, S = Sb * Sk: bra primitive pairs s % Sb, s % Sb + Sb, ... with ket
// primitive pairs s / Sb, s / Sb + Sk, ...
struct SubTask {
  int64_t item0;
  int64_t q0;
  int64_t nq;
  int32_t S;
  int32_t Sk;
};

struct JKArgs {
  const Pair* pairs;
  const PrimPair* prims;
  const ShellXYZ* shells;
  const int2* quartets;
  const SubTask* tasks;
  int ntasks;
  int64_t nitems;
  int64_t item0;        // first item of this launch (set by the launcher, with nitems its end)
  const double* dens;   // [nbd][sum_m n_m^2] Cartesian densities
  double* jp;           // [nbj][...] partial J (J = Jp + Jp^T)
  double* kp;           // [nbd][...] partial K
  const MolInfo* mols;
  int64_t bstride;      // elements per density batch
  int n, nbd, nbj, with_j, with_k;
  // deterministic digestion: [nmol][2] (scale, 1/scale); NULL for FP64 atomics
  const double* det_scale;
};

// Bra-major chunk: quartets [q0, q0+nq) of one sub-task whose bras are the
// consecutive pairs [bra0, bra0+nbra); one workgroup per chunk accumulates the
// exchange rows of those bras (and their J blocks) in LDS.
struct BraChunk {
  int64_t q0;
  int32_t nq;
  int32_t S;
  int32_t bra0;
  int32_t nbra;
  int32_t ket0;   // first ket pair of the chunk's ket window
  int32_t nket;   // window length when the ket-side J is accumulated in LDS (0: global atomics)
  int32_t Sk;     // ket part of the primitive split S (powers of two)
  int32_t mol;    // its molecule
  // partial-sum slab of the chunk (per density): its exchange rows
  // [nbra][ROWS][n_m], then its ket window [nket][NKET]
  int64_t poff;
};

// Copies of each bra slot's J block in LDS: lane l adds into copy l % 8, so
// the lanes of a wavefront (which mostly share one bra) do not serialise on
// the same LDS addresses; the copies are summed at the flush.
constexpr int kJBraCopies = 8;

// What the bra-major kernels read of a ket pair and of its shells, in one
// record (five 16-byte loads a lane, two where both shells are s, in place of
// ten or more loads from the pair, shell and column tables: the address units
// are busy for 46 to 78 % of (ss|ss), (ps|ss) and (ps|ps) even so).
// With the bra records and the staging of all slots at once: 64 water clusters
// 4.70 -> 4.49 ms a build, in-core (H2O)8 cc-pVDZ 470 -> 440 us, (H2O)16 2.72 -> 2.66 ms.
struct alignas(16) KetRec {
  int poff, np;    // primitive-pair range
  int oc, od;      // Cartesian AO offsets inside the molecule
  int kc, kd;      // LDS exchange-row columns of the shells
  int lc, ld;      // segmented-shell indices inside the molecule
  double C[3], CD[3];  // first centre, first minus second
};

// The same of a chunk's bra pairs, one per slot in LDS.
struct BraRec {
  double A[3], AB[3];
  int poff, np, oa, ob, la, lb;
  int first, pad;  // first staged primitive record
};
constexpr int kBraRecDoubles = sizeof(BraRec) / sizeof(double);

struct BraArgs {
  const Pair* pairs;
  const KetRec* kets;   // per pair
  const PrimPair* prims;
  const ShellXYZ* shells;
  const int2* quartets;
  const BraChunk* chunks;
  int nchunks;
  int nbra_max;         // LDS slots per workgroup
  const double* dens;   // [nbd][sum_m n_m^2]
  double* jp;
  double* kp;
  const MolInfo* mols;
  int64_t bstride;
  int n, nbd, nbj, with_j, with_k;  // n: widest molecule (LDS row length)
  // mixed precision: FP32 for quartets with pair_q[bra] pair_q[ket] dmax6 < thr
  int mixed;
  double thr;
  const double* pair_q;  // Schwarz bound per pair
  const double* dmax;    // per molecule [nseg][nseg] max |D| over shell blocks (all batches)
  const PrimCoef* coef;  // column coefficients of a contracted pair set (general patterns)
  int tab_lds;           // stage the class's Rys table slice in LDS (after the slabs)
  int nket_max;          // LDS ket-J window capacity in ket pairs (0: ket-side J by global atomics)
  int threads;           // workgroup size (256 or 512)
  // ket-side J with one 64-byte line per element (element i of jp at
  // jket_pad[8 i]), so atomics to neighbouring J elements do not share a line
  double* jket_pad;
  // in-core integrals: 0 evaluates quartets, 1 evaluates and stores each
  // contracted Cartesian block (the slice of one ket component for split
  // classes) at cache[(quartet * SPLIT + kc) * block], 2 reads them back
  int mode;
  double* cache;
  // partial sums instead of flush atomics: bit 0 stores the exchange rows, bit
  // 1 the ket window, into part[bt * part_stride + chunk.poff + ...] with plain
  // stores; reduction kernels add them into K and J afterwards
  int part_mode;
  int64_t part_stride;
  double* part;
  // exchange-row slab columns: per (molecule, ket mask) the first entry in
  // colmap and the count of the molecule's Cartesian columns whose shell l is
  // in the mask; this class's mask (1 << lc | 1 << ld)
  const int* colmap;
  const int2* cspace;
  int cmask;
  // LDS exchange rows over the same compact columns (segmented sets): per
  // shell and mask its first compact column; NULL: rows over all n columns
  const int* shell_cofs;
  // deterministic digestion: [nmol][2] (scale, 1/scale) of the build; NULL
  // for FP64 atomics (tab_lds 0, mixed 0 and part_mode 0 with it)
  const double* det_scale;
  // bra primitive pairs of the chunk staged in LDS (full-block segmented
  // classes): capacity in records of kStagedPrim doubles, 0 = not staged
  int bra_stage;
};

// Doubles per staged primitive pair: p, P - A (A: the pair's first centre),
// e, 1/p; a bra with general-contraction columns adds c_A[2], c_B[2].
constexpr int kStagedPrim = 6;
constexpr int kStagedPrimCoef = kStagedPrim + 4;

struct ParamArgs {
  const Pair* pairs;
  const PrimPair* prims;
  const PrimAux* aux;
  const ShellXYZ* shells;
  const int* seg_prim0;  // first primitive slot of each segmented shell
  const int2* quartets;
  const SubTask* tasks;
  int ntasks;
  int64_t nitems;
  int64_t item0;         // first item of this launch (set by the launcher, with nitems its end)
  const double* dens;
  const double* cj;
  const double* ck;
  const MolInfo* mols;
  int nprim;             // primitive slots over all segmented shells
  double* gcoef;         // [nprim] dE/d(coefficient incl. s/p factor)
  double* gexp;          // [nprim] dE/d(exponent) at fixed coefficients
};

// Explicit quartet list writing contracted Cartesian blocks:
// out[base + sum_slot (coff[slot] + comp[slot]) * stride[slot]] for class-order slots A,B,C,D.
struct BlockTask {
  int bra, ket;
  int64_t base;
  int stride[4];
  int coff[4];
};

struct BlockArgs {
  const Pair* pairs;
  const PrimPair* prims;
  const ShellXYZ* shells;
  const BlockTask* tasks;
  int64_t ntasks;
  double* out;
};

// ----------------------------------------------------------------------------
// Density-fitting integrals (A B|C u), u the unit function
// ----------------------------------------------------------------------------
constexpr int kDfMaxL = 4;      // auxiliary shells up to g
constexpr int kDfMaxFun = 15;   // functions of one shell
constexpr int kDfMaxTerms = 6;  // Cartesian terms of one real solid harmonic up to g

// One requested-basis function as a sum of its shell's Cartesian components.
struct SphTerm {
  int n;
  int idx[kDfMaxTerms];
  double c[kDfMaxTerms];
};

// Bra pairs [pair0, pair0 + npair) of one class (la, lb) with similar
// primitive counts: T (bra pair, ket shell) tasks per block, each on
// S (x ket components) lanes, blocks from block0 on (negative where the range
// began in an earlier launch: its first task here is -block0 T).
struct DfRange {
  int la, lb;
  int pair0, npair;
  int S, T;
  int64_t block0;
};

// Lanes over ket components: blocks of more than 36 Cartesian components do
// not fit one lane's registers.
__host__ __device__ constexpr int df_ncart(int l) { return (l + 1) * (l + 2) / 2; }
__host__ __device__ constexpr int df_split(int la, int lb, int lc) {
  return df_ncart(la) * df_ncart(lb) * df_ncart(lc) > 36 ? df_ncart(lc) : 1;
}

struct DfArgs {
  const Pair* pairs;
  const PrimPair* prims;
  const ShellXYZ* shells;   // ao: first AO in the requested basis (auxiliary: in the auxiliary set)
  const DfRange* ranges;    // bra ranges of this launch
  int nrange;
  int ket0, nket;           // ket pairs (C, u) of this launch's angular momentum
  int layout;               // 3: out[c][pair(a, b)], 2: out[a][c]
  int64_t np, m;            // row lengths of the two layouts
  const SphTerm* terms;     // [l][kDfMaxFun]
  int nfun[kDfMaxL + 1];
  double* out;
};

// ----------------------------------------------------------------------------
// Packed ERIs
// ----------------------------------------------------------------------------
// Tasks (bra pair, ket pair) of two pair ranges with similar primitive counts
// (tri: one range with itself, ket <= bra): T per block on S = Sb * Sk lanes
// (x ket components) each, blocks from block0 on (negative where the range
// began in an earlier launch: its first task here is -block0 T).
struct EriRange {
  int bra0, nbra, ket0, nket;
  int S, Sk, T, tri;
  int64_t block0;
};

struct EriArgs {
  const Pair* pairs;
  const PrimPair* prims;
  const ShellXYZ* shells;   // ao: first AO in the requested basis
  const EriRange* ranges;   // ranges of this launch
  int nrange;
  int layout;               // 0: symmetric pair matrix, 1: s8 triangle
  int64_t np;
  const SphTerm* terms;     // [l][kDfMaxFun]
  int nfun[kDfMaxL + 1];
  double* out;
};

// Schwarz blocks (pq|pq) of the pairs of one class: q[2 i] = max over the
// requested-basis functions, q[2 i + 1] over the Cartesian components.
struct SchwarzArgs {
  const Pair* pairs;
  const PrimPair* prims;
  const ShellXYZ* shells;
  int npairs;
  const SphTerm* terms;     // [l][kDfMaxFun]
  int nfun[kDfMaxL + 1];
  double* q;
};

// Pair classes for l <= 2: index la*(la+1)/2 + lb with la >= lb.
constexpr int kNumPairClasses = 6;
__host__ __device__ constexpr int pair_class(int la, int lb) { return la * (la + 1) / 2 + lb; }

void launch_jk_class(int la, int lb, int lc, int ld, const JKArgs& a, hipStream_t s);
void launch_jk_bra_class(int la, int lb, int lc, int ld, const BraArgs& a, size_t lds_bytes, hipStream_t s);
struct GradArgs {
  const Pair* pairs;
  const PrimPair* prims;
  const ShellXYZ* shells;
  const int* seg_atom;   // atm row of each segmented shell
  const int2* quartets;
  const SubTask* tasks;
  int ntasks;
  int64_t nitems;
  int64_t item0;         // first item of this launch (set by the launcher, with nitems its end)
  const double* dens;    // Cartesian D, cot_J, cot_K (per molecule n x n); cot may be null
  const double* cj;
  const double* ck;
  const MolInfo* mols;
  int natm;
  double* grad;          // [natm][3]
};

void launch_grad_class(int la, int lb, int lc, int ld, const GradArgs& a, hipStream_t s);
void launch_blocks_class(int la, int lb, int lc, int ld, const BlockArgs& a, hipStream_t s);

}  // namespace gscf
