// Block responses: the scan with T steps at a time.
//
// The map x_{e+1} = M x_e + v_e is linear and time-invariant, so over a block
// of T = 2^lb steps the state at the block's end and the T outputs inside it
// are fixed linear functions of the state at its start and of the block's
// input samples.  A solve then is
//   pass 1: per block, its response from zero at its end  (one product with Q)
//   scan:   the states at the blocks' starts (n_a values a block)
//   pass 2: per block, its T outputs                      (one product with
//           [O H]: the outputs' responses to the state and to the samples)
// in place of T dependent steps, and no state inside a block is formed.
//
// To make a block need only its own samples, the state is shifted by the
// samples that an element and its successors share: with the direct terms
//   Z_e = X_e - sum_{r < taps} D_r u_{e,r},
// Z_{e+1} = M Z_e + G u_e, where u_e are the s samples that element e adds
// (RK4: rows 2e and 2e + 1, taps = 1; ABM: one row, taps = 4), and
// y_e = C x(Z_e) + sum_{r < taps} F_r u_{e,r}.
//
// Everything is FP64 on the matrix cores (v_mfma_f64_16x16x4f64).
// Tables (device, row-major; m inputs, p outputs, kb = s T m):
//   PT [L][na][na]     transposed powers, PT_l = (M^(2^l))^T
//   QT [kb][na]        row (s i + q) m + j: (M^(T-1-i) G_q)[:, j]
//   OT [na][T p]       column i p + o: row o of C E M^i (E: the state block read)
//   Ht [(s (T-1) + taps) m][p]  row d m + j, d = window row - s i + s (T - 1):
//                      the response of output o of step i to input j
//   DL [taps m][na]    the shift of the state
// The factors of column (i, o) for window value k = row m + j are
// Ht[(k + s (T-1-i) m) p + o]: linear in k, so pass 2 needs no row index.
#pragma once
#include "kernels.h"

namespace parode {
namespace k {

struct BlockShape {
    int method = 0, n = 0, m = 0, p = 0, na = 0;
    bool useC = false, useD = false;   // useC false: the outputs are the states (p = n)
    bool mirror = false;               // the reference's float rounding of the map
    int lb = 0, T = 0;                 // steps per block
    int L = 0;                         // powers in PT
    int s = 0, taps = 0;
    bool wide = false;   // the map does not fit one work-group: made by products over many
    // Where P_l lies in PT (in matrices).  Wide: from P_lb on the powers lie in
    // threes, P_l^3, P_{l+1}, P_l (l - lb even): the factors of a radix-4 level
    // of the tree, stacked.
    int slot(int l) const
    {
        return !wide || l < lb ? l : lb + 3 * ((l - lb) / 2) + ((l - lb) & 1 ? 1 : 2);
    }
    int slots() const { return wide ? lb + 3 * ((L - lb) / 2 + 1) : L; }
    bool radix4() const { return wide && na <= 256; }
    int kb() const { return s * T * m; }
    int kh() const { return (s * (T - 1) + taps) * m; }
};

// Block responses of one system: tables and states carved by ScanCore.
struct BlockBufs {
    double *PT = nullptr, *QT = nullptr, *OT = nullptr, *Ht = nullptr, *DL = nullptr;
    double* Z = nullptr;    // [blocks + 1][na]: aggregates
    double* E = nullptr;    // the blocks' start states (Z's place unless wide)
    double* Z2 = nullptr;   // [groups + 1][na]: the same for groups of blocks (wide: for
                            // every level of the tree over the blocks)
    double* W = nullptr;    // wide: the map's intermediate products
};

// Where a batch's samples lie: window row r of block b is the sample row
// b T sL + r g (sL sample rows a step, g = sL / s); rows past `last` (in window
// rows) are not there and count as zero.
struct BlockInput {
    const void* U = nullptr;
    bool isDouble = false;
    long sL = 0;
    long last = 0;
};

// Steps per block for a shape and horizon, 0: this shape keeps the general
// path (see the rule at its definition).
int block_steps_log(int method, int n, int m, int p, bool useC, bool useD, long nScan, long nPad);
BlockShape block_shape(int method, int n, int m, int p, bool useC, bool useD, bool mirror, int lb,
                       int L);
// How a pass is tiled (kBlockAuto: by the rule at pass_tiling).
enum BlockTiling { kBlockAuto = 0, kBlockTile = 1, kBlockSplit4 = 2, kBlockSplit16 = 3, kBlockMid = 4 };
// Groups of blocks that the scan of nb blocks makes first (0: none).
long block_groups(long nb);

// doubles in QT, OT, Ht and DL together; in the states for at most nb blocks; in W
size_t block_table_values(const BlockShape& s);
size_t block_state_values(const BlockShape& s, long nb);
size_t block_scratch_values(const BlockShape& s);
BlockBufs block_carve(const BlockShape& s, double* PT, double* tab, double* z, long nb, double* w);

// ---- wide maps: the launches that make the tables, as operations by phase (an
// operation reads what lower phases wrote)
struct BlkElem {        // element-wise stages of a wide map
    enum Stage { kPrep, kComb, kAsm };
    BlockShape s;
    int stage = 0;
    double h = 0.0;
    Rk4Coef rk;
    AbmCoef ab;
    const float *A, *B, *C, *D, *x0;
    double *PT, *QT, *OT, *DL, *seed;
    double *A64, *B64, *A2, *A3, *A4, *AB, *A2B, *A3B, *CT, *DT, *B1, *VT;
    long count = 0;     // elements
    long gx = 0;
};
struct SeqOp {          // Z = X Y in the reference's float rounding
    int r, kk, c;
    const float *X, *Y;
    float* Z;
};
struct BlockSink {
    virtual void gemm(int phase, const GemmOp& op) = 0;
    virtual void elem(int phase, const BlkElem& e) = 0;
    virtual void seq(int phase, const SeqOp& op) = 0;
    virtual ~BlockSink() = default;
};
// Emits a wide map's operations.  Returns the phase before which pass 1's
// table is not complete.  The powers up to P_last (P_0 .. P_{last}) are made;
// those that pass 1's tables do not need come at the phases they can.  ready, if
// given, receives for each power the phase from which it can be read.
int block_emit(const BlockShape& s, const BlockBufs& b, double h, const float* A, const float* B,
               const float* C, const float* D, const float* x0, double* seed, int last,
               BlockSink& sink, std::vector<int>* ready = nullptr);
// The tree over the blocks' states of a wide map: up products by pairs (level k
// from 0, with the power lb + k), the root's seed, the states at the top one after
// the other (step i from 0), down products (step j from 0).
int block_tree_up_levels(const BlockShape& s, long nb);
int block_tree_top_steps(const BlockShape& s, long nb);
GemmOp block_tree_top(const BlockShape& s, const BlockBufs& b, long nb, int i);
int block_tree_down_steps(const BlockShape& s, long nb);
GemmOp block_tree_up(const BlockShape& s, const BlockBufs& b, long nb, int k);
std::vector<GemmOp> block_tree_down(const BlockShape& s, const BlockBufs& b, long nb, int j);
// the root, the top and the down steps
void block_tree_finish(hipStream_t st, const BlockShape& s, const BlockBufs& b,
                       const BlockInput& in, long nb, const double* seed);
void block_elem(hipStream_t st, const BlkElem& e);

// M, G, the direct terms, the tables (P_0 .. P_lb) and (x0 given) the seed: x0, or
// the ABM start-up's states x_0..x_3 and its three outputs.  (Maps that are not wide.)
void block_tables(hipStream_t st, const BlockShape& s, const BlockBufs& b, double h, const float* A,
                  const float* B, const float* C, const float* D, const float* x0, const void* U,
                  bool uDouble, double* seed, float* Y);
// the outputs of the ABM start-up states (X0: x_0 .. x_3)
void block_start_outputs(hipStream_t st, const BlockShape& s, const float* C, const float* D,
                         const double* X0, const void* U, bool uDouble, float* Y);
// the blocks' responses from zero (and, with powers, the rest of PT)
void block_pass1(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                 long nb, bool powers, int tiling = kBlockAuto);
// the blocks' start states from the seed (in X); Z[nb] is the state after them (of a
// map that is not wide)
void block_scan(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                long nb, const double* seed);
// seedOut = the state (in X) after the blocks
void block_carry(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                 long nb, const double* seed, double* seedOut);
void block_pass2(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                 long nb, long nReal, const double* seed, const float* D, float* Y,
                 int tiling = kBlockAuto);

// ---- the same launches for many systems in one grid (FP64 samples)
namespace g {
void add_block_tables(Phase& ph, const BlockShape& s, const BlockBufs& b, double h, const float* A,
                      const float* B, const float* C, const float* D, const float* x0, double* seed);
void add_block_elem(Phase& ph, const BlkElem& e);
void add_block_start_outputs(Phase& ph, const BlockShape& s, const float* C, const float* D,
                             const double* X0, const double* U, float* Y);
void add_block_pass1(Phase& ph, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                     long nb);
void add_block_pass2(Phase& ph, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                     long nb, long nReal, const double* seed, const float* D, float* Y);
// the scan of a map that is not wide: up and down are used when the blocks go in groups
void add_block_scan(Phase& up, Phase& all, Phase& down, const BlockShape& s, const BlockBufs& b,
                    const BlockInput& in, long nb, const double* seed);
// the root of a wide map's tree
void add_block_root(Phase& ph, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                    long nb, const double* seed);
}  // namespace g

}  // namespace k
}  // namespace parode
