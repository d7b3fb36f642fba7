// rr_kernels.h -- launch descriptors of the fitness kernels (host side of
// the kernels, used by the C-ABI implementation).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/rr_fitness.h"

namespace rr {

// One dataset as the kernels see it.  A launch carries a table of these and,
// per candidate, the index of the one it is scored against (cand_ds; null
// means entry 0 for every candidate), so candidates of independent runs over
// different datasets can share one launch.
struct DsDesc {
  const double* X;    // feature-major FP64, column stride ldx
  const float* X32;   // FP32 copy, same layout
  const double* y;
  int64_t n, ldx;
  double sst, ysum, yy;   // sum (y - mean)^2 (canonical order), sum y, sum y^2
  const double* one;      // ldx ones: the column of the OLS free term
  const double* xnorm;    // per feature: sums of squares over rows >= 0 and >= 1 (chunked order)
};

// Step-synchronous column-pivoted QR over the positions 0..n_pos-1 of a
// launch (sorted by column count, most first; pointers already offset to the
// launch's first position): launch_qr_init, then per step p launch_qr_step
// over the first n_act positions (those with more than p columns) and their
// chunk work items, then launch_qr_solve.  ks: the most columns of any
// position; phys: n_pos x ks ints; cold: 5 x n_pos x ks doubles; part: 2 ks
// doubles per chunk work item.
struct QrState {
  int32_t k, size, p, nonzero, nan_exit, steps, flags, papply;
  int32_t qphys0, qphys1, qapply, pad;   // the third-to-last step: its two A targets, reflector applied
  double thr, tau, den;
  double ptau, pden, ptd0, ptd1;          // the second-to-last step's reflector and dot products
  double qtau, qden, qtd0, qtd1, qtd2;    // the third-to-last step's (targets qphys0, qphys1, y)
};
struct QrLaunch {
  const int32_t* cand_start;
  const DsDesc* ds;
  const int32_t* cand_ds;
  double* coefs;
  rr_fit* fit;
  const int32_t* dead;
  int32_t* info;              // per candidate: -1 (fitness written) or rank | steps << 16 (to be scored)
  const int32_t* order;       // launched position -> candidate
  double* slab;
  const int64_t* slab_off;    // per launched position
  const int32_t* pos_item;    // per launched position: first chunk work item
  int items_per_pos;          // > 0 when every position has that many chunk items
  int n_pos;
  const double* norm_part;    // the evaluation's chunk sums (EvalLaunch::norm_part)
  const int32_t* prog_item;   // per non-bare program: the first evaluation work item of its factor
  const int64_t* prog_kept;   // per program: slab offset of its factor's kept column, or ~v: the bare variable v
  QrState* st;
  int32_t* phys;
  double* cold;
  int ks;
  double* part;
};

// Chunked column-pivoted QR of the FP64 OLS form, for candidates with at most
// TS_MAX_COLS columns (free term included):
//   launch_ts_init   one wave per position: the initial norms (from the
//                    evaluation's chunk sums), the outcome when step 0 would
//                    pivot a non-finite column, the finite columns, the rank
//                    threshold;
//   launch_ts_chunk  per column bucket, a grid of workgroups over the chunk
//                    work items of the bucket's live positions (the lists
//                    launch_alive_fp64 wrote): unpivoted Householder QR of a
//                    chunk of TS_ROWS rows of [finite columns | y], its
//                    triangular factor to rpart;
//   launch_ts_solve  the chunk factors combined in two levels -- one wave
//                    per (position, group of TS_GROUP consecutive chunks)
//                    folds the group's factors in chunk order into the slot
//                    of its first chunk, then one wave per position folds
//                    the group factors in group order -- and on the result
//                    the pivoted steps and the solve; coefficients, info (as
//                    the step-synchronous QR).  max_chunks: the most chunks
//                    of any position in the range.
// Positions pos0..pos1-1 of the arrays (pointers not offset).  Column buckets
// 0 .. 3: up to 10, 7, 5, 3 columns with y (ts_list).  Position p's chunk
// factors sit at rpart + rp_off[p] + chunk * W, W = nc * (nc - 1) words, nc =
// ts_bucket of its columns.
constexpr int TS_MAX_COLS = 9;
constexpr int64_t TS_ROWS = 4096;
constexpr int TS_GRID = 2048;   // workgroups of a chunk launch at most
constexpr int TS_GROUP = 16;    // chunks per group of the two-level combination
constexpr int TS_BUCKETS = 4;   // column buckets of the chunk launches
// The work lists of the chunk launches, of one launch chunk: the live
// positions of each bucket (bucket b's at live + pos0[b], cnt[b] of them, in
// position order).  A bucket's chunk work items are all chunks of its live
// positions, chunk by chunk (items_per_pos > 0: every position has that many;
// a chunk's columns, most of them shared by the candidates of a sweep, are
// then read by all positions at about the same time), or, for positions of
// several datasets, the (position, chunk) pairs at items + 2 item0[b],
// cnt[TS_BUCKETS + b] of them, position p's from base[p] on.
struct TsList {
  int32_t* cnt;     // 2 TS_BUCKETS
  int32_t* live;    // per position
  int32_t* base;    // per position (items_per_pos == 0)
  int32_t* items;   // 2 per chunk work item (items_per_pos == 0)
  int32_t pos0[TS_BUCKETS + 1], item0[TS_BUCKETS];
  int32_t items_per_pos;
};
// What launch_alive_fp64 needs to write one: the positions' candidates and
// datasets.
struct LiveLaunch {
  const int32_t* order;
  const DsDesc* ds;
  const int32_t* cand_ds;
  TsList list;
};
struct TsState {
  int32_t k, kf, size, live;            // live: 1 when the chunk and solve kernels have work
  int32_t fin[TS_MAX_COLS];             // the finite columns, in column order
  int32_t nch, pad;
  int64_t n;
  double thr;
  double nd[TS_MAX_COLS];               // initial column norms
  const double* col[TS_MAX_COLS + 1];   // the finite columns' data, then y
};
struct TsLaunch {
  const int32_t* cand_start;
  const DsDesc* ds;
  const int32_t* cand_ds;
  double* coefs;
  rr_fit* fit;
  const int32_t* dead;
  int32_t* info;
  const int32_t* order;       // position -> candidate
  const double* slab;
  const double* norm_part;
  const int32_t* prog_item;
  const int64_t* prog_kept;
  const int64_t* rp_off;      // per position: offset of its chunk factors in rpart
  TsState* st;
  double* rpart;
  TsList list;
};
hipError_t launch_ts_init(const TsLaunch& L, int pos0, int pos1, hipStream_t s);
// bucket 0 .. 3; max_items: the bucket's chunk work items if every position
// were live
hipError_t launch_ts_chunk(const TsLaunch& L, int bucket, int max_items, hipStream_t s);
hipError_t launch_ts_solve(const TsLaunch& L, int pos0, int pos1, int64_t max_chunks, hipStream_t s);
// the column count with y that fixes the order of the sums of a candidate
// with k columns (free term included, k <= TS_MAX_COLS; the oracle's
// ts_bucket), and the threads of that order (the oracle's ts_dot): 256
// threads of 16 rows for 3 and 5 columns, 1024 of 4 rows for 10
__host__ __device__ inline int ts_bucket(int k) { return k <= 2 ? 3 : k <= 4 ? 5 : 10; }
__host__ __device__ constexpr int ts_threads(int nc) { return nc <= 5 ? 256 : 1024; }
// the launch bucket of a candidate with k columns, the most columns with y it
// takes, and its workgroup: the wide bucket is split so that a chunk of up to
// 7 columns fits the registers of four waves (16 rows a thread); up to 10
// take eight waves (8 rows a thread)
__host__ __device__ inline int ts_list(int k) { return k >= 7 ? 0 : k >= 5 ? 1 : k >= 3 ? 2 : 3; }
__host__ __device__ constexpr int ts_block(int nc) { return nc <= 7 ? 256 : 512; }

// Scoring of the FP64 form: per (launched position, chunk of EVAL_CHUNK_ROWS
// rows) the chunk's sum of squared residuals -- RAW: of the candidate's one
// program; OLS: of the OLS tree from the coefficients and the factor columns
// (prog_kept), for the candidates whose info is >= 0 -- and then per position
// the chunk sums in order into the fitness.  Position p owns work items
// pos_item[p] .. pos_item[p+1]-1 (items_per_pos > 0: p * items_per_pos ..).
//
// ScorePack: the inputs of a small RAW call, at byte offsets of its words, as
// part of the kernel's argument: no staged copy before the kernel.  A staged
// copy is a kernel of its own (5 us and a dependency of the scoring), so a
// call of one tree on 150 rows takes 32.4 us with two copies and 21.6 us with none; the
// limit keeps the argument well inside the 4 KiB a launch can pass, room for
// about a dozen trees of 20 nodes.
constexpr int SCORE_PACK_BYTES = 3072;
struct ScorePack {
  int32_t cand_start, prog_start, code, K, ds, cand_ds, pos_item;   // cand_ds < 0: none
  uint64_t words[SCORE_PACK_BYTES / 8];
};
struct ScoreLaunch {
  const int32_t* cand_start;
  const int32_t* prog_start;
  const uint32_t* code;
  const double* K;
  const DsDesc* ds;
  const int32_t* cand_ds;
  const double* coefs;       // OLS
  const double* slab;        // OLS
  const int64_t* prog_kept;  // OLS, per program (QrLaunch's)
  const int32_t* order;      // launched position -> candidate (null: identity)
  const int32_t* dead;       // or null
  const int32_t* info;       // OLS: written by the QR (k_ts_init / k_ts_solve, or k_qr_init / k_qr_solve)
  const int32_t* pos_item;
  int n_pos;
  int n_items;
  int items_per_pos;
  int raw;
  int rows, form, depth;     // RAW: as EvalLaunch's
  double* part;              // per work item
  rr_fit* fit;
  // RAW, a small call: the input arrays packed in host memory at multiples of
  // 8 bytes and passed with the launch (the pointers above are unused then)
  const ScorePack* pack;
};

// Factor-0 pre-pass of the OLS form: one workgroup per candidate evaluates
// factor 0 in FP64 on rows 0..NAN0_ROWS-1.  A NaN at a row >= 1 fixes the outcome (every
// coefficient NaN, the sentinel fitness; the FP64 kernel reaches the same
// result when it sees it), which is written here; dead[c] = 1 then, else 0.
struct Nan0Launch {
  const int32_t* cand_start;
  const int32_t* prog_start;
  const uint32_t* code;
  const double* K;
  const DsDesc* ds;
  const int32_t* cand_ds;
  double* coefs;
  rr_fit* fit;
  int32_t* dead;
  int n_cands;
};
constexpr int NAN0_ROWS = 64;

// Factor evaluation of the FP64 OLS form into the kept slab columns: one
// workgroup per (unique factor, chunk of EVAL_CHUNK_ROWS rows).  A unique
// factor is a program over a dataset that one or more candidates use;
// factor f is program fac_prog[f] (~fac_prog[f] where negative: a program
// whose operand stack is deeper than EVAL_LDS_SLOTS) over the dataset of
// candidate fac_cand[f],
// kept at slab + fac_kept[f], and owns work items fac_item[f] ..
// fac_item[f+1]-1, n_items in all.  Work item b also leaves the sums of
// squares of its chunk in norm_part[2b], norm_part[2b+1].  Factors with
// alive[f] == 0 (every user candidate settled by the factor-0 pre-pass) are
// skipped.  Must run before the QR launches over the same candidates.
// At four rows a thread the LDS holds EVAL_LDS_SLOTS stack slots, 24 KiB, which
// six workgroups per compute unit fit; the deeper programs (one random tree of
// 50 nodes in 500) take one row at a time.  Sized for the deepest program of
// the launch, a batch of 4000 such trees on 1e5 rows took 1455 us of kernels
// with four programs of depth 4 among them and 1345 without; now 1345.
constexpr int EVAL_LDS_SLOTS = 3;
struct EvalLaunch {
  const int32_t* prog_start;
  const uint32_t* code;
  const double* K;
  const DsDesc* ds;
  const int32_t* cand_ds;
  double* slab;
  const int32_t* fac_prog;
  const int32_t* fac_cand;
  const int32_t* fac_item;
  const int64_t* fac_kept;
  const int32_t* alive;
  int n_facs;
  int n_items;
  int items_per_fac;         // > 0 when every factor has that many items (factor = item / items_per_fac)
  double* norm_part;         // 2 doubles per work item
  int rows;                  // rows per thread per pass: 1, 2 or 4
  int form;                  // 0: operand stack in registers, transcendentals called; 1: stack in LDS, inlined
  int depth;                 // the deepest operand stack of the launch's factor programs
};
constexpr int64_t EVAL_CHUNK_ROWS = 4096;   // the chunk of the norms' order (rrm::NORM_CHUNK)

hipError_t launch_qr_init(const QrLaunch& L, hipStream_t s);
hipError_t launch_qr_step(const QrLaunch& L, int n_act, int n_items, hipStream_t s);
hipError_t launch_qr_solve(const QrLaunch& L, hipStream_t s);
// The same QR (init, every step, solve) in one launch when every position has
// one chunk work item (n <= EVAL_CHUNK_ROWS); n_max: the most rows of any.
hipError_t launch_qr_all1(const QrLaunch& L, int64_t n_max, hipStream_t s);
hipError_t launch_eval_fp64(const EvalLaunch& L, hipStream_t s);
// alive[u] = 1 if some candidate users[ustart[u] .. ustart[u+1]-1] has
// dead == 0, else 0, for u < n; live (or null): the work lists of a launch
// chunk's chunked QR
hipError_t launch_alive_fp64(const int32_t* ustart, const int32_t* users, const int32_t* dead, int32_t n,
                             int32_t* alive, const LiveLaunch* live, hipStream_t s);
hipError_t launch_nan0_fp64(const Nan0Launch& L, hipStream_t s);
hipError_t launch_score_fp64(const ScoreLaunch& L, hipStream_t s);
// feature j of row i at X[j col + i row]
hipError_t launch_predict_fp64(const uint32_t* code, int len, const double* K, const double* X, int64_t n,
                               int64_t col, int64_t row, double* out, hipStream_t s);
// Dataset upload.  launch_place moves `count` values of the flat input [d
// columns of n rows | y], from flat index `at` on, to their padded columns
// (and the FP32 copies); launch_place_stats, after all of them, fills the rows
// past n and the column of ones and leaves xnorm[2f], xnorm[2f+1], the sums of
// squares of feature f's column over rows >= 0 and rows >= 1 in the chunked
// order (rrm::chunk_sum), and out4 = {mean(y), sum((y - mean)^2), sum(y),
// sum(y^2)}.  part: 2 doubles per feature and chunk of EVAL_CHUNK_ROWS rows.
struct DsPlace {
  double* X;
  float* X32;
  double* y;
  double* one;
  int64_t n, ldx;
  int d;
};
hipError_t launch_place(const double* src, int64_t at, int64_t count, const DsPlace& p, hipStream_t s);
hipError_t launch_place_stats(const DsPlace& p, double* part, double* xnorm, double* out4, hipStream_t s);

}  // namespace rr
