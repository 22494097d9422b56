// Host-side plan of the one-launch triangular sweeps (sweep.hip): which
// rows a block walks together, in which order, and which values pass
// between blocks.  No counterpart in the reference, whose sweeps are
// sequential loops over the cells.
#pragma once
#include <string>
#include <vector>

namespace fvk {

// A triangular pattern in the sweep's order: rank k (0 .. n-1) is the k-th
// row of the forward sweep.  Entries keep the order in which the reference
// takes them.  vals: index of the entry's value in the caller's value
// arrays; tvals: index of the transposed entry's value (lower side only).
struct SweepGraph {
  int n = 0;
  std::vector<int> row;          // device row of each rank
  std::vector<int> lptr, lcol, lval, tval;
  std::vector<int> uptr, ucol, uval;
  bool symmetric = false;        // the upper entries are the lower ones transposed
};

// at most kChunk rows are run together by the lanes of one wave
constexpr int kChunk = 64;
// positions a row at most (SweepPlan::width)
constexpr int kPadding = 8;
// LDS of one block: 160 KiB less the kernel's few shared scalars
constexpr int kSweepLds = 163840 - 256;

// The parts, in the order in which the forward sweep may take them (the
// backward sweep takes them from the last to the first).  A part's rows are
// packed into chunks of at most `width` rows that do not depend on each
// other, in an order in which every row follows the rows it depends on; the
// backward sweep walks the chunks from the last to the first.  Position p =
// width chunk + lane.  Inside a part a row's value sits in an LDS slot: own
// rows first, then (per direction) the halo, values of rows of other parts
// in the order in which the chunks need them, a slot that stays zero (for
// padding entries) and one that padding lanes write.
// The width is kChunk unless padding would then take more than kPadding
// positions a row: a chunk of a narrow pattern has few rows (one on a chain),
// and a position costs 148 bytes of tables and more.  Then it is the largest
// power of two that keeps to kPadding; 8 always does.  (A chain of 20,000 rows:
// 64 positions a row -> 8, its context made in 27 ms -> 9, DIC, both sweeps,
// 3.74 ms -> 3.77, for a vector register that holds the shift; 128^3, which
// stays at 64: 205 us both.)
struct SweepPlan {
  int n = 0, P = 0, W = 0, MW = 0, np = 0, levels = 0, width = kChunk;
  int slots = 0, maxh = 0;                 // the most LDS slots and halo values of a part
  bool bricks = false;
  double us = 0, chunk_us = 0;             // both sweeps by this plan (0: bricks of an exactly structured
                                           // numbering) and by chunks of the level order (sweep_plan_us)
  bool chunks_faster() const { return 1.25 * us > chunk_us; }
  std::vector<int> part;                   // 8 ints a part: first chunk, chunks, first row, rows,
                                           // first forward halo, count, first backward halo, count
  std::vector<int> prow, ppos;             // rows of each part ascending: device row, position
  std::vector<unsigned short> pslot;       // ... and LDS byte offset
  struct Dir {
    int NE = 0;                            // values passed between parts
    std::vector<unsigned short> rec;       // record of each position, nrec() words: own LDS byte offset, the
                                           // entries', halo values needed so far, export index (2 words, -1 none)
    std::vector<int> val;                  // MW x np: value index of each entry, -1 padding
    std::vector<int> hsrc;                 // export index of each halo value
  } d[2];                                  // forward, backward
  std::vector<int> tval;                   // MW x np: transposed value index of the lower entries
  int nrec() const { return MW <= 4 ? 8 : 16; }
  int at_need() const { return MW <= 4 ? 5 : 9; }
  // LDS of a block with nc values per slot: the slots and the halo's sources
  size_t lds(int nc) const { return (size_t)8 * nc * slots + (size_t)4 * maxh; }
};

// max_rows: rows of a part at most.  limit: positions at most (0, or more
// than the kernels take: what a 32-bit byte offset into the records reaches,
// 2^28 positions, 2^27 of rows with more than four entries a side).  Empty
// string, or why there is no plan: a row with more than 8 entries on one
// side, or too many positions.
std::string sweep_plan(const SweepGraph &g, int max_rows, SweepPlan &p, long limit = 0);

// us of both sweeps by this plan with one right-hand side, by a model
double sweep_plan_us(const SweepPlan &p);

// Walks the plan as the kernels do and checks that every value is there
// when it is read, that a part only needs parts taken before it, and that
// every row is run once.  Empty string, or the first fault.
std::string sweep_plan_check(const SweepGraph &g, const SweepPlan &p);

}  // namespace fvk
