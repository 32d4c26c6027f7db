// mi_plan.h -- the host-side planning of the transducer-loss library: workspace layout, division constants,
// duration parameter blocks and the choice of kernel shape per problem shape.  Plain C++ with no HIP types, so that a
// CPU-only sanitizer build can exercise it (tests/native/fuzz_host.cpp); mi_transducer.hip includes it inside its
// anonymous namespace, ahead of the device code that uses these types.
#ifndef MI_PLAN_H_
#define MI_PLAN_H_

#include <stddef.h>
#include <stdint.h>

#include "mi_transducer.h"

constexpr int kCoefBase = 8;  // floats per cell in the coefficient buffer before the duration-gradient block
// The prefill segment of the workspace, in ints.  While a lattice kernel runs, HBM idles; "riders" (extra workgroups
// of the same launch) zero-fill the padded cells of the gradient meanwhile, as far as they get.
//   [0, kFillMaxLattice)                  per lattice workgroup: (epoch << 13) | (id of the compute unit it runs on + 1)
//   [kFillMaxLattice, 2*kFillMaxLattice)  per lattice workgroup: the epoch, once it has finished
//   [2*kFillMaxLattice, + kFillMaxRiders) per virtual rider: how many of its items have been filled
// An item is 2^prefill_log_rows rows of one frame (b, t), items are numbered in memory order, and item i is the
// (i / kFillMaxRiders)-th item of virtual rider i % kFillMaxRiders: it is done iff  i / kFillMaxRiders <
// progress[i % kFillMaxRiders].  A launch has a power of two of real riders, each standing for the virtual riders
// congruent to it.  Pass 1 clears the whole segment, and the first two blocks are stamped with an epoch that changes
// with every call, so what an earlier call left there is not mistaken for this call's -- also not in a captured
// graph, where the epoch is frozen -- and a record that no rider of this call wrote says that nothing is filled.
constexpr int kFillMaxLattice = 256;
constexpr int kFillMaxRiders = 4096;
constexpr int kFillProgress = 2 * kFillMaxLattice;
constexpr int kFillInts = kFillProgress + kFillMaxRiders;
constexpr int kFillLogRowsShift = 8;  // the gradient kernels find log2(rows per item) in these bits of `flags`
// Rows per item: eight (the gradient kernels that look at one item span no more rows and straddle no multiple of eight; a
// tile of short rows looks at up to 16 items), fewer for long rows, so that a rider looks at the lattice's state every 64
// KB or so
inline int prefill_log_rows(size_t row_bytes) {
  int log_rows = 3;
  while (log_rows > 0 && (row_bytes << log_rows) > 64 * 1024) --log_rows;
  return log_rows;
}

// ----------------------------------------------------------------------------------------
// Workspace layout
// ----------------------------------------------------------------------------------------
// A cell's arc log-probs are one record of consecutive floats -- blank, label, then the `extras` duration (TDT) or
// big-blank (multi-blank) log-probs -- so that the pass that forms them writes them with one store: 2 floats, or,
// when there are extras, a multiple of 4 (whole 16-byte pieces) whose LAST float is the cell's log-softmax
// denominator (the cell kernels of those losses read it there, and the pass saves the store into `denom`).
constexpr int arc_record_floats(int extras) { return extras <= 0 ? 2 : (3 + extras + 3) / 4 * 4; }

struct Layout {
  int K;    // lattice cells per lane (1,2,4,8,16)
  int Us;   // pitch of a skewed lattice row = 64*K >= U
  int ND;   // number of anti-diagonals of the padded lattice = T+U-1
  int A;    // floats of a cell's record of arc log-probs (arc_record_floats); a skewed row holds Us records
  int CS;   // floats per cell in the coefficient buffer
  size_t off_denom, off_arcs, off_alphas, off_betas, off_ll, off_coef, off_fill, total;
};

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

inline bool make_layout(int B, int T, int U, int D, Layout* L) {
  if (B <= 0 || T <= 0 || U <= 0 || D < 0 || U > MI_TRANSDUCER_MAX_U || D > MI_TRANSDUCER_MAX_DURATIONS) return false;
  int K = 1;
  while (64 * K < U) K *= 2;
  L->K = K;
  L->Us = 64 * K;
  L->ND = T + U - 1;
  L->A = arc_record_floats(D);
  L->CS = kCoefBase + ((D + 3) & ~3);
  const size_t cells = (size_t)B * T * U;
  const size_t skew = (size_t)B * L->ND * L->Us;
  size_t off = 0;
  L->off_denom = off;  off = align256(off + cells * sizeof(float));
  L->off_arcs = off;   off = align256(off + skew * L->A * sizeof(float));
  L->off_alphas = off; off = align256(off + skew * sizeof(double));
  L->off_betas = off;  off = align256(off + skew * sizeof(double));
  L->off_ll = off;     off = align256(off + (size_t)B * 2 * sizeof(double));
  L->off_coef = off;   off = align256(off + cells * L->CS * sizeof(float));
  L->off_fill = off;   off = align256(off + (size_t)kFillInts * sizeof(int));
  L->total = off;
  return true;
}

// n / d for n < 2^31 by one multiply and one shift (the round-up multiplier of Granlund and
// Montgomery, "Division by invariant integers using multiplication"): the hardware has no integer
// divide, and the two divisions that split a workgroup id into (b, t, chunk) would otherwise cost
// some sixty instructions at the head of every wave.
struct FastDiv {
  unsigned mul, shift;
};
inline FastDiv make_fastdiv(unsigned d) {
  unsigned l = 0;
  while ((1ull << l) < d) ++l;
  FastDiv f;
  f.mul = (unsigned)((((unsigned long long)1 << 32) * (((unsigned long long)1 << l) - d)) / d + 1);
  f.shift = l;
  return f;
}
// the two divisions that split a workgroup id into (b, t, chunk), in three words (the shifts share one): this block
// is among the kernel arguments that arrive in registers with the wave, where every word counts
struct GridDiv {
  unsigned mul_chunks, mul_T, shifts;  // shifts = shift of the division by nchunks | shift of the division by T << 8
};
inline FastDiv griddiv_chunks(const GridDiv& g) { return FastDiv{g.mul_chunks, g.shifts & 255u}; }
inline FastDiv griddiv_frames(const GridDiv& g) { return FastDiv{g.mul_T, g.shifts >> 8}; }
inline GridDiv make_griddiv(int nchunks, int T) {
  const FastDiv c = make_fastdiv((unsigned)nchunks), t = make_fastdiv((unsigned)T);
  return GridDiv{c.mul, t.mul, c.shift | (t.shift << 8)};
}


// Consecutive workgroups that one XCD takes per turn (logical_block, mi_device.inc).  Measured on the fwd+bwd step
// with riders (us; B=16, T=375, U=121, V=1025 fp32 / the same as TDT / as multi-blank / B=32, T=750, U=201 bf16 /
// V=16385): 512 -> 1110 / 1181 / 1110 / 3845 / 4996; 1024 -> 1116 / 1186 / 1125 / 3880 / 4990; at the first shape
// 32, 128, 256, 384, 640, 768, 2048, 4096 -> 1123, 1120, 1117, 1115, 1117, 1115, 1133, 1152 (long turns leave XCDs
// idle where an utterance's padding begins; short ones lose the linear walk).
#ifndef MI_XCD_SPAN
#define MI_XCD_SPAN 512
#endif
// The gradient pass over 16-bit rows wants shorter turns (its workgroups hold four rows of 2 KB where the fp32 ones
// hold two of 4 KB): B=32, T=750, U=201, V=1025 bf16: 32 / 64 / 128 / 256 / 512 -> 2556 / 2536 / 2547 / 2575 / 2601 us
// (step 3.76 against 3.83 ms); B=16, T=375, U=121 bf16: 361 / 360 / 359 / 363 / 378 us; the fp32 shapes all lose below
// 512 (T=750, U=201 fp32: 5413 / 5476 / 5328 us at 128 / 256 / 512).  Pass 1 does not care (1038 ... 1043 us).
// MI_XCD_SPAN is a multiple of it (grids are padded to a multiple of 8 * MI_XCD_SPAN).
#ifndef MI_XCD_SPAN_16
#define MI_XCD_SPAN_16 128
#endif
static_assert(MI_XCD_SPAN % MI_XCD_SPAN_16 == 0, "one grid padding must serve both turn lengths");

struct TdtParams {
  int D;
  int dur[MI_TRANSDUCER_MAX_DURATIONS];
  int one_idx;  // index of duration 1 (position 0 or 1)
  int R;        // ring depth
  float sigma;
};


struct MbParams {
  int NB;
  int dur[MI_TRANSDUCER_MAX_BIG_BLANKS];
  int R;  // ring depth: longest blank + 1
  float sigma;
};


inline int make_tdt_params(int D, const int32_t* durations, float sigma, TdtParams* p) {
  if (D <= 0 || D > MI_TRANSDUCER_MAX_DURATIONS || !durations) return MI_TRANSDUCER_INVALID_VALUE;
  p->D = D;
  p->sigma = sigma;
  for (int i = 0; i < MI_TRANSDUCER_MAX_DURATIONS; ++i) p->dur[i] = 0;
  for (int i = 0; i < D; ++i) {
    if (durations[i] < 0 || (i > 0 && durations[i] <= durations[i - 1])) return MI_TRANSDUCER_INVALID_VALUE;
    p->dur[i] = durations[i];
  }
  if (durations[0] == 1) p->one_idx = 0;
  else if (D > 1 && durations[1] == 1) p->one_idx = 1;
  else return MI_TRANSDUCER_INVALID_VALUE;
  p->R = durations[D - 1] + 2;
  return MI_TRANSDUCER_SUCCESS;
}


inline int make_mb_params(int NB, const int32_t* durations, float sigma, MbParams* p) {
  if (NB < 0 || NB > MI_TRANSDUCER_MAX_BIG_BLANKS || (NB > 0 && !durations)) return MI_TRANSDUCER_INVALID_VALUE;
  p->NB = NB;
  p->sigma = sigma;
  int longest = 1;
  for (int i = 0; i < MI_TRANSDUCER_MAX_BIG_BLANKS; ++i) p->dur[i] = 0;
  for (int i = 0; i < NB; ++i) {
    if (durations[i] < 1 || durations[i] > MI_TRANSDUCER_MAX_BLANK_DURATION) return MI_TRANSDUCER_INVALID_VALUE;
    p->dur[i] = durations[i];
    longest = durations[i] > longest ? durations[i] : longest;
  }
  p->R = longest + 1;
  return MI_TRANSDUCER_SUCCESS;
}


// ----------------------------------------------------------------------------------------
// Lattices on probabilities (mi_scaled.inc)
// ----------------------------------------------------------------------------------------
constexpr int kScaledMaxGroups = 4;  // 256 columns
// doubles per cell that a helper leaves in LDS: TDT the two tokens and durations 0 .. maxd, multi-blank the label and the
// blanks of duration 1 .. maxd; in whole pairs, the last of them free
constexpr int scaled_factors(bool tdt, int maxd) { return ((tdt ? 3 + maxd : 1 + maxd) + 1) / 2 * 2; }
constexpr size_t scaled_group_bytes(int factors, int steps) { return (size_t)steps * (1024 * (factors + 1) + 176); }
struct ScaledPlan {
  int longest;  // the longest duration the instantiation holds: 4 or 8; 0: the recursions on logarithms
  int steps;    // anti-diagonals a batch
  int helpers;  // helper waves per group of 64 columns
  int threads;
  size_t lds;
};
// Batches of 8 diagonals and four helpers a group, as far as LDS holds them and for one or two groups; beyond, batches of 4,
// and two helpers: four groups then have the twelve waves that a compute unit gives enough registers.
// longest == 0: longer durations, more than 256 columns (192 with a longest duration above 4), more LDS than there is.
constexpr ScaledPlan scaled_plan(bool tdt, int longest, int U) {
  const int groups = (U + 63) / 64, maxd = longest <= 4 ? 4 : 8, factors = scaled_factors(tdt, maxd);
  ScaledPlan p{0, 0, 0, 0, 0};
  if (longest > 8 || groups > kScaledMaxGroups) return p;
  for (int steps = 8; steps >= 4; steps -= 4) {
    const size_t lds = groups * scaled_group_bytes(factors, steps) + 16;
    if (lds > 160 * 1024 || (steps == 8 && groups > 2)) continue;
    const int helpers = groups > 2 ? 2 : 4;
    return ScaledPlan{maxd, steps, helpers, 64 * groups * (1 + helpers), lds};
  }
  return p;
}
// the largest workgroup that any plan launches an instantiation with
constexpr int scaled_threads(bool tdt, int longest, int steps, int helpers) {
  int most = 0;
  for (int groups = 1; groups <= kScaledMaxGroups; ++groups) {
    const ScaledPlan p = scaled_plan(tdt, longest, 64 * groups);
    if (p.longest == longest && p.steps == steps && p.helpers == helpers && p.threads > most) most = p.threads;
  }
  return most;
}
// offsets into an utterance's records are 32-bit (and run up to 256 diagonals past its end)
inline bool scaled_offsets_fit(const Layout& L) { return (L.ND + 256LL) * L.Us * L.A * 4 < (1LL << 31); }
inline ScaledPlan scaled_plan(const Layout& L, const TdtParams& p, int U) {
  return scaled_offsets_fit(L) ? scaled_plan(true, p.dur[p.D - 1], U) : ScaledPlan{0, 0, 0, 0, 0};
}
// (a blank arc has a factor of its own per duration: the big blanks' durations must differ, also from the standard blank's)
inline ScaledPlan scaled_plan(const Layout& L, const MbParams& p, int U) {
  bool distinct = p.NB > 0 && scaled_offsets_fit(L);
  for (int i = 0; i < p.NB; ++i) {
    distinct = distinct && p.dur[i] >= 2;
    for (int j = 0; j < i; ++j) distinct = distinct && p.dur[j] != p.dur[i];
  }
  return distinct ? scaled_plan(false, p.R - 1, U) : ScaledPlan{0, 0, 0, 0, 0};
}

// ----------------------------------------------------------------------------------------
// Kernel shape per problem shape.  The shape of a call as far as these choices go: logit dtype, tokens per row,
// extra row entries (TDT durations), lattice dimensions, and whether logits and gradients share their 16-byte phase.
// ----------------------------------------------------------------------------------------
struct PlanShape {
  int dt, B, T, U, V, D;
  bool same_phase;
  int vec() const { return dt == MI_DTYPE_F32 ? 4 : 8; }  // elements per 16-byte vector
  int whole_vectors() const { return V / vec(); }
};

#ifndef MI_USE_ROWS
#define MI_USE_ROWS 1
#endif
#ifndef MI_USE_BLOCK_ROWS
#define MI_USE_BLOCK_ROWS 1
#endif
#ifndef MI_ROW_WAVES
#define MI_ROW_WAVES 4
#endif
constexpr int kRowWaves = MI_ROW_WAVES;  // waves (= rows in flight) per workgroup of the row kernels

// Pass 1 of rows beyond 64 vectors, a wave per row: the smallest R of these with floor(V / VEC) <= 64*R, or 0 if the rows are
// too long for the register-resident kernels.
// (3, 5 and 6 as well: a vocabulary just past a power of two -- 1024 tokens, the blank and three big blanks are 257 vectors
// -- then costs 5 vector loads per lane, not 8)
inline int denom_rows_R(const PlanShape& s) {
  if (!MI_USE_ROWS) return 0;
  const int nb = s.whole_vectors();
  for (int r = 1; r <= 8; ++r)
    if (r != 7 && nb <= 64 * r) return r;
  return 0;
}

// Workgroup-per-row kernels: RT threads per row, NVT vectors per thread.  RT == 0: not applicable.
// The denominator pass uses them for rows too long for the register-resident wave-per-row
// kernels (more than 512 whole vectors).  The gradient pass uses them from 65 vectors up, with
// two vectors per thread where the row allows it: of the splits tried (1, 2 and 4 vectors per
// thread) that one streams fastest.
struct BlockPlan {
  int RT, NVT;
  int rows() const { return (RT < 256 ? 256 : RT) / RT; }
  int threads() const { return RT < 256 ? 256 : RT; }
};
inline bool block_rows_ok(const PlanShape& s) { return MI_USE_BLOCK_ROWS && 2 * s.vec() + s.D <= 64; }
inline BlockPlan denom_block_plan(const PlanShape& s) {
  const int nb = s.whole_vectors();
  if (!block_rows_ok(s) || nb <= 512) return BlockPlan{0, 0};
  for (int nvt = 1; nvt <= 8; nvt *= 2)
    if (nb <= 1024 * nvt) return BlockPlan{1024, nvt};
  return BlockPlan{0, 0};
}
inline BlockPlan grad_block_plan(const PlanShape& s) {
  const int nb = s.whole_vectors();
  if (!s.same_phase || !block_rows_ok(s) || nb <= 64) return BlockPlan{0, 0};
  for (int rt = 64; rt <= 1024; rt *= 2) {
    if (nb <= 2 * rt) return BlockPlan{rt, 2};
    // a row just past 2*rt vectors (1024 tokens + blank + big blanks = 257): a third, partly filled vector per
    // thread beats twice the threads with half of them idle -- measured up to about 2.5*rt (V = 1028 ... 2600);
    // towards 3*rt the wider workgroup wins again
    if (nb <= 2 * rt + rt / 2) return BlockPlan{rt, 3};
  }
  for (int nvt = 4; nvt <= 8; nvt *= 2)
    if (nb <= 1024 * nvt) return BlockPlan{1024, nvt};
  return BlockPlan{0, 0};
}
// 1-D grids are rounded up to a whole number of turns of the XCD permutation
inline unsigned padded_grid(long long blocks) {
  const long long turn = 8LL * MI_XCD_SPAN;
  return (unsigned)((blocks + turn - 1) / turn * turn);
}
inline int plan_chunks(const PlanShape& s, const BlockPlan& p) { return (s.U + p.rows() - 1) / p.rows(); }
inline long long plan_blocks(const PlanShape& s, const BlockPlan& p) { return (long long)plan_chunks(s, p) * s.B * s.T; }
// the row kernels: a workgroup takes kRowWaves * rpw consecutive rows of one (b,t)
inline int row_chunks(const PlanShape& s, int rpw) { return (s.U + kRowWaves * rpw - 1) / (kRowWaves * rpw); }
inline long long row_blocks(const PlanShape& s, int rpw) { return (long long)row_chunks(s, rpw) * s.B * s.T; }

// Short rows (at most 64 whole vectors): both passes take tiles of 1 << log_rows consecutive rows of one frame
// (mi_tile.inc), as many as make up to 17 KB -- four 16-byte vectors a thread and a few more, so that the usual vocabulary
// sizes, a power of two and a blank (and durations), do not fall to half a tile -- and no more than a frame needs.  Eight
// rows always fit (they are at most 9 KB).  Longer rows keep the kernels that give a row whole waves: from 65 vectors
// on every lane has work there (measured figures: mi_tile.inc).
constexpr int kTileBytes = 17 * 1024 - 16;
constexpr int kTileMaxRows = 128;
constexpr int kTileThreads = 256;
constexpr int kTileRounds = (kTileBytes + 16) / 16 / kTileThreads;  // aligned vectors a thread moves; a few move one more
static_assert(kTileRounds == 4, "a tile is four vectors a thread, and some");
struct RowTile {
  int log_rows;  // 0: not a short row
  int rows() const { return 1 << log_rows; }
};
inline RowTile row_tile(const PlanShape& s) {
  if (!MI_USE_ROWS || s.whole_vectors() > 64) return RowTile{0};
  const long long row_bytes = (long long)(s.V + s.D) * (16 / s.vec());
  int log_rows = 3;
  while ((2 << log_rows) <= kTileMaxRows && (row_bytes << (log_rows + 1)) <= kTileBytes && (1 << log_rows) < s.U) ++log_rows;
  return RowTile{log_rows};
}
inline int tile_chunks(const PlanShape& s, const RowTile& t) { return (s.U + t.rows() - 1) >> t.log_rows; }
inline long long tile_blocks(const PlanShape& s, const RowTile& t) { return (long long)tile_chunks(s, t) * s.B * s.T; }
// ... but for the gradient of 16-bit rows that give nearly every lane of a wave its vector (grad_rows_kernel): eight elements
// a vector, and a tile selects each element's coefficients (and looks for duration entries among them), which are
// wave-uniform there.  A float32 vector has half the selects for the same bytes, and tiles win.  Measured, step at B=16,
// T=375, U=121 (us, tiles / a wave a row), by whole vectors:
//   RNNT float32 49 279 / 309, 56 295 / 326, 64 322 / 353; bfloat16 36 276 / 310, 49 324 / 330, 56 345 / 345, 60 357 / 352,
//   64 373 / 370; multi-blank bfloat16 49 479 / 489, 56 500 / 506
//   TDT  float32 49 490 / 515, 64 535 / 564; 16 bits, five durations 34 511 / 519, 40 540 / 530, 48 571 / 543, 56 606 / 561,
//   two durations 34 425 / 444, 40 451 / 457, 44 463 / 462, 48 483 / 473
inline bool grad_by_rows(const PlanShape& s) {
  const int nb = s.whole_vectors();
  return MI_USE_ROWS && s.same_phase && s.vec() == 8 && nb > (s.D ? 40 : 56) && nb <= 64;
}
// Pass 1 over them: as many cells, but 16 (or a power of two that holds U) rows of each of several frames.
constexpr int kTileMaxFrames = 16;
// the pieces of a tile's frames each start and end inside a vector
constexpr int kTileVectors = kTileBytes / 16 + 2 * kTileMaxFrames;
// elements of a row a lane reduces (rows * V elements over the workgroup's threads, four at a time)
constexpr int tile_share(int element_bytes) { return (kTileBytes / element_bytes / kTileThreads + 4) / 4 * 4; }
struct DenomTile {
  int log_rows, log_frames;  // log_rows + log_frames: 3 ... 7
  int frame_groups;          // groups of frames per utterance
  int pitch;                 // 16-byte vectors that hold a frame's rows wherever they start
  FastDiv div_pitch;
};
inline DenomTile denom_tile(const PlanShape& s) {
  const long long row_bytes = (long long)(s.V + s.D) * (16 / s.vec());
  int log_cells = 3;
  while ((2 << log_cells) <= kTileMaxRows && (row_bytes << (log_cells + 1)) <= kTileBytes) ++log_cells;
  DenomTile d;
  d.log_rows = 0;
  while (d.log_rows < 4 && d.log_rows < log_cells && (1 << d.log_rows) < s.U) ++d.log_rows;
  d.log_frames = log_cells - d.log_rows;
  if ((1 << d.log_frames) > kTileMaxFrames) d.log_frames = 4;
  d.frame_groups = (s.T + (1 << d.log_frames) - 1) >> d.log_frames;
  d.pitch = (int)(((row_bytes << d.log_rows) + 15) / 16) + 1;
  d.div_pitch = make_fastdiv((unsigned)d.pitch);
  return d;
}
inline int denom_tile_chunks(const PlanShape& s, const DenomTile& d) { return (s.U + (1 << d.log_rows) - 1) >> d.log_rows; }
inline long long denom_tile_blocks(const PlanShape& s, const DenomTile& d) {
  return (long long)denom_tile_chunks(s, d) * s.B * d.frame_groups;
}
// Consecutive tiles per XCD and turn: 64 (a tile's cells read the lattice diagonals of the neighbouring frames', which
// should find them in the same level-2 cache), fewer where the grid would not give every XCD four turns.
inline int tile_log_span(long long blocks) {
  int log_span = 6;
  while (log_span > 0 && (32LL << log_span) > blocks) --log_span;
  return log_span;
}
inline unsigned tile_grid(long long blocks) {
  const long long turn = 8LL << tile_log_span(blocks);
  return (unsigned)((blocks + turn - 1) / turn * turn);
}

#endif  // MI_PLAN_H_
