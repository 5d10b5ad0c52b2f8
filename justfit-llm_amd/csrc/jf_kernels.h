// Shared declarations of the gfx950 sampler: the device parameter records
// the host builds, the scratch records the kernels exchange, and the launch
// entry points of jf_kernels.hip.
#pragma once

#include <stdint.h>

#include "jf_host.h"

struct jf_sample_args;

namespace jf {

// Per-row target policy as the kernels read it (the reference's
// TargetSamplingParams + SamplingPenaltyParams fields of one lane,
// metal/abi/Sampling.h:40-61, 118-129), derived on the host.
struct RowParams {
  uint32_t flags;
  uint32_t top_k;             // effective: the vocabulary when disabled
  float inv_t;                // 1 / temperature
  float top_p;
  float minp_offset;          // temperature * log(min_p); without min-p, how far
                              // below the maximum the weights (with top-p
                              // alone, its boundary) reach (below zero)
  float repetition;
  float repetition_inverse;   // min(1 / repetition, FLT_MAX)
  float presence;
  float frequency;
  uint32_t penalty_row;
  uint32_t extra_count;
  uint32_t extra_offset;      // the row's extra tokens: SampleLaunch::extra + this
  uint32_t draft_index;       // its draft token: draft_tokens[draft_index]
                              // (kNoToken: not drafted)
  uint32_t cand_index;        // its draft distribution: sparse candidates
                              // cand_ids/probs + 16 * this, dense q row this
  uint32_t mask_row;          // its constraint mask: masks + this * mask_stride
  uint32_t fast_row;          // nonzero: a launch split between the two select
                              // kernels selects this row in the fast one
};
static_assert(sizeof(RowParams) == 64, "row params are 64 bytes");

enum RowFlags : uint32_t {
  kRowSampled = 1u,
  kRowConstrained = 2u,
  kRowExcludeStop = 4u,
  kRowPenalized = 8u,
  kRowMinP = 16u,
  kRowTopP = 32u,
  kRowTopK = 64u,
  // A drafted row with no cut, penalty, mask or extra tokens: its residual
  // pass runs in residual_kernel (set by the host).
  kRowLean = 128u,
};

// One block's summary of its chunk of a row.
struct BlockHeader {
  float maximum;       // sampled: largest admitted logit (-FLT_MAX if none)
  uint32_t count;      // sampled: candidates written (wide_row: lanes that
                       // admit a token)
  uint32_t admitted;   // sampled: 1 when the chunk admits a non-NaN token
  uint32_t overflow;   // sampled: candidates did not fit
  float best_value;    // greedy (wide_row: the chunk's least value)
  uint32_t best_id;    // greedy
  uint32_t floor_key;  // sampled: the row's K-th key is at least this
                       // (wide_row: `count` tokens of the chunk reach it)
  uint32_t reserved;
};
static_assert(sizeof(BlockHeader) == 32, "block headers are 32 bytes");

// A row of the cut passes (cut_hist_kernel and the launches after it).
struct RowState {
  uint32_t stage;     // RowStage
  float maximum;
  uint32_t thr_key;   // min-p floor key, 0 without min-p
  float scale;        // bins per unit below the maximum
  uint32_t b0, b1;    // the bins that hold the kept set's end (kCutBins: no cut)
  uint32_t bk;        // the bin of the top-k boundary (kCutBins: top-k cuts nothing)
  uint32_t need_k;    // tokens of bin bk that top-k keeps
  uint64_t mass_b0;   // mass of the bins before b0, before bk, of all
  uint64_t mass_bk;
  uint64_t total;
  uint32_t topp;      // top-p closes the kept set in [b0, b1]
  uint32_t bkey;      // the kept set's last token in (key desc, id asc) order
  uint32_t bid;
  uint32_t kept;      // its size, where kept outputs are asked for
  uint64_t mass3;     // its mass
  float end;          // the row's least value on the bins' scale
  uint32_t reserved[11];
};
static_assert(sizeof(RowState) == 128, "row states are 128 bytes");
enum RowStage : uint32_t {
  kRowDone = 0,
  kRowGather = 1,  // cut_list_kernel found and listed its boundary bins
  kRowEmit = 2,    // cut_draw_kernel found its kept set; outputs or a draft's draw remain
};

struct StagePartial {
  uint64_t v[256];
};

// Geometry of one selection launch.
constexpr int kThreads = 256;
constexpr int kWaves = 4;
constexpr int kBlockCandidates = 1024;
constexpr int kMergeCapacity = 2048;
constexpr uint32_t kMergeItems = 3072;  // tokens of a row the general merge holds
// A sampled row with no min-p floor whose top-k is off or past this takes the
// cut passes; up to it, the candidate lists and the merge. The select pass
// bounds a chunk's K-th token by its waves' ceil(K / 4)-th largest lane maxima
// (64 of them), so the lists grow faster than K: 64 rows x 151,936 fp32 ran
// 33.0 us at top-k 65, 38.4 at 96, 42.0 at 112, 70 at 128 (lists that overflow)
// through the lists, and 46.8-47.5 through the cut passes; in bf16 31.3, 37.2,
// 46.1, 70 against 43.5-44.1. Where the line lies for other batches, at top-k
// 96 through the lists and 97 through the cut passes: 1 row 25.6 and 24.6, 16
// rows 26.9 and 27.4, 256 rows 49.5 and 102.8 (fp32; bf16 26.3 and 24.3, 26.9
// and 26.8, 41.9 and 95.4), 1 row x 248,320 bf16 with top-p 61.1 and 26.9, 64
// rows of it 69.0 and 58.5.
constexpr uint32_t kListTopK = 96;
constexpr uint32_t kCutBins = 512;    // bins of a row's values below its maximum
constexpr uint32_t kCutItems = 6144;  // boundary tokens of a row resolved in LDS
constexpr int kMaxExtra = 16;
constexpr uint32_t kChunkF32 = 8192;
constexpr uint32_t kChunkBF16 = 8192;

// A sampled row of the cut passes by its policy alone (a min-p row past the
// lists joins them too).
__host__ __device__ constexpr bool wide_row(uint32_t flags, uint32_t top_k) {
  return (flags & kRowSampled) && !(flags & kRowMinP) && (flags & (kRowTopP | kRowTopK)) &&
         top_k > kListTopK;
}

constexpr uint32_t kNoGreedyRows = 0xffffffffu;  // SampleLaunch::uniform_row
struct SampleLaunch {
  const void *logits;
  uint64_t stride;
  const uint32_t *masks;
  uint64_t mask_stride;
  const RowParams *params;
  uint32_t vocabulary;
  uint32_t chunks;
  uint32_t rows;
  uint32_t stop0;
  uint32_t stop1;
  uint32_t finish_greedy; // no merge runs: uncut_kernel finishes the greedy
                          // rows
  uint32_t row_indexed;   // drafts are addressed through RowParams'
                          // draft_index/cand_index, not the row number
  uint32_t uniform_row;   // kNoGreedyRows, or, in a launch with greedy rows, a
                          // sampled one (0 without any). A greedy row has no
                          // uniform, and its place in the uniforms or their
                          // index may hold anything: a kernel then reads a
                          // row's uniform only once the row is known to be
                          // sampled
  const uint2 *pen_entries;
  const uint32_t *pen_offsets;
  uint32_t pen_max_entries;
  uint32_t pen_buckets;
  const uint32_t *extra;
  uint64_t extra_stride;
  const float *uniforms;
  const uint32_t *uniform_index;
  uint64_t uniform_offset;
  uint64_t uniform_stride;
  const uint32_t *draft_tokens;
  uint32_t drafted_rows;
  const uint32_t *cand_ids;
  const float *cand_probs;
  const float *dense_q;
  uint64_t q_stride;
  BlockHeader *headers;
  uint64_t *cands;       // key | id << 32
  uint32_t *counters;
  uint64_t *bests;       // all-greedy fast launches: each block's packed best
                         // (zero between calls unless a wait gave up)
  RowState *states;
  StagePartial *partials;
  uint32_t *out_tokens;
  float *out_draft;
  uint32_t *out_kept_counts;
  uint32_t *out_kept_ids;
  float *out_kept_probs;
  uint32_t kept_cap;
  uint32_t q_aligned;     // dense q rows start on 16-byte boundaries
  uint32_t epoch;         // the call's tag of its packed greedy bests (1..4095)
  uint32_t wait_bound;    // reads of a packed best before its wait gives up
  uint32_t *status;       // set to 1 when a wait gave up (host-mapped), or NULL
  // Drafted rows with no cut (kRowLean) in an all-fast fp32 launch: the
  // select pass also stores each token's weight there as pack_yk (row r at
  // r * lean_stride, chunk-major like the logits), and residual_kernel
  // reads it instead of the logits; NULL otherwise.
  uint32_t *lean_weights;
  uint64_t lean_stride;
};

// merge_small_kernel's chunk count with two facts its first loads depend on.
constexpr uint32_t kMergeRowIndexed = 0x80000000u;   // SampleLaunch::row_indexed
constexpr uint32_t kMergeLateUniform = 0x40000000u;  // the uniform waits for the row's record
inline uint32_t merge_chunks_bits(const SampleLaunch &a) {
  return a.chunks | (a.row_indexed ? kMergeRowIndexed : 0u) |
         (a.uniform_row != kNoGreedyRows ? kMergeLateUniform : 0u);
}

// The fast selection launch: the per-row facts every block needs before its
// first load (flags, penalty table row) travel in the kernel arguments, and
// each (table row, chunk) holds its penalty entries in a fixed run of
// `slot_count` 32-bit slots, so a block requests them together with its
// logits and waits on nothing first. Slot = offset in the chunk << 19 |
// prompt bit << 18 | count (< 2^18); an empty slot is 0 (every real entry
// has a count or the prompt bit). A uniform launch (every row the same
// policy, each reading its own penalty row, no row map, no extra tokens)
// carries no per-row facts (FastRows) at all: the kernel-argument segment
// the runtime copies for every launch then stays small.
constexpr int kKernargRows = 256;
struct FastLaunch {
  SampleLaunch a;
  const uint32_t *pen_slots;  // [table rows][chunks][slot_count]
  uint32_t slot_count;        // 256 or 512
  uint32_t row_base;          // sampler row of blockIdx.y == 0
  uint32_t fuse_greedy;       // every row greedy, no merge launch: 1, the
                              // row's last block to arrive finishes it; 2
                              // (set at launch when its rows are fewer than
                              // the blocks the GPU holds at once), the
                              // row's last chunk finishes it
  uint32_t mapped;            // blockIdx.y selects row row_of[blockIdx.y]
                              // (a launch split between the two kernels;
                              // the kernel takes it as a preloaded argument)
  uint32_t lean_bits[kKernargRows / 32];  // bit y: row blockIdx.y stores its
                                          // weights (a.lean_weights)
};
// The per-row facts of a launch that is not uniform, by blockIdx.y.
struct FastRows {
  uint32_t row_info[kKernargRows];  // RowFlags | penalty row << 8
  uint32_t row_of[kKernargRows];
  // Launches whose rows carry extra (verify) penalty tokens: the row's
  // extras are SampleLaunch::extra + (this & kExtraOffsetMask), this >> 27
  // of them (<= kMaxExtra).
  uint32_t row_extra[kKernargRows];
};
// The argument a uniform launch passes in FastRows' place.
struct NoRows {};
// The fast selection's last argument, naming what its finishing blocks do
// beyond selecting: nothing more, draw rows with no cut (UncutFinish), or
// (an AcceptTreeLaunch) run each lane's tree acceptance; StoreWeights is
// NoFinish that also stores the drafted rows' weights (a.lean_weights), a
// separate instantiation since the stores take registers.
struct NoFinish {};
struct UncutFinish {};
struct StoreWeights {};
constexpr uint32_t kExtraOffsetMask = (1u << 27) - 1u;

struct AcceptChainLane {
  uint32_t remaining;
  uint32_t sampled;
};

// Chain acceptance: up to kChainLanesPerLaunch lanes a launch, their
// records in the kernel arguments (no upload); the pointers start at the
// launch's first lane.
constexpr uint32_t kChainLanesPerLaunch = 256;
struct AcceptChainLaunch {
  uint32_t lanes;
  uint32_t verify_rows;
  const uint32_t *proposed;
  const uint32_t *candidates;
  const float *proposal_probs;
  const float *target_draft_probs;
  const float *uniforms;
  uint32_t *target_tokens;
  uint32_t *retained;
  uint32_t *accepted;
  uint32_t stop0;
  uint32_t stop1;
  AcceptChainLane lane_params[kChainLanesPerLaunch];
};

struct TreeLaneParams {
  uint32_t rows;
  uint32_t chain_rows;
  uint32_t remaining;
  uint32_t sampled;
  uint32_t parent[16];
  uint32_t token[16];
  float chain_q[8];
};

// Tree acceptance: up to kTreeLanesPerLaunch lanes a launch, their trees in
// the kernel arguments; the pointers start at the launch's first lane.
constexpr uint32_t kTreeLanesPerLaunch = 16;
struct AcceptTreeLaunch {
  uint32_t lanes;
  uint32_t rows_per_lane;
  const float *target_draft_probs;
  const float *uniforms;
  uint32_t *target_tokens;
  uint32_t *retained;
  uint32_t *accepted;
  uint32_t *path_rows;
  uint32_t stop0;
  uint32_t stop1;
  TreeLaneParams trees[kTreeLanesPerLaunch];
};

// The draft selector (jf_draft.hip): lane geometry of the reference's DFlash
// draft (ExecutionGeometry.h: 8 query rows, 7 proposal positions, 16
// candidates, selector rank 256) and the uniform slots of a lane
// (metal/abi/Sampling.h:19-29).
constexpr uint32_t kDraftQueryRows = 8;
constexpr uint32_t kDraftPositions = 7;
constexpr uint32_t kSamplingUniforms = 40;
constexpr uint32_t kUniformProposals = 1;
struct DraftLaneParams {
  uint32_t anchor;
  float temperature;
  uint32_t sampled;
  uint32_t reserved;
};
struct DraftLaunch {
  const float *logits;        // [lanes * 8][stride]
  uint64_t stride;
  uint32_t vocabulary;
  uint32_t chunks;            // 8192-token chunks per row
  uint32_t lanes;
  const uint16_t *hidden;     // bf16 [lanes * 8][256]
  const uint16_t *pred_codebook;  // bf16 [vocabulary][256]
  const uint16_t *succ_codebook;  // bf16 [vocabulary][256]
  const DraftLaneParams *lane_params;
  const float *uniforms;      // [lanes][40]
  uint32_t *candidates;       // [lanes * 7][16]
  float *unary;               // [lanes * 7][16]
  uint32_t *tokens;           // [lanes * 7]
  float *q_probs;             // [lanes * 7][16], sampled lanes
  uint64_t *part_comp;        // [lanes * 7][chunks][16]
  uint32_t *part_vbits;       // [lanes * 7][chunks][16]
  float *tables;              // [lanes][7][16][16]
  uint32_t *choices;          // [lanes * 7][16]: the walk's pick after each predecessor
  float *choice_q;            // [lanes * 7][16][16]: its probabilities, sampled lanes
  uint32_t *counters;         // [lanes * 8], zero between launches
};

// The tree gather (jf_gather.hip): JustFitTreeGatherParams (TreeVerify.h:54-69)
// in 16-bit units, plus the rows per lane of the tensor.
constexpr uint32_t kGatherDepth = 8;  // path entries per lane
struct GatherLaunch {
  uint16_t *data;
  const uint32_t *path_rows;  // [lanes][8]
  const uint32_t *retained;   // [lanes]
  uint32_t columns, inner, inner_stride, outer_stride;
  uint64_t row_stride, lane_stride, layer_stride;
  uint32_t layers, lanes, rows;
};

// The device scratch of one selection: where its kernels exchange row
// parameters, chunk summaries, candidate lists, arrival counters and packed
// greedy bests (both zero between calls), row states and stage partials. Room for max_rows rows of
// at most max_chunks 8192-token chunks.
struct SampleScratch {
  RowParams *params;        // [max_rows]
  BlockHeader *headers;     // [max_rows * max_chunks]
  uint64_t *cands;          // [max_rows * max_chunks * kBlockCandidates]
  uint32_t *counters;       // [max_rows]
  uint64_t *bests;          // [max_rows * max_chunks], zero between calls
  RowState *states;         // [max_rows]
  StagePartial *partials;   // [max_rows * max_chunks]
  uint32_t max_rows;
  uint32_t max_chunks;
  uint32_t *status;         // device address of a host-mapped word, or NULL
  uint32_t epoch;           // this call's tag (1..4095)
  uint32_t wait_bound;      // reads of a packed best before its wait gives up
  // Room for `rows` drafted rows' stored weights (rows x max_chunks x 8192
  // words), from the owner (called with the upload context), or NULL when
  // the owner keeps none: the residual pass then reads the logits.
  uint32_t *(*lean_weights)(void *ctx, uint32_t rows);
};

// How a selection's host-built row parameters reach scratch.params before
// its kernels run (stream-ordered on `stream`); returns a JF_* status.
typedef int (*ParamUpload)(void *ctx, const RowParams *params, uint32_t rows,
                           RowParams *device, void *stream);

// The body of jf_sample over a given scratch (jf_sampler.cpp): validates the
// call, builds each row's parameters into `params` (host, args->rows
// entries), hands them to `upload`, then enqueues the kernels on `stream`.
// accept: the lanes' tree acceptance to run in the selection's launch if it
// can (*accepted tells whether it did), or NULL.
int sample_core(uint32_t vocabulary, const SampleScratch &scratch,
                const jf_sample_args *args, RowParams *params, ParamUpload upload,
                void *upload_ctx, void *stream, const AcceptTreeLaunch *accept = nullptr,
                bool *accepted = nullptr);

// Launchers (jf_kernels.hip); they return the hipError_t of the launch.
// With both events set, they record the selection kernel's own start and end.
int launch_select(const SampleLaunch &a, uint32_t dtype, void *stream,
                  void *start_event = nullptr, void *stop_event = nullptr);
// `uniform`: when every row of the launch has this policy and penalty table
// row == its own row, or NULL. `fr`: the launch's per-row facts, or NULL for
// a uniform launch with no row map and no extra tokens.
// extras: some row of the launch has extra penalty tokens (fr->row_extra).
// fuse_uncut: every row is sampled with no cut, draft, penalty or extra
// token and no kept outputs are asked for: each row's last chunk block draws
// it (no uncut_kernel launch). accept: the lanes' tree acceptance over this
// launch's rows (greedy lanes, rows = lanes x rows_per_lane), run by the
// row finishers when the launch is uniform, all greedy and finished by
// each row's last chunk; *accepted tells whether it was (else the caller
// launches it).
int launch_select_fast(const FastLaunch &f, const FastRows *fr, uint32_t rows, uint32_t dtype,
                       const RowParams *uniform, bool extras, bool fuse_uncut,
                       const AcceptTreeLaunch *accept, bool *accepted, void *stream,
                       void *start_event = nullptr, void *stop_event = nullptr);
int launch_merge(const SampleLaunch &a, uint32_t dtype, void *stream);
// wide: some cut row of the launch has no min-p floor (longer candidate
// lists); the merge then fetches more list slots a chunk where that helps.
// hold: some min-p row may keep more than 64 tokens.
int launch_merge_small(const SampleLaunch &a, uint32_t dtype, bool wide, bool hold, void *stream);
// Rows with no cut (grid rows x per_row: per_row = chunks when the launch
// has drafted uncut rows, else 1).
int launch_uncut(const SampleLaunch &a, uint32_t dtype, uint32_t per_row, void *stream);
// residual_kernel over the kRowLean rows row_of[0, n_lean) (grid n_lean x
// chunks), before launch_uncut on the same stream; or, with draw set, a
// launch that also draws: each lean row's last chunk block draws that row
// and a share of the rows row_of[n_lean, n_lean + n_plain) (every other row
// of the launch: greedy ones, and sampled ones with no cut, draft, penalty
// or extra token), so no launch_uncut follows (n_lean >= 1, n_lean +
// n_plain <= kKernargRows). Bit 31 of row_of marks a greedy row.
constexpr uint32_t kLeanGreedy = 0x80000000u;
struct LeanLaunch {
  SampleLaunch a;
  uint32_t n_lean;
  uint32_t n_plain;
  uint32_t draw;
  uint32_t row_of[kKernargRows];
};
int launch_residual(const LeanLaunch &l, uint32_t dtype, void *stream);
// The cut passes over the rows that take them: cut_hist_kernel, cut_list_kernel,
// cut_draw_kernel and, for kept outputs or drafted rows, cut_emit_kernel.
struct CutLaunch {
  bool all;      // every row takes them by its policy (wide_row)
  bool plain;    // no row is penalized
  bool drafted;  // some row is drafted
  bool others;   // cut_draw_kernel finishes the listed and greedy rows too (no
                 // merge is launched),
  bool uncut;    // and the uncut rows (no launch_uncut follows)
  bool small;    // its listed rows may take merge_small_row
};
int launch_cut(const SampleLaunch &a, uint32_t dtype, const CutLaunch &c, void *stream);
// Its kernels of one block a (row, chunk) have their chunks in the grid's x and
// their rows in its y, which takes at most 65,535; a sampler has up to
// 4,194,304 rows. So they run a slice of kCutSliceRows rows at a time.
constexpr uint32_t kCutSliceRows = 32768;
inline uint32_t cut_slices(uint32_t rows) { return (rows + kCutSliceRows - 1) / kCutSliceRows; }
inline uint32_t cut_slice_rows(uint32_t rows, uint32_t slice) {
  const uint32_t left = rows - slice * kCutSliceRows;
  return left < kCutSliceRows ? left : kCutSliceRows;
}
int launch_accept_chain(const AcceptChainLaunch &a, void *stream);
int launch_accept_tree(const AcceptTreeLaunch &a, void *stream);
// jf_draft.hip; the events, when set, bracket the top-16 kernel.
int launch_draft_select(const DraftLaunch &d, void *stream,
                        void *start_event = nullptr, void *stop_event = nullptr);
// jf_gather.hip; vec8: 8 columns per thread with 16-byte accesses.
int launch_tree_gather(const GatherLaunch &g, bool vec8, void *stream,
                       void *start_event = nullptr, void *stop_event = nullptr);

// The device penalty table as penalty_count_kernel updates it.
struct PenaltyTableView {
  PenaltyEntry *entries;  // [rows][max_entries]
  uint32_t *offsets;      // [rows][buckets + 1]
  uint32_t *slots;        // [rows][chunks][slot_count]
  uint32_t max_entries;
  uint32_t buckets;
  uint32_t chunks;
  uint32_t slot_count;
};

// Up to kPenaltyOps counted tokens (PenaltyOp, packed), in call order within
// each row; block g applies ops [group_start[g], group_start[g + 1]) to
// table row group_row[g].
constexpr uint32_t kPenaltyOps = 64;
struct PackedPenaltyOp {
  uint32_t token;
  uint32_t word;
  uint32_t index;       // entry index | insert << 31
  uint32_t entries;     // the row's entry count before the op
  uint32_t slot_value;
  uint32_t slot;        // slot index | the chunk's used slots << 16; 0xffff: no slot
};
struct PenaltyOpBatch {
  PackedPenaltyOp op[kPenaltyOps];
  uint32_t group_row[kPenaltyOps];
  uint32_t group_start[kPenaltyOps + 1];
};
static_assert(sizeof(PenaltyOpBatch) <= 2560, "penalty updates travel as kernel arguments");

int launch_penalty_count(const PenaltyTableView &t, const PenaltyOpBatch &b, uint32_t groups,
                         void *stream);
// The same updates read from host-mapped memory (calls of more than
// kPenaltyOps tokens, all in one launch): ops[n], group_row[groups],
// group_start[groups + 1].
int launch_penalty_count_mapped(const PenaltyTableView &t, const PackedPenaltyOp *ops,
                                const uint32_t *group_row, const uint32_t *group_start,
                                uint32_t groups, void *stream);

}  // namespace jf
