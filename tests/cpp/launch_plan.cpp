// The launches jf::sample_core enqueues for a batch, without a GPU: the
// library's own host code over launchers that only record what they were
// given. Prints one JSON object per batch for tests/test_launch_plan.py.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "jf_kernels.h"
#include "jf_sampler.h"

namespace {
std::string g_out;

void add(const char *name, const jf::SampleLaunch &a, const std::string &more = "") {
  if (!g_out.empty()) g_out += ", ";
  g_out += "{\"launch\": \"" + std::string(name) + "\", \"uniform_row\": " +
           std::to_string(a.uniform_row) + more + "}";
}
}  // namespace

namespace jf {
int launch_select(const SampleLaunch &a, uint32_t, void *, void *, void *) {
  add("select", a);
  return 0;
}
int launch_select_fast(const FastLaunch &f, const FastRows *, uint32_t, uint32_t, const RowParams *,
                       bool, bool, const AcceptTreeLaunch *, bool *, void *, void *, void *) {
  add("select_fast", f.a);
  return 0;
}
int launch_merge(const SampleLaunch &a, uint32_t, void *) {
  add("merge", a);
  return 0;
}
int launch_merge_small(const SampleLaunch &a, uint32_t, bool, bool, void *) {
  const uint32_t bits = merge_chunks_bits(a);
  add("merge_small", a,
      ", \"late_uniform\": " + std::to_string((bits & kMergeLateUniform) != 0) +
          ", \"chunks\": " + std::to_string(bits & ~(kMergeRowIndexed | kMergeLateUniform)));
  return 0;
}
int launch_uncut(const SampleLaunch &a, uint32_t, uint32_t, void *) {
  add("uncut", a);
  return 0;
}
int launch_residual(const LeanLaunch &l, uint32_t, void *) {
  std::string rows;
  for (uint32_t i = 0; i < l.n_lean + l.n_plain; ++i)
    rows += (i ? ", " : "") + std::to_string(l.row_of[i]);
  add("residual", l.a, ", \"row_of\": [" + rows + "]");
  return 0;
}
int launch_cut(const SampleLaunch &a, uint32_t, const CutLaunch &, void *) {
  std::string slices;
  for (uint32_t i = 0; i < cut_slices(a.rows); ++i)
    slices += (i ? ", " : "") + std::to_string(cut_slice_rows(a.rows, i));
  add("cut", a, ", \"slices\": [" + slices + "]");
  return 0;
}
int launch_accept_chain(const AcceptChainLaunch &, void *) { return 0; }
int launch_accept_tree(const AcceptTreeLaunch &, void *) { return 0; }
int launch_draft_select(const DraftLaunch &, void *, void *, void *) { return 0; }
int launch_tree_gather(const GatherLaunch &, bool, void *, void *, void *) { return 0; }
int launch_penalty_count(const PenaltyTableView &, const PenaltyOpBatch &, uint32_t, void *) {
  return 0;
}
int launch_penalty_count_mapped(const PenaltyTableView &, const PackedPenaltyOp *, const uint32_t *,
                                const uint32_t *, uint32_t, void *) {
  return 0;
}
}  // namespace jf

namespace {
int upload(void *, const jf::RowParams *, uint32_t, jf::RowParams *, void *) { return JF_OK; }

// One letter a row: g greedy, k top-k 50, n top-p alone, u no cut, d no cut
// and drafted (a dense q). "n:70000": that many rows of the letters, repeated.
void batch(const char *spec) {
  const char *colon = std::strchr(spec, ':');
  const std::string letters(spec, colon ? colon - spec : std::strlen(spec));
  std::string kinds = letters;
  if (colon)
    for (kinds.clear(); kinds.size() < std::strtoul(colon + 1, nullptr, 10);) kinds += letters;
  const uint32_t rows = (uint32_t)kinds.size(), V = 20000;
  static uint64_t memory[64];  // stands for every device buffer; nothing reads it
  std::vector<jf_policy> pol(rows);
  std::vector<uint32_t> draft(rows, JF_NO_TOKEN);
  bool drafted = false;
  for (uint32_t r = 0; r < rows; ++r) {
    jf_policy &p = pol[r];
    p = jf_policy{};
    p.top_p = 1.0f;
    p.repetition = 1.0f;
    p.temperature = kinds[r] == 'g' ? 0.0f : 1.0f;
    if (kinds[r] == 'k') p.top_k = 50;
    if (kinds[r] == 'n') p.top_p = 0.9f;
    if (kinds[r] == 'd') draft[r] = r, drafted = true;
  }
  jf_sample_args a{};
  a.rows = rows;
  a.dtype = JF_DTYPE_F32;
  a.logits = memory;
  a.logits_stride = V;
  a.policies = pol.data();
  a.stop_token_0 = a.stop_token_1 = JF_NO_TOKEN;
  a.uniforms = (const float *)memory;
  a.uniform_index = (const uint32_t *)memory;
  a.out_tokens = (uint32_t *)memory;
  if (drafted) {
    a.draft_tokens = (const uint32_t *)memory;
    a.draft_token_index = draft.data();
    a.draft_q = (const float *)memory;
    a.draft_q_stride = V;
  }
  jf::SampleScratch sc{};
  sc.params = (jf::RowParams *)memory;
  sc.max_rows = rows;
  sc.max_chunks = 3;
  sc.epoch = 1;
  sc.wait_bound = 1;
  std::vector<jf::RowParams> params(rows);
  g_out.clear();
  const int rc = jf::sample_core(V, sc, &a, params.data(), upload, nullptr, nullptr);
  std::printf("{\"batch\": \"%s\", \"rc\": %d, \"launches\": [%s]}\n", spec, rc, g_out.c_str());
}
}  // namespace

int main(int argc, char **argv) {
  for (int i = 1; i < argc; ++i) batch(argv[i]);
  return 0;
}
