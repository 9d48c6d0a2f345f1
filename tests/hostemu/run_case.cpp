// Host build of the lps C ABI (llm-pipeline_amd/csrc/lps.hip, unchanged) over
// the HIP emulation in shim/hip/hip_runtime.h, under AddressSanitizer and
// UndefinedBehaviorSanitizer (array bounds included): test infrastructure for
// tests/test_hostemu.py.
//
//   run_case IN OUT
//
// IN holds one call's inputs, OUT receives its outputs (layouts below,
// little-endian); the first word says which entry point: lps_sample,
// lps_lm_head, lps_softmax, lps_spec_verify or the host's planning rules.  The workspace is calloc'd at its exact size, so an
// access past it, past any input or output array, or past an LDS array of a
// kernel, stops the run with the sanitizer's report.
#include "../../llm-pipeline_amd/csrc/lps.hip"

#include <sanitizer/asan_interface.h>

#include <vector>

namespace {

// IN: int32 header[16] = {magic 0x4C505345, dtype, R, V, H, n_top, flags,
//     use_workspace, logprobs, entropy, skip_draw, 0...}, then
//     logits [R * V] (dtype), temperature f32[R], top_k i32[R], top_p f32[R],
//     min_p f32[R], typical_p f32[R], rep f32[R], pres f32[R], freq f32[R],
//     history i32[R * H], history_len i32[R] (both when H > 0), uniforms f32[R].
// OUT: tokens i64[R], status i32[R], kept_cut f32[R], kept_ties i32[R],
//     kept_count i32[R], row_path i32[R], chosen_logprob f32[R] (logprobs),
//     top_logprobs f32[R * n_top], top_ids i64[R * n_top], entropy f32[R] (when
//     asked), then the workspace's
//     row status words i32[R] (LPS_ROW_DEFERRED | reason << 8 for rows the
//     fast kernels deferred; zeros without a workspace).
template <typename T>
std::vector<T> rd(FILE* f, size_t n) {
  std::vector<T> v(n);
  if (n && fread(v.data(), sizeof(T), n, f) != n) {
    fprintf(stderr, "run_case: short input\n");
    exit(2);
  }
  return v;
}
template <typename T>
void wr(FILE* f, const std::vector<T>& v) {
  if (!v.empty()) fwrite(v.data(), sizeof(T), v.size(), f);
}

// A heap copy of exactly the array's size.
template <typename T>
T* exact(const std::vector<T>& v) {
  T* p = static_cast<T*>(malloc(v.size() * sizeof(T)));
  if (!v.empty()) memcpy(p, v.data(), v.size() * sizeof(T));
  return p;
}
size_t elem(int dtype) { return dtype == LPS_DTYPE_F32 ? 4 : 2; }
int fail(const char* entry, int rc) {
  fprintf(stderr, "run_case: %s returned %d\n", entry, rc);
  return 3;
}

// IN: header {0x4C4D4844, dtype, out_dtype, M, V, H}, x [M * H], w [V * H].
// OUT: out [M * V] (out_dtype), stats f32[M * ceil(V / 128) * 2].
int run_lm_head(const std::vector<int32_t>& h, FILE* f, const char* path) {
  const int M = h[3], V = h[4], H = h[5];
  uint8_t* x = exact(rd<uint8_t>(f, (size_t)M * H * 2));
  uint8_t* w = exact(rd<uint8_t>(f, (size_t)V * H * 2));
  const std::vector<uint8_t> out0((size_t)M * V * elem(h[2]), 0x5A);
  const std::vector<float> stats0((size_t)M * ((V + 127) / 128) * 2, -7.0f);
  uint8_t* out = exact(out0);
  float* stats = exact(stats0);
  lps_lm_head_args a{};
  a.x = x;
  a.w = w;
  a.out = out;
  a.stats = stats;
  a.dtype = h[1];
  a.out_dtype = h[2];
  a.rows = M;
  a.vocab = V;
  a.hidden = H;
  a.x_stride = a.w_stride = H;
  a.out_stride = V;
  const int rc = lps_lm_head(&a, nullptr);
  if (rc != LPS_OK) return fail("lps_lm_head", rc);
  FILE* o = fopen(path, "wb");
  if (!o) return 2;
  fwrite(out, 1, out0.size(), o);
  fwrite(stats, sizeof(float), stats0.size(), o);
  fclose(o);
  free(x);
  free(w);
  free(out);
  free(stats);
  return 0;
}

// IN: header {0x534D4158, dtype, rows, cols, off, stride, causal, row_offset,
// stats_cols}, x [off + (rows - 1) * stride + cols], stats f32[rows * G * 2] (stats_cols > 0,
// G = ceil(cols / stats_cols)).  Row 0 starts at element off of x and of out;
// the bytes of its 16-byte line that lie 8 or more before it are poisoned.
// OUT: out (x's elements, 0x5A where nothing was written), lse f32[rows].
int run_softmax(const std::vector<int32_t>& h, FILE* f, const char* path) {
  const int dtype = h[1], rows = h[2], cols = h[3], off = h[4], stride = h[5], sc = h[8];
  const size_t es = elem(dtype), n = off + (size_t)(rows - 1) * stride + cols;
  const size_t G = sc > 0 ? (cols + sc - 1) / sc : 0;
  uint8_t* x = exact(rd<uint8_t>(f, n * es));
  float* stats = exact(rd<float>(f, rows * G * 2));
  const std::vector<uint8_t> out0(n * es, 0x5A);
  uint8_t* out = exact(out0);
  const std::vector<float> lse0(rows, -7.0f);
  float* lse = exact(lse0);
  const size_t lead = (size_t)off * es / 8 * 8;
  __asan_poison_memory_region(x, lead);
  __asan_poison_memory_region(out, lead);
  lps_softmax_args a{};
  a.x = x + (size_t)off * es;
  a.out = out + (size_t)off * es;
  a.dtype = dtype;
  a.rows = rows;
  a.cols = cols;
  a.x_stride = a.out_stride = stride;
  a.causal = h[6];
  a.seq_len = rows;
  a.row_offset = h[7];
  a.row_lse = lse;
  a.workspace_bytes = lps_softmax_workspace_bytes(rows, cols, dtype);
  void* ws = a.workspace_bytes ? calloc(1, a.workspace_bytes) : nullptr;
  a.workspace = ws;
  if (sc > 0) {
    a.row_stats = stats;
    a.stats_stride = (int64_t)G * 2;
    a.stats_cols = sc;
  }
  const int rc = lps_softmax(&a, nullptr);
  if (rc != LPS_OK) return fail("lps_softmax", rc);
  __asan_unpoison_memory_region(x, lead);
  __asan_unpoison_memory_region(out, lead);
  FILE* o = fopen(path, "wb");
  if (!o) return 2;
  fwrite(out, 1, n * es, o);
  fwrite(lse, sizeof(float), rows, o);
  fclose(o);
  free(x);
  free(stats);
  free(out);
  free(lse);
  free(ws);
  return 0;
}

// IN: header {0x53504543, dtype, B, k, V, residual}, f32 {temperature, top_p},
// target [B * (k + 1) * V], draft [B * k * V], draft tokens i64[B * k],
// u_accept f32[B * k], u_resample f32[B * (k + 1)].
// OUT: n_accepted i32[B], tokens i64[B * (k + 1)], status i32[B * (2 k + 1)].
int run_spec(const std::vector<int32_t>& h, FILE* f, const char* path) {
  const int dtype = h[1], B = h[2], k = h[3], V = h[4];
  const size_t es = elem(dtype), Rt = (size_t)B * (k + 1), Rd = (size_t)B * k;
  const auto tp = rd<float>(f, 2);
  uint8_t* t = exact(rd<uint8_t>(f, Rt * V * es));
  uint8_t* d = exact(rd<uint8_t>(f, Rd * V * es));
  const auto tok = rd<int64_t>(f, Rd);
  const auto ua = rd<float>(f, Rd), ur = rd<float>(f, Rt);
  std::vector<int32_t> n_acc(B, -7), status(Rt + Rd, -7);
  std::vector<int64_t> tokens(Rt, -7);
  lps_spec_args a{};
  a.target_logits = t;
  a.target_stride_b = (int64_t)(k + 1) * V;
  a.target_stride_k = V;
  a.draft_logits = d;
  a.draft_stride_b = (int64_t)k * V;
  a.draft_stride_k = V;
  a.dtype = dtype;
  a.batch = B;
  a.k = k;
  a.vocab = V;
  a.temperature = tp[0];
  a.top_p = tp[1];
  a.residual = h[5];
  a.draft_tokens = tok.data();
  a.u_accept = ua.data();
  a.u_resample = ur.data();
  a.n_accepted = n_acc.data();
  a.tokens = tokens.data();
  a.row_status = status.data();
  a.workspace_bytes = lps_spec_workspace_bytes(B, k, V);
  void* ws = calloc(1, a.workspace_bytes);
  a.workspace = ws;
  const int rc = lps_spec_verify(&a, nullptr);
  if (rc != LPS_OK) return fail("lps_spec_verify", rc);
  FILE* o = fopen(path, "wb");
  if (!o) return 2;
  wr(o, n_acc);
  wr(o, tokens);
  wr(o, status);
  fclose(o);
  free(t);
  free(d);
  free(ws);
  return 0;
}

// IN: header {0x504C414E, n}, n queries i32[4]: {0, dtype, R, V} (a row-group
// plan for misaligned rows), {1, M, V, 0} (an LM-head tile shape).
// OUT: i32[4] each: {logits per thread, chunks, the workspace's chunks, planned},
// {rows, columns of a tile, shape, 0}.
int run_plan(const std::vector<int32_t>& h, FILE* f, const char* path) {
  std::vector<int32_t> out;
  for (int i = 0; i < h[1]; i++) {
    const auto q = rd<int32_t>(f, 4);
    if (q[0] == 0) {
      const RgPlan p = rg_plan(q[1], false, q[2], q[3]);
      out.insert(out.end(), {p.ne, p.G, rg_max_chunks(q[2], q[3]), p.ok ? 1 : 0});
    } else {
      const int s = lmhead_shape(q[1], q[2], device_cus());
      out.insert(out.end(), {LMH_SHAPES[s][0], LMH_SHAPES[s][1], s, 0});
    }
  }
  FILE* o = fopen(path, "wb");
  if (!o) return 2;
  wr(o, out);
  fclose(o);
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc != 3) {
    fprintf(stderr, "usage: run_case IN OUT\n");
    return 2;
  }
  FILE* f = fopen(argv[1], "rb");
  if (!f) return 2;
  const std::vector<int32_t> h = rd<int32_t>(f, 16);
  if (h[0] == 0x4C4D4844) return run_lm_head(h, f, argv[2]);
  if (h[0] == 0x534D4158) return run_softmax(h, f, argv[2]);
  if (h[0] == 0x53504543) return run_spec(h, f, argv[2]);
  if (h[0] == 0x504C414E) return run_plan(h, f, argv[2]);
  if (h[0] != 0x4C505345) return 2;
  const int dtype = h[1], R = h[2], V = h[3], H = h[4], n_top = h[5], flags = h[6], use_ws = h[7], lp = h[8];
  const int want_h = h[9], skip_draw = h[10];
  const size_t es = dtype == LPS_DTYPE_F32 ? 4 : 2;
  // the logits exactly sized (an access past the last row is caught)
  std::vector<uint8_t> logits_v = rd<uint8_t>(f, (size_t)R * V * es);
  void* logits = malloc(logits_v.size());
  memcpy(logits, logits_v.data(), logits_v.size());
  auto T = rd<float>(f, R);
  auto K = rd<int32_t>(f, R);
  auto P = rd<float>(f, R), MP = rd<float>(f, R), TP = rd<float>(f, R);
  auto REP = rd<float>(f, R), PRES = rd<float>(f, R), FREQ = rd<float>(f, R);
  std::vector<int32_t> hist, hlen;
  if (H > 0) {
    hist = rd<int32_t>(f, (size_t)R * H);
    hlen = rd<int32_t>(f, R);
  }
  auto U = rd<float>(f, R);
  fclose(f);

  std::vector<int64_t> tokens(R, -7);
  std::vector<int32_t> status(R, -7), ties(R, -7), count(R, -7), path(R, -7);
  std::vector<float> cut(R, -7.0f), clp(lp ? R : 0, -7.0f), tlp((size_t)R * n_top, -7.0f);
  std::vector<int64_t> tids((size_t)R * n_top, -7);
  std::vector<float> ent(want_h ? R : 0, -7.0f);

  lps_sample_args a{};
  a.logits = logits;
  a.dtype = dtype;
  a.num_rows = R;
  a.vocab = V;
  a.rows_inner = 1;
  a.stride_outer = V;
  a.stride_inner = 0;
  a.temperature = T.data();
  a.top_k = K.data();
  a.top_p = P.data();
  a.min_p = MP.data();
  a.typical_p = TP.data();
  a.repetition_penalty = REP.data();
  a.presence_penalty = PRES.data();
  a.frequency_penalty = FREQ.data();
  if (H > 0) {
    a.history = hist.data();
    a.history_stride = H;
    a.history_len = hlen.data();
  }
  a.uniforms = U.data();
  a.tokens = tokens.data();
  a.chosen_logprob = lp ? clp.data() : nullptr;
  a.top_logprobs = n_top ? tlp.data() : nullptr;
  a.top_ids = n_top ? tids.data() : nullptr;
  a.n_top = n_top;
  a.row_status = status.data();
  a.kept_cut = cut.data();
  a.kept_ties = ties.data();
  a.kept_count = count.data();
  a.row_path = path.data();
  a.entropy = want_h ? ent.data() : nullptr;
  a.skip_draw = skip_draw;
  a.flags = flags;
  void* ws = nullptr;
  if (use_ws) {
    a.workspace_bytes = lps_workspace_bytes(R, V, flags);
    ws = a.workspace_bytes ? calloc(1, a.workspace_bytes) : nullptr;
    a.workspace = ws;
  }
  const int rc = lps_sample(&a, nullptr);
  if (rc != LPS_OK) {
    fprintf(stderr, "run_case: lps_sample returned %d\n", rc);
    return 3;
  }
  FILE* o = fopen(argv[2], "wb");
  if (!o) return 2;
  wr(o, tokens);
  wr(o, status);
  wr(o, cut);
  wr(o, ties);
  wr(o, count);
  wr(o, path);
  wr(o, clp);
  wr(o, tlp);
  wr(o, tids);
  wr(o, ent);
  std::vector<int32_t> wst(R, 0);
  if (ws) memcpy(wst.data(), static_cast<char*>(ws) + rg_counter_bytes(), (size_t)R * 4);
  wr(o, wst);
  fclose(o);
  free(ws);
  free(logits);
  return 0;
}
