// Speculative-decoding kernels: the batched accept test of
// verify_drafts_batched (src/llm_pipeline/inference/speculative_kernel.py:24-87)
// and the per-request epilogue of the accept / reject / resample block
// (src/llm_pipeline/inference/speculative.py:119-174).
#pragma once

#include "lps_generic.h"
#include "lps_wave.h"

namespace lps {

// torch.clamp semantics: NaN propagates (fminf / fmaxf would drop it).
__device__ __forceinline__ float spec_ratio(float p, float q) {
  const float qc = q < 1e-9f ? 1e-9f : q;
  const float r = __fdiv_rn(p, qc);
  return r > 1.0f ? 1.0f : r;
}

// accept[i] = u[i] < min(p[i, tok[i]] / max(q[i], 1e-9), 1)   (speculative_kernel.py:61-87)
template <int DT>
__global__ __launch_bounds__(256) void verify_drafts_kernel(const void* tp, int64_t K, int64_t V, int64_t sk,
                                                            int64_t sv, const float* q, const int64_t* tok,
                                                            const float* u, int8_t* out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= K) return;
  const int64_t t = tok[i];
  const float p = (t >= 0 && t < V) ? load1<DT>(tp, i * sk + t * sv) : 0.0f;
  out[i] = (int8_t)(u[i] < spec_ratio(p, q[i]) ? 1 : 0);
}

// First rejected position of request b (k: every draft accepted); greedy (T <=
// 0) accepts iff the target one-hot is 1 at the draft token
// (speculative.py:130-132).
__device__ __forceinline__ bool spec_accepts(int b, int i, int k, float T, const float* p_t, const float* q_d,
                                             const float* u_acc) {
  const float p = p_t[(int64_t)b * (k + 1) + i];
  if (!(T > 0.0f)) return p == 1.0f;
  return u_acc[(int64_t)b * k + i] < spec_ratio(p, q_d[(int64_t)b * k + i]);
}
__device__ __forceinline__ int spec_first_reject(int b, int k, float T, const float* p_t, const float* q_d,
                                                 const float* u_acc) {
  int j = k;
  for (int i = k - 1; i >= 0; i--) j = spec_accepts(b, i, k, T, p_t, q_d, u_acc) ? j : i;
  return j;
}
struct SpecOut {
  int32_t* n_acc;
  int64_t* tokens;
  int8_t* accept;
  float* p_out;
  float* q_out;
};
// Request b's outputs (one thread): accept bits for every position (as
// verify_drafts_batched computes them), the accepted drafts, then the
// replacement (target draw at the first rejection) or the bonus (target draw
// at k).
__device__ __forceinline__ void spec_epilogue_request(int b, int k, float T, const float* p_t, const float* q_d,
                                                      const int64_t* draws_t, const int64_t* draft_tokens,
                                                      const float* u_acc, const SpecOut& o) {
  int j = k;
  for (int i = 0; i < k; i++) {
    const bool acc = spec_accepts(b, i, k, T, p_t, q_d, u_acc);
    if (o.accept) o.accept[(int64_t)b * k + i] = acc ? 1 : 0;
    if (o.p_out) o.p_out[(int64_t)b * k + i] = p_t[(int64_t)b * (k + 1) + i];
    if (o.q_out) o.q_out[(int64_t)b * k + i] = q_d[(int64_t)b * k + i];
    if (!acc && j == k) j = i;
  }
  o.n_acc[b] = j;
  for (int i = 0; i <= k; i++) {
    int64_t t = -1;
    if (i < j) t = draft_tokens[(int64_t)b * k + i];
    else if (i == j) t = draws_t[(int64_t)b * (k + 1) + i];
    o.tokens[(int64_t)b * (k + 1) + i] = t;
  }
}
__global__ __launch_bounds__(256) void spec_epilogue_kernel(int B, int k, float T, const float* p_t, const float* q_d,
                                                            const int64_t* draws_t, const int64_t* draft_tokens,
                                                            const float* u_acc, SpecOut o) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b < B) spec_epilogue_request(b, k, T, p_t, q_d, draws_t, draft_tokens, u_acc, o);
}

// ---------------------------------------------------------------------------
// Leviathan residual: each request whose first rejection j < k draws from
// norm(max(p_j - q_j, 0)), p and q the kept distributions of target row j and
// draft row j, in vocabulary order with the position's resample uniform.  A
// zero residual keeps the target draw the epilogue wrote, and so does a row
// that could not be sampled.
//
// The row kernels leave each row's kept set as its cut (the least kept scaled
// logit) and the kept ties there; two launches do the rest, RES_CH ids of one
// request a workgroup (a Qwen3 row: 38 chunks):
//   residual_stats_kernel  per chunk and row: the largest scaled logit, the
//                          mass above the cut against it, the ties at the cut;
//                          chunk 0 also writes the request's outputs
//   residual_draw_kernel   combines the chunks (the row's maximum, its kept
//                          mass, the ties before this chunk), sums the chunk's
//                          residual; the request's last chunk to finish finds
//                          the chunk holding u times the total and draws there
// Bound by launches and two dependent passes over 2 rows a request (the second
// from the caches).  Before, the row kernels were the general one (its
// per-row plan held the maximum and mass) and one workgroup per request walked
// both rows twice: 8 requests x 3 drafts of 151936 bf16, 2 x 240 + 284 us.
// ---------------------------------------------------------------------------
constexpr int RES_NT = 256;
constexpr int RES_PT = 16;                // ids per thread
constexpr int RES_CH = RES_NT * RES_PT;   // ids per chunk
__host__ __device__ inline int res_chunks(int V) { return (V + RES_CH - 1) / RES_CH; }

struct ResRec {    // one chunk of one row
  float m;         // its largest scaled logit
  uint32_t ties;   // ids at the cut
  double s;        // sum of mass_f(z, m) over the ids above the cut
};
struct ResParams {
  const void* tl;  // target logits [B, k + 1, V], draft logits [B, k, V]
  int64_t tsb, tsk;
  const void* dl;
  int64_t dsb, dsk;
  int B, k, V;
  float T;
  const float* p_t;         // [B (k + 1)], then [B k]
  const float* q_d;
  const int64_t* draws_t;
  const int64_t* draft_tokens;
  const float* u_acc;
  const float* u_res;
  const float* cut;         // kept sets of the target rows, then the draft rows
  const int32_t* ties;
  const int32_t* status;
  ResRec* rec;              // [B, chunks, 2]
  uint64_t* rsum;           // [B, chunks]: residual mass per chunk (a double's bits)
  uint32_t* count;          // [B]: chunks done
  SpecOut o;
};
struct ResShared {
  float f[RES_NT / 64];
  uint32_t u[RES_NT / 64];
  double d[RES_NT / 64];
  float M[2];
  double Z[2];
  uint32_t before[2];
  int found, last;
  double run;
};
// One of a request's two rows: its logits and its kept set (key > lo, or key
// == lo and tie rank < n_tie).
struct ResRow {
  const char* p;
  uint32_t lo, n_tie;
};
template <int DT>
__device__ __forceinline__ void res_rows(const ResParams& P, int b, int j, ResRow (&row)[2]) {
  constexpr int ES = DT == LPS_DTYPE_F32 ? 4 : 2;
  const int64_t rt = (int64_t)b * (P.k + 1) + j, rd = (int64_t)P.B * (P.k + 1) + (int64_t)b * P.k + j;
  row[0] = ResRow{reinterpret_cast<const char*>(P.tl) + ES * ((int64_t)b * P.tsb + (int64_t)j * P.tsk),
                  f2key(P.cut[rt]), P.ties[rt] < 0 ? kNoTie : (uint32_t)P.ties[rt]};
  row[1] = ResRow{reinterpret_cast<const char*>(P.dl) + ES * ((int64_t)b * P.dsb + (int64_t)j * P.dsk),
                  f2key(P.cut[rd]), P.ties[rd] < 0 ? kNoTie : (uint32_t)P.ties[rd]};
}
// Whether both rows of request b's first rejection were sampled.
__device__ __forceinline__ bool res_rows_ok(const ResParams& P, int b, int j) {
  return P.status[(int64_t)b * (P.k + 1) + j] == 0 &&
         P.status[(int64_t)P.B * (P.k + 1) + (int64_t)b * P.k + j] == 0;
}
// This thread's scaled logits of chunk c: slot v VEC + e is id c RES_CH + (v
// RES_NT + tid) VEC + e; returns the number of slots inside the row, a prefix.
template <int DT, int VEC>
__device__ __forceinline__ int res_load(const char* row, int c, int V, float T, float (&z)[RES_PT]) {
  int n = 0;
#pragma unroll
  for (int v = 0; v < RES_PT / VEC; v++) {
    const int64_t i0 = (int64_t)c * RES_CH + ((int64_t)v * RES_NT + threadIdx.x) * VEC;
    float x[VEC];
#pragma unroll
    for (int e = 0; e < VEC; e++) x[e] = -INFINITY;
    if (i0 < V) {   // (VEC > 1: the row is whole vectors)
      loadv<DT, VEC, false>(row, i0, x);
      n += VEC;
    }
#pragma unroll
    for (int e = 0; e < VEC; e++) z[v * VEC + e] = __fdiv_rn(x[e], T);
  }
  return n;
}
template <typename T, typename Op>
__device__ __forceinline__ T res_reduce(T v, T* slot, Op op) {
  v = wreduce(v, op);
  if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
  __syncthreads();
  T r = slot[0];
#pragma unroll
  for (int w = 1; w < RES_NT / 64; w++) r = op(r, slot[w]);
  __syncthreads();
  return r;
}

template <int DT, int VEC>
__global__ __launch_bounds__(RES_NT) void residual_stats_kernel(ResParams P) {
  __shared__ ResShared S;
  const int G = res_chunks(P.V);
  const int b = (int)blockIdx.x / G, c = (int)blockIdx.x % G;
  if (c == 0 && threadIdx.x == 0) {
    spec_epilogue_request(b, P.k, P.T, P.p_t, P.q_d, P.draws_t, P.draft_tokens, P.u_acc, P.o);
    P.count[b] = 0u;
  }
  const int j = spec_first_reject(b, P.k, P.T, P.p_t, P.q_d, P.u_acc);
  if (j >= P.k || !res_rows_ok(P, b, j)) return;   // uniform over the workgroup
  ResRow row[2];
  res_rows<DT>(P, b, j, row);
#pragma unroll
  for (int q = 0; q < 2; q++) {
    float z[RES_PT];
    const int n = res_load<DT, VEC>(row[q].p, c, P.V, P.T, z);
    float m = -INFINITY;
#pragma unroll
    for (int e = 0; e < RES_PT; e++) m = fmaxf(m, z[e]);
    m = res_reduce(m, S.f, OpMax{});
    double s = 0.0;
    uint32_t t = 0;
#pragma unroll
    for (int e = 0; e < RES_PT; e++) {
      const uint32_t k = f2key(z[e]);
      if (k > row[q].lo && m != -INFINITY) s += (double)mass_f(z[e], m);
      t += e < n && k == row[q].lo ? 1u : 0u;
    }
    s = res_reduce(s, S.d, OpAdd{});
    t = res_reduce(t, S.u, OpAdd{});
    if (threadIdx.x == 0) P.rec[((int64_t)b * G + c) * 2 + q] = ResRec{m, t, s};
  }
}

// The rows' maxima, kept masses and ties before chunk c, from every chunk's
// record (wave q: row q).  Ends with a barrier.
__device__ __forceinline__ void res_combine(const ResParams& P, ResShared& S, const ResRow (&row)[2], int b, int c, int G) {
  const int q = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (q < 2) {
    const ResRec* rec = P.rec + (int64_t)b * G * 2 + q;
    float M = -INFINITY;
    for (int i = l; i < G; i += 64) M = fmaxf(M, rec[2 * i].m);
    M = wreduce(M, OpMax{});
    double Z = 0.0;
    uint32_t tot = 0, before = 0;
    for (int i = l; i < G; i += 64) {
      const ResRec r = rec[2 * i];
      if (r.s > 0.0) Z += r.s * exp((double)r.m - (double)M);
      tot += r.ties;
      before += i < c ? r.ties : 0u;
    }
    Z = wreduce(Z, OpAdd{});
    tot = wreduce(tot, OpAdd{});
    before = wreduce(before, OpAdd{});
    if (l == 0) {
      const uint32_t lo = q ? row[1].lo : row[0].lo, nt = q ? row[1].n_tie : row[0].n_tie;
      const uint32_t kept = nt < tot ? nt : tot;
      S.M[q] = M;
      S.Z[q] = Z + (kept ? (double)kept * (double)mass_f(key2f(lo), M) : 0.0);
      S.before[q] = before;
    }
  }
  __syncthreads();
}
// max(p - q, 0) of this thread's ids of chunk c (0 past the row).
template <int DT, int VEC>
__device__ __forceinline__ void res_residual(const ResParams& P, ResShared& S, const ResRow (&row)[2], int c,
                                             double (&rr)[RES_PT]) {
#pragma unroll
  for (int q = 0; q < 2; q++) {
    float z[RES_PT];
    const int n = res_load<DT, VEC>(row[q].p, c, P.V, P.T, z);
    const uint32_t lo = row[q].lo, n_tie = row[q].n_tie;
    const float M = S.M[q];
    const double inv = 1.0 / S.Z[q];
    uint32_t run = S.before[q];
#pragma unroll
    for (int v = 0; v < RES_PT / VEC; v++) {
      // tie ranks run in vocabulary order: vector v of every thread, then v + 1
      uint32_t nt = 0, tot = 0, rank = run;
      if (n_tie != kNoTie) {   // uniform
#pragma unroll
        for (int e = 0; e < VEC; e++) nt += v * VEC + e < n && f2key(z[v * VEC + e]) == lo ? 1u : 0u;
        rank += gblock_excl_scan<uint32_t>(nt, &tot, S.u, RES_NT);
        run += tot;
      }
#pragma unroll
      for (int e = 0; e < VEC; e++) {
        const int i = v * VEC + e;
        const uint32_t k = f2key(z[i]);
        const bool kept = i < n && (k > lo || (k == lo && (n_tie == kNoTie || rank < n_tie)));
        rank += k == lo ? 1u : 0u;
        const double p = kept ? (double)mass_f(z[i], M) * inv : 0.0;
        if (q == 0) rr[i] = p;
        else rr[i] = rr[i] > p ? rr[i] - p : 0.0;
      }
    }
  }
}

template <int DT, int VEC>
__global__ __launch_bounds__(RES_NT) void residual_draw_kernel(ResParams P) {
  __shared__ ResShared S;
  const int G = res_chunks(P.V);
  const int b = (int)blockIdx.x / G, c = (int)blockIdx.x % G;
  const int j = spec_first_reject(b, P.k, P.T, P.p_t, P.q_d, P.u_acc);
  if (j >= P.k || !res_rows_ok(P, b, j)) return;   // uniform over the workgroup
  const int tid = threadIdx.x;
  ResRow row[2];
  res_rows<DT>(P, b, j, row);
  res_combine(P, S, row, b, c, G);
  double rr[RES_PT];
  res_residual<DT, VEC>(P, S, row, c, rr);
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < RES_PT; e++) s += rr[e];
  s = res_reduce(s, S.d, OpAdd{});
  // publish the chunk's sum, then count it; the request's last chunk goes on
  if (tid == 0) {
    __hip_atomic_store(&P.rsum[(int64_t)b * G + c], __builtin_bit_cast(uint64_t, s), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    S.last = __hip_atomic_fetch_add(&P.count[b], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u == (uint32_t)G;
  }
  __syncthreads();
  if (!S.last) return;   // uniform
  if (tid == 0) {
    auto chunk_sum = [&](int i) {
      return __builtin_bit_cast(double, __hip_atomic_load(&P.rsum[(int64_t)b * G + i], __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT));
    };
    double tot = 0.0;
    for (int i = 0; i < G; i++) tot += chunk_sum(i);
    float u = P.u_res[(int64_t)b * (P.k + 1) + j];
    if (!(u >= 0.0f)) u = 0.0f;
    if (u >= 1.0f) u = 0.99999994f;
    const double target = (double)u * tot;
    // the chunk holding the target (past rounding: the last with any residual)
    int f = -1;
    double run = 0.0, at = 0.0;
    if (tot > 0.0) {
      for (int i = 0; i < G; i++) {
        const double m = chunk_sum(i);
        if (!(m > 0.0)) continue;
        f = i;
        at = run;
        run += m;
        if (target < run) break;
      }
    }
    S.found = f;
    S.run = target - at;
  }
  __syncthreads();
  const int f = S.found;
  if (f < 0) return;     // no residual (uniform)
  const double target = S.run;   // inside the chunk
  if (f != c) {          // (uniform; this workgroup holds chunk c's residuals)
    res_combine(P, S, row, b, f, G);
    res_residual<DT, VEC>(P, S, row, f, rr);
  }
  __syncthreads();       // every thread has read S.found
  if (tid == 0) S.found = -1;
  // the first id whose cumulative residual exceeds the target, in vocabulary
  // order (past rounding: the last with any residual)
  double run = 0.0;
  int last_pos = -1;
#pragma unroll
  for (int v = 0; v < RES_PT / VEC; v++) {
    const int i0 = f * RES_CH + (v * RES_NT + tid) * VEC;
    double t = 0.0;
#pragma unroll
    for (int e = 0; e < VEC; e++) t += rr[v * VEC + e];
    double tot;
    double a = run + gblock_excl_scan<double>(t, &tot, S.d, RES_NT);
#pragma unroll
    for (int e = 0; e < VEC; e++) {
      const double m = rr[v * VEC + e];
      if (m > 0.0) {
        if (a <= target && target < a + m) atomicMax(&S.found, i0 + e);
        last_pos = i0 + e;
      }
      a += m;
    }
    run += tot;
  }
  const int lp = (int)res_reduce((uint32_t)(last_pos + 1), S.u, OpMax{}) - 1;   // (a barrier: S.found is final)
  if (tid == 0) {
    const int t = S.found >= 0 ? S.found : lp;
    if (t >= 0) P.o.tokens[(int64_t)b * (P.k + 1) + j] = t;
  }
}

inline hipError_t launch_residual(int dtype, bool vec, const ResParams& P, hipStream_t s) {
  const dim3 grid((unsigned)P.B * (unsigned)res_chunks(P.V));
#define LPS_RES(DT, VEC)                                                                     \
  do {                                                                                        \
    hipLaunchKernelGGL((residual_stats_kernel<DT, VEC>), grid, dim3(RES_NT), 0, s, P);         \
    hipLaunchKernelGGL((residual_draw_kernel<DT, VEC>), grid, dim3(RES_NT), 0, s, P);          \
  } while (0)
  switch (dtype) {
    case LPS_DTYPE_F32: if (vec) LPS_RES(LPS_DTYPE_F32, 4); else LPS_RES(LPS_DTYPE_F32, 1); break;
    case LPS_DTYPE_BF16: if (vec) LPS_RES(LPS_DTYPE_BF16, 8); else LPS_RES(LPS_DTYPE_BF16, 1); break;
    default: if (vec) LPS_RES(LPS_DTYPE_F16, 8); else LPS_RES(LPS_DTYPE_F16, 1); break;
  }
#undef LPS_RES
  return hipGetLastError();
}

}  // namespace lps
