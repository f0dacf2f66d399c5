// Route scoring: per-row log-sum-exp over the vocabulary and the gather of the
// log-probabilities of the verified tokens, so a verify needs one small
// device-to-host copy instead of one scalar read per token.
#include <algorithm>
#include <cfloat>

#include "common.hpp"

namespace atlas {
namespace {

constexpr int kThreads = 256;

template <int DT>
__device__ __forceinline__ float load_logit(const char* row, int64_t i) {
  if constexpr (DT == ATLAS_DTYPE_F32) {
    return reinterpret_cast<const float*>(row)[i];
  } else if constexpr (DT == ATLAS_DTYPE_F16) {
    return static_cast<float>(reinterpret_cast<const _Float16*>(row)[i]);
  } else {
    return static_cast<float>(reinterpret_cast<const __bf16*>(row)[i]);
  }
}

// 16 bytes of logits -> up to 8 floats.
template <int DT>
struct Vec {
  static constexpr int kElems = DT == ATLAS_DTYPE_F32 ? 4 : 8;
  float x[kElems];
  __device__ __forceinline__ void load(const char* p) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    if constexpr (DT == ATLAS_DTYPE_F32) {
      x[0] = __uint_as_float(u.x);
      x[1] = __uint_as_float(u.y);
      x[2] = __uint_as_float(u.z);
      x[3] = __uint_as_float(u.w);
    } else {
      const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (DT == ATLAS_DTYPE_F16) {
          x[2 * k] = static_cast<float>(__builtin_bit_cast(_Float16, uint16_t(w[k] & 0xffff)));
          x[2 * k + 1] = static_cast<float>(__builtin_bit_cast(_Float16, uint16_t(w[k] >> 16)));
        } else {
          x[2 * k] = __uint_as_float(w[k] << 16);
          x[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
        }
      }
    }
  }
};

// Workgroup (c, r) reads chunk c of logits row r once: the chunk's maximum m
// and the sum of exp(x - m), kept online per thread over batches of kBatch
// 16-byte loads, then reduced over the workgroup.  It stores the pair into its
// slot of the row, waits until the store is acknowledged and counts itself in on
// the row's arrival counter (a row of one chunk needs neither); the
// workgroup that arrives last (the counter held num_chunks - 1) reads every
// slot, combines the pairs in chunk order (a fixed order, so the LSE is the same
// on every run), writes the row LSE and every gather of row r, and empties the
// slots and the counter for the next call.  A slot is (max bits, ~sum bits),
// never zero, and carries its whole message in one agent-scope atomic: the last
// arriver takes a slot as written when it is not zero, whatever order the stores
// of different workgroups become visible in, so no workgroup needs a release (a
// write-back of its XCD's whole L2).  A workgroup stores its slot without waiting
// for anything, so the last arriver finds it, normally at the first read; a slot
// still zero after kSlotTries reads counts as a NaN sum.  Only launches in stream
// order may share a workspace: another launch's pair in a slot is taken as this
// launch's own.
struct GatherArgs {
  const char* logits;
  int64_t row_stride_bytes;
  const char* logits2;          // rows num_rows1 .. come from here (or null)
  int64_t row_stride2_bytes;
  int64_t num_rows1;
  int64_t vocab;
  const int32_t* rows;
  const int64_t* tokens;
  int64_t n;
  float* row_lse;
  float* out;
  uint64_t* slots;     // [num_rows, num_chunks], zero between calls
  uint32_t* arrivals;  // [num_rows], zero between calls
  int num_chunks;
  int64_t chunk_len;  // elements, a multiple of 8 (the last chunk may be shorter)
};

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kFar = 2.3e38f;  // kLog2e * kFar is finite
constexpr int kPre = 2;    // gathers per thread whose logits are loaded ahead of the combine
constexpr int kSlotTries = 1 << 14;  // reads of a slot before it is given up
constexpr int kBatch = 4;  // 16-byte loads a thread has in flight (8 measured slower: 26.9 us against 24.1)

// (m, s) pairs: s is a sum of exp(x - m), and while m is -inf 0, or NaN when a
// NaN has been met: a maximum drops a NaN, so the sum carries it.  exp_ref is
// what exponents are taken relative to: with it, -inf adds 0 and keeps a NaN,
// without a branch.
__device__ __forceinline__ float exp_ref(float m) { return m == -INFINITY ? 0.f : m; }

__device__ __forceinline__ void pair_merge(float& m, float& s, float m2, float s2) {
  const float mn = fmaxf(m, m2);
  const float ref = exp_ref(mn);
  s = s * __builtin_amdgcn_exp2f((m - ref) * kLog2e) + s2 * __builtin_amdgcn_exp2f((m2 - ref) * kLog2e);
  m = mn;
}

// Adds N vectors to a thread's (m, s).
template <int DT, int N>
__device__ __forceinline__ void batch_add(const Vec<DT> (&x)[N], float& m, float& s) {
  constexpr int EPV = Vec<DT>::kElems;
  float mn = m;
#pragma unroll
  for (int b = 0; b < N; ++b)
#pragma unroll
    for (int k = 0; k < EPV; ++k) mn = fmaxf(mn, x[b].x[k]);
  const float ref = exp_ref(mn);
  // (past kFar the product overflows: kept finite, so the sum is 0 and not NaN
  // until a larger logit comes, and folded again at the end if none does)
  const float mb = DT == ATLAS_DTYPE_F16 ? ref * kLog2e : __builtin_amdgcn_fmed3f(ref * kLog2e, -FLT_MAX, FLT_MAX);
  float acc = s * __builtin_amdgcn_exp2f((m - ref) * kLog2e);
#pragma unroll
  for (int b = 0; b < N; ++b) {
    float part = 0.f;
#pragma unroll
    for (int k = 0; k < EPV; ++k) part += __builtin_amdgcn_exp2f(__builtin_fmaf(x[b].x[k], kLog2e, -mb));
    acc += part;
  }
  m = mn;
  s = acc;
}

template <int DT>
__global__ __launch_bounds__(kThreads) void gather_logprobs_kernel(GatherArgs a) {
  __shared__ float red_m[kThreads / 64];
  __shared__ float red_s[kThreads / 64];
  __shared__ int last_sh;
  __shared__ float lse_sh;
  constexpr int EPV = Vec<DT>::kElems;
  const int c = blockIdx.x;
  const int r = blockIdx.y;
  const int t = threadIdx.x;
  const char* row = r < a.num_rows1 ? a.logits + int64_t(r) * a.row_stride_bytes
                                    : a.logits2 + (int64_t(r) - a.num_rows1) * a.row_stride2_bytes;
  const int64_t c0 = int64_t(c) * a.chunk_len;
  const int64_t c1 = min(a.vocab, c0 + a.chunk_len);

  // Row and token of the first kPre * kThreads gathers, requested before the
  // chunk (no branch on them: a branch would wait for them first).
  int32_t grow[kPre];
  int64_t gtok[kPre];
#pragma unroll
  for (int k = 0; k < kPre; ++k) {
    const int64_t i = min(t + int64_t(k) * kThreads, max(a.n - 1, int64_t(0)));
    grow[k] = a.n > 0 ? a.rows[i] : -1;
    gtok[k] = a.n > 0 ? a.tokens[i] : 0;
  }

  // 16-byte loads over the chunk's aligned part [a0, a1); at most EPV - 1 single
  // elements before it and after it (rows of an odd vocabulary start anywhere).
  constexpr int ES = DT == ATLAS_DTYPE_F32 ? 4 : 2;
  const int lead = static_cast<int>((-reinterpret_cast<uintptr_t>(row + c0 * ES) & 15) / ES);
  const int64_t a0 = min(c1, c0 + lead);
  const int64_t nv = (c1 - a0) / EPV;
  const int64_t a1 = a0 + nv * EPV;
  const char* vrow = row + a0 * ES;
  float m = -INFINITY, s = 0.f;
  int64_t v = t;
  // full batches: one running maximum and one rescale per kBatch vectors
  for (; v + int64_t(kBatch - 1) * kThreads < nv; v += int64_t(kBatch) * kThreads) {
    Vec<DT> x[kBatch];
#pragma unroll
    for (int b = 0; b < kBatch; ++b) x[b].load(vrow + (v + int64_t(b) * kThreads) * 16);
    batch_add<DT, kBatch>(x, m, s);
  }
  for (; v < nv; v += kThreads) {
    Vec<DT> x[1];
    x[0].load(vrow + v * 16);
    batch_add<DT, 1>(x, m, s);
  }
  // Nothing but logits masked with the type's lowest value (or a maximum as
  // large): the same vectors again, by difference.
  if (DT != ATLAS_DTYPE_F16 && __builtin_fabsf(m) > kFar && m != -INFINITY) {
    s = 0.f;
#pragma unroll 1
    for (v = t; v < nv; v += kThreads) {
      Vec<DT> x;
      x.load(vrow + v * 16);
#pragma unroll
      for (int k = 0; k < EPV; ++k) s += __builtin_amdgcn_exp2f((x.x[k] - m) * kLog2e);
    }
  }
  const int singles = static_cast<int>((a0 - c0) + (c1 - a1));
  if (t < singles) {
    const int64_t i = t < a0 - c0 ? c0 + t : a1 + (t - (a0 - c0));
    pair_merge(m, s, load_logit<DT>(row, i), 1.f);
  }
  // The gathered logits go out now and land while the pair is published.  Lanes
  // whose gather belongs to another row read the chunk's first logit instead: a
  // read at their own token would fetch a line of this row that nobody needs.
  float gx[kPre];
  bool gmine[kPre];
#pragma unroll
  for (int k = 0; k < kPre; ++k) {
    gmine[k] = t + int64_t(k) * kThreads < a.n && grow[k] == r;
    const bool ok = gtok[k] >= 0 && gtok[k] < a.vocab;
    gx[k] = load_logit<DT>(row, gmine[k] && ok ? gtok[k] : c0);
    if (!ok) gx[k] = NAN;
  }
  // workgroup reduction of (m, s)
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) pair_merge(m, s, __shfl_xor(m, off), __shfl_xor(s, off));
  if ((t & 63) == 0) {
    red_m[t >> 6] = m;
    red_s[t >> 6] = s;
  }
  __syncthreads();
  uint64_t* rs = a.slots + int64_t(r) * a.num_chunks;
  if (t == 0) {
    float bm = red_m[0], bs = red_s[0];
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) pair_merge(bm, bs, red_m[w], red_s[w]);
    if (bs != bs) bs = NAN;  // (one NaN pattern: ~sum is not zero)
    const uint64_t slot = uint64_t(__float_as_uint(bm)) | (uint64_t(~__float_as_uint(bs)) << 32);
    bool last = true;
    if (a.num_chunks > 1) {
      __hip_atomic_store(rs + c, slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // The slot's store is acknowledged before the arrival goes out, so the
      // last arriver finds every slot at its first read.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const uint32_t prev = __hip_atomic_fetch_add(a.arrivals + r, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = prev == uint32_t(a.num_chunks - 1);
    } else {
      lse_sh = bm + __builtin_log2f(bs) * kLn2;
    }
    last_sh = last;
  }
  __syncthreads();
  if (!last_sh) return;

  // The last arriver: combine the row's slots in chunk order (one per lane of
  // wave 0, then a fixed pairwise tree).
  if (t < 64 && a.num_chunks > 1) {
    float cm = -INFINITY, cs = 0.f;
    for (int k = t; k < a.num_chunks; k += 64) {
      // (bounded: launches that share a workspace out of stream order could
      // empty each other's slots; an empty slot reads as a NaN sum)
      uint64_t v = 0;
      for (int tries = 0; v == 0 && tries < kSlotTries; ++tries)
        v = __hip_atomic_load(rs + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      pair_merge(cm, cs, __uint_as_float(uint32_t(v)), __uint_as_float(~uint32_t(v >> 32)));
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) pair_merge(cm, cs, __shfl_xor(cm, off), __shfl_xor(cs, off));
    if (t == 0) lse_sh = cm + __builtin_log2f(cs) * kLn2;
  }
  __syncthreads();
  const float lse = lse_sh;
  if (t == 0 && a.row_lse) a.row_lse[r] = lse;
  if (a.num_chunks > 1) {
    if (t == 0) __hip_atomic_store(a.arrivals + r, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int k = t; k < a.num_chunks; k += kThreads)
      __hip_atomic_store(rs + k, uint64_t(0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int k = 0; k < kPre; ++k)
    if (gmine[k]) a.out[t + int64_t(k) * kThreads] = gx[k] - lse;
  for (int64_t i = t + int64_t(kPre) * kThreads; i < a.n; i += kThreads) {
    if (a.rows[i] != r) continue;
    const int64_t tok = a.tokens[i];
    a.out[i] = (tok >= 0 && tok < a.vocab) ? load_logit<DT>(row, tok) - lse : NAN;
  }
}

}  // namespace
}  // namespace atlas

using namespace atlas;

namespace atlas {
namespace {
// Chunks per row, from the row count and the vocabulary in batches (what a
// workgroup folds in one round: kBatch 16-byte loads per thread, 8192 16-bit or
// 4096 fp32 logits).  A launch takes as long as one workgroup's rounds in series,
// 0.4 to 0.5 us each, plus 1.3 to 1.8 us for slots and arrivals when a row has
// more than one chunk, until rows x chunks fills the device; beyond that each
// further workgroup costs its reduction and its arrival.  So: chunks of few
// batches for few rows, and of more batches the more workgroups there are
// already.  The limits on rows x chunks lie where the next length is faster;
// more than 12 arrivals on one row's counter only pay in small launches; rows of
// up to 4 batches, and 16-bit rows from the stated count on, are faster as
// one chunk.  A chunk is whole batches (what is left of one is folded a vector at a
// time, each a round trip of its own), or the row's even share where that leaves
// half a batch or less.
//
// Measured, us (graph replays over cold logits): this rule against chunks of at
// least 16384 logits for 400 or 512 workgroups, and one chunk per row:
//   x 128256 bf16     1 row  4.8,  6.1, 12.7     5  5.6,  6.8, 13.4    20  7.2,  7.9, 13.8
//                       50   8.5,  9.6, 18.0   100 10.1, 11.3, 18.4   170 13.2, 13.3, 19.5
//                      200  15.4, 16.9, 19.9   300 20.9, 21.6, 22.2   399 24.1, 27.3, 24.0
//                      416  24.4, 24.5, 24.4   (a write-back of L2 per workgroup and
//                      every lane reading its gather's token in every row: 41.4)
//   x 128256 fp32     1      5.0,  7.0, 23.7     5  6.3,  8.1, 26.0    20  7.6,  9.2, 26.9
//                       50  10.8, 12.2, 37.4   100 14.1, 14.4, 38.2   200 23.4, 24.1, 41.4
//                      399  42.1, 42.1, 49.3   512 51.1, 53.2, 53.3
//   x 32001 bf16      1      4.8,  5.7,  4.7    35  6.5,  7.1,  6.5   200  9.1, 10.0,  9.1
//   x 32001 fp32      1      4.6,  5.9,  5.5    35  6.7,  8.4,  9.5   200 11.2, 12.8, 14.1
// Over 1 to 600 rows of 9001 to 152064 logits the rule is within 6 % of the best
// chunk length tried, mostly within 2 %.
struct GatherGeom {
  int num_chunks;
  int64_t chunk_len;
};
GatherGeom gather_geom(int64_t num_rows, int64_t vocab, int esize) {
  const int64_t batch = int64_t(kBatch) * kThreads * (16 / esize);
  const int64_t batches = (vocab + batch - 1) / batch;
  if (batches <= 4 || (esize == 2 && num_rows >= std::max<int64_t>(224, 24 * batches)))
    return GatherGeom{1, (vocab + 7) / 8 * 8};
  const int64_t most16[] = {128, 400, 600, 500, 768}, most32[] = {128, 400, 600, 1024, 1024};
  int64_t per = 1, chunks = batches;
  while (chunks > 1) {
    const int64_t i = std::min<int64_t>(per, 5) - 1;
    if (num_rows * chunks <= (chunks > 12 ? 150 : esize == 4 ? most32[i] : most16[i])) break;
    per = (batches + chunks - 2) / (chunks - 1);  // the next length with fewer chunks
    chunks = (batches + per - 1) / per;
  }
  const int64_t even = (vocab + chunks * 8 - 1) / (chunks * 8) * 8;  // (chunks start on 8 logits)
  return GatherGeom{int(chunks), even % batch <= batch / 2 ? even : per * batch};
}
}  // namespace
}  // namespace atlas

extern "C" int64_t atlas_gather_logprobs_workspace_bytes(int64_t num_rows, int64_t vocab) {
  if (num_rows <= 0 || vocab <= 0 || num_rows >= (int64_t(1) << 31)) return -1;
  const int chunks = std::max(gather_geom(num_rows, vocab, 2).num_chunks, gather_geom(num_rows, vocab, 4).num_chunks);
  // (of either logit size) the slots, then one arrival counter per row
  return int64_t(size_t(num_rows) * chunks * sizeof(uint64_t) + size_t(num_rows) * sizeof(uint32_t));
}

extern "C" int atlas_gather_logprobs(const void* logits_dev, int64_t row_stride, int64_t num_rows,
                                     const void* logits2_dev, int64_t row_stride2, int64_t num_rows2, int64_t vocab,
                                     int dtype, const int32_t* row_dev, const int64_t* token_dev, int64_t n,
                                     float* row_lse_dev, float* out_dev, void* workspace_dev, size_t workspace_bytes,
                                     void* stream) {
  ATLAS_REQUIRE(logits_dev && num_rows > 0 && vocab > 0, "bad logits arguments");
  ATLAS_REQUIRE(num_rows2 >= 0 && (num_rows2 == 0 || logits2_dev != nullptr), "bad second logits arguments");
  ATLAS_REQUIRE(n == 0 || (row_dev && token_dev && out_dev), "gather buffers must not be NULL");
  const int64_t total_rows = num_rows + num_rows2;
  ATLAS_REQUIRE(total_rows < (int64_t(1) << 31), "too many rows");
  const int es = dtype == ATLAS_DTYPE_F32 ? 4 : 2;
  ATLAS_REQUIRE(dtype == ATLAS_DTYPE_F32 || dtype == ATLAS_DTYPE_F16 || dtype == ATLAS_DTYPE_BF16, "bad dtype");
  ATLAS_REQUIRE(row_stride >= vocab && (num_rows2 == 0 || row_stride2 >= vocab),
                "row strides (elements) must cover the vocabulary");
  const int64_t need = atlas_gather_logprobs_workspace_bytes(total_rows, vocab);
  ATLAS_REQUIRE(workspace_dev != nullptr && workspace_bytes >= size_t(need),
                "workspace of %lld bytes needed (atlas_gather_logprobs_workspace_bytes), got %zu", (long long)need,
                workspace_bytes);
  ATLAS_REQUIRE((reinterpret_cast<uintptr_t>(workspace_dev) & 15) == 0, "workspace must be 16-byte aligned");
  const GatherGeom g = gather_geom(total_rows, vocab, es);
  GatherArgs a{};
  a.logits = static_cast<const char*>(logits_dev);
  a.row_stride_bytes = row_stride * es;
  a.logits2 = static_cast<const char*>(logits2_dev);
  a.row_stride2_bytes = row_stride2 * es;
  a.num_rows1 = num_rows;
  a.vocab = vocab;
  a.rows = row_dev;
  a.tokens = token_dev;
  a.n = n;
  a.row_lse = row_lse_dev;
  a.out = out_dev;
  a.slots = static_cast<uint64_t*>(workspace_dev);
  a.arrivals = reinterpret_cast<uint32_t*>(a.slots + total_rows * g.num_chunks);
  a.num_chunks = g.num_chunks;
  a.chunk_len = g.chunk_len;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(g.num_chunks), static_cast<unsigned>(total_rows));
  if (dtype == ATLAS_DTYPE_F32)
    hipLaunchKernelGGL((gather_logprobs_kernel<ATLAS_DTYPE_F32>), grid, dim3(kThreads), 0, s, a);
  else if (dtype == ATLAS_DTYPE_F16)
    hipLaunchKernelGGL((gather_logprobs_kernel<ATLAS_DTYPE_F16>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((gather_logprobs_kernel<ATLAS_DTYPE_BF16>), grid, dim3(kThreads), 0, s, a);
  return launch_status("gather_logprobs_kernel");
}
