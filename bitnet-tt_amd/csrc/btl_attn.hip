// Decode attention between the fused QKV BitLinear and o_proj: RoPE on the new
// q and k rows, KV-cache update at each user's position, and scaled
// dot-product attention of every query head over its key-value head's cached
// positions [0, pos] (src/bitnet_tt/layers/attention.py:1040-1262).  The
// per-(user, key-value head) body is btl_attn_body.h, which the persistent
// decode step runs too.
//
// Layout: qkv [B, (H + 2 Hkv) D] bf16 (Q heads, then K heads, then V heads);
// caches [B, Hkv, S, D] bf16 (the reference's KV-cache shape); output
// [B, H D] bf16 (heads concatenated, o_proj's input).  D = 128.
//
// One workgroup of 8 waves per (user, key-value head), or, where the caller
// gives a scratch for it and the pairs leave most of the chip idle, one per
// split of a pair's context (btl_attn_body.h): each split publishes its partial
// with coherent stores and counts itself, and the last of a pair to arrive
// merges them in split order.  Nothing waits on another workgroup.  (At the 2B
// shape's 160 pairs and 512 positions the store-acknowledge-count-reload chain
// costs more than the extra CUs gain: one split.)
#include <hip/hip_runtime.h>

#include <atomic>

#include "btl.h"
#include "btl_attn_body.h"
#include "btl_common.h"
#include "btl_trace.h"

namespace btl {

struct AttnArgs {
  const uint16_t* qkv;
  int ldq;                 // elements per qkv row
  const int32_t* pos;      // [B] position of each user's new token
  const float* rcos;       // [S, D/2] cos of position x frequency i
  const float* rsin;       // [S, D/2]
  uint16_t* kc;            // [B, Hkv, S, D]
  uint16_t* vc;            // [B, Hkv, S, D]
  uint16_t* out;           // [B, H * D]
  int32_t* error;          // set when a position is outside [0, S)
  int B, H, Hkv, G, S;
  float scale;
  int adjacent;            // 1: RoPE pairs (2i, 2i+1); 0: (i, i + D/2)
  AttnSplits sp;           // sp.smax workgroups per (user, key-value head)
  // sp.smax > 1.  A pair's arrival word is a call's number plus the splits that
  // have arrived, which is zero between calls.  Every split raises the word to
  // its own call's number before it arrives, so that a count left over from two
  // calls that ran at once on one scratch does not outlive them.
  uint64_t* arrive;        // [pairs]
  uint64_t call;           // a multiple of kAttnCallStep, larger in each later call
  float* part;             // [pairs][sp.smax][kAtPartFloats]
};
constexpr uint64_t kAttnCallStep = 16;  // > kAtMaxSplits
static_assert(kAtMaxSplits < (int)kAttnCallStep, "arrivals fit below the call's number");

constexpr int64_t kAttnWorkspace = 256;                // the error word
constexpr int64_t kAttnPart = kAtSplitItems * 8;       // split scratch: the arrival words, then the partials
static_assert(kAttnPart % 16 == 0, "partials aligned");

// Publishes this split's partial; true in the workgroup that arrived last,
// with every split's partial in Ms, Ls, Os.
__device__ bool attn_gather(const AttnArgs& p, const AttnPair& a, int pair, int n, const AttnPartial& mine,
                            int* s_last, float (&Ms)[kAtMaxSplits], float (&Ls)[kAtMaxSplits],
                            float (&Os)[kAtMaxSplits]) {
  const int tid = threadIdx.x, g = tid / kAtD;
  float* const base = p.part + (int64_t)pair * p.sp.smax * kAtPartFloats;
  if (g < a.G) {
    float* const o = base + a.split * kAtPartFloats;
    st_coherent(o + tid, mine.O);
    if (tid % kAtD == 0) {
      st_coherent(o + kAtMaxG * kAtD + 2 * g, mine.M);
      st_coherent(o + kAtMaxG * kAtD + 2 * g + 1, mine.L);
    }
  }
  wait_memory();
  __syncthreads();  // the whole partial is out before the arrival is counted
  if (tid == 0) {
    const uint64_t w = atomicAdd(reinterpret_cast<unsigned long long*>(p.arrive + pair), 1ull);
    const uint64_t arrived = w % kAttnCallStep;
    *s_last = arrived == (uint64_t)(n - 1);
    if (*s_last) st_coherent(p.arrive + pair, w - arrived);  // left clean for the next call
  }
  __syncthreads();
  if (!*s_last) return false;
  const int gc = min(g, a.G - 1);
#pragma unroll
  for (int i = 0; i < kAtMaxSplits; ++i)
    if (i < n) {
      const float* const o = base + i * kAtPartFloats;
      Os[i] = ld_coherent(o + tid);
      Ms[i] = ld_coherent(o + kAtMaxG * kAtD + 2 * gc);
      Ls[i] = ld_coherent(o + kAtMaxG * kAtD + 2 * gc + 1);
    }
  return true;
}

// SPLIT: sp.smax > 1 workgroups per pair.
template <bool SPLIT>
__global__ __launch_bounds__(64 * kAtWaves, 1) void k_decode_attention(AttnArgs p) {
  __shared__ __attribute__((aligned(16))) AttnSmem s;
  __shared__ int s_last;
  const int tid = threadIdx.x;
  BTL_TRACE_AT(0);
  AttnPair a;
  a.rcos = p.rcos;
  a.rsin = p.rsin;
  a.kc = p.kc;
  a.vc = p.vc;
  a.Hkv = p.Hkv;
  a.G = p.G;
  a.S = p.S;
  // grid (Hkv, B, splits), so no index needs a division; every pair's split 0
  // first: they are spread over the XCDs, and where a context is one round they
  // do not queue behind workgroups that only leave
  a.hk = blockIdx.x;
  a.b = blockIdx.y;
  a.split = SPLIT ? blockIdx.z : 0;
  a.sp = SPLIT ? p.sp : AttnSplits{1, 0};
  const int pair = a.b * p.Hkv + a.hk;
  a.scale = p.scale;
  a.adjacent = p.adjacent;
  a.tid = tid;
  AttnRound r;
  if (!att_load_first<true>(a, p.pos + a.b, r)) return;
  BTL_TRACE_AT(1);
  if (!a.pos_ok() && tid == 0 && a.hk == 0 && a.split == 0) st_coherent(p.error, 1);
  // the new token's rows of the group: q rows hk G .. hk G + G - 1, k row hk, v row hk
  const uint16_t* qrow = p.qkv + (int64_t)a.b * p.ldq;
  if (tid < (kAtMaxG + 2) * (kAtD / 8)) {
    const int u = tid / (kAtD / 8), c = tid % (kAtD / 8);
    const int src = u < kAtMaxG ? a.hk * a.G + u : u == kAtMaxG ? p.H + a.hk : p.H + p.Hkv + a.hk;
    if (u >= kAtMaxG || u < a.G)
      *reinterpret_cast<uint4*>(&s.in[u][8 * c]) = *reinterpret_cast<const uint4*>(qrow + (int64_t)src * kAtD + 8 * c);
  }
  __syncthreads();
  BTL_TRACE_AT(2);
  AttnPartial part;
  const int n = SPLIT ? a.n : 1;
  // long before this split's own arrival, which waits for it
  if (SPLIT && n > 1 && tid == 0) atomicMax(reinterpret_cast<unsigned long long*>(p.arrive + pair), p.call);
  uint16_t o = att_body(a, s, r, part, true);
  if (SPLIT && n > 1) {
    float Ms[kAtMaxSplits], Ls[kAtMaxSplits], Os[kAtMaxSplits];
    if (!attn_gather(p, a, pair, n, part, &s_last, Ms, Ls, Os)) return;
    o = tid < a.G * kAtD ? att_merge(s, tid, n, Ms, Ls, Os) : 0;
  }
  if (tid < a.G * kAtD) p.out[(int64_t)a.b * p.H * kAtD + (a.hk * a.G) * kAtD + tid] = o;
  BTL_TRACE_AT(7);
}

}  // namespace btl

using namespace btl;

BTL_TRACE_READ_FN(btl_trace_read_attention)

extern "C" {

int64_t btl_decode_attention_workspace_bytes(int64_t B, int64_t H, int64_t Hkv, int64_t S) {
  if (B <= 0 || Hkv <= 0 || H <= 0 || H % Hkv || H / Hkv > kAtMaxG || S <= 0) return 0;
  return kAttnWorkspace;
}

int64_t btl_decode_attention_split_bytes(int64_t B, int64_t Hkv, int64_t S) {
  if (B <= 0 || Hkv <= 0 || S <= 0) return 0;
  // at most kAtSplitItems splits, on any device
  if (att_max_splits(B * Hkv, S, kAtSplitItems + 32) == 1) return 0;
  return kAttnPart + (int64_t)kAtSplitItems * kAtPartFloats * 4;
}

int64_t btl_decode_attention_error_offset(int64_t B, int64_t Hkv) {
  (void)B;
  (void)Hkv;
  return 0;
}

static int decode_attention(const char* who, const uint16_t* qkv, int64_t B, int64_t H, int64_t Hkv, int64_t D,
                            int64_t S, const int32_t* pos, const float* rope_cos, const float* rope_sin,
                            int rope_adjacent, float scale, uint16_t* k_cache, uint16_t* v_cache, uint16_t* out,
                            void* workspace, size_t workspace_bytes, void* split, size_t split_bytes,
                            btl_stream_t stream) {
  clear_error();
  if (D != kAtD) return set_error(BTL_ERR_SHAPE, "%s: head dim %lld (128 supported)", who, (long long)D);
  if (B <= 0 || B > 4096 || Hkv <= 0 || H <= 0 || H % Hkv || H / Hkv > kAtMaxG || S <= 0 || S > (1 << 20))
    return set_error(BTL_ERR_SHAPE, "%s: B=%lld H=%lld Hkv=%lld S=%lld (H/Hkv <= %d)", who, (long long)B,
                     (long long)H, (long long)Hkv, (long long)S, kAtMaxG);
  if (!qkv || !pos || !rope_cos || !rope_sin || !k_cache || !v_cache || !out || !workspace)
    return set_error(BTL_ERR_NULL, "%s: NULL pointer", who);
  if (!aligned(qkv, 16) || !aligned(k_cache, 16) || !aligned(v_cache, 16) || !aligned(out, 16) ||
      !aligned(workspace, 256) || !aligned(pos, 4) || !aligned(rope_cos, 4) || !aligned(rope_sin, 4) ||
      !aligned(split, 16))
    return set_error(BTL_ERR_ALIGN, "%s: misaligned buffer", who);
  if ((int64_t)workspace_bytes < kAttnWorkspace)
    return set_error(BTL_ERR_WORKSPACE, "%s: workspace %zu < %lld bytes", who, workspace_bytes,
                     (long long)kAttnWorkspace);
  if (split && (int64_t)split_bytes < btl_decode_attention_split_bytes(B, Hkv, S))
    return set_error(BTL_ERR_WORKSPACE, "%s: split scratch %zu < %lld bytes", who, split_bytes,
                     (long long)btl_decode_attention_split_bytes(B, Hkv, S));
  static std::atomic<uint64_t> calls{0};
  AttnArgs a;
  a.qkv = qkv;
  a.ldq = (int)((H + 2 * Hkv) * D);
  a.pos = pos;
  a.rcos = rope_cos;
  a.rsin = rope_sin;
  a.kc = k_cache;
  a.vc = v_cache;
  a.out = out;
  a.B = (int)B;
  a.H = (int)H;
  a.Hkv = (int)Hkv;
  a.G = (int)(H / Hkv);
  a.S = (int)S;
  a.scale = scale;
  a.adjacent = rope_adjacent ? 1 : 0;
  a.error = reinterpret_cast<int32_t*>(workspace);
  a.sp = split ? att_splits(B, H, Hkv, S, device_cus()) : AttnSplits{1, 0};
  a.arrive = nullptr;
  a.call = 0;
  a.part = nullptr;
  if (a.sp.smax > 1) {
    a.arrive = reinterpret_cast<uint64_t*>(split);
    a.call = kAttnCallStep * (calls.fetch_add(1, std::memory_order_relaxed) + 1);
    a.part = reinterpret_cast<float*>(static_cast<char*>(split) + kAttnPart);
  }
  const dim3 grid((unsigned)Hkv, (unsigned)B, (unsigned)a.sp.smax);
  if (a.sp.smax > 1)
    hipLaunchKernelGGL(k_decode_attention<true>, grid, dim3(64 * kAtWaves), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(k_decode_attention<false>, grid, dim3(64 * kAtWaves), 0, (hipStream_t)stream, a);
  return check_launch("decode attention");
}

int btl_decode_attention(const uint16_t* qkv, int64_t B, int64_t H, int64_t Hkv, int64_t D, int64_t S,
                         const int32_t* pos, const float* rope_cos, const float* rope_sin, int rope_adjacent,
                         float scale, uint16_t* k_cache, uint16_t* v_cache, uint16_t* out, void* workspace,
                         size_t workspace_bytes, btl_stream_t stream) {
  return decode_attention("btl_decode_attention", qkv, B, H, Hkv, D, S, pos, rope_cos, rope_sin, rope_adjacent, scale,
                          k_cache, v_cache, out, workspace, workspace_bytes, nullptr, 0, stream);
}

int btl_decode_attention_split(const uint16_t* qkv, int64_t B, int64_t H, int64_t Hkv, int64_t D, int64_t S,
                               const int32_t* pos, const float* rope_cos, const float* rope_sin, int rope_adjacent,
                               float scale, uint16_t* k_cache, uint16_t* v_cache, uint16_t* out, void* workspace,
                               size_t workspace_bytes, void* split, size_t split_bytes, btl_stream_t stream) {
  return decode_attention("btl_decode_attention_split", qkv, B, H, Hkv, D, S, pos, rope_cos, rope_sin, rope_adjacent,
                          scale, k_cache, v_cache, out, workspace, workspace_bytes, split, split_bytes, stream);
}

}  // extern "C"
