// Single-token attention over the generation caches (decode steps).
//
// Reference semantics:
//   * sliding-window GQA decode (parrot/model.py:239-262): the new key and
//     value (RoPE applied) are stored at cache position p, and each query
//     head attends over keys max(0, p - W + 1) .. p of its kv head,
//     softmax(q k^T * scale) v with scale 1/sqrt(head_dim);
//   * MLA decode with absorbed weights (parrot/model.py:362-432): the new
//     latent is stored at p and each head's fp32 query attends over latents
//     0 .. p, which serve as both keys and values, scale head_dim^-0.5; the
//     context stays fp32 for the absorbed output map.
// p is read from device memory, so a decode step has static shapes and can
// be captured once in a HIP graph and replayed as the position advances.
//
// One workgroup per (query head, sequence).  Scores: one key per thread,
// all 16-byte chunks of its row loaded at once, fp32 dot with the query in
// LDS; softmax in fp32 over the scores kept in LDS; values: each thread owns
// one 16-byte chunk of the rows of a key slot, and the slot partials are
// added in a fixed order.  The key and value at p are read from the new rows
// (not from the cache being written), so no workgroup waits for another.
#include "common.h"

namespace parrot {

namespace {

__device__ __forceinline__ float to_f32(uint16_t v) { return __uint_as_float(uint32_t(v) << 16); }
__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ void store_out(uint16_t* p, float v) { *p = f32_to_bf16(v); }
__device__ __forceinline__ void store_out(float* p, float v) { *p = v; }

__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp<0xb1>(v));
  v = fmaxf(v, dpp<0x4e>(v));
  v = fmaxf(v, dpp<0x141>(v));
  v = fmaxf(v, dpp<0x140>(v));
  const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

// Workgroup (4 wavefronts) reductions through `red` [4], fixed order.
__device__ __forceinline__ float block_max(float v, float* red) {
  v = wave_max(v);
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const float r = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  return r;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const float r = ((red[0] + red[1]) + red[2]) + red[3];
  __syncthreads();
  return r;
}

constexpr int kVPre = 8;  // value rows per thread loaded at kernel entry

// Output-projection operands of decode_attention_kernel with Q > 0: the
// [dim, heads x head_dim] bf16 weight and the fp32 per-head contributions
// [batch, heads, dim] it writes.
struct HeadsOut {
  const uint16_t* weight;
  int dim;
  float* contributions;
};

// CH = head_dim / 8 16-byte chunks per key / value row.
//
// Q = 0: one workgroup per (head, sequence) writes the head's output row.
// Q > 0 (bf16 query and output, the deferred residual): Q workgroups per
// (head, sequence) each attend over the window (the same arithmetic, so the
// same bits) and project the head's bf16-rounded output onto a Q-th of the
// output width: contributions[b, h, n] = sum_i out[i] * W[n, h D + i] in
// index order.  Each thread's weight row piece is loaded at entry, so the
// projection's operands arrive during the attention.  The contributions'
// sum over heads is left to the consumer (the reference's PendingResidual).
template <typename QT, typename OT, int CH, int Q>
__global__ __launch_bounds__(256) void decode_attention_kernel(
    const QT* __restrict__ q, const uint16_t* __restrict__ k_new,
    const uint16_t* __restrict__ v_new, uint16_t* __restrict__ k_cache,
    uint16_t* __restrict__ v_cache, const int32_t* __restrict__ position, int heads,
    int kv_heads, int max_pos, int window, float scale, OT* __restrict__ out, HeadsOut ho) {
  constexpr int D = CH * 8;
  constexpr int kSlots = 256 / CH;  // value pass: key slots x chunks
  static_assert(D <= 256, "one query element per thread");
  extern __shared__ float smem[];
  // The kernel arguments in one batch of scalar loads, before any use.
  asm volatile("" ::"s"(q), "s"(k_new), "s"(v_new), "s"(k_cache), "s"(v_cache), "s"(position),
               "s"(heads), "s"(kv_heads), "s"(max_pos), "s"(window), "s"(scale));
  if constexpr (Q > 0) asm volatile("" ::"s"(ho.weight), "s"(ho.dim), "s"(ho.contributions));
  // The device position first, read through the constant address space (it
  // does not change during the launch) so that it is a scalar load: the
  // cache rows' addresses wait for it alone, not for the element loads below
  // (a vector load's wait would cover those too).
  using const_i32 = const __attribute__((address_space(4))) int32_t;
  const int pos = *(const_i32*)(reinterpret_cast<uintptr_t>(position));
  __builtin_amdgcn_sched_barrier(0);
  const int h = Q > 0 ? static_cast<int>(blockIdx.x) / Q : static_cast<int>(blockIdx.x);
  const int part_n = Q > 0 ? static_cast<int>(blockIdx.x) % Q : 0;
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int rep = heads / kv_heads;
  const int kvh = h / rep;
  const int lcap = min(window, max_pos);
  float* s = smem;                 // [lcap] scores, then probabilities
  float* qs = s + lcap;            // [D]
  float* part = qs + D;            // [kSlots][D]
  float* red = part + kSlots * D;  // [4]
  float* ob = red + 4;             // [D] (Q > 0) the head's rounded output

  // Q > 0: thread t < dim / Q owns output column n = part_n dim / Q + t.
  const int nq = Q > 0 ? ho.dim / Q : 0;

  // This thread's elements of the new key / value rows (stored below) and
  // of the query (D <= 256), then the device position: none depends on the
  // position, so they are in flight together, and the cache rows behind
  // them wait for one round trip.  These loads go first, so their uses wait
  // for none of the row loads behind them (loads complete in order).
  const int64_t kv_index = static_cast<int64_t>(b) * kv_heads + kvh;
  const uint16_t* kn = k_new + kv_index * D;
  const uint16_t* vn = v_new + kv_index * D;
  const int ie = min(tid, D - 1);
  const uint16_t kne = kn[ie], vne = vn[ie];
  const float qv = to_f32(q[(static_cast<int64_t>(b) * heads + h) * D + ie]);
  asm volatile("" ::: "memory");
  if (pos < 0 || pos >= max_pos) return;  // uniform: nothing to attend to
  const int lo = max(0, pos - window + 1);
  const int L = pos - lo + 1;
  const uint16_t* kc = k_cache + kv_index * max_pos * D;
  const uint16_t* vc = v_cache + kv_index * max_pos * D;

  // The first pass of key rows (key lo + tid) and the first kVPre value rows
  // of this thread's (slot, chunk) are loaded here, together with the query:
  // none of them depends on another, so the scores and the value pass do not
  // each wait for a memory round trip of their own.
  auto key_row = [&](int key) -> const uint4* {
    return reinterpret_cast<const uint4*>(key == pos ? kn : kc + static_cast<int64_t>(key) * D);
  };
  auto value_row = [&](int key) -> const uint4* {
    return reinterpret_cast<const uint4*>(key == pos ? vn : vc + static_cast<int64_t>(key) * D);
  };
  uint4 kr0[CH];
  {
    const uint4* row = key_row(lo + min(tid, L - 1));
#pragma unroll
    for (int c = 0; c < CH; ++c) kr0[c] = row[c];
  }
  const int chunk = tid % CH;
  const int slot = tid / CH;
  uint4 vpre[kVPre];
#pragma unroll
  for (int u = 0; u < kVPre; ++u)
    vpre[u] = value_row(lo + min(slot + u * kSlots, L - 1))[chunk];

  // Q > 0: the D weights W[n, h D .. h D + D) (16-byte aligned) of this
  // thread's output column, issued after every load the attention waits
  // for, so they arrive during it.
  uint4 wo[Q > 0 ? CH : 1];
  if constexpr (Q > 0) {
    asm volatile("" ::: "memory");
    const uint4* wrow = reinterpret_cast<const uint4*>(
        ho.weight + static_cast<int64_t>(part_n * nq + min(tid, nq - 1)) * heads * D + h * D);
#pragma unroll
    for (int c = 0; c < CH; ++c) wo[c] = wrow[c];
  }
  // The first head of each kv group stores the new key / value row.
  if (h % rep == 0 && part_n == 0 && tid < D) {
    k_cache[(kv_index * max_pos + pos) * D + tid] = kne;
    if (v_cache != k_cache) v_cache[(kv_index * max_pos + pos) * D + tid] = vne;
  }
  if (tid < D) qs[tid] = qv;
  __syncthreads();

  auto score = [&](const uint4 (&kr)[CH]) -> float {
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const float* qc = qs + c * 8;
      acc += lo_bf16(kr[c].x) * qc[0] + hi_bf16(kr[c].x) * qc[1] + lo_bf16(kr[c].y) * qc[2] +
             hi_bf16(kr[c].y) * qc[3] + lo_bf16(kr[c].z) * qc[4] + hi_bf16(kr[c].z) * qc[5] +
             lo_bf16(kr[c].w) * qc[6] + hi_bf16(kr[c].w) * qc[7];
    }
    return acc * scale;
  };

  // Scores: one key per thread per pass, every chunk of its row in flight.
  float mx = -INFINITY;
  if (tid < L) {
    const float acc = score(kr0);
    s[tid] = acc;
    mx = acc;
  }
  for (int j = tid + 256; j < L; j += 256) {
    const uint4* row = key_row(lo + j);
    uint4 kr[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) kr[c] = row[c];
    const float acc = score(kr);
    s[j] = acc;
    mx = fmaxf(mx, acc);
  }
  mx = block_max(mx, red);
  float sum = 0.0f;
  for (int j = tid; j < L; j += 256) {
    const float e = __expf(s[j] - mx);
    s[j] = e;
    sum += e;
  }
  sum = block_sum(sum, red);  // also orders the probability writes before the reads below

  // Values: thread = (key slot, 16-byte chunk); slot k takes keys k,
  // k + kSlots, ...: the first kVPre from the rows loaded at entry, then
  // four rows in flight at a time.  Partials per slot are added in slot
  // order below.
  float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto accumulate = [&](const uint4& vr, float p) {
    a[0] += p * lo_bf16(vr.x);
    a[1] += p * hi_bf16(vr.x);
    a[2] += p * lo_bf16(vr.y);
    a[3] += p * hi_bf16(vr.y);
    a[4] += p * lo_bf16(vr.z);
    a[5] += p * hi_bf16(vr.z);
    a[6] += p * lo_bf16(vr.w);
    a[7] += p * hi_bf16(vr.w);
  };
  if (slot < kSlots) {
#pragma unroll
    for (int u = 0; u < kVPre; ++u) {
      const int j = slot + u * kSlots;
      accumulate(vpre[u], j < L ? s[min(j, L - 1)] : 0.0f);
    }
    for (int j0 = slot + kVPre * kSlots; j0 < L; j0 += 4 * kSlots) {
      uint4 vr[4];
      float p[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = min(j0 + u * kSlots, L - 1);
        const int key = lo + j;
        vr[u] = value_row(key)[chunk];
        p[u] = j0 + u * kSlots < L ? s[j] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) accumulate(vr[u], p[u]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) part[slot * D + chunk * 8 + i] = a[i];
  }
  __syncthreads();
  const float inv = 1.0f / sum;
  if constexpr (Q == 0) {
    for (int i = tid; i < D; i += 256) {
      float o = 0.0f;
      for (int k = 0; k < kSlots; ++k) o += part[k * D + i];
      store_out(out + (static_cast<int64_t>(b) * heads + h) * D + i, o * inv);
    }
  } else {
    // The head's output rounded to bf16, as the output projection of the
    // undeferred path reads it, then this workgroup's output columns.
    for (int i = tid; i < D; i += 256) {
      float o = 0.0f;
      for (int k = 0; k < kSlots; ++k) o += part[k * D + i];
      ob[i] = to_f32(f32_to_bf16(o * inv));
    }
    __syncthreads();
    if (tid < nq) {
      float acc = 0.0f;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const float* oc = ob + c * 8;
        acc += lo_bf16(wo[c].x) * oc[0] + hi_bf16(wo[c].x) * oc[1] + lo_bf16(wo[c].y) * oc[2] +
               hi_bf16(wo[c].y) * oc[3] + lo_bf16(wo[c].z) * oc[4] + hi_bf16(wo[c].z) * oc[5] +
               lo_bf16(wo[c].w) * oc[6] + hi_bf16(wo[c].w) * oc[7];
      }
      ho.contributions[(static_cast<int64_t>(b) * heads + h) * ho.dim + part_n * nq + tid] = acc;
    }
  }
}

template <typename QT, typename OT, int Q = 0>
hipError_t launch_decode(const QT* q, const uint16_t* k_new, const uint16_t* v_new,
                         uint16_t* k_cache, uint16_t* v_cache, const int32_t* position, int batch,
                         int heads, int kv_heads, int head_dim, int max_pos, int window,
                         float scale, OT* out, hipStream_t s, HeadsOut ho = HeadsOut{}) {
  const size_t lds = decode_attention_lds_bytes(window, max_pos, head_dim) +
                     (Q > 0 ? static_cast<size_t>(head_dim) * sizeof(float) : 0);
  const dim3 grid(heads * (Q > 0 ? Q : 1), batch);
#define PARROT_DECODE(CH)                                                                   \
  decode_attention_kernel<QT, OT, CH, Q><<<grid, 256, lds, s>>>(                            \
      q, k_new, v_new, k_cache, v_cache, position, heads, kv_heads, max_pos, window, scale, \
      out, ho)
  switch (head_dim / 8) {
    case 1: PARROT_DECODE(1); break;
    case 2: PARROT_DECODE(2); break;
    case 4: PARROT_DECODE(4); break;
    case 8: PARROT_DECODE(8); break;
    case 12: PARROT_DECODE(12); break;
    case 16: PARROT_DECODE(16); break;
    case 24: PARROT_DECODE(24); break;
    case 32: PARROT_DECODE(32); break;
    default: return hipErrorInvalidValue;
  }
#undef PARROT_DECODE
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Long contexts: the keys split over workgroups.
//
// One workgroup per (head, sequence) streams the whole window through one
// CU: 28.8 us at 2048 keys (b = 1), 31.6 us (b = 8) and 65 us for the latent
// layers at 3900 keys (b = 4), for 1.6, 12.6 and 4 MB of keys and values that the
// chip reads from HBM in 0.3, 2.4 and 0.8 us.
// Here a workgroup takes kSplitKeys = 64 consecutive keys of one kv head for
// all the query heads that share it, so each row is read once (not once per
// head), and leaves (max, sum, unnormalised output) per head in a workspace;
// a second launch merges a head's chunks in chunk order and, for the deferred
// residual, projects its share of the output columns as the one-launch kernel
// does.  64 keys give b = 1 64 workgroups at the 2048-key window and b = 8
// 512; the launch is sized for the whole window, chunks past the position
// exit at once.
//
//   scores    v_mfma_f32_16x16x32_bf16, A = the group's query heads (rows
//             past them zero), B = 16 keys per wavefront straight from the
//             cache rows.  An fp32 query (latent layers) enters as three bf16
//             parts that add up to it exactly, accumulated in fp32, so the
//             products are as exact as the fp32 dot's.
//   softmax   one key per lane per head, fp32, within the wavefront that owns
//             the head.
//   values    staged in LDS once; wavefront w sums heads w, w + 4, ... in
//             fp32 over (key slot, 16-byte chunk) lanes.
constexpr int kSplitKeys = 64;
constexpr int kSplitMaxChunks = 256;  // chunk weights the merge keeps in LDS

// A 16-byte fragment (8 values) of a query row as bf16 parts whose sum is the
// row: one part for a bf16 query, three for an fp32 one (8 + 8 + 8 bits).
template <typename QT>
constexpr int kQueryParts = sizeof(QT) == 4 ? 3 : 1;

__device__ __forceinline__ void query_parts(const uint16_t* p, bool live, bf16x8 (&part)[1]) {
  const uint4 v = *reinterpret_cast<const uint4*>(p);
  part[0] = __builtin_bit_cast(bf16x8, live ? v : make_uint4(0u, 0u, 0u, 0u));
}

__device__ __forceinline__ void query_parts(const float* p, bool live, bf16x8 (&part)[3]) {
  const float4 a = reinterpret_cast<const float4*>(p)[0];
  const float4 b = reinterpret_cast<const float4*>(p)[1];
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int t = 0; t < 3; ++t) w[t][i] = 0u;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float rest = live ? v[2 * i + j] : 0.0f;
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const uint16_t h = f32_to_bf16(rest);
        w[t][i] |= static_cast<uint32_t>(h) << (16 * j);
        // An infinite part leaves no remainder (inf - inf would be NaN).
        const float part_v = bf16_to_f32(h);
        rest = __builtin_isinf(part_v) ? 0.0f : rest - part_v;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 3; ++t)
    part[t] = __builtin_bit_cast(bf16x8, make_uint4(w[t][0], w[t][1], w[t][2], w[t][3]));
}

// CH = head_dim / 8 (a multiple of 4); HPW = query heads per wavefront,
// heads / kv_heads <= 4 HPW <= 16.
template <typename QT, int CH, int HPW>
__global__ __launch_bounds__(256) void decode_split_kernel(
    const QT* __restrict__ q, const uint16_t* __restrict__ k_new,
    const uint16_t* __restrict__ v_new, uint16_t* __restrict__ k_cache,
    uint16_t* __restrict__ v_cache, const int32_t* __restrict__ position, int heads,
    int kv_heads, int max_pos, int window, float scale, float2* __restrict__ part_ml,
    float* __restrict__ part_o) {
  constexpr int D = CH * 8;
  constexpr int KS = D / 32;             // MFMA k steps of a score
  constexpr int kLanes = CH <= 16 ? 16 : 32;  // lanes per key slot in the value pass
  constexpr int kSlots = kWave / kLanes;      // key slots per wavefront
  constexpr int kParts = kQueryParts<QT>;
  constexpr int kPieces = kSplitKeys * CH / 256;  // value pieces staged per thread
  __shared__ __attribute__((aligned(16))) uint16_t v_s[kSplitKeys * D];
  __shared__ float s_s[4 * HPW][kSplitKeys];

  asm volatile("" ::"s"(q), "s"(k_new), "s"(v_new), "s"(k_cache), "s"(v_cache), "s"(position),
               "s"(heads), "s"(kv_heads), "s"(max_pos), "s"(window), "s"(scale), "s"(part_ml),
               "s"(part_o));
  using const_i32 = const __attribute__((address_space(4))) int32_t;
  const int pos = *(const_i32*)(reinterpret_cast<uintptr_t>(position));
  const int chunk = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  if (pos < 0 || pos >= max_pos) return;  // uniform: nothing to attend to
  const int lo = max(0, pos - window + 1);
  const int L = pos - lo + 1;
  const int c0 = chunk * kSplitKeys;
  if (c0 >= L) return;  // uniform: no keys here
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rep = heads / kv_heads;

  const int64_t kv_index = static_cast<int64_t>(b) * kv_heads + kvh;
  const uint16_t* kn = k_new + kv_index * D;
  const uint16_t* vn = v_new + kv_index * D;
  uint16_t* kc = k_cache + kv_index * max_pos * D;
  uint16_t* vc = v_cache + kv_index * max_pos * D;
  // Keys past the last one (of the final chunk) read its row; their scores
  // are masked below.  The row at `pos` comes from the new rows.
  auto row = [&](const uint16_t* cache, const uint16_t* fresh, int j) -> const uint16_t* {
    const int key = lo + min(j, L - 1);
    return key == pos ? fresh : cache + static_cast<int64_t>(key) * D;
  };

  // This wavefront's 16 keys, then its share of the values, then the query heads.
  // The keys' loads are in flight together; at head widths from 96 on the compiler
  // keeps `vr` in scratch memory (64 to 144 bytes per lane), so each value piece is
  // waited for, stored and read back, and each k step waits for its query load.
  const int g = lane >> 4, c = lane & 15;
  bf16x8 kf[KS];
  {
    const uint16_t* kr = row(kc, kn, c0 + 16 * wave + c) + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s)
      kf[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(kr + 32 * s));
  }
  const QT* qrow = q + (static_cast<int64_t>(b) * heads + kvh * rep + min(c, rep - 1)) * D + 8 * g;
  uint4 vr[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int piece = i * 256 + tid;
    vr[i] = *reinterpret_cast<const uint4*>(row(vc, vn, c0 + piece / CH) + (piece % CH) * 8);
  }
  // An fp32 query's leading parts in two chains (even and odd steps) and the
  // other parts in a third, added once: in one chain of twelve products the
  // scores were rounded more often than the one-launch dot's, and an output of
  // 352 to 1000 keys was 1.2-1.4 times as far from fp64 (now 0.6-0.9 times).
  f32x4 sc = {0.f, 0.f, 0.f, 0.f}, odd = {0.f, 0.f, 0.f, 0.f}, rest = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    bf16x8 part[kParts];
    query_parts(qrow + 32 * s, c < rep, part);
    f32x4& lead = kParts > 1 && s % 2 == 1 ? odd : sc;
    lead = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part[0], kf[s], lead, 0, 0, 0);
#pragma unroll
    for (int t = kParts - 1; t >= 1; --t)  // small parts first
      rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part[t], kf[s], rest, 0, 0, 0);
  }
  if constexpr (kParts > 1) {
    // An infinite key makes the leading products infinite, but NaN of a later
    // part that is 0 or of the other sign.
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float lead = sc[r] + odd[r];
      sc[r] = __builtin_isfinite(lead) ? sc[r] + (odd[r] + rest[r]) : lead;
    }
  }
  // The chunk that holds `pos` stores the new rows.
  if (c0 + kSplitKeys >= L && tid < D) {
    kc[static_cast<int64_t>(pos) * D + tid] = kn[tid];
    if (v_cache != k_cache) vc[static_cast<int64_t>(pos) * D + tid] = vn[tid];
  }
#pragma unroll
  for (int i = 0; i < kPieces; ++i)
    *reinterpret_cast<uint4*>(v_s + (i * 256 + tid) * 8) = vr[i];
  // C fragment: lane holds key c of the wavefront's 16, heads 4 g + r.
  const bool valid = c0 + 16 * wave + c < L;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * g + r < 4 * HPW) s_s[4 * g + r][16 * wave + c] = valid ? sc[r] * scale : -INFINITY;
  __syncthreads();

  const int64_t part0 = (static_cast<int64_t>(b) * heads + kvh * rep) * gridDim.x + chunk;
  const int slot = lane / kLanes, vch = lane % kLanes;
  float acc[HPW][8];
#pragma unroll
  for (int i = 0; i < HPW; ++i) {
    const int h = wave + 4 * i;
    const float v = s_s[h][lane];
    const float m = wave_max(v);
    // A chunk whose scores are all -inf weighs nothing; the maximum passes
    // over NaN scores, which stay NaN.
    const float e = m == -INFINITY && v == v ? 0.0f : __expf(v - m);
    const float l = wave_sum(e);
    s_s[h][lane] = e;  // read back by this wavefront only
    if (lane == 0 && h < rep)
      part_ml[part0 + static_cast<int64_t>(h) * gridDim.x] = make_float2(m, l);
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[i][k] = 0.0f;
  }
  const int vlane = min(vch, CH - 1);
#pragma unroll 4
  for (int j = slot; j < kSplitKeys; j += kSlots) {
    const uint4 x = *reinterpret_cast<const uint4*>(v_s + j * D + vlane * 8);
    const float xv[8] = {lo_bf16(x.x), hi_bf16(x.x), lo_bf16(x.y), hi_bf16(x.y),
                         lo_bf16(x.z), hi_bf16(x.z), lo_bf16(x.w), hi_bf16(x.w)};
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
      const float p = s_s[wave + 4 * i][j];
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[i][k] += p * xv[k];
    }
  }
#pragma unroll
  for (int i = 0; i < HPW; ++i) {
    const int h = wave + 4 * i;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if constexpr (kSlots == 4) acc[i][k] += __shfl_xor(acc[i][k], 16);
      acc[i][k] += __shfl_xor(acc[i][k], 32);
    }
    if (slot == 0 && vch < CH && h < rep) {
      float4* o = reinterpret_cast<float4*>(
          part_o + (part0 + static_cast<int64_t>(h) * gridDim.x) * D + vch * 8);
      o[0] = make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
      o[1] = make_float4(acc[i][4], acc[i][5], acc[i][6], acc[i][7]);
    }
  }
}

// Merges a head's chunks: output = sum_c e^(m_c - M) o_c / sum_c e^(m_c - M)
// l_c with M = max_c m_c.  Q as in decode_attention_kernel.
template <typename OT, int CH, int Q>
__global__ __launch_bounds__(256) void decode_merge_kernel(
    const float2* __restrict__ part_ml, const float* __restrict__ part_o,
    const int32_t* __restrict__ position, int heads, int max_pos, int window, int chunks,
    OT* __restrict__ out, HeadsOut ho) {
  constexpr int D = CH * 8;
  constexpr int kVec = D / 4;            // float4 pieces of an output row
  constexpr int kGroups = 256 / kVec;    // chunks summed side by side
  constexpr int kPre = 8;                // pieces per thread loaded at entry
  __shared__ float w_s[kSplitMaxChunks];
  __shared__ float4 part_s[kGroups][kVec];
  __shared__ float ob[D];
  asm volatile("" ::"s"(part_ml), "s"(part_o), "s"(position), "s"(heads), "s"(max_pos),
               "s"(window), "s"(chunks), "s"(out));
  if constexpr (Q > 0) asm volatile("" ::"s"(ho.weight), "s"(ho.dim), "s"(ho.contributions));
  using const_i32 = const __attribute__((address_space(4))) int32_t;
  const int pos = *(const_i32*)(reinterpret_cast<uintptr_t>(position));
  const int h = Q > 0 ? static_cast<int>(blockIdx.x) / Q : static_cast<int>(blockIdx.x);
  const int part_n = Q > 0 ? static_cast<int>(blockIdx.x) % Q : 0;
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int nq = Q > 0 ? ho.dim / Q : 0;
  if (pos < 0 || pos >= max_pos) return;
  const int L = min(pos + 1, window);
  const int n = (L + kSplitKeys - 1) / kSplitKeys;  // live chunks
  const int64_t row = static_cast<int64_t>(b) * heads + h;
  const float2* ml = part_ml + row * chunks;
  const float4* po = reinterpret_cast<const float4*>(part_o + row * chunks * D);

  const float2 ml0 = ml[min(lane, n - 1)];
  const int vec = tid % kVec, grp = tid / kVec;
  float4 pre[kPre];
#pragma unroll
  for (int u = 0; u < kPre; ++u) pre[u] = po[static_cast<int64_t>(min(grp + u * kGroups, n - 1)) * kVec + vec];
  uint4 wo[Q > 0 ? CH : 1];
  if constexpr (Q > 0) {
    asm volatile("" ::: "memory");
    const uint4* wrow = reinterpret_cast<const uint4*>(
        ho.weight + static_cast<int64_t>(part_n * nq + min(tid, nq - 1)) * heads * D + h * D);
#pragma unroll
    for (int c = 0; c < CH; ++c) wo[c] = wrow[c];
  }
  // Every wavefront derives the same maximum and denominator.
  float mx = lane < n ? ml0.x : -INFINITY;
  for (int c = lane + kWave; c < n; c += kWave) mx = fmaxf(mx, ml[c].x);
  mx = wave_max(mx);
  float w0 = lane < n ? __expf(ml0.x - mx) : 0.0f;
  float sum = w0 * (lane < n ? ml0.y : 0.0f);
  if (tid < n && tid < kWave) w_s[tid] = w0;
  for (int c = lane + kWave; c < n; c += kWave) {
    const float2 v = ml[c];
    const float w = __expf(v.x - mx);
    if (tid < kWave) w_s[c] = w;
    sum += w * v.y;
  }
  sum = wave_sum(sum);
  __syncthreads();
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
  auto add = [&](const float4& o, float w) {
    a.x += w * o.x;
    a.y += w * o.y;
    a.z += w * o.z;
    a.w += w * o.w;
  };
  if (grp < kGroups) {
#pragma unroll
    for (int u = 0; u < kPre; ++u) {
      const int c = grp + u * kGroups;
      if (c < n) add(pre[u], w_s[c]);
    }
    for (int c = grp + kPre * kGroups; c < n; c += kGroups) add(po[static_cast<int64_t>(c) * kVec + vec], w_s[c]);
    part_s[grp][vec] = a;
  }
  __syncthreads();
  const float inv = 1.0f / sum;
  const float* ps = reinterpret_cast<const float*>(part_s);
  for (int i = tid; i < D; i += 256) {
    float o = 0.0f;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) o += ps[k * D + i];
    if constexpr (Q == 0) store_out(out + row * D + i, o * inv);
    else ob[i] = to_f32(f32_to_bf16(o * inv));
  }
  if constexpr (Q > 0) {
    __syncthreads();
    if (tid < nq) {
      float acc = 0.0f;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const float* oc = ob + c * 8;
        acc += lo_bf16(wo[c].x) * oc[0] + hi_bf16(wo[c].x) * oc[1] + lo_bf16(wo[c].y) * oc[2] +
               hi_bf16(wo[c].y) * oc[3] + lo_bf16(wo[c].z) * oc[4] + hi_bf16(wo[c].z) * oc[5] +
               lo_bf16(wo[c].w) * oc[6] + hi_bf16(wo[c].w) * oc[7];
      }
      ho.contributions[row * ho.dim + part_n * nq + tid] = acc;
    }
  }
}

// (max, sum) entries of the workspace, padded to whole 16-byte pairs so the
// partial outputs behind them stay aligned.
size_t decode_split_ml_entries(int batch, int heads, int chunks) {
  return (static_cast<size_t>(batch) * heads * chunks + 1) / 2 * 2;
}

int split_chunks(int max_pos, int window) {
  return ((window < max_pos ? window : max_pos) + kSplitKeys - 1) / kSplitKeys;
}

template <typename QT, typename OT, int Q>
hipError_t launch_decode_split(const QT* q, const uint16_t* k_new, const uint16_t* v_new,
                               uint16_t* k_cache, uint16_t* v_cache, const int32_t* position,
                               int batch, int heads, int kv_heads, int head_dim, int max_pos,
                               int window, float scale, OT* out, HeadsOut ho, void* workspace,
                               hipStream_t s) {
  const int chunks = split_chunks(max_pos, window);
  float2* ml = static_cast<float2*>(workspace);
  float* po = reinterpret_cast<float*>(ml + decode_split_ml_entries(batch, heads, chunks));
  const dim3 grid(chunks, kv_heads, batch);
  const dim3 merge_grid(heads * (Q > 0 ? Q : 1), batch);
  const int rep = heads / kv_heads;
#define PARROT_SPLIT(CH, HPW)                                                              \
  decode_split_kernel<QT, CH, HPW><<<grid, 256, 0, s>>>(q, k_new, v_new, k_cache, v_cache, \
                                                        position, heads, kv_heads, max_pos, \
                                                        window, scale, ml, po)
#define PARROT_SPLIT_CH(CH)                                                                \
  if (rep <= 4) PARROT_SPLIT(CH, 1);                                                       \
  else if (rep <= 8) PARROT_SPLIT(CH, 2);                                                  \
  else PARROT_SPLIT(CH, 4);                                                                \
  decode_merge_kernel<OT, CH, Q><<<merge_grid, 256, 0, s>>>(ml, po, position, heads,       \
                                                            max_pos, window, chunks, out, ho)
  switch (head_dim) {
    case 32: PARROT_SPLIT_CH(4); break;
    case 64: PARROT_SPLIT_CH(8); break;
    case 96: PARROT_SPLIT_CH(12); break;
    case 128: PARROT_SPLIT_CH(16); break;
    case 192: PARROT_SPLIT_CH(24); break;
    case 256: PARROT_SPLIT_CH(32); break;
    default: return hipErrorInvalidValue;
  }
#undef PARROT_SPLIT_CH
#undef PARROT_SPLIT
  return hipGetLastError();
}

}  // namespace

bool decode_head_dim_supported(int head_dim) {
  switch (head_dim) {
    case 8: case 16: case 32: case 64: case 96: case 128: case 192: case 256: return true;
    default: return false;
  }
}

size_t decode_attention_lds_bytes(int window, int max_pos, int head_dim) {
  const int lcap = window < max_pos ? window : max_pos;
  const int slots = 256 / (head_dim / 8 > 0 ? head_dim / 8 : 1);
  return (static_cast<size_t>(lcap) + head_dim + static_cast<size_t>(slots) * head_dim + 4) *
         sizeof(float);
}

hipError_t launch_decode_attention(const uint16_t* q, const uint16_t* k_new,
                                   const uint16_t* v_new, uint16_t* k_cache, uint16_t* v_cache,
                                   const int32_t* position, int batch, int heads, int kv_heads,
                                   int head_dim, int max_pos, int window, float scale,
                                   uint16_t* out, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  return launch_decode(q, k_new, v_new, k_cache, v_cache, position, batch, heads, kv_heads,
                       head_dim, max_pos, window, scale, out, s);
}

hipError_t launch_decode_attention_heads(const uint16_t* q, const uint16_t* k_new,
                                         const uint16_t* v_new, uint16_t* k_cache,
                                         uint16_t* v_cache, const int32_t* position, int batch,
                                         int heads, int kv_heads, int head_dim, int max_pos,
                                         int window, float scale, const uint16_t* out_weight,
                                         int dim, float* contributions, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  if (dim % kDecodeHeadsParts != 0 || dim / kDecodeHeadsParts > 256)
    return hipErrorInvalidValue;
  return launch_decode<uint16_t, uint16_t, kDecodeHeadsParts>(
      q, k_new, v_new, k_cache, v_cache, position, batch, heads, kv_heads, head_dim, max_pos,
      window, scale, nullptr, s, HeadsOut{out_weight, dim, contributions});
}

hipError_t launch_decode_attention_latent(const float* q, const uint16_t* latent_new,
                                          uint16_t* latent_cache, const int32_t* position,
                                          int batch, int heads, int latent_dim, int max_pos,
                                          float scale, float* out, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  return launch_decode(q, latent_new, latent_new, latent_cache, latent_cache, position, batch,
                       heads, 1, latent_dim, max_pos, max_pos, scale, out, s);
}

bool decode_split_supported(int heads, int kv_heads, int head_dim, int max_pos, int window) {
  return head_dim % 32 == 0 && decode_head_dim_supported(head_dim) && heads / kv_heads <= 16 &&
         split_chunks(max_pos, window) <= kSplitMaxChunks;
}

size_t decode_split_workspace_bytes(int batch, int heads, int head_dim, int max_pos, int window) {
  const int chunks = split_chunks(max_pos, window);
  return decode_split_ml_entries(batch, heads, chunks) * sizeof(float2) +
         static_cast<size_t>(batch) * heads * chunks * head_dim * sizeof(float);
}

hipError_t launch_decode_attention_split(const uint16_t* q, const uint16_t* k_new,
                                         const uint16_t* v_new, uint16_t* k_cache,
                                         uint16_t* v_cache, const int32_t* position, int batch,
                                         int heads, int kv_heads, int head_dim, int max_pos,
                                         int window, float scale, uint16_t* out,
                                         void* workspace, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  return launch_decode_split<uint16_t, uint16_t, 0>(q, k_new, v_new, k_cache, v_cache, position,
                                                    batch, heads, kv_heads, head_dim, max_pos,
                                                    window, scale, out, HeadsOut{}, workspace, s);
}

hipError_t launch_decode_attention_heads_split(
    const uint16_t* q, const uint16_t* k_new, const uint16_t* v_new, uint16_t* k_cache,
    uint16_t* v_cache, const int32_t* position, int batch, int heads, int kv_heads, int head_dim,
    int max_pos, int window, float scale, const uint16_t* out_weight, int dim,
    float* contributions, void* workspace, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  if (dim % kDecodeHeadsParts != 0 || dim / kDecodeHeadsParts > 256)
    return hipErrorInvalidValue;
  return launch_decode_split<uint16_t, uint16_t, kDecodeHeadsParts>(
      q, k_new, v_new, k_cache, v_cache, position, batch, heads, kv_heads, head_dim, max_pos,
      window, scale, static_cast<uint16_t*>(nullptr), HeadsOut{out_weight, dim, contributions},
      workspace, s);
}

hipError_t launch_decode_attention_latent_split(const float* q, const uint16_t* latent_new,
                                                uint16_t* latent_cache, const int32_t* position,
                                                int batch, int heads, int latent_dim,
                                                int max_pos, float scale, float* out,
                                                void* workspace, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  return launch_decode_split<float, float, 0>(q, latent_new, latent_new, latent_cache,
                                              latent_cache, position, batch, heads, 1, latent_dim,
                                              max_pos, max_pos, scale, out, HeadsOut{}, workspace,
                                              s);
}

}  // namespace parrot
