// Causal (optionally sliding-window) attention for long sequences: the
// arithmetic of causal_attention_kernel (attention.hip) on
// v_mfma_f32_32x32x16_bf16 with K and V shared through LDS.
//
// causal_attention_kernel gives a workgroup 16 queries of one head and lets
// every wavefront read its own key blocks, so a 12 KB block (32 keys of K and V
// at D = 96) that leaves L2 serves 0.2 MFLOP: 18 TB/s at the 290 TFLOP/s it
// reaches on long sequences.  Here a wavefront owns 32 queries, the four of
// a workgroup cover HW heads that share the kv head, and all of them read the
// same key blocks from LDS, filled by direct-to-LDS copies (fragment-order K
// and V are contiguous per block) while the blocks before are computed.
//
//   S^T = K Q^T   A = 32 keys, B = 32 queries: lane l holds the scores of
//                 query l % 32 for 16 of the block's keys.
//   O^T += V^T P^T  P^T comes straight from those registers as the B operand.
//                 Row i of the K operand is key 16 j + 4 (2 s + h) + r of the
//                 block (i = 16 s + 8 j + 4 h + r), so that the 8 scores a
//                 lane holds per 16-key step are the keys
//                 {4 g .. + 3, 16 + 4 g .. + 3}, g = 2 s + l / 32, of one
//                 16-byte piece of the V fragments.
//
// Precision: P enters its product as two bf16 parts (16 bits).  The eight
// wavefronts of causal_attention_kernel have a running maximum each, which makes
// eight large P of a query exactly 1; with one state (or two) and P rounded to
// one bf16, an output was 3-5 % further from fp64 than there.  Relative to that
// kernel's error, 24 x 512 tokens, queries 0.3 / 1 / 3 / 8 / 20 times a normal
// draw: 0.76 / 0.83 / 0.93 / 0.990 / 0.996.  The six products that this adds to a
// block's twelve cost 12-28 % (4 x 4096 93 -> 120 us, 2 x 2047 28 -> 34).  With
// the second part for every other 16 keys only, and the maximum raised by 2^2
// instead of 2^8, it was 106 and 31 us, but the error 1.001 to 1.004 where few keys
// dominate.
//
// What bounds it: 18 MFMAs (576 clocks at D = 96) and about 125 vector
// instructions, 16 of them exp2, per 32 keys and 32 queries; three workgroups
// per CU, out of step with each other, overlap the two in part (4 x 4096 runs at
// 650 TFLOP/s of visible products, 40 % of the MFMA rate with the second part of
// P).  A wavefront alone runs at about half the rate, so a grid's last workgroups
// and small grids wait for the serial chain of the longest queries.  Measured and
// not kept, before P had two parts: 64 queries per wavefront (half the LDS reads,
// two wavefronts per SIMD: 105 against 92 us at 4 x 4096), two blocks interleaved
// in one wavefront (105 us), eight or sixteen wavefronts on one barrier (their
// softmaxes collide: 120 and 150 us), deeper rings of stages (no change).
//
// KG = 2 gives every other block of a stage to a second group of wavefronts,
// merged through LDS at the end: half the queries per workgroup, twice the
// workgroups, half the serial chain, at twice the K / V traffic.
//
// Measured on MI355X (us in graphs of 20 launches, causal_attention_kernel /
// KG = 1 / KG = 2, 8 heads of 96, 2 kv heads, window 2048): 4 x 4096 268 / 119 /
// 121; 3 x 4096 201 / 92 / 94; 2 x 4096 135 / 74 / 68; 16 x 512 80 / 20 / 21;
// 1 x 2000 32 / 44 / 29; 2 x 520 13.7 / 15.2 / 11.9; 1 x 1050 17.2 / 26.1 / 17.8;
// 8 kv heads, causal: 2 x 2047 65 / 47 / 33; 1 x 2047 36 / 45 / 30.
#include "common.h"
#include "extents.h"

namespace parrot {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));


struct TileArgs {
  const uint16_t* q;
  const uint16_t* kf;   // fragment order (kfrag_index)
  const uint16_t* vf;   // fragment order (vfrag_index)
  int64_t qs[3];        // element strides: batch, head, row
  int seq, heads, kv_heads, window;
  float scale_log2;     // |scale| log2(e)
  uint32_t q_sign;      // 0x80008000 for a negative scale (q is negated), else 0
  uint16_t* out;        // [batch, seq, heads, D]
};

// N fragments from LDS at addr + B + S i, landed on return.  By inline asm,
// because the compiler would otherwise wait for the direct-to-LDS copies in
// flight (the next stages) before every read; loads and wait are one block,
// so no register is named before its data is there.
template <int B, int S>
__device__ __forceinline__ void lds_frags(uint32_t addr, bf16x8 (&f)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4 offset:%5\n\tds_read_b128 %1, %4 offset:%6\n\t"
      "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %4 offset:%8\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3])
      : "v"(addr), "i"(B), "i"(B + S), "i"(B + 2 * S), "i"(B + 3 * S));
}

template <int B, int S>
__device__ __forceinline__ void lds_frags(uint32_t addr, bf16x8 (&f)[6]) {
  asm volatile(
      "ds_read_b128 %0, %6 offset:%7\n\tds_read_b128 %1, %6 offset:%8\n\t"
      "ds_read_b128 %2, %6 offset:%9\n\tds_read_b128 %3, %6 offset:%10\n\t"
      "ds_read_b128 %4, %6 offset:%11\n\tds_read_b128 %5, %6 offset:%12\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5])
      : "v"(addr), "i"(B), "i"(B + S), "i"(B + 2 * S), "i"(B + 3 * S), "i"(B + 4 * S),
        "i"(B + 5 * S));
}

template <int B, int S>
__device__ __forceinline__ void lds_frags(uint32_t addr, bf16x8 (&f)[8]) {
  asm volatile(
      "ds_read_b128 %0, %8 offset:%9\n\tds_read_b128 %1, %8 offset:%10\n\t"
      "ds_read_b128 %2, %8 offset:%11\n\tds_read_b128 %3, %8 offset:%12\n\t"
      "ds_read_b128 %4, %8 offset:%13\n\tds_read_b128 %5, %8 offset:%14\n\t"
      "ds_read_b128 %6, %8 offset:%15\n\tds_read_b128 %7, %8 offset:%16\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5]),
        "=&v"(f[6]), "=&v"(f[7])
      : "v"(addr), "i"(B), "i"(B + S), "i"(B + 2 * S), "i"(B + 3 * S), "i"(B + 4 * S),
        "i"(B + 5 * S), "i"(B + 6 * S), "i"(B + 7 * S));
}

// The V fragments of one key block, vf[2 i + s] = 32-dim tile i, 16-key step s
// (bytes 2048 i + 512 s from the lane's piece).
template <int B, int N>
__device__ __forceinline__ void read_values(uint32_t addr, bf16x8 (&vf)[N]) {
  static_assert(N == 4 || N == 6 || N == 8, "two to four 32-dim tiles");
  if constexpr (N == 4)
    asm volatile(
        "ds_read_b128 %0, %4 offset:%5\n\tds_read_b128 %1, %4 offset:%6\n\t"
        "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %4 offset:%8\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(vf[0]), "=&v"(vf[1]), "=&v"(vf[2]), "=&v"(vf[3])
        : "v"(addr), "i"(B), "i"(B + 512), "i"(B + 2048), "i"(B + 2560));
  else if constexpr (N == 6)
    asm volatile(
        "ds_read_b128 %0, %6 offset:%7\n\tds_read_b128 %1, %6 offset:%8\n\t"
        "ds_read_b128 %2, %6 offset:%9\n\tds_read_b128 %3, %6 offset:%10\n\t"
        "ds_read_b128 %4, %6 offset:%11\n\tds_read_b128 %5, %6 offset:%12\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(vf[0]), "=&v"(vf[1]), "=&v"(vf[2]), "=&v"(vf[3]), "=&v"(vf[4]), "=&v"(vf[5])
        : "v"(addr), "i"(B), "i"(B + 512), "i"(B + 2048), "i"(B + 2560), "i"(B + 4096),
          "i"(B + 4608));
  else
    asm volatile(
        "ds_read_b128 %0, %8 offset:%9\n\tds_read_b128 %1, %8 offset:%10\n\t"
        "ds_read_b128 %2, %8 offset:%11\n\tds_read_b128 %3, %8 offset:%12\n\t"
        "ds_read_b128 %4, %8 offset:%13\n\tds_read_b128 %5, %8 offset:%14\n\t"
        "ds_read_b128 %6, %8 offset:%15\n\tds_read_b128 %7, %8 offset:%16\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(vf[0]), "=&v"(vf[1]), "=&v"(vf[2]), "=&v"(vf[3]), "=&v"(vf[4]), "=&v"(vf[5]),
          "=&v"(vf[6]), "=&v"(vf[7])
        : "v"(addr), "i"(B), "i"(B + 512), "i"(B + 2048), "i"(B + 2560), "i"(B + 4096),
          "i"(B + 4608), "i"(B + 6144), "i"(B + 6656));
}

template <int D, int HW, int KG>
__global__ __launch_bounds__(256, 2) void attention_tile_kernel(TileArgs a) {
  constexpr int KU = D / 16;                       // 16-wide k steps of a score
  constexpr int DT = D / 32;                       // 32-dim output tiles
  constexpr int kQTiles = 4 / (HW * KG);           // query tiles per workgroup
  constexpr int SB = KG < 2 ? 2 : KG;              // key blocks per stage
  constexpr int kBlockElems = 32 * D;              // one key block of K (or V)
  constexpr int kStageElems = 2 * SB * kBlockElems;  // the K blocks, then the V blocks
  constexpr int kPieces = kStageElems / 512;       // 1 KB copies per stage
  constexpr int kCopies = kPieces / 4;             // per wavefront
  constexpr int NB = 2;                            // stages in LDS, used in turn
  static_assert(kCopies * 4 == kPieces, "whole copies per wavefront");
  static_assert(KG == 1 || KG == 2, "key groups");
  __shared__ __attribute__((aligned(16))) uint16_t stage[NB][kStageElems];
  __shared__ float ml_s[KG > 1 ? 4 - 4 / KG : 1][2][32];

  asm volatile("" ::"s"(a.q), "s"(a.kf), "s"(a.vf), "s"(a.qs[0]), "s"(a.qs[1]), "s"(a.qs[2]),
               "s"(a.seq), "s"(a.heads), "s"(a.kv_heads), "s"(a.window), "s"(a.scale_log2),
               "s"(a.q_sign), "s"(a.out));
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kw = wave % KG;    // key group
  const int slot = wave / KG;  // (query tile, head) of the workgroup
  const int half = lane >> 5, col = lane & 31;
  const int T = a.seq, W = a.window;
  const int rep = a.heads / a.kv_heads;
  // blockIdx.x = (batch, kv head, head group): consecutive ids, so the
  // workgroups of a kv head share an XCD's L2 when there are eight of them
  // or a multiple; blockIdx.y walks the query tiles from the last (longest).
  const int hgroups = rep / HW;
  const int bh = blockIdx.x / hgroups;
  const int b = bh / a.kv_heads, kvh = bh - b * a.kv_heads;
  const int h = kvh * rep + (blockIdx.x - bh * hgroups) * HW + slot % HW;
  const int wg0 = static_cast<int>(gridDim.y - 1 - blockIdx.y) * (kQTiles * 32);
  const int q0 = wg0 + (slot / HW) * 32;  // this wavefront's first query
  const int nblk = (T + 31) / 32;

  // Key blocks any query of the workgroup sees: from block lo to the last
  // query's.
  const int lo = max(0, wg0 - W + 1) / 32;
  const int stages = ((min(wg0 + kQTiles * 32, T) - 1) / 32 - lo) / SB + 1;
  const int q_last = min(q0 + 32, T) - 1;  // < q0: this wavefront has no rows

  const __amdgpu_buffer_rsrc_t k_rsrc =
      make_rsrc(a.kf + static_cast<int64_t>(bh) * nblk * kBlockElems,
                static_cast<uint32_t>(nblk) * kBlockElems * 2);
  const __amdgpu_buffer_rsrc_t v_rsrc =
      make_rsrc(a.vf + static_cast<int64_t>(bh) * nblk * kBlockElems,
                static_cast<uint32_t>(nblk) * kBlockElems * 2);
  // One stage: SB key blocks of K then of V, 1 KB per wavefront copy.  The
  // second block of an odd last pair is the first once more (no query sees it):
  // the scalar offset that says which block is read lies inside the buffer.
  auto issue = [&](int st, int buf) {
    const int first = lo + st * SB;
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      const int piece = i * 4 + wave;
      const bool is_v = piece >= kPieces / 2;
      buffer_to_lds16(is_v ? v_rsrc : k_rsrc, &stage[buf][piece * 512], lane * 16u,
                      stage_piece_offset(first, is_v ? piece - kPieces / 2 : piece,
                                         kPieces / (2 * SB), nblk));
    }
  };
  issue(0, 0);

  // Q^T as the B operand: lane holds query q0 + col, dims 16 u + 8 half .. + 7.
  bf16x8 qf[KU];
  {
    const uint16_t* row = a.q + b * a.qs[0] + h * a.qs[1] +
                          static_cast<int64_t>(min(q0 + col, T - 1)) * a.qs[2] + 8 * half;
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      uint4 v = *reinterpret_cast<const uint4*>(row + 16 * u);
      v.x ^= a.q_sign;
      v.y ^= a.q_sign;
      v.z ^= a.q_sign;
      v.w ^= a.q_sign;
      qf[u] = __builtin_bit_cast(bf16x8, v);
    }
  }

  // Byte offsets within a block: K row `col` is key 16 j + 4 (2 s + h) + r
  // for col = 16 s + 8 j + 4 h + r; V piece of (16-dim half, group g).
  const int kn = (col >> 3) & 1;
  const int kc = 4 * (2 * (col >> 4) + ((col >> 2) & 1)) + (col & 3);
  const uint32_t k_off =
      static_cast<uint32_t>(kn * (D / 32) * 1024 + half * 256 + kc * 16);
  const uint32_t v_off =
      static_cast<uint32_t>(SB * kBlockElems * 2 + (col >> 4) * 1024 + half * 256 + (col & 15) * 16);

  // The first block in which this lane's query sees a key.  Blocks before it,
  // which other queries of the tile do see, have weight 0 for this one, but 0
  // times an infinite value is not: its sums start from 0 at that block, in
  // `raise`, where m = -inf leaves nothing to scale (a check after every block
  // cost 2-4 %).
  const int first_seen = max(0, q0 + col - W + 1) & ~31;

  // Running maximum m (log2 units) per query, shared by its two lanes and
  // raised only when a score passes it by more than 2^8; each lane sums its
  // own probabilities (see attention.hip).
  constexpr float kLazy = 8.0f;
  float m = -INFINITY, l = 0.0f;
  f32x16 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[i][e] = 0.0f;

  auto scores = [&](const bf16x8 (&kf)[KU]) {
    f32x16 sc;
#pragma unroll
    for (int e = 0; e < 16; ++e) sc[e] = 0.0f;
#pragma unroll
    for (int u = 0; u < KU; ++u)
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[u], qf[u], sc, 0, 0, 0);
    return sc;
  };
  auto mask = [&](f32x16& sc, int k0) {
    // A block that every query of the tile sees whole needs no mask.
    if (k0 + 31 <= q0 && k0 > q_last - W && k0 + 32 <= T) return;
    const int query = q0 + col;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int key = k0 + 16 * ((e >> 2) & 1) + 4 * (2 * (e >> 3) + half) + (e & 3);
      const bool ok = key <= query && key > query - W && key < T;
      sc[e] = ok ? sc[e] : -INFINITY;
    }
  };
  auto max16 = [&](const f32x16& x) {
    float t[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) t[i] = fmaxf(fmaxf(x[3 * i], x[3 * i + 1]), x[3 * i + 2]);
    return fmaxf(fmaxf(fmaxf(t[0], t[1]), t[2]), fmaxf(fmaxf(t[3], t[4]), x[15]));
  };
  auto raise = [&](float mx, int k0) {  // mx: this lane's largest score
    mx *= a.scale_log2;
    if (__ballot(mx > m + kLazy) != 0) {
      const float mn = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32)));
      const float alpha = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
      l *= alpha;
      if (static_cast<uint32_t>(k0 - first_seen) < 32u * KG) {  // the key group's first such block
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[i][e] = 0.0f;
      }
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= alpha;
      m = mn;
    }
  };
  // P of the block as two bf16 parts (see the top): cut off, not rounded, and the
  // rest raised by 2^-20 P, because a rest of 0 or below would make NaN of an
  // infinite value.
  constexpr float kRaise = 1.0f + 0x1p-20f;
  auto probabilities = [&](const f32x16& sc, bf16x8 (&pf)[2], bf16x8 (&rest)[2]) {
    // A query that has seen no key yet has m = -inf and only -inf scores:
    // exp2(-inf - 0) = 0.
    const float neg = m == -INFINITY ? 0.0f : -m;
    float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      uint32_t high[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t bits[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int e = 2 * i + k;
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[8 * s + e], a.scale_log2, neg));
          sum[e & 3] += p;
          bits[k] = __float_as_uint(p);
          rest[s][e] = static_cast<__bf16>(
              __builtin_fmaf(p, kRaise, -__uint_as_float(bits[k] & 0xffff0000u)));
        }
        high[i] = __builtin_amdgcn_perm(bits[1], bits[0], 0x07060302u);  // the upper halves
      }
      pf[s] = __builtin_bit_cast(bf16x8, make_uint4(high[0], high[1], high[2], high[3]));
    }
    l += (sum[0] + sum[1]) + (sum[2] + sum[3]);
  };
  auto values = [&](bf16x8 (&vf)[2 * DT], const bf16x8 (&pf)[2], const bf16x8 (&rest)[2], int k0) {
    // Keys past the sequence: their P is 0, but the padding bytes need not
    // be finite.
    if (k0 + 32 > T) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int key = k0 + 16 * (e >> 2) + 4 * (2 * s + half) + (e & 3);
            if (key >= T) vf[2 * i + s][e] = static_cast<__bf16>(0.0f);
          }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < DT; ++i)
        o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[2 * i + s], pf[s], o[i], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < DT; ++i)
        o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[2 * i + s], rest[s], o[i], 0, 0, 0);
  };
  constexpr int kNext = kBlockElems * 2;  // bytes from one block to the next
  auto block = [&](uint32_t lds, int k0) {
    bf16x8 kf[KU], vf[2 * DT], pf[2], rest[2];
    lds_frags<0, 512>(lds + k_off, kf);
    f32x16 sc = scores(kf);
    __builtin_amdgcn_sched_barrier(0);
    read_values<0>(lds + v_off, vf);
    mask(sc, k0);
    raise(max16(sc), k0);
    probabilities(sc, pf, rest);
    values(vf, pf, rest, k0);
  };

  const uint32_t lds0 = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint16_t*)&stage[0][0]));
  int buf = 0;
  for (int st = 0; st < stages; ++st) {
    // This wavefront's copies of stage st, the only ones in flight, have
    // landed; past the barrier everybody's have, and nobody reads the buffer
    // of stage st - 1 any more.
    wait_vm_barrier<0>();
    if (st + 1 < stages) issue(st + 1, buf ^ 1);
    // Blocks past this wavefront's diagonal or before its window are left out.
    const uint32_t lds = lds0 + buf * (kStageElems * 2);
    const int k0 = (lo + st * SB) * 32;
    auto seen = [&](int k) { return k <= q_last && k + 31 > q0 - W; };
#pragma unroll
    for (int j = kw; j < SB; j += KG)
      if (seen(k0 + 32 * j)) block(lds + j * kNext, k0 + 32 * j);
    buf ^= 1;
  }
  l += __shfl_xor(l, 32);

  // The other key groups hand their states to group 0 through the stage
  // buffers; it adds them in group order.
  if constexpr (KG > 1) {
    constexpr int kState = DT * 16 * kWave;  // floats per wavefront
    static_assert((4 - 4 / KG) * kState * 4 <= NB * kStageElems * 2, "the merge fits the stages");
    float* ob = reinterpret_cast<float*>(&stage[0][0]);
    const int diag = q0 >> 5;
    if ((diag - ((diag - lo - kw) & (KG - 1))) * 32 < first_seen) {  // this key group had none
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] = 0.0f;
    }
    __syncthreads();  // everybody has read the last stage
    if (kw > 0) {
      const int at = slot * (KG - 1) + kw - 1;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) ob[at * kState + (i * 16 + e) * kWave + lane] = o[i][e];
      if (half == 0) {
        ml_s[at][0][col] = m;
        ml_s[at][1][col] = l;
      }
    }
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int g = 1; g < KG; ++g) {
      const int at = slot * (KG - 1) + g - 1;
      const float m1 = ml_s[at][0][col], l1 = ml_s[at][1][col];
      const float mn = fmaxf(m, m1);
      const float f0 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
      const float f1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mn);
      l = l * f0 + l1 * f1;
      m = mn;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          o[i][e] = o[i][e] * f0 + ob[at * kState + (i * 16 + e) * kWave + lane] * f1;
    }
  }
  // C fragment: lane holds query col, dims 32 i + 8 j + 4 half + r.
  const int query = q0 + col;
  if (query >= T) return;
  const float inv = 1.0f / l;
  uint16_t* row = a.out + ((static_cast<int64_t>(b) * T + query) * a.heads + h) * D + 4 * half;
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint2 w;
      w.x = pack_bf16x2(o[i][4 * j] * inv, o[i][4 * j + 1] * inv);
      w.y = pack_bf16x2(o[i][4 * j + 2] * inv, o[i][4 * j + 3] * inv);
      *reinterpret_cast<uint2*>(row + 32 * i + 8 * j) = w;
    }
}

template <int D, int HW, int KG>
hipError_t launch_tile(const TileArgs& a, int batch, hipStream_t s) {
  constexpr int kRows = 4 / (HW * KG) * 32;
  const dim3 grid(batch * a.kv_heads * (a.heads / a.kv_heads / HW), (a.seq + kRows - 1) / kRows);
  attention_tile_kernel<D, HW, KG><<<grid, 256, 0, s>>>(a);
  return hipGetLastError();
}

// KG = 1 from three workgroups per CU: at 768 tiles (3 x 4096 tokens with 8
// heads) 92 against 94 us, at 512 (2 x 4096) 74 against 68.
constexpr int64_t kOneGroupTiles = 768;

template <int D>
hipError_t launch_tile_heads(const TileArgs& a, int batch, hipStream_t s) {
  const int rep = a.heads / a.kv_heads;
  const int64_t tiles = static_cast<int64_t>(batch) * a.heads * ((a.seq + 127) / 128);
  if (tiles >= kOneGroupTiles) {
    if (rep % 4 == 0) return launch_tile<D, 4, 1>(a, batch, s);
    if (rep % 2 == 0) return launch_tile<D, 2, 1>(a, batch, s);
    return launch_tile<D, 1, 1>(a, batch, s);
  }
  if (rep % 2 == 0) return launch_tile<D, 2, 2>(a, batch, s);
  return launch_tile<D, 1, 2>(a, batch, s);
}

}  // namespace

// From where causal_attention_kernel's grid (16 queries of a head per
// workgroup, two workgroups resident per CU) no longer starts at once, and its
// rounds take longer than the serial chain over a query's keys takes here
// (about 12 us per 1000 keys and 5 to start): the more sequences and heads share
// the grid, the sooner.  Measured, that kernel / this (us): 16 heads in all, 528
// workgroups, 520 keys 13.7 / 11.9; 12, 600, 800 keys 15.7 / 14.8; 8, 632, 1250
// keys 19.3 / 19.9, 728, 1450 keys 21.8 / 22.1, 800, 1600 keys 24.9 / 23.9; 4,
// 800, 2048 keys 29.9 / 30.4, 900, 2048 keys 33.9 / 30.5, 900, 3600 keys 43.4 /
// 48.0, 1024, 4096 keys 50.6 / 53.9.  At head width 64 the other kernel's rounds
// are shorter: 8, 728, 1450 keys 16.6 / 18.9, 904, 1800 keys 21.5 / 23.0; 16, 528,
// 520 keys 10.9 / 10.1.
//
// One kv head's fragments must be addressable from every stage's base, the query
// tiles (32 queries at the least) must fit the grid's y, the output takes 8-byte
// stores, and a zero scale is left out (scores are masked before they are scaled
// here).
bool attention_tiles_apply(int batch, int seq, int heads, int head_dim, int window, float scale,
                           const uint16_t* out) {
  const int64_t groups = static_cast<int64_t>(batch) * heads * ((seq + 15) / 16);
  const int keys = min(min(seq, window), 3072);
  const int line = max(512, head_dim == 64 ? 344 + keys / 3 : 384 + keys / 4);
  return scale != 0.0f && groups > line && groups < (int64_t{1} << 31) && seq <= 65535 * 32 &&
         (static_cast<int64_t>(seq) + 256) * head_dim * 2 < (int64_t{1} << 31) &&
         (reinterpret_cast<uintptr_t>(out) & 7u) == 0;
}

hipError_t launch_attention_tiles(const uint16_t* q, const uint16_t* k_frag,
                                  const uint16_t* v_frag, const int64_t* q_strides, int batch,
                                  int seq, int heads, int kv_heads, int head_dim, int window,
                                  float scale, uint16_t* out, hipStream_t s) {
  if (batch == 0 || seq == 0) return hipSuccess;
  TileArgs a{};
  a.q = q;
  a.kf = k_frag;
  a.vf = v_frag;
  for (int i = 0; i < 3; ++i) a.qs[i] = q_strides[i];
  a.seq = seq;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.window = window;
  a.scale_log2 = (scale < 0 ? -scale : scale) * 1.4426950408889634f;
  a.q_sign = scale < 0 ? 0x80008000u : 0u;
  a.out = out;
  switch (head_dim) {
    case 64: return launch_tile_heads<64>(a, batch, s);
    case 96: return launch_tile_heads<96>(a, batch, s);
    case 128: return launch_tile_heads<128>(a, batch, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace parrot
