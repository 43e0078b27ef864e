// Dense projections y = x W^T on v_mfma_f32_16x16x32_bf16: the linear maps of
// the attention layers (packed q|k|v, output, MLA latent and up maps).
//
// Reference semantics: bias-free nn.Linear in bf16 (parrot/model.py:167-230
// for the GQA layers, :331-432 for MLA), the output projection with its
// residual add as the reference's decode kernel computes it,
// bf16(addend + bf16(x W^T)) (parrot/kernels/moe_bf16.metal:1364-1389), and
// for the GQA layers RoPE of q and k plus the head split
// (parrot/model.py:176-230), applied here to the bf16-rounded projection
// exactly as the stand-alone RoPE kernel does.
//
// At prefill sizes (hundreds of rows, K <= 2048, a few MB of weights) a
// library GEMM spends most of its time in a k loop of global -> LDS -> MFMA
// round trips.  Here a workgroup owns 16 rows x 64 columns: the whole A tile
// (16 x K) is copied into LDS once with direct-to-LDS loads, XOR-swizzled as
// in the expert GEMMs, and each of the 4 wavefronts streams the B fragments
// of its 16 columns straight into registers with raw buffer loads from
// weights packed in MFMA fragment order (1 KB contiguous per wavefront
// load): for K = 32 KST with KST in {4, 8, 16, 24} every k step is loaded
// up front (the trip count is a template constant, so the compiler places
// exact per-step waits), for other K through a ring of PF registers.  The A
// loads are issued first and waited for alone (vmcnt(PF)), and the A
// fragments are read from LDS with inline asm so the compiler does not add
// a wait for the whole direct-to-LDS traffic; the k loop has no barrier.
// Measured on MI355X in the bs1 x 512 forward: 16-row tiles beat 32-row
// tiles (more workgroups in flight), and the up-front loads beat the ring.
//
// Workgroups are dispatched round-robin over the 8 XCDs; the tile index is
// remapped so each XCD takes a contiguous run of column-major tiles, and the
// row tiles that share a block of weight columns share that XCD's L2.
//
// Epilogues (the C fragment gives lane l column l % 16 and rows
// 4 (l / 16) + r):
//   kStore    out[row, col] = bf16(acc) or bf16(addend + bf16(acc));
//   kStoreT   per-sequence transpose, out[(b N + col) ld_keys + t], the value
//             layout the attention kernel reads (MLA values);
//   kRopeQkv  columns [0, H d) -> q [b, H, seq, d], [H d, (H + Hk) d) ->
//             k [b, Hk, seq, d], both rotated; the rest -> v, [b, Hk, seq, d]
//             or transposed [b, Hk, d, vt_keys]; and/or k and v in the
//             attention kernel's fragment order (kfrag_index, vfrag_index).
//             Rotation partners (2i, 2i + 1) sit in adjacent lanes: one DPP
//             quad_perm swap.
//   kFrag     the output as attention K or V in fragment order, columns
//             grouped into heads of head_dim, or both from one [Wk; Wv]
//             weight (the MLA up-projections).
#include "common.h"
#include "extents.h"

#include <type_traits>

namespace parrot {

namespace {

constexpr int kProjRows = 16;        // rows per workgroup
constexpr int kProjCols = 64;        // columns per workgroup: 4 wavefronts x 16
constexpr int kProjMaxK = 2048;      // A tile at most 64 KB of LDS

enum ProjEpilogue { kStore = 0, kStoreT = 1, kRopeQkv = 2, kFrag = 3 };

struct ProjArgs {
  const uint16_t* x;
  int64_t lda;
  int rows, K, N;
  const uint16_t* w;       // packed [N / 16][K / 32][64 lanes x 16 B]
  // kStore
  uint16_t* out;
  int64_t ldo;
  const uint16_t* addend;  // optional, [rows, ld_addend]
  int64_t ld_addend;
  // kStoreT and kRopeQkv
  int seq, ld_keys;
  // kRopeQkv
  const float* cos_t;
  const float* sin_t;
  int start, max_positions;
  const int32_t* start_device;
  int heads, kv_heads, head_dim;
  uint16_t* q;
  uint16_t* k;              // optional with kRopeQkv
  uint16_t* v;              // optional with kRopeQkv
  // fragment-order attention operands (kRopeQkv: optional; kFrag: one of them)
  uint16_t* kf;
  uint16_t* vf;
  int nblk;                 // ceil(seq / 32)
};

__device__ __forceinline__ float swap_pair(float v) {  // lanes 2i <-> 2i + 1
  return dpp<0xb1>(v);
}

// One 16-byte MFMA fragment from LDS, read with inline asm: the compiler then
// does not tie it to the direct-to-LDS loads (it would wait for every one of
// them, vmcnt(0), weight loads included); the kernel's own vmcnt wait and
// barrier order it after the A tile, and lds_frag_wait before its use.
__device__ __forceinline__ bf16x8 lds_frag(const uint16_t* p) {
  const uint32_t addr = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint16_t*)p));
  bf16x8 v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}

// Stores one lane's 4 values (rows row0 .. row0 + 3, one column w of kv
// head kvh of kv_heads) as attention values: row-major p.v [b, kv_heads,
// seq, d] or transposed [b, kv_heads, d, ld_keys] when p.v is set, and in
// fragment order when p.vf is set.  When seq % 4 == 0 the 4 rows are
// consecutive positions of one sequence and the transposed and fragment
// stores take them in one 8-byte store.
__device__ __forceinline__ void store_values(const ProjArgs& p, const uint16_t (&bits)[4],
                                             int row0, int kvh, int kv_heads, int w) {
  const int d = p.head_dim;
  if ((p.seq & 3) == 0) {
    const int b = row0 / p.seq;
    const int t0 = row0 - b * p.seq;
    const int64_t bh = static_cast<int64_t>(b) * kv_heads + kvh;
    uint2 u;
    u.x = static_cast<uint32_t>(bits[0]) | (static_cast<uint32_t>(bits[1]) << 16);
    u.y = static_cast<uint32_t>(bits[2]) | (static_cast<uint32_t>(bits[3]) << 16);
    if (p.v != nullptr) {
      if (p.ld_keys > 0) {
        *reinterpret_cast<uint2*>(p.v + (bh * d + w) * p.ld_keys + t0) = u;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) p.v[(bh * p.seq + t0 + r) * d + w] = bits[r];
      }
    }
    if (p.vf != nullptr)
      *reinterpret_cast<uint2*>(p.vf + vfrag_index(bh, p.nblk, t0, w, d / 16)) = u;
    return;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = row0 + r;
    if (row >= p.rows) break;
    const int b = row / p.seq;
    const int tp = row - b * p.seq;
    const int64_t bh = static_cast<int64_t>(b) * kv_heads + kvh;
    if (p.v != nullptr) {
      if (p.ld_keys > 0) p.v[(bh * d + w) * p.ld_keys + tp] = bits[r];
      else p.v[(bh * p.seq + tp) * d + w] = bits[r];
    }
    if (p.vf != nullptr) p.vf[vfrag_index(bh, p.nblk, tp, w, d / 16)] = bits[r];
  }
}

// KST > 0: K == 32 KST and PF == KST (every k step loaded up front);
// KST == 0: a ring of PF stages over K / 32 steps (a multiple of PF).
template <int PF, int EPI, int KST>
__global__ __launch_bounds__(256) void proj_kernel(ProjArgs p) {
  constexpr int BM = kProjRows;
  constexpr int kTilesM = BM / 16;
  static_assert(KST == 0 || KST == PF, "the up-front mode loads every step at once");
  extern __shared__ __attribute__((aligned(16))) uint16_t a_lds[];  // [BM][K], swizzled

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // XCD-aware tile order: hardware id -> (XCD, slot) -> contiguous index j.
  const int total = static_cast<int>(gridDim.x);
  // The prologue's kernel arguments in one batch of scalar loads (a field
  // first read inside a branch or loop costs a scalar round trip of its own).
  asm volatile("" ::"s"(p.x), "s"(p.lda), "s"(p.rows), "s"(p.K), "s"(p.N), "s"(p.w), "s"(total));
  if constexpr (EPI == kStore) asm volatile("" ::"s"(p.addend), "s"(p.ld_addend));
  if constexpr (EPI == kRopeQkv)
    asm volatile("" ::"s"(p.cos_t), "s"(p.sin_t), "s"(p.start), "s"(p.start_device), "s"(p.seq),
                 "s"(p.max_positions), "s"(p.head_dim), "s"(p.heads), "s"(p.kv_heads));
  const int id = static_cast<int>(blockIdx.x);
  const int xcd = id & 7, slot = id >> 3;
  const int q8 = total >> 3, r8 = total & 7;
  const int j = xcd * q8 + min(xcd, r8) + slot;
  const int row_tiles = (p.rows + BM - 1) / BM;
  const int ct = j / row_tiles;
  const int m0 = (j - ct * row_tiles) * BM;
  const int nw = ct * kProjCols + wave * 16;  // this wavefront's first column

  const int K = p.K;
  const int chunks = K / 8;                      // 16-byte chunks per row (multiple of 8)
  const int swz = (chunks & 15) == 0 ? 15 : 7;   // XOR group size - 1
  const int ksteps = KST > 0 ? KST : K / 32;

  // ---- epilogue operands that depend only on this lane's rows and column,
  // loaded before the tile so their round trip overlaps it: read in the
  // epilogue they added one (the residual addend) or two (a device position,
  // then the RoPE tables).  The loads are unconditional (a value loaded
  // inside a branch is waited for at the branch's end): without an addend
  // they read the weights' first row, waves past N clamp their column, and
  // the table indices are clamped into the tables.
  const int ecol = min(nw, p.N - 16) + (lane & 15);
  uint16_t add_v[kTilesM][4];
  float rope_c[kTilesM][4], rope_s[kTilesM][4];
  if constexpr (EPI == kStore) {
    const bool has_addend = p.addend != nullptr;
    const uint16_t* ab = has_addend ? p.addend : p.w;
    const int64_t ald = has_addend ? p.ld_addend : 0;
#pragma unroll
    for (int mi = 0; mi < kTilesM; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = min(m0 + mi * 16 + 4 * (lane >> 4) + r, p.rows - 1);
        add_v[mi][r] = ab[static_cast<int64_t>(row) * ald + ecol];
      }
  }
  if constexpr (EPI == kRopeQkv) {
    const int d = p.head_dim;
    const int w = ecol - (ecol / d) * d;
    const int shift = p.start + (p.start_device != nullptr ? *p.start_device : 0);
#pragma unroll
    for (int mi = 0; mi < kTilesM; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = min(m0 + mi * 16 + 4 * (lane >> 4) + r, p.rows - 1);
        const int tp = row - (row / p.seq) * p.seq;
        const int pos = min(max(shift + tp, 0), p.max_positions - 1);
        const int64_t ti = static_cast<int64_t>(pos) * (d / 2) + w / 2;
        rope_c[mi][r] = p.cos_t[ti];
        rope_s[mi][r] = p.sin_t[ti];
      }
  }

  // ---- A: the whole tile, direct to LDS (rows past the end read the last
  // row).  Buffer loads, not global_load_lds: after a global_load_lds the
  // compiler cannot see that the wait below covered it and turns its own
  // wait for the first weight fragment into vmcnt(0), so no MFMA would start
  // before every weight load of the ring had landed.
  {
    const int tile_rows = min(BM, p.rows - m0);
    const __amdgpu_buffer_rsrc_t x_rsrc =
        make_rsrc(p.x + static_cast<int64_t>(m0) * p.lda,
                  static_cast<uint32_t>(static_cast<int64_t>(tile_rows) * p.lda * 2));
    const int slots = BM * chunks;  // multiple of 64
    for (int i = wave; i < slots / kWave; i += 4) {
      const int s = i * kWave + lane;
      const int r = s / chunks;
      const int pc = s - r * chunks;
      const int c = (pc & ~swz) | ((pc ^ r) & swz);
      const uint32_t off =
          static_cast<uint32_t>((static_cast<int64_t>(min(r, tile_rows - 1)) * p.lda + c * 8) * 2);
      buffer_to_lds16(x_rsrc, a_lds + i * kWave * 8, off, 0);
    }
  }

  asm volatile("" ::: "memory");  // every A load is issued before any B load

  // ---- B: first PF k steps of this lane's fragments (columns past N read 0)
  const __amdgpu_buffer_rsrc_t b_rsrc =
      make_rsrc(p.w, static_cast<uint32_t>(static_cast<int64_t>(p.N) * K * 2));
  const uint32_t b_off = static_cast<uint32_t>((nw / 16) * ksteps * 64 + lane) * 16;
  uint4 bq[PF];
#pragma unroll
  for (int i = 0; i < PF; ++i) bq[i] = buffer_load16(b_rsrc, b_off, static_cast<uint32_t>(i) * 1024);

  // The A tile is complete when at most the PF weight loads issued after it
  // are still in flight.
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(PF) : "memory");

  f32x4 acc[kTilesM];
#pragma unroll
  for (int i = 0; i < kTilesM; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int s0 = 0; s0 < ksteps; s0 += PF) {  // ksteps is a multiple of PF
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int step = s0 + i;
      bf16x8 af[kTilesM];
#pragma unroll
      for (int mi = 0; mi < kTilesM; ++mi) {
        const int r = mi * 16 + (lane & 15);
        const int c = step * 4 + (lane >> 4);
        const int pc = (c & ~swz) | ((c ^ r) & swz);
        af[mi] = lds_frag(&a_lds[(r * chunks + pc) * 8]);
      }
      asm volatile("s_waitcnt lgkmcnt(0)");
#pragma unroll
      for (int mi = 0; mi < kTilesM; ++mi) asm volatile("" : "+v"(af[mi]));
#pragma unroll
      for (int mi = 0; mi < kTilesM; ++mi)
        acc[mi] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            af[mi], __builtin_bit_cast(bf16x8, bq[i]), acc[mi], 0, 0, 0);
      if (step + PF < ksteps)
        bq[i] = buffer_load16(b_rsrc, b_off, static_cast<uint32_t>(step + PF) * 1024);
    }
  }

  // ---- epilogue --------------------------------------------------------------
  const int col = nw + (lane & 15);
  if (nw >= p.N) return;  // whole wavefront past the last column (N % 16 == 0)

  if (EPI == kStore) {
#pragma unroll
    for (int mi = 0; mi < kTilesM; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + mi * 16 + 4 * (lane >> 4) + r;
        if (row >= p.rows) continue;
        uint16_t v = f32_to_bf16(acc[mi][r]);
        if (p.addend != nullptr) v = f32_to_bf16(bf16_to_f32(add_v[mi][r]) + bf16_to_f32(v));
        p.out[static_cast<int64_t>(row) * p.ldo + col] = v;
      }
    return;
  }

  if (EPI == kStoreT) {
    // rows 4 (l / 16) .. + 3 of a lane are consecutive positions of one
    // sequence when seq % 4 == 0: one 8-byte store.
#pragma unroll
    for (int mi = 0; mi < kTilesM; ++mi) {
      const int row0 = m0 + mi * 16 + 4 * (lane >> 4);
      if (row0 >= p.rows) continue;
      const int b = row0 / p.seq;
      const int t0 = row0 - b * p.seq;
      uint16_t* dst = p.out + (static_cast<int64_t>(b) * p.N + col) * p.ld_keys;
      if ((p.seq & 3) == 0) {
        uint2 w;
        w.x = pack_bf16x2(acc[mi][0], acc[mi][1]);
        w.y = pack_bf16x2(acc[mi][2], acc[mi][3]);
        *reinterpret_cast<uint2*>(dst + t0) = w;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = row0 + r;
          if (row >= p.rows) break;
          const int bb = row / p.seq;
          p.out[(static_cast<int64_t>(bb) * p.N + col) * p.ld_keys + (row - bb * p.seq)] =
              f32_to_bf16(acc[mi][r]);
        }
      }
    }
    return;
  }

  if (EPI == kFrag) {
    // With both outputs, columns [0, N / 2) are K and [N / 2, N) are V
    // (N / 2 is a multiple of 16: one side per wavefront).
    const int d = p.head_dim;
    const bool both = p.kf != nullptr && p.vf != nullptr;
    const int half = both ? p.N / 2 : p.N;
    const bool to_v = p.kf == nullptr || (both && nw >= half);
    const int c2 = both && to_v ? col - half : col;
    const int head = c2 / d;
    const int w = c2 - head * d;
    const int heads = half / d;
#pragma unroll
    for (int mi = 0; mi < kTilesM; ++mi) {
      const int row0 = m0 + mi * 16 + 4 * (lane >> 4);
      if (row0 >= p.rows) continue;
      uint16_t bits[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) bits[r] = f32_to_bf16(acc[mi][r]);
      if (!to_v) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = row0 + r;
          if (row >= p.rows) break;
          const int b = row / p.seq;
          p.kf[kfrag_index(static_cast<int64_t>(b) * heads + head, p.nblk, row - b * p.seq, w,
                           d / 32)] = bits[r];
        }
      } else {
        store_values(p, bits, row0, head, heads, w);
      }
    }
    return;
  }

  // kRopeQkv
  const int d = p.head_dim;
  const int head = col / d;  // per lane; a rotation pair never straddles heads (d even)
  const int w = col - head * d;
  const int H = p.heads, Hk = p.kv_heads;
  const bool rotate = head < H + Hk;
  const bool odd = (lane & 1) != 0;
#pragma unroll
  for (int mi = 0; mi < kTilesM; ++mi) {
    float val[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // round as the projection output, then rotate (identical to the
      // stand-alone kernel applied to the stored projection)
      const float self = bf16_to_f32(f32_to_bf16(acc[mi][r]));
      const float other = swap_pair(self);
      val[r] = self;
      if (rotate) {
        const float c = rope_c[mi][r], s = rope_s[mi][r];
        val[r] = odd ? rope_odd(other, self, c, s) : rope_even(self, other, c, s);
      }
    }
    const int row0 = m0 + mi * 16 + 4 * (lane >> 4);
    if (row0 >= p.rows) continue;
    uint16_t bits[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) bits[r] = f32_to_bf16(val[r]);
    if (head < H) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + r;
        if (row >= p.rows) break;
        const int b = row / p.seq;
        const int tp = row - b * p.seq;
        p.q[((static_cast<int64_t>(b) * H + head) * p.seq + tp) * d + w] = bits[r];
      }
    } else if (head < H + Hk) {
      const int kvh = head - H;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + r;
        if (row >= p.rows) break;
        const int b = row / p.seq;
        const int tp = row - b * p.seq;
        if (p.k != nullptr) p.k[((static_cast<int64_t>(b) * Hk + kvh) * p.seq + tp) * d + w] = bits[r];
        if (p.kf != nullptr)
          p.kf[kfrag_index(static_cast<int64_t>(b) * Hk + kvh, p.nblk, tp, w, d / 32)] = bits[r];
      }
    } else {
      store_values(p, bits, row0, head - H - Hk, Hk, w);
    }
  }
}

// ---------------------------------------------------------------------------
// Many rows: BM = 32 or 64 rows per workgroup, all of its columns streamed.
//
// With 16-row tiles every workgroup pulls its 64 columns' weights (96 KB at
// K = 768) through L2 for 16 rows: at 16384 rows the q|k|v projection moved
// 2.3 GB of them and took 128 us, four times its matrix products at the rate
// of a large library GEMM.  Here the A tile (BM x K, in LDS as above) stays
// while the wavefronts walk the columns in blocks of 48, each streaming its
// block's B fragments into a ring of PF register stages that runs on into
// the wavefront's next block, so the k loop has no barrier and no bubble
// between blocks; a fragment loaded feeds BM / 16 products.  Measured on
// MI355X (us, before / now): q|k|v + RoPE with caches 16384 rows 128 / 52
// (560 TFLOP/s), 4094 rows 36 / 20, 1 x 1024 11.4 / 10.0; output projection
// with addend 72 / 34, 20 / 12.6; latent q 79 / 34, 23 / 13.5; latent k, v
// 49 / 22, 15.3 / 9.5.  At 16384 rows each CU runs one workgroup, so its A
// load, products and stores follow each other; that and the 2-byte stores of
// row-major values are what is left.
//
// The accumulation per output is proj_kernel's (one chain of 16x16x32 MFMAs
// in k order), so both give the same bits.  Except for attention values the
// weights are the A operand: lane l then holds row l % 16 of a row tile and
// four consecutive columns, so RoPE's pairs sit in one lane and every store
// is 8 bytes.  Values keep x as the A operand (four consecutive positions of
// one column, what the fragment order wants).  RoPE's cos / sin rows are
// staged in LDS once for all heads.
constexpr int kBlockGroups = 3;             // 16-column groups per block
constexpr int kBlockCols = 16 * kBlockGroups;

// The columns as blocks: [0, n_swap) with the weights as the A operand, then
// [n_swap, N) with x (no block holds both).
struct ColumnBlocks {
  int n_swap, first, total;  // first: blocks of [0, n_swap)
};

__device__ __forceinline__ ColumnBlocks column_blocks(int n_swap, int N) {
  const int first = (n_swap + kBlockCols - 1) / kBlockCols;
  return ColumnBlocks{n_swap, first, first + (N - n_swap + kBlockCols - 1) / kBlockCols};
}

// One workgroup per CU (98 KB of A at BM = 64; two wavefronts per SIMD).
template <int BM, int NW, int KST, int EPI>
__global__ __launch_bounds__(64 * NW, 2) void proj_rows_kernel(ProjArgs p, int splits) {
  constexpr int kTilesM = BM / 16;
  constexpr int K = 32 * KST;
  constexpr int kChunks = K / 8;       // 16-byte chunks per row (a multiple of 16)
  constexpr int PF = 4;
  static_assert(KST % PF == 0 && kChunks % 16 == 0, "whole rings, 16-chunk swizzle");
  __shared__ __attribute__((aligned(16))) uint16_t a_s[BM * K];
  // (cos, sin) of the tile's rows, d / 2 pairs each (d <= 128)
  __shared__ __attribute__((aligned(16))) float2 rope_s[EPI == kRopeQkv ? BM * 64 : 1];

  asm volatile("" ::"s"(p.x), "s"(p.lda), "s"(p.rows), "s"(p.N), "s"(p.w), "s"(splits),
               "s"(p.seq), "s"(p.head_dim));
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int row_tile = static_cast<int>(blockIdx.x) / splits;
  const int split = static_cast<int>(blockIdx.x) - row_tile * splits;
  // Outputs laid out per sequence take row tiles of one sequence each, so a
  // tile's positions start at a multiple of 4 whatever the length.
  int b = 0, t0 = row_tile * BM, seq = p.rows;
  if constexpr (EPI != kStore) {
    const int per_seq = (p.seq + BM - 1) / BM;
    b = row_tile / per_seq;
    t0 = (row_tile - b * per_seq) * BM;
    seq = p.seq;
  }
  const int m0 = b * p.seq + t0;  // first row (b is 0 with plain rows)
  const int tile_rows = min(BM, seq - t0);
  const int d = p.head_dim;
  const int n_swap = EPI == kRopeQkv ? (p.heads + p.kv_heads) * d
                     : EPI == kFrag  ? (p.kf == nullptr ? 0 : p.vf == nullptr ? p.N : p.N / 2)
                                     : p.N;
  const ColumnBlocks cb = column_blocks(n_swap, p.N);
  const int blk_end = (split + 1) * cb.total / splits;
  int blk = split * cb.total / splits + wave;

  // ---- A: the whole tile, direct to LDS (rows past the end read the last row)
  {
    const __amdgpu_buffer_rsrc_t x_rsrc =
        make_rsrc(p.x + static_cast<int64_t>(m0) * p.lda,
                  static_cast<uint32_t>(static_cast<int64_t>(tile_rows) * p.lda * 2));
    for (int i = wave; i < BM * kChunks / kWave; i += NW) {
      const int s = i * kWave + lane;
      const int r = s / kChunks;
      const int pc = s - r * kChunks;
      const int ch = (pc & ~15) | ((pc ^ r) & 15);
      const uint32_t off =
          static_cast<uint32_t>((static_cast<int64_t>(min(r, tile_rows - 1)) * p.lda + ch * 8) * 2);
      buffer_to_lds16(x_rsrc, a_s + i * kWave * 8, off, 0);
    }
  }
  if constexpr (EPI == kRopeQkv) {
    const int half = d / 2;
    const int shift = p.start + (p.start_device != nullptr ? *p.start_device : 0);
    for (int i = tid; i < BM * half; i += 64 * NW) {
      const int r = i / half;
      const int pos = min(max(shift + t0 + r, 0), p.max_positions - 1);
      const int64_t at = static_cast<int64_t>(pos) * half + (i - r * half);
      rope_s[i] = make_float2(p.cos_t[at], p.sin_t[at]);
    }
  }

  // Column block b: first column and 16-column groups (uniform).
  auto first_col = [&](int b) {
    return b < cb.first ? b * kBlockCols : cb.n_swap + (b - cb.first) * kBlockCols;
  };
  const __amdgpu_buffer_rsrc_t b_rsrc =
      make_rsrc(p.w, static_cast<uint32_t>(static_cast<int64_t>(p.N) * K * 2));
  uint4 bq[PF][kBlockGroups];
  // Step `step` of the block whose first column is col0 (groups past the last
  // one read it: the scalar offset stays inside the weights, and what comes of
  // them is not stored).
  auto load_step = [&](uint4 (&dst)[kBlockGroups], int col0, int step) {
#pragma unroll
    for (int j = 0; j < kBlockGroups; ++j)
      dst[j] = buffer_load16(b_rsrc, lane * 16u,
                             column_group_offset(col0, j, p.N, KST, step));
  };
  const int col_first = first_col(min(blk, cb.total - 1));
#pragma unroll
  for (int i = 0; i < PF; ++i) load_step(bq[i], col_first, i);

  // A fragment of k step 4 n + q, row tile mi: element a_off[q] + 128 n +
  // 16 K mi (chunk 4 q + g of the row, swizzled within its group of 16).
  int a_off[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) a_off[q] = c * K + ((4 * q + g) ^ c) * 8;

  __syncthreads();
  bf16x8 af[2][kTilesM];
  auto read_a = [&](bf16x8 (&dst)[kTilesM], int q, int step) {  // q = step % 4
#pragma unroll
    for (int mi = 0; mi < kTilesM; ++mi)
      dst[mi] = *reinterpret_cast<const bf16x8*>(a_s + a_off[q] + (step >> 2) * 128 + mi * 16 * K);
  };
  read_a(af[0], 0, 0);

  auto run_block = [&](auto swap_tag, int col0, int next_col0) {
    constexpr bool SWAP = decltype(swap_tag)::value;
    const int n_end = SWAP ? cb.n_swap : p.N;  // stores stop at the range's end
    uint2 add_v[EPI == kStore ? kTilesM : 1][kBlockGroups];
    if constexpr (EPI == kStore) {
      // loaded before the products, unconditionally (see proj_kernel)
      const bool has = p.addend != nullptr;
      const uint16_t* ab = has ? p.addend : p.w;
      const int64_t ald = has ? p.ld_addend : 0;
#pragma unroll
      for (int mi = 0; mi < kTilesM; ++mi)
#pragma unroll
        for (int j = 0; j < kBlockGroups; ++j) {
          const int row = m0 + min(mi * 16 + c, tile_rows - 1);
          const int col = min(col0 + 16 * j, p.N - 16) + 4 * g;
          add_v[mi][j] = *reinterpret_cast<const uint2*>(ab + static_cast<int64_t>(row) * ald + col);
        }
    }
    f32x4 acc[kTilesM][kBlockGroups];
#pragma unroll
    for (int mi = 0; mi < kTilesM; ++mi)
#pragma unroll
      for (int j = 0; j < kBlockGroups; ++j) acc[mi][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1  // the ring's registers are indexed by i alone
    for (int s0 = 0; s0 < KST; s0 += PF) {
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        const int step = s0 + i;
        const int ahead = step + 1 < KST ? step + 1 : 0;  // A fragments, one step ahead
        read_a(af[(i + 1) & 1], (i + 1) & 3, ahead);
#pragma unroll
        for (int mi = 0; mi < kTilesM; ++mi)
#pragma unroll
          for (int j = 0; j < kBlockGroups; ++j) {
            const bf16x8 bf = __builtin_bit_cast(bf16x8, bq[i][j]);
            acc[mi][j] =
                SWAP ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf, af[i & 1][mi], acc[mi][j], 0, 0, 0)
                     : __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i & 1][mi], bf, acc[mi][j], 0, 0, 0);
          }
        // the slot's refill: this block's step + PF, or the next block's start
        const bool more = s0 + PF < KST;
        load_step(bq[i], more ? col0 : next_col0, more ? step + PF : i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }

    // The tile's first position enters the addresses below afresh for every
    // block: hoisted out of the loop over blocks, those would hold dozens of
    // registers.
    int ta = t0;
    asm volatile("" : "+s"(ta));
#pragma unroll
    for (int j = 0; j < kBlockGroups; ++j) {
      const int nw = col0 + 16 * j;  // uniform
      if (nw >= n_end) continue;
      if constexpr (EPI == kStore) {
#pragma unroll
        for (int mi = 0; mi < kTilesM; ++mi) {
          const int row = ta + mi * 16 + c;
          if (row >= seq) continue;
          uint16_t v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = f32_to_bf16(acc[mi][j][r]);
          if (p.addend != nullptr) {
            const uint2 a = add_v[mi][j];
            v[0] = f32_to_bf16(lo_bf16(a.x) + bf16_to_f32(v[0]));
            v[1] = f32_to_bf16(hi_bf16(a.x) + bf16_to_f32(v[1]));
            v[2] = f32_to_bf16(lo_bf16(a.y) + bf16_to_f32(v[2]));
            v[3] = f32_to_bf16(hi_bf16(a.y) + bf16_to_f32(v[3]));
          }
          *reinterpret_cast<uint2*>(p.out + static_cast<int64_t>(row) * p.ldo + nw + 4 * g) =
              make_uint2(v[0] | static_cast<uint32_t>(v[1]) << 16, v[2] | static_cast<uint32_t>(v[3]) << 16);
        }
      } else if constexpr (SWAP) {
        // queries and keys (kRopeQkv, rotated) or keys (kFrag): one head per group
        const int head = nw / d;
        const int w = nw - head * d + 4 * g;
        const int H = EPI == kRopeQkv ? p.heads : 0;
        const int Hk = EPI == kRopeQkv ? p.kv_heads : n_swap / d;
#pragma unroll
        for (int mi = 0; mi < kTilesM; ++mi) {
          float x[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) x[r] = bf16_round(acc[mi][j][r]);
          if constexpr (EPI == kRopeQkv) {
            const float4 cs = *reinterpret_cast<const float4*>(&rope_s[(mi * 16 + c) * (d / 2) + w / 2]);
            const float e0 = x[0], o0 = x[1], e1 = x[2], o1 = x[3];
            x[0] = rope_even(e0, o0, cs.x, cs.y);
            x[1] = rope_odd(e0, o0, cs.x, cs.y);
            x[2] = rope_even(e1, o1, cs.z, cs.w);
            x[3] = rope_odd(e1, o1, cs.z, cs.w);
          }
          const int t = ta + mi * 16 + c;
          if (t >= seq) continue;
          const uint2 v = make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]));
          if (head < H) {
            *reinterpret_cast<uint2*>(
                p.q + ((static_cast<int64_t>(b) * H + head) * seq + t) * d + w) = v;
          } else {
            const int64_t bh = static_cast<int64_t>(b) * Hk + head - H;
            if (EPI == kRopeQkv && p.k != nullptr)
              *reinterpret_cast<uint2*>(p.k + (bh * seq + t) * d + w) = v;
            if (p.kf != nullptr)
              *reinterpret_cast<uint2*>(p.kf + kfrag_index(bh, p.nblk, t, w, d / 32)) = v;
          }
        }
      } else {
        // values: lane holds column c, positions t .. t + 3 (t % 4 == 0)
        const int head = (nw - n_swap) / d;
        const int w = nw - n_swap - head * d + c;
        const int Hv = EPI == kRopeQkv ? p.kv_heads : (p.N - n_swap) / d;
        const int64_t bh = static_cast<int64_t>(b) * Hv + head;
#pragma unroll
        for (int mi = 0; mi < kTilesM; ++mi) {
          const int t = ta + mi * 16 + 4 * g;
          if (t >= seq) continue;
          uint16_t bits[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) bits[r] = f32_to_bf16(acc[mi][j][r]);
          const uint2 v = make_uint2(bits[0] | static_cast<uint32_t>(bits[1]) << 16,
                                     bits[2] | static_cast<uint32_t>(bits[3]) << 16);
          // (positions past the sequence fall on the last block's padding keys)
          if (p.vf != nullptr)
            *reinterpret_cast<uint2*>(p.vf + vfrag_index(bh, p.nblk, t, w, d / 16)) = v;
          if (EPI == kRopeQkv && p.v != nullptr) {
            if (p.ld_keys > 0 && t + 4 <= seq) {
              *reinterpret_cast<uint2*>(p.v + (bh * d + w) * p.ld_keys + t) = v;
            } else {
#pragma unroll
              for (int r = 0; r < 4; ++r)
                if (t + r < seq)
                  p.v[p.ld_keys > 0 ? (bh * d + w) * p.ld_keys + t + r : (bh * seq + t + r) * d + w] =
                      bits[r];
            }
          }
        }
      }
    }
  };

  for (; blk < blk_end; blk += NW) {
    const int col0 = first_col(blk);
    const int next = first_col(min(blk + NW, cb.total - 1));
    if (blk < cb.first) run_block(std::true_type{}, col0, next);
    else run_block(std::false_type{}, col0, next);
  }
}

// Row tiles of bm rows, of one sequence each where the outputs are laid out
// per sequence.
template <int EPI>
int row_tiles(const ProjArgs& a, int bm) {
  if (EPI == kStore) return (a.rows + bm - 1) / bm;
  return a.rows / a.seq * ((a.seq + bm - 1) / bm);
}

// BM = 32 up to 4096 rows, where 64-row tiles leave a wavefront one block of
// columns and the A tile's load stands out (2 x 2047 rows: q|k|v 22.0 -> 19.8
// us, output 15.3 -> 12.6 us); 64 beyond, for half the weight traffic (2 x
// 4096: 35.7 -> 31.3 and 22.9 -> 20.7 us).
constexpr int kRows32 = 4096;
// From where the tiles beat proj_kernel (16 x 64 per workgroup): a number of
// rows, and of products, since a workgroup here loads its whole A tile first and
// has eight wavefronts to feed with 48-column blocks, which few columns do not
// (hence the growth below a few hundred), and since 8-byte stores and the
// addend's loads weigh more the shorter the k loop is.  Measured in graphs, us,
// that kernel / this.  Plain, K = 768: 1100 x 768 7.9 / 7.0, 1536 x 512 7.5 / 7.4,
// 4096 x 256 8.6 / 8.0, 8192 x 128 8.3 / 9.6, 16384 x 128 14.8 / 9.9; K = 512:
// 1100 x 768 6.4 / 6.4, 4200 x 256 7.1 / 7.7; K = 256: 2048 x 768 6.0 / 6.3, 4096 x
// 768 8.5 / 8.1, with an addend 9.1 / 9.1, 8192 x 512 12.8 / 10.3; K = 128: 4096 x
// 1152 9.2 / 8.9, with an addend 9.6 / 10.1, 8192 x 1536 19.4 / 18.4.  Per sequence:
// q|k|v K = 768 960 x 1152 9.7 / 9.5, K = 512 1024 x 768 7.3 / 8.8, K = 256 2000 x
// 512 6.9 / 8.3; keys and values from a latent of 128, 999 x 1536 6.6 / 5.9, 980 x
// 1536 (7 x 140) 5.8 / 6.2, 2000 x 512 4.8 / 5.2.
constexpr int kRowsFrom = 960, kStoreRowsFrom = 1100;

template <int EPI>
bool enough_products(const ProjArgs& a) {
  const double m = 1e6;
  double need;  // multiply-adds, at very many columns
  if (EPI != kStore) need = a.K == 128 ? 170 * m : a.K == 256 ? 280 * m : a.K == 512 ? 430 * m : 560 * m;
  else need = a.K == 128 ? 400 * m : a.K == 256 ? 500 * m : a.K == 512 ? 400 * m : 560 * m;
  if (EPI == kStore && a.addend != nullptr) need *= a.K == 128 ? 2.7 : a.K == 256 ? 1.7 : 1.0;
  return static_cast<double>(a.rows) * a.N * a.K >= need * (1.0 + 128.0 / a.N);
}

template <int EPI>
bool rows_apply(const ProjArgs& a) {
  const int steps = a.K / 32;
  if (a.K % 32 || (steps != 4 && steps != 8 && steps != 16 && steps != 24)) return false;
  // 8-byte accesses of the row-major operands and outputs
  const auto aligned8 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; };
  if (!enough_products<EPI>(a)) return false;
  if (EPI == kStore)
    return a.rows >= kStoreRowsFrom && a.ldo % 4 == 0 && aligned8(a.out) &&
           (a.addend == nullptr || (a.ld_addend % 4 == 0 && aligned8(a.addend)));
  // whole heads per 16-column group; sequences of at least four tiles, so that
  // their ragged ends stay a small part
  const int bm = a.rows <= kRows32 ? 32 : 64;
  return a.rows >= kRowsFrom && a.seq >= 4 * bm && a.head_dim % 16 == 0 && a.head_dim <= 128 &&
         a.ld_keys % 4 == 0 && aligned8(a.q) && aligned8(a.k) && aligned8(a.v) && aligned8(a.kf) &&
         aligned8(a.vf);
}

template <int BM, int EPI>
hipError_t launch_rows(const ProjArgs& a, hipStream_t s) {
  constexpr int NW = 8;
  const int tiles = row_tiles<EPI>(a, BM);
  // Column splits, each with its own copy of the A tile: the fewest rounds of
  // one workgroup per CU times what one takes (in column blocks of a
  // wavefront: about one for the A tile and the start, its blocks, and a tenth
  // for every block of the workgroup, whose wavefronts share the CU).
  const int blocks = (a.N + kBlockCols - 1) / kBlockCols;
  int splits = 1;
  float best = 0.0f;
  for (int n = 1; n <= 8 && n <= blocks; ++n) {
    const int64_t rounds = (static_cast<int64_t>(tiles) * n + 255) / 256;
    const int per_group = (blocks + n - 1) / n;
    const int per_wave = (per_group + NW - 1) / NW;
    const float cost = static_cast<float>(rounds) *
                       (1.0f + static_cast<float>(per_wave) + 0.1f * static_cast<float>(per_group));
    if (n == 1 || cost < best) {
      splits = n;
      best = cost;
    }
  }
  const int grid = tiles * splits;
  switch (a.K / 32) {
    case 4: proj_rows_kernel<BM, NW, 4, EPI><<<grid, 64 * NW, 0, s>>>(a, splits); break;
    case 8: proj_rows_kernel<BM, NW, 8, EPI><<<grid, 64 * NW, 0, s>>>(a, splits); break;
    case 16: proj_rows_kernel<BM, NW, 16, EPI><<<grid, 64 * NW, 0, s>>>(a, splits); break;
    case 24: proj_rows_kernel<BM, NW, 24, EPI><<<grid, 64 * NW, 0, s>>>(a, splits); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

int ring_depth(int ksteps) {
  for (int pf = 8; pf > 1; pf >>= 1)
    if (ksteps % pf == 0) return pf;
  return 1;
}

template <int EPI>
hipError_t launch_proj(const ProjArgs& a, hipStream_t s) {
  if (a.rows == 0 || a.N == 0) return hipSuccess;
  if constexpr (EPI != kStoreT) {
    if (rows_apply<EPI>(a))
      return a.rows <= kRows32 ? launch_rows<32, EPI>(a, s) : launch_rows<64, EPI>(a, s);
  }
  const int tiles = ((a.rows + kProjRows - 1) / kProjRows) * ((a.N + kProjCols - 1) / kProjCols);
  const size_t lds = static_cast<size_t>(kProjRows) * a.K * 2;
  switch (a.K / 32) {
    case 4: proj_kernel<4, EPI, 4><<<tiles, 256, lds, s>>>(a); break;
    case 8: proj_kernel<8, EPI, 8><<<tiles, 256, lds, s>>>(a); break;
    case 16: proj_kernel<16, EPI, 16><<<tiles, 256, lds, s>>>(a); break;
    case 24: proj_kernel<24, EPI, 24><<<tiles, 256, lds, s>>>(a); break;
    default:
      switch (ring_depth(a.K / 32)) {
        case 8: proj_kernel<8, EPI, 0><<<tiles, 256, lds, s>>>(a); break;
        case 4: proj_kernel<4, EPI, 0><<<tiles, 256, lds, s>>>(a); break;
        default: proj_kernel<2, EPI, 0><<<tiles, 256, lds, s>>>(a); break;
      }
  }
  return hipGetLastError();
}

}  // namespace

bool proj_shape_supported(int k, int n) {
  return k > 0 && k % 64 == 0 && k <= kProjMaxK && n > 0 && n % 16 == 0;
}

hipError_t launch_proj_store(const uint16_t* x, int rows, int k, int64_t lda, const uint16_t* w,
                             int n, const uint16_t* addend, int64_t ld_addend, uint16_t* out,
                             int64_t ldo, hipStream_t s) {
  ProjArgs a{};
  a.x = x; a.lda = lda; a.rows = rows; a.K = k; a.N = n; a.w = w;
  a.out = out; a.ldo = ldo; a.addend = addend; a.ld_addend = ld_addend;
  a.seq = 1;
  return launch_proj<kStore>(a, s);
}

hipError_t launch_proj_transposed(const uint16_t* x, int rows, int seq, int k, const uint16_t* w,
                                  int n, int ld_keys, uint16_t* out, hipStream_t s) {
  ProjArgs a{};
  a.x = x; a.lda = k; a.rows = rows; a.K = k; a.N = n; a.w = w;
  a.out = out; a.seq = seq; a.ld_keys = ld_keys;
  return launch_proj<kStoreT>(a, s);
}

hipError_t launch_proj_rope_qkv(const uint16_t* x, int rows, int seq, int dim, const uint16_t* w,
                                const float* cos_t, const float* sin_t, int start,
                                const int32_t* start_device, int max_positions, int heads,
                                int kv_heads, int head_dim, int vt_keys, uint16_t* q,
                                uint16_t* k, uint16_t* v, uint16_t* kf, uint16_t* vf,
                                hipStream_t s) {
  ProjArgs a{};
  a.kf = kf; a.vf = vf; a.nblk = (seq + 31) / 32;
  a.x = x; a.lda = dim; a.rows = rows; a.K = dim; a.N = (heads + 2 * kv_heads) * head_dim;
  a.w = w; a.seq = seq; a.ld_keys = vt_keys;
  a.cos_t = cos_t; a.sin_t = sin_t; a.start = start; a.start_device = start_device;
  a.max_positions = max_positions;
  a.heads = heads; a.kv_heads = kv_heads; a.head_dim = head_dim;
  a.q = q; a.k = k; a.v = v;
  return launch_proj<kRopeQkv>(a, s);
}

hipError_t launch_proj_frag(const uint16_t* x, int rows, int seq, int k, int64_t lda,
                            const uint16_t* w, int n, int head_dim, uint16_t* kf, uint16_t* vf,
                            hipStream_t s) {
  ProjArgs a{};
  a.x = x; a.lda = lda; a.rows = rows; a.K = k; a.N = n; a.w = w;
  a.seq = seq; a.head_dim = head_dim; a.nblk = (seq + 31) / 32;
  a.kf = kf; a.vf = vf;
  return launch_proj<kFrag>(a, s);
}

}  // namespace parrot
