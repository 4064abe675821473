// Expert GEMMs over long expert segments (chunked prefill, configs with many rows
// per expert) on gfx950 matrix cores: the sorted-segment gather_qmm of the
// reference's prefill (Q36/kernels/gather_qmm_prefill.py:1-257, MLX's quantized
// block loader + tile MMA), whose arithmetic it keeps: every weight is
// dequantized to bf16, w = bf16(s * q + b), and the MMA accumulates bf16
// products in fp32.  Rows are independent, so a row's result does not depend on
// how many rows its expert has.
//
// Work split: a workgroup of WAVES waves (4 or 8) owns 32 WAVES weight rows of one expert (gate||up:
// gate blocks and the up blocks of the same output columns, so SwiGLU is fused) and one chunk of up to
// 16 * TTS tokens of the expert's segment at a time.  Each wave owns 2 row blocks (gate||up: a
// gate block and its up block).  K is walked in steps of one group pair (128 k): the wave
// dequantizes its 2 row blocks' pair into bf16 MFMA B fragments once and uses them against every
// token tile of the chunk, whose activations the workgroup stages in LDS (gathered through pair_row
// for gate||up).  The next steps' packed weights and activations are loaded while the current step
// computes.  fp32 accumulators: TTS x 2 tiles of 16 x 16 per wave.
//
// What bounds it, and the shapes (SegShape).  Long segments are bound by issue: the dequantization
// (vector ALU, the same for any chunk length) and the MFMAs, which two waves a SIMD overlap; 10 tiles a
// chunk spread the dequantization over 160 tokens.  A short segment (a 512-row prompt chunk leaves 32
// pairs an expert) is bound by the latency of its K steps -- barrier, activations, weights -- and wastes
// what it computes past its last token: it takes a chunk of few tiles in workgroups of 4 waves and at
// most 51 KB of LDS, three or four of them a CU, whose steps, prologues and epilogues overlap.
// Deeper rings do not help: loads complete in order, so a wait for a step's activations also waits for
// every weight load issued before them.  128 experts, top-8, 2048 x 768, us (gate||up + down; 10 tiles
// at every size before -> now): 64 rows 130 + 66 -> 49 + 33, 256 rows 124 + 68 -> 60 + 34, 512 rows
// 128 + 70 -> 75 + 42, 1,024 rows 138 + 75 -> 101 + 60, 2,108 rows 153 + 93 -> 144 + 88.
#include <algorithm>
#include <cmath>

#include "qtile.hpp"

namespace {

constexpr int kSegRB = 2;                 // row blocks per wave
constexpr int seg_rows(int waves) { return 16 * kSegRB * waves; }  // weight rows per workgroup
constexpr int kSegRows = seg_rows(8);     // rows a dense matrix or a down stack is a multiple of
#ifndef JIT_SEG_AHEAD
#define JIT_SEG_AHEAD 1
#endif
constexpr int kSegAhead = JIT_SEG_AHEAD;  // token tiles whose fragment reads run ahead of the MFMAs

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // (HIP's uint4 is a union-based struct)

struct SegArgs {
  const uint16_t *x;          // activations [rows, K] bf16
  const int32_t *row_index;   // x row of each sorted position (null: the position itself)
  const int32_t *cnt, *off;   // pairs per expert, first sorted position per expert (null: a
                              // dense matrix, E = 1, rows 0 .. T - 1)
  const uint8_t *w;           // packed stack [E, rows_w, K]
  uint16_t *out;              // [P, N] bf16 in sorted order
  long long w_estride;        // packed bytes per expert
  int K, N;                   // N: output columns (I for gate||up, D for down)
  int T;                      // rows of a dense matrix (cnt null)
  int nx, groups;             // column blocks per group; groups = experts (or a dense matrix's token chunks)
  int dealt;                  // groups of the grid: the experts, and groups that only take dealt chunks
};

// Workgroup -> (group, column block), XCD-aware.  MI355X deals the workgroups of a launch to its
// 8 XCDs round-robin (workgroup i to XCD i % 8), and each XCD has its own L2.  All column blocks
// of one group (an expert's segment, or one token chunk of a dense matrix) read the same
// activation rows, so they are given consecutive slots of one XCD: group g goes to XCD g % 8,
// and its nx blocks follow each other there, resident together, so the rows leave HBM (or the
// last-level cache) once per group instead of once per column block.  The grid is padded to
// 8 * ceil(dealt / 8) groups; the padding's workgroups exit at once.
__device__ __forceinline__ bool seg_block(const SegArgs &a, int &g, int &cb) {
  const int L = blockIdx.x, xcd = L & 7, slot = L >> 3;
  g = xcd + 8 * (slot / a.nx);
  cb = slot % a.nx;
  return g < a.dealt;
}

inline dim3 seg_grid(int nx, int groups) { return dim3(nx * 8 * ((groups + 7) / 8)); }

// 8 packed-order nibbles of a word -> 8 bf16 weights bf16(s * q + b) in natural k order, 19 vector
// instructions: a shift and a mask leave two nibbles in the low bits of a register's halves, where as
// f16 denormals they are q 2^-24; v_fma_mix_f32 takes such a half as an operand, so s2 = 2^24 s (exact
// for |s| < 2^104; dequant_word_wide serves the others) times it plus b is the fp32 fma(s, q, b) in one
// instruction, where a byte conversion and an fma were two (gate||up of 2,108 rows 147 -> 144 us, of 512 rows
// 78 -> 75 us; the same bits).  The weights are rounded in pairs (one v_cvt_pk_bf16_f32 each).
__device__ __forceinline__ Frag8 dequant_word(uint32_t w, float s2, float b) {
  Frag8 f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t u = (w >> (4 * j)) & 0x000F000Fu;  // (q[2j], q[2j + 1])
    float lo, hi;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(lo) : "v"(u), "v"(s2), "v"(b));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(hi) : "v"(u), "v"(s2), "v"(b));
    f.u[j] = pack_bf16x2_rne(lo, hi);
  }
  return f;
}

// The same for any scale.
__device__ __forceinline__ Frag8 dequant_word_wide(uint32_t w, float s, float b) {
  Frag8 f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t u = w >> (4 * j);  // (q[2j] in bits 0-3, q[2j + 1] in bits 16-19)
    f.u[j] = pack_bf16x2_rne(fmaf(s, (float)(u & 15u), b), fmaf(s, (float)((u >> 16) & 15u), b));
  }
  return f;
}

// LDS of a workgroup:
//   activation stages: one K step's activations, 16 TTS token rows of 128 k (256 B, no
//     padding).  Row r's 16 B piece c sits in slot c ^ (r % 16), so the 16 rows one fragment
//     read touches (same piece, rows 16 t .. 16 t + 15) fall in 16 different slots: the reads
//     are free of bank conflicts without the padding the direct global->LDS loads (1 KB = 4
//     whole rows per wave instruction) could not insert;
//   weight stages: per wave its 2 row blocks' nibble tiles of one K step (2 x 1 KB) and their scale
//     tiles (2 x 128 B).
constexpr int kSegWLoads = kSegRB + 1;  // direct loads of a wave's weights per K step
constexpr int kSegWWave = kSegRB * (qtile::kNibbleBytes + qtile::kScaleBytes);

// A shape of the kernel: TTS token tiles a chunk, WAVES waves a workgroup, activations requested DX
// K steps ahead and weights DW steps ahead.
template <int TTS_, int WAVES_, int DX_, int DW_, int OCC_ = 2>
struct SegShape {
  static constexpr int TTS = TTS_, WAVES = WAVES_, DX = DX_, DW = DW_, OCC = OCC_;
  static constexpr int kThreads = 64 * WAVES, kRows = seg_rows(WAVES), kTokens = 16 * TTS;
  static constexpr int kXLoads = 4 * TTS / WAVES;  // a wave's activation loads per K step
  static constexpr int kXStage = kTokens * 256, kWStage = WAVES * kSegWWave;
  static constexpr int kWOff = (DX + 1) * kXStage;
  static constexpr int kLds = kWOff + DW * kWStage;
  // the most loads one of the kernel's waits can leave in flight
  static constexpr int kMaxWait = (DX > DW ? DX : DW) * (kXLoads + kSegWLoads);
  static_assert(WAVES == 4 || WAVES == 8, "a wave stages 4 rows of a token tile: 4 waves a tile");
  static_assert(4 * TTS % WAVES == 0, "the halves of 8 waves stage alternate token tiles");
  static_assert(DX <= DW && kMaxWait < 64, "the waits' steady counts; vmcnt is 6 bits");
  static_assert(kLds <= 160 * 1024, "gfx950 gives a workgroup at most 160 KB of LDS");
};

// s_waitcnt vmcnt(N), nothing else.  Direct loads are counted by hand: the compiler does not see
// the ones issued by inline assembly, and it takes the wait itself for an instruction that touches no
// memory: the fence after it keeps the reads of what has landed behind it.
template <int N>
__device__ __forceinline__ void seg_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
}

// s_waitcnt vmcnt(n) for a count known at run time (uniform), n in [LO, HI): the instruction's count
// is an immediate, so the value is found by bisection over scalar branches.
template <int LO, int HI>
__device__ __forceinline__ void seg_wait_vm_n(int n) {
  if constexpr (HI - LO == 1) {
    seg_wait_vm<LO>();
  } else {
    constexpr int MID = (LO + HI) / 2;
    if (n >= MID)
      seg_wait_vm_n<MID, HI>(n);
    else
      seg_wait_vm_n<LO, MID>(n);
  }
}

// A workgroup barrier that waits for nothing else: every wave has already waited for its own
// direct loads (__syncthreads()'s fence would also wait for the loads still in flight).
__device__ __forceinline__ void seg_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// (the dword form: 256 B a wave)
__device__ __forceinline__ void seg_load_lds4(const void *src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(dst) : "memory", "m0");
}

__device__ __forceinline__ void seg_load_lds(const void *src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(dst) : "memory", "m0");
}

// DENSE: one dense matrix (E = 1, cnt null), one token chunk per group.
//
// Pipeline over the K steps p (one group pair each).  Per wave and step, 4 TTS / WAVES direct loads of
// activations (4 rows of a token tile each; with 8 waves, waves 0-3 stage the even tiles and 4-7 the odd
// ones) and 3 of its packed weights.
//   top of step p: wait for step p's activations, one barrier; request step p + DX's activations and
//     step p + DW's weights into the stages that step p - 1 has left;
//   group 0's token tiles against B fragments dequantized during step p - 1, with the
//     dequantization of this step's group 1 between their MFMAs;
//   wait for step p + 1's weights (the wave's own: no barrier) and read them into registers, then group
//     1's token tiles with the dequantization of step p + 1's group 0 between their MFMAs.
// Each tile's activation fragments are read kSegAhead tiles ahead of its MFMAs.  (Activations are
// mostly L2 hits: an expert's column blocks run on one XCD.)
template <bool SWIGLU, bool DENSE, class S>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu(S::OCC, S::OCC))) void seg_kernel(const SegArgs a) {
  constexpr int TTS = S::TTS, WAVES = S::WAVES, DX = S::DX, DW = S::DW;
  constexpr int kTokens = S::kTokens, kStage = S::kXStage, kXLoads = S::kXLoads;
  extern __shared__ __attribute__((aligned(16))) uint8_t seg_lds[];
  int grp, cb;
  if (!seg_block(a, grp, cb)) return;  // grid padding (uniform over the workgroup)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id();
  // Experts: a workgroup takes its expert's first chunk, and the chunks past the first of all experts are dealt
  // to the column block's workgroups in equal runs, one more to those without a chunk of their own first (runs:
  // the chunks of an expert that follow each other read its weights from L2).  An expert in many rows would
  // otherwise be walked by one workgroup a column block while the chip waits, and in the shorter chunks of
  // the mean segment: 128 experts, every row with the same 8 of them, gate||up + down, us, walked so / walked in
  // 160 tokens / dealt: 100 rows 111 / 57 / 45, 300 rows 184 / 113 / 64, 2,108 rows 707 / 764 / 205.  Even routing pays
  // for the count at the start (64 rows 78.3 -> 79.5).  Every wave counts for itself.
  const int E = a.groups;
  auto chunks_past_first = [&](int c) { return (uint32_t)max(c - 1, 0) / (uint32_t)kTokens; };
  int next = 0, end = 0;  // the chunks past the first that this workgroup is dealt
  int cnt = a.T, off = 0;
  if (!DENSE) {
    // (every load is issued before any is waited for: they are the first thing a workgroup waits for)
    const int own = min(grp, E - 1);
    cnt = a.cnt[own];
    off = a.off[own];
    auto two = [&](int b) {
      const int c0 = a.cnt[min(b + l, E - 1)], c1 = a.cnt[min(b + 64 + l, E - 1)];
      return (b + l < E ? chunks_past_first(c0) : 0u) + (b + 64 + l < E ? chunks_past_first(c1) : 0u);
    };
    uint32_t n = two(0);
    for (int b = 128; b < E; b += 128) n += two(b);
    if (grp >= E) cnt = 0;
    if (__any(n > 0)) {
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) n += __shfl_xor(n, o, 64);
      const int extra = __builtin_amdgcn_readfirstlane(n);
      int none = 0, before = 0;  // experts without a pair; those of them before this workgroup's
      for (int b = 0; b < E; b += 64) {
        const unsigned long long m = __ballot(b + l < E && a.cnt[min(b + l, E - 1)] <= 0);
        none += __builtin_popcountll(m);
        before += __builtin_popcountll(grp >= b + 64 ? m : grp > b ? m & ((1ull << (grp - b)) - 1) : 0ull);
      }
      // the order: the groups past the experts, the experts without a pair, the others
      const int past = a.dealt - E;
      const int turn = grp >= E ? grp - E : cnt <= 0 ? past + before : past + none + grp - before;
      const int each = extra / a.dealt, more = extra % a.dealt;
      next = turn * each + min(turn, more);
      end = next + each + (turn < more ? 1 : 0);
    }
    if (cnt <= 0 && next >= end) return;  // uniform over the workgroup
  }
  const int lr = l & 15, lg = l >> 4;
  const int tid = threadIdx.x;
  const int GP = a.K >> 7;  // K steps (group pairs)
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)seg_lds);

  // the wave's 2 row blocks (index of the first row / 16 inside the expert's stack)
  int rbk[kSegRB];
#pragma unroll
  for (int r = 0; r < kSegRB; r++) {
    if (SWIGLU)  // gate block WAVES cb + wave, and the up block of the same columns
      rbk[r] = (r ? a.N / 16 : 0) + cb * WAVES + wave;
    else
      rbk[r] = kSegRB * (cb * WAVES + wave) + r;
  }
  const uint8_t *wexp, *wnib, *wscl;  // the expert's weights
  const long long tile_row = (long long)GP * qtile::kTileBytes;  // bytes of one row block's tiles
  // weight staging: nibble instruction r moves row block r's tile (lane l: its 16 B piece); the
  // scale instruction's lane l moves word l % 32 of row block l / 32's scale tile
  auto set_expert = [&](int e) {
    wexp = a.w + (long long)e * a.w_estride;
    wnib = wexp + 16 * l;
    const int rb_s = l >> 5 ? rbk[1] : rbk[0];
    wscl = wexp + rb_s * tile_row + (long long)GP * qtile::kNibbleBytes + 4 * (l & 31);
  };
  const uint32_t wlds = lds0 + S::kWOff + wave * kSegWWave;  // + stage * kWStage
  const uint8_t *wmine = seg_lds + S::kWOff + wave * kSegWWave;
  auto load_w = [&](int p) {
    const uint32_t st = wlds + (p % DW) * S::kWStage;
#pragma unroll
    for (int r = 0; r < kSegRB; r++)
      seg_load_lds(wnib + rbk[r] * tile_row + p * qtile::kNibbleBytes, __builtin_amdgcn_readfirstlane(st + r * 1024));
    seg_load_lds4(wscl + p * qtile::kScaleBytes, __builtin_amdgcn_readfirstlane(st + kSegRB * 1024));
  };
  // the lane's staged weights of step p, read into registers half a step before they are dequantized:
  // per row block both groups' two words and the row's scale and bias pairs (each group's dequantization
  // reading its own words would wait on the LDS 16 times a step)
  uint4 rq[kSegRB];
  uint2 rs[kSegRB];
  auto fetch_w = [&](int p) {
    const uint8_t *st = wmine + (p % DW) * S::kWStage;
#pragma unroll
    for (int r = 0; r < kSegRB; r++) {
      rq[r] = *(const uint4 *)(st + r * 1024 + 16 * l);
      rs[r] = *(const uint2 *)(st + kSegRB * 1024 + r * 128 + 8 * lr);
    }
  };
  // B fragment h of group g, row block r: bf16(s q + b) of the lane's word h of the group (the nibble
  // tile's 16 B piece holds group 0's two words, then group 1's)
  auto dequant_at = [&](int g, int r, int h, Frag8 (&bw)[kSegRB][2]) {
    const uint32_t q = g ? (h ? rq[r].w : rq[r].z) : (h ? rq[r].y : rq[r].x);
    const float sc = g ? bf2f_hi(rs[r].x) : bf2f(rs[r].x & 0xffffu);
    const float bi = g ? bf2f_hi(rs[r].y) : bf2f(rs[r].y & 0xffffu);
    bw[r][h] = dequant_word(q, sc * 16777216.0f, bi);
  };
  // activation staging: the wave's instruction i moves rows 4 (wave % 4) .. + 3 (1 KB) of token
  // tile j = (WAVES / 4) i + wave / 4; lane l fetches the piece its slot l % 16 holds in row 16 j + srow
  const int srow = 4 * (wave & 3) + (l >> 4), jhalf = wave >> 2;
  constexpr int kXTile = WAVES / 4;
  const int spiece = (l & 15) ^ srow;
  // fragment reads: lane (lr, lg) reads pieces 8 g + 2 lg and + 1 of row 16 t + lr
  const int frow = lr * 256;

  int c0 = DENSE ? grp * kTokens : 0;
  set_expert(DENSE ? 0 : min(grp, E - 1));
  for (bool own_chunk = DENSE || cnt > 0;; own_chunk = false) {
    if (!DENSE && !own_chunk) {
      if (next >= end) return;
      const int item = next++;
      uint32_t run = 0;
      for (int b = 0;; b += 64) {
        if (b >= E) return;  // (there are more than `item` of them: not reached)
        const uint32_t v = b + l < E ? chunks_past_first(a.cnt[b + l]) : 0u;
        uint32_t incl = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const uint32_t u = __shfl_up(incl, o, 64);
          if (l >= o) incl += u;
        }
        const unsigned long long past = __ballot(run + incl > (uint32_t)item);
        if (past) {
          const int src = __builtin_ctzll(past), e = __builtin_amdgcn_readfirstlane(b + src);
          c0 = (item - __builtin_amdgcn_readfirstlane(__shfl(run + incl - v, src, 64)) + 1) * kTokens;
          cnt = a.cnt[e];
          off = a.off[e];
          set_expert(e);
          break;
        }
        run += __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
      }
      __syncthreads();  // an earlier chunk's reads of the stages are done
    }
    const int nt = min(kTokens, cnt - c0);
    const int last = GP - 1;
    // element offsets of this lane's pieces (x holds < 2^32 elements; rows past the segment re-read its
    // last row)
    uint32_t xsrc[kXLoads];
    auto first_w = [&]() {
#pragma unroll
      for (int i = 0; i < DW; i++)
        if (i <= last) load_w(i);
    };
    if constexpr (kXLoads <= 4) {
      // the first weights go out before the row indices are read (they depend on the expert alone), and
      // the rows come by scalar loads, whose wait does not wait for the weights
      first_w();
#pragma unroll
      for (int i = 0; i < kXLoads; i++) {
        int row[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int pos = off + c0 + min(16 * (kXTile * i + jhalf) + 4 * (wave & 3) + j, nt - 1);
          row[j] = a.row_index ? ((const __attribute__((address_space(4))) int32_t *)a.row_index)[pos] : pos;
        }
        const int rr = lg < 2 ? (lg == 0 ? row[0] : row[1]) : (lg == 2 ? row[2] : row[3]);
        xsrc[i] = (uint32_t)rr * (uint32_t)a.K + 8 * spiece;
      }
    } else {  // (20 or more rows a wave would spill scalar registers)
#pragma unroll
      for (int i = 0; i < kXLoads; i++) {
        const int pos = off + c0 + min(16 * (kXTile * i + jhalf) + srow, nt - 1);
        xsrc[i] = (uint32_t)(a.row_index ? a.row_index[pos] : pos) * (uint32_t)a.K + 8 * spiece;
      }
      first_w();
    }
    auto load_x = [&](int p) {
      const uint32_t st = lds0 + (p % (DX + 1)) * kStage + 4 * (wave & 3) * 256;
#pragma unroll
      for (int i = 0; i < kXLoads; i++)
        seg_load_lds(a.x + xsrc[i] + 128 * p, __builtin_amdgcn_readfirstlane(st + 16 * (kXTile * i + jhalf) * 256));
    };

    f32x4 acc[TTS][kSegRB];
#pragma unroll
    for (int t = 0; t < TTS; t++)
#pragma unroll
      for (int r = 0; r < kSegRB; r++) acc[t][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    Frag8 bw0[kSegRB][2], bw1[kSegRB][2];

    // all TTS token tiles of group g of step p against bw, with no branch (tiles past the
    // chunk compute on rows that are never stored: a branch per tile would keep the
    // dequantization from being scheduled between the MFMAs); side(t) is the dequantization of
    // one B fragment (word t % 2 of row block t / 2) interleaved with tile t's MFMAs (t < 8)
    auto tiles = [&](int p, int g, Frag8 (&bw)[kSegRB][2], auto &&side) {
      const uint8_t *xs = seg_lds + (p % (DX + 1)) * kStage + frow;
      const int pa = 8 * g + 2 * lg;
      const int o0 = 16 * (pa ^ lr), o1 = 16 * ((pa + 1) ^ lr);
      Frag8 xa[kSegAhead + 1][2];
#pragma unroll
      for (int t = 0; t < kSegAhead; t++) {
        xa[t][0].q = *(const uint4 *)(xs + t * 16 * 256 + o0);
        xa[t][1].q = *(const uint4 *)(xs + t * 16 * 256 + o1);
      }
#pragma unroll
      for (int t = 0; t < TTS; t++) {
        if (t + kSegAhead < TTS) {
          Frag8 *n = xa[(t + kSegAhead) % (kSegAhead + 1)];
          n[0].q = *(const uint4 *)(xs + (t + kSegAhead) * 16 * 256 + o0);
          n[1].q = *(const uint4 *)(xs + (t + kSegAhead) * 16 * 256 + o1);
        }
        const Frag8 *c = xa[t % (kSegAhead + 1)];
#pragma unroll
        for (int r = 0; r < kSegRB; r++) {
          acc[t][r] = mfma16x16x32(c[0], bw[r][0], acc[t][r]);
          acc[t][r] = mfma16x16x32(c[1], bw[r][1], acc[t][r]);
        }
        if (t < 2 * kSegRB) side(t);
      }
      // (a chunk of fewer tiles than B fragments runs the rest of them after its tiles)
#pragma unroll
      for (int t = TTS; t < 2 * kSegRB; t++) side(t);
    };

    // Loads are issued as w(0 .. DW - 1), x(0 .. DX - 1), then x(p + DX), w(p + DW) at the top of each
    // step p, as far as the steps exist.  A wait may leave in flight the loads issued after the awaited
    // ones; wait_x and wait_w count exactly those (every wave issues the same sequence).
    auto wait_x = [&](int p) {  // at the top of step p, before its loads: x(p) has landed
      if (p >= DX && p - 1 + DW <= last) {
        seg_wait_vm<(DX - 1) * kXLoads + DX * kSegWLoads>();
        return;
      }
      const int nx = min(p - 1 + DX, last) - p;
      const int nw = min(p - 1 + DW, last) - (p < DX ? DW - 1 : p - DX + DW - 1);
      seg_wait_vm_n<0, S::kMaxWait + 1>(
          __builtin_amdgcn_readfirstlane(max(nx, 0) * kXLoads + max(nw, 0) * kSegWLoads));
    };
    auto wait_w = [&](int p) {  // in step p, after its loads: w(p + 1) has landed
      if (p + 1 >= DW && p + DW <= last && p + DX <= last) {
        seg_wait_vm<(DW - 1) * (kXLoads + kSegWLoads)>();
        return;
      }
      const int nw = min(p + DW, last) - (p + 1);
      const int nx = min(p + DX, last) - (p + 1 < DW ? -1 : p + 1 - DW + DX);
      seg_wait_vm_n<0, S::kMaxWait + 1>(
          __builtin_amdgcn_readfirstlane(max(nx, 0) * kXLoads + max(nw, 0) * kSegWLoads));
    };
#pragma unroll
    for (int i = 0; i < DX; i++)
      if (i <= last) load_x(i);
    wait_w(-1);
    fetch_w(0);
    wait_x(0);
    seg_barrier();
#pragma unroll
    for (int r = 0; r < kSegRB; r++) {
      dequant_at(0, r, 0, bw0);
      dequant_at(0, r, 1, bw0);
    }
    for (int p = 0; p < GP; p++) {
      if (p > 0) {
        wait_x(p);
        seg_barrier();
      }
      if (p + DX <= last) load_x(p + DX);
      if (p + DW <= last) load_w(p + DW);
      tiles(p, 0, bw0, [&](int t) { dequant_at(1, t >> 1, t & 1, bw1); });
      if (p < last) wait_w(p);
      fetch_w(p + 1);  // (after the last step a stale stage, unused)
      tiles(p, 1, bw1, [&](int t) { dequant_at(0, t >> 1, t & 1, bw0); });
    }

    // SwiGLU's sigmoid by table (qtile::swiglu_bf16_tab, exhaustively equal to the bf16 steps): every
    // wave is done with the stages, so the table (7.7 KB) takes the start of the LDS, one entry
    // or so a thread instead of ~45 instructions for each of a lane's ~40 outputs
    // (a short chunk's few outputs cost less by the steps than a table entry or more a thread)
    constexpr bool kTable = SWIGLU && 4 * TTS > qtile::kSigEntries / S::kThreads + 4;
    const uint16_t *sig_tab = (const uint16_t *)seg_lds;
    if constexpr (kTable) {
      __syncthreads();
      for (int i = tid; i < qtile::kSigEntries; i += S::kThreads) ((uint16_t *)seg_lds)[i] = qtile::sigmoid_entry(i);
      __syncthreads();
    }
    // lane l holds C[token 16 t + 4 lg + i][row 16 rbk[r] + lr].  No branch per token: the
    // stores go through a buffer resource (the launch checks that the output spans less than
    // 2 GiB), and a token past the chunk gets an offset past its range, whose store is dropped.
    // (Whole tiles past the chunk are skipped: a branch uniform over the wave.)
    const __amdgpu_buffer_rsrc_t obuf = __builtin_amdgcn_make_buffer_rsrc((void *)a.out, (short)0, 0x7fffffff, 0x00020000);
    const int ntiles = (nt + 15) >> 4;
    auto store_tile = [&](int t, const f32x4 (&c)[kSegRB]) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int tok = 16 * t + 4 * lg + i;
        const uint32_t ro = tok < nt ? (uint32_t)(off + c0 + tok) * (uint32_t)a.N * 2u : 0x80000000u;
        if (SWIGLU) {
          uint32_t hv;
          if constexpr (kTable)
            hv = qtile::swiglu_bf16_tab(c[0][i], c[1][i], sig_tab);
          else
            hv = qtile::swiglu_bf16(c[0][i], c[1][i]);
          __builtin_amdgcn_raw_buffer_store_b16((unsigned short)hv, obuf, (int)(ro + 2u * (16 * rbk[0] + lr)), 0, 0);
        } else {
#pragma unroll
          for (int r = 0; r < kSegRB; r++)
            __builtin_amdgcn_raw_buffer_store_b16((unsigned short)f2bf(c[r][i]), obuf,
                                                  (int)(ro + 2u * (16 * rbk[r] + lr)), 0, 0);
        }
      }
    };
    // A scale past dequant_word's range is infinite there: its group's 64 weights are infinities and NaNs, and
    // with them the sums of its row for every token.  So a token's sums that are not finite say that the wave's
    // sums have to be made again: in the same order, by dequant_word_wide, a tile at a time and straight from
    // memory (no barrier: other waves need not come here).  Inputs that are not finite come here too.
    if (__any(!__builtin_isfinite(acc[0][0][0]) || !__builtin_isfinite(acc[0][1][0]))) {
#pragma unroll 1
      for (int t = 0; t < ntiles; t++) {
        const int pos = off + c0 + min(16 * t + lr, nt - 1);
        const uint16_t *xr = a.x + (uint32_t)(a.row_index ? a.row_index[pos] : pos) * (uint32_t)a.K + 16 * lg;
        f32x4 c[kSegRB] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 1
        for (int pg = 0; pg < 2 * GP; pg++) {
          const int p = pg >> 1, g = pg & 1;
          Frag8 xa[2];
          xa[0].q = *(const uint4 *)(xr + 64 * pg);
          xa[1].q = *(const uint4 *)(xr + 64 * pg + 8);
#pragma unroll
          for (int r = 0; r < kSegRB; r++) {
            const uint8_t *blk = wexp + rbk[r] * tile_row;
            const uint2 q = *(const uint2 *)(blk + p * qtile::kNibbleBytes + 16 * l + 8 * g);
            const uint2 sb = *(const uint2 *)(blk + (long long)GP * qtile::kNibbleBytes + p * qtile::kScaleBytes + 8 * lr);
            const float sc = bf2f((g ? sb.x >> 16 : sb.x) & 0xffffu), bi = bf2f((g ? sb.y >> 16 : sb.y) & 0xffffu);
            c[r] = mfma16x16x32(xa[0], dequant_word_wide(q.x, sc, bi), c[r]);
            c[r] = mfma16x16x32(xa[1], dequant_word_wide(q.y, sc, bi), c[r]);
          }
        }
        store_tile(t, c);
      }
    } else {
#pragma unroll
      for (int t = 0; t < TTS; t++)
        if (t < ntiles) store_tile(t, acc[t]);
    }
    if (DENSE) return;
  }
}

// One launch of a shape: the column blocks of its rows for each of a.groups groups, P pairs in all (the kernels
// take more LDS than the static limit: raise their dynamic limit once).
template <bool SWIGLU, bool DENSE, class S>
void seg_launch(SegArgs a, int rows, hipStream_t st, int P = 0) {
  static const bool done = [] {
    (void)hipFuncSetAttribute((const void *)&seg_kernel<SWIGLU, DENSE, S>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              S::kLds);
    return true;
  }();
  (void)done;
  a.nx = rows / S::kRows;
  if (DENSE) a.groups = (a.T + S::kTokens - 1) / S::kTokens;
  a.dealt = a.groups;
  if (!DENSE) {  // as many groups as dealt chunks may need, where the experts' own leave room on an XCD's CUs
    const int room = 8 * (jit::cu_count() / 8 * (S::WAVES == 4 ? 3 : 1) / a.nx) - a.groups;
    a.dealt += std::max(0, std::min(room, P / S::kTokens));
  }
  seg_kernel<SWIGLU, DENSE, S><<<seg_grid(a.nx, a.dealt), S::kThreads, S::kLds, st>>>(a);
}

// The chunk length of expert segments: the smallest that holds the mean segment plus 2.5 of its
// standard deviations under even routing (sqrt(mean)), so that few experts need a second pass over
// their weights and few tiles are computed past a segment's end.  A shorter chunk re-reads the weights
// (512 rows, mean 32: 2 tiles 103 + 54 us gate||up + down, 3 tiles 75 + 42), a longer one computes
// padding (4 tiles 78 + 43, 6 tiles 95 + 53, 10 tiles 125 + 64).  Every shape gives the same bits.
template <bool SWIGLU>
void seg_experts(const SegArgs &a, int rows, int P, hipStream_t st) {
  const float mean = (float)P / (float)a.groups, need = mean + 2.5f * sqrtf(mean);
  if (need <= 16.0f)
    seg_launch<SWIGLU, false, SegShape<1, 4, 2, 2, 4>>(a, rows, st, P);
  else if (need <= 32.0f)
    seg_launch<SWIGLU, false, SegShape<2, 4, 2, 2, 3>>(a, rows, st, P);
  else if (need <= 48.0f)
    seg_launch<SWIGLU, false, SegShape<3, 4, 1, 2, 3>>(a, rows, st, P);
  else if (need <= 64.0f)
    seg_launch<SWIGLU, false, SegShape<4, 4, 1, 2, 3>>(a, rows, st, P);
  else if (need <= 96.0f)
    seg_launch<SWIGLU, false, SegShape<6, 8, 1, 2>>(a, rows, st, P);
  else
    seg_launch<SWIGLU, false, SegShape<10, 8, 1, 2>>(a, rows, st, P);
}

// The chunk length of a dense matrix (its token chunks spread over workgroups): the least estimated
// time of a K step, from the workgroups L that the busiest CU gets (seg_block deals whole groups to 8
// XCDs).  Up to three workgroups of 4 waves share a CU, 0.38 + L (0.24 + 0.09 tiles) us a step; those of
// 8 waves follow one another, 0.60 + 0.17 tiles each.  Fitted to N = 5120, K = 2048 and N = 2048,
// K = 4096 at 192 .. 2,108 rows, where it picks the fastest shape measured: 192 rows 20 + 25 us, 512
// rows 25 + 26 (36 + 36 before), 1,024 rows 33 + 30, 2,108 rows 56 + 48 (79 + 57 before).
float seg_dense_step_us(int tts, int waves, int T, int N, int cus) {
  const int groups = (T + 16 * tts - 1) / (16 * tts), per_xcd = (N / seg_rows(waves)) * ((groups + 7) / 8);
  const int cu = cus >= 8 ? cus / 8 : 1, L = (per_xcd + cu - 1) / cu;
  if (waves == 8) return (float)L * (0.60f + 0.17f * (float)tts);
  auto round_us = [&](int n) { return n ? 0.38f + (float)n * (0.24f + 0.09f * (float)tts) : 0.0f; };
  return (float)(L / 3) * round_us(3) + round_us(L % 3);
}

void seg_dense(const SegArgs &a, hipStream_t st) {
  static constexpr int kTiles[] = {2, 3, 4, 6, 8, 10};
  const int cus = jit::cu_count();
  int best = 10;
  float best_us = INFINITY;
  for (int t : kTiles) {
    const float us = seg_dense_step_us(t, t <= 4 ? 4 : 8, a.T, a.N, cus);
    if (us < best_us) {
      best_us = us;
      best = t;
    }
  }
  switch (best) {
    case 2: return seg_launch<false, true, SegShape<2, 4, 2, 2, 3>>(a, a.N, st);
    case 3: return seg_launch<false, true, SegShape<3, 4, 1, 2, 3>>(a, a.N, st);
    case 4: return seg_launch<false, true, SegShape<4, 4, 1, 2, 3>>(a, a.N, st);
    case 6: return seg_launch<false, true, SegShape<6, 8, 1, 2>>(a, a.N, st);
    case 8: return seg_launch<false, true, SegShape<8, 8, 1, 2>>(a, a.N, st);
    default: return seg_launch<false, true, SegShape<10, 8, 1, 2>>(a, a.N, st);
  }
}

}  // namespace

extern "C" int jit_moe_gate_up_swiglu_seg(const uint16_t *x, int K, const int32_t *pair_row,
                                          const int32_t *expert_cnt, const int32_t *expert_off, int E,
                                          const void *packed, int I, int P, uint16_t *h, void *stream) {
  if (K <= 0 || I <= 0 || E <= 0 || P < 0)
    return jit::fail(JIT_EINVAL, "moe_gate_up_seg: bad dims K=%d I=%d E=%d P=%d", K, I, E, P);
  if (K % 128 != 0 || I % 128 != 0)
    return jit::fail(JIT_EUNSUPPORTED, "moe_gate_up_seg covers K %% 128 == 0 and I %% 128 == 0, got K=%d I=%d", K,
                     I);
  if (P == 0) return JIT_OK;
  if (!x || !pair_row || !expert_cnt || !expert_off || !packed || !h)
    return jit::fail(JIT_EINVAL, "moe_gate_up_seg: null pointer");
  if ((long long)P * I * 2 >= (1LL << 31))
    return jit::fail(JIT_EUNSUPPORTED, "moe_gate_up_seg: h of %d x %d bf16 exceeds 2 GiB", P, I);
  const SegArgs a{x, pair_row, expert_cnt, expert_off, (const uint8_t *)packed, h, jit_q4_packed_bytes(1, 2 * I, K), K, I,
                  0, 0, E};
  seg_experts<true>(a, 2 * I, P, (hipStream_t)stream);
  return jit::check_launch("jit_moe_gate_up_swiglu_seg");
}

extern "C" int jit_moe_down_seg(const uint16_t *h, int I, const int32_t *expert_cnt, const int32_t *expert_off,
                                int E, const void *packed, int D, int P, uint16_t *r, void *stream) {
  if (I <= 0 || D <= 0 || E <= 0 || P < 0)
    return jit::fail(JIT_EINVAL, "moe_down_seg: bad dims I=%d D=%d E=%d P=%d", I, D, E, P);
  if (I % 128 != 0 || D % kSegRows != 0)
    return jit::fail(JIT_EUNSUPPORTED, "moe_down_seg covers I %% 128 == 0 and D %% %d == 0, got I=%d D=%d", kSegRows,
                     I, D);
  if (P == 0) return JIT_OK;
  if (!h || !expert_cnt || !expert_off || !packed || !r) return jit::fail(JIT_EINVAL, "moe_down_seg: null pointer");
  if ((long long)P * D * 2 >= (1LL << 31))
    return jit::fail(JIT_EUNSUPPORTED, "moe_down_seg: r of %d x %d bf16 exceeds 2 GiB", P, D);
  const SegArgs a{h, nullptr, expert_cnt, expert_off, (const uint8_t *)packed, r, jit_q4_packed_bytes(1, D, I), I, D, 0, 0,
                  E};
  seg_experts<false>(a, D, P, (hipStream_t)stream);
  return jit::check_launch("jit_moe_down_seg");
}

extern "C" int jit_qmm_seg(const uint16_t *x, int T, int K, const void *packed, int N, uint16_t *y, void *stream) {
  if (T < 0 || K <= 0 || N <= 0) return jit::fail(JIT_EINVAL, "qmm_seg: bad dims T=%d K=%d N=%d", T, K, N);
  if (K % 128 != 0 || N % kSegRows != 0)
    return jit::fail(JIT_EUNSUPPORTED, "qmm_seg covers K %% 128 == 0 and N %% %d == 0, got K=%d N=%d", kSegRows, K,
                     N);
  if (T == 0) return JIT_OK;
  if (!x || !packed || !y) return jit::fail(JIT_EINVAL, "qmm_seg: null pointer");
  if ((long long)T * N * 2 >= (1LL << 31))
    return jit::fail(JIT_EUNSUPPORTED, "qmm_seg: y of %d x %d bf16 exceeds 2 GiB", T, N);
  const SegArgs a{x, nullptr, nullptr, nullptr, (const uint8_t *)packed, y, 0, K, N, T, 0, 0};
  seg_dense(a, (hipStream_t)stream);
  return jit::check_launch("jit_qmm_seg");
}
