// Wide tiled expert kernels of the MoE layer (16-bit types): the two grouped SwiGLU contractions
// for batches in which an active expert sees hundreds of tokens.
//
// What bounds them: with random operands the card runs these contractions against its power
// limit (the walk below alone: 2150 TFLOP/s on zeros, 1480-1510 on random bf16; the matrix
// library 2120 and 1510; Mixtral's gate/up call of 8192 tokens 2539 us on zeros, 3059 on random
// data, at a clock of 1.75 GHz), so the rate follows the energy per multiply-add, most of which past
// the matrix cores is LDS and cache traffic. A workgroup of 4 waves owns a 256-row x 256-token
// output tile, alone on its CU, and each wave a 128 x 128 quarter of it with its accumulators
// in 256 AGPRs: per K step of 128 bytes it reads 128 KB from LDS where 8 waves of 128 x 64 read
// 192 KB (same loop, random bf16: 1500 against 1270 TFLOP/s) and the 256 x 128 tiles of
// tiles.hip 192 KB plus 64 KB of register staging. Mixtral, 8192 tokens, 256 x 128 -> 256 x 256
// tiles: gate/up 3607 -> 3060 us, down 1957 -> 1653 us (1257 and 1164 TFLOP/s; 2985 in another run).
//
// Both operands go straight into LDS (buffer_load ... lds, no registers), in two stages of
// 64 KB. One step is two halves, the step's two 64-byte k-groups. While the 64 MFMAs of one half
// run from registers, the fragments of the next half are read into the other register set; the
// DMA of the step after the next goes out one instruction per four MFMAs of the second half
// (issued as one burst it held up the wave's MFMAs). The step's only barrier stands between
// its halves: there every wave has read the whole stage (so that DMA may overwrite it), and
// the next step's DMA has landed.
//
// LDS layout of a stage: row q's 16-byte slot s at slot 8q + (s ^ (q % 8)); fragment reads (16
// rows at one slot) then have no bank conflicts (SQ_LDS_BANK_CONFLICT 0). A DMA instruction
// fills 64 consecutive slots (8 rows) in lane order, so lane l loads slot (l % 8) ^ (l / 8) of
// row l / 8.
//
// The MFMAs are written in assembly with the accumulator as a tied operand: with the builtin
// the register allocator permuted the accumulators over the loop's back edge (~200 AGPR moves
// per two steps; Mixtral 8192 tokens gate/up 3260 us against 2970). The waits that the
// compiler then does not know of (matrix result -> vector read, vector write -> matrix operand)
// are the two s_nop of the loop; no vector instruction stands between them.
//
// A token group's tiles are interleaved over the tile's token rows (tile = group + 2 j), so an
// item of fewer tokens runs fewer tiles per wave (2, 4, 6 or 8).
//
// The arithmetic and rounding points are those of the other expert kernels (and of
// stack_fused_moe, specmoe/layers/fused_moe_kernel.py:319-349); only the fp32 accumulation
// order over K differs.
#include <utility>

#include "expert_items.h"

namespace smx {

constexpr int kXWaves = 4;
constexpr int kXThreads = kXWaves * kWave;
constexpr int kXTokGroups = 2;                   // 2 row groups x 2 token groups of waves
constexpr int kXStep = 128;                      // K bytes per row per step
constexpr int kXSlots = kXStep / 16;             // 16-byte slots per row per step
constexpr int kXRows = 256;                      // weight rows per workgroup
constexpr int kXTiles = 8;                       // 16-row weight tiles per wave
constexpr int kXDmaRows = kXWaves * kWave / kXSlots;  // rows one DMA instruction of all waves fills
constexpr int kXDma = kXRows / kXDmaRows;        // weight DMA instructions per wave and step
constexpr int kXStage = kXRows * kXSlots;        // 16-byte slots per stage and operand
constexpr int kXBlock = 4;                       // token ranges of an expert run side by side

static_assert(kTileGateCols * 2 == kXRows && kTileDownRows == kXRows && kWideTok == kXRows, "the plan's tiles");
static_assert(kXTiles * kRowTile * kXWaves / kXTokGroups == kXRows, "the waves cover the weight rows");
static_assert(kWideTok == 2 * kTileTok, "a wide item is a pair of the routing's ranges");

// What a workgroup's K walk reads: a wave's DMA instruction j fills stage rows 32 j + 8 wave +
// l / 8, the weights' from page offset w_row0[j] + (per lane) w_off, the tokens' from t_off[j].
struct WideSrc {
  __amdgpu_buffer_rsrc_t w, t;
  uint32_t w_off;
  uint32_t w_row0[kXDma];
  uint32_t t_base;
  uint32_t t_off[kXDma];
  int rot, n;  // the walk's step c reads K step (c + rot) mod n
  __device__ __forceinline__ uint32_t at(int c) const {
    const int p = c + rot;
    return static_cast<uint32_t>(p >= n ? p - n : p) * kXStep;
  }
};

// One DMA instruction: 16 bytes per lane into the 64 slots at `lds`, in lane order.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, u32x4* lds, uint32_t lane_off, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds, 16, lane_off, off, 0, 0);
}

// DMA instruction J of a step (K offset kb): the weights', then the tokens'.
template <int J>
__device__ __forceinline__ void wide_dma(const WideSrc& s, u32x4* sa, u32x4* sb, int wave, uint32_t kb) {
  constexpr int j = J % kXDma;
  if constexpr (J < kXDma) dma16(s.w, sa + (j * kXWaves + wave) * kWave, s.w_off, s.w_row0[j] + kb);
  else dma16(s.t, sb + (j * kXWaves + wave) * kWave, s.t_off[j], s.t_base + kb);
}

template <int... Js>
__device__ __forceinline__ void wide_dma_all(const WideSrc& s, u32x4* sa, u32x4* sb, int wave, uint32_t kb,
                                             std::integer_sequence<int, Js...>) {
  (wide_dma<Js>(s, sa, sb, wave, kb), ...);
}

// A and B fragments of one half step.
template <int NT>
struct WideFrags {
  u32x4 a[kXTiles], b[NT];
};

// Stage slot of A tile i of a wave: tiles 0-3 in rows 0-127, 4-7 in rows 128-255.
__device__ __forceinline__ constexpr int wide_a_slot(int i) {
  return ((i < kXTiles / 2 ? 0 : kXRows / 2) + (i % (kXTiles / 2)) * kRowTile) * kXSlots;
}
__device__ __forceinline__ constexpr int wide_b_slot(int j) { return j * kXTokGroups * kTokTile * kXSlots; }

// acc += a . b in place (see the note at the top).
template <int DT>
__device__ __forceinline__ void mfma_acc(f32x4& acc, const u32x4& a, const u32x4& b) {
  if constexpr (DT == kBF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// `count` operations spread over `places`: those at place n are [spread(n), spread(n + 1)).
__device__ constexpr int spread(int n, int count, int places) {
  const int v = (n * count + places - 1) / places;
  return v < count ? v : count;
}

// The MFMAs of one half from `cur`. Between them, the next half's fragments are read into `nxt`
// from this lane's stage slots pa, pb (over the first three quarters of the MFMAs), and kDma
// operations `dma` are issued, evenly spread.
template <int DT, int NT, int kDma, typename F, int... Ns>
__device__ __forceinline__ void wide_half(const WideFrags<NT>& cur, WideFrags<NT>& nxt, const u32x4* pa,
                                          const u32x4* pb, f32x4 (&acc)[kXTiles][NT], F&& dma,
                                          std::integer_sequence<int, Ns...>) {
  constexpr int kM = kXTiles * NT, kR = kXTiles + NT, kRs = kM * 3 / 4;
  auto place = [&](auto nc) {
    constexpr int n = decltype(nc)::value;
    constexpr int r0 = spread(n, kR, kRs), r1 = spread(n + 1, kR, kRs);
#pragma unroll
    for (int q = r0; q < r1; ++q) {
      if (q < NT) nxt.b[q] = pb[wide_b_slot(q)];
      else nxt.a[q - NT] = pa[wide_a_slot(q - NT)];
    }
    constexpr int d0 = spread(n, kDma, kM), d1 = spread(n + 1, kDma, kM);
    static_assert(d1 - d0 <= 1, "at most one DMA instruction per MFMA");
    if constexpr (d0 < d1) dma(std::integral_constant<int, d0>{});
    mfma_acc<DT>(acc[n % kXTiles][n / kXTiles], cur.a[n % kXTiles], cur.b[n / kXTiles]);
    __builtin_amdgcn_sched_barrier(0);
  };
  (place(std::integral_constant<int, Ns>{}), ...);
}

// s_waitcnt: at most n vector-memory operations outstanding, and no LDS read.
constexpr int vm_lgkm0_imm(int n) { return (n & 15) | (7 << 4) | ((n >> 4) << 14); }

// Barrier without a memory fence (a fence would also wait for the DMAs of later steps).
__device__ __forceinline__ void wide_barrier() {
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

struct WideLane {
  int wave, wr, wt;
  int pa[2], pb[2];  // stage slots of the lane's fragments, k-group 0 / 1, tile 0
};

// One step from stage (sa, sb), the next one's stage being (na, nb): see the note at the top.
// kb: K offset of the step whose DMA goes out into (sa, sb).
template <int DT, int NT>
__device__ __forceinline__ void wide_step(const WideSrc& src, u32x4* sa, u32x4* sb, const u32x4* na,
                                          const u32x4* nb, const WideLane& ln, uint32_t kb,
                                          WideFrags<NT>& f0, WideFrags<NT>& f1, f32x4 (&acc)[kXTiles][NT]) {
  constexpr auto kSeq = std::make_integer_sequence<int, kXTiles * NT>{};
  wide_half<DT, NT, 0>(f0, f1, sa + ln.pa[1], sb + ln.pb[1], acc, [](auto) {}, kSeq);
  __builtin_amdgcn_s_waitcnt(vm_lgkm0_imm(0));
  wide_barrier();
  wide_half<DT, NT, kXDma + NT>(f1, f0, na + ln.pa[0], nb + ln.pb[0], acc,
                                [&](auto q) { wide_dma<decltype(q)::value>(src, sa, sb, ln.wave, kb); }, kSeq);
}

// acc += the wave's weight rows . its tokens over n K steps (n even, at least 2). Past the end the
// DMA reloads the last step (in bounds, into stages no later step reads) and the fragment reads
// take what the stage holds (unused), so the body has no branches.
template <int DT, int NT>
__device__ __forceinline__ void wide_walk(const WideSrc& src, u32x4* a0, u32x4* b0, u32x4* a1, u32x4* b1,
                                          const WideLane& ln, f32x4 (&acc)[kXTiles][NT]) {
  constexpr auto kDmas = std::make_integer_sequence<int, kXDma + NT>{};
  static_assert(NT * kXTokGroups * kTokTile == NT * kXDmaRows, "one token DMA instruction per token tile of a wave");
  const int l = src.n - 1;
  WideFrags<NT> f0, f1;
  wide_dma_all(src, a0, b0, ln.wave, src.at(0), kDmas);
  __builtin_amdgcn_sched_barrier(0);
  wide_dma_all(src, a1, b1, ln.wave, src.at(1), kDmas);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(vm_lgkm0_imm(kXDma + NT));
  wide_barrier();
#pragma unroll
  for (int j = 0; j < NT; ++j) f0.b[j] = b0[ln.pb[0] + wide_b_slot(j)];
#pragma unroll
  for (int i = 0; i < kXTiles; ++i) f0.a[i] = a0[ln.pa[0] + wide_a_slot(i)];
  __builtin_amdgcn_sched_barrier(0);
  for (int c = 0; c < src.n; c += 2) {
    asm volatile("s_nop 1");
    __builtin_amdgcn_sched_barrier(0);
    wide_step<DT, NT>(src, a0, b0, a1, b1, ln, src.at(min(c + 2, l)), f0, f1, acc);
    wide_step<DT, NT>(src, a1, b1, a0, b0, ln, src.at(min(c + 3, l)), f0, f1, acc);
    asm volatile("s_nop 15");
    __builtin_amdgcn_sched_barrier(0);
  }
}

__device__ __forceinline__ void wide_lane(WideLane& ln) {
  const int lane = lane_id();
  const int r = lane & 15, g = lane >> 4;
  ln.wave = wave_id();
  ln.wr = ln.wave / kXTokGroups;
  ln.wt = ln.wave % kXTokGroups;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int slot = (4 * u + g) ^ (r & 7);
    ln.pa[u] = (ln.wr * (kXTiles / 2) * kRowTile + r) * kXSlots + slot;
    ln.pb[u] = (ln.wt * kTokTile + r) * kXSlots + slot;
  }
}

// range_group with the ranges taken in blocks of at most kXBlock (of about equal size), each
// block's items over all weight groups before the next block's: the workgroups that run at one
// time on an XCD share a few token panels and a few weight panels. Without it an expert of 23
// ranges streamed 23 token panels at once (Mixtral 8192 tokens: 4910 -> 4885 us).
__device__ __forceinline__ void wide_range_group(int local, int per_item, int nr, int& r, int& g) {
  const int nb = (nr + kXBlock - 1) / kXBlock;
  const int size = (nr + nb - 1) / nb;
  const int blk = local / (size * per_item);
  range_group(local - blk * size * per_item, per_item, min(size, nr - blk * size), r, g);
  r += blk * size;
}

// The work item of workgroup blockIdx.x: up to kWideTok tokens, a pair of the routing's ranges of
// kTileTok sorted positions (the last of an expert may be single). The leading `shared_blocks`
// workgroups run the shared expert. A routed workgroup finds its pair among the range records by
// counting those that begin a pair (an even number of ranges into their expert): every lane
// looks at one record of each 64, one round of loads. False past the batch's pairs.
template <typename S>
__device__ __forceinline__ bool wide_item(const ExpertArgs& a, int shared_blocks, int per_item, WorkItem& w) {
  const int64_t elem = static_cast<int64_t>(sizeof(S));
  const int b = static_cast<int>(blockIdx.x);
  int r, g;
  if (b < shared_blocks) {
    const int nr = a.sh.tok_groups;
    wide_range_group(b, per_item, nr, r, g);
    w.page = static_cast<const char*>(a.sh.page);
    w.page_bytes = 3 * static_cast<int64_t>(a.H) * a.sh.I * elem;
    w.I = a.sh.I;
    w.off = r * kWideTok;
    w.m = min(kWideTok, a.T - w.off);
    w.tg = g;
    w.nr = nr;
    w.rot = g;
    w.shared = true;
    return true;
  }
  const int rb = b - shared_blocks;
  const int want = rb / per_item;
  const int nranges = uniform(a.rb.hdr[0]);
  int seen = 0, j = -1;
  for (int base = 0; base < nranges; base += kWave) {
    const int q = base + lane_id();
    const uint64_t mask = ballot(q < nranges && ((q - a.rb.ranges[min(q, nranges - 1)].j0) & 1) == 0);
    const int cnt = __popcll(mask);
    if (want < seen + cnt) {  // the (want - seen)-th set bit: the lane with that many below it
      const uint64_t below = mask & ((uint64_t{1} << lane_id()) - 1);
      const uint64_t hit = ballot(((mask >> lane_id()) & 1) && __popcll(below) == want - seen);
      j = base + __ffsll(static_cast<unsigned long long>(hit)) - 1;
      break;
    }
    seen += cnt;
  }
  if (j < 0) return false;
  j = uniform(j);
  const RangeRec& rr = a.rb.ranges[j];
  const int off = uniform(rr.off), cnt = uniform(rr.cnt), j0 = uniform(rr.j0);
  const int np = (uniform(rr.nr) + 1) / 2;
  wide_range_group(rb - (want - (j - j0) / 2) * per_item, per_item, np, r, g);
  w.page_bytes = a.page_elems * elem;
  w.page = static_cast<const char*>(a.pool) + uniform64(rr.slot) * w.page_bytes;
  w.I = a.I;
  w.off = off + r * kWideTok;
  w.m = min(kWideTok, cnt - r * kWideTok);
  w.tg = g;
  w.nr = np;
  w.rot = g;
  w.shared = false;
  return true;
}

// Start of a weight group's K walk over n steps: an eighth of the walk per group, so that the
// workgroups of different weight groups, which start together, read different K slices of
// their rows (the row pitches are multiples of 2 KB or 4 KB: at one K step the 256 rows of all
// groups lie on a few HBM channels). A group's token ranges share its order. Measured, without ->
// with: Mixtral 1025 tokens 1001 -> 956 us, Qwen1.5-MoE 3000 tokens 594 -> 574 us,
// DeepSeek-V2-Lite 2047 tokens 465 -> 458 us.
__device__ __forceinline__ int wide_rot(int g, int n) { return (g & 7) * n / 8; }

// Token rows of an item: position q of the range (clamped to the last one; rows past it are
// computed and discarded), per-lane offset of each DMA instruction.
__device__ __forceinline__ void wide_tokens(const ExpertArgs& a, const WorkItem& it, WideSrc& src, int wave,
                                            int64_t row_bytes, bool gather) {
  const int lane = lane_id();
  const uint32_t slot = static_cast<uint32_t>(((lane & 7) ^ (lane >> 3)) * 16);
  int row[kXDma];
#pragma unroll
  for (int j = 0; j < kXDma; ++j) row[j] = it.off + min(j * kXDmaRows + wave * 8 + (lane >> 3), it.m - 1);
  if (gather && !it.shared) {  // one round of loads, then the divisions
    const float rk = 1.0f / static_cast<float>(a.k);
#pragma unroll
    for (int j = 0; j < kXDma; ++j) row[j] = a.rb.sorted_f[row[j]];
#pragma unroll
    for (int j = 0; j < kXDma; ++j) row[j] = div_small(row[j], a.k, rk);
  }
#pragma unroll
  for (int j = 0; j < kXDma; ++j) src.t_off[j] = static_cast<uint32_t>(row[j] * row_bytes) + slot;
}

template <int NT>
__device__ __forceinline__ void wide_zero(f32x4 (&acc)[kXTiles][NT]) {
#pragma unroll
  for (int i = 0; i < kXTiles; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// Two floats rounded (to nearest even) to the activation type, packed; and back.
template <int DT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (DT == kBF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, f16x2));
}
// a.b elementwise, rounded to the activation type, packed. In fp16 with one rounding, from the exact
// product, as the other kernels' conversions of the same products compile to (v_fma_mixlo_f16);
// through pack2 it would be rounded to fp32 first, another bit in 3 of 100 000 products.
template <int DT>
__device__ __forceinline__ uint32_t mul2(const f32x2& a, const f32x2& b) {
  if constexpr (DT == kBF16) return pack2<DT>(a[0] * b[0], a[1] * b[1]);
  else return static_cast<uint32_t>(f32_to_f16(a[0] * b[0])) | static_cast<uint32_t>(f32_to_f16(a[1] * b[1])) << 16;
}
template <int DT>
__device__ __forceinline__ f32x2 unpack2(uint32_t v) {
  if constexpr (DT == kBF16) return f32x2{__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u)};
  else return __builtin_convertvector(__builtin_bit_cast(f16x2, v), f32x2);
}

// g / (1 + e^-g) for a gate that is a 16-bit value, in 15 operations (silu_f32, with expf and an IEEE
// division: ~30). e^-g = 2^hi * 2^lo with hi + lo = -g * log2(e) to twice the precision of hi (the
// remainder of the product by FMA, plus the constant's own remainder); x = 2^hi. The quotient by
// 1 + x is corrected once by its remainder, which takes 2^lo = 1 + lo * ln 2 with it: x itself is
// never rounded again. Numerator and denominator are in eighths, so that the reciprocal of the
// largest finite denominator is not subnormal. From |g| = 88.72, just below where e^-g overflows,
// the first quotient is the result: g itself where x is 0, -0 (NaN for -inf) where x is infinite,
// where lo has no meaning and the remainder would be inf * 0. (The remainder's sign keeps -0.)
// Against 64 bits over all bf16 | fp16 gates above -88.72, in units of 2^-23: largest 1.105 | 1.202,
// rms 0.1814 | 0.3414; silu_f32 1.105 | 1.203, 0.1824 | 0.3417; same results outside, NaN and
// infinities included. With one wave per SIMD nothing covers the epilogue's 128 values per lane,
// 4 cycles per operation. Per call, silu_f32's bits (expf, quotient corrected once) -> this: Mixtral
// 8192 tokens 4812 -> 4776 us, DeepSeek-V2-Lite layer of 2047 tokens 481 -> 475, a bf16 layer of
// hidden 1024 (ffn 2816, 8 experts) at 512 tokens 93.4 -> 91.4.
__device__ __forceinline__ float silu_16(float g) {
  const float hi = g * -1.44269504f;
  const float lo = fmaf(g, -1.92596299e-8f, fmaf(g, -1.44269504f, -hi));
  const float x = __builtin_amdgcn_exp2f(hi);
  const float d = fmaf(x, 0.125f, 0.125f);
  const float n = g * 0.125f;
  const float y = __builtin_amdgcn_rcpf(d);
  const float q = n * y;
  const float r = fmaf(x * (lo * 0.0866433976f), q, fmaf(d, q, -n));  // 0.0866...: ln 2 / 8
  return fabsf(g) < 88.72f ? fmaf(-r, y, q) : q;
}

// Rows of 16 lanes hold 4 consecutive columns each of two 16-column tiles of one output row: `a`
// (tile 0) and `b` (tile 1), packed. Swapping a's odd rows with b's even ones leaves 8 consecutive
// columns in every lane -- of tile g % 2, from column 8 (g / 2), g the row -- so that a store
// writes 16 bytes per lane and 64 contiguous bytes per output row instead of 8 and 32.
__device__ __forceinline__ u32x4 join_tiles(const u32x2& a, const u32x2& b) {
  const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false));
  const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false));
  return u32x4{lo[0], hi[0], lo[1], hi[1]};
}
// The lane's first column of a joined pair of tiles.
__device__ __forceinline__ int join_col(int lane) { return ((lane >> 4) & 1) * kRowTile + (lane >> 5) * 8; }

// A copy of an accumulator, made here: without the assembly the compiler moved all of a wave's 256
// accumulator registers to vector registers ahead of the branches of the epilogue, and spilled 14
// (DeepSeek-V2-Lite 2730 tokens down 189 -> 180 us without, Mixtral 8192 tokens 1707 -> 1692).
__device__ __forceinline__ f32x4 acc_read(const f32x4& acc) {
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(acc[e]));
    v[e] = x;
  }
  return v;
}

struct WideStages {
  u32x4 *a0, *b0, *a1, *b1;
};

template <int DT, int NT>
__device__ __forceinline__ void wide_gateup_item(const ExpertArgs& a, const WorkItem& it, const WideSrc& src,
                                                 const WideStages& st, const WideLane& ln) {
  using S = typename Elem<DT>::S;
  f32x4 acc[kXTiles][NT];
  wide_zero<NT>(acc);
  wide_walk<DT, NT>(src, st.a0, st.b0, st.a1, st.b1, ln, acc);
  S* act = static_cast<S*>(it.shared ? a.sh.act : a.act);
  const int lane = lane_id();
  const int col0 = it.tg * kTileGateCols + ln.wr * (kXTiles / 2) * kRowTile + join_col(lane);
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int q = (ln.wt + kXTokGroups * j) * kTokTile + (lane & 15);
    if (q >= it.m) continue;  // the same for the four lanes of an output row
    const int64_t row = static_cast<int64_t>(it.off + q) * it.I + col0;
#pragma unroll
    for (int i = 0; i < kXTiles / 2; i += 2) {
      u32x2 v[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const f32x4 gacc = acc[i + p][j], uacc = acc[i + p + kXTiles / 2][j];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const f32x2 gate = unpack2<DT>(pack2<DT>(gacc[2 * e], gacc[2 * e + 1]));
          const f32x2 up = unpack2<DT>(pack2<DT>(uacc[2 * e], uacc[2 * e + 1]));
          v[p][e] = mul2<DT>(f32x2{silu_16(gate[0]), silu_16(gate[1])}, up);
        }
      }
      *reinterpret_cast<u32x4*>(act + row + i * kRowTile) = join_tiles(v[0], v[1]);
    }
  }
}

template <int DT, int NT, bool kTerms>
__device__ __forceinline__ void wide_down_item(const ExpertArgs& a, const WorkItem& it, int sp, int h0, int rows,
                                               const WideSrc& src, const WideStages& st, const WideLane& ln) {
  using S = typename Elem<DT>::S;
  const int lane = lane_id();
  // the rows' assignments and weights, loaded before the walk: their two latencies pass under it
  int fs[NT];
  float ws[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int q = it.off + min((ln.wt + kXTokGroups * j) * kTokTile + (lane & 15), it.m - 1);
    fs[j] = it.shared ? q : a.rb.sorted_f[q];
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) ws[j] = kTerms ? a.w[fs[j]] : 0.0f;
  f32x4 acc[kXTiles][NT];
  wide_zero<NT>(acc);
  wide_walk<DT, NT>(src, st.a0, st.b0, st.a1, st.b1, ln, acc);
  float* part = it.shared ? a.sh.part : a.part;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int q = (ln.wt + kXTokGroups * j) * kTokTile + (lane & 15);
    if (q >= it.m) continue;
    const int f = fs[j];
    if constexpr (kTerms) {
      const f32x2 wf = {ws[j], ws[j]};
      S* dst = reinterpret_cast<S*>(part) + static_cast<int64_t>(f) * a.H + join_col(lane);
#pragma unroll
      for (int i = 0; i < kXTiles; i += 2) {
        const int h = h0 + wide_a_slot(i) / kXSlots + ln.wr * (kXTiles / 2) * kRowTile;
        u32x2 v[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const f32x4 d = acc_read(acc[i + p][j]);
          v[p] = u32x2{mul2<DT>(f32x2{d[0], d[1]}, wf), mul2<DT>(f32x2{d[2], d[3]}, wf)};
        }
        const u32x4 o = join_tiles(v[0], v[1]);
        if (h < a.H) *reinterpret_cast<u32x4*>(dst + h) = o;
      }
    } else {
      float* dst = part + (static_cast<int64_t>(sp) * rows + f) * a.H + 4 * (lane >> 4);
#pragma unroll
      for (int i = 0; i < kXTiles; ++i) {
        const int h = h0 + wide_a_slot(i) / kXSlots + ln.wr * (kXTiles / 2) * kRowTile;
        if (h < a.H) *reinterpret_cast<f32x4*>(dst + h) = acc[i][j];
      }
    }
  }
}

// The walk ends with reloads of its last step in flight, DMAs into its LDS stages: the wave waits
// for them before it ends, so that none lands in LDS that a later workgroup has been given.
__device__ __forceinline__ void wide_drain() { __builtin_amdgcn_s_waitcnt(vmcnt_imm(0)); }

// Wave token tiles of an item of m tokens, in quarters of the tile.
__device__ __forceinline__ int wide_quarters(int m) { return (m + kWideTok / 4 - 1) / (kWideTok / 4); }

// Workgroup = (pair of token ranges, 128 intermediate columns): stage rows 0-127 are the columns'
// gate rows (W1), 128-255 the matching up rows (W3 starts I rows later); a wave owns 64 columns
// of both for its token group and writes act = round(silu(round(gate)) * round(up)).
template <int DT>
__global__ __launch_bounds__(kXThreads, 1) void wide_gateup_kernel(ExpertArgs a) {
  using S = typename Elem<DT>::S;
  const bool in_shared = static_cast<int>(blockIdx.x) < a.sh.gateup_blocks;
  const int Iw = in_shared ? a.sh.I : a.I;
  WorkItem it;
  if (!wide_item<S>(a, a.sh.gateup_blocks, Iw / kTileGateCols, it)) return;
  __shared__ u32x4 a0[kXStage], a1[kXStage], b0[kXStage], b1[kXStage];
  const int lane = lane_id();
  WideLane ln;
  wide_lane(ln);
  const int64_t row_bytes = static_cast<int64_t>(a.H) * sizeof(S);
  WideSrc src;
  src.w = make_rsrc(it.page, static_cast<uint32_t>(it.page_bytes));
  src.w_off = static_cast<uint32_t>((lane >> 3) * row_bytes + ((lane & 7) ^ (lane >> 3)) * 16);
#pragma unroll
  for (int j = 0; j < kXDma; ++j) {
    const int q = j * kXDmaRows + ln.wave * 8;
    const int row = (q < kXRows / 2 ? 0 : it.I - kXRows / 2) + it.tg * kTileGateCols + q;
    src.w_row0[j] = static_cast<uint32_t>(row * row_bytes);
  }
  src.t = make_rsrc(a.x, static_cast<uint32_t>(a.T * row_bytes));
  src.t_base = 0;
  wide_tokens(a, it, src, ln.wave, row_bytes, true);
  src.n = static_cast<int>(row_bytes / kXStep);
  src.rot = wide_rot(it.rot, src.n);
  const WideStages st{a0, b0, a1, b1};
  switch (wide_quarters(it.m)) {
    case 1: wide_gateup_item<DT, 2>(a, it, src, st, ln); break;
    case 2: wide_gateup_item<DT, 4>(a, it, src, st, ln); break;
    case 3: wide_gateup_item<DT, 6>(a, it, src, st, ln); break;
    default: wide_gateup_item<DT, 8>(a, it, src, st, ln); break;
  }
  wide_drain();
}

// Workgroup = (pair of token ranges, 256 rows of W2, K split): fp32 partials part[split][f][h],
// summed by the combine; with one split the routed sums are whole, and the kernel rounds them
// times their routing weight (the combine's own rounding) and writes these terms at half the
// bytes, which the combine only adds (per call, fp32 partials -> terms, down + combine:
// DeepSeek-V2-Lite 2047 tokens 159 + 31 -> 153 + 20 us, Mixtral 8192 tokens 1742 + 122 -> 1716 +
// 48; since the epilogue no longer spills 146 + 20 and 1692 + 48). Rows past H (a multiple of 128) are clamped and not stored.
template <int DT, bool kTerms>
__global__ __launch_bounds__(kXThreads, 1) void wide_down_kernel(ExpertArgs a) {
  using S = typename Elem<DT>::S;
  const int rgroups = (a.H + kTileDownRows - 1) / kTileDownRows;
  const bool in_shared = static_cast<int>(blockIdx.x) < a.sh.down_blocks;
  const int splits = in_shared ? a.sh.splits : a.splits;
  const int split_steps = in_shared ? a.sh.split_steps : a.split_steps;  // 64-byte units
  WorkItem it;
  if (!wide_item<S>(a, a.sh.down_blocks, rgroups * splits, it)) return;
  __shared__ u32x4 a0[kXStage], a1[kXStage], b0[kXStage], b1[kXStage];
  const int lane = lane_id();
  WideLane ln;
  wide_lane(ln);
  const int sp = it.tg / rgroups;
  const int h0 = (it.tg - sp * rgroups) * kTileDownRows;
  const int rows = it.shared ? a.T : a.T * a.k;  // rows of act and of one split of part
  const int64_t row_bytes = static_cast<int64_t>(it.I) * sizeof(S);
  const int64_t k0 = static_cast<int64_t>(sp) * split_steps * kStepBytes;
  WideSrc src;
  src.w = make_rsrc(it.page, static_cast<uint32_t>(it.page_bytes));
  src.w_off = static_cast<uint32_t>((lane >> 3) * row_bytes + ((lane & 7) ^ (lane >> 3)) * 16);
  // W2 starts after W1 and W3 (2*I rows of H elements = 2*H rows of I elements)
#pragma unroll
  for (int j = 0; j < kXDma; ++j) {
    const int row = min(h0 + j * kXDmaRows + ln.wave * 8, a.H - 8);
    src.w_row0[j] = static_cast<uint32_t>((2 * static_cast<int64_t>(a.H) + row) * row_bytes + k0);
  }
  src.t = make_rsrc(it.shared ? a.sh.act : a.act, static_cast<uint32_t>(rows * row_bytes));
  src.t_base = static_cast<uint32_t>(k0);
  wide_tokens(a, it, src, ln.wave, row_bytes, false);
  src.n = split_steps * kStepBytes / kXStep;
  src.rot = wide_rot(it.rot, src.n);
  const WideStages st{a0, b0, a1, b1};
  auto item = [&](auto terms) {
    constexpr bool kT = decltype(terms)::value;
    switch (wide_quarters(it.m)) {
      case 1: wide_down_item<DT, 2, kT>(a, it, sp, h0, rows, src, st, ln); break;
      case 2: wide_down_item<DT, 4, kT>(a, it, sp, h0, rows, src, st, ln); break;
      case 3: wide_down_item<DT, 6, kT>(a, it, sp, h0, rows, src, st, ln); break;
      default: wide_down_item<DT, 8, kT>(a, it, sp, h0, rows, src, st, ln); break;
    }
  };
  if constexpr (kTerms) {
    if (!it.shared) item(std::true_type{});
    else item(std::false_type{});
  } else {
    item(std::false_type{});
  }
  wide_drain();
}

template <int DT>
static hipError_t wide_launch(int stage, const ExpertArgs& a, int pairs, hipStream_t s) {
  const int64_t eb = dtype_bytes(DT);
  // the walk consumes K steps in pairs, and the tiles cover whole 128-column groups: the plan
  // gives both (H and I are whole 256-byte chunks, split counts divide half the steps)
  auto odd = [](int64_t bytes) { return bytes <= 0 || bytes % (2 * kXStep) != 0; };
  if (stage == 0) {
    if (odd(a.H * eb) || a.I % kTileGateCols != 0 || a.sh.I % kTileGateCols != 0) return hipErrorInvalidValue;
    const int64_t blocks = tile_grid_blocks(0, a.H, a.I, a.sh.gateup_blocks, pairs, 1);
    wide_gateup_kernel<DT><<<static_cast<unsigned>(blocks), kXThreads, 0, s>>>(a);
  } else {
    if (odd(static_cast<int64_t>(a.split_steps) * kStepBytes) ||
        (a.sh.I > 0 && odd(static_cast<int64_t>(a.sh.split_steps) * kStepBytes)))
      return hipErrorInvalidValue;
    const int64_t blocks = tile_grid_blocks(1, a.H, a.I, a.sh.down_blocks, pairs, a.splits);
    if (a.w != nullptr && a.splits == 1)
      wide_down_kernel<DT, true><<<static_cast<unsigned>(blocks), kXThreads, 0, s>>>(a);
    else
      wide_down_kernel<DT, false><<<static_cast<unsigned>(blocks), kXThreads, 0, s>>>(a);
  }
  return hipGetLastError();
}

hipError_t launch_wide(int stage, int dtype, const ExpertArgs& a, int pairs, hipStream_t s) {
  if (a.rb.span != kTileTok) return hipErrorInvalidValue;
  switch (dtype) {
    case kF16: return wide_launch<kF16>(stage, a, pairs, s);
    case kBF16: return wide_launch<kBF16>(stage, a, pairs, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace smx
