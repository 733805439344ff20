// fp32 Linear (+ exact GELU) forward for gfx950 (MI355X):
//
//   Y[m, n] = act( sum_k X[m, k] * W[n, k] + bias[n] ),   all fp32
//
// - the projections of the fp32 encoder (reference transformer_opt/
// submission.py:484-508: packed QKV, output projection, FFN input with its
// GELU, FFN output) - on the bf16 matrix cores without giving up fp32
// accuracy.
//
// The fp32 MFMA runs at 1/16 of the bf16 rate (157 against 2517 TFLOP/s), so
// each operand is written as the sum of three bf16 numbers, which is exact
// (8 + 8 + 8 significant bits), and the product is formed from the six
// products of terms that matter: x0 w0, x0 w1, x1 w0, x1 w1, x0 w2, x2 w0 (the
// three left out come to at most 2^-24 of |x w|, of random sign: see
// bf16x3.h).  Products of bf16 pairs are exact in fp32, and the
// leading products and the five small ones have an fp32 accumulator each, so
// the leading sum is rounded K / 16 times instead of K / 2 times by the fp32
// MFMA.  Relative error against float64 (2-norm): 1.8e-7 at K = 1024 and
// 3.9e-7 at K = 4096, where the library's fp32 GEMM has 5.7e-7 and 1.15e-6.
// The ceiling is 2517 / 6 = 419 TFLOP/s; with N(0, 1) data the chip's power
// limit holds bf16 MFMAs to about 1.85 PFLOP/s, i.e. 308.
//
// What a bf16 split cannot carry - infinities, values that round to infinity,
// NaN - makes the sum NaN or infinite, and values below 2^-110, which lose
// bits, matter in results as small only: every result that is not finite, or
// not zero and below 2^-80, is recomputed from the fp32 operands (fp32 MFMA or
// fma), which gives what a plain fp32 product gives.
//
// For the tiled kernel W is split by a launch of its own (launch_split_weight),
// in MFMA fragment order: 6 bytes a weight, one contiguous 1 KB copy per
// fragment, no work on it in the main loop.  X is split in registers: 5.5 VALU
// operations per value, in the shadow of the MFMAs.
//
// Tiled kernel (one workgroup = 4 wavefronts, two workgroups per CU; a 128 x
// 128 tile): a wavefront owns 32 tokens x 128 features, as C^T = W . X^T with
// v_mfma_f32_32x32x16_bf16, so no X value is split twice in a workgroup and a
// lane ends holding one token and 4 consecutive features per register group.
// K advances in stages of 32 through a 2-deep LDS ring (X as fp32 rows of 128
// bytes, 16-byte chunks XOR-swizzled by row; W as packed), filled by LDS-DMA;
// operands are read half a k-step ahead and the barrier of a stage sits where
// its last fragments have been read.  The grid is persistent and copies the
// next tile's first stages during the current tile's last.
// Measured, against the library's fp32 GEMM and with the launch that makes W's
// terms: 8192 x 4096 x 1024 485 -> 329 - 338 us (the kernel alone 214 TFLOP/s at
// best; matrix pipe busy 70 % at the 1.7 GHz the power limit leaves), 8192 x 1024 x
// 4096 460 -> 315 us, 32768 x 1536 x 512 368 -> 270 - 277 us, and the GELU, a pass
// of its own of 39 us on the first, costs 6 us in the epilogue.
// 256-token tiles with one workgroup per CU ran 3-6 % slower (no second
// workgroup to cover the epilogue), 128 x 64 and 128 x 32 tiles 15-50 %.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

#include "bf16x3.h"
#include "ttk_common.h"

namespace ttk {
namespace {

constexpr int kFlThreads = 256;  // 4 wavefronts, one per SIMD
constexpr int kFlBK = 32;        // k per stage: 128-byte rows of X
constexpr int kFlTile = 128;     // tokens and features per tile
constexpr int kFlFrag = 1024;    // bytes of one fragment (32 rows x 16 k of one term)

#define TTK_FL_LDS(ptr) ((__attribute__((address_space(3))) void*)(ptr))

__device__ __forceinline__ void fl_dma16(const void* gbase, unsigned voff, unsigned lds) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(gbase), "s"(lds)
               : "memory", "m0");
#pragma clang diagnostic pop
}

// The six products kept, as (term of W, term of X): consecutive ones share an
// operand.  Number 2 is the product of the leading terms.
constexpr int kTermW[6] = {2, 1, 0, 0, 1, 0};
constexpr int kTermX[6] = {0, 0, 0, 1, 1, 2};

template <int N>
__device__ __forceinline__ void fl_vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Output tile of slot `slot`; false for a slot past the last tile of its XCD.
// Workgroups are dealt round-robin to the 8 XCDs, so the slots of one
// workgroup stay on one XCD, which gets a contiguous band of the tile grid
// (group_m token tiles x all feature tiles) and keeps its operands in its L2.
__device__ __forceinline__ bool fl_tile(const LinearF32Params& p, int slot, int& m0, int& n0) {
  const int q = slot >> 3;
  const int o = (slot & 7) * p.per_xcd + q;
  if (q >= p.per_xcd || o >= p.tiles) return false;
  const int span = p.group_m * p.tiles_n;
  const int band = o / span;
  const int first = band * p.group_m;
  const int gs = min(p.group_m, p.tiles_m - first);
  const int rem = o - band * span;
  m0 = (first + rem % gs) * kFlTile;
  n0 = (rem / gs) * kFlTile;
  return true;
}

template <bool GELU, bool BIAS>
__global__ __launch_bounds__(kFlThreads, 2) void linear_f32_kernel(LinearF32Params p) {
  constexpr int R = 2;                         // LDS ring depth
  constexpr int TN = kFlTile / 32;             // feature blocks of a wavefront
  constexpr int kXBytes = kFlTile * kFlBK * 4;
  constexpr int kWFrags = 6 * TN;              // W fragments of a stage
  constexpr int kStage = kXBytes + kWFrags * kFlFrag;
  constexpr int XC = 4;                        // X copies per wavefront per stage
  constexpr int WC = (kWFrags + 3) / 4;        // W copies per wavefront per stage
  constexpr int DMA = XC + WC;
  constexpr int STORES = 4 * TN;               // stores per wavefront per tile
  static_assert((R - 2) * DMA + STORES <= 63, "wait counts fit vmcnt");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[R * kStage];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31;
  const int h = lane >> 5;

  const int grid = static_cast<int>(gridDim.x);
  const int slot_end = 8 * p.per_xcd;
  const int last_fb = (p.N - 1) >> 5;          // last feature block of 32

  // The copy stream runs R stages ahead of the compute stream.  Past the last
  // tile it repeats its last stage (into ring slots that nobody reads any
  // more), so every stage issues the same number of copies.
  int slot = static_cast<int>(blockIdx.x), m0 = 0, n0 = 0;
  while (slot < slot_end && !fl_tile(p, slot, m0, n0)) slot += grid;
  if (slot >= slot_end) return;
  const int NS = p.K / kFlBK;
  int c_slot = slot, c_m0 = m0, c_n0 = n0, c_ks = 0;
  auto c_advance = [&]() __attribute__((always_inline)) {
    if (c_ks + 1 < NS) {
      ++c_ks;
      return;
    }
    int s = c_slot + grid, sm = 0, sn = 0;
    while (s < slot_end && !fl_tile(p, s, sm, sn)) s += grid;
    if (s < slot_end) {
      c_slot = s;
      c_m0 = sm;
      c_n0 = sn;
      c_ks = 0;
    }
  };

  // X copies: lane L of copy c fills row 32 c + 8 wave + L / 8 at physical
  // 16-byte chunk L % 8, which holds logical chunk (L % 8) ^ ((row >> 1) & 7).
  // W copies: one fragment each, as packed.
  const unsigned dchunk = static_cast<unsigned>((lane & 7) ^ (((wave & 1) << 2) | ((lane >> 4) & 3))) * 16u;
  const int drow = 8 * wave + (lane >> 3);
  const unsigned xpitch = static_cast<unsigned>(p.ldx) * 4u;
  const unsigned lane16 = lane * 16;
  const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<size_t>(TTK_FL_LDS(smem)));
  struct Copy {
    const float* x;
    const char* w;
    int xr;           // last row of X, counted from the tile's first
    int wb;           // last feature block of W, counted from the tile's first
    unsigned lds;     // LDS address of the ring slot
  };
  const int64_t wblock = static_cast<int64_t>(NS) * (6 * kFlFrag);  // bytes of a packed feature block
  auto c_stage = [&](unsigned ring) __attribute__((always_inline)) -> Copy {
    return Copy{p.x + static_cast<int64_t>(c_m0) * p.ldx + c_ks * kFlBK,
                static_cast<const char*>(p.wp) + (c_n0 >> 5) * wblock + static_cast<int64_t>(c_ks) * (6 * kFlFrag),
                p.M - 1 - c_m0, last_fb - (c_n0 >> 5), lds0 + ring};
  };
  auto issue_one = [&](const Copy& s, int c) __attribute__((always_inline)) {
    if (c < XC) {
      const int row = min(32 * c + drow, s.xr);
      fl_dma16(s.x, static_cast<unsigned>(__umul24(row, xpitch)) + dchunk, s.lds + wave * 1024 + c * 4096);
    } else {
      const int f = min(wave + 4 * (c - XC), kWFrags - 1);  // fragment of the stage
      const int fb = f / 6;
      const char* src = s.w + min(fb, s.wb) * wblock + (f - 6 * fb) * kFlFrag;
      fl_dma16(src, lane16, s.lds + kXBytes + f * kFlFrag);
    }
  };

  // Fragment addresses: X chunk 4 kk + 2 h + j of row r is stored at
  // chunk ^ ((r >> 1) & 7); W fragments are lane-ordered.
  const int swz = (r32 >> 1) & 7;
  unsigned xfrag[2][2];  // [k-step of the stage][16-byte half]
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      xfrag[kk][j] = (32 * wave + r32) * 128 + 16 * ((4 * kk + 2 * h + j) ^ swz);

  f32x4 rx[2];            // next k-step's X, fp32
  Split8 px[2];           // split X of this and the next k-step
  Split8 pw[TN];          // W
  f32x16 hi[TN], lo[TN];  // sums of the leading and of the other products

  auto load_x = [&](unsigned ring, int kk) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j) rx[j] = *reinterpret_cast<const f32x4*>(smem + (ring + xfrag[kk][j]));
  };
  auto load_w = [&](Split8& d, unsigned ring, int kk, int i, int t) __attribute__((always_inline)) {
    d.t[t] = *reinterpret_cast<const u32x4*>(smem + (ring + lane16) + kXBytes + (6 * i + 3 * kk + t) * kFlFrag);
  };

  // One k-step (P: which of its stage) in two groups of two feature blocks,
  // six products each, the blocks interleaved.  Group 0 reads the W fragments
  // of group 1; group 1 reads those of the next k-step's group 0 and the next
  // k-step's X, and splits it.  So after group 0 of a stage's second k-step
  // nobody reads that stage any more, and what follows is read from stage S +
  // 1: `between` waits for it there, and group 1 then issues the copies of
  // stage S + R into the freed ring slot.
  auto kstep = [&](auto zero, auto step, unsigned ring, auto&& between) __attribute__((always_inline)) {
    constexpr int P = decltype(step)::value;
    unsigned nring = ring;
    Copy copy{};
#pragma unroll
    for (int g = 0; g < 24; ++g) {
      const int grp = g / 12, t = g % 12, pr = t / 2, i = 2 * grp + t % 2;
      if (g == 12) {
        if constexpr (P == 1) {
          between(nring, copy);
        }
        load_x(nring, P ^ 1);
      }
      const u32x4& a = pw[i].t[kTermW[pr]];
      const u32x4& b = px[P].t[kTermX[pr]];
      if (pr == 2) {
        hi[i] = mfma_x3(a, b, decltype(zero)::value ? f32x16{} : hi[i]);
      } else {
        lo[i] = mfma_x3(a, b, decltype(zero)::value && pr == 0 ? f32x16{} : lo[i]);
      }
      if (t < 6) {
        if (grp == 0) load_w(pw[2 + t / 3], ring, P, 2 + t / 3, t % 3);
        else load_w(pw[t / 3], nring, P ^ 1, t / 3, t % 3);
      }
      // The pair splits start once their operands have arrived.
      if (grp == 1 && t >= 4 && t % 2 == 1) {
        const int u = (t - 5) / 2;
        split_pair(px[P ^ 1], u, rx[u >> 1][2 * (u & 1)], rx[u >> 1][2 * (u & 1) + 1]);
      }
      if (P == 1 && grp == 1) {
        static_assert(DMA <= 12, "at most one copy per MFMA");
        if (t * DMA / 12 < (t + 1) * DMA / 12) issue_one(copy, t * DMA / 12);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Bias, activation and store of the wavefront's rows.
  auto epilogue = [&](int tm0, int tn0) __attribute__((always_inline)) {
    int el = lane;
    asm volatile("" : "+v"(el));
    const int eh = el >> 5, er = el & 31;
    const int rows = min(p.M - tm0, kFlTile);
    const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(
        p.y + static_cast<int64_t>(tm0) * p.ldy, static_cast<short>(0),
        static_cast<int>(static_cast<unsigned>((rows - 1) * p.ldy + p.N) * 4u), 0x00020000);
    auto put = [&](int i, int g, f32x4 v) __attribute__((always_inline)) {
      const int f = tn0 + 32 * i + 8 * g + 4 * eh;
      if constexpr (GELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_exact(v[e]);
      }
      const int m = 32 * wave + er;
      const unsigned off = (m < rows && f < p.N)
          ? (static_cast<unsigned>(m) * static_cast<unsigned>(p.ldy) + static_cast<unsigned>(f)) * 4u
          : 0x80000000u;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), yrsrc, static_cast<int>(off), 0, 0);
    };
    // The bias is one more product per feature block: its three terms in k
    // slots 0..2 of lane half 0, times ones.
    if constexpr (BIAS) {
      float bias[TN];
#pragma unroll
      for (int i = 0; i < TN; ++i) bias[i] = p.bias[min(tn0 + 32 * i + er, p.N - 1)];
      const u32x4 ones = {eh ? 0u : 0x3f803f80u, eh ? 0u : 0x00003f80u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const float b1 = bias[i] - high_half(bias[i]);
        const float b2 = b1 - high_half(b1);
        const u32x4 terms = {pack_high(bias[i], b1), __float_as_uint(b2) >> 16, 0u, 0u};
        lo[i] = mfma_x3(terms, ones, lo[i]);
      }
    }
    RedoWatch watch;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = hi[i][4 * g + e] + lo[i][4 * g + e];
          watch.see(v[e]);
        }
        put(i, g, v);
        __builtin_amdgcn_sched_barrier(0);
      }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(watch.any()) != 0, 0)) {
      fl_vm_wait<0>();
#pragma unroll 1
      for (int i = 0; i < TN; ++i) {
        const float* wrow = p.w + static_cast<int64_t>(min(tn0 + 32 * i + er, p.N - 1)) * p.ldw + eh;
        const float* xrow = p.x + static_cast<int64_t>(min(tm0 + 32 * wave + er, p.M - 1)) * p.ldx + eh;
        f32x16 acc{};
#pragma unroll 1
        for (int k = 0; k < p.K; k += 2) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wrow[k], xrow[k], acc, 0, 0, 0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 v = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
          if constexpr (BIAS) v += *reinterpret_cast<const f32x4*>(p.bias + min(tn0 + 32 * i + 8 * g + 4 * eh, p.N - 4));
          put(i, g, v);
        }
      }
    }
  };

  // Prologue: copies of the first R stages; the operands of k-step 0.
#pragma unroll 1
  for (int s = 0; s < R; ++s) {
    const Copy copy = c_stage(s * kStage);
#pragma unroll
    for (int c = 0; c < DMA; ++c) issue_one(copy, c);
    c_advance();
  }
  fl_vm_wait<(R - 1) * DMA>();
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 3; ++t) load_w(pw[i], 0, 0, i, t);
  load_x(0, 0);
#pragma unroll
  for (int u = 0; u < 4; ++u) split_pair(px[0], u, rx[u >> 1][2 * (u & 1)], rx[u >> 1][2 * (u & 1) + 1]);

  constexpr std::integral_constant<int, 0> kStep0{};
  constexpr std::integral_constant<int, 1> kStep1{};
  unsigned ring = 0;    // slot of the current stage
  int since = R;        // stages since the last epilogue
  for (;;) {
    auto stage = [&](auto zero) __attribute__((always_inline)) {
      kstep(zero, kStep0, ring, [](unsigned&, Copy&) {});
      kstep(std::false_type{}, kStep1, ring, [&](unsigned& nring, Copy& copy) __attribute__((always_inline)) {
        // Stage S + 1 has to be in LDS, and every wavefront done reading
        // stage S.  Younger than stage S + 1's copies: those of S + 2 .. S +
        // R - 1, and the stores of an epilogue less than R - 1 stages ago.
        if (since < R - 1) {
          fl_vm_wait<(R - 2) * DMA + STORES>();
        } else {
          fl_vm_wait<(R - 2) * DMA>();
        }
        ++since;
        __syncthreads();
        copy = c_stage(ring);
        nring = ring == static_cast<unsigned>((R - 1) * kStage) ? 0u : ring + kStage;
      });
      ring = ring == static_cast<unsigned>((R - 1) * kStage) ? 0u : ring + kStage;
      c_advance();
    };
    stage(std::true_type{});
    for (int s = 1; s < NS; ++s) stage(std::false_type{});
    epilogue(m0, n0);
    since = 0;
    slot += grid;
    while (slot < slot_end && !fl_tile(p, slot, m0, n0)) slot += grid;
    if (slot >= slot_end) break;
  }
  fl_vm_wait<0>();
}

// Tile o of the small form: bands of group_m rows of tiles.
template <int TB>
__device__ __forceinline__ void small_tile(const LinearF32Params& p, int o, int& m0, int& n0) {
  const int span = p.group_m * p.tiles_n;
  const int first = o / span * p.group_m;
  const int gs = min(p.group_m, p.tiles_m - first);
  const int rem = o % span;
  m0 = (first + rem % gs) * (32 * TB);
  n0 = rem / gs * (32 * TB);
}

// Stores chunk c of the tile at (m0, n0) from its sums: bias, activation, and
// the fp32 operands again where three terms did not do.
template <int TB, bool GELU, bool BIAS>
__device__ __forceinline__ void small_result(const LinearF32Params& p, int m0, int n0, int c, int lane, f32x4 v) {
  const int i = c / (4 * TB), j = (c >> 2) % TB, g = c & 3;
  const int m = m0 + 32 * j + (lane & 31), f = n0 + 32 * i + 8 * g + 4 * (lane >> 5);
  bool redo = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) redo |= redo_x3(v[e]);
  if (m >= p.M || f >= p.N) return;
  if (__builtin_expect(redo, 0)) {
    const float* xr = p.x + static_cast<int64_t>(m) * p.ldx;
#pragma unroll 1
    for (int e = 0; e < 4; ++e) {
      const float* wr = p.w + static_cast<int64_t>(f + e) * p.ldw;
      float a = 0.0f;
#pragma unroll 1
      for (int k = 0; k < p.K; ++k) a = __builtin_fmaf(wr[k], xr[k], a);
      v[e] = a;
    }
  }
  if constexpr (BIAS) v += *reinterpret_cast<const f32x4*>(p.bias + f);
  if constexpr (GELU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = gelu_exact(v[e]);
  }
  *reinterpret_cast<f32x4*>(p.y + static_cast<int64_t>(m) * p.ldy + f) = v;
}

// Small products: one workgroup of NW wavefronts per TB*32 x TB*32 tile, the
// wavefronts splitting K; X and W are both split in registers, so that no terms
// of W have to be made first (a launch of 2.4 us for 256 x 256 weights, 7.5 us
// for 1024 x 4096).  Each wavefront copies its k-steps' 64-byte row pieces by
// LDS-DMA into a ring of its own (no barriers), four lanes a piece: fragments
// loaded straight into registers have every lane in another row, and the L1
// served one of them per cycle (230 cycles a k-step and CU in 32 x 32 tiles,
// 512 in 64 x 64).  Row r's 16-byte chunk c sits at c ^ ((r >> 2) & 3), so the
// 16 rows of a fragment read cover all banks.  The wavefronts' sums are added
// in order through LDS.
// Eight wavefronts, which fill a CU's LDS, or four where two tiles of 32 x 32
// share a CU or K is short: 512 x 1024 x 256 8.0 -> 6.1 us, 512 x 512 x 64 3.9
// -> 3.5; 64 x 1024 x 1024 takes 7.5 with eight and 10.1 with four.
// Fragments in registers -> here: 64 x 1024 x 4096 31 -> 20 us, 256 x 1024 x
// 1024 10.9 -> 9.6, 512 x 1024 x 1024 18.9 -> 14.4, 1024 x 1024 x 1024 21.5 ->
// 18.5, 256 x 256 x 1024 10.0 -> 7.6, 256 x 256 x 256 4.8 -> 4.3.  Bound by the splits' VALU work
// and the MFMAs one after the other (2600 cycles a k-step and SIMD in 64 x 64
// tiles, 1536 of them MFMA): the next k-step's splits between this one's MFMAs
// gained 5 - 13 % from K = 2048 up in few tiles and lost 5 - 20 % elsewhere.
// Few tiles of long K left most CUs idle and one CU reading up to 1 MB of W:
// there p.splits workgroups share a tile's K, each writing its sums to the
// workspace, and linear_f32_join_kernel adds them in order (a launch of its own,
// 2 us in a graph: the kernel boundary makes the sums visible, and nothing has
// to be zeroed before).  In a graph, weights cold in the caches: 16 x 2048 x
// 8192 53 -> 22 us (the library's fp32 GEMM 23), 64 x 2048 x 8192 55 -> 28 (42),
// 16 x 1024 x 4096 27 -> 11 (12), 64 x 1024 x 4096 29 -> 14 (12), 16 x 768 x
// 3072 22 -> 9.3 (11), 16 x 2048 x 2048 16 -> 10.5 (12).
template <int TB, int NW, bool GELU, bool BIAS>
__global__ __launch_bounds__(64 * NW, 2) void linear_f32_small_kernel(LinearF32Params p) {
  constexpr int R = TB == 1 ? 4 : 2;           // ring depth
  constexpr int kHalf = 32 * TB * 64;          // X (then W) of a k-step: rows of 64 bytes
  constexpr int kRing = R * 2 * kHalf;
  constexpr int XC = kHalf / 1024;             // copies of X (and of W) per k-step
  static_assert(TB * TB * 4096 <= kRing, "a wavefront's sums fit its ring");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NW * kRing];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31;
  const int h = lane >> 5;
  // Workgroups are dealt round-robin to the 8 XCDs: each gets a contiguous run
  // of tiles, in bands of group_m rows of tiles, and keeps their operands in
  // its L2 (up to 10 % from two rounds of tiles on).
  const int unit = static_cast<int>(blockIdx.x >> 3);
  const int o = static_cast<int>(blockIdx.x & 7) * p.per_xcd + unit / p.splits;
  if (o >= p.tiles) return;
  const int part = unit % p.splits;  // of the tile's K
  int m0, n0;
  small_tile<TB>(p, o, m0, n0);
  const int KQ = p.K / 16;
  const int share = part * NW + wave, shares = p.splits * NW;
  const int q0 = static_cast<int>(static_cast<int64_t>(KQ) * share / shares);
  const int q1 = static_cast<int>(static_cast<int64_t>(KQ) * (share + 1) / shares);

  // Copy c fills rows 16 c .. + 15; rows past the last repeat it.
  const unsigned chunk = static_cast<unsigned>((lane & 3) ^ ((lane >> 4) & 3)) * 16u;
  unsigned xoff[XC], woff[XC];
#pragma unroll
  for (int c = 0; c < XC; ++c) {
    const int row = 16 * c + (lane >> 2);
    xoff[c] = static_cast<unsigned>(__umul24(min(row, p.M - 1 - m0), static_cast<unsigned>(p.ldx) * 4u)) + chunk;
    woff[c] = static_cast<unsigned>(__umul24(min(row, p.N - 1 - n0), static_cast<unsigned>(p.ldw) * 4u)) + chunk;
  }
  const float* xbase = p.x + static_cast<int64_t>(m0) * p.ldx;
  const float* wbase = p.w + static_cast<int64_t>(n0) * p.ldw;
  unsigned char* const ring = smem + wave * kRing;
  const unsigned ring_lds = static_cast<unsigned>(reinterpret_cast<size_t>(TTK_FL_LDS(smem))) + wave * kRing;
  auto issue = [&](int q, int slot) __attribute__((always_inline)) {
    const int k = 16 * q;
#pragma unroll
    for (int c = 0; c < XC; ++c) fl_dma16(xbase + k, xoff[c], ring_lds + slot * (2 * kHalf) + c * 1024);
#pragma unroll
    for (int c = 0; c < XC; ++c) fl_dma16(wbase + k, woff[c], ring_lds + slot * (2 * kHalf) + kHalf + c * 1024);
  };
  // This lane's 8 values of row 32 b + r32, k = 8 h .. + 7, from row block `at`.
  auto read_split = [&](Split8& d, const unsigned char* at) __attribute__((always_inline)) {
    f32x4 v[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
      v[j] = *reinterpret_cast<const f32x4*>(at + r32 * 64 + 16 * ((2 * h + j) ^ ((r32 >> 2) & 3)));
#pragma unroll
    for (int u = 0; u < 4; ++u) split_pair(d, u, v[u >> 1][2 * (u & 1)], v[u >> 1][2 * (u & 1) + 1]);
  };

  f32x16 hi[TB][TB], lo[TB][TB];
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int j = 0; j < TB; ++j) hi[i][j] = lo[i][j] = f32x16{};
  if (q0 < q1) {
#pragma unroll
    for (int s = 0; s < R - 1; ++s)
      if (q0 + s < q1) issue(q0 + s, s);
    int slot = 0;
    for (int q = q0; q < q1; ++q) {
      // K-step q has to be in LDS (younger: the copies of q + 1 .. q + R - 2, or
      // up to the last), and the reads of k-step q - 1, whose slot is filled
      // next, done.
      if (q + R - 2 < q1) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((R - 2) * 2 * XC) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      }
      if (q + R - 1 < q1) issue(q + R - 1, slot == 0 ? R - 1 : slot - 1);
      const unsigned char* at = ring + slot * (2 * kHalf);
      Split8 x[TB], w[TB];
#pragma unroll
      for (int b = 0; b < TB; ++b) {
        read_split(x[b], at + b * 2048);
        read_split(w[b], at + kHalf + b * 2048);
      }
#pragma unroll
      for (int pr = 0; pr < 6; ++pr)
#pragma unroll
        for (int j = 0; j < TB; ++j)
#pragma unroll
          for (int i = 0; i < TB; ++i) {
            f32x16& c = pr == 2 ? hi[i][j] : lo[i][j];
            c = mfma_x3(w[i].t[kTermW[pr]], x[j].t[kTermX[pr]], c);
          }
      slot = slot == R - 1 ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  f32x4* const sums = reinterpret_cast<f32x4*>(ring) + lane;  // of this wavefront, 64 to a chunk
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int j = 0; j < TB; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = hi[i][j][4 * g + e] + lo[i][j][4 * g + e];
        sums[((i * TB + j) * 4 + g) * 64] = v;
      }
  __syncthreads();
#pragma unroll
  for (int c = wave; c < TB * TB * 4; c += NW) {
    const f32x4* sum = reinterpret_cast<const f32x4*>(smem) + c * 64 + lane;
    f32x4 v = sum[0];
#pragma unroll
    for (int s = 1; s < NW; ++s) v += sum[s * (kRing / 16)];
    if (p.splits > 1) {
      static_cast<f32x4*>(p.part)[((static_cast<int64_t>(part) * p.tiles + o) * (TB * TB * 4) + c) * 64 + lane] = v;
    } else {
      small_result<TB, GELU, BIAS>(p, m0, n0, c, lane, v);
    }
  }
}

// The results of tiles whose K several workgroups share: their sums, added in
// order.  One wavefront per chunk of 64 x 4 results.
template <int TB, bool GELU, bool BIAS>
__global__ __launch_bounds__(kFlThreads) void linear_f32_join_kernel(LinearF32Params p) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int o = static_cast<int>(blockIdx.x) / (TB * TB);
  const int c = static_cast<int>(blockIdx.x) % (TB * TB) * 4 + wave;
  int m0, n0;
  small_tile<TB>(p, o, m0, n0);
  const f32x4* sum = static_cast<const f32x4*>(p.part) + (static_cast<int64_t>(o) * (TB * TB * 4) + c) * 64 + lane;
  const int64_t step = static_cast<int64_t>(p.tiles) * (TB * TB * 4) * 64;
  f32x4 v = sum[0];
#pragma unroll 4
  for (int s = 1; s < p.splits; ++s) v += sum[s * step];
  small_result<TB, GELU, BIAS>(p, m0, n0, c, lane, v);
}

template <int TB, int NW>
hipError_t launch_small(LinearF32Params& p, const LinearF32Plan& plan, void* workspace, bool gelu,
                        hipStream_t stream) {
  p.tiles_n = (p.N - 1) / (32 * TB) + 1;
  p.tiles_m = (p.M - 1) / (32 * TB) + 1;
  p.tiles = p.tiles_m * p.tiles_n;
  p.per_xcd = (p.tiles + 7) / 8;
  // A band is as square as an XCD's share allows.
  p.group_m = 1;
  while (2 * p.group_m <= p.tiles_m && 4 * p.group_m * p.group_m <= p.per_xcd) p.group_m *= 2;
  p.splits = plan.splits;
  p.part = workspace;
  auto launch = [&](auto gelu_tag, auto bias_tag) {
    constexpr bool G = decltype(gelu_tag)::value, B = decltype(bias_tag)::value;
    const dim3 grid(8 * static_cast<unsigned>(p.per_xcd) * static_cast<unsigned>(p.splits));
    linear_f32_small_kernel<TB, NW, G, B><<<grid, dim3(64 * NW), 0, stream>>>(p);
    if (p.splits > 1) {
      linear_f32_join_kernel<TB, G, B><<<dim3(static_cast<unsigned>(p.tiles) * TB * TB), dim3(kFlThreads), 0, stream>>>(p);
    }
    return hipGetLastError();
  };
  if (gelu) return p.bias ? launch(std::true_type{}, std::true_type{}) : launch(std::true_type{}, std::false_type{});
  return p.bias ? launch(std::false_type{}, std::true_type{}) : launch(std::false_type{}, std::false_type{});
}

int fl_cu_count() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

hipError_t launch_tiled(LinearF32Params& p, bool gelu, hipStream_t stream) {
  p.tiles_m = (p.M - 1) / kFlTile + 1;
  p.tiles_n = (p.N - 1) / kFlTile + 1;
  p.tiles = p.tiles_m * p.tiles_n;
  p.per_xcd = (p.tiles + 7) / 8;
  p.group_m = std::max(1, std::min(p.tiles_m, p.per_xcd / p.tiles_n));
  const int slots = fl_cu_count() / 8 * 8 * 2;  // two workgroups per CU
  const dim3 grid(static_cast<unsigned>(std::max(8, std::min(slots, 8 * p.per_xcd)))), blk(kFlThreads);
  if (gelu) {
    if (p.bias) linear_f32_kernel<true, true><<<grid, blk, 0, stream>>>(p);
    else linear_f32_kernel<true, false><<<grid, blk, 0, stream>>>(p);
  } else {
    if (p.bias) linear_f32_kernel<false, true><<<grid, blk, 0, stream>>>(p);
    else linear_f32_kernel<false, false><<<grid, blk, 0, stream>>>(p);
  }
  return hipGetLastError();
}

// W [N, K] fp32 into its three bf16 terms, in MFMA fragment order: 16-byte
// chunk ((fb * K/16 + q) * 3 + t) * 64 + l holds term t of
// W[32 fb + l % 32][16 q + 8 (l / 32) .. + 7]; rows past N are zero.
__global__ __launch_bounds__(256) void split_weight_kernel(const float* w, u32x4* wp, int N, int K, int64_t ldw) {
  const int kq = K / 16;
  const int64_t items = static_cast<int64_t>((N + 31) / 32) * kq * 64;
  for (int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; c < items;
       c += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int l = static_cast<int>(c & 63);
    const int64_t frag = c >> 6;
    const int q = static_cast<int>(frag % kq);
    const int64_t n = 32 * (frag / kq) + (l & 31);
    const int64_t k = 16 * static_cast<int64_t>(q) + 8 * (l >> 5);
    f32x4 v[2] = {};
    if (n < N) {
      v[0] = *reinterpret_cast<const f32x4*>(w + n * ldw + k);
      v[1] = *reinterpret_cast<const f32x4*>(w + n * ldw + k + 4);
    }
    Split8 t;
#pragma unroll
    for (int d = 0; d < 4; ++d) split_pair(t, d, v[d >> 1][2 * (d & 1)], v[d >> 1][2 * (d & 1) + 1]);
#pragma unroll
    for (int i = 0; i < 3; ++i) wp[(frag * 3 + i) * 64 + l] = t.t[i];
  }
}

}  // namespace

namespace {

double tile_count(double M, double N, double side) { return std::ceil(M / side) * std::ceil(N / side); }

// Wavefronts of a 32 x 32 tile (see linear_f32_small_kernel).
bool four_wavefronts(int64_t M, int64_t N, int64_t K) { return K <= 64 || tile_count(M, N, 32.0) > fl_cu_count(); }

}  // namespace

LinearF32Plan plan_linear_f32(int64_t M, int64_t N, int64_t K, int64_t ldw, bool terms_ready) {
  const LinearF32Plan tiled = {LinearF32Form::kTiles128, 1, terms_ready ? 0 : (N + 31) / 32 * 32 * K * 6};
  if (ldw >= int64_t{1} << 22) return tiled;
  // The form with the least expected time (us), from the measured (256 CUs)
  // times of the three over products from 1 x 256 x 256 to 8192 x 4096 x 1024:
  // a launch's fixed cost and the chain of k-steps in one round of tiles, which
  // runs slower the more CUs have a tile, or whole rounds (of two 32 x 32 tiles
  // a CU); for the tiled form also the launch that makes W's terms, unless they
  // are there.  E.g. 256 x 256 x 256: 4.3 us for 32 x 32 tiles, 7.0 for 64 x
  // 64, 15.2 for 128 x 128; 512 x 1024 x 1024: 14.4, 15.7, 46; 1024 x 1024 x
  // 1024: 25.6, 18.5, 45; 4096 x 1024 x 1024: 88, 65, 54.
  const int64_t cu_count = fl_cu_count();
  const double cus = static_cast<double>(cu_count);
  const double m = static_cast<double>(M), n = static_cast<double>(N), k = static_cast<double>(K);
  const double n32 = tile_count(m, n, 32.0), n64 = tile_count(m, n, 64.0), n128 = tile_count(m, n, 128.0);
  const double r64 = std::ceil(n64 / cus), r128 = std::min(std::ceil(n128 / cus), 1.12 * n128 / cus);
  auto one32 = [&](double tiles, double depth) { return 3.0 + depth / 250.0 + tiles / cus * (0.3 + depth / 700.0); };
  auto one64 = [&](double tiles, double depth) { return 4.5 + depth / 113.0 + tiles / cus * (0.9 + depth / 230.0); };
  double t32 = n32 > cus ? 2.4 + std::ceil(n32 / (2.0 * cus)) * (1.6 + k / 100.0) : one32(n32, k);
  double t64 = r64 > 1.0 ? 2.5 + r64 * (3.2 + k / 78.0) : one64(n64, k);
  double t128 = 5.0 + k / kFlBK * (n128 > cus ? 1.37 * r128 : 0.85 + 0.52 * n128 / cus);
  if (!terms_ready) t128 += 3.0 + n * k / 0.6e6;
  int s32 = 1, s64 = 1;
  if (!terms_ready) {
    // Several workgroups to a tile, where tiles leave CUs idle: at least two
    // k-steps a wavefront, a CU each on the tile's XCD, and the launch that
    // joins their sums.  (Among 2 .. 32 workgroups to a tile and both tile
    // sizes, the choice came within 5 % of the best one over 16 .. 512 rows of
    // the projections of d = 256 .. 2048, a few at 10 %.)
    for (int s = 2; s * 256 <= K; ++s) {
      const double join = 2.5 + s * m * n / 0.5e6;
      auto fits = [&](double tiles) { return s * ((static_cast<int64_t>(tiles) + 7) / 8) <= cu_count / 8; };
      if (!fits(n64)) break;
      if (const double t = one64(s * n64, k / s) + join; t < t64) t64 = t, s64 = s;
      if (!fits(n32)) continue;
      if (const double t = one32(s * n32, k / s) + join; t < t32) t32 = t, s32 = s;
    }
  }
  // The small forms have a workgroup per tile: within HIP's limit of 2^32 - 1
  // work-items (the tiled form's grid is persistent).
  constexpr double kMaxTiles = 4294967295.0 / 512.0 - 8.0;
  const bool fits32 = n32 <= kMaxTiles, fits64 = n64 <= kMaxTiles;
  auto small = [](LinearF32Form form, int splits, double tiles, int64_t tile_bytes) {
    return LinearF32Plan{form, splits, splits == 1 ? 0 : splits * static_cast<int64_t>(tiles) * tile_bytes};
  };
  if (fits32 && (t32 <= t64 || !fits64) && t32 <= t128) return small(LinearF32Form::kTiles32, s32, n32, 4096);
  return fits64 && t64 <= t128 ? small(LinearF32Form::kTiles64, s64, n64, 16384) : tiled;
}

hipError_t launch_linear_f32(LinearF32Params& p, const LinearF32Plan& plan, void* workspace, bool gelu,
                             hipStream_t stream) {
  switch (plan.form) {
    case LinearF32Form::kTiles32:
      if (four_wavefronts(p.M, p.N, p.K)) return launch_small<1, 4>(p, plan, workspace, gelu, stream);
      return launch_small<1, 8>(p, plan, workspace, gelu, stream);
    case LinearF32Form::kTiles64: return launch_small<2, 8>(p, plan, workspace, gelu, stream);
    case LinearF32Form::kTiles128: p.wp = workspace; return launch_tiled(p, gelu, stream);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_split_weight(const float* w, void* wp, int N, int K, int64_t ldw, hipStream_t stream) {
  const int64_t items = static_cast<int64_t>((N + 31) / 32) * (K / 16) * 64;
  const int64_t blocks = std::min<int64_t>((items + 255) / 256, 8192);
  split_weight_kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream>>>(w, static_cast<u32x4*>(wp), N, K,
                                                                                  ldw);
  return hipGetLastError();
}

}  // namespace ttk
