// Fused flash-style attention forward for gfx950 (MI355X).
//
// Semantics follow the reference kernel `_attention_fwd`
// (transformer_opt/kernels/attention.py:103-265): BSHD strided q/k/v, fp32
// running max / running sum / output accumulator, keys visited in tiles with
// an online softmax, key mask `valid[b, t]`, causal bound
// `end = min(S, (query_tile + 1) * BLOCK_M)`, and exact zeros for a query row
// without any allowed key.
//
// Design (one workgroup = 4 wavefronts = 128 queries of one (batch, head)):
//
// * Each wavefront owns 32 queries and the full head dimension.  It computes
//   the TRANSPOSED score tile S^T[key, query] = K . Q^T with the 32x32 MFMA.
//   In the 32x32 MFMA result layout a lane holds one column (query = lane%32)
//   and 16 rows (keys 8*(r/4) + 4*(lane/32) + r%4 for register r), so
//     - the softmax row statistics of a query are a reduction over the lane's
//       own registers plus ONE exchange with lane^32 (v_permlane32_swap), and
//     - the probabilities P^T already sit in the B-operand layout of the next
//       MFMA, O^T[d, query] += V^T[d, key] . P^T[key, query]: register r
//       feeds the k-step whose two keys are the ones that register holds in
//       lane halves 0 and 1.  No transpose, no LDS round trip for P.
// * K and V tiles are double-buffered in LDS with one barrier per tile.  K
//   rows are padded by 16 bytes, so the 16-byte MFMA operand reads of 16
//   consecutive key rows start on distinct banks and cover all 64 banks, and
//   every per-step operand address is the lane's base plus an immediate.
//     - fp32, head_dim 32 and up: products of three-term bf16 splits on the
//       bf16 matrix cores, see attn_fwd_x3_kernel.
//     - fp32, head_dim 8 and 16: the next tile's global loads are issued into
//       registers before the current tile's MFMAs and written to the other
//       buffer after them; the fp32 MFMA is 16 passes long, and the softmax
//       VALU of one wavefront runs under the MFMAs of the other wavefront on
//       the SIMD.
//     - bf16/fp16: the 8-pass MFMA leaves the softmax as the bound (per
//       64-key tile of the unmasked steady body a wavefront issues 16
//       (head_dim 64) or 32 (128) MFMAs against 134 other VALU instructions
//       in the compiled head_dim-64 loop: 114 of softmax (32 fma, 32
//       v_exp_f32, 16 conversions, 16 max3, 16 dot2 row-sum steps, the
//       cross-half max), 2 for the lagging-max test and 18 of copy
//       addressing; a masked tile costs ~280), so the loop is
//       software-pipelined.  Unmasked tiles run two phases per tile:
//       Q.K of tile t+1 interleaved with the exp2 and 16-bit rounding of
//       tile t's scores, then the P.V of tile t interleaved with the row max
//       of tile t+1.  Key-masked tiles run one stream interleaving the
//       P.V of tile t-1 with the softmax of tile t.  K and V tiles are
//       copied global->LDS by LDS-DMA (global_load_lds_dwordx4, no register
//       staging), spread over the MFMA groups of the pipelined loop; V stays
//       row-major and the P.V operand is read with the transposing
//       ds_read_b64_tr_b16.
// * Masking: key validity (key mask and key < S) is a wave-uniform 64-bit
//   ballot per tile; with the lane's causal limit it becomes one bit mask per
//   32-key sub-block.  Only tiles that need it (diagonal, ragged end, key
//   mask) take the masked path; interior tiles run unmasked, and key
//   blocks before the first and after the last valid key are not visited
//   (scan_keys).  Causal
//   workgroups stop at their diagonal (future tiles are never loaded) and a
//   wavefront skips the 32-key sub-blocks entirely after its last query.
//   fp32 MFMA kernel: in the last tile of a query tile, wavefront 0
//   (whose rows are complete) takes wavefront 3's diagonal sub-block and
//   hands its partial softmax state over through LDS, so the diagonal costs
//   3 sub-block times instead of 4.
// * fp32 head_dim 8 and 16: P.V runs on 16x16x4 MFMAs (a 32x32 O^T block
//   would leave 3/4 or half of its d-rows empty); v_permlane16_swap of two
//   score registers regroups them by 16 queries, see the tile body.
// * Scheduling: causal query tile i costs i+1 key blocks.  When the grid
//   still fills every workgroup slot of the GPU, a workgroup runs the query
//   tiles nq-1-i and i one after the other, so all workgroups carry the same
//   nq+1 blocks of work and the launch has no tail.  Otherwise the flat grid
//   is ordered heaviest query tile first, or, for an fp32 grid resident in
//   one round, folded so that the two workgroups of a CU hold a heavy and a
//   light tile.  The fp32 MFMA kernel, non-causal with S <= 64, runs two
//   (batch, head) pairs per workgroup (the twin grid).  When B*H is a multiple of 8 all
//   workgroups of one head run on the same XCD (workgroups are dealt
//   round-robin to the 8 XCDs), so a head's K/V is fetched from HBM into one
//   XCD's L2 instead of eight.  The fp32 MFMA kernel alternates wave priority per
//   tile between the two workgroups of a CU (the age order otherwise favours
//   the older one throughout).
// * Output: the 16-bit kernel stages each wavefront's 32 x D tile in LDS so
//   that each store covers whole rows; fp32 stores straight from registers.
//
// fp32 path: fp32 products, exact to 2^-24 of each where they are formed from
// bf16 terms (bf16x3.h), fp32 accumulate.  Q is pre-multiplied by scale*log2(e) so scores
// are already in the exp2 domain.  bf16/fp16 path: v_mfma_f32_32x32x16_{bf16,f16}; scores stay fp32,
// the row max is taken on raw scores and the scale is folded into one fma per
// element before exp2; P is rounded to the input type (v_cvt_pk_bf16_f32 /
// v_cvt_f16_f32) for the P.V product; the 16-bit A operand (8 keys of one d)
// is two transposing 8-byte LDS reads of the row-major V tile.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "bf16x3.h"
#include "ttk_common.h"

namespace ttk {
namespace {

constexpr int kThreads = 256;
constexpr int kBM = 128;  // queries per workgroup (4 wavefronts x 32)

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 mfma_16(BF16, u16x8 a, u16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma_16(F16, u16x8 a, u16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Hardware conversions (round to nearest even) of probabilities to 16 bits.
__device__ __forceinline__ unsigned short to_bits(BF16, float v) {
  return __builtin_bit_cast(unsigned short, static_cast<__bf16>(v));
}
__device__ __forceinline__ unsigned short to_bits(F16, float v) {
  return __builtin_bit_cast(unsigned short, static_cast<_Float16>(v));
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Adds the 16-bit probabilities a lane holds for one tile (NP packed u16x8
// registers of 8 values) to the fp32 row sum acc with v_dot2c_f32_{bf16,f16}
// against (1, 1): one instruction per two values, accumulated straight into
// the running sum (no per-tile partial sums to clear and combine).  Summing
// the rounded P that the P.V product uses makes the weights applied to V sum
// to one exactly in the final division.
__device__ __forceinline__ float dot2_ones(BF16, unsigned pair, float acc) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair),
                                         __builtin_bit_cast(bf16x2, 0x3F803F80u), acc, false);
}
__device__ __forceinline__ float dot2_ones(F16, unsigned pair, float acc) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pair), __builtin_bit_cast(f16x2, 0x3C003C00u),
                                acc, false);
}
// Row sum of the first NU packed registers (all by default).
template <typename T, int NP, int NU = NP>
__device__ __forceinline__ float add_packed(const u16x8 (&pn)[NP], float acc) {
  static_assert(NU <= NP, "registers in use");
#pragma unroll
  for (int i = 0; i < NU; ++i) {
    const u32x4 w = __builtin_bit_cast(u32x4, pn[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = dot2_ones(T{}, w[j], acc);
  }
  return acc;
}

__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

// Max / sum of a value and the same value in lane ^ 32 (v_permlane32_swap:
// exchanges the upper half of the first operand with the lower half of the
// second, so the two results hold {x[l], x[l ^ 32]} in every lane).
// The maximum is one v_max_f32: fmaxf on the swapped words (integers to the
// compiler) would first quiet each of them with a v_max_f32 of its own.
__device__ __forceinline__ float max_with_other_half(float x) {
  const unsigned u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  float m;
  asm("v_max_f32 %0, %1, %2" : "=v"(m) : "v"(r[0]), "v"(r[1]));
  return m;
}
__device__ __forceinline__ float sum_with_other_half(float x) {
  const unsigned u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Per-query value (32x32 result layout: query l % 32, equal in both lane
// halves) re-read for the 16x16 output layout through v_permlane16_swap of
// (x, x), which swaps the odd 16-lane rows of the first operand with the even
// rows of the second: lo = the value of query l % 16, hi = that of query
// 16 + l % 16.
__device__ __forceinline__ void by_query16(float x, float& lo, float& hi) {
  const unsigned u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}

__device__ __forceinline__ f32x4 mfma_f32_16(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// LDS-DMA: each active lane copies the 16 bytes at gbase + voff (gbase
// wave-uniform, voff the lane's byte offset) to lds_base + 16 * lane
// (global_load_lds_dwordx4; lds_base is wave-uniform).  Completion is tracked
// by vmcnt only: callers wait with vm_wait() before the barrier that publishes
// the buffer.  Issued as inline assembly: the compiler cannot tell which LDS
// reads a copy feeds, and with the builtin it waits for every outstanding
// copy before the first LDS read after it - here, the K read right after the
// next tile's copies are issued.  M0 carries the LDS address; the one wait
// state after writing it is required before the copy reads it.
#define TTK_LDS(ptr) ((__attribute__((address_space(3))) void*)(ptr))
__device__ __forceinline__ void dma16(const void* gbase, unsigned voff, void* lds_base) {
  const unsigned lds = static_cast<unsigned>(reinterpret_cast<size_t>(TTK_LDS(lds_base)));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(gbase), "s"(lds)
               : "memory", "m0");
#pragma clang diagnostic pop
}
__device__ __forceinline__ void vm_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Key offset (inside a 32-key sub-block) held by register r of lane half h in
// the 32x32 MFMA result layout.
__device__ __forceinline__ int acc_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// Work of one workgroup: a (batch, head) and one or two query tiles.
struct Work {
  int bh;
  int q_first;   // query tile of the first pass
  int q_second;  // query tile of the second pass (npass == 2)
  int npass;
  int chunk;     // key-split grid: chunk of q_first's key tiles (of nchunk)
  int nchunk;
};

__device__ __forceinline__ Work work_item(const AttnParams& p, bool causal) {
  const int id = blockIdx.x;
  int unit, bh;
  if (p.xcd_swizzle) {
    const int xcd = id & 7;
    const int j = id >> 3;
    const int hpx = p.BH >> 3;  // heads per XCD
    unit = j / hpx;
    bh = xcd + 8 * (j - unit * hpx);
  } else {
    unit = id / p.BH;
    bh = id - unit * p.BH;
  }
  Work w;
  w.bh = bh;
  w.chunk = 0;
  w.nchunk = 1;
  if (causal && p.split) {
    const unsigned e = p.unit_tab[unit];
    w.q_first = static_cast<int>(e & 1023u);
    w.chunk = static_cast<int>((e >> 10) & 7u);
    w.nchunk = static_cast<int>(e >> 13) + 1;
    w.q_second = w.q_first;
    w.npass = 1;
    return w;
  }
  if (causal && p.fold) {
    // Folded order: the first half of the units takes the heavy query tiles
    // (descending), the second half the light ones (ascending), so that the
    // workgroups i and i + CUs that share a CU hold tiles of opposite weight.
    const int half = (p.nq + 1) >> 1;
    w.q_first = unit < half ? p.nq - 1 - unit : unit - half;
  } else {
    w.q_first = causal ? p.nq - 1 - unit : unit;
  }
  w.q_second = unit;
  w.npass = (causal && p.pair && unit < w.q_first) ? 2 : 1;
  return w;
}

// Valid bits of the keys [k0, k0 + 64) that exist (key < S).
__device__ __forceinline__ uint64_t range_bits(int k0, int S) {
  const int n = S - k0;
  return n >= 64 ? ~uint64_t{0} : ((uint64_t{1} << n) - 1);
}

// Allowed-key bits of one 32-key sub-block (first key ks) for this lane, as
// a mask over the lane's registers: bit 8*(r/4) + r%4 <-> register r.
template <bool CAUSAL>
__device__ __forceinline__ uint32_t lane_allowed(uint32_t sub_valid, int ks, int qrow, int h) {
  uint32_t a = sub_valid;
  if constexpr (CAUSAL) {
    const int lim = qrow - ks;  // keys ks + i allowed for i <= lim
    const uint32_t cm = lim >= 31 ? 0xffffffffu : (lim < 0 ? 0u : ((2u << lim) - 1u));
    a &= cm;
  }
  return a >> (4 * h);
}

// Sets scores of disallowed keys to -inf (tile of NSB sub-blocks from k0;
// only the first NL are touched - the caller has not computed the others).
// BITSEL: per register, a signed one-bit field extract of the allowed bit
// gives an all-ones / all-zeros word and a bit-field insert selects the score
// or -inf - two VALU instructions and no compare, so no VCC write that the
// select has to wait for.  Otherwise a compare and a select per register
// (fewer live registers where the kernel is at its register limit).
template <int NSB, bool CAUSAL, bool BITSEL = true, int NL = NSB>
__device__ __forceinline__ void apply_mask(f32x16 (&s)[NSB], int k0, uint64_t kvalid, int qrow, int h) {
#pragma unroll
  for (int sb = 0; sb < NL; ++sb) {
    const uint32_t a =
        lane_allowed<CAUSAL>(static_cast<uint32_t>(kvalid >> (32 * sb)), k0 + sb * 32, qrow, h);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int bit = 8 * (r >> 2) + (r & 3);
      if constexpr (BITSEL) {
        const uint32_t keep = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(a), bit, 1));
        const uint32_t bits = __float_as_uint(s[sb][r]);
        s[sb][r] = __uint_as_float((bits & keep) | (0xff800000u & ~keep));
      } else {
        if (!((a >> bit) & 1u)) s[sb][r] = -INFINITY;
      }
    }
  }
}

// Keys a masked query tile has to visit: those from the first 64-key block with
// a valid key up to the end of the last such block.
struct KeySpan {
  int first;  // a multiple of 64
  int end;
  int full;   // 64-key blocks from the first after which one holds an invalid
              // key (the first itself may): blocks 1 .. full - 1 are whole
};
constexpr int kSpanKeys = 512;  // shorter key ranges are visited whole
constexpr int kSpanLds = 4;     // words of LDS scratch

// Key span of the keys [0, end) of mask row M.  V rows
// that drop out have weight zero, and 0 * V is left out only where V is finite:
// with a non-finite value among them the span stays whole (and full is 0).
//
// Padding otherwise costs what valid keys cost, and a mask is applied to every
// tile (about half as much VALU work again as the softmax).  With the span, the
// 16-bit kernel runs its pipelined body on the whole blocks and applies masks
// only where one has an invalid key.  Measured with prefixes uniform in [S / 2,
// S] (three draws): fp16 [6, 1000, 16, 64] 43 -> 29 - 34 us, bf16 causal [4, 2048,
// 16, 64] 60 -> 49 - 51 us, bf16 [4, 2048, 16, 128] 159 -> 123 - 131 us; fp32 [8,
// 1024, 16, 64] 196 us without and 179 with.  At S = 16384, half of it padding,
// every workgroup reads 8192 dropped V rows, and bf16 causal [1, 16384, 16, 128]
// still takes 811 us where it took 1147.  The scan costs 0.5 - 1 us of a launch: nothing
// on up to 512 keys, where it gained nothing either (bf16 [2, 300, 4, 64] 9.6
// -> 10.1 us with it), and 0 - 7 % where invalid keys are scattered over all
// blocks (bf16 [2, 600, 8, 64] 14.6 -> 15.6 us, bf16 [8, 1000, 16, 64] 56.7 ->
// 58.0 us).
//
// The scan is one dependent load: every wavefront reads the whole row (64 keys
// a lane, as bytes of a bool mask with unit stride), so nothing is exchanged.
template <typename St, unsigned INF, int D>  // INF: magnitude bits of infinity
__device__ __forceinline__ KeySpan scan_keys(const uint8_t* M, const St* V, int64_t vs, int end, int* lds) {
  typedef u32x4 __attribute__((aligned(1))) Bytes16;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  const int nb = (end + 63) >> 6;
  int lo = -1, hi = -1, stop = -1;
  for (int b = 0; b < nb; b += 64) {
    // The last chunk of the row is read as its last 16 bytes: keys of the chunk
    // before count twice, which at most keeps a block.
    unsigned any = 0, zero = 0;
    const int k = 64 * min(b + lane, nb - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4 x = *reinterpret_cast<const Bytes16*>(M + min(k + 16 * i, end - 16));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        any |= x[e];
        zero |= (x[e] - 0x01010101u) & ~x[e] & 0x80808080u;  // set if a byte is zero
      }
    }
    const bool real = b + lane < nb;
    const uint64_t valid = __builtin_amdgcn_ballot_w64(real && any != 0);
    uint64_t bad = __builtin_amdgcn_ballot_w64(real && zero != 0);
    if (valid != 0) {
      if (lo < 0) {
        const int f = __builtin_ctzll(valid);
        lo = b + f;
        bad &= ~((uint64_t{2} << f) - 1);  // blocks after the first
      }
      hi = b + 63 - __builtin_clzll(valid);
    }
    if (lo >= 0 && stop < 0 && bad != 0) stop = b + __builtin_ctzll(bad);
  }
  lo = max(lo, 0);  // no valid key at all: the first block
  hi = max(hi, 0);
  if (stop < 0) stop = nb;
  KeySpan span = {64 * lo, min(end, 64 * (hi + 1)), stop - lo};
  if (lo == 0 && hi == nb - 1) return span;

  // 16-byte chunks of the rows that drop out: the largest magnitude bits.
  constexpr int kChunk = 16 / sizeof(St);
  constexpr int CPR = D / kChunk;
  constexpr int RPP = kThreads / CPR;  // rows per pass
  const int col = kChunk * (static_cast<int>(threadIdx.x) % CPR);
  unsigned top = 0;
  auto scan_v = [&](int r0, int r1) __attribute__((always_inline)) {
    for (int r = r0; r < r1; r += 4 * RPP) {
      u32x4 x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = min(r + u * RPP + static_cast<int>(threadIdx.x) / CPR, r1 - 1);
        x[u] = *reinterpret_cast<const u32x4*>(V + static_cast<int64_t>(row) * vs + col);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (sizeof(St) == 4) {
            top = max(top, x[u][e] & 0x7fffffffu);
          } else {
            typedef unsigned short us2 __attribute__((ext_vector_type(2)));
            top = __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(us2, top),
                                                                         __builtin_bit_cast(us2, x[u][e] & 0x7fff7fffu)));
          }
        }
    }
  };
  if (span.first > 0) scan_v(0, span.first);
  if (span.end < end) scan_v(span.end, end);
  bool odd = sizeof(St) == 4 ? top >= INF : ((top & 0xffffu) >= INF || (top >> 16) >= INF);
  odd = __builtin_amdgcn_ballot_w64(odd) != 0;
  if (lane == 0) lds[wave] = odd;
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(lds[0] | lds[1] | lds[2] | lds[3])) span = KeySpan{0, end, 0};
  return span;
}

// Waves per SIMD the register budget is sized for: two workgroups per CU,
// except fp32 head_dim 128, whose live state does not fit 256 registers and
// runs one workgroup per CU; and 16-bit head_dim <= 64, sized for three (at most 168 VGPRs; the LDS of three workgroups fits).  The 16-bit
// loop is VALU-issue and latency bound, so the third workgroup pays: left to
// itself the compiler gave the causal head_dim-64 kernel 176 VGPRs (two
// workgroups per CU), and capping it at 168 - five registers spilled, reloaded
// only on the accumulator-rescale path - made [4, 2048, 16, 64] 5-7 %
// faster.
template <bool F32, int D>
constexpr int kMinWaves = (D >= 128 && F32) ? 1 : ((!F32 && D <= 64) ? 3 : 2);

// ----------------------------------------------------------------------------
// fp32, head_dim 8 and 16 (fp32 MFMA)
// ----------------------------------------------------------------------------
template <int D>
struct F32Cfg {
  static constexpr int BN = 64;                     // keys per tile
  static constexpr int NSB = BN / 32;               // 32-key sub-blocks per tile
  static constexpr int CPR = D / 4;                 // 16-byte chunks per key row
  static constexpr int KS = D + 4;                  // LDS K row stride (floats, 16-byte pad)
  static constexpr int G = D / 8;                   // Q.K groups of 4 k-steps
  static constexpr int CHUNKS = BN * CPR;
  static constexpr int CPT = (CHUNKS + kThreads - 1) / kThreads;  // chunks per thread
};

template <int D, bool CAUSAL, bool HAS_MASK>
__global__ __launch_bounds__(kThreads, (kMinWaves<true, D>)) void attn_fwd_f32_kernel(AttnParams p) {
  static_assert(D <= 16, "wider heads run attn_fwd_x3_kernel");
  using C = F32Cfg<D>;
  constexpr int BN = C::BN, NSB = C::NSB, CPR = C::CPR, KS = C::KS, CPT = C::CPT, G = C::G;
  __shared__ __attribute__((aligned(16))) float smK[2][BN * KS];
  __shared__ __attribute__((aligned(16))) float smV[2][BN * D];
  // Causal hand-off (two-sub-block tiles): in the last key tile of a query
  // tile only wavefronts 2 (one sub-block) and 3 (two) have keys left, so
  // wavefront 0 - whose rows are complete by then - takes wavefront 3's
  // diagonal sub-block and passes its partial state through smX: per lane
  // 8 accumulator values, the row max and the lane half's row sum, as
  // 16-byte chunks at smX[(chunk * 64 + lane) * 4].
  constexpr bool kHandoff = CAUSAL;
  __shared__ __attribute__((aligned(16))) float smX[kHandoff ? 3 * 256 : 4];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int m = lane & 31;
  const int h = lane >> 5;

  const Work w = work_item(p, CAUSAL);
  // Twin grid (S <= 64, one key tile, rows only for wavefronts 0-1 of a
  // 128-query tile): workgroup i serves (batch, head) pairs 2i (wavefronts
  // 0-1, K/V buffer 0) and 2i + 1 (wavefronts 2-3, buffer 1).  The second
  // pair of the last workgroup may not exist (odd B*H): its wavefronts hold
  // no rows and read nothing.  Built into the non-causal kernels only (the
  // causal ones keep their register budget for the pairing and hand-off).
  constexpr bool kTwin = !CAUSAL;
  const bool twin = kTwin && p.twin != 0;
  const int slot = twin ? (wave >> 1) : 0;
  const int bh = twin ? 2 * static_cast<int>(blockIdx.x) + slot : w.bh;
  const bool head_live = bh < p.BH;
  const int b = head_live ? bh / p.H : 0;
  const int hh = head_live ? bh - b * p.H : 0;
  const int S = p.S;
  const float* __restrict__ Q = static_cast<const float*>(p.q) + b * p.qb + hh * p.qh;
  const float* __restrict__ K = static_cast<const float*>(p.k) + b * p.kb + hh * p.kh;
  const float* __restrict__ V = static_cast<const float*>(p.v) + b * p.vb + hh * p.vh;
  const uint8_t* __restrict__ M = HAS_MASK ? p.mask + b * p.mb : nullptr;

  // Every pass ends with a barrier after its last LDS read, so the next pass
  // may refill both buffers right away.
  f32x4 rk[C::CPT], rv[C::CPT];
  bool rm = false;
  bool staged = false;  // tile 0 of the coming pass already sits in rk / rv
  // Wave priority alternates tile by tile, in opposite phase for workgroups
  // whose index differs by the CU count.  The first grid fills every CU with
  // workgroups i and i + CUs; left to the age order, the older of the two
  // wins every issue conflict and finishes ~15 % earlier, and the younger
  // one runs alone to the end.  Alternating shares the CU evenly; a lone
  // workgroup keeps its CU nearly as busy, so the gain is small (~1 % at
  // S=1024).
  const int prio_phase = (static_cast<int>(blockIdx.x) / max(p.cu_count, 1)) & 1;
  // Folded grid: the heavy workgroup of a CU (the first CU-count workgroups)
  // keeps the high priority throughout and the light one fills its gaps
  // (0.5 % faster than alternating at B*H = 128, S=512).
  const bool fold_fixed = p.fold != 0;
  const bool fold_heavy = prio_phase == 0;
  int tiles_done = 0;
  for (int pass = 0; pass < w.npass; ++pass) {
    const int qb = pass == 0 ? w.q_first : w.q_second;
    // First query of this wavefront (uniform); S, i.e. no rows, for the
    // missing second pair of a twin workgroup.
    const int q0 = !head_live ? S : qb * kBM + (twin ? (wave & 1) : wave) * 32;
    int qrow = q0 + m;                    // query of this lane (wavefront 3's on a hand-off)

    // B operand of S^T = K.Q^T: group g covers d = 8g..8g+7, lane half h
    // holds d = 8g+4h..8g+4h+3 (one element per k-step).  Pre-scaled into
    // exp2 units.
    f32x4 qf[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (qrow < S) {
        qf[g] = *reinterpret_cast<const f32x4*>(Q + qrow * p.qs + 8 * g + 4 * h) * p.scale_log2;
      } else {
        qf[g] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }

    const int kv_end = CAUSAL ? min(S, (qb + 1) * kBM) : S;
    const int ntiles = (kv_end + BN - 1) / BN;
    // Hand-off in this pass: the last tile starts half-way into the query
    // tile and wavefront 3 has rows (and keys of its second sub-block) < S.
    const bool handoff = kHandoff && (ntiles - 1) * BN == qb * kBM + 64 && qb * kBM + 96 < S;
    bool own_done = false;  // wavefront 0 stored its own rows early

    // Global loads of tile t into registers; rows past S read as zeros.
    auto gload = [&](int t) {
      const bool full = (t + 1) * BN <= S;
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int idx = tid + kThreads * i;
        if (C::CHUNKS % kThreads == 0 || idx < C::CHUNKS) {
          const int row = idx / CPR;
          const int c = idx - row * CPR;
          const int key = t * BN + row;
          if (full || key < S) {
            rk[i] = *reinterpret_cast<const f32x4*>(K + key * p.ks + 4 * c);
            rv[i] = *reinterpret_cast<const f32x4*>(V + key * p.vs + 4 * c);
          } else {
            rk[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            rv[i] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
      }
      if constexpr (HAS_MASK) {
        const int key = t * BN + lane;  // every wavefront reads the tile's mask bytes
        rm = lane < BN && key < S && M[key * p.ms] != 0;
      }
    };
    // Writes the staged tile into LDS buffer `buf`; returns the tile's
    // valid-key bits (key mask and key < S) as a wave-uniform 64-bit mask.
    auto lstore = [&](int buf, int t) -> uint64_t {
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int idx = tid + kThreads * i;
        if (C::CHUNKS % kThreads == 0 || idx < C::CHUNKS) {
          const int row = idx / CPR;
          const int c = idx - row * CPR;
          *reinterpret_cast<f32x4*>(&smK[buf][row * KS + 4 * c]) = rk[i];
          *reinterpret_cast<f32x4*>(&smV[buf][row * D + 4 * c]) = rv[i];
        }
      }
      if constexpr (HAS_MASK) {
        return __builtin_amdgcn_ballot_w64(rm);
      } else {
        return range_bits(t * BN, S);
      }
    };

    auto kread = [&](int buf, int sb, int g) -> f32x4 {
      const int row = sb * 32 + m;
      return *reinterpret_cast<const f32x4*>(&smK[buf][row * KS + 8 * g + 4 * h]);
    };
    float m_run = -INFINITY;
    float l_run = 0.0f;  // partial sum over this lane half's keys
    // O^T in two blocks of 16 queries (16x16x4 MFMAs: a 32x32 block would
    // leave 3/4 or half of its d-rows empty).
    f32x4 acc_lo{}, acc_hi{};

    // One tile: S^T = K.Q^T, (mask), online softmax, O^T += V^T.P^T.
    // MASKED: apply the key / causal mask; PARTIAL: only the first of the two
    // sub-blocks holds keys this wavefront may see (the other is skipped).
    // Tiles with every sub-block live keep the branch-free, interleaved
    // sub-block chains even when masked.
    // SB0: index in the LDS tile of the first sub-block processed (k0 and
    // kvalid describe that sub-block onwards).
    auto tile = [&](auto masked_tag, auto partial_tag, auto sb0_tag, int buf, int k0, int nlive,
                    uint64_t kvalid) {
      constexpr bool MASKED = decltype(masked_tag)::value;
      constexpr bool PARTIAL = decltype(partial_tag)::value;
      constexpr int SB0 = decltype(sb0_tag)::value;
      // Live sub-blocks (nlive, 1 on partial tiles, which have two) as a
      // compile-time count in the causal kernels: a run-time one puts every
      // MFMA of sub-block 1 under its own branch, and the compiler copies its
      // operands through each.  Non-causal kernels see partial tiles only at a
      // ragged end and keep the run-time form.
      constexpr bool kStaticLive = CAUSAL;
      constexpr int NL = PARTIAL ? 1 : NSB;
      auto live = [&](int sb) __attribute__((always_inline)) {
        return kStaticLive ? sb < NL : (!PARTIAL || sb < nlive);
      };
      f32x16 s[NSB];
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
        if (!kStaticLive || sb < NL) s[sb] = f32x16{};
      // ---- S^T = K . Q^T (K fragments read one group ahead) --------------
      f32x4 kf[NSB];
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
        if (live(sb)) kf[sb] = kread(buf, SB0 + sb, 0);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        f32x4 kn[NSB];
        if (g + 1 < G) {
#pragma unroll
          for (int sb = 0; sb < NSB; ++sb)
            if (live(sb)) kn[sb] = kread(buf, SB0 + sb, g + 1);
        }
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb) {
          if (!live(sb)) continue;
#pragma unroll
          for (int e = 0; e < 4; ++e) s[sb] = mfma_f32(kf[sb][e], qf[g][e], s[sb]);
        }
        if (g + 1 < G) {
#pragma unroll
          for (int sb = 0; sb < (kStaticLive ? NL : NSB); ++sb) kf[sb] = kn[sb];
        }
        fence();
      }
      constexpr int NS = kStaticLive ? NL : NSB;  // sub-blocks the softmax visits
      if constexpr (MASKED) apply_mask<NSB, CAUSAL, true, NS>(s, k0, kvalid, qrow, h);
      // ---- online softmax (exp2 domain) ------------------------------------
      float mt = s[0][0];
#pragma unroll
      for (int sb = 0; sb < NS; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[sb][r]);
      mt = max_with_other_half(mt);
      const float m_new = fmaxf(m_run, mt);
      // A fully masked row keeps m = -inf; use 0 so exp2(-inf - 0) = 0, never NaN.
      const float m_use = (MASKED && m_new == -INFINITY) ? 0.0f : m_new;
      const float alpha = fast_exp2(m_run - m_use);
      float ls = 0.0f;
#pragma unroll
      for (int sb = 0; sb < NS; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float pr = fast_exp2(s[sb][r] - m_use);
          s[sb][r] = pr;
          ls += pr;
        }
      l_run = __builtin_fmaf(l_run, alpha, ls);
      float a_lo, a_hi;
      by_query16(alpha, a_lo, a_hi);
      acc_lo *= a_lo;
      acc_hi *= a_hi;
      m_run = m_new;
      fence();
      // ---- O^T += V^T . P^T on 16x16x4 MFMAs -----------------------------
      // v_permlane16_swap of score registers r, r + 1 (keys k, k + 1 in lane
      // half 0, k + 4, k + 5 in half 1, k = 8(r/4) + r%4) leaves queries
      // 0-15 in the first and 16-31 in the second, with key k + {0,1,4,5}[g]
      // in 16-lane row g: the B operands of the two 16-query output blocks,
      // sharing one A operand V[key][d = l % 16].  acc_lo holds queries 0-15
      // (d = 4(l/16) + e, query l % 16), acc_hi 16-31; for head_dim 8 the
      // rows d >= 8 multiply zeros.
      const int g16 = lane >> 4;
      const int vkey = (g16 & 1) + 4 * (g16 >> 1);
      const bool d_ok = (lane & 15) < D;
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) {
        if (!live(sb)) continue;
        const float* vb = &smV[buf][((SB0 + sb) * 32 + vkey) * D + (lane & 15 & (D - 1))];
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const float va = d_ok ? vb[(8 * (r >> 2) + (r & 3)) * D] : 0.0f;
          const auto pq = __builtin_amdgcn_permlane16_swap(__float_as_uint(s[sb][r]), __float_as_uint(s[sb][r + 1]),
                                                           false, false);
          acc_lo = mfma_f32_16(va, __uint_as_float(pq[0]), acc_lo);
          acc_hi = mfma_f32_16(va, __uint_as_float(pq[1]), acc_hi);
        }
      }
      fence();
    };

    // O = acc / l: queries base + l % 16 and base + 16 + l % 16, d = 4(l/16) + e.
    auto epilogue = [&]() __attribute__((always_inline)) {
      const float lt = sum_with_other_half(l_run);
      float lt_lo, lt_hi;
      by_query16(lt, lt_lo, lt_hi);
      const float inv_lo = lt_lo > 0.0f ? 1.0f / lt_lo : 0.0f;
      const float inv_hi = lt_hi > 0.0f ? 1.0f / lt_hi : 0.0f;
      const int base = qrow - m;  // first query of the rows held (uniform)
      const int d0 = 4 * (lane >> 4);
      float* __restrict__ O = static_cast<float*>(p.out) + b * p.ob + hh * p.oh + d0;
      const int r_lo = base + (lane & 15), r_hi = r_lo + 16;
      if (d0 >= D) return;  // head_dim 8: d-rows 8-15 are empty
      if (r_lo < S) *reinterpret_cast<f32x4*>(O + r_lo * p.os) = acc_lo * inv_lo;
      if (r_hi < S) *reinterpret_cast<f32x4*>(O + r_hi * p.os) = acc_hi * inv_hi;
    };

    // Twin grid: both pairs' only key tile, pair 2i into buffer 0 and 2i + 1
    // into buffer 1, every load issued before the first LDS store; returns
    // this wavefront's valid-key bits.
    auto twin_stage = [&]() -> uint64_t {
      f32x4 tk[2][CPT], tv[2][CPT];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const int bhx = 2 * static_cast<int>(blockIdx.x) + s2;
        const bool live = bhx < p.BH;
        const int bx = live ? bhx / p.H : 0;
        const int hx = live ? bhx - bx * p.H : 0;
        const float* Kx = static_cast<const float*>(p.k) + bx * p.kb + hx * p.kh;
        const float* Vx = static_cast<const float*>(p.v) + bx * p.vb + hx * p.vh;
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
          const int idx = tid + kThreads * i;
          if (C::CHUNKS % kThreads == 0 || idx < C::CHUNKS) {
            const int row = idx / CPR;  // key: the tile starts at key 0
            const int c = idx - row * CPR;
            if (live && row < S) {
              tk[s2][i] = *reinterpret_cast<const f32x4*>(Kx + row * p.ks + 4 * c);
              tv[s2][i] = *reinterpret_cast<const f32x4*>(Vx + row * p.vs + 4 * c);
            } else {
              tk[s2][i] = f32x4{0.f, 0.f, 0.f, 0.f};
              tv[s2][i] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
          }
        }
      }
      bool valid = head_live && lane < S;
      if constexpr (HAS_MASK) valid = valid && M[lane * p.ms] != 0;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
          const int idx = tid + kThreads * i;
          if (C::CHUNKS % kThreads == 0 || idx < C::CHUNKS) {
            const int row = idx / CPR;
            const int c = idx - row * CPR;
            *reinterpret_cast<f32x4*>(&smK[s2][row * KS + 4 * c]) = tk[s2][i];
            *reinterpret_cast<f32x4*>(&smV[s2][row * D + 4 * c]) = tv[s2][i];
          }
        }
      }
      return HAS_MASK ? __builtin_amdgcn_ballot_w64(valid) : range_bits(0, S);
    };

    uint64_t kvalid;
    if (kTwin && twin) {
      kvalid = twin_stage();
    } else {
      if (!staged) gload(0);
      kvalid = lstore(0, 0);
    }
    __syncthreads();
    staged = false;

    for (int t = 0; t < ntiles; ++t) {
      const int buf = twin ? slot : (t & 1);
      if (fold_fixed ? fold_heavy : (((tiles_done + t) & 1) == prio_phase)) {
        __builtin_amdgcn_s_setprio(1);
      } else {
        __builtin_amdgcn_s_setprio(0);
      }
      if (t + 1 < ntiles) {
        gload(t + 1);
      } else if (pass + 1 < w.npass) {
        gload(0);  // the next pass's key tile 0 (same head, same rows)
        staged = true;
      }
      const int k0 = t * BN;
      if constexpr (kHandoff) {
        if (handoff && t == ntiles - 1 && wave == 0) {
          // Own rows are complete (their last keys were in tile t - 1): store
          // them, then run wavefront 3's second sub-block of this tile on
          // wavefront 3's rows from a fresh state and hand the state over.
          const int frow = qb * kBM + 96 + m;
          f32x4 fq[G];
#pragma unroll
          for (int g = 0; g < G; ++g) {
            fq[g] = frow < S ? *reinterpret_cast<const f32x4*>(Q + frow * p.qs + 8 * g + 4 * h) * p.scale_log2
                             : f32x4{0.f, 0.f, 0.f, 0.f};
          }
          epilogue();
          own_done = true;
          qrow = frow;
#pragma unroll
          for (int g = 0; g < G; ++g) qf[g] = fq[g];
          m_run = -INFINITY;
          l_run = 0.0f;
          acc_lo = acc_hi = f32x4{};
          tile(std::true_type{}, std::true_type{}, std::integral_constant<int, 1>{}, buf, k0 + 32, 1,
               kvalid >> 32);
          *reinterpret_cast<f32x4*>(&smX[lane * 4]) = acc_lo;
          *reinterpret_cast<f32x4*>(&smX[(64 + lane) * 4]) = acc_hi;
          *reinterpret_cast<f32x4*>(&smX[(128 + lane) * 4]) = f32x4{m_run, l_run, 0.f, 0.f};
        }
      }
      if (q0 < S && (!CAUSAL || k0 <= q0 + 31) && !own_done) {
        // Leading sub-blocks that hold any key this wavefront may see.
        int nlive = NSB;
#pragma unroll
        for (int sb = NSB - 1; sb >= 0; --sb) {
          const int ks = k0 + sb * 32;
          if (ks >= S || (CAUSAL && ks > q0 + 31)) nlive = sb;
        }
        // On a hand-off wavefront 3 keeps only the first sub-block of the last
        // tile; its second sub-block's keys are cleared from the valid bits,
        // since the causal mask alone would leave them at score 0.
        uint64_t kv = kvalid;
        if (kHandoff && handoff && t == ntiles - 1 && wave == 3) {
          nlive = 1;
          kv &= 0xffffffffull;
        }
        const bool need_mask = HAS_MASK || (k0 + BN > S) || (CAUSAL && k0 + BN - 1 > q0);
        if (need_mask) {
          if (nlive < NSB) {
            tile(std::true_type{}, std::true_type{}, std::integral_constant<int, 0>{}, buf, k0, nlive, kv);
          } else {
            tile(std::true_type{}, std::false_type{}, std::integral_constant<int, 0>{}, buf, k0, NSB, kv);
          }
        } else {
          tile(std::false_type{}, std::false_type{}, std::integral_constant<int, 0>{}, buf, k0, NSB, kvalid);
        }
      }
      if (t + 1 < ntiles) kvalid = lstore(buf ^ 1, t + 1);
      __syncthreads();
    }

    if constexpr (kHandoff) {
      if (handoff && wave == 3) {
        // Merge wavefront 0's state for the second sub-block of the last
        // tile (written before the loop's final barrier).
        const f32x4 ml = *reinterpret_cast<const f32x4*>(&smX[(128 + lane) * 4]);
        const float mx = fmaxf(m_run, ml[0]);
        const float mu = mx == -INFINITY ? 0.0f : mx;
        const float a = fast_exp2(m_run - mu);
        const float bb = fast_exp2(ml[0] - mu);
        l_run = __builtin_fmaf(l_run, a, ml[1] * bb);
        // Factors per output block (queries l % 16 and 16 + l % 16).
        float a_lo, a_hi, b_lo, b_hi;
        by_query16(a, a_lo, a_hi);
        by_query16(bb, b_lo, b_hi);
        const f32x4 x_lo = *reinterpret_cast<const f32x4*>(&smX[lane * 4]);
        const f32x4 x_hi = *reinterpret_cast<const f32x4*>(&smX[(64 + lane) * 4]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc_lo[e] = __builtin_fmaf(acc_lo[e], a_lo, x_lo[e] * b_lo);
          acc_hi[e] = __builtin_fmaf(acc_hi[e], a_hi, x_hi[e] * b_hi);
        }
        m_run = mx;
      }
    }
    if (!own_done) epilogue();
    tiles_done += ntiles;
  }
  __builtin_amdgcn_s_setprio(0);
}

// ----------------------------------------------------------------------------
// fp32, short sequences: S <= 64, non-causal, head_dim 32 / 64
// ----------------------------------------------------------------------------
// The whole 64-key tile of one (batch, head) fits a wavefront's registers as
// MFMA operands (head_dim 64: K 64 + V 64 + Q 32 VGPRs), so one wavefront
// serves one (batch, head, 32-query half) on its own: no barrier.  The grid
// is persistent (two workgroups per CU); wavefront gw walks the items gw,
// gw + W, ... (item = 2 * (batch * H + head) + half, so the two halves of a
// head run side by side in one workgroup and the second K/V read hits L2).
// While the current item's softmax and P.V run, the next item's K and Q are
// in flight, and the next V while the current rows are stored.
//
// Global traffic is row-coalesced: K, Q and O move as whole rows (64 lanes x
// 16 bytes = 1 KB of consecutive rows per instruction) and are re-laid out
// through an LDS region private to the wavefront (64 rows, 16 KB at head_dim
// 64; 16-byte chunks XOR-swizzled by row so both layouts access LDS without
// bank conflicts): K and Q into the MFMA operand layout (key or query per lane,
// 4 head dims per register), O back from the accumulator layout.  The MFMA
// fragments read with a lane stride of a whole row (32 rows x 32 bytes per
// instruction) cost ~8 % more time at S = 64 than whole rows.  V is read
// straight into its operand layout, 256 contiguous bytes per half-wavefront.
// (fp32 MFMA: the launch is bound by HBM, 4.6 TB/s at [512, 64, 8, 64], so the
// bf16 matrix cores would not shorten it.)
// MASKED: scores need the key mask (HAS_MASK, or S < 64 leaves padded keys).
template <int D>
struct VFrag32 {
  using type = float;
};
template <>
struct VFrag32<64> {
  using type = float2;
};
template <int D, bool HAS_MASK, bool MASKED>
__global__ __launch_bounds__(kThreads, 2) void attn_fwd_f32_short_kernel(AttnParams p) {
  static_assert(D == 32 || D == 64, "short-sequence kernel: head_dim 32 or 64");
  constexpr int NSB = 2, DB = D / 32, G = D / 8;
  constexpr int CPR = D / 4;        // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;     // rows per row-coalesced instruction
  constexpr int NI = 32 / RPI;      // instructions per 32 rows (== G)
  static_assert(NI == G, "32 rows take as many instructions as Q has fragments");
  using VF = typename VFrag32<D>::type;
  __shared__ __attribute__((aligned(16))) float smem[kThreads / 64][64 * D];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 31;
  const int h = lane >> 5;
  const int S = p.S;
  const int hshift = S > 32 ? 1 : 0;  // 32-query halves per head: 2 or 1
  const int items = p.BH << hshift;
  const int stride = static_cast<int>(gridDim.x) * (kThreads / 64);
  int item = static_cast<int>(blockIdx.x) * (kThreads / 64) + wave;
  if (item >= items) return;
  float* const region = smem[wave];

  // Every global access is a buffer access whose resource covers exactly the
  // rows < S of one head (the host checks row stride >= head_dim and that
  // the offsets of all 64 rows a lane may address stay below 2^31): rows past
  // S read as zeros and are not written,
  // without a branch.  The range check covers the VGPR offset (plus the
  // instruction offset) but not soffset, so the row part of every offset is
  // in the VGPR.  The loads of the next item are issued unconditionally -
  // after the last item with an empty resource, which fetches nothing - so
  // every wait count is exact on the one path through the loop and waits only
  // for the operands it needs.
  auto head_of = [&](int it, int& b, int& hh) {
    const int bh = it >> hshift;
    b = bh / p.H;
    hh = bh - b * p.H;
  };
  auto rsrc = [&](const void* base, int64_t bo, int64_t ho, int64_t rs, int it, bool live) {
    int b, hh;
    head_of(it, b, hh);
    const float* ptr = static_cast<const float*>(base) + b * bo + hh * ho;
    const int bytes = live ? static_cast<int>(((S - 1) * rs + D) * 4) : 0;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(ptr), static_cast<short>(0), bytes, 0x00020000);
  };
  // Row-coalesced lane position: instruction j covers rows RPI*j .. RPI*j + RPI - 1.
  const int crow = lane / CPR;
  const int cchunk = lane % CPR;
  // LDS float index of (row, 16-byte chunk) in the wavefront's region.
  auto slot = [](int row, int chunk) { return row * D + 4 * (chunk ^ (row & (CPR - 1))); };
  const int voff0 = static_cast<int>((4 * h * p.vs + DB * m) * 4);

  f32x4 kst[NSB][NI], qst[NI];  // K and Q as loaded (row-coalesced)
  VF vf[NSB][16];
  int key_ok = 0;  // HAS_MASK: this lane's key (= lane) exists and is not masked

  // 32 rows from row0 of one head, row-coalesced (the row offsets of the
  // instructions are added at each load, not hoisted into live registers).
  auto load_rows = [&](f32x4 (&dst)[NI], const __amdgpu_buffer_rsrc_t& rs, int64_t row_stride, int row0) {
    int off = static_cast<int>(((row0 + crow) * row_stride + 4 * cchunk) * 4);
    asm volatile("" : "+v"(off));
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      dst[j] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + static_cast<int>(RPI * j * row_stride * 4), 0, 0));
    }
  };
  auto load_q = [&](int it, bool live) {
    const auto rq = rsrc(p.q, p.qb, p.qh, p.qs, it, live);
    load_rows(qst, rq, p.qs, (it & hshift) << 5);
    if constexpr (HAS_MASK) {
      int b, hh;
      head_of(it, b, hh);
      const int bytes = live ? static_cast<int>((S - 1) * p.ms + 1) : 0;
      const auto rm = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.mask + b * p.mb),
                                                        static_cast<short>(0), bytes, 0x00020000);
      key_ok = __builtin_amdgcn_raw_buffer_load_b8(rm, static_cast<int>(lane * p.ms), 0, 0);
    }
  };
  auto load_k = [&](int it, bool live, int sb) {
    const auto rk = rsrc(p.k, p.kb, p.kh, p.ks, it, live);
    load_rows(kst[sb], rk, p.ks, sb * 32);
  };
  // V as the A operand of O^T += V^T . P^T: register (sb, r) holds key
  // sb * 32 + acc_row(r, h), head dims DB * m .. DB * m + DB - 1.  The
  // per-register row offsets are added at each load (an opaque copy of the
  // lane offset keeps them from being hoisted into 32 live registers).
  auto load_v = [&](int it, bool live, int sb) {
    const auto rv = rsrc(p.v, p.vb, p.vh, p.vs, it, live);
    int voff = voff0;
    asm volatile("" : "+v"(voff));
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int off = voff + static_cast<int>((sb * 32 + acc_row(r, 0)) * p.vs * 4);
      if constexpr (DB == 1) {
        vf[sb][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, off, 0, 0));
      } else {
        vf[sb][r] = __builtin_bit_cast(VF, __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0));
      }
    }
  };
  // Row-coalesced registers -> LDS region rows row0 .. row0 + 31.
  auto put_rows = [&](const f32x4 (&src)[NI], int row0) {
#pragma unroll
    for (int j = 0; j < NI; ++j) *reinterpret_cast<f32x4*>(&region[slot(row0 + RPI * j + crow, cchunk)]) = src[j];
  };
  // MFMA operand fragments from the region: group g of lane (m, h) holds row
  // row0 + m, head dims 8g + 4h .. 8g + 4h + 3 (16-byte chunk 2g + h).
  auto get_frags = [&](f32x4 (&dst)[G], int row0) {
#pragma unroll
    for (int g = 0; g < G; ++g) dst[g] = *reinterpret_cast<const f32x4*>(&region[slot(row0 + m, 2 * g + h)]);
  };

  // Same memory-instruction sequence as the loop body issues before its head
  // (K, Q, NI row stores, V; the stores here go to an empty resource and
  // write nothing): vmcnt counts loads and stores together, so the wait
  // counts the compiler derives at the loop head then fit both paths into it
  // and none of them waits for the previous item's stores.
  load_k(item, true, 0);
  load_k(item, true, 1);
  load_q(item, true);
  {
    const auto none = __builtin_amdgcn_make_buffer_rsrc(p.out, static_cast<short>(0), 0, 0x00020000);
#pragma unroll
    for (int j = 0; j < NI; ++j) __builtin_amdgcn_raw_buffer_store_b128(u32x4{0u, 0u, 0u, 0u}, none, 16 * j, 0, 0);
  }
  load_v(item, true, 0);
  load_v(item, true, 1);
  while (true) {
    const int next_raw = item + stride;
    const bool more = next_raw < items;
    const int next = more ? next_raw : item;
    const int half_row0 = (item & hshift) << 5;
    const int qrow = half_row0 + m;
    const uint64_t kv = HAS_MASK ? __builtin_amdgcn_ballot_w64(lane < S && key_ok != 0) : range_bits(0, S);
    const auto ro = [&] {
      int b, hh;
      head_of(item, b, hh);
      float* ptr = static_cast<float*>(p.out) + b * p.ob + hh * p.oh;
      const int bytes = static_cast<int>(((S - 1) * p.os + D) * 4);
      return __builtin_amdgcn_make_buffer_rsrc(ptr, static_cast<short>(0), bytes, 0x00020000);
    }();

    // ---- S^T = K . Q^T (sub-block by sub-block; each accumulates over d in
    // the same order as the tiled kernel).  Q, then K, passes through the LDS
    // region; one wavefront's LDS accesses complete in program order, so the
    // K rows overwrite Q's only after Q's fragments are read.
    f32x4 qf[G];
    put_rows(qst, 0);
    get_frags(qf, 0);
    put_rows(kst[0], 0);
    put_rows(kst[1], 32);
#pragma unroll
    for (int g = 0; g < G; ++g) qf[g] *= p.scale_log2;
    f32x16 s[NSB];
    f32x4 kf[NSB][G];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) get_frags(kf[sb], 32 * sb);
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) {
      s[sb] = f32x16{};
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[sb] = mfma_f32(kf[sb][g][e], qf[g][e], s[sb]);
    }
    fence();
    // The staging registers of K are free since its rows went to LDS.
    load_k(next, more, 0);
    load_k(next, more, 1);
    fence();

    // ---- softmax (exp2 domain, one tile: the running state starts empty) ----
    if constexpr (MASKED) apply_mask<NSB, false, false>(s, 0, kv, qrow, h);
    float mt = s[0][0];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[sb][r]);
    mt = fmaxf(-INFINITY, max_with_other_half(mt));
    // A fully masked row keeps m = -inf; use 0 so exp2(-inf - 0) = 0, never NaN.
    const float m_use = (MASKED && mt == -INFINITY) ? 0.0f : mt;
    float ls = 0.0f;
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pr = fast_exp2(s[sb][r] - m_use);
        s[sb][r] = pr;
        ls += pr;
      }
    fence();

    // ---- O^T = V^T . P^T ----------------------------------------------------
    f32x16 acc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) acc[i] = f32x16{};
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pr = s[sb][r];
        if constexpr (DB == 1) {
          acc[0] = mfma_f32(vf[sb][r], pr, acc[0]);
        } else {
          acc[0] = mfma_f32(vf[sb][r].x, pr, acc[0]);
          acc[1] = mfma_f32(vf[sb][r].y, pr, acc[1]);
        }
      }
      fence();
    }
    load_q(next, more);
    fence();

    // ---- O = acc / l, through the LDS region into whole rows -----------------
    const float lt = sum_with_other_half(ls);
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
#pragma unroll
    for (int j4 = 0; j4 < 4; ++j4) {
      // Block i holds d = DB * row + i; register 4 * j4 + e holds row 8 * j4 + 4h + e,
      // so a lane's d-values for one j4 form one run of 4 * DB (chunks d0 / 4 ..).
      const int d0 = DB * (8 * j4 + 4 * h);
      float vals[4 * DB];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < DB; ++i) vals[DB * e + i] = acc[i][4 * j4 + e] * inv;
#pragma unroll
      for (int c = 0; c < DB; ++c) {
        *reinterpret_cast<f32x4*>(&region[slot(m, d0 / 4 + c)]) =
            f32x4{vals[4 * c], vals[4 * c + 1], vals[4 * c + 2], vals[4 * c + 3]};
      }
    }
    const int ooff = static_cast<int>(((half_row0 + crow) * p.os + 4 * cchunk) * 4);
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const f32x4 o4 = *reinterpret_cast<const f32x4*>(&region[slot(RPI * j + crow, cchunk)]);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o4), ro,
                                             ooff + static_cast<int>(RPI * j * p.os * 4), 0, 0);
    }
    fence();
    load_v(next, more, 0);
    load_v(next, more, 1);
    if (!more) break;
    item = next;
  }
}

// ----------------------------------------------------------------------------
// bf16 / fp16
// ----------------------------------------------------------------------------
template <int D, int BNK = 64>
struct H16Cfg {
  static constexpr int DK = D < 16 ? 16 : D;         // contraction length of Q.K (zero padded)
  static constexpr int BN = BNK;                     // keys per tile (64, or 32)
  static constexpr int NSB = BN / 32;
  static constexpr int CPR = D / 8;                  // 16-byte chunks per key row (8 elems)
  static constexpr int KS = DK + 8;                  // LDS K row stride (elements, 16-byte pad)
  static constexpr int NDB = (D + 31) / 32;          // output blocks of 32 d-rows
  static constexpr int G = DK / 16;                  // Q.K k-steps of 16
  // LDS V row stride (elements) of the row-major V tile.  The 4 key rows one
  // half-wave reads with the transposing load must fall on disjoint banks.
  // Rows stay unpadded and, for head_dim 64 and 128 (VSWZ), 32-column blocks
  // are permuted per row instead: 16-byte chunk c of row r sits in slot
  // c ^ 4*((r >> 1) & 1) (head_dim 64: 128-byte rows, rows r and r + 2 share
  // banks) or c ^ 4*(r & 3) (head_dim 128: 256-byte rows, every row starts on
  // bank 0).  That copies 8 / 16 chunks per row instead of the 12 / 20 of a
  // padded stride.
  static constexpr bool VSWZ = D == 64 || D == 128;
  static constexpr int VS = D;
  static constexpr int VCH = VS / 8;                 // 16-byte chunks per LDS V row
  // Head dims below 32 read up to d = 31 with the transposing load (rows
  // d >= D of the result are never stored); the slack keeps those reads of
  // the last rows inside the buffer.
  static constexpr int VSLACK = 32;
  static constexpr int NSTEP = NSB * 2 * NDB;        // P.V MFMAs per tile
  // Operand prefetch distances (ring depths) of the K and V fragments.
  static constexpr int PDK = 2;
  static constexpr int PDV = 2;
};

// Transposing LDS read (ds_read_b64_tr_b16).  Within each group of 16 lanes,
// lane 4a+c receives element c of the 8-byte rows addressed by lanes a, a+4,
// a+8 and a+12 of the group (in that order).
__device__ __forceinline__ u16x4 lds_read_tr16(const unsigned short* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)(p));
  return __builtin_bit_cast(u16x4, v);
}

// BNK = 32 (head_dim 128 only): 32-key tiles, sized for three workgroups per
// CU, run with the single-score-buffer body and never key-split - for the
// shorter launches, where more resident wavefronts hide more latency than the
// extra per-tile work costs.
template <typename T, int D, bool CAUSAL, bool HAS_MASK, int BNK = 64>
__global__ __launch_bounds__(kThreads, (BNK == 32 ? (D <= 64 ? 4 : 3) : kMinWaves<false, D>)) void attn_fwd_h16_kernel(AttnParams p) {
  using C = H16Cfg<D, BNK>;
  constexpr int BN = C::BN, NSB = C::NSB, CPR = C::CPR, KS = C::KS,
                NDB = C::NDB, VS = C::VS, VCH = C::VCH, G = C::G, NSTEP = C::NSTEP,
                PDK = C::PDK, PDV = C::PDV;
  static_assert(BNK == 64 || (BNK == 32 && D >= 32), "32-key tiles are built for head_dim 32, 64 and 128");
  // The K region also stages the output tile (4 wavefronts x 32 rows of D + 8).
  constexpr int KBUF = (BN * KS > 64 * (D + 8)) ? BN * KS : 64 * (D + 8);
  __shared__ __attribute__((aligned(16))) unsigned short smK[2][KBUF];
  __shared__ __attribute__((aligned(16))) unsigned short smV[2][BN * VS + C::VSLACK];
  __shared__ int sm_span[HAS_MASK ? kSpanLds : 1];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int m = lane & 31;
  const int h = lane >> 5;

  const Work w = work_item(p, CAUSAL);
  const int b = w.bh / p.H;
  const int hh = w.bh - b * p.H;
  const int S = p.S;
  using St = unsigned short;
  const St* __restrict__ Q = static_cast<const St*>(p.q) + b * p.qb + hh * p.qh;
  const St* __restrict__ K = static_cast<const St*>(p.k) + b * p.kb + hh * p.kh;
  const St* __restrict__ V = static_cast<const St*>(p.v) + b * p.vb + hh * p.vh;
  const uint8_t* __restrict__ M = HAS_MASK ? p.mask + b * p.mb : nullptr;

  // The row max is taken on raw scores, which needs a positive scale: a
  // negative scale is folded into Q as an exact sign flip.
  const bool negate = p.scale_log2 < 0.0f;
  float c = negate ? -p.scale_log2 : p.scale_log2;
  // Scale 0 (uniform weights): masked scores are -inf and -inf * 0 is NaN,
  // so 2^-100 stands in.  Masked scores stay -inf, and every allowed score
  // (|s| < 2^75) gives an exp2 argument below 2^-25, so P = 1 exactly.
  if (c == 0.0f) c = 0x1p-100f;
  // The reference max moves once a row's max passes it by more than 8 / c
  // (8 in log2 units, so P <= 2^8).
  float lag = 8.0f / c;
  // Both are wave-uniform: kept in SGPRs (a VOP3 instruction reads one SGPR
  // operand), they leave two more VGPRs to the loop.
  const unsigned short sign = negate ? 0x8000u : 0u;
  c = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(c)));
  lag = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(lag)));

  // K: LDS-DMA into padded rows of KCH 16-byte chunks; DMA instruction j
  // fills chunks [64j, 64j + 64) and the instructions are dealt round-robin
  // to the wavefronts.  A lane landing on the pad chunk - and for head_dim 8
  // on the zero-padded d 8..15, which meets zero Q entries - copies chunk 0
  // again; keys past S copy row S-1 (finite data that the mask neutralises).
  // The (row, chunk) a lane copies is the same for every tile, so its element
  // byte offset from the tile's first key row is computed once (row < 64 and
  // the ABI bounds the key stride below 2^25 elements, so 2 * (row * ks + col)
  // fits 32 bits); lanes past the tile are marked by pos >= BN * KCH.
  constexpr int KCH = KS / 8;
  constexpr int NK = (BN * KCH + 63) / 64;
  constexpr int NW = kThreads / 64;
  constexpr int KPW = (NK + NW - 1) / NW;
  unsigned koff[KPW];
#pragma unroll
  for (int i = 0; i < KPW; ++i) {
    const int pos = 64 * (wave + NW * i) + lane;
    const int row = pos / KCH;
    const int cc = pos - row * KCH;
    koff[i] = 2u * static_cast<unsigned>(row * static_cast<int>(p.ks) + 8 * (cc < CPR ? cc : 0));
  }
  // V: LDS-DMA into unpadded row-major rows of VCH 16-byte chunks (read back
  // with the transposing load); with VSWZ the lane filling slot (row, cc)
  // copies chunk cc ^ vswz(row).
  static_assert(VCH == CPR, "V rows are unpadded");
  auto vswz = [](int row) { return C::VSWZ ? (D == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1)) : 0; };
  constexpr int NV = (BN * VCH + 63) / 64;
  constexpr int VPW = (NV + NW - 1) / NW;
  unsigned voff[VPW];
#pragma unroll
  for (int i = 0; i < VPW; ++i) {
    const int pos = 64 * (wave + NW * i) + lane;
    const int row = pos / VCH;
    const int cc = pos - row * VCH;
    voff[i] = 2u * static_cast<unsigned>(row * static_cast<int>(p.vs) + 8 * (cc ^ vswz(row)));
  }
  // Per-lane base of the transposing V reads: lane i of 16-lane group g
  // addresses key row 4*(g/2) + i/4 and d = 16*(g%2) + 4*(i%4), so lane
  // (m, h) receives V[4h + 0..3][m] (see lds_read_tr16); P.V step (kstep,
  // db) adds 16*kstep rows and 32*db columns, its upper four keys 8 rows.
  // With VSWZ the rows a lane reads all share their low two bits with lane
  // bits 2-3 (16*kstep and 8 rows leave them alone), so the block permutation
  // is one per-lane XOR of the db offset.
  const int vbase = (4 * h + ((lane & 15) >> 2)) * VS + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int vflip = C::VSWZ ? (D == 128 ? 32 * ((lane >> 2) & 3) : 32 * ((lane >> 3) & 1)) : 0;

  {
    // 16-bit workgroups run one query tile (never paired: a second pass costs
    // this kernel more in register pressure than it gains in balance).
    const int qb = w.q_first;
    const int q0 = qb * kBM + wave * 32;
    const int qrow = q0 + m;

    // Keys count from `off` (0 without a key mask): SK of them exist, those
    // from kv_end on are not visited.  Queries and keys compare as qrow - off.
    int off = 0, SK = S;
    int kv_end = CAUSAL ? min(S, (qb + 1) * kBM) : S;
    int whole = 0;  // 64-key tiles 1 .. whole - 1 have no invalid key
    auto skip_keys = [&](int n) __attribute__((always_inline)) {
      off += n;
      SK -= n;
      kv_end -= n;
    };


    bool rm = false;
    auto dma_k = [&](int buf, int t) __attribute__((always_inline)) {
      if constexpr (HAS_MASK) {
        const int key = t * BN + lane;
        rm = lane < BN && key < SK && M[(off + key) * p.ms] != 0;
      }
      const St* kt = K + static_cast<int64_t>(off + t * BN) * p.ks;
      const bool ragged = (t + 1) * BN > SK;
#pragma unroll
      for (int i = 0; i < KPW; ++i) {
        const int j = wave + NW * i;
        const int pos = 64 * j + lane;
        if (j < NK && pos < BN * KCH) {
          if (!ragged) {
            dma16(kt, koff[i], &smK[buf][512 * j]);
          } else {
            // Keys past the last copy it (at or after the tile's first key).
            const int row = pos / KCH;
            const int cc = pos - row * KCH;
            const int rrel = min(t * BN + row, SK - 1) - t * BN;
            dma16(kt, 2u * static_cast<unsigned>(rrel * static_cast<int>(p.ks) + 8 * (cc < CPR ? cc : 0)),
                  &smK[buf][512 * j]);
          }
        }
      }
    };
    // Valid-key bits (key mask and key < S) of tile t as a wave-uniform mask;
    // with a key mask, call after vm_wait() (the mask bytes load in dma_k).
    auto key_bits = [&](int t) __attribute__((always_inline)) -> uint64_t {
      if constexpr (HAS_MASK) {
        return __builtin_amdgcn_ballot_w64(rm);
      } else {
        return range_bits(t * BN, SK);
      }
    };
    auto dma_v = [&](int buf, int t) __attribute__((always_inline)) {
      const St* vt = V + static_cast<int64_t>(off + t * BN) * p.vs;
      const bool ragged = (t + 1) * BN > SK;
#pragma unroll
      for (int i = 0; i < VPW; ++i) {
        const int j = wave + NW * i;
        const int pos = 64 * j + lane;
        if (j < NV && pos < BN * VCH) {
          if (!ragged) {
            dma16(vt, voff[i], &smV[buf][512 * j]);
          } else {
            const int row = pos / VCH;
            const int cc = pos - row * VCH;
            const int rrel = min(t * BN + row, SK - 1) - t * BN;
            dma16(vt, 2u * static_cast<unsigned>(rrel * static_cast<int>(p.vs) + 8 * (cc ^ vswz(row))),
                  &smV[buf][512 * j]);
          }
        }
      }
    };

    // Copies of a tile that lies wholly before S (no ragged rows): the
    // (row, chunk) offsets computed once, no per-lane range test.  With whole
    // 64-lane DMA instructions (BN * VCH and, for 64-key tiles, BN * KCH
    // multiples of 64) the only guard left is the wave-uniform instruction
    // count; the 32-key K tile of head_dim 128 (544 chunks) ends on half an
    // instruction.
    static_assert((BN * VCH) % 64 == 0 && (BN == 32 || (BN * KCH) % 64 == 0), "whole DMA instructions");
    auto dma_k_full = [&](int buf, int t) __attribute__((always_inline)) {
      if constexpr (HAS_MASK) {
        const int key = t * BN + lane;
        rm = lane < BN && M[(off + key) * p.ms] != 0;
      }
      const St* kt = K + static_cast<int64_t>(off + t * BN) * p.ks;
#pragma unroll
      for (int i = 0; i < KPW; ++i) {
        const int j = wave + NW * i;
        if (j < NK && ((BN * KCH) % 64 == 0 || 64 * j + lane < BN * KCH)) {
          dma16(kt, koff[i], &smK[buf][512 * j]);
        }
      }
    };
    auto dma_v_full = [&](int buf, int t) __attribute__((always_inline)) {
      const St* vt = V + static_cast<int64_t>(off + t * BN) * p.vs;
#pragma unroll
      for (int i = 0; i < VPW; ++i) {
        const int j = wave + NW * i;
        if (j < NV) dma16(vt, voff[i], &smV[buf][512 * j]);
      }
    };

    auto kread = [&](int buf, int sb, int g) __attribute__((always_inline)) -> u16x8 {
      const int row = sb * 32 + m;
      return *reinterpret_cast<const u16x8*>(&smK[buf][row * KS + 16 * g + 8 * h]);
    };
    // A operand of P.V step idx = ((sb * 2 + j) * NDB + db): d-row 32*db + m,
    // keys sb*32 + 16j + 4h + {0..3} and sb*32 + 16j + 8 + 4h + {0..3}.  For
    // head dims below 32 the rows d >= D hold other data; they only reach
    // output rows that are never stored.
    auto vread = [&](int buf, int idx) __attribute__((always_inline)) -> u16x8 {
      const int db = idx % NDB;
      const int kstep = idx / NDB;  // sb * 2 + j
      const int col = C::VSWZ ? vbase + ((32 * db) ^ vflip) : vbase + 32 * db;
      const unsigned short* base = &smV[buf][col + 16 * kstep * VS];
      const u16x4 lo = lds_read_tr16(base);
      const u16x4 hi = lds_read_tr16(base + 8 * VS);
      return u16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };

    u16x8 qf[G];
    float m_run = -INFINITY;  // running max of RAW scores
    float m_exp = -INFINITY;  // ceil(m_run * c), kept with m_run
    float l_run = 0.0f;
    f32x16 acc[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) acc[i] = f32x16{};
    // Probabilities of the pending tile in the B-operand layout of the
    // 32x32x16 MFMA: k-step (sb, j) takes registers 8j..8j+7 of sub-block sb,
    // i.e. keys 16j+4h+{0..3} and 16j+8+4h+{0..3}.
    u16x8 pk[NSB * 2];
#pragma unroll
    for (int i = 0; i < NSB * 2; ++i) pk[i] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};

    // S^T = K(buf) . Q^T.  K fragments run PDK groups ahead in a ring: the
    // slot of group g is refilled with group g + PDK right after group g's
    // MFMAs issue, so an LDS read has PDK - 1 groups of MFMAs to land.
    // Only the first L sub-blocks (a compile-time count: the live ones of a
    // masked tile) are computed; the others are left untouched.  A run-time
    // count would put every MFMA of sub-block 1 under its own branch, and the
    // compiler then copies its 16 accumulators through every branch.
    auto qk = [&](auto live_tag, int buf, f32x16 (&s)[NSB]) {
      constexpr int L = decltype(live_tag)::value;
      static_assert(L >= 1 && L <= NSB, "live sub-blocks");
#pragma unroll
      for (int sb = 0; sb < L; ++sb) s[sb] = f32x16{};
      u16x8 kr[PDK][NSB];
#pragma unroll
      for (int i = 0; i < PDK && i < G; ++i)
#pragma unroll
        for (int sb = 0; sb < L; ++sb) kr[i][sb] = kread(buf, sb, i);
#pragma unroll
      for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int sb = 0; sb < L; ++sb) s[sb] = mfma_16(T{}, kr[g % PDK][sb], qf[g], s[sb]);
        if (g + PDK < G) {
#pragma unroll
          for (int sb = 0; sb < L; ++sb) kr[g % PDK][sb] = kread(buf, sb, g + PDK);
        }
        fence();
      }
    };

    // O^T += V^T(buf) . P^T over the first L sub-blocks (compile-time, as in
    // qk); V fragments run PDV steps ahead in a ring.
    auto pv = [&](int buf, auto live_tag) __attribute__((always_inline)) {
      constexpr int L = decltype(live_tag)::value;
      constexpr int nsteps = L * 2 * NDB;
      u16x8 vr[PDV];
#pragma unroll
      for (int i = 0; i < PDV && i < nsteps; ++i) vr[i] = vread(buf, i);
#pragma unroll
      for (int idx = 0; idx < nsteps; ++idx) {
        acc[idx % NDB] = mfma_16(T{}, vr[idx % PDV], pk[idx / NDB], acc[idx % NDB]);
        if (idx + PDV < nsteps) vr[idx % PDV] = vread(buf, idx + PDV);
        fence();
      }
    };
    // Calls f with the live sub-block count n (1 .. NSB) as a compile-time
    // constant.
    auto with_live = [&](int n, auto&& f) __attribute__((always_inline)) {
      if constexpr (NSB == 2) {
        if (n == 2) {
          f(std::integral_constant<int, 2>{});
        } else {
          f(std::integral_constant<int, 1>{});
        }
      } else {
        f(std::integral_constant<int, NSB>{});
      }
    };
    constexpr std::integral_constant<int, NSB> kAllLive{};

    // Lazy reference max: probabilities are exp2(s * c - ceil(m_run * c))
    // against a per-row reference m_run that moves only when the row's max
    // exceeds it by more than 8 / c (so P <= 2^8); the accumulator and the
    // row sum are rescaled only then, for the whole wavefront at once.  The
    // reference exponent is rounded up to an integer, so P = 2^k * exp2(s * c
    // - ceil(max * c)) for an integer k whatever the lag: rounding P to 16
    // bits lands on the same grid as rounding it against the final row max
    // (a power-of-two scale commutes with rounding), and the rescale factor
    // is an exact power of two.  Call after the P.V MFMAs that use the
    // previous reference have been issued.
    auto rebase = [&](float mt) __attribute__((always_inline)) {
      const bool need = mt - m_run > lag;  // false for two -inf
      if (__builtin_amdgcn_ballot_w64(need) != 0) {
        const float m_new = need ? mt : m_run;
        // 1 where the reference stays (also at -inf, where the difference
        // would be NaN), 0 from -inf, else 2^-k.
        const float e_new = ceilf(m_new * c);
        const float alpha = m_new == m_run ? 1.0f : fast_exp2(m_exp - e_new);
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < NDB; ++i) acc[i] *= alpha;
        m_run = m_new;
        m_exp = e_new;
      }
    };
    // Softmax of the first L sub-blocks of s into pn (registers 2L and up of
    // pn are left as they are: P.V and the row sum of this tile skip them).
    auto softmax = [&](auto masked_tag, auto live_tag, f32x16 (&s)[NSB], u16x8 (&pn)[NSB * 2]) {
      constexpr bool MASKED = decltype(masked_tag)::value;
      constexpr int L = decltype(live_tag)::value;
      float mt = s[0][0];
#pragma unroll
      for (int sb = 0; sb < L; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[sb][r]);
      mt = max_with_other_half(mt);
      rebase(mt);
      const float mc = ceilf(((MASKED && m_run == -INFINITY) ? 0.0f : m_run) * c);
#pragma unroll
      for (int sb = 0; sb < L; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float pr = fast_exp2(__builtin_fmaf(s[sb][r], c, -mc));
          pn[sb * 2 + (r >> 3)][r & 7] = to_bits(T{}, pr);
        }
      l_run = add_packed<T, NSB * 2, 2 * L>(pn, l_run);
    };

    // P.V of the pending tile interleaved with the softmax of s: the first
    // half of the k-steps carries the row max, the second half the exp2 and
    // conversion (the steady body of key-masked tiles).
    auto fused = [&](int buf, f32x16 (&s)[NSB], u16x8 (&pn)[NSB * 2]) __attribute__((always_inline)) {
      constexpr int HALF = NSTEP / 2;
      constexpr int E = NSB * 16;      // score elements per lane
      constexpr int PER = E / HALF;    // elements per step in each phase
      float mt = -INFINITY;
      float m_use = 0.0f, alpha = 1.0f, mc = 0.0f;
      bool rebase_any = false;
      u16x8 vr[PDV];
#pragma unroll
      for (int i = 0; i < PDV && i < NSTEP; ++i) vr[i] = vread(buf, i);
#pragma unroll
      for (int idx = 0; idx < NSTEP; ++idx) {
        acc[idx % NDB] = mfma_16(T{}, vr[idx % PDV], pk[idx / NDB], acc[idx % NDB]);
        if (idx + PDV < NSTEP) vr[idx % PDV] = vread(buf, idx + PDV);
        if (idx < HALF) {
#pragma unroll
          for (int j = 0; j < PER; ++j) {
            const int e = PER * idx + j;
            mt = fmaxf(mt, s[e >> 4][e & 15]);
          }
          if (idx == HALF - 1) {
            mt = max_with_other_half(mt);
            // The reference for this tile: rebased now only if some row needs
            // it (the accumulator rescale waits for the last P.V step).
            const bool need = mt - m_run > lag;
            rebase_any = __builtin_amdgcn_ballot_w64(need) != 0;
            m_use = rebase_any && need ? mt : m_run;
            // 1 where the reference stays: a row still at -inf (no allowed
            // key so far) must not turn its zeros into NaN when another row
            // of the wavefront moves.
            alpha = m_use == m_run ? 1.0f : fast_exp2(m_exp - ceilf(m_use * c));
            mc = ceilf((m_use == -INFINITY ? 0.0f : m_use) * c);
          }
        } else {
#pragma unroll
          for (int j = 0; j < PER; ++j) {
            const int e = PER * (idx - HALF) + j;
            const float pr = fast_exp2(__builtin_fmaf(s[e >> 4][e & 15], c, -mc));
            pn[(e >> 4) * 2 + ((e & 15) >> 3)][e & 7] = to_bits(T{}, pr);
          }
        }
        fence();
      }
      if (rebase_any) {
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < NDB; ++i) acc[i] *= alpha;
        m_run = m_use;
        m_exp = ceilf(m_use * c);
      }
      l_run = add_packed<T>(pn, l_run);
    };
    // Pipelined full tiles (no invalid key).  Q.K runs one tile
    // ahead, so each wavefront has matrix-core work beside its softmax VALU
    // work in both halves of a tile (Q.K on its own was the longest stretch
    // of a tile in which the wavefront could issue nothing else):
    //   phase A: S(t+1) = K(t+1).Q^T, interleaved with the exp2 and 16-bit
    //            conversion of S(t) into P(t) against the reference mc;
    //   phase B: O^T += V(t)^T.P(t), interleaved with the row max of S(t+1);
    //            then the row sum of P(t) and the reference decision for
    //            tile t+1 (with the accumulator rescale when it moves).
    auto phase_a = [&](int kbuf, f32x16 (&sn)[NSB], const f32x16 (&s)[NSB], float mc, auto&& hook)
        __attribute__((always_inline)) {
      constexpr int NQK = G * NSB;  // Q.K MFMAs of a tile
      constexpr int E = NSB * 16;   // score elements per lane
      constexpr int PER = E / NQK;  // exp2 per MFMA
      static_assert(E % NQK == 0, "the softmax work divides over the Q.K steps");
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) sn[sb] = f32x16{};
      u16x8 kr[PDK][NSB];
#pragma unroll
      for (int i = 0; i < PDK && i < G; ++i)
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb) kr[i][sb] = kread(kbuf, sb, i);
#pragma unroll
      for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb) {
          sn[sb] = mfma_16(T{}, kr[g % PDK][sb], qf[g], sn[sb]);
#pragma unroll
          for (int j = 0; j < PER; ++j) {
            const int e = PER * (g * NSB + sb) + j;
            const float pr = fast_exp2(__builtin_fmaf(s[e >> 4][e & 15], c, -mc));
            pk[(e >> 4) * 2 + ((e & 15) >> 3)][e & 7] = to_bits(T{}, pr);
          }
        }
        if (g + PDK < G) {
#pragma unroll
          for (int sb = 0; sb < NSB; ++sb) kr[g % PDK][sb] = kread(kbuf, sb, g + PDK);
        }
        hook(g);
        fence();
      }
    };
    // ADD_SUM: whether P(t) still has to enter the row sum (the generic
    // softmax counts its P when producing it).
    auto phase_b = [&](auto add_sum_tag, int vbuf, const f32x16 (&sn)[NSB], auto&& hook)
        __attribute__((always_inline)) {
      constexpr bool ADD_SUM = decltype(add_sum_tag)::value;
      constexpr int E = NSB * 16;
      constexpr int PER = E / NSTEP;  // max operands per P.V MFMA
      static_assert(E % NSTEP == 0, "the row max divides over the P.V steps");
      float mt = -INFINITY;
      u16x8 vr[PDV];
#pragma unroll
      for (int i = 0; i < PDV && i < NSTEP; ++i) vr[i] = vread(vbuf, i);
#pragma unroll
      for (int idx = 0; idx < NSTEP; ++idx) {
        acc[idx % NDB] = mfma_16(T{}, vr[idx % PDV], pk[idx / NDB], acc[idx % NDB]);
        if (idx + PDV < NSTEP) vr[idx % PDV] = vread(vbuf, idx + PDV);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
          const int e = PER * idx + j;
          mt = fmaxf(mt, sn[e >> 4][e & 15]);
        }
        hook(idx);
        fence();
      }
      if constexpr (ADD_SUM) l_run = add_packed<T>(pk, l_run);
      rebase(max_with_other_half(mt));
    };
    // Reference exponent of the current tile (without a key mask every row
    // of a full tile has finite scores after tile 0).
    auto ref_exp = [&]() __attribute__((always_inline)) -> float { return m_exp; };

    // Keys of this workgroup: all of the query tile's, or one chunk of them on
    // the key-split grid.  The copy of the first tile and the Q loads run under
    // the mask scan (the copy is repeated if the scan moves the first key).
    int kt0 = 0, kt1 = (kv_end + BN - 1) / BN;
    if (w.nchunk > 1) {
      const int csz = (kt1 + w.nchunk - 1) / w.nchunk;
      kt0 = w.chunk * csz;
      kt1 = min(kt1, kt0 + csz);
      if constexpr (HAS_MASK) {
        kv_end = min(kv_end, kt1 * BN);
        skip_keys(kt0 * BN);
        kt1 -= kt0;
        kt0 = 0;
      }
    }
    dma_k(kt0 & 1, kt0);
    // B operand of S^T = K.Q^T: k-step g covers d = 16g..16g+15, lane half h
    // holds d = 16g+8h..16g+8h+7.
    // Without branches, and not used before the scan: rows past S and the zero
    // padding of head_dim 8 load other values and are cleared below.
#pragma unroll
    for (int g = 0; g < G; ++g) {
      qf[g] = *reinterpret_cast<const u16x8*>(Q + min(qrow, S - 1) * p.qs + min(16 * g + 8 * h, D - 8));
    }
    if constexpr (HAS_MASK) {
      if (kv_end > kSpanKeys && p.ms == 1) {
        const KeySpan span = scan_keys<St, std::is_same<T, BF16>::value ? 0x7f80u : 0x7c00u, D>(
            M + off, V + off * p.vs, p.vs, kv_end, sm_span);
        kv_end = __builtin_amdgcn_readfirstlane(span.end);
        whole = __builtin_amdgcn_readfirstlane(span.full);
        if (span.first > 0) {
          skip_keys(__builtin_amdgcn_readfirstlane(span.first));
          vm_wait();
          dma_k(0, 0);
        }
        kt1 = (kv_end + BN - 1) / BN;
      }
    }

#pragma unroll
    for (int g = 0; g < G; ++g) {
      const bool real = qrow < S && 16 * g + 8 * h < D;
      qf[g] = real ? qf[g] ^ sign : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    vm_wait();
    uint64_t kvalid = key_bits(kt0);
    __syncthreads();

    // Tiles before n_full are "full" for this wavefront: every sub-block
    // live, no causal or ragged-end masking (a key mask may still apply).
    // Tiles (kt0, n_full) run a branch-free steady body; tile kt0 and the
    // tail use the generic body.  Every path executes one barrier per tile,
    // so all wavefronts meet kt1 - kt0 barriers.
    const int n_full = q0 >= S ? 0
                               : min(kt1, min(SK / BN, CAUSAL ? max(0, q0 + 1 - off) / BN : kt1));
    bool pending = false;  // a tile's P.V is still to be accumulated (uniform)
    int pend_live = 0;     // its number of live sub-blocks

    auto finish_tile = [&](int t) __attribute__((always_inline)) {
      vm_wait();
      const uint64_t kvalid_next = key_bits(t + 1);
      __syncthreads();
      kvalid = kvalid_next;
    };
    auto generic_tile = [&](int t) __attribute__((always_inline)) {
      const int kb = t & 1;
      // K(t+1) goes to the buffer K(t-1) used, V(t) to the one V(t-2) used;
      // neither is read in this iteration.
      if (t + 1 < kt1) dma_k(kb ^ 1, t + 1);
      dma_v(kb, t);
      const int k0 = t * BN;
      const bool live = q0 < S && (!CAUSAL || k0 <= q0 + 31 - off);
      int nlive = NSB;
#pragma unroll
      for (int sb = NSB - 1; sb >= 0; --sb) {
        const int ks = k0 + sb * 32;
        if (ks >= SK || (CAUSAL && ks > q0 + 31 - off)) nlive = sb;
      }
      if (pending) with_live(pend_live, [&](auto lt) __attribute__((always_inline)) { pv(kb ^ 1, lt); });
      if (live) {
        // pn registers past the live sub-blocks are left unset: P.V and the
        // row sum of this tile never read them.  The copy into pk stays out
        // of the branches (stores to pk that differ per branch would be
        // merged into one store at a selected index, which moves pk to
        // scratch memory).
        u16x8 pn[NSB * 2];
        with_live(nlive, [&](auto lt) __attribute__((always_inline)) {
          f32x16 s[NSB];
          qk(lt, kb, s);
          apply_mask<NSB, CAUSAL, true, decltype(lt)::value>(s, k0, kvalid, qrow - off, h);
          softmax(std::true_type{}, lt, s, pn);
        });
#pragma unroll
        for (int i = 0; i < NSB * 2; ++i) pk[i] = pn[i];
        pend_live = nlive;
      }
      pending = live;
      finish_tile(t);
    };

    generic_tile(kt0);
    constexpr bool kPipe = BNK == 64 && (!HAS_MASK || D >= 64);
    const int n_pipe = HAS_MASK ? min(n_full, whole) : n_full;
    if constexpr (kPipe) if (n_pipe - kt0 >= 2) {
      // Every interval between two barriers copies and reads the same buffers
      // as the generic tile of that index (K(tau+1), V(tau) in; K(tau),
      // V(tau-1) read), so wavefronts on different paths stay in step.
      // S(t) lives in sa when t - kt0 is odd and in sb when it is even.
      f32x16 sa[NSB], sb[NSB];
      const int t1 = kt0 + 1;
      // Tile t1: S(t1) with nothing to overlap, then P.V(kt0) with its row max.
      if (t1 + 1 < n_pipe) {
        dma_k_full((t1 + 1) & 1, t1 + 1);
      } else if (t1 + 1 < kt1) {
        dma_k((t1 + 1) & 1, t1 + 1);
      }
      dma_v_full(t1 & 1, t1);
      qk(kAllLive, t1 & 1, sa);
      phase_b(std::false_type{}, kt0 & 1, sa, [](int) {});
      finish_tile(t1);
      // Tile t + 1 for t = t1 .. n_pipe - 2.
      auto steady = [&](int t, const f32x16 (&cur)[NSB], f32x16 (&nxt)[NSB])
          __attribute__((always_inline)) {
        const int kb = t & 1;
        // The copies of K(t+2) and V(t+1) are spread over the MFMA groups of
        // both phases instead of issued back to back at the top of the tile.
        static_assert(KPW <= G && 2 * VPW - 1 <= NSTEP, "a copy slot for every copy");
        const bool kfull = t + 2 < n_pipe;
        if (!kfull && t + 2 < kt1) dma_k(kb, t + 2);
        const St* kt = K + static_cast<int64_t>(off + (t + 2) * BN) * p.ks;
        const St* vt = V + static_cast<int64_t>(off + (t + 1) * BN) * p.vs;
        phase_a(kb ^ 1, nxt, cur, ref_exp(), [&](int g) __attribute__((always_inline)) {
          if (g < KPW) {
            const int j = wave + NW * g;
            if (kfull && j < NK) dma16(kt, koff[g], &smK[kb][512 * j]);
          }
        });
        phase_b(std::true_type{}, kb, nxt, [&](int idx) __attribute__((always_inline)) {
          if (idx % 2 == 0 && idx / 2 < VPW) {
            const int i = idx / 2;
            const int j = wave + NW * i;
            if (j < NV) dma16(vt, voff[i], &smV[kb ^ 1][512 * j]);
          }
        });
        finish_tile(t + 1);
      };
      int t = t1;
      for (; t + 2 < n_pipe; t += 2) {
        steady(t, sa, sb);
        steady(t + 1, sb, sa);
      }
      if (t + 1 < n_pipe) {
        steady(t, sa, sb);
        ++t;
      }
      // Tile n_pipe - 1: its P becomes the pending P.V of the next tile.
      const float mc = ref_exp();
      auto last_p = [&](const f32x16 (&cur)[NSB]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NSB * 16; ++e) {
          const float pr = fast_exp2(__builtin_fmaf(cur[e >> 4][e & 15], c, -mc));
          pk[(e >> 4) * 2 + ((e & 15) >> 3)][e & 7] = to_bits(T{}, pr);
        }
      };
      if ((t - kt0) & 1) {
        last_p(sa);
      } else {
        last_p(sb);
      }
      l_run = add_packed<T>(pk, l_run);
      pending = true;
      pend_live = NSB;
    }
    if constexpr (HAS_MASK || BNK == 32) {
      // The rest of a key-masked launch - scattered invalid keys, or head dims
      // below 64, where the pipelined body costs an occupancy step (bf16
      // [8, 1024, 16, 32] with scattered keys 45 -> 51 us) - and 32-key tiles,
      // whose three workgroups per CU leave no room for it, keep one score
      // buffer.
      for (int t = kPipe ? max(kt0 + 1, n_pipe) : kt0 + 1; t < n_full; ++t) {
        const int kb = t & 1;
        if (t + 1 < n_full) {
          dma_k_full(kb ^ 1, t + 1);
        } else if (t + 1 < kt1) {
          dma_k(kb ^ 1, t + 1);
        }
        dma_v_full(kb, t);
        f32x16 s[NSB];
        u16x8 pn[NSB * 2];
        qk(kAllLive, kb, s);
        if (HAS_MASK && kvalid != range_bits(0, BN)) apply_mask<NSB, false>(s, t * BN, kvalid, qrow, h);
        fused(kb ^ 1, s, pn);
#pragma unroll
        for (int i = 0; i < NSB * 2; ++i) pk[i] = pn[i];
        finish_tile(t);
      }
    }
    for (int t = max(kt0 + 1, n_full); t < kt1; ++t) generic_tile(t);
    if (pending) with_live(pend_live, [&](auto lt) __attribute__((always_inline)) { pv((kt1 - 1) & 1, lt); });

    if (BNK == 64 && w.nchunk > 1) {
      // Key-split query tile: publish this chunk's state - per lane the
      // integer reference exponent E (-inf for a row with no key yet), the
      // lane half's row sum and the 16 * NDB accumulator values, stored
      // lane-major so every access is coalesced - then count the chunk in.
      // The chunk that arrives last merges all states; E differs between
      // chunks by integers, so every rescale is an exact power of two.
      //
      // Coherence without cache-wide maintenance: the chunks of a tile may
      // run on different XCDs, whose L2 caches are not coherent, and an
      // agent-scope fence would write back and invalidate a whole L2 (the
      // K/V tiles every other workgroup on that XCD streams from).  Instead
      // only the exchanged words are coherent: the states are written and
      // read with system-scope relaxed atomics (write-through stores,
      // cache-bypassing loads), each wavefront waits for its stores to
      // complete (vmcnt) before the barrier that precedes the counter
      // increment, and the last chunk reads the states only after its
      // increment has returned.
      constexpr int NV = NDB * 16 + 2;  // floats per lane
      const int slot = w.bh * p.split_tiles + (qb - p.split_q0);
      float* const base = p.ws_part + static_cast<int64_t>(slot) * p.split_maxch * 4 * NV * 64;
      auto state = [&](int ch) __attribute__((always_inline)) -> float* {
        return base + static_cast<int64_t>(ch * 4 + wave) * NV * 64 + lane;
      };
      auto put = [](float* a, float v) __attribute__((always_inline)) {
        __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      };
      auto get = [](const float* a) __attribute__((always_inline)) -> float {
        return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      };
      const float e_own = m_run == -INFINITY ? -INFINITY : ceilf(m_run * c);
      {
        float* st = state(w.chunk);
        put(st, e_own);
        put(st + 64, l_run);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) put(st + (2 + db * 16 + r) * 64, acc[db][r]);
      }
      vm_wait();
      __syncthreads();
      int* const counter = &p.ws_cnt[slot];
      int* arrival = reinterpret_cast<int*>(&smV[0][0]);  // V buffers are idle now
      if (tid == 0) {
        *arrival = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
      __syncthreads();
      if (*arrival != w.nchunk - 1) return;  // another chunk finishes this tile
      float e_max = -INFINITY;
      for (int ch = 0; ch < w.nchunk; ++ch) e_max = fmaxf(e_max, ch == w.chunk ? e_own : get(state(ch)));
      // Sum the chunks in chunk order, so the result does not depend on which
      // one arrived last.
      f32x16 own[NDB];
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        own[db] = acc[db];
        acc[db] = f32x16{};
      }
      const float l_own = l_run;
      l_run = 0.0f;
      for (int ch = 0; ch < w.nchunk; ++ch) {
        const float* st = state(ch);
        const float e = ch == w.chunk ? e_own : get(st);
        const float a = (e == -INFINITY) ? 0.0f : fast_exp2(e - e_max);
        if (ch == w.chunk) {
          l_run += a * l_own;
#pragma unroll
          for (int db = 0; db < NDB; ++db) acc[db] += a * own[db];
        } else {
          l_run += a * get(st + 64);
#pragma unroll
          for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[db][r] += a * get(st + (2 + db * 16 + r) * 64);
        }
      }
      // Ready for the next launch (the launch boundary orders it).
      if (tid == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }

    // Output through LDS: the accumulator layout gives a lane 4 consecutive
    // d of one query per register group, so direct stores would write 16
    // bytes into each of 32 rows per instruction (partial cache lines).  The
    // wavefront's 32 x D tile goes to its own slice of the K buffers instead
    // (no K read or copy is pending after the loop's last barrier) and comes
    // back as whole 16-byte row chunks, so each store covers whole rows.
    const float lt = sum_with_other_half(l_run);
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    constexpr int OS = D + 8;  // staged row stride (elements; 16-byte pad)
    static_assert(4 * 32 * OS <= 2 * KBUF, "output staging fits the K buffers");
    unsigned short* so = &smK[0][0] + wave * 32 * OS;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int j4 = 0; j4 < 4; ++j4) {
        const int d0 = 32 * db + 8 * j4 + 4 * h;  // 4 consecutive d-rows
        if (D < 32 && d0 >= D) continue;
        u16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = to_bits(T{}, acc[db][4 * j4 + e] * inv);
        *reinterpret_cast<u16x4*>(so + m * OS + d0) = o;
      }
    __builtin_amdgcn_wave_barrier();
    constexpr int OCH = D / 8;  // 16-byte chunks per output row
    St* __restrict__ O = static_cast<St*>(p.out) + b * p.ob + hh * p.oh;
#pragma unroll
    for (int i0 = 0; i0 < 32 * OCH; i0 += 64) {
      const int i = i0 + lane;
      const int row = i / OCH;
      const int cc = i - row * OCH;
      if ((32 * OCH % 64 == 0 || i < 32 * OCH) && q0 + row < S) {
        *reinterpret_cast<u16x8*>(O + (q0 + row) * p.os + 8 * cc) =
            *reinterpret_cast<const u16x8*>(so + row * OS + 8 * cc);
      }
    }
  }
}

// ----------------------------------------------------------------------------
// fp32 on the bf16 matrix cores (head_dim 32, 64, 128)
// ----------------------------------------------------------------------------
// The fp32 MFMA has 1/16 of the bf16 rate, and the fp32 MFMA form of this
// kernel ran at up to 0.79 of its peak.  Here every operand - scaled Q, K, V
// and the probabilities - is the sum of three bf16 terms (bf16x3.h) and each
// product the six products of terms that matter, 16/6 of the fp32 MFMA's rate
// at best.  The small and the leading products of a Q.K have an accumulator
// each, so its sum is rounded D / 16 times, and once more where a VALU addition
// joins the two.  (Leading products accumulated onto the small ones lose more
// than a rounding in the matrix core's alignment: scores of one product each,
// rising to 220 over 512 keys, gave 1.2 - 1.35 times the error of rounded
// products, 1.02 - 1.05 in two sums.  The additions cost no measurable time.)
//
// One workgroup = 4 wavefronts x 32 queries; 32-key tiles.  A tile's K and V
// rows are loaded into registers a tile ahead (16 bytes a lane, through a
// buffer resource that ends with the tile's last row, so no bounds branches),
// split once for the workgroup and written to LDS as three row-major bf16
// planes: K rows padded by 16 bytes, V rows unpadded with permuted column
// blocks and read with the transposing load, as in the 16-bit kernel.  All of
// that sits in the shadow of the Q.K MFMAs (one staged 4-value chunk per six
// MFMAs), the softmax and the split of P in the shadow of the previous tile's
// P.V MFMAs, and the tile's one barrier between the two halves, so fragments
// for the start of either half are read before it.  P's reference max lags
// (see the 16-bit kernel), so the accumulators are rescaled rarely.
//
// It is bound by VALU issue and the power limit together: per wavefront and
// 32-key tile at head_dim 64, 48 MFMAs against ~350 VALU instructions (144 of
// softmax and 88 of P's split for 16 scores a lane, 88 of staging, 16 that join
// the two sums); at [8, 1024, 16, 64] causal 7.7 other VALU instructions are
// issued per MFMA and the matrix pipe is busy 39 % of the cycles.  Against the
// fp32 MFMA kernel: causal [8, 1024, 16, 64] 157 -> 117 us (147 TFLOP/s), [8,
// 4096, 16, 64] 2191 -> 1495 us (184), [8, 1024, 16, 128] 377 -> 235 us, [8, 1024,
// 16, 32] 85 -> 67 us; non-causal key-masked [3, 777, 12, 128] 132 -> 84 us (70 -
// 82 with scan_keys, by the lengths).  Error against float64: 0.5 - 0.8 of the
// fp32 MFMA kernel's.
//
// PACK: heads of up to 64 keys have rows for one or two wavefronts, and a
// workgroup for each of them is a chain of load, split, store and barrier around
// one or two tiles of work.  Up to four of them share a workgroup: their tiles
// follow one another through the same pipeline, and each wavefront works on its
// own head's.  [512, 16, 8, 128] non-causal 152 -> 76 us (102 on the fp32 MFMA
// kernel), causal 162 -> 76 (155); [512, 33, 8, 128] 207 -> 161 (146), causal
// 219 -> 154 (263); causal [512, 16, 8, 64] 52 -> 30 (52), [512, 64, 8, 64]
// key-masked 85 -> 66 (101).
//
// A row with a non-finite operand in reach (or one that rounds to infinity)
// comes out non-finite, and one of values too small for three terms below
// 2^-80; its wavefront then computes its 32 rows again on the fp32 MFMA
// straight from global memory, which gives what plain fp32 arithmetic gives.
template <int D>
struct X3Cfg {
  static constexpr int BN = 32;              // keys per tile
  static constexpr int G = D / 16;           // Q.K k-steps of 16
  static constexpr int NDB = D / 32;         // output blocks of 32 d-rows
  static constexpr int CPR = D / 4;          // 4-value chunks per row
  static constexpr int CPT = D / 32;         // chunks of K (and of V) per thread
  static constexpr int KS = D + 8;           // LDS K row stride (bf16, 16-byte pad)
  static constexpr int KPL = BN * KS;        // one term of a K tile
  static constexpr int VPL = BN * D;         // one term of a V tile
  static constexpr bool VSWZ = D >= 64;      // V column blocks permuted per row (see H16Cfg)
};
// Workgroups per CU: head_dim 128 keeps its Q terms, accumulators and operand
// rings in up to 512 registers.
template <int D>
constexpr int kX3Groups = D >= 128 ? 1 : 2;

template <int D, bool CAUSAL, bool HAS_MASK, bool PACK = false>
__global__ __launch_bounds__(kThreads, kX3Groups<D>) void attn_fwd_x3_kernel(AttnParams p) {
  using C = X3Cfg<D>;
  constexpr int BN = C::BN, G = C::G, NDB = C::NDB, CPR = C::CPR, CPT = C::CPT, KS = C::KS, KPL = C::KPL,
                VPL = C::VPL;
  using St = unsigned short;
  __shared__ __attribute__((aligned(16))) St smK[2][3 * KPL];
  __shared__ __attribute__((aligned(16))) St smV[3][3 * VPL];
  __shared__ int sm_span[HAS_MASK ? kSpanLds : 1];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int m = lane & 31;
  const int h = lane >> 5;

  const int S = p.S;
  // PACK: a head takes tph wavefronts and tiles, tile t is tile t % tph of the
  // workgroup's head t / tph, and a wavefront works on those of its own head
  // from t_lo on.
  const int tph = PACK ? (S > BN ? 2 : 1) : 1;
  const int bh0 = PACK ? static_cast<int>(blockIdx.x) * p.pack : 0;
  const int heads = PACK ? min(p.pack, p.BH - bh0) : 1;
  const int slot = PACK ? wave / tph : 0;
  const int t_lo = PACK ? min(slot, heads) * tph : 0;
  const Work w = PACK ? Work{bh0 + min(slot, heads - 1), 0, 0, 1, 0, 1} : work_item(p, CAUSAL);
  const int b = w.bh / p.H;
  const int hh = w.bh - b * p.H;
  const float* __restrict__ Q = static_cast<const float*>(p.q) + b * p.qb + hh * p.qh;
  const float* K = static_cast<const float*>(p.k) + b * p.kb + hh * p.kh;
  const float* V = static_cast<const float*>(p.v) + b * p.vb + hh * p.vh;
  const uint8_t* M = HAS_MASK ? p.mask + b * p.mb : nullptr;
  // Keys count from `off` (0 without a key mask), SK of them exist.
  int off = 0, SK = S;

  const float* const kt = PACK ? static_cast<const float*>(p.k) : nullptr;
  const float* const vt = PACK ? static_cast<const float*>(p.v) : nullptr;
  // Staging: chunk i of a thread is 4 values of row `srow + i * 256 / CPR`.
  constexpr int RPI = kThreads / CPR;  // rows per staging pass
  const int srow = tid / CPR;
  const int sc = tid - srow * CPR;
  // A tile's rows are read through a buffer resource that ends with row S - 1:
  // rows past it read as zeros (or, where rows overlap, as other rows: the
  // mask neutralises them), without a branch.
  f32x4 rk[CPT], rv[CPT];
  unsigned koff[CPT], voff[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    koff[i] = (static_cast<unsigned>(srow + RPI * i) * static_cast<unsigned>(p.ks) + 4u * sc) * 4u;
    voff[i] = (static_cast<unsigned>(srow + RPI * i) * static_cast<unsigned>(p.vs) + 4u * sc) * 4u;
  }
  // (PACK: `base` is the tensor's and has the strides of its batches and heads.)
  auto tile_rsrc = [&](const float* base, int64_t rs, int64_t bs, int64_t hs, int t) __attribute__((always_inline)) {
    if constexpr (PACK) {
      const int th = min(t / tph, heads), bh = bh0 + th, tb = bh / p.H;
      if (th < heads) base += tb * bs + (bh - tb * p.H) * hs;
      t = th < heads ? t % tph : tph;
    }
    const int rows = min(SK - t * BN, BN);
    const unsigned bytes = rows > 0 ? (static_cast<unsigned>(rows - 1) * static_cast<unsigned>(rs) + D) * 4u : 0u;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + (rows > 0 ? static_cast<int64_t>(t) * BN * rs : 0)),
                                             static_cast<short>(0), static_cast<int>(bytes), 0x00020000);
  };
  auto k_rsrc = [&](int t) __attribute__((always_inline)) { return tile_rsrc(PACK ? kt : K, p.ks, p.kb, p.kh, t); };
  auto v_rsrc = [&](int t) __attribute__((always_inline)) { return tile_rsrc(PACK ? vt : V, p.vs, p.vb, p.vh, t); };
  auto load4 = [](const __amdgpu_buffer_rsrc_t& r, unsigned off) __attribute__((always_inline)) -> f32x4 {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(off), 0, 0));
  };
  auto put = [&](St* dst, int plane, const unsigned (&lo)[3], const unsigned (&hi)[3]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x2*>(dst + t * plane) = u32x2{lo[t], hi[t]};
  };
  unsigned s_lo[3], s_hi[3];  // terms of the chunk being staged
  St* const kdst = &smK[0][srow * KS + 4 * sc];
  // 16-byte chunk c of V row r sits at c ^ 4 ((r >> 1) & 1) (head_dim 64) or
  // c ^ 4 (r & 3) (128); 32 rows per pass of head_dim 32, else a pass adds a
  // multiple of 4 rows for 64 and of 8 for 128.
  const int vswz = C::VSWZ ? (D == 128 ? 4 * (srow & 3) : 4 * ((srow >> 1) & 1)) : 0;
  St* const vdst = &smV[0][srow * D + 8 * ((sc >> 1) ^ vswz) + 4 * (sc & 1)];

  const int vbase = (4 * h + ((lane & 15) >> 2)) * D + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int vflip = C::VSWZ ? (D == 128 ? 32 * ((lane >> 2) & 3) : 32 * ((lane >> 3) & 1)) : 0;
  auto kread = [&](int buf, int term, int g) __attribute__((always_inline)) -> u32x4 {
    return *reinterpret_cast<const u32x4*>(&smK[buf][term * KPL + m * KS + 16 * g + 8 * h]);
  };
  // A operand of P.V: d-row 32 db + m, keys 16 j + 4 h + {0..3} and + 8.
  auto vread = [&](int buf, int term, int j, int db) __attribute__((always_inline)) -> u32x4 {
    const int col = C::VSWZ ? vbase + ((32 * db) ^ vflip) : vbase + 32 * db;
    const St* base = &smV[buf][term * VPL + col + 16 * j * D];
    const u32x2 lo = __builtin_bit_cast(u32x2, lds_read_tr16(base));
    const u32x2 hi = __builtin_bit_cast(u32x2, lds_read_tr16(base + 8 * D));
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };

  // The first tile's pending P is zero; what it multiplies must be finite.
  for (int i = tid; i < 3 * VPL / 8; i += kThreads) reinterpret_cast<u32x4*>(smV[2])[i] = u32x4{0u, 0u, 0u, 0u};

  for (int pass = 0; pass < w.npass; ++pass) {
    const int qb = pass == 0 ? w.q_first : w.q_second;
    const int q0 = PACK ? (slot < heads ? (wave % tph) * 32 : 2 * BN) : qb * kBM + wave * 32;
    const int qrow = q0 + m;
    int kv_end = CAUSAL ? min(S, (qb + 1) * kBM) : S;
    if constexpr (HAS_MASK && !PACK) {
      K -= static_cast<int64_t>(off) * p.ks;
      V -= static_cast<int64_t>(off) * p.vs;
      M -= static_cast<int64_t>(off) * p.ms;
      off = 0;
      if (kv_end > kSpanKeys && p.ms == 1) {
        const KeySpan span = scan_keys<float, 0x7f800000u, D>(M, V, p.vs, kv_end, sm_span);
        off = span.first;
        kv_end = span.end - off;
        K += static_cast<int64_t>(off) * p.ks;
        V += static_cast<int64_t>(off) * p.vs;
        M += static_cast<int64_t>(off) * p.ms;
      }
      SK = S - off;
    }
    const int ntiles = PACK ? heads * tph : (kv_end + BN - 1) / BN;
    // Tiles with keys for this wavefront: up to nlive, of PACK those from t_lo.
    const int own = q0 >= S ? 0 : (CAUSAL ? q0 / BN + 1 : tph);
    const int nlive = PACK ? t_lo + own : q0 >= S ? 0 : (CAUSAL ? min(ntiles, (max(-BN, q0 + 31 - off) + BN) / BN) : ntiles);

    bool rm = false;
    auto load_mask = [&](int t) __attribute__((always_inline)) {
      if constexpr (HAS_MASK) {
        const uint8_t* mrow = PACK ? p.mask + (bh0 + t / tph) / p.H * p.mb : M;
        const int key = (PACK ? t % tph : t) * BN + m;
        rm = h == 0 && key < SK && mrow[key * p.ms] != 0;
      }
    };
    auto key_bits = [&](int t) __attribute__((always_inline)) -> uint64_t {
      if constexpr (HAS_MASK) return __builtin_amdgcn_ballot_w64(rm);
      return range_bits((PACK ? t % tph : t) * BN, SK);
    };

    // Prologue: K(0) into its buffer, K(1) and V(0) into registers.
    load_mask(0);
    {
      const auto r0 = k_rsrc(0);
#pragma unroll
      for (int i = 0; i < CPT; ++i) rk[i] = load4(r0, koff[i]);
    }
    // B operand of S^T = K.Q^T: k-step g, lane half h: d = 16 g + 8 h .. + 7,
    // pre-scaled into exp2 units.
    Split8 qf[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      f32x4 a = {0.f, 0.f, 0.f, 0.f}, c = a;
      if (qrow < S) {
        a = *reinterpret_cast<const f32x4*>(Q + qrow * p.qs + 16 * g + 8 * h) * p.scale_log2;
        c = *reinterpret_cast<const f32x4*>(Q + qrow * p.qs + 16 * g + 8 * h + 4) * p.scale_log2;
      }
      split_pair(qf[g], 0, a[0], a[1]);
      split_pair(qf[g], 1, a[2], a[3]);
      split_pair(qf[g], 2, c[0], c[1]);
      split_pair(qf[g], 3, c[2], c[3]);
    }
    {
      const auto k1 = k_rsrc(1), v0 = v_rsrc(0);
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        split_pair(rk[i][0], rk[i][1], s_lo[0], s_lo[1], s_lo[2]);
        split_pair(rk[i][2], rk[i][3], s_hi[0], s_hi[1], s_hi[2]);
        put(kdst + RPI * i * KS, KPL, s_lo, s_hi);
        rk[i] = load4(k1, koff[i]);
        rv[i] = load4(v0, voff[i]);
      }
    }
    uint64_t kvalid = key_bits(0);
    __syncthreads();

    float m_run = -INFINITY;  // reference max (exp2 units) that P is taken against
    float l_run = 0.0f;       // partial sum over this lane half's keys
    f32x16 acc[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) acc[i] = f32x16{};
    Split8 pk[2];  // pending P: k-step j holds registers 8 j .. 8 j + 7 of S^T
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 3; ++t) pk[j].t[t] = u32x4{0u, 0u, 0u, 0u};

    // Chunk c of the staging work of iteration t (K(t + 1), V(t), interleaved):
    // steps 0 and 1 split its pairs, step 2 writes it to LDS and loads the
    // chunk of the tile after.
    St* kput = kdst + 3 * KPL;  // where K(t + 1) goes
    St* vput = vdst;            // where V(t) goes: V(t) lives in buffer t % 3
    int vb = 2;                 // buffer of V(t - 1)
    __amdgpu_buffer_rsrc_t knext = k_rsrc(2), vnext = v_rsrc(1);
    auto stage = [&](int c, int step) __attribute__((always_inline)) {
      const int i = c >> 1;
      f32x4& r = (c & 1) ? rv[i] : rk[i];
      if (step == 0) {
        split_pair(r[0], r[1], s_lo[0], s_lo[1], s_lo[2]);
      } else if (step == 1) {
        split_pair(r[2], r[3], s_hi[0], s_hi[1], s_hi[2]);
      } else if (c & 1) {
        put(vput + RPI * i * D, VPL, s_lo, s_hi);
        rv[i] = load4(vnext, voff[i]);
      } else {
        put(kput + RPI * i * KS, KPL, s_lo, s_hi);
        rk[i] = load4(knext, koff[i]);
      }
    };
    // P.V products of one k-step, in order of V's term; fragments are read two
    // terms ahead.
    constexpr int kVT[6] = {2, 1, 1, 0, 0, 0};
    constexpr int kPT[6] = {0, 1, 0, 2, 1, 0};
    constexpr int NPV = 12 * NDB;
    u32x4 vr[3][NDB];
    auto v_frag = [&](int vbuf, int s) __attribute__((always_inline)) {  // s: k-step * 3 + (2 - term)
#pragma unroll
      for (int db = 0; db < NDB; ++db) vr[s % 3][db] = vread(vbuf, 2 - s % 3, s / 3, db);
    };
    // MFMA n of P.V: k-step n / (6 NDB), product (n / NDB) % 6, block n % NDB.
    auto pv_mfma = [&](int vbuf, int n) __attribute__((always_inline)) {
      const int j = n / (6 * NDB), pr = (n / NDB) % 6, db = n % NDB;
      const int s = 3 * j + 2 - kVT[pr];
      acc[db] = mfma_x3(vr[s % 3][db], pk[j].t[kPT[pr]], acc[db]);
      if (db == 0 && (pr == 0 || pr == 1 || pr == 3) && s + 2 < 6) v_frag(vbuf, s + 2);
    };
    // K fragments: the two small terms of this and the next k-step, the leading
    // term of every k-step.
    u32x4 kr[2][2], k0f[G];
    auto k_frag = [&](int buf, int g) __attribute__((always_inline)) {
      kr[g & 1][0] = kread(buf, 2, g);
      kr[g & 1][1] = kread(buf, 1, g);
      k0f[g] = kread(buf, 0, g);
    };
    if constexpr (!PACK) k_frag(0, 0);

    // Iteration t: S(t) = K(t).Q^T with the staging of K(t + 1) and V(t) in its
    // shadow; the barrier that publishes them; then P(t - 1).V(t - 1) with the
    // softmax of S(t) in its shadow.  K(t + 1) replaces K(t - 1), read before
    // the previous barrier, and V(t) replaces V(t - 3), read before that
    // barrier too.
    for (int t = 0; t < ntiles; ++t) {
      const int kb = t & 1;
      const int k0 = (PACK ? t % tph : t) * BN;
      const uint64_t kv = kvalid;
      if (HAS_MASK && t + 1 < ntiles) load_mask(t + 1);
      const bool live = t < nlive && (!PACK || t >= t_lo);
      if (PACK && t == t_lo) k_frag(kb, 0);
      f32x16 s[1];
      if (live) {
        // The small products of every k-step first, then the leading ones, in
        // a sum of their own.
        s[0] = f32x16{};
        f32x16 hi;
        constexpr int NQK = 6 * G;
        constexpr int kQT[5] = {0, 1, 0, 2, 1};
#pragma unroll
        for (int n = 0; n < NQK; ++n) {
          if (n < 5 * G) {
            const int g = n / 5, pr = n % 5;
            s[0] = mfma_x3(pr == 0 ? kr[g & 1][0] : (pr < 3 ? kr[g & 1][1] : k0f[g]), qf[g].t[kQT[pr]], s[0]);
            if (pr == 0 && g + 1 < G) k_frag(kb, g + 1);
          } else {
            hi = mfma_x3(k0f[n - 5 * G], qf[n - 5 * G].t[0], n == 5 * G ? f32x16{} : hi);
          }
          // 2 CPT chunks over 6 G = 12 CPT MFMAs: one per six.
          if (n % 6 == 1) stage(n / 6, 0);
          if (n % 6 == 3) stage(n / 6, 1);
          if (n % 6 == 4) stage(n / 6, 2);
          if (n == NQK - 3) v_frag(vb, 0);
          if (n == NQK - 2) v_frag(vb, 1);
          fence();
        }
        s[0] += hi;
      } else {
#pragma unroll
        for (int c = 0; c < 2 * CPT; ++c) {
          stage(c, 0);
          stage(c, 1);
          stage(c, 2);
        }
        if (t == nlive && (!PACK || nlive > t_lo)) {
          v_frag(vb, 0);
          v_frag(vb, 1);
        }
      }
      knext = k_rsrc(t + 3);
      vnext = v_rsrc(t + 2);
      if (t + 1 < ntiles) kvalid = key_bits(t + 1);
      __syncthreads();
      if (live) {
        const bool need_mask = (HAS_MASK && static_cast<uint32_t>(kv) != ~0u) || k0 + BN > SK ||
                               (CAUSAL && k0 + BN - 1 > q0 - off);
        constexpr int N0 = NDB >= 2 ? 4 : 2;  // MFMAs before the exponentials
#pragma unroll
        for (int n = 0; n < N0; ++n) pv_mfma(vb, n);
        fence();
        if (need_mask) apply_mask<1, CAUSAL>(s, k0, kv, qrow - off, h);
        float mt = s[0][0];
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[0][r]);
        mt = max_with_other_half(mt);
        // The reference moves once a row's max passes it by more than 8 (P <=
        // 2^8); the accumulators are rescaled after P.V, in that case only.
        const bool need = mt - m_run > 8.0f;
        const bool rebase = __builtin_amdgcn_ballot_w64(need) != 0;
        const float m_use = need ? mt : m_run;
        const float e_use = m_use == -INFINITY ? 0.0f : m_use;
        Split8 pn[2];
        float ls = 0.0f;
#pragma unroll
        for (int n = N0; n < NPV; ++n) {
          pv_mfma(vb, n);
#pragma unroll
          for (int d = 0; d < 2; ++d) {
            constexpr int R = NPV - N0;
            const int u = (n - N0) * 8 / R + d;
            if (u < (n + 1 - N0) * 8 / R) {
              const float a = fast_exp2(s[0][2 * u] - e_use), c = fast_exp2(s[0][2 * u + 1] - e_use);
              ls += a;
              ls += c;
              split_pair(pn[u >> 2], u & 3, a, c);
            }
          }
          if (n == NPV - 4) k_frag(kb ^ 1, 0);
          fence();
        }
        if (rebase) {
          const float alpha = m_use == m_run ? 1.0f : fast_exp2(m_run - e_use);
          l_run *= alpha;
#pragma unroll
          for (int i = 0; i < NDB; ++i) acc[i] *= alpha;
          m_run = m_use;
        }
        l_run += ls;
#pragma unroll
        for (int j = 0; j < 2; ++j) pk[j] = pn[j];
      } else if (t == nlive && nlive > t_lo) {
#pragma unroll
        for (int n = 0; n < NPV; ++n) pv_mfma(vb, n);
      }
      kput = kb ? kdst + 3 * KPL : kdst;
      vb = vb == 2 ? 0 : vb + 1;
      vput = vb == 2 ? vdst : vput + 3 * VPL;
    }
    if (nlive == ntiles && (!PACK || nlive > t_lo)) {
      // V(ntiles - 1) became visible with the last iteration's barrier.
      v_frag(vb, 0);
      v_frag(vb, 1);
#pragma unroll
      for (int n = 0; n < NPV; ++n) pv_mfma(vb, n);
    }

    // ---- O = acc / l ---------------------------------------------------------
    float* __restrict__ O = static_cast<float*>(p.out) + b * p.ob + hh * p.oh;
    auto store = [&](float lt) __attribute__((always_inline)) {
      const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
      if (qrow < S) {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = acc[db][4 * g + e] * inv;
            *reinterpret_cast<f32x4*>(O + qrow * p.os + 32 * db + 8 * g + 4 * h) = o;
          }
      }
    };
    const float lt = sum_with_other_half(l_run);
    RedoWatch watch;
    watch.see(lt);
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) watch.see(acc[db][r]);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(watch.any()) == 0, 1)) {
      store(lt);
      continue;
    }
    // These rows again on the fp32 MFMA, straight from global memory.
    if (q0 >= S) continue;
    m_run = -INFINITY;
    l_run = 0.0f;
#pragma unroll
    for (int i = 0; i < NDB; ++i) acc[i] = f32x16{};
#pragma unroll 1
    for (int t = 0; t < (PACK ? own : nlive); ++t) {
      const int k0 = t * BN;
      const float* kp = K + static_cast<int64_t>(min(k0 + m, SK - 1)) * p.ks + h;
      const float* qp = Q + static_cast<int64_t>(min(qrow, S - 1)) * p.qs + h;
      f32x16 s[1];
      s[0] = f32x16{};
#pragma unroll 1
      for (int d = 0; d < D; d += 2) s[0] = mfma_f32(kp[d], qp[d] * p.scale_log2, s[0]);
      uint64_t valid = range_bits(k0, SK);
      if constexpr (HAS_MASK) {
        valid = __builtin_amdgcn_ballot_w64(h == 0 && k0 + m < SK && M[(k0 + m) * p.ms] != 0);
      }
      apply_mask<1, CAUSAL>(s, k0, valid, qrow - off, h);
      float mt = s[0][0];
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[0][r]);
      mt = max_with_other_half(mt);
      const float m_new = fmaxf(m_run, mt);
      const float m_use = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = fast_exp2(m_run - m_use);
      float ls = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[0][r] = fast_exp2(s[0][r] - m_use);
        ls += s[0][r];
      }
      l_run = __builtin_fmaf(l_run, alpha, ls);
      m_run = m_new;
#pragma unroll
      for (int i = 0; i < NDB; ++i) acc[i] *= alpha;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + acc_row(r, h);
        const float* vp = V + static_cast<int64_t>(min(key, SK - 1)) * p.vs + m;
#pragma unroll
        for (int i = 0; i < NDB; ++i) acc[i] = mfma_f32(key < SK ? vp[32 * i] : 0.0f, s[0][r], acc[i]);
      }
    }
    store(sum_with_other_half(l_run));
  }
}

// Compute units of the current device (queried once per device).
int device_cu_count() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
      n = 256;
    }
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Key-split plan of a causal 16-bit launch (see AttnParams::split).  When the
// heaviest query tile outweighs the average workgroup slot, the launch lasts
// as long as that workgroup: a query tile that sees more key tiles than the average
// workgroup slot carries is cut into chunks of at most that many (and at
// most 8), and all units are dispatched heaviest first.
struct SplitPlan {
  bool on = false;
  int units = 0;
  int q0 = 0;
  int maxch = 1;
  int64_t cnt_bytes = 0;
  int64_t bytes = 0;
  unsigned short tab[kMaxSplitUnits] = {};
};

// Workgroups of the 16-bit kernel resident per CU (registers / LDS).
int h16_slots_per_cu(int D) { return D >= 128 ? 2 : 3; }

SplitPlan plan_key_split(int dtype, int D, bool causal, int64_t BH, int64_t S) {
  SplitPlan sp;
  if (dtype == 0 || !causal || BH <= 0 || S <= 0) return sp;
  const int64_t nq = (S + kBM - 1) / kBM;
  if (nq < 2 || nq > 1024) return sp;
  const int64_t slots = static_cast<int64_t>(device_cu_count()) * h16_slots_per_cu(D);
  auto tiles = [&](int64_t i) { return (std::min<int64_t>(S, (i + 1) * kBM) + 63) / 64; };
  int64_t total = 0;
  for (int64_t i = 0; i < nq; ++i) total += tiles(i);
  total *= BH;
  const int64_t limit = std::max<int64_t>(8, (total + slots - 1) / slots);
  // Split only when the heaviest query tile carries over 1.5x the average
  // load of a workgroup slot.  Measured on the MI355X: a long-sequence layer
  // (B=4, H=16, S=2048, D=64; 1.41x) ran slower split (62.4 -> 66.6 us: the
  // extra prologues and the state exchange outweigh the shorter tail), as
  // did B=8, H=16, S=1024 (1.33x); B=1, H=4, S=4096 (11.6x) went 51.9 ->
  // 35.4 us and B=2, H=4, S=4096 52.3 -> 42.7 us.
  if (2 * tiles(nq - 1) <= 3 * limit) return sp;
  struct Unit {
    int work, q, c, n;
  };
  Unit units[kMaxSplitUnits];
  int nu = 0;
  int q0 = static_cast<int>(nq);
  for (int64_t i = nq - 1; i >= 0; --i) {
    const int64_t t = tiles(i);
    const int64_t n0 = std::min<int64_t>(8, (t + limit - 1) / limit);
    const int64_t csz = (t + n0 - 1) / n0;
    const int64_t n = (t + csz - 1) / csz;  // every chunk non-empty; ceil(t / n) == csz
    if (n > 1) q0 = static_cast<int>(i);
    for (int64_t c = 0; c < n; ++c) {
      if (nu == kMaxSplitUnits) return SplitPlan{};
      units[nu++] = Unit{static_cast<int>(std::min(t, (c + 1) * csz) - c * csz), static_cast<int>(i),
                         static_cast<int>(c), static_cast<int>(n)};
    }
  }
  std::stable_sort(units, units + nu, [](const Unit& a, const Unit& b) { return a.work > b.work; });
  for (int u = 0; u < nu; ++u) {
    sp.tab[u] = static_cast<unsigned short>(units[u].q | (units[u].c << 10) | ((units[u].n - 1) << 13));
    if (units[u].q == nq - 1) sp.maxch = units[u].n;
  }
  const int64_t nv = ((D + 31) / 32) * 16 + 2;  // floats of partial state per lane
  const int64_t split_tiles = nq - q0;
  // One counter per split slot (batch, head, split query tile), in the fixed
  // block that leads every workspace.
  if (BH * split_tiles > kSplitCounterSlots) return SplitPlan{};
  sp.q0 = q0;
  sp.units = nu;
  sp.cnt_bytes = kSplitCounterBytes;
  sp.bytes = sp.cnt_bytes + BH * split_tiles * sp.maxch * 4 * nv * 64 * 4;
  sp.on = true;
  return sp;
}

template <int D, bool CAUSAL, bool HAS_MASK>
hipError_t launch_d(int dtype, AttnParams& p, void* ws, int64_t ws_bytes, hipStream_t stream) {
  // Causal pairing (fp32 kernel only) halves the grid; use it only while the
  // paired grid still gives every workgroup slot of the GPU (CUs x resident
  // workgroups) one workgroup - below that, the tail of the unpaired grid is
  // cheaper than idle slots.
  const int64_t paired = static_cast<int64_t>((p.nq + 1) / 2) * p.BH;
  p.pair = (dtype == 0 && CAUSAL && p.nq >= 2 &&
            paired >= static_cast<int64_t>(device_cu_count()) * kMinWaves<true, D>) ? 1 : 0;
  p.units = p.pair ? (p.nq + 1) / 2 : p.nq;
  p.cu_count = device_cu_count();
  // Unpaired causal fp32 grid resident in one round (two workgroups per CU):
  // fold the query-tile order so each CU pairs a heavy tile with a light one.
  p.fold = (dtype == 0 && CAUSAL && !p.pair && kMinWaves<true, D> == 2 && p.nq >= 3 &&
            static_cast<int64_t>(p.nq) * p.BH <= 2 * static_cast<int64_t>(p.cu_count) &&
            static_cast<int64_t>(p.nq) * p.BH > static_cast<int64_t>(p.cu_count)) ? 1 : 0;
  // One 64-key tile per head and rows for wavefronts 0-1 only: two heads per
  // workgroup (fp32 non-causal kernels, whose second K/V buffer is free).
  p.twin = (dtype == 0 && D < 32 && !CAUSAL && p.S <= 64) ? 1 : 0;
  // fp32 heads of up to 64 keys, which have rows for one or two wavefronts of
  // a workgroup: up to four or two of them together, once each of them has had
  // a workgroup slot of its own (0: not packed).  The packed kernel has three
  // workgroups per CU at head dim 32, where the plain causal one has two:
  // causal [96, 32, 8, 32] 8.0 -> 6.8 us.
  p.pack = 0;
  if constexpr (D >= 32) {
    if (dtype == 0 && p.S <= 64 && p.BH > p.cu_count * kX3Groups<D>) {
      const int slots = p.cu_count * (D == 32 ? 3 : kX3Groups<D>);
      p.pack = std::min(p.S > 32 ? 2 : 4, (p.BH + slots - 1) / slots);
    }
  }
  p.split = 0;
  if (dtype != 0 && CAUSAL && ws != nullptr) {
    const SplitPlan sp = plan_key_split(dtype, D, true, p.BH, p.S);
    if (sp.on && ws_bytes >= sp.bytes) {
      p.split = 1;
      p.units = sp.units;
      p.split_q0 = sp.q0;
      p.split_tiles = p.nq - sp.q0;
      p.split_maxch = sp.maxch;
      p.ws_cnt = static_cast<int*>(ws);
      p.ws_part = reinterpret_cast<float*>(static_cast<char*>(ws) + sp.cnt_bytes);
      std::copy(sp.tab, sp.tab + sp.units, p.unit_tab);
    }
  }
  if constexpr ((D == 64 || D == 32) && CAUSAL) {
    // 16-bit head_dim 64 and 32, causal, not key-split: 32-key tiles at four
    // workgroups per CU up to S = 1024 (not key-masked head_dim 32, whose
    // 64-key kernel has four workgroups per CU too).
    // Measured against the 64-key kernel (same box, alternating):
    // [16, 512, 16, 64] -13 %, [8, 1024, 16, 64] -4.5 % (key-masked the same
    // time), [4, 2048, 16, 64] +6 % (key-masked +10 to +17 %), key-masked
    // [8, 1500, 16, 64] +4 to +8 %, [1, 8192, 16, 64] +12 %, non-causal
    // launches 6-9 % slower.  Head dim 32: [32, 256, 16, 32] -15 %, [16, 512]
    // -15 %, [8, 1024] -4 %; key-masked [8, 1024, 16, 32] +15 %, [4, 700, 8,
    // 32] +20 %.
    const int bn32_max = HAS_MASK && D == 32 ? 0 : 1024;
    if (dtype != 0 && !p.split && p.S <= bn32_max) {
      const dim3 g(static_cast<unsigned>(p.units) * static_cast<unsigned>(p.BH)), blk(kThreads);
      if (dtype == 1) {
        attn_fwd_h16_kernel<BF16, D, CAUSAL, HAS_MASK, 32><<<g, blk, 0, stream>>>(p);
      } else {
        attn_fwd_h16_kernel<F16, D, CAUSAL, HAS_MASK, 32><<<g, blk, 0, stream>>>(p);
      }
      return hipGetLastError();
    }
  }
  if constexpr (D == 128) {
    // 16-bit head_dim 128, not key-split: 32-key tiles, three workgroups per
    // CU, for causal launches up to S = 4096 and non-causal ones up to 1024.
    // Measured against the 64-key kernel (same box, alternating): causal
    // [16, 512, 16, 128] -19 %, [8, 1024, 16, 128] -9.5 %, [4, 4096, 16, 128]
    // -4 %; non-causal [16, 512, 16, 128] -4 %, [8, 1024, 16, 128] +0.7 %,
    // [4, 2048, 16, 128] +4.6 %, [4, 4096, 16, 128] +4.6 %; causal S = 16384
    // +3.6 %.
    // Key-masked and non-causal from there to 4096, where three workgroups per
    // CU save a round of the grid: without a key span (mask rows of other than
    // unit stride) the 64-key kernel has no whole blocks to run its pipelined
    // body on ([4, 1200, 16, 128] 74.9 us against 63.7, [8, 1800, 16, 128] 256
    // against 244).  With one, the mask decides - prefixes run 1-12 % faster on
    // 64-key tiles, scattered keys 2-15 % slower ([6, 1500, 16, 128] 104.8 us
    // against 113.1 and 147 against 138) - so 32-key tiles are taken only where
    // the second 64-key round would be at most a quarter full: [3, 1500, 16,
    // 128] prefix 65.1 us against 66.1, scattered 95.6 against 82.2; [4, 1200,
    // 16, 128] 54.5 against 57.2, 77.7 against 67.5.  In grids that save no
    // round 64-key tiles win under any mask ([2, 2048, 16, 128] 60.3 against
    // 70.7, 78.7 against 85.2).
    int bn32_max = CAUSAL ? 4096 : 1024;
    if constexpr (HAS_MASK && !CAUSAL) {
      const int64_t groups = static_cast<int64_t>(p.units) * p.BH, cus = p.cu_count;
      const bool saves = (groups + 3 * cus - 1) / (3 * cus) < (groups + 2 * cus - 1) / (2 * cus);
      if (saves && (p.ms != 1 || 2 * groups <= 5 * cus)) bn32_max = 4096;
    }
    if (dtype != 0 && !p.split && p.S <= bn32_max) {
      const dim3 g(static_cast<unsigned>(p.units) * static_cast<unsigned>(p.BH)), blk(kThreads);
      if (dtype == 1) {
        attn_fwd_h16_kernel<BF16, D, CAUSAL, HAS_MASK, 32><<<g, blk, 0, stream>>>(p);
      } else {
        attn_fwd_h16_kernel<F16, D, CAUSAL, HAS_MASK, 32><<<g, blk, 0, stream>>>(p);
      }
      return hipGetLastError();
    }
  }
  if constexpr (!CAUSAL && (D == 32 || D == 64)) {
    // Its buffer resources span rows 0..S-1 of one head, and its lanes
    // address rows 0..63 (rows past S are padding) with 32-bit offsets: rows
    // must not overlap (sequence stride >= head_dim) and the offset of every
    // padded row must stay below 2^31 bytes, or it could wrap back inside the
    // resource instead of reading as zero (or being dropped, for stores).
    auto span_ok = [&](int64_t rs) { return rs >= D && (63 * rs + D) * 4 < (int64_t{1} << 31); };
    if (dtype == 0 && p.S <= 64 && span_ok(p.qs) && span_ok(p.ks) && span_ok(p.vs) && span_ok(p.os) &&
        63 * p.ms < (int64_t{1} << 31) - 1) {
      // Short sequences: one wavefront per (batch, head, 32-query half), a
      // persistent grid of two workgroups per CU (fewer when there are fewer
      // items than wavefronts).
      const int64_t items = static_cast<int64_t>(p.BH) * (p.S > 32 ? 2 : 1);
      const int64_t full = static_cast<int64_t>(p.cu_count) * 2;
      const int64_t groups = std::min<int64_t>((items + 3) / 4, full);
      if (HAS_MASK || p.S < 64) {
        attn_fwd_f32_short_kernel<D, HAS_MASK, true>
            <<<dim3(static_cast<unsigned>(groups)), dim3(kThreads), 0, stream>>>(p);
      } else {
        attn_fwd_f32_short_kernel<D, false, false>
            <<<dim3(static_cast<unsigned>(groups)), dim3(kThreads), 0, stream>>>(p);
      }
      return hipGetLastError();
    }
  }
  const unsigned groups = p.twin ? static_cast<unsigned>((p.BH + 1) / 2)
                                 : static_cast<unsigned>(p.units) * static_cast<unsigned>(p.BH);
  const dim3 g(groups), blk(kThreads);
  switch (dtype) {
    case 0:
      if constexpr (D >= 32) {
        if (p.pack > 0) {
          const dim3 packed(static_cast<unsigned>((p.BH + p.pack - 1) / p.pack));
          attn_fwd_x3_kernel<D, CAUSAL, HAS_MASK, true><<<packed, blk, 0, stream>>>(p);
        } else {
          attn_fwd_x3_kernel<D, CAUSAL, HAS_MASK><<<g, blk, 0, stream>>>(p);
        }
      } else {
        attn_fwd_f32_kernel<D, CAUSAL, HAS_MASK><<<g, blk, 0, stream>>>(p);
      }
      break;
    case 1: attn_fwd_h16_kernel<BF16, D, CAUSAL, HAS_MASK><<<g, blk, 0, stream>>>(p); break;
    case 2: attn_fwd_h16_kernel<F16, D, CAUSAL, HAS_MASK><<<g, blk, 0, stream>>>(p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int D>
hipError_t launch_flags(int dtype, bool causal, bool has_mask, AttnParams& p, void* ws,
                        int64_t ws_bytes, hipStream_t stream) {
  if (causal) {
    return has_mask ? launch_d<D, true, true>(dtype, p, ws, ws_bytes, stream)
                    : launch_d<D, true, false>(dtype, p, ws, ws_bytes, stream);
  }
  return has_mask ? launch_d<D, false, true>(dtype, p, ws, ws_bytes, stream)
                  : launch_d<D, false, false>(dtype, p, ws, ws_bytes, stream);
}

}  // namespace

int attention_block_m(int /*dtype*/, int /*D*/) { return kBM; }

hipError_t launch_attention(int dtype, int D, bool causal, bool has_mask, AttnParams& p,
                            void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  switch (D) {
    case 8: return launch_flags<8>(dtype, causal, has_mask, p, workspace, workspace_bytes, stream);
    case 16: return launch_flags<16>(dtype, causal, has_mask, p, workspace, workspace_bytes, stream);
    case 32: return launch_flags<32>(dtype, causal, has_mask, p, workspace, workspace_bytes, stream);
    case 64: return launch_flags<64>(dtype, causal, has_mask, p, workspace, workspace_bytes, stream);
    case 128: return launch_flags<128>(dtype, causal, has_mask, p, workspace, workspace_bytes, stream);
    default: return hipErrorInvalidValue;
  }
}

int64_t attention_workspace_bytes(int dtype, int D, bool causal, int64_t BH, int64_t S) {
  const SplitPlan sp = plan_key_split(dtype, D, causal, BH, S);
  return sp.on ? sp.bytes : 0;
}

}  // namespace ttk
